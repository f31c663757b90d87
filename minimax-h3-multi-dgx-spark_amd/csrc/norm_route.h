// Which kernels a call of the fused norms or of gate_ runs (rows of N <= 8192
// elements, N % 8 == 0, the default order): one row per workgroup of 256
// threads (norm_row_kernel, gate_row_kernel) or the persistent row streams.
// Plain host C++, so the rules can be checked without a GPU.
#pragma once

#include <stdint.h>

namespace h3mi {

// A launch of S workgroups of 256 threads must stay below 2^32 threads, which
// HIP refuses; the streams' grids do not grow with S.
inline bool rows_launchable(int64_t S) { return S < (int64_t{1} << 24); }

// The norms.  With one table row the streams win once the tensors come from
// memory (with inputs rotated past the caches the two meet at about 16 Mi
// elements, 24 Mi with the quantizer, whose streams have less of a row in
// flight), and, in rows narrower than a workgroup, past about 20 rows per CU
// (at N = 512 9600 rows: norm_mod 12.5 against 14.0 us, norm_mod_q 16.8 against
// 14.6); gate_norm_mod_'s own stream, a workgroup per row and CU, is behind at
// any S for N = 1024 to 2048 (38400 x 1024: 106.7 against 67.9).  With several
// table rows a stream reads most rows' tables from L2 after their x, and the
// lines move: 38400 x 5376 over five, gate_norm_mod_ 470 against 323 us,
// gate_norm_mod_q_ 380 against 325, norm_mod 209 against 201, but norm_mod_q 170
// against 188; over two, gate_norm_mod_ 361 against 325, gate_norm_mod_q_ 175
// against 172 at 19200 rows and 303 against 319 at 38400, norm_mod 30.4 against
// 28.7 at 4800 and 52 against 57 at 9600.
inline bool norm_rows_suit(bool gate, bool quant, int64_t S, int64_t N, int64_t R) {
    if (!rows_launchable(S)) return false;
    const int64_t mi = S * N >> 20;
    if (R > 1) {
        if (gate) return !quant || R > 3 || mi < 100;
        return quant ? mi < 32 : R > 3 || mi < 24;
    }
    if (gate && !quant && N >= 1024 && N <= 2048) return true;
    return S <= 5120 && mi < (quant ? 24 : 16);
}

// gate_: one row per workgroup, except over one table row for wide rows that
// come from memory: 19200 x 5376 107 against 102 us for the stream, 4800 x 5376
// 25 against 30, 19200 x 3072 63 against 75.
inline bool gate_rows_suit(int64_t S, int64_t N, int64_t R) {
    return rows_launchable(S) && (R > 1 || N <= 4096 || S * N <= int64_t{40} << 20);
}

}  // namespace h3mi
