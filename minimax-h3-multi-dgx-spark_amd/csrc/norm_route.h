// Which kernels a call of the fused norms or of gate_ runs (rows of N <= 8192
// elements, N % 8 == 0, the default order): one row per workgroup of 256
// threads (norm_row_kernel, gate_row_kernel) or the persistent row streams.
// Plain host C++, so the rules can be checked without a GPU.
#pragma once

#include <stdint.h>

namespace h3mi {

// A launch of S workgroups of 256 threads must stay below 2^32 threads, which
// HIP refuses; the streams' grids do not grow with S, so they take longer calls
// at every width and number of table rows.
inline bool rows_launchable(int64_t S) { return S < (int64_t{1} << 24); }

// The norms.  Lines between the two routes, each measured on both sides over N
// 8 to 8192, 600 to 200000 rows in one to five runs of table rows, inputs
// rotated past the caches (us below: streams against one row per workgroup).
//
// One table row: the streams win once the tensors come from memory, at about
// 16 Mi elements (20 with the quantizer, whose streams have less of a row in
// flight: 4800 x 5120 23.0 against 23.3; 24 past N = 5632, where they run 16
// chunks a lane), and past about 20 rows per CU, where a workgroup per row costs
// by its row whatever the row's width.
//
// Several table rows: a stream stages one of them and reads the others' from L2
// behind each row's x, so the lines move out, the further the more table rows.
// Narrow rows keep a line in rows for the quantizing norm (N = 512 over two:
// 7200 12.7 against 12.6, 9600 15.1 against 15.7, 38400 41.9 against 52.8).
//
// gate_norm_mod_'s stream is gate_norm_split_kernel at widths of 1024 k and
// 1024 k + 256: a workgroup per row and CU, behind at any S with N <= 2048
// (38400 x 1024: 105.4 against 63.6) or several table rows.  At the other widths
// it is the wave-per-row stream, which wins there with many rows (38400 x 1536
// over one 86.6 against 115.5; 19200 x 2560 over two 80.9 against 89.7).
inline bool norm_rows_suit(bool gate, bool quant, int64_t S, int64_t N, int64_t R) {
    if (!rows_launchable(S)) return false;
    const int64_t mi = S * N >> 20;
    if (gate && !quant) {
        const bool split = N >= 1024 && (N % 1024 == 0 || N % 1024 == 256);
        if (split && (R > 1 || N <= 2048)) return true;
        if (R == 1) return S <= 5120 && mi < 16;
        if (N > 1024 && N < 2048) return R > 2 || S <= 10240;
        return N < 2048 || N > 4096 || S <= 3600 * R;
    }
    if (gate) {
        if (R == 1) return S <= 5120 && mi < 24;
        if (N > 1536 && N < 4608 && S > (N > 2048 ? 5400 : 12000) * R) return false;
        return R > 3 || mi < 100;
    }
    if (quant) {
        if (R == 1) return S <= 5120 && mi < (N > 5632 ? 24 : 20);
        if (N <= 1024) return S <= 7680;
        if (R <= 3 && N > 2048 && N <= 5632) return S <= 10240 && mi < 28;
        return mi < 32;
    }
    return R == 1 ? S <= 5120 && mi < 16 : R > 3 || mi < 24;
}

// gate_: one row per workgroup, except over one table row for wide rows that
// come from memory: 19200 x 5376 107 against 102 us for the stream, 4800 x 5376
// 25 against 30, 19200 x 3072 63 against 75.
inline bool gate_rows_suit(int64_t S, int64_t N, int64_t R) {
    return rows_launchable(S) && (R > 1 || N <= 4096 || S * N <= int64_t{40} << 20);
}

}  // namespace h3mi
