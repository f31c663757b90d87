// Waves per row and passes per wave of the ConvRot quantizer for a row of
// `chunks` 1024-element chunks.  Plain host C++, so the rule can be checked
// without a GPU.
#pragma once

#include <stdint.h>

namespace h3mi {

constexpr int kWprs[] = {1, 2, 4, 8};

// Measured at 19200 rows: the registers of more than 3 passes (4 with
// SwiGLU, whose per-element work is larger) cost more occupancy than the
// extra waves' reductions cost, and workgroups of 3, 6 or 7 waves schedule
// worse than 4 or 8 (7 waves x 1 pass at K = 7168, every lane busy: 84.6
// against 74.9 us for 4 x 2 with one pass slot in 8 empty).  So: the fewest wasted pass slots with at most that many
// passes, ties to fewer waves per row; past 8 waves, 8 waves and more passes.
//
// Few rows (up to 6 a CU, 1.5 with SwiGLU, whose waves each wait for the
// workgroup's copy of the table): the fewest passes that 8 waves allow, since a
// wave's passes are a serial chain while most of the chip is idle.  Before ->
// after: K = 5376 37 rows 5.4 -> 4.0 us, 512 6.4 -> 5.4, 1024 8.2 -> 7.5 (2401
// 13.1 -> 13.7); SwiGLU K = 5376 128 rows 7.2 -> 5.6, K = 14336 37 rows 7.8 -> 6.9.
// Not at 9 to 12 chunks, where 8 waves of 2 passes leave 4 to 7 pass slots of 16
// empty and 4 of 3 none to 3 of 12 (SwiGLU K = 9216 to 12288: 7-9% behind at 96
// to 256 rows; without, 3-12%), and with SwiGLU at 5 and 6 chunks only up to one
// row a CU: there the other shape holds two rows in a workgroup, which keeps one
// workgroup a CU, and 8 waves a row were 5-14% behind at 288 to 384 rows (K = 5376
// 384 rows 8.5 against 9.1 us).
inline void convrot_shape(int chunks, bool swiglu, int64_t rows, int64_t cus, int* wpr, int* passes) {
    const int64_t most = !swiglu ? 6 * cus : chunks == 5 || chunks == 6 ? cus : 3 * cus / 2;
    const bool few = rows <= most && !(chunks > 8 && chunks <= 12);
    const int pmax = few ? (chunks + 7) / 8 : swiglu ? 4 : 3;
    int best_w = 8, best_p = (chunks + 7) / 8, best_slots = 1 << 30;
    for (int w : kWprs) {
        const int p = (chunks + w - 1) / w;
        if (p > pmax) continue;
        if (p * w < best_slots) best_w = w, best_p = p, best_slots = p * w;
    }
    *wpr = best_w;
    *passes = best_p;
}

}  // namespace h3mi
