// W8A8 GEMM for outputs too small to fill the chip with operand-sharing
// tiles: a few rows of X against a whole weight, or any small M x N.
//
// A workgroup computes a small output tile (16 MF rows of X by 16 NF rows of
// W) over the whole K, and its KW waves split K: wave w multiplies the
// 128-byte K slices w, w + KW, ... into its own int32 accumulators, so the
// workgroup reads KW * 128 contiguous bytes of every row at a time.  No
// operand byte is used by two waves, so each wave has a ring of S slices of its
// own in LDS and the K loop has no barrier: a wave waits for its own slice,
// reads it into registers, sends out the load that refills the slot and
// multiplies.  The waves' partial sums meet in LDS once, at the end (int32,
// exact: the bytes equal every other tiling's).
//
// What bounds it: for M up to 16 the stream of W from memory (10240 x 5120 W,
// 52 MB, M = 16: 13.2 us; at the rate of a device copy 10.3), above that the
// bytes per CU into LDS (17-18 TB/s over the chip), so the tile grows with the
// grid (pick_config).  Against the 128x128 tiles that these sizes ran before,
// which left most CUs idle or ran one wave per SIMD: M = 37, 10240 x 5120
// 14.3 from 35 us; M = 37, 3072 x 3072 5.4 from 17.5; M = 16, 5120 x 13824 15
// from 79; M = 256, 3072 x 3072 8.6 from 17.4 (bf16 output, graph replays over
// rotating weights).
//
// v_mfma_i32_16x16x64_i8: the 16-row block is what a few rows of X fill.  The
// operands pass through LDS, although no wave shares them, because a fragment
// is 16 bytes of each of 16 rows: loaded straight into registers, 16
// consecutive lanes touch 16 cache lines (28 against 14.3 us at M = 37,
// 10240 x 5120), while an LDS-DMA load takes whole 128-byte lines of 8 rows.
// Four waves and two slices: 8 waves, or 3 and 4 slices, leave room for fewer
// workgroups per CU and measured the same or up to 15% slower.
#pragma once

template <int MF_, int NF_, int KW_ = 4, int S_ = 2>
struct KTile {
    static constexpr int MF = MF_, NF = NF_, KW = KW_, S = S_;
    static constexpr int BM = 16 * MF_, BN = 16 * NF_, NT = 64 * KW_;
    static constexpr int F = MF_ * NF_;                   // 16x16 blocks of the tile
    static constexpr int CH = F < KW_ ? F : KW_;          // blocks summed per hand-off round, one per wave
    static constexpr int SLOT = (MF_ + NF_) * 2048;       // one K slice of the tile's rows
    static constexpr int LPT = 2 * (MF_ + NF_);           // its 1 KiB loads
    static constexpr int RING = KW_ * S_ * SLOT;
    static constexpr int LDS = RING > KW_ * CH * 1024 ? RING : KW_ * CH * 1024;
    static constexpr int OCC = 160 * 1024 / LDS;          // workgroups per CU, by LDS
    static constexpr int WPE = KW_ * OCC / 4 > 8 ? 8 : KW_ * OCC / 4;
    static_assert(KW_ % 4 == 0 && LDS <= 160 * 1024, "whole SIMDs, within the LDS");
    static_assert(LPT * (S_ - 1) <= 63, "vmcnt range");
};

template <class T, bool OUT_I32>
__global__ __launch_bounds__(T::NT) __attribute__((amdgpu_waves_per_eu(T::WPE, T::WPE))) void w8a8_gemm_kwave_kernel(
    const int8_t* __restrict__ X, const int8_t* __restrict__ W, const float* __restrict__ xs,
    const float* __restrict__ ws, const uint16_t* __restrict__ bias, void* __restrict__ out, int M, int N, int K,
    int ldx, int ldw, int64_t ldo, int tiles_m, int tiles_n) {
#if defined(__HIP_DEVICE_COMPILE__)
    constexpr int KW = T::KW, S = T::S, MF = T::MF, NF = T::NF;
    __shared__ __attribute__((aligned(1024))) uint8_t lds[T::LDS];
    const int lane = threadIdx.x & 63, wid = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int lr = lane & 15, lq = lane >> 4;
    int tm, tn;
    tile_coords<16>(blockIdx.x, tiles_m, tiles_n, tm, tn);
    const int m0 = tm * T::BM, n0 = tn * T::BN;
    // The tile's rows only, so that a row past M or N, and the offset kNone of
    // a slice past this wave's last, is out of range and reads zero
    // (ld * 128 < kNone: gemm_entry).
    constexpr int kNone = 0x40000000;
    const int mr = min(M - m0, T::BM), nr = min(N - n0, T::BN);
    const __amdgpu_buffer_rsrc_t rx =
        make_rsrc(X + static_cast<int64_t>(m0) * ldx, static_cast<int64_t>(mr - 1) * ldx + K);
    const __amdgpu_buffer_rsrc_t rw =
        make_rsrc(W + static_cast<int64_t>(n0) * ldw, static_cast<int64_t>(nr - 1) * ldw + K);
    // Load j of an operand fills rows 8j .. 8j+7 of its part of the slot, lane
    // l the chunk that the swizzle places at row 8j + l/8, slot l%8.  Four
    // loads share one LDS base and step with the instruction offset, which is
    // taken back out of the global offset (8 rows of at least 128 bytes).
    const int slices = K / 128;
    const int mine = wid < slices ? (slices - wid + KW - 1) / KW : 0;
    int vw[2 * NF], vx[2 * MF];
    static_for<2 * NF>([&](auto j_c) {
        constexpr int j = decltype(j_c)::value;
        const int row = 8 * j + (lane >> 3);
        vw[j] = row * ldw + swz<8, true>(row, lane & 7) * 16 - (j & 3) * 1024;
    });
    static_for<2 * MF>([&](auto j_c) {
        constexpr int j = decltype(j_c)::value;
        const int row = 8 * j + (lane >> 3);
        vx[j] = row * ldx + swz<8, true>(row, lane & 7) * 16 - (j & 3) * 1024;
    });
    uint8_t* const ring = lds + wid * S * T::SLOT;
    auto issue = [&](int i, int slot) {
        const bool in = i < mine;  // uniform
        const int k = in ? (i * KW + wid) * 128 : 0;
        uint8_t* base = ring + slot * T::SLOT;
        static_for<2 * NF>([&](auto j_c) {
            constexpr int j = decltype(j_c)::value;
            __builtin_amdgcn_raw_ptr_buffer_load_lds(rw, (lds_ptr_t)(base + (j & ~3) * 1024), 16, in ? vw[j] : kNone, k,
                                                     (j & 3) * 1024, 0);
        });
        static_for<2 * MF>([&](auto j_c) {
            constexpr int j = decltype(j_c)::value;
            __builtin_amdgcn_raw_ptr_buffer_load_lds(rx, (lds_ptr_t)(base + NF * 2048 + (j & ~3) * 1024), 16,
                                                     in ? vx[j] : kNone, k, (j & 3) * 1024, 0);
        });
    };
    // Fragment f of an operand: rows 16f .. 16f+15, this lane's row lr; the
    // swizzle does not depend on f.
    const int o0 = lr * 128 + swz<8, true>(lr, lq) * 16, o1 = lr * 128 + swz<8, true>(lr, 4 + lq) * 16;
    v4i acc[NF][MF];
#pragma unroll
    for (int i = 0; i < NF; ++i)
#pragma unroll
        for (int j = 0; j < MF; ++j) acc[i][j] = v4i{};
    static_for<S>([&](auto s_c) { issue(decltype(s_c)::value, decltype(s_c)::value); });
    for (int i0 = 0; i0 < mine; i0 += S) {
        static_for<S>([&](auto s_c) {
            constexpr int slot = decltype(s_c)::value;
            const uint8_t* base = ring + slot * T::SLOT;
            v4i a[2][NF], b[2][MF];
            wait_vm<T::LPT*(S - 1)>();  // this slot's slice has landed
            asm volatile("" ::: "memory");
#pragma unroll
            for (int f = 0; f < NF; ++f) {
                a[0][f] = *reinterpret_cast<const v4i*>(base + f * 2048 + o0);
                a[1][f] = *reinterpret_cast<const v4i*>(base + f * 2048 + o1);
            }
#pragma unroll
            for (int f = 0; f < MF; ++f) {
                b[0][f] = *reinterpret_cast<const v4i*>(base + (NF + f) * 2048 + o0);
                b[1][f] = *reinterpret_cast<const v4i*>(base + (NF + f) * 2048 + o1);
            }
            wait_lgkm0();  // the slice is in registers: its slot can be filled again
            asm volatile("" ::: "memory");
            issue(i0 + S + slot, slot);
#pragma unroll
            for (int ks = 0; ks < 2; ++ks)
#pragma unroll
                for (int i = 0; i < NF; ++i)
#pragma unroll
                    for (int j = 0; j < MF; ++j)
                        acc[i][j] = __builtin_amdgcn_mfma_i32_16x16x64_i8(a[ks][i], b[ks][j], acc[i][j], 0, 0, 0);
            __builtin_amdgcn_sched_barrier(0);
        });
    }
    wait_vm<0>();  // (the slices past this wave's last, of zeros)
    wg_barrier();  // the ring is free for the hand-off
    uint8_t* const part = lds;

    // Block c of the tile (NF x MF, m fastest) is summed by wave c % KW: every
    // wave leaves its partial block in LDS, and that wave adds the KW of them.
    // A lane holds 4 consecutive n of one row m, as in the other tilings.
    static_for<(T::F + T::CH - 1) / T::CH>([&](auto r_c) {
        constexpr int r0 = decltype(r_c)::value * T::CH;
        if constexpr (r0 > 0) wg_barrier();  // the previous round's sums have been read
        static_for<T::CH>([&](auto c_c) {
            constexpr int c = r0 + decltype(c_c)::value;
            if constexpr (c < T::F)
                *reinterpret_cast<v4i*>(part + (wid * T::CH + (c - r0)) * 1024 + lane * 16) = acc[c / MF][c % MF];
        });
        wait_lgkm0();
        wg_barrier();
        const int c = r0 + wid;
        if (wid < T::CH && c < T::F) {  // uniform
            v4i s = {};
#pragma unroll
            for (int w = 0; w < KW; ++w)
                s += *reinterpret_cast<const v4i*>(part + (w * T::CH + wid) * 1024 + lane * 16);
            const int m = m0 + (c % MF) * 16 + lr, n = n0 + (c / MF) * 16 + lq * 4;
            if (m < M && n < N) {
#pragma clang fp contract(off)  // the products and the bias add round separately
                if constexpr (OUT_I32) {
                    *reinterpret_cast<v4i*>(static_cast<int32_t*>(out) + static_cast<int64_t>(m) * ldo + n) = s;
                } else {
                    const float sx = xs[m];
                    const float4 sw = *reinterpret_cast<const float4*>(ws + n);
                    float v0 = (static_cast<float>(s[0]) * sx) * sw.x;
                    float v1 = (static_cast<float>(s[1]) * sx) * sw.y;
                    float v2 = (static_cast<float>(s[2]) * sx) * sw.z;
                    float v3 = (static_cast<float>(s[3]) * sx) * sw.w;
                    if (bias) {
                        const uint2 bb = *reinterpret_cast<const uint2*>(bias + n);
                        v0 = v0 + bf16_lo(bb.x);
                        v1 = v1 + bf16_hi(bb.x);
                        v2 = v2 + bf16_lo(bb.y);
                        v3 = v3 + bf16_hi(bb.y);
                    }
                    *reinterpret_cast<uint2*>(static_cast<uint16_t*>(out) + static_cast<int64_t>(m) * ldo + n) =
                        make_uint2(bf16x2_bits(v0, v1), bf16x2_bits(v2, v3));
                }
            }
        }
    });
#endif
}
