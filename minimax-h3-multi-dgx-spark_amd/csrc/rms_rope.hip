// q/k RMSNorm + split-half rotary embedding, in place, for gfx950.
//
// Replaces comfy-kitchen's ck.rms_rope_split_half_(q, k, rope_freqs, qw, kw,
// epsilon, rot_dim) as the reference calls it on the [1, s, heads, dim] views
// of the qkv projection (comfyui_nodes/minimax-h3-sp/minimax_sp/
// sp_forward.py:279-296; table from rope_rotation_table, :548).  comfy-kitchen's
// arithmetic is not published with the reference; this kernel implements the
// eager sequence the fused call stands for, bit for bit:
//   y = bf16(w * (rstd * x)) per (token, head) row of D elements -- F.rms_norm
//       of the row: in-thread sequential sums of squares over 4-element
//       chunks, a shuffle tree over the chunks, rstd = rsqrt(tot / D + eps);
//   for i < rot/2, R = tab[token][i] (2 x 2, bf16):
//       out[i]         = bf16(R00 y[i] + R01 y[i + rot/2])
//       out[i + rot/2] = bf16(R10 y[i] + R11 y[i + rot/2])
//     (products and sum each rounded in fp32); out[j] = y[j] for j >= rot.
//
// Layout: a row of D = 8 * LPR elements is LPR lanes x 8 contiguous elements
// (one 16-byte load and store per lane); a wave holds 64 / LPR rows at a time
// and NIT such sets; rows run (token, q heads, k heads), so a wave's rows
// mostly share one token's table.  The
// sum-of-squares order of PyTorch's rms_norm (256 logical threads, 4-element
// chunks, 64-wide shuffle-down tree, then the cross-warp tree) puts chunk t
// in thread t; only D/4 <= 64 threads hold data, so the tree reduces to: lane
// l holds chunks 2l and 2l+1, butterflies over lanes l ^ LPR/2, ..., l ^ 1 sum
// each parity class, and the total is even + odd.  Sums with the zero
// partials of the other threads are exact and are skipped.  The rotation
// partner of element i (< rot/2) sits in the same slot of lane l + rot/16.
#include <type_traits>

#include "common.h"

namespace h3mi {
namespace {

typedef uint32_t v4u_t __attribute__((ext_vector_type(4)));

// n / d for n < 2^31 and d >= 2: (n * mul) >> 32 >> shift, with mul =
// ceil(2^(31+l) / d), 2^(l-1) < d <= 2^l and shift = l - 1 (mul exceeds the
// quotient by less than 1, so the product by less than 2^31 / 2^(31+l) <= 1 / d).
struct Div {
    uint32_t d, mul;
    int shift;
    __device__ __forceinline__ uint32_t operator()(uint32_t n) const { return __umulhi(n, mul) >> shift; }
};

inline Div make_div(uint32_t d) {
    int l = 1;
    while ((uint64_t{1} << l) < d) ++l;
    return {d, static_cast<uint32_t>(((uint64_t{1} << (31 + l)) + d - 1) / d), l - 1};
}

// v of lane l ^ M as a DPP source (no LDS): M = 1 and 2 within 4 lanes, M = 8 the
// rotation by 8 of 16.  For M = 4 the rotation by 4, which reads lane l ^ 4 or
// l ^ 12: for values that lanes 8 apart share.
template <int M>
__device__ __forceinline__ float dpp_xor(float v) {
    constexpr int ctrl = M == 1 ? 0xB1 : M == 2 ? 0x4E : M == 4 ? 0x124 : 0x128;
    static_assert(M == 1 || M == 2 || M == 4 || M == 8, "DPP pattern");
    return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), ctrl, 0xF, 0xF, true));
}

// v plus the v of lane l ^ M, in a butterfly over LPR lanes from LPR / 2 down (so
// that from M = 4 down, lanes 2 M apart hold the same v).
template <int LPR, int M>
__device__ __forceinline__ float butterfly(float v) {
    if constexpr (M == 16 || (M == 4 && LPR == 8)) return v + __shfl_xor(v, M, 64);
    else return v + dpp_xor<M>(v);
}

// One wave handles NIT sets of 64 / LPR rows; every load of the wave is
// issued before the first row is reduced, so a wave keeps NIT x 1 KiB of rows
// in flight.  Branches around memory operations make the compiler drain all
// loads at the join, so a row past the end loads the workgroup's first row instead (unused) and
// only the stores test the row.  RSTD (the per-row rstd output) is for tests;
// ROPE: 0 no rotation (rot = 0), 2 full rotation (rot = D), 1 partial, 3 partial
// with the partner 8 lanes away (rot = 128, D = 256); RN
// selects the correctly rounded rsqrt (else the hardware one, as eager).
//
// The weights (q's then k's) and the table rows of the workgroup's tokens are
// staged in LDS as fp32, the table as four planes of rot/2 coefficients per
// token (R00, R01, R10, R11), so a lane takes its eight pairs' two coefficients
// as four 16-byte reads, ready to multiply.  Four floats between the planes put
// the lower and the upper lanes' reads, 32 bytes apart within a plane, on
// different banks (12 heads of 256 with rot = 128, 2401 tokens 16.3 -> 14.7 us,
// 9600 46.3 -> 43.0).  Loaded per row instead, each
// lane's own eight table words, a wave held 32 registers of them and fetched
// each table line eight times (and one way or the other waited for them before
// the next set's rows went out).  The reduction and, where the partner is 8 lanes
// away, its value are DPP sources; over the LDS crossbar their latency showed
// (19200 tokens of 56 x 128 196 against 182 us; 12 heads of 256 with rot = 128,
// 2401 tokens 14.7 against 14.2).  With the one launch for every row count (the
// rest of the rows was a second, guarded one), before -> after: 56 x 128 37 tokens
// 11.1 -> 3.2 us, 512 8.9 -> 7.5, 2401 32.9 -> 26.4; 12 x 256 with rot = 128, 2401
// tokens 20.0 -> 14.1; long launches, bound by memory (56 x 128 19200 tokens 181
// us, 6.1 TB/s), the same within 2%.
template <int LPR, int NIT, bool RSTD, int ROPE, bool RN>
__global__ __launch_bounds__(256) void rms_rope_kernel(uint16_t* __restrict__ q, uint16_t* __restrict__ k,
                                                       const uint16_t* __restrict__ tab,
                                                       const uint16_t* __restrict__ qw,
                                                       const uint16_t* __restrict__ kw, int S, int H, Div per_tok,
                                                       int64_t ldq, int64_t ldk, int rot, float eps,
                                                       float* __restrict__ rstd_out) {
#pragma clang fp contract(off)
    constexpr int D = LPR * 8;
    constexpr int RPW = 64 / LPR;
    constexpr int RPB = 4 * RPW * NIT;
    static_assert(D <= 256, "one weight element per thread of the workgroup");
    extern __shared__ __attribute__((aligned(16))) float smem[];
    float* const wsh = smem;          // [2][D]
    float* const tsh = smem + 2 * D;  // [tokens][4][rot / 2]
    const int lane = threadIdx.x & 63;
    const int sub = lane % LPR;
    const uint32_t rows = static_cast<uint32_t>(S) * per_tok.d;  // < 2^31 (checked by the caller)
    const uint32_t block0 = blockIdx.x * static_cast<uint32_t>(RPB);
    const uint32_t row0 = block0 + (threadIdx.x >> 6) * (RPW * NIT) + lane / LPR;
    const uint32_t tok0 = per_tok(block0);  // uniform: the workgroup's first token
    // rotation: lanes [0, rot/16) of a row hold the first halves, [rot/16,
    // rot/8) the second halves, the partner lane rot/16 away
    const int hl = rot / 16, half = rot / 2, plane = half + 4;  // floats from one plane to the next
    const bool lower = sub < hl;
    const bool rotated = ROPE == 2 || sub < 2 * hl;
    const int src = rotated ? (lower ? lane + hl : lane - hl) : lane;
    const int pair0 = rotated ? (lower ? sub : sub - hl) * 8 : 0;

    // the weights and the table first (loads complete in order): thread t takes
    // element t % D of both weights (threads past D write the same values again)
    const int wt = static_cast<int>(threadIdx.x) % D;
    const uint16_t wq1 = qw[wt], wk1 = kw[wt];
    const int last = static_cast<int>(per_tok(min(block0 + RPB, rows) - 1) - tok0);  // of its tokens
    const uint2* const pt = reinterpret_cast<const uint2*>(tab) + static_cast<int64_t>(tok0) * half;
    const int pairs = ROPE > 0 ? (last + 1) * half : 0;
    uint2 t0 = make_uint2(0u, 0u);
    if (ROPE > 0 && static_cast<int>(threadIdx.x) < pairs) t0 = pt[threadIdx.x];
    __builtin_amdgcn_sched_barrier(0);  // moved behind the rows' loads, their wait would drain them all

    bool in[NIT], isk[NIT];
    uint32_t rel[NIT];
    uint16_t* px[NIT];
    v4u_t xv[NIT];
#pragma unroll
    for (int it = 0; it < NIT; ++it) {
        const uint32_t row = row0 + it * RPW;
        in[it] = row < rows;
        const uint32_t r = in[it] ? row : block0;
        const uint32_t tok = per_tok(r);
        const int j = static_cast<int>(r - tok * per_tok.d);
        rel[it] = tok - tok0;
        isk[it] = j >= H;
        px[it] = (isk[it] ? k + static_cast<int64_t>(tok) * ldk : q + static_cast<int64_t>(tok) * ldq) +
                 static_cast<int64_t>(isk[it] ? j - H : j) * D + sub * 8;
        xv[it] = __builtin_nontemporal_load(reinterpret_cast<const v4u_t*>(px[it]));
    }
    __builtin_amdgcn_sched_barrier(0);  // every load above is issued before any row is reduced
    wsh[wt] = bf16_f32(wq1);
    wsh[D + wt] = bf16_f32(wk1);
    if constexpr (ROPE > 0) {
        auto stage = [&](int p, uint2 w) {
            float* const d = tsh + (p / half) * 4 * plane + p % half;
            d[0] = bf16_lo(w.x);
            d[plane] = bf16_hi(w.x);
            d[2 * plane] = bf16_lo(w.y);
            d[3 * plane] = bf16_hi(w.y);
        };
        if (static_cast<int>(threadIdx.x) < pairs) stage(threadIdx.x, t0);
        for (int p = threadIdx.x + 256; p < pairs; p += 256) stage(p, pt[p]);  // few heads: many tokens
    }
    wait_lgkm0();  // the writes are done
    wg_barrier();

#pragma unroll
    for (int it = 0; it < NIT; ++it) {
        float x[8];
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            x[2 * i] = bf16_lo(xv[it][i]);
            x[2 * i + 1] = bf16_hi(xv[it][i]);
        }
        // chunks 2*sub (elements 0..3 of the lane) and 2*sub + 1 (4..7)
        float pe = x[0] * x[0], po = x[4] * x[4];
#pragma unroll
        for (int i = 1; i < 4; ++i) {
            pe = pe + x[i] * x[i];
            po = po + x[4 + i] * x[4 + i];
        }
        auto both = [&](auto m_c) {
            constexpr int M = decltype(m_c)::value;
            if constexpr (M < LPR) {
                pe = butterfly<LPR, M>(pe);
                po = butterfly<LPR, M>(po);
            }
        };
        both(std::integral_constant<int, 16>{});
        both(std::integral_constant<int, 8>{});
        both(std::integral_constant<int, 4>{});
        both(std::integral_constant<int, 2>{});
        both(std::integral_constant<int, 1>{});
        // D is a power of two: the product by 1/D is the IEEE quotient
        const float var = (pe + po) * (1.0f / static_cast<float>(D)) + eps;
        const float rstd = RN ? rsqrt_rn(var) : rsqrtf(var);
        if constexpr (RSTD) {
            if (in[it] && sub == 0) rstd_out[row0 + it * RPW] = rstd;
        }

        const float* wr = wsh + (isk[it] ? D : 0) + sub * 8;
        const float4 w0 = *reinterpret_cast<const float4*>(wr), w1 = *reinterpret_cast<const float4*>(wr + 4);
        const float wf[8] = {w0.x, w0.y, w0.z, w0.w, w1.x, w1.y, w1.z, w1.w};
        float y[8];
#pragma unroll
        for (int i = 0; i < 8; ++i) y[i] = wf[i] * (rstd * x[i]);
#pragma unroll
        for (int i = 0; i < 4; ++i) rb2(y[2 * i], y[2 * i + 1]);
        if constexpr (ROPE > 0) {
            // lower lane: out = R00 y + R01 p; upper lane: R10 p + R11 y, the
            // same sum in the other order
            const float* tr = tsh + rel[it] * 4 * plane + pair0;
            const float* const po_ = tr + (lower ? 0 : 3 * plane);
            const float* const pp_ = tr + (lower ? plane : 2 * plane);
            const float4 o0 = *reinterpret_cast<const float4*>(po_), o1 = *reinterpret_cast<const float4*>(po_ + 4);
            const float4 q0 = *reinterpret_cast<const float4*>(pp_), q1 = *reinterpret_cast<const float4*>(pp_ + 4);
            const float co[8] = {o0.x, o0.y, o0.z, o0.w, o1.x, o1.y, o1.z, o1.w};
            const float cp[8] = {q0.x, q0.y, q0.z, q0.w, q1.x, q1.y, q1.z, q1.w};
            float p[8];
#pragma unroll
            for (int i = 0; i < 8; ++i) {
                if constexpr (ROPE == 3 || (ROPE == 2 && LPR == 16)) p[i] = dpp_xor<8>(y[i]);  // rot / 16 = 8 lanes apart
                else p[i] = __shfl(y[i], src, 64);
            }
#pragma unroll
            for (int i = 0; i < 8; ++i) {
                const float u = co[i] * y[i];
                const float v = cp[i] * p[i];
                y[i] = rotated ? u + v : y[i];
            }
        }
        v4u_t ov;
#pragma unroll
        for (int i = 0; i < 4; ++i) ov[i] = bf16x2_bits(y[2 * i], y[2 * i + 1]);
        // opaque: else the compiler moves the rotation into the store's branch
        asm volatile("" : "+v"(ov));
        if (in[it]) __builtin_nontemporal_store(ov, reinterpret_cast<v4u_t*>(px[it]));
    }
}

}  // namespace
}  // namespace h3mi

using namespace h3mi;

extern "C" int h3mi_rms_rope_split_half_bf16(uint16_t* q, uint16_t* k, const uint16_t* tab, const uint16_t* qw,
                                             const uint16_t* kw, int64_t S, int64_t H, int64_t D, int64_t ldq,
                                             int64_t ldk, int64_t rot, float eps, int rsqrt_mode_,
                                             float* rstd_out, void* stream) {
    if (S < 0 || H <= 0) return fail(H3MI_EINVAL, "rms_rope: bad sizes S=%lld H=%lld", (long long)S, (long long)H);
    if (D != 64 && D != 128 && D != 256) return fail(H3MI_EINVAL, "rms_rope: head dim %lld (64, 128 or 256)", (long long)D);
    if (rot < 0 || rot > D || rot % 16) return fail(H3MI_EINVAL, "rms_rope: rot_dim %lld must be a multiple of 16 in [0, %lld]",
                                                    (long long)rot, (long long)D);
    if (rsqrt_mode_ != H3MI_RSQRT_HW && rsqrt_mode_ != H3MI_RSQRT_RN) return fail(H3MI_EINVAL, "rms_rope: unknown rsqrt mode");
    if (ldq < H * D || ldk < H * D || ldq % 8 || ldk % 8)
        return fail(H3MI_EALIGN, "rms_rope: token strides must be >= heads*dim and multiples of 8");
    if (S * 2 * H > 0x7FFFFFFF || H > 0x3FFFFFFF) return fail(H3MI_EINVAL, "rms_rope: more than 2^31 rows");
    if (S == 0) return ok();
    if (!q || !k || !qw || !kw || (rot && !tab)) return fail(H3MI_EINVAL, "rms_rope: null pointer");
    if (!aligned(q, 16) || !aligned(k, 16) || !aligned(qw, 16) || !aligned(kw, 16) || (rot && !aligned(tab, 16)) ||
        (rstd_out && !aligned(rstd_out, 4)))
        return fail(H3MI_EALIGN, "rms_rope: q, k, weights and table need 16-byte alignment");
    const size_t qb = static_cast<size_t>((S - 1) * ldq + H * D) * 2, kb = static_cast<size_t>((S - 1) * ldk + H * D) * 2;
    const size_t tb = static_cast<size_t>(S * rot / 2 * 4) * 2, wb = static_cast<size_t>(D) * 2;
    // q and k may interleave in one qkv buffer: then every token's q heads and
    // every token's k heads must be disjoint, i.e. equal strides and the k
    // offset (mod the stride) at least H*D elements from q on both sides
    if (overlap(q, qb, k, kb)) {
        const intptr_t db = reinterpret_cast<const char*>(k) - reinterpret_cast<const char*>(q);
        const int64_t hd = H * D;
        if (ldq != ldk || db % 2) return fail(H3MI_EALIAS, "rms_rope: q and k overlap");
        const int64_t dm = ((db / 2) % ldq + ldq) % ldq;
        if (dm < hd || dm > ldq - hd) return fail(H3MI_EALIAS, "rms_rope: q and k heads overlap");
    }
    if ((rot && (overlap(q, qb, tab, tb) || overlap(k, kb, tab, tb))) || overlap(q, qb, qw, wb) || overlap(q, qb, kw, wb) ||
        overlap(k, kb, qw, wb) || overlap(k, kb, kw, wb))
        return fail(H3MI_EALIAS, "rms_rope: q/k overlap the table or the weights");
    if (rstd_out) {
        const size_t rb_ = static_cast<size_t>(S * 2 * H) * 4;
        if (overlap(rstd_out, rb_, q, qb) || overlap(rstd_out, rb_, k, kb)) return fail(H3MI_EALIAS, "rms_rope: rstd_out overlaps q/k");
    }
    const int lpr = static_cast<int>(D / 8);
    const int64_t rows = S * 2 * H;
    const Div per_tok = make_div(static_cast<uint32_t>(2 * H));
    // Four sets of rows per wave, or two where four would leave a CU fewer than
    // four workgroups (512 tokens of 56 x 128 7.9 against 8.8 us, 37 4.3 against
    // 4.7; 1024 14.2 against 13.5; before the DPP sources).
    const bool few = rows / (16 * (64 / lpr)) < 4 * static_cast<int64_t>(cu_count());
    auto run4 = [&](auto lpr_c, auto rstd_c, auto rope_c, auto rn_c, auto nit_c) {
        constexpr int L = decltype(lpr_c)::value, NIT = decltype(nit_c)::value, P = decltype(rope_c)::value;
        constexpr bool R = decltype(rstd_c)::value, N = decltype(rn_c)::value;
        constexpr int64_t rows_per_block = 4 * (64 / L) * NIT;
        const unsigned blocks = static_cast<unsigned>((rows + rows_per_block - 1) / rows_per_block);
        // the weights, and the table rows of as many tokens as a workgroup's rows can touch
        const int64_t toks = (rows_per_block - 2) / (2 * H) + 2;
        size_t lds = static_cast<size_t>(2 * D + (rot ? toks * 4 * (rot / 2 + 4) : 0)) * sizeof(float);
        // Rows that come from memory stream faster with five workgroups per CU
        // than with the seven that the registers allow, so the LDS of a long
        // launch is padded: 19200 tokens of 56 x 128 181.5 against 187.5 us, 40 x 128
        // 136.1 against 142.8, 12 x 256 79.8 against 81.4, 9600 of 56 x 128 91.5
        // against 93.9.
        if (rows * D * 2 >= int64_t{48} << 20 && lds < 32768) lds = 32768;
        hipLaunchKernelGGL((rms_rope_kernel<L, NIT, R, P, N>), dim3(blocks), dim3(256), lds, as_stream(stream), q, k, tab,
                           qw, kw, static_cast<int>(S), static_cast<int>(H), per_tok, ldq, ldk, static_cast<int>(rot), eps,
                           rstd_out);
    };
    auto run3 = [&](auto lpr_c, auto rstd_c, auto rope_c, auto rn_c) {
        if (few) run4(lpr_c, rstd_c, rope_c, rn_c, std::integral_constant<int, 2>{});
        else run4(lpr_c, rstd_c, rope_c, rn_c, std::integral_constant<int, 4>{});
    };
    using T = std::true_type;
    using F = std::false_type;
    auto run2 = [&](auto lpr_c, auto rstd_c, auto rope_c) {
        if (rsqrt_mode_ == H3MI_RSQRT_RN) run3(lpr_c, rstd_c, rope_c, T{});
        else run3(lpr_c, rstd_c, rope_c, F{});
    };
    using R0 = std::integral_constant<int, 0>;
    using R1 = std::integral_constant<int, 1>;
    using R2 = std::integral_constant<int, 2>;
    using R3 = std::integral_constant<int, 3>;
    auto run1 = [&](auto lpr_c, auto rstd_c) {
        if constexpr (decltype(lpr_c)::value == 32) {
            if (rot == 128) return run2(lpr_c, rstd_c, R3{});
        }
        if (rot == D) run2(lpr_c, rstd_c, R2{});
        else if (rot) run2(lpr_c, rstd_c, R1{});
        else run2(lpr_c, rstd_c, R0{});
    };
    auto run = [&](auto lpr_c) {
        if (rstd_out) run1(lpr_c, T{});
        else run1(lpr_c, F{});
    };
    if (lpr == 8) run(std::integral_constant<int, 8>{});
    else if (lpr == 16) run(std::integral_constant<int, 16>{});
    else run(std::integral_constant<int, 32>{});
    return check_launch("rms_rope_kernel");
}
