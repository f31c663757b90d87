"""W8A8 linear on the GPU, through the C ABI, against the CPU oracle.

Bar: bit-exact int8 / int32 / scales; bf16 outputs bit-exact (the epilogue
formula fixes every rounding point)."""
import numpy as np
import pytest
import torch

from oracle import oracle as O
from util import bits, from_bits, gemm_inputs

pytestmark = pytest.mark.gpu


def _h3mi():
    import h3mi
    return h3mi


# ------------------------------------------------------------------ quantizer

@pytest.mark.parametrize("M,K", [(1, 8), (37, 256), (64, 3072), (5, 13824), (300, 5120), (3, 32768)])
def test_quant_matches_oracle(M, K):
    h = _h3mi()
    x, _, _, _ = gemm_inputs(M, 8, K, seed=M + K, outliers=0.001)
    if M > 2:
        x[1] = 0                      # all-zero row
        x[2, K // 2] = 3.0e4          # single outlier
    q, s = h.quantize_rowwise(x.cuda())
    oq, os_ = O.quant_rowwise(bits(x))
    assert np.array_equal(q.cpu().numpy(), oq)
    assert np.array_equal(s.cpu().numpy().reshape(-1).view(np.uint32), os_.view(np.uint32))


def _near_half_rows(K, amaxes, seed):
    """Rows whose elements e make fl(e / fl(amax/127)) land on or within 2^-12 of a half-integer: every bf16 value
    in [-amax, amax] is screened in float32 on the CPU and the hits are laid out after the row's amax."""
    g = np.random.default_rng(seed)
    allbits = np.arange(0, 0x8000, dtype=np.uint32) << 16
    vals = allbits.view(np.float32)
    vals = vals[np.isfinite(vals)]
    rows, hits = [], 0
    for amax in amaxes:
        sc = np.float32(amax) / np.float32(127.0)
        c = vals[vals <= np.float32(amax)]
        c = np.concatenate([c, -c])
        qt = (c / sc).astype(np.float32)
        a = np.abs(qt)
        near = np.abs((a - np.trunc(a)) - np.float32(0.5)) < np.float32(2.0 ** -12)
        pick = c[near]
        hits += pick.size
        row = g.choice(pick, size=K) if pick.size else np.zeros(K, np.float32)
        row[0] = np.float32(amax)
        rows.append(row.astype(np.float32))
    x = torch.from_numpy(np.stack(rows)).to(torch.bfloat16)
    assert torch.equal(x.float().abs().amax(1), torch.tensor(amaxes, dtype=torch.float32).to(torch.bfloat16).float())
    return x, hits


@pytest.mark.parametrize("K", [512, 5120, 20480])
def test_quant_near_half_integers(K):
    """The quantizer's fast quotient x * (1/s) must give the IEEE x / s result; these rows consist of the elements
    whose quotients sit on or next to a rounding boundary (ties included), across several scales."""
    h = _h3mi()
    amaxes = [127.0, 100.0, 3.0, 0.75, 1.0e-3, 5.5e4, 2.0 ** -120, 2.0 ** 100]
    x, hits = _near_half_rows(K, amaxes, seed=K)
    assert hits > 100
    q, s = h.quantize_rowwise(x.cuda())
    oq, os_ = O.quant_rowwise(bits(x))
    assert np.array_equal(s.cpu().numpy().reshape(-1).view(np.uint32), os_.view(np.uint32))
    assert np.array_equal(q.cpu().numpy(), oq)


def test_quant_strided_rows():
    h = _h3mi()
    x, _, _, _ = gemm_inputs(40, 8, 512, seed=5)
    big = torch.zeros(40, 640, dtype=torch.bfloat16)
    big[:, :512] = x
    q, s = h.quantize_rowwise(big.cuda()[:, :512])
    oq, os_ = O.quant_rowwise(bits(x))
    assert np.array_equal(q.cpu().numpy(), oq)
    assert np.array_equal(s.cpu().numpy().reshape(-1), os_)


# ------------------------------------------------------------------ GEMM, small/ragged shapes vs oracle

SHAPES = [(1, 4, 128), (37, 72, 256), (64, 64, 128), (300, 260, 384), (257, 520, 1024), (128, 128, 640),
          (512, 10240, 256), (2048, 3072, 3072)]


@pytest.mark.parametrize("M,N,K", SHAPES)
def test_gemm_i32_matches_oracle(M, N, K):
    h = _h3mi()
    g = np.random.default_rng(M * 7 + N)
    a = g.integers(-127, 128, (M, K), dtype=np.int8)
    b = g.integers(-127, 128, (N, K), dtype=np.int8)
    acc = h.int8_mm_i32(torch.from_numpy(a).cuda(), torch.from_numpy(b).cuda()).cpu().numpy()
    ref = O.gemm_i32(a, b)
    assert np.array_equal(acc, ref)


@pytest.mark.parametrize("M,N,K", SHAPES)
def test_gemm_bf16_matches_oracle(M, N, K):
    h = _h3mi()
    x, w, ws, bias = gemm_inputs(M, N, K, seed=M + 3 * N, outliers=0.001)
    ref, oq, os_, acc = O.w8a8_linear(bits(x), w.numpy(), ws.numpy())
    xq = torch.from_numpy(oq).cuda()
    xs = torch.from_numpy(os_).cuda().reshape(M, 1)
    out = h.int8_mm_scaled(xq, w.cuda(), xs, ws.cuda())
    assert np.array_equal(bits(out), ref)
    outb = h.int8_mm_scaled(xq, w.cuda(), xs, ws.cuda(), bias=bias.cuda())
    assert np.array_equal(bits(outb), O.epilogue_bf16(acc, os_, ws.numpy(), bits(bias)))


def test_gemm_extremes_no_overflow():
    h = _h3mi()
    K = 13824
    a = torch.full((64, K), -127, dtype=torch.int8)
    b = torch.full((64, K), -127, dtype=torch.int8)
    b[1::2] = 127
    acc = h.int8_mm_i32(a.cuda(), b.cuda()).cpu()
    assert int(acc[0, 0]) == 127 * 127 * K and int(acc[0, 1]) == -127 * 127 * K


@pytest.mark.parametrize("M,N,K", [(300, 520, 768), (64, 1024, 1280), (257, 388, 2048)])
def test_gemm_leading_dimensions_every_config(M, N, K):
    """Through the C ABI with ldx, ldw > K and ldo > N under every
    configuration: the padding bytes of X and W rows hold large values (a read
    past K would change the sums) and the padding of out a sentinel that must
    survive; the products equal the oracle's on the unpadded operands."""
    from h3mi import _lib as L
    h = _h3mi()
    g = np.random.default_rng(M + N + K)
    ldx, ldw, ldo = K + 48, K + 80, N + 28
    xp = np.full((M, ldx), 127, np.int8)
    wp = np.full((N, ldw), -127, np.int8)
    xp[:, :K] = g.integers(-127, 128, (M, K), dtype=np.int8)
    wp[:, :K] = g.integers(-127, 128, (N, K), dtype=np.int8)
    xs = (0.01 + 0.1 * g.random(M)).astype(np.float32)
    ws = (1e-3 + 9e-3 * g.random(N)).astype(np.float32)
    bias = O.f32_to_bf16_bits((0.02 * g.standard_normal((1, N))).astype(np.float32))[0]
    acc = O.gemm_i32(xp[:, :K], wp[:, :K])
    ref = O.epilogue_bf16(acc, xs, ws, bias)
    xd, wd = torch.from_numpy(xp).cuda(), torch.from_numpy(wp).cuda()
    xsd, wsd = torch.from_numpy(xs).cuda(), torch.from_numpy(ws).cuda()
    bd = torch.from_numpy(bias.view(np.int16)).cuda()
    sentinel = np.int16(0x7F7F)
    try:
        for nm in h.list_configs():
            h.set_config(nm)
            print(f"[ld] {nm} M={M} N={N} K={K}", flush=True)
            out = torch.full((M, ldo), int(sentinel), dtype=torch.int16, device="cuda")
            L.check(L.lib.h3mi_w8a8_gemm_bf16(L.ptr(xd), L.ptr(wd), L.ptr(xsd), L.ptr(wsd), L.ptr(bd), L.ptr(out),
                                              M, N, K, ldx, ldw, ldo, L.stream_of(xd)))
            o = out.cpu().numpy()
            assert np.array_equal(o[:, :N].view(np.uint16), ref), nm
            assert (o[:, N:] == sentinel).all(), nm
            ldc = N + 12
            acc_d = torch.full((M, ldc), -7, dtype=torch.int32, device="cuda")
            L.check(L.lib.h3mi_w8a8_gemm_i32(L.ptr(xd), L.ptr(wd), L.ptr(acc_d), M, N, K, ldx, ldw, ldc,
                                             L.stream_of(xd)))
            a = acc_d.cpu().numpy()
            assert np.array_equal(a[:, :N], acc), nm
            assert (a[:, N:] == -7).all(), nm
    finally:
        h.set_config("auto")


def test_gemm_longest_k_every_config():
    """K = 131072 (1024 K tiles through every configuration's ring): rows of
    -127 against rows of -127 and 127 give sums of +-127^2 K = +-2,114,060,288,
    within 2^31 and exact in fp32 (16129 * 2^17), so the int32 sums and the bf16
    epilogue (xs = ws = 1) are known exactly."""
    h = _h3mi()
    K = 131072
    a = torch.full((64, K), -127, dtype=torch.int8).cuda()
    b = torch.full((96, K), -127, dtype=torch.int8)
    b[1::2] = 127
    b = b.cuda()
    want = torch.tensor([127 * 127 * K, -127 * 127 * K] * 48, dtype=torch.int32).repeat(64, 1)
    one_m = torch.ones(64, 1, dtype=torch.float32, device="cuda")
    one_n = torch.ones(96, dtype=torch.float32, device="cuda")
    want_bf16 = want.float().to(torch.bfloat16)
    try:
        for nm in h.list_configs():
            h.set_config(nm)
            print(f"[long k] {nm}", flush=True)
            assert torch.equal(h.int8_mm_i32(a, b).cpu(), want), nm
            assert torch.equal(h.int8_mm_scaled(a, b, one_m, one_n).cpu(), want_bf16), nm
    finally:
        h.set_config("auto")


@pytest.mark.parametrize("M,N,K", [(300, 520, 768), (1, 4, 128), (257, 260, 128), (64, 1024, 1152)])
def test_every_tile_config_matches(M, N, K):
    h = _h3mi()
    x, w, ws, _ = gemm_inputs(M, N, K, seed=11)
    ref, oq, os_, acc = O.w8a8_linear(bits(x), w.numpy(), ws.numpy())
    xq, xs = torch.from_numpy(oq).cuda(), torch.from_numpy(os_).cuda().reshape(-1, 1)
    names = h.list_configs()
    assert len(names) >= 2
    auto = h.config_for(M, N, K)
    try:
        for nm in names:
            h.set_config(nm)
            # split-K tilings (suffix _k2) take K % 256 == 0 only; other K stay with the heuristic
            assert h.config_for(M, N, K) == (auto if nm.endswith("_k2") and K % 256 else nm)
            assert np.array_equal(h.int8_mm_i32(xq, w.cuda()).cpu().numpy(), acc), nm
            assert np.array_equal(bits(h.int8_mm_scaled(xq, w.cuda(), xs, ws.cuda())), ref), nm
    finally:
        h.set_config("auto")


@pytest.mark.parametrize("M,N,K", [(1, 4, 128), (15, 20, 384), (16, 16, 512), (17, 36, 640), (49, 100, 1152),
                                   (65, 52, 1024), (97, 196, 2176), (37, 1028, 5120)])
def test_wave_split_tilings_match_oracle(M, N, K):
    """Wave-split tilings: one to 40 K slices of 128 bytes over 4 waves of two
    slots each (fewer slices than waves, waves with no slice, odd counts), edges
    of the 16-row blocks and of whole tiles, single rows and columns."""
    h = _h3mi()
    g = np.random.default_rng(M * 11 + N + K)
    xq = g.integers(-127, 128, (M, K), dtype=np.int8)
    w = g.integers(-127, 128, (N, K), dtype=np.int8)
    xs = (0.05 * g.random((M, 1))).astype(np.float32)
    ws = (1e-3 + 9e-3 * g.random(N)).astype(np.float32)
    bias = O.f32_to_bf16_bits((0.02 * g.standard_normal((1, N))).astype(np.float32))[0]
    acc = (xq.astype(np.float64) @ w.astype(np.float64).T).astype(np.int32)
    # operands inside larger buffers whose padding would change the sums if read
    xp, wp = torch.full((M + 1, K + 16), 99, dtype=torch.int8), torch.full((N + 1, K + 48), 77, dtype=torch.int8)
    xp[:M, :K], wp[:N, :K] = torch.from_numpy(xq), torch.from_numpy(w)
    xd, wd, xsd, wsd, bd = (t.cuda() for t in (xp, wp, torch.from_numpy(xs), torch.from_numpy(ws), from_bits(bias)))
    from h3mi._lib import check, lib, ptr, stream_of
    names = [nm for nm in h.list_configs() if nm.startswith("k_")]
    assert len(names) >= 2
    try:
        for nm in names:
            print(f"[wave-split] {nm} M={M} N={N} K={K}", flush=True)
            h.set_config(nm)
            out = torch.full((M, N + 4), 7, dtype=torch.bfloat16, device="cuda")
            check(lib.h3mi_w8a8_gemm_bf16(ptr(xd), ptr(wd), ptr(xsd), ptr(wsd), ptr(bd), ptr(out), M, N, K, K + 16,
                                          K + 48, N + 4, stream_of(xd)))
            assert np.array_equal(bits(out[:, :N]), O.epilogue_bf16(acc, xs, ws, bias)), nm
            assert bool((out[:, N:] == 7).all()), nm
            assert np.array_equal(h.int8_mm_i32(torch.from_numpy(xq).cuda(), torch.from_numpy(w).cuda()).cpu().numpy(),
                                  acc), nm
    finally:
        h.set_config("auto")


SPLITK = ["d_bm128_bn192_bk128_s2_g8_w2x2_sw_k2", "d_bm128_bn128_bk128_s2_g8_w2x2_sw_k2"]


@pytest.mark.parametrize("name", SPLITK)
@pytest.mark.parametrize("M,N,K", [(130, 200, 256), (257, 388, 512), (1, 4, 768), (128, 192, 1024),
                                   (2048, 3072, 3072), (512, 10240, 5120), (300, 4000, 13824)])
def test_split_k_tiling_matches_oracle(name, M, N, K):
    """Split-K tilings: the two K-groups of a workgroup add their int32 partial
    sums through LDS before the epilogue.  One to 27 ring slots of two K tiles,
    ragged M and N edges, a single row, the C0 shape (one tile per CU) and the
    block's cross-attention KV projection (512 x 5120 -> 10240).  int32 against
    an exact float64 product, bf16 with and without bias against the oracle's
    epilogue."""
    h = _h3mi()
    g = np.random.default_rng(M * 7 + N + K)
    xq = g.integers(-127, 128, (M, K), dtype=np.int8)
    w = g.integers(-127, 128, (N, K), dtype=np.int8)
    xs = (0.05 * g.random((M, 1))).astype(np.float32)
    ws = (1e-3 + 9e-3 * g.random(N)).astype(np.float32)
    bias = O.f32_to_bf16_bits((0.02 * g.standard_normal((1, N))).astype(np.float32))[0]
    acc = (xq.astype(np.float64) @ w.astype(np.float64).T).astype(np.int32)
    xd, wd = torch.from_numpy(xq).cuda(), torch.from_numpy(w).cuda()
    xsd, wsd = torch.from_numpy(xs).cuda(), torch.from_numpy(ws).cuda()
    bd = from_bits(bias).cuda()
    print(f"[split-k] {name} M={M} N={N} K={K}", flush=True)
    try:
        h.set_config(name)
        assert h.config_for(M, N, K) == name
        assert np.array_equal(h.int8_mm_i32(xd, wd).cpu().numpy(), acc)
        assert np.array_equal(bits(h.int8_mm_scaled(xd, wd, xsd, wsd)), O.epilogue_bf16(acc, xs, ws))
        assert np.array_equal(bits(h.int8_mm_scaled(xd, wd, xsd, wsd, bias=bd)), O.epilogue_bf16(acc, xs, ws, bias))
    finally:
        h.set_config("auto")


RESIDENT = ["d_bm256_bn384_bk128_s2_g8_w8m_l4_a1_sw_res", "d_bm256_bn256_bk128_s2_g4_w8m_st1_sw_res",
            "d_bm320_bn256_bk128_s2_g4_w8m_st1_sw_res", "d_bm256_bn320_bk128_s2_g4_w4x2_l4_sw_res",
            "d_bm256_bn384_bk128_s2_g4_w8m_l4_a1_sw_res"]


@pytest.mark.parametrize("name", RESIDENT)
@pytest.mark.parametrize("M,N,K", [(12300, 2300, 384), (8200, 3000, 128), (16500, 1540, 256), (40000, 1000, 384)])
def test_resident_tile_loop_matches_oracle(name, M, N, K):
    """Resident configurations: one workgroup per CU loops over 1-3 tiles
    (more tiles than CUs), with the next tile's first K tile loading during
    the epilogue and the ring slots alternating between tiles (K/128 = 1, 2
    or 3 K tiles); ragged M and N edges on both sides.  int32 accumulators
    against an exact float64 product (|acc| <= 127^2 K < 2^53), bf16 with
    and without bias against the oracle's epilogue."""
    h = _h3mi()
    g = np.random.default_rng(M + N + K)
    xq = g.integers(-127, 128, (M, K), dtype=np.int8)
    w = g.integers(-127, 128, (N, K), dtype=np.int8)
    xs = (0.05 * g.random((M, 1))).astype(np.float32)
    ws = (1e-3 + 9e-3 * g.random(N)).astype(np.float32)
    bias = O.f32_to_bf16_bits((0.02 * g.standard_normal((1, N))).astype(np.float32))[0]
    acc = (xq.astype(np.float64) @ w.astype(np.float64).T).astype(np.int32)
    xd, wd = torch.from_numpy(xq).cuda(), torch.from_numpy(w).cuda()
    xsd, wsd = torch.from_numpy(xs).cuda(), torch.from_numpy(ws).cuda()
    bd = from_bits(bias).cuda()
    print(f"[resident] {name} M={M} N={N} K={K}", flush=True)
    try:
        h.set_config(name)
        assert np.array_equal(h.int8_mm_i32(xd, wd).cpu().numpy(), acc)
        assert np.array_equal(bits(h.int8_mm_scaled(xd, wd, xsd, wsd)), O.epilogue_bf16(acc, xs, ws))
        assert np.array_equal(bits(h.int8_mm_scaled(xd, wd, xsd, wsd, bias=bd)), O.epilogue_bf16(acc, xs, ws, bias))
    finally:
        h.set_config("auto")


def test_full_linear_c0_matches_oracle():
    """W8A8 workload C0: X[2048,3072] ~ N(0,1), W[3072,3072], quantize + GEMM + bias."""
    h = _h3mi()
    x, w, ws, bias = gemm_inputs(2048, 3072, 3072, seed=0)
    ref, _, _, _ = O.w8a8_linear(bits(x), w.numpy(), ws.numpy(), bits(bias))
    out = h.w8a8_linear(x.cuda(), w.cuda(), ws.cuda(), bias=bias.cuda())
    assert np.array_equal(bits(out), ref)


# ------------------------------------------------------------------ full-size shapes: properties

@pytest.mark.parametrize("M,N,K", [(32768, 15360, 5120), (32768, 5120, 13824)])
def test_full_size_matches_hipblaslt_and_torch_epilogue(M, N, K):
    """At the workload sizes the CPU oracle is too slow; pin the int32 result
    against torch._int_mm (hipBLASLt, a different implementation) and the bf16
    output against the epilogue computed by separate torch GPU ops (each op a
    single IEEE rounding), on a row sample plus a full-tensor checksum."""
    h = _h3mi()
    g = torch.Generator(device="cuda").manual_seed(M + N)
    xq = torch.randint(-127, 128, (M, K), dtype=torch.int8, device="cuda", generator=g)
    w = torch.randint(-127, 128, (N, K), dtype=torch.int8, device="cuda", generator=g)
    xs = (torch.rand(M, 1, device="cuda", generator=g) * 0.05).contiguous()
    ws = (1e-3 + 9e-3 * torch.rand(N, device="cuda", generator=g)).contiguous()
    acc = h.int8_mm_i32(xq, w)
    ref = torch._int_mm(xq, w.t())
    assert torch.equal(acc, ref)
    out = h.int8_mm_scaled(xq, w, xs, ws)
    ref_out = ((ref.float() * xs) * ws[None, :]).to(torch.bfloat16)
    assert torch.equal(out, ref_out)


def test_allcfg_autotune_picks_a_config_and_keeps_the_bytes(monkeypatch):
    """H3_LINEAR_FAST_ALLCFG=1 (the reference's wider autotune,
    comfyui_nodes/h3-linear-fast/int8_gemm_triton.py:11-21): the first call per
    (N, K, M bucket) times every configuration and caches the fastest; the
    output is the same bytes as the heuristic's."""
    import h3mi
    from h3mi import gemm as G
    M, N, K = 1000, 512, 1024
    g = torch.Generator().manual_seed(5)
    xq = torch.randint(-127, 128, (M, K), generator=g, dtype=torch.int8).cuda()
    w = torch.randint(-127, 128, (N, K), generator=g, dtype=torch.int8).cuda()
    xs = (torch.rand(M, 1, generator=g) * 1e-2).cuda()
    ws = (torch.rand(N, generator=g) * 1e-2).cuda()
    monkeypatch.delenv("H3_LINEAR_FAST_ALLCFG", raising=False)
    ref = h3mi.int8_mm_scaled(xq, w, xs, ws)
    monkeypatch.setenv("H3_LINEAR_FAST_ALLCFG", "1")
    monkeypatch.setattr(G, "_TUNED", {})
    a = h3mi.int8_mm_scaled(xq, w, xs, ws)
    key = (N, K, 1)
    assert key in G._TUNED and G._TUNED[key] in h3mi.list_configs()
    assert G._int8_mm_scaled_kernel.best_config == G._TUNED[key]
    b = h3mi.int8_mm_scaled(xq, w, xs, ws)
    assert torch.equal(a, ref) and torch.equal(b, ref)
    assert h3mi.config_for(M, N, K) == h3mi.config_for(M, N, K)  # the heuristic is restored after each call


@pytest.mark.parametrize("N,ldo,off", [(1000, 1000, 0), (1000, 1028, 0), (1024, 1024, 4), (968, 1024, 0), (1024, 1040, 16), (1024, 1056, 32)])
def test_output_rows_off_half_lines(N, ldo, off):
    """Output rows that start off 64-byte half lines (their length, their stride or
    the first row's address), in an output past the 16 MiB from which they are
    stored through the cache, and rows on them: every configuration writes the
    exact epilogue's bytes, whole tiles and edges, and nothing beside them."""
    h = _h3mi()
    from h3mi._lib import check, lib, ptr, stream_of
    M, K = 8900, 256
    g = torch.Generator(device="cuda").manual_seed(N + ldo + off)
    xq, w = (torch.randint(-127, 128, (r, K), generator=g, device="cuda", dtype=torch.int8) for r in (M, N))
    xs, ws = (torch.rand(r, generator=g, device="cuda") for r in (M, N))
    bias = torch.randn(N, generator=g, device="cuda").to(torch.bfloat16)
    plain = (h.int8_mm_i32(xq, w).float() * xs[:, None]) * ws
    want = {False: plain.to(torch.bfloat16), True: (plain + bias.float()).to(torch.bfloat16)}
    try:
        for name in h.list_configs():
            print(f"[rows off half lines] {name} N={N} ldo={ldo} off={off}", flush=True)
            h.set_config(name)
            for b in (False, True):
                buf = torch.full((M * ldo + off + 64,), 7, dtype=torch.bfloat16, device="cuda")
                out = buf[off:]
                check(lib.h3mi_w8a8_gemm_bf16(ptr(xq), ptr(w), ptr(xs), ptr(ws), ptr(bias) if b else None, ptr(out), M, N, K,
                                              K, K, ldo, stream_of(xq)))
                rows = out[:M * ldo].view(M, ldo)
                assert torch.equal(rows[:, :N], want[b]), (name, b)
                assert bool((rows[:, N:] == 7).all()) and bool((buf[:off] == 7).all()) and bool((out[M * ldo:] == 7).all())
    finally:
        h.set_config("auto")
