"""The fused norms' two routes give the same bytes: a call of many rows (the
row streams) against the same rows in calls of few (one row per workgroup,
which the other norm tests hold against the oracle), on either side of the
lines between them (test_norm_routes.py reads the lines), with rows whose table
index is out of range (left unwritten)."""
import numpy as np
import pytest
import torch

from util import norm_inputs

pytestmark = pytest.mark.gpu

EPS = 1e-6
OPS = ["norm_mod", "norm_mod_q", "gate_norm_mod_", "gate_norm_mod_q_", "gate_"]


def _calls(h, x, w, s1, sh, g, o, ridx):
    """Every norm of the rows: outputs start from a fill, so unwritten rows show."""
    s, n = x.shape
    new = lambda: torch.full_like(x, 3)
    outs = []
    hx = new()
    _, var, rstd = h.norm_mod_ex(x, w, EPS, ridx, s1, sh, stats=True, h=hx)
    ok = (ridx >= 0) & (ridx < s1.shape[0])
    outs += [hx, var[ok], rstd[ok]]
    xa, ha = x.clone(), new()
    h.gate_norm_mod_ex(xa, o, g, w, EPS, ridx, s1, sh, h=ha)
    outs += [xa, ha, h.gate_(x.clone(), o, g, ridx)]
    if n % 8 == 0 and n <= 8192:
        for want in (False, True):
            outs += [t[ok] for t in h.norm_mod_q(x, w, EPS, ridx, s1, sh, want_h=want)]
            xb = x.clone()
            outs += [xb] + [t[ok] for t in h.gate_norm_mod_q_(xb, o, g, w, EPS, ridx, s1, sh, want_h=want)]
    return outs


@pytest.mark.parametrize("S,N,R", [(5125, 8, 1), (5125, 520, 1), (5121, 1032, 1), (5121, 2048, 1), (5600, 3072, 1),
                                   (5000, 5376, 1), (8200, 5120, 1), (3100, 8192, 1), (4800, 5376, 2), (6500, 5376, 2),
                                   (1500, 264, 5), (9800, 3584, 3)])
def test_streams_and_rows_agree(S, N, R):
    import h3mi as h
    x, w, s1, sh, g, o, ridx = norm_inputs(S, N, R, seed=S + N, stress=True)
    if R > 1:
        ridx = (torch.arange(S) * R // S).to(torch.int32)
        ridx[S // 2], ridx[S - 1] = -1, R
    x, w, s1, sh, g, o, ridx = (t.cuda() for t in (x, w, s1, sh, g, o, ridx))
    print(f"[routes] S={S} N={N} R={R}", flush=True)
    whole = _calls(h, x, w, s1, sh, g, o, ridx)
    step = 700
    parts = [_calls(h, x[i:i + step].contiguous(), w, s1, sh, g, o[i:i + step].contiguous(), ridx[i:i + step].contiguous())
             for i in range(0, S, step)]
    for k, t in enumerate(whole):
        ref = torch.cat([p[k] for p in parts])
        assert torch.equal(t.contiguous().view(torch.uint8), ref.contiguous().view(torch.uint8)), k
    if R > 1:  # out-of-range rows keep the fill and x
        assert bool((whole[0][S // 2] == 3).all()) and torch.equal(whole[5][S // 2], x[S // 2])


# (S, N, R) at which the named calls run their streams: test_norm_routes.py
# asserts it.
STREAMS = [
    (8200, 5120, 1, OPS),                                                  # gate_norm_split_kernel, no tail
    (7900, 5376, 1, OPS),                                                  # ... with its 256-element tail
    (8300, 5384, 1, OPS),                                                  # the wave-per-row stream of every norm
    (6001, 520, 1, ["norm_mod", "norm_mod_q", "gate_norm_mod_", "gate_norm_mod_q_"]),
    (8001, 520, 2, ["norm_mod_q"]),                                        # narrow rows over two table rows
    (10301, 1544, 2, ["gate_norm_mod_"]),
    (11001, 2568, 3, ["norm_mod", "norm_mod_q", "gate_norm_mod_"]),
    (11001, 2560, 2, ["norm_mod", "norm_mod_q", "gate_norm_mod_", "gate_norm_mod_q_"]),
    (20001, 5376, 3, ["norm_mod", "norm_mod_q", "gate_norm_mod_q_"]),      # past 100 Mi elements
]


@pytest.mark.parametrize("S,N,R", [c[:3] for c in STREAMS])
def test_streams_with_out_of_range_rows(S, N, R):
    """The streams' per-row table look-up: rows of several table rows in runs of
    unequal length, and rows out of range, single ones, a run, and a workgroup's
    first and last, which it would stage."""
    import h3mi as h
    g = torch.Generator(device="cuda").manual_seed(S + N)
    x, o = (torch.randn(S, N, generator=g, device="cuda").to(torch.bfloat16) for _ in range(2))
    w = torch.randn(N, generator=g, device="cuda").to(torch.bfloat16)
    s1, sh, gt = (torch.randn(R, N, generator=g, device="cuda").to(torch.bfloat16) for _ in range(3))
    rows = torch.arange(S, device="cuda")
    ridx = torch.where(rows < S // 3, 0, torch.where(rows < S // 2, 1, 2)).clamp_(max=R - 1).to(torch.int32)
    for bad in (rows % 97 == 3, (rows > S // 4) & (rows < S // 4 + 300), rows < 40, rows >= S - 40):
        ridx[bad] = torch.where(rows[bad] % 2 == 0, -1, R).to(torch.int32)
    print(f"[streams] S={S} N={N} R={R}", flush=True)
    whole = _calls(h, x, w, s1, sh, gt, o, ridx)
    step = 700
    parts = [_calls(h, x[i:i + step].contiguous(), w, s1, sh, gt, o[i:i + step].contiguous(), ridx[i:i + step].contiguous())
             for i in range(0, S, step)]
    for k, t in enumerate(whole):
        ref = torch.cat([p[k] for p in parts])
        assert torch.equal(t.contiguous().view(torch.uint8), ref.contiguous().view(torch.uint8)), k
    out = (ridx < 0) | (ridx >= R)
    assert bool((whole[0][out] == 3).all()) and torch.equal(whole[5][out], x[out])


@pytest.mark.parametrize("R", [1, 5])
def test_more_rows_than_workgroups_of_one_launch(R):
    """2^24 + 5 narrow rows: a workgroup of 256 threads each would be more than 2^32 threads."""
    import h3mi as h
    S, N, tail = (1 << 24) + 5, 8, 4096
    print(f"[routes] S={S} N={N} R={R}", flush=True)
    g = torch.Generator(device="cuda").manual_seed(R)
    x, o = (torch.randn(S, N, generator=g, device="cuda").to(torch.bfloat16) for _ in range(2))
    w, s1, sh, gt = (torch.randn(r, N, generator=g, device="cuda").to(torch.bfloat16) for r in (1, R, R, R))
    w = w.reshape(-1)
    ridx = (torch.arange(S, device="cuda") * R // S).to(torch.int32)

    def calls(x, o, ridx):
        a, b, c = x.clone(), x.clone(), x.clone()
        return [h.norm_mod(x, w, EPS, ridx, s1, sh), h.gate_norm_mod_(a, o, gt, w, EPS, ridx, s1, sh), a,
                *h.norm_mod_q(x, w, EPS, ridx, s1, sh), *h.gate_norm_mod_q_(b, o, gt, w, EPS, ridx, s1, sh), b,
                h.gate_(c, o, gt, ridx)]

    whole = calls(x, o, ridx)
    for part in (slice(0, tail), slice(S - tail, S)):
        for k, (a, b) in enumerate(zip(whole, calls(x[part].contiguous(), o[part].contiguous(), ridx[part].contiguous()))):
            assert torch.equal(a[part].contiguous().view(torch.uint8), b.view(torch.uint8)), (k, part)
