"""Split prefill over the range of fp32: finite inputs whose magnitudes lie far
apart -- between the values of a row, between head dims, between rows and
between tiles -- against 64 bits, each output column and each query row by
itself, beside the fp32 launches on the same inputs."""
import sys

import numpy as np
import pytest

from common import D

pytestmark = pytest.mark.gpu

HQ, HKV = 8, 2


def case(msg):
    print(f"[case] {msg}", flush=True)
    sys.stdout.flush()


def attend(monkeypatch, split, q, kc, vc, start):
    import torch

    import bitnetrs_amd

    monkeypatch.setenv("BNR_PREFILL_SPLIT", str(split))
    n, n_heads, n_kv, cap = q.shape[0], q.shape[1] // D, kc.shape[0], kc.shape[1]
    gpu = bitnetrs_amd.HipBackend(0)
    out = torch.zeros_like(q)
    gpu.dev_prefill_attention(q, kc, vc, cap, out, n, start, n_heads, n_kv, D)
    torch.cuda.synchronize()
    gpu.close()
    return out


def attend64(q, kc, vc, start):
    """Rows of q [n, heads * D] over cache rows 0 .. start + i in 64 bits."""
    import torch

    n, n_heads, n_kv, rows = q.shape[0], q.shape[1] // D, kc.shape[0], start + q.shape[0]
    hidden = (torch.arange(rows)[None, :] > start + torch.arange(n)[:, None]).to(q.device)
    out = torch.empty(n, n_heads, D, dtype=torch.float64, device=q.device)
    q = q.double().reshape(n, n_heads, D)
    for h in range(n_heads):
        k, v = kc[h * n_kv // n_heads, :rows].double(), vc[h * n_kv // n_heads, :rows].double()
        s = (q[:, h] @ k.t().contiguous()) / D ** 0.5
        out[:, h] = torch.softmax(s.masked_fill(hidden, float("-inf")), 1) @ v
    return out


def normal(n, start, seed, n_heads=HQ, n_kv=HKV):
    import torch

    g = torch.Generator(device="cuda").manual_seed(seed)
    cap = start + n
    return (torch.randn(n, n_heads * D, device="cuda", generator=g),
            torch.randn(n_kv, cap, D, device="cuda", generator=g),
            torch.randn(n_kv, cap, D, device="cuda", generator=g))


def worst(out, ref, by):
    """The largest relative error (2-norm) of any (head, column) or (row, head)."""
    out = out.double().reshape(ref.shape)
    assert bool(out.isfinite().all()), "not finite"
    dim = 0 if by == "column" else 2
    scale = ref.abs().amax().item() or 1.0  # norms of values near fp32's ends
    d, r = ((out - ref) / scale).norm(dim=dim), (ref / scale).norm(dim=dim)
    return (d / r.clamp_min(1e-300)).max().item()


def check(monkeypatch, q, kc, vc, start, by=("column", "row"), rows=None):
    """The split launch is as close to 64 bits as the fp32 launch (half as much
    again: other orders of the same sums) or within fp32's own rounding of a
    product and a sum, 2^-21."""
    ref = attend64(q, kc, vc, start)
    outs = [attend(monkeypatch, split, q, kc, vc, start).reshape(ref.shape) for split in (0, 1)]
    for b in by:
        e0, e1 = (worst(o[rows] if rows else o, ref[rows] if rows else ref, b) for o in outs)
        print(f"[error] by {b}: fp32 {e0:.2e} split {e1:.2e}", flush=True)
        assert e1 <= max(1.5 * e0, 2.0 ** -21), (b, e0, e1)


# a constant V: the output is that value, whatever is added up on the way
@pytest.mark.parametrize("c", [1e30, 1e33, 1e36, 3e38])
@pytest.mark.parametrize("marked", [False, True])
def test_large_v(monkeypatch, c, marked):
    case(f"split prefill, V of {c}, marked tiles {marked}")
    import torch

    n, start = 1024, 1024
    q, kc, vc = normal(n, start, 11)
    q *= 0.1  # weights spread over all keys
    vc.fill_(c)
    if marked:
        vc[:, ::32] = c * 2.0 ** -20  # rows far apart in every tile
    ref = attend64(q, kc, vc, start)
    out = attend(monkeypatch, 1, q, kc, vc, start)
    assert worst(out, ref, "column") <= 2.0 ** -20 and worst(out, ref, "row") <= 2.0 ** -20


# weights of two to a few keys near one another: the exponentials' arguments
# are rounded near 0, not near the power of two that P is scaled by
def test_exponent_rounding(monkeypatch):
    case("split prefill, rounding of the weights' exponents")
    n, start = 512, 0
    q, kc, vc = normal(n, start, 12)
    q *= 0.25
    ref = attend64(q, kc, vc, start)
    outs = [attend(monkeypatch, s, q, kc, vc, start).reshape(ref.shape) for s in (0, 1)]
    e0, e1 = (((o.double() - ref)[1:32].norm() / ref[1:32].norm()).item() for o in outs)
    print(f"[error] fp32 {e0:.2e} split {e1:.2e}", flush=True)
    # a pair leaves out 2^-22 of a product at most; over 128 dims and 32 keys of
    # either sign it is a quarter of that at most
    assert e1 <= e0 + 2.0 ** -24, (e0, e1)


# tiles that set no scale (zeros) or go through fp32 products (rows far apart)
# before V of another magnitude, at the start of the line and inside it
@pytest.mark.parametrize("scale", [1e-10, 1e-17, 1e-20, 1e-25, 1e-30])
@pytest.mark.parametrize("kind", ["zero", "marked", "both"])
def test_first_tiles(monkeypatch, scale, kind):
    case(f"split prefill, {kind} tiles before V of {scale}")
    n, start = 608, 96
    q, kc, vc = normal(n, start, 13)
    vc *= scale
    for t in (0, 1, 5, 6, 11):
        zero = kind == "zero" or (kind == "both" and t % 2 == 0)
        if zero:
            vc[:, 32 * t:32 * t + 32] = 0
        else:
            vc[:, 32 * t + 7] *= 2.0 ** -20
    check(monkeypatch, q, kc, vc, start)


# a sink: its key takes nearly all of the weight and its value is small or zero
@pytest.mark.parametrize("gap,v", [(12.0, 0.0), (25.0, 0.0), (40.0, 0.0), (6.0, 2.0 ** -9), (9.0, 2.0 ** -13),
                                   (14.0, 2.0 ** -20)])
@pytest.mark.parametrize("rows", [1, 32])
def test_sink(monkeypatch, gap, v, rows):
    case(f"split prefill, {rows} sink rows {gap} above the rest, values {v}")
    n, start = 640, 0
    q, kc, vc = normal(n, start, 14)
    q *= 0.5
    q[:, ::D] = 1.0
    kc[:, :, 0] = 0.0
    kc[:, :rows] = 0.0
    kc[:, :rows, 0] = gap * D ** 0.5
    vc[:, :rows] *= v
    check(monkeypatch, q, kc, vc, start, by=("row",), rows=slice(33, None))


# weights that fall and rise again by more than fp16 holds, from tile to tile
@pytest.mark.parametrize("step", [8.0, 20.0])
def test_weights_apart(monkeypatch, step):
    case(f"split prefill, key tiles {step} apart")
    import torch

    n, start = 640, 64
    q, kc, vc = normal(n, start, 15)
    q *= 0.5
    q[:, ::D] = 1.0
    level = torch.arange(start + n, device="cuda") // 32 % 3  # 0, 1, 2, 0, ...
    kc[:, :, 0] = level * step * D ** 0.5
    vc *= torch.exp2(-level * step * 1.4427)[None, :, None]  # all tiles count
    check(monkeypatch, q, kc, vc, start, by=("column", "row"))


RATIOS = [2.0 ** 14, 2.0 ** 20, 2.0 ** 25, 2.0 ** 30, 2.0 ** 40, 2.0 ** 60]


# V: one head dim far above the rest, some rows, dims spread evenly; by column
# where one dim makes up a row's norm (its sum may be near zero)
@pytest.mark.parametrize("r", RATIOS)
@pytest.mark.parametrize("kind", ["dim", "rows", "spread"])
def test_v_apart(monkeypatch, kind, r):
    case(f"split prefill, V {kind} {r} apart")
    import torch

    n, start = 544, 64
    q, kc, vc = normal(n, start, 16)
    if kind == "dim":
        vc[:, :, 5] *= r
    elif kind == "rows":
        vc[:, ::7] *= r
    else:
        vc *= torch.exp2(torch.linspace(0, 1, D, device="cuda") * float(np.log2(r)))
    check(monkeypatch, q, kc, vc, start, by=("column",) if kind == "dim" else ("column", "row"))


# K: one head dim far above the rest, q zero or as far below the rest there
@pytest.mark.parametrize("r", RATIOS)
@pytest.mark.parametrize("other", ["zero", "inverse"])
def test_k_apart(monkeypatch, other, r):
    case(f"split prefill, a K dim of {r}, q {other}")
    n, start = 544, 64
    q, kc, vc = normal(n, start, 16)
    kc[:, :, 5] *= r
    q.view(n, HQ, D)[:, :, 5] *= 0.0 if other == "zero" else 1 / r
    check(monkeypatch, q, kc, vc, start)


# q: one head dim far above the rest, K zero, as far below the rest or 2^-24 of
# the rest there (the line up to which tiles take q's pairs whatever they lost);
# in every row or in a few
@pytest.mark.parametrize("r", RATIOS)
@pytest.mark.parametrize("other", ["zero", "inverse", "line"])
@pytest.mark.parametrize("every", [1, 50])
def test_q_apart(monkeypatch, other, every, r):
    case(f"split prefill, a q dim of {r} in every {every} rows, K {other}")
    n, start = 544, 64
    q, kc, vc = normal(n, start, 16)
    q.view(n, HQ, D)[::every, :, 5] *= r
    kc[:, :, 5] *= {"zero": 0.0, "inverse": 1 / r, "line": max(1 / r, 2.0 ** -24)}[other]
    if other == "line":  # no value of a tile below 2^-24 of its largest
        import torch

        kc[:] = torch.where(kc.abs() < 0.25 * kc.abs().amax(dim=1, keepdim=True), 0.25 * kc.abs().amax(dim=1, keepdim=True), kc)
    check(monkeypatch, q, kc, vc, start)


# q and K spread evenly over the dims, against one another
@pytest.mark.parametrize("r", RATIOS)
def test_q_and_k_spread(monkeypatch, r):
    case(f"split prefill, q and K spread over {r}")
    import torch

    n, start = 544, 64
    q, kc, vc = normal(n, start, 16)
    spread = torch.exp2(torch.linspace(0, 1, D, device="cuda") * float(np.log2(r)))
    q.view(n, HQ, D).mul_(spread)
    check(monkeypatch, q, kc / spread, vc, start)


# magnitudes at the ends of fp32: products of q and K stay in range
@pytest.mark.parametrize("qs,ks", [(2.0 ** 90, 2.0 ** -90), (2.0 ** -90, 2.0 ** 90), (2.0 ** -110, 2.0 ** 110),
                                   (2.0 ** 110, 2.0 ** -110), (2.0 ** -60, 2.0 ** -60)])
def test_magnitudes(monkeypatch, qs, ks):
    case(f"split prefill, q of {qs}, K of {ks}")
    n, start = 544, 64
    q, kc, vc = normal(n, start, 17)
    check(monkeypatch, q * qs, kc * ks, vc, start)


def test_large_q_and_k_apart(monkeypatch):
    """q and K near 2^100 in head dims where the other is zero: their scales'
    product leaves fp32 although every score is small."""
    case("split prefill, q and K of 2^100 apart")
    n, start = 544, 64
    q, kc, vc = normal(n, start, 18)
    qd = q.view(n, HQ, D)
    qd[:, :, 3] = 2.0 ** 100
    kc[:, :, 3] = 0
    kc[:, :, 4] *= 2.0 ** 100
    qd[:, :, 4] = 0
    check(monkeypatch, q, kc, vc, start)


# every head count per kv head the split kernels are built for
@pytest.mark.parametrize("n_heads,n_kv", [(4, 2), (16, 2), (20, 5)])
def test_heads(monkeypatch, n_heads, n_kv):
    case(f"split prefill error at {n_heads}/{n_kv} heads")
    q, kc, vc = normal(700, 45, 19, n_heads, n_kv)
    check(monkeypatch, q, kc, vc, 45)
