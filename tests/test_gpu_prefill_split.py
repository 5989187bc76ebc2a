"""Split prefill (fp16 pairs in place of fp32 operands): edges of its tiles,
units and runs against the oracle, its error against 64 bits beside the fp32
kernels', and the tiles that it takes with fp32 products."""
import sys

import numpy as np
import pytest

import oracle
from common import D, HKV, HQ, THETA, assert_close_scaled, oracle_prefill, prefill_workload

pytestmark = pytest.mark.gpu


def case(msg):
    print(f"[case] {msg}", flush=True)
    sys.stdout.flush()


def dev(a):
    import torch

    return torch.from_numpy(np.ascontiguousarray(a)).to("cuda")


def host(t):
    import torch

    torch.cuda.synchronize()
    return t.cpu().numpy()


def make_backend(monkeypatch, split):
    import bitnetrs_amd

    monkeypatch.setenv("BNR_PREFILL_SPLIT", str(split))
    return bitnetrs_amd.HipBackend(0)


# (heads, kv heads, cached rows, launches in a row): one query, a unit and one
# more or fewer, one and several key tiles, runs that end inside a unit, 2, 4
# and 8 q heads per kv head (128, 32 and 32 queries a unit), a partial first tile
@pytest.mark.parametrize("n_heads,n_kv,start,lens", [
    (20, 5, 0, (1, 31, 32, 33)), (20, 5, 45, (333, 1, 300)), (20, 5, 640, (16, 700)),
    (8, 4, 7, (63, 65, 129, 400)), (16, 2, 45, (32, 333, 47)), (4, 1, 100, (900,))])
def test_split_prefill_shapes(monkeypatch, n_heads, n_kv, start, lens):
    case(f"split prefill heads {n_heads}/{n_kv} start {start} lens {lens}")
    import torch

    gpu = make_backend(monkeypatch, 1)
    try:
        cap = start + sum(lens) + 9
        cache = oracle.KVCache(1, n_kv, D, cap)
        be = oracle.CpuBackend()
        kc = torch.zeros(n_kv, cap, D, device="cuda")
        vc = torch.zeros_like(kc)
        if start:
            oracle_prefill(prefill_workload(51, start, n_heads, n_kv), cache=cache, backend=be,
                           n_heads=n_heads, n_kv=n_kv)
            kc.copy_(torch.from_numpy(cache.k(0).reshape(n_kv, cap, D)))
            vc.copy_(torch.from_numpy(cache.v(0).reshape(n_kv, cap, D)))
        for i, n in enumerate(lens):
            w = prefill_workload(52 + i, n, n_heads, n_kv)
            q_ref, k_ref, cache, out_ref = oracle_prefill(w, start_pos=start, cache=cache, backend=be,
                                                          n_heads=n_heads, n_kv=n_kv)
            q, k = dev(w["q"]), dev(w["k"])
            out = torch.zeros(n, n_heads * D, device="cuda")
            gpu.dev_prefill(q, k, dev(w["v"]), n, start, n_heads, n_kv, D, THETA, kc, vc, cap, out)
            np.testing.assert_array_equal(host(q), q_ref)
            np.testing.assert_array_equal(host(k), k_ref)
            np.testing.assert_array_equal(host(kc).reshape(-1), cache.k(0))
            np.testing.assert_array_equal(host(vc).reshape(-1), cache.v(0))
            assert_close_scaled(host(out), out_ref, f"split {n_heads}/{n_kv} n {n} start {start}")
            # attention alone, over the rows just cached
            again = torch.zeros_like(out)
            gpu.dev_prefill_attention(q, kc, vc, cap, again, n, start, n_heads, n_kv, D)
            assert_close_scaled(host(again), out_ref, f"split attention n {n} start {start}")
            start += n
    finally:
        gpu.close()


def attend64(q, kc, vc, start):
    """Rows of q [n, HQ * D] over cache rows 0 .. start + i in 64 bits."""
    import torch

    n, g, rows = q.shape[0], HQ // HKV, start + q.shape[0]
    hidden = torch.arange(rows)[None, :] > start + torch.arange(n)[:, None]
    out = torch.empty(n, HQ, D, dtype=torch.float64)
    q, kc, vc = q.double().cpu().reshape(n, HQ, D), kc.double().cpu(), vc.double().cpu()
    for h in range(HQ):
        s = (q[:, h] @ kc[h // g, :rows].t()) / D ** 0.5
        out[:, h] = torch.softmax(s.masked_fill(hidden, float("-inf")), 1) @ vc[h // g, :rows]
    return out.reshape(n, HQ * D)


# scales of q, k and v, cached rows and their scale against the new ones': the
# exponents that the pairs are scaled by, V tiles on both sides of what O's
# scale allows, magnitudes far from 1
@pytest.mark.parametrize("qs,ks,vs,start,ps", [(1, 1, 1, 0, 1), (4, 1, 1, 96, 1), (1, 1e-12, 1e-15, 45, 1),
                                               (1e-3, 1e3, 1e20, 64, 1), (1, 1, 1, 320, 2.0 ** -12),
                                               (1, 1, 1, 320, 2.0 ** 12), (1, 1, 1, 320, 1e-30)])
def test_split_error_against_64_bits(monkeypatch, qs, ks, vs, start, ps):
    """Error of split and fp32 launches on the same inputs: the split one is
    no further off (a fifth of slack: sums over another order of tiles)."""
    case(f"split prefill error, scales {qs} {ks} {vs}, start {start} at {ps}")
    import torch

    n, cap = 600, 1024
    g = torch.Generator(device="cuda").manual_seed(97)
    q0 = torch.randn(n, HQ * D, device="cuda", generator=g) * qs
    kc0 = torch.randn(HKV, cap, D, device="cuda", generator=g) * ks
    vc0 = torch.randn(HKV, cap, D, device="cuda", generator=g) * vs
    vc0[:, :start] *= ps
    ref = attend64(q0, kc0, vc0, start)
    err = {}
    for split in (0, 1):
        gpu = make_backend(monkeypatch, split)
        out = torch.zeros(n, HQ * D, device="cuda")
        gpu.dev_prefill_attention(q0, kc0, vc0, cap, out, n, start, HQ, HKV, D)
        err[split] = ((out.double().cpu() - ref).norm() / ref.norm()).item()
        gpu.close()
    assert err[1] <= 1.2 * err[0] and err[1] < 2e-6, err


def test_split_marked_tiles(monkeypatch):
    """Tiles with an infinity or a NaN, and V rows 2^20 apart, go through fp32
    products: NaN where the fp32 kernels give NaN, the same values elsewhere.
    Queries before such a tile are not touched by it."""
    case("split prefill, marked tiles")
    import torch

    n, cap = 640, 640
    g = torch.Generator(device="cuda").manual_seed(98)
    q = torch.randn(n, HQ * D, device="cuda", generator=g)
    kc = torch.randn(HKV, cap, D, device="cuda", generator=g)
    vc = torch.randn(HKV, cap, D, device="cuda", generator=g)
    kc[0, 70, 5] = float("-inf")          # a weight of 0 or NaN, by the sign of q's dim 5
    kc[1, 200] *= 2.0 ** -20              # rows far apart in K ...
    vc[1, 300:310] *= 2.0 ** -20          # ... and in V
    vc[2, 400, 7] = float("inf")
    kc[3, 500, 9] = float("nan")
    outs = []
    for split in (0, 1):
        gpu = make_backend(monkeypatch, split)
        out = torch.zeros(n, HQ * D, device="cuda")
        gpu.dev_prefill_attention(q, kc, vc, cap, out, n, 0, HQ, HKV, D)
        outs.append(host(out).reshape(n, HQ, D))
        gpu.close()
    a, b = outs
    for kv in range(HKV):
        # every row, those before a non-finite one in its own tile too: a masked
        # key's weight of 0 times its infinity is a NaN in either launch
        x, y = a[:, 4 * kv:4 * kv + 4], b[:, 4 * kv:4 * kv + 4]
        np.testing.assert_array_equal(np.isnan(x), np.isnan(y))
        np.testing.assert_array_equal(np.isinf(x), np.isinf(y))
        ok = np.isfinite(x)
        assert_close_scaled(y[ok], x[ok], f"kv head {kv}")
    assert np.isnan(b[384:400, 8:12, 7]).all()
    assert np.isfinite(b[:64]).all() and np.isfinite(b[:, 4:8]).all()
    assert np.isnan(b[70:, 0:4]).any() and np.isinf(b[400:, 8:12]).any() and np.isnan(b[500:, 12:16]).any()
