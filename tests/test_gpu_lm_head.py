"""GPU parity of the i8-weight LM head (Backend::lm_head_matmul_i8_into)
against the oracle, through the C ABI.  fp32 sums in a different order than
the reference's AVX2 lanes: each logit must lie within the fp32 rounding
bound of the exact (fp64) value, 4*K*eps*sum|w*h|*scale, and within
|gpu - oracle| <= 2e-3 + 1e-3*|oracle|."""
import sys

import numpy as np
import pytest

import oracle

pytestmark = pytest.mark.gpu
f32 = np.float32


def case(msg):
    print(f"[gpu case] {msg}", flush=True)
    sys.stdout.flush()


def workload(seed, v, h):
    rng = np.random.default_rng(seed)
    hid = rng.standard_normal(h).astype(f32)
    w = rng.integers(-128, 128, size=(v, h)).astype(np.int8)
    sc = rng.uniform(0.001, 0.03, size=v).astype(f32)
    return hid, w, sc


def check(got, hid, w, sc):
    v, h = w.shape
    ref = np.full(v, np.nan, f32)
    oracle.lm_head_matmul_i8(hid, w, sc, ref, v, h)
    exact = (w.astype(np.float64) @ hid.astype(np.float64)) * sc
    mag = (np.abs(w).astype(np.float64) @ np.abs(hid).astype(np.float64)) * sc
    bound = 4 * max(h, 1) * np.finfo(f32).eps * mag + 1e-30
    assert np.all(np.abs(got.astype(np.float64) - exact) <= bound)
    err = np.abs(got - ref)
    assert np.all(err <= 2e-3 + 1e-3 * np.abs(ref)), float(err.max())
    return float(err.max())


@pytest.mark.parametrize("v,h", [(128256, 2560), (1000, 2560), (129, 100), (300, 4100), (7, 9000)])
def test_host_lm_head(backend, v, h):
    case(f"lm head host vocab {v} hidden {h}")
    hid, w, sc = workload(v + h, v, h)
    out = np.full(v, np.nan, f32)
    backend.lm_head_matmul_i8_into(hid, w.reshape(-1), sc, out, v, h)
    print(f"max |gpu - oracle| {check(out, hid, w, sc):.3e}")


@pytest.mark.parametrize("v,h,offset", [(128256, 2560, 0), (5000, 2560, 4), (333, 2048, 1)])
def test_device_lm_head(backend, v, h, offset):
    """offset shifts the weight pointer by bytes (and hidden by floats) off
    16-byte alignment: the element-wise load path."""
    case(f"lm head device vocab {v} hidden {h} offset {offset}")
    import torch

    hid, w, sc = workload(7 * v + h, v, h)
    wb = torch.zeros(w.size + offset, dtype=torch.int8, device="cuda")
    wb[offset:] = torch.from_numpy(w.reshape(-1)).cuda()
    hb = torch.zeros(h + offset, device="cuda")
    hb[offset:] = torch.from_numpy(hid).cuda()
    out = torch.full((v,), float("nan"), device="cuda")
    backend.dev_lm_head_matmul_i8(hb[offset:], wb[offset:], torch.from_numpy(sc).cuda(), out, v, h)
    torch.cuda.synchronize()
    check(out.cpu().numpy(), hid, w, sc)


def test_lm_head_shape_errors_match_oracle(backend):
    case("lm head errors")
    import bitnetrs_amd

    w = np.zeros(12, np.int8)
    args = [(np.zeros(5, f32), w, np.ones(3, f32), np.zeros(3, f32), 3, 4),
            (np.zeros(4, f32), w, np.ones(2, f32), np.zeros(3, f32), 3, 4),
            (np.zeros(4, f32), w, np.ones(3, f32), np.zeros(4, f32), 3, 4),
            (np.zeros(4, f32), w, np.ones(3, f32), np.zeros(3, f32), 2, 4)]
    for a in args:
        with pytest.raises(oracle.InvalidShape) as oe:
            oracle.lm_head_matmul_i8(*a)
        with pytest.raises(bitnetrs_amd.InvalidShape) as ge:
            backend.lm_head_matmul_i8_into(*a)
        assert str(ge.value) == str(oe.value)


@pytest.mark.parametrize("v,h,kind", [(1, 16, "normal"), (17, 48, "normal"), (63, 512, "normal"),
                                      (4100, 528, "wide"), (70000, 1040, "outlier"), (33, 6144, "wide"),
                                      (20, 6160, "normal"), (65, 2560, "tiny"), (65, 2560, "zero")])
def test_device_lm_head_digits(backend, v, h, kind):
    """The i8 matrix-core form at its edges -- one row, part of a block, several
    blocks per wave, K within and past a set of loads, its largest K and the
    form beyond it -- and over magnitudes: values 2^-40 to 1 (past what fixed
    point holds: fp32 sums), one value 2^30 times the others (and zero weights
    there, so that the rest must survive), subnormals, zeros.  fp32 sums may be
    off by up to K ulp of the products' magnitude; eight exact sums rounded once
    are off by a few."""
    case(f"lm head digits vocab {v} hidden {h} {kind}")
    import torch

    hid, w, sc = workload(v + h, v, h)
    rng = np.random.default_rng(h)
    if kind == "wide":
        hid = (hid * np.exp2(rng.integers(-40, 1, size=h))).astype(f32)
    elif kind == "outlier":
        hid[5] = 2.0 ** 30
        w[:, 5] = 0
    elif kind == "tiny":
        hid = (hid * 1e-40).astype(f32)
    elif kind == "zero":
        hid[:] = 0
    out = torch.full((v,), float("nan"), device="cuda")
    backend.dev_lm_head_matmul_i8(torch.from_numpy(hid).cuda(), torch.from_numpy(w.reshape(-1)).cuda(),
                                  torch.from_numpy(sc).cuda(), out, v, h)
    torch.cuda.synchronize()
    exact = (w.astype(np.float64) @ hid.astype(np.float64)) * sc
    mag = (np.abs(w).astype(np.float64) @ np.abs(hid).astype(np.float64)) * sc
    # 8 roundings of digit sums (the largest at most twice the products'
    # magnitude), 3 additions, the scale; beyond 6144 values the fp32 sums
    ulps = 16 if h <= 6144 else 4 * h
    cut = h * 128 * np.abs(hid).max() * 2.0 ** -61 * sc  # below the last digit
    assert np.all(np.abs(out.cpu().numpy() - exact) <= ulps * 2.0 ** -24 * mag + cut + 1e-44)


@pytest.mark.parametrize("h", [48, 2560, 6144])
@pytest.mark.parametrize("kind", ["above", "below", "both"])
@pytest.mark.parametrize("e", [31, 38, 39, 45, 60, 100])
def test_device_lm_head_range(backend, h, kind, e):
    """One hidden value 2^e above the rest, or a few 2^e below, and rows whose
    weights see only one side: each row is right to the rounding of its own
    products, on both sides of what the fixed point holds (2^38)."""
    case(f"lm head range hidden {h} {kind} 2^{e}")
    import torch

    v = 300
    hid, w, sc = workload(v + h + e, v, h)
    hid = np.where(np.abs(hid) < 0.25, f32(0.5), hid).astype(f32)
    if kind != "below":
        hid[5] = 2.0 ** e
        w[::2, 5] = 0
    if kind != "above":
        hid[20:24] *= f32(2.0 ** -e)
        w[::3] = 0
        w[::3, 20:24] = 77
    out = torch.full((v,), float("nan"), device="cuda")
    backend.dev_lm_head_matmul_i8(torch.from_numpy(hid).cuda(), torch.from_numpy(w.reshape(-1)).cuda(),
                                  torch.from_numpy(sc).cuda(), out, v, h)
    torch.cuda.synchronize()
    exact = (w.astype(np.float64) @ hid.astype(np.float64)) * sc
    mag = (np.abs(w.astype(np.float64)) @ np.abs(hid).astype(np.float64)) * sc
    # fp32 sums of 32 chains: h / 32 roundings and a few at the end
    assert np.all(np.abs(out.cpu().numpy() - exact) <= (h / 32 + 16) * 2.0 ** -24 * mag)


def test_device_lm_head_non_finite(backend):
    """An infinity or a NaN in the hidden vector: what fp32 sums give."""
    case("lm head non-finite hidden")
    import torch

    v, h = 100, 256
    hid, w, sc = workload(3, v, h)
    w[:, 9] = np.arange(v) % 3 - 1  # -, 0, + at the infinity
    for bad in (np.inf, -np.inf, np.nan):
        hid[9] = bad
        out = torch.zeros(v, device="cuda")
        backend.dev_lm_head_matmul_i8(torch.from_numpy(hid).cuda(), torch.from_numpy(w.reshape(-1)).cuda(),
                                      torch.from_numpy(sc).cuda(), out, v, h)
        torch.cuda.synchronize()
        with np.errstate(invalid="ignore"):
            want = w[:, 9].astype(np.float64) * bad
        np.testing.assert_array_equal(out.cpu().numpy(), want.astype(f32))
