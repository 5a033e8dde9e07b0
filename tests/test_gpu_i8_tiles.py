"""GPU parity of the integer prefill kernel with 256 x 256 tiles (8-bit weights over int8 activations) against the CPU oracle
of that arithmetic: forced onto shapes small enough to check every output -- one to nine k-blocks (its stages repeat
every four), row counts around its tile, zero-points, bias, both output types, the gated linear unit, asymmetric
activations -- and K in two parts, which the planner chooses for long rows.  Sums are exact, so f32 outputs are within a few
roundings of the epilogue (1e-6) and equal to the 128-row kernel's."""
import numpy as np
import pytest

from openvino_amd import datagen, fc

pytestmark = pytest.mark.gpu

T = {"u8": 3, "i8": 4}


def reference(oracle, c, x):
    zp = None if c.zp is None else c.zp.astype(np.float32)
    return oracle.fc_dynquant_reference(x, c.w, T[c.w_type], c.scale, zp, c.bias, N=c.N, K=c.K)


@pytest.fixture()
def req():
    d = fc.Device(0)
    r = fc.InferRequest(d)
    yield r
    r.close()
    d.close()


def both(req, monkeypatch, w, x):
    """the call with 256-row tiles and with 128-row tiles"""
    ys = []
    for big in ("1", "0"):
        monkeypatch.setenv("OVFCC_PREFILL_BIG", big)
        ys.append(req.infer(w, x))
        info = req.last_kernel()
        assert info["name"].startswith("fcc_prefill_i8_w8") and info["tile_m"] == (256 if big == "1" else 128), info
        if big == "1":
            split = info["split_k"]
    return ys[0], ys[1], split


@pytest.mark.parametrize("wt,zt,N,K,bias,out,mode", [
    ("u8", "u8", 256, 128, True, "f32", True), ("i8", "none", 512, 256, False, "f16", True),
    ("u8", "none", 256, 384, True, "f32", True), ("u8", "u8", 512, 512, False, "f32", True),
    ("i8", "none", 256, 640, True, "f32", True), ("u8", "u8", 768, 1152, True, "f16", True),
    ("u8", "u8", 256, 1024, True, "f32", "asymmetric"),
    ("u8", "u8", 256, 18432, True, "f32", True),       # K in two parts of 72 k-blocks
    ("i8", "none", 512, 18560, False, "f32", True),    # 73 and 72
])
def test_tiles(oracle, req, monkeypatch, wt, zt, N, K, bias, out, mode):
    monkeypatch.setenv("OVFCC_PREFILL_WIDE", "1")
    c = datagen.make_case(1400 + K, 513, K, N, wt, K, zt, with_bias=bias)
    w = fc.CompressedWeights.from_case(req.device, c, output_type=out, dynamic_quantization=mode)
    try:
        for M in (49, 255, 256, 257, 513):
            print(f"i8 tiles {wt}/{zt} N={N} K={K} M={M} {mode}", flush=True)
            y, y128, split = both(req, monkeypatch, w, c.x[:M])
            assert split == (2 if K >= 18432 else 1)
            assert np.array_equal(y.view(np.uint8), y128.view(np.uint8)) or out == "f16"
            if out == "f16":  # (a conversion may be folded into the multiply-add before it in one of the kernels)
                assert np.mean(y.view(np.uint16) != y128.view(np.uint16)) < 1e-3
            assert np.array_equal(y.view(np.uint8), both(req, monkeypatch, w, c.x[:M])[0].view(np.uint8))
            if mode is True and M in (49, 513):
                rows = np.r_[0:min(M, 40), M - 2:M]
                ref = reference(oracle, c, c.x[rows])
                assert oracle.rel_l2(y[rows].astype(np.float32), ref) < (1e-6 if out == "f32" else 5e-4)
    finally:
        w.close()


@pytest.mark.parametrize("K", [512, 18432])
def test_gated_linear_unit(oracle, req, monkeypatch, K):
    monkeypatch.setenv("OVFCC_PREFILL_WIDE", "1")
    c = datagen.make_case(1450, 300, K, 512, "u8", K, "u8", with_bias=True)
    w = fc.CompressedWeights.from_case(req.device, c, output_type="f32", glu="swish", dynamic_quantization=True)
    try:
        y, y128, _ = both(req, monkeypatch, w, c.x)
        assert y.shape == (300, 256) and np.array_equal(y, y128)
        rows = np.r_[0:30, 254:259, 299]
        assert oracle.rel_l2(y[rows], oracle.glu(reference(oracle, c, c.x[rows]), 1, False)) < 2e-6
    finally:
        w.close()


@pytest.mark.parametrize("N,K,M,tile_m,split", [
    (8192, 8192, 1024, 128, 1),    # 256 tiles of 128 rows: one round
    (10240, 5120, 1076, 256, 1),   # 360: two rounds against one
    (8192, 18432, 1000, 256, 2),   # one round, long rows
])
def test_rule(req, N, K, M, tile_m, split):
    """What the planner gives without overrides."""
    rng = np.random.default_rng(7)
    w = fc.CompressedWeights(req.device, rng.integers(0, 256, N * K, dtype=np.uint8), np.full((N, 1), 0.01, np.float16), None, None,
                             N=N, K=K, group_size=K, w_type="i8", zp_type="none", output_type="f32", dynamic_quantization=True)
    try:
        req.infer(w, rng.standard_normal((M, K)).astype(np.float16))
        info = req.last_kernel()
        assert (info["tile_m"], info["split_k"]) == (tile_m, split), info
    finally:
        w.close()
