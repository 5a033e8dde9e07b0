"""The prefill kernels that run two workgroups on a compute unit (kernel_prefill_pair.hip): every tile height at its edges,
every number of k-blocks that the loop and what follows it treat differently, every form of scales and zero-points."""
import numpy as np
import pytest

from openvino_amd import datagen, fc
from parity import check_parity, glu_reference, oracle_y

pytestmark = pytest.mark.gpu

HEIGHTS = [1, 16, 63, 64, 65, 80, 81, 96, 97, 113, 128]


@pytest.fixture(scope="module")
def dev():
    d = fc.Device(0)
    yield d
    d.close()


@pytest.fixture()
def req(dev):
    r = fc.InferRequest(dev)
    yield r
    r.close()


@pytest.mark.parametrize("kb", [1, 2, 3, 4, 5, 7])
@pytest.mark.parametrize("wt,zt,G,bias", [("u4", "u4", 128, False), ("i4", "none", 128, True), ("u4", "u4", 64, False),
                                          ("i4", "none", 64, False), ("u4", "u4", 32, True), ("i4", "none", 32, False),
                                          ("u4", "u4", 0, False), ("i4", "none", 0, True)])
def test_slices_of_every_height(oracle, dev, req, monkeypatch, wt, zt, G, bias, kb):
    """Grouped launches of slices whose rows end on, before and behind every tile height."""
    monkeypatch.setenv("OVFCC_PREFILL_WIDE", "1")
    monkeypatch.setenv("OVFCC_PREFILL_ROWS", "80" if kb == 4 else "128")
    N, K = 512, 128 * kb
    print(f"pair slices {wt}/{zt} G={G or K} K={K}", flush=True)
    cases = [datagen.make_case(1300 + i, max(HEIGHTS), K, N, wt, G or K, zt, with_bias=bias) for i in range(2)]
    ws = [fc.CompressedWeights.from_case(dev, c) for c in cases]
    try:
        ys = req.infer_grouped([(ws[i % 2], cases[i % 2].x[:m]) for i, m in enumerate(HEIGHTS)])
        info = req.last_kernel()
        assert info["name"] == "fcc_prefill_async_grouped_w4", info
        whole = [oracle_y(oracle, c) for c in cases]
        for i, (m, y) in enumerate(zip(HEIGHTS, ys)):
            check_parity(oracle, y, whole[i % 2][:m], K, f"M={m} {info}", output_rounding_slack=True)
            # a row's result does not depend on the slice it sits in
            tall = ys[-1] if (len(ys) - 1 - i) % 2 == 0 else ys[-2]
            assert np.array_equal(y[:len(tall)].view(np.uint16), tall[:m].view(np.uint16)), m
    finally:
        for w in ws:
            w.close()


SMALL, HEIGHTS_128, MANY = (129, 160, 161, 255, 385, 640, 700), (600, 700, 1000), (2000, 2048)


@pytest.mark.parametrize("wt,zt,G,N,kb,out,glu,rows", [
    ("u4", "u4", 128, 768, 7, "f16", None, SMALL), ("i4", "none", 128, 640, 8, "f32", None, SMALL),  # (640: half a tile of 256)
    ("u4", "u4", 384, 512, 9, "f16", None, SMALL), ("i4", "none", 64, 512, 16, "f16", "swish", SMALL),
    ("u4", "u4", 64, 896, 5, "f32", None, SMALL), ("u4", "u4", 32, 512, 12, "f16", None, SMALL),
    ("u4", "u4", 128, 4096, 8, "f16", None, HEIGHTS_128), ("i4", "none", 128, 4096, 7, "f32", None, HEIGHTS_128),
    ("u4", "u4", 64, 4096, 5, "f16", None, HEIGHTS_128), ("i4", "none", 64, 4096, 3, "f16", "swish", HEIGHTS_128),
    ("u4", "u4", 32, 4096, 4, "f16", None, HEIGHTS_128), ("i4", "none", 32, 4096, 6, "f16", "gelu_tanh", HEIGHTS_128),
    ("u4", "u4", 128, 8192, 8, "f16", None, MANY), ("i4", "none", 64, 8064, 8, "f32", None, MANY)])  # (8064: half a tile)
def test_one_node(oracle, dev, req, monkeypatch, wt, zt, G, N, kb, out, glu, rows):
    """Rows that end on, before and behind the tiles of 64 to 128 rows and 128 or 256 channels, K whole and in parts: the oracle,
    the 8-wave kernel (the same weights, rounded the same way: sums of K products in another order differ by at most K 2^-24
    of the largest sum of magnitudes, below 1e-4 of the 2-norm here also after a tie of the f16 result has moved), and
    repeated launches."""
    K = 128 * kb
    c = datagen.make_case(1400 + kb, max(rows), K, N, wt, G, zt, with_bias=True)
    w = fc.CompressedWeights.from_case(dev, c, output_type=out, **({"glu": glu} if glu else {}))
    seen = set()
    try:
        for M in rows:
            print(f"pair node {wt}/{zt} G={G} N={N} K={K} M={M}", flush=True)
            monkeypatch.setenv("OVFCC_PREFILL_PAIR", "1")
            y = req.infer(w, c.x[:M])
            info = req.last_kernel()
            assert info["name"] == "fcc_prefill_async_w4" and info["block"] == 256, info
            seen.add((info["tile_n"], info["tile_m"], info["split_k"] > 1))
            assert np.array_equal(req.infer(w, c.x[:M]).view(np.uint8), y.view(np.uint8))
            some = np.unique(np.clip(np.r_[0:M:97, 60:68, 78:82, 94:98, 126:130, M - 70:M], 0, M - 1))
            x = np.ascontiguousarray(c.x[some])
            ref, scale = glu_reference(oracle, c, glu, x=x) if glu else (oracle_y(oracle, c, x=x), 1.0)
            check_parity(oracle, y[some], ref, K, f"{info}", output_rounding_slack=True, limit_scale=scale)
            monkeypatch.setenv("OVFCC_PREFILL_PAIR", "0")
            other = req.infer(w, c.x[:M])
            assert req.last_kernel()["block"] == 512 or req.last_kernel()["tile_m"] == 256
            assert oracle.rel_l2(y, other.astype(np.float32)) < 1e-4
        if rows != SMALL:
            assert {(n, m) for n, m, _ in seen} == ({(256, 128)} if rows == MANY else {(128, 80), (128, 96), (128, 128)}), seen
    finally:
        w.close()
