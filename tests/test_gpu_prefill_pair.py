"""The prefill kernels that run two workgroups on a compute unit (kernel_prefill_pair.hip): every tile height at its edges,
every number of k-blocks that the loop and what follows it treat differently, every form of scales and zero-points."""
import numpy as np
import pytest

from openvino_amd import datagen, fc
from parity import check_parity, oracle_y

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
