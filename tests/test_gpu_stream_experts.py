"""GPU parity of the weight-streaming kernel over the slices of a routed launch (4-bit experts of 1 MiB and more, few rows
each): slices of 16 and 32 rows and several slices of one expert, idle experts, K split over workgroups with an odd
number of k-blocks, every group size, rows gathered through the map and rows in place, pairs that name no expert.
Bounds of tests/test_gpu_moe.py and tests/parity.py."""
import numpy as np
import pytest

from openvino_amd import datagen, fc
from parity import check_parity
from test_gpu_grouped_matmul import args_of, make_groups
from test_gpu_moe import check
from test_gpu_parity import gather_matmul_reference
from test_oracle_moe import expert_args, make_layer, routed

pytestmark = pytest.mark.gpu


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


@pytest.mark.parametrize("wt,zt,G,out", [("u4", "u4", 128, "f16"), ("i4", "none", 64, "f32"), ("u4", "u4", 32, "f16")])
def test_moe_block(oracle, dev, req, wt, zt, G, out):
    E, top_k, H, I = 8, 2, 1280, 1664          # ten and thirteen k-blocks
    gu, dn = make_layer(940, E, H, I, wt=wt, zt=zt, G=G)
    wg = [fc.CompressedWeights.from_case(dev, c, glu="swish") for c in gu]
    wd = [fc.CompressedWeights.from_case(dev, c, output_type=out) for c in dn]
    try:
        for M, skewed, height in ((1, False, 16), (5, False, 16), (33, False, 16), (33, True, 16), (70, False, 32),
                                  (80, True, 32)):
            print(f"stream experts {wt}/{zt} G={G} out={out} M={M} skewed={skewed}", flush=True)
            idx, routing = routed(941 + M, M, E, top_k)
            if skewed:                            # every row to the same pair of experts: several slices each
                idx[:] = (6, 1)
            x = (0.25 * np.random.default_rng(942).standard_normal((M, H))).astype(np.float16)  # results of order one
            y = req.moe(wg, wd, x, routing, idx, device_indices=True)
            info = req.last_kernel()
            assert info["name"] == "fcc_stream_grouped_w4" and info["tile_m"] == height, info
            ref = oracle.moe_reference(x, routing, idx, [expert_args(c) for c in gu], [expert_args(c) for c in dn], 1)
            check(oracle, y, ref, max(H, I), f"M={M} skewed={skewed}")
            for _ in range(3):                    # split parts are added in order: the same bits every time
                assert np.array_equal(req.moe(wg, wd, x, routing, idx, device_indices=True).view(np.uint8), y.view(np.uint8))
    finally:
        for w in wg + wd:
            w.close()


@pytest.mark.parametrize("M,a_batches,G", [(1, 1, 128), (9, 2, 1280), (60, 2, 256), (88, 1, 128)])
def test_gather_matmul(oracle, dev, req, M, a_batches, G):
    E, top_k, K, N = 8, 2, 1280, 1792
    cases = [datagen.make_case(950 + e, 1, K, N, "u4", G, "u4", with_bias=True) for e in range(E)]
    ws = [fc.CompressedWeights.from_case(dev, c) for c in cases]
    rng = np.random.default_rng(951 + M)
    indices = np.argsort(rng.standard_normal((M, E)), axis=1)[:, :top_k].astype(np.int32)
    A = rng.standard_normal((a_batches, M, K)).astype(np.float16)
    try:
        print(f"stream gather M={M} a_batches={a_batches} G={G}", flush=True)
        y = req.gather_matmul(ws, A, indices, device_indices=True)
        assert req.last_kernel()["name"] == "fcc_stream_grouped_w4"
        ref = gather_matmul_reference(oracle, cases, A, indices)
        check_parity(oracle, y.reshape(-1, N), ref.reshape(-1, N), K, f"M={M}", output_rounding_slack=True)
        bad = indices.copy()
        bad[0, 0], bad[M - 1, 1] = E, -3
        got = req.gather_matmul(ws, A, bad, device_indices=True, y_fill=7.0)
        assert np.all(got[0, 0].view(np.uint16) == 0) and np.all(got[1, M - 1].view(np.uint16) == 0)
        got[0, 0], got[1, M - 1] = y[0, 0], y[1, M - 1]
        assert np.array_equal(got.view(np.uint16), y.view(np.uint16))
    finally:
        for w in ws:
            w.close()


@pytest.mark.parametrize("tpe,tail", [([0, 50, 0, 0, 3, 0, 17, 0], 9), ([1] * 8, 0)])
def test_offsets_in_device_memory(oracle, dev, req, tpe, tail):
    G, N, K = 8, 1792, 1280
    cases, ws = make_groups(dev, 8700, G, N, K, "u4", "scalar", 128)
    offsets = np.cumsum(tpe).astype(np.int32)
    a = np.random.default_rng(8701).standard_normal((int(offsets[-1]) + tail, K)).astype(np.float16)
    try:
        print(f"stream offsets {tpe} tail {tail}", flush=True)
        y = req.grouped_matmul(ws, a, offsets, y_fill=3.0, device_offsets=True)
        assert req.last_kernel()["name"] == "fcc_stream_grouped_w4"
        assert np.all(y[int(offsets[-1]):] == 0)
        check_parity(oracle, y, oracle.grouped_matmul_reference(a, [args_of(c) for c in cases], offsets), K, f"{tpe}",
                     output_rounding_slack=True)
    finally:
        for w in ws:
            w.close()
