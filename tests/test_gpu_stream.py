"""GPU parity of the weight-streaming kernel (up to 48 rows of large tiled nodes) against the CPU oracle, where it can
go wrong: a last workgroup with channels for some of its waves only, an odd number of k-blocks (half a stage), K split over
workgroups with a short last part, row tiles and their edges, every group size and zero-point form, the gated linear
unit, both output types.  Bounds of tests/parity.py; f32 outputs add no rounding of their own and the weights are exact
in the kernel, so they stay within 1e-5 of the oracle's f32 sums."""
import numpy as np
import pytest

from openvino_amd import datagen, fc
from parity import check_parity, glu_reference, oracle_y

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


CASES = [
    # w_type, zp_type, N, K, G, bias, out, rows
    ("u8", "u8", 272, 1152, 1152, True, "f32", [17, 32, 33, 48]),        # 17 tiles, nine k-blocks
    ("i8", "none", 128, 2176, 2176, False, "f16", [17, 48]),
    ("u8", "u8", 144, 2304, 256, True, "f16", [17, 33]),                 # groups of two k-blocks
    ("i4", "none", 1040, 640, 64, False, "f32", [17, 31, 48]),
    ("u4", "u4", 528, 1152, 64, True, "f16", [17, 33]),
    ("u4", "u4", 1040, 640, 32, True, "f32", [17, 48]),
    ("i4", "none", 528, 1408, 32, False, "f16", [20, 40]),
    ("u4", "u4", 272, 2432, 2432, True, "f32", [17, 48]),                # 4-bit, one scale per channel
    ("i4", "none", 272, 2560, 256, False, "f16", [17, 48]),
    ("u4", "u8", 1296, 4224, 128, True, "f16", [17, 48]),                # 33 k-blocks: no whole number per wave elsewhere
    ("u8", "u8", 4112, 4224, 4224, True, "f32", [5, 16]),                # one row tile: nodes of 16 MB
    ("u4", "u4", 4112, 5504, 64, False, "f16", [5, 16]),
]


def parity(oracle, dev, req, wt, zt, N, K, G, bias, out, rows):
    c = datagen.make_case(2300 + N, max(rows), K, N, wt, G, zt, with_bias=bias)
    ref = oracle_y(oracle, c)
    w = fc.CompressedWeights.from_case(dev, c, output_type=out)
    try:
        for M in rows:
            print(f"stream {wt}/{zt} N={N} K={K} G={G} M={M}", flush=True)
            y = req.infer(w, c.x[:M])
            info = req.last_kernel()
            assert info["name"].startswith("fcc_stream"), info
            check_parity(oracle, y, ref[:M], K, f"{info}", output_rounding_slack=True)
            if out == "f32":
                assert oracle.rel_l2(y, ref[:M]) < 1e-5
            for _ in range(3):      # split parts are added in order: the same bits every time
                assert np.array_equal(y, req.infer(w, c.x[:M]))
    finally:
        w.close()


@pytest.mark.parametrize("wt,zt,N,K,G,bias,out,rows", CASES)
def test_parity(oracle, dev, req, wt, zt, N, K, G, bias, out, rows):
    parity(oracle, dev, req, wt, zt, N, K, G, bias, out, rows)


@pytest.mark.parametrize("wt,zt,N,K,G,bias,out", [case[:7] for case in CASES[:10]])
def test_one_to_four_rows(oracle, dev, req, monkeypatch, wt, zt, N, K, G, bias, out):
    """Most nodes of these sizes run other kernels at so few rows; the kernel itself takes them all."""
    monkeypatch.setenv("OVFCC_STREAM", "1")
    parity(oracle, dev, req, wt, zt, N, K, G, bias, out, [1, 2, 3, 4])


@pytest.mark.parametrize("wt,zt,N,K,G,glu", [
    ("u8", "u8", 2400, 28672, 28672, None),      # 8 bits, K beyond the LDS of the kernel with one tile per workgroup
    ("u4", "u4", 2080, 24576, 64, "swish")])     # a gated linear unit with long K
def test_one_to_four_rows_of_long_nodes(oracle, dev, req, wt, zt, N, K, G, glu):
    c = datagen.make_case(2500 + N, 4, K, N, wt, G, zt, with_bias=True)
    ref, amp = glu_reference(oracle, c, glu) if glu else (oracle_y(oracle, c), 1.0)
    w = fc.CompressedWeights.from_case(dev, c, glu=glu)
    try:
        for M in (1, 2, 4):
            print(f"stream {wt}/{zt} N={N} K={K} G={G} glu={glu} M={M}", flush=True)
            y, info = req.infer(w, c.x[:M]), req.last_kernel()
            assert info["name"].startswith("fcc_stream"), info
            check_parity(oracle, y, ref[:M], K, f"{info}", output_rounding_slack=True, limit_scale=amp)
    finally:
        w.close()


@pytest.mark.parametrize("wt,zt,N,K,G,kind,second", [
    ("u8", "u8", 544, 1152, 1152, "swish", False), ("u4", "u4", 1056, 640, 64, "gelu", True),
    ("i4", "none", 2080, 384, 32, "gelu_tanh", False)])
def test_gated_linear_unit(oracle, dev, req, wt, zt, N, K, G, kind, second):
    c = datagen.make_case(2400 + N, 48, K, N, wt, G, zt, with_bias=True)
    w = fc.CompressedWeights.from_case(dev, c, glu=kind, glu_gate_second=second)
    ref, amp = glu_reference(oracle, c, kind, second)
    try:
        for M in (17, 48):
            print(f"stream glu {wt}/{zt} N={N} K={K} G={G} M={M}", flush=True)
            y = req.infer(w, c.x[:M])
            assert req.last_kernel()["name"].startswith("fcc_stream"), req.last_kernel()
            check_parity(oracle, y, ref[:M], K, f"{req.last_kernel()}", output_rounding_slack=True, limit_scale=amp)
    finally:
        w.close()


@pytest.mark.parametrize("wt,zt,K,G", [("u8", "u8", 8192, 8192), ("i8", "none", 28672, 28672), ("u4", "u4", 14336, 14336),
                                       ("u4", "u4", 8192, 64)])
def test_sums_are_no_less_precise_than_the_small_batch_kernels(oracle, dev, req, monkeypatch, wt, zt, K, G):
    """Both kernels sum exact products in f32, in different orders; 12 288 results, whose mean error varies by 1 %."""
    c = datagen.make_case(2460, 24, K, 512, wt, G, zt)
    exact = oracle_y(oracle, c, acc_f64=True).astype(np.float64)
    w = fc.CompressedWeights.from_case(dev, c, output_type="f32")
    try:
        error = {}
        for stream in ("0", "1"):
            monkeypatch.setenv("OVFCC_STREAM", stream)
            print(f"precision {wt}/{zt} K={K} G={G} OVFCC_STREAM={stream}", flush=True)
            y = req.infer(w, c.x).astype(np.float64)
            assert req.last_kernel()["name"].startswith("fcc_stream" if stream == "1" else "fcc_batch"), req.last_kernel()
            error[stream] = np.linalg.norm(y - exact) / np.linalg.norm(exact)
        print(error)
        assert error["1"] <= 1.1 * error["0"], error
    finally:
        w.close()


@pytest.mark.parametrize("env,M,name,block", [
    ({}, 32, "fcc_stream_w4", 512),
    ({"OVFCC_STREAM": "0"}, 32, "fcc_batch_w4", 512),
    ({"OVFCC_GEMV16": "0"}, 32, "fcc_batch_w4", 512),           # any override about an older kernel keeps it
    ({"OVFCC_DECODE_WAVES": "4"}, 32, "fcc_batch_w4", 256),
    ({"OVFCC_DECODE_RT": "2"}, 32, "fcc_batch_w4", 512),
    ({"OVFCC_DECODE_XLDS": "0"}, 3, "fcc_decode_w4", None),
    ({"OVFCC_STREAM": "1"}, 3, "fcc_stream_w4", 512),
    ({"OVFCC_STREAM": "1", "OVFCC_GEMV16": "0"}, 32, "fcc_stream_w4", 512),
])
def test_overrides(oracle, dev, req, monkeypatch, env, M, name, block):
    c = datagen.make_case(2450, M, 1024, 1024, "u4", 64, "u4")
    w = fc.CompressedWeights.from_case(dev, c)
    try:
        for k, v in env.items():
            monkeypatch.setenv(k, v)
        print(f"overrides {env} M={M}", flush=True)
        y, info = req.infer(w, c.x), req.last_kernel()
        assert info["name"] == name and block in (None, info["block"]), info
        check_parity(oracle, y, oracle_y(oracle, c), 1024, f"{info}", output_rounding_slack=True)
    finally:
        w.close()
