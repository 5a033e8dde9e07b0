"""The register-fed prefill kernels over nodes that end on half a 256-channel tile (N an odd multiple of 128): every
kernel, tile height and cut along K, against the oracle; no byte past the output is written."""
import numpy as np
import pytest
import torch

from openvino_amd import datagen, fc
from parity import check_parity, glu_reference, oracle_y

pytestmark = pytest.mark.gpu

KERNEL = {"async": ("fcc_prefill_async_w4", {"OVFCC_PREFILL_ROWS": "128"}),
          "async64": ("fcc_prefill_async_w4", {"OVFCC_PREFILL_ROWS": "64"}),
          "big": ("fcc_prefill_big_w4", {"OVFCC_PREFILL_ROWS": "128", "OVFCC_PREFILL_BIG": "1"}),
          "direct": ("fcc_prefill_direct_w8", {})}


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


def run_guarded(req, w, x, n_out, out):
    """The call on device buffers, with a page of sentinels behind y."""
    xd = torch.from_numpy(np.ascontiguousarray(x)).cuda()
    dtype = torch.float32 if out == "f32" else torch.float16
    y = torch.full((x.shape[0] * n_out + 4096,), -77.0, dtype=dtype, device="cuda")
    torch.cuda.synchronize()
    req.infer_device(w, xd.data_ptr(), y.data_ptr(), x.shape[0])
    req.sync()
    y = y.cpu().numpy()
    assert np.all(y[x.shape[0] * n_out:] == -77.0)
    return y[:x.shape[0] * n_out].reshape(x.shape[0], n_out)


@pytest.mark.parametrize("N", [384, 896])
@pytest.mark.parametrize("kernel,wt,zt,K,G,out,glu", [
    ("async", "u4", "u4", 384, 128, "f16", None), ("async", "i4", "none", 512, 64, "f32", None),
    ("async", "u4", "u4", 512, 128, "f16", "swish"), ("async64", "u4", "u8", 640, 32, "f16", None),
    ("async64", "u4", "none", 512, 512, "f32", None), ("async64", "i4", "none", 2048, 128, "f16", "gelu"),
    ("big", "u4", "u4", 384, 128, "f16", None), ("big", "i4", "none", 256, 256, "f32", None),
    ("big", "u4", "u4", 512, 128, "f16", "swish"), ("direct", "u8", "u8", 384, 384, "f16", None),
    ("direct", "i8", "none", 512, 128, "f32", None),
    ("direct", "u8", "u8", 2048, 2048, "f32", "swish"),  # (products of 8-bit gate and up reach 1e5: beyond f16)
])
def test_half_tile(oracle, dev, req, monkeypatch, kernel, wt, zt, N, K, G, out, glu):
    name, env = KERNEL[kernel]
    monkeypatch.setenv("OVFCC_PREFILL_WIDE", "1")
    for k, v in env.items():
        monkeypatch.setenv(k, v)
    c = datagen.make_case(77, 300, K, N, wt, G, zt, with_bias=True)
    w = fc.CompressedWeights.from_case(dev, c, output_type=out, **({"glu": glu} if glu else {}))
    try:
        for M in (129, 256, 300):
            print(f"half tile {kernel} N={N} M={M}", flush=True)
            y = run_guarded(req, w, c.x[:M], N // 2 if glu else N, out)
            info = req.last_kernel()
            assert info["name"] == name, info
            ref, scale = glu_reference(oracle, c, glu, x=c.x[:M]) if glu else (oracle_y(oracle, c, x=c.x[:M]), 1.0)
            check_parity(oracle, y, ref, K, f"{info}", output_rounding_slack=True, limit_scale=scale)
    finally:
        w.close()


@pytest.mark.parametrize("wt,zt,N,K,G,M,name", [
    ("u4", "u4", 5760, 1024, 128, 700, "fcc_prefill_async_w4"), ("i4", "none", 1152, 4096, 64, 300, "fcc_prefill_async_w4"),
    ("u8", "u8", 4480, 1024, 1024, 600, "fcc_prefill_direct_w8"), ("i4", "none", 128, 1024, 128, 8192, "fcc_prefill_w4"),
])
def test_half_tile_rule(oracle, dev, req, wt, zt, N, K, G, M, name):
    """What the planner gives such nodes by itself; a node of half a tile keeps the square kernel."""
    c = datagen.make_case(78, M, K, N, wt, G, zt)
    w = fc.CompressedWeights.from_case(dev, c)
    try:
        y = run_guarded(req, w, c.x, N, "f16")
        assert req.last_kernel()["name"] == name, req.last_kernel()
        some = np.r_[0:64, M - 70:M]
        check_parity(oracle, y[some], oracle_y(oracle, c, x=c.x[some]), K, name, output_rounding_slack=True)
    finally:
        w.close()


@pytest.mark.parametrize("wt,zt,N,K,G", [("u4", "u4", 4224, 4096, 128), ("i4", "none", 6528, 2048, 64),
                                         ("u8", "u8", 4480, 8192, 8192)])
def test_half_tile_nodes_of_up_to_128_rows_keep_their_decode_launches(dev, req, wt, zt, N, K, G):
    """... whose weights are not rounded after scaling: f32 results as close to 64 bits as f32 sums over K allow."""
    c = datagen.make_case(79, 128, K, N, wt, G, zt)
    w = fc.CompressedWeights.from_case(dev, c, output_type="f32")
    q = c.w.astype(np.int64) if wt == "u8" else datagen.unpack_nibbles(c.w.reshape(-1), N * K).astype(np.int64)
    q = np.where(q > 7, q - 16, q) if wt == "i4" else q
    z = 0 if c.zp is None else c.zp.reshape(N, -1, 1) if wt == "u8" else datagen.unpack_nibbles(c.zp.reshape(-1), N * K // G).reshape(N, -1, 1)
    full = (q.reshape(N, K // G, G) - np.asarray(z, np.int64)) * c.scale.astype(np.float64).reshape(N, -1, 1)
    ref = c.x.astype(np.float64) @ full.reshape(N, K).T
    try:
        for M in (49, 96, 97, 128):
            print(f"half tile, decode launches {wt} N={N} K={K} M={M}", flush=True)
            y = run_guarded(req, w, c.x[:M], N, "f32")
            assert not req.last_kernel()["name"].startswith("fcc_prefill"), req.last_kernel()
            # a rounding of f16 weights would show as 2^-12; a sum of K terms in f32 is within sqrt(K) 2^-24 = 5.4e-6 of exact
            assert np.linalg.norm(y - ref[:M]) < 2e-5 * np.linalg.norm(ref[:M])
    finally:
        w.close()
