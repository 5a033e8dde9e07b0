"""GPU: a call with host tensors gives what the same call on device buffers gives, at transfer sizes around the sixteen bytes
and the 4096 bytes of a workgroup of the kernel that fetches staged activations, and around the size from which tensors are
copied directly; the bytes that the previous, larger call left behind it do not show."""
import numpy as np
import pytest

from openvino_amd import datagen, fc

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("K,rows", [
    (8, [1, 255, 256, 257, 3]),      # 16 bytes; 4096 and a piece less and more
    (9, [1, 8, 227, 228, 455, 2]),   # 18 bytes; odd tails on both sides of 4096
    (1161, [3, 1, 7]),
    (2048, [126, 127, 128, 1]),      # x and y around 1 MiB together
])
def test_host_and_device_calls_agree(K, rows):
    import torch
    N = 1024
    c = datagen.make_case(2400 + K, max(rows), K, N, "i8", K, "none", with_bias=True)
    dev = fc.Device(0)
    req = fc.InferRequest(dev)
    w = fc.CompressedWeights.from_case(dev, c, output_type="f32")
    try:
        for M in rows:
            x = np.ascontiguousarray(c.x[:M])
            xd = torch.from_numpy(x).cuda()
            yd = torch.empty((M, N), dtype=torch.float32, device="cuda")
            torch.cuda.synchronize()
            y = req.infer(w, x)
            req.infer_device(w, xd.data_ptr(), yd.data_ptr(), M)
            req.sync()
            assert np.array_equal(y, yd.cpu().numpy()), (K, M)
            ref = x.astype(np.float64) @ (c.w.reshape(N, K).astype(np.int8).astype(np.float64) * c.scale.reshape(N, 1).astype(np.float64)).T
            ref += c.bias.reshape(1, N).astype(np.float64)
            assert np.linalg.norm(y - ref) < 1e-5 * np.linalg.norm(ref), (K, M)  # K 2^-24 of the magnitudes summed, K <= 2048
    finally:
        w.close()
        req.close()
        dev.close()
