"""A request's first launch that splits K allocates its scratch buffers: that must work, and leave the capture whole, while
another library's stream (here torch's) is under graph capture."""
import numpy as np
import pytest

from openvino_amd import datagen, fc
from parity import check_parity, oracle_y

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("wt,N,K,G,M,name", [
    ("i8", 1160, 1160, 1160, 577, "fcc_ragged_tile_w8"),
    ("u4", 1024, 1152, 64, 32, "fcc_stream_w4")])
@pytest.mark.parametrize("mode", ["global", "thread_local"])
def test_first_call_while_a_stream_is_captured(oracle, wt, N, K, G, M, name, mode):
    torch = pytest.importorskip("torch")
    c = datagen.make_case(2600, M, K, N, wt, G, "none")
    dev = fc.Device(0)
    req = fc.InferRequest(dev)
    w = fc.CompressedWeights.from_case(dev, c, output_type="f32")
    x_ptr, y_ptr = dev.malloc(c.x.nbytes), dev.malloc(4 * M * N)
    try:
        dev.upload(x_ptr, c.x)
        a = torch.ones(1000, device="cuda")
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph, capture_error_mode=mode):
            b = a + 1
            print(f"first call under {mode} capture: {wt} N={N} K={K} M={M}", flush=True)
            req.infer_device(w, x_ptr, y_ptr, M)
        info = req.last_kernel()
        assert info["name"] == name and info["split_k"] > 1, info
        for k in range(3):
            a.fill_(k)
            graph.replay()
            torch.cuda.synchronize()
            assert bool((b == k + 1).all())
        req.sync()
        rows = np.unique(np.r_[0:M:19, M - 1])
        y = dev.download(y_ptr, (M, N), np.float32)
        check_parity(oracle, y[rows], oracle_y(oracle, c, x=c.x[rows]), K, f"{info}", output_rounding_slack=True)
    finally:
        dev.free(x_ptr)
        dev.free(y_ptr)
        w.close()
        req.close()
        dev.close()
