"""Routing and weighted sum of the expert block where their kernels can go wrong: expert counts that are no power of two
(a reduction across lanes), as many as one launch takes, one expert; one to five selections (sums of one, two and four
at a time, and the rest); rows that end inside a workgroup's 1024 channels, in one or two of them."""
import numpy as np
import pytest

from openvino_amd import fc
from test_gpu_moe import check, dev, req  # noqa: F401
from test_oracle_moe import expert_args, make_layer, routed

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("E,top_k,H,I,M", [(1, 1, 256, 256, 3), (3, 2, 1280, 256, 5), (5, 3, 1024, 256, 130), (6, 4, 256, 256, 64),
                                           (7, 5, 2304, 256, 60), (33, 2, 256, 256, 20), (64, 1, 256, 256, 300)])
@pytest.mark.parametrize("out", ["f16", "f32"])
def test_moe_routed_counts(oracle, dev, req, E, top_k, H, I, M, out):  # noqa: F811
    print(f"moe routed E={E} top_k={top_k} H={H} M={M} out={out}", flush=True)
    gu, dn = make_layer(970 + E, E, H, I)
    wg = [fc.CompressedWeights.from_case(dev, c, glu="swish") for c in gu]
    wd = [fc.CompressedWeights.from_case(dev, c, output_type=out) for c in dn]
    idx, routing = routed(971 + E, M, E, top_k)
    x = np.random.default_rng(972).standard_normal((M, H)).astype(np.float16)
    try:
        y = req.moe(wg, wd, x, routing, idx, device_indices=True)
        ref = oracle.moe_reference(x, routing, idx, [expert_args(c) for c in gu], [expert_args(c) for c in dn], 1)
        check(oracle, y, ref, max(H, I), f"E={E} top_k={top_k}")
        # an index that names no expert adds nothing, whatever its weight
        bad = idx.copy()
        bad[M // 2, top_k - 1], bad[0, 0] = E, -1
        zeroed = routing.copy()
        zeroed[M // 2, top_k - 1], zeroed[0, 0] = 0, 0
        got = req.moe(wg, wd, x, routing, bad, device_indices=True)
        ref = oracle.moe_reference(x, zeroed, idx, [expert_args(c) for c in gu], [expert_args(c) for c in dn], 1)
        check(oracle, got, ref, max(H, I), f"E={E} top_k={top_k}, bad indices")
    finally:
        for w in wg + wd:
            w.close()
