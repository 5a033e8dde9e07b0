"""GPU parity of nodes with one scale per channel whose widths fit no tile (matrix-core kernels over weights in operand
order, activations as given) against the CPU oracle: tails of K and N, the rows kernel and the tile kernel with the
edges of their row tiles, K split over workgroups (the tile kernel only), every zero-point form, both output types.
Weights are exact integers in the kernels and the products are summed in f32, so f32 outputs agree with a float64 sum
to K 2^-24 of the sum of magnitudes, here bounded as 1e-5 relative in the 2-norm; f16 outputs add their own rounding
(the bounds of tests/parity.py)."""
import numpy as np
import pytest

from openvino_amd import datagen, fc
from parity import check_parity, oracle_y

pytestmark = pytest.mark.gpu

MS = [1, 15, 16, 17, 32, 33, 63, 64, 65, 130]


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


@pytest.mark.parametrize("wt,zt,N,K,bias,out,scalar", [
    ("i8", "none", 1000, 2048, True, "f32", False),   # a classifier head: N % 16 == 8
    ("u8", "u8", 40, 200, False, "f16", False),       # K % 128 != 0
    ("i8", "u8", 67, 1161, True, "f16", False),       # both odd: single halves at the end of a row, 2-byte rows
    ("u8", "none", 5, 8, False, "f32", False),        # one chunk of eight inputs
    ("i8", "none", 63, 9, True, "f32", False),
    ("u8", "u8", 130, 4300, True, "f16", True),       # long K: three k-blocks to a wave
    ("i4", "none", 65, 1160, True, "f32", False),     # nibbles
    ("u4", "u4", 33, 650, False, "f16", False),
    ("i4", "u8", 17, 4102, False, "f32", False),
    ("u4", "u4", 300, 130, True, "f16", True),
])
def test_widths_that_fit_no_tile(oracle, dev, req, wt, zt, N, K, bias, out, scalar):
    c = datagen.make_case(2100 + N, max(MS), K, N, wt, K, zt, with_bias=bias)
    if scalar:
        c.zp = c.zp[:1].copy()
        c.zp_scalar = True
    ref = oracle_y(oracle, c)
    w = fc.CompressedWeights.from_case(dev, c, output_type=out)
    try:
        assert not w.tiled
        for M in MS:
            print(f"ragged {wt}/{zt} N={N} K={K} M={M}", flush=True)
            y = req.infer(w, c.x[:M])
            info = req.last_kernel()
            kernel = "rows" if info["tile_n"] == 16 else "tile"
            assert info["name"] == f"fcc_ragged_{kernel}_w{wt[1]}", info
            check_parity(oracle, y, ref[:M], K, f"{wt}/{zt} N={N} K={K} M={M}", output_rounding_slack=True)
            if out == "f32":
                assert oracle.rel_l2(y, ref[:M]) < 1e-5
            assert np.array_equal(y, req.infer(w, c.x[:M]))
    finally:
        w.close()


@pytest.mark.parametrize("wt,zt,N,K,bias,out,scalar,runs", [
    # runs: {M: parts of K}.  One channel of the last tile of 64, one row of the last row tile, tails of K.
    ("i8", "none", 1160, 1160, True, "f16", False, {577: 2, 640: 2, 641: 2}),    # parts of five k-blocks
    ("u8", "u8", 1161, 1161, True, "f32", False, {577: 2, 1300: 1}),             # ten k-blocks, the last of nine inputs
    ("u4", "u4", 1160, 4300, False, "f32", False, {577: 4}),                     # parts of 9, 9, 9 and 7 k-blocks
    ("i4", "none", 100, 4302, True, "f32", False, {1500: 7}),                    # parts of five, the last of four
    ("i8", "u8", 1161, 200, False, "f16", False, {577: 1}),
    ("i4", "none", 1160, 8, True, "f16", False, {577: 1}),                       # one chunk of one k-block
    ("u4", "u8", 2113, 300, True, "f32", False, {63: 1, 64: 1, 65: 1, 577: 1}),  # three k-blocks
    ("u8", "none", 4300, 394, False, "f16", False, {17: 1, 33: 1}),              # less than one row tile
    ("u8", "u8", 1089, 1161, False, "f16", True, {577: 2}),
    ("u4", "u4", 1090, 650, True, "f32", True, {577: 1}),
])
def test_tiles(oracle, dev, req, wt, zt, N, K, bias, out, scalar, runs):
    """The tile kernel, unsplit and with K split, over even and odd numbers of k-blocks."""
    c = datagen.make_case(2150 + N + K, max(runs), K, N, wt, K, zt, with_bias=bias)
    if scalar:
        c.zp = c.zp[:1].copy()
        c.zp_scalar = True
    w = fc.CompressedWeights.from_case(dev, c, output_type=out)
    try:
        for M, parts in runs.items():
            print(f"ragged tiles {wt}/{zt} N={N} K={K} M={M}", flush=True)
            y, info = req.infer(w, c.x[:M]), req.last_kernel()
            assert info["name"] == f"fcc_ragged_tile_w{wt[1]}" and (info["tile_m"], info["tile_n"]) == (64, 64), info
            assert info["split_k"] == parts, info
            rows = np.unique(np.clip(np.r_[0:M:37, 60:68, M - 66:M], 0, M - 1))
            ref = oracle_y(oracle, c, x=c.x[rows])
            check_parity(oracle, y[rows], ref, K, f"{wt}/{zt} N={N} K={K} M={M}", output_rounding_slack=True)
            if out == "f32":
                assert oracle.rel_l2(y[rows], ref) < 1e-5
            assert np.array_equal(y, req.infer(w, c.x[:M]))
    finally:
        w.close()


def test_rows_keep_to_themselves(dev, req):
    """A row's result does not see its neighbours: what a lane loads beyond the end of a row is the next row, here
    infinities and NaNs."""
    for N, M, kernel in ((50, 3, "rows"), (50, 40, "rows"), (1161, 577, "tile")):
        c = datagen.make_case(2200, M, 203, N, "i8", 203, "none")
        w = fc.CompressedWeights.from_case(dev, c, output_type="f32")
        try:
            clean = req.infer(w, c.x)
            assert req.last_kernel()["name"] == f"fcc_ragged_{kernel}_w8"
            x = c.x.copy()
            x[1::2] = np.inf
            x[1, 0] = np.nan
            dirty = req.infer(w, x)
            assert np.array_equal(clean[0::2], dirty[0::2]) and not np.isfinite(dirty[1::2]).any()
        finally:
            w.close()


@pytest.mark.parametrize("wt,zt,N,K,M,bias", [
    ("i8", "none", 3480, 1160, 577, True),   # rows of 16-byte pieces
    ("u8", "u8", 3474, 394, 577, False),     # the row ends inside a piece, one dword of it left
    ("i4", "none", 4225, 262, 514, True),    # ... three dwords left, two rows in the last row tile
    ("u4", "u4", 4300, 388, 521, False),     # ... two
    ("i8", "u8", 1161, 4300, 577, True),     # parts of nine k-blocks, the last of seven
    ("u8", "none", 8300, 14, 257, False),    # one k-block, two pieces
])
def test_tiles_loaded_straight_to_lds_and_through_registers(oracle, dev, req, monkeypatch, capfd, wt, zt, N, K, M, bias):
    """Activations at a multiple of four bytes take the kernel that loads them straight to LDS, those at an odd multiple
    of two the one that loads through registers: the same bits, and a row's result does not see its neighbours.  (The
    first kernel takes launches of more than two workgroups to a compute unit, 512 here.)"""
    import torch
    c = datagen.make_case(2300 + K, M, K, N, wt, K, zt, with_bias=bias)
    w = fc.CompressedWeights.from_case(dev, c, output_type="f32")
    monkeypatch.setenv("OVFCC_VERBOSE", "1")

    def run(x, shift):
        buf = torch.zeros(M * K + 8, dtype=torch.float16, device="cuda")
        buf[shift:shift + M * K] = torch.from_numpy(x).cuda().reshape(-1)
        y = torch.full((M, N), float("nan"), dtype=torch.float32, device="cuda")
        torch.cuda.synchronize()
        capfd.readouterr()
        req.infer_device(w, buf.data_ptr() + 2 * shift, y.data_ptr(), M)
        req.sync()
        launch, = [line for line in capfd.readouterr().err.splitlines() if line.startswith("ovfcc: launch")]
        assert launch.endswith(" to_lds") == (shift % 2 == 0), launch
        assert req.last_kernel()["name"] == f"fcc_ragged_tile_w{wt[1]}"
        return y.cpu().numpy()

    try:
        y = run(c.x, 0)
        check_parity(oracle, y, oracle_y(oracle, c), K, f"{wt}/{zt} N={N} K={K} M={M}", output_rounding_slack=True)
        assert np.array_equal(y, run(c.x, 2))  # four bytes further
        assert np.array_equal(y, run(c.x, 1))  # two
        x = c.x.copy()
        x[1::2] = np.inf
        x[1, 0] = np.nan
        dirty = run(x, 0)
        assert np.array_equal(y[0::2], dirty[0::2]) and not np.isfinite(dirty[1::2]).any()
    finally:
        w.close()


def blob_fields(blob, at=0):
    """(version, flags, bytes of the weights) of the header that begins at byte `at`, as views into the blob."""
    head = int(blob[at + 12:at + 16].view(np.uint32)[0])
    return (blob[at + 8:at + 12].view(np.uint32), blob[at + head - 36:at + head - 32].view(np.int32),
            blob[at + head - 32:at + head - 24].view(np.uint64))


def pad16(n):
    return (n + 15) // 16 * 16


def version_2(blob, given):
    """The blob of a node that fits no tile as version 2 wrote it: the weights as given, no flag."""
    head = int(blob[12:16].view(np.uint32)[0])
    old = blob[:pad16(head)].copy()
    rest = blob[pad16(head) + pad16(int(blob_fields(blob)[2][0])):]
    version, flags, w_bytes = blob_fields(old)
    version[0], flags[0], w_bytes[0] = 2, 0, given.size
    return np.concatenate([old, given, np.zeros(pad16(given.size) - given.size, np.uint8), rest])


@pytest.mark.parametrize("wt,zt,N,K", [("i8", "u8", 128, 256),    # as many bytes in operand order as in OpenVINO's
                                       ("u8", "u8", 67, 1161), ("i4", "none", 65, 1160), ("u4", "u4", 33, 651)])
def test_blob_with_the_weights_as_given(dev, req, wt, zt, N, K):
    """A blob of version 2, written before these nodes had an order of their own, holds the weights as OpenVINO packs
    them: it gives the same node, as does a blob of version 3 in operand order.  Each version's flag is held to."""
    c = datagen.make_case(2250 + N, 20, K, N, wt, K, zt, with_bias=True)
    w = fc.CompressedWeights.from_case(dev, c, output_type="f32")
    blob = np.asarray(w.export_blob()).copy()
    version, flags, _ = blob_fields(blob)
    assert version[0] == 3 and flags[0] == 4
    old = version_2(blob, np.ascontiguousarray(c.w).view(np.uint8).reshape(-1))
    nodes = [w]
    try:
        y = req.infer(w, c.x)
        for b in (blob, old):
            nodes.append(fc.CompressedWeights.import_blob(dev, b))
            assert np.array_equal(req.infer(nodes[-1], c.x), y)
        assert np.array_equal(np.asarray(nodes[-1].export_blob()), blob)
        blob_fields(old)[1][0] = 4          # version 2 with the flag of version 3
        with pytest.raises(fc.OvfccError):
            fc.CompressedWeights.import_blob(dev, old)
        # version 3 without it (operand order, as one would write before there was a flag), tiled, or as version 1 or 4
        for v, f in ((3, 0), (3, 1), (3, 5), (1, 4), (4, 4)):
            version[0], flags[0] = v, f
            with pytest.raises(fc.OvfccError):
                fc.CompressedWeights.import_blob(dev, blob)
    finally:
        for n in nodes:
            n.close()


def test_version_2_blobs_of_other_nodes(dev, req):
    """Tiled nodes, MLP nodes and nodes with several groups per channel have the same blob in both versions."""
    plain = datagen.make_case(2260, 6, 200, 40, "u4", 50, "u4")
    tiled = datagen.make_case(2261, 6, 512, 256, "i4", 128, "none", with_bias=True)
    gate_up = fc.CompressedWeights.from_case(dev, datagen.make_case(2262, 6, 512, 512, "u4", 128, "u4"), glu="swish")
    down = fc.CompressedWeights.from_case(dev, datagen.make_case(2263, 6, 256, 128, "u4", 128, "u4"))
    nodes = [gate_up, down, fc.CompressedWeights.from_case(dev, plain), fc.CompressedWeights.from_case(dev, tiled)]
    try:
        nodes.append(fc.CompressedWeights.mlp(gate_up, down))
        for w in list(nodes[2:]):
            x = np.random.default_rng(2264).standard_normal((6, w.K)).astype(np.float16)
            blob = np.asarray(w.export_blob()).copy()
            magic, at = blob[:8].tobytes(), 0
            while at >= 0:                  # an MLP node: its down projection's blob as well
                blob_fields(blob, at)[0][0] = 2
                at = blob.tobytes().find(magic, at + 8)
            nodes.append(fc.CompressedWeights.import_blob(dev, blob))
            assert np.array_equal(req.infer(nodes[-1], x), req.infer(w, x))
    finally:
        for n in nodes:
            n.close()
