"""The dequantise-then-fp32 GEMM (W4A16 / W8A16) on the GPU against the CPU oracle.  GPU only.

Reference: gemm_w4a16_naive / gemm_w4a16_tiled / gemm_w8a16_naive (include/gemm_cuda_naive.cuh:
66-150, include/gemm_cuda_tiled.cuh:108-190), their CPU references (include/gemm_reference.h:
73-147) and the harness oracle of the fp32-activation definitions (llm_kernel_test/reference/
gemm_ref.py:51-97).  Bars: integer-valued inputs (d = 1, integer activations, all sums below
2^24) exact, np.array_equal, on both tiles, split and unsplit; random inputs within the fp32
accumulation bound of the fp64 dequantised product (|y - ref| <= 2^-24 * K * sum |a w|), and
within max relative error 1e-3 of the reference's own fp32 loop; identical results run to run.
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

TOL = 1e-3


@pytest.fixture(scope="module")
def dev():
    import torch
    assert torch.cuda.is_available(), "gpu tests need a GPU"
    from ksq import _lib
    _lib.lib()
    return torch.device("cuda:0")


def _t(a, dev):
    import torch
    return torch.from_numpy(np.ascontiguousarray(a)).to(dev)


def _rel_err(y, ref):
    y = np.asarray(y, np.float64)
    ref = np.asarray(ref, np.float64)
    floor = 1e-3 * np.abs(ref).max(axis=-1, keepdims=True) + 1e-30
    return float((np.abs(y - ref) / np.maximum(np.abs(ref), floor)).max())


def _int_weights(wtype, g, N, K):
    nb = K // 32
    if wtype == 0:
        w = np.zeros((N, nb, 18), np.uint8)
        w[..., 0:2] = np.frombuffer(np.float16(1).tobytes(), np.uint8)
        w[..., 2:18] = g.integers(0, 256, size=(N, nb, 16), dtype=np.uint8)
        qs = w[..., 2:18].astype(np.int64)
        vals = np.concatenate([qs & 15, qs >> 4], axis=-1) - 8
    else:
        w = np.zeros((N, nb, 34), np.uint8)
        w[..., 0:2] = np.frombuffer(np.float16(1).tobytes(), np.uint8)
        w[..., 2:34] = g.integers(-128, 128, size=(N, nb, 32)).astype(np.int8).view(np.uint8)
        vals = w[..., 2:34].view(np.int8).astype(np.int64)
    return w, vals.reshape(N, K)


def _run(dev, wtype, x, w, M, N, K, workspace=False):
    import torch
    from ksq import ops
    ws = None
    if workspace:
        nbytes = ops.gemm_w16_workspace_size(M, N, K)
        ws = torch.empty(max(nbytes, 1), dtype=torch.uint8, device=dev) if nbytes else None
    y = ops.gemm_w16(wtype, _t(x, dev), _t(w, dev), M, N, K, workspace=ws)
    eng = ops.last_engines()
    torch.cuda.synchronize()
    return y.cpu().numpy(), eng


@pytest.mark.parametrize("wtype", [0, 1])
@pytest.mark.parametrize("M,N,K", [(1, 256, 1024), (2, 300, 1024), (3, 520, 2048), (4, 130, 8320),
                                   (1, 4096, 14336), (7, 200, 320), (32, 384, 2048), (45, 130, 576),
                                   (300, 256, 1024), (129, 1024, 4096),
                                   # the decode form's 16 and 8 weight rows per workgroup (512+ workgroups)
                                   # with ragged last workgroups: 16 rows at N = 14336 and N = 8200
                                   # (8 rows past N), 8 rows at N = 4100 (4 past N)
                                   (1, 14336, 4096), (4, 8200, 1024), (2, 4100, 2048)])
def test_w16_integer_inputs_exact(dev, wtype, M, N, K):
    from ksq import ops
    g = np.random.default_rng(500 + 7 * M + wtype)
    w, vals = _int_weights(wtype, g, N, K)
    amax = 40 if wtype == 0 else 3            # sum |a w| < 2^24 at K = 4096
    x = g.integers(-amax, amax + 1, size=(M, K)).astype(np.float32)
    want = (x.astype(np.int64) @ vals.T)
    assert (np.abs(x.astype(np.int64)) @ np.abs(vals).T).max() < 2 ** 24
    y, eng = _run(dev, wtype, x, w, M, N, K)
    assert np.array_equal(y, want.astype(np.float32)), (wtype, M, N, K, float(np.abs(y - want).max()))
    assert "w16" in eng
    assert ("splitk" in eng) == (ops.gemm_w16_workspace_size(M, N, K) > 0)


@pytest.mark.parametrize("wtype", [0, 1])
@pytest.mark.parametrize("M,N,K", [(1, 4096, 4096), (3, 1000, 8192), (16, 512, 2048), (96, 640, 1536),
                                   (512, 512, 4096)])
def test_w16_random_vs_oracle(dev, oracle, wtype, M, N, K):
    from ksq import refcheck
    g = np.random.default_rng(600 + M + wtype)
    x = g.standard_normal((M, K), dtype=np.float32)
    if M > 1:
        x[0] *= np.float32(1e30)                 # wide range: the three-term split keeps products exact
        x[1] *= np.float32(1e-30)
    quant = oracle.quantize_q4_0 if wtype == 0 else oracle.quantize_q8_0
    w = quant(g.standard_normal((N, K), dtype=np.float32)).reshape(N, K // 32, -1)
    y, _ = _run(dev, wtype, x, w, M, N, K, workspace=True)
    wd = refcheck.dequantize(wtype, w)
    ref64 = x.astype(np.float64) @ wd.T
    bound = np.abs(x.astype(np.float64)) @ np.abs(wd).T
    assert np.all(np.abs(y - ref64) <= 2.0 ** -24 * K * bound)
    rows = np.unique(np.linspace(0, M - 1, min(M, 6)).astype(int))
    ref32 = oracle.gemm_w16(wtype, x[rows], w, len(rows), N, K)
    assert _rel_err(y[rows], ref32) < TOL
    y2, _ = _run(dev, wtype, x, w, M, N, K)
    assert np.array_equal(y, y2)


def test_w16_baseline_shapes(dev, oracle):
    """BASELINE config 0 and config 2 shapes (M = 1 and M = 2048, N = K = 4096) through the
    reference launchers' form (ksq_gemm_w4a16 / ksq_gemm_w8a16, library pool), sampled rows
    against the reference's fp32 loop."""
    import torch
    from ksq import _lib
    L = _lib.lib()
    N = K = 4096
    for wtype, entry in ((0, "ksq_gemm_w4a16"), (1, "ksq_gemm_w8a16")):
        for M in (1, 2048):
            g = np.random.default_rng(700 + M + wtype)
            x = g.standard_normal((M, K), dtype=np.float32)
            quant = oracle.quantize_q4_0 if wtype == 0 else oracle.quantize_q8_0
            w = quant(g.standard_normal((N, K), dtype=np.float32) * 0.02).reshape(N, K // 32, -1)
            xt, wt = _t(x, dev), _t(w, dev)
            y = torch.full((M, N), float("nan"), dtype=torch.float32, device=dev)
            assert getattr(L, entry)(xt.data_ptr(), wt.data_ptr(), y.data_ptr(), M, N, K, None) == 0
            torch.cuda.synchronize()
            rows = np.unique(np.linspace(0, M - 1, min(M, 8)).astype(int))
            ref = oracle.gemm_w16(wtype, x[rows], w, len(rows), N, K)
            assert _rel_err(y.cpu().numpy()[rows], ref) < TOL, (entry, M)


# one row past the small-batch form, rows and columns one short of and one past a tile, one K step, an odd
# number of K steps, split along K: the 64 x 128 tile's edges but for (2047, 4095, 64), which takes 128 x 256
@pytest.mark.parametrize("wtype", [0, 1])
@pytest.mark.parametrize("M,N,K", [(33, 1, 64), (64, 127, 128), (65, 129, 64), (33, 200, 1088), (257, 383, 192),
                                   (1000, 4100, 128), (1025, 4097, 64), (2047, 4095, 64), (2048, 4097, 192)])
def test_w16_tile_edges_exact(dev, wtype, M, N, K):
    g = np.random.default_rng(900 + M + wtype)
    w, vals = _int_weights(wtype, g, N, K)
    amax = 250 if wtype == 0 else 15          # sum |a w| < 2^24, activations with two-term bf16 splits
    x = g.integers(-amax, amax + 1, size=(M, K)).astype(np.float32)
    want = x.astype(np.float64) @ vals.astype(np.float64).T
    assert amax * (8 if wtype == 0 else 128) * K < 2 ** 24
    y, eng = _run(dev, wtype, x, w, M, N, K, workspace=True)
    assert np.array_equal(y, want.astype(np.float32)), (wtype, M, N, K, float(np.abs(y - want).max()))
    assert "w16" in eng


# M, N, K, tile (1: 64 x 128, 2: 128 x 128, 3: 128 x 256), splits: each tile's edges in rows and columns, one
# K step, an odd and an even number of them, split along K into equal and unequal parts
TILE_CASES = [(65, 129, 704, 1, 2), (63, 161, 512, 1, 2),
              (383, 5503, 64, 2, 1), (257, 6529, 128, 2, 1), (3327, 513, 192, 2, 1), (2687, 129, 1024, 2, 4),
              (127, 5247, 1536, 2, 5),
              (385, 14113, 64, 3, 1), (385, 14081, 128, 3, 1), (3327, 1793, 192, 3, 1), (639, 3327, 1152, 3, 3),
              (257, 6655, 1024, 3, 3)]


@pytest.mark.parametrize("wtype", [0, 1])
@pytest.mark.parametrize("M,N,K,tile,splits", TILE_CASES)
def test_w16_every_tile_exact(dev, wtype, M, N, K, tile, splits):
    """The tile and split count that the shape is listed for, and exact integer results."""
    from ksq import _lib
    assert _lib.lib().ksq_debug_w16_plan(M, N, K) == tile + 16 * splits
    g = np.random.default_rng(930 + M + wtype)
    w, vals = _int_weights(wtype, g, N, K)
    amax = 250 if wtype == 0 else 15
    x = g.integers(-amax, amax + 1, size=(M, K)).astype(np.float32)
    assert amax * (8 if wtype == 0 else 128) * K < 2 ** 24
    # exact in fp32 in any order: every partial sum is an integer below 2^24
    want = x @ vals.astype(np.float32).T
    y, eng = _run(dev, wtype, x, w, M, N, K, workspace=True)
    assert np.array_equal(y, want), float(np.abs(y - want).max())
    assert eng == {"w16"} | ({"splitk"} if splits > 1 else set()), eng


@pytest.mark.parametrize("M,N,K,tile", [(130, 300, 256, 1), (257, 6529, 128, 2), (385, 14081, 128, 3)])
def test_w16_three_term_split(dev, M, N, K, tile):
    """Activations that need all 24 bits: a = 2^23 + odd integers against quants of -1, 0 and 1 (Q4_0
    nibbles 7, 8, 9), one non-zero per row, so every output is plus or minus one activation, exactly."""
    from ksq import _lib
    assert _lib.lib().ksq_debug_w16_plan(M, N, K) % 16 == tile
    g = np.random.default_rng(77)
    x = (g.integers(2 ** 23, 2 ** 24, size=(M, K)) | 1).astype(np.float32) * g.choice([-1.0, 1.0], size=(M, K)).astype(np.float32)
    w = np.zeros((N, K // 32, 18), np.uint8)
    w[..., 0:2] = np.frombuffer(np.float16(1).tobytes(), np.uint8)
    w[..., 2:] = 0x88
    pick, sign = g.integers(0, K, size=N), g.choice([-1, 1], size=N)
    for n, k in enumerate(pick):
        b, e = divmod(int(k), 32)
        q = 8 + int(sign[n])
        w[n, b, 2 + e % 16] = 0x80 | q if e < 16 else q << 4 | 8
    y, _ = _run(dev, 0, x, w, M, N, K)
    assert np.array_equal(y, x[:, pick] * sign.astype(np.float32))


def _plane_bytes(M, N, splits):
    return (splits * M * N * 4 + 255) // 256 * 256


# (the plan takes 15, 5 and 6 splits)
@pytest.mark.parametrize("wtype", [0, 1])
@pytest.mark.parametrize("M,N,K,least", [(34, 6092, 4736, 11), (46, 17713, 1280, 4), (34, 13136, 1920, 5)])
def test_w16_smaller_workspace_exact(dev, wtype, M, N, K, least):
    """A workspace, or under capture a pool, that holds fewer splits than the plan takes, but as many as
    bring the 128 x 128 grid to 512 workgroups: fewer splits, exact results; one byte less is refused."""
    import torch
    from ksq import _lib, ops
    g = np.random.default_rng(950 + wtype)
    w, vals = _int_weights(wtype, g, N, K)
    amax = 250 if wtype == 0 else 15
    x = g.integers(-amax, amax + 1, size=(M, K)).astype(np.float32)
    want = (x.astype(np.float64) @ vals.astype(np.float64).T).astype(np.float32)
    assert amax * (8 if wtype == 0 else 128) * K < 2 ** 24
    assert ops.gemm_w16_workspace_size(M, N, K) > _plane_bytes(M, N, least) and least == -(-512 // -(-N // 128))
    xt, wt = _t(x, dev), _t(w, dev)
    ws = torch.empty(_plane_bytes(M, N, least), dtype=torch.uint8, device=dev)
    assert np.array_equal(ops.gemm_w16(wtype, xt, wt, M, N, K, workspace=ws).cpu().numpy(), want)
    with pytest.raises(_lib.KsqError) as err:
        ops.gemm_w16(wtype, xt, wt, M, N, K, workspace=ws[:-1])
    assert _lib.STATUS[err.value.status] == "KSQ_ERR_WORKSPACE"
    # a pool of about that size: fewer columns of the same layer
    n = next(n for n in range(N - 32, 64, -32)
             if _plane_bytes(M, N, least) <= ops.gemm_w16_workspace_size(M, n, K) < ops.gemm_w16_workspace_size(M, N, K))
    torch.cuda.synchronize()
    _lib.lib().ksq_release()
    own = torch.cuda.Stream()
    with torch.cuda.stream(own):
        ops.gemm_w16(wtype, xt, wt[:n], M, n, K)
    out = torch.empty((M, N), dtype=torch.float32, device=dev)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=own):
        ops.gemm_w16(wtype, xt, wt, M, N, K, out=out)
    for _ in range(3):
        out.fill_(float("nan"))
        torch.cuda.synchronize()
        graph.replay()
        torch.cuda.synchronize()
        assert np.array_equal(out.cpu().numpy(), want)
    del graph
