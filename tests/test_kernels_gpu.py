"""GPU parity of every direct kernel entry point against the CPU oracle.

Inputs are seeded; the HIP path runs through the C ABI (ferrograd_amd);
torch tensors serve only as device memory.  Tolerances (BASELINE.json
north_star): GEMM outputs max normwise relative error 1e-5*sqrt(K);
elementwise / softmax / optimiser 1e-5; argmax and integer outputs
bit-exact; SGD and Adam are held to bit-exactness, which their kernels are
written to give.
"""
import math
import sys

import numpy as np
import pytest

import oracle as O
from conftest import golden, normwise_rel

pytestmark = pytest.mark.gpu

f32 = np.float32


def _torch():
    import torch
    return torch


def dev(a):
    torch = _torch()
    return torch.from_numpy(np.ascontiguousarray(a)).cuda()


def host(t):
    _torch().cuda.synchronize()
    return t.cpu().numpy()


def note(msg):
    print(msg, flush=True)
    sys.stdout.flush()


def empty(shape, dtype=None):
    torch = _torch()
    return torch.empty(shape, dtype=dtype or torch.float32, device="cuda")


# ------------------------------------------------------------------ GEMM
SHAPES = [(17, 33, 29), (64, 256, 784), (64, 10, 256), (300, 260, 100), (128, 1000, 512),
          (512, 512, 512), (256, 2048, 64), (1, 1, 1)]


def storage(layout, A, B):
    """(A_stored, B_stored) for a logical C = A.B in the given layout."""
    if layout == O.NN:
        return A, B
    if layout == O.NT:
        return A, np.ascontiguousarray(B.T)
    return np.ascontiguousarray(A.T), B


def run_gemm(ctx, layout, A, B, bias=None, act=0, want_z=True):
    M, K = A.shape
    N = B.shape[1]
    As, Bs = storage(layout, A, B)
    dA, dB = dev(As), dev(Bs)
    dC = empty((M, N))
    dZ = empty((M, N)) if want_z else None
    db = dev(bias) if bias is not None else None
    ctx.gemm(layout, M, N, K, dA, As.shape[1], dB, Bs.shape[1], dC, N, bias=db, act=act,
             Z=dZ, ldz=N)
    return host(dC), (host(dZ) if want_z else None)


@pytest.mark.parametrize("layout", [O.NN, O.NT, O.TN], ids=["NN", "NT", "TN"])
@pytest.mark.parametrize("shape", SHAPES, ids=lambda s: "x".join(map(str, s)))
@pytest.mark.parametrize("act", [O.ACT_NONE, O.ACT_RELU, O.ACT_GELU], ids=["none", "relu", "gelu"])
def test_gemm_forward_parity(gpu_ctx, layout, shape, act):
    M, N, K = shape
    note(f"gemm fwd layout={layout} M={M} N={N} K={K} act={act}")
    rng = np.random.default_rng(M * 7 + N * 13 + K + layout)
    A = rng.standard_normal((M, K)).astype(f32)
    B = rng.standard_normal((K, N)).astype(f32)
    bias = (0.1 * rng.standard_normal(N)).astype(f32)
    C, Z = run_gemm(gpu_ctx, layout, A, B, bias, act)
    Zr, Hr = O.bias_act(O.gemm(O.NN, A, B), bias, act)
    tol = 1e-5 * math.sqrt(K)
    assert normwise_rel(Z, Zr) < tol
    assert normwise_rel(C, Hr) < tol


@pytest.mark.parametrize("layout", [O.NN, O.NT, O.TN], ids=["NN", "NT", "TN"])
def test_gemm_bias_and_activation_exact_on_zero_product(gpu_ctx, layout):
    """A = 0: the output is act(bias) per column, so a bias indexing slip
    cannot hide under the GEMM tolerance."""
    M, N, K = 70, 130, 36
    note(f"gemm zero-product bias layout={layout}")
    A = np.zeros((M, K), f32)
    B = np.random.default_rng(1).standard_normal((K, N)).astype(f32)
    bias = np.linspace(-2, 2, N).astype(f32)
    for act in (O.ACT_NONE, O.ACT_RELU):
        C, Z = run_gemm(gpu_ctx, layout, A, B, bias, act)
        assert np.array_equal(Z, np.tile(bias, (M, 1)))
        assert np.array_equal(C, np.tile(O.act(act, bias), (M, 1)))
    C, _ = run_gemm(gpu_ctx, layout, A, B, bias, O.ACT_GELU)
    assert np.max(np.abs(C - np.tile(O.act(O.ACT_GELU, bias), (M, 1)))) < 1e-6


def test_gemm_k_zero_and_accumulate(gpu_ctx):
    torch = _torch()
    note("gemm K=0 and accumulate")
    M, N = 40, 24
    bias = np.arange(N, dtype=f32)
    dC = empty((M, N))
    dummy = empty((4,))
    gpu_ctx.gemm(O.NN, M, N, 0, dummy, 1, dummy, N, dC, N, bias=dev(bias), act=O.ACT_RELU)
    assert np.array_equal(host(dC), np.tile(bias, (M, 1)))
    rng = np.random.default_rng(3)
    A = rng.standard_normal((M, 50)).astype(f32)
    B = rng.standard_normal((50, N)).astype(f32)
    C0 = rng.standard_normal((M, N)).astype(f32)
    dC = dev(C0)
    gpu_ctx.gemm(O.NN, M, N, 50, dev(A), 50, dev(B), N, dC, N, accumulate=True)
    assert normwise_rel(host(dC), C0 + O.gemm(O.NN, A, B)) < 1e-5 * math.sqrt(50)
    del torch


@pytest.mark.parametrize("layout", [O.NN, O.NT, O.TN], ids=["NN", "NT", "TN"])
@pytest.mark.parametrize("act", [O.ACT_NONE, O.ACT_RELU, O.ACT_GELU], ids=["none", "relu", "gelu"])
def test_gemm_backward_epilogue_parity(gpu_ctx, layout, act):
    """C = (op(A).op(B)) * act'(Zs): the dA GEMM with the upstream activation
    derivative fused in."""
    M, N, K = 200, 136, 300
    note(f"gemm bwd layout={layout} act={act}")
    rng = np.random.default_rng(11 + layout * 3 + act)
    A = rng.standard_normal((M, K)).astype(f32)
    B = rng.standard_normal((K, N)).astype(f32)
    Zs = rng.standard_normal((M, N)).astype(f32)
    As, Bs = storage(layout, A, B)
    dC = empty((M, N))
    gpu_ctx.gemm_bwd(layout, M, N, K, dev(As), As.shape[1], dev(Bs), Bs.shape[1], dC, N, act=act,
                     Zs=dev(Zs), ldzs=N)
    ref = O.act_bwd(act, O.gemm(O.NN, A, B), Zs)
    assert normwise_rel(host(dC), ref) < 1e-5 * math.sqrt(K)


def test_gemm_c2_full_size_sampled(gpu_ctx):
    """Config 2 at its real shape, 4096^3, on the configuration's inputs
    (library generator, seed 1: A, B ~ N(0,1), bias ~ N(0, 0.1^2), dC ~
    N(0,1)): forward C = ReLU(A.B + bias) in one NN launch, then the
    backward through the ReLU mask, dZ = dC * [Z > 0], dA = dZ.B^T,
    dB = A^T.dZ, dbias = colsum(dZ), with the mask applied as the NT and TN
    GEMMs load dC (fg_linear_bwd_f32; the forward output C stands in for Z,
    [C > 0] == [Z > 0]).  Checked against float64 on 24 sampled rows
    (forward, dA) and 24 sampled columns (dB, dbias); the mask of the
    float64 reference is the GPU forward's own (a sign decided by fp32
    rounding would otherwise flip single terms)."""
    import ferrograd_amd as fa
    n = 4096
    note("gemm c2 4096^3 sampled: forward, masked dA / dB / dbias")
    A, B, G = empty((n, n)), empty((n, n)), empty((n, n))
    bias = empty((n,))
    gpu_ctx.rng_normal(1, 0, 0.0, 1.0, A, n * n)
    gpu_ctx.rng_normal(1, 1, 0.0, 1.0, B, n * n)
    gpu_ctx.rng_normal(1, 2, 0.0, 0.1, bias, n)
    gpu_ctx.rng_normal(1, 3, 0.0, 1.0, G, n * n)
    C, dX, dW, db = empty((n, n)), empty((n, n)), empty((n, n)), empty((n,))
    gpu_ctx.gemm(fa.NN, n, n, n, A, n, B, n, C, n, bias=bias, act=fa.ACT_RELU)
    # Both ways of applying the mask: dZ materialised by one pass, and the
    # prologue on the GEMMs' dC tiles (dZ never stored).
    dZ = empty((n, n))
    gpu_ctx.linear_bwd(fa.ACT_RELU, n, n, n, A, n, B, n, C, n, G, n, dX=dX, lddx=n, dW=dW,
                       lddw=n, dbias=db, dZ=dZ, lddz=n)
    pX, pW, pb = empty((n, n)), empty((n, n)), empty((n,))
    gpu_ctx.linear_bwd(fa.ACT_RELU, n, n, n, A, n, B, n, C, n, G, n, dX=pX, lddx=n, dW=pW,
                       lddw=n, dbias=pb)
    sel = np.random.default_rng(5)
    rows = np.sort(sel.choice(n, 24, replace=False))
    cols = np.sort(sel.choice(n, 24, replace=False))
    A64, B64, G64 = (host(t).astype(np.float64) for t in (A, B, G))
    Ch, bh = host(C), host(bias).astype(np.float64)
    tol = 1e-5 * math.sqrt(n)
    Zr = A64[rows] @ B64 + bh
    assert normwise_rel(Ch[rows], np.maximum(Zr, 0)) < tol
    dZr = G64[rows] * (Ch[rows] > 0)
    assert normwise_rel(host(dX)[rows], dZr @ B64.T) < tol
    dZc = G64[:, cols] * (Ch[:, cols] > 0)
    assert normwise_rel(host(dW)[:, cols], A64.T @ dZc) < tol
    assert normwise_rel(host(db)[cols], dZc.sum(axis=0)) < tol
    # The mask matters: without it dbias would be the plain column sums.
    assert normwise_rel(host(db)[cols], G64[:, cols].sum(axis=0)) > 1e-2
    # The materialised dZ is exactly dC or 0; the prologue path agrees.
    dZh = host(dZ)
    assert np.array_equal(dZh[rows], host(G)[rows] * (Ch[rows] > 0))
    assert normwise_rel(host(pX)[rows], host(dX)[rows]) < tol
    assert normwise_rel(host(pW)[:, cols], host(dW)[:, cols]) < tol
    assert normwise_rel(host(pb), host(db)) < tol


@pytest.mark.parametrize("case", [
    # (M, N, K, act, outputs, accumulate, workspace): C = act(X.W + b) with
    # X[M][K], W[K][N]; dX = dZ.W^T (NT, prologue on A), dW = X^T.dZ (TN,
    # prologue on B, dbias from its tiles).
    (17, 33, 29, O.ACT_RELU, "xwb", False, False),     # element loads, edge tiles
    (17, 33, 29, O.ACT_GELU, "xwb", True, False),
    (200, 136, 300, O.ACT_GELU, "xwb", False, False),  # any-shape kernel, K off tiles
    (512, 512, 512, O.ACT_RELU, "xwb", False, False),  # pipelined 128x128 / 128x64
    (256, 1000, 2048, O.ACT_GELU, "xwb", False, False),  # NT K = 1000: any-shape
    (2048, 4096, 1024, O.ACT_RELU, "xwb", True, False),  # 256x128 8-wave pipe (NT)
    (2048, 1024, 4096, O.ACT_GELU, "xwb", False, False),  # c5-like hidden shapes
    (64, 4096, 256, O.ACT_RELU, "x", False, True),     # dX splits K (own workspace)
    (300, 260, 100, O.ACT_RELU, "b", False, False),    # dbias alone: masked reduction
    (300, 260, 100, O.ACT_GELU, "wb", True, False),
    (128, 96, 64, O.ACT_NONE, "xwb", False, False),    # no activation: no prologue
], ids=lambda c: f"{c[0]}x{c[1]}x{c[2]}-act{c[3]}-{c[4]}{'-acc' if c[5] else ''}"
                 f"{'-ws' if c[6] else ''}")
@pytest.mark.parametrize("mat", [False, True], ids=["prologue", "dZ"])
def test_linear_bwd_parity(gpu_ctx, case, mat):
    """fg_linear_bwd_f32 against the oracle: dZ = act_bwd(dC, Z) on the CPU,
    then the oracle's NT / TN GEMMs and column sums.  The GPU either scales
    the dC tiles by act'(Z) as the GEMMs load them (prologue; dZ never
    stored) or materialises dZ in one pass that also sums its columns (dZ
    checked too: bit-exact for ReLU, 1e-5 for GELU).  GEMM tolerance
    1e-5*sqrt(reduction length)."""
    torch = _torch()
    import ferrograd_amd as fa
    M, N, K, act, outs, acc, ws = case
    note(f"linear_bwd M={M} N={N} K={K} act={act} outputs={outs} acc={acc} ws={ws} mat={mat}")
    rng = np.random.default_rng(M + 7 * N + 3 * K + act)
    X = rng.standard_normal((M, K)).astype(f32)
    W = (rng.standard_normal((K, N)) / math.sqrt(K)).astype(f32)
    Z = rng.standard_normal((M, N)).astype(f32)
    dC = rng.standard_normal((M, N)).astype(f32)
    dX0 = rng.standard_normal((M, K)).astype(f32)
    dW0 = rng.standard_normal((K, N)).astype(f32)
    db0 = rng.standard_normal(N).astype(f32)
    dZ = O.act_bwd(act, dC, Z) if act != O.ACT_NONE else dC
    ref_x = O.gemm(O.NT, dZ, W) + (dX0 if acc else 0)
    ref_w = O.gemm(O.TN, X, dZ) + (dW0 if acc else 0)
    ref_b = O.bias_grad(dZ) + (db0 if acc else 0)
    ctx = gpu_ctx
    own = None
    if ws:
        own = fa.Context(0, torch.cuda.current_stream().cuda_stream)
        own.reserve_workspace(16 << 20)
        ctx = own
    try:
        gx = dev(dX0) if "x" in outs else None
        gw = dev(dW0) if "w" in outs else None
        gb = dev(db0) if "b" in outs else None
        gz = empty((M, N)) if mat else None
        ctx.linear_bwd(act, M, N, K, dev(X), K, dev(W), N, dev(Z), N, dev(dC), N, dX=gx,
                       lddx=K, dW=gw, lddw=N, dbias=gb, accumulate=acc, dZ=gz, lddz=N)
        if mat and act != O.ACT_NONE:
            if act == O.ACT_RELU:
                assert np.array_equal(host(gz), dZ)
            else:
                assert normwise_rel(host(gz), dZ) < 1e-5
        if "x" in outs:
            assert normwise_rel(host(gx), ref_x) < 1e-5 * math.sqrt(N)
        if "w" in outs:
            assert normwise_rel(host(gw), ref_w) < 1e-5 * math.sqrt(M)
        if "b" in outs:
            assert normwise_rel(host(gb), ref_b) < 1e-5 * math.sqrt(M)
    finally:
        if own is not None:
            own.sync()
            own.close()


@pytest.mark.parametrize("case", [
    # (M, N, K, act, accumulate)
    (2048, 4096, 4096, O.ACT_GELU, False),  # hidden layer: the 8-wave tiles' pair
    (2048, 4096, 1024, O.ACT_NONE, False),  # first layer: the 128x64 tiles' pair
    (2048, 1000, 4096, O.ACT_GELU, False),  # 1000-wide head (dX's last K tile partial): two launches
    (64, 256, 784, O.ACT_RELU, True),       # c1's first layer: the small kernels' pair
    (100, 33, 17, O.ACT_GELU, True),        # unaligned rows: two launches
], ids=lambda c: f"{c[0]}x{c[1]}x{c[2]}-act{c[3]}{'-acc' if c[4] else ''}")
def test_matmul_bwd_matches_separate_calls(case):
    """fg_matmul_bwd_f32 (dW = X^T.dZ + dbias, dX = (dZ.W^T) * act'(Zs), one
    launch where the two kernels pair) against fg_gemm_dw_f32 and
    fg_gemm_bwd_f32 on the same context and workspace: every output equal
    bit for bit.  Shapes the oracle finishes quickly are also checked
    against it (GEMM tolerance 1e-5*sqrt(reduction length))."""
    torch = _torch()
    import ferrograd_amd as fa
    M, N, K, act, acc = case
    note(f"matmul_bwd M={M} N={N} K={K} act={act} acc={acc}")
    rng = np.random.default_rng(M + 5 * N + 11 * K)
    X = rng.standard_normal((M, K)).astype(f32)
    W = (rng.standard_normal((K, N)) / math.sqrt(K)).astype(f32)
    dZ = rng.standard_normal((M, N)).astype(f32)
    Zs = rng.standard_normal((M, K)).astype(f32)
    dX0, dW0, db0 = (rng.standard_normal(s).astype(f32) for s in ((M, K), (K, N), (N,)))
    own = fa.Context(0, torch.cuda.current_stream().cuda_stream)
    try:
        own.reserve_workspace(1 << 20)
        gX, gW, gdZ, gZs = dev(X), dev(W), dev(dZ), dev(Zs)
        outs = []
        for fused in (True, False):
            gx, gw, gb = dev(dX0), dev(dW0), dev(db0)
            if fused:
                own.matmul_bwd(M, N, K, gX, K, gW, N, gdZ, N, gx, K, gw, N, dbias=gb, act=act,
                               Zs=gZs, ldzs=K, accumulate=acc)
            else:
                own.gemm_dw(K, N, M, gX, K, gdZ, N, gw, N, accumulate=acc, colsum=gb,
                            colsum_accumulate=acc)
                own.gemm_bwd(fa.NT, M, K, N, gdZ, N, gW, N, gx, K, act=act, Zs=gZs, ldzs=K,
                             accumulate=acc)
            own.sync()
            outs.append([host(gx), host(gw), host(gb)])
        for a, b in zip(*outs):
            assert np.array_equal(a, b)
        if M * N * K <= 1 << 24:
            ref_x = O.gemm(O.NT, dZ, W)
            ref_x = (O.act_bwd(act, ref_x, Zs) if act != O.ACT_NONE else ref_x) + (
                dX0 if acc else 0)
            ref_w = O.gemm(O.TN, X, dZ) + (dW0 if acc else 0)
            ref_b = O.bias_grad(dZ) + (db0 if acc else 0)
            gx, gw, gb = outs[0]
            assert normwise_rel(gx, ref_x) < 1e-5 * math.sqrt(N)
            assert normwise_rel(gw, ref_w) < 1e-5 * math.sqrt(M)
            assert normwise_rel(gb, ref_b) < 1e-5 * math.sqrt(M)
    finally:
        own.sync()
        own.close()


def test_matmul_bwd_rejects_bad_arguments(gpu_ctx):
    """fg_matmul_bwd_f32 / _x16 report a missing operand, a leading
    dimension below its row length and an activation without Zs as
    INVALID_ARGUMENT, launching nothing."""
    import ferrograd_amd as fa
    M, N, K = 64, 32, 16
    X, W, dZ, dX, dW = (empty(s) for s in ((M, K), (K, N), (M, N), (M, K), (K, N)))
    for kw, bad in ((dict(ldx=K - 1), "ld"), (dict(X=None), "null"), (dict(act=O.ACT_GELU), "zs")):
        a = dict(X=X, ldx=K, W=W, ldw=N, dZ=dZ, lddz=N, dX=dX, lddx=K, dW=dW, lddw=N, act=0)
        a.update(kw)
        with pytest.raises(fa.FgError) as e:
            gpu_ctx.matmul_bwd(M, N, K, a["X"], a["ldx"], a["W"], a["ldw"], a["dZ"], a["lddz"],
                               a["dX"], a["lddx"], a["dW"], a["lddw"], act=a["act"])
        assert e.value.code == 1, bad
        with pytest.raises(fa.FgError) as e:
            gpu_ctx.matmul_bwd_x16(fa.DTYPE_BF16, M, N, K, a["X"], a["ldx"], a["W"], a["ldw"],
                                   a["dZ"], a["lddz"], a["dX"], a["lddx"], a["dW"], a["lddw"],
                                   act=a["act"])
        assert e.value.code == 1, bad


@pytest.mark.parametrize("mat", [False, True], ids=["prologue", "dZ"])
def test_linear_bwd_relu_mask_from_output(gpu_ctx, mat):
    """For ReLU the forward output C = max(Z, 0) gives the same mask as Z,
    including Z == 0 exactly (gradient 0, the [z > 0] convention): the
    results with Zs = C and Zs = Z are identical bit for bit."""
    M, N, K = 256, 512, 384
    rng = np.random.default_rng(3)
    X = rng.standard_normal((M, K)).astype(f32)
    W = rng.standard_normal((K, N)).astype(f32)
    Z = rng.standard_normal((M, N)).astype(f32)
    Z[rng.random((M, N)) < 0.05] = 0.0
    Cm = np.maximum(Z, 0)
    dC = rng.standard_normal((M, N)).astype(f32)
    res = []
    for zs in (Z, Cm):
        gx, gw, gb = empty((M, K)), empty((K, N)), empty((N,))
        gz = empty((M, N)) if mat else None
        gpu_ctx.linear_bwd(O.ACT_RELU, M, N, K, dev(X), K, dev(W), N, dev(zs), N, dev(dC), N,
                           dX=gx, lddx=K, dW=gw, lddw=N, dbias=gb, dZ=gz, lddz=N)
        res.append([host(gx), host(gw), host(gb)])
    for a, b in zip(*res):
        assert np.array_equal(a, b)


@pytest.mark.parametrize("case", [
    # (layout, M, N, K, mode): shapes that select each configuration of the
    # pipelined kernel (k_gemm.hip pick_cfg), edge tiles included.
    (O.NN, 2000, 4000, 4096, "fwd"),   # 256x128, 8 waves; partial M and N tiles
    (O.NT, 2048, 4096, 4096, "bwd"),   # 256x128, 8 waves; GELU' epilogue
    (O.TN, 4096, 4096, 2048, "fwd"),   # 256x128, 4 waves (c5 dW)
    (O.NT, 2048, 2000, 1024, "fwd"),   # 128x128
    (O.NN, 2048, 1000, 4096, "fwd"),   # 128x64 (c5 head)
    (O.TN, 1000, 4096, 2048, "bwd"),   # 128x64; partial M tile
    (O.NN, 2048, 4096, 32, "fwd"),     # one K tile (256x128, 8 waves, BK 32)
    (O.TN, 4096, 4096, 16, "fwd"),     # one K tile (256x128, 4 waves, BK 16)
    # K % BK != 0: the register-staged kernel with the same tiles
    (O.NT, 2048, 4096, 1000, "bwd"),   # 256x128, 8 waves (c5 head dA)
    (O.NT, 2048, 4096, 1020, "bwd"),   # a 28-deep tail: every MFMA group of the tail tile
    (O.TN, 1024, 4096, 1000, "fwd"),   # 128x64, row-contiguous operands
    (O.TN, 1024, 4096, 1001, "fwd"),   # odd K: a lane half past K in the last tail step
    (O.TN, 4096, 4096, 2020, "bwd"),   # 256x128, 8 waves, interleaved TN fragments
    (O.NN, 2048, 4096, 20, "fwd"),     # K below one tile
    (O.NT, 2048, 4096, 12, "bwd"),     # K below one tile, NT
    (O.NN, 2000, 4000, 1000, "fwd"),   # K tail on partial M and N edge tiles
    (O.NT, 1000, 1000, 996, "bwd"),    # 64x64 tiles, BK 16, a 4-deep tail, partial tiles
], ids=lambda c: f"{['NN', 'NT', 'TN'][c[0]]}-{c[1]}x{c[2]}x{c[3]}-{c[4]}")
def test_gemm_pipe_configs_sampled(gpu_ctx, case):
    """The large tile configurations at full size (and the same tiles for K
    not a multiple of the tile depth), checked on 32 sampled output rows
    against float64 dot products: forward with bias + GELU (C and Z), or
    backward with the GELU derivative of a saved Zs."""
    torch = _torch()
    layout, M, N, K, mode = case
    note(f"gemm pipe config layout={layout} M={M} N={N} K={K} mode={mode}")
    g = torch.Generator(device="cuda").manual_seed(M + N + K + layout)
    a_shape = (K, M) if layout == O.TN else (M, K)
    b_shape = (N, K) if layout == O.NT else (K, N)
    dA = torch.randn(a_shape, device="cuda", generator=g)
    dB = 0.05 * torch.randn(b_shape, device="cuda", generator=g)
    dC, dZ = empty((M, N)), empty((M, N))
    lda, ldb = a_shape[1], b_shape[1]
    if mode == "fwd":
        dbias = 0.1 * torch.randn((N,), device="cuda", generator=g)
        gpu_ctx.gemm(layout, M, N, K, dA, lda, dB, ldb, dC, N, bias=dbias, act=O.ACT_GELU,
                     Z=dZ, ldz=N)
    else:
        dZs = torch.randn((M, N), device="cuda", generator=g)
        gpu_ctx.gemm_bwd(layout, M, N, K, dA, lda, dB, ldb, dC, N, act=O.ACT_GELU, Zs=dZs,
                         ldzs=N)
    rows = np.sort(np.random.default_rng(M * 3 + N).choice(M, 32, replace=False))
    rows[-1] = M - 1  # the last row sits in the edge tile when M is not a tile multiple
    A = host(dA).astype(np.float64)
    B = host(dB).astype(np.float64)
    Ar = A[:, rows].T if layout == O.TN else A[rows]
    Bf = B.T if layout == O.NT else B
    P = Ar @ Bf
    tol = 1e-5 * math.sqrt(K)
    if mode == "fwd":
        Zr = P + host(dbias).astype(np.float64)
        assert normwise_rel(host(dZ)[rows], Zr) < tol
        assert normwise_rel(host(dC)[rows], O.act(O.ACT_GELU, Zr)) < tol
    else:
        ref = O.act_bwd(O.ACT_GELU, P, host(dZs)[rows].astype(np.float64))
        assert normwise_rel(host(dC)[rows], ref) < tol


@pytest.mark.parametrize("layout", [O.NN, O.NT, O.TN], ids=["NN", "NT", "TN"])
@pytest.mark.parametrize("shape", [(2048, 4096, 512), (1024, 1024, 256), (200, 136, 64)],
                         ids=lambda s: "x".join(map(str, s)))
def test_gemm_pipe_strided_accumulate(gpu_ctx, layout, shape):
    """The pipelined kernel on operands and output with leading dimensions
    wider than their rows (padding filled with NaN, which must not be
    read into valid outputs) and C += A.B into a NaN-free C: checked in full
    against float64, padding of C untouched."""
    torch = _torch()
    M, N, K = shape
    note(f"gemm pipe strided accumulate layout={layout} M={M} N={N} K={K}")
    rng = np.random.default_rng(M + 3 * N + 7 * K + layout)
    A = rng.standard_normal((M, K)).astype(f32)
    B = (0.05 * rng.standard_normal((K, N))).astype(f32)
    As, Bs = storage(layout, A, B)
    pa, pb, pc = 8, 4, 12
    Ap = np.full((As.shape[0], As.shape[1] + pa), np.nan, f32)
    Ap[:, :As.shape[1]] = As
    Bp = np.full((Bs.shape[0], Bs.shape[1] + pb), np.nan, f32)
    Bp[:, :Bs.shape[1]] = Bs
    C0 = rng.standard_normal((M, N)).astype(f32)
    Cp = np.full((M, N + pc), -7.0, f32)
    Cp[:, :N] = C0
    dC = dev(Cp)
    gpu_ctx.gemm(layout, M, N, K, dev(Ap), Ap.shape[1], dev(Bp), Bp.shape[1], dC, N + pc,
                 accumulate=True)
    got = host(dC)
    ref = C0.astype(np.float64) + A.astype(np.float64) @ B.astype(np.float64)
    assert normwise_rel(got[:, :N], ref) < 1e-5 * math.sqrt(K)
    assert np.array_equal(got[:, N:], Cp[:, N:])
    del torch


@pytest.mark.parametrize("case", [
    # (layout, M, N, K, mode, act, accumulate): outputs of a few tiles with
    # long K, which split K over workgroups when the workspace holds the slots
    (O.NN, 64, 256, 784, "fwd", O.ACT_RELU, False),   # c1 layer 1 (4 tiles)
    (O.NN, 64, 10, 1024, "fwd", O.ACT_NONE, False),   # N = 10 past the skinny kernel's K
    (O.NT, 64, 784, 256, "bwd", O.ACT_NONE, False),   # c1 dX
    (O.NN, 100, 200, 3000, "fwd", O.ACT_GELU, False),  # edge tiles, K off the tile depth
    (O.NT, 96, 128, 4096, "bwd", O.ACT_GELU, False),   # act' of a saved Zs
    (O.TN, 128, 64, 2048, "fwd", O.ACT_NONE, True),    # C += A^T.B
], ids=lambda c: f"{['NN', 'NT', 'TN'][c[0]]}-{c[1]}x{c[2]}x{c[3]}-{c[4]}-act{c[5]}"
                 f"{'-acc' if c[6] else ''}")
def test_gemm_split_k(gpu_ctx, case):
    """Split-K GEMMs (slots summed in a fixed order, then the epilogue):
    against float64 with the CPU oracle's epilogue, bit-identical on a
    second run, and within tolerance of the unsplit kernel (a context with
    no workspace) but not bit-identical to it (the split did happen).  The
    workspace is reserved on a context of the test's own, so the shared
    context's direct GEMMs keep their unsplit path."""
    torch = _torch()
    import ferrograd_amd as fa
    layout, M, N, K, mode, act, acc = case
    note(f"gemm split-K layout={layout} M={M} N={N} K={K} mode={mode} act={act} acc={acc}")
    rng = np.random.default_rng(M * 5 + N + K + layout)
    A = rng.standard_normal((M, K)).astype(f32)
    B = (0.05 * rng.standard_normal((K, N))).astype(f32)
    bias = (0.1 * rng.standard_normal(N)).astype(f32)
    Zs = rng.standard_normal((M, N)).astype(f32)
    C0 = rng.standard_normal((M, N)).astype(f32)
    As, Bs = storage(layout, A, B)
    dA, dB, db, dZs = dev(As), dev(Bs), dev(bias), dev(Zs)

    def run(ctx):
        dC = dev(C0) if acc else empty((M, N))
        dZ = empty((M, N))
        if mode == "fwd":
            ctx.gemm(layout, M, N, K, dA, As.shape[1], dB, Bs.shape[1], dC, N,
                     bias=None if acc else db, act=act, Z=None if acc else dZ, ldz=N,
                     accumulate=acc)
        else:
            ctx.gemm_bwd(layout, M, N, K, dA, As.shape[1], dB, Bs.shape[1], dC, N, act=act,
                         Zs=dZs, ldzs=N)
        return host(dC), host(dZ)

    stream = torch.cuda.current_stream().cuda_stream
    split = fa.Context(0, stream)
    try:
        split.reserve_workspace(16 << 20)
        C1, Z1 = run(split)
        C2, Z2 = run(split)
    finally:
        split.sync()
        split.close()
    assert np.array_equal(C1, C2)
    P = A.astype(np.float64) @ B.astype(np.float64)
    tol = 1e-5 * math.sqrt(K)
    if mode == "fwd" and acc:
        assert normwise_rel(C1, C0 + P) < tol
    elif mode == "fwd":
        Zr = P + bias
        assert normwise_rel(Z1, Zr) < tol
        assert normwise_rel(C1, O.act(act, Zr)) < tol
    else:
        assert normwise_rel(C1, O.act_bwd(act, P, Zs)) < tol
    plain = fa.Context(0, stream)  # no workspace: no split
    try:
        C3, _ = run(plain)
    finally:
        plain.sync()
        plain.close()
    assert normwise_rel(C1, C3) < tol
    # Another summation order: some of the M*N sums round differently.
    assert not np.array_equal(C1, C3)


# ----------------------------------------------------- bias grad, act bwd
@pytest.mark.parametrize("shape", [(2048, 4096), (64, 10), (1, 5), (1000, 1000), (3, 4097),
                                   (4096, 1000)], ids=lambda s: "x".join(map(str, s)))
def test_bias_grad_parity(gpu_ctx, shape):
    M, N = shape
    note(f"bias_grad M={M} N={N}")
    dZ = np.random.default_rng(M + N).standard_normal((M, N)).astype(f32)
    out = empty((N,))
    gpu_ctx.bias_grad(M, N, dev(dZ), N, out)
    ref = O.bias_grad(dZ)
    assert normwise_rel(host(out), ref) < 1e-5
    # accumulate
    gpu_ctx.bias_grad(M, N, dev(dZ), N, out, accumulate=True)
    assert normwise_rel(host(out), 2 * ref.astype(np.float64)) < 1e-5


@pytest.mark.parametrize("shape", [(256, 4096, 2048), (1024, 4096, 2048), (96, 128, 64),
                                   (784, 256, 64), (37, 29, 300), (130, 200, 33), (4096, 1000, 2048),
                                   (1024, 4096, 1000), (256, 512, 999)],
                         ids=lambda s: "x".join(map(str, s)))
def test_gemm_dw_fused_bias_grad(gpu_ctx, shape):
    """dW = A^T.dZ and dbias = column sums of dZ in one launch (TN layout):
    dW to the GEMM tolerance, dbias to 1e-5 of the float64 column sums, both
    with and without accumulation.  The shapes cover the pipelined path
    (K a multiple of 32, and K = 1000, 999 with the K tail's rows added to
    the column sums after the whole tiles') and the other kernel (K = 300,
    33, whose M is not a multiple of 4)."""
    M, N, K = shape  # dW is M x N; the reduction runs over K rows
    note(f"gemm_dw M={M} N={N} K={K}")
    rng = np.random.default_rng(M + 3 * N + K)
    A = rng.standard_normal((K, M)).astype(f32)
    dZ = rng.standard_normal((K, N)).astype(f32)
    C, db = empty((M, N)), empty((N,))
    gpu_ctx.gemm_dw(M, N, K, dev(A), M, dev(dZ), N, C, N, colsum=db)
    refC = O.gemm(O.TN, A, dZ)
    refb = O.bias_grad(dZ)
    assert normwise_rel(host(C), refC) < 1e-5 * math.sqrt(K)
    assert normwise_rel(host(db), refb) < 1e-5
    gpu_ctx.gemm_dw(M, N, K, dev(A), M, dev(dZ), N, C, N, accumulate=True, colsum=db,
                    colsum_accumulate=True)
    assert normwise_rel(host(C), 2 * refC.astype(np.float64)) < 1e-5 * math.sqrt(K)
    assert normwise_rel(host(db), 2 * refb.astype(np.float64)) < 1e-5


SKINNY = [(64, 10, 256), (1, 1, 1), (130, 16, 255), (200, 3, 17), (64, 16, 1), (257, 10, 64)]


@pytest.mark.parametrize("layout", [O.NN, O.NT, O.TN], ids=["NN", "NT", "TN"])
@pytest.mark.parametrize("shape", SKINNY, ids=lambda s: "x".join(map(str, s)))
def test_gemm_skinny_parity(gpu_ctx, layout, shape):
    """Shapes with N <= 16 and K <= 256 (the second layer and head gradients
    of a small MLP) take the one-round-trip kernel of k_gemm_skinny.hip.
    Against the oracle: the forward epilogue (bias + GELU, Z stored), bias
    placement exactly (A = 0 gives Z = bias), the act' backward epilogue,
    accumulate, and for TN the fused column sums, plain and accumulated.  M
    up to five 64-row workgroups, N from 1 to 16, K from 1 to 256."""
    M, N, K = shape
    note(f"gemm skinny layout={layout} M={M} N={N} K={K}")
    rng = np.random.default_rng(M * 5 + N * 11 + K + layout)
    A = rng.standard_normal((M, K)).astype(f32)
    B = rng.standard_normal((K, N)).astype(f32)
    bias = (0.1 * rng.standard_normal(N)).astype(f32)
    tol = 1e-5 * math.sqrt(K)
    C, Z = run_gemm(gpu_ctx, layout, A, B, bias, O.ACT_GELU)
    Zr, Hr = O.bias_act(O.gemm(O.NN, A, B), bias, O.ACT_GELU)
    assert normwise_rel(Z, Zr) < tol
    assert normwise_rel(C, Hr) < tol
    C0, Z0 = run_gemm(gpu_ctx, layout, np.zeros_like(A), B, bias, O.ACT_RELU)
    assert np.array_equal(Z0, np.tile(bias, (M, 1)))
    assert np.array_equal(C0, np.tile(np.maximum(bias, 0), (M, 1)))
    As, Bs = storage(layout, A, B)
    Zs = rng.standard_normal((M, N)).astype(f32)
    dC = empty((M, N))
    gpu_ctx.gemm_bwd(layout, M, N, K, dev(As), As.shape[1], dev(Bs), Bs.shape[1], dC, N,
                     act=O.ACT_GELU, Zs=dev(Zs), ldzs=N)
    assert normwise_rel(host(dC), O.act_bwd(O.ACT_GELU, O.gemm(O.NN, A, B), Zs)) < tol
    Cin = rng.standard_normal((M, N)).astype(f32)
    dC = dev(Cin)
    gpu_ctx.gemm(layout, M, N, K, dev(As), As.shape[1], dev(Bs), Bs.shape[1], dC, N,
                 accumulate=True)
    assert normwise_rel(host(dC), Cin + O.gemm(O.NN, A, B)) < tol
    if layout == O.TN:
        # dW = X^T.dZ with dbias = column sums of dZ: here X = As ([K][M]), dZ = Bs.
        C, db = empty((M, N)), empty((N,))
        gpu_ctx.gemm_dw(M, N, K, dev(As), M, dev(Bs), N, C, N, colsum=db)
        refb = O.bias_grad(Bs)
        assert normwise_rel(host(C), O.gemm(O.TN, As, Bs)) < tol
        assert normwise_rel(host(db), refb) < 1e-5
        gpu_ctx.gemm_dw(M, N, K, dev(As), M, dev(Bs), N, C, N, accumulate=True, colsum=db,
                        colsum_accumulate=True)
        assert normwise_rel(host(db), 2 * refb.astype(np.float64)) < 1e-5


@pytest.mark.parametrize("n", [1, 7, 4096, 1000003])
def test_act_bwd_parity(gpu_ctx, n):
    note(f"act_bwd n={n}")
    rng = np.random.default_rng(n)
    dH = rng.standard_normal(n).astype(f32)
    Z = (3 * rng.standard_normal(n)).astype(f32)
    out = empty((n,))
    gpu_ctx.act_bwd(O.ACT_RELU, n, dev(dH), dev(Z), out)
    assert np.array_equal(host(out), O.act_bwd(O.ACT_RELU, dH, Z))
    gpu_ctx.act_bwd(O.ACT_GELU, n, dev(dH), dev(Z), out)
    ref = O.act_bwd(O.ACT_GELU, dH, Z)
    assert np.max(np.abs(host(out) - ref) / np.maximum(np.abs(ref), 1.0)) < 1e-5


# Few-row GEMMs: a whole step, its remainders, the columns' and rows' edges,
# odd rows; 4100 and more of K split it.
@pytest.mark.parametrize("place", ["plain", "padded", "offset"])
@pytest.mark.parametrize("layout", [O.NN, O.NT], ids=["NN", "NT"])
@pytest.mark.parametrize("dtype", [0, 1, 2], ids=["f32", "f16", "bf16"])
def test_gemm_few_rows(gpu_ctx, dtype, layout, place):
    """Small-integer operands (every sum exact in fp32, whatever its order),
    with NaN around every row (padded) and before and after the tensors:
    outputs bit for bit, forward with bias + ReLU + Z, backward through a ReLU
    mask, C +=."""
    torch = _torch()
    dt = [torch.float32, torch.float16, torch.bfloat16][dtype]
    gpu_ctx.reserve_workspace(8 << 20)
    g = torch.Generator().manual_seed(7)

    def ints(r, c, lim):  # a [r][c] tensor inside NaN, its leading dimension
        ld = c + (3 if place == "padded" else 0)
        off = 1 if place == "offset" else 64
        v = torch.randint(-lim, lim + 1, (r, c), generator=g).to(dt)
        buf = torch.full((off + r * ld + 64,), float("nan"), dtype=dt)
        buf[off:off + r * ld].view(r, ld)[:, :c] = v
        buf = buf.cuda()
        return v.double(), buf, buf[off:], ld

    for M, N, K in [(1, 2, 1), (1, 33, 129), (16, 31, 64), (17, 100, 63), (33, 64, 517),
                    (64, 95, 1024), (7, 1000, 4100), (32, 129, 8191), (64, 2100, 2050)]:
        if dtype == 0 and M > 32 and N * K < 1 << 22:
            M = 30  # (the fp32 kernel's range)
        note(f"gemm_few_rows {dtype} {layout} {place} {M}x{N}x{K}")
        a, _ka, A, lda = ints(M, K, 2)
        b, _kb, B, ldb = ints(*((K, N) if layout == O.NN else (N, K)), 2)
        bias, _kc, dbias, _ = ints(1, N, 4)
        zs, _kd, dZs, ldzs = ints(M, N, 1)
        old, _ke, C, ldc = ints(M, N, 8)
        v = (a @ (b if layout == O.NN else b.T)).to(dt)
        z = (v.double() + bias).to(dt)
        Z = torch.empty(M, N, dtype=dt, device="cuda")

        def got(t, ld):
            torch.cuda.synchronize()
            return t[:M * ld].view(M, ld)[:, :N].cpu()

        def call(mode, acc, act):
            kw = dict(act=act, accumulate=acc)
            if mode == 0:
                kw.update(bias=dbias, Z=Z, ldz=N)
            else:
                kw.update(Zs=dZs, ldzs=ldzs)
            args = (layout, M, N, K, A, lda, B, ldb, C, ldc)
            if dtype == 0:
                (gpu_ctx.gemm if mode == 0 else gpu_ctx.gemm_bwd)(*args, **kw)
            else:
                (gpu_ctx.gemm_x16 if mode == 0 else gpu_ctx.gemm_bwd_x16)(dtype, *args, **kw)

        call(0, True, O.ACT_NONE)
        assert torch.equal(got(C, ldc), (z.double() + old).to(dt))
        call(0, False, O.ACT_RELU)
        assert torch.equal(got(C, ldc), z.clamp(min=0))
        assert torch.equal(Z.cpu(), z)
        call(1, False, O.ACT_RELU)
        assert torch.equal(got(C, ldc), torch.where(zs > 0, v, torch.zeros_like(v)))


# fp32 tiles on rows of any alignment: every K remainder of the tile pipeline
# (1 to 9 tiles of 16 and a tail), rows that end between 16-byte chunks (whose
# last one the K tail takes), edges of 64- and 128-wide tiles, K slices with
# column sums.
@pytest.mark.parametrize("place", ["plain", "padded", "offset"])
@pytest.mark.parametrize("layout", [O.NN, O.NT, O.TN], ids=["NN", "NT", "TN"])
def test_gemm_f32_any_rows(gpu_ctx, layout, place):
    """Small-integer operands (every sum exact in fp32, whatever its order),
    with NaN around every row (padded) and before and after the tensors:
    outputs and column sums bit for bit."""
    torch = _torch()
    gpu_ctx.reserve_workspace(64 << 20)
    g = torch.Generator().manual_seed(11)

    def ints(r, c):
        ld = c + (3 if place == "padded" else 0)
        off = 1 if place == "offset" else 64
        v = torch.randint(-3, 4, (r, c), generator=g).float()
        buf = torch.full((off + r * ld + 64,), float("nan"))
        buf[off:off + r * ld].view(r, ld)[:, :c] = v
        buf = buf.cuda()
        return v.double(), buf[off:], ld

    shapes = [(65, 67, 16 * t + x) for t in range(1, 10) for x in (0, 5)]
    shapes += [(4, 4, 1), (5, 7, 15), (63, 4, 33), (129, 130, 64), (128, 66, 256),
               (100, 201, 3000), (500, 1000, 1500), (1000, 1501, 400)]
    for M, N, K in shapes:
        if layout != O.TN and M <= 32:
            continue  # (few rows: another kernel)
        note(f"gemm_f32_any_rows {layout} {place} {M}x{N}x{K}")
        a, A, lda = ints(*((K, M) if layout == O.TN else (M, K)))
        b, B, ldb = ints(*((N, K) if layout == O.NT else (K, N)))
        old, C, ldc = ints(M, N)
        ref = (a.T if layout == O.TN else a) @ (b.T if layout == O.NT else b)

        def got():
            torch.cuda.synchronize()
            return C[:M * ldc].view(M, ldc)[:, :N].cpu().double()

        gpu_ctx.gemm(layout, M, N, K, A, lda, B, ldb, C, ldc, accumulate=True)
        assert torch.equal(got(), ref + old)
        if layout == O.TN:
            cs, S, _ = ints(1, N)
            gpu_ctx.gemm_dw(M, N, K, A, lda, B, ldb, C, ldc, colsum=S, colsum_accumulate=True)
            assert torch.equal(got(), ref)
            assert torch.equal(S[:N].cpu().double(), (cs + b.sum(0)).reshape(-1))
        else:
            zs, Zs, ldzs = ints(M, N)
            gpu_ctx.gemm_bwd(layout, M, N, K, A, lda, B, ldb, C, ldc, act=O.ACT_RELU, Zs=Zs,
                             ldzs=ldzs)
            assert torch.equal(got(), torch.where(zs > 0, ref, torch.zeros_like(ref)))


@pytest.mark.parametrize("layout", [O.NN, O.NT, O.TN], ids=["NN", "NT", "TN"])
def test_gemm_f32_deep_k(gpu_ctx, layout):
    """Few outputs of a K so deep that it takes more than 16 slices (odd counts of
    them, a last slice of any length): small-integer operands, outputs and column
    sums bit for bit."""
    torch = _torch()
    gpu_ctx.reserve_workspace(64 << 20)
    g = torch.Generator().manual_seed(23)
    for M, N, K in ((56, 64, 40000), (130, 70, 20011), (64, 200, 65536), (256, 64, 9001)):
        note(f"gemm_f32_deep_k {layout} {M}x{N}x{K}")
        a = torch.randint(-3, 4, (K, M) if layout == O.TN else (M, K), generator=g).float()
        b = torch.randint(-3, 4, (N, K) if layout == O.NT else (K, N), generator=g).float()
        ref = ((a.T if layout == O.TN else a).double() @
               (b.T if layout == O.NT else b).double()).float()
        A, B = a.cuda(), b.cuda()
        C, S = empty((M, N)), empty((N,))
        gpu_ctx.gemm(layout, M, N, K, A, A.shape[1], B, B.shape[1], C, N)
        torch.cuda.synchronize()
        assert torch.equal(C.cpu(), ref)
        if layout == O.TN:
            gpu_ctx.gemm_dw(M, N, K, A, M, B, N, C, N, colsum=S)
            torch.cuda.synchronize()
            assert torch.equal(C.cpu(), ref)
            assert torch.equal(S.cpu().double(), b.double().sum(0))


@pytest.mark.parametrize("dims", [(448, 1024, 448), (640, 2992, 88), (512, 512, 64), (64, 256, 784),
                                  (300, 700, 130), (67, 378, 2229), (496, 960, 128)],
                         ids=lambda d: "x".join(map(str, d)))
def test_matmul_bwd_slices(gpu_ctx, dims):
    """dW (+ dbias) and dX whose K splits, together or apart: small-integer
    operands, every gradient bit for bit, with and without accumulation; and on
    normal ones the bits of the two calls."""
    torch = _torch()
    gpu_ctx.reserve_workspace(64 << 20)
    M, N, K = dims
    g = torch.Generator().manual_seed(29)
    x, w, dz, zs, dx0, dw0, db0 = (torch.randint(-3, 4, s, generator=g).float() for s in
                                   ((M, K), (K, N), (M, N), (M, K), (M, K), (K, N), (N,)))
    X, W, dZ, Zs = (t.cuda() for t in (x, w, dz, zs))
    dw, db = (x.T.double() @ dz.double()).float(), dz.double().sum(0).float()
    dx = torch.where(zs > 0, (dz.double() @ w.T.double()).float(), torch.zeros(M, K))
    for acc in (False, True):
        dX, dW, dB = dx0.cuda(), dw0.cuda(), db0.cuda()
        gpu_ctx.matmul_bwd(M, N, K, X, K, W, N, dZ, N, dX, K, dW, N, dbias=dB, act=O.ACT_RELU,
                           Zs=Zs, ldzs=K, accumulate=acc)
        torch.cuda.synchronize()
        assert torch.equal(dW.cpu(), dw + dw0 if acc else dw)
        assert torch.equal(dB.cpu(), db + db0 if acc else db)
        assert torch.equal(dX.cpu(), dx + dx0 if acc else dx)
    X, W, dZ, Zs = (torch.randn(t.shape, generator=g).cuda() for t in (x, w, dz, zs))
    a, b = ([empty((M, K)), empty((K, N)), empty((N,))] for _ in range(2))
    gpu_ctx.matmul_bwd(M, N, K, X, K, W, N, dZ, N, a[0], K, a[1], N, dbias=a[2], act=O.ACT_GELU,
                       Zs=Zs, ldzs=K)
    gpu_ctx.gemm_dw(K, N, M, X, K, dZ, N, b[1], N, colsum=b[2])
    gpu_ctx.gemm_bwd(O.NT, M, K, N, dZ, N, W, N, b[0], K, act=O.ACT_GELU, Zs=Zs, ldzs=K)
    torch.cuda.synchronize()
    for p, q in zip(a, b):
        assert torch.equal(p, q)


# 16-bit tiles on rows of any alignment, as test_gemm_f32_any_rows: K
# remainders of the tile pipeline (1 to 6 tiles of 32 and a tail), rows that end
# between chunks, even and odd leading dimensions, K slices, edges of tiles.
@pytest.mark.parametrize("place", ["plain", "even", "odd", "offset"])
@pytest.mark.parametrize("layout", [O.NN, O.NT, O.TN], ids=["NN", "NT", "TN"])
@pytest.mark.parametrize("dtype", [1, 2], ids=["f16", "bf16"])
def test_gemm_x16_any_rows(gpu_ctx, dtype, layout, place):
    """Small-integer operands (sums exact in fp32 and every fp32 sum below the
    types' first rounding reproduced by one), with NaN around every row (even:
    ld + 2, odd: ld + 3) and the tensors: outputs and column sums bit for bit."""
    torch = _torch()
    dt = [None, torch.float16, torch.bfloat16][dtype]
    gpu_ctx.reserve_workspace(64 << 20)
    g = torch.Generator().manual_seed(13)

    def ints(r, c):
        ld = c + {"even": 2, "odd": 3}.get(place, 0)
        off = 1 if place == "offset" else 64
        v = torch.randint(-3, 4, (r, c), generator=g).to(dt)
        buf = torch.full((off + r * ld + 64,), float("nan"), dtype=dt)
        buf[off:off + r * ld].view(r, ld)[:, :c] = v
        buf = buf.cuda()
        return v.double(), buf[off:], ld

    shapes = [(129, 130, 32 * t + x) for t in range(1, 7) for x in (0, 1, 18)]
    shapes += [(72, 8, 1), (65, 9, 7), (257, 66, 256), (128, 256, 64), (100, 201, 3000),
               (500, 1000, 1500), (600, 2001, 400), (2048, 2050, 300)]
    for M, N, K in shapes:
        note(f"gemm_x16_any_rows {dtype} {layout} {place} {M}x{N}x{K}")
        a, A, lda = ints(*((K, M) if layout == O.TN else (M, K)))
        b, B, ldb = ints(*((N, K) if layout == O.NT else (K, N)))
        old, C, ldc = ints(M, N)
        ref = ((a.T if layout == O.TN else a) @ (b.T if layout == O.NT else b)).to(dt)

        def got():
            torch.cuda.synchronize()
            return C[:M * ldc].view(M, ldc)[:, :N].cpu()

        gpu_ctx.gemm_x16(dtype, layout, M, N, K, A, lda, B, ldb, C, ldc, accumulate=True)
        assert torch.equal(got(), (ref.double() + old).to(dt))
        if layout == O.TN:
            cs, S, _ = ints(1, N)
            gpu_ctx.gemm_dw_x16(dtype, M, N, K, A, lda, B, ldb, C, ldc, colsum=S,
                                colsum_accumulate=True)
            assert torch.equal(got(), ref)
            assert torch.equal(S[:N].cpu(), (cs + b.sum(0)).reshape(-1).to(dt))
        else:
            zs, Zs, ldzs = ints(M, N)
            gpu_ctx.gemm_bwd_x16(dtype, layout, M, N, K, A, lda, B, ldb, C, ldc, act=O.ACT_RELU,
                                 Zs=Zs, ldzs=ldzs)
            assert torch.equal(got(), torch.where(zs > 0, ref, torch.zeros_like(ref)))
            bias, Bi, _ = ints(1, N)
            Z = torch.empty(M, N + 1, dtype=dt, device="cuda")
            gpu_ctx.gemm_x16(dtype, layout, M, N, K, A, lda, B, ldb, C, ldc, bias=Bi,
                             act=O.ACT_RELU, Z=Z, ldz=N + 1)
            z = (ref.double() + bias).to(dt)
            assert torch.equal(got(), z.clamp(min=0))
            assert torch.equal(Z[:, :N].cpu(), z)


@pytest.mark.parametrize("reserved", [0, 64 << 20], ids=["no-workspace", "workspace"])
@pytest.mark.parametrize("dtype", [1, 2], ids=["f16", "bf16"])
def test_gemm_x16_short_k(dtype, reserved):
    """K around the lengths where the 64x64 tiles, the pipelined tiles and their
    K tails take over from each other, each call captured on a context that holds
    no workspace (and must not ask for one then) or enough: small-integer operands,
    outputs and column sums bit for bit."""
    torch = _torch()
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    import ferrograd_amd as fa

    dt = [None, torch.float16, torch.bfloat16][dtype]
    g = torch.Generator().manual_seed(19)
    before = torch.cuda.current_stream()
    ctx, st = fa.torch_context(0)
    try:
        if reserved:
            ctx.reserve_workspace(reserved)
        for M, N in ((100, 99), (16, 1216), (512, 57), (130, 256), (300, 407)):
            for K in (1, 2, 3, 31, 32, 33, 96, 129, 250, 512, 513):
                for layout in (O.NN, O.NT, O.TN):
                    if layout != O.TN and M <= 64:
                        continue  # (few rows: another kernel)
                    note(f"gemm_x16_short_k {dtype} {reserved} {layout} {M}x{N}x{K}")
                    a = torch.randint(-2, 3, (K, M) if layout == O.TN else (M, K), generator=g)
                    b = torch.randint(-2, 3, (N, K) if layout == O.NT else (K, N), generator=g)
                    ref = ((a.T if layout == O.TN else a).double() @
                           (b.T if layout == O.NT else b).double())
                    A, B = a.to(dt).cuda(), b.to(dt).cuda()
                    C = torch.zeros(M, N, dtype=dt, device="cuda")
                    S = torch.zeros(N, dtype=dt, device="cuda")
                    lda, ldb = A.shape[1], B.shape[1]
                    torch.cuda.synchronize()
                    graph = torch.cuda.CUDAGraph()
                    with torch.cuda.graph(graph, stream=st):
                        if layout == O.TN:
                            ctx.gemm_dw_x16(dtype, M, N, K, A, lda, B, ldb, C, N, colsum=S)
                        else:
                            ctx.gemm_x16(dtype, layout, M, N, K, A, lda, B, ldb, C, N)
                    for _ in range(2):
                        C.zero_(), S.zero_()
                        graph.replay()
                        torch.cuda.synchronize()
                        assert torch.equal(C.cpu(), ref.to(dt))
                        if layout == O.TN:
                            assert torch.equal(S.cpu(), b.double().sum(0).to(dt))
    finally:
        torch.cuda.set_stream(before)
        ctx.sync()
        ctx.close()


@pytest.mark.parametrize("dtype", [0, 1, 2], ids=["f32", "f16", "bf16"])
@pytest.mark.parametrize("pad", [0, 1, 2])
def test_bias_grad_any_rows(gpu_ctx, dtype, pad):
    """Column sums of small integers (exact in fp32) over rows of any length and
    alignment, NaN between them: 1 to 63 row splits, columns at the edges of
    the summing workgroups."""
    torch = _torch()
    dt = [torch.float32, torch.float16, torch.bfloat16][dtype]
    g = torch.Generator().manual_seed(17)
    for M, N in [(1, 1), (15, 3), (17, 63), (64, 65), (200, 257), (1000, 130)]:
        ld = N + pad
        v = torch.randint(-3, 4, (M, N), generator=g).to(dt)
        buf = torch.full((M * ld + 9,), float("nan"), dtype=dt)
        buf[pad:pad + M * ld].view(M, ld)[:, :N] = v
        buf = buf.cuda()
        old = torch.randint(-9, 10, (N,), generator=g).to(dt)
        for acc in (False, True):
            out = old.clone().cuda()
            gpu_ctx.bias_grad(M, N, buf[pad:], ld, out, accumulate=acc, dtype=dtype)
            torch.cuda.synchronize()
            ref = v.double().sum(0) + (old.double() if acc else 0.0)
            assert torch.equal(out.cpu(), ref.to(dt)), (M, N, acc)


# --------------------------------------------------------- softmax + CE
def check_softmax_ce(ctx, x, labels, scale=1.0):
    torch = _torch()
    R, C = x.shape
    dx, dl = dev(x), dev(labels.astype(np.uint32).view(np.int32))
    loss, mean, dlog = empty((R,)), empty((1,)), empty((R, C))
    am = empty((R,), torch.int32)
    ctx.softmax_ce(dx, C, dl, R, C, scale, row_loss=loss, mean_loss=mean, dlogits=dlog, ldd=C,
                   argmax=am)
    rl, d, a, m = O.softmax_ce(x, labels.astype(np.uint32), scale)
    assert np.array_equal(host(am).view(np.uint32), a)
    got = host(loss)
    assert np.max(np.abs(got - rl) / np.maximum(np.abs(rl), 1.0)) < 1e-5
    assert normwise_rel(host(dlog), d) < 1e-5
    assert abs(float(host(mean)[0]) - m) <= 1e-5 * max(1.0, abs(m))


def test_softmax_ce_mean_across_paths(gpu_ctx):
    """Calls of changing row counts, on the register path (C % 4 == 0, 256
    and 512 threads), the streaming path (C = 10) and the 16-bit path: each
    mean loss matches the float64 mean of the row losses the same call
    wrote, and a mean requested without row losses (the row losses then go
    to the context's workspace) is the same value."""
    torch = _torch()
    import ferrograd_amd as fa
    rng = np.random.default_rng(5)
    for R, C, dt in [(8192, 1000, None), (3, 10, None), (1, 32000, None), (600, 10, None),
                     (1024, 16, None), (257, 1000, fa.DTYPE_BF16), (2, 64, fa.DTYPE_BF16),
                     (37, 12, fa.DTYPE_BF16), (65, 20000, None)]:
        note(f"softmax_ce mean R={R} C={C} dtype={dt}")
        x = (2 * rng.standard_normal((R, C))).astype(f32)
        lab = rng.integers(0, C, R).astype(np.uint32)
        dl = dev(lab.view(np.int32))
        loss, mean, mean2 = empty((R,)), empty((1,)), empty((1,))
        dx = dev(x) if dt is None else dev(x).to(torch.bfloat16)
        dt = fa.DTYPE_F32 if dt is None else dt
        gpu_ctx.softmax_ce(dx, C, dl, R, C, 1.0, row_loss=loss, mean_loss=mean, dtype=dt)
        gpu_ctx.softmax_ce(dx, C, dl, R, C, 1.0, mean_loss=mean2, dtype=dt)
        rl = host(loss).astype(np.float64)
        m, m2 = float(host(mean)[0]), float(host(mean2)[0])
        assert abs(m - rl.mean()) <= 1e-6 * max(1.0, abs(rl.mean())), (R, C, m, rl.mean())
        assert m2 == m


def test_softmax_ce_fixture(gpu_ctx):
    note("softmax_ce fixture 9x37")
    g = golden("softmax_ce_9x37.npz")
    check_softmax_ce(gpu_ctx, g["x"], g["labels"])


@pytest.mark.parametrize("shape", [(64, 10), (1024, 16), (100, 16), (33, 17), (1024, 64), (1025, 10),
                                   (5, 1), (7, 1024), (2048, 1000),
                                   (256, 32000), (16, 40000), (33, 4100), (5, 8192)],
                         ids=lambda s: "x".join(map(str, s)))
def test_softmax_ce_parity(gpu_ctx, shape):
    R, C = shape
    note(f"softmax_ce R={R} C={C}")
    rng = np.random.default_rng(R * C)
    x = (2 * rng.standard_normal((R, C))).astype(f32)
    x[0, C // 3] = x[0, C // 2] = 50.0   # tie: argmax must be the first
    # Ties 2048 columns apart fall to one thread of a 256- or 512-thread row
    # in different chunks; rows start their chunk walk at different places,
    # so some rows meet the higher column first.  The lowest must still win.
    for r in range(1, min(R, 17)):
        a = 28 + 2048 * (r % 4)
        b = a + 2048 * (1 + r % 6)
        if b < C:
            x[r, a] = x[r, b] = 60.0
    labels = rng.integers(0, C, R)
    check_softmax_ce(gpu_ctx, x, labels, scale=1.0)
    check_softmax_ce(gpu_ctx, x, labels, scale=1.0 / R)


def test_softmax_ce_c3_full_size(gpu_ctx):
    """Config 3 at its real shape: logits [8192, 32000] ~ N(0, 2^2), seed 2."""
    torch = _torch()
    R, C = 8192, 32000
    note("softmax_ce c3 8192x32000")
    x = empty((R, C))
    lab = empty((R,), torch.int32)
    gpu_ctx.rng_normal(2, 0, 0.0, 2.0, x, R * C)
    gpu_ctx.rng_int(2, 1, C, lab, R)
    check_softmax_ce(gpu_ctx, host(x), host(lab).view(np.uint32))


def test_softmax_and_backward(gpu_ctx):
    note("softmax / softmax_bwd")
    # std_wgsl.rs:97-187 closed form: uniform rows of 64 -> 1/64, backward 0.
    x = np.full((16, 64), 5.0, f32)
    y = empty((16, 64))
    gpu_ctx.softmax(dev(x), 16, 64, y)
    yh = host(y)
    assert np.all(yh == f32(1 / 64))
    dx = empty((16, 64))
    gpu_ctx.softmax_bwd(y, dev(np.ones((16, 64), f32)), 16, 64, dx)
    assert np.all(host(dx) == 0.0)
    rng = np.random.default_rng(4)
    for (R, C) in [(33, 1000), (3, 37), (2, 40000)]:
        x = rng.standard_normal((R, C)).astype(f32)
        dy = rng.standard_normal((R, C)).astype(f32)
        y = empty((R, C))
        gpu_ctx.softmax(dev(x), R, C, y)
        assert normwise_rel(host(y), O.softmax(x)) < 1e-5
        dx = empty((R, C))
        gpu_ctx.softmax_bwd(y, dev(dy), R, C, dx)
        assert normwise_rel(host(dx), O.softmax_bwd(host(y), dy)) < 1e-5


# Columns at the edges of the row kernels' capacities: 64 / 128 / 256 / 512 /
# 1024 / 2048 / 4096 / 8192 chunks of 4 (fp32) or 8 (16-bit) elements, and past.
@pytest.mark.parametrize("place", ["aligned", "offset", "out-of-phase", "in-place"])
@pytest.mark.parametrize("dtype", [0, 1, 2], ids=["f32", "f16", "bf16"])
@pytest.mark.parametrize("chunks", [1, 64, 128, 256, 512, 1024, 2048, 4096, 8192, 12000])
def test_softmax_rows_any(gpu_ctx, chunks, dtype, place):
    """softmax + CE and the plain softmax's backward on rows of any length,
    against float64: rows that start anywhere against 16-byte boundaries,
    outputs that start elsewhere than the logits, outputs over the logits; a
    row half -inf, a row of the type's lowest value, ties."""
    torch = _torch()
    E, dt = (4, torch.float32) if dtype == 0 else (8, [None, torch.float16, torch.bfloat16][dtype])
    # Unit of the stored type (round to nearest: half of it), and its least spacing.
    unit = {0: 2.0 ** -24, 1: 2.0 ** -11, 2: 2.0 ** -8}[dtype]
    tiny = {0: 0.0, 1: 2.0 ** -25, 2: 0.0}[dtype]
    off = 0 if place == "aligned" else 1
    for C in (chunks * E - 1, chunks * E, chunks * E + E + 3):
        R = 6 if C > 70 else 1030  # (few short rows take the one-workgroup kernels)
        note(f"softmax_rows_any dtype={dtype} C={C} {place}")
        g = torch.Generator().manual_seed(C)
        x = (2 * torch.randn(R, C, generator=g)).to(dt)
        x[1, : C // 2] = float("-inf")
        x[2, :] = torch.finfo(dt).min
        x[3, C // 3] = x[3, C // 2] = 60.0
        lab = torch.randint(0, C, (R,), generator=g, dtype=torch.int32)
        lab[1] = C - 1
        xd = x.double()
        m = xd.max(1, keepdim=True).values
        e = torch.exp(xd - m)
        s = e.sum(1, keepdim=True)
        p = e / s
        rows = (m + torch.log(s)).squeeze(1) - xd.gather(1, lab.long()[:, None]).squeeze(1)
        ref = p.clone()
        ref[torch.arange(R), lab.long()] -= 1.0
        first = (xd == m).int().argmax(1)

        def put(t, at):  # t in device memory, `at` elements past an aligned start
            b = torch.zeros(t.numel() + 64, dtype=t.dtype, device="cuda")
            b[at:at + t.numel()] = t.reshape(-1).cuda()
            return b, b[at:at + t.numel()]

        _, dx = put(x, off)
        if place == "in-place":
            out = dx
        else:
            _, out = put(torch.zeros_like(x), off + (1 if place == "out-of-phase" else 0))
        dl = lab.cuda()
        loss, am = empty((R,)), empty((R,), torch.int32)
        gpu_ctx.softmax_ce(dx, C, dl, R, C, 1.0, row_loss=loss, dlogits=out, ldd=C, argmax=am,
                           dtype=dtype)
        torch.cuda.synchronize()
        assert torch.equal(am.cpu().long(), first)
        fin = torch.isfinite(rows)
        # The loss is (max + log s) - x_label in fp32: the first sum rounds at
        # the maximum's magnitude.
        bound = 1e-6 * rows.abs().clamp(min=1) + 2.0 ** -23 * m.squeeze(1).abs()
        assert ((loss.cpu().double() - rows).abs() <= bound)[fin].all()
        err = (out.view(R, C).cpu().double() - ref).abs()
        # p in fp32 is off by its exponential's argument rounding: 2.5e-7.
        assert (err <= unit * ref.abs() + tiny + 2.5e-7).all(), float(err.max())
        if place == "in-place":
            continue
        # Plain softmax of the same logits, then its backward.
        _, y = put(torch.zeros_like(x), off + (1 if place == "out-of-phase" else 0))
        gpu_ctx.softmax(dx, R, C, y, dtype=dtype)
        torch.cuda.synchronize()
        yh = y.view(R, C).cpu()
        assert ((yh.double() - p).abs() <= unit * p + tiny + 2.5e-7).all()
        dy = torch.randn(R, C, generator=g).to(dt)
        old = torch.randn(R, C, generator=g).to(dt)
        _, ddy = put(dy, off)
        for acc in (False, True):
            _, gx = put(old, off)
            gpu_ctx.softmax_bwd(y, ddy, R, C, gx, accumulate=acc, dtype=dtype)
            torch.cuda.synchronize()
            yd, dyd = yh.double(), dy.double()
            rb = yd * (dyd - (yd * dyd).sum(1, keepdim=True)) + (old.double() if acc else 0.0)
            # fp32 dot product of terms y * dy (sum of |y| is 1), then one rounding.
            big = dyd.abs().amax(1, keepdim=True)
            e2 = (gx.view(R, C).cpu().double() - rb).abs()
            assert (e2 <= unit * rb.abs() + tiny + 1e-6 * (yd * big + acc)).all(), float(e2.max())


# ------------------------------------------------------------ optimisers
SIZES = [1, 3, 4096, 4097, 100003, 262144]


def make_list(rng, sizes, misalign):
    """Host arrays plus device tensors; misalign shifts every device tensor
    by one float so the 16-byte path is not taken."""
    torch = _torch()
    hs, ds = [], []
    for n in sizes:
        h = rng.standard_normal(n).astype(f32)
        base = torch.empty(n + 1, dtype=torch.float32, device="cuda")
        d = base[1:] if misalign else base[:n]
        d.copy_(torch.from_numpy(h))
        hs.append(h)
        ds.append(d)
    return hs, ds


@pytest.mark.parametrize("misalign", [False, True], ids=["aligned", "misaligned"])
def test_sgd_multi_tensor_bit_exact(gpu_ctx, misalign):
    import ferrograd_amd as fa
    note(f"sgd multi-tensor misalign={misalign}")
    rng = np.random.default_rng(21)
    W, dW = make_list(rng, SIZES, misalign)
    G, dG = make_list(rng, SIZES, misalign)
    mt = fa.MultiTensor(gpu_ctx, dW, dG)
    lr = f32(0.01)
    mt.sgd(float(lr), zero_grad=True)
    for w, g, dw, dg in zip(W, G, dW, dG):
        O.sgd_(w, g, lr, True)
        assert np.array_equal(host(dw), w)
        assert np.all(host(dg) == 0)
    mt.close()


@pytest.mark.parametrize("misalign", [False, True], ids=["aligned", "misaligned"])
def test_adam_multi_tensor_bit_exact_10_steps(gpu_ctx, misalign):
    import ferrograd_amd as fa
    torch = _torch()
    note(f"adam multi-tensor misalign={misalign}")
    rng = np.random.default_rng(22)
    P, dP = make_list(rng, SIZES, misalign)
    G, dG = make_list(rng, SIZES, misalign)
    Mh = [np.zeros_like(p) for p in P]
    Vh = [np.zeros_like(p) for p in P]
    dM = [torch.zeros_like(d) for d in dP]
    dV = [torch.zeros_like(d) for d in dP]
    if misalign:
        dM = [torch.zeros(d.numel() + 1, device="cuda")[1:] for d in dP]
        dV = [torch.zeros(d.numel() + 1, device="cuda")[1:] for d in dP]
    mt = fa.MultiTensor(gpu_ctx, dP, dG, dM, dV)
    b1, b2, eps, lr = f32(0.9), f32(0.999), f32(1e-8), f32(1e-3)
    for step in range(1, 11):
        for h, d in zip(G, dG):
            h[:] = (1e-3 * rng.standard_normal(h.size)).astype(f32)
            d.copy_(torch.from_numpy(h))
        mt.adam(float(lr), float(b1), float(b2), float(eps), step)
        s, r = O.adam_scalars(lr, b1, b2, step)
        for p, g, m, v in zip(P, G, Mh, Vh):
            O.adam_(p, g, m, v, b1, b2, eps, s, r)
    for p, m, v, dp, dm, dv in zip(P, Mh, Vh, dP, dM, dV):
        assert np.array_equal(host(dp), p)
        assert np.array_equal(host(dm), m)
        assert np.array_equal(host(dv), v)
    mt.close()


def test_adam_c4_full_size_sampled(gpu_ctx):
    """Config 4 at its real shape: 64 tensors x 4 Mi parameters, 10 steps
    with fresh N(0, 1e-3^2) grads (device generator), bit-exact against the
    oracle on a sample of 4 tensors."""
    import ferrograd_amd as fa
    torch = _torch()
    note("adam c4 64x4Mi 10 steps (sampled)")
    nt, n = 64, 4 * 1024 * 1024
    P = [empty((n,)) for _ in range(nt)]
    G = [empty((n,)) for _ in range(nt)]
    M = [torch.zeros(n, device="cuda") for _ in range(nt)]
    V = [torch.zeros(n, device="cuda") for _ in range(nt)]
    for i, p in enumerate(P):
        gpu_ctx.rng_normal(3, i, 0.0, 0.02, p, n)
    sample = [0, 21, 42, 63]
    hp = {i: host(P[i]).copy() for i in sample}
    hm = {i: np.zeros(n, f32) for i in sample}
    hv = {i: np.zeros(n, f32) for i in sample}
    mt = fa.MultiTensor(gpu_ctx, P, G, M, V)
    b1, b2, eps, lr = f32(0.9), f32(0.999), f32(1e-8), f32(1e-3)
    for step in range(1, 11):
        for i, g in enumerate(G):
            gpu_ctx.rng_normal(3, 1000 * step + i, 0.0, 1e-3, g, n)
        hg = {i: host(G[i]) for i in sample}
        mt.adam(float(lr), float(b1), float(b2), float(eps), step)
        s, r = O.adam_scalars(lr, b1, b2, step)
        for i in sample:
            O.adam_(hp[i], hg[i], hm[i], hv[i], b1, b2, eps, s, r)
    for i in sample:
        assert np.array_equal(host(P[i]), hp[i]), i
        assert np.array_equal(host(M[i]), hm[i]), i
        assert np.array_equal(host(V[i]), hv[i]), i
    mt.close()


def test_device_rng_matches_host(gpu_ctx):
    import ferrograd_amd as fa
    torch = _torch()
    note("device rng vs host rng")
    n = 100000
    x = empty((n,))
    gpu_ctx.rng_uniform(9, 4, -1.0, 1.0, x, n)
    assert np.array_equal(host(x), fa.rng_uniform(9, 4, (n,), -1.0, 1.0))
    k = empty((n,), torch.int32)
    gpu_ctx.rng_int(9, 5, 1000, k, n)
    assert np.array_equal(host(k).view(np.uint32), fa.rng_int(9, 5, (n,), 1000))
    gpu_ctx.rng_normal(9, 6, 0.0, 1.0, x, n)
    # Box-Muller in double: device and host libm may differ in the last
    # double ulp, which almost never survives rounding to fp32.
    hx = fa.rng_normal(9, 6, (n,))
    assert np.mean(host(x) == hx) > 0.999
    assert np.max(np.abs(host(x) - hx)) < 1e-5


def test_softmax_row_sum_order(gpu_ctx):
    """A one-wave row's sum (fp32, 1024 columns) adds its chunks' sums, not one
    long chain a lane: with 256 columns at the maximum and the rest 15.5 below
    it (1.9e-7 each, under half a unit of a lane's first four), a chain loses
    all of the rest.  Chunk sums and the six steps are exact but for units of
    the small ones; the three sums added to the first, 1 / s and the product
    round by half a unit each.  And the label's gradient is the rounded
    probability less one."""
    torch = _torch()
    R, C = 6, 1024
    x = torch.full((R, C), -15.5)
    x[:, :256] = 0.0
    x[3:] += 2.0
    y, d, loss = empty((R, C)), empty((R, C)), empty((R,))
    lab = torch.arange(0, 32 * R, 32, dtype=torch.int32)
    xd = x.cuda()
    gpu_ctx.softmax(xd, R, C, y)
    gpu_ctx.softmax_ce(xd, C, lab.cuda(), R, C, 1.0, row_loss=loss, dlogits=d, ldd=C)
    torch.cuda.synchronize()
    p = torch.softmax(x.double(), 1)
    assert ((y.cpu().double() - p).abs() <= 5 * 2.0 ** -24 * p)[:, :256].all()
    cols = lab.long()[:, None]
    assert torch.equal(d.cpu().gather(1, cols), y.cpu().gather(1, cols) - 1.0)


@pytest.mark.parametrize("C,active", [(2048, 1024), (32768, 8192), (131072, 8192)])
@pytest.mark.parametrize("dtype", [1, 2], ids=["f16", "bf16"])
def test_softmax_exponential_16bit(gpu_ctx, dtype, C, active):
    """The fp32 row loss of 16-bit rows shows the exponential's own error: one
    logit 0, `active` of -D, the rest -inf, so that all sums but a few are exact and
    the loss is log(1 + active exp(-D)), for 64 D around 8.  In units of 2^-24: 1.5
    for the exponential, half a unit for each of at most 3 sums and of the loss, 2
    for the logarithm."""
    torch = _torch()
    dt = [None, torch.float16, torch.bfloat16][dtype]
    D = (torch.arange(64) / 32 + 7).to(dt)
    x = torch.full((64, C), float("-inf"), dtype=dt)
    x[:, :active] = -D[:, None]
    x[:, C - 5] = 0.0
    lab = torch.full((64,), C - 5, dtype=torch.int32).cuda()
    loss, d = empty((64,)), torch.empty(64, C, dtype=dt, device="cuda")
    gpu_ctx.softmax_ce(x.cuda(), C, lab, 64, C, 1.0, row_loss=loss, dlogits=d, ldd=C, dtype=dtype)
    torch.cuda.synchronize()
    ref = torch.log1p(active * torch.exp(-D.double()))
    err = (loss.cpu().double() - ref).abs().max().item() * 2.0 ** 24
    assert err <= 5.5, err


def test_softmax_bf16_subnormal(gpu_ctx):
    """Probabilities under 2^-126 keep bf16's subnormal values: within one unit of
    them (the fp32 value rounds once before)."""
    torch = _torch()
    x = torch.full((64, 2048), -88.0, dtype=torch.bfloat16)
    x -= torch.arange(64, dtype=torch.bfloat16)[:, None] / 16
    x[:, 7] = 0.0
    y = torch.empty(64, 2048, dtype=torch.bfloat16, device="cuda")
    gpu_ctx.softmax(x.cuda(), 64, 2048, y, dtype=2)
    torch.cuda.synchronize()
    p = torch.softmax(x.double(), 1)
    assert p[:, 0].min() > 2.0 ** -133 and p[:, 0].max() < 2.0 ** -126
    assert ((y.cpu().double() - p).abs() <= 2.0 ** -133)[:, 8:].all()
