"""The wave-split kernel (FFK_LATENCY convs, the FC head from a few faces on)
at the edges of its tiles and of its launch rules, bit for bit against the
oracle."""
import ctypes as C

import numpy as np
import pytest

import fastface_amd as fa
import gpu_util
from gpu_util import params_block, run_conv, run_fc
from test_gpu_kernels import F32, _pair_desc, _special_params, rng

pytestmark = pytest.mark.gpu

# (cin, cout, k, stride, H, batch, workgroups): every tile, from one short row
# tile to the last grid it takes, ragged last row tiles, one K step up to 72
CASES = [
    (512, 512, 3, 1, 7, 1, 4 * 16), (512, 512, 3, 1, 7, 5, 16 * 16),                       # 16x32
    (64, 128, 1, 1, 28, 1, 49 * 4), (256, 512, 1, 1, 7, 5, 16 * 16),
    (256, 256, 3, 1, 14, 5, 31 * 8), (64, 64, 3, 2, 112, 1, 98 * 2),                       # 32x32
    (256, 256, 3, 1, 14, 8, 49 * 4), (64, 128, 3, 1, 56, 1, 98 * 2), (256, 256, 3, 2, 28, 10, 62 * 4),   # 32x64
    (256, 256, 3, 1, 14, 11, 45 * 4), (512, 512, 3, 2, 14, 31, 32 * 8),                    # 48x64
    (256, 256, 3, 2, 28, 17, 53 * 4), (512, 512, 3, 1, 7, 41, 32 * 8),                     # 64x64
]

# the K-group patch kernel's tiles past those, at the first and last batch
# each one takes (64x64, 128x64, then 128x128), also as one of two halves
SH = fa.FFK_SHARED_GPU
PATCH_CASES = [
    (256, 256, 3, 1, 14, 16, 49 * 4, 0), (256, 256, 3, 1, 14, 20, 62 * 4, 0),
    (256, 256, 3, 1, 14, 21, 33 * 4, 0), (256, 256, 3, 1, 14, 41, 63 * 4, 0), (256, 256, 3, 1, 14, 42, 65 * 2, 0),
    (256, 256, 3, 1, 14, 20, 31 * 4, SH), (256, 256, 3, 1, 14, 10, 31 * 4, SH),
    (256, 512, 3, 1, 14, 8, 25 * 8, 0), (256, 512, 3, 1, 14, 10, 31 * 8, 0),
    (256, 512, 3, 1, 14, 11, 17 * 8, 0), (256, 512, 3, 1, 14, 20, 31 * 8, 0),
    (128, 128, 3, 1, 28, 11, 68 * 2, 0), (128, 128, 3, 1, 28, 20, 123 * 2, 0), (128, 128, 3, 1, 28, 21, 129, 0),
    (128, 256, 3, 1, 28, 6, 37 * 4, 0), (128, 256, 3, 1, 28, 10, 62 * 4, 0),
    (512, 512, 3, 1, 7, 42, 17 * 8, 0), (512, 512, 3, 1, 7, 83, 32 * 8, 0),
]


def _desc(cin, cout, k, s, H, B, flags):
    d = fa.ffk_conv_desc()
    d.batch, d.cin, d.cout, d.kh, d.kw, d.stride, d.pad, d.hin, d.win = B, cin, cout, k, k, s, k // 2, H, H
    d.flags = flags
    return C.byref(d)


@pytest.mark.parametrize("mode", ["raw", "all", "bn_only", "inscale"])
@pytest.mark.parametrize("cin,cout,k,s,H,B,grid", CASES)
def test_wavek_conv(gpu_lib, oracle, cin, cout, k, s, H, B, grid, mode):
    _check_conv(gpu_lib, oracle, cin, cout, k, s, H, B, grid, mode, fa.FFK_LATENCY, b"wavek")


@pytest.mark.parametrize("mode", ["raw", "all"])
@pytest.mark.parametrize("cin,cout,k,s,H,B,grid,shared", PATCH_CASES)
def test_latency_patch_tiles(gpu_lib, oracle, cin, cout, k, s, H, B, grid, shared, mode):
    _check_conv(gpu_lib, oracle, cin, cout, k, s, H, B, grid, mode, fa.FFK_LATENCY | shared, b"patch_kg")


def _check_conv(lib, oracle, cin, cout, k, s, H, B, grid, mode, L, kind):
    assert lib.ffk_conv_variant(_desc(cin, cout, k, s, H, B, L)) == kind
    assert lib.ffk_conv_grid(_desc(cin, cout, k, s, H, B, L)) == grid
    assert lib.ffk_conv_workspace_bytes(_desc(cin, cout, k, s, H, B, L)) == 0
    r = rng(3100 + cin + cout + k + H + B)
    x = r.integers(-128, 128, size=(B, H, H, cin), dtype=np.int8)
    w = r.integers(-128, 128, size=(cout, cin, k, k), dtype=np.int8)
    x[0] = -128                                        # the largest sums
    w[-1] = -128
    acc = oracle.conv_i32(x, w, s, k // 2)
    if mode == "raw":
        assert np.array_equal(run_conv(lib, x, w, s, k // 2, raw=True, split=False, flags=L), acc)
        return
    ws, bias, inv = _special_params(r, cout)           # ties, NaN, infinities, denormals
    if mode == "inscale":
        got, _ = run_conv(lib, x, w, s, k // 2, params=params_block(cout, ws=ws, bias=bias, inv=inv), split=False,
                          flags=fa.FFK_EPI_BIAS | fa.FFK_EPI_INSCALE | L, in_scale=0.0173)
        assert np.array_equal(got, oracle.fused_epilogue(acc, ws=ws, bias=bias, in_scale=0.0173, inv_pc=inv))
        return
    ho = acc.shape[1]
    slope = r.uniform(0, 1.5, cout).astype(F32)
    adds = r.uniform(1e-3, 5e-2, cout).astype(F32)
    add = r.integers(-128, 128, size=acc.shape, dtype=np.int8)
    bsin = r.uniform(1e-3, 5e-2, cout).astype(F32)
    bns = r.uniform(0.5, 1.5, cout).astype(F32)
    bno = r.normal(0, 0.05, cout).astype(F32)
    binv = (1.0 / r.uniform(0.01, 0.1, cout)).astype(F32)
    P = params_block(cout, ws=ws, bias=bias, inv=inv, slope=slope, adds=adds, bn_sin=bsin, bn_s=bns, bn_o=bno,
                     bn_inv=binv)
    flags = fa.FFK_EPI_BIAS | fa.FFK_EPI_PRELU | fa.FFK_EPI_ADD | fa.FFK_EPI_BN | L
    exp = oracle.fused_epilogue(acc, ws=ws, bias=bias, prelu=slope, add_src=add, add_scale_pc=adds, inv_pc=inv)
    exp_bn = oracle.bn_prelu_requant(exp, in_scale_pc=bsin, bn_scale=bns, bn_offset=bno, inv_pc=binv)
    for x_even in ([False, True] if mode == "all" and ho % 2 == 0 else [False]):
        got, got_bn = run_conv(lib, x, w, s, k // 2, params=P, flags=flags, add=add, want_x=mode == "all",
                               want_bn=True, split=False, x_even=x_even)
        if mode == "all":
            assert np.array_equal(got, exp[:, ::2, ::2] if x_even else exp)
        assert np.array_equal(got_bn, exp_bn)


# batches at the ends of every tile and K split of the rule, with the
# workspace the call asks for and without one (whole K, from 5 faces); past
# 704 faces the call's own workspace is the 128x128 GEMM's
@pytest.mark.parametrize("B", [3, 4, 5, 16, 17, 64, 65, 128, 129, 256, 257, 512, 513, 704, 1024])
@pytest.mark.parametrize("split", [True, False])
def test_wavek_fc(gpu_lib, oracle, B, split):
    r = rng(3200 + B)
    K, N = 25088, 512
    a = r.integers(-128, 128, size=(B, K), dtype=np.int8)
    W = r.integers(-127, 128, size=(N, K), dtype=np.int8)
    a[0] = -128
    W[-1] = -127
    ws = r.uniform(1e-7, 1e-5, N).astype(F32)
    bias = r.normal(0, 0.05, N).astype(F32)
    kernel = (b"gemm" if B > 704 else b"wavek") if split else b"matvec" if B < 5 else b"wavek"
    got = run_fc(gpu_lib, a, W, ws, bias, a_scale=0.37, split=split, kernel=kernel)
    for b in sorted({0, B // 2, B - 1}):
        assert np.array_equal(got[b], oracle.fc(a[b], W, ws, bias, 0.37)), b


@pytest.mark.parametrize("B,K,N,split", [(12, 64, 12, False), (7, 192, 500, True), (33, 4096, 512, True), (70, 1024, 40, True),
                                         (3, 64, 600, True), (3, 24640, 20, True), (17, 33024, 64, False), (9, 128, 20000, False)])
def test_wavek_fc_other_heads(gpu_lib, oracle, B, K, N, split):
    """Heads of other sizes: fewer K steps than waves, columns past N."""
    r = rng(3300 + B)
    a = r.integers(-128, 128, size=(B, K), dtype=np.int8)
    W = r.integers(-128, 128, size=(N, K), dtype=np.int8)
    ws = r.uniform(1e-7, 1e-5, N).astype(F32)
    bias = r.normal(0, 0.05, N).astype(F32)
    got = run_fc(gpu_lib, a, W, ws, bias, split=split, kernel=b"wavek")
    for b in range(B):
        assert np.array_equal(got[b], oracle.fc(a[b], W, ws, bias)), b


@pytest.mark.parametrize("via_io", [False, True])
@pytest.mark.parametrize("skew", [1, 2, 3])
def test_wavek_fc_at_any_float(gpu_lib, oracle, skew, via_io):
    """Scales, biases and outputs at addresses aligned to one float only."""
    r = rng(3320 + skew)
    B, K, N = 40, 1024, 72
    a = r.integers(-128, 128, size=(B, K), dtype=np.int8)
    W = r.integers(-128, 128, size=(N, K), dtype=np.int8)
    ws = r.uniform(1e-7, 1e-5, N).astype(F32)
    bias = r.normal(0, 0.05, N).astype(F32)
    got = run_fc(gpu_lib, a, W, ws, bias, kernel=b"wavek", via_io=via_io, skew=skew)
    assert np.array_equal(got, np.stack([oracle.fc(a[b], W, ws, bias) for b in range(B)]))


@pytest.mark.parametrize("B,N,kernel", [(5, 4194368, b"matvec"), (65, 46340 * 64, b"wavek")])
def test_fc_wide_heads(gpu_lib, oracle, B, N, kernel):
    """Millions of outputs: the widest grid of two row tiles whose block
    indices divide exactly, and a head past it, which the matvec runs."""
    K = 64
    d = fa.ffk_fc_desc()
    d.batch, d.n, d.k = B, N, K
    assert gpu_lib.ffk_fc_variant(C.byref(d)) == kernel
    r = rng(3350 + B)
    a = r.integers(-128, 128, size=(B, K), dtype=np.int8)
    W = r.integers(-128, 128, size=(N, K), dtype=np.int8)
    ws = r.uniform(1e-7, 1e-5, N).astype(F32)
    bias = r.normal(0, 0.05, N).astype(F32)
    got = run_fc(gpu_lib, a, W, ws, bias)
    for b in sorted({0, min(B, 64) - 1, B - 1}):
        assert np.array_equal(got[b], oracle.fc(a[b], W, ws, bias)), b


# (cin, cout, H, shortcut's cin, batch): a stride-2 conv and its shortcut as
# one launch, on every tile it takes, ragged last row tiles, one to four
# shortcut steps, the first conv's steps a multiple of the waves or not
PAIRS = [(64, 64, 112, 64, 1), (128, 128, 56, 64, 1), (128, 128, 56, 64, 2), (256, 256, 28, 128, 1), (256, 256, 28, 128, 7),
         (256, 256, 28, 128, 13), (512, 512, 14, 256, 1), (512, 512, 14, 256, 9), (512, 512, 14, 256, 31)]


@pytest.mark.parametrize("form", ["x_bn", "x", "bn", "x_even"])
@pytest.mark.parametrize("cin,cout,H,cx,B", PAIRS)
def test_wavek_pair_equals_two_launches(gpu_lib, cin, cout, H, cx, B, form):
    lib, L = gpu_lib, fa.FFK_LATENCY
    Ho = H // 2
    if form == "x_even" and Ho % 2:
        pytest.skip("odd output image")
    r = rng(3400 + cin + H + B)
    x = r.integers(-128, 128, size=(B, H, H, cin), dtype=np.int8)
    w = r.integers(-128, 128, size=(cout, cin, 3, 3), dtype=np.int8)
    xc = r.integers(-128, 128, size=(B, Ho, Ho, cx), dtype=np.int8)
    w2 = r.integers(-128, 128, size=(cout, cx, 1, 1), dtype=np.int8)
    x[0] = -128
    w[-1] = -128
    ws, bias, inv = _special_params(r, cout)
    P1 = params_block(cout, ws=ws, bias=bias, inv=inv)
    ws2, bias2, inv2 = _special_params(r, cout)
    P2 = params_block(cout, ws=ws2, bias=bias2, inv=inv2, adds=r.uniform(1e-3, 5e-2, cout).astype(F32),
                      bn_sin=r.uniform(1e-3, 5e-2, cout).astype(F32), bn_s=r.uniform(0.5, 1.5, cout).astype(F32),
                      bn_o=r.normal(0, 0.05, cout).astype(F32), bn_inv=(1.0 / r.uniform(0.01, 0.1, cout)).astype(F32))
    want_bn = form != "x"
    f1 = fa.FFK_EPI_BIAS
    f2 = fa.FFK_EPI_BIAS | fa.FFK_EPI_ADD | (fa.FFK_EPI_BN if want_bn else 0)
    R, _ = run_conv(lib, x, w, 2, 1, params=P1, flags=f1, split=False)
    X_exp, BN_exp = run_conv(lib, xc, w2, 1, 0, params=P2, flags=f2, add=R, want_bn=want_bn, split=False)

    keep = []
    n = B * Ho * Ho * cout
    dR, dX, dBN = (gpu_util.Dev(lib, host=np.full(n, 0x5A, np.uint8)) for _ in range(3))
    keep += [dR, dX, dBN]
    c = _pair_desc(lib, keep, B, cin, cout, 3, 2, 1, H, x, w, P1, f1 | L, dR.ptr)
    sc = _pair_desc(lib, keep, B, cx, cout, 1, 1, 0, Ho, xc, w2, P2,
                    f2 | L | (fa.FFK_OUT_X_EVEN if form == "x_even" else 0), None if form == "bn" else dX.ptr,
                    out_bn=dBN.ptr if want_bn else None, add=dR.ptr)
    assert lib.ffk_conv_s2_shortcut(C.byref(c), C.byref(sc), None) == 1
    gpu_util.check(lib, lib.ffk_stream_sync(None))
    X = dX.get(np.int8, (n,))
    if form == "x_even":
        ne = n // 4
        assert np.array_equal(X[:ne].reshape(B, Ho // 2, Ho // 2, cout), X_exp[:, ::2, ::2])
        assert (X[ne:].view(np.uint8) == 0x5A).all()
    elif form != "bn":
        assert np.array_equal(X.reshape(X_exp.shape), X_exp)
    if want_bn:
        assert np.array_equal(dBN.get(np.int8, BN_exp.shape), BN_exp)
