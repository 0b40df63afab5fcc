"""The generic conv's epilogue at the edges of its vector widths: channel
counts of every divisibility, tensors at odd addresses, both tile widths, bit
for bit against the oracle."""
import ctypes as C

import numpy as np
import pytest

import fastface_amd as fa
from gpu_util import Dev, check, make_bn_lut, pack_conv, params_block
from test_gpu_kernels import F32, _special_params, rng

pytestmark = pytest.mark.gpu


# (cin, cout, k, pad, H, B): 16-, 8-, 4- and 1-byte channel runs and outputs,
# tiles of 64 and 128 channels with ragged last blocks, 64 and 128 pixels
@pytest.mark.parametrize("cin,cout,k,pad,H,B", [
    (32, 16, 3, 1, 9, 2), (32, 80, 3, 1, 9, 2), (16, 136, 1, 0, 12, 3), (24, 104, 3, 1, 10, 2), (48, 36, 3, 1, 9, 2),
    (20, 100, 3, 1, 9, 2), (7, 5, 3, 1, 10, 2), (16, 131, 3, 1, 8, 2), (32, 128, 1, 0, 60, 10), (48, 60, 3, 1, 58, 12),
    # small grids with 12 K steps or more (the wave-split tiles): steps that
    # span taps and steps of one tap, one and two column halves, ragged ends
    (80, 64, 3, 1, 9, 3), (48, 100, 5, 2, 11, 2), (16, 72, 7, 3, 8, 1), (128, 36, 3, 1, 9, 2), (192, 260, 3, 0, 9, 2),
    (112, 128, 3, 1, 37, 11)])
@pytest.mark.parametrize("offsets", [(0, 0, 0), (8, 8, 8), (16, 4, 0), (0, 16, 1), (3, 0, 16)])
def test_generic_epilogue_vector_widths(gpu_lib, oracle, cin, cout, k, pad, H, B, offsets):
    _check(gpu_lib, oracle, cin, cout, k, pad, H, B, offsets)


# the same shapes' small grids with the BN tables at addresses that allow 8-,
# 4- and 1-byte accesses only
@pytest.mark.parametrize("cin,cout,k,pad,H,B", [(80, 64, 3, 1, 9, 3), (128, 36, 3, 1, 9, 2), (48, 100, 5, 2, 11, 2),
                                                (32, 80, 3, 1, 9, 2)])
@pytest.mark.parametrize("lut_offset", [8, 4, 1])
def test_generic_bn_table_at_any_address(gpu_lib, oracle, cin, cout, k, pad, H, B, lut_offset):
    _check(gpu_lib, oracle, cin, cout, k, pad, H, B, (0, 0, 0), lut_offset)


# X at its even pixels only, beside BN at all of them, for every vector width,
# 64- and 128-row tiles and the register-staged operands
@pytest.mark.parametrize("cin,cout,k,pad,H,B", [(32, 33, 3, 1, 10, 2), (16, 131, 1, 0, 12, 3), (24, 36, 3, 1, 10, 2),
                                                (32, 136, 3, 1, 12, 2), (16, 67, 1, 0, 58, 12), (7, 5, 3, 1, 10, 2)])
@pytest.mark.parametrize("offsets", [(0, 0, 0), (3, 4, 1)])
def test_generic_x_even(gpu_lib, oracle, cin, cout, k, pad, H, B, offsets):
    _check(gpu_lib, oracle, cin, cout, k, pad, H, B, offsets, x_even=True)


def _check(lib, oracle, cin, cout, k, pad, H, B, offsets, lut_offset=0, x_even=False):
    r = rng(4100 + cin + cout * 3 + H)
    ho = H + 2 * pad - k + 1
    x = r.integers(-128, 128, size=(B, H, H, cin), dtype=np.int8)
    w = r.integers(-128, 128, size=(cout, cin, k, k), dtype=np.int8)
    if cout >= 6:
        ws, bias, inv = _special_params(r, cout)
    else:
        ws, bias, inv = (r.uniform(1e-3, 1e-2, cout).astype(F32) for _ in range(3))
    slope = r.uniform(0, 1.5, cout).astype(F32)
    adds, bsin = (r.uniform(1e-3, 5e-2, cout).astype(F32) for _ in range(2))
    add = r.integers(-128, 128, size=(B, ho, ho, cout), dtype=np.int8)
    bns = r.uniform(0.5, 1.5, cout).astype(F32)
    bno = r.normal(0, 0.05, cout).astype(F32)
    binv = (1.0 / r.uniform(0.01, 0.1, cout)).astype(F32)
    P = params_block(cout, ws=ws, bias=bias, inv=inv, slope=slope, adds=adds, bn_sin=bsin, bn_s=bns, bn_o=bno, bn_inv=binv)
    n = add.size
    # outputs and residual at the given offsets, guard bytes around the outputs
    guard = np.full(n + 64, 0x5a, np.int8)
    res = np.concatenate([np.zeros(offsets[2], np.int8), add.reshape(-1)])
    dx, dw, dp = Dev(lib, host=x), Dev(lib, host=pack_conv(lib, w)), Dev(lib, host=P)
    lut = np.concatenate([np.zeros(lut_offset, np.int8), make_bn_lut(lib, P).reshape(-1)])
    dl, da = Dev(lib, host=lut), Dev(lib, host=res)
    do, db = Dev(lib, host=guard), Dev(lib, host=guard)
    d = fa.ffk_conv_desc()
    d.batch, d.cin, d.cout, d.kh, d.kw, d.stride, d.pad, d.hin, d.win = B, cin, cout, k, k, 1, pad, H, H
    d.in_, d.w, d.params, d.bn_lut = dx.ptr, dw.ptr, dp.ptr, dl.ptr + lut_offset
    d.add_src, d.out, d.out_bn = da.ptr + offsets[2], do.ptr + offsets[0], db.ptr + offsets[1]
    d.flags = fa.FFK_EPI_BIAS | fa.FFK_EPI_PRELU | fa.FFK_EPI_ADD | fa.FFK_EPI_BN
    if x_even:
        d.flags |= fa.FFK_OUT_X_EVEN
    assert lib.ffk_conv_variant(C.byref(d)) == b"generic"
    check(lib, lib.ffk_conv(C.byref(d), None))
    check(lib, lib.ffk_stream_sync(None))
    exp = oracle.fused_epilogue(oracle.conv_i32(x, w, 1, pad), ws=ws, bias=bias, prelu=slope, add_src=add,
                                add_scale_pc=adds, inv_pc=inv)
    exp_bn = oracle.bn_prelu_requant(exp, in_scale_pc=bsin, bn_scale=bns, bn_offset=bno, inv_pc=binv)
    for dev, off, e in ((do, offsets[0], exp[:, ::2, ::2] if x_even else exp), (db, offsets[1], exp_bn)):
        got = dev.get(np.int8, (n + 64,))
        assert np.array_equal(got[off:off + e.size].reshape(e.shape), e)
        assert (got[:off] == 0x5a).all() and (got[off + e.size:] == 0x5a).all()
