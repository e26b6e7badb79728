"""Prompt sizes on token-blocked codes at their edges: row chunks and unaligned
inputs beside whole aligned ones, NaN and infinities, one row tile mostly in 16
bits among light ones in the split kernel."""
from __future__ import annotations

from types import SimpleNamespace

import numpy as np
import pytest
import torch

from helpers import assert_gemm_close, complement, make_w, make_x, oracle_pack, uniform_fp16_ids, values
from oracle import native as onat
from oracle import numerics as nm
from tilequant_amd.gemm_rows_splitk_64x64 import gemm_mixed_rows_blocked, gemm_mixed_rows_splitk
from tilequant_amd.mixed_linear import MixedLinear
from tilequant_amd.pack import pack_weight_from_tile_ids
from tilequant_amd.quant_utils import quantize_activation_tile_absmax
from tilequant_amd.quantize_activation import quantize_activation_blocked

pytestmark = pytest.mark.gpu


def _cfg(**extra):
    return SimpleNamespace(quant_style="gi", dtype_out="bf16", **extra)


def _pack(m, k, ids16, seed):
    W = make_w(m, k, seed=seed)
    n_tr, n_tc = -(-m // 64), k // 64
    return W, pack_weight_from_tile_ids(
        W, n_tr=n_tr, n_tc=n_tc, int8_tile_ids=torch.from_numpy(complement(ids16, n_tr * n_tc)),
        fp16_tile_ids=torch.from_numpy(np.asarray(ids16, np.int64)), cfg=_cfg())


def _kw(p):
    return dict(int8_tiles=p.int8_tiles, int8_scales=p.int8_scales, int8_tile_ids=p.int8_tile_ids,
                int8_row_ptr=p.int8_row_ptr, fp16_tiles=p.fp16_tiles, fp16_tile_ids=p.fp16_tile_ids,
                fp16_row_ptr=p.fp16_row_ptr, M=p.M_orig, K=p.K_orig, n_tr=p.n_tr, n_tc=p.n_tc,
                out_dtype=torch.bfloat16, tile_layout=p.tile_layout)


def _check(y, W, p, ids16, x, rows):
    """Rows of ``y`` against the oracle on the scales of the whole input."""
    op = oracle_pack(W, ids16)
    q, s = nm.act_quant(values(x))
    _, acc, sab = onat.gemm_mixed(q[rows], s, values(x[rows]), op.int8_tiles, op.int8_scales, op.int8_tile_ids,
                                  op.int8_row_ptr, nm.bf16_bits_to_f32(op.fp16_tiles), op.fp16_tile_ids,
                                  op.fp16_row_ptr, p.n_tr, p.n_tc, p.M_orig, p.K_orig, want_f64=True)
    assert_gemm_close(y[torch.from_numpy(rows).cuda()], acc, sab, p.n_tc)


@pytest.mark.parametrize("n,k,chunk,bitwise", [
    (1500, 640, 512, True),        # whole lists in both, no chunk of 64 rows or fewer: the same sums
    (1400, 6144, 700, True),       # the same past the long lists' split limit
    (300, 640, 100, False),        # split lists as a whole, row-major kernels in chunks
    (1050, 640, 500, False),       # a last chunk of 50 rows runs the decode kernels
    (1000, 6144, 600, False)])
def test_row_chunks_and_unaligned_inputs(n, k, chunk, bitwise):
    """A chunked input and one whose rows are not 16-byte aligned have the
    scales and codes of the whole aligned input and its outputs bit for bit
    where the same sums are formed; elsewhere the partial sums differ, each
    result within the oracle's bound."""
    m = 320
    ids16 = uniform_fp16_ids(m // 64, k // 64, 0.1, seed=n)
    W, p = _pack(m, k, ids16, seed=n)
    x = make_x(n, k, seed=n)
    x[n - 2:, :64] *= 40                       # the last chunk holds the first tile's absmax
    xd = x.cuda()
    whole = MixedLinear(p, None, _cfg())(xd)
    parts = MixedLinear(p, None, _cfg(activation_row_chunk_size=chunk))(xd)
    shifted = torch.empty(n * k + 1, dtype=x.dtype, device="cuda")[1:].view(n, k).copy_(xd)
    assert shifted.data_ptr() % 16
    moved = MixedLinear(p, None, _cfg())(shifted)
    rows = np.unique(np.r_[0:3, chunk - 1:chunk + 2, n - 3:n])
    for y in (whole, parts, moved):
        _check(y, W, p, ids16, x, rows)
    if bitwise:
        assert torch.equal(parts, whole) and torch.equal(moved, whole)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("n", [65, 129, 257, 512, 513])
def test_quantizer_on_nan_and_infinities(n, dtype):
    """Column tiles with a NaN, an infinity, both, nothing but infinities, the
    type's lowest value: codes and scales of the row-major quantizer, bit for
    bit."""
    x = make_x(n, 384, seed=n, dtype=dtype)
    x[n // 2, 3] = float("nan")
    x[n - 1, 70] = float("inf")
    x[0, 130], x[n - 1, 131] = float("nan"), float("-inf")
    x[:, 192:256] = float("-inf")
    x[:, 256:320] = torch.finfo(dtype).min
    xd = x.cuda()
    ref_q, ref_s = quantize_activation_tile_absmax(xd)
    q, s = quantize_activation_blocked(xd)
    nb = -(-n // 16)
    rows = q.view(6, nb, 4, 16, 16).permute(1, 3, 0, 2, 4).reshape(16 * nb, 384)
    assert torch.equal(rows[:n], ref_q) and not rows[n:].any()
    assert torch.equal(s.view(torch.int32), ref_s.view(torch.int32))


@pytest.mark.parametrize("n", [100, 400, 2100])
def test_gemm_on_nan_and_infinities(n):
    """Non-finite activations through the split (100 rows) and whole-list
    kernels: NaN and infinities exactly where the row-major kernel has them --
    one token's where the weight holds the column in 16 bits, every token's
    where in INT8 (the scale is theirs too).  Finite outputs: the same bits
    from whole lists; from split lists a bf16 rounding (2^-7) and the fp32
    error of K = 256 products on each side apart."""
    m, k = (16384, 256) if n == 2100 else (192, 256)     # 2100 rows: 128-token workgroups
    n_tr, n_tc = m // 64, k // 64
    ids16 = np.r_[1, 2, 3, n_tc + 2]                     # row tile 0: columns 1..3, row tile 1: column 2
    W, p = _pack(m, k, ids16, seed=n)
    x = make_x(n, k, seed=n)
    x[7, 70], x[n - 1, 140], x[n // 2, 200] = float("inf"), float("nan"), float("-inf")
    for cols in (slice(0, 0), slice(64, 128), slice(128, 192)):
        xd = x.clone()
        xd[:, cols] = 0                                  # without column 1's or 2's: more row tiles stay finite
        xd = xd.cuda()
        xq, sx = quantize_activation_tile_absmax(xd)
        ref = gemm_mixed_rows_splitk(x_fp=xd, x_int8=xq, sx=sx, **_kw(p))
        xb, sb = quantize_activation_blocked(xd)
        y = gemm_mixed_rows_blocked(x_fp=xd, x_blocked=xb, sx=sb, **_kw(p))
        assert torch.equal(y.isnan(), ref.isnan()) and torch.equal(y.isinf(), ref.isinf())
        assert ref.isnan().any() and ref[:, :64].isfinite().any()
        keep = ref.isfinite()
        if n > 384:
            assert torch.equal(y[keep], ref[keep]) and torch.equal(y[ref.isinf()], ref[ref.isinf()])
        else:
            half_code = sx.nan_to_num(0, 0, 0).repeat_interleave(64).double() / 2    # |code * scale| <= |value| + half a step
            sab = (xd.nan_to_num(0, 0, 0).abs().double() + half_code) @ (W.cuda().abs().double().T + W.abs().max().item() / 254)
            bound = ref.double().abs() * 2 ** -7 + 2 * k * 2 ** -24 * sab
            assert bool(((y.double() - ref.double()).abs() <= bound)[keep].all())


@pytest.mark.parametrize("n,m,k", [(65, 320, 640), (128, 512, 3072), (384, 1472, 320), (100, 256, 8192),
                                   (1280, 192, 6144)])
def test_split_kernel_with_one_heavy_row_tile(n, m, k):
    """One row tile all in 16 bits and one with two thirds of its tiles in 16
    bits among light ones, as clustered masks give (half and whole row tiles,
    4 and 8 waves)."""
    n_tr, n_tc = m // 64, k // 64
    ids16 = np.unique(np.r_[uniform_fp16_ids(n_tr, n_tc, 0.02, seed=n), np.arange(n_tc, 2 * n_tc),
                            (n_tr - 1) * n_tc + np.arange(0, n_tc, 3), (n_tr - 1) * n_tc + np.arange(1, n_tc, 3)])
    W, p = _pack(m, k, ids16, seed=n)
    x = make_x(n, k, seed=n + 1)
    xd = x.cuda()
    xb, sx = quantize_activation_blocked(xd)
    y = gemm_mixed_rows_blocked(x_fp=xd, x_blocked=xb, sx=sx, **_kw(p))
    assert torch.equal(y, gemm_mixed_rows_blocked(x_fp=xd, x_blocked=xb, sx=sx, **_kw(p)))
    _check(y, W, p, ids16, x, np.unique(np.r_[0:4, n // 2, n - 4:n]))
