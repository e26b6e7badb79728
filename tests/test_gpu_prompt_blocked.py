"""Prompt sizes on token-blocked codes (tq_act_quant_blocked, tq_gemm_mixed_blocked).

The whole-list kernel forms the row-major prefill kernels' sums: bitwise equal
outputs.  The split kernel adds W wave partials: outputs within the oracle's
tolerance (2 bf16 ulp + the fp32 accumulation bound, oracle.numerics), and its
INT32 tile products equal to the oracle's bit for bit.
"""
from __future__ import annotations

from types import SimpleNamespace

import numpy as np
import pytest
import torch

from helpers import assert_gemm_close, complement, make_w, make_x, oracle_pack, uniform_fp16_ids, values
from oracle import native as onat
from oracle import numerics as nm
from tilequant_amd.gemm_rows_splitk_64x64 import gemm_mixed_rows_blocked, gemm_mixed_rows_splitk, prefill_plan
from tilequant_amd.mixed_linear import MixedLinear, MixedLinearGroup
from tilequant_amd.pack import pack_weight_from_tile_ids
from tilequant_amd.quant_utils import quantize_activation_tile_absmax
from tilequant_amd.quantize_activation import quantize_activation_blocked

pytestmark = pytest.mark.gpu
CFG = SimpleNamespace(quant_style="gi", dtype_out="bf16")
SPLIT_TOKENS, SPLIT_LONG_TOKENS, SPLIT_LONG_TILES = 384, 1280, 96   # the schedule's limits (tq_prefill.hip)


def _pack(m, k, ids16, seed, dtype=torch.bfloat16, layout="mfma"):
    W = make_w(m, k, seed=seed, dtype=dtype)
    n_tr, n_tc = -(-m // 64), k // 64
    return W, pack_weight_from_tile_ids(
        W, n_tr=n_tr, n_tc=n_tc, int8_tile_ids=torch.from_numpy(complement(ids16, n_tr * n_tc)),
        fp16_tile_ids=torch.from_numpy(np.asarray(ids16, np.int64)), cfg=CFG, tile_layout=layout)


def _ids(m, k, frac, seed):
    n_tr, n_tc = -(-m // 64), k // 64
    return uniform_fp16_ids(n_tr, n_tc, frac, seed=seed) if frac > 0 else np.zeros(0, np.int64)


def _kw(p, out_dtype, bias=None):
    return dict(int8_tiles=p.int8_tiles, int8_scales=p.int8_scales, int8_tile_ids=p.int8_tile_ids,
                int8_row_ptr=p.int8_row_ptr, fp16_tiles=p.fp16_tiles, fp16_tile_ids=p.fp16_tile_ids,
                fp16_row_ptr=p.fp16_row_ptr, M=p.M_orig, K=p.K_orig, n_tr=p.n_tr, n_tc=p.n_tc, out_dtype=out_dtype,
                bias=bias, tile_layout=p.tile_layout)


def _blocked(codes):
    n, k = codes.shape
    nb = -(-n // 16)
    padded = np.zeros((16 * nb, k), np.int8)
    padded[:n] = codes
    return padded.reshape(nb, 16, k // 64, 4, 16).transpose(2, 0, 3, 1, 4).reshape(-1)


@pytest.mark.parametrize("n", [1, 64, 65, 127, 128, 129, 256, 257, 500, 512, 513, 769])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_blocked_quantizer_matches_the_oracle(n, dtype):
    x = make_x(n, 192, seed=n, dtype=dtype)
    x[:, 64:128] = 0                                   # an all-zero column tile: scale 1, codes 0
    wide = torch.zeros((n, 256), dtype=dtype, device="cuda")
    wide[:, :192] = x.cuda()
    q, s = quantize_activation_blocked(wide[:, :192])   # a row stride of its own
    q_ref, s_ref = nm.act_quant(values(x), dtype == torch.bfloat16)
    assert np.array_equal(q.cpu().numpy(), _blocked(q_ref))
    assert np.array_equal(s.cpu().numpy().view(np.uint32), np.asarray(s_ref, np.float32).view(np.uint32))


@pytest.mark.parametrize("n,m,k,frac,dtype,layout,heavy", [
    (385, 64, 64, 0.0, torch.bfloat16, "mfma", False),         # one tile
    (400, 200, 640, 0.2, torch.bfloat16, "mfma", False),       # ragged last row tile, four row tiles
    (449, 320, 192, 1.0, torch.float16, "row_major", False),   # no INT8 tile at all
    (513, 704, 4160, 0.3, torch.bfloat16, "mfma", True),       # 65 column tiles: two windows, an odd count
    (1000, 8192, 320, 0.1, torch.bfloat16, "row_major", True),
    (2049, 16384, 128, 0.1, torch.float16, "mfma", False),     # 128-token workgroups
    (2100, 16384, 192, 0.2, torch.bfloat16, "mfma", False),    # the last one with 52 tokens: half of its blocks
    (2052, 16384, 256, 0.1, torch.bfloat16, "mfma", True),     # a short last one beside row tiles in 16 bits
    (1281, 192, 8192, 0.1, torch.bfloat16, "mfma", False),     # long lists past the split limit
    (1300, 128, 19456, 0.05, torch.bfloat16, "mfma", False),   # the most column tiles it takes
])
def test_whole_list_kernel_is_bitwise_the_row_major_kernel(n, m, k, frac, dtype, layout, heavy):
    ids16 = _ids(m, k, frac, seed=n)
    if heavy:                                          # a row tile entirely in 16 bits, and a column of them
        n_tc = k // 64
        ids16 = np.union1d(ids16, np.r_[n_tc:2 * n_tc, np.arange(-(-m // 64)) * n_tc + 3])
    _, p = _pack(m, k, ids16, seed=m + k, dtype=dtype, layout=layout)
    x = make_x(n, k, seed=n + 1, dtype=dtype).cuda()
    xq, sx = quantize_activation_tile_absmax(x)
    xb, sb = quantize_activation_blocked(x)
    assert torch.equal(sb, sx)
    order = torch.randperm(p.n_tr + 3, generator=torch.Generator().manual_seed(n)).to(torch.int32)
    order[order >= p.n_tr] = -1                        # empty slots
    order = order.cuda()
    for out_dtype, biased in ((torch.bfloat16, False), (torch.float16, True)):
        bias = (torch.randn(m, generator=torch.Generator().manual_seed(n)) * 0.5).to(out_dtype).cuda() if biased else None
        kw = _kw(p, out_dtype, bias)
        ref = gemm_mixed_rows_splitk(x_fp=x, x_int8=xq, sx=sx, **kw)
        wide = torch.full((n, m + 3), 5.0, dtype=out_dtype, device="cuda")   # rows that forbid 16-byte stores
        gemm_mixed_rows_blocked(x_fp=x, x_blocked=xb, sx=sb, out=wide[:, :m], **kw)
        assert torch.equal(wide[:, :m], ref) and torch.all(wide[:, m:] == 5)
        y = gemm_mixed_rows_blocked(x_fp=x, x_blocked=xb, sx=sb, row_order=order, **kw)
        assert torch.equal(y, ref)


@pytest.mark.parametrize("n,m,k,frac,layout", [
    (65, 64, 64, 0.0, "mfma"), (65, 200, 640, 0.3, "row_major"), (128, 512, 3072, 0.05, "mfma"),
    (384, 320, 320, 0.5, "mfma"), (100, 256, 19456, 0.1, "mfma"), (257, 192, 8192, 0.2, "mfma"),
    (1280, 64, 6144, 0.1, "mfma"), (300, 128, 512, 1.0, "mfma"),
    # more than 128 row tiles x 64-token blocks: whole row tiles per workgroup
    (65, 4160, 192, 0.4, "mfma"), (384, 1500, 256, 0.3, "row_major"), (200, 3072, 6144, 0.02, "mfma")])
def test_split_kernel_products_and_outputs(n, m, k, frac, layout):
    assert n <= (SPLIT_LONG_TOKENS if k // 64 >= SPLIT_LONG_TILES else SPLIT_TOKENS)
    ids16 = _ids(m, k, frac, seed=n)
    W, p = _pack(m, k, ids16, seed=m + k, layout=layout)
    op = oracle_pack(W, ids16)
    x = make_x(n, k, seed=n + 2)
    xd = x.cuda()
    xb, sx = quantize_activation_blocked(xd)
    q_ref, s_ref = nm.act_quant(values(x))
    bias = (torch.randn(m, generator=torch.Generator().manual_seed(n)) * 0.5).to(torch.bfloat16)
    kw = dict(x_fp=xd, x_blocked=xb, sx=sx, **_kw(p, torch.bfloat16, bias.cuda()))
    y = gemm_mixed_rows_blocked(**kw)
    assert torch.equal(gemm_mixed_rows_blocked(**kw), y)
    T8 = int(p.int8_tiles.shape[0])
    rows = np.unique(np.r_[0:4, n // 2, n - 4:n])
    if T8:
        prod = torch.full((T8, n, 64), -2**31, dtype=torch.int32, device="cuda")
        assert torch.equal(gemm_mixed_rows_blocked(**kw, _products=(prod, 0, n)), y)
        ref = onat.tile_products_i32(q_ref[rows], op.int8_tiles, op.int8_tile_ids, p.n_tc, K=k)
        assert np.array_equal(prod[:, torch.from_numpy(rows).cuda()].cpu().numpy(), ref)
        assert int((prod == -2**31).sum()) == 0
    w16 = nm.bf16_bits_to_f32(op.fp16_tiles)
    _, acc, sab = onat.gemm_mixed(q_ref[rows], s_ref, values(x[rows]), op.int8_tiles, op.int8_scales, op.int8_tile_ids,
                                  op.int8_row_ptr, w16, op.fp16_tile_ids, op.fp16_row_ptr, p.n_tr, p.n_tc, m, k,
                                  want_f64=True)
    assert_gemm_close(y[torch.from_numpy(rows).cuda()], acc, sab, p.n_tc, bias=values(bias))


@pytest.mark.parametrize("n,m,k", [(600, 320, 640), (2100, 16384, 128)])
def test_whole_list_kernel_products(n, m, k):
    """INT32 products of both token-block sizes, on rows of the first and last workgroups."""
    ids16 = _ids(m, k, 0.2, seed=n)
    W, p = _pack(m, k, ids16, seed=m + k)
    op = oracle_pack(W, ids16)
    x = make_x(n, k, seed=n + 2)
    xb, sx = quantize_activation_blocked(x.cuda())
    kw = dict(x_fp=x.cuda(), x_blocked=xb, sx=sx, **_kw(p, torch.bfloat16))
    y = gemm_mixed_rows_blocked(**kw)
    q_ref, _ = nm.act_quant(values(x))
    for r0, cnt in ((0, 40), (n - 20, 20)):
        prod = torch.full((int(p.int8_tiles.shape[0]), cnt, 64), -2**31, dtype=torch.int32, device="cuda")
        assert torch.equal(gemm_mixed_rows_blocked(**kw, _products=(prod, r0, cnt)), y)
        ref = onat.tile_products_i32(q_ref[r0:r0 + cnt], op.int8_tiles, op.int8_tile_ids, p.n_tc, K=k)
        assert np.array_equal(prod.cpu().numpy(), ref)


@pytest.mark.parametrize("n", [65, 300, 400, 1500])
def test_mixed_linear_prompts_group_capture_and_plan(n):
    """Through MixedLinear: a stacked group equals its members bitwise, a
    captured call replays to the eager result, and a work plan (a row tile all
    in 16 bits) changes nothing."""
    mods = []
    for i, m in enumerate((640, 128, 128)):
        ids16 = np.union1d(_ids(m, 3072, 0.05, seed=i), np.arange(48, 96))
        mods.append(MixedLinear(_pack(m, 3072, ids16, seed=i)[1], None, CFG))
    plan = prefill_plan(int8_tile_ids=mods[0].int8_tile_ids, int8_row_ptr=mods[0].int8_row_ptr,
                        fp16_row_ptr=mods[0].fp16_row_ptr, n_tr=mods[0].n_tr, n_tc=48)
    assert plan.row_order[:4].tolist() == [1, -1, -1, -1]            # the 16-bit row tile has a workgroup of its own
    assert sorted(plan.row_order.tolist())[3:] == list(range(10))
    x = make_x(n, 3072, seed=n).cuda()
    group = MixedLinearGroup(mods)
    with torch.inference_mode():
        stacked, parts = group.output_for(x, 0), [m(x) for m in mods]
        assert torch.equal(stacked, torch.cat(parts, dim=1))
        s = torch.cuda.Stream()
        s.wait_stream(torch.cuda.current_stream())
        with torch.cuda.stream(s):
            group.linear(x)
        torch.cuda.synchronize()
        g = torch.cuda.CUDAGraph()
        with torch.cuda.graph(g, stream=s):
            y = group.linear(x)
        for _ in range(3):
            x.add_(0)                                  # eager work between the replays
            g.replay()
            torch.cuda.synchronize()
            assert torch.equal(y, stacked)


def test_mixed_linear_prompt_descriptors_follow_their_module():
    """Cached prompt descriptors: siblings share one quantization under
    inference mode, in-place bias and input updates are seen, a replaced weight
    is used, and a module still copies."""
    import copy

    _, p = _pack(256, 320, _ids(256, 320, 0.1, seed=1), seed=1)
    x = make_x(700, 320, seed=3).cuda()
    lin = MixedLinear(p, torch.ones(256, device="cuda", dtype=torch.float16), CFG)   # a bias of another dtype
    plain = lambda mod, v: gemm_mixed_rows_splitk(   # noqa: E731
        x_fp=v, x_int8=quantize_activation_tile_absmax(v)[0], sx=quantize_activation_tile_absmax(v)[1],
        **_kw(mod.to_pack(), torch.bfloat16, mod.bias.to(torch.bfloat16)))
    twin = copy.deepcopy(lin)
    with torch.inference_mode():
        assert torch.equal(lin(x), plain(lin, x)) and torch.equal(twin(x), plain(lin, x))
        lin.bias.mul_(3)
        assert torch.equal(lin(x), plain(lin, x))
    y = x.clone()
    assert torch.equal(lin(y), plain(lin, y))
    y.mul_(0.5)
    assert torch.equal(lin(y), plain(lin, y))
    assert torch.equal(lin(y.view(7, 100, 320)).view(700, 256), plain(lin, y))
    other = copy.deepcopy(lin)
    for name in ("int8_tiles", "int8_scales", "fp16_tiles"):
        setattr(other, name, getattr(other, name) * 2 if name != "int8_tiles" else getattr(other, name).clone())
    assert torch.equal(other(y), plain(other, y)) and not torch.equal(other(y), lin(y))
    wide = torch.zeros((700, 384), device="cuda", dtype=torch.bfloat16)
    wide[:, :320] = y                                  # not contiguous: copied first, as before
    assert torch.equal(lin(wide[:, :320]), plain(lin, y))


def test_blocked_gemm_refuses_what_it_cannot_take():
    _, p = _pack(128, 128, np.zeros(0, np.int64), seed=1)
    x = make_x(65, 128, seed=2).cuda()
    xb, sx = quantize_activation_blocked(x)
    kw = _kw(p, torch.bfloat16)
    with pytest.raises(ValueError):
        gemm_mixed_rows_blocked(x_fp=x[:64], x_blocked=xb, sx=sx, **kw)
    with pytest.raises(ValueError):
        gemm_mixed_rows_blocked(x_fp=x, x_blocked=xb[:-1], sx=sx, **kw)
    with pytest.raises(ValueError):
        gemm_mixed_rows_blocked(x_fp=x, x_blocked=xb, sx=sx, **dict(kw, K=100))
    with pytest.raises(ValueError):
        gemm_mixed_rows_blocked(x_fp=x, x_blocked=xb, sx=sx, row_order=torch.arange(3).cuda(), **kw)
    with pytest.raises(ValueError):
        quantize_activation_blocked(x[:, :100])
