"""Sibling projections that share one activation's codes, on the GPU: every
output is that of a module that quantizes for itself."""
from __future__ import annotations

from types import SimpleNamespace

import pytest
import torch

from helpers import complement, make_w, make_x, uniform_fp16_ids
from tilequant_amd.mixed_linear import MixedLinear, MixedLinearGroup
from tilequant_amd.pack import pack_weight_from_tile_ids

pytestmark = pytest.mark.gpu
CFG = SimpleNamespace(quant_style="gi", dtype_out="bf16")
K = 640
SIZES = [40, 100, 600]      # the two-launch path, one and two quantizer launches of the prompt path


def _siblings(count=2, m=192):
    mods = []
    for seed in range(count):
        ids16 = uniform_fp16_ids(m // 64, K // 64, 0.1, seed=seed)
        ids8 = complement(ids16, (m // 64) * (K // 64))
        mods.append(MixedLinear(pack_weight_from_tile_ids(
            make_w(m, K, seed=seed), n_tr=m // 64, n_tc=K // 64, int8_tile_ids=torch.from_numpy(ids8),
            fp16_tile_ids=torch.from_numpy(ids16), cfg=CFG), None, CFG))
    return mods


def _alone(lin, x):
    with torch.no_grad():              # nothing is shared outside inference mode
        return lin(x.clone())


@pytest.mark.parametrize("n", SIZES)
def test_in_place_changes_of_inference_tensors_are_seen(n):
    a, b = _siblings()
    with torch.inference_mode():
        x = make_x(n, K, seed=n).cuda()
        a(x)
        x.mul_(-0.5)
        y = b(x)
    assert torch.equal(y, _alone(b, x))
