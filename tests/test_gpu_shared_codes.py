"""Sibling projections that share one activation's codes, on the GPU: every
output is that of a module that quantizes for itself."""
from __future__ import annotations

from types import SimpleNamespace

import pytest
import torch

from helpers import complement, make_w, make_x, uniform_fp16_ids
from tilequant_amd import _native as nat
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


def _capture(fn, stream):
    g = torch.cuda.CUDAGraph()
    torch.cuda.synchronize()
    with torch.cuda.graph(g, stream=stream):
        out = fn()
    return g, out


@pytest.mark.parametrize("n", SIZES)
@pytest.mark.parametrize("grouped", [False, True])
def test_captures_and_eager_calls_do_not_serve_each_other(n, grouped):
    """Two siblings on one stream and one input: the first eager and the second
    captured, each in a graph of its own, the first captured and the second
    eager.  The input is refilled before every replay."""
    mods = _siblings()
    if grouped:
        group = MixedLinearGroup(mods)
        bounds = group.bounds
        call = lambda i, x: group.output_for(x, i)[:, bounds[i][0]:bounds[i][1]]   # noqa: E731
    else:
        call = lambda i, x: mods[i](x)   # noqa: E731
    x = make_x(n, K, seed=n).cuda()
    s = torch.cuda.Stream()
    s.wait_stream(torch.cuda.current_stream())
    with torch.inference_mode(), torch.cuda.stream(s):
        for m in mods:
            m(x.clone())                       # plans and workspaces before the captures
        if grouped:
            group.linear(x.clone())
        call(0, x)                             # eager, then its sibling captured
        graphs = [_capture(lambda: call(1, x), s)]
        graphs.append(_capture(lambda: call(0, x), s))
        assert torch.equal(call(1, x), _alone(mods[1], x))   # captured, then its sibling eager
        graphs.append(_capture(lambda: call(0, x), s))       # ... and two graphs one after the other
        graphs.append(_capture(lambda: call(1, x), s))
        for rep in range(3):
            x.copy_(make_x(n, K, seed=100 * n + rep))
            want = [_alone(m, x) for m in mods]
            for which, (g, y) in zip((1, 0, 0, 1), graphs):
                g.replay()
                torch.cuda.synchronize()
                assert torch.equal(y, want[which]), (rep, which)


@pytest.mark.parametrize("n", SIZES)
def test_siblings_of_one_capture_share_and_replay(n):
    a, b = _siblings()
    x = make_x(n, K, seed=n).cuda()
    s = torch.cuda.Stream()
    s.wait_stream(torch.cuda.current_stream())
    with torch.inference_mode(), torch.cuda.stream(s):
        a(x.clone()), b(x.clone())
        g, (ya, yb) = _capture(lambda: (a(x), b(x)), s)
        for rep in range(3):
            x.copy_(make_x(n, K, seed=100 * n + rep))
            want = _alone(a, x), _alone(b, x)
            g.replay()
            torch.cuda.synchronize()
            assert torch.equal(ya, want[0]) and torch.equal(yb, want[1])


def test_capture_ids():
    s, side = torch.cuda.Stream(), torch.cuda.Stream()
    x = torch.zeros(64, device="cuda")
    seen = []

    def body():
        seen.append(nat.capture_id(s.cuda_stream))
        side.wait_stream(s)
        seen.append(nat.capture_id(side.cuda_stream))
        x.add_(1)
        s.wait_stream(side)

    assert nat.capture_id(s.cuda_stream) == 0 and nat.capture_id(0) == 0
    graphs = [_capture(body, s) for _ in range(2)]
    assert nat.capture_id(s.cuda_stream) == 0
    assert seen[0] == seen[1] and seen[2] == seen[3] and 0 < seen[0] != seen[2] > 0
    del graphs
