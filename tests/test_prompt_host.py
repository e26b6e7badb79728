"""Host logic of the prompt GEMM (no GPU): the slot order of a weight's row tiles."""
from __future__ import annotations

import os
import re
import struct
import subprocess
from pathlib import Path
from types import SimpleNamespace

import numpy as np
import pytest
import torch

from tilequant_amd import _native as nat


def _slots(counts, n_tc):
    rp = np.concatenate(([0], np.cumsum(counts))).astype(np.int32)
    out = np.full(len(counts) + 3, 77, np.int32)
    n = nat.load().tq_gemm_row_order(rp.ctypes.data, len(counts), n_tc, out.ctypes.data, out.size)
    return out[:n].tolist(), out[n:].tolist()


@pytest.mark.parametrize("seed", range(6))
def test_row_order_covers_every_row_tile_and_groups_the_heavy_ones(seed):
    rng = np.random.default_rng(seed)
    n_tr, n_tc = int(rng.integers(1, 60)), int(rng.integers(1, 80))
    counts = rng.integers(0, max(1, n_tc // 2), n_tr)
    counts[rng.random(n_tr) < 0.1 * seed] = n_tc
    slots, rest = _slots(counts, n_tc)
    heavy = [r for r in range(n_tr) if 3 * counts[r] >= 2 * n_tc]
    whole = -(-len(heavy) // 4) * 4
    assert len(slots) == n_tr + whole - len(heavy) and set(rest) <= {77}
    assert sorted(s for s in slots if s >= 0) == list(range(n_tr))
    assert sorted(s for s in slots[:whole] if s >= 0) == heavy and all(s >= 0 for s in slots[whole:])
    ordered = [counts[s] for s in slots if s >= 0]
    assert ordered == sorted(ordered, reverse=True)


def test_row_order_rejects_bad_arguments():
    lib = nat.load()
    rp, out = np.zeros(5, np.int32), np.zeros(7, np.int32)
    assert lib.tq_gemm_row_order(None, 4, 4, out.ctypes.data, 7) == -1
    assert lib.tq_gemm_row_order(rp.ctypes.data, 4, 4, out.ctypes.data, 6) == -1
    assert lib.tq_gemm_row_order(rp.ctypes.data, 0, 4, out.ctypes.data, 7) == -1


def test_prompt_entries_reject_bad_arguments_before_any_launch():
    lib = nat.load()
    assert lib.tq_act_quant_blocked(None, 64, 0, 0, 64, None, None, None, 0, None) == -1
    assert lib.tq_act_quant_blocked(1 << 20, 100, 0, 4, 100, 1 << 20, 1 << 20, None, 0, None) == -1
    assert lib.tq_act_quant_blocked(1 << 20, 68, 0, 100, 64, 1 << 20, 1 << 20, None, 0, None) == -3
    assert lib.tq_act_quant_blocked(1 << 20, 64, 0, 600, 64, 1 << 20, 1 << 20, None, 0, None) == -4
    fake = 1 << 20
    args = [fake, fake, fake, fake, fake, fake, fake, 128, 0, None, None, None, fake, 64, 0, None, 100, 64, 128, 1, 2, 1,
            None, 0, None, 0, 0, None]
    for at, value, code in ((16, -1, -1), (18, 100, -1), (8, 7, -2), (21, 5, -2), (13, 60, -1), (0, fake + 8, -3),
                            (2, fake + 4, -3), (5, None, -1)):
        bad = list(args)
        bad[at] = value
        assert lib.tq_gemm_mixed_blocked(*bad) == code, (at, value)
    assert lib.tq_gemm_mixed_blocked(*[fake if i == 22 else a for i, a in enumerate(args)]) == -1   # no slots
    assert lib.tq_prompt_forward(None) == -1


def _blocked_kernel_listings(tmp_path):
    """{symbol: instructions} of the whole-list prompt kernels in the library
    built from this tree (its gfx950 code objects, listed by llvm-objdump)."""
    llvm = Path(os.environ.get("ROCM_PATH", "/opt/rocm")) / "llvm" / "bin"
    fat = tmp_path / "fatbin"
    subprocess.run([llvm / "llvm-objcopy", f"--dump-section=.hip_fatbin={fat}", nat.LIB_PATH, tmp_path / "rest"],
                   check=True)
    data, magic, listings = fat.read_bytes(), b"__CLANG_OFFLOAD_BUNDLE__", {}
    for found in re.finditer(magic, data):
        base, at = found.start(), found.end()
        (entries,) = struct.unpack_from("<Q", data, at)
        at += 8
        for _ in range(entries):
            offset, size, id_len = struct.unpack_from("<QQQ", data, at)
            at += 24 + id_len
            code = data[base + offset:base + offset + size]
            if b"gfx950" not in data[at - id_len:at] or b"gemm_prefill_blocked_kernel" not in code:
                continue
            obj = tmp_path / "code.o"
            obj.write_bytes(code)
            text = subprocess.run([llvm / "llvm-objdump", "-d", "--no-show-raw-insn", obj], check=True,
                                  capture_output=True, text=True).stdout
            for part in re.split(r"\n(?=[0-9a-f]+ <[^>]+>:\n)", text):
                head = re.match(r"([0-9a-f]+) <([^>]+)>:\n", part)
                if head and "gemm_prefill_blocked_kernel" in head[2]:
                    ins = re.findall(r"^\s+([a-z]\w+.*?)\s*//\s*([0-9A-F]+):", part, flags=re.M)
                    listings[head[2]] = [(int(addr, 16), text) for text, addr in ins]
    return listings


@pytest.mark.skipif(not Path("/opt/rocm/llvm/bin/llvm-objdump").exists(), reason="no llvm-objdump")
def test_ring_slices_land_before_the_first_barrier_publishes_them(tmp_path):
    """The whole-list kernel's waves fill each LDS ring stage together, so a
    wave's own loads of the first two slices must have landed before its first
    ring barrier.  In the built code: after the prologue's 6 XL LDS loads (XL
    per slice), the waits before that barrier leave in flight no more than the
    vector memory operations issued after the first 2 XL."""
    listings = _blocked_kernel_listings(tmp_path)
    assert len(listings) == 6            # bf16 and fp16 x 64 and 128 tokens, and the bf16 dumps
    for name, ins in listings.items():
        xl = 2 if "ELi4E" in name else 1
        index = {addr: i for i, (addr, _) in enumerate(ins)}
        vmem = [bool(re.match(r"(global|buffer|flat)_", text)) for _, text in ins]
        loads = [i for i, v in enumerate(vmem) if v]
        bodies = 0
        for first in range(len(loads)):
            run = loads[first:first + 6 * xl + 1]
            lds = ["_lds_" in ins[i][1] for i in run]
            if first and "_lds_" in ins[loads[first - 1]][1] or lds != [True] * (6 * xl) + [False]:
                continue
            bodies += 1
            i, since, landed, hops = run[2 * xl - 1] + 1, 0, False, 0
            while not ins[i][1].startswith("s_barrier"):
                text = ins[i][1]
                since += vmem[i]
                wait = re.match(r"s_waitcnt.*vmcnt\((\d+)\)", text)
                landed = landed or bool(wait) and int(wait[1]) <= since
                jump = re.match(r"s_branch (\S+)", text)
                i += 1
                if jump:
                    hops += 1
                    assert hops < 20, name
                    i = index[ins[i - 1][0] + 4 + 4 * ((int(jump[1], 0) + 0x8000) % 0x10000 - 0x8000)]
            assert landed, f"{name}: the first ring barrier is passed with {since} later operations and no wait"
        assert bodies >= 3, name         # 1, 2 or 4 token blocks, and the 16-bit-heavy row tiles


def test_modules_saved_whole_before_prompt_descriptors_still_load():
    """A module object pickled by a version without prompt descriptors and slot
    orders lacks both in its state."""
    import pickle

    from test_host_logic import _cpu_pack

    from tilequant_amd.gemm_rows_splitk_64x64 import PrefillPlan
    from tilequant_amd.mixed_linear import MixedLinear

    lin = MixedLinear(_cpu_pack(128, 192, 0.3, 1)[0], None, SimpleNamespace(dtype_out="bf16"))
    state = dict(lin.__dict__, _launches={})
    del state["_prompts"]
    old = MixedLinear.__new__(MixedLinear)
    old.__setstate__(state)
    assert old._prompts == {} and torch.equal(old.int8_tiles, lin.int8_tiles)
    again = pickle.loads(pickle.dumps(old))
    assert again._prompts == {} and again._launches == {}
    units = torch.arange(3, dtype=torch.int32)
    plan = PrefillPlan.__new__(PrefillPlan)
    plan.__setstate__((None, {"units": units, "n_first": 1, "n_tr": 3}))
    assert plan.units is units and (plan.n_first, plan.n_tr, plan.row_order) == (1, 3, None)
    plan = pickle.loads(pickle.dumps(PrefillPlan(units, 2, 3, row_order=units)))
    assert (plan.n_first, plan.row_order.tolist()) == (2, [0, 1, 2])


@pytest.mark.parametrize("heavy,n16,rest", [([5], 33, 2), (list(range(28)), 48, 0), (list(range(0, 48, 2)), 48, 0)])
def test_plans_order_heavy_row_tiles_that_split_no_pair(heavy, n16, rest):
    """Row tiles mostly in 16 bits get slots of their own also where the pair
    plan of the row-major kernel splits nothing (48 x 48 tiles: one row tile
    with 33 in 16 bits among others with 2, the first 28 all in 16 bits, every
    second one)."""
    from test_host_logic import _plan_from_ids16

    plan = _plan_from_ids16(np.concatenate([r * 48 + np.arange(n16 if r in heavy else rest) for r in range(48)]), 48, 48)
    assert plan.units is None and plan.n_tr == 48
    slots = plan.row_order.tolist()
    whole = -(-len(heavy) // 4) * 4
    assert slots[:whole] == heavy + [-1] * (whole - len(heavy))
    assert slots[whole:] == [r for r in range(48) if r not in heavy]
