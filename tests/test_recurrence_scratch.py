"""Scratch memory of the recurrent layers: asked for only by steps that use it, and set aside when the caches are sized."""
import re
import shutil
import struct
import subprocess

import pytest
import torch
import torch.nn as nn

from nanovllm_amd import _lib, ops
from nanovllm_amd.engine.cache_spec import PagedKVSpec, SlotStateSpec
from nanovllm_amd.engine.model_runner import ModelRunner
from nanovllm_amd.layers.delta_rule import GatedDeltaRule
from nanovllm_amd.layers.gated_memory import GatedWriteMemory
from nanovllm_amd.layers.general_delta import GeneralDeltaRule

H, D = 4, 128


class _Model(nn.Module):
    def __init__(self):
        super().__init__()
        self.rules = nn.ModuleList([GatedDeltaRule(H, H, D, D, 1e-5), GeneralDeltaRule(H, D, 1e-5), GatedWriteMemory(H, D, D, 1e-5),
                                    GatedDeltaRule(H, H, 40, D, 1e-5)])

    def cache_specs(self):
        return [PagedKVSpec(2, 64, 64)] + [SlotStateSpec({"state": ((H, D, D), torch.float32)})] * 3

    def bind_caches(self, caches):
        pass


@pytest.mark.parametrize("rows", [0, 1, 5000])
def test_caches_leave_room_for_the_scratch_of_the_largest_step(monkeypatch, rows):
    runner = ModelRunner(_Model(), None, 16, 3, device="cpu", num_state_slots=6, max_num_batched_tokens=rows)
    free, total = 3 << 30, 4 << 30
    monkeypatch.setattr(torch.cuda, "mem_get_info", lambda device: (free, total))
    need = [_lib.mixers().nv_recurrence_workspace_bytes(form, rows, H, D, D, 6, 0, _lib.DTYPE_BF16) for form in range(3)]
    assert (min(need) > 0) == (rows > 0)
    left = int(total * 0.9) - (total - free) - 3 * 6 * H * D * D * 4 - max(need)
    assert runner._spec_blocks_that_fit(0.9) == left // (16 * 2 * 128 * 2)


def test_sizes_without_a_launch_in_chunks_need_none():
    assert _Model().rules[3].step_scratch_bytes(5000, 6, torch.bfloat16) == 0


@pytest.mark.parametrize("max_rows,lead,portions", [(1, 0, 7), (0, 3, 7), (0, 1, 1), (0, 0, 0)])
def test_single_tokens_allocate_nothing(max_rows, lead, portions):
    """All sequences of one row each, known as such by any of the step's three hints."""
    assert ops._portions(None, 0, None, 3, H, D, D, 3, max_rows, lead, portions)[2] is None


def _need(form, T, seqs, lead=0, heads=16, d=D):
    return _lib.mixers().nv_recurrence_workspace_bytes(form, T, heads, d, d, seqs, lead, _lib.DTYPE_BF16)


def _bytes(form, tokens, T, seqs, heads=16, d=D):
    """Records of `tokens` tokens with their rows of V, read-outs and flags of a step."""
    words = (1 if form == 2 else 2) * tokens * d + (2 if form == 1 else 1) * tokens * d + d
    words += {8: (384, 384, 64), 16: (512, 1024, 256)}[tokens][form]
    records = (T + (tokens - 1) * seqs) // tokens + 1
    return heads * (records * (words * 4 + tokens * d * 2 + 4) + T * d * 4)


@pytest.mark.parametrize("form", range(3))
@pytest.mark.parametrize("seqs,rows", [(256, 2), (256, 5), (8, 17), (64, 24)])
def test_short_portions_take_small_records(form, seqs, rows):
    """A record of 16 tokens for a portion of a few is twice the memory and, for many of them, up to 1.6 times the time."""
    assert _need(form, seqs * rows, seqs) == _bytes(form, 8, seqs * rows, seqs)
    assert _need(form, seqs * rows + 7, seqs + 7, 7) == _bytes(form, 8, seqs * rows + 7, seqs)        # single tokens in front


@pytest.mark.parametrize("form,seqs,rows,tokens", [(0, 4, 191, 8), (0, 4, 192, 16), (0, 16, 255, 8), (0, 16, 256, 16), (0, 1, 96, 16), (1, 4, 511, 8),
                                                   (1, 4, 512, 16), (1, 16, 512, 8), (1, 1, 128, 16), (2, 8, 63, 8), (2, 8, 64, 16), (2, 1, 25, 16)])
def test_long_portions_take_chunks_of_16(form, seqs, rows, tokens):
    T = seqs * rows
    assert _need(form, T, seqs) == max(_bytes(form, 8, T, seqs), _bytes(form, tokens, T, seqs))


@pytest.mark.parametrize("form", range(3))
@pytest.mark.parametrize("d", [64, 128])
def test_no_step_needs_more_than_the_layers_say(form, d):
    most = {n: ops.recurrence_scratch_bytes(form, 4096, 16, d, d, n, torch.bfloat16) for n in (1, 5, 40)}
    for n, bound in most.items():
        for seqs in range(1, n + 1):
            for T in (seqs, 2 * seqs, 33, 95 * seqs, 128 * seqs - 1, 255 * seqs, 256 * seqs, 511 * seqs, 4095, 4096):
                if seqs <= T <= 4096:
                    assert _need(form, T, seqs, heads=16, d=d) <= bound, (seqs, T)
    assert ops.recurrence_scratch_bytes(form, 4096, 16, d, d, 0, torch.bfloat16) == 0


READELF = shutil.which("llvm-readelf", path="/opt/rocm/llvm/bin")


@pytest.mark.skipif(READELF is None, reason="no llvm-readelf")
def test_kernels_keep_their_registers(tmp_path):
    """No kernel of the recurrences in chunks has private memory: none spills, and none indexes an array by a lane's number."""
    data = open(_lib.MIXERS_LIB_PATH, "rb").read()
    magic, at, sizes = b"__CLANG_OFFLOAD_BUNDLE__", 0, {}
    while (at := data.find(magic, at)) >= 0:           # one bundle per source file: code objects by target
        (entries,), p = struct.unpack_from("<Q", data, at + 24), at + 32
        for _ in range(entries):
            off, size, chars = struct.unpack_from("<QQQ", data, p)
            target, p = data[p + 24:p + 24 + chars], p + 24 + chars
            code = data[at + off:at + off + size]
            if target.endswith(b"gfx950") and b"recurrence_states_kernel" in code:
                (tmp_path / "code").write_bytes(code)
                notes = subprocess.run([READELF, "--notes", tmp_path / "code"], capture_output=True, text=True, check=True).stdout
                for name, n in re.findall(r"\.name: +(\S*recurrence\S*)\n.*?\.private_segment_fixed_size: (\d+)", notes, re.S):
                    sizes[name] = int(n)
        at += 24
    assert len(sizes) > 100
    assert not {name: n for name, n in sizes.items() if n}
