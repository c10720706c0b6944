"""Host logic of the ragged / long-step attention section on the CPU.

attention_section_rows and the long-chunk branch of attention_section run one
launch per count of new tokens, over the sequences with that count. Checked
here:

* the launch list covers every new-token row exactly once, with the block
  table row and context length of its own sequence, and says which groups lie
  in consecutive rows and how long their contexts are;
* the oracle's causal rule (the reference's bottom-right mask,
  kernels/ref/flash_attention_ref.py:35-39) gives a prompt prefilled in chunks
  over several steps the rows of the whole prompt: chunk [i0, i1) of c new
  tokens is the i1 - i0 newest tokens of a context of length ctx - c + i1, and
  a wrong length (ctx - c + i0, or ctx) fails it."""

from __future__ import annotations

import pytest
import torch

from engine.cache import StepBatch
from engine.model.block import _launches
from oracle import flash_attention_ref


def _step(counts, lengths, width=4):
    B = len(counts)
    bt = torch.arange(B * width, dtype=torch.int32).view(B, width)
    cu = [0]
    for c in counts:
        cu.append(cu[-1] + c)
    return StepBatch(block_tables=bt, context_lens=torch.tensor(lengths, dtype=torch.int32),
                     cu_new=torch.tensor(cu, dtype=torch.int32),
                     starts=torch.tensor([n - c for n, c in zip(lengths, counts)], dtype=torch.int32),
                     num_new=-1, max_context=max(lengths), starts_host=tuple(n - c for n, c in zip(lengths, counts)),
                     lengths_host=tuple(lengths), new_counts=tuple(counts))


@pytest.mark.parametrize("counts,spans", [
    ([300, 1, 1, 0, 5, 700, 64, 1], {300: 0, 1: None, 5: 302, 700: 307, 64: 1007}),  # the last 1 is apart
    ([4, 4, 4], {4: 0}), ([1], {1: 0}), ([0, 7, 0, 0, 7, 2], {7: 0, 2: 14}),  # zeros in between stay consecutive
    ([2, 3, 2, 3], {2: None, 3: None}), ([129, 128, 127, 0], {129: 0, 128: 129, 127: 257}), ([0, 0], {}), ([], {})])
def test_launches_cover_every_row_once(counts, spans):
    lengths = [c + 37 * b for b, c in enumerate(counts)]
    step = _step(counts, lengths or [0])
    launches = _launches(step, torch.device("cpu"))
    cu = [0]
    for c in counts:
        cu.append(cu[-1] + c)
    seen = []
    for tables, rows, lens, L, r0, longest in launches:
        n = tables.shape[0]
        assert rows.numel() == n * L and lens.shape[0] == n and lens.dtype == torch.int32
        for j in range(n):
            b = int(tables[j, 0]) // 4
            assert torch.equal(tables[j], step.block_tables[b]) and counts[b] == L
            assert rows[j * L:(j + 1) * L].tolist() == list(range(cu[b], cu[b + 1]))
            assert int(lens[j]) == lengths[b]
        seen += rows.tolist()
        assert r0 == spans[L] and longest == int(lens.max())
        if r0 is not None:
            assert rows.tolist() == list(range(r0, r0 + n * L))
    assert sorted(seen) == list(range(sum(counts))) and sorted(launch[3] for launch in launches) == sorted(spans)


@pytest.mark.parametrize("c,hist,chunk", [(300, 200, 64), (97, 0, 32), (5, 1000, 2)])
def test_chunked_causal_rows_equal_the_whole_block(c, hist, chunk):
    g = torch.Generator().manual_seed(c)
    ctx = hist + c
    q = torch.randn(1, 4, c, 32, generator=g)
    k = torch.randn(1, 2, ctx, 32, generator=g)
    v = torch.randn(1, 2, ctx, 32, generator=g)
    whole = flash_attention_ref(q, k, v, causal=True)
    parts = []
    for i0 in range(0, c, chunk):
        i1 = min(c, i0 + chunk)
        n = ctx - c + i1  # the chunk's context length
        parts.append(flash_attention_ref(q[:, :, i0:i1], k[:, :, :n], v[:, :, :n], causal=True))
    assert torch.allclose(torch.cat(parts, dim=2), whole, atol=1e-6, rtol=0)
    # a planted mistake: the chunk's length taken as ctx - c + i0 shifts every mask by the chunk size
    i0, i1 = 0, min(c, chunk)
    wrong = flash_attention_ref(q[:, :, i0:i1], k[:, :, :ctx - c + i0 + 1], v[:, :, :ctx - c + i0 + 1],
                                causal=True)
    if i1 - i0 > 1:
        assert not torch.allclose(wrong.nan_to_num(9.0), whole[:, :, i0:i1], atol=1e-3)


def test_step_flags_follow_the_host_copies():
    """fresh, aligned and total_new are found once per step, and again when a
    program moves the step on by replacing its host copies."""
    step = _step([4, 4], [4, 4])
    assert step.fresh and step.aligned and step.total_new == 8
    step.starts_host, step.lengths_host = (4, 4), (8, 8)
    assert not step.fresh and step.aligned
    step.lengths_host = (9, 8)
    assert not step.aligned
    step.new_counts = (4, 3)
    assert step.total_new == 7
