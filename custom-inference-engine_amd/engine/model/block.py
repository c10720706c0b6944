"""The attention section of the reference's ``Attention.forward``
(``engine/model/block.py:53-75``) on the paged path, for a batch.

The reference, per layer and for one sequence (``B == 1`` is asserted at
``block.py:48``): rotates q and k at ``positions`` (``:53-54``), appends
the rotated k and v at ``positions[0]`` (``:57-64``), gathers the whole
history into dense tensors (``:65-67``, ``kv_cache.py:141-165``), runs
causal ``flash_attention`` with scale ``1/sqrt(head_dim)`` (``:69-71``) and
returns ``(1, L, Hq * D)`` (``:72-74``) for the output projection.
:func:`attention_section` does the same for B sequences of L new tokens
each, with RoPE fused into the kernels when the model's tables are given:

* a prefill of fresh sequences (every history is just the new tokens):
  one rotary append that also returns the rotated K densely, then prefill
  attention over the new tokens with q rotated as it is loaded;
* decode / verify ((Hq/Hk) * L <= 256 query rows per kv head, 128 at
  head_dim 256: ``paged_max_rows``): one rotary append, then paged attention
  reading K/V in place with q rotated as it is loaded;
* a long chunk on top of a history (more query rows per kv head): the rotary
  append, then the prefill kernels over the paged history
  (``paged_prefill``) -- the history is never gathered.

:func:`attention_section_rows` takes a ragged step (a different number of
new tokens per sequence, e.g. a prefill chunk next to decode tokens) as
packed rows: one append for all, then one launch per group of sequences with
equal counts, ``paged_attention`` or ``paged_prefill`` by the same bound.

The Lq new tokens of a sequence of context length ctx sit at positions
ctx - Lq .. ctx - 1 (the reference appends before it attends,
block.py:57-65), and row i sees keys <= ctx - Lq + i.

The Q/K/V projections and the output projection around it are unchanged.
"""

from __future__ import annotations

import math

import torch

from engine import _lib
from engine.attention import flash_attention, paged_attention, paged_max_rows, paged_prefill
from engine.cache import PagedKVCache, StepBatch


def attention_section(q: torch.Tensor, k: torch.Tensor, v: torch.Tensor, layer_idx: int, cache: PagedKVCache,
                      step: StepBatch, rope: tuple[torch.Tensor, torch.Tensor] | None = None,
                      fuse_append: bool = True) -> torch.Tensor:
    """q: (B, Hq, L, D), k/v: (B, Hk, L, D): the L new tokens of each
    sequence, at positions ``starts[b] + 0..L-1``, after RoPE when ``rope``
    is None, before it when ``rope`` is the model's (cos, sin) tables
    (``RotaryEmbedding.tables``). ``step`` is ``cache.prepare_step(tables,
    L, starts)``, made once per engine step before the first layer: it
    allocates the blocks, extends the lengths (so the history includes the
    new tokens, as in the reference, which appends before it attends) and
    holds the step's device metadata. Returns (B, L, Hq * D).

    With ``fuse_append`` (default) a step whose new tokens are the newest of
    every sequence appends inside the paged attention launch pair
    (``paged_attention(new_kv=..., rope=rope)``), bit-identical to
    ``append_step`` followed by ``paged_attention``."""
    B, Hq, L, D = q.shape
    if step.context_lens.shape[0] != B or k.shape[0] != B or v.shape[0] != B or step.num_new != L:
        raise ValueError(f"step of {step.context_lens.shape[0]} sequences x {step.num_new} tokens "
                         f"for q of shape {tuple(q.shape)}")
    Hk = k.shape[1]
    fused = fuse_append and not step.fresh and step.aligned and (Hq // Hk) * L <= paged_max_rows(D)
    if fused:  # decode / verify: append and attention in one call
        plan = step.plan_for(True)
        cos, sin = rope if rope is not None else (None, None)
        done = _lib.host().section(q, k, v, cache.k[layer_idx], cache.v[layer_idx], step.block_tables,
                                   step.context_lens, step.max_context, cos, sin,
                                   *((plan.data, plan.split, plan.key) if plan is not None else (None, None, None)))
        if done is not None:
            return _lib.checked(done)
    scale = 1.0 / math.sqrt(D)
    # the kernels write (B, L, Hq, D) directly: the reference's
    # transpose(1, 2).contiguous() of the output (block.py:72-74) is free
    out_rows = torch.empty((B, L, Hq, D), dtype=q.dtype, device=q.device)
    out = out_rows.transpose(1, 2)
    # the rows of sequence b are consecutive in (B*L, Hk, D)
    k_rows = k.transpose(1, 2).reshape(B * L, Hk, D)
    v_rows = v.transpose(1, 2).reshape(B * L, Hk, D)

    if step.fresh:
        # history == the new tokens: attend over them directly (the gathered
        # history of the reference is bit-identical to them)
        if rope is None:
            cache.append_step(layer_idx, step, k_rows, v_rows)
            flash_attention(q, k, v, causal=True, scale=scale, out=out)
        else:
            k_rot = torch.empty_like(k_rows)
            cache.append_step(layer_idx, step, k_rows, v_rows, rope=rope, k_out=k_rot)
            flash_attention(q, k_rot.view(B, L, Hk, D).transpose(1, 2), v, causal=True, scale=scale, rope=rope,
                            out=out)  # positions 0..L-1
    elif fused:
        cache._validate(k_rows)
        cache._validate(v_rows)
        paged_attention(q, cache.k[layer_idx], cache.v[layer_idx], step.block_tables, step.context_lens,
                        causal=True, scale=scale, max_context=step.max_context, rope=rope, out=out,
                        new_kv=(k_rows, v_rows), plan=step.plan_for(True))
    elif (Hq // Hk) * L <= paged_max_rows(D):
        cache.append_step(layer_idx, step, k_rows, v_rows, rope=rope)
        q_rope = rope
        if rope is not None and not step.aligned:
            # positions start + i differ from context_len - L + i: rotate q first
            from engine.model.rope import rope_apply

            pos = step.starts[:, None] + torch.arange(L, device=q.device, dtype=torch.int32)[None, :]
            q, q_rope = rope_apply(q, rope[0], rope[1], positions=pos), None
        paged_attention(q, cache.k[layer_idx], cache.v[layer_idx], step.block_tables, step.context_lens,
                        causal=True, scale=scale, max_context=step.max_context, rope=q_rope, out=out,
                        plan=step.plan_for(False))
    else:
        cache.append_step(layer_idx, step, k_rows, v_rows, rope=rope)
        _paged_rows(q.transpose(1, 2).reshape(B * L, Hq, D), layer_idx, cache, step, rope,
                    out_rows.view(B * L, Hq, D))
    return out_rows.view(B, L, Hq * D)


def attention_section_rows(q: torch.Tensor, k: torch.Tensor, v: torch.Tensor, layer_idx: int,
                           cache: PagedKVCache, step: StepBatch,
                           rope: tuple[torch.Tensor, torch.Tensor] | None = None) -> torch.Tensor:
    """The attention section for a step of any shape, ragged ones included:
    q (T, Hq, D), k / v (T, Hk, D) hold the new tokens of all sequences as
    packed rows, sequence b's ``step.new_counts[b]`` rows consecutive (the
    layout of ``step.cu_new``), at positions ``starts[b] + i``, un-rotated
    when ``rope`` is given. ``step`` is ``cache.prepare_step(tables,
    counts)``. Returns (T, Hq * D), row for row. One append for every
    sequence, then one attention launch per group of sequences with equal
    counts."""
    T, Hq, D = q.shape
    Hk = k.shape[1]
    if T != step.total_new or k.shape[0] != T or v.shape[0] != T or k.shape[1:] != (Hk, D) \
            or tuple(v.shape) != tuple(k.shape):
        raise ValueError(f"step of {step.total_new} new tokens for q {tuple(q.shape)}, k {tuple(k.shape)}, "
                         f"v {tuple(v.shape)}")
    out = torch.empty((T, Hq, D), dtype=q.dtype, device=q.device)
    cache.append_step(layer_idx, step, k, v, rope=rope)
    _paged_rows(q, layer_idx, cache, step, rope, out)
    return out.view(T, Hq * D)


def _paged_rows(q_rows: torch.Tensor, layer_idx: int, cache: PagedKVCache, step: StepBatch,
                rope: tuple[torch.Tensor, torch.Tensor] | None, out_rows: torch.Tensor) -> None:
    """Paged attention of the packed new-token rows of ``step`` (already
    appended) over each sequence's history, into ``out_rows`` (T, Hq, D): one
    launch per count of new tokens, ``paged_attention`` up to
    ``paged_max_rows(D)`` query rows per kv head and ``paged_prefill`` above
    (1000 new tokens on 4600, 32/8 heads, D=128 bf16: the whole section 119 us,
    against 1030 with paged_attention launches of that many rows each, which
    reread the history once per 64 tokens). A group whose rows are consecutive is read and
    written in place, others through an index (two more launches). The
    device index tensors of each launch are built on the first call of the
    step and reused by every layer."""
    T, Hq, D = q_rows.shape
    Hk = cache.cfg.num_kv_heads
    scale = 1.0 / math.sqrt(D)
    dev = q_rows.device
    if rope is not None and not step.aligned:
        # positions start + i differ from context_len - count + i: rotate q first
        from engine.model.rope import rope_apply

        key = ("positions",)
        if key not in step.cache:
            pos = [s0 + i for s0, c in zip(step.starts_host, step.new_counts) for i in range(c)]
            step.cache[key] = torch.tensor(pos, dtype=torch.int32).to(dev)
        q_rows = rope_apply(q_rows.transpose(0, 1).unsqueeze(0), rope[0], rope[1],
                            positions=step.cache[key])[0].transpose(0, 1)
        rope = None
    key = ("launches",)
    if key not in step.cache:
        step.cache[key] = _launches(step, dev)
    for tables, rows, lens, L, r0, max_context in step.cache[key]:
        n = lens.shape[0]
        # (a group of more query heads per kv head than paged_attention takes is refused there)
        attend = paged_prefill if Hq // Hk <= paged_max_rows(D) < Hq // Hk * L else paged_attention
        qs = (q_rows[rows] if r0 is None else q_rows[r0:r0 + n * L]).view(n, L, Hq, D).transpose(1, 2)
        out = None if r0 is None else out_rows[r0:r0 + n * L].view(n, L, Hq, D).transpose(1, 2)
        o = attend(qs, cache.k[layer_idx], cache.v[layer_idx], tables, lens, causal=True, scale=scale,
                   max_context=max_context, rope=rope, out=out)
        if r0 is None:
            out_rows[rows] = o.transpose(1, 2).reshape(-1, Hq, D)


def _group_span(step: StepBatch, seqs: list[int], count: int) -> tuple[int | None, int]:
    """First packed row of the sequences ``seqs`` with ``count`` new tokens
    each when their rows are consecutive (else None), and their longest
    context."""
    between = step.new_counts[seqs[0]:seqs[-1] + 1]
    contiguous = all(c in (count, 0) for c in between)
    return (sum(step.new_counts[:seqs[0]]) if contiguous else None), max(step.lengths_host[b] for b in seqs)


def _launches(step: StepBatch, dev: torch.device) -> list:
    """(block tables (B', max_blocks), packed row indices (B' * L,), context
    lengths (B',), L, first packed row or None, longest context) per count L of
    new tokens in the step; the indices are uploaded in one copy."""
    groups: dict[int, list[int]] = {}
    for b, c in enumerate(step.new_counts):
        if c > 0:
            groups.setdefault(c, []).append(b)
    if not groups:
        return []
    cu = [0]
    for c in step.new_counts:
        cu.append(cu[-1] + c)
    flat = []
    for c, seqs in sorted(groups.items()):
        flat += seqs + [cu[b] + i for b in seqs for i in range(c)] + [step.lengths_host[b] for b in seqs]
    flat = torch.tensor(flat, dtype=torch.int64).to(dev)
    out, p = [], 0
    for c, seqs in sorted(groups.items()):
        n = len(seqs)
        out.append((step.block_tables[flat[p:p + n]], flat[p + n:p + n + n * c],
                    flat[p + n + n * c:p + 2 * n + n * c].to(torch.int32), c, *_group_span(step, seqs, c)))
        p += 2 * n + n * c
    return out
