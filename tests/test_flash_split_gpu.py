"""GPU parity of the prefill kernels with key splits (cie_flash_fwd_ex) and over
a paged history (cie_flash_paged) against the CPU oracle: every head_dim, split
counts from one to more splits than key tiles, context lengths around the tile
edges, block sizes on both copy paths (one block per wave's rows, several), more
block ids than the kernel stages, and invalid lengths and block ids (NaN rows of
that sequence only). Tolerances are those of the unsplit kernels: a split only
reorders fp32 sums."""

from __future__ import annotations

import ctypes
import math

import pytest
import torch

from engine import _lib
from engine.attention import flash_attention, paged_attention, paged_prefill
from engine.model.rope import build_rope_cache
from oracle import flash_attention_ref, gather_ref, rope_ref

pytestmark = pytest.mark.gpu
DEV = "cuda"
TOL = {torch.float16: 2e-3, torch.bfloat16: 1e-2}


def _randn(g, *shape, dtype):
    return torch.randn(shape, generator=g).to(dtype)


def _close(out, ref, tol, what):
    out, ref = out.float().cpu(), ref.float()
    assert torch.equal(torch.isnan(out), torch.isnan(ref)), f"{what}: NaN pattern"
    err = (out - ref).nan_to_num().abs().max().item()
    assert err <= tol, f"{what}: {err:.3e}"


def _flash(q, k, v, causal, splits):
    lib = _lib.load()
    B, Hq, Lq, D = q.shape
    Hk, Lk = k.shape[1], k.shape[2]
    nbytes = lib.cie_flash_workspace_bytes(B, Hq, Hk, Lq, Lk, D, int(causal), splits)
    assert (nbytes > 0) == (splits > 1)
    ws = torch.empty(max(nbytes, 16), dtype=torch.uint8, device=DEV)
    o = torch.full((B, Hq, Lq, D), 7.0, dtype=q.dtype, device=DEV)
    _lib.check(lib.cie_flash_fwd_ex(
        q.data_ptr(), k.data_ptr(), v.data_ptr(), o.data_ptr(), *(_lib.strides(t) for t in (q, k, v, o)), B, Hq, Hk,
        Lq, Lk, D, ctypes.c_float(1.0 / math.sqrt(D)), int(causal), _lib.DTYPE_CODES[q.dtype], None, None, 0, 0, None,
        splits, ws.data_ptr(), nbytes, _lib.stream_handle(q.device)))
    return o


@pytest.mark.parametrize("D", [16, 32, 64, 128, 256])
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("Lq,Lk,causal", [(1, 1, True), (5, 129, True), (33, 300, False), (130, 257, True),
                                          (200, 70, True), (1, 2049, True)])
def test_splits_match_oracle(D, dtype, Lq, Lk, causal):
    g = torch.Generator().manual_seed(D + Lq + Lk)
    q, k, v = _randn(g, 2, 4, Lq, D, dtype=dtype), _randn(g, 2, 2, Lk, D, dtype=dtype), _randn(g, 2, 2, Lk, D, dtype=dtype)
    ref = flash_attention_ref(q.float(), k.float(), v.float(), causal=causal)
    q, k, v = q.to(DEV), k.to(DEV), v.to(DEV)
    for splits in (1, 2, 3, 7, 32):
        _close(_flash(q, k, v, causal, splits), ref, TOL[dtype], f"splits={splits}")


@pytest.mark.parametrize("D", [64, 128])
def test_split_short_query_equals_expanded_heads_bitwise(D):
    """flash_attention of a few rows over a long history splits its keys; the
    split depends on B * Hq, not on the group, so GQA equals expanded MHA."""
    g = torch.Generator().manual_seed(D)
    q, k, v = (_randn(g, 1, h, n, D, dtype=torch.float16).to(DEV) for h, n in ((8, 5), (2, 3001), (2, 3001)))
    assert _lib.load().cie_flash_workspace_bytes(1, 8, 2, 5, 3001, D, 1, 0) > 0
    a = flash_attention(q, k, v, causal=True)
    assert torch.equal(a, flash_attention(q, k.repeat_interleave(4, 1), v.repeat_interleave(4, 1), causal=True))
    _close(a, flash_attention_ref(q.cpu().float(), k.cpu().float(), v.cpu().float(), causal=True), 2e-3, "short query")
    # an infinite score stays in its row, as in one pass over the keys
    q[0, 1, 2, 0] = float("inf")
    bad = flash_attention(q, k, v, causal=True)
    assert torch.isnan(bad[0, 1, 2]).all()
    keep = torch.ones(8, 5, dtype=torch.bool)
    keep[1, 2] = False
    _close(bad[0].cpu()[keep], a[0].cpu()[keep], 2e-3, "rows beside an infinite score")


@pytest.mark.parametrize("D,bs,dtype", [(16, 16, torch.float16), (32, 32, torch.bfloat16), (64, 16, torch.float16),
                                        (64, 5, torch.bfloat16), (128, 8, torch.float16), (128, 16, torch.bfloat16),
                                        (256, 48, torch.float16), (128, 1, torch.bfloat16)])
@pytest.mark.parametrize("rope", [False, True])
def test_paged_prefill_matches_oracle(D, bs, dtype, rope):
    Hq, Hk, Lq = 4, 2, 140
    lens = [140, 161, 256, 1100, 300, 200]  # 1100 one-token blocks: more ids than are staged
    g = torch.Generator().manual_seed(D + bs)
    width = -(-max(lens) // bs)
    need = [-(-n // bs) for n in lens]
    ids = torch.randperm(sum(need), generator=g).tolist()
    bt = torch.zeros(len(lens), width, dtype=torch.int32)
    for b, n in enumerate(need):
        bt[b, :n] = torch.tensor([ids.pop() for _ in range(n)])
    kp, vp = (_randn(g, sum(need), bs, Hk, D, dtype=dtype) for _ in range(2))
    q = _randn(g, len(lens), Hq, Lq, D, dtype=dtype)
    cos, sin = build_rope_cache(2048, D)
    ref = []
    for b, n in enumerate(lens):
        kh, vh = (gather_ref(p, bt[b, :need[b]].tolist(), n).transpose(0, 1).unsqueeze(0).float() for p in (kp, vp))
        qb = rope_ref(q[b:b + 1], cos, sin, torch.arange(n - Lq, n)) if rope else q[b:b + 1]
        ref.append(flash_attention_ref(qb.float(), kh, vh, causal=True))
    ref = torch.cat(ref)
    lt = torch.tensor(lens, dtype=torch.int32)
    bad_bt = bt.clone()
    bad_bt[4, 2] = sum(need)   # the block of sequence 4's third block lies outside the pool
    bad_lens = lt.clone()
    bad_lens[5] = width * bs + 1
    qd, kd, vd = q.to(DEV), kp.to(DEV), vp.to(DEV)
    tabs = (cos.to(DEV), sin.to(DEV)) if rope else None
    out = paged_prefill(qd, kd, vd, bt.to(DEV), lt.to(DEV), rope=tabs)
    _close(out, ref, TOL[dtype], "paged_prefill")
    # rows whose keys touch no invalid block keep their value or are NaN; a whole invalid sequence is NaN
    got = paged_prefill(qd, kd, vd, bad_bt.to(DEV), bad_lens.to(DEV), rope=tabs).cpu()
    assert torch.equal(got[:4], out[:4].cpu()) and torch.isnan(got[5]).all()
    last = lens[4] - 1  # its last row sees every block
    assert torch.isnan(got[4, :, Lq - 1]).all() and last >= 2 * bs
    # every split count gives the oracle's rows too, and NaN where it must
    lib = _lib.load()
    for splits in (1, 2, 5, 32):
        nbytes = lib.cie_flash_paged_workspace_bytes(len(lens), Hq, Hk, Lq, D, 0, bs, width, splits)
        ws = torch.empty(max(nbytes, 16), dtype=torch.uint8, device=DEV)
        for t, n, want in ((bt, lt, ref), (bad_bt, bad_lens, None)):
            o = torch.full_like(qd, 7.0)
            td, nd = t.to(DEV), n.to(DEV)
            rp = (tabs[0].data_ptr(), tabs[1].data_ptr(), 2048, 2) if rope else (None, None, 0, 0)
            _lib.check(lib.cie_flash_paged(
                qd.data_ptr(), kd.data_ptr(), vd.data_ptr(), td.data_ptr(), nd.data_ptr(), o.data_ptr(),
                *(_lib.strides(x) for x in (qd, kd, vd, o)), len(lens), Hq, Hk, Lq, D, sum(need), bs, width, 0,
                ctypes.c_float(1.0 / math.sqrt(D)), 1, _lib.DTYPE_CODES[dtype], *rp, splits, ws.data_ptr(), nbytes,
                _lib.stream_handle(qd.device)))
            if want is not None:
                _close(o, want, TOL[dtype], f"splits={splits}")
            else:
                assert torch.isnan(o[5]).all() and torch.isnan(o[4, :, Lq - 1]).all()


@pytest.mark.parametrize("D", [16, 32, 64, 128, 256])
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("rising", [False, True])
def test_paged_prefill_error_is_the_rounding_of_its_output(D, dtype, rising):
    """P in two 16-bit parts leaves about 16 (bf16) to 22 (fp16) of its bits and
    the row sums stay in fp32, so against 64 bits the result is off by its one
    rounding to 16 bits and little else (with P rounded to 16 bits it would be
    1.4 times that). rising: scores that grow along the keys past 2^10 take the
    recompute of the running max."""
    Hq, Hk, Lq, n, bs = 4, 2, 150, 1203, 16
    g = torch.Generator().manual_seed(D)
    nb = -(-n // bs)
    kp, vp = (_randn(g, nb, bs, Hk, D, dtype=dtype) for _ in range(2))
    q = _randn(g, 1, Hq, Lq, D, dtype=dtype)
    if rising:
        q = q.abs()
        kp = (kp.abs() * torch.linspace(0, 24 / D ** 0.5, nb).view(-1, 1, 1, 1)).to(dtype)
    bt = torch.randperm(nb, generator=g).view(1, nb).int()
    kh, vh = (gather_ref(p, bt[0].tolist(), n).transpose(0, 1).double().repeat_interleave(Hq // Hk, 0) for p in (kp, vp))
    s = q[0].double() @ kh.transpose(1, 2).contiguous() / math.sqrt(D)
    s.masked_fill_(torch.arange(n) > torch.arange(Lq).unsqueeze(1) + n - Lq, -math.inf)
    ref = torch.softmax(s, -1) @ vh
    rel = lambda x: ((x.double() - ref).norm() / ref.norm()).item()  # noqa: E731
    out = paged_prefill(q.to(DEV), kp.to(DEV), vp.to(DEV), bt.to(DEV), torch.tensor([n], dtype=torch.int32, device=DEV))
    assert rel(out[0].cpu()) <= 1.05 * rel(ref.to(dtype))


@pytest.mark.parametrize("D,bs", [(16, 16), (64, 5), (128, 16), (256, 8)])
@pytest.mark.parametrize("kw", [{}, {"causal": False}, {"max_context": 200}, {"scale": -0.4}, {"scale": 0.0}])
@pytest.mark.parametrize("rope", [False, True])
def test_paged_prefill_answers_as_paged_attention(D, bs, kw, rope):
    """The route of long chunks against the one of short ones over the lengths
    both take: empty, shorter than the new tokens, at tile edges, at and past
    the table's and the hint's limit, negative, with a pool of other strides;
    NaN and zero rows in the same places."""
    Hq, Hk, Lq = 4, 2, 40
    lens = [0, 1, 39, 40, 41, 63, 64, 65, 199, 200, 201, 256, 300, 301, -1, 2 ** 30]
    g = torch.Generator().manual_seed(D + bs)
    width = -(-300 // bs)
    # ids of lengths within the table (-(-300 // bs) * bs tokens); any valid ids do for the others
    bt = torch.randint(0, 70, (len(lens), width), generator=g).int().to(DEV)
    pool = torch.randn(2, 70, Hk, bs, D + 8, generator=g).half().to(DEV)
    kp, vp = pool[0, ..., :D].transpose(1, 2), pool[1, ..., :D].transpose(1, 2)
    q = _randn(g, len(lens), Lq, Hq, D, dtype=torch.float16).to(DEV).transpose(1, 2)
    lt = torch.tensor(lens, dtype=torch.int32, device=DEV)
    tabs = tuple(t.to(DEV) for t in build_rope_cache(250, D)) if rope else None  # positions from 250 on are NaN rows
    a = paged_attention(q, kp, vp, bt, lt, rope=tabs, **kw)
    b = paged_prefill(q, kp, vp, bt, lt, rope=tabs, **kw)
    _close(b, a.cpu(), 2e-3, "paged_prefill")
    assert torch.isnan(a[-1]).all() and (a[0] == 0).all()
