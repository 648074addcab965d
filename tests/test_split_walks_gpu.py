"""Calls with few 32-row tiles split each tile's walk over a workgroup's waves
(split_walks, dil_walk.hpp), and fp32 / split operands take the dq pass in
groups of 4 tiles instead of 8 (query_few).

Forward, demand and gradients against the fp64 oracle at the edges of a tile
and on both sides of each type's limit, with the bounds of the forward's and
backward's own tests: fp32 operands 1e-4 max-abs, bf16 operands 2e-2 for the
output and 5e-2 for the gradients.
"""

from __future__ import annotations

import pytest
import torch

from gpu_helpers import max_abs, needs_gpu
from oracle import dilution_oracle as orc

pytestmark = [pytest.mark.gpu, needs_gpu]

# head dim, operand type, and the limit in tiles of that pair
LIMITS = [(16, "bf16", 2048), (32, "bf16", 2048), (64, "bf16", 1280), (128, "bf16", 768), (64, "ieee", 2048),
          (128, "ieee", 1024), (32, "tf32", 1024), (64, "tf32", 640), (128, "tf32", 640)]


def _check(q, k, v, do, prec, slices):
    """One call over all slices; the named slices against the oracle."""
    from dilution import kernels

    xs = [t.cuda().requires_grad_(True) for t in (q, k, v)]
    out = kernels.dilution_attention(*xs, dot_precision=prec)
    out.backward(do.cuda())
    _, aux = kernels.dilution_attention_forward(*(x.detach() for x in xs), dot_precision=prec, return_aux=True)
    b16 = prec == "bf16"
    for s in slices:
        one = [t[:, s:s + 1].double() for t in (q, k, v, do)]
        want, _ = orc.grads_closed_form_f64(*(t.numpy() for t in one))
        assert max_abs(out.detach()[:, s:s + 1], orc.attention_f64(*one[:3])) < (2e-2 if b16 else 1e-4)
        for name, x, w in zip(("dq", "dk", "dv"), xs, want):
            assert max_abs(x.grad[:, s:s + 1], torch.as_tensor(w)) < (5e-2 if b16 else 1e-4), (name, s)
        scores = (one[0] @ one[1].transpose(-1, -2)) / q.shape[-1] ** 0.5
        t = q.shape[-2]
        total = scores.masked_fill(torch.ones(t, t, dtype=torch.bool).triu(1), float("-inf")).softmax(-1).sum(-2)
        # the columns of p: fp32 exponentials (and, for bf16 operands, exact products of the given values)
        assert max_abs(aux["committed_total"][:, s:s + 1], total) < 1e-5 * max(1.0, t ** 0.5)


@pytest.mark.parametrize("dim,prec", [(d, p) for d, p, _ in LIMITS])
@pytest.mark.parametrize("seq", [1, 31, 33, 129, 300])
def test_tile_edges(dim, prec, seq):
    dtype = torch.bfloat16 if prec == "bf16" else torch.float32
    q, k, v, do = orc.make_inputs((1, 2, seq, dim), seed=seq + dim, qk_scale=0.5, with_dout=True, dtype=dtype)
    _check(q, k, v, do, prec, (0, 1))


@pytest.mark.parametrize("over", [0, 1])
@pytest.mark.parametrize("dim,prec,limit", LIMITS)
def test_both_sides_of_the_limit(dim, prec, limit, over):
    """As many slices of 65 rows (3 tiles) as the limit takes, and one more."""
    dtype = torch.bfloat16 if prec == "bf16" else torch.float32
    heads = limit // 3 + over
    q, k, v, do = orc.make_inputs((1, heads, 65, dim), seed=dim + over, qk_scale=0.5, with_dout=True, dtype=dtype)
    _check(q, k, v, do, prec, (0, heads // 2, heads - 1))


@pytest.mark.parametrize("prec", ["bf16", "ieee", "tf32"])
@pytest.mark.parametrize("chunk", [37, 96])
def test_prefill_chunks(prec, chunk):
    """Chunks whose first row lies inside a tile, with demand carried in."""
    from dilution import cache, kernels

    dtype = torch.bfloat16 if prec == "bf16" else torch.float32
    q, k, v = (t.cuda() for t in orc.make_inputs((1, 2, 300, 64), seed=chunk, qk_scale=0.5, dtype=dtype))
    got, state = cache.begin_cache(q, k, v, capacity=300, chunk=chunk, dot_precision=prec)
    assert max_abs(got, orc.attention_f64(q.cpu(), k.cpu(), v.cpu())) < (2e-2 if prec == "bf16" else 1e-4)
    _, aux = kernels.dilution_attention_forward(q, k, v, dot_precision=prec, return_aux=True)
    assert max_abs(state["committed"].reshape(1, 2, 300), aux["committed_total"].cpu()) < 2e-4


def _check_chunk(heads, dim, prec, start, rows, slices):
    """One prefill chunk over `heads` slices with demand carried in; the named
    slices' checkpoints, totals and outputs against fp64."""
    from dilution import kernels

    dtype = torch.bfloat16 if prec == "bf16" else torch.float32
    g = torch.Generator(device="cuda").manual_seed(start + dim)
    length, blocks = start + rows, (rows + 31) // 32
    q = (0.5 * torch.randn(1, heads, rows, dim, device="cuda", generator=g)).to(dtype)
    k, v = ((s * torch.randn(1, heads, length, dim, device="cuda", generator=g)).to(dtype) for s in (0.5, 1.0))
    before = torch.zeros(1, heads, length + 9, device="cuda")
    before[..., :start] = 3 * torch.rand(1, heads, start, device="cuda", generator=g)
    kc, vc = (torch.cat([x, torch.zeros_like(x[:, :, :1]).expand(-1, -1, 9, -1)], dim=2) for x in (k, v))
    committed = before.clone()
    out, aux = kernels.dilution_prefill_chunk(q, kc, vc, committed, start, dot_precision=prec, return_aux=True)
    future = torch.arange(length, device="cuda")[None, :] > start + torch.arange(rows, device="cuda")[:, None]
    for s in slices:
        scores = (q[0, s].double() @ k[0, s].double().T.contiguous()) / dim ** 0.5
        p = scores.masked_fill(future, float("-inf")).softmax(-1)
        demand = before[0, s, :length].double() + p.cumsum(-2)            # after each row
        share = p / (demand + 1e-9)
        want = (share / (share.sum(-1, keepdim=True) + 1e-9)) @ v[0, s].double()
        carry = aux["carry"].reshape(heads, blocks, length)[s]
        assert torch.equal(carry[0, :start], before[0, s, :start]), s
        for b in range(1, blocks):
            end = min(length, start + 32 * (b + 1))
            assert (carry[b, :end].double() - demand[32 * b - 1, :end]).abs().max() < 2e-5, (s, b)
        assert (committed[0, s, :length].double() - demand[-1]).abs().max() < 2e-5, s
        assert (out[0, s].double() - want).abs().max() < (2e-2 if prec == "bf16" else 1e-4), s
    assert torch.equal(committed[..., length:], before[..., length:])


@pytest.mark.parametrize("dim,prec,start,rows", [(64, "ieee", 1000, 300), (64, "tf32", 1000, 300), (64, "bf16", 1000, 300),
                                                 (64, "bf16", 1024, 300), (32, "bf16", 37, 100), (128, "tf32", 70, 130)])
def test_carried_demand_is_read_before_it_is_advanced(dim, prec, start, rows):
    """A chunk's demand pass takes the carried demand from the memory that it
    advances (committed): all 4 waves of a key tile have to read it before one
    of them stores the new total.  Every checkpoint against fp64, the first one
    (the carried demand itself) bit for bit, over 6 slices' key tiles at once.

    Tolerance: the demand is below 4; its terms p <= 1 carry about 1e-5
    relative (hardware exp2, scores rounded to fp32) and sum to less than 1 per
    key beside the diagonal's few: 2e-5; outputs as in the tests above."""
    _check_chunk(6, dim, prec, start, rows, range(6))


@pytest.mark.parametrize("over", [0, 1])
@pytest.mark.parametrize("dim,prec,limit", [(16, "bf16", 2048), (64, "bf16", 640), (128, "bf16", 384), (64, "ieee", 640),
                                            (128, "ieee", 512), (32, "tf32", 512), (64, "tf32", 320)])
def test_both_sides_of_the_key_tile_limit(dim, prec, limit, over):
    """A chunk past row 0 counts key tiles for its demand pass: as many slices
    of 8 key tiles (5 row blocks) as the limit takes, and one more; and chunks of
    3 and 4 row blocks."""
    heads = limit // 8 + over
    _check_chunk(heads, dim, prec, 97, 147, (0, heads // 2, heads - 1))
    _check_chunk(2, dim, prec, 130, 96 + over, (0, 1))
    if (dim, prec) == (16, "bf16"):                            # 16 row blocks or more: twice the key tiles
        _check_chunk(128 + over, dim, prec, 500, 512, (0, 127))


@pytest.mark.parametrize("dim,prec,limit", [(64, "ieee", 2048), (64, "tf32", 640), (128, "bf16", 768), (32, "bf16", 2048)])
def test_groups_have_the_bits_of_the_whole_call(dim, prec, limit):
    """A call without aux whose checkpoint scratch is over its budget runs its
    slices in groups: a call just above the limit in groups below it, and one
    below the limit."""
    from dilution import kernels

    dtype = torch.bfloat16 if prec == "bf16" else torch.float32
    g = torch.Generator(device="cuda").manual_seed(dim)
    for heads in (limit // 3 + 1, limit // 3 - 1):                        # 3 row tiles per slice
        q, k, v = (torch.randn(1, heads, 90, dim, device="cuda", generator=g).to(dtype) for _ in range(3))
        whole = kernels.dilution_attention_forward(q, k, v, dot_precision=prec)
        for rows in (heads // 2, heads - 1, 1 if heads < 300 else heads // 7):
            budget = (rows + 0.5) * 3 * 90 * 4 / 2 ** 30
            assert torch.equal(whole, kernels.dilution_attention_forward(q, k, v, dot_precision=prec,
                                                                         scratch_budget_gib=budget)), (heads, rows)


def test_long_row_keeps_the_full_demand_walk():
    """One slice of more row blocks than the split demand pass holds the sums of
    (256) takes the statistics and the output split and the demand whole."""
    from dilution import kernels

    q, k, v = (t.cuda() for t in orc.make_inputs((1, 1, 8225, 32), seed=5, qk_scale=0.5, dtype=torch.float32))
    out, aux = kernels.dilution_attention_forward(q, k, v, dot_precision="ieee", return_aux=True)
    head, head_aux = kernels.dilution_attention_forward(*(x[:, :, :8192].contiguous() for x in (q, k, v)),
                                                        dot_precision="ieee", return_aux=True)
    # fp32 sums of the same terms in another order: 8192 demand terms below 1, in fp64
    assert max_abs(out[:, :, :8192], head.cpu()) < 1e-5
    p = (q[:, :, 8192:].double() @ k.double().transpose(-1, -2).contiguous()) / 32 ** 0.5
    mask = torch.ones(8225, 8225, dtype=torch.bool, device="cuda").triu(1)[8192:]
    tail = p.masked_fill(mask, float("-inf")).softmax(-1).sum(-2)
    assert max_abs(aux["committed_total"][..., :8192].double() - head_aux["committed_total"].double(),
                   tail[..., :8192].cpu()) < 1e-4
