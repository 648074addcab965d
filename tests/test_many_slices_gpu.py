"""More (batch * head) slices than a grid's y dimension holds (65535): the
kernels that put the slice on grid y are launched in batches of slices.
Forward, backward and the decode step over 65600 slices of a short sequence
against the fp64 oracle (fp32 tolerances)."""

from __future__ import annotations

import pytest
import torch

from gpu_helpers import max_abs, needs_gpu
from oracle import dilution_oracle as orc

pytestmark = [pytest.mark.gpu, needs_gpu]

SHAPE = (4, 16400, 8, 16)          # n = 65600 slices


def test_forward_backward_past_grid_y_limit():
    from dilution import kernels

    q, k, v, do = orc.make_inputs(SHAPE, seed=31, with_dout=True)
    xs = [t.cuda().requires_grad_(True) for t in (q, k, v)]
    out = kernels.dilution_attention(*xs, dot_precision="ieee")
    out.backward(do.cuda())
    assert max_abs(out.detach(), orc.attention_f64(q, k, v)) < 1e-4
    want, _ = orc.grads_closed_form_f64(q.numpy(), k.numpy(), v.numpy(), do.numpy())
    for name, x, w in zip(("dq", "dk", "dv"), xs, want):
        assert max_abs(x.grad, torch.from_numpy(w)) < 1e-4, name


def test_decode_past_grid_y_limit():
    from dilution import kernels

    q, k, v = orc.make_inputs(SHAPE, seed=32)
    t = SHAPE[2]
    _, aux = kernels.dilution_attention_forward(q[:, :, :t - 1].cuda(), k[:, :, :t - 1].cuda(),
                                                v[:, :, :t - 1].cuda(), return_aux=True)
    committed = torch.zeros(*SHAPE[:2], t, device="cuda")
    committed[:, :, :t - 1] = aux["committed_total"]
    y = kernels.dilution_decode_step(q[:, :, t - 1:].contiguous().cuda(), k.cuda(), v.cuda(), committed, t)
    assert max_abs(y[:, :, 0], orc.attention_f64(q, k, v)[:, :, t - 1]) < 1e-4
    assert max_abs(committed, orc.demand_totals(q, k)) < 1e-5


@pytest.mark.parametrize("seq", [2049, 2560, 4097])
def test_key_group_size_does_not_change_the_bits(seq):
    """Above 2048 keys the forward's key pass takes groups of 256 or 512 keys
    by the size of the call (keyout_waves); a slice's outputs, row sums and
    demand totals have the same bits alone (256-key groups) and among many
    slices (512)."""
    from dilution import kernels

    many = 2 ** 19 // seq
    g = torch.Generator(device="cuda").manual_seed(seq)
    q, k, v = (torch.randn(1, many, seq, 64, device="cuda", generator=g, dtype=torch.float32).to(torch.bfloat16)
               for _ in range(3))
    out, aux = kernels.dilution_attention_forward(q, k, v, dot_precision="bf16", return_aux=True)
    for s in (0, many // 2, many - 1):
        one, one_aux = kernels.dilution_attention_forward(q[:, s:s + 1], k[:, s:s + 1], v[:, s:s + 1],
                                                          dot_precision="bf16", return_aux=True)
        assert torch.equal(one[0, 0], out[0, s])
        assert torch.equal(one_aux["ssum"][0], aux["ssum"][s])
        assert torch.equal(one_aux["committed_total"][0, 0], aux["committed_total"][0, s])


@pytest.mark.parametrize("heads,seq,pk", [(1, 1, True), (3, 33, True), (4, 257, False), (4, 256, False), (64, 2048, True),
                                          (65, 2048, True), (2, 2048, False), (512, 256, True), (513, 256, True)])
def test_few_short_rows_forward(heads, seq, pk):
    """Few short rows take the three-pass forward (few_short_rows), the others
    the key pass: on both sides of each limit of the rule the outputs, the row
    sums and the demand are the reference's, with and without checkpoints kept,
    and a call without aux has the bits of the call with it."""
    from dilution import kernels

    g = torch.Generator(device="cuda").manual_seed(seq + heads)
    q, k, v = (torch.randn(1, heads, seq, 64, device="cuda", generator=g, dtype=torch.float32).to(torch.bfloat16)
               for _ in range(3))
    out, aux = kernels.dilution_attention_forward(q, k, v, dot_precision="bf16", return_aux=True, _save_pk=pk)
    if not pk:
        assert torch.equal(out, kernels.dilution_attention_forward(q, k, v, dot_precision="bf16"))
    for s in sorted({0, heads // 2, heads - 1}):
        xs = [x[:, s:s + 1].double() for x in (q, k, v)]
        a = (xs[0] @ xs[1].transpose(-1, -2).contiguous()) / 8
        p = a.masked_fill(torch.ones(seq, seq, dtype=torch.bool, device="cuda").triu(1), float("-inf")).softmax(-1)
        total = p.cumsum(-2)
        share = p / (total + 1e-9)
        want = (share / (share.sum(-1, keepdim=True) + 1e-9)) @ xs[2]
        assert (out[:, s:s + 1] - want).abs().max() < 2e-2
        assert ((aux["ssum"][s] - share.sum(-1)[0, 0]) / share.sum(-1)[0, 0]).abs().max() < 1e-2
        assert (aux["committed_total"][:, s] - total[:, 0, -1]).abs().max() < 1e-5 * max(1, seq ** 0.5)


@pytest.mark.parametrize("seq,few,many", [(4096, 32, 48), (4096, 3, 200), (2048, 65, 96), (2048, 64, 96), (2048, 8, 65), (300, 40, 500)])
def test_a_workspace_for_more_slices_runs_fewer(seq, few, many):
    """A C caller that sizes its workspace once, for its largest batch: smaller
    calls run in it with the bits of a call in their own (larger) one."""
    from dilution import _hip

    lib = _hip.lib()
    g = torch.Generator(device="cuda").manual_seed(seq)
    q, k, v = (torch.randn(few, seq, 64, device="cuda", generator=g).to(torch.bfloat16) for _ in range(3))
    sizes = [lib.dil_forward_workspace_bytes(n, seq, 64, 1, 2, 0) for n in (few, many)]
    assert lib.dil_prefill_workspace_bytes(many, seq, 0, 64, 1, 2) == sizes[1]
    got = []
    for size in sizes:
        out = torch.empty(few, seq, 64, device="cuda")
        stats = [torch.empty(few, seq, device="cuda") for _ in range(4)]
        ws = torch.empty(size, dtype=torch.uint8, device="cuda")
        _hip.check(lib.dil_forward(q.data_ptr(), k.data_ptr(), v.data_ptr(), few, seq, 64, 1, 2, out.data_ptr(),
                                   *(s.data_ptr() for s in stats[:3]), None, stats[3].data_ptr(), None, ws.data_ptr(),
                                   size, torch.cuda.current_stream().cuda_stream), "dil_forward")
        got.append([out, *stats])
    assert all(torch.equal(a, b) for a, b in zip(*got))
