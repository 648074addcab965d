"""q, k, v, dout and gradients at strided rows (dil_rows): a call on views
gives the bits of the same call on contiguous copies, in every layout that the
rule takes to the strided kernels and in those that it copies."""

from __future__ import annotations

import ctypes

import pytest
import torch

from dilution import _hip, cache, kernels, kernels_bid

# layout -> (B, H, T, D) view of new memory holding the values of x
LAYOUTS = {
    "packed": lambda x: _packed(x, 3 * x.shape[1] * x.shape[3], 0),          # views of a (B, T, 3 H D) projection
    "packed_last": lambda x: _packed(x, 3 * x.shape[1] * x.shape[3], 2 * x.shape[1] * x.shape[3]),
    "bthd": lambda x: x.transpose(1, 2).contiguous().transpose(1, 2),
    "hbtd": lambda x: x.transpose(0, 1).contiguous().transpose(0, 1),        # heads outermost
    "row_gap": lambda x: torch.cat([x, x], dim=3)[..., : x.shape[3]],        # rows 2 D apart
    "misaligned": lambda x: torch.cat([x[..., :1], x], dim=3)[..., 1:],      # odd strides and start: copied
    "dthb": lambda x: x.permute(3, 2, 1, 0).contiguous().permute(3, 2, 1, 0),  # head dims not contiguous: copied
    "row_major_t": lambda x: x.transpose(2, 3).contiguous().transpose(2, 3),   # head dims T apart: copied
}


def _packed(x, width, at):
    b, h, t, d = x.shape
    buf = torch.full((b, t, width), 3.0, dtype=x.dtype, device=x.device)
    view = buf[..., at : at + h * d].view(b, t, h, d).transpose(1, 2)
    view.copy_(x)
    return view


def _rows(x):
    return _hip.Rows(x.data_ptr(), *x.stride()[:3])


def _inputs(shape, dtype, device="cuda"):
    g = torch.Generator().manual_seed(5)
    xs = [torch.randn(shape, generator=g) * s for s in (0.5, 0.5, 1.0)]
    return [x.to(dtype).to(device) for x in xs], torch.randn(shape, generator=g).to(device)


@pytest.mark.parametrize("layout", list(LAYOUTS))
def test_rule_matches_the_library(layout):
    """strided_rows says which views dil_forward_rows takes: the library's
    own check refuses the others (-4) before any launch, and passes the
    accepted ones on to its next check (a missing output, also -4, or a
    workspace that is too small, -3)."""
    x = LAYOUTS[layout](torch.randn(2, 3, 40, 64).to(torch.bfloat16))
    lib = _hip.lib()
    fake = [ctypes.c_void_p(0x1000 * (i + 1)) for i in range(8)]
    row = _rows(x)
    status = lib.dil_forward_rows(row, row, row, 2, 3, 40, 64, 1, 2, 0, 1, 1.0, *fake[:6], None, fake[6], 0, None)
    taken = kernels._native().strided_rows(x) and x.stride(3) == 1
    assert taken == (layout not in ("misaligned", "dthb", "row_major_t"))
    if x.stride(3) == 1:                      # the library is told nothing of the head dims' stride
        assert status == (-3 if taken else -4)


def test_slice_limits_and_gradient_order():
    assert kernels._native().slice_dims(4, 16) == (4, 16)
    assert kernels._native().slice_dims(3, 1 << 16) == (3 << 16, 1)
    assert kernels._native().slice_dims(200, 10000) == (200 * 10000, 1)
    lib = _hip.lib()
    x = torch.zeros(1, 1, 8, 64, dtype=torch.bfloat16)
    row = _rows(x)
    assert lib.dil_forward_rows(row, row, row, 200, 10000, 8, 64, 1, 2, 0, 1, 1.0, *[None] * 8, 0, None) == -4
    packed = LAYOUTS["packed"](torch.zeros(2, 3, 5, 64))
    grad = kernels._native().empty_as(packed, torch.float32)
    assert grad.shape == packed.shape and grad.transpose(1, 2).is_contiguous()
    assert kernels._native().empty_as(LAYOUTS["hbtd"](torch.zeros(2, 3, 5, 64)), torch.float32).is_contiguous()


def _train(q, k, v, dout, prec, ops=kernels, **kw):
    leaves = [x.detach().requires_grad_(True) for x in (q, k, v)]
    out = ops.dilution_attention(*leaves, dot_precision=prec, **kw)
    return [out.detach(), *torch.autograd.grad(out, leaves, dout)]


@pytest.mark.gpu
@pytest.mark.parametrize("layout", list(LAYOUTS))
@pytest.mark.parametrize("shape,dtype,prec", [
    ((2, 3, 1, 64), torch.bfloat16, "bf16"),
    ((3, 5, 33, 64), torch.bfloat16, "bf16"),
    ((2, 3, 545, 64), torch.bfloat16, "bf16"),
    ((1, 4, 130, 128), torch.bfloat16, "bf16"),
    ((2, 2, 97, 16), torch.bfloat16, "bf16"),
    ((2, 3, 161, 64), torch.float32, "tf32"),
    ((2, 2, 70, 32), torch.float32, "ieee"),
    ((2, 3, 65, 64), torch.float16, "bf16"),
    ((1, 2, 65, 256), torch.bfloat16, "bf16"),
])
def test_training_on_views_equals_contiguous(layout, shape, dtype, prec):
    xs, dout = _inputs(shape, dtype)
    want = _train(*xs, dout, prec)
    got = _train(*(LAYOUTS[layout](x) for x in xs), LAYOUTS[layout](dout), prec)
    for w, g in zip(want, got):
        assert g.shape == w.shape and torch.equal(w, g)


@pytest.mark.gpu
def test_mixed_layouts_variants_and_expanded_dout():
    xs, dout = _inputs((2, 3, 200, 64), torch.bfloat16)
    want = _train(*xs, dout, "bf16")
    got = _train(LAYOUTS["packed"](xs[0]), xs[1], LAYOUTS["hbtd"](xs[2]), LAYOUTS["bthd"](dout), "bf16")
    assert all(torch.equal(w, g) for w, g in zip(want, got))
    # a loss that is a plain sum: dout of zero strides
    ones = torch.ones((), device="cuda").expand(2, 3, 200, 64)
    want = _train(*xs, ones.contiguous(), "bf16")
    got = _train(*(LAYOUTS["packed"](x) for x in xs), ones, "bf16")
    assert all(torch.equal(w, g) for w, g in zip(want, got))
    want = _train(*xs, dout, "bf16", kernels_bid, bid="relu")
    got = _train(*(LAYOUTS["packed"](x) for x in xs), LAYOUTS["packed"](dout), "bf16", kernels_bid, bid="relu")
    assert all(torch.equal(w, g) for w, g in zip(want, got))


@pytest.mark.gpu
@pytest.mark.parametrize("chunk,prec,dtype,dim", [(512, "bf16", torch.bfloat16, 64), (200, "bf16", torch.bfloat16, 64),
                                                  (96, "tf32", torch.float32, 64), (300, "bf16", torch.float16, 32)])
def test_prefill_on_views_writes_its_rows(chunk, prec, dtype, dim):
    """begin_cache on views of a projection: every chunk reads its queries
    where they lie and writes its rows of y, in y's type."""
    xs, _ = _inputs((2, 3, 700, dim), dtype)
    y, c = cache.begin_cache(*(LAYOUTS["packed"](x) for x in xs), capacity=750, chunk=chunk, dot_precision=prec)
    parts, ref = [], cache.alloc_cache(xs[1], xs[2], 750)
    for a in range(0, 700, chunk):
        b = min(a + chunk, 700)
        parts.append(kernels.dilution_prefill_chunk(xs[0][:, :, a:b].contiguous(), ref["k"], ref["v"],
                                                    ref["committed"], a, dot_precision=prec))
    assert y.dtype == dtype and y.is_contiguous()
    assert torch.equal(y, torch.cat(parts, dim=2).to(dtype))
    assert torch.equal(c["committed"], ref["committed"])


@pytest.mark.gpu
@pytest.mark.parametrize("layout", list(LAYOUTS))
@pytest.mark.parametrize("shape,bid", [((1, 4, 1, 64), "softmax"), ((1, 4, 1, 64), "relu"), ((1, 2, 1, 32), "sigmoid"),
                                       ((3, 1, 1, 64), "softplus"), ((1, 3, 1, 256), "softmax"), ((1, 1, 1, 16), "minshift")])
def test_one_row_has_no_stride(layout, shape, bid):
    """A call of one row takes views whatever torch says of the row's stride (a
    (1, H, 1, D) view of a projection is contiguous to torch and keeps the
    projection's): the variants and head_dim 256, which are built for rows
    head_dim apart, among them."""
    xs, dout = _inputs(shape, torch.bfloat16)
    ops, kw = (kernels, {}) if bid == "softmax" else (kernels_bid, {"bid": bid})
    want = _train(*xs, dout, "bf16", ops, **kw)
    got = _train(*(LAYOUTS[layout](x) for x in xs), LAYOUTS[layout](dout), "bf16", ops, **kw)
    for w, g in zip(want, got):
        assert g.shape == w.shape and torch.equal(w, g)


@pytest.mark.gpu
@pytest.mark.parametrize("dim,bid_kw", [(256, {}), (64, {"bid": "relu"})])
def test_one_row_prompts_and_chunks(dim, bid_kw):
    """begin_cache on a projection's views: a prompt of one token, and a last
    chunk of one row."""
    for seq, chunk in ((1, None), (1, 8), (9, 8)):
        if bid_kw and chunk:
            continue
        xs, _ = _inputs((1, 2, seq, dim), torch.bfloat16)
        want, c0 = cache.begin_cache(*xs, capacity=12, chunk=chunk, **bid_kw)
        got, c1 = cache.begin_cache(*(LAYOUTS["packed"](x) for x in xs), capacity=12, chunk=chunk, **bid_kw)
        assert torch.equal(got, want) and torch.equal(c0["committed"], c1["committed"])


@pytest.mark.gpu
@pytest.mark.parametrize("dim,bid", [(64, 1), (256, 0)])
def test_refused_rows_launch_nothing(dim, bid):
    """Strided rows where only the contiguous form is built are an argument
    error (-4) of the C ABI before any launch, forward and backward."""
    lib, n, t = _hip.lib(), 6, 40
    x = LAYOUTS["packed"](torch.randn(2, 3, t, dim, device="cuda").to(torch.bfloat16))
    flat = torch.empty(2, 3, t, dim, device="cuda", dtype=torch.bfloat16)
    f32 = [torch.empty(n * t * max(dim, 64), device="cuda") for _ in range(7)]
    ws = torch.empty(lib.dil_forward_workspace_bytes(n, t, dim, 1, 2, 1) + lib.dil_backward_workspace_bytes(n, t, dim, 1, 2),
                     dtype=torch.uint8, device="cuda")
    row, out, ptr = _rows(x), _rows(flat), [b.data_ptr() for b in f32]
    stream = torch.cuda.current_stream().cuda_stream
    with _hip.kernel_timing() as kt:
        forward = lib.dil_forward_rows(row, row, row, 2, 3, t, dim, 1, 2, bid, 1, 1.0, *ptr, ws.data_ptr(), ws.numel(), stream)
        backward = lib.dil_backward_rows(row, row, row, row, *ptr[:6], 2, 3, t, dim, 1, 1, 1, 2, bid, 1, 1.0, out, out, out,
                                         ws.data_ptr(), ws.numel(), stream)
    assert (forward, backward) == (-4, -4) and not kt.result
