"""Slices of short contexts take the decode step in one workgroup (dec_one,
one_max_keys); longer ones in chunks.

Outputs and demand against an fp64 evaluation of the step on the kernel's
inputs, on both sides of the limit of each row of the rule, and the
device-resident length's bits against the host length's there.  Tolerances:
the output is a share-weighted mean of v (|v| < 6), its terms and sums in fp32
with hardware exp2 and reciprocal: 1e-5 relative per share, so 1e-4 max-abs,
plus half a unit in the last place of 16-bit outputs (2^-9 relative of 6); the
demand adds one p <= 1 in fp32 to values below 4: 1e-5.
"""

from __future__ import annotations

import pytest
import torch

from gpu_helpers import needs_gpu

pytestmark = [pytest.mark.gpu, needs_gpu]


def _limit(n, dim, elt):
    """one_max_keys of the library."""
    key_bytes = 2 * dim * elt
    if n >= 512 or 160 <= n <= 256:
        return 16384
    if n > 256:
        return (768 << 10) // key_bytes
    return min(4096, (((256 + n) if elt == 4 else (272 + 3 * n)) << 10) // key_bytes)


def _case(n, length, dim, dtype, spare, seed):
    g = torch.Generator(device="cuda").manual_seed(seed)
    q1 = torch.randn(1, n, 1, dim, device="cuda", generator=g).to(dtype)
    kc, vc = (torch.randn(1, n, length + spare, dim, device="cuda", generator=g).to(dtype) for _ in range(2))
    c = torch.rand(1, n, length + spare, device="cuda", generator=g) * 3
    c[..., length - 1] = 0
    return q1, kc, vc, c


def _check(q1, kc, vc, c0, length, out, c):
    n, dim = q1.shape[1], q1.shape[-1]
    for s in sorted({0, n // 2, n - 1}):
        q, k, v = q1[0, s, 0].double(), kc[0, s, :length].double(), vc[0, s, :length].double()
        p = ((k * q).sum(-1) / dim ** 0.5).softmax(0)
        cm = c0[0, s, :length].double()
        share = p / (cm + p + 1e-9)
        want = (share[:, None] * v).sum(0) / (share.sum() + 1e-9)
        tol = 1e-4 + (0.0 if out.dtype == torch.float32 else 6 * 2.0 ** -9)
        assert (out[0, s].reshape(-1).double() - want).abs().max() < tol, (s, length)
        assert (c[0, s, :length].double() - (cm + p)).abs().max() < 1e-5, (s, length)
    assert torch.equal(c[..., length:], c0[..., length:])


@pytest.mark.parametrize("dim,dtype", [(16, torch.bfloat16), (32, torch.float16), (64, torch.bfloat16),
                                       (64, torch.float32), (128, torch.bfloat16), (256, torch.float32)])
@pytest.mark.parametrize("n", [1, 159, 160, 257])
def test_both_sides_of_the_limit(n, dim, dtype):
    from dilution import kernels

    limit = _limit(n, dim, 4 if dtype == torch.float32 else 2)
    lengths = [1, 65, 1025, limit, limit + 1] if limit < 16384 else [1, 65, 1025, 3000]
    for length in lengths:
        q1, kc, vc, c0 = _case(n, length, dim, dtype, 3, length)
        c_host, c_dev = c0.clone(), c0.clone()
        out = kernels.dilution_decode_step(q1, kc, vc, c_host, length)
        _check(q1, kc, vc, c0, length, out, c_host)
        # the live length in device memory, with room for more
        got = kernels.decode_step_device_length(q1, kc, vc, c_dev, torch.tensor([length], device="cuda"), length + 3)
        assert torch.equal(got.reshape(-1), out.reshape(-1)) and torch.equal(c_dev, c_host), length


def test_largest_context_in_one_workgroup():
    from dilution import kernels

    for length in (16384, 16385):
        q1, kc, vc, c0 = _case(160, length, 64, torch.bfloat16, 40, length)
        c_host, c_dev = c0.clone(), c0.clone()
        out = kernels.dilution_decode_step(q1, kc, vc, c_host, length)
        _check(q1, kc, vc, c0, length, out, c_host)
        got = kernels.decode_step_device_length(q1, kc, vc, c_dev, torch.tensor([length], device="cuda"), length + 40)
        assert torch.equal(got.reshape(-1), out.reshape(-1)) and torch.equal(c_dev, c_host)


def test_masked_affinities_and_zero_length():
    """Keys whose affinity is -inf take no share and leave the demand as it is;
    a live length of 0 writes zeros and nothing else."""
    from dilution import kernels

    q1, kc, vc, c0 = _case(4, 700, 64, torch.float32, 0, 9)
    q1[..., 0] = 1.0
    kc[:, :, 100:600, 0] = float("-inf")
    c = c0.clone()
    out = kernels.dilution_decode_step(q1, kc, vc, c, 700)
    keep = torch.cat([torch.arange(100), torch.arange(600, 700)]).cuda()
    c_part = c0[..., keep].contiguous()
    want = kernels.dilution_decode_step(q1, kc[:, :, keep].contiguous(), vc[:, :, keep].contiguous(), c_part, 200)
    assert (out - want).abs().max() < 1e-4
    assert torch.equal(c[..., 100:600], c0[..., 100:600])
    assert (c[..., keep] - c_part).abs().max() < 1e-5
    for cap in (500, 700):
        c = c0.clone()
        got = kernels.decode_step_device_length(q1, kc, vc, c, torch.tensor([0], device="cuda"), cap)
        assert (got == 0).all() and torch.equal(c, c0)


@pytest.mark.parametrize("n,length,room", [(160, 2000, 20000), (9, 65, 70000), (3, 1, 300), (65, 1025, 4096), (257, 600, 33000)])
def test_short_live_length_under_a_long_maximum(n, length, room):
    """A graph's grid has a workgroup per slice and chunk of the longest length;
    the first ones take a slice each when the live length is short: every slice
    once, with the bits of the host length's step."""
    from dilution import kernels

    q1, kc, vc, c0 = _case(n, length, 32, torch.bfloat16, 3, length)
    kc, vc = (torch.cat([x, x.new_zeros(1, n, room - x.shape[2], 32)], dim=2) for x in (kc, vc))
    c0 = torch.cat([c0, c0.new_zeros(1, n, room - c0.shape[2])], dim=2)
    c_host, c_dev = c0.clone(), c0.clone()
    want = kernels.dilution_decode_step(q1, kc, vc, c_host, length)
    _check(q1, kc, vc, c0, length, want, c_host)
    got = kernels.decode_step_device_length(q1, kc, vc, c_dev, torch.tensor([length], device="cuda"), room)
    assert torch.equal(got.reshape(-1), want.reshape(-1)) and torch.equal(c_dev, c_host)


@pytest.mark.parametrize("n,dim,dtype,limit", [(513, 64, torch.bfloat16, 4096), (623, 64, torch.float32, 2048),
                                               (624, 16, torch.bfloat16, 16384), (770, 128, torch.bfloat16, 4096),
                                               (1039, 32, torch.float16, 16384), (300, 16, torch.bfloat16, 12288)])
def test_partial_last_round_of_workgroups(n, dim, dtype, limit):
    """More than one round of 256 workgroups with a last one that leaves more
    than 3/16 of their places empty: at most 768 KiB, 1 MiB (three rounds) or 2 MiB
    of K and V a slice."""
    from dilution import kernels

    for length in (33, limit, limit + 1):
        q1, kc, vc, c0 = _case(n, length, dim, dtype, 1, length)
        c_host, c_dev = c0.clone(), c0.clone()
        out = kernels.dilution_decode_step(q1, kc, vc, c_host, length)
        _check(q1, kc, vc, c0, length, out, c_host)
        got = kernels.decode_step_device_length(q1, kc, vc, c_dev, torch.tensor([length], device="cuda"), length + 1)
        assert torch.equal(got.reshape(-1), out.reshape(-1)) and torch.equal(c_dev, c_host)
