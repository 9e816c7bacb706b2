"""Paged decode at the edges of its work split and of its LDS tiles, against the fp32 oracle:
contexts around the 32-token step and the 16-token half, pages whose size is not a power of
two, more sequences than one launch's tables hold, row strides beyond 32-bit offsets, and
values that a split of the softmax weights into parts could spoil (infinities in V).

Tolerance (TOL, atol 2e-2): outputs are bf16 averages of up to some hundred N(0, 1) values,
|o| < 4, whose rounding is at most 2^-7; the fp32 sums and the exact three-part weights add
below 1e-4.  Longer contexts, whose averages are small, take a tolerance of their own.
"""

import math

import pytest
import torch

from oracle import kvpath_oracle as ref
from oracle import layers_oracle as lref
from tests.helpers import TOL, contiguous_caches, gen, random_block_tables, randn_bf16
from tests.test_fused_decode import _case as fused_case, _fused, _separate
from tests.test_paged_decode import SCALE, _case as decode_case, _check, _decode

pytestmark = pytest.mark.gpu

EDGES = [1, 15, 16, 17, 31, 32, 33, 63, 64, 65, 95, 96, 97, 127, 128, 129, 191, 192, 193, 383, 385]


@pytest.mark.parametrize("G", [1, 2, 4, 5, 8])
@pytest.mark.parametrize("bs", [64, 192])
def test_step_and_page_edges(cuda_device, G, bs):
    g = gen(700 + G + bs)
    hkv = 3 if G < 8 else 5  # waves past the last kv head, one and two head groups
    nb = sum(math.ceil(c / bs) for c in EDGES) + 2
    kc, vc = contiguous_caches(nb, bs, hkv, 128, g)
    bt = random_block_tables(EDGES, bs, nb, g)
    q = randn_bf16((len(EDGES), G * hkv, 128), g)
    _check(cuda_device, q, kc, vc, bt, torch.tensor(EDGES, dtype=torch.int32))


@pytest.mark.parametrize("steps", [2, 4, 5, 19, 20, 21, 100])
def test_one_sequence_in_many_ranges(cuda_device, steps):
    """A lone sequence is cut into short ranges, one step each where the table is as wide as four
    times its context: their states merge in rounds of 4 and 16.  Step r alone has a value in dim
    r, of size `steps`, so that a step lost or weighed wrongly changes that dim by its weight, of
    order 1: |o| is a few units, rounded to bf16 (2^-8 at most), on noise of 0.05 / sqrt(tokens)."""
    bs, hkv, G, ctx = 64, 2, 4, 32 * steps - 5
    g, n = gen(900 + steps), -(-ctx // bs)
    kc, vc = contiguous_caches(n, bs, hkv, 128, g)
    vc.mul_(0.05)
    at = torch.arange(n * bs)
    vc.view(-1, hkv, 128)[at, :, at // 32] = float(steps)
    bt = torch.full((1, 4 * n), -1, dtype=torch.int32)
    bt[0, :n] = torch.arange(n)
    q, lens, d = randn_bf16((1, G * hkv, 128), g), torch.tensor([ctx], dtype=torch.int32), cuda_device
    out = _decode(q.to(d), kc.to(d), vc.to(d), lens.to(d), bt.to(d)).cpu().float()
    want = ref.paged_decode(q, kc, vc, bt, lens, SCALE)
    assert bool((want[..., :steps] > 0.02).all())
    torch.testing.assert_close(out, want, atol=2e-3, rtol=5e-3)


@pytest.mark.parametrize("G", [1, 2, 4, 5, 8])
def test_one_launch_step_at_the_edges(cuda_device, G):
    """Append, q and attention of the one-launch step where the new token opens, fills or
    closes a step, a page or a range."""
    hkv, bs = 3, 64
    host, d1 = fused_case(cuda_device, 800 + G, G * hkv, hkv, bs, EDGES, pad=2)
    d2 = {k: v.clone() for k, v in d1.items()}
    sep, one = _separate(d1, G * hkv, hkv, bs), _fused(d2, G * hkv, hkv, bs)
    torch.cuda.synchronize()
    assert torch.equal(d1["pool"].cpu(), d2["pool"].cpu())
    torch.testing.assert_close(one.cpu().float(), sep.cpu().float(), **TOL)


def test_more_sequences_than_one_launch(cuda_device):
    B, hkv, bs = 1030, 2, 64
    g = gen(9)
    ctx = torch.randint(0, 90, (B,), generator=g, dtype=torch.int32)
    nb = sum(math.ceil(int(c) / bs) for c in ctx) + 2
    kc, vc = contiguous_caches(nb, bs, hkv, 128, g)
    bt = random_block_tables([int(c) for c in ctx], bs, nb, g)
    _check(cuda_device, randn_bf16((B, 4 * hkv, 128), g), kc, vc, bt, ctx)


@pytest.mark.parametrize("G,hkv,B", [(1, 32, 2300), (2, 32, 2300), (8, 8, 2100)])
def test_many_short_sequences_per_wave(cuda_device, G, hkv, B):
    """More sequences than a wave's window of 64 holds and than a launch's tables, with runs of
    empty ones across the windows' borders.  All sequences share eight pages."""
    g, bs = gen(12 + G), 64
    ctx = torch.randint(0, 41, (B,), generator=g, dtype=torch.int32)
    ctx[100:300] = 0
    ctx[1000:1064] = 0
    ctx[B - 70:] = 0
    kc, vc = contiguous_caches(8, bs, hkv, 128, g)
    bt = torch.randint(0, 8, (B, 1), generator=g, dtype=torch.int32)
    d = cuda_device
    q = randn_bf16((B, G * hkv, 128), g)
    out = _decode(q.to(d), kc.to(d), vc.to(d), ctx.to(d), bt.to(d)).cpu().float()
    # all pages' keys at once, masked per sequence: [B, heads, 8 * bs]
    qd, kd, vd = q.to(d).float(), kc.to(d).float(), vc.to(d).float()
    s = torch.stack([torch.mm(qd[:, h], kd[:, :, h // G].reshape(-1, 128).t().contiguous()) for h in range(G * hkv)], 1)
    at = torch.arange(8 * bs, device=d)
    seen = (at[None] // bs == bt.to(d)) & (at[None] % bs < ctx.to(d)[:, None])
    w = torch.softmax((s * SCALE).masked_fill(~seen[:, None], -math.inf), -1).nan_to_num(0.0)
    want = torch.stack([torch.mm(w[:, h], vd[:, :, h // G].reshape(-1, 128)) for h in range(G * hkv)], 1)
    torch.testing.assert_close(out, want.cpu(), **TOL)
    assert torch.count_nonzero(out[ctx == 0]) == 0


@pytest.mark.parametrize("G,hkv,B", [(1, 32, 2300), (2, 32, 1500), (8, 8, 1100)])
def test_one_launch_step_of_many_short_sequences(cuda_device, G, hkv, B):
    """The same for the one-launch step, against the separate launches: a page per sequence."""
    d, g, hq, bs = cuda_device, gen(40 + G), G * hkv, 64
    ctx = torch.randint(1, 41, (B,), generator=g, dtype=torch.int32)
    ctx[90:170] = 0
    pages = torch.randperm(B, generator=g).to(torch.int32)
    slots = torch.where(ctx > 0, pages * bs + ctx - 1, -1)
    dg = torch.Generator(device=d).manual_seed(G)

    def rand(*shape):
        return torch.randn(*shape, generator=dg, device=d, dtype=torch.bfloat16)

    d1 = dict(pool=rand(B, 2 * bs * hkv * 128).view(torch.uint8), qkv=rand(B, (hq + 2 * hkv) * 128), qw=rand(128),
              kw=rand(128), table=lref.rope_table(128, 64, 1e6).to(d), bt=pages[:, None].contiguous().to(d),
              ctx=ctx.to(d), pos=(ctx - 1).clamp(min=0).to(d), slots=slots.to(torch.int32).to(d))
    d2 = {k: v.clone() for k, v in d1.items()}
    sep, one = _separate(d1, hq, hkv, bs), _fused(d2, hq, hkv, bs)
    torch.cuda.synchronize()
    assert torch.equal(d1["pool"], d2["pool"])
    torch.testing.assert_close(one.float(), sep.float(), **TOL)
    assert torch.count_nonzero(one[90:170]) == 0


def test_strides_beyond_32_bit_offsets(cuda_device):
    """Token rows and q heads further apart than 32 rows of 32-bit byte offsets reach: the
    tiles are filled through registers and give the same bits."""
    g, d = gen(10), cuda_device
    hkv, G, bs, far = 1, 2, 64, (1 << 24) + 8
    kc, vc = contiguous_caches(1, bs, hkv, 128, g)
    q = randn_bf16((1, G, 128), g)
    ctx, bt = torch.tensor([61], dtype=torch.int32), torch.zeros(1, 1, dtype=torch.int32)
    near = _decode(q.to(d), kc.to(d), vc.to(d), ctx.to(d), bt.to(d))
    big = [torch.empty(bs * far, dtype=torch.bfloat16, device=d).as_strided((1, bs, hkv, 128), (bs * far, far, 128, 1))
           for _ in range(2)]
    big[0].copy_(kc)
    big[1].copy_(vc)
    qf = torch.empty(G * far, dtype=torch.bfloat16, device=d).as_strided((1, G, 128), (G * far, far, 1))
    qf.copy_(q)
    out = _decode(qf, big[0], big[1], ctx.to(d), bt.to(d))
    torch.cuda.synchronize()
    assert torch.equal(out.view(torch.int16), near.view(torch.int16))


@pytest.mark.parametrize("G", [2, 5, 8])
def test_infinite_values_stay_infinite(cuda_device, G):
    """An infinity in V gives that infinity (a weight's lower parts times it are inf - inf),
    and touches no other dim."""
    g, d = gen(11), cuda_device
    hkv, bs = 2, 64
    ctx = torch.tensor([50, 40], dtype=torch.int32)
    kc, vc = contiguous_caches(3, bs, hkv, 128, g)
    vc[1, 20, 0, 5] = float("inf")
    vc[1, 21, 1, 77] = float("-inf")
    bt = torch.tensor([[1], [2]], dtype=torch.int32)
    q = randn_bf16((2, G * hkv, 128), g)
    out = _decode(q.to(d), kc.to(d), vc.to(d), ctx.to(d), bt.to(d)).cpu().float()
    want = ref.paged_decode(q, kc, vc, bt, ctx, SCALE)
    assert torch.equal(torch.isinf(out), torch.isinf(want)) and not torch.isnan(out).any()
    assert torch.all(out[0, :G, 5] == float("inf")) and torch.all(out[0, G:, 77] == float("-inf"))
    fin = torch.isfinite(want)
    torch.testing.assert_close(out[fin], want[fin], **TOL)


@pytest.mark.parametrize("G", [1, 2, 4, 5, 8])
def test_infinity_in_the_last_token(cuda_device, G):
    """Rows of a step past the context carry weight 0; an infinity in the context's last token
    stays that infinity in its own dim and touches no other, from both entry points."""
    hkv, bs, ctxs = 2, 64, [1, 17, 31, 32, 33, 48, 63, 64, 80, 129]
    hq = G * hkv
    host, d = fused_case(cuda_device, 820 + G, hq, hkv, bs, ctxs)
    v = host["qkv"].view(len(ctxs), hq + 2 * hkv, 128)[:, hq + hkv:]
    v[:, 0, 9], v[:, 1, 100] = float("inf"), float("-inf")
    d["qkv"].copy_(host["qkv"])
    d2 = {k: t.clone() for k, t in d.items()}
    for out in (_separate(d, hq, hkv, bs), _fused(d2, hq, hkv, bs)):
        out = out.cpu().float()
        want = torch.zeros(out.shape)
        want[:, :G, 9], want[:, G:, 100] = float("inf"), float("-inf")
        assert torch.equal(torch.where(torch.isfinite(out), 0.0, out), want)
