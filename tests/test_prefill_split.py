"""Prefill of few query tiles on long keys, whose key ranges the launch cuts into chunks
(prefill_split_plan_kernel, prefill_merge_kernel), against the fp32 oracle and against the
uncut launch, which a workspace without the split area gives.

An average of thousands of N(0, 1) values is small, so a fixed tolerance would pass a merge that
weighs its chunks wrongly.  The keys' scale therefore changes every 300 tokens (their scores'
maxima differ by many units, and so do the chunks' weights), the values carry a constant that
changes every 200, and outputs are compared within a bound of their own: the kernel rounds each
weight p of a key and the output to bf16 (8 significant bits: 2^-8 relative at most) and keeps
all sums in fp32, so an output sum(p v) is within 2^-8 sum(p |v|) + 2^-8 |sum(p v)| <=
2^-7 sum(p |v|) of the exact one; 1e-4 beside it covers the fp32 sums of both sides (values and
constants are below 8).  A merge that weighs its chunks alike is 15 to 75 times further off,
one that loses a chunk of a thirtieth of the weight 4 times.
"""

import itertools
import math

import pytest
import torch

from kavor_amd import _lib
from kavor_amd.layers import attention
from oracle import kvpath_oracle as ref
from tests.helpers import bits_equal, gen, interleaved_pool, randn_bf16

pytestmark = pytest.mark.gpu
SCALE = 128 ** -0.5


def _cu(lens):
    return torch.tensor([0] + list(itertools.accumulate(lens)), dtype=torch.int32)


def _check(out, q, k, v, cq, ck, bt=None):
    """out against the oracle within 2^-7 sum(p |v|) (see above)."""
    want, weight = (ref.varlen_prefill(q, k, x, cq, ck, SCALE, block_tables=bt).cpu() for x in (v, v.abs()))
    err = (out.cpu().float() - want).abs()
    assert bool((err <= 2.0 ** -7 * weight + 1e-4).all()), float((err / (weight + 1e-4)).max() * 128)


def _uneven(k, v, t):
    """k and v [n, heads, 128] of the tokens t: scales and constants that change along the keys."""
    scale = 0.2 + 0.7 * ((t // 300) * 5 % 4).float()
    shift = ((t // 200) * 3 % 5 - 2).float()
    return (k * scale[:, None, None]).to(torch.bfloat16), (v + shift[:, None, None]).to(torch.bfloat16)


def _paged(seed, qlens, prefixes, G, hkv, bs):
    g = gen(seed)
    klens = [a + b for a, b in zip(qlens, prefixes)]
    need = [math.ceil(k / bs) for k in klens]
    nb = sum(need) + 2
    _, kc, vc = interleaved_pool(nb, bs, hkv, 128, g)
    ids = torch.randperm(nb, generator=g).tolist()
    bt = torch.full((len(qlens), max(need)), -1, dtype=torch.int32)
    for s, n in enumerate(need):
        bt[s, :n] = torch.tensor(ids[:n], dtype=torch.int32)
        ids = ids[n:]
        if n:
            rows = bt[s, :n].long()
            k, v = _uneven(kc[rows].view(-1, hkv, 128), vc[rows].view(-1, hkv, 128), torch.arange(n * bs))
            kc[rows], vc[rows] = k.view(n, bs, hkv, 128), v.view(n, bs, hkv, 128)
    return randn_bf16((sum(qlens), G * hkv, 128), g), kc, vc, bt, _cu(qlens), _cu(klens)


def _run(dev, q, k, v, bt, cq, ck, max_q):
    out = attention.varlen_prefill(*(t.to(dev) for t in (q, k, v)), max_q, cq.to(dev), 0, ck.to(dev), SCALE,
                                   causal=True, block_table=None if bt is None else bt.to(dev))
    torch.cuda.synchronize()
    return out.cpu()


def _launch(dev, q, k, v, bt, cq, ck, max_q, split=True):
    """The C entry point in a workspace with or without the split area: the output, and the
    split plan's units and cut tiles (None: the launch was not a split one)."""
    lib = _lib.lib()
    n, (Tq, hq, D), hkv = cq.numel() - 1, q.shape, k.shape[-2]
    plain = lib.kvp_prefill_workspace_bytes(n, max_q, hq, hkv)
    size = lib.kvp_prefill_split_workspace_bytes(n, max_q, hq, hkv) if split else plain
    ws = torch.full((size,), 0xFF, dtype=torch.uint8, device=dev)
    q, k, v, cq, ck = (t.to(dev) for t in (q, k, v, cq, ck))
    out = torch.empty_like(q)
    if bt is None:
        ks, vs, table = (0, k.stride(0), k.stride(1)), (0, v.stride(0), v.stride(1)), (0, 0, 0, 0, 0)
    else:
        bt = bt.to(dev)
        ks, vs = k.stride()[:3], v.stride()[:3]
        table = bt.data_ptr(), bt.stride(0), k.shape[0], k.shape[1], bt.shape[1]
    _lib.check("prefill", lib.kvp_varlen_prefill_bf16(
        q.data_ptr(), q.stride(0), q.stride(1), k.data_ptr(), *ks, v.data_ptr(), *vs, *table, cq.data_ptr(),
        ck.data_ptr(), n, max_q, hq, hkv, D, SCALE, 1, out.data_ptr(), out.stride(0), out.stride(1), ws.data_ptr(),
        size, torch.cuda.current_stream(dev).cuda_stream))
    torch.cuda.synchronize()
    at = -(-plain // 256) * 256  # the split area: unit and cut counts, from int 64 the units, 8 ints each
    area = ws[at:at + 4 * (64 + 8 * 1024)].view(torch.int32).tolist() if split else [-1]
    if area[0] < 0:
        return out.cpu(), None, None
    return out.cpu(), [area[64 + 8 * i:72 + 8 * i] for i in range(area[0] // hkv)], area[1]


CASES = [
    # one tile on many keys, one row past a tile, a tile of one row; chunks off block borders
    (2, 8, 256, [64], [4000]), (2, 8, 64, [65], [1500]), (4, 8, 192, [1], [3000]),
    # ragged turns, an empty sequence, a short one beside long ones
    (4, 8, 256, [300, 17, 0, 158], [6000, 2048, 700, 5]), (5, 8, 64, [100, 30], [2500, 64]),
    (8, 4, 64, [70, 33], [1111, 4096]), (1, 4, 256, [200, 129], [1024, 0]),
    # no prefix: causal tiles of 1 .. n key tiles, some cut and some not
    (2, 8, 256, [1500], [0]), (2, 2, 64, [2100, 700], [0, 900]),
]


@pytest.mark.parametrize("G,hkv,bs,qlens,prefixes", CASES)
def test_split_paged_matches_oracle(cuda_device, G, hkv, bs, qlens, prefixes):
    args = _paged(40 + G + len(qlens), qlens, prefixes, G, hkv, bs)
    q, kc, vc, bt, cq, ck = args
    d = cuda_device
    out, units, cuts = _launch(d, *args, max(qlens))
    assert cuts > 0 and len(units) > cuts
    dev = [t.to(d) for t in (q, kc, vc)]
    _check(out, *dev, cq, ck, bt.to(d))
    uncut, units, _ = _launch(d, *args, max(qlens), split=False)
    assert units is None
    _check(uncut, *dev, cq, ck, bt.to(d))
    assert bits_equal(_run(d, *args, max(qlens)), out)  # the Python layer takes the split launch


def test_split_dense_matches_oracle(cuda_device):
    g, d = gen(60), cuda_device
    qlens, hkv, G = [1400, 321], 8, 2
    cu = _cu(qlens)
    q, k, v = (randn_bf16((sum(qlens), h, 128), g) for h in (G * hkv, hkv, hkv))
    k, v = _uneven(k, v, torch.cat([torch.arange(n) for n in qlens]))
    out, _, cuts = _launch(d, q, k, v, None, cu, cu, max(qlens))
    assert cuts > 0
    dev = [t.to(d) for t in (q, k, v)]
    _check(out, *dev, cu, cu)
    _check(_launch(d, q, k, v, None, cu, cu, max(qlens), split=False)[0], *dev, cu, cu)


def test_split_understated_max_seqlen_and_rows_without_keys(cuda_device):
    """A sequence longer than max_seqlen_q is computed in full (its units stride over tiles);
    rows before the first key (more queries than keys) are zeros; a bad block id poisons its
    own sequence only."""
    qlens, klens, bs, hkv, G = [500, 90, 40], [3000, 50, 2000], 64, 8, 2
    q, kc, vc, bt, cq, ck = _paged(70, qlens, [k - a for a, k in zip(qlens, klens)], G, hkv, bs)
    bt[2, 20] = 10 ** 6
    out, _, cuts = _launch(cuda_device, q, kc, vc, bt, cq, ck, 100)
    assert cuts > 0
    good = slice(0, 590)
    _check(out[good], q[good], kc, vc, cq[:3], ck[:3], bt[:2])
    assert torch.count_nonzero(out[500:540]) == 0
    assert torch.isnan(out[590:].float()).all()


def test_split_replays_in_a_graph(cuda_device):
    """Captured with one batch's lengths, replayed with others: plan, units and merge follow
    the lengths on the device."""
    d, hkv, G, bs, width = cuda_device, 8, 2, 64, 80
    g = gen(80)
    _, kc, vc, bt, _, _ = (None, *_paged(80, [1], [width * bs - 1], G, hkv, bs)[1:])
    kc, vc, bt = kc.to(d), vc.to(d), bt.to(d)
    q = randn_bf16((256, G * hkv, 128), g).to(d)
    cq, ck = torch.zeros(2, dtype=torch.int32, device=d), torch.zeros(2, dtype=torch.int32, device=d)
    out = torch.zeros_like(q)
    attention.reserve_prefill_workspace(1, 256, G * hkv, hkv, d)

    def call(o):
        return attention.varlen_prefill(q, kc, vc, 256, cq, 0, ck, SCALE, causal=True, block_table=bt, out=o)

    cq[1], ck[1] = 256, 4000
    call(out)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        call(out)
    for ql, kl in ((30, 5000), (256, 1200), (1, 64), (200, 4444)):
        cq[1], ck[1] = ql, kl
        out.fill_(float("nan"))
        torch.cuda.synchronize()
        graph.replay()
        torch.cuda.synchronize()
        got = out[:ql].clone()
        eager = call(torch.zeros_like(q))[:ql]
        torch.cuda.synchronize()
        assert torch.equal(got.view(torch.int16), eager.view(torch.int16))
        _check(got, q[:ql], kc, vc, cq, ck, bt)


def test_smaller_workspace_is_accepted_inside_a_capture(cuda_device, monkeypatch):
    """A workspace that holds the work list but no split area (reserved for a wide batch by an
    older caller) still serves a captured call, uncut."""
    d = cuda_device
    q, kc, vc, bt, cq, ck = (t.to(d) for t in _paged(90, [100], [2000], 2, 8, 64))
    base = attention.prefill_workspace_bytes(1, 100, 16, 8)
    assert _lib.lib().kvp_prefill_split_workspace_bytes(1, 100, 16, 8) > base
    for pool in (attention._prefill_pool, attention._split_pool):
        for name in ("default", "side", "captured"):
            monkeypatch.setattr(pool, name, {})
    attention._prefill_pool.default[d.index] = torch.empty(base, dtype=torch.uint8, device=d)
    out = torch.zeros_like(q)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        attention.varlen_prefill(q, kc, vc, 100, cq, 0, ck, SCALE, causal=True, block_table=bt, out=out)
    assert not attention._split_pool.captured
    for _ in range(2):
        graph.replay()
        torch.cuda.synchronize()
    _check(out, q, kc, vc, cq, ck, bt)


@pytest.mark.parametrize("qlens,prefixes", [([250] * 8, [1024] * 8), ([100] * 32, [2048] * 32),
                                            ([500, 490, 450, 500], [512] * 4), ([1300] * 3, [0] * 3)])
def test_neighbouring_tiles_rank_side_by_side(cuda_device, qlens, prefixes):
    """Where the plan cuts nothing, tiles 2j and 2j + 1 of a sequence follow each other in its list,
    as the pairs of an uncut launch do, so that they are claimed one after the other on one XCD
    and read their keys together."""
    q, kc, vc, bt, cq, ck = _paged(33, qlens, prefixes, 2, 8, 64)
    _, units, cuts = _launch(cuda_device, q, kc, vc, bt, cq, ck, max(qlens))
    assert cuts == 0
    at = {(s, tile): i for i, (s, tile, *_) in enumerate(units)}
    assert len(at) == len(units) and sorted(at) == [(s, t) for s, n in enumerate(qlens) for t in range(-(-n // 64))]
    for (s, tile), i in at.items():
        if (s, tile ^ 1) in at:
            assert abs(at[s, tile ^ 1] - i) == 1, (s, tile)


def test_a_batch_bound_by_its_keys_arrival_is_not_cut(cuda_device):
    """32 one-tile sequences on 33 key tiles of their own: two chunks each would fit the workgroup
    slots, but the K/V take longer to arrive than the longest unit to compute."""
    args = _paged(34, [60] * 32, [2048] * 32, 2, 8, 256)
    _, units, cuts = _launch(cuda_device, *args, 60)
    assert cuts == 0 and len(units) == 32
    _, units, cuts = _launch(cuda_device, *_paged(35, [60] * 8, [2048] * 8, 2, 8, 256), 60)
    assert cuts == 8 and len(units) > 16
