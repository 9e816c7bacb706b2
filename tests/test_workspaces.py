"""The device workspaces that the Python layer keeps for decode and prefill: how they grow, who
shares them, and what a captured graph holds."""

import pytest
import torch

from kavor_amd.layers import attention, fused, workspace
from tests.helpers import bits_equal, gen, interleaved_pool, randn_bf16

pytestmark = pytest.mark.gpu
SCALE = 128 ** -0.5


KINDS = (attention._decode_workspaces, attention._prefill_pool, attention._split_pool, fused._argmax_pool)


@pytest.fixture
def fresh(cuda_device, monkeypatch):
    """Starts a test without workspaces; those of graphs captured earlier stay alive."""
    for kind in KINDS:
        for name in ("default", "side", "captured"):
            monkeypatch.setattr(kind, name, {})
    monkeypatch.setattr(workspace, "retired", [])
    return cuda_device


def _decode_args(d, B, hq, hkv, width, bs=256, seed=1):
    """Arguments of a decode of B one-page sequences under a block table of `width` pages."""
    g = gen(seed)
    kc, vc = (randn_bf16((4, bs, hkv, 128), g).to(d) for _ in range(2))
    bt = torch.zeros(B, width, dtype=torch.int32, device=d)
    ctx = torch.full((B,), 40, dtype=torch.int32, device=d)
    return randn_bf16((B, hq, 128), g).to(d), kc, vc, ctx, bt, SCALE


def _decode(*args):
    return attention.paged_decode(*_decode_args(*args))


def test_growing_step_by_step_retires_less_than_is_held(fresh):
    """Calls whose block tables widen page by page, then whose batches grow: the buffers that
    were outgrown add up to less than the one in use."""
    d = fresh
    for width in range(1, 129):
        _decode(d, 1, 64, 8, width)
    for batch in range(1, 65):
        _decode(d, batch, 64, 8, 36)
    held = attention._decode_workspaces.default[d.index].numel()
    assert sum(t.numel() for t in workspace.retired) < held
    need = attention.decode_workspace_bytes(64, 64, 128, 4 * 36, 256)
    assert need <= held <= 2 * need


def test_captures_that_grow_retire_less_than_is_held(fresh):
    """Graphs captured for ever larger batches, each after an eager call: the buffers that the
    smaller graphs keep add up to less than the last one."""
    d, graphs = fresh, []
    for batch in range(1, 33):
        _decode(d, batch, 64, 8, 4)
        args = _decode_args(d, batch, 64, 8, 4)
        graphs.append(torch.cuda.CUDAGraph())
        with torch.cuda.graph(graphs[-1]):
            attention.paged_decode(*args)
    held = attention._decode_workspaces.captured[d.index].numel()
    assert sum(t.numel() for t in workspace.retired) < held


def _reserve_all(d):
    return [attention.reserve_decode_workspace(4, 16, 128, 8, 256, d),
            attention.reserve_prefill_workspace(2, 300, 16, 8, d), fused.argmax_workspace(d)]


def test_streams_have_buffers_of_their_own(fresh):
    """Another stream's calls get another buffer, the same one each time; the streams that keep
    one are bounded."""
    d = fresh
    side = torch.cuda.Stream(d)
    mine = _reserve_all(d)
    with torch.cuda.stream(side):
        theirs = _reserve_all(d)
        again = _reserve_all(d)
    for a, b, c, e in zip(mine, theirs, again, _reserve_all(d)):
        assert a.data_ptr() != b.data_ptr() and b.data_ptr() == c.data_ptr() and a.data_ptr() == e.data_ptr()
    fused._argmax_pool.side = {(d.index, -n): mine[2] for n in range(1, 200)}  # streams that came and went
    with torch.cuda.stream(side):
        last = fused.argmax_workspace(d)
        assert len(fused._argmax_pool.side) == workspace._SIDE_STREAMS
        assert fused.argmax_workspace(d).data_ptr() == last.data_ptr()


def _prefill(d, num_seqs, new, keys, bs=256, max_seqlen_k=0, causal=True):
    """An eager prefill of num_seqs sequences, 16 query heads over 8, on one shared prefix."""
    g = gen(3)
    kc, vc = (randn_bf16((2, bs, 8, 128), g).to(d) for _ in range(2))
    bt = torch.zeros(num_seqs, -(-keys // bs), dtype=torch.int32, device=d)
    cu = torch.arange(num_seqs + 1, dtype=torch.int32, device=d)
    q = randn_bf16((num_seqs * new, 16, 128), g).to(d)
    return attention.varlen_prefill(q, kc, vc, new, cu * new, max_seqlen_k, cu * keys, SCALE, causal=causal,
                                    block_table=bt)


def test_partial_states_are_held_only_where_a_batch_may_be_split(fresh):
    """A launch of too many query tiles, one on few keys (by its table or by the stated length) and
    one without the causal mask hold a work list alone; the launches that may be split share one
    buffer of 69 MB."""
    d, split, lists = fresh, attention._split_pool, attention._prefill_pool
    _prefill(d, 33, 128, 2048)
    _prefill(d, 2, 100, 700)
    _prefill(d, 2, 100, 2048, max_seqlen_k=900)
    _prefill(d, 2, 100, 2048, causal=False)
    assert not split.default and lists.default[d.index].numel() <= 16384
    _prefill(d, 2, 100, 2048)
    held = split.default[d.index]
    assert held.numel() <= 70 << 20
    for n, new, keys in ((1, 1, 1024), (8, 512, 1024), (64, 60, 4096)):
        _prefill(d, n, new, keys)
        assert split.default[d.index] is held
    assert lists.default[d.index].numel() <= 16384


@pytest.mark.parametrize("heads", [(4, 8), (24, 8), (256, 1), (8, 0)])
def test_head_counts_without_a_kernel_are_still_refused(fresh, heads):
    hq, hkv = heads
    q = torch.zeros(8, hq, 128, dtype=torch.bfloat16, device=fresh)
    k = torch.zeros(8, hkv, 128, dtype=torch.bfloat16, device=fresh)
    cu = torch.tensor([0, 8], dtype=torch.int32, device=fresh)
    with pytest.raises(RuntimeError, match="kvp_varlen_prefill_bf16"):
        attention.varlen_prefill(q, k, k, 2000, cu, None, cu, SCALE)


def test_a_capture_takes_the_buffer_over(fresh):
    d = fresh
    args = _decode_args(d, 4, 16, 8, 8)
    mine = attention.reserve_decode_workspace(4, 16, 128, 8, 256, d)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        attention.paged_decode(*args)
    assert attention._decode_workspaces.captured[d.index].data_ptr() == mine.data_ptr()
    assert attention.reserve_decode_workspace(4, 16, 128, 8, 256, d).data_ptr() != mine.data_ptr()
    with pytest.raises(RuntimeError, match="reserved before graph capture"):
        big = _decode_args(d, 64, 64, 8, 64)
        with torch.cuda.graph(torch.cuda.CUDAGraph()):
            attention.paged_decode(*big)


def test_calls_on_two_streams_and_a_replay_at_once(fresh):
    """Decode with partial states, split prefill and split-row sampling, eagerly on two streams
    and as graph replays on a third, none ordered against the others: every output is the one
    that the call gives alone."""
    d, hkv, G, bs = fresh, 8, 2, 64
    g = gen(5)
    jobs = []
    for n in range(3):  # per stream: inputs of its own
        _, kc, vc = (t.to(d) for t in interleaved_pool(130, bs, hkv, 128, g))
        bt = torch.randperm(128, generator=g).to(torch.int32).view(2, 64).to(d)
        ctx = torch.tensor([4000 - 700 * n, 900 + 500 * n], dtype=torch.int32, device=d)
        q, qp = randn_bf16((2, G * hkv, 128), g).to(d), randn_bf16((90, G * hkv, 128), g).to(d)
        cq = torch.tensor([0, 40 + 9 * n, 90], dtype=torch.int32, device=d)
        ck = torch.tensor([0, 3000 + 300 * n, 6500], dtype=torch.int32, device=d)
        logits = randn_bf16((4, 32000), g, 3.0).to(d)

        def job(q=q, qp=qp, kc=kc, vc=vc, ctx=ctx, bt=bt, cq=cq, ck=ck, logits=logits):
            return (attention.paged_decode(q, kc, vc, ctx, bt, SCALE),
                    attention.varlen_prefill(qp, kc, vc, 80, cq, 0, ck, SCALE, block_table=bt),
                    fused.greedy_argmax(logits))

        jobs.append(job)
    want = [[t.clone() for t in job()] for job in jobs]
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        replayed = jobs[2]()
    streams = [torch.cuda.default_stream(d), torch.cuda.Stream(d), torch.cuda.Stream(d)]
    torch.cuda.synchronize()
    outs = []
    for _ in range(40):
        for n in (0, 1):
            with torch.cuda.stream(streams[n]):
                outs.append((n, jobs[n]()))
        with torch.cuda.stream(streams[2]):
            graph.replay()
            outs.append((2, [t.clone() for t in replayed]))
    torch.cuda.synchronize()
    for n, got in outs:
        for a, b in zip(got, want[n]):
            assert torch.equal(a, b) if a.dtype == torch.int64 else bits_equal(a, b)
