"""HIP-graph capture of the operators.

* Replays of captured ring-share, distributed-KV decode, key-split prefill and layer-op calls
  equal the eager results on every replay, with eager work on the device between the
  replays (the kernels write every scratch value they read in the same call and record no
  memset).
* The operators' scratch: what a capture recorded belongs to its graph, so replays never write
  into memory the allocator has handed out again, graphs captured on one stream can be replayed
  on two, and calls of two threads on one stream do not share it.
"""

import threading

import pytest
import torch

pytestmark = pytest.mark.gpu


def _attn_inputs(dev, s, seed, hq=4, hkv=2, d=128):
    g = torch.Generator().manual_seed(seed)
    q = torch.randn(1, s, hq, d, generator=g).to(torch.bfloat16).to(dev)
    k = torch.randn(1, s, hkv, d, generator=g).to(torch.bfloat16).to(dev)
    v = torch.randn(1, s, hkv, d, generator=g).to(torch.bfloat16).to(dev)
    pos = torch.arange(s).view(1, s).to(dev)
    return q, k, v, pos


def test_captured_workspace_survives_growth(cea, dev):
    s = torch.cuda.Stream(dev)
    q, k, v, pos = _attn_inputs(dev, 256, 1)
    bq, bk, bv, bpos = _attn_inputs(dev, 16384, 2)  # 256 tiles: more scratch
    with torch.cuda.stream(s):
        ref_o, ref_l = cea.attention_with_lse(q, k, v, pos, pos)
    s.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=s):
        out, lse = cea.attention_with_lse(q, k, v, pos, pos)
    with torch.cuda.stream(s):
        cea.attention_with_lse(bq, bk, bv, bpos, bpos)
        fillers = [torch.full((4096,), 7, dtype=torch.uint8, device=dev) for _ in range(32)]
    s.synchronize()
    for i in range(3):
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, ref_o) and torch.equal(lse, ref_l), f"replay {i}"
        assert all(bool((f == 7).all()) for f in fillers), f"replay {i} wrote into reused memory"
        with torch.cuda.stream(s):
            cea.attention_with_lse(bq, bk, bv, bpos, bpos)
        s.synchronize()


def _replays_match(fn, eager_work, n=3):
    """Captures fn() (a tuple of tensors), replays it n times with eager_work() between the
    replays, and checks every replay against the eager result."""
    ref = [t.clone() for t in fn()]
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        outs = fn()
    for i in range(n):
        for t in outs:
            t.fill_(0)
        graph.replay()
        torch.cuda.synchronize()
        for a, b in zip(outs, ref):
            assert torch.equal(a, b), f"replay {i}"
        eager_work()
        torch.cuda.synchronize()


def test_ring_share_replays(cea, dev):
    g = torch.Generator().manual_seed(3)
    sizes, hq, hkv, d = [300, 257, 64, 1000], 8, 2, 128
    group, start = cea.LocalGroup(len(sizes), 1), 0
    for r, n in enumerate(sizes):
        k = torch.randn(1, n, hkv, d, generator=g).to(torch.bfloat16).to(dev)
        v = torch.randn(1, n, hkv, d, generator=g).to(torch.bfloat16).to(dev)
        group.set_shard(r, k=k, v=v, pos=torch.arange(start, start + n).view(1, n).to(dev))
        start += n
    own = group.shard(1)
    q = torch.randn(1, sizes[1], hq, d, generator=g).to(torch.bfloat16).to(dev)

    def share():
        out, lse = cea.sequence_parallel.ring_attention_with_lse(
            q, own["k"], own["v"], own["pos"], own["pos"], group, sizes)
        plain = cea.ring_attention(q, own["k"], own["v"], own["pos"], own["pos"], group, sizes)
        return out, lse, plain

    bq, bk, bv, bpos = _attn_inputs(dev, 4096, 4)
    _replays_match(share, lambda: cea.attention_with_lse(bq, bk, bv, bpos, bpos))


def test_distributed_kv_decode_replays(cea, dev):
    w = cea.workloads.kv_decode(device=dev, batch=[0, 5, 9, 30], cap=4096, min_len=64)
    parts = w.partitions()

    def step():
        out, lse = cea.partitioned_attention(w.q, w.q_pos, parts, return_lse=True)
        return out, lse, cea.partitioned_attention(w.q, w.q_pos, parts)

    bq, bk, bv, bpos = _attn_inputs(dev, 2048, 5)
    _replays_match(step, lambda: cea.attention_with_lse(bq, bk, bv, bpos, bpos))


def test_layer_ops_replays(cea, dev):
    g = torch.Generator().manual_seed(6)
    x = torch.randn(64, 1024, generator=g).to(torch.bfloat16).to(dev)
    w = (1 + 0.02 * torch.randn(1024, generator=g)).to(torch.bfloat16).to(dev)
    pos = torch.arange(64).to(dev)
    inv = cea.layers.rope_inv_freq(128, 10000.0).to(dev)
    gate = torch.randn(64, 2048, generator=g).to(torch.bfloat16).to(dev)
    up = torch.randn(64, 2048, generator=g).to(torch.bfloat16).to(dev)

    def step():
        y = cea.rmsnorm_rope(x, w, 1e-5, pos, inv, 8)
        h = cea.gated_mul(gate, up, "silu")
        return y, h

    _replays_match(step, lambda: cea.gated_mul(up, gate, "gelu"))


def test_key_split_and_subgroup_decode_replays(cea, dev):
    """A prefill chunk that takes the key-split route (partials in the workspace, then the
    list merge) and a decode step with 32 query heads on one KV head (sub-group units)."""
    q, k, v, pos = _attn_inputs(dev, 6000, 7, hq=8, hkv=2)
    qc, qpc = q[:, -96:], pos[:, -96:]
    g = torch.Generator().manual_seed(8)
    dq = torch.randn(2, 1, 32, 128, generator=g).to(torch.bfloat16).to(dev)
    dk = torch.randn(2, 3000, 1, 128, generator=g).to(torch.bfloat16).to(dev)
    dv = torch.randn(2, 3000, 1, 128, generator=g).to(torch.bfloat16).to(dev)
    dkp = torch.arange(3000).repeat(2, 1).to(dev)
    dqp = torch.full((2, 1), 2999).to(dev)

    def step():
        out, lse = cea.attention_with_lse(qc, k, v, qpc, pos)
        plain = cea.attention.attention(qc, k, v, qpc, pos)
        dout, dlse = cea.attention_with_lse(dq, dk, dv, dqp, dkp)
        return out, lse, plain, dout, dlse

    bq, bk, bv, bpos = _attn_inputs(dev, 2048, 9)
    _replays_match(step, lambda: cea.attention_with_lse(bq, bk, bv, bpos, bpos))


@pytest.mark.parametrize("tokens", [20, 300])
def test_graph_of_projections(cea, dev, tokens):
    """The few-token kernel and a K-split launch (its sums in the graph's memory) captured
    together: replays on changed inputs, with eager calls of another size between them, equal
    the eager results."""
    g = torch.Generator().manual_seed(tokens)
    x = torch.randn(tokens, 2048, generator=g).to(torch.bfloat16).to(dev)
    w = (torch.randn(512, 2048, generator=g) / 45).to(torch.bfloat16).to(dev)
    wd = (torch.randn(2048, 256, generator=g) / 16).to(torch.bfloat16).to(dev)
    step = lambda t: cea.linear(cea.linear_gated(t, w[:256], w[256:]), wd)
    stream = torch.cuda.Stream()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.stream(stream):
        step(x)
        stream.synchronize()
        with torch.cuda.graph(graph, stream=stream):
            y = step(x)
    for i in range(3):
        x.copy_(torch.randn(tokens, 2048, generator=g).to(torch.bfloat16))
        want = step(x).clone()
        torch.cuda.synchronize()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(y, want), i
        step(torch.randn(900, 2048, device=dev).to(torch.bfloat16))
        torch.cuda.synchronize()


# calls of several launches that pass scratch from one to the next: a K-split projection (plain and
# gated), key-split prefill, one-launch prefill and split-KV decode
def _scratch_calls(cea, dev, seed):
    g = torch.Generator().manual_seed(seed)
    rand = lambda *s: torch.randn(*s, generator=g).to(torch.bfloat16).to(dev)
    x, w, wd = rand(300, 2048), rand(1024, 2048) / 45, rand(512, 4096) / 64
    xd = rand(300, 4096)
    q, k, v, pos = _attn_inputs(dev, 3000, seed + 1, hq=8, hkv=2)
    return [
        lambda: cea.linear(xd, wd),
        lambda: cea.linear_gated(x, w[:512], w[512:]),
        lambda: cea.attention.attention(q[:, -96:], k, v, pos[:, -96:], pos),
        lambda: cea.attention.attention(q[:, :700], k[:, :700], v[:, :700], pos[:, :700], pos[:, :700]),
        lambda: cea.attention.attention(q[:, -1:], k, v, pos[:, -1:], pos),
    ]


def test_two_threads_on_one_stream(cea, dev):
    """Each thread gets its own results, whatever call of the other thread is enqueued between
    the launches of one of its calls."""
    calls = [_scratch_calls(cea, dev, 10), _scratch_calls(cea, dev, 20)]
    want = [[f() for f in c] for c in calls]
    torch.cuda.synchronize()
    wrong, start = [], threading.Barrier(2)

    def work(t):
        with torch.cuda.stream(stream):
            start.wait(timeout=30)
            for i in range(40):
                for j in range(len(calls[t])):
                    f = calls[t][(j + t) % len(calls[t])]
                    got.append((t, (j + t) % len(calls[t]), f()))

    stream = torch.cuda.Stream(dev)
    got = []
    threads = [threading.Thread(target=work, args=(t,)) for t in range(2)]
    for t in threads:
        t.start()
    for t in threads:
        t.join(timeout=60)
        assert not t.is_alive()
    torch.cuda.synchronize()
    assert len(got) == 2 * 40 * 5
    wrong = [(t, j) for t, j, y in got if not torch.equal(y, want[t][j])]
    assert not wrong, wrong[:10]


def test_graphs_of_one_stream_replayed_on_two(cea, dev):
    """Two graphs captured on the same stream own their scratch: replayed at the same time on two
    streams, with eager calls on the capture stream, each gives its own results."""
    calls = [_scratch_calls(cea, dev, 30), _scratch_calls(cea, dev, 40)]
    want = [[f() for f in c] for c in calls]
    torch.cuda.synchronize()
    capture = torch.cuda.Stream(dev)
    graphs, outs = [], []
    for c in calls:
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph, stream=capture):
            outs.append([f() for f in c])
        graphs.append(graph)
    streams = [torch.cuda.Stream(dev) for _ in graphs]
    for i in range(10):
        for ys in outs:
            for y in ys:
                y.zero_()
        torch.cuda.synchronize()
        for graph, s in zip(graphs, streams):
            with torch.cuda.stream(s):
                graph.replay()
        with torch.cuda.stream(capture):
            eager = [f() for f in calls[0]]
        torch.cuda.synchronize()
        for ys, ws in zip(outs + [eager], want + [want[0]]):
            for j, (y, w) in enumerate(zip(ys, ws)):
                assert torch.equal(y, w), (i, j)
