"""The spark GPU sampler over fp32 measures (ds41_spark_verify_gpu_v2 /
ds41_spark_sample_gpu_v2, engine/third_party/spark/src/sampling.cu:6-49) on the
GPU against the oracle's restatement of the reference kernel, through the C ABI.

Bar: accept/reject decisions and token ids bit-exact.
The measures are random fp32 rows whose fp64 sums round, so the kernel's
summation orders (strided mass + tree, chunked draw prefix) are exercised; the
oracle itself is pinned to the compiled reference host sampler on exact sums
(tests/test_oracle_sampler.py)."""
import numpy as np
import pytest

import oracle as O

pytestmark = pytest.mark.gpu


def measures(rng, rows, V, kind):
    if kind == "softmax":
        x = rng.standard_normal((rows, V)) * 2.5
        return np.exp(x - x.max(axis=1, keepdims=True)).astype(np.float32)
    if kind == "sparse":  # long zero runs: empty chunks, fallbacks to the last positive index
        m = (rng.random((rows, V)) * (rng.random((rows, V)) < 0.01)).astype(np.float32)
        m[:, 0] += 1e-3
        return m
    return rng.random((rows, V)).astype(np.float32) * 1e-3 + np.float32(1e-30)


def run_gpu(gpu, d, q, p, greedy, seed, step):
    import torch
    import ds41_gfx950 as G
    out = torch.full((10,), 7, dtype=torch.int32, device=gpu)
    dd = torch.from_numpy(np.ascontiguousarray(d, np.int32)).to(gpu) if d is not None and len(d) else None
    qd = torch.from_numpy(np.ascontiguousarray(q)).to(gpu) if q is not None else None
    G.verify_gpu_v2(dd, qd, torch.from_numpy(np.ascontiguousarray(p)).to(gpu), greedy, seed, step, out)
    torch.cuda.synchronize()
    return G.result_raw(out)


@pytest.mark.parametrize("V,k,kind", [(129280, 3, "softmax"), (129280, 5, "uniform"), (4097, 2, "sparse"),
                                      (300, 1, "softmax"), (257, 4, "sparse"), (7, 2, "uniform"), (1, 0, "uniform")])
def test_verify_gpu_v2_bitexact_vs_oracle(gpu, V, k, kind):
    rng = np.random.default_rng(V * 10 + k)
    steps = 40 if V > 10000 else 120
    mism = 0
    for step in range(steps):
        p = measures(rng, k + 1, V, kind)
        q = measures(rng, k, V, kind) if k else None
        greedy = int(step % 5 == 4)
        seed = int(rng.integers(0, 1 << 63))
        # drafts as the drafter samples them: from q (slot j, purpose Draft) with the same sampler
        d = np.array([O.sample_gpu_v2(q[j], seed, step, j, 1) for j in range(k)], np.int32)
        want = O.verify_gpu_v2(d, q, p, k, V, greedy, seed, step).raw()
        got = run_gpu(gpu, d, None if greedy else q, p, greedy, seed, step)
        mism += got != want
    assert mism == 0


@pytest.mark.parametrize("V,k", [(2047, 2), (2048, 2), (2049, 5), (4095, 2), (4096, 2), (4097, 5), (5119, 1), (5120, 1), (5121, 4),
                                 (65537, 1), (131072, 2), (131073, 3), (200001, 5)])
def test_verify_gpu_v2_wide_edges(gpu, V, k):
    """Around the row lengths where calls spread over workgroups, and where a chain of 256 strided
    or contiguous entries passes one staged block (131,072 entries, 512 per chain)."""
    rng = np.random.default_rng(V + k)
    for step, kind in enumerate(("softmax", "sparse", "uniform", "softmax", "sparse", "uniform")):
        p, q = measures(rng, k + 1, V, kind), measures(rng, k, V, kind)
        if kind == "softmax":  # close rows: drafts are accepted and later rows reached
            q = (p[:k] * rng.uniform(0.95, 1.05, (k, V))).astype(np.float32)
        seed, greedy = int(rng.integers(0, 1 << 63)), int(step == 3)
        d = (p[:k].argmax(1).astype(np.int32) if greedy
             else np.array([O.sample_gpu_v2(q[j], seed, step, j, 1) for j in range(k)], np.int32))
        want = O.verify_gpu_v2(d, q, p, k, V, greedy, seed, step).raw()
        assert run_gpu(gpu, d, None if greedy else q, p, greedy, seed, step) == want, (kind, greedy)


@pytest.mark.parametrize("V", [10239, 10240, 10241])
def test_single_row_wide_edges(gpu, V):
    """The row length from which a call of one row spreads over workgroups: sample, and verify of no draft."""
    import torch
    import ds41_gfx950 as G
    rng = np.random.default_rng(V)
    tok = torch.zeros(1, dtype=torch.int32, device=gpu)
    for step, kind in enumerate(("softmax", "sparse", "uniform")):
        p = measures(rng, 1, V, kind)
        for greedy in (0, 1):
            want = O.verify_gpu_v2(None, None, p, 0, V, greedy, 21, step).raw()
            assert run_gpu(gpu, None, None, p, greedy, 21, step) == want, (kind, greedy)
        G.sample_gpu_v2(torch.from_numpy(p[0]).to(gpu), 21, step, 2, 1, tok)
        torch.cuda.synchronize()
        assert int(tok.item()) == O.sample_gpu_v2(p[0], 21, step, 2, 1), kind


def slots_in_use(gpu, hold=0):
    """Scratch slots that calls own; hold: takes the free ones first."""
    import torch
    import ds41_gfx950 as G
    n = torch.full((1,), -1, dtype=torch.int32, device=gpu)
    G.spark_scratch_hold(hold, n)
    torch.cuda.synchronize()
    return int(n.item())


def accepting_call(gpu, rng, V, k, seed, step):
    """A call whose rows are close, so that drafts are accepted: its arrays, and the same on the device."""
    import torch
    p = measures(rng, k + 1, V, "softmax")
    q = (p[:k] * rng.uniform(0.95, 1.05, (k, V))).astype(np.float32)
    d = np.array([O.sample_gpu_v2(q[j], seed, step, j, 1) for j in range(k)], np.int32)
    return (d, q, p), [torch.from_numpy(a).to(gpu) for a in (d, q, p)]


@pytest.mark.parametrize("V", [1000, 20000])
def test_verify_gpu_v2_drafts_inside_result(gpu, V):
    """The drafts lie in the result's own tokens: both ways of running a call read them before it is written."""
    import torch
    import ds41_gfx950 as G
    rng = np.random.default_rng(V)
    k = 3
    for step in range(6):
        (d, q, p), (_, qd, pd) = accepting_call(gpu, rng, V, k, 9, step)
        for greedy in (0, 1):
            if greedy:
                d = p[:k].argmax(1).astype(np.int32)
            out = torch.full((10,), 7, dtype=torch.int32, device=gpu)
            out[:k] = torch.from_numpy(d).to(gpu)
            G.verify_gpu_v2(out[:k], None if greedy else qd, pd, greedy, 9, step, out)
            torch.cuda.synchronize()
            assert G.result_raw(out) == O.verify_gpu_v2(d, None if greedy else q, p, k, V, greedy, 9, step).raw()


def test_wide_calls_with_one_result_buffer(gpu):
    """The same call on several streams into one result: whatever order the launches take, each finds its own
    slot, the result is the call's, and every slot is free in the end."""
    import torch
    import ds41_gfx950 as G
    rng = np.random.default_rng(12)
    V, k = 20000, 3
    host, dev = accepting_call(gpu, rng, V, k, 3, 4)
    want = O.verify_gpu_v2(*host, k, V, 0, 3, 4).raw()
    out, tok = torch.zeros(10, dtype=torch.int32, device=gpu), torch.zeros(1, dtype=torch.int32, device=gpu)
    streams = [torch.cuda.Stream() for _ in range(8)]
    torch.cuda.synchronize()
    for r in range(12):
        for s in streams:
            G.verify_gpu_v2(*dev, 0, 3, 4, out, s)
            G.sample_gpu_v2(dev[2][0], 3, 4, 0, 0, tok, s)
    torch.cuda.synchronize()
    assert G.result_raw(out) == want
    assert int(tok.item()) == O.sample_gpu_v2(host[2][0], 3, 4, 0, 0)
    assert slots_in_use(gpu) == 0


def test_wide_calls_without_a_free_slot(gpu):
    """With every slot taken, verify (greedy and not) and sample run on one workgroup, with the same results."""
    import torch
    import ds41_gfx950 as G
    rng = np.random.default_rng(13)
    V, k = 20000, 3
    host, dev = accepting_call(gpu, rng, V, k, 5, 6)
    top = host[2][:k].argmax(1).astype(np.int32)
    topd = torch.from_numpy(top).to(gpu)
    outs = [torch.zeros(10, dtype=torch.int32, device=gpu) for _ in range(4)]
    toks = [torch.zeros(1, dtype=torch.int32, device=gpu) for _ in range(2)]
    try:
        for i in range(2):  # all taken, then all free
            assert slots_in_use(gpu, hold=1 - i) == 0
            G.verify_gpu_v2(*dev, 0, 5, 6, outs[2 * i])
            G.verify_gpu_v2(topd, None, dev[2], 1, 5, 6, outs[2 * i + 1])
            G.sample_gpu_v2(dev[2][1], 5, 6, 1, 0, toks[i])
            torch.cuda.synchronize()
    finally:
        slots_in_use(gpu, hold=0)
    for i in range(2):
        assert G.result_raw(outs[2 * i]) == O.verify_gpu_v2(*host, k, V, 0, 5, 6).raw()
        assert G.result_raw(outs[2 * i + 1]) == O.verify_gpu_v2(top, None, host[2], k, V, 1, 5, 6).raw()
        assert int(toks[i].item()) == O.sample_gpu_v2(host[2][1], 5, 6, 1, 0)
    assert slots_in_use(gpu) == 0


def test_wide_call_replayed(gpu):
    """A captured call finds its slot again at every replay, with eager calls between and new inputs in place."""
    import torch
    import ds41_gfx950 as G
    rng = np.random.default_rng(14)
    V, k = 20000, 2
    _, dev = accepting_call(gpu, rng, V, k, 7, 8)
    out, eager = (torch.zeros(10, dtype=torch.int32, device=gpu) for _ in range(2))
    stream = torch.cuda.Stream()
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=stream):
        G.verify_gpu_v2(*dev, 0, 7, 8, out, stream)
    for _ in range(4):
        host, new = accepting_call(gpu, rng, V, k, 7, 8)
        for a, b in zip(dev, new):
            a.copy_(b)
        torch.cuda.synchronize()
        G.verify_gpu_v2(*dev, 0, 7, 8, eager)
        graph.replay()
        torch.cuda.synchronize()
        assert G.result_raw(out) == G.result_raw(eager) == O.verify_gpu_v2(*host, k, V, 0, 7, 8).raw()
    assert slots_in_use(gpu) == 0


def test_verify_gpu_v2_overlapping_streams(gpu):
    """Calls on more streams than there are scratch slots, each several times over; every slot is free again
    in the end (the hardware's queues decide how many of them are in flight together)."""
    import torch
    import ds41_gfx950 as G
    rng = np.random.default_rng(11)
    V, k, n = 20000, 3, 24
    calls = []
    for i in range(n):
        p, q = measures(rng, k + 1, V, "softmax"), measures(rng, k, V, "softmax")
        d = np.array([O.sample_gpu_v2(q[j], i, 5, j, 1) for j in range(k)], np.int32)
        dev = [torch.from_numpy(a).to(gpu) for a in (d, q, p)]
        calls.append((dev, torch.zeros((4, 10), dtype=torch.int32, device=gpu), torch.cuda.Stream(),
                      O.verify_gpu_v2(d, q, p, k, V, 0, i, 5).raw()))
    torch.cuda.synchronize()
    for r in range(4):
        for i, (dev, out, stream, _) in enumerate(calls):
            G.verify_gpu_v2(*dev, 0, i, 5, out[r], stream)
    torch.cuda.synchronize()
    for _, out, _, want in calls:
        assert all(G.result_raw(out[r]) == want for r in range(4))
    assert slots_in_use(gpu) == 0


def test_verify_gpu_v2_invalid_inputs_match_oracle(gpu):
    rng = np.random.default_rng(3)
    V = 5000
    p = measures(rng, 3, V, "softmax")
    q = measures(rng, 2, V, "softmax")
    d = np.array([10, 20], np.int32)
    # a row is checked when the step reaches it (sampling.cu:29-33): row 0 and draft 0 always are
    cases = []
    bad = p.copy(); bad[0, 77] = np.nan; cases.append((d, q, bad))
    neg = p.copy(); neg[0, 5] = -1.0; cases.append((d, q, neg))
    qz = q.copy(); qz[0, 10] = 0.0; cases.append((d, qz, p))
    cases.append((np.array([V, 10], np.int32), q, p))
    zero = p.copy(); zero[0] = 0.0; cases.append((d, q, zero))
    qnan = q.copy(); qnan[0, 3] = np.inf; cases.append((d, qnan, p))
    for dd, qq, pp in cases:
        want = O.verify_gpu_v2(dd, qq, pp, 2, V, 0, 1, 2).raw()
        assert run_gpu(gpu, dd, qq, pp, 0, 1, 2) == want
        assert want[1] == -1
    # an invalid row past the step's end takes no part in it (its entries may be read): the step is valid
    late = p.copy(); late[2, 9] = np.nan
    want = O.verify_gpu_v2(np.array([0, 1], np.int32), q, late, 2, V, 0, 1, 2).raw()
    assert run_gpu(gpu, np.array([0, 1], np.int32), q, late, 0, 1, 2) == want


def test_sample_gpu_v2_bitexact_vs_oracle(gpu):
    import torch
    import ds41_gfx950 as G
    rng = np.random.default_rng(4)
    out = torch.zeros(1, dtype=torch.int32, device=gpu)
    for V, kind in ((129280, "softmax"), (1000, "sparse"), (3, "uniform")):
        for step in range(30):
            p = measures(rng, 1, V, kind)[0]
            seed, slot, purpose = int(rng.integers(0, 1 << 63)), step % 6, step % 4
            G.sample_gpu_v2(torch.from_numpy(p).to(gpu), seed, step, slot, purpose, out)
            torch.cuda.synchronize()
            assert int(out.item()) == O.sample_gpu_v2(p, seed, step, slot, purpose), (V, kind, step)
    with pytest.raises(RuntimeError):
        G.sample_gpu_v2(torch.zeros(4, device=gpu), 0, 0, 6, 0, out)  # slot > 5
