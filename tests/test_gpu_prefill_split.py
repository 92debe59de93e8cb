"""Prefill over a context cut into splits (and over 128-column workgroups)
against float64 causal attention: chunks on both sides of the lengths that
stay whole, ragged batches whose shorter sequences leave splits empty, split
edges inside a chunk's causal diagonal, a rejected page in one split, and a
first call under capture, which keeps the context in one piece."""
import numpy as np
import pytest

from gpu_util import Populated, rel_err_rows, seeded

pytestmark = pytest.mark.gpu

# as in test_gpu_decode_plan: scores of at most ~16 from operands split to a
# relative 2^-21, sums in float32, one more float32 rounding per split
TOL = 2e-5


def causal64(q, k, v, H, kvh, hd, start, scale):
    m, n, G = q.shape[0], k.shape[0], H // kvh
    q = q.astype(np.float64).reshape(m, kvh, G, hd)
    k = k.astype(np.float64).reshape(n, kvh, hd)
    v = v.astype(np.float64).reshape(n, kvh, hd)
    out = np.empty((m, kvh, G, hd))
    dead = np.arange(n)[None, :] > start + np.arange(m)[:, None]
    for h in range(kvh):
        s = np.einsum("mgd,nd->gmn", q[:, h], k[:, h]) * scale
        s[:, dead] = -np.inf
        p = np.exp(s - s.max(axis=2, keepdims=True))
        p /= p.sum(axis=2, keepdims=True)
        out[:, h] = np.einsum("gmn,nd->mgd", p, v[:, h])
    return out.reshape(m, H * hd)


SHAPES = [
    (16, 4, 128, 16, [0, 700, 1300], 45), (8, 2, 128, 32, [2040], 64), (8, 2, 128, 64, [449], 64),
    (16, 4, 128, 16, [448], 65), (8, 4, 64, 16, [321, 1000], 64), (16, 2, 64, 32, [320], 64),
    (8, 8, 64, 64, [1531], 130), (4, 4, 128, 16, [5, 3001], 1), (8, 1, 128, 16, [250], 515),
    (32, 8, 128, 16, [0, 900], 257),  # wide splits: 144 workgroups of 128 columns on 256 CUs
]


@pytest.mark.parametrize("kv_type", [0, 1, 2, 3], ids=["f32", "f16", "q8_0", "q4_0"])
@pytest.mark.parametrize("H,kvh,hd,P,starts,chunk", SHAPES)
def test_prefill_splits(gi, oracle, dev, kv_type, H, kvh, hd, P, starts, chunk):
    import torch
    lens = [s + chunk for s in starts]
    pop = Populated(gi, dev, kv_type, 1, kvh, hd, P, lens, seed=91)
    bt = pop.block_tables()
    sp = torch.tensor(starts, dtype=torch.int32, device=dev)
    qd, q = seeded((len(starts), chunk, H * hd), 92, dev)
    scale = oracle.attn_scale(hd)
    wants = []
    for i, s in enumerate(starts):
        ks, vs = pop.stored(0, i)
        wants.append(causal64(q[i], oracle.widen(kv_type, kvh * hd, ks), oracle.widen(kv_type, kvh * hd, vs),
                              H, kvh, hd, s, scale))
    for _ in range(2):  # the second call finds the first one's partials in the workspace
        out = torch.full_like(qd, float("nan"))
        pop.pool.AttentionGQABatch(out, qd, 0, bt, sp, H, scale, chunk)
        pop.pool.synchronize()
        o = out.cpu().numpy()
        for i in range(len(starts)):
            assert float(rel_err_rows(o[i], wants[i], H, hd).max()) <= TOL, i

    # the same without a workspace: a fresh pool's first call is captured
    fresh = Populated(gi, dev, kv_type, 1, kvh, hd, P, lens, seed=91)
    if fresh.pool.attention_plan(1, H, 1)["prefill_kernel"] == 0:
        return
    stream = torch.cuda.Stream(dev)
    fresh.pool.set_stream(stream.cuda_stream)
    out = torch.full_like(qd, float("nan"))
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=stream):
        fresh.pool.AttentionGQABatch(out, qd, 0, bt, sp, H, scale, chunk)
    for _ in range(2):
        out.fill_(float("nan"))
        torch.cuda.synchronize()
        graph.replay()
        torch.cuda.synchronize()
        o = out.cpu().numpy()
        for i in range(len(starts)):
            assert float(rel_err_rows(o[i], wants[i], H, hd).max()) <= TOL, i


@pytest.mark.parametrize("kv_type", [0, 1, 2, 3], ids=["f32", "f16", "q8_0", "q4_0"])
def test_prefill_splits_skip_a_bad_page(gi, oracle, dev, kv_type):
    """Every page of one split's 256 tokens rejected: its partial is empty
    and the others carry the row."""
    import torch
    H, kvh, hd, P, start, chunk = 8, 2, 128, 16, 1200, 48
    pop = Populated(gi, dev, kv_type, 1, kvh, hd, P, [start + chunk], seed=93)
    bt = pop.block_tables()
    lo, hi = 512 // P, 1024 // P
    bt[0, lo:hi] = pop.pool.num_pages + 3
    keep = np.r_[0:lo * P, hi * P:start + chunk]
    qd, q = seeded((1, chunk, H * hd), 94, dev)
    scale = oracle.attn_scale(hd)
    ks, vs = pop.stored(0, 0)
    want = causal64(q[0], oracle.widen(kv_type, kvh * hd, ks)[keep], oracle.widen(kv_type, kvh * hd, vs)[keep],
                    H, kvh, hd, start - (hi - lo) * P, scale)
    out = torch.full_like(qd, float("nan"))
    pop.pool.AttentionGQABatch(out, qd, 0, bt, torch.tensor([start], dtype=torch.int32, device=dev), H, scale, chunk)
    with pytest.raises(gi.GIError) as e:
        pop.pool.synchronize()
    assert e.value.code == -7
    assert float(rel_err_rows(out[0].cpu().numpy(), want, H, hd).max()) <= TOL


# q4_0 pages at head dimension 64 run on the vector kernel, which cuts nothing
@pytest.mark.parametrize("kv_type,hd", [(0, 64), (0, 128), (1, 64), (1, 128), (2, 64), (2, 128), (3, 128)])
def test_prefill_splits_queries_before_position_0(gi, oracle, dev, kv_type, hd):
    """Queries that attend no token get zeros, in a sequence of which every
    workgroup holds only such queries and in one that crosses position 0,
    beside a sequence long enough to be cut."""
    import torch
    H, kvh, P, starts, chunk = 8, 2, 16, [-300, -20, 1000], 64
    lens = [max(0, s + chunk) for s in starts]
    pop = Populated(gi, dev, kv_type, 1, kvh, hd, P, lens, seed=95)
    bt = pop.block_tables()
    qd, q = seeded((len(starts), chunk, H * hd), 96, dev)
    scale = oracle.attn_scale(hd)
    out = torch.full_like(qd, float("nan"))
    pop.pool.AttentionGQABatch(out, qd, 0, bt, torch.tensor(starts, dtype=torch.int32, device=dev), H, scale, chunk)
    pop.pool.synchronize()
    o = out.cpu().numpy()
    for i, s in enumerate(starts):
        skip = min(chunk, max(0, -s))  # queries before position 0
        assert not o[i, :skip].any(), i
        if skip == chunk:
            continue
        ks, vs = pop.stored(0, i)
        want = causal64(q[i, skip:], oracle.widen(kv_type, kvh * hd, ks), oracle.widen(kv_type, kvh * hd, vs),
                        H, kvh, hd, s + skip, scale)
        assert float(rel_err_rows(o[i, skip:], want, H, hd).max()) <= TOL, i


# 16 heads per kv head (fp16 pages; the others run on the vector kernel), and
# an odd number of rows in an odd number of splits, whose (maximum, sum) part
# is no multiple of 16 bytes
@pytest.mark.parametrize("kv_type,H,kvh,hd,start,chunk", [
    (1, 16, 1, 128, 1500, 77), (1, 32, 2, 128, 700, 130), (0, 9, 9, 128, 760, 45), (1, 9, 9, 64, 760, 45),
    (2, 9, 9, 64, 760, 45), (3, 9, 9, 128, 760, 45)])
def test_prefill_splits_of_other_head_layouts(gi, oracle, dev, kv_type, H, kvh, hd, start, chunk):
    import torch
    pop = Populated(gi, dev, kv_type, 1, kvh, hd, 16, [start + chunk], seed=97)
    qd, q = seeded((1, chunk, H * hd), 98, dev)
    scale = oracle.attn_scale(hd)
    out = torch.full_like(qd, float("nan"))
    pop.pool.AttentionGQABatch(out, qd, 0, pop.block_tables(), torch.tensor([start], dtype=torch.int32, device=dev),
                               H, scale, chunk)
    pop.pool.synchronize()
    ks, vs = pop.stored(0, 0)
    want = causal64(q[0], oracle.widen(kv_type, kvh * hd, ks), oracle.widen(kv_type, kvh * hd, vs), H, kvh, hd, start,
                    scale)
    assert float(rel_err_rows(out[0].cpu().numpy(), want, H, hd).max()) <= TOL
