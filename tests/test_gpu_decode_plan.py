"""The decode split plan at the edges of its rules, against float64 softmax
attention over the stored K/V, and the calls whose scratch cannot hold the
plan's partials: those run with the coarse plan instead of failing."""
import numpy as np
import pytest

from gpu_util import Populated, rel_err_rows, seeded

pytestmark = pytest.mark.gpu

# Scores are exact products of split operands (relative 2^-21 of |q||k|, here
# |score| <= ~16 after scaling, so at most 16 * 2^-21 = 8e-6 in the exponent)
# and sums in float32; 2e-5 of a row's largest output covers both.
TOL = 2e-5


def attend64(q, k, v, H, kvh, hd, scale):
    G = H // kvh
    n = k.shape[0]
    s = np.einsum("hgd,nhd->hgn", q.astype(np.float64).reshape(kvh, G, hd), k.astype(np.float64).reshape(n, kvh, hd))
    s = s * scale
    p = np.exp(s - s.max(axis=2, keepdims=True))
    p /= p.sum(axis=2, keepdims=True)
    return np.einsum("hgn,nhd->hgd", p, v.astype(np.float64).reshape(n, kvh, hd)).reshape(H * hd)


# (kv type, H, kvh, hd, page, rows, tokens): unsplit and split on both sides
# of 256, 512 and 1024 tokens, splits of 128 with a short last one, merges of
# up to 8, up to 32 and more splits, one and two workgroups per CU, and the
# splits of batches that half fill a second round.
@pytest.mark.parametrize("kv_type,H,kvh,hd,P,rows,n", [
    (1, 32, 8, 128, 16, 1, 512), (1, 32, 8, 128, 16, 1, 513), (0, 32, 8, 128, 16, 1, 257),
    (0, 32, 4, 64, 16, 1, 513), (3, 32, 4, 64, 32, 2, 700), (2, 32, 8, 128, 16, 1, 1025),
    (1, 16, 1, 128, 16, 1, 8200), (1, 8, 1, 64, 16, 1, 33000), (3, 16, 2, 128, 16, 1, 4097),
    (1, 32, 8, 128, 16, 12, 1025), (0, 32, 8, 128, 16, 12, 1100), (2, 32, 8, 128, 16, 17, 1030),
    (0, 32, 8, 128, 16, 20, 1100), (1, 32, 8, 128, 16, 36, 4097), (3, 32, 8, 128, 16, 48, 2561)])
def test_decode_plan_edges(gi, oracle, dev, kv_type, H, kvh, hd, P, rows, n):
    import torch
    pop = Populated(gi, dev, kv_type, 1, kvh, hd, P, [n], seed=71)
    ks, vs = pop.stored(0, 0)
    k, v = oracle.widen(kv_type, kvh * hd, ks), oracle.widen(kv_type, kvh * hd, vs)
    # row r attends the first lens[r] tokens of the one sequence
    lens = [max(1, n - 37 * r) for r in range(rows)]
    bt = pop.block_tables()[torch.zeros(rows, dtype=torch.long, device=dev)].contiguous()
    sl = torch.tensor(lens, dtype=torch.int32, device=dev)
    qd, q = seeded((rows, H * hd), 72, dev)
    out = torch.full_like(qd, float("nan"))
    scale = oracle.attn_scale(hd)
    pop.pool.AttentionGQA(out, qd, 0, bt, sl, H, scale, n)
    pop.pool.synchronize()
    o = out.cpu().numpy()
    for r in sorted({0, rows // 2, rows - 1}):
        want = attend64(q[r], k[:lens[r]], v[:lens[r]], H, kvh, hd, scale)
        assert float(rel_err_rows(o[r], want, H, hd).max()) <= TOL, (r, lens[r])


def test_scratch_that_cannot_hold_the_plan_takes_the_coarse_one(gi, oracle, dev):
    """102 rows x 1 kv head of 16 query heads: five splits each would need
    4.24 MB, over the fixed 4 MiB scratch; three splits (2.5 MB) fit, so the
    allocate-nothing call is still served.  And a first call made while the
    stream captures: 600 tokens are cut into splits only where the workspace
    exists, so it needs none."""
    import torch
    H, kvh, hd, P, n, rows = 16, 1, 128, 16, 2300, 102
    if torch.cuda.get_device_properties(dev).multi_processor_count != 256:
        pytest.skip("the shape is worked out for a 256-CU device")
    pop = Populated(gi, dev, 1, 1, kvh, hd, P, [n], seed=73)
    scale = oracle.attn_scale(hd)
    plan = pop.pool.attention_plan(rows, H, n)
    assert rows * plan["decode_splits"] * H * (hd + 2) * 4 > 4 << 20, plan
    bt = pop.block_tables()[torch.zeros(rows, dtype=torch.long, device=dev)].contiguous()
    sl = torch.full((rows,), n, dtype=torch.int32, device=dev)
    qd, q = seeded((rows, H * hd), 74, dev)
    out = torch.full_like(qd, float("nan"))
    pop.pool.AttentionGQANoAlloc(out, qd, 0, bt, sl, H, scale)
    pop.pool.synchronize()
    ks, vs = pop.stored(0, 0)
    k, v = oracle.widen(1, kvh * hd, ks), oracle.widen(1, kvh * hd, vs)
    for r in (0, rows - 1):
        want = attend64(q[r], k, v, H, kvh, hd, scale)
        assert float(rel_err_rows(out[r].cpu().numpy(), want, H, hd).max()) <= TOL, r

    fresh = Populated(gi, dev, 1, 1, 8, hd, P, [600], seed=75)
    assert fresh.pool.attention_plan(1, 32, 600)["decode_splits"] > 1
    stream = torch.cuda.Stream(dev)
    fresh.pool.set_stream(stream.cuda_stream)
    bt = fresh.block_tables()
    sl = torch.tensor([600], dtype=torch.int32, device=dev)
    qd, q = seeded((1, 32 * hd), 76, dev)
    out = torch.full_like(qd, float("nan"))
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=stream):
        fresh.pool.AttentionGQA(out, qd, 0, bt, sl, 32, scale, 600)
    ks, vs = fresh.stored(0, 0)
    want = attend64(q[0], oracle.widen(1, 8 * hd, ks), oracle.widen(1, 8 * hd, vs), 32, 8, hd, scale)
    for _ in range(3):
        out.fill_(float("nan"))
        torch.cuda.synchronize()
        graph.replay()
        torch.cuda.synchronize()
        assert float(rel_err_rows(out[0].cpu().numpy(), want, 32, hd).max()) <= TOL
