"""The split workspaces of a pool: one allocation serves a whole generation,
and one that grows all the same keeps captured graphs valid."""
import numpy as np
import pytest

from gpu_util import Populated, rel_err_rows, seeded

pytestmark = pytest.mark.gpu


def _free():
    import torch
    torch.cuda.synchronize()
    return torch.cuda.mem_get_info()[0]


def test_one_allocation_serves_a_generation(gi, oracle, dev):
    """Decode of one sequence of 8 kv heads x 16 query heads from 513 to 8000
    tokens (partials of 8.3 KB, 40 of them and then 256) and prefill of
    growing contexts: the device's free memory stands still after the first
    split call of each."""
    import torch
    H, kvh, hd, P, n = 128, 8, 128, 16, 8000
    pop = Populated(gi, dev, 1, 1, kvh, hd, P, [n], seed=3)
    bt = pop.block_tables()
    lens = [400, 513, 900, 2000, 4000, n]
    sls = [torch.full((1,), x, dtype=torch.int32, device=dev) for x in lens]
    qd, _ = seeded((1, H * hd), 5, dev)
    out = torch.empty_like(qd)
    scale = oracle.attn_scale(hd)
    splits, free = [], []
    for x, sl in zip(lens, sls):
        splits.append(pop.pool.attention_plan(1, H, x)["decode_splits"])
        pop.pool.AttentionGQA(out, qd, 0, bt, sl, H, scale, x)
        free.append(_free())
    assert splits[0] == 1 and splits[1] > 1 and splits[-1] > 2 * splits[1], splits
    assert free[1:] == free[1:2] * (len(lens) - 1), (splits, free)
    C = 16
    qp, _ = seeded((1, C, H * hd), 6, dev)
    op = torch.empty_like(qp)
    starts = [torch.tensor([x - C], dtype=torch.int32, device=dev) for x in lens]
    tables = [bt[:1, :(x + P - 1) // P].contiguous() for x in lens]
    free = []
    for sp, t in zip(starts, tables):
        pop.pool.AttentionGQABatch(op, qp, 0, t, sp, H, scale, C)
        free.append(_free())
    assert free[2:] == free[2:3] * (len(lens) - 2), free


def test_no_plan_asks_for_more_than_the_first_growth(gi, dev):
    """Slots of either plan never pass two per CU up to one pair per CU, and
    6.25 per CU in all (the room the first growth makes, and the header's
    bound)."""
    import torch
    cus = torch.cuda.get_device_properties(dev).multi_processor_count
    for kv_type in range(4):
        for kvh, hd in ((1, 128), (4, 64), (8, 128)):
            pool = gi.PagedKVCache(1, kvh, hd, 16, 1, kv_type)
            for batch in sorted({max(1, f * cus // (8 * kvh)) + d for f in range(1, 17) for d in (0, 1)}):
                pairs = batch * kvh
                most = 2 * cus if pairs <= cus else min(5 * pairs, 25 * cus // 4)
                for n in (1, 257, 513, 1025, 2561, 4097, 9000, 40000, 200000):
                    s = pool.attention_plan(batch, 8 * kvh, n)["decode_splits"]
                    coarse = max(1, min(-(-cus // pairs), -(-n // 1024)))
                    assert max(s, coarse) * pairs <= most or (s == 1 and coarse == 1), (kv_type, kvh, batch, n, s)
            pool.close()


def test_growth_after_a_capture_keeps_the_graph(gi, oracle, dev):
    """A graph captured over 32 query heads replays bit for bit after an eager
    call over 64 grew the workspace it reads."""
    import torch
    H, kvh, hd, P, n = 32, 8, 128, 16, 1100
    pop = Populated(gi, dev, 1, 1, kvh, hd, P, [n], seed=7)
    stream = torch.cuda.Stream(dev)
    pop.pool.set_stream(stream.cuda_stream)
    bt = pop.block_tables()
    sl = torch.tensor([n], dtype=torch.int32, device=dev)
    qd, q = seeded((1, H * hd), 8, dev)
    out = torch.empty_like(qd)
    scale = oracle.attn_scale(hd)
    with torch.cuda.stream(stream):
        pop.pool.AttentionGQA(out, qd, 0, bt, sl, H, scale, n)
    torch.cuda.synchronize()
    ref = out.clone()
    ks, vs = pop.stored(0, 0)
    k, v = oracle.widen(1, kvh * hd, ks), oracle.widen(1, kvh * hd, vs)
    assert float(rel_err_rows(ref.cpu().numpy(), oracle.attention_decode(q[0], k, v, H, kvh, hd, n, scale),
                              H, hd).max()) <= 1e-3
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=stream):
        pop.pool.AttentionGQA(out, qd, 0, bt, sl, H, scale, n)
    q2, q2h = seeded((1, 2 * H * hd), 9, dev)
    o2 = torch.empty_like(q2)
    for r in range(3):
        out.fill_(float("nan"))
        torch.cuda.synchronize()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, ref), r
        with torch.cuda.stream(stream):
            pop.pool.AttentionGQA(o2, q2, 0, bt, sl, 2 * H, scale, n)
        torch.cuda.synchronize()
        assert float(rel_err_rows(o2.cpu().numpy(),
                                  oracle.attention_decode(q2h[0], k, v, 2 * H, kvh, hd, n, scale),
                                  2 * H, hd).max()) <= 1e-3, r


def test_wide_tables_alone_do_not_split_a_full_device(gi, oracle, dev):
    """Where (sequence, kv head) pairs fill the CUs 1 to 1.6 times, contexts
    are cut for a caller that says they are long, not because the tables are
    wide: without max_seq_len such a call takes no workspace.  Both give the
    same attention."""
    import torch
    cus = torch.cuda.get_device_properties(dev).multi_processor_count
    H, kvh, hd, P, n, wide = 32, 8, 128, 16, 300, 6000
    rows = cus * 9 // 8 // kvh
    pop = Populated(gi, dev, 1, 1, kvh, hd, P, [n], seed=11)
    bt = torch.zeros(rows, wide // P, dtype=torch.int32, device=dev)
    bt[:, :pop.max_blocks] = pop.block_tables()
    sl = torch.full((rows,), n, dtype=torch.int32, device=dev)
    qd, q = seeded((rows, H * hd), 12, dev)
    scale = oracle.attn_scale(hd)
    ks, vs = pop.stored(0, 0)
    k, v = oracle.widen(1, kvh * hd, ks), oracle.widen(1, kvh * hd, vs)
    want = oracle.attention_decode(q[rows - 1], k, v, H, kvh, hd, n, scale)
    out = torch.empty_like(qd)
    before = _free()
    for hint, grows in ((0, False), (wide, True)):
        out.fill_(float("nan"))
        pop.pool.AttentionGQA(out, qd, 0, bt, sl, H, scale, hint)
        pop.pool.synchronize()
        assert (_free() < before) == grows, hint
        assert float(rel_err_rows(out[rows - 1].cpu().numpy(), want, H, hd).max()) <= 1e-3, hint


def test_short_contexts_at_head_dimension_64_stay_whole(gi, dev):
    """A third round of 256-token blocks costs less than a merge there."""
    import torch
    if torch.cuda.get_device_properties(dev).multi_processor_count != 256:
        pytest.skip("the shapes are worked out for a 256-CU device")
    for kv_type, batch, whole in ((1, 1, 640), (1, 8, 640), (1, 16, 896), (2, 16, 640), (3, 4, 640), (0, 4, 512)):
        pool = gi.PagedKVCache(1, 4, 64, 16, 1, kv_type)
        assert pool.attention_plan(batch, 32, whole)["decode_splits"] == 1, (kv_type, batch)
        assert pool.attention_plan(batch, 32, whole + 1)["decode_splits"] > 1, (kv_type, batch)
        pool.close()
