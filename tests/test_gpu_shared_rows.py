"""Decode steps whose rows share pages: draft tokens of one sequence verified
as rows of one batch (the same block table at lengths n + 1, n + 2, ...), and
a row that reads the page they write at another place of its own table.  Every
token of a step is stored before any row attends, so the step must leave the
bits of the append followed by the attention: q, the pages and the output."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


# H, kvh, hd, P, n, rows: one split and several, eight- and four-wave
# workgroups, pages whose lines two waves read (64) and that blocks straddle
# (48), more rows than lanes of a wave, 16 heads per kv head; contexts whose
# pages go through the hash, and more of them than lanes
@pytest.mark.parametrize("kv_type", [0, 1, 2, 3], ids=["f32", "f16", "q8_0", "q4_0"])
@pytest.mark.parametrize("H,kvh,hd,P,n,rows", [
    (32, 8, 128, 16, 45, 5), (32, 8, 128, 32, 700, 4), (32, 4, 64, 64, 100, 3), (16, 2, 64, 16, 20, 70),
    (32, 8, 128, 16, 30, 40), (16, 1, 128, 48, 200, 6), (32, 8, 128, 16, 1200, 40), (32, 8, 128, 32, 4200, 52)])
@pytest.mark.parametrize("rope", [False, True], ids=["step", "rope"])
def test_rows_of_a_step_see_each_others_tokens(gi, oracle, dev, kv_type, H, kvh, hd, P, n, rows, rope):
    import torch
    kv_dim = kvh * hd
    # the last row's table starts with the page of the first draft token
    lens = [n + 1 + r for r in range(rows)] + [P + 5]
    blocks = (n + rows + P - 1) // P
    pages = blocks + 3
    ids = np.random.default_rng(3).permutation(pages).astype(np.int32)
    bt = np.zeros((rows + 1, max(blocks, 2)), np.int32)
    bt[:rows, :blocks] = ids[:blocks]
    bt[rows, :2] = ids[n // P], ids[blocks]
    btd = torch.from_numpy(bt).to(dev)
    sl = torch.tensor(lens, dtype=torch.int32, device=dev)
    t = np.arange(pages * P)
    old = [torch.from_numpy(oracle.normal(s, (pages * P, kv_dim))).to(dev) for s in (4, 5)]
    pools = []
    for _ in range(2):
        pool = gi.PagedKVCache(1, kvh, hd, P, pages, kv_type)
        pool.SetRoPE(10000.0, 0, max(lens))
        pool.Write(0, torch.from_numpy((t // P).astype(np.int32)).to(dev),
                   torch.from_numpy((t % P).astype(np.int32)).to(dev), *old)
        pools.append(pool)
    fused, parts = pools
    plan = fused.attention_plan(rows + 1, H, max(lens))
    assert plan["decode_kernel"] == 0 or plan["decode_step_fused"], plan  # what this test is about
    q = torch.from_numpy(oracle.normal(7, (rows + 1, H * hd))).to(dev)
    k = torch.from_numpy(oracle.normal(8, (rows + 1, kv_dim))).to(dev)
    v = torch.from_numpy(oracle.normal(9, (rows + 1, kv_dim))).to(dev)
    scale = oracle.attn_scale(hd)
    qf, of = q.clone(), torch.full_like(q, float("nan"))
    step = fused.RoPEDecodeStep if rope else fused.DecodeStep
    step(of, qf, k, v, 0, btd, sl, H, scale, max(lens))
    fused.synchronize()
    qp, op = q.clone(), torch.full_like(q, float("nan"))
    if rope:
        parts.RoPEWriteAtLen(0, btd, sl, qp, k, v)
    else:
        parts.WriteAtLen(0, btd, sl, k, v)
    parts.AttentionGQA(op, qp, 0, btd, sl, H, scale, max(lens))
    parts.synchronize()
    assert torch.equal(qf, qp)
    every = torch.arange(pages, dtype=torch.int32, device=dev)
    for x, y in zip(fused.Get(0, every, pages * P), parts.Get(0, every, pages * P)):
        assert torch.equal(x, y)
    assert torch.equal(of, op)
