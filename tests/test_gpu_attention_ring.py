"""bf16 paged attention with head_dim 64 and 128 (attn_ring_kernel) against the
oracle, at the edges of its 16-position tiles, 64-position chunks, 256- to
1024-position splits and blocks of 1, 2 and 4 waves.

The output projection is the identity, so the output is the attention itself
rounded to bf16 once (2^-9 relative); q is carried to about 16 significant
bits, which moves a score of order 1 by 2^-16 of the sum of its products'
magnitudes (under 1e-3 here) and an output by less than half a percent of its
RMS: 1e-2 in all."""

from __future__ import annotations

import numpy as np
import pytest
import torch

from oracle import attention as oa
from oracle import numerics as nm
from helpers import assert_close_rms

pytestmark = pytest.mark.gpu

EDGES = [0, 1, 15, 16, 17, 63, 64, 65, 127, 191, 192, 255, 256, 257, 320, 449, 511, 512, 513, 769]


# (lens, n_embd, H, Hkv, block_size): every query group size with both head
# sizes, block sizes that no tile divides; 64 sequences x 8 heads, whose splits
# hold 512 and 1024 positions (contexts up to 520 and 1100, the short last
# splits behind the full ones); more than 512 pairs of at most 64 and 128
# positions (blocks of one and two waves); 8 query heads x 128: more than 256
# pairs of at most 64 and 300, 1024 of at most 200 (one wave per 256
# positions), and 128 pairs of 1250, in splits of 768.
@pytest.mark.parametrize("lens,n_embd,H,Hkv,bs", [
    (EDGES, 128, 1, 1, 16), (EDGES, 128, 2, 1, 5), (EDGES, 256, 4, 1, 32), (EDGES, 512, 8, 1, 7),
    (EDGES, 128, 2, 2, 64), (EDGES, 256, 2, 1, 3), (EDGES, 512, 4, 1, 16), (EDGES, 1024, 8, 1, 1),
    ([520] + [1 + 8 * i for i in range(64)] + [513], 512, 8, 8, 16),
    ([1100, 1025, 1024, 1023, 961, 960, 4] + [17 * i for i in range(57)], 512, 8, 8, 32),
    ([64, 63, 17, 4] + [i % 65 for i in range(62)], 512, 8, 8, 16),
    ([64, 1, 0, 33] + [i % 65 for i in range(62)], 1024, 8, 8, 16),
    ([128, 127, 65, 64] + [2 * i % 129 for i in range(62)], 512, 8, 8, 16),
    ([128, 64, 0, 66] + [2 * i % 129 for i in range(62)], 2048, 16, 8, 16),
    ([64, 63, 17, 4] + [i % 65 for i in range(130)], 2048, 16, 2, 16),
    ([300, 257, 256, 200, 65] + [3 * i % 301 for i in range(125)], 2048, 16, 2, 16),
    ([200, 65, 64, 129, 193] + [i % 201 for i in range(1020)], 1024, 8, 1, 16),
    ([1250, 769, 768, 767, 1024] + [20 * i for i in range(59)], 2048, 16, 2, 16),
])
def test_ring_edges(fm, lens, n_embd, H, Hkv, bs):
    rng = np.random.default_rng(len(lens) * n_embd + bs)
    B, D, max_ctx = len(lens), n_embd // H, max(lens)
    bf = lambda a: nm.bf16_round(np.asarray(a, np.float32))  # noqa: E731
    per = max_ctx // bs + 1
    n_blocks = B * per
    tables = rng.permutation(n_blocks).reshape(1, B, per).astype(np.int32)
    kp, vp = (bf(rng.standard_normal((n_blocks, bs, Hkv, D))) for _ in range(2))
    # entries outside the pool read as zero rows: a whole sequence, and one
    # block in the middle of another
    tables[0, 3, :] = n_blocks
    tables[0, B - 1, per // 2] = -1
    w = [bf(rng.standard_normal((n_embd, n)) * n_embd ** -0.5) for n in (n_embd, Hkv * D, Hkv * D)]
    w.append(np.eye(n_embd, dtype=np.float32))
    x = bf(rng.standard_normal((B, n_embd)))
    pos = np.asarray(lens, np.int64)
    lens2 = np.asarray(lens, np.int32).reshape(1, B)
    slot_b, slot_p = np.full(B, -1, np.int32), np.zeros(B, np.int32)  # no write-back
    dev = lambda a: torch.from_numpy(np.ascontiguousarray(a)).cuda().bfloat16()  # noqa: E731
    blk = fm.AttentionBlockDecode(*(dev(m) for m in w), n_head=H, n_head_kv=Hkv, n_embd=n_embd,
                                  act_dtype=torch.bfloat16)
    kd, vd = dev(kp), dev(vp)
    out, _, _ = blk.paged(dev(x), pos, kd, vd, 0, tables, lens2, max_ctx, slot_b, slot_p)
    # the oracle indexes the pool directly: a zero block stands in for the
    # entries outside it
    zb = np.zeros((1, bs, Hkv, D), np.float32)
    t2 = np.where((tables < 0) | (tables >= n_blocks), n_blocks, tables)
    kc = oa.kv_gather(np.concatenate([kp, zb]), 0, t2, lens2, max_ctx)
    vc = oa.kv_gather(np.concatenate([vp, zb]), 0, t2, lens2, max_ctx)
    ref, _, _ = oa.attention_block_decode(x, pos, kc, vc, *w, None, None, None, None, False, H, Hkv, n_embd)
    got = out.float().cpu().numpy()
    for b in range(B):
        assert_close_rms(got[b], ref[b], 1e-2, what=f"context {lens[b]}")
    assert torch.equal(kd, dev(kp)) and torch.equal(vd, dev(vp))


def test_ring_does_not_use_rows_past_the_context(fm):
    """NaN and infinity in the pool's other rows stay out of the result."""
    rng = np.random.default_rng(5)
    B, n_embd, H, Hkv, bs, D = 2, 256, 2, 1, 16, 128
    kp, vp = (torch.full((8, bs, Hkv, D), float("nan")).cuda().bfloat16() for _ in range(2))
    vp[:, 1::2] = float("inf")
    tables = np.array([[[6, 2, 4], [5, 1, 3]]], np.int32)
    lens = np.array([[33, 7]], np.int32)
    for b in range(B):
        for j in range(lens[0, b]):
            kp[tables[0, b, j // bs], j % bs] = torch.from_numpy(rng.standard_normal((Hkv, D))).cuda().bfloat16()
            vp[tables[0, b, j // bs], j % bs] = torch.from_numpy(rng.standard_normal((Hkv, D))).cuda().bfloat16()
    w = [torch.from_numpy(rng.standard_normal((n_embd, n)).astype(np.float32) * n_embd ** -0.5).cuda().bfloat16()
         for n in (n_embd, D, D, n_embd)]
    blk = fm.AttentionBlockDecode(*w, n_head=H, n_head_kv=Hkv, n_embd=n_embd, act_dtype=torch.bfloat16)
    x = torch.from_numpy(rng.standard_normal((B, n_embd)).astype(np.float32)).cuda().bfloat16()
    out, _, _ = blk.paged(x, lens[0].astype(np.int64), kp, vp, 0, tables, lens, 40, np.full(B, -1, np.int32),
                          np.zeros(B, np.int32))
    assert torch.isfinite(out).all()


@pytest.mark.parametrize("D", [64, 128])
@pytest.mark.parametrize("masked", [(0, 64), (64, 128), (0, 256), (256, 300), (0, 300), (10, 290)])
def test_ring_scores_of_minus_infinity(fm, D, masked):
    """Cached keys of bf16's lowest value whose scores overflow to minus
    infinity take no part, also where they fill a 64-position chunk of a wave,
    a whole split, or the whole context."""
    bs, ctx, q0 = 16, 300, 1000.0
    rng = np.random.default_rng(D + masked[0])
    w, zero = torch.zeros((D, D)), torch.zeros((D, D))
    w[0, 0] = 1.0  # the query is x's first channel, the new token's key and value are zero
    blk = fm.AttentionBlockDecode(*(m.cuda().bfloat16() for m in (w, zero, zero, torch.eye(D))), n_head=1, n_head_kv=1,
                                  n_embd=D, act_dtype=torch.bfloat16)
    x = torch.zeros((1, D))
    x[0, 0] = q0
    n_blocks = ctx // bs + 1
    k = np.zeros((n_blocks * bs, D), np.float32)
    v = nm.bf16_round(rng.standard_normal((n_blocks * bs, D)).astype(np.float32))
    k[:, 0] = nm.bf16_round((rng.standard_normal(n_blocks * bs) * 1e-2).astype(np.float32))
    k[masked[0]:masked[1], 0] = torch.finfo(torch.bfloat16).min
    kd, vd = (torch.from_numpy(a).cuda().bfloat16().view(n_blocks, bs, 1, D) for a in (k, v))
    out, _, _ = blk.paged(x.cuda().bfloat16(), np.zeros(1, np.int64), kd, vd, 0,
                          np.arange(n_blocks, dtype=np.int32).reshape(1, 1, n_blocks), np.array([[ctx]], np.int32), ctx,
                          np.full(1, -1, np.int32), np.zeros(1, np.int32))
    keep = np.r_[0:masked[0], masked[1]:ctx]
    score = np.append(q0 * D ** -0.5 * k[keep, 0].astype(np.float64), 0.0)  # the last: the new token's
    p = np.exp(score - score.max())
    assert_close_rms(out.float().cpu().numpy()[0], p[:-1] @ v[keep] / p.sum(), 1e-2)
