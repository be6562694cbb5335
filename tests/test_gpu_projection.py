"""The decode attention's projections at 17 to 128 rows (gemm_proj_kernel:
bias + RoPE, and bias + residual, in its epilogue), and with fp8 weights at
any row count up to that, against the float64 oracle, on both sides of the
lines to the split product and to the register kernel.

Bounds.  v_new is one product: K exact bf16 products summed in fp32 in any
order (at most K 2^-24 sum |x w|), then one rounding to bf16 (2^-8 |v|).  k_new
is two such products turned by an angle whose cosine and sine are rounded to
fp32.  fp8 weights are e4m3 values times a power of two with every column's
largest at 448 of it, so that their quantisation is exact."""

from __future__ import annotations

import numpy as np
import pytest
import torch

from oracle import attention as oa
from oracle import numerics as nm
from helpers import assert_close_rms

pytestmark = pytest.mark.gpu


def _bf16(a):
    return nm.bf16_round(np.asarray(a, np.float32))


def _weights(rng, n_in, n_out, fp8):
    if not fp8:
        return _bf16(rng.standard_normal((n_in, n_out)) * n_in ** -0.5)
    w = np.clip(rng.standard_normal((n_in, n_out)).astype(np.float32) * 100, -448, 448)  # above 464 torch gives NaN
    w = torch.from_numpy(w).to(torch.float8_e4m3fn).float()
    w[rng.integers(0, n_in, n_out), np.arange(n_out)] = 448.0
    # std about n_in^-0.5, so that the scores stay of order 1 and the softmax
    # does not amplify the rounding of the normalised rows
    return (w * 2.0 ** round(np.log2(n_in ** -0.5 / 100))).numpy()


# B: both sides of each row-tile count; n_embd 64 and 192: fewer units than
# waves, and a wave without any; 4160 columns of Q/K/V: two column groups per
# block; head sizes below and above a column group.  The last two rows: both
# sides of the row limits (96 and 64 rows of Q/K/V 4096 -> 6144, 96 and 128 of
# 3072 -> 4608), and 9216 columns of Q/K/V at 12 and 13 rows with fp8 weights
# (288 blocks of two column groups, a second round nearly empty).
@pytest.mark.parametrize("B,n_embd,H,Hkv,fp8,bias", [
    (17, 64, 4, 2, False, True), (32, 192, 6, 6, False, False), (33, 2560, 40, 10, False, True),
    (48, 512, 4, 4, False, False), (49, 256, 16, 2, False, True), (64, 2560, 20, 20, False, True),
    (65, 512, 4, 2, False, True), (96, 128, 2, 1, False, False), (97, 2560, 40, 10, False, False),
    (128, 256, 8, 1, False, True), (129, 256, 8, 1, False, True),
    (1, 64, 4, 2, True, True), (16, 2560, 40, 10, True, False), (17, 192, 6, 6, True, True),
    (64, 2560, 20, 20, True, False), (100, 256, 2, 2, True, True),
    (96, 4096, 32, 8, False, True), (97, 4096, 32, 8, False, True), (65, 4096, 32, 8, True, False),
    (97, 3072, 24, 6, True, True), (12, 3072, 24, 24, True, True), (13, 3072, 24, 24, True, True),
])
def test_projections(fm, B, n_embd, H, Hkv, fp8, bias):
    rng = np.random.default_rng(B * 31 + n_embd)
    D, nkv = n_embd // H, Hkv * (n_embd // H)
    ws = [_weights(rng, n_embd, n, fp8) for n in (n_embd, nkv, nkv, n_embd)]
    bs = [(rng.standard_normal(n) * 0.1).astype(np.float32) for n in (n_embd, nkv, nkv, n_embd)]
    x = _bf16(rng.standard_normal((B, n_embd)))
    res = _bf16(rng.standard_normal((B, n_embd)))
    kc, vc = (_bf16(rng.standard_normal((B, 3, Hkv, D))) for _ in range(2))
    pos = rng.integers(0, 100000, B).astype(np.int64)
    dev = lambda a: torch.from_numpy(np.ascontiguousarray(a)).cuda().bfloat16()  # noqa: E731
    blk = fm.AttentionBlockDecode(*(dev(w) for w in ws), *(torch.from_numpy(b).cuda() for b in bs), use_bias=bias,
                                  n_head=H, n_head_kv=Hkv, n_embd=n_embd, act_dtype=torch.bfloat16,
                                  weight_dtype="fp8" if fp8 else None)
    out, k_new, v_new = (t.float().cpu().numpy() for t in blk(dev(x), pos, dev(kc), dev(vc)))
    barg = bs if bias else [None] * 4
    ref, rk, rv = oa.attention_block_decode(x, pos, kc, vc, *ws, *barg, bias, H, Hkv, n_embd)
    mag = [np.abs(x).astype(np.float64) @ np.abs(w) + (np.abs(b) if bias else 0) for w, b in zip(ws[1:3], bs[1:3])]
    km, vm = (((n_embd + 2) * 2.0 ** -24 * m).reshape(B, Hkv, D) for m in mag)
    assert np.all(np.abs(v_new - rv) <= vm + 2.0 ** -8 * np.abs(rv))
    turned = np.repeat(km.reshape(B, Hkv, D // 2, 2).sum(-1), 2, axis=-1).reshape(B, Hkv, D)
    length = np.repeat(np.sqrt((rk**2).reshape(B, Hkv, D // 2, 2).sum(-1)), 2, axis=-1).reshape(B, Hkv, D)
    assert np.all(np.abs(k_new - rk) <= turned + 2.0 ** -8 * np.abs(rk) + 2.0 ** -21 * length)
    assert_close_rms(out, ref, 2e-2, what=f"output B={B}")

    # the residual added after the rounded output, in place
    nw = _bf16(np.ones(n_embd))
    n_blocks, table = B, np.arange(B, dtype=np.int32).reshape(1, B, 1)
    kp, vp = (np.concatenate([c, np.zeros((B, 1, Hkv, D), np.float32)], axis=1) for c in (kc, vc))
    lens = np.full((1, B), 3, np.int32)
    r = dev(res)
    got, _, _ = blk.paged_sublayer(r, dev(nw), 1e-5, pos, dev(kp), dev(vp), 0, table, lens, 3,
                                   np.arange(n_blocks, dtype=np.int32), np.full(B, 3, np.int32), out=r)
    ref, *_ = oa.attention_sublayer_decode_paged(res, nw, 1e-5, pos, kp, vp, 0, table, lens, 3,
                                                 np.arange(n_blocks), np.full(B, 3), *ws, *barg, bias, H, Hkv, n_embd)
    assert_close_rms(got.float().cpu().numpy(), ref, 2e-2, what=f"sub-layer B={B}")
