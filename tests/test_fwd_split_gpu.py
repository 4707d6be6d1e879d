"""The forward on grids too small for the chip: two wave groups per workgroup
share a query block's keys, and with fa_fwd_args.split_ws several workgroups do
(fwd_plan).  Against the oracle at the sizes where the shares end (odd block
counts, fewer blocks than shares for some rows, rows without keys, one query),
GQA against expanded MHA bit for bit, and whichever workgroup comes last."""

import ctypes

import pytest
import torch

import fa_capi
import flash_attention_interface as fai
from helpers import assert_2x, assert_lse, check_varlen, cu_from_lengths, kv_oracle, randn16
from oracle.attention import attention_fwd
from oracle.twin import fwd_twin


def _fa(b, sq, sk, h, hk, hd, causal):
    a = fa_capi.FaFwdArgs()
    a.batch, a.seqlen_q, a.seqlen_k, a.nheads, a.nheads_k = b, sq, sk, h, hk
    a.head_dim, a.lse_seqlen, a.causal = hd, sq, int(causal)
    return fa_capi.load().fa_fwd_split_bytes(ctypes.byref(a))


# batch, sq, sk, h, hk, hd, causal, whether workgroups share (2 to 16 of them).  Without: one group on one key block,
# two groups of 2 row waves (64-row blocks, from two key blocks to the most of that plan), then of 4.
CASES = [
    (1, 130, 2500, 8, 2, 128, True, True),
    (1, 40, 5000, 6, 2, 64, False, True),
    (1, 300, 2100, 4, 4, 128, True, True),
    (1, 1800, 1750, 2, 1, 128, True, True),
    (2, 1, 2000, 16, 16, 128, False, True),
    (1, 17, 9000, 2, 2, 128, True, True),
    (1, 20, 30, 2, 1, 128, False, False),
    (1, 65, 64, 6, 2, 64, True, False),
    (1, 20, 65, 2, 1, 128, False, False),
    (2, 70, 100, 6, 2, 64, True, False),
    (1, 509, 509, 32, 8, 128, True, False),
    (2, 512, 777, 6, 2, 64, False, False),
    (3, 257, 520, 4, 4, 128, True, False),
    (1, 900, 700, 4, 1, 64, True, False),
    (2, 500, 333, 16, 4, 128, True, False),
    (1, 1020, 1030, 32, 4, 64, True, False),
    (1, 1020, 1030, 32, 4, 128, True, False),
    (1, 2100, 2100, 28, 4, 128, True, False),
]


@pytest.mark.gpu
@pytest.mark.parametrize("b,sq,sk,h,hk,hd,causal,split", CASES)
def test_fwd_shares(device, b, sq, sk, h, hk, hd, causal, split):
    assert (_fa(b, sq, sk, h, hk, hd, causal) > 0) == split
    g = torch.Generator().manual_seed(8500 + sq + 3 * sk + h + hd)
    q, k, v = randn16((b, sq, h, hd), g), randn16((b, sk, hk, hd), g), randn16((b, sk, hk, hd), g)
    k[:, sk // 2:] *= 4  # the row maxima differ between the shares
    s = hd ** -0.5
    print(f"case shares b={b} sq={sq} sk={sk} h={h} hk={hk} hd={hd} causal={causal}", flush=True)
    qd, kd, vd = (t.to(device) for t in (q, k, v))
    out, lse = fai._flash_attn_forward(qd, kd, vd, s, causal)
    again, lse2 = fai._flash_attn_forward(qd, kd, vd, s, causal)
    wide = [t.repeat_interleave(h // hk, dim=2).contiguous() for t in (kd, vd)]
    mha, lse_m = fai._flash_attn_forward(qd, *wide, s, causal)
    torch.cuda.synchronize()
    assert torch.equal(out, again) and torch.equal(lse, lse2)
    assert torch.equal(out, mha) and torch.equal(lse, lse_m)
    o_ref, l_ref = attention_fwd(q, k, v, s, causal)
    assert_2x("out", out.cpu(), o_ref, fwd_twin(q, k, v, s, causal)[0])
    assert_lse(lse.cpu(), l_ref)
    if causal and sq > sk:
        assert not out[:, : sq - sk].any() and not lse[:, :, : sq - sk].any()
    # Without the workspace: one workgroup per query block, the same values to rounding.
    o1, l1 = torch.full_like(qd, 7.0), torch.full_like(lse, 7.0)
    fa_capi.call("fa_fwd", fa_capi.fwd_args(qd, kd, vd, o1, l1, s, causal))
    torch.cuda.synchronize()
    assert_2x("out", o1.cpu(), o_ref, fwd_twin(q, k, v, s, causal)[0])
    assert_lse(l1.cpu(), l_ref)


# Few queries of many heads: packed into 128-row workgroups a group's heads leave CUs idle, expanded they fill the
# chip (in 256-row blocks at head_dim 64).  Both take the same plan, one group, two, or shares, which the expanded form's
# workgroups walk several of in turn (all of them; two of three or four).
PACKED = [
    (32, 16, 2048, 16, 2, 64, False, False),
    (32, 100, 2100, 16, 4, 64, True, False),
    (16, 64, 1300, 32, 8, 128, True, False),
    (16, 2, 6500, 16, 4, 128, False, True),
    (8, 33, 4100, 16, 2, 128, True, True),
    (4, 150, 4000, 16, 4, 64, True, True),
]


@pytest.mark.gpu
@pytest.mark.parametrize("b,sq,sk,h,hk,hd,causal,split", PACKED)
def test_packed_heads_have_the_expanded_heads_bits(device, b, sq, sk, h, hk, hd, causal, split):
    assert (_fa(b, sq, sk, h, hk, hd, causal) > 0) == split
    assert (_fa(b, sq, sk, h, h, hd, causal) > 0) == split
    g = torch.Generator().manual_seed(8550 + sq + 3 * sk + h + hd)
    q, k, v = randn16((b, sq, h, hd), g), randn16((b, sk, hk, hd), g), randn16((b, sk, hk, hd), g)
    k[:, sk // 2:] *= 4
    s = hd ** -0.5
    print(f"case packed b={b} sq={sq} sk={sk} h={h} hk={hk} hd={hd} causal={causal}", flush=True)
    qd, kd, vd = (t.to(device) for t in (q, k, v))
    out, lse = fai._flash_attn_forward(qd, kd, vd, s, causal)
    mha, lse_m = fai._flash_attn_forward(
        qd, *(t.repeat_interleave(h // hk, dim=2).contiguous() for t in (kd, vd)), s, causal)
    torch.cuda.synchronize()
    assert torch.equal(out, mha) and torch.equal(lse, lse_m)
    for i in (0, b - 1):
        o_ref, l_ref = attention_fwd(q[i:i + 1], k[i:i + 1], v[i:i + 1], s, causal)
        assert_2x("out", out[i:i + 1].cpu(), o_ref, fwd_twin(q[i:i + 1], k[i:i + 1], v[i:i + 1], s, causal)[0])
        assert_lse(lse[i:i + 1].cpu(), l_ref)


@pytest.mark.gpu
def test_fwd_groups_varlen(device):
    lens_q, lens_k, h, hk, hd, s = [700, 0, 33, 512], [800, 50, 0, 500], 8, 2, 128, 128 ** -0.5
    g = torch.Generator().manual_seed(8600)
    cu_q, cu_k = cu_from_lengths(lens_q), cu_from_lengths(lens_k)
    q = randn16((sum(lens_q), h, hd), g)
    k, v = randn16((sum(lens_k), hk, hd), g), randn16((sum(lens_k), hk, hd), g)
    out, lse = fai._flash_attn_varlen_forward(q.to(device), k.to(device), v.to(device), cu_q.to(device),
                                              cu_k.to(device), 700, 800, s, True)
    torch.cuda.synchronize()
    check_varlen("groups varlen", cu_q, cu_k, q, k, v, None, out.cpu(), lse.cpu(), None, s, True)


@pytest.mark.gpu
def test_fwd_shares_kvcache_chunk(device):
    """A contiguous cache's multi-token call: per-sequence key counts (an empty one, one below the share count)."""
    b, sq, h, hk, hd, cap = 3, 7, 4, 4, 128, 3000
    g = torch.Generator().manual_seed(8700)
    q, k, v = (randn16((b, sq, n, hd), g) for n in (h, hk, hk))
    kc, vc = randn16((b, cap, hk, hd), g), randn16((b, cap, hk, hd), g)
    seqlens = torch.tensor([2993, 0, 100], dtype=torch.int32)
    kd, vd = kc.clone().to(device), vc.clone().to(device)
    out, lse = fai.flash_attn_with_kvcache(q.to(device), kd, vd, k.to(device), v.to(device),
                                           cache_seqlens=seqlens.to(device), causal=True, num_splits=1,
                                           return_softmax_lse=True)
    torch.cuda.synchronize()
    o_ref, l_ref, kc_ref, vc_ref = kv_oracle(q, kc, vc, k, v, seqlens, None, None, True, 1, None)
    assert torch.equal(kd.cpu(), kc_ref) and torch.equal(vd.cpu(), vc_ref)
    # This path rounds P to fp16, which the bound's rounded oracle does not.
    for i in range(b):
        n = int(seqlens[i]) + sq
        tw = fwd_twin(q[i:i + 1], kc_ref[i:i + 1, :n], vc_ref[i:i + 1, :n], hd ** -0.5, True)[0]
        assert_2x("out", out[i:i + 1].cpu(), o_ref[i:i + 1], tw)
    assert_lse(lse.cpu(), l_ref)
