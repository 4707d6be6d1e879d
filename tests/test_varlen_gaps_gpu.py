"""Packed rows that no sequence covers read 0 in outputs and gradients: the
kernels zero them (o_rows, dq_rows, dkv_rows) in tensors that start with other
values, and touch no other row."""

import ctypes

import pytest
import torch

import fa_capi
import flash_attention_interface as fai
from helpers import randn16


def _poisoned(shape, device):
    """Leave sevens where the caching allocator takes the next tensors of this size from."""
    for _ in range(3):
        torch.full(shape, 7.0, dtype=torch.float16, device=device)


# (cumulative offsets, rows, max_seqlen): no gap and an empty sequence; rows before and after the sequences; a long
# tail; more sequences than the 1024 gaps looked at at a time, with the end's gap in the second lot.
CASES = [
    ([0, 70, 70, 200], 200, 130),
    ([5, 70, 203], 260, 133),
    ([0, 3], 5000, 3),
    ([3 * i for i in range(1501)], 4510, 3),
]


@pytest.mark.gpu
@pytest.mark.parametrize("h,hk,hd", [(4, 2, 64), (3, 3, 128)])
@pytest.mark.parametrize("case", range(len(CASES)))
def test_uncovered_rows(device, case, h, hk, hd):
    cu, rows, longest = CASES[case]
    g = torch.Generator().manual_seed(8800 + case)
    q, do = randn16((rows, h, hd), g).to(device), randn16((rows, h, hd), g).to(device)
    k, v = randn16((rows, hk, hd), g).to(device), randn16((rows, hk, hd), g).to(device)
    cud = torch.tensor(cu, dtype=torch.int32, device=device)
    b, s = len(cu) - 1, hd ** -0.5
    print(f"case gaps {case} h={h} hd={hd}", flush=True)

    def run(fill, flag, ordered):
        o, dq, dk, dv = (torch.full_like(t, fill) for t in (q, q, k, v))
        lse = torch.empty((b, h, longest), device=device)
        dsum = torch.empty((2, b, h, longest), device=device)
        fa = fa_capi.fwd_args(q, k, v, o, lse, s, True, cud, cud, longest, longest)
        ba = fa_capi.bwd_args(q, k, v, o, lse, do, dq, dk, dv, dsum, s, True, cud, cud, longest, longest)
        fo = torch.empty(fa_capi.load().fa_fwd_order_len(ctypes.byref(fa)), dtype=torch.int32, device=device)
        bo = torch.empty(fa_capi.load().fa_bwd_order_len(ctypes.byref(ba)), dtype=torch.int32, device=device)
        if ordered:
            fa.work_order, ba.work_order = fo.data_ptr(), bo.data_ptr()
        if flag:
            fa.o_rows = ba.dq_rows = ba.dkv_rows = rows
        fa_capi.call("fa_fwd", fa)
        fa_capi.call("fa_bwd", ba)
        torch.cuda.synchronize()
        return o, dq, dk, dv

    ref = run(0.0, False, True)
    for ordered in (True, False):
        for x, r in zip(run(7.0, True, ordered), ref):
            assert torch.equal(x, r), "the rows of no sequence, and only those, are zeroed"
    covered = torch.zeros(rows, dtype=torch.bool)
    for x, y in zip(cu, cu[1:]):
        covered[x:y] = True
    for t in (q, do, k, v):
        _poisoned(t.shape, device)
    qg, kg, vg = (t.clone().requires_grad_() for t in (q, k, v))
    out = fai.flash_attn_varlen_func(qg, kg, vg, cud, cud, longest, longest, causal=True)
    out.backward(do)
    for t in (out.detach(), qg.grad, kg.grad, vg.grad):
        assert not t[~covered.to(device)].any()
    kv = torch.stack([k, v], 1).requires_grad_()
    _poisoned(kv.shape, device)
    fai.flash_attn_varlen_kvpacked_func(q.clone().requires_grad_(), kv, cud, cud, longest, longest,
                                        causal=True).backward(do)
    assert torch.equal(kv.grad[:, 0], kg.grad) and torch.equal(kv.grad[:, 1], vg.grad)
