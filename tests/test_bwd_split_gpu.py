"""dK/dV with several workgroups on each key block (fa_bwd_args.split_ws): the
shares of a block's steps are cut anywhere, across query heads and through the
causal diagonal, and their fp32 partial sums added in order.  Against the
unsplit kernel (the same fp16 products, fp32 sums in another order) and the
oracle."""

import ctypes

import pytest
import torch

import fa_capi
import flash_attention_interface as fai
from helpers import assert_2x, check_fwd_bwd, check_varlen, cu_from_lengths, randn16
from oracle.attention import attention_bwd, attention_fwd, bwd_fp32_noise
from oracle.twin import bwd_twin, fwd_twin


def _args(q, k, v, do, s, causal, cu_q=None, cu_k=None, mq=0, mk=0):
    o, grads = torch.empty_like(q), [torch.full_like(t, 7.0) for t in (q, k, v)]
    shape = (q.shape[0], q.shape[2], q.shape[1]) if cu_q is None else (cu_q.numel() - 1, q.shape[1], mq)
    lse = torch.empty(shape, device=q.device)
    dsum = torch.empty((2,) + shape, device=q.device)
    fa_capi.call("fa_fwd", fa_capi.fwd_args(q, k, v, o, lse, s, causal, cu_q, cu_k, mq, mk))
    return fa_capi.bwd_args(q, k, v, o, lse, do, *grads, dsum, s, causal, cu_q, cu_k, mq, mk), o, lse, grads


def _split_ws(ba, device):
    n = fa_capi.load().fa_bwd_split_bytes(ctypes.byref(ba))
    assert n > 0, "the shape must select the split kernel"
    ws = torch.full((n,), 255, dtype=torch.uint8, device=device)
    ba.split_ws, ba.split_ws_bytes = ws.data_ptr(), n
    return ws


# batch, sq, sk, h, hk, hd, causal: shares through the diagonal and across heads; ragged ends; sq != sk both
# ways (keys that no query sees, queries that see no key); more shares than steps; both head dims; S from 2 to 16.
CASES = [
    (1, 512, 512, 8, 2, 128, True),
    (1, 257, 500, 12, 1, 128, True),
    (1, 700, 300, 6, 2, 64, True),
    (1, 33, 900, 32, 2, 128, False),
    (1, 2050, 2060, 2, 2, 64, True),
    (1, 1000, 130, 8, 1, 64, False),
    (2, 129, 129, 16, 4, 128, True),
    (1, 1100, 1100, 16, 16, 128, True),
]


@pytest.mark.gpu
@pytest.mark.parametrize("b,sq,sk,h,hk,hd,causal", CASES)
def test_split_dkdv(device, b, sq, sk, h, hk, hd, causal):
    g = torch.Generator().manual_seed(8100 + sq + 3 * sk + h + hd)
    q, do = randn16((b, sq, h, hd), g), randn16((b, sq, h, hd), g)
    k, v = randn16((b, sk, hk, hd), g), randn16((b, sk, hk, hd), g)
    s = hd ** -0.5
    print(f"case split b={b} sq={sq} sk={sk} h={h} hk={hk} hd={hd} causal={causal}", flush=True)
    ba, o, lse, grads = _args(*(t.to(device) for t in (q, k, v, do)), s, causal)
    fa_capi.call("fa_bwd", ba)
    plain = [t.clone() for t in grads]
    ws = _split_ws(ba, device)
    for entry in ("fa_bwd", "fa_bwd_dkdv", "fa_bwd_preprocess"):  # the counters are left cleared, or cleared again
        for t in grads[1:]:
            t.fill_(7.0)
        fa_capi.call(entry, ba)
        if entry == "fa_bwd_preprocess":
            ws.fill_(255)
            fa_capi.call(entry, ba)
            fa_capi.call("fa_bwd_dkdv", ba)
        torch.cuda.synchronize()
        got = [t.clone() for t in grads]
        assert torch.equal(got[0], plain[0])
        if entry == "fa_bwd":
            first = got
        elif entry == "fa_bwd_dkdv":  # D from the same kernel: the same bits whichever workgroup comes last
            assert torch.equal(got[1], first[1]) and torch.equal(got[2], first[2])
        o_ref, l_ref = attention_fwd(q, k, v, s, causal)
        g_ref = attention_bwd(q, k, v, o_ref, l_ref, do, s, causal)
        o_tw, l_tw = fwd_twin(q, k, v, s, causal)
        g_tw = bwd_twin(q, k, v, o_tw, l_tw, do, s, causal)
        noise = bwd_fp32_noise(q, k, v, o_ref, l_ref, do, s, causal)
        for name, x, r, t, n in zip(("dq", "dk", "dv"), got, g_ref, g_tw, noise):
            assert_2x(name, x.cpu(), r, t, n)


@pytest.mark.gpu
@pytest.mark.parametrize("ordered", [False, True])
def test_split_dkdv_varlen(device, ordered):
    """Sequences of mixed lengths, one without queries and one without keys, in natural and device-built order."""
    lens_q, lens_k, h, hk, hd, s = [300, 0, 77, 640, 33], [290, 50, 0, 700, 33], 8, 2, 128, 128 ** -0.5
    g = torch.Generator().manual_seed(8200)
    cu_q, cu_k = cu_from_lengths(lens_q), cu_from_lengths(lens_k)
    q, do = randn16((sum(lens_q), h, hd), g), randn16((sum(lens_q), h, hd), g)
    k, v = randn16((sum(lens_k), hk, hd), g), randn16((sum(lens_k), hk, hd), g)
    ba, o, lse, grads = _args(*(t.to(device) for t in (q, k, v, do)), s, True, cu_q.to(device), cu_k.to(device), 640,
                              700)
    if ordered:
        order = torch.empty(fa_capi.load().fa_bwd_order_len(ctypes.byref(ba)), dtype=torch.int32, device=device)
        ba.work_order = order.data_ptr()
    ws = _split_ws(ba, device)  # noqa: F841  (kept alive)
    fa_capi.call("fa_bwd", ba)
    torch.cuda.synchronize()
    check_varlen("split varlen", cu_q, cu_k, q, k, v, do, o.cpu(), lse.cpu(), tuple(t.cpu() for t in grads), s, True)


@pytest.mark.gpu
@pytest.mark.parametrize("short_by", [1, None])
def test_small_workspace_is_not_touched(device, short_by):
    """A split_ws below fa_bwd_split_bytes (by a byte, or all but 8 bytes of it) gives the unsplit kernel's bits and is
    not written (the buffer behind the pointer has the whole size)."""
    b, sq, sk, h, hk, hd = 1, 512, 512, 8, 2, 128
    g = torch.Generator().manual_seed(8300)
    q, do = randn16((b, sq, h, hd), g).to(device), randn16((b, sq, h, hd), g).to(device)
    k, v = randn16((b, sk, hk, hd), g).to(device), randn16((b, sk, hk, hd), g).to(device)
    print(f"case small workspace short_by={short_by}", flush=True)
    ba, o, lse, grads = _args(q, k, v, do, hd ** -0.5, True)
    fa_capi.call("fa_bwd", ba)
    plain = [t.clone() for t in grads]
    ws = _split_ws(ba, device)
    ba.split_ws_bytes = ws.numel() - short_by if short_by else 8
    for entry in ("fa_bwd", "fa_bwd_preprocess"):
        fa_capi.call(entry, ba)
        torch.cuda.synchronize()
        assert bool((ws == 255).all()), entry
        assert all(torch.equal(x, y) for x, y in zip(grads, plain))


def test_split_bytes_rule():
    """Sizes that fill the chip by themselves take no workspace; the partials stay within 256 MiB."""
    def size(b, sq, sk, h, hk, hd, causal):
        ba = fa_capi.FaBwdArgs()
        ba.batch, ba.seqlen_q, ba.seqlen_k, ba.nheads, ba.nheads_k = b, sq, sk, h, hk
        ba.head_dim, ba.lse_seqlen, ba.causal = hd, sq, int(causal)
        return fa_capi.load().fa_bwd_split_bytes(ctypes.byref(ba))

    assert size(4, 4096, 4096, 16, 16, 128, True) == 0
    assert size(4, 1024, 1024, 16, 16, 128, True) == 0
    assert size(0, 64, 64, 2, 2, 64, True) == 0 and size(1, 0, 64, 2, 2, 64, True) == 0
    assert size(1, 8192, 8192, 32, 8, 128, True) > 0
    for case in CASES + [(1, 1 << 20, 1 << 20, 8, 1, 128, True), (1, 16384, 16384, 32, 8, 128, True)]:
        assert size(*case) <= (256 << 20) + (1 << 20)


@pytest.mark.gpu
@pytest.mark.parametrize("b,sq,sk,h,hk,hd", [(3, 700, 700, 16, 16, 64), (3, 600, 777, 20, 20, 128)])
def test_paired_items(device, b, sq, sk, h, hk, hd):
    """Causal grids between one and two workgroups per CU, whose second layer is taken backwards (an odd number of
    items in it): every query and key block once, against the oracle."""
    cus = torch.cuda.get_device_properties(0).multi_processor_count
    for blocks in ((sq + 127) // 128, (sk + 127) // 128):
        assert cus < blocks * b * h <= 2 * cus and sk > 512, "the shape must select the pairing"
    g = torch.Generator().manual_seed(8900 + sq + hd)
    q, do = randn16((b, sq, h, hd), g), randn16((b, sq, h, hd), g)
    k, v = randn16((b, sk, hk, hd), g), randn16((b, sk, hk, hd), g)
    s = hd ** -0.5
    print(f"case paired sq={sq} sk={sk} hd={hd}", flush=True)
    ba, o, lse, grads = _args(*(t.to(device) for t in (q, k, v, do)), s, True)
    fa_capi.call("fa_bwd", ba)
    torch.cuda.synchronize()
    check_fwd_bwd("paired", q, k, v, do, o.cpu(), lse.cpu(), tuple(t.cpu() for t in grads), s, True)


@pytest.mark.gpu
@pytest.mark.parametrize("before", ["fa_bwd_dq", "fa_bwd_preprocess"])
def test_dkdv_clears_its_own_counters(device, before):
    """fa_bwd_dkdv with a workspace that the call before it did not have, then once more on the same one."""
    b, sq, sk, h, hk, hd = 1, 512, 400, 8, 2, 64
    g = torch.Generator().manual_seed(8400)
    q, do = randn16((b, sq, h, hd), g).to(device), randn16((b, sq, h, hd), g).to(device)
    k, v = randn16((b, sk, hk, hd), g).to(device), randn16((b, sk, hk, hd), g).to(device)
    print(f"case own counters before={before}", flush=True)
    ba, o, lse, grads = _args(q, k, v, do, hd ** -0.5, True)
    fa_capi.call(before, ba)
    ws = _split_ws(ba, device)  # its counters hold -1
    got = []
    for _ in range(2):
        for t in grads[1:]:
            t.fill_(7.0)
        fa_capi.call("fa_bwd_dkdv", ba)
        torch.cuda.synchronize()
        got.append([t.clone() for t in grads[1:]])
    fa_capi.call(before, ba)
    ws.zero_()
    fa_capi.call("fa_bwd_dkdv", ba)
    torch.cuda.synchronize()
    for x, y, z in zip(*got, grads[1:]):
        assert torch.equal(x, z) and torch.equal(y, z)


@pytest.mark.gpu
def test_split_workspace_is_optional_memory(device):
    """A training step that fits in memory without the shares' workspace still runs: the extension does without it."""
    b, sq, h, hk, hd = 1, 8192, 32, 8, 128
    g = torch.Generator().manual_seed(8500)
    q, do = randn16((b, sq, h, hd), g).to(device), randn16((b, sq, h, hd), g).to(device)
    k, v = randn16((b, sq, hk, hd), g).to(device), randn16((b, sq, hk, hd), g).to(device)
    s = hd ** -0.5
    print("case optional workspace", flush=True)
    ba, o, lse, grads = _args(q, k, v, do, s, True)
    need = fa_capi.load().fa_bwd_split_bytes(ctypes.byref(ba))
    fa_capi.call("fa_bwd", ba)  # unshared
    torch.cuda.synchronize()
    torch.cuda.empty_cache()
    room = sum(t.numel() * t.element_size() for t in grads) + (32 << 20)
    assert need > room
    total = torch.cuda.get_device_properties(device).total_memory
    torch.cuda.set_per_process_memory_fraction((torch.cuda.memory_reserved() + room) / total)
    try:
        got = fai._flash_attn_backward(do, q, k, v, o, lse, s, True)
        torch.cuda.synchronize()
    finally:
        torch.cuda.set_per_process_memory_fraction(1.0)
    assert all(torch.equal(x, y) for x, y in zip(got, grads))
