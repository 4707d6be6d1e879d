"""KV-cache calls with many query rows per KV head (kv_chunk_kernel: 128-row
tiles over shared 64-key blocks) against the oracle, at the sizes where its
tiles, blocks, splits and masks end; the same logical cache contiguous, remapped
and paged must give the same bits."""

import pytest
import torch

import flash_attention_interface as fai
from helpers import assert_2x, assert_lse, kv_oracle, randn16
from oracle import kvcache as okv
from test_capi_paths_gpu import _kv_capi
from test_kvcache_gpu import _paged_from_contiguous

# batch, queries, heads, kv heads, head_dim, capacity, appended, lengths before the append, splits, causal, options.
# 64 rows (the least), 65, 127 - 129, a group of 3; keys at block and page edges, an empty cache, fewer keys than
# splits; windows smaller than a tile's positions, keys before a leftpad, every option at once.  (Softcap and ALiBi on
# so few tiles are the split kernel's; test_chunk_ranked has them on this one.)
CASES = [
    (2, 16, 8, 2, 128, 512, 16, (0, 496), 1, True, {}),
    (2, 13, 10, 2, 64, 768, 5, (64, 700), 3, True, {}),
    (1, 43, 3, 1, 128, 1024, 43, (213,), 4, True, {}),
    (3, 32, 8, 2, 64, 512, 0, (512, 1, 0), 5, False, {}),
    (2, 127, 2, 2, 128, 768, 127, (1, 641), 0, True, {}),
    (1, 300, 4, 4, 64, 1280, 300, (900,), 0, True, {}),
    (1, 100, 6, 2, 128, 2048, 100, (1500,), 2, False, {}),
    (2, 33, 8, 2, 128, 1024, 33, (900, 40), 3, True, {"window": (70, -1)}),
    (2, 64, 4, 2, 64, 1024, 64, (950, 100), 2, False, {"window": (5, 200)}),
    (2, 40, 4, 1, 128, 768, 40, (300, 700), 2, True, {"softcap": 15.0, "alibi": True}),
    (2, 40, 4, 1, 64, 768, 40, (300, 700), 0, False, {"leftpad": (33, 650), "alibi": True}),
    (2, 50, 6, 2, 128, 768, 50, (130, 700), 3, True, {"rotary": 64, "window": (200, 0), "softcap": 20.0,
                                                      "leftpad": (100, 0)}),
]


def _call(device, q, kc, vc, k, v, lens, idx, table, splits, causal, kw):
    dev = lambda t: None if t is None else t.to(device)  # noqa: E731
    kcd, vcd = kc.clone().to(device), vc.clone().to(device)
    out, lse = fai.flash_attn_with_kvcache(
        q.to(device), kcd, vcd, k=dev(k), v=dev(v), cache_seqlens=lens.to(device), cache_batch_idx=dev(idx),
        block_table=dev(table), causal=causal, num_splits=splits, return_softmax_lse=True,
        **{n: dev(x) if isinstance(x, torch.Tensor) else x for n, x in kw.items()})
    torch.cuda.synchronize()
    return out.cpu(), lse.cpu(), kcd.cpu(), vcd.cpu()


@pytest.mark.gpu
@pytest.mark.parametrize("case", range(len(CASES)))
def test_kvcache_chunk(device, case):
    b, sq, h, hk, hd, cap, new, lens, splits, causal, opt = CASES[case]
    g = torch.Generator().manual_seed(8300 + case)
    print(f"case chunk {CASES[case]}", flush=True)
    q, kc, vc = randn16((b, sq, h, hd), g), randn16((b, cap, hk, hd), g), randn16((b, cap, hk, hd), g)
    k = randn16((b, new, hk, hd), g) if new else None
    v = randn16((b, new, hk, hd), g) if new else None
    seqlens = torch.tensor(lens, dtype=torch.int32)
    ends = seqlens + new
    window, softcap = opt.get("window", (-1, -1)), opt.get("softcap", 0.0)
    slopes = 2.0 ** -torch.arange(1, h + 1, dtype=torch.float32) if opt.get("alibi") else None
    leftpad = torch.tensor(opt["leftpad"], dtype=torch.int32) if "leftpad" in opt else None
    kw = dict(window_size=window, softcap=softcap, alibi_slopes=slopes, cache_leftpad=leftpad)
    q_ref, k_ref = q, k
    if "rotary" in opt:
        angle = torch.rand((cap, opt["rotary"] // 2), generator=g) * 6.0
        kw.update(rotary_cos=angle.cos().half(), rotary_sin=angle.sin().half(), rotary_interleaved=False)
        pos = seqlens.long()[:, None]
        step = torch.arange(sq)[None, :]
        q_ref = okv.rotary_embed(q, kw["rotary_cos"], kw["rotary_sin"], pos + step, False)
        k_ref = okv.rotary_embed(k, kw["rotary_cos"], kw["rotary_sin"], pos + step[:, :new], False)
    _, _, kc_ref, vc_ref = kv_oracle(q, kc, vc, k_ref, v, seqlens, None, None, causal, 1, None)
    ku, vu = okv.materialize(kc_ref, vc_ref, ends, None, None)
    o_ref, l_ref = okv.splitkv_attention(q_ref, ku, vu, ends, hd ** -0.5, causal, 1, window=window, softcap=softcap,
                                         alibi_slopes=slopes, leftpad=leftpad)
    kp, vp, table = _paged_from_contiguous(kc, vc, torch.full_like(seqlens, cap - new), 256, g)
    perm = torch.randperm(b + 2, generator=g)[:b].to(torch.int32)
    kr, vr = randn16((b + 2, cap, hk, hd), g), randn16((b + 2, cap, hk, hd), g)
    kr[perm.long()], vr[perm.long()] = kc, vc
    got = _call(device, q, kp, vp, k, v, seqlens, None, table, splits, causal, kw)
    assert_2x("out", got[0], o_ref, o_ref.to(torch.float16))
    assert_lse(got[1], l_ref)
    again = _call(device, q, kp, vp, k, v, seqlens, None, table, splits, causal, kw)
    assert torch.equal(got[0], again[0]) and torch.equal(got[1], again[1]), "whichever split finishes last"
    if splits > 1 or opt:  # contiguous caches take this kernel too
        plain = _call(device, q, kc, vc, k, v, seqlens, None, None, splits, causal, kw)
        remap = _call(device, q, kr, vr, k, v, seqlens, perm, None, splits, causal, kw)
        assert torch.equal(plain[2], kc_ref) and torch.equal(plain[3], vc_ref)
        if splits > 1:
            for x in (plain, remap):
                assert torch.equal(x[0], got[0]) and torch.equal(x[1], got[1])
        else:  # the heuristic may cut another capacity into another number of splits
            assert_2x("out", plain[0], o_ref, o_ref.to(torch.float16))
            assert_2x("out", remap[0], o_ref, o_ref.to(torch.float16))


@pytest.mark.gpu
@pytest.mark.parametrize("splits", [1, 2])
def test_chunk_over_1024_pages(device, splits):
    """1100 shuffled pages of 64 tokens: one split of this kernel holds their ids in LDS; the contiguous cache of the
    same tokens gives the same bits (18 KV heads of one tile: this kernel)."""
    g = torch.Generator().manual_seed(8400)
    pages, page, sq, h, hd = 1100, 64, 64, 18, 64
    cap, lens = pages * page, torch.tensor([pages * page - 21], dtype=torch.int32)
    q = randn16((1, sq, h, hd), g)
    gd = torch.Generator(device=device).manual_seed(8401)
    kc, vc = (torch.randn((1, cap, h, hd), generator=gd, device=device, dtype=torch.float16) for _ in range(2))
    table = torch.randperm(pages, generator=g).to(torch.int32)
    kp, vp = (torch.empty((pages, page, h, hd), dtype=torch.float16, device=device) for _ in range(2))
    for dst, src in ((kp, kc), (vp, vc)):
        dst[table.long().to(device)] = src.view(pages, page, h, hd)
    print(f"case over 1024 pages splits={splits}", flush=True)
    kw = dict(causal=True, splits=splits, order=True, fused=splits > 1, calls=("fa_fwd_kvcache",))
    out, lse, _, _ = _kv_capi(device, q, kp, vp, None, None, lens, table.view(1, pages), **kw)
    out2, lse2, _, _ = _kv_capi(device, q, kc, vc, None, None, lens, None, **kw)
    assert torch.equal(out, out2) and torch.equal(lse, lse2)
    for i in (0, h - 1):
        ku, vu = okv.materialize(kc[:, :, i:i + 1].cpu(), vc[:, :, i:i + 1].cpu(), lens, None, None)
        o_ref, l_ref = okv.splitkv_attention(q[:, :, i:i + 1], ku, vu, lens, hd ** -0.5, True, 1)
        assert_2x("out", out[:, :, i:i + 1], o_ref, o_ref.to(torch.float16))
        assert_lse(lse[:, i:i + 1], l_ref)


# Batches of chunks in more items than CUs (12 sequences x 8 KV heads x 2 tiles x 3 splits): sequences in the order of
# their lengths, an empty one among them, later items starting while earlier ones merge.
@pytest.mark.gpu
@pytest.mark.parametrize("hd,opt", [(128, ""), (64, "softcap alibi"), (128, "alibi window"), (64, "leftpad"),
                                    (128, "rotary softcap window leftpad")])
def test_chunk_ranked(device, hd, opt):
    b, sq, h, hk, cap, new, splits = 12, 33, 32, 8, 640, 33, 3
    assert b * hk * 2 * splits > torch.cuda.get_device_properties(0).multi_processor_count, "items must be ranked"
    g = torch.Generator().manual_seed(8500 + hd + len(opt))
    q, kc, vc = randn16((b, sq, h, hd), g), randn16((b, cap, hk, hd), g), randn16((b, cap, hk, hd), g)
    k, v = randn16((b, new, hk, hd), g), randn16((b, new, hk, hd), g)
    seqlens = torch.tensor([0, 607, 31, 300, 64, 600, 1, 450, 128, 95, 520, 200], dtype=torch.int32)
    ends = seqlens + new
    kw = dict(window_size=(150, 0) if "window" in opt else (-1, -1), softcap=15.0 if "softcap" in opt else 0.0,
              alibi_slopes=2.0 ** -torch.arange(1, h + 1, dtype=torch.float32) / 4 if "alibi" in opt else None,
              cache_leftpad=torch.arange(b, dtype=torch.int32) * 3 if "leftpad" in opt else None)
    print(f"case ranked hd={hd} {opt}", flush=True)
    q_ref, k_ref = q, k
    if "rotary" in opt:
        # Quarter turns: exact, so that no element hangs on a rounding by way of fp32 or not.
        turn = torch.randint(0, 4, (cap, 32), generator=g)
        kw.update(rotary_cos=torch.tensor([1.0, 0.0, -1.0, 0.0])[turn].half(),
                  rotary_sin=torch.tensor([0.0, 1.0, 0.0, -1.0])[turn].half(), rotary_interleaved=True)
        at = seqlens.long()[:, None] + torch.arange(sq)[None, :]
        q_ref = okv.rotary_embed(q, kw["rotary_cos"], kw["rotary_sin"], at, True)
        k_ref = okv.rotary_embed(k, kw["rotary_cos"], kw["rotary_sin"], at, True)
    _, _, kc_ref, vc_ref = kv_oracle(q, kc, vc, k_ref, v, seqlens, None, None, True, 1, None)
    ku, vu = okv.materialize(kc_ref, vc_ref, ends, None, None)
    o_ref, l_ref = okv.splitkv_attention(q_ref, ku, vu, ends, hd ** -0.5, True, 1, window=kw["window_size"],
                                         softcap=kw["softcap"], alibi_slopes=kw["alibi_slopes"],
                                         leftpad=kw["cache_leftpad"])
    got = _call(device, q, kc, vc, k, v, seqlens, None, None, splits, True, kw)
    again = _call(device, q, kc, vc, k, v, seqlens, None, None, splits, True, kw)
    assert torch.equal(got[2], kc_ref) and torch.equal(got[3], vc_ref)
    assert torch.equal(got[0], again[0]) and torch.equal(got[1], again[1])
    assert_2x("out", got[0], o_ref, o_ref.to(torch.float16))
    assert_lse(got[1], l_ref)


@pytest.mark.gpu
@pytest.mark.parametrize("pad,window", [((32, 96), (-1, -1)), ((33, 127), (-1, -1)), ((0, 0), (40, 0))])
def test_chunk_ignores_what_unseen_keys_hold(device, pad, window):
    """Keys before a sequence's leftpad, or before the window of every query, share a key block with the first one
    seen; NaN in them reaches no output."""
    b, sq, h, hk, hd, cap, lens = 2, 70, 4, 4, 128, 512, (300, 450)
    g = torch.Generator().manual_seed(8600 + sum(pad))
    q, kc, vc = randn16((b, sq, h, hd), g), randn16((b, cap, hk, hd), g), randn16((b, cap, hk, hd), g)
    seqlens, leftpad = torch.tensor(lens, dtype=torch.int32), torch.tensor(pad, dtype=torch.int32)
    print(f"case unseen keys pad={pad} window={window}", flush=True)
    o_ref, l_ref = okv.splitkv_attention(q, *okv.materialize(kc, vc, seqlens, None, None), seqlens, hd ** -0.5, True, 1,
                                         window=window, leftpad=leftpad)
    for i in range(b):
        first = pad[i] if window[0] < 0 else lens[i] - sq - window[0]
        assert first > 0 and first % 64
        kc[i, :first], vc[i, :first] = float("nan"), float("nan")
    for splits in (1, 3):
        out, lse = _call(device, q, kc, vc, None, None, seqlens, None, None, splits, True,
                         dict(window_size=window, cache_leftpad=leftpad))[:2]
        assert_2x("out", out, o_ref, o_ref.to(torch.float16))
        assert_lse(lse, l_ref)
