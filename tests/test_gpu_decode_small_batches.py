"""GPU parity of the decode of small batches (the library's own choice for up to 64 rows; up to 16 rows: 128-token
chunks, listed from the rows' lengths where their grid is more than one workgroup a CU; 17 to 64: the row kernel).

* against the oracle (bf16 output within max-abs 2e-2 and mean-abs 2e-3 of the fp32-softmax restatement of
  engine/talker.py:82-88) at the edges of the ranges: the smallest and largest batch and table, one lane short of a wave,
  rows of 0, 1, a tile, a tile and a token, and full tables, all rows full (the longest lists) and all rows empty but one;
* the plain form bit-identical to the append form on the same tokens, and that with the norm/rope form on +-1 rows,
  whose normalised rows are exact (the same decomposition in all three);
* a row's bits do not depend on the other rows' lengths, and waves of two tiles round the output alone to bf16;
* the shapes beside the ranges bit-identical to the path that serves them;
* 17 to 64 rows need no workspace (q3a_paged_decode_workspace_bytes of split_tokens 0 is 0) and so write none, whatever
  buffer the call is handed: a caller may share it between streams.
"""
import numpy as np
import pytest
import torch

import q3attn
from helpers import decode_oracle, to_np
from oracle import attention as ora
from q3attn import _lib
from q3attn import workloads as W


def _ctx(B, cap, kind):
    rng = np.random.default_rng(B * 7 + cap)
    if kind == "full":
        return np.full(B, cap)
    if kind == "lone":
        c = np.zeros(B, np.int64)
        c[B // 2] = cap
        return c
    c = np.rint(np.exp(rng.uniform(0, np.log(cap), size=B))).astype(np.int64)
    c[:5] = [0, 1, 16, 17, cap]
    return rng.permutation(c)


@pytest.mark.gpu
@pytest.mark.parametrize("kind", ["ragged", "full", "lone"])
@pytest.mark.parametrize("B,cap", [(5, 272), (5, 2048), (6, 144), (6, 768), (8, 512), (16, 256), (16, 272), (16, 1040), (16, 2048), (17, 528),
                                   (32, 1040), (33, 208), (33, 544), (63, 1024), (64, 2048)])
def test_small_batches_vs_oracle_and_append(cuda_device, B, cap, kind):
    ctx = _ctx(B, cap, kind)
    wl = W.make_decode("bal", cuda_device, ctx=ctx, num_pages=2 * B * (cap // 16 + 1), max_ctx=cap, seed=B + cap)
    L = wl.layers[0]
    out = q3attn.paged_decode(L.q, wl.k_cache, wl.v_cache, wl.cache_seqlens, L.block_table, wl.scale)
    ok, st = ora.compare(to_np(out), decode_oracle(wl))
    assert ok, (B, cap, kind, st)
    assert not out[torch.from_numpy(ctx == 0).to(cuda_device)].float().abs().sum().item()
    # The append form, its slots poisoned: same bits, and the pool as index_copy_ leaves it.
    page = wl.page_size
    bt = L.block_table.cpu().numpy().astype(np.int64)
    live = ctx > 0
    pos = np.maximum(ctx - 1, 0)
    slots = torch.from_numpy((bt[np.arange(B), pos // page] * page + pos % page)[live]).to(cuda_device)
    rows = torch.from_numpy(np.flatnonzero(live)).to(cuda_device)
    kf, vf = (x.view(-1, W.HKV, W.HEAD_DIM) for x in (wl.k_cache, wl.v_cache))
    k, v = torch.zeros((2, B, W.HKV, W.HEAD_DIM), dtype=torch.bfloat16, device=cuda_device)
    k[rows], v[rows] = kf[slots], vf[slots]
    ref_k, ref_v = wl.k_cache.clone(), wl.v_cache.clone()
    kf[slots], vf[slots] = float("nan"), float("nan")
    old = torch.from_numpy(ctx - 1).to(torch.int32).to(cuda_device)
    app = q3attn.paged_decode_append(L.q, k, v, wl.k_cache, wl.v_cache, old, L.block_table, wl.scale)
    assert torch.equal(app, out)
    assert torch.equal(wl.k_cache, ref_k) and torch.equal(wl.v_cache, ref_v)


@pytest.mark.gpu
@pytest.mark.parametrize("B", [12, 20])
def test_rope_form_exact_rows(cuda_device, B):
    dev = cuda_device
    ctx = _ctx(B, 1024, "ragged")
    wl = W.make_decode("bal_rope", dev, ctx=ctx, num_pages=4096, max_ctx=1024, seed=7)
    rng = np.random.default_rng(5)
    r = lambda x: ora.bf16_round(np.asarray(x, np.float32))
    t = lambda x: torch.from_numpy(np.ascontiguousarray(x, np.float32)).to(dev).to(torch.bfloat16)
    q, k = (r(rng.choice([-1.0, 1.0], size=(B, h, W.HEAD_DIM))) for h in (W.HQ, W.HKV))
    v = r(rng.standard_normal((B, W.HKV, W.HEAD_DIM)))
    qn, kn = (r(rng.uniform(0.5, 1.5, W.HEAD_DIM)) for _ in range(2))
    cos_t, sin_t = ora.rope_tables(1024)
    pos = np.maximum(ctx - 1, 0)
    cos, sin = r(cos_t[pos]), r(sin_t[pos])
    qq, kk = (ora.norm_rope(x, w, cos[:, None], sin[:, None], 0.0, eager=False) for x, w in ((q, qn), (k, kn)))
    old = torch.from_numpy(ctx - 1).to(torch.int32).to(dev)
    L = wl.layers[0]
    kc, vc = wl.k_cache.clone(), wl.v_cache.clone()
    out = q3attn.paged_decode_append_rope(t(q), t(k), t(v), t(qn), t(kn), t(cos), t(sin), wl.k_cache, wl.v_cache, old,
                                          L.block_table, wl.scale, 0.0)
    ref = q3attn.paged_decode_append(t(qq), t(kk), t(v), kc, vc, old, L.block_table, wl.scale)
    assert torch.equal(out, ref) and torch.equal(kc, wl.k_cache) and torch.equal(vc, wl.v_cache)


@pytest.mark.gpu
@pytest.mark.parametrize("B,cap", [(6, 768), (16, 272), (12, 1280), (16, 2048), (20, 1024)])
def test_a_row_does_not_depend_on_its_neighbours(cuda_device, B, cap):
    wl = W.make_decode("bal_nb", cuda_device, ctx=_ctx(B, cap, "ragged"), num_pages=2 * B * (cap // 16 + 1), max_ctx=cap, seed=B)
    L = wl.layers[0]
    run = lambda lens: q3attn.paged_decode(L.q, wl.k_cache, wl.v_cache, lens, L.block_table, wl.scale)
    out = run(wl.cache_seqlens)
    for other in (0, 17, cap // 2 + 3, cap):
        lens = wl.cache_seqlens.clone()
        lens[1::2] = other
        assert torch.equal(run(lens)[::2], out[::2]), other


@pytest.mark.gpu
@pytest.mark.parametrize("B,cap", [(6, 768), (16, 272), (16, 1280), (3, 144), (8, 256), (24, 192), (64, 256)])
def test_two_tiles_a_wave_round_the_output_alone(cuda_device, B, cap):
    """Listed chunks and tables of 9 to 16 tiles: q, k and v are exact in bf16 and the probabilities stay in fp32, so an output is within half a unit in the last place
    (2^-8 of it) of the float64 result, but for the fp32 sums: 128 products of a score (about 1e-6 of p each) and the
    tokens' sum, 2e-5 at the outputs' scale.  Probabilities rounded to bf16 are 7e-4 of the outputs' root mean square off."""
    wl = W.make_decode("bal_p", cuda_device, ctx=_ctx(max(B, 5), cap, "ragged")[:B], num_pages=2 * B * (cap // 16 + 1), max_ctx=cap, seed=cap)
    L = wl.layers[0]
    out = to_np(q3attn.paged_decode(L.q, wl.k_cache, wl.v_cache, wl.cache_seqlens, L.block_table, wl.scale)).astype(np.float64)
    ref = np.asarray(decode_oracle(wl, acc=np.float64), np.float64)
    over = np.abs(out - ref) - (2.0 ** -8 * np.abs(ref) + 2e-5)
    assert over.max() <= 0, over.max()


@pytest.mark.gpu
@pytest.mark.parametrize("hkv,B,cap", [(8, 33, 272), (8, 40, 1040), (8, 63, 2048), (8, 64, 528), (16, 17, 272), (16, 20, 1040),
                                       (16, 32, 2048), (5, 60, 528), (4, 64, 528)])
def test_rows_in_the_order_of_their_lengths(cuda_device, hkv, B, cap):
    """A batch whose rows fill the CUs more than once goes in the order of the lengths: each row as in a call of a few rows
    (index order), ties, empty rows and rows past the capacity among them, in the plain and in the append form."""
    g = torch.Generator(device=cuda_device).manual_seed(B)
    pages = B * (cap // 16)
    rnd = lambda *s: torch.randn(s, generator=g, device=cuda_device).to(torch.bfloat16)
    kc, vc, q = rnd(pages, 16, hkv, 128), rnd(pages, 16, hkv, 128), rnd(B, 2 * hkv, 128)
    k, v = rnd(B, hkv, 128), rnd(B, hkv, 128)
    bt = torch.randperm(pages, generator=g, device=cuda_device).view(B, -1).to(torch.int32)
    ctx = _ctx(B, cap, "ragged")
    ctx[5:9] = [cap, cap, cap + 9, 17]
    few = lambda f: torch.cat([f(slice(i, min(i + 8, B))) for i in range(0, B, 8)])
    for lens in (ctx, np.full(B, cap // 2), np.where(np.arange(B) == B - 1, cap, 0)):
        sl = torch.from_numpy(lens).to(torch.int32).to(cuda_device)
        out = q3attn.paged_decode(q, kc, vc, sl, bt, 0.1)
        assert torch.equal(out, few(lambda r: q3attn.paged_decode(q[r], kc, vc, sl[r], bt[r], 0.1, q3attn.DECODE_ROW)))
        c1 = (kc.clone(), vc.clone())
        app = q3attn.paged_decode_append(q, k, v, kc, vc, sl, bt, 0.1)
        assert torch.equal(app, few(lambda r: q3attn.paged_decode_append(q[r], k[r], v[r], *c1, sl[r], bt[r], 0.1,
                                                                         q3attn.DECODE_ROW)))
        assert torch.equal(kc, c1[0]) and torch.equal(vc, c1[1])


ROW, CHUNKS, SK = q3attn.DECODE_ROW, q3attn.DECODE_CHUNKS, q3attn.DECODE_STREAMK


@pytest.mark.gpu
@pytest.mark.parametrize("B,cap,path", [(4, 1024, CHUNKS), (65, 1024, SK), (8, 256, ROW), (17, 512, ROW), (17, 528, ROW),
                                        (28, 1024, ROW), (33, 2048, ROW), (64, 2048, ROW), (8, 2064, CHUNKS)])
def test_shapes_beside_its_range(cuda_device, B, cap, path):
    wl = W.make_decode("bal_no", cuda_device, ctx=_ctx(max(B, 5), cap, "ragged")[:B], num_pages=4 * B * 130, max_ctx=cap, seed=B)
    L = wl.layers[0]
    out = q3attn.paged_decode(L.q, wl.k_cache, wl.v_cache, wl.cache_seqlens, L.block_table, wl.scale)
    ok, st = ora.compare(to_np(out), decode_oracle(wl))
    assert ok, st
    forced = q3attn.paged_decode(L.q, wl.k_cache, wl.v_cache, wl.cache_seqlens, L.block_table, wl.scale, path)
    assert torch.equal(out, forced)


@pytest.mark.gpu
def test_batches_past_the_grid_limit(cuda_device):
    """Narrow tables with more rows than a grid dimension holds (65,535) go in slices of rows: the rows around the cut and the
    last one as in a call of those rows alone, plain, append and norm/rope form, and the slots that they wrote."""
    B, dev = 65600, cuda_device
    g = torch.Generator(device=dev).manual_seed(65)
    rnd = lambda *s: torch.randn(s, generator=g, device=dev, dtype=torch.bfloat16)
    kc, vc = rnd(B, 16, 8, 128), rnd(B, 16, 8, 128)
    qkv, qn, kn, cos, sin = rnd(B, 32 * 128), rnd(128), rnd(128), rnd(B, 128), rnd(B, 128)
    q, k, v = qkv[:, :2048].view(B, 16, 128), qkv[:, 2048:3072].view(B, 8, 128), qkv[:, 3072:].view(B, 8, 128)
    bt = torch.randperm(B, generator=g, device=dev).to(torch.int32).view(B, 1)
    lens = torch.randint(0, 16, (B,), generator=g, device=dev, dtype=torch.int32)
    r = torch.tensor([0, 1, 65533, 65534, 65535, 65536, 65537, B - 2, B - 1], device=dev)
    pages = bt[r, 0].long()

    def forms(x):
        pools = [(kc.clone(), vc.clone()) for _ in range(2)] if x is not None else [(kc, vc)] * 2
        s = (lambda t: t[x]) if x is not None else (lambda t: t)
        return (q3attn.paged_decode(s(q), kc, vc, s(lens), s(bt), 0.1),
                lambda: (q3attn.paged_decode_append(s(q), s(k), s(v), *pools[0], s(lens), s(bt), 0.1), *pools[0]),
                lambda: (q3attn.paged_decode_append_rope(s(q), s(k), s(v), qn, kn, s(cos), s(sin), *pools[1], s(lens), s(bt), 0.1,
                                                         1e-6), *pools[1]))

    few = forms(r)
    few = [few[0], few[1](), few[2]()]
    clean = kc[pages].clone(), vc[pages].clone()
    big = forms(None)
    assert torch.equal(big[0][r], few[0])
    for f, want in zip(big[1:], few[1:]):
        out, pk, pv = f()
        assert torch.equal(out[r], want[0])
        assert torch.equal(pk[pages], want[1][pages]) and torch.equal(pv[pages], want[2][pages])
        kc[pages], vc[pages] = clean


def _c_decode(fn, wl, out, *ws):
    L = wl.layers[0]
    return fn(L.q.data_ptr(), L.q.stride(0), L.q.stride(1), wl.k_cache.data_ptr(), wl.v_cache.data_ptr(),
              *wl.k_cache.stride()[:3], wl.k_cache.shape[0], wl.page_size, wl.cache_seqlens.data_ptr(),
              L.block_table.data_ptr(), L.block_table.stride(0), L.block_table.shape[1], out.data_ptr(), out.stride(0),
              out.stride(1), *ws, wl.batch, W.HQ, W.HKV, W.HEAD_DIM, wl.scale, 0, torch.cuda.current_stream().cuda_stream)


@pytest.mark.gpu
@pytest.mark.parametrize("B,cap", [(17, 2048), (20, 1024), (33, 544), (64, 2048)])
def test_no_workspace_is_touched_from_17_rows(cuda_device, B, cap):
    """Without a workspace, with a large one (left as it was) and through the entry point that shares one array between
    all its calls: the row kernel, bit for bit."""
    wl = W.make_decode("bal_ws", cuda_device, ctx=_ctx(B, cap, "ragged"), num_pages=2 * B * (cap // 16 + 1), max_ctx=cap, seed=3)
    L, lib = wl.layers[0], _lib.lib()
    row = q3attn.paged_decode(L.q, wl.k_cache, wl.v_cache, wl.cache_seqlens, L.block_table, wl.scale, ROW)
    out = torch.full_like(L.q, float("nan"))
    assert _c_decode(lib.q3a_paged_decode, wl, out, None, 0) == 0 and torch.equal(out, row)
    arena = torch.full((8 << 20,), 0x5A, dtype=torch.uint8, device=cuda_device)
    out.fill_(float("nan"))
    assert _c_decode(lib.q3a_paged_decode, wl, out, arena.data_ptr(), arena.numel()) == 0 and torch.equal(out, row)
    assert bool((arena == 0x5A).all())
    out.fill_(float("nan"))
    assert _c_decode(lib.q3a_paged_decode_noalloc, wl, out) == 0 and torch.equal(out, row)


def test_workspace_query():
    """Up to 16 rows: the records of 128-token chunks; 17 to 64 rows of up to 2,048 tokens: none, for every head count."""
    ws = lambda B, pages, split, hkv=8: _lib.lib().q3a_paged_decode_workspace_bytes(B, 2 * hkv, hkv, 128, pages, 16, split)
    assert ws(16, 128, 0) == 16 * 16 * 8 * 1040 and ws(5, 17, 0) == 5 * 3 * 8 * 1040
    for B in (17, 32, 33, 64):
        for pages in (9, 16, 17, 33, 65, 128):
            for hkv in (1, 8, 16):
                assert ws(B, pages, 0, hkv) == 0
