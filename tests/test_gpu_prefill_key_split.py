"""GPU parity of the key-split prefill kernel (few workgroups with long key-tile chains: four teams of 32 query tokens,
or two of 64, merged in LDS).

Against the oracle (bf16 output within max-abs 2e-2 and mean-abs 2e-3 of the fp32-softmax restatement of
engine/talker.py:163-167): the smallest shapes that take it, lengths around a tile and a team, the table's second
64-page window, sequences much shorter than the longest (whole workgroups and teams without a key), no mask, and
query rows that see no key.  K/V packed, paged and with the pool write give the same bits (one decomposition), the
pool holds the rows, and the norm/rope form agrees with the append form on the oracle's rows.
"""
import numpy as np
import pytest
import torch

import q3attn
from helpers import to_np
from oracle import attention as ora
from q3attn import workloads as W
from test_gpu_prefill_append import _run_both, _table

pytestmark = pytest.mark.gpu


def check(out, ref, what):
    ok, st = ora.compare(to_np(out), ref)
    print(f"[parity] key split {what} {st}", flush=True)
    assert ok, (what, st)


def varlen(wl, k=None, v=None, bt=None, causal=True):
    return q3attn.flash_attn_varlen_func(wl.q, wl.k if k is None else k, wl.v if v is None else v, wl.cu_seqlens,
                                         wl.cu_seqlens, wl.max_len, wl.max_len, softmax_scale=wl.scale, causal=causal,
                                         block_table=bt)


@pytest.mark.parametrize("lens", [
    [384], [385], [415, 1], [1024], [33, 510],     # four teams
    [384, 353, 5], [352, 352, 31, 352], [1057], [2047],  # two
])
def test_varlen_forms(cuda_device, lens):
    wl = W.make_prefill(cuda_device, lens, seed=sum(lens), paged=True)
    out = varlen(wl)
    cu = wl.cu_seqlens.cpu().numpy()
    check(out, ora.prefill_varlen(to_np(wl.q), to_np(wl.k), to_np(wl.v), cu, wl.scale), lens)
    assert torch.equal(out, varlen(wl, wl.k_cache, wl.v_cache, wl.block_table)), "paged differs"
    kc, vc = torch.zeros_like(wl.k_cache), torch.zeros_like(wl.v_cache)
    app = q3attn.prefill_append(wl.q, wl.k, wl.v, wl.cu_seqlens, wl.cu_seqlens, wl.max_len, kc, vc, wl.block_table,
                                wl.scale, True)
    assert torch.equal(app, out), "append differs"
    assert torch.equal(kc, _scattered(wl, wl.k)) and torch.equal(vc, _scattered(wl, wl.v)), "pool differs"


def _scattered(wl, x):
    """A zeroed pool with each token's row of x [T, Hkv, D] at its slot."""
    cu, bt, page = wl.cu_seqlens.cpu().numpy(), wl.block_table.cpu().numpy().astype(np.int64), wl.k_cache.shape[1]
    slots = np.concatenate([bt[s, np.arange(n) // page] * page + np.arange(n) % page
                            for s, n in enumerate(np.diff(cu))])
    pool = torch.zeros_like(wl.k_cache)
    pool.view(-1, W.HKV, W.HEAD_DIM)[torch.from_numpy(slots).to(x.device)] = x
    return pool


@pytest.mark.parametrize("lens", [[400, 37], [353, 353, 353, 100]])
def test_not_causal(cuda_device, lens):
    wl = W.make_prefill(cuda_device, lens, seed=9, paged=False)
    out = varlen(wl, causal=False)
    cu = wl.cu_seqlens.cpu().numpy()
    q, k, v = to_np(wl.q), to_np(wl.k), to_np(wl.v)
    ref = np.zeros_like(q)
    for s in range(len(lens)):
        r = slice(cu[s], cu[s + 1])
        for h in range(W.HQ):
            a = q[r, h] @ k[r, h // 2].T * wl.scale
            p = np.exp(a - a.max(-1, keepdims=True))
            ref[r, h] = (p / p.sum(-1, keepdims=True)) @ v[r, h // 2]
    check(out, ref, f"not causal {lens}")


@pytest.mark.parametrize("S,R,n", [(1, 1, 288), (1, 290, 288), (4, 200, 352), (6, 210, 380), (2, 300, 331), (1, 320, 289)])
def test_dense_prefix_and_append(cuda_device, S, R, n):
    dev = cuda_device
    g = torch.Generator(device=dev).manual_seed(S * 1000 + R)
    q = torch.randn(S, R, 16, 128, generator=g, device=dev).to(torch.bfloat16)
    K = torch.randn(S, n, 8, 128, generator=g, device=dev).to(torch.bfloat16)
    V = torch.randn(S, n, 8, 128, generator=g, device=dev).to(torch.bfloat16)
    scale = 128 ** -0.5
    out = q3attn.flash_attn_func(q, K, V, softmax_scale=scale, causal=True)
    qf, kf, vf = to_np(q), to_np(K), to_np(V)
    ref = np.zeros_like(qf)
    see = np.arange(n)[None, :] <= n - R + np.arange(R)[:, None]
    for s in range(S):
        for h in range(16):
            a = np.where(see, qf[s, :, h] @ kf[s, :, h // 2].T * scale, -np.inf)
            p = np.exp(a - np.maximum(a.max(-1, keepdims=True), -1e30))
            ref[s, :, h] = (p / np.maximum(p.sum(-1, keepdims=True), 1e-30)) @ vf[s, :, h // 2]
    check(out, ref, f"dense {S}x{R} over {n}")
    if R > n:
        assert not out[:, :R - n].float().abs().sum().item(), "rows that see no key must be zeros"
        return
    w = -(-n // 16)
    bt = torch.randperm(S * w, generator=torch.Generator().manual_seed(1)).to(torch.int32).view(S, w).to(dev)
    kc, vc = torch.zeros((2, S * w, 16, 8, 128), dtype=torch.bfloat16, device=dev)
    app = q3attn.prefill_dense_append(q, K, V, kc, vc, bt, scale, True)
    assert torch.equal(app, out)
    for c, x in ((kc, K), (vc, V)):
        assert torch.equal(c[bt.long()].view(S, w * 16, 8, 128)[:, :n], x)


@pytest.mark.parametrize("lens", [[400], [384, 353, 40]])
def test_norm_rope_form(cuda_device, lens):
    dev = cuda_device
    wl = W.make_prefill(dev, lens, seed=21, paged=True)
    rng = np.random.default_rng(4)
    t = lambda x: torch.from_numpy(np.ascontiguousarray(x, np.float32)).to(dev).to(torch.bfloat16)
    r = lambda x: ora.bf16_round(np.asarray(x, np.float32))
    qn, kn = (r(rng.uniform(0.5, 1.5, W.HEAD_DIM)) for _ in range(2))
    cos_t, sin_t = ora.rope_tables(2048)
    pos = np.concatenate([np.arange(n) for n in lens])
    cos, sin = r(cos_t[pos]), r(sin_t[pos])
    eps = 1e-6
    qq, kk = (ora.norm_rope(to_np(x), w, cos[:, None], sin[:, None], eps, eager=True) for x, w in ((wl.q, qn), (wl.k, kn)))
    pools = [torch.zeros_like(wl.k_cache) for _ in range(4)]
    out = q3attn.prefill_append_rope(wl.q, wl.k, wl.v, t(qn), t(kn), t(cos), t(sin), wl.cu_seqlens, wl.max_len, pools[0],
                                     pools[1], wl.block_table, wl.scale, True, eps)
    ref = q3attn.prefill_append(t(qq), t(kk), wl.v, wl.cu_seqlens, wl.cu_seqlens, wl.max_len, pools[2], pools[3],
                                wl.block_table, wl.scale, True)
    check(out, to_np(ref), f"norm/rope {lens}")
    assert torch.equal(pools[1], pools[3])
    assert (pools[0].float() - pools[2].float()).abs().max().item() <= 2 ** -6 * pools[2].float().abs().max().item()


@pytest.mark.parametrize("lens,bound", [([42], 1024), ([200], 1024), ([100, 100], 1000), ([50, 30, 50, 50], 500), ([400], 2048)])
def test_a_loose_bound_takes_the_same_kernel(cuda_device, lens, bound):
    """max_seqlen above every length, in the packed, the append and the norm/rope form: the bits of the exact bound (teams
    of waves for a chain that no sequence has merged in another order, and cost a short prompt 10 to 40 %)."""
    wl = W.make_prefill(cuda_device, lens, seed=5, paged=True)
    g = torch.Generator(device=cuda_device).manual_seed(1)
    rnd = lambda *s: torch.randn(s, generator=g, device=cuda_device).to(torch.bfloat16)
    T = int(wl.q.shape[0])
    qn, kn, cos, sin = rnd(128), rnd(128), rnd(T, 128), rnd(T, 128)

    def forms(mx):
        pool = lambda: (torch.zeros_like(wl.k_cache), torch.zeros_like(wl.v_cache))
        p, r = pool(), pool()
        return (q3attn.flash_attn_varlen_func(wl.q, wl.k, wl.v, wl.cu_seqlens, wl.cu_seqlens, mx, mx, softmax_scale=wl.scale,
                                              causal=True),
                q3attn.prefill_append(wl.q, wl.k, wl.v, wl.cu_seqlens, wl.cu_seqlens, mx, *p, wl.block_table, wl.scale, True),
                q3attn.prefill_append_rope(wl.q, wl.k, wl.v, qn, kn, cos, sin, wl.cu_seqlens, mx, *r, wl.block_table, wl.scale,
                                           True, 1e-6), *p, *r)
    for a, b in zip(forms(max(lens)), forms(bound)):
        assert torch.equal(a, b)


@pytest.mark.parametrize("causal", [True, False])
@pytest.mark.parametrize("lens,prefix", [([400], [37]), ([384, 100], [32, 50]),      # four teams
                                         ([384, 353, 5], [0, 45, 300]), ([1057], [3])])  # two
def test_packed_append_after_a_prefix(cuda_device, lens, prefix, causal):
    """Keys before the first query (a multiple of a tile or not), with and without the mask: the pool rows go out through the
    prologue's copies, or from the stages of the last tiles.  Output and pool as in scatter + packed prefill, bit for bit,
    and the output against the fp32 softmax."""
    dev, g = cuda_device, torch.Generator().manual_seed(sum(lens))
    Lq, Lk = np.array(lens), np.array(lens) + np.array(prefix)
    cu_q, cu_k = (np.concatenate([[0], np.cumsum(x)]).astype(np.int32) for x in (Lq, Lk))
    rnd = lambda n, h: torch.randn(n, h, 128, generator=g).to(torch.bfloat16).to(dev)
    q, k, v = rnd(cu_q[-1], 16), rnd(cu_k[-1], 8), rnd(cu_k[-1], 8)
    P = -(-int(Lk.max()) // 16)
    out, _, _, n = _run_both(dev, q, k, v, cu_q, cu_k, int(Lq.max()), _table(len(lens), P, 4 * P * len(lens), False, 7), 16,
                             4 * P * len(lens), 0.09, causal)
    assert n == Lq.sum()
    qf, kf, vf = to_np(q), to_np(k), to_np(v)
    ref = np.zeros_like(qf)
    for s in range(len(lens)):
        r, c = slice(cu_q[s], cu_q[s + 1]), slice(cu_k[s], cu_k[s + 1])
        see = np.arange(Lk[s])[None, :] <= (prefix[s] + np.arange(Lq[s])[:, None] if causal else Lk[s])
        for h in range(16):
            a = np.where(see, qf[r, h] @ kf[c, h // 2].T * 0.09, -np.inf)
            p = np.exp(a - a.max(-1, keepdims=True))
            ref[r, h] = (p / p.sum(-1, keepdims=True)) @ vf[c, h // 2]
    check(out, ref, f"packed {lens} after {prefix}, causal {causal}")
