"""GPU parity: causal GQA attention prefill over the paged KV cache.

The reference prefills by running one decode step per prompt token
(qwen36_chat_batch.py:255-258 -> qwen36_attention_cache.py:306-317), so the
oracle is `oracle.chunked.causal_attention_prefill` (pinned against that
token-by-token recurrence in test_oracle_chunked.py).  Covered here: ragged
prompt lengths over shuffled pages, a prompt continued after resident
context, fp16 activations with fp16 pages, GQA groups below 8, the pages the
prefill writes (bit-exact against the decode append), prefill == decode
steps, and a 16384-token prompt checked row-by-row on sampled tokens.
"""

from __future__ import annotations

import pytest
import torch

from conftest import announce
from helpers import assert_act_close
from oracle import chunked as OC
from oracle import qwen36_cpu as O
from router_ia import kernels as K
from router_ia.batched_state import rope_inv_freq
from router_ia.paged_kv import PagedKVCache

SCALE = 256 ** -0.5


def _inputs(seed, length, hq=16, hkv=2, dtype=torch.bfloat16):
    g = torch.Generator().manual_seed(seed)
    q = torch.randn((length, hq, 256), generator=g).to(dtype)
    k = torch.randn((length, hkv, 256), generator=g).to(dtype)
    v = torch.randn((length, hkv, 256), generator=g).to(dtype)
    gate = torch.randn((length, hq, 256), generator=g).to(dtype)
    return q, k, v, gate


def _cache(dev, tokens, hkv=2, dtype=torch.bfloat16, shuffle_seed=5):
    pages = (tokens + 15) // 16 + 3
    kv = PagedKVCache(1, pages, 1, pages, num_kv_heads=hkv, device=dev, shuffle_seed=shuffle_seed, dtype=dtype)
    kv.ensure(0, tokens)
    return kv


def _run(dev, kv, q, k, v, gate, start, staged=False, phase=None):
    inv = rope_inv_freq(10_000_000.0, 64).to(dev)
    length, hkv = int(q.shape[0]), int(k.shape[1])
    stage = torch.empty(K.prefill_stage_bytes(length, hkv), dtype=torch.uint8, device=dev) if staged else None
    qd, kd, vd, gd = q.to(dev), k.to(dev), v.to(dev), gate.to(dev)
    if phase is None:
        return K.attn_prefill(qd, kd, vd, gd, kv.k[0], kv.v[0], kv.page_table[0], start=start, inv_freq=inv,
                              scale=SCALE, stage=stage)
    from router_ia import _native as nat
    out = K.attn_prefill(qd, kd, vd, gd, kv.k[0], kv.v[0], kv.page_table[0], start=start, inv_freq=inv,
                         scale=SCALE, stage=stage, phase=nat.RIA_PREFILL_APPEND)
    return K.attn_prefill(qd, kd, vd, gd, kv.k[0], kv.v[0], kv.page_table[0], out, start=start, inv_freq=inv,
                          scale=SCALE, stage=stage, phase=nat.RIA_PREFILL_ATTEND)


@pytest.mark.gpu
@pytest.mark.parametrize("length", [1, 15, 16, 17, 300, 1000])
def test_attn_prefill_matches_oracle(gpu, length):
    announce(f"attn_prefill: L={length}, bf16, shuffled pages")
    q, k, v, gate = _inputs(100 + length, length)
    kv = _cache(gpu, length)
    out = _run(gpu, kv, q, k, v, gate, 0)
    want, kr = OC.causal_attention_prefill(q, k, v, gate, torch.arange(length))
    assert_act_close(out, want, f"L={length}")
    # the pages hold v exactly and the rotated keys rounded once to bf16
    kg, vg = K.kv_gather(kv.k[0], kv.v[0], kv.page_table, batch=1, start=0, count=length)
    assert torch.equal(vg[0].cpu(), v.transpose(0, 1))
    torch.testing.assert_close(kg[0].cpu().float(), kr.transpose(0, 1).to(torch.bfloat16).float(),
                               rtol=8e-3, atol=1e-5)


@pytest.mark.gpu
@pytest.mark.parametrize("length,hq,hkv,phases", [(1, 16, 2, False), (17, 16, 2, True), (300, 16, 2, False),
                                                   (1000, 16, 2, True), (130, 6, 2, False)])
def test_attn_prefill_staged_fp16_keys(gpu, length, hq, hkv, phases):
    # a prompt from slot 0 with an fp16 stage: the pages get exactly what the unstaged append writes, the
    # attention reads the prompt's fp16 keys (single fp16 MFMA operands) and matches the oracle
    announce(f"attn_prefill staged: L={length}, Hq={hq}, Hkv={hkv}, {'two phases' if phases else 'one call'}")
    q, k, v, gate = _inputs(200 + length, length, hq, hkv)
    kv_s, kv_u = _cache(gpu, length, hkv=hkv), _cache(gpu, length, hkv=hkv)
    out_s = _run(gpu, kv_s, q, k, v, gate, 0, staged=True, phase=phases or None)
    out_u = _run(gpu, kv_u, q, k, v, gate, 0)
    assert torch.equal(kv_s.k, kv_u.k) and torch.equal(kv_s.v, kv_u.v), "pages differ from the unstaged append"
    want, _ = OC.causal_attention_prefill(q, k, v, gate, torch.arange(length), num_kv_groups=hq // hkv)
    assert_act_close(out_s, want, f"staged L={length}")


@pytest.mark.gpu
def test_attn_prefill_continues_after_resident_context(gpu):
    """Prompt of 157 tokens on top of 100 prefilled ones == one 257-token prompt."""
    announce("attn_prefill: 100 + 157 tokens in two calls")
    n0, n1 = 100, 157
    q, k, v, gate = _inputs(7, n0 + n1)
    kv = _cache(gpu, n0 + n1)
    out0 = _run(gpu, kv, q[:n0], k[:n0], v[:n0], gate[:n0], 0, staged=True)
    # (a stage is ignored past slot 0: the resident keys are only in the pages)
    out1 = _run(gpu, kv, q[n0:], k[n0:], v[n0:], gate[n0:], n0, staged=True)
    want, _ = OC.causal_attention_prefill(q, k, v, gate, torch.arange(n0 + n1))
    assert_act_close(torch.cat([out0.cpu(), out1.cpu()]), want, "two-call prefill")


@pytest.mark.gpu
def test_attn_prefill_fp16_pages(gpu):
    announce("attn_prefill: L=333, fp16 activations and fp16 pages")
    length = 333
    q, k, v, gate = _inputs(9, length, dtype=torch.float16)
    kv = _cache(gpu, length, dtype=torch.float16)
    out = _run(gpu, kv, q, k, v, gate, 0)
    assert out.dtype == torch.float16
    want, _ = OC.causal_attention_prefill(q, k, v, gate, torch.arange(length))
    assert_act_close(out, want, "fp16")


@pytest.mark.gpu
@pytest.mark.parametrize("hq,hkv", [(8, 2), (6, 2), (4, 4), (1, 1)])
def test_attn_prefill_gqa_groups(gpu, hq, hkv):
    announce(f"attn_prefill: Hq={hq}, Hkv={hkv}, L=130")
    length = 130
    q, k, v, gate = _inputs(11 + hq, length, hq, hkv)
    kv = _cache(gpu, length, hkv=hkv)
    out = _run(gpu, kv, q, k, v, gate, 0)
    want, _ = OC.causal_attention_prefill(q, k, v, gate, torch.arange(length), num_kv_groups=hq // hkv)
    assert_act_close(out, want, f"Hq={hq} Hkv={hkv}")


@pytest.mark.gpu
def test_attn_prefill_equals_decode_steps(gpu):
    """The prefill writes the same pages as per-token appends, and its outputs match per-token decode."""
    announce("attn_prefill vs decode steps: L=200")
    length = 200
    q, k, v, gate = _inputs(13, length)
    inv = rope_inv_freq(10_000_000.0, 64).to(gpu)
    kv_a = _cache(gpu, length, shuffle_seed=1)
    out_p = _run(gpu, kv_a, q, k, v, gate, 0)
    kv_b = _cache(gpu, length, shuffle_seed=2)
    ws = torch.empty(K.attn_decode_workspace_bytes(1, 16, 2, length, 64) // 4 + 64, dtype=torch.float32,
                     device=gpu)
    outs = []
    for t in range(length):
        K.kv_append(k[t:t + 1].to(gpu), v[t:t + 1].to(gpu), kv_b.k[0], kv_b.v[0], kv_b.page_table, positions=t,
                    slots=t, inv_freq=inv)
        o = torch.empty((1, 16, 256), dtype=torch.float32, device=gpu)
        K.attn_decode(q[t:t + 1].to(gpu), gate[t:t + 1].to(gpu), kv_b.k[0], kv_b.v[0], kv_b.page_table, o,
                      positions=t, ctx_lens=t + 1, max_ctx=length, inv_freq=inv, scale=SCALE, workspace=ws,
                      split_tokens=64)
        outs.append(o.cpu())
    dec = torch.cat(outs)
    assert_act_close(out_p, dec, "prefill vs decode")
    ka, va = K.kv_gather(kv_a.k[0], kv_a.v[0], kv_a.page_table, batch=1, start=0, count=length)
    kb, vb = K.kv_gather(kv_b.k[0], kv_b.v[0], kv_b.page_table, batch=1, start=0, count=length)
    assert torch.equal(ka, kb) and torch.equal(va, vb)


def _row_reference(qr, kr, v, gate, t, group=8):
    """fp64 attention of query token t over keys 0..t (all heads)."""
    kx = kr[: t + 1].double().repeat_interleave(group, dim=1)  # [t+1, Hq, d]
    vx = v[: t + 1].double().repeat_interleave(group, dim=1)
    s = torch.einsum("hd,thd->ht", qr[t].double(), kx) * SCALE
    p = torch.softmax(s, dim=-1)
    return torch.einsum("ht,thd->hd", p, vx) * torch.sigmoid(gate[t].double())


@pytest.mark.gpu
@pytest.mark.parametrize("staged", [False, True], ids=["pages", "stage"])
def test_attn_prefill_16384_sampled_rows(gpu, staged):
    """Full-size prompt: 16384 tokens, 48 sampled query rows against fp64 attention."""
    announce(f"attn_prefill: L=16384, sampled rows vs fp64, keys from the {'stage' if staged else 'pages'}")
    length = 16384
    q, k, v, gate = _inputs(17, length)
    kv = _cache(gpu, length)
    out = _run(gpu, kv, q, k, v, gate, 0, staged=staged).cpu()
    torch.cuda.synchronize()
    g = torch.Generator().manual_seed(3)
    rows = sorted(set([0, 1, 15, 16, 4095, 8191, length - 1] + torch.randint(0, length, (41,), generator=g).tolist()))
    qr = torch.empty(len(rows), 16, 256)
    kr = torch.empty(length, 2, 256)
    for t in range(length):  # each key rotated at its own position
        _, kt = O.apply_rope(k[t:t + 1].float(), k[t:t + 1].float(), t)
        kr[t] = kt[0]
    for i, t in enumerate(rows):
        qt, _ = O.apply_rope(q[t:t + 1].float(), q[t:t + 1].float(), t)
        qr[i] = qt[0]
    for i, t in enumerate(rows):
        qfull = torch.zeros(t + 1, 16, 256)
        qfull[t] = qr[i]
        want = _row_reference(qfull, kr, v.float(), gate.float(), t)
        assert_act_close(out[t], want.float(), f"row {t}")


@pytest.mark.gpu
@pytest.mark.parametrize("staged,bound", [(False, 0.7), (True, 0.35)], ids=["pages", "stage"])
def test_attn_prefill_keeps_its_tolerance_margin(gpu, staged, bound):
    """The worst error against the oracle stays well inside the activation
    tolerance across seeds and lengths (bf16 pages: q and P run as bf16 hi + lo
    pairs, a single bf16 P reached the tolerance itself on short prompts; fp16
    stage: single fp16 q and P over keys rounded once to fp16)."""
    announce(f"attn_prefill: error / tolerance over 9 prompts, keys from the {'stage' if staged else 'pages'}")
    from helpers import ACT_ATOL, ACT_RTOL
    worst = 0.0
    for length in (17, 300, 1000):
        for seed in (7, 42, 100 + length):
            q, k, v, gate = _inputs(seed, length)
            kv = _cache(gpu, length)
            out = _run(gpu, kv, q, k, v, gate, 0, staged=staged).float().cpu()
            want, _ = OC.causal_attention_prefill(q, k, v, gate, torch.arange(length))
            ratio = ((out - want.float()).abs() / (ACT_ATOL + ACT_RTOL * want.float().abs())).max().item()
            worst = max(worst, ratio)
    print(f"worst error / tolerance: {worst:.3f}", flush=True)
    assert worst <= bound, f"worst error is {worst:.3f} of the tolerance"


@pytest.mark.gpu
@pytest.mark.parametrize("length,start,hq,hkv", [(1, 1300, 16, 2), (17, 2047, 16, 2), (100, 1000, 6, 2),
                                                  (517, 0, 16, 2), (500, 7900, 16, 2), (1000, 0, 16, 2), (130, 813, 4, 4)])
def test_attn_prefill_split_keys(gpu, length, start, hq, hkv):
    """Query blocks whose keys are split between workgroups against the unsplit
    launch, fp32 activations.  Both round the probabilities (fp16: 2^-11,
    bf16 hi + lo: 2^-16 relative, about different maxima) in products and
    normaliser alike, so each output moves at most 2 * 2 * u * max |v|."""
    announce(f"attn_prefill split: {length} after {start}, Hq={hq}, Hkv={hkv}")
    _, k0, v0, _ = _inputs(7, max(start, 1), hq, hkv, torch.float32)
    q, k, v, gate = _inputs(8 + length, length, hq, hkv, torch.float32)
    inv = rope_inv_freq(10_000_000.0, 64).to(gpu)
    for kv_dtype, staged in ((torch.bfloat16, start == 0), (torch.float16, False)):
        kv = _cache(gpu, start + length, hkv, kv_dtype)
        if start:
            K.kv_append_seq(k0.to(gpu), v0.to(gpu), kv.k[0], kv.v[0], kv.page_table[0], start=0, inv_freq=inv)
        fp16 = staged or kv_dtype == torch.float16
        need = K.prefill_attn_workspace_bytes(length, hq, hkv, start, fp16)
        assert need > 0, "a split case"
        ws = torch.full((need,), 0xFF, dtype=torch.uint8, device=gpu)  # NaN partials where nothing is written
        args = (q.to(gpu), k.to(gpu), v.to(gpu), gate.to(gpu), kv.k[0], kv.v[0], kv.page_table[0])
        stage = torch.empty(K.prefill_stage_bytes(length, hkv), dtype=torch.uint8, device=gpu) if staged else None
        kw = dict(start=start, inv_freq=inv, scale=SCALE, stage=stage)
        whole = K.attn_prefill(*args, **kw)
        split = K.attn_prefill(*args, **kw, workspace=ws)
        small = K.attn_prefill(*args, **kw, workspace=ws[:need - 16])  # too small: unsplit
        assert torch.equal(whole, small)
        vmax = float(max(v.abs().max(), v0.abs().max()))
        tol = 4 * vmax * (2.0 ** -11 if fp16 else 2.0 ** -16) + 1e-5
        assert float((split - whole).abs().max()) <= tol


@pytest.mark.gpu
@pytest.mark.parametrize("length,hq,hkv", [(6017, 16, 2), (6031, 16, 2), (6048, 6, 2)])
@pytest.mark.parametrize("staged", [False, True], ids=["fp16 pages", "stage"])
def test_attn_prefill_32_token_blocks(gpu, length, hq, hkv, staged):
    """Long fp16-key prompts run in query blocks of 32 tokens.  Their first and
    last tokens (remainders of 1, 15 and 32) against the same tokens in blocks
    of 16: a short prompt of the first ones, and the last ones continued over
    the prompt's own pages.  Same bound as the split launches; the stage's fp16
    keys are compared on pages that hold the same fp16 values."""
    announce(f"attn_prefill 32-token blocks: L={length}, Hq={hq}, {'stage' if staged else 'fp16 pages'}")
    q, k, v, gate = (x.to(gpu) for x in _inputs(9 + length, length, hq, hkv, torch.float32))
    inv = rope_inv_freq(10_000_000.0, 64).to(gpu)
    kv = _cache(gpu, length, hkv, torch.float16)
    stage = torch.empty(K.prefill_stage_bytes(length, hkv), dtype=torch.uint8, device=gpu) if staged else None
    kw = dict(inv_freq=inv, scale=SCALE)
    out = K.attn_prefill(q, k, v, gate, kv.k[0], kv.v[0], kv.page_table[0], start=0, stage=stage, **kw)
    tol = 4 * float(v.abs().max()) * 2.0 ** -11 + 1e-5
    n = 70
    t0 = length - n
    last = K.attn_prefill(q[t0:], k[t0:], v[t0:], gate[t0:], kv.k[0], kv.v[0], kv.page_table[0], start=t0, **kw)
    first = K.attn_prefill(q[:n], k[:n], v[:n], gate[:n], kv.k[0], kv.v[0], kv.page_table[0], start=0, **kw)
    assert float((out[t0:] - last).abs().max()) <= tol
    assert float((out[:n] - first).abs().max()) <= tol


@pytest.mark.gpu
@pytest.mark.parametrize("length,start,token", [(6048, 0, 3000), (6035, 0, 6033), (6048, 13, 2995), (6048, 16, 2987)])
def test_attn_prefill_infinite_value_reaches_no_earlier_block(gpu, length, start, token):
    """A value of infinity: the queries before its block of 16 tokens, which
    the causal mask keeps from it, give the bits they give without it, also
    where two blocks of 16 share a workgroup."""
    announce(f"attn_prefill: infinite V at token {token} of {length} after {start}")
    q, k, v, gate = (x.to(gpu) for x in _inputs(31, length, dtype=torch.float16))
    k0, v0 = (x.to(gpu) for x in _inputs(32, max(start, 1), dtype=torch.float16)[1:3])
    outs = []
    for value in (1.0, float("inf")):
        v[token] = value
        kv = _cache(gpu, start + length, dtype=torch.float16)
        inv = rope_inv_freq(10_000_000.0, 64).to(gpu)
        if start:
            K.kv_append_seq(k0, v0, kv.k[0], kv.v[0], kv.page_table[0], start=0, inv_freq=inv)
        outs.append(_run(gpu, kv, q, k, v, gate, start))
    before = token // 16 * 16
    assert bool(torch.isfinite(outs[0]).all())
    assert torch.equal(outs[1][:before], outs[0][:before])
    assert bool((~torch.isfinite(outs[1][token:])).any(-1).all())


@pytest.mark.gpu
@pytest.mark.parametrize("length,start", [(500, 7900), (64, 4000)])
def test_attn_prefill_split_with_infinite_keys(gpu, length, start):
    """Resident keys that score -inf for every query, whole pieces of the split
    among them, weigh nothing in the merge: the unsplit launch's result."""
    announce(f"attn_prefill split: {length} after {start}, keys 40 .. {start - 1} score -inf")
    _, k0, v0, _ = _inputs(41, start, dtype=torch.float32)
    q, k, v, gate = (x.to(gpu) for x in _inputs(42, length, dtype=torch.float32))
    q[..., 100] = q[..., 100].abs() + 0.5  # past the rotary dims
    k0[40:, :, 100] = float("-inf")
    inv = rope_inv_freq(10_000_000.0, 64).to(gpu)
    kv = _cache(gpu, start + length, dtype=torch.float16)
    K.kv_append_seq(k0.to(gpu), v0.to(gpu), kv.k[0], kv.v[0], kv.page_table[0], start=0, inv_freq=inv)
    need = K.prefill_attn_workspace_bytes(length, 16, 2, start, True)
    assert need > 0, "a split case"
    ws = torch.empty(need, dtype=torch.uint8, device=gpu)
    args = (q, k, v, gate, kv.k[0], kv.v[0], kv.page_table[0])
    kw = dict(start=start, inv_freq=inv, scale=SCALE)
    whole = K.attn_prefill(*args, **kw)
    split = K.attn_prefill(*args, **kw, workspace=ws)
    assert bool(torch.isfinite(whole).all())
    vmax = float(max(v.abs().max(), v0.abs().max()))
    assert float((split - whole).abs().max()) <= 4 * vmax * 2.0 ** -11 + 1e-5  # fp16 probabilities of both


def _assert_same_but_rounding(got, want, vmax, fp16_keys):
    """Two launches whose query blocks or pieces differ: the probabilities' rounding about different maxima
    (2^-11 relative with fp16 keys, 2^-16 hi + lo, in products and normaliser of both), then each output's own
    rounding to a 16-bit type (half a unit in the last place of both)."""
    got, want, dt = got.float(), want.float(), want.dtype
    ulp = {torch.float32: 0.0, torch.float16: 2.0 ** -10, torch.bfloat16: 2.0 ** -7}[dt]
    tol = 4 * vmax * (2.0 ** -11 if fp16_keys else 2.0 ** -16) + 1e-5
    assert bool(((got - want).abs() <= tol + ulp * torch.maximum(got.abs(), want.abs())).all())


def _norms(gpu, seed):
    g = torch.Generator().manual_seed(seed)
    return {n: (0.1 * torch.randn(256, generator=g)).to(gpu) for n in ("q_norm_weight", "k_norm_weight")}


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16], ids=["bf16", "fp16"])
@pytest.mark.parametrize("length,start,pages", [(1000, 0, torch.bfloat16), (500, 7900, torch.bfloat16),
                                                (500, 7900, torch.float16), (33, 1024, torch.float16)])
def test_attn_prefill_split_16_bit_activations_and_norms(gpu, length, start, pages, dtype):
    """16-bit q, k, v and gate with q_norm and k_norm, in pieces of 16 and 32 tokens, against the unsplit launch."""
    staged = start == 0
    announce(f"attn_prefill split with norms: {length} after {start}, {dtype} over {pages} pages")
    _, k0, v0, _ = _inputs(51, max(start, 1), dtype=dtype)
    q, k, v, gate = (x.to(gpu) for x in _inputs(52 + length, length, dtype=dtype))
    inv = rope_inv_freq(10_000_000.0, 64).to(gpu)
    kv = _cache(gpu, start + length, dtype=pages)
    if start:
        K.kv_append_seq(k0.to(gpu), v0.to(gpu), kv.k[0], kv.v[0], kv.page_table[0], start=0, inv_freq=inv)
    fp16 = staged or pages == torch.float16
    need = K.prefill_attn_workspace_bytes(length, 16, 2, start, fp16)
    assert need > 0, "a split case"
    args = (q, k, v, gate, kv.k[0], kv.v[0], kv.page_table[0])
    stage = torch.empty(K.prefill_stage_bytes(length, 2), dtype=torch.uint8, device=gpu) if staged else None
    kw = dict(start=start, inv_freq=inv, scale=SCALE, stage=stage, **_norms(gpu, 53))
    whole = K.attn_prefill(*args, **kw)
    pages_whole = kv.k.clone(), kv.v.clone()
    split = K.attn_prefill(*args, **kw, workspace=torch.full((need,), 0xFF, dtype=torch.uint8, device=gpu))
    assert torch.equal(kv.k, pages_whole[0]) and torch.equal(kv.v, pages_whole[1])
    _assert_same_but_rounding(split, whole, float(max(v.abs().max(), v0.abs().max())), fp16)


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16], ids=["bf16", "fp16"])
def test_attn_prefill_32_token_blocks_with_norms(gpu, dtype):
    """q_norm in a 32-token block's prologue: a long prompt's first and last tokens against blocks of 16."""
    length, n = 6031, 70
    announce(f"attn_prefill 32-token blocks with norms: L={length}, {dtype}, fp16 pages")
    q, k, v, gate = (x.to(gpu) for x in _inputs(61, length, dtype=dtype))
    kv = _cache(gpu, length, dtype=torch.float16)
    kw = dict(inv_freq=rope_inv_freq(10_000_000.0, 64).to(gpu), scale=SCALE, **_norms(gpu, 62))
    cache = (kv.k[0], kv.v[0], kv.page_table[0])
    out = K.attn_prefill(q, k, v, gate, *cache, start=0, **kw)
    t0 = length - n
    last = K.attn_prefill(q[t0:], k[t0:], v[t0:], gate[t0:], *cache, start=t0, **kw)
    first = K.attn_prefill(q[:n], k[:n], v[:n], gate[:n], *cache, start=0, **kw)
    vmax = float(v.abs().max())
    _assert_same_but_rounding(out[t0:], last, vmax, True)
    _assert_same_but_rounding(out[:n], first, vmax, True)
