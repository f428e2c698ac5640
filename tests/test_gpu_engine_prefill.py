"""GPU parity: prompt prefill through the batched engine, then decode.

Two rows of a BatchedAttentionState (one DeltaNet and one attention layer)
take prompts of different lengths with the prefill kernels, then decode three
tokens together; every output is compared with the oracle running the same
sequences token by token, as the reference does
(qwen36_chat_batch.py:255-258 -> qwen36_attention_cache.py:176-317).
"""

from __future__ import annotations

import pytest
import torch

from conftest import announce
from helpers import assert_act_close, assert_state_close
from oracle import qwen36_cpu as O
from router_ia import _native as nat
from router_ia import kernels as K
from router_ia import workloads as W
from router_ia.batched_state import BatchedAttentionState

pytestmark = pytest.mark.gpu


def test_engine_prefill_then_decode(gpu):
    announce("engine: rows prefilled with 100 and 37 tokens, then 3 decode steps")
    prompts = [100, 37]
    steps = 3
    total = max(prompts) + steps
    params = W.gdn_layer_params(61)
    lin = W.gdn_step_inputs(62, total, 2)    # [T, 2, ...]
    att = W.attn_step_inputs(63, total, 2)
    st = BatchedAttentionState(2, 256, num_linear_layers=1, num_full_layers=1, device=gpu, page_shuffle_seed=5,
                               prefill_segment_tokens=64)
    st.set_positions([0, 0])
    dev = gpu
    cw, alog, dtb = params["conv_weight"].to(dev), params["A_log"].to(dev), params["dt_bias"].to(dev)
    got_lin = [[] for _ in prompts]
    got_att = [[] for _ in prompts]
    for row, n in enumerate(prompts):
        st.begin_prefill(row, n)
        o_lin = st.linear_prefill(0, row, lin["mixed"][:n, row].to(dev), cw, lin["a_raw"][:n, row].to(dev),
                                  lin["b_raw"][:n, row].to(dev), gate_mode=nat.RIA_GATE_RAW, A_log=alog,
                                  dt_bias=dtb, out_dtype=torch.float32)
        o_att = st.full_prefill(0, row, att["q"][:n, row].to(dev), att["k"][:n, row].to(dev),
                                att["v"][:n, row].to(dev), att["gate"][:n, row].to(dev))
        st.end_prefill(row, n)
        got_lin[row] += list(o_lin.cpu())
        got_att[row] += list(o_att.float().cpu())
    # decode: row r feeds its own next inputs (token prompts[r] + i)
    st.reserve(steps)
    for i in range(steps):
        idx = [n + i for n in prompts]
        mixed = torch.stack([lin["mixed"][t, r] for r, t in enumerate(idx)]).to(dev)
        a = torch.stack([lin["a_raw"][t, r] for r, t in enumerate(idx)]).to(dev)
        b = torch.stack([lin["b_raw"][t, r] for r, t in enumerate(idx)]).to(dev)
        o_lin = st.linear_step(0, mixed, cw, a, b, gate_mode=nat.RIA_GATE_RAW, A_log=alog, dt_bias=dtb,
                               out_dtype=torch.float32)
        qkvg = {name: torch.stack([att[name][t, r] for r, t in enumerate(idx)]).to(dev)
                for name in ("q", "k", "v", "gate")}
        o_att = st.full_step(0, qkvg["q"], qkvg["k"], qkvg["v"], qkvg["gate"], out_dtype=torch.float32)
        st.advance()
        for r in range(2):
            got_lin[r].append(o_lin[r].cpu())
            got_att[r].append(o_att[r].cpu())
    for r, n in enumerate(prompts):
        s = O.SequenceState()
        for t in range(n + steps):
            beta, g = O.gating(lin["a_raw"][t, r:r + 1], lin["b_raw"][t, r:r + 1], params["A_log"], params["dt_bias"])
            want, s.conv[0], s.linear[0] = O.linear_decode_step(s.conv.get(0), s.linear.get(0),
                                                                 lin["mixed"][t, r:r + 1], params["conv_weight"],
                                                                 beta, g)
            assert_act_close(got_lin[r][t], want[0], f"row {r} DeltaNet token {t}")
            want, s.keys[0], s.values[0] = O.full_decode_step(s.keys.get(0), s.values.get(0), att["q"][t, r:r + 1],
                                                              att["k"][t, r:r + 1], att["v"][t, r:r + 1],
                                                              att["gate"][t, r:r + 1], t)
            assert_act_close(got_att[r][t], want[0], f"row {r} attention token {t}")
        assert_state_close(st.linear_states[0, r].cpu()[None], s.linear[0], f"row {r} final state")


def test_rows_prefilled_on_two_streams(gpu):
    """Two prompts from empty rows, their layers issued in turn on two streams: the serial result's bits."""
    announce("engine: rows prefilled with 1500 and 1100 tokens on two streams, then serially")
    prompts, layers = [1500, 1100], 3
    params = W.gdn_layer_params(71)
    cw, alog, dtb = (params[n].to(gpu) for n in ("conv_weight", "A_log", "dt_bias"))
    g = torch.Generator(device=gpu)
    g.manual_seed(72)
    rows = [[torch.randn((n, *shape), generator=g, device=gpu).to(dt) for shape, dt in (
        ((W.CONV_DIM,), torch.bfloat16), ((32,), torch.float32), ((32,), torch.float32), ((16, 256), torch.bfloat16),
        ((2, 256), torch.bfloat16), ((2, 256), torch.bfloat16), ((16, 256), torch.bfloat16))] for n in prompts]

    def run(streams):
        st = BatchedAttentionState(2, 1600, num_linear_layers=layers, num_full_layers=layers, device=gpu,
                                   prefill_segment_tokens=512)
        st.set_positions([0, 0])
        for row, n in enumerate(prompts):
            st.begin_prefill(row, n)
        torch.cuda.synchronize()
        outs = []
        for layer in range(layers):
            for row, (mixed, a, b, q, k, v, gate) in enumerate(rows):
                with torch.cuda.stream(streams[row]):
                    outs.append(st.linear_prefill(layer, row, mixed, cw, a, b, gate_mode=nat.RIA_GATE_RAW, A_log=alog,
                                                  dt_bias=dtb))
                    outs.append(st.full_prefill(layer, row, q, k, v, gate))
        torch.cuda.synchronize()
        return outs + [st.linear_states, st.conv_rings, st.kv.k, st.kv.v]

    serial = torch.cuda.current_stream()
    want = run([serial, serial])
    got = run([torch.cuda.Stream(), torch.cuda.Stream()])
    assert all(torch.equal(x, y) for x, y in zip(got, want))


def test_full_prefill_splits_short_prompts(gpu):
    """A prompt of 1000 tokens and a turn of 300 after it through the engine, which splits their keys, against
    unsplit launches over a second engine's pages: the same pages, outputs within the probabilities' rounding
    (fp16 keys in the first prompt: 2^-11 relative, bf16 hi + lo after it: 2^-16, in products and normaliser of
    both launches)."""
    announce("engine: full_prefill of 1000 + 300 tokens with split keys")
    g = torch.Generator(device=gpu)
    g.manual_seed(81)
    one, other = (BatchedAttentionState(1, 1400, num_linear_layers=0, num_full_layers=1, device=gpu,
                                        page_shuffle_seed=3) for _ in range(2))
    start = 0
    for n, u in ((1000, 2.0 ** -11), (300, 2.0 ** -16)):
        assert K.prefill_attn_workspace_bytes(n, 16, 2, start, start == 0) > 0, "a split case"
        q, k, v, gate = (torch.randn((n, h, 256), generator=g, device=gpu) for h in (16, 2, 2, 16))
        for st in (one, other):
            st.begin_prefill(0, n)
        got = one.full_prefill(0, 0, q, k, v, gate)
        stage = torch.empty(K.prefill_stage_bytes(n, 2), dtype=torch.uint8, device=gpu) if start == 0 else None
        want = K.attn_prefill(q, k, v, gate, *other.kv.layer(0), other.kv.page_table[0], start=start,
                              inv_freq=other.inv_freq, scale=other.scale, stage=stage)
        assert torch.equal(one.kv.k, other.kv.k) and torch.equal(one.kv.v, other.kv.v)
        # values of every key so far are standard normal, below 6
        assert float((got - want).abs().max()) <= 4 * 6 * u + 1e-5
        for st in (one, other):
            st.end_prefill(0, n)
        start += n


def test_recorded_prefill_replays_beside_eager_prompts(gpu):
    """One row's two layers in a HIP graph, replayed with longer eager prompts of the other row on the same stream
    between (they grow the eager scratch): every replay gives the eager bits."""
    announce("engine: recorded prefill of 700 tokens, replayed three times beside eager prompts of 900 .. 1500")
    n = 700
    params = W.gdn_layer_params(91)
    cw, alog, dtb = (params[x].to(gpu) for x in ("conv_weight", "A_log", "dt_bias"))
    g = torch.Generator(device=gpu)
    g.manual_seed(92)
    mixed = torch.randn((1500, W.CONV_DIM), generator=g, device=gpu).to(torch.bfloat16)
    a, b = (torch.randn((1500, 32), generator=g, device=gpu) for _ in range(2))
    q, k, v, gate = (torch.randn((1500, h, 256), generator=g, device=gpu).to(torch.bfloat16) for h in (16, 2, 2, 16))
    st = BatchedAttentionState(2, 1600, num_linear_layers=1, num_full_layers=1, device=gpu)
    st.set_positions([0, 0])
    st.begin_prefill(0, n)
    st.begin_prefill(1, 1500)

    def run(row, m):
        return [st.linear_prefill(0, row, mixed[:m], cw, a[:m], b[:m], gate_mode=nat.RIA_GATE_RAW, A_log=alog,
                                  dt_bias=dtb), st.full_prefill(0, row, q[:m], k[:m], v[:m], gate[:m])]

    stream = torch.cuda.Stream()
    with torch.cuda.stream(stream):
        want = [x.clone() for x in run(0, n)]
        state = st.linear_states[0, 0].clone()
        torch.cuda.synchronize()
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph, stream=stream):
            outs = run(0, n)
        for m in (900, 1200, 1500):
            run(1, m)
            st.linear_states[0, 0].zero_()
            st.conv_rings[0, 0].zero_()
            graph.replay()
            torch.cuda.synchronize()
            assert all(torch.equal(x, y) for x, y in zip(outs, want))
            assert torch.equal(st.linear_states[0, 0], state)
