"""Scratch memory of the engine's prompt prefill, on the host (the kernels are replaced by recorders).

Prompts in flight on two streams, or in a recorded graph and outside it, must
not share memory that one of them still computes in.
"""

from __future__ import annotations

from types import SimpleNamespace

import pytest
import torch

from router_ia import kernels as K
from router_ia.batched_state import BatchedAttentionState


class _Calls:
    """A state without a GPU and the scratch tensors of its prefill calls."""

    def __init__(self, monkeypatch, seen: list[int]):
        self.stream, self.capturing, self.held = 1, False, []
        monkeypatch.setattr(K, "gdn_prefill", self._record)
        monkeypatch.setattr(K, "attn_prefill", self._record)
        monkeypatch.setattr(torch._C, "_cuda_getCurrentRawStream", lambda device: self.stream, raising=False)
        monkeypatch.setattr(torch.cuda, "is_current_stream_capturing", lambda: self.capturing)
        st = self.st = object.__new__(BatchedAttentionState)  # only what the prefill methods read
        st.device = torch.device("cpu")
        st.num_k_heads, st.num_v_heads, st.num_q_heads, st.num_kv_heads = 16, 32, 16, 2
        st.prefill_segment_tokens, st._prefill_scratch, st._device_index = 4096, {}, 0
        st.linear_states = st.conv_rings = torch.zeros((1, 2, 1))
        st.inv_freq, st.scale, st._host_seen = None, 1.0, seen
        st.kv = SimpleNamespace(layer=lambda i: (None, None), page_table=[None, None], dtype=torch.bfloat16)

    def _record(self, *args, **kw):
        self.held.extend(t for t in (kw.get("workspace"), kw.get("stage")) if t is not None)

    def prefill(self, row: int, length: int) -> set[int]:
        """Addresses of the scratch of one row's two layers (every tensor so far stays alive)."""
        first, q = len(self.held), torch.empty((length, 0))
        self.st.linear_prefill(0, row, q, None, None, None, out=q)
        self.st.full_prefill(0, row, q, None, None, None, out=q)
        return {t.data_ptr() for t in self.held[first:]}


@pytest.mark.parametrize("seen", [[0, 0], [700, 900]], ids=["from empty", "continued"])
@pytest.mark.parametrize("length", [64, 300, 5000])
def test_streams_share_no_scratch(monkeypatch, seen, length):
    calls = _Calls(monkeypatch, seen)
    one = calls.prefill(0, length)
    calls.stream = 2
    other = calls.prefill(1, length)
    assert one and other and not one & other


def test_scratch_of_a_recorded_graph_is_its_own(monkeypatch):
    calls = _Calls(monkeypatch, [0, 0])
    eager = calls.prefill(0, 300)
    calls.capturing = True
    recorded = calls.prefill(0, 300)
    calls.capturing = False
    assert not recorded & (eager | calls.prefill(1, 300))
