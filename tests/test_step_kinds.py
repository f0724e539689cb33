"""Which steps count as steps of single tokens."""
from __future__ import annotations

import pytest

import llama_cu_amd  # noqa: F401
from llama_cu_amd.engine.batch import StepContext


@pytest.mark.parametrize("q_lens,single", [([1], True), ([1, 1, 1], True), ([1, 2], False), ([1, 0, 1], False), ([1, 0], False), ([], False)])
def test_single_tokens(q_lens, single):
    """Kernels that take row r for request r's are chosen by it: a request that feeds nothing moves the rows behind it."""
    step = StepContext(n=sum(q_lens), n_req=len(q_lens), tokens=None, positions=None, req_of_token=None, q_start=None, ctx_len=None, state_slot=None,
                       logit_rows=None, n_logits=0, block_tables=[], slot_maps=[], q_lens=q_lens, ctx_lens=[3] * len(q_lens))
    assert step.decode_only == single
