"""Which prefill layers take q and k through the one-pass launch (fdms_prefill_qk)."""
import pytest
import torch

from fastdms_amd.engine.dms import prefill_qk_supported
from fastdms_amd.layers.layernorm import RMSNorm

TOKENS, HQ, HKV, D = 3, 4, 2, 128


def _views(d=D, k_tokens=TOKENS):
    rows = torch.zeros(TOKENS, (HQ + 2 * HKV) * d, dtype=torch.bfloat16)
    q = rows[:, :HQ * d].view(-1, HQ, d)
    return q, rows[:k_tokens, HQ * d:(HQ + HKV) * d].view(-1, HKV, d)


def _norms(d=D):
    norms = (RMSNorm(d), RMSNorm(d))
    for n in norms:
        n.weight.data = n.weight.data.to(torch.bfloat16)
    return norms


def test_prefill_qk_takes_matching_rows():
    q, k = _views()
    assert prefill_qk_supported(q, k, torch.zeros(16, 1, D), _norms())
    assert prefill_qk_supported(q, k, torch.zeros(16, 1, D))


@pytest.mark.parametrize("what", ["narrow table", "wide table", "q norm", "k norm", "k tokens", "k width"])
def test_prefill_qk_refuses_rows_it_would_read_past(what):
    """The kernel reads head_dim values of a table row and of each norm weight,
    and as many k rows as q rows: anything narrower would be read out of range."""
    q, k = _views(k_tokens=TOKENS - 1 if what == "k tokens" else TOKENS)
    norms = _norms()
    table = torch.zeros(16, 1, {"narrow table": D // 2, "wide table": 2 * D}.get(what, D))
    if what == "q norm":
        norms = (_norms(D // 2)[0], norms[1])
    if what == "k norm":
        norms = (norms[0], _norms(D // 2)[1])
    if what == "k width":
        k = _views(D // 2)[1]
    assert not prefill_qk_supported(q, k, table, norms)
