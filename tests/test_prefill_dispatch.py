"""Which prefill layers take q and k through the one-pass launch
(fdms_prefill_qk), and which key blocks a prefill attention wave works on."""
import shutil
import subprocess
from pathlib import Path

import pytest
import torch

from native_emulator import cpu_engine
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



@pytest.mark.parametrize("what", ["no tokens", "head width", "fp32 q", "fp16 k", "odd token stride", "odd head stride",
                                  "odd offset", "strided dim", "heads", "lanes", "table type", "strided table",
                                  "odd table rows", "norm type", "strided norm", "odd norm offset"])
def test_prefill_qk_refuses_rows_it_cannot_move(what):
    """Types, strides and alignments its 16-byte moves do not take."""
    hq, hkv = (256, 16) if what == "lanes" else (4, 3) if what == "heads" else (HQ, HKV)
    d = 32 if what == "head width" else D
    tokens = 0 if what == "no tokens" else TOKENS
    width = (hq + 2 * hkv) * d + (4 if what == "odd token stride" else 0)
    store = torch.zeros(TOKENS * 2 * width + 16, dtype=torch.bfloat16)
    offset = 4 if what == "odd offset" else 0
    rows = store[offset:offset + tokens * width].view(tokens, width)
    q, k = rows[:, :hq * d].view(-1, hq, d), rows[:, hq * d:(hq + hkv) * d].view(-1, hkv, d)
    if what == "odd head stride":
        q = store.as_strided((tokens, hq, d), (width, d + 4, 1))
    if what == "strided dim":
        k = store.as_strided((tokens, hkv, d), (2 * width, 2 * d, 2))
    q = q.float() if what == "fp32 q" else q
    k = k.half() if what == "fp16 k" else k
    table = torch.zeros(16, 1, d)
    if what == "table type":
        table = table.double()
    if what == "strided table":
        table = torch.zeros(16, 1, 2 * d)[..., ::2]
    if what == "odd table rows":
        table = torch.zeros(16, 1, d + 2)[..., :d]
    norms = _norms(d)
    if what == "norm type":
        norms[0].weight.data = norms[0].weight.data.float()
    if what == "strided norm":
        norms[1].weight.data = torch.ones(2 * d, dtype=torch.bfloat16)[::2]
    if what == "odd norm offset":
        norms[1].weight.data = torch.ones(d + 4, dtype=torch.bfloat16)[4:]
    assert not prefill_qk_supported(q, k, table, norms)

def _prefill(hooked=(), replace=None):
    """Prefill logits of a two-layer QK-norm model with forward hooks on the
    named modules of layer 1; returns (logits, hook calls, kernel calls)."""
    with cpu_engine() as emu:
        from fastdms_amd import LLM, SamplingParams
        llm = LLM("tiny-qwen3", max_model_len=512, max_num_seqs=2, max_num_batched_tokens=512, enforce_eager=True,
                  fused_greedy_head=False, dms_window_size=32, dms_alpha_scale=10.0, dms_alpha_offset=5.0)
        attn = llm.model_runner.model.model.layers[1].self_attn
        seen, handles = [], []
        for name in hooked:
            def hook(module, args, output, name=name):
                if not (name == "qkv_proj" and seen):
                    seen.append((name, output, output.clone() if name == "qkv_proj" else None))
            handles.append(getattr(attn, name).register_forward_hook(hook))
        if replace:
            replace(attn)
        llm.add_request(list(range(1, 150)), SamplingParams(temperature=0.0, max_tokens=2, ignore_eos=True))
        emu.calls.clear()
        llm.step()
        for h in handles:
            h.remove()
        logits = llm.model_runner.model.lm_head.last_logits.clone()
        calls = list(emu.calls)
        llm.exit()
    return logits, seen, calls


def test_prefill_hooks_see_their_modules():
    """A forward hook on q_norm, k_norm or rotary_emb is called at prefill, and
    one on qkv_proj keeps rows that the norms left alone; the results stay."""
    want, _, calls = _prefill()
    assert calls.count("fdms_prefill_qk") == 2
    for name in ("q_norm", "k_norm", "rotary_emb", "qkv_proj"):
        got, seen, calls = _prefill((name,))
        assert [s[0] for s in seen][:1] == [name]
        # the rotary module is shared by the layers
        assert calls.count("fdms_prefill_qk") == (0 if name == "rotary_emb" else 1)
        assert torch.equal(got, want)
        if name == "qkv_proj":
            assert torch.equal(seen[0][1], seen[0][2])


def test_prefill_runs_replaced_modules():
    """A norm of another class, or with its own forward, is called."""
    want, _, _ = _prefill()
    called = []

    class Wrapped(torch.nn.Module):
        def __init__(self, inner):
            super().__init__()
            self.inner = inner

        def forward(self, x):
            called.append("class")
            return self.inner(x)

    def other_class(attn):
        attn.q_norm = Wrapped(attn.q_norm)

    def own_forward(attn):
        plain = attn.k_norm.forward
        attn.k_norm.forward = lambda x: (called.append("forward"), plain(x))[1]

    for replace, name in ((other_class, "class"), (own_forward, "forward")):
        got, _, _ = _prefill(replace=replace)
        assert name in called
        assert torch.equal(got, want)


def test_prefill_attention_block_ranges(tmp_path):
    """Every row's visible keys and no others, the same barriers in every wave of
    a workgroup, no work in a wave past the sequence's end."""
    gxx = shutil.which("g++")
    if gxx is None:
        pytest.skip("g++ not available")
    root = Path(__file__).resolve().parents[1]
    exe = tmp_path / "prefill_blocks_check"
    subprocess.run([gxx, "-std=c++17", "-O1", "-I", str(root / "fastdms_amd" / "csrc"),
                    str(root / "tests" / "prefill_blocks_check.cpp"), "-o", str(exe)], check=True)
    res = subprocess.run([str(exe)], capture_output=True, text=True, timeout=120)
    assert res.returncode == 0 and res.stdout.strip() == "ok", res.stdout + res.stderr
