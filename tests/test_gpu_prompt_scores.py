"""GPU: a prompt's scores in one call (odmkv_prompt_scores, odmkv_project_rows) against the same stages one by one."""
from types import SimpleNamespace

import pytest
import torch
from torch import nn

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("batch,rows,cols", [(1, 1, 8), (2, 7, 520), (3, 128, 2048), (7, 1025, 4104)])
def test_projected_rows(batch, rows, cols, dtype):
    from kvquant import _lib
    g = torch.Generator(device="cuda").manual_seed(rows)
    w = (torch.randn(rows, cols + 8, generator=g, device="cuda") * cols ** -0.5).to(dtype)[:, :cols]
    x, bias = (torch.randn(n, generator=g, device="cuda").to(dtype) for n in ((batch, cols), (rows,)))
    for b in (None, bias):
        want = x.double() @ w.double().t().contiguous() + (0 if b is None else b.double())
        for out_dtype in (dtype, torch.float32):
            out = torch.empty(batch, rows, dtype=out_dtype, device="cuda")
            _lib.check(_lib.lib.odmkv_project_rows(w.data_ptr(), w.stride(0), _lib.ptr(b), x.data_ptr(), _lib._DT[dtype], batch, rows, cols,
                                                   out.data_ptr(), _lib.dtype_code(out), _lib.stream_ptr(out.device)))
            step = {torch.float16: 2 ** -11, torch.bfloat16: 2 ** -8}[dtype]
            assert ((out.double() - want).abs() <= step * want.abs() + 1e-5).all() and torch.equal(out, out.to(dtype).to(out_dtype))


@pytest.mark.parametrize("rope", [True, False])
@pytest.mark.parametrize("B,Hq,Hkv,T,dtype,gap", [(1, 4, 4, 5, torch.float16, 0), (2, 8, 2, 300, torch.bfloat16, 0), (3, 7, 1, 777, torch.float16, 0),
                                                  (2, 16, 2, 1030, torch.float16, 3)])
def test_scores_of_all_sequences(B, Hq, Hkv, T, dtype, gap, rope):
    from kvquant import RiskScorer
    g = torch.Generator(device="cuda").manual_seed(T)
    hidden = 256
    module = nn.Module()
    module.config = SimpleNamespace(num_attention_heads=Hq, head_dim=128)
    module.q_proj = nn.Linear(hidden, Hq * 128, bias=Hq == 7, device="cuda", dtype=dtype)
    asked = []
    if rope:
        def rotary(x, pos):
            asked.append(1)
            a = pos[..., None].float() * (500000.0 ** (-torch.arange(0, 128, 2, device="cuda").float() / 128))
            a = torch.cat((a, a), dim=-1)
            return a.cos().to(x.dtype), a.sin().to(x.dtype)
        module.rotary_emb = rotary
    h = (torch.randn(B, T, hidden, generator=g, device="cuda") + 0.3).to(dtype)
    k, v = (torch.randn(B, Hkv + gap, T, 128, generator=g, device="cuda").to(dtype)[:, gap:] for _ in range(2))
    scorer = RiskScorer(n_future_positions=64, n_sink=4, epsilon=1e-2)
    scorer.normalize_grain = "global"
    tables = {}
    with torch.inference_mode():
        got = [scorer.score_prompt(k, v, i, module=module, hidden_states=h, rope_tables=tables) for i in range(2)][1]
        assert len(asked) == (1 if rope else 0)                                   # the layers of a forward share the tables
        for b in range(B):
            want = scorer.score_prefill(k[b], v[b], 0, module=module, hidden_states=h[b:b + 1])
            assert (got[b] - want).norm() <= 2e-3 * want.norm()                    # (mean queries may land one step of the type apart)
            assert torch.equal(got[b][:, :4], got[b][:, 4:].max().expand(Hkv, 4))   # the sinks take their own sequence's largest
        module.q_norm = nn.Identity()
        assert scorer.score_prompt(k, v, 0, module=module, hidden_states=h) is None


@pytest.mark.parametrize("T", [8193, 8196, 8197])
def test_prompts_whose_mean_is_cut_otherwise_without_the_sinks(T):
    test_scores_of_all_sequences(2, 4, 2, T, torch.float16, 0, True)


@pytest.mark.parametrize("gap", [0, 1])
def test_a_batch_scored_in_turns(gap):
    # 4.2 MB of workspace a sequence, 15 sequences a turn (64 MB)
    from kvquant import _lib
    assert _lib.lib.odmkv_prompt_scores_workspace_bytes(17, 100001, 256, 8, 1) < 17 * _lib.lib.odmkv_prompt_scores_workspace_bytes(1, 100001, 256, 8, 1) / 1.1
    test_scores_of_all_sequences(17, 8, 1, 100001, torch.float16, gap, True)


def test_a_projection_that_is_watched_or_cast_is_called():
    from kvquant import RiskScorer
    module = nn.Module()
    module.config = SimpleNamespace(num_attention_heads=2, head_dim=128)
    module.q_proj = nn.Linear(64, 256, bias=False, device="cuda", dtype=torch.float16)
    k = torch.randn(1, 2, 40, 128, device="cuda", dtype=torch.float16)
    h = torch.randn(1, 40, 64, device="cuda", dtype=torch.float16)
    scorer = RiskScorer(n_future_positions=8, n_sink=4, epsilon=1e-2)
    scorer.normalize_grain = "global"
    call = lambda: scorer.score_prompt(k, k, 0, module=module, hidden_states=h)
    with torch.inference_mode():
        assert call() is not None
        with torch.autocast("cuda", dtype=torch.bfloat16):
            assert call() is None
        handle = nn.modules.module.register_module_forward_hook(lambda m, i, o: None)
        try:
            assert call() is None
        finally:
            handle.remove()
        handle = module.q_proj.register_forward_hook(lambda m, i, o: None)
        assert call() is None
        handle.remove()
        assert call() is not None
