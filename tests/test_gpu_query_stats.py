"""GPU: the mean over a prompt's hidden states (odmkv_token_mean) and the averaged RoPE (odmkv_average_rope) against torch."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16, torch.float32])
@pytest.mark.parametrize("b,t,hidden", [(1, 1, 8), (2, 17, 264), (1, 515, 4096), (3, 2049, 2056), (1, 40000, 128)])
def test_token_mean(b, t, hidden, dtype):
    from kvquant.attention_utils import _token_mean
    g = torch.Generator(device="cuda").manual_seed(t)
    x = (torch.randn(b, t + 4, hidden, generator=g, device="cuda") + 0.5).to(dtype)[:, 4:]
    got, want = _token_mean(x), x.double().mean(dim=1, keepdim=True)
    assert got.dtype == dtype and got.shape == want.shape
    step = {torch.float16: 2 ** -11, torch.bfloat16: 2 ** -8, torch.float32: 1e-6}[dtype]
    assert ((got.double() - want).abs() <= step * want.abs() + 1e-6).all()


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16, torch.float32])
@pytest.mark.parametrize("heads,positions", [(1, 1), (28, 37), (40, 512)])
def test_averaged_rope(heads, positions, dtype):
    from types import SimpleNamespace
    from kvquant.attention_utils import _apply_avg_rope
    g = torch.Generator(device="cuda").manual_seed(heads)
    mu = torch.randn(1, heads, 128, generator=g, device="cuda").to(dtype)

    def rotary(x, pos):
        a = pos.cpu()[..., None].float() * (500000.0 ** (-torch.arange(0, 128, 2).float() / 128))
        a = torch.cat((a, a), dim=-1)
        return a.cos().to(x), a.sin().to(x)                        # (one table for both: the device's cos differs in the last bit)
    got, _ = _apply_avg_rope(SimpleNamespace(rotary_emb=rotary), mu, None, 600, positions)
    want, _ = _apply_avg_rope(SimpleNamespace(rotary_emb=rotary), mu.cpu(), None, 600, positions)     # the tensor operations
    # the rounding points are the same; a mean of cos or sin may land one step of the type away, elements near zero by that noise
    step = {torch.float16: 2 ** -10, torch.bfloat16: 2 ** -7, torch.float32: 2e-6}[dtype]
    assert ((got.cpu() - want.float()).abs() <= 2 * step * (want.float().abs() + 0.1)).all()


def _rotary(x, pos):
    a = pos.cpu()[..., None].float() * (500000.0 ** (-torch.arange(0, 128, 2).float() / 128))
    a = torch.cat((a, a), dim=-1)
    return a.cos().to(x), a.sin().to(x)


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("heads,t,rope", [(1, 1, False), (3, 17, True), (8, 1023, True), (32, 4097, False), (2, 40001, True)])
def test_query_covariance(heads, t, rope, dtype):
    from types import SimpleNamespace
    from kvquant.attention_utils import _apply_avg_rope
    from kvquant.scorer import _query_covariance
    g = torch.Generator(device="cuda").manual_seed(t)
    q = torch.randn(1, t, heads, 128, generator=g, device="cuda")
    q = (q * torch.rand(128, generator=g, device="cuda") + 4.0 * torch.randn(128, generator=g, device="cuda")).to(dtype).transpose(1, 2)
    module = SimpleNamespace(rotary_emb=_rotary) if rope else SimpleNamespace()
    mu, cov = _query_covariance(module, q, 77, 64)
    d = q.double().cpu()
    want_mu = d.mean(dim=2)
    c = d - want_mu.unsqueeze(2)
    want_mu, want_cov = _apply_avg_rope(module, want_mu, c.transpose(-1, -2).contiguous() @ c / t, 77, 64)
    assert (mu.cpu().double() - want_mu).abs().max() <= 2e-6 * want_mu.abs().max()
    # means of up to twelve times the deviation: they must not cost the covariance anything
    assert (cov.cpu().double() - want_cov).abs().max() <= 3e-6 * (want_cov.abs().max() + 1e-3)
    assert torch.equal(cov, cov.transpose(-1, -2)) or rope


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16, torch.float32])
@pytest.mark.parametrize("heads,w", [(1, 1), (28, 64), (5, 33)])
def test_window_queries_rotated(heads, w, dtype):
    from kvquant import _lib
    from kvquant.attention_utils import _apply_rotary_pos_emb_q
    g = torch.Generator(device="cuda").manual_seed(w)
    q = torch.randn(1, w, heads, 128, generator=g, device="cuda").to(dtype).transpose(1, 2)
    cos, sin = _rotary(q, torch.arange(900, 900 + w)[None])
    out = torch.empty(heads, w, 128, dtype=dtype, device="cuda")
    _lib.check(_lib.lib.odmkv_rotate_queries(q.data_ptr(), _lib.dtype_code(q), heads, w, q.stride(1), q.stride(2), cos.data_ptr(),
                                             sin.data_ptr(), out.data_ptr(), _lib.stream_ptr(q.device)))
    assert torch.equal(out, _apply_rotary_pos_emb_q(q, cos, sin)[0])


@pytest.mark.parametrize("rows,cols,pad", [(1, 1, 0), (3, 255, 4), (8, 32764, 4), (2, 1000, 0)])
def test_scores_normalised_on_the_device(rows, cols, pad):
    from kvquant.scorer import _normalize_scores, _scale_on_device
    x = torch.randn(rows, cols, generator=torch.Generator().manual_seed(cols))
    for y in (x, torch.full_like(x, 3.0)):
        padded = torch.cat([y.max().expand(rows, pad), y], dim=1)
        assert torch.equal(_scale_on_device(y.cuda(), pad, False).cpu(), padded)
        assert torch.allclose(_scale_on_device(y.cuda(), pad, True).cpu(), _normalize_scores(padded), rtol=1e-6, atol=1e-7)
    x[0, cols // 2] = float("nan")
    assert _scale_on_device(x.cuda(), pad, True).isnan().all()


def test_rotary_modules_see_mean_queries():
    # a rotary module may read the dimension, the heads or the type off the tensor it is handed
    from types import SimpleNamespace
    from kvquant import ExpectedAttentionScorer, RiskScorer
    seen = []

    def rotary(x, pos):
        seen.append((tuple(x.shape), x.dtype))
        a = pos[..., None].float() * (500000.0 ** (-torch.arange(0, x.shape[-1], 2, device=x.device).float() / x.shape[-1]))
        a = torch.cat((a, a), dim=-1)
        return a.cos().to(x.dtype), a.sin().to(x.dtype)
    module = torch.nn.Module()
    module.config = SimpleNamespace(num_attention_heads=4, head_dim=128)
    module.q_proj = torch.nn.Linear(64, 512, bias=False, device="cuda", dtype=torch.float16)
    module.rotary_emb = rotary
    k = torch.randn(1, 2, 60, 128, device="cuda", dtype=torch.float16)
    h = torch.randn(1, 60, 64, device="cuda", dtype=torch.float16)
    risk = RiskScorer(n_future_positions=16, n_sink=4, epsilon=1e-2)
    risk.normalize_grain = "global"
    with torch.inference_mode():
        assert risk.score_prompt(k, k, 0, module=module, hidden_states=h) is not None
        risk.score_prefill(k[0], k[0], 0, module=module, hidden_states=h)
        ExpectedAttentionScorer(n_future_positions=16, n_sink=4).score_prefill(k[0], k[0], 0, module=module, hidden_states=h)
    assert seen == [((1, 4, 128), torch.float16)] * 2 + [((1, 4, 128), torch.float32)]


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("t", [597, 8192, 32764])
def test_means_of_queries_are_no_further_from_fp64_than_fp32_means(t, dtype):
    # relative 2-norm errors over 32 x 128 means: 0.5 to 0.9e-7 in fp32 (torch)
    from types import SimpleNamespace
    from kvquant.scorer import _query_covariance
    g = torch.Generator(device="cuda").manual_seed(t)
    q = (torch.randn(1, 32, t, 128, generator=g, device="cuda") + 0.5 * torch.randn(1, 32, 1, 128, generator=g, device="cuda")).to(dtype)
    mu, _ = _query_covariance(SimpleNamespace(), q, t, 0)
    want = q.double().mean(dim=2)
    off = lambda x: float((x.double() - want).norm() / want.norm())
    assert off(mu) <= 1.2 * off(q.float().mean(dim=2))
