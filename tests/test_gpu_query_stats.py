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
