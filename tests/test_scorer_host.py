"""CPU: what the scorers' host side hands to the library (workspaces, which calls it takes), no kernels run."""
import pytest


@pytest.mark.parametrize("batch,cols", [(1, 4096), (1, 3584), (2, 256), (7, 1024), (600, 64)])
def test_the_mean_of_a_prompt_without_its_sinks_fits_the_workspace_of_the_whole_prompt(batch, cols):
    # a prompt's workspace is asked for with all its tokens, the mean then leaves the sinks (up to 64 tokens) out
    from kvquant import _lib
    need = _lib.lib.odmkv_token_mean_workspace_bytes
    for rows in [*range(1, 700), *range(8100, 8500), 32768, 65537, 131072 + 4]:
        whole = need(batch, rows, cols)
        assert all(need(batch, rows - n, cols) <= whole for n in range(1, min(rows, 65)))


@pytest.mark.parametrize("batch,cols", [(1, 4096), (1, 3584), (2, 256), (7, 1024), (600, 64)])
def test_the_mean_workspace_holds_every_run_of_rows(batch, cols):
    # the kernel's cut: runs of 16 to 256 rows, as many as put two workgroups on each of 256 compute units
    from kvquant import _lib
    for per_thread in (8, 4):
        runs = max(1, 512 // (batch * -(-cols // (256 * per_thread))))
        for rows in (1, 15, 16, 17, 4095, 4097, 8189, 8193, 65537, 131073, 131072 * 2 + 1):
            chunk = min(256, max(16, -(-rows // runs)))
            assert _lib.lib.odmkv_token_mean_workspace_bytes(batch, rows, cols) >= batch * -(-rows // chunk) * cols * 4


class _Fake:
    """The face of a GPU tensor: what the covering checks of RiskScorer.score_prompt look at."""
    is_cuda = True

    def __init__(self, shape, dtype, device):
        import torch
        self.shape, self.dtype, self.device = torch.Size(shape), dtype, torch.device(device)

    def dim(self):
        return len(self.shape)

    def stride(self, i=None):
        s = [1]
        for n in reversed(self.shape[1:]):
            s.insert(0, s[0] * n)
        return tuple(s) if i is None else s[i]

    def data_ptr(self):
        return 4096


@pytest.mark.parametrize("away", ["keys", "values", "hidden", "weight", "bias", None])
def test_a_prompt_spread_over_devices_is_left_to_the_general_path(away, monkeypatch):
    import torch
    from types import SimpleNamespace
    from kvquant import RiskScorer, scorer as sc

    class Reached(Exception):
        pass

    def reached(*args, **kw):
        raise Reached

    where = {n: "cuda:1" if n == away else "cuda:0" for n in ("keys", "values", "hidden", "weight", "bias")}
    f16, B, H, T, hidden, n_q = torch.float16, 2, 2, 40, 64, 4
    keys, values = (_Fake((B, H, T, 128), f16, where[n]) for n in ("keys", "values"))
    h = _Fake((B, T, hidden), f16, where["hidden"])
    w, b = _Fake((n_q * 128, hidden), f16, where["weight"]), _Fake((n_q * 128,), f16, where["bias"])
    monkeypatch.setattr(sc, "_plain_projection", lambda module: (w, b))
    monkeypatch.setattr(sc, "lib", SimpleNamespace(odmkv_prompt_scores_workspace_bytes=reached, odmkv_prompt_scores=reached))
    module = SimpleNamespace(config=SimpleNamespace(num_attention_heads=n_q, head_dim=128))
    scorer = RiskScorer(n_future_positions=8, n_sink=4, epsilon=1e-2)
    scorer.normalize_grain = "global"
    call = lambda: scorer.score_prompt(keys, values, 0, module=module, hidden_states=h, out=object())
    if away is None:
        with pytest.raises(Reached):                       # the same call on one device is the library's
            call()
    else:
        assert call() is None


@pytest.mark.parametrize("where", ["class", "instance", "nowhere"])
@pytest.mark.parametrize("grain", ["layer", "global", "head"])
def test_a_window_scorers_own_normalisation_is_asked(grain, where, monkeypatch):
    import torch
    from types import SimpleNamespace
    from kvquant import WindowRiskScorer, scorer as sc
    core = torch.arange(12.0).reshape(2, 6)

    class Halved(WindowRiskScorer):
        def _maybe_normalize(self, raw):
            return raw / 2

    scorer = (Halved if where == "class" else WindowRiskScorer)(window=4, n_future_positions=8, n_sink=2, epsilon=1e-2)
    if where == "instance":
        scorer._maybe_normalize = lambda raw: raw / 2
    scorer.normalize_grain = grain
    monkeypatch.setattr(sc, "_launch_window_attention", lambda *a: None)
    monkeypatch.setattr(sc, "_launch_score", lambda *a: core)
    monkeypatch.setattr(sc, "_scale_on_device", lambda scores, pad, scale: "on the device")
    monkeypatch.setattr(scorer, "_window_queries", lambda module, h, w: None)
    keys = torch.zeros(2, 8, 128)
    got = scorer.score_prefill(keys, keys, 0, module=SimpleNamespace(), hidden_states=torch.zeros(1, 8, 64))
    padded = torch.cat([torch.full((2, 2), 11.0), core], dim=1)
    if where == "nowhere":
        assert got == "on the device" if grain != "head" else torch.equal(got, sc._normalize_scores(padded, grain=grain))
    else:
        assert torch.equal(got, padded / 2)


def test_a_batch_of_long_prompts_does_not_grow_the_workspace():
    from kvquant import _lib
    need = _lib.lib.odmkv_prompt_scores_workspace_bytes
    for T, hidden, n_q, n_kv in ((131072, 4096, 32, 8), (32768, 3584, 28, 4), (4096, 2048, 16, 2), (100, 1024, 8, 8)):
        one = need(1, T, hidden, n_q, n_kv)
        assert one > T * (n_q + n_kv) * 4
        for B in (2, 3, 16, 64, 300, 9000):
            assert need(B, T, hidden, n_q, n_kv) <= max(one, 64 << 20)
    assert need(2, 8192, 4096, 32, 8) > need(1, 8192, 4096, 32, 8)          # (short ones are still scored together)
