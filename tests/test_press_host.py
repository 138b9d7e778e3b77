"""CPU: host logic of the press classes and the attention patch (no kernels run)."""
import numpy as np
import pytest
import torch


def _scorer():
    from kvquant import RiskScorer
    return RiskScorer(n_future_positions=512, n_sink=4, use_vnorm=True, epsilon=1e-2)


def test_package_exports_reference_names():
    import kvquant
    for name in ("scores_to_bits", "ratio_scores_to_bits", "optimal_scores_to_bits", "calibrate_epsilon",
                 "effective_bits", "DEFAULT_BIT_LEVELS", "BaseScorer", "ExpectedAttentionScorer", "RiskScorer",
                 "TurboQuantBackendPress", "TurboQuantPerTokenPress", "TurboQuantPerTokenBackendPress"):
        assert hasattr(kvquant, name), name


def test_constructor_errors_follow_reference():
    from kvquant import TurboQuantPerTokenBackendPress, TurboQuantPerTokenPress
    with pytest.raises(ValueError, match="explicit scorer"):
        TurboQuantPerTokenPress()
    with pytest.raises(ValueError, match="below 2"):
        TurboQuantPerTokenBackendPress(scorer=_scorer(), bit_levels=(0, 1, 2, 16), key_quantizer="prod")
    p = TurboQuantPerTokenBackendPress(scorer=_scorer(), bit_levels=(0, 2, 3, 4, 8, 16), key_quantizer="mse",
                                       value_quantizer="mse", target_avg_bits=2.0)
    assert p._decode_bit_levels == (2, 3, 4, 8, 16) and p.decode_quant and p.buffer_size == 128
    q = TurboQuantPerTokenBackendPress(scorer=_scorer(), bit_levels=(0, 2, 16), key_quantizer="mse",
                                       value_quantizer="mse", allow_decode_eviction=True)
    assert q._decode_bit_levels == (0, 2, 16)


def test_sink_mask_and_uniform_partition():
    from kvquant import TurboQuantPerTokenPress
    p = TurboQuantPerTokenPress(scorer=_scorer(), bit_levels=(0, 2, 4, 16), sink_tokens=4, value_quantizer="mse")
    m = p._build_sink_mask(3, 10, "cpu")
    assert m.shape == (3, 10) and m[:, :4].all() and not m[:, 4:].any()
    assert TurboQuantPerTokenPress(scorer=_scorer(), value_quantizer="mse")._build_sink_mask(2, 5, "cpu") is None
    s = torch.tensor([[0.0, 0.1, 0.3, 0.6, 0.9, 1.0, 0.2, 0.4, 0.7, 0.99]]).repeat(3, 1)
    bits = p._compute_bits(s, m)               # neither ratios nor target: uniform partition, sinks 16
    assert bits[:, :4].eq(16).all()
    assert bits[0, 4:].tolist() == [16, 16, 0, 2, 4, 16]


def test_search_hyperplane_gives_negative_logits():
    from kvquant.attention_patch import search_hyperplane
    g = torch.Generator().manual_seed(0)
    x = torch.randn(6, 12, 128, generator=g) + 0.5
    y = search_hyperplane(x)
    assert y.shape == (6, 128)
    logits = torch.einsum("nmd,nd->nm", x, y)
    assert (logits < -1e3).all()


def test_group_and_scalar_value_quantisers():
    from kvquant.press import _qd_scalar, _qd_values_group
    g = torch.Generator().manual_seed(1)
    x = torch.randn(5, 128, generator=g)
    for b in (2, 4, 8):
        y = _qd_values_group(x, b, 32)
        xg = x.numpy().reshape(5, 4, 32)
        lo, hi = xg.min(-1, keepdims=True), xg.max(-1, keepdims=True)
        sc = np.maximum((hi - lo) / (2 ** b - 1), 1e-10)
        want = (np.clip(np.round((xg - lo) / sc), 0, 2 ** b - 1) * sc + lo).reshape(5, 128)
        assert np.allclose(y.numpy(), want, atol=1e-6)
        assert (y - x).abs().max() <= (hi - lo).max() / (2 ** b - 1) * 0.5 + 1e-6
        z = _qd_scalar(x, b)
        assert (z - x).abs().max() <= (x.amax(-1) - x.amin(-1)).max() / (2 ** b - 1) * 0.5 + 1e-6
    assert torch.equal(_qd_values_group(x[:, :100], 2, 32), _qd_scalar(x[:, :100], 2))   # d not divisible: per-vector


def test_observed_ratios_and_cached_allocation():
    from kvquant import TurboQuantPerTokenBackendPress
    p = TurboQuantPerTokenBackendPress(scorer=_scorer(), bit_levels=(0, 2, 4, 16), key_quantizer="mse",
                                       value_quantizer="mse", target_avg_bits=2.0, sink_tokens=4, buffer_size=8)
    T = 4 + 40 + 8
    bits = torch.full((1, 2, T), 16, dtype=torch.int32)
    bits[0, 0, 4:44] = torch.tensor([0] * 10 + [2] * 20 + [4] * 10)
    bits[0, 1, 4:44] = torch.tensor([2] * 30 + [4] * 10)
    p._record_observed_ratios(3, bits)
    assert p._observed_ratios[(3, 0)] == ((0, 0.25), (2, 0.5), (4, 0.25))
    assert p._observed_ratios[(3, 1)] == ((2, 0.75), (4, 0.25))
    # flush allocation from the cached ratios, eviction not allowed at decode: level 0 dropped, rest renormalised
    n = 12
    pos = torch.stack([torch.zeros(2 * n, dtype=torch.long), torch.arange(2).repeat_interleave(n),
                       torch.arange(n).repeat(2)], dim=-1)
    scores = torch.linspace(0, 1, 2 * n)
    out = p._allocate_bits_via_cached_ratios(scores, pos, 2, 3, {2, 4, 16})
    assert out[:n].tolist() == [2] * 8 + [4] * 4          # 2/3 and 1/3 of 12
    assert out[n:].tolist() == [2] * 9 + [4] * 3
    assert p._allocate_bits_via_cached_ratios(scores, pos, 2, 5, {2, 4, 16}) is None     # layer without a record
    # the one-sort form taken when the caller vouches for the (batch, head, position) order: same levels
    assert torch.equal(p._allocate_bits_via_cached_ratios(scores, pos, 2, 3, {2, 4, 16}, batch_size=1), out)
    B, H, n = 3, 2, 37
    g = torch.Generator().manual_seed(5)
    scores = torch.rand(B * H * n, generator=g)
    scores[7] = scores[9]                                  # a tie keeps index order in both forms
    pos = torch.stack([torch.arange(B).repeat_interleave(H * n), torch.arange(H).repeat_interleave(n).repeat(B),
                       torch.arange(n).repeat(B * H)], dim=-1)
    for allowed in ({0, 2, 4, 16}, {2, 4}):
        loop = p._allocate_bits_via_cached_ratios(scores, pos, H, 3, allowed)
        assert torch.equal(p._allocate_bits_via_cached_ratios(scores, pos, H, 3, allowed, batch_size=B), loop)


def test_rank_table_follows_the_shares_of_the_latest_prefill():
    """A press object that is used for a second prompt must flush with the second prompt's level shares:
    the expanded rank table is cached, and the cache has to notice that the shares changed."""
    from kvquant import TurboQuantPerTokenBackendPress
    p = TurboQuantPerTokenBackendPress(scorer=_scorer(), bit_levels=(0, 2, 4, 16), key_quantizer="mse",
                                       value_quantizer="mse", target_avg_bits=2.0, sink_tokens=4, buffer_size=8)
    p._decode_bit_levels = {2, 4, 16}
    T = 4 + 40 + 8

    def prompt(n2):
        bits = torch.full((1, 1, T), 16, dtype=torch.int32)
        bits[0, 0, 4:44] = torch.tensor([2] * n2 + [4] * (40 - n2))
        p._record_observed_ratios(0, bits)

    prompt(30)
    table, counts = p._by_rank_table(0, 1, 16, "cpu")
    assert table[0].tolist() == [2] * 12 + [4] * 4 and counts[0].tolist() == [0, 12, 0, 4, 0, 0]
    assert p._by_rank_table(0, 1, 16, "cpu")[0] is table            # same shares: the cached table
    prompt(10)                                                      # the next prompt: 25 % / 75 %
    table2, counts2 = p._by_rank_table(0, 1, 16, "cpu")
    assert table2[0].tolist() == [2] * 4 + [4] * 12 and counts2[0].tolist() == [0, 4, 0, 12, 0, 0]
    p._decode_bit_levels = {4, 16}                                  # and another set of allowed levels
    assert p._by_rank_table(0, 1, 16, "cpu")[0][0].tolist() == [4] * 16


def test_backend_press_rejects_unbuilt_quantisers():
    from kvquant import TurboQuantBackendPress
    with pytest.raises(NotImplementedError):
        TurboQuantBackendPress()                       # min-max values by default
    TurboQuantBackendPress(key_quantizer="mse", value_quantizer="mse")


class _FakeStore:
    """What PackedCacheLayer needs of a packed store: a length, dense rows on request, truncation."""
    def __init__(self, keys, values):
        self.k, self.v = keys.clone(), values.clone()

    @property
    def seq_len(self):
        return self.k.shape[2]

    def append(self, k, v):
        self.k, self.v = torch.cat([self.k, k], 2), torch.cat([self.v, v], 2)

    def materialize(self):
        return self.k, self.v

    def truncate(self, n):
        self.k, self.v = self.k[:, :, :n], self.v[:, :, :n]


def test_packed_cache_layer_aliases_the_newest_token():
    from kvquant.hf_cache import PackedCacheLayer, is_aliased
    g = torch.Generator().manual_seed(0)
    k0, v0 = torch.randn(2, 3, 10, 8, generator=g), torch.randn(2, 3, 10, 8, generator=g)
    store = _FakeStore(k0, v0)
    layer = PackedCacheLayer(store, k0, v0)
    assert layer.get_seq_length() == 10 and layer.get_mask_sizes(1) == (11, 0)
    assert is_aliased(layer.keys) and layer.keys.untyped_storage().nbytes() == 2 * 3 * 8 * 4
    # one token: shapes in step, every position aliases the new token, nothing is concatenated
    k1, v1 = torch.randn(2, 3, 1, 8, generator=g), torch.randn(2, 3, 1, 8, generator=g)
    keys, values = layer.update(k1, v1)
    assert keys.shape == (2, 3, 11, 8) and is_aliased(keys) and torch.equal(keys[:, :, -1:], k1)
    assert torch.equal(values[:, :, -1:], v1) and layer.recent[0] is k1
    store.append(k1, v1)                                   # what the attention path does with the token
    # several tokens: the new tokens alone, tagged with the number of tokens the store holds (the attention patch takes
    # the stored part from the fused kernel: nothing is dequantised), views afterwards
    k2, v2 = torch.randn(2, 3, 4, 8, generator=g), torch.randn(2, 3, 4, 8, generator=g)
    store.materialize = None                               # must not be called
    keys, values = layer.update(k2, v2)
    assert keys is k2 and values is v2 and keys._odmkv_store_len == 11 and values._odmkv_store_len == 11
    assert layer.get_seq_length() == 15 and is_aliased(layer.keys) and torch.equal(layer.recent[0], k2)
    store.append(k2, v2)
    # out of step: refused rather than answered from the wrong rows
    store.truncate(14)
    with pytest.raises(RuntimeError, match="in step"):
        layer.update(k2, v2)
    store.append(k2[:, :, -1:], v2[:, :, -1:])
    # crop, both spellings
    layer.crop(-2)
    assert layer.get_seq_length() == 13 and store.seq_len == 13
    layer.crop(12)
    assert layer.get_seq_length() == 12 and store.seq_len == 12
    layer.crop(40)
    assert layer.get_seq_length() == 12
    with pytest.raises(NotImplementedError):
        layer.reorder_cache(torch.tensor([0, 1]))
    with pytest.raises(ValueError, match="holds"):
        PackedCacheLayer(store, k0, v0)


def test_release_dense_cache_needs_decode_quant():
    from kvquant import TurboQuantPerTokenBackendPress
    with pytest.raises(ValueError, match="release_dense_cache"):
        TurboQuantPerTokenBackendPress(scorer=_scorer(), bit_levels=(0, 2, 4, 16), key_quantizer="mse",
                                       value_quantizer="mse", target_avg_bits=2.0, decode_quant=False,
                                       release_dense_cache=True)


class _CountingScorer:
    """Scores a prompt in one call, on any device: every score is the scorer's own number."""
    def __init__(self, number):
        self.number, self.calls = number, 0

    def score_prefill(self, keys, values, layer_idx, *, module=None, hidden_states=None):
        raise AssertionError("the one-call form covers this prompt")

    def score_decode(self, key, value, layer_idx, *, module=None, hidden_states=None):
        return torch.ones(key.shape[0])

    def score_prompt(self, keys, values, layer_idx, *, module, hidden_states, out=None, rope_tables=None):
        self.calls += 1
        return torch.full(keys.shape[:3], self.number)


def test_a_scorer_assigned_after_construction_scores_the_next_prompt():
    from kvquant import TurboQuantPerTokenPress
    first, second = _CountingScorer(1.0), _CountingScorer(2.0)
    press = TurboQuantPerTokenPress(scorer=first, bit_levels=(0, 2, 4, 16), value_quantizer="mse", layerwise=True, target_avg_bits=2.0)
    press._finalize_prefill = lambda cache: None
    keys = torch.zeros(2, 3, 10, 128)
    press._prefill_hook(torch.nn.Module(), None, torch.zeros(2, 10, 64), 0, keys, keys)
    press.scorer = second
    press._prefill_hook(torch.nn.Module(), None, torch.zeros(2, 10, 64), 1, keys, keys)
    assert (first.calls, second.calls) == (1, 1)
    assert (press._prefill_scores[0] == 1.0).all() and (press._prefill_scores[1] == 2.0).all()


def test_an_overridden_allocation_finds_the_sink_masks():
    from kvquant import TurboQuantPerTokenPress
    seen = {}

    class Own(TurboQuantPerTokenPress):
        def _allocate_bits_for_prefill(self):
            seen.update(self._prefill_sink_masks)
            return {}

    press = Own(scorer=_CountingScorer(1.0), bit_levels=(0, 2, 4, 16), value_quantizer="mse", layerwise=True, target_avg_bits=2.0, sink_tokens=4)
    keys = torch.zeros(1, 3, 10, 128)
    press._prefill_hook(torch.nn.Module(), None, torch.zeros(1, 10, 64), 0, keys, keys)
    assert torch.equal(seen[0], torch.arange(10).expand(3, 10) < 4)


def test_the_uniform_press_refuses_cpu_tensors(monkeypatch):
    from types import SimpleNamespace
    from kvquant import TurboQuantBackendPress, backend_press

    def launched(*args):
        raise AssertionError("addresses of host memory handed to a kernel")

    monkeypatch.setattr(backend_press, "_lib", SimpleNamespace(
        lib=SimpleNamespace(odmkv_round_trip_workspace_bytes=lambda n: 1, odmkv_round_trip_rows=launched),
        workspace=lambda *a: torch.empty(1), stream_ptr=lambda d: 0, check=lambda rc: None, dtype_code=lambda t: 0))
    press = TurboQuantBackendPress(key_bits=3, value_bits=2, value_quantizer="mse")
    k, v = torch.zeros(1, 2, 20, 128, dtype=torch.float16), torch.zeros(1, 2, 20, 128, dtype=torch.float16)
    with pytest.raises(RuntimeError, match="must live on the GPU"):
        press._quantise_span(0, k, v, 0, 10)


@pytest.mark.parametrize("decode_quant,fp16_layers,counted", [(True, 0, True), (False, 0, False), (True, 1, False)])
def test_the_short_way_through_the_hook_counts_what_the_long_way_counts(decode_quant, fp16_layers, counted):
    from types import SimpleNamespace
    from kvquant import TurboQuantPerTokenBackendPress
    press = TurboQuantPerTokenBackendPress(scorer=_scorer(), bit_levels=(0, 2, 4, 16), key_quantizer="mse", value_quantizer="mse",
                                           target_avg_bits=2.0, initial_layers_fp16=fp16_layers)
    press.decode_quant = decode_quant
    for fast in (object(), None):                             # a store with the native step armed, and one without
        state = SimpleNamespace(_fast=fast, exact_decode_append=True, seq_len=41)
        press._states, press._buffer_counts, press._buffer_start_seqs = {0: state}, {}, {0: 40}
        module = torch.nn.Module()
        module.layer_idx, module._odmkv_state = 0, state
        keys = torch.zeros(1, 2, 41, 8)
        cache = SimpleNamespace(layers=[SimpleNamespace(keys=keys, values=keys, _tq_backend_state=state)])
        press._forward_hook(module, (), {"past_key_values": cache, "hidden_states": torch.zeros(1, 1, 16)}, None)
        assert press._buffer_counts.get(0, 0) == int(counted)


def test_a_prefill_that_fails_waits_for_the_counts_it_asked_for(monkeypatch):
    from types import SimpleNamespace
    from kvquant import TurboQuantPerTokenBackendPress, _lib, adaptive_backend_press as abp
    calls = []
    monkeypatch.setattr(abp, "_lib", SimpleNamespace(
        lib=SimpleNamespace(odmkv_finish_levels_chunks=lambda n: 1, odmkv_finish_levels=lambda *a: calls.append("launched") or 0),
        check=_lib.check, stream_ptr=lambda d: 0, LEVEL_ORDER=_lib.LEVEL_ORDER))

    class Event:
        def record(self, stream): calls.append("recorded")
        def synchronize(self): calls.append("waited")

    empty = torch.empty
    monkeypatch.setattr(abp.torch, "empty", lambda *a, pin_memory=False, **kw: empty(*a, **kw))
    monkeypatch.setattr(abp.torch.cuda, "Event", Event)
    monkeypatch.setattr(abp.torch.cuda, "current_stream", lambda d=None: None)
    monkeypatch.setattr(abp.torch.cuda, "device", lambda d: __import__("contextlib").nullcontext())
    press = TurboQuantPerTokenBackendPress(scorer=_scorer(), bit_levels=(0, 2, 4, 16), key_quantizer="mse", value_quantizer="mse",
                                           target_avg_bits=2.0, layerwise=True)
    press._allocate_bits_for_prefill = lambda: {0: torch.full((1, 2, 200), 2, dtype=torch.int32)}
    keys = torch.zeros(1, 2, 200, 128)
    cache = SimpleNamespace(layers=[SimpleNamespace(keys=keys, values=keys)])
    with pytest.raises(RuntimeError, match="no CPU path"):        # the store lives on the GPU
        press._finalize_prefill(cache)
    assert calls == ["launched", "recorded", "waited"]


def test_aliases_of_what_is_no_cache_layer_are_refused():
    from kvquant import _lib
    k = torch.arange(24.0).reshape(1, 2, 3, 4)
    a, b = _lib._native.alias(k, k + 1, 7)
    assert a.shape == b.shape == (1, 2, 7, 4) and torch.equal(a, k[:, :, -1:].expand(1, 2, 7, 4)) and torch.equal(b, a + 1)
    for bad in (k[0], k[:, :, :0], torch.zeros(3)):
        with pytest.raises(ValueError, match="alias"):
            _lib._native.alias(k, bad, 7)
    with pytest.raises(RuntimeError):
        _lib._native.alias(k, k, -1)


@pytest.mark.parametrize("inference", [False, True])
@pytest.mark.parametrize("additive", [False, True])
def test_a_mask_written_to_between_forwards_is_looked_at_again(inference, additive, monkeypatch):
    from kvquant import attention_patch as ap
    looks = []
    monkeypatch.setattr(ap, "bool", lambda x: looks.append(1) or x.item(), raising=False)
    with torch.inference_mode(inference):
        mask = torch.zeros(1, 1, 3, 13) if additive else torch.ones(1, 1, 3, 13, dtype=torch.bool)
        assert [ap._store_part_is_open(mask, 10, layer) for layer in (0, 1, 5)] == [True] * 3
        assert len(looks) == 1                                # the layers of one forward share the look
        mask[0, 0, 1, 4] = float("-inf") if additive else False
        assert [ap._store_part_is_open(mask, 10, layer) for layer in (0, 1, 5)] == [False] * 3      # the question after a rewind
        assert len(looks) == 2 and ap._store_part_is_open(mask, 4, 6) and len(looks) == 3
        assert ap._store_part_is_open(mask, 4) and ap._store_part_is_open(mask, 4) and len(looks) == 5   # (no layer index)
    if not inference:
        assert ap._store_part_is_open(mask, 4, 7) and len(looks) == 6
        mask[0, 0, 1, 2] = float("-inf") if additive else False
        assert not ap._store_part_is_open(mask, 4, 8)


def test_rows_that_share_memory_do_not_take_the_one_pass_kernel():
    """The kernel rewrites a row while others are still to be read.  Layouts of caches pass; expanded tensors, overlapping windows of one
    sequence, and keys that are the values or begin inside them do not.  Against a count of every element's address."""
    from kvquant.backend_press import _rows_apart
    base = torch.zeros(1 << 16, dtype=torch.float16)

    def view(at, B, H, n, strides):
        return base.as_strided((B, H, n, 8), (*strides, 1), at)

    def apart(k, v):
        index = torch.arange(base.numel())
        return torch.cat([index.as_strided(t.shape, t.stride(), t.storage_offset()).flatten() for t in (k, v)]).bincount().max() == 1

    some = []
    for B, H, n, strides in [(1, 4, 6, (192, 48, 8)), (2, 4, 6, (192, 48, 8)), (1, 4, 6, (192, 8, 32)), (2, 3, 6, (480, 160, 16)), (1, 4, 6, (384, 16, 64)),
                             (1, 4, 6, (0, 0, 8)), (1, 4, 6, (32, 8, 8)), (1, 4, 6, (96, 24, 8)), (1, 1, 6, (8, 8, 8)), (2, 1, 6, (24, 24, 8)), (1, 1, 1, (8, 8, 8))]:
        k = view(0, B, H, n, strides)
        for off in (0, 4, 8, 16, 32, 184, 192, 4096):
            v = view(off, B, H, n, strides)
            for a, b in ((k, v), (v, k)):
                assert apart(a, b) or not _rows_apart(a, b), (strides, off)
            some.append((_rows_apart(k, v), bool(apart(k, v)), strides, off))
    assert (True, True, (192, 48, 8), 4096) in some and (True, True, (192, 8, 32), 192) in some       # one behind the other
    assert (True, True, (384, 16, 64), 8) in some                                                     # keys and values of a token side by side
    assert not any(fast for fast, _, strides, _ in some if strides in ((0, 0, 8), (32, 8, 8), (96, 24, 8)))
