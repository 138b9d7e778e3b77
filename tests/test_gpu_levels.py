"""GPU: a layer's levels between allocation and store (odmkv_finish_levels) and the list of evicted positions
(odmkv_evicted_indices), against torch, at the edges of their 4096-token chunks."""
import pytest
import torch

pytestmark = pytest.mark.gpu
LEVELS = torch.tensor((0, 2, 3, 4, 8, 16))


@pytest.mark.parametrize("B,H,T,tail", [(1, 1, 1, 0), (1, 3, 130, 128), (2, 2, 4095, 128), (1, 8, 4096, 0), (3, 1, 4097, 4097),
                                        (2, 4, 8193, 128)])
def test_levels_counted_overridden_and_written_down(B, H, T, tail):
    from kvquant import _lib
    g = torch.Generator().manual_seed(T)
    bits = LEVELS[torch.randint(0, 6, (B, H, T), generator=g)].to(torch.int32)
    dev = bits.cuda()
    room = (T + 300 + 3) & ~3
    levels = torch.full((B, H, room), 77, dtype=torch.uint8, device="cuda")
    counts = torch.full((B * H, _lib.lib.odmkv_finish_levels_chunks(room), 2, 6), -1, dtype=torch.int32, pin_memory=True)
    lo, hi = min(4, T - 1), max(T - tail, 1)
    _lib.check(_lib.lib.odmkv_finish_levels(dev.data_ptr(), B * H, T, lo, hi, T - tail, levels.data_ptr(), room, counts.data_ptr(),
                                            _lib.stream_ptr(dev.device)))
    torch.cuda.synchronize()
    bulk, stored = counts.sum(dim=1).swapaxes(0, 1)
    want = torch.stack([(bits[..., lo:hi] == b).sum(-1) for b in LEVELS.tolist()], dim=-1).reshape(B * H, 6)
    assert torch.equal(bulk.long(), want)
    if tail:
        bits[..., T - tail:] = 16
    assert torch.equal(dev.cpu(), bits)
    assert torch.equal(levels[..., :T].cpu().int(), bits) and (levels[..., T:] == 16).all()
    assert torch.equal(stored.long(), torch.stack([(bits == b).sum(-1) for b in LEVELS.tolist()], dim=-1).reshape(B * H, 6))
    want = (bits == 0).nonzero(as_tuple=True)
    n = want[0].numel()
    if n:
        out = torch.empty(3, n, dtype=torch.long, device="cuda")
        ws = torch.empty(_lib.lib.odmkv_evicted_workspace_bytes(B, H, T), dtype=torch.uint8, device="cuda")
        _lib.check(_lib.lib.odmkv_evicted_indices(levels.data_ptr(), B, H, T, room, n, out.data_ptr(), ws.data_ptr(), ws.numel(),
                                                  _lib.stream_ptr(dev.device)))
        assert all(torch.equal(a.cpu(), b) for a, b in zip(out, want))


@pytest.mark.parametrize("T,skip", [(4, 1), (4096, 2), (4097, 2), (8200, 3), (8200, 4)])
def test_levels_that_start_anywhere(T, skip):
    # (a group of layers inside one allocation: its first row starts where the layers before it end)
    from kvquant import _lib
    g = torch.Generator().manual_seed(T + skip)
    bits = LEVELS[torch.randint(0, 6, (3, T), generator=g)].to(torch.int32)
    dev = torch.zeros(skip + 3 * T, dtype=torch.int32, device="cuda")
    dev[skip:] = bits.reshape(-1).cuda()
    room = (T + 3) & ~3
    levels = torch.empty((3, room), dtype=torch.uint8, device="cuda")
    counts = torch.full((3, _lib.lib.odmkv_finish_levels_chunks(room), 2, 6), -1, dtype=torch.int32, pin_memory=True)
    _lib.check(_lib.lib.odmkv_finish_levels(dev.data_ptr() + 4 * skip, 3, T, 1, T, T - 3, levels.data_ptr(), room, counts.data_ptr(),
                                            _lib.stream_ptr(dev.device)))
    torch.cuda.synchronize()
    bulk = torch.stack([(bits[:, 1:] == b).sum(-1) for b in LEVELS.tolist()], dim=-1)
    bits[:, T - 3:] = 16
    assert torch.equal(dev[skip:].cpu(), bits.reshape(-1)) and (dev[:skip] == 0).all() and torch.equal(levels[:, :T].cpu().int(), bits)
    assert torch.equal(counts.sum(dim=1)[:, 0].long(), bulk)
    assert torch.equal(counts.sum(dim=1)[:, 1].long(), torch.stack([(bits == b).sum(-1) for b in LEVELS.tolist()], dim=-1))


def test_a_prompt_whose_first_layer_stays_in_fp16_has_groups_that_start_anywhere():
    # two kv-heads of 333 tokens: the second layer's levels start 8 bytes off a multiple of 16
    from types import SimpleNamespace
    from kvquant import RiskScorer, TurboQuantPerTokenBackendPress
    scorer = RiskScorer(n_future_positions=16, n_sink=4, epsilon=1e-2)
    scorer.normalize_grain = "global"
    press = TurboQuantPerTokenBackendPress(scorer=scorer, bit_levels=(0, 2, 3, 4, 8, 16), target_avg_bits=2.0, eviction_cost=0.5,
                                           key_quantizer="mse", value_quantizer="mse", sink_tokens=4, layerwise=True, buffer_size=128,
                                           initial_layers_fp16=1)
    g = torch.Generator(device="cuda").manual_seed(1)
    k, v = (torch.randn(1, 2, 333, 128, generator=g, device="cuda").half() for _ in range(2))
    cache = SimpleNamespace(layers=[SimpleNamespace(keys=k.clone(), values=v.clone()) for _ in range(2)])
    press._head_dim = 128
    press._prefill_scores = {i: torch.rand(1, 2, 333, generator=g, device="cuda") for i in range(2)}
    press._finalize_prefill(cache)
    assert press._states[0].level_counts()[16] == 2 * 333
    counts = press._states[1].level_counts()
    assert sum(counts.values()) == 2 * 333 and counts[16] < 2 * 333 and not press._states[1].masked_key_indices() is None


@pytest.mark.parametrize("rows,T", [(65532, 4), (65533, 3), (65536, 4), (131073, 1)])
def test_more_rows_than_a_launch_takes(rows, T):
    from kvquant import _lib
    g = torch.Generator().manual_seed(rows)
    bits = LEVELS[torch.randint(0, 6, (rows, T), generator=g)].to(torch.int32)
    dev = bits.cuda()
    levels = torch.empty((rows, 8), dtype=torch.uint8, device="cuda")
    counts = torch.full((rows, 1, 2, 6), -1, dtype=torch.int32, pin_memory=True)
    _lib.check(_lib.lib.odmkv_finish_levels(dev.data_ptr(), rows, T, 0, T, T - 1, levels.data_ptr(), 8, counts.data_ptr(),
                                            _lib.stream_ptr(dev.device)))
    torch.cuda.synchronize()
    assert torch.equal(counts[:, 0, 0].long(), torch.stack([(bits == b).sum(-1) for b in LEVELS.tolist()], dim=-1))
    bits[:, T - 1:] = 16
    assert torch.equal(dev.cpu(), bits) and torch.equal(levels[:, :T].cpu().int(), bits) and (levels[:, T:] == 16).all()
    assert torch.equal(counts[:, 0, 1].long(), torch.stack([(bits == b).sum(-1) for b in LEVELS.tolist()], dim=-1))


def test_levels_that_a_subclass_keeps_are_left_as_they_were():
    from types import SimpleNamespace
    from kvquant import RiskScorer, TurboQuantPerTokenBackendPress

    class Keeping(TurboQuantPerTokenBackendPress):
        def _allocate_bits_for_prefill(self):
            self.kept = super()._allocate_bits_for_prefill()
            self.copies = {i: b.clone() for i, b in self.kept.items()}
            return self.kept

    press = Keeping(scorer=RiskScorer(n_future_positions=16, n_sink=4, epsilon=1e-2), bit_levels=(0, 2, 3, 4, 8, 16), target_avg_bits=2.0,
                    eviction_cost=0.5, key_quantizer="mse", value_quantizer="mse", sink_tokens=4, layerwise=True, buffer_size=128)
    g = torch.Generator(device="cuda").manual_seed(2)
    k, v = (torch.randn(1, 2, 400, 128, generator=g, device="cuda").half() for _ in range(2))
    cache = SimpleNamespace(layers=[SimpleNamespace(keys=k.clone(), values=v.clone()) for _ in range(2)])
    press._head_dim = 128
    press._prefill_scores = {i: torch.rand(1, 2, 400, generator=g, device="cuda") for i in range(2)}
    press._finalize_prefill(cache)
    assert all(torch.equal(press.kept[i], press.copies[i]) for i in range(2)) and (press.kept[0][..., -128:] != 16).any()
    assert press._states[0].level_counts()[16] >= 2 * 128


@pytest.mark.parametrize("buffer_size", [-200, 0])
def test_a_prompt_without_a_decode_buffer(buffer_size):
    from types import SimpleNamespace
    from kvquant import RiskScorer, TurboQuantPerTokenBackendPress
    press = TurboQuantPerTokenBackendPress(scorer=RiskScorer(n_future_positions=16, n_sink=4, epsilon=1e-2), bit_levels=(0, 2, 3, 4, 8, 16),
                                           target_avg_bits=2.0, key_quantizer="mse", value_quantizer="mse", sink_tokens=4, layerwise=True,
                                           buffer_size=buffer_size)
    g = torch.Generator(device="cuda").manual_seed(2)
    k, v = (torch.randn(1, 2, 300, 128, generator=g, device="cuda").half() for _ in range(2))
    press._head_dim = 128
    press._prefill_scores = {0: torch.rand(1, 2, 300, generator=g, device="cuda")}
    press._finalize_prefill(SimpleNamespace(layers=[SimpleNamespace(keys=k, values=v)]))
    assert sum(press._states[0].level_counts().values()) == 600
