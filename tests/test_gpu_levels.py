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
