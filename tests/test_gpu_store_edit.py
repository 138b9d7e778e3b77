"""GPU: a store edited in place (blocks of exact tokens, truncation) against one filled at once, and a question's own part of
its attention (odmkv_block_merge) against torch, at the edges of tiles and of the kernel's 64-key rounds."""
import pytest
import torch

pytestmark = pytest.mark.gpu
LEVELS = (0, 2, 3, 4, 8, 16)


def _store(k, v, bits):
    from kvquant.tq_adaptive_backend import TurboQuantAdaptiveKVCacheState
    st = TurboQuantAdaptiveKVCacheState(128, LEVELS, device="cuda", dtype=k.dtype, key_quantizer="mse", value_quantizer="mse")
    st.prefill(k, v, bits)
    return st


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("T,blocks,cut", [(1, (63, 1, 2), 64), (130, (29, 300), 131), (400, (1, 64, 5), 399), (257, (500,), 3)])
def test_blocks_of_exact_tokens_and_truncation(T, blocks, cut, dtype):
    g = torch.Generator().manual_seed(T)
    total = T + sum(blocks)
    k, v = (torch.randn(2, 3, total, 128, generator=g).to(dtype).cuda() for _ in range(2))
    bits = torch.tensor(LEVELS)[torch.randint(0, 6, (2, 3, total), generator=g)].to(torch.int32)
    bits[:, :, T:] = 16
    st = _store(k[:, :, :T], v[:, :, :T], bits[:, :, :T].cuda())
    at = T
    for n in blocks:
        st.append_all_exact(k[:, :, at:at + n], v[:, :, at:at + n])
        at += n
    whole = _store(k, v, bits.cuda())
    q = torch.randn(2, 6, 128, generator=g).to(dtype).cuda()

    def same(a, b):
        assert a.seq_len == b.seq_len and a.level_counts() == b.level_counts()
        assert all(torch.equal(x, y) for x, y in zip(a.materialize(), b.materialize()))
        assert (a.decode_attention(q) - b.decode_attention(q)).abs().max() < 2e-4      # (work lists may be cut differently)
    same(st, whole)
    st.truncate(cut)
    same(st, _store(k[:, :, :cut], v[:, :, :cut], bits[:, :, :cut].cuda()))
    st.append_all_exact(k[:, :, cut:cut + 1], v[:, :, cut:cut + 1])                    # and it goes on from there
    assert st.seq_len == cut + 1 and torch.equal(st.materialize()[0][:, :, -1], k[:, :, cut])


@pytest.mark.parametrize("qt,kt", [(torch.float16, torch.float16), (torch.bfloat16, torch.bfloat16), (torch.float32, torch.float16)])
@pytest.mark.parametrize("L,G,masked", [(1, 1, False), (29, 4, True), (64, 7, False), (65, 8, True), (256, 3, False)])
def test_a_blocks_own_tokens_merged_with_the_stores_part(L, G, masked, qt, kt):
    from kvquant import _lib
    g = torch.Generator(device="cuda").manual_seed(L)
    B, H, D = 2, 2, 128
    q = torch.randn(B, L, H * G, D, generator=g, device="cuda").to(qt).transpose(1, 2)
    k, v = (torch.randn(B, H, L + 3, D, generator=g, device="cuda").to(kt)[:, :, 3:] for _ in range(2))
    out_s, lse_s = torch.randn(B, H * G, L, D, generator=g, device="cuda"), torch.randn(B, H * G, L, generator=g, device="cuda")
    lse_s[0, 0, 0] = float("-inf")                             # a store without a visible token
    mask = torch.ones(B, 1, L, L + 5, dtype=torch.bool, device="cuda").tril(5)
    if masked:
        mask[1, 0, L // 2:, 5] = False
    tail = mask[..., 5:] if masked else None
    out = torch.empty(B, L, H * G, D, dtype=qt, device="cuda")
    _lib.check(_lib.lib.odmkv_block_merge(
        q.data_ptr(), _lib.dtype_code(q), *q.stride()[:3], k.data_ptr(), *k.stride()[:3], v.data_ptr(), *v.stride()[:3],
        _lib.dtype_code(k), _lib.ptr(tail), 0 if tail is None else tail.stride(0), 0 if tail is None else tail.stride(2),
        B, H * G, H, L, 0.07, out_s.data_ptr(), lse_s.data_ptr(), out.data_ptr(), _lib.stream_ptr(q.device)))
    kr, vr = k.double().repeat_interleave(G, 1).cpu(), v.double().repeat_interleave(G, 1).cpu()
    logits = (q.double().cpu() @ kr.transpose(-1, -2).contiguous()) * 0.07
    logits = logits.masked_fill(~mask[..., 5:].cpu(), float("-inf"))
    both = torch.cat([lse_s.double().cpu().unsqueeze(-1), logits], -1).softmax(-1)
    want = (both[..., :1] * out_s.double().cpu() + both[..., 1:] @ vr).transpose(1, 2)
    tol = {torch.float32: 2e-5, torch.float16: 1e-3, torch.bfloat16: 8e-3}[qt]
    assert ((out.double().cpu() - want).norm(dim=-1) <= tol * (want.norm(dim=-1) + 1e-3)).all()


@pytest.mark.parametrize("B,H,G", [(1, 2, 4), (2, 1, 7), (64, 2, 4)])             # (the last: the merge by groups of heads)
def test_a_step_into_full_exact_segments_leaves_their_counts(B, H, G):
    import ctypes as C
    from kvquant import _lib
    from kvquant.tq_adaptive_backend import TurboQuantAdaptiveKVCacheState
    g = torch.Generator(device="cuda").manual_seed(B)
    k, v = (torch.randn(B, H, 128, 128, generator=g, device="cuda").half() for _ in range(2))
    bits = torch.full((B, H, 128), 16, dtype=torch.int32, device="cuda")
    bits[:, :, 64:] = 3                                        # 64 exact tokens a pair: one tile, and no room beside them
    st = TurboQuantAdaptiveKVCacheState(128, LEVELS, device="cuda", dtype=k.dtype, key_quantizer="mse", value_quantizer="mse", exact_slack=0)
    st.prefill(k, v, bits)
    q = torch.randn(B, H * G, 128, generator=g, device="cuda").half()
    want = st.decode_attention(q)
    ws = torch.empty(_lib.lib.odmkv_decode_workspace_bytes(B, H * G, st._items[2]), dtype=torch.uint8, device="cuda")
    step = _lib.Step(C.pointer(st._packed), C.pointer(st._worklist), st._pi_k_ops.data_ptr(), st.pi_v.data_ptr(), st._decode_cb.data_ptr(),
                     st._decode_cb_host, st._decode_inv, ws.data_ptr(), ws.numel(), B, H * G, _lib.F16, _lib.F32, 128 ** -0.5)
    token = torch.full((B, H, 128), 9.0, dtype=torch.float16, device="cuda")
    out = torch.empty_like(want)
    for _ in range(2):
        _lib.check(_lib.lib.odmkv_decode_step(C.byref(step), q.data_ptr(), token.data_ptr(), token.data_ptr(), token.stride(0), token.stride(1),
                                              128, out.data_ptr(), None, _lib.stream_ptr(out.device)))
        assert torch.equal(out, want) and (st._bufs["seg_count"][4] == 64).all()
    assert torch.equal(st.materialize()[0][:, :, :64], k[:, :, :64])


@pytest.mark.parametrize("B,Hq,H,L", [(1, 8, 8, 627), (1, 8, 8, 628), (3, 28, 4, 193), (3, 28, 4, 194), (2, 4, 2, 2)])
def test_blocks_on_either_side_of_the_native_limit(B, Hq, H, L):
    # 3 << 20 pairs: 627 tokens of 8 heads, 193 tokens of 3 x 28
    from types import SimpleNamespace
    from kvquant import attention_patch as ap
    g = torch.Generator(device="cuda").manual_seed(L)
    q = torch.randn(B, L, Hq, 128, generator=g, device="cuda").half().transpose(1, 2)
    k, v = (torch.randn(B, L, H, 128, generator=g, device="cuda").half().transpose(1, 2) for _ in range(2))
    out_s, lse_s = torch.randn(B, Hq, L, 128, generator=g, device="cuda"), torch.randn(B, Hq, L, generator=g, device="cuda")
    state = SimpleNamespace(seq_len=50, decode_attention_block=lambda query, scaling: (out_s, lse_s))
    with torch.inference_mode():
        got = ap._fused_block(state, q, k, v, None, 0.08, 50 + L)
        logits = (q.float() @ k.float().repeat_interleave(Hq // H, 1).transpose(-1, -2).contiguous()) * 0.08
        keep = torch.ones(L, L, dtype=torch.bool, device="cuda").tril()
        both = torch.cat([lse_s.unsqueeze(-1), logits.masked_fill(~keep, float("-inf"))], -1).softmax(-1)
        want = both[..., :1] * out_s + both[..., 1:] @ v.float().repeat_interleave(Hq // H, 1)
    assert got.shape == (B, L, Hq, 128) and (got.float() - want.transpose(1, 2)).norm() <= 1e-3 * want.norm()
