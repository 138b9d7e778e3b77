"""GPU: rows outside the store.  The matrix-core quantiser gives the exact quantiser's codes (the same numbers as fp32 rows take
the exact kernel), in bytes and in the container; the in-place round trip gives dequantize(quantize(x))."""
import pytest
import torch

pytestmark = pytest.mark.gpu


def _rows(n, dtype, seed):
    x = torch.randn(n, 128, generator=torch.Generator().manual_seed(seed))
    if n > 40:
        x[3], x[4], x[5, 7], x[6, 9] = 0.0, 1e-6, float("inf"), float("nan")
        x[7] *= 3e3
        x[8, 1:] = 0.0
    return x.to(dtype).cuda()


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("bits", [2, 3, 4, 8])
@pytest.mark.parametrize("n", [1, 63, 64, 65, 700, 33000])
def test_codes_of_16_bit_rows(n, bits, dtype):
    from kvquant.tq_backend import TurboQuantMSE, _pack_indices
    x = _rows(n, dtype, 10 * n + bits)
    q = TurboQuantMSE(128, bits, device="cuda", dtype=dtype, seed=7)
    codes, norms = q.quantize_codes(x)
    exact, exact_norms = q.quantize_codes(x.float())
    assert torch.equal(codes, exact) and torch.equal(norms.view(torch.int32), exact_norms.view(torch.int32))
    mq = q.quantize(x)
    assert torch.equal(mq.indices, _pack_indices(exact, bits)) and torch.equal(mq.norms.view(torch.int32), norms.view(torch.int32))
    strided = torch.zeros(n, 256, dtype=dtype, device="cuda")
    strided[:, 128:] = x
    assert torch.equal(q.quantize_codes(strided[:, 128:])[0], exact)


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("bits", [2, 3, 4])
@pytest.mark.parametrize("move", [2e-7, 1.6e-6, 3e-6, 3e-3, -0.1])
def test_codes_of_16_bit_rows_by_tables_that_do_not_mirror(move, bits, dtype):
    """Either side of the 1e-6 by which a threshold (it moves by half as much as a centroid) may be off its mirror image, and far."""
    from kvquant.tq_backend import TurboQuantMSE, _pack_indices
    x = _rows(33000, dtype, bits)
    q = TurboQuantMSE(128, bits, device="cuda", dtype=dtype, seed=7)
    q.centroids = q.centroids.clone()
    q.centroids[0 if move < 0 else -1] += move
    codes, _ = q.quantize_codes(x)
    exact, _ = q.quantize_codes(x.float())
    assert torch.equal(codes, exact) and torch.equal(q.quantize(x).indices, _pack_indices(exact, bits))


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("B,H,T,lo,hi,bits", [(1, 1, 1, 0, 1, (3, 2)), (2, 3, 90, 17, 81, (2, 4)), (1, 8, 1300, 0, 1172, (3, 2)), (2, 2, 70, 0, 70, (8, 3))])
def test_round_trip_in_place(B, H, T, lo, hi, bits, dtype):
    from kvquant import TurboQuantBackendPress
    g = torch.Generator().manual_seed(T)
    k, v = (torch.randn(B, H, T, 128, generator=g).to(dtype).cuda() for _ in range(2))
    press = TurboQuantBackendPress(key_bits=bits[0], value_bits=bits[1], value_quantizer="mse")
    want = []
    for x, b, seed in ((k, bits[0], 42), (v, bits[1], 2042)):
        q = press._q(b, seed, x)
        y = x.clone()
        y[:, :, lo:hi] = q.dequantize(q.quantize(x[:, :, lo:hi].reshape(-1, 128))).reshape(B, H, hi - lo, 128).to(dtype)
        want.append(y)
    got_k, got_v = k.clone(), v.clone()
    press._quantise_span(0, got_k, got_v, lo, hi)
    # one step of the type: the sums are formed from fp16 pairs on the matrix cores here, in fp32 there (about 1e-7 of the row's norm
    # either way, so that elements next to a rounding boundary may fall on the other side)
    step = 2 ** -10 if dtype == torch.float16 else 2 ** -7
    for got, y in zip((got_k, got_v), want):
        assert torch.equal(got[:, :, :lo], y[:, :, :lo]) and torch.equal(got[:, :, hi:], y[:, :, hi:])
        assert ((got.float() - y.float()).abs() <= step * y.float().abs() + 1e-5).all()


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("bits", [2, 3, 4])
@pytest.mark.parametrize("n,shift", [(1, 0.0), (64, 0.0), (65, 0.0), (40000, 0.0), (130, 3e-3)])
def test_round_trip_takes_the_quantiser_s_codes(n, shift, bits, dtype):
    """In one pass over the rows, every code is the one that the quantiser gives: ordinary rows, rows of zeros, one element, tiny and large ones, tiles with
    more values next to a threshold than the list holds, and infinities; tables that mirror and one that does not; whole tiles, one row and one
    row more, several tiles a wavefront."""
    from kvquant import TurboQuantBackendPress
    x = _rows(n, dtype, bits)
    press = TurboQuantBackendPress(key_bits=bits, value_bits=bits, value_quantizer="mse")
    kq, vq = press._q(bits, 42, x), press._q(bits, 2042, x)
    kq.centroids = kq.centroids.clone()
    kq.centroids[0] -= shift
    if n >= 130:                                                 # (the first tile holds rows without a norm already)
        mid = float((kq.centroids[0] + kq.centroids[1]) / 2)     # on the first threshold after the rotation: 128 listed values a row
        x[70:78] = (torch.full((8, 128), mid, device="cuda") @ kq.pi).to(dtype)
        x[79] = 0.0
    k, v = x.view(1, 1, n, 128).clone(), x.view(1, 1, n, 128).clone()
    press._quantise_span(0, k, v, 0, n)
    step = 2 ** -10 if dtype == torch.float16 else 2 ** -7
    for got, q in ((k, kq), (v, vq)):
        codes, norms = q.quantize_codes(x.float())
        want = (q.centroids.double()[codes.long()] @ q.pi.double()) * norms.double()[:, None]
        finite = torch.isfinite(want).all(dim=-1)
        assert finite.sum() >= n - 2 and not torch.isfinite(got.view(n, 128)[~finite]).any()
        # a code more or less moves the row by a centroid's distance, some tenths of a percent of its norm at the least
        scale = norms.double()[finite, None].abs()
        assert ((got.view(n, 128)[finite].double() - want[finite]).abs() <= step * want[finite].abs() + 1e-6 * scale + 1e-7).all()


@pytest.mark.parametrize("kind", [torch.uint8, torch.int16, torch.int32, torch.int64])
@pytest.mark.parametrize("bits,pad", [(2, 0), (3, 0), (4, 5), (8, 0), (2, 3)])
def test_indices_in_wider_types_and_padded_rows(bits, pad, kind):
    from kvquant.tq_backend import MSEQuantized, TurboQuantMSE, _unpack_indices
    x = _rows(70, torch.float16, bits)
    x[5, 7], x[6, 9] = 1.0, 2.0
    q = TurboQuantMSE(128, bits, device="cuda", dtype=x.dtype, seed=7)
    got = q.quantize(x.view(2, 35, 128))
    want = q.dequantize(got)
    indices = torch.cat([got.indices.to(kind), torch.full((2, 35, pad), 85, dtype=kind, device="cuda")], dim=-1)
    assert torch.equal(_unpack_indices(indices, bits, 128), _unpack_indices(got.indices, bits, 128))
    assert torch.equal(q.dequantize(MSEQuantized(indices, got.norms, bits)), want)
    with pytest.raises(ValueError):
        q.dequantize(MSEQuantized(got.indices[..., :-1], got.norms, bits))


def test_rows_that_are_shared_or_recorded_are_refused_as_by_torch():
    from kvquant import TurboQuantBackendPress
    press = TurboQuantBackendPress(key_bits=3, value_bits=2, value_quantizer="mse")
    make = lambda heads=2, **kw: torch.randn(1, heads, 40, 128, device="cuda", dtype=torch.float16, **kw)
    for k, v in ((make(1).expand(1, 2, 40, 128), make(1).expand(1, 2, 40, 128)),              # one row for two heads
                 (make(requires_grad=True), make()), (make(), make(requires_grad=True))):     # leaves of a graph
        before = k.detach().clone()
        with pytest.raises(RuntimeError):
            press._quantise_span(0, k, v, 0, 30)
            torch.cuda.synchronize()
        assert not k.requires_grad or torch.equal(k.detach(), before)
    # and what a gradient is recorded for is recorded: the quantised rows pass none on
    k, leaf = make(), make(requires_grad=True)
    values = leaf * 1.0
    press._quantise_span(0, k, values, 0, 30)
    values.float().sum().backward()
    assert (leaf.grad[:, :, :30] == 0).all() and (leaf.grad[:, :, 30:] == 1).all()
    # [B, T, H, D] in memory, as a projection leaves it
    k = torch.randn(1, 40, 2, 128, device="cuda", dtype=torch.float16).transpose(1, 2)
    a, b = k.contiguous(), k.contiguous()
    press._quantise_span(0, a, b, 0, 30)
    v = k.contiguous().transpose(1, 2).contiguous().transpose(1, 2)
    press._quantise_span(0, k, v, 0, 30)
    assert torch.equal(k, a) and torch.equal(v, b)


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("bits", [(3, 2), (4, 3), (8, 8)])
@pytest.mark.parametrize("heavy", [False, True])
def test_the_round_trip_is_no_further_from_fp64_than_fp32_sums(bits, heavy, dtype):
    # elements that are not the nearest value of the type to the fp64 result: of the in-place kernels, and of fp32 sums rounded once
    # (of 4.2 million elements 600 to 11000; the bound leaves six standard deviations of such a count at the least)
    from kvquant import TurboQuantBackendPress
    g = torch.Generator(device="cuda").manual_seed(bits[0])
    k, v = (torch.randn(1, 4, 4096, 128, generator=g, device="cuda") for _ in range(2))
    if heavy:
        k[..., [11, 37, 64, 101]] *= 20.0
    k, v = k.to(dtype), v.to(dtype)
    press = TurboQuantBackendPress(key_bits=bits[0], value_bits=bits[1], value_quantizer="mse")
    wrong, wrong32 = 0, 0
    got_k, got_v = k.clone(), v.clone()
    press._quantise_span(0, got_k, got_v, 0, 4096)
    for x, got, b, seed in ((k, got_k, bits[0], 42), (v, got_v, bits[1], 2042)):
        q = press._q(b, seed, x)
        codes, norms = q.quantize_codes(x.view(-1, 128))
        exact = ((q.centroids.double()[codes.long()] @ q.pi.double()) * norms.double()[:, None]).float().to(dtype)
        wrong += int((got.view(-1, 128) != exact).sum())
        wrong32 += int((q.dequantize(q.quantize(x.view(-1, 128))).to(dtype) != exact).sum())
    assert wrong <= 1.25 * wrong32


@pytest.mark.parametrize("bits", [2, 3, 4])
def test_codes_of_fp16_rows_below_the_normal_numbers(bits):
    """Rows of a few units of 2^-24 an element up to norms of 1e-3, outside a store and in the round trip: the definition's codes."""
    from kvquant import TurboQuantBackendPress
    n, g = 16384, torch.Generator().manual_seed(bits)
    x = torch.randn(n, 128, generator=g) * torch.logspace(-24, -14, n, base=2.0)[torch.randperm(n, generator=g)][:, None]
    x[::5, 8:] = 0.0
    x = x.half().cuda()
    press = TurboQuantBackendPress(key_bits=bits, value_bits=bits, value_quantizer="mse")
    kq, vq = press._q(bits, 42, x), press._q(bits, 2042, x)
    assert torch.equal(kq.quantize_codes(x)[0], kq.quantize_codes(x.float())[0])
    k, v = x.view(1, 1, n, 128).clone(), x.view(1, 1, n, 128).clone()
    press._quantise_span(0, k, v, 0, n)
    for got, q in ((k, kq), (v, vq)):
        codes, norms = q.quantize_codes(x.float())
        want = (q.centroids.double()[codes.long()] @ q.pi.double()) * norms.double()[:, None]
        # half a unit of fp16's smallest numbers, or a step; another code moves the row by some tenths of a percent of its norm at the least
        err = (got.view(n, 128).double() - want).abs()
        assert (err <= 2.0 ** -25 + 2.0 ** -10 * want.abs() + 1e-6 * norms.double()[:, None]).all()


@pytest.mark.parametrize("bits", [(2, 2), (4, 3), (8, 3), (2, 8), (8, 8)])
def test_the_round_trip_takes_a_workspace_for_8_bits_alone(bits, monkeypatch):
    from kvquant import TurboQuantBackendPress, _lib
    asked, workspace = [], _lib.workspace
    monkeypatch.setattr(_lib, "workspace", lambda device, size, name, *a: (asked.append(size) if name == "round_trip" else None) or workspace(device, size, name, *a))
    k, v = (torch.randn(1, 2, 300, 128, generator=torch.Generator().manual_seed(s)).half().cuda() for s in (1, 2))
    press = TurboQuantBackendPress(key_bits=bits[0], value_bits=bits[1], value_quantizer="mse")
    got_k, got_v = k.clone(), v.clone()
    press._quantise_span(0, got_k, got_v, 0, 300)
    assert asked == ([_lib.lib.odmkv_round_trip_workspace_bytes(600)] if 8 in bits else [])
    for got, x, b, seed in ((got_k, k, bits[0], 42), (got_v, v, bits[1], 2042)):
        q = press._q(b, seed, x)
        want = q.dequantize(q.quantize(x.view(-1, 128))).view(x.shape)
        assert ((got.float() - want).abs() <= 2 ** -10 * want.abs() + 1e-5).all()       # (as in test_round_trip_in_place)
    kq, vq = press._q(bits[0], 42, k), press._q(bits[1], 2042, v)
    rc = _lib.lib.odmkv_round_trip_rows(k.data_ptr(), v.data_ptr(), _lib.dtype_code(k), 2, 300, 300 * 128, 128, kq.bits, vq.bits, kq.pi.data_ptr(),
                                        vq.pi.data_ptr(), kq.centroids.data_ptr(), vq.centroids.data_ptr(), None, 0, _lib.stream_ptr(k.device))
    torch.cuda.synchronize()
    assert rc == (-1 if 8 in bits else 0)
    assert 8 in bits or (torch.equal(k, got_k) and torch.equal(v, got_v))
