"""GPU parity: NVFP4 quantize / dequantize through the C ABI against the CPU oracle and the golden
vectors.  Bar: bit-exact packed nibbles, scale bytes and amax."""
import ctypes

import numpy as np
import pytest
import torch

import nvfp4_oracle as o
from helpers import activations, bits_of, from_bits, hardware_convert, u8, weights
from longlive_amd import _native
from longlive_amd.fouroversix import QuantizationConfig, QuantizedTensor, quantize_to_fp4

pytestmark = pytest.mark.gpu
RULES = list(o.SCALE_RULES)


def _check(x_bits, rule, dev):
    q = quantize_to_fp4(from_bits(x_bits, dev), QuantizationConfig(scale_rule=rule))
    v, s, a, pad = o.quantize_to_fp4(x_bits, rule)
    assert q.padded_shape == pad
    assert float(q.amax.cpu()) == float(a)
    sg = u8(q.scale_factors)
    assert np.array_equal(sg, s), f"{rule}: {(sg != s).sum()} scale bytes differ"
    vg = u8(q.values)
    assert np.array_equal(vg, v), f"{rule}: {(vg != v).sum()} value bytes differ"
    return q


def test_hardware_e4m3_conversion_matches_software_codec(gpu):
    x = np.concatenate([np.linspace(0, 448, 200001, dtype=np.float32),
                        o.e4m3_decode(np.arange(127, dtype=np.uint8)),
                        np.array([2**-10, 2**-10 * 1.001, 3 * 2**-10, 2**-9 * 2.5, 17.0, 19.0, 27.0], dtype=np.float32)])
    got = hardware_convert(torch.from_numpy(x).to(gpu), 0).cpu().numpy()
    assert np.array_equal(got, o.e4m3_encode(x))


def test_hardware_e2m1_conversion_matches_reference_rounding(gpu):
    x = np.concatenate([np.linspace(-6.9, 6.9, 400001, dtype=np.float32),
                        np.array([0.25, 0.75, 1.25, 1.75, 2.5, 3.5, 5.0, -0.25, -2.5, -5.0, -0.1, 0.0], dtype=np.float32)])
    got = hardware_convert(torch.from_numpy(x).to(gpu), 1).cpu().numpy()
    ref = o._codes_from_fake_quantized(o._fake_quantize_e2m1(x))
    assert np.array_equal(got, ref)


@pytest.mark.parametrize("rule", RULES)
def test_golden_vectors(golden, gpu, rule):
    for name in golden["case_names"]:
        q = quantize_to_fp4(from_bits(golden[f"{name}/x"], gpu), QuantizationConfig(scale_rule=rule))
        assert float(q.amax.cpu()) == float(golden[f"{name}/{rule}/amax"][0]), name
        assert np.array_equal(u8(q.scale_factors), golden[f"{name}/{rule}/scales"]), name
        assert np.array_equal(u8(q.values), golden[f"{name}/{rule}/values"]), name


@pytest.mark.parametrize("rule", RULES)
@pytest.mark.parametrize("shape,seed", [((128, 64), 0), ((256, 192), 1), ((130, 70), 2), ((1, 16), 3), ((257, 1000), 4)])
def test_random_and_ragged_shapes(gpu, rule, shape, seed):
    _check(bits_of(activations(shape, seed)), rule, gpu)


@pytest.mark.parametrize("rule", ["mse", "static_6"])
def test_input_classes_of_the_reference_test(gpu, rule):
    g = torch.Generator().manual_seed(0)
    for x in (torch.zeros(512, 1024), torch.ones(512, 1024), torch.rand(512, 1024, generator=g),
              torch.randn(1024, 512, generator=g)):
        _check(bits_of(x.bfloat16()), rule, gpu)


def test_edge_values(gpu):
    x = torch.randn(128, 128, generator=torch.Generator().manual_seed(5))
    x[0, :16] = -0.0                      # negative zeros -> code 0
    x[1, :16] = torch.tensor([-1e-4] * 16)  # negatives that round to zero -> code 8
    x[2, :] *= 1e-6                       # blocks with sub-normal / zero e4m3 scales
    x[3, :] *= 3e-5
    x[4, 0] = 250.0                       # sets amax; other blocks far below
    for rule in RULES:
        _check(bits_of(x.bfloat16()), rule, gpu)
    tiny = (torch.randn(128, 64, generator=torch.Generator().manual_seed(6)) * 1e-30).bfloat16()
    huge = (torch.randn(128, 64, generator=torch.Generator().manual_seed(7)) * 1e30).bfloat16()
    for t in (tiny, huge):
        for rule in ("mse", "static_6"):
            _check(bits_of(t), rule, gpu)


def test_benchmark_activation_full_size(gpu):
    """Config 1 activation [2640, 3072], seed 0, rule mse: full-size bit-exact comparison."""
    _check(bits_of(activations((2640, 3072), 0)), "mse", gpu)


@pytest.mark.parametrize("rule", ["mse", "mae"])
def test_ffn_down_activation_full_size_bit_exact(gpu, rule):
    """The activation with the most blocks, [2640, 14336] (2.4 million blocks of 16, the input of the FFN-down
    linear), against the CPU oracle bit for bit: every block whose four-over-six choice the kernel takes from its
    error estimate instead of the reference's arithmetic is one more chance for a wrong confident decision to show."""
    _check(bits_of(activations((2640, 14336), 10)), rule, gpu)


def test_strided_input_and_given_amax(gpu):
    big = activations((200, 512), 8).to(gpu)
    view = big[:, 128:384]  # row stride 512, 256 columns
    q = quantize_to_fp4(view)
    v, s, a, _ = o.quantize_to_fp4(bits_of(view), "mse")
    assert np.array_equal(u8(q.values), v) and np.array_equal(u8(q.scale_factors), s)
    amax = torch.tensor([float(a) * 2], device=gpu)
    vals, sc, am = _native.quantize(view, "mse", amax=amax)
    v2, s2, a2, _ = o.quantize_to_fp4(bits_of(view), "mse", amax=np.float32(float(a) * 2))
    assert np.array_equal(u8(vals), v2) and np.array_equal(u8(sc), s2) and float(am.cpu()) == float(a2)


@pytest.mark.parametrize("rule,factor", [(r, f) for r in ("mse", "mae", "static_6", "abs_max") for f in (1.0, 1.7, 30.0)]
                         + [(r, 0.9) for r in ("mse", "mae", "abs_max")])   # the static rules put the amax itself at 448, the end of e4m3
def test_caller_supplied_amax_bit_exact(gpu, rule, factor):
    """A precomputed amax (quantize/pytorch/reference.py:244) that is the true maximum, larger than it, or a little
    smaller (the blocks above the given amax, here by up to 11 %, get scales above 256 that e4m3 still holds; they
    take the reference's own arithmetic block by block, the others the fast path), against the oracle bit for bit.
    An amax so far below the maximum that block scales leave the e4m3 range (NaN in the reference) is not a
    supported input."""
    x = activations((384, 1024), 23).to(gpu)
    true_amax = float(x.float().abs().max())
    given = np.float32(true_amax * factor)
    vals, sc, am = _native.quantize(x, rule, amax=torch.tensor([given], device=gpu))
    v, s, a, _ = o.quantize_to_fp4(bits_of(x), rule, amax=given)
    assert float(am.cpu()) == float(a) == float(given)
    assert np.array_equal(u8(sc), s)
    assert np.array_equal(u8(vals), v)


def test_rejects_non_bf16_and_cpu_input(gpu):
    with pytest.raises(ValueError, match="bfloat16"):
        quantize_to_fp4(torch.zeros(128, 64, device=gpu))


@pytest.mark.parametrize("rule", ["mse", "static_6", "static_4"])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16, torch.float16])
def test_dequantize_matches_oracle(gpu, rule, dtype):
    x = activations((130, 200), 9)
    q = quantize_to_fp4(x.to(gpu), QuantizationConfig(scale_rule=rule))
    got = q.dequantize(dtype)
    assert got.shape == (130, 200) and got.dtype == dtype
    ref = o.dequantize(u8(q.values), u8(q.scale_factors), np.float32(q.amax.item()), rule, q.padded_shape, (130, 200))
    if dtype == torch.float32:
        assert np.array_equal(got.cpu().numpy(), ref)
    else:
        assert torch.equal(got.cpu(), torch.from_numpy(ref).to(dtype))


@pytest.mark.parametrize("shape", [(1, 16), (31, 250), (32, 256), (129, 264), (256, 520)])
@pytest.mark.parametrize("amax", [0.0, 1e-35, 1.7, 3e35])
def test_dequantize_every_code_and_scale_byte(gpu, shape, amax):
    """Random bytes (all codes, all finite scale bytes of both signs) at the edges of the kernel's 32 x 256 tiles, with
    amax values inside and outside the range in which it scales by powers of two: equal to the oracle's divisions."""
    from longlive_amd._native import padded_shape
    rng = np.random.default_rng(5)
    mp, kp = padded_shape(shape)
    v = rng.integers(0, 256, (mp, kp // 2), dtype=np.uint8)
    s = rng.integers(0, 256, mp * kp // 16, dtype=np.uint8)
    s[(s & 0x7F) == 0x7F] = 0x7E
    q = QuantizedTensor(torch.from_numpy(v).to(gpu), torch.from_numpy(s).to(gpu).view(torch.float8_e4m3fn),
                        torch.tensor([amax], device=gpu), "nvfp4", shape, "mse", (mp, kp))
    ref = o.dequantize(v, s, np.float32(amax), "mse", (mp, kp), shape)
    got = q.dequantize(torch.float32).cpu().numpy()
    assert np.array_equal(got.view(np.uint32), np.ascontiguousarray(ref).view(np.uint32))
    assert torch.equal(q.dequantize(torch.bfloat16).cpu(), torch.from_numpy(ref).bfloat16())


def test_dequantize_golden(golden, gpu):
    for name, shape in (("randn_128x512_s1", (128, 512)), ("weights_256x512_s2", (256, 512))):
        v, s, a = (golden[f"{name}/mse/{k}"] for k in ("values", "scales", "amax"))
        qt = QuantizedTensor(torch.from_numpy(v).to(gpu), torch.from_numpy(s).to(gpu).view(torch.float8_e4m3fn),
                             torch.from_numpy(a).to(gpu), "nvfp4", shape, "mse", shape)
        assert np.array_equal(qt.dequantize(torch.float32).cpu().numpy(), golden[f"{name}/mse/deq_f32"])
        assert np.array_equal(bits_of(qt.dequantize(torch.bfloat16)), golden[f"{name}/mse/deq_bf16"])


def test_round_trip_property_at_full_ffn_size(gpu):
    """Size-independent property at the largest benchmark activation [2640, 14336]: dequantize(quantize(x))
    re-quantized with the same amax and a static rule reproduces the same bytes (idempotence), and the
    relative error of the four-over-six result is not worse than plain NVFP4."""
    x = activations((2640, 14336), 10).to(gpu)
    q6 = quantize_to_fp4(x, QuantizationConfig(scale_rule="static_6"))
    d6 = q6.dequantize(torch.float32)
    qm = quantize_to_fp4(x, QuantizationConfig(scale_rule="mse"))
    dm = qm.dequantize(torch.float32)
    e6 = (d6 - x.float()).pow(2).sum().item()
    em = (dm - x.float()).pow(2).sum().item()
    assert em <= e6 * 1.0001
    assert float(qm.amax.cpu()) == float(x.float().abs().max().cpu())
    assert q6.values.shape == (2688, 7168) and not q6.values[2640:].any()


@pytest.mark.parametrize("rule", ["mse", "mae", "abs_max"])
def test_four_over_six_choice_on_ties_and_near_ties(gpu, rule):
    """The kernel decides most blocks from error estimates in units of the block's step and falls back to the
    reference's own arithmetic when the two candidates are close.  Inputs built to make them close or equal:
    values on a coarse lattice (many exact ties), lattice values nudged by one bf16 ulp, blocks repeated at
    many magnitudes, a tensor amax far from the blocks' size, and blocks far below the tensor amax (scale byte 0)."""
    rng = np.random.default_rng(7)
    rows, cols = 1024, 256
    lattice = rng.integers(-12, 13, size=(rows, cols)).astype(np.float32) * 0.25
    nudged = lattice * (1.0 + rng.choice([-2.0 ** -8, 0.0, 2.0 ** -8], size=lattice.shape)).astype(np.float32)
    magn = rng.standard_normal((rows, cols)).astype(np.float32) * np.exp2(rng.integers(-12, 6, size=(rows, 1))).astype(np.float32)
    two_level = np.where(rng.random((rows, cols)) < 0.5, 1.0, 1.5).astype(np.float32) * rng.choice([-1.0, 1.0], size=(rows, cols)).astype(np.float32)
    tiny = rng.standard_normal((rows, cols)).astype(np.float32) * 1e-7
    tiny[0, 0] = 300.0  # tensor amax: the other blocks get scale byte 0 or subnormal scale bytes
    for x in (lattice, nudged, magn, two_level, tiny):
        _check(bits_of(torch.from_numpy(x).bfloat16()), rule, gpu)


@pytest.mark.parametrize("rows,C,rule", [(300, 256, "mse"), (2640, 3072, "mse"), (130, 128, "static_6")])
def test_two_tensors_in_one_launch_equal_the_oracle(gpu, rows, C, rule):
    """The K and V of a chunk go into the cache as one launch (two tensors of one shape, each with the amax its
    producer left in a sink of its own): bytes and amax of both equal the oracle's, i.e. those of two launches."""
    g = torch.Generator().manual_seed(rows + C)
    xs = [(torch.randn(rows, C, generator=g) * s).bfloat16().to(gpu) for s in (1.0, 7.0)]
    sinks = [_native.PrivateAmaxSink(gpu), _native.PrivateAmaxSink(gpu)]
    tickets = [s.ticket() for s in sinks]
    ys = [_native.layer_norm(x, None, None, amax_out=t).reshape(-1, 128) for x, t in zip(xs, tickets)]
    Mp, Kp = _native.padded_shape(tuple(ys[0].shape))
    outs = [(torch.empty((Mp, Kp // 2), dtype=torch.uint8, device=gpu),
             torch.empty(Mp * Kp // 16, dtype=torch.uint8, device=gpu),
             torch.empty(1, dtype=torch.float32, device=gpu)) for _ in range(2)]
    _native.quantize_pair(ys[0], ys[1], rule, tickets[0], tickets[1], outs[0], outs[1])
    for y, (values, scales, amax) in zip(ys, outs):
        v, s, a, _ = o.quantize_to_fp4(bits_of(y), rule)
        assert float(amax.cpu()) == float(a)
        assert np.array_equal(u8(scales), s) and np.array_equal(u8(values), v)
    with pytest.raises(ValueError, match="two sink buffers"):
        t = sinks[0].ticket()
        _native.layer_norm(xs[0], None, None, amax_out=t)
        _native.quantize_pair(ys[0], ys[1], rule, t, t, outs[0], outs[1])


@pytest.mark.parametrize("rule", ["mse", "static_6", "static_4", "mae", "abs_max"])
@pytest.mark.parametrize("M,K,pad", [(1, 64, 0), (48, 256, 0), (129, 192, 8), (512, 3072, 0), (1173, 1536, 0), (4096, 512, 0), (130, 8192, 24)])
def test_small_tensors_in_one_launch_have_the_bytes_of_the_two_launches(gpu, rule, M, K, pad):
    """Up to 256 tiles of 128 x 64, one workgroup each: ragged rows, rows with a stride, one tile, as many as the rule takes;
    several calls on one sink with the maximum falling; with the wait's way out (every workgroup computes all maxima);
    a tensor of zeros and one with maxima outside the fast path."""
    lib, stream, code = _native.load(), torch.cuda.current_stream().cuda_stream, _native.RULE_IDS[rule]
    g = torch.Generator(device=gpu).manual_seed(M + K)
    Mp, Kp = -(-M // 128) * 128, K
    parts = torch.zeros(1024, dtype=torch.int64, device=gpu)
    for i, (scale, spin) in enumerate([(1e3, 64), (1.0, 64), (0.01, -1), (0.0, 64), (1e35, 64), (1.0, 0)]):
        x = (torch.randn((M, K + pad), generator=g, device=gpu) * scale).bfloat16()[:, :K]
        x[0, -1] *= 30
        outs = []
        for once in (True, False):
            v, s, a = (torch.full((n,), 7, dtype=t, device=gpu) for n, t in ((Mp * Kp // 2, torch.uint8), (Mp * Kp // 16, torch.uint8),
                                                                            (1, torch.float32)))
            ws = torch.empty(1024, dtype=torch.float32, device=gpu)
            args = (x.data_ptr(), M, K, x.stride(0), code, v.data_ptr(), s.data_ptr(), a.data_ptr())
            if once:
                sink = _native.AmaxSinkStruct(parts.data_ptr(), i + 1, None)
                rc = lib.ll_nvfp4_quantize_once(*args, ctypes.byref(sink), spin, stream)
            else:
                rc = lib.ll_nvfp4_quantize(*args, 0, ws.data_ptr(), stream)
            assert rc == 0, lib.ll_last_error()
            outs.append((v, s, a))
        assert all(torch.equal(p, q) for p, q in zip(*outs)), (i, scale, spin)
    assert lib.ll_nvfp4_quantize_once(x.data_ptr(), 128 * 257, 64, 64, *args[4:], ctypes.byref(sink), 64, stream) == -3   # refused on the host


@pytest.mark.parametrize("rule", ["mse", "static_4", "abs_max"])
@pytest.mark.parametrize("M,K,pad,tensors", [(1, 64, 0, 2), (1173, 2112, 8, 1), (16384, 256, 0, 1), (5888, 128, 0, 2), (16321, 128, 8, 2), (32768, 128, 0, 2)])
def test_one_pass_has_the_bytes_of_the_two_launches(gpu, rule, M, K, pad, tensors):
    """One or two tensors of up to 512 tiles, one or two tiles per workgroup: an odd number of them, as many as the rule takes,
    ragged rows and rows with a stride; several calls on one sink with the maxima falling, with the wait's way out, and with
    zeros and maxima outside the fast path.  The two tensors differ in scale, so that neither may see the other's maximum."""
    lib, stream, code = _native.load(), torch.cuda.current_stream().cuda_stream, _native.RULE_IDS[rule]
    g = torch.Generator(device=gpu).manual_seed(M + K)
    Mp = -(-M // 128) * 128
    parts = torch.zeros(1024, dtype=torch.int64, device=gpu)
    ws = torch.empty(1024, dtype=torch.float32, device=gpu)

    def buffers():
        return [torch.full((n,), 7, dtype=t, device=gpu) for n, t in ((Mp * K // 2, torch.uint8), (Mp * K // 16, torch.uint8), (1, torch.float32))]

    for i, (scale, spin) in enumerate([(1e3, 64), (1.0, 64), (0.01, -1), (0.0, 64), (1e35, 64), (1.0, 0)]):
        xs = [(torch.randn((M, K + pad), generator=g, device=gpu) * scale * f).bfloat16()[:, :K] for f in (1.0, 0.3, 5.0)[i % 2:][:tensors]]
        xs[0][0, -1] *= 30
        got, want = [buffers() for _ in xs], [buffers() for _ in xs]
        sink = _native.AmaxSinkStruct(parts.data_ptr(), i + 1, None)
        two = [(x, o) for x, o in zip(xs, got)] if tensors == 2 else [(xs[0], got[0]), (None, [None] * 3)]
        ptr = lambda t: t.data_ptr() if t is not None else None
        args = [v for j in range(3) for v in (ptr(two[0][1][j]), ptr(two[1][1][j]))]
        assert lib.ll_nvfp4_quantize_one_pass(xs[0].data_ptr(), ptr(two[1][0]), M, K, xs[0].stride(0), code, *args, ctypes.byref(sink), spin,
                                              stream) == 0, lib.ll_last_error()
        for x, (v, s, a) in zip(xs, want):
            assert lib.ll_nvfp4_quantize(x.data_ptr(), M, K, x.stride(0), code, v.data_ptr(), s.data_ptr(), a.data_ptr(), 0, ws.data_ptr(), stream) == 0
        assert all(torch.equal(p, q) for a, b in zip(got, want) for p, q in zip(a, b)), (i, scale, spin)
    assert lib.ll_nvfp4_quantize_one_pass(xs[0].data_ptr(), None, 128 * 513, 64, 64, code, *args, ctypes.byref(sink), 64, stream) == -3   # refused on the host


def test_small_quantization_recorded_into_a_graph(gpu):
    """While a stream is being captured the two launches are recorded: replays on a falling maximum equal the eager bytes."""
    cfg = QuantizationConfig(scale_rule="mse")
    xs = [(torch.randn(200, 512, generator=torch.Generator().manual_seed(i)) * s).bfloat16().to(gpu) for i, s in enumerate((8.0, 1.0, 0.1))]
    eager = [quantize_to_fp4(x, cfg) for x in xs]
    static, side = xs[0].clone(), torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        quantize_to_fp4(static, cfg)
    torch.cuda.current_stream().wait_stream(side)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=side):
        q = quantize_to_fp4(static, cfg)
    for x, ref in zip(xs, eager):
        static.copy_(x)
        graph.replay()
        torch.cuda.synchronize()
        quantize_to_fp4(x, cfg)
        assert torch.equal(q.values, ref.values) and torch.equal(q.amax, ref.amax)
        assert torch.equal(q.scale_factors.view(torch.uint8), ref.scale_factors.view(torch.uint8))
