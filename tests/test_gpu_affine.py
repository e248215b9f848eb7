"""Affine group-wise quantize / dequantize on the GPU vs the CPU restatement
of MLX's algorithm: bit-exact codes, scales and biases."""
import json
from pathlib import Path

import numpy as np
import pytest

import mlxq
import oracle as orc
from helpers import bf16_weights, dev, host

pytestmark = pytest.mark.gpu
KAT = json.loads((Path(__file__).resolve().parent / "golden" / "gguf_kat.json").read_text())


def gpu_quantize(w, gs, bits, bf16):
    import torch

    wq, s, b = mlxq.quantize(dev(w, bf16=bf16), gs, bits)
    torch.cuda.synchronize()
    return host(wq), host(s), host(b)


@pytest.mark.parametrize("bits", [4, 8])
@pytest.mark.parametrize("gs", [32, 64, 128])
@pytest.mark.parametrize("bf16", [True, False])
def test_codes_bit_exact(torch_gpu, bits, gs, bf16):
    rows, cols = 96, 1024
    w = bf16_weights(1000 + bits + gs, rows, cols)
    if not bf16:
        w = orc.normal(2000 + bits + gs, rows * cols, 0.0, 0.02).reshape(rows, cols)
    w = w.copy()
    # edge cases: constant group, zero group, one outlier, exact ramp
    if bf16:
        w[0, :gs] = orc.f32_to_bf16(np.float32([0.25]))[0]
        w[1, :gs] = 0
        w[2, 5] = orc.f32_to_bf16(np.float32([3.0]))[0]
    else:
        w[0, :gs] = 0.25
        w[1, :gs] = 0
        w[2, 5] = 3.0
        w[3, :gs] = np.arange(gs) % 16
    ref = orc.affine_quantize(w, gs, bits, orc.BF16 if bf16 else orc.F32)
    got = gpu_quantize(w, gs, bits, bf16)
    for r, g in zip(ref, got):
        assert np.array_equal(np.asarray(r).view(np.uint8), np.asarray(g).view(np.uint8))


@pytest.mark.parametrize("bits", [4, 8])
def test_dequantize_bit_exact(torch_gpu, bits):
    import torch

    w = bf16_weights(31 + bits, 64, 512)
    wq, s, b = orc.affine_quantize(w, 64, bits, orc.BF16)
    ref = orc.affine_dequantize(wq, s, b, 64, bits, orc.BF16)
    got = mlxq.dequantize(dev(wq), dev(s, bf16=True), dev(b, bf16=True), 64, bits)
    torch.cuda.synchronize()
    assert np.array_equal(host(got), ref)
    wf = orc.normal(40 + bits, 64 * 512, 0, 0.02).reshape(64, 512)
    wq, s, b = orc.affine_quantize(wf, 64, bits, orc.F32)
    ref = orc.affine_dequantize(wq, s, b, 64, bits, orc.F32)
    got = mlxq.dequantize(dev(wq), dev(s), dev(b), 64, bits)
    torch.cuda.synchronize()
    assert np.array_equal(host(got).view(np.uint32), ref.view(np.uint32))


def test_reference_roundtrip_q8(torch_gpu):
    import torch

    a = KAT["affine"]["roundtrip_q8"]  # quant.rs:91-107
    w = np.float32(a["w"]).reshape(a["shape"])
    wq, s, b = mlxq.quantize(dev(w), 64, 8)
    back = host(mlxq.dequantize(wq, s, b, 64, 8))
    torch.cuda.synchronize()
    assert np.max(np.abs(back - w)) < a["max_abs_err"]


@pytest.mark.parametrize("shape", [(4096, 4096), (14336, 4096), (4096, 14336)])
@pytest.mark.parametrize("bits", [4, 8])
def test_llama_shapes_bit_exact(torch_gpu, shape, bits):
    n, k = shape
    w = bf16_weights(0x5EED0000 + n + k + bits, n, k)
    ref = orc.affine_quantize(w, 64, bits, orc.BF16)
    got = gpu_quantize(w, 64, bits, True)
    for r, g in zip(ref, got):
        assert np.array_equal(r.view(np.uint8), g.view(np.uint8))


@pytest.mark.parametrize("bits", [4, 8])
@pytest.mark.parametrize("factor", [1.0, 0.02, 3.0e-5, 7.0, 0.0123457, 3.3e-3, 1.7e-6, 0.7071068, 511.3, 9.9e-2,
                                    3.1e20, 2.0e30])
def test_codes_at_rounding_ties(torch_gpu, bits, factor):
    """Groups whose quotients (w - bias) / scale sit on or within a few ulps
    of half-integers: min 0 and max n_bins (times `factor`) make scale
    -factor and bias max, so every element j + 1/2 (times `factor`) lands on a
    tie of the code rounding; with factor not a power of two the f32 products
    put the quotients a few ulps to either side of it.  The two largest
    factors give scales above 2^60, where the quantizer takes the division
    instead of its unscaled form of it."""
    rng = np.random.default_rng(77 + bits)
    n_bins = (1 << bits) - 1
    gs, rows, cols = 64, 64, 512
    half = rng.integers(0, 2 * n_bins + 1, size=(rows, cols)).astype(np.float32) / 2
    half = half.reshape(rows, cols // gs, gs)
    half[:, :, 0] = 0
    half[:, :, 1] = n_bins
    w = (half.reshape(rows, cols) * np.float32(factor)).astype(np.float32)
    ref = orc.affine_quantize(w, gs, bits, orc.F32)
    got = gpu_quantize(w, gs, bits, False)
    for r, g in zip(ref, got):
        assert np.array_equal(np.asarray(r).view(np.uint8), np.asarray(g).view(np.uint8))


@pytest.mark.parametrize("bits", [4, 8])
@pytest.mark.parametrize("gs", [32, 64, 128])
@pytest.mark.parametrize("bf16", [True, False])
def test_groups_outside_the_ordinary_range(torch_gpu, bits, gs, bf16):
    """Groups that leave the short quotient's range or sit on its edges: huge,
    tiny and subnormal values, infinities, single NaN elements, a scale whose
    mantissa is all ones with a quotient next to one half, and a row count
    whose last workgroup is partial.  Codes bit-exact, scales and biases too
    except for the payload of a NaN."""
    rng = np.random.default_rng(5 + gs)
    n_bins = (1 << bits) - 1
    s1 = np.float32(float.fromhex("0x1.fffffep-7"))
    half = (n_bins + 1) // 2
    groups = [rng.normal(0, f, gs) for f in (1e-30, 1e-42, 1e-8, 3e-7, 2e18, 1e25, 1e37, 1e38)]
    groups += [np.where(rng.random(gs) < 0.5, -3e38, 3e38), np.full(gs, -0.0)]
    for bad in (np.inf, -np.inf, np.nan):
        g = rng.normal(0, 0.02, gs)
        g[gs // 2 + 3] = bad
        groups.append(g)
    edge = np.full(gs, float(half * s1))  # scale = edge / half: all mantissa bits set
    edge[1] = float(-(half - 1) * s1)
    edge[2::2] = float(half * s1) - 2.0**-7  # quotient 0.5 rounded from just above
    groups += [edge, -edge]
    rows = 37
    w = rng.normal(0, 0.02, (rows, 4 * gs)).astype(np.float32)
    flat = w.reshape(-1, gs)
    for i, g in enumerate(groups):
        with np.errstate(over="ignore", under="ignore"):
            flat[5 * i] = g.astype(np.float32)
    w = flat.reshape(rows, 4 * gs)
    if bf16:
        w = orc.f32_to_bf16(w).reshape(rows, 4 * gs)
    ref = orc.affine_quantize(w, gs, bits, orc.BF16 if bf16 else orc.F32)
    got = gpu_quantize(w, gs, bits, bf16)
    assert np.array_equal(ref[0], got[0].view(np.uint32))
    for r, g in zip(ref[1:], got[1:]):
        r = orc.bf16_to_f32(np.asarray(r)) if bf16 else np.asarray(r)
        g = orc.bf16_to_f32(np.asarray(g).view(np.uint16)) if bf16 else np.asarray(g)
        assert np.array_equal(r.reshape(-1), g.reshape(-1), equal_nan=True)


@pytest.mark.parametrize("bits", [4, 8])
@pytest.mark.parametrize("gs", [32, 64, 128])
@pytest.mark.parametrize("bf16", [True, False])
def test_narrow_groups_of_one_sign(torch_gpu, bits, gs, bf16):
    """Groups whose values have one sign and a small spread: edge / scale runs
    from the number of bins to 2^30 (constant groups: scale 1e-7), far past
    the quotients of a group around zero.  The first values are the constant
    groups for which a reciprocal one ulp off changes the last bit of the
    scale.  Codes, scales and biases bit-exact."""
    rng = np.random.default_rng(0x51 + gs)
    hard = [float.fromhex("0x1.b5b6b2p-1") * 2.0**e for e in range(12)]
    level = np.float32(hard + list(np.exp(rng.uniform(np.log(1e-3), np.log(1e3), 500))))
    spread = np.where(np.arange(512) % 4 == 0, 0.0, np.exp(rng.uniform(np.log(1e-7), np.log(0.9), 512)))
    spread[:len(hard)] = 0
    sign = np.where(np.arange(512) % 2, -1.0, 1.0)
    w = level[:, None] * (1.0 - spread[:, None] * rng.random((512, gs))) * sign[:, None]
    w = w.astype(np.float32).reshape(128, 4 * gs)
    if bf16:
        w = orc.f32_to_bf16(w).reshape(128, 4 * gs)
    ref = orc.affine_quantize(w, gs, bits, orc.BF16 if bf16 else orc.F32)
    got = gpu_quantize(w, gs, bits, bf16)
    for r, g in zip(ref, got):
        assert np.array_equal(np.asarray(r).view(np.uint8), np.asarray(g).view(np.uint8))


@pytest.mark.parametrize("bits", [4, 8])
@pytest.mark.parametrize("gs", [32, 64, 128])
@pytest.mark.parametrize("bf16", [True, False])
@pytest.mark.parametrize("rows,cols", [(1, 128), (3, 384), (33, 640)])
def test_dequantize_partial_workgroups(torch_gpu, bits, gs, bf16, rows, cols):
    import torch

    w = bf16_weights(77 + bits, rows, cols)
    if not bf16:
        w = orc.normal(78 + bits, rows * cols, 0, 0.02).reshape(rows, cols)
    dt = orc.BF16 if bf16 else orc.F32
    wq, s, b = orc.affine_quantize(w, gs, bits, dt)
    ref = orc.affine_dequantize(wq, s, b, gs, bits, dt)
    got = mlxq.dequantize(dev(wq), dev(s, bf16=bf16), dev(b, bf16=bf16), gs, bits)
    torch.cuda.synchronize()
    assert np.array_equal(host(got).view(np.uint8), np.asarray(ref).view(np.uint8))


@pytest.mark.parametrize("bits", [4, 8])
@pytest.mark.parametrize("bf16", [True, False])
def test_quantize_codes_at_word_alignment(torch_gpu, bits, bf16):
    """The code words may start at any 4-byte (Q8: 8-byte) boundary, although
    a lane stores up to four of them at once: bit-exact, and nothing before or
    after the array is written."""
    import torch

    n, k, gs = 33, 640, 64
    w = bf16_weights(0x61 + bits, n, k)
    if not bf16:
        w = orc.normal(0x62 + bits, n * k, 0.0, 0.02).reshape(n, k)
    ref = orc.affine_quantize(w, gs, bits, orc.BF16 if bf16 else orc.F32)
    words, step = n * k * bits // 32, bits // 4
    for off in range(step, 5, step):
        buf = torch.full((words + 8,), -1, dtype=torch.int32, device="cuda")
        x = dev(w, bf16=bf16)
        s = torch.empty((n, k // gs), dtype=x.dtype, device="cuda")
        b = torch.empty_like(s)
        mlxq.check(mlxq.lib().mlxq_quantize(x.data_ptr(), mlxq.BF16 if bf16 else mlxq.F32, n, k, gs, bits,
                                            buf.data_ptr() + 4 * off, s.data_ptr(), b.data_ptr(), mlxq._stream()))
        got = host(buf)
        assert np.array_equal(got[off:off + words], ref[0].reshape(-1).view(np.uint32)), off
        assert np.all(got[:off] == 0xFFFFFFFF) and np.all(got[off + words:] == 0xFFFFFFFF)
