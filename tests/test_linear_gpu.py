"""PackedLinear forward on the GPU, every kind of weight, against the CPU oracle (max |y - ref| <=
1e-3 * max |ref|); more than 16 rows take the many-row kernels, or 16-row calls where those decline."""
import numpy as np
import pytest
import torch

import oracle
from conftest import assert_close
from ishizuki_amd import exl3, ggml, gguf, synth
from ishizuki_amd.linear import PackedLinear

pytestmark = pytest.mark.gpu
DEV = "cuda:0"
dev = lambda a: torch.from_numpy(a).to(DEV)


@pytest.mark.parametrize("rows", [1, 3, 20])
def test_rotated_affine_2bit(rows):
    N, K = 300, 1024
    codes, s, b = synth.affine_pack(N, K, group=64, seed=rows)
    signs = synth.hadamard_signs(K, seed=3)
    x = synth.fp16_normal((rows, K), seed=rows + 1)
    xr = oracle.hadamard(x.astype(np.float32), 128, signs).astype(np.float16).astype(np.float32)
    ref = oracle.affine_matmul(xr, codes, s.view(np.uint16), b.view(np.uint16), N, 2, 64)
    lin = PackedLinear(dev(codes.view(np.int32)), dev(s), dev(b), signs=torch.from_numpy(signs), block=128,
                       group_size=64, bits=2)
    y = lin(dev(x))
    assert y is not None and y.shape == (rows, N)
    assert_close(y.float().cpu().numpy(), ref, what=f"PackedLinear affine rows={rows}")


def test_affine_4bit_three_dim_input():
    N, K = 200, 512
    codes, s, b = synth.affine_pack_bits(N, K, 4, group=128, seed=9)
    x = synth.fp16_normal((2, 3, K), seed=10)
    ref = oracle.affine_matmul(x.reshape(6, K).astype(np.float32), codes, s.view(np.uint16), b.view(np.uint16), N, 4,
                               128).reshape(2, 3, N)
    lin = PackedLinear(dev(codes.view(np.int32)), dev(s), dev(b), group_size=128, bits=4)
    y = lin(dev(x))
    assert y is not None and y.shape == (2, 3, N)
    assert_close(y.float().cpu().numpy(), ref, what="PackedLinear affine 4-bit")


@pytest.mark.parametrize("bits,group", [(2, 64), (4, 64), (4, 128), (8, 64), (4, 32)])
@pytest.mark.parametrize("dt", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("rows", [1, 2, 4, 16, 17])
def test_unrotated_affine_bf16_fp32(bits, group, dt, rows):
    """A pack without a rotation and x of another type than fp16: no workspace but for the bf16 rows' image."""
    N, K = 96, 512
    codes, s, b = (synth.affine_pack(N, K, group=group, seed=rows) if bits == 2 else
                   synth.affine_pack_bits(N, K, bits, group=group, seed=rows))
    x = torch.from_numpy(synth.fp16_normal((rows, K), seed=rows + 1)).to(dt)
    lin = PackedLinear(dev(codes.view(np.int32)), dev(s), dev(b), group_size=group, bits=bits)
    y = lin(x.to(DEV))
    assert y is not None and y.shape == (rows, N) and y.dtype == dt
    xf = x.float().numpy().astype(np.float64)
    W = oracle.affine_dequant(codes, s.view(np.uint16), b.view(np.uint16), N, K, bits, group).astype(np.float64)
    ref = xf @ W.T
    # fp32 sums of exact products (1e-4 of sum |x||w|, as every matmul here), then the output's rounding
    lim = 1e-4 * (np.abs(xf) @ np.abs(W).T) + (2.0 ** -8 if dt == torch.bfloat16 else 0) * np.abs(ref)
    assert (np.abs(y.float().cpu().numpy() - ref) <= lim).all()


def test_ggml_blocks():
    N, K, rows = 96, 1024, 5
    blk = synth.ggml_blocks(ggml.Q6_K, N, K, seed=11)
    x = synth.fp16_normal((rows, K), seed=12)
    ref = oracle.ggml_matmul(ggml.Q6_K, x.astype(np.float32), blk, N)
    lin = PackedLinear.from_ggml(gguf.GGUFBlocks(dev(blk), ggml.Q6_K, (N, K)))
    y = lin(dev(x))
    assert y is not None
    assert_close(y.float().cpu().numpy(), ref, what="PackedLinear ggml")


@pytest.mark.parametrize("t", [ggml.Q4_K, ggml.Q6_K, ggml.Q4_0])
@pytest.mark.parametrize("rows,first", [(40, 96), (95, 96), (96, 96)])
def test_ggml_prompt_on_both_sides_of_the_line(monkeypatch, t, rows, first):
    """Up to 95 rows in 16-row calls, a remainder among them, and the expansion from 96 on: both within the
    bound of the other."""
    monkeypatch.setattr(ggml, "dense_from_rows", lambda *a: first)
    N, K = 48, 512
    blk = synth.ggml_blocks(t, N, K, seed=rows)
    x = synth.fp16_normal((rows, K), seed=rows + 1)
    y = PackedLinear.from_ggml(gguf.GGUFBlocks(dev(blk), t, (N, K)))(dev(x))
    assert_close(y.float().cpu().numpy(), oracle.ggml_matmul(t, x.astype(np.float32), blk, N), what=f"ggml prompt t={t} rows={rows}")


def test_exl3_and_dense():
    K, N, rows = 512, 256, 3
    t, suh, svh = synth.exl3_pack(K, N, bits2=4, seed=13)
    ten = exl3.EXL3Tensor(dev(t), dev(suh), dev(svh))
    x = synth.fp16_normal((rows, K), seed=14)
    ref = oracle.exl3_apply(x.astype(np.float32), t, suh, svh, 4, 0)
    y = PackedLinear.from_exl3(ten)(dev(x))
    assert y is not None
    assert_close(y.float().cpu().numpy(), ref, what="PackedLinear exl3")
    w = synth.fp16_normal((N, K), seed=15)
    yd = PackedLinear.dense(dev(w))(dev(x))
    refd = x.astype(np.float32) @ w.astype(np.float32).T
    assert_close(yd.float().cpu().numpy(), refd, what="PackedLinear dense")


@pytest.mark.parametrize("K", [512, 384])
@pytest.mark.parametrize("shape", [(17,), (40,), (2, 65)])
def test_exl3_prompt(K, shape):
    """More than 16 rows of an EXL3 projection: the many-row kernel, and 16-row calls for a K it declines."""
    N = 256
    t, suh, svh = synth.exl3_pack(K, N, bits2=4, seed=K)
    ten = exl3.EXL3Tensor(dev(t), dev(suh), dev(svh))
    x = synth.fp16_normal((*shape, K), seed=16)
    rows = x.reshape(-1, K)
    assert (exl3.apply_rows(dev(rows), ten) is None) == (K == 384)
    ref = np.concatenate([oracle.exl3_apply(rows[r:r + 16].astype(np.float32), t, suh, svh, 4, 0) for r in range(0, len(rows), 16)])
    y = PackedLinear.from_exl3(ten)(dev(x))
    assert y is not None and y.shape == (*shape, N)
    assert_close(y.float().cpu().numpy().reshape(-1, N), ref, what=f"PackedLinear exl3 prompt K={K} {shape}")
