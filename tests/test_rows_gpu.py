"""Many-row products (prompts: PackedLinear with more than 16 rows) against the CPU oracle: row counts at
the edges of the 16-row tiles and the 128-row workgroups, column counts that do not fill a workgroup, a K
split into parts, gathered groups, every width and trellis rate the kernels take, fp16 and bf16.

Products of the exact codes are summed in fp32, as in the kernels for up to 16 rows: held to the same
per-element bound, 1e-4 of sum |x||w| plus the rounding of the output."""
import numpy as np
import pytest
import torch

import oracle
from ishizuki_amd import affine, exl3, synth

pytestmark = pytest.mark.gpu
DEV = "cuda:0"
dev = lambda a: torch.from_numpy(a).to(DEV)


def act(M, K, seed, dt):
    x = np.random.default_rng(seed).standard_normal((M, K)).astype(np.float32)
    if dt == torch.bfloat16:
        x[1] *= 1.0e6
        x[2] *= 1.0e-7
    t = torch.from_numpy(x).to(dt)
    return t.to(DEV), t.float().numpy()


def check(y, ref, bound, dt, what):
    y, ref = y.float().cpu().numpy().astype(np.float64), np.asarray(ref, np.float64)
    assert np.isfinite(y).all(), what
    lim = 1e-4 * bound + (2.0 ** -8 if dt == torch.bfloat16 else 2.0 ** -10) * np.abs(ref) + 1e-30
    bad = np.abs(y - ref) > lim
    assert not bad.any(), f"{what}: {int(bad.sum())} outside; worst {np.max(np.abs(y - ref) / lim):.3g}x the bound"


@pytest.mark.parametrize("bits,group,dt,M,N,K", [
    (2, 64, torch.float16, 17, 130, 256), (2, 64, torch.float16, 128, 128, 512), (2, 128, torch.bfloat16, 129, 300, 1024),
    (2, 64, torch.float16, 300, 257, 2816), (4, 64, torch.float16, 33, 96, 512), (4, 128, torch.float16, 200, 40, 768),
    (4, 64, torch.bfloat16, 31, 513, 4096), (6, 64, torch.float16, 18, 100, 512), (8, 64, torch.bfloat16, 144, 129, 768),
    (8, 128, torch.float16, 17, 16, 1280)])
@pytest.mark.parametrize("sdt", [torch.float16, torch.bfloat16])
def test_affine_rows(bits, group, dt, M, N, K, sdt):
    print(f"affine rows bits={bits} group={group} M={M} N={N} K={K} {dt} scales {sdt}", flush=True)
    if bits == 2:
        codes, s, b = synth.affine_pack(N, K, group=group, seed=bits + M)
    else:
        codes, s, b = synth.affine_pack_bits(N, K, bits, group=group, seed=bits + M)
    x, xf = act(M, K, M + K, dt)
    if sdt == torch.float16:
        sd, bd = dev(s), dev(b)
        W = oracle.affine_dequant(codes, s.view(np.uint16), b.view(np.uint16), N, K, bits, group)
    else:  # the same values rounded to bf16: W = s q + b from the exact codes
        sd, bd = dev(s).to(sdt), dev(b).to(sdt)
        q = oracle.affine_dequant(codes, np.full(s.shape, 0x3C00, np.uint16), np.zeros(s.shape, np.uint16), N, K, bits, group)
        W = q * np.repeat(sd.float().cpu().numpy(), group, 1) + np.repeat(bd.float().cpu().numpy(), group, 1)
    y = affine.linear_rows(x, dev(codes.view(np.int32)), sd, bd, group_size=group, bits=bits)
    assert y is not None and y.dtype == dt and y.shape == (M, N)
    W = W.astype(np.float64)
    check(y, xf @ W.T, np.abs(xf) @ np.abs(W).T, dt, f"affine rows bits={bits} M={M} N={N} K={K}")


def test_affine_rows_match_the_verify_calls():
    """The rotated forward of 40 rows equals the calls of 16 rows up to the rounding of the output."""
    N, K = 300, 1024
    codes, s, b = synth.affine_pack(N, K, group=64, seed=4)
    args = (dev(codes.view(np.int32)), dev(s), dev(b))
    x, _ = act(40, K, 5, torch.float16)
    kw = dict(signs=torch.from_numpy(synth.hadamard_signs(K, seed=3)), block=128, group_size=64, bits=2)
    y = affine.linear_rows(x, *args, **kw).float()
    ref = torch.cat([affine.linear(x[r:r + 16], *args, **kw) for r in range(0, 40, 16)]).float()
    assert (y - ref).abs().max() <= 2.0 ** -9 * ref.abs().max()


def test_affine_rows_declines():
    codes, s, b = synth.affine_pack_bits(32, 512, 3, group=64, seed=1)
    args = (dev(codes.view(np.int32)), dev(s), dev(b))
    x, _ = act(20, 512, 1, torch.float16)
    assert affine.linear_rows(x, *args, bits=3) is None          # odd widths
    codes, s, b = synth.affine_pack(32, 384, group=64, seed=1)
    args = (dev(codes.view(np.int32)), dev(s), dev(b))
    assert affine.linear_rows(x[:, :384], *args) is None         # K not a multiple of 256
    codes, s, b = synth.affine_pack(32, 512, group=64, seed=1)
    args = (dev(codes.view(np.int32)), dev(s), dev(b))
    assert affine.linear_rows(x.float(), *args) is None          # fp32 x


@pytest.mark.parametrize("bits2,cb,dt,M,K,N", [
    (2, 0, torch.float16, 17, 256, 128), (3, 2, torch.float16, 40, 512, 256), (4, 0, torch.float16, 129, 512, 384),
    (4, 1, torch.bfloat16, 64, 1280, 128), (4, 2, torch.float16, 31, 2048, 128), (5, 2, torch.float16, 20, 256, 256),
    (6, 0, torch.float16, 33, 512, 128), (7, 2, torch.bfloat16, 20, 512, 128), (8, 1, torch.float16, 300, 768, 128),
    (10, 0, torch.float16, 17, 512, 128), (12, 2, torch.float16, 17, 512, 128), (14, 1, torch.float16, 17, 512, 128),
    (16, 0, torch.bfloat16, 130, 512, 256),
    # eight row tiles a workgroup and K in parts of uneven length (2 of 11 steps, 5 of 21)
    (4, 0, torch.float16, 129, 2816, 256), (8, 2, torch.bfloat16, 129, 2816, 128), (4, 1, torch.float16, 70, 5376, 256),
    (4, 2, torch.bfloat16, 70, 5376, 256)])
def test_exl3_rows(bits2, cb, dt, M, K, N):
    print(f"exl3 rows bits2={bits2} cb={cb} M={M} K={K} N={N} {dt}", flush=True)
    tr, suh, svh = synth.exl3_pack(K, N, bits2=bits2, seed=bits2 + M)
    t = exl3.EXL3Tensor(dev(tr), dev(suh), dev(svh), codebook=cb)
    x, xf = act(M, K, M + K, dt)
    y = exl3.apply_rows(x, t)
    assert y is not None and y.dtype == dt and y.shape == (M, N)
    W = oracle.exl3_dequant(tr, bits2, cb).astype(np.float64)
    xr = oracle.hadamard(xf * suh.astype(np.float32), 128)
    xr = torch.from_numpy(xr).to(dt).float().numpy()
    ref = oracle.hadamard((xr.astype(np.float64) @ W).astype(np.float32), 128) * svh.astype(np.float32)
    bh = np.abs(xr).astype(np.float64) @ np.abs(W)
    bound = np.repeat(bh.reshape(M, N // 128, 128).sum(2), 128, 1) / np.sqrt(128.0) * np.abs(svh.astype(np.float64))
    # one rounding of a rotated value to x's dtype may go the other way (fp32 butterfly order)
    check(y, ref, bound * (40 if dt == torch.bfloat16 else 5), dt, f"exl3 rows bits2={bits2} cb={cb} M={M}")


def test_rows_decline_what_lds_loads_cannot_read():
    """The many-row kernels read weights 16 bytes at a time straight into LDS (scales 4): other alignments are
    declined before any launch, and PackedLinear takes the calls of 16 rows."""
    N, K = 64, 512
    codes, s, b = synth.affine_pack(N, K, group=64, seed=1)
    x, _ = act(20, K, 1, torch.float16)
    c, sd, bd = dev(codes.view(np.int32)), dev(s), dev(b)
    off = torch.zeros(c.numel() + 1, dtype=torch.int32, device=DEV)[1:].view_as(c)
    assert affine.linear_rows(x, off, sd, bd) is None
    off = torch.zeros(sd.numel() + 1, dtype=torch.float16, device=DEV)[1:].view_as(sd)
    assert affine.linear_rows(x, c, off, bd) is None and affine.linear_rows(x, c, sd, off) is None
    tr, suh, svh = synth.exl3_pack(K, 128, bits2=4, seed=2)
    t = exl3.EXL3Tensor(dev(tr), dev(suh), dev(svh))
    t.trellis = torch.zeros(t.trellis.numel() + 2, dtype=torch.int16, device=DEV)[2:].view_as(t.trellis)
    assert exl3.apply_rows(x, t) is None


def test_packed_linear_in_blocks_of_rows():
    """More than 4096 rows go in blocks; the rows are independent, so they equal a call of their own."""
    from ishizuki_amd.linear import PackedLinear
    N, K = 32, 256
    codes, s, b = synth.affine_pack(N, K, group=64, seed=1)
    lin = PackedLinear(dev(codes.view(np.int32)), dev(s), dev(b), group_size=64, bits=2)
    x, _ = act(4100, K, 1, torch.float16)
    y = lin(x)
    assert y.shape == (4100, N)
    assert torch.equal(y[4096:], lin(x[4000:])[96:]) and torch.equal(y[:64], lin(x[:64]))


@pytest.mark.parametrize("kind,M", [("affine", 1_500_017), ("exl3", 2_100_001)])
def test_more_rows_than_a_32_bit_tile_product(kind, M):
    """Row tile times row block passes 2^31 from 1.48 million rows (four row tiles a workgroup) and 2.1 million
    (eight): every row equals the same row of a smaller call."""
    K = 256
    if kind == "affine":
        codes, s, b = synth.affine_pack(16, K, group=64, seed=1)
        args = (dev(codes.view(np.int32)), dev(s), dev(b))
        call = lambda x: affine.linear_rows(x, *args)
    else:
        t = exl3.EXL3Tensor(*(dev(a) for a in synth.exl3_pack(K, 128, bits2=2, seed=2)))
        call = lambda x: exl3.apply_rows(x, t)
    print(f"rows {kind} M={M}", flush=True)
    x = torch.randn(M, K, dtype=torch.float16, device=DEV, generator=torch.Generator(DEV).manual_seed(M))
    y, step = call(x), 1 << 18
    for r in range(0, M, step):
        assert torch.equal(y[r:r + step], call(x[r:r + step])), r
    torch.cuda.empty_cache()
