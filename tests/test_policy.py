"""Host-side dispatch policy (no GPU): the row-count thresholds measured on MI355X, and workspace sizes."""
import pytest
import torch

from ishizuki_amd import _lib, affine, ggml


def test_minimum_rows_is_two_at_every_size():
    # VerifyMatmul.minimumRows re-measured: one M-row verify call beats M GEMVs from M = 2
    for nbytes in (1_000, 1_638_400, 9_830_400, 27_852_800, 397_312_000):
        assert affine.minimum_rows(nbytes) == 2


def test_dense_from_rows():
    assert ggml.dense_from_rows(2_949_120) == 32
    assert ggml.dense_from_rows(73_728_000) == 48
    assert ggml.dense_from_rows(10_000_000) == 48


@pytest.mark.parametrize("N,K", [(5120, 25600), (7000, 8192), (1024, 8192), (2048, 32768), (17408, 5120), (100, 256)])
@pytest.mark.parametrize("t", ggml.SUPPORTED)
def test_ggml_workspace_serves_fewer_rows(t, N, K):
    """One workspace for up to 16 rows splits K for fewer rows as their own would: the size never falls with
    the rows, and past the activation image never below what a kernel for fewer rows asks for."""
    L = _lib.lib()
    size = [L.ishz_ggml_workspace_size(t, M, K, N) for M in range(1, 17)]
    image = [(2 * M * K + 255) // 256 * 256 for M in range(1, 17)]
    parts = [s - i for s, i in zip(size, image)]
    assert size == sorted(size)
    assert parts[1:4] == sorted(parts[1:4]) and max(parts[:4]) <= min(parts[4:])


H, B, F = torch.float16, torch.bfloat16, torch.float32


@pytest.mark.parametrize("t,N,K,dt,first", [
    # long rows of large weights: later, by format and size
    (ggml.Q4_K, 5120, 25600, H, 96), (ggml.IQ2_XS, 5120, 25600, B, 96), (ggml.Q6_K, 5120, 25600, H, 81),
    (ggml.Q4_0, 5120, 25600, B, 81), (ggml.Q4_K, 4096, 17408, H, 65), (ggml.Q6_K, 4096, 17408, H, 48),
    # IQ1_M, fp32 x, small weights and other proportions: by bytes alone
    (ggml.IQ1_M, 5120, 25600, H, 48), (ggml.Q4_K, 5120, 25600, F, 48), (ggml.Q4_K, 2560, 10240, H, 48),
    (ggml.Q4_K, 1024, 4096, H, 32), (ggml.Q4_K, 17408, 5120, H, 48), (ggml.Q4_K, 1024, 65536, H, 48),
    (ggml.Q4_0, 1024, 5120, B, 32)])
def test_apply_follows_dense_from_rows(monkeypatch, t, N, K, dt, first):
    """16-row calls up to the row before the line, one expansion from it on."""
    calls = []

    def matvec(x, blocks, type_, n):
        calls.append("rows")
        return x.new_empty(x.shape[0], n)

    def dequantize(blocks, type_, shape, dtype):
        calls.append("dense")
        return torch.empty(1, dtype=dtype).expand(K, N).t()
    monkeypatch.setattr(ggml, "matvec", matvec)
    monkeypatch.setattr(ggml, "dequantize", dequantize)
    monkeypatch.setattr(torch.Tensor, "__matmul__", lambda x, w: x.new_empty(x.shape[0], w.shape[1]))
    blocks = torch.empty(N * ggml.row_bytes(t, K), dtype=torch.uint8, device="meta")
    assert ggml.dense_from_rows(blocks.numel(), t, N, K, dt) == first
    for rows, want in ((17, ["rows"] * 2), (first - 1, ["rows"] * ((first + 14) // 16)), (first, ["dense"])):
        calls.clear()
        assert ggml.apply(torch.empty(rows, K, dtype=dt, device="meta"), blocks, t, N).shape == (rows, N)
        assert calls == want
