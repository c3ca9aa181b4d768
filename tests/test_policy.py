"""Host-side dispatch policy (no GPU): the row-count thresholds measured on MI355X, and workspace sizes."""
import pytest

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
