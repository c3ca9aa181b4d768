"""What the Python calls pass to the library, and what they refuse before any launch (no GPU: the library is a
recorder)."""
import pytest
import torch

from ishizuki_amd import _lib, affine, exl3
from ishizuki_amd.linear import PackedLinear


class Recorder:
    """Stands in for the library: every call but the `declined` ones succeeds; all are listed."""

    def __init__(self):
        self.calls, self.args, self.declined = [], [], ()

    def __getattr__(self, name):
        def call(*args):
            if name.endswith("_size"):
                return 256
            self.calls.append(name)
            self.args.append(args)
            return _lib.DECLINED if name in self.declined else _lib.OK
        return call


@pytest.fixture
def library(monkeypatch):
    lib = Recorder()
    monkeypatch.setattr(_lib, "lib", lambda: lib)
    for m in (affine, exl3):
        monkeypatch.setattr(m, "require_cuda", lambda *ts: None)
        monkeypatch.setattr(m, "stream", lambda: None)
    return lib


def exl3_tensor(K=512, N=128):
    return exl3.EXL3Tensor(torch.zeros(K // 16, N // 16, 32, dtype=torch.int16), torch.ones(K), torch.ones(N))


def pack(N=8, K=512, bits=2):
    return (torch.zeros(N, K * bits // 32, dtype=torch.int32), torch.ones(N, K // 64, dtype=torch.float16),
            torch.zeros(N, K // 64, dtype=torch.float16))


@pytest.mark.parametrize("rows", [3, 20, 5000])
@pytest.mark.parametrize("width", [256, 384, 500, 640, 1024])
def test_exl3(library, rows, width):
    t = exl3_tensor()
    x = torch.zeros(rows, width, dtype=torch.float16)
    with pytest.raises(RuntimeError):
        PackedLinear.from_exl3(t)(x)
    with pytest.raises(RuntimeError):
        exl3.apply_rows(x, t)
    with pytest.raises(RuntimeError):
        exl3.matvec(x, t)
    if rows > 16:
        assert library.calls == []


@pytest.mark.parametrize("rows", [1, 3, 20, 5000])
@pytest.mark.parametrize("width", [256, 384, 640, 1024])
@pytest.mark.parametrize("bits", [2, 4])
def test_affine(library, rows, width, bits):
    p = pack(bits=bits)
    x = torch.zeros(rows, width, dtype=torch.float16)
    with pytest.raises(RuntimeError):
        PackedLinear(*p, group_size=64, bits=bits)(x)
    for f in (affine.linear_rows, affine.linear, affine.quantized_matmul):
        with pytest.raises(RuntimeError):
            f(x, *p, group_size=64, bits=bits)
    assert library.calls == []


def test_the_right_width_is_launched(library):
    x = torch.zeros(20, 512, dtype=torch.float16)
    assert PackedLinear.from_exl3(exl3_tensor())(x).shape == (20, 128)
    assert PackedLinear(*pack(), group_size=64)(x).shape == (20, 8)
    assert PackedLinear(*pack(), group_size=64)(x[:5]).shape == (5, 8)
    assert library.calls == ["ishz_exl3_apply_rows", "ishz_affine_linear_rows", "ishz_affine_linear"]


def test_what_the_library_declines_is_left_to_it(library):
    """Dtypes, groups and widths it refuses reach it whatever the pack's width: the answer stays None."""
    w, s, b = pack(K=1024)
    x = torch.zeros(1, 512, dtype=torch.float16)
    for kw, xx in (({"group_size": 48}, x), ({"group_size": 64}, x.to(torch.int16)), ({"group_size": 64}, x[:, :500])):
        affine.quantized_matmul(xx, w, s, b, **kw)
    assert library.calls == ["ishz_affine_matmul"] * 3


@pytest.mark.parametrize("dt,M,block,needed", [(torch.float16, 1, 0, False), (torch.float16, 4, 0, False), (torch.bfloat16, 1, 0, False),
                                               (torch.bfloat16, 2, 0, True), (torch.bfloat16, 16, 0, True), (torch.float32, 4, 0, False),
                                               (torch.bfloat16, 1, 128, True), (torch.float32, 1, 128, True)])
def test_affine_linear_workspace(library, dt, M, block, needed):
    """The rotated rows and the image of two and more bf16 rows take a workspace; nothing else asks for one."""
    affine.linear(torch.zeros(M, 512, dtype=dt), *pack(bits=4), signs=torch.ones(512), block=block, bits=4)
    assert (library.args[0][-3] is not None) == needed and (library.args[0][-2] > 0) == needed


def test_declined_prompts_allocate_nothing(library):
    """fp32 x, odd widths, other groups and K the many-row kernels do not take: no output and no workspace is made."""
    library.declined = ("ishz_affine_linear_rows", "ishz_exl3_apply_rows")
    x = torch.zeros(20, 512, dtype=torch.float16)
    grouped = tuple(t.repeat_interleave(2, 1) if t.dtype == torch.float16 else t for t in pack())  # groups of 32
    narrow = torch.zeros(20, 384, dtype=torch.float16)
    assert affine.linear_rows(x.float(), *pack()) is None
    assert affine.linear_rows(x, *pack(bits=3), bits=3) is None
    assert affine.linear_rows(x, *grouped, group_size=32) is None
    assert affine.linear_rows(narrow, *pack(K=384)) is None
    assert exl3.apply_rows(x.float(), exl3_tensor()) is None
    assert exl3.apply_rows(narrow, exl3_tensor(K=384)) is None
    for args in library.args:
        assert args[-4:-1] == (None, None, 0)


def test_a_declined_prompt_is_asked_once(library):
    library.declined = ("ishz_affine_linear_rows",)
    x = torch.zeros(9000, 512, dtype=torch.float32)
    assert PackedLinear(*pack(), group_size=64)(x).shape == (9000, 8)
    assert library.calls == ["ishz_affine_linear_rows"] + ["ishz_affine_linear"] * 563
