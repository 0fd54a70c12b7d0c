"""Where `linear_bf16` sends operands (CPU: a library that notes its launches stands for the GPU's, torch's own product runs for the vendor's)."""
import ctypes

import pytest
import torch

from xinfer_amd import kernels


class _Noted:
    """The kernel library with its products' launches noted and not made."""

    def __init__(self, real, launches):
        self.real, self.launches = real, launches

    def __getattr__(self, name):
        if name not in ("xi_linear_tile", "xi_linear_mid", "xi_linear_skinny", "xi_linear_thin"):
            return getattr(self.real, name)

        def launch(*args):
            self.launches.append((name, [a.value if isinstance(a, ctypes.c_void_p) else a for a in args]))
            return 0
        return launch


@pytest.fixture
def launches(monkeypatch):
    noted = []
    real = kernels.lib()
    monkeypatch.setattr(kernels, "lib", lambda: _Noted(real, noted))
    monkeypatch.setattr(kernels, "_dev", lambda *a: None)
    monkeypatch.setattr(kernels, "_stream", lambda: ctypes.c_void_p(0))
    return noted


def _rows(*shape):
    g = torch.Generator().manual_seed(len(shape))
    return torch.randn(*shape, generator=g).to(torch.bfloat16)


@pytest.mark.parametrize("M", [17, 64, 65, 128, 129, 256, 300, 1025])
@pytest.mark.parametrize("x_shape,w_shape", [((64,), (1024, 64, 2)), ((64,), (1024, 64, 1)), ((64,), (1024, 64, 0)), ((64,), (64,)), ((64,), (0, 64)),
                                             ((0,), (1024, 0)), ((128,), (1024, 64)), ((64, 64), (1024, 64))])
def test_operands_that_are_no_product_of_the_tiles(launches, M, x_shape, w_shape):
    """A weight of one or three dimensions, empty sizes, lengths that do not match, x of three dimensions: the library's answer or its refusal, and
    no kernel of tiles is launched."""
    x, w = _rows(M, *x_shape), _rows(*w_shape)
    try:
        want = torch.nn.functional.linear(x, w)
    except (RuntimeError, IndexError):
        want = None
    if want is None:
        with pytest.raises((RuntimeError, IndexError)):
            kernels.linear_bf16(x, w)
    else:
        assert torch.equal(kernels.linear_bf16(x, w), want)
    assert not launches


@pytest.mark.parametrize("M,asked,kernel", [(17, 64, "xi_linear_skinny"), (64, 64, "xi_linear_skinny"), (48, 48, "xi_linear_skinny"), (32, 17, "xi_linear_tile"),
                                            (32, None, "xi_linear_tile"), (65, 100, "xi_linear_tile")])
def test_rows_for_the_streaming_kernel(launches, M, asked, kernel):
    """`skinny_rows` is a caller's choice, up to the 64 rows that the streaming kernel takes: what is whole goes there up to that many."""
    x, w = _rows(M, 1024), _rows(4096, 1024)
    kernels.linear_bf16(x, w, **({} if asked is None else {"skinny_rows": asked}))
    assert [name for name, _ in launches] == [kernel]
