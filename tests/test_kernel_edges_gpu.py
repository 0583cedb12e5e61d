"""Kernels and branches of dispatches at the sizes where they can go wrong: edges of tiles, remainders, the smallest and the
largest of their ranges, each against the same operation in float64."""
import pytest
import torch

from rbitnet_amd.csrc.lib import kernels

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


@pytest.fixture(scope="module")
def lib():
    return kernels()


def _within(got, want, bound):
    """Every number of `got` is within `bound` (a tensor of the same shape, or a number) of `want`."""
    off = (got.double().cpu() - want.cpu()).abs()
    assert torch.isfinite(got).all()
    assert (off <= (bound.cpu() if torch.is_tensor(bound) else bound)).all(), float(off.max())


# ---------------------------------------------------------------- float32 products of many tokens
@pytest.mark.parametrize("m", [17, 64, 65, 127, 129, 257])
@pytest.mark.parametrize("n,k", [(1, 32), (63, 64), (65, 96), (130, 160), (300, 32), (16, 128), (80, 128), (144, 256), (272, 384)])
def test_float32_tiles(lib, m, n, k):
    g = torch.Generator().manual_seed(m * 31 + n + k)
    a, w = torch.randn(m, k, generator=g), torch.randn(n, k, generator=g)
    want = a.double() @ w.double().T
    # K products of 24 bits each, summed one after another: K 2^-24 of the sum of the absolute products at the most
    bound = k * 2.0 ** -24 * (a.double().abs() @ w.double().abs().T) + 1e-30
    layouts = [False] + ([True] if n % 16 == 0 and k % 128 == 0 else [])
    ad, wd = a.to(DEV), w.to(DEV)
    for frag in layouts:
        wl = wd
        if frag:
            wl = torch.empty_like(wd)
            lib.place_rows(wd, wl, frag=True)
        c = torch.full((m, n), float("nan"), device=DEV)
        lib.gemm_generic(ad, wl, c, w_frag=frag)
        _within(c, want, bound)


@pytest.mark.parametrize("m,n,k", [(70, 40, 64), (200, 130, 96)])
def test_float32_tiles_of_operands_at_odd_addresses(lib, m, n, k):
    """Operands that do not start at a multiple of 16 bytes take the kernels that do not ask for it."""
    a, w = torch.randn(m * k + 1, device=DEV)[1:].view(m, k), torch.randn(n * k + 1, device=DEV)[1:].view(n, k)
    c = torch.full((m, n), float("nan"), device=DEV)
    lib.gemm_generic(a, w, c)
    _within(c, a.double() @ w.double().T, k * 2.0 ** -24 * (a.double().abs() @ w.double().abs().T))
