"""Kernels and branches of dispatches at the sizes where they can go wrong: edges of tiles, remainders, the smallest and the
largest of their ranges, each against the same operation in float64."""
from types import SimpleNamespace

import pytest
import torch

from rbitnet_amd.cache import Cache
from rbitnet_amd.config.spec import PartSpec
from rbitnet_amd.csrc.lib import kernels
from rbitnet_amd.engine.context import StepBatch, StepContext
from rbitnet_amd.errors import KernelError
from rbitnet_amd.parts.base import BuildEnv, build_part

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


def _least_time(run, rounds=7, calls=8):
    times = []
    for _ in range(rounds):
        begin, end = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
        begin.record()
        for _ in range(calls):
            run()
        end.record()
        end.synchronize()
        times.append(begin.elapsed_time(end) / calls)
    return min(times)


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


# ---------------------------------------------------------------- tiles of eight waves that take turns
@pytest.mark.parametrize("tile", [4, 5, 6, 8, 9, 11])
@pytest.mark.parametrize("m,n,k", [(130, 208, 64), (257, 400, 128), (70, 272, 192), (300, 1000, 320), (259, 521, 448)])
def test_turn_taking_tiles(lib, tile, m, n, k):
    """One K tile, two, odd numbers of them; row and token counts that end inside a tile, a wave's share and a piece of 16; rows that
    begin at whole vectors and not; float32 and bfloat16 outputs, an activation on the way out, W as rows and
    fragment-major (N a multiple of 16 only)."""
    g = torch.Generator().manual_seed(1000 * tile + m + n + k)
    a, w = torch.randn(m, k, generator=g).bfloat16(), (torch.randn(n, k, generator=g) * k ** -0.5).bfloat16()
    want, size = a.double() @ w.double().T, a.double().abs() @ w.double().abs().T
    sums = 2.0 ** -24 * k * size                           # products of bfloat16 are exact in float32: the sums' rounding, K of them
    half = 2.0 ** -8                                       # and bfloat16's where the output is that
    ad, wd = a.to(DEV), w.to(DEV)
    layouts = [(wd, False)]
    if n % 16 == 0:
        wf = torch.empty_like(wd)
        lib.place_rows(wd, wf, frag=True)
        layouts.append((wf, True))
    relu2 = torch.tensor([float("nan"), 1.0], device=DEV)
    try:
        lib._lib.rb_tune_tiles(tile, 1)
        got = []
        for weights, frag in layouts:
            for offset in (0, 1):                          # an output whose first element lies at an odd place
                for dtype, act in ((torch.float32, None), (torch.bfloat16, None), (torch.bfloat16, relu2), (torch.float32, relu2)):
                    room = torch.full((m * n + 1,), float("nan"), device=DEV, dtype=dtype)
                    c = room[offset:offset + m * n].view(m, n)
                    lib.gemm_bf16(ad, weights, c, 0, w_frag=frag, act=act)
                    exact = want if act is None else want.clamp(min=0) ** 2
                    slack = sums if act is None else 2 * want.abs() * sums + sums ** 2 + 2.0 ** -23 * exact
                    if dtype == torch.bfloat16:
                        slack = slack + half * (exact.abs() + slack)
                    assert ((c.double().cpu() - exact).abs() <= slack).all(), (frag, offset, dtype, act is not None)
                    got.append(c.cpu())
        for other in got[8:]:                              # either layout: the same bits
            assert any(torch.equal(other, first) for first in got[:8])
    finally:
        lib._lib.rb_tune_tiles(0, 0)


@pytest.mark.parametrize("tile", [4, 5, 6, 7, 8, 9, 10, 11, 13])
@pytest.mark.parametrize("m,n,k", [(70, 224, 128), (130, 416, 64), (259, 992, 320), (300, 1376, 384)])
@pytest.mark.parametrize("limits", [None, (1.5, 1.702)])
def test_gated_tiles(lib, tile, m, n, k, limits):
    """Gated pairs for row counts that are multiples of 32 and fill no tile (with three pieces a half a pair's rows lie in two halves),
    W as rows and fragment-major, outputs that begin at whole vectors and not, the plain gate and the one with limits."""
    if tile == 13 and k % 128:
        pytest.skip("K tiles of 128")
    g = torch.Generator().manual_seed(100 * tile + m)
    a, w = torch.randn(m, k, generator=g).bfloat16(), (torch.randn(n, k, generator=g) * 2 * k ** -0.5).bfloat16()
    sums, size = a.double() @ w.double().T, a.double().abs() @ w.double().abs().T
    gate, up = (sums.view(m, n // 32, 2, 16)[:, :, i].reshape(m, n // 2) for i in (0, 1))
    off = 2.0 ** -24 * k * size.view(m, n // 32, 2, 16).amax(2).reshape(m, n // 2)      # the sums' rounding, either of a pair
    act = None
    if limits is None:
        exact = gate * torch.sigmoid(gate) * up
        slack = 1.1 * off * up.abs() + off * gate.abs() + 1.1 * off * off               # |silu'| <= 1.1, |silu(x)| <= |x|
    else:
        act = torch.tensor(limits, device=DEV)
        lim, alpha = (float(x) for x in act.cpu())
        cut, moved = gate.clamp(max=lim), up.clamp(-lim, lim) + 1
        exact = cut * torch.sigmoid(alpha * cut) * moved
        slack = 1.1 * off * moved.abs() + off * cut.abs() + 1.1 * off * off             # g sigmoid(alpha g) has the same slopes
    slack = slack + 2.0 ** -20 * exact.abs()               # the hardware's exponential and reciprocal, 1 ulp each
    ad, wd = a.to(DEV), w.to(DEV)
    wf = torch.empty_like(wd)
    lib.place_rows(wd, wf, frag=True)
    try:
        lib._lib.rb_tune_tiles(tile, 1)
        for weights, frag in ((wd, False), (wf, True)):
            for offset in (0, 1):
                for dtype in (torch.float32, torch.bfloat16):
                    room = torch.full((m * n // 2 + 1,), float("nan"), device=DEV, dtype=dtype)
                    c = room[offset:offset + m * n // 2].view(m, n // 2)
                    lib.gemm_bf16(ad, weights, c, 1, w_frag=frag, act=act)
                    bound = slack if dtype == torch.float32 else slack + 2.0 ** -8 * (exact.abs() + slack)
                    _within(c, exact, bound)
    finally:
        lib._lib.rb_tune_tiles(0, 0)


@pytest.mark.parametrize("m,n,k,gated", [(256, 2176, 2048, False), (250, 2160, 2048, False), (250, 2155, 2048, False), (256, 2112, 2048, True)])
def test_products_in_two_launches(lib, m, n, k, gated):
    """Whole rounds of a large tile (of 8 compute units, for small operands) and the rows that are left: the bits of one launch of the
    large tile, or within what float32 sums in another order differ by where the rest's MFMAs are other ones.  (K is long enough for
    a second launch to be worth its price by the planner's estimate, which counts both launches' own; the bound goes with K.)"""
    g = torch.Generator().manual_seed(m + n)
    a, w = torch.randn(m, k, generator=g).bfloat16().to(DEV), (torch.randn(n, k, generator=g) * 0.05).bfloat16().to(DEV)
    layouts = [(w, False)]
    if n % 16 == 0:
        wf = torch.empty_like(w)
        lib.place_rows(w, wf, frag=True)
        layouts.append((wf, True))
    size = a.double().abs() @ w.double().abs().T
    cols = n // 2 if gated else n
    if gated:
        size = size.view(m, n // 32, 2, 16).amax(2).reshape(m, cols)
    dtypes = (torch.float32, torch.bfloat16)
    try:
        for weights, frag in layouts:
            for dtype in dtypes:
                c, whole = (torch.full((m, cols), float("nan"), device=DEV, dtype=dtype) for _ in range(2))
                lib._lib.rb_tune_tiles(4, 1)
                lib.gemm_bf16(a, weights, whole, int(gated), w_frag=frag)
                lib._lib.rb_tune_tiles(0, 0)
                lib._lib.rb_tune_compute_units(8)
                assert lib._lib.rb_tune_plan(m, n, k, int(gated)) >= 10000
                lib.gemm_bf16(a, weights, c, int(gated), w_frag=frag)
                lib._lib.rb_tune_compute_units(0)
                assert torch.equal(c[:, :1024], whole[:, :1024])
                bound = 2 * k * 2.0 ** -24 * size
                if gated:                                  # both factors move: |silu'| <= 1.1, |silu(x)| <= |x|
                    bound = 3 * bound * (1 + size)
                if dtype == torch.bfloat16:
                    bound = bound + 2.0 ** -7 * whole.double().abs()
                _within(c, whole.double(), bound)
    finally:
        lib._lib.rb_tune_tiles(0, 0)
        lib._lib.rb_tune_compute_units(0)


def test_planner_prices_slices_by_who_adds_them_up(lib):
    """A product that is not cut into slices for a kernel that reads its terms is not cut for itself, whatever the sizes and the
    machine (its launch has no workspace then); and where a launch of its own would add two slices up for more than they save, it is one."""
    import random
    rng = random.Random(5)
    try:
        for units in (8, 64, 256, 304):
            lib._lib.rb_tune_compute_units(units)
            for _ in range(3000):
                m, n, k = int(2 ** rng.uniform(4.1, 13.5)), 16 * int(2 ** rng.uniform(2, 13)), 64 * int(2 ** rng.uniform(0, 8.2))
                parts = int(lib._lib.rb_gemm_workspace_floats(m, n, k, 0)) / (m * n)
                assert parts == 0 or lib.gemm_bf16_terms_count(m, n, k) > 1, (units, m, n, k, parts)
    finally:
        lib._lib.rb_tune_compute_units(0)


@pytest.mark.parametrize("m,n,k", [(700, 3072, 2048), (850, 3072, 2048), (1286, 2048, 2048), (512, 1024, 1024)])
def test_planner_of_products_that_add_up_their_slices(lib, m, n, k):
    """The planner's choice beside every tile with 1, 2 and 4 slices forced in turn.  (Its estimate is within 5 % of the best at these
    sizes, and a time is within 3 % of itself; with the reader's price for slices it was off by 24 to 32 %.)"""
    a, c = torch.randn(m, k, device=DEV).bfloat16(), torch.empty(m, n, device=DEV)
    w = torch.empty(n, k, dtype=torch.bfloat16, device=DEV)
    lib.place_rows((torch.randn(n, k, device=DEV) * 0.02).bfloat16(), w, frag=True)
    run = lambda: lib.gemm_bf16(a, w, c, 0, w_frag=True)
    times = {}
    try:
        for cfg in (0, 4, 5, 6, 7, 8, 9, 10, 11, 13, 0):
            for parts in (1, 2, 4) if cfg else (0,):
                lib._lib.rb_tune_tiles(cfg, parts)
                graph = torch.cuda.CUDAGraph()
                run()
                torch.cuda.synchronize()
                with torch.cuda.graph(graph):
                    for _ in range(10):
                        run()
                times[cfg, parts] = min(_least_time(graph.replay, calls=3), times.get((cfg, parts), 1e9))
    finally:
        lib._lib.rb_tune_tiles(0, 0)
    assert times[0, 0] <= 1.15 * min(times.values()), (lib._lib.rb_tune_plan(m, n, k, 0), times)


@pytest.mark.parametrize("tile", [1, 2, 3, 4, 5, 6, 7])
@pytest.mark.parametrize("m,n,k", [(70, 160, 32), (131, 200, 64), (300, 333, 96), (131, 208, 128), (300, 400, 640)])
def test_float32_tiles_forced(lib, tile, m, n, k):
    """Every float32 tile: one, two, three, four and twenty K tiles, ends inside a tile, both layouts where K is a multiple of 128."""
    g = torch.Generator().manual_seed(100 * tile + m)
    a, w = torch.randn(m, k, generator=g), torch.randn(n, k, generator=g)
    want, size = a.double() @ w.double().T, a.double().abs() @ w.double().abs().T
    ad, wd = a.to(DEV), w.to(DEV)
    layouts = [(wd, False)]
    if n % 16 == 0 and k % 128 == 0:
        wf = torch.empty_like(wd)
        lib.place_rows(wd, wf, frag=True)
        layouts.append((wf, True))
    try:
        lib._lib.rb_tune_f32_tile(tile)
        for weights, frag in layouts:
            c = torch.full((m, n), float("nan"), device=DEV)
            lib.gemm_generic(ad, weights, c, w_frag=frag)
            assert ((c.double().cpu() - want).abs() <= 2.0 ** -24 * (k + 1) * size).all()
    finally:
        lib._lib.rb_tune_f32_tile(0)


@pytest.mark.parametrize("tile", [1, 2, 3, 4, 5])
@pytest.mark.parametrize("m,n,k", [(131, 200, 32), (300, 333, 160), (300, 400, 256)])
def test_float32_tiles_in_parts(lib, tile, m, n, k):
    """Tiles whose operands go as three bfloat16 parts: as close as float32 sums are, and what is not finite, or as large as
    float32 numbers get, is what the float32 product makes of it, in the places it reaches and nowhere else."""
    g = torch.Generator().manual_seed(tile + m)
    a, w = torch.randn(m, k, generator=g), torch.randn(n, k, generator=g)
    a[5, 7], a[m - 1, 3], a[100, 0] = float("inf"), float("-inf"), float("nan")
    w[:, 7], w[n - 3, 11] = 1.0, float("inf")
    a[:, 11] = a[:, 11].abs()
    a[17], a[40], w[77, 9] = 0.0, 0.0, 1.0
    a[17, 20], a[40, 9] = 3e38, 3.3999e38                  # the nearest bfloat16 to the latter is infinite
    exact = (a.double()[:, None] * w.double()[None]).sum(-1)
    want = exact.float()
    size = (a.double().abs()[:, None] * w.double().abs()[None]).sum(-1)
    ad, wd = a.to(DEV), w.to(DEV)
    layouts = [(wd, False)]
    if n % 16 == 0 and k % 128 == 0:
        wf = torch.empty_like(wd)
        lib.place_rows(wd, wf, frag=True)
        layouts.append((wf, True))
    try:
        lib._lib.rb_tune_f32_tile(tile)
        for weights, frag in layouts:
            c = torch.full((m, n), 7.0, device=DEV)
            lib.gemm_generic(ad, weights, c, w_frag=frag)
            c = c.cpu()
            finite = torch.isfinite(want)
            assert ((c.double() - exact).abs() <= 2.0 ** -24 * (k + 1) * size)[finite].all(), frag
            assert torch.equal(torch.isnan(c), torch.isnan(want)) and torch.equal(torch.isinf(c), torch.isinf(want)), frag
            assert torch.equal(torch.sign(c[torch.isinf(c)]), torch.sign(want[torch.isinf(want)])), frag
    finally:
        lib._lib.rb_tune_f32_tile(0)


def _both_layouts(lib, w):
    wf = torch.empty_like(w)
    lib.place_rows(w, wf, frag=True)
    return ((w, False), (wf, True))


@pytest.mark.parametrize("tile", [1, 2, 3, 4, 5, 6, 7])
def test_float32_tiles_hold_every_bit_of_a_product(lib, tile):
    """One depth value of a token is not zero, another one for every token, so that a result is one product and no bound grows with
    K: 12 K tiles, those whose sums are turned among them, both layouts, numbers of 24 bits and the pair whose left-out
    products of parts are largest."""
    m, n, k = 131, 208, 384
    g = torch.Generator().manual_seed(tile)
    bits = lambda *size: (torch.randint(0, 1 << 22, size, generator=g) * 2 + (1 << 23) + 1).float() * 2.0 ** -23
    a, w = torch.zeros(m, k), bits(n, k) * torch.randint(0, 2, (n, k), generator=g).mul(2).sub(1)
    at = torch.arange(m) * 3 % k
    a[torch.arange(m), at] = bits(m)
    a[7, at[7]] = a[90, at[90]] = 1.0039138793945312
    w[5, at[7]], w[6, at[90]] = 1.0039138793945312, -1.0039138793945312
    want = a.double() @ w.double().T
    # the last of six additions rounds down, 2^-23 of the result at most, the products left out are 2^-24, the other additions 2^-30 each
    bound = (2.0 ** -23 + 2.0 ** -24 + 2.0 ** -27) * want.abs()
    two = lambda x: x.bfloat16().double() + (x - x.bfloat16().float()).bfloat16().double()
    assert ((two(a) @ two(w).T - want).abs() > bound).double().mean() > 0.5          # two parts would not pass
    try:
        lib._lib.rb_tune_f32_tile(tile)
        for weights, frag in _both_layouts(lib, w.to(DEV)):
            c = torch.full((m, n), float("nan"), device=DEV)
            lib.gemm_generic(a.to(DEV), weights, c, w_frag=frag)
            _within(c, want, bound)
    finally:
        lib._lib.rb_tune_f32_tile(0)


@pytest.mark.parametrize("tile", [1, 2, 3, 4, 5, 6, 7])
@pytest.mark.parametrize("scale", [1e-30, 1e-36, 1e-40, 1e31])
def test_float32_tiles_over_the_range_of_exponents(lib, tile, scale):
    """Operands near the ends of the exponents' range, one side at a time: as close as float32 sums of them are, down to numbers
    that are subnormal."""
    m, n, k = 131, 208, 384
    g = torch.Generator().manual_seed(tile)
    for small in (0, 1):
        a, w = torch.randn(m, k, generator=g), torch.randn(n, k, generator=g)
        if small:
            a = a * scale
        else:
            w = w * scale
        want, size = a.double() @ w.double().T, a.double().abs() @ w.double().abs().T
        try:
            lib._lib.rb_tune_f32_tile(tile)
            for weights, frag in _both_layouts(lib, w.to(DEV)):
                c = torch.full((m, n), float("nan"), device=DEV)
                lib.gemm_generic(a.to(DEV), weights, c, w_frag=frag)
                _within(c, want, 2.0 ** -24 * (k + 1) * size + 2.0 ** -149)
                off = (c.double().cpu() - want).norm() / want.norm()
                # K roundings, each to 24 bits or to a subnormal's last place, are as good as independent: a tenth of what they could add up to
                assert off <= 0.1 * k * (2.0 ** -24 + 2.0 ** -149 / want.square().mean().sqrt()), (small, frag, float(off))
        finally:
            lib._lib.rb_tune_f32_tile(0)


@pytest.mark.parametrize("frag", [False, True])
def test_float32_product_with_an_undefined_token_costs_no_multiple(lib, frag):
    """A token that is no number is computed again on the float32 matrix core: about three times the product's time where every
    token is one; other tokens keep their bits."""
    m, n, k = 1000, 4096, 3072
    g = torch.Generator().manual_seed(3)
    a, w = torch.randn(m, k, generator=g).to(DEV), torch.randn(n, k, generator=g).to(DEV)
    if frag:
        rows, w = w, torch.empty_like(w)
        lib.place_rows(rows, w, frag=True)

    def run(x):
        c, times = torch.empty(m, n, device=DEV), []
        for _ in range(5):
            begin, end = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
            begin.record()
            lib.gemm_generic(x, w, c, w_frag=frag)
            end.record()
            end.synchronize()
            times.append(begin.elapsed_time(end))
        return c, min(times)

    whole, finite = run(a)
    bad = a.clone()
    bad[37, 5] = float("nan")
    c, with_one = run(bad)
    assert torch.isnan(c[37]).all()
    keep = torch.arange(m, device=DEV) != 37
    assert torch.equal(c[keep], whole[keep])
    c, with_all = run(torch.full_like(a, float("nan")))
    assert torch.isnan(c).all()
    assert with_one < 4 * finite and with_all < 8 * finite, (finite, with_one, with_all)


@pytest.mark.parametrize("m,n", [(256, 2112), (250, 2100), (256, 3600), (250, 1590), (256, 4352)])
def test_float32_product_in_two_launches(lib, m, n):
    """Whole rounds of a large tile (of 8 compute units, for small operands), and the rows that are left with another tile; 4,352 rows
    are whole rounds but for one tile and stay one launch."""
    k = 3072
    a, w = torch.randn(m, k, device=DEV), torch.randn(n, k, device=DEV)
    layouts = [(w, False)]
    if n % 16 == 0:
        wf = torch.empty_like(w)
        lib.place_rows(w, wf, frag=True)
        layouts.append((wf, True))
    try:
        lib._lib.rb_tune_compute_units(8)
        assert (lib._lib.rb_tune_f32_plan(m, n, k) >= 10) == (n != 4352)
        for weights, frag in layouts:
            c = torch.full((m, n), float("nan"), device=DEV)
            lib.gemm_generic(a, weights, c, w_frag=frag)
            _within(c, a.double() @ w.double().T, k * 2.0 ** -24 * (a.double().abs() @ w.double().abs().T))
    finally:
        lib._lib.rb_tune_compute_units(0)


@pytest.mark.parametrize("m,n,k", [(300, 16384, 512), (1286, 8192, 256), (300, 16384, 2048), (2000, 1536, 1024), (1286, 5120, 3072)])
def test_float32_planner_over_k(lib, m, n, k):
    """The planner's choice beside every tile forced in turn, at a K of its own for each size: rounds cost what K says.  (Its estimate
    is within 7 % of the best over the sizes it was fitted to; prices of one K for all were off by 12 to 19 % at the first four.)"""
    a, w, c = torch.randn(m, k, device=DEV), torch.randn(n, k, device=DEV), torch.empty(m, n, device=DEV)
    run = lambda: lib.gemm_generic(a, w, c)
    times = []
    try:
        for tile in (0, 1, 2, 3, 4, 5, 6, 7, 0):
            lib._lib.rb_tune_f32_tile(tile)
            times.append(_least_time(run))
    finally:
        lib._lib.rb_tune_f32_tile(0)
    assert min(times[0], times[-1]) <= 1.12 * min(times), (lib._lib.rb_tune_f32_plan(m, n, k), times)


@pytest.mark.parametrize("m,n,k", [(70, 40, 64), (200, 130, 96)])
def test_float32_tiles_of_operands_at_odd_addresses(lib, m, n, k):
    """Operands that do not start at a multiple of 16 bytes take the kernels that do not ask for it."""
    a, w = torch.randn(m * k + 1, device=DEV)[1:].view(m, k), torch.randn(n * k + 1, device=DEV)[1:].view(n, k)
    c = torch.full((m, n), float("nan"), device=DEV)
    lib.gemm_generic(a, w, c)
    _within(c, a.double() @ w.double().T, k * 2.0 ** -24 * (a.double().abs() @ w.double().abs().T))


# ---------------------------------------------------------------- products of few tokens that add to the stream
@pytest.mark.parametrize("m", [1, 5, 16])
@pytest.mark.parametrize("n,k", [(48, 96), (64, 128), (272, 768), (8192, 2048)])
def test_stream_products_do_not_depend_on_addresses(lib, m, n, k):
    """The stream's new rows, what the next norm takes of them and their sums of squares are the same bits where columns leave four at a
    time and one by one; a sum of squares is one of products that are not rounded, in the order of the columns."""
    g = torch.Generator().manual_seed(m + n)
    a, w = torch.randn(m, k, generator=g).bfloat16().to(DEV), (torch.randn(n, k, generator=g) * 0.02).bfloat16().to(DEV)
    c0, gain0 = torch.randn(m, n, generator=g).to(DEV), torch.randn(n, generator=g).to(DEV)
    got = []
    for off in (0, 1):
        c, gain = torch.empty(m * n + off, device=DEV)[off:].view(m, n), torch.empty(n + off, device=DEV)[off:]
        gained = torch.empty(m * n + off, dtype=torch.bfloat16, device=DEV)[off:].view(m, n)
        squares = torch.full((m, n // 16), float("nan"), device=DEV)
        c.copy_(c0)
        gain.copy_(gain0)
        lib.gemm_bf16_few(a, w, c, 3, gain=gain, gained=gained, squares_out=squares)
        got.append((c, gained, squares))
    for x, y in zip(*got):
        assert torch.equal(x, y)
    v = got[0][0].double().cpu().view(m, n // 16, 4, 4)
    four = torch.zeros(m, n // 16, 4)
    for i in range(4):                       # float64 holds the product and the sum of one fused operation but for ties of ties
        four = (four.double() + v[..., i] * v[..., i]).float()
    want = (four[..., 0] + four[..., 1]) + (four[..., 2] + four[..., 3])
    assert torch.equal(got[0][2].cpu(), want)


# ---------------------------------------------------------------- float32 attention on the matrix cores
def _paged(lengths, heads, dim, generator, spare=7):
    """Keys (or values) of sequences of these lengths in pages that are handed out in a mixed order, NaN where nothing was written."""
    need = [(n + 63) // 64 for n in lengths]
    order = torch.randperm(sum(need) + spare, generator=generator).tolist()
    pages = torch.full((sum(need) + spare, heads, 64, dim), float("nan"))
    rows, at = [], 0
    table = torch.zeros(len(lengths), max(need), dtype=torch.int32)
    for b, n in enumerate(lengths):
        mine = order[at:at + need[b]]
        at += need[b]
        table[b, :need[b]] = torch.tensor(mine, dtype=torch.int32)
        x = torch.randn(n, heads, dim, generator=generator)
        for j in range(n):
            pages[mine[j // 64], :, j % 64] = x[j]
        rows.append(x)
    return pages, table, rows


def _attention64(q, k, v, pos, scale, window=0, keep=0, cap=0.0, sinks=None, chunk=0, sig=None):
    """q [T, H, D] at positions pos [T] over k, v [N, G, D] in float64."""
    t, h, _ = q.shape
    rep = h // k.shape[1]
    s = torch.einsum("thd,nhd->htn", q.double(), k.double().repeat_interleave(rep, 1)) * scale
    if cap > 0:
        s = cap * torch.tanh(s / cap)
    i, j = pos[:, None], torch.arange(k.shape[0])[None, :]
    seen = j <= i
    if window:
        seen = seen & ((i - j < window) | (j < keep))
    if chunk:
        seen = seen & (i // chunk == j // chunk)
    if sig is not None:
        w = torch.sigmoid(s + sig.double()[:, None, None]) * seen
    else:
        s = s.masked_fill(~seen, float("-inf"))
        top = s.amax(-1, keepdim=True)
        if sinks is not None:
            top = torch.maximum(top, sinks.double()[:, None, None])
        w = torch.exp(s - top)
        w = w / (w.sum(-1, keepdim=True) + (0 if sinks is None else torch.exp(sinks.double()[:, None, None] - top)))
    return torch.einsum("htn,nhd->thd", w, v.double().repeat_interleave(rep, 1))


@pytest.mark.parametrize("heads,kv,dim", [(4, 1, 24), (3, 3, 4), (24, 8, 128), (16, 1, 64), (40, 2, 100), (6, 2, 32)])
@pytest.mark.parametrize("past,new", [([0], [1]), ([62, 0, 130, 31], [1, 1, 1, 1]), ([0, 0, 0], [5, 17, 77]), ([40, 129], [70, 3]),
                                      ([0, 500], [600, 1])])
@pytest.mark.parametrize("more", [{}, {"window": 50, "keep": 9, "cap": 3.0}, {"sinks": True, "chunk": 48}, {"sig": True, "chunk": 64}])
def test_float32_attention(lib, heads, kv, dim, past, new, more):
    g = torch.Generator().manual_seed(heads * 7 + dim + len(past) + sum(new))
    more = dict(more)
    lengths = [p + n for p, n in zip(past, new)]
    kp, table, ks = _paged(lengths, kv, dim, g)
    vp, vs = torch.full_like(kp, float("nan")), []
    for b, n in enumerate(lengths):
        x = torch.randn(n, kv, dim, generator=g)
        for j in range(n):
            vp[table[b, j // 64], :, j % 64] = x[j]
        vs.append(x)
    q = torch.randn(sum(new), heads, dim, generator=g)
    pos = torch.cat([torch.arange(p, p + n) for p, n in zip(past, new)])
    seq = torch.repeat_interleave(torch.arange(len(new)), torch.tensor(new))
    for name in ("sinks", "sig"):
        if more.get(name):
            more[name] = torch.randn(heads, generator=g)
    scale = dim ** -0.5
    want = torch.cat([_attention64(q[seq == b], ks[b], vs[b], pos[seq == b], scale, **more) for b in range(len(new))])
    out = torch.full((sum(new), heads * dim), float("nan"), device=DEV)
    i32 = lambda x: x.to(torch.int32).to(DEV)
    dev = lambda x: None if x is None else x.to(DEV)
    lib.attention_opts(q.to(DEV), kp.to(DEV), vp.to(DEV), out, i32(pos), i32(seq), table.to(DEV), heads, kv, dim, scale,
                       more.get("window", 0), more.get("keep", 0), more.get("cap", 0.0), dev(more.get("sinks")), more.get("chunk", 0),
                       dev(more.get("sig")))
    # scores are sums of `dim` products of a few units: their error, at most dim 2^-24 of the sum of absolute products, moves a
    # weight by as much relatively, and the outputs are sums of weights times values of a few units
    _within(out.view(want.shape), want, 64 * 2.0 ** -24 * max(4.0, float(want.abs().max())) * 4)


@pytest.mark.parametrize("heads,kv,dim", [(8, 8, 32), (6, 2, 32), (12, 4, 64), (24, 8, 128), (5, 5, 100)])
@pytest.mark.parametrize("past,new", [([0, 40, 130, 0], [301, 7, 2, 303]), ([70, 3, 0], [1, 1, 1]), ([0], [90])])
@pytest.mark.parametrize("more", [{}, {"window": 50, "keep": 9}, {"sig": True, "chunk": 48}])
@pytest.mark.parametrize("bad", ["none", "values", "keys"])
def test_float32_attention_keeps_tokens_apart(lib, heads, kv, dim, past, new, more, bad):
    """Blocks over the boundaries of sequences, two and three in a block; an infinite or undefined key or value comes to the queries that
    see it and to no other token's, of its sequence or the next, and an undefined value to its own number of a head alone."""
    g = torch.Generator().manual_seed(heads * 7 + dim + sum(new))
    more = dict(more)
    lengths = [p + n for p, n in zip(past, new)]
    kp, table, ks = _paged(lengths, kv, dim, g)
    vp, vs = torch.full_like(kp, float("nan")), []
    for b, n in enumerate(lengths):
        x = torch.randn(n, kv, dim, generator=g)
        for j in range(n):
            vp[table[b, j // 64], :, j % 64] = x[j]
        vs.append(x)
    where = {}                                                    # sequence -> position, kv head and number of what is not finite
    if bad != "none":
        for b, n in enumerate(lengths):
            if b % 2 == 0:
                j, head, d = max(past[b], n - 1 - n // 3), b % kv, (5 * b) % dim
                where[b] = (j, head, d)
                (vp if bad == "values" else kp)[table[b, j // 64], head, j % 64, d] = float("inf") if b else float("nan")
    q = torch.randn(sum(new), heads, dim, generator=g)
    pos = torch.cat([torch.arange(p, p + n) for p, n in zip(past, new)])
    seq = torch.repeat_interleave(torch.arange(len(new)), torch.tensor(new))
    if more.get("sig"):
        more["sig"] = torch.randn(heads, generator=g)
    scale = dim ** -0.5
    want = torch.cat([_attention64(q[seq == b], ks[b], vs[b], pos[seq == b], scale, **more) for b in range(len(new))])
    out = torch.full((sum(new), heads * dim), float("nan"), device=DEV)
    i32 = lambda x: x.to(torch.int32).to(DEV)
    lib.attention_opts(q.to(DEV), kp.to(DEV), vp.to(DEV), out, i32(pos), i32(seq), table.to(DEV), heads, kv, dim, scale,
                       more.get("window", 0), more.get("keep", 0), 0.0, None, more.get("chunk", 0),
                       None if more.get("sig") is None else more["sig"].to(DEV))
    got = out.view(want.shape).cpu()
    touched = torch.zeros(want.shape, dtype=torch.bool)           # what may differ from the result with finite keys and values
    for b, (j, head, d) in where.items():
        seen = (seq == b) & (pos >= j)
        if more.get("window"):
            seen &= (pos - j < more["window"]) | (j < more["keep"])
        if more.get("chunk"):
            seen &= pos // more["chunk"] == j // more["chunk"]
        mine = slice(head * (heads // kv), (head + 1) * (heads // kv))
        assert seen.any()
        if bad == "values":
            touched[seen, mine, d] = True
            assert not torch.isfinite(got[seen][:, mine, d]).any()
        else:
            touched[seen, mine] = True
    _within(torch.where(touched, 0.0, got), torch.where(touched, 0.0, want), 64 * 2.0 ** -24 * max(4.0, float(want.abs().max())) * 4)


@pytest.mark.parametrize("heads,kv,dim", [(8, 8, 32), (12, 4, 64), (24, 8, 128)])
@pytest.mark.parametrize("more", [{}, {"window": 50, "keep": 9}])
@pytest.mark.parametrize("order", ["falling", "mixed", "twice", "without a position"])
def test_float32_attention_of_tokens_in_any_order(lib, heads, kv, dim, more, order):
    """Every token is answered from its own position and sequence, whatever its neighbours in the step are; a token without a position
    (a negative one) sees nothing."""
    g = torch.Generator().manual_seed(heads + dim)
    lengths = [300, 90]
    kp, table, ks = _paged(lengths, kv, dim, g)
    vp, vs = torch.full_like(kp, float("nan")), []
    for b, n in enumerate(lengths):
        x = torch.randn(n, kv, dim, generator=g)
        for j in range(n):
            vp[table[b, j // 64], :, j % 64] = x[j]
        vs.append(x)
    pos, seq = torch.cat([torch.arange(n) for n in lengths]), torch.repeat_interleave(torch.arange(2), torch.tensor(lengths))
    if order == "falling":
        pos, seq = pos.flip(0), seq.flip(0)
    elif order == "mixed":
        at = torch.randperm(len(pos), generator=g)
        pos, seq = pos[at], seq[at]
    elif order == "twice":
        pos, seq = pos.repeat_interleave(2), seq.repeat_interleave(2)
    else:
        pos = torch.where(torch.rand(len(pos), generator=g) < 0.3, -1, pos)
    q = torch.randn(len(pos), heads, dim, generator=g)
    want = torch.zeros(q.shape, dtype=torch.float64)
    for b in range(2):
        at = (seq == b) & (pos >= 0)
        want[at] = _attention64(q[at], ks[b], vs[b], pos[at], dim ** -0.5, **more)
    out = torch.full((len(pos), heads * dim), float("nan"), device=DEV)
    lib.attention_opts(q.to(DEV), kp.to(DEV), vp.to(DEV), out, pos.int().to(DEV), seq.int().to(DEV), table.to(DEV), heads, kv, dim,
                       dim ** -0.5, more.get("window", 0), more.get("keep", 0), 0.0, None)
    _within(out.view(want.shape), want, 64 * 2.0 ** -24 * max(4.0, float(want.abs().max())) * 4)


@pytest.mark.parametrize("heads,kv,dim,n_splits", [(24, 8, 128, 8), (40, 2, 100, 3), (16, 1, 64, 4), (6, 2, 24, 2)])
@pytest.mark.parametrize("more", [{}, {"window": 300, "keep": 9, "cap": 3.0, "sinks": True}, {"sig": True, "chunk": 512}])
def test_float32_tokens_whose_keys_are_shared(lib, heads, kv, dim, n_splits, more):
    """Contexts in which no, some and all workgroups have keys: 8 units of 32 keys are one workgroup's, 9 two's.  The counters are zeros
    again after every launch."""
    g = torch.Generator().manual_seed(heads + dim + n_splits)
    more = dict(more)
    lengths = [1, 256, 257, 700, 2081, 64]
    kp, table, ks = _paged(lengths, kv, dim, g)
    vp, vs = torch.full_like(kp, float("nan")), []
    for b, n in enumerate(lengths):
        x = torch.randn(n, kv, dim, generator=g)
        for j in range(n):
            vp[table[b, j // 64], :, j % 64] = x[j]
        vs.append(x)
    n = len(lengths)
    q = torch.randn(n, heads, dim, generator=g)
    pos, seq = torch.tensor(lengths) - 1, torch.arange(n)
    for name in ("sinks", "sig"):
        if more.get(name):
            more[name] = torch.randn(heads, generator=g)
    want = torch.cat([_attention64(q[b:b + 1], ks[b], vs[b], pos[b:b + 1], dim ** -0.5, **more) for b in range(n)])
    i32 = lambda x: x.to(torch.int32).to(DEV)
    dev = lambda x: None if x is None else x.to(DEV)
    workspace = torch.zeros(n * heads * (1 + n_splits * (dim + 2)), device=DEV)
    args = [q.to(DEV), kp.to(DEV), vp.to(DEV), None, i32(pos), i32(seq), table.to(DEV), heads, kv, dim, dim ** -0.5, more.get("window", 0),
            more.get("keep", 0), more.get("cap", 0.0), dev(more.get("sinks")), more.get("chunk", 0), dev(more.get("sig"))]
    for _ in range(3):
        args[3] = torch.full((n, heads * dim), float("nan"), device=DEV)
        lib.attention_opts(*args, n_seqs=n, shared=(n_splits, workspace))
        _within(args[3].view(want.shape), want, 64 * 2.0 ** -24 * max(4.0, float(want.abs().max())) * 4)
        assert not workspace[:n * heads].view(torch.int32).any()
    with pytest.raises(KernelError):
        lib.attention_opts(*args, n_seqs=n, shared=(n_splits + 1, workspace))


@pytest.mark.parametrize("heads,kv,dim", [(32, 32, 128), (4, 2, 24), (24, 8, 128), (16, 16, 64)])
@pytest.mark.parametrize("past,new", [([70] * 3, [1] * 3), ([70, 3, 129, 0] * 9, [1] * 36), ([0], [6]), ([100], [40]), ([0, 9, 0], [16, 16, 16]),
                                      ([0], [130])])
def test_float32_attention_by_how_many_sequences_a_step_has(lib, heads, kv, dim, past, new):
    """Single-token steps, one prompt and several, on either side of the lines between the kernels and the splits; the count decides between
    kernels and not what is computed."""
    g = torch.Generator().manual_seed(heads + dim + sum(new))
    lengths = [p + n for p, n in zip(past, new)]
    kp, table, ks = _paged(lengths, kv, dim, g)
    vp, vs = torch.full_like(kp, float("nan")), []
    for b, n in enumerate(lengths):
        x = torch.randn(n, kv, dim, generator=g)
        for j in range(n):
            vp[table[b, j // 64], :, j % 64] = x[j]
        vs.append(x)
    q, sinks = torch.randn(sum(new), heads, dim, generator=g), torch.randn(heads, generator=g)
    pos = torch.cat([torch.arange(p, p + n) for p, n in zip(past, new)])
    seq = torch.repeat_interleave(torch.arange(len(new)), torch.tensor(new))
    want = torch.cat([_attention64(q[seq == b], ks[b], vs[b], pos[seq == b], dim ** -0.5, sinks=sinks) for b in range(len(new))])
    for n_seqs in (0, len(new)):
        for more in ({}, {"keep_first": 0, "softcap": 0.0}):
            out = torch.full((sum(new), heads * dim), float("nan"), device=DEV)
            args = [q.to(DEV), kp.to(DEV), vp.to(DEV), out, pos.int().to(DEV), seq.int().to(DEV), table.to(DEV), heads, kv, dim, dim ** -0.5, 0]
            (lib.attention_opts if more else lib.attention_sinks)(*args, *more.values(), sinks.to(DEV), n_seqs=n_seqs)
            _within(out.view(want.shape), want, 64 * 2.0 ** -24 * max(4.0, float(want.abs().max())) * 4)


@pytest.mark.parametrize("heads,kv,dim", [(24, 8, 128), (16, 4, 64), (8, 2, 32), (32, 16, 20)])
@pytest.mark.parametrize("past,new", [([0, 0], [131, 387]), ([400, 131, 300, 520, 900, 77, 30, 2000], [1] * 8), ([500], [60])])
def test_float32_attention_is_as_exact_as_on_the_vector_units(lib, heads, kv, dim, past, new):
    """The error against float64 is not larger than that of the kernel that takes the keys one by one on the vector units.  The relative
    errors of 2,000 numbers and more are random ones of the same size: their norms are known to a few hundredths."""
    g = torch.Generator().manual_seed(dim + sum(new))
    lengths = [p + n for p, n in zip(past, new)]
    kp, table, ks = _paged(lengths, kv, dim, g)
    vp, vs = torch.full_like(kp, float("nan")), []
    for b, n in enumerate(lengths):
        x = torch.randn(n, kv, dim, generator=g)
        for j in range(n):
            vp[table[b, j // 64], :, j % 64] = x[j]
        vs.append(x)
    q = torch.randn(sum(new), heads, dim, generator=g)
    pos = torch.cat([torch.arange(p, p + n) for p, n in zip(past, new)])
    seq = torch.repeat_interleave(torch.arange(len(new)), torch.tensor(new))
    want = torch.cat([_attention64(q[seq == b], ks[b], vs[b], pos[seq == b], dim ** -0.5) for b in range(len(new))])
    args = [q.to(DEV), kp.to(DEV), vp.to(DEV)], [pos.int().to(DEV), seq.int().to(DEV), table.to(DEV), heads, kv, dim, dim ** -0.5, 0, None]
    error = {}
    try:
        for mode in (1, 2):
            lib._lib.rb_tune_attention_vec(mode)
            out = torch.full((sum(new), heads * dim), float("nan"), device=DEV)
            lib.attention_sinks(*args[0], out, *args[1])
            error[mode] = float((out.view(want.shape).double().cpu() - want).norm() / want.norm())
    finally:
        lib._lib.rb_tune_attention_vec(1)
    assert error[1] <= 1.1 * error[2], error


# ---------------------------------------------------------------- products per head on the matrix cores
@pytest.mark.parametrize("tokens", [1, 4, 16, 17, 200])
@pytest.mark.parametrize("heads,k,n,more", [(1, 32, 16, {}), (3, 64, 96, {"rot": 32, "pad": 128}), (16, 128, 128, {}),
                                            (5, 96, 64, {"gate": True, "wide": 128}), (2, 128, 48, {"gate": True})])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_products_per_head(lib, tokens, heads, k, n, more, dtype):
    if dtype == torch.bfloat16 and "rot" in more:
        pytest.skip("a rotated part rides with float32 inputs")
    g = torch.Generator().manual_seed(tokens + heads + k)
    rot, x_head, y_head = more.get("rot", 0), more.get("wide", k) + more.get("rot", 0), more.get("pad", n)
    x = torch.randn(tokens, heads, x_head, generator=g).to(dtype)
    w = torch.randn(heads, n, k, generator=g).bfloat16()
    if dtype == torch.float32:                                    # a number whose rounding to bfloat16 would be an infinity
        x[0, 0, 0], w[0, :, 0] = 3.4e38, w[0, :, 0] * 0.125
    want = torch.einsum("thk,hnk->thn", x[..., :k].double(), w.double())
    size = torch.einsum("thk,hnk->thn", x[..., :k].double().abs(), w.double().abs())
    wf = torch.empty_like(w, device=DEV)
    for i in range(heads):
        lib.place_rows(w[i].to(DEV).contiguous(), wf[i], frag=True)
    y = torch.full((tokens, heads * y_head), float("nan"), dtype=torch.bfloat16, device=DEV)
    gate = torch.randn(tokens, heads + 3, generator=g)
    pos = torch.randint(0, 50, (tokens,), generator=g, dtype=torch.int32)
    angles = torch.rand(50, max(1, rot // 2), generator=g) * 6.0
    cos, sin = torch.cos(angles), torch.sin(angles)
    rope = (k, rot, cos.to(DEV), sin.to(DEV), 0, n, pos.to(DEV)) if rot else None
    lib.heads_linear_part(x.reshape(tokens, -1).to(DEV), x_head, wf, y, y_head, gate=gate.to(DEV) if "gate" in more else None,
                          gate_col=2, rope=rope, w_frag=True)
    got = y.view(tokens, heads, y_head).double().cpu()
    if "gate" in more:
        factor = torch.sigmoid(gate[:, 2:2 + heads].double())[..., None]
        want, size = want * factor, size * factor
    # the output's rounding to 8 bits, and float32 sums of exact products (three parts each)
    _within(got[..., :n], want, want.abs() * 2.0 ** -8 + size * 3 * k * 2.0 ** -24 + 1e-30)
    if rot:
        c, s = cos[pos.long()].double()[:, None], sin[pos.long()].double()[:, None]
        a, b = x[..., k:k + rot:2].double(), x[..., k + 1:k + rot:2].double()
        turned = torch.stack([a * c - b * s, b * c + a * s], -1).flatten(-2)
        _within(got[..., n:n + rot], turned, 2.0 ** -7 * (a.abs().max() + b.abs().max()))
        assert (got[..., n + rot:] == 0).all()


def test_infinite_inputs_of_products_per_head(lib):
    """An infinite or undefined input makes its own sums so and no other token's or head's."""
    x = torch.ones(20, 2, 32)
    x[3, 1, 5], x[7, 0, 1] = float("inf"), float("nan")
    w = torch.ones(2, 16, 32).bfloat16()
    wf = torch.empty_like(w, device=DEV)
    for i in range(2):
        lib.place_rows(w[i].to(DEV), wf[i], frag=True)
    y = torch.empty(20, 32, dtype=torch.bfloat16, device=DEV)
    lib.heads_linear_part(x.reshape(20, -1).to(DEV), 32, wf, y, 16, w_frag=True)
    got = y.float().cpu().view(20, 2, 16)
    assert torch.isinf(got[3, 1]).all() and torch.isnan(got[7, 0]).all()
    got[3, 1] = got[7, 0] = 32.0
    assert (got == 32.0).all()


# ---------------------------------------------------------------- experts on the dense product's tiles
@pytest.mark.parametrize("tokens,top,experts,width,ff", [(70, 1, 2, 64, 64), (150, 2, 2, 128, 192), (131, 3, 3, 64, 320), (1600, 2, 2, 64, 64)])
@pytest.mark.parametrize("gated,limit", [(True, None), (True, 1.5), (False, None)])
def test_experts_on_tiles_with_weighted_inputs(lib, tokens, top, experts, width, ff, gated, limit):
    """The router's weight counts the expert's input: runs padded to 64, 128 and 256 rows, against 64 bits."""
    g = torch.Generator().manual_seed(tokens + ff)
    r = lambda *s, f=1.0: (torch.randn(*s, generator=g) * f).bfloat16()
    h, gate, up, down = r(tokens, width), r(experts, ff, width, f=width ** -0.5 * 2), r(experts, ff, width, f=width ** -0.5 * 2), r(experts, width, ff, f=ff ** -0.5)
    z = torch.randn(tokens, experts, generator=g)
    place = lambda src, dst, *at: [lib.place_rows(src[e].to(DEV), dst[e], *at, frag=True) for e in range(experts)]
    wu, wd = torch.empty(experts, 2 * ff if gated else ff, width, dtype=torch.bfloat16, device=DEV), torch.empty(experts, width, ff, dtype=torch.bfloat16, device=DEV)
    if gated:
        place(gate, wu, 0, 16, 32)
        place(up, wu, 16, 16, 32)
    else:
        place(up, wu)
    place(down, wd)
    act = torch.tensor([float("nan"), 1.0], device=DEV) if not gated else None if limit is None else torch.tensor([limit, 1.702], device=DEV)
    for unit in (64, 128, 256):
        rows = lib.routed_rows(tokens, top, experts, unit)
        i32 = lambda n: torch.empty(n, dtype=torch.int32, device=DEV)
        sel, row_pair, tile_expert = i32(tokens * top), i32(rows), i32(2 * (rows // unit))
        weight = torch.empty(tokens * top, device=DEV)
        lib.route_choose(z.to(DEV), experts, experts, top, 0, None, sel, weight, row_pair, tile_expert, unit=unit)
        y = torch.full((rows, ff), float("nan"), dtype=torch.bfloat16, device=DEV)
        out = torch.full((tokens * top, width), float("nan"), device=DEV)
        lib.routed_experts_tiled(h.to(DEV), top, row_pair, tile_expert, unit, wu, wd, gated, act, y, out, weight)
        s, x = sel.cpu().long(), h.double().repeat_interleave(top, 0) * weight.double().cpu()[:, None]
        for e in range(experts):
            at = torch.nonzero(s == e)[:, 0]
            a, b = x[at] @ gate[e].double().T, x[at] @ up[e].double().T
            if not gated:
                u = b.clamp(min=0) ** 2
            elif limit is not None:
                a, b = a.clamp(max=limit), b.clamp(-limit, limit)
                u = a * torch.sigmoid(float(torch.tensor(1.702)) * a) * (b + 1)
            else:
                u = a * torch.sigmoid(a) * b
            # the units are rounded to 8 bits, everything else is float32
            _within(out[at], u @ down[e].double().T, (u.abs() * 2.0 ** -8 + 1e-4) @ down[e].double().abs().T)


@pytest.mark.parametrize("tokens,top,experts,width,ff", [(112, 1, 1, 64, 64), (150, 2, 2, 128, 192), (131, 3, 3, 64, 320), (1600, 2, 2, 64, 64),
                                                         (700, 4, 16, 256, 128)])
@pytest.mark.parametrize("limit", [None, 1.5])
def test_gated_experts_on_tiles(lib, tokens, top, experts, width, ff, limit):
    from rbitnet_amd.parts.routed import tile_rows
    g = torch.Generator().manual_seed(tokens + ff)
    r = lambda *s, f=1.0: (torch.randn(*s, generator=g) * f).bfloat16()
    h, gate, up, down = r(tokens, width), r(experts, ff, width, f=width ** -0.5 * 2), r(experts, ff, width, f=width ** -0.5 * 2), r(experts, width, ff, f=ff ** -0.5)
    z = torch.randn(tokens, experts, generator=g)
    unit = tile_rows(tokens * top, experts)
    rows = lib.routed_rows(tokens, top, experts, unit)
    i32 = lambda n: torch.empty(n, dtype=torch.int32, device=DEV)
    sel, row_pair, tile_expert = i32(tokens * top), i32(rows), i32(2 * (rows // unit))
    weight = torch.empty(tokens * top, device=DEV)
    lib.route_choose(z.to(DEV), experts, experts, top, 0, None, sel, weight, row_pair, tile_expert, unit=unit)
    both, wd = torch.empty(experts, 2 * ff, width, dtype=torch.bfloat16, device=DEV), torch.empty(experts, width, ff, dtype=torch.bfloat16, device=DEV)
    for e in range(experts):
        lib.place_rows(gate[e].to(DEV), both[e], 0, 16, 32, frag=True)
        lib.place_rows(up[e].to(DEV), both[e], 16, 16, 32, frag=True)
        lib.place_rows(down[e].to(DEV), wd[e], frag=True)
    act = None if limit is None else torch.tensor([limit, 1.702], device=DEV)
    y = torch.full((rows, ff), float("nan"), dtype=torch.bfloat16, device=DEV)
    out = torch.full((tokens * top, width), float("nan"), device=DEV)
    lib.routed_experts_tiled(h.to(DEV), top, row_pair, tile_expert, unit, both, wd, True, act, y, out)
    s = sel.cpu().long()
    x = h.double().repeat_interleave(top, 0)
    for e in range(experts):
        at = torch.nonzero(s == e)[:, 0]
        a, b = x[at] @ gate[e].double().T, x[at] @ up[e].double().T
        if limit is not None:
            a, b = a.clamp(max=limit), b.clamp(-limit, limit)
            u = a * torch.sigmoid(float(torch.tensor(1.702)) * a) * (b + 1)
        else:
            u = a * torch.sigmoid(a) * b
        want = u @ down[e].double().T
        # the units are rounded to 8 bits, everything else is float32
        _within(out[at], want, (u.abs() * 2.0 ** -8 + 1e-4) @ down[e].double().abs().T)
    # the kernels for few tokens and for runs of a few rows read the same interleaved matrices
    for n in (1, 9, 40, 100):
        n = min(n, tokens)
        few_rows = lib.routed_rows(n, top, experts)
        sel2, row2, tile2, weight2 = i32(n * top), i32(few_rows), i32(2 * (few_rows // 16)), torch.empty(n * top, device=DEV)
        lib.route_choose(z[:n].to(DEV), experts, experts, top, 0, None, sel2, weight2, row2, tile2)
        y2 = torch.empty((few_rows, ff + width), dtype=torch.bfloat16, device=DEV)
        out2 = torch.full((n * top, width), float("nan"), device=DEV)
        lib.routed_experts(h[:n].to(DEV), None, top, row2, tile2, both, None, wd, y2, out2, limit or 0.0, 1.702,
                           w_frag=True)
        _within(out2, out[:n * top].double(), 0.05)


# ---------------------------------------------------------------- single-token attention over several pages a wave
@pytest.mark.parametrize("dim,heads,kv,length,splits", [(128, 32, 8, 8001, 8), (128, 16, 1, 1500, 1), (64, 8, 2, 4000, 2), (128, 4, 4, 2100, 1)])
def test_single_token_attention_over_many_pages(lib, dim, heads, kv, length, splits):
    """Every wave walks three pages and more: the same bits every time, and the weighted sum of every row of every page."""
    g = torch.Generator().manual_seed(length)
    n = (length + 63) // 64
    order = torch.randperm(n, generator=g)
    k = torch.randn(n * 64, kv, dim, generator=g).bfloat16()
    v = torch.randn(n * 64, kv, dim, generator=g).bfloat16()
    # pages that differ much from one another: a row of another page in the place of one's own shows
    v = (v.float() + 40.0 * torch.randn(n, 1, 1, generator=g).repeat_interleave(64, 0)).bfloat16()
    paged = lambda x: x.view(n, 64, kv, dim).transpose(1, 2).contiguous()[torch.argsort(order)]
    kp, vp = paged(k).to(DEV), paged(v).to(DEV)
    q = torch.randn(1, heads, dim, generator=g).bfloat16()
    table = order.to(torch.int32)[None].to(DEV)
    pos = torch.tensor([length - 1], dtype=torch.int32)
    ws = torch.empty(heads * splits * (dim + 2), device=DEV)
    outs = []
    for _ in range(20):
        out = torch.full((1, heads * dim), float("nan"), dtype=torch.bfloat16, device=DEV)
        lib.attention_decode_bf16(q.to(DEV), kp, vp, out, pos.to(DEV), table, heads, kv, dim, 0.05, None, splits, ws)
        outs.append(out)
    want = _attention64(q.float(), k[:length].float(), v[:length].float(), pos, 0.05)
    # weights and outputs are rounded to 8 bits each
    _within(outs[0].view(want.shape), want, 2.0 ** -7 * float(v.abs().max()))
    for out in outs[1:]:
        assert torch.equal(out, outs[0])


@pytest.mark.parametrize("heads,kv,dim", [(32, 8, 128), (16, 1, 64), (8, 8, 128)])
@pytest.mark.parametrize("splits", [1, 3, 8, 9, 16, 65])
@pytest.mark.parametrize("sink", [False, True])
def test_single_token_attention_dealt_to_many_workgroups(lib, heads, kv, dim, splits, sink):
    """The kernel that rotates and stores, and the combination behind it: fewer and more workgroups than pages, than loads in flight and than
    lanes, with sequences of one page beside longer ones."""
    g = torch.Generator().manual_seed(heads + splits)
    lengths = [1, 70, 1500]
    kp, table, ks = _paged(lengths, kv, dim, g)
    vp, vs = torch.full_like(kp, float("nan")), []
    for b, n in enumerate(lengths):
        x = torch.randn(n, kv, dim, generator=g)
        for j in range(n):
            vp[table[b, j // 64], :, j % 64] = x[j]
        vs.append(x)
    q = torch.randn(3, heads, dim, generator=g)
    last = lambda rows: torch.stack([x[-1] for x in rows])
    qkv = torch.cat([q.flatten(1), last(ks).flatten(1), last(vs).flatten(1)], 1)
    sinks = torch.randn(heads, generator=g) if sink else None
    pos = torch.tensor(lengths, dtype=torch.int32) - 1
    r = lambda x: x.bfloat16().float()
    want = torch.cat([_attention64(r(q[b:b + 1]), r(ks[b]), r(vs[b]), pos[b:b + 1].long(), 0.1, sinks=sinks) for b in range(3)])
    kd, vd = kp.bfloat16().to(DEV), vp.bfloat16().to(DEV)
    for b, n in enumerate(lengths):                               # the token itself is the kernel's to store
        for pages in (kd, vd):
            pages[table[b, (n - 1) // 64], :, (n - 1) % 64] = float("nan")
    cos, sin = torch.ones(1600, dim // 2, device=DEV), torch.zeros(1600, dim // 2, device=DEV)
    ws = torch.full((3 * heads * splits * (dim + 2),), float("nan"), device=DEV)
    out = torch.full((3, heads * dim), float("nan"), dtype=torch.bfloat16, device=DEV)
    lib.attention_decode_fused_bf16(qkv.to(DEV), cos, sin, 1, kd, vd, out, pos.to(DEV), table.to(DEV), heads, kv, dim, 0.1, None, splits, ws,
                                    sinks=None if sinks is None else sinks.to(DEV))
    # weights and outputs are rounded to 8 bits each
    _within(out.view(want.shape), want, 2.0 ** -7 * float(max(x.abs().max() for x in vs)))


# ---------------------------------------------------------------- float32 products of few tokens, any depth
@pytest.mark.parametrize("m", [1, 4, 16])
@pytest.mark.parametrize("n,k", [(1, 4), (15, 12), (16, 20), (17, 96), (33, 124), (48, 132), (96, 252), (40, 260), (144, 500), (10, 516), (5, 1348)])
@pytest.mark.parametrize("odd", [0, 1])
def test_float32_products_of_few_tokens_and_any_depth(lib, m, n, k, odd):
    """Depths around the stages of 128 and the four waves; operands also at addresses that are multiples of 4 bytes only; what lies behind
    the operands is NaN."""
    g = torch.Generator().manual_seed(m * 31 + n + k)
    a, w = torch.randn(m, k, generator=g), torch.randn(n, k, generator=g)

    def placed(x):
        room = torch.full((x.numel() + 260,), float("nan"), device=DEV)
        room[odd:odd + x.numel()] = x.flatten().to(DEV)
        return room[odd:odd + x.numel()].view(x.shape)

    c = torch.full((m, n), float("nan"), device=DEV)
    lib.gemm_generic(placed(a), placed(w), c)
    # K products of 24 bits each, summed one after another: K 2^-24 of the sum of the absolute products at the most
    _within(c, a.double() @ w.double().T, k * 2.0 ** -24 * (a.double().abs() @ w.double().abs().T) + 1e-30)


# ---------------------------------------------------------------- the choice and the sort of a step of few tokens
@pytest.mark.parametrize("tokens", [1, 5, 17, 32])
@pytest.mark.parametrize("outputs,experts,top", [(1, 1, 1), (16, 16, 4), (20, 16, 3), (64, 64, 8), (64, 60, 64), (63, 63, 1), (8, 0, 2)])
@pytest.mark.parametrize("score", [0, 1, 2])
@pytest.mark.parametrize("extra", [False, True])
def test_choice_of_a_step_of_few_tokens(lib, tokens, outputs, experts, top, score, extra):
    """One launch of a rank per lane chooses and weighs, bit for bit, as the launch for many tokens does, which 40 tokens take: with ties,
    both zeros, infinities, NaN, and rows in which fewer outputs than are chosen have a score; and every pair has its row."""
    g = torch.Generator().manual_seed(tokens * 100 + outputs + score)
    z = torch.randn(40, outputs + 3, generator=g)
    z[1::4] = z[1::4].round()                                   # ties
    z[2::8] = torch.where(torch.rand(z[2::8].shape, generator=g) < 0.7, torch.tensor(-float("inf")), z[2::8])
    z[3::8, ::3] = float("nan")
    z[5] = -0.0
    z[6, outputs // 2] = float("inf")
    z[7] = -float("inf")
    z[0, :] = torch.where(torch.rand(z[0].shape, generator=g) < 0.3, torch.tensor(torch.finfo(torch.float32).min), z[0])
    z = z.to(DEV)
    bias = torch.randn(outputs, generator=g).to(DEV) if extra else None
    correction = torch.randn(outputs, generator=g).to(DEV) if extra and score == 1 else None
    res = []
    for n in (tokens, 40):
        rows = lib.routed_rows(n, top, experts, 16)
        sel, weight = torch.full((n * top,), -7, dtype=torch.int32, device=DEV), torch.full((n * top,), -7.0, device=DEV)
        pair, tile = torch.full((rows,), -7, dtype=torch.int32, device=DEV), torch.full((2 * (rows // 16),), -7, dtype=torch.int32, device=DEV)
        lib.route_choose(z[:n], outputs, experts, top, score, correction, sel, weight, pair, tile, bias=bias)
        res.append((sel.cpu(), weight.cpu(), pair.cpu(), tile.cpu()))
    few, many = res
    assert torch.equal(few[0], many[0][:tokens * top])
    assert torch.equal(few[1].view(torch.int32), many[1][:tokens * top].view(torch.int32))
    sel, _, pair, tile = few
    runs = pair.view(-1, 16)
    expert, position = tile.view(2, -1)
    at = 0
    for e in range(experts):
        wanted = (sel == e).nonzero().flatten().tolist()
        n_tiles = (len(wanted) + 15) // 16
        got = runs[at:at + n_tiles].flatten().tolist()
        assert sorted(p for p in got if p >= 0) == wanted and expert[at:at + n_tiles].tolist() == [e] * n_tiles
        assert got[len(wanted):] == [-1] * (16 * n_tiles - len(wanted)) and position[at:at + n_tiles].tolist() == list(range(n_tiles))
        at += n_tiles
    assert (runs[at:] == -1).all() and (expert[at:] == -1).all()


# ---------------------------------------------------------------- layer norm over copies of the stream
@pytest.mark.parametrize("copies", [1, 2, 3, 4, 7])
@pytest.mark.parametrize("width", [4, 252, 2048, 4096, 4100, 9000])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("kind", ["plain", "rows", "update"])
def test_layernorm_over_copies(lib, copies, width, dtype, kind):
    """One row of values a thread and several; every number of copies that has a kernel of its own and some that have none."""
    g = torch.Generator().manual_seed(copies * width)
    n, eps = 5, 1e-5
    x, weight, bias = torch.randn(copies, n, width, generator=g), torch.randn(width, generator=g), torch.randn(width, generator=g)
    coef, mix = torch.randn(copies, generator=g), torch.randn(copies, copies, generator=g)
    out_coef, y, scale, delta = torch.randn(copies, generator=g), torch.randn(n, width, generator=g), torch.randn(width, generator=g), torch.randn(n, width, generator=g)
    d = [t.to(DEV) for t in (x, coef, weight, bias, mix, out_coef, y, scale, delta)]
    rows = torch.tensor([3, 0, 3], dtype=torch.int32) if kind == "rows" else None
    want_x, v = x.double(), None
    if kind == "update":
        want_x = torch.einsum("sk,stw->ktw", mix.double(), x.double()) + out_coef.double()[:, None, None] * (scale.double() * y.double())
    v = (coef.double()[:, None, None] * want_x).sum(0)
    if kind != "update":
        v = v + delta.double()
        if copies == 1 and rows is None:
            want_x = v[None]
    v = v if rows is None else v[rows.long()]
    norm = (v - v.mean(-1, keepdim=True)) / (v.var(-1, unbiased=False, keepdim=True) + eps).sqrt()
    want = norm * weight.double() + bias.double()
    out = torch.full((v.shape[0], width), float("nan"), dtype=dtype, device=DEV)
    lib.streams_layernorm(d[0], d[1], d[2], d[3], eps, None if rows is None else rows.to(DEV), out, delta=None if kind == "update" else d[8],
                          update=(d[4], d[5], d[6], d[7]) if kind == "update" else None)
    # a value is a sum of (copies + 1)^2 products at the most, a mean and a variance are sums of `width` terms: each is off by that many
    # roundings of the largest thing it is made of; then the rounding of the result's type
    big = (coef.abs().double()[:, None, None] * (want_x.abs() + (x.abs().sum(0) * mix.abs().max() + (scale * y).abs() * out_coef.abs().max()).double())).sum(0).max()
    sd = (v.var(-1, unbiased=False, keepdim=True) + eps).sqrt()
    bound = weight.abs().double() * (((copies + 1) ** 2 + 30) * 2.0 ** -23 * big / sd * (1 + norm.abs() * norm.abs().amax(-1, keepdim=True)))
    bound = bound + want.abs() * (2.0 ** -8 if dtype is torch.bfloat16 else 2.0 ** -22) + 1e-6
    _within(out, want, bound)
    _within(d[0], want_x, ((copies + 3) * 2.0 ** -23) * (x.abs().double().sum(0) * mix.abs().max() + (scale * y).abs().double() * out_coef.abs().max()
                                                      + x.abs().double().sum(0) * (1 + coef.abs().max()) + delta.abs().double()).max())


# ---------------------------------------------------------------- the gated delta rule, token after token
@pytest.mark.parametrize("dim", [8, 32, 64, 68, 100, 128, 200, 384])
@pytest.mark.parametrize("lengths", [[1], [1, 1, 1], [15, 16, 17], [70]])
@pytest.mark.parametrize("heads,per_head", [(2, True), (64, False)])
@pytest.mark.parametrize("rule", ["delta", "plain"])
def test_recurrences_of_every_key_size(lib, dim, lengths, heads, per_head, rule):
    """Every split of a column over lanes, both layouts of a column in LDS, chunks that are whole, in part and of one token; 64 heads fill
    the GPU and take the longer shares of a column."""
    from types import SimpleNamespace
    g = torch.Generator().manual_seed(dim + heads + sum(lengths))
    n, vdim = sum(lengths), 20 if heads == 2 else 128
    qkv = torch.randn(n, 2 * heads * dim + heads * vdim, generator=g)
    unit = torch.nn.functional.normalize(qkv[:, :2 * heads * dim].view(n, 2 * heads, dim), dim=-1)
    qkv[:, :2 * heads * dim] = unit.view(n, -1)
    decay = 0.8 + 0.2 * torch.rand(n, heads * (1 if per_head else dim), generator=g)
    beta = torch.rand(n, heads, generator=g)
    state = torch.randn(len(lengths) + 1, heads, vdim, dim, generator=g)
    slots = list(range(len(lengths), 0, -1))
    want, want_state, most, at = torch.empty(n, heads, vdim, dtype=torch.float64), state.double(), 1.0, 0
    for b, length in enumerate(lengths):
        S = want_state[slots[b]].transpose(1, 2).clone()              # [H, dim, vdim]
        for t in range(at, at + length):
            q, k = unit[t, :heads].double(), unit[t, heads:].double()
            v = qkv[t, 2 * heads * dim:].view(heads, vdim).double()
            S = S * decay[t].double().view(heads, -1, 1)
            u = beta[t].double()[:, None] * (v - torch.einsum("hiv,hi->hv", S, k)) if rule == "delta" else v
            S = S + k[:, :, None] * u[:, None, :]
            want[t] = torch.einsum("hiv,hi->hv", S, q)
            most = max(most, float(S.norm(dim=1).max()))
        want_state[slots[b]] = S.transpose(1, 2)
        at += length
    cu = torch.tensor([0] + torch.tensor(lengths).cumsum(0).tolist(), dtype=torch.int32, device=DEV)
    ctx = SimpleNamespace(n_tokens=n, n_seqs=len(lengths), cu_seqlens=cu, slots=torch.tensor(slots, dtype=torch.int32, device=DEV))
    dev_state, out = state.to(DEV), torch.full((n, heads * vdim), float("nan"), device=DEV)
    lib.linear_recurrence(qkv.to(DEV), heads, dim, heads, vdim, decay.to(DEV), 0, per_head, beta.to(DEV) if rule == "delta" else None,
                          dev_state, ctx, out)
    # unit keys and decays below 1 do not enlarge an error: each token adds the roundings of two sums over `dim` of a column
    bound = max(lengths) * (2 * dim + 8) * 2.0 ** -24 * most
    _within(out, want.view(n, -1), bound)
    _within(dev_state, want_state, bound)


# ---------------------------------------------------------------- what enters a recurrence
@pytest.mark.parametrize("tokens", [1, 5, 128, 129])
@pytest.mark.parametrize("heads,dim,per_head", [(1, 4, True), (2, 100, False), (16, 128, False), (40, 256, True), (3, 300, False), (24, 512, False)])
@pytest.mark.parametrize("unit", [0, 1])
def test_what_enters_a_recurrence(lib, tokens, heads, dim, per_head, unit):
    """Heads that fit registers and longer ones, one workgroup a token and several, down to fewer threads than there is work."""
    g = torch.Generator().manual_seed(tokens + dim)
    cols = heads if per_head else heads * dim
    qk, a, b = torch.randn(tokens, 2 * heads * dim + 3, generator=g), torch.randn(tokens, cols + 1, generator=g), torch.randn(tokens, heads, generator=g)
    bias, a_log = torch.randn(cols, generator=g), 0.3 * torch.randn(heads, generator=g)
    d = [t.to(DEV) for t in (qk, a, b, bias, a_log)]
    beta = torch.full((tokens, heads), float("nan"), device=DEV)
    lib._ok(lib._lib.rb_recurrence_prep(d[0].data_ptr(), qk.shape[1], heads, dim, unit, 0.25, 1e-6, d[1].data_ptr(), a.shape[1], cols, 0,
                                        d[3].data_ptr(), d[4].data_ptr(), 1.0, heads, d[2].data_ptr(), heads, beta.data_ptr(), tokens, lib._stream()))
    v = qk[:, :2 * heads * dim].double().view(tokens, 2, heads, dim)
    scale = torch.tensor([0.25, 1.0], dtype=torch.float64).view(1, 2, 1, 1)
    want = v * scale / ((v * v).sum(-1, keepdim=True) + 1e-6).sqrt() if unit else v * scale
    # a sum of `dim` squares over 64 lanes, a root and a quotient: dim / 64 + 12 roundings
    _within(d[0][:, :2 * heads * dim], want.view(tokens, -1), (dim / 64 + 12) * 2.0 ** -24 * want.view(tokens, -1).abs() + 1e-30)
    assert torch.equal(d[0][:, 2 * heads * dim:].cpu(), qk[:, 2 * heads * dim:]) and torch.equal(d[1][:, cols:].cpu(), a[:, cols:])
    rate = a_log.double().exp().repeat_interleave(cols // heads) * torch.nn.functional.softplus(a[:, :cols].double() + bias.double())
    # the exponent has the roundings of a sum, an exponential, a softplus and a product, the result those of its exponential
    _within(d[1][:, :cols], (-rate).exp(), 32 * 2.0 ** -24 * (1 + rate) * (-rate).exp() + 2.0 ** -22 * (-rate).exp() + 1e-37)
    _within(beta, b.double().sigmoid(), 2.0 ** -20)


# ---------------------------------------------------------------- single-token attention: one query head on a kv head, many sequences
@pytest.mark.parametrize("dim", [64, 128])
@pytest.mark.parametrize("kv,lengths,window,splits", [(3, [1, 64, 65, 700], 0, 1), (2, [130, 5, 1000], 100, 1), (2, [2000, 63], 0, 5), (1, [500], 130, 3),
                                                      (16, [(97 * i) % 400 + 1 for i in range(20)], 0, 1), (16, [(61 * i) % 190 + 1 for i in range(40)], 0, 1),
                                                      (33, [300] * 8, 0, 2)])
def test_single_token_attention_of_heads_of_their_own(lib, dim, kv, lengths, window, splits):
    """Weights in float32: what is left of the error is that of float32 scores and of the output's 8 bits.  Up to 256 workgroups, up to
    512 (sequences taken by length) and more (two waves each); windows that begin inside a page, behind an infinite value."""
    g = torch.Generator().manual_seed(dim + kv + len(lengths))
    kp, table, ks = _paged(lengths, kv, dim, g)
    vp, _, vs = _paged(lengths, kv, dim, torch.Generator().manual_seed(dim + kv + len(lengths)))
    rows = lambda xs: [x.bfloat16().float() for x in xs]
    ks, vs = rows(ks), rows(vs)
    pos = torch.tensor([n - 1 for n in lengths], dtype=torch.int32)
    q = torch.randn(len(lengths), kv, dim, generator=g).bfloat16()
    want = torch.cat([_attention64(q[b:b + 1].float(), ks[b], vs[b], pos[b:b + 1], 0.1, window) for b in range(len(lengths))])
    vd = vp.bfloat16()
    if window:                                             # a key that no query sees any more
        for b, n in enumerate(lengths):
            if n > window:
                gone = n - window - 1
                vd[table[b, gone // 64], :, gone % 64] = float("inf")
    out = torch.full((len(lengths), kv * dim), float("nan"), dtype=torch.bfloat16, device=DEV)
    ws = torch.full((len(lengths) * kv * splits * (dim + 2),), float("nan"), device=DEV)
    lib.attention_decode_bf16(q.to(DEV), kp.bfloat16().to(DEV), vd.to(DEV), out, pos.to(DEV), table.to(DEV), kv, kv, dim, 0.1, window, splits, ws)
    _within(out.view(want.shape), want, 2.0 ** -8 * want.abs() + 2.0 ** -14 * float(max(x.abs().max() for x in vs)))


@pytest.mark.parametrize("length", [60, 200])
def test_float32_weights_cost_a_short_context_little(lib, length):
    """A step whose heads have a key head each, short contexts: beside the same heads with weights of 8 bits.  (Rows of zeros that
    nothing read, a second trip to memory behind them and lane moves made it 1.2 to 1.25 of that.)"""
    heads, dim = 32, 128
    pages = (length + 63) // 64
    kp = torch.randn(pages, heads, 64, dim, device=DEV).bfloat16()
    vp = torch.randn_like(kp)
    table = torch.arange(pages, dtype=torch.int32, device=DEV)[None]
    pos = torch.tensor([length - 1], dtype=torch.int32, device=DEV)
    qkv = torch.randn(1, 3 * heads * dim, device=DEV)
    cos, sin = torch.ones(256, dim // 2, device=DEV), torch.zeros(256, dim // 2, device=DEV)
    out, ws = torch.empty(1, heads * dim, dtype=torch.bfloat16, device=DEV), torch.empty(heads * (dim + 2), device=DEV)
    run = lambda: lib.attention_decode_fused_bf16(qkv, cos, sin, 1, kp, vp, out, pos, table, heads, heads, dim, 0.1, 0, 1, ws)
    times = [1e9, 1e9]
    try:
        for mode in (0, 1, 0, 1):
            lib._lib.rb_tune_decode_mfma(mode)
            graph = torch.cuda.CUDAGraph()
            run()
            torch.cuda.synchronize()
            with torch.cuda.graph(graph):
                for _ in range(20):
                    run()
            times[mode] = min(times[mode], _least_time(graph.replay, calls=3))
    finally:
        lib._lib.rb_tune_decode_mfma(0)
    assert times[0] <= 1.13 * times[1], times


@pytest.mark.parametrize("hook,value", [("rb_tune_decode_waves", 8), ("rb_tune_decode_waves", 3), ("rb_tune_decode_mfma", 2)])
def test_forced_choices_of_single_token_attention_that_are_not_built_are_refused(lib, hook, value):
    from rbitnet_amd.errors import KernelError
    kp = torch.zeros(1, 2, 64, 64, dtype=torch.bfloat16, device=DEV)
    i32 = lambda *x: torch.tensor(x, dtype=torch.int32, device=DEV)
    call = lambda: lib.attention_decode_bf16(torch.zeros(1, 4, 64, dtype=torch.bfloat16, device=DEV), kp, torch.zeros_like(kp),
                                             torch.empty(1, 256, dtype=torch.bfloat16, device=DEV), i32(5), i32(0)[None], 4, 2, 64, 0.1, 0, 1,
                                             torch.empty(4 * 66, device=DEV))
    try:
        getattr(lib._lib, hook)(value)
        with pytest.raises(KernelError):
            call()
    finally:
        getattr(lib._lib, hook)(0)
    call()


def test_single_token_attention_of_an_infinite_value(lib):
    """An infinity among the visible values comes out in its own place, whatever the weights' parts are, and nowhere else."""
    kv, dim, n = 2, 128, 200
    g = torch.Generator().manual_seed(3)
    kp, table, ks = _paged([n], kv, dim, g)
    vp, _, vs = _paged([n], kv, dim, torch.Generator().manual_seed(3))
    vp = vp.bfloat16()
    vp[table[0, 1], 1, 7, 50] = float("-inf")
    q = torch.randn(1, kv, dim, generator=g).bfloat16()
    out = torch.full((1, kv * dim), float("nan"), dtype=torch.bfloat16, device=DEV)
    pos = torch.tensor([n - 1], dtype=torch.int32)
    lib.attention_decode_bf16(q.to(DEV), kp.bfloat16().to(DEV), vp.to(DEV), out, pos.to(DEV), table.to(DEV), kv, kv, dim, 0.1, 0, 1,
                              torch.empty(kv * (dim + 2), device=DEV))
    got = out.float().cpu().view(kv, dim)
    assert got[1, 50] == float("-inf")
    got[1, 50] = 0.0
    assert torch.isfinite(got).all()


@pytest.mark.parametrize("heads,kv,count", [(32, 16, 18), (32, 16, 33), (32, 8, 70), (16, 16, 18), (16, 16, 40)])
@pytest.mark.parametrize("sink", [False, True])
def test_single_token_attention_of_many_sequences(lib, heads, kv, count, sink):
    """The kernel that rotates and stores with more workgroups than compute units: sequences by length, and two waves each; what it
    stored is there."""
    dim = 128
    lengths = [(83 * i) % 210 + 1 for i in range(count)]
    g = torch.Generator().manual_seed(heads + count)
    kp, table, ks = _paged(lengths, kv, dim, g)
    vp, _, vs = _paged(lengths, kv, dim, torch.Generator().manual_seed(heads + count))
    pos = torch.tensor([n - 1 for n in lengths], dtype=torch.int32)
    qkv = torch.randn(count, (heads + 2 * kv) * dim, generator=g)
    angle = torch.randn(256, dim // 2, generator=g)
    cos, sin = torch.cos(angle).to(DEV), torch.sin(angle).to(DEV)
    sinks = torch.randn(heads, generator=g) if sink else None
    kd, vd = kp.bfloat16().to(DEV), vp.bfloat16().to(DEV)
    out = torch.full((count, heads * dim), float("nan"), dtype=torch.bfloat16, device=DEV)
    lib.attention_decode_fused_bf16(qkv.to(DEV), cos, sin, 1, kd, vd, out, pos.to(DEV), table.to(DEV), heads, kv, dim, 0.1, None, 1,
                                    torch.empty(count * heads * (dim + 2), device=DEV), sinks=None if sinks is None else sinks.to(DEV))

    def turned(x, at):                                     # [H, D], halves together
        a, c, s = x.double(), torch.cos(angle[at]).double(), torch.sin(angle[at]).double()
        u, v = a[:, :dim // 2], a[:, dim // 2:]
        return torch.cat([u * c - v * s, v * c + u * s], 1).bfloat16().float()
    want = []
    for b, n in enumerate(lengths):
        row = qkv[b].view(heads + 2 * kv, dim)
        k, v = ks[b].bfloat16().float().clone(), vs[b].bfloat16().float().clone()
        k[n - 1], v[n - 1] = turned(row[heads:heads + kv], n - 1), row[heads + kv:].bfloat16().float()
        want.append(_attention64(turned(row[:heads], n - 1)[None], k, v, pos[b:b + 1], 0.1, sinks=sinks))
        page, at = int(table[b, (n - 1) // 64]), (n - 1) % 64
        assert torch.equal(vd[page, :, at].float().cpu(), v[n - 1])
        # the rotation rounds to 8 bits; a number between two of them may go either way
        _within(kd[page, :, at], k[n - 1].double(), 2.0 ** -7 * k[n - 1].abs().double() + 1e-6)
    want = torch.cat(want)
    _within(out.view(want.shape), want, 2.0 ** -6 * float(max(x.abs().max() for x in vs)))


# ---------------------------------------------------------------------------- single tokens through a recurrence, in one launch
ONE_LAUNCH = [("channel_delta", dict(heads=h, kv_heads=k, dim=d, vdim=v, conv=c, eps=1e-5, decay_rank=16, gate_rank=16))
              for h, k, d, v, c in ((1, 1, 64, 64, 4), (3, 3, 128, 64, 2), (4, 2, 128, 128, 3), (4, 1, 64, 128, 1))]
ONE_LAUNCH += [("gated_delta", dict(heads=h, kv_heads=k, dim=d, vdim=v, conv=c, eps=1e-5))
               for h, k, d, v, c in ((2, 2, 64, 192, 4), (4, 1, 128, 128, 4), (7, 1, 64, 64, 3), (6, 2, 128, 64, 1))]
ONE_LAUNCH += [("decay_attention", dict(heads=h, dim=d, vdim=v, tau=8.0, decay_rank=16, eps=1e-5)) for h, d, v in ((2, 64, 128), (1, 128, 448), (3, 128, 64))]
ONE_LAUNCH += [("time_mix", dict(heads=h, dim=d, decay_rank=16, eps=1e-5)) for h, d in ((1, 64), (3, 128))]
ONE_LAUNCH += [("state_space", dict(heads=h, vdim=v, state=d, groups=g, conv=c, norm_groups=n, eps=1e-5))
               for h, v, d, g, c, n in ((8, 64, 128, 1, 4, 1), (4, 64, 64, 2, 2, 4), (2, 128, 128, 2, 3, 4), (5, 64, 128, 1, 1, 5))]


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("kind,params", ONE_LAUNCH)
def test_single_tokens_through_a_recurrence_in_one_launch_beside_launches_of_their_own(lib, kind, params, dtype):
    """The same mixer, states and tokens both ways, three steps of three sequences, by formula: 1e-5 of the largest value bounds any order
    of float32 sums of at most 512 numbers, and bfloat16 outputs may round the other way once.  (That the order is the same: below.)"""
    gen = torch.Generator().manual_seed(11)
    hidden = 64
    part = build_part("mixer", PartSpec(kind, params), BuildEnv(hidden_size=hidden, dtype=dtype, device=torch.device(DEV), lib=lib))
    assert part.one_launch
    part.load({n: (torch.randn(ts.shape, generator=gen) * (0.5 if len(ts.shape) < 2 or min(ts.shape) < 8 else ts.shape[-1] ** -0.5))
               .to(torch.float32 if ts.role == "gain" else dtype).to(DEV) for n, ts in part.tensor_specs().items()})
    caches = [Cache([part.cache_requests()], 3, 64 * 4, dtype, DEV) for _ in range(2)]
    slots = [2, 0, 1]
    for c in caches:
        assert sorted(c.alloc_slot() for _ in range(3)) == [0, 1, 2]
    for g, other in zip(caches[0].state_groups, caches[1].state_groups):
        g.data.copy_(torch.randn(g.data.shape, generator=gen) * 0.3)
        other.data.copy_(g.data)
    for step in range(3):
        h = torch.randn(3, hidden, generator=gen).to(dtype).to(DEV)
        outs = []
        for one, c in zip((True, False), caches):
            part.one_launch = one
            c.reserve(slots, [1, 1, 1])
            ctx = StepContext.for_batch(DEV, StepBatch(slots, [c.length(s) for s in slots], [[1]] * 3, [0, 1, 2], c.block_tables(slots)),
                                        n_compute_units=lib.n_compute_units)
            outs.append(part.forward(h, ctx, c.view(0, ctx.block_tables)).float())
            c.commit(slots, [1, 1, 1])
        worst = lambda got, want: float((got - want).abs().max() / want.abs().max())
        assert worst(*outs) < (1e-5 if dtype == torch.float32 else 1e-2)
        for g, other in zip(caches[0].state_groups, caches[1].state_groups):
            assert worst(g.data[:, slots], other.data[:, slots]) < 1e-5
    assert not lib.recurrence_step_ok(2, 2, 96, 64) and not lib.recurrence_step_ok(2, 2, 64, 96) and not lib.recurrence_step_ok(9, 1, 64, 64)


@pytest.mark.parametrize("units", [0, 1])
@pytest.mark.parametrize("kind,params", ONE_LAUNCH + [("state_space", dict(heads=8, vdim=64, state=128, groups=1, conv=4, norm_groups=n, eps=1e-5)) for n in (2, 8)])
def test_single_tokens_through_a_recurrence_in_one_launch_give_the_same_bits(lib, kind, params, units, monkeypatch):
    """Sums are taken in the order of the launches that this one stands for, by whichever number of lanes those deal a column to (units:
    how many compute units decide that; 1: as if the sequences filled the GPU)."""
    gen = torch.Generator().manual_seed(5)
    monkeypatch.setattr(type(lib), "recurrence_step_pays", staticmethod(lambda *a: True))
    part = build_part("mixer", PartSpec(kind, params), BuildEnv(hidden_size=64, dtype=torch.float32, device=torch.device(DEV), lib=lib))
    part.load({n: (torch.randn(ts.shape, generator=gen) * (0.5 if len(ts.shape) < 2 or min(ts.shape) < 8 else ts.shape[-1] ** -0.5)).to(DEV)
               for n, ts in part.tensor_specs().items()})
    cache = Cache([part.cache_requests()], 3, 64, torch.float32, DEV)
    slots, h = [cache.alloc_slot() for _ in range(3)], torch.randn(3, 64, generator=gen).to(DEV)
    states = [torch.randn(g.data.shape, generator=gen).to(DEV) * 0.3 for g in cache.state_groups]
    ctx = StepContext.for_batch(DEV, StepBatch(slots, [0] * 3, [[1]] * 3, [0, 1, 2], {}), n_compute_units=lib.n_compute_units)
    got = []
    try:
        lib._lib.rb_tune_compute_units(units)
        for one in (True, False):
            part.one_launch = one
            for g, s in zip(cache.state_groups, states):
                g.data.copy_(s)
            got.append([part.forward(h, ctx, cache.view(0, {}))] + [g.data[:, slots].clone() for g in cache.state_groups])
    finally:
        lib._lib.rb_tune_compute_units(0)
    for a, b in zip(*got):
        assert torch.equal(a, b)


# ---------------------------------------------------------------------------- recurrences: whole chunks of 16 tokens and what is left
@pytest.mark.parametrize("dim,vdim", [(64, 12), (64, 36), (128, 12), (128, 24), (128, 33), (96, 36)])
@pytest.mark.parametrize("per_head", [False, True])
@pytest.mark.parametrize("delta", [False, True])
def test_recurrences_of_whole_and_partial_chunks_with_one_and_two_columns_a_lane(lib, dim, vdim, per_head, delta):
    """Against the equations in float64 (1e-5 of the largest value bounds any order of float32 sums of 128 numbers over 50 tokens whose
    decays shrink what came before).  How many compute units there are decides about two columns a lane of 8, one, and one of 16 lanes: the
    first two give the same bits, and so does a step in two pieces."""
    gen = torch.Generator().manual_seed(dim + vdim)
    heads, kv, lengths, cuts = 4, 2, [1, 15, 16, 17, 31, 32, 33, 50], [1, 7, 16, 1, 16, 31, 17, 33]
    n, cu = sum(lengths), [sum(lengths[:i]) for i in range(len(lengths) + 1)]
    q, k = (torch.nn.functional.normalize(torch.randn(n, kv, dim, generator=gen), dim=-1) for _ in range(2))
    v, beta = torch.randn(n, heads, vdim, generator=gen), torch.rand(n, heads, generator=gen)
    g = 0.5 + 0.5 * torch.rand(n, heads, 1 if per_head else dim, generator=gen)
    start = torch.randn(len(lengths), heads, vdim, dim, generator=gen) * 0.3

    def run(units, steps):
        state, out = start.to(DEV), torch.full((n, heads * vdim), float("nan"), device=DEV)
        try:
            lib._lib.rb_tune_compute_units(units)
            for spans in steps:
                pick = torch.cat([torch.arange(cu[b] + lo, cu[b] + hi) for b, (lo, hi) in enumerate(spans)])
                seqs = [hi - lo for lo, hi in spans]
                ctx = SimpleNamespace(n_tokens=len(pick), n_seqs=len(seqs), slots=torch.arange(len(seqs), dtype=torch.int32, device=DEV),
                                      cu_seqlens=torch.tensor([sum(seqs[:i]) for i in range(len(seqs) + 1)], dtype=torch.int32, device=DEV))
                qkv = torch.cat([t[pick].reshape(len(pick), -1) for t in (q, k, v)], 1).to(DEV)
                part = torch.full((len(pick), heads * vdim), float("nan"), device=DEV)
                lib.linear_recurrence(qkv, kv, dim, heads, vdim, g[pick].reshape(len(pick), -1).to(DEV), 0, per_head,
                                      beta[pick].to(DEV) if delta else None, state, ctx, part)
                out[pick.to(DEV)] = part
        finally:
            lib._lib.rb_tune_compute_units(0)
        return out, state

    whole = [[(0, m) for m in lengths]]
    waves = lambda cols: len(lengths) * heads * -(-vdim // cols)
    between = (waves(16) + waves(8)) // 2 // 4               # four SIMDs a compute unit
    assert waves(16) < 4 * between <= waves(8) < 4 * 256
    out, state = run(1, whole)
    for other in (run(between, whole), run(1, [[(0, c) for c in cuts], [(c, m) for c, m in zip(cuts, lengths)]])):
        assert torch.equal(out, other[0]) and torch.equal(state, other[1])
    more_lanes = run(0, whole)
    want, wanted = torch.empty(n, heads, vdim, dtype=torch.float64), start.double().clone()
    for b, m in enumerate(lengths):
        s = wanted[b]                                          # [H, vdim, dim]
        for t in range(cu[b], cu[b] + m):
            kk, qq = (x[t].double().repeat_interleave(heads // kv, 0)[:, None] for x in (k, q))
            s *= g[t].double()[:, None]
            u = v[t].double()
            if delta:
                u = beta[t].double()[:, None] * (u - (s * kk).sum(-1))
            s += u[..., None] * kk
            want[t] = (s * qq).sum(-1)
    for got, ref in ((out, want), (state, wanted), (more_lanes[0], want), (more_lanes[1], wanted)):
        _within(got.view(ref.shape), ref, 1e-5 * float(ref.abs().max()))


@pytest.mark.parametrize("dim,vdim", [(64, 12), (64, 36), (128, 24), (128, 33), (96, 36)])
@pytest.mark.parametrize("kind", ["bonus", "silu", "selective"])
def test_other_recurrences_of_whole_and_partial_chunks_with_one_and_two_columns_a_lane(lib, dim, vdim, kind):
    """As above for time mixing, silu on the inputs and the selective scan, against the equations in float64.  Sums: as above.  A decay made in float32 is off by a few
    2^-24 of itself and what it multiplies shrinks by it, so that a state that has forgotten half of a value after 14 tokens (x = 0.05) is off by
    2 / x of these: 5e-6."""
    gen = torch.Generator().manual_seed(dim + vdim)
    heads, lengths, cuts = 4, [1, 15, 16, 17, 31, 32, 33, 50], [1, 7, 16, 1, 16, 31, 17, 33]
    n, cu = sum(lengths), [sum(lengths[:i]) for i in range(len(lengths) + 1)]
    kv = 2 if kind == "selective" else heads
    q, k = (torch.nn.functional.normalize(torch.randn(n, kv, dim, generator=gen), dim=-1) * (3.0 if kind == "silu" else 1.0) for _ in range(2))
    v, start = torch.randn(n, heads, vdim, generator=gen), torch.randn(len(lengths), heads, vdim, dim, generator=gen) * 0.3
    g, u = 0.5 + 0.5 * torch.rand(n, heads, dim, generator=gen), torch.randn(heads, dim, generator=gen)
    constant = 0.5 + 0.45 * torch.rand(heads, generator=gen)
    dt, dt_bias, a_log, d = (torch.randn(*shape, generator=gen) for shape in ((n, heads), (heads,), (heads,), (heads,)))

    def run(units, steps):
        state, out = start.to(DEV), torch.full((n, heads * vdim), float("nan"), device=DEV)
        try:
            lib._lib.rb_tune_compute_units(units)
            for spans in steps:
                pick = torch.cat([torch.arange(cu[b] + lo, cu[b] + hi) for b, (lo, hi) in enumerate(spans)])
                seqs = [hi - lo for lo, hi in spans]
                ctx = SimpleNamespace(n_tokens=len(pick), n_seqs=len(seqs), slots=torch.arange(len(seqs), dtype=torch.int32, device=DEV),
                                      cu_seqlens=torch.tensor([sum(seqs[:i]) for i in range(len(seqs) + 1)], dtype=torch.int32, device=DEV))
                rows = lambda *ts: torch.cat([t[pick].reshape(len(pick), -1) for t in ts], 1).to(DEV)
                part = torch.full((len(pick), heads * vdim), float("nan"), device=DEV)
                if kind == "bonus":
                    lib.time_mix_recurrence(rows(q), rows(k), rows(v), rows(g), u.to(DEV), state, ctx, part, heads, dim, vdim)
                elif kind == "silu":
                    lib.lightning_recurrence(rows(q, k, v), dim, heads, vdim, constant.to(DEV), state, ctx, part)
                else:
                    lib.selective_scan(rows(v, k, q), dim, kv, heads, vdim, rows(dt), 0, dt_bias.to(DEV), a_log.to(DEV), d.to(DEV), state, ctx, part)
                out[pick.to(DEV)] = part
        finally:
            lib._lib.rb_tune_compute_units(0)
        return out, state

    whole = [[(0, m) for m in lengths]]
    waves = lambda cols: len(lengths) * heads * -(-vdim // cols)
    between = (waves(16) + waves(8)) // 2 // 4               # four SIMDs a compute unit
    assert waves(16) < 4 * between <= waves(8) < 4 * 256
    out, state = run(1, whole)
    for other in (run(between, whole), run(1, [[(0, c) for c in cuts], [(c, m) for c, m in zip(cuts, lengths)]])):
        assert torch.equal(out, other[0]) and torch.equal(state, other[1])
    want, wanted = torch.empty(n, heads, vdim, dtype=torch.float64), start.double().clone()
    silu = torch.nn.functional.silu
    for b, m in enumerate(lengths):
        s = wanted[b]                                          # [H, vdim, dim]
        for t in range(cu[b], cu[b] + m):
            qq, kk = (x[t].double().repeat_interleave(heads // kv, 0)[:, None] for x in (q, k))
            vv = v[t].double()
            if kind == "bonus":
                write = vv[..., None] * kk
                want[t] = ((s + u.double()[:, None] * write) * qq).sum(-1)
                s *= g[t].double()[:, None]
                s += write
            elif kind == "silu":
                s *= constant.double()[:, None, None]
                s += silu(vv)[..., None] * silu(kk)
                want[t] = (s * silu(qq)).sum(-1)
            else:
                step = torch.nn.functional.softplus(dt[t].double() + dt_bias.double())
                s *= torch.exp(-torch.exp(a_log.double()) * step)[:, None, None]
                s += (step[:, None] * vv)[..., None] * kk
                want[t] = (s * qq).sum(-1) + d.double()[:, None] * vv
    more_lanes = run(0, whole)
    for got, ref in ((out, want), (state, wanted), (more_lanes[0], want), (more_lanes[1], wanted)):
        _within(got.view(ref.shape), ref, 1e-5 * float(ref.abs().max()))


def test_a_recurrence_of_more_workgroups_than_a_launch_takes(lib):
    """A launch has fewer than 2^32 threads, here a wave a (sequence, head).  States of one number, against the rule in float64: the state is off by two roundings of
    numbers up to 5, and what is read by those of g S q (2 and 2), of k q times v (8) and of the sum (10), 2^-24 of each."""
    seqs, heads = 16400, 4096
    gen = torch.Generator(device=DEV).manual_seed(3)
    qkv = torch.randn(seqs, 2 + heads, generator=gen, device=DEV).clamp_(-2.0, 2.0)
    g = torch.rand(seqs, heads, generator=gen, device=DEV)
    state = torch.rand(seqs, heads, 1, 1, generator=gen, device=DEV)
    out = torch.empty(seqs, heads, device=DEV)
    ctx = SimpleNamespace(n_tokens=seqs, n_seqs=seqs, slots=torch.arange(seqs, dtype=torch.int32, device=DEV),
                          cu_seqlens=torch.arange(seqs + 1, dtype=torch.int32, device=DEV))
    kept = state.clone()
    lib.linear_recurrence(qkv, 1, 1, heads, 1, g, 0, True, None, state, ctx, out)
    want = g.double() * kept.view(seqs, heads) + qkv[:, 1:2].double() * qkv[:, 2:]
    assert float((state.view(seqs, heads) - want).abs().max()) <= 10 * 2.0 ** -24
    assert float((out - want * qkv[:, :1]).abs().max()) <= 22 * 2.0 ** -24


# ---------------------------------------------------------------------------- the router's product and the choice in one launch
@pytest.mark.parametrize("n", [1, 3, 16])
@pytest.mark.parametrize("rows,outputs,experts,top,k", [(16, 16, 16, 4, 2048), (17, 16, 16, 2, 1024), (8, 8, 8, 8, 1152), (64, 64, 64, 6, 1280),
                                                       (33, 32, 30, 5, 8192), (48, 48, 48, 1, 3200)])
def test_router_product_and_choice_in_one_launch_beside_two(lib, n, rows, outputs, experts, top, k):
    """The same bits as a product and a choice of their own: the product's sums are taken in the same order.  A token whose logits
    are not numbers, every score, rows of W behind the outputs, W as rows and fragment-major.  (Which row of an expert's run a pair
    gets is the waves' to say: a run is compared as a set.)"""
    gen = torch.Generator().manual_seed(rows + k)
    h = torch.randn(n, k, generator=gen).to(torch.bfloat16)
    if n > 2:
        h[1] = float("nan")
    h, w = h.to(DEV), (torch.randn(rows, k, generator=gen) * k ** -0.5).to(torch.bfloat16).to(DEV)
    bias = (torch.randn(outputs, generator=gen) * 0.1).to(DEV)
    correction = (torch.randn(outputs, generator=gen) * 0.1).to(DEV)
    assert lib.route_linear_ok(h, rows, outputs)
    for frag in (False, True) if rows % 16 == 0 and k % 64 == 0 else (False,):
        wd = w
        if frag:
            wd = torch.empty_like(w)
            lib.place_rows(w, wd, frag=True)
        for score, corr, b in ((0, None, None), (1, correction, bias), (1, None, None), (2, None, bias)):
            room = lib.routed_rows(n, top, experts)
            got, want = ([torch.zeros(n, rows, device=DEV), torch.empty(n * top, dtype=torch.int32, device=DEV), torch.empty(n * top, device=DEV),
                          torch.empty(room, dtype=torch.int32, device=DEV), torch.zeros(2 * (room // 16), dtype=torch.int32, device=DEV)]
                         for _ in range(2))
            lib.route_linear(h, wd, frag, got[0], outputs, experts, top, score, corr, got[1], got[2], got[3], got[4], bias=b)
            lib.gemm_bf16(h, wd, want[0], 0, w_frag=frag)
            lib.route_choose(want[0], outputs, experts, top, score, corr, want[1], want[2], want[3], want[4], bias=b)
            for i, (x, y) in enumerate(zip(got, want)):
                if i != 3:
                    assert torch.equal(x.nan_to_num(7.0) if x.is_floating_point() else x, y.nan_to_num(7.0) if y.is_floating_point() else y), i
            runs = lambda pair, tile: {e: sorted(p for t in range(room // 16) if tile[t] == e for p in pair[16 * t:16 * t + 16]) for e in set(tile[:room // 16])}
            assert runs(got[3].tolist(), got[4].tolist()) == runs(want[3].tolist(), want[4].tolist())
    assert not lib.route_linear_ok(h, 65, 65) and not lib.route_linear_ok(h[:, :k - 64].contiguous(), rows, outputs)
    assert not lib.route_linear_ok(h.float(), rows, outputs)



@pytest.mark.parametrize("experts,n,one", [(16, 16, True), (17, 8, True), (32, 8, True), (32, 9, False), (33, 1, False), (64, 4, False)])
def test_routers_of_many_rows_keep_a_product_of_their_own(lib, monkeypatch, experts, n, one):
    """On either side of where one workgroup is no faster any more; the outputs are the same bits."""
    gen = torch.Generator().manual_seed(experts + n)
    params = {"experts": experts, "top": 2, "intermediate_size": 32, "limit": 7.0}
    part = build_part("feed_forward", PartSpec("routed_experts", params), BuildEnv(hidden_size=1024, dtype=torch.bfloat16, device=torch.device(DEV), lib=lib))
    part.load({name: (torch.randn(ts.shape, generator=gen) * 0.03).to(torch.float32 if ts.role == "gain" else torch.bfloat16).to(DEV)
               for name, ts in part.tensor_specs().items()})
    h = torch.randn(n, 1024, generator=gen).bfloat16().to(DEV)
    calls, real = [], lib.route_linear
    monkeypatch.setattr(lib, "route_linear", lambda *a, **kw: (calls.append(1), real(*a, **kw)))
    got = part.forward(h)
    assert bool(calls) == one
    monkeypatch.setattr(type(lib), "route_linear_pays", staticmethod(lambda *a: not one))
    assert torch.equal(part.forward(h), got)


# ---------------------------------------------------------------------------- products of few tokens: packed loads, halves of tiles
@pytest.mark.parametrize("n,k", [(16, 128), (48, 384), (2048, 1024), (2064, 256), (1040, 2048), (96, 8192), (544, 5120), (4112, 128)])
def test_a_row_of_a_product_has_the_same_bits_however_its_operands_are_loaded(lib, n, k):
    """4, 2 or 1 blocks of the tokens a load by how many tokens there are, whole tiles of W and halves: 16 tokens with whole tiles, a block a load, and
    the same rows among fewer, for every end.  (That those are right: the tests against float64 above and in test_kernels_gpu.py.)"""
    gen = torch.Generator().manual_seed(n + k)
    x = torch.randn(16, k, generator=gen).bfloat16().to(DEV)
    rows = (torch.randn(n, k, generator=gen) * k ** -0.5).bfloat16().to(DEV)
    w = torch.empty_like(rows)
    lib.place_rows(rows, w, frag=True)
    act, gain = torch.tensor([0.3, -0.2], device=DEV), torch.randn(n, generator=gen).to(DEV)
    before, squares = torch.randn(16, n, generator=gen).to(DEV), torch.rand(16, (k + 15) // 16, generator=gen).to(DEV) * 16

    def all_ends(m, pick=None):
        at = slice(0, m) if pick is None else pick
        outs = []
        for dtype, epilogue, a in ((torch.float32, 0, None), (torch.bfloat16, 0, act), (torch.bfloat16, 1, None)):
            if epilogue == 1 and n % 32:
                continue
            out = torch.empty(m, n // 2 if epilogue == 1 else n, dtype=dtype, device=DEV)
            lib.gemm_bf16(x[at].contiguous(), w, out, epilogue, w_frag=True, act=a)
            outs.append(out)
        if lib.gemm_bf16_few_ok(m, n, k):
            for epilogue in (2, 3):
                out, g, s = before[at].clone(), torch.zeros(m, n, dtype=torch.bfloat16, device=DEV), torch.zeros(m, (n + 15) // 16, device=DEV)
                lib.gemm_bf16_few(x[at].contiguous(), w, out, epilogue, w_frag=True, **(dict(gain=gain, gained=g, squares_out=s) if epilogue == 3 else {}))
                outs += [out, g, s]
            out = torch.empty(m, n, device=DEV)
            chosen = None if pick is None else torch.tensor(pick, dtype=torch.int32, device=DEV)
            lib.gemm_bf16_few(x if pick is not None else x[at].contiguous(), w, out, 0, squares=squares if pick is not None else squares[at].contiguous(), eps=1e-5,
                              rows=chosen, w_frag=True)
            outs.append(out)
        return outs
    try:
        lib._lib.rb_tune_parts(1)
        whole = all_ends(16)
        for parts in (0, 1, 2):
            lib._lib.rb_tune_parts(parts)
            for m, pick in ((16, None), (9, None), (8, None), (5, None), (4, None), (3, None), (1, None), (3, [7, 2, 11]), (6, [15, 0, 3, 3, 9, 1])):
                for got, want in zip(all_ends(m, pick), whole):
                    assert torch.equal(got, want[:m] if pick is None else want[pick]), (parts, m, pick)
    finally:
        lib._lib.rb_tune_parts(0)


@pytest.mark.parametrize("n,k", [(2064, 1280), (9216, 5120)])
def test_a_row_of_a_product_has_the_same_bits_whether_its_operands_are_set_aside(lib, n, k):
    """As above where 9 to 16 tokens set their operands aside with one row tile a wave, with two and with four, and 8 and fewer do not."""
    assert lib._lib.rb_tune_few_aside(n, k, 1) and lib._lib.rb_tune_few_aside(n, k, 2)
    test_a_row_of_a_product_has_the_same_bits_however_its_operands_are_loaded(lib, n, k)


# ---------------------------------------------------------------------------- splits of attention put together by the product that reads them
@pytest.mark.parametrize("n", [1, 4, 7, 8])
@pytest.mark.parametrize("heads,width,k,n_out,splits,sink,gated", [(16, 128, 128, 128, 2, True, False), (32, 128, 96, 64, 16, False, True),
                                                                   (3, 64, 64, 16, 5, False, False), (2, 128, 32, 272, 70, True, True), (1, 64, 32, 64, 9, False, True)])
def test_splits_put_together_by_the_product_per_head_give_the_bits_of_two_launches(lib, n, heads, width, k, n_out, splits, sink, gated):
    gen = torch.Generator().manual_seed(heads + n)
    lengths = [(97 * i) % 400 + 1 for i in range(n)]         # fewer pages than splits: some are empty
    pages, table, _ = _paged(lengths, 1, width, gen)
    pos = torch.tensor([m - 1 for m in lengths], dtype=torch.int32, device=DEV)
    q = torch.randn(n, heads, width, generator=gen).bfloat16().to(DEV)
    rows = (torch.randn(heads * n_out, k, generator=gen) * k ** -0.5).bfloat16().to(DEV)
    w = torch.empty(heads, n_out, k, dtype=torch.bfloat16, device=DEV)
    lib.place_rows(rows, w.view(-1, k), frag=True)
    sinks = torch.randn(heads, generator=gen).to(DEV) if sink else None
    gate = torch.randn(n, heads + 3, generator=gen).to(DEV) if gated else None
    assert lib.heads_combined_ok(n, splits, width, n_out, k, True)
    assert not lib.heads_combined_ok(9, splits, width, n_out, k, True) and not lib.heads_combined_ok(n, 1, width, n_out, k, True)
    ws = [torch.full((n * heads * splits * (width + 2),), float("nan"), device=DEV) for _ in range(2)]
    attend = lambda out, scratch: lib.attention_decode_bf16(q, pages.bfloat16().to(DEV), pages.bfloat16().to(DEV), out, pos, table.to(DEV), heads, 1, width, 0.1,
                                                            None, splits, scratch, sinks=sinks)
    x, want, got = torch.empty(n, heads * width, dtype=torch.bfloat16, device=DEV), *(torch.empty(n, heads * n_out, dtype=torch.bfloat16, device=DEV) for _ in range(2))
    attend(x, ws[0])
    lib.heads_linear_part(x, width, w, want, n_out, gate=gate, gate_col=2, w_frag=True)
    attend(None, ws[1])
    lib.heads_combined(ws[1], splits, sinks, width, w, got, n_out, gate=gate, gate_col=2)
    assert torch.isfinite(want.float()).all() and torch.equal(got, want)


@pytest.mark.parametrize("n,k", [(16, 128), (48, 384), (2048, 256), (2064, 512), (1040, 2048), (96, 8192), (4096, 640), (4112, 128), (6144, 384)])
def test_a_row_of_a_float32_product_has_the_same_bits_however_its_operands_are_loaded(lib, n, k):
    """As above, with one and two stages in registers besides (up to and beyond a workgroup a compute unit); against float64 as well: a sum of K products
    is off by K 2^-24 of the sum of their sizes at the most."""
    gen = torch.Generator().manual_seed(n + k)
    x, rows = torch.randn(16, k, generator=gen), torch.randn(n, k, generator=gen) * k ** -0.5
    w = torch.empty(n, k, device=DEV)
    lib.place_rows(rows.to(DEV), w, frag=True)

    def product(m):
        out = torch.full((m, n), float("nan"), device=DEV)
        lib.gemm_generic(x[:m].contiguous().to(DEV), w, out, w_frag=True)
        return out
    try:
        lib._lib.rb_tune_f32_parts(1)
        whole = product(16)
        _within(whole, x.double() @ rows.double().T, k * 2.0 ** -24 * (x.double().abs() @ rows.double().abs().T))
        for parts in (0, 1, 2):
            lib._lib.rb_tune_f32_parts(parts)
            for units in (0, 1, 1024):                       # workgroups that share a compute unit, and none that do
                lib._lib.rb_tune_compute_units(units)
                for m in (16, 9, 8, 5, 4, 1):
                    assert torch.equal(product(m), whole[:m]), (parts, units, m)
    finally:
        lib._lib.rb_tune_f32_parts(0)
        lib._lib.rb_tune_compute_units(0)


@pytest.mark.parametrize("ff,k,frag", [(16, 128, True), (256, 96, False), (48, 500, False), (4096, 100, False), (2048, 512, True), (4112, 768, True), (1024, 3072, True),
                                       (80, 8192, True)])
def test_a_float32_gate_on_its_products_sums_gives_the_bits_of_two_launches(lib, ff, k, frag):
    gen = torch.Generator().manual_seed(ff + k)
    rows = torch.randn(2 * ff, k, generator=gen) * k ** -0.5
    rows[:8] *= 300.0                                        # gates whose exponentials are none
    w = rows.to(DEV)
    if frag:
        w = torch.empty(2 * ff, k, device=DEV)
        lib.place_rows(rows.to(DEV), w, frag=True)
    for m in (1, 4, 5, 8, 9, 16):
        x = torch.randn(m, k, generator=gen).to(DEV)
        got, gu, want = torch.full((m, ff), float("nan"), device=DEV), torch.empty(m, 2 * ff, device=DEV), torch.empty(m, ff, device=DEV)
        if not lib.gemm_f32_gated_ok(m, ff, k, frag):
            assert not frag and k > 128 and m <= 8           # (many rows of a longer depth: another kernel's)
            continue
        lib.gemm_f32_gated(x, w, got, w_frag=frag)
        lib.gemm_generic(x, w, gu, w_frag=frag)
        lib.swiglu(gu, want)
        assert torch.isfinite(want).all() and torch.equal(got, want)
    assert not lib.gemm_f32_gated_ok(17, ff, k, frag) and not lib.gemm_f32_gated_ok(4, ff + 8, k, frag)


# ---------------------------------------------------------------------------- experts of few tokens: packed loads
@pytest.mark.parametrize("hidden,ff", [(96, 64), (64, 192), (128, 128), (384, 640), (2048, 256)])
@pytest.mark.parametrize("params", [dict(score="softmax", weight_on="output", unit="squared_relu"), dict(score="chosen", weight_on="output"),
                                    dict(limit=7.0), dict(score="softmax", weight_on="output", unit="squared_relu", shared={"intermediate_size": 128, "gate": False})])
def test_a_tokens_experts_give_the_same_bits_however_many_tokens_a_load_brings(lib, hidden, ff, params):
    """4, 2 or 1 blocks of depth a load by how many tokens there are: 16 tokens in a step, a block a load, and the same tokens in smaller ones."""
    if params.get("shared") and (hidden % 128 or ff < 128):
        params = dict(params, shared=None)
    gen = torch.Generator().manual_seed(hidden + ff)
    part = build_part("feed_forward", PartSpec("routed_experts", dict(params, experts=4, top=2, intermediate_size=ff)),
                      BuildEnv(hidden_size=hidden, dtype=torch.bfloat16, device=torch.device(DEV), lib=lib))
    part.load({name: (torch.randn(ts.shape, generator=gen) * ts.shape[-1] ** -0.5).to(torch.float32 if ts.role == "gain" else torch.bfloat16).to(DEV)
               for name, ts in part.tensor_specs().items()})
    h = torch.randn(16, hidden, generator=gen).bfloat16().to(DEV)
    want = part.forward(h)
    assert torch.isfinite(want).all()
    for at in (slice(0, 1), slice(3, 6), slice(8, 12), slice(0, 5), slice(8, 16), slice(2, 11)):
        assert torch.equal(part.forward(h[at].contiguous()), want[at])


@pytest.mark.parametrize("hidden,ff", [(96, 64), (64, 192), (384, 640)])
@pytest.mark.parametrize("params", [dict(score="softmax", weight_on="output", unit="squared_relu"), dict(score="chosen", weight_on="output"),
                                    dict(limit=7.0), dict(score="softmax", weight_on="output", unit="squared_relu", shared={"intermediate_size": 128, "gate": False})])
def test_a_token_of_nan_changes_nothing_in_the_tokens_beside_it(lib, hidden, ff, params):
    """Its router's logits are none, and it chooses the first expert every time: a run with more rows than the step has tokens."""
    if params.get("shared") and (hidden % 128 or ff < 128):
        params = dict(params, shared=None)
    gen = torch.Generator().manual_seed(hidden + ff)
    part = build_part("feed_forward", PartSpec("routed_experts", dict(params, experts=4, top=4, intermediate_size=ff)),
                      BuildEnv(hidden_size=hidden, dtype=torch.bfloat16, device=torch.device(DEV), lib=lib))
    part.load({name: (torch.randn(ts.shape, generator=gen) * ts.shape[-1] ** -0.5).to(torch.float32 if ts.role == "gain" else torch.bfloat16).to(DEV)
               for name, ts in part.tensor_specs().items()})
    h = torch.randn(16, hidden, generator=gen).bfloat16().to(DEV)
    want = part.forward(h)
    for n in (3, 4, 7, 8, 16):
        for bad in (0, 1, n - 1):
            some = h[:n].clone()
            some[bad] = float("nan")
            got, others = part.forward(some), [i for i in range(n) if i != bad]
            assert torch.equal(got[others], want[others])


# ---------------------------------------------------------------------------- a norm with the convolution behind it
@pytest.mark.parametrize("width", [4, 260, 2048, 4096])
@pytest.mark.parametrize("taps,copies,update,biased,dtype", [(2, 1, False, True, torch.bfloat16), (3, 2, True, True, torch.float32),
                                                             (4, 2, True, False, torch.bfloat16), (4, 3, True, True, torch.bfloat16), (4, 4, False, True, torch.bfloat16)])
def test_a_norm_with_the_convolution_behind_it_gives_the_bits_of_two_launches(lib, width, taps, copies, update, biased, dtype):
    gen = torch.Generator().manual_seed(width + taps)
    n, r = 5, lambda *shape: torch.randn(*shape, generator=gen).to(DEV)
    x, coef, weight, bias, w = r(copies, n, width), r(copies), r(width), r(width) if biased else None, r(width, taps)
    todo = (r(copies, copies), r(copies), r(n, width), r(width)) if update else None
    state, slots = r(7, taps - 1, width), torch.tensor([3, 0, 6, 1, 4], dtype=torch.int32, device=DEV)
    ctx = SimpleNamespace(n_tokens=n, n_seqs=n, max_q_len=1, slots=slots, tok_pos=torch.zeros(n, dtype=torch.int32, device=DEV),
                          tok_seq=torch.arange(n, dtype=torch.int32, device=DEV), cu_seqlens=torch.arange(n + 1, dtype=torch.int32, device=DEV))
    assert lib.streams_conv_ok(width, taps) and not lib.streams_conv_ok(4100, taps) and not lib.streams_conv_ok(width, 5)
    one, two = (tuple(t.clone() for t in (x, state)) for _ in range(2))
    got, want, row = torch.empty(n, width, dtype=dtype, device=DEV), torch.empty(n, width, dtype=dtype, device=DEV), torch.empty(n, width, device=DEV)
    lib.streams_layernorm(one[0], coef, weight, bias, 1e-5, None, got, update=todo, conv=(w, one[1], ctx))
    lib.streams_layernorm(two[0], coef, weight, bias, 1e-5, None, row, update=todo)
    lib.short_conv(row, 0, width, w, two[1], ctx, want, True, 0)
    for a, b in ((got, want), (one[0], two[0]), (one[1], two[1])):
        assert torch.equal(a, b)
    odd = torch.empty(width * taps + 1, device=DEV)[1:].view(width, taps)      # weights at an odd address go in two launches
    odd.copy_(w)
    x2, s2 = x.clone(), state.clone()
    lib.streams_layernorm(x2, coef, weight, bias, 1e-5, None, got, update=todo, conv=(odd, s2, ctx))
    assert torch.equal(got, want) and torch.equal(s2, two[1])


# ---------------------------------------------------------------------------- a shared expert in the chosen experts' launches
@pytest.mark.parametrize("n", [1, 4, 16, 17])
@pytest.mark.parametrize("hidden,ff,shared,along", [(128, 128, 128, True), (384, 256, 128, True), (2048, 1024, 1024, True), (1152, 640, 640, True),
                                                    (256, 128, 256, False), (256, 192, 160, False)])
def test_a_shared_expert_in_the_chosen_experts_launches_gives_the_bits_of_its_own(lib, n, hidden, ff, shared, along):
    gen = torch.Generator().manual_seed(hidden + n)
    params = {"experts": 4, "top": 2, "intermediate_size": ff, "score": "softmax", "weight_on": "output", "unit": "squared_relu",
              "shared": {"intermediate_size": shared, "gate": False}}
    part = build_part("feed_forward", PartSpec("routed_experts", params), BuildEnv(hidden_size=hidden, dtype=torch.bfloat16, device=torch.device(DEV), lib=lib))
    part.load({name: (torch.randn(ts.shape, generator=gen) * ts.shape[-1] ** -0.5).to(torch.float32 if ts.role == "gain" else torch.bfloat16).to(DEV)
               for name, ts in part.tensor_specs().items()})
    h = torch.randn(n, hidden, generator=gen).bfloat16().to(DEV)
    assert part.shared_along == (shared % 64 == 0)
    assert lib.routed_shared_ok(n, hidden, ff, shared) == (along and n <= 16)
    got = part.forward(h, pairs=True)
    part.shared_along = False
    want = part.forward(h, pairs=True)
    for a, b in ((got.outputs, want.outputs), (got.weights, want.weights), (got.shared, want.shared)):
        assert torch.equal(a, b)


# ---------------------------------------------------------------------------- products of few tokens in one launch
@pytest.mark.parametrize("m", [1, 4, 16])
@pytest.mark.parametrize("k", [128, 384, 2048, 8192])
@pytest.mark.parametrize("rows,frag", [((16, 64, 1024), True), ((1, 37, 16, 250, 3), False), ((4096, 1024, 16, 16, 16, 16), True), ((2050,), False)])
def test_products_in_one_launch(lib, m, k, rows, frag):
    """Products of inputs, matrices and ends of their own against each in float64: a float32 sum of K products of bfloat16 numbers is off
    by K 2^-24 of the sum of their sizes at the most, and bfloat16 results by half a unit in their last place besides."""
    gen = torch.Generator().manual_seed(k + m + len(rows))
    ends = ["float32", "bfloat16", "tanh"]
    products, wants = [], []
    for i, n in enumerate(rows):
        x = torch.randn(m, k, generator=gen).to(torch.bfloat16)
        w = (torch.randn(n, k, generator=gen) * k ** -0.5).to(torch.bfloat16)
        end, wd = ends[(i + m) % 3], w.to(DEV)
        if frag:
            rows_of, wd = wd, torch.empty_like(wd)
            lib.place_rows(rows_of, wd, frag=True)
        want, size = x.double() @ w.double().T, k * 2.0 ** -24 * (x.double().abs() @ w.double().abs().T)
        if end == "tanh":
            want = want.tanh()
        wants.append((want, size + (0 if end == "float32" else 2.0 ** -8 * want.abs()) + 1e-7))
        products.append((x.to(DEV), wd, torch.full((m, n), 9.0, dtype=torch.float32 if end == "float32" else torch.bfloat16, device=DEV), end))
    lib.gemm_bf16_group(products, frag)
    for (_, _, c, _), (want, bound) in zip(products, wants):
        _within(c, want, bound)
    assert not lib.gemm_bf16_group_ok(17, 128) and not lib.gemm_bf16_group_ok(4, 192)


@pytest.mark.parametrize("m", [1, 16])
@pytest.mark.parametrize("k,rows", [(128, (16, 4112)), (2048, (6160, 256, 1024)), (4096, (4096, 4112, 64)), (4096, (8192, 8208)), (5120, (5120, 1024)),
                                    (8192, (4112, 16))])
def test_products_in_one_launch_give_the_bits_of_each_alone(lib, m, k, rows):
    """Wherever a product is said to gain among others its sums are those it has alone, on either side of as many row tiles as compute
    units; what is left out (other row tiles a wave, resident tokens) goes alone."""
    gen = torch.Generator(device=DEV).manual_seed(k + m)
    x = torch.randn(m, k, generator=gen, device=DEV).bfloat16()
    ws = [torch.randn(n, k, generator=gen, device=DEV).bfloat16() for n in rows]
    pays = [lib.gemm_bf16_group_pays(m, n, k) for n in rows]
    if k in (128, 2048, 8192):
        assert all(pays)
    assert lib.gemm_bf16_group_pays(m, 8192, 4096) and not lib.gemm_bf16_group_pays(m, 8208, 4096)
    assert not lib.gemm_bf16_group_pays(17, 64, 2048) and not lib.gemm_bf16_group_pays(m, 64, 192)
    alone, ends = [], ["float32", "bfloat16", "tanh"]
    for w in ws:
        c = torch.empty(m, w.shape[0], device=DEV)
        lib.gemm_bf16(x, w, c, 0)
        alone.append(c)
    end = lambda i: "float32" if not pays[i] else ends[i % 3]
    got = [torch.empty(m, w.shape[0], dtype=torch.float32 if end(i) == "float32" else torch.bfloat16, device=DEV) for i, w in enumerate(ws)]
    lib.gemm_bf16_group([(x, w, c, end(i)) for i, (w, c) in enumerate(zip(ws, got))], False)
    for i, (c, a) in enumerate(zip(got, alone)):
        if not pays[i]:
            continue
        if end(i) == "tanh":
            z, a = a, torch.empty_like(c)
            lib.tanh_cast(z, a)
        assert torch.equal(c, a.to(c.dtype)), rows[i]


@pytest.mark.parametrize("m", [1, 4, 5, 8, 9, 16])
@pytest.mark.parametrize("k,rows", [(128, (16, 1024)), (256, (1024,) * 5), (768, (768, 48)), (1024, (16, 4096)), (2048, (16, 1040)), (2048, (4096, 64)), (2560, (2560, 16)),
                                    (4096, (2048, 128)), (8192, (6144, 1024))])
def test_products_in_one_launch_give_the_bits_of_each_alone_however_tokens_are_loaded(lib, m, k, rows):
    gen = torch.Generator(device=DEV).manual_seed(k + m)
    products, alone = [], []
    for n in rows:
        x, plain = torch.randn(m, k, generator=gen, device=DEV).bfloat16(), torch.randn(n, k, generator=gen, device=DEV).bfloat16()
        w = torch.empty_like(plain)
        lib.place_rows(plain, w, frag=True)
        products.append((x, w, torch.full((m, n), 9.0, device=DEV), "float32"))
        alone.append(torch.empty(m, n, device=DEV))
        assert lib.gemm_bf16_group_pays(m, n, k)
        lib.gemm_bf16(x, w, alone[-1], 0, w_frag=True)
    lib.gemm_bf16_group(products, True)
    for (_, _, c, _), want in zip(products, alone):
        assert torch.equal(c, want)


# ---------------------------------------------------------------------------- float32 products of few tokens: sums and norms in their launches
@pytest.mark.parametrize("n,k,frag", [(16, 128, True), (96, 96, False), (257, 96, False), (90, 500, False), (384, 1000, False), (130, 384, False), (2048, 512, True),
                                      (4096, 768, True), (4112, 1280, True), (3072, 3072, True), (256, 8192, True)])
def test_float32_products_of_few_tokens_take_sum_and_norm_along(lib, n, k, frag):
    """Against the same in 64 bits.  A product's error is at most (K + 3) units of 2^-24 of its sum of magnitudes, a random walk of them in fact:
    2^-24 sqrt(K) times that sum covers it and the few more roundings (residual sum, gain, factor)."""
    gen = torch.Generator().manual_seed(n + k)
    rows = torch.randn(n, k, generator=gen) * k ** -0.5
    w = rows.to(DEV)
    if frag:
        w = torch.empty(n, k, device=DEV)
        lib.place_rows(rows.to(DEV), w, frag=True)
    unit, eps = 2.0 ** -24 * max(4.0, k ** 0.5), 1e-5
    nan = float("nan")

    def close(got, want, size):
        assert torch.isfinite(got).all()
        assert ((got.double().cpu() - want).abs() <= unit * size).all()

    for m in (1, 4, 5, 8, 9, 16):
        if not lib.gemm_f32_few_ok(m, n, k, frag, 0):
            assert not frag and k > 128 and m <= 8           # (many rows of a longer depth: another kernel's)
            continue
        x, gain, before = torch.randn(m + 2, k, generator=gen) * 3.0, torch.randn(k, generator=gen), torch.randn(m, n, generator=gen)
        x[0] *= 1e-4                                         # (a row that eps decides)
        gained = (x * gain).to(DEV)
        padded = torch.zeros(m + 2, (k + 7) // 8 * 8)
        padded[:, :k] = x * x
        squares = padded.view(m + 2, -1, 8).sum(-1).to(DEV)
        pick = torch.randperm(m + 2, generator=gen)[:m].to(torch.int32)
        # rows that a norm prepared, all of the step's or some of them
        for rows_of, src in ((None, torch.arange(m)), (pick, pick.long())):
            normed = (x.double() * gain.double() / (x.double().square().mean(-1, keepdim=True) + eps).sqrt())[src]
            got = torch.full((m, n), nan, device=DEV)
            a = gained if rows_of is not None else gained[:m].contiguous()
            lib.gemm_f32_few(a, w, got, 0, squares=squares if rows_of is not None else squares[:m].contiguous(), eps=eps,
                             rows=None if rows_of is None else rows_of.to(DEV), w_frag=frag)
            close(got, normed @ rows.double().T, normed.abs() @ rows.double().abs().T)
        # the residual sum, and what the next norm needs; columns at whole vectors and not
        g2 = torch.randn(n, generator=gen)
        want = before.double() + x[:m].double() @ rows.double().T
        size = before.double().abs() + x[:m].double().abs() @ rows.double().abs().T
        for off in (0, 1):
            c = torch.empty(m * n + off, device=DEV)[off:].view(m, n)
            c.copy_(before)
            alone = c.clone()
            out, sq = torch.full((m, n), nan, device=DEV), torch.full((m, (n + 7) // 8), nan, device=DEV)
            lib.gemm_f32_few(x[:m].contiguous().to(DEV), w, c, 3, gain=g2.to(DEV), gained=out, squares_out=sq, w_frag=frag)
            close(c, want, size)
            assert torch.equal(out, c * g2.to(DEV))
            full = torch.zeros(m, (n + 7) // 8 * 8, dtype=torch.float64)
            full[:, :n] = c.double().cpu().square()
            torch.testing.assert_close(sq.double().cpu(), full.view(m, -1, 8).sum(-1), rtol=8 * 2.0 ** -24, atol=0.0)
            lib.gemm_f32_few(x[:m].contiguous().to(DEV), w, alone, 2, w_frag=frag)
            assert torch.equal(alone, c)
        # the gate on prepared rows
        if n % 32 == 0 and lib.gemm_f32_few_ok(m, n, k, frag, 1):
            got = torch.full((m, n // 2), nan, device=DEV)
            normed = x[:m].double() * gain.double() / (x[:m].double().square().mean(-1, keepdim=True) + eps).sqrt()
            lib.gemm_f32_few(gained[:m].contiguous(), w, got, 1, squares=squares[:m].contiguous(), eps=eps, w_frag=frag)
            g, u = (normed @ rows.double().T).split(n // 2, dim=1)
            sg, su = (normed.abs() @ rows.double().abs().T).split(n // 2, dim=1)
            close(got, g * torch.sigmoid(g) * u, 1.1 * sg * u.abs() + (g.abs() + 1.0) * su)
    assert not lib.gemm_f32_few_ok(17, n, k, frag, 0) and not lib.gemm_f32_few_ok(4, n, k + 2, frag, 2)


@pytest.mark.parametrize("k,frag", [(96, False), (128, True), (1000, False), (1024, True), (2048, True)])
def test_float32_products_multiply_by_a_norms_factor_as_64_bits_have_it(lib, k, frag):
    """Rows of W that pick a column each, sums of squares that float32 adds up exactly: what is left is the rounding of the result, half a unit of 2^-23, and
    what one step from the root's estimate of 2^-23 leaves (2^-45).  An infinite sum of squares makes zeros, as the norm's own launch does."""
    gen = torch.Generator().manual_seed(k)
    pick = torch.randperm(k, generator=gen)[:64]
    rows = torch.zeros(64, k)
    rows[torch.arange(64), pick] = 1.0
    w = rows.to(DEV)
    if frag:
        w = torch.empty(64, k, device=DEV)
        lib.place_rows(rows.to(DEV), w, frag=True)
    for m in (1, 4, 8, 16):
        if not lib.gemm_f32_few_ok(m, 64, k, frag, 0):
            continue
        for eps in (1e-5, 0.0):
            gained = torch.randn(m, k, generator=gen)
            squares = torch.randint(1, 4096, (m, (k + 7) // 8), generator=gen).float()
            want = gained[:, pick].double() / (squares.double().sum(-1, keepdim=True) / k + torch.tensor(eps).double()).sqrt()
            if m == 4:
                squares[2] = float("inf")
                want[2] = 0.0
            got = torch.full((m, 64), float("nan"), device=DEV)
            lib.gemm_f32_few(gained.to(DEV), w, got, 0, squares=squares.to(DEV), eps=eps, w_frag=frag)
            assert ((got.double().cpu() - want).abs() <= 2.0 ** -24 * 1.00001 * want.abs()).all()


# ---------------------------------------------------------------------------- a norm that adds up the outputs of a token's experts
@pytest.mark.parametrize("width", [4, 101, 2048, 4104])
@pytest.mark.parametrize("terms", [1, 2, 3, 4, 5, 9])
def test_a_norm_adds_up_the_outputs_of_a_tokens_experts_to_the_bits_of_two_launches(lib, width, terms):
    gen = torch.Generator().manual_seed(width + terms)
    r = lambda *shape: torch.randn(*shape, generator=gen).to(DEV)
    n, rows = 5, torch.tensor([4, 0, 3], dtype=torch.int32, device=DEV)
    x, a, pairs, weight, bias = r(n, width), r(n, width), r(n * terms, width), r(width), r(width)
    total = torch.empty(n, width, device=DEV)
    if terms > 1:
        lib.pairs_sum(pairs, terms, total)
    else:
        total.copy_(pairs)
    for some in (None, rows):
        for dtype in (torch.float32, torch.bfloat16):
            one, two = x.clone(), x.clone()
            got, want = (torch.full((n if some is None else 3, width), float("nan"), dtype=dtype, device=DEV) for _ in range(2))
            lib.layernorm_residual(one, a, pairs.view(n, terms, width), 0.6, weight, bias, 1e-5, some, got)
            lib.layernorm_residual(two, a, total, 0.6, weight, bias, 1e-5, some, want)
            assert torch.isfinite(want.float()).all() and torch.equal(got, want) and torch.equal(one, two)
            assert torch.equal(one, x) == (some is not None)


# ---------------------------------------------------------------------------- products of several depths in one launch
@pytest.mark.parametrize("m", [1, 4, 7, 16])
@pytest.mark.parametrize("sizes", [((2048, 2048), (2048, 1024)), ((16, 128), (4112, 4096), (64, 384)), ((1024, 8192), (1024, 128))])
def test_products_of_several_depths_in_one_launch_give_the_bits_of_each_alone(lib, m, sizes):
    gen = torch.Generator(device=DEV).manual_seed(m + sizes[0][1])
    products, alone = [], []
    for n, k in sizes:
        x, rows = torch.randn(m, k, generator=gen, device=DEV).bfloat16(), (torch.randn(n, k, generator=gen, device=DEV) * k ** -0.5).bfloat16()
        w, c = torch.empty_like(rows), torch.empty(m, n, device=DEV)
        lib.place_rows(rows, w, frag=True)
        lib.gemm_bf16(x, w, c, 0, w_frag=True)
        alone.append(c if lib.gemm_bf16_group_pays(m, n, k) else None)
        products.append((x, w, torch.full((m, n), float("nan"), device=DEV), "float32"))
    assert any(c is not None for c in alone)
    lib.gemm_bf16_group(products, True)
    for (_, _, got, _), want in zip(products, alone):
        assert want is None or torch.equal(got, want)
    with pytest.raises(KernelError):
        lib.gemm_bf16_group([products[0], (products[0][0][:, :96].contiguous(), products[0][1][:, :96].contiguous(), products[0][2], "float32")], True)
