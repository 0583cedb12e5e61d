"""Which kernels the products of a step's few tokens go to, over sizes: rules that no result shows, for a GPU of 256 compute units."""
import ctypes

import pytest
import torch

from rbitnet_amd.csrc import build
from rbitnet_amd.parts import linear


@pytest.fixture(scope="module")
def lib():
    lib = ctypes.CDLL(build.ensure_built())
    lib.rb_tune_compute_units(256)
    yield lib
    lib.rb_tune_compute_units(0)


# rows, K, end, prepared by a norm -> blocks of depth a load of 4 and of 8 tokens, and what a load of the other kind took longer where that was timed
@pytest.mark.parametrize("n,k,end,prepared,four,eight", [
    (3072, 3072, 0, 0, 4, 2), (6144, 4096, 2, 0, 4, 2), (4096, 14336, 3, 0, 4, 2), (8192, 8192, 1, 0, 4, 2),
    (2048, 2048, 0, 1, 1, 1), (6144, 4096, 0, 1, 1, 1), (8192, 8192, 0, 1, 1, 1),          # 2, 1 and 5 %
    (5120, 5120, 0, 1, 4, 2), (10240, 8192, 0, 1, 4, 2),                                  # 5 and 1 %
    (8192, 2048, 1, 1, 1, 1), (8192, 8192, 1, 1, 1, 1), (57344, 8192, 1, 1, 1, 2),         # 2, 5 and 2 %
    (4096, 4096, 1, 1, 4, 2), (4096, 14336, 1, 1, 4, 2),                                  # 4 and 5 %
    (12288, 8192, 0, 0, 1, 1), (10240, 8192, 3, 0, 1, 1), (12288, 7168, 0, 0, 4, 2),       # 5, 3 and 4 %
    (16384, 8192, 3, 0, 1, 1), (16384, 6144, 3, 0, 4, 2), (15360, 5120, 0, 0, 1, 1),       # 4, 1 and 2 %
    (12288, 6144, 1, 0, 4, 2), (16384, 6144, 1, 0, 1, 1),                                 # 4 and 1 %
    (3072, 1024, 0, 0, 4, 1), (3072, 1024, 2, 0, 4, 1), (3072, 1024, 1, 0, 4, 1),          # 5, 4 and 4 % (8 tokens)
    (2560, 1280, 0, 0, 4, 2), (2560, 1280, 1, 0, 4, 2), (27648, 5120, 1, 0, 4, 2), (27648, 5120, 0, 1, 1, 1),      # 5, 6, 7 and 4 %
])
def test_tokens_are_packed_where_that_was_the_faster_load(lib, n, k, end, prepared, four, eight):
    blocks = [lib.rb_tune_few_blocks(m, n, k, end, prepared) for m in (1, 4, 5, 8, 9, 16)]
    assert blocks == [four, four, eight, eight, 1, 1]


# rows, K, end -> workgroups a tile of 16 rows for 1, 4, 8, 9 and 16 tokens, and what the other number took longer
@pytest.mark.parametrize("n,k,end,parts", [
    (2048, 512, 0, (1, 1, 1, 1, 1)), (2048, 768, 0, (1, 2, 2, 1, 1)), (2048, 1024, 0, (2, 2, 2, 1, 1)), (1024, 1280, 0, (2, 2, 2, 2, 2)),      # 5, 7, 8 and 7 %
    (2048, 512, 2, (1, 1, 2, 2, 2)), (2048, 896, 2, (2, 2, 2, 1, 1)), (2048, 2048, 2, (2, 2, 2, 2, 2)), (2064, 2048, 0, (1, 1, 1, 1, 1)),      # 8, 5, 7 and 6 %
])
def test_a_tile_of_rows_has_two_workgroups_where_that_was_the_faster(lib, n, k, end, parts):
    assert tuple(lib.rb_tune_few_parts(m, n, k, end) for m in (1, 4, 8, 9, 16)) == parts


# rows, K -> whether products of 9 to 16 tokens set their operands aside: stored, the gate, added to C, and with the next norm's rows; what the other way took longer
@pytest.mark.parametrize("n,k,aside", [
    (3072, 512, (0, 0, 1, 1)), (3072, 896, (0, 0, 0, 0)), (4096, 1024, (0, 0, 0, 0)), (3072, 1152, (1, 1, 1, 1)), (2560, 1280, (1, 1, 1, 1)),      # 10, 6, 9, 6 and 13 %
    (6144, 4096, (0, 1, 1, 0)), (8192, 8192, (1, 1, 1, 1)), (57344, 8192, (1, 1, 0, 1)),                                     # 9, 10 and 11 %
    (10240, 8192, (0, 1, 1, 0)), (16384, 8192, (0, 0, 1, 0)),                                                              # 5 and 20 %
])
def test_operands_are_set_aside_where_that_was_the_faster(lib, n, k, aside):
    assert tuple(lib.rb_tune_few_aside(n, k, end) for end in range(4)) == aside


# K, row tiles -> 4 or 2 blocks a load, 1: one, multiplied where it was loaded, 0: set aside, for 1, 4, 5, 8, 9 and 16 tokens, and what another took longer
@pytest.mark.parametrize("k,tiles,forms", [
    (768, 99, (1, 1, 1, 1, 1, 1)), (1024, 68, (4, 4, 1, 1, 1, 1)), (1024, 260, (4, 4, 2, 2, 1, 1)),       # 7, 2 to 6 and 2 to 3 %
    (256, 320, (4, 4, 2, 2, 0, 0)), (1536, 262, (4, 4, 2, 2, 0, 0)), (2560, 323, (4, 4, 0, 0, 1, 1)),       # 8, 3 and 2 to 4 %
    (2048, 209, (0, 0, 0, 0, 1, 1)), (2048, 401, (0, 0, 0, 0, 1, 1)), (4096, 136, (4, 4, 2, 2, 1, 1)), (4096, 401, (4, 4, 0, 0, 1, 1)),       # 2, 4, 2 and 4 %
    (8192, 260, (4, 4, 2, 2, 1, 1)), (8192, 448, (1, 1, 1, 1, 1, 1)),                                    # 7 and 2 to 3 %
])
def test_products_in_one_launch_load_their_tokens_as_was_the_faster(lib, k, tiles, forms):
    assert tuple(lib.rb_tune_group_form(m, k, tiles) for m in (1, 4, 5, 8, 9, 16)) == forms


# units, K, stored fragment-major -> whether 1, 8, 9 and 16 float32 tokens go through gate, way up and the gate in one launch, and what the other way took longer
@pytest.mark.parametrize("ff,k,frag,one", [
    (1024, 512, 1, (1, 1, 1, 1)), (256, 96, 0, (1, 1, 1, 1)), (5120, 500, 0, (0, 0, 1, 1)),            # 22, 50 and 24 % (9 tokens)
    (1024, 1024, 1, (0, 0, 0, 0)), (1024, 4096, 1, (0, 0, 0, 0)), (2048, 8192, 1, (0, 0, 0, 0)), (2048, 1000, 0, (0, 0, 0, 0)),      # 18, 70, 40 and 4 %
    (3072, 4096, 1, (1, 1, 1, 1)), (4096, 3072, 1, (1, 1, 1, 1)), (8192, 3072, 1, (1, 1, 1, 1)),       # 12, 9 and 5 %
    (5120, 3072, 1, (0, 0, 0, 0)), (6144, 8192, 1, (0, 0, 0, 0)), (14336, 4096, 1, (0, 0, 0, 0)),      # 7 to 20, 9 to 20, 0 to 8 %
    (5120, 1024, 1, (1, 1, 0, 0)), (16384, 4096, 1, (1, 1, 1, 1)),
])
def test_the_float32_gate_is_in_its_products_launch_where_no_unit_gets_more_rows(lib, ff, k, frag, one):
    assert tuple(lib.rb_gemm_f32_gated_pays(m, ff, k, frag) for m in (1, 8, 9, 16)) == one
    assert lib.rb_gemm_f32_gated_pays(17, ff, k, frag) == 0


def test_a_second_float32_stage_is_under_way_where_that_was_the_faster(lib):
    """By tiles of 16 rows: up to which number of tokens (3 to 11 % at 200 tiles and 1 to 6 % at 224 with up to 8; 240 and 256 gain nothing)."""
    for tiles, most in ((1, 12), (136, 12), (192, 12), (200, 8), (208, 8), (224, 8), (225, 0), (240, 0), (256, 0), (1024, 0)):
        for n in (16 * tiles, 16 * tiles - 15):
            assert [m for m in range(1, 17) if lib.rb_tune_f32_ahead(m, n)] == list(range(1, most + 1)), tiles


def test_a_float32_norm_is_left_to_its_products_where_that_was_the_faster(lib):
    for width, most in ((96, 16), (2048, 16), (2052, 8), (3072, 8), (3076, 0), (4096, 0), (5120, 0)):
        assert [m for m in range(0, 18) if lib.rb_gemm_f32_fold_pays(m, width)] == list(range(1, most + 1)), width


def test_float32_products_with_their_neighbours_refuse_operands_between_whole_pieces_of_16_bytes(lib):
    """Host checks in front of the launch (addresses that nothing reads)."""
    lib.rb_last_error.restype = ctypes.c_char_p
    at, p, f = 1 << 20, ctypes.c_void_p, ctypes.c_float
    for a, w, squares in ((at + 4, at, at), (at, at + 8, at), (at, at, at + 4)):
        assert lib.rb_gemm_f32_few(p(a), p(squares), f(1e-5), None, p(w), 1, p(at), 0, None, None, None, 4, 128, 128, None) != 0
        assert b"16-byte aligned" in lib.rb_last_error()
    for a, w in ((at + 4, at), (at, at + 8)):
        assert lib.rb_gemm_f32_gated(p(a), p(w), 1, p(at), 4, 128, 128, None) != 0
        assert b"16-byte aligned" in lib.rb_last_error()


def test_float32_operands_between_whole_pieces_of_16_bytes_go_to_the_products_that_take_any(lib):
    class Products:
        calls = []
        gemm_f32_few_ok = staticmethod(lambda *sizes: True)
        gemm_f32_gated_pays = staticmethod(lambda *sizes: True)
        gemm_f32_fold_pays = staticmethod(lambda *sizes: True)

        def __getattr__(self, name):
            return lambda *args, **kwargs: self.calls.append(name)

    aligned, between = torch.zeros(4, 128), torch.zeros(4 * 128 + 1)[1:].view(4, 128)
    w, w_between, kernels = torch.zeros(128, 128), torch.zeros(128 * 128 + 1)[1:].view(128, 128), Products()
    assert aligned.data_ptr() % 16 == 0 and w.data_ptr() % 16 == 0
    for x, m, calls in ((aligned, w, ["gemm_f32_gated", "gemm_f32_few"]), (between, w, ["gemm_generic", "swiglu", "gemm_generic"]),
                        (aligned, w_between, ["gemm_generic", "swiglu", "gemm_generic"])):
        kernels.calls.clear()
        linear.gated_linear(kernels, x, m, 64, fused=False)
        linear.linear_to_stream(kernels, x, m, torch.zeros(4, 128))
        assert kernels.calls == calls
