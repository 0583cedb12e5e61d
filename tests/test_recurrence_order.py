"""In which order the workgroups of single tokens take the states of a recurrence: a rule that no result shows."""
import ctypes

import pytest

from rbitnet_amd.csrc import build


# heads, keys, values -> from how many sequences on the order of prompts is the faster, and what the other order took longer on either side
@pytest.mark.parametrize("heads,dim,vdim,most", [(16, 128, 128, 96), (32, 128, 128, 48), (8, 256, 128, 96), (4, 512, 64, 192),            # 3 to 15 and 3 to 30 %
                                                 (64, 128, 64, 8), (64, 64, 64, 16), (32, 64, 64, 32), (8, 64, 128, 64)])               # 0 to 3 and 2 to 95 %
def test_single_tokens_take_states_in_the_faster_order(heads, dim, vdim, most):
    lib = ctypes.CDLL(build.ensure_built())
    assert [n for n in range(1, 300) if lib.rb_tune_singles_by_seq(n, heads, dim, vdim)] == list(range(1, most))
