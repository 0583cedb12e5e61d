"""How many workgroups walk a (sequence, kv head) pair's pages in a single-token step, over sizes."""
import pytest

from rbitnet_amd.engine.context import decode_splits, decode_workgroups


@pytest.mark.parametrize("units", [64, 128, 256, 304])
@pytest.mark.parametrize("heads", [1, 2, 8, 32])
def test_more_workgroups_only_where_the_gpu_has_room(units, heads):
    for seqs in (1, 2, 3, 8, 16, 64, 300):
        before = 0
        for bucket in (1, 2, 4, 8, 16, 64):
            n = decode_workgroups(seqs, heads, bucket, units)
            plain = decode_splits(seqs, heads, bucket, units)
            assert plain <= n <= max(plain, 16)
            assert n == plain or n * seqs * heads <= units           # at most one a compute unit
            assert bucket > 1 or n == plain                          # short contexts: one launch and its walk
            assert n >= before                                       # longer contexts never fewer
            before = n
