"""The linear-attention work split: segments and ranges cover the chunks, one
workgroup per CU, never dearer than the long segments by its own time model."""

import pytest

from nkipy_amd.dispatch import launchers as LA


@pytest.mark.parametrize("bh", [1, 3, 8, 24, 64, 127, 128, 129, 256, 1000])
@pytest.mark.parametrize("chunks", [1, 2, 7, 12, 16, 97, 128, 160, 1024])
def test_split_covers_the_sequence(bh, chunks):
    nseg, rchunks, nranges = LA.linear_attention_split(bh, 64 * chunks)
    long = LA._linattn_long_split(bh, 64 * chunks)
    assert chunks % nseg == 0 and (chunks // nseg) % rchunks == 0
    assert nranges == (nseg - 1) * (chunks // nseg // rchunks)
    assert (nseg, rchunks) == long or (2 <= nseg and bh * nseg <= LA.LINATTN_TARGET_WGS)
    cost = LA._linattn_cost(bh, chunks, nseg, rchunks)
    assert (nseg, rchunks) == long or cost < LA._linattn_cost(bh, chunks, *long)
    assert LA.linear_attention_workspace_bytes(bh, 64 * chunks) >= bh * nranges * 129 * 128 * 4
