"""The linear-attention work split: segments and ranges cover the chunks, one
workgroup per CU, never dearer than the long segments by its own time model."""

import ctypes

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


def test_c_abi_ignores_a_workspace_it_does_not_need():
    """A shape that needs no workspace takes any pointer as one: the shorter
    segments use it only where it is aligned and large enough.  Without a
    device the call passes its checks and stops at the missing runtime."""
    from nkipy_amd.runtime.hip import load_library

    lib = load_library()
    flag = ctypes.c_int()
    assert lib.nkh_is_initialized(ctypes.byref(flag)) == 0
    if flag.value:
        pytest.skip("the call would launch")
    bh, t, size = 24, 768, ctypes.c_size_t()
    assert LA._linattn_long_split(bh, t)[0] == 1 and LA.linear_attention_split(bh, t)[0] > 1
    assert lib.nkh_linear_attention_workspace_size(bh, t, ctypes.byref(size)) == 0
    p = 1 << 20
    codes = {lib.nkh_linear_attention(p, p, p, p, bh, t, ws, n)
             for ws, n in ((None, 0), (p, size.value), (p + 8, size.value), (p + 8, 16))}
    assert codes == {lib.nkh_linear_attention(p, p, p, p, bh, 64, None, 0)}
    # one that needs a workspace wants it aligned
    assert lib.nkh_linear_attention(p, p, p, p, 1, 4096, p + 8, 1 << 30) == 2


def test_launcher_without_a_workspace():
    """The launcher needs a workspace only where the long segments do; without
    one the sequences run unsegmented."""
    p = 1 << 20
    plain = LA.linear_attention(p, p, p, p, 24, 768)
    assert [l.symbol for l in plain] == ["nk_linattn_c64_d128"] and plain[0].args.nseg == 1
    assert len(LA.linear_attention(p, p, p, p, 24, 768, part_ptr=p)) == 2
    with pytest.raises(LA.LaunchError):
        LA.linear_attention(p, p, p, p, 1, 4096)
