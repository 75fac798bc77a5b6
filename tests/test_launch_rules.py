"""Rules that choose a launch shape on the host."""
import ctypes

import pytest

I64 = ctypes.c_int64


@pytest.mark.parametrize("asked", [0, 1, 2, 3, 4, -1])
@pytest.mark.parametrize("nb,bpw", [(1, 0), (1, 1), (1, 8), (3, 3), (3, 8), (3, 2), (65, 8), (2, 0)])
@pytest.mark.parametrize("ntiles", [1, 7, 8, 63, 64, 511, 512, 7680])
def test_tile_map(pkg, asked, nb, bpw, ntiles):
    """The caller's map wherever one workgroup takes all blocks of its tile; runs of
    tiles per XCD for several blocks otherwise; else the identity."""
    f = pkg.lib().rsvdt_hip_tile_map
    f.argtypes = [I64, I64, I64, ctypes.c_int]
    got = f(nb, bpw, ntiles, asked)
    if 1 <= asked <= 3 and (nb == 1 or bpw >= nb) and ntiles >= 8:
        assert got == asked
    elif nb > 1 and ntiles >= 64:
        assert got == (2 if ntiles >= 512 else 1)
    else:
        assert got == 0


@pytest.mark.parametrize("n", [65536, 70000])
def test_identity_beyond_one_launch(pkg, n):
    """Refused before anything is launched: a launch has less than 2^32 threads."""
    f = pkg.lib().rsvdt_hip_identity
    f.argtypes = [I64, ctypes.c_void_p, ctypes.c_void_p]
    assert f(n, None, None) == 102
