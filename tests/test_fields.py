"""Word forms of field elements on the host (halo2_amd/fields.py)."""
import numpy as np
import pytest

from halo2_amd import fields as F


@pytest.mark.parametrize("x", [0, 5, -5, True, F.R_MOD - 1, (1 << 300) + 7, np.uint64(2**64 - 1), np.array(9, dtype=np.uint64)])
def test_limbs_of_every_integer_type(x):
    """Python integers of any size and sign (mod 2^256) and numpy's unsigned 64-bit scalars."""
    got = F.limbs(x)
    assert got.dtype == np.uint64 and got.flags.writeable
    assert [int(w) for w in got] == [(int(x) >> (64 * i)) & (2**64 - 1) for i in range(4)]
    assert F.from_limbs(got) == int(x) % F.MONT
