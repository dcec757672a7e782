"""The scratch that an MSM asks for does not fall as its length grows, so that a caller can keep
one scratch for its longest polynomial: over a table of any size, over plain bases up to 2^19
points and in batches, around the lengths where the plan changes (runs of 8 or 16 entries a
thread at 2^19 digits, work-groups per sort tile, window widths at powers of two). Host only."""
import ctypes

import pytest


@pytest.fixture(scope="module")
def lib():
    import torch  # noqa: F401  one HIP runtime with torch

    from halo2_amd import _lib

    return _lib.load()


def _lengths(top: int) -> list[int]:
    near = {(1 << k) + d for k in range(1, 21) for d in (-1, 0, 1)}  # widths
    near |= {4096 * t + d for t in range(1, 130) for d in (0, 1)}  # tiles of a sort
    near |= {(1 << 19) // w + d for w in range(12, 64) for d in (0, 1)}  # 2^19 digits in w windows
    return sorted(n for n in near | set(range(1, 1 << 17, 331)) if n <= top)


def _rises(sizes: list[int]) -> bool:
    return all(a <= b for a, b in zip(sizes, sizes[1:]))


@pytest.mark.parametrize("log_table", [8, 13, 15, 16, 17, 18, 20, 22])
def test_table_scratch_serves_shorter_lengths(lib, log_table):
    n = 1 << log_table
    size = lib.h2amd_multiexp_precomputed_workspace_size
    assert _rises([int(size(m, n)) for m in _lengths(min(n, 1 << 18)) + [n]])


def test_plain_scratch_serves_shorter_lengths(lib):
    ns = _lengths((1 << 19) - 1)
    for size in (lib._halo2_multiexp_device_scalars_device_bases_workspace_size,
                 lib._halo2_multiexp_device_bases_workspace_size, lib._halo2_multiexp_workspace_size):
        assert _rises([int(size(n)) for n in ns])


@pytest.mark.parametrize("count", [1, 3, 64])
def test_batch_scratch_serves_shorter_lengths(lib, count):
    def words(n):
        return (ctypes.c_uint64 * count)(*([n] * count))

    ns = _lengths((1 << 19) // count)
    assert _rises([int(lib.h2amd_multiexp_batch_workspace_size(words(n), count)) for n in ns])
    assert _rises([int(lib.h2amd_multiexp_batch_precomputed_workspace_size(words(n), count, 1 << 20)) for n in ns])
