"""Lookup permutation pair and lookup product on the device against the oracle
(src/cuda/tests.rs:978-1141 and 2340-2548 of the reference): all-distinct,
mixed-duplicate, all-same and small-value (keys equal in the high words) inputs,
usable_rows = n - blinding - 1 with garbage in the blinding rows, sizes across
the 2048-key sort tile and many merge passes; bit-exact."""
import numpy as np
import pytest

from conftest import rand_fr

pytestmark = pytest.mark.gpu


def _case(co, U, pattern, seed):
    from halo2_amd.fields import mont_limbs

    rng = np.random.default_rng(seed)
    if U == 0:
        z = np.zeros((0, 4), dtype=np.uint64)
        return z, z
    if pattern == "small":
        alpha = min(U, 1000)
        alphabet = np.stack([mont_limbs(v) for v in range(alpha)])
    else:
        alpha = {"distinct": U, "mixed": max(1, U // 3), "same": 1}[pattern]
        alphabet = rand_fr(co, alpha, seed)
    table = np.concatenate([alphabet, alphabet[rng.integers(0, alpha, U - alpha)]])
    table = table[rng.permutation(U)]
    if pattern == "distinct":
        inp = alphabet[rng.permutation(U)]
    else:
        inp = alphabet[rng.integers(0, alpha, U)]
    return np.ascontiguousarray(inp), np.ascontiguousarray(table)


CASES = [(4, 5, "distinct"), (4, 0, "same"), (10, 5, "mixed"), (11, 5, "small"), (12, 0, "distinct"),
         (12, 3, "mixed"), (13, 7, "same"), (16, 5, "mixed"), (16, 5, "small"), (20, 5, "distinct"),
         (20, 5, "mixed")]


@pytest.mark.parametrize("log_n,blinding,pattern", CASES)
def test_permute_expression_pair(lib, co, log_n, blinding, pattern):
    from halo2_amd import device as dv
    from halo2_amd.lookup import permute_expression_pair_device

    n = 1 << log_n
    U = n - blinding - 1 if blinding else n
    print(f"permute n={n} U={U} {pattern}", flush=True)
    inp, table = _case(co, U, pattern, 31 * log_n + blinding)
    pad_i = np.concatenate([inp, rand_fr(co, n - U, 7)])
    pad_t = np.concatenate([table, rand_fr(co, n - U, 8)])
    exp_i, exp_t = co.permute_expression_pair(pad_i, pad_t, n, U)
    d_pi = dv.to_device(np.full((n, 4), 0x5A, dtype=np.uint64))
    d_pt = dv.to_device(np.full((n, 4), 0x5A, dtype=np.uint64))
    permute_expression_pair_device(dv.to_device(pad_i), dv.to_device(pad_t), d_pi, d_pt, n, U)
    assert (dv.to_host(d_pi) == exp_i).all()
    assert (dv.to_host(d_pt) == exp_t).all()


def test_permute_expression_pair_edges(lib, co):
    """usable_rows 0 and 1 (outputs all zero / one row), and usable_rows > n rejected."""
    from halo2_amd import _lib, device as dv
    from halo2_amd.lookup import permute_expression_pair_device

    n = 64
    a, t = rand_fr(co, n, 1), rand_fr(co, n, 2)
    t[0] = a[0]
    for U in (0, 1):
        exp_i, exp_t = co.permute_expression_pair(a, t, n, U)
        d_pi, d_pt = dv.to_device(np.ones((n, 4), dtype=np.uint64)), dv.to_device(np.ones((n, 4), dtype=np.uint64))
        permute_expression_pair_device(dv.to_device(a), dv.to_device(t), d_pi, d_pt, n, U)
        assert (dv.to_host(d_pi) == exp_i).all() and (dv.to_host(d_pt) == exp_t).all()
    d = dv.to_device(a)
    err = lib._halo2_permute_expression_pair(dv.ptr(d), dv.ptr(d), dv.ptr(d), dv.ptr(d), 4, 5, None, 0, dv.stream())
    with pytest.raises(_lib.Halo2GpuError):
        _lib.check(err)


@pytest.mark.parametrize("free_bytes", [None, 200_000])
def test_lookup_product_mirrors(lib, co, free_bytes):
    from halo2_amd import device as dv, fields as F
    from halo2_amd.lookup import lookup_product_device, lookup_product_gpu

    n = 9000
    pi, pt, ci, ct = (rand_fr(co, n, 40 + i) for i in range(4))
    beta, gamma = 0xB37A, 0x6A33A
    exp = co.lookup_product(pi, pt, ci, ct, F.mont_limbs(beta), F.mont_limbs(gamma))
    assert (lookup_product_gpu(pi, pt, ci, ct, beta, gamma, free_bytes=free_bytes) == exp).all()
    got = lookup_product_device(*(dv.to_device(x) for x in (pi, pt, ci, ct)), beta, gamma)
    assert (dv.to_host(got) == exp).all()


@pytest.mark.parametrize("U", [2, 63, 8191, 8192, 8193, 3 * 8192 + 1])
@pytest.mark.parametrize("pattern", ["low_and_high", "window", "top"])
def test_permute_sort_windows(lib, co, U, pattern):
    """Columns whose keys a tile cannot order by one 51-bit window: they differ in high bits
    and, where those agree, in low ones only (every window of the tile is needed); or exactly
    in the bits of one window; or only in the top word; around the 8192-key tile."""
    from halo2_amd import device as dv
    from halo2_amd.fields import R_MOD, mont_limbs
    from halo2_amd.lookup import permute_expression_pair_device

    rng = np.random.default_rng(U)
    small = [int(v) for v in rng.integers(0, 97, U)]
    high = [int(v) for v in rng.integers(0, 5, U)]
    if pattern == "low_and_high":
        vals = [(h << 250) + (s << 100) + (h ^ s) for h, s in zip(high, small)]
    elif pattern == "window":
        vals = [s << 60 for s in small]
    else:
        vals = [(R_MOD - 1) - (s << 195) for s in small]
    table = np.stack([mont_limbs(v % R_MOD) for v in vals])
    inp = table[rng.integers(0, U, U)]
    exp_i, exp_t = co.permute_expression_pair(inp, table, U, U)
    d_pi, d_pt = dv.empty_u64(4 * U), dv.empty_u64(4 * U)
    permute_expression_pair_device(dv.to_device(inp), dv.to_device(table), d_pi, d_pt, U, U)
    assert (dv.to_host(d_pi) == exp_i).all()
    assert (dv.to_host(d_pt) == exp_t).all()


@pytest.mark.parametrize("U", [5, 1023, 8191, 8193, 3 * 8192 + 1])
@pytest.mark.parametrize("pattern", ["signed", "signed_wide", "three_groups", "packed", "powers", "groups_of_many", "late_tie",
                                     "two_ends", "levels"])
def test_permute_sort_bit_choices(lib, co, U, pattern):
    """Columns for every way in which a tile finds the bits that order its keys: signed numbers
    (small and 100 bits), three far groups, packed bytes and two values (few differing bits),
    powers of two (lengths), many lengths with long rests or with several levels of ties (further
    rounds of ranks), and a tie in the window that no two neighbours of the input show."""
    from halo2_amd import device as dv
    from halo2_amd.fields import R_MOD, mont_limbs
    from halo2_amd.lookup import permute_expression_pair_device

    rng = np.random.default_rng(U)

    def wide(bits):
        return [int.from_bytes(rng.bytes(32), "little") >> (256 - bits) for _ in range(U)]

    if pattern in ("signed", "signed_wide"):
        vals = [v if v & 1 else -v for v in wide(12 if pattern == "signed" else 100)]
    elif pattern == "three_groups":
        vals = [v + (g % 3) * (R_MOD // 2 - 1500) for v, g in zip(wide(11), wide(8))]
    elif pattern == "packed":
        vals = [sum((v >> (8 * j) & 255) << (61 * j) for j in range(4)) for v in wide(32)]
    elif pattern == "powers":
        vals = [1 << (v % 254) for v in wide(16)]
    elif pattern == "groups_of_many":
        vals = [(1 << (253 - v % 40)) + w for v, w in zip(wide(16), wide(100))]
    elif pattern == "levels":
        b, c = wide(60)[:3], wide(60)[:3]
        vals = [(1 << (253 - v % 40)) + (b[v >> 6 & 1] << 100) + (c[v >> 7 & 1] << 20) + (v >> 8 & 3) for v in wide(16)]
    elif pattern == "late_tie":
        vals = wide(253)
        vals[0], vals[-1], vals[U // 2] = vals[1] ^ 5, vals[1] ^ 3, vals[1] ^ (1 << 150)
    else:
        vals = [0 if v & 1 else R_MOD - 1 for v in wide(8)]
    table = np.stack([mont_limbs(v % R_MOD) for v in vals])
    inp = table[rng.integers(0, U, U)]
    exp_i, exp_t = co.permute_expression_pair(inp, table, U, U)
    d_pi, d_pt = dv.empty_u64(4 * U), dv.empty_u64(4 * U)
    permute_expression_pair_device(dv.to_device(inp), dv.to_device(table), d_pi, d_pt, U, U)
    assert (dv.to_host(d_pi) == exp_i).all()
    assert (dv.to_host(d_pt) == exp_t).all()
