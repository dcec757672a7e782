"""The bounds that the NTT's matrix steps rest on (halo2-gpu_amd/csrc/ntt_mfma.h), from the
mathematics: balanced digits of the centred residues of g^e 2^(8b), column sums that let a
pair of digits fit an int32, and the value range that the Montgomery steps take."""
import numpy as np
import pytest

from halo2_amd.fields import R_MOD as M

G16 = pow(7, (M - 1) // 16, M)


def _digits(v: int) -> list[int]:
    out, carry = [], 0
    for byte in (v % (1 << 256)).to_bytes(32, "little"):
        s = byte + carry
        carry = int(s >= 128)
        out.append(s - 256 * carry)
    assert sum(d << (8 * i) for i, d in enumerate(out)) == v
    return out


@pytest.fixture(scope="module")
def matrices():
    def centred(v):
        return v if 2 * v <= M else v - M

    return np.array([[_digits(centred(pow(G16, e, M) * pow(256, b, M) % M)) for b in range(32)] for e in range(16)])


@pytest.mark.parametrize("r", [16, 8])
def test_column_sums(matrices, r):
    # data bytes are x - 128 in [-128, 127]; y_0 gets 128 r back on every digit
    worst = max(int(np.abs(matrices[[a * j * (16 // r) % 16 for a in range(r)]]).sum(axis=(0, 1)).max()) * 128 + 128 * r
                for j in range(r))
    assert worst * 257 < 1 << 31 and worst < 2 ** 21.91


@pytest.mark.parametrize("seed", range(6))
def test_column_sums_of_scaled_matrices(seed):
    """The last step's matrices hold 2^29 s w^e for the caller's scale s: inverse powers of
    two, arbitrary ones and ones whose own digits are all extreme. (Over all s the sums are
    those of 512 digits that nobody chooses, mean 2^22; 2^23 is 39 standard deviations off.)"""
    rng = np.random.default_rng(seed)
    extreme = sum(-128 << (8 * i) for i in range(31)) % M
    scales = [pow(2, -(4 * seed + 5), M), int.from_bytes(rng.bytes(32), "little") % M, extreme,
              extreme * pow(G16, seed, M) % M]
    for s in scales:
        cols = [[pow(G16, e, M) * s * pow(256, b, M) % M for b in range(32)] for e in range(16)]
        digits = np.array([[_digits(v if 2 * v <= M else v - M) for v in row] for row in cols])
        for r in (16, 8):
            for j in range(r):
                sums = np.abs(digits[[a * j * (16 // r) % 16 for a in range(r)]]).sum(axis=(0, 1)) * 128
                assert int(sums.max()) * 257 < 1 << 31


@pytest.mark.parametrize("k", range(0, 29))
def test_column_sums_of_inverse_transforms(k):
    """The scales that the transforms themselves use, 1 and every 2^-k: the sums fit for certain."""
    s = pow(2, -k, M)
    cols = [[pow(G16, e, M) * s * pow(2, 29, M) * pow(256, b, M) % M for b in range(32)] for e in range(16)]
    digits = np.abs(np.array([[_digits(v if 2 * v <= M else v - M) for v in row] for row in cols]))
    for r in (16, 8):
        for j in range(r):
            assert int(digits[[a * j * (16 // r) % 16 for a in range(r)]].sum(axis=(0, 1)).max()) * 128 * 257 < 1 << 31


def test_dft_by_digits(matrices):
    """The steps' arithmetic in Python integers: shifted bytes through the matrices, the shift
    given back to y_0 only, against the DFT itself."""
    rng = np.random.default_rng(5)
    xs = [int.from_bytes(rng.bytes(32), "little") for _ in range(16)]
    shifted = np.array([[b - 128 for b in x.to_bytes(32, "little")] for x in xs])
    for j in range(16):
        cols = sum(shifted[a] @ matrices[a * j % 16] for a in range(16))
        v = sum(int(c) << (8 * i) for i, c in enumerate(cols))
        assert abs(v) <= 16 * 32 * 128 * (M // 2 + 1)
        if j == 0:
            v += 16 * sum(128 << (8 * b) for b in range(32))
        assert v % M == sum(x * pow(G16, a * j, M) for a, x in enumerate(xs)) % M
