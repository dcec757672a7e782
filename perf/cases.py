"""What a prover spends its time on, as calls of this library's public entry points.

Every case is one kind of call at one size. The kinds are the steps of a KZG / SHPLONK
proof over BN254 (transforms between coefficient, Lagrange and coset form; commitments;
the lookup argument; the opening) and the proof itself; sizes run from the calls where
launches and latency are all there is to the largest that one proof makes.

Field elements are 4 little-endian 64-bit words in Montgomery form (a * 2^256 mod m) and
every result is a whole number mod r or mod p, fully reduced, so every case is exact.
"""
from __future__ import annotations

import ctypes
import functools
import math
import os
import random
import sys

import numpy as np
import torch

_PKG = os.path.abspath("halo2-gpu_amd")
if _PKG not in sys.path:
    sys.path.insert(0, _PKG)

from halo2_amd import _lib, device as dv, fields, lookup, msm, ntt, polyops, prover, shplonk  # noqa: E402
from halo2_amd.domain import EvaluationDomain, coeff_to_extended_batch_device  # noqa: E402

R = 0x30644E72E131A029B85045B68181585D2833E84879B9709143E1F593F0000001  # scalar field
P = 0x30644E72E131A029B85045B68181585D97816A916871CA8D3C208C16D87CFD47  # base field
DEGREE = 4  # constraint degree of the standard-gate circuit: the extended domain is 4 n
BLINDING = 6  # rows of a column that hold no witness values


# ------------------------------------------------------------------ the cases


def listed() -> list[dict]:
    return [
        # one short column to coefficient form: launches and latency are all there is
        {"name": "ifft_1x2^10", "kind": "ifft", "k": 10, "count": 1},
        # the columns of a proof of the most frequent served size, moved to one coset part of h(X)
        {"name": "coset_part_9x2^16", "kind": "coset_part", "k": 16, "count": 9},
        # the largest single transform that is benchmarked: a coset NTT out of place
        {"name": "coset_ntt_2^24", "kind": "coset", "k": 24},
        # polynomials of different circuits extended together
        {"name": "extend_uneven", "kind": "extend", "ks": "14,20,15,16,18,14,21,17,19,16,15,18"},
        # best_multiexp of a small circuit's column, scalars and points in host memory
        {"name": "msm_host_1500", "kind": "msm_host", "n": 1500},
        # an MSM of a ragged length over bases that have no table
        {"name": "msm_50003", "kind": "msm", "n": 50003},
        {"name": "msm_3000001", "kind": "msm", "n": 3_000_001},
        # the advice commitments of a 2^20-row proof against the resident SRS: five columns,
        # one of them 16-bit values, the last one shorter
        {"name": "commit_5x2^20", "kind": "commit", "k": 20, "count": 5, "small": 1, "short": 4097},
        # a range lookup: the permuted pair and its grand product
        {"name": "lookup_2^20", "kind": "lookup", "k": 20},
        # the evaluations of a proof's polynomials and their SHPLONK opening
        {"name": "opening_2^18", "kind": "opening", "k": 18},
        # whole proofs of the standard-gate circuit: the smallest served size and the benchmarked one
        {"name": "proof_2^16", "kind": "proof", "k": 16},
        {"name": "proof_2^20", "kind": "proof", "k": 20},
    ]


def _log_uniform(rng: random.Random, lo: int, hi: int) -> int:
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng: random.Random) -> dict:
    kind = rng.choice(["ifft", "coset_part", "coset", "extend", "msm_host", "msm", "msm", "commit", "lookup", "opening",
                       "proof"])
    if kind in ("ifft", "coset_part"):
        k = rng.randint(6, 21)
        return {"kind": kind, "k": k, "count": rng.randint(1, min(12, 1 << (23 - k)))}
    if kind == "coset":
        return {"kind": kind, "k": rng.randint(5, 24)}
    if kind == "extend":
        return {"kind": kind, "ks": ",".join(str(rng.randint(8, 20)) for _ in range(rng.randint(2, 16)))}
    if kind == "msm_host":
        return {"kind": kind, "n": _log_uniform(rng, 30, 1 << 17)}
    if kind == "msm":
        return {"kind": kind, "n": _log_uniform(rng, 100, 3_000_000)}
    if kind == "commit":
        k, count = rng.randint(10, 20), rng.randint(1, 6)
        return {"kind": kind, "k": k, "count": count, "small": rng.randint(0, count),
                "short": rng.randint(0, 1 << (k - 1))}
    if kind == "lookup":
        return {"kind": kind, "k": rng.randint(8, 20)}
    if kind == "opening":
        return {"kind": kind, "k": rng.randint(8, 19)}
    return {"kind": "proof", "k": rng.randint(12, 19)}


# --------------------------------------------------------------------- inputs


def _uniform(n: int, seed: int) -> torch.Tensor:
    """n field elements: words of a value below m, the top word below m's own top word."""
    g = torch.Generator(device="cuda").manual_seed(seed)
    out = torch.randint(-(1 << 63), (1 << 63) - 1, (n, 4), generator=g, device="cuda", dtype=torch.int64)
    out[:, 3] = torch.randint(0, R >> 192, (n,), generator=g, device="cuda", dtype=torch.int64)
    return out.reshape(-1)


@functools.lru_cache(maxsize=1)
def _range_table() -> np.ndarray:
    """The words of 0 .. 2^16 - 1 in Montgomery form."""
    one, v, rows = (1 << 256) % R, 0, []
    for _ in range(1 << 16):
        rows.append(v.to_bytes(32, "little"))
        v = (v + one) % R
    return np.frombuffer(b"".join(rows), dtype=np.int64).reshape(-1, 4)


def _range_column(n: int, seed: int, table: torch.Tensor) -> torch.Tensor:
    """n values drawn from the range table (a witness column of small values)."""
    g = torch.Generator(device="cuda").manual_seed(seed)
    return table[torch.randint(0, table.shape[0], (n,), generator=g, device="cuda")].reshape(-1)


def _table_rows(limit: int) -> torch.Tensor:
    return torch.from_numpy(_range_table()[:limit].copy()).cuda()


def _scalar(rng: random.Random) -> int:
    return rng.randrange(1, R)


def _opening_plan(k: int, x: int) -> list[tuple[int, int]]:
    """(polynomial, point) of the standard-gate circuit's queries, in halo2's open order:
    5 advice, 2 permutation products, lookup product and permuted pair, 5 fixed, 4 sigma, h."""
    w = fields.omega(k)
    w_inv = pow(w, -1, R)
    nxt, prev, last = x * w % R, x * w_inv % R, x * pow(w_inv, BLINDING, R) % R
    plan = [(i, x) for i in range(5)] + [(5, x), (5, nxt), (6, x), (6, nxt), (5, last)]
    plan += [(7, x), (8, x), (9, x), (8, prev), (7, nxt)]
    return plan + [(10 + i, x) for i in range(10)]


_OPENED = 20  # polynomials of _opening_plan


def prepare(case: dict, seed: int) -> dict:
    kind, rng = case["kind"], random.Random(seed)
    st = {"case": case}
    if kind in ("ifft", "coset_part"):
        st["domain"] = EvaluationDomain(DEGREE, case["k"])
        st["polys"] = [_uniform(1 << case["k"], seed * 64 + i) for i in range(case["count"])]
        st["factor"] = pow(st["domain"].extended_omega, rng.randint(0, 3), R)
    elif kind == "coset":
        st["omega"], st["shift"] = fields.omega(case["k"]), _scalar(rng)
        st["poly"] = _uniform(1 << case["k"], seed * 64)
    elif kind == "extend":
        ks = [int(v) for v in case["ks"].split(",")]
        st["domains"] = [EvaluationDomain(DEGREE, k) for k in ks]
        st["polys"] = [_uniform(1 << k, seed * 64 + i) for i, k in enumerate(ks)]
    elif kind in ("msm", "msm_host"):
        n = case["n"]
        st["scalars"], st["logs"] = _uniform(n, seed * 64), _uniform(n, seed * 64 + 1)
        st["bases"] = msm.g1_mul_generator(st["logs"], n)
        if kind == "msm_host":
            st["scalars"], st["bases"] = dv.to_host(st["scalars"]), dv.to_host(st["bases"], cols=8)
    elif kind == "commit":
        n, table = 1 << case["k"], _table_rows(1 << 16)
        st["tau"] = _scalar(rng)
        st["params"] = msm.ParamsKZG(case["k"], st["tau"])
        lens = [n] * (case["count"] - 1) + [n - case["short"]]
        st["polys"] = [_range_column(m, seed * 64 + i, table) if i < case["small"] else _uniform(m, seed * 64 + i)
                       for i, m in enumerate(lens)]
        st["params"].commit_device(st["polys"][0])  # builds the table that the parameters keep
    elif kind == "lookup":
        n = 1 << case["k"]
        usable = n - BLINDING
        rows = _table_rows(min(1 << 16, usable))
        st["input"] = _range_column(n, seed * 64, rows)
        st["table"] = torch.zeros(n, 4, dtype=torch.int64, device="cuda")
        st["table"][: rows.shape[0]] = rows
        st["table"] = st["table"].reshape(-1)
        st["blinders"] = _uniform(3 * BLINDING, seed * 64 + 1).view(3, BLINDING, 4)
        st["beta"], st["gamma"] = _scalar(rng), _scalar(rng)
        st["usable"] = usable
    elif kind == "opening":
        n = 1 << case["k"]
        st["params"] = msm.ParamsKZG(case["k"], _scalar(rng))
        st["polys"] = [_uniform(n, seed * 64 + i) for i in range(_OPENED)]
        st["plan"] = _opening_plan(case["k"], _scalar(rng))
        st["challenges"] = [_scalar(rng) for _ in range(3)]
        st["params"].commit_device(st["polys"][0])
    elif kind == "proof":
        st["circuit"] = prover.synthesize_standard(case["k"], seed)
        st["params"] = msm.ParamsKZG(case["k"], _scalar(rng))
        st["pk"] = prover.keygen(st["circuit"], st["params"])
        st["seed"] = seed % 100003 + 1
        st["params"].commit_device(st["circuit"].advice[0])  # both tables of the parameters
    else:
        raise ValueError(f"no kind {kind!r}")
    return st


# ------------------------------------------------------------------- one pass


def run(st: dict):
    kind = st["case"]["kind"]
    if kind == "ifft":
        return st["domain"].lagrange_to_coeff_many_device_inputs(st["polys"])
    if kind == "coset_part":
        return st["domain"].coeff_to_extended_part_many_device(st["polys"], st["factor"])
    if kind == "coset":
        out = dv.empty_u64(st["poly"].numel())
        ntt.fft_normal_device(ntt.COSET_FFT_PART, st["case"]["k"], st["poly"], out, st["omega"], st["shift"])
        return out
    if kind == "extend":
        return coeff_to_extended_batch_device(st["domains"], st["polys"])
    if kind == "msm_host":
        return msm.best_multiexp(st["scalars"], st["bases"])
    if kind == "msm":
        return msm.multiexp_device_scalars_device_bases(st["scalars"], st["bases"], st["case"]["n"])
    if kind == "commit":
        return st["params"].commit_many_device(st["polys"])
    if kind == "lookup":
        return _run_lookup(st)
    if kind == "opening":
        polys, plan = st["polys"], st["plan"]
        y, v, u = st["challenges"]
        evals = [fields.value_of(e) for e in polyops.batch_eval_polynomial_d2h([polys[i] for i, _ in plan],
                                                                               [p for _, p in plan])]
        out = shplonk.create_proof_device(st["params"], [shplonk.ProverQuery(p, polys[i], i) for i, p in plan], y, v,
                                          lambda h: u, evals=evals)
        return {"evals": np.stack([fields.limbs(e) for e in evals]), "h": out["h"], "h_final": out["h_final"],
                "h_x": out["h_x"], "h_x_final": out["h_x_final"]}
    out = prover.create_proof(st["params"], st["pk"], st["circuit"], seed=st["seed"])
    return {"proof": np.frombuffer(out["proof"], dtype=np.uint8), "holds": all(out["checks"].values())}


def _run_lookup(st: dict) -> dict:
    """The lookup argument of a proof: the permuted pair with its blinding rows, the
    product column and its running product."""
    lib, usable = _lib.load(), st["usable"]
    n = st["input"].numel() // 4
    p_in, p_tab, z = dv.empty_u64(4 * n), dv.empty_u64(4 * n), dv.empty_u64(4 * n)
    lookup.permute_expression_pair_device(st["input"], st["table"], p_in, p_tab, n, usable)
    p_in.view(-1, 4)[usable:] = st["blinders"][0]
    p_tab.view(-1, 4)[usable:] = st["blinders"][1]
    ratio = lookup.lookup_product_device(p_in, p_tab, st["input"], st["table"], st["beta"], st["gamma"])
    one = dv.to_device(fields.mont_limbs(1).reshape(1, 4))
    z.view(-1, 4)[:1].copy_(one.view(1, 4))
    z.view(-1, 4)[1:].copy_(ratio.view(-1, 4)[: n - 1])
    _lib.check(lib._halo2_grand_product_device_inputs(ctypes.byref(_lib.obj(dv.ptr(z))),
                                                      ctypes.byref(_lib.obj(dv.ptr(one))), n, 0, dv.stream()),
               "_halo2_grand_product_device_inputs")
    z.view(-1, 4)[n - BLINDING:] = st["blinders"][2]
    return {"permuted_input": p_in, "permuted_table": p_tab, "z": z}


# ----------------------------------------------------------------------- work

_MUL = 2 * 136  # operations of a 256-bit modular product: 64 + 64 + 8 32-bit multiply-adds


def _ntt_work(k: int, n_in: int) -> tuple[int, int]:
    n = 1 << k
    return 32 * (n_in + n), _MUL * (n * k // 2 + n)


def _msm_work(n: int) -> int:
    """Bucket additions of a window method of half log2 n + 2 bits, 10 products each."""
    c = int(math.log2(n)) // 2 + 2
    return -(-254 // c) * 10 * n * _MUL


def work(case: dict) -> dict:
    kind = case["kind"]
    if kind in ("ifft", "coset_part"):
        b, f = _ntt_work(case["k"], 1 << case["k"])
        return {"bytes": b * case["count"], "flops": f * case["count"]}
    if kind == "coset":
        b, f = _ntt_work(case["k"], 1 << case["k"])
        return {"bytes": b, "flops": f}
    if kind == "extend":
        parts = [_ntt_work(int(k) + 2, 1 << int(k)) for k in case["ks"].split(",")]
        return {"bytes": sum(b for b, _ in parts), "flops": sum(f for _, f in parts)}
    if kind in ("msm", "msm_host"):
        return {"bytes": 96 * case["n"], "flops": _msm_work(case["n"])}
    n = 1 << case["k"]
    if kind == "commit":
        total = n * case["count"] - case["short"]
        return {"bytes": 64 * n + 32 * total, "flops": _msm_work(n) * total // n}
    if kind == "lookup":  # two columns in; permuted pair and z out; ~10 products a row
        return {"bytes": 32 * 5 * n, "flops": 10 * n * _MUL}
    opening = (3 * _OPENED + 20) * n * _MUL + 2 * _msm_work(n)
    if kind == "opening":
        return {"bytes": 32 * (_OPENED + 2) * n, "flops": opening}
    # proof: 15 commitments, 11 columns to coefficients and 10 to 4 coset parts, the inverse of the
    # extended size, ~40 products a row of identities on 4 parts, the opening
    return {"bytes": 32 * 45 * n,
            "flops": 13 * _msm_work(n) + 51 * _ntt_work(case["k"], n)[1] + _ntt_work(case["k"] + 2, n)[1]
            + 160 * n * _MUL + opening}


def tolerance(case: dict):
    return "exact"  # whole numbers mod r or mod p and bytes


# -------------------------------------------------- the same from Python integers


def _ints(words) -> list[int]:
    """Canonical values of Montgomery words."""
    raw = (words.cpu().numpy() if isinstance(words, torch.Tensor) else np.asarray(words)).tobytes()
    inv = pow(1 << 256, -1, R)
    return [int.from_bytes(raw[i:i + 32], "little") * inv % R for i in range(0, len(raw), 32)]


def _words(values, m: int) -> np.ndarray:
    return np.frombuffer(b"".join((v * (1 << 256) % m).to_bytes(32, "little") for v in values), dtype=np.int64)


def _dft(a: list[int], w: int) -> list[int]:
    if len(a) == 1:
        return a
    even, odd = _dft(a[0::2], w * w % R), _dft(a[1::2], w * w % R)
    half, out, t = len(a) // 2, [0] * len(a), 1
    for i in range(half):
        v = t * odd[i] % R
        out[i], out[i + half] = (even[i] + v) % R, (even[i] - v) % R
        t = t * w % R
    return out


def _times_generator(s: int) -> np.ndarray:
    """s (1, 2) on y^2 = x^3 + 3 as (x, y, 1) in Montgomery words, (0, 1, 0) for the identity."""
    acc, base = None, (1, 2)

    def add(p, q):
        if p is None or q is None:
            return q if p is None else p
        if p[0] == q[0]:
            if (p[1] + q[1]) % P == 0:
                return None
            lam = 3 * p[0] * p[0] * pow(2 * p[1], -1, P) % P
        else:
            lam = (q[1] - p[1]) * pow(q[0] - p[0], -1, P) % P
        x = (lam * lam - p[0] - q[0]) % P
        return x, (lam * (p[0] - x) - p[1]) % P

    while s:
        if s & 1:
            acc = add(acc, base)
        base, s = add(base, base), s >> 1
    return _words((0, 1, 0) if acc is None else (*acc, 1), P).view(np.uint64)


def exact(case: dict, seed: int):
    """The transforms of up to 2^13 points in all, and every MSM and commitment of up to 2^20
    points: bases are known multiples of the generator, so the result is one multiple of it."""
    kind = case["kind"]
    if kind in ("ifft", "coset_part", "coset") and case.get("count", 1) << case["k"] <= 1 << 13:
        st = prepare(case, seed)
        k, n = case["k"], 1 << case["k"]
        w = pow(7, (R - 1) >> k, R)
        zeta = fields.ZETA
        outs = []
        for p in (st["polys"] if kind != "coset" else [st["poly"]]):
            a = _ints(p)
            if kind == "ifft":
                n_inv = pow(n, -1, R)
                vals = [v * n_inv % R for v in _dft(a, pow(w, -1, R))]
            else:
                g = zeta * st["factor"] % R if kind == "coset_part" else st["shift"]
                vals = _dft([v * pow(g, i, R) % R for i, v in enumerate(a)], w)
            outs.append(torch.from_numpy(_words(vals, R).copy()).cuda())
        return outs if kind != "coset" else outs[0]
    if kind in ("msm", "msm_host") and case["n"] <= 1 << 20:
        st = prepare(case, seed)
        return _times_generator(sum(a * b for a, b in zip(_ints(st["scalars"]), _ints(st["logs"]))) % R)
    if kind == "commit" and case["count"] << case["k"] <= 1 << 21:
        st = prepare(case, seed)
        rows = []
        for p in st["polys"]:
            acc = 0
            for v in reversed(_ints(p)):
                acc = (acc * st["tau"] + v) % R
            rows.append(_times_generator(acc))
        return np.stack(rows)
    return None
