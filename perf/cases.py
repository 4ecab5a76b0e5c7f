"""The work whose speed this framework is judged by.

Each case is one pass through the public entry points on operands that are
already on the GPU, as a DF-MP2 or tensor-contraction program holds them. The
listed cases walk the range from the smallest calls (a 24-orbital molecule, a
32 x 96 pair block) over mid-sized molecules with odd extents (21 occupied,
150 virtual, 555 auxiliary functions: nothing is a multiple of a tile) to the
largest configurations of bench.py; `draw` gives more of the same ranges.

Kinds of case:
  pairs    einsum("ap,bp->ab", B[i], B[j]) for every ordered pair (the
           einsum-loop form of DF-MP2: many launches of one tiny product)
  mp2      mp2_energy(B, eps_occ, eps_vir)
  ao2mo    ao_to_mo_transform(eri, C_occ, C_vir)
  matmul   einsum of two matrices, or of two batches of them, in one of the
           four operand layouts, with or without alpha/beta/out
  path     einsum("ia,jb,abP,ijP->") in the default (greedy) order
  permute  einsum of one operand, a permutation of its three letters
"""

from __future__ import annotations

import math

import numpy as np
import torch

import trntensor_amd as tt

_DTYPES = {"f32": torch.float32, "f64": torch.float64, "bf16": torch.bfloat16, "f16": torch.float16}
_SIZE = {"f32": 4, "f64": 8, "bf16": 2, "f16": 2}

# Operand layouts of a matrix product: A stored [m][k] or [k][m], B stored
# [k][n] or [n][k]; a leading "b" is the batch.
_LAYOUTS = ("ij,jk->ik", "ij,kj->ik", "ji,jk->ik", "ji,kj->ik")
_BATCH_LAYOUTS = ("bij,bjk->bik", "bij,bkj->bik", "bji,bjk->bik", "bji,bkj->bik")
_PERMUTATIONS = ("ijk->kji", "ijk->ikj", "ijk->jki", "ijk->kij")


def listed() -> list[dict]:
    return [
        # The einsum-loop DF-MP2 harness (8 occupied, 32 virtual, 96
        # auxiliary functions): 64 calls whose kernels are microseconds long.
        {"name": "pair_loop_f32", "kind": "pairs", "dtype": "f32", "nocc": 8, "nvir": 32, "naux": 96},
        # Smallest molecule: one call, 15 occupied pairs.
        {"name": "mp2_small_f64", "kind": "mp2", "dtype": "f64", "nocc": 5, "nvir": 19, "naux": 72},
        # A mid-sized molecule in single precision, every extent ragged.
        {"name": "mp2_mid_f32", "kind": "mp2", "dtype": "f32", "nocc": 21, "nvir": 150, "naux": 555},
        # bench.py's headline configuration.
        {"name": "mp2_large_f64", "kind": "mp2", "dtype": "f64", "nocc": 64, "nvir": 320, "naux": 1200},
        # The mid-sized molecule's integral transform (171 basis functions).
        {"name": "ao2mo_mid_f64", "kind": "ao2mo", "dtype": "f64", "nbasis": 171, "nocc": 21, "nvir": 150,
         "naux": 555},
        # bench.py's full transform, in single precision (1.6 GB of integrals).
        {"name": "ao2mo_large_f32", "kind": "ao2mo", "dtype": "f32", "nbasis": 512, "nocc": 64, "nvir": 320,
         "naux": 1536},
        # One large product of ragged matrices with the whole epilogue.
        {"name": "matmul_ragged_f32", "kind": "matmul", "dtype": "f32", "sub": "ij,jk->ik", "batch": 0, "m": 1999,
         "n": 3001, "k": 1201, "epilogue": True, "precision": "fast"},
        # The 16-bit product at bench.py's GEMM size.
        {"name": "matmul_bf16", "kind": "matmul", "dtype": "bf16", "sub": "ij,jk->ik", "batch": 0, "m": 4096,
         "n": 4096, "k": 4096, "epilogue": False, "precision": "fast"},
        # The mid-sized molecule's diagonal pair blocks "iap,ibp->iab", batched.
        {"name": "bmm_pairs_f64", "kind": "matmul", "dtype": "f64", "sub": "bij,bkj->bik", "batch": 21, "m": 150,
         "n": 150, "k": 555, "epilogue": False, "precision": "fast"},
        # A product whose sums need more than double precision.
        {"name": "matmul_dd", "kind": "matmul", "dtype": "f64", "sub": "ij,jk->ik", "batch": 0, "m": 500, "n": 700,
         "k": 900, "epilogue": False, "precision": "dd"},
        # A four-operand energy expression in its default order.
        {"name": "path_f64", "kind": "path", "dtype": "f64", "nocc": 30, "nvir": 130, "naux": 450},
        # Reordering a three-index tensor: memory traffic only.
        {"name": "permute_f64", "kind": "permute", "dtype": "f64", "sub": "ijk->kji", "shape": "405,350,471"},
    ]


def _log_int(rng, lo: int, hi: int) -> int:
    """An integer in [lo, hi], its logarithm uniform."""
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


# Most work a drawn case of each kind may have (its listed cases' largest;
# flops, or bytes for the kinds that only move data).
_LIMIT = {"pairs": 1.0e8, "mp2": 5.2e11, "ao2mo": 1.1e11, "f32": 6.0e10, "f64": 2.0e10, "half": 1.4e11, "dd": 2.0e9,
          "path": 1.0e11, "permute": 1.1e9}


def draw(rng) -> dict:
    """One more case of the listed ranges."""
    kind = rng.choice(("pairs", "mp2", "mp2", "ao2mo", "f32", "half", "f64", "dd", "path", "permute"))
    while True:
        if kind == "pairs":
            case = {"kind": "pairs", "dtype": rng.choice(("f32", "f64")), "nocc": rng.randint(3, 10),
                    "nvir": _log_int(rng, 12, 64), "naux": _log_int(rng, 40, 160)}
        elif kind == "mp2":
            case = {"kind": "mp2", "dtype": rng.choice(("f32", "f64")), "nocc": _log_int(rng, 4, 64),
                    "nvir": _log_int(rng, 16, 320), "naux": _log_int(rng, 60, 1200)}
        elif kind == "ao2mo":
            nbasis = _log_int(rng, 24, 512)
            nocc = max(2, int(nbasis * rng.uniform(0.1, 0.25)))
            case = {"kind": "ao2mo", "dtype": rng.choice(("f32", "f64")), "nbasis": nbasis, "nocc": nocc,
                    "nvir": nbasis - nocc, "naux": int(nbasis * rng.uniform(2.5, 4.0))}
        elif kind in ("f32", "half", "dd"):
            lo, hi = {"f32": (100, 4096), "half": (128, 6144), "dd": (64, 1500)}[kind]
            case = {"kind": "matmul", "dtype": {"f32": "f32", "half": rng.choice(("bf16", "f16")), "dd": "f64"}[kind],
                    "sub": rng.choice(_LAYOUTS), "batch": 0, "m": _log_int(rng, lo, hi), "n": _log_int(rng, lo, hi),
                    "k": _log_int(rng, lo, hi), "epilogue": kind != "dd" and rng.random() < 0.5,
                    "precision": "dd" if kind == "dd" else "fast"}
        elif kind == "f64":
            nvir = _log_int(rng, 20, 320)
            case = {"kind": "matmul", "dtype": rng.choice(("f32", "f64")), "sub": rng.choice(_BATCH_LAYOUTS),
                    "batch": rng.randint(4, 64), "m": nvir, "n": nvir if rng.random() < 0.5 else _log_int(rng, 20, 320),
                    "k": _log_int(rng, 60, 1200), "epilogue": rng.random() < 0.5, "precision": "fast"}
        elif kind == "path":
            case = {"kind": "path", "dtype": rng.choice(("f32", "f64")), "nocc": _log_int(rng, 8, 48),
                    "nvir": _log_int(rng, 30, 200), "naux": _log_int(rng, 90, 700)}
        else:
            case = {"kind": "permute", "dtype": rng.choice(("f32", "f64")), "sub": rng.choice(_PERMUTATIONS),
                    "shape": ",".join(str(_log_int(rng, 60, 900)) for _ in range(3))}
        w = work(case)
        if max(w["flops"], w["bytes"] if kind == "permute" else 0) <= _LIMIT[kind]:
            return case


def _rand(g, *shape, scale=1.0):
    return torch.randn(shape, generator=g, dtype=torch.float64, device="cuda") * scale


def _energies(g, n, lo, hi):
    return torch.sort(lo + (hi - lo) * torch.rand(n, generator=g, dtype=torch.float64, device="cuda"))[0]


def _matmul_shapes(case):
    ext = {"b": case["batch"], "i": case["m"], "j": case["k"], "k": case["n"]}
    lhs, out = case["sub"].split("->")
    return [tuple(ext[c] for c in term) for term in lhs.split(",")] + [tuple(ext[c] for c in out)]


def prepare(case: dict, seed: int) -> dict:
    g = torch.Generator(device="cuda").manual_seed(seed)
    dt = _DTYPES[case["dtype"]]
    kind = case["kind"]
    if kind == "pairs":
        return {"case": case, "B": _rand(g, case["nocc"], case["nvir"], case["naux"], scale=0.1).to(dt)}
    if kind == "mp2":
        nocc, nvir, naux = case["nocc"], case["nvir"], case["naux"]
        return {"case": case, "B": _rand(g, nocc, nvir, naux, scale=0.05).to(dt),
                "eo": _energies(g, nocc, -20.0, -0.3).to(dt), "ev": _energies(g, nvir, 0.1, 5.0).to(dt)}
    if kind == "ao2mo":
        nb = case["nbasis"]
        eri = torch.randn((nb, nb, case["naux"]), generator=g, dtype=dt, device="cuda")
        eri = eri.add_(eri.transpose(0, 1).clone()).mul_(0.1)  # (mu nu | P) is symmetric in mu, nu
        scale = 1.0 / math.sqrt(nb)  # orbital coefficients: columns of about unit length
        return {"case": case, "eri": eri, "Co": _rand(g, nb, case["nocc"], scale=scale).to(dt),
                "Cv": _rand(g, nb, case["nvir"], scale=scale).to(dt)}
    if kind == "matmul":
        sa, sb, sd = _matmul_shapes(case)
        A, B = _rand(g, *sa), _rand(g, *sb)
        if case["precision"] == "dd":
            # Products over 16 binary orders of magnitude: sums that cancel.
            A = A * torch.exp2(torch.randint(-8, 9, sa, generator=g, device="cuda").double())
            B = B * torch.exp2(torch.randint(-8, 9, sb, generator=g, device="cuda").double())
        out = _rand(g, *sd, scale=math.sqrt(case["k"])).to(dt) if case["epilogue"] else None
        return {"case": case, "A": A.to(dt), "B": B.to(dt), "out": out}
    if kind == "path":
        nocc, nvir, naux = case["nocc"], case["nvir"], case["naux"]
        # Positive means, so that the energy is no sum of cancelling noise.
        return {"case": case, "ops": [(_rand(g, *s) + 1.0).to(dt) for s in
                                      ((nocc, nvir), (nocc, nvir), (nvir, nvir, naux), (nocc, nocc, naux))]}
    shape = tuple(int(x) for x in case["shape"].split(","))
    return {"case": case, "x": torch.randn(shape, generator=g, dtype=dt, device="cuda")}


def run(state: dict):
    case = state["case"]
    kind = case["kind"]
    if kind == "pairs":
        B = state["B"]
        n = case["nocc"]
        return [tt.einsum("ap,bp->ab", B[i], B[j]) for i in range(n) for j in range(n)]
    if kind == "mp2":
        return tt.mp2_energy(state["B"], state["eo"], state["ev"])
    if kind == "ao2mo":
        return tt.ao_to_mo_transform(state["eri"], state["Co"], state["Cv"])
    if kind == "matmul":
        if case["epilogue"]:
            return tt.einsum(case["sub"], state["A"], state["B"], alpha=1.5, beta=0.5, out=state["out"],
                             precision=case["precision"])
        return tt.einsum(case["sub"], state["A"], state["B"], precision=case["precision"])
    if kind == "path":
        return tt.einsum("ia,jb,abP,ijP->", *state["ops"])
    return tt.einsum(case["sub"], state["x"])


def work(case: dict) -> dict:
    es = _SIZE[case["dtype"]]
    kind = case["kind"]
    if kind == "pairs":
        no, nv, nx = case["nocc"], case["nvir"], case["naux"]
        return {"bytes": es * (no * nv * nx + no * no * nv * nv), "flops": 2 * no * no * nv * nv * nx}
    if kind == "mp2":
        # T_ij and T_ji are transposes of each other: the pairs i <= j.
        no, nv, nx = case["nocc"], case["nvir"], case["naux"]
        return {"bytes": es * (no * nv * nx + no + nv), "flops": no * (no + 1) // 2 * 2 * nv * nv * nx}
    if kind == "ao2mo":
        nb, no, nv, nx = case["nbasis"], case["nocc"], case["nvir"], case["naux"]
        return {"bytes": es * (nb * nb * nx + nb * (no + nv) + no * nv * nx),
                "flops": 2 * nx * (nb * nb * no + nb * no * nv)}
    if kind == "matmul":
        b, m, n, k = max(1, case["batch"]), case["m"], case["n"], case["k"]
        return {"bytes": es * b * (m * k + k * n + m * n * (2 if case["epilogue"] else 1)), "flops": 2 * b * m * n * k}
    if kind == "path":
        # The plan's order: the outer product, abP,ijP->abij, and the dot.
        no, nv, nx = case["nocc"], case["nvir"], case["naux"]
        return {"bytes": es * (2 * no * nv + nv * nv * nx + no * no * nx), "flops": 2 * nv * nv * no * no * (nx + 1)}
    total = math.prod(int(x) for x in case["shape"].split(","))
    return {"bytes": 2 * es * total, "flops": 0}


def tolerance(case: dict):
    """About four times what the path differs by from a float64 evaluation
    over the ranges above (matrix products 6e-7 f32, 1.1e-15 f64, 1.7e-3 bf16,
    2.1e-4 f16, 8e-18 dd; the scalar energies 5e-8 f32, 3e-16 f64, whose own
    last place is about that wide, so a little more)."""
    kind, dt = case["kind"], case["dtype"]
    if kind == "permute":
        return "exact"
    if case.get("precision") == "dd":
        return {"rel": 4e-17}
    if dt in ("bf16", "f16"):
        return {"rel": 7e-3 if dt == "bf16" else 9e-4}
    if kind in ("mp2", "path"):
        return {"rel": 3e-7 if dt == "f32" else 2e-15}
    return {"rel": 2.5e-6 if dt == "f32" else 4.5e-15}


def exact(case: dict, seed: int):
    s = prepare(case, seed)
    kind = case["kind"]
    if kind == "pairs":
        B = s["B"].double()
        n = case["nocc"]
        return [B[i] @ B[j].T.contiguous() for i in range(n) for j in range(n)]
    if kind == "mp2":
        B, eo, ev = s["B"].double(), s["eo"].double(), s["ev"].double()
        nocc, nvir, naux = B.shape
        flat = B.reshape(nocc * nvir, naux).T.contiguous()
        e = torch.zeros((), dtype=torch.float64, device="cuda")
        for i in range(nocc):
            T = (B[i] @ flat).reshape(nvir, nocc, nvir)  # [a, j, b]
            den = (eo[i] + eo)[None, :, None] - ev[:, None, None] - ev[None, None, :]
            e += (T * (2 * T - T.transpose(0, 2)) / den).sum()
        return e
    if kind == "ao2mo":
        Co, Cv = s["Co"].double(), s["Cv"].double()
        nb, no, nv, nx = case["nbasis"], case["nocc"], case["nvir"], case["naux"]
        X = (Co.T.contiguous() @ s["eri"].double().reshape(nb, nb * nx)).reshape(no, nb, nx)
        CvT = Cv.T.contiguous()
        return torch.stack([CvT @ X[i] for i in range(no)])
    if kind == "matmul":
        lhs = case["sub"].split("->")[0].split(",")
        A = s["A"].transpose(-2, -1) if lhs[0].endswith("ji") else s["A"]
        B = s["B"].transpose(-2, -1) if lhs[1].endswith("kj") else s["B"]
        if case["precision"] == "dd":
            a, b = (x.cpu().numpy().astype(np.longdouble) for x in (A, B))
            return torch.from_numpy((a @ b).astype(np.float64)).cuda()
        D = torch.matmul(A.double().contiguous(), B.double().contiguous())
        return 1.5 * D + 0.5 * s["out"].double() if case["epilogue"] else D
    if kind == "path":
        A, B, W, V = (x.double() for x in s["ops"])
        nocc, nvir, naux = case["nocc"], case["nvir"], case["naux"]
        ibP = (A @ W.reshape(nvir, nvir * naux)).reshape(nocc, nvir, naux)
        return sum(((B @ ibP[i]) * V[i]).sum() for i in range(nocc))
    order = [case["sub"].split("->")[0].index(c) for c in case["sub"].split("->")[1]]
    return s["x"].double().permute(order).contiguous()
