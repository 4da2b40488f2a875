"""Performance cases of the block-tridiagonal solver: what its users run, at their sizes.

A case is one call sequence of a user's program through the package's public entry
points, on inputs that stay on the GPU; `run` is one pass of it.  The kinds are

  plan      a plan of same-shape systems: new right-hand sides, factorize, solve
  combined  the same through the one-call factorize_solve
  resolve   new right-hand sides against factors that stay resident: solve only
  smoother  a state-space smoother request: blocks built on the device from the model,
            then factorize_solve
  group     systems of one block size and different lengths in one group plan
  batch     systems of different lengths and block sizes in one uneven batch

Inputs are the repository's own generators restated on the device: A_i = G G^T + n I,
B_i ~ N(0,1), d ~ U(0,1) (well conditioned, symmetric positive definite), or the normal
equations of a linear smoother (smoother requests and FP64 groups).
"""
import math
import random

import numpy as np
import torch

import blockstructuredsolvers_amd as bss
from blockstructuredsolvers_amd import serving, workloads

SIZES = (16, 32, 48, 64, 96, 128)


def _case(name, kind, mode, N, n, nrhs, nsys, schedule="auto"):
    """mode: "f64" and "f32" (plain solves in that type) or "mixed" (FP32 factors with FP64
    refinement).  group, batch: N is the longest system, sizes are drawn from 1/32 of
    it on; batch: n = 0 stands for a mix of all block sizes."""
    return {"name": name, "kind": kind, "mode": mode, "N": N, "n": n, "nrhs": nrhs,
            "nsys": nsys, "schedule": schedule}


def listed():
    return [
        # the smallest request: one filter horizon, its blocks built from the model
        _case("smoother_n16", "smoother", "f64", 300, 16, 1, 1),
        # the small system of the reference's own tests: latency and launches
        _case("small_n32", "plan", "f64", 100, 32, 1, 1),
        # one long system, the reference's batched path as its callers use it
        _case("single_n64", "plan", "f64", 8192, 64, 1, 1),
        # the largest blocks with a full set of right-hand sides
        _case("single_n128_rhs16", "plan", "f64", 8192, 128, 16, 1),
        # throughput: many systems resident in one plan, plain FP64 and mixed (the
        # benchmark's default workload)
        _case("batch_n64_f64", "plan", "f64", 8192, 64, 1, 32),
        _case("batch_n64_mixed", "plan", "mixed", 8192, 64, 1, 32),
        # refinement with several right-hand sides
        _case("mixed_n64_rhs16", "plan", "mixed", 4096, 64, 16, 8),
        # a block size between the powers of two, mixed
        _case("mixed_n96", "plan", "mixed", 2048, 96, 1, 8),
        # odd length, single precision, the reference's schedule (padded levels), the
        # combined call
        _case("ragged_n48_f32", "combined", "f32", 777, 48, 3, 7, "reference"),
        # an uneven batch over all block sizes in one call
        _case("uneven_mixed", "batch", "mixed", 4096, 0, 1, 64),
        # what the request loop runs: one coalesced group of smoother systems
        _case("group_n32_rhs4", "group", "f64", 4096, 32, 4, 24, "serve"),
        # repeated solves with resident factors
        _case("resolve_n64", "resolve", "f64", 8192, 64, 1, 8),
    ]


def _caps():
    works = [work(c) for c in listed()]
    return max(w["bytes"] for w in works), max(w["flops"] for w in works)


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["plan", "plan", "plan", "combined", "resolve", "smoother", "group", "batch"])
    mode = rng.choice(["f64", "mixed", "mixed", "f32"])
    n = rng.choice(SIZES)
    nrhs = rng.choice([1, 1, 1, 2, 3, 4, 7, 8, 16])
    N = _log_int(rng, 40, 8192)
    nsys = _log_int(rng, 1, 32)
    schedule = rng.choice(["auto", "auto", "auto", "reference"])
    if kind == "smoother":
        n, nsys, schedule, mode = rng.choice([16, 32, 64]), 1, "auto", "f64"
        N = _log_int(rng, 128, 4096)
    elif kind == "group":
        n, nsys, schedule = rng.choice([16, 32, 64]), rng.randint(2, 40), "serve"
        N, mode = _log_int(rng, 1024, 4096), rng.choice(["f64", "mixed"])
    elif kind == "batch":
        n, nsys, schedule, nrhs = 0, rng.randint(12, 64), "auto", 1
        N, mode = _log_int(rng, 1024, 4096), rng.choice(["f64", "mixed"])
    case = _case("", kind, mode, N, n, nrhs, nsys, schedule)
    del case["name"]
    top_bytes, top_flops = _caps()
    while case["nsys"] > 1 or case["N"] > 40:  # no more work than the largest listed case
        w = work(case)
        if w["bytes"] <= top_bytes and w["flops"] <= top_flops:
            break
        if case["nsys"] > 1:
            case["nsys"] -= max(1, case["nsys"] // 8)
        else:
            case["N"] -= max(1, case["N"] // 8)
    return case


def _sizes(case):
    """(N, n) of every system."""
    if case["kind"] in ("group", "batch"):
        r = random.Random(case["N"] * 1009 + case["nsys"])
        Ns = [_log_int(r, max(2, case["N"] // 32), case["N"]) for _ in range(case["nsys"])]
        ns = [r.choice(SIZES) if case["n"] == 0 else case["n"] for _ in Ns]
        return list(zip(Ns, ns))
    return [(case["N"], case["n"])] * case["nsys"]


def work(case):
    s = 4 if case["mode"] == "f32" else 8
    nrhs, nbytes, flops = case["nrhs"], 0.0, 0.0
    for N, n in _sizes(case):
        nbytes += 2 * N * n * nrhs * s  # right-hand sides in, solutions out
        flops += 6 * N * n * n * nrhs
        if case["kind"] == "resolve":  # the factors U (triangle) and C
            nbytes += (N * n * (n + 1) / 2 + (N - 1) * n * n) * s
        else:
            flops += 7 / 3 * N * n**3
            if case["kind"] == "smoother":  # F, H, Q^-1, R^-1
                nbytes += 2.75 * n * n * s
            else:  # A and B
                nbytes += (2 * N - 1) * n * n * s
    return {"bytes": nbytes, "flops": flops}


def _dtype(case):
    return torch.float32 if case["mode"] == "f32" else torch.float64


def _systems(case, seed):
    """Every system's (A, B, d) on the device, one after the other, block index first:
    A (N, row, col), B (N-1, col, row) as the solver stores it, d (N, rhs, row)."""
    g = torch.Generator(device="cuda").manual_seed(seed)
    dt, dev, f64 = _dtype(case), "cuda", torch.float64
    smooth = case["kind"] in ("group", "smoother") and case["mode"] == "f64"
    for k, (N, n) in enumerate(_sizes(case)):
        if smooth:
            m = _model(n, seed, k)
            Ai, Bi = m.blocks()
            A = torch.from_numpy(np.ascontiguousarray(Ai)).to(dev).expand(N, n, n)
            B = torch.from_numpy(np.ascontiguousarray(Bi.T)).to(dev).expand(N - 1, n, n)
        else:
            G = torch.randn((N, n, n), generator=g, device=dev, dtype=f64)
            A = torch.bmm(G, G.transpose(1, 2).contiguous())
            A.diagonal(dim1=1, dim2=2).add_(n)
            B = torch.randn((N - 1, n, n), generator=g, device=dev, dtype=f64)
        d = torch.rand((N, case["nrhs"], n), generator=g, device=dev, dtype=f64)
        yield A.to(dt), B.to(dt), d.to(dt)


def _model(n, seed, k):
    return workloads.smoother_model(n, np.random.default_rng([seed, k]))


def _data(case):
    mode = "mixed" if case["mode"] == "mixed" else "plain"
    kw = {"nrhs": case["nrhs"], "mode": mode}
    dt, sizes = _dtype(case), _sizes(case)
    if case["kind"] == "batch":
        return bss.initialize_batch([N for N, _ in sizes], [n for _, n in sizes], dt, "cuda", **kw)
    if case["kind"] == "group":
        return bss.initialize_batched_group([N for N, _ in sizes], case["n"], dt, "cuda",
                                            tuned=False, **serving.SERVE_SCHEDULE, **kw)
    return bss.initialize_batched(case["N"], case["n"], dt, "cuda", nsys=case["nsys"],
                                  schedule=case["schedule"], **kw)


def _views(data, case):
    """Per-system (A, B, d) views of the plan's tensors, block index first, the padding of
    the reference schedule left out."""
    if case["kind"] in ("group", "batch"):
        trip = zip(data.A_tensors, data.B_tensors, data.d_tensors)
    elif case["nsys"] == 1:
        trip = [(data.A_tensor, data.B_tensor, data.d_tensor)]
    else:
        trip = [(data.A_tensor[..., s], data.B_tensor[..., s], data.d_tensor[..., s])
                for s in range(case["nsys"])]
    for (N, _), (A, B, d) in zip(_sizes(case), trip):
        yield (A[:, :, :N].permute(2, 1, 0), B[:, :, :N - 1].permute(2, 1, 0),
               d[:, :, :N].permute(2, 1, 0))


def prepare(case, seed):
    data = _data(case)
    state = {"kind": case["kind"], "data": data}
    if case["kind"] in ("group", "batch"):
        state["x"] = data.d_tensors
    else:  # the reference schedule pads a system behind its last block
        state["x"] = data.d_tensor[:, :, :case["N"]]
    for (A, B, d), (Av, Bv, dv) in zip(_systems(case, seed), _views(data, case)):
        if case["kind"] != "smoother":
            Av.copy_(A)
            Bv.copy_(B)
        dv.copy_(d)
    if case["kind"] == "smoother":
        state["model"] = _model(case["n"], seed, 0)
    if case["kind"] in ("group", "batch"):
        state["d"] = data.d_tensors
    else:
        state["d"] = [data.d_tensor]
    # the right-hand sides a program keeps, since a solve overwrites d with the solution
    state["d0"] = [v.clone() for v in state["d"]]
    if case["kind"] == "resolve":
        bss.factorize(data)
    return state


def run(state):
    kind, data = state["kind"], state["data"]
    if kind == "smoother":
        bss.build_smoother(data, state["model"])
    torch._foreach_copy_(state["d"], state["d0"])
    if kind == "resolve":
        bss.solve(data)
    elif kind in ("combined", "smoother"):
        bss.factorize_solve(data)
    else:
        bss.factorize(data)
        bss.solve(data)
    return state["x"]


def _spd_solve(A, R):
    """A^-1 R for a stack of symmetric positive-definite blocks, by Gauss-Jordan elimination
    in steps of 16 rows."""
    n = A.shape[1]
    M = torch.cat([A, R], dim=2)
    for j in range(0, n, 16):
        D = torch.cat([M[:, j:j + 16, j:j + 16],
                       torch.eye(16, dtype=A.dtype, device=A.device).expand(len(A), 16, 16)], dim=2)
        for i in range(16):
            row = D[:, i:i + 1] / D[:, i:i + 1, i:i + 1]
            D -= D[:, :, i:i + 1] * row
            D[:, i:i + 1] = row
        P = torch.bmm(D[:, :, 16:].contiguous(), M[:, j:j + 16].contiguous())
        M -= torch.bmm(M[:, :, j:j + 16].contiguous(), P)
        M[:, j:j + 16] = P
    return M[:, :, n:]


def _block_solve(A, B, d):
    """x of tridiag(B^T, A, B) x = d by odd-even block reduction: A (N, n, n), B (N-1, n, n)
    in (row, col) order, d (N, n, nrhs)."""
    N, n = A.shape[0], A.shape[1]
    if N == 1:
        return _spd_solve(A, d)
    Bt = B.transpose(1, 2).contiguous()
    odd = torch.arange(1, N, 2, device=A.device)
    right = torch.zeros((len(odd), n, n), dtype=A.dtype, device=A.device)
    k = (N - 1) // 2  # odd blocks with a right neighbour
    right[:k] = B[1::2][:k]
    left = Bt[0::2]  # B_{j-1}^T of the odd blocks
    P = _spd_solve(A[1::2], torch.cat([left, right, d[1::2]], dim=2))
    PL, PR, Pd = [p.contiguous() for p in (P[:, :, :n], P[:, :, n:2 * n], P[:, :, 2 * n:])]
    A2, d2 = A[0::2].clone(), d[0::2].clone()
    m = len(odd)  # the even block on the left of odd block q is q, on its right q + 1
    Bl = B[0::2].contiguous()
    A2[:m] -= torch.bmm(Bl, PL)
    d2[:m] -= torch.bmm(Bl, Pd)
    Br = Bt[1::2][:k].contiguous()
    A2[1:k + 1] -= torch.bmm(Br, PR[:k])
    d2[1:k + 1] -= torch.bmm(Br, Pd[:k])
    xe = _block_solve(A2, -torch.bmm(Bl[:k], PR[:k]), d2)
    x = torch.empty_like(d)
    x[0::2] = xe
    xo = Pd - torch.bmm(PL, xe[:m])
    xo[:k] -= torch.bmm(PR[:k], xe[1:k + 1])
    x[1::2] = xo
    return x


def _residual(A, B, x, d):
    r = d - torch.bmm(A, x)
    r[:-1] -= torch.bmm(B, x[1:].contiguous())
    r[1:] -= torch.bmm(B.transpose(1, 2).contiguous(), x[:-1].contiguous())
    return r


def exact(case, seed):
    out = []
    for A, B, d in _systems(case, seed):
        A, d = A.double().contiguous(), d.double().transpose(1, 2).contiguous()
        B = B.double().transpose(1, 2).contiguous()
        x = _block_solve(A, B, d)
        x = x + _block_solve(A, B, _residual(A, B, x, d))
        out.append(x.permute(1, 2, 0))  # (n, nrhs, N)
    if case["kind"] in ("group", "batch"):
        return out
    return out[0] if case["nsys"] == 1 else torch.stack(out, dim=3)
