"""The work whose speed this repository keeps an eye on, as calls of its public entry points.

The library is used to solve A x = b with conjugate gradients for the sparse
matrices of finite elements: the matrix and its preconditioner schedule stay
on the GPU in a `capi.System`, and right-hand sides come and go.  Beside that
stand the calls with host arrays (the drop-in form), the engine that advances
many systems together (`capi.Batch`), and the matrix-vector product alone.

A case is a dict:

  kind    "solve" (System.solve), "mixed" (System.solve_mixed: FP32 inner
          solves, FP64 refinement), "call" (a ConjugateGradientSolverCSR_* call
          with host arrays), "batch" (capi.Batch) or "apply" (System.apply)
  family  the matrix: "p1_2d" / "p1_3d" (P1 stiffness in the numbering of a
          uniformly refined mesh, `size` cells per axis, a power of two),
          "lagrange" (degree `degree` in dimension `dim`, any `size`),
          "hcurl" (Whitney 1-forms in 3D, any `size`)
  method  "rainbow" (multicolour SSOR), "ssor" (natural order), "cg"
  omega   the SSOR relaxation
  systems, rhs, mixed   batch only: `systems` matrices of degrees 1..3 with up
          to `size` cells per axis, `rhs` right-hand sides each; FP64 or mixed

Every solve starts from x = 0 and stops at a reduction of 1e-10, the setting
of the benchmark.  The right-hand sides are uniform in [-1, 1) on the free
unknowns; the matrix is scaled by a seeded material constant.
"""
import functools

import numpy as np
import torch  # before the library: both then use one HIP runtime

from simplefem_amd import capi
from simplefem_amd import systems as S

PRECISION = 1e-10
METHODS = {"rainbow": capi.METHOD_RAINBOW, "ssor": capi.METHOD_SSOR, "cg": capi.METHOD_CG}
KINDS = ("solve", "mixed", "call", "batch", "apply")


def _case(name, kind, family, size, method="rainbow", omega=1.0, dim=0, degree=1, systems=0,
          rhs=1, mixed=False):
    c = {"kind": kind, "family": family, "size": size, "method": method, "omega": omega,
         "dim": dim, "degree": degree, "systems": systems, "rhs": rhs, "mixed": mixed}
    return dict(c, name=name) if name else c


def listed():
    return [
        # the smallest solves: a coarse mesh, or one time step of a small model
        _case("ssor_2d_33", "solve", "p1_2d", 32, "ssor"),
        # the same class of problem through the drop-in call with host arrays
        _case("call_2d_33", "call", "p1_2d", 32, "rainbow", 1.2),
        # natural-order SSOR on a 129^2 mesh, the benchmark's 2D configuration
        _case("ssor_2d_129", "solve", "p1_2d", 128, "ssor"),
        # plain CG, two launches per iteration, on a middle-sized 3D mesh
        _case("cg_3d_33", "solve", "p1_3d", 32, "cg"),
        # higher degree: more colours, rows of uneven length
        _case("rainbow_3d_p2_33", "solve", "lagrange", 16, "rainbow", 1.0, 3, 2),
        # the benchmark's headline configuration, 64^3 cubes
        _case("rainbow_3d_65", "solve", "p1_3d", 64),
        # H(curl), the ill-conditioned operator, at a middle and at full size
        _case("rainbow_hcurl_24", "solve", "hcurl", 24),
        _case("rainbow_hcurl_48", "solve", "hcurl", 48),
        # the same operator to a true residual of 1e-10 in mixed precision
        _case("mixed_hcurl_24", "mixed", "hcurl", 24),
        # many small systems with four right-hand sides each, advanced together
        _case("batch_fp64_12x4", "batch", "lagrange", 64, dim=2, systems=12, rhs=4),
        _case("batch_mixed_12x4", "batch", "lagrange", 64, dim=2, systems=12, rhs=4, mixed=True),
        # the matrix-vector product on its own
        _case("apply_3d_65", "apply", "p1_3d", 64),
    ]


def _log_int(rng, lo, hi):
    return int(round(lo * (hi / lo) ** rng.random()))


def draw(rng):
    kind = rng.choice(("solve", "solve", "solve", "mixed", "call", "batch", "apply"))
    omega = rng.choice((1.0, 1.2))
    if kind == "batch":
        return _case("", "batch", "lagrange", _log_int(rng, 8, 64), "rainbow", omega, 2, 1,
                     rng.randint(2, 16), rng.randint(1, 4), rng.random() < 0.5)
    if kind == "call":  # small meshes, any number of cells
        return _case("", "call", "lagrange", _log_int(rng, 8, 64), rng.choice(("rainbow", "ssor")),
                     omega, 2, 1)
    method = "rainbow" if kind == "mixed" else rng.choice(("rainbow", "rainbow", "ssor", "cg"))
    if method != "ssor" and rng.random() < 0.3:
        return _case("", kind, "hcurl", _log_int(rng, 4, 36), method, omega)
    dim, degree = rng.choice((2, 3)), rng.choice((1, 2, 3))
    # nodes per axis, so that every degree covers the same range of unknowns; the levels of a
    # natural-order sweep on these meshes grow with the nodes per axis, so it gets the smaller ones
    nodes = _log_int(rng, 24, 64 if method == "ssor" else 500) if dim == 2 else \
        _log_int(rng, 8, 14 if method == "ssor" else 60)
    return _case("", kind, "lagrange", max(2, nodes // degree), method, omega, dim, degree)


# ------------------------------------------------------------------ matrices


@functools.lru_cache(maxsize=None)
def _matrix(family, size, dim, degree):
    if family == "p1_2d":
        return S.poisson2d_p1(size.bit_length() - 1, numbering="reference")
    if family == "p1_3d":
        return S.poisson3d_p1_kuhn(size, numbering="reference")
    if family == "hcurl":
        return S.hcurl3d_whitney_kuhn(size)
    return S.lagrange_pr(dim, size, degree)


def _members(case):
    """The matrices of a case: one, or the systems of a batch, from small to large."""
    if case["kind"] != "batch":
        return [_matrix(case["family"], case["size"], case["dim"], case["degree"])]
    out = []
    for k in range(case["systems"]):
        degree = 1 + k % 3
        nodes = max(4, case["size"] * (k + 1) // case["systems"])
        out.append(_matrix("lagrange", max(2, nodes // degree), case["dim"], degree))
    return out


def _inputs(case, seed):
    """Per member: the matrix, its scaled values, and the right-hand sides (rhs, n)."""
    rng = np.random.default_rng([seed, 20])
    out = []
    for s in _members(case):
        V = s.V * rng.uniform(0.5, 2.0)
        b = rng.uniform(-1.0, 1.0, (case["rhs"], s.n))
        if case["kind"] != "apply":
            b[:, s.dirichlet] = 0.0
        out.append((s, V, b))
    return out


class _Vector:
    """A torch vector as the library's device buffers are passed: by address."""

    def __init__(self, t):
        self.t, self.n, self.dtype, self.address = t, t.numel(), np.float64, t.data_ptr()


def _vector(a):
    return _Vector(torch.from_numpy(np.ascontiguousarray(a)).cuda())


def prepare(case, seed):
    made = _inputs(case, seed)
    if case["kind"] == "batch":
        batch = capi.Batch(mixed=case["mixed"], max_slots=case["systems"] * 4)
        jobs = []
        for s, V, b in made:
            rb = capi.Rainbow(s.n, s.A, s.C)
            mid = batch.add_matrix(s.n, s.A, s.C, V, capi.get_diagonal(s.n, s.A, s.C, V),
                                   case["omega"], rb.num_colors, rb.F, rb.B, rb.R)
            jobs.append((mid, s.n, list(b)))
        return {"kind": "batch", "batch": batch, "jobs": jobs}
    s, V, b = made[0]
    colours = (0, None, None, None)
    if case["method"] == "rainbow":
        rb = capi.Rainbow(s.n, s.A, s.C)
        colours = (rb.num_colors, rb.F, rb.B, rb.R)
    diagonal = capi.get_diagonal(s.n, s.A, s.C, V) if case["method"] != "cg" else None
    if case["kind"] == "call":
        return {"kind": "call", "matrix": s, "V": V, "b": b[0], "diagonal": diagonal,
                "omega": case["omega"], "colours": colours, "method": case["method"]}
    system = capi.System(METHODS[case["method"]], s.n, s.A, s.C, V, diagonal, case["omega"],
                         *colours, fp32_inner=case["kind"] == "mixed")
    zero = np.zeros(s.n)
    return {"kind": case["kind"], "system": system, "b": _vector(b[0]), "x": _vector(zero),
            "residual": _vector(zero)}


def run(state):
    """The solution and whether the solve reports success (apply: the product).

    The residual that the solvers also return is what is left of b - A x after
    a reduction by 1e10: its own digits follow where the iteration happened to
    stop, so it stands behind `success` and not beside x.
    """
    kind = state["kind"]
    if kind == "batch":
        batch, slots = state["batch"], []
        for mid, n, bs in state["jobs"]:
            slots.append((n, batch.submit_group(mid, bs, precision=PRECISION)))
        while batch.run(0) > 0:
            pass
        batch.finished()
        out = {"x": [], "success": []}
        for n, group in slots:
            got = [batch.collect(slot, n) for slot in group]
            out["x"].append(np.stack([x for x, _ in got]))
            out["success"].append(np.array([i["success"] for _, i in got]))
        return out
    if kind == "call":
        s, info = state["matrix"], {}
        x, residual = np.zeros(s.n), np.zeros(s.n)
        args = (s.n, x, state["b"], s.A, s.C, state["V"], residual, PRECISION, -3,
                state["diagonal"], state["omega"])
        if state["method"] == "rainbow":
            capi.ConjugateGradientSolverCSR_Rainbow(*args, *state["colours"], info=info)
        else:
            capi.ConjugateGradientSolverCSR_SSOR(*args, info=info)
        return {"x": x, "success": info["success"]}
    system, x = state["system"], state["x"]
    if kind == "apply":
        system.apply(x, state["b"])
        return {"y": x.t}
    x.t.zero_()
    if kind == "mixed":
        info = system.solve_mixed(x, state["b"], PRECISION)
    else:
        state["residual"].t.zero_()
        info = {}
        system.solve(x, state["b"], state["residual"], PRECISION, info=info)
    return {"x": x.t, "success": info["success"]}


def _iterations(case, s):
    """About the iterations CG needs at this reduction: proportional to the nodes per axis."""
    if case["kind"] == "apply":
        return 0
    nodes = case["size"] * case["degree"]
    per_node = 25.0 if case["family"] == "hcurl" else 2.0
    if case["kind"] == "batch":
        nodes, per_node = s.n ** 0.5, 2.0
    return per_node * nodes * (2.0 if case["method"] == "cg" else 1.0)


def work(case):
    total = {"bytes": 0.0, "flops": 0.0}
    for s in _members(case):
        # the CSR arrays and b in, x out: each once
        total["bytes"] += 12.0 * s.nnz + 4.0 * s.n + 16.0 * s.n * case["rhs"]
        # a product is 2 flops an entry; the two triangles of an SSOR step are as much again
        per = 2.0 * s.nnz + (0.0 if case["method"] == "cg" else 2.0 * s.nnz) + 10.0 * s.n
        total["flops"] += case["rhs"] * (2.0 * s.nnz + per * _iterations(case, s))
    return total


def tolerance(case):
    """What the stopping rule leaves open: the loop ends at sqrt(z.r) <= max(1e-10 |b|, 2^-26), and
    another order of the dot products may end it an iteration earlier or later.  Measured against
    exact(): 1e-12 to 6.7e-9, the largest on the smallest systems, where the floor 2^-26 decides."""
    if case["kind"] == "apply":
        return {"rel": 1e-14}
    return {"rel": 3e-8}


def exact(case, seed):
    """The solution itself, from Jacobi-preconditioned CG in float64 with torch's own sparse
    product, run to 1e-13; 64-bit numbers have none better at these condition numbers."""
    out = []
    for s, V, b in _inputs(case, seed):
        matrix = torch.sparse_csr_tensor(torch.from_numpy(s.A.astype(np.int64)),
                                         torch.from_numpy(s.C.astype(np.int64)),
                                         torch.from_numpy(V), size=(s.n, s.n)).cuda()
        if case["kind"] == "apply":
            return {"y": matrix @ torch.from_numpy(b[0]).cuda()}
        rows = torch.repeat_interleave(torch.arange(s.n), torch.from_numpy(np.diff(s.A).astype(np.int64)))
        on = rows == torch.from_numpy(s.C.astype(np.int64))
        diagonal = torch.zeros(s.n, dtype=torch.float64).index_add_(
            0, rows[on], torch.from_numpy(V)[on]).cuda()
        free = diagonal != 0
        inverse = torch.where(free, 1.0 / torch.where(free, diagonal, 1.0), 0.0)
        found = []
        for right in torch.from_numpy(b).cuda():
            x, r = torch.zeros_like(right), right.clone()
            z = inverse * r
            d, zr, stop = z.clone(), torch.dot(z, r), 1e-13 * float(right.norm())
            for k in range(20000):
                q = matrix @ d
                alpha = zr / torch.dot(d, q)
                x += alpha * d
                r -= alpha * q
                if k % 32 == 31 and not float(r.norm()) > stop:
                    break
                z = inverse * r
                new = torch.dot(z, r)
                d = z + (new / zr) * d
                zr = new
            found.append(x)
        out.append(torch.stack(found))
    if case["kind"] == "batch":
        return {"x": out, "success": [None] * len(out)}
    return {"x": out[0][0], "success": None}
