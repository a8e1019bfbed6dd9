"""The work that users of this framework have it do, as cases to be timed.

A case is a dict of plain values with a "kind":

  step     one complex-double implicit step of a resident context (Step.step):
           what a time march runs thousands of times after one set-up
  refined  one step with complex-float factors and one complex-double defect
           correction (Step.step_refined_fixed)
  march    a chunk of complex-double steps of one receptivity request, sponge
           and local time steps on, replayed as one graph (the serving loop's
           unit of work)
  batch    uneven instances stepped together by one staged graph, the solve
           kernels chosen by the batch tuner as the batch driver does
  lines    a line solve of a factored handle (Penta.solve), the drop-in solver's
           device form: layout 1 has the lines along the last index, layout 2
           along the one before it
  periodic the same for lines that close on themselves
  factor   a new matrix factored and one right-hand side solved (a caller whose
           operator changes each step)

States are seeded: disturbances, matrices and right-hand sides differ by seed,
grids and physics are the case's.
"""
from __future__ import annotations

import math

import torch

from lns3d_amd.batch import Batch, draw_instances, pin_variants, tune_batch
from lns3d_amd.config import (Params, disturbance_envelope, make_disturbance_device, make_grid,
                              make_mean)
from lns3d_amd.native import MODE_BATCHED, MODE_FP64, Graph, Penta, Step
from lns3d_amd.serve import request_cfl, sponge_profiles

# bytes per grid point that each part cannot do without: coefficients, state
# and residual of the right-hand side; factors and right-hand side of a line
# solve in both precisions; the update; the line operator of a correction
RHS, SOLVE, SOLVE32, UPDATE, OPERATOR = 1224, 2160, 1160, 240, 1224
STEP = RHS + 2 * SOLVE + UPDATE
# a refined step: two pairs of complex-float solves, one application of the
# complex-double operator in both directions
REFINED = RHS + 4 * SOLVE32 + 2 * OPERATOR + UPDATE
# operations per point: a complex line solve (126 complex multiply-adds), the
# residual or operator (four real 5x5 blocks on complex values and stencils)
F_SOLVE, F_RHS = 1008, 1000


def listed():
    return [
        # the smallest grid the batches and the tests step: launches and the
        # serial chain of one short line
        dict(name="step_65x33", kind="step", nx=65, ny=33, wall=0, wallt=0, loctime=0, xper=0),
        # the small validation grid, stepped alone in parameter studies
        dict(name="step_129x65", kind="step", nx=129, ny=65, wall=0, wallt=0, loctime=0, xper=0),
        # the reference's receptivity grid, no-slip wall rows, local time steps
        dict(name="step_384x127_wall", kind="step", nx=384, ny=127, wall=1, wallt=1, loctime=1, xper=0),
        # the benchmark grid
        dict(name="step_1025x257", kind="step", nx=1025, ny=257, wall=0, wallt=0, loctime=0, xper=0),
        # temporal stability: periodic streamwise direction
        dict(name="step_periodic_257x97", kind="step", nx=257, ny=97, wall=0, wallt=0, loctime=0, xper=1),
        # mixed precision, an ordinary and the benchmark grid
        dict(name="refined_257x129", kind="refined", nx=257, ny=129, wall=0, wallt=0, loctime=0, xper=0),
        dict(name="refined_1025x257", kind="refined", nx=1025, ny=257, wall=0, wallt=0, loctime=0, xper=0),
        # a served request on the grid most requests use
        dict(name="march_129x65", kind="march", nx=129, ny=65, steps=50),
        # a parameter sweep: uneven grids of 65x33 to 513x257
        dict(name="batch_24", kind="batch", count=24, steps=10, which=0),
        # the line solver by itself: short lines and many of them, as the wall
        # normal direction has; long periodic lines
        dict(name="lines_700x301", kind="lines", layout=1, lines=700, rows=301),
        dict(name="periodic_512x1024", kind="periodic", layout=2, lines=512, rows=1024),
        # an operator that changes: factor and solve
        dict(name="factor_257x513", kind="factor", layout=2, lines=257, rows=513),
    ]


def draw(rng):
    def logint(lo, hi):
        return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))

    kind = rng.choice(("step", "step", "step", "refined", "refined", "march", "batch", "lines", "lines",
                       "periodic", "factor"))
    if kind in ("step", "refined"):
        wall = rng.choice((0, 1, 2))
        return dict(kind=kind, nx=logint(65, 1025), ny=logint(33, 257), wall=wall,
                    wallt=rng.choice((0, 1)) if wall else 0, loctime=rng.choice((0, 1)),
                    xper=int(kind == "step" and rng.random() < 0.15))
    if kind == "march":
        return dict(kind=kind, nx=logint(65, 257), ny=logint(33, 129), steps=rng.randint(10, 50))
    if kind == "batch":
        return dict(kind=kind, count=rng.randint(4, 20), steps=rng.randint(2, 10), which=rng.randint(1, 1 << 20))
    lines = logint(33, 1025)
    rows = logint(33, 1025 if lines < 300 else 300 if lines > 600 else 600)
    return dict(kind=kind, layout=rng.choice((1, 2)), lines=lines, rows=rows)


def _params(case):
    return Params(nx=case["nx"], ny=case["ny"], kz=0.3, wall=case["wall"], wallt=case["wallt"],
                  loctime=case["loctime"], xper=case["xper"])


def _disturbance(p, x, seed):
    env = torch.from_numpy(disturbance_envelope(x).reshape(-1, order="F")).to(torch.complex128).cuda()
    return make_disturbance_device(env, seed)


def _lines(case, seed):
    """seeded diagonally dominant lines: mat (row, line or line, row; c, r,
    slot) and a right-hand side, in the drop-in solver's storage order"""
    L, n = case["lines"], case["rows"]
    g = torch.Generator(device="cuda")
    g.manual_seed(int(seed))
    mat = torch.randn((L * n, 5, 5, 5), dtype=torch.complex128, generator=g, device="cuda") * 0.14
    for k in range(5):
        mat[:, k, k, 2] += 3.0
    rhs = torch.randn((L * n, 5), dtype=torch.complex128, generator=g, device="cuda")
    return mat, rhs


def prepare(case, seed):
    kind = case["kind"]
    s = {"kind": kind}
    if kind in ("step", "refined"):
        p = _params(case)
        x, y, met = make_grid(p)
        s["st"] = st = Step(p, precision=int(kind == "refined"))
        st.setup(met, make_mean(p, y))
        st.factor()
        s["v"] = _disturbance(p, x, seed)
        st.itrbc3d(s["v"])
        s["dv"] = torch.zeros_like(s["v"])
    elif kind == "march":
        p = Params(nx=case["nx"], ny=case["ny"], kz=0.4, omega=0.08, Ma=0.5, Re=100.0, loctime=1,
                   cflmax=request_cfl(case["nx"]))
        x, y, met = make_grid(p)
        s["st"] = st = Step(p)
        s["v"] = _disturbance(p, x, seed)
        s["dv"] = torch.zeros_like(s["v"])
        st.setup(met, make_mean(p, y))
        spg, spg2 = sponge_profiles(x)
        st.set_sponge(2, spg, spg2, x, None, 0.0)
        st.factor()
        st.itrbc3d(s["v"])
        s["norms"] = torch.zeros(case["steps"], dtype=torch.float64, device="cuda")
        st.set_residual_output(s["norms"], case["steps"])
        s["graph"] = Graph([st], [s["v"]], [s["dv"]], nsteps=case["steps"], mode=MODE_FP64)
        # a served request runs on a stream of its own
        s["stream"] = torch.cuda.Stream()
        torch.cuda.synchronize()
    elif kind == "batch":
        params = draw_instances(case["count"], case["which"])
        tune_batch(params, precision=1, seed=seed)
        s["batch"] = Batch(params, precision=1, seed=seed)
        s["graph"] = s["batch"].capture(case["steps"], MODE_BATCHED, 1)
        pin_variants(params, None)
    else:
        periodic = kind == "periodic"
        s["mat"], s["rhs"] = _lines(case, seed)
        s["x"] = torch.empty_like(s["rhs"])
        s["penta"] = Penta(int(periodic), case["layout"], case["lines"], case["rows"], exact=int(periodic))
        if kind != "factor":
            s["penta"].factor(s.pop("mat"))
    return s


def run(s):
    kind = s["kind"]
    if kind == "step":
        s["st"].step(s["v"], s["dv"])
        return {"v": s["v"], "dv": s["dv"]}
    if kind == "refined":
        s["st"].step_refined_fixed(s["v"], s["dv"], 1)
        return {"v": s["v"], "dv": s["dv"]}
    if kind == "march":
        # the stream takes up the state where the caller's stream left it, and
        # hands it back
        s["stream"].wait_stream(torch.cuda.current_stream())
        s["graph"].launch(s["stream"])
        torch.cuda.current_stream().wait_stream(s["stream"])
        return {"v": s["v"], "norms": s["norms"]}
    if kind == "batch":
        s["graph"].launch()
        return {"v%d" % k: v for k, v in enumerate(s["batch"].v)}
    # the solve is in place: a new right-hand side each pass
    s["x"].copy_(s["rhs"])
    if kind == "factor":
        s["penta"].factor(s["mat"])
    s["penta"].solve(s["x"])
    return s["x"]


def work(case):
    kind = case["kind"]
    if kind == "batch":
        P = sum(p.nx * p.ny for p in draw_instances(case["count"], case["which"]))
        n = P * case["steps"]
        return {"bytes": REFINED * n, "flops": (4 * F_SOLVE + 3 * F_RHS) * n}
    if kind in ("step", "refined", "march"):
        n = case["nx"] * case["ny"] * case.get("steps", 1)
        if kind == "refined":
            return {"bytes": REFINED * n, "flops": (4 * F_SOLVE + 3 * F_RHS) * n}
        # a periodic line's factors hold two border blocks more per row
        return {"bytes": (STEP + (1600 if case.get("xper") else 0)) * n, "flops": (2 * F_SOLVE + F_RHS) * n}
    n = case["lines"] * case["rows"]
    if kind == "lines":
        return {"bytes": SOLVE * n, "flops": F_SOLVE * n}
    if kind == "periodic":
        return {"bytes": (SOLVE + 1600) * n, "flops": 2 * F_SOLVE * n}
    # the matrix in, the factors out for later solves, one solve's vectors;
    # a block row costs about 14 products of 5x5 blocks
    return {"bytes": (2000 + 2000 + 160) * n, "flops": 14 * 1000 * n}


def exact(case, seed):
    """Line solves: the solution by 25x25 block elimination in 64 bits.  A
    step's outputs are held to the start's alone: its operator is the whole
    discretisation of the linearized equations, boundary closures included,
    which no short formula restates."""
    if case["kind"] not in ("lines", "periodic", "factor"):
        return None
    L, n = case["lines"], case["rows"]
    mat, rhs = _lines(case, seed)

    def line_first(a):
        a = a.reshape((n, L) + a.shape[1:]) if case["layout"] == 1 else a.reshape((L, n) + a.shape[1:])
        return a.transpose(0, 1) if case["layout"] == 1 else a

    periodic = case["kind"] == "periodic"
    m, b = line_first(mat), line_first(rhs)
    nu = n - 1 if periodic else n          # the last row of a periodic line repeats the first

    def columns(i):
        if periodic:
            return [(i - 2 + k) % nu for k in range(5)]
        # the rows next to an end keep five blocks in the line's first or last
        # five columns, wrapped so that slot k holds column i - 2 + k where
        # that is on the line
        return [(i - 2 + k) % 5 if i < 2 else nu - 5 + (i - 2 + k - (nu - 5)) % 5 if i > nu - 3 else i - 2 + k
                for k in range(5)]

    # super-rows of five rows (the last one five to nine): block tridiagonal,
    # plus corners that couple a periodic line's last super-row to the first
    starts = list(range(0, nu - nu % 5, 5))
    ends = starts[1:] + [nu]
    K = len(starts)
    of = [min(i // 5, K - 1) for i in range(nu)]

    def block(I, J):
        A = torch.zeros((L, (ends[I] - starts[I]) * 5, (ends[J] - starts[J]) * 5), dtype=mat.dtype, device=mat.device)
        for i in range(starts[I], ends[I]):
            for k, c in enumerate(columns(i)):
                if of[c] == J:
                    r0, c0 = (i - starts[I]) * 5, (c - starts[J]) * 5
                    A[:, r0:r0 + 5, c0:c0 + 5] += m[:, i, :, :, k].transpose(1, 2)
        return A

    def rows_of(I):
        return b[:, starts[I]:ends[I]].reshape(L, -1, 1)

    # eliminate super-rows 0..K-2 with the right-hand side and, beside it, the
    # coupling to the last super-row, then solve that one
    last = K - 1
    D, B, up = None, [], []
    for I in range(last):
        A = block(I, I)
        R = torch.cat([rows_of(I), block(I, last) if periodic and I == 0 or I == last - 1 else
                       torch.zeros((L, A.shape[1], (ends[last] - starts[last]) * 5), dtype=mat.dtype, device=mat.device)], 2)
        if I:
            low = block(I, I - 1)
            A = A - low @ up[-1]
            R = R - low @ B[-1]
        lu = torch.linalg.lu_factor(A)
        B.append(torch.linalg.lu_solve(*lu, R))
        up.append(torch.linalg.lu_solve(*lu, block(I, I + 1)) if I + 1 < last else None)
    for I in range(last - 2, -1, -1):
        B[I] = B[I] - up[I] @ B[I + 1]
    D, r = block(last, last), rows_of(last)
    for J in {0, last - 1} if periodic else {last - 1}:
        low = block(last, J)
        D = D - low @ B[J][:, :, 1:]
        r = r - low @ B[J][:, :, :1]
    xl = torch.linalg.solve(D, r)
    x = torch.cat([B[I][:, :, :1] - B[I][:, :, 1:] @ xl for I in range(last)] + [xl], 1).reshape(L, nu, 5)
    if periodic:
        x = torch.cat([x, x[:, :1]], 1)
    return (x.transpose(0, 1) if case["layout"] == 1 else x).reshape(L * n, 5).contiguous()
