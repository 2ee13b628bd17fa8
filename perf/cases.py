"""Workloads of the solver for timing: what they are, their inputs, one pass
of each through the public entry points, and the same results in plain torch
FP64.

A case is a dict of plain values.  kind:
  flow   `steps` time steps (compute_dt + step, as the time loop runs them),
         then the velocity field as the output routine takes it
         (snapshot_begin / snapshot_end, or download on a tiny grid);
         `rows` also filters the DNS onto an LES grid and returns the
         closure's training rows
  stats  the statistics interval: z means, monitor sums, Cf, divergence
  train  Adam steps of the learned closure on the device dataset
Grids are tanh-stretched with x from 1 and nu for Re_theta = 300 at the inlet;
theta is the unit of the box lengths.
"""
import ctypes
import functools
import importlib.util
import math
import os

import numpy as np
import torch

THETA = 1.469653e-3
NU = 4.898844e-6
ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
F64 = torch.float64


@functools.lru_cache(maxsize=1)
def blgpu():
    """The product's Python binding (the package directory's name is not an importable module name)."""
    spec = importlib.util.spec_from_file_location("blgpu", os.path.join(ROOT, "boundary-layer-gpu_amd", "blgpu.py"))
    mod = importlib.util.module_from_spec(spec)
    spec.loader.exec_module(mod)
    return mod


def device():
    return torch.device("cuda" if torch.cuda.is_available() else "cpu")


# ------------------------------------------------------------------ cases ----
def flow(nx, ny, nz, steps, box=(400.0, 40.0, 40.0), cfl=0.5, precision="fp64", scheme=3, les=0, modes=0, inflow=1,
         wall=0, rows=False):
    return dict(kind="flow", nx=nx, ny=ny, nz=nz, lx=box[0], ly=box[1], lz=box[2], steps=steps, cfl=cfl,
                precision=precision, scheme=scheme, les=les, modes=modes, inflow=inflow, wall=wall, rows=rows)


def listed():
    c = {
        # one step of the smallest test grid: launches and latency only (a
        # regression run, a coupled code that steps the solver)
        "step_tiny": flow(24, 16, 8, 1, (102.0, 10.2, 4.1), cfl=-2e-4),
        # the laminar validation grid, 20 steps between outputs
        "laminar": flow(192, 32, 8, 20, (100.0, 10.0, 4.0), cfl=-1e-4),
        # transition run: inflow modes, RK2, odd sizes with no small factors
        "transition_rk2_odd": flow(131, 75, 53, 10, (64.0, 12.0, 11.0), scheme=2, modes=3),
        # the DNS that feeds the closure: steps, then filtering onto the LES grid
        "dns_training_rows": flow(513, 97, 130, 20, rows=True),
        # the throughput configuration, in both precisions
        "dns_full_fp64": flow(814, 257, 193, 40),
        "dns_full_mixed": flow(814, 257, 193, 40, precision="mixed"),
        # a span wider than the folded z transforms take, RK2, FP32 fields
        "dns_wide_mixed_rk2": flow(262, 66, 230, 10, (128.0, 10.2, 48.0), precision="mixed", scheme=2),
        # LES of the study grid with dynamic Smagorinsky, and the learned
        # closure on the smaller one
        "les_dynamic_mixed": flow(257, 97, 64, 10, precision="mixed", les=2),
        "les_learned_mixed": flow(129, 49, 34, 10, precision="mixed", les=4, cfl=0.3),
        # constant-coefficient Smagorinsky with a wall model and random inflow
        "les_wall_model": flow(161, 57, 42, 10, (80.0, 10.0, 9.0), cfl=-1e-4, les=1, wall=11, inflow=4),
        # the statistics interval of the throughput configuration
        "statistics_full": dict(kind="stats", nx=814, ny=257, nz=193, precision="fp64"),
        # closure training: batches of the study's size
        "closure_train": dict(kind="train", rows=400000, batch=65536, steps=10),
    }
    return [dict(v, name=k) for k, v in c.items()]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _x_fits(n):
    """Whether the x transform takes n = nx - 2 points: a divisor not too far from its square root."""
    n1 = max(a for a in range(1, int(n ** 0.5) + 1) if n % a == 0)
    return n <= 200 or n1 >= 4


def draw(rng):
    kind = rng.choice(["flow"] * 8 + ["stats", "train"])
    if kind == "train":
        return dict(kind="train", rows=_log(rng, 3000, 400000), batch=_log(rng, 256, 65536), steps=rng.randint(2, 10))
    precision = rng.choice(["fp64", "mixed"])
    while True:
        nx, ny, nz = _log(rng, 24, 820), _log(rng, 14, 290), _log(rng, 8, 240)
        if _x_fits(nx - 2) and nx * ny * nz <= 814 * 257 * 193:
            break
    if kind == "stats":
        return dict(kind="stats", nx=nx, ny=ny, nz=nz, precision=precision)
    cells = nx * ny * nz
    les = rng.choice([0, 0, 0, 1, 2, 3, 4])
    if les and cells > 4000000:
        les = 0
    steps = max(1, min(rng.randint(2, 20), 800000000 // cells))
    box = (nx * 0.49, max(10.0, 40.0 * (ny - 1) / 256.0), nz * 0.21)
    return flow(nx, ny, nz, steps, box, cfl=0.5 if ny >= 64 and les == 0 else -1e-4, precision=precision,
                scheme=rng.choice([2, 3, 3]), les=les, modes=rng.choice([0, 0, 3]) if les == 0 else 0,
                inflow=4 if les == 1 else 1, wall=11 if les == 1 else 0)


# ----------------------------------------------------------------- inputs ----
def grid(case):
    box = [case.get(k, d) * THETA for k, d in (("lx", 400.0), ("ly", 40.0), ("lz", 40.0))]
    nx, ny, nz = case["nx"], case["ny"], case["nz"]
    x, y, z = blgpu().grid_tanh(nx, ny, nz, box[0], box[1], box[2], 2.0, 1.0)
    eta, f, df = blgpu().blasius_profile()
    return x, y, z, blgpu().blasius_tables(x, y, NU, eta, f, df), (eta, f, df)


def initial(case, seed, amp=0.05):
    """Blasius + uniform noise on the interior, periodic in z: tensors (z, y, x) on the device."""
    x, y, z, tables, prof = grid(case)
    dev = device()
    gen = torch.Generator(device=dev)
    gen.manual_seed(int(seed))
    base = blgpu().blasius_field(x, y, z[:5], NU, *prof)  # uniform in z
    out = []
    for q, b in enumerate(base):
        nk = z.size if q == 2 else z.size + 1
        plane = torch.from_numpy(np.ascontiguousarray(b[:, :, 0].T)).to(dev)
        a = plane.expand(nk, *plane.shape).contiguous()
        r = torch.rand((nk - 2, plane.shape[0] - 2, plane.shape[1] - 2), generator=gen, device=dev, dtype=F64)
        a[1:-1, 1:-1, 1:-1] += amp * (2.0 * r - 1.0)
        _periodic(a, q == 2)
        out.append(a)
    return x, y, z, tables, out


def _periodic(a, faces):
    if faces:
        a[0], a[-1] = a[-2].clone(), a[1].clone()
    else:
        a[0], a[-2], a[-1] = a[-3].clone(), a[1].clone(), a[2].clone()


def modes_of(case, y, seed):
    """Inflow modes that decay from the wall, 2 in z by `modes` in time."""
    if not case["modes"]:
        return None
    rng = np.random.default_rng(seed + 77)
    yg = np.concatenate(([2 * y[0] - 0.5 * (y[0] + y[1])], 0.5 * (y[1:] + y[:-1]), [1.5 * y[-1] - 0.5 * y[-2]]))
    m = dict(zmode=2 * np.pi / (case["lz"] * THETA) * np.arange(1, 3), tmode=60.0 * np.arange(1, case["modes"] + 1))
    for key, grid_y in (("qu", yg), ("qv", y), ("qw", yg)):
        amp = 1e-3 * (rng.standard_normal((2, case["modes"])) + 1j * rng.standard_normal((2, case["modes"])))
        shape = np.clip(grid_y / (2 * THETA), 0, None) * np.exp(-grid_y / (2 * THETA))
        m[key] = np.asfortranarray(shape[:, None, None] * amp[None])
    return m


def closure_rows(n, seed):
    """Training rows: features of a normalised gradient tensor and wall distance, a smooth target, weights of both signs of scale."""
    rng = np.random.default_rng(seed)
    rows = np.zeros((n, 28), dtype=np.float32)
    g = rng.standard_normal((n, 9))
    rows[:, :9] = g / np.linalg.norm(g, axis=1, keepdims=True)
    rows[:, 9] = 8.0 * rng.random(n) ** 2
    rows[:, 10] = 0.02 * (1.0 + rows[:, 1] * rows[:, 3] + 0.5 * rows[:, 0] ** 2) * (1.0 - np.exp(-rows[:, 9]))
    rows[:, 11] = np.where(rng.random(n) < 0.05, 0.0, rng.random(n) + 0.1)
    rows[:, 12] = 1e-5
    return rows


def params0(seed):
    """Initial network parameters: uniform weights with half the He bound, zero biases."""
    rng = np.random.default_rng(seed + 5)
    parts = []
    for fan, shape in ((10, 640), (0, 64), (64, 4096), (0, 64), (64, 4096), (0, 64), (64, 64), (0, 1)):
        lim = 0.5 * math.sqrt(6.0 / fan) if fan else 0.0
        parts.append(rng.uniform(-lim, lim, size=shape) if fan else np.zeros(shape))
    return np.concatenate(parts).astype(np.float32)


def _host(a):
    return np.asfortranarray(a.cpu().numpy().T)


def prepare(case, seed):
    B = blgpu()
    if case["kind"] == "train":
        c = B.Closure(case["rows"], case["batch"])
        c.add_rows(closure_rows(case["rows"], seed))
        c.params = params0(seed)
        return dict(case=case, closure=c, seed=seed, theta=params0(seed))
    x, y, z, tables, f = initial(case, seed)
    prec = B.PREC_MIXED if case["precision"] == "mixed" else B.PREC_FP64
    if case["kind"] == "stats":
        s = B.Solver(x, y, z, NU, tables, precision=prec)
        s.set_fields(*[_host(a) for a in f])
        gen = torch.Generator(device=device())
        gen.manual_seed(int(seed) + 3)
        s.upload(B.FIELD_P, _host(torch.rand((z.size + 1, y.size + 1, x.size + 1), generator=gen, device=device(),
                                             dtype=F64)))
        return dict(case=case, solver=s)
    s = B.Solver(x, y, z, NU, tables, scheme=case["scheme"], les=case["les"], cfl=case["cfl"], precision=prec,
                 modes=modes_of(case, y, seed))
    if case["inflow"] != 1:
        s.set_boundary(inflow_flag=case["inflow"], amplitude=0.02, seed=seed)
    if case["wall"]:
        s.set_wall_model(case["wall"], istress_model=1)
    s.set_fields(*[_host(a) for a in f])
    st = dict(case=case, solver=s)
    if case["les"] == 4:
        c = B.Closure(4096, 4096)
        c.add_rows(closure_rows(4096, seed))
        c.params = 0.3 * params0(seed)
        c.install(s, 7.5 * THETA, 3.0)
        st["closure"] = c
    if case["rows"]:
        nc = ((case["nx"] - 1) // 4 + 1, (case["ny"] - 1) // 2 + 1, (case["nz"] - 2) // 4 + 2)
        xc, yc, zc, tc, _ = grid(dict(case, nx=nc[0], ny=nc[1], nz=nc[2]))
        st["les"] = B.Solver(xc, yc, zc, NU, tc, les=2)
        st["closure"] = B.Closure((nc[0] - 1) * (nc[1] - 1) * (nc[2] - 2), 4096)
    if prec == B.PREC_MIXED:
        # FP32 fields are kept as FP32
        st["f32"] = [torch.empty(sh[::-1], dtype=torch.float32) for sh in s.shapes[:3]]
    return st


# ------------------------------------------------------------------- pass ----
def velocity(st):
    """U, V, W of the current state in the snapshot's pinned host memory."""
    s, B = st["solver"], blgpu()
    s.snapshot_begin()
    ptr = [ctypes.POINTER(ctypes.c_double)() for _ in range(5)]
    if B.lib().bl_snapshot_end(s.h, *[ctypes.byref(p) for p in ptr]):
        raise RuntimeError(B.lib().bl_last_error())
    out = []
    for q in range(3):
        sh = s.shapes[q][::-1]
        buf = (ctypes.c_double * int(np.prod(sh))).from_address(ctypes.addressof(ptr[q].contents))
        buf.owner = s  # the memory is the solver's
        a = np.frombuffer(buf, dtype=np.float64).reshape(sh)
        out.append(st["f32"][q].copy_(torch.from_numpy(a)) if "f32" in st else a)
    return out


def run(state):
    case = state["case"]
    if case["kind"] == "train":
        c = state["closure"]
        c.params = state["theta"]
        hist = c.train(case["steps"], case["batch"], lr=1e-3, seed=state["seed"])
        return [c.params, hist]
    s = state["solver"]
    if case["kind"] == "stats":
        st = s.statistics()
        return [st[k] for k in s.STAT_NAMES] + [st["Cf"], s.monitor()[[0, 1, 4, 5, 6]], s.max_divergence()]
    for _ in range(case["steps"]):
        s.compute_dt()
        s.step()
    if case["rows"]:
        c = state["closure"]
        c.clear()
        c.samples_from(s, state["les"], 4, 2, 4, 7.5 * THETA, 1e-3 / THETA)
        return velocity(state) + [c.rows()]
    if case["nx"] * case["ny"] * case["nz"] < 20000:
        out = s.fields()
        return [a.astype(np.float32) for a in out] if case["precision"] == "mixed" else list(out)
    return velocity(state)


def work(case):
    if case["kind"] == "train":
        n = case["batch"] * case["steps"]
        return dict(bytes=n * 12 * 4.0, flops=n * 6.0 * 9089)
    cells = float(case["nx"] * case["ny"] * case["nz"])
    e = 4.0 if case["precision"] == "mixed" else 8.0
    if case["kind"] == "stats":
        return dict(bytes=cells * 4 * e + 9 * 8.0 * case["nx"] * case["ny"], flops=cells * 40.0)
    # every stage reads and writes the three velocities; its pressure solve couples all cells
    stages = case["steps"] * case["scheme"]
    per = 250.0 + 5.0 * math.log2(case["nx"]) + 5.0 * math.log2(case["nz"])
    if case["les"]:
        per += 300.0 if case["les"] < 4 else 300.0 + 2.0 * 9089
    return dict(bytes=stages * 6.0 * e * cells, flops=stages * per * cells)


# ------------------------------------------------------------ exact values ----
class Exact:
    """The solver's algorithm in torch FP64: arrays are (z, y, x), indices 0-based with one ghost cell on each side."""

    def __init__(self, case, seed):
        self.c = case
        x, y, z, tb, (self.U, self.V, self.W) = initial(case, seed)
        dev = self.dev = self.U.device
        if case["precision"] == "mixed":
            self.U, self.V, self.W = (a.float().double() for a in (self.U, self.V, self.W))
        t = lambda a: torch.as_tensor(np.ascontiguousarray(a), dtype=F64, device=dev)  # noqa: E731
        cen = lambda a: np.concatenate(([1.5 * a[0] - 0.5 * a[1]], 0.5 * (a[1:] + a[:-1]), [1.5 * a[-1] - 0.5 * a[-2]]))  # noqa: E731
        xg, yg, zg = cen(x), cen(y), cen(z)
        self.x, self.y, self.z, self.xg, self.yg, self.zg = x, y, z, xg, yg, zg
        self.dx, self.dy, self.dz = (t(np.diff(a)) for a in (x, y, z))
        self.dxg, self.dyg, self.dzg = (t(np.diff(a)) for a in (xg, yg, zg))
        self.w0 = t((yg[1:] - y) / np.diff(yg))
        self.w1 = 1.0 - self.w0
        self.tb = {k: t(v) for k, v in tb.items()}
        self.uc = float(tb["U_top"][-1])
        self.modes = modes_of(case, y, seed)
        self.time = 0.0
        nx, ny, nz = x.size, y.size, z.size
        self.N, self.NM, self.M = nx - 2, ny - 1, nz - 2
        N, NM, M = self.N, self.NM, self.M
        mins = [np.diff(a).min() for a in (xg, yg, zg)]
        self.mins = mins
        kxx = t(2 * (np.cos(np.pi * np.arange(N) / N) - 1) / mins[0] ** 2)
        kzz = t(2 * (np.cos(2 * np.pi * np.arange(M // 2 + 1) / M) - 1) / mins[2] ** 2)
        self.lam = kzz[:, None] + kxx[None, :]
        a = 1 / np.diff(y) / np.diff(yg)[1:]      # to the cell above
        c = 1 / np.diff(y) / np.diff(yg)[:-1]     # to the cell below
        b = -a - c
        b[0], b[-1] = b[0] + c[0], b[-1] + a[-1]
        self.tri = (a, b, c)
        self.rot = torch.exp(-1j * np.pi * torch.arange(N, device=dev, dtype=F64) / (2 * N))

    def nu_eff(self):
        les = self.c["les"]
        return None if les == 0 else self.dynamic(les == 3)

    # -- momentum right-hand sides on the cells (1..nzg-2, 1..nyg-2, 1..nxg-2)
    def rhs(self):
        U, V, W, N = self.U, self.V, self.W, self.N
        dx, dy, dz, dxg, dyg, dzg = self.dx, self.dy[:, None], self.dz[:, None, None], self.dxg, self.dyg[:, None], self.dzg[:, None, None]
        w0, w1 = self.w0[:, None], self.w1[:, None]
        nt = self.nu_eff()
        I, A, Bk = slice(1, -1), slice(2, None), slice(None, -2)
        # u at faces 1..nx-3
        up, ue, uw = U[I, I, 1:N], U[I, I, 2:N + 1], U[I, I, 0:N - 1]
        un, us, ut, ub = U[I, A, 1:N], U[I, Bk, 1:N], U[A, I, 1:N], U[Bk, I, 1:N]
        if nt is None:
            ex = ew = en = es = et = eb = NU
        else:
            yav = w0 * nt[:, :-1] + w1 * nt[:, 1:]  # at y faces
            ed = 0.5 * (yav[:, :, :-1] + yav[:, :, 1:])
            xz = 0.25 * (nt[:-1, :, :-1] + nt[:-1, :, 1:] + nt[1:, :, :-1] + nt[1:, :, 1:])
            ew, ex = NU + nt[I, I, 1:N], NU + nt[I, I, 2:N + 1]
            es, en = NU + ed[I, :-1, 1:N], NU + ed[I, 1:, 1:N]
            eb, et = NU + xz[:-1, I, 1:N], NU + xz[1:, I, 1:N]
        r = -((0.5 * (up + ue)) ** 2 - (0.5 * (uw + up)) ** 2) / dxg[1:N]
        vn = 0.5 * (V[I, 1:, 1:N] + V[I, 1:, 2:N + 1])
        vs = 0.5 * (V[I, :-1, 1:N] + V[I, :-1, 2:N + 1])
        r -= ((w0[1:] * up + w1[1:] * un) * vn - (w0[:-1] * us + w1[:-1] * up) * vs) / dy
        wt = 0.5 * (W[1:, I, 1:N] + W[1:, I, 2:N + 1])
        wb = 0.5 * (W[:-1, I, 1:N] + W[:-1, I, 2:N + 1])
        r -= (0.5 * (up + ut) * wt - 0.5 * (ub + up) * wb) / dz
        r += (ex * (ue - up) / dx[1:N] - ew * (up - uw) / dx[0:N - 1]) / dxg[1:N]
        r += (en * (un - up) / dyg[1:] - es * (up - us) / dyg[:-1]) / dy
        r += (et * (ut - up) / dzg[1:] - eb * (up - ub) / dzg[:-1]) / dz
        fu = r
        # v at x centres 1..nxg-3, y faces 1..ny-2
        C = slice(1, N + 1)
        J = slice(1, -1)
        vp, ve, vw = V[I, J, C], V[I, J, 2:N + 2], V[I, J, 0:N]
        vn, vs, vt, vb = V[I, A, C], V[I, Bk, C], V[A, J, C], V[Bk, J, C]
        if nt is None:
            ex = ew = en = es = et = eb = NU
        else:
            ew, ex = NU + ed[I, J, 0:N], NU + ed[I, J, 1:N + 1]
            es, en = NU + nt[I, 1:-2, C], NU + nt[I, 2:-1, C]
            eb, et = NU + 0.5 * (yav[:-2, J, C] + yav[1:-1, J, C]), NU + 0.5 * (yav[1:-1, J, C] + yav[2:, J, C])
        r = -((0.5 * (vp + vn)) ** 2 - (0.5 * (vs + vp)) ** 2) / dyg[J]
        uy = w0[J] * U[I, 1:-2] + w1[J] * U[I, 2:-1]
        r -= (uy[:, :, 1:N + 1] * 0.5 * (vp + ve) - uy[:, :, 0:N] * 0.5 * (vw + vp)) / dx[0:N]
        wy = w0[J] * W[:, 1:-2, C] + w1[J] * W[:, 2:-1, C]
        r -= (0.5 * (vp + vt) * wy[1:] - 0.5 * (vb + vp) * wy[:-1]) / dz
        r += (ex * (ve - vp) / dxg[1:N + 1] - ew * (vp - vw) / dxg[0:N]) / dx[0:N]
        r += (en * (vn - vp) / dy[1:] - es * (vp - vs) / dy[:-1]) / dyg[J]
        r += (et * (vt - vp) / dzg[1:] - eb * (vp - vb) / dzg[:-1]) / dz
        fv = r
        # w at x centres 1..nxg-3, z faces 1..nz-2
        wp, we, ww = W[J, I, C], W[J, I, 2:N + 2], W[J, I, 0:N]
        wn, ws, wt, wb = W[J, A, C], W[J, Bk, C], W[A, I, C], W[Bk, I, C]
        if nt is None:
            ex = ew = en = es = et = eb = NU
        else:
            zav = 0.5 * (nt[1:-2] + nt[2:-1])
            yz = 0.5 * (yav[1:-2] + yav[2:-1])
            ew, ex = NU + xz[1:-1, I, 0:N], NU + xz[1:-1, I, 1:N + 1]
            es, en = NU + yz[:, :-1, C], NU + yz[:, 1:, C]
            eb, et = NU + nt[1:-2, I, C], NU + nt[2:-1, I, C]
            del zav
        r = -((0.5 * (wp + wt)) ** 2 - (0.5 * (wb + wp)) ** 2) / dzg[J]
        uz = 0.5 * (U[1:-2, I] + U[2:-1, I])
        r -= (uz[:, :, 1:N + 1] * 0.5 * (wp + we) - uz[:, :, 0:N] * 0.5 * (ww + wp)) / dx[0:N]
        vz = 0.5 * (V[1:-2, :, C] + V[2:-1, :, C])
        r -= (vz[:, 1:] * (w0[1:] * wp + w1[1:] * wn) - vz[:, :-1] * (w0[:-1] * ws + w1[:-1] * wp)) / dy
        r += (ex * (we - wp) / dxg[1:N + 1] - ew * (wp - ww) / dxg[0:N]) / dx[0:N]
        r += (en * (wn - wp) / dyg[1:] - es * (wp - ws) / dyg[:-1]) / dy
        r += (et * (wt - wp) / dz[1:] - eb * (wp - wb) / dz[:-1]) / dzg[J]
        return fu, fv, r

    def add(self, old, f):
        """old + f on the cells that a stage moves."""
        N = self.N
        n = [a.clone() for a in old]
        n[0][1:-1, 1:-1, 1:N] += f[0]
        n[1][1:-1, 1:-1, 1:N + 1] += f[1]
        n[2][1:-1, 1:-1, 1:N + 1] += f[2]
        return n

    # -- boundary planes
    def boundary(self, old, stage, dt, t):
        U, V, W, tb = self.U, self.V, self.W, self.tb
        coef = (8 / 15, 2 / 3, 1.0)[stage] * dt * self.uc
        ui, vi, wi = tb["U_inlet"][None, :], tb["V_inlet"][None, :], tb["W_inlet"][None, :]
        if self.modes:
            zc, zf = torch.as_tensor(self.zg, device=self.dev), torch.as_tensor(self.z, device=self.dev)
            for n, bz in enumerate(self.modes["zmode"]):
                for m, om in enumerate(self.modes["tmode"]):
                    q = [torch.as_tensor(np.ascontiguousarray(self.modes[k][:, n, m]), device=self.dev)[None] for k in ("qu", "qv", "qw")]
                    ec = torch.exp(1j * (float(bz) * zc - float(om) * t))[:, None]
                    ef = torch.exp(1j * (float(bz) * zf - float(om) * t))[:, None]
                    ui, vi, wi = ui + (q[0] * ec).real, vi + (q[1] * ec).real, wi + (q[2] * ef).real
        U[:, :, 0], V[:, :, 0], W[:, :, 0] = ui, vi, wi
        for a, o, h in ((U, old[0], self.x[-2] - self.x[-3]), (V, old[1], self.xg[-2] - self.xg[-3]), (W, old[2], self.xg[-2] - self.xg[-3])):
            v = o[:, :, -2] - coef * (o[:, :, -2] - o[:, :, -3]) / h
            a[:, :, -2], a[:, :, -1] = v, v
        Q = ((U[1:-2, 1:-1, 0] - U[1:-2, 1:-1, -2]) * self.dy[None]).sum()
        for a, faces in ((U, False), (V, False), (W, True)):
            _periodic(a, faces)
        U[:, -1], V[:, -1], W[:, -1] = tb["U_top"], tb["V_top"], tb["W_top"]
        U[:, 0], V[:, 0], W[:, 0] = -U[:, 1], 0.0, -W[:, 1]
        Q = Q - (tb["V_top"][1:-2] * self.dx[:-1]).sum() * self.M
        U[:, :, -2] += Q / (self.y[-1] - self.y[0]) / self.M
        U[:, :, -1] = U[:, :, -2]

    # -- pressure projection
    def project(self):
        U, V, W, N, NM, M = self.U, self.V, self.W, self.N, self.NM, self.M
        kz, ix = slice(1, M + 1), slice(1, N + 1)
        r = (U[kz, 1:-1, 1:N + 1] - U[kz, 1:-1, 0:N]) / self.dx[:N]
        r += (V[kz, 1:, ix] - V[kz, :-1, ix]) / self.dy[:, None]
        r += (W[1:M + 1, 1:-1, ix] - W[0:M, 1:-1, ix]) / self.dz[:M, None, None]
        r = (torch.fft.rfft(torch.cat((r, r.flip(2)), 2), dim=2)[:, :, :N] * self.rot).real  # cosine transform
        r = torch.fft.rfft(r, dim=0)
        a, b, c = self.tri
        up = []
        for j in range(NM):
            p = b[j] + self.lam
            if j == 0:
                p[0, 0] *= 1.5
            else:
                p -= c[j] * up[-1]
                r[:, j] -= c[j] * r[:, j - 1]
            p = 1.0 / p
            r[:, j] *= p
            up.append(a[j] * p)
        for j in range(NM - 2, -1, -1):
            r[:, j] -= up[j] * r[:, j + 1]
        del up
        r = torch.fft.irfft(r, n=M, dim=0)
        r = torch.cat((r * self.rot.conj(), torch.zeros((M, NM, 1), dtype=torch.complex128, device=self.dev)), 2)
        r = torch.fft.irfft(r, n=2 * N, dim=2)[:, :, :N]
        phi = torch.cat((r, r[:1]), 0)                   # cells 1..M, and M+1 = 1
        phi = torch.cat((phi, phi[:, :, -1:]), 2)        # cells 1..N, and N+1 = N
        U[1:-1, 1:-1, 1:N + 1] -= (phi[:, :, 1:] - phi[:, :, :-1]) / self.dxg[1:N + 1]
        V[1:-1, 1:-1, 1:-1] -= (phi[:, 1:] - phi[:, :-1]) / self.dyg[1:-1, None]
        W[1:-1, 1:-1, 1:-1] -= (phi[1:] - phi[:-1]) / self.dzg[1:-1, None, None]

    def dt(self):
        if self.c["cfl"] < 0:
            return -self.c["cfl"]
        I = slice(1, -1)
        conv = min(float((d / a.abs()).max()) for d, a in (
            (self.dxg[1:], self.U[I, I, 1:]), (self.dyg[1:, None], self.V[I, 1:, I]), (self.dzg[1:, None, None], self.W[1:, I, I])))
        return self.c["cfl"] * min(conv, min(h ** 2 / NU for h in self.mins))

    def step(self):
        dt, t0, rk3 = self.dt(), self.time, self.c["scheme"] == 3
        old = [self.U, self.V, self.W]
        f1 = None
        for s in range(3 if rk3 else 2):
            f = self.rhs()
            if s == 0:
                f1, co = f, (0.0, 8 / 15 if rk3 else 0.5)
            else:
                co = ((0.25, 5 / 12), (0.25, 0.75))[s - 1] if rk3 else (0.0, 1.0)
            self.U, self.V, self.W = self.add(old, [dt * (co[0] * p + co[1] * q) for p, q in zip(f1, f)])
            ts = t0 + ((8 / 15, 2 / 3, 1.0) if rk3 else (0.5, 1.0))[s] * dt
            self.boundary(old, s, dt, ts)
            self.project()
            self.boundary(old, s, dt, ts)
            self.time = ts

    # -- dynamic Smagorinsky eddy viscosity (z-averaged, or per cell)
    def dynamic(self, percell):
        U, V, W = self.U, self.V, self.W
        n3, n2, n1 = U.shape[0], U.shape[1], V.shape[2]
        ar = lambda n: torch.arange(n, device=self.dev)  # noqa: E731

        def ends(n, first, *last):
            k = ar(n)
            k[0] = first
            for q, v in enumerate(last):
                k[n - len(last) + q] = v
            return k

        zc, zf = ends(n3, n3 - 3, 1, 2), ends(n3 - 1, n3 - 3, 1)
        xc = ends(n1, n1 - 3, 1, 2) if percell else ar(n1).clamp(1, n1 - 2)
        xf = ends(n1 - 1, n1 - 3, 1) if percell else ar(n1 - 1).clamp(1, n1 - 3)

        def test_filter(g, lo, hi):
            y = g.clone()
            y[:, lo + 1:hi] = g[:, lo:hi - 1] / 6 + 2 / 3 * g[:, lo + 1:hi] + g[:, lo + 2:hi + 1] / 6
            y[:, lo], y[:, hi] = 2 / 3 * g[:, lo] + g[:, lo + 1] / 3, g[:, hi - 1] / 3 + 2 / 3 * g[:, hi]
            out = torch.zeros_like(y)
            v = y[:, :, :-2] / 6 + 2 / 3 * y[:, :, 1:-1] + y[:, :, 2:] / 6
            out[1:-1, :, 1:-1] = v[:-2] / 6 + 2 / 3 * v[1:-1] + v[2:] / 6
            return out

        def strain(u, v, w):
            dx, dy, dz = self.dx, self.dy[:, None], self.dz[:, None, None]
            dxg, dyg, dzg = self.dxg, self.dyg[:, None], self.dzg[:, None, None]
            s = [(u[1:-1, 1:-1].diff(dim=2)) / dx, (v[1:-1, :, 1:-1].diff(dim=1)) / dy, (w[:, 1:-1, 1:-1].diff(dim=0)) / dz]
            a = 0.5 * (u[1:-1].diff(dim=1) / dyg + v[1:-1].diff(dim=2) / dxg)
            b = 0.5 * (u[:, 1:-1].diff(dim=0) / dzg + w[:, 1:-1].diff(dim=2) / dxg)
            c = 0.5 * (v[:, :, 1:-1].diff(dim=0) / dzg + w[:, :, 1:-1].diff(dim=1) / dyg)
            s.append(0.25 * (a[:, :-1, :-1] + a[:, :-1, 1:] + a[:, 1:, :-1] + a[:, 1:, 1:]))
            s.append(0.25 * (b[:-1, :, :-1] + b[:-1, :, 1:] + b[1:, :, :-1] + b[1:, :, 1:]))
            s.append(0.25 * (c[:-1, :-1] + c[:-1, 1:] + c[1:, :-1] + c[1:, 1:]))
            return s, torch.sqrt(2 * (s[0] ** 2 + s[1] ** 2 + s[2] ** 2) + 4 * (s[3] ** 2 + s[4] ** 2 + s[5] ** 2))

        def pad(a):
            return torch.nn.functional.pad(a, (1, 1, 1, 1, 1, 1))

        remap = lambda g: g[zc][:, :, xc]  # noqa: E731
        filt = lambda g: test_filter(g, 1, n2 - 2)[1:-1, 1:-1, 1:-1]  # noqa: E731
        cu = 0.5 * (U[:, :, xc - 1] + U[:, :, xc])
        cv = torch.zeros((n3, n2, n1), dtype=F64, device=self.dev)
        cv[:, 1:-1] = 0.5 * (V[:, :-1] + V[:, 1:])
        cw = 0.5 * (W[zc - 1] + W[zc])
        h = [filt(a) for a in (cu, cv, cw)]
        p = [remap(a) for a in (cu, cv, cw)]
        pairs = ((0, 0), (1, 1), (2, 2), (0, 1), (0, 2), (1, 2))
        L = [filt(p[a] * p[b]) - h[a] * h[b] for a, b in pairs]
        s, S = strain(U, V, W)
        hs = [filt(remap(pad(S * q))) for q in s]
        Uf = test_filter(U, 0, n2 - 1)[zc][:, :, xf]
        Vf = test_filter(V, 0, n2 - 2)[zc][:, :, xc]
        Wf = test_filter(W, 0, n2 - 1)[zf][:, :, xc]
        sh, Sh = strain(Uf, Vf, Wf)
        M = [4 * Sh * a - b for a, b in zip(sh, hs)]
        g = (1, 1, 1, 2, 2, 2)
        lm = sum(q * a * b for q, a, b in zip(g, M, L))
        mm = sum(q * a * a for q, a in zip(g, M))
        if percell:
            nt = remap(pad(-0.5 * lm / mm * S))
        else:
            nt = pad(-0.5 * (lm[:-1].mean(0) / mm[:-1].mean(0)) * S)
        nt = torch.nan_to_num(nt, nan=0.0).clamp(min=0.0)
        nt[:, 0], nt[:, -1] = nt[:, 1], nt[:, -2]
        return nt


def exact_train(case, seed):
    """Adam on weighted batches drawn by the library's counter hash of (seed, step, slot)."""
    dev, n, B = device(), case["rows"], case["batch"]
    rows = torch.from_numpy(closure_rows(n, seed)).to(dev).double()
    w = rows[:, 11] * ((rows[:, 11] > 0).sum() / rows[:, 11].sum())
    th = torch.from_numpy(params0(seed)).to(dev).double()
    m, v, hist = torch.zeros_like(th), torch.zeros_like(th), []
    u64 = np.uint64

    def mix(a):
        a = a + u64(0x9E3779B97F4A7C15)
        a = (a ^ (a >> u64(30))) * u64(0xBF58476D1CE4E5B9)
        a = (a ^ (a >> u64(27))) * u64(0x94D049BB133111EB)
        return a ^ (a >> u64(31))

    for step in range(case["steps"]):
        with np.errstate(over="ignore"):
            slot = np.arange(B, dtype=u64) + u64(step * 0x100000001B3)
            pick = mix(u64(seed) ^ mix(slot)) % u64(n)
        pick = torch.from_numpy(pick.astype(np.int64)).to(dev)
        X, t, wb = rows[pick, :10], rows[pick, 10], w[pick]
        p = th.clone().requires_grad_(True)
        W1, b1, W2, b2, W3, b3, W4, b4 = torch.split(p, [640, 64, 4096, 64, 4096, 64, 64, 1])
        act = torch.nn.functional.silu
        h = act(X @ W1.view(64, 10).T + b1)
        h = act(h @ W2.view(64, 64).T + b2)
        h = act(h @ W3.view(64, 64).T + b3)
        loss = (wb * (h @ W4 + b4 - t) ** 2).mean()
        g, = torch.autograd.grad(loss, p)
        hist.append(float(loss.detach()))
        m, v = 0.9 * m + 0.1 * g, 0.999 * v + 0.001 * g * g
        th = th - 1e-3 * (m / (1 - 0.9 ** (step + 1))) / (torch.sqrt(v / (1 - 0.999 ** (step + 1))) + 1e-8)
    return [th, np.array(hist)]


def exact_stats(case, seed):
    x, y, z, _, (U, V, W) = initial(case, seed)
    gen = torch.Generator(device=device())
    gen.manual_seed(int(seed) + 3)
    P = torch.rand((z.size + 1, y.size + 1, x.size + 1), generator=gen, device=device(), dtype=F64)
    if case["precision"] == "mixed":
        U, V, W, P = (a.float().double() for a in (U, V, W, P))
    t = lambda a: torch.as_tensor(np.ascontiguousarray(a), dtype=F64, device=U.device)  # noqa: E731
    yg = np.concatenate(([1.5 * y[0] - 0.5 * y[1]], 0.5 * (y[1:] + y[:-1]), [1.5 * y[-1] - 0.5 * y[-2]]))
    w0 = t((yg[1:] - y) / np.diff(yg))[:, None]
    u = w0 * U[1:-1, :-1] + (1 - w0) * U[1:-1, 1:]
    v = 0.5 * (V[1:-1, :, :-1] + V[1:-1, :, 1:])
    w = 0.5 * (W[:-2, :, :-1] + W[:-2, :, 1:])
    w = w0 * w[:, :-1] + (1 - w0) * w[:, 1:]
    p = P[1:-1, :-1, :-1]
    nz = z.size - 2
    means = [u.mean(0), v.mean(0), w.sum(0) / nz, (u * u).mean(0), (v * v).mean(0), (w * w).sum(0) / nz, (u * v).mean(0), p.mean(0), (p * p).mean(0)]
    cf = 2 * (NU * (U[1:-1, 1] - U[1:-1, 0]).mean(0) / (yg[1] - yg[0]) - (u[:, 0] * v[:, 0]).mean(0))
    I = slice(1, -1)
    ui, vi, wi = U[I, I, 1:-1], V[I, 1:-1, I], W[1:-1, I, I]
    mon = torch.stack((ui.sum(), vi.sum(), ui.max(), vi.max(), wi.max()))
    div = U[I, I].diff(dim=2)[:, :, :-1] / t(np.diff(x))[:-1]
    div = div + V[I, :, 1:-2].diff(dim=1) / t(np.diff(y))[:, None] + W[:, I, 1:-2].diff(dim=0) / t(np.diff(z))[:, None, None]
    return [a.T for a in means] + [cf, mon, float(div.abs().max())]


def exact(case, seed):
    if case["kind"] == "train":
        return exact_train(case, seed)
    if case["kind"] == "stats":
        return exact_stats(case, seed)
    if case["les"] in (1, 4):  # a random stream, and a network in 16 bits: no such values
        return None
    e = Exact(case, seed)
    for _ in range(case["steps"]):
        e.step()
    out = [e.U, e.V, e.W]
    if case["nx"] * case["ny"] * case["nz"] < 20000:
        out = [np.asfortranarray(a.cpu().numpy().T) for a in out]
    return out + ([None] if case["rows"] else [])
