"""Measured cases of the ECSIM cycle on one GPU.

listed() holds the cases, draw() more of the same ranges; prepare() makes what
a run has in hand (a context with its particles and fields on the GPU, started),
run() is one pass through the public entry points, work() what the pass cannot
do without, exact() the same pass in plain torch.

The plasmas are those of the repository's decks, tests and benchmark:
- "magnetised": cells of 0.25 d_i, electrons (q/m -64, thermal 0.045) and ions
  (q/m 1, thermal 0.0056), B0 = 0.01 z plus a seeded spectrum of 1e-3 B0,
  dt 0.1;
- "twostream": two electron beams of +-0.2 with thermal 0.01 on a line of
  cells of 0.245, dt 0.1;
- "weibel": electrons with thermal (0.3, 0.1, 0.3) and ions (q/m 0.01, thermal
  0.01) on cells of 0.1, dt 0.05.
Particles are loaded as the dense load does: (sub + U)/ppc per axis in each
cell, Maxwellian velocities, equal charges, load order.
"""
import math

import numpy as np
import torch

import tpic_amd
from tpic_amd import gradient as G
from tpic_amd import runtime as R

FOUR_PI = 4.0 * math.pi
THETA = 0.5

PLASMAS = {
    "magnetised": dict(spacing=0.25, q_over_m=(-64.0, 1.0), rho=(1.0, 1.0), dt=0.1,
                       thermal=((0.045,) * 3, (0.0056,) * 3), drift=((0.0, 0.0, 0.0), (0.0, 0.0, 0.0)),
                       b0=(0.0, 0.0, 0.01), b_wave=1e-5, e_wave=1e-6),
    "twostream": dict(spacing=0.2454369260617026, q_over_m=(-1.0, -1.0), rho=(0.5, 0.5), dt=0.1,
                      thermal=((0.01,) * 3, (0.01,) * 3), drift=((0.2, 0.0, 0.0), (-0.2, 0.0, 0.0)),
                      b0=(0.0, 0.0, 0.0), b_wave=1e-5, e_wave=1e-3),
    "weibel": dict(spacing=0.1, q_over_m=(-1.0, 0.01), rho=(1.0, 1.0), dt=0.05,
                   thermal=((0.3, 0.1, 0.3), (0.01,) * 3), drift=((0.0, 0.0, 0.0), (0.0, 0.0, 0.0)),
                   b0=(0.0, 0.0, 0.0), b_wave=1e-3, e_wave=1e-4),
}
MASS = {"fp64": R.MASS_FP64, "fp32": R.MASS_FP32, "bf16x3": R.MASS_BF16X3}
# Field faces per axis (both faces alike); a closed axis mirrors its particles.
PERIODIC = (R.FACE_PERIODIC, R.FACE_PERIODIC)
FACES = {"periodic": (PERIODIC,) * 3,
         "pec_y": (PERIODIC, (R.FACE_PEC, R.FACE_PEC), PERIODIC),
         "pmc_xz": ((R.FACE_PMC, R.FACE_PMC), PERIODIC, (R.FACE_PMC, R.FACE_PEC))}
SMOOTHING = {"none": None, "face7": (R.SMOOTH_FACE7, 3, 0.5), "binomial27": (R.SMOOTH_BINOMIAL27, 2, 0.0)}
ATTRIBUTES = ("rx", "ry", "rz", "u", "v", "w", "q", "cell", "id")


def _case(call, plasma, cells, ppc, mass="fp64", faces="periodic", smoothing="none", scalars=False, cycles=1, name=None):
    c = dict(call=call, plasma=plasma, nx=cells[0], ny=cells[1], nz=cells[2], px=ppc[0], py=ppc[1], pz=ppc[2],
             mass=mass, faces=faces, smoothing=smoothing, scalars=scalars, cycles=cycles)
    if name:
        c["name"] = name
    return c


def listed():
    return [
        # The smallest 3D box of the tests and decks, as run for quick studies: latency and launches.
        _case("cycle", "magnetised", (16, 16, 16), (4, 4, 4), name="cycle_16cube"),
        # A 1D two-stream run of the full-size tests: a line of cells, many particles in each.
        _case("cycle", "twostream", (1024, 1, 1), (1000, 1, 1), name="cycle_1d_twostream"),
        # A 2D Weibel run at the full size of the tests: one cell across, ordinary counts.
        _case("cycle", "weibel", (512, 512, 1), (10, 10, 1), name="cycle_2d_weibel"),
        # An odd box with few particles a cell, single precision mass products.
        _case("cycle", "magnetised", (45, 37, 29), (3, 3, 3), mass="fp32", name="cycle_ragged_fp32"),
        # A middle-sized production run that reports its scalars every cycle (DiagnosticsOutputCycle 1).
        _case("cycle", "magnetised", (64, 64, 64), (4, 4, 4), mass="bf16x3", scalars=True, name="cycle_64cube_scalars"),
        # A closed box: conducting walls in y, mirrored particles, odd sizes.
        _case("cycle", "magnetised", (61, 47, 33), (3, 3, 3), faces="pec_y", name="cycle_walls"),
        # Energy-conserving smoothing, as decks ask for it.
        _case("cycle", "magnetised", (48, 48, 48), (3, 3, 3), smoothing="face7", name="cycle_smoothed"),
        # The stages called one by one, as a caller with its own pipeline does.
        _case("stages", "magnetised", (56, 40, 48), (4, 4, 2), name="stages"),
        # A gradient through cycles of a small two-stream line: forward, checkpoints, adjoint.
        _case("gradient", "twostream", (1024, 1, 1), (100, 1, 1), cycles=20, name="gradient_1d"),
        # A gradient through cycles of a 2D Weibel plane.
        _case("gradient", "weibel", (192, 160, 1), (5, 5, 1), cycles=10, name="gradient_2d"),
        # The benchmark's box, in both of the forms that it reports first and last.
        _case("cycle", "magnetised", (128, 128, 128), (4, 4, 4), name="cycle_128cube"),
        _case("cycle", "magnetised", (128, 128, 128), (4, 4, 4), mass="bf16x3", name="cycle_128cube_bf16x3"),
    ]


def _log_int(rng, low, high):
    return int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))


def draw(rng):
    """3D boxes of 12 to 128 cells a side, planes of 32 to 640, lines of 128 to 4096, 8 to 64 particles a cell
    and species (lines up to 1200), every mass form, closed faces and smoothing in FP64."""
    kind = rng.choice(("box", "box", "box", "closed", "smoothed", "plane", "line", "stages", "gradient_line",
                       "gradient_plane"))
    if kind in ("line", "gradient_line"):
        small = kind == "gradient_line"
        nx = _log_int(rng, 128, 1536 if small else 4096)
        ppc = _log_int(rng, 24, 160 if small else 1200)
        mass = "fp64" if small else rng.choice(("fp64", "fp64", "fp32", "bf16x3"))
        return _case("gradient" if small else "cycle", "twostream", (nx, 1, 1), (ppc, 1, 1), mass=mass,
                     cycles=rng.choice((8, 12, 16)) if small else 1)
    if kind in ("plane", "gradient_plane"):
        small = kind == "gradient_plane"
        nx, ny = (_log_int(rng, 32, 192 if small else 640) for _ in range(2))
        p = rng.randint(3, 5 if small else 10)
        return _case("gradient" if small else "cycle", "weibel", (nx, ny, 1), (p, p, 1),
                     cycles=rng.choice((4, 6, 8)) if small else 1)
    high = 128 if kind == "box" else 72
    cells = tuple(_log_int(rng, 12, high) for _ in range(3))
    ppc = rng.choice(((2, 2, 2), (3, 3, 3), (4, 3, 2), (4, 4, 2), (4, 4, 4)))
    if kind == "box":
        return _case("cycle", "magnetised", cells, ppc, mass=rng.choice(("fp64", "fp64", "fp32", "bf16x3")),
                     scalars=rng.random() < 0.5)
    if kind == "closed":
        return _case("cycle", "magnetised", cells, ppc, faces=rng.choice(("pec_y", "pmc_xz")))
    if kind == "smoothed":
        return _case("cycle", "magnetised", cells, ppc, smoothing=rng.choice(("face7", "binomial27")))
    return _case("stages", "magnetised", cells, ppc)


# ---- inputs, in plain torch ------------------------------------------------

def _cells(case):
    return case["nx"], case["ny"], case["nz"]


def _per_cell(case):
    return case["px"] * case["py"] * case["pz"]


def _particles(case, species, seed):
    """(attribute, values) of one species, one attribute at a time, on the GPU."""
    p, (nx, ny, nz), ppc = PLASMAS[case["plasma"]], _cells(case), (case["px"], case["py"], case["pz"])
    per, n = _per_cell(case), nx * ny * nz * _per_cell(case)
    gen = torch.Generator(device="cuda").manual_seed(1000003 * int(seed) + 101 * species + 12345)
    index = torch.arange(n, device="cuda")
    sub = index % per
    below = (1, ppc[0], ppc[0] * ppc[1])
    for a, name in enumerate(("rx", "ry", "rz")):
        u = torch.rand(n, generator=gen, device="cuda", dtype=torch.float64)
        yield name, u.add_((sub // below[a]) % ppc[a]).mul_(1.0 / ppc[a]).clamp_(max=1.0 - 2.0 ** -53)
    del sub
    for a, name in enumerate(("u", "v", "w")):
        v = torch.randn(n, generator=gen, device="cuda", dtype=torch.float64)
        yield name, v.mul_(p["thermal"][species][a]).add_(p["drift"][species][a])
    sign = 1.0 if p["q_over_m"][species] > 0 else -1.0
    charge = sign * p["spacing"] ** 3 / per * p["rho"][species] / FOUR_PI
    yield "q", torch.full((n,), charge, dtype=torch.float64, device="cuda")
    cell = index // per
    key = (cell % nx + 2) + (nx + 4) * ((cell // nx % ny + 2) + (ny + 4) * (cell // (nx * ny) + 2))
    yield "cell", key.to(torch.int32)
    del cell, key
    yield "id", index + species * n


def _waves(case, seed, centre, amplitude, base):
    """[3, nz, ny, nx]: base plus four transverse waves of seeded phases, at the cell centres or lower nodes."""
    nx, ny, nz = _cells(case)
    rng = np.random.default_rng(int(seed) * 2 + centre)
    s = [((torch.arange(m, device="cuda", dtype=torch.float64) + 0.5 * centre) / m) for m in (nx, ny, nz)]
    out = torch.zeros((3, nz, ny, nx), dtype=torch.float64, device="cuda")
    for c in range(3):
        out[c] = base[c]
    for _ in range(4):
        k = rng.integers(1, 4, 3).astype(float) * np.array([1.0, ny > 1, nz > 1])
        pol = np.cross(rng.uniform(-1.0, 1.0, 3), k)
        pol /= max(float(np.linalg.norm(pol)), 1e-3)
        phase = rng.uniform(0.0, 2.0 * math.pi)
        wave = torch.cos(2.0 * math.pi * (k[0] * s[0][None, None, :] + k[1] * s[1][None, :, None]
                                          + k[2] * s[2][:, None, None]) + phase)
        for c in range(3):
            out[c] += amplitude * float(pol[c]) * wave
    return out


def _pad(v):
    """Unique nodes [3, nz, ny, nx] with their periodic duplicates."""
    v = torch.cat((v, v[..., :1]), 3)
    v = torch.cat((v, v[..., :1, :]), 2)
    return torch.cat((v, v[:, :1]), 1)


def _fields(case, seed):
    """E at nodes (with duplicates) and B at cells; a closed box starts without E."""
    p = PLASMAS[case["plasma"]]
    b = _waves(case, seed, 1, p["b_wave"], p["b0"])
    e = _pad(_waves(case, seed, 0, p["e_wave"], (0.0, 0.0, 0.0)))
    if case["faces"] != "periodic":
        e.zero_()
    return e.reshape(-1).contiguous(), b.reshape(-1).contiguous()


# ---- the framework's side --------------------------------------------------

class _Pointer:
    """A device array of a context; the tensor made of it keeps it, and so the context, alive."""

    def __init__(self, owner, address, count, kind):
        self.owner = owner
        self.__cuda_array_interface__ = {"data": (address, False), "shape": (count,), "typestr": kind, "version": 2,
                                         "strides": None}


class _State:
    """A context and torch views of its device arrays (the particle slots alternate, so a view is kept per address)."""

    def __init__(self, sim, run=None, inputs=None):
        self.sim, self.gradient, self.inputs, self.views = sim, run, inputs, {}
        self.scalars, self.stages = False, False

    def view(self, address, count, kind="<f8"):
        v = self.views.get(address)
        if v is None:
            v = self.views[address] = torch.as_tensor(_Pointer(self.sim, address, count, kind), device="cuda")
        return v

    def field(self, which):
        return self.view(self.sim.device_field(which), 3 * (self.sim.ncells if which == R.FIELD_B else self.sim.nodes))

    def particles(self, s):
        n = self.sim.species[s][1]
        return {name: self.view(self.sim.device_particles(s, a), n, {"cell": "<i4", "id": "<i8"}.get(name, "<f8"))
                for a, name in enumerate(ATTRIBUTES)}


def _simulation(case, tolerance=1e-10, iterations=100):
    p, cells = PLASMAS[case["plasma"]], _cells(case)
    n = cells[0] * cells[1] * cells[2] * _per_cell(case)
    faces = FACES[case["faces"]]
    return tpic_amd.Simulation(cells, [m * p["spacing"] for m in cells], [(q, n) for q in p["q_over_m"]], dt=p["dt"],
                               theta=THETA, gmres_tolerance=tolerance, gmres_max_iterations=iterations,
                               particle_periodic=[int(f == PERIODIC) for f in faces], mass_kernel=MASS[case["mass"]],
                               field_faces=faces, smoothing=SMOOTHING[case["smoothing"]])


def prepare(case, seed):
    e, b = _fields(case, seed)
    if case["call"] == "gradient":
        sim = _simulation(case, tolerance=1e-13, iterations=400)
        base = [{k: v.cpu().numpy() for k, v in _particles(case, s, seed)} for s in range(2)]
        n = sim.species[0][1]
        run = G.Run(sim, base, [0, n], case["cycles"], (case["cycles"] + 1) // 2, weight_e=1.0, weight_b=1.0)
        v = torch.from_numpy(np.concatenate([np.stack([x["u"], x["v"], x["w"]], axis=1) for x in base]))
        q = torch.from_numpy(np.concatenate([x["q"] for x in base]))
        return _State(sim, run, [x.requires_grad_() for x in (v, q, e.cpu(), b.cpu())])
    sim = _simulation(case)
    state = _State(sim)
    state.scalars, state.stages = case["scalars"], case["call"] == "stages"
    for s in range(2):
        slot = state.particles(s)
        for name, values in _particles(case, s, seed):
            slot[name].copy_(values)
    state.field(R.FIELD_E).copy_(e)
    state.field(R.FIELD_B).copy_(b)
    torch.cuda.synchronize()
    sim.initialize()
    sim.synchronize()
    return state


def run(state):
    sim = state.sim
    if state.gradient is not None:
        value = G.FieldEnergy.apply(*state.inputs, state.gradient)
        grads = torch.autograd.grad(value, state.inputs)
        return {"value": value.detach(), "v": grads[0], "q": grads[1], "e": grads[2], "b": grads[3]}
    out = {}
    if state.stages:
        sim.solve()
        for s in range(2):
            sim.move(s)
        sim.advance_fields()
        for s in range(2):
            sim.sort(s)
        sim.deposit()
        sim.assemble()
    else:
        sim.cycle(1)
    if state.scalars:
        out["scalars"] = sim.scalars()
    out["etheta"] = state.field(R.FIELD_ETHETA)
    out["e"], out["b"], out["j"] = (state.field(f) for f in (R.FIELD_E, R.FIELD_B, R.FIELD_J))
    out["particles"] = [state.particles(s) for s in range(2)]
    return out


def work(case):
    """Per cycle: 312 B a particle (mover 112, sort copy 144, deposition 56) and 648 flop (27 moments x 12 columns,
    2 each); per node the matrix and current written and B read (1056 B, 552 B with a matrix in 32 bits), and eight
    solver steps that read the matrix and their vectors. A reported scalar sample reads 60 B a particle. A gradient
    repeats each forward cycle (run, replayed, solved again) and walks it backwards once (two passes over 68 B of
    particle and 112 B of adjoint each, a solve)."""
    nx, ny, nz = _cells(case)
    particles, nodes = 2 * nx * ny * nz * _per_cell(case), (nx + 1) * (ny + 1) * (nz + 1)
    matrix = 1008 if case["mass"] == "fp64" else 504
    steps = 8
    solve = steps * nodes * (matrix + 96 + 24 * (steps + 5))
    cycle = 312 * particles + (matrix + 48) * nodes + solve
    flops = 648 * particles + steps * nodes * 486
    if case["call"] == "gradient":
        back = 2 * (68 + 112) * particles + 2 * solve
        return {"bytes": case["cycles"] * (2 * cycle + back), "flops": 2 * case["cycles"] * flops}
    return {"bytes": cycle + (60 * particles if case["scalars"] else 0), "flops": flops}


# ---- the same pass in plain torch, 64 bits ---------------------------------

CORNERS = [(a & 1, (a >> 1) & 1, (a >> 2) & 1) for a in range(8)]


def _shift(v, d, sign):
    """v at (i + sign d0, j + sign d1, k + sign d2), periodic, of a [..., nz, ny, nx] array."""
    return torch.roll(v, shifts=(-sign * d[2], -sign * d[1], -sign * d[0]), dims=(-3, -2, -1))


def _curl(v, h, sign):
    """Curl with four-edge differences: nodes to cells (sign 1) or cells to nodes (sign -1)."""
    at = [_shift(v, d, sign) for d in CORNERS]

    def d(c, axis):
        total = 0.0
        for a, corner in enumerate(CORNERS):
            total = total + (at[a][c] if corner[axis] else -at[a][c])
        return sign * 0.25 / h * total

    return torch.stack((d(2, 1) - d(1, 2), d(0, 2) - d(2, 0), d(1, 0) - d(0, 1)))


def _to_nodes(b):
    return sum(_shift(b, d, -1) for d in CORNERS) / 8.0


def _corner_values(v):
    """[8, 3, cells] of a node vector."""
    return torch.stack([_shift(v, d, 1).reshape(3, -1) for d in CORNERS])


def _weights(r):
    return torch.stack([(r[0] if x else 1 - r[0]) * (r[1] if y else 1 - r[1]) * (r[2] if z else 1 - r[2])
                        for x, y, z in CORNERS])


def _alpha(o):
    """Response rows of omega [3, n]."""
    x, y, z = o
    inv = 1.0 / (1.0 + x * x + y * y + z * z)
    return [[(1 + x * x) * inv, (x * y + z) * inv, (x * z - y) * inv],
            [(x * y - z) * inv, (1 + y * y) * inv, (y * z + x) * inv],
            [(x * z + y) * inv, (y * z - x) * inv, (1 + z * z) * inv]]


CHUNK = 1 << 21


def _deposit(case, parts, bn, moments):
    """Moments [cells, 27, 12] (the last three columns the current) of every species' particles, any order. Without
    `moments` the corner currents [cells, 8, 3] alone."""
    p, ncells = PLASMAS[case["plasma"]], case["nx"] * case["ny"] * case["nz"]
    volume, corners = p["spacing"] ** 3, _corner_values(bn)
    shape = (ncells * 27, 12) if moments else (ncells * 8, 3)
    total = torch.zeros(shape, dtype=torch.float64, device="cuda")
    for s, q_over_m in enumerate(p["q_over_m"]):
        beta = q_over_m * p["dt"] / 2
        n = parts[s]["cell"].numel()
        for at in range(0, n, CHUNK):
            pick = slice(at, min(n, at + CHUNK))
            cell = parts[s]["cell"][pick]
            r = [parts[s][k][pick] for k in ("rx", "ry", "rz")]
            v = [parts[s][k][pick] for k in ("u", "v", "w")]
            q, w = parts[s]["q"][pick], _weights(r)
            b = sum(w[a] * corners[a][:, cell] for a in range(8))
            al = _alpha(beta * b)
            t = [q / volume * (al[c][0] * v[0] + al[c][1] * v[1] + al[c][2] * v[2]) for c in range(3)]
            if moments:
                t = [beta * q * al[i][j] for i in range(3) for j in range(3)] + t
                powers = [((1 - x) * (1 - x), x * (1 - x), x * x) for x in r]
            t = torch.stack(t, 1)
            for m in range(27 if moments else 8):
                f = powers[0][m % 3] * powers[1][m // 3 % 3] * powers[2][m // 9] if moments else w[m]
                total.index_add_(0, cell * (27 if moments else 8) + m, t * f[:, None])
    return total.reshape(ncells, -1, shape[1])


def _sum_corners(case, values):
    """Node vector of [cells, 8, 3] corner values."""
    nx, ny, nz = _cells(case)
    out = 0.0
    for a, d in enumerate(CORNERS):
        out = out + _shift(values[:, a].T.reshape(3, nz, ny, nx), d, -1)
    return out


def _moment(a, b):
    return sum((CORNERS[a][x] + CORNERS[b][x]) * 3 ** x for x in range(3))


def _mass_times(case, k, v):
    """M v from the cells' moments k [27][cells, 3, 3]."""
    at = _corner_values(v).permute(0, 2, 1).contiguous()
    out = torch.zeros((at.shape[1], 8, 3), dtype=torch.float64, device="cuda")
    for a in range(8):
        for b in range(8):
            out[:, a] += (k[_moment(a, b)] * at[b][:, None, :]).sum(2)
    return _sum_corners(case, out)


def _gmres(apply, b, x, steps=60):
    """Modified Gram-Schmidt GMRES run to rounding."""
    for _ in range(2):
        r = b - apply(x)
        norm = float(r.norm())
        basis, h, columns = [r / norm], np.zeros((steps + 1, steps)), 0
        for j in range(steps):
            w = apply(basis[j])
            for i in range(j + 1):
                h[i, j] = float((basis[i] * w).sum())
                w = w - h[i, j] * basis[i]
            h[j + 1, j] = float(w.norm())
            columns = j + 1
            rhs = np.zeros(j + 2)
            rhs[0] = norm
            y, *_ = np.linalg.lstsq(h[:j + 2, :j + 1], rhs, rcond=None)
            if np.linalg.norm(h[:j + 2, :j + 1] @ y - rhs) < 1e-15 * float(b.norm()):
                break
            basis.append(w / h[j + 1, j])
        for i in range(columns):
            x = x + float(y[i]) * basis[i]
    return x


def exact(case, seed):
    if (case["call"] == "gradient" or case["faces"] != "periodic" or case["smoothing"] != "none"
            or 2 * _per_cell(case) * case["nx"] * case["ny"] * case["nz"] > 60_000_000):
        return None
    p, (nx, ny, nz) = PLASMAS[case["plasma"]], _cells(case)
    h, dt = p["spacing"], p["dt"]
    delta, kappa = THETA * dt, FOUR_PI * THETA * dt
    e, b = _fields(case, seed)
    e = e.reshape(3, nz + 1, ny + 1, nx + 1)[:, :nz, :ny, :nx].contiguous()
    b = b.reshape(3, nz, ny, nx)
    parts = []
    for s in range(2):
        got = dict(_particles(case, s, seed))
        key = got["cell"].long()
        i, j, k = key % (nx + 4) - 2, key // (nx + 4) % (ny + 4) - 2, key // ((nx + 4) * (ny + 4)) - 2
        got["cell"] = i + nx * (j + ny * k)
        parts.append(got)
    bn = _to_nodes(b)
    moments = _deposit(case, parts, bn, True)
    corners = torch.stack([sum(moments[:, _moment(a, c), 9:] for c in range(8)) for a in range(8)], 1)
    j = _sum_corners(case, corners)
    tensor = [moments[:, m, :9].reshape(-1, 3, 3).contiguous() for m in range(27)]
    del moments, corners

    def apply(x):
        return x + delta * delta * _curl(_curl(x, h, 1), h, -1) + kappa / h ** 3 * _mass_times(case, tensor, x)

    etheta = _gmres(apply, e + delta * _curl(b, h, -1) - kappa * j, e)
    del tensor
    at_b, at_e = _corner_values(bn), _corner_values(etheta)
    extent = torch.tensor([nx, ny, nz], device="cuda")
    for s, q_over_m in enumerate(p["q_over_m"]):
        beta, got = q_over_m * dt / 2, parts[s]
        n = got["cell"].numel()
        for at in range(0, n, CHUNK):
            pick = slice(at, min(n, at + CHUNK))
            cell = got["cell"][pick]
            r, v = [torch.stack([got[k][pick] for k in names]) for names in (("rx", "ry", "rz"), ("u", "v", "w"))]
            w = _weights(r)
            bp, ep = (sum(w[a] * f[a][:, cell] for a in range(8)) for f in (at_b, at_e))
            al = _alpha(beta * bp)
            x = v + beta * ep
            v = torch.stack([2.0 * (al[c][0] * x[0] + al[c][1] * x[1] + al[c][2] * x[2]) - v[c] for c in range(3)])
            moved = r + dt / h * v
            shift = torch.floor(moved)
            r = moved - shift
            ijk = torch.stack((cell % nx, cell // nx % ny, cell // (nx * ny))) + shift.long()
            ijk = torch.remainder(ijk, extent[:, None])
            for c in range(3):
                got[("rx", "ry", "rz")[c]][pick], got[("u", "v", "w")[c]][pick] = r[c], v[c]
            got["cell"][pick] = ijk[0] + nx * (ijk[1] + ny * ijk[2])
        order = torch.argsort(got["cell"], stable=True)
        parts[s] = {k: x[order] for k, x in got.items()}
    e_next = (etheta - (1.0 - THETA) * e) / THETA
    b_next = b - dt * _curl(etheta, h, 1)
    j = _sum_corners(case, _deposit(case, parts, _to_nodes(b_next), False))
    out = {"etheta": _pad(etheta), "e": _pad(e_next), "b": b_next, "j": _pad(j)}
    out = {k: x.reshape(-1).contiguous() for k, x in out.items()}
    if case["scalars"]:
        volume = h ** 3
        rows = [float((e_next * e_next).sum()) * volume / (2 * FOUR_PI),
                float((b_next * b_next).sum()) * volume / (2 * FOUR_PI)]
        for q_over_m, got in zip(p["q_over_m"], parts):
            m = got["q"] / q_over_m
            rows += [float((m * (got["u"] ** 2 + got["v"] ** 2 + got["w"] ** 2)).sum()) / 2, float(got["q"].sum())]
            rows += [float((m * got[k]).sum()) for k in ("u", "v", "w")]
        out["scalars"] = np.array(rows)
    # The mixed forms push with a field that differs by their operands' rounding: a particle may then end in the next
    # cell, and the sorted order with it, so only the fields have a value that can be compared place by place.
    same = case["mass"] == "fp64"
    out["particles"] = [{k: got[k] if same and k not in ("cell", "id") else None for k in ATTRIBUTES} for got in parts]
    return out
