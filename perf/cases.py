"""The work that users of this package have it do, as cases that can be timed and compared.

A case is a dict of plain values: `path` says which public calls one pass makes, the rest are sizes
and options.  The listed cases span the package's range from the reference's smallest call (the stars'
field at the 512 cells of one leaf block) to whole bridge directions between 10,000 stars and about a
million AMR cells; sizes follow the c1, c2 and c4 workloads of torch_amd.workloads and the tests.
Inputs are those workloads' (Plummer / Kroupa clusters with hard binaries, AMR leaf blocks of a
lognormal field), made from the seed and resident on the GPU, in pc, Msun and km/s.  Calls use the
package's defaults: input validation on, the committed tune cache.

    block_call   StellarGravityField.get_gravity_at_point at one leaf block's cell centres: the
                 reference's bridge makes one such call per leaf block, with the stars set once.
    bridge       a whole small bridge step (c1): both source sets loaded, the stars' field on the cells
                 and the gas field on the stars, on explicit arrays.
    points       the stars' acceleration and potential at scattered points in no block order (other
                 stars, tracers), star set loaded in the same pass.
    forward      stars -> AMR cells: leaf blocks with the gas kick fused, or explicit cell centres.
    potential    get_potential_at_point of the stars at the cells (explicit centres).
    reverse      AMR cells -> stars: the blocks (or explicit cells) loaded, then the stars' acceleration.
    plan         uneven independent problems in one batch plan replayed from its graph.
    fused        the two-way pass over all (cell, star) pairs.
    flash        FLASH's spline or linear softening, cells as leaf blocks -> stars, isolated boundaries.
    periodic     the same kernels with the periodic image sum, explicit cells -> stars.
    mesh         the particle-mesh pieces: mass deposit, grid kick from the potential, and the
                 particles' long-range force.
"""
import math

import numpy as np
import torch

from torch_amd import GasGravityField, GravityField, LeafBlocks, ParticleMesh, StellarGravityField
from torch_amd import workloads as W
from torch_amd.batch import BatchPlan
from torch_amd.blocks import block_centres

G = W.G_PC_MSUN_KMS
DT = 0.01                 # kick interval, pc / (km/s)
RSOFT = 0.078125          # FLASH's global softening radius: 2.5 cells of the finest c2 level
BOX = 4.0


def listed():
    return [
        # one leaf block of the reference's per-block bridge loop; thousands of these in a row
        dict(name="block_call_fp64", path="block_call", mode="fp64", stars=1024, blocks=1),
        # c1, the smallest configuration, both directions
        dict(name="bridge_c1_mixed", path="bridge", mode="mixed", stars=1024, grid=16),
        # unsoftened cluster members onto scattered points; no count is a multiple of a tile
        dict(name="points_fp64", path="points", mode="fp64", stars=5003, points=20011, eps="none"),
        # c2's forward direction with the gas kick
        dict(name="forward_blocks_mixed", path="forward", mode="mixed", stars=10000, blocks=2000, form="blocks"),
        # half of c2 as the reference hands it over: explicit cell centres
        dict(name="forward_centres_fp64", path="forward", mode="fp64", stars=10000, blocks=1000, form="centres"),
        # c2's reverse direction
        dict(name="reverse_blocks_mixed", path="reverse", mode="mixed", stars=10000, blocks=2000, form="blocks"),
        # the stars' potential on the cells, a legacy function of its own
        dict(name="potential_fp64", path="potential", mode="fp64", stars=10000, blocks=1000),
        # a quarter of c4's problem count at its sizes
        dict(name="plan_mixed", path="plan", mode="mixed", problems=16, max_stars=50000, max_points=1000000, sizes=4),
        # c2's fused pass on half of its blocks
        dict(name="fused_mixed", path="fused", mode="mixed", stars=10000, blocks=1000),
        # gas onto stars with FLASH's own kernel and the reference's potential
        dict(name="flash_spline", path="flash", stars=10000, blocks=1000, kernel="spline", quirks=True),
        # c1 reverse in a periodic box
        dict(name="periodic_c1", path="periodic", stars=1024, grid=16, nrep=6, quirks=True),
        # c2's leaf blocks with 4 guard layers and its stars
        dict(name="mesh_c2", path="mesh", stars=10000, blocks=2000, guard=4),
    ]


PAIRS = 1.0e10            # no drawn case has more pairs than half of c2's forward direction and back


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    path = rng.choice(["block_call", "bridge", "points", "forward", "potential", "reverse", "plan", "fused",
                       "flash", "periodic", "mesh"])
    mode = rng.choice(["fp64", "mixed"])
    stars = _log_int(rng, 100, 20000)
    if path == "block_call":
        return dict(path=path, mode=mode, stars=_log_int(rng, 100, 10000), blocks=rng.randint(1, 8))
    if path == "bridge":
        return dict(path=path, mode=mode, stars=_log_int(rng, 100, 4000), grid=rng.randint(6, 24))
    if path == "points":
        return dict(path=path, mode=mode, stars=stars, points=_log_int(rng, 1, 100000),
                    eps=rng.choice(["none", "source", "point"]))
    if path in ("forward", "potential", "reverse", "fused"):
        most = PAIRS / 512 / stars / (2.2 if mode == "fp64" else 1.0)
        case = dict(path=path, mode=mode, stars=stars, blocks=_log_int(rng, 8, max(9, min(2000, int(most)))))
        if path in ("forward", "reverse"):
            case["form"] = rng.choice(["blocks", "centres"])
        return case
    if path == "plan":
        return dict(path=path, mode=mode, problems=rng.randint(2, 16), max_stars=_log_int(rng, 1000, 20000),
                    max_points=_log_int(rng, 4000, 300000), sizes=rng.randint(0, 10 ** 6))
    if path == "flash":
        return dict(path=path, stars=stars, blocks=_log_int(rng, 8, max(9, min(2000, int(PAIRS / 1100 / stars)))),
                    kernel=rng.choice(["spline", "linear"]), quirks=rng.random() < 0.5)
    if path == "periodic":
        return dict(path=path, stars=_log_int(rng, 20, 1024), grid=rng.randint(4, 16), nrep=rng.randint(2, 6),
                    quirks=rng.random() < 0.5)
    return dict(path=path, stars=stars, blocks=_log_int(rng, 8, 2000), guard=rng.randint(1, 4))


# ------------------------------------------------------------------------ inputs ----
def _dev(a):
    return torch.as_tensor(np.ascontiguousarray(a), device="cuda")


def _stars(rng, n, binary=0.2, eps=0.01):
    s = W.star_cluster(rng, n, r_vir=1.0, binary_frac=binary, eps=eps)
    return {k: _dev(s[k]) for k in ("x", "y", "z", "m", "eps")}, s


def _gas(rng, n):
    """n leaf blocks of 8^3 cells covering (or, below 512 of them, taken from) a 4 pc box."""
    base = 8 if n >= 512 else 4 if n >= 64 else 2
    c = W.gas_cells(rng, BOX, base, n, 1.5, 64, 100.0, min_size=0.0625)
    return c, dict(origin=_dev(c["block_origin"]), dx=_dev(c["block_size"] / 8), x=_dev(c["x"]), y=_dev(c["y"]),
                   z=_dev(c["z"]), m=_dev(c["m"]), rho=_dev(c["rho"]), dx_cell=_dev(c["dx"]))


def _grid(rng, n):
    """A uniform n^3 grid of gas cells over the 4 pc box (c1's cells)."""
    x, y, z, dx = W.uniform_grid(n, BOX)
    rho = W.lognormal_field(rng, n, 1.5).ravel() * 100.0
    d = np.full(x.size, dx)
    return dict(x=_dev(x), y=_dev(y), z=_dev(z), dx=_dev(d), rho=_dev(rho), m=_dev(rho * dx ** 3))


def _plan_sizes(case):
    """[(sources, leaf blocks)] of a plan's problems, log-uniform as c4 draws them."""
    rng = W.rng_for(case["sizes"])
    return [(int(10.0 ** rng.uniform(2.0, math.log10(case["max_stars"]))),
             int(math.ceil(10.0 ** rng.uniform(3.0, math.log10(case["max_points"])) / 512)))
            for _ in range(case["problems"])]


def _plan_problems(rng, case):
    """Uneven problems as c4's: cluster stars or gas cells as sources, leaf blocks as targets."""
    out = []
    for p, (ns, nblk) in enumerate(_plan_sizes(case)):
        if p % 2 == 0:
            s = W.star_cluster(rng, ns, r_vir=1.0)
            src = dict(x=s["x"], y=s["y"], z=s["z"], m=s["m"])
        else:
            sblk = -(-ns // 512)
            o = rng.uniform(-2.0, 1.5, (sblk, 3))
            size = 10.0 ** rng.uniform(np.log10(0.03125), np.log10(0.5), sblk)
            x, y, z, dx = block_centres(o, size / 8)
            rho = 100.0 * np.exp(1.5 * rng.normal(size=x.size) - 1.125)
            src = dict(x=x[:ns], y=y[:ns], z=z[:ns], m=(rho * dx ** 3)[:ns])
        src["eps"] = rng.uniform(0.005, 0.1, ns)
        o = rng.uniform(-2.0, 1.5, (nblk, 3))
        size = 10.0 ** rng.uniform(np.log10(0.03125), np.log10(0.5), nblk)
        out.append(dict(sources={k: _dev(v) for k, v in src.items()},
                        targets=dict(block_origin=_dev(o), block_dx=_dev(size / 8))))
    return out


def _inputs(case, seed):
    """The arrays of a case, on the GPU."""
    rng = W.rng_for(seed)
    path, I = case["path"], {}
    if path == "plan":
        I["problems"] = _plan_problems(rng, case)
        return I
    eps = case.get("eps", "source")
    I["s"], host = _stars(rng, case["stars"])
    if eps == "none":
        I["s"]["eps"] = None
    if path == "block_call":
        o = rng.uniform(-1.0, 0.75, (case["blocks"], 3))
        x, y, z, _ = block_centres(o, np.full(case["blocks"], 0.03125))
        I["t"] = dict(x=_dev(x), y=_dev(y), z=_dev(z))
    elif path in ("bridge", "periodic"):
        I["g"] = _grid(rng, case["grid"])
        if path == "periodic":       # positions wrapped into the box
            for k in "xyz":
                I["s"][k] = torch.remainder(I["s"][k] + BOX / 2, BOX) - BOX / 2
    elif path == "points":
        n = case["points"]
        t, _ = _stars(rng, max(n, 2), binary=0.0)
        I["t"] = {k: t[k][:n].contiguous() for k in "xyz"}
        I["t"]["eps"] = _dev(rng.uniform(0.005, 0.05, n)) if eps == "point" else None
    else:
        c, I["g"] = _gas(rng, case["blocks"])
        if path == "forward" and case["form"] == "blocks":
            I["v"] = [_dev(rng.normal(0.0, 3.0, case["blocks"] * 512)) for _ in range(3)]
        if path == "mesh":
            blk = W.containing_block(host["x"], host["y"], host["z"], c["block_origin"], c["block_size"])
            out = np.flatnonzero(blk < 0)          # stars outside the mesh go to random places in it
            blk[out] = rng.integers(0, case["blocks"], out.size)
            at = c["block_origin"][blk[out]] + c["block_size"][blk[out], None] * rng.uniform(0, 1, (out.size, 3))
            for a, k in enumerate("xyz"):
                host[k][out] = at[:, a]
            I["p"] = {k: _dev(host[k]) for k in ("x", "y", "z", "m")}
            I["p"]["blk"] = _dev(blk)
            I["B"] = LeafBlocks(_dev(c["block_origin"]), _dev(c["block_size"]), nb=8, ng=case["guard"])
            B = I["B"]
            h = B.size / B.nb
            idx = torch.arange(B.nbg, dtype=torch.float64, device="cuda") - B.ng + 0.5
            r2 = 0.36
            for a in range(3):           # x is the fastest axis of a block
                shape = [1, 1, 1, 1]
                shape[3 - a] = B.nbg
                q = B.origin[:, a].reshape(-1, 1, 1, 1) + h.reshape(-1, 1, 1, 1) * idx.reshape(shape)
                r2 = r2 + q * q
            I["phi"] = (-500.0 / torch.sqrt(r2)).reshape(-1).contiguous()
            gen = torch.Generator(device="cuda").manual_seed(int(seed))
            I["v"] = [3.0 * torch.randn(B.ncell, dtype=torch.float64, device="cuda", generator=gen)
                      for _ in range(3)]
    return I


def prepare(case, seed):
    S = dict(_inputs(case, seed), case=case)
    path, mode = case["path"], case.get("mode", "fp64")
    if path == "block_call":
        S["f"] = StellarGravityField(mode)
        S["f"].set_stars(*(S["s"][k] for k in ("x", "y", "z", "m", "eps")))
    elif path == "bridge":
        S["f"], S["h"] = StellarGravityField(mode), GasGravityField(mode)
    elif path in ("points", "forward", "potential"):
        S["f"] = StellarGravityField(mode)
    elif path == "reverse":
        S["f"] = GasGravityField(mode)
    elif path == "plan":
        S["f"] = GravityField(mode)
        S["plan"] = BatchPlan(S["f"], S["problems"])
    elif path == "fused":
        S["f"] = GravityField(mode)
    elif path in ("flash", "periodic"):
        S["f"] = GasGravityField("fp64")
        S["f"].set_softening(case.get("kernel", "spline"), RSOFT, quirks=case["quirks"])
        if path == "periodic":
            S["f"].set_periodic((BOX, BOX, BOX), nrep=case["nrep"])
    else:
        S["f"] = ParticleMesh()
    return S


# ---------------------------------------------------------------------- one pass ----
def run(S):
    case, f = S["case"], S["f"]
    path = case["path"]
    if path == "plan":
        return [list(o) for o in S["plan"].run()]
    s, g = S["s"], S.get("g")
    stars = [s[k] for k in ("x", "y", "z", "m", "eps")]
    at_stars = [s[k] for k in "xyz"]
    if path == "block_call":
        t = S["t"]
        return f.get_gravity_at_point(0.0, t["x"], t["y"], t["z"])
    if path == "bridge":
        f.set_stars(*stars)
        on_gas = f.evaluate(0.0, g["x"], g["y"], g["z"])
        S["h"].set_cells(g["x"], g["y"], g["z"], g["rho"], g["dx"])
        return on_gas, S["h"].get_accel_gas_on_particles(0.0, *at_stars)
    if path == "points":
        t = S["t"]
        f.set_stars(*stars)
        return f.evaluate(t["eps"], t["x"], t["y"], t["z"])
    if path == "forward":
        f.set_stars(*stars)
        if case["form"] == "blocks":
            return f.evaluate_blocks(g["origin"], g["dx"], dt=DT, vel=S["v"]), S["v"]
        return f.get_gravity_at_point(0.0, g["x"], g["y"], g["z"])
    if path == "potential":
        f.set_stars(*stars)
        return f.get_potential_at_point(0.0, g["x"], g["y"], g["z"])
    if path == "reverse":
        if case["form"] == "blocks":
            f.set_blocks(g["origin"], g["dx"], g["m"])
        else:
            f.set_cells(g["x"], g["y"], g["z"], g["rho"], g["dx_cell"])
        return f.get_accel_gas_on_particles(0.0, *at_stars)
    if path == "fused":
        return f.bidirectional_blocks(g["origin"], g["dx"], g["m"], g["dx"], *stars)
    if path == "flash":
        f.set_blocks(g["origin"], g["dx"], g["m"])
        return f.evaluate(0.0, *at_stars)
    if path == "periodic":
        f.set_cells(g["x"], g["y"], g["z"], g["rho"], g["dx"])
        return f.evaluate(0.0, *at_stars)
    p, B = S["p"], S["B"]
    rho = f.update_grid_var(p["x"], p["y"], p["z"], p["m"], p["blk"], B)
    f.accel_list_of_blocks(S["phi"], B, dt=DT, vel=S["v"], store=False)
    acc = f.long_range_force(p["x"], p["y"], p["z"], p["blk"], B, S["phi"])
    return rho, S["v"], acc


# ------------------------------------------------------------------- what it needs ----
def work(case):
    """Bytes: every input read and every output written once (FP64).  Flop per pair: 21 for acceleration
    and potential, 19 for the acceleration, 12 for the potential alone, 34 both ways."""
    path = case["path"]
    ns, nc = case.get("stars", 0), 512 * case.get("blocks", 0)
    if path == "plan":
        sizes = _plan_sizes(case)
        return {"bytes": sum(40.0 * n + 32.0 * 512 * b for n, b in sizes),
                "flops": sum(21.0 * n * 512 * b for n, b in sizes)}
    if path in ("bridge", "periodic"):
        nc = case["grid"] ** 3
    if path == "block_call":
        return {"bytes": 40.0 * ns + 48.0 * nc, "flops": 19.0 * ns * nc}
    if path == "bridge":
        return {"bytes": 2 * (40.0 * ns + 40.0 * nc) + 32.0 * nc + 24.0 * ns, "flops": 40.0 * ns * nc}
    if path == "points":
        return {"bytes": 40.0 * ns + 56.0 * case["points"], "flops": 21.0 * ns * case["points"]}
    if path == "forward":
        out = 32 + 48 if case["form"] == "blocks" else 24 + 24
        return {"bytes": 40.0 * ns + float(out) * nc, "flops": (21.0 if case["form"] == "blocks" else 19.0) * ns * nc}
    if path == "potential":
        return {"bytes": 40.0 * ns + 32.0 * nc, "flops": 12.0 * ns * nc}
    if path == "reverse":
        return {"bytes": (8.0 if case["form"] == "blocks" else 40.0) * nc + 48.0 * ns, "flops": 19.0 * ns * nc}
    if path == "fused":
        return {"bytes": 40.0 * nc + 72.0 * ns, "flops": 34.0 * ns * nc}
    if path == "flash":
        return {"bytes": 8.0 * nc + 56.0 * ns, "flops": 21.0 * ns * nc}
    if path == "periodic":          # images inside the cutoff sphere of nrep boxes around the star
        return {"bytes": 40.0 * nc + 56.0 * ns, "flops": 21.0 * ns * nc * 4.18879 * case["nrep"] ** 3}
    cells = case["blocks"] * float((8 + 2 * case["guard"]) ** 3)
    # rho out; phi in, velocities in and out; per particle its record twice and 32 potential values
    return {"bytes": cells * (8 + 8 + 48) + ns * (40 + 32 + 256 + 24.0), "flops": cells * 15.0 + ns * 200.0}


# ---------------------------------------------------------------- 64-bit reference ----
def _pairs(t, s, te2, se2, m, acc=True, pot=True):
    """Softened sums over all pairs in 64 bits: (ax, ay, az, phi) at the points t[3] from sources s[3]."""
    n, ns = t[0].numel(), s[0].numel()
    out = [torch.zeros(n, dtype=torch.float64, device="cuda") for _ in range(4)]
    step = max(1, (1 << 25) // ns)
    for a in range(0, n, step):
        b = min(n, a + step)
        d = [s[q][None, :] - t[q][a:b, None] for q in range(3)]
        r2 = d[0] * d[0] + d[1] * d[1] + d[2] * d[2]
        if se2 is not None:
            r2 += se2[None, :]
        if te2 is not None:
            r2 += te2[a:b, None]
        y = torch.where(r2 > 0, 1.0 / torch.sqrt(r2), 0.0)   # a coincident pair contributes nothing
        mr = m[None, :] * y
        if pot:
            out[3][a:b] = -G * mr.sum(1)
        if acc:
            w = mr * y * y
            for q in range(3):
                out[q][a:b] = G * (w * d[q]).sum(1)
    return out


def _flash_kernels(r2, kernel, quirks):
    """FLASH's force and potential kernels at separation^2 r2."""
    r = torch.sqrt(r2)
    soft = r < RSOFT
    kv, pk = 1.0 / (r2 * r), 1.0 / r
    if not bool(soft.any()):
        return kv, pk
    rs, h = r[soft], 2.0 / RSOFT
    if kernel == "spline":
        q = rs * h
        k1 = torch.where(q > 1e-5, h * h * (4 / 3 * q - 1.2 * q ** 3 + 0.5 * q ** 4) / rs,
                         h ** 3 * (4 / 3 - 1.2 * q ** 2 + 0.5 * q ** 3))
        k2 = h * h * (8 / 3 * q - 3 * q ** 2 + 1.2 * q ** 3 - q ** 4 / 6 - 1 / (15 * q ** 2)) / rs
        p1 = h * (2 / 3 * q ** 2 - (0.1 if quirks else 0.3) * q ** 4 + 0.1 * q ** 5 - 1.4)
        p2 = h * (4 / 3 * q ** 2 - q ** 3 + 0.3 * q ** 4 - q ** 5 / 30 - 1.6 + 1 / (15 * q))
        sign = 1.0 if quirks else -1.0
        kv[soft], pk[soft] = torch.where(q < 1, k1, k2), sign * torch.where(q < 1, p1, p2)
    else:
        slope = 1.0 / RSOFT ** 3
        kv[soft] = slope
        pk[soft] = slope if quirks else (3.0 * RSOFT ** 2 - rs * rs) * (0.5 * slope)
    return kv, pk


def _flash(t, s, m, kernel, quirks, nrep=0):
    n, ns = t[0].numel(), s[0].numel()
    out = [torch.zeros(n, dtype=torch.float64, device="cuda") for _ in range(4)]
    shifts = np.arange(-nrep, nrep + 1)
    step = max(1, (1 << 23) // ns)
    for a in range(0, n, step):
        b = min(n, a + step)
        d = [t[q][a:b, None] - s[q][None, :] for q in range(3)]
        A = [torch.zeros_like(d[0]) for _ in range(4)]
        for nx in shifts:
            for ny in shifts:
                for nz in shifts:
                    if nrep and math.dist((abs(nx), abs(ny), abs(nz)), (0, 0, 0)) > nrep + 1.75:
                        continue
                    e = [d[0] + nx * BOX, d[1] + ny * BOX, d[2] + nz * BOX] if nrep else d
                    r2 = (e[0] * e[0] + e[1] * e[1]) + e[2] * e[2]
                    kv, pk = _flash_kernels(r2, kernel, quirks)
                    if nrep:
                        inside = torch.sqrt(r2) < nrep * BOX
                        kv = torch.where(inside, kv, 0.0)
                        A[3] = torch.where(inside, pk, A[3] if quirks else 0.0) + (0.0 if quirks else A[3])
                    else:
                        A[3] = pk
                    for q in range(3):
                        A[q] += kv * e[q]
        for q in range(3):
            out[q][a:b] = -G * (m[None, :] * A[q]).sum(1)
        out[3][a:b] = -G * (m[None, :] * A[3]).sum(1)
    return out


def _mesh(I):
    """(deposited density, kicked velocities, particle accelerations) of the mesh path."""
    p, B = I["p"], I["B"]
    n, dl = B.nbg, B.size / B.nb
    u = [(p[k] - B.origin[:, a][p["blk"]]) / dl[p["blk"]] - 0.5 + B.ng for a, k in enumerate("xyz")]
    i0 = [torch.floor(q) for q in u]
    w = [(1.0 - (q - i), q - i) for q, i in zip(u, i0)]
    corners = []
    for dk in (0, 1):
        for dj in (0, 1):
            for di in (0, 1):
                cell = ((p["blk"] * n + i0[2].long() + dk) * n + i0[1].long() + dj) * n + i0[0].long() + di
                corners.append((cell, (w[0][di] * w[1][dj]) * w[2][dk]))
    md = p["m"] / dl[p["blk"]] ** 3
    rho = torch.zeros(B.ncell, dtype=torch.float64, device="cuda")
    for cell, wt in corners:
        rho.index_add_(0, cell, md * wt)
    phi = I["phi"].reshape(-1, n, n, n)
    g = []
    for axis in (3, 2, 1):               # x, y, z; the two end cells of a row copy their neighbour
        i = torch.arange(n, device="cuda").clamp(1, n - 2)
        diff = phi.index_select(axis, i - 1) - phi.index_select(axis, i + 1)
        g.append(((0.5 * B.nb / B.size).reshape(-1, 1, 1, 1) * diff).reshape(-1))
    vel = [v + DT * a for v, a in zip(I["v"], g)]
    return rho, vel, [sum(wt * a[cell] for cell, wt in corners) for a in g]


def exact(case, seed):
    I = _inputs(case, seed)
    path = case["path"]
    if path == "plan":
        out = []
        for p in I["problems"]:
            s, t = p["sources"], p["targets"]
            x, y, z, _ = block_centres(t["block_origin"].cpu().numpy(), t["block_dx"].cpu().numpy())
            out.append(_pairs([_dev(q) for q in (x, y, z)], [s[k] for k in "xyz"], None, s["eps"] ** 2, s["m"]))
        return out
    s, g = I["s"], I.get("g")
    at_s = [s[k] for k in "xyz"]
    se2 = None if s["eps"] is None else s["eps"] ** 2
    if path == "mesh":
        return _mesh(I)
    at_g = [g[k] for k in "xyz"] if g else None
    if path == "periodic":
        return _flash(at_s, at_g, g["m"], "spline", case["quirks"], case["nrep"])
    if path == "flash":
        return _flash(at_s, at_g, g["m"], case["kernel"], case["quirks"])
    if path == "block_call":
        return _pairs([I["t"][k] for k in "xyz"], at_s, None, se2, s["m"], pot=False)[:3]
    if path == "points":
        t = I["t"]
        return _pairs([t[k] for k in "xyz"], at_s, None if t["eps"] is None else t["eps"] ** 2, se2, s["m"])
    if path == "bridge":
        return (_pairs(at_g, at_s, None, se2, s["m"]),
                _pairs(at_s, at_g, None, g["dx"] ** 2, g["m"], pot=False)[:3])
    if path == "forward" and case["form"] == "blocks":
        a = _pairs(at_g, at_s, None, se2, s["m"])
        return a, [v + DT * q for v, q in zip(I["v"], a)]
    if path == "forward":
        return _pairs(at_g, at_s, None, se2, s["m"], pot=False)[:3]
    if path == "potential":
        return _pairs(at_g, at_s, None, se2, s["m"], acc=False)[3]
    if path == "reverse":
        return _pairs(at_s, at_g, None, g["dx_cell"] ** 2, g["m"], pot=False)[:3]
    a = _pairs(at_g, at_s, g["dx_cell"] ** 2, se2, s["m"])
    return a, _pairs(at_s, at_g, se2, g["dx_cell"] ** 2, g["m"])
