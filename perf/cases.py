"""Performance cases of the Z4c evolution path, through the public Python surface.

A case is what one call (or one output event) of a numerical-relativity run
does on one GPU: right-hand sides, whole bt_rk4 steps with each kind of ghost
handling, the constraint output, and the adjoints.  Sizes follow the
repository's configurations (one 32^3 block; the 64^3 gauge wave; 2048 uneven
blocks; 2:1-balanced trees of 16^3 blocks; 64 cotangents of one 32^3 block)
and spread from one 8^3 block to those, with ragged and odd blocks between.

``exact`` evaluates the same right-hand side, step and constraints in float64
torch tensor algebra written here, differentiated by torch.autograd for the
adjoints.
"""
from __future__ import annotations

import functools
import math
import os
import sys

import numpy as np
import torch

_ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
sys.path.insert(0, os.path.join(_ROOT, "gr-athena_amd"))

from z4c_amd import Params  # noqa: E402
from z4c_amd.initial_data import balanced_octree_blocks  # noqa: E402
from z4c_amd.z4c import MeshBlockGeom, Z4c  # noqa: E402

NG = 4
DEV = "cuda"

# Counted arithmetic of one right-hand side and of the rest of one bt_rk4 step
# per interior vertex (the repository's counted totals for 16^3 .. 32^3 blocks),
# of one constraint evaluation, and the reverse sweep at twice the forward's.
FLOP_RHS = 7500.0
FLOP_STEP = 4.0 * FLOP_RHS + 1800.0
FLOP_CON = 3500.0


# --------------------------------------------------------------------- cases
def listed():
    return [
        # a unit-test sized evolution block: latency and launches are all there is
        dict(name="rhs_one_8", kind="rhs", nx="8", nblocks=1, data="bumps", faces=0, matter=0),
        # the single-block right-hand side of the parity configuration
        dict(name="rhs_one_32", kind="rhs", nx="32", nblocks=1, data="bumps", faces=0, matter=0),
        # an odd-sized, non-cubic batch with matter sources and Sommerfeld faces,
        # as a host code that integrates with its own driver calls it
        dict(name="rhs_ragged_matter", kind="rhs", nx="37x19x24,11x29x16,22x13x35,9x10x51",
             nblocks=90, data="punctures", faces=1, matter=1),
        # the periodic 64^3 gauge wave (convergence tests): one block, graph replay
        dict(name="step_wave_64", kind="step", ghosts="periodic", nx="64", nblocks=1,
             data="wave", graph=1, faces=0),
        # the same wave on a small odd grid, issued eagerly (parameter studies)
        dict(name="step_wave_21", kind="step", ghosts="periodic", nx="21x17x13", nblocks=1,
             data="wave", graph=0, faces=0),
        # puncture blocks of ragged sizes with Sommerfeld faces on some, eager
        dict(name="step_ragged_faces", kind="step", ghosts="frozen", nx="26x18x14,33x12x20,15x21x27",
             nblocks=60, data="punctures", graph=0, faces=1),
        # the headline batch: 2048 uneven blocks, graph replay
        dict(name="step_uneven_2048", kind="step", ghosts="frozen", nx="16*7,24*2,32*1",
             nblocks=2048, data="punctures", graph=1, faces=0),
        # a refined binary: balanced tree, ghost update across levels, outflow faces
        dict(name="step_tree_1000", kind="step", ghosts="tree", nx="16", nblocks=1000,
             data="punctures", graph=1, faces=0),
        # what a run does at its constraint output: Z4cToADM, ADMConstraints, history sums
        dict(name="constraints_400", kind="constraints", nx="16*7,24*2,32*1", nblocks=400,
             data="punctures"),
        # the adjoint of one right-hand side with 64 cotangents in one call
        dict(name="vjp_rhs_32_64", kind="vjp_rhs", nx="32", nblocks=1, nw=64, data="bumps"),
        # the adjoint of one step of a batch of 16^3 blocks, one cotangent
        dict(name="vjp_step_320", kind="vjp_step", ghosts="frozen", nx="16", nblocks=320, nw=1,
             data="punctures"),
        # the adjoint of one step of a refined tree through its ghost update
        dict(name="vjp_step_tree_200", kind="vjp_step", ghosts="tree", nx="16", nblocks=200, nw=1,
             data="punctures"),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _draw_sizes(rng, lo, hi):
    """One to four block sizes, cubic or ragged, each axis in [lo, hi]."""
    out = []
    for _ in range(rng.randint(1, 4)):
        if rng.random() < 0.4:
            out.append(str(_log_int(rng, lo, hi)))
        else:
            out.append("x".join(str(_log_int(rng, lo, hi)) for _ in range(3)))
    return ",".join(out)


def _cap_blocks(nx, nblocks, vertices):
    """nblocks lowered until the batch holds at most ``vertices`` vertices."""
    per = np.mean([np.prod([n + 1 + 2 * NG for n in s]) for s in _sizes(nx)])
    return int(max(1, min(nblocks, vertices / per)))


def draw(rng):
    kind = rng.choice(["rhs", "rhs", "step", "step", "step", "step", "constraints", "vjp_rhs",
                       "vjp_step"])
    if kind == "rhs":
        nx = _draw_sizes(rng, 8, 48)
        n = _cap_blocks(nx, _log_int(rng, 1, 400), 8e6)
        return dict(kind=kind, nx=nx, nblocks=n, data=rng.choice(["bumps", "punctures"]),
                    faces=rng.randint(0, 1), matter=rng.randint(0, 1))
    if kind == "step":
        ghosts = rng.choice(["periodic", "frozen", "frozen", "tree"])
        graph = rng.randint(0, 1)
        if ghosts == "periodic":
            return dict(kind=kind, ghosts=ghosts, nx=_draw_sizes(rng, 9, 64).split(",")[0],
                        nblocks=1, data="wave", graph=graph, faces=0)
        if ghosts == "tree":
            return dict(kind=kind, ghosts=ghosts, nx=str(rng.choice([8, 10, 12, 16, 20])),
                        nblocks=_log_int(rng, 64, 500), data="punctures", graph=graph, faces=0)
        nx = _draw_sizes(rng, 8, 36)
        n = _cap_blocks(nx, _log_int(rng, 2, 2048), 24e6)
        return dict(kind=kind, ghosts=ghosts, nx=nx, nblocks=n, data="punctures", graph=graph,
                    faces=0 if graph else rng.randint(0, 1))
    if kind == "constraints":
        nx = _draw_sizes(rng, 8, 36)
        return dict(kind=kind, nx=nx, nblocks=_cap_blocks(nx, _log_int(rng, 1, 400), 8e6),
                    data="punctures")
    if kind == "vjp_rhs":
        nx = _draw_sizes(rng, 8, 32)
        nw = _log_int(rng, 1, 64)
        return dict(kind=kind, nx=nx, nblocks=_cap_blocks(nx, _log_int(rng, 1, 64), 4e6 / nw), nw=nw,
                    data="bumps")
    if rng.random() < 0.5:
        return dict(kind=kind, ghosts="tree", nx=str(rng.choice([8, 12, 16])),
                    nblocks=_log_int(rng, 64, 160), nw=1, data="punctures")
    nx = _draw_sizes(rng, 8, 32)
    nw = rng.randint(1, 3)
    return dict(kind=kind, ghosts="frozen", nx=nx,
                nblocks=_cap_blocks(nx, _log_int(rng, 1, 400), 6e6 / nw), nw=nw, data="punctures")


def work(case):
    """Bytes and operations of one pass, counted on the vertices the blocks
    own or hold: state in and out (22 fields), the registers a classical RK4
    step cannot do without, the constraint fields, the cotangents."""
    blocks = _blocks(case)[0]
    padded = float(sum(g.npts for g in blocks))
    inner = float(sum((g.nx[0] + 1) * (g.nx[1] + 1) * (g.nx[2] + 1) for g in blocks))
    kind = case["kind"]
    field = 22 * 8.0
    if kind == "rhs":
        extra = 10 * 8.0 * inner if case["matter"] else 0.0
        return {"bytes": field * (padded + inner) + extra, "flops": FLOP_RHS * inner}
    if kind == "step":
        # each stage reads its state and writes the next; one running register
        return {"bytes": field * (2 * padded + 13 * inner), "flops": FLOP_STEP * inner}
    if kind == "constraints":
        # u in; ADM out and in; constraints out; history sums in
        return {"bytes": 8.0 * (22 * padded + 17 * padded + 7 * 2 * inner),
                "flops": FLOP_CON * inner}
    nw = case["nw"]
    if kind == "vjp_rhs":
        return {"bytes": field * (padded + nw * (inner + padded)),
                "flops": FLOP_RHS * inner * (1 + 2 * nw)}
    # forward sweep once, then the reverse sweep per cotangent
    return {"bytes": field * (padded * (1 + 2 * nw) + 13 * inner * (1 + nw)),
            "flops": FLOP_STEP * inner * (1 + 2 * nw)}


# -------------------------------------------------------------------- blocks
def _sizes(spec):
    """'16*7,24*2' -> [(16,16,16)]*7 + [(24,24,24)]*2; '9x10x51' is one block."""
    out = []
    for item in str(spec).split(","):
        dims, _, rep = item.partition("*")
        n = [int(v) for v in dims.split("x")]
        out += [tuple(n * 3 if len(n) == 1 else n)] * int(rep or 1)
    return out


@functools.lru_cache(maxsize=4)
def _tree(nblocks, cells):
    return balanced_octree_blocks(nblocks=nblocks, seed=0, cells=cells)


def _blocks(case):
    """Block list of a case and, for a tree, the corners of its box."""
    if case.get("ghosts") == "tree":
        return _tree(case["nblocks"], int(case["nx"]))
    sizes = _sizes(case["nx"])
    if case["data"] != "punctures":
        out = []
        for b in range(case["nblocks"]):
            n = sizes[b % len(sizes)]
            h = tuple(1.0 / v for v in n)
            out.append(MeshBlockGeom(n, h, (-0.5, -0.5, -0.5),
                                     sommerfeld_faces=21 if case.get("faces") else 0))
        return out, None, None
    # blocks scattered around the two punctures on levels 0..7, spacing 2^-level
    rng = np.random.default_rng(len(sizes) * 7919 + case["nblocks"])
    order = rng.permutation(case["nblocks"])
    out = []
    for b in range(case["nblocks"]):
        n = sizes[int(order[b]) % len(sizes)]
        level = int(rng.integers(0, 8))
        h = 0.5 ** level
        c = rng.normal(size=3) * 24.0 * h
        c[0] += 5.0 if rng.random() < 0.5 else -5.0
        faces = int(rng.integers(0, 64)) if case.get("faces") and b % 4 == 0 else 0
        if faces:       # an outer-boundary block
            c = c / np.linalg.norm(c) * 96.0
        lo = (np.floor(c / h) - np.array(n) // 2) * h
        out.append(MeshBlockGeom(n, (h, h, h), tuple(float(v) for v in lo), level=level,
                                 sommerfeld_faces=faces))
    return out, None, None


def _groups(blocks):
    """{shape: [block index, ...]} of equal-shaped blocks, at most about two
    million vertices per group."""
    by = {}
    for b, g in enumerate(blocks):
        by.setdefault(g.shape, []).append(b)
    out = []
    for shape, ids in by.items():
        step = max(1, int(1e6 // np.prod(shape)))
        out += [(shape, ids[q:q + step]) for q in range(0, len(ids), step)]
    return out


def _coords(blocks, ids):
    """x, y, z (broadcastable to nblocks, nn3, nn2, nn1) of equal-shaped blocks."""
    out = []
    for d in range(3):
        n = blocks[ids[0]].nn[d]
        i = torch.arange(n, dtype=torch.float64, device=DEV) - NG
        lo = torch.tensor([blocks[b].xmin[d] for b in ids], dtype=torch.float64, device=DEV)
        h = torch.tensor([blocks[b].dx[d] for b in ids], dtype=torch.float64, device=DEV)
        v = lo[:, None] + i[None, :] * h[:, None]
        shape = [len(ids), 1, 1, 1]
        shape[3 - d] = n
        out.append(v.view(shape))
    return out


# ---------------------------------------------------------------------- data
def _params(case):
    if case["data"] == "wave":
        # harmonic slicing, no shift
        return Params(lapse_oplog=0.0, lapse_harmonicf=1.0, lapse_harmonic=1.0, lapse_advect=0.0,
                      shift_Gamma=0.0, shift_advect=0.0, shift_eta=0.0, diss=0.02)
    # the step's gradient runs keep AlgConstr away from its branch switch at
    # det g~ = 1 + eps_floor, where the step has no derivative
    eps = -0.5 if case["kind"] == "vjp_step" else 1e-12
    return Params(lapse_oplog=2.0, lapse_harmonicf=1.0, lapse_advect=1.0, shift_Gamma=1.0,
                  shift_advect=1.0, shift_eta=2.0, diss=0.02, damp_kappa1=0.02,
                  chi_div_floor=1e-5, eps_floor=eps)


def _bumps(x, y, z, amp, rng, scale, dx):
    """Sum of four separable Gaussian bumps around the blocks' coordinates."""
    out = 0.0
    for _ in range(4):
        c = rng.uniform(-0.5, 0.5, 3) * scale + np.array([dx, 0.0, 0.0])
        w = rng.uniform(0.2, 0.5) * scale
        a = amp * rng.uniform(0.2, 1.0) * rng.choice([-1.0, 1.0])
        e = [torch.exp(-((v - c[d]) / w) ** 2) for d, v in enumerate((x, y, z))]
        out = out + a * (e[0] * e[1] * e[2])
    return out


def _state(case, blocks, ids, shape, seed):
    """(22, len(ids), nn3, nn2, nn1) initial state of equal-shaped blocks."""
    x, y, z = _coords(blocks, ids)
    u = torch.zeros((22, len(ids)) + shape, dtype=torch.float64, device=DEV)
    rng = np.random.default_rng(1000 + seed)
    if case["data"] == "wave":
        amp = 0.01 * (1.0 + 0.1 * rng.random())
        phase = 2 * math.pi * (x + rng.random())
        H = 1.0 - amp * torch.sin(phase)
        Kxx = -math.pi * amp * torch.cos(phase) / torch.sqrt(H)
        chi = H ** (-1.0 / 3.0)
        K = Kxx / H
        u[0] = chi
        u[1] = chi * H
        u[4] = u[6] = chi
        u[7] = K
        u[8] = chi * (Kxx - H * K / 3.0)
        u[11] = -chi * K / 3.0
        u[13] = -chi * K / 3.0
        u[18] = torch.sqrt(H)
        return u
    if case["data"] == "bumps":
        for n in range(22):
            u[n] = _bumps(x, y, z, 1e-3, rng, 1.0, 0.0)
        for n in (0, 1, 4, 6, 18):
            u[n] += 1.0
        return u
    off = 0.5 * 2.0 ** -7
    m = 0.5 + 0.05 * rng.uniform(-1.0, 1.0, 2)
    r = [torch.sqrt((x - off - s) ** 2 + (y - off) ** 2 + (z - off) ** 2) for s in (5.0, -5.0)]
    psi = 1.0 + m[0] / (2 * r[0]) + m[1] / (2 * r[1])
    for n in range(22):
        u[n] = _bumps(x, y, z, 1e-3, rng, 8.0, 5.0 * rng.choice([-1.0, 1.0]))
    u[0] += psi ** -4
    u[0].abs_()
    for n in (1, 4, 6):
        u[n] += 1.0
    u[18] += psi ** -2
    return u


def _fill(z, case, seed, make, nvar):
    """Flat device buffer of ``nvar`` fields from make(ids, shape)."""
    buf = z.empty(nvar)
    for shape, ids in _groups(z.blocks):
        val = make(ids, shape)
        for q, b in enumerate(ids):
            z.block_view(buf, b, nvar).copy_(val[:, q])
    return buf


def _matter(z, case, seed):
    def make(ids, shape):
        x, y, zz = _coords(z.blocks, ids)
        rng = np.random.default_rng(7 + seed)
        return torch.stack([_bumps(x, y, zz, 1e-3, rng, 8.0, 0.0).expand((len(ids),) + shape)
                            for _ in range(10)])
    return _fill(z, case, seed, make, 10)


def prepare(case, seed):
    blocks, lo, hi = _blocks(case)
    z = Z4c(blocks, _params(case))
    u = _fill(z, case, seed, lambda ids, shape: _state(case, blocks, ids, shape, seed), 22)
    z.AlgConstr(u)
    st = dict(z=z, u=u, kind=case["kind"])
    gen = torch.Generator(device=DEV).manual_seed(4242 + seed)
    if case["kind"] == "rhs":
        st["mat"] = _matter(z, case, seed) if case["matter"] else None
        st["rhs"], st["faces"] = z.zeros(), case["faces"]
    elif case["kind"] == "step":
        st["work"] = z.make_step_work()
    elif case["kind"] == "constraints":
        st["adm"], st["con"] = z.zeros(17), z.zeros(7)
        st["hist"] = torch.zeros(8, dtype=torch.float64, device=DEV)
    else:
        # cotangents of interior vertices, as an objective over owned vertices gives them
        nw = case["nw"]
        w = torch.zeros(nw * 22 * z.total_points, dtype=torch.float64, device=DEV)
        for q in range(nw):
            reg = w[q * 22 * z.total_points:(q + 1) * 22 * z.total_points]
            for b in range(len(blocks)):
                v = z.block_view(reg, b, 22)[:, NG:-NG, NG:-NG, NG:-NG]
                v.copy_(torch.randn(v.shape, generator=gen, dtype=torch.float64, device=DEV))
        st["w"], st["nw"] = w, nw
    if case["kind"] in ("step", "vjp_step"):
        st["dt"] = z.NewBlockTimeStep(0.25)
        st["ghosts"] = dict(periodic=case["ghosts"] == "periodic", exchange=case["ghosts"] == "tree",
                            physical=case["ghosts"] == "tree")
        st["graph"] = bool(case.get("graph"))
        if case["ghosts"] == "tree":
            z.set_exchange(lo, hi, periodic=False)
    return st


def run(state):
    z, kind = state["z"], state["kind"]
    if kind == "rhs":
        z.Z4cRHS(state["u"], state["mat"], state["rhs"])
        if state["faces"]:
            z.Z4cBoundaryRHS(state["u"], state["mat"], state["rhs"])
        return state["rhs"]
    if kind == "step":
        z.rk4_step_fused(state["dt"], state["u"], state["work"], graph=state["graph"],
                         **state["ghosts"])
        return state["u"]
    if kind == "constraints":
        z.Z4cToADM(state["u"], state["adm"])
        z.ADMConstraints(state["con"], state["adm"], None, state["u"])
        z.history_noalloc(state["u"], state["con"], state["hist"])
        return {"adm": state["adm"], "con": state["con"], "hist": state["hist"]}
    if kind == "vjp_rhs":
        return z.rhs_vjp(state["u"], state["w"], nw=state["nw"])
    if state["ghosts"]["exchange"]:
        return z.rk4_step_ghosts_vjp(state["dt"], state["u"], state["w"], nw=state["nw"],
                                     physical=True)
    return z.rk4_step_vjp(state["dt"], state["u"], state["w"], nw=state["nw"])


# ------------------------------------------------------- exact, in torch f64
# Fields carry their component indices first and (block, z, y, x) last.
SYM = ((0, 1, 2), (1, 3, 4), (2, 4, 5))
PAIRS = ((0, 0), (0, 1), (0, 2), (1, 1), (1, 2), (2, 2))


def _full(s):
    return torch.stack([torch.stack([s[SYM[a][b]] for b in range(3)]) for a in range(3)])


def _pack(t):
    return torch.stack([t[a, b] for a, b in PAIRS])


def _at(f, d, m):
    """f at offset m along axis d (x = 0), on the vertices 4 in from its ends."""
    ax = f.dim() - 1 - d
    return f.narrow(ax, NG + m, f.shape[ax] - 2 * NG)


def _crop(f, axes=(0, 1, 2)):
    for d in axes:
        f = _at(f, d, 0)
    return f


def _lin(f, d, weights):
    out = 0.0
    for m, c in weights:
        out = out + c * _at(f, d, m)
    return out


_D1 = ((-3, -1 / 60), (-2, 9 / 60), (-1, -45 / 60), (1, 45 / 60), (2, -9 / 60), (3, 1 / 60))
_D2 = ((-3, 2 / 180), (-2, -27 / 180), (-1, 270 / 180), (0, -490 / 180), (1, 270 / 180),
       (2, -27 / 180), (3, 2 / 180))
_KO = ((-4, 1.), (-3, -8.), (-2, 28.), (-1, -56.), (0, 70.), (1, -56.), (2, 28.), (3, -8.), (4, 1.))
_LEFT = ((-4, 1 / 60), (-3, -8 / 60), (-2, 30 / 60), (-1, -80 / 60), (0, 35 / 60), (1, 24 / 60),
         (2, -2 / 60))
_RIGHT = tuple((-m, -c) for m, c in _LEFT)


class _Grid:
    """Differences on a group of equal-shaped blocks of spacings h[d] (block,)."""

    def __init__(self, blocks, ids):
        self.h = [torch.tensor([blocks[b].dx[d] for b in ids], dtype=torch.float64,
                               device=DEV).view(-1, 1, 1, 1) for d in range(3)]

    def one(self, f, d):
        return _lin(f, d, _D1) / self.h[d]

    def grad(self, f):
        return torch.stack([_crop(self.one(f, d), [e for e in range(3) if e != d])
                            for d in range(3)])

    def hess(self, f):
        rows = {}
        for a, b in PAIRS:
            if a == b:
                rows[a, a] = _crop(_lin(f, a, _D2) / self.h[a] ** 2,
                                   [e for e in range(3) if e != a])
            else:
                rows[a, b] = rows[b, a] = _crop(self.one(self.one(f, b), a), [3 - a - b])
        return torch.stack([torch.stack([rows[a, b] for b in range(3)]) for a in range(3)])

    def advect(self, f, beta):
        out = 0.0
        for d in range(3):
            rest = [e for e in range(3) if e != d]
            left = _crop(_lin(f, d, _LEFT), rest)
            right = _crop(_lin(f, d, _RIGHT), rest)
            out = out + beta[d] * torch.where(beta[d] < 0, left, right) / self.h[d]
        return out

    def dissipate(self, f, diss):
        return sum(_crop(_lin(f, d, _KO), [e for e in range(3) if e != d]) / self.h[d]
                   for d in range(3)) * (-diss / 256.0)


def _ein(spec, *t):
    """einsum over leading component indices (each index once per operand),
    operand by operand, as broadcast products and sums."""
    ins, out = spec.split("->")
    ins = ins.split(",")
    cur, idx = t[0], ins[0]
    for q in range(1, len(t)):
        every = "".join(sorted(set(idx + ins[q])))

        def spread(v, names):
            v = v.permute([names.index(c) for c in sorted(names)] + list(range(len(names), v.dim())))
            return v[tuple(slice(None) if c in names else None for c in every)]
        cur = spread(cur, idx) * spread(t[q], ins[q])
        later = out + "".join(ins[q + 1:])
        drop = [every.index(c) for c in every if c not in later]
        cur = cur.sum(drop) if drop else cur
        idx = "".join(c for c in every if c in later)
    return cur.permute([idx.index(c) for c in out] + list(range(len(out), cur.dim())))


def _det_inv(g):
    c = torch.stack([torch.stack([g[(a + 1) % 3, (b + 1) % 3] * g[(a + 2) % 3, (b + 2) % 3]
                                  - g[(a + 1) % 3, (b + 2) % 3] * g[(a + 2) % 3, (b + 1) % 3]
                                  for b in range(3)]) for a in range(3)])
    det = g[0, 0] * c[0, 0] + g[0, 1] * c[0, 1] + g[0, 2] * c[0, 2]
    return det, c / det


def _christoffel(gi, dg):
    """Gamma_{c,ab}, Gamma^c_ab from dg[c, a, b] = d_c g_ab."""
    low = 0.5 * (dg.permute(2, 0, 1, *range(3, dg.dim())) + dg.permute(2, 1, 0, *range(3, dg.dim()))
                 - dg)
    return low, _ein("cd,dab->cab", gi, low)


def _rhs(u, grid, p, mat=None, eta=None, kappa1=None, kappa2=None):
    """Right-hand sides (22, block, interior) of states u (22, block, padded)."""
    eta = p.shift_eta if eta is None else eta
    k1 = p.damp_kappa1 if kappa1 is None else kappa1
    k2 = p.damp_kappa2 if kappa2 is None else kappa2
    c = _crop(u)
    g, A, Gam, beta = _full(c[1:7]), _full(c[8:14]), c[14:17], c[19:22]
    Kh, Th, al = c[7], c[17], c[18]
    chi = torch.clamp(c[0], min=p.chi_div_floor)
    det, gi = _det_inv(g)
    dgs = torch.stack([grid.grad(u[1 + n]) for n in range(6)])          # (ab, c)
    dg = torch.stack([_full(dgs[:, d]) for d in range(3)])              # c, a, b
    low, up = _christoffel(gi, dg)
    Gd = _ein("bc,abc->a", gi, up)
    lap = _full(torch.stack([_ein("cd,cd->", gi, grid.hess(u[1 + n])) for n in range(6)]))
    dGam = torch.stack([grid.grad(u[14 + n]) for n in range(3)])        # c, b
    t = _ein("ca,cb->ab", g, dGam)
    q = _ein("c,abc->ab", Gd, low)
    R = -0.5 * lap + 0.5 * (t + t.transpose(0, 1)) + 0.5 * (q + q.transpose(0, 1))
    gu = _ein("cd,eca->dea", gi, up)                                    # g^cd Gamma^e_ca
    s = _ein("dea,bed->ab", gu, low)
    R = R + s + s.transpose(0, 1) + _ein("cd,ead,ecb->ab", gi, up, low)
    dchi = grid.grad(u[0])
    dphi = dchi / (chi * p.chi_psi_power)
    Dphi = (grid.hess(u[0]) / (chi * p.chi_psi_power)
            - p.chi_psi_power * dphi[:, None] * dphi[None, :] - _ein("cab,c->ab", up, dphi))
    tr = _ein("cd,cd->", gi, Dphi + 2 * dphi[:, None] * dphi[None, :])
    R = R + 4 * dphi[:, None] * dphi[None, :] - 2 * Dphi - 2 * g * tr
    dal = grid.grad(u[18])
    Da = grid.hess(u[18]) - 2 * (dphi[:, None] * dal[None, :] + dal[:, None] * dphi[None, :])
    Da = Da + 2 * g * _ein("cd,c,d->", gi, dphi, dal) - _ein("cab,c->ab", up, dal)
    psi4i = chi                                                         # chi_psi_power = -4
    trDa = psi4i * _ein("ab,ab->", gi, Da)
    Rs = psi4i * _ein("ab,ab->", gi, R)
    Aud = _ein("cd,db->cb", gi, A)
    AA = _ein("ac,cb->ab", A, Aud)
    trAA = _ein("ab,ab->", gi, AA)
    Auu = _ein("ac,bc->ab", Aud, gi)
    dK, dT = grid.grad(u[7]), grid.grad(u[17])
    DA = (6 / p.chi_psi_power) * _ein("ab,b->a", Auu, dchi) / chi
    DA = DA - _ein("ab,b->a", gi, 2 * dK + dT) / 3 + _ein("abc,bc->a", up, Auu)
    K = Kh + 2 * Th
    Ht = Rs + 2 / 3 * K * K - trAA
    db = torch.stack([grid.grad(u[19 + n]) for n in range(3)]).transpose(0, 1)   # b, a
    div = db[0, 0] + db[1, 1] + db[2, 2]
    hb = [grid.hess(u[19 + n]) for n in range(3)]
    adv = [1.0] * 22
    adv[18], adv[19:22] = p.lapse_advect, [p.shift_advect] * 3
    LD = [adv[n] * grid.advect(u[n], beta) + grid.dissipate(u[n], p.diss) for n in range(22)]
    rho, S, Sd = 0.0, None, None
    trS = 0.0
    if mat is not None:
        m = _crop(mat)
        rho, S, Sd = m[0], m[1:4], _full(m[4:10])
        trS = psi4i * _ein("ab,ab->", gi, Sd)
    pi = math.pi
    out = [None] * 22
    out[0] = LD[0] + p.chi_psi_power / 6 * chi * (div - al * K)
    out[7] = (LD[7] - trDa + al * (trAA + K * K / 3) + k1 * (1 - k2) * al * Th
              + 4 * pi * al * (trS + rho))
    out[17] = LD[17] + al * (0.5 * Ht - (2 + k2) * k1 * Th) - 8 * pi * al * rho
    ddb = torch.stack([sum(hb[b][a, b] for b in range(3)) for a in range(3)]) / 3
    dG = _ein("ab,b->a", gi, ddb) - _ein("b,ba->a", Gd, db) + 2 / 3 * Gd * div
    dG = dG + torch.stack([_ein("bc,bc->", gi, hb[a]) for a in range(3)])
    dG = dG + 2 * al * DA - 2 * al * k1 * (Gam - Gd) - 2 * _ein("ab,b->a", Auu, dal)
    if S is not None:
        dG = dG - 16 * pi * al * _ein("ab,b->a", gi, S)
    gb, Ab = _ein("ac,bc->ab", db, g), _ein("bc,ac->ab", db, A)
    rg = gb + gb.transpose(0, 1) - 2 / 3 * g * div - 2 * al * A
    rA = Ab + Ab.transpose(0, 1) - 2 / 3 * A * div
    rA = rA + psi4i * (al * R - Da) - g / 3 * (al * Rs - trDa) + al * (K * A - 2 * AA)
    if S is not None:
        rA = rA - 8 * pi * al * (psi4i * Sd - trS * g / 3)
    for n, (a, b) in enumerate(PAIRS):
        out[1 + n] = LD[1 + n] + rg[a, b]
        out[8 + n] = LD[8 + n] + rA[a, b]
    f = p.lapse_oplog * p.lapse_harmonicf + p.lapse_harmonic * al
    out[18] = LD[18] - f * al * (Kh + 2 * p.lapse_K * Th)
    for a in range(3):
        out[14 + a] = LD[14 + a] + dG[a]
        out[19 + a] = LD[19 + a] + p.shift_Gamma * Gam[a] - eta * beta[a]
    return torch.stack([o.expand_as(c[0]) for o in out])


def _sommerfeld(rhs, u, blocks, ids, grid):
    """Radiative rows on the flagged faces: -c (u + x^a d_a u) / r, 2nd order."""
    faces = torch.tensor([blocks[b].sommerfeld_faces for b in ids], device=DEV).view(-1, 1, 1, 1)
    if not bool((faces != 0).any()):
        return rhs
    xyz = [_crop(v.expand(u.shape[1:])) for v in _coords(blocks, ids)]
    r = torch.sqrt(sum(v * v for v in xyz))
    on = torch.zeros_like(r, dtype=torch.bool)
    for d in range(3):
        i = torch.arange(r.shape[3 - d], device=DEV).view([-1 if q == 3 - d else 1
                                                            for q in range(4)])
        on |= ((faces >> (2 * d)) & 1).bool() & (i == 0)
        on |= ((faces >> (2 * d + 1)) & 1).bool() & (i == r.shape[3 - d] - 1)
    rows = list(rhs)
    for n in (17, 7, 14, 15, 16, 8, 9, 10, 11, 12, 13):
        c = math.sqrt(2.0) if n == 7 else 1.0
        v = -_crop(u[n]) / r
        for d in range(3):
            du = _crop(_lin(u[n], d, ((-1, -0.5), (1, 0.5))) / grid.h[d],
                       [e for e in range(3) if e != d])
            v = v - xyz[d] / r * du
        rows[n] = torch.where(on, c * v, rows[n])
    return torch.stack(rows)


def _constrain(u, eps):
    """det g~ = 1 (a constant factor below the floor) and trace-free A~."""
    g, A = _full(u[1:7]), _full(u[8:14])
    det, _ = _det_inv(g)
    det = torch.where(det > 0, det, torch.ones_like(det))
    low = det - 1.0 < eps
    fac = torch.where(low, torch.full_like(det, 1.0 - eps / 3.0),
                      torch.where(low, torch.ones_like(det), det) ** (-1.0 / 3.0))
    g = g * fac
    d, gi = _det_inv(g)
    A = A - d * _ein("ab,ab->", gi, A) * g / 3.0
    return torch.cat([u[:1], _pack(g), u[7:8], _pack(A), u[14:]])


def _pad(k):
    return torch.nn.functional.pad(k, (NG, NG) * 3)


def _periodic(u):
    """VC periodic fill of one block: shared vertices averaged, then ghosts."""
    for d in range(3):
        ax = u.dim() - 1 - d
        n = u.shape[ax] - 2 * NG - 1
        inner = u.narrow(ax, NG, n + 1)
        mean = 0.5 * (inner.narrow(ax, 0, 1) + inner.narrow(ax, n, 1))
        body = torch.cat([mean, inner.narrow(ax, 1, n - 1)], ax)
        idx = (torch.arange(-NG, n + NG + 1, device=u.device)) % n
        u = body.index_select(ax, idx)
    return u


def _step(u, grid, p, dt, after, rhs, **kw):
    """One bt_rk4 step; ``after`` follows each stage's sum (before the
    algebraic constraints)."""
    a, b = (0.5, 0.5, 1.0), (1 / 6, 1 / 3, 1 / 3, 1 / 6)
    v, acc = u, u
    for s in range(4):
        k = _pad(rhs(v, **kw))
        acc = acc + (b[s] * dt) * k
        v = _constrain(after(u + (a[s] * dt) * k if s < 3 else acc), p.eps_floor)
    return v


def _adm(u):
    psi4 = 1.0 / u[0]
    G = psi4 * u[1:7]
    K = psi4 * u[8:14] + (u[7] + 2 * u[17]) / 3 * G
    return torch.cat([u[18:22], G, K, psi4[None]])


def _constraints(u, adm, grid, p):
    """C, H, M, Z, M_x, M_y, M_z on the interior of the blocks."""
    c, ad = _crop(u), _crop(adm)
    gt, G, Kd = _full(c[1:7]), _full(ad[4:10]), _full(ad[10:16])
    chi = torch.clamp(c[0], min=p.chi_div_floor)
    dchi, hchi = grid.grad(u[0]), grid.hess(u[0])
    dgt = torch.stack([grid.grad(u[1 + n]) for n in range(6)])
    dgt = torch.stack([_full(dgt[:, d]) for d in range(3)])
    hgt = torch.stack([grid.hess(u[1 + n]) for n in range(6)])
    hgt = torch.stack([torch.stack([_full(hgt[:, a, b]) for b in range(3)]) for a in range(3)])
    dg = (dgt - gt * dchi[:, None, None] / chi) / chi
    dd = (hgt - (dchi[:, None, None, None] * dgt[None] + dchi[None, :, None, None] * dgt[:, None]
                 + hchi[:, :, None, None] * gt) / chi
          + 2 * dchi[:, None, None, None] * dchi[None, :, None, None] * gt / chi ** 2) / chi
    _, gi = _det_inv(G)
    low, up = _christoffel(gi, dg)
    R = (_ein("ef,cae,cbf->ab", gi, up, low) - _ein("ef,cab,cef->ab", gi, up, low)
         + 0.5 * (-_ein("cd,bacd->ab", gi, dd) + _ein("cd,dabc->ab", gi, dd)
                  + _ein("cd,dbac->ab", gi, dd) - _ein("cd,dcab->ab", gi, dd)))
    Kud = _ein("ac,cb->ab", gi, Kd)
    K = Kud[0, 0] + Kud[1, 1] + Kud[2, 2]
    H = _ein("ab,ab->", gi, R) + K * K - _ein("ab,ba->", Kud, Kud)
    dK = torch.stack([grid.grad(adm[10 + n]) for n in range(6)])
    dK = torch.stack([_full(dK[:, d]) for d in range(3)])
    DK = dK - _ein("dab,dc->abc", up, Kd) - _ein("dac,bd->abc", up, Kd)
    DKu = _ein("ad,dbc->abc", gi, DK)
    Mu = _ein("ab,b->a", gi, sum(DKu[c, :, c] for c in range(3))) - _ein("bc,abc->a", gi, DKu)
    Md = _ein("ab,b->a", G, Mu)
    _, cgi = _det_inv(gt)
    _, cup = _christoffel(cgi, dgt)
    Gd = c[14:17] - _ein("bc,abc->a", cgi, cup)
    M = _ein("ab,a,b->", G, Mu, Mu)
    Z = 0.25 * _ein("ab,a,b->", G, Gd, Gd)
    C = H * H + M + c[17] ** 2 + 4 * Z
    return torch.stack([C, H, M, Z, Md[0], Md[1], Md[2]])


def _gather(buf, blocks, ids, offsets, nvar):
    return torch.stack([buf[offsets[b] * nvar:(offsets[b] + blocks[b].npts) * nvar]
                        .view((nvar,) + blocks[b].shape) for b in ids], dim=1)


def _scatter(buf, val, blocks, ids, offsets, nvar):
    for q, b in enumerate(ids):
        buf[offsets[b] * nvar:(offsets[b] + blocks[b].npts) * nvar].view(
            (nvar,) + blocks[b].shape).copy_(val[:, q])


def exact(case, seed):
    kind, ghosts = case["kind"], case.get("ghosts")
    if ghosts == "tree":
        return None      # the update across levels takes minutes in plain torch
    st = prepare(case, seed)
    z, p, u0 = st["z"], st["z"].params, st["u"]
    blocks, off = z.blocks, z.offsets
    inner = sum((g.nx[0] + 1) * (g.nx[1] + 1) * (g.nx[2] + 1) for g in blocks)
    cost = inner * {"rhs": 1, "step": 4, "constraints": 1, "vjp_rhs": 3 * case.get("nw", 1),
                    "vjp_step": 12 * case.get("nw", 1)}[kind]
    if cost > 2e7:
        return None      # over the time a check may take
    groups = []
    for shape, ids in _groups(blocks):
        cut = max(1, int(4e5 // np.prod(shape)))
        groups += [ids[q:q + cut] for q in range(0, len(ids), cut)]

    if kind == "constraints":
        out = {"adm": torch.zeros_like(st["adm"]), "con": torch.zeros_like(st["con"]),
               "hist": torch.zeros_like(st["hist"])}
        for ids in groups:
            grid = _Grid(blocks, ids)
            u = _gather(u0, blocks, ids, off, 22)
            adm = _adm(u)
            con = _constraints(u, adm, grid, p)
            _scatter(out["adm"], adm, blocks, ids, off, 17)
            _scatter(out["con"], _pad(con), blocks, ids, off, 7)
            vol = grid.h[0] * grid.h[1] * grid.h[2]
            cell = con[:, :, :-1, :-1, :-1] * torch.ones_like(vol)
            th = _crop(u[17])[:, :-1, :-1, :-1]
            cols = [cell[1] ** 2, cell[2].abs(), cell[4] ** 2, cell[5] ** 2, cell[6] ** 2,
                    cell[3].abs(), th ** 2, cell[0].abs()]
            out["hist"] += torch.stack([(vol * v).sum() for v in cols])
        return out

    def rhs_of(ids, grid):
        return lambda v, **kw: _sommerfeld(_rhs(v, grid, p, **kw), v, blocks, ids, grid)

    if kind == "rhs":
        out = torch.zeros_like(u0)
        for ids in groups:
            grid = _Grid(blocks, ids)
            mat = _gather(st["mat"], blocks, ids, off, 10) if case["matter"] else None
            r = rhs_of(ids, grid)(_gather(u0, blocks, ids, off, 22), mat=mat)
            _scatter(out, _pad(r), blocks, ids, off, 22)
        return out
    after = _periodic if ghosts == "periodic" else (lambda v: v)
    if kind == "step":
        out = torch.zeros_like(u0)
        for ids in groups:
            grid = _Grid(blocks, ids)
            v = _step(_gather(u0, blocks, ids, off, 22), grid, p, st["dt"], after,
                      rhs_of(ids, grid))
            _scatter(out, v, blocks, ids, off, 22)
        return out
    nw, size = case["nw"], 22 * z.total_points
    ubar = torch.zeros(nw * size, dtype=torch.float64, device=DEV)
    pbar = torch.zeros(nw, 3, dtype=torch.float64, device=DEV)
    for ids in groups:
        grid = _Grid(blocks, ids)
        u = _gather(u0, blocks, ids, off, 22).requires_grad_(True)
        par = torch.tensor([p.shift_eta, p.damp_kappa1, p.damp_kappa2], dtype=torch.float64,
                           device=DEV, requires_grad=True)
        kw = dict(eta=par[0], kappa1=par[1], kappa2=par[2])
        if kind == "vjp_rhs":
            v = _pad(_rhs(u, grid, p, **kw))
        else:
            v = _step(u, grid, p, st["dt"], after, rhs_of(ids, grid), **kw)
        for q in range(nw):
            w = _gather(st["w"][q * size:(q + 1) * size], blocks, ids, off, 22)
            du, dp = torch.autograd.grad(v, (u, par), w, retain_graph=q + 1 < nw)
            _scatter(ubar[q * size:(q + 1) * size], du, blocks, ids, off, 22)
            pbar[q] += dp
        del v
    return ubar, pbar
