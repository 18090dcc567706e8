"""The work that a user of this package has it do, as cases that can be timed.

A case is a dict of plain values; its ``kind`` says which public entry points one pass calls:

* ``md``     one ``VerletIntegrator.run(steps)`` (NVE, NVT with a Nose-Hoover chain or the
             Langevin thermostat, NPT with the chain and the MTK barostat);
* ``batch``  one ``BatchVerlet.run(steps)`` over replicas of uneven size;
* ``force``  one force evaluation: ``MicMecForceField.compute`` on host arrays, or
             ``ForcePartMechanical.compute_device`` on device tensors;
* ``relax``  one ``CGOptimizer.run(steps)`` from the strained, noisy start;
* ``fit``    one forward and backward pass of ``FitProblem.loss`` (parameter gradients);
* ``grad``   ``micmec_energy`` and the gradients of a function of its three outputs with respect
             to positions, domain vectors and parameters.

``prepare`` makes the inputs from the seed and holds what such a program keeps (system, field,
integrator); ``run`` is one pass; ``work`` the bytes and operations a pass cannot do without;
``exact`` the same outputs from plain torch and numpy in 64 bits.
"""

import numpy as np
import torch

# Cell types of the package's own workloads: cubic rest cells (edge in angstrom) and elasticity
# (C11, C12, C44 in GPa) of every metastable state; the states combine at 300 K.
TYPES = {1: [(20.7, (40.0, 20.0, 10.0))],
         2: [(20.9, (30.0, 18.0, 7.0)), (0.97 * 20.9, (24.0, 14.4, 5.6))]}
T_EFF = 300.0
CELL_MASS_AMU = 8 * 6000.0
# offsets of a cell's eight corners, and the three edges (lower, upper corner) through each
OFF = np.array([(0, 0, 0), (1, 0, 0), (0, 1, 0), (0, 0, 1),
                (1, 1, 0), (1, 0, 1), (0, 1, 1), (1, 1, 1)])
LO = [[0, 0, 0], [0, 1, 1], [2, 0, 2], [3, 3, 0], [2, 1, 4], [3, 5, 1], [6, 3, 2], [6, 5, 4]]
HI = [[1, 2, 3], [1, 4, 5], [4, 2, 6], [5, 6, 3], [4, 4, 7], [5, 7, 5], [7, 6, 6], [7, 7, 7]]
VOIGT = [(0, 0), (1, 1), (2, 2), (1, 2), (0, 2), (0, 1)]


def listed():
    return [
        # the smallest system of the package's configurations: a host-launched run of a 3^3
        # crystal, where a step costs its launches
        dict(name="nve 3^3", kind="md", ensemble="nve", nx=3, ny=3, nz=3, p_b=0.0, p_hole=0.0,
             pbc=True, steps=50),
        # the mid-size configuration: constant temperature, a fifth of the cells two-state
        dict(name="nvt 32^3", kind="md", ensemble="nvt", nx=32, ny=32, nz=32, p_b=0.2,
             p_hole=0.0, pbc=True, steps=40),
        # the headline configuration: constant temperature and pressure at 128^3, with voids
        dict(name="npt 128^3", kind="md", ensemble="npt", nx=128, ny=128, nz=128, p_b=0.2,
             p_hole=0.05, pbc=True, steps=20),
        # constant pressure on an ordinary, uneven box with a tenth of the cells missing
        dict(name="npt 24x19x27", kind="md", ensemble="npt", nx=24, ny=19, nz=27, p_b=0.3,
             p_hole=0.1, pbc=True, steps=20),
        # a finite crystal (open boundaries) under the stochastic thermostat
        dict(name="langevin open 40x36x47", kind="md", ensemble="langevin", nx=40, ny=36, nz=47,
             p_b=0.2, p_hole=0.05, pbc=False, steps=20),
        # many small systems of uneven size and composition in one engine
        dict(name="batch 192", kind="batch", replicas=192, nmin=4, nmax=24, steps=20),
        # the plain plugin call on host arrays, as a script or an optimiser of one's own makes it
        dict(name="force host 5^3", kind="force", nx=5, ny=5, nz=5, p_b=0.2, p_hole=0.0,
             pbc=True, model="corner8", where="host", gradient=True),
        # one evaluation of the averaged-matrix model on device tensors, odd sizes
        dict(name="force original 61x64x67", kind="force", nx=61, ny=64, nz=67, p_b=0.2,
             p_hole=0.05, pbc=True, model="original", where="device", gradient=True),
        # one evaluation of a large system on device tensors, most of it two-state
        dict(name="force 72x80x96", kind="force", nx=72, ny=80, nz=96, p_b=0.7, p_hole=0.0,
             pbc=True, model="corner8", where="device", gradient=True),
        # geometry optimisation from a strained start
        dict(name="relax 48^3", kind="relax", nx=48, ny=48, nz=48, p_b=0.2, p_hole=0.05,
             pbc=True, steps=6),
        # the parameter fit: 64 configurations of 16^3 cells, one loss and its gradients
        dict(name="fit 64x16^3", kind="fit", count=64, n=16, p_b=0.2, model="corner8"),
        # gradients of a few small systems with respect to every input
        dict(name="grad 5x7^3", kind="grad", count=5, n=7, p_b=0.4, model="original"),
    ]


def draw(rng):
    """One more case of these ranges: edges of 3 to 56 cells, spread over their logarithm."""
    def edge(lo, hi):
        return max(lo, min(hi, int(round(lo * (hi / lo) ** rng.random()))))

    kind = rng.choice(["md", "md", "md", "batch", "force", "force", "relax", "fit", "grad"])
    model = rng.choice(["corner8", "corner8", "original"])
    mix = dict(p_b=round(rng.choice([0.0, 0.2, rng.random(), 1.0]), 3),
               p_hole=round(rng.choice([0.0, 0.3 * rng.random()]), 3))
    box = dict(nx=edge(3, 56), ny=edge(3, 56), nz=edge(3, 56))
    if kind == "md":
        ensemble = rng.choice(["nve", "nvt", "npt", "langevin"])
        pbc = True if ensemble in ("npt", "nvt") else rng.random() < 0.7
        return dict(kind=kind, ensemble=ensemble, pbc=pbc, steps=rng.randint(5, 40), **box, **mix)
    if kind == "batch":
        nmin = rng.randint(3, 8)
        return dict(kind=kind, replicas=edge(4, 96), nmin=nmin, nmax=nmin + rng.randint(0, 12),
                    steps=rng.randint(5, 30))
    if kind == "force":
        where = "host" if box["nx"] * box["ny"] * box["nz"] < 3000 else "device"
        return dict(kind=kind, pbc=rng.random() < 0.7, model=model, where=where,
                    gradient=rng.random() < 0.8, **box, **mix)
    if kind == "relax":
        return dict(kind=kind, pbc=True, steps=rng.randint(3, 6), nx=edge(5, 40), ny=edge(5, 40),
                    nz=edge(5, 40), **mix)
    return dict(kind=kind, count=edge(2, 24), n=edge(3, 14),
                p_b=round(0.1 + 0.6 * rng.random(), 3), model=model)


# ------------------------------------------------------------------------------------- inputs
def _grid(shape, p_b, p_hole, rng):
    """Type grid: 2 with probability p_b, otherwise 1; 0 (empty) with probability p_hole. One
    cell of each type that the probabilities allow is always there. The empty sites belong to the
    case (the number of nodes follows from them), everything else to the seed."""
    g = np.where(rng.random(shape) < p_b, 2, 1)
    if p_hole > 0:
        g[np.random.default_rng([7, *shape]).random(shape) < p_hole] = 0
    if p_b < 1.0:
        g.flat[0] = 1
    if p_b > 0.0:
        g.flat[1] = 2
    return g


def _shape(case):
    return (case["nx"], case["ny"], case["nz"])


def _noise(pos, rvecs, rng, noise, strain):
    """Positions with Gaussian noise (angstrom), and a random symmetric strain of everything."""
    from micmec_amd import units
    pos = pos + rng.normal(0.0, noise * units.angstrom, pos.shape)
    if strain:
        e = rng.uniform(-strain, strain, (3, 3))
        F = np.identity(3) + 0.5 * (e + e.T)
        pos, rvecs = pos @ F, (rvecs @ F if len(rvecs) else rvecs)
    return pos, rvecs


def _system(shape, p_b, p_hole, pbc, rng, noise=0.05, strain=0.0):
    from micmec_amd.system import System
    from micmec_amd.topology import build_system_device
    from micmec_amd.workloads import type_a, type_b
    grid = _grid(shape, p_b, p_hole, rng)
    types = {1: type_a(), 2: type_b()}
    out = build_system_device({t: types[t] for t in (1, 2) if (grid == t).any()}, grid, pbc=pbc)
    out["pos"], out["rvecs"] = _noise(out["pos"], out["rvecs"], rng, noise, strain)
    return System.from_dict(out)


def _md_start(masses, pos, open_, rng):
    """Maxwell-Boltzmann velocities at 300 K without momentum (and, of a finite system, without
    angular momentum), chain velocities and a symmetric barostat velocity, as a run that
    continues an earlier one has them."""
    from micmec_amd import units
    kT = units.boltzmann * 300.0
    vel = rng.normal(0.0, 1.0, pos.shape) * np.sqrt(kT / masses)[:, None]
    vel -= (masses @ vel) / masses.sum()
    if open_:
        x = pos - (masses @ pos) / masses.sum()
        m = masses[:, None]
        inertia = np.identity(3) * (m * x ** 2).sum() - x.T @ (m * x)
        vel -= np.cross(np.linalg.solve(inertia, np.cross(x, m * vel).sum(0)), x)
    chain, baro = rng.normal(0.0, 1.0, 3), rng.normal(0.0, 1.0, (3, 3))
    ndof = pos.size - (6 if open_ else 3)
    w = 2 * np.pi / (100 * units.femtosecond)
    mass = kT / w ** 2 * np.array([ndof, 1.0, 1.0])
    wb = 2 * np.pi / (1000 * units.femtosecond)
    mass_press = (ndof + 9) * kT / wb ** 2
    return dict(vel=vel, ndof=ndof, chain_mass=mass, chain=chain * np.sqrt(kT / mass),
                mass_press=mass_press,
                vel_press=0.5 * (baro + baro.T) * np.sqrt(kT / mass_press))


# -------------------------------------------------------------------------------------- cases
def prepare(case, seed):
    from micmec_amd import units
    from micmec_amd.pes import ForcePartMechanical, MicMecForceField
    rng = np.random.default_rng(seed)
    kind = case["kind"]
    fs = units.femtosecond
    if kind == "md":
        from micmec_amd.sampling import (LangevinThermostat, MTKBarostat, NHCThermostat,
                                         VerletIntegrator)
        system = _system(_shape(case), case["p_b"], case["p_hole"], case["pbc"], rng)
        mmf = MicMecForceField(system, [ForcePartMechanical(system)])
        m = np.asarray(system.masses)
        st = _md_start(m, np.asarray(system.pos), not case["pbc"], rng)
        hooks = []
        if case["ensemble"] in ("nvt", "npt"):
            hooks.append(NHCThermostat(temp=300.0, timecon=100 * fs, chainlength=3,
                                       chain_pos0=np.zeros(3), chain_vel0=st["chain"],
                                       restart=True))
        if case["ensemble"] == "npt":
            hooks.append(MTKBarostat(mmf, temp=300.0, press=units.bar, timecon=1000 * fs,
                                     vel_press0=st["vel_press"], restart=True))
        if case["ensemble"] == "langevin":
            hooks.append(LangevinThermostat(temp=300.0, timecon=100 * fs, seed=seed))
        verlet = VerletIntegrator(mmf, timestep=fs, hooks=hooks, vel0=st["vel"])
        return dict(case=case, verlet=verlet)
    if kind == "batch":
        from micmec_amd.batch import BatchVerlet
        systems, temps = [], []
        sizes = np.random.default_rng([11, case["replicas"]])
        for _ in range(case["replicas"]):
            n = int(sizes.integers(case["nmin"], case["nmax"] + 1))
            p_b, p_hole = float(rng.uniform(0.0, 1.0)), float(sizes.uniform(0.0, 0.3))
            systems.append(_system((n, n, n), p_b, p_hole, True, rng))
            temps.append(float(rng.uniform(100.0, 500.0)))
        batch = BatchVerlet(systems, fs, temps, [seed + k for k in range(len(systems))])
        return dict(case=case, batch=batch)
    if kind == "force":
        system = _system(_shape(case), case["p_b"], case["p_hole"], case["pbc"], rng,
                         noise=0.1, strain=0.02)
        fpm = ForcePartMechanical(system, model=case["model"])
        if case["where"] == "host":
            return dict(case=case, mmf=MicMecForceField(system, [fpm]),
                        pos=np.array(system.pos), gpos=np.zeros(system.pos.shape),
                        vtens=np.zeros((3, 3)))
        kw = dict(dtype=torch.float64, device=fpm.device)
        rv = np.zeros((3, 3))
        rv[:len(system.domain.rvecs)] = system.domain.rvecs
        return dict(case=case, fpm=fpm, pos=torch.tensor(np.asarray(system.pos), **kw),
                    rvecs=torch.tensor(rv, **kw), energy=torch.zeros(1, **kw),
                    gpos=torch.zeros(system.pos.shape, **kw), vtens=torch.zeros((3, 3), **kw))
    if kind == "relax":
        system = _system(_shape(case), case["p_b"], case["p_hole"], case["pbc"], rng,
                         strain=0.02)
        mmf = MicMecForceField(system, [ForcePartMechanical(system)])
        return dict(case=case, mmf=mmf, pos=np.array(system.pos))
    from micmec_amd.adjoint import DiffField, FitProblem
    n, count = case["n"], case["count"]
    systems = [_system((n, n, n), case["p_b"], 0.0, True, rng, noise=0.1, strain=0.03)
               for _ in range(count)]
    field = DiffField(systems, model=case["model"])
    pos, rvecs = field.positions()
    params = field.initial_params()
    dev = dict(dtype=torch.float64, device=pos.device)
    if kind == "fit":
        target = field.initial_params()
        target.cv = target.cv * torch.tensor(_cv_noise(target.cv.shape, rng), **dev)
        a = torch.zeros_like(params.cv, requires_grad=True)
        b = torch.zeros_like(params.h0, requires_grad=True)
        return dict(case=case, problem=FitProblem(field, pos, rvecs, target), params=params,
                    a=a, b=b)
    weights = _cotangents(count, pos.shape, rng)
    return dict(case=case, field=field, params=params, pos=pos.requires_grad_(True),
                rvecs=rvecs.requires_grad_(True), w=[torch.tensor(x, **dev) for x in weights])


def _cv_noise(shape, rng):
    """Relative symmetric changes of up to 10% of every elasticity entry."""
    x = rng.uniform(-0.1, 0.1, tuple(shape))
    return 1.0 + 0.5 * (x + np.swapaxes(x, -1, -2))


def _cotangents(count, shape, rng):
    """Random derivatives of a scalar with respect to energies, node gradients and virials."""
    return (rng.normal(0.0, 1.0, count), rng.normal(0.0, 1.0, tuple(shape)),
            rng.normal(0.0, 1.0, (count, 3, 3)))


def run(state):
    case = state["case"]
    kind = case["kind"]
    if kind == "md":
        v = state["verlet"]
        v.run(case["steps"])
        # the trajectory's arrays where the integrator holds them; the scalars as attributes
        eng = v._engine
        return dict(pos=eng.pos, vel=eng.vel, gpos=eng.gpos, vtens=v.vtens, rvecs=v.rvecs,
                    scalars=np.array([v.epot, v.ekin, v.etot]), econs=np.float64(v.econs))
    if kind == "batch":
        b = state["batch"]
        b.run(case["steps"])
        return dict(pos=b.pos, vel=b.vel, gpos=b.gpos, epot=b.scalars("EPOT"),
                    ekin=b.scalars("EKIN"), econs=b.scalars("ECONS"))
    if kind == "force":
        if case["where"] == "host":
            mmf, gpos, vtens = state["mmf"], state["gpos"], state["vtens"]
            mmf.update_pos(state["pos"])
            if not case["gradient"]:
                return dict(energy=np.float64(mmf.compute()))
            gpos[:] = 0.0
            vtens[:] = 0.0
            return dict(energy=np.float64(mmf.compute(gpos, vtens)), gpos=gpos, vtens=vtens)
        out = dict(energy=state["energy"])
        if case["gradient"]:
            out.update(gpos=state["gpos"], vtens=state["vtens"])
        state["fpm"].compute_device(state["pos"], state["rvecs"], out["energy"],
                                    out.get("gpos"), out.get("vtens"))
        return out
    if kind == "relax":
        from micmec_amd.sampling import CartesianDOF, CGOptimizer
        state["mmf"].update_pos(state["pos"])
        dof = CartesianDOF(state["mmf"], gpos_rms=1e-30, dpos_rms=1e-30)
        opt = CGOptimizer(dof)
        opt.run(case["steps"])
        return dict(pos=opt.minimizer.x, gpos=opt.minimizer.g, epot=np.float64(opt.epot))
    from micmec_amd.adjoint import CellParams, micmec_energy
    p = state["params"]
    if kind == "fit":
        # one step's loss and gradients of the relative corrections, as ``fit`` forms them
        a, b = state["a"], state["b"]
        a.grad = b.grad = None
        now = CellParams(p.cv * (1.0 + 0.5 * (a + a.transpose(-1, -2))), p.h0 * (1.0 + b),
                         p.free, p.teff, p.nstates, p.type_ids)
        loss = state["problem"].loss(now)
        loss.backward()
        return dict(loss=loss, a=a.grad, b=b.grad)
    leaves = [state["pos"], state["rvecs"]] + [t.clone().requires_grad_(True)
                                               for t in p.tensors()]
    e, g, v = micmec_energy(state["field"], leaves[0], leaves[1],
                            CellParams(*leaves[2:], p.nstates, p.type_ids))
    wE, wG, wV = state["w"]
    grads = torch.autograd.grad((wE * e).sum() + (wG * g).sum() + (wV * v).sum(), leaves)
    return dict(energy=e, gpos=g, vtens=v, grads=list(grads))


def work(case):
    """Bytes and operations one pass cannot do without (a fused multiply-add counts as two).

    Per cell of the eight-corner model: edges, their products and the vertex sums 1010; per
    metastable state 48 strains, 66 x 8 stress and 11 x 8 energy operations. The averaged model
    forms one matrix instead of eight. Per node and step, position and velocity are read and
    written and the mass read (104 bytes), per further force evaluation the positions read and
    the gradient written (48 bytes); per cell one byte of type. Derivatives along a direction
    take three times the operations of the values."""
    kind = case["kind"]
    averaged = case.get("model") == "original"

    def per_cell(p_b):
        states = 1.0 + p_b
        return (290.0 + 85.0 * states) if averaged else (1010.0 + 664.0 * states)

    if kind == "batch":
        n = np.arange(case["nmin"], case["nmax"] + 1, dtype=float)
        nodes = case["replicas"] * float((n ** 3).mean())
        cells = 0.85 * nodes
        return {"bytes": case["steps"] * (104.0 * nodes + cells),
                "flops": case["steps"] * (cells * per_cell(0.5) + 60.0 * nodes)}
    if kind in ("fit", "grad"):
        nodes = cells = case["count"] * float(case["n"]) ** 3
        return {"bytes": 2 * (48.0 * nodes + cells),
                "flops": cells * per_cell(case["p_b"]) * 4.0}
    nodes = float(case["nx"] * case["ny"] * case["nz"])
    cells = nodes * (1.0 - case["p_hole"])
    one = cells * per_cell(case["p_b"])
    if kind == "md":
        evals = 3 if case["ensemble"] == "npt" else 1
        return {"bytes": case["steps"] * ((104.0 + 48.0 * (evals - 1)) * nodes + cells),
                "flops": case["steps"] * (evals * one + 60.0 * nodes)}
    if kind == "relax":
        return {"bytes": 2 * case["steps"] * (120.0 * nodes + cells),
                "flops": 2 * case["steps"] * one}
    return {"bytes": (48.0 if case["gradient"] else 24.0) * nodes + cells, "flops": one}


# ---------------------------------------------------------------------- the same in plain torch
class _Plain(object):
    """Energy, gradients and dynamics of one system from the definitions: per corner the strain
    e of the cell matrix against the rest matrix and det(h0)/8 e.C.e/2 (or once, of the averaged
    matrix), the states combined by their free energy; gradients by automatic differentiation."""

    def __init__(self, grid, pbc, model):
        cells = np.argwhere(grid != 0)
        dims = np.array(grid.shape)
        lattice = dims if pbc else dims + 1
        at = cells[:, None, :] + OFF[None]
        flat = np.ravel_multi_index(tuple(np.moveaxis(at % lattice, -1, 0)), tuple(lattice))
        used, inverse = np.unique(flat, return_inverse=True)
        self.sn = torch.from_numpy(inverse.reshape(flat.shape))
        self.shift = torch.from_numpy((at // lattice).astype(float))
        self.node_ijk = np.stack(np.unravel_index(used, tuple(lattice)), 1)
        self.types = grid[grid != 0]
        self.sel = {t: torch.from_numpy(np.nonzero(self.types == t)[0])
                    for t in (1, 2) if (self.types == t).any()}
        self.model = model
        counts = np.bincount(grid.ravel(), minlength=3)[1:]
        self.spacing = _parameters()[int(np.argmax(counts)) + 1][0][0][0, 0].item()
        self.dims, self.pbc = dims, pbc
        from micmec_amd import units
        touching = np.zeros(len(used))
        np.add.at(touching, inverse.reshape(-1), 0.125 * CELL_MASS_AMU * units.amu)
        self.masses = touching

    def lattice(self):
        pos = self.node_ijk * self.spacing
        rvecs = np.diag(self.dims * self.spacing) if self.pbc else np.zeros((0, 3))
        return pos, rvecs

    def energy(self, pos, rvecs, params, D=None):
        """pos [N, 3], rvecs [3, 3], params {type: [(h0, Cv)]}; D deforms every edge."""
        from micmec_amd import units
        p = pos[self.sn]
        r = p - p[:, :1] + self.shift @ rvecs
        if D is not None:
            r = r @ D
        M = r[:, torch.tensor(HI)] - r[:, torch.tensor(LO)]            # [C, 8, 3, 3]
        if self.model == "original":
            M = M.mean(1, keepdim=True)
        total = 0.0
        for t, sel in self.sel.items():
            states, free, teff = params[t]
            kT = units.boltzmann * teff
            es = []
            for s, (h0, cv) in enumerate(states):
                B = torch.linalg.inv(h0) @ M[sel]
                eps = 0.5 * (B @ B.transpose(-1, -2) - torch.eye(3, dtype=torch.float64))
                e = torch.stack([eps[..., i, j] * (1.0 if i == j else 2.0) for i, j in VOIGT], -1)
                u = 0.5 * ((e @ cv) * e).sum(-1).mean(-1)
                es.append(torch.linalg.det(h0) * u + free[s])
            es = torch.stack(es, -1)
            total = total + (es if es.shape[-1] == 1
                             else -kT * torch.logsumexp(-es / kT, -1)).sum()
        return total

    def force(self, pos, rvecs, params=None):
        """Energy, node gradient and virial (numpy)."""
        x = torch.tensor(pos, requires_grad=True)
        D = torch.eye(3, dtype=torch.float64, requires_grad=True)
        rv = torch.from_numpy(np.array(rvecs)) if len(rvecs) else torch.zeros((3, 3),
                                                                              dtype=torch.float64)
        e = self.energy(x, rv, params or _plain_params(), D)
        g, v = torch.autograd.grad(e, [x, D])
        return e.item(), g.numpy(), v.t().numpy().copy()


def _parameters():
    """{type: [(h0, Cv)]} of TYPES in atomic units."""
    from micmec_amd import units
    out = {}
    for t, states in TYPES.items():
        out[t] = []
        for edge, (c11, c12, c44) in states:
            cv = np.zeros((6, 6))
            cv[:3, :3] = c12
            np.fill_diagonal(cv, [c11] * 3 + [c44] * 3)
            out[t].append((torch.from_numpy(edge * units.angstrom * np.identity(3)),
                           torch.from_numpy(cv * units.gigapascal)))
    return out


def _plain_params():
    return {t: (states, [0.0] * len(states), T_EFF) for t, states in _parameters().items()}


def _plain_system(shape, p_b, p_hole, pbc, rng, model, noise=0.05, strain=0.0):
    """The system that ``_system`` makes from the same generator."""
    plain = _Plain(_grid(shape, p_b, p_hole, rng), pbc, model)
    pos, rvecs = _noise(*plain.lattice(), rng, noise, strain)
    return plain, pos, rvecs


def _expm(A):
    w, Q = np.linalg.eigh(A)
    return (Q * np.exp(w)) @ Q.T


def _exact_md(case, seed):
    from micmec_amd import units
    rng = np.random.default_rng(seed)
    plain, x, rv = _plain_system(_shape(case), case["p_b"], case["p_hole"], case["pbc"], rng,
                                 "corner8")
    m = plain.masses
    st = _md_start(m, x, not case["pbc"], rng)
    dt, kT, v = units.femtosecond, units.boltzmann * 300.0, st["vel"]
    nvt, npt = case["ensemble"] != "nve", case["ensemble"] == "npt"
    ndof = st["ndof"] if nvt else x.size
    Q, xi_v, W, vg = st["chain_mass"], st["chain"].copy(), st["mass_press"], st["vel_press"]
    xi = np.zeros(3)
    mm = m[:, None]
    ekin = 0.0
    svv = np.zeros((3, 3))

    def sums():
        nonlocal ekin, svv
        svv = v.T @ (mm * v)
        ekin = 0.5 * np.trace(svv)

    def chain():
        """Half a step of the Nose-Hoover chain; the velocities are scaled by its factor."""
        nonlocal v, xi, ekin, svv
        g1 = W * (vg ** 2).sum() - 6 * kT if npt else 0.0

        def bead(k, e):
            g = (2 * e - ndof * kT + g1 if k == 0 else Q[k - 1] * xi_v[k - 1] ** 2 - kT) / Q[k]
            f = np.exp(-xi_v[k + 1] * dt / 8) if k < 2 else 1.0
            xi_v[k] = (xi_v[k] * f + g * dt / 4) * f
        for k in (2, 1, 0):
            bead(k, ekin)
        xi = xi + xi_v * dt / 2
        f = np.exp(-xi_v[0] * dt / 2)
        v, ekin, svv = v * f, ekin * f * f, svv * f * f
        for k in (0, 1, 2):
            bead(k, ekin)

    def barostat():
        """Half a step of the cell: its velocity, positions and cell, velocities, and again."""
        nonlocal x, v, rv, vg, epot, g, vt
        damp = np.exp(-dt * xi_v[0] / 8)

        def kick():
            nonlocal vg
            G = svv - vt
            G = 0.5 * (G + G.T) + (2 * ekin / ndof
                                   - units.bar * abs(np.linalg.det(rv))) * np.identity(3)
            vg = (vg * damp + G / W * dt / 4) * damp
        kick()
        R = _expm(vg * dt / 2)
        x, rv = x @ R, rv @ R
        epot, g, vt = plain.force(x, rv)
        v = v @ _expm(-(vg + np.trace(vg) / ndof * np.identity(3)) * dt / 2)
        sums()
        kick()

    epot, g, vt = plain.force(x, rv)
    sums()
    for _ in range(case["steps"]):
        if npt:
            barostat()
        if nvt:
            chain()
        v = v - 0.5 * dt * g / mm
        x = x + dt * v
        epot, g, vt = plain.force(x, rv)
        v = v - 0.5 * dt * g / mm
        sums()
        if nvt:
            chain()
        if npt:
            barostat()
    return dict(pos=x, vel=v, gpos=g, vtens=vt, rvecs=np.array(rv),
                scalars=np.array([epot, ekin, epot + ekin]), econs=None)


def _exact_differentiated(case, seed):
    """The loss (or weighted sum) and its gradients, one configuration at a time."""
    rng = np.random.default_rng(seed)
    n, count = case["n"], case["count"]
    systems = [_plain_system((n, n, n), case["p_b"], 0.0, True, rng, case["model"], 0.1, 0.03)
               for _ in range(count)]
    ids = [t for t in (1, 2) if any(t in s[0].sel for s in systems)]
    table = _parameters()
    S = max(len(table[t]) for t in ids)
    cv = torch.zeros((len(ids), S, 6, 6), dtype=torch.float64)
    h0 = torch.eye(3, dtype=torch.float64).repeat(len(ids), S, 1, 1)
    for r, t in enumerate(ids):
        for s, (h, c) in enumerate(table[t]):
            h0[r, s], cv[r, s] = h, c
    free = torch.zeros((len(ids), S), dtype=torch.float64)
    teff = torch.full((len(ids),), T_EFF, dtype=torch.float64)

    def params(cv, h0, free, teff):
        return {t: ([(h0[r, s], cv[r, s]) for s in range(len(table[t]))], free[r], teff[r])
                for r, t in enumerate(ids)}

    def outputs(s, x, rv, p):
        D = torch.eye(3, dtype=torch.float64, requires_grad=True)
        e = s.energy(x, rv, p, D)
        g, v = torch.autograd.grad(e, [x, D], create_graph=True)
        return e, g, v.t()

    inputs = [(s, torch.from_numpy(x).requires_grad_(True),
               torch.from_numpy(rv).requires_grad_(True)) for s, x, rv in systems]
    nodes = sum(len(x) for _, x, _ in inputs)
    if case["kind"] == "fit":
        target = params(cv * torch.from_numpy(_cv_noise(cv.shape, rng)), h0, free, teff)
        want = [[t.detach() for t in outputs(*i, target)] for i in inputs]
        vol = [abs(torch.linalg.det(rv.detach())) for _, _, rv in inputs]
        f_scale = sum((g ** 2).sum() for _, g, _ in want) / (3 * nodes)
        s_scale = sum(((v / V) ** 2).sum() for (_, _, v), V in zip(want, vol)) / (9 * count)
        a = torch.zeros_like(cv, requires_grad=True)
        b = torch.zeros_like(h0, requires_grad=True)
        total = 0.0
        for i, (_, gt, vt), V in zip(inputs, want, vol):
            now = params(cv * (1.0 + 0.5 * (a + a.transpose(-1, -2))), h0 * (1.0 + b), free, teff)
            _, g, v = outputs(*i, now)
            loss = ((g - gt) ** 2).sum() / (3 * nodes) / f_scale \
                + (((v - vt) / V) ** 2).sum() / (9 * count) / s_scale
            loss.backward()
            total += loss.item()
        return dict(loss=np.float64(total), a=a.grad, b=b.grad)
    wE, wG, wV = [torch.from_numpy(w) for w in _cotangents(count, (nodes, 3), rng)]
    leaves = [t.clone().requires_grad_(True) for t in (cv, h0, free, teff)]
    got, at = [], 0
    for k, i in enumerate(inputs):
        e, g, v = outputs(*i, params(*leaves))
        ((wE[k] * e) + (wG[at:at + len(g)] * g).sum() + (wV[k] * v).sum()).backward()
        got.append((e.detach(), g.detach(), v.detach()))
        at += len(g)
    grad = [leaves[0].grad, leaves[1].grad, leaves[2].grad, leaves[3].grad]
    grad[0] = 0.5 * (grad[0] + grad[0].transpose(-1, -2))
    return dict(energy=torch.stack([x[0] for x in got]), gpos=torch.cat([x[1] for x in got]),
                vtens=torch.stack([x[2] for x in got]),
                grads=[torch.cat([x.grad for _, x, _ in inputs]),
                       torch.stack([rv.grad for _, _, rv in inputs])] + grad)


def exact(case, seed):
    """The outputs of ``run`` on a new state. None where the draws are the framework's own
    (Langevin noise, the replicas' start), where they depend on a search's trials, and where
    plain torch takes too long."""
    kind = case["kind"]
    if kind in ("batch", "relax") or case.get("ensemble") == "langevin":
        return None
    if kind in ("fit", "grad"):
        return _exact_differentiated(case, seed)
    cells = case["nx"] * case["ny"] * case["nz"]
    if kind == "md":
        evals = case["steps"] * (3 if case["ensemble"] == "npt" else 1)
        return _exact_md(case, seed) if evals * (cells + 2000) < 2e6 else None
    rng = np.random.default_rng(seed)
    plain, pos, rvecs = _plain_system(_shape(case), case["p_b"], case["p_hole"], case["pbc"], rng,
                                      case["model"], 0.1, 0.02)
    e, g, v = plain.force(pos, rvecs)
    e = np.array([e]) if case["where"] == "device" else np.float64(e)
    return dict(energy=e, gpos=g, vtens=v) if case["gradient"] else dict(energy=e)
