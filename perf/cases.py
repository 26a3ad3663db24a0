"""The work that users of this framework have it do, as measurable cases.

Kinds of work (the values of a case's "kind"):

  md        LJSystem.run: a block of velocity-Verlet (NVE) or Langevin (NVT) steps of a plain
            Lennard-Jones liquid or gas, one type or a two-type mixture
  actions   LJSystem.run with energy records: the same loop action by action, the form of the
            reference's examples and of C++ programs on the drop-in headers
  evaluate  exchange, ghosts, Verlet list, forces, energy and virial of a given configuration
  adress    AdResSSystem.run: a block of steps of the LJ / ideal-gas AdResS slab
  ensemble  Ensemble.run: a block of steps of many replicas, then their frame and energies
  fit       force matching: LJForce forward and backward (forces and their adjoint)

Starts are liquids: a small box is melted by plain torch dynamics and repeated in space, and
every atom draws its own velocity and a small displacement, so that neighbour counts, list
lifetimes and velocities are those of a running simulation.  Everything is FP64, the only
precision the framework computes in.
"""
import ctypes
import math

import numpy as np
import torch

RC, DT = 2.5, 0.005

# ------------------------------------------------------------------------------------------
# the cases


def listed():
    return [
        # the smallest calls: the 4,000-atom NVE system, where launches and latency count
        dict(name="nve_4k", kind="md", atoms=4000, density=0.8442, temperature=0.72, nvt=False, permute=False,
             cap=0.0, types=1, skin=0.3, steps=50),
        # an argon-like gas of odd size with a thin skin and the capped potential, NVE
        dict(name="nve_gas_62k", kind="md", atoms=61731, density=0.35, temperature=1.2, nvt=False, permute=False,
             cap=0.7, types=1, skin=0.1, steps=30),
        # an ordinary liquid, Langevin, atoms kept in cell order
        dict(name="nvt_256k", kind="md", atoms=256000, density=0.8442, temperature=1.0, nvt=True, permute=True,
             cap=0.0, types=1, skin=0.3, steps=20),
        # the headline throughput system: 4,000,000 atoms, Langevin, atoms kept in cell order
        dict(name="nvt_4m", kind="md", atoms=4000000, density=0.8442, temperature=1.0, nvt=True, permute=True,
             cap=0.0, types=1, skin=0.3, steps=20),
        # a two-type mixture (80/20, Lorentz-Berthelot) as sampled for force matching
        dict(name="mixture_32k", kind="md", atoms=32000, density=0.8, temperature=1.0, nvt=True, permute=False,
             cap=0.0, types=2, skin=0.3, steps=20),
        # the example program's loop: one call per action, energies recorded on the way
        dict(name="actions_108k", kind="actions", atoms=108001, density=0.7, temperature=1.0, nvt=False,
             permute=True, cap=0.0, types=1, skin=0.3, steps=10),
        # one configuration scored from scratch: the neighbour list dominates
        dict(name="evaluate_500k", kind="evaluate", atoms=500009, density=0.8442, temperature=1.0, nvt=False,
             permute=False, cap=0.0, types=1, skin=0.3, steps=1),
        # the AdResS slab of 160,000 molecules in a 200 x 40 x 40 box
        dict(name="adress_160k", kind="adress", atoms=160000, density=0.5, temperature=1.0, cap=0.7, skin=0.3,
             steps=20),
        # a small slab of odd size
        dict(name="adress_21k", kind="adress", atoms=21277, density=0.6, temperature=1.0, cap=0.7, skin=0.3,
             steps=20),
        # the 256-replica ensemble, a frame read every 100 steps
        dict(name="ensemble_256", kind="ensemble", replicas=256, smallest=500, largest=50000, steps=100),
        # a parameter sweep over a few small replicas
        dict(name="ensemble_24", kind="ensemble", replicas=24, smallest=500, largest=3000, steps=100),
        # one force-matching evaluation of a 32,000-atom mixture: forces and their adjoint
        dict(name="fit_32k", kind="fit", atoms=32000, density=0.8, temperature=1.0, types=2, skin=0.3, cap=0.0),
    ]


def draw(rng):
    def log(lo, hi):
        return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))

    kind = rng.choice(["md", "md", "md", "actions", "evaluate", "adress", "ensemble", "fit"])
    density, temperature = round(rng.uniform(0.3, 0.9), 4), round(rng.uniform(0.7, 1.5), 4)
    skin = rng.choice([0.1, 0.3, 0.3])
    if kind == "ensemble":
        smallest = log(500, 4000)
        return dict(kind=kind, replicas=log(8, 128), smallest=smallest, largest=smallest * rng.randint(2, 10),
                    steps=100)
    if kind == "adress":
        return dict(kind=kind, atoms=log(12000, 300000), density=round(rng.uniform(0.35, 0.8), 4),
                    temperature=temperature, cap=0.7, skin=skin, steps=rng.randint(10, 25))
    if kind == "fit":
        return dict(kind=kind, atoms=log(4000, 100000), density=round(rng.uniform(0.6, 0.85), 4),
                    temperature=temperature, types=rng.choice([1, 2]), skin=skin, cap=0.0)
    case = dict(kind=kind, atoms=log(3000, 1500000 if kind == "md" else 600000), density=density,
                temperature=temperature, nvt=rng.random() < 0.5, permute=rng.random() < 0.5,
                cap=rng.choice([0.0, 0.0, 0.7]), types=rng.choice([1, 1, 2]), skin=skin, steps=1)
    if kind == "md":
        case["steps"] = rng.randint(15, 30)
    if kind == "actions":
        case["steps"] = rng.randint(6, 12)
    return case


def tolerance(case):
    # Sums of some 50 FP64 pair terms in another order differ by 1e-15 to 1e-14 of a force;
    # a block of steps multiplies that by the growth of neighbouring trajectories.  The
    # AdResS partners' forces and the density sums arrive by atomics, in any order.
    # Against exact(): evaluate and fit up to 7e-15 (largest value 3e-13), blocks of steps up
    # to 5e-14 (1.4e-12); ensembles, 200 steps with the start's, 1.2e-10 (4e-8 at 110,000
    # atoms, growing with their number).
    if case["kind"] in ("evaluate", "fit"):
        return {"rel": 4e-14, "max": 2e-12}
    if case["kind"] == "ensemble":
        return {"rel": 5e-10, "max": 2e-7}
    return {"rel": 2e-13, "max": 8e-12}


def work(case):
    """One pass: every atom's position, velocity and force read and written once per step, a
    partner index (2 B) per list entry read per step and written once per list, 24 FLOP per
    pair inside the cutoff and 8 per other listed pair, each pair once."""
    if case["kind"] == "ensemble":
        sizes = _ensemble_parameters(case, 0)
        n = float(sum(r["n"] for r in sizes))
        density = sum(r["n"] * r["density"] for r in sizes) / n
        skin, steps = 0.3, case["steps"]
    else:
        n, density, skin = float(case["atoms"]), case["density"], case["skin"]
        steps = case.get("steps", 1)
    share = 0.25 if case["kind"] == "adress" else (0.6 if case["kind"] == "ensemble" else 1.0)
    listed_pairs = 0.5 * n * share * density * 4.0 / 3.0 * math.pi * (RC + skin) ** 3
    pairs = listed_pairs * (RC / (RC + skin)) ** 3
    force_flops = 8.0 * listed_pairs + 24.0 * pairs
    if case["kind"] == "fit":
        # positions and upstream in, forces and gradients out; forward and adjoint pair terms
        return {"bytes": n * 4 * 24.0 + 4.0 * listed_pairs, "flops": 3.0 * force_flops}
    if case["kind"] == "evaluate":
        return {"bytes": n * 72.0 + 4.0 * listed_pairs, "flops": force_flops + 8.0 * 3.0 * listed_pairs}
    return {"bytes": steps * (n * 136.0 + 2.0 * listed_pairs), "flops": steps * force_flops}


# ------------------------------------------------------------------------------------------
# starting configurations (plain torch, made from the seed alone)

_DEVICE = "cuda" if torch.cuda.is_available() else "cpu"
_MIX_EPS, _MIX_SIGMA = (1.0, 0.5), (1.0, 0.88)


def _generator(seed, salt):
    g = torch.Generator(device=_DEVICE)
    g.manual_seed((int(seed) * 1000003 + salt) % (1 << 62))
    return g


def _lattice(n, box, g):
    """n sites of a simple cubic lattice that fills the box, each moved by up to 4 % of the
    lattice spacing"""
    box = torch.as_tensor(box, dtype=torch.float64, device=_DEVICE)
    spacing = float((box.prod() / n) ** (1.0 / 3.0))
    while True:
        cells = [max(1, int(float(e) / spacing)) for e in box]
        if cells[0] * cells[1] * cells[2] >= n:
            break
        spacing *= 0.995
    sites = torch.randperm(cells[0] * cells[1] * cells[2], generator=g, device=_DEVICE)[:n].sort().values
    ijk = torch.stack([sites // (cells[1] * cells[2]), sites // cells[2] % cells[1], sites % cells[2]], 1)
    edge = box / torch.tensor(cells, dtype=torch.float64, device=_DEVICE)
    jitter = (torch.rand((n, 3), generator=g, device=_DEVICE, dtype=torch.float64) - 0.5) * 0.08
    return (ijk + 0.5 + jitter) * edge


def _melt(n, box, temperature, g, steps=500):
    """a liquid of n atoms: a lattice run for `steps` strongly thermostatted steps with the
    pair force softened below 0.8 sigma"""
    box = torch.as_tensor(box, dtype=torch.float64, device=_DEVICE)
    x = _lattice(n, box, g)

    def normal():
        return torch.randn((n, 3), generator=g, device=_DEVICE, dtype=torch.float64)

    v = normal() * math.sqrt(2.0 * temperature)
    away = torch.eye(n, device=_DEVICE, dtype=torch.float64) * 1e6
    damping = math.exp(-2.0 * DT)
    for _ in range(steps):
        d = x[:, None, :] - x[None, :, :]
        d = d - box * torch.round(d / box)
        r2 = (d * d).sum(2) + away
        f2 = 1.0 / r2.clamp(min=0.64)
        f6 = f2 * f2 * f2
        ff = torch.where(r2 <= RC * RC, (48.0 * f6 * f6 - 24.0 * f6) * f2, 0.0)
        v = v + DT * (ff[:, :, None] * d).sum(1)
        v = v * damping + math.sqrt(temperature * (1.0 - damping * damping)) * normal()
        x = x + DT * v
    return x - box * torch.floor(x / box)


def _liquid(case, seed):
    """(positions, velocities, types, box edges) of a single-system case: a melted box
    repeated along the axes, then single atoms taken out to reach the exact count"""
    n, density = case["atoms"], case["density"]
    g = _generator(seed, 1)
    stretch = 5 if case["kind"] == "adress" else 1  # Lx : Ly : Lz = 5 : 1 : 1 for the slab
    k = max(1, round((n / stretch / 500.0) ** (1.0 / 3.0)))
    copies = (stretch * k, k, k)
    total = copies[0] * copies[1] * copies[2]
    base = -(-n // total)
    edge = (base / density) ** (1.0 / 3.0)
    # vacancies are spread over the whole box, which is scaled to the exact density
    edge *= (n / (base * total)) ** (1.0 / 3.0)
    x = _melt(base, [edge] * 3, case["temperature"], g)
    shift = torch.stack(torch.meshgrid(*[torch.arange(c, device=_DEVICE) for c in copies], indexing="ij"), -1)
    x = (shift.reshape(-1, 1, 3) * edge + x[None]).reshape(-1, 3)
    keep = torch.randperm(x.shape[0], generator=g, device=_DEVICE)[:n].sort().values
    x = x[keep]
    box = torch.tensor([c * edge for c in copies], dtype=torch.float64, device=_DEVICE)
    x = x + 0.04 * (torch.rand(x.shape, generator=g, device=_DEVICE, dtype=torch.float64) - 0.5)
    x = x - box * torch.floor(x / box)
    x = torch.where(x >= box, torch.zeros_like(x), x)
    v = torch.randn(x.shape, generator=g, device=_DEVICE, dtype=torch.float64) * math.sqrt(case["temperature"])
    v = v - v.mean(0)
    types = torch.zeros(n, dtype=torch.int64, device=_DEVICE)
    if case.get("types", 1) == 2:
        types = (torch.rand(n, generator=g, device=_DEVICE) < 0.2).to(torch.int64)
    return x, v, types, box


def _pair_tables(case):
    """row-major sigma and epsilon tables of the case's types"""
    if case.get("types", 1) == 1:
        return [1.0], [1.0]
    (ea, eb), (sa, sb) = _MIX_EPS, _MIX_SIGMA
    return [sa, 0.5 * (sa + sb), 0.5 * (sa + sb), sb], [ea, math.sqrt(ea * eb), math.sqrt(ea * eb), eb]


def _slab_table(box, density):
    """a converged thermodynamic force on 1-sigma bins: smooth, odd about the slab's centre,
    acting in the hybrid regions"""
    length = float(box[0])
    nbins = math.ceil(length)
    x = (np.arange(nbins) + 0.5) * (length / nbins) - 0.5 * length
    at, hy = 0.075 * length, 0.05 * length
    inside = (np.abs(x) > at) & (np.abs(x) < at + hy)
    return np.where(inside, np.sign(x) * 2.0 * density * np.sin(math.pi * (np.abs(x) - at) / hy), 0.0)


def _ensemble_parameters(case, seed):
    """per replica: atoms (log-uniform), density, temperature, AdResS or plain (the first
    half are slabs), box edges; the counts belong to the case, not to the seed"""
    from random import Random
    r = Random(2024 + case["replicas"])
    out = []
    for k in range(case["replicas"]):
        n = int(round(math.exp(r.uniform(math.log(case["smallest"]), math.log(case["largest"])))))
        density, temperature = r.uniform(0.3, 0.9), r.uniform(0.7, 1.5)
        adress = k < case["replicas"] // 2
        volume, low = n / density, 2.0 * (RC + 0.3) + 1e-6
        short = max((volume / (5.0 if adress else 1.0)) ** (1.0 / 3.0), low)
        box = [max(volume / (short * short), low), short, short] if adress else [short] * 3
        out.append(dict(n=n, density=density, temperature=temperature, adress=adress, box=box,
                        seed=int(seed) * 1000 + k))
    return out


# ------------------------------------------------------------------------------------------
# the framework's side

_context = None


def _ctx():
    global _context
    if _context is None:
        import mrmd_amd
        _context = mrmd_amd.Context(0)
    return _context


class _DeviceArray:
    """device memory of the library as torch sees it; keeps its owner alive"""

    def __init__(self, owner, ptr, shape, strides):
        self.owner = owner
        self.__cuda_array_interface__ = dict(shape=shape, strides=strides, typestr="<f8", data=(ptr, False), version=3)


def _view(state, field):
    """the local atoms' positions (n x 3), velocities or forces (3 x n), in place"""
    from mrmd_amd import POS, _L
    atoms = state["system"].atoms
    n = state["n"]
    ptr, stride = ctypes.c_void_p(), ctypes.c_int64()
    atoms.ctx.check(_L.mrmd_atoms_device_ptr(atoms.h, field, ctypes.byref(ptr), ctypes.byref(stride)))
    key = (field, ptr.value, stride.value)
    if key not in state["views"]:
        array = (_DeviceArray(atoms, ptr.value, (n, 3), (32, 8)) if field == POS
                 else _DeviceArray(atoms, ptr.value, (3, n), (8 * stride.value, 8)))
        state["views"][key] = torch.as_tensor(array, device="cuda")
        state["views"][key].owner = atoms  # the memory outlives the view, also without the state
    return state["views"][key]


def prepare(case, seed):
    from mrmd_amd.adjoint import Snapshot, make_force_function
    from mrmd_amd.drivers import AdResSSystem, LJSystem
    from mrmd_amd.ensemble import Ensemble, replica
    ctx = _ctx()
    if case["kind"] == "ensemble":
        parameters = _ensemble_parameters(case, seed)
        reps = [replica(p["n"], p["box"], p["temperature"], p["seed"], adress=p["adress"]) for p in parameters]
        ensemble = Ensemble(ctx, reps, RC, 0.3)
        ensemble.set_lj(cap=0.7)
        x, v = _ensemble_start(parameters, seed)
        ensemble.upload(0, x.cpu().numpy())
        ensemble.upload(1, v.cpu().numpy())
        ensemble.run(100, 10)
        return dict(case=case, ensemble=ensemble)
    x, v, types, box = _liquid(case, seed)
    edges = box.cpu().numpy()
    if case["kind"] == "fit":
        sigma, eps = _pair_tables(case)
        pos = x.cpu().numpy()
        snap = Snapshot(ctx, pos, types.cpu().numpy(), float(edges[0]), case["types"], np.array(eps),
                        np.array(sigma), RC, case["skin"])
        up = torch.randn(x.shape, generator=_generator(seed, 2), device=_DEVICE, dtype=torch.float64).cpu()
        leaves = [torch.from_numpy(pos).requires_grad_(), torch.tensor(eps, dtype=torch.float64, requires_grad=True),
                  torch.tensor(sigma, dtype=torch.float64, requires_grad=True)]
        return dict(case=case, snap=snap, function=make_force_function(), leaves=leaves, up=up)
    if case["kind"] == "adress":
        length = float(edges[0])
        system = AdResSSystem(ctx, x.cpu().numpy(), v.cpu().numpy(), edges, 0.15 * length, 0.05 * length, 1, rc=RC,
                              skin=case["skin"], cap=case["cap"], temperature=case["temperature"], seed=seed)
        system.tf.set_force(_slab_table(edges, case["density"])[:, None])
    else:
        sigma, eps = _pair_tables(case)
        system = LJSystem(ctx, x.cpu().numpy(), v.cpu().numpy(), edges, rc=RC, skin=case["skin"],
                          sigma=np.array(sigma), epsilon=np.array(eps), cap=case["cap"], shifted=True,
                          langevin=case["nvt"], gamma=1.0, temperature=case["temperature"], seed=seed,
                          permute=case["permute"], types=types.cpu().numpy(), num_types=case["types"],
                          type_stride=case["types"])
    return dict(case=case, system=system, n=case["atoms"], views={})


def run(state):
    from mrmd_amd import FORCE, POS, VEL
    case, kind = state["case"], state["case"]["kind"]
    if kind == "ensemble":
        ensemble = state["ensemble"]
        ensemble.run(case["steps"], 10)
        potential, kinetic = ensemble.energies()
        return dict(positions=ensemble.download(POS), velocities=ensemble.download(VEL), potential=potential,
                    kinetic=kinetic)
    if kind == "fit":
        pos, eps, sigma = state["leaves"]
        forces = state["function"].apply(pos, eps, sigma, state["snap"])
        grads = torch.autograd.grad(forces, (pos, eps, sigma), state["up"])
        return dict(forces=forces.detach(), pos=grads[0], epsilon=grads[1], sigma=grads[2])
    system = state["system"]
    out = {}
    if kind == "evaluate":
        system.rebuild()
        system.atoms.set_force(0.0)
        system.lj.apply(system.atoms, system.vl)
        system.ghosts.contribute_back_ghost_to_real(system.atoms)
        out["energy_virial"] = np.array(system.lj.energy_virial())
        out["forces"] = _view(state, FORCE)
        return out
    if kind == "actions":
        out["energies"] = system.run(case["steps"], DT, energy_every=2)
    else:
        system.run(case["steps"], DT)
    out["positions"], out["velocities"], out["forces"] = (_view(state, f) for f in (POS, VEL, FORCE))
    if kind == "adress":
        out["energy"] = np.float64(system.energy)
    return out


def _ensemble_start(parameters, seed):
    g = _generator(seed, 3)
    x = torch.cat([_lattice(p["n"], p["box"], g) for p in parameters])
    v = []
    for p in parameters:
        w = torch.randn((p["n"], 3), generator=g, device=_DEVICE, dtype=torch.float64) * math.sqrt(p["temperature"])
        v.append(w - w.mean(0))
    return x, torch.cat(v)


# ------------------------------------------------------------------------------------------
# the same work in plain torch, FP64


def _philox(c0, c1, c2, c3, k0, k1):
    """Philox4x32-10 (Salmon et al., SC'11) on int64 tensors that hold 32-bit words"""
    low = 0xFFFFFFFF
    for _ in range(10):
        p0, p1 = c0 * 0xD2511F53, c2 * 0xCD9E8D57
        c0, c1, c2, c3 = ((p1 >> 32) & low) ^ c1 ^ k0, p1 & low, ((p0 >> 32) & low) ^ c3 ^ k1, p0 & low
        k0, k1 = (k0 + 0x9E3779B9) & low, (k1 + 0xBB67AE85) & low
    return c0, c1, c2, c3


def _noise(seed, index, call):
    """the Langevin noise: three normals per atom, Philox words keyed by (seed, atom, call) in
    Marsaglia's polar method, accepted pairs taken in the order of their rounds"""
    n = index.shape[0]
    out = torch.zeros((n, 4), dtype=torch.float64, device=index.device)
    have = torch.zeros(n, dtype=torch.int64, device=index.device)
    todo, r = torch.arange(n, device=index.device), 0
    while todo.numel():
        i, s = index[todo], seed[todo]
        o = _philox(i, torch.full_like(i, call & 0xFFFFFFFF), torch.full_like(i, call >> 32), torch.full_like(i, r),
                    s & 0xFFFFFFFF, (s >> 32) & 0xFFFFFFFF)
        u, w = (((a << 20) ^ (b >> 12)).double().add(0.5).mul(2.0 ** -51).sub(1.0) for a, b in (o[:2], o[2:]))
        q = u * u + w * w
        ok = (q < 1.0) & (q > 0.0)
        f = torch.sqrt(-2.0 * torch.log(torch.where(ok, q, 0.5)) / torch.where(ok, q, 0.5))
        t, place = todo[ok], have[todo[ok]]
        out[t, 2 * place], out[t, 2 * place + 1] = (u * f)[ok], (w * f)[ok]
        have[t] += 1
        todo = todo[have[todo] < 2]
        r += 1
    return out[:, :3]


class _Reference:
    """periodic replicas advanced together; all arrays are per atom but box (per replica)"""

    def __init__(self, x, v, replica, box, types, tables, cap, skin, dt=DT, damping=None, sigma=None, seeds=None,
                 slabs=None, tf_every=0):
        self.x, self.v, self.rep, self.box, self.types = x, v, replica, box, types
        self.sigma_table, self.eps_table = (torch.tensor(t, dtype=torch.float64, device=x.device) for t in tables)
        self.nt = int(round(math.sqrt(self.sigma_table.numel())))
        self.cap, self.skin, self.dt = cap, skin, dt
        self.damping, self.noise_sigma, self.seeds = damping, sigma, seeds
        self.slabs, self.tf_every = slabs, tf_every  # slabs: dict of per-replica tensors and tables
        self.f = torch.zeros_like(x)
        self.index = torch.arange(x.shape[0], device=x.device)
        self.index = self.index - torch.cat([torch.zeros(1, dtype=torch.int64, device=x.device),
                                             torch.bincount(replica).cumsum(0)[:-1]])[replica]
        self.moved = torch.full((box.shape[0],), float("inf"), dtype=torch.float64, device=x.device)
        self.since, self.rows, self.steps = float("inf"), None, 0

    # ---- neighbour rows of radius RC + 0.5, remade when an atom may have moved 0.25
    def neighbours(self):
        radius = RC + 0.5
        x, box = self.x, self.box
        n, dev = x.shape[0], x.device
        w = x - box[self.rep] * torch.floor(x / box[self.rep])
        cells = torch.clamp((box / radius).floor().long(), min=1)
        count = cells.prod(1)
        first = torch.cat([torch.zeros(1, dtype=torch.int64, device=dev), count.cumsum(0)[:-1]])
        ijk = torch.minimum((w / (box / cells)[self.rep]).long(), cells[self.rep] - 1)
        c = first[self.rep] + (ijk[:, 0] * cells[self.rep, 1] + ijk[:, 1]) * cells[self.rep, 2] + ijk[:, 2]
        order = torch.argsort(c, stable=True)
        occupied = torch.bincount(c, minlength=int(count.sum()))
        start = occupied.cumsum(0) - occupied
        width = int(occupied.max())
        place = torch.arange(n, device=dev) - start[c[order]]
        table = torch.full((occupied.numel(), width), -1, dtype=torch.int32, device=dev)
        table[c[order], place] = order.to(torch.int32)
        offsets = torch.tensor([(a, b, d) for a in (-1, 0, 1) for b in (-1, 0, 1) for d in (-1, 0, 1)], device=dev)
        kept, most = [], 0
        chunk = max(1024, int(1.5e8) // (27 * width))
        for lo in range(0, n, chunk):
            i = order[lo:lo + chunk]
            nc = cells[self.rep[i]][:, None, :]
            # an axis of two cells has one neighbour cell, an axis of one cell none
            ok = ((offsets[None] != -1) | (nc > 2)) & ((offsets[None] != 1) | (nc > 1))
            k = (ijk[i][:, None, :] + offsets[None]) % nc
            cell = first[self.rep[i]][:, None] + (k[..., 0] * nc[..., 1] + k[..., 1]) * nc[..., 2] + k[..., 2]
            j = torch.where(ok.all(2)[..., None], table[cell], -1).reshape(i.numel(), -1)
            near = j >= 0
            jj = j.clamp(min=0).long()
            r2 = torch.zeros(j.shape, dtype=torch.float64, device=dev)
            for d in range(3):
                e = box[self.rep[i], d][:, None]
                t = x[i, d][:, None] - x[jj, d]
                r2 += (t - e * torch.round(t / e)) ** 2
            near &= (r2 <= radius * radius) & (jj != i[:, None])
            del r2, jj
            cnt = near.sum(1)
            m = int(cnt.max())
            rank = near.cumsum(1) - 1
            r = torch.full((i.numel(), max(m, 1)), -1, dtype=torch.int32, device=dev)
            a, b = near.nonzero(as_tuple=True)
            r[a, rank[a, b]] = j[a, b]
            kept.append((i, r))
            most = max(most, m)
        self.rows, self.since = kept, 0.0

    def weights(self):
        s = self.slabs
        one, zero = torch.ones_like(self.x[:, 0]), torch.zeros_like(self.x[:, 0])
        if s is None:
            return one, one, zero
        half, hy = 0.5 * s["at"][self.rep], s["hy"][self.rep]
        dx = self.x[:, 0] - s["centre"][self.rep]
        far = dx.abs()
        arg = math.pi / (2.0 * hy) * (far - half)
        base, hybrid = torch.cos(arg), (far >= half) & (far <= half + hy)
        lam = torch.where(far < half, one, torch.where(hybrid, base * base, zero))
        grad = torch.where(hybrid, -math.pi / (2.0 * hy) * 2.0 * torch.sin(arg) * base / far * dx, zero)
        plain = ~s["adress"][self.rep]
        return torch.where(plain, one, lam), torch.where(plain, one, lam), torch.where(plain, zero, grad)

    def forces(self):
        """pair forces, energy per replica and virial; with slabs the weighted forces, the
        drift and the compensation terms of LJ_IdealGas"""
        if self.since >= 0.25:
            self.neighbours()
        lam, mod, grad = self.weights()
        f = torch.zeros_like(self.x)
        e_atom, w_atom, e_plain = (torch.zeros_like(self.x[:, 0]) for _ in range(3))
        shift_f2 = (self.sigma_table / RC) ** 6
        shift = 4.0 * self.eps_table * (shift_f2 * shift_f2 - shift_f2)
        for i, rows in self.rows:
            step = max(1, int(4e7) // max(rows.shape[1], 1))
            for lo in range(0, i.numel(), step):
                ii, j = i[lo:lo + step], rows[lo:lo + step]
                jj = j.clamp(min=0).long()
                d, r2 = [], 0.0
                for a in range(3):
                    e = self.box[self.rep[ii], a][:, None]
                    t = self.x[ii, a][:, None] - self.x[jj, a]
                    t = t - e * torch.round(t / e)
                    d.append(t)
                    r2 = r2 + t * t
                inside = (j >= 0) & (r2 <= RC * RC)
                if self.slabs is not None:
                    inside &= (mod[ii][:, None] > 0.0) | (mod[jj] > 0.0)
                r2 = torch.where(inside, r2, 1.0)
                t = self.types[ii][:, None] * self.nt + self.types[jj]
                sig, eps = self.sigma_table[t], self.eps_table[t]
                f6 = (sig * sig / r2) ** 3
                ff = eps * (48.0 * f6 * f6 - 24.0 * f6) / r2
                en = 4.0 * eps * (f6 * f6 - f6) - shift[t]
                if self.cap > 0.0:
                    c6 = (sig / self.cap) ** 6
                    slope = eps * (48.0 * c6 * c6 - 24.0 * c6) / self.cap
                    r = torch.sqrt(r2)
                    below = r2 < self.cap * self.cap
                    ff = torch.where(below, slope / r, ff)
                    en = torch.where(below, 4.0 * eps * (c6 * c6 - c6) - (r - self.cap) * slope - shift[t], en)
                ff, en = torch.where(inside, ff, 0.0), torch.where(inside, en, 0.0)
                w = 0.5 * (mod[ii][:, None] + mod[jj]) if self.slabs is not None else 1.0
                for a in range(3):
                    f[ii, a] = (d[a] * ff * w).sum(1)
                e_atom[ii] = 0.5 * (en * w).sum(1)
                e_plain[ii] = 0.5 * en.sum(1)
                w_atom[ii] = -0.25 * (ff * r2).sum(1)
        if self.slabs is not None:
            f[:, 0] += self.drift(lam, mod, grad, e_plain)
        self.f = f
        energy = torch.zeros(self.box.shape[0], dtype=torch.float64, device=f.device).index_add_(0, self.rep, e_atom)
        return energy, float(w_atom.sum())

    def drift(self, lam, mod, grad, v):
        """-V_i grad(lambda_i) and the mean compensation energy (200 lambda bins per replica,
        sampled every 200 calls, averaged in every 20,000)"""
        s = self.slabs
        hybrid = (mod > 0.0) & (mod < 1.0)
        cell = self.rep * 200 + (lam * 200.0).floor().long().clamp(0, 199)
        out = torch.where(hybrid, (s["mean"][cell] - v) * grad, 0.0)
        if s["calls"] % 200 == 0:
            s["comp"].index_add_(0, cell[hybrid], v[hybrid])
            s["count"].index_add_(0, cell[hybrid], torch.ones_like(v[hybrid]))
        if s["calls"] % 20000 == 0:
            some = s["count"] > 0.5
            s["mean"] = torch.where(some, (10.0 * s["mean"] + s["comp"] / s["count"].clamp(min=1.0)) / 11.0, s["mean"])
            s["comp"].zero_()
            s["count"].zero_()
        s["calls"] += 1
        return out

    def thermodynamic_force(self):
        """density sample on 1-sigma x-bins, update every tf_every steps, application"""
        s = self.slabs
        nbins, first = s["nbins"], s["first"]
        width = self.box[:, 0] / nbins
        bins = (self.x[:, 0] / width[self.rep]).floor().long()
        ok = s["adress"][self.rep] & (bins >= 0) & (bins < nbins[self.rep])
        cell = first[self.rep] + torch.where(ok, bins, 0)
        s["density"].index_add_(0, cell[ok], torch.ones_like(self.x[:, 0])[ok])
        s["samples"] += 1
        self.steps += 1
        if self.tf_every and self.steps % self.tf_every == 0:
            for r in range(nbins.numel()):
                if not bool(s["adress"][r]):
                    continue
                nb, a = int(nbins[r]), int(first[r])
                w, edge = float(width[r]), [float(t) for t in self.box[r]]
                rho = s["density"][a:a + nb].cpu().numpy() / (edge[1] * edge[2] * w * s["samples"])
                rho = 0.5 * (rho + rho[::-1])
                reach = np.arange(-int(6.0 / w), int(6.0 / w) + 1)
                kernel = np.exp(-((reach * w / 2.0) ** 2))
                at = (np.arange(nb)[:, None] + reach[None, :])
                at = np.where(at < 0, at + nb, np.where(at >= nb, at - nb, at))
                smooth = (rho[at] * kernel).sum(1) / kernel.sum()
                slope = (np.roll(smooth, -1) - np.roll(smooth, 1)) / (2.0 * w) / float(s["target"][r])
                far = np.abs((np.arange(nb) + 0.5) * w - float(s["centre"][r]))
                half, hy = 0.5 * float(s["at"][r]), float(s["hy"][r])
                slope = np.where((far >= half) & (far < half + hy), slope, 0.0)
                s["force"][a:a + nb] -= torch.from_numpy(slope).to(s["force"].device)
            s["density"].zero_()
            s["samples"] = 0
        self.f[:, 0] += torch.where(ok, s["force"][cell], 0.0)

    def wrap(self, which):
        """PeriodicMapping of the atoms of the replicas in `which`"""
        edge = self.box[self.rep]
        x = torch.where(self.x >= edge, (self.x - edge).clamp(min=0.0), self.x)
        up = x + edge
        x = torch.where(x < 0.0, torch.where(up >= edge, torch.zeros_like(x), up), x)
        self.x = torch.where(which[self.rep][:, None], x, self.x)

    def permute(self):
        """Atoms::permute by the linked cells of edge >= RC + skin (one system)"""
        n = torch.floor(self.box[0] * (1.0 / (RC + self.skin)))
        c = torch.minimum(torch.floor(self.x * (1.0 / (self.box[0] / n))), n - 1).long()
        n = n.long()
        order = torch.argsort((c[:, 0] * n[1] + c[:, 1]) * n[2] + c[:, 2], stable=True)
        self.x, self.v, self.types, self.f = self.x[order], self.v[order], self.types[order], self.f[order]
        self.since = float("inf")

    def step(self, call, permute=False):
        half = 0.5 * self.dt
        old = self.x
        v = self.v + half * self.f
        if self.damping is None:
            self.x = old + self.dt * v
        else:
            self.x = old + half * v
            v = v * self.damping[self.rep][:, None]
            v = v + self.noise_sigma[self.rep][:, None] * _noise(self.seeds[self.rep], self.index, call)
            self.x = self.x + half * v
        self.v = v
        r2 = ((old - self.x) ** 2).sum(1)
        far = torch.sqrt(torch.zeros_like(self.moved).scatter_reduce(0, self.rep, r2, "amax"))
        self.since += float(far.max())
        self.moved += far
        which = self.moved >= 0.5 * self.skin
        self.moved = torch.where(which, 0.0, self.moved)
        if bool(which.any()):
            self.wrap(which)
            if permute:
                self.permute()
        energy, virial = self.forces()
        if self.slabs is not None:
            self.thermodynamic_force()
        self.v = self.v + half * self.f
        return energy, virial


def _langevin(temperature, gamma=1.0, dt=DT):
    return math.exp(-gamma * dt), math.sqrt(temperature * (1.0 - math.exp(-2.0 * gamma * dt)))


def _slabs(box, adress, density, device):
    """the slab parameters of every replica: atomistic diameter 0.15 Lx, hybrid width 0.05 Lx"""
    box = box.to(device)
    nbins = torch.ceil(box[:, 0]).long()
    bins = int(nbins.sum())
    cells = box.shape[0] * 200
    zeros = lambda n: torch.zeros(n, dtype=torch.float64, device=device)  # noqa: E731
    return dict(at=0.15 * box[:, 0], hy=0.05 * box[:, 0], centre=0.5 * box[:, 0],
                adress=torch.tensor(adress, device=device), target=density, nbins=nbins,
                first=nbins.cumsum(0) - nbins, density=zeros(bins), force=zeros(bins), samples=0, mean=zeros(cells),
                comp=zeros(cells), count=zeros(cells), calls=0)


def exact(case, seed):
    if case["kind"] == "ensemble":
        return _exact_ensemble(case, seed)
    x, v, types, box = _liquid(case, seed)
    if case["kind"] == "fit":
        return _exact_fit(case, seed, x, types, box)
    n, dev = case["atoms"], x.device
    rep = torch.zeros(n, dtype=torch.int64, device=dev)
    tables = _pair_tables(case)
    options = {}
    if case.get("nvt") or case["kind"] == "adress":
        damping, sigma = _langevin(case["temperature"])
        options = dict(damping=torch.tensor([damping], dtype=torch.float64, device=dev),
                       sigma=torch.tensor([sigma], dtype=torch.float64, device=dev),
                       seeds=torch.tensor([seed], dtype=torch.int64, device=dev))
    if case["kind"] == "adress":
        density = n / float(np.prod(box.cpu().numpy()))
        slabs = _slabs(box[None], [True], torch.tensor([density]), dev)
        slabs["force"] += torch.from_numpy(_slab_table(box.cpu().numpy(), case["density"])).to(dev)
        options.update(slabs=slabs, tf_every=100)
    ref = _Reference(x, v, rep, box[None], types, tables, case["cap"], case["skin"], **options)
    if case["kind"] == "evaluate":
        ref.wrap(torch.ones(1, dtype=torch.bool, device=dev))
        if case["permute"]:
            ref.permute()
        energy, virial = ref.forces()
        return dict(energy_virial=np.array([float(energy), virial]), forces=ref.f.T.contiguous())
    records = []
    for k in range(case["steps"]):
        energy, virial = ref.step(k, case.get("permute", False))
        if case["kind"] == "actions" and k % 2 == 0:
            records.append((float(energy), 0.5 * float((ref.v ** 2).sum()), virial))
    out = dict(positions=ref.x, velocities=ref.v.T.contiguous(), forces=ref.f.T.contiguous())
    if case["kind"] == "actions":
        out["energies"] = np.array(records)
    if case["kind"] == "adress":
        out["energy"] = np.float64(float(energy))
    return out


def _exact_ensemble(case, seed):
    parameters = _ensemble_parameters(case, seed)
    if sum(p["n"] for p in parameters) > 150000:
        return None  # minutes of plain torch
    x, v = _ensemble_start(parameters, seed)
    dev = x.device
    rep = torch.cat([torch.full((p["n"],), k, dtype=torch.int64) for k, p in enumerate(parameters)]).to(dev)
    box = torch.tensor([p["box"] for p in parameters], dtype=torch.float64, device=dev)
    factors = torch.tensor([_langevin(p["temperature"]) for p in parameters], dtype=torch.float64, device=dev)
    target = torch.tensor([p["n"] / float(np.prod(p["box"])) for p in parameters])
    ref = _Reference(x, v, rep, box, torch.zeros_like(rep), ([1.0], [1.0]), 0.7, 0.3, damping=factors[:, 0],
                     sigma=factors[:, 1], seeds=torch.tensor([p["seed"] for p in parameters], device=dev),
                     slabs=_slabs(box, [p["adress"] for p in parameters], target, dev), tf_every=100)
    for k in range(100 + case["steps"]):
        energy, _ = ref.step(k)
    kinetic = torch.zeros_like(energy).index_add_(0, rep, 0.5 * (ref.v ** 2).sum(1))
    return dict(positions=ref.x, velocities=ref.v, potential=energy, kinetic=kinetic)


def _exact_fit(case, seed, x, types, box):
    up = torch.randn(x.shape, generator=_generator(seed, 2), device=_DEVICE, dtype=torch.float64)
    sigma, eps = _pair_tables(case)
    rep = torch.zeros(x.shape[0], dtype=torch.int64, device=x.device)
    ref = _Reference(x, torch.zeros_like(x), rep, box[None], types, (sigma, eps), 0.0, case["skin"])
    ref.neighbours()
    pairs = []
    for i, rows in ref.rows:
        a, b = ((rows >= 0) & (rows > i[:, None])).nonzero(as_tuple=True)
        pairs.append(torch.stack([i[a], rows[a, b].long()]))
    i, j = torch.cat(pairs, 1)
    pos = x.clone().requires_grad_()
    eps = torch.tensor(eps, dtype=torch.float64, device=x.device, requires_grad=True)
    sigma = torch.tensor(sigma, dtype=torch.float64, device=x.device, requires_grad=True)
    nt = case["types"]
    tij, tji = types[i] * nt + types[j], types[j] * nt + types[i]
    e, s = 0.5 * (eps[tij] + eps[tji]), 0.5 * (sigma[tij] + sigma[tji])
    d = pos[i] - pos[j]
    d = d - box * torch.round((d / box).detach())
    r2 = (d * d).sum(1)
    inside = (r2 <= RC * RC).detach()
    f6 = (s * s / r2) ** 3
    energy = torch.where(inside, 4.0 * e * (f6 * f6 - f6), 0.0).sum()
    forces = -torch.autograd.grad(energy, pos, create_graph=True)[0]
    grads = torch.autograd.grad(forces, (pos, eps, sigma), up)
    return dict(forces=forces.detach(), pos=grads[0], epsilon=grads[1], sigma=grads[2])
