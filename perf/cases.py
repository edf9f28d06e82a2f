"""Timed cases of the engine: the runs that its users make, over the range of
sizes that they make them at.

Every case goes through the public entry points (the `sopgpu` bindings of the
C ABI).  `prepare` makes the input and the handles that a program holds on to
(an engine with its jobs admitted, a matrix in device memory, a parameter
file with its topology), `run` is one pass: a stretch of dynamics whose end
coordinates the program reads, one factorisation, one evaluation of forces
and energies, or one whole run of the command-line program.
"""
import math
import os
import sys
import tempfile

import numpy as np
import torch

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
if os.path.join(ROOT, "sop-gpu_amd") not in sys.path:
    sys.path.insert(0, os.path.join(ROOT, "sop-gpu_amd"))

import sopgpu as S  # noqa: E402

H_TAU = 0.16              # 40 ps
TAU_H_PS = 250.0
PN_PER_KCAL_A = 69.48
DENSITY = 175.0           # A^3 per bead of a compact globule

# SOP force field and cadence that the benchmark and the tests use: Verlet
# lists rebuilt every 10 steps, possible pairs every 100.
BASE = dict(kspring_cov=14.0, R_limit=2.0, a=3.8, el=1.0, pairs_cutoff=20.0, pairlist_cutoff=20.0,
            pairs_threshold=32.0, pairs_freq=10, possiblepairs_freq=100, timestep=H_TAU, zeta=50.0,
            temperature=0.6, nav=1000, outputtiming=10000, dcdfreq=10000)
FOREVER = 1 << 40         # jobs that a pass never ends


def listed():
    return [
        # Many short trajectories of one small peptide on one GPU (22 beads,
        # 350 runs: the reference's many-runs benchmark): launches and
        # latency are all there is.
        dict(name="peptide_runs", kind="runs", n=22, jobs=350, steps=4000, tune=False),
        # One domain-sized chain under force-ramp pulling, the small
        # configuration of the benchmark, launch shapes tuned as its program
        # tunes them.
        dict(name="chain_1000", kind="runs", n=1000, jobs=1, steps=4000, tune=True),
        # The benchmark's mix: 512 chains of 200 to 5,000 beads stepped
        # together, force-ramp pulling.
        dict(name="mix_512", kind="mix", lo=200, hi=5000, jobs=512, steps=1000),
        # One assembly of mid size under an indentation tip (a request of
        # the serving mix).
        dict(name="assembly_18k", kind="shell", n=300, jobs=60, steps=1000),
        # The capsid shell of 100,000 beads under an indentation tip.
        dict(name="capsid_100k", kind="shell", n=500, jobs=200, steps=400),
        # A protein of two domains with hydrodynamics by the truncated
        # expansion (TEA), nine trajectories together (1,062 beads: the
        # reference's many-runs hydrodynamics).
        dict(name="tea_runs", kind="tea", n=1062, jobs=9, steps=400, listed=False, tune=False),
        # TEA on one long chain (the benchmark's hydrodynamics chain), tuned.
        dict(name="tea_4096", kind="tea", n=4096, jobs=1, steps=200, listed=False, tune=True),
        # Exact hydrodynamics: the tensor factored anew at every step (the
        # reference's rule), split-BF16 updates (the default).
        dict(name="exact_hi_1400", kind="exact", n=1400, mode=0, freq=1, steps=20),
        # The factorisation alone on a matrix in device memory, at the
        # benchmark's order, and in FP32 at a ragged one.
        dict(name="cholesky_12288", kind="chol", n=12288, mode=0),
        dict(name="cholesky_f32_4001", kind="chol", n=4001, mode=1),
        # Analysis of a frame: lists, forces and energies of every bead at
        # given coordinates.
        dict(name="readout_18k", kind="readout", n=300, jobs=60),
        # The command-line program on a parameter file: eight runs of a
        # 144-bead protein with its output files.
        dict(name="program_144", kind="program", n=144, jobs=8, steps=2000),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    """One more case of the same kinds: trajectories of 20 to 5,000 beads, 1
    to 512 together; assemblies of 2,000 to 60,000 beads; TEA chains of 300
    to 4,096 beads; exact hydrodynamics of 100 to 1,400; factorisations of
    order 64 to 8,192."""
    kind = rng.choice(["runs", "runs", "chain", "mix", "shell", "shell", "tea", "tea", "exact", "chol", "chol",
                       "readout", "program"])
    if kind == "runs":
        n = _log_int(rng, 20, 3000)
        jobs = max(1, min(512, _log_int(rng, 1, max(2, 150000 // n))))
        return dict(kind="runs", n=n, jobs=jobs, steps=1000, tune=rng.random() < 0.3)
    if kind == "chain":
        return dict(kind="runs", n=_log_int(rng, 3000, 20000), jobs=1, steps=1000, tune=rng.random() < 0.3)
    if kind == "mix":
        lo = _log_int(rng, 50, 500)
        return dict(kind="mix", lo=lo, hi=_log_int(rng, 1000, 5000), jobs=_log_int(rng, 16, 256), steps=400)
    if kind == "shell":
        return dict(kind="shell", n=rng.randint(101, 499), jobs=_log_int(rng, 20, 120), steps=400)
    if kind == "tea":
        n = _log_int(rng, 300, 4096)
        return dict(kind="tea", n=n, jobs=rng.randint(1, max(1, min(9, 6000 // n))), steps=100,
                    listed=rng.random() < 0.25, tune=rng.random() < 0.3)
    if kind == "exact":
        return dict(kind="exact", n=_log_int(rng, 100, 1400), mode=rng.randint(0, 1), freq=rng.choice([1, 1, 3, 10]),
                    steps=20)
    if kind == "chol":
        return dict(kind="chol", n=_log_int(rng, 64, 8192), mode=rng.randint(0, 1))
    if kind == "readout":
        return dict(kind="readout", n=rng.randint(101, 499), jobs=_log_int(rng, 2, 80))
    return dict(kind="program", n=_log_int(rng, 30, 400), jobs=rng.randint(1, 12), steps=1000)


# ---------------------------------------------------------------------------
# inputs
# ---------------------------------------------------------------------------
def _ramp(n, seed, speed=1.0, kappa=35.0):
    """Force-ramp pulling at `speed` um/s with a cantilever of `kappa` pN/nm."""
    return S.make_params(**BASE, seed=seed, pulling=1, fixedEnd=0, pulledEnd=n - 1, pullFreq=1000,
                         deltax=speed * 1e-8 * 1000 * H_TAU * TAU_H_PS, k_trans=kappa * 0.1 / PN_PER_KCAL_A)


def _clamp(n, seed, **hi):
    """Force clamp of 100 pN with hydrodynamics."""
    return S.make_params(**BASE, seed=seed, pulling=1, fixedEnd=0, pulledEnd=n - 1, fconst=100.0 / PN_PER_KCAL_A,
                         hi_on=1, hi_a=1.9, **hi)


def _ends(system):
    system.fixed = np.array([0], np.int32)
    system.pulled = np.array([system.n - 1], np.int32)
    return system


def _shell(case, seed):
    """Chains on a sphere at the capsid's areal density (100,000 beads at 140 A)."""
    beads = case["n"] * case["jobs"]
    return S.synth_shell(case["jobs"], case["n"], seed=seed, radius=140.0 * math.sqrt(beads / 100000.0))


def _indent(system, seed):
    z = system.coords[:, 2]
    top, bot, tip = float(z.max()), float(z.min()), 50.0
    at = (0.0, 0.0, top + tip + 4.0)
    return S.make_params(**BASE, max_possiblePairs=1024, seed=seed, indentation=1, indTip=at, indChip=at,
                         indDirection=(0.0, 0.0, -1.0), indSurfR0=(0.0, 0.0, bot - 4.0), indSurfN=(0.0, 0.0, 1.0),
                         indTipR=tip, indKs=0.07, indDeltaX=1e-8 * 1000 * H_TAU * TAU_H_PS, indTipZeta=5000.0,
                         indTipA=0.0, indTipB=1.0)


def _frame(case, seed):
    """An assembly with thermal displacements (0.1 A in each direction)."""
    system = _shell(case, seed)
    rng = np.random.default_rng(seed)
    system.coords[:, :3] += rng.normal(0.0, 0.1, (system.n, 3)).astype(np.float32)
    return system


def _rpy_matrix(n, seed):
    """The leading n rows and columns of the Rotne-Prager-Yamakawa tensor
    (D_ij / D_ii, a = 1.9 A) of a confined random walk with 3.8 A bonds, in
    FP64 on the GPU."""
    m, a = (n + 2) // 3, 1.9
    rng = np.random.default_rng(seed)
    step = rng.normal(size=(m, 3))
    step *= 3.8 / np.linalg.norm(step, axis=1, keepdims=True)
    side = (m * DENSITY) ** (1.0 / 3.0) + 7.6
    x = np.cumsum(step, axis=0)
    x = np.abs((x + side / 2) % (2 * side) - side)          # walls reflect
    x = torch.from_numpy(x).cuda()
    D = torch.empty(3 * m, 3 * m, dtype=torch.float64, device="cuda")
    eye = torch.eye(3, dtype=torch.float64, device="cuda")
    for b in range(0, m, 256):
        e = min(m, b + 256)
        d = x[None, :, :] - x[b:e, None, :]
        r = d.square().sum(-1).sqrt()
        s = torch.where(r > 0, r, torch.ones_like(r))
        far = r > 2 * a
        cii = torch.where(far, 3 * a / (4 * s) * (1 + 2 * a * a / (3 * s * s)), 1 - 9 * s / (32 * a))
        crr = torch.where(far, 3 * a / (4 * s) * (1 - 2 * a * a / (s * s)), 3 * s / (32 * a))
        u = d / s[..., None]
        blk = crr[..., None, None] * u[..., :, None] * u[..., None, :] + cii[..., None, None] * eye
        at = torch.arange(b, e, device="cuda")
        blk[at - b, at] = eye
        D[3 * b:3 * e] = blk.permute(0, 2, 1, 3).reshape(3 * (e - b), 3 * m)
    return D[:n, :n].float()


def _write_topology(path, system):
    """A .top file: atoms, bonds and native contacts."""
    out = ["; synthetic chain\n[ atoms ]\n"]
    for i in range(system.n):
        out.append("%5d CA %4d ALA CA A 0.00 0.00\n" % (i, i + 1))
    out.append("\n[ bonds ]\n")
    out += ["%5d %5d 1 %.6f\n" % (b[0], b[1], r) for b, r in zip(system.bonds, system.bond_r0)]
    out.append("\n[ native ]\n")
    out += ["%5d %5d 1 %.6f %.6f\n" % (c[0], c[1], r, e)
            for c, r, e in zip(system.natives, system.nat_r0, system.nat_eh)]
    with open(path, "w") as f:
        f.write("".join(out))


def _program(case, seed):
    folder = tempfile.mkdtemp(prefix="sop_case_")
    at = lambda name: os.path.join(folder, name)  # noqa: E731
    n = case["n"]
    system = S.synth_chain(n, seed=seed)
    _write_topology(at("chain.top"), system)
    with open(at("chain.xyz"), "w") as f:
        f.write("%d\n\n" % n)
        f.write("".join("CA\t%.3f\t%.3f\t%.3f\n" % tuple(c[:3]) for c in system.coords))
    conf = dict(name="chain", topology=at("chain.top"), coordinates=at("chain.xyz"), runnum=case["jobs"], firstrun=1,
                numsteps=case["steps"], timestep=H_TAU, seed=1 + seed % 100000, temperature=0.6, nav=1000,
                outputtiming=1000, dcdfreq=1000, restartfreq=1000, pairs_freq=10, possiblepairs_freq=100,
                pairs_threshold=32.0, kspring_cov=14.0, pulling="on", fixed=0, pulled=n - 1, fixedEnd=0,
                pulledEnd=n - 1, deltax=0.0004, k_trans=0.05, pullFreq=1000, outputname=at("energy_<run>.dat"),
                pullOutput=at("pull_<run>.dat"), DCDfile=at("traj_<run>.dcd"), finalcoord=at("final_<run>.pdb"),
                reffilename=at("ref.pdb"), restartname=at("restart_<run>.pdb"))
    with open(at("run.sop"), "w") as f:
        f.write("".join("%s\t\t%s\n" % kv for kv in conf.items()))
    return folder


def prepare(case, seed):
    kind = case["kind"]
    if kind == "chol":
        n, mp = case["n"], -(-case["n"] // 64) * 64
        A = torch.zeros(mp, mp, dtype=torch.float32, device="cuda")
        A[:n, :n] = _rpy_matrix(n, seed)
        return dict(case=case, A=A, mp=mp)
    if kind == "program":
        return dict(case=case, folder=_program(case, seed))
    eng = S.Engine(0, 24 << 30)
    ids, rng = [], np.random.default_rng(seed)
    if kind == "runs":
        n = case["n"]
        system = _ends(S.synth_chain(n, seed=seed))
        for k in range(case["jobs"]):
            ids.append(eng.add_job(_ramp(n, 1 + (seed + 7919 * k) % 1000000), system, FOREVER))
    elif kind == "mix":
        # one set of sizes for a case; the chains, speeds and springs are the seed's
        sizes = np.exp(np.random.default_rng(2024).uniform(math.log(case["lo"]), math.log(case["hi"]), case["jobs"]))
        sizes = sizes.round().astype(int)
        speeds = np.exp(rng.uniform(math.log(0.1), math.log(10.0), case["jobs"]))
        kappas = rng.uniform(10.0, 70.0, case["jobs"])
        for k in range(case["jobs"]):
            n = int(sizes[k])
            system = _ends(S.synth_chain(n, seed=seed * 1009 + k))
            p = _ramp(n, 1 + (seed + 7919 * k) % 1000000, float(speeds[k]), float(kappas[k]))
            ids.append(eng.add_job(p, system, FOREVER))
    elif kind == "shell":
        system = _shell(case, seed)
        ids.append(eng.add_job(_indent(system, 1 + seed % 1000000), system, FOREVER))
    elif kind == "readout":
        system = _frame(case, seed)
        ids.append(eng.add_job(S.make_params(**BASE, max_possiblePairs=1024, seed=1 + seed % 1000000), system, FOREVER))
    elif kind == "tea":
        n = case["n"]
        system = _ends(S.synth_chain(n, seed=seed))
        for k in range(case["jobs"]):
            p = _clamp(n, 1 + (seed + 7919 * k) % 1000000, hi_epsilon_freq=10, hi_capricious=0,
                       hi_unlisted=0 if case["listed"] else 1)
            ids.append(eng.add_job(p, system, FOREVER))
    elif kind == "exact":
        n = case["n"]
        eng.set_chol_mode(case["mode"])
        system = _ends(S.synth_chain(n, seed=seed))
        ids.append(eng.add_job(_clamp(n, 1 + seed % 1000000, hi_exact=1, hi_chol_freq=case["freq"]), system, FOREVER))
    if case.get("tune"):
        eng.autotune()
    eng.synchronize()
    return dict(case=case, eng=eng, ids=ids, blocks=case.get("steps", 0) // eng.block_steps())


# ---------------------------------------------------------------------------
# one pass
# ---------------------------------------------------------------------------
def run(state):
    case = state["case"]
    kind = case["kind"]
    if kind == "chol":
        L = state["A"].clone()
        S.check(S.lib.sop_chol_factor_noalloc(0, case["n"], L.data_ptr(), state["mp"], case["mode"],
                                              torch.cuda.current_stream().cuda_stream))
        return L[:case["n"], :case["n"]]
    if kind == "program":
        folder = state["folder"]
        S.run_config(os.path.join(folder, "run.sop"))
        finals, rows = [], []
        for r in range(1, 1 + case["jobs"]):
            with open(os.path.join(folder, "final_%d.pdb" % r)) as f:
                finals.append([[float(s[30:38]), float(s[38:46]), float(s[46:54])] for s in f if s.startswith("ATOM")])
            rows.append(np.loadtxt(os.path.join(folder, "energy_%d.dat" % r), ndmin=2)[:, :6])
        return dict(finals=np.array(finals, np.float32), energies=np.array(rows, np.float32))
    eng, ids = state["eng"], state["ids"]
    if kind == "readout":
        eng.rebuild(ids[0])
        forces = eng.forces(ids[0])
        per_bead, sums = eng.energies(ids[0])
        return dict(forces=forces, energies=per_bead, sums=sums)
    eng.run_blocks(state["blocks"])
    coords = np.concatenate([eng.coords(j) for j in ids])
    if kind == "shell":
        return dict(coords=coords, tip=eng.indentation(ids[0]))
    return dict(coords=coords)


# ---------------------------------------------------------------------------
# what a pass cannot do without
# ---------------------------------------------------------------------------
def _pairs(n):
    """Verlet partners of a bead of a compact globule of n beads (about 140 in
    a large one)."""
    return min(n - 1.0, 160.0 * n / (n + 150.0))


def _step_work(n, jobs):
    """Bytes and operations of one step: coordinates, generator state and
    temperature read and written, list entries read (2 bytes each; natives
    10, bonds 6), about 25 operations per repulsive pair."""
    b = n * jobs
    return b * (32 + 32 + 8 + 12 + 2 * 6 + 9 * 10 + 2 * _pairs(n)), b * (25 * _pairs(n) + 9 * 35 + 300)


def work(case):
    kind, n = case["kind"], case["n"] if "n" in case else 0
    if kind == "chol":
        return dict(bytes=4.0 * n * n, flops=n ** 3 / 3.0)
    if kind == "mix":
        mean = (case["hi"] - case["lo"]) / math.log(case["hi"] / case["lo"])
        b, f = _step_work(mean, case["jobs"])
    elif kind in ("shell", "readout"):
        b, f = _step_work(n * case["jobs"], 1)
    else:
        b, f = _step_work(n, case.get("jobs", 1))
    if kind == "readout":
        return dict(bytes=2.0 * b, flops=2.0 * f)
    if kind == "tea":
        terms = case["jobs"] * (n * 160.0 if case["listed"] else float(n) * n)
        b, f = b + 64.0 * n * case["jobs"], f + 75.0 * terms
    if kind == "exact":
        m = 3.0 * n
        b, f = b + 4 * m * m / 2, f + 75.0 * n * n + m * m + m ** 3 / 3.0 / case["freq"]
    return dict(bytes=float(b * case["steps"]), flops=float(f * case["steps"]))


# ---------------------------------------------------------------------------
# the same in 64 bits
# ---------------------------------------------------------------------------
def _exact_readout(case, seed):
    system = _frame(case, seed)
    n = system.n
    t = lambda a, k: torch.from_numpy(np.ascontiguousarray(a)).cuda().to(k)  # noqa: E731
    x = t(system.coords[:, :3], torch.float64)
    force = torch.zeros(n, 4, dtype=torch.float64, device="cuda")
    energy = torch.zeros(3, n, dtype=torch.float64, device="cuda")

    def both(term, i, j, d, f, e):
        """A pair's force f (on i; -f on j) and its energy e, on both beads."""
        force[:, :3].index_add_(0, i, f)
        force[:, :3].index_add_(0, j, -f)
        energy[term].index_add_(0, i, e)
        energy[term].index_add_(0, j, e)

    ks, R2, a2, el = BASE["kspring_cov"], BASE["R_limit"] ** 2, BASE["a"] ** 2, BASE["el"]
    i, j = t(system.bonds[:, 0], torch.int64), t(system.bonds[:, 1], torch.int64)
    r0 = t(system.bond_r0, torch.float64)
    d = x[j] - x[i]
    r = d.square().sum(1).sqrt()
    w = r - r0
    both(0, i, j, d, (ks * w / (r * (1 - w * w / R2)))[:, None] * d, -0.5 * ks * R2 * torch.log(1 - w * w / R2))
    i, j = t(system.natives[:, 0], torch.int64), t(system.natives[:, 1], torch.int64)
    r0, eh = t(system.nat_r0, torch.float64), t(system.nat_eh, torch.float64)
    d = x[j] - x[i]
    q = r0 * r0 / d.square().sum(1)
    p6 = q ** 3
    both(1, i, j, d, (-12 * eh / (r0 * r0) * q * (p6 * p6 - p6))[:, None] * d, eh * (p6 * p6 - 2 * p6))
    bonded = torch.cat([t(system.bonds, torch.int64), t(system.natives, torch.int64)])
    keys = torch.unique(torch.cat([bonded[:, 0] * n + bonded[:, 1], bonded[:, 1] * n + bonded[:, 0]]))
    cut = min(BASE["pairs_cutoff"], BASE["pairlist_cutoff"]) ** 2
    for b in range(0, n, 512):
        e = min(n, b + 512)
        d = x[None, :, :] - x[b:e, None, :]
        d2 = d.square().sum(-1)
        at = torch.arange(b, e, device="cuda")
        ok = d2 < cut
        ok[at - b, at] = False
        mine = keys[(keys >= b * n) & (keys < e * n)]
        ok[mine // n - b, mine % n] = False
        q = torch.where(ok, a2 / torch.where(ok, d2, torch.ones_like(d2)), torch.zeros_like(d2))
        force[b:e, :3] += ((-6 * el / a2) * q ** 4)[..., None].mul(d).sum(1)
        energy[2, b:e] = el * (q ** 3).sum(1)
    return dict(forces=force, energies=energy, sums=0.5 * energy.sum(1))


def exact(case, seed):
    if case["kind"] == "chol":
        A = _rpy_matrix(case["n"], seed)
        return torch.linalg.cholesky(A.double()).tril() + A.double().triu(1)
    if case["kind"] == "readout":
        return _exact_readout(case, seed)
    return None  # trajectories: thousands of steps of noise have no value to be compared with
