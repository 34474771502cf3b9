"""Workloads that stand for what a user of moldyn_amd has it do.

Every case goes through the package's public entry points (Engine, FrameWriter,
StateToSave, mlp.lj_labels, mlp.Trainer) with the host arrays a program hands
over and takes back.  Sizes, lattice edges, controls and step counts are those
of the benchmark and the commands (argon, dt 0.002, lattice edge 3.338339 nm
for the gas, 0.47 nm for the liquid).

Kinds of a case:
  loop      one step of a resident system and its new positions, velocities
            and box: a program that looks at every state
  run       a whole job: the state uploaded, forces, `steps` steps under the
            given controls, the state downloaded
  batch     the same for `replicas` independent systems in one engine
  force     the state uploaded, update_force, the per-atom results downloaded
  label     mlp.lj_labels of one frame: FP64 energies and forces for training
  epoch     one training epoch of the surrogate, and its new parameters
  gradient  loss and gradient of the surrogate over a data set
  files     the state saved to data/<n>.csv + bb.csv and read back
"""
import math
import tempfile

import numpy as np
import torch

import moldyn_amd as M
from moldyn_amd import mlp
from moldyn_amd.engine import L
from moldyn_amd.frames import FrameWriter, StateToSave

MASS = 66.335
SIGMA, EPS = 0.3418, 1.712
RC = 2.5 * SIGMA
K_B = 1.380648528
DT = 0.002
A_GAS, A_LIQUID = 3.338339, 0.47
# second component of the mixture: a lighter, slightly smaller species
MASS2, SIGMA2, EPS2 = 33.5, 0.29, 0.9


def listed():
    return [
        # the benchmark's smallest system, driven one step at a time by a
        # program that looks at every state: latency of a step call and of a
        # small download
        {"name": "loop_1k_gas", "kind": "loop", "n_side": 10, "a": A_GAS, "mode": "fp64_list"},
        # argon gas NVE in FP32, the benchmark's 64,000-atom system: an
        # ordinary production run of a small system
        {"name": "run_64k_gas_nve", "kind": "run", "n_side": 40, "a": A_GAS, "mode": "fp32_list", "temp": 120.0,
         "steps": 2000, "thermostat": "none", "barostat": False, "types": 1},
        # the headline workload: one million atoms under Berendsen NPT, 5,000 steps
        {"name": "run_1M_gas_npt", "kind": "run", "n_side": 100, "a": A_GAS, "mode": "fp32_list", "temp": 273.15,
         "steps": 5000, "thermostat": "berendsen", "barostat": True, "types": 1},
        # the benchmark's dense liquid: about 35 list entries per atom
        {"name": "run_262k_liquid", "kind": "run", "n_side": 64, "a": A_LIQUID, "mode": "fp32_list", "temp": 150.0,
         "steps": 500, "thermostat": "berendsen", "barostat": True, "types": 1},
        # a two-component liquid under Nose-Hoover on the path that restates
        # the reference bit by bit: several types, odd size
        {"name": "run_36k_mixture_fp64", "kind": "run", "n_side": 33, "a": A_LIQUID, "mode": "fp64_list",
         "temp": 120.0, "steps": 400, "thermostat": "nose_hoover", "barostat": False, "types": 2},
        # the learned surrogate in deployment: 262,144 atoms, NPT, BF16 network
        {"name": "run_262k_surrogate", "kind": "run", "n_side": 64, "a": A_LIQUID, "mode": "mlp", "temp": 150.0,
         "steps": 300, "thermostat": "berendsen", "barostat": True, "types": 1},
        # the benchmark's batch: 256 replicas of 500 to 32,768 atoms
        {"name": "batch_256", "kind": "batch", "replicas": 256, "n_min": 500, "n_max": 32768, "steps": 500},
        # the reference's own force benchmark at its largest size on the
        # restatement of its algorithm (all pairs, FP64)
        {"name": "force_27k_allpairs", "kind": "force", "n_side": 30, "a": A_LIQUID, "mode": "fp64_allpairs"},
        # labelling one 4,096-atom training frame
        {"name": "label_4k", "kind": "label", "n_side": 16, "a": 0.42},
        # one epoch of surrogate training, 4,096-atom frames in minibatches of 16
        {"name": "epoch_64x4k", "kind": "epoch", "frames": 64, "n_side": 16, "a": 0.42, "batch": 16},
        # loss and gradient over a small data set of odd sizes
        {"name": "gradient_13x1331", "kind": "gradient", "frames": 13, "n_side": 11, "a": 0.47, "batch": 5},
        # checkpoint and restart through the reference's state files
        {"name": "files_125k", "kind": "files", "n_side": 50, "a": A_GAS},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["loop", "run", "run", "run", "batch", "force", "label", "epoch", "gradient", "files"])
    if kind == "loop":
        return {"kind": kind, "n_side": rng.randint(5, 24), "a": round(rng.uniform(3.0, 4.2), 3),
                "mode": rng.choice(["fp64_list", "fp32_list"])}
    if kind == "run":
        dense = rng.random() < 0.5
        mode = rng.choice(["fp32_list", "fp64_list", "mlp"] if dense else ["fp32_list", "fp64_list"])
        n_side = round(_log_int(rng, 1000, 262144 if dense else 1000000) ** (1.0 / 3.0))
        types = rng.choice([1, 2]) if mode != "mlp" else 1
        return {"kind": kind, "n_side": n_side, "mode": mode, "types": types,
                "a": round(rng.uniform(0.42, 0.55) if dense else rng.uniform(3.0, 4.2), 3),
                "temp": round(rng.uniform(80.0, 400.0), 1),
                "steps": rng.randint(50, 300) if dense else rng.randint(200, 2000),
                "thermostat": rng.choice(["none", "berendsen", "nose_hoover"]),
                "barostat": types == 1 and rng.random() < 0.5}
    if kind == "batch":
        return {"kind": kind, "replicas": _log_int(rng, 2, 256), "n_min": 500, "n_max": _log_int(rng, 1000, 32768),
                "steps": rng.randint(50, 500)}
    if kind == "force":
        mode = rng.choice(["fp64_allpairs", "fp64_list", "fp32_list"])
        hi = 27000 if mode == "fp64_allpairs" else 262144
        return {"kind": kind, "n_side": round(_log_int(rng, 1000, hi) ** (1.0 / 3.0)),
                "a": round(rng.uniform(0.42, 0.75), 3), "mode": mode}
    if kind == "label":
        return {"kind": kind, "n_side": rng.randint(8, 30), "a": round(rng.uniform(0.38, 0.7), 3)}
    if kind in ("epoch", "gradient"):
        n_side = rng.randint(6, 16)
        return {"kind": kind, "frames": rng.randint(3, 64), "n_side": n_side, "a": round(rng.uniform(0.38, 0.7), 3),
                "batch": rng.randint(1, 16)}
    return {"kind": kind, "n_side": round(_log_int(rng, 500, 262144) ** (1.0 / 3.0)),
            "a": round(rng.uniform(0.42, 4.2), 3)}


# ------------------------------------------------------------------ inputs


def _rng(seed, salt):
    return np.random.default_rng([int(seed) & 0xFFFFFFFF, salt])


def _positions(rng, n_side, a, jitter=0.1):
    """A simple-cubic lattice with each site moved by up to `jitter` edges, wrapped."""
    x = M.lattice("u", [n_side] * 3, a)
    box = np.full(3, n_side * a)
    return np.mod(x + rng.uniform(-jitter, jitter, x.shape) * a, box), box


def _velocities(rng, n, temp, mass):
    """Maxwell-Boltzmann with zero net momentum."""
    v = rng.normal(0.0, math.sqrt(K_B * temp * 0.01 / mass), (n, 3))
    return v - v.mean(axis=0)


def _surrogate(rng):
    """Network parameters that stand for the Lennard-Jones pair energy: a
    least-squares fit of it in the radial basis, spread over dense weight
    matrices (silu(z) - silu(-z) = z carries a linear map through each layer)."""
    r = np.linspace(0.75 * SIGMA, RC, 500)
    mu = SIGMA * (0.8 + 1.7 * np.arange(32) / 31.0)
    g = np.exp(-(r[:, None] - mu) ** 2 / (2 * (0.1 * SIGMA) ** 2)) * (0.5 * (np.cos(np.pi * r / RC) + 1.0))[:, None]
    rr = np.maximum(r, 0.88 * SIGMA)  # the core continued linearly
    s6 = (SIGMA / rr) ** 6
    phi = 2.0 * EPS * (s6 * s6 - s6 + (6.0 * s6 - 12.0 * s6 * s6) / rr * (r - rr))
    scale = 1.0 + np.abs(phi)
    lhs = np.vstack([g / scale[:, None], 0.005 * np.eye(32)])
    coef = np.linalg.lstsq(lhs, np.concatenate([phi / scale, np.zeros(32)]), rcond=None)[0]
    g_mean, g_std = np.full(32, 1.0), np.full(32, 0.5)
    a = coef * g_std
    e_scale = float(np.linalg.norm(a))
    q1, _ = np.linalg.qr(rng.normal(size=(64, 32)))
    q2, _ = np.linalg.qr(rng.normal(size=(64, 64)))
    w1 = np.concatenate([q1, -q1])
    w2 = np.block([[q2, -q2], [-q2, q2]])
    u = q2 @ (q1 @ (a / e_scale))
    theta = np.concatenate([w1.ravel(), np.zeros(128), w2.ravel(), np.zeros(128), u, -u, [0.0]])
    return mlp.Surrogate(theta.astype(np.float32), g_mean.astype(np.float32), (1.0 / g_std).astype(np.float32),
                         np.full(32, -10.0, np.float32), np.full(32, 100.0, np.float32), e_scale, float(coef @ g_mean))


def _lj(x, box, chunk=1024):
    """FP64 Lennard-Jones energies (Particle::potential / 2), forces and
    virials of one frame by plain torch, all pairs."""
    dev = "cuda" if torch.cuda.is_available() else "cpu"
    x = torch.as_tensor(x, dtype=torch.float64, device=dev)
    b = torch.as_tensor(np.broadcast_to(box, 3).copy(), dtype=torch.float64, device=dev)
    u_cut = 4 * EPS * ((SIGMA / RC) ** 12 - (SIGMA / RC) ** 6)
    pot, force, vir = [], [], []
    for i0 in range(0, len(x), chunk):
        d = x[None, :, :] - x[i0:i0 + chunk, None, :]
        d = torch.where(d < -b / 2, d + b, torch.where(d > b / 2, d - b, d))
        r2 = d.square().sum(-1)
        k = torch.arange(len(d), device=dev)
        r2[k, i0 + k] = math.inf
        near = r2 <= RC * RC
        r = torch.where(near, r2, torch.ones_like(r2)).sqrt()
        s6 = (SIGMA / r) ** 6
        u = torch.where(near, 4 * EPS * (s6 * s6 - s6) - u_cut, torch.zeros_like(r))
        f = torch.where(near, 24 * EPS / r * (s6 - 2 * s6 * s6), torch.zeros_like(r))
        pot.append(u.sum(1))
        force.append((d * (f / r)[..., None]).sum(1))
        vir.append((f * r).sum(1))
    return torch.cat(pot).cpu().numpy(), torch.cat(force).cpu().numpy(), torch.cat(vir).cpu().numpy()


def _frames(case, seed):
    rng = _rng(seed, 7)
    f, n = case["frames"], case["n_side"] ** 3
    pos, box, e, fr = np.empty((f, n, 3)), np.empty((f, 3)), np.empty((f, n)), np.empty((f, n, 3))
    for k in range(f):
        pos[k], box[k] = _positions(rng, case["n_side"], case["a"] * rng.uniform(0.98, 1.05), 0.08)
        p, fr[k], _ = _lj(pos[k], box[k])
        e[k] = p / 2.0
    return mlp.Frames(pos, box, e, fr)


def _train_inputs(case, seed, frames):
    """Parameters, normalisation, scales and loss weights as mlp.train sets them."""
    w_e = 1.0 / max(float(np.var(frames.e_ref)), 1e-12)
    w_f = 1.0 / max(float(np.var(frames.f_ref)), 1e-12)
    return (mlp.init_params(seed % 100003), np.full(32, 1.0, np.float32), np.full(32, 2.0, np.float32),
            float(np.std(frames.e_ref)), float(np.mean(frames.e_ref)), w_e, w_f,
            _rng(seed, 8).permutation(case["frames"]))


LR = 1e-3


def _run_inputs(case, seed):
    rng = _rng(seed, 1)
    x, box = _positions(rng, case["n_side"], case["a"], 0.08)
    n = len(x)
    temp = case.get("temp", 273.15)
    if case.get("types", 1) == 2:
        n2 = n // 3
        v = np.concatenate([_velocities(rng, n - n2, temp, MASS), _velocities(rng, n2, temp, MASS2)])
        order = rng.permutation(n)  # the species are mixed over the sites
        return [n - n2, n2], [MASS, MASS2], x[order], v, box
    return [n], [MASS], x, _velocities(rng, n, temp, MASS), box


def _counts(case):
    """Atoms of each replica, log-uniform in [n_min, n_max]: the batch is part of the case."""
    u = np.random.default_rng(case["replicas"]).uniform(0.0, 1.0, case["replicas"])
    return np.rint(case["n_min"] * (case["n_max"] / case["n_min"]) ** u).astype(np.int64)


def _engine(case, counts, masses, box):
    e = M.Engine(counts, masses, box, force_mode=case["mode"])
    if len(counts) == 2:
        e.set_pair_potential(1, 1, SIGMA2, EPS2)
        e.set_pair_potential(0, 1, 0.5 * (SIGMA + SIGMA2), math.sqrt(EPS * EPS2))
    return e


def prepare(case, seed):
    kind = case["kind"]
    if kind in ("loop", "run", "force"):
        counts, masses, x, v, box = _run_inputs(case, seed)
        e = _engine(case, counts, masses, box)
        if case["mode"] == "mlp":
            _surrogate(_rng(seed, 2)).apply(e)
        if kind == "loop":
            e.upload(x, v, box)
            e.update_force()
        return {"case": case, "engine": e, "x": x, "v": v, "box": box}
    if kind == "batch":
        rng = _rng(seed, 3)
        r = case["replicas"]
        counts = _counts(case)
        a, temp = rng.uniform(3.0, 4.2, r), rng.uniform(80.0, 400.0, r)
        xs, vs, boxes = [], [], []
        for k in range(r):
            x, box = _positions(rng, int(math.ceil(counts[k] ** (1.0 / 3.0) - 1e-9)), a[k], 0.02)
            xs.append(x[:counts[k]])
            vs.append(_velocities(rng, int(counts[k]), temp[k], MASS))
            boxes.append(box)
        boxes = np.array(boxes)
        e = M.Engine(counts[:, None], [MASS], boxes, force_mode="fp32_list")
        return {"case": case, "engine": e, "x": np.concatenate(xs), "v": np.concatenate(vs), "box": boxes,
                "temp": temp, "pressure": rng.uniform(0.5, 5.0, r)}
    if kind == "label":
        x, box = _positions(_rng(seed, 4), case["n_side"], case["a"], 0.08)
        return {"case": case, "x": x, "box": box}
    if kind in ("epoch", "gradient"):
        frames = _frames(case, seed)
        tr = mlp.Trainer(frames)
        theta, g_mean, g_inv_std, e_scale, e_shift, w_e, w_f, order = _train_inputs(case, seed, frames)
        tr.set_params(theta, g_mean, g_inv_std, e_scale, e_shift)
        return {"case": case, "trainer": tr, "w": (w_e, w_f), "order": order}
    counts, masses, x, v, box = _run_inputs(case, seed)
    e = M.Engine(counts, masses, box)
    e.upload(x, v, box)
    folder = tempfile.TemporaryDirectory(prefix="moldyn_files_")
    return {"case": case, "engine": e, "folder": folder, "writer": FrameWriter(e, folder.name)}


# ------------------------------------------------------------------ one pass


def _controls(case):
    th = {"none": lambda: None,
          "berendsen": lambda: M.thermostat("berendsen", tau=1.0, target_t=case["temp"]),
          "nose_hoover": lambda: M.thermostat("nose_hoover", tau=1.0, target_t=case["temp"])}[case["thermostat"]]()
    if not case["barostat"]:
        return th, None
    if case["a"] > 1.0:  # gas: the benchmark's controls
        return th, M.barostat("berendsen", beta=1.0, tau=5.0, target_p=1.01325)
    return th, M.barostat("berendsen", beta=1.0, tau=50.0, target_p=11.0)


def run(s):
    case = s["case"]
    kind = case["kind"]
    if kind == "loop":
        e = s["engine"]
        e.step(DT, 1, M.thermostat("berendsen", tau=10.0, target_t=300.0))
        return e.download(("x", "v", "box"))
    if kind == "run":
        e = s["engine"]
        th, ba = _controls(case)
        e.upload(s["x"], s["v"], s["box"])
        e.update_force()
        e.step(DT, case["steps"], th, ba)
        return e.download()
    if kind == "batch":
        e, r = s["engine"], case["replicas"]
        e.upload(s["x"], s["v"], s["box"])
        e.update_force()
        th = (L.MdThermostat * r)(*[M.thermostat("berendsen", 10.0, float(t)) for t in s["temp"]])
        ba = (L.MdBarostat * r)(*[M.barostat("berendsen", 1.0, 5.0, float(p)) for p in s["pressure"]])
        if r == 1:
            th, ba = th[0], ba[0]
        e.step(DT, case["steps"], th, ba)
        return e.download()
    if kind == "force":
        e = s["engine"]
        e.upload(s["x"], s["v"], s["box"])
        e.update_force()
        return e.download(("force", "pot", "virial"))
    if kind == "label":
        return mlp.lj_labels(s["x"], s["box"])
    if kind == "epoch":
        tr = s["trainer"]
        loss = tr.epoch(case["batch"], LR, *s["w"], order=s["order"])
        # the losses are means of FP32 terms: FP32 is what they hold
        return {"loss": loss.astype(np.float32), "theta": tr.params()}
    if kind == "gradient":
        loss, grad = s["trainer"].loss(*s["w"], batch_frames=case["batch"], grad=True)
        return {"loss": loss.astype(np.float32), "grad": grad}
    s["writer"].save(0)
    s["writer"].flush()
    got = StateToSave.load_from_file(s["folder"].name, 0)
    return {"ids": got.ids, "x": got.x, "v": got.v, "box": got.boundary_box}


# ------------------------------------------------------------------ what a pass cannot do without


def work(case):
    kind = case["kind"]
    if kind in ("epoch", "gradient"):
        rows = case["frames"] * case["n_side"] ** 3
        pairs = 4.0 / 3.0 * math.pi * (RC / case["a"]) ** 3
        # multiply-adds of the 32-128-128-1 network: forward, force backward,
        # the double backward and the four weight products; about ten
        # operations per basis value and pair, with the force and its adjoint
        net = 2.0 * (7 * 128 * 128 + 7 * 32 * 128) * rows
        return {"bytes": rows * (24.0 + 16.0 + 4.0 * 32), "flops": net + rows * pairs * 32 * 2 * 10.0}
    if kind == "batch":
        n, a, steps = int(_counts(case).sum()), 3.6, case["steps"]
    else:
        n, a, steps = case["n_side"] ** 3, case["a"], case.get("steps", 1)
    near = 4.0 / 3.0 * math.pi * (RC / a) ** 3
    if kind == "files":
        return {"bytes": n * (48.0 + 118.0 + 118.0 + 50.0), "flops": 0.0}
    if kind in ("force", "label"):
        return {"bytes": n * (48.0 + 40.0), "flops": n * near * 45.0 + n * (n * 9.0 if case.get("mode") == "fp64_allpairs" else 0.0)}
    if case.get("mode") == "mlp":
        flops = n * (2.0 * 2 * (32 * 128 + 128 * 128) + near * 32 * 2 * 6.0)
    else:
        flops = n * (40.0 + near * 45.0)
    # per step the state in and out; the job's arrays in and out once
    return {"bytes": n * (96.0 * steps + (48.0 + 88.0 if kind != "loop" else 48.0)), "flops": flops * steps}


# ------------------------------------------------------------------ the same in 64 bits


def _exact_loop(case, seed):
    _, _, x, v, box = _run_inputs(case, seed)
    n = len(x)
    f = _lj(x, box)[1]
    c = DT / (2.0 * MASS)
    com = v.mean(axis=0)
    t = MASS * np.square(v - com).sum() / (3.0 * n * K_B) * 100.0
    lam = math.sqrt(1.0 + DT / 10.0 * (300.0 / t - 1.0))
    v = (v + f * c) * lam
    x = x + v * DT
    x = np.where(x < 0, x + box, np.where(x >= box, x - box, x))
    return {"x": x, "v": v + _lj(x, box)[1] * c, "box": box}


def _batch_loss(theta, norm, frames, idx, w_e, w_f, n_total):
    """w_e sum (E - E_ref)^2 + w_f sum (F - F_ref)^2 / 3 over n_total atoms of
    the frames idx, as a differentiable function of theta, and the two sums."""
    dev = theta.device
    g_mean, g_inv_std, e_scale, e_shift = norm
    mu = torch.as_tensor(SIGMA * (0.8 + 1.7 * np.arange(32) / 31.0), device=dev)
    w1, b1 = theta[:4096].reshape(128, 32), theta[4096:4224]
    w2, b2 = theta[4224:20608].reshape(128, 128), theta[20608:20736]
    w3, b3 = theta[20736:20864], theta[20864]
    se = sf = torch.zeros((), dtype=torch.float64, device=dev)
    for k in idx:
        x = torch.as_tensor(frames.pos[k], device=dev)
        b = torch.as_tensor(frames.box[k], device=dev)
        ii, jj = [], []
        with torch.no_grad():
            for i0 in range(0, len(x), 1024):
                d = x[None] - x[i0:i0 + 1024, None]
                d = torch.where(d < -b / 2, d + b, torch.where(d > b / 2, d - b, d))
                i, j = torch.nonzero(d.square().sum(-1) < RC * RC, as_tuple=True)
                ii.append(i + i0)
                jj.append(j)
            i, j = torch.cat(ii), torch.cat(jj)
            i, j = i[i != j], j[i != j]
            d = x[j] - x[i]
            d = torch.where(d < -b / 2, d + b, torch.where(d > b / 2, d - b, d))
            r = d.square().sum(-1).sqrt()
            fc = 0.5 * (torch.cos(math.pi * r / RC) + 1.0)
            dfc = -0.5 * math.pi / RC * torch.sin(math.pi * r / RC)
            u = r[:, None] - mu
            e = torch.exp(-u * u / (2 * (0.1 * SIGMA) ** 2))
            g = torch.zeros(len(x), 32, dtype=torch.float64, device=dev).index_add_(0, i, e * fc[:, None])
            dg = e * (dfc[:, None] - u / (0.1 * SIGMA) ** 2 * fc[:, None])
            dirs = d / r[:, None]
            e_ref = torch.as_tensor(frames.e_ref[k].astype(np.float32), device=dev).double()
            f_ref = torch.as_tensor(frames.f_ref[k].astype(np.float32), device=dev).double()
        # backward of the network written out, so that autograd goes through it once
        a1 = (g - g_mean) * g_inv_std @ w1.T + b1
        s1 = torch.sigmoid(a1)
        a2 = (a1 * s1) @ w2.T + b2
        s2 = torch.sigmoid(a2)
        energy = e_scale * ((a2 * s2) @ w3 + b3) + e_shift
        d2 = w3 * (s2 * (1 + a2 * (1 - s2)))
        d1 = (d2 @ w2) * (s1 * (1 + a1 * (1 - s1)))
        gam = e_scale * g_inv_std * (d1 @ w1)
        c = ((gam[i] + gam[j]) * dg).sum(1)
        force = torch.zeros_like(x).index_add(0, i, c[:, None] * dirs)
        se = se + (energy - e_ref).square().sum()
        sf = sf + (force - f_ref).square().sum()
    return w_e * se / n_total + w_f * sf / (3.0 * n_total), se.detach(), sf.detach()


def _exact_training(case, seed):
    frames = _frames(case, seed)
    theta, g_mean, g_inv_std, e_scale, e_shift, w_e, w_f, order = _train_inputs(case, seed, frames)
    dev = "cuda" if torch.cuda.is_available() else "cpu"
    norm = (torch.as_tensor(g_mean, device=dev).double(), torch.as_tensor(g_inv_std, device=dev).double(), e_scale, e_shift)
    theta = torch.as_tensor(theta, device=dev).double()
    f, n = frames.e_ref.shape
    if case["kind"] == "gradient":
        grad, se, sf = torch.zeros_like(theta), 0.0, 0.0
        for k in range(f):
            p = theta.clone().requires_grad_(True)
            loss, a, b = _batch_loss(p, norm, frames, [k], w_e, w_f, f * n)
            grad += torch.autograd.grad(loss, p)[0]
            se, sf = se + float(a), sf + float(b)
        se, sf = se / (f * n), sf / (3.0 * f * n)
        return {"loss": np.array([w_e * se + w_f * sf, se, sf]), "grad": grad.cpu().numpy()}
    m, v, losses, step = torch.zeros_like(theta), torch.zeros_like(theta), [], 0
    for b0 in range(0, f, case["batch"]):
        idx = order[b0:b0 + case["batch"]]
        grad, se, sf = torch.zeros_like(theta), 0.0, 0.0
        for k in idx:
            p = theta.clone().requires_grad_(True)
            loss, a, b = _batch_loss(p, norm, frames, [k], w_e, w_f, len(idx) * n)
            grad += torch.autograd.grad(loss, p)[0]
            se, sf = se + float(a), sf + float(b)
        se, sf = se / (len(idx) * n), sf / (3.0 * len(idx) * n)
        losses.append([w_e * se + w_f * sf, se, sf])
        step += 1
        m = 0.9 * m + 0.1 * grad
        v = 0.999 * v + 0.001 * grad * grad
        theta = theta - LR * (m / (1 - 0.9 ** step)) / ((v / (1 - 0.999 ** step)).sqrt() + 1e-8)
    return {"loss": np.mean(losses, axis=0), "theta": theta.cpu().numpy()}


def exact(case, seed):
    kind = case["kind"]
    if kind == "loop":
        return _exact_loop(case, seed)
    if kind in ("epoch", "gradient"):
        return _exact_training(case, seed)
    if kind == "label":
        x, box = _positions(_rng(seed, 4), case["n_side"], case["a"], 0.08)
        pot, force, _ = _lj(x, box)
        return pot / 2.0, force
    if kind == "force":
        _, _, x, _, box = _run_inputs(case, seed)
        pot, force, vir = _lj(x, box, 256)
        return {"force": force, "pot": pot, "virial": vir}
    if kind == "files":
        _, _, x, v, box = _run_inputs(case, seed)
        return {"ids": None, "x": x, "v": v, "box": box}
    return None  # a trajectory of many steps
