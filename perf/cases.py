"""Workloads that stand for what users run on the octree_hip solver.

Each case goes through the public Python surface (`OctreeHip`, the ctypes
binding for the device-pointer sort) with the state a program keeps between
calls: a handle with its particles uploaded, or host arrays where the call
takes those. A kind of case is one use of the library:

  forces   one force evaluation of a resident state, accelerations to the host
  coupled  a host program that owns the particles: upload, forces back
  steps    a leapfrog run: K steps on the resident state, then a snapshot
  block    the same with dyadic block time steps (one base step)
  treepm   a periodic TreePM box: short-range walk and particle mesh
  lff      forces with the learned far-field correction (a given network)
  lffgrad  gradient of the correction's network on a batch (its training)
  direct   FP64 direct sum on sampled targets (force-error measurements)
  sort     the allocation-free key/value sort on device pointers
"""
import ctypes
import math

import numpy as np
import torch

import blitzar_amd as B

LFF_SIZES = (32 * 64, 64, 64 * 64, 64, 64 * 3, 3)  # W1 b1 W2 b2 W3 b3


def listed():
    return [
        # The smallest real problem: the 2,000-particle cloud, one force pass.
        {"name": "forces_cloud_2k", "kind": "forces", "scene": "cube", "n": 2000,
         "criterion": "com", "theta": 0.5, "order": 2, "alpha": 0.0, "mono": 0.0},
        # A small interactive run, odd size, where launches and latency count.
        {"name": "steps_plummer_4k", "kind": "steps", "scene": "plummer", "n": 4099,
         "theta": 0.5, "eps": 0.01, "dt": 1e-3, "steps": 10},
        # The small reference configuration: Plummer 65,536, theta 0.5, KDK.
        {"name": "steps_plummer_64k", "kind": "steps", "scene": "plummer", "n": 65536,
         "theta": 0.5, "eps": 0.01, "dt": 1e-3, "steps": 10},
        # The middle configuration: Plummer 1,048,576.
        {"name": "steps_plummer_1m", "kind": "steps", "scene": "plummer", "n": 1048576,
         "theta": 0.5, "eps": 0.005, "dt": 5e-4, "steps": 4},
        # The benchmark's state and opening criterion: 8,388,608 particles, relative
        # criterion with point-mass cells.
        {"name": "forces_merger_8m", "kind": "forces", "scene": "merger", "n": 8388608,
         "criterion": "relative", "theta": 2.0, "order": 2, "alpha": 0.0125, "mono": 0.2},
        # A program that owns its particles (the reference's dirty-host path):
        # new positions in, accelerations out, the reference's bounds criterion.
        {"name": "coupled_bounds_300k", "kind": "coupled", "scene": "plummer", "n": 300001,
         "criterion": "bounds", "theta": 0.5, "order": 2, "alpha": 0.0, "mono": 0.0},
        # Block time steps: one base step of 2^-6 in up to 256 slices.
        {"name": "block_plummer_100k", "kind": "block", "n": 100003, "theta": 0.5, "levels": 8},
        # A periodic cosmological box: 128^3 Zel'dovich lattice, mesh 128.
        {"name": "treepm_128", "kind": "treepm", "ng": 128, "mesh": 128, "theta": 0.6},
        # Learned far-field correction over a merger, a network loaded beforehand.
        {"name": "lff_merger_512k", "kind": "lff", "n": 524288, "band": 0.75},
        # One gradient of that network (a large training batch).
        {"name": "lff_gradient_64k", "kind": "lffgrad", "n": 65536},
        # Force-error check of a run: 4,096 targets against every particle, FP64.
        {"name": "direct_4096_of_1m", "kind": "direct", "n": 1048576, "targets": 4096},
        # A key/value sort inside a loop that may not allocate.
        {"name": "sort_device_1500k", "kind": "sort", "n": 1500000, "bits": 63},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["forces", "forces", "coupled", "steps", "steps", "block", "treepm", "lff",
                       "lffgrad", "direct", "sort"])
    if kind in ("forces", "coupled"):
        crit = rng.choice(["com", "bounds", "extent", "relative", "relative"])
        n = _log_int(rng, 1000, 4000000 if kind == "forces" else 600000)
        c = {"kind": kind, "scene": rng.choice(["plummer", "merger", "cube"]), "n": n,
             "criterion": crit, "theta": round(rng.uniform(0.4, 0.8), 2),
             "order": rng.choice([2, 2, 1]), "alpha": 0.0, "mono": 0.0}
        if crit == "relative":
            c.update(theta=round(rng.uniform(1.0, 2.0), 2), order=2,
                     alpha=round(rng.uniform(0.004, 0.02), 4), mono=rng.choice([0.0, 0.1, 0.2]))
        return c
    if kind == "steps":
        return {"kind": kind, "scene": rng.choice(["plummer", "merger"]),
                "n": _log_int(rng, 1000, 1048576), "theta": round(rng.uniform(0.4, 0.8), 2),
                "eps": 0.01, "dt": rng.choice([2.0 ** -10, 5e-4]), "steps": rng.randint(1, 6)}
    if kind == "block":
        return {"kind": kind, "n": _log_int(rng, 2000, 150000),
                "theta": round(rng.uniform(0.5, 0.8), 2), "levels": rng.choice([5, 8])}
    if kind == "treepm":
        ng = rng.randint(24, 120)
        return {"kind": kind, "ng": ng, "mesh": 2 * ((ng + 1) // 2),
                "theta": round(rng.uniform(0.4, 0.7), 2)}
    if kind == "lff":
        return {"kind": kind, "n": _log_int(rng, 50000, 800000),
                "band": round(rng.uniform(0.65, 0.8), 2)}
    if kind == "lffgrad":
        return {"kind": kind, "n": _log_int(rng, 2000, 200000)}
    if kind == "direct":
        return {"kind": kind, "n": _log_int(rng, 10000, 2000000),
                "targets": _log_int(rng, 100, 4096)}
    return {"kind": kind, "n": _log_int(rng, 1000, 2097152), "bits": rng.choice([30, 63, 64])}


# -- inputs ---------------------------------------------------------------------

def _scene(scene, n, seed):
    if scene == "plummer":
        return B.plummer(n, seed=seed)
    if scene == "cube":
        return B.uniform_cube(n, seed=seed)
    pos, vel, m = B.hernquist_merger((n + 1) // 2, seed=seed, separation=20.0, pericentre=2.0)
    return (np.ascontiguousarray(pos[:n]), np.ascontiguousarray(vel[:n]),
            np.ascontiguousarray(m[:n]))


def _lff_params(seed):
    """A network of a trained one's magnitude: fan-in scaled layers, a small output."""
    rng = np.random.default_rng([seed, 5])
    w1, b1, w2, b2, w3, b3 = (rng.standard_normal(k) for k in LFF_SIZES)
    return np.concatenate([w1 / math.sqrt(32), 0.1 * b1, w2 / 8.0, 0.1 * b2, 2e-3 * w3,
                           0.0 * b3]).astype(np.float32)


def _lff_rows(n, seed):
    """Feature rows (three zero pads) and targets of unit variance."""
    rng = np.random.default_rng([seed, 6])
    x = rng.standard_normal((n, 32)).astype(np.float32)
    x[:, 29:] = 0.0
    return x, rng.standard_normal((n, 3)).astype(np.float32)


def _targets(case, seed):
    rng = np.random.default_rng([seed, 7])
    k = min(case["targets"], case["n"])
    return np.sort(rng.choice(case["n"], k, replace=False)).astype(np.uint32)


def prepare(case, seed):
    kind = case["kind"]
    st = {"kind": kind, "case": case}
    if kind in ("forces", "coupled"):
        pos, vel, m = _scene(case["scene"], case["n"], seed)
        more = {}
        if case["criterion"] == "relative":
            more = {"relative_alpha": case["alpha"], "relative_mono": case["mono"]}
        s = B.OctreeHip(case["n"], theta=case["theta"], softening=0.01,
                        multipole_order=case["order"], criterion=case["criterion"], **more)
        st["solver"] = s
        if kind == "coupled":
            st["host"] = (pos, vel, m)
        else:
            s.upload(pos, vel, m)
            if case["criterion"] == "relative":  # |a| of an earlier evaluation, as in a run
                s.compute_accelerations(to_host=False)
        return st
    if kind == "steps":
        s = B.OctreeHip(case["n"], theta=case["theta"], softening=case["eps"],
                        integrator="leapfrog")
        s.upload(*_scene(case["scene"], case["n"], seed))
        st["solver"] = s
        return st
    if kind == "block":
        s = B.OctreeHip(case["n"], theta=case["theta"], softening=0.01, integrator="leapfrog",
                        adaptive_max_level=case["levels"], adaptive_eta=0.02, adaptive_flags=0)
        s.upload(*_scene("plummer", case["n"], seed))
        st["solver"] = s
        return st
    if kind == "treepm":
        ng = case["ng"]
        h = 1.0 / case["mesh"]
        n = ng ** 3
        s = B.OctreeHip(n, theta=case["theta"], softening=0.05 * h, treepm_split_scale=1.25 * h,
                        treepm_cutoff=4.5 * 1.25 * h, periodic_box=1.0, pm_mesh=case["mesh"])
        s.upload(B.zeldovich_lattice(ng, seed=seed), None, np.full(n, 1.0 / n, np.float32))
        st["solver"] = s
        return st
    if kind == "lff":
        s = B.OctreeHip(case["n"], theta=0.9, softening=0.01)
        s.lff_configure(theta=0.9, band=case["band"], min_count=64)
        s.lff_set_params(_lff_params(seed))
        s.lff_enable(True)
        s.upload(*_scene("merger", case["n"], seed))
        st["solver"] = s
        return st
    if kind == "lffgrad":
        st["solver"] = s = B.OctreeHip(1024, theta=0.9, softening=0.01)
        s.lff_configure(theta=0.9, band=0.75, min_count=64)
        st["rows"] = _lff_rows(case["n"], seed)
        st["params"] = _lff_params(seed)
        return st
    if kind == "direct":
        st["solver"] = s = B.OctreeHip(case["n"], softening=0.01)
        s.upload(*_scene("plummer", case["n"], seed))
        st["targets"] = _targets(case, seed)
        return st
    g = torch.Generator(device="cuda").manual_seed(seed)
    # keys over the whole range of the sorted bits (the top one set in half of a 64-bit set)
    keys = torch.randint(-(2 ** 63), 2 ** 63 - 1, (case["n"],), dtype=torch.int64, device="cuda",
                         generator=g)
    if case["bits"] < 64:
        keys &= (1 << case["bits"]) - 1
    st["keys"] = keys
    st["vals"] = torch.arange(case["n"], dtype=torch.int32, device="cuda")
    st["keys_out"] = torch.empty_like(keys)
    st["vals_out"] = torch.empty_like(st["vals"])
    return st


# -- one pass -------------------------------------------------------------------

def run(st):
    kind, case = st["kind"], st["case"]
    if kind in ("forces", "treepm", "lff"):
        return {"acc": st["solver"].compute_accelerations()}
    if kind == "coupled":
        st["solver"].upload(*st["host"])
        return {"acc": st["solver"].compute_accelerations()}
    if kind == "steps":
        st["solver"].step(case["dt"], case["steps"])
        pos, vel = st["solver"].download()
        return {"pos": pos, "vel": vel}
    if kind == "block":
        st["solver"].step(2.0 ** -6, 1)
        pos, vel = st["solver"].download()
        return {"pos": pos, "vel": vel}
    if kind == "lffgrad":
        grad, loss = st["solver"].lff_gradient(*st["rows"], st["params"])
        return {"grad": grad, "loss": loss}
    if kind == "direct":
        return {"acc": st["solver"].direct_forces_fp64(st["targets"])}
    p = lambda t: t.data_ptr()  # noqa: E731
    err = ctypes.create_string_buffer(256)
    stream = torch.cuda.current_stream().cuda_stream
    rc = B.lib().bh_hip_sort_pairs_noalloc(p(st["keys"]), p(st["vals"]), case["n"], case["bits"],
                                           p(st["keys_out"]), p(st["vals_out"]), stream, err, 256)
    if rc != 0:
        raise RuntimeError(f"sort_pairs_noalloc: {rc} {err.value.decode(errors='replace')}")
    return {"keys": st["keys_out"], "vals": st["vals_out"]}


# -- what a pass cannot do without -----------------------------------------------

def _interactions(case):
    """Interactions per target of a tree walk: the Barnes-Hut count
    28 pi / (3 theta^3) log8(n) for the geometric criteria, at most n; about a
    thousand under the relative criterion."""
    n = case.get("n") or case["ng"] ** 3
    if case.get("criterion") == "relative":
        return min(n, 1000.0)
    theta = {"lff": 0.9}.get(case["kind"], case.get("theta", 0.9))
    return min(float(n), 28.0 * math.pi / (3.0 * theta ** 3) * math.log(max(n, 8), 8))


def work(case):
    kind = case["kind"]
    if kind == "sort":
        return {"bytes": 24.0 * case["n"], "flops": 0.0}
    if kind == "lffgrad":
        macs = 32 * 64 + 64 * 64 + 64 * 3
        return {"bytes": case["n"] * 35 * 4.0 + 2 * 6467 * 4.0, "flops": 6.0 * macs * case["n"]}
    if kind == "direct":
        return {"bytes": 28.0 * case["n"] + 28.0 * case["targets"],
                "flops": 20.0 * case["n"] * case["targets"]}
    n = case["ng"] ** 3 if kind == "treepm" else case["n"]
    per_walk = 20.0 * n * _interactions(case)
    if kind == "steps":  # state in, state out; the first pass also primes the force
        return {"bytes": 52.0 * n + 48.0 * n, "flops": per_walk * case["steps"]}
    if kind == "block":  # every particle steps at least once per base step
        return {"bytes": 52.0 * n + 48.0 * n, "flops": per_walk}
    if kind == "treepm":  # short-range neighbours of a 4.5 r_s sphere at most, plus the mesh
        per_walk = 20.0 * n * min(n, 4.0 / 3.0 * math.pi * (4.5 * 1.25) ** 3)
        per_walk += 4 * 2.5 * case["mesh"] ** 3 * 3 * math.log2(case["mesh"])
    return {"bytes": 28.0 * n + 12.0 * n, "flops": per_walk}


# -- 64-bit results ----------------------------------------------------------------

def _direct_sum(pos, m, eps, targets=None):
    """Softened direct sum in FP64 (G = 1) on the GPU, n x 3."""
    x = torch.as_tensor(np.asarray(pos, np.float64), device="cuda")
    m = torch.as_tensor(np.asarray(m, np.float64), device="cuda")
    t = x if targets is None else x[torch.as_tensor(targets.astype(np.int64), device="cuda")]
    out = torch.empty((t.shape[0], 3), dtype=torch.float64, device="cuda")
    rows = max(1, min(t.shape[0], (1 << 26) // x.shape[0]))
    for a in range(0, t.shape[0], rows):
        q = t[a:a + rows]
        d = [x[None, :, k] - q[:, None, k] for k in range(3)]
        w = torch.addcmul(torch.addcmul(torch.addcmul(
            torch.full_like(d[0], eps * eps), d[0], d[0]), d[1], d[1]), d[2], d[2])
        w = w.rsqrt_()
        w = w * w * w * m[None, :]
        for k in range(3):
            out[a:a + rows, k] = (w * d[k]).sum(1)
    return out


def exact(case, seed):
    kind = case["kind"]
    if kind in ("forces", "coupled") and case["n"] <= 320000:
        pos, _, m = _scene(case["scene"], case["n"], seed)
        return {"acc": _direct_sum(pos, m, float(np.float32(0.01))).cpu().numpy()}
    if kind == "direct":
        pos, _, m = _scene("plummer", case["n"], seed)
        return {"acc": _direct_sum(pos, m, float(np.float32(0.01)),
                                   _targets(case, seed)).cpu().numpy()}
    if kind == "steps" and case["n"] ** 2 * (case["steps"] + 1) <= 6e10:
        pos, vel, m = _scene(case["scene"], case["n"], seed)
        x, v = (torch.as_tensor(a, device="cuda") for a in (pos, vel))
        eps, dt = float(np.float32(case["eps"])), case["dt"]
        acc = _direct_sum(pos, m, eps)
        for _ in range(case["steps"]):
            v = v + 0.5 * dt * acc
            x = x + dt * v
            acc = _direct_sum(x.cpu().numpy(), m, eps)
            v = v + 0.5 * dt * acc
        return {"pos": x.cpu().numpy(), "vel": v.cpu().numpy()}
    if kind == "lffgrad":
        x, y = (torch.as_tensor(a.astype(np.float64), device="cuda")
                for a in _lff_rows(case["n"], seed))
        p = torch.as_tensor(_lff_params(seed).astype(np.float64), device="cuda")
        p.requires_grad_(True)
        w1, b1, w2, b2, w3, b3 = torch.split(p, LFF_SIZES)
        h = torch.nn.functional.silu(x @ w1.view(32, 64) + b1)
        h = torch.nn.functional.silu(h @ w2.view(64, 64) + b2)
        loss = ((h @ w3.view(64, 3) + b3 - y) ** 2).sum(1).mean()
        loss.backward()
        return {"grad": p.grad.cpu().numpy(), "loss": float(loss.detach())}
    return None
