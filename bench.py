"""Benchmark: J-tensor grid points/s on one MI355X, mixed precision vs FP64.

Workload (one step): the full J tensor on every point of a 128^3 grid
(0.12 bohr spacing) around a 60-atom carbon cage (truncated icosahedron,
radius 6.7 bohr) with a 4s3p2d1f spherical basis per atom (nbf 1800),
nocc 180, seeded synthetic densities.  Points and results stay in HBM.
`value` is the mixed-precision rate (FP32 operands split into three BF16
parts, six BF16 MFMA products, FP32 accumulation, FP64 tensor assembly); the FP64 GPU path, the plane-flux error of mixed against FP64, the
contraction kernel's roofline position and the reference CPU code timed on
this host are reported beside it.

    python bench.py [--steps K] [--warmup W] [--gpus 1]

Other workloads (one JSON line each; not the headline):
    --workload scan      256 uneven Gauss-Lobatto planes across a bond of a
                         30-atom sheet, one hipGraph launch per scan
    --workload openshell 200-atom sheet, alpha/beta densities (8 matrices),
                         charge and spin current on a 192x192x96 grid
    --workload surrogate learned J field of the 60-atom cage on a 256^3 grid
                         with exact-kernel fallback
    --workload property  shielding of all 60 nuclei and the magnetizability of
                         the cage on per-atom product grids (jfield.f90:584-929)
"""
import argparse
import json
import os
import sys
import tempfile
import time

import numpy as np

ROOT = os.path.dirname(os.path.abspath(__file__))
sys.path.insert(0, ROOT)

PEAK_TFLOPS = {"mixed": 2500.0, "fp64": 78.6, "fp32": 157.3}  # MI355X dense MFMA (bf16, fp64, fp32)
HBM_GBS = 8000.0


def log(*a):
    print(*a, file=sys.stderr, flush=True)


def plane_grid(system):
    """bond plane through the cage: atoms 1 and its nearest neighbour"""
    from gimic_amd import grid as gridmod
    c = np.asarray(system.coords)
    d = np.linalg.norm(c - c[0], axis=1)
    d[0] = np.inf
    j = int(np.argmin(d))
    kw = {"_arg": "bond", "type": "lobatto", "gauss_order": 7, "bond": [1, j + 1],
          "fixcoord": [0.0, 0.0, 0.0], "distance": float(d[j] / 2), "height": [-7.0, 7.0],
          "width": [-7.0, 7.0], "grid_points": [140, 140, 0]}
    g = gridmod.new_grid(kw, c)
    return g, gridmod.get_magnet(g, "X")


def time_steps(ctx, d_pts, out, precision, steps, warmup):
    import torch
    for _ in range(warmup):
        ctx.jtensor_device(d_pts, precision=precision, out=out)
    torch.cuda.synchronize()
    e0 = torch.cuda.Event(enable_timing=True)
    e1 = torch.cuda.Event(enable_timing=True)
    t0 = time.perf_counter()
    e0.record()
    for _ in range(steps):
        ctx.jtensor_device(d_pts, precision=precision, out=out)
    e1.record()
    torch.cuda.synchronize()
    wall = time.perf_counter() - t0
    return e0.elapsed_time(e1) / steps, wall


def kernel_roofline(ctx, d_pts, out, precision, nbf):
    """Two extra passes: one that counts the screening lists of every row
    tile (a tile of R rows with k live 8-function groups multiplies
    R x 8k by 8k x 7*8k: 14 R (8 k)^2 flops; the mixed kernel walks these
    groups along N and K, the FP64 kernel the live granules of four functions
    in them, up to a fifth fewer pairs, so its figure is an upper bound), and
    one with event timing around each kernel launch.  achieved = listed flops per launch / average launch time; the
    dense product would need 14 nbf^2 per point."""
    import torch
    # these passes measure the mixed contraction kernel alone: the FP64 pass
    # over points next to a nucleus (counted in the step time) is left out
    radius = ctx.fp64_refined()[0]
    ctx.set_fp64_radius(0.0)
    ctx.set_tile_stats(True)
    ctx.jtensor_device(d_pts, precision=precision, out=out)
    torch.cuda.synchronize()
    ts = ctx.tile_stats()
    ctx.set_tile_stats(False)
    ctx.set_timing(True)
    ctx.jtensor_device(d_pts, precision=precision, out=out)
    torch.cuda.synchronize()
    t = ctx.get_timing()
    ctx.set_timing(False)
    ctx.set_fp64_radius(radius)
    ms, launches = t["contract"]
    npts = d_pts.shape[0]
    dense = 14.0 * nbf * nbf * npts
    if ts["tiles"] > 0:
        # live 8-function groups along N and K (FP64: an upper bound)
        pairs = ts["groups_sq"] * 64.0
        flop = 14.0 * ts["tile_rows"] * pairs
        block_pairs = pairs / (ts["tiles"] * (32.0 * ts["nblk"]) ** 2)
    else:  # a dense kernel
        flop, block_pairs = dense, 1.0
    avg_ms = ms / launches
    achieved = flop / launches / avg_ms / 1e9  # TFLOP/s per launch average
    return dict(bound="mfma", achieved=round(achieved, 2), peak=PEAK_TFLOPS[precision],
                unit="TFLOP/s", frac=round(achieved / PEAK_TFLOPS[precision], 4), traffic=None,
                kernel="contract_mx2_kernel" if precision != "fp64" else "contract_f64_kernel",
                avg_launch_ms=round(avg_ms, 3), launches=launches,
                flop_per_launch=flop / launches, dense_flop_per_launch=dense / launches,
                listed_block_pairs=round(block_pairs, 4),
                points_per_launch=npts / launches), t


def measured_traffic(kernel, split, points_per_launch):
    """HBM-side bytes per launch from the committed rocprofv3 --pmc summary
    (FETCH_SIZE and WRITE_SIZE of the same kernel and split on this workload,
    calibrated against a 1 GiB copy), or None when none matches"""
    path = os.path.join(ROOT, "profiles", "contract_mx2_traffic_cage60.md")
    if not os.path.exists(path):
        return None
    for line in open(path):
        f = line.split()
        if len(f) == 4 and f[0] == "traffic_bytes_per_point" and f[1] == kernel and \
                f[2] == f"split={split}":
            return float(f[3]) * points_per_launch
    return None


def cpu_baseline(system, budget_s=15.0):
    """reference (flang-built oracle/_ref/ref_driver) on a bounded sample"""
    from oracle import molio, refrun, sph
    if not refrun.available():
        return None
    # every core this process may use: the OpenMP thread count the host
    # sets for it (a GPU host gives one GPU's job its share of the cores),
    # else the cores in its affinity mask
    nproc = os.cpu_count() or 1
    threads = int(os.environ.get("OMP_NUM_THREADS") or len(os.sched_getaffinity(0)) or 1)
    b = molio.Basis()
    b.symbols, b.charges, b.coords = system.symbols, system.charges, system.coords
    b.shell_atom, b.shell_l, b.shell_nprim, b.shell_poff = (system.shell_atom, system.shell_l,
                                                             system.shell_nprim, system.shell_poff)
    b.exps, b.coefs = system.exps, system.coefs
    dcart = sph.to_cartesian(system.dens, system.shell_l)
    rng = np.random.default_rng(3)
    from gimic_amd import synth
    pts = synth.cube_grid(128, 0.12, -7.62)
    with tempfile.TemporaryDirectory() as td:
        mol = os.path.join(td, "MOL")
        molio.write_mol(mol, b)
        flat = molio.pack_dens(dcart)
        sample = pts[rng.choice(len(pts), 64, replace=False)]
        _, t = refrun.ref_jtensor(mol, sample, dens=flat, screening=1e-8, threads=threads,
                                  return_time=True)
        n = int(min(len(pts), max(64, budget_s / max(t, 1e-6) * 64)))
        n = (n // threads) * threads or threads
        sample = pts[rng.choice(len(pts), n, replace=False)]
        _, t = refrun.ref_jtensor(mol, sample, dens=flat, screening=1e-8, threads=threads,
                                  return_time=True)
        if t < 0.5 * budget_s and n < len(pts):
            # the small probe overstates the time per point (thread start-up):
            # size the sample once more from this run
            n = int(min(len(pts), n * budget_s / max(t, 1e-6)))
            n = (n // threads) * threads or threads
            sample = pts[rng.choice(len(pts), n, replace=False)]
            _, t = refrun.ref_jtensor(mol, sample, dens=flat, screening=1e-8, threads=threads,
                                      return_time=True)
    return {"value": round(n / t, 2), "unit": "points/s", "cores": threads, "kind": "reference",
            "nproc": nproc, "affinity_cores": len(os.sched_getaffinity(0)),
            "sample": f"{n} random points of the 128^3 grid, flang-built reference "
                      f"(oracle/_ref/ref_driver, -O3 -fopenmp, OpenMP over points on {threads} "
                      f"threads), cartesian-equivalent density D_cart = T^T D T, loop time "
                      f"{t:.2f} s"}


def bench_scan(args):
    """A scan step is one flux_plane_grids call: the device generates every
    plane's points and weights from its 1-D rules, evaluates the tensors and
    sums the flux, in one hipGraph launch.  The same planes passed as host
    point arrays (flux_planes) are timed beside it."""
    import torch
    from gimic_amd import flux, synth
    system = synth.sheet30()
    ctx = system.context(screening=1e-8)
    ctx.set_chunk_bytes(-1)  # the large chunk: a third of device memory
    scan = synth.scan_planes(system)
    grids, fields = [g for g, _ in scan], [b for _, b in scan]
    planes = [flux.plane_of(g, b) for g, b in scan]
    npts = sum(len(p["weights"]) for p in planes)
    res = {}
    for prec in ("mixed", "fp64"):
        out = {}
        for mode in ("eager", "graph", "graph_host_arrays"):
            ctx.set_graph(mode != "eager")
            if mode == "graph_host_arrays":
                call = lambda: ctx.flux_planes(planes, precision=prec, modulus=True)
            else:
                call = lambda: ctx.flux_plane_grids(grids, fields, precision=prec, modulus=True)
            for _ in range(args.warmup):
                call()
            t0 = time.perf_counter()
            for _ in range(args.steps):
                f, m = call()
            out[mode] = (time.perf_counter() - t0) / args.steps
            if mode == "graph":
                fg = f
            elif mode == "graph_host_arrays":
                assert np.array_equal(f, fg), "device-generated and host planes differ"
        res[prec] = dict(flux=fg, ms=out)
    ctx.close()
    f64, fmx = res["fp64"]["flux"], res["mixed"]["flux"]
    rel = np.abs(fmx[:, 0] - f64[:, 0]) / np.maximum(np.abs(f64[:, 0]), 1e-300)
    big = np.abs(f64[:, 0]) >= 1e-3 * np.abs(f64[:, 0]).max()
    t = res["mixed"]["ms"]["graph"]
    return {
        "metric": "plane-scan J-tensor points/s (planes generated on the device, one hipGraph "
                  "launch per scan)",
        "value": round(npts / t, 1), "unit": "points/s", "n_gpus": 1, "steps": args.steps,
        "warmup": args.warmup, "ms_per_step": round(1e3 * t, 3), "higher_is_better": True,
        "dtype": "fp32 (bf16x6 MFMA), fp64 assembly", "data": "synthetic",
        "config": {"workload": "sheet30 tetracene C18H12, nbf 312, nocc 60; 256 planes "
                               "perpendicular to bond 1-2, offsets -6..+6 bohr, order-7 "
                               "Lobatto, 40..120 x 60..200 points per plane",
                   "points_per_step": int(npts), "planes": len(planes)},
        "wall_ms": {p: {m: round(1e3 * v, 3) for m, v in res[p]["ms"].items()} for p in res},
        "mixed_over_fp64": round(res["fp64"]["ms"]["graph"] / t, 3),
        "error": {"flux_rel_max": float(rel[big].max()), "flux_rel_median": float(np.median(rel)),
                  "planes_checked": int(big.sum())},
    }


def bench_openshell(args):
    import torch
    from gimic_amd import synth
    system = synth.sheet200()
    ctx = system.context(screening=1e-8)
    ctx.set_chunk_bytes(-1)  # the large chunk: a third of device memory
    pts = np.stack(np.meshgrid(0.2 * np.arange(192) - 19.1, 0.2 * np.arange(192) - 19.1,
                               0.2 * np.arange(96) - 9.5, indexing="ij"), -1)
    pts = pts.transpose(2, 1, 0, 3).reshape(-1, 3)  # x fastest
    d_pts = torch.tensor(pts, dtype=torch.float64, device="cuda")
    npts = len(pts)
    spins = ["total", "spindens"]  # charge and spin current, 8 matrices
    out = torch.empty((2, npts, 9), dtype=torch.float64, device="cuda")
    ms = {}
    for prec in ("mixed", "fp64"):
        for _ in range(args.warmup):
            ctx.jtensor_multi_device(d_pts, spins, precision=prec, out=out)
        torch.cuda.synchronize()
        t0 = time.perf_counter()
        for _ in range(args.steps):
            ctx.jtensor_multi_device(d_pts, spins, precision=prec, out=out)
        torch.cuda.synchronize()
        ms[prec] = 1e3 * (time.perf_counter() - t0) / args.steps
        if prec == "mixed":
            Jm = out.clone()
    err = {}
    for k, name in enumerate(("charge", "spin")):
        d = torch.linalg.norm(Jm[k] - out[k], dim=1)
        nb = torch.linalg.norm(out[k], dim=1)
        e = (d / torch.clamp(nb, min=1e-3 * float(nb.max()))).cpu().numpy()
        err[name] = {"tensor_rel_max": float(e.max()), "tensor_rel_p99": float(np.quantile(e, 0.99)),
                     "field_rel": float(torch.linalg.norm(Jm[k] - out[k]) / torch.linalg.norm(out[k]))}
    ctx.close()
    return {
        "metric": "open-shell J-tensor points/s (charge + spin, 8 matrices)",
        "value": round(npts / (ms["mixed"] / 1e3), 1), "unit": "points/s", "n_gpus": 1,
        "steps": args.steps, "warmup": args.warmup, "ms_per_step": round(ms["mixed"], 3),
        "higher_is_better": True, "dtype": "fp32 (bf16x6 MFMA), fp64 assembly",
        "data": "synthetic",
        "config": {"workload": "sheet200 C180H20, nbf 2620, alpha/beta nocc 610/600, "
                               "192x192x96 grid at 0.2 bohr", "points_per_step": npts,
                   "nbf": system.nbf},
        "fp64_gpu": {"value": round(npts / (ms["fp64"] / 1e3), 1), "ms_per_step": round(ms["fp64"], 3)},
        "mixed_over_fp64": round(ms["fp64"] / ms["mixed"], 3),
        "error": err,
    }


def atom_product_grids(coords, rmax=6.0, nr=24, nt=12, nphi=24):
    """per atom a product grid: Gauss-Legendre in r on [0, rmax] and in
    cos(theta), trapezoid in phi (a stand-in for numgrid's per-atom blocks)"""
    xr, wr = np.polynomial.legendre.leggauss(nr)
    rr = 0.5 * rmax * (xr + 1.0)
    wr = 0.5 * rmax * wr * rr ** 2
    ct, wt = np.polynomial.legendre.leggauss(nt)
    ph = 2.0 * np.pi * np.arange(nphi) / nphi
    R, CT, PH = np.meshgrid(rr, ct, ph, indexing="ij")
    W = (wr[:, None, None] * wt[None, :, None] * (2.0 * np.pi / nphi)).repeat(nphi, axis=2)
    st = np.sqrt(1.0 - CT ** 2)
    local = np.stack([R * st * np.cos(PH), R * st * np.sin(PH), R * CT], axis=-1).reshape(-1, 3)
    pts = np.concatenate([local + c for c in coords])
    return pts, np.tile(W.reshape(-1), len(coords)), np.full(len(coords), local.shape[0])


def bench_property(args):
    """shielding of all 60 nuclei + magnetizability (jfield.f90:584-929) on
    per-atom product grids of the cage: J at every point and the 61 weighted
    sums per point block; host arrays in and out, as the drop-in reads them
    from numgrid files"""
    from gimic_amd import synth
    system = synth.cage60()
    ctx = system.context(screening=1e-8)
    ctx.set_chunk_bytes(-1)  # the large chunk: a third of device memory
    coords = np.asarray(system.coords)
    pts, w, sizes = atom_product_grids(coords)
    npts = len(pts)
    ms, res = {}, {}
    # "mixed_all": the mixed path without the FP64 pass near the nuclei
    # (radius 0), which on atom-centred grids covers many points
    radius = ctx.fp64_refined()[0]
    for prec in ("mixed", "fp64", "mixed_all"):
        ctx.set_fp64_radius(0.0 if prec == "mixed_all" else radius)
        p = "mixed" if prec == "mixed_all" else prec
        for _ in range(args.warmup):
            ctx.properties(pts, w, sizes, coords, precision=p)
        t0 = time.perf_counter()
        for _ in range(args.steps):
            res[prec] = ctx.properties(pts, w, sizes, coords, precision=p)
        ms[prec] = 1e3 * (time.perf_counter() - t0) / args.steps
        if prec == "mixed":
            refined = ctx.fp64_refined()[1]
    iso = {p: res[p]["shield"].sum(axis=1)[:, :3].sum(axis=1) / 3.0 for p in res}
    chi = {p: res[p]["magnet"].sum(axis=0)[:3].sum() / 3.0 for p in res}
    ctx.close()
    return {
        "metric": "property-grid points/s (J + shielding of every nucleus + magnetizability)",
        "value": round(npts / (ms["mixed"] / 1e3), 1), "unit": "points/s", "n_gpus": 1,
        "steps": args.steps, "warmup": args.warmup, "ms_per_step": round(ms["mixed"], 3),
        "higher_is_better": True, "dtype": "fp32 (bf16x6 MFMA), fp64 assembly and sums",
        "data": "synthetic",
        "config": {"workload": "cage60 (nbf 1800), 60 per-atom product grids of 24 x 12 x 24 points "
                               "(r <= 6 bohr), shielding of all 60 nuclei and the magnetizability; "
                               "host arrays in and out", "points_per_step": npts},
        "fp64_gpu": {"value": round(npts / (ms["fp64"] / 1e3), 1), "ms_per_step": round(ms["fp64"], 3)},
        "mixed_over_fp64": round(ms["fp64"] / ms["mixed"], 3),
        "fp64_near_nuclei": {"radius_bohr": radius, "points_per_step": refined,
                             "fraction": round(refined / npts, 4)},
        "mixed_without_fp64_near_nuclei": {
            "value": round(npts / (ms["mixed_all"] / 1e3), 1), "ms_per_step": round(ms["mixed_all"], 3),
            "over_fp64": round(ms["fp64"] / ms["mixed_all"], 3),
            "shielding_vs_fp64_max_abs_ppm": float(np.abs(iso["mixed_all"] - iso["fp64"]).max()),
            "magnetizability_vs_fp64_rel": float(abs(chi["mixed_all"] - chi["fp64"]) / abs(chi["fp64"]))},
        "results": {"shielding_iso_ppm_fp64": [round(float(iso["fp64"].min()), 4),
                                               round(float(iso["fp64"].max()), 4)],
                    "magnetizability_iso_au_fp64": float(chi["fp64"]),
                    "shielding_mixed_vs_fp64_max_abs_ppm": float(np.abs(iso["mixed"] - iso["fp64"]).max()),
                    "magnetizability_mixed_vs_fp64_rel": float(abs(chi["mixed"] - chi["fp64"]) /
                                                               abs(chi["fp64"]))},
    }


def bench_surrogate(args):
    """The learned surrogate on the 60-atom cage, 256^3 visualisation grid
    over [-7.68, 7.68]^3 bohr.  'stated': the workload as given -- exact
    kernel within 0.4 bohr of every nucleus, 2M training points (uniform plus
    Gaussian clouds of 1 bohr around the nuclei), 1% held out, a cell of the
    8^3 served only where its held-out error is within 1e-3.  'far_field'
    beside it: exact within 3 bohr, uniform samples, reported at looser
    tolerances, where the network does serve.  Each line times the hybrid
    evaluation (network on served points, exact mixed kernel on the rest)
    against the exact kernel alone and audits the served points with the
    exact FP64 kernel."""
    import torch
    from gimic_amd import synth
    from gimic_amd.surrogate import Surrogate
    system = synth.cage60()
    ctx = system.context(screening=1e-8)
    ctx.set_chunk_bytes(-1)  # the large chunk: a third of device memory
    half = 7.68
    ax = torch.linspace(-half, half, 256, dtype=torch.float64, device="cuda")
    z, y, x = torch.meshgrid(ax, ax, ax, indexing="ij")
    grid = torch.stack([x.ravel(), y.ravel(), z.ravel()], 1)
    del x, y, z
    n = grid.shape[0]
    out = torch.empty((n, 9), dtype=torch.float64, device="cuda")
    ctx.jtensor_device(grid, precision="mixed", out=out)
    torch.cuda.synchronize()
    t0 = time.perf_counter()
    ctx.jtensor_device(grid, precision="mixed", out=out)
    torch.cuda.synchronize()
    t_ex = time.perf_counter() - t0
    runs = {}
    for name, excl, near_frac in (("stated", 0.4, 0.5), ("far_field", 3.0, 0.0)):
        log(f"surrogate {name}")
        sg = Surrogate(ctx, np.asarray(system.coords), -half * np.ones(3), half * np.ones(3),
                       tol=1e-3, ncell=8, sigma=args.sigma, seed=3, exclusion=excl)
        st = sg.fit(n_train=2_000_000, steps=args.train_steps, batch=16384, lr=2e-3,
                    near_frac=near_frac)
        st.pop("loss_history", None)
        per_tol = {}
        for tol in (1e-3, 1e-2, 3e-2):
            sg.set_tolerance(tol)
            sg.evaluate(grid, out=out)
            torch.cuda.synchronize()
            t0 = time.perf_counter()
            J, served = sg.evaluate(grid, out=out)
            torch.cuda.synchronize()
            t_h = time.perf_counter() - t0
            per_tol[f"{tol:g}"] = {"served_fraction": round(float(served.float().mean()), 4),
                                   "points_per_s": round(n / t_h, 1),
                                   "gain_over_exact": round(t_ex / t_h, 3),
                                   "audit": sg.audit(grid, J, served)}
        runs[name] = {"exclusion_bohr": excl, "near_frac": near_frac, "training": st,
                      "by_tolerance": per_tol}
        sg.net.close()
    ctx.close()
    head = runs["stated"]["by_tolerance"]["0.001"]
    return {
        "metric": "visualisation-grid J-tensor points/s with learned surrogate + exact fallback",
        "value": head["points_per_s"], "unit": "points/s", "n_gpus": 1, "steps": 1, "warmup": 1,
        "higher_is_better": True,
        "dtype": "bf16 MFMA (fp32 master weights); fallback fp32 (bf16x6 MFMA)",
        "data": "synthetic",
        "config": {"workload": "cage60 (nbf 1800) on a 256^3 grid over [-7.68, 7.68]^3 bohr; "
                               "2M exact-kernel training points, 1% held out, 8^3 cells; "
                               "tolerance 1e-3, exact within 0.4 bohr of every nucleus",
                   "points_per_step": n},
        "tolerance_1e-3": head, "exact_only_points_per_s": round(n / t_ex, 1), "runs": runs,
    }


def main():
    ap = argparse.ArgumentParser()
    ap.add_argument("--gpus", type=int, default=1)
    ap.add_argument("--steps", type=int, default=3)
    ap.add_argument("--warmup", type=int, default=1)
    ap.add_argument("--no-cpu", action="store_true", help="skip the CPU reference baseline")
    ap.add_argument("--points", type=int, default=0, help="limit points (profiling)")
    ap.add_argument("--workload", default="cage60",
                    choices=["cage60", "scan", "openshell", "surrogate", "property"])
    ap.add_argument("--train-steps", type=int, default=12000, help="surrogate training steps")
    ap.add_argument("--sigma", type=float, default=1.0, help="surrogate Fourier frequency scale")
    args = ap.parse_args()
    if args.gpus != 1 or int(os.environ.get("WORLD_SIZE", "1")) > 1:
        print("bench.py measures one GPU only: the workload is sharded by point tiles "
              "across GPUs by design but this build runs on a single MI355X.", file=sys.stderr)
        sys.exit(2)
    import torch
    from gimic_amd import flux, synth
    assert torch.cuda.is_available(), "no GPU"
    if args.workload != "cage60":
        fn = {"scan": bench_scan, "openshell": bench_openshell, "surrogate": bench_surrogate,
              "property": bench_property}
        print(json.dumps(fn[args.workload](args)))
        return
    dev = torch.device("cuda:0")
    log("setup cage60")
    system = synth.cage60()
    nbf = system.nbf
    pts = synth.cube_grid(128, 0.12, -7.62)
    if args.points:
        pts = pts[:args.points]
    npts = len(pts)
    ctx = system.context(screening=1e-8)
    # the large chunk (a third of device memory): the whole grid in one
    # mixed launch; the library's default is a modest 8 GiB
    ctx.set_chunk_bytes(-1)
    d_pts = torch.tensor(pts, dtype=torch.float64, device=dev)
    out = torch.empty((npts, 9), dtype=torch.float64, device=dev)

    log("timing mixed")
    ms_mixed, wall_mixed = time_steps(ctx, d_pts, out, "mixed", args.steps, args.warmup)
    fp64_radius, fp64_refined = ctx.fp64_refined()
    J_mixed_sample = out[:: max(1, npts // 65536)].cpu().numpy()
    roof, ktimes = kernel_roofline(ctx, d_pts, out, "mixed", nbf)
    variant, split, tune_ms = ctx.tuning()
    tuning_log = [[v, sp, round(t, 3)] for v, sp, t in ctx.tuning_log()]
    roof["kernel"] = {3: "contract_mx2_kernel<2,2,4>", 4: "contract_mx2_kernel<3,2,4>",
                      5: "contract_mx2_kernel<2,4,4>", 8: "contract_mx2_kernel<2,2,8>",
                      9: "contract_mx2_kernel<3,2,8>"}.get(variant, "?")
    roof["split"] = split
    # the mixed kernels issue six BF16 MFMA products per algorithmic product
    # (FP32 operands split into three BF16 parts): matrix-pipe use is 6x frac
    roof["mfma_issued_tflops"] = round(6.0 * roof["achieved"], 1)
    roof["mfma_issued_frac"] = round(6.0 * roof["achieved"] / roof["peak"], 4)
    # the arithmetic emulated is FP32 (products of FP32 operands, FP32
    # accumulation): against MI355X's dense FP32 matrix peak
    roof["over_fp32_mfma_peak"] = round(roof["achieved"] / PEAK_TFLOPS["fp32"], 3)
    roof["traffic"] = measured_traffic(roof["kernel"], split, roof["points_per_launch"])
    if roof["traffic"] is not None:
        roof["traffic_note"] = ("L2-miss bytes per launch (Infinity Cache + HBM), rocprofv3 FETCH_SIZE/"
                                "WRITE_SIZE calibrated on a 1 GiB copy; profiles/contract_mx2_traffic_cage60.md")
    log("timing fp64")
    ms_f64, wall_f64 = time_steps(ctx, d_pts, out, "fp64", args.steps, args.warmup)
    J_f64_sample = out[:: max(1, npts // 65536)].cpu().numpy()
    roof64, _ = kernel_roofline(ctx, d_pts, out, "fp64", nbf)
    roof64["flop_count"] = ("upper bound: live 8-function groups; the kernel walks the live "
                            "granules of four functions in them")

    nb = np.linalg.norm(J_f64_sample, axis=1)
    e = np.linalg.norm(J_mixed_sample - J_f64_sample, axis=1) / np.maximum(nb, 1e-3 * nb.max())
    log("host buffers")
    # PCIe-inclusive rate: host points in, host tensors out through
    # gimic_jtensor_batch (the second of two calls: the first sizes its
    # staging buffers; the headline keeps both in HBM)
    ctx.jtensor(pts, precision="mixed")
    t0 = time.perf_counter()
    ctx.jtensor(pts, precision="mixed")
    host_s = time.perf_counter() - t0
    log("plane flux")
    g, B = plane_grid(system)
    f64 = np.array(flux.integrate_current(ctx, g, B, precision="fp64"))
    fmx = np.array(flux.integrate_current(ctx, g, B, precision="mixed"))
    flux_err = float(abs(fmx[0] - f64[0]) / abs(f64[0]))
    ctx.close()

    cpu = None
    if not args.no_cpu:
        log("cpu baseline")
        cpu = cpu_baseline(system)

    value = npts / (ms_mixed / 1e3)
    res = {
        "metric": "J-tensor grid points/s, mixed vs FP64 GPU at <=1e-6 rel plane-flux error",
        "value": round(value, 1), "unit": "points/s", "n_gpus": 1, "steps": args.steps,
        "warmup": args.warmup, "ms_per_step": round(ms_mixed, 3), "higher_is_better": True,
        "scaling": "weak", "vs_baseline": None,
        "dtype": "fp32 (bf16x6 MFMA), fp64 assembly; fp64 within %.2f bohr of a nucleus" % fp64_radius,
        "data": "synthetic (seeded basis and densities)",
        "config": {"workload": "cage60 C60 truncated icosahedron r=6.7 bohr, 4s3p2d1f spherical "
                               "(nbf 1800), nocc 180, 128^3 grid at 0.12 bohr",
                   "points_per_step": npts, "nbf": nbf, "precision": "mixed (bf16x6 MFMA emulating fp32)"},
        "fp64_near_nuclei": {"radius_bohr": fp64_radius, "points_per_step": fp64_refined,
                             "fraction": round(fp64_refined / npts, 5),
                             "note": "points this close to a nucleus are evaluated again in FP64 "
                                     "inside the timed step"},
        "fp64_gpu": {"value": round(npts / (ms_f64 / 1e3), 1), "unit": "points/s",
                     "ms_per_step": round(ms_f64, 3), "roofline": roof64},
        "mixed_over_fp64": round(ms_f64 / ms_mixed, 3),
        "error": {"plane_flux_rel": flux_err, "plane_flux_fp64": f64.tolist(),
                  "plane_flux_mixed": fmx.tolist(), "tensor_rel_max": float(e.max()),
                  "tensor_rel_p99": float(np.quantile(e, 0.99)),
                  "tensor_sample_points": int(len(e))},
        "kernel_ms": {k: round(v[0], 3) for k, v in ktimes.items()},
        "mixed_kernel_tuning": {"chosen": variant, "split": split,
                                "candidates_ms": tuning_log},
        "roofline": roof,
        "cpu_baseline": cpu,
        "wall_s": {"mixed": round(wall_mixed, 3), "fp64": round(wall_f64, 3)},
        "host_buffers": {"points_per_s": round(npts / host_s, 1), "ms": round(1e3 * host_s, 3),
                         "note": "mixed, host points in and host tensors out (PCIe-inclusive)"},
    }
    print(json.dumps(res))


if __name__ == "__main__":
    main()
