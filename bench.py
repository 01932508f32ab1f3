"""Benchmark of the fused direct-minimisation evaluation on one MI355X.

One step = one energy + gradient evaluation (QR orthonormalisation,
G-sphere scatter, batched 3D FFTs, density, Hartree / external / kinetic /
LDA-x energies, potential and the full adjoint back to dE/dw) of the
8-atom conventional diamond Si cube: a = 10.26 bohr, Z = 14 Coulomb nuclei,
64^3 grid, 4x4x4 Monkhorst-Pack k-mesh (64 k), 32 bands, spherical cutoff
48 Ha (G_n = 17071), parameters N(0,1) from seed 0, FP64 throughout.

A second measurement, "convergence", times direct minimisation to
|E - E*| < 1e-6 Ha from the seeded start on the held-out strained 8-atom
cell (Z = 4, 64 k-points): preconditioned CG with the plain Teter-Payne-
Allan preconditioner against the learned preconditioner (with and without
the learned warm start).

Prints ONE JSON line (rank 0).  Flags: --gpus N (only 1 is supported: the
path runs on one GPU), --steps K, --warmup W, --no-cpu-baseline,
--cpu-seconds S (target length of the CPU baseline sample),
--no-convergence, --conv-seconds S (time cap of each convergence run),
--no-batch, --batch-steps K (the uneven-structure batch section),
--traffic-probe (the workload of the rocprofv3 counter runs),
--no-large-cell, --large-cell-steps K, --large-cell-probe (the 128^3 /
128-band section and its rocprofv3 workload), --no-small-cell,
--no-band-structure, --band-probe (the band-mode rocprofv3 workload),
--no-normcons, --normcons-probe (the norm-conserving rocprofv3 workload).

A third section, "batch", times Adam steps (energy + gradient + update) of
16 uneven structures run as one batch: eager, over several streams, and as
a replayed hipGraph.

A fifth, "small_cell", times the reference's own CPU-sized case (2-atom FCC
Si, 32^3, 8 k, 8 bands) launched eagerly and replayed as a captured HIP
graph.

A fourth, "large_cell", times evaluations of the 64-atom Si cell at the
Gamma point (128^3 box, 128 bands) with the FP64 MFMA rate of its QR
passes.

A sixth, "band_structure", runs the band driver on the reference's Si band
example (60-point path, 28 bands, 64^3): its whole Adam schedule, and the
path with CG at each k-point.

A seventh, "normcons", times evaluations of the reference's
norm-conserving diamond example (48^3, 8 k, 14 bands, local part and
non-local projectors).
"""
import argparse
import json
import os
import sys
import time

METRIC = ("wall-time to |ΔE|<1e-6 Ha (learned vs plain precond); "
          "energy+grad evals/s")
HBM_PEAK_GBS = 8000.0


def algorithmic_bytes(cls, plan, chunks):
  """Algorithmic HBM bytes of ALL launches of one kernel class in one
  evaluation (each array read or written once; complex128 = 16 B)."""
  S = plan.ns * plan.nk * plan.nb
  ng = plan.num_g
  nx, ny, nz = plan.grid_sizes
  N = nx * ny * nz
  P = plan.ns * plan.nk
  nxa = plan.active_planes
  if getattr(plan, "row_path", False):
    # row buffer R[state][z][row]: z-transformed mask rows of all states
    T = S * nz * plan.num_rows * 16
  else:
    T = S * nxa * ny * nz * 16    # intermediate planes of all states
  Q = S * ng * 16                 # orthonormal coefficients
  W = 2 * S * ng * 8              # planar parameters (or gradient)
  rho = plan.ns * N * 8
  # (T: the plane buffer, or on the row path the row buffer R)
  if cls in ("plane_ifft", "row_ifft"):   # reads Q, writes T, per sweep
    return (1 if plan.keep_planes else 2) * (Q + T)
  if cls in ("xline_density", "zplane_density"):  # read T; rho per chunk
    return T + chunks * 2 * rho
  if cls in ("xline_vpsi", "zplane_vpsi"):  # read T, write T, read v
    return 2 * T + chunks * rho
  if cls in ("plane_fft_gather", "row_fft_gather"):  # T, Q in; Qbar out
    return T + 2 * Q
  if cls == "qr_gram":            # two Gram passes over W
    return 2 * W
  if cls == "qr_apply":           # read W, write Q
    return W + Q
  if cls == "qr_bwd_gram":        # read Q, Qbar
    return 2 * Q
  if cls == "qr_bwd_apply":       # read Q, Qbar, write dW
    return 2 * Q + W
  return None


def cpu_host():
  """Host facts the CPU figure depends on."""
  model = None
  try:
    with open("/proc/cpuinfo") as f:
      model = next((ln.split(":", 1)[1].strip() for ln in f
                    if ln.startswith("model name")), None)
  except OSError:
    pass
  return {"nproc": os.cpu_count(), "cpu_model": model,
          "OMP_NUM_THREADS": os.environ.get("OMP_NUM_THREADS")}


def cpu_band_step(target_s, nthreads):
  """Band-mode steps (trace and gradient, oracle/band.py) of the Si band
  example's first k-point on the host, per second; the same synthetic
  density as band_structure_bench, built on the host by the oracle."""
  sys.path.insert(0, os.path.dirname(os.path.abspath(__file__)))
  import numpy as np
  from threadpoolctl import threadpool_limits
  from jrystal_amd import band
  from oracle import adjoint as OA
  from oracle import band as OB
  from oracle import grid as OG
  from oracle import pw as OP
  from oracle.crystal import Crystal
  OP.set_workers(nthreads)
  limits = threadpool_limits(limits=nthreads)
  cr = Crystal.create_from_file(os.path.join(
    os.path.dirname(os.path.abspath(__file__)), "jrystal_amd", "geometry",
    "si.xyz"))
  gs = [64, 64, 64]
  mask = OG.spherical_mask(cr.cell_vectors, gs, 100.0)
  g = OG.g_vectors(cr.cell_vectors, gs)
  k0 = band.get_k_path(cr.cell_vectors, "LGXL", 60)[0:1]
  gsprob = OA.Problem(mask=mask, g_vector_grid=g, kpts=np.zeros((1, 3)),
                      vol=cr.vol, occupation=2.0 * np.ones((1, 1, 14)),
                      positions=cr.positions,
                      charges=np.asarray(cr.charges, float))
  rho = OA.energy_and_grad(OP.param_init(0, 14, 1, mask, dist="uniform"),
                           gsprob, want_grad=False)[2]
  prob = OA.Problem(mask=mask, g_vector_grid=g, kpts=k0, vol=cr.vol,
                    occupation=np.ones((1, 1, 28)), positions=cr.positions,
                    charges=np.asarray(cr.charges, float))
  v = OB.effective_potential(rho, prob)
  p = OP.param_init(123, 28, 1, mask, dist="uniform")
  OB.hamiltonian_trace(p, prob, v)  # warm-up
  n, t0 = 0, time.perf_counter()
  while time.perf_counter() - t0 < target_s:
    OB.hamiltonian_trace(p, prob, v)
    n += 1
  t = time.perf_counter() - t0
  limits.unregister()
  return {"value": n / t, "unit": "band-mode trace+gradient evaluations/s",
          "cores": nthreads, "kind": "port",
          "sample": (f"{n} evaluations ({t:.2f} s) of the Si band example's "
                     f"first k-point (12939 coefficients x 28 bands, 64^3); "
                     f"oracle/ NumPy+SciPy FP64, scipy.fft workers="
                     f"{nthreads}")}


def cpu_baseline(wl, params, target_s, nthreads):
  """Oracle (NumPy/SciPy restatement of the reference) on a k-point subset
  of the same workload, scaled to whole evaluations per second; FFT
  workers and BLAS threads both set to nthreads."""
  sys.path.insert(0, os.path.dirname(os.path.abspath(__file__)))
  import numpy as np
  from threadpoolctl import threadpool_limits
  from oracle import adjoint as OA
  from oracle import grid as OG
  from oracle import occupation as OO
  from oracle import pw as OP
  OP.set_workers(nthreads)
  limits = threadpool_limits(limits=nthreads)
  cr = wl.crystal
  nk_full = wl.kpts.shape[0]

  def problem(nk_s):
    kp = OG.k_vectors(cr.cell_vectors, wl.k_grid)[:nk_s]
    occ = OO.uniform(nk_full, cr.num_electron, 0, wl.num_bands)[:, :nk_s]
    return OA.Problem(mask=OG.spherical_mask(cr.cell_vectors,
                                             list(wl.grid_sizes),
                                             wl.cutoff_energy),
                      g_vector_grid=OG.g_vectors(cr.cell_vectors,
                                                 list(wl.grid_sizes)),
                      kpts=kp, vol=cr.vol, occupation=occ,
                      positions=cr.positions,
                      charges=np.asarray(cr.charges, float))

  def run(nk_s):
    prob = problem(nk_s)
    p = {k: v[:, :nk_s] for k, v in params.items()}
    t = time.perf_counter()
    OA.energy_and_grad(p, prob, k_chunk=min(nk_s, 8))
    return time.perf_counter() - t

  run(1)  # warm-up (FFT plans, page-in)
  t1 = run(1)
  nk_s = int(max(1, min(nk_full, round(target_s / max(t1, 1e-3)))))
  t = run(nk_s)
  limits.unregister()
  evals_per_s = nk_s / (t * nk_full)
  return {"value": evals_per_s, "unit": "energy+gradient evaluations/s",
          "cores": nthreads, "kind": "port",
          "sample": (f"one energy+gradient evaluation of the same system "
                     f"restricted to {nk_s} of {nk_full} k-points "
                     f"({t:.2f} s), scaled by {nk_full}/{nk_s}; oracle/ "
                     f"NumPy+SciPy FP64 restatement, scipy.fft workers="
                     f"{nthreads}, BLAS threads {nthreads}")}


def time_to(history, e_star, tol):
  """First (seconds, index) of a (seconds, energy) history within tol."""
  for i, (t, e) in enumerate(history):
    if e - e_star < tol:
      return t, i
  return None, None


def convergence(time_cap, tol=1e-6):
  """Wall time to |E - E*| < tol from the seeded start, plain (TPA) against
  learned preconditioning, on the held-out strained 8-atom cell (Z = 4,
  64^3 grid, 4x4x4 k-mesh, 32 bands, 48 Ha): E* = the lowest energy any of
  the runs reaches (each run continues to convergence or time_cap).  The
  clock of every run starts with the seeded start resident on the device;
  the warm start's own evaluation and network pass are inside it."""
  import torch
  from jrystal_amd import learned, workloads
  from jrystal_amd.minimize import PLAIN_RESTART, Minimizer
  from jrystal_amd.objective import EnergyPlan
  if not os.path.exists(learned.DEFAULT_MODEL):
    print("bench: no trained preconditioner model; convergence skipped",
          file=sys.stderr)
    return None, None
  wl = workloads.si8_strained(4.0, k=4)
  plan = EnergyPlan.from_workload(wl)
  net = learned.PrecondNet.load(learned.DEFAULT_MODEL)
  runs = {}
  e_best = None
  p = wl.params(0)
  start = {k: torch.tensor(p[k], device=plan.device) for k in ("w_re", "w_im")}
  # untimed first use of every kernel and torch operation the runs share
  # (the first run would otherwise pay the loading for all of them)
  plan.evaluate(start["w_re"], start["w_im"], grad=True)
  warm = learned.LearnedFactor(plan, net)
  learned.density_stats(plan, warm.stats)
  learned.apply(plan, net, warm.stats,
                gap=learned.band_gaps(plan) if net.use_gap else None,
                factor=warm.factor)
  # and short runs of both minimisers (CG vector kernels, gauge resets,
  # the factor from its first refresh on): the first timed run would
  # otherwise pay the loading of everything it shares with the others
  Minimizer(plan, start, restart=PLAIN_RESTART).run(max_iter=40)
  Minimizer(plan, start, factor_fn=learned.LearnedFactor(plan, net),
            restart=learned.LEARNED_RESTART,
            first_restart=learned.LEARNED_FIRST_RESTART).run(max_iter=40)
  torch.cuda.synchronize()
  for mode in ("learned", "learned_warm", "plain"):
    print(f"bench: convergence run {mode}", file=sys.stderr, flush=True)
    torch.cuda.synchronize()
    t0 = time.perf_counter()
    p0 = start
    if mode == "learned_warm":
      p0 = learned.warm_start(plan, net, p0)
    fn = None if mode == "plain" else learned.LearnedFactor(plan, net)
    if mode == "plain":
      m = Minimizer(plan, p0, restart=PLAIN_RESTART)
    else:
      m = Minimizer(plan, p0, factor_fn=fn, restart=learned.LEARNED_RESTART,
                    first_restart=learned.LEARNED_FIRST_RESTART)
    t_setup = time.perf_counter() - t0
    stop = None if e_best is None else e_best + 0.1 * tol
    r = m.run(max_iter=100000, time_limit=time_cap, e_stop=stop)
    r.history = [(t + t_setup, e) for t, e in r.history]
    runs[mode] = r
    e_best = r.energy if e_best is None else min(e_best, r.energy)
  e_star = min(r.energy for r in runs.values())
  out = {"workload": wl.name, "tol_Ha": tol, "E_star_Ha": e_star,
         "time_cap_s": time_cap,
         "schedule": {"plain_restart": PLAIN_RESTART,
                      "learned_restart": learned.LEARNED_RESTART,
                      "learned_plain_first_cycle": (
                        learned.LEARNED_FIRST_RESTART),
                      "line_search": "parabola"}}
  for mode, r in runs.items():
    t, i = time_to(r.history, e_star, tol)
    out[mode] = {"seconds": t, "iterations": i,
                 "evaluations_total": r.evaluations,
                 "final_E_Ha": r.energy, "status": r.status,
                 "fallbacks": r.fallbacks}
  tp, tl = out["plain"]["seconds"], out["learned"]["seconds"]
  out["speedup_learned_vs_plain"] = (tp / tl) if tp and tl else None
  tw = out["learned_warm"]["seconds"]
  out["speedup_learned_warm_vs_plain"] = (tp / tw) if tp and tw else None
  return out, (wl, runs["plain"])


def batch_bench(steps, warmup, streams=4):
  """Adam steps of the 16 uneven structures of workloads.batch_cells(3)
  (grids 36^3-80^3, 1-64 k-points, 4-47 bands): eager on one stream, eager
  over `streams` streams, and the hipGraph-captured step replayed."""
  import numpy as np
  import torch
  from jrystal_amd import workloads
  from jrystal_amd.batch import BatchStep
  wls = workloads.batch_cells(seed=3, n=16)
  out = {"workload": "batch_cells(seed=3): 16 structures",
         "parameters": int(sum(np.prod(w.shape) for w in wls)),
         "states": int(sum(w.shape[0] * w.shape[1] * w.shape[3]
                           for w in wls))}
  for mode, ns, graph in (("eager_1_stream", 0, False),
                          (f"eager_{streams}_streams", streams, False),
                          (f"graph_{streams}_streams", streams, True)):
    print(f"bench: batch {mode}", file=sys.stderr, flush=True)
    bs = BatchStep(wls, streams=ns)
    if graph:
      bs.capture()
    run = bs.replay if graph else bs.step
    for _ in range(warmup):
      run()
    torch.cuda.synchronize()
    t0 = time.perf_counter()
    for _ in range(steps):
      run()
    torch.cuda.synchronize()
    dt = (time.perf_counter() - t0) / steps
    e = bs.energies()
    if not np.all(np.isfinite(e)):
      raise RuntimeError(f"batch {mode}: non-finite energies")
    out[mode] = {"ms_per_step": dt * 1e3,
                 "structure_evals_per_s": len(wls) / dt}
    bs.close()
    del bs
    torch.cuda.empty_cache()
  return out


FP64_MFMA_PEAK_TFLOPS = 78.6


def qr_flops(cls, plan):
  """Algorithmic real flops of one evaluation's launches of a QR class
  (complex multiply-add = 8 flops; triangular factors count their nonzero
  half): the Gram pass computes the nb(nb+1)/2 entries of a Hermitian
  matrix, the forward apply multiplies by an upper-triangular R^-1, the
  backward Gram is a full nb x nb product and the backward apply a
  triangular plus a full one."""
  P = plan.ns * plan.nk
  ng, nb = plan.num_g, plan.nb
  per = {"qr_gram": nb * (nb + 1) / 2, "qr_apply": nb * (nb + 1) / 2,
         "qr_bwd_gram": nb * nb, "qr_bwd_apply": nb * (nb + 1) / 2 + nb * nb}
  if cls not in per:
    return None
  return 8.0 * P * ng * per[cls]


def small_cell_bench(steps, warmup):
  """Energy + gradient evaluations of the reference's own CPU-sized case
  (2-atom FCC Si, 32^3, 8 k-points, 8 bands, 24 Ha): launched eagerly from
  the host, and replayed as one captured HIP graph (the case is bound by
  launch latency)."""
  import numpy as np
  import torch
  from jrystal_amd import workloads
  from jrystal_amd.objective import EnergyPlan
  wl = workloads.si2_fcc(14.0)
  p = wl.params(0)
  plan = EnergyPlan.from_workload(wl)
  wr = torch.tensor(p["w_re"], device=plan.device)
  wi = torch.tensor(p["w_im"], device=plan.device)
  out = {}
  print(f"bench: small cell {wl.name}", file=sys.stderr, flush=True)
  res = {"workload": wl.name, "grid": list(wl.grid_sizes),
         "num_kpts": int(plan.nk), "num_bands": int(plan.nb),
         "num_g": int(plan.num_g), "steps": steps}
  for _ in range(warmup):
    plan.evaluate(wr, wi, grad=True, out=out)
  torch.cuda.synchronize()
  t0 = time.perf_counter()
  for _ in range(steps):
    plan.evaluate(wr, wi, grad=True, out=out)
  torch.cuda.synchronize()
  dt = (time.perf_counter() - t0) / steps
  res["eager"] = {"ms_per_eval": dt * 1e3, "evals_per_s": 1.0 / dt}
  graph, gout = plan.capture(wr, wi)
  for _ in range(warmup):
    graph.replay()
  torch.cuda.synchronize()
  t0 = time.perf_counter()
  for _ in range(steps):
    graph.replay()
  torch.cuda.synchronize()
  dt = (time.perf_counter() - t0) / steps
  res["graph"] = {"ms_per_eval": dt * 1e3, "evals_per_s": 1.0 / dt}
  e = gout["energies"].tolist()
  if not np.all(np.isfinite(e)) or e != out["energies"].tolist():
    raise RuntimeError("small cell: graph replay differs from eager")
  res["energy_total_Ha"] = e[4]
  del graph
  plan.close()
  torch.cuda.empty_cache()
  return res


BAND_WORKLOAD = "si-fcc-64^3-100Ha-28b-LGXL-60k"


def _band_setup(num_kpoints=60, adam_first=10000, adam_rest=400):
  """(config, driver module, density, mask) of the reference's all-electron
  Si band example (tests/all_electron/si/config.yaml: geometry/si.xyz,
  64^3, spherical 100 Ha, 28 bands, the 60-point path LGXL, Adam with
  lr 0.001, 10000 steps at the first k-point and 400 at each of the
  others), with a synthetic fixed density: that of 14 seeded orbitals at
  Gamma (the cost of a band step does not depend on the density's
  values)."""
  import importlib
  import tempfile
  import numpy as np
  from jrystal_amd import config as C
  from jrystal_amd import pw
  from jrystal_amd.objective import EnergyPlan
  BD = importlib.import_module("jrystal_amd.calc.band_all_electrons")
  cfg = C.get_config()
  cfg.update(crystal="si", grid_sizes=64, cutoff_energy=100.0,
             freq_mask_method="spherical", empty_bands=14,
             band_structure_empty_bands=14, xc="lda_x",
             k_path_special_points="LGXL", num_kpoints=num_kpoints,
             band_structure_epoch=adam_first,
             k_path_fine_tuning_epoch=adam_rest, optimizer="adam",
             optimizer_args={"learning_rate": 0.001, "b1": 0.9, "b2": 0.99},
             seed=123, save_dir=tempfile.mkdtemp(prefix="jrx_band_"),
             verbose=False)
  cr = BD.create_crystal(cfg)
  mask = BD.create_freq_mask(cfg, cr)
  gsp = EnergyPlan(cr.positions, cr.charges, cr.cell_vectors, mask,
                   np.zeros((1, 3)), 2.0 * np.ones((1, 1, 14)))
  p0 = pw.param_init(0, 14, 1, mask)
  rho = gsp.evaluate(p0["w_re"], p0["w_im"], grad=False,
                     density=True)["density"].clone()
  gsp.close()
  return cfg, BD, rho, mask


class _GroundState:
  def __init__(self, density):
    self.density = density
    self.total_energy = 0.0


def band_structure_bench(adam_first=10000, adam_rest=400, num_kpoints=60,
                         chunked=0):
  """The band driver on the reference's Si band example (_band_setup): the
  whole Adam schedule on one chunk (the reference on one device), with
  ``chunked`` > 1 also on that many chunks at once (the reference's
  parallel_over_k_path on that many devices), and the path with
  preconditioned CG at each k-point."""
  import numpy as np
  import torch
  cfg, BD, rho, mask = _band_setup(num_kpoints, adam_first, adam_rest)
  _GS = _GroundState
  res = {"workload": BAND_WORKLOAD,
         "num_g": int(np.sum(np.asarray(mask))), "num_bands": 28,
         "num_kpoints": num_kpoints, "density": "synthetic (14 seeded "
         "orbitals at Gamma)"}
  runs = {}
  for chunks in (1, chunked) if chunked > 1 else (1,):
    print(f"bench: band structure (Adam schedule, {chunks} chunk(s))",
          file=sys.stderr, flush=True)
    cfg.update(k_path_chunks=chunks)
    r = BD.calc_with_output(cfg, ground_state=_GS(rho))
    per = num_kpoints // chunks
    res[f"adam_{chunks}_chunk" + ("s" if chunks > 1 else "")] = {
      "k_path_chunks": chunks,
      "steps": adam_first + (per - 1) * adam_rest,
      "evaluations": r.evaluations, "seconds": r.seconds,
      "ms_per_step": 1e3 * r.seconds / r.evaluations,
      "k_points_per_s": num_kpoints / r.seconds}
    runs[chunks] = r
  adam = runs[1]
  cfg.update(optimizer="cg", band_structure_epoch=400,
             k_path_fine_tuning_epoch=200, k_path_chunks=1)
  print("bench: band structure (CG)", file=sys.stderr, flush=True)
  cg = BD.calc_with_output(cfg, ground_state=_GS(rho))
  res["cg"] = {"evaluations": cg.evaluations, "seconds": cg.seconds,
               "k_points_per_s": num_kpoints / cg.seconds,
               "max_iter": [400, 200]}
  d = np.abs(adam.eigenvalues - cg.eigenvalues)
  res["max_abs_eig_diff_adam_vs_cg_Ha"] = float(np.max(d))
  res["trace_sum_lowest_adam_minus_cg_Ha"] = float(
    np.max(np.sum(adam.eigenvalues - cg.eigenvalues, axis=-1)))
  torch.cuda.empty_cache()
  return res


def large_cell_bench(steps, warmup):
  """Energy + gradient evaluations of the 64-atom Si cell at the Gamma
  point (128^3 box, 128 bands, 48 Ha, 137059 coefficients per band), with
  per-class durations, the HBM rate of the FFT passes and the FP64 MFMA
  rate of the QR passes."""
  import numpy as np
  import torch
  from jrystal_amd import workloads
  from jrystal_amd.objective import EnergyPlan
  wl = workloads.si64()
  p = wl.params(0)
  plan = EnergyPlan.from_workload(wl)
  wr = torch.tensor(p["w_re"], device=plan.device)
  wi = torch.tensor(p["w_im"], device=plan.device)
  out = {}
  print(f"bench: large cell {wl.name}", file=sys.stderr, flush=True)
  for _ in range(warmup):
    plan.evaluate(wr, wi, grad=True, out=out)
  torch.cuda.synchronize()
  t0 = time.perf_counter()
  for _ in range(steps):
    plan.evaluate(wr, wi, grad=True, out=out)
  torch.cuda.synchronize()
  dt = (time.perf_counter() - t0) / steps
  e = out["energies"].tolist()
  if not np.all(np.isfinite(e)):
    raise RuntimeError(f"large cell: non-finite energies {e}")
  plan.set_timing(True)
  nprof = 3
  for _ in range(nprof):
    plan.evaluate(wr, wi, grad=True, out=out)
  timing = plan.read_timing()
  plan.set_timing(False)
  if plan.row_path:
    timing = {ROW_PATH_CLASSES.get(k, k): v for k, v in timing.items()}
  res = {"workload": wl.name, "atoms": int(wl.crystal.num_atom),
         "grid": list(wl.grid_sizes), "num_bands": int(plan.nb),
         "num_g": int(plan.num_g), "steps": steps,
         "ms_per_eval": dt * 1e3, "evals_per_s": 1.0 / dt,
         "energy_total_Ha": e[4],
         "kernel_ms_per_eval": {k: round(v[0] / nprof, 4)
                                for k, v in timing.items()},
         "fft_hbm": {}, "qr_fp64_mfma": {}}
  chunks = plan.ns * max(1, -(-plan.nk * plan.nb // plan.chunk_states))
  for k, (ms, n) in timing.items():
    sec = ms / nprof * 1e-3
    b = algorithmic_bytes(k, plan, chunks)
    f = qr_flops(k, plan)
    if f is not None:
      tf = f / sec / 1e12
      res["qr_fp64_mfma"][k] = {"alg_tflops": tf,
                                "frac_of_peak": tf / FP64_MFMA_PEAK_TFLOPS}
    elif b is not None:
      gbs = b / sec / 1e9
      res["fft_hbm"][k] = {"alg_gbs": gbs, "frac_of_peak": gbs / HBM_PEAK_GBS}
  res["fp64_mfma_peak_tflops"] = FP64_MFMA_PEAK_TFLOPS
  res["mfma_counters"] = measured_mfma()
  plan.close()
  del plan, out, wr, wi
  torch.cuda.empty_cache()
  return res


MFMA_PROFILE = os.path.join(
  os.path.dirname(os.path.abspath(__file__)), "profiles",
  "qr_si64-128^3-gamma-128b_pmc-mfma.md")


def measured_mfma():
  """Per-kernel FP64 MFMA figures of the large cell from the committed
  rocprofv3 counter summary (SQ_INSTS_VALU_MFMA_MOPS_F64 x 512 flops over
  the kernel's traced duration), or None."""
  if not os.path.exists(MFMA_PROFILE):
    return None
  text = open(MFMA_PROFILE).read()
  start = text.find("```json")
  if start < 0:
    return None
  end = text.find("```", start + 7)
  return json.loads(text[start + 7:end])


NC_WORKLOAD = "nc-diamond-48^3-100Ha-8k-14b"


def _normcons_setup():
  """The reference's norm-conserving diamond example
  (tests/normconserving/diamond/config.yaml: C2 FCC, 48^3, spherical
  100 Ha, 2x2x2 k, ceil(8/2) + 10 = 14 bands, LDA exchange, uniform
  occupation of the 8 valence electrons), as a plan with the local part and
  the projectors set, and seeded parameters."""
  import numpy as np
  from jrystal_amd import pseudopotential as PS
  from jrystal_amd.objective import EnergyPlan
  params, (cr, pp, g, mask, kpts, occ) = _normcons_inputs()
  plan = EnergyPlan(cr.positions, cr.charges, cr.cell_vectors, mask, kpts,
                    occ)
  plan.set_external_potential(PS.potential_local_reciprocal(pp, g, cr.vol))
  plan.set_nonlocal(PS.potential_nonlocal_psi_reciprocal(pp, g, mask, kpts))
  return plan, params, (cr, pp, g, mask, kpts, occ)


def _normcons_inputs():
  """Host inputs of _normcons_setup: seeded parameters (numpy, the draws
  of pw.param_init) and (crystal, pseudopotential, G grid, mask, k-points,
  occupation)."""
  import numpy as np
  from jrystal_amd import grid, occupation, pseudopotential as PS
  from jrystal_amd.crystal import Crystal
  here = os.path.dirname(os.path.abspath(__file__))
  cr = Crystal.create_from_file(os.path.join(here, "jrystal_amd", "geometry",
                                             "diamond.xyz"))
  pp = PS.NormConservingPseudopotential.create(cr)
  gs = grid.proper_grid_size(48)
  g = np.asarray(grid.g_vectors(cr.cell_vectors, gs))
  mask = np.asarray(grid.spherical_mask(cr.cell_vectors, gs, 100.0))
  kpts = np.asarray(grid.k_vectors(cr.cell_vectors, grid.proper_grid_size(2)))
  nb = 14
  occ = occupation.uniform(kpts.shape[0], pp.total_valence_charge, 0, nb)
  occ = np.asarray(occ.cpu() if hasattr(occ, "cpu") else occ, np.float64)
  rng = np.random.default_rng(0)
  shape = (1, kpts.shape[0], int(mask.sum()), nb)
  params = {"w_re": rng.random(shape), "w_im": rng.random(shape)}
  return params, (cr, pp, g, mask, kpts, occ)


def normcons_bench(steps=200, warmup=10):
  """Energy + gradient evaluations of the norm-conserving diamond example
  (local pseudopotential, non-local projectors), eager, with the per-class
  times of one evaluation."""
  import torch
  plan, params, _ = _normcons_setup()
  params = {k: torch.tensor(v, device=plan.device) for k, v in params.items()}
  out = {}
  print(f"bench: norm-conserving {NC_WORKLOAD}", file=sys.stderr, flush=True)
  for _ in range(warmup):
    plan.evaluate(params["w_re"], params["w_im"], grad=True, out=out)
  torch.cuda.synchronize()
  t0 = time.perf_counter()
  for _ in range(steps):
    plan.evaluate(params["w_re"], params["w_im"], grad=True, out=out)
  torch.cuda.synchronize()
  dt = (time.perf_counter() - t0) / steps
  plan.set_timing(True)
  plan.evaluate(params["w_re"], params["w_im"], grad=True, out=out)
  torch.cuda.synchronize()
  cls = {k: round(v[0], 4) for k, v in plan.read_timing().items() if v[1]}
  plan.set_timing(False)
  e = out["energies"].tolist()
  res = {"workload": NC_WORKLOAD, "num_g": int(plan.num_g),
         "num_kpts": int(plan.nk), "num_bands": int(plan.nb),
         "projectors": int(plan.num_projectors), "steps": steps,
         "ms_per_eval": dt * 1e3, "evals_per_s": 1.0 / dt,
         "class_ms_one_eval": cls, "energy_total_Ha": e[4]}
  plan.close()
  torch.cuda.empty_cache()
  return res


def normcons_probe(evals=20):
  """The workload of the norm-conserving rocprofv3 runs."""
  import torch
  plan, params, _ = _normcons_setup()
  params = {k: torch.tensor(v, device=plan.device) for k, v in params.items()}
  out = {}
  for _ in range(evals):
    plan.evaluate(params["w_re"], params["w_im"], grad=True, out=out)
  torch.cuda.synchronize()
  print(json.dumps({"probe": NC_WORKLOAD, "evaluations": evals,
                    "energy_total_Ha": float(out["energies"][4])}))


def cpu_normcons(target_s, nthreads):
  """The oracle's norm-conserving evaluation of the diamond example on a
  k-point subset, scaled to whole evaluations per second (projector
  tables built before the timed region)."""
  sys.path.insert(0, os.path.dirname(os.path.abspath(__file__)))
  import numpy as np
  from threadpoolctl import threadpool_limits
  from oracle import adjoint as OA
  from oracle import pseudopotential as OPP
  from oracle import pw as OP
  OP.set_workers(nthreads)
  limits = threadpool_limits(limits=nthreads)
  params, (cr, pp, g, mask, kpts, occ) = _normcons_inputs()
  opp = OPP.create(cr.symbols, cr.positions, os.path.join(
    os.path.dirname(os.path.abspath(__file__)), "jrystal_amd", "data",
    "pseudopotential", "normconserving"))
  vloc = OPP.local_potential_reciprocal(opp, np.asarray(g), cr.vol)
  nk_full = kpts.shape[0]
  p_np = params

  def run(nk_s):
    kp = np.asarray(kpts)[:nk_s]
    prob = OA.Problem(mask=np.asarray(mask), g_vector_grid=np.asarray(g),
                      kpts=kp, vol=cr.vol, occupation=occ[:, :nk_s],
                      positions=cr.positions,
                      charges=np.asarray(cr.charges, float), v_ext_rec=vloc,
                      projectors=OPP.projectors(opp, np.asarray(g), mask, kp))
    p = {k: v[:, :nk_s] for k, v in p_np.items()}
    t = time.perf_counter()
    OA.energy_and_grad(p, prob)
    return time.perf_counter() - t

  run(1)
  t1 = run(1)
  nk_s = int(max(1, min(nk_full, round(target_s / max(t1, 1e-3)))))
  t = run(nk_s)
  limits.unregister()
  return {"value": nk_s / (t * nk_full),
          "unit": "energy+gradient evaluations/s", "cores": nthreads,
          "kind": "port",
          "sample": (f"the norm-conserving diamond example restricted to "
                     f"{nk_s} of {nk_full} k-points ({t:.2f} s), scaled by "
                     f"{nk_full}/{nk_s}; oracle/ NumPy+SciPy FP64")}


def band_probe(steps=100):
  """The workload of the band-mode rocprofv3 runs: ``steps`` Adam steps of
  the band driver's objective at the first k-point of the Si band example
  (one band-mode evaluation and the Adam kernel each)."""
  import torch
  from jrystal_amd import band, pw
  from jrystal_amd.hamiltonian import band_plan
  from jrystal_amd.optim import Adam
  cfg, BD, rho, mask = _band_setup()
  cr = BD.create_crystal(cfg)
  k = band.get_k_path(cr.cell_vectors, "LGXL", 60)[0:1]
  plan = band_plan(cr.positions, cr.charges, cr.cell_vectors, mask, rho, k,
                   28)
  params = pw.param_init(123, 28, 1, mask)
  opt = Adam(params, **cfg.optimizer_args)
  out = {}
  for _ in range(steps):
    plan.evaluate(params["w_re"], params["w_im"], grad=True, out=out)
    opt.step(params, {"w_re": out["dw_re"], "w_im": out["dw_im"]})
  torch.cuda.synchronize()
  print(json.dumps({"probe": BAND_WORKLOAD, "steps": steps,
                    "trace_Ha": float(out["energies"][4])}))


def large_cell_probe():
  """Workload of the large-cell rocprofv3 runs: eight energy + gradient
  evaluations of the 64-atom Gamma cell."""
  import torch
  from jrystal_amd import workloads
  from jrystal_amd.objective import EnergyPlan
  wl = workloads.si64()
  p = wl.params(0)
  plan = EnergyPlan.from_workload(wl)
  wr = torch.tensor(p["w_re"], device="cuda")
  wi = torch.tensor(p["w_im"], device="cuda")
  out = {}
  for _ in range(8):
    plan.evaluate(wr, wi, grad=True, out=out)
  torch.cuda.synchronize()
  print(f"large cell probe done: E = {float(out['energies'][4]):.10f}",
        flush=True)


TRAFFIC_PROFILE = os.path.join(
  os.path.dirname(os.path.abspath(__file__)), "profiles",
  "energy_grad_si8-cube-64k-32b_pmc-traffic.md")
KERNEL_NAMES = {"xline_vpsi": "jrx::xline_vpsi64_kernel",
                "plane_ifft": "jrx::plane_ifft64_kernel",
                "xline_density": "jrx::xline_density64_kernel",
                "plane_fft_gather": "jrx::plane_fft_gather64_kernel",
                "zplane_vpsi": "jrx::zplane_vpsi_kernel<64, 2, 4, true, true>",
                "row_ifft": "jrx::row_ifft_kernel<64, 2>",
                "zplane_density": "jrx::zplane_density_kernel<64, 2, 4, true>",
                "row_fft_gather": "jrx::row_fft_gather_kernel<64, 2, false>"}
# On the row-buffer path the four FFT timing classes hold these kernels.
ROW_PATH_CLASSES = {"plane_ifft": "row_ifft",
                    "xline_density": "zplane_density",
                    "xline_vpsi": "zplane_vpsi",
                    "plane_fft_gather": "row_fft_gather"}


SQ_PROFILE = os.path.join(
  os.path.dirname(os.path.abspath(__file__)), "profiles",
  "energy_grad_si8-cube-64k-32b_pmc-sq.md")
FP64_VALU_PEAK_TFLOPS = 78.6


def measured_sq(cls):
  """Per-launch SQ figures of a kernel class from the committed rocprofv3
  SQ counter summary (valu_f64_flop = 64 lanes x (ADD + MUL + 2 FMA) F64
  instructions, valu_instr = VALU instructions), or None."""
  name = KERNEL_NAMES.get(cls)
  if name is None or not os.path.exists(SQ_PROFILE):
    return None
  text = open(SQ_PROFILE).read()
  start = text.find("```json")
  if start < 0:
    return None
  end = text.find("```", start + 7)
  return json.loads(text[start + 7:end]).get(name)


def measured_traffic(cls):
  """HBM bytes per launch of a kernel class from the committed rocprofv3
  FETCH_SIZE / WRITE_SIZE summary (calibrated against a copy kernel), or
  None."""
  name = KERNEL_NAMES.get(cls)
  if name is None or not os.path.exists(TRAFFIC_PROFILE):
    return None
  text = open(TRAFFIC_PROFILE).read()
  start = text.find("```json")
  if start < 0:
    return None
  end = text.find("```", start + 7)
  table = json.loads(text[start + 7:end])
  return table.get(name)


def traffic_probe():
  """Workload of the rocprofv3 counter runs: a calibration kernel of known
  traffic (jrx_vec_axpby on 2^27 float64: reads 2 GiB, writes 1 GiB), then
  twelve energy+gradient evaluations of the benchmark workload (enough for
  the clocks to settle, so the traced durations match the live ones)."""
  import ctypes
  import torch
  from jrystal_amd import _lib, workloads
  from jrystal_amd.objective import EnergyPlan
  n = 1 << 27
  x = torch.ones(n, dtype=torch.float64, device="cuda")
  y = torch.ones(n, dtype=torch.float64, device="cuda")
  z = torch.empty(n, dtype=torch.float64, device="cuda")
  for _ in range(2):
    _lib.check(_lib.lib().jrx_vec_axpby(
      ctypes.c_double(1.0), x.data_ptr(), ctypes.c_double(2.0), y.data_ptr(),
      z.data_ptr(), n, _lib.stream_ptr()))
  torch.cuda.synchronize()
  del x, y, z
  wl = workloads.si8_cube(14.0, k=4)
  p = wl.params(0)
  plan = EnergyPlan.from_workload(wl)
  wr = torch.tensor(p["w_re"], device="cuda")
  wi = torch.tensor(p["w_im"], device="cuda")
  out = {}
  for _ in range(12):
    plan.evaluate(wr, wi, grad=True, out=out)
  torch.cuda.synchronize()
  print(f"traffic probe done: E = {float(out['energies'][4]):.10f}",
        flush=True)


def main():
  ap = argparse.ArgumentParser()
  ap.add_argument("--gpus", type=int, default=1)
  ap.add_argument("--steps", type=int, default=20)
  ap.add_argument("--warmup", type=int, default=3)
  ap.add_argument("--no-cpu-baseline", action="store_true")
  ap.add_argument("--cpu-seconds", type=float, default=12.0)
  ap.add_argument("--chunk-states", type=int, default=0)
  ap.add_argument("--no-convergence", action="store_true")
  ap.add_argument("--conv-seconds", type=float, default=30.0)
  ap.add_argument("--no-batch", action="store_true")
  ap.add_argument("--batch-steps", type=int, default=5)
  ap.add_argument("--traffic-probe", action="store_true",
                  help="run the rocprofv3 counter workload and exit")
  ap.add_argument("--no-small-cell", action="store_true")
  ap.add_argument("--no-band-structure", action="store_true")
  ap.add_argument("--band-probe", action="store_true",
                  help="only the band-mode rocprofv3 workload")
  ap.add_argument("--no-normcons", action="store_true")
  ap.add_argument("--normcons-probe", action="store_true",
                  help="only the norm-conserving rocprofv3 workload")
  ap.add_argument("--no-large-cell", action="store_true")
  ap.add_argument("--large-cell-steps", type=int, default=5)
  ap.add_argument("--large-cell-probe", action="store_true",
                  help="run the large-cell rocprofv3 workload and exit")
  args = ap.parse_args()
  if args.traffic_probe:
    traffic_probe()
    return
  if args.band_probe:
    band_probe()
    return
  if args.normcons_probe:
    normcons_probe()
    return
  if args.large_cell_probe:
    large_cell_probe()
    return
  if args.gpus != 1:
    print(f"bench.py: --gpus {args.gpus} is not supported; this path runs "
          "on one GPU (k-point sharding across GPUs is a design note only).",
          file=sys.stderr)
    sys.exit(2)

  import numpy as np
  import torch

  from jrystal_amd import workloads
  from jrystal_amd.objective import EnergyPlan

  wl = workloads.si8_cube(14.0, k=4)
  params = wl.params(seed=0)
  plan = EnergyPlan.from_workload(wl, chunk_states=args.chunk_states)
  dev = plan.device
  wr = torch.tensor(params["w_re"], device=dev)
  wi = torch.tensor(params["w_im"], device=dev)
  out = {}
  print(f"bench: workload {wl.name} G_n={plan.num_g} warmup={args.warmup} "
        f"steps={args.steps}", file=sys.stderr, flush=True)
  for _ in range(args.warmup):
    plan.evaluate(wr, wi, grad=True, out=out)
  torch.cuda.synchronize()
  ev0 = torch.cuda.Event(enable_timing=True)
  ev1 = torch.cuda.Event(enable_timing=True)
  t0 = time.perf_counter()
  ev0.record()
  for _ in range(args.steps):
    plan.evaluate(wr, wi, grad=True, out=out)
  ev1.record()
  torch.cuda.synchronize()
  wall = time.perf_counter() - t0
  gpu_ms = ev0.elapsed_time(ev1)
  ms_per_step = gpu_ms / args.steps
  value = args.steps / (wall)
  energies = out["energies"].tolist()
  if not np.all(np.isfinite(energies)):
    raise RuntimeError(f"non-finite energies {energies}")

  # Per-kernel-class durations, HIP events on the launch stream.
  plan.set_timing(True)
  nprof = 3
  for _ in range(nprof):
    plan.evaluate(wr, wi, grad=True, out=out)
  timing = plan.read_timing()
  plan.set_timing(False)
  if plan.row_path:
    timing = {ROW_PATH_CLASSES.get(k, k): v for k, v in timing.items()}
  chunks = plan.ns * max(1, -(-plan.nk * plan.nb // plan.chunk_states))
  dom = max(timing, key=lambda k: timing[k][0])
  ms, launches = timing[dom]
  per_eval_ms = ms / nprof
  bytes_eval = algorithmic_bytes(dom, plan, chunks)
  roofline = None
  if bytes_eval is not None:
    per_launch_bytes = bytes_eval / (launches / nprof)
    per_launch_ms = ms / launches
    achieved = per_launch_bytes / (per_launch_ms * 1e-3) / 1e9
    roofline = {"kernel": dom, "bound": "hbm", "achieved": achieved,
                "peak": HBM_PEAK_GBS, "unit": "GB/s",
                "frac": achieved / HBM_PEAK_GBS,
                "traffic": measured_traffic(dom),
                "avg_launch_ms": per_launch_ms,
                "algorithmic_bytes_per_launch": per_launch_bytes}
    sq = measured_sq(dom)
    if sq and sq.get("valu_f64_flop"):
      # the FFT passes' other bound: the FP64 VALU (counted flops of one
      # launch over the live launch duration; an FP64 add occupies an issue
      # slot like an FMA, so the issue fraction is given as well: VALU
      # instructions x 4 cycles per wave64 over 1024 SIMDs x 2.4 GHz)
      t = per_launch_ms * 1e-3
      tf = sq["valu_f64_flop"] / t / 1e12
      roofline["fp64_valu"] = {
        "achieved": tf, "peak": FP64_VALU_PEAK_TFLOPS, "unit": "TFLOP/s",
        "frac": tf / FP64_VALU_PEAK_TFLOPS,
        "flop_per_launch": sq["valu_f64_flop"],
        "issue_frac": sq.get("valu_instr", 0) * 4 / (1024 * 2.4e9 * t)}
  breakdown = {k: round(v[0] / nprof, 4) for k, v in timing.items()}
  config = {"workload": wl.name, "atoms": int(wl.crystal.num_atom),
            "Z": 14, "grid": list(wl.grid_sizes), "k_mesh": list(wl.k_grid),
            "num_kpts": int(plan.nk), "num_bands": int(plan.nb),
            "num_g": int(plan.num_g), "cutoff_Ha": wl.cutoff_energy,
            "chunk_states": int(plan.chunk_states),
            "keep_planes": bool(plan.keep_planes),
            "energy_total_Ha": energies[4]}

  plan.close()
  del plan, out, wr, wi
  torch.cuda.empty_cache()

  batch = None
  if not args.no_batch:
    batch = batch_bench(args.batch_steps, 1)

  small = None
  if not args.no_small_cell:
    small = small_cell_bench(200, 20)

  large = None
  if not args.no_large_cell:
    large = large_cell_bench(args.large_cell_steps, 1)

  bands = None
  if not args.no_band_structure:
    bands = band_structure_bench()

  nc = None
  if not args.no_normcons:
    nc = normcons_bench()

  conv = None
  if not args.no_convergence:
    conv, conv_ctx = convergence(args.conv_seconds)

  cpu = None
  if not args.no_cpu_baseline:
    nthreads = int(os.environ.get("OMP_NUM_THREADS", "0")) or os.cpu_count()
    cpu = cpu_baseline(wl, params, args.cpu_seconds, nthreads)
    cpu["host"] = cpu_host()
    # the reference's own thread setting (opt_utils.py:45-47)
    c4 = cpu_baseline(wl, params, args.cpu_seconds / 2, 4)
    cpu["value_4_threads"] = c4["value"]
    cpu["sample_4_threads"] = c4["sample"]
    if bands is not None:
      cpu["band_structure_step"] = cpu_band_step(args.cpu_seconds / 2,
                                                 nthreads)
    if nc is not None:
      cpu["normcons"] = cpu_normcons(args.cpu_seconds / 2, nthreads)
    if conv is not None:
      # CPU seconds per evaluation of the convergence cell, times the
      # evaluations the plain method needed on the GPU
      cwl, plain = conv_ctx
      c2 = cpu_baseline(cwl, cwl.params(0), args.cpu_seconds / 2, nthreads)
      i = conv["plain"]["iterations"]
      if i is not None and plain.history:
        frac = i / max(1, len(plain.history) - 1)
        evals = frac * plain.evaluations
        conv["cpu_estimate_plain_s"] = evals / c2["value"]
        conv["cpu_estimate_note"] = (
          "estimate: evaluations the plain method used on the GPU up to the "
          f"tolerance ({evals:.0f}) / CPU evaluations per second of the "
          f"oracle restatement on this cell ({c2['value']:.4g}/s, "
          f"{c2['sample']})")

  line = {
    "metric": METRIC, "value": value,
    "unit": "energy+gradient evaluations/s", "n_gpus": 1,
    "steps": args.steps, "warmup": args.warmup,
    "ms_per_step": ms_per_step, "higher_is_better": True, "scaling": "weak",
    "vs_baseline": None, "dtype": "f64", "data": "synthetic",
    "config": config,
    "roofline": roofline,
    "kernel_ms_per_eval": breakdown,
    "cpu_baseline": cpu,
    "convergence": conv,
    "batch": batch,
    "small_cell": small,
    "large_cell": large,
    "band_structure": bands,
    "normcons": nc,
  }
  print(json.dumps(line))


if __name__ == "__main__":
  main()
