"""Benchmark of the XCorr search path on one MI355X.

Workload (default): tryptic-20k-20k, the dense-block workload -- 20,000
seeded random proteins, tryptic digest with up to 2 missed cleavages and
fixed carbamidomethyl Cys, 20,000 synthetic spectra at 2+/3+ (50/50; 3+
spectra also carry doubly charged fragments), no variable modifications,
+-3 Da precursor window, top-5 per spectrum.

A step is one pass of the scoring stage over the whole batch with the
database and the preprocessed spectra resident in HBM: precursor windows ->
theoretical peaks -> XCorr of every (spectrum, candidate) pair -> per-spectrum
top-N with exact re-score.  Three forms are timed:
  plain          hfx_window + hfx_xcorr_sparse + hfx_topn (the drop-in: a call
                 of this size writes the theoretical rows its windows need and
                 contracts them with blocks of sixteen spectra in 32-bit fixed
                 point, rounded once to FP32; every step writes them anew);
  batched fp32   hfx_batch_* in its FP32 form (the same contraction over the
                 rows the per-database peptide index keeps);
  batched bf16x2 hfx_batch_* in its BF16 form (blocks of up to eight spectra,
                 BF16 weights x hi+lo BF16 spectra, FP32 accumulation);
  batched i8x3   hfx_batch_* in its integer form (blocks of up to sixteen
                 spectra, int8 weights x three base-256 digits);
each with its top-N and exact re-score.
Each batched step runs every per-batch step on the device -- windows,
spectrum order, block cut, the spectra's digits or hi/lo planes, scoring,
top-N -- captured once in a hipGraph and replayed.  The per-database peptide
index (b ladders, ion lists) is built once before the loop and its build
time is reported beside the step (`db_setup_ms`); its theoretical rows are
added by the first batch that runs on it, before its timed steps; the one-off
plan (allocation) time is reported too.
value = scored pairs per second of the batched BF16-split form (whole job,
one GPU); every form's top-N must equal the plain form's.

Prints one JSON line.  --gpus N > 1 exits: the benchmark runs on one GPU.
"""
from __future__ import annotations

import argparse
import json
import os
import sys
import time

import numpy as np

ROOT = os.path.dirname(os.path.abspath(__file__))
sys.path.insert(0, ROOT)

METRIC = "XCorr peptide-spectrum scores/sec, plain FP32 vs batched BF16-split, top-5 match"
HBM_PEAK_GBS = 8000.0
BF16_PEAK_TFLOPS = 2500.0  # dense MFMA, no sparsity
INT8_PEAK_TOPS = 5000.0    # dense int8 MFMA, no sparsity
I8_K = 6                   # integer form: operations per padded bin and scored pair


def measured_traffic(kernel: str, workload: str):
    """HBM bytes per launch of `kernel` on `workload`, as measured by the
    counter runs summarised in profiles/<kernel>_counters_<workload>.md (the
    line 'HBM traffic per launch (bytes): N': rocprofv3 FETCH_SIZE plus
    WRITE_SIZE, each scaled by a copy kernel of known size), or None."""
    import re
    path = os.path.join(ROOT, "profiles", f"{kernel}_counters_{workload}.md")
    try:
        with open(path) as f:
            m = re.search(r"HBM traffic per launch \(bytes\): ([0-9,]+)", f.read())
    except OSError:
        return None
    if not m:
        return None
    return {"bytes": int(m.group(1).replace(",", "")),
            "source": os.path.relpath(path, ROOT)}


def log(msg):
    print(f"[bench] {msg}", file=sys.stderr, flush=True)


def setup(workload: str):
    from hfx_amd import pipeline, synth

    w = synth.WORKLOADS[workload]
    t0 = time.time()
    prot = synth.make_proteins(w["proteins"], seed=w["seed"])
    mass = pipeline.mass_table(w["static"])
    r, tc, tn = pipeline.digest(prot.seq, prot.seg, mass, 1, w["missed"], 400.0, 7200.0,
                                w["p_rule"], w["min_len"], w["max_len"])
    log(f"database: {prot.count} proteins, {len(prot.seq)} residues, {len(r)} peptides "
        f"({time.time() - t0:.1f}s)")
    sp = synth.make_spectra(prot, r, tc, tn, w["spectra"], seed=w["seed"] + 100,
                            charges=w["charges"], charge_p=w["charge_p"], static_mods=w["static"],
                            double_for_3plus=w["double3"])
    log(f"spectra: {sp.count} ({len(sp.mz)} peaks, {time.time() - t0:.1f}s)")
    ctx = pipeline.Ctx(0)
    db = pipeline.DeviceDB(pipeline.HostDB(prot.seq, r, tc, tn, mass))
    dsp = pipeline.DeviceSpectra(ctx, sp.pcr, sp.charge, sp.mz, sp.inten, sp.off, 2112)
    st = dsp.status()
    if (st != 0).any():
        raise SystemExit(f"preprocessing failed for {int((st != 0).sum())} spectra")
    log(f"device resident ({time.time() - t0:.1f}s)")
    return dict(w=w, prot=prot, mass=mass, r=r, tc=tc, tn=tn, sp=sp, ctx=ctx, db=db, dsp=dsp)


def bench_mods(steps, warmup, workload="mods-2k-50k"):
    """The modified-candidate search (Search.hs:282-622) on the uneven
    workload: hfx_mod_windows for every spectrum, the reference ABI's
    enumeration stages (findModablePeptides, calcTotalModCands,
    prepareGenMod, genModCands: each synchronises the host for its count, as
    in the reference), hfx_mpep_offsets, hfx_xcorr_sparse_mod and
    hfx_topn_mod.  Wall time per run (host synchronisations and copies
    included; a run reuses the previous run's device buffers when they are
    large enough) and the scoring and top-N kernels by events."""
    from hfx_amd import pipeline, synth

    w = synth.WORKLOADS[workload]
    t0 = time.time()
    prot = synth.make_proteins(w["proteins"], seed=w["seed"])
    mass = pipeline.mass_table(w["static"])
    r, tc, tn = pipeline.digest(prot.seq, prot.seg, mass, 1, w["missed"], 400.0, 7200.0,
                                w["p_rule"], w["min_len"], w["max_len"])
    sp = synth.make_spectra(prot, r, tc, tn, w["spectra"], seed=w["seed"] + 100,
                            charges=w["charges"], charge_p=w["charge_p"],
                            double_for_3plus=w["double3"], var_mods=w["var"])
    ctx = pipeline.Ctx(0)
    mi = pipeline.mod_info(w["var"], w["max_ma"])
    db = pipeline.DeviceDB(pipeline.HostDB(prot.seq, r, tc, tn, mass), ma=mi.ma)
    dsp = pipeline.DeviceSpectra(ctx, sp.pcr, sp.charge, sp.mz, sp.inten, sp.off, 2112)
    log(f"mods workload: {len(r)} peptides, {mi.num_mod} modifications, {dsp.num_spec} spectra "
        f"({time.time() - t0:.1f}s)")
    ms = pipeline.ModSearch(ctx, db, dsp, mi, eps=3.0, topn=w["topn"])
    for _ in range(warmup):
        res = ms.run(keep_stages=False)
    pipeline.sync()
    t0 = time.perf_counter()
    for _ in range(steps):
        res = ms.run(keep_stages=False)
    pipeline.sync()
    el = (time.perf_counter() - t0) / max(steps, 1)
    n = np.diff(res.mp_off).astype(np.int64)
    return res, {"workload": workload, "spectra": int(dsp.num_spec), "peptides": int(len(r)),
                 "modifications": int(mi.num_mod), "modified_candidates": int(res.num_mpep),
                 "per_spectrum": {"min": int(n.min()), "median": int(np.median(n)),
                                  "p99": int(np.percentile(n, 99)), "max": int(n.max())},
                 "ms_per_run": el * 1e3, "value": res.num_mpep / el,
                 "unit": "modified-candidate scores/s"}


def algorithmic_bytes(env, res) -> float:
    """Compulsory HBM bytes of the scoring stage for the scored pairs: per
    pair the candidate's residues + 16 bytes of index/terminal/residual words
    + 8 bytes out (score + index), plus each spectrum read once (4 B/bin)."""
    tc, tn = env["tc"], env["tn"]
    idx = env["db"].idx_sorted()
    nres = (tn.astype(np.int64) - tc.astype(np.int64)).clip(min=0)
    per_pos = nres[idx] + 16 + 8
    cs = np.concatenate([[0], np.cumsum(per_pos)])
    b, n = res.begin.astype(np.int64), res.num.astype(np.int64)
    cand = float(np.sum(cs[b + n] - cs[b]))
    spec = float(4 * env["dsp"].lengths().astype(np.int64).sum())
    return cand + spec


def same_topn(a, b, n=None) -> bool:
    S = len(a.top_cnt) if n is None else n
    if not (a.top_cnt[:S] == b.top_cnt[:S]).all():
        return False
    return all(a.top_pos[s, : a.top_cnt[s]].tolist() == b.top_pos[s, : b.top_cnt[s]].tolist()
               and (a.top_exact[s, : a.top_cnt[s]] == b.top_exact[s, : b.top_cnt[s]]).all()
               for s in range(S))


def _cpu_model() -> str:
    try:
        with open("/proc/cpuinfo") as f:
            for line in f:
                if line.startswith("model name"):
                    return line.split(":", 1)[1].strip()
    except OSError:
        pass
    return "unknown"


def cpu_baseline(env, res, topn, target_s=1.0, reps=5):
    """The oracle (C++ restatement of the reference's path: window ->
    per-candidate dense row with max per bin -> FP32 dot, plus the exact
    fixed-point score -> top-N; -O3 -march=x86-64-v3 -ffp-contract=off,
    OpenMP over spectra) on a bounded sample of the same spectra: best of
    `reps` timed runs after one warm-up, with all the threads this process
    may use (OMP_NUM_THREADS, else the cores the OS reports, at most 16: the
    host share of one GPU) and with one thread.  Every sampled spectrum's
    top-N is compared with the GPU's."""
    from oracle import oracle as orc

    nproc = os.cpu_count() or 1
    threads = int(os.environ.get("OMP_NUM_THREADS", "0") or 0) or min(nproc, 16)
    dsp = env["dsp"]
    X = dsp.x()
    lens = dsp.lengths()
    idx = env["db"].idx_sorted()
    ions = env["db"].packed_ions()
    S = dsp.num_spec
    args = (ions, env["r"], env["tc"], env["tn"], env["mass"], idx)
    # spread the sample over the whole order of precursor masses
    perm = np.random.default_rng(7).permutation(S)

    def run(n, nt):
        sel = np.sort(perm[:n])
        t0 = time.perf_counter()
        ref = orc.search_plain(*args, X[sel], lens[sel], dsp.zmax[sel], dsp.mass[sel], 3.0, topn,
                               nthreads=nt)
        return time.perf_counter() - t0, sel, ref

    def timed(nt):
        n = 4 * nt
        dt, _, _ = run(n, nt)  # warm-up and size probe
        n = int(min(S, max(4 * nt, n * target_s / max(dt, 1e-3))))
        best, sel, ref = None, None, None
        for _ in range(reps):
            dt, sel, ref = run(n, nt)
            best = dt if best is None else min(best, dt)
        return best, sel, ref

    dt_all, sel, ref = timed(threads)
    scores = int(ref["num"].sum())
    same = all(
        int(res.top_cnt[s]) == int(ref["top_cnt"][i])
        and res.top_pos[s, : res.top_cnt[s]].tolist() == ref["top_pos"][i, : ref["top_cnt"][i]].tolist()
        and (res.top_exact[s, : res.top_cnt[s]] ==
             orc.fx_to_double(ref["top_fx"][i, : ref["top_cnt"][i]])).all()
        for i, s in enumerate(sel))
    dt_one, sel1, ref1 = timed(1)
    scores1 = int(ref1["num"].sum())
    acc = score_error(orc, args, X, lens, dsp, sel, res, topn, threads)
    return dict(value=scores / dt_all, unit="scores/s", cores=threads, kind="port",
                sample=f"{len(sel)} of {S} spectra drawn across the mass range ({scores} scored "
                       f"pairs): oracle dense-row scoring with exact top-{topn}, OpenMP over "
                       f"spectra, best of {reps} after a warm-up, {dt_all:.2f}s",
                nproc=nproc, cpu_model=_cpu_model(),
                one_thread=dict(value=scores1 / dt_one, unit="scores/s", cores=1,
                                sample=f"{len(sel1)} spectra ({scores1} scored pairs), best of "
                                       f"{reps}, {dt_one:.2f}s"),
                build="g++ -O3 -march=x86-64-v3 -ffp-contract=off -fopenmp",
                topn_identical_to_gpu=bool(same), accuracy=acc)


def score_error(orc, args, X, lens, dsp, sel, res, topn, threads):
    """Every score of the sampled spectra from the measured form against the
    oracle's exact score of the same pair (outside the timed runs): the
    relative error with the floor the full-size tests use (|exact| or a
    quarter of the pair's sum w|x|, whichever is larger) and the plain
    relative error."""
    if res.scores is None:
        return None
    ex = orc.search_plain(*args, X[sel], lens[sel], dsp.zmax[sel], dsp.mass[sel], 3.0, topn,
                          want_all=True, nthreads=threads)
    ab = orc.search_plain(*args, np.abs(X[sel]), lens[sel], dsp.zmax[sel], dsp.mass[sel], 3.0,
                          topn, want_all=True, nthreads=threads)
    if not (np.diff(ex["off"].astype(np.int64)) == res.num[sel]).all():
        raise SystemExit("sampled windows differ from the measured form's")
    e = orc.fx_to_double(ex["all_fx"])[: int(ex["off"][-1])]
    scale = orc.fx_to_double(ab["all_fx"])[: int(ex["off"][-1])]
    g = np.concatenate([res.scores[int(res.off[s]):int(res.off[s + 1])] for s in sel])
    d = np.abs(g.astype(np.float64) - e)
    rel = d / np.maximum(np.abs(e), 0.25 * scale)
    nz = np.abs(e) > 0
    return dict(pairs=int(len(e)), max_rel=float(rel.max(initial=0.0)),
                within_1e4=float((rel <= 1e-4).mean()) if len(e) else 1.0,
                max_rel_of_exact=float((d[nz] / np.abs(e[nz])).max(initial=0.0)),
                within_1e4_of_exact=float((d[nz] <= 1e-4 * np.abs(e[nz])).mean()) if nz.any() else 1.0,
                rule="rel = |score - exact| / max(|exact|, 0.25 * sum w|x| of the pair); "
                     "of_exact: |score - exact| / |exact| over pairs with exact != 0")


def calib_read(mib: int):
    """Streams mib MiB of floats through k_mvm_rows (reads A once, x from
    cache, writes 4 bytes per row): a kernel of known HBM traffic whose byte
    counters scale the counters of the search kernels."""
    from hfx_amd import check, lib, pipeline

    n = 4096
    m = mib * 1024 * 1024 // (4 * n)
    A = pipeline.empty(4 * m * n)
    A.zero()
    x = pipeline.dev(np.ones(n, np.float32))
    y = pipeline.empty(4 * m)
    ctx = pipeline.Ctx(0)
    for _ in range(3):
        check(lib().hfx_mvm_rows(ctx.h, y.p, A.p, n, x.p, m, n, None), "hfx_mvm_rows")
    pipeline.sync()
    print(json.dumps({"calib_read_bytes": 4 * m * n, "calib_write_bytes": 4 * m,
                      "launches": 3}), flush=True)


def bench_plain(env, topn, steps, warmup, margin=0):
    from hfx_amd import pipeline

    srch = pipeline.PlainSearch(env["ctx"], env["db"], env["dsp"], eps=3.0, topn=topn,
                                margin=margin)

    def step(ev=None):
        srch.window()
        if ev is not None:
            ev[0].record(pipeline.stream_handle())
        srch.score()
        if ev is not None:
            ev[1].record(pipeline.stream_handle())
        srch.select()

    for _ in range(warmup):
        step()
    pipeline.sync()
    evs = [(pipeline.Event(), pipeline.Event()) for _ in range(steps)]
    t0 = time.perf_counter()
    for k in range(steps):
        step(evs[k])
    pipeline.sync()
    elapsed = time.perf_counter() - t0
    kern_ms = float(np.mean([a.elapsed_ms(b) for a, b in evs]))
    flagged = len(srch.flagged())
    res = srch.run()
    return res, elapsed, kern_ms, flagged, srch


def bench_stats(srch, steps, res):
    """E-value fit over every score of the batch (hfx_evalue_fit, one
    workgroup per spectrum) and the SP ion counts of the top N
    (hfx_sp_ions_topn: peak flags, then one match per thread), each timed
    with events on the stream they run on, after the plain search."""
    import ctypes as C

    import hfx_amd
    from hfx_amd import pipeline

    L = hfx_amd.lib()
    S, N = srch.sp.num_spec, srch.topn
    t_fit, t_np, t_nu = pipeline.empty(16 * S), pipeline.empty(4 * S), pipeline.empty(8 * S)
    outs = [pipeline.empty(4 * S * N) for _ in range(3)]
    st = pipeline.stream_handle()

    def fit():
        hfx_amd.check(L.hfx_evalue_fit(srch.ctx.h, t_fit.p, t_np.p, t_nu.p, srch.t_scores.p,
                                       srch.t_off.p, None, None, S, 350, 3.0, st),
                      "hfx_evalue_fit")

    def ions():
        hfx_amd.check(L.hfx_sp_ions_topn(srch.ctx.h, *[o.p for o in outs], srch.t_pos.p,
                                         srch.t_cnt.p, srch.t_begin.p, N, C.byref(srch.db.desc),
                                         C.byref(srch.sp.desc), 1, st), "hfx_sp_ions_topn")

    fit()
    ions()
    pipeline.sync()
    evs = [(pipeline.Event(), pipeline.Event(), pipeline.Event()) for _ in range(max(steps, 3))]
    for e in evs:
        e[0].record(st)
        fit()
        e[1].record(st)
        ions()
        e[2].record(st)
    pipeline.sync()
    fit_ms = float(np.mean([a.elapsed_ms(b) for a, b, _ in evs]))
    ions_ms = float(np.mean([b.elapsed_ms(c) for _, b, c in evs]))
    total = int(res.off[-1])
    npts = pipeline.host(t_np, np.uint32, S)
    fit_bytes = 4.0 * total + 16.0 * S + 16.0 * S   # scores read once, offsets, fits
    return {"evalue_fit": {"kernel": "k_evfit", "ms": fit_ms, "scores": total,
                           "spectra_with_fit": int((npts >= 2).sum()),
                           "algorithmic_bytes": fit_bytes,
                           "achieved_gbs": fit_bytes / (fit_ms * 1e-3) / 1e9,
                           "frac_hbm": fit_bytes / (fit_ms * 1e-3) / 1e9 / HBM_PEAK_GBS},
            "sp_ions": {"kernels": ["k_sp_topn"], "ms": ions_ms,
                        "matches": int(res.top_cnt.sum())}}


DENSE_K = 2176  # padded bins of a dense row (the kernel's row length)


def dense_flops(env, res, k_per_pair=4) -> tuple[float, float]:
    """(executed, useful) MFMA operations of one dense pass by the per-pair
    figures of the precision form: executed = k_per_pair K per scored pair
    (BF16 form: 4 K, hi and lo columns over the padded row, K = 2176 bins;
    integer form: 6 K, three digit contractions; the groups of 256 bins that no
    peak of a tile reaches are skipped, not subtracted here), useful = 2 len_s
    per scored pair (one product per bin of the spectrum)."""
    dsp = env["dsp"]
    z = dsp.zmax.astype(np.int64)
    scored = (z <= 4) & (z > 0)
    n = res.num.astype(np.int64)
    lens = np.minimum(dsp.lengths().astype(np.int64), DENSE_K)
    executed = float(np.sum(float(k_per_pair) * DENSE_K * n * scored))
    useful = float(np.sum(2.0 * lens * n * scored))
    return executed, useful


def bench_batched(env, topn, steps, warmup, index, precision=0, margin=0):
    from hfx_amd import pipeline

    t0 = time.perf_counter()
    bs = pipeline.BatchSearch(env["ctx"], env["db"], env["dsp"], eps=3.0, topn=topn,
                              margin=margin, index=index)
    bs.set_precision(precision)
    bs.stream.sync()
    plan_ms = (time.perf_counter() - t0) * 1e3
    t0 = time.time()
    cfg = bs.autotune()
    log(f"autotune ({'dense' if precision else 'sparse'}): G={cfg[0]} C={cfg[1]} "
        f"threads={cfg[2]} ({time.time() - t0:.1f}s)")
    bs.capture()
    for _ in range(warmup):
        bs.replay()
    bs.stream.sync()
    t0 = time.perf_counter()
    for _ in range(steps):
        bs.replay()
    bs.stream.sync()
    elapsed = time.perf_counter() - t0
    res = bs.results(keep_scores=precision != 0)
    # the same per-batch pipeline run phase by phase, with events on the
    # batch's stream around each phase and around the scoring kernel itself
    ph = [bs.time_phases() for _ in range(max(steps, 3))]
    phases = {k: float(np.mean([p[k] for p in ph])) for k in ph[0]}
    info = bs.info()
    if precision:
        info["dense_blocks"] = int(len(bs.dense_blocks()) - 1)
    return res, elapsed, phases, cfg, info, plan_ms


def main():
    ap = argparse.ArgumentParser()
    ap.add_argument("--gpus", type=int, default=1)
    ap.add_argument("--steps", type=int, default=10)
    ap.add_argument("--warmup", type=int, default=3)
    ap.add_argument("--workload", default="tryptic-20k-20k")
    ap.add_argument("--no-cpu", action="store_true")
    ap.add_argument("--margin", type=int, default=0,
                    help="extra candidates re-scored exactly beyond the top N")
    ap.add_argument("--path", choices=("all", "plain", "batched", "dense", "i8", "mods"),
                    default="all")
    ap.add_argument("--calib-read", type=int, default=0, metavar="MIB",
                    help="only run a streaming read of MIB MiB (k_mvm_rows over a "
                         "row matrix) to calibrate HBM byte counters, then exit")
    args = ap.parse_args()
    if args.gpus != 1:
        print(json.dumps({"error": "the benchmark runs on one GPU; --gpus must be 1"}))
        raise SystemExit(2)
    if args.calib_read:
        calib_read(args.calib_read)
        return

    from hfx_amd import pipeline

    if args.path == "mods":
        _, m = bench_mods(args.steps, args.warmup)
        print(json.dumps({"metric": "modified-candidate XCorr scores/sec (uneven workload)",
                          "value": m["value"], "unit": m["unit"], "n_gpus": 1,
                          "steps": args.steps, "warmup": args.warmup,
                          "ms_per_step": m["ms_per_run"], "higher_is_better": True,
                          "scaling": "weak", "vs_baseline": None, "dtype": "f32",
                          "data": "synthetic", "config": m}), flush=True)
        return
    env = setup(args.workload)
    topn = env["w"]["topn"]
    out = {"metric": METRIC, "unit": "scores/s", "n_gpus": 1, "steps": args.steps,
           "warmup": args.warmup, "higher_is_better": True, "scaling": "weak",
           "vs_baseline": None, "dtype": "f32", "data": "synthetic"}
    paths = {}
    plain_res = None
    if args.path in ("all", "plain"):
        plain_res, el, kern_ms, flagged, psrch = bench_plain(env, topn, args.steps,
                                                             args.warmup, args.margin)
        sc = int(plain_res.off[-1])
        ab = algorithmic_bytes(env, plain_res)
        paths["plain_fp32_sparse"] = dict(
            value=sc * args.steps / el, ms_per_step=el * 1e3 / args.steps, scores_per_step=sc,
            kernel="k_rw_build + k_rw_mm", kernel_ms=kern_ms,
            kernel_gbs=ab / (kern_ms * 1e-3) / 1e9, algorithmic_bytes=ab,
            flagged_spectra_per_step=flagged)
        log(f"plain: {paths['plain_fp32_sparse']['value']:.3e} scores/s, kernel {kern_ms:.2f} ms")
        stats = bench_stats(psrch, args.steps, plain_res)
        log(f"stats: {stats}")
        del psrch
    # the per-database peptide index, built once
    index = None
    forms = 0
    if args.path in ("all", "batched"):
        forms |= pipeline.PepIndex.IONS
    if args.path in ("all", "dense", "i8"):
        forms |= pipeline.PepIndex.LADDER
    db_setup = {}
    if forms:
        pipeline.sync()
        t0 = time.perf_counter()
        index = pipeline.PepIndex(env["ctx"], env["db"], forms=forms, levels=4, max_len=4096)
        pipeline.sync()
        db_setup = dict(ms=(time.perf_counter() - t0) * 1e3, **index.info())
        log(f"peptide index: {db_setup}")
    batch_res = None
    if args.path in ("all", "batched"):
        batch_res, el, phases, cfg, info, plan_ms = bench_batched(
            env, topn, args.steps, args.warmup, index, 0, args.margin)
        sc = int(batch_res.off[-1])
        ab = algorithmic_bytes(env, batch_res)
        paths["batched_fp32_sparse"] = dict(
            value=sc * args.steps / el, ms_per_step=el * 1e3 / args.steps, scores_per_step=sc,
            kernel="k_rw_mm", kernel_ms=phases["kernel"], phases_ms=phases,
            kernel_gbs=ab / (phases["kernel"] * 1e-3) / 1e9,
            config=dict(G=cfg[0], C=cfg[1], threads=cfg[2]), info=info, plan_ms=plan_ms,
            graph="every per-batch step captured once, replayed per step",
            flagged_spectra=int(len(batch_res.flagged)))
        log(f"batched fp32: {paths['batched_fp32_sparse']['value']:.3e} scores/s {phases}")
    dense_res = None
    if args.path in ("all", "dense"):
        dense_res, el, phases, cfg, info, plan_ms = bench_batched(
            env, topn, args.steps, args.warmup, index, 1, args.margin)
        sc = int(dense_res.off[-1])
        ex, useful = dense_flops(env, dense_res)
        paths["batched_bf16x2_dense"] = dict(
            value=sc * args.steps / el, ms_per_step=el * 1e3 / args.steps, scores_per_step=sc,
            kernel="k_rw_mm", kernel_ms=phases["kernel"], phases_ms=phases,
            mfma_flops_executed=ex, mfma_flops_useful=useful,
            config=dict(chunk=cfg[1], threads=cfg[2], spectra_per_block_max=8,
                        blocks=info["dense_blocks"]), plan_ms=plan_ms,
            graph="every per-batch step captured once, replayed per step",
            flagged_spectra=int(len(dense_res.flagged)))
        log(f"batched bf16x2: {paths['batched_bf16x2_dense']['value']:.3e} scores/s {phases}")
    i8_res = None
    if args.path in ("all", "i8"):
        i8_res, el, phases, cfg, info, plan_ms = bench_batched(
            env, topn, args.steps, args.warmup, index, 2, args.margin)
        sc = int(i8_res.off[-1])
        ex, useful = dense_flops(env, i8_res, k_per_pair=I8_K)
        paths["batched_i8x3_dense"] = dict(
            value=sc * args.steps / el, ms_per_step=el * 1e3 / args.steps, scores_per_step=sc,
            kernel="k_rw_mm", kernel_ms=phases["kernel"], phases_ms=phases,
            mfma_ops_executed=ex, mfma_ops_useful=useful,
            config=dict(chunk=cfg[1], threads=cfg[2], spectra_per_block_max=16,
                        blocks=info["dense_blocks"]), plan_ms=plan_ms,
            graph="every per-batch step captured once, replayed per step",
            flagged_spectra=int(len(i8_res.flagged)), short_spectra=int(len(i8_res.short)))
        log(f"batched i8x3: {paths['batched_i8x3_dense']['value']:.3e} scores/s {phases}")
    ref = plain_res
    for key, r in (("batched_fp32_sparse", batch_res), ("batched_bf16x2_dense", dense_res),
                   ("batched_i8x3_dense", i8_res)):
        if r is not None and ref is not None:
            paths[key]["topn_identical_to_plain"] = same_topn(ref, r)
    # the headline: the faster dense form whose rankings match the plain form's
    dense_forms = [(k, r) for k, r in (("batched_i8x3_dense", i8_res),
                                       ("batched_bf16x2_dense", dense_res))
                   if r is not None and paths[k].get("topn_identical_to_plain", True)]
    if dense_forms:
        main_key, res = max(dense_forms, key=lambda kr: paths[kr[0]]["value"])
    elif batch_res is not None:
        main_key, res = "batched_fp32_sparse", batch_res
    else:
        main_key, res = "plain_fp32_sparse", plain_res
    p = paths[main_key]
    if main_key == "batched_i8x3_dense":
        achieved = p["mfma_ops_executed"] / (p["kernel_ms"] * 1e-3) / 1e12
        tr = measured_traffic("k_rw_mm_i8x3", args.workload)
        roofline = {"kernel": p["kernel"], "bound": "mfma", "achieved": achieved,
                    "peak": INT8_PEAK_TOPS, "unit": "TOP/s",
                    "frac": achieved / INT8_PEAK_TOPS,
                    "traffic": tr["bytes"] if tr else None,
                    "kernel_ms": p["kernel_ms"], "ops_per_launch": p["mfma_ops_executed"],
                    "ops_rule": f"{I8_K} K per scored pair, K = {DENSE_K} padded bins (three "
                                "int8 digit contractions, 2 ops a multiply-add); groups of 256 bins "
                                "past a tile's last peak are skipped, not subtracted",
                    "ops_useful": p["mfma_ops_useful"]}
        if tr:
            roofline["traffic_source"] = tr["source"]
        dtype = "i8x3"
    elif main_key == "batched_bf16x2_dense":
        achieved = p["mfma_flops_executed"] / (p["kernel_ms"] * 1e-3) / 1e12
        tr = measured_traffic("k_rw_mm_bf16x2", args.workload)
        roofline = {"kernel": p["kernel"], "bound": "mfma", "achieved": achieved,
                    "peak": BF16_PEAK_TFLOPS, "unit": "TFLOP/s",
                    "frac": achieved / BF16_PEAK_TFLOPS,
                    "traffic": tr["bytes"] if tr else None,
                    "kernel_ms": p["kernel_ms"], "flops_per_launch": p["mfma_flops_executed"],
                    "flops_rule": f"4 K per scored pair, K = {DENSE_K} padded bins (hi and lo "
                                  "BF16 columns); groups of 256 bins past a tile's last peak "
                                  "are skipped, not subtracted",
                    "flops_useful": p["mfma_flops_useful"]}
        if tr:
            roofline["traffic_source"] = tr["source"]
        dtype = "bf16x2"
    else:
        ab = algorithmic_bytes(env, res)
        achieved = ab / (p["kernel_ms"] * 1e-3) / 1e9
        roofline = {"kernel": p["kernel"], "bound": "hbm", "achieved": achieved,
                    "peak": HBM_PEAK_GBS, "unit": "GB/s", "frac": achieved / HBM_PEAK_GBS,
                    "traffic": None, "kernel_ms": p["kernel_ms"], "algorithmic_bytes": ab}
        dtype = "f32"
    out.update(
        value=p["value"], ms_per_step=p["ms_per_step"], dtype=dtype,
        config={"workload": args.workload, "proteins": env["w"]["proteins"],
                "peptides": int(len(env["r"])), "spectra": int(env["dsp"].num_spec),
                "window_da": 3.0, "bin_width": 1.0005079,
                "max_len": int(env["dsp"].lengths().max()), "topn": topn, "margin": args.margin,
                "path": main_key, "scores_per_step": p["scores_per_step"]},
        roofline=roofline, db_setup_ms=db_setup.get("ms"), db_setup=db_setup, paths=paths)
    if "plain_fp32_sparse" in paths:
        out["stats"] = stats
    if args.path == "all":
        # the modified-candidate search on the uneven workload (not the headline)
        _, m = bench_mods(min(args.steps, 3), min(args.warmup, 1))
        paths["mods_fp32_sparse"] = m
        log(f"mods: {m['value']:.3e} modified-candidate scores/s, {m['ms_per_run']:.1f} ms a run")
    if "plain_fp32_sparse" in paths and main_key != "plain_fp32_sparse":
        out["batched_over_plain"] = p["value"] / paths["plain_fp32_sparse"]["value"]
        out["target_batched_over_plain"] = 10.0
    if not args.no_cpu:
        log("cpu baseline ...")
        out["cpu_baseline"] = cpu_baseline(env, res, topn)
    print(json.dumps(out), flush=True)


if __name__ == "__main__":
    main()
