"""The search core's own work, as its users have it done, for measurement.

listed()            the cases; each is a dict of plain values.
draw(rng)           one more case of the same ranges.
prepare(case, seed) what a search program holds before the call: the database on the device,
                    preprocessed spectra, the peptide index and batch plan.
run(state)          one pass through the public entry points, and its outputs.
work(case)          bytes and operations that a pass cannot do without.
exact(case, seed)   the same outputs in 64 bits from plain torch and numpy.

A database is fixed by its rules and its size, as a user searches many spectra against one
database.  The precursors of a case are fixed too, up to their order, so that every seed has as
many scores; their order and every peak, score or residual follow from the seed.
"""
from __future__ import annotations

import ctypes as C
import functools
import math

import numpy as np
import torch

from hfx_amd import check, lib, pipeline, synth

STRIDE = 2112   # floats a preprocessed spectrum takes, as the benchmark has it
EPS = 3.0       # precursor window, +- Da
DB_SEED = 29

# digestion rules of the repository's two kinds of workload: every tryptic peptide with up to
# two missed cleavages; peptides of 7 to 30 residues, no cleavage before proline
RULES = {
    "tryptic": dict(missed=2, p_rule=0, min_len=0, max_len=0, static={"C": 57.02146}),
    "short": dict(missed=1, p_rule=1, min_len=7, max_len=30, static={}),
}
# candidates in a spectrum's window, and ladder positions a candidate, by these rules
PAIRS_PER_PROTEIN = {"tryptic": 0.232, "short": 0.183}
PEPTIDES_PER_PROTEIN = {"tryptic": 136.6, "short": 57.5}
POSITIONS = {"tryptic": 17.5, "short": 14.0}
MODS = {"M": 15.9949, "S": 79.9663, "T": 79.9663, "Y": 79.9663}
MAX_MA = 4                    # modification vectors summing below 4
MODDED_PER_PROTEIN = 1.07     # modified candidates a spectrum, per protein
CHARGES = {"tryptic": ((2, 3), (0.5, 0.5)), "short": ((2, 3), (0.7, 0.3)),
           "mods": ((1, 2, 3, 4), (0.1, 0.4, 0.35, 0.15))}
FORMS = {"fp32": pipeline.BatchSearch.FP32_SPARSE, "bf16": pipeline.BatchSearch.BF16X2_DENSE,
         "i8": pipeline.BatchSearch.I8X3_DENSE}


def listed():
    return [
        # the reference's own driver over its C ABI: a group of 16 spectra, their windows and
        # candidate lists, then dense rows, matrix-vector product and sort for each
        dict(name="abi-group", kind="abi", rules="short", proteins=2000, spectra=16),
        # a small file against a small database, scored as it comes
        dict(name="plain-small", kind="plain", rules="short", proteins=2000, spectra=100, topn=5),
        # a whole run against a whole proteome, without an index
        dict(name="plain-large", kind="plain", rules="tryptic", proteins=20000, spectra=10000,
             topn=10),
        # batched searches against an indexed database, in the three forms: planned and run,
        # or captured once and replayed for each new set of spectra of the same size
        dict(name="batch-fp32", kind="batch", form="fp32", rules="tryptic", proteins=20000,
             spectra=4000, topn=5, graph=False, tune=False),
        dict(name="batch-bf16", kind="batch", form="bf16", rules="tryptic", proteins=20000,
             spectra=6000, topn=10, graph=True, tune=False),
        dict(name="batch-i8-small", kind="batch", form="i8", rules="tryptic", proteins=20000,
             spectra=250, topn=5, graph=False, tune=False),
        # the benchmark's own step: 20,000 spectra, tuned and captured
        dict(name="batch-i8-large", kind="batch", form="i8", rules="tryptic", proteins=20000,
             spectra=20000, topn=5, graph=True, tune=True),
        # variable modifications: the whole modified search of a batch
        dict(name="mods", kind="mods", rules="short", proteins=2000, spectra=5000, topn=5),
        # peak lists as an instrument writes them, to correlation-ready arrays
        dict(name="preprocess", kind="preprocess", rules="tryptic", proteins=2000, spectra=20000,
             mean_mode=1),
        # what follows a search: E-values from every score, ion counts of the matches
        dict(name="evalues", kind="evalues", spectra=10000, mean_scores=4600, topn=5),
        dict(name="sp-ions", kind="ions", rules="tryptic", proteins=20000, spectra=10000, topn=5),
        # a new database: residues packed, peptides sorted by residual mass
        dict(name="db-sort", kind="sort", rules="tryptic", proteins=20000),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["abi", "plain", "plain", "batch", "batch", "batch", "mods", "preprocess",
                       "evalues", "ions", "sort"])
    rules = rng.choice(["tryptic", "short"])
    proteins = _log_int(rng, 1000, 20000)
    case = dict(kind=kind, rules=rules, proteins=proteins)
    if kind == "abi":
        return dict(case, rules="short", proteins=_log_int(rng, 500, 4000),
                    spectra=rng.randint(1, 16))
    if kind == "plain":
        return dict(case, spectra=_log_int(rng, 50, 8000), topn=rng.choice([1, 5, 6, 10, 25]))
    if kind == "batch":
        form = rng.choice(sorted(FORMS))
        return dict(case, form=form, spectra=_log_int(rng, 64, 4000 if form == "fp32" else 15000),
                    topn=rng.choice([1, 5, 10]), graph=rng.random() < 0.5, tune=False)
    if kind == "mods":
        return dict(case, rules="short", proteins=_log_int(rng, 500, 2000),
                    spectra=_log_int(rng, 50, 4000), topn=rng.choice([3, 5, 10]))
    if kind == "preprocess":
        return dict(case, proteins=2000, spectra=_log_int(rng, 100, 20000),
                    mean_mode=rng.randint(0, 1))
    if kind == "evalues":
        return dict(kind=kind, spectra=_log_int(rng, 100, 10000),
                    mean_scores=_log_int(rng, 100, 10000), topn=rng.choice([1, 5, 10]))
    if kind == "ions":
        return dict(case, spectra=_log_int(rng, 100, 10000), topn=rng.choice([1, 5, 10]))
    return case


def work(case):
    """Inputs read once, outputs written once; two operations for each peak of a theoretical
    spectrum (ten peaks a ladder position and fragment charge) that a score sums."""
    k = case["kind"]
    S, N = case.get("spectra", 0), case.get("topn", 0)
    spec = 4.0 * STRIDE * S
    top = 20.0 * S * N
    if k == "evalues":
        return dict(bytes=4.0 * S * case["mean_scores"] + 16 * S * N + 40.0 * S,
                    flops=8.0 * S * case["mean_scores"])
    P = case["proteins"] * PEPTIDES_PER_PROTEIN[case["rules"]]
    db = 16 * P + 450.0 * case["proteins"]
    if k == "sort":
        return dict(bytes=12 * P + 900.0 * case["proteins"], flops=P)
    if k == "preprocess":
        return dict(bytes=spec + 8 * 165.0 * S, flops=30.0 * 2000 * S)
    if k == "ions":
        return dict(bytes=spec + 12.0 * S * N + 30.0 * S * N, flops=1.5 * 4 * 20.0 * S * N)
    per = PAIRS_PER_PROTEIN[case["rules"]] * case["proteins"]
    if k == "mods":
        per = MODDED_PER_PROTEIN * case["proteins"]
    peaks = 10 * POSITIONS[case["rules"]] * (1.75 if k == "mods" else 1.4)
    if k == "abi":  # its dense rows are outputs
        return dict(bytes=db + spec + S * per * (4.0 * 1400 + 8), flops=2 * 1400.0 * S * per)
    return dict(bytes=db + spec + top + 4.0 * S * per, flops=2 * peaks * S * per)


# ---------------------------------------------------------------------------- inputs


@functools.lru_cache(maxsize=3)
def _database(rules, proteins):
    w = RULES[rules]
    prot = synth.make_proteins(proteins, seed=DB_SEED)
    mass = pipeline.mass_table(w["static"])
    r, tc, tn = pipeline.digest(prot.seq, prot.seg, mass, 1, w["missed"], 400.0, 7200.0,
                                w["p_rule"], w["min_len"], w["max_len"])
    return prot, pipeline.HostDB(prot.seq, r, tc, tn, mass)


@functools.lru_cache(maxsize=2)
def _device_db(rules, proteins, ma):
    return pipeline.DeviceDB(_database(rules, proteins)[1], ma=ma)


@functools.lru_cache(maxsize=1)
def _mod_info():
    return pipeline.mod_info(MODS, MAX_MA)


@functools.lru_cache(maxsize=1)
def _program():
    """The context and stream that a search program opens once."""
    return pipeline.Ctx(0), pipeline.Stream()


def _spectra(case, seed):
    """Synthetic spectra as synth.make_spectra describes them, made all at once: a peptide's b
    and y ions (doubly charged ones too from 3+ on, intensities 0.2 to 1), three times as many
    noise peaks; with modifications, every second spectrum's peptide carries some.
    Returns (precursor m/z, charge, m/z, intensity, offsets)."""
    prot, h = _database(case["rules"], case["proteins"])
    rng, fixed = np.random.default_rng([seed, 1]), np.random.default_rng(DB_SEED)
    S = case["spectra"]
    mods = case["kind"] == "mods"
    charges, p = CHARGES["mods" if mods else case["rules"]]
    order = rng.permutation(S)
    src = fixed.integers(0, len(h.r), S)[order]
    z = fixed.choice(np.asarray(charges), S, p=p)[order]
    tc, tn = h.tc[src].astype(np.int64), h.tn[src].astype(np.int64)
    ends = np.asarray(prot.seg[1:], np.int64)
    end = ends[np.searchsorted(ends, tc, side="right")]
    n = np.where(tn == end, tn, tn + 1) - tc          # a protein's last piece ends before tn
    first = np.concatenate([[0], np.cumsum(n)])
    sp = np.repeat(np.arange(S), n)
    res = h.ions[np.arange(first[-1]) - first[sp] + tc[sp]]
    m = h.mass.astype(np.float64)[res - 65]
    if mods:
        sites = (fixed.random((S, int(n.max()))) < 0.12) & (fixed.random((S, 1)) < 0.5)
        hit = sites[order][sp, np.arange(len(m)) - first[sp]]
        for a, d in MODS.items():
            m += np.where(hit & (res == ord(a)), d, 0.0)
    cum = np.cumsum(m)
    before = np.concatenate([[0.0], cum])[first[:-1]]
    total = cum[first[1:] - 1] - before
    pcr = ((total + synth.H2O + z * synth.PROTON) / z).astype(np.float32)
    keep = np.arange(len(m)) != first[sp + 1] - 1     # n - 1 ladder positions
    b, s1 = (cum - before[sp])[keep], sp[keep]
    y = total[s1] - b + synth.H2O
    d = z[s1] >= 3
    mz = np.concatenate([b + synth.PROTON, y + synth.PROTON, b[d] / 2 + synth.PROTON,
                         y[d] / 2 + synth.PROTON])
    ss = np.concatenate([s1, s1, s1[d], s1[d]])
    ok = mz <= 2000.0
    mz, ss = mz[ok], ss[ok]
    noise = 3 * np.maximum(np.bincount(ss, minlength=S), 1)
    inten = np.concatenate([rng.uniform(0.2, 1.0, len(mz)), rng.uniform(0.0, 0.3, noise.sum())])
    mz = np.concatenate([mz, rng.uniform(50.0, 2000.0, noise.sum())])
    ss = np.concatenate([ss, np.repeat(np.arange(S), noise)])
    o = np.argsort(ss * 4096.0 + mz)
    off = np.concatenate([[0], np.cumsum(np.bincount(ss, minlength=S))]).astype(np.uint32)
    return pcr, z.astype(np.float32), mz[o].astype(np.float32), inten[o].astype(np.float32), off


def _cuda(a):
    return torch.from_numpy(np.ascontiguousarray(a)).cuda()


class _Memory:
    """Device memory of the library as a tensor, kept while the tensor lives."""

    def __init__(self, p, shape, kind, owner):
        self.owner = owner
        self.__cuda_array_interface__ = dict(shape=tuple(shape), typestr=kind, data=(int(p), False),
                                             version=2)


def _tensor(p, shape, kind, owner):
    if 0 in shape:
        return torch.empty(shape, dtype={"<f4": torch.float32, "<f8": torch.float64,
                                         "<i4": torch.int32, "<i8": torch.int64}[kind])
    return torch.as_tensor(_Memory(p, shape, kind, owner), device="cuda")


# ---------------------------------------------------------------------------- prepare, run


def prepare(case, seed):
    return _PREPARE[case["kind"]](case, seed)


def run(state):
    return state["run"](state)


def _prepare_searched(case, seed, ma=b""):
    ctx, stream = _program()
    db = _device_db(case["rules"], case["proteins"], ma)
    sp = pipeline.DeviceSpectra(ctx, *_spectra(case, seed), STRIDE)
    return dict(ctx=ctx, stream=stream, db=db, sp=sp, case=case)


def _prepare_plain(case, seed):
    st = _prepare_searched(case, seed)
    s = st["search"] = pipeline.PlainSearch(st["ctx"], st["db"], st["sp"], EPS, case["topn"])
    for b in (s.t_pos, s.t_exact, s.t_f32, s.t_cnt):
        b.zero()
    pipeline.sync()
    st["run"] = _run_plain
    return st


def _run_plain(st):
    s = st["search"]
    s.window()
    s.score()
    s.select()
    S, N = s.sp.num_spec, s.topn
    return dict(begin=_tensor(s.t_begin.p, [S], "<i4", s), num=_tensor(s.t_num.p, [S], "<i4", s),
                scores=_tensor(s.t_scores.p, [s.total], "<f4", s.t_scores),
                top_pos=_tensor(s.t_pos.p, [S, N], "<i4", s),
                top_exact=_tensor(s.t_exact.p, [S, N], "<f8", s),
                top_f32=_tensor(s.t_f32.p, [S, N], "<f4", s),
                top_cnt=_tensor(s.t_cnt.p, [S], "<i4", s))


def _prepare_batch(case, seed):
    st = _prepare_searched(case, seed)
    forms = pipeline.PepIndex.IONS if case["form"] == "fp32" else pipeline.PepIndex.LADDER
    st["index"] = pipeline.PepIndex(st["ctx"], st["db"], forms=forms)
    b = st["batch"] = pipeline.BatchSearch(st["ctx"], st["db"], st["sp"], EPS, case["topn"],
                                           stream=st["stream"], index=st["index"])
    b.set_precision(FORMS[case["form"]])
    ptrs = (C.c_void_p * 10)()
    check(lib().hfx_batch_outputs(b.h, ptrs), "hfx_batch_outputs")
    S, N = case["spectra"], case["topn"]
    for i, size in ((0, 4 * S * N), (1, 8 * S * N), (2, 4 * S * N), (3, 4 * S)):
        check(lib().hfx_memset(ptrs[i], 0, size, b.stream.p), "hfx_memset")
    if case["tune"]:
        b.autotune()
    if case["graph"]:
        b.capture()
    b.stream.sync()
    total = b.info()["scores"]
    st["out"] = dict(begin=_tensor(ptrs[7], [S], "<i4", st), num=_tensor(ptrs[8], [S], "<i4", st),
                     scores=_tensor(ptrs[5], [total], "<f4", st),
                     top_pos=_tensor(ptrs[0], [S, N], "<i4", st),
                     top_exact=_tensor(ptrs[1], [S, N], "<f8", st),
                     top_f32=_tensor(ptrs[2], [S, N], "<f4", st),
                     top_cnt=_tensor(ptrs[3], [S], "<i4", st))
    st["run"] = _run_batch
    return st


def _run_batch(st):
    if st["case"]["graph"]:
        st["batch"].replay()
    else:
        st["batch"].run()
    return dict(st["out"])


def _prepare_mods(case, seed):
    mi = _mod_info()
    st = _prepare_searched(case, seed, mi.ma)
    st["search"] = pipeline.ModSearch(st["ctx"], st["db"], st["sp"], mi, EPS, case["topn"])
    st["run"] = _run_mods
    return st


def _run_mods(st):
    ms = st["search"]
    r = ms.run(keep_stages=False)
    there = np.arange(ms.topn) < r.top_cnt[:, None]   # entries past the count are not written
    scores, _, n = ms._scored
    return dict(spec_cand=r.spec_cand, mp_off=r.mp_off, top_cnt=r.top_cnt,
                top_pos=np.where(there, r.top_pos, 0), top_exact=np.where(there, r.top_exact, 0.0),
                top_f32=np.where(there, r.top_f32, np.float32(0)),
                scores=_tensor(scores.p, [n], "<f4", scores))


def _prepare_preprocess(case, seed):
    ctx, _ = _program()
    pcr, charge, mz, inten, off = _spectra(case, seed)
    S = case["spectra"]
    t = dict(pcr=_cuda(pcr), charge=_cuda(charge), mz=_cuda(mz), inten=_cuda(inten),
             off=_cuda(off.astype(np.int32)), x=torch.zeros(S, STRIDE, device="cuda"),
             len=torch.zeros(S, dtype=torch.int32, device="cuda"),
             status=torch.zeros(S, dtype=torch.int32, device="cuda"))
    return dict(ctx=ctx, t=t, case=case, run=_run_preprocess)


def _run_preprocess(st):
    t, case = st["t"], st["case"]
    check(lib().hfx_preprocess(st["ctx"].h, t["x"].data_ptr(), STRIDE, t["len"].data_ptr(),
                               t["status"].data_ptr(), t["mz"].data_ptr(), t["inten"].data_ptr(),
                               t["off"].data_ptr(), t["pcr"].data_ptr(), t["charge"].data_ptr(),
                               case["spectra"], 1, 1, case["mean_mode"], None), "hfx_preprocess")
    return dict(x=t["x"], len=t["len"], status=t["status"])


def _score_sets(case, seed):
    """Scores as a search leaves them: most near zero with a long upper tail, a number of them
    for each spectrum that varies as precursor windows do; and the best N of each."""
    S, N = case["spectra"], case["topn"]
    n = case["mean_scores"] * np.random.default_rng(DB_SEED).lognormal(-0.18, 0.6, S)
    n = np.maximum(np.rint(n), 1).astype(np.int64)[np.random.default_rng([seed, 2]).permutation(S)]
    off = np.concatenate([[0], np.cumsum(n)])
    g = torch.Generator(device="cuda").manual_seed(seed)
    k = int(off[-1])
    u = torch.rand(k, generator=g, device="cuda").clamp_(1e-9)
    scores = torch.randn(k, generator=g, device="cuda") * 1800.0 - 900.0 * torch.log(u)
    best = torch.rand(S, N, generator=g, device="cuda", dtype=torch.float64) * 30000.0
    return scores, off, best


def _prepare_evalues(case, seed):
    ctx, _ = _program()
    S, N = case["spectra"], case["topn"]
    scores, off, best = _score_sets(case, seed)
    f8 = dict(dtype=torch.float64, device="cuda")
    t = dict(scores=scores, off=_cuda(off), best=best, fit=torch.zeros(S, 2, **f8),
             npts=torch.zeros(S, dtype=torch.int32, device="cuda"),
             nused=torch.zeros(S, dtype=torch.int64, device="cuda"), ev=torch.zeros(S, N, **f8))
    return dict(ctx=ctx, t=t, case=case, run=_run_evalues)


def _run_evalues(st):
    t, S, N, h = st["t"], st["case"]["spectra"], st["case"]["topn"], st["ctx"].h
    check(lib().hfx_evalue_fit(h, t["fit"].data_ptr(), t["npts"].data_ptr(), t["nused"].data_ptr(),
                               t["scores"].data_ptr(), t["off"].data_ptr(), None, None, S, 350,
                               3.0, None), "hfx_evalue_fit")
    check(lib().hfx_evalues(h, t["ev"].data_ptr(), t["fit"].data_ptr(), t["best"].data_ptr(), None,
                            N, S, None), "hfx_evalues")
    return dict(fit=t["fit"], npts=t["npts"], nused=t["nused"], ev=t["ev"])


def _prepare_ions(case, seed):
    st = _prepare_searched(case, seed)
    S, N = case["spectra"], case["topn"]
    s = pipeline.PlainSearch(st["ctx"], st["db"], st["sp"], EPS, N)
    s.window()
    num = _tensor(s.t_num.p, [S], "<i4", s).cpu()
    begin = _tensor(s.t_begin.p, [S], "<i4", s).clone()
    rng = np.random.default_rng([seed, 3])
    cnt = np.minimum(num.numpy(), N)
    pos = np.zeros((S, N), np.int32)
    for k in range(N):   # distinct positions all over the window
        pos[:, k] = np.maximum(num.numpy().astype(np.int64) - 1, 0) * (k + rng.random(S)) / N
    out = [torch.zeros(S, N, dtype=torch.int32, device="cuda") for _ in range(3)]
    return dict(st, begin=begin, pos=_cuda(pos), cnt=_cuda(cnt), out=out, run=_run_ions)


def _run_ions(st):
    nb, ny, tot = st["out"]
    check(lib().hfx_sp_ions_topn(st["ctx"].h, nb.data_ptr(), ny.data_ptr(), tot.data_ptr(),
                                 st["pos"].data_ptr(), st["cnt"].data_ptr(),
                                 st["begin"].data_ptr(), st["case"]["topn"],
                                 C.byref(st["db"].desc), C.byref(st["sp"].desc), 1, None),
          "hfx_sp_ions_topn")
    return dict(nb=nb, ny=ny, total=tot)


def _residuals(case, seed):
    """A database's residuals as another one of its size has them: in protein order."""
    h = _database(case["rules"], case["proteins"])[1]
    return np.roll(h.r, seed % len(h.r)), np.roll(h.ions, seed % len(h.ions))


def _prepare_sort(case, seed):
    r, ions = _residuals(case, seed)
    t = dict(r=_cuda(r), ions=_cuda(ions))
    t["idx"] = torch.zeros(len(r), dtype=torch.int32, device="cuda")
    return dict(t=t, case=case, run=_run_sort)


def _run_sort(st):
    t = st["t"]
    keys, packed = t["r"].clone(), t["ions"].clone()   # both calls work in place
    lib().prepare_ions(packed.data_ptr(), packed.numel(), None, 0)
    lib().sort_idx_f(keys.data_ptr(), t["idx"].data_ptr(), keys.numel(), 0)
    return dict(keys=keys, idx=t["idx"], ions=packed)


def _prepare_abi(case, seed):
    st = _prepare_searched(case, seed)
    S = case["spectra"]
    i4 = dict(dtype=torch.int32, device="cuda")
    st["t"] = dict(begin=torch.zeros(S, **i4), end=torch.zeros(S, **i4), num=torch.zeros(S, **i4))
    blas = C.c_void_p()
    check(lib().hfx_blas_create(C.byref(blas)), "hfx_blas_create")
    st["lens"] = [int(v) for v in st["sp"].lengths()]
    return dict(st, blas=blas, run=_run_abi)


def _run_abi(st):
    """Search.hs's sequence over algorithms.h, spectrum by spectrum."""
    L, db, sp, t = lib(), st["db"], st["sp"], st["t"]
    S = sp.num_spec
    total = L.findSpecCandsByMass(t["begin"].data_ptr(), t["end"].data_ptr(), t["num"].data_ptr(),
                                  db.t_r.p, db.t_idx.p, db.num_pep, sp.t_mass.p, S, EPS)
    num = t["num"].tolist()
    idx = torch.empty(max(total, 1), dtype=torch.int32, device="cuda")
    scores = torch.empty(max(total, 1), dtype=torch.float32, device="cuda")
    L.prepare_scoring(idx.data_ptr(), db.t_idx.p, t["begin"].data_ptr(), t["num"].data_ptr(), S)
    rows = torch.empty(max(n * k for n, k in zip(num, st["lens"])) or 1, device="cuda")
    o = 0
    for s, (n, k) in enumerate(zip(num, st["lens"])):
        at = idx.data_ptr() + 4 * o
        y = scores.data_ptr() + 4 * o
        L.addIons(rows.data_ptr(), db.t_r.p, db.t_mass.p, db.t_ions.p, db.t_tc.p, db.t_tn.p, at, n,
                  int(sp.zmax[s]), k)
        L.mvm_ff(st["blas"], y, rows.data_ptr(), sp.t_x.p + 4 * s * sp.x_stride, n, k)
        L.sort_b40c_f(y, at, n)
        o += n
    return dict(num=t["num"], scores=scores[:total], idx=idx[:total])


_PREPARE = dict(abi=_prepare_abi, plain=_prepare_plain, batch=_prepare_batch, mods=_prepare_mods,
                preprocess=_prepare_preprocess, evalues=_prepare_evalues, ions=_prepare_ions,
                sort=_prepare_sort)

# ---------------------------------------------------------------------------- in 64 bits

H, H2O, NH3, CO = (np.float32(v) for v in (1.0078246, 18.01056, 17.02655, 27.9949))
HOST_H, HOST_H2O = np.float32(1.007276), np.float32(18.010565)
BIN = np.float32(1.0005079)


def exact(case, seed):
    f = _EXACT.get(case["kind"])
    return f(case, seed) if f else None


def _exact_preprocess(case, seed, dtype=np.float64):
    """x of every spectrum, [S, STRIDE]: binned square roots, ten regions scaled to 50, less the
    mean of 151 bins around (bins and cut-offs by the 32-bit rule that defines them)."""
    pcr, charge, mz, inten, off = _spectra(case, seed)
    S = len(pcr)
    f4 = np.float32
    cut = np.minimum(f4(50) + pcr * charge,
                     (np.trunc(mz[off[1:].astype(np.int64) - 1] / f4(10)) * f4(10)).astype(f4))
    ln = (f4(75) + np.ceil(cut)).astype(np.int64)
    sp = np.repeat(np.arange(S), np.diff(off.astype(np.int64)))
    keep = (mz <= cut[sp]) & ((mz <= (pcr - f4(15))[sp]) | ((pcr + f4(15))[sp] <= mz))
    at = np.rint(mz / BIN).astype(np.int64)
    keep &= at < ln[sp]
    e = torch.zeros(S * STRIDE, dtype=torch.float64)
    e.scatter_reduce_(0, torch.from_numpy((sp * STRIDE + at)[keep]),
                      torch.from_numpy(np.sqrt(inten.astype(dtype))[keep].astype(np.float64)), "amax")
    e = e.numpy().reshape(S, STRIDE).astype(dtype)
    sel = (ln - 75) // 10
    x = np.zeros((S, STRIDE), dtype)
    i = np.arange(STRIDE)
    for s in range(S):
        n, k = int(ln[s]), int(sel[s])
        if n < 85 or n > STRIDE:
            continue
        a = np.zeros(n, dtype)
        top = e[s, : 10 * k].reshape(10, k).max(1)
        a[: 10 * k] = (dtype(50) * np.divide(e[s, : 10 * k].reshape(10, k), top[:, None],
                                             out=np.zeros((10, k), dtype),
                                             where=top[:, None] > 1e-6)).reshape(-1)
        c = np.concatenate([[0.0], np.cumsum(a, dtype=np.float64)])
        w0 = np.maximum(i[:n] - 75, 0)
        mean = (c[np.minimum(w0 + 151, n)] - c[w0]) / 150.0
        x[s, :n] = a - mean
    return x


def _exact_x(case, seed):
    return _exact_preprocess(case, seed, dtype=np.float32)


def _div(a, d):
    """a / d correctly rounded to 32 bits (twice 24 bits and two more fit in 53)."""
    return (a.double() / float(d)).float()


def _weights(b, r, n, z, K):
    """Dense theoretical rows [C, K] for the 32-bit b ladders b [C, P] with n positions,
    residuals r, fragment charges 1..z: the largest of 10, 25, 50 that falls on a bin."""
    Cn, P = b.shape
    there = torch.arange(P, device=b.device)[None, :] < n[:, None]
    y = r[:, None] - b
    rows = torch.zeros(Cn, K + 1, device=b.device)
    base = torch.arange(Cn, device=b.device)[:, None] * (K + 1)

    def put(at, w, live):
        ok = live & (at >= 0) & (at < K)
        where = (base + torch.where(ok, at, torch.full_like(at, K).long())).reshape(-1)
        rows.view(-1).scatter_reduce_(0, where, torch.full_like(where, w, dtype=torch.float32),
                                      "amax")

    def bins(m):
        return torch.round(_div(m, BIN)).long()

    for c in range(1, int(z.max()) + 1):
        live = there & (z >= c)[:, None]
        f = np.float32(c)
        zh, h2o, nh3 = float(H * f), float(H2O / f), float(NH3 / f)
        mb = _div(b + zh, f)
        my = _div((y + float(H2O)) + zh, f)
        for m in (_div((b - float(CO)) + zh, f), mb - h2o, mb - nh3, my - nh3):
            put(bins(m), 10.0, live)
        for m in (mb, my):
            at = bins(m)
            for q, w in ((at, 50.0), (at - 1, 25.0), (at + 1, 25.0)):
                put(q, w, live)
    return rows[:, :K]


def _ladders(ions, mass, tc, n):
    """32-bit running sums of residue masses, left to right, [C, longest]."""
    P = max(int(n.max()), 1) if len(n) else 1
    j = torch.arange(P, device=ions.device)
    at = torch.clamp(tc[:, None] + j, max=len(ions) - 1)
    m = mass[ions[at].long() - 65]
    b = torch.empty_like(m)
    run_ = torch.zeros(len(tc), device=ions.device)
    for k in range(P):
        run_ = run_ + m[:, k]
        b[:, k] = run_
    return b


class _Exact64:
    """A database on the device for the 64-bit scores."""

    def __init__(self, case):
        h = _database(case["rules"], case["proteins"])[1]
        order = np.argsort(h.r, kind="stable")
        self.r_sorted = h.r[order]
        self.ions, self.mass = _cuda(h.ions), _cuda(h.mass)
        tc, tn = h.tc[order].astype(np.int64), h.tn[order].astype(np.int64)
        self.tc, self.n = _cuda(tc), _cuda(np.maximum(tn - tc, 0))
        self.r, self.host = _cuda(self.r_sorted), h
        self.order = order

    def windows(self, mass):
        lo, hi = mass - np.float32(EPS), mass + np.float32(EPS)
        b = np.searchsorted(self.r_sorted, lo, "left")
        return b, np.searchsorted(self.r_sorted, hi, "right") - b


def _masses(case, seed):
    pcr, charge = _spectra(case, seed)[:2]
    m = (pcr * charge - (charge - np.float32(1)) * HOST_H) - (HOST_H + HOST_H2O)
    return m.astype(np.float32), np.maximum(1, np.rint(charge - 1)).astype(np.int64)


def _exact_scores(case, seed):
    """Every score of every window, spectrum after spectrum, and the windows."""
    q = _Exact64(case)
    mass, z = _masses(case, seed)
    begin, num = q.windows(mass)
    off = np.concatenate([[0], np.cumsum(num)])
    X = _cuda(_exact_x(case, seed)).double()
    out = torch.zeros(int(off[-1]), dtype=torch.float64, device="cuda")
    for level in np.unique(z):
        group = np.nonzero(z == level)[0]
        group = group[np.argsort(begin[group], kind="stable")]
        for g0 in range(0, len(group), 128):
            block = [s for s in group[g0:g0 + 128] if num[s]]
            if not block:
                continue
            at = int(begin[block].min())
            end = int((begin[block] + num[block]).max())
            for p0 in range(at, end, 60000):
                p1 = min(p0 + 60000, end)
                n = q.n[p0:p1]
                b = _ladders(q.ions, q.mass, q.tc[p0:p1], n)
                w = _weights(b, q.r[p0:p1], n, torch.full_like(n, int(level)), STRIDE)
                got = w.double() @ X[_cuda(np.asarray(block))].t().contiguous()
                for k, s in enumerate(block):
                    lo, hi = max(int(begin[s]), p0), min(int(begin[s] + num[s]), p1)
                    if lo < hi:
                        o = int(off[s]) + lo - int(begin[s])
                        out[o:o + hi - lo] = got[lo - p0:hi - p0, k]
    return out, off


def _best(scores, off, N):
    """The N best of each spectrum's scores, best first, zeros where there are fewer."""
    S = len(off) - 1
    seg = torch.repeat_interleave(torch.arange(S, device="cuda"), _cuda(np.diff(off)))
    s, o = torch.sort(scores, descending=True, stable=True)
    s = s[torch.sort(seg[o], stable=True).indices]
    j = torch.arange(N, device="cuda")[None, :]
    at = _cuda(off[:-1])[:, None] + j
    ok = j < _cuda(np.diff(off))[:, None]
    return torch.where(ok, s[at.clamp(max=max(len(s) - 1, 0))], 0.0)


def _exact_search(case, seed):
    scores, off = _exact_scores(case, seed)
    top = _best(scores, off, case["topn"])
    return dict(begin=None, num=None, scores=scores, top_pos=None, top_exact=top, top_f32=top,
                top_cnt=None)


def _exact_abi(case, seed):
    scores, off = _exact_scores(case, seed)
    for s in range(len(off) - 1):
        part = scores[int(off[s]):int(off[s + 1])]
        part.copy_(torch.sort(part.clone()).values)
    return dict(num=None, scores=scores, idx=None)


def _subsets(n, k):
    """The k-subsets of n sites as bit masks in the reference's order of ranks: the largest site
    first, ranks past the middle mirrored."""
    total, out = math.comb(n, k), []
    for rank in range(total):
        mirrored = rank > total // 2
        x, a, m = (total - 1 - rank if mirrored else rank), n, 0
        for left in range(k, 0, -1):
            v = a - 1
            while math.comb(v, left) > x:
                v -= 1
            x, a = x - math.comb(v, left), v
            m |= 1 << (n - 1 - v if mirrored else v)
        out.append(m)
    return out


def _exact_mods(case, seed):
    """Scores of all modified candidates: per spectrum and modification the peptides of the
    shifted window that hold the sites, each expanded to its subsets of sites."""
    q, mi = _Exact64(case), _mod_info()
    mass, z = _masses(case, seed)
    S, M, A = len(mass), mi.num_mod, mi.num_ma
    delta, need = mi.mod_delta, _cuda(mi.mod_ma_count.astype(np.int64))
    lo = (mass - np.float32(EPS))[:, None] - delta[None, :]
    hi = (mass + np.float32(EPS))[:, None] - delta[None, :]
    b = np.searchsorted(q.r_sorted, lo.reshape(-1), "left")
    cnt = np.searchsorted(q.r_sorted, hi.reshape(-1), "right") - b
    # acids of each peptide's ladder, and how many of each modifiable one
    P = int(q.n.max())
    res = q.ions[torch.clamp(q.tc[:, None] + torch.arange(P, device="cuda"), max=len(q.ions) - 1)]
    inside = torch.arange(P, device="cuda")[None, :] < q.n[:, None]
    acid = torch.full(res.shape, -1, dtype=torch.int64, device="cuda")
    for a, ch in enumerate(mi.ma):
        acid[(res == ch) & inside] = a
    have = torch.stack([(acid == a).sum(1) for a in range(A)], 1)
    # subset tables
    top_n, top_k = int(have.max()), int(need.max())
    start = torch.zeros(top_n + 1, top_k + 1, dtype=torch.int64)
    choose = torch.zeros(top_n + 1, top_k + 1, dtype=torch.int64)
    masks = []
    for n in range(top_n + 1):
        for k in range(min(n, top_k) + 1):
            start[n, k], choose[n, k] = len(masks), math.comb(n, k)
            masks += _subsets(n, k)
    start, choose = start.cuda(), choose.cuda()
    masks = torch.tensor(masks, dtype=torch.int64, device="cuda")
    X = _cuda(_exact_x(case, seed)).double()
    zt, rs = _cuda(z), q.r
    ma_mass, dl = _cuda(mi.ma_mass), _cuda(delta.astype(np.float32))
    parts, per = [], np.zeros(S, np.int64)
    rows = np.concatenate([[0], np.cumsum(cnt)])
    step = 256
    for s0 in range(0, S, step):
        s1 = min(s0 + step, S)
        lo_r, hi_r = s0 * M, s1 * M
        c = _cuda(cnt[lo_r:hi_r])
        pair = torch.repeat_interleave(torch.arange(lo_r, hi_r, device="cuda"), c)
        pos = _cuda(b)[pair] + torch.arange(len(pair), device="cuda") + int(rows[lo_r]) - _cuda(rows)[pair]
        mod, spec = pair % M, pair // M
        ok = (have[pos] >= need[mod]).all(1)
        pos, mod, spec = pos[ok], mod[ok], spec[ok]
        ways = choose[have[pos], need[mod]]
        many = ways.prod(1)
        row = torch.repeat_interleave(torch.arange(len(pos), device="cuda"), many)
        rank = torch.arange(len(row), device="cuda") - (torch.cumsum(many, 0) - many)[row]
        per[s0:s1] = torch.bincount(spec[row] - s0, minlength=s1 - s0).cpu().numpy()
        for c0 in range(0, len(row), 150000):
            rr, x = row[c0:c0 + 150000], rank[c0:c0 + 150000]
            p, m, s = pos[rr], mod[rr], spec[rr]
            bits = []
            for a in range(A):
                rest = ways[rr][:, a + 1:].prod(1)
                bits.append(masks[start[have[p, a], need[m, a]] + x // rest])
                x = x % rest
            n = q.n[p]
            Pm = max(int(n.max()), 1)
            run_ = torch.zeros(len(p), device="cuda")
            lad = torch.empty(len(p), Pm, device="cuda")
            seen = torch.zeros(len(p), A, dtype=torch.int64, device="cuda")
            for k in range(Pm):
                w = q.mass[res[p, k].long() - 65]
                for a in range(A):
                    is_a = acid[p, k] == a
                    hit = is_a & ((bits[a] >> seen[:, a]) & 1).bool()
                    w = torch.where(hit, w + ma_mass[a], w)
                    seen[:, a] += is_a
                run_ = run_ + w
                lad[:, k] = run_
            wt = _weights(lad, rs[p] + dl[m], n, zt[s], STRIDE)
            parts.append((wt.double() * X[s]).sum(1))
    scores = torch.cat(parts) if parts else torch.zeros(0, dtype=torch.float64, device="cuda")
    top = _best(scores, np.concatenate([[0], np.cumsum(per)]), case["topn"])
    return dict(spec_cand=None, mp_off=None, top_cnt=None, top_pos=None, top_exact=top, top_f32=top,
                scores=scores)


def _exact_evalues(case, seed):
    scores, off, best = _score_sets(case, seed)
    scores, best = scores.cpu().numpy(), best.cpu().numpy()
    S, w = case["spectra"], 350.0
    fit = np.full((S, 2), np.nan)
    for s in range(S):
        x = np.sort(scores[off[s]:off[s + 1]].astype(np.float64))
        n = len(x)
        end = int(np.rint((np.float32(1) - np.float32(3) / np.float32(100)) * np.float32(n)))
        y = (x + 1.0 - x[0])[int(np.rint(0.3 * n)):end]
        k, c = np.unique(np.ceil(y[y > 4000.0] / w), return_counts=True)
        if len(k) < 2:
            continue
        px, py = (k * w - w / 2) / 10000.0, np.log10(c / w)
        dx, dy = px - px.mean(), py - py.mean()
        beta = (dx @ dy) / (dx @ dx)
        fit[s] = py.mean() - beta * px.mean(), beta
    ev = 10.0 ** (fit[:, :1] + fit[:, 1:] * (best / 10000.0))
    return dict(fit=fit, npts=None, nused=None, ev=ev)


_EXACT = dict(
    abi=_exact_abi, plain=_exact_search, batch=_exact_search, mods=_exact_mods,
    evalues=_exact_evalues,
    preprocess=lambda case, seed: dict(x=_exact_preprocess(case, seed), len=None, status=None),
    sort=lambda case, seed: dict(keys=np.sort(_residuals(case, seed)[0]).astype(np.float64),
                                 idx=None, ions=None),
)
