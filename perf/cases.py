"""The work that programs using gsbn_amd have it do, as cases to measure.

Four kinds, each through the package's public entry points:

net     one network's whole run: build a Solver from its prototxt, present the
        patterns (training), optionally recall partial cues (each recall
        window after a reset window, so the learning rate switches twice per
        cue), read the learned weights, the biases and the population state,
        close.  Structural options: sparse connections with several delays,
        16-bit trace storage, the separate spike exchange, rewiring.
batch   many independent networks of uneven sizes in lock-step in one Solver.
recall  frozen weights: partial cues of one trained population through a
        Recall handle, with float weights in the reference's order ("exact")
        or bfloat16 weights on the matrix cores ("mfma").
gemm    the support product on its own (gsbn_spike_gemm), on device buffers.
sweep   the full catch-up of every synapse of a projection to a target step
        (gsbn_proj_all), on device buffers.

Sizes are those of gsbn_amd.configs, the tests and bench.py (10 x 10 and
100 x 100 networks, batches of 8-64 HCUs x 16-128 MCUs with connection
probabilities 0.1, 0.5, 0.9, 8192 cues x 50 steps) and odd ones between them.
"""

from __future__ import annotations

import ctypes
import math
import shutil
import tempfile

import numpy as np
import torch

from gsbn_amd import Solver, configs, lib
from gsbn_amd import recall as rc

DT = 0.001
EPS = 0.001


def listed():
    return [
        # the smallest interactive use: one cue of a 10 x 10 network
        dict(name="recall_one_cue", kind="recall", H=10, M=10, cues=1, steps=50, mode="exact",
             frac=0.5),
        # the 10 x 10 experiment from end to end: 2600 steps where launches count
        dict(name="net_10x10", kind="net", H=10, M=10, patterns=10, train=100, quiet=10, recall=100,
             frac=0.5, prec="fp32", p=1.0, delays=1, direct=1, rewire=0),
        # an odd-sized network, half connected with delays of 1 to 8 steps, fp16 traces
        dict(name="net_ragged_fp16", kind="net", H=37, M=53, patterns=12, train=50, quiet=10,
             recall=50, frac=0.3, prec="fp16", p=0.5, delays=8, direct=1, rewire=0),
        # the 100 x 100 network's whole training phase (9.9e7 synapses, 6000 steps)
        dict(name="net_100x100_train", kind="net", H=100, M=100, patterns=100, train=50, quiet=10,
             recall=0, frac=0.3, prec="fp32", p=1.0, delays=1, direct=1, rewire=0),
        # 100 x 100 trained and recalled, 16-bit traces (40 learning-rate switches)
        dict(name="net_100x100_bf16", kind="net", H=100, M=100, patterns=20, train=50, quiet=10,
             recall=50, frac=0.3, prec="bf16", p=1.0, delays=1, direct=1, rewire=0),
        # a small batch of networks, trained and recalled
        dict(name="batch_24", kind="batch", nets=24, layout=1, patterns=10, train=50, quiet=10, recall=50,
             frac=0.5, prec="fp32"),
        # a large batch (0.66e9 synapses)
        dict(name="batch_128", kind="batch", nets=128, layout=2, patterns=6, train=50, quiet=10, recall=50,
             frac=0.5, prec="fp32"),
        # the serving form at full size: 8192 cues x 50 steps, float weights
        dict(name="recall_exact_8192", kind="recall", H=100, M=100, cues=8192, steps=50,
             mode="exact", frac=0.4),
        # the same on the matrix cores
        dict(name="recall_mfma_8192", kind="recall", H=100, M=100, cues=8192, steps=50,
             mode="mfma", frac=0.4),
        # a few hundred cues of an odd-sized population on the matrix cores
        dict(name="recall_mfma_ragged", kind="recall", H=37, M=53, cues=300, steps=50, mode="mfma",
             frac=0.4),
        # the support product alone at the recall shape
        dict(name="gemm_8192", kind="gemm", B=8192, N=10000, K=10000, active=0.001),
        # one full catch-up sweep of a mid-sized projection after 50 steps
        dict(name="sweep_64x80", kind="sweep", H=64, M=80, prec="fp32", gap=50),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    """One more case of the same ranges."""
    kind = rng.choice(["net", "net", "net", "batch", "recall", "recall", "recall", "gemm", "sweep"])
    if kind == "net":
        H, M = _log_int(rng, 6, 100), _log_int(rng, 6, 100)
        small = H * M <= 1200
        prec = rng.choice(["fp32", "fp32", "bf16", "fp16"])
        p = rng.choice([1.0, 1.0, 0.5, 0.1])
        return dict(kind="net", H=H, M=M, patterns=rng.randint(4, 14), train=rng.randint(30, 100),
                    quiet=rng.choice([0, 7, 10, 20]), recall=rng.choice([0, 40, 50, 90]),
                    frac=rng.choice([0.3, 0.5]), prec=prec, p=p, delays=rng.choice([1, 1, 3, 8]),
                    direct=0 if rng.random() < 0.2 else 1,
                    rewire=1 if small and rng.random() < 0.2 else 0)
    if kind == "batch":
        return dict(kind="batch", nets=_log_int(rng, 2, 96), layout=rng.randint(3, 999), patterns=rng.randint(3, 6),
                    train=rng.randint(30, 60), quiet=rng.choice([0, 10]),
                    recall=rng.choice([0, 40, 50]), frac=0.5,
                    prec=rng.choice(["fp32", "fp32", "bf16"]))
    if kind == "recall":
        mode = rng.choice(["exact", "mfma"])
        return dict(kind="recall", H=_log_int(rng, 8, 90), M=_log_int(rng, 8, 90),
                    cues=_log_int(rng, 1, 6000), steps=rng.randint(20, 60), mode=mode,
                    frac=rng.choice([0.3, 0.4, 0.5]))
    if kind == "gemm":
        N = _log_int(rng, 100, 9000)
        return dict(kind="gemm", B=_log_int(rng, 1, 8000), N=N, K=N,
                    active=rng.choice([0.001, 0.01, 0.1]))
    return dict(kind="sweep", H=_log_int(rng, 5, 80), M=_log_int(rng, 5, 90),
                prec=rng.choice(["fp32", "bf16", "fp16"]), gap=rng.randint(1, 200))


# ---------------------------------------------------------------- networks

def _population(H, M):
    return configs.PopSpec(hcu=H, mcu=M, wtagain=4.0, wgain=8.0, snoise=0.1)


def _projection(src, dest, C):
    return configs.ProjSpec(src=src, dest=dest, tauzi=0.01, tauzj=0.01, taue=0.02, taup=1.0,
                            slot_num=float(C))


def _dense(H, M):
    """Every source unit outside the HCU, ascending."""
    src = np.arange(H * M, dtype=np.int32)
    ii = np.stack([src[src // M != h] for h in range(H)])
    return ii.reshape(-1), np.ones(ii.size, np.int32), (H - 1) * M


def _sparse(rng, H, M, p):
    """A fixed share p of the units outside the HCU, ascending; the last slot
    of every HCU left empty."""
    src = np.arange(H * M)
    n = max(1, int(p * (H - 1) * M))
    ii = np.full((H, n + 1), -1, np.int32)
    for h in range(H):
        ii[h, :n] = np.sort(rng.permutation(src[src // M != h])[:n])
    return ii.reshape(-1), (ii >= 0).astype(np.int32).reshape(-1), n + 1


def _stimuli(rng, H, M, n_pat, frac):
    """Patterns, one row of no input, cues; masks: training, one per cue."""
    pats = configs.random_patterns(rng, n_pat, H, M)
    cues, masks = pats.copy(), np.zeros((n_pat, H), np.float32)
    n_clamp = int(round(frac * H))
    for i in range(n_pat):
        free = rng.permutation(H)[n_clamp:]
        cues[i, free] = configs.UNCLAMPED
        masks[i, free] = 1.0
    quiet = np.full((1, H), configs.UNCLAMPED, np.uint32)
    return (np.concatenate([pats, quiet, cues]),
            np.concatenate([np.zeros((1, H), np.float32), masks]))


def _modes(case):
    modes = configs.recall_schedule(case["patterns"], case["train"], case["quiet"],
                                    max(case["recall"], 1), reset=50, dt=DT)
    if case["recall"] == 0:
        modes = modes[:case["patterns"] * (2 if case["quiet"] > 0 else 1)]
    return modes


def _net_spec(case, seed):
    rng = np.random.Generator(np.random.Philox(seed))
    H, M = case["H"], case["M"]
    if case["p"] >= 1.0:
        ii, di, C = _dense(H, M)
    else:
        ii, di, C = _sparse(rng, H, M, case["p"])
    if case["delays"] > 1:
        di = np.where(ii >= 0, rng.integers(1, case["delays"] + 1, ii.size), 0).astype(np.int32)
    stim, mask = _stimuli(rng, H, M, case["patterns"], case["frac"])
    spec = configs.NetSpec(dt=DT, pops=[_population(H, M)], projs=[_projection(0, 0, C)],
                           modes=_modes(case), stim=stim, mask=mask, conn=[[]], conn_arrays=[(ii, di)],
                           seed=seed, name="net", trace_precision=case["prec"],
                           exchange_direct=bool(case["direct"]))
    if case["rewire"]:
        spec.structural = configs.StructuralSpec(period=100, pruning_period=200, seed=seed)
    return spec


def _batch_spec(case, seed):
    """Network sizes and connections by the case's layout, each network's
    patterns, cues and random streams by the seed."""
    spec = configs.batched_nets(case["nets"], n_pat=case["patterns"], train=case["train"],
                                quiet=case["quiet"], recall=max(case["recall"], 1),
                                clamp_frac=case["frac"], seed=case["layout"])
    rng = np.random.Generator(np.random.Philox(seed))
    stimuli = [_stimuli(rng, p.hcu, p.mcu, case["patterns"], case["frac"]) for p in spec.pops]
    spec.stim = np.concatenate([s for s, _ in stimuli], axis=1)
    spec.mask = np.concatenate([m for _, m in stimuli], axis=1)
    spec.seed = seed
    spec.modes = _modes(case)
    spec.trace_precision = case["prec"]
    return spec


class _Directory:
    """A temporary directory that goes with the state that holds it."""

    def __init__(self):
        self.path = tempfile.mkdtemp(prefix="gsbn_case_")

    def __del__(self):
        shutil.rmtree(self.path, ignore_errors=True)


def _prepare_solver(spec, names):
    d = _Directory()
    return dict(dir=d, spec=spec, path=configs.write(spec, d.path), names=names)


def _run_solver(st):
    """The program's run: build, step to the end of the schedule, read."""
    with Solver(st["path"]) as s:
        configs.apply_conn_arrays(s, st["spec"])
        s.run()
        out = {n: np.concatenate([s.vector(v) for v in vs]) if len(vs) > 1 else s.vector(vs[0])
               for n, vs in st["names"].items() if vs}
        correct, total, flags = s.check()
        out["check"] = np.concatenate([np.array([correct, total], np.int32), flags])
    return out


POP_STATE = ("spike", "dsup", "act", "epsc", "bj")
UNIT_STATE = ("pj", "ej", "zj")
SYN_STATE = ("wij", "pij", "eij", "zi2", "zj2", "tij")


def _net_names(case):
    # beyond a few million synapses a program reads the weights only
    syn = SYN_STATE if case["H"] * case["H"] * case["M"] * case["M"] <= 1 << 23 else SYN_STATE[:1]
    return {n: ["%s_0" % n] for n in POP_STATE + UNIT_STATE + syn}


def _batch_names(spec):
    """Every network's population state; the weights of the first networks,
    up to 2^25 (a program reads those of the networks it goes on with)."""
    nets = range(len(spec.pops))
    names = {n: ["%s_%d" % (n, i) for i in nets] for n in POP_STATE + UNIT_STATE}
    total, names["wij"] = 0, []
    for i, (p, q) in enumerate(zip(spec.pops, spec.projs)):
        total += int(p.hcu * p.mcu * q.slot_num)
        if total > 1 << 25:
            break
        names["wij"].append("wij_%d" % i)
    return names


# ------------------------------------------------------------------ recall

def _frozen(H, M, seed):
    """Weights and biases of a population that learned H-wide one-of-M
    patterns: Wij = log(Pij / (Pi Pj)) with recency-weighted pattern
    statistics and a noise floor.  Returns the [Nsrc, N] weights on the
    device, bj [N] and the patterns."""
    g = torch.Generator().manual_seed(seed)
    n_pat = 40
    pats = torch.randint(0, M, (n_pat, H), generator=g)
    x = torch.zeros(n_pat, H * M)
    x.scatter_(1, pats + M * torch.arange(H)[None, :], 1.0)
    age = torch.linspace(0.2, 1.0, n_pat)[:, None]
    x = (x * age).cuda()
    gd = torch.Generator(device="cuda").manual_seed(seed)
    norm = float((age ** 2).sum())
    pij = (x.t() @ x) / norm
    pij = pij * (1 + 0.1 * torch.rand(pij.shape, generator=gd, device="cuda")) + 2e-5
    pi = x.square().sum(0) / norm + 4e-3
    w = torch.log((pij + 1e-6) / ((pi[:, None] + EPS) * (pi[None, :] + EPS)))
    return w, torch.log(pi + EPS).cpu().numpy(), pats.numpy()


def _prepare_recall(case, seed):
    H, M = case["H"], case["M"]
    w, bj, pats = _frozen(H, M, seed)
    ii, di, C = _dense(H, M)
    wij = torch.empty(H, C, M, device="cuda")
    for h in range(H):
        cols = w[:, h * M:(h + 1) * M]
        wij[h, :h * M] = cols[:h * M]
        wij[h, h * M:] = cols[(h + 1) * M:]
    spec = configs.NetSpec(dt=DT, pops=[_population(H, M)], projs=[_projection(0, 0, C)], modes=[],
                           stim=np.zeros((0, H)), mask=np.zeros((0, H)), conn=[[]])
    mode = rc.EXACT if case["mode"] == "exact" else rc.MFMA
    handle = rc.Recall(H, M, C, ii, di, wij.cpu().numpy(), bj, rc.population_params(spec),
                       case["cues"], mode, seed)
    clamp, wmask, _ = rc.cues(pats, case["cues"], case["frac"], seed)
    return dict(recall=handle, clamp=clamp, wmask=wmask, steps=case["steps"],
                raster=case["cues"] * H * M * case["steps"] <= 1 << 21)


def _run_recall(st):
    idx, cnt, raster, _ = st["recall"].run(st["clamp"], st["wmask"], st["steps"],
                                           raster=st["raster"])
    return dict(idx=idx, cnt=cnt, raster=raster)


# ---------------------------------------------------- kernels on own buffers

def _pad(n, m):
    return (n + m - 1) // m * m


def _stream():
    return ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)


def _gemm_inputs(case, seed):
    B, N, K = case["B"], case["N"], case["K"]
    g = torch.Generator(device="cuda").manual_seed(seed)
    kp = _pad(K, 64)
    s = torch.zeros(_pad(B, 256), kp, dtype=torch.bfloat16, device="cuda")
    s[:B, :K] = (torch.rand(B, K, generator=g, device="cuda") < case["active"]).to(torch.bfloat16)
    wt = torch.zeros(_pad(N, 256), kp, dtype=torch.bfloat16, device="cuda")
    wt[:N, :K] = (1.5 * torch.randn(N, K, generator=g, device="cuda")).to(torch.bfloat16)
    e = torch.randn(B, N, generator=g, device="cuda")
    return s, wt, e, kp


def _prepare_gemm(case, seed):
    rc._setup(lib())
    s, wt, e, kp = _gemm_inputs(case, seed)
    return dict(s=s, wt=wt, e=e, kp=kp, B=case["B"], N=case["N"], beta=0.9)


def _run_gemm(st):
    code = lib().gsbn_spike_gemm(st["B"], st["N"], st["kp"], st["s"].data_ptr(), st["wt"].data_ptr(),
                                 st["e"].data_ptr(), st["beta"], _stream())
    if code != 0:
        raise RuntimeError("gsbn_spike_gemm failed with code %d" % code)
    return st["e"]


class _AllArgs(ctypes.Structure):
    """gsbn_all_args of include/gsbn_amd.h."""
    _fields_ = [("H", ctypes.c_int32), ("M", ctypes.c_int32), ("C", ctypes.c_int32),
                ("target", ctypes.c_int32), ("kp", ctypes.c_float), ("wgain", ctypes.c_float),
                ("eps", ctypes.c_float), ("eps2", ctypes.c_float), ("table", ctypes.c_void_p),
                ("table_len", ctypes.c_int32), ("syn", ctypes.c_void_p),
                ("rowst", ctypes.c_void_p), ("pj", ctypes.c_void_p), ("prec", ctypes.c_int32),
                ("syn16", ctypes.c_void_p), ("wij", ctypes.c_void_p), ("p_scale", ctypes.c_float),
                ("e_scale", ctypes.c_float), ("ii", ctypes.c_void_p), ("dhist", ctypes.c_void_p),
                ("dcnt", ctypes.c_void_p), ("dK", ctypes.c_int32), ("kftj", ctypes.c_float)]


KZ, KE, KP = DT / 0.01, DT / 0.02, DT / 1.0
PREC = {"fp32": 0, "bf16": 1, "fp16": 2}
F16_SCALE = 512.0


def _sweep_values(case, seed):
    """Traces of a projection in training: Zi Zj products decayed by a few
    time constants, their averages, last updates up to `gap` steps back."""
    H, M = case["H"], case["M"]
    C = (H - 1) * M
    R = H * C
    g = torch.Generator(device="cuda").manual_seed(seed)

    def rand(*shape):
        return torch.rand(*shape, generator=g, device="cuda")

    v = dict(zi2=rand(R, M) ** 4, zj2=rand(R, M) ** 4)
    v["eij"] = 0.2 * rand(R, M) ** 3
    v["pij"] = 1e-6 + 0.05 * rand(R, M) ** 4
    v["tij"] = torch.randint(0, case["gap"], (R, M), generator=g, device="cuda", dtype=torch.int32)
    v["pi"], v["ei"], v["zi"] = 0.02 * rand(R) + 1e-4, 0.2 * rand(R), rand(R)
    v["ti"] = torch.randint(0, case["gap"], (R,), generator=g, device="cuda", dtype=torch.int32)
    v["pj"] = 0.02 * rand(H * M) + 1e-4
    v["wij"] = torch.log((v["pij"] + 1e-6) / 1e-4)
    return v


def _store16(prec, x):
    """The 16-bit code of a trace (bfloat16, or binary16 scaled)."""
    x = x.to(torch.bfloat16) if prec == "bf16" else (x * F16_SCALE).to(torch.float16)
    return x.view(torch.int16)


def _load16(prec, code):
    if prec == "bf16":
        return code.view(torch.bfloat16).to(torch.float64)
    return code.view(torch.float16).to(torch.float64) / F16_SCALE


def _prepare_sweep(case, seed):
    from gsbn_amd import coeff_entry
    H, M, prec = case["H"], case["M"], case["prec"]
    C = (H - 1) * M
    v = _sweep_values(case, seed)
    if prec == "fp32":
        syn = torch.zeros(H * C, M, 8, device="cuda")
        for k, n in enumerate(("pij", "eij", "zi2", "zj2", "wij")):
            syn[..., k] = v[n]
        syn[..., 5] = v["tij"].view(torch.float32)
        wij = None
    else:
        syn = torch.zeros(H * C, M, 8, dtype=torch.int16, device="cuda")
        syn[..., 0], syn[..., 1] = _store16(prec, v["pij"]), _store16(prec, v["eij"])
        words = syn.view(torch.int32)
        words[..., 1], words[..., 2] = v["zi2"].view(torch.int32), v["zj2"].view(torch.int32)
        words[..., 3] = v["tij"]
        wij = v["wij"].clone()
    row = torch.stack([v["pi"], v["ei"], v["zi"], v["ti"].view(torch.float32)], dim=1).contiguous()
    gaps = case["gap"] + 2
    table = torch.from_numpy(np.stack([coeff_entry(KZ, KZ, KE, KP, d) for d in range(gaps)])).cuda()
    a = _AllArgs()
    a.H, a.M, a.C, a.target = H, M, C, 0
    a.kp, a.wgain, a.eps, a.eps2 = KP, 1.0, KP, KP * KP
    a.table, a.table_len = table.data_ptr(), gaps
    a.rowst, a.pj, a.prec = row.data_ptr(), v["pj"].data_ptr(), PREC[prec]
    a.p_scale = a.e_scale = F16_SCALE if prec == "fp16" else 1.0
    if prec == "fp32":
        a.syn = syn.data_ptr()
    else:
        a.syn16, a.wij = syn.data_ptr(), wij.data_ptr()
    lib().gsbn_proj_all.argtypes = [ctypes.c_void_p, ctypes.c_void_p]
    return dict(args=a, syn=syn, wij=wij, row=row, pj=v["pj"], table=table, gap=case["gap"],
                prec=prec)


def _run_sweep(st):
    """The next sweep, `gap` steps after the last one."""
    st["args"].target += st["gap"]
    code = lib().gsbn_proj_all(ctypes.byref(st["args"]), _stream())
    if code != 0:
        raise RuntimeError("gsbn_proj_all failed with code %d" % code)
    syn, row = st["syn"], st["row"]
    if st["prec"] == "fp32":
        out = dict(traces=syn[..., :5], tij=syn[..., 5].view(torch.int32))
    else:
        words = syn.view(torch.int32)
        kind = torch.bfloat16 if st["prec"] == "bf16" else torch.float16
        out = dict(traces=syn[..., :2].view(kind), z=words[..., 1:3].view(torch.float32),
                   tij=words[..., 3], wij=st["wij"])
    out.update(rows=row[:, :3], ti=row[:, 3].view(torch.int32))
    return out


# ------------------------------------------------------------- the interface

def prepare(case, seed):
    kind = case["kind"]
    if kind == "net":
        st = _prepare_solver(_net_spec(case, seed), _net_names(case))
    elif kind == "batch":
        spec = _batch_spec(case, seed)
        st = _prepare_solver(spec, _batch_names(spec))
    else:
        st = {"recall": _prepare_recall, "gemm": _prepare_gemm, "sweep": _prepare_sweep}[kind](case, seed)
    st["kind"] = kind
    return st


def run(state):
    kind = state["kind"]
    if kind in ("net", "batch"):
        return _run_solver(state)
    return {"recall": _run_recall, "gemm": _run_gemm, "sweep": _run_sweep}[kind](state)


def _schedule_steps(case):
    n = case["patterns"] * (case["train"] + case["quiet"])
    return n + (case["patterns"] * (50 + case["recall"]) if case["recall"] else 0)


def work(case):
    """Bytes: the population state once per step (73 B a unit), 44 B per
    synapse updated (an HCU's units spike with about 0.1 per step while
    stimulated, a spike updates its unit's rows and column once), the initial
    state written and what is read back; the recall's state and the product's
    operands once."""
    kind = case["kind"]
    if kind in ("net", "batch"):
        if kind == "net":
            H, M, p, nets = case["H"], case["M"], case["p"], 1
        else:
            H, M, p, nets = 36, 72, 0.5, case["nets"]
        N, C = H * M, (H - 1) * M * p
        steps = _schedule_steps(case)
        spikes = 0.08 * H * steps
        syn = H * C * M
        upd = spikes * 2 * C * 1.0
        return dict(bytes=nets * (73.0 * N * steps + 44 * upd + 28 * syn), flops=nets * upd * 30.0)
    if kind == "recall":
        N, B, T = case["H"] * case["M"], case["cues"], case["steps"]
        bytes_ = 24.0 * B * N * T + 4.0 * N * N
        if case["mode"] == "exact":
            return dict(bytes=bytes_, flops=(100 + 0.1 * case["H"]) * B * N * T)
        return dict(bytes=bytes_, flops=2.0 * B * N * N * max(T - 3, 0))
    if kind == "gemm":
        B, N, K = case["B"], case["N"], case["K"]
        return dict(bytes=2.0 * B * K + 2.0 * N * K + 8.0 * B * N, flops=2.0 * B * N * K)
    H, M = case["H"], case["M"]
    syn = H * (H - 1) * M * M
    return dict(bytes=(44.0 if case["prec"] == "fp32" else 36.0) * syn, flops=40.0 * syn)


def _exact_gemm(case, seed):
    s, wt, e, _ = _gemm_inputs(case, seed)
    B, N = case["B"], case["N"]
    beta = float(np.float32(0.9))
    return beta * e.double() + s[:B].double() @ wt[:N].double().t()


def _exact_sweep(case, seed):
    """The catch-up in closed form: dz = -kz z, de = ke (z - e), dp = kp (e - p)
    over D steps, z the product Zi Zj for a synapse and Zi for a row."""
    H, M, prec = case["H"], case["M"], case["prec"]
    C = (H - 1) * M
    v = _sweep_values(case, seed)
    f = {k: x.double() for k, x in v.items()}
    if prec != "fp32":
        f["pij"], f["eij"] = (_load16(prec, _store16(prec, v[n])) for n in ("pij", "eij"))

    def catch_up(z, e, p, D, kz):
        a = KE / (KE - kz)
        ez, ee, ep = torch.exp(-kz * D), torch.exp(-KE * D), torch.exp(-KP * D)
        b, c = KP / (KP - kz) * a, KP / (KP - KE)
        p1 = ep * p + b * z * (ez - ep) + c * (e - a * z) * (ee - ep)
        return ee * e + a * z * (ez - ee), p1

    D = case["gap"] - f["tij"]
    eij, pij = catch_up(f["zi2"] * f["zj2"], f["eij"], f["pij"], D, 2 * KZ)
    Dr = case["gap"] - f["ti"]
    ei, pi = catch_up(f["zi"], f["ei"], f["pi"], Dr, KZ)
    zi2, zj2 = f["zi2"] * torch.exp(-KZ * D), f["zj2"] * torch.exp(-KZ * D)
    pj = f["pj"].view(H, 1, M).expand(H, C, M).reshape(H * C, M)
    wij = torch.log((pij + KP * KP) / ((pi[:, None] + KP) * (pj + KP)))
    rows = torch.stack([pi, ei, f["zi"] * torch.exp(-KZ * Dr)], dim=1)
    if prec == "fp32":
        return dict(traces=torch.stack([pij, eij, zi2, zj2, wij], dim=-1), tij=None, rows=rows, ti=None)
    scale = F16_SCALE if prec == "fp16" else 1.0
    return dict(traces=torch.stack([pij, eij], dim=-1) * scale, z=torch.stack([zi2, zj2], dim=-1),
                tij=None, wij=wij, rows=rows, ti=None)


def exact(case, seed):
    """Simulated spiking has no value beyond its own arithmetic (a rounding
    decides a spike): nets, batches and recalls are compared as they are."""
    if case["kind"] == "gemm":
        return _exact_gemm(case, seed)
    if case["kind"] == "sweep":
        return _exact_sweep(case, seed)
    return None
