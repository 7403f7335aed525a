"""Performance cases of the decoder: what its users have it do, through its
public entry points, from one syndrome to the largest batches.

``listed()`` names the cases, ``draw()`` gives further ones of the same
ranges, ``prepare()`` makes what a program holds before the call (inputs on
the GPU from a seed, compiled decoders, output buffers), ``run()`` is one
pass, ``work()`` its unavoidable bytes and operations and ``exact()`` the
same results in 64 bits by a method of its own: a sweep over the error
variables that keeps the joint weight of the open parities, which is exact
for every code and detector error model here and shares nothing with the
contraction.

Reduced-precision decodes return class posteriors, the FP32 quantity that
programs read from them; the exact FP64 decode returns its marginals.
"""
import functools
import math
import os
import sys

import numpy as np
import torch

_ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
_PKG = os.path.join(_ROOT, "tensorqec.jl_amd")
if _PKG not in sys.path:
    sys.path.insert(0, _PKG)

from tensorqec import decoders as D  # noqa: E402
from tensorqec import learned  # noqa: E402
from tensorqec import lib as L  # noqa: E402
from tensorqec import planio, tnmap  # noqa: E402
from tensorqec.circuits import detector_error_model_from_stim, rotated_memory_z  # noqa: E402
from tensorqec.codes import CSSTannerGraph, ShorCode, SteaneCode, SurfaceCode, ToricCode  # noqa: E402
from tensorqec.errors import iid_error  # noqa: E402
from tensorqec.gf2 import gf2_right_inverse, logical_operator  # noqa: E402

DEV = "cuda:0"
HIDDEN = 512

# Multiply-adds per syndrome of the contraction trees that the planner finds
# for these problems (sum-product; "map": max-product), and of one sample,
# recovery and check of the logical-error loop (bit operations).
MACS = {"steane": 496, "shor": 48, "surface3": 272, "surface5": 3216, "surface7": 21328, "toric3": 312448,
        "toric5": 1329914864, "dem3x3": 262672, "dem5x2": 15210656}
MAP_MACS = {"surface3": 332, "surface5": 2652}
# (syndrome bits, error variables, classes)
SIZES = {"steane": (6, 14, 4), "shor": (8, 18, 4), "surface3": (8, 18, 4), "surface5": (24, 50, 4),
         "surface7": (48, 98, 4), "toric3": (16, 36, 16), "toric5": (48, 100, 16), "dem3x3": (24, 197, 2),
         "dem5x2": (48, 415, 2)}


def listed():
    return [
        # one shot in a feedback loop: a host program decodes one syndrome with the default decoder
        {"name": "one_d5", "kind": "one", "code": "surface5", "p": 0.05, "n": 1},
        # a data set read from a file, decoded from host arrays with the default decoder
        {"name": "host_d7_3000", "kind": "host", "code": "surface7", "p": 0.05, "n": 3000},
        # a small online batch already on the GPU: latency of one launch
        {"name": "small_d3_100", "kind": "decode", "code": "surface3", "p": 0.05, "n": 100},
        # the headline workload: the committed d=7 plan, 65,536 syndromes on the GPU
        {"name": "batch_d7_65536", "kind": "decode", "code": "surface7", "p": 0.05, "n": 65536},
        # exact FP64 decoding of a ragged batch
        {"name": "exact_d7_10007", "kind": "exact64", "code": "surface7", "p": 0.05, "n": 10007},
        # circuit-level noise: detector error model of a d=5, 2-round memory experiment
        {"name": "circuit_d5r2_4096", "kind": "decode", "code": "dem5x2", "p": 0.001, "n": 4096},
        # the widest network decoded without slicing
        {"name": "toric5_512", "kind": "decode", "code": "toric5", "p": 0.09, "n": 512},
        # most probable error instead of most probable class
        {"name": "map_d5_16384", "kind": "map", "code": "surface5", "p": 0.05, "n": 16384},
        # one point of a threshold plot: sample, decode, recover, check, on the GPU
        {"name": "ler_d7_262144", "kind": "ler", "code": "surface7", "p": 0.05, "n": 262144},
        # inference of the learned front-end on the d=9 code's 80 syndrome bits
        {"name": "mlp_d9_65536", "kind": "mlp", "inputs": 80, "classes": 4, "n": 65536},
        # one training step's loss and gradients at the trainer's batch size
        {"name": "train_d7_8192", "kind": "train", "inputs": 48, "classes": 4, "n": 8192},
        # a window of a stream: batches of uneven size of several codes in one launch
        {"name": "stream_24", "kind": "stream", "p": 0.05, "n": 4096, "batches": 24},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["one", "host", "decode", "decode", "decode", "exact64", "wide", "map", "ler", "mlp", "train",
                       "stream"])
    p = rng.choice([0.02, 0.05, 0.08])
    if kind == "one":
        return {"kind": kind, "code": rng.choice(["surface3", "surface5", "surface7"]), "p": p, "n": 1}
    if kind == "host":
        return {"kind": kind, "code": rng.choice(["surface3", "surface5", "surface7"]), "p": p,
                "n": _log_int(rng, 2, 8000)}
    if kind in ("decode", "exact64"):
        return {"kind": kind, "code": rng.choice(["surface3", "surface5", "surface7"]), "p": p,
                "n": _log_int(rng, 1, 65536)}
    if kind == "wide":
        code = rng.choice(["toric3", "dem3x3", "dem5x2", "toric5"])
        most = {"toric3": 16384, "dem3x3": 16384, "dem5x2": 4096, "toric5": 512}[code]
        return {"kind": "decode", "code": code, "p": 0.001 if code.startswith("dem") else 0.09,
                "n": _log_int(rng, 16, most)}
    if kind == "map":
        return {"kind": kind, "code": rng.choice(["surface3", "surface5"]), "p": p, "n": _log_int(rng, 1, 65536)}
    if kind == "ler":
        return {"kind": kind, "code": rng.choice(["surface3", "surface5", "surface7", "dem3x3"]),
                "p": rng.choice([0.02, 0.05, 0.08]), "n": _log_int(rng, 4096, 262144)}
    if kind == "mlp":
        return {"kind": kind, "inputs": rng.choice([24, 48, 80]), "classes": rng.choice([2, 4]),
                "n": _log_int(rng, 16, 65536)}
    if kind == "train":
        return {"kind": kind, "inputs": rng.choice([24, 48, 80]), "classes": rng.choice([2, 4]),
                "n": 32 * _log_int(rng, 8, 256)}
    return {"kind": kind, "p": p, "n": _log_int(rng, 64, 4096), "batches": rng.randint(4, 48)}


# ---------------------------------------------------------------------------
# Problems and compiled decoders (kept for the life of a program)
# ---------------------------------------------------------------------------

STREAM_CODES = ("steane", "shor", "surface3", "surface5", "toric3")


def _code(name):
    return {"steane": SteaneCode, "shor": ShorCode}[name]() if name in ("steane", "shor") else \
        (SurfaceCode if name.startswith("surface") else ToricCode)(int(name[-1]), int(name[-1]))


@functools.lru_cache(None)
def problem(code, p):
    """The decoding problem as arrays: what each elementary outcome of each
    error variable does.  A variable's outcomes are (probability, flipped
    checks, flipped logical bits)."""
    if code.startswith("dem"):
        dem = detector_error_model_from_stim(rotated_memory_z(int(code[3]), int(code[5]), p))
        Dm, Lm = np.asarray(dem.detector_matrix()), np.asarray(dem.logical_matrix())
        var = [[(1 - r, (), ()), (r, tuple(np.flatnonzero(Dm[:, j])), tuple(np.flatnonzero(Lm[:, j])))]
               for j, r in enumerate(dem.error_rates)]
        return {"dem": dem, "vars": var, "ns": Dm.shape[0], "nl": Lm.shape[0]}
    t = CSSTannerGraph.from_code(_code(code))
    em = iid_error(p / 3, p / 3, p / 3, t.nq)
    lx, lz = logical_operator(t)
    Hx, Hz, k, nsx = np.asarray(t.stgx.H), np.asarray(t.stgz.H), lx.shape[0], t.stgx.ns
    var = []
    for j in range(t.nq):
        x = tuple(nsx + np.flatnonzero(Hz[:, j])), tuple(k + np.flatnonzero(lz[:, j]))
        z = tuple(np.flatnonzero(Hx[:, j])), tuple(np.flatnonzero(lx[:, j]))
        y = tuple(np.concatenate([x[0], z[0]]).astype(int)), tuple(np.concatenate([x[1], z[1]]).astype(int))
        var.append([(1 - p, (), ()), (p / 3, *x), (p / 3, *y), (p / 3, *z)])
    return {"tanner": t, "em": em, "lx": lx, "lz": lz, "vars": var, "ns": t.ns, "nl": 2 * k}


def _wide(code):
    return code.startswith("dem") or code == "toric5"


@functools.lru_cache(None)
def decoder(code, p):
    """``compile(TNMMAP(), ...)``: the default decoder, and the
    nested-dissection optimizer for the wide networks."""
    q = problem(code, p)
    opt = {"optimizer": D.Dissection()} if _wide(code) else {}
    if code.startswith("dem"):
        return D.compile(D.TNMMAP(**opt), q["dem"])
    if code == "toric5":
        opt["tabulate_bits"] = 0
    return D.compile(D.TNMMAP(**opt), q["tanner"], q["em"])


@functools.lru_cache(None)
def plan(code, p):
    """Library plan of a device-side decode; d=7 from the committed plan files."""
    if code == "surface7":
        path = os.path.join(_PKG, "plans", "surface_d7_p%03d_seed11.json" % round(1000 * p))
        return L.HipPlan(planio.load_plan(path)[0], tabulate_bits=8)
    return decoder(code, p).hip


@functools.lru_cache(None)
def map_decoder(code, p):
    q = problem(code, p)
    return D.compile(tnmap.TNMAP(factorize=True), q["tanner"], q["em"])


@functools.lru_cache(None)
def ler_loop(code, p, batch):
    q = problem(code, p)
    if "dem" in q:
        dem, ct = q["dem"], decoder(code, p)
        smp = L.HipSampler.flips(dem.error_rates, dem.detector_matrix(), dem.logical_matrix())
        rec = L.HipRecovery.dem(ct.pure, ct.l2q_mask)
    else:
        t = q["tanner"]
        smp = L.HipSampler.css(t, q["em"], q["lx"], q["lz"])
        rec = L.HipRecovery.css(t, gf2_right_inverse(t.stgz.H), gf2_right_inverse(t.stgx.H), q["lx"], q["lz"])
    return L.HipLER(plan(code, p), smp, rec, batch=batch)


@functools.lru_cache(None)
def stream_executor(p, max_batches, max_rows):
    mx = L.HipMixed([decoder(c, p).hip for c in STREAM_CODES], max_batches=max_batches, max_rows=max_rows)
    mx.set_kernel(True)
    return mx


# ---------------------------------------------------------------------------
# Inputs
# ---------------------------------------------------------------------------


def syndromes(code, p, n, seed):
    """n syndrome rows (uint8, on the GPU) of errors drawn from the noise model."""
    q = problem(code, p)
    gen = torch.Generator(device=DEV).manual_seed(seed)
    nv = len(q["vars"])
    cum = torch.tensor(np.cumsum([[o[0] for o in v] for v in q["vars"]], axis=1), device=DEV)
    flips = torch.zeros((nv * (cum.shape[1] - 1), q["ns"]), device=DEV)
    for j, v in enumerate(q["vars"]):
        for i, o in enumerate(v[1:]):
            flips[(i * nv) + j, list(o[1])] = 1
    rows = torch.empty((n, q["ns"]), dtype=torch.uint8, device=DEV)
    for a in range(0, n, 65536):
        m = min(65536, n - a)
        u = torch.rand((m, nv), generator=gen, device=DEV, dtype=torch.float64)
        kind = (u[:, :, None] >= cum[None, :, :-1]).sum(dim=2)
        e = torch.cat([(kind == i + 1) for i in range(cum.shape[1] - 1)], dim=1).float()
        rows[a:a + m] = (e @ flips).remainder(2).to(torch.uint8)
    return rows


def _buffers(n, nout):
    return (torch.empty((n, nout), dtype=torch.float64, device=DEV), torch.empty(n, dtype=torch.int32, device=DEV),
            torch.empty(n, dtype=torch.uint8, device=DEV), torch.empty((n, nout), dtype=torch.float32, device=DEV))


def _stream_table(case, seed):
    """(code index, rows) of each batch: codes uniform, sizes log-uniform."""
    rng = np.random.default_rng(case["n"] * 1000 + case["batches"])   # the window's shape belongs to the case
    codes = rng.integers(0, len(STREAM_CODES), case["batches"])
    sizes = np.maximum(1, np.floor(np.exp(rng.uniform(0, np.log(case["n"] + 1), case["batches"])))).astype(int)
    return [(int(c), int(s)) for c, s in zip(codes, sizes)]


def _features(case, seed):
    """Syndrome rows of the learned front-end: sparse bits, as at a few percent of noise."""
    gen = torch.Generator(device=DEV).manual_seed(seed)
    return (torch.rand((case["n"], case["inputs"]), generator=gen, device=DEV) < 0.15).to(torch.uint8)


def _targets(case, seed):
    """Class posteriors, mostly confident."""
    gen = torch.Generator(device=DEV).manual_seed(seed + 1)
    return torch.softmax(6 * torch.randn((case["n"], case["classes"]), generator=gen, device=DEV), dim=1)


def prepare(case, seed):
    kind, n = case["kind"], case["n"]
    s = {"kind": kind, "n": n, "stream": torch.cuda.current_stream().cuda_stream}
    if kind in ("one", "host"):
        code, p = case["code"], case["p"]
        s["ct"] = decoder(code, p)
        rows = syndromes(code, p, n, seed).cpu().numpy()
        nsx = problem(code, p)["tanner"].stgx.ns
        s["syndrome"] = D.CSSSyndrome(rows[0, :nsx], rows[0, nsx:]) if kind == "one" else rows
    elif kind in ("decode", "exact64"):
        code, p = case["code"], case["p"]
        s["mode"] = "spec_f32" if kind == "decode" else "spec_f64"
        s["plan"] = plan(code, p)
        s["rows"] = syndromes(code, p, n, seed)
        s["classes"] = SIZES[code][2]
        s["mar"], s["cls"], s["tie"], s["post"] = _buffers(n, s["classes"])
    elif kind == "map":
        code, p = case["code"], case["p"]
        s["ct"] = map_decoder(code, p)
        s["rows"] = syndromes(code, p, n, seed)
        s["config"] = torch.empty((n, s["ct"].qubit_num), dtype=torch.uint8, device=DEV)
        s["logp"] = torch.empty(n, dtype=torch.float64, device=DEV)
    elif kind == "ler":
        s["ler"] = ler_loop(case["code"], _ler_p(case), min(65536, n))
        s["seed"] = seed
    elif kind in ("mlp", "train"):
        s["mlp"] = learned.HipMLP(case["inputs"], case["classes"], hidden=HIDDEN, seed=seed)
        s["rows"] = _features(case, seed)
        if kind == "mlp":
            s["logits"] = torch.empty((n, case["classes"]), dtype=torch.float32, device=DEV)
        else:
            s["targets"] = _targets(case, seed)
            s["grad"] = torch.empty(s["mlp"].nparams, dtype=torch.float32, device=DEV)
    else:
        table, p = _stream_table(case, seed), case["p"]
        s["mx"] = stream_executor(p, len(table), sum(m for _, m in table))
        s["table"], s["parts"] = [], {}
        for nout in (4, 16):
            mine = [(i, c, m) for i, (c, m) in enumerate(table) if SIZES[STREAM_CODES[c]][2] == nout]
            if not mine:
                continue
            buf = s["parts"][nout] = _buffers(sum(m for _, _, m in mine), nout)
            at = 0
            for i, c, m in mine:
                rows = syndromes(STREAM_CODES[c], p, m, seed * 64 + i)
                s["table"].append((c, m, rows, *(b[at:at + m] for b in buf[:3])))
                at += m
    return s


def _ler_p(case):
    return 0.001 if case["code"].startswith("dem") else case["p"]


# ---------------------------------------------------------------------------
# One pass
# ---------------------------------------------------------------------------


def run(s):
    kind, n, st = s["kind"], s["n"], s["stream"]
    if kind == "one":
        e = D.decode(s["ct"], s["syndrome"]).error_pattern
        return {"x": e.xerror, "z": e.zerror}
    if kind == "host":
        r = D.decode_batch(s["ct"], s["syndrome"])
        return {"marginals": r.marginals, "classes": r.classes, "ties": r.ties, "x": r.error_patterns.xerror,
                "z": r.error_patterns.zerror}
    if kind in ("decode", "exact64"):
        s["plan"].decode_device(s["rows"].data_ptr(), n, s["mode"], s["mar"].data_ptr(), s["cls"].data_ptr(),
                                s["tie"].data_ptr(), st)
        if kind == "exact64":
            return {"marginals": s["mar"], "classes": s["cls"], "ties": s["tie"]}
        learned.posteriors(s["mar"].data_ptr(), n, s["classes"], s["post"].data_ptr(), st)
        return {"posteriors": s["post"], "classes": s["cls"], "ties": s["tie"]}
    if kind == "map":
        s["ct"].hip.map_decode_device(s["rows"].data_ptr(), n, s["ct"].qubit_num, s["config"].data_ptr(),
                                      s["logp"].data_ptr(), st)
        return {"config": s["config"], "logp": s["logp"]}
    if kind == "ler":
        return s["ler"].run("spec_f32", s["seed"], 0, n, st)
    if kind == "mlp":
        s["mlp"].forward(s["rows"].data_ptr(), n, s["logits"].data_ptr(), st)
        return {"logits": s["logits"]}
    if kind == "train":
        loss = s["mlp"].gradients(s["rows"].data_ptr(), s["targets"].data_ptr(), n, s["grad"].data_ptr(), st)
        return {"loss": loss, "grad": s["grad"]}
    s["mx"].decode_device([(c, m, *(x.data_ptr() for x in t)) for c, m, *t in s["table"]], st)
    out = {}
    for nout, (mar, cls, tie, post) in s["parts"].items():
        learned.posteriors(mar.data_ptr(), len(cls), nout, post.data_ptr(), st)
        out["of %d" % nout] = {"posteriors": post, "classes": cls, "ties": tie}
    return out


def work(case):
    kind, n = case["kind"], case["n"]
    if kind in ("mlp", "train"):
        kin, c = (case["inputs"] + 31) // 32 * 32, case["classes"]
        weights = kin * HIDDEN + 2 * HIDDEN * HIDDEN + HIDDEN * c
        params = weights + 3 * HIDDEN + c
        if kind == "mlp":
            return {"bytes": n * (case["inputs"] + 4 * c) + 2 * params, "flops": 2 * n * weights}
        # forward, weight gradients, and input gradients of all layers but the first
        return {"bytes": n * (case["inputs"] + 4 * c) + 8 * params,
                "flops": 2 * n * (2 * weights + weights - kin * HIDDEN)}
    if kind == "stream":
        w = {"bytes": 0, "flops": 0}
        for c, m in _stream_table(case, 0):
            ns, _, nout = SIZES[STREAM_CODES[c]]
            w["bytes"] += m * (ns + 12 * nout + 5)
            w["flops"] += 2 * m * MACS[STREAM_CODES[c]]
        return w
    code = case["code"]
    ns, nv, nout = SIZES[code]
    if kind == "map":
        return {"bytes": n * (ns + nv + 8), "flops": 2 * n * MAP_MACS[code]}
    if kind == "ler":
        # nothing but the counts has to leave the chip
        return {"bytes": 64, "flops": n * (2 * MACS[code] + 60 * nv)}
    if kind in ("one", "host"):
        return {"bytes": n * (ns + 8 * nout + 5 + nv), "flops": 2 * n * MACS[code]}
    return {"bytes": n * (ns + (8 if kind == "exact64" else 4) * nout + 5), "flops": 2 * n * MACS[code]}


# ---------------------------------------------------------------------------
# The same results in 64 bits
# ---------------------------------------------------------------------------


@functools.lru_cache(None)
def _sweep_order(code, p):
    """Order of the error variables that keeps few parities open (greedy, the best of several starts)."""
    touched = [sorted({c for o in v for c in o[1]}) for v in problem(code, p)["vars"]]
    uses = {}
    for t in touched:
        for c in t:
            uses[c] = uses.get(c, 0) + 1
    best = None
    for start in range(0, len(touched), max(1, len(touched) // 24)):
        left, cnt, open_, seq, cost, nxt = set(range(len(touched))), dict(uses), set(), [], 0.0, start
        while left:
            if nxt is None:
                near = [j for j in left if any(c in open_ for c in touched[j])] or sorted(left)
                nxt = min(near, key=lambda j: (sum(c not in open_ for c in touched[j]) -
                                               sum(cnt[c] == 1 for c in touched[j]), j))
            left.discard(nxt)
            seq.append(nxt)
            open_.update(touched[nxt])
            cost += 2.0 ** len(open_)
            for c in touched[nxt]:
                cnt[c] -= 1
                if cnt[c] == 0:
                    open_.discard(c)
            nxt = None
        if best is None or cost < best[0]:
            best = (cost, seq)
    return best[1]


def joint(code, p, rows, best=False):
    """P(syndrome, class) of each row (or, with `best`, the largest weight of
    one error): float64, (n, classes), column-major class order."""
    q = problem(code, p)
    seq = _sweep_order(code, p)
    last = {}
    for i, j in enumerate(seq):
        for o in q["vars"][j]:
            for c in o[1]:
                last[c] = i
    nl = 0 if best else q["nl"]
    peak = _peak_open(q, seq, last) + nl
    out = torch.empty((len(rows), 1 << nl), dtype=torch.float64, device=DEV)
    step = max(1, (1 << 27) >> peak)
    for a in range(0, len(rows), step):
        r = rows[a:a + step].to(torch.int64)
        slots = []
        T = torch.zeros((len(r), 1 << nl), dtype=torch.float64, device=DEV)
        T[:, 0] = 1
        for i, j in enumerate(seq):
            for c in sorted({c for o in q["vars"][j] for c in o[1]}):
                if c not in slots:
                    slots.append(c)
                    T = torch.cat([T, torch.zeros_like(T)], dim=1)
            idx = torch.arange(T.shape[1], device=DEV)
            new = None
            for w, cs, ls in q["vars"][j]:
                m = 0
                for c in cs:
                    m ^= 1 << (nl + slots.index(c))
                for b in (() if best else ls):
                    m ^= 1 << int(b)
                part = w * T[:, idx ^ m]
                new = part if new is None else torch.maximum(new, part) if best else new + part
            T = new
            for c in [c for c in slots if last[c] == i]:
                k = nl + slots.index(c)
                V = T.view(len(r), -1, 2, 1 << k)
                T = V.gather(2, r[:, c].view(-1, 1, 1, 1).expand(-1, V.shape[1], 1, V.shape[3])).reshape(len(r), -1)
                slots.remove(c)
        out[a:a + step] = T
    return out


def _peak_open(q, seq, last):
    open_, peak = set(), 0
    for i, j in enumerate(seq):
        open_ |= {c for o in q["vars"][j] for c in o[1]}
        peak = max(peak, len(open_))
        open_ = {c for c in open_ if last[c] > i}
    return peak


def _network(case, seed):
    """The front-end's network in 64 bits: (parameters, logits)."""
    mlp = learned.HipMLP(case["inputs"], case["classes"], hidden=HIDDEN, seed=seed)
    w = {k: torch.tensor(v, dtype=torch.float64, device=DEV, requires_grad=True)
         for k, v in mlp.unflatten(mlp.init_params(seed)).items()}
    x = torch.zeros((case["n"], mlp.kin), dtype=torch.float64, device=DEV)
    x[:, :case["inputs"]] = _features(case, seed)
    for i in (1, 2, 3):
        x = torch.relu(x @ w["W%d" % i] + w["b%d" % i])
    return [w[k] for k, _ in mlp.layout()], x @ w["W4"] + w["b4"]


def exact(case, seed):
    kind, n = case["kind"], case["n"]
    if kind in ("one", "ler"):
        return None
    if kind == "mlp":
        with torch.no_grad():
            return {"logits": _network(case, seed)[1]}
    if kind == "train":
        w, z = _network(case, seed)
        loss = -(_targets(case, seed).double() * torch.log_softmax(z, dim=1)).sum() / n
        g = torch.autograd.grad(loss, w)
        return {"loss": float(loss), "grad": torch.cat([x.reshape(-1) for x in g])}
    if kind == "stream":
        out = {}
        table, p = _stream_table(case, seed), case["p"]
        for nout in (4, 16):
            mar = [joint(STREAM_CODES[c], p, syndromes(STREAM_CODES[c], p, m, seed * 64 + i))
                   for i, (c, m) in enumerate(table) if SIZES[STREAM_CODES[c]][2] == nout]
            if mar:
                mar = torch.cat(mar)
                out["of %d" % nout] = {"posteriors": mar / mar.sum(dim=1, keepdim=True), "classes": None, "ties": None}
        return out
    code, p = case["code"], case["p"]
    rows = syndromes(code, p, n, seed)
    if kind == "map":
        return {"config": None, "logp": joint(code, p, rows, best=True)[:, 0].log()}
    mar = joint(code, p, rows)
    if kind == "host":
        return {"marginals": mar, "classes": None, "ties": None, "x": None, "z": None}
    if kind == "exact64":
        return {"marginals": mar, "classes": None, "ties": None}
    return {"posteriors": mar / mar.sum(dim=1, keepdim=True), "classes": None, "ties": None}
