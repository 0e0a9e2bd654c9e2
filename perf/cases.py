"""Performance cases: the work users have this engine do, through its public entry points.

Kinds of case, by what calls them in earnest:

* ``host``         ``Engine.eigenvalues_by_seed``: host seeds in, host eigenvalues out, the form
                   ``calculate_eigenvalues`` and interactive use take (one walk to some thousands);
* ``device``       ``Engine.eigenvalues_by_seed_device``: seeds and eigenvalues resident on the GPU,
                   enqueued on torch's stream (batch simulation, the benchmark's headline);
* ``sweep``        ``Engine.eigenvalues_by_seed_models_device``: the five models of one dim over the
                   same walks, the compute of the production sweep (models 0-4 x dims 1-12);
* ``query``        ``Server.submit`` + ``Server.wait``: one critical-value query;
* ``normals``      ``Engine.walk_normals_device``: the random stream itself, written to memory;
* ``percentiles``  ``Engine.percentiles_device``: quantiles of a finished statistics array.

The sizes are the repository's own workloads: plain runs (model 0, dim 2, T = 1,000, 100,000 walks;
model 2, dim 5, T = 5,000, 1,000,000 walks), the headline (model 4, dim 12, T = 10,000, 1,000,000
walks), the wide dims of the benchmark (20 and 32), the served mix (T log-uniform over 100..10,000,
10,000..1,000,000 walks) and single walks.  The .dat files of a whole simulation are host and disk
work over seeds that are always 1..runs, so they are not a case here; their device work is ``sweep``.
"""
import importlib
import math

import numpy as np
import torch

jne = importlib.import_module("johansen-null-eigenspectra_amd")

QS = (0.90, 0.95, 0.99)
# one engine and one server for the whole program, as a user's program keeps them
_kept = {}


def _engine():
    if "engine" not in _kept:
        _kept["engine"] = jne.Engine(0)
    return _kept["engine"]


def _server():
    if "server" not in _kept:
        _kept["server"] = jne.Server(0, hbm_budget_bytes=1 << 30)
    return _kept["server"]


def listed():
    return [
        # calculate_eigenvalues: one walk, launch and serial latency
        dict(name="one walk d5 T1000", kind="host", model=2, dim=5, steps=1000, n=1, precision="fp64"),
        # the smallest class of served query, submit to answer
        dict(name="query d3 T1000 10k", kind="query", model=4, dim=3, steps=1000, n=10_000, precision="auto"),
        # the plain CPU workload's size on the device
        dict(name="plain d2 T1000 100k", kind="device", model=0, dim=2, steps=1000, n=100_000, precision="fp64"),
        # the plain GPU FP64 workload
        dict(name="plain d5 T5000 1M", kind="device", model=2, dim=5, steps=5000, n=1_000_000, precision="fp64"),
        # the FP64 side of the headline comparison
        dict(name="fp64 d12 T10000 64k", kind="device", model=4, dim=12, steps=10_000, n=65_536, precision="fp64"),
        # the headline
        dict(name="mixed d12 T10000 1M", kind="device", model=4, dim=12, steps=10_000, n=1_000_000,
             precision="mfma_fp16x2"),
        # an odd-sized served chunk in the middle of the mix (auto: the mixed pass)
        dict(name="auto d9 T1237 30011", kind="device", model=3, dim=9, steps=1237, n=30_011, precision="auto"),
        # short FP64 walks at a middle dim, ragged: the eigen solve counts
        dict(name="fp64 d7 T333 50001", kind="device", model=1, dim=7, steps=333, n=50_001, precision="fp64"),
        # one dim of the production sweep
        dict(name="sweep d6 T10000 128k", kind="sweep", model=-1, dim=6, steps=10_000, n=131_072, precision="auto"),
        # the wide dims: the benchmark's largest, and a short ragged batch
        dict(name="wide d32 T10000 16k", kind="device", model=4, dim=32, steps=10_000, n=16_384, precision="fp64"),
        # the stream for callers that consume it on the device (the benchmark's shape)
        dict(name="normals d12 T10000 16k", kind="normals", model=-1, dim=12, steps=10_000, n=16_384, precision="fp64"),
        # the analysis step over a finished run's statistics
        dict(name="percentiles 1M", kind="percentiles", model=-1, dim=12, steps=1, n=1_000_000, precision="fp64"),
    ]


# normals one drawn case draws at most (the largest listed case: 1.2e11)
_MOST_NORMALS = 1.5e10


def _log_int(rng, lo, hi):
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    kind = rng.choices(["device", "host", "query", "sweep", "normals", "percentiles"], [10, 3, 3, 2, 1, 1])[0]
    if kind == "percentiles":
        return dict(kind=kind, model=-1, dim=rng.randint(1, 12), steps=1, n=_log_int(rng, 100, 10_000_000),
                    precision="fp64")
    wide = kind in ("device", "host") and rng.random() < 0.25
    dim = rng.randint(13, 32) if wide else rng.randint(1, 12)
    steps = _log_int(rng, 100, 10_000)
    precision = "fp64" if wide else rng.choice(["fp64", "auto", "mfma_fp16x2"])
    lo, hi = {"device": (1, 1_000_000), "host": (1, 5_000), "query": (10_000, 1_000_000), "sweep": (1_000, 500_000),
              "normals": (1, 100_000)}[kind]
    most = _MOST_NORMALS / (4 if wide or kind == "sweep" else 8 if kind == "normals" else 1)
    n = _log_int(rng, lo, max(lo, min(hi, int(most / (steps * dim)))))
    model = -1 if kind in ("sweep", "normals") else rng.randint(0, 4)
    return dict(kind=kind, model=model, dim=dim, steps=steps, n=n, precision=precision)


def _models(case):
    return list(range(5)) if case["kind"] == "sweep" else [case["model"]]


def _nf(model, dim):
    return dim + 1 if model in (1, 3) else dim


def _host_seeds(case, seed):
    return np.random.default_rng([seed, 77]).integers(1, 2**32, case["n"], dtype=np.uint32)


def _values(case, seed):
    g = torch.Generator("cuda").manual_seed(seed)
    v = torch.zeros(case["n"], dtype=torch.float64, device="cuda")
    for _ in range(case["dim"] + 1):  # a skewed positive statistic, as traces and largest eigenvalues are
        v += torch.randn(case["n"], dtype=torch.float64, device="cuda", generator=g).square()
    return v


def prepare(case, seed):
    s = dict(case, engine=_engine(), prec=jne.PRECISIONS[case["precision"]])
    if case["kind"] == "query":
        s["server"] = _server()
        s["seed"] = (seed * 2654435761 + 12345) & 0xFFFFFFFF
    elif case["kind"] == "percentiles":
        s["values"] = _values(case, seed)
    else:
        h = _host_seeds(case, seed)
        s["seeds"] = h if case["kind"] == "host" else torch.from_numpy(h.view(np.int32)).cuda()
        if case["kind"] in ("device", "sweep"):
            s["out"] = [torch.empty((case["n"], _nf(m, case["dim"])), dtype=torch.float64, device="cuda")
                        for m in _models(case)]
        elif case["kind"] == "normals":
            s["out"] = torch.empty((case["n"], case["steps"], case["dim"]), dtype=torch.float32, device="cuda")
    return s


def run(s):
    e, kind, n = s["engine"], s["kind"], s["n"]
    if kind == "host":
        return e.eigenvalues_by_seed(s["model"], s["dim"], s["steps"], s["seeds"], precision=s["prec"])
    if kind == "query":
        srv = s["server"]
        return srv.wait(srv.submit(s["model"], s["dim"], s["steps"], n, s["seed"], s["precision"]))[0]
    st = torch.cuda.current_stream().cuda_stream
    if kind == "percentiles":
        return e.percentiles_device(s["values"].data_ptr(), n, QS, hip_stream=st)
    if kind == "normals":
        e.walk_normals_device(s["dim"], s["steps"], s["seeds"].data_ptr(), n, s["out"].data_ptr(), hip_stream=st)
    elif kind == "sweep":
        e.eigenvalues_by_seed_models_device(_models(s), s["dim"], s["steps"], s["seeds"].data_ptr(), n,
                                            [o.data_ptr() for o in s["out"]], precision=s["prec"], hip_stream=st)
    else:
        e.eigenvalues_by_seed_device(s["model"], s["dim"], s["steps"], s["seeds"].data_ptr(), n,
                                     s["out"][0].data_ptr(), precision=s["prec"], hip_stream=st)
    return s["out"]


def work(case):
    """Seeds in, results out; the stream's float operations (about 30 per normal) and, per walk, the
    contractions 2 T nF (nF + dim) of S11 and S01."""
    n, d, T = case["n"], case["dim"], case["steps"]
    if case["kind"] == "percentiles":
        return dict(bytes=8.0 * n, flops=2.0 * n)
    flops = 30.0 * n * T * d
    if case["kind"] == "normals":
        return dict(bytes=4.0 * n + 4.0 * n * T * d, flops=flops)
    nb = 0.0 if case["kind"] == "query" else 4.0 * n
    for m in _models(case):
        f = _nf(m, d)
        nb += 48.0 if case["kind"] == "query" else 8.0 * n * f
        flops += 2.0 * n * T * f * (f + d)
    return dict(bytes=nb, flops=flops)


# ---------------------------------------------------------------------------
# The same results in 64 bits: the stream by its definition (Philox4x32-10,
# Box-Muller in float32 operations), the walk, F, S11, S01 and the
# eigenproblem in float64.
# ---------------------------------------------------------------------------
_M32 = 0xFFFFFFFF
_hex = float.fromhex
_LN = [_hex(c) for c in ("0x1.15425cp-4", "-0x1.d962f2p-4", "0x1.e3d33ap-4", "-0x1.fcc1aep-4", "0x1.237a56p-3",
                         "-0x1.5559e6p-3", "0x1.99a13p-3", "-0x1.000008p-2", "0x1.55554ep-2", "-0x1p-1")]
_SIN = [_hex(c) for c in ("0x1.d53624p-14", "-0x1.b1de6p-9", "0x1.cda0f6p-5", "-0x1.d3ba5cp-2", "0x1.1c5832p+0")]
_COS = [_hex(c) for c in ("-0x1.26d016p-16", "0x1.54c234p-11", "-0x1.e36a9ep-7", "0x1.6f5a4ap-3", "-0x1.bea5b6p-1",
                          "0x1.6a09e6p-1")]


def _fma(a, b, c):
    """float32 fma on float64 tensors that hold float32 values (the product of two is exact)."""
    return (a * b + c).float().double()


def _mul(a, b):
    return (a * b).float().double()


def _philox(q, seeds, stream):
    c0, c1, c2, c3 = (q + 0 * seeds) & _M32, (q >> 32) + 0 * seeds, seeds + 0 * q, 0 * (seeds + q)
    k0, k1 = int(stream), 0x4A4E4531
    for _ in range(10):
        p0, p1 = c0 * 0xD2511F53, c2 * 0xCD9E8D57  # the low 64 bits; the shifts below mask the sign
        c0, c1, c2, c3 = (((p1 >> 32) & _M32) ^ c1 ^ k0, p1 & _M32, ((p0 >> 32) & _M32) ^ c3 ^ k1, p0 & _M32)
        k0, k1 = (k0 + 0x9E3779B9) & _M32, (k1 + 0xBB67AE85) & _M32
    return c0, c1, c2, c3


def _normal_pair(wa, wb):
    u = _fma(wa.float().double(), 2.0**-32, 2.0**-33)
    mant, ex = torch.frexp(u)  # mant in [1/2, 1)
    low = mant <= _hex("0x1.6a09e6p-1")
    m = torch.where(low, 2.0 * mant, mant)
    e = torch.where(low, ex - 1, ex).double()
    f = m - 1.0
    q = torch.full_like(f, _LN[0])
    for c in _LN[1:]:
        q = _fma(q, f, c)
    lnm = _fma(_mul(f, f), q, f)
    ln = _fma(e, _hex("0x1.62e43p-1"), _fma(e, _hex("-0x1.05c61p-29"), lnm))
    r = (-2.0 * ln).sqrt().float().double()
    g = ((wb & 0x3FFFFFFF) - 0x20000000).float().double() * 2.0**-30
    x = _mul(g, g)
    sp, cp = torch.full_like(g, _SIN[0]), torch.full_like(g, _COS[0])
    for c in _SIN[1:]:
        sp = _fma(sp, x, c)
    for c in _COS[1:]:
        cp = _fma(cp, x, c)
    s = _mul(g, sp)
    co, si = (cp - s).float().double(), (cp + s).float().double()
    t = wb >> 30
    z0 = torch.where(t == 0, co, torch.where(t == 1, -si, torch.where(t == 2, -co, si)))
    z1 = torch.where(t == 0, si, torch.where(t == 1, co, torch.where(t == 2, -si, -co)))
    return _mul(r, z0), _mul(r, z1)


def _stream(seeds, stream, T, d):
    """Normals (n, T, d) in float64 of the walks `seeds` (int64, 0 <= seed < 2^32)."""
    calls = (T * d + 3) // 4
    w = _philox(torch.arange(calls, device=seeds.device)[None, :], seeds[:, None], stream)
    z = torch.stack(_normal_pair(w[0], w[1]) + _normal_pair(w[2], w[3]), dim=2)
    return z.reshape(len(seeds), 4 * calls)[:, :T * d].reshape(len(seeds), T, d)


def _f_rows(model, b):
    """F of the walks b (n, T, d) (B before each step) as (n, T, nF)."""
    n, T, d = b.shape
    u = (torch.arange(1, T + 1, dtype=torch.float64, device=b.device) / T)[None, :, None].expand(n, T, 1)
    if model == 0:
        return b
    if model == 1:
        return torch.cat([b, torch.ones_like(u)], 2)
    if model in (2, 3):
        x = b[:, :, :d - 1] if model == 2 else b
        return torch.cat([x - x.mean(1, keepdim=True), u - 0.5], 2)
    x = torch.cat([b[:, :, :d - 1], u * u], 2)
    z = torch.cat([torch.ones_like(u), u], 2)
    zt = z.transpose(1, 2).contiguous()
    return x - z.contiguous() @ torch.linalg.solve((zt @ z).cpu(), (zt @ x).cpu()).to(b.device)


def _eigenvalues(models, T, d, z):
    b = torch.cumsum(torch.cat([torch.zeros_like(z[:, :1]), z * math.sqrt(1.0 / T)], 1), 1)
    prev, db = b[:, :T].contiguous(), (b[:, 1:] - b[:, :T]).contiguous()
    outs = []
    for m in models:
        f = _f_rows(m, prev).contiguous()
        ft = f.transpose(1, 2).contiguous()
        s11, s10 = ((ft @ f) / T).cpu(), (ft @ db).cpu()
        w = torch.linalg.solve_triangular(torch.linalg.cholesky(s11), s10, upper=False)
        ev = torch.linalg.eigvalsh(w.transpose(1, 2).contiguous() @ w).abs().sort(1, descending=True).values
        if m in (1, 3):
            ev = torch.cat([ev, torch.zeros_like(ev[:, :1])], 1)
        outs.append(ev)
    return outs


def _quantiles(v):
    v = np.sort(np.asarray(v, dtype=np.float64))
    got = []
    for p in QS:
        rank = p * (len(v) - 1)
        lo, hi = math.floor(rank), math.ceil(rank)
        got.append(float(v[lo]) if lo == hi else float(v[lo] * (1.0 - (rank - lo)) + v[hi] * (rank - lo)))
    return got


def exact(case, seed):
    n, d, T, kind = case["n"], case["dim"], case["steps"], case["kind"]
    if kind == "percentiles":
        return _quantiles(_values(case, seed).cpu().numpy())
    # about 2e8 normals/s in all, and the host's eigen solves
    if n * T * d > 1.2e9 or n * len(_models(case)) * d**2 > 1.5e7:
        return None
    dev = torch.device("cuda" if torch.cuda.is_available() else "cpu")
    if kind == "query":
        seeds, stream = torch.arange(1, n + 1, device=dev), prepare(case, seed)["seed"]
    else:
        seeds, stream = torch.from_numpy(_host_seeds(case, seed).astype(np.int64)).to(dev), 0
    step = max(1, min(4096, int(1.6e7 / (T * (d + 4)))))
    parts = []
    for at in range(0, n, step):
        z = _stream(seeds[at:at + step], stream, T, d)
        parts.append([z.cpu()] if kind == "normals" else _eigenvalues(_models(case), T, d, z))
    outs = [torch.cat([p[k] for p in parts]) for k in range(len(parts[0]))]
    if kind == "query":
        ev = outs[0].numpy()
        return np.array(_quantiles(ev.sum(1)) + _quantiles(ev.max(1)))
    return outs[0].numpy() if kind == "host" else outs[0] if kind == "normals" else outs
