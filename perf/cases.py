"""Workloads of the phase-space library that its speed is judged by.

Each case is one call (or pair of calls) of the C ABI as a program makes it:

  generate    hpsp_generate into momentum columns and the PhaseSpaceWeight
              column, what a filled Decays container holds
  unweight    hpsp_generate_unweight(_mixed): Generate + Unweight() of one
              container, the accept-reject study's step
  reweight    hpsp_unweight with a functor over stored events: Unweight(F) of
              a Dalitz model with the maximum found over the events
  average     hpsp_average_on of a sum of Breit-Wigners (an integral)
  evaluate    hpsp_evaluate of the weight and three functors per event
  histogram   hpsp_histogram_fill_events: a Dalitz plot of stored events, each
              with its PhaseSpaceWeight
  range       hpsp_histogram_fill_range: a lazy phase_space_range filled into
              an invariant-mass histogram

`exact` restates each of them with plain torch operations in double precision:
the counter-based engines, the GENBOD chain and the partition.
"""
import ctypes
import math

import torch

from hydra_amd import capi

DEV = "cuda:0"
UW_SEED = 0x180EC6D33CFD0ABA  # Decays::Unweight's default
M3, MASSES3 = 5.279, [3.0969, 0.493677, 0.13957]  # B0 -> J/psi K pi
MK, MPI = 0.493677, 0.13957061  # K+ -> 3 pi
BW3 = [(0.892, 0.05, 0.4967141530, -0.1382643012, 1, 2),
       (1.43, 0.11, 0.6476885381, 1.5230298564, 1, 2),
       (0.775, 0.149, -0.2341533747, -0.2341368981, 0, 2)]
BW2 = BW3[:1] + BW3[2:]


# ---- the cases ----------------------------------------------------------------

def listed():
    return [
        # the smallest request a generator service gets: a two-body decay of a
        # thousand events in single precision columns; launch latency counts
        {"name": "generate_2body_mixed_1e3", "path": "generate", "N": 2, "n": 1000,
         "engine": "squares3", "prec": "mixed", "decay": "flat"},
        # the plain toy study: 10^6 weighted three-body events, FP64
        {"name": "generate_3body_1e6", "path": "generate", "N": 3, "n": 1000000,
         "engine": "squares3", "prec": "fp64", "decay": "jpsikpi"},
        # the arithmetic-heavy end: ten pions from 10 GeV, FP64
        {"name": "generate_10body_2p24", "path": "generate", "N": 10, "n": 1 << 24,
         "engine": "squares3", "prec": "fp64", "decay": "pions"},
        # the same multiplicity just above threshold in mixed precision, a
        # ragged count
        {"name": "generate_10body_threshold_mixed", "path": "generate", "N": 10,
         "n": (1 << 24) + 33, "engine": "squares3", "prec": "mixed", "decay": "threshold"},
        # a four-body decay on one of the Random123 engines
        {"name": "generate_4body_threefry_3e6", "path": "generate", "N": 4, "n": 3000007,
         "engine": "threefry", "prec": "fp64", "decay": "flat"},
        # a small accept-reject sample
        {"name": "unweight_3body_1e5", "path": "unweight", "N": 3, "n": 100000,
         "engine": "squares3", "prec": "fp64", "decay": "jpsikpi"},
        # the large production step: 2^27 events generated and unweighted
        {"name": "unweight_3body_2p27", "path": "unweight", "N": 3, "n": 1 << 27,
         "engine": "squares3", "prec": "fp64", "decay": "jpsikpi"},
        # a Dalitz model sampled from stored flat events
        {"name": "reweight_3body_1e7", "path": "reweight", "N": 3, "n": 10000000,
         "decay": "jpsikpi"},
        # one 2^24-event chunk of the Dalitz integral, FP64
        {"name": "average_3body_bw_2p24", "path": "average", "N": 3, "n": 1 << 24,
         "engine": "squares3", "prec": "fp64", "decay": "jpsikpi"},
        # a small integration request in mixed precision
        {"name": "average_5body_mixed_6e4", "path": "average", "N": 5, "n": 60001,
         "engine": "squares3", "prec": "mixed", "decay": "flat"},
        # per-event variables without the momenta
        {"name": "evaluate_3body_1e7", "path": "evaluate", "N": 3, "n": 10000001,
         "engine": "squares3", "decay": "jpsikpi"},
        # the Dalitz plot of a stored sample, 100 x 100 bins
        {"name": "histogram_3body_5e6", "path": "histogram", "N": 3, "n": 5000011,
         "decay": "jpsikpi", "bins": 100},
    ]


def draw(rng):
    path = rng.choice(["generate", "generate", "generate", "unweight", "unweight", "unweight",
                       "reweight", "average", "average", "evaluate", "histogram", "range"])
    # the counts of a generator service, and larger ones where the container
    # is filled or unweighted
    top = 7.0
    N = rng.randint(2, 12)
    if path in ("generate", "unweight"):
        top = math.log10((1 << 27) / max(N, 4))
    elif path in ("reweight", "histogram"):
        N = rng.choice([3, 3, 4, 5])
    elif path in ("average", "evaluate"):
        N = rng.randint(3, 8)
    elif path == "range":
        N = 3
    if rng.random() < 0.3 and path in ("generate", "unweight", "evaluate"):
        N = 3
    n = int(10 ** rng.uniform(3.0, top)) | 1
    case = {"path": path, "N": N, "n": n}
    if path == "range":
        return dict(case, decay="kaon", bins=rng.choice([10, 50, 100]))
    case["decay"] = "jpsikpi" if N == 3 else rng.choice(["flat", "flat", "pions"])
    if path in ("generate", "unweight", "average", "evaluate"):
        case["engine"] = rng.choice(["squares3"] * 6 + ["squares4", "philox", "philox_long",
                                                        "threefry", "threefry_long"])
    if path in ("generate", "unweight", "average"):
        case["prec"] = rng.choice(["fp64", "mixed"])
    if path == "histogram":
        case["bins"] = rng.choice([20, 50, 100])
    return case


def masses_of(case):
    """(mother mass, daughter masses) of a case."""
    N = case["N"]
    if case["decay"] == "jpsikpi":
        return M3, list(MASSES3)
    if case["decay"] == "kaon":
        return MK, [MPI] * 3
    if case["decay"] == "pions":
        return float(N), [0.13957] * N
    if case["decay"] == "threshold":
        return 10.0, [0.999 * 10.0 / N] * N
    m = [0.1 + 0.9 * ((7 * i + 3) % 11) / 11.0 for i in range(N)]
    return 1.7 * sum(m), m


def functors_of(case):
    """(kind, terms) of the functors an evaluate case writes."""
    N = case["N"]
    return [(capi.F_MASS2, (0, N - 1)), (capi.F_MASS2, (1, N - 1)), (capi.F_COS_HELICITY, (1, 2))]


def plot_of(case):
    """Axis limits of a histogram case: m^2(0, 1) and m^2(1, 2), or the range's m(0, 1)."""
    M, m = masses_of(case)
    rest = sum(m)
    if case["path"] == "range":
        return [m[0] + m[1]], [M - m[2]]
    return ([(m[0] + m[1]) ** 2, (m[1] + m[2]) ** 2],
            [(M - rest + m[0] + m[1]) ** 2, (M - rest + m[1] + m[2]) ** 2])


def average_terms(case):
    return BW3 if case["decay"] == "jpsikpi" else BW2


def work(case):
    N, n, path = case["N"], case["n"], case["path"]
    genbod = (3 * (3 * N - 4) + 3 * N + 15 * (N - 1) + 4 + 5 * N
              + sum(11 + 12 * (i + 1) for i in range(1, N))
              + sum(5 + 53 * (i + 1) for i in range(1, N - 1)))
    column = 4 if case.get("prec") == "mixed" else 8
    if path == "generate":
        return {"bytes": n * (4 * N * column + 8), "flops": n * (genbod + 39 * (N - 1))}
    if path == "unweight":
        return {"bytes": n * 4 * N * column, "flops": n * genbod}
    if path == "reweight":
        return {"bytes": n * 64 * N, "flops": n * (39 * (N - 1) + 60)}
    if path == "average":
        return {"bytes": 24, "flops": n * (genbod + 75)}
    if path == "evaluate":
        return {"bytes": n * 32, "flops": n * (genbod + 90)}
    if path == "histogram":
        return {"bytes": n * 96, "flops": n * (39 * (N - 1) + 30)}
    return {"bytes": 8 * (case["bins"] + 2), "flops": n * (genbod + 20)}


# ---- the framework's side -------------------------------------------------------

def padded(n):
    """Column stride of the containers: whole cache lines."""
    return (n + 63) // 64 * 64


def columns(rows, n, dtype=torch.float64):
    return torch.empty((rows, padded(n)), dtype=dtype, device=DEV)


def workspace(size):
    return torch.empty(int(size), dtype=torch.uint8, device=DEV)


def prepare(case, seed):
    lib = capi.lib()
    N, n, path = case["N"], case["n"], case["path"]
    M, masses = masses_of(case)
    s = {"path": path, "n": n, "seed": 159753 + 1000003 * seed,
         "prec": capi.MIXED if case.get("prec") == "mixed" else capi.FP64}
    if path == "range":
        s["decay"] = capi.make_range([M, 0.0, 0.0, 0.0], masses)
    else:
        s["decay"] = capi.make_decay(M, masses, case.get("engine", "squares3"))
    dtype = torch.float32 if s["prec"] == capi.MIXED else torch.float64
    if path == "generate":
        s["cols"] = columns(4 * N, n, dtype)
        s["weights"] = torch.empty(n, dtype=torch.float64, device=DEV)
    elif path == "unweight":
        s["cols"] = columns(4 * N, n, dtype)
        s["ws"] = workspace(lib.hpsp_generate_unweight_workspace_size(n))
        s["accepted"] = torch.zeros(1, dtype=torch.int64, device=DEV)
    elif path == "reweight":
        s["events"] = stored_events(case, seed)
        s["cols"] = columns(4 * N, n)
        s["ws"] = workspace(lib.hpsp_unweight_workspace_size(n))
        s["accepted"] = torch.zeros(1, dtype=torch.int64, device=DEV)
        s["functor"] = capi.make_functor(capi.F_BW_SUM, BW3)
    elif path == "average":
        s["functor"] = capi.make_functor(capi.F_BW_SUM, average_terms(case))
        s["ws"] = workspace(lib.hpsp_average_on_workspace_size(n))
        s["stats"] = torch.empty(3, dtype=torch.float64, device=DEV)
    elif path == "evaluate":
        s["functors"] = capi.functor_array([capi.make_functor(k, t) for k, t in functors_of(case)])
        s["out"] = columns(4, n)
    else:
        lower, upper = plot_of(case)
        s["histogram"] = capi.make_histogram([case["bins"]] * len(lower), lower, upper)
        s["contents"] = torch.empty(case["bins"] ** len(lower) + 2, dtype=torch.float64, device=DEV)
        if path == "histogram":
            s["events"] = stored_events(case, seed)
            s["axes"] = capi.functor_array([capi.make_functor(capi.F_MASS2, (0, 1)),
                                            capi.make_functor(capi.F_MASS2, (1, 2))])
        else:
            s["axes"] = capi.functor_array([capi.make_functor(capi.F_MASS, (0, 1))])
    return s


def run(s):
    lib, n, path = capi.lib(), s["n"], s["path"]
    dec, stream = ctypes.byref(s["decay"]), capi.stream_handle()
    if path == "generate":
        cols = s["cols"]
        capi.check(lib.hpsp_generate(dec, s["seed"], 0, n, s["prec"], capi.ptr(cols),
                                     cols.shape[1], int(cols.dtype == torch.float32), None,
                                     capi.ptr(s["weights"]), stream), "hpsp_generate")
        return cols[:, :n], s["weights"]
    if path == "unweight":
        cols, ws = s["cols"], s["ws"]
        fn = (lib.hpsp_generate_unweight_mixed if s["prec"] == capi.MIXED
              else lib.hpsp_generate_unweight)
        capi.check(fn(dec, s["seed"], 0, n, UW_SEED, capi.ptr(cols), cols.shape[1], None, None,
                      capi.ptr(ws), ws.numel(), capi.ptr(s["accepted"]), stream),
                   "hpsp_generate_unweight")
        return cols[:, :n], s["accepted"]
    if path == "reweight":
        cols, ws, events = s["cols"], s["ws"], s["events"]
        capi.check(lib.hpsp_unweight(dec, ctypes.byref(s["functor"]), -1.0, UW_SEED,
                                     capi.ptr(events), events.shape[1], n, None, capi.ptr(cols),
                                     cols.shape[1], None, None, capi.ptr(ws), ws.numel(),
                                     capi.ptr(s["accepted"]), stream), "hpsp_unweight")
        return cols[:, :n], s["accepted"]
    if path == "average":
        ws = s["ws"]
        capi.check(lib.hpsp_average_on(dec, ctypes.byref(s["functor"]), s["seed"], 0, n, s["prec"],
                                       capi.ptr(ws), ws.numel(), capi.ptr(s["stats"]), stream),
                   "hpsp_average_on")
        return s["stats"]
    if path == "evaluate":
        out, fs = s["out"], s["functors"]
        capi.check(lib.hpsp_evaluate(dec, fs, len(fs), s["seed"], 0, n, capi.ptr(out),
                                     out.shape[1], stream), "hpsp_evaluate")
        return out[:, :n]
    hist, contents = ctypes.byref(s["histogram"]), s["contents"]
    if path == "histogram":
        events = s["events"]
        capi.check(lib.hpsp_histogram_fill_events(hist, dec, s["axes"], capi.ptr(events),
                                                  events.shape[1], n, capi.HIST_WEIGHT_PHSP, None,
                                                  capi.ptr(contents), stream),
                   "hpsp_histogram_fill_events")
    else:
        capi.check(lib.hpsp_histogram_fill_range(hist, dec, s["seed"], s["axes"], 0, n,
                                                 capi.HIST_WEIGHT_GENERATION, capi.ptr(contents),
                                                 stream), "hpsp_histogram_fill_range")
    return contents


# ---- plain double precision restatement ------------------------------------------
# 64-bit words are int64 tensors (two's complement: products and sums wrap as
# unsigned ones do; logical shifts mask the sign).

CHUNK = 1 << 22
MASK32 = 0xFFFFFFFF


def i64(x):
    """A Python integer's low 64 bits as a signed value."""
    x &= (1 << 64) - 1
    return x - (1 << 64) if x >> 63 else x


def shr(x, k):
    return (x >> k) & ((1 << (64 - k)) - 1)


def rotl(x, k):
    return (x << k) | shr(x, 64 - k)


def mulhi(a, b):
    """High 64 bits of the unsigned product of a constant and a tensor."""
    a0, a1 = a & MASK32, (a >> 32) & MASK32
    b0, b1 = b & MASK32, shr(b, 32)
    # every partial product is below 2^64; carries through its halves
    p00, p01, p10, p11 = a0 * b0, a0 * b1, a1 * b0, a1 * b1
    mid = shr(p00, 32) + (p01 & MASK32) + (p10 & MASK32)
    return p11 + shr(p01, 32) + shr(p10, 32) + shr(mid, 32)


def keys(seed, count):
    """SplitMix64 draws from a seed, as Python integers."""
    out, full = [], (1 << 64) - 1
    x = seed & full
    for _ in range(count):
        x = (x + 0x9E3779B97F4A7C15) & full
        z = ((x ^ (x >> 30)) * 0xBF58476D1CE4E5B9) & full
        z = ((z ^ (z >> 27)) * 0x94D049BB133111EB) & full
        out.append(z ^ (z >> 31))
    return out


def squares(seed, counter, rounds):
    key = i64(keys(seed, 1)[0])
    y = key * counter
    z = y + key
    x = y * y + y
    x = rotl(x, 32)
    x = x * x + z
    x = rotl(x, 32)
    if rounds == 4:
        x = rotl(x * x + y, 32)
        return shr(x * x + z, 32)
    return shr(x * x + y, 32)


def philox(key, c):
    k = list(key)
    for r in range(7):
        if r:
            k[0] = i64(k[0] + 0x9E3779B97F4A7C15)
            if len(k) > 1:
                k[1] = i64(k[1] + 0xBB67AE8584CAA73B)
        if len(c) == 2:
            m = i64(0xD2B74407B1CE6E93)
            c = [mulhi(m, c[0]) ^ k[0] ^ c[1], m * c[0]]
        else:
            m0, m1 = i64(0xD2E7470EE14C6C93), i64(0xCA5A826395121157)
            c = [mulhi(m1, c[2]) ^ c[1] ^ k[0], m1 * c[2],
                 mulhi(m0, c[0]) ^ c[3] ^ k[1], m0 * c[0]]
    return c


def threefry(key, x):
    w = len(x)
    parity = 0x1BD11BDAA9FC1A22
    for k in key:
        parity ^= k & ((1 << 64) - 1)
    ks = [i64(k) for k in key] + [i64(parity)]
    rot2 = (16, 42, 12, 31, 16, 32, 24, 21)
    rot4 = ((14, 16), (52, 57), (23, 40), (5, 37), (25, 33), (46, 12), (58, 22), (32, 32))
    x = [x[i] + ks[i] for i in range(w)]
    for r in range(12):
        if w == 2:
            x[0] = x[0] + x[1]
            x[1] = rotl(x[1], rot2[r % 8]) ^ x[0]
        else:
            a, b = (1, 3) if r % 2 == 0 else (3, 1)
            x[0] = x[0] + x[a]
            x[a] = rotl(x[a], rot4[r % 8][0]) ^ x[0]
            x[2] = x[2] + x[b]
            x[b] = rotl(x[b], rot4[r % 8][1]) ^ x[2]
        if r % 4 == 3:
            i = (r + 1) // 4
            x = [x[j] + ks[(i + j) % (w + 1)] for j in range(w)]
            x[w - 1] = x[w - 1] + i
    return x


def uniforms(engine, seed, N, first, count):
    """The 3N - 4 uniforms of events first .. first + count - 1 (a column each)."""
    base = torch.arange(count, dtype=torch.int64, device=DEV) + (first + 3 * N)
    W = 3 * N - 4
    if engine == "minstd":
        a, m = 48271, (1 << 31) - 1
        x0 = (seed & MASK32) % m or 1
        lane = torch.ones(count + W, dtype=torch.int64, device=DEV)
        have = 1
        while have < count + W:  # powers of a by doubling
            take = min(have, count + W - have)
            lane[have:have + take] = lane[:take] * pow(a, have, m) % m
            have += take
        x = lane * (x0 * pow(a, first + 3 * N + 1, m) % m) % m
        return [(x[j:j + count] - 1).double() / 2147483646.0 for j in range(W)]
    if engine in ("squares3", "squares4"):
        rounds = 3 if engine == "squares3" else 4
        return [squares(seed, base + j, rounds).double() * 2.0 ** -32 for j in range(W)]
    arity = 4 if engine.endswith("long") else 2
    words = []
    for b in range((W + arity - 1) // arity):
        ctr = [base + 1 + b] + [torch.zeros_like(base) for _ in range(arity - 1)]
        if engine.startswith("philox"):
            words += philox([i64(k) for k in keys(seed, arity // 2)], ctr)
        else:
            words += threefry(keys(seed, arity), ctr)
    return [(shr(w, 32).double() * 2.0 ** 32 + (w & MASK32).double()) * 2.0 ** -64
            for w in words[:W]]


def pdk(a, b, c):
    x = (a - b - c) * (a + b + c) * (a - b + c) * (a + b - c)
    return torch.sqrt(x) / (2 * a)


def max_weight(M, masses):
    ecm = M - sum(masses)
    emmax, emmin, w = ecm + masses[0], 0.0, 1.0
    for i in range(1, len(masses)):
        emmin += masses[i - 1]
        emmax += masses[i]
        x = ((emmax - emmin - masses[i]) * (emmax + emmin + masses[i])
             * (emmax - emmin + masses[i]) * (emmax + emmin - masses[i]))
        w *= math.sqrt(x) / (2 * emmax)
    return 1.0 / w


def genbod(M, masses, u):
    """Momenta (N lists of E, px, py, pz) and generation weights from uniforms."""
    N = len(masses)
    mass_u = torch.stack(u[:N - 2]).sort(dim=0).values if N > 2 else []
    ecm = M
    for m in masses:
        ecm -= m
    rno = [torch.zeros_like(u[0])] + list(mass_u) + [torch.ones_like(u[0])]
    inv, total = [], 0.0
    for i in range(N):
        total += masses[i]
        inv.append(rno[i] * ecm + total)
    pd = [pdk(inv[i + 1], inv[i], masses[i + 1]) for i in range(N - 1)]
    wt = torch.full_like(u[0], max_weight(M, masses))
    for q in pd:
        wt = wt * q
    zero = torch.zeros_like(u[0])
    p = [[torch.sqrt(pd[0] ** 2 + masses[0] ** 2), zero, pd[0], zero]]
    for i in range(1, N):
        p.append([torch.sqrt(pd[i - 1] ** 2 + masses[i] ** 2), zero, -pd[i - 1], zero])
        cz = 2 * u[N - 2 + 2 * (i - 1)] - 1
        sz = torch.sqrt((1 - cz) * (1 + cz))
        angle = 2 * math.pi * u[N - 2 + 2 * (i - 1) + 1]
        cy, sy = torch.cos(angle), torch.sin(angle)
        for v in p:
            x, y = cz * v[1] - sz * v[2], sz * v[1] + cz * v[2]
            v[1], v[2], v[3] = cy * x - sy * v[3], y, sy * x + cy * v[3]
        if i < N - 1:
            g, gb = torch.sqrt(pd[i] ** 2 + inv[i] ** 2) / inv[i], pd[i] / inv[i]
            for v in p:
                v[0], v[2] = g * v[0] + gb * v[2], gb * v[0] + g * v[2]
    return p, wt


def generated(case, seed, first, count):
    M, masses = masses_of(case)
    engine = "minstd" if case["path"] == "range" else case["engine"]
    return genbod(M, masses, uniforms(engine, 159753 + 1000003 * seed, case["N"], first, count))


def stored_events(case, seed):
    """Momentum columns of n flat phase-space events, as a container holds them."""
    M, masses = masses_of(case)
    n = case["n"]
    cols = columns(4 * case["N"], n)
    gen = torch.Generator(device=DEV).manual_seed(seed)
    for b in range(0, n, CHUNK):
        e = min(n, b + CHUNK)
        u = torch.rand((3 * case["N"] - 4, e - b), generator=gen, dtype=torch.float64, device=DEV)
        p, _ = genbod(M, masses, list(u))
        for i, v in enumerate(p):
            for c in range(4):
                cols[4 * i + c, b:e] = v[c]
    cols[:, n:] = 0.0
    return cols


def dot(a, b):
    return a[0] * b[0] - a[1] * b[1] - a[2] * b[2] - a[3] * b[3]


def add(a, b):
    return [x + y for x, y in zip(a, b)]


def phsp_weight(M, masses, p):
    total = p[0]
    w = torch.full_like(p[0][0], max_weight(M, masses))
    before = torch.sqrt(dot(total, total))
    for i in range(1, len(masses)):
        total = add(total, p[i])
        now = torch.sqrt(dot(total, total))
        w = w * pdk(now, masses[i], before)
        before = now
    return w


def breit_wigners(terms, p):
    re, im = 0.0, 0.0
    for m, g, cr, ci, a, b in terms:
        v = add(p[a], p[b])
        dr, di = m * m - dot(v, v), -(m * g)
        den = dr * dr + di * di
        br, bi = dr / den, -di / den
        re, im = re + cr * br - ci * bi, im + cr * bi + ci * br
    return re * re + im * im


def cos_helicity(p, a, b):
    P = p[0]
    for v in p[1:]:
        P = add(P, v)
    d, q = p[a], add(p[a], p[b])
    num = dot(P, d) * dot(q, q) - dot(P, q) * dot(q, d)
    den = ((dot(P, q) ** 2 - dot(q, q) * dot(P, P)) * (dot(q, d) ** 2 - dot(q, q) * dot(d, d)))
    return num / torch.sqrt(den)


def partition(cols, accept):
    """Accepted events first, both parts in their order; the column buffer is reused."""
    order = torch.cat([accept.nonzero().squeeze(1), (~accept).nonzero().squeeze(1)])
    for i in range(cols.shape[0]):
        cols[i] = cols[i][order]
    return cols


def chunks(n):
    return [(b, min(n, b + CHUNK)) for b in range(0, n, CHUNK)]


def rows_of(cols, b, e):
    return [[cols[4 * i + c, b:e] for c in range(4)] for i in range(cols.shape[0] // 4)]


def accept_uniforms(b, e):
    k = torch.arange(b, e, dtype=torch.int64, device=DEV)
    return squares(UW_SEED, k, 3).double() * 2.0 ** -32


def exact(case, seed):
    M, masses = masses_of(case)
    N, n, path = case["N"], case["n"], case["path"]
    if path in ("generate", "unweight"):
        cols = torch.empty((4 * N, n), dtype=torch.float64, device=DEV)
        wts = torch.empty(n, dtype=torch.float64, device=DEV)
        accept = torch.empty(n, dtype=torch.bool, device=DEV)
        top = max_weight(M, masses)
        for b, e in chunks(n):
            p, wt = generated(case, seed, b, e - b)
            for i, v in enumerate(p):
                for c in range(4):
                    cols[4 * i + c, b:e] = v[c]
            wts[b:e] = wt
            if path == "unweight":
                # the mixed container's weights are the generation weights
                w = wt if case["prec"] == "mixed" else phsp_weight(M, masses, p)
                accept[b:e] = w / top > accept_uniforms(b, e)
        return (cols, wts) if path == "generate" else (partition(cols, accept), None)
    if path == "reweight":
        cols = stored_events(case, seed)[:, :n].contiguous()
        value = torch.empty(n, dtype=torch.float64, device=DEV)
        for b, e in chunks(n):
            p = rows_of(cols, b, e)
            value[b:e] = phsp_weight(M, masses, p) * breit_wigners(BW3, p)
        top = value.max()
        accept = torch.empty(n, dtype=torch.bool, device=DEV)
        for b, e in chunks(n):
            accept[b:e] = value[b:e] / top > accept_uniforms(b, e)
        return partition(cols, accept), None
    if path == "average":
        f = torch.empty(n, dtype=torch.float64, device=DEV)
        w = torch.empty(n, dtype=torch.float64, device=DEV)
        for b, e in chunks(n):
            p, wt = generated(case, seed, b, e - b)
            f[b:e], w[b:e] = breit_wigners(average_terms(case), p), wt
        total = w.sum()
        mean = (w * f).sum() / total
        return torch.stack([total, mean, (w * (f - mean) ** 2).sum()])
    if path == "evaluate":
        out = torch.empty((4, n), dtype=torch.float64, device=DEV)
        for b, e in chunks(n):
            p, wt = generated(case, seed, b, e - b)
            out[0, b:e] = wt
            for j, (kind, t) in enumerate(functors_of(case)):
                if kind == capi.F_MASS2:
                    v = add(p[t[0]], p[t[1]])
                    out[1 + j, b:e] = dot(v, v)
                else:
                    out[1 + j, b:e] = cos_helicity(p, *t)
        return out
    lower, upper = plot_of(case)
    g = case["bins"]
    contents = torch.zeros(g ** len(lower) + 2, dtype=torch.float64, device=DEV)
    events = stored_events(case, seed) if path == "histogram" else None
    for b, e in chunks(n):
        if path == "histogram":
            p = rows_of(events, b, e)
            w = phsp_weight(M, masses, p)
            s, t = add(p[0], p[1]), add(p[1], p[2])
            axes = [dot(s, s), dot(t, t)]
        else:
            p, w = generated(case, seed, b, e - b)
            s = add(p[0], p[1])
            axes = [torch.sqrt(dot(s, s))]
        # every value lies inside the axes but for rounding at their ends
        key = torch.zeros(e - b, dtype=torch.int64, device=DEV)
        for x, lo, hi in zip(axes, lower, upper):
            key = key * g + ((x - lo) * g / (hi - lo)).long().clamp(0, g)
        contents.index_add_(0, key, w)
    return contents
