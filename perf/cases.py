"""The work that users of muca_amd have it do, as cases that can be timed.

Five kinds of case, each one pass through the public entry points:

  loop     the host weight loop of the drop-in `multigpu_weight`: Context,
           init_lattice, compute_state, weight_iteration
  batch    the device weight loop: Batch, init, iterate (graph replay)
  produce  a production run with reweighting, as the drop-in `produce_gpu`
           does it: a thermalisation launch, a production launch, reweight
  train    one epoch of the surrogate's training: set_data, train
  predict  ln W outputs of the surrogate for every D of one lattice
  gradient the loss and gradient over a whole corpus, as training ends with

Every pass starts from the same state (lattices drawn anew from the case's
seed), so that passes can be repeated and cost the same.
"""
import math

import numpy as np

import muca_amd as M
from muca_amd import surrogate as S

DELTAS = np.round(np.linspace(1.90, 2.00, 11), 4)


def listed():
    return [
        # the smallest call: a small lattice with few walkers in the host loop,
        # where launches, copies and the latency of one chain are all there is
        dict(name="loop_L16_W16", kind="loop", L=16, walkers=16, iters=10, nup=1, recursive=False,
             seeded=False, fp64=False, T=0.5),
        # the headline workload: plain weight iterations, L = 72, 4096 walkers
        dict(name="batch_L72_W4096", kind="batch", Ls="72", walkers=4096, iters=20, nup=1,
             recursive=True, seeded=False, T=0.5),
        # the same engine at the headline's larger lattice, seeded weights and
        # a sweep of NUPDATES (lattices too large for LDS)
        dict(name="batch_L128_W4096", kind="batch", Ls="128", walkers=4096, iters=8, nup=16384,
             recursive=False, seeded=True, T=0.55),
        # 96 weight problems of a (L, T, Delta) grid in one batch
        dict(name="batch_96", kind="batch", Ls=",".join(str(L) for L in (32, 48, 64, 72, 96, 128)
                                                        for _ in range(16)),
             walkers=4096, iters=4, nup=1, recursive=True, seeded=False, T=0.5),
        # the drop-in program's default walker count (one per hardware thread)
        dict(name="loop_L72_W524288", kind="loop", L=72, walkers=524288, iters=3, nup=1,
             recursive=False, seeded=False, fp64=False, T=0.5),
        # an even lattice size that is no multiple of 8, ragged walker count
        dict(name="loop_L100_W4100", kind="loop", L=100, walkers=4100, iters=3, nup=1,
             recursive=False, seeded=True, fp64=False, T=0.6),
        # an odd lattice size
        dict(name="loop_L45_W2000", kind="loop", L=45, walkers=2000, iters=3, nup=2025,
             recursive=True, seeded=True, fp64=False, T=0.6),
        # production at the headline's size with joint H(D, M), ten blocks
        dict(name="produce_L72_W4096", kind="produce", L=72, walkers=4096, therm=5184, nup=10368,
             blocks=10, moments=False, T=0.55),
        # large production with exact per-D moments, ten blocks
        dict(name="produce_L256_W16384", kind="produce", L=256, walkers=16384, therm=65536,
             nup=65536, blocks=10, moments=True, T=0.5),
        # the drop-in production program's defaults: one walker per hardware
        # thread, one joint histogram
        dict(name="produce_L64_W524288", kind="produce", L=64, walkers=524288, therm=4096,
             nup=4096, blocks=1, moments=False, T=0.5),
        # one epoch over the shipped corpus at the default minibatch
        dict(name="train_4096", kind="train", samples=49152, batch=4096),
        # the seed of one L = 128 weight problem
        dict(name="predict_L128", kind="predict", L=128, T=0.5),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _draw_L(rng, lo, hi):
    L = _log_int(rng, lo, hi)
    u = rng.random()
    if u < 0.5:
        return max(lo, min(hi, 8 * round(L / 8)))
    if u < 0.8:
        return max(lo, min(hi, 2 * round(L / 2)))
    return L


# most attempts a drawn case makes (about a tenth of a second of the largest
# listed case's rate, less for odd L, which runs on one lane per walker)
_ATTEMPTS, _ATTEMPTS_ODD, _STEPS = 2.0e9, 2.5e8, 40000


def _fit(L, walkers, iters, nup):
    """Walkers, iterations and NUPDATES cut until the case is small enough."""
    most = _ATTEMPTS_ODD if L % 2 else _ATTEMPTS
    N = L * L
    while iters > 1 and iters * (N + nup) > _STEPS:
        iters -= 1
    if iters * (N + nup) > _STEPS:
        nup = max(1, _STEPS - N)
    walkers = max(1, min(walkers, int(most / (iters * (N + nup)))))
    return walkers, iters, nup


def draw(rng):
    T = rng.choice((0.5, 0.55, 0.6, 0.7, 0.8))
    kind = rng.choice(("loop", "loop", "loop", "batch", "batch", "produce", "produce", "produce",
                       "train", "predict", "gradient"))
    if kind == "loop":
        L = _draw_L(rng, 8, 128)
        seeded = rng.random() < 0.5
        nup = rng.choice((1, L * L // 2 + 3, L * L, 2 * L * L + 1)) if seeded else 1
        walkers, iters, nup = _fit(L, _log_int(rng, 16, 262144), rng.randint(1, 6), nup)
        return dict(kind="loop", L=L, walkers=walkers, iters=iters, nup=nup,
                    recursive=rng.random() < 0.5, seeded=seeded, fp64=rng.random() < 0.2, T=T)
    if kind == "batch":
        n = rng.choice((1, 1, 2, 4, 8, 16))
        step = 8 if rng.random() < 0.7 else 2
        Ls = [max(8, min(128, step * round(_log_int(rng, 16, 128) / step))) for _ in range(n)]
        seeded = rng.random() < 0.5
        nup = rng.choice((1, 500, 4096)) if seeded else 1
        walkers, iters, nup = _fit(max(Ls), _log_int(rng, 32, 8192), rng.randint(1, 20), nup)
        return dict(kind="batch", Ls=",".join(map(str, Ls)), walkers=walkers, iters=iters, nup=nup,
                    recursive=rng.random() < 0.5, seeded=seeded, T=T)
    if kind == "produce":
        moments = rng.random() < 0.5
        L = _draw_L(rng, 8, 160 if moments else 72)
        N = L * L
        walkers, _, nup = _fit(L, _log_int(rng, 64, 131072), 1, rng.choice((N, 2 * N + 5, 4 * N)))
        return dict(kind="produce", L=L, walkers=walkers, therm=N, nup=nup,
                    blocks=min(walkers, rng.choice((1, 4, 10))), moments=moments, T=T)
    if kind == "predict":
        return dict(kind="predict", L=_log_int(rng, 16, 256), T=T)
    samples = _log_int(rng, 1000, 60000)
    if kind == "gradient":
        return dict(kind="gradient", samples=samples)
    return dict(kind="train", samples=samples,
                batch=min(rng.choice((1024, 2048, 4096, 8192)), samples // 64 * 64))


# ---- inputs ---------------------------------------------------------------

def _curve(L, T, rng):
    """ln W(D) of an (L, T) problem from the shipped converged curves (the
    curve of the nearest T and largest L, scaled by N), with a smooth error of
    the size a surrogate's seed has."""
    d = np.load(S.CORPUS_PATH)
    keys = [(int(k.split("_")[0][1:]), float(k.split("_T")[1]), k) for k in d.files]
    k = min(keys, key=lambda q: (abs(q[1] - T), q[0] != L, -q[0]))[2]
    f = d[k]
    n0, N = len(f) - 1, L * L
    m = np.arange(N + 1) / N
    lnw = np.interp(m * n0, np.arange(n0 + 1), f / n0) * N
    lnw = lnw + 0.3 * np.sin(2 * np.pi * (rng.uniform(1, 3) * m + rng.uniform()))
    return lnw - lnw[0]


def _chain_inputs(case, seed):
    rng = np.random.default_rng(seed)
    key = int(rng.integers(1, 1 << 30))
    return rng, key


def _samples(case, seed):
    """Shuffled corpus samples (features, targets, weights) and start parameters."""
    rng = np.random.default_rng(seed)
    X, t, w = S.corpus(S.load_corpus())
    at = rng.permutation(len(X))
    n = case["samples"]
    at = np.resize(at, n)
    t = t[at] + rng.normal(0, 1e-3, n).astype(np.float32)
    return X[at], t.astype(np.float32), w[at], S.init_params(seed % (1 << 31))


def prepare(case, seed):
    kind = case["kind"]
    st = dict(case=case)
    if kind == "loop":
        rng, st["seed"] = _chain_inputs(case, seed)
        st["ctx"] = M.Context(case["L"], case["walkers"], beta=1.0 / case["T"],
                              precision=M.FP64 if case["fp64"] else M.REF32)
        st["lnw"] = _curve(case["L"], case["T"], rng) if case["seeded"] else None
    elif kind == "batch":
        rng, key = _chain_inputs(case, seed)
        Ls = [int(x) for x in case["Ls"].split(",")]
        st["batch"] = M.Batch([dict(L=L, walkers=case["walkers"], seed=key + i,
                                    beta=1.0 / case["T"], recursion=case["recursive"],
                                    init_nup=case["nup"]) for i, L in enumerate(Ls)])
        st["lnw"] = [_curve(L, case["T"], rng) for L in Ls] if case["seeded"] else None
    elif kind == "produce":
        rng, st["seed"] = _chain_inputs(case, seed)
        st["ctx"] = M.Context(case["L"], case["walkers"], beta=1.0 / case["T"], precision=M.FP64,
                              keying=M.KEYING_PRODUCE, joint_blocks=case["blocks"],
                              observables=M.OBS_MOMENTS if case["moments"] else M.OBS_JOINT)
        st["lnw"] = _curve(case["L"], case["T"], rng)
    elif kind == "predict":
        st["net"] = M.Mlp()
        st["net"].set_params(S.init_params(seed % (1 << 31)))
        st["x"] = _features(case, seed)
    else:
        st["x"], st["t"], st["w"], st["p"] = _samples(case, seed)
        st["net"] = M.Mlp()
        st["net"].set_params(st["p"])
    return st


def _features(case, seed):
    N = case["L"] ** 2
    delta = np.random.default_rng(seed).uniform(S.DELTAS[0], S.DELTAS[-1])
    return S.features(np.arange(N + 1) / N, case["L"], 1.0 / case["T"], delta)


# ---- one pass -------------------------------------------------------------

def run(st):
    case = st["case"]
    kind = case["kind"]
    if kind == "loop":
        ctx = st["ctx"]
        ctx.init_lattice(mm=0, gpu=0, seed=st["seed"], stratified=case["seeded"])
        ctx.compute_state()
        lnw, recs = M.weight_iteration(ctx, case["iters"], seed=st["seed"], init_nup=case["nup"],
                                       recursion=case["recursive"], lnw_init=st["lnw"])
        E, D, Mg = ctx.get_state()
        return dict(lnw=lnw, hist=np.stack([r["hist"] for r in recs]).astype(np.int64),
                    E=E, D=D, M=Mg)
    if kind == "batch":
        b = st["batch"]
        b.init(0, stratified=case["seeded"])
        if st["lnw"] is not None:
            for i, lw in enumerate(st["lnw"]):
                b.set_log_weight(i, lw)
        b.iterate(case["iters"])
        state = [b.get_state(i) for i in range(b.n)]
        return dict(lnw=np.concatenate([b.get_log_weight(i) for i in range(b.n)]),
                    hist=np.concatenate([b.get_hist(i) for i in range(b.n)]).astype(np.int64),
                    E=np.concatenate([s[0] for s in state]),
                    D=np.concatenate([s[1] for s in state]),
                    M=np.concatenate([s[2] for s in state]))
    if kind == "produce":
        ctx = st["ctx"]
        ctx.init_lattice(mm=0, gpu=0, seed=st["seed"], stratified=True)
        ctx.compute_state()
        ctx.set_log_weight(st["lnw"])
        ctx.run(0, st["seed"] + 1000, case["therm"], 0, want_hist=False)
        hist, _ = ctx.run(1, st["seed"] + 2000, 0, case["nup"])
        absM, chi, binder = ctx.reweight(DELTAS)
        E, D, Mg = ctx.get_state()
        return dict(hist=hist.astype(np.int64), absM=absM, chi=chi, binder=binder, E=E, D=D, M=Mg)
    if kind == "predict":
        return st["net"].predict(st["x"])
    if kind == "gradient":
        g, loss = st["net"].gradient(st["x"], st["t"])
        return dict(grad=g, loss=loss)
    net = st["net"]
    net.set_params(st["p"])
    net.set_data(st["x"], st["t"], st["w"])
    loss, _ = net.train(max(1, case["samples"] // case["batch"]), case["batch"], 2e-3, 1.9e-3)
    return dict(params=net.get_params(), loss=loss)


# ---- the work of a pass ---------------------------------------------------

_PARAMS = 4 * 128 + 128 + 2 * (128 * 128 + 128) + 128 + 1
# per attempt: half a Philox4x32-7 block (two keys, four attempts a block:
# 7 rounds of two products, four xors and two key additions) and the
# proposal, energy and acceptance
_OPS = 28 + 12


def work(case):
    kind = case["kind"]
    if kind in ("loop", "batch"):
        Ls = [case["L"]] if kind == "loop" else [int(x) for x in case["Ls"].split(",")]
        W, n, nup = case["walkers"], case["iters"], case["nup"]
        b = f = 0
        for L in Ls:
            N = L * L
            # the lattice written once at the start, read and written by each launch
            b += N * W * (1 + 2 * n) + 12 * W * (1 + 2 * n) + 20 * (N + 1) * n
            f += n * W * (N + nup) * _OPS
        return dict(bytes=b, flops=f)
    if kind == "produce":
        N, W = case["L"] ** 2, case["walkers"]
        acc = (8 * (N + 1) if case["moments"] else (N + 1) * (N + 2) // 2) * 8 * case["blocks"]
        return dict(bytes=5 * N * W + 5 * 12 * W + 2 * acc,
                    flops=W * (case["therm"] + case["nup"]) * _OPS)
    if kind == "predict":
        n = case["L"] ** 2 + 1
        return dict(bytes=20 * n + 2 * _PARAMS, flops=2 * n * _PARAMS)
    n = case["samples"]
    if kind == "gradient":
        return dict(bytes=20 * n + 6 * _PARAMS, flops=6 * n * _PARAMS)
    steps = max(1, n // case["batch"])
    return dict(bytes=24 * n + steps * 24 * _PARAMS, flops=6 * steps * case["batch"] * _PARAMS)


# ---- the same in plain numpy ----------------------------------------------

_M0, _M1 = np.uint64(0xD2511F53), np.uint64(0xCD9E8D57)
_LOW, _S32 = np.uint64(0xFFFFFFFF), np.uint64(32)


def _philox(c, k):
    """Philox4x32-7 (Salmon et al., SC'11) over arrays: c of four words, k of two."""
    c = [np.asarray(x, np.uint64) for x in c]
    k0, k1 = (np.asarray(x, np.uint64) for x in k)
    for _ in range(7):
        p0, p1 = _M0 * c[0], _M1 * c[2]
        c = [(p1 >> _S32) ^ c[1] ^ k0, p1 & _LOW, (p0 >> _S32) ^ c[3] ^ k1, p0 & _LOW]
        k0 = (k0 + np.uint64(0x9E3779B9)) & _LOW
        k1 = (k1 + np.uint64(0xBB67AE85)) & _LOW
    return np.stack(np.broadcast_arrays(*c))


def _uniform(r):
    return (np.uint64(1) | (r >> np.uint64(8))).astype(np.float64) * 2.0 ** -24


class _Chains:
    """W Metropolis chains on an L x L lattice in the order of sites and with
    the random numbers that the programs document."""

    def __init__(self, L, W, seed, produce, stratified, beta):
        self.L, self.N, self.W, self.produce, self.beta = L, L * L, W, produce, beta
        N = self.N
        w = np.arange(W, dtype=np.uint64)
        self.w = w
        s = np.empty((N, W), np.int64)
        p = (np.arange(W) + 0.5) / W
        for blk in range((N + 3) // 4):
            if produce:
                r = _philox((0, seed, blk + 1, 0xBADCAFE3), (10 * w, 0xdecafbad))
            else:
                r = _philox((blk + 1, seed, 0xBADCAB1E, 0xBADC0DED), (10 * w, 0xdecafbad))
            u = _uniform(r)
            v = (np.where(u < p, np.where(u < 0.5 * p, -1, 1), 0) if stratified
                 else (u < 1 / 3.0).astype(np.int64) + (u < 2 / 3.0) - 1)
            s[4 * blk:min(4 * blk + 4, N)] = v[:N - 4 * blk]
        self.s = s
        a = s.reshape(L, L, W)
        self.E = -(a * (np.roll(a, 1, 0) + np.roll(a, 1, 1))).sum((0, 1))
        self.D = (a * a).sum((0, 1))
        self.M = a.sum((0, 1))
        i = np.arange(N)
        half = N // 2
        self.order = np.where((i // half) % 2 == 0, (2 * i) % N, (2 * i + 1) % N)

    def go(self, n, c0, it, seed, lnw, T, record):
        """n attempts per walker; returns the next block counter."""
        L, N, w, s = self.L, self.N, self.w, self.s
        k1 = (w if self.produce else 2 * w, 0xdecafbad)
        k3 = (w + 40000, 0xdecafead) if self.produce else (2 * w + 50000, 0x11cafead)
        lnw = lnw.astype(T)
        for i in range(n):
            if i % 4 == 0:
                c0 += 1
                lg = np.log(_uniform(_philox((c0, seed, it, 0xBADC0DED), k1))).astype(np.float32)
                r3 = _philox((c0, seed, it, 0xBADC0DED), k3)
            at = self.order[i % N]
            x, y = at % L, at // L
            old = s[at].copy()
            nb = (s[y * L + (x + 1) % L] + s[y * L + (x - 1) % L] + s[(y + 1) % L * L + x] +
                  s[(y - 1) % L * L + x])
            new = old + np.where(r3[i % 4] < 0x80000000, 1, -1)
            new = np.where(new == 2, -1, np.where(new == -2, 1, new))
            dE = -(new - old) * nb
            dD = new * new - old * old
            diff = ((-dE.astype(np.float64) * self.beta).astype(T) + lnw[self.D + dD]) - lnw[self.D]
            ok = lg[i % 4].astype(T) < diff
            s[at] = np.where(ok, new, old)
            self.E += np.where(ok, dE, 0)
            self.D += np.where(ok, dD, 0)
            self.M += np.where(ok, new - old, 0)
            if record is not None:
                record(self)
        return c0


def _exact_loop(case, seed):
    rng, key = _chain_inputs(case, seed)
    L, W = case["L"], case["walkers"]
    N = L * L
    T = np.float64 if case["fp64"] else np.float32
    lnw = _curve(L, case["T"], rng) if case["seeded"] else np.zeros(N + 1)
    c = _Chains(L, W, key, False, case["seeded"], 1.0 / case["T"])
    p_acc, width, nup = np.zeros(N + 1), 10, case["nup"]
    for it in range(case["iters"]):
        if width == N:
            nup = int((nup + 1) * 1.01)
        h = np.zeros(N + 1, np.int64)

        def record(q):
            np.add.at(h, q.D, 1)

        c0 = c.go(N, 0, it, key, lnw, T, None)
        c.go(nup, c0, it, key, lnw, T, record)
        at = np.nonzero(h > 1)[0]
        start, end = (int(at[0]), int(at[-1])) if len(at) else (0, 0)
        width = max(width, end - start)
        hp = h[h > 0] / h.sum()
        if width == N and (hp * np.log(hp * len(hp))).sum() < 1e-4:
            break
        if case["recursive"]:
            old = lnw.copy()
            for i in range(start, end):
                if h[i] and h[i + 1]:
                    q = float(h[i] * h[i + 1]) / float(h[i] + h[i + 1])
                    lnw[i + 1] = lnw[i] + (old[i + 1] - old[i] +
                                           q / (q + p_acc[i]) * math.log(h[i] / h[i + 1]))
                    p_acc[i] += q
        else:
            lnw = lnw - np.where(h > 1, np.log(np.maximum(h, 1)), 0.0)
        lnw = lnw - lnw[0]
    return dict(lnw=lnw, hist=None, E=None, D=None, M=None)


def _exact_produce(case, seed):
    rng, key = _chain_inputs(case, seed)
    L, W, B, beta = case["L"], case["walkers"], case["blocks"], 1.0 / case["T"]
    N = L * L
    lnw = _curve(L, case["T"], rng)
    c = _Chains(L, W, key, True, True, beta)
    c.go(case["therm"], 0, 0, key + 1000, lnw, np.float64, None)
    block = np.arange(W) // ((W + B - 1) // B)
    S_ = np.zeros((4, B, N + 1))

    def record(q):
        m = np.minimum(np.abs(q.M), q.D).astype(np.float64)
        for k, v in enumerate((np.ones(W), m, m * m, m ** 4)):
            np.add.at(S_[k], (block, q.D), v)

    c.go(case["nup"], 0, 1, key + 2000, lnw, np.float64, record)
    out = np.empty((3, len(DELTAS), B))
    for i, delta in enumerate(DELTAS):
        e = -beta * delta * np.arange(N + 1) - lnw
        for b in range(B):
            seen = S_[0, b] > 0
            z = np.where(seen, np.exp(np.minimum(e - e[seen].max(), 0)), 0) if seen.any() else e * 0
            with np.errstate(invalid="ignore", divide="ignore"):
                m1, m2, m4 = ((z * S_[k, b]).sum() / (z * S_[0, b]).sum() for k in (1, 2, 3))
                out[:, i, b] = m1, (m2 - m1 * m1) * beta / N, 1 - m4 / (3 * m2 * m2)
    return dict(hist=None, absM=out[0], chi=out[1], binder=out[2], E=None, D=None, M=None)


def _net(p):
    """The packed parameters as float64 arrays W1, b1, W2, b2, W3, b3, w4, b4."""
    at, out = 0, []
    for shape in ((128, 4), (128,), (128, 128), (128,), (128, 128), (128,), (128,), (1,)):
        n = int(np.prod(shape))
        out.append(p[at:at + n].astype(np.float64).reshape(shape))
        at += n
    return out


def _forward(q, x):
    W1, b1, W2, b2, W3, b3, w4, b4 = q
    sig = lambda z: 1 / (1 + np.exp(-z))  # noqa: E731
    z1 = x @ W1.T + b1
    a1 = z1 * sig(z1)
    z2 = a1 @ W2.T + b2
    a2 = z2 * sig(z2)
    z3 = a2 @ W3.T + b3
    a3 = z3 * sig(z3)
    y = a3 @ w4 + b4[0]

    def back(dy):
        d = lambda z: sig(z) * (1 + z * (1 - sig(z)))  # noqa: E731
        dz3 = dy[:, None] * w4 * d(z3)
        dz2 = (dz3 @ W3) * d(z2)
        dz1 = (dz2 @ W2) * d(z1)
        g = (dz1.T @ x, dz1.sum(0), dz2.T @ a1, dz2.sum(0), dz3.T @ a2, dz3.sum(0), a3.T @ dy,
             dy.sum(keepdims=True))
        return np.concatenate([v.ravel() for v in g])

    return y, back


def _exact_train(case, seed):
    x, t, w, p = _samples(case, seed)
    B = case["batch"]
    steps = max(1, case["samples"] // B)
    p = p.astype(np.float64)
    m, v = np.zeros_like(p), np.zeros_like(p)
    for s in range(steps):
        at = slice(s % (case["samples"] // B) * B, s % (case["samples"] // B) * B + B)
        lr = 1.9e-3 + 0.5 * (2e-3 - 1.9e-3) * (1 + math.cos(math.pi * s / steps))
        y, back = _forward(_net(p), x[at].astype(np.float64))
        d = y - t[at]
        g = back(2.0 / B * w[at] * d)
        m = 0.9 * m + 0.1 * g
        v = 0.999 * v + 0.001 * g * g
        p = p - lr * (m / (1 - 0.9 ** (s + 1))) / (np.sqrt(v / (1 - 0.999 ** (s + 1))) + 1e-8)
    return dict(params=p, loss=float((w[at] * d * d).sum() / B))


def exact(case, seed):
    kind = case["kind"]
    if kind in ("loop", "produce"):
        n = (case["iters"] * (case["L"] ** 2 + case["nup"]) if kind == "loop"
             else case["therm"] + case["nup"])
        if n * (1.5e-4 + 2e-7 * case["walkers"]) > 16:   # seconds
            return None
        return _exact_loop(case, seed) if kind == "loop" else _exact_produce(case, seed)
    if kind == "batch":
        return None
    if kind == "predict":
        return _forward(_net(S.init_params(seed % (1 << 31))),
                        _features(case, seed).astype(np.float64))[0]
    if kind == "gradient":
        x, t, _, p = _samples(case, seed)
        y, back = _forward(_net(p), x.astype(np.float64))
        d = y - t
        return dict(grad=back(2.0 / len(t) * d), loss=float((d * d).mean()))
    return _exact_train(case, seed)
