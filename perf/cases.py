"""Workloads of the solver and of the warm-start network, through the Python entry points.

A case is a dict of plain values.  ``prepare`` builds what a program holds before the call (an uploaded
``Solver`` or ``Batch``, a network and its data), ``run`` is one pass as such a program makes it, ``exact`` the
same pass in plain torch / numpy at 64 bits and ``work`` its arithmetic and the bytes of its inputs and outputs.

Kinds:
  solver   one instance at its default launch settings: fields in, n_rt round trips, fields and power history
           out (what the cuOPO executable does with each chunk of round trips)
  noalloc  the same on the caller's device buffers (opo_run_noalloc)
  batch    a sweep of instances in one tuned batch, round trips with or without the steady-state test, then
           every instance's fields and power (what the sweep and data-set drivers do)
  fit      one epoch of the warm-start network's training on minibatches
  predict  the network's outputs for a set of sweep points
"""
import ctypes as C
import math

import numpy as np
import torch

import cuopo_amd as P
from cuopo_amd import surrogate as S
from cuopo_amd import sweep as SW

WIDTH, DEPTH, N_IN, N_OUT = 256, 4, 5, 4096  # the network the package trains


def listed():
    return [
        # The smallest grid in use: two equations, 2^12 samples, 32 slices, one chunk of a converging run.
        dict(name="two_wave_4k", kind="solver", family="c1", N=1 << 12, NZ=32, n_rt=50, fp32=False),
        # The same on device buffers the caller owns, a few round trips per call (code that cannot allocate).
        dict(name="noalloc_4k", kind="noalloc", family="c1", N=1 << 12, NZ=32, n_rt=5, fp32=False),
        # The ordinary continuous-wave run: three equations, 2^14 samples, 100 slices, one instance.
        dict(name="three_wave_16k", kind="solver", family="c2", N=1 << 14, NZ=100, n_rt=50, fp32=False),
        # A pulsed run at a medium grid in the FP32-complex variant (phase modulator and GDD on).
        dict(name="pulsed_64k_fp32c", kind="solver", family="c5", N=1 << 16, NZ=100, n_rt=20, fp32=True),
        # The largest grid: nanosecond pulses on 2^18 samples, 200 slices, phase modulator and GDD on.
        dict(name="pulsed_256k", kind="solver", family="c5", N=1 << 18, NZ=200, n_rt=10, fp32=False),
        # The sweep of the benchmark's headline: 256 warm-started points on one grid, FP64.
        dict(name="sweep_256x16k", kind="batch", family="sppl", N=1 << 14, count=256, NZ=100, n_rt=20, check=0,
             start="warm", fp32=False),
        # The sweep over four grid sizes (2^12..2^15), 256 points, FP64 ...
        dict(name="sweep_256_mixed", kind="batch", family="ppln", N=0, count=256, NZ=100, n_rt=20, check=0,
             start="noise", fp32=False),
        # ... and in the FP32-complex variant, as the sweep driver runs it by default.
        dict(name="sweep_256_mixed_fp32c", kind="batch", family="ppln", N=0, count=256, NZ=100, n_rt=10, check=0,
             start="noise", fp32=True),
        # One chunk of the training-set generation: 512 points at 4096 x 25 with the steady-state test, FP32C.
        dict(name="dataset_512x4k_fp32c", kind="batch", family="sppl", N=1 << 12, count=512, NZ=25, n_rt=100,
             check=50, start="noise", fp32=True),
        # The tail of a sweep, or a sweep of a few points: seven instances still iterating.
        dict(name="sweep_7x16k", kind="batch", family="sppl", N=1 << 14, count=7, NZ=100, n_rt=50, check=25,
             start="warm", fp32=False),
        # Training of the warm-start network: one epoch of eight minibatches of 256.
        dict(name="fit_256", kind="fit", points=2048, batch=256),
        # Inference for one sweep of 256 points.
        dict(name="predict_256", kind="predict", points=256),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    """Another case of the same ranges; every grid is a power of two (the solver takes no other), slice, round
    trip and instance counts and batch sizes are any number."""
    kind = rng.choice(["solver", "solver", "noalloc", "batch", "batch", "batch", "fit", "predict"])
    if kind == "solver":
        fam = rng.choice(["c1", "c2", "c5"])
        L = rng.randint(12, 18) if fam == "c5" else rng.randint(10, 15)
        NZ = rng.randint(20, 120)
        return dict(kind="solver", family=fam, N=1 << L, NZ=NZ, fp32=rng.random() < 0.4,
                    n_rt=max(2, min(60, int(50 * 2 ** 16 * 20 / ((1 << L) + (1 << 16)) / NZ))) + rng.randint(0, 5))
    if kind == "noalloc":
        return dict(kind="noalloc", family=rng.choice(["c1", "c2"]), N=1 << rng.randint(10, 15),
                    NZ=rng.randint(16, 100), n_rt=rng.randint(1, 9), fp32=rng.random() < 0.4)
    if kind == "batch":
        fp32 = rng.random() < 0.5
        fam = rng.choice(["sppl", "ppln"])
        L = rng.choice([0, 12, 13, 14, 15]) if fam == "ppln" else rng.randint(11, 14)
        count = _log_int(rng, 2, 4096 if L and L < 13 else 160)
        count = min(count, 512, (1 << 22) // (1 << (L or 14)))
        return dict(kind="batch", family=fam, N=(1 << L) if L else 0, count=count, NZ=rng.randint(20, 100),
                    n_rt=rng.randint(4, 12), check=rng.choice([0, 3]), start=rng.choice(["noise", "warm"]), fp32=fp32)
    if kind == "fit":
        b = _log_int(rng, 16, 256)
        return dict(kind="fit", points=b * rng.randint(3, 7) + rng.randint(0, b - 1), batch=b)
    return dict(kind="predict", points=_log_int(rng, 1, 700))


# ------------------------------------------------------------------ inputs

def _args(case, rng):
    """The instances' command-line arguments: the physics is drawn from the seed, as a sweep's points are."""
    fam, NZ, NRT = case["family"], case["NZ"], case["n_rt"] + 4
    one = dict(N=case["N"], NZ=NZ, NRT=NRT, lp_nm=532.0)
    if fam == "c1":  # two equations, MgO:PPLN, 5 mm, 2 W of pump
        a = P.Args(three_eqs=False, regime=P.CW, crystal=P.PPLN, Lambda=6.97, Nth=1.0,
                   R_pct=float(rng.uniform(96, 99)), lcr_mm=5.0, **one)
        a.Nth = 2.0 / P.derive(a).Pth
        return [a]
    if fam == "c2":  # three equations, sPPLT, 20 mm, 3 x threshold, detuned
        return [P.Args(three_eqs=True, regime=P.CW, crystal=P.SPPLT, Lambda=7.97, Nth=3.0, R_pct=98.0,
                       delta=float(rng.uniform(0, 0.2)), lcr_mm=20.0, ls_um=1.0, pm_mode=P.PM_THREE_WAVE, **one)]
    if fam == "c5":  # nanosecond pulses, three equations, phase modulator and GDD compensation
        return [P.Args(three_eqs=True, regime=P.NS, crystal=P.PPLN, Lambda=6.97, Nth=float(rng.uniform(3, 5)),
                       R_pct=98.0, gdd_pct=100.0, upm=1, md=0.8 / np.pi, fm=4.0, lcr_mm=5.0, **one)]
    if fam == "sppl":  # the training family: pump, detuning, crystal length, GDD and reflectivity all vary
        pts = S.sample_points(case["count"], int(rng.integers(1 << 30)))
        return [S.family_args(*p, N=case["N"], NZ=NZ, NRT=NRT) for p in pts]
    pts = SW.sweep_points(case["count"], int(rng.integers(1 << 30)))  # the degenerate PPLN sweep
    return [S.sweep_args(*p[1:], N=N, NZ=NZ, NRT=NRT) for p, N in zip(pts, _grids(case))]


def _grids(case):
    """The instances' grid sizes: one, or the benchmark sweep's mix of four."""
    if case["N"]:
        return [case["N"]] * case.get("count", 1)
    return [p[0] for p in SW.sweep_points(case["count"], 3)]


def _instances(case, seed):
    """Per instance: (params, w, T, Ap_in, As, Ai), everything a run is given."""
    rng = np.random.default_rng(seed)
    out, roots = [], {}
    for a in _args(case, rng):
        d = P.derive(a)
        p = P.params_from(d, P.FP32C if case["fp32"] else P.FP64)
        T, w = P.grids(d)
        Ap_in = P.pump_input(d)
        s = int(rng.integers(1 << 40))
        if case.get("start") == "warm":  # one mode pair at a fraction of the pump, over weak noise
            m = int(rng.integers(-40, 40))
            amp = d.Ap0 * rng.uniform(0.05, 0.6)
            if d.N not in roots:
                roots[d.N] = np.exp(2j * np.pi * np.arange(d.N) / d.N)
            tone = roots[d.N][(m * np.arange(d.N)) % d.N]
            As = amp * tone + P.noise(s, 0, 1e-6 * amp, d.N)
            Ai = amp * np.conj(tone) + P.noise(s, 1, 1e-6 * amp, d.N) if a.three_eqs else None
        else:
            As = P.noise(s, 0, 1e-20, d.N)
            Ai = P.noise(s, 1, 1e-20, d.N) if a.three_eqs else None
        out.append((p, w, T, Ap_in, As, Ai))
    return out


def _network_data(case, seed):
    """Features in the encoder's range, targets as the encoder lays them out: a few spectral lines of unit norm
    and a constant log power, signal then idler."""
    rng = np.random.default_rng(seed)
    n, nb = case["points"], N_OUT // 4
    X = rng.uniform(-1, 1, (n, N_IN)).astype(np.float32)
    Y = np.zeros((n, N_OUT), np.float32)
    for f in (0, 1):
        at = np.clip(nb // 2 + np.rint(rng.normal(0, 6, (n, 4))).astype(int), 0, nb - 1)
        amp = rng.uniform(0.05, 1.0, (n, 4))
        amp /= np.linalg.norm(amp, axis=1, keepdims=True)
        for k in range(4):
            Y[np.arange(n), 2 * f * nb + at[:, k]] = amp[:, k]
        Y[:, (2 * f + 1) * nb:(2 * f + 2) * nb] = rng.uniform(-0.4, 0.1, (n, 1))
    dims = [N_IN] + [WIDTH] * DEPTH + [N_OUT]
    w0 = []
    for i, o in zip(dims[:-1], dims[1:]):
        w0 += [rng.normal(0, math.sqrt(2.0 / i), o * i), rng.normal(0, 0.02, o)]
    return X, Y, np.concatenate(w0).astype(np.float32)


# ------------------------------------------------------------------ the passes

def prepare(case, seed):
    kind = case["kind"]
    if kind in ("fit", "predict"):
        X, Y, w0 = _network_data(case, seed)
        sur = S.Surrogate(seed=0, max_batch=256)
        sur.net.set_weights(w0)
        return dict(case=case, sur=sur, X=X, Y=Y, w0=w0)
    made = _instances(case, seed)
    if kind == "solver":
        p, w, T, Ap_in, As, Ai = made[0]
        s = P.Solver(p)
        s.upload(w, T, Ap_in, Ap_in[: p.N].copy(), As, Ai)
        return dict(case=case, solver=s, start=(Ap_in[: p.N].copy(), As, Ai))
    if kind == "noalloc":
        p, w, T, Ap_in, As, Ai = made[0]
        dt = torch.complex64 if case["fp32"] else torch.complex128
        f0 = torch.from_numpy(np.stack([x for x in (Ap_in[: p.N], As, Ai) if x is not None])).to("cuda", dt)
        return dict(case=case, params=p, w=w, T=T, pump=torch.from_numpy(Ap_in).to("cuda", dt), f0=f0,
                    fields=f0.clone())
    b = P.Batch([m[0] for m in made])
    for k, (p, w, T, Ap_in, As, Ai) in enumerate(made):
        b.upload(k, w, T, Ap_in, Ap_in[: p.N].copy(), As, Ai)
    b.autotune(iters=3)
    return dict(case=case, batch=b, start=[(m[1], m[2], m[3], m[3][: m[0].N].copy(), m[4], m[5]) for m in made])


def _single(case, x):
    """FP32C fields come back widened; they hold 32-bit values, and are kept as such."""
    return x.astype(np.complex64) if case["fp32"] else x


def run(state):
    case = state["case"]
    kind = case["kind"]
    if kind == "fit":
        state["sur"].net.set_weights(state["w0"])
        hist = state["sur"].fit(state["X"], state["Y"], epochs=1, batch=case["batch"], lr=1e-3, seed=1)
        return dict(loss=hist.astype(np.float32), weights=state["sur"].net.get_weights())
    if kind == "predict":
        return state["sur"].predict(state["X"])
    n = case["n_rt"]
    if kind == "solver":
        s = state["solver"]
        s.set_fields(*state["start"])
        s.run(0, n)
        power = s.power_history(n)
        return dict(fields=[_single(case, x) for x in s.download() if x is not None],
                    power=power.astype(np.float32) if case["fp32"] else power)
    if kind == "noalloc":
        fields = state["fields"]
        fields.copy_(state["f0"])
        power = np.zeros(n)
        st = torch.cuda.current_stream().cuda_stream
        P._check(P.lib().opo_run_noalloc(C.byref(state["params"]), P._ptr(state["w"]), P._ptr(state["T"]),
                                         C.c_void_p(state["pump"].data_ptr()), state["pump"].numel(),
                                         C.c_void_p(fields.data_ptr()), 0, n, P._ptr(power), C.c_void_p(st)))
        return dict(fields=fields, power=power.astype(np.float32) if case["fp32"] else power)
    # a batch goes on from where its last pass ended, as consecutive chunks of a sweep do
    b = state["batch"]
    rts, states = b.run_ex(n, check_every=case["check"], tol=1e-12 if case["check"] else 0.0)
    got = [b.download(k) for k in range(b.count)]
    power = b.power()
    sizes = sorted({x[0].size for x in got})
    fields = {}
    for N in sizes:
        for f, name in enumerate(("pump", "signal", "idler")):
            fields["%s_%d" % (name, N)] = _single(case, np.stack([x[f] for x in got if x[0].size == N]))
    return dict(fields=fields, power=power.astype(np.float32) if case["fp32"] else power, rts=rts, states=states)


# ------------------------------------------------------------------ 64-bit results

def _propagate(insts, n_rt):
    """n_rt round trips of instances that share the grid size, the equations and the slices: per slice a
    nonlinear half step, inverse transform, linear phase, forward transform, nonlinear half step; then the phase
    modulator, the GDD phase and the mirrors.  Returns the fields [field, instance, sample] and the signal power
    after each round trip."""
    dev = "cuda" if torch.cuda.is_available() else "cpu"
    ps = [i[0] for i in insts]
    N, NZ, three, ns = ps[0].N, ps[0].NZ, bool(ps[0].three_eqs), ps[0].regime == P.NS
    nf = 3 if three else 2
    real = lambda v: torch.tensor(np.array(v, np.float64), device=dev).reshape(-1, 1)  # noqa: E731
    par = lambda name: real([getattr(p, name) for p in ps])  # noqa: E731
    cplx = lambda v: torch.tensor(np.stack(v).astype(np.complex128), device=dev)  # noqa: E731
    w = torch.tensor(np.stack([i[1] for i in insts]), device=dev)
    pump = cplx([i[3] for i in insts])
    A = [pump[:, :N].clone(), cplx([i[4] for i in insts])] + ([cplx([i[5] for i in insts])] if three else [])
    dz, dk = par("dz"), par("dk")
    kap = [par(k) for k in (("kp", "ks", "ki") if three else ("kp", "ks"))]
    if three:  # the signal's frame; the pump's walk-off is taken against the idler, as the solver's model does
        walk = [1 / par("vp") - 1 / par("vi"), 0 * dz, 1 / par("vi") - 1 / par("vs")]
    else:
        walk = [1 / par("vp") - 1 / par("vs"), 0 * dz]
    lin = []
    for f, c in enumerate("psi"[:nf]):
        ph = dz * w * (walk[f] + 0.5 * w * par("b2" + c) + w * w * par("b3" + c) / 6)
        lin.append(torch.polar(torch.exp(-0.5 * par("alpha_cr" + c) * dz) * torch.ones_like(ph), ph))
    e = lambda x: torch.polar(torch.ones_like(x), x)  # noqa: E731
    gdd = par("GDD")
    any_gdd = bool((gdd != 0).any())
    comp = []
    for t, c in (("TODscomp", "s"), ("TODicomp", "i")):
        tod = par(t) * (par("b3" + c) != 0)
        comp.append(e(torch.where(gdd == 0, torch.zeros_like(w), 0.5 * w * (w * gdd + w * w * tod / 3.0))))
    eom = None
    if any(p.use_eom for p in ps):
        T = torch.tensor(np.stack([i[2] for i in insts]), device=dev)
        eom = e(par("use_eom") * par("mod_depth") * torch.sin(2 * math.pi * par("fpm") * T))
    mir = e(math.pi * par("delta"))
    amp = [None, torch.sqrt(par("Rs")), torch.sqrt(par("Ri"))]
    inv = lambda x: torch.fft.ifft(x)  # e^{+i} with 1/N  # noqa: E731

    def half(A, z):
        h = dz / 2
        if three:  # every stage sees the unchanged fields, so the stages differ by their phase only
            a, b, c = z, z + dz / 4, z + dz / 2
            em = e(-dk * a) + 4 * e(-dk * b) + e(-dk * c)
            ep = e(dk * a) + 4 * e(dk * b) + e(dk * c)
            p, s, i = A
            return [p + 1j * kap[0] * em * h / 6 * s * i, s + 1j * kap[1] * ep * h / 6 * p * i.conj(),
                    i + 1j * kap[2] * ep * h / 6 * p * s.conj()]
        p, s = A
        f = lambda x, y, zz: (1j * kap[0] * y * y * e(dk * zz), 1j * kap[1] * x * y.conj() * e(-dk * zz))  # noqa: E731
        k1 = f(p, s, z)
        k2 = f(p + k1[0] / 2, s + k1[1] / 2, z + dz / 4)
        k3 = f(p + k2[0] / 2, s + k2[1] / 2, z + dz / 4)
        k4 = f(p + k3[0], s + k3[1], z + dz / 2)
        return [x + h / 6 * (a + 2 * b + 2 * c + d) for x, a, b, c, d in zip((p, s), k1, k2, k3, k4)]

    power = []
    for rt in range(n_rt):
        if ns:
            nrt = ps[0].NRT
            off = 0 if rt == 0 else (rt * N if rt < nrt - 1 else N * nrt - 1 - N)
            A[0] = pump[:, off:off + N].clone()
        else:
            A[0] = pump[:, :N].clone()
        z = torch.zeros_like(dz)
        for _ in range(NZ):
            A = half(A, z)
            A = [torch.fft.fft(inv(x) * q) for x, q in zip(A, lin)]
            A = half(A, z)
            z = z + dz
        if eom is not None:
            A = [A[0]] + [x * eom for x in A[1:]]
        if any_gdd:
            A = [A[0]] + [torch.fft.fft(inv(x) * q) for x, q in zip(A[1:], comp)]
        A = [A[0]] + [x * g * mir for x, g in zip(A[1:], amp[1:])]
        power.append((A[1].abs() ** 2).sum(1))
    return torch.stack(A), torch.stack(power)


def _exact_network(case, seed):
    X, Y, w0 = _network_data(case, seed)
    dims = [N_IN] + [WIDTH] * DEPTH + [N_OUT]
    dev = "cuda" if torch.cuda.is_available() else "cpu"
    X, Y = torch.tensor(X, device=dev, dtype=torch.float64), torch.tensor(Y, device=dev, dtype=torch.float64)
    w = torch.tensor(w0, device=dev, dtype=torch.float64).requires_grad_(case["kind"] == "fit")

    def net(x, w):
        o = 0
        for k, (i, j) in enumerate(zip(dims[:-1], dims[1:])):
            W, b = w[o:o + i * j].reshape(j, i), w[o + i * j:o + i * j + j]
            o += i * j + j
            x = x @ W.t() + b
            if k < DEPTH:
                x = torch.nn.functional.gelu(x)
        return x

    if case["kind"] == "predict":
        return net(X, w)
    n, b = X.shape[0], case["batch"]
    order = np.random.default_rng(1).permutation(n)
    m, v, tot, t = torch.zeros_like(w), torch.zeros_like(w), 0.0, 0
    for s in range(0, n - b + 1 if n >= b else 1, b):
        idx = torch.tensor(order[s:s + b], device=dev)
        loss = ((net(X[idx], w) - Y[idx]) ** 2).mean()
        g, = torch.autograd.grad(loss, w)
        t += 1
        with torch.no_grad():
            m, v = 0.9 * m + 0.1 * g, 0.999 * v + 0.001 * g * g
            w -= 1e-3 * (m / (1 - 0.9 ** t)) / (torch.sqrt(v / (1 - 0.999 ** t)) + 1e-8)
        tot += float(loss) * len(idx)
    return dict(loss=np.array([tot / max(1, (n // b) * b if n >= b else n)]), weights=w.detach())


def exact(case, seed):
    if case["kind"] in ("fit", "predict"):
        return _exact_network(case, seed)
    insts = _instances(case, seed)
    n = case["n_rt"]
    if case["kind"] in ("solver", "noalloc"):
        A, power = _propagate(insts, n)
        fields = A[:, 0] if case["kind"] == "noalloc" else [x[0] for x in A]
        return dict(fields=fields, power=power[:, 0])
    fields, last = {}, np.zeros(len(insts))
    for N in sorted({i[0].N for i in insts}):
        who = [k for k, i in enumerate(insts) if i[0].N == N]
        A, power = _propagate([insts[k] for k in who], n)
        for f, name in enumerate(("pump", "signal", "idler")):
            fields["%s_%d" % (name, N)] = A[f]
        last[who] = power[-1].cpu().numpy()
    return dict(fields=fields, power=last, rts=None, states=None)


def work(case):
    """Transforms at 5 N log2 N, six operations per sample of linear phase, and the nonlinear half steps (14 per
    field with three equations, about 100 per field with two); fields and tables read once, fields written once."""
    kind = case["kind"]
    if kind in ("fit", "predict"):
        par = N_IN * WIDTH + (DEPTH - 1) * WIDTH * WIDTH + WIDTH * N_OUT
        if kind == "predict":
            return dict(flops=2.0 * par * case["points"], bytes=4.0 * case["points"] * (N_IN + N_OUT) + 2.0 * par)
        n = max(1, case["points"] // case["batch"]) * min(case["batch"], case["points"])
        steps = max(1, case["points"] // case["batch"])
        return dict(flops=6.0 * par * n, bytes=4.0 * n * (N_IN + N_OUT) + 28.0 * par * steps)
    three = case["family"] != "c1"
    nf = 3 if three else 2
    sc = 8 if case["fp32"] else 16
    flops = total = 0.0
    for N in _grids(case):
        per = nf * N * (10 * math.log2(N) + 6) + 2 * N * (42 if three else 200)
        flops += case["n_rt"] * (case["NZ"] * per + 20 * N)
        total += sc * N * (3 * nf + (case["n_rt"] if case["family"] == "c5" else 1))
    return dict(flops=flops, bytes=total)
