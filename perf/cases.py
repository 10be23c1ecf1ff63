"""The work that programs have this framework do, as cases that can be timed.

A case is a dict of plain values.  Its "kind" says which part of the public
interface a pass goes through (cudamica_amd.engine):

  fit      a recording that the engine already holds whitened: load a model
           state, run some EM iterations as a replayed graph, read the state
           and the log back
  job      a whole decomposition from the raw recording: load, centre and
           sphere, EM iterations, then the model in sensor space
  batch    some EM iterations of many recordings in one batch, every
           recording's state read back
  score    per-sample log-likelihoods of a fixed model (amica_ll_forward)
  serve    the same through the allocation-free call (amica_ll_forward_noalloc)
  adjoint  log-likelihoods and the gradients of every parameter

listed() holds the shapes of this repository's workloads and tests and some
generic ones; draw() gives more of the same ranges.  Engine results are
handed back as the float32 that the density math of every engine precision
has (a program applies them to float32 recordings); the likelihood calls'
results in the precision they were asked to compute in, and what
preprocessing computes in float64 as float64.
"""
import math

import numpy as np
import torch

from cudamica_amd import engine as amica

PRECISION = {"fp32": amica.PREC_FP32, "plain": amica.PREC_FP32_PLAIN,
             "bf16": amica.PREC_BF16, "fp8": amica.PREC_FP8}
LOG2 = 0.693147180559945   # the constant of the density (include/amica_adjoint.h)


def listed():
    return [
        # scoring one short window of 32 channels inside a serving loop
        dict(name="serve_n32_T4k", kind="serve", bits=32, n=32, T=4096, M=1, m=3),
        # the small reference recording: each kernel is short, launches count;
        # rho held at 1.5 as for a parameter file without update_rho
        dict(name="fit_n16_T20k", kind="fit", precision="fp32", n=16, T=20_000, M=1, m=3, iters=5,
             update_rho=0),
        # an EEG recording of 64 channels, one model, the parity precision
        dict(name="fit_n64_T1M", kind="fit", precision="fp32", n=64, T=1_000_000, M=1, m=3, iters=2,
             update_rho=0),
        # an odd channel and sample count, two models
        dict(name="fit_n71_T200k", kind="fit", precision="bf16", n=71, T=200_003, M=2, m=3, iters=2,
             update_rho=0),
        # the headline workload: 128 channels, 4 models, mixed precision
        dict(name="fit_n128_T2M_M4", kind="fit", precision="bf16", n=128, T=2_000_000, M=4, m=3, iters=1,
             update_rho=1),
        # the largest: 256 channels, whitened data stored as FP8, 4 components
        dict(name="fit_n256_T4M_M2", kind="fit", precision="fp8", n=256, T=4_000_000, M=2, m=4, iters=1,
             update_rho=1),
        # from a raw 128-channel recording to the first iterations' model
        dict(name="job_n128_T1M", kind="job", precision="bf16", n=128, T=1_000_000, M=1, m=3, iters=2,
             update_rho=0, sphere=1, host=False),
        # the same for a MEG-like channel count, past one workgroup's channels
        dict(name="job_n260_T50k", kind="job", precision="fp32", n=260, T=50_000, M=2, m=3, iters=1,
             update_rho=1, sphere=1, host=False),
        # recordings of several subjects side by side
        dict(name="batch_8", kind="batch", precision="bf16", recordings=8, sizes=3, m=3, iters=2),
        # scoring a long recording in double precision
        dict(name="score_n100_T200k", kind="score", bits=64, n=100, T=200_000, M=2, m=3),
        # a gradient step of a program that optimises the likelihood itself
        dict(name="adjoint_n128_T500k", kind="adjoint", bits=32, n=128, T=500_000, M=2, m=3),
        # the same in double precision on a short segment
        dict(name="adjoint64_n40_T30k", kind="adjoint", bits=64, n=40, T=30_011, M=2, m=4),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["fit", "fit", "fit", "job", "job", "batch", "score", "serve", "adjoint", "adjoint"])
    if kind == "batch":
        return dict(kind=kind, precision=rng.choice(["bf16", "fp32"]), recordings=rng.randint(2, 12),
                    sizes=rng.randrange(1 << 20), m=3, iters=rng.randint(1, 3))
    M, m = rng.choice([1, 1, 2, 3, 4]), rng.choice([1, 2, 3, 3, 4])
    if kind == "serve":
        n = _log_int(rng, 8, 128)
        return dict(kind=kind, bits=rng.choice([32, 64]), n=n, T=_log_int(rng, 256, 50_000),
                    M=min(M, 65536 // (n * n)), m=m)
    if kind in ("score", "adjoint"):
        n = _log_int(rng, 8, 280)
        T = _log_int(rng, 2_000, max(4_000, min(1_000_000, 60_000_000 // (n * M))))
        return dict(kind=kind, bits=rng.choice([32, 32, 64]), n=n, T=T, M=M, m=m)
    if kind == "fit":
        n = _log_int(rng, 8, 256)
        T = _log_int(rng, 60 * n, max(120 * n, min(2_000_000, 500_000_000 // (n * M * m))))
        rho = rng.randint(0, 1)
        return dict(kind=kind, precision=rng.choice(["fp32", "fp32", "plain", "bf16", "bf16", "fp8"]), n=n, T=T,
                    M=M, m=m, iters=1 if rho else rng.randint(1, 3), update_rho=rho)
    n = _log_int(rng, 8, 200)
    T = _log_int(rng, 60 * n, max(120 * n, min(1_000_000, 150_000_000 // (n * M))))
    return dict(kind=kind, precision=rng.choice(["fp32", "bf16", "fp8"]), n=n, T=T, M=M, m=m, iters=1,
                update_rho=1, sphere=rng.choice([1, 1, 1, 2]), host=n * T <= 4_000_000 and rng.random() < 0.5)


def _batch_sizes(case):
    rng = np.random.default_rng(case["sizes"])
    return [(int(rng.choice((32, 64, 128))), int(rng.integers(100_000, 500_001)))
            for _ in range(case["recordings"])]


# inputs -----------------------------------------------------------------------

def _recording(n, T, seed, nmix=1):
    """T x n float32 on the GPU: super-Gaussian sources, mixed by matrices of
    condition number 30 that alternate over blocks of samples, plus a constant
    offset per channel."""
    g = torch.Generator("cuda").manual_seed(seed)
    rng = np.random.default_rng(seed)
    s = torch.randn((T, n), generator=g, device="cuda")
    s = torch.sign(s) * s.abs().pow(1.0 + 0.8 * torch.rand(n, generator=g, device="cuda"))
    block = -(-T // (8 * nmix))
    mixes = []
    for _ in range(nmix):
        q1, q2 = (np.linalg.qr(rng.standard_normal((n, n)))[0] for _ in range(2))
        mixes.append(torch.tensor((q1 * np.logspace(0.0, -1.48, n)) @ q2, dtype=torch.float32, device="cuda"))
    x = torch.empty_like(s)
    for k, t in enumerate(range(0, T, block)):
        torch.mm(s[t:t + block], mixes[k % nmix].T, out=x[t:t + block])
    x += 5.0 * torch.randn(n, generator=g, device="cuda")
    return x


def _model(n, M, m, seed):
    """A model in the middle of its fit, with W = A^-1 in the layout of the likelihood calls."""
    st = amica.synth_init(n, M, m, seed, fix_init=0)
    rng = np.random.default_rng(seed)
    a = rng.uniform(0.5, 1.5, (M, m, n))
    A = st["A"].reshape(M, n, n)                       # transposed: column-major models
    return dict(W=np.linalg.inv(A), c=0.1 * st["c"].reshape(M, n), alpha=a / a.sum(1, keepdims=True),
                mu=np.arange(m).reshape(1, m, 1) - (m - 1) / 2 + 0.1 * rng.standard_normal((M, m, n)),
                beta=rng.uniform(0.5, 1.5, (M, m, n)), rho=rng.uniform(1.1, 1.9, (M, m, n)),
                gm=np.full(M, 1.0 / M))


def _samples(case, seed):
    """Whitened samples (float32 or float64) and the upstream gradient of their likelihoods."""
    g = torch.Generator("cuda").manual_seed(seed)
    s = torch.randn((case["T"], case["n"]), generator=g, device="cuda", dtype=torch.float64)
    x = 1.2 * torch.sign(s) * s.abs().pow(1.4)
    dll = 0.5 + torch.rand(case["T"], generator=g, device="cuda", dtype=torch.float64)
    return x.to(torch.float64 if case["bits"] == 64 else torch.float32), dll


def _options(case, n, T):
    return amica.options(n, T, case.get("M", 1), case["m"], precision=PRECISION[case["precision"]],
                         max_iter=16, update_rho=case.get("update_rho", 0))


def _open(engine, x, sphere=1):
    if isinstance(x, np.ndarray):
        engine.load_raw(x)
    else:
        engine.load_raw_device(x.data_ptr())
    engine.preprocess(sphere)


def prepare(case, seed):
    kind = case["kind"]
    if kind in ("fit", "job"):
        n, T, M, m = (case[k] for k in ("n", "T", "M", "m"))
        x = _recording(n, T, seed, M)
        state = dict(case=case, init=amica.synth_init(n, M, m, seed), engine=amica.Engine(_options(case, n, T)))
        torch.cuda.synchronize()
        if kind == "fit":
            _open(state["engine"], x)
            S, state["mean"], _ = state["engine"].sphere()
            state["unsphere"] = np.linalg.inv(S.reshape(n, n))
        else:
            state["x"] = x.cpu().numpy() if case["host"] else x
        return state
    if kind == "batch":
        sizes = _batch_sizes(case)
        batch = amica.Batch([_options(case, n, T) for n, T in sizes])
        init, unsphere, mean = [], [], []
        for r, ((n, T), e) in enumerate(zip(sizes, batch.engines)):
            x = _recording(n, T, seed + 1000 * r)
            torch.cuda.synchronize()
            _open(e, x)
            S, mu, _ = e.sphere()
            unsphere.append(np.linalg.inv(S.reshape(n, n)))
            mean.append(mu)
            init.append(amica.synth_init(n, 1, case["m"], seed + 1000 * r))
        return dict(case=case, batch=batch, init=init, unsphere=unsphere, mean=mean)
    x, dll = _samples(case, seed)
    model = {k: torch.tensor(v, dtype=torch.float64, device="cuda").contiguous()
             for k, v in _model(case["n"], case["M"], case["m"], seed).items()}
    return dict(case=case, x=x, dll=dll, model=model, address={k: v.data_ptr() for k, v in model.items()},
                ll=torch.empty(case["T"], dtype=torch.float64, device="cuda"),
                grad=torch.empty(sum(v.numel() for v in model.values()), dtype=torch.float64, device="cuda"))


# one pass ---------------------------------------------------------------------

def _results(engine, iters, mean, unsphere):
    """The fitted model (its centres in sensor space) and its history, float32."""
    st, log = engine.get_state(), engine.log(iters)
    st["c"] = mean + st["c"].reshape(-1, len(mean)) @ unsphere
    st.update(ll=log["ll"], lrate=log["lrate"], vsum=log["vsum"])
    return {k: v.ravel().astype(np.float32) for k, v in st.items()}


def run(state):
    case, kind = state["case"], state["case"]["kind"]
    if kind == "fit":
        e = state["engine"]
        e.set_state(state["init"])
        e.iterate(case["iters"], graph=True)
        return _results(e, case["iters"], state["mean"], state["unsphere"])
    if kind == "job":
        e = state["engine"]
        _open(e, state["x"], case["sphere"])
        e.set_state(state["init"])
        e.iterate(case["iters"], graph=True)
        st, log = e.get_state(), e.log(case["iters"])
        A, c = e.output()
        S, mean, ldetS = e.sphere()
        out = dict(A=A, c=c, ll=log["ll"], vsum=log["vsum"],
                   **{k: st[k] for k in ("W", "alpha", "mu", "beta", "rho", "gm")})
        return dict({k: v.ravel().astype(np.float32) for k, v in out.items()}, S=S, mean=mean, ldetS=ldetS)
    if kind == "batch":
        batch = state["batch"]
        for e, init in zip(batch.engines, state["init"]):
            e.set_state(init)
        batch.iterate(case["iters"])
        got = [_results(e, case["iters"], mean, un)
               for e, mean, un in zip(batch.engines, state["mean"], state["unsphere"])]
        return {k: np.concatenate([r[k] for r in got]) for k in got[0]}
    n, T, M, m, bits = (case[k] for k in ("n", "T", "M", "m", "bits"))
    real = torch.float64 if bits == 64 else torch.float32
    args = (bits, state["x"].data_ptr(), T, n, M, m, state["address"], 0.0)
    if kind == "serve":
        amica.ll_forward_noalloc(*args, state["ll"].data_ptr())
        return state["ll"].to(real)
    if kind == "score":
        amica.ll_forward(*args, state["ll"].data_ptr())
        return state["ll"].to(real)
    at, grads = state["grad"].data_ptr(), {}
    for k, v in state["model"].items():
        grads[k] = at
        at += 8 * v.numel()
    amica.ll_adjoint(*args, state["dll"].data_ptr(), grads, state["ll"].data_ptr())
    parts = torch.split(state["grad"].to(real), [v.numel() for v in state["model"].values()])
    return dict(zip(("d" + k for k in state["model"]), parts), ll=state["ll"].to(real))


# what a pass cannot do without ---------------------------------------------------

def work(case):
    kind, m = case["kind"], case["m"]
    if kind == "batch":
        parts = [work(dict(case, kind="fit", n=n, T=T, M=1)) for n, T in _batch_sizes(case)]
        return {k: sum(p[k] for p in parts) for k in ("bytes", "flops")}
    n, T, M = case["n"], case["T"], case["M"]
    gemm, state = 2.0 * T * M * n * n, 8.0 * M * n * (2 * n + 4 * m + 1)
    if kind in ("fit", "job"):
        # unmixing and statistic products; about 40 operations per density and its sums
        flops = case["iters"] * (2 * gemm + 40.0 * T * M * n * m)
        data = case["iters"] * float(T) * n * (1 if case["precision"] == "fp8" else 4)
        if kind == "job":
            flops += 3.0 * T * n * n          # covariance (one triangle) and sphering
            data += 4.0 * T * n
        return {"bytes": data + 2 * state, "flops": flops}
    values = T * n * (8.0 if case["bits"] == 64 else 4.0) + 8.0 * T + state
    if kind == "adjoint":
        return {"bytes": values + 8.0 * T + state, "flops": 2 * gemm + 50.0 * T * M * n * m}
    return {"bytes": values, "flops": gemm + 20.0 * T * M * n * m}


# the same in 64 bits, plainly -------------------------------------------------------

def _components(b, p, h):
    """y, |y| and the component log-densities Q (t, m, n) of model h at b (t, n)."""
    y = p["beta"][h].sqrt() * (b[:, None, :] - p["mu"][h])
    ay = y.abs()
    Q = (p["alpha"][h].log() + 0.5 * p["beta"][h].log() - LOG2 - torch.lgamma(1.0 + 1.0 / p["rho"][h])
         - (p["rho"][h] * ay.log()).exp())
    return y, ay, Q


def _likelihood(x, p, ldetS):
    """b and log-density sums per model, and the models' log-likelihoods (M, t)."""
    bs, L = [], []
    for h in range(len(p["gm"])):
        b = x @ p["W"][h].T - p["W"][h] @ p["c"][h]
        L.append(p["gm"][h].log() + torch.linalg.slogdet(p["W"][h])[1] + ldetS
                 + torch.logsumexp(_components(b, p, h)[2], 1).sum(1))
        bs.append(b)
    return bs, torch.stack(L)


def _em_step(x, p, ldetS, update_rho, lrate, ll_prev, first):
    """One EM iteration with the natural-gradient step; p is replaced in place."""
    T, n = x.shape
    M, m = p["alpha"].shape[:2]
    z = lambda *s: torch.zeros(s, dtype=torch.float64, device=x.device)  # noqa: E731
    p["W"] = torch.linalg.inv(p["A"])
    names = ("u", "mn", "md", "bd", "rn")
    s = {k: z(M, m, n) for k in names}
    cnew, phi, vsum, total = z(M, n), z(M, n, n), z(M), 0.0
    step = max(1, (1 << 27) // (n * m * M))
    for t in range(0, T, step):
        xt = x[t:t + step]
        bs, L = _likelihood(xt, p, ldetS)
        P = torch.logsumexp(L, 0)
        total += float(P.sum())
        v = (L - P).exp()
        vsum += v.sum(1)
        for h in range(M):
            y, ay, Q = _components(bs[h], p, h)
            u = v[h][:, None, None] * torch.softmax(Q, 1)
            rho, sb = p["rho"][h], p["beta"][h].sqrt()
            lay = ay.log()
            w = rho * ((rho - 2.0) * lay).exp()            # f / y
            f = w * y
            uf = u * f
            s["u"][h] += u.sum(0)
            s["mn"][h] += uf.sum(0)
            s["md"][h] += sb * (u * w).sum(0)
            s["bd"][h] += (uf * y).sum(0)
            yr = (rho * lay).exp()
            s["rn"][h] += (u * torch.where(yr > 0, yr * rho * lay, 0.0)).sum(0)
            cnew[h] += v[h] @ xt
            phi[h] += (sb * uf).sum(1).T @ bs[h]
    ll = total / (n * T)
    if not first and ll < ll_prev:
        lrate *= 0.5
    used, lrate = lrate, min(0.1, lrate + min(0.1, lrate))
    p["gm"] = vsum / T
    p["alpha"] = s["u"] / vsum[:, None, None]
    mu, beta, rho = p["mu"] + s["mn"] / s["md"], p["beta"] * s["u"] / s["bd"], p["rho"]
    if update_rho:
        rho = (rho + 0.1 * (1.0 - rho / torch.digamma(1.0 + 1.0 / rho) * s["rn"] / s["u"])).clamp(1.0, 2.0)
    cnew /= vsum[:, None]
    eye = torch.eye(n, dtype=torch.float64, device=x.device)
    A = p["A"] - lrate * p["A"] @ (eye - phi / vsum[:, None, None])
    nu = A.norm(dim=1)
    shift = torch.stack([p["W"][h] @ (cnew[h] - p["c"][h]) for h in range(M)])
    p.update(A=A / nu[:, None, :], mu=mu * nu[:, None, :] - shift[:, None, :], beta=beta / nu[:, None, :] ** 2,
             rho=rho, c=cnew)
    return ll, used, lrate, vsum


def _sphere(x, how):
    """S, mean, log-determinant term and the whitened data of a raw recording."""
    T, n = x.shape
    parts = [x[t:t + (1 << 18)] for t in range(0, T, 1 << 18)]
    mean = sum(q.double().sum(0) for q in parts) / T
    C = sum((q.double() - mean).T @ (q.double() - mean) for q in parts) / T
    if how == 1:
        d, V = np.linalg.eigh(C.cpu().numpy())
        S = (V * (2.0 / np.sqrt(d))) @ V.T
    else:
        S = np.diag(1.0 / np.sqrt(np.diag(C.cpu().numpy()) * T / (T - 1)))
    ldetS = -np.linalg.slogdet(S)[1]
    St = torch.tensor(S, device=x.device)
    return S, mean, ldetS, torch.cat([(q.double() - mean) @ St.T for q in parts])


def _exact_fit(case, n, T, M, x, init):
    m = case["m"]
    S, mean, ldetS, xw = _sphere(x, case.get("sphere", 1))
    shape = dict(A=(M, n, n), c=(M, n), gm=(M,))
    p = {k: torch.tensor(v, device="cuda").reshape(shape.get(k, (M, m, n))) for k, v in init.items()}
    p["A"] = p["A"].transpose(1, 2).contiguous()
    lrate, ll, hist = 0.1, -math.inf, []
    for it in range(case["iters"]):
        ll, used, lrate, vsum = _em_step(xw, p, ldetS, case.get("update_rho", 0), lrate, ll, it == 0)
        hist.append((ll, used, vsum))
    flat = lambda t: t.cpu().numpy().ravel()  # noqa: E731
    out = {k: flat(p[k]) for k in ("alpha", "mu", "beta", "rho", "gm")}
    out["W"] = flat(p["W"].transpose(1, 2))
    unsphere = torch.linalg.inv(torch.tensor(S, device="cuda"))
    out["c"] = flat(mean + p["c"] @ unsphere.T)
    A = p["A"]
    if case["kind"] == "job":
        A = unsphere @ A
        A = A / A.norm(dim=1, keepdim=True)
        out.update(S=S.T.ravel(), mean=flat(mean), ldetS=float(ldetS))
    else:
        out["lrate"] = np.array([h[1] for h in hist])
    out["A"] = flat(A.transpose(1, 2))
    out["ll"] = np.array([h[0] for h in hist])
    out["vsum"] = np.concatenate([flat(h[2]) for h in hist])
    return out


def exact(case, seed):
    kind = case["kind"]
    if kind in ("fit", "job"):
        n, T, M = case["n"], case["T"], case["M"]
        return _exact_fit(case, n, T, M, _recording(n, T, seed, M), amica.synth_init(n, M, case["m"], seed))
    if kind == "batch":
        got = [_exact_fit(case, n, T, 1, _recording(n, T, seed + 1000 * r),
                          amica.synth_init(n, 1, case["m"], seed + 1000 * r))
               for r, (n, T) in enumerate(_batch_sizes(case))]
        return {k: np.concatenate([r[k] for r in got]) for k in got[0]}
    n, T, M, m = (case[k] for k in ("n", "T", "M", "m"))
    x, dll = _samples(case, seed)
    p = {k: torch.tensor(v, device="cuda") for k, v in _model(n, M, m, seed).items()}
    leaf = {k: v.clone().requires_grad_(kind == "adjoint") for k, v in p.items()}
    q = dict(leaf, W=leaf["W"].transpose(1, 2))
    ll = torch.empty(T, dtype=torch.float64, device="cuda")
    step = max(1, (1 << 26) // (n * m * M))
    for t in range(0, T, step):
        part = torch.logsumexp(_likelihood(x[t:t + step].double(), q, 0.0)[1], 0)
        if kind == "adjoint":
            (dll[t:t + step] * part).sum().backward()
        ll[t:t + step] = part.detach()
    if kind != "adjoint":
        return ll
    return dict({"d" + k: leaf[k].grad.reshape(-1) for k in p}, ll=ll)
