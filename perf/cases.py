"""The timed cases: what a user of the transform has it do, through the public
entry points.

Band limits run over 32..1024 (the range the request loop is quoted on),
azimuthal band limits over 1..8, dilations 2 and 3.  ``path`` is one of

- ``analysis`` / ``synthesis``: a device-resident plan (`core.Plan`), the
  coefficients staying in GPU memory;
- ``split``: the analysis of a plan with the split-precision contraction;
- ``moments``: analysis reduced to the per-scale moments (the statistics
  pipeline), through `analysis_moments` where the plan offers it;
- ``dropin``: the host-array procedures of the Fortran module's mirror, an
  analysis followed by a synthesis of its result;
- ``serve``: a batch of mixed requests through the request loop.
"""
import math

import numpy as np
import torch

from s2dw_amd import core
from s2dw_amd.serve import Server

DEV = "cuda"


# ------------------------------------------------------------------ the cases
def _case(name, path, L, N, alpha=2, jmin=0, red=False, graphs=False):
    c = {"path": path, "L": L, "N": N, "alpha": alpha, "jmin": jmin, "red": red, "graphs": graphs}
    return {"name": name, **c} if name else c


def listed():
    return [
        # the smallest calls: the round-trip test program's size, one transform at a time (latency, launches)
        _case("analysis_64", "analysis", 64, 3),
        _case("synthesis_64", "synthesis", 64, 3),
        # ordinary sizes that are no power of two: the middle of the served range, dilation 3
        _case("analysis_181_a3", "analysis", 181, 4, alpha=3),
        _case("synthesis_397", "synthesis", 397, 6),
        # the benchmark's configuration, replayed from the plan's graphs as the benchmark does
        _case("analysis_512", "analysis", 512, 8, jmin=2, red=True, graphs=True),
        _case("synthesis_512", "synthesis", 512, 8, jmin=2, red=True, graphs=True),
        # the same with the split-precision contraction
        _case("split_512", "split", 512, 8, jmin=2, red=True),
        # the largest served transforms: the full range's end, and a ragged one beside it
        _case("analysis_1024", "analysis", 1024, 8, red=True),
        _case("synthesis_899_a3", "synthesis", 899, 5, alpha=3),
        # statistics of the coefficients of an odd-sized map
        _case("moments_300", "moments", 300, 8, red=True),
        # a Fortran host program's call on its own arrays: analysis, then synthesis
        _case("dropin_256", "dropin", 256, 5),
        # a batch of every L in 64..512 with every N in 1, 3, 5, 8 through the request loop
        _case("serve_mix", "serve", 512, 8),
    ]


def draw(rng):
    path = rng.choice(["analysis"] * 3 + ["synthesis"] * 3 + ["moments", "split", "dropin"])
    top = {"dropin": 256, "split": 512}.get(path, 900)  # none costs more than the listed transforms of L = 1024
    L = min(top, int(round(math.exp(rng.uniform(math.log(32), math.log(top))))))
    return _case(None, path, L, rng.randint(1, 8), alpha=rng.choice([2, 3]), jmin=rng.choice([0, 0, 1, 2]),
                 red=rng.random() < 0.5, graphs=path in ("analysis", "synthesis") and rng.random() < 0.25)


def _serve_mix():
    return [(L, N) for L in (64, 128, 256, 512) for N in (1, 3, 5, 8)]


# ------------------------------------------------------------------ geometry
def _near_int(x):
    y = round(x)
    return y if abs(x - y) < 1e-5 else None


def _limits(j, L, alpha):
    xh, xl = L / float(alpha) ** (j - 1), L / float(alpha) ** (j + 1)
    hi, lo = _near_int(xh), _near_int(xl)
    hi = math.ceil(xh) if hi is None else hi
    lo = math.floor(xl) if lo is None else lo
    return min(hi, L), max(lo, 0)


def _jmax(L, alpha):
    y = math.log(L) / math.log(alpha)
    n = _near_int(y)
    return math.ceil(y) if n is None else n


def _geometry(case):
    """J, per-scale (hi, lo) and the band limit of the scaling coefficients."""
    L, alpha = case["L"], case["alpha"]
    J = max(1, _jmax(L, alpha) - case["jmin"])
    x = L / float(alpha) ** J
    bl = _near_int(x)
    return J, [_limits(j, L, alpha) for j in range(J + 1)], math.ceil(x) if bl is None else bl


# ------------------------------------------------------------------ the inputs
def _gen(seed):
    g = torch.Generator(device=DEV)
    g.manual_seed(int(seed))
    return g


def _flm(L, seed, red):
    """flm[m, l] (l fastest, the Fortran order) of a real signal: Re, Im ~ N(0, 1) for m <= l, f_l0 real; a red
    spectrum falls as 1/(l+1)."""
    f = torch.randn((L, L), dtype=torch.complex128, device=DEV, generator=_gen(seed)) * math.sqrt(2.0)
    f[0].imag.zero_()
    f = torch.triu(f)
    if red:
        f = f / torch.arange(1, L + 1, device=DEV, dtype=torch.float64)
    return f.contiguous()


def _wav(case, seed):
    """Packed wavelet coefficients, N(0, 1) (with a red spectrum falling towards the finest scales) and scaling
    coefficients, as a program holds them after thresholding or simulation."""
    J, lim, bl = _geometry(case)
    g = _gen(seed)
    parts = []
    for j, (h, _) in enumerate(lim):
        w = torch.randn((2 * h - 1) * 2 * h * case["N"], dtype=torch.float64, device=DEV, generator=g)
        parts.append(w * (2.0 ** (j - J) if case["red"] else 1.0))
    return torch.cat(parts), _flm(bl, seed + 1, case["red"])


class _Requests:
    """A running request loop and the batch a client submits to it."""

    def __init__(self, seed):
        self.mix = [(L, N, _jmax(L, 2)) for L, N in _serve_mix()]
        self.server = Server(hbm_budget_bytes=64 << 30, max_inflight=8)
        self.flm = None
        self.load(seed + 1)
        for _ in range(2):  # a running service: its plans and buffers are there
            self.batch()
        self.load(seed)

    def load(self, seed):
        self.flm = [np.asfortranarray(_flm(L, 64 * seed + i, True).cpu().numpy().T)
                    for i, (L, _, _) in enumerate(self.mix)]

    def batch(self):
        s = self.server
        ana = [s.submit_analysis(L, N, J, 2.0, f, keep_resident=True, want_wav=False)
               for (L, N, J), f in zip(self.mix, self.flm)]
        syn = [s.submit_synthesis(L, N, J, 2.0, wav_from=t) for (L, N, J), t in zip(self.mix, ana)]
        out = [s.result(t) for t in syn]
        sc = [s.result(t)[1] for t in ana]
        for t in ana:
            s.release(t)
        return {"flm": out, "scoeff": sc}

    def __del__(self):
        try:
            self.server.close()
        except Exception:
            pass


class _Device:
    """A plan and the device buffers of one program."""


def prepare(case, seed):
    if case["path"] == "serve":
        return _Requests(seed)
    L, N, alpha = case["L"], case["N"], float(case["alpha"])
    J, _, _ = _geometry(case)
    K, Phi2, bl = core.s2dw_core_init_kernels(J, L, alpha)
    S = core.s2dw_core_init_directionality(L, N)
    st = _Device()
    st.path = case["path"]
    if st.path == "dropin":
        st.args = (K, S, J, L, N, bl, alpha)
        st.Phi2 = Phi2
        st.flm = np.asfortranarray(_flm(L, seed, case["red"]).cpu().numpy().T)
        return st
    st.plan = core.Plan(L, N, J, alpha, K, Phi2, S, precision=core.PREC_SPLIT if st.path == "split" else core.PREC_FP64)
    st.plan.set_graphs(case["graphs"])
    if st.path == "synthesis":
        st.wav, st.sc = _wav(case, seed)
        st.flm = st.plan.empty_flm()
        return st
    st.flm = _flm(L, seed, case["red"])
    st.sc = st.plan.empty_scoeff()
    st.fused = st.path == "moments" and st.plan.moments_fusable
    st.wav = None if st.fused else st.plan.empty_wav()
    if st.path == "moments":
        st.out = torch.empty((8, J + 1), dtype=torch.float64, device=DEV)
    return st


def run(st):
    if isinstance(st, _Requests):
        return st.batch()
    if st.path == "dropin":
        K, S, J, L, N, bl, alpha = st.args
        wav, sc = core.s2dw_core_analysis_flm2wav_dynamic(st.flm, K, S, J, L, N, bl, alpha)
        flm = core.s2dw_core_synthesis_wav2flm_dynamic(wav, sc, K, st.Phi2, S, J, L, N, bl, alpha)
        return {"wav": wav, "scoeff": sc, "flm": flm}
    if st.path == "synthesis":
        st.plan.synthesis(st.wav, st.sc, st.flm)
        return {"flm": st.flm}
    if st.path == "moments":
        if st.fused:
            st.plan.analysis_moments(st.flm, st.sc, st.out)
        else:
            st.plan.analysis(st.flm, st.wav, st.sc)
            st.plan.stat_moments(st.wav, None, st.out)
        return {"scoeff": st.sc, **{n: st.out[i] for i, n in enumerate(st.plan.MOMENT_ROWS)}}
    st.plan.analysis(st.flm, st.wav, st.sc)
    return {"wav": st.wav, "scoeff": st.sc}


# ------------------------------------------------------------------ what a pass cannot do without
def _work_one(L, N, lim, bl, analysis, stored=True):
    nwav = sum((2 * h - 1) * 2 * h * N for h, _ in lim)
    nbytes = 16.0 * L * (L + 1) / 2 + 16.0 * bl * bl + (8.0 * nwav if stored else 0.0)
    flops = 0.0
    for h, lo in lim:
        for l in range(lo + 1, h):
            ns = [n for n in range(-(N - 1) if analysis else 0, N) if (N + n) % 2 and abs(n) <= l]
            flops += 8.0 * len(ns) * (l + 1) ** 2  # complex multiply-adds of the l-contraction
        na, nb = 2 * h - 1, 2 * h
        flops += 2.5 * N * nb * na * math.log2(max(2, na)) + 5.0 * N * h * nb * math.log2(nb)
    return nbytes, flops


def work(case):
    if case["path"] == "serve":
        b = f = 0.0
        for L, N in _serve_mix():
            g = _geometry(_case(None, "serve", L, N))
            for ana in (True, False):
                # the coefficients stay resident between the two requests; f_lm goes in and comes out
                x, y = _work_one(L, N, g[1], g[2], ana)
                b, f = b + x, f + y
        return {"bytes": b, "flops": f}
    J, lim, bl = _geometry(case)
    L, N, path = case["L"], case["N"], case["path"]
    b, f = _work_one(L, N, lim, bl, path != "synthesis", path != "moments")
    if path == "dropin":
        x, y = _work_one(L, N, lim, bl, False)
        b, f = b + x, f + y
    return {"bytes": b, "flops": f}


# ------------------------------------------------------------------ the same in plain torch and numpy, 64 bits
def _kernels(J, L, alpha):
    """K_j(l) and Phi^2(l) by the extended trapezoid / Simpson refinement that defines them (relative stopping
    tolerance 1e-12 after at least six refinements, limits moved in by 1e-12)."""
    alpha = float(alpha)

    def integrand(k, bw, lo):
        t = 2.0 * ((k - lo) / float(bw - lo)) - 1.0
        return np.exp(-2.0 / (1.0 - t * t)) / k

    def simpson(a, b, bw, lo):
        s = os = ost = 0.0
        for j in range(1, 41):
            if j == 1:
                s = 0.5 * (b - a) * float(integrand(np.float64(a), bw, lo) + integrand(np.float64(b), bw, lo))
            else:
                n = 1 << (j - 2)
                d = (b - a) / n
                x = np.full(n, d)
                x[0] = a + 0.5 * d
                s = 0.5 * (s + (b - a) * float(np.cumsum(integrand(np.cumsum(x), bw, lo))[-1]) / n)
            v = (4.0 * s - ost) / 3.0
            if j > 5 and (abs(v - os) < 1e-12 * abs(os) or v == os == 0.0):
                return v
            os, ost = v, s
        return v

    K, prev = np.zeros((J + 1, L)), None
    for j in range(J + 2):
        x = L / alpha ** (j - 1)
        bw = _near_int(x)
        bw = math.ceil(x) if bw is None else bw
        lo = _near_int(bw / alpha)
        lo = math.floor(bw / alpha) if lo is None else lo
        whole = simpson(lo + 1e-12, bw - 1e-12, bw, lo)
        cur = np.zeros(L)
        cur[: min(L, lo + 1)] = 1.0
        for l in range(lo + 1, min(L, bw)):
            cur[l] = simpson(float(l), bw - 1e-12, bw, lo) / whole
        if prev is not None:
            K[j - 1] = np.sqrt(np.maximum(prev - cur, 0.0))
        prev = cur
    return K, prev


def _directions(L, N):
    """S(l, n) for 0 <= n < N."""
    S = np.zeros((L, N), dtype=np.complex128)
    for l in range(1, L):
        g = min(N - 1, l - (1 if (N + l) % 2 == 0 else 0))
        for n in range(min(l, N - 1) + 1):
            if (N + n) % 2:
                r = (g - n) // 2
                c = math.comb(g, r) if 0 <= r <= g else 0
                S[l, n] = math.sqrt(c / 2.0 ** g) * (1.0 if (N - 1) % 2 == 0 else 1j)
    return S


def _wigner(L):
    """Planes d^l_{m'm}(pi/2), 0 <= m', m <= l, one l at a time, by the three-term recursion in l from its exact
    edge values."""
    m = torch.arange(L, device=DEV, dtype=torch.float64)
    big, small = torch.maximum(m[:, None], m[None, :]), torch.minimum(m[:, None], m[None, :])
    edge = 0.5 * (torch.lgamma(2 * big + 1) - torch.lgamma(big + small + 1) - torch.lgamma(big - small + 1))
    edge = torch.exp(edge - big * math.log(2.0))
    edge = torch.where((m[:, None] > m[None, :]) & (((m[:, None] - m[None, :]) % 2) == 1), -edge, edge)
    mm, pp = m[None, :], m[:, None]
    cur, last = torch.zeros_like(edge), torch.zeros_like(edge)
    for l in range(L):
        cur = torch.where(big == l, edge, cur)
        yield l, cur[: l + 1, : l + 1]
        den = torch.sqrt(torch.clamp((l + 1.0) ** 2 - mm * mm, min=1.0) * torch.clamp((l + 1.0) ** 2 - pp * pp, min=1.0))
        nxt = -(2 * l + 1.0) * pp * mm / max(l, 1) * cur
        if l:
            nxt = nxt - (l + 1.0) / l * torch.sqrt(torch.clamp(l * l - mm * mm, min=0.0)
                                                    * torch.clamp(l * l - pp * pp, min=0.0)) * last
        last, cur = cur, torch.where(big <= l, nxt / den, torch.zeros_like(cur))


def _beta_angles(h):
    k = torch.arange(h, device=DEV)[None, :] * (2 * torch.arange(2 * h, device=DEV)[:, None] + 1) % (8 * h)
    return k.to(torch.float64) * (math.pi / (4.0 * h))  # m' beta_b, [b, m']


def _mm(a, z):
    """Real (p x q) times complex (q x ...)."""
    v = torch.view_as_real(z.contiguous())
    return torch.view_as_complex((a @ v.reshape(a.shape[1], -1)).reshape(a.shape[0], *v.shape[1:]).contiguous())


def _exact_analysis(L, N, alpha, J, lim, flm):
    """Per-scale coefficients w[g, b, a] of flm[m, l]."""
    K, _ = _kernels(J, L, alpha)
    S = _directions(L, N)
    ns = [n for n in range(-(N - 1), N) if (N + n) % 2]
    T = [torch.zeros((len(ns), h, h), dtype=torch.complex128, device=DEV) for h, _ in lim]
    for l, d in _wigner(L):
        x = d * flm[: l + 1, l][None, :]
        for j, (h, lo) in enumerate(lim):
            if not lo < l < h:
                continue
            w = torch.zeros((len(ns), l + 1), dtype=torch.complex128, device=DEV)
            for i, n in enumerate(ns):
                if abs(n) > l:
                    continue
                s = K[j, l] * S[l, abs(n)]
                s = (-1) ** n * s if n < 0 else s.conjugate()
                # d^l_{m',-n} = (-1)^{l+m'} d^l_{m',n} at pi/2
                col = d[:, abs(n)]
                if n < 0:
                    col = col * torch.where((torch.arange(l + 1, device=DEV) + l) % 2 == 1, -1.0, 1.0)
                w[i] = col * complex(s)
            T[j][:, : l + 1, : l + 1].addcmul_(w[:, :, None], x[None])
    out = []
    for j, (h, _) in enumerate(lim):
        m = torch.arange(h, device=DEV)
        ph = torch.tensor([1, 1j, -1, -1j], dtype=torch.complex128, device=DEV)
        t = torch.zeros((N, h, h), dtype=torch.complex128, device=DEV)
        for i, n in enumerate(ns):
            z = T[j][i] * ph[(n - m) % 4][None, :]
            for g in range(N):
                a = math.pi * (n * g % (2 * N)) / N
                t[g] += z * complex(math.cos(a), math.sin(a))
        T[j] = None
        ang = _beta_angles(h)
        ec, es = 2.0 * torch.cos(ang), 2.0 * torch.sin(ang)
        ec[:, 0] = 1.0
        es[:, 0] = 0.0
        even = ((m + N - 1) % 2 == 0)
        w = torch.empty((N, 2 * h, 2 * h - 1), dtype=torch.float64, device=DEV)
        for g in range(N):
            c = _mm(ec, t[g])
            # the odd class carries i sin, and 1 at m' = 0
            s = _mm(es, t[g]) * 1j + t[g][0][None, :]
            w[g] = torch.fft.irfft(torch.where(even[None, :], c, s), n=2 * h - 1, dim=1, norm="forward")
        out.append(w)
    return out


def _exact_synthesis(L, N, alpha, J, lim, bl, wavs, sc):
    K, Phi2 = _kernels(J, L, alpha)
    S = _directions(L, N)
    ns = [n for n in range(N) if (N + n) % 2]
    V = []
    for j, (h, lo) in enumerate(lim):
        if lo + 1 > h - 1:
            V.append(None)
            continue
        v = torch.fft.rfft(wavs[j].reshape(N, 2 * h, 2 * h - 1), dim=2) * (4 * math.pi ** 2 / N / (2 * h - 1))
        beta = (2 * torch.arange(2 * h, device=DEV, dtype=torch.float64) + 1) * (math.pi / (4 * h))
        k = 2 * torch.arange(h, device=DEV, dtype=torch.float64) + 1
        wq = (2.0 / h) * torch.sin(beta) * (torch.sin(k[None, :] * beta[:, None]) / k[None, :]).sum(1)
        ang = _beta_angles(h).T
        c, s = torch.cos(ang), torch.sin(ang)
        m = torch.arange(h, device=DEV)
        rows = []
        for n in ns:
            u = torch.zeros((2 * h, h), dtype=torch.complex128, device=DEV)
            for g in range(N):
                a = -math.pi * (n * g % (2 * N)) / N
                u += v[g] * complex(math.cos(a), math.sin(a))
            u = u * wq[:, None]
            plus = ((m + n) % 2 == 0)[None, :]
            x, y = _mm(c, u), _mm(s, u)
            z = torch.where(plus, 2.0 * x, -2j * y)  # m' plus sign times -m'
            z[0] = x[0]
            rows.append(z)
        V.append(torch.stack(rows))
    flm = torch.zeros((L, L), dtype=torch.complex128, device=DEV)
    for l, d in _wigner(L):
        for j, (h, lo) in enumerate(lim):
            if not lo < l < h:
                continue
            for i, n in enumerate(ns):
                if n > l:
                    continue
                q = (V[j][i, : l + 1, : l + 1] * (d * d[:, n][:, None])).sum(0)
                m = torch.arange(l + 1, device=DEV)
                ph = torch.tensor([1, -1j, -1, 1j], dtype=torch.complex128, device=DEV)[(n - m) % 4]
                e = (1.0 if n == 0 else 2.0) * (2 * l + 1) / (8 * math.pi ** 2)
                flm[: l + 1, l] += q * ph * complex(e * K[j, l] * S[l, n])
    flm[:bl, :bl] += torch.from_numpy(Phi2[:bl]).to(DEV)[None, :] * sc
    return flm


def _exact_moments(wavs):
    rows = {n: [] for n in core.Plan.MOMENT_ROWS}
    for w in wavs:
        n, mean = w.numel(), w.mean()
        d = w - mean
        var = float((d * d).sum() / (n - 1))
        flat = var < 1e-12
        p = [0.0 if flat else float((d ** k).mean()) / var ** (k / 2) for k in (3, 4, 5, 6)]
        vals = [float(mean), var, p[0], 0.0 if flat else p[1] - 3.0, p[2], 0.0 if flat else p[3] - 15.0, n, float(flat)]
        for k, v in zip(rows, vals):
            rows[k].append(v)
    return {k: torch.tensor(v, dtype=torch.float64) for k, v in rows.items()}


def exact(case, seed):
    if case["path"] == "serve":
        flm, scs = [], []
        for i, (L, N) in enumerate(_serve_mix()):
            f = _flm(L, 64 * seed + i, True)
            g = _geometry(_case(None, "serve", L, N))
            # synthesis inverts analysis exactly (the m = 0 column, l < 1 of no scale, comes with scoeff)
            flm.append(f.cpu().numpy().T)
            scs.append(f[: g[2], : g[2]].cpu().numpy().T)
        return {"flm": flm, "scoeff": scs}
    L, N, alpha = case["L"], case["N"], case["alpha"]
    J, lim, bl = _geometry(case)
    if case["path"] == "synthesis":
        wav, sc = _wav(case, seed)
        sizes = [(2 * h - 1) * 2 * h * N for h, _ in lim]
        return {"flm": _exact_synthesis(L, N, alpha, J, lim, bl, torch.split(wav, sizes), sc)}
    flm = _flm(L, seed, case["red"])
    wavs = _exact_analysis(L, N, alpha, J, lim, flm)
    sc = flm[:bl, :bl].contiguous()
    if case["path"] == "moments":
        return {"scoeff": sc, **_exact_moments(wavs)}
    if case["path"] == "dropin":
        return {"wav": [w.cpu().numpy().T for w in wavs], "scoeff": sc.cpu().numpy().T, "flm": flm.cpu().numpy().T}
    return {"wav": torch.cat([w.reshape(-1) for w in wavs]), "scoeff": sc}
