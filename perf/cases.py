"""What the framework's speed is measured on: calls that its users make, through its public entry points.

``listed()`` names the cases, ``draw(rng)`` gives one more of the same ranges, ``prepare`` builds
what a program holds before the call, ``run`` is one call, ``work`` what the call cannot do
without, and ``exact`` its value by another route in 64-bit torch / numpy.

A case's ``kind`` names the entry point:

=============  =====================================================================================
``call``       ``hafnian(A, loop, method)``: one matrix, host in, number out (the drop-in)
``batch``      ``DeviceBatch``: many all-ones requests resident in HBM, one plan
``served``     ``Server.submit``: a mixed stream through the continuous-batching engine
``repeated``   ``DeviceBatch`` of ``hafnian_repeated`` requests (Fock amplitudes, density elements)
``sampler``    ``loop_hafnian_batch``: one chain-rule step of the photon-number sampler
``threshold``  ``loop_hafnian_batch_gamma``: one step of the threshold sampler (fanout rows)
``montrealer`` ``mtl`` / ``lmtl``: one cumulant
``tensor``     ``hafnian_batched``: every Fock amplitude below the cutoffs
=============  =====================================================================================
"""
import math
from collections import Counter

import numpy as np
import torch

import thewalrus_amd as tw
from thewalrus_amd._hermite_multidimensional import hafnian_batched
from thewalrus_amd.batch import DeviceBatch, prepare as prepare_matrix, prepare_repeated
from thewalrus_amd.loop_hafnian_batch import loop_hafnian_batch
from thewalrus_amd.loop_hafnian_batch_gamma import loop_hafnian_batch_gamma
from thewalrus_amd.serve import Server


# ---------------------------------------------------------------------------------- the cases
def listed():
    return [
        # the smallest request: a few-photon amplitude of a displaced state, all latency
        {"name": "call_n8_loop", "kind": "call", "n": 8, "loop": True, "real": False, "method": "glynn"},
        # one ordinary call: the 20 x 20 complex hafnian of the benchmark's first configuration
        {"name": "call_n20", "kind": "call", "n": 20, "loop": False, "real": False, "method": "glynn"},
        # an odd photon number: half of all amplitudes of a displaced state
        {"name": "call_n23_loop", "kind": "call", "n": 23, "loop": True, "real": False, "method": "glynn"},
        # the largest single call: the benchmark's third configuration
        {"name": "call_n40_loop", "kind": "call", "n": 40, "loop": True, "real": False, "method": "glynn"},
        # many real matrices of one size (perfect matchings of graphs; the second configuration,
        # a quarter of its count)
        {"name": "batch_real_n24", "kind": "batch", "count": 1024, "n": 24, "loop": False, "real": True},
        # the serving stream: even n mixed, half of them loop hafnians (the fifth configuration)
        {"name": "served_mixed", "kind": "served", "count": 96, "nmin": 8, "nmax": 30},
        # amplitudes with repeated photons: 8 modes, 32 photons (the fourth configuration)
        {"name": "repeated_8_modes", "kind": "repeated", "count": 1024, "modes": 8, "photons_min": 32,
         "photons_max": 32, "loop": True, "real": False, "glynn": True},
        # amplitudes of a wider device: 12 modes, odd and even photon numbers mixed
        {"name": "repeated_12_modes", "kind": "repeated", "count": 256, "modes": 12, "photons_min": 18,
         "photons_max": 23, "loop": True, "real": False, "glynn": True},
        # the photon-number sampler's step: 16 modes, about 1.5 photons in each, up to 12 in the next
        {"name": "sampler_16_modes", "kind": "sampler", "modes": 16, "photons": 22, "cutoff": 12},
        # the threshold sampler's step: 16 modes, 11 clicks, ten fanout rows
        {"name": "threshold_16_modes", "kind": "threshold", "modes": 16, "clicks": 11, "fanout": 10, "cutoff": 1},
        # a 14-mode cumulant of a displaced state (beyond 15 modes the alternating subset sum leaves
        # fewer digits than double precision comparisons need)
        {"name": "montrealer_14", "kind": "montrealer", "modes": 14, "loop": True, "real": False},
        # all amplitudes of 6 modes below 10 photons in each (10^6 entries)
        {"name": "tensor_6_modes", "kind": "tensor", "modes": 6, "cutoff": 10, "real": False, "renorm": True},
    ]


def draw(rng):
    kind = rng.choice(["call", "call", "batch", "served", "repeated", "repeated", "sampler", "threshold",
                       "montrealer", "tensor"])
    if kind == "call":
        loop = rng.random() < 0.5
        real = rng.random() < 0.25
        if loop and rng.random() < 0.5:
            return {"kind": kind, "n": 2 * rng.randint(3, 13) + 1, "loop": True, "real": real, "method": "glynn"}
        if not loop and rng.random() < 0.25:
            return {"kind": kind, "n": 2 * rng.randint(3, 11), "loop": False, "real": real, "method": "inclexcl"}
        return {"kind": kind, "n": 2 * rng.randint(3, 19), "loop": loop, "real": real, "method": "glynn"}
    if kind == "batch":
        n = 2 * rng.randint(4, 13)
        # counts over a logarithm, fewer of the large matrices
        most = min(2048, 2 ** (22 - n // 2))
        return {"kind": kind, "count": int(8 * (most / 8) ** rng.random()), "n": n, "loop": rng.random() < 0.5,
                "real": rng.random() < 0.5}
    if kind == "served":
        return {"kind": kind, "count": int(16 * 8 ** rng.random()), "nmin": 8, "nmax": 2 * rng.randint(8, 15)}
    if kind == "repeated":
        modes = rng.randint(4, 12)
        photons = rng.randint(8, 32 if modes <= 8 else 24)
        loop = rng.random() < 0.7
        if not loop:
            photons -= photons % 2
        return {"kind": kind, "count": int(32 * (512 / 32) ** rng.random()) + 1, "modes": modes, "photons_min": photons,
                "photons_max": photons + (rng.randint(0, 1) if loop else 0), "loop": loop,
                "real": rng.random() < 0.25, "glynn": rng.random() < 0.8}
    if kind == "sampler":
        modes = rng.randint(5, 18)
        return {"kind": kind, "modes": modes, "photons": rng.randint(2, 22), "cutoff": rng.randint(2, 12)}
    if kind == "threshold":
        modes = rng.randint(6, 20)
        return {"kind": kind, "modes": modes, "clicks": rng.randint(2, min(13, modes - 1)),
                "fanout": rng.randint(2, 10), "cutoff": 1}
    if kind == "montrealer":
        return {"kind": kind, "modes": rng.randint(4, 15), "loop": rng.random() < 0.5, "real": rng.random() < 0.25}
    modes = rng.randint(2, 6)
    top = int(round((10 ** 6) ** (1.0 / modes)))
    return {"kind": kind, "modes": modes, "cutoff": rng.randint(3, max(3, min(top, 40))), "real": rng.random() < 0.5,
            "renorm": rng.random() < 0.5}


# ------------------------------------------------------------------------------------- inputs
def _normal(r, scale2, size, real):
    if real:
        return r.normal(scale=math.sqrt(scale2), size=size)
    s = math.sqrt(scale2 / 2.0)
    return r.normal(scale=s, size=size) + 1j * r.normal(scale=s, size=size)


def _symmetric(r, n, real):
    """Entries of variance about 1/n, as the adjacency matrix of a Gaussian state has."""
    B = _normal(r, 1.0 / n, (n, n), real)
    return (B + B.T) / 2


def _inputs(case, seed):
    r = np.random.default_rng([int(seed), 20])
    kind = case["kind"]
    if kind == "call":
        return _symmetric(r, case["n"], case["real"])
    if kind == "batch":
        return [_symmetric(r, case["n"], case["real"]) for _ in range(case["count"])]
    if kind == "served":
        out = []
        for k in range(case["count"]):
            # every seed has the same sizes, in an order of its own
            n = case["nmin"] + 2 * (k // 2 % ((case["nmax"] - case["nmin"]) // 2 + 1))
            out.append((_symmetric(r, n, False), bool(k % 2)))
        return [out[i] for i in r.permutation(len(out))]
    if kind == "repeated":
        # the photon patterns belong to the case (a program asks for a list of patterns), the
        # matrices and displacements to the seed
        pat = np.random.default_rng([case["modes"], case["photons_min"], case["count"]])
        m = case["modes"]
        span = case["photons_max"] - case["photons_min"] + 1
        return [(_symmetric(r, m, case["real"]),
                 [int(x) for x in pat.multinomial(case["photons_min"] + k % span, [1.0 / m] * m)],
                 _normal(r, 1.0, m, case["real"]) if case["loop"] else None) for k in range(case["count"])]
    if kind == "sampler":
        m = case["modes"]
        pat = np.random.default_rng([m, case["photons"], case["cutoff"]])
        fixed = [int(x) for x in pat.multinomial(case["photons"], [1.0 / (m - 1)] * (m - 1))]
        return _symmetric(r, m, False), _normal(r, 1.0, m, False), fixed
    if kind == "threshold":
        m = case["modes"]
        pat = np.random.default_rng([m, case["clicks"], case["fanout"]])
        fixed = [0] * (m - 1)
        for i in pat.permutation(m - 1)[: case["clicks"]]:
            fixed[int(i)] = 1
        return _symmetric(r, m, False), _normal(r, 1.0, (case["fanout"], m), False), fixed
    if kind == "montrealer":
        m = 2 * case["modes"]
        return _symmetric(r, m, case["real"]), _normal(r, 1.0, m, case["real"]) if case["loop"] else None
    m = case["modes"]
    return 0.4 * _symmetric(r, m, case["real"]), 0.3 * _normal(r, 1.0, m, case["real"])


_server = None


def _the_server():
    """A program keeps one server for its lifetime."""
    global _server
    if _server is None:
        _server = Server()
    return _server


def prepare(case, seed):
    x = _inputs(case, seed)
    kind = case["kind"]
    state = {"case": case, "x": x}
    if kind == "batch":
        state["plan"] = DeviceBatch([prepare_matrix(A, loop=case["loop"]) for A in x])
    elif kind == "repeated":
        state["plan"] = DeviceBatch([prepare_repeated(A, rpt, mu=mu, loop=case["loop"], glynn=case["glynn"])
                                     for A, rpt, mu in x])
    elif kind == "served":
        state["server"] = _the_server()
    return state


def run(state):
    case, x, kind = state["case"], state["x"], state["case"]["kind"]
    if kind == "call":
        return tw.hafnian(x, loop=case["loop"], method=case["method"])
    if kind in ("batch", "repeated"):
        state["plan"].run()
        return state["plan"].results()
    if kind == "served":
        futures = [state["server"].submit(A, loop=loop) for A, loop in x]
        return np.array([f.result() for f in futures])
    if kind == "sampler":
        A, D, fixed = x
        return loop_hafnian_batch(A, D, fixed, case["cutoff"])
    if kind == "threshold":
        A, D, fixed = x
        return loop_hafnian_batch_gamma(A, D, fixed, case["cutoff"])
    if kind == "montrealer":
        A, zeta = x
        return tw.mtl(A) if zeta is None else tw.lmtl(A, zeta)
    A, mu = x
    return hafnian_batched(A, case["cutoff"], mu=mu, renorm=case["renorm"])


# --------------------------------------------------------------------------------- least work
def _edges(rpt):
    """Modes paired into edges: the photons sorted by how often their mode is hit, the first
    half matched with the second.  Returns ([(mode, mode)], [multiplicity], unpaired mode)."""
    photons = [i for i in sorted(range(len(rpt)), key=lambda i: -rpt[i]) for _ in range(rpt[i])]
    odd = photons.pop() if len(photons) % 2 else None
    h = len(photons) // 2
    pairs = Counter(zip(photons[:h], photons[h:]))
    return list(pairs), list(pairs.values()), odd


def _fewest_terms(rpt):
    """Edge multiplicities of a pairing with few sieve terms: the two fullest modes together, a
    mode with more than twice the next one's photons with itself.  Returns (them, odd photon left)."""
    left, mult = sorted((r for r in rpt if r), reverse=True), []
    while len(left) > 1 or (left and left[0] > 1):
        top, second = left[0], left[1] if len(left) > 1 else 0
        if top > 2 * second:
            mult.append(top // 2)
            left = [top % 2] + left[1:]
        else:
            mult.append(second)
            left = [top - second] + left[2:]
        left = sorted((r for r in left if r), reverse=True)
    return mult, bool(left)


def _sieve_flops(mult, photons, real, glynn):
    """A sieve's matrix products: half the powers of the term matrix, each power symmetric (its
    upper triangle); 8 flops for a complex multiply-add, 2 for a real one."""
    if not mult:
        return 0.0
    terms = float(np.prod([e + 1.0 for e in mult]))
    if glynn:
        terms /= 2
    side, h = 2 * len(mult), (photons + 1) // 2
    products = max(0, (h + 1) // 2 - 1)
    return terms * products * (2.0 if real else 8.0) * side * (side + 1) / 2 * side


def work(case):
    kind = case["kind"]
    cx = 16.0
    if kind == "call":
        n = case["n"]
        mult = [1] * ((n + 1) // 2)
        return {"bytes": n * n * (8.0 if case["real"] else cx) + cx,
                "flops": _sieve_flops(mult, n, case["real"], True)}
    if kind == "batch":
        n = case["n"]
        return {"bytes": case["count"] * (n * n * (8.0 if case["real"] else cx) + cx),
                "flops": case["count"] * _sieve_flops([1] * (n // 2), n, case["real"], True)}
    if kind == "served":
        reqs = _inputs(case, 0)
        return {"bytes": sum(A.shape[0] ** 2 * cx + cx for A, _ in reqs),
                "flops": sum(_sieve_flops([1] * (A.shape[0] // 2), A.shape[0], False, True) for A, _ in reqs)}
    if kind == "repeated":
        b = f = 0.0
        for A, rpt, _ in _inputs(case, 0):
            mult, odd = _fewest_terms(rpt)
            f += _sieve_flops(mult + [1] * odd, sum(rpt), case["real"], case["glynn"])
            b += A.size * cx + 2 * len(rpt) * cx + cx
        return {"bytes": b, "flops": f}
    if kind in ("sampler", "threshold"):
        A, D, fixed = _inputs(case, 0)
        mult, odd = _fewest_terms(fixed)
        mult = mult + [1] * odd + [max(1, case["cutoff"] // 2)]
        # the term matrices are the diagonals' alike
        return {"bytes": A.size * cx + D.size * cx + (case["cutoff"] + 1) * D.size / A.shape[0] * cx,
                "flops": _sieve_flops(mult, sum(fixed) + case["cutoff"], False, False)}
    if kind == "montrealer":
        n = case["modes"]
        # one power trace of every principal submatrix, by repeated squaring up to half the order
        per = max(1, math.ceil(math.log2(max(2, n))) - 1)
        f = sum(math.comb(n, s) * (2.0 * s) ** 3 for s in range(1, n + 1))
        return {"bytes": 4.0 * n * n * cx + cx, "flops": f * per * (2.0 if case["real"] else 8.0)}
    n, c = case["modes"], case["cutoff"]
    return {"bytes": n * n * cx + n * cx + float(c) ** n * (8.0 if case["real"] else cx),
            "flops": float(c) ** n * (n + 1) / 2 * (2.0 if case["real"] else 8.0)}


# -------------------------------------------------------------------------- values by another route
def _power_series(p, v, h):
    """[eta^h] exp(sum_k (p_k / 2k + v_k / 2) eta^k) for a batch of terms (lists of vectors)."""
    e = [torch.ones_like(p[1])]
    for k in range(1, h + 1):
        s = torch.zeros_like(p[1])
        for i in range(1, k + 1):
            s = s + (p[i] / 2 + i * v[i] / 2) * e[k - i]
        e.append(s / k)
    return e[h]


def _fsum(values):
    values = values.cpu().numpy()
    return complex(math.fsum(values.real.tolist()), math.fsum(values.imag.tolist()))


def _loop_hafnian(A, rpt, mu):
    """(Loop) hafnian of A with mode i repeated rpt[i] times and loop weights mu (None: no
    loops), by the finite-difference sieve over zero-padded term matrices.  An odd photon number
    is made even by one more mode that couples to nothing and carries a loop of weight 1."""
    A = np.asarray(A, dtype=np.complex128)
    rpt = list(rpt)
    if sum(rpt) == 0:
        return 1.0 + 0j
    if sum(rpt) % 2:
        if mu is None:
            return 0j
        A = np.pad(A, ((0, 1), (0, 1)))
        mu = np.append(np.asarray(mu, dtype=np.complex128), 1.0)
        rpt = rpt + [1]
    pairs, mult, _ = _edges(rpt)
    E, h = len(pairs), sum(mult)
    order = [a for a, _ in pairs] + [b for _, b in pairs]
    dev = "cuda" if torch.cuda.is_available() else "cpu"
    Ax = torch.from_numpy(A[np.ix_(order, order)].copy()).to(dev)
    swap = list(range(E, 2 * E)) + list(range(E))
    M = Ax[:, swap].contiguous()
    D = None if mu is None else torch.from_numpy(np.asarray(mu, dtype=np.complex128)[order].copy()).to(dev)
    terms = int(np.prod([e + 1 for e in mult], dtype=np.int64))
    block = max(1, min(terms, (1 << 25) // (4 * E * E)))
    total = []
    for t0 in range(0, terms, block):
        t = torch.arange(t0, min(terms, t0 + block), dtype=torch.int64, device=dev)
        sign = torch.ones(t.shape, dtype=torch.float64, device=dev)
        rest, ksum, cols = t, torch.zeros_like(t), []
        for e in mult:
            k = rest % (e + 1)
            rest = rest // (e + 1)
            ksum = ksum + k
            binom = torch.tensor([float(math.comb(e, i)) for i in range(e + 1)], dtype=torch.float64, device=dev)
            sign = sign * binom[k]
            cols.append((2 * k - e).to(torch.float64))
        sign = torch.where((h - ksum) % 2 == 0, sign, -sign)
        d = torch.stack(cols + cols, dim=1).to(torch.complex128)
        B = (M[None] * d[:, None, :]).contiguous()
        zero = torch.zeros(t.shape, dtype=torch.complex128, device=dev)
        p, v = [zero], [zero]
        P = B
        left = None if D is None else (D[swap][None] * d)[:, None, :].contiguous()
        for k in range(1, h + 1):
            p.append(torch.diagonal(P, dim1=1, dim2=2).sum(1))
            if left is not None:
                v.append((left[:, 0, :] * D).sum(1))
                left = torch.bmm(left, B)
            else:
                v.append(zero)
            if k < h:
                P = torch.bmm(P, B)
        total.append((_power_series(p, v, h) * sign).cpu())
    return _fsum(torch.cat(total)) / 2.0 ** h


def _montrealer(A, zeta):
    A = np.asarray(A, dtype=np.complex128)
    n2 = A.shape[0]
    n = n2 // 2
    dev = "cuda" if torch.cuda.is_available() else "cpu"
    S = torch.from_numpy(np.concatenate([A[n:], A[:n]])).to(dev)
    z = None if zeta is None else torch.from_numpy(np.asarray(zeta, dtype=np.complex128)).to(dev)
    total, block = [], max(1, (1 << 25) // (n2 * n2))
    for t0 in range(0, 1 << n, block):
        t = torch.arange(t0, min(1 << n, t0 + block), dtype=torch.int64, device=dev)
        on = torch.stack([(t >> i) & 1 for i in range(n)], dim=1)
        d = torch.cat([on, on], dim=1).to(torch.complex128)
        sign = torch.where((on.sum(1) + n) % 2 == 0, 1.0, -1.0).to(torch.float64)
        B = (S[None] * d[:, None, :]).contiguous()
        P = B
        for _ in range(n - 1):
            P = torch.bmm(P, B)
        f = torch.diagonal(P, dim1=1, dim2=2).sum(1) / (2 * n)
        if z is not None:
            x = (d * z)[:, :, None].contiguous()
            for _ in range(n - 1):
                x = torch.bmm(B, x)
            f = f + (d * z.conj() * x[:, :, 0]).sum(1) / 2
        total.append((f * sign).cpu())
    return _fsum(torch.cat(total))


def _tensor(A, mu, cutoff, renorm):
    """G[k] = loop hafnian with mode i repeated k_i times, axis by axis."""
    n = len(mu)
    G = np.zeros((cutoff,) * n, dtype=np.complex128)
    G[(0,) * n] = 1.0
    for i in range(n - 1, -1, -1):
        sub = G[(0,) * i]  # axes i .. n-1
        for v in range(1, cutoff):
            new = mu[i] * sub[v - 1]
            if v > 1:
                new = new + A[i, i] * (v - 1) * sub[v - 2]
            for l in range(i + 1, n):
                ax = l - i - 1
                k = np.arange(cutoff, dtype=np.float64).reshape([-1 if j == ax else 1 for j in range(n - i - 1)])
                new = new + A[i, l] * k * np.roll(sub[v - 1], 1, axis=ax)
            sub[v] = new
    if renorm:
        f = np.sqrt(np.array([float(math.factorial(k)) for k in range(cutoff)]))
        for l in range(n):
            G = G / f.reshape([-1 if j == l else 1 for j in range(n)])
    return G


def exact(case, seed):
    x = _inputs(case, seed)
    kind = case["kind"]
    if kind == "call":
        if case["n"] > 30 and not torch.cuda.is_available():
            return None
        return np.array(_loop_hafnian(x, [1] * case["n"], np.diag(x) if case["loop"] else None))
    if kind == "batch":
        return np.array([_loop_hafnian(A, [1] * case["n"], np.diag(A) if case["loop"] else None) for A in x])
    if kind == "served":
        return np.array([_loop_hafnian(A, [1] * len(A), np.diag(A) if loop else None) for A, loop in x])
    if kind == "repeated":
        return np.array([_loop_hafnian(A, rpt, mu) for A, rpt, mu in x])
    if kind == "sampler":
        A, D, fixed = x
        return np.array([_loop_hafnian(A, fixed + [q], D) for q in range(case["cutoff"] + 1)])
    if kind == "threshold":
        A, D, fixed = x
        return np.array([[_loop_hafnian(A, fixed + [q], row) for q in range(case["cutoff"] + 1)] for row in D])
    if kind == "montrealer":
        return np.array(_montrealer(*x))
    A, mu = x
    G = _tensor(A, mu, case["cutoff"], case["renorm"])
    return G.real.copy() if case["real"] else G
