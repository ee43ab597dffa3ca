"""The work that users of this package have it do, as cases that can be timed.

listed() are the workloads of this repository's configurations, tests and
benchmark: HMC trajectories from 8^4 to 48^3 x 96 in both storage types and
with both integrator forms, the Wilson action's forward / backward pair,
checkerboard Metropolis, heat-bath and overrelaxation sweeps, the field
strength, batched chains and the projected momentum refresh.  draw() gives one
more of the same ranges, odd and ragged extents among them.

prepare() makes the lattice from a seed, run() is one pass through the public
entry points, exact() restates that pass in 64-bit torch from the same seed
(the Philox4x32-10 streams of Salmon et al., SC'11, included).

Passes on a lattice return the gradient of the Wilson action of the links they
leave behind (n_links x 8, on the GPU): the form in which the updated links
reach a program that keeps working on the device.  FP32 lattices give it in
FP32, the precision that its values have there.
"""
import math
import os
import sys

import numpy as np
import torch

sys.path.insert(1, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "lattice-qcd-rs_amd"))
import lqcd  # noqa: E402

F = lqcd._ffi
F32, F64 = lqcd.F32, lqcd.F64
ADDITIVE, EXP = lqcd.DRIFT_ADDITIVE, lqcd.DRIFT_EXP
REFERENCE, LEAPFROG = lqcd.SCHEME_REFERENCE, lqcd.SCHEME_LEAPFROG


# ------------------------------------------------------------------- cases

def _hmc(name, extents, precision, integrator, steps, dt, beta):
    c = {"kind": "hmc", "extents": extents, "precision": precision, "integrator": integrator, "steps": steps,
         "dt": dt, "beta": beta}
    return dict(c, name=name) if name else c


def _lattice(name, kind, extents, precision, beta):
    c = {"kind": kind, "extents": extents, "precision": precision, "beta": beta}
    return dict(c, name=name) if name else c


def listed():
    return [
        # a test-sized lattice: a trajectory is many launches of a few waves each
        _hmc("hmc_8x4_f64", "8x8x8x8", "f64", "reference", 20, 0.01, 6.0),
        # the reference's own integrator form (kick-drift-kick, additive drift) at a common size
        _hmc("hmc_16x4_f64", "16x16x16x16", "f64", "reference", 20, 0.01, 5.7),
        # odd, ragged extents: no power of two, no whole rows per wavefront
        _hmc("hmc_15x13x11x17_f64", "15x13x11x17", "f64", "leapfrog", 20, 0.02, 6.0),
        # the headline trajectory in both storage types
        _hmc("hmc_32x4_f32", "32x32x32x32", "f32", "leapfrog", 40, 0.025, 6.0),
        _hmc("hmc_32x4_f64", "32x32x32x32", "f64", "leapfrog", 40, 0.025, 6.0),
        # the largest configured lattice
        _hmc("hmc_48x3x96_f32", "48x48x48x96", "f32", "leapfrog", 50, 0.02, 6.2),
        # action and gradient, as a program that drives its own integrator asks for them
        _lattice("pair_16x4_f64", "pair", "16x16x16x16", "f64", 5.7),
        # D = 3 Metropolis sweeps of a large lattice
        _lattice("metropolis_128x3_f64", "metropolis", "128x128x128", "f64", 6.0),
        # a quenched update of a thermalised lattice: heat bath, normalisation, four overrelaxation sweeps
        _lattice("quenched_32x4_f64", "quenched", "32x32x32x32", "f64", 6.0),
        # F_mu_nu of every site, kept on the GPU for the observables built on it
        _lattice("field_32x4_f32", "field", "32x32x32x32", "f32", 6.0),
        # many independent chains of four sizes, one trajectory of each
        {"name": "batched_64_f32", "kind": "batched", "sizes": "8,12,16,20", "per_size": 16, "precision": "f32",
         "steps": 20, "dt": 0.01},
        # momenta drawn, projected on Gauss's law and read back (the start of a user's own integration)
        _lattice("refresh_16x4_f64", "refresh", "16x16x16x16", "f64", 6.0),
    ]


def _draw_extents(rng, d, low, high, even=False):
    """d extents whose volume is spread over its logarithm from low^d to high^d, each its own."""
    side = math.exp(rng.uniform(math.log(low), math.log(high)))
    ext = []
    for _ in range(d):
        x = int(round(side * math.exp(rng.uniform(-0.3, 0.3))))
        x = min(max(x, low), high)
        ext.append(min(high, x + x % 2) if even else x)
    return "x".join(str(x) for x in ext)


def draw(rng):
    kind = rng.choice(["hmc"] * 5 + ["pair", "metropolis", "quenched", "field", "batched", "refresh"])
    prec = rng.choice(["f32", "f64"])
    beta = round(rng.uniform(5.5, 6.2), 3)
    if kind == "hmc":
        d, low, high = rng.choice([(4, 5, 32), (4, 5, 32), (4, 5, 32), (3, 8, 96)])
        return _hmc(None, _draw_extents(rng, d, low, high), prec, rng.choice(["leapfrog", "reference"]),
                    rng.randint(10, 40), round(rng.uniform(0.01, 0.025), 4), beta)
    if kind == "batched":
        sizes = sorted(rng.sample(range(4, 21, 2), 3))
        return {"kind": "batched", "sizes": ",".join(map(str, sizes)), "per_size": rng.randint(1, 16),
                "precision": prec, "steps": rng.randint(10, 20), "dt": round(rng.uniform(0.01, 0.02), 4)}
    if kind == "metropolis":
        d, low, high = rng.choice([(3, 8, 128), (4, 6, 32)])
        return _lattice(None, kind, _draw_extents(rng, d, low, high, even=True), prec, beta)
    if kind == "quenched":
        return _lattice(None, kind, _draw_extents(rng, 4, 6, 32, even=True), prec, beta)
    if kind == "refresh":
        return _lattice(None, kind, _draw_extents(rng, 4, 5, 20), prec, beta)
    return _lattice(None, kind, _draw_extents(rng, 4, 6, 32), prec, beta)


def _extents(case):
    return [int(x) for x in case["extents"].split("x")]


def _precision(case):
    return F32 if case["precision"] == "f32" else F64


def _chains(case, seed):
    """The chains of a batched case: beta rises from 5.6 to 6.2 over them, each has its own seed."""
    sizes = [int(x) for x in case["sizes"].split(",")]
    n = len(sizes) * case["per_size"]
    return [(sizes[k // case["per_size"]], 5.6 + 0.6 * k / max(1, n - 1), seed * 1000 + k) for k in range(n)]


# --------------------------------------------------------------------- run

# heat-bath sweeps from the cold start before a quenched update
_THERMALISE = 4


class _Gradient:
    """A torch tensor where the package takes a device buffer."""

    def __init__(self, shape):
        self.tensor = torch.empty(shape, dtype=torch.float64, device="cuda")
        self.nbytes, self.ptr = self.tensor.numel() * 8, self.tensor.data_ptr()


def prepare(case, seed):
    s = {"case": case, "kind": case["kind"]}
    if case["kind"] == "batched":
        specs = [lqcd.ChainSpec([n] * 4, b, k) for n, b, k in _chains(case, seed)]
        s["chains"] = lqcd.BatchedChains(specs, 4, _precision(case))
        s["chains"].hot_start()
        return s
    ext = _extents(case)
    if case["kind"] == "quenched":
        st = lqcd.LatticeStateDefault.new_cold(1.0, case["beta"], ext, len(ext), _precision(case))
    else:
        st = lqcd.LatticeStateDefault.new_determinist(1.0, case["beta"], ext, seed, len(ext), _precision(case))
    s["state"] = st
    n = st.lattice().number_of_canonical_links_space()
    if case["kind"] == "field":
        s["out"] = torch.empty((n // len(ext), len(ext), len(ext), 3, 3, 2), dtype=torch.float64, device="cuda")
    elif case["kind"] == "refresh":
        s["seed"] = seed
    else:
        s["gradient"] = _Gradient((n, 8))
    if case["kind"] == "hmc":
        form = (EXP, LEAPFROG) if case["integrator"] == "leapfrog" else (ADDITIVE, REFERENCE)
        s["update"] = lqcd.HybridMonteCarloDiagnostic(case["dt"], case["steps"], lqcd.SymplecticEulerGpu(*form), seed,
                                                      project_gauss=False)
    elif case["kind"] == "metropolis":
        s["update"] = lqcd.MetropolisHastingsSweep(1, 0.1, seed)
    elif case["kind"] == "quenched":
        s["update"] = lqcd.HeatBathSweep(seed)
        s["relax"] = lqcd.OverrelaxationSweepRotation()
        for _ in range(_THERMALISE):
            st.monte_carlo_step(s["update"])
            st.normalize_link_matrices()
    torch.cuda.synchronize()
    return s


def _gradient(s):
    """The gradient at the state's links.  An FP32 one is a conversion on
    torch's stream: it has to be done with the buffer before the package,
    which has a stream of its own, writes there again."""
    g = s["gradient"]
    if s["case"]["precision"] == "f64":
        return s["state"].wilson_backward_device(g).tensor
    torch.cuda.current_stream().synchronize()
    return s["state"].wilson_backward_device(g).tensor.to(torch.float32)


def run(s):
    kind, case = s["kind"], s["case"]
    if kind == "batched":
        b = s["chains"]
        stats = b.hmc(case["dt"], case["steps"], 1, reunitarize=True)[0]
        real = np.float32 if case["precision"] == "f32" else np.float64
        return {"h_old": stats["h_old"].astype(real), "h_new": stats["h_new"].astype(real),
                "plaquette": stats["plaquette"].astype(real), "accepted": stats["accepted"].copy(),
                "links_first": b.link_matrix(0).astype(real)}
    st = s["state"]
    if kind == "pair":
        return {"action": st.wilson_forward(), "gradient": _gradient(s)}
    if kind == "field":
        out = s["out"]
        lqcd._raise(F.lib().lqcd_field_strength_device(st.handle, F.FIELD_F_MU_NU, out.data_ptr(), out.numel()))
        return {"field": out}
    if kind == "refresh":
        ef = lqcd.LatticeStateEFSyncDefault.new_random_e_state(st, s["seed"])
        return {"e_field": ef.e_field().astype(np.float32 if case["precision"] == "f32" else np.float64, copy=False)}
    u = s["update"]
    st.monte_carlo_step(u)
    if kind == "metropolis":
        return {"probability": u.prob_replace_mean(), "replaced": u.number_replace_last(), "gradient": _gradient(s)}
    st.normalize_link_matrices()
    if kind == "quenched":
        for _ in range(4):
            st.monte_carlo_step(s["relax"])
        return {"exhausted": u.exhausted_last(), "plaquette": st.average_trace_plaquette().real / 3.0,
                "gradient": _gradient(s)}
    return {"h_old": u.last_stats.h_old, "h_new": u.last_stats.h_new, "accepted": int(u.has_replace_last()),
            "plaquette": st.average_trace_plaquette().real / 3.0, "gradient": _gradient(s)}


# -------------------------------------------------------------------- work

# multiply-adds of two flops each, per link: a product of 3x3 complex matrices is 108 of them
_PRODUCT = 216


def _md_work(nlink, d, real, steps, exp):
    # per link and step: links and momenta read and written once (a link of SU(3) is 12
    # reals); per site the products of the shared staples, per link U Sigma and the drift
    reals = 40 if exp else 52
    force = (d - 1) * 2 * _PRODUCT * 23 / 24 + _PRODUCT
    return {"bytes": steps * nlink * reals * real, "flops": steps * nlink * (force + (5 if exp else 1) * _PRODUCT)}


def work(case):
    real = 4 if case["precision"] == "f32" else 8
    if case["kind"] == "batched":
        links = sum(4 * n ** 4 for n, _, _ in _chains(case, 0))
        return _md_work(links, 4, real, case["steps"], True)
    ext = _extents(case)
    d, nsite = len(ext), math.prod(_extents(case))
    nlink = nsite * d
    gradient = {"bytes": nlink * (18 * real + 64), "flops": nlink * ((d - 1) * 2 * _PRODUCT + _PRODUCT)}
    if case["kind"] == "hmc":
        w = _md_work(nlink, d, real, case["steps"], case["integrator"] == "leapfrog")
    elif case["kind"] == "pair":
        w = {"bytes": 0, "flops": nlink * (d - 1) / 2 * 2.2 * _PRODUCT}
    elif case["kind"] in ("metropolis", "quenched"):
        # a sweep is 2 D classes; each reads the links of its staples and writes its own
        sweeps = 1 if case["kind"] == "metropolis" else 5
        w = {"bytes": sweeps * nlink * (2 * d * 12 + 18) * real, "flops": sweeps * nlink * ((d - 1) * 4 + 5) * _PRODUCT}
    elif case["kind"] == "field":
        return {"bytes": nsite * (18 * d * real + d * d * 144), "flops": nsite * d * (d - 1) / 2 * 12 * _PRODUCT}
    else:
        # about thirty checks of four steps, each over E (held in 64 bits) and the links
        return {"bytes": 120 * nlink * (18 * real + 128), "flops": 120 * nlink * 4 * _PRODUCT}
    return {"bytes": w["bytes"] + gradient["bytes"], "flops": w["flops"] + gradient["flops"]}


# ------------------------------------------------- the same in 64-bit torch

_M = 0xFFFFFFFF


def _device():
    return "cuda" if torch.cuda.is_available() else "cpu"


def _philox(link, block, n, seed):
    """Philox4x32-10 of link's counter {lo32(l), hi16(l) | block << 16, lo32(n), hi32(n)}, key seed."""
    c = [link & _M, ((link >> 32) & 0xFFFF) | (block << 16), torch.full_like(link, n & _M),
         torch.full_like(link, (n >> 32) & _M)]
    k = [seed & _M, (seed >> 32) & _M]
    for _ in range(10):
        p0, p1 = c[0] * 0xD2511F53, c[2] * 0xCD9E8D57
        c = [((p1 >> 32) & _M) ^ c[1] ^ k[0], p1 & _M, ((p0 >> 32) & _M) ^ c[3] ^ k[1], p0 & _M]
        k = [(k[0] + 0x9E3779B9) & _M, (k[1] + 0xBB67AE85) & _M]
    return c


def _uniforms(link, blocks, n, seed):
    """Two 53-bit uniforms of [0, 1) from each block."""
    out = []
    for b in blocks:
        o = _philox(link, b, n, seed)
        out += [(((o[i] >> 5) << 26) | (o[i + 1] >> 6)).double() * 2.0 ** -53 for i in (0, 2)]
    return out


def _mm(a, b):
    return sum(a[..., :, k:k + 1] * b[..., k:k + 1, :] for k in range(3))


def _dag(a):
    return a.conj().transpose(-1, -2)


def _tr(a):
    return a[..., 0, 0] + a[..., 1, 1] + a[..., 2, 2]


def _normalized(m):
    """Gram-Schmidt of the columns; the third is the conjugated cross product."""
    a, b = m[..., :, 0], m[..., :, 1]
    a = a / torch.linalg.vector_norm(a, dim=-1, keepdim=True)
    b = b - a * (a.conj() * b).sum(-1, keepdim=True)
    b = b / torch.linalg.vector_norm(b, dim=-1, keepdim=True)
    return torch.stack([a, b, torch.cross(a.conj(), b.conj(), dim=-1)], -1)


class _Lattice:
    """Links u[mu] of shape (L_{D-1}, .., L_0, 3, 3), sites in storage order."""

    def __init__(self, ext, precision, seed):
        self.ext, self.d, self.f32, self.seed = ext, len(ext), precision == "f32", seed
        site = torch.arange(math.prod(ext), device=_device()).reshape(ext[::-1])
        self.index = [site * self.d + mu for mu in range(self.d)]
        self.u = [self.stored(self.hot(l)) for l in self.index]

    def cold(self):
        self.u = [torch.eye(3, dtype=torch.complex128, device=_device()).expand_as(x).clone() for x in self.u]

    def normalize(self):
        self.u = [self.stored(_normalized(x)) for x in self.u]

    def stored(self, x):
        return x.to(torch.complex64).to(torch.complex128) if self.f32 else x

    def hot(self, link):
        w = [2.0 * x - 1.0 for x in _uniforms(link, range(16, 22), 0, self.seed)]
        v = [torch.complex(w[2 * i], w[2 * i + 1]) for i in range(6)]
        col = [torch.stack(v[:3], -1), torch.stack(v[3:], -1)]
        return _normalized(torch.stack([col[0], col[1], col[1]], -1))

    def momenta(self, n, seed, sigma):
        out = []
        for link in self.index:
            w = _uniforms(link, range(4), n, seed)
            e = []
            for j in range(4):
                rad = torch.sqrt(-2.0 * torch.log(1.0 - w[2 * j])) * sigma
                e += [rad * torch.cos(2.0 * math.pi * w[2 * j + 1]), rad * torch.sin(2.0 * math.pi * w[2 * j + 1])]
            e = torch.stack(e, -1)
            out.append(e.float().double() if self.f32 else e)
        return out

    def up(self, x, mu, k=1):
        """x at the site k steps along mu."""
        return torch.roll(x, -k, self.d - 1 - mu)

    def staple(self, mu):
        """Sum of U_nu(x+mu) U_mu(x+nu)^+ U_nu(x)^+ and its mirror images."""
        u, out = self.u, 0
        for nu in range(self.d):
            if nu != mu:
                out = out + _mm(_mm(self.up(u[nu], mu), _dag(self.up(u[mu], nu))), _dag(u[nu]))
                low = _mm(_dag(_mm(u[mu], self.up(u[nu], mu))), u[nu])
                out = out + self.up(low, nu, -1)
        return out

    def force(self):
        """Im Tr(T^a U Sigma) for every link."""
        return [_projections(_mm(self.u[mu], self.staple(mu))) for mu in range(self.d)]

    def gradient(self, beta):
        # dS / dw^a = (beta / 3) Im Tr(T^a U Sigma), links in storage order
        return torch.stack(self.force(), -2).reshape(-1, 8) * (beta / 3.0)

    def plaquettes(self):
        """Sum of Re Tr P over the plaquettes, and how many there are."""
        total, n = 0.0, 0
        for i in range(self.d):
            for j in range(i + 1, self.d):
                a, b = _mm(self.u[i], self.up(self.u[j], i)), _mm(self.u[j], self.up(self.u[i], j))
                total += float((a * b.conj()).sum().real)
                n += self.index[0].numel()
        return total, n

    def energy(self, beta, e=None):
        total, n = self.plaquettes()
        return beta * (n - total / 3.0) + (beta * 0.5 * sum(float((x * x).sum()) for x in e) if e else 0.0)

    def mean_plaquette(self):
        total, n = self.plaquettes()
        return total / n / 3.0

    def parity(self):
        grid = torch.meshgrid(*[torch.arange(n, device=_device()) for n in self.ext[::-1]], indexing="ij")
        return sum(grid) % 2

    def classes(self):
        p = self.parity()
        for mu in range(self.d):
            for par in range(2):
                yield mu, p == par


def _projections(m):
    r3 = 1.0 / (2.0 * math.sqrt(3.0))
    re, im = m.real, m.imag
    return torch.stack([(im[..., 0, 1] + im[..., 1, 0]) / 2, (re[..., 0, 1] - re[..., 1, 0]) / 2,
                        (im[..., 0, 0] - im[..., 1, 1]) / 2, (im[..., 0, 2] + im[..., 2, 0]) / 2,
                        (re[..., 0, 2] - re[..., 2, 0]) / 2, (im[..., 1, 2] + im[..., 2, 1]) / 2,
                        (re[..., 1, 2] - re[..., 2, 1]) / 2,
                        r3 * (im[..., 0, 0] + im[..., 1, 1] - 2 * im[..., 2, 2])], -1)


def _hermitian(e):
    """sum_a e^a T^a (T^a = Gell-Mann / 2)."""
    r3 = 1.0 / (2.0 * math.sqrt(3.0))
    c = [e[..., a] / 2 for a in range(7)] + [e[..., 7] * r3]
    z = torch.zeros_like(c[0])
    rows = [[torch.complex(c[2] + c[7], z), torch.complex(c[0], -c[1]), torch.complex(c[3], -c[4])],
            [torch.complex(c[0], c[1]), torch.complex(c[7] - c[2], z), torch.complex(c[5], -c[6])],
            [torch.complex(c[3], c[4]), torch.complex(c[5], c[6]), torch.complex(-2 * c[7], z)]]
    return torch.stack([torch.stack(r, -1) for r in rows], -2)


def _exp_times(x, u):
    """exp(x) u, summed to where 64 bits end for |x| < 1."""
    out = term = u
    for k in range(1, 20):
        term = _mm(x, term) / k
        out = out + term
    return out


def _trajectory(lat, e, case):
    """steps of the case's integrator from the momenta e."""
    dt, n, exp = case["dt"], case["steps"], case.get("integrator", "leapfrog") == "leapfrog"
    kick = -math.sqrt(2.0 / 3.0)
    for k in range(n):
        f = lat.force()
        # the half kicks of neighbouring steps see the same links
        e = [x + (0.5 if k == 0 else 1.0) * dt * kick * y for x, y in zip(e, f)]
        for mu in range(lat.d):
            x = 1j * dt * math.sqrt(6.0) * _hermitian(e[mu])
            lat.u[mu] = _exp_times(x, lat.u[mu]) if exp else lat.u[mu] + _mm(x, lat.u[mu])
    return [x + 0.5 * dt * kick * y for x, y in zip(e, lat.force())]


def _splitmix64(x):
    m = (1 << 64) - 1
    z = (x + 0x9E3779B97F4A7C15) & m
    z = ((z ^ (z >> 30)) * 0xBF58476D1CE4E5B9) & m
    z = ((z ^ (z >> 27)) * 0x94D049BB133111EB) & m
    return z ^ (z >> 31)


def _step(lat, case, beta, seed, word):
    """A trajectory with its accept decision: H before and after, whether it was accepted."""
    e = lat.momenta(0, seed, 0.5 / beta)
    before, h_old = list(lat.u), lat.energy(beta, e)
    e = _trajectory(lat, e, case)
    h_new = lat.energy(beta, e)
    accepted = h_new <= h_old or word < math.exp(h_old - h_new) * 2.0 ** 64
    if not accepted:
        lat.u = before
    return h_old, h_new, int(accepted)


def _host_links(lat):
    """The links in the host layout: column-major matrices, re and im interleaved."""
    u = torch.stack(lat.u, -3).transpose(-1, -2).reshape(-1, 9)
    return torch.view_as_real(u.contiguous()).reshape(-1, 18)


def _exact_batched(case, seed):
    rows, first = [], None
    for n, beta, k in _chains(case, seed):
        lat = _Lattice([n] * 4, case["precision"], k)
        one = torch.zeros(1, dtype=torch.int64, device=_device())
        o = _philox(one, 62, 0, k)
        rows.append(_step(lat, case, beta, k, (int(o[0]) << 32) | int(o[1])))
        rows[-1] += (lat.mean_plaquette(),)
        if first is None:
            lat.u = [_normalized(x) for x in lat.u]
            first = _host_links(lat).cpu().numpy()
    cols = [np.array(c) for c in zip(*rows)]
    return {"h_old": cols[0], "h_new": cols[1], "plaquette": cols[3], "accepted": cols[2].astype(np.int32),
            "links_first": first}


def _su2_near_one(w, spread):
    r = [2.0 * x - 1.0 for x in w[:3]]
    n = torch.sqrt(r[0] ** 2 + r[1] ** 2 + r[2] ** 2)
    x = [v / n * spread for v in r]
    x0 = torch.sqrt(1.0 - (x[0] ** 2 + x[1] ** 2 + x[2] ** 2))
    return _quaternion(torch.where(w[3] < 0.5, x0, -x0), x)


def _quaternion(x0, x):
    """x0 + i x . sigma in the reference's form, whose sigma_3 is the identity."""
    return [torch.complex(x0, x[2]), torch.complex(x[1], x[0]), torch.complex(-x[1], x[0]), torch.complex(x0, x[2])]


_BLOCKS = ((0, 1), (0, 2), (1, 2))


def _embed(m, rows):
    """The 2x2 matrix m (row-major list) in the given rows and columns of the identity."""
    out = torch.zeros(m[0].shape + (3, 3), dtype=torch.complex128, device=m[0].device)
    i, j = rows
    k = 3 - i - j
    out[..., k, k] = 1.0
    out[..., i, i], out[..., i, j], out[..., j, i], out[..., j, j] = m
    return out


def _metropolis(lat, beta, seed, spread):
    p_sum, replaced = 0.0, 0
    for mu, mask in lat.classes():
        a, u, link = lat.staple(mu)[mask], lat.u[mu][mask], lat.index[mu][mask]
        w = _uniforms(link, range(64, 71), 0, seed)
        r = _embed(_su2_near_one(w[0:4], spread), _BLOCKS[0])
        r = _mm(r, _embed(_su2_near_one(w[4:8], spread), _BLOCKS[1]))
        r = _mm(r, _embed(_su2_near_one(w[8:12], spread), _BLOCKS[2]))
        r = torch.where((w[12] < 0.5)[..., None, None], _dag(r), r)
        new = _mm(_normalized(r), u)
        ds = -(((new - u) * a.transpose(-1, -2)).sum((-1, -2))).real * beta / 3.0
        p = torch.exp(-ds).clamp(0.0, 1.0)
        o = _philox(link, 63, 0, seed)
        # the word's leading 53 bits decide
        ok = (p >= 1.0) | (((o[0] << 21) | (o[1] >> 11)).double() * 2.0 ** -53 < p)
        lat.u[mu][mask] = lat.stored(torch.where(ok[..., None, None], new, u))
        p_sum += float(p.sum())
        replaced += int(ok.sum())
    return p_sum / (lat.d * lat.index[0].numel()), replaced


def _heat_bath_su2(st, beta, link, group, seed, counter):
    base = 0x8000 + 256 * group
    k = torch.sqrt((st[0] * st[3] - st[1] * st[2]).real)
    x0, todo = torch.zeros_like(k), torch.ones_like(k, dtype=torch.bool)
    for t in range(64):
        w = _uniforms(link, (base + 2 * t, base + 2 * t + 1), counter, seed)
        c = torch.cos(2.0 * math.pi * (1.0 - w[2]))
        lam2 = -(torch.log(1.0 - w[1]) + c * c * torch.log(1.0 - w[3])) / (2.0 * beta * k)
        ok = todo & (w[0] * w[0] <= 1.0 - lam2)
        x0 = torch.where(ok, 1.0 - 2.0 * lam2, x0)
        todo = todo & ~ok
        if not bool(todo.any()):
            break
    w = _uniforms(link, (base + 128, base + 129), counter, seed)
    x = [2.0 * v - 1.0 for v in w[:3]]
    scale = torch.sqrt(1.0 - x0 * x0) / torch.sqrt(x[0] ** 2 + x[1] ** 2 + x[2] ** 2)
    q = _quaternion(x0, [v * scale for v in x])
    v = [st[0].conj() / k, st[2].conj() / k, st[1].conj() / k, st[3].conj() / k]
    out = [q[0] * v[0] + q[1] * v[2], q[0] * v[1] + q[1] * v[3], q[2] * v[0] + q[3] * v[2], q[2] * v[1] + q[3] * v[3]]
    one = [1.0, 0.0, 0.0, 1.0]
    return [torch.where(todo, torch.full_like(z, i), z) for z, i in zip(out, one)], int(todo.sum())


def _heat_bath(lat, beta, seed, counter):
    exhausted = 0
    for mu, mask in lat.classes():
        a, u, link = lat.staple(mu)[mask], lat.u[mu][mask], lat.index[mu][mask]
        for group, (i, j) in enumerate(_BLOCKS):
            w = _mm(u, a)
            m = [w[..., i, i], w[..., i, j], w[..., j, i], w[..., j, j]]
            tr = (m[0] + m[3]).conj()
            su2 = [tr, m[1] - m[2].conj(), m[2] - m[1].conj(), tr]
            su2[0], su2[3] = tr + m[0] - m[0].conj(), tr + m[3] - m[3].conj()
            f, n = _heat_bath_su2(su2, beta, link, group, seed, counter)
            u = _mm(_embed(f, (i, j)), u)
            exhausted += n
        lat.u[mu][mask] = lat.stored(u)
    return exhausted


def _adjugate(m):
    r = [m[..., k, :] for k in range(3)]
    return torch.stack([torch.cross(r[1], r[2], dim=-1), torch.cross(r[2], r[0], dim=-1),
                        torch.cross(r[0], r[1], dim=-1)], -1)


def _polar(m):
    """The unitary factor of m, by Newton's iteration scaled with the determinant."""
    for _ in range(30):
        adj = _adjugate(m)
        det = (m[..., 0, :] * adj[..., :, 0]).sum(-1)[..., None, None]
        g = det.abs() ** (-1.0 / 3.0)
        new = 0.5 * (g * m + _dag(adj / det) / g)
        done = float((new - m).abs().max()) < 1e-15
        m = new
        if done:
            break
    return m


def _overrelax(lat):
    for mu, mask in lat.classes():
        rot = _polar(_dag(lat.staple(mu)[mask]))
        lat.u[mu][mask] = lat.stored(_mm(_mm(rot, _dag(lat.u[mu][mask])), rot))


def _field_strength(lat):
    d, zero = lat.d, torch.zeros_like(lat.u[0])
    out = [[zero] * d for _ in range(d)]

    def link(y, mu, sign):
        """Links along +-mu of the field y (a link field), at every site."""
        return y if sign > 0 else _dag(lat.up(y, mu, -1))

    for i in range(d):
        for j in range(i + 1, d):
            c = 0
            for (a, sa), (b, sb) in (((i, 1), (j, 1)), ((j, 1), (i, -1)), ((i, -1), (j, -1)), ((j, -1), (i, 1))):
                ua, ub = link(lat.u[a], a, sa), link(lat.u[b], b, sb)
                # P_ab = U_a(x) U_b(x+a) U_a(x+b)^+ U_b(x)^+
                c = c + _mm(_mm(ua, lat.up(ub, a, sa)), _dag(_mm(ub, lat.up(ua, b, sb))))
            out[i][j] = (c - _dag(c)) / 8.0
            out[j][i] = -out[i][j]
    f = torch.stack([torch.stack(r, -3) for r in out], -4).transpose(-1, -2)
    return torch.view_as_real(f.contiguous()).reshape(-1, d, d, 3, 3, 2)


def _gauss(lat, e):
    g = 0
    for i in range(lat.d):
        h = _hermitian(e[i])
        g = g + h - lat.up(_mm(_mm(_dag(lat.u[i]), h), lat.u[i]), i, -1)
    return g


def _projected(lat, e):
    """The Gauss projection: a step, then four more while the deviation is above its threshold."""
    threshold = 2.220446049250313e-16 * lat.index[0].numel() * 320
    sums = torch.ones(8, dtype=torch.float64, device=_device())
    total = _hermitian(sums)

    def step(e):
        g = _gauss(lat, e)
        return [x + 2.0 * 0.12 * _projections(1j * (_mm(_mm(_mm(u, g), _dag(u)), lat.up(g, i)) - g))
                for i, (x, u) in enumerate(zip(e, lat.u))]

    e = step(e)
    for _ in range(1000):
        if float((total * _gauss(lat, e).transpose(-1, -2)).sum((-1, -2)).abs().sum()) <= threshold:
            return e
        for _ in range(4):
            e = step(e)
    return None


def exact(case, seed):
    kind = case["kind"]
    if kind == "batched":
        return _exact_batched(case, seed)
    ext = _extents(case)
    if math.prod(ext) > 1 << 21:
        return None  # minutes in plain torch
    lat, beta = _Lattice(ext, case["precision"], seed), case["beta"]
    if kind == "pair":
        return {"action": lat.energy(beta), "gradient": lat.gradient(beta)}
    if kind == "field":
        return {"field": _field_strength(lat)}
    if kind == "refresh":
        e = _projected(lat, lat.momenta(0, seed, 0.5 / beta))
        return e and {"e_field": torch.stack(e, -2).reshape(-1, 8).cpu().numpy()}
    if kind == "metropolis":
        p, n = _metropolis(lat, beta, seed, 0.1)
        return {"probability": p, "replaced": n, "gradient": lat.gradient(beta)}
    if kind == "quenched":
        lat.cold()
        for k in range(_THERMALISE + 1):
            n = _heat_bath(lat, beta, seed, k)
            lat.normalize()
        for _ in range(4):
            _overrelax(lat)
        return {"exhausted": n, "plaquette": lat.mean_plaquette(), "gradient": lat.gradient(beta)}
    h_old, h_new, accepted = _step(lat, case, beta, seed, _splitmix64(seed))
    lat.u = [_normalized(x) for x in lat.u]
    return {"h_old": h_old, "h_new": h_new, "accepted": accepted, "plaquette": lat.mean_plaquette(),
            "gradient": lat.gradient(beta)}
