"""The work that programs have this library do, as measurable cases.

A case names a kind of system, its grid and the steps of one call.  `run`
advances the prepared system (or batch) by those steps and takes the device
spectra of its fields, as a program does that goes on with its own kernels
(analysis, structure factors, output) every few steps.  Every following pass
advances the same state further.

`exact` steps the same equations in 64 bits with torch.fft on full complex
arrays: constraint fields first, then the dynamic fields, each updated field
made real again, dealiased copies of the product factors (zero before a
field's first update), noise from the documented Philox streams.
"""
import ctypes
import math

import numpy as np
import torch

import cupss_amd as C

# ------------------------------------------------------------------ systems
#
# A system: fields (name, dynamic), implicit operators, terms (field, factors,
# prefactors), noise amplitudes; a prefactor is (c, q2n, iqx, iqy, iqz, invq):
# c q^(2 q2n) (i qx)^iqx (i qy)^iqy (i qz)^iqz |q|^-invq.


def _diffusion(rng):
    d = float(rng.uniform(0.5, 1.5))
    return dict(dt=0.01, fields=[("phi", True)], implicit={"phi": [(-d, 1)]}, terms=[("phi", [], [(0.0,)])])


def _cahn_hilliard(rng, noise=False):
    s = dict(dt=0.01, fields=[("phi", True)], implicit={"phi": [(1.0, 1), (-1.0, 2)]},
             terms=[("phi", ["phi"] * 3, [(-1.0, 1)])])
    if noise:  # conserved noise: amplitude 2 D q^2
        s["noise"] = {"phi": (0.02, 1)}
    return s


def _kpz(rng, ndim, linear=False):
    nu = float(rng.uniform(0.5, 2.0))
    lam = 0.0 if linear else float(rng.uniform(0.5, 2.0))
    axes = ["x", "y", "z"][:ndim]
    fields, terms = [("h", True)], []
    for a, ax in enumerate(axes):
        fields.append(("d" + ax, False))
        terms.append(("h", ["d" + ax] * 2, [(0.5 * lam,)]) if lam else ("h", [], [(0.0,)]))
    if not lam:
        terms = terms[:1]
    for a, ax in enumerate(axes):
        p = [1.0, 0, 0, 0, 0]
        p[2 + a] = 1
        terms.append(("d" + ax, ["h"], [tuple(p)]))
    return dict(dt=0.005, fields=fields, implicit={"h": [(-nu, 1)]}, terms=terms, noise={"h": (0.02,)})


def _model_h(rng):
    ka = -4.0
    terms = [("phi", ["phi"] * 3, [(-1.0, 1)]), ("phi", ["dx", "vx"], [(-1.0,)]), ("phi", ["dy", "vy"], [(-1.0,)]),
             ("dx", ["phi"], [(1.0, 0, 1)]), ("dy", ["phi"], [(1.0, 0, 0, 1)]),
             ("sxx", ["dx", "dx"], [(-0.5 * ka,)]), ("sxx", ["dy", "dy"], [(0.5 * ka,)]),
             ("sxy", ["dx", "dy"], [(-ka,)]),
             ("vx", ["sxx"], [(1.0, 0, 1), (1.0, 0, 3, 0, 0, 2), (-1.0, 0, 1, 2, 0, 2)]),
             ("vx", ["sxy"], [(1.0, 0, 0, 1), (1.0, 0, 2, 1, 0, 2), (1.0, 0, 2, 1, 0, 2)]),
             ("vy", ["sxy"], [(1.0, 0, 1), (1.0, 0, 1, 2, 0, 2), (1.0, 0, 1, 2, 0, 2)]),
             ("vy", ["sxx"], [(-1.0, 0, 0, 1), (-1.0, 0, 0, 3, 0, 2), (1.0, 0, 2, 1, 0, 2)]),
             ("w", ["vy"], [(0.5, 0, 1)]), ("w", ["vx"], [(-0.5, 0, 0, 1)])]
    fields = [("phi", True)] + [(n, False) for n in ("dx", "dy", "sxx", "sxy", "vx", "vy", "w")]
    return dict(dt=0.01, fields=fields, implicit={"phi": [(1.0, 1), (-4.0, 2)], "vx": [(1.0, 1)], "vy": [(1.0, 1)]},
                terms=terms)


def _gray_scott(rng):
    F, k = 0.035, 0.065
    return dict(dt=0.5, fields=[("u", True), ("v", True)], implicit={"u": [(-0.16, 1)], "v": [(-0.08, 1)]},
                terms=[("u", ["u", "v", "v"], [(-1.0,)]), ("u", [], [(F,)]), ("u", ["u"], [(-F,)]),
                       ("v", ["u", "v", "v"], [(1.0,)]), ("v", ["v"], [(-(F + k),)])])


def _uniform(rng, n, lo, hi):
    return rng.random(n, dtype=np.float32) * np.float32(hi - lo) + np.float32(lo)


def _system(kind, dims, rng):
    """The equations and the starting real fields of one system."""
    n = dims[0] * dims[1] * dims[2]
    ndim = 1 + (dims[1] > 1) + (dims[2] > 1)
    if kind == "diffusion":
        s = _diffusion(rng)
        init = {"phi": _uniform(rng, n, 0.0, 1.0)}
    elif kind in ("ch", "chnoise"):
        s = _cahn_hilliard(rng, kind == "chnoise")
        init = {"phi": _uniform(rng, n, -0.1, 0.1)}
    elif kind in ("kpz", "ew"):
        s = _kpz(rng, ndim, kind == "ew")
        init = {"h": np.zeros(n, np.float32)}
    elif kind == "modelh":
        s = _model_h(rng)
        init = {"phi": _uniform(rng, n, -0.1, 0.1)}
    else:
        s = _gray_scott(rng)
        u = np.ones((dims[1], dims[0]), np.float32)
        v = np.zeros((dims[1], dims[0]), np.float32)
        mid = tuple(slice(m // 2 - m // 8, m // 2 + m // 8) for m in (dims[1], dims[0]))
        u[mid], v[mid] = 0.5, 0.25
        init = {"u": u.ravel() + _uniform(rng, n, -0.02, 0.02), "v": v.ravel() + _uniform(rng, n, -0.02, 0.02)}
    s["dims"], s["init"], s["seed"] = dims, init, int(rng.integers(1, 1 << 40))
    return s


def _members(case):
    """(kind, dims) of every member of a case; a single system is one member."""
    if case["kind"] == "ensemble":  # Edwards-Wilkinson and KPZ instances of mixed sides, half and half
        sides = [64, 128, 256, 512][:case["sides"]]
        return [("kpz" if (i // len(sides)) % 2 else "ew", (sides[i % len(sides)],) * 2 + (1,))
                for i in range(case["members"])]
    if case["kind"] == "modelh_mix":  # the jobs a server holds at once
        sides = [128, 256, 512, 1024][:case["sides"]]
        return [("modelh", (sides[i % len(sides)],) * 2 + (1,)) for i in range(case["members"])]
    return [(case["kind"], (case["sx"], case["sy"], case["sz"]))]


def _all_systems(case, seed):
    rng = np.random.default_rng(seed)
    return [_system(kind, dims, rng) for kind, dims in _members(case)]


# ------------------------------------------------------------------ cases


def _single(name, kind, dims, steps, noise="real"):
    return {"name": name, "kind": kind, "sx": dims[0], "sy": dims[1], "sz": dims[2], "steps": steps, "noise": noise}


def listed():
    return [
        # the C++ advanceTime() loop of a light linear system: one step per call, all latency
        _single("diffusion_256_one_step", "diffusion", (256, 256, 1), 1),
        # growth of a line interface, the smallest of the noisy systems
        _single("kpz_line_1024", "kpz", (1024, 1, 1), 100),
        # one small noisy interface alone, with the default draw
        _single("kpz_128", "kpz", (128, 128, 1), 100),
        # phase separation at an everyday size and at the benchmark's
        _single("ch_256", "ch", (256, 256, 1), 100),
        _single("ch_1024", "ch", (1024, 1024, 1), 100),
        # phase separation in a box
        _single("ch3d_256", "ch", (256, 256, 256), 11),
        # model B with its conserved noise in a box, the default draw
        _single("chnoise3d_128", "chnoise", (128, 128, 128), 20),
        # binary fluid: many constraint fields, many products
        _single("modelh_1024", "modelh", (1024, 1024, 1), 50),
        # two reacting species on a rectangle
        _single("grayscott_1024x512", "grayscott", (1024, 512, 1), 50),
        # the resident jobs of a serving run, advanced together by the server's default quantum
        {"name": "modelh_mix", "kind": "modelh_mix", "members": 8, "sides": 4, "steps": 100, "noise": "real"},
        # a parameter sweep with the default noise draw
        {"name": "sweep_48", "kind": "ensemble", "members": 48, "sides": 4, "steps": 20, "noise": "real"},
        # the benchmark's ensemble: 512 instances, noise drawn in spectral space
        {"name": "ensemble_512", "kind": "ensemble", "members": 512, "sides": 4, "steps": 20, "noise": "spectral"},
    ]


def draw(rng):
    kind = rng.choice(["diffusion", "kpz", "ch", "ch3d", "chnoise3d", "modelh", "grayscott", "modelh_mix", "ensemble",
                       "line"])

    def side(lo, hi):  # a power of two
        return 1 << rng.randint(int(math.log2(lo)), int(math.log2(hi)))

    noise = rng.choice(["real", "spectral"])
    steps = int(round(math.exp(rng.uniform(math.log(5), math.log(100)))))
    if kind == "line":
        c = _single("", "kpz", (side(64, 4096), 1, 1), steps)
    elif kind == "ch3d":
        c = _single("", "ch", (side(32, 256), side(32, 256), side(32, 256)), 1 + steps // 12)
    elif kind == "chnoise3d":
        c = _single("", "chnoise", (side(32, 128), side(32, 128), side(32, 128)), 1 + steps // 6, noise)
    elif kind == "modelh_mix":
        c = {"kind": kind, "members": rng.randint(2, 12), "sides": rng.randint(1, 3), "steps": steps, "noise": "real"}
    elif kind == "ensemble":
        c = {"kind": kind, "members": rng.randint(8, 200), "sides": rng.randint(1, 4), "steps": 5 + steps // 5,
             "noise": noise}
    elif kind == "diffusion":
        c = _single("", kind, (side(64, 2048), side(64, 2048), 1), rng.randint(1, 9))
    elif kind == "kpz":
        c = _single("", kind, (side(32, 1024), side(32, 1024), 1), steps, noise)
    elif kind == "ch":
        c = _single("", kind, (side(32, 2048), side(32, 1024), 1), steps)
    elif kind == "modelh":
        c = _single("", kind, (side(64, 1024), side(64, 1024), 1), 1 + steps // 2)
    else:
        c = _single("", kind, (side(64, 1024), side(64, 1024), 1), 1 + steps // 2)
    c.pop("name", None)
    return c


def work(case):
    """Per step: each dynamic field's spectrum read and written once (8 B a
    point), one real transform per dealiased factor, product sum and
    real-space noise draw (2.5 n log2 n operations), ten operations a point.
    A system without products advances all its steps on one read and write."""
    nbytes = flops = 0.0
    for kind, dims in _members(case):
        n = float(dims[0] * dims[1] * dims[2])
        ndim = 1 + (dims[1] > 1) + (dims[2] > 1)
        dyn = 2 if kind == "grayscott" else 1
        nt = {"diffusion": 0, "ew": 0, "kpz": ndim + 1, "ch": 2, "chnoise": 2, "modelh": 9, "grayscott": 3}[kind]
        if kind in ("ew", "kpz", "chnoise") and case["noise"] == "real":
            nt += 1
        nbytes += 8.0 * n * dyn * (case["steps"] if nt else 1)
        flops += case["steps"] * (nt * 2.5 * n * math.log2(n) + 10.0 * n * dyn)
    return {"bytes": nbytes, "flops": flops}


# ------------------------------------------------------------------ running


class _Span:
    """A device span of a system as an array (torch.as_tensor reads it, and
    holds it, so the system lives as long as the tensor)."""

    def __init__(self, system, ptr, shape):
        self.system = system
        self.__cuda_array_interface__ = {"shape": shape, "typestr": "<f4", "data": (ptr, False), "version": 2,
                                         "strides": None}


class _Fields:
    """The device spectra of some fields of a system, by (pointer, shape)."""

    def __init__(self, system, ids):
        self.system, self.ids, self.seen = system, ids, {}
        sx, sy, sz = system.dims
        self.shape = (sz, sy, sx // 2 + 1, 2)

    def now(self):
        got, p = [], ctypes.c_void_p()
        for f in self.ids:
            C.check(self.system.L.cupss_field_spectrum_device(self.system.h, f, ctypes.byref(p)))
            t = self.seen.get(p.value)
            if t is None:
                t = self.seen[p.value] = torch.as_tensor(_Span(self.system, p.value, self.shape), device="cuda")
            got.append(t)
        return got


_stream = None


def _program_stream():
    """The one stream of the program: the library's work and torch's on its
    results are in order without waiting."""
    global _stream
    if _stream is None:
        _stream = torch.cuda.Stream()
    return _stream


class _StreamBatch(C.Batch):
    """A batch on the caller's stream."""

    def __init__(self, stream, graph_steps):
        self.L, self.h, self.members = C.lib(), ctypes.c_void_p(), []
        C.check(self.L.cupss_batch_create(ctypes.c_void_p(stream.cuda_stream), ctypes.byref(self.h)))
        C.check(self.L.cupss_batch_set_graph_steps(self.h, graph_steps))


def _build(spec, noise):
    sx, sy, sz = spec["dims"]
    s = C.System(sx, sy, sz, 1.0, 1.0, 1.0, spec["dt"])
    ids = {name: s.add_field(dyn) for name, dyn in spec["fields"]}
    for name, plist in spec["implicit"].items():
        for p in plist:
            s.add_implicit(ids[name], C.pres(*p))
    for name, factors, plist in spec["terms"]:
        s.add_term(ids[name], [ids[f] for f in factors], [C.pres(*p) for p in plist])
    for name, p in spec.get("noise", {}).items():
        s.set_noise(ids[name], C.pres(*p), spec["seed"])
    for name, x in spec["init"].items():
        s.set_real(ids[name], x)
    if noise == "spectral":
        s.set_noise_mode(1)
    C.check(s.L.cupss_system_set_stream(s.h, ctypes.c_void_p(_program_stream().cuda_stream)))
    s.prepare()
    return s, ids


def prepare(case, seed):
    specs = _all_systems(case, seed)
    built = [_build(spec, case["noise"]) for spec in specs]
    if "members" not in case:
        s, ids = built[0]
        return {"system": s, "steps": case["steps"], "fields": _Fields(s, list(ids.values()))}
    stream = _program_stream()
    batch = _StreamBatch(stream, graph_steps=20)
    dyn, sides = [], {}
    for spec, (s, ids) in zip(specs, built):
        batch.add(s)
        dyn.append(_Fields(s, [ids[name] for name, d in spec["fields"] if d]))
        sides.setdefault(spec["dims"][0], []).append(len(dyn) - 1)
    return {"batch": batch, "steps": case["steps"], "fields": dyn, "sides": sides, "stream": stream}


def run(state):
    if "system" in state:
        state["system"].step(state["steps"])
        return state["fields"].now()
    state["batch"].step(state["steps"])
    with torch.cuda.stream(state["stream"]):
        return {str(n): torch.cat([t for i in members for t in state["fields"][i].now()])
                for n, members in state["sides"].items()}


# ------------------------------------------------------------------ 64 bits


def _philox(c, key, rounds=10):
    """Philox4x32-10 of int64 counter and key arrays holding 32-bit words."""
    m32 = 0xFFFFFFFF
    k0, k1 = key

    def mulhilo(a, b):  # a: 32-bit constant, b: 32-bit words
        p, q = a * (b & 0xFFFF), a * (b >> 16)  # below 2^48
        s = p + ((q & 0xFFFF) << 16)
        return ((q >> 16) + (s >> 32)) & m32, s & m32

    for _ in range(rounds):
        h0, l0 = mulhilo(0xD2511F53, c[0])
        h1, l1 = mulhilo(0xCD9E8D57, c[2])
        c = [h1 ^ c[1] ^ k0, l1, h0 ^ c[3] ^ k1, l0]
        k0, k1 = (k0 + 0x9E3779B9) & m32, (k1 + 0xBB67AE85) & m32
    return c


def _normal_pairs(o):
    """The two Box-Muller pairs of a Philox output."""
    u = [(2 * (x >> 9) + 1).double() * 2.0 ** -24 for x in o]
    got = []
    for a, b in ((u[0], u[1]), (u[2], u[3])):
        r = torch.sqrt(-2.0 * torch.log(a))
        got.append((r * torch.cos(2 * math.pi * b), r * torch.sin(2 * math.pi * b)))
    return got


def _noise_hat(dims, mode, seeds, step, stream):
    """The full transforms of one step's noise fields, one for each seed."""
    sx, sy, sz = dims
    n, m, dev = sx * sy * sz, len(seeds), seeds.device
    key = ((seeds & 0xFFFFFFFF)[:, None], (seeds >> 32)[:, None])
    if mode == "real":
        c = torch.arange((n + 3) // 4, device=dev).expand(m, -1)
        z = torch.zeros_like(c)
        (a0, a1), (b0, b1) = _normal_pairs(_philox([c, z + step, z, z + stream], key))
        return _fft(torch.stack([a0, a1, b0, b1], -1).reshape(m, -1)[:, :n].reshape(m, sz, sy, sx))
    nc, hy = sx // 2, sy // 2 if sy >= 2 else 1
    c = torch.arange(sz * (nc + 1) * hy, device=dev).expand(m, -1)  # (kz, kx, j)
    z = torch.zeros_like(c)
    pairs = _normal_pairs(_philox([c, z + step, z, z + (stream | 0x80000000)], key))
    v = torch.cat([torch.complex(*p).reshape(m, sz, nc + 1, hy) for p in (pairs if sy >= 2 else pairs[:1])], -1)
    v = v.transpose(2, 3).contiguous()  # (kz, ky, kx)
    iz, iy = torch.meshgrid(torch.arange(sz, device=dev), torch.arange(sy, device=dev), indexing="ij")
    pz, py = (sz - iz) % sz, (sy - iy) % sy
    own, partner = iz * sy + iy, pz * sy + py
    full = torch.zeros(m, sz, sy, sx, dtype=torch.complex128, device=dev)
    full[..., :nc + 1] = v * math.sqrt(0.5 * n)
    for k in (0, nc):  # the planes that hold both partners
        e = v[..., k]
        full[..., k] = torch.where(partner == own, (e.real * math.sqrt(n)).to(e.dtype),
                                   torch.where(partner < own, e[:, pz, py].conj(), e) * math.sqrt(0.5 * n))
    full[..., nc + 1:] = full[:, pz, py][..., 1:nc].flip(-1).conj()
    return full


def _fft(x):
    return torch.fft.fftn(x, dim=(-3, -2, -1))


def _ifft_real(x):
    return torch.fft.ifftn(x, dim=(-3, -2, -1)).real


def _f32(x):
    return float(np.float32(x))


def _exact_systems(specs, steps, noise, dev):
    """The half spectra of every field of like systems (same fields, terms
    and grid), stacked, after `steps` steps."""
    first = specs[0]
    sx, sy, sz = dims = first["dims"]
    m, n = len(specs), sx * sy * sz
    shape = (m, sz, sy, sx)
    pi = np.float32(3.1415926535)

    def axis(s):  # wave numbers and |mode| of an axis
        k = torch.arange(s, device=dev)
        step = float(np.float32(2.0) * pi / np.float32(s))
        return torch.where(k < (s + 1) // 2, k, k - s).double() * step, torch.where(k > s // 2, k - s, k).abs()

    (qz, mz), (qy, my), (qx, mx) = axis(sz), axis(sy), axis(sx)
    qz, qy, qx = qz[:, None, None], qy[None, :, None], qx[None, None, :]
    q2 = qx * qx + qy * qy + qz * qz
    iq = torch.where(q2 > 0, 1.0 / torch.sqrt(q2), torch.zeros_like(q2))

    def multiplier(lists):  # of each system's prefactor list
        total = 0
        for ps in zip(*lists):
            _, q2n, a, b, cz, invq = (tuple(ps[0]) + (0,) * 6)[:6]
            f = torch.tensor([_f32(p[0]) for p in ps], dtype=torch.complex128, device=dev)[:, None, None, None]
            for q, k in ((q2, q2n), (1j * qx, a), (1j * qy, b), (1j * qz, cz), (iq, invq)):
                for _ in range(k):
                    f = f * q
            total = total + f
        return total

    mult = [multiplier([s["terms"][t][2] for s in specs]) for t in range(len(first["terms"]))]
    imp = {name: multiplier([s["implicit"][name] for s in specs]).real for name in first["implicit"]}
    dt = _f32(first["dt"])
    order = {}
    for _, factors, _ in first["terms"]:
        if len(factors) >= 2:
            for f in factors:
                order[f] = max(order.get(f, 0), len(factors))
    keep = {f: (mz <= sz // (p + 1))[:, None, None] & (my <= sy // (p + 1))[None, :, None] &
            (mx <= sx // (p + 1))[None, None, :] for f, p in order.items()}
    hat = {name: torch.zeros(shape, dtype=torch.complex128, device=dev) for name, _ in first["fields"]}
    for name in first["init"]:
        x = np.stack([s["init"][name] for s in specs])
        hat[name] = _fft(torch.from_numpy(x).to(dev).double().reshape(shape))
    real = {f: torch.zeros(shape, dtype=torch.float64, device=dev) for f in order}
    seeds = torch.tensor([s["seed"] for s in specs], device=dev)
    amp = {name: math.sqrt(dt * _f32(p[0])) * torch.sqrt(q2) ** (p[1] if len(p) > 1 else 0)
           for name, p in first.get("noise", {}).items()}
    for step in range(steps):
        for dynamic in (False, True):
            new = {}
            for i, (name, dyn) in enumerate(first["fields"]):
                if dyn != dynamic:
                    continue
                acc = torch.zeros_like(hat[name])
                for (target, factors, _), f in zip(first["terms"], mult):
                    if target != name:
                        continue
                    if len(factors) >= 2:
                        prod = real[factors[0]]
                        for g in factors[1:]:
                            prod = prod * real[g]
                        acc += f * _fft(prod)
                    elif factors:
                        acc += f * hat[factors[0]]
                    else:
                        acc[:, 0, 0, 0] += f[:, 0, 0, 0] * n
                if dyn:
                    acc = hat[name] + dt * acc
                    if name in amp:
                        acc += amp[name] * _noise_hat(dims, noise, seeds, step, i)
                    if name in imp:
                        acc /= 1.0 - dt * imp[name]
                elif name in imp:
                    acc = torch.where(q2 > 0, acc / torch.where(q2 > 0, imp[name], torch.ones_like(q2)), acc)
                new[name] = _fft(_ifft_real(acc))
            for name, s in new.items():
                hat[name] = s
                if name in order:
                    real[name] = _ifft_real(torch.where(keep[name], s, torch.zeros_like(s)))
    return {name: torch.view_as_real(h[..., :sx // 2 + 1].contiguous()).cpu() for name, h in hat.items()}


def exact(case, seed):
    dev = "cuda" if torch.cuda.is_available() else "cpu"
    specs, like = _all_systems(case, seed), {}
    for i, (spec, member) in enumerate(zip(specs, _members(case))):
        like.setdefault(member, []).append(i)
    got = [None] * len(specs)
    for members in like.values():
        both = _exact_systems([specs[i] for i in members], case["steps"], case["noise"], dev)
        for j, i in enumerate(members):
            got[i] = {name: h[j] for name, h in both.items()}
    if "members" not in case:
        return [got[0][name] for name, _ in specs[0]["fields"]]
    sides = {}
    for spec, g in zip(specs, got):
        sides.setdefault(str(spec["dims"][0]), []).extend(g[name] for name, d in spec["fields"] if d)
    return {n: torch.cat(v) for n, v in sides.items()}
