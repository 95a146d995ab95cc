"""Performance cases of the field pipeline: what a program that makes initial
conditions with this package has it do, through its public entry points.

Kinds of case:

  ic         one whole realisation (ICGenerator.run): noise, phi(1..3), A(3),
             FP64 positions and velocities left in device memory
  batch      several small realisations as one captured graph (Batch)
  eulerian   a realisation with the semiclassical density and velocities
  lpt        the nLPT sources of a potential (OrszagConvolver.lpt_sources)
  convolve   the same 2LPT source through the named convolutions, as host code
             written against the reference's convolver calls them
  fft        a forward and a backward transform of a real grid
  panphasia  the white noise of a Panphasia descriptor on a grid

All work is issued on the one context (stream) that such a program keeps.
Outputs are views of the library's own device buffers.
"""
import ctypes
import math

import numpy as np
import torch

import monofonic_amd as M
from monofonic_amd import _lib

H0, OMEGA_M, OMEGA_B, N_S = 70.0, 0.3, 0.045, 0.96
DESCRIPTOR = "[Panph6,L20,({x},{y},{z}),S1,KK0,CH-999,field]"


def listed():
    return [
        # the smallest whole run: launches and latency decide
        {"name": "ic-64-2lpt-f64", "kind": "ic", "n": 64, "order": 2, "prec": "double", "gen": "MUSIC1"},
        # the FP64 production run of a small box
        {"name": "ic-256-3lpt-f64", "kind": "ic", "n": 256, "order": 3, "prec": "double", "gen": "MUSIC1"},
        # the headline run: 3LPT at 512^3 with FP32 bulk
        {"name": "ic-512-3lpt-f32", "kind": "ic", "n": 512, "order": 3, "prec": "float", "gen": "MUSIC1"},
        # a grid size that is no power of two: a box chosen by particle mass
        {"name": "ic-200-3lpt-f64", "kind": "ic", "n": 200, "order": 3, "prec": "double", "gen": "NGENIC"},
        # many small uneven boxes (training sets, covariances): throughput of one graph
        {"name": "batch-96-128-192-f32", "kind": "batch", "sizes": "96,128,192", "copies": 3, "order": 2,
         "prec": "float"},
        # the semiclassical fields of a grid code's initial conditions
        {"name": "eulerian-256-f64", "kind": "eulerian", "n": 256, "order": 2, "prec": "double"},
        # the sources alone, for host code that does its own noise and output
        {"name": "lpt-384-3lpt-f32", "kind": "lpt", "n": 384, "order": 3, "prec": "float"},
        {"name": "lpt-96-3lpt-f64", "kind": "lpt", "n": 96, "order": 3, "prec": "double"},
        # a host program that keeps the reference's call sequence
        {"name": "convolve-160-f32", "kind": "convolve", "n": 160, "prec": "float"},
        # transforms: a large cube, and a slab with unequal, non-power-of-two sides
        {"name": "fft-512-f32", "kind": "fft", "n0": 512, "n1": 512, "n2": 512, "prec": "float"},
        {"name": "fft-250x162x300-f64", "kind": "fft", "n0": 250, "n1": 162, "n2": 300, "prec": "double"},
        # a public descriptor field of a zoom parent box
        {"name": "panphasia-256-f32", "kind": "panphasia", "n": 256, "prec": "float"},
    ]


def _smooth(rng, lo, hi, step):
    """a multiple of `step`, its size spread over the logarithm, whose other
    factors are at most 7: the sizes that people choose for transforms"""
    while True:
        n = step * round(math.exp(rng.uniform(math.log(lo), math.log(hi))) / step)
        r = n
        for f in (2, 3, 5, 7):
            while r and r % f == 0:
                r //= f
        if r == 1 and lo <= n <= hi:
            return n


def draw(rng):
    kind = rng.choice(["ic", "ic", "batch", "eulerian", "lpt", "lpt", "convolve", "fft", "fft", "panphasia"])
    prec = rng.choice(["float", "double"])
    order = rng.choice([2, 3])
    if kind == "ic":
        if rng.random() < 0.5:
            return {"kind": kind, "n": rng.choice([32, 64, 128, 256]), "order": rng.choice([1, 2, 3]), "prec": prec,
                    "gen": "MUSIC1"}
        return {"kind": kind, "n": _smooth(rng, 32, 256, 4), "order": order, "prec": prec, "gen": "NGENIC"}
    if kind == "batch":
        sizes = [_smooth(rng, 32, 192, 4) for _ in range(rng.choice([2, 3]))]
        return {"kind": kind, "sizes": ",".join(map(str, sizes)), "copies": rng.choice([2, 3]), "order": order,
                "prec": prec}
    if kind == "eulerian":
        return {"kind": kind, "n": rng.choice([48, 64, 96, 128, 192, 256]), "order": rng.choice([1, 2]), "prec": prec}
    if kind == "lpt":
        return {"kind": kind, "n": _smooth(rng, 32, 384, 4), "order": order, "prec": prec}
    if kind == "convolve":
        return {"kind": kind, "n": _smooth(rng, 32, 320, 4), "prec": prec}
    if kind == "fft":
        return {"kind": kind, "n0": _smooth(rng, 16, 512, 1), "n1": _smooth(rng, 16, 512, 1),
                "n2": _smooth(rng, 16, 512, 2), "prec": prec}
    return {"kind": kind, "n": _smooth(rng, 32, 256, 4), "prec": prec}


# ---------------------------------------------------------------- the program
_ctx = None
_tuned = set()


def _context():
    """the program's one context"""
    global _ctx
    if _ctx is None:
        _ctx = M.Context(0)
    return _ctx


def _tune(n, prec):
    """the convolver's transform lengths, timed once per context (ICGenerator does this by itself)"""
    if (n, prec) not in _tuned:
        _context().autotune(n, prec)
        _tuned.add((n, prec))


class _Buffer:
    def __init__(self, ptr, shape, typestr, owner):
        self.__cuda_array_interface__ = {"data": (ptr, False), "shape": tuple(shape), "typestr": typestr,
                                         "version": 2}
        self.owner = owner  # the handle that holds the memory


def _view(ptr, shape, typestr, owner):
    return torch.as_tensor(_Buffer(ptr.value, shape, typestr, owner), device="cuda")


def _grid_view(g, space):
    """a grid's device buffer: padded real rows, or complex modes"""
    p = ctypes.c_void_p()
    _lib.call("mfx_grid_data", g.handle, ctypes.byref(p))
    n0, n1, n2 = g.n_
    real = "<f8" if g.dtype == np.float64 else "<f4"
    v = _view(p, (n0, n1, n2 + 2), real, g)
    return v if space == "real" else torch.view_as_complex(v.view(n0, n1, n2 // 2 + 1, 2))


def _particles(ic, what):
    n = ic.n
    return [_view(ic.particles_dev(w), (n, n, n), "<f8", ic) for w in what]


def _boxlen(n):
    return 2.0 * n  # 2 Mpc/h between particles


def _zstart(case):
    return 24.0 if case["kind"] != "eulerian" else 49.0


def _spectrum(n):
    """A(k) at k = kf sqrt(q), q = 0 .. 3 (n/2)^2, of a cold dark matter spectrum (the fit of Bardeen et al. 1986),
    as a caller tabulates that of any Boltzmann code"""
    k = 2 * np.pi / _boxlen(n) * np.sqrt(np.arange(3 * (n // 2) ** 2 + 1, dtype=np.float64))
    h = H0 / 100
    q = np.maximum(k, 1e-12) / (OMEGA_M * h * math.exp(-OMEGA_B * (1 + math.sqrt(2 * h) / OMEGA_M)))
    t = np.log1p(2.34 * q) / (2.34 * q) * (1 + 3.89 * q + (16.1 * q) ** 2 + (5.46 * q) ** 3 + (6.71 * q) ** 4) ** -0.25
    a = k ** (0.5 * N_S) * t
    a[0] = 0.0
    return 210.0 * a


def _noise_seed(seed, i=0):
    return 1000 + (seed * 7919 + 104729 * i) % 1000000


def _generator(case, n, seed):
    kw = {"generic_out_eulerian": True, "field_output": True} if case["kind"] == "eulerian" else {}
    return M.ICGenerator(_context(), n, _boxlen(n), _zstart(case), LPTorder=case["order"], precision=case["prec"],
                         generator=case.get("gen", "NGENIC"), seed=seed, H0=H0, Omega_m=OMEGA_M, Omega_b=OMEGA_B,
                         n_s=N_S, ZeroRadiation=True, amplitude_table=_spectrum(n), **kw)


def _device():
    return torch.device("cuda" if torch.cuda.is_available() else "cpu")


def _normal(shape, seed, i=0):
    g = torch.Generator(device=_device())
    g.manual_seed(_noise_seed(seed, i))
    return torch.randn(shape, generator=g, device=_device(), dtype=torch.float64)


def _real_dtype(case):
    return torch.float32 if case["prec"] == "float" else torch.float64


def _round(x, case):
    """complex modes rounded to the case's precision"""
    return x.to(torch.complex64 if case["prec"] == "float" else torch.complex128)


def _modes_of_noise(x):
    return torch.fft.rfftn(x) / math.sqrt(x.numel())


def _potential(case, seed):
    """phi(1) of a Gaussian realisation, as the caller's own noise gives it"""
    n = case["n"]
    return _round(_phi1(_modes_of_noise(_normal((n, n, n), seed)), n), case)


def _fft_inputs(case, seed):
    shape = (case["n0"], case["n1"], case["n2"])
    x = _normal(shape, seed).to(_real_dtype(case))
    return x, _round(_modes_of_noise(_normal(shape, seed, 1)), case)


def prepare(case, seed):
    kind, prec, ctx = case["kind"], case["prec"], _context()
    if kind in ("ic", "eulerian"):
        return {"kind": kind, "ic": _generator(dict(case, gen=case.get("gen", "MUSIC1" if _pow2(case["n"]) else
                                                                       "NGENIC")), case["n"], _noise_seed(seed))}
    if kind == "batch":
        gens = [_generator(case, int(n), _noise_seed(seed, i)) for i, n in enumerate(_batch_sizes(case))]
        return {"kind": kind, "batch": M.Batch(gens, nstreams=len(gens)),
                "seeds": [_noise_seed(seed, i) for i in range(len(gens))]}
    if kind == "panphasia":
        r = np.random.default_rng(seed).integers(0, 1 << 19, 3)
        return {"kind": kind, "grid": M.Grid_FFT(ctx, case["n"], _boxlen(case["n"]), prec),
                "noise": M.RNG_panphasia(DESCRIPTOR.format(x=r[0], y=r[1], z=r[2]))}
    if kind == "fft":
        shape = (case["n0"], case["n1"], case["n2"])
        x, k = _fft_inputs(case, seed)
        grids = [M.Grid_FFT(ctx, shape, shape, prec, initialspace=s)
                 for s in (M.rspace_id, M.rspace_id, M.kspace_id, M.kspace_id)]
        _grid_view(grids[0], "real")[:, :, :shape[2]] = x
        _grid_view(grids[2], "modes").copy_(k)
        torch.cuda.synchronize()
        return {"kind": kind, "grids": grids}
    n = case["n"]
    _tune(n, prec)
    grids = [M.Grid_FFT(ctx, n, _boxlen(n), prec, initialspace=M.kspace_id)
             for _ in range(6 if case.get("order") == 3 else 2)]
    _grid_view(grids[0], "modes").copy_(_potential(case, seed))
    torch.cuda.synchronize()
    return {"kind": kind, "grids": grids, "conv": M.OrszagConvolver(ctx, n, _boxlen(n), prec),
            "order": case.get("order", 2)}


def _pow2(n):
    return n & (n - 1) == 0


def _batch_sizes(case):
    return [n for n in case["sizes"].split(",") for _ in range(case["copies"])]


def run(state):
    kind = state["kind"]
    if kind == "ic":
        state["ic"].run()
        return _particles(state["ic"], range(6))
    if kind == "eulerian":
        state["ic"].run()
        return _particles(state["ic"], (6, 3, 4, 5))
    if kind == "batch":
        b = state["batch"]
        for g, s in zip(b.gens, state["seeds"]):
            g.set_seed(s)
        b.launch()
        return [_particles(g, range(6)) for g in b.gens]
    if kind == "panphasia":
        state["noise"].Fill_Grid(state["grid"])
        return _grid_view(state["grid"], "modes")
    if kind == "fft":
        x, xk, k, kx = state["grids"]
        xk.copy_from(x)
        xk.FourierTransformForward()
        kx.copy_from(k)
        kx.FourierTransformBackward()
        return [_grid_view(xk, "modes"), _grid_view(kx, "real")]
    conv, (phi, phi2, *rest) = state["conv"], state["grids"]
    if kind == "lpt":
        if state["order"] == 3:
            conv.lpt_sources(phi, phi2, rest[0], tuple(rest[1:]), order=3)
        else:
            conv.lpt_sources(phi, phi2, order=2)
        return [_grid_view(g, "modes") for g in state["grids"][1:]]
    op = M.op
    conv.convolve_SumOfHessians(phi, (0, 0), phi, (1, 1), (2, 2), op.assign_to(phi2))
    conv.convolve_Hessians(phi, (1, 1), phi, (2, 2), op.add_to(phi2))
    conv.convolve_Hessians(phi, (0, 1), phi, (0, 1), op.subtract_from(phi2))
    conv.convolve_Hessians(phi, (0, 2), phi, (0, 2), op.subtract_from(phi2))
    conv.convolve_Hessians(phi, (1, 2), phi, (1, 2), op.subtract_from(phi2))
    phi2.apply_InverseLaplacian()
    return [_grid_view(phi2, "modes")]


# ---------------------------------------------------------------- work
def _fft_flops(n):
    return 2.5 * n * math.log2(max(n, 2))


def _lpt_flops(n, order):
    # padded real transforms: 6 Hessian components and 1 source for 2LPT; 3LPT has those of phi(2), the four
    # intermediates both ways and four more sources
    m = (3 * n // 2) ** 3
    return (7 if order == 2 else 7 + 6 + 8 + 4) * _fft_flops(m) + 40 * m


def _ic_work(n, order, prec):
    lpt = _lpt_flops(n, order) if order > 1 else 0
    return 6 * 8 * n ** 3, lpt + 7 * _fft_flops(n ** 3) + 60 * n ** 3


def work(case):
    kind, p = case["kind"], 4 if case["prec"] == "float" else 8
    if kind == "ic":
        b, f = _ic_work(case["n"], case["order"], p)
    elif kind == "batch":
        each = [_ic_work(int(n), case["order"], p) for n in _batch_sizes(case)]
        b, f = (sum(x) for x in zip(*each))
    elif kind == "eulerian":
        n = case["n"]
        b = 4 * 8 * n ** 3
        f = (_lpt_flops(n, 2) if case["order"] > 1 else 0) + 3 * _fft_flops(n ** 3) + 14 * _fft_flops(n ** 3)
    elif kind == "panphasia":
        n = case["n"]
        # 84 coefficients for each cell of the (n/2)^3 cube, from 84 counter blocks each (Threefry, Box-Muller)
        b, f = n ** 3 * p, (n / 2) ** 3 * 84 * 200 + 84 * _fft_flops((n / 2) ** 3)
    elif kind == "fft":
        n = case["n0"] * case["n1"] * case["n2"]
        b, f = 4 * n * p, 2 * _fft_flops(n)
    else:
        n, order = case["n"], case.get("order", 2)
        b, f = (2 if order == 2 else 6) * n ** 3 * p, _lpt_flops(n, order)
    return {"bytes": b, "flops": f}


# ---------------------------------------------------------------- the same in 64 bits
def _index(n, nyquist):
    """signed mode indices; the one at n/2 kept positive, or zero as in a gradient"""
    i = torch.arange(n, device=_device(), dtype=torch.float64)
    i = torch.where(i > n // 2, i - n, i)
    if n % 2 == 0 and not nyquist:
        i[n // 2] = 0.0
    return i


def _waves(n, nyquist, half=True):
    """wave numbers along the three axes, shaped to broadcast over the modes"""
    k = 2 * math.pi / _boxlen(n) * _index(n, nyquist)
    kz = k[:n // 2 + 1] if half else k
    return k.view(n, 1, 1), k.view(1, n, 1), kz.view(1, 1, -1)


def _k2(n, half=True):
    kx, ky, kz = _waves(n, True, half)
    return kx * kx + ky * ky + kz * kz


def _over_k2(f, n):
    """-f / k^2, the k = 0 mode zero"""
    k2 = _k2(n)
    k2[0, 0, 0] = 1.0
    f = -f / k2
    f[0, 0, 0] = 0
    return f


def _phi1(modes, n):
    i = _index(n, True)
    q = (i.view(n, 1, 1) ** 2 + i.view(1, n, 1) ** 2 + i[:n // 2 + 1].view(1, 1, -1) ** 2).long()
    return _over_k2(modes * torch.from_numpy(_spectrum(n)).to(_device())[q], n)


def _to_real(f, m):
    """unnormalised inverse transform of half-spectrum modes onto m points along the last axis; the imaginary parts
    that a real field cannot have are dropped"""
    x = torch.fft.ifftn(f, dim=(0, 1), norm="forward")
    x[:, :, 0] = x[:, :, 0].real.to(x.dtype)
    if m % 2 == 0 and x.shape[2] == m // 2 + 1:
        x[:, :, -1] = x[:, :, -1].real.to(x.dtype)
    return torch.fft.irfft(x, n=m, dim=2, norm="forward")


def _positions(n):
    """where the padded grid holds the n modes along x and y"""
    i = torch.arange(n, device=_device())
    return torch.where(i > n // 2, i + n // 2, i)


class _Sources:
    """the nLPT sources with 3/2 padding (ic_generator.cc:464-547)"""

    def __init__(self, n):
        self.n, self.m, self.at = n, 3 * n // 2, _positions(n)
        self.g = _waves(n, False)

    def padded(self, f):
        p = torch.zeros(self.m, self.m, self.n // 2 + 1, dtype=torch.complex128, device=f.device)
        p[self.at[:, None], self.at[None, :]] = f
        return _to_real(p, self.m) / math.sqrt(self.n ** 3)

    def hessian(self, f):
        g = self.g
        return {a + b: self.padded(-f * g["xyz".index(a)] * g["xyz".index(b)]) for a, b in
                ("xx", "yy", "zz", "xy", "xz", "yz")}

    def truncated(self, x):
        n = self.n
        f = torch.fft.fftn(torch.fft.rfft(x, dim=2)[:, :, :n // 2 + 1], dim=(0, 1))
        f = f[self.at[:, None], self.at[None, :]] * (math.sqrt(n ** 3) / self.m ** 3)
        f[n // 2], f[:, n // 2], f[:, :, n // 2] = 0, 0, 0
        return f

    def __call__(self, phi, order):
        n, p = self.n, self.hessian(phi)
        s2 = p["xx"] * (p["yy"] + p["zz"]) + p["yy"] * p["zz"] - p["xy"] ** 2 - p["xz"] ** 2 - p["yz"] ** 2
        phi2 = _over_k2(self.truncated(s2), n)
        if order < 3:
            return [phi2]
        again = lambda x: self.padded(self.truncated(x))  # noqa: E731
        s3 = again(p["xx"] * p["yy"] - p["xy"] ** 2) * p["zz"] + 2 * again(p["xy"] * p["xz"]) * p["yz"]
        s3 -= again(p["yz"] ** 2) * p["xx"]
        s3 -= again(p["xz"] ** 2) * p["yy"]
        h = self.hessian(phi2)
        s3 -= 5 / 7 * (p["xx"] * (h["yy"] + h["zz"]) + p["yy"] * (h["xx"] + h["zz"]) + p["zz"] * (h["xx"] + h["yy"]))
        s3 += 10 / 7 * (p["xy"] * h["xy"] + p["xz"] * h["xz"] + p["yz"] * h["yz"])
        out = [phi2, _over_k2(self.truncated(s3), n)]
        of = lambda f, a, b: f["".join(sorted("xyz"[a] + "xyz"[b]))]  # noqa: E731
        for i in range(3):
            j, k = (i + 1) % 3, (i + 2) % 3
            a = of(h, i, j) * of(p, i, k) - of(h, i, k) * of(p, i, j)
            a += of(p, j, k) * (of(h, j, j) - of(h, k, k)) - of(h, j, k) * (of(p, j, j) - of(p, k, k))
            out.append(_over_k2(self.truncated(a), n))
        return out


def _growth(a):
    """D+(a) / D+(1) and f a H / h of a flat universe of matter and a cosmological constant"""
    x, w = np.polynomial.legendre.leggauss(64)

    def integral(b):  # of da / (a E)^3 from 0 to b, with a = u^2
        u = 0.5 * math.sqrt(b) * (x + 1)
        return float(np.sum(w * 2 * u ** 4 / (OMEGA_M + (1 - OMEGA_M) * u ** 6) ** 1.5)) * 0.5 * math.sqrt(b)

    e = lambda b: math.sqrt(OMEGA_M / b ** 3 + 1 - OMEGA_M)  # noqa: E731
    f = -1.5 * OMEGA_M / a ** 3 / e(a) ** 2 + a / ((a * e(a)) ** 3 * integral(a))
    return e(a) * integral(a) / integral(1.0), f * a * 100 * e(a)


def _music1(n, seed, cube=32):
    """the MUSIC1 noise: per cube one MT19937 stream through Leva's ratio method"""
    cube = min(cube, n)
    nc, want = n // cube, cube ** 3
    out = np.empty((nc, nc, nc, cube, cube, cube))
    for c in range(nc ** 3):
        words = np.random.RandomState(seed + c)
        got, have = [], 0
        while have < want:
            u = np.frombuffer(words.bytes(4 * 624 * (2 * (want - have) // 400 + 2)), "<u4") / 4294967296.0
            s, t = 1 - u[0::2], (u[1::2] - 0.5) * 1.7156
            px, py = s - 0.449871, np.abs(t) + 0.386595
            q = px * px + py * (0.196 * py - 0.25472 * px)
            ok = q < 0.27597
            edge = np.flatnonzero(~ok & (q <= 0.27846))
            ok[edge] = t[edge] ** 2 <= -4 * s[edge] ** 2 * np.log(s[edge])
            got.append(t[ok] / s[ok])
            have += len(got[-1])
        out[c // nc ** 2, c // nc % nc, c % nc] = np.concatenate(got)[:want].reshape(cube, cube, cube)
    return torch.from_numpy(out.transpose(0, 3, 1, 4, 2, 5).reshape(n, n, n)).to(_device())


class _Ranlux:
    """ranlxd1 streams side by side: one per column of the state"""

    def __init__(self, seeds):
        seeds = np.where(seeds == 0, 1, seeds).astype(np.int64)
        bit = [(seeds >> k) & 1 for k in range(31)]
        i, j, self.x = 0, 18, []
        for _ in range(12):
            x = np.zeros(len(seeds), np.int64)
            for _ in range(48):
                x = 2 * x + (1 - bit[i])
                bit[i] = bit[i] ^ bit[j]
                i, j = (i + 1) % 31, (j + 1) % 31
            self.x.append(torch.from_numpy(x).to(_device() if len(seeds) > 1 else "cpu"))
        if len(seeds) == 1:  # a single stream is quicker in plain integers
            self.x = [int(x) for x in self.x]
        self.carry, self.ir, self.jr, self.end = 0 * self.x[0], 11, 7, 0

    def __call__(self):
        """the next draw of each stream, times 2^48"""
        self.ir = (self.ir + 1) % 12
        if self.ir == self.end:
            for _ in range(202):
                y = self.x[self.jr] - self.x[self.ir] - self.carry
                self.carry = (y >> 48) & 1
                self.x[self.ir] = y & ((1 << 48) - 1)
                self.ir, self.jr = (self.ir + 1) % 12, (self.jr + 1) % 12
            self.end = self.ir
        return self.x[self.ir]


def _ngenic(n, seed):
    """the NGenIC noise, drawn mode by mode from one stream per (x, y) column"""
    one, table = _Ranlux(np.array([seed])), np.zeros((n, n), np.int64)
    draws = lambda count: [int(0x7fffffff * (one() / 2.0 ** 48)) for _ in range(count)]  # noqa: E731
    for i in range(n // 2):
        r = n - 1 - i
        table[i, :i] = draws(i)
        table[:i + 1, i] = draws(i + 1)
        table[r, :i] = draws(i)
        table[n - 1 - np.arange(i + 1), i] = draws(i + 1)
        table[i, n - 1 - np.arange(i)] = draws(i)
        table[:i + 1, r] = draws(i + 1)
        table[r, n - 1 - np.arange(i)] = draws(i)
        table[n - 1 - np.arange(i + 1), r] = draws(i + 1)
    streams = _Ranlux(table.reshape(-1))
    f = torch.zeros(n, n, n // 2 + 1, dtype=torch.complex128, device=_device())
    for k in range(n // 2 + 1):
        phase, ampl = (streams().double() / 2.0 ** 48 for _ in range(2))
        f[:, :, k] = torch.polar(torch.sqrt(-torch.log(ampl)), 2 * math.pi * phase).view(n, n)
    f[n // 2], f[:, n // 2], f[:, :, n // 2] = 0, 0, 0
    # kz = 0: the lower half plane holds the conjugates
    h, back = n // 2, torch.remainder(-torch.arange(n, device=_device()), n)
    z = f[:, :, 0].clone()
    mirror = z[back][:, back].conj()
    f[h + 1:, :, 0] = mirror[h + 1:]
    f[0, h + 1:, 0] = mirror[0, h + 1:]
    f[0, 0, 0] = 0
    return f


def _ic_potentials(case, n, gen, seed):
    volfac = (_boxlen(n) / n / 2 / math.pi) ** 1.5
    noise = _modes_of_noise(_music1(n, seed)) if gen == "MUSIC1" else _ngenic(n, seed)
    phi = _phi1(noise / volfac, n)
    return phi, _Sources(n)(phi, case["order"]) if case["order"] > 1 else []


def _exact_ic(case, n, gen, seed):
    order, D_vfact = case["order"], _growth(1 / (1 + _zstart(case)))
    D, vfact = D_vfact
    phi, rest = _ic_potentials(case, n, gen, seed)
    terms = [-D * phi] + ([-3 / 7 * D * D * rest[0]] if order > 1 else [])
    terms += [D ** 3 / 3 * rest[1]] if order > 2 else []
    A = [D ** 3 / 7 * a for a in rest[2:]]
    del phi, rest
    g, q, out = _waves(n, False), torch.arange(n, device=_device(), dtype=torch.float64) / n, []
    for kind in range(2):
        pot = sum(t * ((o + 1) * vfact if kind else 1) for o, t in enumerate(terms))
        for d in range(3):
            j, k = (d + 1) % 3, (d + 2) % 3
            f = g[d] * pot
            if A:
                f = f + (3 * vfact if kind else 1) * (g[j] * A[k] - g[k] * A[j])
            x = _to_real(1j * f, n) / (math.sqrt(n ** 3) * _boxlen(n))
            out.append(x if kind else x + q.view([n if a == d else 1 for a in range(3)]))
    return out


def _exact_eulerian(case, seed):
    n = case["n"]
    D, vfact = _growth(1 / (1 + _zstart(case)))
    phi, rest = _ic_potentials(case, n, "MUSIC1" if _pow2(n) else "NGENIC", seed)
    phi = _to_real(-D * phi, n) / math.sqrt(n ** 3)
    phi2 = _to_real(-3 / 7 * D * D * rest[0], n) / math.sqrt(n ** 3) if rest else torch.zeros_like(phi)
    steps = [(phi.roll(-1, a) - phi)[:n - 1].abs().max() for a in range(3)]
    hbar = float(max(steps)) / math.pi / D * 1.01
    k = _waves(n, True, half=False)
    psi = torch.exp(1j * (phi + phi2) / (hbar * D))
    psi = torch.fft.ifftn(torch.fft.fftn(psi) * torch.exp(-0.5j * hbar * D * _k2(n, half=False)))
    if rest:
        psi = psi * torch.exp(1j * phi2 / (hbar * D))
    rho = psi.real ** 2 + psi.imag ** 2
    f, out = torch.fft.fftn(psi), [rho - 1]
    for d in range(3):
        out.append(D * vfact / _boxlen(n) * hbar * (psi.conj() * torch.fft.ifftn(1j * k[d] * f)).imag / rho)
    return out


def exact(case, seed):
    kind = case["kind"]
    if kind == "ic":
        return _exact_ic(case, case["n"], case["gen"], _noise_seed(seed))
    if kind == "batch":
        return [_exact_ic(case, int(n), "NGENIC", _noise_seed(seed, i)) for i, n in enumerate(_batch_sizes(case))]
    if kind == "eulerian":
        return _exact_eulerian(case, _noise_seed(seed))
    if kind == "fft":
        x, k = (t.to(torch.float64) if t.is_floating_point() else t.to(torch.complex128)
                for t in _fft_inputs(case, seed))
        norm = math.sqrt(x.numel())
        return [torch.fft.rfftn(x) / norm, torch.nn.functional.pad(_to_real(k, case["n2"]) / norm, (0, 2))]
    if kind in ("lpt", "convolve"):
        return _Sources(case["n"])(_potential(case, seed).to(torch.complex128), case.get("order", 2))
    return None  # the octree field of a descriptor has no short restatement
