"""The work that users of this framework have it do, as timed cases.

A case is one pass through a public entry point on one view of the plane:

* ``"frame"``: a whole frame on device buffers (``GpuContext.tile_device``),
  the path of the benchmark and of programs that keep results on the GPU;
* ``"tile"``: one tile of ``settings.chunk_size`` pixels a side through
  ``Fractal.compute_tile``, host arrays in and out, as a tiled renderer calls
  it (the reference's per-tile call);
* ``"layers"``: the continuous-iteration, distance-estimate and normal-map
  layers of a finished frame (``fsg_postproc_device``);
* ``"serve"``: a burst of mixed tile requests through ``TileServer``.

The views are the seeded locations of ``fractalshades_amd.configs`` (the
benchmark's), at their own width and at wider ones.  Every state is a
slightly panned view of its location, iterated around the location's own
reference orbit, as a user's next frame of the same place is; the device
context (derivative paths, BLA table) is made anew for each.
"""
import functools
import math
import random
import types

import numpy as np
import torch

from fractalshades_amd import _native, configs, serving, settings
from fractalshades_amd.postproc import post_desc

DEVICE = "cuda:0"

# A view: seeded location, width, and per pixel of a frame the plain steps,
# BLA jumps, BLA lookups and rebases that the perturbation loop takes there
# (measured with all of the view's outputs on; a property of the algorithm,
# from which work() prices a pass).  "pan": how far, in widths, a seed moves
# the frame's centre.
VIEWS = {
    # z^2 + c, binary64 deltas
    "m2_1e-12": dict(at="C1", width="1e-12", steps=(35.9, 2.0, 7.7, 0.9)),
    "m2_1e-40": dict(at="C1", width="1e-40", steps=(36.0, 6.0, 12.1, 2.0)),
    "m2_1e-150": dict(at="C2_2000", width="1e-150", steps=(39.7, 6.4, 12.5, 1.0)),
    # z^2 + c, extended-range deltas
    "m2_1e-300": dict(at="C2", width="1e-300", steps=(35.7, 8.2, 14.1, 1.2)),
    "m2_1e-800": dict(at="C2_2000", width="1e-800", steps=(41.6, 11.9, 18.6, 1.6)),
    "m2_1e-2000": dict(at="C2_2000", width="1e-2000", steps=(37.5, 13.2, 19.1, 1.2)),
    # a minibrot fills the frame's centre: most pixels stop on the interior test
    "m2_interior": dict(at="C2_int", width="5e-601", pan=0.02, steps=(616.4, 367.5, 450.6, 40.8)),
    # z^d + c
    "m3_1e-60": dict(at="C3_d3", width="1e-60", steps=(30.8, 5.0, 10.0, 1.5)),
    "m3_1e-800": dict(at="C3_d3", width="1e-800", steps=(38.1, 11.0, 17.0, 1.8)),
    "m4_1e-800": dict(at="C3_d4", width="1e-800", steps=(30.0, 12.9, 17.8, 1.0)),
    "m6_1e-800": dict(at="C3_d6", width="1e-800", steps=(22.8, 10.0, 13.9, 0.8)),
    # burning ship
    "bs_1e-60": dict(at="C3_bs", width="1e-60", steps=(43.8, 5.5, 11.3, 0.1)),
    "bs_1e-800": dict(at="C3_bs", width="1e-800", steps=(65.1, 10.0, 18.8, 0.8)),
}
PRECISIONS = {"fp64": _native.FSG_PREC_FP64, "fp32x": _native.FSG_PREC_FP32X}
BACKSHIFT = 3

# one burst of the serving case: (columns, rows, width exponent) of each
# request; the even ones on the seeded boundary location (exterior frames),
# the odd ones on a resident nucleus (interior frames)
BURST = ((256, 256, -31), (512, 512, -145), (256, 256, -260), (1024, 1024, -420), (512, 512, -700),
         (256, 256, -980), (4096, 256, -1210), (512, 512, -1430), (1024, 1024, -1590), (256, 256, -1760),
         (512, 512, -1880), (4096, 256, -1990))


def listed():
    frame = dict(form="frame", precision="fp64", interior=False, orbit=False)
    return [
        # the smallest call: one tile of a shallow zoom, host arrays both ways
        dict(frame, name="tile_200_m2_1e-12", form="tile", view="m2_1e-12", nx=800, ny=600),
        # an ordinary preview, binary64 deltas
        dict(frame, name="m2_512_1e-40", view="m2_1e-40", nx=512, ny=512),
        # a ragged frame with the orbit points that field-line colouring reads
        dict(frame, name="m2_orbit_1001x667_1e-150", view="m2_1e-150", nx=1001, ny=667, orbit=True),
        # the benchmark's frames: deep zooms with interior detection
        dict(frame, name="m2_2048_1e-300", view="m2_1e-300", nx=2048, ny=2048, interior=True),
        dict(frame, name="m2_2048_1e-2000", view="m2_1e-2000", nx=2048, ny=2048, interior=True),
        # an interior-dominated frame: the longest pixels, the largest case
        dict(frame, name="m2_2048_interior", view="m2_interior", nx=2048, ny=2048, interior=True),
        # the other model families at full-HD
        dict(frame, name="m3_1920_1e-800", view="m3_1e-800", nx=1920, ny=1080),
        dict(frame, name="m6_1920_1e-800", view="m6_1e-800", nx=1920, ny=1080),
        dict(frame, name="bs_1920_1e-800", view="bs_1e-800", nx=1920, ny=1080),
        # the binary32 form, on an odd-sized frame
        dict(frame, name="fp32x_1279x719_1e-300", view="m2_1e-300", nx=1279, ny=719, interior=True,
             precision="fp32x"),
        # layers of a finished frame
        dict(name="layers_2048", form="layers", nx=2048, ny=2048, holomorphic=True),
        # a tile service: a burst of requests on resident references
        dict(name="serve_burst", form="serve", max_iter=50000),
    ]


def _log_uniform(rng, lo, hi):
    return math.exp(rng.uniform(math.log(lo), math.log(hi)))


def draw(rng):
    kind = rng.random()
    aspect = _log_uniform(rng, 0.5, 2.)
    if kind < 0.1:
        px = _log_uniform(rng, 256 ** 2, 2048 ** 2)
        return dict(form="layers", nx=max(2, int(math.sqrt(px * aspect))), ny=max(2, int(math.sqrt(px / aspect))),
                    holomorphic=rng.random() < 0.6)
    if kind < 0.15:
        return dict(form="serve", max_iter=int(_log_uniform(rng, 1000, 200000)))
    # frames from a thumbnail to the benchmark's size; the interior view's
    # pixels are the longest and its frames stay below the listed one
    view = rng.choice(sorted(VIEWS))
    px = _log_uniform(rng, 96 ** 2, (1500 if view == "m2_interior" else 2048) ** 2)
    tile = rng.random() < 0.15
    orbit = not tile and rng.random() < 0.12
    case = dict(form="tile" if tile else "frame", view=view, nx=max(64, int(math.sqrt(px * aspect))),
                ny=max(64, int(math.sqrt(px / aspect))), interior=False, orbit=orbit, precision="fp64")
    if _model(view) != "BS":
        case["interior"] = view == "m2_interior" or rng.random() < 0.4
    if not orbit and rng.random() < 0.15:
        case["precision"] = "fp32x"
    return case


# ---- preparation -----------------------------------------------------------

def _model(view):
    return configs.WORKLOADS[VIEWS[view]["at"]].model


@functools.lru_cache(maxsize=None)
def _reference(at, xrange):
    """(reference point, order, orbit, first invalid index, Xrange register)
    of a seeded location: what a program computes once per place it visits."""
    w = configs.WORKLOADS[at]
    x, y, _, _ = configs.center_for(at, compute=False)
    f = configs.new_model(w)
    f.zoom(precision=w.digits, x=x, y=y, dx=w.width if at == "C1" or xrange else "1e-100", nx=w.nx, xy_ratio=1.,
           theta_deg=0.)
    f.M_divergence = 1.e3
    f.max_iter = w.max_iter
    f.no_newton = at not in ("C1", "C2_int")  # those two: the orbit is a nucleus's cycle; else it escapes
    f.get_FP_orbit()
    p = f.FP_params
    return p["ref_point"], p["order"], f.Zn_path, p["div_iter"], p["xr"]


def _pan(case, seed):
    rng = random.Random(seed * 7919 + 17)
    pan = VIEWS[case["view"]].get("pan", 0.1)
    return rng.uniform(-pan, pan), rng.uniform(-pan, pan)


def _panned(at, view, ox, oy):
    """The panned frame's centre, as decimal texts."""
    import decimal
    w = configs.WORKLOADS[at]
    x, y, _, _ = configs.center_for(at, compute=False)
    with decimal.localcontext() as ctx:
        ctx.prec = w.digits + 10
        width = decimal.Decimal(VIEWS[view]["width"])
        return (str(decimal.Decimal(x) + decimal.Decimal(ox) * width),
                str(decimal.Decimal(y) + decimal.Decimal(oy) * width))


def _calculation(case, seed):
    """The model with its calculation "view" set up on the panned frame."""
    v = VIEWS[case["view"]]
    w = configs.WORKLOADS[v["at"]]
    x, y = _panned(v["at"], case["view"], *_pan(case, seed))
    f = configs.new_model(w)
    f.zoom(precision=w.digits, x=x, y=y, dx=v["width"], nx=case["nx"], xy_ratio=case["nx"] / case["ny"], theta_deg=0.)
    f.max_iter = w.max_iter
    f.set_reference(*_reference(v["at"], f.xr_detect_activated))
    options = dict(calc_name="view", subset=None, max_iter=w.max_iter, M_divergence=1.e3, BLA_eps=1.e-6)
    if w.model == "BS":
        options["calc_hessian"] = True
    else:
        options.update(epsilon_stationnary=1.e-3, interior_detect=case["interior"], calc_dzndc=True)
    if case["orbit"]:
        options.update(calc_orbit=True, backshift=BACKSHIFT)
    f.calc_std_div(**options)
    return f, f._calc_data["view"]["cycle_indep_args"].with_fields(precision=PRECISIONS[case["precision"]])


@functools.lru_cache(maxsize=4)
def _pixels(nx, ny):
    """The pixel offsets of an nx x ny frame, on the device."""
    f = configs.new_model(configs.WORKLOADS["C1"])
    f.zoom(precision=60, x="0", y="0", dx="1e-5", nx=nx, xy_ratio=nx / ny, theta_deg=0.)
    c_pix = np.ascontiguousarray(np.ravel(f.chunk_pixel_pos((0, nx, 0, ny))))
    return torch.from_numpy(c_pix.view(np.float64)).to(DEVICE)


class _Frame:
    """A frame's context and its device buffers."""

    def __init__(self, case, seed):
        f, self.args = _calculation(case, seed)
        fields = self.args.fields
        self.ctx = self.args.ctx
        self.nx = f.nx
        self.pix = _pixels(f.nx, f.ny)
        self.n = n = self.pix.numel() // 2
        planes = _native.n_z_fields(fields)
        z_words = planes * n * (1 if fields["kind"] == _native.FSG_KIND_BS else 2)
        self.Z = torch.empty(z_words, dtype=torch.float64, device=DEVICE)
        self.U = torch.empty(n, dtype=torch.int32, device=DEVICE)
        self.reason = torch.empty(n, dtype=torch.int8, device=DEVICE)
        self.iters = torch.empty(n, dtype=torch.int32, device=DEVICE)
        self.work = torch.zeros(_native.work_bytes() // 8, dtype=torch.int64, device=DEVICE)

    def run(self):
        self.ctx.tile_device(self.pix.data_ptr(), self.n, self.Z.data_ptr(), self.U.data_ptr(),
                             self.reason.data_ptr(), self.iters.data_ptr(), self.work.data_ptr(),
                             torch.cuda.current_stream().cuda_stream, grid_w=self.nx)
        return {"Z": self.Z, "U": self.U, "stop_reason": self.reason, "stop_iter": self.iters}


class _Tile:
    """One tile of a frame, through host arrays."""

    def __init__(self, case, seed):
        self.f, args = _calculation(case, seed)
        self.f._calc_data["view"]["cycle_indep_args"] = args
        args.ctx                                       # the context of the frame
        tiles = list(self.f.chunk_slices())
        self.tile = tiles[len(tiles) // 2]

    def run(self):
        _, (_, Z, U, reason, iters) = self.f.compute_tile("view", self.tile)
        return {"Z": Z, "U": U, "stop_reason": reason, "stop_iter": iters}


class _Layers:
    """The raw results of an escape-time frame (made up: escaped values just
    past the escape radius, derivatives over many orders of magnitude, one
    pixel in ten not escaped) and the layers computed from them."""

    def __init__(self, case, seed):
        self.n = n = case["nx"] * case["ny"]
        g = torch.Generator(DEVICE).manual_seed(seed)
        made = dict(generator=g, device=DEVICE, dtype=torch.float64)
        mod = 10. ** (3. + 3. * torch.rand(n, **made))
        arg = 2. * math.pi * torch.rand(n, **made)
        if case["holomorphic"]:
            dmod = 10. ** (-2. + 10. * torch.rand(n, **made))
            darg = 2. * math.pi * torch.rand(n, **made)
            z = torch.stack((mod * torch.cos(arg), mod * torch.sin(arg)), 1)
            d = torch.stack((dmod * torch.cos(darg), dmod * torch.sin(darg)), 1)
            self.Z = torch.stack((z, d)).contiguous()                     # [2, n] complex rows
        else:
            d = torch.randn(4, n, **made) * 10. ** (-2. + 10. * torch.rand(n, **made))
            self.Z = torch.cat((torch.stack((mod * torch.cos(arg), mod * torch.sin(arg))), d)).contiguous()
        self.iters = torch.randint(100, 100000, (n,), generator=g, device=DEVICE, dtype=torch.int32)
        kind = torch.rand(n, **made)
        self.reason = torch.where(kind < 0.9, 1, torch.where(kind < 0.95, 0, 2)).to(torch.int8)
        self.desc = _native.PostDesc(int(case["holomorphic"]), 1 if case["holomorphic"] else 2, 2., 1., 1.e3, 0., 0.)
        for i, s in enumerate((1., 0., 0., 1.)):
            self.desc.skew[i] = s
        self.nu = torch.empty(n, dtype=torch.float32, device=DEVICE)
        self.dem = torch.empty(n, dtype=torch.float32, device=DEVICE)
        self.normal = torch.empty(n, 2, dtype=torch.float32, device=DEVICE)

    def run(self):
        _native.check(_native.load().fsg_postproc_device(
            self.desc, self.Z.data_ptr(), self.n, self.n, None, self.iters.data_ptr(), self.reason.data_ptr(),
            self.nu.data_ptr(), self.dem.data_ptr(), self.normal.data_ptr(), torch.cuda.current_stream().cuda_stream))
        return {"nu": self.nu, "dem": self.dem, "normal": self.normal}


@functools.lru_cache(maxsize=1)
def _service():
    """The running tile server and its resident centres: two nuclei and the
    boundary location, one base context per centre and arithmetic."""
    server = serving.TileServer(lanes=3, chunk_px=65536, hbm_budget=2 << 30)
    return server, serving.serve_centres(2) + [serving.boundary_centre()], {}


def _pinned(c_pix):
    """A request's buffers, as a LayerTile holds them, in pinned memory that
    lives as long as any of its arrays."""
    def empty(shape, dtype):
        return torch.empty(shape, dtype=dtype, pin_memory=True).numpy()
    n = c_pix.size
    tile = types.SimpleNamespace(
        c_pix=empty(n, torch.complex128), nu=empty(n, torch.float32), dem=empty(n, torch.float32), normal=None,
        stop_reason=empty((1, n), torch.int8), stop_iter=empty((1, n), torch.int32))
    tile.c_pix[:] = c_pix
    return tile


class _Burst:
    """Requests returning the nu / dem layers, all submitted at once."""

    def __init__(self, case, seed):
        self.server, centres, bases = _service()
        rng = random.Random(seed * 104729 + 5)
        self.requests = []
        for k, (nx, ny, exponent) in enumerate(BURST):
            spec = serving.RequestSpec(2 if k % 2 == 0 else rng.randrange(2), nx, ny,
                                       f"{rng.uniform(1., 9.):.6f}e{exponent}", case["max_iter"],
                                       rng.uniform(-0.3, 0.3), rng.uniform(-0.3, 0.3))
            f, args, c_pix = serving.build_request(spec, centres)
            base = bases.setdefault(args.resident_key, args)
            if base is not args:
                args = args.shared_with(base.ctx)
            tile = _pinned(c_pix)
            self.requests.append((args.ctx, tile, post_desc(f, "serve"), nx))
            if base is args:
                args.ctx                                    # stays resident with the service

    def run(self):
        tickets = [self.server.submit_layers(ctx, tile, post, grid_w=nx) for ctx, tile, post, nx in self.requests]
        for t in tickets:
            self.server.wait(t)
        return [{"nu": t.nu, "dem": t.dem, "stop_reason": t.stop_reason, "stop_iter": t.stop_iter}
                for _, t, _, _ in self.requests]


def prepare(case, seed):
    return {"frame": _Frame, "tile": _Tile, "layers": _Layers, "serve": _Burst}[case["form"]](case, seed)


def run(state):
    return state.run()


# ---- what a pass cannot do without -----------------------------------------

def _flops(model, degree, dc, dz):
    """Flops (add / multiply / square root = 1) of a plain step, a BLA jump,
    a BLA lookup and a rebase."""
    if model == "BS":
        return 71, 26, 4, 4
    z = 12 if model == "M2" else 12 + 16 * (degree - 2)
    return z + 5 + 18 * dc + 23 * dz, 14 + 6 * dc + 6 * dz, 4, 2 * dc + 2 * dz


def work(case):
    if case["form"] == "layers":
        n = case["nx"] * case["ny"]
        # a value and a derivative (or a 2x2 Jacobian) in, four floats out
        return {"bytes": n * ((32 if case["holomorphic"] else 48) + 5 + 16), "flops": 60. * n}
    if case["form"] == "serve":
        n = sum(nx * ny for nx, ny, _ in BURST)
        return {"bytes": n * (16 + 13), "flops": 58. * 40. * n}
    w = configs.WORKLOADS[VIEWS[case["view"]]["at"]]
    if case["form"] == "tile":
        n = min(settings.chunk_size, case["nx"]) * min(settings.chunk_size, case["ny"])
    else:
        n = case["nx"] * case["ny"]
    planes = (2 + 4 + 2 * case["orbit"]) / 2. if w.model == "BS" else 2 + case["interior"] + case["orbit"]
    per_px = sum(c * f for c, f in zip(VIEWS[case["view"]]["steps"], _flops(w.model, w.degree, 1, case["interior"])))
    return {"bytes": n * (16 + 16 * planes + 9), "flops": n * per_px}


# ---- the same outputs in 64 bits, without the framework's code --------------

def _exact_layers(case, seed):
    """The layers by their formulas, in numpy."""
    s = _Layers(case, seed)
    Z, n = s.Z.cpu().numpy(), s.iters.cpu().numpy().astype(np.float64)
    escaped = s.reason.cpu().numpy() == 1
    with np.errstate(all="ignore"):
        if case["holomorphic"]:
            z, d = Z[0, :, 0] + 1j * Z[0, :, 1], Z[1, :, 0] + 1j * Z[1, :, 1]
            size, normal = np.abs(d), z / d
        else:
            z, (a, b, c, d) = Z[0] + 1j * Z[1], Z[2:]
            size = 0.5 * (np.hypot(a + d, b - c) + np.hypot(a - d, b + c))
            normal = (a * z.real + c * z.imag) + 1j * (b * z.real + d * z.imag)
        x = np.log(np.log(np.abs(z)) / np.log(1.e3)) / np.log(2.)
        nu = n - np.floor(x) - (x - np.floor(x))
        dem = np.abs(z) * np.log(np.abs(z)) / size
        normal = normal / np.abs(normal)
    out = {"nu": nu, "dem": dem, "normal": np.stack((normal.real, normal.imag), 1)}
    for v in out.values():
        v[~escaped] = np.nan
    return {k: torch.from_numpy(v) for k, v in out.items()}


def _fixed_orbit(x, y, digits, n_max):
    """z^2 + c from 0 at c = x + iy in fixed-point integers: the orbit up to
    its escape, rounded to binary64."""
    from fractions import Fraction
    bits = int(digits * 3.33) + 64
    cx, cy = (round(Fraction(v) * (1 << bits)) for v in (x, y))
    a = b = 0
    out = []
    for _ in range(n_max):
        out.append(complex(a / (1 << bits), b / (1 << bits)))
        a, b = ((a * a - b * b) >> bits) + cx, ((2 * a * b) >> bits) + cy
        if a * a + b * b > 10 ** 8 << (2 * bits):
            break
    return np.array(out)


def _exact_frame(case, seed):
    """Escaped z and dz/dc of a shallow z^2 + c view, iterated without any
    skipping as Z_n + z_n around the frame's own centre."""
    v = VIEWS[case["view"]]
    w = configs.WORKLOADS[v["at"]]
    nx, ny = case["nx"], case["ny"]
    x, y = _panned(v["at"], case["view"], *_pan(case, seed))
    orbit = _fixed_orbit(x, y, w.digits, w.max_iter)
    cs = settings.chunk_size
    ix, ixx, iy, iyy = 0, nx, 0, ny
    if case["form"] == "tile":
        tiles = [(i, min(i + cs, nx), j, min(j + cs, ny)) for i in range(0, nx, cs) for j in range(0, ny, cs)]
        ix, ixx, iy, iyy = tiles[len(tiles) // 2]
    px = np.linspace(0.5 * (2 * ix - nx + 1) / (nx - 1), 0.5 * (2 * ixx - nx - 1) / (nx - 1), ixx - ix)
    py = np.linspace(0.5 * (2 * iy - ny + 1) / (ny - 1), 0.5 * (2 * iyy - ny - 1) / (ny - 1), iyy - iy)
    dx = float(v["width"])
    c = np.ravel(px[None, :] - 1j * py[:, None] * ny / nx) * dx
    out = np.zeros((2, c.size), dtype=np.complex128)
    at = np.arange(c.size)
    z, d = np.zeros_like(c), np.zeros_like(c)
    full, k = np.zeros_like(c), np.zeros(c.size, dtype=np.int64)
    for _ in range(w.max_iter):
        d = 2. * full * d + dx
        z = z * (z + 2. * orbit[k]) + c
        k += 1
        full = orbit[k] + z
        gone = full.real ** 2 + full.imag ** 2 > 1.e6
        if gone.any():
            out[0, at[gone]], out[1, at[gone]] = full[gone], d[gone]
            left = ~gone
            at, z, d, c, full, k = at[left], z[left], d[left], c[left], full[left], k[left]
            if not at.size:
                break
        back = ((np.abs(full.real) <= np.abs(z.real)) & (np.abs(full.imag) <= np.abs(z.imag))) | (k >= len(orbit) - 1)
        z[back], k[back] = full[back], 0
    out = out if case["form"] == "tile" else torch.from_numpy(out.view(np.float64).reshape(-1))
    return {"Z": out, "U": None, "stop_reason": None, "stop_iter": None}


def exact(case, seed):
    if case["form"] == "layers":
        return _exact_layers(case, seed)
    if (case["form"] in ("frame", "tile") and case["view"] in ("m2_1e-12", "m2_1e-40") and case["precision"] == "fp64"
            and not case["interior"] and not case["orbit"] and case["nx"] * case["ny"] <= 500000):
        return _exact_frame(case, seed)
    return None
