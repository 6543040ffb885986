"""Cases by which the speed of this framework is measured: the calls that a
visibility simulation makes per time sample and channel, through the public
C-ABI, from a few stations and a few hundred sources to the headline
workload of 512 stations and a million sources.

Kinds:
  direct    oskar_cross_correlate on Jones matrices (or Stokes-I scalars)
            of every (station, source): point and Gaussian sources, with and
            without bandwidth and time smearing, FP32 and FP64, both phase
            conventions.  This is the correlator every simulation runs.
  shared    oskar_cross_correlate_factorised: one station beam shared by
            all stations, point sources.
  stations  oskar_cross_correlate_factorised_jones: one beam per station.
  beam      oskar_station_beam of an aperture array of crossed dipoles.
  step      one whole time sample and channel in double precision:
            oskar_evaluate_jones_E (every station its own layout),
            oskar_evaluate_jones_K, oskar_jones_join, oskar_cross_correlate
            and oskar_auto_correlate.
  clip      oskar_sky_horizon_clip of an all-sky catalogue.

Every correlation clears its visibilities first, as a simulation does for
each new block.
"""
import ctypes as C
import math

import numpy as np
import torch

from oskar_amd import capi, lib
from oskar_amd.mem import (OSKAR_COMPLEX, OSKAR_DOUBLE, OSKAR_GPU,
                           OSKAR_MATRIX, OSKAR_SINGLE, Jones, Mem, Sky,
                           StationView, Station, StationWork, Telescope,
                           check_status)

C0 = 299792458.0
FREQ_HZ = 150e6
RADEC, AZEL, ENU_DIR = 2, 4, 1
RA0, DEC0, GAST = 0.4, -0.5, 1.3
POINTING = (0.0, math.radians(60.0))        # azimuth, elevation
MJD = 60000.0
OMEGA_EARTH = 7.272205217e-5

# Sky columns of a catalogue: RA, Dec, I, Q, U, V, reference frequency,
# spectral index, rotation measure, major, minor, PA, l, m, n, a, b, c.
CLIP_COLUMNS = (1, 2, 3, 4, 5, 6, 7, 8, 9, 10, 11, 12,
                0x103, 0x104, 0x105, 0x100, 0x101, 0x102)


# --- the cases --------------------------------------------------------------

def _direct(name, precision, stations, sources, matrix=True, gaussian=False,
            bandwidth_hz=0.0, time_s=0.0, casa=False, radius_m=35000.0):
    return dict(name=name, kind="direct", precision=precision,
                stations=stations, sources=sources, matrix=matrix,
                gaussian=gaussian, bandwidth_hz=bandwidth_hz, time_s=time_s,
                casa=casa, radius_m=radius_m)


def listed():
    return [
        # A small array and a short catalogue in double precision with every
        # factor on, the size of a first simulation: launches and latency.
        _direct("direct_small_f64", "f64", 30, 277, gaussian=True,
                bandwidth_hz=10e3, time_s=1.0, radius_m=3000.0),
        # The default settings of a simulation (double precision, point
        # sources, no smearing) on an array of SKA1-Mid's size.
        _direct("direct_point_f64", "f64", 197, 30011, radius_m=20000.0),
        # The plain FP32 correlator at SKA1-Low's 512 stations.
        _direct("direct_point_f32", "f32", 512, 100000),
        # Extended sources with bandwidth and time smearing, both precisions.
        _direct("direct_gauss_smear_f32", "f32", 512, 20000, gaussian=True,
                bandwidth_hz=10e3, time_s=1.0),
        _direct("direct_smear_f64", "f64", 255, 10007, bandwidth_hz=10e3,
                time_s=1.0, casa=True, radius_m=20000.0),
        # Stokes-I only simulation (scalar mode) with bandwidth smearing.
        _direct("direct_scalar_f32", "f32", 351, 50001, matrix=False,
                bandwidth_hz=10e3, radius_m=20000.0),
        # The headline workload: one beam shared by 512 stations, 1M sources.
        dict(name="shared_512", kind="shared", precision="f32", mode=0,
             stations=512, sources=1000000, radius_m=35000.0),
        # The same path at the size of a small array and a bright catalogue.
        dict(name="shared_small", kind="shared", precision="f32", mode=0,
             stations=97, sources=12007, radius_m=10000.0),
        # Every station its own beam.
        dict(name="stations_512", kind="stations", precision="f32", mode=0,
             stations=512, sources=150000, radius_m=35000.0),
        # One station's beam: 256 dipoles over a million directions in FP32
        # (the step below holds 60 smaller ones in FP64).
        dict(name="beam_f32", kind="beam", precision="f32", elements=256,
             sources=1000000),
        # A whole time sample and channel of a 60-station array in FP64.
        dict(name="step_f64", kind="step", precision="f64", elements=96,
             stations=60, sources=16385, radius_m=10000.0),
        # All-sky catalogue clipped to the local sky, once per time sample.
        dict(name="clip_1m", kind="clip", precision="f32", sources=1000000),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["direct"] * 6 + ["shared"] * 2 + ["stations"] +
                      ["beam"] * 2 + ["step"] + ["clip"])
    precision = rng.choice(["f32", "f64"])
    stations = _log_int(rng, 20, 512)
    pairs = stations * (stations - 1) // 2
    radius = math.exp(rng.uniform(math.log(3000.0), math.log(35000.0)))
    if kind == "direct":
        matrix = rng.random() < 0.75
        smear = rng.random() < 0.5
        c = _direct("", precision, stations, 0, matrix=matrix,
                    gaussian=smear and rng.random() < 0.5,
                    bandwidth_hz=10e3 if smear else 0.0,
                    time_s=1.0 if smear and rng.random() < 0.5 else 0.0,
                    casa=rng.random() < 0.3, radius_m=radius)
        most = {("f32", False): 1.2e10, ("f32", True): 2.5e9,
                ("f64", False): 2.5e9, ("f64", True): 8e8}[(precision, smear)]
        c["sources"] = min(_log_int(rng, 200, 100000), int(most / pairs))
    elif kind == "shared":
        c = dict(kind=kind, precision=precision, mode=rng.choice([0, 0, 1]),
                 stations=stations, sources=_log_int(rng, 1000, 900000),
                 radius_m=radius)
    elif kind == "stations":
        c = dict(kind=kind, precision="f32", mode=0, stations=stations,
                 sources=_log_int(rng, 1000, 140000), radius_m=radius)
    elif kind == "beam":
        c = dict(kind=kind, precision=precision,
                 elements=_log_int(rng, 16, 256),
                 sources=_log_int(rng, 1000, 900000 if precision == "f32"
                                  else 200000))
    elif kind == "step":
        c = dict(kind=kind, precision="f64", elements=_log_int(rng, 16, 128),
                 stations=min(stations, 60), sources=_log_int(rng, 500, 16000),
                 radius_m=radius)
    else:
        c = dict(kind=kind, precision="f32",
                 sources=_log_int(rng, 10000, 1000000))
    c.pop("name", None)
    return c


def work(case):
    """Bytes: inputs read once, outputs written once.  Operations: the
    contraction itself (a complex multiply-add is 8), plus what the smearing
    factors of an evaluation and the terms of a beam take."""
    s = case["sources"]
    fp = 4 if case["precision"] == "f32" else 8
    kind = case["kind"]
    if kind == "beam":
        return {"bytes": s * (3 * fp + 8 * fp),
                "flops": 12.0 * s * case["elements"]}
    if kind == "clip":
        return {"bytes": s * 3 * fp + s / 2 * 2 * (18 * fp + 80), "flops": 0}
    n = case["stations"]
    pairs = n * (n - 1) // 2
    if kind == "direct":
        nr = 8 if case["matrix"] else 2
        factors = bool(case["gaussian"]) + bool(case["bandwidth_hz"]) + \
            bool(case["time_s"])
        per = 4 * nr * nr // 4 if case["matrix"] else 8
        per += 8 * factors + (nr if factors else 0)
        return {"bytes": fp * (n * s * nr + s * 10 + pairs * nr),
                "flops": float(per) * pairs * s}
    if kind == "shared":
        return {"bytes": fp * (s * (8 + 4 + 3) + pairs * 8),
                "flops": 32.0 * pairs * s}
    if kind == "stations":
        return {"bytes": fp * (n * s * 8 + s * 7 + pairs * 8),
                "flops": 64.0 * pairs * s}
    # step: beams, K, join, cross- and auto-correlation.  The Jones matrices
    # are intermediate values; only the sky and the visibilities have to
    # cross memory.
    return {"bytes": fp * (s * 7 + (pairs + n) * 8),
            "flops": 12.0 * n * s * case["elements"] + 64.0 * n * s +
            64.0 * (pairs + n) * s}


def tolerance(case):
    """About four times the largest relative error against exact() that the
    sizes of draw() showed."""
    kind, single = case["kind"], case["precision"] == "f32"
    if kind == "clip":
        return "exact"
    if kind in ("shared", "stations"):
        return {"rel": 2e-5} if case["mode"] == 0 else {"rel": 4e-5}
    if kind == "beam":
        return {"rel": 1e-5} if single else {"rel": 1e-12}
    if kind == "step":
        return {"rel": 4e-12}
    smear = case["gaussian"] or case["bandwidth_hz"] or case["time_s"]
    if single:
        return {"rel": 4e-6} if smear else {"rel": 8e-7}
    return {"rel": 1e-13}


# --- inputs -----------------------------------------------------------------

def _types(case):
    if case["precision"] == "f64":
        return OSKAR_DOUBLE, torch.float64
    return OSKAR_SINGLE, torch.float32


def _sky(gen, n, dtype):
    """Directions uniform over the sky above the horizon, Stokes I from a
    power law (index -1.8, 0.01-10 Jy), up to 20 % polarised."""
    def uni(*shape):
        return torch.rand(*shape, generator=gen, device="cuda",
                          dtype=torch.float64)
    z = uni(n).clamp_min(1e-4)
    ph = uni(n) * (2 * math.pi)
    r = torch.sqrt(1 - z * z)
    a = -0.8
    flux = (0.01 ** a + uni(n) * (10.0 ** a - 0.01 ** a)) ** (1.0 / a)
    d = torch.randn(3, n, generator=gen, device="cuda", dtype=torch.float64)
    d = d / d.norm(dim=0) * (0.2 * uni(n) * flux)
    return dict(dir=torch.stack([r * torch.sin(ph), r * torch.cos(ph),
                                 z]).to(dtype),
                flux=torch.cat([flux[None], d]).to(dtype))


def _gaussians(gen, n, dtype):
    """a, b, c of the sources: 30 % Gaussian, FWHM 5-60 arcsec."""
    def uni():
        return torch.rand(n, generator=gen, device="cuda",
                          dtype=torch.float64)
    on = uni() < 0.3
    major = torch.where(on, (5 + 55 * uni()) * (math.pi / 648000), 0.0)
    minor = major * (0.2 + 0.8 * uni())
    pa = uni() * math.pi
    k = math.pi ** 2 / (4 * math.log(2.0))
    s, c = torch.sin(pa), torch.cos(pa)
    return torch.stack([k * ((major * s) ** 2 + (minor * c) ** 2),
                        k * (major ** 2 - minor ** 2) * s * c,
                        k * ((major * c) ** 2 + (minor * s) ** 2)]).to(dtype)


def _uvw(seed, n, radius, dtype):
    """Log-radial station layout out to `radius`, w within +-20 m."""
    rng = np.random.default_rng(1000 + seed)
    r = np.exp(rng.uniform(np.log(0.003 * radius), np.log(radius), n))
    t = rng.uniform(0, 2 * np.pi, n)
    a = np.stack([r * np.cos(t), r * np.sin(t), rng.uniform(-20, 20, n)])
    return torch.from_numpy(a).to(dtype)


def _jones(gen, n, s, nr, dtype):
    """Jones values of every (station, source): a unit phasor (the geometric
    phase) times a beam near the identity, reals interleaved."""
    j = torch.randn(n, s, nr // 2, 2, generator=gen, device="cuda",
                    dtype=dtype).mul_(0.3)
    j[:, :, 0, 0] += 1
    if nr == 8:
        j[:, :, 3, 0] += 1
    ph = torch.rand(n, s, 1, generator=gen, device="cuda",
                    dtype=dtype).mul_(2 * math.pi)
    z = torch.view_as_complex(j)
    z *= torch.polar(torch.ones_like(ph), ph)
    return j.reshape(n, s, nr)


def _elements(seed, n, dtype):
    """Element layout: uniform in a disc that holds one element per 4 m^2,
    in the station's plane."""
    rng = np.random.default_rng(5000 + seed)
    r = math.sqrt(4.0 * n / math.pi) * np.sqrt(rng.uniform(size=n))
    t = rng.uniform(0, 2 * np.pi, n)
    a = np.stack([r * np.cos(t), r * np.sin(t), np.zeros(n)])
    return torch.from_numpy(a).to(dtype)


def _inputs(case, seed):
    """The numbers of a case, made from the seed alone."""
    _, dtype = _types(case)
    gen = torch.Generator(device="cuda").manual_seed(77777 + seed)
    s, kind = case["sources"], case["kind"]
    x = _sky(gen, s, dtype)
    if "stations" in case:
        x["uvw"] = _uvw(seed, case["stations"], case["radius_m"], dtype)
    if kind == "direct":
        x["ext"] = _gaussians(gen, s, dtype)
        x["jones"] = _jones(gen, case["stations"], s,
                            8 if case["matrix"] else 2, dtype)
    elif kind == "shared":
        x["beam"] = _jones(gen, 1, s, 8, dtype)[0]
    elif kind == "stations":
        x["jones"] = _jones(gen, case["stations"], s, 8, dtype)
    elif kind in ("beam", "step"):
        x["elements"] = [_elements(seed * 1000 + i, case["elements"], dtype)
                         for i in range(case.get("stations", 1))]
    return x


def _mem(tensor, type_code, keep):
    """An oskar_Mem over a device tensor."""
    st = C.c_int(0)
    n = tensor.numel()
    n //= (2 if type_code & OSKAR_COMPLEX else 1) * \
        (4 if type_code & OSKAR_MATRIX else 1)
    m = Mem(type_code, OSKAR_GPU, n, ptr=lib.oskar_mem_create_alias_from_raw(
        C.c_void_p(tensor.data_ptr()), type_code, OSKAR_GPU, n, C.byref(st)))
    check_status(st, "alias")
    keep.append((tensor, m))
    return m


def _three(t, type_code, keep):
    t = t.cuda()
    return capi.MEM3(*[_mem(t[i], type_code, keep).ptr for i in range(3)])


def _fill_jones(tensor, type_code, keep):
    """An oskar_Jones holding a copy of the tensor's values."""
    j = Jones(type_code, OSKAR_GPU, tensor.shape[0], tensor.shape[1])
    src = _mem(tensor, type_code, [])
    st = C.c_int(0)
    lib.oskar_mem_copy_contents(lib.oskar_jones_mem(j.ptr), src.ptr, 0, 0,
                                len(src), C.byref(st))
    check_status(st, "jones")
    torch.cuda.synchronize()
    keep.append(j)
    return j


class _Device:
    """A device array of the library, for torch.as_tensor: the tensor keeps
    this object, and so the array's owner, for as long as it lives."""

    def __init__(self, owner, ptr, shape, code):
        self.owner = owner
        self.__cuda_array_interface__ = dict(
            shape=shape, typestr=code, data=(ptr, False), version=2)


def _telescope(case, x, prec, keep):
    n = case["stations"]
    tel = Telescope(prec, OSKAR_GPU, n)
    keep.append(tel)
    xyz = x["uvw"].double().numpy()
    tel.set_station_ecef(xyz[0], xyz[1], np.zeros(n))
    return tel


def _set_station(station, elements):
    st = C.c_int(0)
    station.set_coords(elements.double().numpy())
    lib.oskar_station_set_phase_centre(station.ptr, AZEL, *POINTING)
    lib.oskar_station_set_normalise_array_pattern(station.ptr, 0)
    lib.oskar_station_set_normalise_final_beam(station.ptr, 1)
    check_status(st, "station")


def prepare(case, seed):
    prec, dtype = _types(case)
    kind, s = case["kind"], case["sources"]
    if kind == "clip":
        return _prepare_clip(case, seed, prec, dtype)
    x = _inputs(case, seed)
    keep = [x]
    matrix = prec | OSKAR_COMPLEX | OSKAR_MATRIX
    p = dict(keep=keep, kind=kind, status=C.c_int(0))
    p["ref"] = C.byref(p["status"])
    flux = x["flux"]
    p["flux"] = capi.MEMA(*[_mem(flux[i], prec, keep).ptr for i in range(4)])
    p["dir"] = _three(x["dir"], prec, keep)
    p["s"] = s
    if kind == "beam":
        station = Station(prec, OSKAR_GPU, case["elements"])
        _set_station(station, x["elements"][0])
        p["station"], p["work"] = station, StationWork(prec, OSKAR_GPU)
        p["out"] = torch.zeros(s, 8, dtype=dtype, device="cuda")
        p["mem"] = _mem(p["out"], matrix, keep).ptr
        return p
    n = case["stations"]
    nb = n * (n - 1) // 2
    p["uvw"] = _three(x["uvw"], prec, keep)
    tel = _telescope(case, x, prec, keep)
    p["tel"] = tel.ptr
    nr = 8 if case.get("matrix", True) else 2
    vt = matrix if nr == 8 else prec | OSKAR_COMPLEX
    p["out"] = torch.zeros(nb, nr, dtype=dtype, device="cuda")
    p["vis"] = _mem(p["out"], vt, keep).ptr
    if kind == "direct":
        lib.oskar_telescope_set_channel_bandwidth(tel.ptr,
                                                  case["bandwidth_hz"])
        lib.oskar_telescope_set_time_average(tel.ptr, case["time_s"])
        lib.oskar_telescope_set_phase_centre(tel.ptr, RADEC, RA0, DEC0)
        p["ext"] = _three(x["ext"], prec, keep)
        p["jones"] = _fill_jones(x.pop("jones"), vt, keep).ptr
        p["casa"], p["gaussian"] = int(case["casa"]), int(case["gaussian"])
    elif kind == "shared":
        p["mode"] = case["mode"]
        p["beam"] = _mem(x["beam"], matrix, keep).ptr
    elif kind == "stations":
        p["mode"] = case["mode"]
        p["jones"] = _fill_jones(x.pop("jones"), matrix, keep).ptr
    else:
        lib.oskar_telescope_resize_station_array(tel.ptr, n, p["ref"])
        lib.oskar_telescope_set_phase_centre(tel.ptr, AZEL, *POINTING)
        for i in range(n):
            view = StationView(lib.oskar_telescope_station(tel.ptr, i), prec)
            lib.oskar_station_resize(view.ptr, case["elements"], p["ref"])
            _set_station(view, x["elements"][i])
        p["work"] = StationWork(prec, OSKAR_GPU)
        e = Jones(matrix, OSKAR_GPU, n, s)
        k = Jones(prec | OSKAR_COMPLEX, OSKAR_GPU, n, s)
        keep += [e, k]
        p["E"], p["K"] = e.ptr, k.ptr
        p["auto"] = torch.zeros(n, 8, dtype=dtype, device="cuda")
        p["vis_auto"] = _mem(p["auto"], matrix, keep).ptr
        p["ext"] = p["dir"]
    check_status(p["status"], kind)
    return p


def _prepare_clip(case, seed, prec, dtype):
    s = case["sources"]
    gen = torch.Generator(device="cuda").manual_seed(99999 + seed)

    def uni():
        return torch.rand(s, generator=gen, device="cuda",
                          dtype=torch.float64)
    ra, dec = uni() * (2 * math.pi), torch.asin(2 * uni() - 1)
    dec0 = math.radians(-30.0)
    cd, sd = math.cos(dec0), math.sin(dec0)
    flux = 0.01 + 10 * uni()
    value = {1: ra, 2: dec, 3: flux, 4: 0.1 * (uni() - 0.5),
             5: 0.1 * (uni() - 0.5), 6: 0.1 * (uni() - 0.5),
             7: torch.full_like(ra, 1e8), 8: -0.7 + 0.1 * uni(),
             0x103: torch.cos(dec) * torch.sin(ra),
             0x104: cd * torch.sin(dec) -
             sd * torch.cos(dec) * torch.cos(ra),
             0x105: sd * torch.sin(dec) +
             cd * torch.cos(dec) * torch.cos(ra)}
    zero = torch.zeros_like(ra)
    sky, out = (Sky(prec, OSKAR_GPU, s) for _ in range(2))
    st = C.c_int(0)
    for c in CLIP_COLUMNS:
        sky.column(c)
        out.column(c)
    for c in CLIP_COLUMNS:
        src = _mem(value.get(c, zero).to(dtype), prec, [])
        lib.oskar_mem_copy_contents(sky.column(c).ptr, src.ptr, 0, 0, s,
                                    C.byref(st))
        torch.cuda.synchronize()
    check_status(st, "sky")
    sky.set_reference(0.0, dec0)
    capacity = out.attr(Sky.CAPACITY)
    code = "<f4" if dtype == torch.float32 else "<f8"
    table = torch.as_tensor(_Device(out, out.column(CLIP_COLUMNS[0]).data_ptr(),
                                    (len(CLIP_COLUMNS), capacity), code),
                            device="cuda")
    tel = Telescope(prec, OSKAR_GPU, 4)
    lib.oskar_telescope_resize_station_array(tel.ptr, 1, C.byref(st))
    lib.oskar_station_set_position(lib.oskar_telescope_station(tel.ptr, 0),
                                   math.radians(116.7), math.radians(-26.7),
                                   0.0, 0.0, 0.0, 0.0)
    check_status(st, "clip")
    return dict(kind="clip", sky=sky, out=out, table=table, tel=tel,
                work=StationWork(prec, OSKAR_GPU), status=st,
                ref=C.byref(st), gast=0.37 * seed % (2 * math.pi))


def run(p):
    kind, ref = p["kind"], p["ref"]
    if kind == "direct":
        lib.oskar_mem_clear_contents(p["vis"], ref)
        lib.oskar_cross_correlate(p["casa"], p["gaussian"], p["s"],
                                  p["jones"], p["flux"], p["dir"], p["ext"],
                                  p["tel"], p["uvw"], GAST, FREQ_HZ, 0,
                                  p["vis"], ref)
        out = p["out"]
    elif kind == "shared":
        lib.oskar_mem_clear_contents(p["vis"], ref)
        lib.oskar_cross_correlate_factorised(
            0, p["s"], p["beam"], p["flux"], p["dir"], p["tel"], p["uvw"],
            FREQ_HZ, p["mode"], 0, p["vis"], ref)
        out = p["out"]
    elif kind == "stations":
        lib.oskar_mem_clear_contents(p["vis"], ref)
        lib.oskar_cross_correlate_factorised_jones(
            0, p["s"], p["jones"], p["flux"], p["dir"], p["tel"], p["uvw"],
            FREQ_HZ, p["mode"], 0, p["vis"], ref)
        out = p["out"]
    elif kind == "beam":
        lib.oskar_station_beam(p["station"].ptr, p["work"].ptr, ENU_DIR,
                               p["s"], p["dir"], 0.0, 0.0, AZEL, POINTING[0],
                               POINTING[1], 0, MJD, MJD, FREQ_HZ, 0,
                               p["mem"], ref)
        out = p["out"]
    elif kind == "step":
        lib.oskar_evaluate_jones_E(p["E"], ENU_DIR, p["s"], p["dir"], 0.0,
                                   0.0, p["tel"], 0, MJD, MJD, FREQ_HZ,
                                   p["work"].ptr, ref)
        d, u = p["dir"], p["uvw"]
        lib.oskar_evaluate_jones_K(p["K"], p["s"], d[0], d[1], d[2], u[0],
                                   u[1], u[2], FREQ_HZ, p["flux"][0], -1e30,
                                   1e30, 0, ref)
        lib.oskar_jones_join(p["E"], p["K"], p["E"], ref)
        lib.oskar_mem_clear_contents(p["vis"], ref)
        lib.oskar_mem_clear_contents(p["vis_auto"], ref)
        lib.oskar_cross_correlate(0, 0, p["s"], p["E"], p["flux"], d,
                                  p["ext"], p["tel"], u, GAST, FREQ_HZ, 0,
                                  p["vis"], ref)
        lib.oskar_auto_correlate(p["s"], p["E"], p["flux"], 0, p["vis_auto"],
                                 ref)
        out = {"cross": p["out"], "auto": p["auto"]}
    else:
        lib.oskar_sky_horizon_clip(p["out"].ptr, p["sky"].ptr, p["tel"].ptr,
                                   p["gast"], p["work"].ptr, ref)
        kept = lib.oskar_sky_int(p["out"].ptr, Sky.NUM_SOURCES)
        out = {"kept": kept, "table": p["table"]}
    check_status(p["status"], kind)
    return out


# --- the same in 64 bits, in plain torch ------------------------------------

def _brightness(flux):
    i, q, u, v = flux.double()
    b = torch.stack([i + q, u + 1j * v, u - 1j * v, i - q], dim=1)
    return b.reshape(-1, 2, 2).to(torch.complex128)


def _phasor(uvw, d):
    """K of every (station, source)."""
    u, dd = uvw.double().cuda(), d.double().clone()
    dd[2] -= 1
    return torch.polar(torch.ones(u.shape[1], dd.shape[1], device="cuda",
                                  dtype=torch.float64),
                       (2 * math.pi * FREQ_HZ / C0) * (u.T @ dd))


def _pick(full, n, casa):
    """The baselines of a product of all station pairs (n, 2, n, 2)."""
    q, p = torch.triu_indices(n, n, 1, device="cuda")
    full = full.reshape(n, 2, n, 2)
    out = full[q, :, p, :] if casa else full[p, :, q, :]
    return torch.view_as_real(out.contiguous()).reshape(-1, 8)


def _contract(jones_of, bright, n, s, casa):
    """sum_s J_p B J_q^H over chunks of sources; jones_of(a, b) gives
    (n, b - a, 2, 2)."""
    full = torch.zeros(2 * n, 2 * n, device="cuda", dtype=torch.complex128)
    step = max(1, (1 << 23) // n)
    auto = torch.zeros(n, 2, 2, device="cuda", dtype=torch.complex128)
    for a in range(0, s, step):
        b = min(s, a + step)
        j = jones_of(a, b)
        # (n, s, 2, 2) x (s, 2, 2), written out per element.
        w = bright[a:b]
        m = torch.stack([j[..., 0] * w[:, 0, 0, None] +
                         j[..., 1] * w[:, 1, 0, None],
                         j[..., 0] * w[:, 0, 1, None] +
                         j[..., 1] * w[:, 1, 1, None]], dim=-1)
        left = m.permute(0, 2, 1, 3).reshape(2 * n, -1)
        right = j.permute(0, 2, 1, 3).reshape(2 * n, -1)
        full += left @ right.conj().T.contiguous()
    for i in range(2):
        for k in range(2):
            idx = torch.arange(n, device="cuda")
            auto[:, i, k] = full.reshape(n, 2, n, 2)[idx, i, idx, k]
    return _pick(full, n, casa), torch.view_as_real(auto).reshape(n, 8)


def _sinc(x):
    return torch.where(x.abs() < 1e-6, 1 - x * x / 6, torch.sin(x) /
                       torch.where(x == 0, 1.0, x))


def _exact_direct(case, x):
    n, s = case["stations"], case["sources"]
    nr = 8 if case["matrix"] else 2
    smear = case["gaussian"] or case["bandwidth_hz"] or case["time_s"]
    jones = x["jones"]
    if case["matrix"]:
        bright = _brightness(x["flux"])

        def cut(a, b):
            j = jones[:, a:b].double().reshape(n, b - a, 2, 2, 2)
            return torch.view_as_complex(j.contiguous())
        if not smear:
            return _contract(cut, bright, n, s, case["casa"])[0]
    u = x["uvw"].double().cuda()
    d = x["dir"].double().clone()
    d[2] -= 1
    ext = x["ext"].double()
    inv_wl = FREQ_HZ / C0
    frac = case["bandwidth_hz"] / FREQ_HZ
    ha0 = GAST - RA0
    out = []
    step = max(1, (1 << 24) // n)
    full = [0] * n
    for a in range(0, s, step):
        b = min(s, a + step)
        l, m, n1 = d[:, a:b]
        if case["matrix"]:
            j, w = cut(a, b), bright[a:b]
            left = j @ w
        else:
            j = torch.view_as_complex(jones[:, a:b].double().reshape(
                n, b - a, 2).contiguous())
            left = j * x["flux"][0, a:b].double()
        for q in range(n - 1):
            uu, vv, ww = (u[:, q + 1:] - u[:, q:q + 1])[:, :, None] * inv_wl
            f = torch.ones(n - 1 - q, b - a, device="cuda",
                           dtype=torch.float64)
            if case["gaussian"]:
                f *= torch.exp(-(ext[0, a:b] * uu ** 2 +
                                 2 * ext[1, a:b] * uu * vv +
                                 ext[2, a:b] * vv ** 2))
            if case["bandwidth_hz"]:
                f *= _sinc(math.pi * frac * (uu * l + vv * m + ww * n1))
            if case["time_s"]:
                # Rates of change of u, v, w from the Earth's rotation; the
                # station's ECEF x, y are its u, v here.
                xx, yy = math.pi * uu, math.pi * vv
                rot = OMEGA_EARTH * case["time_s"]
                t = (xx * math.sin(ha0) + yy * math.cos(ha0)) * rot
                du = (xx * math.cos(ha0) - yy * math.sin(ha0)) * rot
                f *= _sinc(du * l + t * math.sin(DEC0) * m -
                           t * math.cos(DEC0) * n1)
            first, second = (left[q:q + 1], j[q + 1:]) if case["casa"] else \
                (left[q + 1:], j[q:q + 1])
            if case["matrix"]:
                v = torch.stack(
                    [(f * (first[..., i, 0] * second[..., k, 0].conj() +
                           first[..., i, 1] * second[..., k, 1].conj()))
                     .sum(-1) for i in range(2) for k in range(2)], dim=-1)
            else:
                v = (f * (first * second.conj())).sum(-1)[:, None]
            full[q] = full[q] + v
    out = torch.cat(full[:n - 1])
    return torch.view_as_real(out).reshape(-1, nr)


def _exact_beam(elements, d):
    """The normalised beam of an array of half-wave crossed dipoles."""
    kk = 2 * math.pi * FREQ_HZ / C0
    az, el = POINTING
    point = torch.tensor([[math.cos(el) * math.sin(az)],
                          [math.cos(el) * math.cos(az)], [math.sin(el)]],
                         dtype=torch.float64, device="cuda")
    xyz = elements.double().cuda()
    weight = -kk * (point.T @ xyz)

    def beam(d):
        af = torch.zeros(d.shape[1], dtype=torch.complex128, device="cuda")
        step = max(1, (1 << 25) // xyz.shape[1])
        for a in range(0, d.shape[1], step):
            t = kk * (d[:, a:a + step].T @ xyz) + weight
            af[a:a + step] = torch.polar(torch.ones_like(t), t).sum(1)
        theta = torch.atan2(torch.hypot(d[0], d[1]), d[2])
        phi = torch.atan2(d[1], d[0])
        out = torch.zeros(d.shape[1], 4, dtype=torch.complex128,
                          device="cuda")
        for row, p in enumerate((phi, phi + math.pi / 2)):
            c, st, ct = torch.cos(p), torch.sin(theta), torch.cos(theta)
            t = torch.cos(math.pi / 2 * c * st) / (1 + c * c * (ct * ct - 1))
            out[:, 2 * row] = -c * ct * t * af
            out[:, 2 * row + 1] = torch.sin(p) * t * af
        return out
    norm = (beam(point).abs() ** 2).sum() / 2
    return beam(d) / torch.sqrt(norm)


def exact(case, seed):
    if case["kind"] == "clip":
        return None
    x = _inputs(case, seed)
    n, s, kind = case.get("stations"), case["sources"], case["kind"]
    if kind == "direct":
        return _exact_direct(case, x)
    if kind == "beam":
        b = _exact_beam(x["elements"][0], x["dir"].double())
        return torch.view_as_real(b).reshape(s, 8)
    bright = _brightness(x["flux"])
    if kind == "shared":
        e = torch.view_as_complex(x["beam"].double().reshape(s, 2, 2, 2)
                                  .contiguous())
        c = (e @ bright) @ e.mH
        full = torch.zeros(n, 2, n, 2, device="cuda", dtype=torch.complex128)
        step = 1 << 16
        for a in range(0, s, step):
            k = _phasor(x["uvw"], x["dir"][:, a:a + step])
            for i in range(2):
                for j in range(2):
                    full[:, i, :, j] += (k * c[a:a + step, i, j]) @ \
                        k.conj().T.contiguous()
        return _pick(full, n, False)
    if kind == "stations":
        jones = x["jones"]

        def cut(a, b):
            j = jones[:, a:b].double().reshape(n, b - a, 2, 2, 2)
            k = _phasor(x["uvw"], x["dir"][:, a:b])
            return torch.view_as_complex(j.contiguous()) * k[..., None, None]
        return _contract(cut, bright, n, s, False)[0]

    def cut(a, b):
        d = x["dir"][:, a:b]
        e = torch.stack([_exact_beam(el, d.double()).reshape(-1, 2, 2)
                         for el in x["elements"]])
        return e * _phasor(x["uvw"], d)[..., None, None]
    cross, auto = _contract(cut, bright, n, s, False)
    return {"cross": cross, "auto": auto}
