"""Performance cases of the sparse 3D FFT: what programs have this library do.

A case is one pass through the public entry points on device-resident data.

  call      "pair"      backward into a dense field, then forward with full
                        scaling (a plane-wave code applying a local potential)
            "backward"  sparse set -> field (a density put on its grid)
            "forward"   field -> sparse set, full scaling (a density analysed)
            "bands"     a pair over several bands with one multi_transform
                        call per direction
            "gradient"  energy sum V |psi|^2 of several bands and its gradient
                        with respect to the coefficients, through autograd
  nx ny nz  grid; fill = radius of the index ellipsoid over the grid size
            (0.25: wavefunctions on a density grid; near 0.5: densities)
  bands     transforms of the call (bands, gradient)
  order     "xyz": values sorted by x, y, z; "shells": by |G|, as codes that
            work with G-vector shells store them
  sync      the library's default, synchronous execution mode, else the
            asynchronous one
"""
import math

import numpy as np
import torch

import spfft_amd as sp
from spfft_amd.autograd import sparse_energy_batch


def _case(name, call, nx, ny, nz, dtype, fill, r2c=False, bands=1, order="xyz", sync=False):
    case = {"call": call, "nx": nx, "ny": ny, "nz": nz, "dtype": dtype, "fill": fill, "r2c": r2c,
            "bands": bands, "order": order, "sync": sync}
    return dict(case, name=name) if name else case


def listed():
    return [
        # a small molecule's or unit cell's grid: launches and host time count
        _case("cell_20_f64", "pair", 20, 20, 20, "f64", 0.3),
        # the density of a medium cell, G-vectors kept by shells, default mode
        _case("density_72_r2c_f64", "forward", 72, 72, 72, "f64", 0.47, r2c=True, order="shells",
              sync=True),
        # an elongated cell (a surface slab with its vacuum)
        _case("slab_40_48_150_f64", "pair", 40, 48, 150, "f64", 0.3),
        # a grid size that is no smooth number (taken from a cutoff as it came)
        _case("odd_97_f64", "pair", 97, 97, 97, "f64", 0.3),
        # the size of the reference's own largest unit test
        _case("grid_100_f64", "pair", 100, 100, 100, "f64", 0.3),
        # the headline workload: 128^3, sphere of radius 40
        _case("grid_128_f64", "pair", 128, 128, 128, "f64", 0.3125),
        # a real density put on a large grid in single precision
        _case("density_180_r2c_f32", "backward", 180, 180, 180, "f32", 0.33, r2c=True),
        # the single-band form of the 192^3, radius 60 configuration
        _case("grid_192_f64", "pair", 192, 192, 192, "f64", 0.3125),
        # the largest grid: a big supercell
        _case("grid_256_f64", "pair", 256, 256, 256, "f64", 0.3),
        # bands of a k-point in single precision, one fused call per direction
        _case("bands_96_f32_x16", "bands", 96, 96, 96, "f32", 0.3125, bands=16),
        # bands in double precision at the headline size
        _case("bands_128_f64_x8", "bands", 128, 128, 128, "f64", 0.3125, bands=8),
        # differentiated energy of a few bands
        _case("gradient_60_f64_x6", "gradient", 60, 60, 60, "f64", 0.3, bands=6),
    ]


def _smooth(n):
    """The next size without prime factors above 13 (and 11, 13 at most once)."""
    while True:
        m = n
        for p in (2, 3, 5, 7):
            while m % p == 0:
                m //= p
        if m in (1, 11, 13):
            return n
        n += 1


def _size(rng, largest, smooth):
    n = round(math.exp(rng.uniform(math.log(16), math.log(largest))))
    return _smooth(n) if smooth else n


def draw(rng):
    call = rng.choice(["pair"] * 5 + ["backward", "forward", "bands", "bands", "gradient"])
    # most programs round a grid up to a smooth size, some take it as it comes
    smooth = rng.random() < 0.75
    top = {"pair": 240, "backward": 240, "forward": 240, "bands": 144, "gradient": 112}[call]
    if not smooth:
        top = min(top, 128)
    nx = _size(rng, top, smooth)
    if rng.random() < 0.3:
        ny, nz = (_size(rng, top, smooth) for _ in range(2))
    else:
        ny = nz = nx
    r2c = call not in ("gradient",) and rng.random() < 0.3
    dtype = rng.choice(["f64", "f32"])
    density = call in ("backward", "forward") and r2c
    fill = round(rng.uniform(0.3, 0.48) if density else rng.uniform(0.24, 0.36), 3)
    bands = 1
    if call in ("bands", "gradient"):
        most = max(2, min(32, 12_000_000 // (nx * ny * nz)))
        bands = round(math.exp(rng.uniform(math.log(2), math.log(most))))
    order = "shells" if rng.random() < 0.25 else "xyz"
    return _case("", call, nx, ny, nz, dtype, fill, r2c, bands, order, rng.random() < 0.2)


def _triplets(case):
    """Centred triplets of the ellipsoid |G_d| <= fill * n_d (its hermitian
    half for R2C), int32 (n, 3)."""
    g = []
    for n in (case["nx"], case["ny"], case["nz"]):
        half = min(int(math.ceil(case["fill"] * n)), (n - 1) // 2)
        g.append(np.arange(-half, half + 1))
    r = [max(1.0, case["fill"] * n) for n in (case["nx"], case["ny"], case["nz"])]
    if case["r2c"]:
        g[0] = g[0][g[0] >= 0]
    x, y, z = g[0][:, None, None], g[1][None, :, None], g[2][None, None, :]
    norm = (x / r[0]) ** 2 + (y / r[1]) ** 2 + (z / r[2]) ** 2
    keep = norm <= 1.0 + 1e-9
    if case["r2c"]:
        keep &= (x > 0) | (y > 0) | ((y == 0) & (z >= 0))
    at = np.nonzero(keep)
    t = np.stack([g[d][at[d]] for d in range(3)], axis=1).astype(np.int32)
    if case["order"] == "shells":
        t = t[np.argsort(norm[keep], kind="stable")]
    return np.ascontiguousarray(t)


def _dtypes(case):
    return ((torch.float64, torch.complex128) if case["dtype"] == "f64"
            else (torch.float32, torch.complex64))


def _inputs(case, seed, count, device):
    """Coefficients (bands, count), field(s) and potential of the case, each
    from the seed alone; only what the case's call takes."""
    rng = np.random.default_rng(seed)
    real, cplx = _dtypes(case)
    shape = (case["nz"], case["ny"], case["nx"])
    made = {}
    if case["call"] == "forward":
        field = rng.standard_normal(shape)
        if not case["r2c"]:
            field = field + 1j * rng.standard_normal(shape)
        made["field"] = torch.from_numpy(field).to(device, real if case["r2c"] else cplx)
        return made
    c = rng.standard_normal((case["bands"], count)) + 1j * rng.standard_normal((case["bands"], count))
    if case["r2c"]:
        # the coefficient of G = 0 of a real field is real
        zero = np.nonzero(np.all(_triplets(case) == 0, axis=1))[0]
        c[:, zero] = c[:, zero].real
    made["coeff"] = torch.from_numpy(c).to(device, cplx)
    if case["call"] == "gradient":
        made["potential"] = torch.from_numpy(rng.standard_normal(shape)).to(device, real)
    return made


def prepare(case, seed):
    triplets = _triplets(case)
    device = "cuda"
    count = len(triplets)
    real, cplx = _dtypes(case)
    kind = sp.Transform if case["dtype"] == "f64" else sp.TransformFloat
    first = kind(-1, sp.SPFFT_PU_GPU, sp.SPFFT_TRANS_R2C if case["r2c"] else sp.SPFFT_TRANS_C2C,
                 case["nx"], case["ny"], case["nz"], count, sp.SPFFT_INDEX_TRIPLETS, triplets)
    transforms = [first] + [first.clone() for _ in range(case["bands"] - 1)]
    for t in transforms:
        t.set_execution_mode(sp.SPFFT_EXEC_SYNCHRONOUS if case["sync"]
                             else sp.SPFFT_EXEC_ASYNCHRONOUS)
    state = {"case": case, "transforms": transforms, **_inputs(case, seed, count, device)}
    shape = (case["bands"], case["nz"], case["ny"], case["nx"])
    if case["call"] == "gradient":
        state["coeff"].requires_grad_(True)
    else:
        if "field" not in state:
            state["space"] = torch.empty(shape, dtype=real if case["r2c"] else cplx, device=device)
        if case["call"] != "backward":
            state["out"] = torch.empty((case["bands"], count), dtype=cplx, device=device)
    if case["call"] == "bands":
        # one tensor per band, as band codes hold them
        for name in ("coeff", "space", "out"):
            state[name + "_bands"] = list(state[name])
    return state


def run(state):
    case, transforms = state["case"], state["transforms"]
    if case["call"] == "gradient":
        coeff = state["coeff"]
        coeff.grad = None
        energy = sparse_energy_batch(coeff, state["potential"], transforms,
                                     (case["nx"], case["ny"], case["nz"]))
        energy.backward()
        return {"energy": energy.detach(), "gradient": coeff.grad}
    if case["call"] == "bands":
        sp.multi_transform_backward(transforms, state["coeff_bands"], state["space_bands"])
        sp.multi_transform_forward(transforms, state["space_bands"], state["out_bands"],
                                   [sp.SPFFT_FULL_SCALING] * case["bands"])
        return {"field": state["space"], "values": state["out"]}
    t = transforms[0]
    if case["call"] == "forward":
        t.forward(state["field"], state["out"], sp.SPFFT_FULL_SCALING)
        return {"values": state["out"]}
    t.backward(state["coeff"], state["space"])
    if case["call"] == "backward":
        return {"field": state["space"]}
    t.forward(state["space"], state["out"], sp.SPFFT_FULL_SCALING)
    return {"field": state["space"], "values": state["out"]}


def work(case):
    """Values, their int32 index map and the dense field, each once per
    direction; the radix-2 operation count of the pruned transforms."""
    t = _triplets(case)
    real = 8 if case["dtype"] == "f64" else 4
    nx, ny, nz = case["nx"], case["ny"], case["nz"]
    points = nx * ny * nz
    sticks = len(np.unique(t[:, 0].astype(np.int64) * 4096 + t[:, 1]))
    columns = len(np.unique(t[:, 0]))
    directions = 1 if case["call"] in ("backward", "forward") else 2
    dense = points * real * (1 if case["r2c"] else 2)
    one_way = (2 * real * len(t) + dense) * case["bands"] + 4 * len(t)
    x_lines = ny * nz * (0.5 if case["r2c"] else 1.0)
    flops = 5.0 * (sticks * nz * math.log2(nz) + columns * nz * ny * math.log2(ny)
                   + x_lines * nx * math.log2(nx)) * case["bands"]
    extra = 0
    if case["call"] == "gradient":
        extra = points * real
    return {"bytes": float(directions * one_way + extra), "flops": float(directions * flops)}


def exact(case, seed):
    triplets = _triplets(case)
    dims = (case["nx"], case["ny"], case["nz"])
    made = {k: v.to(torch.float64 if not v.is_complex() else torch.complex128)
            for k, v in _inputs(case, seed, len(triplets), "cpu").items()}
    at = torch.from_numpy(triplets.astype(np.int64) % np.array(dims))
    at = (at[:, 2] * dims[1] + at[:, 1]) * dims[0] + at[:, 0]
    shape = (dims[2], dims[1], dims[0])
    points = dims[0] * dims[1] * dims[2]

    def synthesis(c):
        grid = torch.zeros(points, dtype=torch.complex128)
        grid[at] = c
        if case["r2c"]:
            # f(r) = Re(c_0 + 2 sum over the half of c_G exp(i G r))
            grid = grid * 2.0
            grid[0] = grid[0] * 0.5
        field = torch.fft.ifftn(grid.reshape(shape), norm="forward")
        return field.real.contiguous() if case["r2c"] else field

    def analysis(field):
        return torch.fft.fftn(field.to(torch.complex128)).reshape(-1)[at]

    if case["call"] == "forward":
        return {"values": (analysis(made["field"]) / points)[None]}
    if case["call"] == "gradient":
        energy, gradient = 0.0, []
        for c in made["coeff"]:
            psi = synthesis(c)
            energy = energy + torch.sum(made["potential"] * (psi.real ** 2 + psi.imag ** 2))
            gradient.append(2.0 * analysis(made["potential"] * psi))
        return {"energy": energy, "gradient": torch.stack(gradient)}
    fields = torch.stack([synthesis(c) for c in made["coeff"]])
    if case["call"] == "backward":
        return {"field": fields}
    return {"field": fields, "values": torch.stack([analysis(f) / points for f in fields])}
