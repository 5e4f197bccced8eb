"""Performance cases of the reconstruction path, through the package's public entry points.

A case is a dict of plain values; its "kind" names the call a user's program makes:

- "sense":    the batched Toeplitz SENSE normal operator (native.SenseNormalToeplitz.apply),
              the call of every CG or prox-gradient iteration;
- "cg":       a whole CG-SENSE solve (native.cg_solve on that operator);
- "adjoint":  a type-1 NUFFT (samples to image, native.NufftPlan.execute), the gridding step;
- "forward":  a type-2 NUFFT (image to samples), the forward model, several coils at once;
- "explicit": the drop-in SenseNormal (a type-2 and a type-1 NUFFT per coil);
- "toeplitz": the FP64 build of a trajectory's Toeplitz kernel (native.toeplitz_build);
- "llr":      the locally-low-rank prox over all frames (native.llr_normal_blocks);
- "l1dct":    the L1-DCT prox over the encodings' volumes (native.l1dct_prox_).

Images are ellipsoid phantoms with a little noise, coil maps are smooth Gaussian-magnitude,
linear-phase maps with unit sum of squares, trajectories are golden-means kooshballs.
"""
from __future__ import annotations

import math

import torch

from hastycompute_amd import native

DEV = "cuda:0"
PHI1 = 0.465571231876768  # 3-D golden means
PHI2 = 0.682327803828019


# ---------------------------------------------------------------------------------------
# cases
# ---------------------------------------------------------------------------------------
def listed():
    return [
        # one small volume with the operator's default batches: a low-resolution preview or
        # coil calibration, where launches and latency are what the caller sees
        {"name": "sense_small", "kind": "sense", "dims": "32,32,32", "coils": 8, "problems": 1, "kernels": 1,
         "coil_batch": 4, "problem_batch": 1, "own_maps": False, "spokes": 600, "readout": 64},
        # the five velocity encodings of one cardiac frame of a 4D-flow scan, 128^3 x 16
        {"name": "sense_flow", "kind": "sense", "dims": "128,128,128", "coils": 16, "problems": 5, "kernels": 1,
         "coil_batch": 16, "problem_batch": 4, "own_maps": False, "spokes": 1150, "readout": 128},
        # two requests of the largest served matrix in one launch, each with its own coil
        # maps, coil count and kernel, as the request server batches them
        {"name": "sense_large", "kind": "sense", "dims": "160,160,160", "coils": 20, "problems": 2, "kernels": 2,
         "coil_batch": 16, "problem_batch": 4, "own_maps": True, "spokes": 1000, "readout": 160},
        # an anisotropic matrix as slabs and reduced fields of view give it
        {"name": "sense_odd", "kind": "sense", "dims": "72,100,90", "coils": 10, "problems": 2, "kernels": 1,
         "coil_batch": 4, "problem_batch": 1, "own_maps": False, "spokes": 900, "readout": 128},
        # one whole reconstruction at 64^3 x 8 coils: 10 CG iterations on A + l2 I
        {"name": "cg_recon", "kind": "cg", "dims": "64,64,64", "coils": 8, "problems": 1, "iters": 10,
         "coil_batch": 8, "problem_batch": 1, "spokes": 2000, "readout": 64},
        # gridding of one cardiac frame's samples (one coil) at 128^3
        {"name": "nufft_adjoint", "kind": "adjoint", "dims": "128,128,128", "ntransf": 1, "tol": 1e-6,
         "spokes": 1150, "readout": 128},
        # forward model of four coils on an anisotropic matrix at the drop-in classes' tolerance
        {"name": "nufft_forward", "kind": "forward", "dims": "72,100,90", "ntransf": 4, "tol": 1e-5,
         "spokes": 1500, "readout": 100},
        # the explicit normal operator as programs written for the reference call it
        {"name": "sense_explicit", "kind": "explicit", "dims": "64,64,64", "coils": 8, "spokes": 2000, "readout": 64},
        # set-up of one served request: the FP64 kernel of a weighted trajectory
        {"name": "toeplitz_build", "kind": "toeplitz", "dims": "96,96,96", "spokes": 2500, "readout": 192,
         "tol": 1e-8, "weighted": True},
        # one prox of the LLR-regularised 4D-flow reconstruction: 100 frames in one Casorati matrix
        {"name": "llr_flow", "kind": "llr", "dims": "128,128,128", "frames": 100, "enc": 1, "block": 16, "iters": 1},
        # the five-point form: 20 frames, the encodings stacked in the rows, a reduced field
        # of view and two shifted passes
        {"name": "llr_five", "kind": "llr", "dims": "60,96,77", "frames": 20, "enc": 5, "block": 12, "iters": 2},
        # sparsity prox of the five encodings
        {"name": "l1dct_five", "kind": "l1dct", "dims": "96,128,128", "batch": 5},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _smooth_even(n, hi):
    """Nearest size <= hi whose double has no prime factor above 5."""
    for d in range(hi):
        for m in (n - d, n + d):
            k = m
            for p in (2, 3, 5):
                while k > 1 and k % p == 0:
                    k //= p
            if k == 1 and 8 <= m <= hi:
                return m
    return hi


def _draw_dims(rng, lo, hi, smooth):
    pick = (lambda: _smooth_even(_log_int(rng, lo, hi), hi)) if smooth else (lambda: _log_int(rng, lo, hi))
    n = pick()
    if rng.random() < 0.5:  # isotropic
        d = [n, n, n]
    else:
        d = [pick(), pick(), pick()]
    if smooth and rng.random() < 0.35:  # the matrices scanners are set to most often
        m = rng.choice([32, 64, 96, 128, 160])
        d = [m, m, m] if m <= hi else d
    return ",".join(str(v) for v in d)


def draw(rng):
    kind = rng.choice(["sense", "sense", "cg", "adjoint", "forward", "explicit", "toeplitz", "llr", "l1dct"])
    c = {"kind": kind}
    if kind == "sense":
        c.update(dims=_draw_dims(rng, 24, 160, True), coils=rng.randint(3, 24), problems=rng.randint(1, 5), kernels=1,
                 coil_batch=rng.choice([4, 8, 16]), problem_batch=rng.choice([1, 4]), own_maps=rng.random() < 0.3,
                 spokes=_log_int(rng, 200, 1500), readout=_log_int(rng, 48, 200))
        c["kernels"] = rng.randint(1, c["problems"])
        while work(c)["flops"] > 4.0e10 and c["problems"] * c["coils"] > 1:
            if c["problems"] > 1:
                c["problems"] -= 1
                c["kernels"] = min(c["kernels"], c["problems"])
            else:
                c["coils"] -= 1
    elif kind == "cg":
        c.update(dims=_draw_dims(rng, 24, 80, True), coils=rng.randint(3, 12), problems=rng.randint(1, 3),
                 iters=rng.randint(4, 12), coil_batch=rng.choice([4, 8, 16]), problem_batch=rng.choice([1, 4]),
                 spokes=_log_int(rng, 400, 2500), readout=_log_int(rng, 48, 128))
        while work(c)["flops"] > 4.0e10 and c["coils"] > 1:
            c["coils"] -= 1
    elif kind in ("adjoint", "forward"):
        c.update(dims=_draw_dims(rng, 24, 160, False), ntransf=rng.randint(1, 6), tol=rng.choice([1e-4, 1e-5, 1e-6]),
                 spokes=_log_int(rng, 100, 2500), readout=_log_int(rng, 40, 200))
        vox = math.prod(_dims(c))
        c["ntransf"] = max(1, min(c["ntransf"], int(1.2e7 / vox)))
    elif kind == "explicit":
        c.update(dims=_draw_dims(rng, 24, 96, False), coils=rng.randint(2, 8), spokes=_log_int(rng, 200, 2500),
                 readout=_log_int(rng, 40, 128))
        c["coils"] = max(1, min(c["coils"], int(4.0e6 / math.prod(_dims(c)))))
    elif kind == "toeplitz":
        c.update(dims=_draw_dims(rng, 24, 96, True), spokes=_log_int(rng, 200, 2500), readout=_log_int(rng, 48, 192),
                 tol=rng.choice([1e-8, 1e-10]), weighted=rng.random() < 0.5)
    elif kind == "llr":
        c.update(dims=",".join(str(rng.randint(40, 100)) for _ in range(3)), frames=_log_int(rng, 5, 100),
                 enc=rng.choice([1, 1, 5]), block=rng.choice([8, 12, 16]), iters=rng.randint(1, 2))
        while c["enc"] * c["frames"] * math.prod(_dims(c)) > 1.0e8:
            c["enc"], c["frames"] = 1, max(5, int(c["frames"] * 0.8))
    else:
        c.update(dims=_draw_dims(rng, 24, 128, False), batch=rng.randint(1, 5))
    return c


def _dims(c):
    return [int(v) for v in c["dims"].split(",")]


# ---------------------------------------------------------------------------------------
# inputs
# ---------------------------------------------------------------------------------------
def _gen(seed, device="cpu"):
    g = torch.Generator(device=device)
    g.manual_seed(seed)
    return g


def _randn(shape, seed):
    return torch.randn(shape, dtype=torch.complex64, device=DEV, generator=_gen(seed, DEV))


def _kooshball(spokes, readout, offset):
    n = torch.arange(offset, offset + spokes, dtype=torch.float64, device=DEV)
    uz = torch.remainder(n * PHI1, 1.0) * 2.0 - 1.0
    th = 2.0 * math.pi * torch.remainder(n * PHI2, 1.0)
    r = torch.sqrt(torch.clamp(1.0 - uz * uz, min=0.0))
    dirs = torch.stack([uz, r * torch.cos(th), r * torch.sin(th)])
    t = -math.pi + 2.0 * math.pi * torch.arange(readout, dtype=torch.float64, device=DEV) / readout
    return (dirs[:, :, None] * t[None, None, :]).reshape(3, -1).to(torch.float32).contiguous()


def _coords(c, seed, k=0):
    return _kooshball(c["spokes"], c["readout"], 1 + (seed % 1000) * 7 + 4001 * k)


def _axes(dims):
    ax = [(torch.arange(n, dtype=torch.float32, device=DEV) - n / 2) / n for n in dims]
    return ax[0][:, None, None], ax[1][None, :, None], ax[2][None, None, :]


def _phantom(dims, seed, nell=6):
    g = _gen(seed)
    z, y, x = _axes(dims)
    img = torch.zeros(dims, dtype=torch.complex64, device=DEV)
    for _ in range(nell):
        c = ((torch.rand(3, generator=g) - 0.5) * 0.4).tolist()
        a = (0.05 + 0.2 * torch.rand(3, generator=g)).tolist()
        m, p = torch.rand(2, generator=g).tolist()
        v = complex((0.2 + 0.8 * m) * math.cos(2 * math.pi * p), (0.2 + 0.8 * m) * math.sin(2 * math.pi * p))
        img += v * (((z - c[0]) / a[0]) ** 2 + ((y - c[1]) / a[1]) ** 2 + ((x - c[2]) / a[2]) ** 2 <= 1.0)
    return img


def _images(count, dims, seed):
    x = torch.stack([_phantom(dims, seed * 131 + p) for p in range(count)])
    return x + 0.01 * _randn(x.shape, seed * 131 + 97)


def _coil_maps(coils, dims, seed):
    g = _gen(seed + 5)
    z, y, x = _axes(dims)
    maps = torch.empty((coils, *dims), dtype=torch.complex64, device=DEV)
    for c in range(coils):
        r = (torch.rand(7, generator=g) - 0.5).tolist()
        w = 0.45 + 0.3 * r[3]
        mag = torch.exp(-((z - r[0]) ** 2 + (y - r[1]) ** 2 + (x - r[2]) ** 2) / (2 * w * w))
        maps[c] = torch.polar(mag, 6.0 * (r[4] * z + r[5] * y + r[6] * x))
    maps /= torch.sqrt((maps.abs() ** 2).sum(0, keepdim=True))
    return maps


def _ncoil(c):
    """Coils of each problem: alternating full and about two thirds when every problem brings its own."""
    if not c.get("own_maps"):
        return [c["coils"]] * c["problems"]
    return [c["coils"] if p % 2 == 0 else max(1, (2 * c["coils"] + 2) // 3) for p in range(c["problems"])]


def _kernel_index(c):
    return [p * c["kernels"] // c["problems"] for p in range(c["problems"])]


def _sense_inputs(c, seed):
    dims = _dims(c)
    coords = [_coords(c, seed, k) for k in range(c.get("kernels", 1))]
    sets = c["problems"] if c.get("own_maps") else 1
    smaps = torch.cat([_coil_maps(c["coils"], dims, seed + 11 * s) for s in range(sets)])
    return dims, coords, smaps, _images(c["problems"], dims, seed)


def _sense_operator(c, dims, coords, smaps):
    kern = torch.stack([native.toeplitz_build(co, dims, tol=1e-8, diag=False)[1] for co in coords])
    return native.SenseNormalToeplitz(smaps, kern, coils=list(range(c["coils"])), coil_batch=c["coil_batch"],
                                      problem_batch=c["problem_batch"])


def _l2(c):
    return 0.1 * c["spokes"]  # about a tenth of the kooshball operator's largest eigenvalue


def _weights(c, coords):
    """Radial density compensation, |k|^2 with a floor at the centre."""
    if not c["weighted"]:
        return None
    k2 = (coords.double() ** 2).sum(0) / math.pi ** 2
    return (k2 + 1.0 / c["readout"] ** 2).to(torch.float32)


def _llr_inputs(c, seed):
    dims, F, E = _dims(c), c["frames"], c["enc"]
    ph = _phantom(dims, seed).reshape(1, -1)
    comp = torch.cat([ph.repeat(1, E)] + [ph.repeat(1, E) * 0.2 * _randn((1, E * ph.shape[1]), seed + 20 + i)
                                          for i in range(4)])
    temp = _randn((F, 5), seed + 31) / math.sqrt(5.0)
    x = (temp @ comp).reshape(F, E, *dims)
    x += 0.01 * _randn(x.shape, seed + 32)
    g = _gen(seed + 33)
    shifts = torch.randint(0, c["block"] // 2 + 1, (3, c["iters"]), generator=g).tolist()
    # a little above the noise's largest singular value, about 0.01 of the signal's
    rows = E * c["block"] ** 3
    thresh = 0.015 * (math.sqrt(rows) + math.sqrt(F))
    return x, shifts, thresh


def _l1dct_inputs(c, seed):
    dims = _dims(c)
    x = _images(c["batch"], dims, seed)
    return x, 0.02 * math.sqrt(8.0 * math.prod(dims))


def prepare(case, seed):
    c, kind = case, case["kind"]
    if kind == "sense":
        dims, coords, smaps, x = _sense_inputs(c, seed)
        op = _sense_operator(c, dims, coords, smaps)
        return {"case": c, "op": op, "x": x, "out": torch.empty_like(x), "kidx": _kernel_index(c),
                "ncoil": _ncoil(c) if c["own_maps"] else None, "stride": c["coils"] if c["own_maps"] else 0}
    if kind == "cg":
        dims, coords, smaps, b = _sense_inputs(c, seed)
        return {"case": c, "op": _sense_operator(c, dims, coords, smaps), "b": b, "x0": torch.zeros_like(b)}
    if kind in ("adjoint", "forward"):
        dims = _dims(c)
        co = _coords(c, seed)
        nt, scale = c["ntransf"], 1.0 / math.sqrt(math.prod(dims))
        if kind == "adjoint":
            plan = native.NufftPlan(co, dims, 1, +1, nt, c["tol"], scale)
            return {"case": c, "plan": plan, "c": _randn((nt, co.shape[1]), seed + 3),
                    "f": torch.empty((nt, *dims), dtype=torch.complex64, device=DEV)}
        plan = native.NufftPlan(co, dims, 2, -1, nt, c["tol"], scale)
        return {"case": c, "plan": plan, "f": _images(nt, dims, seed),
                "c": torch.empty((nt, co.shape[1]), dtype=torch.complex64, device=DEV)}
    if kind == "explicit":
        from hastycompute_amd.ffi import hasty_sense

        dims = _dims(c)
        co = _coords(c, seed)
        x = _images(1, dims, seed)
        return {"case": c, "op": hasty_sense.SenseNormal(co, [1, *dims]), "x": x, "out": torch.empty_like(x),
                "smaps": _coil_maps(c["coils"], dims, seed), "coils": list(range(c["coils"]))}
    if kind == "toeplitz":
        co = _coords(c, seed)
        return {"case": c, "coords": co, "w": _weights(c, co)}
    if kind == "llr":
        x, shifts, thresh = _llr_inputs(c, seed)
        b = (c["block"],) * 3
        return {"case": c, "x": x, "out": torch.empty_like(x), "shifts": shifts, "thresh": thresh, "block": b}
    x, thresh = _l1dct_inputs(c, seed)
    return {"case": c, "x": x, "out": torch.empty_like(x), "thresh": thresh}


# ---------------------------------------------------------------------------------------
# one pass
# ---------------------------------------------------------------------------------------
def run(state):
    c = state["case"]
    kind = c["kind"]
    if kind == "sense":
        return state["op"].apply(state["x"], out=state["out"], kernel_index=state["kidx"],
                                 problem_ncoil=state["ncoil"], coil_problem_stride=state["stride"])
    if kind == "cg":
        op = state["op"]
        x, cg_state = native.cg_solve(lambda v, out: op.apply(v, out=out), state["b"], state["x0"], c["iters"],
                                      l2=_l2(c))
        return [x, cg_state]
    if kind == "adjoint":
        state["plan"].execute(state["c"], state["f"])
        return state["f"]
    if kind == "forward":
        state["plan"].execute(state["c"], state["f"])
        return state["c"]
    if kind == "explicit":
        state["op"].apply(state["x"], state["out"], state["smaps"], state["coils"])
        return state["out"]
    if kind == "toeplitz":
        return native.toeplitz_build(state["coords"], _dims(c), weights=state["w"], tol=c["tol"], diag=False)[1]
    # the proxes work in place on the solver's fresh gradient step
    state["out"].copy_(state["x"])
    if kind == "llr":
        return native.llr_normal_blocks(state["out"], state["block"], state["block"], c["iters"], state["thresh"], True,
                                        shifts=state["shifts"])
    return native.l1dct_prox_(state["out"], (True, True, True), state["thresh"])


# ---------------------------------------------------------------------------------------
# what a pass cannot do without
# ---------------------------------------------------------------------------------------
def _fft_flops(lines, L):
    return lines * 5.0 * L * math.log2(max(2, L))


def _toeplitz_apply_flops(n):
    """One zero-padded convolution: the lines that are not zero, there and back."""
    L = [2 * v for v in n]
    return 2 * (_fft_flops(n[0] * n[1], L[2]) + _fft_flops(n[0] * L[2], L[1]) + _fft_flops(L[1] * L[2], L[0]))


def _nufft_flops(n, M, tol):
    """The doubled grid's pruned FFT lines and the kernel's cells of every sample."""
    ns = max(2, min(16, math.ceil(-math.log10(tol / 10.0))))
    L = [2 * v for v in n]
    return (_fft_flops(n[0] * n[1], L[2]) + _fft_flops(n[0] * L[2], L[1]) + _fft_flops(L[1] * L[2], L[0])
            + 4.0 * M * ns ** 3)


def work(case):
    c, n = case, _dims(case)
    vox = math.prod(n)
    M = c.get("spokes", 0) * c.get("readout", 0)
    kind = c["kind"]
    if kind in ("sense", "cg"):
        nc = _ncoil(c)
        applies = c.get("iters", 1)
        maps = sum(nc) if c.get("own_maps") else c["coils"]
        return {"bytes": 16.0 * vox * c["problems"] + 8.0 * vox * maps + 32.0 * vox * c.get("kernels", 1),
                "flops": applies * sum(nc) * (_toeplitz_apply_flops(n) + 16.0 * vox)}
    if kind in ("adjoint", "forward"):
        return {"bytes": 12.0 * M + c["ntransf"] * 8.0 * (M + vox), "flops": c["ntransf"] * _nufft_flops(n, M, c["tol"])}
    if kind == "explicit":
        return {"bytes": 12.0 * M + 16.0 * vox + 8.0 * vox * c["coils"],
                "flops": c["coils"] * (2 * _nufft_flops(n, M, 1e-5) + 16.0 * vox)}
    if kind == "toeplitz":
        return {"bytes": (16.0 if c["weighted"] else 12.0) * M + 32.0 * vox,
                "flops": _nufft_flops([2 * v for v in n], M, c["tol"])
                + _fft_flops(4 * n[0] * n[1], 2 * n[2]) + _fft_flops(4 * n[0] * n[2], 2 * n[1])
                + _fft_flops(4 * n[1] * n[2], 2 * n[0])}
    if kind == "llr":
        F, E = c["frames"], c["enc"]
        nblk = math.prod((v // c["block"]) for v in n)
        return {"bytes": 16.0 * F * E * vox,
                "flops": c["iters"] * nblk * (16.0 * E * c["block"] ** 3 * F * F + 8.0 * F ** 3)}
    # the three cosine transforms there and back at an FFT's cost
    return {"bytes": 16.0 * c["batch"] * vox,
            "flops": 2.0 * c["batch"] * sum(_fft_flops(vox // v, v) for v in n)}


# ---------------------------------------------------------------------------------------
# tolerances
# ---------------------------------------------------------------------------------------
def tolerance(case):
    """About four times the distance from the 64-bit result on an MI355X (in comments)."""
    kind = case["kind"]
    if kind == "sense":
        return {"rel": 5e-7}  # 7e-8 .. 1.2e-7: float32 FFTs
    if kind == "cg":
        return {"rel": 5e-6}  # 1.2e-6 after 10 iterations
    if kind in ("adjoint", "forward"):
        return {"rel": 6.0 * case["tol"]}  # 0.4 .. 1.6 tol: the spreading kernel's own error
    if kind == "explicit":
        return {"rel": 3e-5}  # 7.7e-6, at the drop-in classes' default tolerance of 1e-5
    if kind == "toeplitz":
        return {"rel": 1.5e-7}  # 3.1e-8: the rounding to float32
    if kind == "llr":
        return {"rel": 8e-5}  # 1e-5 .. 2e-5: float32 Gram matrices square the conditioning
    return {"rel": 2e-6}  # 5.5e-7: float32 sums of up to 128 terms per axis, there and back


# ---------------------------------------------------------------------------------------
# the same results in 64 bits, by plain torch
# ---------------------------------------------------------------------------------------
def _phases(coords, dims, sign, lo=None):
    """exp(sign i m x) per axis, [n, M] complex128, m = index - n // 2."""
    out = []
    for d, n in enumerate(dims):
        m = torch.arange(n, dtype=torch.float64, device=DEV) - n // 2
        ang = sign * m[:, None] * coords[d].double()[None, :]
        out.append(torch.polar(torch.ones_like(ang), ang))
    return out


def _chunks(M, rows):
    step = max(256, int(6.0e7 / rows))
    return [slice(a, min(M, a + step)) for a in range(0, M, step)]


def _direct_type1(coords, values, dims, sign=+1):
    out = torch.zeros((dims[0] * dims[1], dims[2]), dtype=torch.complex128, device=DEV)
    for s in _chunks(coords.shape[1], dims[0] * dims[1]):
        e0, e1, e2 = _phases(coords[:, s], dims, sign)
        a = ((e0 * values[s][None, :])[:, None, :] * e1[None, :, :]).reshape(dims[0] * dims[1], -1)
        out += a @ e2.T.contiguous()
    return out.reshape(dims)


def _direct_type2(coords, img, dims, sign=-1):
    out = torch.empty(coords.shape[1], dtype=torch.complex128, device=DEV)
    f = img.reshape(dims[0] * dims[1], dims[2])
    for s in _chunks(coords.shape[1], dims[0] * dims[1]):
        e0, e1, e2 = _phases(coords[:, s], dims, sign)
        t = (f @ e2).reshape(dims[0], dims[1], -1)
        out[s] = ((t * e1[None, :, :]).sum(1) * e0).sum(0)
    return out


def _exact_kernel(coords, dims, weights=None):
    """Eigenvalues of the doubled circulant embedding, over prod N."""
    L = [2 * n for n in dims]
    w = torch.ones(coords.shape[1], dtype=torch.float64, device=DEV) if weights is None else weights.double()
    psf = _direct_type1(coords, w.to(torch.complex128), L)
    psf[0], psf[:, 0], psf[:, :, 0] = 0, 0, 0  # never reach a cropped output
    return torch.fft.fftn(torch.fft.ifftshift(psf)).real / math.prod(dims)


def _exact_normal(x, smaps, kern):
    L, n = list(kern.shape), list(x.shape)
    out = torch.zeros_like(x)
    for s in smaps:
        s = s.to(torch.complex128)
        y = torch.fft.ifftn(torch.fft.fftn(s * x, s=L) * kern)
        out += s.conj() * y[:n[0], :n[1], :n[2]]
    return out


def _direct_cost(c):
    """Complex multiply-adds of the direct sums."""
    n, M = _dims(c), c.get("spokes", 0) * c.get("readout", 0)
    doubled = 8 if c["kind"] in ("sense", "cg", "toeplitz") else 1
    times = {"explicit": 2 * c.get("coils", 1), "adjoint": c.get("ntransf", 1), "forward": c.get("ntransf", 1)}
    return doubled * math.prod(n) * M * times.get(c["kind"], c.get("kernels", 1))


def exact(case, seed):
    c, kind = case, case["kind"]
    if _direct_cost(c) > 1.6e13:  # direct sums of more than about 20 seconds
        return None
    if kind == "sense":
        dims, coords, smaps, x = _sense_inputs(c, seed)
        kern = [_exact_kernel(co, dims) for co in coords]
        out = torch.empty(x.shape, dtype=torch.complex128, device=DEV)
        for p, (k, nc) in enumerate(zip(_kernel_index(c), _ncoil(c))):
            first = p * c["coils"] if c["own_maps"] else 0
            out[p] = _exact_normal(x[p].to(torch.complex128), smaps[first:first + nc], kern[k])
        return out
    if kind == "cg":
        dims, coords, smaps, b = _sense_inputs(c, seed)
        kern = _exact_kernel(coords[0], dims)
        xs = []
        for p in range(c["problems"]):
            r = b[p].to(torch.complex128)
            x, q = torch.zeros_like(r), r.clone()
            rz = torch.vdot(r.flatten(), r.flatten()).real
            for _ in range(c["iters"]):
                Aq = _exact_normal(q, smaps, kern) + _l2(c) * q
                alpha = rz / torch.vdot(q.flatten(), Aq.flatten()).real
                x, r = x + alpha * q, r - alpha * Aq
                rz_new = torch.vdot(r.flatten(), r.flatten()).real
                q = r + (rz_new / rz) * q
                rz = rz_new
            xs.append(x)
        return [torch.stack(xs), None]
    if kind in ("adjoint", "forward"):
        dims, co = _dims(c), _coords(c, seed)
        scale = 1.0 / math.sqrt(math.prod(dims))
        if kind == "adjoint":
            v = _randn((c["ntransf"], co.shape[1]), seed + 3).to(torch.complex128)
            return torch.stack([scale * _direct_type1(co, t, dims) for t in v])
        f = _images(c["ntransf"], dims, seed).to(torch.complex128)
        return torch.stack([scale * _direct_type2(co, t, dims) for t in f])
    if kind == "explicit":
        dims, co = _dims(c), _coords(c, seed)
        x = _images(1, dims, seed)[0].to(torch.complex128)
        out = torch.zeros_like(x)
        for s in _coil_maps(c["coils"], dims, seed):
            s = s.to(torch.complex128)
            out += s.conj() * _direct_type1(co, _direct_type2(co, s * x, dims), dims)
        return (out / math.prod(dims))[None]
    if kind == "toeplitz":
        co = _coords(c, seed)
        # native.toeplitz_build's kernel also carries the inverse transform's 1 / prod 2N
        return _exact_kernel(co, _dims(c), _weights(c, co)) / math.prod(2 * v for v in _dims(c))
    if kind == "llr":
        return _exact_llr(c, seed)
    x, thresh = _l1dct_inputs(c, seed)
    y = x.to(torch.complex128)
    mats = [_dct_matrix(n) for n in _dims(c)]
    for d, m in enumerate(mats):
        y = _along(y, m, d + 1)
    mag = y.abs()
    y = y * torch.where(mag > thresh, (mag - thresh) / mag, torch.zeros_like(mag))
    for d, m in enumerate(mats):
        y = _along(y, torch.linalg.inv(m), d + 1)
    return y


def _dct_matrix(n):
    i = torch.arange(n, dtype=torch.float64, device="cpu")
    return 2.0 * torch.cos(math.pi * i[:, None] * (2.0 * i[None, :] + 1.0) / (2.0 * n))


def _along(y, m, dim):
    m = m.to(device=y.device, dtype=y.dtype)
    t = y.movedim(dim, 0).contiguous()
    return (m @ t.reshape(t.shape[0], -1)).reshape(t.shape).movedim(0, dim).contiguous()


def _exact_llr(c, seed):
    x, shifts, thresh = _llr_inputs(c, seed)
    x = x.to(torch.complex128)
    dims, b, F = _dims(c), c["block"], c["frames"]
    for it in range(c["iters"]):
        corners = [[v for v in range(shifts[d][it], (dims[d] // b - 1) * b + shifts[d][it] + 1, b) if v + b < dims[d]]
                   for d in range(3)]
        where = [(i, j, k) for i in corners[0] for j in corners[1] for k in corners[2]]
        mats = [x[:, :, i:i + b, j:j + b, k:k + b].reshape(F, -1) for i, j, k in where]
        if not mats:
            continue
        grams = torch.stack([a @ a.conj().T.contiguous() for a in mats]).cpu()  # frames x frames
        lam, vec = torch.linalg.eigh(grams)
        s = torch.sqrt(torch.clamp(lam, min=0.0))
        g = torch.where(s > thresh, (s - thresh) / torch.clamp(s, min=1e-300), torch.zeros_like(s))
        w = ((vec * g[:, None, :]) @ vec.conj().transpose(1, 2).contiguous()).to(x.device)
        for (i, j, k), a, m in zip(where, mats, w):
            x[:, :, i:i + b, j:j + b, k:k + b] = (m @ a).reshape(F, c["enc"], b, b, b)
    return x
