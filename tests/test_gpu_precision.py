"""Precision study on the plain single-volume shapes (64^3, 8 coils, kooshball 2000 spokes
x 64 samples, NUFFT tolerance 1e-6): per step, the relative L2 error against the FP64
oracle of the build's path (FP32 data, FP64 Toeplitz-kernel build, FP64 CG scalars) and
of an all-FP32 variant (FP32 PSF NUFFT for the kernel, FP32 CG scalars on the host).

Bounds: NUFFT type-1/type-2 1e-5; normal operator 1e-5 (the FP64-built kernel must also
beat the FP32-built one).

CG image after 15 iterations (ConjugateGradient::run, lib/op/opalgs.cpp:50-96):
- On the raw kooshball system the 15th iterate is ill-conditioned in its inputs: the
  oracle's own FP64 CG moves by ~3.5e-5 when b is scaled by (1 + 1e-15), and any
  perturbation of 1e-10 or more (complex64 operator outputs, complex64 vectors, FP32
  dot products, FP64 with 1e-7 noise) lands ~3.3e-2 away, the same for every kind. The
  device CG is therefore held to the envelope of the oracle's FP64 CG under such
  perturbations (complex64-rounded operator inputs/outputs, and Gaussian output noise at
  3x the device operator's measured error, three seeds): at most 1.25x the largest
  distance, and a phantom error within 2 % of the largest.
- On the reference's Tikhonov-regularised operator l2_reg_linop(A, lambda) = A + lambda I
  (python/python/hastypy/base/opalg.py:626-627) with lambda = 0.1 lambda_max the system
  is well posed and the device CG image is held to 1e-5 of the FP64 CG.
"""
import math

import numpy as np
import pytest
import torch

from oracle import oracle as O

pytestmark = [pytest.mark.gpu, pytest.mark.slow]


@pytest.fixture(scope="module")
def setup():
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    from hastycompute_amd import native

    n, C = 64, 8
    co = O.kooshball(2000, 64)
    co32 = co.astype(np.float32)
    cod = co32.astype(np.float64)
    S = O.coil_maps(C, n, seed=1)
    x_true = O.ellipsoid_phantom(n, seed=2)
    return dict(native=native, n=n, C=C, co32=co32, cod=cod, S=S, x_true=x_true)


def rel(a, b):
    return O.rel_l2(np.asarray(a, dtype=np.complex128), np.asarray(b, dtype=np.complex128))


def test_precision_study(setup):
    N = setup["native"]
    n, C, co32, cod, S, x_true = (setup[k] for k in ("n", "C", "co32", "cod", "S", "x_true"))
    dev = torch.device("cuda:0")
    cog = torch.as_tensor(co32).to(dev)
    nvox = n ** 3
    rows = []

    # NUFFT type-2 / type-1 (scaled as CUDANufft::apply)
    f = (x_true * S[0][None]).astype(np.complex64)
    k_gpu = N.nufft(cog, torch.as_tensor(f).to(dev), [n] * 3, 2, -1, 1e-6, 1 / math.sqrt(nvox)).cpu().numpy()
    k_ref = O.nufft_type2(cod, f[0].astype(np.complex128), -1, 1e-12) / math.sqrt(nvox)
    e2 = rel(k_gpu[0], k_ref)
    rng = np.random.default_rng(3)
    c = (rng.standard_normal(cod.shape[1]) + 1j * rng.standard_normal(cod.shape[1])).astype(np.complex64)
    im_gpu = N.nufft(cog, torch.as_tensor(c[None]).to(dev), [n] * 3, 1, 1, 1e-6, 1 / math.sqrt(nvox)).cpu().numpy()
    im_ref = O.nufft_type1(cod, c.astype(np.complex128), [n] * 3, 1, 1e-12) / math.sqrt(nvox)
    e1 = rel(im_gpu[0], im_ref)
    rows += [("NUFFT type-2", e2, None), ("NUFFT type-1", e1, None)]
    print(f"precision: NUFFT done ({e2:.2e}, {e1:.2e})", flush=True)

    # Toeplitz kernels: FP64 build (the path) and an FP32 PSF (all-FP32 variant)
    _, kern64 = N.toeplitz_build(cog, [n] * 3, tol=1e-8, diag=False)
    L = 2 * n
    ones = torch.ones((1, cog.shape[1]), dtype=torch.complex64, device=dev)
    psf32 = N.nufft(cog, ones, [L] * 3, 1, 1, 1e-6, 1.0)[0] / float(L ** 3)
    psf32[0, :, :] = 0
    psf32[:, 0, :] = 0
    psf32[:, :, 0] = 0
    # the operator's real kernel: Re DFT(ifftshift(psf)) / N^d, psf carrying (2N)^-d
    kern32 = (torch.fft.fftn(torch.fft.ifftshift(psf32)).real / float(nvox)).contiguous()
    diag = O.toeplitz_diagonal(cod, [1, n, n, n])
    Sg = torch.as_tensor(S).to(torch.complex64).to(dev)
    xg = torch.as_tensor(x_true).to(torch.complex64).to(dev)
    ref_normal = O.sense_normal_toeplitz(diag, x_true, S, list(range(C)), workers=O.default_threads())
    op64 = N.SenseNormalToeplitz(Sg, kern64[None].contiguous())
    op32 = N.SenseNormalToeplitz(Sg, kern32[None].contiguous())
    en64 = rel(op64.apply(xg).cpu().numpy(), ref_normal)
    en32 = rel(op32.apply(xg).cpu().numpy(), ref_normal)
    rows += [("normal op", en64, en32)]
    print(f"precision: normal op done ({en64:.2e}, {en32:.2e})", flush=True)

    print("\nprecision vs FP64 oracle (relative L2): step | this path | all-FP32 variant", flush=True)
    for name, a, b_ in rows:
        print(f"  {name:18s} {a:.3e}  {'' if b_ is None else f'{b_:.3e}'}", flush=True)
    assert e1 < 1e-5 and e2 < 1e-5
    assert en64 < 1e-5 and en64 <= en32


@pytest.fixture(scope="module")
def cg_setup(setup):
    """b = A^H (A x_true + noise) (sigma = 1e-3 per sample) with exact NUFFTs, the
    oracle operator, and the device operator with the FP64-built kernel."""
    N = setup["native"]
    n, C, co32, cod, S, x_true = (setup[k] for k in ("n", "C", "co32", "cod", "S", "x_true"))
    dev = torch.device("cuda:0")
    cog = torch.as_tensor(co32).to(dev)
    nvox = n ** 3
    rng = np.random.default_rng(4)
    noise = 1e-3 * (rng.standard_normal((C, cod.shape[1])) + 1j * rng.standard_normal((C, cod.shape[1])))
    y = np.stack([O.nufft_type2(cod, (x_true[0] * S[ci]), -1, 1e-12) / math.sqrt(nvox) for ci in range(C)]) + noise
    b = sum(np.conj(S[ci])[None] * O.nufft_type1(cod, y[ci], [n] * 3, 1, 1e-12)[None] / math.sqrt(nvox)
            for ci in range(C))
    diag = O.toeplitz_diagonal(cod, [1, n, n, n])
    Aref = lambda v: O.sense_normal_toeplitz(diag, v, S, list(range(C)), workers=O.default_threads())
    _, kern64 = N.toeplitz_build(cog, [n] * 3, tol=1e-8, diag=False)
    op = N.SenseNormalToeplitz(torch.as_tensor(S).to(torch.complex64).to(dev), kern64[None].contiguous())
    bg = torch.as_tensor(b).to(torch.complex64).to(dev)
    return dict(N=N, b=b, bg=bg, Aref=Aref, op=op, x_true=x_true, cog=cog, S=S)


def test_precision_cg_raw_kooshball(cg_setup):
    N, b, bg, Aref, op, x_true = (cg_setup[k] for k in ("N", "b", "bg", "Aref", "op", "x_true"))
    c64 = lambda a: a.astype(np.complex64).astype(np.complex128)
    ref = O.conjugate_gradient(Aref, b, np.zeros_like(b), 15)
    ulp = O.conjugate_gradient(Aref, b * (1 + 1e-15), np.zeros_like(b), 15) / (1 + 1e-15)
    rounded = O.conjugate_gradient(lambda v: c64(Aref(c64(v))), b, np.zeros_like(b), 15)
    e_op = O.rel_l2(op.apply(bg).cpu().numpy(), Aref(b))
    noisy = []
    for seed in range(3):
        r = np.random.default_rng(seed)

        def Anoisy(v, r=r):
            y = Aref(v)
            return y + 3 * e_op * np.linalg.norm(y) / math.sqrt(y.size) * (
                r.standard_normal(y.shape) + 1j * r.standard_normal(y.shape)) / math.sqrt(2)

        noisy.append(O.conjugate_gradient(Anoisy, b, np.zeros_like(b), 15))
    x, st = N.cg_solve(lambda v, o: op.apply(v, out=o), bg, torch.zeros_like(bg), 15)
    xd = x.cpu().numpy()
    # all-FP32 variant: FP32 scalars read back every iteration
    x32 = torch.zeros_like(bg)
    r = bg - op.apply(x32)
    p = r.clone()
    rz = torch.vdot(r.flatten(), r.flatten()).real
    for _ in range(15):
        Ap = op.apply(p)
        alpha = rz / torch.vdot(p.flatten(), Ap.flatten()).real
        x32 += alpha * p
        r -= alpha * Ap
        rz_new = torch.vdot(r.flatten(), r.flatten()).real
        p = r + (rz_new / rz) * p
        rz = rz_new
    e_dev, e_32 = O.rel_l2(xd, ref), O.rel_l2(x32.cpu().numpy(), ref)
    e_ulp, e_rnd = O.rel_l2(ulp, ref), O.rel_l2(rounded, ref)
    e_noise = [O.rel_l2(xn, ref) for xn in noisy]
    env_d = max([e_rnd] + e_noise)
    env_ph = max(O.rel_l2(xn, x_true) for xn in [ref, rounded] + noisy)
    ph_dev, ph_ref = O.rel_l2(xd, x_true), O.rel_l2(ref, x_true)
    print(f"\nCG 15 it, raw kooshball, vs FP64 CG: device {e_dev:.3e}, all-FP32 {e_32:.3e}; oracle FP64 CG with "
          f"b*(1+1e-15) {e_ulp:.3e}, with complex64-rounded operator {e_rnd:.3e}, with output noise at 3x the "
          f"device operator error ({e_op:.2e}) {', '.join(f'{v:.3e}' for v in e_noise)}; phantom error device "
          f"{ph_dev:.4f}, FP64 CG {ph_ref:.4f}, envelope {env_ph:.4f}", flush=True)
    assert e_dev <= 1.25 * env_d
    assert ph_dev <= 1.02 * env_ph


def test_precision_cg_l2_regularised(cg_setup):
    N, b, bg, Aref, op = (cg_setup[k] for k in ("N", "b", "bg", "Aref", "op"))
    # lambda_max by power iteration on the device operator; the same lambda on both sides
    v = bg.clone()
    for _ in range(30):
        w = op.apply(v)
        lmax = float(torch.linalg.vector_norm(w))
        v = w / lmax
    lam = 0.1 * lmax
    ref = O.conjugate_gradient(lambda u: Aref(u) + lam * u, b, np.zeros_like(b), 15)
    x, st = N.cg_solve(lambda u, o: op.apply(u, out=o), bg, torch.zeros_like(bg), 15, l2=lam)
    xg, _ = N.cg_solve(lambda u, o: op.apply(u, out=o), bg, torch.zeros_like(bg), 15, l2=lam, graph=True)
    e = O.rel_l2(x.cpu().numpy(), ref)
    print(f"\nCG 15 it on A + {lam:.4g} I (0.1 lambda_max): device vs FP64 CG {e:.3e}", flush=True)
    assert e < 1e-5
    assert torch.equal(x, xg)


@pytest.mark.parametrize("dims,M", [((20, 24, 30), 3000), ((64, 64, 64), 0), ((9, 30), 500), ((18,), 40)])
@pytest.mark.parametrize("fp64,weighted", [(False, True), (True, False)])
def test_toeplitz_build_workspace(dims, M, fp64, weighted):
    """The kernel and the diagonal do not depend on where the build's memory comes from: the
    caller's whole workspace, a part of it (unaligned), or none."""
    import torch

    from hastycompute_amd import _capi as C

    gen = torch.Generator(device="cuda:0")
    gen.manual_seed(M + len(dims))
    co = ((torch.rand((len(dims), M), dtype=torch.float64, device="cuda:0", generator=gen) * 2 - 1) * 3.1415926)
    co = co if fp64 else co.to(torch.float32)
    w = torch.rand(M, dtype=torch.float32, device="cuda:0", generator=gen) if weighted else None
    L = [2 * n for n in dims]
    size = int(C.lib().hasty_toeplitz_workspace_size(M, len(dims), C.i64arr(dims), 1e-10))
    assert size > 0
    ws = torch.empty(size + 8, dtype=torch.uint8, device="cuda:0")
    outs = []
    for off, nbytes in ((0, size), (8, size), (8, size // 3), (0, 100), (0, 0)):
        d = torch.empty(L, dtype=torch.complex64, device="cuda:0")
        k = torch.empty(L, dtype=torch.float32, device="cuda:0")
        C.call("hasty_toeplitz_build_ws", co.data_ptr(), int(fp64), M, len(dims), C.i64arr(dims), C.ptr(w), d.data_ptr(),
               k.data_ptr(), 1e-10, ws.data_ptr() + off, nbytes, C.stream_ptr())
        outs.append((d, k))
    scale = float(outs[-1][1].abs().max()) + 1e-30
    for d, k in outs[:-1]:  # tile spreaders add in another order from run to run: 1e-13, below float32
        assert float((k - outs[-1][1]).abs().max()) <= 1e-7 * scale
        assert torch.allclose(d, outs[-1][0], rtol=1e-6, atol=1e-6 * float(outs[-1][0].abs().max()))


@pytest.mark.parametrize("dims", [(32, 24, 32), (20, 24, 30)])
def test_toeplitz_build_waits_for_its_stream(dims):
    """The workspace may still be in use by what its owner queued on the build's stream (a
    block that torch's caching allocator hands on): some 30 ms of fills of the workspace are
    queued before a build on a side stream, which gives the default stream's kernel."""
    from hastycompute_amd import _capi as C

    gen = torch.Generator(device="cuda:0")
    gen.manual_seed(5)
    M = 5000
    co = (torch.rand((3, M), dtype=torch.float32, device="cuda:0", generator=gen) * 2 - 1) * 3.1415926
    L = [2 * n for n in dims]
    size = int(C.lib().hasty_toeplitz_workspace_size(M, 3, C.i64arr(dims), 1e-10))
    ks = []
    torch.cuda.synchronize()
    for stream in (torch.cuda.default_stream(), torch.cuda.Stream()):
        with torch.cuda.stream(stream):
            ws = torch.empty(size, dtype=torch.uint8, device="cuda:0")
            k = torch.empty(L, dtype=torch.float32, device="cuda:0")
            for _ in range(1000):
                ws.fill_(255)  # NaN in every table it would reach
            C.call("hasty_toeplitz_build_ws", co.data_ptr(), 0, M, 3, C.i64arr(dims), None, None, k.data_ptr(), 1e-10,
                   ws.data_ptr(), size, C.stream_ptr())
            ks.append(k)
        stream.synchronize()
    # the tile spreader of the second size adds in another order from run to run
    assert float((ks[1] - ks[0]).abs().max()) <= 1e-7 * float(ks[0].abs().max())


def test_toeplitz_build_without_torch_memory():
    """The workspace is an estimate and comes from torch: where torch has no room for it the
    build allocates what it needs, through the Python wrapper and the C++ operator alike."""
    from hastycompute_amd import native
    from hastycompute_amd.ffi import hasty_sense

    n, M = 64, 20000
    gen = torch.Generator(device="cuda:0")
    gen.manual_seed(7)
    co = (torch.rand((3, M), dtype=torch.float32, device="cuda:0", generator=gen) * 2 - 1) * 3.1415926
    S = torch.randn((1, n, n, n), dtype=torch.complex64)
    x = torch.randn((1, 1, n, n, n), dtype=torch.complex64)

    def both():
        out = torch.zeros_like(x)
        hasty_sense.BatchedSenseNormal([co], S).apply(x, out)
        return native.toeplitz_build(co, [n] * 3, diag=False)[1], out

    k, out = both()
    torch.cuda.synchronize()
    torch.cuda.empty_cache()
    total = torch.cuda.get_device_properties(0).total_memory
    # room for the images, kernels and the operator's grids (some 100 MB), not for 500 MB more
    torch.cuda.set_per_process_memory_fraction((torch.cuda.memory_reserved() + 2**28) / total)
    held = []
    try:
        with pytest.raises(torch.OutOfMemoryError):
            while len(held) < 64:  # blocks of that size that other tests left inside reserved memory
                held.append(torch.empty(2**29 - 2**26, dtype=torch.uint8, device="cuda:0"))
        k2, out2 = both()
    finally:
        torch.cuda.set_per_process_memory_fraction(1.0)
        del held
    assert torch.equal(k, k2) and torch.equal(out, out2)


def test_failed_toeplitz_build_leaves_its_stream_idle():
    """The workspace is free again when the call returns, also when the build refuses its
    sizes after its first launches (a 1-D grid of 20000): what was queued is through."""
    from hastycompute_amd import _capi as C

    M, n = 1000, C.i64arr([5000])
    co = torch.zeros((1, M), dtype=torch.float32, device="cuda:0")
    k = torch.empty(10000, dtype=torch.float32, device="cuda:0")
    ws = torch.empty(2**27, dtype=torch.uint8, device="cuda:0")
    stream = torch.cuda.Stream()
    torch.cuda.synchronize()
    with torch.cuda.stream(stream):
        for _ in range(1000):
            ws.fill_(0)
        with pytest.raises(C.HastyError, match="fine grid too large"):
            C.call("hasty_toeplitz_build_ws", co.data_ptr(), 0, M, 1, n, None, None, k.data_ptr(), 1e-8, ws.data_ptr(),
                   ws.numel(), C.stream_ptr())
        assert stream.query()
    stream.synchronize()
