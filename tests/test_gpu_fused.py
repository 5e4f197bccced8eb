"""GPU parity of the fused three-kernel Toeplitz SENSE normal operator (layouts 1 and 2)
against the FP64 oracle and against the generic five-pass path (layout 0)."""
import numpy as np
import pytest
import torch

from oracle import oracle as O

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def N():
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    from hastycompute_amd import native

    return native


def g(a, dtype=torch.complex64):
    return torch.as_tensor(np.ascontiguousarray(a)).to(dtype).cuda()


def h(t):
    torch.cuda.synchronize()
    return t.detach().cpu().numpy().astype(np.complex128)


def rnd(rng, shape):
    return rng.standard_normal(shape) + 1j * rng.standard_normal(shape)


def maps(rng, C, shape):
    m = rnd(rng, (C,) + shape) * 0.3 + 1.0
    return m / np.sqrt(np.sum(np.abs(m) ** 2, axis=0, keepdims=True))


@pytest.mark.parametrize("N0,Nn,C,cb,P", [(32, 32, 3, 2, 2), (40, 64, 4, 4, 3), (24, 96, 2, 1, 1), (20, 32, 5, 3, 4),
                                         (8, 128, 3, 2, 3),
                                         # N = 160: coset kernels one coset per step, the
                                         # inverse in two row halves (N0 = 20: a short last
                                         # group of 8 planes); 2 N0 = 320 and 300 z lines
                                         (8, 160, 3, 2, 3), (20, 160, 2, 1, 2), (160, 32, 2, 2, 2),
                                         (150, 32, 2, 1, 1)])
def test_fused_vs_oracle(N, N0, Nn, C, cb, P):
    rng = np.random.default_rng(N0 + Nn + C)
    shape = (N0, Nn, Nn)
    S = maps(rng, C, shape)
    cos = [rng.uniform(-np.pi, np.pi, (3, 3000)) for _ in range(2)]
    kern = []
    diags = []
    for co in cos:
        _, k = N.toeplitz_build(g(co, torch.float32), list(shape), diag=False)
        kern.append(k)
        diags.append(O.toeplitz_diagonal(co.astype(np.float32).astype(np.float64), [1, *shape]))
    K = torch.stack(kern)
    x = rnd(rng, (P,) + shape)
    sub = rnd(rng, (P,) + shape)
    kidx = [p % 2 for p in range(P)][::-1]
    coils = list(range(C))[::-1]
    op = N.SenseNormalToeplitz(g(S), K, coils=coils, coil_batch=cb, problem_batch=2)
    assert op.layout != 0
    out = h(op.apply(g(x), kernel_index=kidx))
    outs = h(op.apply(g(x), kernel_index=kidx, sub=g(sub)))
    for p in range(P):
        ref = O.sense_normal_toeplitz(diags[kidx[p]], x[p:p + 1], S, coils)
        e = O.rel_l2(out[p:p + 1], ref)
        es = O.rel_l2(outs[p:p + 1], ref - sub[p:p + 1])
        print(f"fused N0={N0} N={Nn} C={C} cb={cb} p={p}: {e:.2e} (sub {es:.2e})", flush=True)
        assert e < 1e-5 and es < 1e-5


def test_fused_matches_generic_and_oracle_at_128(N):
    # the benchmark size: 128^3, two coils, kooshball kernel; the oracle gets the GPU-built
    # complex diagonal, so this pins the fused FFT pipeline itself at L = 256
    rng = np.random.default_rng(128)
    n, C = 128, 2
    co = O.kooshball(1000, 128)
    cog = g(co, torch.float32)
    diag, kern = N.toeplitz_build(cog, [n, n, n], tol=1e-8)
    S = g(maps(rng, C, (n, n, n)))
    x = g(rnd(rng, (1, n, n, n)))
    fused = N.SenseNormalToeplitz(S, kern, coil_batch=2)
    generic = N.SenseNormalToeplitz(S, kern, coil_batch=2, fused=False)
    assert fused.layout != 0 and generic.layout == 0
    of = h(fused.apply(x))
    og = h(generic.apply(x))
    e_fg = O.rel_l2(of, og)
    ref = O.sense_normal_toeplitz(h(diag)[None], h(x), h(S), [0, 1], workers=O.default_threads())
    e_f = O.rel_l2(of, ref)
    print(f"128^3: fused vs generic {e_fg:.2e}, fused vs oracle FFT pipeline {e_f:.2e}", flush=True)
    assert e_fg < 1e-5 and e_f < 1e-5


def test_fused_repeatable(N):
    # same inputs, same launch sequence -> identical bits (no atomics in the fused path)
    rng = np.random.default_rng(3)
    shape = (32, 64, 64)
    S = g(maps(rng, 3, shape))
    co = rng.uniform(-np.pi, np.pi, (3, 2000))
    _, k = N.toeplitz_build(g(co, torch.float32), list(shape), diag=False)
    op = N.SenseNormalToeplitz(S, k, coil_batch=3)
    x = g(rnd(rng, (2,) + shape))
    a = op.apply(x).clone()
    b = op.apply(x).clone()
    assert torch.equal(a, b)


def test_fused_160_every_variant_runs_the_coset_kernels(N):
    # at N1 = N2 = 160 only the coset kernels fit in LDS: every sense_xy_variant value
    # prepares layout 1 and gives the same bits, which match the oracle
    from hastycompute_amd import _capi as C

    rng = np.random.default_rng(16)
    shape = (12, 160, 160)
    Sn = maps(rng, 3, shape)
    co = rng.uniform(-np.pi, np.pi, (3, 6000))
    _, k = N.toeplitz_build(g(co, torch.float32), list(shape), diag=False)
    x = rnd(rng, (2,) + shape)
    prev = C.get_option("sense_xy_variant")
    outs = []
    try:
        for v in (0, 1, 2, 3):
            C.set_option("sense_xy_variant", v)
            op = N.SenseNormalToeplitz(g(Sn), k, coil_batch=2, problem_batch=2)
            assert op.layout == 1
            outs.append(op.apply(g(x)).clone())
    finally:
        C.set_option("sense_xy_variant", prev)
    assert all(torch.equal(outs[0], o) for o in outs[1:])
    diag = O.toeplitz_diagonal(co.astype(np.float32).astype(np.float64), [1, *shape])
    got = h(outs[0])
    for p in range(2):
        e = O.rel_l2(got[p:p + 1], O.sense_normal_toeplitz(diag, x[p:p + 1], Sn, [0, 1, 2]))
        print(f"160: problem {p}: {e:.2e}", flush=True)
        assert e < 1e-5


def test_prepared_layout_survives_option_change(N):
    # kernels prepared for the register plane kernels (layout 2 at N1 = N2 = 128) keep
    # running them after the sense_xy_variant option changes, and coset-prepared kernels
    # (layout 1) keep the coset order; both agree with the oracle-checked default
    from hastycompute_amd import _capi as C

    rng = np.random.default_rng(8)
    shape = (8, 128, 128)
    S = g(maps(rng, 2, shape))
    co = rng.uniform(-np.pi, np.pi, (3, 3000))
    _, k = N.toeplitz_build(g(co, torch.float32), list(shape), diag=False)
    x = g(rnd(rng, (1,) + shape))
    prev = C.get_option("sense_xy_variant")
    try:
        C.set_option("sense_xy_variant", 2)
        op2 = N.SenseNormalToeplitz(S, k, coil_batch=2)
        C.set_option("sense_xy_variant", 1)
        op1 = N.SenseNormalToeplitz(S, k, coil_batch=2)
        assert (op2.layout, op1.layout) == (2, 1)
        a = h(op2.apply(x))  # option now 1: still the register kernels
        b = h(op1.apply(x))
        C.set_option("sense_xy_variant", 2)
        c = h(op1.apply(x))  # option now 2: still the coset kernels
    finally:
        C.set_option("sense_xy_variant", prev)
    assert O.rel_l2(a, b) < 1e-5 and O.rel_l2(c, b) < 1e-5


@pytest.mark.parametrize("N0", [128, 160])
@pytest.mark.parametrize("variant", [0, 1, 2, 3])
def test_zconv_variants_vs_oracle(N, variant, N0):
    # every z-convolution kernel at N0 = 128 (2N0 = 256): 16 or 8 columns per workgroup,
    # one or two LDS transpose buffers; at N0 = 160 (2N0 = 320) the 20 x 16 register form
    # with one (0) or two (2) buffers and the LDS Stockham form (1, 3); three problems with
    # their own kernels
    from hastycompute_amd import _capi as C

    rng = np.random.default_rng(40 + variant)
    shape = (N0, 32, 32)
    S = maps(rng, 3, shape)
    cos = [rng.uniform(-np.pi, np.pi, (3, 3000)) for _ in range(2)]
    kern, diags = [], []
    for co in cos:
        _, k = N.toeplitz_build(g(co, torch.float32), list(shape), diag=False)
        kern.append(k)
        diags.append(O.toeplitz_diagonal(co.astype(np.float32).astype(np.float64), [1, *shape]))
    x = rnd(rng, (3,) + shape)
    kidx = [1, 0, 1]
    prev = C.get_option("sense_zconv_variant")
    try:
        C.set_option("sense_zconv_variant", variant)
        op = N.SenseNormalToeplitz(g(S), torch.stack(kern), coil_batch=3, problem_batch=3)
        out = h(op.apply(g(x), kernel_index=kidx))
    finally:
        C.set_option("sense_zconv_variant", prev)
    for p in range(3):
        e = O.rel_l2(out[p:p + 1], O.sense_normal_toeplitz(diags[kidx[p]], x[p:p + 1], S, [0, 1, 2]))
        print(f"z-conv variant {variant} problem {p}: {e:.2e}", flush=True)
        assert e < 1e-5


@pytest.mark.parametrize("n", [32, 64, 96, 128])
@pytest.mark.parametrize("coil_batch", [2, 5])
def test_split_launches_equal_whole_launches(N, n, coil_batch):
    """A few problems split the plane kernels by coils (coil images, then a coil sum), many
    do not; a problem's result is the same to the bit either way, with coil chunks that
    accumulate, uneven coil counts and a subtracted term."""
    C, P = 5, {32: 16, 64: 8, 96: 3, 128: 2}[n]  # P problems fill the GPU, one does not
    gen = torch.Generator(device="cuda:0")
    gen.manual_seed(n + coil_batch)
    smaps = torch.randn((C, n, n, n), dtype=torch.complex64, device="cuda:0", generator=gen)
    kern = torch.rand((2 * n, 2 * n, 2 * n), dtype=torch.float32, device="cuda:0", generator=gen)
    x = torch.randn((P, n, n, n), dtype=torch.complex64, device="cuda:0", generator=gen)
    sub = torch.randn((P, n, n, n), dtype=torch.complex64, device="cuda:0", generator=gen)
    op = N.SenseNormalToeplitz(smaps, kern, coil_batch=coil_batch, problem_batch=P)
    counts = [C - p % 4 for p in range(P)]
    whole = op.apply(x, sub=sub)
    uneven = op.apply(x, sub=sub, problem_ncoil=counts)
    for p in (0, 1, P - 1):
        xp, sp = x[p:p + 1].contiguous(), sub[p:p + 1].contiguous()
        assert torch.equal(op.apply(xp, sub=sp)[0], whole[p])
        assert torch.equal(op.apply(xp, sub=sp, problem_ncoil=counts[p:p + 1])[0], uneven[p])
    # the split result against the same convolution in FP64
    ref = torch.zeros((n, n, n), dtype=torch.complex128, device="cuda:0")
    kd = kern.double()
    for s in smaps.to(torch.complex128):
        y = torch.fft.ifftn(torch.fft.fftn(s * x[0], s=[2 * n] * 3) * kd) * float((2 * n) ** 3)
        ref += s.conj() * y[:n, :n, :n]
    ref -= sub[0]
    err = float(torch.linalg.vector_norm(whole[0] - ref) / torch.linalg.vector_norm(ref))
    assert err < 1e-6, err


@pytest.mark.parametrize("n,n0,P,C,split", [
    (128, 128, 1, 16, True), (128, 128, 1, 2, True), (128, 96, 2, 2, False), (128, 160, 1, 2, False), (128, 96, 2, 3, False),
    (96, 160, 1, 2, False), (96, 96, 1, 3, True), (64, 64, 1, 8, True), (64, 96, 4, 3, False), (64, 96, 2, 4, True),
    (32, 32, 1, 4, True), (32, 32, 1, 2, False), (32, 48, 4, 2, False), (128, 128, 2, 8, False)])
def test_inverse_split_by_coils_where_it_pays(N, n, n0, P, C, split):
    """The inverse plane launch writes coil images and sums them only where that was measured
    to be faster; the result is the same to the bit (see the test above)."""
    gen = torch.Generator(device="cuda:0")
    gen.manual_seed(n0)
    smaps = torch.randn((C, n0, n, n), dtype=torch.complex64, device="cuda:0", generator=gen)
    kern = torch.rand((2 * n0, 2 * n, 2 * n), dtype=torch.float32, device="cuda:0", generator=gen)
    x = torch.randn((P, n0, n, n), dtype=torch.complex64, device="cuda:0", generator=gen)
    op = N.SenseNormalToeplitz(smaps, kern, coil_batch=C, problem_batch=P)
    assert op.layout != 0
    op.apply(x)
    N.timing_enable(True)
    op.apply(x)
    torch.cuda.synchronize()
    names = N.timing_read()
    N.timing_enable(False)
    assert ("sense_coil_sum" in names) == split, names


@pytest.mark.parametrize("n0", [32, 64, 96, 128, 160])
@pytest.mark.parametrize("narrow", [False, True])
def test_z_convolution_lengths(N, n0, narrow):
    """The register z-convolutions (2 N0 = 64 .. 320; coil groups of one and of several
    coils, one and two problems per launch) against the same convolution in FP64. Float32
    FFTs of 15 levels there and back stay below 15 * 2^-23 = 1.8e-6."""
    from hastycompute_amd import _capi

    C, n = 5, 32
    gen = torch.Generator(device="cuda:0")
    gen.manual_seed(n0)
    smaps = torch.randn((C, n0, n, n), dtype=torch.complex64, device="cuda:0", generator=gen)
    kern = torch.rand((2, 2 * n0, 2 * n, 2 * n), dtype=torch.float32, device="cuda:0", generator=gen)
    x = torch.randn((2, n0, n, n), dtype=torch.complex64, device="cuda:0", generator=gen)
    prev = _capi.get_option("sense_zconv_variant")
    _capi.set_option("sense_zconv_variant", 1 if narrow else 2)
    try:
        outs = [N.SenseNormalToeplitz(smaps, kern, coil_batch=cb, problem_batch=pb).apply(x, kernel_index=[1, 0])
                for cb, pb in ((5, 2), (2, 1))]
    finally:
        _capi.set_option("sense_zconv_variant", prev)
    for p in range(2):
        ref = torch.zeros((n0, n, n), dtype=torch.complex128, device="cuda:0")
        for s in smaps.to(torch.complex128):
            y = torch.fft.ifftn(torch.fft.fftn(s * x[p], s=[2 * n0, 2 * n, 2 * n]) * kern[1 - p].double())
            ref += s.conj() * y[:n0, :n, :n] * float(8 * n0 * n * n)
        for out in outs:
            err = float(torch.linalg.vector_norm(out[p] - ref) / torch.linalg.vector_norm(ref))
            assert err < 1.8e-6, err


@pytest.mark.parametrize("n", [50, 75, 80, 81, 96, 100, 108, 120, 125, 128, 135, 144, 150, 160])
def test_long_register_lines_equal_lds_passes(N, n):
    """The lengths with a step of more than 16 values, which take the register form from some
    number of lines on: passes above it (convolved, strided, contiguous), as below."""
    from hastycompute_amd import _capi

    gen = torch.Generator(device="cuda:0")
    gen.manual_seed(n)
    for dims in ([n, 25, 24], [72, n, 60], [125, 108, n] if n > 50 else [162, 162, n]):
        smaps = torch.randn([2] + dims, dtype=torch.complex64, device="cuda:0", generator=gen)
        kern = torch.rand([2 * d for d in dims], dtype=torch.float32, device="cuda:0", generator=gen)
        x = torch.randn([1] + dims, dtype=torch.complex64, device="cuda:0", generator=gen)
        op = N.SenseNormalToeplitz(smaps, kern, coil_batch=2, fused=False)
        prev = _capi.get_option("fft_r16")
        outs = []
        try:
            for v in (0, 1):
                _capi.set_option("fft_r16", v)
                outs.append(op.apply(x))
        finally:
            _capi.set_option("fft_r16", prev)
        if any(2 * d in (128, 192, 256, 320) for d in dims):  # four-step plain passes, see below
            err = float(torch.linalg.vector_norm(outs[0] - outs[1]) / torch.linalg.vector_norm(outs[0]))
            assert err < 2e-6, err
        else:
            assert torch.equal(outs[0], outs[1])


@pytest.mark.parametrize("dims", [(16, 16, 50), (16, 16, 100), (16, 16, 144), (16, 16, 160), (160, 8, 8), (8, 108, 8)])
def test_short_launches_of_long_lines(N, dims):
    """Passes of few long lines run no slower than on the LDS kernel (a fifth allowed for the
    clock; two register steps for every pass took 1.2 to 1.5 times as long)."""
    from hastycompute_amd import _capi

    gen = torch.Generator(device="cuda:0")
    gen.manual_seed(1)
    smaps = torch.randn((8, *dims), dtype=torch.complex64, device="cuda:0", generator=gen)
    kern = torch.rand([2 * d for d in dims], dtype=torch.float32, device="cuda:0", generator=gen)
    x = torch.randn((1, *dims), dtype=torch.complex64, device="cuda:0", generator=gen)
    op = N.SenseNormalToeplitz(smaps, kern, coil_batch=4, fused=False)
    prev = _capi.get_option("fft_r16")
    best = {}
    try:
        for v in (0, 1) * 6:
            _capi.set_option("fft_r16", v)
            op.apply(x)
            N.timing_enable(True)
            for _ in range(5):
                op.apply(x)
            torch.cuda.synchronize()
            ms = N.timing_read()["fft_axis"][0]
            best[v] = min(ms, best.get(v, ms))
    finally:
        N.timing_enable(False)
        _capi.set_option("fft_r16", prev)
    print(f"passes of {dims} x 8 coils: {200 * best[0]:.0f} us LDS, {200 * best[1]:.0f} us as chosen", flush=True)
    assert best[1] <= 1.2 * best[0], best


@pytest.mark.parametrize("n", [24, 30, 32, 36, 40, 45, 48, 50, 54, 60, 64, 72, 75, 80, 81, 90, 96, 100, 108, 120, 125,
                               128, 135, 144, 150, 160])
def test_register_lines_equal_lds_passes(N, n):
    """Generic normal operator (multiplied, plain, convolved and accumulated passes; each
    axis in turn as the long one; line counts that are no multiple of a bundle): the
    two-step register lines give the LDS passes' bits. Lengths 128, 192, 256 and 320 also
    have a four-step form for the plain passes, with its own roundings: there 15 levels
    there and back bound the distance, 2e-6."""
    from hastycompute_amd import _capi

    gen = torch.Generator(device="cuda:0")
    gen.manual_seed(n)
    for dims in ([n, 10, 15], [10, n, 15], [10, 15, n]):
        smaps = torch.randn([3] + dims, dtype=torch.complex64, device="cuda:0", generator=gen)
        kern = torch.rand([2 * d for d in dims], dtype=torch.float32, device="cuda:0", generator=gen)
        x = torch.randn([2] + dims, dtype=torch.complex64, device="cuda:0", generator=gen)
        op = N.SenseNormalToeplitz(smaps, kern, coil_batch=2, fused=False)
        prev = _capi.get_option("fft_r16")
        outs = []
        try:
            for v in (0, 1):
                _capi.set_option("fft_r16", v)
                outs.append(op.apply(x, sub=x))
        finally:
            _capi.set_option("fft_r16", prev)
        if 2 * n in (128, 192, 256, 320):
            err = float(torch.linalg.vector_norm(outs[0] - outs[1]) / torch.linalg.vector_norm(outs[0]))
            assert err < 2e-6, err
        else:
            assert torch.equal(outs[0], outs[1])
