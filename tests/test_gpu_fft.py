"""HIP FFTs against numpy's pocketfft with DFTpy's normalisation
(field.py:373-390,739-764): forward * dV, inverse / dV."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu

SHAPES = [(8, 8, 8), (6, 10, 15), (20, 30, 22), (36, 36, 72), (7, 11, 13), (1, 6, 10), (5, 1, 9), (32, 32, 32),
          (27, 25, 49), (96, 96, 96), (128, 64, 56)]


def _grid(shape, dtype, full=False):
    from dftpy_amd import DirectGrid
    lat = np.array([[7.1, 0.2, 0.0], [0.3, 8.0, 0.1], [0.0, 0.5, 9.3]])
    return DirectGrid(lat, shape, full=full, dtype=dtype)


def _tol(dtype):
    return 1e-12 if dtype == torch.float64 else 2e-6


@pytest.mark.parametrize("shape", SHAPES)
@pytest.mark.parametrize("dtype", [torch.float64, torch.float32])
def test_r2c_c2r(shape, dtype):
    from dftpy_amd import DirectField
    g = _grid(shape, dtype)
    rng = np.random.default_rng(hash(shape) % 2 ** 32)
    f = rng.standard_normal(shape)
    F = DirectField(g, data=f).fft()
    ref = np.fft.rfftn(f) * g.dV
    got = F.data.cpu().numpy()
    assert got.shape == ref.shape
    assert np.max(np.abs(got - ref)) <= _tol(dtype) * np.max(np.abs(ref)) * 4
    back = F.ifft().data.cpu().numpy()
    assert np.max(np.abs(back - f)) <= _tol(dtype) * np.max(np.abs(f)) * 8
    # irfftn semantics on a spectrum that is not Hermitian at k=0 / Nyquist
    spec = np.fft.rfftn(f) * g.dV + 0.3j
    from dftpy_amd import ReciprocalField
    got = ReciprocalField(g.get_reciprocal(), data=torch.as_tensor(spec)).ifft().data.cpu().numpy()
    ref = np.fft.irfftn(spec, s=shape, axes=(0, 1, 2)) / g.dV
    assert np.max(np.abs(got - ref)) <= _tol(dtype) * np.max(np.abs(ref)) * 8


@pytest.mark.parametrize("shape", [(8, 8, 8), (6, 10, 15), (16, 26, 18), (7, 11, 13), (32, 32, 32), (64, 48, 40)])
@pytest.mark.parametrize("dtype", [torch.float64, torch.float32])
def test_c2c(shape, dtype):
    from dftpy_amd import DirectField
    g = _grid(shape, dtype, full=True)
    rng = np.random.default_rng(3)
    f = rng.standard_normal(shape) + 1j * rng.standard_normal(shape)
    fld = DirectField(g, data=torch.as_tensor(f), cplx=True)
    F = fld.fft()
    ref = np.fft.fftn(f) * g.dV
    got = F.data.cpu().numpy()
    assert np.max(np.abs(got - ref)) <= _tol(dtype) * np.max(np.abs(ref)) * 4
    back = F.ifft().data.cpu().numpy()
    assert np.max(np.abs(back - f)) <= _tol(dtype) * np.max(np.abs(f)) * 8


def test_gaussian_pair():
    # examples/test/test_field.py:247-285 (a 2/3/5-smooth grid instead of 51^3)
    from dftpy_amd import DirectField, DirectGrid
    nr = (50, 50, 50)
    g = DirectGrid(np.eye(3) * 10.0, nr, full=False)
    r = g.r.cpu().numpy()
    c = r[:, 25, 25, 25]
    s = 0.5
    a = r - c[:, None, None, None]
    df = (s * np.sqrt(2 * np.pi)) ** -3 * np.exp(-0.5 * np.einsum("lijk,lijk->ijk", a, a) / s ** 2)
    F = DirectField(g, data=df).fft()
    gv = g.get_reciprocal().g.cpu().numpy()
    gg = (gv ** 2).sum(0)
    ref = np.exp(-s ** 2 * gg / 2.0) * np.exp(-1j * np.einsum("lijk,l->ijk", gv, c))
    assert np.allclose(F.data.cpu().numpy(), ref, atol=1e-8)
    assert np.isclose(DirectField(g, data=df).integral(), 1.0)


def test_160_cube_fp32_fp64():
    from dftpy_amd import DirectField
    for dt, tol in ((torch.float64, 1e-12), (torch.float32, 3e-6)):
        g = _grid((160, 160, 160), dt)
        rng = np.random.default_rng(11)
        f = rng.random((160, 160, 160))
        F = DirectField(g, data=f).fft()
        ref = np.fft.rfftn(f) * g.dV
        assert np.max(np.abs(F.data.cpu().numpy() - ref)) <= tol * np.max(np.abs(ref))


@pytest.mark.parametrize("shape", [(160, 160, 160), (96, 72, 100), (48, 80, 64), (128, 120, 144), (32, 256, 240)])
@pytest.mark.parametrize("dtype", [torch.float64, torch.float32])
def test_fixed_and_generic_kernels_agree(shape, dtype):
    """The size-specialised passes against pocketfft and against the generic
    mixed-radix kernels on the same input."""
    from dftpy_amd import DirectField, _lib
    g = _grid(shape, dtype)
    rng = np.random.default_rng(5)
    f = rng.standard_normal(shape)
    fld = DirectField(g, data=f)
    plan = g.plan(dtype)
    _lib.check(_lib.lib.ofdft_plan_set_fft_kernels(plan.handle, 1))
    F1 = fld.fft().data.clone()
    b1 = DirectField(g, data=f).fft().ifft().data.clone()
    _lib.check(_lib.lib.ofdft_plan_set_fft_kernels(plan.handle, 0))
    F0 = fld.fft().data.clone()
    _lib.check(_lib.lib.ofdft_plan_set_fft_kernels(plan.handle, 1))
    ref = np.fft.rfftn(f) * g.dV
    tol = _tol(dtype) * np.max(np.abs(ref)) * 4
    assert np.max(np.abs(F1.cpu().numpy() - ref)) <= tol
    assert np.max(np.abs(F0.cpu().numpy() - ref)) <= tol
    assert np.max(np.abs(b1.cpu().numpy() - f)) <= _tol(dtype) * 8 * np.max(np.abs(f))


@pytest.mark.parametrize("shape", [(160, 160, 160), (96, 72, 100), (64, 48, 32)])
@pytest.mark.parametrize("dtype", [torch.float64, torch.float32])
def test_tile_variants_agree(shape, dtype):
    """Both tiles of each size-specialised pass (the autotuner's search space),
    one pass at a time, against tile 0 of all: the same transforms bit for bit,
    and the same WT evaluation to the order in which its mean density is
    summed.  The variants past 1 are the same two tiles by other numbers; they
    are accepted, and the autotuner's choice is one of the two."""
    from dftpy_amd import DirectField, _lib
    from dftpy_amd.functional import Functional
    g = _grid(shape, dtype)
    rng = np.random.default_rng(9)
    f = 0.02 + 0.01 * rng.random(shape)
    plan = g.plan(dtype)
    print("autotuned", plan.variants, plan.variant_ms.tolist())

    def run(v):
        plan.set_variants(v)
        F = DirectField(g, data=f).fft().data.cpu().numpy()
        o = Functional(type="KEDF", name="WT")(DirectField(g, data=f))
        return F, o.energy, o.potential.numpy()

    tuned = list(plan.variants)
    assert all(v in (0, 1) for v in tuned)
    F0, e0, p0 = run([0, 0, 0, 0])
    for v in ([1, 0, 0, 0], [0, 1, 0, 0], [0, 0, 1, 0], [0, 0, 0, 1], [1, 1, 1, 1], tuned, [2, 2, 5, 4]):
        F, e, p = run(v)
        assert np.array_equal(F, F0)
        assert abs(e - e0) <= 1e-12 * abs(e0)
        assert np.max(np.abs(p - p0)) <= 1e-12 * np.max(np.abs(p0))
    with pytest.raises(_lib.OFDFTError):
        plan.set_variants([3, 0, 0, 0])
    plan.set_variants([0, 0, 0, 0])


# every length with size-specialised passes (16 to 256, even, primes up to 13; not 242),
# beside odd and generic lengths on the other axes
def _smooth(n):
    for p in (2, 3, 5, 7, 11, 13):
        while n % p == 0:
            n //= p
    return n == 1


LENGTHS = [n for n in range(16, 257, 2) if _smooth(n)]


@pytest.mark.parametrize("n", LENGTHS)
def test_each_length_on_each_axis(n):
    from dftpy_amd import DirectField
    for dtype in (torch.float64, torch.float32):
        for shape in ((n, 5, 18), (7, n, 20), (3, 5, n)):
            rng = np.random.default_rng(n)
            f = rng.standard_normal(shape)
            g = _grid(shape, dtype)
            F = DirectField(g, data=f).fft()
            ref = np.fft.rfftn(f) * g.dV
            assert np.max(np.abs(F.data.cpu().numpy() - ref)) <= _tol(dtype) * np.max(np.abs(ref)) * 4
            assert np.max(np.abs(F.ifft().data.cpu().numpy() - f)) <= _tol(dtype) * np.max(np.abs(f)) * 8
            gc = _grid(shape, dtype, full=True)
            z = f + 1j * rng.standard_normal(shape)
            fld = DirectField(gc, data=torch.as_tensor(z), cplx=True)
            C = fld.fft()
            ref = np.fft.fftn(z) * gc.dV
            assert np.max(np.abs(C.data.cpu().numpy() - ref)) <= _tol(dtype) * np.max(np.abs(ref)) * 4
            assert np.max(np.abs(C.ifft().data.cpu().numpy() - z)) <= _tol(dtype) * np.max(np.abs(z)) * 8


@pytest.mark.parametrize("shape", [(16, 18, 20), (22, 26, 28), (52, 78, 104), (36, 15, 98), (27, 32, 40), (162, 20, 30)])
@pytest.mark.parametrize("full", [False, True])
@pytest.mark.parametrize("dtype", [torch.float64, torch.float32])
def test_evaluation_on_fixed_and_generic_passes(shape, full, dtype):
    """TF + vW + WT + LDA + Hartree with the size-specialised passes (the x
    pass with the multiply) and with the generic kernels.  FP64 to the
    transforms' rounding, which vW's G^2 multiplies: G_max^2 / 2 times a few
    ulps of sqrt(rho) over sqrt(rho), 1e-12 of the potential here; FP32
    likewise, 4e-4."""
    from dftpy_amd import DirectField, _lib
    from dftpy_amd.functional import Functional, TotalFunctional
    g = _grid(shape, dtype, full)
    rng = np.random.default_rng(2)
    rho = DirectField(g, data=0.02 + 0.01 * rng.random(shape))
    ev = TotalFunctional(KE=Functional(type="KEDF", name="WT"), XC=Functional(type="XC", name="LDA"),
                         H=Functional(type="HARTREE"))
    out = []
    for fixed in (1, 0):
        _lib.check(_lib.lib.ofdft_plan_set_fft_kernels(g.plan().handle, fixed))
        o = ev(rho)
        out.append((o.energy, o.potential.numpy().astype(np.float64), ev(rho, calcType={"E"}).energy))
    (e1, v1, x1), (e0, v0, x0) = out
    tol = 1e-12 if dtype == torch.float64 else 4e-4
    assert np.max(np.abs(v1 - v0)) <= tol * np.max(np.abs(v0))
    etol = 1e-12 if dtype == torch.float64 else 1e-5
    assert abs(e1 - e0) <= etol * abs(e0) and abs(x1 - x0) <= etol * abs(x0) and abs(x1 - e1) <= etol * abs(e1)


@pytest.mark.parametrize("shape", [(16, 18, 20), (26, 50, 52), (22, 15, 30), (27, 32, 40), (1, 24, 36)])
@pytest.mark.parametrize("dtype", [torch.float64, torch.float32])
@pytest.mark.parametrize("maxiter", [100, 3])
def test_cn_batch_on_fixed_and_generic_passes(shape, dtype, maxiter):
    """Lock-step Crank-Nicolson solves with the fused passes and with the
    generic kernels: three runs that need different numbers of iterations (one
    of them a constant), and a stop at maxiter.  Converged runs: both residuals
    are within atol and |A^-1| <= 1 (H is Hermitian), so the solutions differ
    by 2 atol in the 2-norm at most, besides the rounding of the recursion;
    after three steps, which amplify nothing much, by rounding alone."""
    from dftpy_amd import _lib
    from dftpy_amd.td import CrankNicholsonBatch
    g = _grid(shape, dtype, full=True)
    ct = torch.complex128 if dtype == torch.float64 else torch.complex64
    rng = np.random.default_rng(4)
    psi = torch.as_tensor(np.stack([np.full(shape, 0.1 + 0.0j),
                                    rng.standard_normal(shape) + 1j * rng.standard_normal(shape),
                                    0.1 + 0.01 * rng.standard_normal(shape)])).to(ct).cuda()
    v = torch.as_tensor(np.stack([np.full(shape, 0.3), rng.random(shape), 0.1 * rng.random(shape)])).to(dtype).cuda()
    tol = 1e-9 if dtype == torch.float64 else 1e-5
    out = []
    for fixed in (1, 0):
        _lib.check(_lib.lib.ofdft_plan_set_fft_kernels(g.plan().handle, fixed))
        cn = CrankNicholsonBatch(0.005, tol=tol, maxiter=maxiter)
        y, status = cn(g, psi, v)
        out.append((y.clone(), status, [d["iterations"] for d in cn.last_info]))
    (y1, s1, k1), (y0, s0, k0) = out
    assert s1 == s0 and all(abs(a - b) <= 1 for a, b in zip(k1, k0))
    eps = torch.finfo(dtype).eps
    for r in range(3):
        diff = float((y1[r] - y0[r]).abs().square().sum().sqrt())
        size = float(y0[r].abs().square().sum().sqrt())
        assert diff <= (2 * cn.last_info[r]["atol"] if s0[r] == 0 else 0.0) + 100 * eps * size


@pytest.mark.parametrize("nx,full", [(28, False), (52, False), (104, False), (36, True), (32, True), (160, True)])
def test_f32_multiply_keeps_f64_factors(nx, full):
    """FP32 grids whose G-space factors are FP64 ones (full grids, and half
    grids of the later x lengths), on a density whose transforms are exact: 1
    + cos(G.r) of period 4 along y and z and constant along x.  The Hartree
    potential is then 4 pi / G^2 cos(G.r) with the one rounding of the
    multiply, 2^-24, and what the x transforms of a constant leave, which the
    mean over x takes to a quarter of it."""
    from dftpy_amd import DirectField, DirectGrid
    from dftpy_amd.functional import Functional, TotalFunctional
    rng = np.random.default_rng(1)
    ev = TotalFunctional(H=Functional(type="HARTREE"))
    yz = (np.arange(4)[:, None] + np.arange(4)[None, :]) % 4
    cos = np.array([1.0, 0.0, -1.0, 0.0])[yz]
    for _ in range(24):
        lat = np.diag([7.1, 8.0, 9.3]) + 0.4 * rng.standard_normal((3, 3))
        g = DirectGrid(lat, (nx, 4, 4), full=full, dtype=torch.float32)
        v = ev(DirectField(g, data=np.broadcast_to(1.0 + cos, (nx, 4, 4)).copy())).potential.data
        v = v.double().mean(0).cpu().numpy()
        B = 2.0 * np.pi * np.linalg.inv(lat).T
        exact = 4.0 * np.pi / np.sum((B[1] + B[2]) ** 2)
        assert np.abs(v - exact * cos).max() <= 1.25 * 2.0 ** -24 * exact


@pytest.mark.parametrize("nx", [26, 50, 52])
def test_f32_kinetic_keeps_f64_factors(nx):
    """The kinetic operator of FP32 Crank-Nicolson steps on a plane wave of
    period 4 along z, exact but for the rounding of the multiply as above:
    after no iteration the workspace holds b = psi - i dt/2 G^2/2 psi."""
    from dftpy_amd import DirectGrid
    from dftpy_amd.td import CrankNicholsonBatch
    rng = np.random.default_rng(1)
    psi = torch.tensor([1, 1j, -1, -1j], dtype=torch.complex64).repeat(nx, 1, 4)[None].cuda().contiguous()
    v = torch.zeros((1, nx, 1, 16), device="cuda")
    for _ in range(24):
        lat = np.diag([71.0, 8.0, 9.3]) + 0.4 * rng.standard_normal((3, 3))  # small G_x: it amplifies what x leaves
        g = DirectGrid(lat, (nx, 1, 16), full=True, dtype=torch.float32)
        cn = CrankNicholsonBatch(4.0, maxiter=0, sigma=0.0)
        cn(g, psi, v)
        n = 16 * nx
        b = next(iter(cn._work.values())).view(torch.complex64)[n:2 * n].view(nx, 16)[:, ::4]
        exact = np.sum((4 * 2.0 * np.pi * np.linalg.inv(lat).T[2]) ** 2)
        err = np.abs(-b.imag.double().mean(0).cpu().numpy() - exact).max()
        assert err <= 1.25 * 2.0 ** -24 * exact


@pytest.mark.parametrize("shape", [(9, 15, 27), (27, 32, 40), (16, 18, 20)])
@pytest.mark.parametrize("dtype", [torch.float64, torch.float32])
def test_cn_batch_leaves_out_products_of_converged_runs(shape, dtype):
    """A solve that starts converged applies the Hamiltonian twice (right side,
    first residual): the workspace has the fields of one stopped there, and the
    product of the first iteration was not written."""
    from dftpy_amd.td import CrankNicholsonBatch
    g = _grid(shape, dtype, full=True)
    ct = torch.complex128 if dtype == torch.float64 else torch.complex64
    rng = np.random.default_rng(5)
    psi = torch.as_tensor(rng.standard_normal((2,) + shape) + 1j * rng.standard_normal((2,) + shape)).to(ct).cuda()
    v = torch.as_tensor(rng.random((2,) + shape)).to(dtype).cuda()
    n, out = int(np.prod(shape)), []
    for tol, maxiter in ((1e-6, 0), (1e3, 50)):
        cn = CrankNicholsonBatch(0.005, tol=tol, maxiter=maxiter)
        cn(g, psi, v)
        work = next(iter(cn._work.values())).view(ct)
        work.fill_(7.0)
        cn(g, psi, v)
        assert [d["iterations"] for d in cn.last_info] == [0, 0]
        assert bool((work[8 * n:] == 7.0).all())
        out.append(work.clone())
    assert torch.equal(out[0], out[1])


@pytest.mark.parametrize("n", [210, 224, 234, 240, 250, 252, 256])
def test_f32_full_grids_of_the_longest_axes(n):
    """The x pass with FP64 factors needs the most LDS here (130 KB at 256 with
    the second tile): both tiles against the generic kernels, to FP32 rounding
    that vW's G^2 multiplies."""
    from dftpy_amd import DirectField, _lib
    from dftpy_amd.functional import Functional, TotalFunctional
    shape = (n, 4, 18)
    g = _grid(shape, torch.float32, full=True)
    rho = DirectField(g, data=0.02 + 0.01 * np.random.default_rng(2).random(shape))
    ev = TotalFunctional(KE=Functional(type="KEDF", name="WT"), H=Functional(type="HARTREE"))
    out = []
    for fixed, tile in ((1, 0), (1, 1), (0, 0)):
        _lib.check(_lib.lib.ofdft_plan_set_fft_kernels(g.plan().handle, fixed))
        g.plan().set_variants([tile] * 4)
        out.append(ev(rho).potential.numpy().astype(np.float64))
    for v in out[:2]:
        assert np.max(np.abs(v - out[2])) <= 4e-4 * np.max(np.abs(out[2]))
