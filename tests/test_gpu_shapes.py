"""Default launch shapes, batch item lists and row-range sums at the sizes
where they change: results against one step per launch, single-field runs and
FP64 sums."""
import numpy as np
import pytest

from symphas_amd import abi, inputs, models
from symphas_amd.solver import FDBatch, FDPlan, MultiPlan, RegionalPlan, interior_shape

pytestmark = pytest.mark.gpu


def field(shape, seed, dtype):
    return inputs.uniform(shape[::-1], seed=seed).astype(
        np.float32 if dtype == abi.F32 else np.float64)


def run(d, psi, steps, shape=None):
    with FDPlan(d) as p:
        if shape:
            p.tune(*shape)
        p.upload(psi)
        p.step(steps)
        return p.download()


@pytest.mark.parametrize("dtype", [abi.F32, abi.F64])
@pytest.mark.parametrize("n", [(4, 3), (64, 64), (66, 5), (2, 700), (1030, 9), (1700, 1300)])
def test_default_shape_2d(gpu_lib, n, dtype):
    if n[0] < 3:
        n = (4, n[1])
    for model in (models.model_b, models.allen_cahn):
        d = model(n, dtype=dtype)
        psi = field(n, 51, dtype)
        vec = 2 if dtype == abi.F32 else 1
        assert np.array_equal(run(d, psi, 7), run(d, psi, 7, (1, 16, 0, vec)))


@pytest.mark.parametrize("dtype", [abi.F32, abi.F64])
@pytest.mark.parametrize("n", [(3, 4, 5), (65, 13, 3), (60, 61, 62), (200, 70, 90),
                               (236, 232, 240), (300, 280, 250)])
def test_default_shape_3d(gpu_lib, n, dtype):
    for model, kw in ((models.model_b, {"dt": 0.005}), (models.allen_cahn, {})):
        d = model(n, dtype=dtype, stencil=models.Stencil3d2h(7, 10, 25), **kw)
        psi = field(n, 52, dtype)
        assert np.array_equal(run(d, psi, 5), run(d, psi, 5, (1, 4, 8, 0)))


@pytest.mark.parametrize("n,L", [((4, 3), 5), ((130, 700), 5), ((6, 5, 4), 7), ((64, 33, 50), 7)])
@pytest.mark.parametrize("model", [models.gray_scott, models.model_c, models.turing, models.mixed])
def test_default_shape_coupled(gpu_lib, orc, model, n, L):
    # the models with known polynomial classes and one without, FP64 against
    # the oracle: rounding of a few steps
    st = models.Stencil2d2h(5, 6, 13) if L == 5 else models.Stencil3d2h(7, 10, 25)
    d = model(n, dt=0.002, stencil=st)
    f = [inputs.uniform(n[::-1], seed=s, lo=0.1, hi=0.9) for s in (53, 54)]
    want = orc.mrun(d, f, 5, 8)
    with MultiPlan(d) as p:
        assert p.query()[0] == abi.PATH_FUSED
        for i in range(2):
            p.upload(i, f[i])
        p.step(5)
        for i in range(2):
            err = np.linalg.norm(p.download(i) - want[i]) / np.linalg.norm(want[i])
            assert err <= 1e-13, (i, err)


@pytest.mark.parametrize("sizes", [[(4, 3)], [(512, 512)], [(130, 6), (64, 640)],
                                   [(128, 128)] * 9 + [(384, 200), (2, 90)] + [(96, 61)] * 20])
def test_batch_items_and_sums(gpu_lib, sizes):
    sizes = [(max(4, x), y) for x, y in sizes]
    descs = [(models.model_b if i % 2 else models.allen_cahn)(
        n, h=1.0, dt=0.01, dtype=abi.F32, path=abi.PATH_FUSED) for i, n in enumerate(sizes)]
    psi = [field(n, 60 + i, abi.F32) for i, n in enumerate(sizes)]
    with FDBatch(descs) as b:
        for i, f in enumerate(psi):
            b.upload(i, f)
        b.step(9)
        mass, energy = b.reduce()
        got = [b.download(i) for i in range(len(sizes))]
    for i, (d, f) in enumerate(zip(descs, psi)):
        assert np.array_equal(got[i], run(d, f, 9)), sizes[i]
        g = got[i].astype(np.float64)
        e = (-0.5 * g ** 2 + 0.25 * g ** 4 + 0.5 * (np.roll(g, -1, 0) - g) ** 2
             + 0.5 * (np.roll(g, -1, 1) - g) ** 2)
        # FP64 sums of N terms in another order: N eps of the terms' magnitude
        tol = g.size * 2.0 ** -52
        assert abs(mass[i] - g.sum()) <= tol * np.abs(g).sum()
        assert abs(energy[i] - e.sum()) <= tol * np.abs(e).sum()


@pytest.mark.parametrize("dtype", [abi.F32, abi.F64])
@pytest.mark.parametrize("gradient", [abi.GRAD_FORWARD, abi.GRAD_CENTRAL])
@pytest.mark.parametrize("n", [(4, 3), (5, 7), (2056, 1500), (1030, 3), (6, 5, 4), (68, 40, 33),
                               (3, 700, 5)])
def test_row_sums(gpu_lib, n, gradient, dtype):
    st = models.Stencil2d2h() if len(n) == 2 else models.Stencil3d2h()
    d = models.model_b(n, h=0.7, dtype=dtype, stencil=st)
    psi = field(n, 55, dtype)
    with FDPlan(d) as p:
        p.set_energy(models.landau_energy(d, gradient=gradient, c1=0.7, c2=1.9, kappa=2.5))
        p.upload(psi)
        mass, energy = p.reduce()
    g = psi.astype(np.float64)
    e = -0.35 * g ** 2 + 0.475 * g ** 4
    for a in range(g.ndim):
        diff = (np.roll(g, -1, a) - g) / 0.7 if gradient == abi.GRAD_FORWARD else \
            (np.roll(g, -1, a) - np.roll(g, 1, a)) / 1.4
        e = e + 1.25 * diff ** 2
    e = e * 0.7 ** g.ndim
    # N eps of the terms' magnitude, the density itself a few eps
    tol = (g.size + 16) * 2.0 ** -52
    assert abs(mass - g.sum()) <= tol * np.abs(g).sum()
    assert abs(energy - e.sum()) <= tol * np.abs(e).sum() * 4


@pytest.mark.parametrize("dtype", [abi.F32, abi.F64])
@pytest.mark.parametrize("blob", [(820, 790), (1210, 1300), (1700, 61)])
def test_regional_box_chunks(gpu_lib, blob, dtype):
    """Boxes whose chunk height is above the least one (7, 14 and more rows; a
    short last chunk): four steps per launch against one, bit for bit."""
    d = models.model_b((2048, 1600), dt=0.01, dtype=dtype, path=abi.PATH_FUSED)
    psi = np.zeros(interior_shape(d), np.float32 if dtype == abi.F32 else np.float64)
    psi[60:60 + blob[1], 50:50 + blob[0]] = 0.4 + field(blob, 31, dtype) * 0.05
    got = {}
    for spl in (1, 4):
        with RegionalPlan(d, abi.Regional(1e-6, 1.1, 1.0, 1, spl, 0.05)) as rp:
            rp.upload(psi)
            rp.step(23)
            info = rp.region()
            assert blob[0] <= info.dims[0] < d.n[0] and blob[1] <= info.dims[1] < d.n[1]
            got[spl] = rp.download()
    assert np.array_equal(got[1], got[4])


@pytest.mark.parametrize("dtype", [abi.F32, abi.F64])
@pytest.mark.parametrize("n", [(64, 48), (260, 31), (36, 10, 9)])
def test_sums_wherever_the_field_lies(gpu_lib, n, dtype):
    # a caller's field may start at any value of an allocation: the sums are
    # those of the plan bit for bit, in the order that the sizes alone set
    import ctypes

    import torch
    st = {"stencil": models.Stencil3d2h(7, 10, 25), "dt": 0.005} if len(n) == 3 else {}
    d = models.model_b(n, dtype=dtype, **st)
    psi = field(n, 57, dtype)
    energy = abi.Energy(0.7, 1.3, 1.9, abi.GRAD_CENTRAL, 0)
    with FDPlan(d) as p:
        p.upload(psi)
        p.set_energy(energy)
        want = p.reduce()
    sums = torch.empty(2, device="cuda", dtype=torch.float64)
    for shift in (0, 1, 3):
        buf = torch.zeros(psi.size + 8, device="cuda",
                          dtype=torch.float32 if dtype == abi.F32 else torch.float64)
        buf[shift:shift + psi.size] = torch.from_numpy(psi.ravel()).to("cuda")
        nn = (ctypes.c_int32 * 3)(*(list(n) + [1] * (3 - len(n))))
        torch.cuda.synchronize()
        abi.check(gpu_lib.sps_fd_reduce_device(
            d.dim, dtype, nn, d.h, ctypes.byref(energy),
            ctypes.c_void_p(buf[shift:].data_ptr()), ctypes.c_void_p(sums.data_ptr()), None))
        torch.cuda.synchronize()
        assert tuple(sums.cpu().tolist()) == want, shift
