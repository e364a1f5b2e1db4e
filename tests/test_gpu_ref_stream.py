"""The stream form of the reference-order step against the one-site kernel and
the CPU oracle, bit for bit.

`FDPlan.equation` evaluates the right-hand side with the one-site kernel, so
psi + dt * equation(psi), rounded like the kernel's Euler update, is what one
step of the stream has to give in either type.
"""
import itertools

import numpy as np
import pytest

from symphas_amd import abi, inputs, models
from symphas_amd.models import Stencil2d2h, Stencil3d2h, TermSpec
from symphas_amd.solver import FDPlan, MultiPlan

pytestmark = pytest.mark.gpu

LAP = TermSpec(abi.OP_LAP, 0.9, models.PSI)
LAP3 = TermSpec(abi.OP_LAP, 1.1, models.PSI3)
LAPP = TermSpec(abi.OP_LAP, -0.7, (0.3, 0.5, -0.25, 0.125, 0.0, 0.0625, -0.4))
BI = TermSpec(abi.OP_BILAP, -0.8, models.PSI)
ID = TermSpec(abi.OP_ID, 1.0, (0.0, 1.0, 0.0, -1.0))
IDP = TermSpec(abi.OP_ID, 0.6, (0.2, 0.0, -0.3, 0.0, 0.7))
ID1 = TermSpec(abi.OP_ID, -1.3, models.PSI)
ID0 = TermSpec(abi.OP_ID, 1.3, (0.0,))
SETS = [[LAP], [LAP3], [LAPP], [BI], [IDP], [ID0]]
SETS += [list(s) for s in itertools.permutations([LAP, ID], 2)]
SETS += [[BI, LAPP], [LAP3, IDP], [LAP, LAP3], [BI, ID1], [LAPP, BI]]
SETS += [list(s) for s in itertools.permutations([BI, LAP, LAP3], 3)]
SETS += [[LAP, LAPP, IDP], [ID, BI, LAP], [ID1, LAP3, BI], [LAP3, ID, BI]]
# lists that are no set of kinds keep the one-site kernel
SETS += [[BI, LAP, LAP3, ID], [LAP, LAP], [LAP, TermSpec(abi.OP_BILAP, 0.1, models.PSI3)]]


def field(desc, seed):
    shape = tuple(desc.n[a] for a in reversed(range(desc.dim)))
    psi = inputs.uniform(shape, seed=seed, lo=-1.0, hi=1.0)
    return psi.astype(np.float32 if desc.dtype == abi.F32 else np.float64)


@pytest.mark.parametrize("dtype", [abi.F32, abi.F64])
@pytest.mark.parametrize("shape", [(3, 3), (7, 4), (60, 5), (61, 9), (59, 33), (121, 70)])
def test_step_equals_one_site_kernel(gpu_lib, shape, dtype):
    print("[case] ref stream", shape, dtype, flush=True)
    t = np.float32 if dtype == abi.F32 else np.float64
    for terms in SETS:
        for L, G, B in ((5, 6, 13), (9, 6, 13), (5, 6, 17), (9, 6, 17), (5, 6, 21), (9, 6, 21)):
            d = models.make_desc(shape, Stencil2d2h(L, G, B), 0.8, 0.003, terms, dtype,
                                 abi.PATH_REFERENCE)
            psi = field(d, 31)
            with FDPlan(d) as p:
                p.upload(psi)
                rhs = p.equation()
                p.step(1)
                got = p.download()
            assert np.array_equal(got, psi + t(0.003) * rhs), (terms, L, B)


@pytest.mark.parametrize("dtype", [abi.F32, abi.F64])
# up to 512 workgroups (FP32; FP64 256) the one-site kernel takes the step
@pytest.mark.parametrize("shape", [(3, 4, 5), (3, 4, 3500), (60, 5, 150), (61, 220, 3), (125, 33, 26),
                                   (60, 5, 257), (61, 685, 3), (125, 33, 29)])
def test_3d_step_equals_one_site_kernel(gpu_lib, shape, dtype):
    print("[case] ref stream 3D", shape, dtype, flush=True)
    t = np.float32 if dtype == abi.F32 else np.float64
    for terms in SETS:
        # 19 and 41 points keep the one-site kernel
        for L, G, B in ((7, 10, 25), (15, 10, 25), (19, 10, 25), (15, 10, 41)):
            d = models.make_desc(shape, Stencil3d2h(L, G, B), 0.8, 0.003, terms, dtype,
                                 abi.PATH_REFERENCE)
            psi = field(d, 33)
            with FDPlan(d) as p:
                p.upload(psi)
                rhs = p.equation()
                p.step(1)
                got = p.download()
            assert np.array_equal(got, psi + t(0.003) * rhs), (terms, L, B)


def test_tall_chunks_equal_oracle(gpu_lib, orc):
    # 6144 chunks' worth of rows is passed: chunks above the lowest height,
    # the last one shorter
    d = models.model_b((1201, 2011), dt=0.01, stencil=Stencil2d2h(), dtype=abi.F64,
                       path=abi.PATH_REFERENCE)
    psi = field(d, 32) * 0.1
    with FDPlan(d) as p:
        p.upload(psi)
        p.step(3)
        got = p.download()
    assert np.array_equal(got, orc.unpad(d, orc.run(d, psi, 3, 8)))


@pytest.mark.parametrize("model", [models.model_c, models.gray_scott, models.turing])
@pytest.mark.parametrize("shape", [(3, 5), (61, 9), (130, 77), (3, 4, 5), (61, 10, 23)])
def test_coupled_forms_equal_oracle(gpu_lib, orc, model, shape):
    stencils = [Stencil2d2h(L, G, B) for L, G, B in
                ((5, 6, 13), (9, 6, 17), (9, 6, 13), (5, 6, 21))]
    if len(shape) == 3:
        stencils = [Stencil3d2h(L, 10, B) for L, B in ((7, 25), (15, 25), (15, 21))]
    for st in stencils:
        d = model(shape, dt=0.01, stencil=st, dtype=abi.F64, path=abi.PATH_REFERENCE)
        f = [inputs.uniform(shape[::-1], seed=s, lo=-1.0, hi=1.0) for s in (41, 42)]
        want = orc.mrun(d, f, 4, 8)
        with MultiPlan(d) as p:
            for i in range(2):
                p.upload(i, f[i])
            p.step(4)
            for i in range(2):
                assert np.array_equal(p.download(i), want[i]), (st, i)
        # FP32: four steps round each site a few tens of times
        d32 = model(shape, dt=0.01, stencil=st, dtype=abi.F32, path=abi.PATH_REFERENCE)
        with MultiPlan(d32) as p:
            for i in range(2):
                p.upload(i, f[i].astype(np.float32))
            p.step(4)
            for i in range(2):
                err = np.abs(p.download(i) - want[i]).max() / np.abs(want[i]).max()
                assert err <= 100 * 2.0 ** -24, (st, i, err)
