"""x and y sweeps of z planes held in LDS (csrc/resident.hip) against the separate sweep kernels,
which an explicit launch shape selects, and against the oracle: the same bits in FP64 and in FP32
storage.  Shapes: the largest planes that fit (and the ones that just do not), the denser LDS
layout, lines around multiples of the batch and the wavefront, one-voxel axes."""
import numpy as np
import pytest

import casefile as cf
import oracle as orc

pytestmark = pytest.mark.gpu

SEPARATE = 1 << 30  # a grid for every tile: the separate sweeps' default shape


def _case(shape, seed, nagents=60, nsteps=2, **kw):
    return cf.make_case(*shape, seed=seed, nagents=nagents, nsteps=nsteps, shared_voxels=True, **kw)


def _solver(c, precision, separate=False):
    from biofvmb import LODSolver
    s = LODSolver(c.nx, c.ny, c.nz, c.nsub, c.dx, precision)
    s.set_coefficients(c.D, c.decay, c.dt)
    dv, da = cf.effective_dirichlet(c)
    s.set_dirichlet(dv, da)
    if c.dnodes is not None:
        s.set_dirichlet_nodes(*c.dnodes)
    s.upload(c.init)
    voxel, t1, t2 = orc.agent_tables(c)
    s.set_agents(voxel, t1, t2)
    if separate:
        s.set_launch(0, SEPARATE, 0, 0)
    return s


def _fields(c, precision):
    out = []
    for separate in (False, True):
        s = _solver(c, precision, separate)
        s.run(c.nsteps)
        out.append(s.download())
        s.close()
    return out


# (139, 139) and (140, 145) in FP64: the largest square, one that fits no more
FP64 = [(1, 1, 3, 1), (2, 1, 3, 2), (1, 7, 4, 2), (3, 5, 4, 2), (4, 4, 3, 1), (5, 9, 3, 2), (12, 13, 3, 2), (63, 64, 3, 1),
        (65, 66, 2, 1), (16, 130, 2, 1), (200, 20, 2, 1), (20, 200, 2, 1), (100, 101, 2, 1), (139, 139, 3, 1),
        (140, 145, 2, 1), (142, 136, 3, 1), (256, 70, 2, 1), (70, 256, 2, 1), (50, 50, 30, 3)]
FP32 = [(2, 1, 3, 1), (5, 6, 3, 2), (64, 64, 3, 1), (120, 119, 3, 1), (150, 160, 2, 1), (200, 200, 3, 1), (200, 199, 2, 1),
        (192, 205, 2, 1), (201, 201, 2, 1), (256, 150, 2, 1)]


@pytest.mark.parametrize("shape", FP64)
def test_fp64_planes_match_separate_sweeps_and_oracle(shape):
    c = _case(shape, seed=7)
    print(f"[gpu] planes fp64 {shape}", flush=True)
    planes, separate = _fields(c, "fp64")
    assert np.array_equal(planes, separate)
    assert np.array_equal(planes, orc.run(c))


@pytest.mark.parametrize("shape", FP32)
def test_fp32_planes_match_separate_sweeps(shape):
    c = _case(shape, seed=8)
    print(f"[gpu] planes fp32 {shape}", flush=True)
    planes, separate = _fields(c, "fp32")
    assert np.array_equal(planes, separate)


@pytest.mark.parametrize("precision", ["fp64", "fp32"])
@pytest.mark.parametrize("shape", [(17, 12, 5, 3), (139, 100, 3, 2), (40, 1, 6, 2)])
def test_dirichlet_nodes_on_planes(shape, precision):
    c = _case(shape, seed=9, dactive=[1, 0, 1][:shape[3]])
    rng = np.random.default_rng(3)
    nv = shape[0] * shape[1] * shape[2]
    c.dnodes = (rng.permutation(nv)[:nv // 3].astype(np.int32), rng.uniform(0.0, 9.0, (nv // 3, shape[3])))
    planes, separate = _fields(c, precision)
    assert np.array_equal(planes, separate)


def test_signed_zero_and_tiny_fields():
    """Zeros, negative zeros, tiny and huge values in some planes: those take true divisions, the
    others do not, and every bit is the separate sweeps'."""
    c = _case((40, 33, 9, 2), seed=11, nagents=0)
    c.init[:, :, 1] = 0.0
    c.init[:, :, 2] = -0.0
    c.init[3, 4, 3] = 1e-310
    c.init[5:9, :, 4] = 1e-290
    c.init[7, 7, 5] = -1e300
    c.init[:, :, 6] *= -1.0
    planes, separate = _fields(c, "fp64")
    assert np.array_equal(planes.view(np.uint64), separate.view(np.uint64))


def test_zero_dirichlet_values():
    c = _case((36, 48, 7, 2), seed=12, dactive=[1, 1])
    c.dvalue[:] = 0.0
    planes, separate = _fields(c, "fp64")
    assert np.array_equal(planes, separate) and np.array_equal(planes, orc.run(c))


def test_substrate_without_reciprocal_pair():
    """Coefficients whose denominators include one that no reciprocal pair divides by exactly
    (about one in a thousand): that substrate's planes take the corrected product."""
    import ctypes
    import biofvmb._lib as L
    fn = ctypes.CDLL(L.LIB_PATH)["_ZN5bfvmb15reciprocal_pairEdPdS0_"]
    fn.restype, fn.argtypes = ctypes.c_bool, [ctypes.c_double] + [ctypes.POINTER(ctypes.c_double)] * 2
    hi, lo = ctypes.c_double(), ctypes.c_double()
    c = _case((21, 30, 6, 2), seed=13)
    rng = np.random.default_rng(5)
    found = 0
    for _ in range(20000):  # the first denominator of every axis is 1 + c1 + decay*dt/3
        D, decay = float(rng.uniform(1e3, 1e5)), float(rng.uniform(0.01, 1.0))
        a = D * c.dt / c.dx / c.dx
        if not fn((1.0 + a) + decay * c.dt / 3.0, ctypes.byref(hi), ctypes.byref(lo)):
            found, c.D[1], c.decay[1] = 1, D, decay
            break
    assert found
    planes, separate = _fields(c, "fp64")
    assert np.array_equal(planes, separate) and np.array_equal(planes, orc.run(c))


@pytest.mark.parametrize("precision", ["fp64", "fp32"])
@pytest.mark.parametrize("shape", [(24, 31, 9, 2), (130, 139, 4, 2), (200, 196, 3, 1)])
def test_adjoint_order_on_planes(shape, precision):
    """The reverse pass (y before x on the plane) gives the separate sweeps' gradients."""
    c = _case(shape, seed=14, nsteps=3, dactive=[1, 0][:shape[3]])
    seed = np.random.default_rng(2).normal(size=shape)
    out = []
    for separate in (False, True):
        s = _solver(c, precision, separate)
        s.adjoint_forward(c.nsteps, 2)
        out.append(s.adjoint_backward(seed))
        s.close()
    for a, b in zip(*out):
        assert np.array_equal(a, b)


@pytest.mark.parametrize("precision", ["fp64", "fp32"])
def test_batch_of_resident_and_other_members(precision):
    """Members of every size class beside members whose planes do not fit, eager and as a graph,
    against each member alone."""
    from biofvmb import Batch
    shapes = [(20, 21, 5, 2), (60, 60, 4, 1), (100, 90, 3, 2), (139, 130, 3, 1), (230, 210, 2, 1), (200, 200, 2, 1),
              (2, 3, 4, 1)]
    cases = [_case(sh, seed=20 + i, nagents=0 if i == 2 else 50) for i, sh in enumerate(shapes)]
    for graph in (False, True):
        b = Batch(shapes, cases[0].dx, precision)
        for i, c in enumerate(cases):
            b.set_coefficients(i, c.D, c.decay, c.dt)
            b.set_dirichlet(i, *cf.effective_dirichlet(c))
            b.upload(i, c.init)
            b.set_agents(i, *orc.agent_tables(c))
        for _ in range(2):
            b.run(3, graph=graph)
        got = [b.download(i) for i in range(len(shapes))]
        b.close()
        for c, g in zip(cases, got):
            s = _solver(c, precision, separate=True)
            s.run(6)
            assert np.array_equal(g, s.download())
            s.close()


@pytest.mark.parametrize("precision,shapes", [
    ("fp64", [(240, 60, 5, 1), (133, 120, 6, 2), (60, 240, 3, 1)]),   # 256 solvers leave 256 loaders
    ("fp64", [(200, 30, 5, 1), (95, 95, 6, 2), (30, 200, 3, 1)]),     # more threads than a workgroup
    ("fp32", [(320, 70, 5, 1), (190, 190, 4, 2), (70, 320, 3, 1)])])
def test_batch_of_long_and_large_planes(precision, shapes):
    """Members of one size class, some with many lines, some with many values: the launch has the
    solvers of the former and then too few loaders to hold the latter's planes in registers."""
    from biofvmb import Batch
    cases = [_case(sh, seed=60 + i) for i, sh in enumerate(shapes)]
    b = Batch(shapes, cases[0].dx, precision)
    for i, c in enumerate(cases):
        b.set_coefficients(i, c.D, c.decay, c.dt)
        b.set_dirichlet(i, *cf.effective_dirichlet(c))
        b.upload(i, c.init)
        b.set_agents(i, *orc.agent_tables(c))
    b.run(3)
    got = [b.download(i) for i in range(len(shapes))]
    b.close()
    for c, g in zip(cases, got):
        s = _solver(c, precision, separate=True)
        s.run(3)
        assert np.array_equal(g, s.download())
        s.close()
