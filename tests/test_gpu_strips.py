"""The x sweep by strips of rows held in LDS (csrc/resident.hip), for planes that do not fit there,
against the separate sweep kernel, which an explicit launch shape selects, and the oracle: the
same bits (FP32 storage keeps the separate sweep, beside them in a batch too).  Shapes: two workgroups per CU and one, one and two
wavefronts of rows, ragged last strips, strips over several planes, the longest rows that fit."""
import numpy as np
import pytest

import casefile as cf
import oracle as orc
from test_gpu_planes import _case, _fields, _solver

pytestmark = pytest.mark.gpu

FP64 = [(150, 140, 3, 2), (161, 130, 5, 1), (200, 111, 3, 1), (300, 70, 4, 2), (311, 66, 3, 1), (400, 60, 3, 2),
        (401, 53, 5, 1), (640, 37, 3, 1), (2, 1500, 3, 1), (31, 700, 4, 1), (66, 400, 3, 1)]
FP32 = [(230, 200, 3, 2), (300, 250, 140, 1), (301, 150, 3, 1), (400, 113, 5, 2), (640, 70, 3, 1), (2, 1500, 3, 1), (800, 57, 3, 1)]


@pytest.mark.parametrize("shape", FP64)
def test_fp64_strips_match_separate_sweep_and_oracle(shape):
    c = _case(shape, seed=31, nagents=300)
    print(f"[gpu] strips fp64 {shape}", flush=True)
    strips, separate = _fields(c, "fp64")
    assert np.array_equal(strips, separate)
    assert np.array_equal(strips, orc.run(c))


@pytest.mark.parametrize("shape", FP32)
def test_fp32_strips_match_separate_sweep(shape):
    c = _case(shape, seed=32, nagents=300)
    print(f"[gpu] strips fp32 {shape}", flush=True)
    strips, separate = _fields(c, "fp32")
    assert np.array_equal(strips, separate)


@pytest.mark.parametrize("precision", ["fp64", "fp32"])
def test_dense_agents_on_strips(precision):
    """More occupied voxels in a strip than loading threads, many agents to a voxel."""
    c = _case((210, 205, 4, 2), seed=33, nagents=60000, agent_box=(np.zeros(3), np.array([4200.0, 500.0, 40.0])))
    strips, separate = _fields(c, precision)
    assert np.array_equal(strips, separate)


@pytest.mark.parametrize("precision", ["fp64", "fp32"])
@pytest.mark.parametrize("shape", [(170, 140, 5, 2), (401, 160, 3, 1), (260, 190, 3, 2)])
def test_dirichlet_nodes_on_strips(shape, precision):
    c = _case(shape, seed=34, dactive=[1, 0][:shape[3]])
    rng = np.random.default_rng(3)
    nv = shape[0] * shape[1] * shape[2]
    c.dnodes = (rng.permutation(nv)[:nv // 3].astype(np.int32), rng.uniform(0.0, 9.0, (nv // 3, shape[3])))
    strips, separate = _fields(c, precision)
    assert np.array_equal(strips, separate)


def test_signed_zero_and_tiny_rows():
    """Zero, tiny, huge and negative rows: their wavefront's rows take true divisions, with the
    agents applied again, the others do not."""
    c = _case((180, 150, 5, 2), seed=35, nagents=500)
    c.init[:, 3:9, 1] = 0.0
    c.init[:, 9:12, 1] = -0.0
    c.init[7, 80, 2] = 1e-310
    c.init[:, 20:25, 3] = 1e-290
    c.init[11, 70, 1] = -1e300
    c.init[:, 100:110, 2] *= -1.0
    strips, separate = _fields(c, "fp64")
    assert np.array_equal(strips.view(np.uint64), separate.view(np.uint64))


@pytest.mark.parametrize("precision", ["fp64", "fp32"])
def test_adjoint_on_strips(precision):
    c = _case((220, 201, 3, 2), seed=36, nsteps=3, dactive=[1, 0])
    seed = np.random.default_rng(2).normal(size=(220, 201, 3, 2))
    out = []
    for separate in (False, True):
        s = _solver(c, precision, separate)
        s.adjoint_forward(c.nsteps, 2)
        out.append(s.adjoint_backward(seed))
        s.close()
    for a, b in zip(*out):
        assert np.array_equal(a, b)


@pytest.mark.parametrize("precision", ["fp64", "fp32"])
def test_batch_of_planes_strips_and_others(precision):
    """Members of every path in one batch, eager and as a graph, against each member alone."""
    from biofvmb import Batch
    shapes = [(20, 21, 5, 2), (230, 210, 2, 1), (900, 50, 3, 1), (150, 141, 3, 2), (401, 130, 2, 1), (1700, 30, 2, 1)]
    cases = [_case(sh, seed=40 + i, nagents=0 if i == 3 else 50) for i, sh in enumerate(shapes)]
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
