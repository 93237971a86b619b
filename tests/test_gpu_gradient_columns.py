"""Density gradients (csrc/gradient.hip) against numpy's differences and divisions, bit for bit, at
the edges of the kernel's split: one plane to many per thread, planes smaller and larger than a
block, one-voxel axes, and differences that the reciprocal pair does not cover."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _reference(f, dx):
    out = np.zeros(f.shape + (3,))
    with np.errstate(all="ignore"):
        for a in range(3):
            n = f.shape[a]
            if n == 1:
                continue
            v, g = np.moveaxis(f, a, 0), np.moveaxis(out[..., a], a, 0)
            g[0] = (v[1] - v[0]) / dx
            g[n - 1] = (v[n - 1] - v[n - 2]) / dx
            g[1:n - 1] = (v[2:] - v[:-2]) / (dx * 2.0)
    return out


def _check(f, dx, precision):
    from biofvmb import LODSolver
    s = LODSolver(*f.shape, dx, precision)
    s.set_coefficients(np.full(f.shape[3], 1e3), np.full(f.shape[3], 0.1), 0.01)
    s.upload(f)
    s.compute_gradients()
    got, held = s.download_gradients(), s.download()
    s.close()
    ref = _reference(held, dx)
    if precision == "fp32":
        with np.errstate(all="ignore"):
            ref = ref.astype(np.float32).astype(np.float64)
    got = got.reshape(ref.shape)
    assert np.array_equal(np.isnan(got), np.isnan(ref))
    ok = ~np.isnan(ref)
    assert np.array_equal(got[ok].view(np.uint64), ref[ok].view(np.uint64))


# at most 2^17 values: one plane per thread; above: 4 to 16, with ragged ends
SHAPES = [(1, 1, 1, 1), (1, 1, 5, 2), (5, 1, 1, 1), (1, 9, 1, 2), (2, 2, 2, 1), (31, 17, 9, 2), (64, 64, 32, 1),
          (64, 64, 33, 1), (300, 219, 2, 1), (3, 1, 60001, 1), (1, 300, 501, 1), (101, 103, 17, 3), (97, 113, 61, 4),
          (160, 161, 67, 5)]


@pytest.mark.parametrize("precision", ["fp64", "fp32"])
@pytest.mark.parametrize("shape", SHAPES)
def test_split_edges(shape, precision):
    print(f"[gpu] gradients {shape} {precision}", flush=True)
    _check(np.random.default_rng(1).lognormal(size=shape), 20.0, precision)


@pytest.mark.parametrize("dx", [1.0, 0.3, 1e-13, 1e14])
def test_divisors(dx):
    """A power of two, an ordinary one, and two that no pair is made for."""
    _check(np.random.default_rng(2).lognormal(size=(60, 61, 40, 1)), dx, "fp64")


@pytest.mark.parametrize("precision", ["fp64", "fp32"])
def test_zero_tiny_huge_and_nonfinite(precision):
    f = np.random.default_rng(3).lognormal(size=(40, 70, 50, 1))
    f[:, :, 3:9] = 0.0
    f[:, :, 9:14] = -0.0
    f[:, 5:9, 20:25] = 1e-310
    f[:, 9:12, 20:25] *= 1e-290
    f[:, 12:15, 20:25] = np.random.default_rng(4).uniform(-1.0, 1.0, (40, 3, 5, 1)) * 1.7e308
    f[7, 8, 30], f[9, 9, 31], f[11, 12, 33] = np.inf, -np.inf, np.nan
    with np.errstate(all="ignore"):
        _check(f, 20.0, precision)
