"""Statistics of an ensemble of trajectories on the device (level probabilities with
their variance, expectation values) against numpy, from one trajectory of one level
to more levels than a block's and more trajectories than its chunks."""
import ctypes

import numpy as np
import pytest

import quac_amd as qa

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("levels", [1, 2, 20, 64, 65, 131])
@pytest.mark.parametrize("count", [1, 2, 5, 1030, 2500])
def test_ensemble_statistics(levels, count):
    rng = np.random.default_rng(levels + 7 * count)
    a = (rng.normal(size=(count, levels)) + 1j * rng.normal(size=(count, levels))) * rng.uniform(0.1, 1.0, (count, 1))
    v = qa.DeviceVec(count * levels, qa.FP64)
    v.set(a.reshape(-1))
    L = qa.lib()
    dbl, i64, vp = ctypes.c_double, ctypes.c_int64, ctypes.c_void_p
    L.qh_ens_probs.argtypes = [vp, i64, i64, ctypes.POINTER(dbl), ctypes.POINTER(dbl)]
    L.qh_ens_expect.argtypes = [vp, i64, i64, ctypes.c_int, vp, ctypes.c_int, vp, ctypes.POINTER(dbl),
                                ctypes.POINTER(dbl)]
    mean, var = (dbl * levels)(), (dbl * levels)()
    assert L.qh_ens_probs(v.h, count, levels, mean, var) == 0
    q = np.abs(a) ** 2
    q /= q.sum(1, keepdims=True)
    ref_mean, ref_var = q.mean(0), ((q - q.mean(0)) ** 2).sum(0) / max(count - 1, 1)
    # sums of `levels` and of `count` non-negative numbers, each a few roundings
    tol = (levels + count + 16) * 2.0 ** -53
    assert np.abs(np.array(mean) - ref_mean).max() <= tol * ref_mean.max()
    assert np.abs(np.array(var) - ref_var).max() <= 4 * tol
    # the level number (one operator of `levels` levels), and its lowering
    n = np.arange(levels)
    low = np.sqrt(np.arange(1.0, levels + 1))
    for table, ref in (([(k, k, float(k), 0.0) for k in range(levels)], (q * n).sum(1).mean()),
                       ([(k + 1 if k + 1 < levels else -1, k - 1, low[k], 0.0) for k in range(levels)],
                        ((a[:, :-1].conj() * a[:, 1:] * low[:-1]).sum(1) / (np.abs(a) ** 2).sum(1)).mean())):
        lev = (qa.QhLevel * levels)()
        for k, (nx, pv, re, im) in enumerate(table):
            lev[k].next, lev[k].prev, lev[k].re, lev[k].im = nx, pv, re, im
        op = qa.QhOp()
        op.stride, op.levels, op.tab = 1, levels, 0
        re, im = dbl(), dbl()
        assert L.qh_ens_expect(v.h, count, levels, 1, ctypes.addressof(op), levels, ctypes.addressof(lev),
                               ctypes.byref(re), ctypes.byref(im)) == 0
        assert abs(re.value + 1j * im.value - ref) <= 4 * tol * max(levels, 1)


# a workgroup of 256 and of 1024 threads a trajectory; the most amplitudes that the host
# sums, and one trajectory more; enough short trajectories for a wavefront each
@pytest.mark.parametrize("levels,count", [(257, 5), (300, 100), (1000, 9), (4096, 3), (4097, 2), (16384, 4), (513, 600),
                                          (64, 128), (64, 129), (260, 8192)])
def test_long_trajectories(levels, count):
    test_ensemble_statistics(levels, count)
