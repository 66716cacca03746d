"""The launch schedule measured for a set of sizes is kept for the process. Legacy and plain calls of the same sizes run
different kernels with different candidates (the register-resident kernel holds no legacy code), so neither may take the
choice measured for the other: a plain volume large enough to be measured, then legacy calls of those sizes, and the
other way round."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

M, N, TE, T2R = 24, 64, 10e-3, (10e-3, 2.0)
# split candidates exist at these sizes (3 workgroups per CU with every row in LDS), so a volume of this size is measured
LARGE, SMALL = (64, 64, 16), (9, 7, 2)


def _run(dmi, shape, K, seed, **kw):
    img, _ = dmi.synth_mse(shape, M, TE, ncomp=3, mask_fraction=1.0, seed=seed)
    opts = dmi.T2mapOptions.from_image(img, TE=TE, nT2=N, T2Range=T2R, Reg="chi2", Chi2Factor=1.02, nRefAngles=K,
                                       nRefAnglesMin=5, SaveRegParam=True, SaveResidualNorm=True, Silent=True, **kw)
    maps, dist = dmi.T2mapSEcorr(img, opts)
    return maps, dist, dmi.context(0).stats()


def _same(a, b):
    assert np.array_equal(a[1], b[1], equal_nan=True)
    for k in a[0]:
        assert np.array_equal(a[0][k], b[0][k], equal_nan=True), k
    assert a[2]["nnls_solves"] == b[2]["nnls_solves"] and a[2]["fp64_flops"] == b[2]["fp64_flops"]


def test_legacy_call_after_a_measured_plain_volume(dmi):
    print("[legacy-schedule] plain volume, then legacy", flush=True)
    _, _, st = _run(dmi, LARGE, 9, 1)
    assert st["lds_rows"] == 0  # the register-resident schedule won
    ref = _run(dmi, SMALL, 9, 2, legacy=True, schedule="lds")
    got = _run(dmi, SMALL, 9, 2, legacy=True)
    assert got[2]["lds_rows"] != 0
    _same(ref, got)


def test_plain_call_after_a_measured_legacy_volume(dmi):
    print("[legacy-schedule] legacy volume, then plain", flush=True)
    _, _, st = _run(dmi, LARGE, 10, 3, legacy=True)
    assert st["lds_rows"] != 0
    ref = _run(dmi, SMALL, 10, 4, schedule="lds")
    got = _run(dmi, SMALL, 10, 4)
    assert got[2]["lds_rows"] == 0
    _same(ref, got)
