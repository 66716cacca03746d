"""The register-resident voxel kernel (the automatic schedule where a size class holds the train) against the
memory-resident one with every workspace row in LDS: the same arithmetic in the same order, so every output is equal
bit for bit. Sizes on both sides of each class edge, the smallest and the largest, each regularization and basis
source."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

CASES = [
    # nTE, nT2, Reg, register-resident, other options
    (4, 2, "mdp", True, dict(nRefAngles=2)),
    (5, 64, "none", True, {}),
    (32, 40, "chi2", True, {}),
    (33, 37, "gcv", True, {}),
    (48, 64, "lcurve", True, {}),
    (49, 2, "chi2", True, {}),
    (56, 60, "lcurve", True, {}),
    (57, 63, "gcv", True, {}),
    (64, 64, "mdp", True, {}),
    (64, 64, "lcurve", True, dict(SetFlipAngle=150.0)),
    (65, 40, "mdp", False, {}),
    (80, 64, "none", True, dict(RefConAngle=165.0)),
    (81, 64, "none", False, {}),
    (47, 33, "chi2", True, dict(precision="mixed", SaveNNLSBasis=True)),
    (25, 64, "gcv", True, dict(b1=True)),
    (61, 7, "chi2", True, dict(precision="mixed", b1=True)),
]


@pytest.mark.parametrize("m,n,reg,resident,extra", CASES)
def test_register_schedule_is_bit_identical(dmi, m, n, reg, resident, extra):
    print(f"[register] m={m} n={n} {reg} {extra}", flush=True)
    extra = dict(extra)
    shape = (7, 5, 2)
    img, _ = dmi.synth_mse(shape, m, 8e-3, ncomp=4, mask_fraction=0.9, seed=100 + m)
    alpha = np.asfortranarray(np.random.default_rng(m).uniform(120, 180, shape)) if extra.pop("b1", False) else None
    K = extra.pop("nRefAngles", 24)
    kw = dict(TE=8e-3, nT2=n, T2Range=(8e-3, 2.0), Reg=reg, nRefAngles=K, nRefAnglesMin=min(5, K), SaveRegParam=True,
              SaveResidualNorm=True, SaveDecayCurve=True, Silent=True, Chi2Factor=1.02, NoiseLevel=2e-3, **extra)
    res = {}
    for sched in ("lds", "auto"):
        maps, dist = dmi.T2mapSEcorr(img, dmi.T2mapOptions.from_image(img, schedule=sched, **kw), alpha=alpha)
        res[sched] = (maps, dist, dmi.context(0).stats())
    (ml, dl, sl), (ma, da, sa) = res["lds"], res["auto"]
    assert sl["lds_rows"] == m + n and sa["lds_rows"] == (0 if resident else m + n)
    assert np.isfinite(dl).any() and np.array_equal(dl, da, equal_nan=True)
    for k in ml:
        assert np.array_equal(ml[k], ma[k], equal_nan=True), k
    assert sl["nnls_solves"] == sa["nnls_solves"] and sl["fp64_flops"] == sa["fp64_flops"]
