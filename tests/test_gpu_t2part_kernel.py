"""The T2part kernel's two forms (two voxels per thread with 16-byte loads, one voxel per thread) against the oracle:
even and odd volumes, a distribution that is not 16-byte aligned, bin counts around the rows read at once (12), the
smallest and the largest count, NaN and empty voxels, the sigmoid weights."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("shape,n,offset", [
    ((6, 5, 2), 40, 0), ((7, 5, 3), 40, 0), ((6, 5, 2), 40, 1), ((64, 9, 1), 12, 0), ((31, 17, 1), 13, 0),
    ((2, 1, 1), 2, 0), ((1, 1, 1), 64, 0), ((130, 4, 1), 64, 1),
])
@pytest.mark.parametrize("sigmoid", [None, 5e-3])
def test_t2part_forms_match_oracle(dmi, oracle, shape, n, offset, sigmoid):
    import torch

    from decaes_amd import device as D

    rng = np.random.default_rng(n + shape[0])
    V = int(np.prod(shape))
    dist = np.asfortranarray(rng.uniform(0, 1, (*shape, n)) * (rng.uniform(0, 1, (*shape, n)) > 0.5))
    if V > 2:
        dist[0, 0, 0, n - 1] = np.nan
        dist[1, 0, 0, :] = 0.0
    T2R, SP, MP = (10e-3, 2.0), (10e-3, 40e-3 if n > 2 else 2.0), (40e-3 if n > 2 else 10e-3, 2.0)
    buf = torch.zeros(V * n + 1, dtype=torch.float64, device="cuda")
    d = buf[offset:offset + V * n].view(n, *shape[::-1])
    d.copy_(torch.from_numpy(np.ascontiguousarray(dist.T)))
    assert (d.data_ptr() % 16 == 0) == (offset == 0)
    opts = dmi.T2partOptions(MatrixSize=shape, nT2=n, T2Range=T2R, SPWin=SP, MPWin=MP, Sigmoid=sigmoid, Silent=True)
    out = {k: torch.full(shape[::-1], float("nan"), dtype=torch.float64, device="cuda") for k in ("sfr", "sgm", "mfr", "mgm")}
    D.t2part_device(d, opts, out)
    o = oracle.t2part(dist, T2R, SP, MP, Sigmoid=sigmoid)
    for k in out:
        g, e = out[k].cpu().numpy().T, o[k]
        assert np.array_equal(np.isnan(g), np.isnan(e)), k
        ok = ~np.isnan(e)
        # sums of at most 64 terms in the same order, one exp: 1e-12 as the other T2part tests
        assert np.all(np.abs(g[ok] - e[ok]) <= 1e-12 * np.maximum(np.abs(e[ok]), 1e-300)), k
