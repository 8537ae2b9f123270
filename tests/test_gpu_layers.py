"""The layer kernel on its own (fsg_postproc_device) against the formulas in
numpy: sizes off the block size, both derivative forms, a skew, potentials
with |a_d| != 1, and values at which a square leaves binary64's range or a
logarithm is near zero (the form by squares hands those to the general one).

Each layer is a binary64 value of a few roundings stored as binary32: half a
unit of binary32 (2^-24, relative) plus 1e-13 of the terms."""
import ctypes

import numpy as np
import pytest

from fractalshades_amd import _native
from fractalshades_amd.postproc import continuous_iter, dem, normal_map

HALF_ULP = 2. ** -24 * (1. + 1e-6)


def run(Z, si, sr, desc):
    import torch
    n = si.size
    dev = [torch.from_numpy(np.ascontiguousarray(a)).cuda() for a in (Z.view(np.float64), si, sr)]
    nu, dm = (torch.empty(n, dtype=torch.float32, device="cuda") for _ in range(2))
    nrm = torch.empty(n, 2, dtype=torch.float32, device="cuda")
    _native.check(_native.load().fsg_postproc_device(
        ctypes.byref(desc), dev[0].data_ptr(), n, n, None, dev[1].data_ptr(), dev[2].data_ptr(), nu.data_ptr(),
        dm.data_ptr(), nrm.data_ptr(), torch.cuda.current_stream().cuda_stream))
    torch.cuda.synchronize()
    return nu.cpu().numpy(), dm.cpu().numpy(), nrm.cpu().numpy()


@pytest.mark.gpu
@pytest.mark.parametrize("holo", [True, False], ids=["holomorphic", "jacobian"])
@pytest.mark.parametrize("n,d,a_d,M,skew", [
    (1, 2., 1., 1e3, None), (63, 2., 1., 1e3, (1., 0., 0., 1.)), (257, 3., 8., 1e3, (0.6, -0.8, 1.1, 0.4)),
    (4099, 6., 1. / 32., 30., (1., 0.5, 0., 1.))])
def test_layers(holo, n, d, a_d, M, skew):
    rng = np.random.default_rng(n + holo)
    # |z| from just past 1 / k to beyond the root of the largest value
    log_mod = rng.uniform(0.5, 10., n)
    log_mod[rng.random(n) < 0.1] = rng.uniform(0.02, 0.6)
    log_mod[rng.random(n) < 0.1] = rng.uniform(200., 600.)
    z = np.exp(log_mod + 2j * np.pi * rng.random(n)) / min(1., a_d ** (1. / (d - 1.)))
    scale = np.where(rng.random(n) < 0.2, rng.uniform(-190., 190.), rng.uniform(-3., 9., n))
    der = rng.normal(size=(4, n)) * 10. ** scale
    if not holo:
        der[:, ::7] = np.stack((der[0, ::7], -der[1, ::7], der[1, ::7], der[0, ::7]))  # one singular value twice
    if holo:
        Z = np.stack((z, der[0] + 1j * der[1]))
    else:
        Z = np.concatenate((np.stack((z.real, z.imag)), der))
    si = rng.integers(1, 100000, n).astype(np.int32)
    sr = np.where(rng.random(n) < 0.9, 1, rng.integers(0, 3, n)).astype(np.int8)
    desc = _native.PostDesc(int(holo), 1 if holo else 2, d, a_d, M, 0., 0.)
    for i, s in enumerate(skew or (0.,) * 4):
        desc.skew[i] = s
    nu, dm, nrm = run(Z, si, sr, desc)
    esc = sr == 1
    for out in (nu, dm, nrm):
        assert np.isnan(out[~esc]).all()
    kw = dict(dzndc=Z[1][esc]) if holo else dict(jac=der[:, esc])
    nu_ref = continuous_iter(z[esc], si[esc], d=d, a_d=a_d, M=M)
    assert (np.abs(nu[esc] - nu_ref) <= HALF_ULP * np.abs(nu_ref) + 1e-13 * (si[esc] + 20.)).all()
    dem_ref = dem(z[esc], **kw)
    with np.errstate(over="ignore"):
        in_range = (dem_ref > 1.2e-38) & (dem_ref < 3.4e38)
        assert (np.abs(dm[esc] - dem_ref) <= (HALF_ULP + 1e-13) * dem_ref)[in_range].all()
        assert (dm[esc][~in_range] == dem_ref[~in_range].astype(np.float32)).all()
    small = np.ldexp(1., -np.frexp(np.abs(der[:2] if holo else der).max(0))[1])   # keeps z / d in range
    kw = dict(dzndc=(Z[1] * small)[esc]) if holo else dict(jac=(der * small)[:, esc])
    zs = z * np.ldexp(1., -np.frexp(np.abs(z))[1])
    nrm_ref = normal_map(zs[esc], skew=None if skew is None else np.reshape(skew, (2, 2)), **kw)
    # J^T z and the skew may cancel: 1e-13 of the terms, not of the sum
    assert (np.abs(nrm[esc][:, 0] - np.real(nrm_ref)) <= HALF_ULP + 1e-11).all()
    assert (np.abs(nrm[esc][:, 1] - np.imag(nrm_ref)) <= HALF_ULP + 1e-11).all()
