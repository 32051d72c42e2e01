"""Transform lengths with prime factors above 13 (matrix-core stages) in the
refocus and the screen filter, against the FP64 CPU oracles.

Tolerance: a stage of R terms rounds like sqrt(R) eps, R <= 2039, a few
operations a term and two transforms: below 1e-13; 1e-12 relative L2.
"""
import json

import numpy as np
import pytest

import oracle
import viewer_oracle as vo
from nemaktis_amd import bpm_backend, fields, viewer

pytestmark = pytest.mark.gpu

TOL = 1e-12


# one prime (a last k tile of 1 to 16 rows), a prime and small factors, two primes (twiddles before the second stage),
# 8, 4 and 2 lines per block, the longest
@pytest.mark.parametrize("Nx,Ny", [(17, 31), (29, 19), (161, 46), (289, 34), (323, 37), (127, 251), (257, 62),
                                   (509, 85), (1021, 3), (5, 1021), (2039, 2), (3, 2039), (2047, 4), (4, 2023)])
def test_refocus(Nx, Ny):
    print("[gpu case] focus", (Nx, Ny), flush=True)
    of = viewer.OpticalFields(wavelengths=[0.55], max_NA_objective=0.6, max_NA_condenser=0.0, N_radial_wavevectors=1,
                              n_out=1.1, mesh_lengths=(0.1 * (Nx - 1), 0.1 * (Ny - 1)), mesh_dimensions=(Nx, Ny))
    rng = np.random.default_rng(Nx)
    of.vals = rng.standard_normal(of.vals.shape) + 1j * rng.standard_normal(of.vals.shape)
    of.focus_fields(1.3)
    dx, dy = of.get_mesh_spacings()
    want = vo.focus(of.vals, dx, dy, of.get_wavelengths(), np.array([1.1]), of.get_wavevectors(), of._NA, 1.3, 0.0)
    got = of.focused_vals
    a, b = (v.reshape(-1, Nx * Ny) for v in (got, want))
    assert (np.linalg.norm(a - b, axis=1) / np.linalg.norm(b, axis=1)).max() < TOL


def test_a_line_with_a_nan_leaves_the_others_alone():
    """the tiles of a stage hold several lines side by side"""
    Nx, Ny = 161, 24
    of = viewer.OpticalFields(wavelengths=[0.55], max_NA_objective=0.6, max_NA_condenser=0.0, N_radial_wavevectors=1,
                              n_out=1.0, mesh_lengths=(16.0, 2.3), mesh_dimensions=(Nx, Ny))
    rng = np.random.default_rng(3)
    of.vals = rng.standard_normal(of.vals.shape) + 1j * rng.standard_normal(of.vals.shape)
    of.focus_fields(0.7)
    want = of.focused_vals.reshape(4, -1).copy()
    v = of.vals.copy().reshape(4, Ny, Nx)
    v[2, 5, 17] = np.nan
    of.vals = v.reshape(of.vals.shape)
    of.focus_fields(0.7)
    got = of.focused_vals.reshape(4, -1)
    assert np.isnan(got[2]).all()
    assert np.array_equal(got[[0, 1, 3]], want[[0, 1, 3]])


@pytest.mark.parametrize("dims", [(8, 323, 3), (161, 23, 3), (6, 2039, 2)])
def test_screen_filter(dims):
    print("[gpu case]", dims, flush=True)
    lc = fields.twisted_nematic(*dims)
    s = fields.make_settings(dims, (0.1, 0.1, 0.1), [0.6], wavevectors=((0.05, 0.1),))
    got = bpm_backend.propagate(json.dumps(s), lc)
    want = oracle.propagate(s, lc)
    a, b = (v.reshape(4, -1) for v in (got, want))
    # planes without a field (no twist within the mesh) have no relative error
    keep = np.linalg.norm(b, axis=1) > 1e-6
    assert keep.sum() >= 2
    assert (np.linalg.norm(a - b, axis=1)[keep] / np.linalg.norm(b, axis=1)[keep]).max() < 1e-10


# rows and columns of enough lines for the stages on the matrix cores (single planes of the meshes above go by the direct
# sum along one axis): 16, 8, 4 and 2 lines a block, one prime and a prime with small factors
@pytest.mark.parametrize("Nx,Ny,nwl", [(17, 64, 16), (34, 64, 17), (71, 64, 8), (127, 33, 16), (161, 128, 1), (251, 64, 4),
                                       (509, 64, 4), (1021, 32, 8), (1042, 6, 1), (64, 1409, 2), (6, 17, 8)])
def test_refocus_of_many_lines(Nx, Ny, nwl):
    print("[gpu case] focus", (Nx, Ny, nwl), flush=True)
    wl = list(np.linspace(0.5, 0.6, nwl))
    of = viewer.OpticalFields(wavelengths=wl, max_NA_objective=0.6, max_NA_condenser=0.0, N_radial_wavevectors=1,
                              n_out=1.1, mesh_lengths=(0.1 * (Nx - 1), 0.1 * (Ny - 1)), mesh_dimensions=(Nx, Ny))
    rng = np.random.default_rng(Nx)
    of.vals = rng.standard_normal(of.vals.shape) + 1j * rng.standard_normal(of.vals.shape)
    of.focus_fields(1.3)
    dx, dy = of.get_mesh_spacings()
    want = vo.focus(of.vals, dx, dy, of.get_wavelengths(), np.full(nwl, 1.1), of.get_wavevectors(), of._NA, 1.3, 0.0)
    a, b = (v.reshape(-1, Nx * Ny) for v in (of.focused_vals, want))
    assert (np.linalg.norm(a - b, axis=1) / np.linalg.norm(b, axis=1)).max() < TOL


@pytest.mark.parametrize("dims", [(8, 1042, 2), (9, 521, 2), (161, 130, 2), (40, 51, 2)])
def test_screen_filter_of_many_lines(dims):
    print("[gpu case]", dims, flush=True)
    lc = fields.twisted_nematic(*dims)
    s = fields.make_settings(dims, (0.1, 0.1, 0.1), [0.6], wavevectors=((0.05, 0.1), (0.0, 0.1), (0.1, 0.0)))
    got, want = (v.reshape(12, -1) for v in (bpm_backend.propagate(json.dumps(s), lc), oracle.propagate(s, lc)))
    keep = np.linalg.norm(want, axis=1) > 1e-6
    assert keep.sum() >= 6
    assert (np.linalg.norm(got - want, axis=1)[keep] / np.linalg.norm(want, axis=1)[keep]).max() < 1e-10
