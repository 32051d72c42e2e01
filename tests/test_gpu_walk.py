"""The walking line solvers (FP64, built-in shapes) against the solvers on
stored stencils, which explicit launch shapes ask for and which are held to
the CPU oracle: the same operators in another order of the same FP64
operations, so the two differ by round-off.

Tolerance: a slab applies about 100 rounded operations of a few ulp to a field
value, with condition numbers of the line systems near 1 (diagonal 1 + O(mu)):
1e-13 relative L2 over up to 6 slabs, taken ten times larger.
"""
import json

import numpy as np
import pytest

import oracle
from nemaktis_amd import bpm_backend, fields

pytestmark = pytest.mark.gpu

TOL = 1e-12


def _director(dims, seed):
    """smooth periodic director with some noise in all components"""
    Nx, Ny, Nz = dims
    rng = np.random.default_rng(seed)
    z, y, x = np.meshgrid(np.arange(Nz), np.arange(Ny) / max(1, Ny - 1), np.arange(Nx) / max(1, Nx - 1), indexing="ij")
    n = np.stack([np.cos(2 * np.pi * x + 0.3 * z), np.sin(2 * np.pi * y - 0.2 * z),
                  0.8 + 0.5 * np.cos(2 * np.pi * (x + y))], -1)
    n += 0.2 * rng.standard_normal(n.shape)
    return n / np.linalg.norm(n, axis=-1, keepdims=True)


def _compare(dims, lc, s, mask=None, formula="", E_in=None, **kw):
    print("[gpu case]", dims, flush=True)
    js = json.dumps(s)
    chunks = 64 if max(dims) <= 1025 else 128  # of at most 16 points
    stored = {"x_chunks": chunks, "x_rows": 1, "y_chunks": chunks, "y_cols": 2}
    a = bpm_backend.propagate(js, lc, mask_vals=mask, mask_formula=formula, E_in=E_in, **kw)
    b = bpm_backend.propagate(js, lc, mask_vals=mask, mask_formula=formula, E_in=E_in, tuning=stored)
    assert np.isfinite(a).all()
    a, b = (v.reshape(v.shape[0], v.shape[1], 2, -1) for v in (a, b))
    err = np.linalg.norm(a - b, axis=-1) / np.linalg.norm(b, axis=-1)
    assert err.max() < TOL, err.max()


# march lines of Nx - 1 and Ny - 1 points around the ends of the launch shapes, with last strips of one line; strips that
# are long along x, and lines above 1024 points, take the stored stencils on both sides
@pytest.mark.parametrize("Nx,Ny", [(17, 17), (18, 33), (16, 40), (40, 16), (34, 130), (129, 66), (200, 97), (258, 50),
                                   (400, 19), (512, 18), (513, 20), (514, 21), (25, 769), (1024, 17), (18, 1025),
                                   (1026, 17)])
def test_line_lengths(Nx, Ny):
    dims = (Nx, Ny, 4)
    s = fields.make_settings(dims, (0.1, 0.13, 0.1), [0.6], wavevectors=((0.0, 0.0), (0.11, -0.07)), nhost="1.5")
    _compare(dims, _director(dims, Nx + Ny), s)


@pytest.mark.parametrize("nw", [0, 1, 2, 3])
def test_neumann_depths_batched(nw):
    """several wavelengths and pairs in one batch"""
    dims = (67, 45, 6)
    s = fields.make_settings(dims, (0.1, 0.1, 0.1), [0.5, 0.62], wavevectors=((0.0, 0.0), (0.1, 0.05), (-0.2, 0.1)),
                             ne_imag="0.002", n_woodbury=nw)
    _compare(dims, _director(dims, nw), s, wl_batch=0)


@pytest.mark.parametrize("field_type", ["Director", "Q-tensor"])
def test_masked_fields(field_type):
    """formula weights at the droplet's surface, a host medium, caller fields"""
    dims = (35, 50, 6)
    lc, mask, formula = fields.droplet(*dims, (0.1, 0.1, 0.1), 1.2)
    lc = np.asarray(lc).reshape(dims[2], dims[1], dims[0], 3)
    if field_type != "Director":
        x, y, z = (lc[..., i] for i in range(3))
        lc = np.stack([x * x - 1 / 3, y * y - 1 / 3, z * z - 1 / 3, x * y, x * z, y * z], -1)
    s = fields.make_settings(dims, (0.1, 0.1, 0.1), [0.55], wavevectors=((0.0, 0.0), (0.15, 0.1)), nhost="1.55",
                             field_type=field_type, beam_profile="GaussianBeam(2.0)")
    _compare(dims, lc, s, mask=mask, formula=formula)
    rng = np.random.default_rng(7)
    E = rng.standard_normal(fields.output_shape(s)) + 1j * rng.standard_normal(fields.output_shape(s))
    s["Physics settings"]["Initial conditions"]["Beam profile"] = "None"
    _compare(dims, lc, s, mask=mask, E_in=E)


@pytest.mark.parametrize("use_graph", [False, True])
def test_retuning_to_stored_stencils_and_back(use_graph):
    """a resident job whose solvers change gives each route's own result"""
    dims = (40, 36, 5)
    s = fields.make_settings(dims, (0.1, 0.1, 0.1), [0.6], wavevectors=((0.0, 0.0), (0.1, 0.05)))
    lc = _director(dims, 11)
    shape = fields.output_shape(s)
    out = []
    with bpm_backend.Context(json.dumps(s), lc, int(np.prod(shape)), precision=64, use_graph=use_graph) as ctx:
        for tuning in (None, {"x_chunks": 16, "x_rows": 2, "y_chunks": 16, "y_cols": 8}, None):
            if out:
                ctx.set_tuning(tuning)
            for _ in range(2):
                ctx.propagate()
            out.append(ctx.download(np.empty(shape, np.complex128)))
    assert np.array_equal(out[0], out[2])
    assert np.linalg.norm(out[0] - out[1]) < TOL * np.linalg.norm(out[1])


# thin lines of points in thick slabs couple strongly (mu / dx^2 near 1), so that the reduction carries weight
@pytest.mark.parametrize("dims", [(200, 120, 40), (66, 514, 30), (129, 129, 60)])
def test_no_further_from_the_oracle_than_the_stored_stencils(dims):
    """The reduced systems are solved with corrections to the right-hand side:
    rescaled at every stage, it was 1.9 to 3.1 times as far off here.  Two
    routes of equal round-off are equally far from the oracle, whose own is of
    the same order; half as much again is allowed for."""
    s = fields.make_settings(dims, (0.05, 0.05, 0.2), [0.55], no="1.5", ne="1.55")
    lc = fields.random_smooth(*dims, (0.05, 0.05, 0.2), seed=2, corr_length=0.6)
    js, want = json.dumps(s), oracle.propagate(s, lc)
    walk = bpm_backend.propagate(js, lc)
    stored = bpm_backend.propagate(js, lc, tuning={"x_chunks": 64, "x_rows": 1, "y_chunks": 64, "y_cols": 2})
    assert np.linalg.norm(walk - want) < 1.5 * np.linalg.norm(stored - want)


# mesh, directions a wavelength, wavelengths: every kernel instance of the walk (chunks of 2 to 8 points with 16, 8, 4 and 2
# lines a block) along x and along y, of whole chunks or with shorter ones (tests/test_walk_route_host.py looks them up)
SHAPES = [(9, 9, 1, 1), (10, 10, 1, 1), (14, 14, 1, 1), (17, 17, 1, 1), (18, 18, 1, 1), (26, 26, 1, 1), (33, 33, 1, 1),
          (34, 34, 1, 1), (50, 50, 1, 1), (66, 66, 1, 1), (82, 82, 1, 1), (98, 98, 1, 1), (130, 130, 1, 1),
          (162, 162, 1, 1), (82, 82, 7, 1), (66, 66, 19, 1), (66, 770, 1, 1), (770, 66, 1, 1), (9, 898, 1, 1),
          (898, 65, 1, 1), (86, 386, 1, 3), (386, 86, 1, 3), (98, 450, 1, 3), (450, 98, 1, 3), (114, 338, 1, 3),
          (338, 114, 1, 3), (194, 194, 1, 3), (226, 226, 1, 3), (1025, 65, 1, 1), (66, 1024, 1, 1)]


@pytest.mark.parametrize("Nx,Ny,nq,nwl", SHAPES)
def test_every_kernel_instance(Nx, Ny, nq, nwl):
    dims = (Nx, Ny, 3)
    s = fields.make_settings(dims, (0.1, 0.13, 0.1), [0.5 + 0.06 * k for k in range(nwl)],
                             wavevectors=[(0.11 - 0.01 * k, 0.02 * k - 0.07) for k in range(nq)], nhost="1.5")
    _compare(dims, _director(dims, Nx + Ny), s, wl_batch=0)
