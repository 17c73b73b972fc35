"""The tile kernel of the elevation modes and the further shapes against the per-lane kernel:
both round every operation alike, so the fields are equal, whatever the grid's sides and
spacing (tiles inside one lattice cell, tiles over so many that an octave runs per lane, ends
of rows and planes)."""
import pytest

from unnatural_planets_amd import spec as S

pytestmark = pytest.mark.gpu

GRIDS = [((2, 2, 2), 900.0), ((63, 5, 3), 17.0), ((64, 8, 2), 0.5), ((65, 9, 3), 61.0), ((130, 3, 4), 8.0), ((129, 131, 126), 8.0),
         ((200, 2, 2), 700.0)]


def _grid(dims, spacing):
    g = S.Grid()
    for a in range(3):
        g.dims[a] = dims[a]
        g.spacing[a] = spacing * (1.0, 1.3, 0.7)[a]
        g.origin[a] = -0.47 * spacing * dims[a] + (11.0, -903.0, 250.0)[a]
    return g


def _check(upf, s, dims, spacing):
    import torch
    g = _grid(dims, spacing)
    rows = upf.field_eval_grid(s, g, variant=upf.EVAL_AUTO)
    lanes = upf.field_eval_grid(s, g, variant=upf.EVAL_PER_LANE)
    assert torch.isfinite(lanes).all()
    assert torch.equal(rows, lanes)


@pytest.mark.parametrize("dims,spacing", GRIDS)
@pytest.mark.parametrize("mode", ["none", "simple", "legacy", "lakes", "islands", "craters"])
@pytest.mark.parametrize("compose", ["land", "water", "navigation", "elevation", "elevation_raw"])
def test_modes(upf, mode, compose, dims, spacing):
    _check(upf, S.spec_elevation_mode(mode, 5, "torus", (1200.0, 450.0), compose), dims, spacing)


@pytest.mark.parametrize("dims,spacing", GRIDS)
@pytest.mark.parametrize("shape,params", [("gear", ()), ("knot", ()), ("asteroid", (0.7, 1234.0)), ("bowl", ())])
def test_shapes_and_layers(upf, shape, params, dims, spacing):
    layers = [S.layer("gradient", "ridged", 5, 0.002, 2.1, -0.4, 3.0, 7), S.layer("value", "none", 1, 0.004, weight=0.5, seed=9, blend="mask"),
              S.layer("cellular", "fbm", 2, 0.003, weight=2.0, seed=11, jitter=0.8, blend="lerp"),
              S.layer("simplex", "fbm", 3, 0.002, weight=1.5, seed=13)]
    s = S.field_spec(shape, params, layers, "land", 0.1)
    if shape == "bowl":  # a composition runs the exact form with an elevation mode only
        s = S.spec_elevation_mode("lakes", 3, shape, params)
    _check(upf, s, dims, spacing)


def test_signs_and_mesh(upf):
    """The fused sign words give the mesh of the stored field."""
    import torch
    s, g = S.spec_elevation_mode("lakes", 8), S.grid_reference(71)
    f, ws, nv, nt = upf.field_mesh_count(s, g)
    a = upf.mc_emit_counted(f, g, 0.0, ws, nv, nt)
    b = upf.mc_extract(f, g)
    assert nv > 0 and torch.equal(a.positions, b.positions) and torch.equal(a.indices, b.indices)
