"""The band kernels (eight rows a wave, four, and the adjoint's four) against the row pairs, whose
values they share: each grid's planes evaluated again in parts of too few bands.  The counts
that the dispatch goes by are asserted, so that a moved bound cannot turn a comparison into one
of a kernel with itself.  Ragged rows, row ends and last bands; planes of few rows, on both
sides of the bounds; cells whose rows are too far apart to share their points."""
import pytest

from unnatural_planets_amd import spec as S

pytestmark = pytest.mark.gpu

FIELD8, FIELD4, GRAD4 = 8192, 2048, 4096  # fewest bands of a grid's field (eight rows, four) and adjoint


def _bands(dims, rows):
    return -(-dims[0] // 64) * -(-dims[1] // rows) * dims[2]


def _layers(kind):
    if kind == "blends":
        return [S.layer("gradient", "ridged", 6, 0.002, 2.1, -0.4, 3.0, 7), S.layer("value", "none", 1, 0.004, weight=0.5, seed=9, blend="mask"),
                S.layer("cellular", "fbm", 2, 0.001, weight=2.0, seed=11, jitter=0.8, blend="lerp"),
                S.layer("value", "fbm", 3, 0.003, weight=1.5, seed=13)]
    if kind == "sum":
        return [S.layer("gradient", "ridged", 4, 0.002, 2.1, -0.4, 3.0, 7), S.layer("value", "fbm", 3, 0.003, weight=1.5, seed=13),
                S.layer("cellular", "none", 1, 0.004, weight=2.0, seed=11, jitter=0.8)]
    if kind == "columns":  # up to 15, 30 or 60 columns an octave over 64 nodes at 0.5, 1 and 2 m
        return [S.layer("gradient", "fbm", 3, 0.12, weight=2.0, seed=21), S.layer("value", "fbm", 2, 0.24, weight=1.0, seed=22)]
    if kind == "cells":
        return [S.layer("cellular", "ridged", 2, 0.012, weight=2.0, seed=11), S.layer("gradient", "fbm", 3, 0.01, weight=1.0, seed=12)]
    return []


def _grid(dims, spacing, k0=0, n=None):
    """The grid, or n of its planes from plane k0 on (spacings are multiples of an eighth: exact)."""
    g = S.Grid()
    for a in range(3):
        g.dims[a], g.spacing[a] = dims[a], spacing[a]
        g.origin[a] = -round(0.5 * dims[a]) * spacing[a] + (11.0, -896.0, 256.0)[a]
    if n:
        g.dims[2] = n
        g.origin[2] += k0 * g.spacing[2]
    return g


def _parts(dims, rows, bound):
    """Plane ranges of fewer than `bound` bands that cover the grid, of two planes at least."""
    step = (bound - 1) // _bands((dims[0], dims[1], 1), rows)
    assert step >= 2 and _bands((dims[0], dims[1], step), rows) < bound
    for k in range(0, dims[2], step):
        n = min(step, dims[2] - k)
        yield (k, n) if n > 1 else (k - 1, 2)


def _check_field(upf, kind, compose, dims, spacing):
    import torch
    s = S.field_spec("torus", (1200.0, 450.0), _layers(kind), compose, 0.1)
    whole = upf.field_eval_grid(s, _grid(dims, spacing))
    assert torch.isfinite(whole).all()
    for k, n in _parts(dims, 4, FIELD4):
        assert torch.equal(whole[k:k + n], upf.field_eval_grid(s, _grid(dims, spacing, k, n)))


@pytest.mark.parametrize("dims,eight", [((64, 64, 1024), True), ((64, 64, 1023), False), ((65, 37, 820), True), ((130, 17, 911), True),
                                        ((257, 66, 184), True), ((3, 13, 4100), True), ((3, 12, 4100), False), ((193, 39, 1050), True)])
@pytest.mark.parametrize("kind,step", [("blends", 0.5), ("blends", 8.0), ("columns", 0.5), ("columns", 2.0), ("cells", 1.0)])
def test_eight_rows(upf, kind, step, dims, eight):
    assert (_bands(dims, 8) >= FIELD8 and dims[1] >= 13) == eight and _bands(dims, 4) >= FIELD4
    _check_field(upf, kind, "land", dims, (step, 1.5 * step, 0.5 * step))


@pytest.mark.parametrize("rows", [2, 3, 4, 5, 6, 7, 8, 12, 13, 14])
@pytest.mark.parametrize("kind,compose", [("blends", "land"), ("cells", "elevation_raw"), ("none", "land"), ("blends", "water")])
def test_planes_of_few_rows(upf, rows, kind, compose):
    dims = (70, rows, 4200)
    assert _bands(dims, 8) >= FIELD8
    _check_field(upf, kind, compose, dims, (1.0, 1.0, 1.0))


# rows 0.1 to 6 cells apart, over few cells along x or many
@pytest.mark.parametrize("apart", [4.0, 24.0, 26.0, 33.0, 34.0, 52.0, 53.0, 256.0])
@pytest.mark.parametrize("step", [0.5, 8.0])
def test_rows_far_apart(upf, step, apart):
    import torch
    dims = (130, 17, 911)
    _check_field(upf, "cells", "land", dims, (step, apart, 1.0))
    s = S.field_spec("none", (), _layers("cells"), "elevation_raw")
    f, dfdx, _ = upf.field_adjoint_grid(s, _grid(dims, (step, apart, 1.0)), None)
    for k, n in _parts(dims, 4, GRAD4):
        pf, pd, _ = upf.field_adjoint_grid(s, _grid(dims, (step, apart, 1.0), k, n), None)
        assert torch.equal(f[k:k + n], pf) and torch.equal(dfdx[k:k + n], pd)


def test_signs_and_mesh(upf):
    """The sign words that the eight-row kernel writes give the mesh of the stored field."""
    import torch
    s, g = S.spec_torus_ridged_voronoi(8), S.grid_torus(163)
    assert _bands((163, 163, 163), 8) >= FIELD8
    f, ws, nv, nt = upf.field_mesh_count(s, g)
    a = upf.mc_emit_counted(f, g, 0.0, ws, nv, nt)
    b = upf.mc_extract(f, g)
    assert nv > 0 and torch.equal(a.positions, b.positions) and torch.equal(a.indices, b.indices)


@pytest.mark.parametrize("dims", [(64, 16, 1024), (65, 37, 210), (130, 3, 1400), (257, 201, 34)])
@pytest.mark.parametrize("kind,step", [("sum", 0.5), ("sum", 8.0), ("columns", 0.5), ("cells", 8.0)])
@pytest.mark.parametrize("shape,params,compose", [("torus", (1200.0, 450.0), "land"), ("none", (), "elevation_raw"), ("capsule", (900.0, 300.0), "elevation")])
@pytest.mark.parametrize("theta", [True, False])
def test_adjoint_bands(upf, theta, shape, params, compose, kind, step, dims):
    """f and df/dp equal the row form's, and dL/dtheta the parts' sum within 1e-4 of its scale, as
    the grid adjoint is held to elsewhere."""
    import torch
    assert _bands(dims, 4) >= GRAD4
    spacing = (step, 1.5 * step, 0.5 * step)
    s = S.field_spec(shape, params, _layers(kind), compose, 0.1)
    w = torch.randn(dims[::-1], device="cuda", generator=torch.Generator("cuda").manual_seed(5)) if theta else None
    f, dfdx, th = upf.field_adjoint_grid(s, _grid(dims, spacing), w)
    assert torch.isfinite(f).all() and torch.isfinite(dfdx).all()
    total, done = 0.0, 0
    for k, n in _parts(dims, 4, GRAD4):
        part = None
        if theta:
            part = w[k:k + n].clone()
            part[:done - k] = 0  # planes that the part before has counted
        pf, pd, pt = upf.field_adjoint_grid(s, _grid(dims, spacing, k, n), part)
        assert torch.equal(f[k:k + n], pf) and torch.equal(dfdx[k:k + n], pd)
        total, done = (total + pt.double() if theta else 0.0), k + n
    if theta:
        assert float((th.double() - total).abs().max()) <= 1e-4 * max(float(total.abs().max()), 1e-6)
