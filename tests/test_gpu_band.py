"""Grids of many rows are evaluated in bands of eight or four rows, small ones two rows at a time:
the same values.  A large grid is compared with its planes evaluated a few at a time, over
ragged sides, all layer kinds and blends, spacings at which a wave spans few cells, more
columns than a band's share and more than fit at all, bands over several cells and cells
past the pairs' reach.  The adjoint's bands of four rows likewise."""
import pytest

from unnatural_planets_amd import spec as S

pytestmark = pytest.mark.gpu

# the fewest bands of eight, one fewer plane, the fewest of four, ragged rows and row ends, one
# band a plane, too few rows for eight
DIMS = [(64, 64, 1024), (64, 32, 1023), (64, 16, 512), (65, 37, 300), (3, 9, 1030), (130, 5, 700), (130, 4, 700), (257, 66, 90)]


def _layers(kind):
    if kind == "blends":
        return [S.layer("gradient", "ridged", 6, 0.002, 2.1, -0.4, 3.0, 7), S.layer("value", "none", 1, 0.004, weight=0.5, seed=9, blend="mask"),
                S.layer("cellular", "fbm", 3, 0.001, weight=2.0, seed=11, jitter=0.8, blend="lerp"),
                S.layer("value", "fbm", 3, 0.003, weight=1.5, seed=13)]
    if kind == "cells":
        return [S.layer("cellular", "ridged", 2, 0.003, weight=2.0, seed=11), S.layer("cellular", "none", 1, 0.0625, weight=1.0, seed=12)]
    if kind == "cells8":  # more octaves than the pairs hold
        return [S.layer("cellular", "fbm", 8, 0.0005, weight=2.0, seed=11)]
    if kind == "wide":
        return [S.layer("gradient", "fbm", 3, 0.12, weight=2.0, seed=21), S.layer("value", "fbm", 2, 0.9, weight=1.0, seed=22)]
    return [S.layer("simplex", "fbm", 3, 0.002, weight=1.5, seed=13)]


def _grid(dims, spacing, k0=0, n=None):
    """The grid, or n of its planes from plane k0 on."""
    g = S.Grid()
    for a in range(3):
        g.dims[a] = dims[a]
        g.spacing[a] = spacing * (1.0, 1.5, 0.5)[a]
        g.origin[a] = -round(0.5 * dims[a]) * g.spacing[a] + (11.0, -896.0, 256.0)[a]
    if n:
        g.dims[2] = n
        g.origin[2] += k0 * g.spacing[2]  # exact: multiples of an eighth
    return g


@pytest.mark.parametrize("variant", ["rows", "lanes"])
@pytest.mark.parametrize("first", ["bands", "pairs"])
def test_batch_of_both_kinds(upf, first, variant):
    """Chunks in bands between chunks in row pairs (too few rows, an octave too fine for the
    spacing), small ones of several a workgroup: each as its own grid."""
    import torch
    from unnatural_planets_amd.batch import Batch
    sizes = [((65, 37, 300), 8.0, "blends"), ((9, 7, 5), 8.0, "blends"), ((130, 4, 70), 8.0, "blends"), ((3, 9, 530), 8.0, "cells"),
             ((2, 2, 2), 8.0, "blends"), ((2, 6, 2), 8.0, "wide"), ((64, 65, 66), 61.0, "wide"), ((70, 31, 90), 8.0, "simplex"),
             ((5, 5, 5), 0.5, "cells"), ((128, 64, 250), 0.5, "wide")]
    if first == "pairs":
        sizes = sizes[::-1]
    chunks = (S.Chunk * len(sizes))()
    for c, (dims, spacing, kind) in zip(chunks, sizes):
        c.spec = S.field_spec("torus", (1200.0, 450.0), _layers(kind), "land", 0.1)
        c.grid = _grid(dims, spacing)
        c.iso = 900.0
    v = upf.EVAL_ROWS if variant == "rows" else upf.EVAL_PER_LANE
    b = Batch(chunks, S.BatchOpts(v, 0, 0, 0))
    b.size_outputs()
    b.run()
    table = b.mesh_table()
    for i, c in enumerate(chunks):
        f = upf.field_eval_grid(c.spec, c.grid, variant=v)
        assert torch.equal(b.field_of(i), f), sizes[i]
        m, bm = upf.mc_extract(f, c.grid, 900.0), b.mesh_of(i, table)
        assert torch.equal(bm.indices, m.indices) and torch.equal(bm.positions, m.positions), sizes[i]


@pytest.mark.parametrize("dims", DIMS)
@pytest.mark.parametrize("spacing", [0.5, 8.0, 9.5, 61.0])
@pytest.mark.parametrize("kind", ["blends", "cells", "cells8", "wide", "simplex"])
@pytest.mark.parametrize("shape,params,compose", [("torus", (1200.0, 450.0), "land"), ("pipe", (), "navigation"), ("none", (), "elevation_raw"),
                                                  ("hemispheres", (), "water"), ("sphere", (900.0,), "elevation")])
def test_bands_are_rows(upf, shape, params, compose, kind, spacing, dims):
    import torch
    s = S.field_spec(shape, params, _layers(kind), compose, 0.1)
    whole = upf.field_eval_grid(s, _grid(dims, spacing))
    assert torch.isfinite(whole).all()
    for k in range(0, dims[2], 30):  # planes too few for bands
        k = min(k, dims[2] - 30)
        part = upf.field_eval_grid(s, _grid(dims, spacing, k, 30))
        assert torch.equal(whole[k:k + 30], part)


def test_signs_and_mesh(upf):
    """The sign words that the band kernel writes give the mesh of the stored field."""
    import torch
    s, g = S.spec_torus_ridged_voronoi(8), S.grid_torus(133)
    f, ws, nv, nt = upf.field_mesh_count(s, g)
    a = upf.mc_emit_counted(f, g, 0.0, ws, nv, nt)
    b = upf.mc_extract(f, g)
    assert nv > 0 and torch.equal(a.positions, b.positions) and torch.equal(a.indices, b.indices)


# the fewest bands of four rows, ragged, one band a plane, more rows than planes
GRAD_DIMS = [(64, 16, 1024), (65, 37, 210), (130, 3, 1400), (257, 201, 34)]


@pytest.mark.parametrize("dims", GRAD_DIMS)
@pytest.mark.parametrize("spacing", [0.5, 8.0, 61.0])
@pytest.mark.parametrize("kind", ["sum", "cells", "cells8", "wide"])
@pytest.mark.parametrize("shape,params,compose", [("torus", (1200.0, 450.0), "land"), ("none", (), "elevation_raw"), ("box", (700.0, 500.0, 300.0, 90.0), "water"),
                                                  ("capsule", (900.0, 300.0), "elevation")])
@pytest.mark.parametrize("theta", [True, False])
def test_adjoint_bands_are_rows(upf, theta, shape, params, compose, kind, spacing, dims):
    """f and df/dp of a large grid equal those of its planes taken a few at a time (rows), and
    dL/dtheta their sum within 1e-4 of its scale, as the grid adjoint is held to elsewhere."""
    import torch
    layers = _layers(kind) if kind != "sum" else [S.layer("gradient", "ridged", 4, 0.002, 2.1, -0.4, 3.0, 7),
                                                  S.layer("value", "fbm", 3, 0.003, weight=1.5, seed=13),
                                                  S.layer("cellular", "none", 1, 0.004, weight=2.0, seed=11, jitter=0.8)]
    s = S.field_spec(shape, params, layers, compose, 0.1)
    w = torch.randn(dims[::-1], device="cuda", generator=torch.Generator("cuda").manual_seed(5)) if theta else None
    f, dfdx, th = upf.field_adjoint_grid(s, _grid(dims, spacing), w)
    assert torch.isfinite(f).all() and torch.isfinite(dfdx).all()
    total = 0.0
    for k in range(0, dims[2], 34):
        n = min(34, dims[2] - k)
        if n < 2:
            k, n = k - 1, 2
        pf, pd, pt = upf.field_adjoint_grid(s, _grid(dims, spacing, k, n), w[k:k + n].contiguous() if theta else None)
        assert torch.equal(f[k:k + n], pf) and torch.equal(dfdx[k:k + n], pd)
        if theta:
            if (k % 34) and n == 2:  # the plane before is counted already
                zero = w[k:k + n].clone()
                zero[0] = 0
                pt = upf.field_adjoint_grid(s, _grid(dims, spacing, k, n), zero)[2]
            total = total + pt.double()
    if theta:
        assert float((th.double() - total).abs().max()) <= 1e-4 * max(float(total.abs().max()), 1e-6)
