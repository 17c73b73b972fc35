"""The exact form's kernels over grids on both sides of the bounds that choose between them (few
rows, few planes, numbers of nodes): one-plane tiles, four-plane tiles and the per-lane form
round every operation alike, so the fields are the per-lane form's."""
import pytest

from unnatural_planets_amd import spec as S

pytestmark = pytest.mark.gpu

# 2^21 nodes and more of 2 to 9 rows or planes; a little below and above 2^21 and 2^22
DIMS = [(1040, n, 2100 // n * 2) for n in (2, 3, 5, 9)] + [(1040, 4200 // n, n) for n in (2, 3, 5, 9)] + \
       [(512, 2, 600), (127, 127, 128), (133, 132, 128), (163, 160, 159), (167, 164, 160), (2, 1030, 1025)]


def _spec(name):
    if name == "gear lattices":
        return S.field_spec("gear", (), [S.layer("gradient", "ridged", 5, 0.002, 2.1, -0.4, 3.0, 7), S.layer("value", "fbm", 2, 0.004, weight=2.0, seed=9)], "land", 0.1)
    if name == "gear cells":
        return S.field_spec("gear", (), [S.layer("cellular", "fbm", 2, 0.003, weight=2.0, seed=11, jitter=0.8)], "land", 0.1)
    if name == "gear mixed":
        return S.field_spec("gear", (), [S.layer("gradient", "ridged", 3, 0.002, weight=3.0, seed=7), S.layer("simplex", "fbm", 3, 0.002, weight=1.5, seed=13)], "land", 0.1)
    if name == "knot":
        return S.field_spec("knot", (), [], "land", 0.1)
    if name == "lakes water":
        return S.spec_elevation_mode("lakes", 5, "torus", (1200.0, 450.0), "water")
    return S.spec_elevation_mode(name, 5, "torus", (1200.0, 450.0))


@pytest.mark.parametrize("dims", DIMS)
@pytest.mark.parametrize("name", ["none", "simple", "legacy", "lakes", "islands", "craters", "lakes water", "gear lattices", "gear cells", "gear mixed", "knot"])
def test_thin_grids(upf, name, dims):
    import torch
    g = S.Grid()
    for a in range(3):
        g.dims[a], g.spacing[a] = dims[a], (3.0, 2.5, 4.0)[a]
        g.origin[a] = -0.47 * g.spacing[a] * dims[a] + (11.0, -903.0, 250.0)[a]
    s = _spec(name)
    lanes = upf.field_eval_grid(s, g, variant=upf.EVAL_PER_LANE)
    assert torch.isfinite(lanes).all()
    assert torch.equal(upf.field_eval_grid(s, g), lanes)
