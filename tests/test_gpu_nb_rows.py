"""The narrow band's sign masks and records of brick rows, on fields that cross nearly every
edge (rows full of vertices, cells of up to five triangles) and on grids of one block, of one
block along an axis and of several: the dense mesh, vertex for vertex."""
import numpy as np
import pytest

from test_gpu_nb import canonical, canon_tris
from unnatural_planets_amd import spec as S

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dims", [(9, 9, 9), (25, 9, 9), (9, 17, 9), (9, 9, 33), (41, 33, 25)])
@pytest.mark.parametrize("noise,freq", [("value", 0.9), ("simplex", 0.4), ("gradient", 0.23), ("modes", 0.0)])
@pytest.mark.parametrize("iso", [0.0, 0.1])
def test_rows_against_dense(upf, dims, noise, freq, iso):
    g = S.Grid()
    for a in range(3):
        g.dims[a], g.spacing[a], g.origin[a] = dims[a], 1.0, (-7.0, 3.0, 11.0)[a]
    if noise == "modes":
        for a in range(3):
            g.spacing[a], g.origin[a] = 2600.0 / max(dims), -1300.0 * dims[a] / max(dims)
        s = S.spec_elevation_mode("lakes", 2, "sphere", (900.0,))
    else:
        s = S.field_spec("none", (), [S.layer(noise, "none", 1, freq, weight=1.0, seed=5)], "elevation_raw")
    mesh, keys, st = upf.nb_extract(s, g, 1e9, iso=iso, keys=True)
    dense = upf.mc_extract(upf.field_eval_grid(s, g), g, iso)
    assert st.active_blocks == st.blocks and st.unresolved == 0 and mesh.n_triangles > 0
    _, pos, _, tri = canonical(keys.cpu().numpy(), mesh.positions.cpu().numpy(), None, mesh.indices.cpu().numpy().astype(np.int64))
    np.testing.assert_array_equal(pos, dense.positions.cpu().numpy())
    np.testing.assert_array_equal(tri, canon_tris(dense.indices.cpu().numpy().astype(np.int64)))
