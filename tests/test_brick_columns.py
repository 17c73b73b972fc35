"""The narrow band's bricks keep a layer's lattice columns in LDS where a bound says that they
fit (brick_columns_fit).  The bound itself against the count of columns, in a sanitized host
build of the function (built by build(), tests/sanitize/Makefile); and, far from the origin,
where the coordinates' rounding moves whole lattice cells, a narrow-band mesh against the
dense one."""
import os
import subprocess

import numpy as np
import pytest

from test_gpu_nb import canon_tris, canonical
from unnatural_planets_amd import spec as S

EXE = os.path.join(os.path.dirname(os.path.abspath(__file__)), "sanitize", "_build", "brick_check")


def test_bound_covers_the_count():
    assert os.path.exists(EXE), "run build() (make -C tests/sanitize)"
    r = subprocess.run([EXE], capture_output=True, text=True, timeout=300)
    assert r.returncode == 0 and "brick_check: ok" in r.stdout, r.stdout + r.stderr


# cells a node on both sides of the limit (24 columns a row of 9 nodes), and origins at which
# one ulp of a coordinate is 2^-21, 1/8, and 1 to 4 nodes
@pytest.mark.gpu
@pytest.mark.parametrize("nodes", [2.0 ** 3, 2.0 ** 21, 2.0 ** 24.5, 2.0 ** 26])
@pytest.mark.parametrize("octaves,cells", [(1, 2.4), (1, 2.9), (4, 0.12), (4, 0.3)])
@pytest.mark.parametrize("noise", ["gradient", "value"])
def test_far_origins_against_dense(upf, noise, octaves, cells, nodes):
    g = S.Grid()
    for a in range(3):
        g.dims[a], g.spacing[a], g.origin[a] = (41, 17, 25)[a], 0.2023, (0.2023 * nodes if a == 0 else 1.5 * a)
    s = S.field_spec("none", (), [S.layer(noise, "fbm", octaves, cells / 0.2023, weight=1.0, seed=5)], "elevation_raw")
    iso = 0.01
    mesh, keys, st = upf.nb_extract(s, g, 1e9, iso=iso, keys=True, normals=False)
    assert st.active_blocks == st.blocks and st.unresolved == 0 and mesh.n_triangles > 0
    _, pos, _, tri = canonical(keys.cpu().numpy(), mesh.positions.cpu().numpy(), None, mesh.indices.cpu().numpy().astype(np.int64))
    # a brick takes its values from columns or, where they do not fit, per lane: each vertex is
    # the one of the dense mesh of either form, whose sums round apart by a few ulps
    same = np.zeros(len(pos), bool)
    for variant in (upf.EVAL_ROWS, upf.EVAL_PER_LANE):
        dense = upf.mc_extract(upf.field_eval_grid(s, g, variant=variant), g, iso)
        np.testing.assert_array_equal(tri, canon_tris(dense.indices.cpu().numpy().astype(np.int64)))
        same |= (pos == dense.positions.cpu().numpy()).all(axis=1)
    assert same.all()
