"""The material stack's shared lattices (slots, boxes, per lane) give the oracle's tiles:
points from one lattice cell to the whole planet, waves that are not full, textures whose
sides are not multiples of a wave's 8 x 8 texels.  Bar: bit for bit, as for every tile."""
import numpy as np
import pytest

import unnatural_planets_amd as upfm
from unnatural_planets_amd import spec as S

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 63, 64, 65, 700])
@pytest.mark.parametrize("spread", [0.0, 0.5, 4.0, 15.0, 60.0, 900.0])
@pytest.mark.parametrize("purpose", ["land", "water"])
def test_tiles_at_every_spread(upf, oracle, n, spread, purpose):
    import torch
    rng = np.random.default_rng(n + int(10 * spread))
    m = S.material_spec(S.spec_elevation_mode("islands", 4), "default", purpose, seed=33)
    d = rng.standard_normal(3)
    centre = 1100.0 * d / np.linalg.norm(d)
    pos = (centre + spread * rng.uniform(-1, 1, (n, 3))).astype(np.float32)
    nrm = (pos / np.linalg.norm(pos, axis=1, keepdims=True)).astype(np.float32)
    got = upf.material_tiles(m, torch.from_numpy(pos).cuda(), torch.from_numpy(nrm).cuda()).cpu().numpy()
    ref = oracle.material_tiles(m, pos, nrm)
    np.testing.assert_array_equal(got[:, :13].view(np.int32), ref[:, :13].view(np.int32))


@pytest.mark.parametrize("shape", ["box", "gear"])  # a primitive, one of the further shapes
@pytest.mark.parametrize("w,h", [(97, 151), (250, 129)])
def test_bake_of_ragged_sides(upf, oracle, shape, w, h):
    params = {"box": (700.0, 700.0, 700.0, 200.0), "gear": ()}[shape]
    f = S.spec_elevation_mode("lakes", 9, shape, params)
    mesh = upfm.mesh_generate_generic(f, S.grid_reference(24))
    m = S.material_spec(f, "default", "land", seed=3)
    uv = upfm.atlas_per_triangle(mesh.n_triangles, w, h)
    tri = upfm.bake_rasterize(uv, w, h)
    tri[0, :5] = -1
    out = upfm.bake_material(m, mesh, uv, tri)
    ref = oracle.bake_material(m, mesh.positions.cpu().numpy(), mesh.normals.cpu().numpy(), mesh.indices.cpu().numpy(),
                               uv.cpu().numpy(), tri.cpu().numpy())
    for x, y in zip(out, ref):
        x = x.cpu().numpy()
        nan = np.isnan(y)
        assert 0 < nan.sum() < nan.size
        np.testing.assert_array_equal(np.isnan(x), nan)
        np.testing.assert_array_equal(x[~nan].view(np.int32), y[~nan].view(np.int32))
