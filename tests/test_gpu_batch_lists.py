"""A batch whose chunks run as row pairs, in bands of eight rows and in bands of four (cellular
layers over many cells, rows of cells far apart), mixed and of ragged sizes: each chunk as its
own grid, in either order, with the field form switched after the batch is made, and replayed
from a captured graph."""
import pytest

from unnatural_planets_amd import spec as S

pytestmark = pytest.mark.gpu

# (dims, spacing along x and z, along y, layers)
CHUNKS = [((128, 64, 520), 8.0, 8.0, "plain"), ((70, 31, 90), 8.0, 8.0, "wide"), ((9, 7, 5), 8.0, 8.0, "wide"), ((65, 6, 40), 8.0, 8.0, "wide"),
          ((3, 9, 130), 1.0, 300.0, "near"), ((130, 4, 70), 8.0, 8.0, "wide"), ((2, 2, 2), 8.0, 8.0, "plain"), ((129, 13, 33), 8.0, 100.0, "wide"),
          ((64, 37, 21), 0.5, 0.5, "near"), ((33, 65, 2), 8.0, 8.0, "simplex"), ((5, 5, 5), 8.0, 8.0, "plain")]


def _layers(kind):
    if kind == "wide":
        return [S.layer("gradient", "fbm", 3, 0.004, weight=40.0, seed=3), S.layer("cellular", "fbm", 2, 0.012, weight=30.0, seed=9)]
    if kind == "near":
        return [S.layer("value", "fbm", 2, 0.004, weight=40.0, seed=3), S.layer("cellular", "none", 1, 0.006, weight=30.0, seed=9)]
    if kind == "simplex":
        return [S.layer("simplex", "fbm", 3, 0.004, weight=40.0, seed=3)]
    return [S.layer("gradient", "ridged", 5, 0.002, weight=60.0, seed=7)]


@pytest.mark.parametrize("order", [1, -1])
@pytest.mark.parametrize("variants", [("rows", "lanes"), ("lanes", "rows")])
def test_chunks_of_every_list(upf, order, variants):
    import torch
    from unnatural_planets_amd.batch import Batch
    form = {"rows": upf.EVAL_ROWS, "lanes": upf.EVAL_PER_LANE}
    chunks = (S.Chunk * len(CHUNKS))()
    for c, (dims, sx, sy, kind) in zip(chunks, CHUNKS[::order]):
        c.spec, c.iso = S.field_spec("torus", (1200.0, 450.0), _layers(kind), "land", 0.1), 900.0
        for a in range(3):
            c.grid.dims[a], c.grid.spacing[a] = dims[a], (sx, sy, sx)[a]
            c.grid.origin[a] = -round(0.5 * dims[a]) * c.grid.spacing[a] + (11.0, -896.0, 256.0)[a]
    b = Batch(chunks, S.BatchOpts(form[variants[0]], 0, 0, 0))
    b.size_outputs(1.05)  # the forms differ by ulps
    side = torch.cuda.Stream()
    for v in variants:
        b.set_opts(S.BatchOpts(form[v], 0, 0, 0))
        want = [upf.field_eval_grid(c.spec, c.grid, variant=form[v]) for c in chunks]
        b.run()
        table = b.mesh_table()
        for i, c in enumerate(chunks):
            assert torch.equal(b.field_of(i), want[i]), CHUNKS[::order][i]
            m, bm = upf.mc_extract(want[i], c.grid, 900.0), b.mesh_of(i, table)
            assert torch.equal(bm.indices, m.indices) and torch.equal(bm.positions, m.positions), CHUNKS[::order][i]
        torch.cuda.synchronize()
        b.capture(side)
        for _ in range(3):
            b.field.zero_()
            torch.cuda.synchronize()
            b.replay(side)
            torch.cuda.synchronize()
            for i in range(len(chunks)):
                assert torch.equal(b.field_of(i), want[i]), CHUNKS[::order][i]
