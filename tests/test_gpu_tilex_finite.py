"""The lakes and islands modes with layers that overflow: the masks that are 0 do not hide an
infinite or undefined layer, the field is the per-lane form's bit for bit, NaN included."""
import pytest

from unnatural_planets_amd import spec as S

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [40, 132])
@pytest.mark.parametrize("mode", ["lakes", "islands"])
@pytest.mark.parametrize("layer", [1, 2, 3])
@pytest.mark.parametrize("what", ["amplitude", "frequency", "jitter"])
def test_overflowing_layers(upf, what, layer, mode, n):
    import torch
    s, g = S.spec_elevation_mode(mode, 5, "torus", (1200.0, 450.0)), S.uniform_grid(-2000.0, 2000.0, n)
    L = s.layers[layer]
    if what == "amplitude":
        L.fractal, L.octaves = S.FRACTAL["fbm"], 2
        L.amp[0] = L.amp[1] = 3e38
        L.freq[1] = 2 * L.freq[0]
    elif what == "frequency":
        L.freq[0] = 3e38
    else:
        L.noise, L.jitter = S.NOISE["cellular"], 3e38
    lanes = upf.field_eval_grid(s, g, variant=upf.EVAL_PER_LANE)
    assert torch.equal(upf.field_eval_grid(s, g).view(torch.int32), lanes.view(torch.int32))
