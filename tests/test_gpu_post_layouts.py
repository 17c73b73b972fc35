"""texture_post over the layouts of its images: a roughness of any strides (the special map is made
from it), an albedo or bump with gaps (copied); a dense transposed albedo or bump is refused."""
import pytest

import unnatural_planets_amd as upfm

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("rounds", [0, 7, 9])
@pytest.mark.parametrize("layout", ["transposed", "gaps", "expanded", "every second row"])
def test_roughness_of_any_strides(upf, layout, rounds):
    import torch
    gen = torch.Generator("cuda").manual_seed(1)
    h, w = 45, 61
    base = torch.rand((w, h), device="cuda", generator=gen)
    base[torch.rand((w, h), device="cuda", generator=gen) < 0.4] = float("nan")
    rough = {"transposed": base.t(), "gaps": base.repeat(2, 2)[:h, :w], "expanded": base[:w, :1].t().expand(h, w),
             "every second row": torch.cat([base.t(), base.t()], 1).reshape(2 * h, w)[::2]}[layout]
    assert tuple(rough.shape) == (h, w)
    albedo, bump = torch.rand((h, w, 3), device="cuda", generator=gen), torch.rand((h, w), device="cuda", generator=gen)
    got = upfm.texture_post(upfm.Textures(albedo, bump, rough, None, None), rounds)
    want = upfm.texture_post(upfm.Textures(albedo, bump, rough.contiguous(), None, None), rounds)
    special = torch.stack([rough, torch.where(torch.isnan(rough), rough, torch.zeros_like(rough))], 2).contiguous()
    steps = upfm.image_to_u8(upfm.image_dilate(special, rounds))
    for g, x in zip(got, want):
        assert torch.equal(g, x)
    assert torch.equal(got[1], steps)


def test_albedo_and_bump(upf):
    import torch
    h, w = 45, 61
    rough = torch.rand((h, w), device="cuda")
    albedo, bump = torch.rand((h, w, 4), device="cuda")[..., :3], torch.rand((h, 2 * w), device="cuda")[:, ::2][:, :w]
    got = upfm.texture_post(upfm.Textures(albedo, bump, rough, None, None))
    want = upfm.texture_post(upfm.Textures(albedo.contiguous(), bump.contiguous(), rough, None, None))
    for g, x in zip(got, want):
        assert torch.equal(g, x)
    for a, b in ((torch.rand((w, h, 3), device="cuda").transpose(0, 1), bump), (albedo, torch.rand((w, h), device="cuda").t())):
        with pytest.raises(ValueError):
            upfm.texture_post(upfm.Textures(a, b, rough, None, None))
