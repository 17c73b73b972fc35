"""upf_images_post (dilation and U8 conversion in one pass) against the oracle's dilation and
conversion, byte for byte: sizes at the edges of its tiles and of its vector rows, images
without a NaN, with nothing but NaN, with one valid texel, and mixed ones."""
import numpy as np
import pytest

import unnatural_planets_amd as upfm

pytestmark = pytest.mark.gpu


def _image(w, h, c, kind, seed):
    rng = np.random.default_rng(seed)
    a = rng.uniform(-0.2, 1.2, (h, w, c)).astype(np.float32)
    if kind == "nan":
        a[:] = np.nan
    elif kind == "one":
        keep = a[h // 2, w // 2].copy()
        a[:] = np.nan
        a[h // 2, w // 2] = keep
    elif kind == "mixed":
        a[rng.random((h, w)) < 0.7] = np.nan
        a[: h // 3, : w // 3] = rng.uniform(0, 1, c).astype(np.float32)  # a covered corner
        a[rng.random((h, w)) < 0.01, c - 1] = np.nan  # a NaN past the first channel does not count
    return a


def _want(oracle, a, rounds):
    return oracle.image_to_u8(oracle.image_dilate(a.copy(), rounds))


@pytest.mark.parametrize("w,h", [(1, 1), (31, 33), (32, 32), (40, 64), (97, 65), (132, 70)])
@pytest.mark.parametrize("kind", ["full", "nan", "one", "mixed"])
@pytest.mark.parametrize("rounds", [0, 1, 7])
def test_channels_against_oracle(upf, oracle, w, h, kind, rounds):
    import torch
    images = [_image(w, h, c, kind, 10 * w + c) for c in (1, 2, 3, 4)]
    dev = [torch.from_numpy(a).cuda() for a in images]
    before = [d.clone() for d in dev]
    got = upfm._images_post(dev[:3], (None,) * 3, rounds, None) + upfm._images_post(dev[3:], (None,), rounds, None)
    for a, d, b, g in zip(images, dev, before, got):
        np.testing.assert_array_equal(g.cpu().numpy(), _want(oracle, a, rounds))
        assert torch.equal(d.view(torch.int32), b.view(torch.int32))  # the input is not written


@pytest.mark.parametrize("w,h", [(40, 33), (37, 41)])
def test_zero_channels_and_unaligned_rows(upf, oracle, w, h):
    import torch
    a = _image(w, h, 1, "mixed", 3)
    want = _want(oracle, np.concatenate([a, np.where(np.isnan(a), a, 0)], 2).astype(np.float32), 5)
    flat = torch.empty(w * h + 1, device="cuda")
    for off in (0, 1):  # off 1: neither the reads nor the writes are aligned
        d = flat[off:off + w * h].view(h, w)
        d.copy_(torch.from_numpy(a[:, :, 0]))
        np.testing.assert_array_equal(upfm._images_post((d,), (2,), 5, None)[0].cpu().numpy(), want)


@pytest.mark.parametrize("rounds", [0, 7, 9])
def test_texture_post_is_its_steps(upf, rounds):
    import torch
    w, h = 150, 70
    albedo, rough, bump = (torch.from_numpy(_image(w, h, c, "mixed", 5)).cuda() for c in (3, 1, 1))
    tex = upfm.Textures(albedo, bump[:, :, 0].contiguous(), rough[:, :, 0].contiguous(), None, None)
    special = torch.stack([tex.roughness, torch.where(torch.isnan(tex.roughness), tex.roughness, 0 * tex.bump.nan_to_num())], 2)
    want = [upfm.image_to_u8(upfm.image_dilate(i.clone().contiguous(), rounds)) for i in (albedo, special, tex.bump)]
    for got in (upfm.texture_post(tex, rounds), upfm.texture_post_images(albedo, special, tex.bump, rounds)):
        for g, x in zip(got, want):
            assert torch.equal(g, x)
