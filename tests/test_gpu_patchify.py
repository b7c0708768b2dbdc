"""Patch extraction of bf16 and fp32 latents against tensor reshapes (exact)."""
import pytest
import torch

pytestmark = pytest.mark.gpu

if torch.cuda.is_available():
    from ditserve_amd import ops


@pytest.mark.parametrize("c,f,h,w,patch", [(16, 9, 60, 104, (1, 2, 2)), (48, 1, 2, 2, (1, 2, 2)), (3, 2, 6, 10, (1, 2, 2)),
                                           (16, 1, 34, 66, (1, 2, 2)), (4, 4, 6, 9, (2, 2, 3)), (5, 3, 4, 4, (1, 1, 1))])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_patchify_matches_reshapes(c, f, h, w, patch, dtype):
    g = torch.Generator(device="cuda").manual_seed(c + h)
    full = torch.randn((c, f, h, w + 2), generator=g, device="cuda").to(dtype)
    full[0, 0, 0, :4] = torch.tensor([float("inf"), -0.0, 3.4e38, 1e-40], dtype=dtype, device="cuda")
    pt, ph, pw = patch
    for lat in (full[..., :w], full[..., :w].contiguous()):
        want = lat.to(torch.bfloat16).reshape(c, f // pt, pt, h // ph, ph, w // pw, pw).permute(1, 3, 5, 0, 2, 4, 6)
        got = (ops.patchify_f32 if dtype == torch.float32 else ops.patchify)(lat, patch)
        assert torch.equal(got.view(torch.int16), want.reshape(got.shape).view(torch.int16))
