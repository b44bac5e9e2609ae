"""The convolution that cuts its channels between work-groups (few images, many channels), against float64: strips and whole images per
work-group, parts of different lengths, channels out and planes of no whole tiles or vectors, with and without bias.

fp32 sums of n terms, in parts and then added: the error of a result is below n eps sum|x w|, and near sqrt(n) eps of the
result's size for random operands; 1e-5 of the largest result holds a factor of ten for n = 9 x 512."""
import os

import pytest
import torch
import torch.nn.functional as F

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("N,C,OC,H,W,k,stride,pad,bias", [
    (1, 256, 256, 14, 14, 3, 1, 1, True),      # strips of one image
    (1, 16, 65, 9, 9, 3, 1, 1, False),         # two chunks: too few to cut
    (1, 72, 70, 13, 11, 3, 1, 0, True),        # nine chunks, a ragged last tile of channels, planes of 99 pixels
    (3, 512, 64, 7, 7, 3, 1, 1, True),         # several images per work-group, one of them missing
    (2, 136, 33, 15, 17, 3, 2, 1, True),       # steps of two, a result of no whole vectors
    (1, 512, 96, 9, 9, 1, 2, 0, True),         # 1x1 with steps of two
    (1, 320, 48, 40, 40, 3, 1, 1, False),
])
def test_channels_in_parts(rt, monkeypatch, N, C, OC, H, W, k, stride, pad, bias):
    g = torch.Generator().manual_seed(C + OC)
    x, w = torch.randn(N, C, H, W, generator=g), torch.randn(OC, C, k, k, generator=g) * (C * k * k) ** -0.5
    b = torch.randn(OC, generator=g) if bias else None
    ref = F.conv2d(x.double(), w.double(), b.double() if bias else None, stride=stride, padding=pad)
    dx, dw, db = x.cuda(), w.cuda(), b.cuda() if bias else None
    y = torch.full(ref.shape, float("nan"), device="cuda")
    for choice in (None, None, "direct"):       # the last: the strips where the choice is Winograd's form
        if choice and not os.environ.get("DOCC_ROCM_CONV"):
            monkeypatch.setenv("DOCC_ROCM_CONV", choice)
        rt.conv2d_f32(N, C, H, W, OC, k, k, (stride, stride), (pad, pad), (1, 1), dx.data_ptr(), dw.data_ptr(), db.data_ptr() if bias else 0, y.data_ptr())
        torch.cuda.synchronize()
        assert (y.cpu().double() - ref).abs().max() <= 1e-5 * ref.abs().max()


# the form and the number of parts given: as few chunks as can be cut, parts of different lengths, both strip sizes, whole images
# (tests/test_launcher_memory.py holds the launchers to the kernels' names)
@pytest.mark.parametrize("form", ["t4-parts2", "t2-parts2", "t4m-parts2", "t2m-parts2", "t4-parts3", "t2-parts4", "t4m-parts3", "t2m-parts4"])
@pytest.mark.parametrize("k,stride,pad", [(3, 1, 1), (3, 2, 1), (1, 2, 0)])
def test_forms_in_parts(rt, monkeypatch, form, k, stride, pad):
    monkeypatch.setenv("DOCC_ROCM_CONV", "halo-" + form)
    for C, N in ((32 if "2" in form[-1] else 72, 3), (72, 5)):
        test_channels_in_parts(rt, monkeypatch, N, C, 70, 9, 7, k, stride, pad, True)
