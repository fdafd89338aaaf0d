"""fp32 3x3 layers in tiles of 32 consecutive pixels (conv3x3_split.hip): tiles that end inside a row, an image, the batch; several images a
tile; one image of exactly a tile; six slabs, the fewest, and many; the widest rows; against torch in 64 bits, and what is not finite."""
import numpy as np
import pytest
import torch

from test_gpu_conv3x3_split import layer_and_reference

pytestmark = pytest.mark.gpu

CASES = [(6, 512, 512, 8, 10, "flat"), (7, 512, 512, 8, 9, "flat"), (9, 512, 512, 7, 8, "flat"), (20, 448, 448, 5, 5, "flat"),
         (12, 512, 512, 4, 8, "flat"), (16, 512, 512, 4, 7, "flat"), (3, 448, 512, 10, 16, "flat"), (55, 512, 512, 3, 3, "flat"), (4, 512, 512, 5, 24, "flat"),
         (64, 192, 256, 8, 2, "flat"), (3, 192, 512, 7, 24, "flat"), (24, 192, 64, 10, 17, "flat"), (1, 256, 512, 22, 23, "flat"), (12, 256, 512, 14, 3, "flat"), (16, 256, 512, 32, 1, "flat")]


@pytest.mark.parametrize("case", CASES, ids=lambda c: "x".join(map(str, c[:5])))
def test_matches_double(case):
    got, want, tags = layer_and_reference(case, 1)
    assert tags == ["conv3x3_split<f32,flat>"], tags
    err = ((got.double() - want).norm() / want.norm()).item()
    # 9 C / 16 additions of half an ulp at most in a row, as a random walk, and a few ulp at the end
    assert err < 2.0 ** -25 * (9 * case[1] / 48) ** 0.5 + 2.0 ** -24, err
    assert ((got.double() - want).abs().amax((0, 2, 3)) < 1e-4 * want.abs().amax()).all()


def test_values_that_bf16_does_not_hold():
    N, C, F, H, W, _ = case = CASES[0]

    def spoil(x, w):
        x[0, 3, 4, 5] = float("inf")
        x[1, 0, 0, 0] = float("nan")
        x[2, C - 1, H - 1, W - 1] = 3.4e38  # rounds to infinity in bf16
        w[5] *= 1e-3

    got, want, tags = layer_and_reference(case, 2, spoil)
    assert tags == ["conv3x3_split<f32,flat>"], tags
    want32 = want.float()
    fin = torch.isfinite(want32)
    assert torch.equal(torch.isnan(got), torch.isnan(want32))
    assert torch.equal(got[torch.isinf(want32)], want32[torch.isinf(want32)])
    large = fin & (want.abs() > 1e6)
    assert large.any() and ((got[large].double() - want[large]).abs() <= 1e-5 * want[large].abs()).all()
    rest = fin & ~large
    assert ((got[rest].double() - want[rest]).norm() / want[rest].norm()).item() < 1e-6
