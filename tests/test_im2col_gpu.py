"""Windows of a 3x3 convolution side by side: image borders, 16-byte pixels, both tap orders; and the convolutions made of them."""
import pytest
import torch
import torch.nn.functional as F

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16, torch.float32])
@pytest.mark.parametrize("B,H,W,C", [(1, 1, 1, 8), (2, 1, 5, 16), (3, 7, 1, 24), (2, 13, 11, 8), (1, 64, 63, 72)])
def test_im2col3x3(B, H, W, C, dtype):
    from pfeife_amd.hip import HipKernels

    hip = HipKernels(0)
    src = torch.randn(B, H, W, C, generator=torch.Generator().manual_seed(C)).to(dtype).cuda()
    pad = F.pad(src, (0, 0, 1, 1, 1, 1))
    for flip in (0, 1):
        whole = torch.full((B * H * W * 9 * C + 64,), 7.0, dtype=dtype, device="cuda")
        dst = whole[:-64].view(B, H, W, 9, C)
        hip.run("im2col3x3", src, dst, B, H, W, C, flip)
        torch.cuda.synchronize()
        for t in range(9):
            i, j = (2 - t // 3, 2 - t % 3) if flip else (t // 3, t % 3)
            assert torch.equal(dst[:, :, :, t], pad[:, i:i + H, j:j + W])
        assert (whole[-64:] == 7).all()


def test_im2col_refuses():
    from pfeife_amd.hip import HipKernels

    hip = HipKernels(0)
    t, out = torch.zeros(1, 4, 4, 12, dtype=torch.float16, device="cuda"), torch.zeros(1, 4, 4, 9, 12, dtype=torch.float16, device="cuda")
    with pytest.raises(RuntimeError, match="16-byte"):
        hip.run("im2col3x3", t, out, 1, 4, 4, 12)
    u = torch.zeros(1 * 4 * 4 * 16 + 8, dtype=torch.float16, device="cuda")[4:-4]
    with pytest.raises(RuntimeError, match="16-byte"):
        hip.run("im2col3x3", u, out, 1, 4, 4, 16)
