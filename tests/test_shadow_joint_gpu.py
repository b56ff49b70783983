"""Transposed shadows of several weight matrices side by side, and the refresh of joint and single ones in one launch."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_transposed_shadows_side_by_side(dtype):
    from pfeife_amd.executor.lowering import ParamStore
    from pfeife_amd.hip import HipKernels

    hip = HipKernels(0)
    store = ParamStore(hip, torch.device("cuda", 0))
    g = torch.Generator().manual_seed(3)
    for sizes, cols in (((8, 72, 64), 40), ((128, 128, 136), 200), ((64,), 64), ((1000, 24), 8)):
        ws = [torch.randn(n, cols, generator=g).cuda() for n in sizes]
        joint = store.shadow_joint(ws, dtype)
        joint_t = store.shadow_joint_t(ws, dtype)
        own = store.shadow_t(ws[0], dtype)          # one of them alone as well
        joint.fill_(7), joint_t.fill_(7), own.fill_(7)
        assert store.shadow(ws[-1], dtype).data_ptr() == joint[-sizes[-1]:].data_ptr()
        for launch in store.refresh_launches():
            launch(torch.cuda.current_stream().cuda_stream)
        torch.cuda.synchronize()
        want = torch.cat(ws).to(dtype)
        assert torch.equal(joint, want) and torch.equal(joint_t, want.t()) and torch.equal(own, ws[0].to(dtype).t())


def test_transposed_fp32_copies():
    """fp32 weights' transposed copies, all in one launch; one whose size does not allow 16-byte accesses on its own."""
    from pfeife_amd.executor.lowering import ParamStore
    from pfeife_amd.hip import HipKernels

    hip = HipKernels(0)
    store = ParamStore(hip, torch.device("cuda", 0))
    g = torch.Generator().manual_seed(3)
    ws = [torch.randn(*s, generator=g).cuda() for s in ((4, 4), (64, 64), (68, 132), (1536, 384), (384, 1152), (12, 2000), (30, 10))]
    copies = [store.shadow_t(w, torch.float32) for w in ws]
    launches = store.refresh_launches()
    assert len(launches) == 2
    for launch in launches:
        launch(torch.cuda.current_stream().cuda_stream)
    torch.cuda.synchronize()
    for w, c in zip(ws, copies):
        assert torch.equal(c, w.t())
