"""Workspaces kept between calls go back when a program asks for them."""
import pytest

pytestmark = pytest.mark.gpu


def test_release_frees_what_waits():
    import torch

    from tom_amd import api
    dev = torch.device("cuda:0")
    g = torch.Generator(device=dev)
    g.manual_seed(2)
    V = torch.randn((128, 256, 256), generator=g, device=dev)
    T = torch.randn((16, 16, 16), generator=g, device=dev)
    M = torch.ones((16, 16, 16), device=dev)
    ref = api.tom_os3_corr(V, T, M)
    torch.cuda.synchronize()
    ctx = api.context()
    held = torch.cuda.mem_get_info()[0]
    ctx.release_workspaces()
    # two FP64 spectra of the volume at the least
    assert torch.cuda.mem_get_info()[0] - held > 2 * 16 * V.numel()
    assert torch.equal(api.tom_os3_corr(V, T, M), ref)
