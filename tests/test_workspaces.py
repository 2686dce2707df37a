"""Workspaces kept between calls: calls on several streams and threads that
share them return what they return alone (the same kernels: the same bits),
and what waits for the next call stays within its bound of 4 GiB."""
import threading

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def test_threads_and_streams_share_workspaces():
    import torch

    from tom_amd import api
    dev = torch.device("cuda:0")
    n = 16
    rng = np.random.default_rng(1)
    T = torch.from_numpy(rng.standard_normal((n, n, n)).astype(np.float32)).to(dev)
    M = torch.ones((n, n, n), device=dev)
    V = [torch.from_numpy(rng.standard_normal((64, 64, 64)).astype(np.float32)).to(dev) for _ in range(2)]
    torch.cuda.synchronize()
    ref = [api.tom_os3_corr(v, T, M).clone() for v in V]
    torch.cuda.synchronize()
    bad = []

    def work(k):
        ctx = api.Context(0)
        try:
            with torch.cuda.stream(torch.cuda.Stream(device=dev)):
                for i in range(6):
                    out = api.tom_os3_corr(V[(k + i) % 2], T, M, ctx=ctx)
                    if not torch.equal(out, ref[(k + i) % 2]):
                        bad.append((k, i))
        except Exception as e:  # reported by the main thread
            bad.append((k, repr(e)))
        finally:
            ctx.close()

    ts = [threading.Thread(target=work, args=(k,)) for k in range(3)]
    for t in ts:
        t.start()
    for t in ts:
        t.join()
    assert not bad


def test_kept_workspaces_are_bounded():
    import torch

    from tom_amd import api
    dev = torch.device("cuda:0")
    T = torch.randn((16, 16, 16), device=dev)
    M = torch.ones((16, 16, 16), device=dev)
    vols = [torch.randn(s, device=dev) for s in ((128, 256, 256), (192, 256, 256), (256, 256, 384), (64, 512, 512))]
    torch.cuda.synchronize()
    torch.cuda.empty_cache()
    free0 = torch.cuda.mem_get_info()[0]
    for v in vols + vols:
        del_me = api.tom_os3_corr(v, T, M)
        del del_me
    torch.cuda.synchronize()
    torch.cuda.empty_cache()
    # the pool's bound, and room for what the driver rounds
    assert free0 - torch.cuda.mem_get_info()[0] < (4 << 30) + (512 << 20)
