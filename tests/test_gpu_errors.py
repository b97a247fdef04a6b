"""Errors that a launch leaves for a later call: each is reported once, by the
first status or blocking call after it, and no later call is blamed for it."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

LOSSLESS = ((1, 1, 1, 1), 1.0)


# one workgroup per tile, and the persistent kernel (257 tiles of 256 blocks)
@pytest.mark.parametrize("shape", [(2, 60, 70), (1, 2048, 2056)], ids=["small", "persistent"])
def test_replayed_u32_range_error(gpu, orc, shape):
    """A captured uint32 compression runs without its host call: a value of 2^31
    met by a replay is reported after that replay, not after a good one."""
    import torch
    rng = np.random.default_rng(8)
    vol = rng.poisson(0.4, shape).astype(np.uint32) << 9
    st, ref, refn = orc.compress_u32(vol, *LOSSLESS)
    assert st == 0
    d = torch.from_numpy(vol.view(np.int32)).cuda()
    out = torch.zeros(gpu.max_compressed_bytes_u32(shape), dtype=torch.uint8, device="cuda")
    size = torch.zeros(1, dtype=torch.int64, device="cuda")
    s = torch.cuda.Stream()
    s.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(s):
        gpu.compress_u32_async(d, shape, *LOSSLESS, out, size)   # scratch outside the capture
    assert gpu.stream_status(s) == gpu.OK
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g, stream=s):
        gpu.compress_u32_async(d, shape, *LOSSLESS, out, size)
    last = d.view(-1)[-1:]
    good = last.clone()
    for bad in (False, False, True, False, True, True, False):
        last.copy_(torch.full_like(last, -(1 << 31)) if bad else good)
        out.zero_()
        size.zero_()
        s.wait_stream(torch.cuda.current_stream())
        with torch.cuda.stream(s):
            g.replay()
        assert gpu.stream_status(s) == (gpu.ERR_RANGE if bad else gpu.OK)
        if not bad:
            assert int(size.item()) == refn and np.array_equal(out[:refn].cpu().numpy(), ref)
    # a good blocking call right after an unread bad replay gets that error, the next one none
    last.copy_(torch.full_like(last, -(1 << 31)))
    s.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(s):
        g.replay()
    s.synchronize()
    last.copy_(good)
    s.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(s):
        with pytest.raises(gpu.LscompError) as e:
            gpu.compress_u32(d, shape, *LOSSLESS, out=out)
        assert e.value.status == gpu.ERR_RANGE
        _, n = gpu.compress_u32(d, shape, *LOSSLESS, out=out)
    assert n == refn and np.array_equal(out[:n].cpu().numpy(), ref)
