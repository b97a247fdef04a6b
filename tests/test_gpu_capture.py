"""Single-volume calls captured in a HIP graph: every replay gives what an eager
call gives, with new data, with eager calls of other sizes on the same stream's
scratch area in between, small volumes (one workgroup per tile) and persistent
kernels alike."""
import numpy as np
import pytest

from lsc_helpers import MODES, synth

pytestmark = pytest.mark.gpu

# 1, 64, 128 and 189 tiles of 64 to 512 blocks; 257 tiles compress on the persistent
# kernel, 705 decompress on it
SHAPES = [(1, 8, 60), (1, 512, 512), (4, 512, 510), (3, 1000, 1030), (1, 8, 8 * 131073), (1, 8, 8 * 360449)]


def _np16(t):
    return t.cpu().numpy().view(np.uint16)


@pytest.mark.parametrize("entry", ["async", "noalloc"])
@pytest.mark.parametrize("shape", SHAPES, ids=lambda s: "x".join(map(str, s)))
def test_replays(gpu, orc, shape, entry):
    import torch
    bins, p = MODES["lossless"]
    s = torch.cuda.Stream()
    compress = gpu.compress_async if entry == "async" else gpu.compress_noalloc_async
    vols = [synth(kind, shape, seed=40 + i) for i, kind in enumerate(("sparse", "mixed", "sparse"))]
    refs = [orc.compress(v, bins, p)[1] for v in vols]
    d = torch.zeros(shape, dtype=torch.int16, device="cuda")
    back = torch.zeros_like(d)
    out = torch.zeros(gpu.max_compressed_bytes(shape), dtype=torch.uint8, device="cuda")
    size = torch.zeros(1, dtype=torch.int64, device="cuda")
    other = torch.from_numpy(synth("sparse", (2, 700, 900), seed=9).view(np.int16)).cuda()
    _, other_ref, _ = orc.compress(other.cpu().numpy().view(np.uint16), bins, p)
    cap = refs[0].size   # the decode's stream length is fixed in the graph: that of the first volume
    stream0 = torch.from_numpy(refs[0]).cuda()
    torch.cuda.synchronize()
    with torch.cuda.stream(s):   # scratch outside the capture
        compress(d, shape, bins, p, out, size)
        gpu.decompress_async(stream0, cap, shape, bins, back)
    assert gpu.stream_status(s) == gpu.OK
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g, stream=s):
        compress(d, shape, bins, p, out, size)
        gpu.decompress_async(stream0, cap, shape, bins, back)
    for i in (0, 1, 2, 0, 1):
        d.copy_(torch.from_numpy(vols[i].view(np.int16)))
        out.fill_(0x77)
        size.zero_()
        back.fill_(0x55)
        s.wait_stream(torch.cuda.current_stream())
        with torch.cuda.stream(s):
            g.replay()
        assert gpu.stream_status(s) == gpu.OK
        n = int(size.item())
        assert n == refs[i].size and np.array_equal(out[:n].cpu().numpy(), refs[i])
        assert np.array_equal(_np16(back), vols[0])
        with torch.cuda.stream(s):   # an eager call in between
            o, m = gpu.compress(other, other.shape, bins, p)
        assert m == other_ref.size and np.array_equal(o[:m].cpu().numpy(), other_ref)
