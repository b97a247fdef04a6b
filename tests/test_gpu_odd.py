"""Volumes whose rows are only 2-byte aligned, above the sizes of the small-volume
kernels, and decodes above them at every stream alignment.

Odd widths load and store the rows at 2 mod 4 through the neighbour lane: the
shapes put a wave's blocks on one row, across rows and across frames whose rows
have other parities, with 1, 3, 5 and 7 elements in the block at a row's end and
partial block rows; a volume of even width at 2 mod 4 takes the general code.
Streams and decoded volumes are byte-equal to the oracle's and nothing outside
the volume is written."""
import numpy as np
import pytest

from lsc_helpers import MODES, synth

pytestmark = pytest.mark.gpu

# more than 704 tiles of 512 blocks each
SHAPES = [(12, 2000, 1999), (70, 621, 621), (10000, 61, 33), (2900, 81, 91), (70, 621, 622)]


@pytest.mark.parametrize("kind,mode", [("cssi", "lossless"), ("uniform", "lossless"), ("cssi", "b3-5-10-15_p0.5"),
                                       ("mixed", "b1-2-4-8_p0")])
@pytest.mark.parametrize("off", [0, 1])
@pytest.mark.parametrize("shape", SHAPES, ids=lambda s: "x".join(map(str, s)))
def test_odd_rows(gpu, orc, shape, off, kind, mode):
    import torch
    bins, p = MODES[mode]
    vol = synth(kind, shape, seed=31)
    n = vol.size
    st, ref, refn = orc.compress(vol, bins, p, omp=True)
    assert st == 0
    big = torch.zeros(n + 16, dtype=torch.int16, device="cuda")
    d_in = big[off:off + n].view(shape)
    d_in.copy_(torch.from_numpy(vol.view(np.int16)))
    out, got = gpu.compress(d_in, shape, bins, p)
    assert got == refn and np.array_equal(out[:got].cpu().numpy(), ref)
    big.fill_(0x5A5A)
    gpu.decompress(out, got, shape, bins, out=d_in)
    _, want = orc.decompress(ref, shape, bins, omp=True)
    host = big.cpu().numpy().view(np.uint16)
    assert np.array_equal(host[off:off + n], want.ravel())
    assert np.all(host[:off] == 0x5A5A) and np.all(host[off + n:] == 0x5A5A)


@pytest.mark.parametrize("off", [0, 4, 8, 12])
@pytest.mark.parametrize("mode", ["lossless", "b3-5-10-15_p0.5"])
def test_large_decode_stream_offsets(gpu, orc, off, mode):
    import torch
    bins, p = MODES[mode]
    shape = (24, 1000, 1030)   # 756 tiles
    vol = synth("cssi", shape, seed=21)
    _, ref, refn = orc.compress(vol, bins, p, omp=True)
    _, want = orc.decompress(ref, shape, bins, omp=True)
    buf = torch.full((refn + 64,), 0xC3, dtype=torch.uint8, device="cuda")
    buf[off:off + refn].copy_(torch.from_numpy(ref))
    got = gpu.decompress(buf[off:off + refn], refn, shape, bins)
    assert np.array_equal(got.cpu().numpy().view(np.uint16), want)
