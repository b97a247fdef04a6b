"""Small volumes (one workgroup per tile, no tile ids).  Compression: byte-equal
to the oracle at the edges of the tile choice and of the path itself, over
calls whose sizes go up and down on one scratch area.  Workgroups that form
totals they find missing themselves are in test_gpu_help.py: the number of probes
before they do is an argument there, and the environment variable that the last
test here sets has no effect on the library."""
import os
import subprocess
import sys

import numpy as np
import pytest

from lsc_helpers import MODES, synth

pytestmark = pytest.mark.gpu

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
# blocks on both sides of each tile size's range (64, 128, 256, 512 blocks per
# tile) and of 256 tiles, and less than a wave
EDGES = (1, 63, 65, 4096, 4097, 16384, 16385, 49152, 49153, 131072, 131073)


def _check(gpu, orc, vol, bins, p):
    import torch
    want_st, ref, refn = orc.compress(vol, bins, p)
    assert want_st == 0
    out, n = gpu.compress(torch.from_numpy(vol.view(np.int16)).cuda(), vol.shape, bins, p)
    assert n == refn and np.array_equal(out[:n].cpu().numpy(), ref)


@pytest.mark.parametrize("mode", ["lossless", "b3-5-10-15_p0.5", "b1-2-4-8_p0"])
def test_small_edges(gpu, orc, mode):
    bins, p = MODES[mode]
    for n in EDGES + EDGES[::-1]:   # up, then down: stale totals of a larger volume
        _check(gpu, orc, synth("mixed" if n < 20000 else "sparse", (1, 7, 8 * n - 3), seed=n), bins, p)


@pytest.mark.parametrize("n", [1, 65, 4096, 4097, 16384, 16385, 65536, 65537])
def test_small_edges_u32(gpu, orc, n):
    import torch
    rng = np.random.default_rng(n)
    vol = (rng.poisson(0.4, (1, 8, 8 * n - 2)).astype(np.uint32) << 9) * 3
    for bins, p in (((1, 1, 1, 1), 1.0), ((3, 5, 10, 15), 0.5)):
        st, ref, refn = orc.compress_u32(vol, bins, p)
        assert st == 0
        out, got = gpu.compress_u32(torch.from_numpy(vol.view(np.int32)).cuda(), vol.shape, bins, p)
        assert got == refn and np.array_equal(out[:got].cpu().numpy(), ref)


# decompression: the edges of its tile sizes (64, 128, 256, 512 blocks) and of
# the path (704 tiles of 512 blocks; 448 for uint32), sparse and dense payloads
@pytest.mark.parametrize("kind", ["sparse", "uniform"])
@pytest.mark.parametrize("n", [1, 63, 65, 4096, 4097, 16384, 16385, 65536, 65537, 704 * 512, 704 * 512 + 1])
def test_small_decode_edges(gpu, orc, kind, n):
    import torch
    vol = synth(kind, (1, 7, 8 * n - 3), seed=n)
    for bins, p in (MODES["lossless"], MODES["b3-5-10-15_p0.5"]):
        _, ref, refn = orc.compress(vol, bins, p)
        _, want = orc.decompress(ref, vol.shape, bins)
        got = gpu.decompress(torch.from_numpy(ref).cuda(), refn, vol.shape, bins)
        assert np.array_equal(got.cpu().numpy().view(np.uint16), want)


@pytest.mark.parametrize("n", [65, 4096, 4097, 16385, 65537, 448 * 512, 448 * 512 + 1])
def test_small_decode_edges_u32(gpu, orc, n):
    import torch
    vol = np.random.default_rng(n).poisson(0.4, (1, 8, 8 * n - 2)).astype(np.uint32) << 12
    _, ref, refn = orc.compress_u32(vol, (1, 1, 1, 1), 1.0)
    got = gpu.decompress_u32(torch.from_numpy(ref).cuda(), refn, vol.shape)
    assert np.array_equal(got.cpu().numpy().view(np.uint32), vol)


def test_small_missing_totals_are_formed(gpu):
    """The same streams when no workgroup waits for another's total."""
    code = ("import sys; sys.path[:0] = [%r, %r, %r]\n"
            "import lscomp, oracle, test_gpu_small as t\n"
            "from lsc_helpers import MODES, synth\n"
            "for n in (100, 4096, 16384, 40000, 131072):\n"
            "    for m in ('lossless', 'b3-5-10-15_p0.5'):\n"
            "        t._check(lscomp, oracle.get(), synth('sparse', (1, 8, 8 * n), n), *MODES[m])\n"
            "print('equal')\n") % (ROOT, os.path.join(ROOT, "sc25-lscomp_amd"), os.path.join(ROOT, "tests"))
    r = subprocess.run([sys.executable, "-c", code], env=dict(os.environ, LSCOMP_HELP_PROBES="0"),
                       capture_output=True, text=True, timeout=100)
    assert r.returncode == 0 and "equal" in r.stdout, r.stdout[-500:] + r.stderr[-2000:]
