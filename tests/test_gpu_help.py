"""The small-volume compression where a workgroup finds earlier tiles' totals
missing: it forms them itself, after the number of probes that the call gives (0:
after the first), and streams stay byte-equal to the oracle's."""
import ctypes

import numpy as np
import pytest

from lsc_helpers import MODES, synth


def _entry(lscomp):
    f = lscomp._lib.lscomp_internal_compress_u16_async
    f.restype = ctypes.c_int
    f.argtypes = [ctypes.c_void_p, ctypes.c_void_p, ctypes.c_size_t, ctypes.c_void_p, lscomp.Dim3, lscomp.Bins4,
                  ctypes.c_float, ctypes.c_uint32, ctypes.c_void_p]
    return f


def test_no_switch_in_the_environment():
    """The wait for a missing total is not a setting of the process."""
    import lscomp
    with open(lscomp.LIB_PATH, "rb") as f:
        assert b"LSCOMP_HELP_PROBES" not in f.read()


@pytest.mark.gpu
@pytest.mark.parametrize("mode", ["lossless", "b3-5-10-15_p0.5"])
@pytest.mark.parametrize("n", [1, 65, 4096, 16384, 40000, 131072])
def test_missing_totals_are_formed(gpu, orc, n, mode):
    import torch
    f = _entry(gpu)
    bins, p = MODES[mode]
    vol = synth("sparse", (1, 8, 8 * n), seed=n)
    _, ref, refn = orc.compress(vol, bins, p)
    d = torch.from_numpy(vol.view(np.int16)).cuda()
    size = torch.zeros(1, dtype=torch.int64, device="cuda")
    for help_probes in (0, 3, 0xffffffff):   # the last: as many as any call
        out = torch.full((refn + 64,), 0x6B, dtype=torch.uint8, device="cuda")
        size.zero_()
        st = f(d.data_ptr(), out.data_ptr(), refn, size.data_ptr(), gpu._dims(vol.shape), gpu._bins(bins), p,
               help_probes, torch.cuda.current_stream().cuda_stream)
        assert st == gpu.OK and gpu.stream_status() == gpu.OK
        got = out.cpu().numpy()
        assert int(size.item()) == refn and np.array_equal(got[:refn], ref) and np.all(got[refn:] == 0x6B)
