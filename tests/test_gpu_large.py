"""Volumes above the sizes that run with one workgroup per tile (uint16: 256 tiles
of 512 blocks to compress, 704 to decompress; uint32: 256 tiles of 256 and 448 of
512), through every persistent kernel: each way of finding the tile offsets, each
tile size, window and counter count, even and odd rows, dense and sparse payloads
(the pipelined and the sparse decoder), streams at each alignment, and what these
kernels report: short capacity, truncated streams and values out of range.  Streams
and volumes are the oracle's byte for byte."""
import numpy as np
import pytest

from lsc_helpers import MODES, synth

pytestmark = pytest.mark.gpu

SETTINGS = [MODES["lossless"], MODES["b3-5-10-15_p0.5"]]   # dense and sparse payloads
# 756 tiles of 512 (rows at 4-byte boundaries), 832 (odd rows whose parities differ
# between frames, partial block rows)
SHAPES = [(24, 1000, 1030), (70, 621, 621)]
SHAPE32 = (8, 1500, 1240)   # 911 tiles of 256, 456 of 512
GUARD = 0xC3
_refs = {}


def _case(orc, shape, k):
    """(volume, stream, decoded volume) of a shape and setting, by the oracle."""
    if (shape, k) not in _refs:
        bins, p = SETTINGS[k]
        vol = synth("cssi", shape, seed=31)
        st, ref, refn = orc.compress(vol, bins, p, omp=True)
        assert st == 0 and refn == ref.size
        _refs[shape, k] = vol, ref, orc.decompress(ref, shape, bins, omp=True)[1]
    return _refs[shape, k]


def _case32(orc, k):
    if k not in _refs:
        bins, p = SETTINGS[k]
        vol = synth("cssi", SHAPE32, seed=33).astype(np.uint32) * 4099
        st, ref, refn = orc.compress_u32(vol, bins, p)
        assert st == 0 and refn == ref.size
        _refs[k] = vol, ref, orc.decompress_u32(ref, SHAPE32, bins)[1]
    return _refs[k]


def _dev(a):
    import torch
    a = np.ascontiguousarray(a)
    return torch.from_numpy(a if a.itemsize == 1 else a.view(np.int16 if a.itemsize == 2 else np.int32)).cuda()


def _check(gpu, orc, shape, k):
    vol, ref, want = _case(orc, shape, k)
    out, n = gpu.compress(_dev(vol), shape, *SETTINGS[k])
    assert n == ref.size and np.array_equal(out[:n].cpu().numpy(), ref)
    dec = gpu.decompress(out, n, shape, SETTINGS[k][0])
    assert np.array_equal(dec.cpu().numpy().view(np.uint16), want)


@pytest.fixture
def keep_shapes(gpu):
    saved = [gpu.get_launch_shape_ex(k) for k in (gpu.COMPRESS, gpu.DECOMPRESS)]
    mode = gpu.set_decode_prepass(1)
    yield
    gpu.set_decode_prepass(mode)
    for k, s in zip((gpu.COMPRESS, gpu.DECOMPRESS), saved):
        gpu.set_launch_shape_ex(k, **s)


@pytest.mark.parametrize("shape", SHAPES, ids=lambda s: "x".join(map(str, s)))
@pytest.mark.parametrize("tile", [128, 256, 512])
@pytest.mark.parametrize("mode", [0, 1, 2])
def test_offset_modes(gpu, orc, keep_shapes, mode, tile, shape):
    """Look-back in the decode (0), the decode's offset phase (1), the pre-pass kernel (2)."""
    for k in (gpu.COMPRESS, gpu.DECOMPRESS):
        gpu.set_launch_shape(k, tile)
    gpu.set_decode_prepass(mode)
    for k in range(2):
        _check(gpu, orc, shape, k)


@pytest.mark.parametrize("shape", SHAPES, ids=lambda s: "x".join(map(str, s)))
@pytest.mark.parametrize("mode", sorted(MODES))
def test_settings(gpu, orc, mode, shape):
    """Compression has a kernel per kind of settings."""
    bins, p = MODES[mode]
    vol = _case(orc, shape, 0)[0]
    st, ref, refn = orc.compress(vol, bins, p, omp=True)
    out, n = gpu.compress(_dev(vol), shape, bins, p)
    assert st == 0 and n == refn and np.array_equal(out[:n].cpu().numpy(), ref)
    dec = gpu.decompress(out, n, shape, bins)
    assert np.array_equal(dec.cpu().numpy().view(np.uint16), orc.decompress(ref, shape, bins, omp=True)[1])


@pytest.mark.parametrize("shape", SHAPES, ids=lambda s: "x".join(map(str, s)))
@pytest.mark.parametrize("launch", [(128, 1, 128, 1), (256, 1, 256, 16), (512, 1, 512, 8), (512, 0, 64, 3), (512, 2, 256, 1)],
                         ids=lambda v: "-".join(map(str, v)))
def test_launch_shapes(gpu, orc, keep_shapes, launch, shape):
    for k in (gpu.COMPRESS, gpu.DECOMPRESS):
        gpu.set_launch_shape_ex(k, *launch)
    for mode in (1, 0):
        gpu.set_decode_prepass(mode)
        for k in range(2):
            _check(gpu, orc, shape, k)


@pytest.mark.parametrize("mode", [0, 1, 2])
def test_u32_offset_modes(gpu, orc, keep_shapes, mode):
    gpu.set_decode_prepass(mode)
    for k in range(2):
        vol, ref, want = _case32(orc, k)
        out, n = gpu.compress_u32(_dev(vol), SHAPE32, *SETTINGS[k])
        assert n == ref.size and np.array_equal(out[:n].cpu().numpy(), ref)
        dec = gpu.decompress_u32(out, n, SHAPE32, SETTINGS[k][0])
        assert np.array_equal(dec.cpu().numpy().view(np.uint32), want)


@pytest.mark.parametrize("k", [0, 1], ids=["lossless", "lossy"])
@pytest.mark.parametrize("off", [0, 4, 8, 12])
def test_u32_stream_offsets(gpu, orc, off, k):
    import torch
    vol, ref, want = _case32(orc, k)
    n = ref.size
    big = torch.full((n + off + 64,), GUARD, dtype=torch.uint8, device="cuda")
    _, got = gpu.compress_u32(_dev(vol), SHAPE32, *SETTINGS[k], out=big[off:off + n])
    host = big.cpu().numpy()
    assert got == n and np.array_equal(host[off:off + n], ref)
    assert np.all(host[:off] == GUARD) and np.all(host[off + n:] == GUARD)
    dec = gpu.decompress_u32(big[off:off + n], n, SHAPE32, SETTINGS[k][0])
    assert np.array_equal(dec.cpu().numpy().view(np.uint32), want)


def _short_capacity(gpu, compress, vol, dims, setting, ref):
    """Refused with the size it needs, nothing past the capacity; the exact size is enough."""
    import torch
    n = ref.size
    buf = torch.full((n + 64,), GUARD, dtype=torch.uint8, device="cuda")
    for cap in (n - 4, n - 100, n // 2):
        with pytest.raises(gpu.LscompError) as e:
            compress(vol, dims, *setting, out=buf[:cap])
        assert e.value.status == gpu.ERR_CAPACITY and e.value.required == n
        assert bool((buf[cap:] == GUARD).all())
        buf.fill_(GUARD)
    _, got = compress(vol, dims, *setting, out=buf[:n])
    assert got == n and np.array_equal(buf[:n].cpu().numpy(), ref) and bool((buf[n:] == GUARD).all())


@pytest.mark.parametrize("shape", SHAPES, ids=lambda s: "x".join(map(str, s)))
def test_short_capacity(gpu, orc, shape):
    vol, ref, _ = _case(orc, shape, 0)
    _short_capacity(gpu, gpu.compress, _dev(vol), shape, SETTINGS[0], ref)


def test_u32_short_capacity(gpu, orc):
    vol, ref, _ = _case32(orc, 0)
    _short_capacity(gpu, gpu.compress_u32, _dev(vol), SHAPE32, SETTINGS[0], ref)


def test_u32_value_out_of_range(gpu, orc):
    vol, ref, _ = _case32(orc, 0)
    d = _dev(vol)
    at = d.view(-1)
    for i in (0, vol.size // 2, vol.size - 1):   # the first tile, one between, the last
        was = int(at[i])
        at[i] = -(1 << 31)
        with pytest.raises(gpu.LscompError) as e:
            gpu.compress_u32(d, SHAPE32, *SETTINGS[0])
        assert e.value.status == gpu.ERR_RANGE
        at[i] = was
        out, n = gpu.compress_u32(d, SHAPE32, *SETTINGS[0])   # and the next call is clean
        assert n == ref.size and np.array_equal(out[:n].cpu().numpy(), ref)


@pytest.mark.parametrize("mode", [0, 1, 2])
def test_truncated_streams(gpu, orc, keep_shapes, mode):
    """The pipelined, the sparse and the look-back decoder, and uint32's: the error is
    reported by the call, and the next call is clean."""
    gpu.set_decode_prepass(mode)
    for k in range(2):
        _, ref, want = _case(orc, SHAPES[0], k)
        d = _dev(ref)
        with pytest.raises(gpu.LscompError) as e:
            gpu.decompress(d, ref.size - 8, SHAPES[0], SETTINGS[k][0])
        assert e.value.status == gpu.ERR_CORRUPT
        dec = gpu.decompress(d, ref.size, SHAPES[0], SETTINGS[k][0])
        assert np.array_equal(dec.cpu().numpy().view(np.uint16), want)
    _, ref, want = _case32(orc, 0)
    with pytest.raises(gpu.LscompError) as e:
        gpu.decompress_u32(_dev(ref), ref.size - 8, SHAPE32)
    assert e.value.status == gpu.ERR_CORRUPT
    dec = gpu.decompress_u32(_dev(ref), ref.size, SHAPE32)
    assert np.array_equal(dec.cpu().numpy().view(np.uint32), want)
