"""tg_hip_matmul_dev over its dispatch: every format at row lengths of each form
in which the launch cuts a row, partial q8 blocks and rows past what the
staged kernel holds, row counts around a wave's groups and past one grid, and
input row counts that quantize in the kernel, in a launch of their own, and in
several staged chunks.  Bar: max|d| <= 1e-5 max|ref| against the oracle, whose
sums run in another order."""

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

Q4K, F16, Q6K, MXFP4, Q80 = 0, 1, 2, 3, 4


def _matrix(tg, rng, fmt, nrows, ncols):
    import tinygiant_amd.synth as S
    if fmt == F16:
        return (rng.standard_normal(nrows * ncols) * 0.05).astype(np.float16).view(np.uint8)
    return S.matrix_host(fmt, int(rng.integers(1 << 40)), nrows, ncols)


@pytest.mark.parametrize("fmt,nrows,ncols,k,bias", [
    (Q4K, 1, 256, 1, True), (Q4K, 33, 512, 2, False), (Q6K, 63, 768, 5, True), (Q6K, 7, 2048, 3, False),
    (Q4K, 130, 4096, 16, True), (Q6K, 41, 12288, 1, True), (Q4K, 9, 16384, 4, False), (Q4K, 9, 16640, 2, True),
    (Q4K, 40001, 256, 1, False), (Q6K, 40001, 256, 3, True),
    (Q80, 5, 32, 1, True), (Q80, 65, 288, 3, True), (Q80, 100, 2880, 1, True), (Q80, 31, 2880, 9, False),
    (Q80, 17, 4096, 1, False), (Q80, 13, 8192, 9, True), (Q80, 13, 8224, 2, True),
    (MXFP4, 77, 2880, 16, True), (MXFP4, 8, 96, 1, False), (MXFP4, 19, 5888, 2, True),
    (F16, 3, 32, 1, True), (F16, 70, 1056, 5, False), (F16, 33, 2880, 4, True), (F16, 21, 8192, 3, True),
    (F16, 9, 8224, 2, False), (F16, 1025, 512, 1, True)])
def test_matmul_dev_forms(tg, orc, fmt, nrows, ncols, k, bias):
    _check_matmul(tg, orc, fmt, nrows, ncols, k, bias)


# a row's items on 8, 16, 32 and 64 lanes, 1 to 4 a lane (up to 16 for F16), as the launch cuts it: a row length of
# each form, the longest or one with lanes left over
K_COLS = [512, 1280, 1536, 768, 2304, 2560, 3328, 3584, 1792, 4352, 7168, 3840, 7936, 8448, 12544]
BLOCK32_COLS = [96, 544, 288, 1056, 1568, 800, 2080, 3104, 1824, 3872, 4128, 6176]
F16_COLS = [32, 160, 288, 544, 96, 352, 608, 1056, 224, 736, 1248, 2080, 480, 992, 1504, 2016, 2528, 4128]


@pytest.mark.parametrize("fmt,ncols", [(f, c) for f in (Q4K, Q6K) for c in K_COLS] +
                         [(f, c) for f in (Q80, MXFP4) for c in BLOCK32_COLS] + [(F16, c) for c in F16_COLS])
def test_matmul_dev_every_row_form(tg, orc, fmt, ncols):
    """Each form with one row (quantized by the launch), two (quantized by it
    up to eight blocks a row) and nineteen (in q8 before it)."""
    for k in (1, 2, 19):
        _check_matmul(tg, orc, fmt, 37, ncols, k, k == 2)


def _check_matmul(tg, orc, fmt, nrows, ncols, k, bias):
    print(f"matmul fmt {fmt} {nrows} x {ncols}, {k} rows, bias {bias}", flush=True)
    lib = tg.lib()
    rng = np.random.default_rng(fmt * 1000 + nrows + ncols + k)
    w = _matrix(tg, rng, fmt, nrows, ncols)
    x = rng.standard_normal((k, ncols)).astype(np.float32)
    b = (rng.standard_normal(nrows) * 0.1).astype(np.float32) if bias else None
    bufs = []

    def dev(a):
        d = tg.DeviceArray(a.nbytes)
        d.upload(a)
        bufs.append(d)
        return d

    guard = np.full((k, nrows + 8), 7.0, np.float32)   # the rows lie densely: what follows must stay
    y, wd, xd, bd = dev(guard), dev(w), dev(x), dev(b) if bias else None
    sc = dev(np.zeros(lib.tg_hip_matmul_scratch_bytes(k, ncols), np.uint8))
    lib.tg_hip_clear_error()
    lib.tg_hip_matmul_dev(fmt, wd.ptr, bd.ptr if bias else None, xd.ptr, y.ptr, nrows, ncols, k, sc.ptr, None)
    lib.tg_hip_synchronize()
    assert tg.last_error() == ""
    flat = y.download(np.float32, guard.size)
    for d in bufs:
        d.free()
    got = flat[:k * nrows].reshape(k, nrows)
    assert (flat[k * nrows:] == 7.0).all()
    for j in range(k):
        ref = orc.matmul(fmt, w, b, x[j], nrows, ncols)
        assert np.abs(got[j] - ref).max() <= 1e-5 * np.abs(ref).max(), j


@pytest.mark.parametrize("fmt,size", [(Q4K, 144), (Q6K, 210)])
@pytest.mark.parametrize("byte", [0x00, 0x7F, 0x80, 0xFF])
def test_scale_products_at_their_largest(tg, orc, fmt, size, byte):
    """Blocks whose codes and scales are all one byte against rows of one
    sign (every q8 code 127) and of alternating signs: the integer sums and
    their products with the scales at the ends of their ranges (below 2^18
    and 2^26).  They are exact, so only the f32 terms' order differs: two
    blocks a row, 1e-6."""
    lib = tg.lib()
    nrows, ncols = 3, 512
    w = np.full((nrows * ncols // 256, size), byte, np.uint8)
    half = np.array([0.0371], np.float16).view(np.uint8)
    if fmt == Q4K:
        w[:, 0:2] = half
        w[:, 2:4] = half
    else:
        w[:, 208:210] = half
    w = w.reshape(-1)
    x = np.full((2, ncols), 1.7, np.float32)
    x[1, ::2] = -1.7
    print("scale products", fmt, byte, flush=True)
    bufs = [tg.DeviceArray(n) for n in (w.nbytes, x.nbytes, 2 * nrows * 4, lib.tg_hip_matmul_scratch_bytes(2, ncols))]
    bufs[0].upload(w)
    bufs[1].upload(x)
    lib.tg_hip_clear_error()
    lib.tg_hip_matmul_dev(fmt, bufs[0].ptr, None, bufs[1].ptr, bufs[2].ptr, nrows, ncols, 2, bufs[3].ptr, None)
    lib.tg_hip_synchronize()
    assert tg.last_error() == ""
    got = bufs[2].download(np.float32, 2 * nrows).reshape(2, nrows)
    for b in bufs:
        b.free()
    for j in range(2):
        ref = orc.matmul(fmt, w, None, x[j], nrows, ncols)
        assert np.abs(got[j] - ref).max() <= 1e-6 * max(np.abs(ref).max(), 1e-3), (j, got[j], ref)


@pytest.mark.parametrize("fmt,nrows,ncols,k,shift", [
    (Q4K, 2048, 2048, 1, 0), (Q6K, 8192, 8192, 1, 0), (Q80, 2880, 2880, 1, 0), (MXFP4, 4096, 512, 8, 0),
    (Q4K, 768, 2048, 1, 1500), (Q4K, 768, 2048, 1, -700), (Q80, 100, 288, 3, 860), (Q6K, 512, 512, 9, 0)])
@pytest.mark.parametrize("alloc", [True, False])
def test_matmul_dev_over_its_inputs(tg, fmt, nrows, ncols, k, shift, alloc):
    """Outputs that lie over the inputs (in place, and shifted by `shift`
    values either way) are the bits of a call with buffers apart: one row and
    few blocks, whose launch would quantize the rows while others write, and
    more, which are in q8 before."""
    print(f"matmul over its inputs: fmt {fmt} {nrows} x {ncols}, {k} rows, shift {shift}", flush=True)
    lib = tg.lib()
    rng = np.random.default_rng(fmt + nrows + ncols + k)
    x = rng.standard_normal((k, ncols)).astype(np.float32)
    nx, ny, pad = k * ncols, k * nrows, max(0, -shift)
    wd = tg.DeviceArray(nrows * lib.tg_row_bytes(fmt, ncols))
    wd.upload(_matrix(tg, rng, fmt, nrows, ncols))
    room = tg.DeviceArray(4 * (pad + max(nx, max(shift, 0) + ny)))
    apart = tg.DeviceArray(4 * ny)
    sc = tg.DeviceArray(lib.tg_hip_matmul_scratch_bytes(k, ncols))

    def call(y):
        room.upload(np.concatenate([np.zeros(pad, np.float32), x.reshape(-1)]))
        if alloc:
            lib.tg_hip_matmul_dev(fmt, wd.ptr, None, room.ptr + 4 * pad, y, nrows, ncols, k, sc.ptr, None)
        else:
            lib.tg_hip_matmul_dev_noalloc(fmt, wd.ptr, None, room.ptr + 4 * pad, y, nrows, ncols, k, None)
        lib.tg_hip_synchronize()
        assert tg.last_error() == ""

    lib.tg_hip_clear_error()
    lib.tg_hip_init()
    call(apart.ptr)
    call(room.ptr + 4 * (pad + shift))
    ref = apart.download(np.float32, ny)
    got = room.download(np.float32, room.nbytes // 4)[pad + shift:][:ny]
    for d in (wd, room, apart, sc):
        d.free()
    assert got.tobytes() == ref.tobytes()
