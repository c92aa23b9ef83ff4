"""GPU parity of the corner turns either side of the beamformer, through the
C ABI, against the oracle: the TUSE beam corner turn
(meerkat/tuse/src/transpose_to_dada.cpp:19-48) and the F-engine heap reorder
(meerkat/tools/src/feng_to_dada.cu:54-80).  Byte moves: bit-exact."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _dev(capi, a):
    return capi.DeviceBuffer.from_array(np.ascontiguousarray(a))


@pytest.mark.parametrize("C,S,F,B,G,b0,nb", [
    (128, 64, 32, 4, 10, 0, 4),     # the reference's default geometry (transpose_to_dada.cpp:13-16), 4 beams
    (64, 128, 16, 6, 2, 0, 6),      # 16-byte units, full 16 x 16 element tiles
    (64, 40, 13, 3, 2, 1, 2),       # partial tiles, a beam range
    (12, 33, 17, 2, 3, 1, 1),       # 4-byte units, element 12 bytes
    (3, 9, 70, 4, 2, 2, 2),         # 1-byte units, odd element size, > 64 bands
    (4096, 4, 3, 2, 2, 0, 2),       # large elements: one element per tile
    (16, 1, 1, 1, 1, 0, 1),         # degenerate 1 x 1 matrix
])
def test_tuse_transpose_bit_exact(gpu, oracle, C, S, F, B, G, b0, nb):
    capi = gpu
    rng = np.random.default_rng(C * 7 + S)
    blk = rng.integers(-128, 128, G * B * F * S * C).astype(np.int8)
    d_in = _dev(capi, blk)
    d_out = capi.DeviceBuffer(nb * G * S * F * C)
    capi.tuse_transpose(d_in, d_out, C, S, F, B, G, b0, nb)
    np.testing.assert_array_equal(d_out.download(), oracle.tuse_transpose(blk, C, S, F, B, G, b0, nb))


def test_tuse_transpose_full_size_against_numpy(gpu):
    """The bench workload: 512 beams x 16 bands x 512 samples (4 groups of
    128) x 64 channels, 256 MiB; checked against numpy's transpose of the
    same block."""
    capi = gpu
    C, S, F, B, G = 64, 128, 16, 512, 4
    n = G * B * F * S * C
    blk = capi.synth_gaussian_int8(99, 30.0, n)
    d_in = _dev(capi, blk)
    d_out = capi.DeviceBuffer(n)
    capi.tuse_transpose(d_in, d_out, C, S, F, B, G)
    got = d_out.download()
    ref = blk.reshape(G, B, F, S, C).transpose(1, 0, 3, 2, 4).reshape(-1)
    assert np.array_equal(got, ref)


def test_tuse_transpose_rejects_bad_sizes(gpu):
    capi = gpu
    C, S, F, B, G = 16, 8, 4, 3, 2
    d_in = capi.DeviceBuffer(G * B * F * S * C)
    with pytest.raises(RuntimeError, match="geometry needs"):
        capi.tuse_transpose(capi.DeviceBuffer(100), capi.DeviceBuffer(B * G * S * F * C), C, S, F, B, G)
    with pytest.raises(RuntimeError, match="output must be"):
        capi.tuse_transpose(d_in, capi.DeviceBuffer(7), C, S, F, B, G)
    with pytest.raises(RuntimeError, match="beam range"):
        capi.tuse_transpose(d_in, capi.DeviceBuffer(2 * G * S * F * C), C, S, F, B, G, 2, 2)


@pytest.mark.parametrize("nchans,nts", [(32, 3), (4096, 2), (96, 5), (40, 1), (1, 4)])
def test_feng_to_dada_bit_exact(gpu, oracle, nchans, nts):
    capi = gpu
    rng = np.random.default_rng(nchans + nts)
    w = rng.integers(-2**31, 2**31, nts * nchans * 256, dtype=np.int64).astype(np.int32)
    d_in = _dev(capi, w)
    d_out = capi.DeviceBuffer(w.nbytes)
    capi.feng_to_dada(d_in, d_out, nchans)
    np.testing.assert_array_equal(d_out.download(np.int32), oracle.feng_to_dada(w, nchans))


def test_feng_to_dada_rejects_bad_sizes(gpu):
    capi = gpu
    d = capi.DeviceBuffer(32 * 256 * 4 * 2)
    with pytest.raises(RuntimeError, match="bytes per timestamp"):
        capi.call("fbf_feng_to_dada", d.ptr, capi.DeviceBuffer(d.nbytes).ptr, d.nbytes - 4, 32, None)
    with pytest.raises(RuntimeError, match="distinct"):
        capi.feng_to_dada(d, d, 32)


@pytest.mark.parametrize("C,S,F,B,G,b0,nb", [
    (23, 92, 44, 3, 2, 1, 2),        # bytes, odd elements, partial tiles both ways
    (1, 300, 7, 2, 1, 0, 2),         # single bytes, fewer bands than a tile has rows
    (148, 70, 41, 2, 2, 0, 2),       # 4-byte units, 37 to an element
    (4, 289, 54, 2, 3, 0, 1),        # one 4-byte unit, rows of no 16-byte multiple
    (48, 133, 5, 7, 2, 2, 5),        # 16-byte units, three to an element, few bands
    (256, 64, 32, 33, 1, 0, 33),     # 16 MiB and more: stored past the cache
    (36, 512, 64, 15, 1, 0, 15),     # the same in 4-byte units
    (64, 100, 1, 6, 3, 1, 5),        # one band: rows of four units
    (1, 300, 2, 5, 4, 0, 5),         # two bands of single bytes
    (5, 77, 3, 4, 2, 0, 4), (17, 33, 1, 3, 2, 0, 3),   # 15 and 17 units
    (8, 22, 3, 7, 2, 0, 7), (4, 63, 4, 3, 1, 0, 3), (4, 64, 4, 3, 1, 0, 3),   # whole matrices of few units
])
def test_tuse_transpose_tile_shapes_bit_exact(gpu, C, S, F, B, G, b0, nb):
    """Tile shapes by unit size, bands and block size against numpy."""
    capi = gpu
    rng = np.random.default_rng(C + S + F)
    x = rng.integers(-128, 128, (G, B, F, S, C), dtype=np.int8)
    d_out = capi.DeviceBuffer(G * nb * F * S * C)
    capi.tuse_transpose(_dev(capi, x), d_out, C, S, F, B, G, beam0=b0, nbeams_out=nb)
    ref = np.ascontiguousarray(x[:, b0:b0 + nb].transpose(1, 0, 3, 2, 4))
    np.testing.assert_array_equal(d_out.download(), ref.reshape(-1))


@pytest.mark.parametrize("C,S,F,B,G", [
    (7, 900, 40, 2, 1), (3, 64, 64, 8, 4),     # few tiles: shrunk to two units a thread
    (5, 7, 5, 300, 3),                         # a matrix smaller than a tile
    (13, 37, 41, 3, 2),                        # steps: a tile's last rows and columns in bytes
    (36, 50, 17, 4, 3),                        # the same in 4-byte units, nine to an element
    (1, 4000, 2, 40, 20),                      # rows: output rows of two bytes
    (20, 530, 33, 2, 40),                      # rows: the last tile holds one row
    (52, 166, 2, 30, 15),                      # rows: fewer than a work-group has waves
    (64, 61, 9, 3, 2), (48, 61, 9, 3, 2),      # 16-byte units, shifts and multiplications, partial tiles
    (512, 9, 5, 3, 2),                         # two elements a tile row
    (112, 77, 19, 30, 2),                      # 8 MiB and more: past the cache, no power of two
    (4, 4, 4, 3, 2), (4, 68, 60, 3, 2), (4, 260, 132, 2, 3),   # word tiles: partial rows and columns
    (4, 1024, 96, 24, 1),                      # word tiles of whole lines past the cache, partial rows
    (4, 1024, 100, 24, 1),                     # and cached, rows of no whole lines
])
def test_tuse_transpose_every_walk_bit_exact(gpu, C, S, F, B, G):
    """Each way a tile is walked, at its edges, against numpy."""
    capi = gpu
    rng = np.random.default_rng(C + S + F + 1)
    x = rng.integers(-128, 128, (G, B, F, S, C), dtype=np.int8)
    d_out = capi.DeviceBuffer(G * B * F * S * C)
    capi.tuse_transpose(_dev(capi, x), d_out, C, S, F, B, G)
    ref = np.ascontiguousarray(x.transpose(1, 0, 3, 2, 4))
    np.testing.assert_array_equal(d_out.download(), ref.reshape(-1))


@pytest.mark.parametrize("C,n", [(96, 200), (193, 100), (1056, 16), (1024, 140)])
def test_feng_to_dada_large_blocks_bit_exact(gpu, C, n):
    """F-engine blocks of 16 MiB and more (a partial tile of 32 channels, odd
    channels, 33 lines to a row) and one of 140 MiB."""
    capi = gpu
    rng = np.random.default_rng(C)
    x = rng.integers(0, 1 << 32, (n, C, 256), dtype=np.uint32)
    d_out = capi.DeviceBuffer(x.nbytes)
    capi.feng_to_dada(_dev(capi, x), d_out, C)
    np.testing.assert_array_equal(d_out.download(np.uint32), x.transpose(0, 2, 1).reshape(-1))
