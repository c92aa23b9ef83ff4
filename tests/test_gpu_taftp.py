"""Coherent beams straight from TAFTP (fbf_cb_beamform_taftp) and the
incoherent beam with the weights in one launch (fbf_ib_beamform_weights).

The oracle for fbf_cb_beamform_taftp is the reference's pair as its Pipeline
calls it (Pipeline.cu:166-168): the oracle's split-transpose of the plan's
antennas, then the oracle's coherent beamformer; bit-exact.  Cases cover the
direct path (the kernel stages the TAFTP runs and transposes them in LDS:
64 or 128 beams per wave, antennas padded to a multiple of 16, subarrays at
any antenna offset, tscrunch 4 to 64, heaps of 16 to 512 samples, weight
components of -128 on the exact path) and the fallback through the plan's
FTPA buffer (geometries the direct path does not take: fscrunch above 1,
32 beams per wave, the other kernels, heaps that are not a power of two).
"""
import numpy as np
import pytest

from conftest import gaussian_int8, unit_weights

pytestmark = pytest.mark.gpu


def _dev(capi, arr):
    return capi.DeviceBuffer.from_array(arr)


def _levels(oracle, A, ts, fs, F):
    cbo, cbs, _, _ = oracle.power_levels(16.0, 24.0, A, ts, fs, 64, 16, 1)
    Fo = F // fs
    return np.full(Fo, cbo, np.float32), np.full(Fo, cbs, np.float32)


def _check_taftp(capi, oracle, Atot, A, a0, F, nhg, B, ts, fs, S, variant, direct, seed, weights=None):
    T = nhg * S
    taftp = gaussian_int8(seed, nhg * Atot * F * S * 4, 16.0)
    w = unit_weights(seed + 1, F * B * A) if weights is None else weights
    off, sc = _levels(oracle, A, ts, fs, F)
    plan = capi.CbPlan(A, B, F, ts, fs, off, sc, nsamples_per_heap_out=T // ts)
    plan.set_variant(variant)
    assert plan.taftp_direct(Atot, T, S) == direct
    ftpa = oracle.split_transpose(taftp, nhg, Atot, A, a0, F, nsamples_per_heap=S)
    ref = oracle.cb_tbtf(oracle.cb_power(ftpa, w, F, T, A, B, ts, fs), off, sc, T // ts)
    d_t, d_w = _dev(capi, taftp), _dev(capi, w)
    d_o = capi.DeviceBuffer((F // fs) * (T // ts) * B)
    d_o.fill(0x5A)
    plan.beamform_taftp(d_t, d_w, d_o, nantennas_total=Atot, start_antenna=a0, nsamples_per_heap=S)
    np.testing.assert_array_equal(d_o.download(), ref)
    return plan, d_t, d_w, d_o


@pytest.mark.parametrize("Atot,A,a0,F,nhg,B,ts,fs,S,variant", [
    (64, 64, 0, 8, 2, 512, 16, 1, 256, 0),     # the bench geometry (channels and heaps cut)
    (64, 64, 0, 4, 2, 512, 16, 1, 256, 11),    # 128 beams per wave
    (64, 40, 0, 8, 2, 96, 16, 1, 256, 11),     # 40 antennas: rows 40..47 padded
    (64, 64, 0, 4, 2, 256, 4, 1, 256, 9),      # tscrunch 4 (four windows a tile)
    (64, 32, 32, 4, 2, 128, 4, 1, 256, 9),     # upper half, tscrunch 4
    (64, 16, 40, 8, 2, 64, 16, 1, 256, 9),     # subarray at antenna 40
    (64, 8, 56, 4, 2, 64, 8, 1, 256, 9),       # last 8 antennas, one K step
    (128, 64, 64, 2, 2, 256, 32, 1, 256, 9),   # upper half of a 128-antenna block, tscrunch 32
    (64, 48, 8, 4, 2, 200, 64, 1, 256, 11),    # tscrunch 64 (four tiles a window), ragged beams
    (64, 64, 0, 4, 4, 512, 16, 1, 128, 9),     # 128-sample heaps
    (64, 64, 0, 2, 1, 256, 16, 1, 512, 9),     # 512-sample heaps
    (32, 24, 4, 4, 16, 64, 16, 1, 16, 11),     # 16-sample heaps: one tile a heap
    (64, 64, 0, 4, 3, 512, 8, 1, 256, 11),     # three heap groups, tscrunch 8
])
def test_cb_taftp_direct_bit_exact(gpu, oracle, Atot, A, a0, F, nhg, B, ts, fs, S, variant):
    _check_taftp(gpu, oracle, Atot, A, a0, F, nhg, B, ts, fs, S, variant, True, 2000 + A + a0 + S)


@pytest.mark.parametrize("Atot,A,a0,F,nhg,B,ts,fs,S,variant", [
    (64, 40, 0, 8, 2, 96, 4, 2, 256, 0),       # 40 antennas: the automatic pick is the wave-private kernel
    (128, 128, 0, 2, 1, 32, 8, 1, 256, 0),     # 128 antennas: 32 beams per wave
    (64, 20, 3, 4, 2, 64, 16, 1, 256, 0),      # 20 antennas (the LDS kernel)
    (64, 64, 0, 4, 2, 512, 16, 1, 96, 9),      # 96-sample heaps (not a power of two)
    (64, 64, 0, 4, 2, 256, 16, 1, 256, 5),     # the LDS variant chosen explicitly
    (64, 32, 16, 8, 2, 128, 8, 4, 256, 9),     # fscrunch 4
    (64, 64, 0, 4, 2, 512, 32, 2, 256, 8),     # fscrunch 2, 32 beams per wave
])
def test_cb_taftp_fallback_bit_exact(gpu, oracle, Atot, A, a0, F, nhg, B, ts, fs, S, variant):
    _check_taftp(gpu, oracle, Atot, A, a0, F, nhg, B, ts, fs, S, variant, False, 2100 + A + a0 + S)


@pytest.mark.parametrize("variant,Atot,A,a0", [(9, 128, 64, 32), (11, 64, 48, 8)])
def test_cb_taftp_minus128_weights_exact(gpu, oracle, variant, Atot, A, a0):
    """Weight components of -128 on the direct path: the work-groups that
    hold one compute their outputs on the exact int32 path, which then reads
    the TAFTP block itself (antenna stride F * S * 4 bytes)."""
    F, nhg, B, ts, fs, S = 4, 2, 256, 16, 1, 256
    w = unit_weights(2201, F * B * A).reshape(F, B, A, 2).copy()
    w[0, 3, 5, 1] = -128
    w[F - 1, B - 7, 0, 1] = -128
    w[F - 1, B - 7, 1, 0] = -128
    w[1, B // 2, A - 1, :] = -128
    _check_taftp(gpu, oracle, Atot, A, a0, F, nhg, B, ts, fs, S, variant, True, 2200, weights=w.reshape(-1))


def test_cb_taftp_direct_needs_block_below_4gib(gpu, oracle):
    """The direct path addresses the block with 32-bit tile offsets, so a
    block of 4 GiB or more takes the split-transpose path (a query only: no
    such block is allocated)."""
    capi = gpu
    A, F, B, ts, S = 64, 64, 512, 16, 256
    off, sc = _levels(oracle, A, ts, 1, F)
    plan = capi.CbPlan(A, B, F, ts, 1, off, sc)
    hg = 4 * A * F * S                    # bytes per heap group
    below = ((1 << 32) - 1) // hg          # heap groups of the largest block below 4 GiB
    assert plan.taftp_direct(A, below * S, S)
    assert not plan.taftp_direct(A, (below + 1) * S, S)


def test_cb_taftp_matches_ftpa_path_and_repeats(gpu, oracle):
    """The direct path equals split-transpose + fbf_cb_beamform on the GPU
    at a larger block (64 channels, 4 heap groups, 512 beams), on two calls
    in a row (the second with other voltages), and a forced fallback (the
    LDS variant) equals both."""
    capi = gpu
    Atot, A, F, nhg, B, ts, S = 64, 64, 64, 4, 512, 16, 256
    T = nhg * S
    off, sc = _levels(oracle, A, ts, 1, F)
    plan = capi.CbPlan(A, B, F, ts, 1, off, sc, nsamples_per_heap_out=T // ts)
    assert plan.taftp_direct(Atot, T, S)
    w = unit_weights(2301, F * B * A)
    d_w = _dev(capi, w)
    d_f = capi.DeviceBuffer(F * T * 2 * A * 2)
    d_a = capi.DeviceBuffer(F * (T // ts) * B)
    d_b = capi.DeviceBuffer(F * (T // ts) * B)
    for seed in (2302, 2303):
        d_t = _dev(capi, gaussian_int8(seed, nhg * Atot * F * S * 4, 16.0))
        capi.split_transpose(d_t, d_f, Atot, A, 0, F)
        plan.beamform(d_f, d_w, d_a)
        d_b.fill(0x5A)
        plan.beamform_taftp(d_t, d_w, d_b, nantennas_total=Atot)
        np.testing.assert_array_equal(d_b.download(), d_a.download())
    plan.set_variant(5)
    assert not plan.taftp_direct(Atot, T, S)
    d_b.fill(0x5A)
    plan.beamform_taftp(d_t, d_w, d_b, nantennas_total=Atot)
    np.testing.assert_array_equal(d_b.download(), d_a.download())


def test_cb_taftp_rejects_bad_arguments(gpu):
    capi = gpu
    A, B, F, ts, S = 16, 32, 4, 16, 256
    off, sc = np.full(F, 1.0, np.float32), np.full(F, 1.0, np.float32)
    plan = capi.CbPlan(A, B, F, ts, 1, off, sc, nsamples_per_heap_out=S // ts)
    d_t = capi.DeviceBuffer(32 * F * S * 4)       # one heap group of 32 antennas
    d_w = capi.DeviceBuffer(F * B * A * 2)
    d_o = capi.DeviceBuffer(F * (S // ts) * B)
    with pytest.raises(capi.FbfError):            # antennas past the block's
        plan.beamform_taftp(d_t, d_w, d_o, nantennas_total=32, start_antenna=20)
    with pytest.raises(capi.FbfError):            # not a whole number of heap groups
        plan.beamform_taftp(d_t, d_w, d_o, nantennas_total=48)
    with pytest.raises(capi.FbfError):            # weights size
        plan.beamform_taftp(d_t, capi.DeviceBuffer(F * B * A * 2 - 2), d_o, nantennas_total=32)
    with pytest.raises(capi.FbfError):            # output size
        plan.beamform_taftp(d_t, d_w, capi.DeviceBuffer(F * (S // ts) * B + 1), nantennas_total=32)
    plan.set_variant(5)                           # the fallback checks sizes before it launches
    with pytest.raises(capi.FbfError):
        plan.beamform_taftp(d_t, capi.DeviceBuffer(F * B * A * 2 - 2), d_o, nantennas_total=32)
    with pytest.raises(capi.FbfError):
        plan.beamform_taftp(d_t, d_w, capi.DeviceBuffer(F * (S // ts) * B + 1), nantennas_total=32)
    plan.beamform_taftp(d_t, d_w, d_o, nantennas_total=32, start_antenna=16)


@pytest.mark.parametrize("A,F,nhg,ts,fs,B", [(64, 64, 4, 16, 1, 512), (40, 8, 2, 32, 2, 96), (8, 16, 3, 1, 1, 7),
                                             (24, 4, 1, 4, 4, 33)])
def test_ib_beamform_weights_fused(gpu, oracle, A, F, nhg, ts, fs, B):
    """The incoherent beam and the weights in one launch equal
    fbf_ib_beamform and fbf_weights_generate byte for byte, and the IB
    output equals the oracle's."""
    capi = gpu
    taftp = gaussian_int8(2400 + A, nhg * A * F * 256 * 4, 16.0)
    _, _, ibo, ibs = oracle.power_levels(16.0, 24.0, A, 16, 1, A, ts, fs)
    Fo = F // fs
    ioff, isc = np.full(Fo, ibo, np.float32), np.full(Fo, ibs, np.float32)
    ib = capi.IbPlan(A, F, ts, fs, ioff, isc)
    freqs = capi.channel_frequencies_f64(1284e6, 856e6, F)
    wp = capi.WeightsPlan(A, B, F, freqs)
    delays = np.zeros((B * A, 2), np.float32)
    delays[:, 0] = capi.synth_uniform_f32(2401, -1e-9, 1e-9, B * A)
    delays[:, 1] = capi.synth_uniform_f32(2402, -1e-6, 1e-6, B * A)
    d_t, d_d = _dev(capi, taftp), _dev(capi, delays.reshape(-1))
    d_ib, d_ib2 = capi.DeviceBuffer(ib.output_bytes(d_t.nbytes)), capi.DeviceBuffer(ib.output_bytes(d_t.nbytes))
    d_w, d_w2 = capi.DeviceBuffer(F * B * A * 2), capi.DeviceBuffer(F * B * A * 2)
    ib.beamform(d_t, d_ib)
    wp.generate(d_d, 12.5, d_w)
    d_ib2.fill(0x5A)
    d_w2.fill(0x5A)
    ib.beamform_weights(d_t, d_ib2, wp, d_d, 12.5, d_w2)
    np.testing.assert_array_equal(d_ib2.download(), d_ib.download())
    np.testing.assert_array_equal(d_w2.download(), d_w.download())
    ref = oracle.ib_tf(oracle.ib_power(taftp, F, ts, fs, nhg, A), ioff, isc)
    np.testing.assert_array_equal(d_ib2.download(), ref.reshape(-1))


def test_ib_beamform_weights_rejects_channel_mismatch(gpu):
    capi = gpu
    A, F, B = 8, 16, 8
    ib = capi.IbPlan(A, F, 16, 1, np.zeros(F, np.float32), np.ones(F, np.float32))
    wp = capi.WeightsPlan(A, B, F // 2, capi.channel_frequencies_f64(1284e6, 856e6, F // 2))
    d_t = capi.DeviceBuffer(A * F * 256 * 4)
    d_ib = capi.DeviceBuffer(ib.output_bytes(d_t.nbytes))
    d_d = capi.DeviceBuffer(B * A * 8)
    d_w = capi.DeviceBuffer((F // 2) * B * A * 2)
    with pytest.raises(capi.FbfError):
        ib.beamform_weights(d_t, d_ib, wp, d_d, 0.0, d_w)


def _check_cb_ib(capi, oracle, A, F, nhg, B, ts, ib_ts, ib_fs, S, variant, fused, seed, weights=None):
    """fbf_cb_ib_beamform_taftp against the oracle: the coherent beams as in
    _check_taftp, the incoherent beam as the oracle's ib_power + ib_tf over
    all antennas (IncoherentBeamformer.cu:10-69)."""
    T = nhg * S
    taftp = gaussian_int8(seed, nhg * A * F * S * 4, 16.0)
    w = unit_weights(seed + 1, F * B * A) if weights is None else weights
    off, sc = _levels(oracle, A, ts, 1, F)
    _, _, ibo, ibs = oracle.power_levels(16.0, 24.0, A, ts, 1, A, ib_ts, ib_fs)
    Fo = F // ib_fs
    ioff, isc = np.full(Fo, ibo, np.float32), np.full(Fo, ibs, np.float32)
    plan = capi.CbPlan(A, B, F, ts, 1, off, sc, nsamples_per_heap_out=T // ts)
    if variant:
        plan.set_variant(variant)
    ib = capi.IbPlan(A, F, ib_ts, ib_fs, ioff, isc, nsamples_per_heap=S)
    assert plan.ib_fused(ib, T, S) == fused
    ftpa = oracle.split_transpose(taftp, nhg, A, A, 0, F, nsamples_per_heap=S)
    ref = oracle.cb_tbtf(oracle.cb_power(ftpa, w, F, T, A, B, ts, 1), off, sc, T // ts)
    ib_ref = oracle.ib_tf(oracle.ib_power(taftp, F, ib_ts, ib_fs, nhg, A, nsamples_per_heap=S), ioff, isc)
    d_t, d_w = _dev(capi, taftp), _dev(capi, w)
    d_o = capi.DeviceBuffer(F * (T // ts) * B)
    d_tf = capi.DeviceBuffer(ib.output_bytes(d_t.nbytes))
    for _ in range(2):   # a second call finds the partials buffer in use
        d_o.fill(0x5A)
        d_tf.fill(0x5A)
        plan.ib_beamform_taftp(ib, d_t, d_w, d_o, d_tf, nsamples_per_heap=S)
        np.testing.assert_array_equal(d_o.download(), ref)
        np.testing.assert_array_equal(d_tf.download(), ib_ref.reshape(-1))


@pytest.mark.parametrize("A,F,nhg,B,ts,ib_ts,ib_fs,S,variant", [
    (64, 8, 2, 512, 16, 16, 1, 256, 0),     # the bench geometry (channels and heaps cut)
    (64, 4, 2, 256, 4, 1, 1, 256, 0),       # IB per sample, CB tscrunch 4
    (64, 4, 3, 512, 8, 256, 2, 256, 0),     # IB windows of a whole heap, fscrunch 2
    (64, 8, 2, 1024, 32, 8, 4, 256, 0),     # two beam groups (only the first leaves partials), IB fscrunch 4
    (40, 8, 2, 200, 16, 16, 1, 256, 11),    # antennas 40..47 padded; waves without beams
    (48, 4, 2, 128, 64, 32, 1, 256, 11),    # three K slices: the fourth wave's slot holds zeros
    (16, 4, 4, 128, 16, 16, 1, 256, 11),    # one K slice
])
def test_cb_ib_fused_bit_exact(gpu, oracle, A, F, nhg, B, ts, ib_ts, ib_fs, S, variant):
    _check_cb_ib(gpu, oracle, A, F, nhg, B, ts, ib_ts, ib_fs, S, variant, True, 2500 + A + B + ib_ts)


@pytest.mark.parametrize("A,F,nhg,B,ts,ib_ts,ib_fs,S,variant", [
    (64, 4, 2, 256, 16, 16, 1, 256, 9),     # 64 beams per wave: the two beamformers in turn
    (40, 8, 2, 96, 16, 16, 2, 256, 0),      # the automatic pick at 40 antennas
])
def test_cb_ib_unfused_bit_exact(gpu, oracle, A, F, nhg, B, ts, ib_ts, ib_fs, S, variant):
    _check_cb_ib(gpu, oracle, A, F, nhg, B, ts, ib_ts, ib_fs, S, variant, False, 2600 + A + B + ib_ts)


def test_cb_ib_fused_minus128_weights_exact(gpu, oracle):
    """Work-groups with a weight component of -128 take the exact path and
    leave the incoherent-beam partials from the TAFTP block themselves."""
    A, F, nhg, B = 64, 4, 2, 512
    w = unit_weights(2701, F * B * A).reshape(F, B, A, 2).copy()
    w[0, 3, 5, 1] = -128
    w[F - 1, B - 7, 0, 1] = -128
    w[2, 100, :, :] = -128
    _check_cb_ib(gpu, oracle, A, F, nhg, B, 16, 16, 1, 256, 0, True, 2700, weights=w.reshape(-1))


@pytest.mark.parametrize("A,B,variant,alias", [(64, 512, 0, True), (64, 256, 0, False), (64, 256, 9, True)])
def test_cb_ib_next_weights(gpu, oracle, A, B, variant, alias):
    """fbf_cb_ib_beamform_taftp_next equals fbf_cb_ib_beamform_taftp followed
    by fbf_weights_generate at the next epoch: beams from this block's
    weights, then the next block's weights, also when they overwrite this
    block's (alias) and on the unfused path (variant 9)."""
    capi = gpu
    F, nhg, ts, S = 8, 2, 16, 256
    T = nhg * S
    taftp = gaussian_int8(2800 + B, nhg * A * F * S * 4, 16.0)
    off, sc = _levels(oracle, A, ts, 1, F)
    _, _, ibo, ibs = oracle.power_levels(16.0, 24.0, A, ts, 1, A, 16, 1)
    plan = capi.CbPlan(A, B, F, ts, 1, off, sc, nsamples_per_heap_out=T // ts)
    if variant:
        plan.set_variant(variant)
    ib = capi.IbPlan(A, F, 16, 1, np.full(F, ibo, np.float32), np.full(F, ibs, np.float32))
    assert plan.ib_fused(ib, T) == (variant == 0)
    freqs = capi.channel_frequencies_f64(1284e6, 856e6, F)
    wp = capi.WeightsPlan(A, B, F, freqs)
    delays = np.zeros((B * A, 2), np.float32)
    delays[:, 0] = capi.synth_uniform_f32(2801, -1e-9, 1e-9, B * A)
    delays[:, 1] = capi.synth_uniform_f32(2802, -1e-6, 1e-6, B * A)
    d_t, d_d = _dev(capi, taftp), _dev(capi, delays.reshape(-1))
    d_w = capi.DeviceBuffer(F * B * A * 2)
    wp.generate(d_d, 3.0, d_w)
    w_now = d_w.download()
    d_wn = capi.DeviceBuffer(F * B * A * 2)
    wp.generate(d_d, 3.0 + 0.0392, d_wn)
    w_next = d_wn.download()
    d_cb, d_tf = capi.DeviceBuffer(F * (T // ts) * B), capi.DeviceBuffer(ib.output_bytes(d_t.nbytes))
    d_cb2, d_tf2 = capi.DeviceBuffer(F * (T // ts) * B), capi.DeviceBuffer(ib.output_bytes(d_t.nbytes))
    plan.ib_beamform_taftp(ib, d_t, d_w, d_cb, d_tf)
    d_out_w = d_w if alias else capi.DeviceBuffer(F * B * A * 2)
    d_cb2.fill(0x5A)
    d_tf2.fill(0x5A)
    plan.ib_beamform_taftp_next(ib, d_t, d_w, d_cb2, d_tf2, wp, d_d, 3.0 + 0.0392, d_out_w)
    np.testing.assert_array_equal(d_cb2.download(), d_cb.download())
    np.testing.assert_array_equal(d_tf2.download(), d_tf.download())
    np.testing.assert_array_equal(d_out_w.download(), w_next)
    if not alias:
        np.testing.assert_array_equal(d_w.download(), w_now)
    ftpa = oracle.split_transpose(taftp, nhg, A, A, 0, F)
    ref = oracle.cb_tbtf(oracle.cb_power(ftpa, w_now, F, T, A, B, ts, 1), off, sc, T // ts)
    np.testing.assert_array_equal(d_cb2.download(), ref)


def test_cb_plan_timing_events(gpu, oracle):
    """fbf_cb_plan_set_timing: the plan records the events around the
    coherent kernel alone, inside the call's own span, on every later call
    until unset; a half-set pair is refused."""
    capi = gpu
    A, F, nhg, B, ts, S = 64, 8, 2, 512, 16, 256
    T = nhg * S
    off, sc = _levels(oracle, A, ts, 1, F)
    plan = capi.CbPlan(A, B, F, ts, 1, off, sc, nsamples_per_heap_out=T // ts)
    _, _, ibo, ibs = oracle.power_levels(16.0, 24.0, A, ts, 1, A, 16, 1)
    ib = capi.IbPlan(A, F, 16, 1, np.full(F, ibo, np.float32), np.full(F, ibs, np.float32))
    d_t = _dev(capi, gaussian_int8(2900, nhg * A * F * S * 4, 16.0))
    d_w = _dev(capi, unit_weights(2901, F * B * A))
    d_cb, d_tf = capi.DeviceBuffer(F * (T // ts) * B), capi.DeviceBuffer(ib.output_bytes(d_t.nbytes))
    s = capi.Stream()
    c0, c1, k0, k1 = capi.Event(), capi.Event(), capi.Event(), capi.Event()
    plan.set_timing(k0, k1)
    c0.record(s)
    plan.ib_beamform_taftp(ib, d_t, d_w, d_cb, d_tf, stream=s)
    c1.record(s)
    s.sync()
    kern, call, before = k0.elapsed_ms(k1), c0.elapsed_ms(c1), c0.elapsed_ms(k0)
    assert 0 < kern <= call and 0 <= before <= call - kern
    plan.set_timing(None, None)
    plan.ib_beamform_taftp(ib, d_t, d_w, d_cb, d_tf, stream=s)
    s.sync()
    assert k0.elapsed_ms(k1) == kern   # not recorded again
    with pytest.raises(capi.FbfError):
        capi.call("fbf_cb_plan_set_timing", plan.handle, k0.handle, None)


def test_cb_ib_next_weights_rejects_other_geometry(gpu, oracle):
    """A weights plan of other channels with the same byte count (half the
    channels, twice the beams) is refused before anything is launched.  (A
    plan of another antennas x beams split with the same product gives the
    same bytes: the generator works per (beam, antenna) index.)"""
    capi = gpu
    A, B, F, ts, S = 64, 256, 4, 16, 256
    off, sc = _levels(oracle, A, ts, 1, F)
    plan = capi.CbPlan(A, B, F, ts, 1, off, sc, nsamples_per_heap_out=S // ts)
    ib = capi.IbPlan(A, F, 16, 1, np.zeros(F, np.float32), np.ones(F, np.float32))
    freqs = capi.channel_frequencies_f64(1284e6, 856e6, F)
    wp_other = capi.WeightsPlan(A, 2 * B, F // 2, freqs[: F // 2])   # same bytes, other channels
    d_t = capi.DeviceBuffer(A * F * S * 4)
    d_w = capi.DeviceBuffer(F * B * A * 2)
    d_d = capi.DeviceBuffer(2 * B * A * 8)
    d_cb, d_tf = capi.DeviceBuffer(F * (S // ts) * B), capi.DeviceBuffer(ib.output_bytes(d_t.nbytes))
    with pytest.raises(capi.FbfError):
        plan.ib_beamform_taftp_next(ib, d_t, d_w, d_cb, d_tf, wp_other, d_d, 1.0, d_w)


@pytest.mark.parametrize("A,F,nhg,B,ts,ib_ts,ib_fs", [
    (12, 4, 2, 104, 16, 16, 1),     # one K step, half a slice padded, beams just past the direct path's line
    (20, 4, 2, 136, 4, 4, 1),       # two K steps, four windows a tile
    (44, 4, 2, 128, 64, 1, 1),      # three K steps
    (60, 8, 2, 400, 16, 16, 1),     # four K steps, a partial group of beams
    (68, 4, 3, 264, 16, 256, 1),    # five K steps: 64 beams per wave, the last wave with 8
    (92, 4, 1, 40, 8, 16, 4),       # six K steps, one partly filled wave
    (108, 4, 2, 256, 64, 64, 1),    # seven K steps
    (124, 4, 2, 72, 4, 8, 1),       # eight K steps, four windows a tile
    (128, 4, 2, 512, 32, 16, 2),    # eight whole K steps, two beam groups
])
def test_cb_one_pass_any_antennas(gpu, oracle, A, F, nhg, B, ts, ib_ts, ib_fs):
    """Antennas a multiple of 4 only and above 64 on the one-pass path, the
    automatic pick; and as a subset of a wider block from an antenna that is
    no multiple of 4, with a few weight components of -128."""
    _check_cb_ib(gpu, oracle, A, F, nhg, B, ts, ib_ts, ib_fs, 256, 0, True, 3100 + A + B)
    w = unit_weights(3201 + A, F * B * A).reshape(F, B, A, 2).copy()
    w[0, B - 1, A - 1, 1] = -128
    _check_taftp(gpu, oracle, A + 12, A, 5, F, nhg, B, ts, 1, 128, 0, True, 3200 + A, weights=w.reshape(-1))


@pytest.mark.parametrize("A,F,nhg,B,ts,ib_ts", [
    (16, 16, 3, 32, 16, 16),    # 32 beams per wave, one K step
    (40, 4, 2, 24, 4, 1),       # three K steps, four windows a tile, a wave with unused beams
    (64, 4, 2, 8, 64, 256),     # four K steps, one window over four tiles
    (20, 4, 2, 64, 8, 4),       # 64 beams per wave, antennas in fours
    (60, 4, 1, 40, 16, 16),
    (48, 8, 2, 96, 32, 64),     # 128 beams per wave, four time slots
    (64, 4, 2, 200, 16, 16),    # two beam groups, two time slots
    (32, 4, 2, 640, 16, 16),    # five beam groups: one to a work-group
    (128, 4, 2, 32, 16, 16),    # 64 beams per wave over eight K steps, half empty
    (76, 4, 1, 136, 4, 1),      # three beam groups in pairs
])
def test_cb_one_pass_few_beams(gpu, oracle, A, F, nhg, B, ts, ib_ts):
    """The one-pass path where few beams share their waves out over time
    slots, against the oracle."""
    _check_cb_ib(gpu, oracle, A, F, nhg, B, ts, ib_ts, 1, 256, 0, True, 3400 + A + B)


@pytest.mark.parametrize("A,B,ib_ts,ib_fs,variant", [
    (16, 32, 16, 1, 10),    # the incoherent beam in the split-transpose's pass
    (20, 64, 32, 1, 5),     # antennas in fours: the LDS-staged kernel
    (128, 32, 1, 1, 8),     # 32 beams per wave
    (40, 96, 64, 1, 10),    # windows longer than the split-transpose's tiles: a pass of its own
    (24, 40, 16, 2, 0),     # two channels to an output channel: likewise
])
def test_cb_ib_next_weights_split_transposed(gpu, oracle, A, B, ib_ts, ib_fs, variant):
    """Blocks that are split-transposed: the coherent beams, the incoherent
    beam and the next block's weights, written over this block's, of one call
    equal the oracle's beams and fbf_weights_generate."""
    capi = gpu
    from psrdada_cpp_amd import workloads as wl
    F, nhg, ts, S = 8, 2, 16, 256
    T = nhg * S
    taftp = gaussian_int8(3300 + A, nhg * A * F * S * 4, 16.0)
    off, sc = _levels(oracle, A, ts, 1, F)
    _, _, ibo, ibs = oracle.power_levels(16.0, 24.0, A, ts, 1, A, ib_ts, ib_fs)
    ioff, isc = np.full(F // ib_fs, ibo, np.float32), np.full(F // ib_fs, ibs, np.float32)
    plan = capi.CbPlan(A, B, F, ts, 1, off, sc, nsamples_per_heap_out=T // ts)
    plan.set_variant(variant)
    ib = capi.IbPlan(A, F, ib_ts, ib_fs, ioff, isc)
    assert not plan.ib_fused(ib, T, S)
    wp = capi.WeightsPlan(A, B, F, capi.channel_frequencies_f64(wl.L_BAND_CENTRE_HZ, F * wl.CHANNEL_BW_HZ, F))
    d_d = _dev(capi, wl.synth_delays(B, A, 3301, 1e-6, rate_max=1e-9))
    d_w, d_next = capi.DeviceBuffer(F * B * A * 2), capi.DeviceBuffer(F * B * A * 2)
    wp.generate(d_d, 7.5, d_w)
    wp.generate(d_d, 8.25, d_next)
    w = d_w.download()
    ftpa = oracle.split_transpose(taftp, nhg, A, A, 0, F)
    ref = oracle.cb_tbtf(oracle.cb_power(ftpa, w, F, T, A, B, ts, 1), off, sc, T // ts)
    ib_ref = oracle.ib_tf(oracle.ib_power(taftp, F, ib_ts, ib_fs, nhg, A), ioff, isc)
    d_t, d_o = _dev(capi, taftp), capi.DeviceBuffer(F * (T // ts) * B)
    d_tf = capi.DeviceBuffer(ib.output_bytes(d_t.nbytes))
    plan.ib_beamform_taftp_next(ib, d_t, d_w, d_o, d_tf, wp, d_d, 8.25, d_w)
    np.testing.assert_array_equal(d_o.download(), ref)
    np.testing.assert_array_equal(d_tf.download(), ib_ref.reshape(-1))
    np.testing.assert_array_equal(d_w.download(), d_next.download())


@pytest.mark.parametrize("A,F,nhg,B,ts,ohs,ib_ts,over,m128", [
    (16, 16, 8, 32, 16, 128, 16, "", False),     # one output heap
    (40, 4, 3, 24, 4, 16, 1, "", False),         # many output heaps, unused beams, a window per sample
    (60, 12, 2, 64, 16, 4, 2, "", False),        # 64 beams per wave, antennas in fours
    (64, 4, 3, 40, 64, 3, 8, "", False),         # windows over four tiles
    (20, 8, 2, 8, 8, 32, 4, "", True),           # a weight of -128: the exact path
    (16, 64, 8, 64, 16, 128, 16, "", False),     # the largest outputs written directly (512 KiB)
    (16, 64, 9, 64, 16, 16, 16, "", False),      # just above
    (72, 8, 2, 136, 16, 16, 4, "", False),       # more than 64 antennas: beam groups, over five K steps
    (128, 4, 2, 72, 4, 32, 16, "", False),
    (100, 8, 2, 72, 32, 16, 8, "", True),
    (16, 16, 2, 32, 16, 16, 32, "", False),      # windows longer than a tile: partials
    (16, 16, 2, 32, 16, 32, 16, "weights", False),   # next weights over this block's
    (16, 16, 2, 32, 4, 16, 16, "block", False),  # beams over the block
])
def test_small_block_outputs_in_one_launch(gpu, oracle, A, F, nhg, B, ts, ohs, ib_ts, over, m128):
    """Small blocks of few beams, whose kernel writes TBTF, the incoherent beam
    and the next weights itself (unless its outputs lie over its inputs or are
    too large): TAFTP and FTPA entry points against the oracle."""
    capi = gpu
    S = 256
    T = nhg * S
    taftp = gaussian_int8(3600 + A + B, nhg * A * F * S * 4, 16.0)
    off, sc = _levels(oracle, A, ts, 1, F)
    _, _, ibo, ibs = oracle.power_levels(16.0, 24.0, A, ts, 1, A, ib_ts, 1)
    ioff, isc = np.full(F, ibo, np.float32), np.full(F, ibs, np.float32)
    w = unit_weights(3601 + A, F * B * A).reshape(F, B, A, 2).copy()
    if m128:
        w[1, 3, 5, 1] = -128
    w = w.reshape(-1)
    ftpa = oracle.split_transpose(taftp, nhg, A, A, 0, F)
    ref = oracle.cb_tbtf(oracle.cb_power(ftpa, w, F, T, A, B, ts, 1), off, sc, ohs)
    ib_ref = oracle.ib_tf(oracle.ib_power(taftp, F, ib_ts, 1, nhg, A), ioff, isc)
    wp = capi.WeightsPlan(A, B, F, capi.channel_frequencies_f64(1284e6, 856e6, F))
    delays = np.stack([capi.synth_uniform_f32(3602, -1e-9, 1e-9, B * A),
                       capi.synth_uniform_f32(3603, -1e-6, 1e-6, B * A)], axis=1)
    d_d, d_gen = _dev(capi, delays.reshape(-1)), capi.DeviceBuffer(F * B * A * 2)
    wp.generate(d_d, 8.25, d_gen)
    plan = capi.CbPlan(A, B, F, ts, 1, off, sc, nsamples_per_heap_out=ohs)
    ib = capi.IbPlan(A, F, ib_ts, 1, ioff, isc)
    d_t, d_w, d_f = _dev(capi, taftp), _dev(capi, w), _dev(capi, ftpa)
    d_o, d_tf = capi.DeviceBuffer(F * (T // ts) * B), capi.DeviceBuffer(ib.output_bytes(d_t.nbytes))

    for call in (lambda: plan.beamform_taftp(d_t, d_w, d_o), lambda: plan.beamform(d_f, d_w, d_o)):
        d_o.fill(0x5A)
        call()
        np.testing.assert_array_equal(d_o.download(), ref)

    d_next = d_w if over == "weights" else capi.DeviceBuffer(d_gen.nbytes)
    d_out = d_t if over == "block" else d_o
    d_tf.fill(0x5A)
    plan.ib_beamform_taftp_next(ib, d_t, d_w, _View(d_out.ptr, d_o.nbytes), d_tf, wp, d_d, 8.25, d_next)
    np.testing.assert_array_equal(d_out.download(count=ref.size), ref)
    np.testing.assert_array_equal(d_tf.download(), ib_ref.reshape(-1))
    np.testing.assert_array_equal(d_next.download(), d_gen.download())


class _View:
    def __init__(self, ptr, nbytes):
        self.ptr, self.nbytes = ptr, nbytes


def _captured(capi, stream, call):
    """The call captured into an executable graph; returns its launcher."""
    import ctypes as C
    hip = capi.lib()   # (finds the HIP runtime's functions through its dependencies)
    graph, execg = C.c_void_p(), C.c_void_p()
    assert hip.hipStreamBeginCapture(stream.handle, 1) == 0
    try:
        call()
    finally:
        e = hip.hipStreamEndCapture(stream.handle, C.byref(graph))
    assert e == 0 and hip.hipGraphInstantiate(C.byref(execg), graph, None, None, C.c_size_t(0)) == 0
    return lambda: hip.hipGraphLaunch(execg, stream.handle)


@pytest.mark.parametrize("warm,captured,Atot,A,a0,F,nhg,nhg_warm,B,ts", [
    ("ftpa", "ftpa over the block", 16, 16, 0, 4, 2, 2, 32, 4),   # first in one launch, then staged
    ("taftp", "both", 40, 40, 0, 4, 2, 2, 136, 16),               # the incoherent beam on its own
    ("taftp", "both", 16, 16, 0, 16, 3, 3, 32, 16),
    ("both", "taftp", 72, 72, 0, 4, 4, 4, 16, 16),                # small blocks that are split-transposed
    ("taftp", "taftp", 24, 16, 5, 4, 2, 6, 40, 16),               # after a larger block that was not
    ("taftp", "both", 44, 44, 0, 4, 2, 6, 64, 8),
])
def test_calls_captured_after_other_calls(gpu, oracle, warm, captured, Atot, A, a0, F, nhg, nhg_warm, B, ts):
    """A call that is captured uses the scratch that other calls of its plan
    have left: one call runs eagerly, another is captured on a block of at most
    that size and replayed on new voltages, against the oracle."""
    capi = gpu
    S = 256
    off, sc = _levels(oracle, A, ts, 1, F)
    _, _, ibo, ibs = oracle.power_levels(16.0, 24.0, 8, ts, 1, Atot, 16, 1)
    ioff, isc = np.full(F, ibo, np.float32), np.full(F, ibs, np.float32)
    plan = capi.CbPlan(A, B, F, ts, 1, off, sc, nsamples_per_heap_out=S // ts)
    ib = capi.IbPlan(Atot, F, 16, 1, ioff, isc)
    w = unit_weights(3800 + A, F * B * A)
    d_w = _dev(capi, w)
    s = capi.Stream()

    def call(name, d_t, d_o, d_tf):
        if name == "both":
            plan.ib_beamform_taftp(ib, d_t, d_w, d_o, d_tf, stream=s)
        elif name == "taftp":
            plan.beamform_taftp(d_t, d_w, d_o, nantennas_total=Atot, start_antenna=a0, stream=s)
        else:
            plan.beamform(d_t, d_w, d_o, stream=s)

    def buffers(n):
        return (capi.DeviceBuffer(n * Atot * F * S * 4), capi.DeviceBuffer(F * (n * S // ts) * B),
                capi.DeviceBuffer(F * n * 16))

    bufs = buffers(nhg_warm)
    bufs[0].fill(1, s)
    call(warm, *bufs)
    s.sync()
    d_t, d_o, d_tf = buffers(nhg)
    d_out = _View(d_t.ptr, d_o.nbytes) if captured.endswith("block") else d_o
    replay = _captured(capi, s, lambda: call(captured.split()[0], d_t, d_out, d_tf))
    T = nhg * S
    for rep in range(3):
        taftp = gaussian_int8(3801 + rep, nhg * Atot * F * S * 4, 16.0)
        ftpa = oracle.split_transpose(taftp, nhg, Atot, A, a0, F)
        d_t.upload(ftpa if captured.startswith("ftpa") else taftp, s)
        d_o.fill(0x5A, s)
        d_tf.fill(0x5A, s)
        s.sync()
        assert replay() == 0
        s.sync()
        ref = oracle.cb_tbtf(oracle.cb_power(ftpa, w, F, T, A, B, ts, 1), off, sc, S // ts)
        got = (d_t if captured.endswith("block") else d_o).download(count=ref.size)
        np.testing.assert_array_equal(got, ref, err_msg=f"replay {rep}")
        if captured == "both":
            np.testing.assert_array_equal(d_tf.download(),
                                          oracle.ib_tf(oracle.ib_power(taftp, F, 16, 1, nhg, Atot), ioff, isc))


@pytest.mark.parametrize("A,F,nhg,B,ts,ib_ts,m128", [
    (48, 4, 4, 96, 256, 16, False),    # long windows, waves of 32 beams in three groups
    (60, 4, 3, 136, 64, 256, False),   # five groups of 32, the last with 8
    (16, 4, 2, 72, 32, 1, True),       # a weight of -128
    (20, 8, 2, 136, 16, 16, False),    # waves of 64 beams in three groups
    (40, 4, 1, 96, 4, 4, True),
    (12, 64, 4, 192, 16, 16, False),   # the most that run in two rounds
    (12, 64, 4, 200, 16, 16, False),   # just above: 128 beams
    (12, 64, 8, 192, 32, 16, False),   # 32 beams would not fit in one round: 64
])
def test_small_blocks_of_narrow_waves(gpu, oracle, A, F, nhg, B, ts, ib_ts, m128):
    """Small blocks of more than 64 beams on waves of 32 and 64: both beams from
    TAFTP, a subset of a wider block and FTPA, against the oracle."""
    capi = gpu
    w = unit_weights(3901 + A, F * B * A).reshape(F, B, A, 2).copy()
    if m128:
        w[1, B - 1, 5, 1] = -128
    w = w.reshape(-1)
    _check_cb_ib(capi, oracle, A, F, nhg, B, ts, ib_ts, 1, 256, 0, True, 3900 + A, weights=w)
    T = nhg * 256
    off, sc = _levels(oracle, A, ts, 1, F)
    plan = capi.CbPlan(A, B, F, ts, 1, off, sc, nsamples_per_heap_out=T // ts)
    taftp = gaussian_int8(3902 + A, nhg * (A + 8) * F * 256 * 4, 16.0)
    ftpa = oracle.split_transpose(taftp, nhg, A + 8, A, 3, F)
    ref = oracle.cb_tbtf(oracle.cb_power(ftpa, w, F, T, A, B, ts, 1), off, sc, T // ts)
    d_w, d_o = _dev(capi, w), capi.DeviceBuffer(ref.size)
    for call in (lambda: plan.beamform_taftp(_dev(capi, taftp), d_w, d_o, nantennas_total=A + 8, start_antenna=3),
                 lambda: plan.beamform(_dev(capi, ftpa), d_w, d_o)):
        d_o.fill(0x5A)
        call()
        np.testing.assert_array_equal(d_o.download(), ref)


@pytest.mark.parametrize("A,B,F,T,ts,fs,m128", [
    (64, 104, 2, 64, 32, 2, False),       # two windows, a ragged beam group
    (64, 264, 6, 512, 256, 2, True),      # one pass of long windows, a weight of -128
    (44, 168, 4, 768, 16, 2, False),      # 4 antennas past a multiple of 8
    (52, 104, 2, 4352, 16, 2, False),     # passes over six groups, the last with two
    (20, 400, 8, 256, 64, 4, False),      # four channels to a sum
    (32, 136, 4, 128, 128, 4, True),      # one window
    (28, 1032, 4, 1344, 16, 4, False),    # 33 x 7 work-groups, one round
    (28, 1032, 4, 1360, 16, 4, False),    # 33 x 8, more than one: 128 beams a wave
    (64, 1024, 32, 96, 16, 2, False),     # 16 x 16 = 256 work-groups
    (64, 1032, 32, 96, 16, 2, False),     # 16 x 17: 128 beams a wave
])
def test_small_blocks_of_summed_channels(gpu, oracle, A, B, F, T, ts, fs, m128):
    """Small blocks with channels summed over and more than 96 beams (32 beams per
    wave, three time slots to a work-group) in FTPA and as a subarray of a wider
    FTPA block, 4 antennas in, against the oracle."""
    capi = gpu
    w = unit_weights(4101 + A, F * B * A).reshape(F, B, A, 2).copy()
    if m128:
        w[1, B - 1, 5, 1] = -128
    w = w.reshape(-1)
    off, sc = _levels(oracle, A, ts, fs, F)
    plan = capi.CbPlan(A, B, F, ts, fs, off, sc, nsamples_per_heap_out=T // ts)
    wide = gaussian_int8(4102 + A, F * T * 2 * (A + 8) * 2, 16.0).reshape(F, 2 * T, A + 8, 2)
    ftpa = np.ascontiguousarray(wide[:, :, 4:4 + A]).reshape(-1)
    ref = oracle.cb_tbtf(oracle.cb_power(ftpa, w, F, T, A, B, ts, fs), off, sc, T // ts)
    d_w, d_o = _dev(capi, w), capi.DeviceBuffer(ref.size)
    for call in (lambda: plan.beamform(_dev(capi, ftpa), d_w, d_o),
                 lambda: plan.beamform_subarray(_dev(capi, wide.reshape(-1)), A + 8, 4, d_w, d_o)):
        d_o.fill(0x5A)
        call()
        np.testing.assert_array_equal(d_o.download(), ref)
