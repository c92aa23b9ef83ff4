"""The beamformer's work as a user's program calls it, for timing and comparison.

Every case names one call of the public Python binding (``psrdada_cpp_amd.capi``)
on device buffers: the buffers here are torch tensors, whose addresses go
through the C ABI as any device pointer does.  A case is a dict of plain
values; ``kind`` says which call it is:

  block     both beams of one TAFTP block and the next block's weights
            (``CbPlan.ib_beamform_taftp_next``), the step of a running pipeline
  taftp     coherent beams of an antenna subset of a TAFTP block
            (``CbPlan.beamform_taftp``)
  ftpa      coherent beams of split-transposed voltages (``CbPlan.beamform``)
  batch     several subarrays of one block and its incoherent beam
            (``Batch.run`` with its graph)
  split     split-transpose of an antenna subset (``split_transpose``)
  ib        incoherent beam (``IbPlan.beamform``)
  weights   weights of a delay model (``WeightsPlan.generate``)
  tuse      beam corner turn after the beamformer (``tuse_transpose``)
  feng      F-engine heap reorder before it (``feng_to_dada``)

Voltages are rounded, clamped Gaussians and weights unit phasors at int8
amplitude 127, as the beamformer meets them; moved bytes are uniformly random.
"""
from __future__ import annotations

import ctypes
import math

import numpy as np
import torch

from psrdada_cpp_amd import capi

SAMPLES_PER_HEAP = 256
INPUT_LEVEL = 16.0       # sigma of the voltages' re and im
OUTPUT_LEVEL = 24.0      # sigma of the quantised beams
BAND_CENTRE_HZ = 1284e6
CHANNEL_BW_HZ = 1712e6 / 8192
TAU_MAX_S = 2e-6
RATE_MAX = 1e-9
OUTPUT_HEAP_BYTES = 8192
COHERENT_MAX = 64 * 8192 * 128 * 1024    # channels x samples x antennas x beams of the largest listed case
MOVED_MAX = 1 << 28                      # bytes of a block that is only moved


def listed():
    return [
        # A small array's block: 16 antennas, 16 channels, 2048 spectra.  Launches and latency are most of it.
        dict(name="block_16ant_32beams", kind="block", antennas=16, chans=16, heaps=8, beams=32, ts=16, fs=1,
             ib_ts=16),
        # The full array of 64 antennas with 512 beams, the repository's headline block.
        dict(name="block_64ant_512beams", kind="block", antennas=64, chans=64, heaps=32, beams=512, ts=16, fs=1,
             ib_ts=16),
        # The array with some antennas out: no multiple of 8, and beams that fill no whole group.
        dict(name="block_60ant_400beams", kind="block", antennas=60, chans=64, heaps=16, beams=400, ts=16, fs=1,
             ib_ts=16),
        # The widest array that the coherent beamformer takes, with twice the headline's beams.
        dict(name="block_128ant_1024beams", kind="block", antennas=128, chans=64, heaps=32, beams=1024, ts=16, fs=1,
             ib_ts=16),
        # A subarray beamformed straight from the full array's block, long integrations.
        dict(name="taftp_40of64_768beams", kind="taftp", total=64, antennas=40, start=0, chans=64, heaps=32,
             beams=768, ts=64, fs=1),
        # The coherent operator on its own at the antennas, beams and scrunch of the reference's test.
        dict(name="ftpa_44ant_1024beams_fs4", kind="ftpa", antennas=44, chans=64, samples=8192, beams=1024, ts=16,
             fs=4),
        # One block shared by three subarrays of uneven sizes, in one graph launch.
        dict(name="batch_40_16_8", kind="batch", chans=64, heaps=32, antennas="40,16,8", beams="768,256,64", ts=16),
        # The split-transpose operator at the reference's default geometry, 44 of 64 antennas.
        dict(name="split_44of64", kind="split", total=64, antennas=44, start=0, chans=64, heaps=12),
        # The incoherent operator on its own, two channels to an output channel.
        dict(name="ib_64ant_fs2", kind="ib", antennas=64, chans=64, heaps=32, ts=16, fs=2),
        # New weights for every beam after a delay update.
        dict(name="weights_64ant_1024beams", kind="weights", antennas=64, beams=1024, chans=64),
        # The reference's default corner turn: 128 channels, 64 samples, 32 bands, 10 groups.
        dict(name="tuse_64beams", kind="tuse", chans=128, samples=64, bands=32, beams=64, groups=10),
        # A wide-band F-engine's heaps of 4096 channels.
        dict(name="feng_4096ch", kind="feng", chans=4096, stamps=16),
    ]


def _log(rng, lo, hi):
    """A whole number in [lo, hi], spread over the logarithm."""
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def _log_of(rng, step, lo, hi):
    """A multiple of step in [lo, hi], spread over the logarithm."""
    return max(lo, min(hi, step * max(1, int(round(_log(rng, lo, hi) / step)))))


def draw(rng):
    kind = rng.choice(["block", "block", "block", "taftp", "taftp", "ftpa", "ftpa", "batch", "split", "ib",
                       "weights", "tuse", "feng"])
    if kind in ("block", "taftp", "ftpa"):
        while True:
            antennas = rng.choice([_log_of(rng, 4, 8, 128), 8 * rng.randint(1, 16)])
            chans = _log_of(rng, 4, 4, 128)
            heaps = _log(rng, 1, 48)
            beams = _log_of(rng, 8, 8, 1024)
            # At most half the largest listed case's work: not every geometry runs at its rate.
            inputs = chans * heaps * SAMPLES_PER_HEAP * antennas
            if 4 * inputs <= MOVED_MAX and 2 * inputs * beams <= COHERENT_MAX:
                break
        ts = rng.choice([4, 8, 16, 16, 32, 64])
        c = dict(kind=kind, antennas=antennas, chans=chans, beams=beams, ts=ts, fs=1)
        if kind == "ftpa":
            c["fs"] = rng.choice([1, 1, 2, 4])
            c["ts"] = ts = rng.choice([ts, ts, ts, 1, 2, 3, 10, 24])
            c["samples"] = ts * max(1, heaps * SAMPLES_PER_HEAP // ts)
        elif kind == "taftp":
            c["total"] = antennas + rng.choice([0, 4, 8, 24, 64])
            c["start"] = rng.randint(0, (c["total"] - antennas) // 4) * 4
            c["heaps"] = heaps
        else:
            c["heaps"] = heaps
            c["ib_ts"] = rng.choice([4, 16, 16, 64])
        return c
    if kind == "batch":
        cut = sorted(rng.sample(range(1, 8), rng.choice([1, 2, 3])))
        sizes = [8 * (b - a) for a, b in zip([0] + cut, cut + [8])]
        return dict(kind=kind, chans=_log_of(rng, 4, 8, 64), heaps=_log(rng, 1, 32),
                    antennas=",".join(str(a) for a in sizes),
                    beams=",".join(str(_log_of(rng, 8, 16, 12 * a)) for a in sizes), ts=rng.choice([4, 16, 64]))
    if kind == "split":
        total = _log(rng, 8, 128)
        antennas = rng.randint(max(1, total // 8), total)
        chans = _log(rng, 4, 128)
        heaps = _log(rng, 1, max(1, min(48, MOVED_MAX // 2 // (1024 * total * chans))))
        return dict(kind=kind, total=total, antennas=antennas, start=rng.randint(0, total - antennas), chans=chans,
                    heaps=heaps)
    if kind == "ib":
        fs = rng.choice([1, 1, 2, 4, 8])
        antennas = _log(rng, 4, 128)
        chans = _log_of(rng, max(4, fs), max(4, fs), 128)
        heaps = _log(rng, 1, max(1, min(48, MOVED_MAX // 2 // (1024 * antennas * chans))))
        return dict(kind=kind, antennas=antennas, chans=chans, heaps=heaps, ts=rng.choice([1, 4, 16, 16, 64, 256]),
                    fs=fs)
    if kind == "weights":
        return dict(kind=kind, antennas=_log(rng, 4, 128), beams=_log(rng, 8, 1024), chans=_log(rng, 1, 128))
    if kind == "tuse":
        chans = rng.choice([1 << rng.randint(2, 8), 4 * rng.randint(1, 64), _log(rng, 1, 256)])
        samples, bands, groups = _log(rng, 16, 512), _log(rng, 1, 64), rng.randint(1, 10)
        most = MOVED_MAX // 2 if chans % 4 == 0 else MOVED_MAX // 8
        beams = _log(rng, 1, max(1, min(1024, most // (chans * samples * bands * groups))))
        return dict(kind=kind, chans=chans, samples=samples, bands=bands, beams=beams, groups=groups)
    chans = rng.choice([1 << rng.randint(4, 12), _log(rng, 8, 4096)])
    return dict(kind=kind, chans=chans, stamps=_log(rng, 1, max(1, min(1024, MOVED_MAX // 2 // (1024 * chans)))))


# ---------------------------------------------------------------------------
# Inputs and sizes
# ---------------------------------------------------------------------------
class _Buf:
    """A torch tensor's memory as the binding's calls take it."""

    def __init__(self, tensor):
        self.tensor = tensor
        self.nbytes = tensor.numel() * tensor.element_size()
        self.ptr = ctypes.c_void_p(tensor.data_ptr())


def _gen(seed):
    return torch.Generator(device="cuda").manual_seed(int(seed))


def _voltages(gen, nbytes):
    out = torch.empty(nbytes, dtype=torch.int8, device="cuda")
    step = 1 << 26
    for i in range(0, nbytes, step):
        n = min(step, nbytes - i)
        out[i:i + n] = (torch.randn(n, device="cuda", generator=gen) * INPUT_LEVEL).round_().clamp_(-127, 127)
    return out


def _weights(gen, chans, beams, antennas):
    """FBA [chans][beams][antennas][re, im]."""
    th = torch.rand((chans, beams, antennas), device="cuda", generator=gen) * (2 * math.pi)
    return torch.stack(((127 * th.cos()).round_(), (127 * th.sin()).round_()), dim=-1).to(torch.int8)


def _bytes(gen, nbytes):
    return torch.randint(-128, 128, (nbytes,), dtype=torch.int8, device="cuda", generator=gen)


def _delays(gen, beams, antennas):
    """[beams][antennas][rate, offset] float32."""
    u = torch.rand((beams, antennas, 2), device="cuda", generator=gen) * 2 - 1
    return (u * torch.tensor([RATE_MAX, TAU_MAX_S], device="cuda")).contiguous()


def _epoch(seed):
    return float(seed % 600) + 0.25


def _freqs(chans):
    return BAND_CENTRE_HZ + CHANNEL_BW_HZ * (np.arange(chans) - 0.5 * (chans - 1))


def _cb_level(antennas, ts, fs):
    """Offset and scale of a coherent output channel's detected power."""
    s, dof = (127.0 * INPUT_LEVEL) ** 2 * antennas, 4.0 * ts * fs
    return np.float32(s * dof), np.float32(s * math.sqrt(2 * dof) / OUTPUT_LEVEL)


def _ib_level(antennas, ts, fs):
    s, dof = INPUT_LEVEL ** 2, 4.0 * ts * fs * antennas
    return np.float32(s * dof), np.float32(s * math.sqrt(2 * dof) / OUTPUT_LEVEL)


def _full(n, level):
    return np.full(n, level[0], np.float32), np.full(n, level[1], np.float32)


def _samples(case):
    return case["samples"] if case["kind"] == "ftpa" else case["heaps"] * SAMPLES_PER_HEAP


def _ohs(case, fs=1):
    """Output samples per heap: the largest count within an 8 KiB heap that the block fills whole."""
    return math.gcd(_samples(case) // case["ts"], max(1, OUTPUT_HEAP_BYTES // (case["chans"] // fs)))


def _subs(case):
    """(start, antennas, beams) of a batch's subarrays."""
    start, out = 0, []
    for a, b in zip(case["antennas"].split(","), case["beams"].split(",")):
        out.append((start, int(a), int(b)))
        start += int(a)
    return out


def _empty(nbytes):
    return _Buf(torch.empty(nbytes, dtype=torch.int8, device="cuda"))


_streams = []


def _stream():
    """The program's processing stream: blocks are taken one after the other, as a pipeline takes them."""
    if not _streams:
        _streams.append(capi.Stream())
    return _streams[0]


def prepare(case, seed):
    gen, kind = _gen(seed), case["kind"]
    st = {"kind": kind, "case": case, "stream": _stream()}
    if kind in ("block", "taftp", "ftpa"):
        A, F, B, ts, fs, T = case["antennas"], case["chans"], case["beams"], case["ts"], case["fs"], _samples(case)
        total = case.get("total", A)
        st["volts"] = _Buf(_voltages(gen, 4 * total * F * T))
        st["weights"] = _Buf(_weights(gen, F, B, A))
        st["cb"] = capi.CbPlan(A, B, F, ts, fs, *_full(F // fs, _cb_level(A, ts, fs)),
                               nsamples_per_heap_out=_ohs(case, fs))
        st["out"] = _empty(T // ts * B * (F // fs))
        if kind == "block":
            its = case["ib_ts"]
            st["ib"] = capi.IbPlan(A, F, its, 1, *_full(F, _ib_level(A, its, 1)))
            st["tf"] = _empty(T // its * F)
            st["wplan"] = capi.WeightsPlan(A, B, F, _freqs(F))
            st["delays"] = _Buf(_delays(gen, B, A))
            st["epoch"] = _epoch(seed)
            st["next"] = _empty(2 * A * B * F)
    elif kind == "batch":
        F, T, ts = case["chans"], _samples(case), case["ts"]
        subs = _subs(case)
        total = sum(a for _, a, _ in subs)
        st["volts"] = _Buf(_voltages(gen, 4 * total * F * T))
        st["weights"] = [_Buf(_weights(gen, F, b, a)) for _, a, b in subs]
        st["batch"] = capi.Batch(total, F, case["heaps"],
                                 [dict(start_antenna=s, nantennas=a, nbeams=b, tscrunch=ts, fscrunch=1,
                                       nsamples_per_heap_out=_ohs(case)) for s, a, b in subs],
                                 [_full(F, _cb_level(a, ts, 1)) for _, a, _ in subs])
        st["batch"].enable_ib(16, 1, *_full(F, _ib_level(total, 16, 1)))
        st["out"] = [_empty(T // ts * b * F) for _, _, b in subs] + [_empty(T // 16 * F)]
    elif kind == "split":
        n = 4 * case["chans"] * case["heaps"] * SAMPLES_PER_HEAP
        st["volts"] = _Buf(_voltages(gen, n * case["total"]))
        st["out"] = _empty(n * case["antennas"])
    elif kind == "ib":
        A, F, ts, fs, T = case["antennas"], case["chans"], case["ts"], case["fs"], _samples(case)
        st["volts"] = _Buf(_voltages(gen, 4 * A * F * T))
        st["ib"] = capi.IbPlan(A, F, ts, fs, *_full(F // fs, _ib_level(A, ts, fs)))
        st["out"] = _empty(T // ts * (F // fs))
    elif kind == "weights":
        A, F, B = case["antennas"], case["chans"], case["beams"]
        st["wplan"] = capi.WeightsPlan(A, B, F, _freqs(F))
        st["delays"] = _Buf(_delays(gen, B, A))
        st["epoch"] = _epoch(seed)
        st["out"] = _empty(2 * A * B * F)
    elif kind == "tuse":
        n = case["chans"] * case["samples"] * case["bands"] * case["beams"] * case["groups"]
        st["volts"], st["out"] = _Buf(_bytes(gen, n)), _empty(n)
    elif kind == "feng":
        n = case["chans"] * 1024 * case["stamps"]
        st["volts"], st["out"] = _Buf(_bytes(gen, n)), _empty(n)
    else:
        raise ValueError(f"unknown kind {kind!r}")
    torch.cuda.synchronize()     # the inputs are made on torch's stream
    return st


def run(st):
    kind, case, s = st["kind"], st["case"], st["stream"]
    if kind == "block":
        st["cb"].ib_beamform_taftp_next(st["ib"], st["volts"], st["weights"], st["out"], st["tf"], st["wplan"],
                                        st["delays"], st["epoch"], st["next"], stream=s)
        return {"beams": st["out"].tensor, "incoherent": st["tf"].tensor, "next_weights": st["next"].tensor}
    if kind == "taftp":
        st["cb"].beamform_taftp(st["volts"], st["weights"], st["out"], nantennas_total=case["total"],
                                start_antenna=case["start"], stream=s)
    elif kind == "ftpa":
        st["cb"].beamform(st["volts"], st["weights"], st["out"], stream=s)
    elif kind == "batch":
        st["batch"].run(st["volts"], st["weights"], st["out"], use_graph=True, stream=s)
        return {"beams": [o.tensor for o in st["out"][:-1]], "incoherent": st["out"][-1].tensor}
    elif kind == "split":
        capi.split_transpose(st["volts"], st["out"], case["total"], case["antennas"], case["start"], case["chans"],
                             stream=s)
    elif kind == "ib":
        st["ib"].beamform(st["volts"], st["out"], stream=s)
    elif kind == "weights":
        st["wplan"].generate(st["delays"], st["epoch"], st["out"], stream=s)
    elif kind == "tuse":
        capi.tuse_transpose(st["volts"], st["out"], case["chans"], case["samples"], case["bands"], case["beams"],
                            case["groups"], stream=s)
    else:
        capi.feng_to_dada(st["volts"], st["out"], case["chans"], stream=s)
    return st["out"].tensor


def work(case):
    kind = case["kind"]
    if kind in ("block", "taftp", "ftpa"):
        A, F, B, T = case["antennas"], case["chans"], case["beams"], _samples(case)
        b = 4 * A * F * T + 2 * A * F * B + T // case["ts"] * B * (F // case["fs"])
        if kind == "block":
            b += T // case["ib_ts"] * F + 8 * A * B + 2 * A * F * B
        return {"bytes": b, "flops": 16 * F * T * A * B}
    if kind == "batch":
        F, T, subs = case["chans"], _samples(case), _subs(case)
        total = sum(a for _, a, _ in subs)
        b = 4 * total * F * T + T // 16 * F + sum(2 * F * a * b + T // case["ts"] * b * F for _, a, b in subs)
        return {"bytes": b, "flops": sum(16 * F * T * a * b for _, a, b in subs)}
    if kind == "split":
        return {"bytes": 8 * case["antennas"] * case["chans"] * _samples(case), "flops": 0}
    if kind == "ib":
        n = case["antennas"] * case["chans"] * _samples(case)
        return {"bytes": 4 * n + _samples(case) // case["ts"] * (case["chans"] // case["fs"]), "flops": 8 * n}
    if kind == "weights":
        n = case["antennas"] * case["beams"]
        return {"bytes": 8 * n + 2 * n * case["chans"], "flops": 0}
    if kind == "tuse":
        return {"bytes": 2 * case["chans"] * case["samples"] * case["bands"] * case["beams"] * case["groups"],
                "flops": 0}
    return {"bytes": 2048 * case["chans"] * case["stamps"], "flops": 0}


# ---------------------------------------------------------------------------
# The same in 64 bits
# ---------------------------------------------------------------------------
def _quantise(power, level):
    v = (power - float(level[0])) / float(level[1])
    return (torch.sign(v) * torch.floor(v.abs() + 0.5)).clamp_(-128, 127).to(torch.int64)


def _aftp(volts, total, F, heaps):
    return volts.reshape(heaps, total, F, SAMPLES_PER_HEAP, 2, 2)


def _ftpa(volts, total, start, A, F, heaps):
    v = _aftp(volts, total, F, heaps)[:, start:start + A]
    return v.permute(2, 0, 3, 4, 1, 5).reshape(F, heaps * SAMPLES_PER_HEAP, 2, A, 2)


def _coherent(ftpa, weights, ts, fs, ohs):
    """FTPA [F][T][2][A][2] and FBA [F][B][A][2] to TBTF in 64 bits."""
    F, T, _, A, _ = ftpa.shape
    B, Fo, To = weights.shape[1], F // fs, T // ts
    out = torch.empty((To // ohs, B, ohs, Fo), dtype=torch.int64, device="cuda")
    for fo in range(Fo):
        power = torch.zeros((To, B), dtype=torch.float64, device="cuda")
        for f in range(fo * fs, fo * fs + fs):
            v, w = ftpa[f].reshape(T * 2, A, 2).double(), weights[f].double()
            vr, vi = v[..., 0].contiguous(), v[..., 1].contiguous()
            wr, wi = w[..., 0].t().contiguous(), w[..., 1].t().contiguous()
            re = vr @ wr - vi @ wi
            im = vi @ wr + vr @ wi
            power += (re * re + im * im).reshape(To, ts * 2, B).sum(1)
        out[..., fo] = _quantise(power, _cb_level(A, ts, fs)).reshape(To // ohs, ohs, B).permute(0, 2, 1)
    return out.reshape(-1)


def _incoherent(volts, A, F, heaps, ts, fs):
    """TAFTP to TF in 64 bits."""
    out = torch.empty((heaps * SAMPLES_PER_HEAP // ts, F // fs), dtype=torch.int64, device="cuda")
    n = SAMPLES_PER_HEAP // ts
    for hg, block in enumerate(_aftp(volts, A, F, heaps)):
        p = block.to(torch.int32).square().sum((0, 3, 4), dtype=torch.int64)     # [F][256]
        p = p.reshape(F // fs, fs, n, ts).sum((1, 3))
        out[hg * n:(hg + 1) * n] = _quantise(p.double(), _ib_level(A, ts, fs)).t()
    return out.reshape(-1)


def _phasors(delays, freqs, epoch):
    """[F][B][A][re, im] in 64 bits."""
    d = delays.double()
    tau = d[..., 0] * epoch + d[..., 1]
    out = []
    for f in freqs:
        x = tau * float(f)
        x = (x - torch.round(x)) * (2 * math.pi)
        out.append(torch.stack((torch.round(127 * x.cos()), torch.round(127 * x.sin())), dim=-1).to(torch.int64))
    return torch.stack(out).reshape(-1)


def exact(case, seed):
    gen, kind = _gen(seed), case["kind"]
    if kind in ("block", "taftp", "ftpa"):
        A, F, B, ts, fs, T = case["antennas"], case["chans"], case["beams"], case["ts"], case["fs"], _samples(case)
        total = case.get("total", A)
        volts = _voltages(gen, 4 * total * F * T)
        weights = _weights(gen, F, B, A)
        ftpa = (volts.reshape(F, T, 2, A, 2) if kind == "ftpa"
                else _ftpa(volts, total, case.get("start", 0), A, F, case["heaps"]))
        beams = _coherent(ftpa, weights, ts, fs, _ohs(case, fs))
        if kind != "block":
            return beams
        return {"beams": beams, "incoherent": _incoherent(volts, A, F, case["heaps"], case["ib_ts"], 1),
                "next_weights": _phasors(_delays(gen, B, A), _freqs(F), _epoch(seed))}
    if kind == "batch":
        F, T, subs = case["chans"], _samples(case), _subs(case)
        total = sum(a for _, a, _ in subs)
        volts = _voltages(gen, 4 * total * F * T)
        weights = [_weights(gen, F, b, a) for _, a, b in subs]
        return {"beams": [_coherent(_ftpa(volts, total, s, a, F, case["heaps"]), w, case["ts"], 1, _ohs(case))
                          for (s, a, _), w in zip(subs, weights)],
                "incoherent": _incoherent(volts, total, F, case["heaps"], 16, 1)}
    if kind == "split":
        volts = _voltages(gen, 4 * case["chans"] * case["heaps"] * SAMPLES_PER_HEAP * case["total"])
        return _ftpa(volts, case["total"], case["start"], case["antennas"], case["chans"], case["heaps"]).reshape(-1)
    if kind == "ib":
        volts = _voltages(gen, 4 * case["antennas"] * case["chans"] * _samples(case))
        return _incoherent(volts, case["antennas"], case["chans"], case["heaps"], case["ts"], case["fs"])
    if kind == "weights":
        return _phasors(_delays(gen, case["beams"], case["antennas"]), _freqs(case["chans"]), _epoch(seed))
    if kind == "tuse":
        C, S, F, B, G = (case[k] for k in ("chans", "samples", "bands", "beams", "groups"))
        return _bytes(gen, C * S * F * B * G).reshape(G, B, F, S, C).permute(1, 0, 3, 2, 4).reshape(-1)
    w = _bytes(gen, case["chans"] * 1024 * case["stamps"]).reshape(case["stamps"], case["chans"], 256, 4)
    return w.permute(0, 2, 1, 3).reshape(-1)
