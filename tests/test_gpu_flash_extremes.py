"""The small-launch flash kernels (csrc/kernels/flash_w.h) on scores far below
the running max the .ph sources start from (-65504 for f16, -3e8 for f32):
each key group starts its own softmax, so a block of such scores may be a
group's first.  Held to a plain f64 softmax by the kernels' bounds (2e-2 for
f16, 1e-4 for f32), each entry launched by itself and through the built-in
plan."""
import ctypes
import os

import numpy as np
import pytest

import oracle
from test_gpu_flash_small import D, ENTRIES, FILES, TOL, _Heads, _inputs, _launch

pytestmark = pytest.mark.gpu

STEP = {"flash_w4": {16: 64, 32: 32}, "flash_w2x4": {16: 64}, "flash_w8": {32: 32}}
GROUPS = {"flash_w4": 4, "flash_w2x4": 4, "flash_w8": 8}


def _softmax(q, k, v, scale):
    """f64 attention of every head; a key whose score is -inf has no weight."""
    with np.errstate(invalid="ignore"):
        s = scale * (q.astype(np.float64) @ k.astype(np.float64).transpose(0, 2, 1))
    p = np.exp(s - s.max(axis=-1, keepdims=True))
    return (p / p.sum(axis=-1, keepdims=True)) @ v.astype(np.float64)


class _Entry:
    """One small-launch entry over dense heads, launched with its own grid."""

    def __init__(self, px, stream, bits, entry, q, k, v, scale):
        self.px, self.stream, self.bits, self.scale = px, stream, bits, scale
        _, self.qb, self.threads = next(e for e in ENTRIES[bits] if e[0] == entry)
        with open(os.path.join(px.LIB_DIR, FILES[bits]), "rb") as f:
            self.mod = px.module_load_data(f.read())
        self.fn = px.module_get_function(self.mod, entry)
        self.combine = px.module_get_function(self.mod, "flash_combine")
        self.BH, self.Nq, self.Nk = q.shape[0], q.shape[1], k.shape[1]
        self.ops = [_Heads(px, bits, t) for t in (q, k, v)]

    def run(self, sp):
        px = self.px
        nkb = -(-self.Nk // 64)
        chunk = -(-nkb // min(sp, nkb)) * 64
        sp = -(-self.Nk // chunk)
        do = _Heads(px, self.bits, np.zeros((self.BH, self.Nq, D), np.float32))
        ws = px.DeviceBuffer(sp * self.BH * self.Nq * (D + 2) * 4)
        i64, u64 = ctypes.c_int64, ctypes.c_uint64
        ts = self.ops + [do]
        vals = [u64(t.buf.ptr) for t in ts] + [u64(ws.ptr)]
        vals += [i64(x) for x in [self.BH, self.Nq, self.Nk] + [t.ld for t in ts] +
                 [t.hs for t in ts] + [chunk]]
        vals += [ctypes.c_int32(sp), ctypes.c_float(self.scale)]
        _launch(px, self.stream, self.fn, (-(-self.Nq // self.qb) * self.BH, sp, 1), self.threads,
                vals)
        if sp > 1:
            vals = [u64(ws.ptr), ctypes.c_int32(sp), u64(do.buf.ptr)]
            vals += [i64(x) for x in (self.BH, self.Nq, do.ld, do.hs)]
            _launch(px, self.stream, self.combine, (-(-self.BH * self.Nq * 16 // 256), 1, 1), 256,
                    vals)
        self.stream.synchronize()
        return do.get()

    def close(self):
        self.px.module_unload(self.mod)


def _rel(got, want):
    return (np.abs(got - want) / np.maximum(np.abs(want), 0.1)).max()


def _all_entries():
    return [(bits, e[0]) for bits in (16, 32) for e in ENTRIES[bits]]


@pytest.mark.parametrize("low", ["finite", "-inf"])
@pytest.mark.parametrize("bits,entry", _all_entries())
def test_a_key_group_starts_on_a_padded_block(px_gpu, stream, bits, entry, low):
    # padding keys score -8e5 (f16) or -1e11 (f32), or -inf, for every query;
    # in turn each group's first block is all padding, then all but one
    # group's first blocks are, and (Nk a block longer) a later block too
    px, step, kg = px_gpu, STEP[entry][bits], GROUPS[entry]
    pad = -np.inf if low == "-inf" else (-65504.0 if bits == 16 else -1e10)
    for Nk in (kg * step, kg * step + 70):
        q, k, v = _inputs(bits, 1, 40, Nk, 131)
        q[:, :, 0], k[:, :, 0] = 100.0, 0.0
        for blocks in [[g] for g in range(kg)] + [list(range(1, kg)), [kg - 1, kg]]:
            kp = k.copy()
            for b in blocks:
                kp[:, b * step:(b + 1) * step, 0] = pad
            e = _Entry(px, stream, bits, entry, q, kp, v, 0.125)
            want = _softmax(q, kp, v, 0.125)
            for sp in (1, 2):
                got = e.run(sp)
                assert _rel(got, want) < TOL[bits], (Nk, blocks, sp)
            e.close()


@pytest.mark.parametrize("bits", [16, 32])
def test_planned_launch_with_padded_keys(px_gpu, stream, bits):
    # through the public entry: 32 queries over 256 keys, the last 64 padding
    px = px_gpu
    Nq, Nk = 32, 256
    q, k, v = (t[0] for t in _inputs(bits, 1, Nq, Nk, 141))
    q[:, 0], k[:, 0] = 100.0, 0.0
    k[192:, 0] = -65504.0 if bits == 16 else -1e10
    up = oracle.f16_bits if bits == 16 else np.ascontiguousarray
    dq, dk, dv = (px.DeviceBuffer.from_array(up(t)) for t in (q, k, v))
    do = px.DeviceBuffer(Nq * D * bits // 8)
    px.launch_flash(stream, px.FLASH_FP16 if bits == 16 else px.FLASH_FP32, dq, dk, dv, do, Nq, Nk,
                    D, 0.125)
    stream.synchronize()
    got = (oracle.f16_to_f32(do.download(np.uint16, Nq * D)).reshape(Nq, D) if bits == 16
           else do.download(np.float32, (Nq, D)))
    assert _rel(got, _softmax(q[None], k[None], v[None], 0.125)[0]) < TOL[bits]


@pytest.mark.parametrize("bits,entry", _all_entries())
@pytest.mark.parametrize("Nk", [1, 40, 100, 320, 520])
def test_every_key_far_below_the_initial_max(px_gpu, stream, bits, entry, Nk):
    # every score is -102400 (f16) or -6.4e8 (f32), in f16 one key's 3.75 more
    # (the scores are exact; a max of this size in log2 units is rounded by up
    # to 2^-7, which weighs its group 0.5% wrong), in groups with blocks and
    # without (Nk under KG steps)
    px, (qv, kv), scale = px_gpu, ((40.0, -40.0) if bits == 16 else (1e3, -1e4)), 1.0
    q, k, v = _inputs(bits, 2, 33, Nk, 151)
    q[:], k[:] = qv, kv
    if bits == 16:
        k[:, Nk // 2, 0] += 3.0 / 32.0
    e = _Entry(px, stream, bits, entry, q, k, v, scale)
    want = _softmax(q, k, v, scale)
    for sp in (1, 2, 3):
        assert _rel(e.run(sp), want) < TOL[bits], sp
    e.close()


@pytest.mark.parametrize("bits", [16, 32])
def test_planned_launch_far_below_the_initial_max(px_gpu, stream, bits):
    px, (qv, kv) = px_gpu, ((40.0, -40.0) if bits == 16 else (1e3, -1e4))
    Nq, Nk = 32, 200
    v = _inputs(bits, 1, 1, Nk, 161)[2][0]
    q, k = np.full((Nq, D), qv, np.float32), np.full((Nk, D), kv, np.float32)
    up = oracle.f16_bits if bits == 16 else np.ascontiguousarray
    dq, dk, dv = (px.DeviceBuffer.from_array(up(t)) for t in (q, k, v))
    do = px.DeviceBuffer(Nq * D * bits // 8)
    px.launch_flash(stream, px.FLASH_FP16 if bits == 16 else px.FLASH_FP32, dq, dk, dv, do, Nq, Nk,
                    D, 1.0)
    stream.synchronize()
    got = (oracle.f16_to_f32(do.download(np.uint16, Nq * D)).reshape(Nq, D) if bits == 16
           else do.download(np.float32, (Nq, D)))
    assert _rel(got, np.broadcast_to(v.astype(np.float64).mean(axis=0), got.shape)) < TOL[bits]


@pytest.mark.parametrize("bits", [16, 32])
@pytest.mark.parametrize("splits", [1, 2, 3, 4, 5, 6, 7])
def test_an_infinite_value_stays_infinite(px_gpu, stream, monkeypatch, bits, splits):
    # V holds one infinity per sign: every output of its column is that
    # infinity, whatever the number of chunks flash_combine merges (it reads
    # them in batches of four)
    px = px_gpu
    monkeypatch.setenv("PHX_FLASH_SPLIT", str(splits))
    Nq, Nk = 40, 448
    q, k, v = (t[0] for t in _inputs(bits, 1, Nq, Nk, 171))
    v[3, 5], v[440, 9] = np.inf, -np.inf
    up = oracle.f16_bits if bits == 16 else np.ascontiguousarray
    dq, dk, dv = (px.DeviceBuffer.from_array(up(t)) for t in (q, k, v))
    do = px.DeviceBuffer(Nq * D * bits // 8)
    px.launch_flash(stream, px.FLASH_FP16 if bits == 16 else px.FLASH_FP32, dq, dk, dv, do, Nq, Nk,
                    D, 0.125)
    stream.synchronize()
    got = (oracle.f16_to_f32(do.download(np.uint16, Nq * D)).reshape(Nq, D) if bits == 16
           else do.download(np.float32, (Nq, D)))
    assert (got[:, 5] == np.inf).all() and (got[:, 9] == -np.inf).all()
    rest = [d for d in range(D) if d not in (5, 9)]
    want = _softmax(q[None], k[None], v[None][:, :, rest], 0.125)[0]
    assert _rel(got[:, rest], want) < TOL[bits]
