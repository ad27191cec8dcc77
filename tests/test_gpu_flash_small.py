"""The small-launch flash kernels (csrc/kernels/flash_w.h) at the edges of
their query blocks, key groups and key steps, each entry launched by itself
with one key chunk and with several (merged by flash_combine), against the f64
oracle by the kernels' bounds (|err| / max(|want|, 0.1) <= 2e-2 for f16, 1e-4
for f32, test_gpu_flash.py), over rows and heads with gaps between them."""
import ctypes
import os

import numpy as np
import pytest

import oracle

pytestmark = pytest.mark.gpu

D = 64
ENTRIES = {16: [("flash_w4", 32, 256), ("flash_w2x4", 64, 512)],
           32: [("flash_w4", 32, 256), ("flash_w8", 32, 512)]}
FILES = {16: "flash_attention_fp16.hsaco", 32: "flash_attention_fp32.hsaco"}
TOL = {16: 2e-2, 32: 1e-4}
GAP = 8  # elements after every row, and a row after every head


class _Heads:
    """[BH, N, D] rows GAP elements apart in a buffer of NaN."""

    def __init__(self, px, bits, x):
        BH, N, _ = x.shape
        self.dt = np.uint16 if bits == 16 else np.uint32
        self.bits, self.shape = bits, (BH, N, D)
        self.ld, self.hs = D + GAP, (N + 1) * (D + GAP)
        self.host = np.full((BH, N + 1, D + GAP), 0x7E00 if bits == 16 else 0x7FC00000, self.dt)
        self.host[:, :N, :D] = (oracle.f16_bits(x) if bits == 16
                                else x.astype(np.float32).view(np.uint32)).reshape(x.shape)
        self.buf = px.DeviceBuffer.from_array(self.host)

    def get(self):
        out = self.buf.download(self.dt, self.host.shape)
        N = self.shape[1]
        assert np.array_equal(out[:, N:], self.host[:, N:]), "store past the head"
        assert np.array_equal(out[:, :, D:], self.host[:, :, D:]), "store past a row"
        got = np.ascontiguousarray(out[:, :N, :D])
        return oracle.f16_to_f32(got).reshape(got.shape) if self.bits == 16 else got.view(np.float32)


def _inputs(bits, BH, Nq, Nk, seed):
    t = [oracle.normal_f32(seed + i, BH * n * D).reshape(BH, n, D)
         for i, n in enumerate((Nq, Nk, Nk))]
    return [oracle.f16_round(x).reshape(x.shape) for x in t] if bits == 16 else t


def _void(vals):
    return (ctypes.c_void_p * len(vals))(*[ctypes.cast(ctypes.byref(v), ctypes.c_void_p)
                                           for v in vals])


def _launch(px, stream, fn, grid, block, vals):
    u3 = ctypes.c_uint32 * 3
    px.check(px.lib().phx_launch(fn, u3(*grid), u3(block, 1, 1), 0, stream.handle, _void(vals)))


@pytest.mark.parametrize("bits", [16, 32])
@pytest.mark.parametrize("BH,Nq,Nk,scale", [
    (1, 1, 1, 0.125), (2, 31, 31, 0.125), (1, 32, 33, -0.2), (3, 33, 64, 0.125),
    (1, 64, 65, 0.125), (2, 65, 129, 0.0), (1, 63, 255, 0.125), (1, 40, 257, 8.0),
    (2, 97, 320, 0.125), (1, 128, 577, -0.125), (1, 35, 1100, 0.125)])
def test_small_launch_kernels(px_gpu, stream, bits, BH, Nq, Nk, scale):
    px = px_gpu
    q, k, v = _inputs(bits, BH, Nq, Nk, 101)
    dq, dk, dv = (_Heads(px, bits, t) for t in (q, k, v))
    want = np.stack([oracle.flash_rows(np.arange(Nq), q[h], k[h], v[h], scale) for h in range(BH)])
    nkb = -(-Nk // 64)
    ws = px.DeviceBuffer(4 * BH * Nq * (D + 2) * 4)
    with open(os.path.join(px.LIB_DIR, FILES[bits]), "rb") as f:
        mod = px.module_load_data(f.read())
    i64, u64 = ctypes.c_int64, ctypes.c_uint64
    for entry, qb, threads in ENTRIES[bits]:
        fn = px.module_get_function(mod, entry)
        for sp in sorted({1, min(2, nkb), min(4, nkb)}):
            chunk = -(-nkb // sp) * 64
            sp = -(-Nk // chunk)
            do = _Heads(px, bits, np.zeros((BH, Nq, D), np.float32))
            vals = [u64(b) for b in (dq.buf.ptr, dk.buf.ptr, dv.buf.ptr, do.buf.ptr, ws.ptr)]
            vals += [i64(x) for x in (BH, Nq, Nk, dq.ld, dk.ld, dv.ld, do.ld, dq.hs, dk.hs, dv.hs,
                                      do.hs, chunk)]
            vals += [ctypes.c_int32(sp), ctypes.c_float(scale)]
            _launch(px, stream, fn, (-(-Nq // qb) * BH, sp, 1), threads, vals)
            if sp > 1:
                vals = [u64(ws.ptr), ctypes.c_int32(sp), u64(do.buf.ptr)]
                vals += [i64(x) for x in (BH, Nq, do.ld, do.hs)]
                _launch(px, stream, px.module_get_function(mod, "flash_combine"),
                        (-(-BH * Nq * 16 // 256), 1, 1), 256, vals)
            stream.synchronize()
            err = (np.abs(do.get() - want) / np.maximum(np.abs(want), 0.1)).max()
            assert err < TOL[bits], (entry, sp, err)
    px.module_unload(mod)


@pytest.mark.parametrize("bits", [16, 32])
@pytest.mark.parametrize("BH,Nq,Nk", [(16, 529, 128), (1, 1024, 1024), (4, 300, 700), (8, 1000, 1000)])
def test_planned_launches_meet_the_oracle(px_gpu, stream, bits, BH, Nq, Nk):
    # through the built-in plan, with the session stream's workspace and
    # without one
    px = px_gpu
    q, k, v = _inputs(bits, BH, Nq, Nk, 111)
    kern = px.FLASH_FP16_BH if bits == 16 else px.FLASH_FP32_BH
    up = (lambda t: oracle.f16_bits(t)) if bits == 16 else (lambda t: np.ascontiguousarray(t))
    dq, dk, dv = (px.DeviceBuffer.from_array(up(t)) for t in (q, k, v))
    esz = bits // 8
    rows = np.unique(np.linspace(0, Nq - 1, 24).astype(np.int64))
    want = {h: oracle.flash_rows(rows, q[h], k[h], v[h], 0.125) for h in (0, BH - 1)}
    bare = px.Stream()
    for s in (stream, bare):
        do = px.DeviceBuffer(BH * Nq * D * esz)
        px.launch_flash_bh(s, kern, dq, dk, dv, do, BH, Nq, Nk, D, 0.125)
        s.synchronize()
        if bits == 16:
            got = oracle.f16_to_f32(do.download(np.uint16, BH * Nq * D)).reshape(BH, Nq, D)
        else:
            got = do.download(np.float32, (BH, Nq, D))
        for h, w in want.items():
            err = (np.abs(got[h][rows] - w) / np.maximum(np.abs(w), 0.1)).max()
            assert err < TOL[bits], (h, err)
    bare.destroy()
