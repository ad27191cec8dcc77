"""The smaller output tiles of the GEMMs at the edges of their tiles:
gemm_fp16 and gemm_fp16tc_fp32acc (csrc/kernels/gemm_tiles.h), gemm_fp32 and
the cluster step leaf (gemm_s_tiles.h), and their split-K forms.

An output is an f32 sum of K exact products in some order, so it lies within
K eps of the sum of their magnitudes (K * 2^-24 * |A|@|B|) of the f64 oracle,
plus the epilogue's roundings: 2^-22 relative for f32 outputs, one rounding to
f16 (2^-11, doubled for ties on the wrong side of the f32 error) for
gemm_fp16.  Small integers are exact in every order.
"""
import ctypes
import os

import numpy as np
import pytest

import oracle

pytestmark = pytest.mark.gpu

M_ENTRIES = {"gemm_m64": (64, 64), "gemm_m128x64": (128, 64), "gemm_m128": (128, 128)}
S_ENTRIES = {"s64": (64, 64), "s64x32": (64, 32), "s32": (32, 32)}
KERNELS = {"GEMM_FP16": ("gemm_fp16.hsaco", M_ENTRIES),
           "GEMM_FP16TC_FP32ACC": ("gemm_fp16tc_fp32acc.hsaco", M_ENTRIES),
           "GEMM_FP32": ("gemm_fp32.hsaco", {"gemm_" + n: t for n, t in
                                             {**S_ENTRIES, "s32a4": (32, 32)}.items()}),
           "MATMUL": ("matmul_cluster_fp32.hsaco", {"matmul_" + n: t for n, t in S_ENTRIES.items()})}
# one row and the smallest N and K, whole tiles, one past a tile, one K step
# and one past it, a K of every stage of the rings, a partial last K step
SHAPES = [(1, 8, 8), (64, 64, 64), (65, 72, 72), (128, 128, 128), (129, 136, 200),
          (63, 56, 320), (200, 264, 456), (257, 320, 1000)]


class _Case:
    """A, B, C in buffers with row pitches beyond their extents (pad elements
    of NaN after every row) and a C whose pad must come back untouched."""

    def __init__(self, px, kern, M, N, K, pad, seed=5):
        self.px, self.kern, self.dims = px, kern, (M, N, K)
        self.f16 = kern == px.GEMM_FP16
        self.idx = ctypes.c_int32 if kern in (px.GEMM_FP32, px.MATMUL) else ctypes.c_int64
        A = oracle.f16_round(oracle.normal_f32(seed, M * K, 1 / np.sqrt(K))).reshape(M, K)
        B = oracle.f16_round(oracle.normal_f32(seed + 1, K * N, 1 / np.sqrt(K))).reshape(K, N)
        C = oracle.f16_round(oracle.normal_f32(seed + 2, M * N)).reshape(M, N)
        self.A, self.B, self.C = A, B, C
        self.dt = np.uint16 if self.f16 else np.uint32
        self.host = [self._padded(t, pad) for t in (A, B, C)]
        self.dev = [px.DeviceBuffer.from_array(t) for t in self.host]

    def _padded(self, t, pad):
        bits = oracle.f16_bits(t) if self.f16 else t.astype(np.float32).view(np.uint32)
        out = np.full((t.shape[0], t.shape[1] + pad), 0x7E00 if self.f16 else 0x7FC00000, self.dt)
        out[:, :t.shape[1]] = bits.reshape(t.shape)
        return out

    def args(self, alpha, beta):
        vals = []
        for t, buf, (r, c) in zip(self.host, self.dev, (self.A.shape, self.B.shape, self.C.shape)):
            vals += [ctypes.c_uint64(buf.ptr), ctypes.c_uint64(buf.ptr)]
            vals += [self.idx(v) for v in (0, r, c, t.shape[1], 1)]
        vals += [ctypes.c_float(alpha), ctypes.c_float(beta)]
        return vals, (ctypes.c_void_p * len(vals))(
            *[ctypes.cast(ctypes.byref(v), ctypes.c_void_p) for v in vals])

    def launch(self, stream, fn, grid, block, alpha, beta):
        """The bits of C after the launch, its pad checked."""
        self.dev[2].upload(self.host[2])
        keep, arr = self.args(alpha, beta)
        u3 = ctypes.c_uint32 * 3
        self.px.check(self.px.lib().phx_launch(fn, u3(grid, 1, 1), u3(block, 1, 1), 0,
                                               stream.handle, arr))
        stream.synchronize()
        out = self.dev[2].download(self.dt, self.host[2].shape)
        N = self.dims[1]
        assert np.array_equal(out[:, N:], self.host[2][:, N:]), "store outside C"
        return out[:, :N].copy()

    def values(self, bits):
        return oracle.f16_to_f32(bits) if self.f16 else bits.view(np.float32)


def _check(case, bits, alpha, beta):
    if case.kern == case.px.MATMUL:
        beta = 1.0  # the step leaf's, whatever it is passed
    got = case.values(bits).reshape(case.C.shape)
    ref = oracle.gemm_full(case.A, case.B, case.C, alpha, beta, round16=True)
    K = case.dims[2]
    mag = abs(alpha) * (np.abs(case.A) @ np.abs(case.B)) + abs(beta) * np.abs(case.C)
    bound = K * 2.0 ** -24 * mag + (2.0 ** -10 if case.f16 else 2.0 ** -22) * np.abs(ref)
    # an f16 result below 2^-14 is subnormal: its step is 2^-24
    assert (np.abs(got - ref) <= bound + (2.0 ** -24 if case.f16 else 1e-30)).all()
    return got


@pytest.mark.parametrize("pad", [0, 8])
@pytest.mark.parametrize("M,N,K", SHAPES)
@pytest.mark.parametrize("kern_name", list(KERNELS))
def test_each_tile_meets_the_oracle(px_gpu, stream, kern_name, M, N, K, pad):
    # every entry launched by itself, one workgroup per tile and with fewer
    # workgroups than tiles (the block-stride walk), C read and not read
    px = px_gpu
    case = _Case(px, getattr(px, kern_name), M, N, K, pad)
    with open(os.path.join(px.LIB_DIR, KERNELS[kern_name][0]), "rb") as f:
        mod = px.module_load_data(f.read())  # launched with the test's own grids
    for alpha, beta in ((1.0, 0.0), (0.75, -0.5)):
        for entry, (tm, tn) in KERNELS[kern_name][1].items():
            fn = px.module_get_function(mod, entry)
            tiles = -(-M // tm) * -(-N // tn)
            outs = [case.launch(stream, fn, grid, 256, alpha, beta)
                    for grid in (tiles, max(1, tiles // 2), min(8, tiles))]
            _check(case, outs[0], alpha, beta)
            assert all(np.array_equal(outs[0], o) for o in outs), entry
    px.module_unload(mod)


@pytest.mark.parametrize("chunk", [32, 96, 160])
@pytest.mark.parametrize("M,N,K", [(1, 8, 40), (65, 72, 200), (130, 136, 264), (200, 264, 328),
                                   (257, 320, 1000)])
@pytest.mark.parametrize("kern_name", [k for k in KERNELS if k != "MATMUL"])
def test_each_split_form_meets_the_oracle(px_gpu, stream, kern_name, M, N, K, chunk):
    # every split-K entry launched by itself over its own grid, then the reduce
    # kernel: chunks of an odd number of 32 columns (a partial step of the 64
    # deep tiles), the last one shorter, guard words behind the planes
    px = px_gpu
    case = _Case(px, getattr(px, kern_name), M, N, K, 8)
    with open(os.path.join(px.LIB_DIR, KERNELS[kern_name][0]), "rb") as f:
        mod = px.module_load_data(f.read())
    reduce = px.module_get_function(mod, "gemm_splitk_reduce")
    chunks = -(-K // chunk)
    planes = chunks * M * N
    guard = np.full(planes + 1024, 0x7FC00001, np.uint32)
    ws = px.DeviceBuffer.from_array(guard)
    i64, u64, u3 = ctypes.c_int64, ctypes.c_uint64, ctypes.c_uint32 * 3

    def launch(fn, grid, vals):
        arr = (ctypes.c_void_p * len(vals))(
            *[ctypes.cast(ctypes.byref(v), ctypes.c_void_p) for v in vals])
        px.check(px.lib().phx_launch(fn, u3(*grid), u3(256, 1, 1), 0, stream.handle, arr))

    ld = [t.shape[1] for t in case.host]
    for entry, (tm, tn) in KERNELS[kern_name][1].items():
        if entry == "gemm_s32a4":  # runs unsplit only
            continue
        ws.upload(guard)
        case.dev[2].upload(case.host[2])
        launch(px.module_get_function(mod, entry + "_splitk"),
               (-(-M // tm) * -(-N // tn), chunks, 1),
               [u64(case.dev[0].ptr), u64(case.dev[1].ptr), u64(ws.ptr)] +
               [i64(x) for x in (ld[0], ld[1], M, N, K, chunk)])
        launch(reduce, (-(-M * N // 1024), 1, 1),
               [u64(ws.ptr), ctypes.c_int32(chunks), u64(case.dev[2].ptr), i64(ld[2]), i64(M),
                i64(N), ctypes.c_float(0.75), ctypes.c_float(-0.5)])
        stream.synchronize()
        w = ws.download(np.uint32, planes + 1024)
        assert (w[planes:] == guard[planes:]).all(), (entry, "store past the planes")
        assert np.isfinite(w[:planes].view(np.float32)).all(), (entry, "plane not written")
        out = case.dev[2].download(case.dt, case.host[2].shape)
        assert np.array_equal(out[:, N:], case.host[2][:, N:]), (entry, "store outside C")
        _check(case, out[:, :N].copy(), 0.75, -0.5)
    px.module_unload(mod)


@pytest.mark.parametrize("kern_name", list(KERNELS))
@pytest.mark.parametrize("M,N,K", [(64, 64, 4096), (65, 72, 2056), (200, 520, 3000),
                                   (1000, 1000, 1000), (1208, 1208, 64), (300, 4096, 512),
                                   (2100, 2056, 40), (1100, 1064, 104)])
def test_rule_launches_meet_the_oracle(px_gpu, stream, kern_name, M, N, K):
    # through the built-in plan: the tile it picks, split over K into the
    # bound workspace where that is cheaper, and on a stream without one
    px = px_gpu
    kern = getattr(px, kern_name)
    case = _Case(px, kern, M, N, K, 8)
    bare = px.Stream()
    for s in (stream, bare):
        _check(case, case.launch(s, px.builtin_function(kern), 1, 256, 0.75, -0.5), 0.75, -0.5)
    bare.destroy()


def test_rows_that_overlap_run_the_256_tile(px_gpu, stream):
    # a row stride shorter than the row (the descriptors allow it) is left to
    # the 256 x 256 kernels, which take any stride: A's rows here are the
    # same 64 elements shifted by 8
    px = px_gpu
    M, N, K, lda = 64, 64, 64, 8
    case = _Case(px, px.GEMM_FP16, M, N, K, 0)
    flat = case.A.ravel()
    case.A = np.stack([flat[i * lda:i * lda + K] for i in range(M)])
    vals, arr = case.args(1.0, 0.0)
    vals[5].value = lda  # A's row stride
    case.dev[2].upload(case.host[2])
    u3 = ctypes.c_uint32 * 3
    px.check(px.lib().phx_launch(px.builtin_function(px.GEMM_FP16), u3(1, 1, 1), u3(256, 1, 1), 0,
                                 stream.handle, arr))
    stream.synchronize()
    _check(case, case.dev[2].download(case.dt, case.host[2].shape), 1.0, 0.0)


# extents whose built-in split has shorter chains than a small tile's
# accumulator sets would have
@pytest.mark.parametrize("kern_name,M,N,K", [
    ("GEMM_FP16TC_FP32ACC", 1536, 1536, 4096), ("GEMM_FP16TC_FP32ACC", 1304, 728, 1864),
    ("GEMM_FP16TC_FP32ACC", 1760, 448, 2840), ("GEMM_FP16TC_FP32ACC", 284, 2528, 3432),
    ("GEMM_FP16TC_FP32ACC", 1280, 1280, 1280), ("GEMM_FP16TC_FP32ACC", 1000, 1000, 1000),
    ("GEMM_FP32", 400, 96, 376), ("GEMM_FP32", 113, 104, 400), ("GEMM_FP32", 564, 64, 392),
    ("GEMM_FP32", 96, 80, 344)])
def test_small_tiles_sum_no_less_exactly_than_the_split(px_gpu, stream, monkeypatch, kern_name, M,
                                                        N, K):
    # root mean square error against f64 of the tile the built-in plan picks
    # and of the split it names on the 256 x 256 tile: within 5% (the root mean
    # square of 7680 errors scatters by 1%, and sum_noise fits within 3%)
    px = px_gpu
    kern = getattr(px, kern_name)
    case = _Case(px, kern, M, N, K, 0)
    ref = case.A.astype(np.float64) @ case.B.astype(np.float64)
    fn = px.builtin_function(kern)

    def rms():
        got = case.values(case.launch(stream, fn, 1, 256, 1.0, 0.0)).reshape(ref.shape)
        return np.sqrt(np.mean((got - ref) ** 2))

    splits = px.split_plan(kern, [M, N, K])[0]
    assert splits > 1
    picked = rms()
    monkeypatch.setenv("PHX_GEMM_SPLIT", str(splits))
    assert picked <= 1.05 * rms()


def test_more_tiles_than_a_launch_takes_workgroups(px_gpu, stream):
    # 2^31 - 1 rows of gemm_fp16 in 128 x 64 tiles would be 2^24 workgroups of
    # 256 threads, one more than a launch takes; A of equal elements, so every
    # row of C is the same, over a C of NaN (32 GiB each, checked at both ends
    # and in between)
    px = px_gpu
    M, N, K = 2 ** 31 - 1, 8, 8
    dA, dC = px.DeviceBuffer(M * K * 2), px.DeviceBuffer(M * N * 2)
    px.check(px.lib().phx_memset_async(dA.ptr, 0x38, M * K * 2, None))
    px.check(px.lib().phx_memset_async(dC.ptr, 0xFF, M * N * 2, None))
    px.synchronize()
    B = (np.arange(K * N, dtype=np.float32) / 8).reshape(K, N)
    dB = px.DeviceBuffer.from_array(oracle.f16_bits(B))
    print(f"gemm_fp16 M={M} N={N} K={K}", flush=True)
    px.launch_gemm(stream, px.GEMM_FP16, dA, dB, dC, M, N, K, 1.0, 0.0)
    stream.synchronize()
    a = oracle.f16_to_f32(np.uint16([0x3838]))[0]
    want = oracle.f16_bits((a * B.sum(axis=0)).astype(np.float32))  # the sums are exact in f32
    rows = 1 << 16
    for r in [0, M // 3, 1 << 30, M - 5 * rows, M - rows]:
        out = np.empty((rows, N), np.uint16)
        px.check(px.lib().phx_memcpy_d2h(out.ctypes.data, dC.ptr + r * N * 2, out.nbytes))
        assert (out == want.reshape(1, N)).all(), r
    for b in (dA, dB, dC):
        b.free()
