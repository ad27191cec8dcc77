"""The launch path's own state: argument lists longer than the words a launch
keeps on its stack, and entry points remembered per thread, which a shutdown
must forget (in a child process, as it unloads every module)."""
import os
import subprocess
import sys

import numpy as np
import pytest

import oracle

pytestmark = pytest.mark.gpu

_AGAIN = """
import sys, threading
sys.path[:0] = [{root!r} + "/phobos-lang_amd"]
import numpy as np, phobos_amd as px
M, N, K = 64, 64, 2048
a, b = px.normal_f32(1, M * K), px.normal_f32(2, K * N)

def run():
    s = px.Stream()
    px.bind_workspace(s, 1 << 22)  # K is split: entries no .ph kernel names
    bufs = [px.DeviceBuffer.from_array(x) for x in (a, b)] + [px.DeviceBuffer(4 * M * N)]
    bufs[2].zero(s)
    px.launch_gemm(s, px.GEMM_FP32, *bufs, M, N, K, 1.0, 0.0)
    s.synchronize()
    out = bufs[2].download(np.float32, (M, N))
    px.bind_workspace(s, 0)
    s.destroy()
    return out

px.init(0)
first = run()
want = a.reshape(M, K).astype(np.float64) @ b.reshape(K, N)
assert np.abs(first - want).max() <= 1e-5 * K ** 0.5 * 4
for _ in range(2):
    px.synchronize()
    px.check(px.lib().phx_shutdown())
    px.check(px.lib().phx_init(0, px.LIB_DIR.encode()))
    assert np.array_equal(run(), first)
    got = []
    t = threading.Thread(target=lambda: got.append(run()))  # a thread that remembers nothing
    t.start()
    t.join()
    assert np.array_equal(got[0], first)
print("same")
"""


def test_entries_are_found_again_after_a_shutdown():
    root = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
    r = subprocess.run([sys.executable, "-c", _AGAIN.format(root=root)], capture_output=True,
                       text=True, timeout=100)
    assert r.returncode == 0 and "same" in r.stdout, r.stderr[-2000:]


# words of a COMPUTE list: saxpy's three tiles (5 each) and alpha, then further
# tiles the kernel does not read; a launch keeps 48 on its stack, of the
# tiles * 9 + 1 it makes room for
@pytest.mark.parametrize("extra", [0, 2, 3, 20])
def test_long_argument_lists(px_gpu, stream, extra):
    px = px_gpu
    n = 1000
    x, y = oracle.normal_f32(1, n), oracle.normal_f32(2, n)
    bx, by = px.DeviceBuffer.from_array(x), px.DeviceBuffer.from_array(y)
    out = px.DeviceBuffer(4 * n)
    tiles = [(b.ptr, (n,)) for b in (bx, by, out)] + [(bx.ptr, (n,))] * extra
    px.compute(px.builtin_function(px.SAXPY_FP32), 32, tiles, [(3, 4, px.f32_bits(2.5))],
               (1, 1, 1), (256, 1, 1), stream)
    stream.synchronize()
    # one rounding of the product and one of the sum, or a single fused one
    want = 2.5 * x.astype(np.float64) + y
    bound = 2.0 ** -24 * (np.abs(2.5 * x) + np.abs(want)) * 1.01
    assert np.all(np.abs(out.download(np.float32, n) - want) <= bound)
