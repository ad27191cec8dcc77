"""The work this backend's users have it do, as cases that can be timed and
compared: the leaf kernels through the launch helpers of phobos_amd, on a
stream of the program's own with a split workspace bound to it, as bench.py
and the pod executor set theirs up.

A case names its "op" and sizes:
  saxpy   out = 2.5 x + y over n elements;
  gemm    C = alpha A@B + beta C, kernel gemm_fp32, gemm_fp16tc or gemm_fp16;
  flash   attention over D = 64, one head (the .ph entry, heads 0) or a batch
          of heads in one launch, f16 or f32;
  leaves  what a pod computes for one C supertile of a matmul_cluster job: the
          init leaf, then one step leaf per K supertile.
Operands are dense torch tensors made on the GPU from the seed: N(0, 1) where
the BASELINE configs draw normals, GEMM operands scaled by 1/sqrt(K) (1/64 at
4096), so that outputs are of order one.
"""
import math
import os
import sys

import torch

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
if os.path.join(ROOT, "phobos-lang_amd") not in sys.path:
    sys.path.insert(0, os.path.join(ROOT, "phobos-lang_amd"))
import phobos_amd as px  # noqa: E402

D = 64
SCALE = 0.125
WORKSPACE = 256 << 20  # the split workspace the tests and bench.py's shapes bind

GEMMS = {"gemm_fp32": px.GEMM_FP32, "gemm_fp16tc": px.GEMM_FP16TC_FP32ACC,
         "gemm_fp16": px.GEMM_FP16}


def _saxpy(n, **kw):
    return dict(kw, op="saxpy", n=n)


def _gemm(kernel, M, N, K, alpha=1.0, beta=0.0, **kw):
    return dict(kw, op="gemm", kernel=kernel, M=M, N=N, K=K, alpha=alpha, beta=beta)


def _flash(bits, heads, Nq, Nk, **kw):
    return dict(kw, op="flash", bits=bits, heads=heads, Nq=Nq, Nk=Nk)


def _leaves(M, N, K, steps, **kw):
    # beta below 1, so that a supertile run over and over stays finite
    return dict(kw, op="leaves", M=M, N=N, K=K, steps=steps, alpha=0.125, beta=0.5)


def listed():
    return [
        # the smallest calls: a vector of odd length, where the launch is the cost
        _saxpy(100_003, name="saxpy_100003"),
        # the BASELINE saxpy, an HBM stream
        _saxpy(1 << 24, name="saxpy_16m"),
        # a small exact-f32 product with C accumulated
        _gemm("gemm_fp32", 512, 512, 512, 0.5, 0.25, name="gemm_fp32_512"),
        # the BASELINE f32 GEMM size
        _gemm("gemm_fp32", 4096, 4096, 4096, name="gemm_fp32_4096"),
        # f32 storage, f16 products, no extent a multiple of a tile
        _gemm("gemm_fp16tc", 1000, 1000, 1000, name="gemm_fp16tc_1000"),
        # the BASELINE headline
        _gemm("gemm_fp16tc", 4096, 4096, 4096, name="gemm_fp16tc_4096"),
        # f16 storage at an ordinary size, and at the BASELINE size
        _gemm("gemm_fp16", 1024, 1024, 1024, 0.5, 0.25, name="gemm_fp16_1024"),
        _gemm("gemm_fp16", 4096, 4096, 4096, name="gemm_fp16_4096"),
        # the reference bench's own flash launch: one head of 4096 queries
        _flash(16, 0, 4096, 4096, name="flash_fp16_one_head"),
        # the BASELINE flash: B4 x H16
        _flash(16, 64, 4096, 4096, name="flash_fp16_64_heads"),
        # exact-f32 attention of a few heads, ragged queries and keys
        _flash(32, 4, 1000, 4133, name="flash_fp32_ragged"),
        # a pod's leaves for one C supertile
        _leaves(1024, 1024, 1024, 4, name="pod_leaves_1024"),
    ]


def _size(rng, lo, hi, mult=1):
    """A size in [lo, hi], even in its logarithm; half of them multiples of 64."""
    v = int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))
    if rng.random() < 0.5:
        v = v // 64 * 64
    return max(mult, lo // mult * mult, min(v, hi) // mult * mult)


def draw(rng):
    op = rng.choice(["saxpy", "gemm", "gemm", "gemm", "gemm", "flash", "flash", "leaves"])
    if op == "saxpy":
        return _saxpy(int(round(math.exp(rng.uniform(math.log(1000), math.log(1 << 24))))))
    if op == "gemm":
        kernel = rng.choice(sorted(GEMMS))
        M, N, K = (_size(rng, 64, 4096, m) for m in (1, 8, 8))
        return _gemm(kernel, M, N, K, *rng.choice([(1.0, 0.0), (0.5, 0.25)]))
    if op == "flash":
        bits = rng.choice([16, 32])
        Nq, Nk = _size(rng, 64, 4096), _size(rng, 64, 4096)
        heads = rng.choice([0, 1, 2, 4, 8, 12, 16] + ([32, 64] if bits == 16 else []))
        return _flash(bits, heads, Nq, Nk)
    M, N, K = (_size(rng, 256, 2048, 4) for _ in range(3))
    return _leaves(M, N, K, rng.choice([1, 2, 4]))


_stream = None


def _launch_stream():
    """The program's stream, its split workspace bound."""
    global _stream
    if _stream is None:
        px.init(0)
        _stream = px.Stream()
        px.bind_workspace(_stream, WORKSPACE)
    return _stream


def _inputs(case, seed):
    g = torch.Generator(device="cuda").manual_seed(int(seed))

    def normal(*shape, scale=1.0, dtype=torch.float32):
        return (torch.randn(*shape, generator=g, device="cuda") * scale).to(dtype)

    op = case["op"]
    if op == "saxpy":
        return {"x": normal(case["n"]), "y": normal(case["n"])}
    if op == "flash":
        t = torch.float16 if case["bits"] == 16 else torch.float32
        lead = (case["heads"],) if case["heads"] else ()
        return {k: normal(*lead, case[n], D, dtype=t)
                for k, n in (("q", "Nq"), ("k", "Nk"), ("v", "Nk"))}
    M, N, K = case["M"], case["N"], case["K"]
    t = torch.float16 if op == "gemm" and case["kernel"] == "gemm_fp16" else torch.float32
    if op == "gemm":
        return {"a": normal(M, K, scale=K ** -0.5, dtype=t),
                "b": normal(K, N, scale=K ** -0.5, dtype=t),
                "c": normal(M, N, dtype=t)}
    # a pod's tiles: A [M, K] and B [K, N] per step, scaled to the whole sum
    s = (K * case["steps"]) ** -0.5
    return {"a": [normal(M, K, scale=s) for _ in range(case["steps"])],
            "b": [normal(K, N, scale=s) for _ in range(case["steps"])],
            "c": normal(M, N)}


def prepare(case, seed):
    state = dict(_inputs(case, seed), case=case, stream=_launch_stream())
    if case["op"] == "saxpy":
        state["out"] = torch.empty_like(state["x"])
    elif case["op"] == "flash":
        state["out"] = torch.empty_like(state["q"])
    elif case["op"] == "gemm":
        state["kernel"] = GEMMS[case["kernel"]]
    else:
        state["init"] = px.builtin_function(px.MATMUL_INIT)
        state["step"] = px.builtin_function(px.MATMUL)
    torch.cuda.synchronize()  # the inputs were made on torch's stream
    return state


def run(state):
    case, s = state["case"], state["stream"]
    op = case["op"]
    if op == "saxpy":
        px.launch_saxpy(s, state["x"].data_ptr(), state["y"].data_ptr(), state["out"].data_ptr(),
                        case["n"], 2.5)
        return state["out"]
    if op == "gemm":
        px.launch_gemm(s, state["kernel"], state["a"].data_ptr(), state["b"].data_ptr(),
                       state["c"].data_ptr(), case["M"], case["N"], case["K"], case["alpha"],
                       case["beta"])
        return state["c"]
    if op == "flash":
        p = [state[k].data_ptr() for k in ("q", "k", "v", "out")]
        f16 = case["bits"] == 16
        if case["heads"]:
            px.launch_flash_bh(s, px.FLASH_FP16_BH if f16 else px.FLASH_FP32_BH, *p,
                               case["heads"], case["Nq"], case["Nk"], D, SCALE)
        else:
            px.launch_flash(s, px.FLASH_FP16 if f16 else px.FLASH_FP32, *p, case["Nq"],
                            case["Nk"], D, SCALE)
        return state["out"]
    # the job's beta scales C once; then each step adds its product, with the
    # leaf grid and cta a scheduler sends (supertile / 32, 256 threads)
    M, N, K = case["M"], case["N"], case["K"]
    grid, cta = (M // 32, N // 32, 1), (256, 1, 1)
    c = (state["c"].data_ptr(), (M, N))
    alpha, beta = px.f32_bits(case["alpha"]), px.f32_bits(case["beta"])
    px.compute(state["init"], 32, [c], [(1, 4, beta)], grid, cta, s)
    for a, b in zip(state["a"], state["b"]):
        px.compute(state["step"], 32, [(a.data_ptr(), (M, K)), (b.data_ptr(), (K, N)), c],
                   [(3, 4, alpha), (4, 4, beta)], grid, cta, s)
    return state["c"]


def work(case):
    op = case["op"]
    if op == "saxpy":
        return {"bytes": 12 * case["n"], "flops": 2 * case["n"]}
    if op == "flash":
        bh = max(1, case["heads"])
        return {"bytes": bh * (2 * case["Nq"] + 2 * case["Nk"]) * D * case["bits"] // 8,
                "flops": 4 * bh * case["Nq"] * case["Nk"] * D}
    M, N, K = case["M"], case["N"], case["K"]
    if op == "gemm":
        e = 2 if case["kernel"] == "gemm_fp16" else 4
        return {"bytes": e * (M * K + K * N + (2 if case["beta"] else 1) * M * N),
                "flops": 2 * M * N * K}
    # C is read and written by every leaf: each is a call of its own
    steps = case["steps"]
    return {"bytes": 4 * (steps * (M * K + K * N) + 2 * (steps + 1) * M * N),
            "flops": 2 * M * N * K * steps}


def tolerance(case):
    op = case["op"]
    if op == "saxpy":
        return "exact"  # the multiply and the add round separately, in every implementation
    if op == "flash":
        # f16: O rounds to f16, and P for P.V; f32: sums over the keys and D
        return {"rel": 1.5e-3} if case["bits"] == 16 else {"rel": 4e-6}
    if op == "gemm" and case["kernel"] == "gemm_fp16":
        return {"rel": 1e-3}  # one rounding of C to f16
    return {"rel": 4e-6}  # f32 sums over K


def exact(case, seed):
    i = _inputs(case, seed)
    op = case["op"]
    if op == "saxpy":
        return 2.5 * i["x"].double() + i["y"].double()
    if op == "gemm":
        a, b = i["a"], i["b"]
        if case["kernel"] == "gemm_fp16tc":  # the kernel's operands: f32 rounded to f16
            a, b = a.half(), b.half()
        out = case["alpha"] * (a.double() @ b.double())
        return out + case["beta"] * i["c"].double() if case["beta"] else out
    if op == "leaves":
        out = case["beta"] * i["c"].double()
        for a, b in zip(i["a"], i["b"]):
            out = out + case["alpha"] * (a.double() @ b.double())
        return out
    q, k, v = (i[n].reshape(-1, i[n].shape[-2], D).double() for n in ("q", "k", "v"))
    out = torch.empty_like(q)
    for h in range(q.shape[0]):
        out[h] = torch.softmax(SCALE * (q[h] @ k[h].t().contiguous()), dim=-1) @ v[h]
    return out.reshape(i["q"].shape)
