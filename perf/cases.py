"""The calls that programs built on this library make, at the sizes they make them at.

A case names an operator of `fastgate_amd.speedgate`, a number of activation rows M, a weight shape
(N outputs, K inputs, both multiples of 128) and nothing else; weights are random, activations
N(0, 1).  The operators cover both fp16 weight layouts ([N,K] and [K,N]), overwrite and accumulate,
the feed-forward pair with its fused bias and activation, and the int8, int4 and int8 x int8 weight
paths.  Rows run from one (decoding one sequence) over 2 .. 16 (small batches, the sixteen tokens of
the DiT feed-forward pair) to 256 (large decode batches, prompt chunks); the quantised operators
take 16, 4 and 8 rows at most.
"""
import torch

from fastgate_amd import speedgate as sg

# kind -> (most rows the operator takes, bytes of one weight)
KINDS = {
    "gemv": (1, 2.0),         # fastgemv: weights [N,K], weight first
    "edgemm": (256, 2.0),     # edgemm_m8n128k64x4: weights [K,N], overwrites
    "edgemm_bt": (256, 2.0),  # edgemm_m8n128k64x4_bt: weights [N,K], overwrites
    "residual": (256, 2.0),   # flat_gemm_m8n128k64x4_bz1: weights [K,N], adds into C
    "residual_bt": (256, 2.0),  # gemm_m8n32k256x8_bt: weights [N,K], adds into C
    "ffn_bt": (256, 2.0),     # two [N,K] products, bias and GELU between them
    "int8": (16, 1.0),        # fastgemv_int8 with a scale per output channel
    "int4": (4, 0.5),         # fastgemv_int4 with a scale per output channel and a zero point
    "w8a8": (8, 1.0),         # gemv_i8i8_i32 followed by dequant_i32_f16
}
MOST_WEIGHTS = 13824 * 5120  # of one matrix; the largest listed


def listed():
    return [
        # smallest calls: launch latency and host work, one token through a narrow feed-forward pair
        {"name": "ffn_m1_small", "kind": "ffn_bt", "M": 1, "N": 2048, "K": 1024},
        # one token through a 4096-wide attention projection
        {"name": "gemv_4096", "kind": "gemv", "M": 1, "N": 4096, "K": 4096},
        # batch of eight through an up-projection, weights as a checkpoint's [in, out] matrix
        {"name": "edgemm_m8_up", "kind": "edgemm", "M": 8, "N": 11008, "K": 4096},
        # the library's headline shape with sixteen rows, both layouts
        {"name": "edgemm_m16_8192", "kind": "edgemm", "M": 16, "N": 8192, "K": 8192},
        {"name": "edgemm_bt_m16_8192", "kind": "edgemm_bt", "M": 16, "N": 8192, "K": 8192},
        # feed-forward block of a text-to-video DiT: up-projection, bias, GELU, down-projection, bias
        {"name": "ffn_m16_dit", "kind": "ffn_bt", "M": 16, "N": 12288, "K": 3072},
        # one token against int8 weights, and a batch of eight
        {"name": "int8_m1_8192", "kind": "int8", "M": 1, "N": 8192, "K": 8192},
        {"name": "int8_m8_up", "kind": "int8", "M": 8, "N": 14336, "K": 4096},
        # four sequences against int4 weights, down-projection
        {"name": "int4_m4_down", "kind": "int4", "M": 4, "N": 4096, "K": 14336},
        # int8 activations, exact integer sums, then scales
        {"name": "w8a8_m4_5120", "kind": "w8a8", "M": 4, "N": 5120, "K": 5120},
        # a decode batch of 48 through a down-projection that adds into the residual stream
        {"name": "residual_bt_m48_down", "kind": "residual_bt", "M": 48, "N": 4096, "K": 11008},
        # a prompt chunk of 256 tokens through an up-projection
        {"name": "edgemm_m256_up", "kind": "edgemm", "M": 256, "N": 13824, "K": 5120},
    ]


def _log_uniform(rng, low, high):
    return low * (high / low) ** rng.random()


def draw(rng):
    kind = rng.choice(sorted(KINDS))
    rows = int(_log_uniform(rng, 1, KINDS[kind][0] + 0.999))
    while True:
        n = 128 * round(_log_uniform(rng, 1024, 28672) / 128)
        k = 128 * round(_log_uniform(rng, 1024, 16384) / 128)
        # the feed-forward pair holds two matrices
        if 2 ** 22 <= n * k * (2 if kind == "ffn_bt" else 1) <= MOST_WEIGHTS:
            return {"kind": kind, "M": rows, "N": n, "K": k}


def prepare(case, seed):
    dev = torch.device("cuda")
    g = torch.Generator(device=dev)
    g.manual_seed(seed)
    kind, M, N, K = case["kind"], case["M"], case["N"], case["K"]

    def normal(shape, std=1.0):
        return (torch.randn(shape, generator=g, device=dev) * std).half()

    st = {"kind": kind}
    if kind == "w8a8":
        st["x"] = torch.randint(-127, 128, (M, K), generator=g, device=dev, dtype=torch.int8)
        st["x_scale"] = 3.0 / 127.0
    else:
        st["x"] = normal((M, K))
    if kind in ("int8", "w8a8"):
        st["w"] = torch.randint(-127, 128, (N, K), generator=g, device=dev, dtype=torch.int8)
    elif kind == "int4":
        st["w"] = torch.randint(0, 256, (N, K // 2), generator=g, device=dev, dtype=torch.uint8)
    else:
        st["w"] = normal((K, N) if kind in ("edgemm", "residual") else (N, K), 0.02)
    if kind in ("int8", "int4", "w8a8"):
        st["scale"] = (torch.rand(N, generator=g, device=dev) * 0.009 + 0.001).half()
    if kind == "w8a8":
        st["acc"] = torch.empty((M, N), device=dev, dtype=torch.int32)
    if kind in ("residual", "residual_bt"):
        st["residual"] = normal((M, N))
    if kind == "ffn_bt":
        st["b1"] = normal(N, 0.02)
        st["w2"] = normal((K, N), 0.02)
        st["b2"] = normal(K, 0.02)
        st["h"] = torch.empty((M, N), device=dev, dtype=torch.half)
        st["c"] = torch.empty((M, K), device=dev, dtype=torch.half)
    else:
        st["c"] = torch.empty((M, N), device=dev, dtype=torch.half)
    return st


def run(st):
    kind, x, w, c = st["kind"], st["x"], st["w"], st["c"]
    if kind == "gemv":
        sg.fastgemv(w, x, c)
    elif kind == "edgemm":
        sg.edgemm_m8n128k64x4(x, w, c)
    elif kind == "edgemm_bt":
        sg.edgemm_m8n128k64x4_bt(x, w, c)
    elif kind == "residual":
        c.copy_(st["residual"])
        sg.flat_gemm_m8n128k64x4_bz1(x, w, c, 1)
    elif kind == "residual_bt":
        c.copy_(st["residual"])
        sg.gemm_m8n32k256x8_bt(x, w, c)
    elif kind == "ffn_bt":
        sg.ffn_bt(x, w, st["b1"], st["w2"], st["b2"], st["h"], c, "gelu")
        return {"h": st["h"], "c": c}
    elif kind == "int8":
        sg.fastgemv_int8(w, x, c, st["scale"])
    elif kind == "int4":
        sg.fastgemv_int4(w, x, c, st["scale"], 1.0, 8.0)
    else:
        sg.gemv_i8i8_i32(w, x, st["acc"])
        sg.dequant_i32_f16(st["acc"], st["scale"], st["x_scale"], c)
        return {"acc": st["acc"], "c": c}
    return c


def work(case):
    kind, M, N, K = case["kind"], case["M"], case["N"], case["K"]
    x_bytes = 1 if kind == "w8a8" else 2
    n = {"bytes": KINDS[kind][1] * N * K + x_bytes * M * K + 2 * M * N, "flops": 2.0 * M * N * K}
    if kind in ("int8", "int4", "w8a8"):
        n["bytes"] += 2 * N
    if kind in ("residual", "residual_bt"):
        n["bytes"] += 2 * M * N
    if kind == "w8a8":
        n["bytes"] += 4 * M * N
    if kind == "ffn_bt":
        n["bytes"] += 2 * N * K + 2 * M * K + 2 * (N + K)
        n["flops"] *= 2
    return n


def tolerance(case):
    # fp32 sums rounded once to fp16 (twice along the feed-forward pair), measured against the same
    # formulas in 64 bits over the listed cases: rel 2.1e-4, max 4.9e-4 (half a unit in the last
    # place), the pair 3.1e-4 and 1.4e-3.  Integer sums are exact.
    if case["kind"] == "ffn_bt":
        return {"rel": 1.2e-3, "max": 6e-3}
    return {"rel": 8e-4, "max": 2e-3}


def exact(case, seed):
    # the operator's formula in float64, no rounding between the products of the feed-forward pair
    st = prepare(case, seed)
    kind, x = st["kind"], st["x"].double()
    if kind == "int4":
        nibbles = torch.stack((st["w"] & 15, st["w"] >> 4), dim=-1)  # even element in the low nibble
        w = nibbles.flatten(1).double().sub_(8.0)
    else:
        w = st["w"].double()
    sums = x @ (w if kind in ("edgemm", "residual") else w.t())
    if kind == "ffn_bt":
        h = torch.nn.functional.gelu(sums + st["b1"].double())
        return {"h": h, "c": h @ st["w2"].double().t() + st["b2"].double()}
    if kind == "w8a8":
        return {"acc": sums.round().int(), "c": sums * st["scale"].double() * st["x_scale"]}
    if kind in ("int8", "int4"):
        return sums * st["scale"].double()
    if kind in ("residual", "residual_bt"):
        return sums + st["residual"].double()
    return sums
