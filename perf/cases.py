"""The work that users of this library have it do, as cases whose time can be taken: the quantized matrix products of a
language model's layers, through the public entry points (arcinferzero_amd.Engine), from one token to a prompt chunk.

A case is one of three kinds of call sequence:
  proj  one projection: quantize the chunk's f32 rows, multiply with one weight matrix (attention projections, output
        heads, the decode step's building block)
  ffn   a feed-forward block: RMS norm + quantization, gate and up (one launch for one token; SwiGLU fused into the up
        product for chunks), SwiGLU + quantization, down
  moe   a mixture-of-experts layer: quantize the chunk, route, the experts' gate / up / down, combine into the residual

listed() names twelve of them, draw() gives more of the same ranges.
"""
import math

import numpy as np
import torch

import arcinferzero_amd as az
from arcinferzero_amd.binding import lib

TYPES = {"Q4_K": az.Q4_K, "Q5_K": az.Q5_K, "Q6_K": az.Q6_K, "Q8_0": az.Q8_0, "Q4_0": az.Q4_0, "IQ4_XS": az.IQ4_XS,
         "IQ4_NL": az.IQ4_NL, "MXFP4": az.MXFP4, "Q3_K": az.Q3_K, "IQ3_S": az.IQ3_S, "IQ3_XXS": az.IQ3_XXS}
EPS = 1e-6


def listed():
    return [
        # -- one token: a decode step
        # a small model's attention projection: as short as a call gets, launches and host work are most of it
        dict(name="proj_2048x2048_q4k_1", kind="proj", type="Q4_K", N=2048, K=2048, T=1),
        # the dense benchmark model's FFN in the usual 4-bit mix (gate and up Q4_K, down Q6_K)
        dict(name="ffn_5120x17408_q4k_1", kind="ffn", type="Q4_K", down="Q6_K", E=5120, F=17408, T=1, two_pass=False),
        # its output head: the largest matrix of a model, read once per token
        dict(name="head_151936x5120_q6k_1", kind="proj", type="Q6_K", N=151936, K=5120, T=1),
        # one token through a mixture-of-experts layer (128 experts, 8 used)
        dict(name="moe_128x8_q4k_1", kind="moe", type="Q4_K", down="Q4_K", NE=128, NU=8, E=2048, F=768, T=1),
        # -- a few tokens: speculative or batched decode
        # two-pass inputs (the more exact activation mode), two sequences, 8-bit weights
        dict(name="ffn_4096x12288_q8_0_2_two_pass", kind="ffn", type="Q8_0", down="Q8_0", E=4096, F=12288, T=2, two_pass=True),
        # a batch of eight sequences through a dense FFN
        dict(name="ffn_5120x17408_q5k_8", kind="ffn", type="Q5_K", down="Q5_K", E=5120, F=17408, T=8, two_pass=False),
        # a batch of forty through an expert layer: few tokens for each expert
        dict(name="moe_128x8_iq4xs_40", kind="moe", type="IQ4_XS", down="IQ4_XS", NE=128, NU=8, E=2048, F=768, T=40),
        # -- prompt chunks
        # a prompt of an odd length, most of a tile of padding
        dict(name="ffn_5120x17408_q4k_300", kind="ffn", type="Q4_K", down="Q6_K", E=5120, F=17408, T=300, two_pass=False),
        # the first benchmark configuration
        dict(name="proj_4096x4096_q8_0_512", kind="proj", type="Q8_0", N=4096, K=4096, T=512),
        # a longer one in a 3-bit model
        dict(name="ffn_4096x12288_q3k_1000", kind="ffn", type="Q3_K", down="Q5_K", E=4096, F=12288, T=1000, two_pass=False),
        # the expert-layer benchmark configuration
        dict(name="moe_128x8_q4k_4096", kind="moe", type="Q4_K", down="Q4_K", NE=128, NU=8, E=2048, F=768, T=4096),
        # the headline benchmark configuration: the largest chunk
        dict(name="proj_17408x5120_q4k_8192", kind="proj", type="Q4_K", N=17408, K=5120, T=8192),
    ]


def _log(rng, lo, hi, step=1):
    """A whole multiple of `step` between lo and hi, even over the logarithm."""
    v = math.exp(rng.uniform(math.log(lo), math.log(hi)))
    return max(lo, min(hi, int(round(v / step)) * step))


def draw(rng):
    while True:
        kind = rng.choice(("proj", "proj", "ffn", "moe"))
        # (the K-quants and Q8_0 are what most models come in; the others are seen less often)
        t = rng.choice(("Q4_K", "Q4_K", "Q4_K", "Q6_K", "Q6_K", "Q5_K", "Q5_K", "Q8_0", "Q8_0", "Q4_0", "IQ4_XS", "IQ4_NL",
                        "MXFP4", "Q3_K", "IQ3_S", "IQ3_XXS"))
        if kind == "proj":
            # N need not be whole tiles: router-sized and vocabulary-sized matrices are not
            c = dict(kind=kind, type=t, N=_log(rng, 256, 17408, rng.choice((1, 16, 128))), K=_log(rng, 1024, 17408, 256), T=_log(rng, 1, 8192))
            if rng.random() < 0.1:
                c.update(N=_log(rng, 32000, 151936), K=_log(rng, 1024, 5120, 256), T=_log(rng, 1, 64))
        elif kind == "ffn":
            e = _log(rng, 1024, 5120, 256)
            c = dict(kind=kind, type=t, down=t if rng.random() < 0.6 else "Q6_K", E=e, F=_log(rng, 2 * e, 7 * e // 2, 256), T=_log(rng, 1, 4096), two_pass=False)
            c["two_pass"] = rng.random() < 0.1
        else:
            c = dict(kind=kind, type=t, down=t, NE=rng.choice((32, 64, 128)), NU=rng.choice((4, 8)), E=_log(rng, 1024, 3072, 256),
                     F=_log(rng, 512, 1536, 256), T=_log(rng, 1, 4096))
        w = work(c)
        held = work(dict(c, T=4096))["bytes"] if kind == "moe" else w["bytes"]   # (every expert's weights, used or not)
        # (never more than the headline case: the slower types and two passes are allowed half of its products)
        if w["flops"] * (2 if c.get("two_pass") else 1) <= 7e11 and held <= 1.0e9:
            return c


# ---------------------------------------------------------------- what a pass cannot do without
def work(case):
    T = case["T"]
    if case["kind"] == "proj":
        N, K = case["N"], case["K"]
        return {"bytes": az.gguf_bytes(TYPES[case["type"]], N, K) + 4 * T * (K + N), "flops": 2.0 * T * N * K}
    E, F = case["E"], case["F"]
    gu, dn = az.gguf_bytes(TYPES[case["type"]], 2 * F, E), az.gguf_bytes(TYPES[case["down"]], E, F)
    if case["kind"] == "ffn":
        return {"bytes": gu + dn + 4 * T * 2 * E + 4 * E, "flops": 2.0 * T * 3 * E * F}
    NE, NU = case["NE"], case["NU"]
    hit = NE * (1.0 - (1.0 - NU / NE) ** T)   # experts that T tokens reach, on average
    return {"bytes": hit * (gu + dn) + 4 * T * (3 * E + NE), "flops": 2.0 * T * NU * 3 * E * F}


def tolerance(case):
    # one projection: exact integer block sums, f32 from there on
    if case["kind"] == "proj":
        return {"rel": 1e-5}
    # a block quantizes again in the middle: values on a rounding boundary of the int8 grid may fall either way when the
    # f32 sums in front of it are added in another order (about one in 10^5, each worth 1/127 of its block's maximum)
    return {"rel": 5e-4}


# ---------------------------------------------------------------- a user's buffers
class _Array:
    """A device buffer of the library, seen by torch without a copy; freed with the last of its tensors."""

    def __init__(self, shape):
        self.shape = tuple(shape)
        self.buf = az.Runtime.alloc(4 * int(np.prod(self.shape)))
        self.__cuda_array_interface__ = {"shape": self.shape, "typestr": "<f4", "version": 2,
                                         "data": (int(lib.arcz_mem_ptr(self.buf.h)), False)}

    def tensor(self):
        return torch.as_tensor(self, device="cuda")

    def __del__(self):
        self.buf.free()


def _rows(shape, gen, std=1.0, outliers=False):
    a = _Array(shape)
    t = torch.randn(shape, generator=gen, device="cuda") * std
    if outliers:   # activations have a few large values: one in 97 four times its size
        t *= 1.0 + 3.0 * (torch.rand(shape, generator=gen, device="cuda") < 1.0 / 97)
    a.tensor().copy_(t)
    return a


_pools = {}


def _weights(name, rows, K, gen):
    """GGUF rows of normal weights: every superblock drawn from a pool of 4096 that the library's quantizer made."""
    q = TYPES[name]
    if name not in _pools:
        _pools[name] = torch.from_numpy(az.gen_weights(q, 7, 16, 65536, 0.02)).view(4096, -1).cuda()
    pool = _pools[name]
    out = np.empty((rows * (K // 256), pool.shape[1]), np.uint8)
    for i in range(0, out.shape[0], 1 << 20):
        n = min(1 << 20, out.shape[0] - i)
        out[i:i + n] = pool[torch.randint(4096, (n,), generator=gen, device="cuda")].cpu().numpy()
    return out.reshape(-1)


def _chunk_rows(T):
    """The rows that a chunk of T tokens is laid out for: whole 16s, from 128 tokens on whole 128s."""
    return (T + 15) // 16 * 16 if T < 128 else (T + 127) // 128 * 128


class _State:
    def __init__(self, case):
        self.case, self.eng = case, None

    def __del__(self):
        if self.eng is not None:
            self.eng.close()   # (its weights with it)


def prepare(case, seed):
    az.Runtime.init(0)
    gen = torch.Generator(device="cuda")
    gen.manual_seed(seed)
    s = _State(case)
    T = s.T = case["T"]
    Mp = s.Mp = _chunk_rows(T)
    out_rows = Mp if T > 8 else T
    if case["kind"] == "proj":
        N, K = case["N"], case["K"]
        s.eng = az.Engine(Mp, K)
        s.w = s.eng.make_weight(TYPES[case["type"]], N, K, _weights(case["type"], N, K, gen))
        s.x = _rows((T, K), gen, outliers=True)
        s.y = _Array((out_rows, N))
    elif case["kind"] == "ffn":
        E, F = case["E"], case["F"]
        s.eng = az.Engine(Mp, max(E, F))
        if case["two_pass"]:
            s.eng.two_pass(True)
        s.g, s.u = (s.eng.make_weight(TYPES[case["type"]], F, E, _weights(case["type"], F, E, gen)) for _ in range(2))
        s.d = s.eng.make_weight(TYPES[case["down"]], E, F, _weights(case["down"], E, F, gen))
        s.x = _rows((T, E), gen, outliers=True)
        s.norm = _rows((E,), gen, std=0.1)
        s.norm.tensor().add_(1.0)
        s.gu = _Array((out_rows, 2 * F))
        s.y = _Array((out_rows, E))
    else:
        NE, E, F = case["NE"], case["E"], case["F"]
        s.eng = az.Engine(Mp, max(E, F))
        q = TYPES[case["type"]]
        s.layer = s.eng.make_moe_layer(q, _weights(case["type"], NE * F, E, gen), _weights(case["type"], NE * F, E, gen),
                                       _weights(case["down"], NE * E, F, gen), NE, case["NU"], E, F)
        s.h = _rows((T, E), gen, outliers=True)
        s.logits = _rows((T, NE), gen)
        s.y = _rows((T, E), gen, std=0.5)   # the residual stream the layer adds to
    s.out = s.y.tensor()[:T]
    torch.cuda.synchronize()
    return s


def run(s):
    c, eng, T, Mp = s.case, s.eng, s.T, s.Mp
    if c["kind"] == "proj":
        eng.quantize(s.x.buf, c["K"], c["K"], Mp, T)
        eng.matmul("proj", s.w, Mp, s.y.buf, c["N"])
    elif c["kind"] == "ffn":
        E, F = c["E"], c["F"]
        eng.rmsnorm_quant(s.x.buf, 0, s.norm.buf, E, Mp, T, EPS)
        if T > 8 and not c["two_pass"]:
            eng.matmul("ffn_gate", s.g, Mp, s.gu.buf, F)
            eng.matmul("ffn_up", s.u, Mp, s.gu.buf, F, 0, 2)   # silu(gate) * up in the product's epilogue
            eng.swiglu_quant(s.gu.buf, F, Mp, T, fused=1)
        else:
            if T != 1 or not eng.gemv_gu(s.g, s.u, Mp, s.gu.buf):
                eng.matmul("ffn_gate", s.g, Mp, s.gu.buf, 2 * F)
                eng.matmul("ffn_up", s.u, Mp, s.gu.buf, 2 * F, F)
            eng.swiglu_quant(s.gu.buf, F, Mp, T)
        eng.matmul("ffn_down", s.d, Mp, s.y.buf, E)
    else:
        eng.quantize(s.h.buf, c["E"], c["E"], Mp, T)
        eng.layer_moe(s.layer, s.logits.buf, c["NE"], s.y.buf, T, Mp)
    return s.out
