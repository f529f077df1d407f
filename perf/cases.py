"""The work that a user of this backend has it do, as cases to be timed: dense matrices of every weight format from one token to a
prefill chunk, routed-expert layer steps over the same range, and decode attention over the latent KV cache.

Everything goes through the entry points a host calls: the kc_* functions of libnslm_hip.so (include/kernels_hip.h) on device
pointers and the default stream, and moe.MoeStack, the expert layer host.  Inputs live in torch tensors on the GPU."""
import ctypes as C
import math

import torch

from nanoseedlm_amd import backend, moe, packs

BF16, P3, Q8, Q4, P4 = packs.MF_BF16, packs.MF_SEED4, packs.MF_Q8, packs.MF_Q4, packs.MF_SEED4P4
FORMATS = {"bf16": BF16, "p3": P3, "q8": Q8, "q4": Q4, "p4": P4}
BYTES_A_WEIGHT = {"bf16": 2.0, "p3": 0.5, "q8": 1.0 + 4.0 / 64, "q4": 0.5 + 4.0 / 64, "p4": 36.0 / 64}
MV_MAXT = 8            # tokens up to which a host takes the matvec (kernels_hip.h)
N_HEAD, LATENT, ROPE = 16, 512, 64   # the latent attention's shape
SPLITS, CHUNK = 32, 128              # key splits and their least length, as the whole-model host passes them
MOST_FLOPS = 1.5e11    # a drawn case's bound: the largest listed one's


def listed():
    return [
        # one token through a projection of a 2048-wide model: the smallest call a decode step makes
        dict(name="mv_p4_one", kind="mv", fmt="p4", T=1, R=2048, K=2048),
        # a few sequences decoding together, rows whose 64-weight chunks (45) fill no wave
        dict(name="mv_p3_rows", kind="mv", fmt="p3", T=6, R=2880, K=2880),
        # a decode batch too large for the matvec through a square projection
        dict(name="mm_p4_batch", kind="mm", fmt="p4", T=48, R=4096, K=4096),
        # a prefill chunk through an up projection
        dict(name="mm_p4_prefill", kind="mm", fmt="p4", T=512, R=14336, K=4096),
        # a prompt of no round length through an affine int4 projection
        dict(name="mm_q4_ragged", kind="mm", fmt="q4", T=301, R=2880, K=2880),
        # the vocabulary's logits of a decode batch
        dict(name="head_bf16", kind="mm", fmt="bf16", T=16, R=151936, K=2048),
        # an expert layer step for one token, the layers of a stack one after the other: the latency of single-user decode
        dict(name="moe_p4_one", kind="moe", fmt="p4", router="softmax", T=1, layers=4, E=128, k=8, d=2048, ff=768),
        # the same for a small decode batch
        dict(name="moe_p4_rows", kind="moe", fmt="p4", router="softmax", T=8, layers=2, E=128, k=8, d=2048, ff=768),
        # few, wide experts in the three-coefficient format
        dict(name="moe_p3_rows", kind="moe", fmt="p3", router="softmax", T=3, layers=1, E=64, k=4, d=2880, ff=2880),
        # a server's decode batch
        dict(name="moe_p4_batch", kind="moe", fmt="p4", router="softmax", T=64, layers=1, E=128, k=8, d=2048, ff=768),
        # a prefill chunk
        dict(name="moe_p4_prefill", kind="moe", fmt="p4", router="softmax", T=2048, layers=1, E=128, k=8, d=2048, ff=768),
        # decode attention: sequences of different lengths over an FP8 latent cache
        dict(name="attn_fp8", kind="attn", fmt="fp8", T=16, ctx=4096),
    ]


def _log(rng, lo, hi):
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    """A case of the listed ones' ranges: any token count, output widths down to odd ones, input widths in whole 64-weight chunks."""
    kind = rng.choice(("mv", "mm", "mm", "moe", "moe", "moe", "attn"))
    if kind == "attn":
        while True:
            c = dict(kind=kind, fmt=rng.choice(("fp8", "fp8", "bf16")), T=_log(rng, 1, 32), ctx=_log(rng, 100, 16384))
            if c["T"] * c["ctx"] <= 200000:
                return c
    if kind == "moe":
        # (the sigmoid router is the three-coefficient family's, too; either format takes either)
        c = dict(kind=kind, fmt=rng.choice(("p4", "p4", "p3")), router=rng.choice(("softmax", "softmax", "softmax", "sigmoid")), T=_log(rng, 1, 2048))
        c["E"] = rng.choice((16, 32, 64, 128))
        c["k"] = rng.choice((2, 4, 8))
        c["layers"] = rng.choice((1, 2, 4)) if c["T"] <= 8 else 1
        while True:
            c["d"], c["ff"] = 64 * _log(rng, 8, 64), 64 * _log(rng, 4, 48)
            if c["d"] * c["ff"] <= 2880 * 2880 and c["layers"] * work(c)["flops"] <= MOST_FLOPS:
                return c
    while True:
        fmt = rng.choice(("p4", "p4", "p4", "p3", "p3", "q4", "q8", "bf16"))
        T = _log(rng, 1, MV_MAXT) if kind == "mv" else _log(rng, MV_MAXT + 1, 2048)
        c = dict(kind=kind, fmt=fmt, T=T, R=_log(rng, 64, 152000 if fmt == "bf16" else 16384), K=64 * _log(rng, 4, 224))
        if c["R"] * c["K"] <= 320e6 and work(c)["flops"] <= MOST_FLOPS:
            return c


# ---- inputs -----------------------------------------------------------------------------------------------------------------

def _ptr(t):
    return C.c_void_p(t.data_ptr())


def _words(g, n):
    """n uniform 16-bit words as an int16 tensor."""
    return torch.randint(-32768, 32768, (n,), dtype=torch.int16, device="cuda", generator=g)


def _matrix(g, fmt, R, K):
    """A weight matrix [R][K] of seeded random records: (WSlice, the tensors that hold its streams)."""
    w, nb = backend.WSlice(), R * K // 8
    if fmt in ("p4", "p3"):
        seeds = _words(g, nb)
        seeds[seeds == 0] = 1
        keep = [seeds, _words(g, nb)]
        w.eb = -22
        if fmt == "p4":
            keep.append(torch.randint(0, 256, ((nb + 1) // 2,), dtype=torch.uint8, device="cuda", generator=g))
            w.p[3] = keep[2].data_ptr()
        w.p[0], w.p[1] = keep[0].data_ptr(), keep[1].data_ptr()
    elif fmt in ("q4", "q8"):
        n = R * (K // 64)
        top = 16 if fmt == "q4" else 256
        scale = (0.005 + 0.015 * torch.rand(n, device="cuda", generator=g)) * (16.0 / top)
        scale = scale.bfloat16()
        zero = torch.randint(0, top, (n,), device="cuda", generator=g).float()
        keep = [_words(g, R * K // (4 if fmt == "q4" else 2)), scale, (-zero * scale.float()).bfloat16()]
        w.gs = 6
        for i in range(3):
            w.p[i] = keep[i].data_ptr()
    else:
        keep = [torch.empty(R, K, dtype=torch.bfloat16, device="cuda").normal_(0.0, 0.02, generator=g)]
        w.p[0] = keep[0].data_ptr()
    return w, keep


def _rows(g, T, n):
    """Activations: BF16 values held in f32, as an engine hands them over."""
    return torch.randn(T, n, device="cuda", generator=g).bfloat16().float()


class _Mv:
    """kc_mv: y[t] = bf16(W x[t]) for up to MV_MAXT tokens."""

    def __init__(self, c, g):
        w, self.keep = _matrix(g, c["fmt"], c["R"], c["K"])
        self.x = _rows(g, c["T"], c["K"])
        self.y = torch.empty(c["T"], c["R"], device="cuda")
        self.call = backend.hip().kc_mv
        self.args = (None, FORMATS[c["fmt"]], w, c["K"], c["R"], _ptr(self.x), c["K"], _ptr(self.y), c["R"], c["T"], 0, None)

    def run(self):
        self.call(*self.args)
        return self.y


class _Mm:
    """kc_mm_packed: the same product for more tokens, activations as BF16 bits."""

    def __init__(self, c, g):
        w, self.keep = _matrix(g, c["fmt"], c["R"], c["K"])
        self.x = torch.randn(c["T"], c["K"], device="cuda", generator=g).bfloat16()
        self.y = torch.empty(c["T"], c["R"], device="cuda")
        self.call = backend.hip().kc_mm_packed
        self.args = (None, FORMATS[c["fmt"]], w, c["K"], c["R"], _ptr(self.x), c["K"], _ptr(self.y), c["R"], c["T"], 0, None)

    def run(self):
        self.call(*self.args)
        return self.y


class _Moe:
    """A stack of routed-expert layers, all experts resident: a pass is one step through each layer."""

    def __init__(self, c, g, seed):
        self.T, self.sigmoid = c["T"], c["router"] == "sigmoid"
        self.st = moe.MoeStack(c["layers"], c["E"], c["k"], c["d"], c["ff"], fmt=FORMATS[c["fmt"]], max_rows=c["T"],
                               router=moe.ROUTE_SIGMOID if self.sigmoid else moe.ROUTE_SOFTMAX)
        backend.check(self.st.L.nslm_moe_fill_random(self.st.h, C.c_uint64(seed * 2654435761 + 1), -22, C.c_float(0.035)), "nslm_moe_fill_random")
        self.st.finalize()
        self.xs = [_rows(g, c["T"], c["d"]) for _ in range(c["layers"])]
        self.res = [_rows(g, c["T"], c["d"]) for _ in range(c["layers"])] if self.sigmoid else None
        self.out = [torch.empty(c["T"], c["d"], device="cuda") for _ in range(c["layers"])]

    def run(self):
        for l, (x, y) in enumerate(zip(self.xs, self.out)):
            if self.sigmoid:   # this composition adds to the residual stream in place
                y.copy_(self.res[l])
            self.st.step(None, l, _ptr(x), self.T, _ptr(y))
        return self.out

    def __del__(self):
        if hasattr(self, "st"):
            self.st.close()


class _Attn:
    """kc_mla_attn: absorbed latent attention of one new token for each of T sequences, between half of ctx and ctx positions long.
    The cache is written by kc_mla_rope, as a prefill writes it."""

    def __init__(self, c, g):
        T, ctx, L, fp8 = c["T"], c["ctx"], backend.hip(), c["fmt"] == "fp8"
        e = 1 if fp8 else 2
        self.k = torch.zeros(T * ctx * ROPE * e, dtype=torch.uint8, device="cuda")
        self.v = torch.zeros(T * ctx * LATENT * e, dtype=torch.uint8, device="cuda")
        self.ks = torch.zeros(T * ctx * ROPE // 32, dtype=torch.uint8, device="cuda")
        self.vs = torch.zeros(T * ctx * LATENT // 32, dtype=torch.uint8, device="cuda")
        kv = backend.KvView()
        kv.a.k, kv.a.v, kv.a.ks, kv.a.vs = self.k.data_ptr(), self.v.data_ptr(), self.ks.data_ptr(), self.vs.data_ptr()
        kv.nv, kv.fmt = T * ctx, backend.KV_FP8 if fp8 else backend.KV_BF16
        a = backend.MlaArgs(N_HEAD, LATENT, CHUNK, SPLITS, 1.0 / math.sqrt(128 + ROPE))
        a.pad[0] = ROPE
        inv = 10000.0 ** (-2.0 * torch.arange(ROPE // 2, device="cuda") / ROPE)
        slot = torch.zeros(ctx, 4, dtype=torch.int32, device="cuda")   # RowInfo: position, the sequence's first cache row
        slot[:, 0] = torch.arange(ctx, device="cuda")
        qr = torch.zeros(ctx, N_HEAD * ROPE, device="cuda")
        for t in range(T):
            slot[:, 1] = t * ctx
            kr, lat = _rows(g, ctx, ROPE), _rows(g, ctx, LATENT)
            L.kc_mla_rope(None, a, _ptr(qr), _ptr(kr), _ptr(lat), kv, _ptr(slot), _ptr(inv), ctx)
        self.ri = torch.zeros(T, 4, dtype=torch.int32, device="cuda")
        self.ri[:, 0] = torch.randint(ctx // 2, ctx, (T,), device="cuda", generator=g)
        self.ri[:, 1] = torch.arange(T, device="cuda") * ctx
        self.ql, self.qr = 0.25 * _rows(g, T, N_HEAD * LATENT), _rows(g, T, N_HEAD * ROPE)
        self.part = torch.empty(T * N_HEAD * SPLITS * (LATENT + 2), device="cuda")
        self.o = torch.empty(T, N_HEAD, LATENT, device="cuda")
        self.call = L.kc_mla_attn
        self.args = (None, a, _ptr(self.ql), _ptr(self.qr), kv, _ptr(self.ri), _ptr(self.part), _ptr(self.o), T)

    def run(self):
        self.call(*self.args)
        return self.o


def prepare(case, seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    if case["kind"] == "moe":
        return _Moe(case, g, seed)
    return {"mv": _Mv, "mm": _Mm, "attn": _Attn}[case["kind"]](case, g)


def run(state):
    return state.run()


# ---- what a pass cannot do without ---------------------------------------------------------------------------------------------

def work(case):
    T = case["T"]
    if case["kind"] == "attn":   # every cached position of every sequence once, at the mean length
        n, row = 0.75 * T * case["ctx"], LATENT + ROPE
        cached = row * (1 + 1 / 32) if case["fmt"] == "fp8" else 2 * row
        return {"bytes": n * cached + 4 * T * N_HEAD * (row + LATENT), "flops": 2.0 * n * N_HEAD * (row + LATENT)}
    if case["kind"] == "moe":    # the distinct experts that T tokens choose, the router, the rows
        E, k, d, ff = case["E"], case["k"], case["d"], case["ff"]
        distinct = E * (1 - (1 - k / E) ** T)
        one = distinct * 3 * d * ff * BYTES_A_WEIGHT[case["fmt"]] + 2 * E * d + 8 * T * d
        return {"bytes": case["layers"] * one, "flops": case["layers"] * 2.0 * T * (3 * k * d * ff + E * d)}
    R, K = case["R"], case["K"]
    return {"bytes": R * K * BYTES_A_WEIGHT[case["fmt"]] + T * K * (4 if case["kind"] == "mv" else 2) + 4 * T * R, "flops": 2.0 * T * R * K}


def tolerance(case):
    """Every path rounds its results to BF16 (8 bits).  The matvec keeps weights, activations and sums in f32 before that, so another
    order of the sums moves few results, by one unit; the others also take BF16 activations, weights or probabilities."""
    return {"rel": 2e-3} if case["kind"] == "mv" else {"rel": 1e-2}
