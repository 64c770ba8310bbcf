"""The work that a serving program has this library do, as cases that can be timed and compared.

Each case is one pass through the public entry points as such a program calls them: single linears from one token to a
chunk of a prompt, the four projections of a prefill step, decode attention over the cache layouts, filling a cache,
a mixture-of-experts layer, and whole decode steps recorded once and replayed.  Device memory comes from torch; the
library sees plain pointers.
"""
import ctypes
import math
import os
import random
import sys

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.getcwd(), "mojo-linuxperiments_amd"))
import mi355_int8 as mi  # noqa: E402  (after torch: both then share one HIP runtime)
import workload  # noqa: E402

D = 128          # head dimension
PAGE = 64        # tokens of a page of the tiled cache
ROW_PAGE = 16    # tokens of a page of the row-major cache
PROJECTIONS = {name: (K, N) for name, K, N in workload.PROJECTIONS}


# ---- the cases -------------------------------------------------------------------------------------------------------

def listed():
    return [
        # one generated token through the fused QKV projection: the smallest call of a decode loop
        dict(name="linear_m1_qkv", kind="linear", M=1, K=4096, N=6144),
        # a square projection for a batch of 32 sequences
        dict(name="linear_m32", kind="linear", M=32, K=4096, N=4096),
        # the gate projection for a short prompt: too many rows for the decode kernels, too few to fill the chip with tiles
        dict(name="linear_m200_gate", kind="linear", M=200, K=4096, N=14336),
        # a ragged chunk of a prompt through the four projections of a layer
        dict(name="prefill_m509", kind="prefill", M=509),
        # the same for 2048 tokens: the largest contraction
        dict(name="prefill_m2048", kind="prefill", M=2048),
        # a prompt of 2048 tokens on its way into the cache: keys and values rotated, quantized and laid out
        dict(name="kv_prefill_t2048", kind="kv_prefill", B=1, Hkv=8, T=2048),
        # decode attention of 16 sequences of equal length, dense cache
        dict(name="attention_b16_t4096", kind="attention", layout="tiled", B=16, Hq=32, Hkv=8, T=4096, ragged=False,
             append=False),
        # the same as a server with a page table has it: 24 sequences of mixed lengths, the new token appended first
        dict(name="attention_paged_b24", kind="attention", layout="tiled_paged", B=24, Hq=32, Hkv=8, T=3001, ragged=True,
             append=True),
        # a mixture-of-experts layer over 512 tokens
        dict(name="moe_t512", kind="moe", T=512, H=2048, I=768, E=128, topk=8),
        # a whole decode step of 16 sequences (four decoder layers, recorded and replayed)
        dict(name="decode_b16_t4096", kind="decode", B=16, T=4096, layers=4, moe=False),
        # the same for a single conversation: latency
        dict(name="decode_b1_t1531", kind="decode", B=1, T=1531, layers=4, moe=False),
        # a decode step of 16 sequences whose layers have experts in place of the dense FFN
        dict(name="decode_moe_b16_t1024", kind="decode", B=16, T=1024, layers=2, moe=True),
    ]


def _log(rng, lo, hi):
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    kind = rng.choice(["linear", "linear", "linear", "prefill", "kv_prefill", "attention", "attention", "moe", "decode"])
    if kind == "linear":
        if rng.random() < 0.5:
            K, N = rng.choice(list(PROJECTIONS.values()) + [(4096, 4096)])
        else:
            K, N = 128 * _log(rng, 8, 112), 16 * _log(rng, 32, 896)
        return dict(kind=kind, M=_log(rng, 1, 1024), K=K, N=N)
    if kind == "prefill":
        return dict(kind=kind, M=_log(rng, 256, 2048))
    if kind == "kv_prefill":
        return dict(kind=kind, B=rng.randint(1, 4), Hkv=rng.choice([4, 8]), T=_log(rng, 16, 4096))
    if kind == "attention":
        Hkv, group = rng.choice([4, 8]), rng.choice([1, 2, 4])
        return dict(kind=kind, layout=rng.choice(["tiled", "tiled", "tiled_paged", "tiled_paged", "rows", "rows_paged"]),
                    B=_log(rng, 1, 32), Hq=Hkv * group, Hkv=Hkv, T=_log(rng, 48, 4096), ragged=rng.random() < 0.5,
                    append=rng.random() < 0.5)
    if kind == "moe":
        return dict(kind=kind, T=_log(rng, 1, 512), H=rng.choice([1024, 2048]), I=rng.choice([512, 768]),
                    E=rng.choice([64, 128]), topk=rng.choice([4, 8]))
    return dict(kind=kind, B=_log(rng, 1, 16), T=_log(rng, 64, 4096), layers=rng.randint(1, 2), moe=rng.random() < 0.4)


# ---- device memory from torch, in the shape the package's objects take it --------------------------------------------

class Memory:
    """What mi.GemmBatch and mi.DecoderLayer ask of a device: buffers.  Every buffer is a torch tensor."""

    def __init__(self):
        self.kept = []

    def hold(self, t, shape=None, dtype=None):
        self.kept.append(t)
        if dtype is None:
            dtype = {torch.float32: np.float32, torch.int8: np.int8, torch.int32: np.int32, torch.uint8: np.uint8}[t.dtype]
        return mi.DevBuf(t.data_ptr(), shape if shape is not None else t.shape, dtype)

    def empty(self, shape, dtype):
        shape = tuple(int(s) for s in (shape if isinstance(shape, (tuple, list)) else (shape,)))
        kind = {"float32": torch.float32, "int8": torch.int8, "int32": torch.int32, "uint8": torch.uint8}[np.dtype(dtype).name]
        return self.hold(torch.empty(shape, dtype=kind, device="cuda"))

    def upload(self, a):
        return self.hold(a.contiguous() if isinstance(a, torch.Tensor) else torch.from_numpy(np.ascontiguousarray(a)).cuda())

    def mark(self):
        return len(self.kept)

    def reset_to(self, mark):
        del self.kept[mark:]

    def sync(self):
        torch.cuda.synchronize()

    def tensor(self, buf):
        return next(t for t in self.kept if t.data_ptr() == buf.ptr and t.numel() * t.element_size() == buf.nbytes)


class State:
    """Whatever a case keeps between passes; gives native handles back when it goes."""

    def __init__(self, case):
        self.case, self.mem, self.graph, self.batch = dict(case), Memory(), None, None

    def __del__(self):
        if sys.is_finalizing():
            return
        torch.cuda.synchronize()                 # passes may still be in flight
        for handle in (self.graph, self.batch):
            if handle is not None:
                handle.destroy()


def _activations(g, M, K):
    """fp32 [M,K] ~ N(0,1), 0.1 % of the channels 20 times as large."""
    x = torch.randn(M, K, generator=g, device="cuda")
    ch = torch.randperm(K, generator=g, device="cuda")[: math.ceil(0.001 * K)]
    x[:, ch] *= 20.0
    return x


def _weights(g, *shape):
    return torch.randn(*shape, generator=g, device="cuda").mul_(0.02)


def _quantized(mem, rows, block):
    """Codes and scales of fp32 rows [..., K] (rotated in blocks)."""
    rows = rows.contiguous()
    K = rows.shape[-1]
    q = torch.empty(rows.shape, dtype=torch.int8, device="cuda")
    s = torch.empty(rows.shape[:-1], dtype=torch.float32, device="cuda")
    n = rows.numel() // K
    mi.fwht_quant(mi.DevBuf(rows.data_ptr(), (n, K), np.float32), mi.DevBuf(q.data_ptr(), (n, K), np.int8),
                  mi.DevBuf(s.data_ptr(), (n,), np.float32), block)
    torch.cuda.synchronize()
    return mem.hold(q), mem.hold(s)


def _lengths(case, seed):
    """Sequence lengths: all T, or spread from T down to T/4 and dealt in an order that the seed gives."""
    B, T = case["B"], case["T"]
    n = [T - (3 * T * i) // (4 * B) if case.get("ragged") else T for i in range(B)]
    random.Random(seed).shuffle(n)
    return n


def _round64(t):
    return (t + 63) // 64 * 64


def _cache_rows(mem, g, *lead):
    """Keys or values ~ N(0,1) of shape [*lead, D], rotated and quantized."""
    return _quantized(mem, torch.randn(*lead, D, generator=g, device="cuda"), D)


def _tiled(mem, kq, vq, rows, T):
    kt, vt = mem.empty((rows, T, D), np.int8), mem.empty((rows, T, D), np.int8)
    mi.check(mi.lib.mi_kv_tiled_from_rows_i8(kq.ptr, vq.ptr, kt.ptr, vt.ptr, rows, T, T, T, None), "mi_kv_tiled_from_rows_i8")
    torch.cuda.synchronize()
    return kt, vt


# ---- what a program has in hand before the call ----------------------------------------------------------------------

def prepare(case, seed):
    st = State(case)
    g = torch.Generator(device="cuda").manual_seed(int(seed))
    {"linear": _prepare_linear, "prefill": _prepare_prefill, "kv_prefill": _prepare_kv_prefill, "attention": _prepare_attention,
     "moe": _prepare_moe, "decode": _prepare_decode}[case["kind"]](st, case, g, int(seed))
    torch.cuda.synchronize()
    return st


def _prepare_linear(st, c, g, seed):
    mem, M, K, N = st.mem, c["M"], c["K"], c["N"]
    st.x = mem.upload(_activations(g, M, K))
    st.qw, st.sw = _quantized(mem, _weights(g, N, K), workload.HADAMARD_BLOCK)
    st.y = mem.empty((M, N), np.float32)
    st.ws = mem.empty(mi.lib.mi_w8a8_linear_workspace_bytes(M, N, K), np.uint8)
    st.out = mem.tensor(st.y)


def _prepare_prefill(st, c, g, seed):
    mem, M = st.mem, c["M"]
    f, i8 = np.float32, np.int8
    w = {name: _quantized(mem, _weights(g, N, K), workload.HADAMARD_BLOCK) for name, (K, N) in PROJECTIONS.items()}
    y = {name: mem.empty((M, N), f) for name, (K, N) in PROJECTIONS.items()}
    st.sets, codes = [], {}
    for name in ("qkv", "gate", "down"):        # gate and up take the same input
        K = PROJECTIONS[name][0]
        codes[name] = (mem.empty((M, K), i8), mem.empty(M, f))
        st.sets.append((mem.upload(_activations(g, M, K)),) + codes[name])
    codes["up"] = codes["gate"]
    st.ops = [codes[name] + w[name] + (y[name],) for name in PROJECTIONS]
    st.batch = mi.GemmBatch(mem, [(M, N, K) for K, N in PROJECTIONS.values()])
    st.out = {name: mem.tensor(b) for name, b in y.items()}


def _prepare_kv_prefill(st, c, g, seed):
    mem, B, Hkv, T = st.mem, c["B"], c["Hkv"], c["T"]
    rows, cap = B * Hkv, _round64(T)
    st.k = mem.upload(torch.randn(rows * T, D, generator=g, device="cuda"))
    st.v = mem.upload(torch.randn(rows * T, D, generator=g, device="cuda"))
    st.kq, st.vq = mem.empty((rows * T, D), np.int8), mem.empty((rows * T, D), np.int8)
    st.ks, st.vs = mem.empty(rows * T, np.float32), mem.empty(rows * T, np.float32)
    st.kt, st.vt = mem.empty((rows, cap, D), np.int8), mem.empty((rows, cap, D), np.int8)
    st.out = {n: mem.tensor(getattr(st, n)) for n in ("kt", "vt", "ks", "vs")}


def _prepare_attention(st, c, g, seed):
    mem, B, Hq, Hkv, T, layout = st.mem, c["B"], c["Hq"], c["Hkv"], c["T"], c["layout"]
    lens = _lengths(c, seed)
    page = {"tiled_paged": PAGE, "rows_paged": ROW_PAGE}.get(layout)
    if page:
        st.max_pages = (T + page - 1) // page
        pages = sum((n + page - 1) // page for n in lens)
        order = list(range(pages))
        random.Random(seed + 1).shuffle(order)   # pages were handed out as sequences grew side by side
        table, at = np.zeros((B, st.max_pages), np.int32), 0
        for b, n in enumerate(lens):
            k = (n + page - 1) // page
            table[b, :k] = order[at:at + k]
            at += k
        st.table = mem.upload(table)
        lead = (pages, Hkv, page)
    else:
        st.cap = _round64(T)
        lead = (B, Hkv, st.cap)
    kq, st.ks = _cache_rows(mem, g, *lead)
    vq, st.vs = _cache_rows(mem, g, *lead)
    st.kq, st.vq = _tiled(mem, kq, vq, lead[0] * Hkv, lead[2]) if layout.startswith("tiled") else (kq, vq)
    st.q = mem.upload(torch.randn(B, Hq, D, generator=g, device="cuda"))
    st.k_new = mem.upload(torch.randn(B, Hkv, D, generator=g, device="cuda"))
    st.v_new = mem.upload(torch.randn(B, Hkv, D, generator=g, device="cuda"))
    st.lens = mem.upload(np.array(lens, np.int32))
    st.pos = mem.upload(np.array(lens, np.int32) - 1)
    st.o = mem.empty((B, Hq, D), np.float32)
    st.ws = mem.empty(mi.lib.mi_gqa_decode_workspace_bytes(B, Hq, Hkv, D, T), np.uint8)
    st.out = {"o": mem.tensor(st.o)}
    if c["append"]:
        st.out.update({n: mem.tensor(getattr(st, n)) for n in ("kq", "ks", "vq", "vs")})


def _experts(mem, g, H, I, E):
    wg, sg = _quantized(mem, _weights(g, E, I, H), workload.HADAMARD_BLOCK)
    wu, su = _quantized(mem, _weights(g, E, I, H), workload.HADAMARD_BLOCK)
    wd, sd = _quantized(mem, _weights(g, E, H, I), workload.MOE_INNER_BLOCK)
    return dict(wr=mem.upload(_weights(g, E, H)), wg=wg, sg=sg, wu=wu, su=su, wd=wd, sd=sd)


def _prepare_moe(st, c, g, seed):
    mem, T, H, I, E, topk = st.mem, c["T"], c["H"], c["I"], c["E"], c["topk"]
    st.x = mem.upload(_activations(g, T, H))
    st.w = _experts(mem, g, H, I, E)
    st.y = mem.empty((T, H), np.float32)
    st.ws = mem.empty(mi.lib.mi_moe_layer_workspace_bytes(T, H, I, E, topk), np.uint8)
    st.out = mem.tensor(st.y)


def _decode_shape(moe):
    return dict(H=2048, Hq=16, Hkv=4, I=768) if moe else dict(H=4096, Hq=32, Hkv=8, I=14336)


def _prepare_decode(st, c, g, seed):
    mem, B, T = st.mem, c["B"], c["T"]
    s = _decode_shape(c["moe"])
    H, Hq, Hkv, I, cap = s["H"], s["Hq"], s["Hkv"], s["I"], _round64(T)
    angle = torch.arange(cap, device="cuda")[:, None] * (10000.0 ** (-torch.arange(D // 2, device="cuda") * (2.0 / D)))[None]
    cos, sin = angle.cos().float(), angle.sin().float()
    st.layers = []
    for _ in range(c["layers"]):
        ones = lambda: 1.0 + 0.1 * torch.randn(H, generator=g, device="cuda")  # noqa: E731
        moe = dict(_experts(mem, g, H, I, workload.MOE["E"]), topk=workload.MOE["topk"]) if c["moe"] else None
        layer = mi.DecoderLayer(mem, B, H, Hq, Hkv, I, cap, _weights(g, (Hq + 2 * Hkv) * D, H), _weights(g, H, Hq * D),
                                None if moe else _weights(g, 2 * I, H), None if moe else _weights(g, H, I), ones(), ones(),
                                cos, sin, tiled=True, moe=moe)
        kq, ks = _cache_rows(mem, g, B, Hkv, cap)
        vq, vs = _cache_rows(mem, g, B, Hkv, cap)
        kt, vt = _tiled(mem, kq, vq, B * Hkv, cap)
        for to, of in ((layer.kq, kt), (layer.vq, vt), (layer.ks, ks), (layer.vs, vs)):
            mem.tensor(to).view(-1).copy_(mem.tensor(of).view(-1))
        torch.cuda.synchronize()
        for b in (kq, ks, vq, vs, kt, vt):
            mem.kept = [t for t in mem.kept if t.data_ptr() != b.ptr]
        st.layers.append(layer)
    st.x = mem.upload(_activations(g, B, H))
    lens = _lengths(c, seed)
    st.lens = mem.upload(np.array(lens, np.int32))
    st.pos = mem.upload(np.array(lens, np.int32) - 1)
    st.y = mem.empty((B, H), np.float32)

    def step(stream):
        x, residual = st.x, None
        for k, layer in enumerate(st.layers):
            layer.step(x, st.pos, st.lens, T, st.y if k + 1 == len(st.layers) else None, stream, residual)
            x, residual = layer.dn, layer.h1

    step(None)                                   # once as it is: one-time kernel attributes
    torch.cuda.synchronize()
    side = torch.cuda.Stream()
    st.graph = mi.Graph(ctypes.c_void_p(side.cuda_stream))
    with st.graph:
        step(st.graph.stream)
    st.out = {"y": mem.tensor(st.y)}
    for k, layer in enumerate(st.layers):
        st.out.update({"%s%d" % (n, k): mem.tensor(getattr(layer, n)) for n in ("kq", "ks", "vq", "vs")})


# ---- one pass --------------------------------------------------------------------------------------------------------

def run(st):
    c, lib = st.case, mi.lib
    kind = c["kind"]
    if kind == "linear":
        mi.linear(st.x, st.qw, st.sw, st.y, workload.HADAMARD_BLOCK, st.ws)
    elif kind == "prefill":
        mi.fwht_quant_batch(st.sets, workload.HADAMARD_BLOCK)
        st.batch.run_f32(st.ops)
    elif kind == "kv_prefill":
        rows = c["B"] * c["Hkv"]
        mi.fwht_quant(st.k, st.kq, st.ks, D)
        mi.fwht_quant(st.v, st.vq, st.vs, D)
        mi.check(lib.mi_kv_tiled_from_rows_i8(st.kq.ptr, st.vq.ptr, st.kt.ptr, st.vt.ptr, rows, c["T"], c["T"], _round64(c["T"]),
                                              None), "mi_kv_tiled_from_rows_i8")
    elif kind == "attention":
        _run_attention(st, c, lib)
    elif kind == "moe":
        w = st.w
        mi.moe_layer(st.x, w["wr"], w["wg"], w["sg"], w["wu"], w["su"], w["wd"], w["sd"], st.y, c["topk"], st.ws)
    else:
        mi.check(lib.mi_graph_launch(st.graph.h, None), "mi_graph_launch")
    return st.out


def _run_attention(st, c, lib):
    B, Hq, Hkv, T, layout = c["B"], c["Hq"], c["Hkv"], c["T"], c["layout"]
    cache = (st.kq.ptr, st.ks.ptr, st.vq.ptr, st.vs.ptr)
    new = (st.k_new.ptr, st.v_new.ptr, Hkv * D)
    ws = (st.ws.ptr, st.ws.nbytes, None)
    if layout == "tiled":
        if c["append"]:
            mi.check(lib.mi_kv_append_tiled_f32_i8(*new, *cache, st.pos.ptr, B, Hkv, D, st.cap, None))
        mi.check(lib.mi_gqa_decode_attn_tiled(st.q.ptr, *cache, st.o.ptr, B, Hq, Hkv, D, st.cap,
                                              st.lens.ptr if c["ragged"] else None, T, 0, *ws))
    elif layout == "tiled_paged":
        if c["append"]:
            mi.check(lib.mi_kv_append_tiled_paged_f32_i8(*new, *cache, st.table.ptr, st.max_pages, st.pos.ptr, B, Hkv, D, None))
        mi.check(lib.mi_gqa_decode_attn_tiled_paged(st.q.ptr, *cache, st.o.ptr, st.table.ptr, st.max_pages, B, Hq, Hkv, D,
                                                    st.lens.ptr, T, 0, *ws))
    elif layout == "rows":
        if c["append"]:
            mi.check(lib.mi_kv_append_f32_i8(*new, *cache, st.pos.ptr, B, Hkv, D, st.cap, None))
        mi.check(lib.mi_gqa_decode_attn_cache(st.q.ptr, *cache, st.o.ptr, B, Hq, Hkv, D, st.cap, st.lens.ptr, T, 0, *ws))
    else:
        if c["append"]:
            mi.check(lib.mi_kv_append_paged_f32_i8(*new, *cache, st.table.ptr, st.max_pages, ROW_PAGE, st.pos.ptr, B, Hkv, D,
                                                   None))
        mi.check(lib.mi_gqa_decode_attn_paged(st.q.ptr, *cache, st.o.ptr, st.table.ptr, st.max_pages, ROW_PAGE, B, Hq, Hkv, D,
                                              st.lens.ptr, T, 0, *ws))


# ---- what a pass cannot do without -----------------------------------------------------------------------------------

def _linear_work(M, K, N, x_bytes=4, y_bytes=4):
    return N * K + 4 * N + x_bytes * M * K + y_bytes * M * N, 2 * M * N * K


def _attention_work(B, Hq, Hkv, tokens):
    return 2 * Hkv * tokens * (D + 4) + 8 * B * Hq * D, 4 * Hq * tokens * D


def _moe_work(T, H, I, E, topk):
    """Weights of the experts that T tokens reach when routed evenly, the router, tokens in and out."""
    reached = E * (1.0 - (1.0 - topk / E) ** T)
    return reached * (3 * H * I + 8 * I + 4 * H) + 4 * E * H + 8 * T * H, 2 * T * E * H + 6 * T * topk * H * I


def work(case):
    c, kind = case, case["kind"]
    if kind == "linear":
        b, f = _linear_work(c["M"], c["K"], c["N"])
    elif kind == "prefill":
        parts = [_linear_work(c["M"], K, N, x_bytes=0 if name == "up" else 4) for name, (K, N) in PROJECTIONS.items()]
        b, f = sum(p[0] for p in parts), sum(p[1] for p in parts)
    elif kind == "kv_prefill":
        n = 2 * c["B"] * c["Hkv"] * c["T"]
        b, f = n * (5 * D + 4), n * D * 7
    elif kind == "attention":
        b, f = _attention_work(c["B"], c["Hq"], c["Hkv"], sum(_lengths(c, 0)))
    elif kind == "moe":
        b, f = _moe_work(c["T"], c["H"], c["I"], c["E"], c["topk"])
    else:
        B, s = c["B"], _decode_shape(c["moe"])
        H, Hq, Hkv, I = s["H"], s["Hq"], s["Hkv"], s["I"]
        parts = [_linear_work(B, H, (Hq + 2 * Hkv) * D, 0, 0), _linear_work(B, Hq * D, H, 0, 0),
                 _attention_work(B, Hq, Hkv, B * c["T"])]
        if c["moe"]:
            parts.append(_moe_work(B, H, I, workload.MOE["E"], workload.MOE["topk"]))
        else:
            parts += [_linear_work(B, H, 2 * I, 0, 0), _linear_work(B, I, H, 0, 0)]
        b, f = (c["layers"] * sum(p[k] for p in parts) for k in (0, 1))
        b += 8 * B * H
    return {"bytes": b, "flops": f}


def tolerance(case):
    """About four times what the same pass shows with its sums in another order (row-major against tiled cache kernels, the
    kernels against sums in C on the host)."""
    kind = case["kind"]
    if kind in ("linear", "prefill", "kv_prefill"):
        return "exact"       # codes, integer sums and two fp32 products per result: IEEE operations in a fixed order
    if kind == "attention":  # fp32 sums; measured 9e-7 and 2e-5.  Appended codes are exact
        return {"rel": 4e-6, "max": 1e-4}
    if kind == "moe":        # measured 5e-8 over 64 tokens; an ulp in a SwiGLU value can move an int8 code, 1/127 of its row's range
        return {"rel": 1e-4, "max": 1e-2}
    # decode: an ulp in the attention output moves int8 codes, and every later layer quantizes what that left.  Measured
    # dense 1.2e-3, 6.6e-3, 1.3e-2 behind 1, 2, 4 layers (largest 0.12), with experts 7e-4 (largest 5e-3); cache codes of
    # the new token up to 0.23 % of a 64-token cache
    if case["moe"]:
        return {"rel": 3e-3, "max": 2e-2, "differ": 5e-3}
    return {"rel": 5e-3 if case["layers"] == 1 else 3e-2, "max": 0.08 if case["layers"] == 1 else 0.4, "differ": 9e-3}
