"""The measured cases: what a host of this library has it do, through ``vybforge_amd.ops``.

Families (``family`` of a case), and what each stands for in real use:
  gemv     one packed GEMV of a decoding token, called eagerly: launch latency and host cost
  stack    a whole decode token of a q4_0 model's linear stack (fused q|k|v, o, fused gate|up,
           down per layer), captured once as a graph as a decode loop keeps it
  xq8      decode MLPs on quantized activations: RMSNorm with its q8 copy, gate|up, SwiGLU with
           its q8 copy, down with the residual; graph
  batch    batched or speculative decode: an MLP's gate|up and down at 2..48 rows (the GEMV entry
           up to its 8 rows, the GEMM above); graph
  prefill  a prompt chunk through an MLP's gate, up and down, fp16 matrix path or (q8 = True) the
           int8 path with its activation quantizer; eager
  exl3     decode MLPs of EXL3 4-bpw linears at batch 1..16; graph
  moe      a GLM-5-shaped MoE layer with GGUF experts, 1..256 tokens; eager
  moe_exl3 a GLM-5.3-shaped MoE layer with EXL3 experts and a bf16 shared expert; eager
Sizes are those of the benchmark (Qwen3-4B stack 2560/4096/1024/9728, MLP 5120/17408, GLM-5
6144/2048/256, GLM-5.3 4096/2048/288). Weights of the decode families exceed the 256 MB cache, as a
model's do.
"""

import json
import math
import os

import torch

from vybforge_amd import ops

F32, F16, BF16 = torch.float32, torch.float16, torch.bfloat16
DT = {"f32": F32, "f16": F16, "bf16": BF16}
Q4_0, Q8_0, Q4_K, Q5_K, Q6_K, IQ2_S = 2, 8, 12, 13, 14, 22
BLOCK = {Q4_0: (32, 18), Q8_0: (32, 34), Q4_K: (256, 144), Q5_K: (256, 176), Q6_K: (256, 210), IQ2_S: (256, 82)}
SCALE_AT = {Q4_0: (0,), Q8_0: (0,), Q4_K: (0, 2), Q5_K: (0, 2), Q6_K: (208,), IQ2_S: (0,)}
SCALE_STD = {Q4_0: 1e-2, Q8_0: 1e-3, Q4_K: 1e-4, Q5_K: 1e-4, Q6_K: 1e-5, IQ2_S: 1e-4}
DATA = os.path.join(os.path.dirname(os.path.abspath(ops.__file__)), "data")


def listed():
    return [
        # the smallest call: a key projection of one token
        dict(name="gemv_q4_0", family="gemv", ty=Q4_0, N=1024, K=2560, x="f16"),
        # one decoded token of a 4B q4_0 model
        dict(name="stack_q4_0", family="stack", H=2560, Q=4096, KV=1024, I=9728, L=36, x="f16"),
        # the default decode path of a 27B mixed-quant model: IQ2_S gate|up, Q4_K down
        dict(name="xq8_iq2s_q4k", family="xq8", gu=IQ2_S, down=Q4_K, H=5120, I=17408, L=4),
        # 24 sequences decoded together
        dict(name="batch24_q4k_q6k", family="batch", gu=Q4_K, down=Q6_K, M=24, H=5120, I=17408, L=3, x="bf16"),
        # a prompt chunk of a Q8_0 model
        dict(name="prefill512_q8_0", family="prefill", gu=Q8_0, down=Q8_0, M=512, H=5120, I=17408, x="bf16", q8=False),
        # a long, ragged prompt of a Q4_K_M model
        dict(name="prefill1999_q4k_q6k", family="prefill", gu=Q4_K, down=Q6_K, M=1999, H=5120, I=17408, x="bf16",
             q8=False),
        # one sequence, and a full batch, through EXL3 linears
        dict(name="exl3_b1", family="exl3", B=1, H=5120, I=17408, L=2, x="f16"),
        dict(name="exl3_b16", family="exl3", B=16, H=5120, I=17408, L=2, x="f16"),
        # MoE layers: a small decode batch and a prefill chunk of GGUF experts
        dict(name="moe_q4_0_T16", family="moe", ty=Q4_0, T=16, H=6144, I=2048, E=256, x="bf16", bias=False),
        dict(name="moe_q4_0_T256", family="moe", ty=Q4_0, T=256, H=6144, I=2048, E=256, x="bf16", bias=False),
        # one token, and a prefill chunk, of the production layer with EXL3 experts
        dict(name="moe_exl3_T1", family="moe_exl3", T=1, H=4096, I=2048, E=288, x="bf16", bias=True),
        dict(name="moe_exl3_T256", family="moe_exl3", T=256, H=4096, I=2048, E=288, x="bf16", bias=True),
    ]


def draw(rng):
    def log(a, b, step=1):
        v = math.exp(rng.uniform(math.log(a), math.log(b)))
        return min(max(int(round(v / step)) * step, -(-a // step) * step), b // step * step)

    every = (Q4_0, Q8_0, Q4_K, Q5_K, Q6_K, IQ2_S)
    family = rng.choice(("gemv", "stack", "xq8", "batch", "batch", "prefill", "prefill", "exl3", "exl3", "moe", "moe",
                         "moe_exl3", "moe_exl3"))
    if family == "gemv":
        ty = rng.choice(every)
        return dict(family=family, ty=ty, N=log(200, 9728), K=log(1024, 9728, 64 if ty in (Q4_0, Q8_0) else 256),
                    x=rng.choice(("f32", "f16", "bf16")))
    if family == "stack":
        return dict(family=family, H=log(1024, 2560, 64), Q=log(1024, 4096, 64), KV=log(256, 1024, 64),
                    I=log(3072, 9728, 64), L=rng.randint(24, 36), x=rng.choice(("f16", "bf16")))
    if family == "xq8":
        return dict(family=family, gu=rng.choice((IQ2_S, Q4_K, Q5_K)), down=rng.choice((IQ2_S, Q4_K, Q5_K)),
                    H=log(2048, 5120, 256), I=log(6144, 17408, 256), L=4)
    if family == "batch":
        return dict(family=family, gu=rng.choice(every), down=rng.choice(every), M=log(2, 48), H=log(2048, 5120, 256),
                    I=log(6144, 17408, 256), L=3, x=rng.choice(("f16", "bf16", "f32")))
    if family == "prefill":
        q8 = rng.random() < 0.25
        gu, down = (Q8_0, Q8_0) if q8 else (rng.choice(every), rng.choice(every))
        return dict(family=family, gu=gu, down=down, M=log(64, 1999), H=log(2048, 5120, 256), I=log(6144, 17408, 256),
                    x=rng.choice(("f16", "bf16", "bf16")), q8=q8)
    if family == "exl3":
        return dict(family=family, B=log(1, 16), H=log(2048, 5120, 128), I=log(6144, 17408, 128), L=2,
                    x=rng.choice(("f16", "bf16", "f32")))
    if family == "moe":
        return dict(family=family, ty=rng.choice((Q4_0, Q4_0, Q8_0)), T=log(1, 256), H=log(2048, 6144, 256),
                    I=log(512, 2048, 256), E=rng.choice((64, 128, 160)), x=rng.choice(("f16", "bf16", "bf16")),
                    bias=rng.random() < 0.5)
    return dict(family=family, T=log(1, 256), H=log(2048, 4096, 128), I=log(768, 2048, 128),
                E=rng.choice((96, 160, 288)), x=rng.choice(("f16", "bf16", "bf16")), bias=rng.random() < 0.7)


# ---- inputs -----------------------------------------------------------------------------------

TOPK, ROUTE_SCALE, LIMIT, EPS = 8, 2.5, 10.0, 1e-6


class _Gen:
    """Tensors of one seed on the GPU, in a fixed order."""

    def __init__(self, seed):
        self.g = torch.Generator(device="cuda")
        self.g.manual_seed(int(seed))

    def normal(self, *shape, dt=F32, std=1.0):
        return (torch.randn(*shape, generator=self.g, device="cuda") * std).to(dt)

    def bytes(self, n):
        words = torch.randint(-(1 << 63), (1 << 63) - 1, ((n + 7) // 8,), generator=self.g, device="cuda")
        return words.view(torch.uint8)[:n]

    def packed(self, ty, rows, K):
        """Packed rows: uniform quants, the fp16 scale fields |N(0, std)|."""
        nw, nb = BLOCK[ty]
        n = rows * (K // nw)
        blk = self.bytes(n * nb).view(n, nb)
        for at in SCALE_AT[ty]:
            blk[:, at:at + 2] = self.normal(n, dt=F16, std=SCALE_STD[ty]).abs().view(torch.uint8).view(n, 2)
        return blk.view(-1)

    def signed(self, n):
        """EXL3 suh / svh of one side: +-|N(0, 0.12)|, matrices of about N(0, 0.02)."""
        return self.normal(n, dt=F16, std=0.12)

    def exl3(self, K, N):
        t = self.bytes(K * N // 2).view(torch.int16).view(K // 16, N // 16, 64)
        return t, self.signed(K), self.signed(N)


def _graph(calls):
    """The calls as one captured graph, warmed once."""
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        calls()
    torch.cuda.current_stream().wait_stream(side)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        calls()
    return graph


def _inputs(case, seed):
    """The plain tensors of a case (weights, activations), before any handle of the library."""
    g, f, d = _Gen(seed), case["family"], dict(case)
    x = DT[case.get("x", "f32")]
    if f == "gemv":
        d.update(W=g.packed(case["ty"], case["N"], case["K"]), X=g.normal(case["K"], dt=x))
    elif f == "stack":
        H, Q, KV, I = (case[k] for k in ("H", "Q", "KV", "I"))
        shapes = dict(q=(Q, H), k=(KV, H), v=(KV, H), o=(H, Q), gate=(I, H), up=(I, H), down=(H, I))
        d.update(shapes=shapes, W=[{k: g.packed(Q4_0, *s) for k, s in shapes.items()} for _ in range(case["L"])],
                 X={k: g.normal(n, dt=x) for k, n in (("attn", H), ("o", Q), ("mlp", H), ("down", I))})
    elif f == "xq8":
        H, I = case["H"], case["I"]
        d.update(W=[dict(gate=g.packed(case["gu"], I, H), up=g.packed(case["gu"], I, H),
                         down=g.packed(case["down"], H, I), norm=1 + g.normal(H, std=0.1)) for _ in range(case["L"])],
                 X=[g.normal(H) for _ in range(case["L"])])
    elif f in ("batch", "prefill"):
        H, I, M = case["H"], case["I"], case["M"]
        d.update(W=[dict(gate=g.packed(case["gu"], I, H), up=g.packed(case["gu"], I, H),
                         down=g.packed(case["down"], H, I)) for _ in range(case.get("L", 1))],
                 X=g.normal(M, H, dt=x), XD=g.normal(M, I, dt=x), R=g.normal(M, H, dt=x))
    elif f == "exl3":
        H, I = case["H"], case["I"]
        d.update(W=[dict(gate=g.exl3(H, I), up=g.exl3(H, I), down=g.exl3(I, H)) for _ in range(case["L"])],
                 X=g.normal(case["B"], H, dt=x), XD=g.normal(case["B"], I, dt=x))
    else:
        T, H, I, E = (case[k] for k in ("T", "H", "I", "E"))
        if f == "moe":
            ty = case["ty"]
            d.update(W=(g.packed(ty, E * I, H), g.packed(ty, E * I, H), g.packed(ty, E * H, I)),
                     S=(g.packed(ty, I, H), g.packed(ty, I, H), g.packed(ty, H, I)))
        else:
            t = g.bytes(E * 3 * H * I // 2).view(torch.int16).view(E, 3, H * I // 4)
            sh, si = g.signed(E * 3 * H).view(E, 3, H), g.signed(E * 3 * I).view(E, 3, I)
            up, dn = (H // 16, I // 16, 64), (I // 16, H // 16, 64)
            d.update(W=[(t[e, 0].view(up), sh[e, 0], si[e, 0], t[e, 1].view(up), sh[e, 1], si[e, 1],
                         t[e, 2].view(dn), si[e, 2], sh[e, 2]) for e in range(E)],
                     S=tuple(g.normal(*s, dt=BF16, std=0.02) for s in ((I, H), (I, H), (H, I))))
        d.update(X=g.normal(T, H, dt=x), logits=g.normal(T, E),
                 B=g.normal(E, std=0.05) if case["bias"] else None)
    return d


def prepare(case, seed):
    s = _inputs(case, seed)
    f, dt = case["family"], DT[case.get("x", "f32")]
    buf = lambda *shape, dt=dt: torch.empty(*shape, dtype=dt, device="cuda")  # noqa: E731
    if f == "stack":
        L, X, shapes = case["L"], s["X"], s["shapes"]
        Y = {k: buf(L, n) for k, (n, _) in shapes.items()}

        def token():
            for i, W in enumerate(s["W"]):
                seg = lambda k, i=i, W=W: (W[k], Y[k][i], shapes[k][0])  # noqa: E731
                ops.gemv_q4_0_seg3(X["attn"], case["H"], [seg("q"), seg("k"), seg("v")])
                ops.gemv(Q4_0, W["o"], X["o"], *shapes["o"], out=Y["o"][i])
                ops.gemv_q4_0_seg3(X["mlp"], case["H"], [seg("gate"), seg("up")])
                ops.gemv(Q4_0, W["down"], X["down"], *shapes["down"], out=Y["down"][i])
        s.update(Y=Y, graph=_graph(token))
    elif f == "xq8":
        L, H, I = case["L"], case["H"], case["I"]
        Y = dict(gate=buf(L, I), up=buf(L, I), down=buf(L, H))

        def token():
            for i, W in enumerate(s["W"]):
                _, _, q, d = ops.rmsnorm_q8(s["X"][i], W["norm"], EPS)
                ops.gemv_xq8_seg3(case["gu"], q, d, H, [(W["gate"], Y["gate"][i], I), (W["up"], Y["up"][i], I)])
                _, q, d = ops.swiglu_q8(Y["gate"][i], Y["up"][i], h_dtype=None)
                ops.gemv_xq8(case["down"], W["down"], q, d, H, I, residual=s["X"][i], out=Y["down"][i])
        s.update(Y=Y, graph=_graph(token))
    elif f == "batch":
        L, H, I, M = case["L"], case["H"], case["I"], case["M"]
        Y = dict(gate=buf(L, M, I), up=buf(L, M, I), down=buf(L, M, H))
        ws = [ops.GemmWorkspace([(M, n, k)], "cuda", ty) for ty, n, k in ((case["gu"], I, H), (case["down"], H, I))]

        def token():
            for i, W in enumerate(s["W"]):
                if M <= 8:
                    ops.gemv_seg3(case["gu"], s["X"], H, [(W["gate"], Y["gate"][i], I), (W["up"], Y["up"][i], I)])
                    ops.gemv(case["down"], W["down"], s["XD"], H, I, residual=s["R"], out=Y["down"][i])
                else:
                    ops.gemm(case["gu"], W["gate"], s["X"], I, H, out=Y["gate"][i], workspace=ws[0])
                    ops.gemm(case["gu"], W["up"], s["X"], I, H, out=Y["up"][i], workspace=ws[0])
                    ops.gemm(case["down"], W["down"], s["XD"], H, I, residual=s["R"], out=Y["down"][i], workspace=ws[1])
        s.update(Y=Y, ws=ws, graph=_graph(token))
    elif f == "prefill":
        H, I, M = case["H"], case["I"], case["M"]
        s["ws"] = [ops.GemmWorkspace([(M, n, k)], "cuda", ty, int8=case["q8"])
                   for ty, n, k in ((case["gu"], I, H), (case["down"], H, I))]
    elif f == "exl3":
        L, B, H, I = case["L"], case["B"], case["H"], case["I"]
        Y = dict(gate=buf(L, B, I), up=buf(L, B, I), down=buf(L, B, H))
        s["lin"] = [{k: ops.Exl3Linear(*W[k], *kn, max_batch=B) for k, kn in
                     (("gate", (H, I)), ("up", (H, I)), ("down", (I, H)))} for W in s["W"]]

        def token():
            for i, lin in enumerate(s["lin"]):
                lin["gate"](s["X"], out=Y["gate"][i])
                lin["up"](s["X"], out=Y["up"][i])
                lin["down"](s["XD"], out=Y["down"][i])
        s.update(Y=Y, graph=_graph(token))
    elif f == "moe":
        s["layer"] = ops.MoeLayer(case["ty"], *s["W"], case["H"], case["I"], case["E"], TOPK, shared=s["S"],
                                  scale=ROUTE_SCALE, limit=LIMIT, bias=s["B"])
    elif f == "moe_exl3":
        s["layer"] = ops.MoeExl3Layer(s["W"], case["H"], case["I"], TOPK, shared=s["S"], scale=ROUTE_SCALE, limit=LIMIT,
                                      bias=s["B"])
    return s


def run(s):
    f = s["family"]
    if "graph" in s:
        s["graph"].replay()
        return s["Y"]
    dt = DT[s["x"]]
    if f == "gemv":
        return ops.gemv(s["ty"], s["W"], s["X"], s["N"], s["K"], y_dtype=dt)
    if f == "prefill":
        H, I, W, (gu, dn) = s["H"], s["I"], s["W"][0], s["ws"]
        if s["q8"]:
            q, d = ops.quant_q8_act(s["X"])
            gate = ops.gemm_q8_0_i8(W["gate"], q, d, I, H, y_dtype=dt, workspace=gu)
            up = ops.gemm_q8_0_i8(W["up"], q, d, I, H, y_dtype=dt, workspace=gu)
            q, d = ops.quant_q8_act(s["XD"])
            return dict(gate=gate, up=up,
                        down=ops.gemm_q8_0_i8(W["down"], q, d, H, I, y_dtype=dt, residual=s["R"], workspace=dn))
        return dict(gate=ops.gemm(s["gu"], W["gate"], s["X"], I, H, y_dtype=dt, workspace=gu),
                    up=ops.gemm(s["gu"], W["up"], s["X"], I, H, y_dtype=dt, workspace=gu),
                    down=ops.gemm(s["down"], W["down"], s["XD"], H, I, y_dtype=dt, residual=s["R"], workspace=dn))
    return s["layer"](s["X"], s["logits"], out_dtype=dt)


# ---- what a pass cannot do without ----------------------------------------------------------------

def _hit(case):
    """Expected number of distinct experts T tokens select (random logits)."""
    T, E = case["T"], case["E"]
    return E * (1 - (1 - TOPK / E) ** T)


def work(case):
    f = case["family"]
    e = {"f32": 4, "f16": 2, "bf16": 2}[case.get("x", "f32")]
    rows = lambda ty, n, k: n * (k // BLOCK[ty][0]) * BLOCK[ty][1]  # noqa: E731
    if f == "gemv":
        N, K = case["N"], case["K"]
        return dict(bytes=rows(case["ty"], N, K) + e * (N + K), flops=2 * N * K)
    if f == "stack":
        H, Q, KV, I, L = (case[k] for k in ("H", "Q", "KV", "I", "L"))
        shapes = ((Q, H), (KV, H), (KV, H), (H, Q), (I, H), (I, H), (H, I))
        return dict(bytes=L * sum(rows(Q4_0, n, k) + e * n for n, k in shapes) + L * e * (2 * H + Q + I),
                    flops=2 * L * sum(n * k for n, k in shapes))
    if f in ("xq8", "batch", "prefill", "exl3"):
        H, I, L = case["H"], case["I"], case.get("L", 1)
        M = case.get("M", case.get("B", 1))
        if f == "exl3":
            w = 3 * (H * I // 2 + 2 * (H + I))
        else:
            w = 2 * rows(case["gu"], I, H) + rows(case["down"], H, I)
        acts = e * M * (H + I + 2 * I + H + (H if f in ("batch", "prefill") else 0))
        if f == "xq8":
            acts = e * (H + H + 2 * I + H)
        return dict(bytes=L * (w + acts), flops=2 * L * M * 3 * H * I)
    T, H, I, E = (case[k] for k in ("T", "H", "I", "E"))
    per = 3 * rows(case["ty"], I, H) if f == "moe" else 3 * (H * I // 2 + 2 * (H + I))
    shared = per if f == "moe" else 6 * H * I
    return dict(bytes=_hit(case) * per + shared + T * (2 * e * H + 4 * E), flops=2 * T * (TOPK + 1) * 3 * H * I)


def tolerance(case):
    """About four times the measured distance to exact(). An output of bf16 is its own rounding, 1.7e-3; fp16 and
    float32 outputs of activations that the kernels take as fp16 are 2e-4 to 3.7e-4 off. The int8 products of the
    xq8 path are exact and their float32 sums 1e-7 off, but a sum that falls on the other side of a rounding moves one
    of the int8 activations that down reads by one step: 1.8e-4 of its result."""
    if case["family"] == "xq8":
        return {"rel": 7e-4}
    return {"rel": 7e-3 if case.get("x") == "bf16" else 1.5e-3}


# ---- the same in 64 bits ---------------------------------------------------------------------------

def _f16_at(b, at):
    return b[:, at:at + 2].contiguous().view(F16)[:, 0].double()


def _scales_k4(b):
    """The eight 6-bit scales and mins of Q4_K / Q5_K super-blocks."""
    s = b[:, 4:16].long()
    sc = torch.cat([s[:, 0:4] & 63, (s[:, 8:12] & 15) | (s[:, 0:4] >> 6 << 4)], 1)
    mn = torch.cat([s[:, 4:8] & 63, (s[:, 8:12] >> 4) | (s[:, 4:8] >> 6 << 4)], 1)
    return sc.double(), mn.double()


_GRID = None


def _grid():
    global _GRID
    if _GRID is None:
        with open(os.path.join(DATA, "iq2s_grid.json")) as fh:
            words = [int(h, 16) for h in json.load(fh)["grid_u64_hex"]]
        _GRID = torch.tensor([[w >> (8 * j) & 255 for j in range(8)] for w in words], dtype=torch.float64, device="cuda")
    return _GRID


def _decode(ty, raw, rows, K):
    """Packed rows -> float64 [rows, K]."""
    nw, nb = BLOCK[ty]
    b = raw.view(-1, nb)
    n = b.shape[0]
    if ty == Q4_0:
        q = torch.cat([b[:, 2:] & 15, b[:, 2:] >> 4], 1).double() - 8
        w = q * _f16_at(b, 0)[:, None]
    elif ty == Q8_0:
        w = b[:, 2:].contiguous().view(torch.int8).double() * _f16_at(b, 0)[:, None]
    elif ty in (Q4_K, Q5_K):
        sc, mn = _scales_k4(b)
        qs = b[:, 16 if ty == Q4_K else 48:].reshape(n, 4, 1, 32)
        q = torch.cat([qs & 15, qs >> 4], 2).reshape(n, 8, 32).double()
        if ty == Q5_K:
            j = torch.arange(8, device=b.device, dtype=torch.uint8).view(1, 8, 1)
            q += 16.0 * ((b[:, None, 16:48] >> j) & 1)
        w = (_f16_at(b, 0)[:, None] * sc)[:, :, None] * q - (_f16_at(b, 2)[:, None] * mn)[:, :, None]
    elif ty == Q6_K:
        ql, qh = b[:, :128].reshape(n, 2, 2, 32), b[:, 128:192].reshape(n, 2, 1, 32)
        lo = torch.cat([ql & 15, ql >> 4], 2)
        sh = torch.arange(0, 8, 2, device=b.device, dtype=torch.uint8).view(1, 1, 4, 1)
        q = (lo | (((qh >> sh) & 3) << 4)).double() - 32
        sc = b[:, 192:208].contiguous().view(torch.int8).double().view(n, 2, 4, 2, 1)
        w = q.view(n, 2, 4, 2, 16) * sc * _f16_at(b, 208).view(n, 1, 1, 1, 1)
    else:
        qh = b[:, 66:74].long().view(n, 8, 1)
        l2 = torch.arange(0, 8, 2, device=b.device).view(1, 1, 4)
        idx = b[:, 2:34].long().view(n, 8, 4) | (((qh >> l2) & 3) << 8)
        s8 = b[:, 74:82]
        nib = torch.stack([s8 & 15, s8 & 15, s8 >> 4, s8 >> 4], 2).double()
        db = _f16_at(b, 0).view(n, 1, 1) * (0.5 + nib) * 0.25
        j = torch.arange(8, device=b.device, dtype=torch.uint8)
        neg = (b[:, 34:66].reshape(n, 8, 4, 1) >> j) & 1
        w = db[..., None] * _grid()[idx] * (1.0 - 2.0 * neg)
    return w.reshape(rows, K)


def _mul(x, ty, raw, N, K):
    """x [M, K] float64 times packed rows [N, K], in slices of rows."""
    nw, nb = BLOCK[ty]
    rb, step = K // nw * nb, max(1, (1 << 25) // K)
    out = [x @ _decode(ty, raw[a * rb:min(a + step, N) * rb], min(step, N - a), K).t().contiguous()
           for a in range(0, N, step)]
    return torch.cat(out, 1)


_SLOTS = None


def _slots():
    global _SLOTS
    if _SLOTS is None:
        with open(os.path.join(DATA, "exl3_slot_composition.json")) as fh:
            slots = json.load(fh)["slots"]
        nib, pos = torch.zeros(256, 4, dtype=torch.long), torch.zeros(256, 4, dtype=torch.long)
        for r, c, members in slots:
            for i, (a, p) in enumerate(members):
                nib[16 * r + c, i], pos[16 * r + c, i] = a, p
        _SLOTS = nib.cuda(), pos.cuda()
    return _SLOTS


def _hadamard():
    h = torch.ones(1, 1, dtype=torch.float64, device="cuda")
    for _ in range(7):
        h = torch.cat([torch.cat([h, h], 1), torch.cat([h, -h], 1)])
    return h / math.sqrt(128.0)


def _rotate(x):
    return (x.reshape(-1, 128) @ _hadamard()).reshape(x.shape)


def _exl3_mul(x, trellis, suh, svh, K, N):
    """x [M, K] float64 times an EXL3 matrix, in slices of 16-row tile rows."""
    nib, pos = _slots()
    z = torch.zeros(x.shape[0], N, dtype=torch.float64, device="cuda")
    xr = _rotate(x * suh.double())
    step = max(1, (1 << 22) // (16 * N))
    for a in range(0, K // 16, step):
        t = trellis[a:a + step].reshape(-1, 64).view(torch.uint8).int()       # [tiles, 128]
        n = torch.stack([t & 15, t >> 4], 2).reshape(-1, 256)                 # nibbles, low first
        w = sum(n[:, nib[:, i]].long() << (4 * pos[:, i]) for i in range(4))  # [tiles, 256] windows
        y = (w * 0xCBAC1FED & 0x8FFF8FFF) ^ 0x3B603B60
        half = lambda v: v.to(torch.int16).view(F16).float()                  # noqa: E731
        lo, hi = half(((y & 0xFFFF) ^ 0x8000) - 0x8000), half(((y >> 16) ^ 0x8000) - 0x8000)
        v = (lo + hi).to(F16).double().view(-1, N // 16, 16, 16).transpose(1, 2).reshape(-1, N)
        z += xr[:, 16 * a:16 * a + v.shape[0]].contiguous() @ v
    return _rotate(z) * svh.double()


def _q8(x):
    """The q8 activation format: float32 scale a / 127 per 32 values, int8 round-half-even."""
    b = x.float().view(*x.shape[:-1], -1, 32)
    a = b.abs().amax(-1, keepdim=True)
    q = torch.where(a > 0, torch.round(b * (127.0 / a)), torch.zeros_like(b)).clamp(-128, 127)
    return (q.double() * (a / 127.0).double()).view(x.shape)


def _swiglu(g, u, limit=None):
    if limit is not None:
        g, u = g.clamp(max=limit), u.clamp(-limit, limit)
    return g * torch.sigmoid(g) * u


def exact(case, seed):
    s, f = _inputs(case, seed), case["family"]
    if f == "gemv":
        return _mul(s["X"].double()[None], case["ty"], s["W"], case["N"], case["K"])[0]
    if f == "stack":
        src = dict(q="attn", k="attn", v="attn", o="o", gate="mlp", up="mlp", down="down")
        return {k: torch.cat([_mul(s["X"][src[k]].double()[None], Q4_0, W[k], *shape) for W in s["W"]])
                for k, shape in s["shapes"].items()}
    if f == "xq8":
        H, I, out = case["H"], case["I"], dict(gate=[], up=[], down=[])
        for x, W in zip(s["X"], s["W"]):
            x = x.double()
            q = _q8(x / torch.sqrt((x * x).mean() + EPS) * W["norm"].double())[None]
            gate, up = (_mul(q, case["gu"], W[k], I, H) for k in ("gate", "up"))
            down = _mul(_q8(_swiglu(gate, up)), case["down"], W["down"], H, I) + x
            for k, v in (("gate", gate), ("up", up), ("down", down)):
                out[k].append(v)
        return {k: torch.cat(v) for k, v in out.items()}
    if f in ("batch", "prefill"):
        H, I, got = case["H"], case["I"], dict(gate=[], up=[], down=[])
        x, xd, r = (s[k].double() for k in ("X", "XD", "R"))
        if case.get("q8"):
            x, xd = _q8(s["X"]), _q8(s["XD"])
        for W in s["W"]:
            got["gate"].append(_mul(x, case["gu"], W["gate"], I, H))
            got["up"].append(_mul(x, case["gu"], W["up"], I, H))
            got["down"].append(_mul(xd, case["down"], W["down"], H, I) + r)
        return {k: torch.stack(v) if f == "batch" else v[0] for k, v in got.items()}
    if f == "exl3":
        H, I = case["H"], case["I"]
        x, xd = s["X"].double(), s["XD"].double()
        return dict(gate=torch.stack([_exl3_mul(x, *W["gate"], H, I) for W in s["W"]]),
                    up=torch.stack([_exl3_mul(x, *W["up"], H, I) for W in s["W"]]),
                    down=torch.stack([_exl3_mul(xd, *W["down"], I, H) for W in s["W"]]))
    T, H, I = (case[k] for k in ("T", "H", "I"))
    x, score = s["X"].double(), torch.sigmoid(s["logits"].double())
    idx = torch.topk(score if s["B"] is None else score + s["B"].double(), TOPK, dim=1).indices
    w = score.gather(1, idx)
    w = w / (w.sum(1, keepdim=True) + 1e-20) * ROUTE_SCALE
    if f == "moe":
        ty = case["ty"]
        rh, ri = (k // BLOCK[ty][0] * BLOCK[ty][1] for k in (H, I))
        ffn = lambda v, g, u, d: _mul(_swiglu(_mul(v, ty, g, I, H), _mul(v, ty, u, I, H), LIMIT), ty, d, H, I)  # noqa: E731
        out = ffn(x, *s["S"])
        expert = lambda v, e: ffn(v, *(m[e * n:(e + 1) * n] for m, n in zip(s["W"], (I * rh, I * rh, H * ri))))  # noqa: E731
    else:
        g, u, d = (m.double().t().contiguous() for m in s["S"])
        out = _swiglu(x @ g, x @ u, LIMIT) @ d
        expert = lambda v, e: _exl3_mul(_swiglu(_exl3_mul(v, *s["W"][e][0:3], H, I), _exl3_mul(v, *s["W"][e][3:6], H, I),  # noqa: E731
                                                LIMIT), *s["W"][e][6:9], I, H)
    for e in torch.unique(idx).tolist():
        t, k = torch.nonzero(idx == e, as_tuple=True)
        out.index_add_(0, t, w[t, k][:, None] * expert(x[t], e))
    return out
