"""What a program does with this package, as cases that can be timed and compared: sizes, inputs, one pass, and the
work of a pass.

A case is a dict of plain values. `kind` names the path and the other fields its sizes and options:

  decode   one generation step: for every layer of the stack the router's picks, then the fused expert layer, added
           into the residual stream
  prefill  a prompt through the expert layers, inference only: route, group by expert, gather + gate|up + SwiGLU, down,
           combine; the group sizes come back to the host between grouping and GEMMs, as the problem lists need them
  train    one expert layer forward and backward on bf16 activations: as prefill, with the pre-activations kept, then
           gate gradient, the two backward flushes (weight gradient beside input gradient), combine
  ffn32    an expert FFN on fp32 activations with fp32 arithmetic: up, down, both input gradients, both weight
           gradients, then one optimizer step on the matrices
  step     the optimizer's share of a training step: gradient norm, clip factor, integer AdamW or Lion over all spans
  codec    weights entering and leaving the 4-bit form on the GPU: encode, scale servo, render
  export   the checkpoint wire format on the host: write and read back

D is the model width, F the width of an expert, E the experts of a layer, K the experts of a token, N the tokens of a pass.
"""
import importlib
import math

import numpy as np
import torch

PROB = np.dtype([("A", "<u8"), ("B", "<u8"), ("C", "<u8"), ("wq", "<u8"), ("wg", "<u8"), ("M", "<i4"), ("beta", "<f4")])
DMAX = 7
MODES = ("gate", "up", "down", "g2", "d2", "g13", "d1", "d3")


def listed():
    return [
        # a chat answered token by token, the step recorded as a graph: launch latency and the chain inside a layer
        dict(name="decode_one", kind="decode", N=1, E=32, K=2, D=768, F=2048, layers=8, graph=True),
        # the same model serving sixteen sequences, called eagerly
        dict(name="decode_batch", kind="decode", N=16, E=32, K=2, D=768, F=2048, layers=8, graph=False),
        # the wide model (64 experts, top-4) serving an odd number of sequences
        dict(name="decode_wide", kind="decode", N=11, E=64, K=4, D=2048, F=1408, layers=4, graph=True),
        # a short prompt: a dozen rows per expert, too many for the decode path and far from a full tile
        dict(name="prefill_prompt", kind="prefill", N=193, E=32, K=2, D=768, F=2048, layers=4, skew=0.0),
        # a long prompt on the wide model
        dict(name="prefill_long", kind="prefill", N=3001, E=64, K=4, D=2048, F=1408, layers=1, skew=0.0),
        # fine-tuning a small model on a small ragged batch
        dict(name="train_small", kind="train", N=1000, E=8, K=1, D=512, F=1536, skew=0.0),
        # the training layer of the 32-expert model, 8 x 1024 tokens, Zipf load
        dict(name="train_layer", kind="train", N=8192, E=32, K=2, D=768, F=2048, skew=1.1),
        # a layer of the wide model, 16 x 2048 tokens, Zipf load
        dict(name="train_large", kind="train", N=32768, E=64, K=4, D=2048, F=1408, skew=1.1),
        # the fp32 path, what a caller gets who binds the GEMMs without asking for the matrix-core types
        dict(name="ffn_fp32", kind="ffn32", N=1024, E=1, D=512, F=1536, group=128),
        # the optimizer over all weights of the 120 M model
        dict(name="step_sweep", kind="step", n=125829120, spans=3, group=128, adam=True, lrmode=0, render=False),
        # an expert stack quantised at start-up, its scales served once, the fp32 view written for an evaluation
        dict(name="codec_stack", kind="codec", n=150994944, spans=3, group=128),
        # a checkpoint: rendered expert weights on the 4-bit grid with a share of parameters that are not on it
        dict(name="export_shard", kind="export", n=4000037, group=128, raw=0.1),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _width(rng, lo, hi):
    return 128 * max(1, round(_log(rng, lo, hi) / 128))


def draw(rng):
    kind = rng.choice(("decode", "decode", "decode", "prefill", "prefill", "train", "train", "train", "ffn32", "step", "step", "codec", "export"))
    if kind in ("decode", "prefill", "train"):
        E = rng.choice((8, 16, 32, 64))
        K = rng.choice((1, 2, 4))
        D, F = _width(rng, 256, 2048), _width(rng, 512, 2816)
        weights = 3 * E * D * F
        if kind == "decode":
            layers = max(1, min(8, 1200000000 // weights))
            return dict(kind=kind, N=_log(rng, 1, min(32, 64 // K)), E=E, K=K, D=D, F=F, layers=layers, graph=rng.random() < 0.5)
        skew = rng.choice((0.0, 0.0, 1.1))
        if kind == "prefill":
            N = _log(rng, 70, 4096)
            return dict(kind=kind, N=N, E=E, K=K, D=D, F=F, layers=max(1, min(4, 600000000 // weights, 4096 // N)), skew=skew)
        most = 32768 * 4 * 2048 * 1408 // (K * D * F)
        return dict(kind=kind, N=_log(rng, 250, min(32768, most)), E=E, K=K, D=D, F=F, skew=skew)
    if kind == "ffn32":
        return dict(kind=kind, N=_log(rng, 16, 4096), E=rng.choice((1, 1, 4, 8)), D=_width(rng, 256, 1024), F=_width(rng, 512, 2048),
                    group=rng.choice((64, 128)))
    if kind == "step":
        return dict(kind=kind, n=32 * _log(rng, 2048, 3932160), spans=rng.randint(1, 24), group=rng.choice((64, 128, 128, 128)),
                    adam=rng.random() < 0.75, lrmode=rng.choice((0, 0, 1)), render=rng.random() < 0.25)
    if kind == "codec":
        return dict(kind=kind, n=32 * _log(rng, 8192, 4718592), spans=rng.randint(1, 24), group=rng.choice((64, 128, 128, 128)))
    return dict(kind=kind, n=_log(rng, 50000, 4000000), group=rng.choice((64, 128, 128)), raw=rng.choice((0.0, 0.1, 0.5)))


# ------------------------------------------------------------------------------------------------ inputs
class Maker:
    """Arrays made on the GPU from one seed."""

    def __init__(self, seed):
        self.dev = torch.device("cuda")
        self.g = torch.Generator(device=self.dev)
        self.g.manual_seed(seed)

    def normal(self, *shape, scale=1.0, dtype=torch.float32):
        return torch.randn(*shape, device=self.dev, generator=self.g).mul_(scale).to(dtype)

    def scales(self, n, mean):
        return torch.rand(n, device=self.dev, generator=self.g).add_(0.5).mul_(mean)

    def whole(self, n, lo, hi, dtype):
        return torch.randint(lo, hi + 1, (n,), device=self.dev, generator=self.g, dtype=torch.int16).to(dtype)

    def digits(self, n):
        """n packed 4-bit codes of -7..7, as an encoder leaves them"""
        b = torch.randint(0, 225, (n // 2,), device=self.dev, generator=self.g, dtype=torch.uint8)
        lo, hi = b % 15 - 7 & 15, b // 15 - 7 & 15
        return (lo | hi << 4).view(torch.int8)

    def logits(self, N, E, skew):
        """Router logits ~ N(0, 1); with a skew, such that the top-K picks follow p_e ~ (e + 1)^-skew without replacement."""
        if skew == 0.0:
            return self.normal(N, E)
        u = torch.rand(N, E, device=self.dev, generator=self.g).clamp_(1e-7, 1 - 1e-7)
        rank = torch.arange(1, E + 1, device=self.dev, dtype=torch.float32)
        return -torch.log(-torch.log(u)) - skew * torch.log(rank)

    def empty(self, *shape, dtype=torch.float32):
        return torch.empty(*shape, device=self.dev, dtype=dtype)

    def zeros(self, *shape, dtype=torch.float32):
        return torch.zeros(*shape, device=self.dev, dtype=dtype)


def _package():
    return importlib.import_module("cudalm-c_amd")


def _spans(P, n, count, group):
    """`count` tensors of n elements in all, sizes in a ratio of up to three and multiples of 32, back to back"""
    share = [1.0 + 2.0 * ((i * 7) % 5) / 5 for i in range(count)]
    sizes = [int(n * w / sum(share)) // 32 * 32 for w in share]
    sizes[-1] += n - sum(sizes)
    tab = np.zeros(count, dtype=P.SPAN_DTYPE)
    at = groups = 0
    for i, m in enumerate(sizes):
        ng = -(-m // group)
        tab[i] = (at, at, at, m, groups, ng, 0.01, 0)
        at, groups = at + m, groups + ng
    return tab, groups


def _optimizer(m, n, groups):
    return dict(r=m.whole(n, -64, 64, torch.int8), m8=m.whole(n, -127, 127, torch.int8), v8=m.whole(n, 0, 255, torch.uint8),
                m8s=m.scales(groups, 3e-3 / 127), v8s=m.scales(groups, 3e-3 / 255), t=0)


class State:
    """What a program keeps between passes: attributes only."""

    def __init__(self, case, **more):
        self.__dict__.update(case)
        self.__dict__.update(more)


def prepare(case, seed):
    P = _package()
    if case["kind"] == "export":
        return _prepare_export(P, case, seed)
    s = State(case, q=P.load(), P=P, m=Maker(seed))
    return {"decode": _prepare_decode, "prefill": _prepare_grouped, "train": _prepare_grouped, "ffn32": _prepare_ffn32,
            "step": _prepare_step, "codec": _prepare_codec}[case["kind"]](s)


def _layer_weights(s):
    """w1 | w3 | w2 of a layer's experts, back to back"""
    n = 3 * s.E * s.D * s.F
    return s.m.digits(n), s.m.scales(n // 128, 0.02 * 3 / 7)


def _prepare_decode(s):
    m, L = s.m, s.layers
    s.w = [_layer_weights(s) for _ in range(L)]
    s.x = [m.normal(s.N, s.D) for _ in range(L)]
    s.logits = [m.normal(s.N, s.E) for _ in range(L)]
    s.h = m.normal(s.N, s.D)
    s.rprobs = m.empty(s.N, s.E)
    s.assign = [m.empty(s.K, s.N, dtype=torch.int32) for _ in range(L)]
    s.gates = [m.empty(s.K, s.N) for _ in range(L)]
    s.tape = None
    if s.graph:
        h = s.h.clone()
        side = torch.cuda.Stream()
        side.wait_stream(torch.cuda.current_stream())
        with torch.cuda.stream(side):
            _decode_step(s, side.cuda_stream)
            side.synchronize()
            s.tape = torch.cuda.CUDAGraph()
            with torch.cuda.graph(s.tape, stream=side):
                _decode_step(s, side.cuda_stream)
        torch.cuda.current_stream().wait_stream(side)
        s.h.copy_(h)
    return s


def _prepare_grouped(s):
    m, E, D, F, N = s.m, s.E, s.D, s.F, s.N
    R = N * s.K
    s.L = s.layers if s.kind == "prefill" else 1
    s.w = [_layer_weights(s) for _ in range(s.L)]
    s.logits = [m.logits(N, E, s.skew) for _ in range(s.L)]
    bf = torch.bfloat16
    s.x = [m.normal(N, D, dtype=bf if s.kind == "prefill" else torch.float32) for _ in range(s.L)]
    s.h = m.normal(N, D)
    s.rprobs, s.gates = m.empty(N, E), m.empty(s.K, N)
    s.assign, s.perm, s.tok, s.inv = (m.empty(R, dtype=torch.int32) for _ in range(4))
    s.off = m.empty(E + 1, dtype=torch.int32)
    s.ws = m.empty(s.q.moe_perm_workspace(R, E, 1), dtype=torch.uint8)
    s.act, s.y = m.empty(R, F, dtype=bf), m.empty(R, D)
    if s.kind == "train":
        s.dout, s.dx = m.normal(N, D), m.zeros(N, D)
        s.xp, s.dyp = m.empty(R, D, dtype=bf), m.empty(R, D, dtype=bf)
        s.gp, s.up = m.empty(R, F), m.empty(R, F)
        s.dgp, s.dup = m.empty(R, F, dtype=bf), m.empty(R, F, dtype=bf)
        s.dxp, s.dgate = m.empty(R, D), m.empty(s.K, N)
        s.G = m.empty(3 * E * D * F)
    # the problem lists: the columns that name weights stay, the others are filled in from the group sizes
    s.table, s.col = {}, {}
    for name in MODES if s.kind == "train" else MODES[:3]:
        n = 2 * E if name == "g13" else E
        s.table[name] = (s.P.GemmProb * n)()
        c = s.col[name] = np.frombuffer(s.table[name], dtype=PROB)
        matrix = {"gate": 0, "up": 1, "down": 2, "g2": 2, "d2": 2, "g13": 0, "d1": 0, "d3": 1}[name]
        at = (matrix * E + np.arange(n, dtype=np.uint64)) * np.uint64(D * F)
        if name in ("g2", "g13"):
            c["C"] = np.uint64(s.G.data_ptr()) + at * np.uint64(4)
        else:
            c["wq"], c["wg"] = at, at // np.uint64(128)
        if name == "d3":
            c["beta"] = 1.0
    return s


def _prepare_ffn32(s):
    m, E, D, F = s.m, s.E, s.D, s.F
    n = E * D * F
    rows = np.random.RandomState(s.m.g.initial_seed() % (1 << 31)).multinomial(s.N, [1.0 / E] * E)
    s.rows, s.at = rows, np.concatenate([[0], np.cumsum(rows)[:-1]])
    s.d, s.s = m.digits(2 * n), m.scales(2 * n // s.group, 0.02 * 3 / 7)
    s.x, s.dy = m.normal(s.N, D), m.normal(s.N, D)
    s.hid, s.y, s.dhid, s.dx = m.empty(s.N, F), m.empty(s.N, D), m.empty(s.N, F), m.empty(s.N, D)
    s.G = m.empty(2 * n)
    s.grad = m.normal(2 * n, scale=1e-3)
    groups = 2 * n // s.group
    s.tab = np.zeros(2, dtype=s.P.SPAN_DTYPE)
    for i in range(2):
        s.tab[i] = (i * n, i * n, i * n, n, i * groups // 2, groups // 2, 0.02 * 3 / 7, 0)
    s.sp = torch.from_numpy(s.tab.view(np.uint8)).cuda()
    s.groups = groups
    s.opt = _optimizer(m, 2 * n, groups)

    def problems(A, a, B, b, C, c, w):
        return s.q.problems([(A.data_ptr() + int(s.at[e]) * a * 4, None if B is None else B.data_ptr() + int(s.at[e]) * b * 4,
                              C.data_ptr() + ((w * n + e * D * F) * 4 if C is s.G else int(s.at[e]) * c * 4),
                              w * n + e * D * F, (w * n + e * D * F) // s.group, int(rows[e]), 0.0) for e in range(E)])
    s.up, s.down = problems(s.x, D, None, 0, s.hid, F, 0), problems(s.hid, F, None, 0, s.y, D, 1)
    s.d2, s.d1 = problems(s.dy, D, None, 0, s.dhid, F, 1), problems(s.dhid, F, None, 0, s.dx, D, 0)
    s.g2, s.g1 = problems(s.hid, F, s.dy, D, s.G, 0, 1), problems(s.x, D, s.dhid, F, s.G, 0, 0)
    return s


def _prepare_step(s):
    m = s.m
    s.tab, s.groups = _spans(s.P, s.n, s.spans, s.group)
    s.sp = torch.from_numpy(s.tab.view(np.uint8)).cuda()
    s.d, s.s = m.digits(s.n), m.scales(s.groups, 0.02 * 3 / 7)
    s.grad = m.normal(s.n, scale=1e-3)
    s.view = m.empty(s.n) if s.render else None
    s.part, s.clip = m.empty(64), m.empty(2)
    s.opt = _optimizer(m, s.n, s.groups)
    return s


def _prepare_codec(s):
    m = s.m
    s.tab, s.groups = _spans(s.P, s.n, s.spans, s.group)
    s.sp = torch.from_numpy(s.tab.view(np.uint8)).cuda()
    s.w = m.normal(s.n, scale=0.02)
    s.d, s.r, s.s = m.zeros(s.n // 2, dtype=torch.int8), m.zeros(s.n, dtype=torch.int8), m.zeros(s.groups)
    s.view = m.empty(s.n)
    return s


def _prepare_export(P, case, seed):
    rng = np.random.default_rng(seed)
    n, g = case["n"], case["group"]
    groups = -(-n // g)
    digit = rng.integers(-DMAX, DMAX + 1, groups * g, dtype=np.int8).reshape(groups, g)
    scale = (0.02 * 3 / 7 * (0.5 + rng.random(groups, dtype=np.float32))).astype(np.float32)
    v = digit.astype(np.float32) * scale[:, None]
    off = rng.permutation(groups - 1)[:round(case["raw"] * groups)]
    v[off] = 0.02 * rng.standard_normal((len(off), g), dtype=np.float32)
    return State(case, q=P.Qlmx(init=False), v=np.ascontiguousarray(v.reshape(-1)[:n]))


# ------------------------------------------------------------------------------------------------ one pass
def run(s):
    return {"decode": _run_decode, "prefill": _run_prefill, "train": _run_train, "ffn32": _run_ffn32, "step": _run_step,
            "codec": _run_codec, "export": _run_export}[s.kind](s)


def _decode_step(s, stream):
    q, nw = s.q, s.E * s.D * s.F
    for l, (d, sc) in enumerate(s.w):
        q.router_topk(s.logits[l], s.rprobs, s.assign[l], s.gates[l], s.N, s.E, s.K, None, 0, stream)
        q.decode_forward(s.x[l], s.assign[l], s.gates[l], s.h, d, sc, 128, 0, nw, 2 * nw, s.N, s.K, s.E, s.D, s.F, stream)


def _run_decode(s):
    if s.tape is not None:
        s.tape.replay()
    else:
        _decode_step(s, torch.cuda.current_stream().cuda_stream)
    return {"h": s.h, "assign": s.assign, "gates": s.gates}


def _group(s, l, stream):
    """Route and group the tokens by expert; the first row of every expert, on the host."""
    q, N, E, K = s.q, s.N, s.E, s.K
    q.router_topk(s.logits[l], s.rprobs, s.assign, s.gates, N, E, K, None, 0, stream)
    q.moe_perm(s.assign, N * K, E, 1, s.perm, s.off, s.ws, stream)
    q.moe_merge_rows(s.perm, N, K, s.tok, s.inv, stream)
    off = s.off.cpu().numpy().astype(np.uint64)
    first, rows = off[:-1], np.diff(off)

    def fill(name, **columns):
        c = s.col[name]
        c["M"] = rows
        for key, (base, width) in columns.items():
            c[key] = np.uint64(base.data_ptr()) + first * np.uint64(width * base.element_size())
        return s.table[name]
    return fill, first, rows


def _run_prefill(s):
    q, P, E, D, F, N = s.q, s.P, s.E, s.D, s.F, s.N
    stream = torch.cuda.current_stream().cuda_stream
    for l, (d, sc) in enumerate(s.w):
        fill, _, _ = _group(s, l, stream)
        gate, up = fill("gate", A=(s.tok, 1)), fill("up", B=(s.act, F))
        q.gemm_nn_gather_swiglu(d, sc, 128, gate, up, E, D, F, s.x[l], stream)
        q.gemm_nn(d, sc, 128, fill("down", A=(s.act, F), C=(s.y, D)), E, F, D, P.ACT_BF16, P.MATH_MFMA_F16, stream)
        q.moe_combine(s.y, s.inv, s.gates, s.h, N, s.K, D, stream)
    return {"h": s.h, "assign": s.assign, "tok": s.tok}


def _run_train(s):
    q, P, E, D, F, N, K = s.q, s.P, s.E, s.D, s.F, s.N, s.K
    stream = torch.cuda.current_stream().cuda_stream
    bf, (d, sc) = P.ACT_BF16, s.w[0]
    fill, first, rows = _group(s, 0, stream)
    # forward
    q.moe_gather(s.x[0], s.tok, s.xp, N * K, D, bf, stream)
    q.gemm_nn_swiglu(d, sc, 128, fill("gate", A=(s.xp, D), C=(s.gp, F)), fill("up", B=(s.act, F), C=(s.up, F)), E, D, F, bf, P.MATH_MFMA_F16, stream)
    q.gemm_nn(d, sc, 128, fill("down", A=(s.act, F), C=(s.y, D)), E, F, D, bf, P.MATH_MFMA_F16, stream)
    q.moe_combine(s.y, s.inv, s.gates, s.h, N, K, D, stream)
    # backward
    q.moe_dgate_merged(s.dout, s.y, s.perm, s.gates, s.dgate, s.dyp, N, K, D, bf, stream)
    q.pair_begin(stream)
    q.gemm_nt(fill("g2", A=(s.act, F), B=(s.dyp, D)), E, F, D, bf, P.MATH_MFMA, stream)
    q.gemm_tn_swiglu_bwd(d, sc, 128, fill("d2", A=(s.dyp, D), C=(s.gp, F)), E, D, F, s.gp, s.up, s.dgp, s.dup, stream)
    q.pair_end(stream)
    g13 = s.col["g13"]
    g13["M"] = np.tile(rows, 2)
    g13["A"] = np.uint64(s.xp.data_ptr()) + np.tile(first, 2) * np.uint64(D * 2)
    g13["B"][:E] = np.uint64(s.dgp.data_ptr()) + first * np.uint64(F * 2)
    g13["B"][E:] = np.uint64(s.dup.data_ptr()) + first * np.uint64(F * 2)
    d1, d3 = fill("d1", A=(s.dgp, F), C=(s.dxp, D)), fill("d3", A=(s.dup, F), C=(s.dxp, D))
    q.pair_begin(stream)
    q.gemm_nt(s.table["g13"], 2 * E, D, F, bf, P.MATH_MFMA, stream)
    q.gemm_tn_pair(d, sc, 128, d1, d3, E, F, D, bf, P.MATH_MFMA, stream)
    q.pair_end(stream)
    q.moe_combine(s.dxp, s.inv, None, s.dx, N, K, D, stream)
    return {"h": s.h, "dx": s.dx, "dgate": s.dgate, "G": s.G, "tok": s.tok}


def _optimize(s, gscale, gsp, view, adam, lrmode, stream):
    o = s.opt
    o["t"] += 1
    t, b1, b2 = o["t"], 0.9, 0.95
    s.q.step(view, s.grad, s.d, o["r"], s.s, o["m8"], o["m8s"], o["v8"], o["v8s"], s.sp, len(s.tab), s.group, DMAX, 3e-4, b1, b2, 0.1,
             gscale, gsp, 1.0 / (1.0 - b1 ** t), 1.0 / (1.0 - b2 ** t) ** 0.5, lrmode, t, int(adam), None, 1, 0, s.groups, 0, stream)
    return {"d": s.d, "r": o["r"], "m8": o["m8"], "m8s": o["m8s"], "v8": o["v8"], "v8s": o["v8s"]}


def _run_ffn32(s):
    q, P, E, D, F, g = s.q, s.P, s.E, s.D, s.F, s.group
    stream = torch.cuda.current_stream().cuda_stream
    f = P.ACT_F32, P.MATH_F32, stream
    q.gemm_nn(s.d, s.s, g, s.up, E, D, F, *f)
    q.gemm_nn(s.d, s.s, g, s.down, E, F, D, *f)
    q.gemm_nt(s.g2, E, F, D, *f)
    q.gemm_tn(s.d, s.s, g, s.d2, E, D, F, *f)
    q.gemm_nt(s.g1, E, D, F, *f)
    q.gemm_tn(s.d, s.s, g, s.d1, E, F, D, *f)
    return dict(_optimize(s, 1.0, None, None, True, 0, stream), y=s.y, dx=s.dx, G=s.G)


def _run_step(s):
    stream = torch.cuda.current_stream().cuda_stream
    s.q.sqsum(s.grad, s.n, s.part, stream)
    s.q.gnorm(s.part, 0, 0, s.clip, stream)
    out = _optimize(s, 1.0, s.clip, s.view, s.adam, s.lrmode, stream)
    out["clip"] = s.clip
    if s.view is not None:
        out["P"] = s.view
    return out


def _run_codec(s):
    q, a = s.q, (s.sp, len(s.tab), s.group)
    stream = torch.cuda.current_stream().cuda_stream
    q.encode(s.w, s.d, s.r, s.s, *a, DMAX, 1, s.groups, stream)
    q.servo(s.d, s.r, s.s, *a, DMAX, 0.02, 0.002, 1, s.groups, stream)
    q.render(s.view, s.d, s.s, *a, 1, 0, s.groups, stream)
    return {"d": s.d, "r": s.r, "s": s.s, "P": s.view}


def _run_export(s):
    wire, raw = s.q.q4n_quantize(s.v, s.group)
    back, used = s.q.q4n_dequantize(wire, s.n, s.group)
    return {"wire": wire, "raw": raw, "back": back, "used": used}


# ------------------------------------------------------------------------------------------------ work, tolerance
def work(case):
    c = State(case)
    if c.kind in ("decode", "prefill", "train"):
        per_expert = 3 * c.D * c.F * (0.5 + 4 / 128)
        route = c.N * c.E * 8 + c.N * c.K * 8
        R = c.N * c.K
        hit = c.E * (1.0 - (1.0 - c.K / c.E) ** c.N)      # experts that a layer's tokens reach, evenly routed
        if c.kind == "decode":
            return {"bytes": c.layers * (hit * per_expert + 12 * c.N * c.D + route), "flops": c.layers * 6 * R * c.D * c.F}
        if c.kind == "prefill":
            return {"bytes": c.layers * (hit * per_expert + 10 * c.N * c.D + route), "flops": c.layers * 6 * R * c.D * c.F}
        # x, dout, h, dx; the kept pre-activations and activation written once and read once; digits for both directions once; G
        return {"bytes": hit * per_expert + 24 * c.N * c.D + 2 * R * c.F * 10 + 3 * c.E * c.D * c.F * 4 + route, "flops": 18 * R * c.D * c.F}
    if c.kind == "ffn32":
        n = 2 * c.E * c.D * c.F
        # x, dy, y, dx; the hidden rows written once and read once; G; then the optimizer's state and gradient
        return {"bytes": c.N * (16 * c.D + 8 * c.F) + 4 * n + n * (11 + 20 / c.group), "flops": 12 * c.N * c.D * c.F}
    if c.kind == "step":
        moments = 4 if c.adam else 2
        # the norm has to be known before the first weight moves, so the gradient is read twice
        return {"bytes": c.n * (8 + 1 + 2 + moments + 4 * int(c.render) + 4 * (1 + moments) / c.group), "flops": 0}
    if c.kind == "codec":
        return {"bytes": c.n * (4 + 0.5 + 1 + 4 + 4 / c.group), "flops": 0}
    groups = -(-c.n // c.group)
    wire = 4 * groups + c.n * ((1 - c.raw) * 0.5 + c.raw * 4)
    return {"bytes": 8 * c.n + 2 * wire, "flops": 0}


def tolerance(case):
    kind = case["kind"]
    if kind in ("step", "codec", "export"):
        return "exact"
    if kind in ("decode", "ffn32"):
        return {"rel": 1e-5}
    # bf16 activations between the GEMMs: 2^-9 a rounding, five of them in a row at most
    return {"rel": 5e-3, "max": 0.2}
