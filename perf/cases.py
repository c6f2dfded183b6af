"""The work that a user of the palettized-linear library has it do, as measurable cases.

Sizes are those of the benchmark and the tests: the seven linears of a decoder layer with hidden
size 2560, 32 query and 8 kv heads of 128 and an MLP of 9728, at 1..16 tokens (decode), at prompt
lengths (prefill) and at 32 x 512 tokens (training), plus odd sizes of the same ranges.

  decode       grouped GEMVs on packed 2-bit weights: a layer's four launches, or a stage of layers
  prefill      hard forward of a layer's seven linears with LoRA, without gradients
  hard         lut_linear forward + backward (x, palette, bias, LoRA)
  soft         soft_lut_linear forward + backward (x, palette, logits, LoRA), supplied noise
  dropin_hard  QwenLoRA(PalettizedLinear) forward + backward on frozen indices
  dropin_soft  QwenLoRA(PalettizedLinear) forward + backward on index logits (LCG noise)
  attention    causal grouped-query attention forward + backward
  layer        one distillation training step of a palettized decoder layer
"""
import math
import os
import sys

import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))),
                                "qwen-palettize_amd"))

from palettize_hip import fused_lut_linear_cuda as FL  # noqa: E402
from palettize_hip import lut_linear, ops, soft_lut_linear  # noqa: E402
from palettize_hip.layer import LayerConfig, LayerTrainer, attention  # noqa: E402
from palettize_hip.qwen_model import PalettizedLinear, QwenLoRA  # noqa: E402

# (K, N, LoRA rank) of a layer's q, k, v, o, gate, up, down, by hidden size
LINEARS = {2560: ((2560, 4096, 16), (2560, 1024, 16), (2560, 1024, 16), (4096, 2560, 32),
                  (2560, 9728, 16), (2560, 9728, 16), (9728, 2560, 32)),
           1024: ((1024, 2048, 16), (1024, 1024, 16), (1024, 1024, 16), (2048, 1024, 32),
                  (1024, 3072, 16), (1024, 3072, 16), (3072, 1024, 32))}
# the linears that share one input, i.e. one grouped decode launch each
DECODE_GROUPS = ((0, 1, 2), (3,), (4, 5), (6,))


# ---- the cases ------------------------------------------------------------------------------
def listed():
    return [
        # one token through one layer: q/k/v, o, gate/up and down depend on each other, so a
        # decode loop issues four grouped launches; the smallest call, where latency counts
        dict(name="decode_layer_m1", kind="decode", hidden=2560, M=1, layers=1,
             stage=False),
        # the whole weight stream of a nine-layer pipeline stage in one grouped launch, one token
        # and a full batch of sixteen
        dict(name="decode_stage_m1", kind="decode", hidden=2560, M=1, layers=9,
             stage=True),
        dict(name="decode_stage_m16", kind="decode", hidden=2560, M=16, layers=9,
             stage=True),
        # a decode batch too large for the GEMV (or a speculative window), and a ragged prompt
        dict(name="prefill_m48", kind="prefill", hidden=2560, M=48),
        dict(name="prefill_m777", kind="prefill", hidden=2560, M=777),
        # palette + LoRA training: a small ragged microbatch on q, the full batch on gate
        dict(name="hard_m1000_q", kind="hard", M=1000, K=2560, N=4096, rank=16, bias=False),
        dict(name="hard_m16384_gate", kind="hard", M=16384, K=2560, N=9728, rank=16, bias=False),
        # index training (Gumbel softmax) of the gate projection at the full batch
        dict(name="soft_m16384_gate", kind="soft", M=16384, K=2560, N=9728, rank=16, tau=0.5),
        # the modules that a training script of the original project constructs, in its layouts:
        # a microbatch of 4 x 512 tokens on q with the modules' default LoRA rank
        dict(name="dropin_hard_m2048_q", kind="dropin_hard", B=4, S=512, K=2560, N=4096, rank=32,
             bias=False),
        dict(name="dropin_soft_m2048_q", kind="dropin_soft", B=4, S=512, K=2560, N=4096, rank=32,
             bias=False, tau=1.0),
        # the layer step's attention by itself
        dict(name="attention_b32_s512", kind="attention", B=32, S=512, Hq=32, Hkv=8),
        # the whole training step: teacher, student, loss, backward, clipping, optimizer
        dict(name="layer_b32_s512", kind="layer", B=32, S=512, hidden=2560, heads=32, kv_heads=8,
             intermediate=9728),
    ]


def _log(rng, lo, hi):
    """A whole number whose logarithm is uniform over lo..hi."""
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def _shape(rng):
    """(K, N, rank) of one of the layer's linears, or a generic one (K in 256s, N in 8s)."""
    if rng.random() < 0.6:
        return rng.choice(LINEARS[2560])
    return 256 * _log(rng, 1, 38), 8 * _log(rng, 16, 1216), rng.choice((8, 16, 32))


def draw(rng):
    kind = rng.choice(("decode", "decode", "prefill", "prefill", "hard", "hard", "soft",
                       "dropin_hard", "dropin_soft", "attention", "attention", "layer"))
    if kind == "decode":
        stage = rng.random() < 0.6
        return dict(kind=kind, hidden=rng.choice((2560, 2560, 1024)),
                    M=rng.randint(1 if stage else 2, 16), layers=rng.randint(2, 9) if stage else 1,
                    stage=stage)
    if kind == "prefill":
        return dict(kind=kind, hidden=rng.choice((2560, 2560, 1024)), M=_log(rng, 17, 4096))
    if kind in ("hard", "soft"):
        K, N, rank = _shape(rng)
        c = dict(kind=kind, M=_log(rng, 64, 16384), K=K, N=N, rank=rank)
        if kind == "hard":
            c["bias"] = rng.random() < 0.3
        else:
            c["tau"] = rng.choice((2.0, 1.0, 0.5))
        return c
    if kind in ("dropin_hard", "dropin_soft"):
        K, N, _ = _shape(rng)
        c = dict(kind=kind, B=rng.randint(1, 8), S=_log(rng, 32, 1024), K=K, N=N,
                 rank=rng.choice((16, 32)), bias=rng.random() < 0.3)
        if kind == "dropin_soft":
            c["tau"] = rng.choice((2.0, 1.0, 0.5))
        return c
    if kind == "attention":
        S = 128 * _log(rng, 1, 32)
        Hq, Hkv = rng.choice(((32, 8), (16, 8), (8, 8), (16, 2)))
        return dict(kind=kind, B=rng.randint(1, max(1, 16384 // S)), S=S, Hq=Hq, Hkv=Hkv)
    S = 128 * _log(rng, 1, 16)
    cfg = rng.choice((dict(hidden=2560, heads=32, kv_heads=8, intermediate=9728),
                      dict(hidden=1024, heads=16, kv_heads=8, intermediate=3072)))
    return dict(kind=kind, B=rng.randint(1, 16384 // S), S=S, **cfg)


# ---- inputs -----------------------------------------------------------------------------------
def _bf(gen, *shape, std=1.0):
    return (torch.randn(*shape, generator=gen, device="cuda") * std).to(torch.bfloat16)


def _packed(gen, N, K):
    """Uniform 2-bit indices, packed: every 32-bit word is sixteen of them."""
    return torch.randint(-2 ** 31, 2 ** 31, (N, K // 16), generator=gen, device="cuda",
                         dtype=torch.int64).to(torch.int32)


def _palette(gen, N, G):
    return torch.sort(torch.randn(N, G, 4, generator=gen, device="cuda") * 0.02, -1).values


def _weight(gen, K, N):
    return _packed(gen, N, K), _palette(gen, N, K // 256).contiguous()


def _gumbel(gen, *shape):
    u = torch.rand(*shape, generator=gen, device="cuda").clamp_(1e-7, 1 - 6e-8)
    return -torch.log(-torch.log(u))


def _inputs(case, seed):
    """The tensors of a case, the same ones for prepare() and exact()."""
    g = torch.Generator(device="cuda").manual_seed(int(seed))
    kind, d = case["kind"], {}
    if kind in ("decode", "prefill"):
        layers = case["layers"] if kind == "decode" else 1
        linears = LINEARS[case["hidden"]]
        d["weights"] = [[_weight(g, K, N) for K, N, _ in linears] for _ in range(layers)]
        d["x"] = []
        for _ in range(layers):
            xs = [None] * len(linears)
            for grp in DECODE_GROUPS:
                x = _bf(g, case["M"], linears[grp[0]][0])
                for i in grp:
                    xs[i] = x
            d["x"].append(xs)
        if kind == "prefill":
            d["lora"] = [(_bf(g, r, K, std=0.01), _bf(g, N, r, std=0.01)) for K, N, r in linears]
        return d
    if kind in ("hard", "soft"):
        M, K, N, r = case["M"], case["K"], case["N"], case["rank"]
        d["x"], d["gy"] = _bf(g, M, K), _bf(g, M, N)
        d["a"], d["b"] = _bf(g, r, K, std=0.01), _bf(g, N, r, std=0.01)
        if kind == "hard":
            d["packed"], d["pal"] = _weight(g, K, N)
            d["bias"] = _bf(g, N, std=0.1) if case["bias"] else None
        else:
            d["pal"] = _palette(g, N, K // 256).contiguous()
            d["logits"] = _bf(g, N, K, 4)
            d["noise"] = _gumbel(g, N, K, 4)
        return d
    if kind in ("dropin_hard", "dropin_soft"):
        B, S, K, N, r = case["B"], case["S"], case["K"], case["N"], case["rank"]
        d["x"], d["gy"] = _bf(g, B, S, K), _bf(g, B, S, N)
        d["idx"] = torch.randint(0, 4, (K, N), generator=g, device="cuda")
        d["pal"] = _palette(g, -(-N // 256), 1)[:, 0].to(torch.bfloat16)
        d["a"], d["b"] = _bf(g, K, r, std=0.01), _bf(g, N, r, std=0.01)
        d["bias"] = _bf(g, N, std=0.1) if case["bias"] else None
        if kind == "dropin_soft":
            # part-way through training: the planes' mass still leans to one index
            d["logits"] = torch.randn(4, K, N, generator=g, device="cuda")
            d["logits"].scatter_add_(0, d["idx"][None], torch.full((1, K, N), 3.0, device="cuda"))
            d["logits"] = d["logits"].to(torch.float16)
        return d
    if kind == "attention":
        B, S, Hq, Hkv = case["B"], case["S"], case["Hq"], case["Hkv"]
        d["q"], d["go"] = _bf(g, B, S, Hq, 128), _bf(g, B, S, Hq * 128)
        d["k"], d["v"] = _bf(g, B, S, Hkv, 128), _bf(g, B, S, Hkv, 128)
        return d
    d["hs"] = _bf(g, case["B"], case["S"], case["hidden"])
    return d


def _leaf(t):
    return t.detach().requires_grad_(True)


class _Shape:
    """What PalettizedLinear reads of the linear that it replaces."""

    def __init__(self, K, N, bias):
        self.in_features, self.out_features = K, N
        self.bias = None if bias is None else torch.nn.Parameter(bias, requires_grad=False)


def prepare(case, seed):
    d = _inputs(case, seed)
    kind = case["kind"]
    if kind == "decode":
        if case["stage"]:
            groups = [[(l, i) for l in range(case["layers"]) for i in range(7)]]
        else:
            groups = [[(0, i) for i in grp] for grp in DECODE_GROUPS]
        return kind, [ops.GemvGroup([(d["x"][l][i], *d["weights"][l][i]) for l, i in grp])
                      for grp in groups]
    if kind == "prefill":
        return kind, d["x"][0], d["weights"][0], d["lora"]
    if kind in ("hard", "soft"):
        for n in ("x", "pal", "a", "b", "bias", "logits"):
            if d.get(n) is not None:
                d[n] = _leaf(d[n])
        return kind, d, case.get("tau")
    if kind in ("dropin_hard", "dropin_soft"):
        soft = kind == "dropin_soft"
        base = PalettizedLinear(_Shape(case["K"], case["N"], d["bias"]), d["idx"],
                                d["pal"].shape[0], 4, 256, False, initial_palette=d["pal"],
                                use_soft_indices=soft)
        mod = QwenLoRA(base, rank=case["rank"], alpha=64, init="random").cuda().train()
        with torch.no_grad():
            mod.lora_A.copy_(d["a"])
            mod.lora_B.copy_(d["b"])
            if soft:
                base.index_logits.copy_(d["logits"])
                base.tau = case["tau"]
                # the noise follows a counter of forwards, which a resumed run sets
                FL._SOFT_STEP_SEED = _step_seed(seed)
        return kind, mod, _leaf(d["x"]), d["gy"]
    if kind == "attention":
        return kind, _leaf(d["q"]), _leaf(d["k"]), _leaf(d["v"]), d["go"]
    cfg = LayerConfig(hidden=case["hidden"], heads=case["heads"], kv_heads=case["kv_heads"],
                      intermediate=case["intermediate"])
    trainer = LayerTrainer(cfg, torch.device("cuda"), seed=int(seed) % 1000, lora_b_std=0.01)
    return kind, trainer, d["hs"]


def _step_seed(seed):
    return 1000 + int(seed) % 100000


# ---- one pass -----------------------------------------------------------------------------------
def run(state):
    kind = state[0]
    if kind == "decode":
        return [y for grp in state[1] for y in grp.run()]
    if kind == "prefill":
        _, xs, weights, lora = state
        with torch.no_grad():
            return [lut_linear(x, packed, pal, None, a, b, 1.0)
                    for x, (packed, pal), (a, b) in zip(xs, weights, lora)]
    if kind == "hard":
        d = state[1]
        y = lut_linear(d["x"], d["packed"], d["pal"], d["bias"], d["a"], d["b"], 1.0)
        wrt = [d[n] for n in ("x", "pal", "a", "b", "bias") if d[n] is not None]
        return [y, *torch.autograd.grad(y, wrt, d["gy"])]
    if kind == "soft":
        d = state[1]
        y = soft_lut_linear(d["x"], d["pal"], d["logits"], d["noise"], state[2], None, d["a"],
                            d["b"], 1.0)
        return [y, *torch.autograd.grad(y, [d[n] for n in ("x", "pal", "logits", "a", "b")],
                                        d["gy"])]
    if kind in ("dropin_hard", "dropin_soft"):
        _, mod, x, gy = state
        y = mod(x)
        wrt = [x, mod.base.palette, mod.lora_A, mod.lora_B]
        if kind == "dropin_soft":
            wrt.append(mod.base.index_logits)
        return [y, *torch.autograd.grad(y, wrt, gy)]
    if kind == "attention":
        _, q, k, v, go = state
        o = attention(q, k, v, q.shape[2], k.shape[2])
        return [o, *torch.autograd.grad(o, (q, k, v), go)]
    _, trainer, hs = state
    loss, l_cos = trainer.step(hs)
    params = trainer.logits + trainer.others
    return [loss, l_cos] + [p.grad for p in params] + [p.detach() for p in params]


# ---- work and tolerance -------------------------------------------------------------------------
def work(case):
    kind = case["kind"]
    if kind in ("decode", "prefill"):
        M, layers, linears = case["M"], case.get("layers", 1), LINEARS[case["hidden"]]
        nbytes = flops = 0
        for K, N, r in linears:
            nbytes += N * K // 4 + N * (K // 256) * 16 + 2 * M * N
            flops += 2 * M * N * K
            if kind == "prefill":
                nbytes += 2 * r * (K + N)
                flops += 2 * M * r * (K + N)
        nbytes += sum(2 * M * linears[grp[0]][0] for grp in DECODE_GROUPS)
        return {"bytes": layers * nbytes, "flops": layers * flops}
    if kind == "attention":
        B, S, Hq, Hkv = case["B"], case["S"], case["Hq"], case["Hkv"]
        # q, grad_o read, o, grad_q written; k, v read, grad_k, grad_v written; half of S x S
        return {"bytes": 2 * B * S * 128 * (4 * Hq + 4 * Hkv),
                "flops": 7 * B * Hq * S * S * 128}
    if kind == "layer":
        B, S, h, f, r = case["B"], case["S"], case["hidden"], case["intermediate"], 16
        M, q, kv = B * S, case["heads"] * 128, case["kv_heads"] * 128
        lin = ((h, q), (h, kv), (h, kv), (q, h), (h, f), (h, f), (f, h))
        # student forward, grad_x (not of q, k, v) and dW; teacher forward; LoRA; attention of
        # the student (forward and backward) and the teacher
        flops = sum(8 * M * k * n + 6 * M * r * (k + n) for k, n in lin)
        flops -= sum(2 * M * k * n for k, n in lin[:3])
        flops += 9 * B * case["heads"] * S * S * 128
        weights = sum(k * n for k, n in lin)
        # logits, masters and moments read and written, gradients written, teacher weights, hs
        return {"bytes": weights * (4 * (2 + 2 + 12 + 12 + 2) + 2) + 2 * M * h, "flops": flops}
    K, N, r = case["K"], case["N"], case["rank"]
    M = case["M"] if "M" in case else case["B"] * case["S"]
    # x, gy read, y, gx written; LoRA factors read, their gradients written
    nbytes = 4 * M * (K + N) + 4 * r * (K + N)
    if kind == "hard":
        nbytes += N * K // 4 + 2 * 16 * N * (K // 256)
    elif kind == "soft":
        nbytes += N * K * (8 + 16 + 8) + 2 * 16 * N * (K // 256)
    elif kind == "dropin_hard":
        nbytes += N * K  # int8 indices
    else:
        nbytes += N * K * 16  # fp16 logits and their gradient
    return {"bytes": nbytes, "flops": 6 * M * K * N + 6 * M * r * (K + N)}


def tolerance(case):
    # bf16 outputs of fp32 sums, LoRA intermediates and attention probabilities rounded to bf16:
    # 1.7e-3 to 2.5e-3 from exact()
    return {"rel": 1e-2}


# ---- the same in 64 bits ------------------------------------------------------------------------
def _unpack(packed):
    s = torch.arange(0, 32, 2, device=packed.device, dtype=torch.int32)
    return ((packed[:, :, None] >> s) & 3).reshape(packed.shape[0], -1).long()


def _class_sums(dw, idx, N, K):
    """[N, K/256, 4]: dw summed per group and class."""
    out = torch.zeros(N, K // 256, 4, dtype=torch.float64, device=dw.device)
    return out.scatter_add_(2, idx.view(N, K // 256, 256), dw.view(N, K // 256, 256))


def _dequant(packed, pal):
    N, G = pal.shape[:2]
    return torch.gather(pal.to(torch.bfloat16).double(), 2,
                        _unpack(packed).view(N, G, 256)).view(N, G * 256)


def _lcg_gumbel(seed, K, N):
    """The original sampler's noise for (4, K, N) planes: a 32-bit hash of (k N + n) 4 + c, with
    u = its low 24 bits / 2^24 and -log(-log(max(u, 1e-7)))."""
    m = 0xFFFFFFFF
    x = torch.arange(K * N * 4, device="cuda", dtype=torch.int64)
    x = (x * 0x9E3779B9 & m) ^ (seed & m)
    x = x ^ (x >> 13)
    x = x * 1103515245 + 12345 & m
    x = x ^ (x >> 17)
    x = x * 1103515245 + 12345 & m
    u = ((x & 0xFFFFFF).double() / 2 ** 24).clamp_(min=1e-7)
    return (-torch.log(-torch.log(u))).view(K, N, 4).permute(2, 0, 1)


def _attention64(q, k, v, go):
    """One batch entry: q [S, Hq, D], k, v [S, Hkv, D], go [S, Hq, D] -> o, dq, dk, dv."""
    S, Hq, D = q.shape
    rep = Hq // k.shape[1]
    mask = torch.ones(S, S, dtype=torch.bool, device=q.device).triu(1)
    outs = [torch.empty_like(q), torch.empty_like(q), torch.zeros_like(k), torch.zeros_like(v)]
    for h in range(Hq):
        qh, kh, vh, gh = q[:, h], k[:, h // rep], v[:, h // rep], go[:, h]
        p = torch.softmax((qh @ kh.T * D ** -0.5).masked_fill_(mask, -math.inf), -1)
        o = p @ vh
        dp = gh @ vh.T
        ds = p * (dp - (gh * o).sum(-1, keepdim=True)) * D ** -0.5
        outs[0][:, h], outs[1][:, h] = o, ds @ kh
        outs[2][:, h // rep] += ds.T @ qh
        outs[3][:, h // rep] += p.T @ gh
    return outs


def exact(case, seed):
    kind = case["kind"]
    if kind == "layer":
        # the step draws its noise inside the library and rounds between its parts, each of
        # which has a case of its own here
        return None
    d = _inputs(case, seed)
    if kind == "decode":
        # the order of run(): layer after layer, and the groups within a layer
        return [d["x"][l][i].double() @ _dequant(*d["weights"][l][i]).T
                for l in range(case["layers"]) for i in range(7)]
    if kind == "prefill":
        return [x.double() @ _dequant(*w).T + (x.double() @ a.double().T) @ b.double().T
                for x, w, (a, b) in zip(d["x"][0], d["weights"][0], d["lora"])]
    if kind == "attention":
        B, S = case["B"], case["S"]
        got = [_attention64(*(d[n][i].double().view(S, -1, 128) for n in ("q", "k", "v", "go")))
               for i in range(B)]
        o, dq, dk, dv = (torch.stack(t) for t in zip(*got))
        return [o.reshape(B, S, -1), dq, dk, dv]
    x, gy = (d[n].double().view(-1, d[n].shape[-1]) for n in ("x", "gy"))
    a, b = d["a"].double(), d["b"].double()
    scale = 1.0
    if kind in ("dropin_hard", "dropin_soft"):
        a, scale = a.T, 64.0 / case["rank"]
    (M, K), N = x.shape, gy.shape[1]
    dw = gy.T @ x
    grad_logits = None
    if kind == "hard":
        w = _dequant(d["packed"], d["pal"])
        grad_pal = _class_sums(dw, _unpack(d["packed"]), N, K)
    elif kind == "soft":
        pal = d["pal"].double()[:, :, None, :].expand(N, K // 256, 256, 4).reshape(N, K, 4)
        p = torch.softmax((d["logits"].double() + d["noise"].double()) / case["tau"], -1)
        w = torch.gather(pal, 2, p.argmax(-1, keepdim=True))[..., 0].to(torch.bfloat16).double()
        grad_logits = dw[..., None] * p * (pal - (p * pal).sum(-1, keepdim=True))
        grad_pal = (dw[..., None] * p).view(N, K // 256, 256, 4).sum(2)
    else:
        pal = d["pal"].double().repeat_interleave(256, 0)[:N]  # [N, 4]
        if kind == "dropin_hard":
            w = torch.gather(pal, 1, d["idx"].T)
            per_row = torch.zeros(N, 4, dtype=torch.float64, device="cuda")
            per_row.scatter_add_(1, d["idx"].T, dw)
        else:
            p = (d["logits"].double() + _lcg_gumbel(_step_seed(seed) + 1, K, N)) / case["tau"]
            p = torch.softmax(p, 0).permute(2, 1, 0)  # [N, K, 4]
            w = torch.gather(pal, 1, p.argmax(-1))
            soft = (p * pal[:, None]).sum(-1, keepdim=True)
            grad_logits = (dw[..., None] * p * (pal[:, None] - soft)).permute(2, 1, 0)
            per_row = (dw[..., None] * p).sum(1)
        grad_pal = torch.zeros(d["pal"].shape, dtype=torch.float64, device="cuda")
        grad_pal.index_add_(0, torch.arange(N, device="cuda") // 256, per_row)
    y = x @ w.T + scale * (x @ a.T) @ b.T
    gb = gy @ b
    grad_x = gy @ w + scale * gb @ a
    grad_a, grad_b = scale * gb.T @ x, scale * gy.T @ (x @ a.T)
    if d.get("bias") is not None:
        y = y + d["bias"].double()
    if kind == "hard":
        out = [y, grad_x, grad_pal, grad_a, grad_b]
        return out + ([gy.sum(0)] if d["bias"] is not None else [])
    if kind == "soft":
        return [y, grad_x, grad_pal, grad_logits, grad_a, grad_b]
    lead = d["x"].shape[:-1]
    out = [y.view(*lead, N), grad_x.view(*lead, K), grad_pal, grad_a.T, grad_b]
    return out + ([grad_logits] if kind == "dropin_soft" else [])
