"""Timed cases of the library: attention, linear layers, the VAE mid-block and the weight decode,
through the Python binding of the C ABI on torch device buffers.

Sizes come from the models whose layers these are (DiT: 14 blocks of 9 heads x 64 over 256 tokens,
width 576, MLP 2304; T5 encoder: 12 layers of 12 heads x 64; VAE mid-block: one head over 512
channels), at the batches the benchmark and the tests use, and ragged ones between them. Values are
those of the repository's workloads: activations ~ N(0, 1), weights ~ N(0, 1/K), biases ~ N(0, 0.1^2).
"""

import math
import os
import sys

import numpy as np
import torch
import torch.nn.functional as F

sys.path.insert(0, os.path.join(os.getcwd(), "supra2-img-web_amd"))

from supra_attn import AttnArgs, LinearArgs, _lib, attention, bucket_lut, linear, load, workspace_bytes  # noqa: E402

TOKENS, DIM, MLP, HEADS, HEAD_DIM, BLOCKS = 256, 576, 2304, 9, 64, 14
T5_HEADS, T5_LAYERS, T5_BUCKETS, T5_DISTANCE = 12, 12, 32, 128

# One layer's weights of the DiT checkpoint, repeated per block by the decode case
BLOCK_WEIGHTS = [(3 * DIM, DIM), (3 * DIM,), (DIM, DIM), (DIM,), (DIM, DIM), (DIM,), (2 * DIM, DIM), (2 * DIM,),
                 (DIM, DIM), (DIM,), (MLP, DIM), (MLP,), (DIM, MLP), (DIM,), (6 * DIM, DIM), (6 * DIM,)]


def listed():
    return [
        # a prompt through the T5 encoder: each layer's self-attention, 128 tokens of which 40 are padding
        dict(name="t5_prompt", kind="t5", B=1, L=128, pad=40, layers=T5_LAYERS, bias="relpos"),
        # a batch of ragged prompts with the dense position bias the JS encoder passes
        dict(name="t5_dense_ragged", kind="t5", B=3, L=333, pad=55, layers=1, bias="dense"),
        # one image with guidance: a denoising step's attention, 14 blocks of self then cross, the
        # prompt at 77 tokens and the empty one at 1
        dict(name="dit_step_b2", kind="dit_step", B=2, keys="guided", layers=BLOCKS),
        # a few images at once: batched self-attention at a batch that fills no whole round
        dict(name="dit_self_b13", kind="dit_self", B=13, layers=1),
        # the throughput batch: self-attention of one block
        dict(name="dit_self_b64", kind="dit_self", B=64, layers=1),
        # and cross-attention, prompts of 1 to 128 tokens
        dict(name="dit_cross_b64", kind="dit_cross", B=64, keys="uniform", layers=1),
        # the operator's other fused head dim, ragged lengths on both sides
        dict(name="attn_d128", kind="attn", B=4, H=8, D=128, Lq=1000, Lk=777, bias="none"),
        # the VAE mid-block of a 256 x 256 image (32 x 32 latent), and of a 512 x 512 one
        dict(name="vae_block_32", kind="vae", HW=1024),
        dict(name="vae_block_64", kind="vae", HW=4096),
        # the linear layers of one DiT block (qkv, proj, q, cproj, fc1, fc2): one image with guidance,
        # and the throughput batch
        dict(name="dit_linears_b2", kind="linears", B=2),
        dict(name="dit_linears_b64", kind="linears", B=64),
        # a model load: every tensor of a bfloat16 DiT checkpoint decoded to float32
        dict(name="decode_bf16", kind="decode", dtype="BF16", blocks=BLOCKS),
    ]


def _log(rng, lo, hi):
    return min(hi, max(lo, round(math.exp(rng.uniform(math.log(lo), math.log(hi + 0.5))))))


def draw(rng):
    kind = rng.choice(["t5", "dit_step", "dit_self", "dit_cross", "attn", "vae", "linear", "linears", "decode"])
    if kind == "t5":
        L = _log(rng, 8, 512)
        return dict(kind=kind, B=rng.randint(1, 4), L=L, pad=rng.randint(0, L // 2), layers=rng.choice([1, T5_LAYERS]),
                    bias=rng.choice(["relpos", "dense"]))
    if kind == "dit_step":
        return dict(kind=kind, B=rng.randint(1, 8), keys="uniform", layers=rng.randint(1, 4))
    if kind == "dit_self":
        return dict(kind=kind, B=_log(rng, 1, 64), layers=1)
    if kind == "dit_cross":
        return dict(kind=kind, B=_log(rng, 1, 64), keys=rng.choice(["uniform", "full"]), layers=1)
    if kind == "attn":
        return dict(kind=kind, B=rng.randint(1, 4), H=rng.randint(1, 12), D=rng.choice([64, 128]), Lq=_log(rng, 1, 1024),
                    Lk=_log(rng, 1, 1024), bias=rng.choice(["none", "dense"]))
    if kind == "vae":
        return dict(kind=kind, HW=_log(rng, 16, 64) * _log(rng, 16, 64))
    if kind == "linear":
        N, K = rng.choice([(3 * DIM, DIM), (2 * DIM, DIM), (DIM, DIM), (MLP, DIM), (DIM, MLP), (768, 768), (2048, 768), (1536, 512)])
        return dict(kind=kind, M=_log(rng, 1, 16384), N=N, K=K, act=rng.choice(["none", "gelu", "gelu_tanh", "silu"]))
    if kind == "linears":
        return dict(kind=kind, B=_log(rng, 1, 63))
    return dict(kind=kind, dtype=rng.choice(["BF16", "F16", "F32"]), blocks=rng.randint(1, BLOCKS))


# ---- inputs, made from the seed alone

def _rng(seed):
    return torch.Generator(device="cuda").manual_seed(int(seed))


def _normal(g, *shape, std=1.0):
    return torch.randn(*shape, generator=g, device="cuda", dtype=torch.float32) * std


def _key_lengths(case, seed):
    B = case["B"]
    if case["keys"] == "guided":
        return np.array([77, 1] * ((B + 1) // 2), dtype=np.int32)[:B].copy()
    if case["keys"] == "full":
        return np.full(B, 77, dtype=np.int32)
    return np.random.default_rng([int(seed), 999]).integers(1, 129, size=B, dtype=np.int32)


def _self_inputs(case, g):
    return [_normal(g, case["B"] * TOKENS, 3 * DIM) for _ in range(case["layers"])]


def _cross_inputs(case, g, lens):
    Lk = int(lens.max())
    return [(_normal(g, case["B"] * TOKENS, DIM), _normal(g, case["B"] * Lk, 2 * DIM)) for _ in range(case["layers"])]


def _t5_inputs(case, g):
    B, L, C = case["B"], case["L"], T5_HEADS * HEAD_DIM
    qkv = [tuple(_normal(g, B * L, C) for _ in range(3)) for _ in range(case["layers"])]
    table = _normal(g, T5_BUCKETS, T5_HEADS, std=0.5)
    lut = torch.from_numpy(bucket_lut(L, L, T5_BUCKETS, T5_DISTANCE, True)).cuda()
    mask = torch.ones(B, L, dtype=torch.uint8, device="cuda")
    for b in range(B):  # the first prompt has all the padding, the others less
        mask[b, L - case["pad"] // (b + 1):] = 0
    return qkv, table, lut, mask


def _dense_bias(table, lut, L):
    i = torch.arange(L, device="cuda")
    return table[lut.long()[i[None, :] - i[:, None] + L - 1]].permute(2, 0, 1).contiguous()  # [H, L, L]


def _attn_inputs(case, g):
    B, H, D, Lq, Lk = (case[k] for k in ("B", "H", "D", "Lq", "Lk"))
    q, k, v = _normal(g, B * Lq, H * D), _normal(g, B * Lk, H * D), _normal(g, B * Lk, H * D)
    return q, k, v, _normal(g, H, Lq, Lk) if case["bias"] == "dense" else None


def _vae_inputs(case, g):
    HW, C = case["HW"], 512
    return dict(x=_normal(g, HW, C), gamma=1 + _normal(g, C, std=0.1), beta=_normal(g, C, std=0.1),
                wqkv=_normal(g, 3 * C, C, std=C ** -0.5), bqkv=_normal(g, 3 * C, std=0.1),
                wo=_normal(g, C, C, std=C ** -0.5), bo=_normal(g, C, std=0.1))


LAYERS = {  # name: (N, K, act, epilogue)
    "qkv": (3 * DIM, DIM, _lib.SA_ACT_NONE, _lib.SA_EPI_STORE),
    "proj": (DIM, DIM, _lib.SA_ACT_NONE, _lib.SA_EPI_RESID_GATE),
    "q": (DIM, DIM, _lib.SA_ACT_NONE, _lib.SA_EPI_STORE),
    "cproj": (DIM, DIM, _lib.SA_ACT_NONE, _lib.SA_EPI_RESID),
    "fc1": (MLP, DIM, _lib.SA_ACT_GELU_TANH, _lib.SA_EPI_STORE),
    "fc2": (DIM, MLP, _lib.SA_ACT_NONE, _lib.SA_EPI_RESID_GATE),
}
ACTS = {"none": _lib.SA_ACT_NONE, "gelu": _lib.SA_ACT_GELU, "gelu_tanh": _lib.SA_ACT_GELU_TANH, "silu": _lib.SA_ACT_SILU}


def _linears_inputs(case, g):
    R = case["B"] * TOKENS
    w = {n: (_normal(g, N, K, std=K ** -0.5), _normal(g, N, std=0.1)) for n, (N, K, _, _) in LAYERS.items()}
    h, a, h2, c, h3 = (_normal(g, R, DIM) for _ in range(5))
    return w, dict(qkv=h, proj=a, q=h2, cproj=c, fc1=h3), _normal(g, R, DIM), _normal(g, 6 * DIM)


def _linear_inputs(case, g):
    return _normal(g, case["M"], case["K"]), _normal(g, case["N"], case["K"], std=case["K"] ** -0.5), _normal(g, case["N"], std=0.1)


def _decode_inputs(case, g):
    shapes = BLOCK_WEIGHTS * case["blocks"]
    kind = {"BF16": torch.bfloat16, "F16": torch.float16, "F32": torch.float32}[case["dtype"]]
    return shapes, _normal(g, sum(math.prod(s) for s in shapes), std=0.05).to(kind)


# ---- what a program has in hand before the call

def _attn_call(hold, q, k, v, o, *, scale, B, H, D, Lq, Lk, **kw):
    args = AttnArgs(B=B, H=H, D=D, Lq=Lq, Lk=Lk, q=q.data_ptr(), k=k.data_ptr(), v=v.data_ptr(), o=o.data_ptr(),
                    ldo=H * D, so=Lq * H * D, scale=scale, **kw)
    need = workspace_bytes(args)
    if need > 0:
        ws = torch.empty(need, dtype=torch.uint8, device="cuda")
        hold.append(ws)
        args.workspace, args.workspace_bytes = ws.data_ptr(), need
    hold += [q, k, v, o]
    return args


def _self_calls(case, hold, inputs):
    calls, outs = [], []
    for qkv in inputs:
        o = torch.empty(case["B"] * TOKENS, DIM, device="cuda")
        s = TOKENS * 3 * DIM
        calls.append(_attn_call(hold, qkv, qkv, qkv, o, scale=HEAD_DIM ** -0.5, B=case["B"], H=HEADS, D=HEAD_DIM, Lq=TOKENS,
                                Lk=TOKENS, k_off=DIM, v_off=2 * DIM, ldq=3 * DIM, ldk=3 * DIM, ldv=3 * DIM, sq=s, sk=s, sv=s))
        outs.append(o)
    return calls, outs


def _cross_calls(case, hold, inputs, lens):
    calls, outs = [], []
    Lk = int(lens.max())
    dev_lens = torch.from_numpy(lens).cuda()
    hold += [lens, dev_lens]
    for q, kv in inputs:
        o = torch.empty(case["B"] * TOKENS, DIM, device="cuda")
        calls.append(_attn_call(hold, q, kv, kv, o, scale=HEAD_DIM ** -0.5, B=case["B"], H=HEADS, D=HEAD_DIM, Lq=TOKENS, Lk=Lk,
                                v_off=DIM, ldq=DIM, ldk=2 * DIM, ldv=2 * DIM, sq=TOKENS * DIM, sk=Lk * 2 * DIM, sv=Lk * 2 * DIM,
                                mask_mode=_lib.SA_MASK_KEY_LEN, key_len=dev_lens.data_ptr(), key_len_host=lens.ctypes.data))
        outs.append(o)
    return calls, outs


def _linear_call(hold, x, w, b, y, N, K, act, epi, gate=None, gate_off=0):
    hold += [x, w, b, y, gate]
    return LinearArgs(M=x.shape[0], N=N, K=K, x=x.data_ptr(), w=w.data_ptr(), bias=b.data_ptr(), act=act, epilogue=epi,
                      y=y.data_ptr(), gate=gate.data_ptr() if gate is not None else None, gate_off=gate_off)


def prepare(case, seed):
    kind, g, hold = case["kind"], _rng(seed), []
    state = dict(kind=kind, hold=hold)
    if kind == "dit_self":
        state["calls"], state["outs"] = _self_calls(case, hold, _self_inputs(case, g))
    elif kind == "dit_cross":
        lens = _key_lengths(case, seed)
        state["calls"], state["outs"] = _cross_calls(case, hold, _cross_inputs(case, g, lens), lens)
    elif kind == "dit_step":
        lens = _key_lengths(case, seed)
        sc, so = _self_calls(case, hold, _self_inputs(case, g))
        cc, co = _cross_calls(case, hold, _cross_inputs(case, g, lens), lens)
        state["calls"] = [c for pair in zip(sc, cc) for c in pair]
        state["outs"] = [o for pair in zip(so, co) for o in pair]
    elif kind == "t5":
        B, L, C = case["B"], case["L"], T5_HEADS * HEAD_DIM
        qkv, table, lut, mask = _t5_inputs(case, g)
        hold += [table, lut, mask]
        if case["bias"] == "dense":
            bias = _dense_bias(table, lut, L)
            hold.append(bias)
            kw = dict(bias_mode=_lib.SA_BIAS_DENSE, bias=bias.data_ptr())
        else:
            kw = dict(bias_mode=_lib.SA_BIAS_RELPOS, bias=table.data_ptr(), bucket_lut=lut.data_ptr(), num_buckets=T5_BUCKETS)
        outs = [torch.empty(B * L, C, device="cuda") for _ in qkv]
        state["calls"] = [_attn_call(hold, q, k, v, o, scale=1.0, B=B, H=T5_HEADS, D=HEAD_DIM, Lq=L, Lk=L, ldq=C, ldk=C, ldv=C,
                                     sq=L * C, sk=L * C, sv=L * C, mask_mode=_lib.SA_MASK_KEY_MASK, key_mask=mask.data_ptr(), smask=L, **kw)
                          for (q, k, v), o in zip(qkv, outs)]
        state["outs"] = outs
    elif kind == "attn":
        B, H, D, Lq, Lk = (case[k] for k in ("B", "H", "D", "Lq", "Lk"))
        q, k, v, bias = _attn_inputs(case, g)
        o = torch.empty(B * Lq, H * D, device="cuda")
        kw = {}
        if bias is not None:
            hold.append(bias)
            kw = dict(bias_mode=_lib.SA_BIAS_DENSE, bias=bias.data_ptr())
        state["calls"] = [_attn_call(hold, q, k, v, o, scale=D ** -0.5, B=B, H=H, D=D, Lq=Lq, Lk=Lk, ldq=H * D, ldk=H * D, ldv=H * D,
                                     sq=Lq * H * D, sk=Lk * H * D, sv=Lk * H * D, **kw)]
        state["outs"] = [o]
    elif kind == "vae":
        t = _vae_inputs(case, g)
        out = torch.empty_like(t["x"])
        args = _lib.VaeAttnArgs(HW=case["HW"], C=512, out=out.data_ptr(), **{k: v.data_ptr() for k, v in t.items()})
        need = _lib.vae_workspace_bytes(args)
        ws = torch.empty(need, dtype=torch.uint8, device="cuda")
        args.workspace, args.workspace_bytes = ws.data_ptr(), need
        hold += [t, ws]
        state["args"], state["outs"] = args, out
    elif kind == "linears":
        w, x, resid, gates = _linears_inputs(case, g)
        R = resid.shape[0]
        stream = torch.empty_like(resid)  # the residual stream that proj, cproj and fc2 add to
        y = {n: torch.empty(R, LAYERS[n][0], device="cuda") for n in ("qkv", "q", "fc1")}
        x["fc2"] = y["fc1"]
        gate_off = dict(proj=2 * DIM, fc2=5 * DIM)
        state["calls"] = [_linear_call(hold, x[n], *w[n], y.get(n, stream), N, K, act, epi,
                                       gates if n in gate_off else None, gate_off.get(n, 0)) for n, (N, K, act, epi) in LAYERS.items()]
        state["resid"], state["stream"], state["outs"] = resid, stream, [y["qkv"], y["q"], y["fc1"], stream]
    elif kind == "linear":
        x, w, b = _linear_inputs(case, g)
        y = torch.empty(case["M"], case["N"], device="cuda")
        state["calls"] = [_linear_call(hold, x, w, b, y, case["N"], case["K"], ACTS[case["act"]], _lib.SA_EPI_STORE)]
        state["outs"] = y
    else:
        shapes, blob = _decode_inputs(case, g)
        dtype, size, at, calls, outs = _lib.SA_DT[case["dtype"]], blob.element_size(), 0, [], []
        arena = torch.empty(blob.numel(), device="cuda")
        for s in shapes:
            n = math.prod(s)
            calls.append((blob.data_ptr() + at * size, dtype, n, arena.data_ptr() + 4 * at))
            at += n
        hold.append(blob)
        state["calls"], state["outs"] = calls, arena
    return state


def run(state):
    stream = torch.cuda.current_stream().cuda_stream
    kind = state["kind"]
    if kind == "vae":
        _lib.vae_attention(state["args"], stream)
    elif kind in ("linears", "linear"):
        if kind == "linears":
            state["stream"].copy_(state["resid"])
        for c in state["calls"]:
            linear(c, stream)
    elif kind == "decode":
        to_f32 = load().sa_to_f32
        for src, dtype, n, dst in state["calls"]:
            _lib.check(to_f32(src, dtype, n, dst, stream))
    else:
        for c in state["calls"]:
            attention(c, stream)
    return state["outs"]


# ---- the work a pass cannot do without

def _attn_work(B, H, D, Lq, keys, extra=0):
    """keys: the attended keys of all sequences together."""
    return {"bytes": 4 * (2 * B * Lq * H * D + 2 * keys * H * D) + extra, "flops": 4 * D * H * Lq * keys}


def _plus(*works):
    return {k: sum(w[k] for w in works) for k in ("bytes", "flops")}


def _linear_work(M, N, K, resid=False):
    return {"bytes": 4 * (M * K + N * K + N + M * N * (2 if resid else 1)), "flops": 2 * M * N * K}


def work(case):
    kind = case["kind"]
    if kind in ("dit_self", "dit_cross", "dit_step"):
        B = case["B"]
        one = {"bytes": 0, "flops": 0}
        if kind != "dit_cross":
            one = _plus(one, _attn_work(B, HEADS, HEAD_DIM, TOKENS, B * TOKENS))
        if kind != "dit_self":
            keys = {"guided": 77 * ((B + 1) // 2) + B // 2, "full": 77 * B}.get(case["keys"], 64.5 * B)
            one = _plus(one, _attn_work(B, HEADS, HEAD_DIM, TOKENS, keys))
        return {k: v * case["layers"] for k, v in one.items()}
    if kind == "t5":
        B, L = case["B"], case["L"]
        keys = sum(L - case["pad"] // (b + 1) for b in range(B))
        bias = 4 * T5_HEADS * L * L if case["bias"] == "dense" else 4 * T5_BUCKETS * T5_HEADS + 8 * L
        one = _attn_work(B, T5_HEADS, HEAD_DIM, L, keys, bias + B * L)
        return {k: v * case["layers"] for k, v in one.items()}
    if kind == "attn":
        bias = 4 * case["H"] * case["Lq"] * case["Lk"] if case["bias"] == "dense" else 0
        return _attn_work(case["B"], case["H"], case["D"], case["Lq"], case["B"] * case["Lk"], bias)
    if kind == "vae":
        HW, C = case["HW"], 512
        return {"bytes": 4 * (2 * HW * C + 4 * C * C + 6 * C), "flops": 8 * HW * C * C + 4 * C * HW * HW}
    if kind == "linears":
        R = case["B"] * TOKENS
        return _plus(*(_linear_work(R, N, K, epi != _lib.SA_EPI_STORE) for N, K, _, epi in LAYERS.values()))
    if kind == "linear":
        return _linear_work(case["M"], case["N"], case["K"])
    n = sum(math.prod(s) for s in BLOCK_WEIGHTS) * case["blocks"]
    return {"bytes": n * (4 + (4 if case["dtype"] == "F32" else 2)), "flops": 0}


def tolerance(case):
    # About four times the distance from 64 bits: float32 sums, and for the T5 encoder unscaled
    # logits (standard deviation 8), whose rounding the exponential passes on.
    if case["kind"] == "decode":
        return "exact"
    if case["kind"] == "t5":
        return {"rel": 4e-6, "max": 2e-4}
    return {"rel": 1e-6 if case["kind"] == "vae" else 2e-6, "max": 8e-5}


# ---- the same in 64 bits

def _attn64(q, k, v, scale, bias=None, keep=None):
    """q [B, H, Lq, D], k and v [B, H, Lk, D]; keep [B, Lk] (attended keys)."""
    s = (q.double() * scale) @ k.double().transpose(-1, -2).contiguous()
    if bias is not None:
        s = s + bias.double()
    if keep is not None:
        s = s.masked_fill(~keep[:, None, None, :], -math.inf)
    return torch.softmax(s, dim=-1) @ v.double()


def _heads(x, B, L, H, D):
    return x.reshape(B, L, H, D).transpose(1, 2)


def _rows(o):
    B, H, L, D = o.shape
    return o.transpose(1, 2).reshape(B * L, H * D)


def _self64(case, inputs):
    B = case["B"]
    return [_rows(_attn64(*(_heads(x, B, TOKENS, HEADS, HEAD_DIM) for x in qkv.split(DIM, dim=1)), HEAD_DIM ** -0.5)) for qkv in inputs]


def _cross64(case, inputs, lens):
    B, Lk = case["B"], int(lens.max())
    keep = torch.arange(Lk, device="cuda")[None, :] < torch.from_numpy(lens).cuda()[:, None]
    res = []
    for q, kv in inputs:
        k, v = kv.split(DIM, dim=1)
        res.append(_rows(_attn64(_heads(q, B, TOKENS, HEADS, HEAD_DIM), _heads(k, B, Lk, HEADS, HEAD_DIM),
                                 _heads(v, B, Lk, HEADS, HEAD_DIM), HEAD_DIM ** -0.5, keep=keep)))
    return res


def exact(case, seed):
    kind, g = case["kind"], _rng(seed)
    if kind == "dit_self":
        return _self64(case, _self_inputs(case, g))
    if kind in ("dit_cross", "dit_step"):
        lens = _key_lengths(case, seed)
        if kind == "dit_cross":
            return _cross64(case, _cross_inputs(case, g, lens), lens)
        so = _self64(case, _self_inputs(case, g))
        co = _cross64(case, _cross_inputs(case, g, lens), lens)
        return [o for pair in zip(so, co) for o in pair]
    if kind == "t5":
        B, L = case["B"], case["L"]
        qkv, table, lut, mask = _t5_inputs(case, g)
        bias = _dense_bias(table, lut, L)
        return [_rows(_attn64(*(_heads(x, B, L, T5_HEADS, HEAD_DIM) for x in t), 1.0, bias, mask != 0)) for t in qkv]
    if kind == "attn":
        B, H, D, Lq, Lk = (case[k] for k in ("B", "H", "D", "Lq", "Lk"))
        q, k, v, bias = _attn_inputs(case, g)
        return [_rows(_attn64(_heads(q, B, Lq, H, D), _heads(k, B, Lk, H, D), _heads(v, B, Lk, H, D), D ** -0.5, bias))]
    if kind == "vae":
        t = {k: v.double() for k, v in _vae_inputs(case, g).items()}
        n = F.group_norm(t["x"].t()[None], 32, t["gamma"], t["beta"], 1e-6)[0].t().contiguous()
        q, k, v = (F.linear(n, t["wqkv"], t["bqkv"])).split(512, dim=1)
        a = torch.softmax(q @ k.t().contiguous() * 512 ** -0.5, dim=-1) @ v
        return t["x"] + F.linear(a, t["wo"], t["bo"])
    act64 = {_lib.SA_ACT_NONE: lambda r: r, _lib.SA_ACT_GELU: F.gelu, _lib.SA_ACT_SILU: F.silu,
             _lib.SA_ACT_GELU_TANH: lambda r: F.gelu(r, approximate="tanh")}
    if kind == "linears":
        w, x, resid, gates = _linears_inputs(case, g)
        r = {}
        for n, (N, K, act, _) in LAYERS.items():
            src = r["fc1"] if n == "fc2" else x[n].double()
            r[n] = act64[act](F.linear(src, w[n][0].double(), w[n][1].double()))
        gd = gates.double()
        stream = resid.double() + gd[2 * DIM:3 * DIM] * r["proj"] + r["cproj"] + gd[5 * DIM:] * r["fc2"]
        return [r["qkv"], r["q"], r["fc1"], stream]
    if kind == "linear":
        x, w, b = _linear_inputs(case, g)
        return act64[ACTS[case["act"]]](F.linear(x.double(), w.double(), b.double()))
    _, blob = _decode_inputs(case, g)
    return blob.double()
