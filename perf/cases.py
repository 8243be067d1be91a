"""Performance cases of the library: the calls a program that runs a qwen35moe-shaped
model on it makes, through the entry points of qmag.py, with inputs and weights of
the shapes and distributions such a model has.

  matmul       qmag_matmul_dev, the projections and the LM head (one token: decode;
               several: the prompt, a batch)
  group        qmag_matmul_group_dev, the projections of one activation vector
  matmul_f32   qmag_matmul_f32_dev, the fp32 form (no activation quantisation)
  moe          qmag_moe_ffn_dev, one MoE FFN layer (one token, a small batch, a
               prompt chunk)
  moe_f32      qmag_moe_ffn_f32_dev, its fp32 form
  stack        qmag_moe_stack_dev, one token through a stack of MoE layers (decode)
  sample       qmag_sampler_*_dev, the next token from the logits

Weights are block bytes drawn directly in the two GGUF formats, with the nibble, scale
and minimum statistics that quantising N(0, 0.02) gives; activations are N(0, 1).
"""
import math
import os
import sys
from types import SimpleNamespace

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.getcwd(), "qwen-mobile-agent_amd"))
import qmag  # noqa: E402

DEV = "cuda:0"
WTYPE = {"q4_K": qmag.TYPE_Q4_K, "q6_K": qmag.TYPE_Q6_K}
BLOCK = {"q4_K": 144, "q6_K": 210}
MASK64 = (1 << 64) - 1
MOE = dict(n_embd=2048, n_ff=512, n_expert=256, n_used=8)


def listed():
    return [
        # one projection of one decoded token (the attention output's size class): a
        # few microseconds, where the launch counts
        dict(name="proj_t1", kind="matmul", n_in=2048, n_out=2048, T=1, wtype="q4_K", repacked=False),
        # q, k and v of one token in one launch, two weight types
        dict(name="qkv_group_t1", kind="group", n_in=2048, mats="8192:q4_K,512:q4_K,512:q6_K"),
        # one token, a row length that is no power of two and an odd row count
        dict(name="proj_odd_t1", kind="matmul", n_in=5120, n_out=1537, T=1, wtype="q6_K", repacked=False),
        # the LM head of one token, as the file holds it
        dict(name="head_t1", kind="matmul", n_in=2048, n_out=151936, T=1, wtype="q6_K", repacked=False),
        # the widest projection over a full prompt chunk
        dict(name="proj_t512", kind="matmul", n_in=2048, n_out=8192, T=512, wtype="q4_K", repacked=False),
        # the output projection over a short ragged prompt
        dict(name="proj_t37", kind="matmul", n_in=4096, n_out=2048, T=37, wtype="q6_K", repacked=False),
        # the fp32 form over a short prompt
        dict(name="proj_f32_t24", kind="matmul_f32", n_in=2048, n_out=2048, T=24, wtype="q4_K"),
        # one layer over a handful of tokens (a few sequences decoded together, the
        # last tokens of a prompt)
        dict(name="moe_t5", kind="moe", T=5, down="q4_K", bias=False, **MOE),
        # one layer over a full prompt chunk, experts chosen unevenly
        dict(name="moe_t512", kind="moe", T=512, down="q6_K", bias=True, **MOE),
        # the fp32 form of a layer over a few tokens
        dict(name="moe_f32_t12", kind="moe_f32", T=12, down="q6_K", bias=False, **MOE),
        # one decoded token through the model's layers
        dict(name="stack_t1", kind="stack", n_layer=40, down="q6_K", **MOE),
        # the next token of the engine's vocabulary: top-40 and the pick
        dict(name="sample", kind="sample", n_vocab=248320, top_k=40, temp=0.7, penalty=1.1, n_last=64, pick=True),
    ]


def _log_int(rng, lo, hi):
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    kind = rng.choice(["matmul_t1", "matmul_tn", "matmul_tn", "group", "matmul_f32", "moe_t1", "moe_tn", "moe_tn",
                       "moe_f32", "stack", "sample"])
    wtype = rng.choice(["q4_K", "q6_K"])
    if kind == "matmul_t1":
        n_in = 256 * _log_int(rng, 2, 32)
        repacked = wtype == "q6_K" and n_in % 2048 == 0 and rng.random() < 0.5
        n_out = _log_int(rng, 32, min(151936, 151936 * 2048 // n_in))
        return dict(kind="matmul", n_in=n_in, n_out=n_out, T=1, wtype=wtype, repacked=repacked)
    if kind == "matmul_tn":
        n_in, T = 256 * _log_int(rng, 2, 32), _log_int(rng, 2, 512)
        n_out = _log_int(rng, 32, max(32, min(16384, 2048 * 8192 * 512 // (n_in * T))))
        return dict(kind="matmul", n_in=n_in, n_out=n_out, T=T, wtype=wtype, repacked=False)
    if kind == "group":
        n_in = rng.choice([1024, 2048, 4096])
        mats = ",".join("%d:%s" % (_log_int(rng, 32, 8192), rng.choice(["q4_K", "q6_K"]))
                        for _ in range(rng.randint(2, 4)))
        return dict(kind="group", n_in=n_in, mats=mats)
    if kind == "matmul_f32":
        return dict(kind="matmul_f32", n_in=256 * _log_int(rng, 2, 16), n_out=_log_int(rng, 32, 4096),
                    T=_log_int(rng, 1, 48), wtype=wtype)
    shape = dict(MOE)
    if kind in ("moe_tn", "moe_f32") and rng.random() < 0.5:
        shape = dict(n_embd=rng.choice([1024, 2048, 4096]), n_ff=rng.choice([256, 512]),
                     n_expert=rng.choice([64, 128, 200]), n_used=rng.choice([4, 6, 8]))
    if kind == "moe_t1":
        return dict(kind="moe", T=1, down=wtype, bias=rng.random() < 0.5, **shape)
    if kind == "moe_tn":
        return dict(kind="moe", T=_log_int(rng, 2, 512), down=wtype, bias=rng.random() < 0.5, **shape)
    if kind == "moe_f32":
        return dict(kind="moe_f32", T=_log_int(rng, 1, 16), down=wtype, bias=rng.random() < 0.5, **shape)
    if kind == "stack":
        return dict(kind="stack", n_layer=_log_int(rng, 2, 40), down=wtype, **shape)
    return dict(kind="sample", n_vocab=_log_int(rng, 32000, 262144), top_k=rng.choice([1, 20, 40]),
                temp=rng.choice([0.0, 0.6, 1.0]), penalty=rng.choice([1.0, 1.1]), n_last=rng.randint(0, 64),
                pick=rng.random() < 0.7)


# ------------------------------------------------------------------ inputs --

def _gen(seed, tag):
    g = torch.Generator(device=DEV)
    g.manual_seed((seed * 1000003 + tag * 7919 + 1) & 0x7FFFFFFFFFFFFFFF)
    return g


def _f16_bytes(v):
    return v.to(torch.float16).view(torch.uint8).reshape(-1, 2)


def _blocks(g, n_blocks, wtype):
    """Block bytes [n_blocks, 144 or 210] of weights ~ N(0, 0.02)."""
    out = torch.empty((n_blocks, BLOCK[wtype]), dtype=torch.uint8, device=DEV)
    step = 1 << 19
    for a in range(0, n_blocks, step):
        n = min(step, n_blocks - a)
        o = out[a:a + n]
        spread = 0.9 + 0.2 * torch.rand((n, 1), device=DEV, generator=g)

        def normal(cols, std, mid, lo, hi):
            v = torch.randn((n, cols), device=DEV, generator=g, dtype=torch.float16)
            return v.mul_(std).add_(mid).round_().clamp_(lo, hi)

        if wtype == "q4_K":
            o[:, 0:2] = _f16_bytes(0.276 * 0.02 / 52 * spread)
            o[:, 2:4] = _f16_bytes(2.07 * 0.02 / 52 * spread)
            sc = torch.randint(41, 64, (n, 8), device=DEV, generator=g, dtype=torch.uint8)
            mn = torch.randint(41, 64, (n, 8), device=DEV, generator=g, dtype=torch.uint8)
            o[:, 4:8] = sc[:, :4] | ((sc[:, 4:] >> 4) << 6)
            o[:, 8:12] = mn[:, :4] | ((mn[:, 4:] >> 4) << 6)
            o[:, 12:16] = (sc[:, 4:] & 15) | ((mn[:, 4:] & 15) << 4)
            o[:, 16:] = normal(128, 3.6, 7.5, 0, 15).to(torch.uint8) | (normal(128, 3.6, 7.5, 0, 15).to(torch.uint8) << 4)
        else:
            q = normal(256, 18.0, 32.0, 0, 63).to(torch.uint8).view(n, 2, 4, 32)     # [half][quarter][l]
            o[:, 0:128] = ((q[:, :, :2] & 15) | ((q[:, :, 2:] & 15) << 4)).reshape(n, 128)
            hi = q >> 4
            o[:, 128:192] = (hi[:, :, 0] | (hi[:, :, 1] << 2) | (hi[:, :, 2] << 4) | (hi[:, :, 3] << 6)).reshape(n, 64)
            sc = torch.randint(80, 128, (n, 16), device=DEV, generator=g, dtype=torch.int16)
            sign = torch.randint(0, 2, (n, 16), device=DEV, generator=g, dtype=torch.int16) * 2 - 1
            o[:, 192:208] = (sc * sign).to(torch.int8).view(torch.uint8)
            o[:, 208:210] = _f16_bytes(0.02 / 18.0 / 104 * spread)
    return out


def _matrix(seed, tag, n_in, n_out, wtype):
    return _blocks(_gen(seed, tag), n_out * n_in // 256, wtype)


def _normal(seed, tag, shape, std=1.0):
    return torch.randn(shape, device=DEV, generator=_gen(seed, tag)) * std


def _layer_tensors(case, seed, il):
    N, F, E = case["n_embd"], case["n_ff"], case["n_expert"]
    t = 100 + 20 * il
    w = dict(gate_inp=_normal(seed, t + 1, (E, N), 0.02), gate_exps=_matrix(seed, t + 2, N, E * F, "q4_K"),
             up_exps=_matrix(seed, t + 3, N, E * F, "q4_K"), down_exps=_matrix(seed, t + 4, F, E * N, case["down"]),
             gate_inp_shexp=_normal(seed, t + 5, (N,), 0.02), gate_shexp=_matrix(seed, t + 6, N, F, "q4_K"),
             up_shexp=_matrix(seed, t + 7, N, F, "q4_K"), down_shexp=_matrix(seed, t + 8, F, N, case["down"]))
    w["router_bias"] = _normal(seed, t + 9, (E,)) if case.get("bias") else None
    return SimpleNamespace(**w)


def _layer(case, w):
    t_down = WTYPE[case["down"]]
    return qmag.MoeLayer(case["n_embd"], case["n_ff"], case["n_expert"], case["n_used"], w.gate_inp.data_ptr(),
                         w.router_bias.data_ptr() if w.router_bias is not None else None, w.gate_exps.data_ptr(),
                         w.up_exps.data_ptr(), w.down_exps.data_ptr(), t_down, w.gate_inp_shexp.data_ptr(),
                         w.gate_shexp.data_ptr(), w.up_shexp.data_ptr(), w.down_shexp.data_ptr(), t_down)


def _mats(case):
    for i, m in enumerate(case["mats"].split(",")):
        n_out, wtype = m.split(":")
        yield i, int(n_out), wtype


def _logits(case, seed):
    return _normal(seed, 1, (case["n_vocab"],), 2.5)


def _history(case, seed):
    g = torch.Generator()
    g.manual_seed(seed)
    return torch.randint(0, case["n_vocab"], (case["n_last"],), generator=g).tolist()


class _Buf:
    """A tensor as the binding's calls take a device buffer."""

    def __init__(self, t):
        self.t, self.ptr = t, t.data_ptr()


def prepare(case, seed):
    qmag.init(0)
    k = case["kind"]
    s = SimpleNamespace(case=case)
    if k in ("matmul", "matmul_f32"):
        s.x = _Buf(_normal(seed, 1, (case["T"], case["n_in"])))
        s.W = _Buf(_matrix(seed, 2, case["n_in"], case["n_out"], case["wtype"]))
        s.wtype = WTYPE[case["wtype"]]
        s.out = _Buf(torch.zeros((case["T"], case["n_out"]), device=DEV))
        torch.cuda.synchronize()
        if case.get("repacked"):        # once, when the weights are loaded
            qmag.repack_q6k_dev(s.W, s.W, case["n_in"], case["n_out"])
            s.wtype = qmag.TYPE_Q6_K_R
            qmag.sync()
    elif k == "group":
        s.x = _Buf(_normal(seed, 1, (case["n_in"],)))
        s.mats = [(_Buf(_matrix(seed, 2 + i, case["n_in"], n, w)), n, WTYPE[w]) for i, n, w in _mats(case)]
        s.outs = [_Buf(torch.zeros(n, device=DEV)) for _, n, _ in s.mats]
    elif k in ("moe", "moe_f32"):
        s.w = _layer_tensors(case, seed, 0)
        s.layer = _layer(case, s.w)
        s.x = _normal(seed, 1, (case["T"], case["n_embd"]))
        s.out = torch.zeros_like(s.x)
    elif k == "stack":
        s.w = [_layer_tensors(case, seed, il) for il in range(case["n_layer"])]
        s.layers = [_layer(case, w) for w in s.w]
        s.x0 = _normal(seed, 1, (1, case["n_embd"]))
        s.x = torch.zeros_like(s.x0)
    else:
        s.logits = _logits(case, seed)
        s.state = qmag.Sampler.init(seed=seed + 1, temp=case["temp"], top_k=case["top_k"], top_p=0.95,
                                    repeat_penalty=case["penalty"], last=_history(case, seed))
    torch.cuda.synchronize()            # the library works on a stream of its own
    return s


def run(s):
    case, k = s.case, s.case["kind"]
    if k == "matmul":
        qmag.matmul_dev(s.x, s.W, case["n_in"], case["n_out"], case["T"], s.wtype, s.out)
        return s.out.t
    if k == "matmul_f32":
        qmag.matmul_f32_dev(s.x, s.W, case["n_in"], case["n_out"], case["T"], s.wtype, s.out)
        return s.out.t
    if k == "group":
        qmag.matmul_group_dev(s.x, case["n_in"], s.mats, s.outs)
        return [o.t for o in s.outs]
    if k == "moe":
        qmag.moe_ffn_dev(s.layer, s.x.data_ptr(), s.out.data_ptr(), case["T"])
        return s.out
    if k == "moe_f32":
        qmag.moe_ffn_f32_dev(s.layer, s.x.data_ptr(), s.out.data_ptr(), case["T"])
        return s.out
    if k == "stack":
        # the token's embedding arrives in x, which the stack updates in place
        qmag.check(qmag.lib().qmag_d2d(s.x.data_ptr(), s.x0.data_ptr(), 4 * case["n_embd"]))
        qmag.moe_stack_dev(s.layers, s.x.data_ptr(), 1)
        return s.x
    state = qmag.Sampler.from_buffer_copy(s.state)
    if not case["pick"]:
        ids, vals = qmag.sampler_candidates_dev(s.logits.data_ptr(), case["n_vocab"], state)
        return {"ids": ids, "values": vals}
    token = qmag.sampler_sample_dev(s.logits.data_ptr(), case["n_vocab"], state)
    return {"token": token, "seed_hi": int(state.seed >> 32), "seed_lo": int(state.seed & 0xFFFFFFFF),
            "last": np.array(state.last_tokens[:state.n_last], dtype=np.int64)}


# -------------------------------------------------------------------- work --

def _experts_read(case):
    """Distinct routed experts of T tokens whose logits are N(0, 0.9) plus the bias."""
    T, E, K = case["T"], case["n_expert"], case["n_used"]
    r = np.random.RandomState(7)
    lg = r.randn(T, E) * 0.02 * math.sqrt(case["n_embd"])
    if case["bias"]:
        lg += r.randn(E)
    return len(np.unique(np.argpartition(-lg, K - 1, axis=1)[:, :K]))


def work(case):
    k = case["kind"]
    if k in ("matmul", "matmul_f32"):
        n_in, n_out, T = case["n_in"], case["n_out"], case["T"]
        return {"bytes": n_in * n_out // 256 * BLOCK[case["wtype"]] + 4 * T * (n_in + n_out), "flops": 2 * n_in * n_out * T}
    if k == "group":
        n_in = case["n_in"]
        return {"bytes": sum(n_in // 256 * n * BLOCK[w] + 4 * n for _, n, w in _mats(case)) + 4 * n_in,
                "flops": sum(2 * n_in * n for _, n, _ in _mats(case))}
    if k == "sample":
        return {"bytes": 4 * case["n_vocab"], "flops": 2 * case["n_vocab"]}
    N, F, E, K = (case[n] for n in ("n_embd", "n_ff", "n_expert", "n_used"))
    expert = 2 * F * N // 256 * 144 + N * F // 256 * BLOCK[case["down"]]
    T = case.get("T", 1)
    per_token = 2 * (E * N + N + 3 * (K + 1) * N * F)
    if k == "stack":
        return {"bytes": case["n_layer"] * (4 * N * (E + 1) + (K + 1) * expert) + 8 * N, "flops": case["n_layer"] * per_token}
    return {"bytes": 4 * N * (E + 1) + (_experts_read(case) + 1) * expert + 8 * T * N, "flops": T * per_token}


def tolerance(case):
    k = case["kind"]
    if k in ("matmul", "matmul_f32", "group"):
        # fp32 sums in any order over exact integer block sums (fp32: over the products)
        return {"rel": 1e-5, "max": 1e-4}
    if k == "moe_f32":
        return {"rel": 1e-5, "max": 1e-4}
    if k == "moe":
        # Q8_K(h) rounds a value of h that lies on a rounding boundary to either side: one
        # step (amax / 127) of one of 512 values moves an expert's output by up to 2e-3 of
        # its norm, which for one token may be most of the result
        return {"rel": 4e-3, "max": 3e-2}
    if k == "stack":
        # such steps change x, then Q8_K(x) and now and then a near-tied expert of the
        # layers behind: 0.02 of the norm after 40 layers against 64-bit sums
        return {"rel": 1.5e-3 * case["n_layer"], "max": 7.5e-3 * case["n_layer"]}
    return {"rel": 1e-6, "max": 1e-6}


# ------------------------------------------------------------------- exact --

def _deq(b, wtype):
    """float64 weights [n_blocks, 256] of block bytes."""
    n = b.shape[0]
    if wtype == "q4_K":
        d = b[:, 0:2].contiguous().view(torch.float16).double()
        dmin = b[:, 2:4].contiguous().view(torch.float16).double()
        s, m, x = b[:, 4:8], b[:, 8:12], b[:, 12:16]
        sc = torch.cat([s & 63, (x & 15) | ((s >> 6) << 4)], 1).double()
        mn = torch.cat([m & 63, (x >> 4) | ((m >> 6) << 4)], 1).double()
        qs = b[:, 16:].reshape(n, 4, 32)
        q = torch.stack([qs & 15, qs >> 4], 2).reshape(n, 8, 32).double()
        return (q * (d * sc)[:, :, None] - (dmin * mn)[:, :, None]).reshape(n, 256)
    ql, qh = b[:, 0:128].reshape(n, 2, 2, 32), b[:, 128:192].reshape(n, 2, 32)
    lo = torch.cat([ql & 15, ql >> 4], 2)                                          # [n][half][quarter][l]
    hi = torch.stack([(qh >> (2 * Q)) & 3 for Q in range(4)], 2)
    q = (lo | (hi << 4)).double() - 32.0
    sc = b[:, 192:208].contiguous().view(torch.int8).double()                       # per 16 values
    d = b[:, 208:210].contiguous().view(torch.float16).double()
    return (q.reshape(n, 16, 16) * (d * sc)[:, :, None]).reshape(n, 256)


def _rows(b, n_in, wtype):
    return _deq(b, wtype).reshape(-1, n_in)


def _q8(x):
    """The values Q8_K(x) stands for, in float64; the format's own steps are fp32."""
    v = x.float().reshape(-1, 256)
    amax = v.abs().amax(1, keepdim=True)
    d = torch.where(amax > 0, amax / 127.0, torch.ones_like(amax))
    t = (v * (1.0 / d)).double()
    q = (torch.sign(t) * torch.floor(t.abs() + 0.5)).clamp(-127, 127)
    return (q * d.double()).reshape(x.shape)


def _product(x, b, n_in, wtype):
    per = max(1, (1 << 26) // n_in) * (n_in // 256)
    return torch.cat([x @ _rows(b[a:a + per], n_in, wtype).T for a in range(0, b.shape[0], per)], 1)


def _moe(case, w, x, quantise):
    """One layer in float64; x [T, n_embd] float64."""
    N, F, E, K, T = case["n_embd"], case["n_ff"], case["n_expert"], case["n_used"], x.shape[0]
    gb, db = F * N // 256, N * F // 256
    q = _q8 if quantise else (lambda v: v)
    lg = x @ w.gate_inp.double().T
    if w.router_bias is not None:
        lg = lg + w.router_bias.double()
    top, sel = lg.topk(K, dim=1)
    wt = torch.softmax(top, 1)
    xq = q(x)

    def ffn(v, g, u, dn):
        gg, uu = v @ _rows(g, N, "q4_K").T, v @ _rows(u, N, "q4_K").T
        return q(gg / (1 + torch.exp(-gg)) * uu) @ _rows(dn, F, case["down"]).T

    out = torch.sigmoid(xq @ w.gate_inp_shexp.double())[:, None] * ffn(xq, w.gate_shexp, w.up_shexp, w.down_shexp)
    for e in sel.unique().tolist():
        t, k = (sel == e).nonzero(as_tuple=True)
        y = ffn(xq[t], w.gate_exps[e * gb:(e + 1) * gb], w.up_exps[e * gb:(e + 1) * gb],
                w.down_exps[e * db:(e + 1) * db])
        out.index_add_(0, t, wt[t, k][:, None] * y)
    return out


def _sample(case, seed):
    lg = _logits(case, seed).cpu().numpy().astype(np.float64)
    for i in _history(case, seed):
        lg[i] = lg[i] * case["penalty"] if lg[i] < 0 else lg[i] / case["penalty"]
    if case["temp"] > 0:
        lg /= case["temp"]
    k = min(case["top_k"], 40)
    ids = np.lexsort((np.arange(lg.size), -lg))[:k]
    if not case["pick"]:
        return {"ids": ids.astype(np.int32), "values": lg[ids]}
    st, last = seed + 1, _history(case, seed)
    if case["temp"] <= 0:
        token = int(ids[0])
    else:
        p = np.exp(lg[ids] - lg[ids[0]])
        c = np.cumsum(p / p.sum())
        kept = min(k, int(np.searchsorted(c, np.float32(0.95))) + 1)
        st ^= st >> 12
        st ^= (st << 25) & MASK64
        st ^= st >> 27
        r = float(((st * 0x2545F4914F6CDD1D) & MASK64) >> 11) / 2.0 ** 53
        token = int(ids[min(int(np.searchsorted(c[:kept], r, side="right")), kept - 1)])
        last = (last + [token])[-64:]
    return {"token": token, "seed_hi": st >> 32, "seed_lo": st & 0xFFFFFFFF, "last": np.array(last, dtype=np.int64)}


def exact(case, seed):
    k = case["kind"]
    if k in ("matmul", "matmul_f32"):
        x = _normal(seed, 1, (case["T"], case["n_in"])).double()
        W = _matrix(seed, 2, case["n_in"], case["n_out"], case["wtype"])
        return _product(x if k == "matmul_f32" else _q8(x), W, case["n_in"], case["wtype"])
    if k == "group":
        x = _q8(_normal(seed, 1, (1, case["n_in"])).double())
        return [_product(x, _matrix(seed, 2 + i, case["n_in"], n, w), case["n_in"], w)[0] for i, n, w in _mats(case)]
    if k in ("moe", "moe_f32"):
        x = _normal(seed, 1, (case["T"], case["n_embd"])).double()
        return _moe(case, _layer_tensors(case, seed, 0), x, k == "moe")
    if k == "stack":
        x = _normal(seed, 1, (1, case["n_embd"])).double()
        for il in range(case["n_layer"]):
            x = x + _moe(case, _layer_tensors(case, seed, il), x, True)
        return x
    return _sample(case, seed)
