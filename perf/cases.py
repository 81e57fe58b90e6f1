"""The calls this library is measured on: what a training or rollout program for the policy networks asks
of it, through the C ABI (include/talos_hip.h) by way of the ctypes binding.

Kinds of call, each with the sizes it is used at:

* policy  -- one PPO minibatch, forward + backward (talos_ppo_minibatch_f32): the reference's own actor-critic
             (one MLA layer, d 64, ReLU, 5 actions) and the d 128 policy (two layers, 4 heads x 32, GELU, causal,
             3 actions), full sequences or right-padded ragged ones.
* forward -- the same networks' logits and values alone (talos_ppo_forward_n_f32), as the rollout's old
             log-probs need them.
* block   -- one pre-norm transformer block, forward + backward (talos_block_fwd_bwd_f32).
* mla     -- one multi-head-latent-attention block, forward + backward (talos_mla_fwd_bwd_f32), fp32 or with
             bf16 operands.
* linear  -- one Linear layer as the tape calls it: y = xW, dX = dY W^T, dW = x^T dY, db = column sums
             (talos_gemm_f32 or talos_gemm_bf16acc_f32, talos_bias_grad_f32).
* attention -- fused attention, forward + backward, on separate q / k / v tensors (talos_attn_fwd_f32, _bwd_f32).
* rows    -- the row operations of the tape on one activation: RMSNorm, causal softmax and RoPE, each forward
             and backward.
* rollout -- an episode of the KV-cache decoder: one token per environment and step, caches reset at the
             first (talos_ppo_decoder_step_f32).

The calling thread is in the asynchronous mode with a scratch workspace bound, as a training loop sets
itself up; everything runs on the default stream.
"""
import ctypes
import math
import os
import sys

import numpy as np
import torch

_PKG = os.path.join(os.getcwd(), "talos-xii_amd")
if _PKG not in sys.path:
    sys.path.insert(0, _PKG)

import talos_hip as th  # noqa: E402

# in_dim, d_model, layers, heads, head_dim, ffn, actions, causal, activation, eps, MLA widths (0: standard)
_NETS = {
    "reference": dict(I=8, d=64, L=1, H=4, hd=16, F=128, A=5, causal=0, act=th.ACT_RELU, lat=32, r=16, vd=16),
    "policy128": dict(I=8, d=128, L=2, H=4, hd=32, F=512, A=3, causal=1, act=th.ACT_GELU, lat=0, r=0, vd=0),
}
_EPS, _BASE, _CLIP, _VC, _EC = 1e-5, 10000.0, 0.2, 0.5, 0.01
_WORKSPACE_BYTES = 256 << 20
_workspace = None


def listed():
    return [
        # a Linear layer of the value networks at their replay batch: launch latency is all of it
        {"name": "linear_256x64x64", "kind": "linear", "M": 256, "K": 64, "N": 64, "prec": "fp32"},
        # a wide projection over a whole batch of tokens: the tape's GEMMs at full size
        {"name": "linear_16384x512x2048", "kind": "linear", "M": 16384, "K": 512, "N": 2048, "prec": "fp32"},
        # the reference trainer's own minibatch: 256 samples of its context length, of varying lengths
        {"name": "actor_critic_256x16_ragged", "kind": "policy", "net": "reference", "B": 256, "S": 16, "ragged": True},
        # the same network over a large batched rollout
        {"name": "actor_critic_4096x16", "kind": "policy", "net": "reference", "B": 4096, "S": 16, "ragged": False},
        # the headline minibatch
        {"name": "policy_4096x32", "kind": "policy", "net": "policy128", "B": 4096, "S": 32, "ragged": False},
        # a mid-size minibatch at no round number, right-padded
        {"name": "policy_700x21_ragged", "kind": "policy", "net": "policy128", "B": 700, "S": 21, "ragged": True},
        # one standard block at a longer context
        {"name": "block_512x64_d128", "kind": "block", "B": 512, "S": 64, "d": 128, "H": 4, "F": 512,
         "causal": 1},
        # the latent-attention block at its full size, in both precisions
        {"name": "mla_64x256_d512", "kind": "mla", "B": 64, "S": 256, "d": 512, "H": 8, "lat": 128, "r": 32, "hd": 64,
         "vd": 64, "causal": 0, "prec": "fp32"},
        {"name": "mla_64x256_d512_bf16", "kind": "mla", "B": 64, "S": 256, "d": 512, "H": 8, "lat": 128, "r": 32,
         "hd": 64, "vd": 64, "causal": 0, "prec": "bf16"},
        # attention by itself, as the tape's modules call it, at a ragged length
        {"name": "attention_24x200_8x64", "kind": "attention", "B": 24, "S": 200, "H": 8, "dk": 64, "dv": 64,
         "causal": 1},
        # the tape's row operations on one layer's activations
        {"name": "rows_4096x256", "kind": "rows", "R": 4096, "C": 256, "S": 64, "hd": 64},
        # an episode of the rollout decoder over a full set of environments
        {"name": "rollout_4096_w16", "kind": "rollout", "net": "reference", "n": 4096, "window": 16, "T": 20},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["linear", "linear", "policy", "policy", "policy", "forward", "block", "block", "mla", "mla",
                       "attention", "rows", "rollout"])
    if kind == "linear":
        c = {"kind": kind, "M": _log_int(rng, 64, 65536), "K": _log_int(rng, 8, 2048), "N": _log_int(rng, 8, 2048),
             "prec": rng.choice(["fp32", "fp32", "bf16"])}
        while 6 * c["M"] * c["K"] * c["N"] > 1.5e11:
            c["M"] //= 2
        return c
    if kind in ("policy", "forward"):
        net = rng.choice(["reference", "policy128"])
        S = rng.randint(4, 32)
        return {"kind": kind, "net": net, "B": min(_log_int(rng, 64, 4096), 131072 // S), "S": S,
                "ragged": rng.random() < 0.5}
    if kind == "block":
        d, H = rng.choice([(64, 4), (128, 4), (128, 8), (256, 8)])
        S = rng.randint(8, 128)
        tokens = _log_int(rng, 1024, 32768)
        return {"kind": kind, "B": max(1, tokens // S), "S": S, "d": d, "H": H, "F": d * rng.choice([2, 4]),
                "causal": rng.randint(0, 1)}
    if kind == "mla":
        d, H, lat, r, hd, vd = rng.choice([(512, 8, 128, 32, 64, 64), (256, 4, 64, 32, 64, 64),
                                           (256, 8, 64, 16, 16, 32)])
        S = rng.randint(48, 256)
        return {"kind": kind, "B": max(1, _log_int(rng, 1024, 16384) // S), "S": S, "d": d, "H": H, "lat": lat, "r": r,
                "hd": hd, "vd": vd, "causal": rng.randint(0, 1), "prec": rng.choice(["fp32", "bf16"])}
    if kind == "attention":
        dk, dv = rng.choice([(32, 32), (64, 64), (96, 64), (128, 128)])
        S = rng.randint(8, 256)
        H = rng.choice([4, 8])
        return {"kind": kind, "B": max(1, _log_int(rng, 512, 16384) // S), "S": S, "H": H, "dk": dk, "dv": dv,
                "causal": rng.randint(0, 1)}
    if kind == "rows":
        hd = rng.choice([16, 32, 64])
        C = hd * rng.randint(2, 16)
        S = rng.randint(16, 256)
        return {"kind": kind, "R": max(1, _log_int(rng, 256, 32768) // S) * S, "C": C, "S": S, "hd": hd}
    net = rng.choice(["reference", "reference", "policy128"])
    return {"kind": "rollout", "net": net, "n": _log_int(rng, 64, 4096), "window": rng.randint(4, 16), "T": 20}


# ---------------------------------------------------------------------------------------------------------
# Inputs (made on the GPU from the seed; the same tensors for run and exact)
# ---------------------------------------------------------------------------------------------------------

class _Draws:
    def __init__(self, seed):
        self.g = torch.Generator(device="cuda")
        self.g.manual_seed(1000003 * (seed + 1))

    def normal(self, *shape, std=1.0):
        return torch.randn(*shape, generator=self.g, device="cuda") * std

    def uniform(self, lo, hi, *shape):
        return torch.rand(*shape, generator=self.g, device="cuda") * (hi - lo) + lo

    def integers(self, lo, hi, *shape):
        return torch.randint(lo, hi, shape, generator=self.g, device="cuda", dtype=torch.int32)

    def xavier(self, fan_in, fan_out, cols=None):
        lim = math.sqrt(6.0 / (fan_in + fan_out))
        return self.uniform(-lim, lim, fan_in, cols or fan_out)


def _mha_block_params(g, d, F):
    return [("g1", g.uniform(0.9, 1.1, d)), ("wqkv", g.xavier(d, d, 3 * d)), ("wo", g.xavier(d, d)),
            ("g2", g.uniform(0.9, 1.1, d)), ("w1", g.xavier(d, F)), ("b1", g.normal(F, std=0.02)),
            ("w2", g.xavier(F, d)), ("b2", g.normal(d, std=0.02))]


def _mla_params(g, d, H, lat, r, hd, vd):
    return [("g1", g.uniform(0.9, 1.1, d)), ("wdkv", g.xavier(d, lat)), ("wuk", g.xavier(lat, H * hd)),
            ("wuv", g.xavier(lat, H * vd)), ("wq", g.xavier(d, H * hd)), ("wkr", g.xavier(d, H * r)),
            ("wqr", g.xavier(d, H * r)), ("wo", g.xavier(H * vd, d))]


def _net_params(g, n):
    d, F = n["d"], n["F"]
    out = [("we", g.xavier(n["I"], d)), ("be", g.normal(d, std=0.02))]
    for i in range(n["L"]):
        if n["lat"]:
            b = _mla_params(g, d, n["H"], n["lat"], n["r"], n["hd"], n["vd"])
            b += _mha_block_params(g, d, F)[3:]
        else:
            b = _mha_block_params(g, d, F)
        out += [("%d.%s" % (i, k), v) for k, v in b]
    return out + [("gf", g.uniform(0.9, 1.1, d)), ("wout", g.xavier(d, d)), ("bout", g.normal(d, std=0.02)),
                  ("wa", g.xavier(d, n["A"])), ("ba", g.normal(n["A"], std=0.02)), ("wc", g.xavier(d, 1)),
                  ("bc", g.normal(1, std=0.02))]


def _flat(params):
    return torch.cat([v.reshape(-1) for _, v in params])


def _states(g, B, S):
    """Gacha states: pity, guarantee flag, log currency, pulls, pity x flag, pull phase and its square, noise."""
    pity = g.integers(0, 80, B, S).float() / 80.0
    flag = g.integers(0, 2, B, S).float()
    cur = torch.log1p(g.uniform(0, 1e4, B, S)) / math.log1p(1e4)
    pulls = g.uniform(0, 300, B, S)
    phase = torch.remainder(pulls, 120.0) / 120.0
    return torch.stack([pity, flag, cur, pulls / 300.0, pity * flag, phase, phase * phase, g.uniform(-1, 1, B, S)],
                       -1).contiguous()


def _inputs(case, seed):
    g = _Draws(seed)
    k = case["kind"]
    if k in ("policy", "forward"):
        n, B, S = _NETS[case["net"]], case["B"], case["S"]
        x = {"params": _net_params(g, n), "states": _states(g, B, S),
             "lengths": g.integers(1, S + 1, B) if case["ragged"] else None,
             "actions": g.integers(0, n["A"], B), "adv": g.normal(B), "ret": g.normal(B),
             # log-probs of a policy somewhat older than this one
             "old": -math.log(n["A"]) + g.normal(B, std=0.1)}
        return x
    if k == "block":
        B, S, d = case["B"], case["S"], case["d"]
        return {"params": _mha_block_params(g, d, case["F"]), "x": g.normal(B, S, d), "gout": g.normal(B, S, d)}
    if k == "mla":
        B, S, d = case["B"], case["S"], case["d"]
        return {"params": _mla_params(g, d, case["H"], case["lat"], case["r"], case["hd"], case["vd"]),
                "x": g.normal(B, S, d), "gout": g.normal(B, S, d)}
    if k == "linear":
        M, K, N = case["M"], case["K"], case["N"]
        return {"x": g.normal(M, K), "w": g.xavier(K, N), "dy": g.normal(M, N)}
    if k == "attention":
        B, S, H, dk, dv = (case[c] for c in ("B", "S", "H", "dk", "dv"))
        return {"q": g.normal(B, S, H, dk), "k": g.normal(B, S, H, dk), "v": g.normal(B, S, H, dv),
                "do": g.normal(B, S, H, dv)}
    if k == "rows":
        R, C = case["R"], case["C"]
        return {"x": g.normal(R, C), "w": g.uniform(0.9, 1.1, C), "dy": g.normal(R, C)}
    n, E, T = _NETS[case["net"]], case["n"], case["T"]
    return {"params": _net_params(g, n), "tokens": _states(g, T, E), "uniforms": g.uniform(0, 1, T, E)}


# ---------------------------------------------------------------------------------------------------------
# The calls
# ---------------------------------------------------------------------------------------------------------

def _ppo_cfg(n, B, S):
    return th.PpoCfg(B, S, n["I"], n["d"], n["L"], n["H"], n["hd"], n["F"], n["A"], n["causal"], n["act"], _EPS, _BASE,
                     _CLIP, _VC, _EC, th.ATTN_MLA if n["lat"] else th.ATTN_MHA, n["lat"], n["r"], n["vd"])


def _empty(*shape, dtype=torch.float32):
    return torch.empty(*shape, device="cuda", dtype=dtype)


def _p(t):
    return None if t is None else t.data_ptr()


def prepare(case, seed):
    global _workspace
    if _workspace is None:
        _workspace = _empty(_WORKSPACE_BYTES // 4)
    th.call("talos_set_async", 1)
    th.call("talos_workspace_bind", _workspace.data_ptr(), _WORKSPACE_BYTES)
    s = {"case": dict(case), "in": _inputs(case, seed)}
    i, k = s["in"], case["kind"]
    if "params" in i:
        i["flat"] = _flat(i.pop("params"))
    if k in ("policy", "forward"):
        n, B = _NETS[case["net"]], case["B"]
        s["plan"] = th.Plan("ppo", _ppo_cfg(n, B, case["S"]))
        if k == "policy":
            s["out"] = {"loss": _empty(1), "dparams": torch.empty_like(i["flat"])}
        else:
            s["out"] = {"logits": _empty(B, n["A"]), "values": _empty(B)}
    elif k == "block":
        s["plan"] = th.Plan("block", th.BlockCfg(case["B"], case["S"], case["d"], case["H"], case["d"] // case["H"],
                                                 case["F"], case["causal"], th.ACT_GELU, _EPS, _BASE))
        s["out"] = {"out": torch.empty_like(i["x"]), "dparams": torch.empty_like(i["flat"]),
                    "dx": torch.empty_like(i["x"])}
    elif k == "mla":
        prec = th.PREC_BF16 if case["prec"] == "bf16" else th.PREC_FP32
        s["plan"] = th.Plan("mla", th.MlaCfg(case["B"], case["S"], case["d"], case["H"], case["lat"], case["r"],
                                             case["hd"], case["vd"], case["causal"], prec, _EPS, _BASE))
        s["out"] = {"out": torch.empty_like(i["x"]), "dparams": torch.empty_like(i["flat"]),
                    "dx": torch.empty_like(i["x"])}
    elif k == "linear":
        s["out"] = {"y": torch.empty_like(i["dy"]), "dx": torch.empty_like(i["x"]), "dw": torch.empty_like(i["w"]),
                    "db": _empty(case["N"])}
    elif k == "attention":
        s["out"] = {"o": torch.empty_like(i["v"]), "lse": _empty(case["B"], case["H"], case["S"]),
                    "dq": torch.empty_like(i["q"]), "dk": torch.empty_like(i["k"]), "dv": torch.empty_like(i["v"])}
    elif k == "rows":
        s["rstd"] = _empty(case["R"])
        s["out"] = {a: torch.empty_like(i["x"]) for a in ("norm", "dnorm", "soft", "dsoft", "rope", "drope")}
        s["out"]["dw"] = _empty(case["C"])
    else:
        n, E, T = _NETS[case["net"]], case["n"], case["T"]
        s["dec"] = _Decoder(_ppo_cfg(n, 1, case["window"]), E, case["window"])
        s["pos"] = torch.arange(T, device="cuda", dtype=torch.int32)[:, None].expand(T, E).contiguous()
        s["reset"] = torch.ones(E, device="cuda", dtype=torch.uint8)
        s["logp"] = _empty(T, E)
        # logp is the chosen action's entry of log_softmax(logits), so it is not returned beside them
        s["out"] = {"logits": _empty(T, E, n["A"]), "values": _empty(T, E), "actions": _empty(T, E, dtype=torch.int32)}
    return s


class _Decoder:
    """The decoder handle, on caller-owned buffers."""

    def __init__(self, cfg, n, window):
        self.h = ctypes.c_void_p()
        th.call("talos_ppo_decoder_create", ctypes.byref(cfg), n, window, 256, ctypes.byref(self.h))

    def __del__(self):
        th.lib().talos_ppo_decoder_destroy(self.h)


def run(s):
    c, i, o, call = s["case"], s["in"], s["out"], th.call
    k = c["kind"]
    if k == "policy":
        call("talos_ppo_minibatch_f32", s["plan"].h, c["B"], _p(i["flat"]), _p(i["states"]), _p(i["lengths"]),
             _p(i["actions"]), _p(i["adv"]), _p(i["ret"]), _p(i["old"]), _p(o["loss"]), _p(o["dparams"]), None, 0, None)
    elif k == "forward":
        call("talos_ppo_forward_n_f32", s["plan"].h, c["B"], _p(i["flat"]), _p(i["states"]), _p(i["lengths"]),
             _p(o["logits"]), _p(o["values"]), None)
    elif k in ("block", "mla"):
        call("talos_%s_fwd_bwd_f32" % k, s["plan"].h, _p(i["flat"]), _p(i["x"]), _p(i["gout"]), _p(o["out"]),
             _p(o["dparams"]), _p(o["dx"]), None)
    elif k == "linear":
        M, K, N = c["M"], c["K"], c["N"]
        gemm = "talos_gemm_f32" if c["prec"] == "fp32" else "talos_gemm_bf16acc_f32"
        call(gemm, 0, 0, M, N, K, 1.0, _p(i["x"]), K, _p(i["w"]), N, 0.0, _p(o["y"]), N, None)
        call(gemm, 0, 1, M, K, N, 1.0, _p(i["dy"]), N, _p(i["w"]), N, 0.0, _p(o["dx"]), K, None)
        call(gemm, 1, 0, K, N, M, 1.0, _p(i["x"]), K, _p(i["dy"]), N, 0.0, _p(o["dw"]), N, None)
        call("talos_bias_grad_f32", M, N, _p(i["dy"]), 0.0, _p(o["db"]), None)
    elif k == "attention":
        B, S, H, dk, dv = (c[a] for a in ("B", "S", "H", "dk", "dv"))
        sc, q, v = 1.0 / math.sqrt(dk), H * dk, H * dv
        call("talos_attn_fwd_f32", B, S, H, dk, dv, sc, c["causal"], _p(i["q"]), q, _p(i["k"]), q, _p(i["v"]), v,
             _p(o["o"]), v, _p(o["lse"]), None)
        call("talos_attn_bwd_f32", B, S, H, dk, dv, sc, c["causal"], _p(i["q"]), q, _p(i["k"]), q, _p(i["v"]), v,
             _p(o["o"]), v, _p(o["lse"]), _p(i["do"]), v, _p(o["dq"]), q, _p(o["dk"]), q, _p(o["dv"]), v, None)
    elif k == "rows":
        R, C, x, dy = c["R"], c["C"], _p(i["x"]), _p(i["dy"])
        call("talos_rmsnorm_fwd_f32", R, C, _EPS, x, _p(i["w"]), _p(o["norm"]), _p(s["rstd"]), None)
        call("talos_rmsnorm_bwd_f32", R, C, x, _p(i["w"]), _p(s["rstd"]), dy, 0.0, _p(o["dnorm"]), 0.0, _p(o["dw"]),
             None)
        call("talos_softmax_fwd_f32", R, C, 1, x, _p(o["soft"]), None)
        call("talos_softmax_bwd_f32", R, C, 1, _p(o["soft"]), dy, 0.0, _p(o["dsoft"]), None)
        rope = (R // c["S"], c["S"], C // c["hd"], c["hd"], 0, _BASE)
        call("talos_rope_fwd_f32", *rope, x, _p(o["rope"]), None)
        call("talos_rope_bwd_f32", *rope, dy, 0.0, _p(o["drope"]), None)
    else:
        E, A = c["n"], _NETS[c["net"]]["A"]
        tok, pos, uni = _p(i["tokens"]), _p(s["pos"]), _p(i["uniforms"])
        lg, vl, ac, lp = _p(o["logits"]), _p(o["values"]), _p(o["actions"]), _p(s["logp"])
        for t in range(c["T"]):
            at = 4 * t * E
            call("talos_ppo_decoder_step_f32", s["dec"].h, E, _p(i["flat"]), tok + 8 * at, pos + at,
                 _p(s["reset"]) if t == 0 else None, uni + at, lg + A * at, vl + at, ac + at, lp + at, None)
    return o


# ---------------------------------------------------------------------------------------------------------
# What a pass cannot do without
# ---------------------------------------------------------------------------------------------------------

def _net_size(n):
    d, F = n["d"], n["F"]
    if n["lat"]:
        att = d * n["lat"] + n["lat"] * n["H"] * (n["hd"] + n["vd"]) + d * n["H"] * (n["hd"] + 2 * n["r"])
        att += n["H"] * n["vd"] * d
    else:
        att = 4 * d * d
    return n["I"] * d + d + n["L"] * (att + 2 * d + 2 * d * F + F + d) + d + d * d + d + (d + 1) * (n["A"] + 1)


def _pairs(S, causal):
    return S * (S + 1) / 2 if causal else S * S


def _net_flops(n, B, S):
    """Forward flops the loss depends on: after the last layer's attention only the last token of each sample."""
    M, d, F, H = B * S, n["d"], n["F"], n["H"]
    if n["lat"]:
        keys = d * n["lat"] + n["lat"] * H * (n["hd"] + n["vd"]) + d * H * n["r"]
        query, dk, dv = d * H * (n["hd"] + n["r"]), n["hd"] + n["r"], n["vd"]
    else:
        keys, query, dk, dv = 2 * d * d, d * d, n["hd"], n["hd"]
    after = H * dv * d + 2 * d * F
    full = 2 * M * (keys + query + after) + 2 * B * H * (dk + dv) * _pairs(S, n["causal"])
    last = 2 * M * keys + 2 * B * (query + after) + 2 * B * H * (dk + dv) * S
    return 2 * M * n["I"] * d + (n["L"] - 1) * full + last + 2 * B * d * (d + n["A"] + 1)


def work(case):
    k = case["kind"]
    if k in ("policy", "forward"):
        n, B, S = _NETS[case["net"]], case["B"], case["S"]
        tokens = (S + 1) / 2 if case["ragged"] else S
        f, p = _net_flops(n, B, tokens), 4 * _net_size(n)
        states = 4 * B * tokens * n["I"]
        if k == "policy":
            return {"bytes": states + 2 * p + 16 * B, "flops": 3 * f}
        return {"bytes": states + p + 4 * B * (n["A"] + 1), "flops": f}
    if k == "block":
        B, S, d, F = case["B"], case["S"], case["d"], case["F"]
        w = 4 * d * d + 2 * d * F
        return {"bytes": 16 * B * S * d + 8 * w, "flops": 3 * (2 * B * S * w + 4 * B * d * _pairs(S, case["causal"]))}
    if k == "mla":
        B, S, d, H, lat, r, hd, vd = (case[a] for a in ("B", "S", "d", "H", "lat", "r", "hd", "vd"))
        w = d * lat + lat * H * (hd + vd) + d * H * (hd + 2 * r) + H * vd * d
        return {"bytes": 16 * B * S * d + 8 * w,
                "flops": 3 * (2 * B * S * w + 2 * B * H * (hd + r + vd) * _pairs(S, case["causal"]))}
    if k == "linear":
        M, K, N = case["M"], case["K"], case["N"]
        return {"bytes": 4 * (2 * M * K + 2 * M * N + 2 * K * N + N), "flops": 6 * M * K * N}
    if k == "attention":
        B, S, H, dk, dv = (case[a] for a in ("B", "S", "H", "dk", "dv"))
        return {"bytes": 4 * B * S * H * (4 * dk + 4 * dv + 1),
                "flops": 2 * B * H * _pairs(S, case["causal"]) * (4 * dk + 3 * dv)}
    if k == "rows":
        R, C = case["R"], case["C"]
        return {"bytes": 4 * 8 * R * C, "flops": 0}
    n, E, T = _NETS[case["net"]], case["n"], case["T"]
    return {"bytes": 4 * (T * E * (n["I"] + n["A"] + 4) + _net_size(n)), "flops": 2 * T * E * _net_size(n)}


def tolerance(case):
    """About four times and more what fp32 shows against 64 bits (1e-7 .. 1.6e-6 over the ranges), and with bf16
    operands (2.4e-3 for one product, 6.6e-3 for the weight gradients of the latent-attention block)."""
    k = case["kind"]
    if case.get("prec") == "bf16":
        return {"rel": 1e-2 if k == "linear" else 2e-2}
    if k == "policy" and _NETS[case["net"]]["act"] == th.ACT_RELU:
        # a unit whose input is within rounding of 0 passes its gradient on one side of the kink only: one such
        # unit of one sample moves the gradient by about this much (a ReLU block over 20875 rows showed 7e-4)
        return {"rel": 0.1 / math.sqrt(case["B"])}
    if k == "rollout":
        return {"rel": 1e-5, "differ": 1e-4}
    return {"rel": 1e-5}


# ---------------------------------------------------------------------------------------------------------
# The same results in 64 bits, in plain torch
# ---------------------------------------------------------------------------------------------------------

def _norm64(x, w):
    return x * torch.rsqrt((x * x).mean(-1, keepdim=True) + _EPS) * w


def _rope64(x):
    """x [..., S, H, D], pairs (2i, 2i + 1) rotated by the position along S; the fp32 cos / sin table of the
    library's definition."""
    S, D = x.shape[-3], x.shape[-1]
    theta = 1.0 / (_BASE ** (torch.arange(0, D, 2, device=x.device, dtype=torch.float64) / D))
    ang = torch.arange(S, device=x.device, dtype=torch.float64)[:, None] * theta
    co, si = (f(ang).float().double()[:, None, :] for f in (torch.cos, torch.sin))
    a, b = x[..., 0::2], x[..., 1::2]
    return torch.stack([a * co - b * si, a * si + b * co], -1).reshape(x.shape)


def _attend64(q, k, v, scale, mask):
    """q, k [B, S, H, dk], v [B, S, H, dv]; mask [1 or B, S, S] of the pairs that are kept."""
    q, k, v = (t.transpose(1, 2).contiguous() for t in (q, k, v))
    s = torch.matmul(q, k.transpose(-1, -2).contiguous()) * scale
    s = s.masked_fill(~mask[:, None], float("-inf"))
    return torch.matmul(torch.softmax(s, -1), v).transpose(1, 2), torch.logsumexp(s, -1)


def _mask(S, causal, lengths=None, window=None):
    i = torch.arange(S, device="cuda")
    m = (i[None, :] <= i[:, None]) if causal else torch.ones(S, S, device="cuda", dtype=torch.bool)
    if window is not None:
        m = m & (i[None, :] >= i[:, None] - window)
    m = m[None]
    return m if lengths is None else m & (i[None, None, :] < lengths[:, None, None])


def _mha64(x, p, H, mask):
    B, S, d = x.shape
    q, k, v = (t.reshape(B, S, H, d // H) for t in (_norm64(x, p["g1"]) @ p["wqkv"]).split(d, -1))
    o, _ = _attend64(_rope64(q), _rope64(k), v, 1.0 / math.sqrt(d // H), mask)
    return x + o.reshape(B, S, d) @ p["wo"]


def _mla64(x, p, H, r, hd, vd, mask):
    B, S, _ = x.shape
    xn = _norm64(x, p["g1"])
    lat = xn @ p["wdkv"]
    q = torch.cat([(xn @ p["wq"]).reshape(B, S, H, hd), _rope64((xn @ p["wqr"]).reshape(B, S, H, r))], -1)
    k = torch.cat([(lat @ p["wuk"]).reshape(B, S, H, hd), _rope64((xn @ p["wkr"]).reshape(B, S, H, r))], -1)
    o, _ = _attend64(q, k, (lat @ p["wuv"]).reshape(B, S, H, vd), 1.0 / math.sqrt(hd + r), mask)
    return x + o.reshape(B, S, H * vd) @ p["wo"]


def _mlp64(h, p, act):
    u = _norm64(h, p["g2"]) @ p["w1"] + p["b1"]
    a = torch.relu(u) if act == th.ACT_RELU else 0.5 * u * (1.0 + torch.erf(u / math.sqrt(2.0)))
    return h + a @ p["w2"] + p["b2"]


def _net64(states, p, n, mask):
    """The output rows [B, S, d] of the backbone."""
    h = states @ p["we"] + p["be"]
    for i in range(n["L"]):
        b = {k.split(".")[1]: v for k, v in p.items() if k.startswith("%d." % i)}
        h = _mla64(h, b, n["H"], n["r"], n["hd"], n["vd"], mask) if n["lat"] else _mha64(h, b, n["H"], mask)
        h = _mlp64(h, b, n["act"])
    return _norm64(h, p["gf"]) @ p["wout"] + p["bout"]


def _leaves64(params):
    return {k: v.double().requires_grad_() for k, v in params}


def _grads(p):
    return torch.cat([v.grad.reshape(-1) for v in p.values()])


def exact(case, seed):
    i = {k: v.double() if torch.is_tensor(v) and v.is_floating_point() else v for k, v in _inputs(case, seed).items()}
    k = case["kind"]
    if k in ("policy", "forward"):
        n, S = _NETS[case["net"]], case["S"]
        p = _leaves64(i["params"])
        rows = _net64(i["states"], p, n, _mask(S, n["causal"], i["lengths"]))
        end = torch.full((case["B"],), S, device="cuda") if i["lengths"] is None else i["lengths"].long()
        last = rows[torch.arange(case["B"], device="cuda"), end - 1]
        logits, values = last @ p["wa"] + p["ba"], (last @ p["wc"] + p["bc"])[:, 0]
        if k == "forward":
            return {"logits": logits.detach(), "values": values.detach()}
        lp = torch.log_softmax(logits, -1)
        ratio = torch.exp(lp.gather(1, i["actions"].long()[:, None])[:, 0] - i["old"])
        s1, s2 = ratio * i["adv"], torch.clamp(ratio, 1.0 - _CLIP, 1.0 + _CLIP) * i["adv"]
        loss = (-torch.where(s1 < s2, s1, s2) + _VC * (values - i["ret"]) ** 2
                + _EC * (torch.exp(lp) * lp).sum(-1)).mean()
        loss.backward()
        return {"loss": loss.detach().reshape(1), "dparams": _grads(p)}
    if k in ("block", "mla"):
        p, x = _leaves64(i["params"]), i["x"].requires_grad_()
        mask = _mask(case["S"], case["causal"])
        if k == "block":
            out = _mlp64(_mha64(x, p, case["H"], mask), p, th.ACT_GELU)
        else:
            out = _mla64(x, p, case["H"], case["r"], case["hd"], case["vd"], mask)
        out.backward(i["gout"])
        return {"out": out.detach(), "dparams": _grads(p), "dx": x.grad}
    if k == "linear":
        return {"y": i["x"] @ i["w"], "dx": i["dy"] @ i["w"].t().contiguous(), "dw": i["x"].t().contiguous() @ i["dy"],
                "db": i["dy"].sum(0)}
    if k == "attention":
        q, kk, v = (i[a].requires_grad_() for a in ("q", "k", "v"))
        o, lse = _attend64(q, kk, v, 1.0 / math.sqrt(case["dk"]), _mask(case["S"], case["causal"]))
        o.backward(i["do"])
        return {"o": o.detach(), "lse": lse.detach(), "dq": q.grad, "dk": kk.grad, "dv": v.grad}
    if k == "rows":
        R, C, S, hd = (case[a] for a in ("R", "C", "S", "hd"))
        x, w, dy = i["x"].requires_grad_(), i["w"].requires_grad_(), i["dy"]
        norm = _norm64(x, w)
        dnorm, dw = torch.autograd.grad(norm, [x, w], dy)
        keep = torch.arange(C, device="cuda")[None, :] <= (torch.arange(R, device="cuda") % C)[:, None]
        soft = torch.softmax(x.masked_fill(~keep, float("-inf")), -1)
        # the backward reads the forward's fp32 rows; its own 64-bit value from the 64-bit rows is as close
        (dsoft,) = torch.autograd.grad(soft, x, dy)
        rot = _rope64(x.reshape(R // S, S, C // hd, hd)).reshape(R, C)
        (drope,) = torch.autograd.grad(rot, x, dy)
        return {"norm": norm.detach(), "dnorm": dnorm, "soft": soft.detach(), "dsoft": dsoft, "rope": rot.detach(),
                "drope": drope, "dw": dw}
    n, E = _NETS[case["net"]], case["n"]
    p = {a: v.double() for a, v in i["params"]}
    rows = _net64(i["tokens"].transpose(0, 1), p, n, _mask(case["T"], True, window=case["window"])).transpose(0, 1)
    return {"logits": rows @ p["wa"] + p["ba"], "values": (rows @ p["wc"] + p["bc"])[..., 0], "actions": None}
