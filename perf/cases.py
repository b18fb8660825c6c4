"""The work that a serving program has this package do, as measurable cases: one pass through the public entry points each.

Four kinds of pass:
  step          one decode or verify step of the decoder stack for B sequences (two periods of its 3 GatedDeltaNet layers + 1
                attention layer, each with its MLP): what every generated token costs.  `graph`: the program has captured the
                step in a HIP graph, as the benchmark does, and replays it; otherwise it makes the calls each time
  prefill_gdn   the GatedDeltaNet layer core over the T tokens of a prompt
  prefill_attn  a full-attention layer over the S rows of a prompt (or of the part of it that follows `prefix` cached rows),
                between its qkv and o projections
  admit         a request whose prompt hits the prefix cache: lookup, restore, admission of the state into its slot

Sizes are those of the package's model configuration (qwen_tailor_amd.model.Cfg), its benchmark and its tests."""
from __future__ import annotations

import math

import numpy as np
import torch

import qwen_tailor_amd as qt

BF16 = torch.bfloat16
HV, DK, DV, CD, PW, QKV = 16, 128, 128, 6144, 8224, 5120
STEP_LAYERS = 8                    # two periods of the stack: their weights and state exceed the last-level cache, as the whole stack's do
EPS = 1e-6


def listed():
    return [
        # one user, one token: latency and the number of launches
        {"name": "step_b1", "kind": "step", "B": 1, "M": 1, "lo": 300, "hi": 301, "graph": True},
        # a few users with short contexts and three draft tokens each, launched eagerly (a batch whose make-up changes too often
        # to be captured)
        {"name": "step_b5_m3_eager", "kind": "step", "B": 5, "M": 3, "lo": 90, "hi": 900, "graph": False},
        # the benchmark's long-context batch
        {"name": "step_b16_long", "kind": "step", "B": 16, "M": 1, "lo": 512, "hi": 32768, "graph": True},
        # the benchmark's speculative batch
        {"name": "step_b16_m4", "kind": "step", "B": 16, "M": 4, "lo": 1024, "hi": 8192, "graph": True},
        # the benchmark's full batch, chat-length contexts
        {"name": "step_b64", "kind": "step", "B": 64, "M": 1, "lo": 200, "hi": 2000, "graph": True},
        # a short question, an ordinary prompt, a long document
        {"name": "prefill_gdn_61", "kind": "prefill_gdn", "T": 61},
        {"name": "prefill_gdn_2048", "kind": "prefill_gdn", "T": 2048},
        {"name": "prefill_gdn_8192", "kind": "prefill_gdn", "T": 8192},
        # the next turn of a conversation, an ordinary prompt, a long document
        {"name": "prefill_attn_333_on_1500", "kind": "prefill_attn", "S": 333, "prefix": 1500},
        {"name": "prefill_attn_2048", "kind": "prefill_attn", "S": 2048, "prefix": 0},
        {"name": "prefill_attn_8192", "kind": "prefill_attn", "S": 8192, "prefix": 0},
        # a cached system prompt and a cached turn, admitted into a slot of 4096 positions
        {"name": "admit_2048", "kind": "admit", "pos": 2048, "max_len": 4096},
    ]


def _log(rng, lo, hi):
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    kind = rng.choice(["step", "step", "prefill_gdn", "prefill_attn", "admit"])
    if kind == "step":
        M = rng.choice([1, 1, 1, 2, 3, 4, 5])
        B = _log(rng, 1, 64 if M == 1 else 16)
        hi = _log(rng, 64, min(32768, 17 * 32768 // (B + 1)))
        if M > 1:
            hi = min(hi, 17 * 8192 // (B + 1))
        return {"kind": kind, "B": B, "M": M, "lo": max(1, int(hi * rng.uniform(0.02, 0.7))), "hi": hi, "graph": rng.random() < 0.7}
    if kind == "prefill_gdn":
        return {"kind": kind, "T": _log(rng, 17, 8192)}
    if kind == "prefill_attn":
        S = _log(rng, 17, 8192)
        return {"kind": kind, "S": S, "prefix": rng.choice([0, _log(rng, 64, 8192)]) if S <= 2048 else 0}
    pos = _log(rng, 64, 4096)
    return {"kind": kind, "pos": pos, "max_len": rng.choice([m for m in (512, 2048, 4096) if m >= pos])}


# ---- what a program has in hand ---------------------------------------------------------------------------------------

def _randn(gen, shape, scale=1.0, dtype=BF16):
    return torch.empty(shape, dtype=dtype, device="cuda").normal_(0.0, scale, generator=gen)


def _near_one(gen, n):
    return (1.0 + _randn(gen, (n,), 0.1, torch.float32)).to(BF16)


def _gdn_params(gen):
    return {"cw": _randn(gen, (CD, 4, 1), 0.5), "A_log": torch.empty(HV, device="cuda").uniform_(0.0, 2.7, generator=gen),
            "dtb": _randn(gen, (HV,), 0.1, torch.float32), "gw": 1.0 + _randn(gen, (DV,), 0.1, torch.float32)}


def _prepare_step(case, gen):
    cfg = qt.model.Cfg(layers=STEP_LAYERS)
    B, M, lo, hi = case["B"], case["M"], case["lo"], case["hi"]
    H, I = cfg.hidden, cfg.inter
    branch = (2 * qt.model.Cfg().layers) ** -0.5                  # the residual stream dominates what one layer adds to it
    layers = []
    for i in range(cfg.layers):
        p = {"linear": cfg.is_linear(i), "ln1": _near_one(gen, H), "ln2": _near_one(gen, H),
             "gate_up": _randn(gen, (2 * I, H), H ** -0.5), "down": _randn(gen, (H, I), branch * I ** -0.5)}
        if p["linear"]:
            p.update(_gdn_params(gen), w_in=_randn(gen, (PW, H), H ** -0.5), w_out=_randn(gen, (H, HV * DV), branch * (HV * DV) ** -0.5))
        else:
            p.update(w_in=_randn(gen, (QKV, H), H ** -0.5), w_out=_randn(gen, (H, 2048), branch * 2048 ** -0.5), q_norm=_near_one(gen, 256),
                     k_norm=_near_one(gen, 256))
        layers.append(p)
    P = qt.batch.Pools(cfg, B, hi + 16)
    slots = torch.randperm(B, generator=gen, device="cuda").to(torch.int32)
    pos = torch.randint(lo, max(hi, lo + 1), (B,), generator=gen, device="cuda").to(torch.int32)
    s = {"case": case, "layers": layers, "P": P, "slots": slots, "pos": pos, "x": _randn(gen, (B * M, H))}
    R = P
    if M > 1:
        s["SP"] = R = qt.batch_spec.SpecPools(cfg, B, B, M, hi + 16)
        s["sels"] = torch.randint(0, M, (B,), generator=gen, device="cuda").to(torch.int32)
        s["pars"] = torch.randint(0, 2, (B,), generator=gen, device="cuda").to(torch.int32)
    if case["graph"]:
        side = torch.cuda.Stream()
        side.wait_stream(torch.cuda.current_stream())
        with torch.cuda.stream(side):
            _step(s)                                              # once outside the capture: tables and scratch buffers exist
            side.synchronize()
            s["graph"] = torch.cuda.CUDAGraph()
            with torch.cuda.graph(s["graph"], stream=side):
                s["out"] = _step(s)
        torch.cuda.current_stream().wait_stream(side)
    # the state goes in last: the step above has run on empty pools
    for pool in P.K + P.V:
        pool.normal_(0.0, 1.0, generator=gen)
    for conv, ssm in zip(R.conv, R.ssm):
        conv.normal_(0.0, 1.0, generator=gen)
        ssm.normal_(0.0, 0.02, generator=gen)
    return s


def _prepare_prefill_gdn(case, gen):
    T = case["T"]
    return dict(_gdn_params(gen), case=case, proj=_randn(gen, (T, PW)), conv=_randn(gen, (1, 3, CD)),
                ssm=_randn(gen, (1, HV, DV, DK), 0.02, torch.float32))


def _prepare_prefill_attn(case, gen):
    S, prefix = case["S"], case["prefix"]
    max_len = prefix + S + 64                                     # room for the answer
    return {"case": case, "qkv": _randn(gen, (S, QKV)), "q_norm": _near_one(gen, 256), "k_norm": _near_one(gen, 256),
            "K": _randn(gen, (1, 2, max_len, 256)), "V": _randn(gen, (1, 2, max_len, 256)),
            "pos": torch.full((1,), prefix, dtype=torch.int32, device="cuda")}


def _prepare_admit(case, gen):
    cfg = qt.model.Cfg()
    pos, max_len = case["pos"], case["max_len"]
    nl = sum(cfg.is_linear(i) for i in range(cfg.layers))
    st = {"kv": [(_randn(gen, (1, cfg.n_kv, pos, 256)), _randn(gen, (1, cfg.n_kv, pos, 256))) for _ in range(cfg.layers - nl)],
          "conv": [_randn(gen, (1, 3, CD)) for _ in range(nl)],
          "ssm": [_randn(gen, (1, HV, DV, DK), 0.02, torch.float32) for _ in range(nl)]}
    ids = np.arange(pos + 100, dtype=np.int32)                    # the prompt: the cached rows and a new question
    cache = qt.prefix_cache.PrefixCache(budget_mb=4096)
    head = cache.insert(None, ids, max(1, pos // 3), st)          # a system prompt ...
    cache.insert(head, ids, pos, st)                              # ... and the conversation so far
    return {"case": case, "cache": cache, "ids": ids, "P": qt.batch.Pools(cfg, 4, max_len), "slot": 2}


def prepare(case, seed):
    gen = torch.Generator(device="cuda").manual_seed(int(seed))
    return {"step": _prepare_step, "prefill_gdn": _prepare_prefill_gdn, "prefill_attn": _prepare_prefill_attn,
            "admit": _prepare_admit}[case["kind"]](case, gen)


# ---- one pass ---------------------------------------------------------------------------------------------------------

def _step(s):
    M, P, slots, pos, x = s["case"]["M"], s["P"], s["slots"], s["pos"], s["x"]
    gemv = qt.kernels.fused_gemv
    R = P if M == 1 else s["SP"]
    lin = att = 0
    for p in s["layers"]:
        proj = gemv(p["w_in"], x, nw=p["ln1"])
        if p["linear"]:
            if M == 1:
                o = qt.batch.deltanet_b_gnorm(proj, P.conv[lin], p["cw"], p["A_log"], p["dtb"], P.ssm[lin], slots, pos, p["gw"])
            else:
                y = qt.batch_spec.deltanet_bm(proj, R.conv[lin], p["cw"], p["A_log"], p["dtb"], R.ssm[lin], slots, s["sels"], s["pars"], M)
                o = qt.batch.gnorm_rows(y, proj, p["gw"])
            lin += 1
        else:
            o = qt.batch.attn_layer_b(proj, p["q_norm"], p["k_norm"], P.K[att], P.V[att], slots, pos, M)
            att += 1
        x = gemv(p["w_out"], o, res=x)
        x = gemv(p["down"], gemv(p["gate_up"], x, nw=p["ln2"], swiglu=True), res=x)
    return {"x": x, "conv": R.conv, "ssm": R.ssm, "K": P.K, "V": P.V}


def _run_step(s):
    if not s["case"]["graph"]:
        return _step(s)
    s["graph"].replay()
    return s["out"]


def _run_prefill_gdn(s):
    return qt.prefill.gdn_core(s["proj"], s["conv"], s["ssm"], s["cw"], s["A_log"], s["dtb"], s["gw"])


def _run_prefill_attn(s):
    S, at = s["case"]["S"], s["case"]["prefix"]
    n, K, V, qkv = at + S, s["K"], s["V"], s["qkv"]
    q, k, v = qt.attention.qkv_prep(qkv, s["q_norm"], s["k_norm"], s["pos"], M=S, max_pos=n)
    K[0, :, at:n], V[0, :, at:n] = k.transpose(0, 1), v.transpose(0, 1)
    o = qt.attention.scaled_dot_product_attention(q.transpose(0, 1)[None], K[:, :, :n], V[:, :, :n], scale=256 ** -0.5, mask="causal")
    return {"o": qt.attention.out_gate(o[0].transpose(0, 1).contiguous(), qkv), "K": K, "V": V}


def _run_admit(s):
    node, _ = s["cache"].lookup(s["ids"])
    st, _ = s["cache"].restore(node, s["case"]["max_len"])
    s["P"].load(s["slot"], st, node.pos)
    return s["P"].as_tree()


def run(state):
    return {"step": _run_step, "prefill_gdn": _run_prefill_gdn, "prefill_attn": _run_prefill_attn, "admit": _run_admit}[state["case"]["kind"]](state)


# ---- what a pass cannot do without ------------------------------------------------------------------------------------

def work(case):
    cfg = qt.model.Cfg()
    H, I = cfg.hidden, cfg.inter
    if case["kind"] == "step":
        B, M = case["B"], case["M"]
        R, mean = B * M, (case["lo"] + max(case["hi"], case["lo"] + 1) - 1) / 2
        lin, att = STEP_LAYERS * 3 // 4, STEP_LAYERS // 4
        w = STEP_LAYERS * 3 * I * H + lin * (PW + HV * DV) * H + att * (QKV + 2048) * H
        state = HV * DV * DK * 4
        gdn = B * ((1 + M) * state + (1 + M) * 3 * CD * 2) + CD * 4 * 2
        kv = B * mean * 2 * 2 * 256 * 2
        return {"bytes": w * 2 + lin * gdn + att * kv + 2 * R * H * 2,
                "flops": 2.0 * R * w + lin * R * HV * 6.0 * DV * DK + att * 4.0 * R * 8 * 256 * mean}
    if case["kind"] == "prefill_gdn":
        T = case["T"]
        return {"bytes": T * (PW + HV * DV) * 2 + 2 * (HV * DV * DK * 4 + 3 * CD * 2), "flops": 2621440.0 * T}
    if case["kind"] == "prefill_attn":
        S, prefix = case["S"], case["prefix"]
        return {"bytes": S * (QKV + 2048) * 2 + S * 1024 * 2 + prefix * 1024 * 2, "flops": 4.0 * 8 * 256 * (S * prefix + S * (S + 1) / 2)}
    nl = sum(cfg.is_linear(i) for i in range(cfg.layers))
    rec, row = nl * (HV * DV * DK * 4 + 3 * CD * 2), (cfg.layers - nl) * 2 * 2 * 256 * 2
    return {"bytes": 3 * rec + row * (2 * case["pos"] + case["max_len"]), "flops": 0.0}     # cache -> fresh state -> slot


def tolerance(case):
    if case["kind"] == "admit":
        return "exact"
    # bf16 outputs of eight layers.  A sum taken in another order moves single bf16 roundings, which the following layers carry
    # on: the step with its products summed by another fp32 matrix product differs by 4.2e-3 .. 7.2e-3, largest 0.157
    if case["kind"] == "step":
        return {"rel": 2.8e-2, "max": 0.6}
    # half-precision operands inside the chunked form: the sequential form of the same layer differs by 1.47e-3, largest 0.0148
    if case["kind"] == "prefill_gdn":
        return {"rel": 6e-3, "max": 6e-2}
    # bf16 outputs of an attention in fp32 differ by 2.7e-3, largest 0.030
    return {"rel": 1e-2, "max": 0.12}
