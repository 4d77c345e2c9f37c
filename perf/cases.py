"""What is timed: the Gated DeltaNet and KDA operators as a model's layer calls them, from one decoded token to a long
training sequence.

Head counts: 16 q/k and 32 value heads of 128 are the layer's; with the heads sharded over P ranks each rank has
16/P and 32/P of them on the full sequence.  The smallest decode batches and short prompts are bound by latency, the
large ones by memory and matrix work."""
import math
import os
import sys

import torch

sys.path.insert(1, os.path.join(os.getcwd(), "mindspeed-mm_amd"))

import mindspeed_mm_amd as gdn  # noqa: E402

CONV_WIDTH = 4
CHUNK = 64
_DTYPES = {"bf16": torch.bfloat16, "fp32": torch.float32}


def _case(name, kind, B, T, Hqk, Hv, K=128, V=128, dtype="bf16", lengths="", keep=False, slow=False):
    """kind: decode (the layer's one-token step), prefill (the layer's chain without gradients), layer (the same chain
    forward and backward), rule (the chunked rule alone, forward and backward), kda (its sibling with one decay per key
    channel, forward and backward), kda_prefill.  lengths: packed sequences, comma-separated, "" for B rows of T tokens.
    keep: skip_recompute=True.  slow: slowly decaying heads (long memory)."""
    case = dict(kind=kind, B=B, T=T, Hqk=Hqk, Hv=Hv, K=K, V=V, dtype=dtype, lengths=lengths, keep=keep, slow=slow)
    return case if name is None else dict(case, name=name)


# 24 packed sequences of 172 to 4096 tokens, 32768 in all
_PACKED_24 = ("903,2685,209,241,441,1560,881,4096,772,1550,514,627,172,271,420,986,2016,3057,265,403,1890,4096,617,"
              "4096")


def listed():
    return [
        # one user's next token: two small launches, so latency and host work are all there is
        _case("decode_1", "decode", 1, 1, 16, 32),
        # a full serving batch: the fp32 states in and out
        _case("decode_256", "decode", 256, 1, 16, 32),
        # one short prompt, ragged
        _case("prefill_360", "prefill", 1, 360, 16, 32),
        # prompts of very different lengths packed into one row
        _case("prefill_packed_32832", "prefill", 1, 32832, 16, 32, lengths="14012,12588,6166,66"),
        # pretraining micro-batch, the forward workspace kept for the backward pass
        _case("rule_2x8192", "rule", 2, 8192, 16, 32, keep=True),
        # fine-tuning micro-batch of short samples, the operator's default call
        _case("rule_4x1024", "rule", 4, 1024, 16, 32),
        # a long sequence with the heads sharded over four ranks: few heads, many dependent chunks
        _case("rule_32768_4ranks", "rule", 1, 32768, 4, 8),
        # the largest: long context, wide value heads, slow decay
        _case("rule_65536_wide", "rule", 1, 65536, 16, 64, V=256, keep=True, slow=True),
        # the layer between its projections, trained on a packed batch
        _case("layer_packed_24", "layer", 1, 32768, 16, 32, lengths=_PACKED_24),
        # the linear-attention layer with one decay per key channel: training and a prompt
        _case("kda_2x8192", "kda", 2, 8192, 32, 32),
        _case("kda_prefill_4608", "kda_prefill", 1, 4608, 32, 32),
        # full precision, as numerical comparisons run it
        _case("rule_512_fp32", "rule", 1, 512, 4, 4, K=64, V=64, dtype="fp32"),
    ]


def _spread(rng, lo, hi):
    """A whole number spread evenly over the logarithm of [lo, hi]; odd as often as even."""
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def _lengths(rng, total):
    """Between 2 and 24 sequences of at least one token that add up to `total`."""
    n = rng.randint(2, min(24, max(2, total // 64)))
    cuts = sorted(rng.sample(range(1, total), n - 1))
    return ",".join(str(b - a) for a, b in zip([0] + cuts, cuts + [total]))


def draw(rng):
    kind = rng.choice(["decode", "decode", "prefill", "prefill", "rule", "rule", "rule", "layer", "kda", "kda_prefill",
                       "fp32"])
    ranks = rng.choice([1, 1, 2, 4, 8])
    Hqk, Hv = 16 // ranks, 32 // ranks
    if kind == "decode":
        return _case(None, kind, _spread(rng, 1, 256), 1, Hqk, Hv)
    if kind in ("prefill", "layer"):
        T = _spread(rng, 64 if kind == "prefill" else 512, 32768)
        return _case(None, kind, 1, T, Hqk, Hv, lengths=_lengths(rng, T) if T >= 128 and rng.random() < 0.5 else "")
    if kind == "rule":
        B = rng.choice([1, 1, 2, 4])
        T = _spread(rng, 256, 32768 // B)
        wide, expanded = rng.random() < 0.2, rng.random() < 0.25   # expanded: q, k already repeated to the value heads
        return _case(None, kind, B, T, Hv if expanded else Hqk, Hv, V=256 if wide else 128, keep=rng.random() < 0.5,
                     slow=rng.random() < 0.25, lengths=_lengths(rng, T) if B == 1 and rng.random() < 0.4 else "")
    if kind in ("kda", "kda_prefill"):
        B = rng.choice([1, 1, 2])
        T = _spread(rng, 128, 16384 // B)
        return _case(None, kind, B, T, Hv, Hv, lengths=_lengths(rng, T) if B == 1 and rng.random() < 0.3 else "")
    d = rng.choice([64, 128])
    return _case(None, "rule", rng.choice([1, 2]), _spread(rng, 64, 1024), rng.choice([2, 4]), 4, K=d, V=d, dtype="fp32")


def _sequences(case):
    return len(case["lengths"].split(",")) if case["lengths"] else case["B"]


def prepare(case, seed):
    dev = torch.device("cuda")
    gen = torch.Generator(device=dev).manual_seed(seed)
    B, T, Hqk, Hv, K, V = (case[n] for n in ("B", "T", "Hqk", "Hv", "K", "V"))
    N, kind, dt = _sequences(case), case["kind"], _DTYPES[case["dtype"]]
    D = 2 * Hqk * K + Hv * V
    a_log, bias = ((0.5, 2.0), (-6.0, -4.0)) if case["slow"] else ((1.0, 16.0), (-4.0, -2.0))

    def normal(*shape, std=1.0, dtype=dt):
        return (torch.randn(*shape, generator=gen, device=dev) * std).to(dtype)

    def uniform(n, lo, hi):
        return torch.rand(n, generator=gen, device=dev) * (hi - lo) + lo

    s = dict(case=case, cu=None)
    if case["lengths"]:
        cu = [0]
        for n in case["lengths"].split(","):
            cu.append(cu[-1] + int(n))
        s["cu"] = torch.tensor(cu, dtype=torch.int64, device=dev)
    A_log = uniform(Hv, math.log(a_log[0]), math.log(a_log[1]))
    if kind in ("decode", "prefill", "layer"):
        grad = kind == "layer"
        s["x"] = normal(B, T, D).requires_grad_(grad)
        s["a"], s["b"] = normal(B, T, Hv).requires_grad_(grad), normal(B, T, Hv).requires_grad_(grad)
        s["A_log"], s["dt_bias"] = A_log.requires_grad_(grad), uniform(Hv, *bias).requires_grad_(grad)
        taps = (CONV_WIDTH ** -0.5)
        if kind == "decode":
            s["conv_w"], s["conv_b"] = normal(D, CONV_WIDTH, std=taps), normal(D, std=0.1)
            s["conv_state"] = normal(B, D, CONV_WIDTH)
            s["state"] = normal(B, Hv, K, V, std=0.1, dtype=torch.float32)
            return s
        s["conv_w"] = normal(CONV_WIDTH, D, std=taps).requires_grad_(grad)
        s["conv_b"] = normal(D, std=0.1).requires_grad_(grad)
        s["z"] = normal(B, T, Hv, V).requires_grad_(grad)
        s["norm_w"] = (1 + normal(V, std=0.1, dtype=torch.float32)).to(dt).requires_grad_(grad)
        if grad:
            s["dy"] = normal(B, T, Hv, V)
        return s
    grad = kind != "kda_prefill"
    s["q"], s["k"] = normal(B, T, Hqk, K).requires_grad_(grad), normal(B, T, Hqk, K).requires_grad_(grad)
    s["v"] = normal(B, T, Hv, V).requires_grad_(grad)
    if kind == "rule":
        raw = normal(B, T, Hv, dtype=torch.float32) + uniform(Hv, *bias)
        s["g"] = (-A_log.exp() * torch.nn.functional.softplus(raw)).requires_grad_(grad)
        s["beta"] = torch.sigmoid(normal(B, T, Hv, dtype=torch.float32)).to(dt).requires_grad_(grad)
        s["h0"] = normal(N, Hv, K, V, std=0.02, dtype=torch.float32).requires_grad_(grad)
    else:
        s["g"], s["beta"] = normal(B, T, Hv, K).requires_grad_(grad), normal(B, T, Hv).requires_grad_(grad)
        s["A_log"], s["dt_bias"] = A_log.requires_grad_(grad), uniform(Hv * K, *bias).requires_grad_(grad)
        s["h0"] = normal(N, Hv, V, K, std=0.02, dtype=torch.float32).requires_grad_(grad)
    if grad:
        s["do"] = normal(B, T, Hv, V)
    return s


def _layer(s):
    """The layer between its input projections and its output projection."""
    c = s["case"]
    x, conv_state = gdn.causal_conv1d(s["x"], s["conv_w"], s["conv_b"], activation="silu", cu_seqlens=s["cu"],
                                      output_final_state=c["kind"] == "prefill")
    g, beta = gdn.gdn_gates(s["a"], s["b"], s["A_log"], s["dt_bias"])
    y, state = gdn.chunk_gated_delta_rule_qkv(x, g, beta, c["Hqk"], c["Hv"], c["K"], c["V"],
                                              output_final_state=c["kind"] == "prefill", use_qk_l2norm_in_kernel=True,
                                              cu_seqlens=s["cu"], gate=s["z"], norm_weight=s["norm_w"])
    return y, conv_state, state


def _kda(s):
    return gdn.chunk_kda(s["q"], s["k"], s["v"], s["g"], s["beta"], initial_state=s["h0"], output_final_state=True,
                         use_qk_l2norm_in_kernel=True, use_gate_in_kernel=True, use_beta_sigmoid_in_kernel=True,
                         transpose_state_layout=True, cu_seqlens=s["cu"], A_log=s["A_log"], dt_bias=s["dt_bias"])


def run(state):
    s, c = state, state["case"]
    kind = c["kind"]
    if kind == "decode":
        with torch.no_grad():
            o = gdn.decode_step(s["x"], s["a"], s["b"], s["conv_state"], s["state"], s["conv_w"], s["conv_b"], s["A_log"],
                                s["dt_bias"], c["Hqk"], c["Hv"], c["K"], c["V"])
        return o, s["conv_state"], s["state"]
    if kind == "prefill":
        with torch.no_grad():
            return _layer(s)
    if kind == "kda_prefill":
        with torch.no_grad():
            return _kda(s)
    if kind == "layer":
        y, _, ht = _layer(s)
        names, dy = ("x", "a", "b", "A_log", "dt_bias", "conv_w", "conv_b", "z", "norm_w"), s["dy"]
    elif kind == "rule":
        y, ht = gdn.chunk_gated_delta_rule(s["q"], s["k"], s["v"], s["g"], s["beta"], initial_state=s["h0"],
                                           output_final_state=True, use_qk_l2norm_in_kernel=True, cu_seqlens=s["cu"],
                                           skip_recompute=c["keep"])
        names, dy = ("q", "k", "v", "g", "beta", "h0"), s["do"]
    else:
        y, ht = _kda(s)
        names, dy = ("q", "k", "v", "g", "beta", "A_log", "dt_bias", "h0"), s["do"]
    return (y.detach(), None if ht is None else ht.detach(), *torch.autograd.grad([y], [s[n] for n in names], [dy]))


def work(case):
    """Matrix work by the chunked form's usual count (chunks of 64 tokens), backward twice the forward."""
    B, T, Hqk, Hv, K, V = (case[n] for n in ("B", "T", "Hqk", "Hv", "K", "V"))
    N, kind, tokens, es = _sequences(case), case["kind"], B * T, 2 if case["dtype"] == "bf16" else 4
    D, state = 2 * Hqk * K + Hv * V, 4 * N * Hv * K * V
    rule = 2 * tokens * Hv * (3 * V * CHUNK + 2 * K * CHUNK + 3 * K * V)
    conv = 2 * CONV_WIDTH * tokens * D
    if kind == "decode":
        return {"bytes": 2 * state + es * (B * (D + 2 * Hv + Hv * V + 2 * CONV_WIDTH * D) + (CONV_WIDTH + 1) * D),
                "flops": 6 * K * V * Hv * B + 2 * CONV_WIDTH * D * B}
    if kind == "prefill":   # in: conv input, gate projections, z; out: y and both states
        return {"bytes": es * tokens * (D + 2 * Hv + 2 * Hv * V) + state + es * N * D * CONV_WIDTH, "flops": rule + conv}
    if kind == "layer":     # in: the same and dy; out: y and a gradient for each input
        return {"bytes": es * tokens * (2 * D + 4 * Hv + 4 * Hv * V), "flops": 3 * (rule + conv)}
    if kind == "rule":      # in: q, k, v, g, beta, the state, do; out: o, the final state and a gradient for each input
        return {"bytes": tokens * (es * (4 * Hqk * K + 4 * Hv * V + 2 * Hv) + 8 * Hv) + 3 * state, "flops": 3 * rule}
    if kind == "kda_prefill":
        return {"bytes": es * tokens * Hv * (3 * K + 2 * V + 1) + 2 * state, "flops": rule}
    return {"bytes": es * tokens * Hv * (6 * K + 4 * V + 2) + 3 * state, "flops": 3 * rule}


# largest (rel, max) of any output: four times what the path differs by from itself run in float32 on the same values
# (float32: from the same rule in float64), capped where a sum over all tokens (the gradients of A_log and dt_bias) or an
# output that is small beside a sum it passed through (a gated row, a decay's gradient) would go beyond 0.03 and 0.9
_OFF = {"decode": (1e-2, 0.12), "prefill": (2e-2, 0.9), "rule": (2e-2, 0.25), "layer": (3e-2, 0.9), "kda": (3e-2, 0.9),
        "kda_prefill": (2e-2, 0.25)}


def tolerance(case):
    rel, most = _OFF[case["kind"]] if case["dtype"] == "bf16" else (5e-6, 5e-5)
    return {"rel": rel, "max": most}
