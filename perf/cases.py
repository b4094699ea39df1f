"""The work that a user of this package has it do, as cases that can be timed: the operators at the sizes of the benchmark's
configurations, the hybrid layers at the published head geometries in prefill, generation and training.

listed() names the cases, draw() gives more of the same ranges, prepare() makes what a program holds before the call, run() is
one pass through the public entry points, work() what a pass cannot do without, tolerance() how far two correct
implementations may differ.
"""
import math
from statistics import NormalDist

import torch
import torch.nn.functional as F

from neuralattentionsearchlinear_amd import nats_util
from neuralattentionsearchlinear_amd.cache import NAtSCache, NAtSMamba2Cache
from neuralattentionsearchlinear_amd.mixed_attn_gdn import nats_mixed_attn_gdn, nats_mixed_attn_gdn_recurrent
from neuralattentionsearchlinear_amd.mixed_attn_mamba import nats_mixed_attn_mamba, nats_mixed_attn_mamba_recurrent
from neuralattentionsearchlinear_amd.natsl_attn_gdn import NeuralAttentionSearchLinearAttnGDN
from neuralattentionsearchlinear_amd.natsl_attn_mamba2 import NeuralAttentionSearchLinearAttnMamba

DEV = "cuda:0"

# Layer geometries: the two published Gated DeltaNet configurations, and a Mamba2-SSD layer with the state and head widths of
# the benchmark's Mamba configuration.
GEOMETRY = {
    "gdn_340M": dict(hidden_size=1024, expand_v=2, head_dim=128, num_heads=6, num_attn_heads=12),
    "gdn_760M": dict(hidden_size=1536, expand_v=2, head_dim=192, num_heads=6, num_attn_heads=18),
    "mamba": dict(hidden_size=1024, expand_v=0.5, head_dim=128, num_heads=16, num_attn_heads=16),
}


def listed():
    return [
        # one token for each of eight sequences on cached states and keys: a serving loop's inner step, at the operator
        dict(name="decode_gdn_b8", task="decode", kind="gdn", B=8, ctx=8192, H=16, K=128, V=128, p_attn=0.25, block=64, n_in=17),
        # one user's answer through a layer: the prompt, then token by token (latency and launches count)
        dict(name="generate_gdn_340M_b1", task="generate", geometry="gdn_340M", B=1, T=777, new=32),
        # the same for a small batch on the Mamba layer, with a longer prompt
        dict(name="generate_mamba_b8", task="generate", geometry="mamba", B=8, T=2000, new=16),
        # the smallest configuration of the operator, in fp32: a unit test's or a notebook's call
        dict(name="forward_small_fp32", task="forward", kind="gdn", B=1, T=256, H=2, K=64, V=64, p_attn=0.5, block=64, dtype="float32",
             packed=False),
        # every block routed to the linear branch
        dict(name="forward_gdn_only", task="forward", kind="gdn", B=4, T=4096, H=16, K=128, V=128, p_attn=0.0, block=64, dtype="bfloat16",
             packed=False),
        # the headline shape
        dict(name="forward_headline", task="forward", kind="gdn", B=8, T=8192, H=16, K=128, V=128, p_attn=0.25, block=64, dtype="bfloat16",
             packed=False),
        # long context, four documents packed in one row
        dict(name="forward_packed_long", task="forward", kind="gdn", B=1, T=65536, H=32, K=128, V=128, p_attn=0.10, block=64,
             dtype="bfloat16", packed=True),
        # the Mamba2-SSD variant with its long selector blocks
        dict(name="forward_mamba", task="forward", kind="mamba", B=4, T=8192, H=32, K=128, V=64, p_attn=0.25, block=256, dtype="bfloat16",
             packed=False),
        # a batch of prompts through a layer into an empty cache, and the first token that is fed back
        dict(name="prefill_gdn_340M", task="prefill", geometry="gdn_340M", B=8, T=4096, new=1),
        # forward and backward of the Mamba operator
        dict(name="train_op_mamba", task="train_op", kind="mamba", B=4, T=8192, H=32, K=128, V=64, p_attn=0.25, block=256),
        # a training step's share of one layer at both published geometries, the second with sequences of an uneven length
        dict(name="train_layer_gdn_340M", task="train_layer", geometry="gdn_340M", B=8, T=4096),
        dict(name="train_layer_gdn_760M", task="train_layer", geometry="gdn_760M", B=2, T=3000),
    ]


def _log_int(rng, lo, hi):
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def _estimate(case):
    """A rough time in seconds, to keep drawn cases below the largest listed ones."""
    w = work(case)
    return w["flops"] / 3e14 + w["bytes"] / 1e12 + 7e-4 * case.get("new", 0)


def draw(rng):
    task = rng.choice(["decode", "generate", "forward", "forward", "prefill", "train_op", "train_layer"])
    odd = rng.random() < 0.5                            # a length that no tile or block divides, or a multiple of the block
    if task in ("decode", "forward", "train_op"):
        kind = rng.choice(["gdn", "gdn", "mamba"])
        case = dict(task=task, kind=kind, B=_log_int(rng, 1, 64 if task == "decode" else 16), H=rng.choice([2, 4, 6, 8, 12, 16, 24, 32]))
        case["K"], case["V"] = rng.choice([(64, 64), (128, 128), (128, 128), (128, 64), (64, 128)])
        case["p_attn"] = round(rng.uniform(0.05, 0.5), 3)
        case["block"] = rng.choice([64, 64, 64, 128, 256])
        if task == "decode":
            case["ctx"] = _log_int(rng, 256, 32768)
            case["n_in"] = rng.randrange(case["block"] - 1)
        else:
            T = _log_int(rng, 64, 65536)
            case["T"] = T if odd else max(1, T // case["block"]) * case["block"]
            if task == "forward":
                case["dtype"] = "float32" if rng.random() < 0.15 else "bfloat16"
                case["packed"] = kind == "gdn" and rng.random() < 0.25 and case["T"] >= 512
                if case["packed"]:
                    case["B"] = 1
    else:
        case = dict(task=task, geometry=rng.choice(sorted(GEOMETRY)), B=_log_int(rng, 1, 16))
        if task == "generate":
            case["T"], case["new"] = _log_int(rng, 64, 4096), rng.randint(4, 32)
        else:
            if task == "prefill":
                case["new"] = 1
            T = _log_int(rng, 128, 16384)
            case["T"] = T if odd else T // 64 * 64
    most = max(_estimate(c) for c in listed() if c["task"] == task)
    size = "ctx" if task == "decode" else "T"
    while _estimate(case) > most:                       # fewer sequences first, then shorter ones
        if case["B"] > 1:
            case["B"] = max(1, case["B"] // 2)
        else:
            case[size] = max(64, int(case[size] * 0.7)) if odd else max(case.get("block", 64), case[size] // 128 * 64)
    return case


# ---------------------------------------------------------------------------------------------------------------------------
def _selector_bias(p):
    """What is added to the linear op's logit so that attention wins with probability p between two N(0,1) logits."""
    return 30.0 if p <= 0.0 else -math.sqrt(2.0) * NormalDist().inv_cdf(p)


def _boundaries(case):
    """The packed sequences of a row of T tokens: eighths 1, 2, 2, 3 (uneven ones where T is)."""
    T = case["T"]
    return [0, T // 8, 3 * T // 8, 5 * T // 8, T]


def _n_blocks(case):
    if case.get("packed"):
        cu = _boundaries(case)
        return sum(-(-(b - a) // case["block"]) for a, b in zip(cu[:-1], cu[1:]))
    return -(-case["T"] // case["block"])


def _operator_inputs(case, g):
    B, T, H, K, V = (case[n] for n in ("B", "T", "H", "K", "V"))
    dt = getattr(torch, case.get("dtype", "bfloat16"))
    rn = lambda *s: torch.randn(*s, device=DEV, generator=g)
    s = {}
    if case["kind"] == "mamba":
        # B and C: one group shared by all heads; log-decay dt * A with dt = softplus(N(0,1) - 4), A = -exp(U(0, log 16)).  The
        # linear branch takes X * dt as its values, the attention branch X itself.
        s["q"] = rn(B, T, 1, K).to(dt).expand(B, T, H, K).contiguous()
        s["k"] = rn(B, T, 1, K).to(dt).expand(B, T, H, K).contiguous()
        x, step = rn(B, T, H, V), F.softplus(rn(B, T, H) - 4.0)
        s["g"] = -torch.exp(torch.rand(H, device=DEV, generator=g) * math.log(16.0)) * step
        s["v"], s["v_l"] = x.to(dt), (x * step[..., None]).to(dt)
        s["beta"] = None
    else:
        s["q"], s["k"], s["v"] = rn(B, T, H, K).to(dt), rn(B, T, H, K).to(dt), rn(B, T, H, V).to(dt)
        s["v_l"] = s["v"]
        s["beta"] = torch.sigmoid(rn(B, T, H)).to(dt)
        s["g"] = -F.softplus(rn(B, T, H))
    logits = rn(B, _n_blocks(case), H, 2)
    logits[..., 1] += _selector_bias(case["p_attn"])
    s["logits"] = logits.to(dt)
    return s


def _layer(case, seed):
    torch.manual_seed(seed)
    cfg = dict(GEOMETRY[case["geometry"]], nats_block_size=64, ops_for_incomplete_chunks="all", layer_idx=0)
    if case["geometry"] == "mamba":
        layer = NeuralAttentionSearchLinearAttnMamba(norm_eps=1e-5, decay_for_non_mamba_blocks=True, **cfg)
    else:
        layer = NeuralAttentionSearchLinearAttnGDN(norm_eps=1e-6, decay_for_non_gdn_blocks=True, **cfg)
    return layer.to(DEV).to(torch.bfloat16).train(case["task"] == "train_layer")


def prepare(case, seed):
    task = case["task"]
    g = torch.Generator(device=DEV).manual_seed(seed)
    rn = lambda *s: torch.randn(*s, device=DEV, generator=g)
    s = dict(case=case)
    if task == "decode":
        B, H, K, V = (case[n] for n in ("B", "H", "K", "V"))
        kept = max(1, int(case["ctx"] * case["p_attn"]) // case["block"])
        n_keys = kept * case["block"] + case["n_in"] + 1
        s.update(q=rn(B, 1, H, K).bfloat16(), k=rn(B, 1, H, K).bfloat16(), v=rn(B, 1, H, V).bfloat16(),
                 k_cache=rn(B, n_keys, H, K).bfloat16(), v_cache=rn(B, n_keys, H, V).bfloat16(),
                 state=rn(B, H, K, V) * 0.1, state0=rn(B, H, K, V) * 0.1, g=-F.softplus(rn(B, 1, H)),
                 g_cumsum=-torch.rand(B, H, device=DEV, generator=g) * 5, beta=torch.sigmoid(rn(B, 1, H)).bfloat16(),
                 types=torch.ones(B, 1, H, 2, device=DEV, dtype=torch.bfloat16))
        # every head keeps its own number of blocks, the fullest one all of them; then come the block's tokens
        own = torch.randint(kept // 2, kept + 1, (B, H, 1), device=DEV, generator=g)
        own[:, 0] = kept
        at = torch.arange(n_keys, device=DEV) // case["block"]
        s["mask"] = ((at < own) | (at == kept)).unsqueeze(2)
    elif task in ("forward", "train_op"):
        s.update(_operator_inputs(case, g))
        if case.get("packed"):
            cu = _boundaries(case)
            s["cu_seqlens"] = torch.tensor(cu, dtype=torch.int32, device=DEV)
            s["seqs"] = nats_util.pack_sequences(cu, None, case["block"], DEV)
        if task == "train_op":
            s["do_l"], s["do_a"] = rn(*s["v"].shape).bfloat16(), rn(*s["v"].shape).bfloat16()
            for n in ("q", "k", "v", "v_l", "beta", "g", "logits"):
                if s[n] is not None:
                    s[n].requires_grad_(True)
    else:
        s["layer"] = _layer(case, seed)
        hidden = GEOMETRY[case["geometry"]]["hidden_size"]
        s["x"] = rn(case["B"], case["T"], hidden).bfloat16()
        if task in ("generate", "prefill"):
            s["tokens"] = [rn(case["B"], 1, hidden).bfloat16() for _ in range(case["new"])]
        if task == "train_layer":
            s["x"].requires_grad_(True)
            s["do"] = rn(*s["x"].shape).bfloat16()
    return s


# ---------------------------------------------------------------------------------------------------------------------------
def _operator(s):
    case = s["case"]
    types, counts = nats_util.hard_select(s["logits"], force_last_block=True, seqs=s.get("seqs"))
    qkv = (s["q"], s["k"], s["v"], s["q"], s["k"], s["v_l"])
    if case["kind"] == "mamba":
        return nats_mixed_attn_mamba(*qkv, None, s["g"], types, counts, scale_lattn=1.0, nats_block_size=case["block"],
                                     ops_for_incomplete_chunks="all", output_final_state_mamba=True, decay_for_non_mamba_blocks=True,
                                     compute_dnats_for_invalid_blocks_linear_att=False)
    return nats_mixed_attn_gdn(*qkv, None, s["g"], s["beta"], types, counts, cu_seqlens=s.get("cu_seqlens"), nats_block_size=case["block"],
                               ops_for_incomplete_chunks="all", output_final_state_gated_delta=True, decay_for_non_gdn_blocks=True,
                               compute_dnats_for_invalid_blocks_linear_att=False)


def _decode(s):
    case = s["case"]
    common = dict(n_tokens_in_current_block=case["n_in"], nats_block_size=case["block"], ops_for_incomplete_chunks="all")
    if case["kind"] == "mamba":
        return nats_mixed_attn_mamba_recurrent(s["q"], s["k_cache"], s["v_cache"], s["q"], s["k"], s["v"], s["mask"], s["state"], s["state0"],
                                               s["g"], s["g_cumsum"], s["types"], scale_lattn=1.0, decay_for_non_mamba_blocks=True, **common)
    return nats_mixed_attn_gdn_recurrent(s["q"], s["k_cache"], s["v_cache"], s["q"], s["k"], s["v"], s["mask"], s["state"], s["state0"],
                                         s["g"], s["g_cumsum"], s["beta"], s["types"], decay_for_non_gdn_blocks=True, **common)


def _into_cache(s):
    """The prompt through the layer into an empty cache -> (outputs, the layer's cache, a call that feeds more tokens)."""
    if s["case"]["geometry"] == "mamba":
        holder = NAtSMamba2Cache()
        feed = lambda x: s["layer"](x, cache_params=holder, use_cache=True)
        o = feed(s["x"])
        return o, holder.nats_cache[0], feed
    holder = NAtSCache()
    feed = lambda x: s["layer"](x, past_key_values=holder, use_cache=True)[0]
    o = feed(s["x"])
    return o, holder[0], feed


def run(s):
    task = s["case"]["task"]
    if task == "train_op":
        leaves = [s[n] for n in ("q", "k", "v", "v_l", "beta", "g", "logits") if s[n] is not None]
        for t in leaves:
            t.grad = None
        o_l, o_a, state = _operator(s)
        torch.autograd.backward([o_l, o_a], [s["do_l"], s["do_a"]])
        return [o_l.detach(), o_a.detach(), state.detach()] + [t.grad for t in leaves if t.grad is not None]
    if task == "train_layer":
        s["x"].grad = None
        s["layer"].zero_grad(set_to_none=True)
        o = s["layer"](s["x"])
        o = o[0] if isinstance(o, tuple) else o
        o.backward(s["do"])
        return [o.detach(), s["x"].grad] + [p.grad for p in s["layer"].parameters()]
    with torch.no_grad():
        if task == "decode":
            return _decode(s)
        if task == "forward":
            return _operator(s)
        o, cache, feed = _into_cache(s)
        return [o] + [feed(t) for t in s["tokens"]] + [cache.recurrent_state, cache.n_attn_blocks]


# ---------------------------------------------------------------------------------------------------------------------------
def _branch_flops(kind, B, T, H, K, V, HA, KA, VA, p, block, sequences=1):
    """Operations of the two branches' forward: what the visible keys and the 64-token chunks need."""
    n, blocks = T / sequences, T / sequences / block
    pairs = sequences * (n * (block + 1) / 2 + p * block * block * blocks * max(0.0, blocks - 1) / 2)
    soft = 2.0 * (KA + VA) * B * HA * pairs
    C, chunks = 64, B * H * T / 64
    if kind == "gdn":
        lin = (2 * C * C * (3 * K + 2 * V) + 2.0 / 3.0 * C ** 3 + 6 * C * K * V) * chunks
    else:
        lin = (2 * C * C * (K + V) + 4 * C * K * V) * chunks
    return soft, lin


def work(case):
    task, B = case["task"], case["B"]
    if task == "decode":
        H, K, V = case["H"], case["K"], case["V"]
        n_keys = max(1, int(case["ctx"] * case["p_attn"]) // case["block"]) * case["block"] + case["n_in"] + 1
        return {"bytes": B * H * (K * V * 4 * 3 + n_keys * ((K + V) * 2 + 1) + (2 * K + 2 * V) * 2 * 2), "flops": B * H * (8 * K * V + 2 * n_keys * (K + V))}
    T = case["T"]
    if task in ("forward", "train_op"):
        H, K, V = case["H"], case["K"], case["V"]
        size = 4 if case.get("dtype") == "float32" else 2
        mamba = case["kind"] == "mamba"
        soft, lin = _branch_flops(case["kind"], B, T, H, K, V, H, K, V, case["p_attn"], case["block"], 4 if case.get("packed") else 1)
        values = 2 if mamba else 1                       # X and X * dt
        inputs = B * T * H * ((2 * K + values * V) * size + 4 + (0 if mamba else size))
        outputs = B * T * H * 2 * V * size + B * H * K * V * 4
        if task == "forward":
            return {"bytes": inputs + outputs, "flops": soft + lin}
        return {"bytes": 3 * inputs + 2 * outputs, "flops": 3.5 * soft + 3 * lin}
    geo = GEOMETRY[case["geometry"]]
    D, H, K, HA = geo["hidden_size"], geo["num_heads"], geo["head_dim"], geo["num_attn_heads"]
    V = int(K * geo["expand_v"])
    kind = "mamba" if case["geometry"] == "mamba" else "gdn"
    weights = D * (2 * H * K + 3 * H * V + 4 * H) + 2 * HA * H * K
    soft, lin = _branch_flops(kind, B, T, H, K, V, HA, H * K // HA, H * V // HA, 0.5, 64)
    dense = 2.0 * B * T * weights
    act = B * T * D * 2
    if task == "train_layer":
        return {"bytes": 3 * act + 4 * weights + act, "flops": 3 * dense + 3.5 * soft + 3 * lin}
    kept = B * T * H * (K + V)                           # half of the keys and values, bf16
    prefill = {"bytes": 2 * act + 2 * weights + kept + B * H * K * V * 4, "flops": dense + soft + lin}
    new = case["new"]
    per_token = 2 * weights + kept + B * H * K * V * 4 * 2
    return {"bytes": prefill["bytes"] + new * per_token, "flops": prefill["flops"] + new * (2.0 * B * weights + 8.0 * B * H * K * V + kept)}


def tolerance(case):
    """bf16 operands with fp32 sums: an output of one operator is within 3e-3 to 5e-3 of exact arithmetic, so two right ones are
    within 1e-2 of each other; a layer rounds to bf16 a few times more on the way, and a gradient passes twice the steps."""
    if case["task"] in ("decode", "forward"):
        return {"rel": 1e-2}
    return {"rel": 1.5e-2 if case["task"] in ("prefill", "generate") else 2e-2}
