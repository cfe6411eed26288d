"""Performance cases of the FP8 expert path and the operators around it.

A case is a dict of plain values; ``kind`` names the part of a training program it stands for:

  experts     stage 3 of a MoE layer (group rows by expert, gate/up, activation, down, un-permute),
              forward and backward, the weights quantised in the pass as after every optimizer step
  operators   the same layer spelled with the single operators (scatter, three grouped linears,
              ``silu_mul``, gather), which is what a program gets that swaps only the imports
  block       a whole MoE block: router gate, experts, shared experts, weighted sum; training
              (forward and backward) or evaluation (forward only, quantised weights kept)
  ep_rank     one rank of an expert-parallel group: dispatch indices and the gather of the rows to
              send, stage 3 on deduplicated received rows, weighted combine of the returned rows
  linear      a dense FP8 linear of the decoder layer, forward and backward
  mla         FP8 decompression of an MLA latent block and its backward
  loss        the loss head: cross-entropy on the logits, forward and backward

Sizes are those of the repository's benchmark workloads and tests, or lie between them.
"""

import math

import torch

from pith_train_amd.dualpipe_utils import FP8WeightCacheControl
from pith_train_amd.modules.experts import DeepSeekV2Experts, GptOssExperts, Qwen3MoeExperts, Qwen35MoeExperts, forward_stage3
from pith_train_amd.modules.moe import DeepSeekV2MoE, GptOssMoE, Qwen3MoeMoE, Qwen35MoeSparseMoeBlock
from pith_train_amd.operators.cross_entropy import cross_entropy
from pith_train_amd.operators.deepgemm_quantize import fp8cast_blockwise_transpose
from pith_train_amd.operators.ep_dispatch import adjust_expand_idx, build_expert_idxs, fused_dedup_prepare_dispatch
from pith_train_amd.operators.linear import FP8Linear
from pith_train_amd.operators.mla_decompress import mla_decompress, mla_decompress_backward
from pith_train_amd.operators.moe_combine import moe_combine_ep
from pith_train_amd.operators.silu_mul import silu_mul
from pith_train_amd.operators.token_scatter import padded_index_gather, precompute_group_indices, scatter_for_grouped_gemm

BF16 = torch.bfloat16


# ------------------------------------------------------------------------------------------------
# the cases
# ------------------------------------------------------------------------------------------------
def listed():
    return [
        # the toy layer of the tests: a step of some twenty launches, bound by latency and host work
        dict(name="experts_toy", kind="experts", model="qwen3", hidden=256, inter=512, experts=8, top_k=2, tokens=1024, zipf=0.0, dedup=0.0),
        # the headline workload: a Qwen3-30B-A3B layer, fused gate/up weight, 8192 tokens
        dict(name="experts_qwen3", kind="experts", model="qwen35", hidden=2048, inter=768, experts=128, top_k=8, tokens=8192, zipf=0.0, dedup=0.0),
        # a GPT-OSS-20B layer: biases, clamped SwiGLU, widths that are no multiple of 128
        dict(name="experts_gpt_oss", kind="experts", model="gpt_oss", hidden=2880, inter=2880, experts=32, top_k=4, tokens=16384, zipf=0.0, dedup=0.0),
        # the largest: a 32k-token layer whose routed rows re-use a quarter of the received rows
        dict(name="experts_dedup_32k", kind="experts", model="qwen35", hidden=2048, inter=768, experts=128, top_k=8, tokens=32768, zipf=0.0, dedup=0.25),
        # a drop-in user's layer: every operator by itself, the group sizes read back to the host
        dict(name="operators_qwen3", kind="operators", hidden=2048, inter=768, experts=64, top_k=8, tokens=4096, zipf=0.0),
        # a DeepSeek-V2-Lite block in training: skewed routing (idle and crowded experts), shared experts
        dict(name="block_dsv2_lite", kind="block", model="dsv2", hidden=2048, inter=1408, experts=64, top_k=6, tokens=8192, zipf=1.2, train=True),
        # an evaluation batch of odd length through a Qwen3 block: few rows per expert, forward only
        dict(name="block_qwen3_eval", kind="block", model="qwen3", hidden=2048, inter=768, experts=128, top_k=8, tokens=333, zipf=0.0, train=False),
        # one rank of eight in an expert-parallel group
        dict(name="ep_rank_qwen3", kind="ep_rank", hidden=2048, inter=768, experts=128, top_k=8, tokens=4096, ranks=8),
        # the query projection of the 32k-token decoder layer
        dict(name="linear_q_32k", kind="linear", fin=2048, fout=4096, tokens=32768),
        # a key/value projection on a short batch of odd length
        dict(name="linear_kv_odd", kind="linear", fin=2048, fout=512, tokens=1001),
        # one 4096-row latent block of DeepSeek-V2-Lite's attention
        dict(name="mla_block", kind="mla", batch=1, rows=4096, heads=16, nope=128, vdim=128, rank=512),
        # the loss head on 4096 rows of a 151 936-entry vocabulary
        dict(name="loss_head", kind="loss", tokens=4096, vocab=151936, dtype="bfloat16"),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    """One more case: the kind at random, token counts over the logarithm of their range, widths and
    expert counts from what the model families use."""
    kind = rng.choice(["experts", "experts", "experts", "operators", "block", "block", "ep_rank", "linear", "linear", "mla", "loss"])
    if kind == "linear":
        fin, fout = rng.choice([(2048, 4096), (2048, 512), (4096, 2048), (2048, 2816), (2816, 2048), (2880, 4096), (512, 4096), (1024, 1536)])
        return dict(kind=kind, fin=fin, fout=fout, tokens=_log_int(rng, 128, 32768))
    if kind == "mla":
        heads, nope, rank = rng.choice([16, 4]), rng.choice([128, 64]), rng.choice([512, 256])
        return dict(kind=kind, batch=rng.choice([1, 2]), rows=_log_int(rng, 256, 4096) // 16 * 16, heads=heads, nope=nope, vdim=nope, rank=rank)
    if kind == "loss":
        return dict(kind=kind, tokens=_log_int(rng, 256, 4096), vocab=rng.choice([32000, 50257, 151936, 201088]), dtype=rng.choice(["bfloat16", "bfloat16", "float32"]))
    while True:
        hidden, inter, experts, top_k = rng.choice([
            (256, 512, 8, 2), (1024, 512, 32, 4), (2048, 768, 128, 8), (2048, 768, 64, 8), (2048, 768, 16, 8),
            (2048, 1408, 64, 6), (2048, 512, 128, 8), (2880, 2880, 32, 4), (2880, 2880, 8, 4), (1536, 1024, 16, 2)])
        tokens = _log_int(rng, 96, 16384)
        zipf = rng.choice([0.0, 0.0, 1.2])
        if kind == "experts":
            model = "gpt_oss" if hidden == 2880 else rng.choice(["qwen3", "qwen35", "dsv2"])
            dedup = rng.choice([0.0, 0.0, 0.25]) if model != "gpt_oss" else 0.0
            return dict(kind=kind, model=model, hidden=hidden, inter=inter, experts=experts, top_k=top_k, tokens=tokens, zipf=zipf, dedup=dedup)
        if kind == "operators" and hidden != 2880:
            return dict(kind=kind, hidden=hidden, inter=inter, experts=experts, top_k=top_k, tokens=tokens, zipf=zipf)
        if kind == "block":
            model = "gpt_oss" if hidden == 2880 else rng.choice(["qwen3", "dsv2", "qwen35"])
            return dict(kind=kind, model=model, hidden=hidden, inter=inter, experts=experts, top_k=top_k, tokens=tokens, zipf=zipf, train=rng.random() < 0.6)
        if kind == "ep_rank" and hidden != 2880:
            ranks = rng.choice([2, 4, 8])
            return dict(kind=kind, hidden=hidden, inter=inter, experts=experts, top_k=top_k, tokens=min(tokens, 8192), ranks=ranks)


# ------------------------------------------------------------------------------------------------
# inputs and weights
# ------------------------------------------------------------------------------------------------
class _Draw:
    """Seeded values on the GPU: activations and gradients ~ N(0, 1), weights ~ N(0, 0.02)."""

    def __init__(self, seed):
        self.g = torch.Generator(device="cuda").manual_seed(seed)

    def normal(self, *shape, std=1.0, dtype=BF16):
        return torch.empty(shape, device="cuda", dtype=dtype).normal_(0.0, std, generator=self.g)

    def fill(self, module):
        with torch.no_grad():
            for p in module.parameters():
                p.normal_(0.0, 0.02, generator=self.g)
        return module

    def popularity(self, experts, zipf):
        """Router bias of every expert: zero, or the centred log-probabilities of a Zipf ranking,
        steep enough that some experts get nothing and some several times the mean."""
        if not zipf:
            return torch.zeros(experts, device="cuda")
        ranks = torch.randperm(experts, device="cuda", generator=self.g).float() + 1.0
        logp = -1.5 * zipf * ranks.log()
        return logp - logp.mean()

    def routing(self, tokens, experts, top_k, zipf=0.0):
        logits = torch.randn((tokens, experts), device="cuda", generator=self.g) + self.popularity(experts, zipf)
        return torch.topk(logits.softmax(-1), k=top_k, dim=-1)


    def limited_routing(self, tokens, experts, top_k, ranks, per_token):
        """Top-k within the ``per_token`` ranks that score highest for a token (group-limited
        routing), at least one expert on each of them."""
        logits = torch.randn((tokens, ranks, experts // ranks), device="cuda", generator=self.g)
        best = logits.max(-1)
        chosen = torch.zeros((tokens, ranks), device="cuda").scatter_(1, best.values.topk(per_token, dim=1).indices, 1.0)
        first = torch.nn.functional.one_hot(best.indices, experts // ranks)
        key = (logits + 100.0 * first + 1000.0 * chosen.unsqueeze(-1)).view(tokens, experts)
        idx = key.topk(top_k, dim=-1).indices
        return idx, logits.view(tokens, experts).softmax(-1).gather(1, idx)


def _ranks_per_token(case):
    """Ranks that hold one of a token's experts, as many as evenly spread choices would reach."""
    n, k = case["ranks"], case["top_k"]
    return min(n, k, round(n * (1 - (1 - 1 / n) ** k)))


def _on_gpu(make):
    with torch.device("cuda"):
        return make().to(BF16)


def _experts(case):
    make = {"qwen3": Qwen3MoeExperts, "dsv2": DeepSeekV2Experts, "qwen35": Qwen35MoeExperts, "gpt_oss": GptOssExperts}[case["model"]]
    return _on_gpu(lambda: make(case["hidden"], case["inter"], case["experts"]))


def _block(case):
    H, I, E, k = case["hidden"], case["inter"], case["experts"], case["top_k"]
    if case["model"] == "qwen3":
        return _on_gpu(lambda: Qwen3MoeMoE(H, I, E, k))
    if case["model"] == "dsv2":
        return _on_gpu(lambda: DeepSeekV2MoE(H, I, E, k, n_shared_experts=2))
    if case["model"] == "qwen35":
        return _on_gpu(lambda: Qwen35MoeSparseMoeBlock(H, I, E, k, I))
    return _on_gpu(lambda: GptOssMoE(H, I, E, k))


def prepare(case, seed):
    """Inputs, weights and upstream gradients of one pass."""
    kind, d = case["kind"], _Draw(seed)
    s = {"case": case}
    if kind in ("experts", "operators"):
        T, k, E, H = case["tokens"], case["top_k"], case["experts"], case["hidden"]
        rows = T * k
        s["experts"] = d.fill(_experts(case if kind == "experts" else dict(case, model="qwen3")))
        s["expert_idxs"] = d.routing(T, E, k, case["zipf"]).indices.reshape(-1)
        s["expand_idx"] = None
        if case.get("dedup"):
            # the received rows are unique; every one is used at least once, the rest are repeats
            unique = rows - int(rows * case["dedup"])
            again = torch.randint(0, unique, (rows - unique,), device="cuda", generator=d.g)
            idx = torch.cat([torch.arange(unique, device="cuda"), again])
            s["expand_idx"] = idx[torch.randperm(rows, device="cuda", generator=d.g)]
            s["tokens"] = d.normal(unique, H)
        else:
            s["tokens"] = d.normal(T, H).repeat_interleave(k, dim=0)
        s["grad"] = d.normal(rows, H)
    elif kind == "block":
        T, H = case["tokens"], case["hidden"]
        s["block"] = d.fill(_block(case))
        gate = s["block"].router if case["model"] == "gpt_oss" else s["block"].gate
        with torch.no_grad():
            # hidden states share a direction; the router's weights along it make experts popular
            gate.weight[:, 0] = d.popularity(case["experts"], case["zipf"]) / 4.0
        s["hidden"] = d.normal(T, H)
        s["hidden"][:, 0] += 4.0
        s["grad"] = d.normal(T, H)
    elif kind == "ep_rank":
        T, k, E, H, n = case["tokens"], case["top_k"], case["experts"], case["hidden"], case["ranks"]
        local = E // n
        s["experts"] = d.fill(_on_gpu(lambda: Qwen3MoeExperts(H, case["inter"], local)))
        s["residual"], s["grad"] = d.normal(T, H), d.normal(T, H)
        u = _ranks_per_token(case)
        s["topk_idx"], s["topk_weight"] = d.limited_routing(T, E, k, n, u)
        # what rank 0 receives from every rank: unique token rows, rows per local expert, and the
        # unique row of each of them (every unique row is used at least once)
        rows_each, unique_each = T * k // n, T * u // n
        owner = torch.randint(0, local, (n, rows_each), device="cuda", generator=d.g)
        s["recv_counts"] = torch.nn.functional.one_hot(owner, local).sum(1).reshape(-1)
        s["recv_unique"] = torch.full((n,), unique_each, device="cuda")
        again = torch.randint(0, unique_each, (n, rows_each - unique_each), device="cuda", generator=d.g)
        expand = torch.cat([torch.arange(unique_each, device="cuda").expand(n, -1), again], dim=1)
        order = torch.rand(n, rows_each, device="cuda", generator=d.g).argsort(dim=1)
        s["recv_expand"] = expand.gather(1, order).reshape(-1)
        s["recv_tokens"] = d.normal(n * unique_each, H)
        s["recv_grad"] = d.normal(n * rows_each, H)
        # expert outputs that come back for this rank's own rows, and the gradient of what it sent
        s["returned"] = d.normal(T * k, H)
        s["sent_grad"] = d.normal(T * u, H)
    elif kind == "linear":
        s["linear"] = d.fill(_on_gpu(lambda: FP8Linear(case["fin"], case["fout"], bias=False)))
        s["x"], s["grad"] = d.normal(case["tokens"], case["fin"]), d.normal(case["tokens"], case["fout"])
    elif kind == "mla":
        b, n, h, dk, dv, r = (case[x] for x in ("batch", "rows", "heads", "nope", "vdim", "rank"))
        s["weight"] = d.normal(h * (dk + dv), r, std=0.02)
        s["quantised"] = fp8cast_blockwise_transpose(s["weight"])  # once per micro-batch, kept over the ring's hops
        s["latent"] = d.normal(b, n, r)
        s["grad_k"], s["grad_v"] = d.normal(b, n, h, dk), d.normal(b, n, h, dv)
    else:
        T, V = case["tokens"], case["vocab"]
        s["logits"] = d.normal(T, V, std=2.0, dtype=getattr(torch, case["dtype"]))
        s["target"] = torch.randint(0, V, (T,), device="cuda", generator=d.g)
        s["target"][torch.rand(T, device="cuda", generator=d.g) < 0.02] = -100
    return s


# ------------------------------------------------------------------------------------------------
# one pass
# ------------------------------------------------------------------------------------------------
def _fresh(module):
    """The start of a step: weights changed by the optimizer, gradients cleared."""
    FP8WeightCacheControl.step()
    module.zero_grad(set_to_none=True)


def _backward(out, x, grad, module):
    """Gradients of ``x`` and of every parameter.  Grouped weights get theirs written to ``.grad`` by
    the weight-gradient GEMM; the others, and ``x``, are taken from autograd (``x`` is an inner
    tensor of a training program, not a leaf that accumulates)."""
    names, params = zip(*module.named_parameters())
    gx, *gp = torch.autograd.grad(out, [x, *params], grad, allow_unused=True)
    return {"out": out.detach(), "grad_x": gx, **{n: p.grad if g is None else g for n, p, g in zip(names, params, gp)}}


def run(state):
    case = state["case"]
    kind = case["kind"]
    if kind == "experts":
        m = state["experts"]
        _fresh(m)
        x = state["tokens"].detach().requires_grad_(True)
        out = forward_stage3(m, x, state["expert_idxs"], case["experts"], expand_idx=state["expand_idx"])
        return _backward(out, x, state["grad"], m)
    if kind == "operators":
        m = state["experts"]
        _fresh(m)
        x = state["tokens"].detach().requires_grad_(True)
        rows, reverse, offs, ks, ks_tensor = scatter_for_grouped_gemm(x, state["expert_idxs"], case["experts"])
        kw = dict(grouped_mm_offs=offs, ks=ks, ks_tensor=ks_tensor, group_indices=precompute_group_indices(offs, rows.shape[0]))
        out = padded_index_gather(m.down_proj(silu_mul(m.gate_proj(rows, **kw), m.up_proj(rows, **kw)), **kw), reverse)
        return _backward(out, x, state["grad"], m)
    if kind == "block":
        m = state["block"]
        if not case["train"]:
            with torch.no_grad():
                return m.reference_forward(state["hidden"])
        _fresh(m)
        x = state["hidden"].detach().requires_grad_(True)
        return _backward(m.reference_forward(x), x, state["grad"], m)
    if kind == "ep_rank":
        return _run_ep_rank(case, state)
    if kind == "linear":
        m = state["linear"]
        _fresh(m)
        x = state["x"].detach().requires_grad_(True)
        return _backward(m(x), x, state["grad"], m)
    if kind == "mla":
        w_fp8, w_scale, w_t_fp8, w_t_scale = state["quantised"]
        k_nope, value = mla_decompress(state["latent"], state["weight"], case["heads"], case["nope"], case["vdim"], use_fp8=True,
                                       weight_fp8=w_fp8, scale_weight=w_scale)
        d_latent, d_weight = mla_decompress_backward(state["grad_k"], state["grad_v"], state["latent"], w_t_fp8, w_t_scale)
        return k_nope, value, d_latent, d_weight
    # the loss overwrites the logits, which the head's GEMM writes anew in every step: a copy stands for it
    logits = state["logits"].clone().requires_grad_(True)
    loss = cross_entropy(logits, state["target"])
    (grad,) = torch.autograd.grad(loss * 0.125, logits)  # 0.125: an eighth of the step, as with eight micro-batches
    return loss.detach(), grad


def _run_ep_rank(case, s):
    E, n = case["experts"], case["ranks"]
    local = E // n
    m = s["experts"]
    _fresh(m)
    # stage 1: index construction and the rows to send
    hidden = s["residual"].detach().requires_grad_(True)
    per_rank, unique, send_idx, slots, expand, meta = fused_dedup_prepare_dispatch(s["topk_idx"], E, n, local)
    counts = s["recv_counts"]
    expert_idxs, splits = build_expert_idxs(counts, n, local, case["tokens"] * case["top_k"] * n)
    unique_host, splits_host = unique.tolist(), splits.tolist()  # the all-to-all's split sizes
    sent = padded_index_gather(hidden, send_idx[: sum(unique_host)])
    # stage 3 on what the other ranks sent
    expand_idx = adjust_expand_idx(s["recv_expand"], s["recv_unique"], splits)
    recv = s["recv_tokens"].detach().requires_grad_(True)
    out = forward_stage3(m, recv, expert_idxs[: sum(splits_host)], local, expand_idx=expand_idx)
    # stage 5 on what they returned
    returned, weight = s["returned"].detach().requires_grad_(True), s["topk_weight"].detach().requires_grad_(True)
    combined = moe_combine_ep(returned, slots, weight, hidden)
    grad_returned, grad_weight, grad_residual = torch.autograd.grad(combined, [returned, weight, hidden], s["grad"])
    stage3 = _backward(out, recv, s["recv_grad"], m)
    (grad_hidden,) = torch.autograd.grad(sent, hidden, s["sent_grad"])
    return {**stage3, "combined": combined.detach(), "sent": sent.detach(), "per_rank": per_rank, "slots": slots, "expand": expand, "meta": meta,
            "expand_idx": expand_idx, "grad_returned": grad_returned, "grad_weight": grad_weight, "grad_residual": grad_residual,
            "grad_hidden": grad_hidden}


# ------------------------------------------------------------------------------------------------
# what a pass cannot do without, and how close results have to be
# ------------------------------------------------------------------------------------------------
def work(case):
    """Inputs read once, outputs written once; multiply-adds of the linear maps, padding not counted."""
    kind = case["kind"]
    if kind == "linear":
        T, a, b = case["tokens"], case["fin"], case["fout"]
        return {"bytes": 2 * (2 * T * a + 2 * T * b + 2 * a * b), "flops": 6 * T * a * b}
    if kind == "mla":
        T, r, o = case["batch"] * case["rows"], case["rank"], case["heads"] * (case["nope"] + case["vdim"])
        return {"bytes": 2 * (2 * T * r + 2 * T * o) + 2 * r * o + 4 * (T * r + r * o), "flops": 6 * T * r * o}
    if kind == "loss":
        size = 2 if case["dtype"] == "bfloat16" else 4
        return {"bytes": 2 * size * case["tokens"] * case["vocab"] + 8 * case["tokens"], "flops": 0}
    T, k, E, H, I = (case[x] for x in ("tokens", "top_k", "experts", "hidden", "inter"))
    if kind in ("experts", "operators"):
        rows = T * k
        unique = rows - int(rows * case.get("dedup", 0.0))
        return {"bytes": 2 * (2 * 3 * E * H * I + 2 * rows * H + 2 * unique * H) + 8 * rows, "flops": 18 * rows * H * I}
    if kind == "ep_rank":
        n = case["ranks"]
        rows = T * k
        unique = T * _ranks_per_token(case)
        nbytes = 2 * (2 * 3 * (E // n) * H * I + 2 * rows * H + 2 * unique * H)  # stage 3
        nbytes += 2 * (2 * rows * H + 4 * T * H) + 2 * 2 * unique * H + 8 * (4 * rows)  # combine, sent rows, indices
        return {"bytes": nbytes, "flops": 18 * rows * H * I}
    # block: the routed weights, the dense ones, the hidden states
    shared = {"dsv2": 2 * I, "qwen35": I}.get(case["model"], 0)
    weights = 3 * E * H * I + 3 * H * shared + E * H
    macs = 3 * T * k * H * I + 3 * T * H * shared + T * E * H
    if not case["train"]:
        return {"bytes": 2 * (2 * T * H) + 3 * E * H * I + 3 * H * shared + 2 * E * H, "flops": 2 * macs}  # weights kept as FP8 bytes
    return {"bytes": 2 * (4 * T * H + 2 * weights), "flops": 6 * macs}


def tolerance(case):
    if case["kind"] == "loss":
        # one rounding of the logits' type per entry, 32-bit sums for the loss
        return {"rel": 4e-3, "max": 1.6e-2} if case["dtype"] == "bfloat16" else {"rel": 1e-5, "max": 1e-4}
    # bf16 results of sums over FP8 products; an intermediate one bf16 step apart may be quantised to the
    # neighbouring FP8 value; index outputs are whole numbers and the same
    return {"rel": 1e-2, "max": 1e-1}
