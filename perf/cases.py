"""The work that users of this framework have it do, as measurable cases.

An actor or critic update meets the framework at five places, and each is a ``kind`` of case here:

* ``score``: log-probs and entropies of a micro-batch under ``no_grad`` (``compute_log_prob`` of the old and the
  reference policy), through ``linear_cross_entropy``;
* ``train``: the same with gradients to the hidden states and the weight (``update_policy``); with ``prompt`` > 0 the
  loss masks that share of every sequence out, so its upstream gradients are zero;
* ``rows``: log-probs and entropies of logits that a model without the fused head has materialised, with gradients;
* ``actor``: GRPO advantages of a batch, then the policy loss, the entropy bonus and the KL loss with one backward;
* ``ppo``: GAE with whitening, then the clipped value loss and the clipped policy loss, each with its backward;
* ``stats``: what the driver computes on a whole batch between rollout and update: KL-penalised rewards, the rollout
  correction's token weights and diagnostics, and the data metrics.

Token counts are those of micro-batches: one short response up to the 16384 tokens of the benchmark (``score`` somewhat
more, as no gradient is held).  Head shapes are those of the benchmark's three models.  Batches are ``rows`` responses
padded to ``cols`` tokens, lengths uniform.
"""
from __future__ import annotations

import math

import numpy as np
import torch

from verl_amd.trainer.ppo import core_algos, metric_utils, ray_trainer, rollout_corr_helper
from verl_amd.utils import torch_functional
from verl_amd.utils.kernel.linear_cross_entropy import linear_cross_entropy

# (hidden_size, vocab) of the benchmark's heads: Qwen2.5-0.5B, Qwen2.5-7B, Llama-3-8B
HEADS = ((896, 151936), (3584, 152064), (4096, 128256))
MASKS = {"int64": torch.int64, "bool": torch.bool, "float32": torch.float32}
GROUP = 8   # responses per prompt


def listed():
    return [
        # one short response of an evaluation or a straggler micro-batch: the whole weight is read for 93 tokens
        _score("score_one_response", 93, HEADS[0]),
        # the forward-only benchmark: log-probs of a 2048-token micro-batch of the small model
        _score("score_small_model", 2048, HEADS[0]),
        # a dynamic micro-batch filled up to a token budget, so its total is no multiple of anything; sampling temperature
        _score("score_token_budget", 21503, HEADS[2], 0.7),
        # one response of average length in an update with a micro-batch of one, small model
        _train("train_one_response", 777, HEADS[0]),
        # the headline benchmark: forward and backward at the 7B head with a full 16384-token micro-batch
        _train("train_full_batch", 16384, HEADS[1]),
        # an update on packed prompt + response sequences: a third of the tokens is prompt and carries no gradient
        _train("train_with_prompts", 11290, HEADS[1], seqs=9, prompt=0.35),
        # the default model path without the fused head: materialised bf16 logits of one 3000-token micro-batch
        {"name": "rows_bf16", "kind": "rows", "tokens": 3001, "vocab": 152064, "dtype": "bfloat16"},
        # the losses of one micro-batch of eight short responses: launches and host work
        _actor("actor_micro_batch", 8, 513),
        # the GRPO benchmark configuration
        _actor("actor_grpo_batch", 512, 4096, mask="float32"),
        # long reasoning responses padded to the longest of the batch, an odd length
        _actor("actor_long_responses", 1000, 11999),
        # the PPO benchmark configuration
        {"name": "ppo_batch", "kind": "ppo", "rows": 512, "cols": 4096, "mask": "float32"},
        # the driver's bookkeeping for one training step
        {"name": "step_statistics", "kind": "stats", "rows": 1024, "cols": 3072, "prompt_cols": 512, "mask": "int64"},
    ]


def _score(name, tokens, head, temperature=1.0):
    return {"name": name, "kind": "score", "tokens": tokens, "hidden": head[0], "vocab": head[1],
            "temperature": temperature}


def _train(name, tokens, head, temperature=1.0, seqs=1, prompt=0.0):
    return {"name": name, "kind": "train", "tokens": tokens, "hidden": head[0], "vocab": head[1],
            "temperature": temperature, "seqs": seqs, "prompt": prompt}


def _actor(name, rows, cols, loss="vanilla", agg="token-mean", mask="int64"):
    return {"name": name, "kind": "actor", "rows": rows, "cols": cols, "loss": loss, "agg": agg, "mask": mask}


def _log_int(rng, low, high):
    return int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))


def draw(rng):
    kind = rng.choice(("score", "score", "train", "train", "train", "rows", "actor", "actor", "ppo", "stats"))
    if kind in ("score", "train"):
        hidden, vocab = rng.choice(HEADS)
        case = {"kind": kind, "tokens": _log_int(rng, 64, 22000 if kind == "score" else 16000), "hidden": hidden,
                "vocab": vocab, "temperature": rng.choice((1.0, 1.0, 0.7))}
        if kind == "train":
            with_prompts = rng.random() < 0.4
            case["seqs"] = max(1, case["tokens"] // rng.randint(500, 3000))
            case["prompt"] = round(rng.uniform(0.1, 0.6), 3) if with_prompts else 0.0
        return case
    if kind == "rows":
        dtype = rng.choice(("bfloat16", "bfloat16", "float32"))
        return {"kind": kind, "tokens": _log_int(rng, 64, 3000 if dtype == "bfloat16" else 1500),
                "vocab": rng.choice(HEADS)[1], "dtype": dtype}
    cols = _log_int(rng, 256, 12000)
    rows = GROUP * _log_int(rng, 1, max(1, min(256, 9_000_000 // (GROUP * cols))))
    case = {"kind": kind, "rows": rows, "cols": cols, "mask": rng.choice(tuple(MASKS))}
    if kind == "actor":
        case["loss"] = rng.choice(("vanilla", "vanilla", "vanilla", "gspo", "cispo", "geo_mean"))
        case["agg"] = rng.choice(("token-mean", "token-mean", "seq-mean-token-mean", "seq-mean-token-sum-norm"))
    elif kind == "stats":
        case["prompt_cols"] = rng.randint(32, 1024)
    return case


class _Config:
    """The fields of the actor configuration that the losses read."""

    clip_ratio = 0.2
    clip_ratio_low = None
    clip_ratio_high = None
    global_batch_info: dict = {}

    def get(self, key, default=None):
        return getattr(self, key, default)


class _Batch:
    """The two fields of the trainer's batch object that the driver-side functions read."""

    def __init__(self, batch):
        self.batch = batch
        self.non_tensor_batch = {}


def _prompt_spans(case):
    """[start, end) of the prompt part of every packed sequence."""
    n, seqs = case["tokens"], case["seqs"]
    starts = [n * i // seqs for i in range(seqs + 1)]
    return [(a, a + int((b - a) * case["prompt"])) for a, b in zip(starts, starts[1:])]


def prepare(case, seed):
    dev = torch.device("cuda")
    g = torch.Generator(device=dev).manual_seed(seed)
    normal = lambda *shape: torch.randn(shape, generator=g, device=dev)
    kind = case["kind"]
    if kind in ("score", "train"):
        n, h, v = case["tokens"], case["hidden"], case["vocab"]
        s = {"hidden": normal(n, h).bfloat16(), "weight": (normal(v, h) * 0.02).bfloat16(),
             "labels": torch.randint(0, v, (n,), generator=g, device=dev)}
        if kind == "train":
            s["hidden"].requires_grad_()
            s["weight"].requires_grad_()
            s["g_logprobs"] = normal(n)
            s["g_entropy"] = torch.full((n,), 0.001, device=dev)
            for a, b in _prompt_spans(case):
                s["g_logprobs"][a:b] = 0.0
                s["g_entropy"][a:b] = 0.0
    elif kind == "rows":
        n, v = case["tokens"], case["vocab"]
        s = {"logits": (normal(n, v) * 1.5).to(getattr(torch, case["dtype"])).requires_grad_(),
             "labels": torch.randint(0, v, (n,), generator=g, device=dev), "g_logprobs": normal(n),
             "g_entropy": torch.full((n,), 0.001, device=dev)}
    else:
        s = _batch_state(case, g, dev, normal)
    s["case"] = case
    return s


def _batch_state(case, g, dev, normal):
    B, L, kind = case["rows"], case["cols"], case["kind"]
    lens = torch.randint(min(64, L), L + 1, (B,), generator=g, device=dev)
    mask = torch.arange(L, device=dev)[None, :] < lens[:, None]
    s = {"mask": mask.to(MASKS[case["mask"]])}
    at_end = torch.zeros((B, L), device=dev)
    every = torch.arange(B, device=dev)
    old = normal(B, L) * 0.5 - 1
    new = old + normal(B, L) * 0.05
    if kind == "actor":
        at_end[every, lens - 1] = torch.randint(0, 2, (B,), generator=g, device=dev).float()
        names = [f"prompt-{int(i)}" for i in torch.randint(0, 1 << 30, (B // GROUP,), generator=g, device=dev)]
        s.update(rewards=at_end, uid=np.array([x for x in names for _ in range(GROUP)], dtype=object), old=old,
                 new=new.requires_grad_(), ref=new.detach() + normal(B, L) * 0.1,
                 entropy=(normal(B, L) * 0.3 + 1).abs().requires_grad_(), config=_Config())
    elif kind == "ppo":
        at_end[every, lens - 1] = normal(B)
        values = normal(B, L)
        s.update(rewards=at_end, values=values, vpreds=(values + normal(B, L) * 0.4).requires_grad_(), old=old,
                 new=new.requires_grad_(), config=_Config())
    else:
        at_end[every, lens - 1] = normal(B)
        prompt = torch.ones((B, case["prompt_cols"]), dtype=torch.bool, device=dev)
        attention = torch.cat((prompt, mask), dim=1).to(torch.int64)
        s["data"] = _Batch({"response_mask": s["mask"], "attention_mask": attention, "token_level_scores": at_end,
                            "responses": torch.zeros((B, L), dtype=torch.int64, device=dev), "old_log_probs": old,
                            "ref_log_prob": old + normal(B, L) * 0.1, "rollout_log_probs": new,
                            "advantages": normal(B, L), "returns": normal(B, L), "values": normal(B, L)})
        s["kl"] = core_algos.FixedKLController(0.05)
    return s


def run(state):
    return _RUN[state["case"]["kind"]](state)


def _run_score(s):
    with torch.no_grad():
        return linear_cross_entropy(s["hidden"], s["weight"], s["labels"], s["case"]["temperature"])


def _run_train(s):
    logprobs, entropy = linear_cross_entropy(s["hidden"], s["weight"], s["labels"], s["case"]["temperature"])
    grads = torch.autograd.grad((logprobs, entropy), (s["hidden"], s["weight"]), (s["g_logprobs"], s["g_entropy"]))
    return logprobs.detach(), entropy.detach(), *grads


def _run_rows(s):
    logprobs = torch_functional.logprobs_from_logits(s["logits"], s["labels"], inplace_backward=False)
    entropy = torch_functional.entropy_from_logits(s["logits"])
    (d,) = torch.autograd.grad((logprobs, entropy), (s["logits"],),
                               (s["g_logprobs"].to(logprobs.dtype), s["g_entropy"].to(entropy.dtype)))
    return logprobs.detach(), entropy.detach(), d


def _run_actor(s):
    case = s["case"]
    advantages, _ = core_algos.compute_grpo_outcome_advantage(s["rewards"], s["mask"], s["uid"])
    loss_fn = core_algos.get_policy_loss_fn(case["loss"])
    pg_loss, metrics = loss_fn(s["old"], s["new"], advantages, s["mask"], case["agg"], s["config"])
    entropy_loss = core_algos.agg_loss(s["entropy"], s["mask"], case["agg"])
    kl_loss = core_algos.compute_kl_loss(s["new"], s["ref"], s["mask"], "low_var_kl", case["agg"])
    loss = pg_loss - 0.001 * entropy_loss + 0.001 * kl_loss
    d_logprob, d_entropy = torch.autograd.grad(loss, (s["new"], s["entropy"]))
    return advantages, pg_loss.detach(), metrics, entropy_loss.detach(), kl_loss.detach(), d_logprob, d_entropy


def _run_ppo(s):
    advantages, returns = core_algos.compute_gae_advantage_return(s["rewards"], s["values"], s["mask"], 1.0, 0.95)
    vf_loss, vf_clipfrac = core_algos.compute_value_loss(s["vpreds"], returns, s["values"], s["mask"], 0.5)
    (d_vpreds,) = torch.autograd.grad(vf_loss, (s["vpreds"],))
    pg_loss, metrics = core_algos.compute_policy_loss_vanilla(s["old"], s["new"], advantages, s["mask"], "token-mean",
                                                              s["config"])
    (d_logprob,) = torch.autograd.grad(pg_loss, (s["new"],))
    return (advantages, returns, vf_loss.detach(), vf_clipfrac.detach(), d_vpreds, pg_loss.detach(), metrics,
            d_logprob)


def _run_stats(s):
    data = s["data"]
    b = data.batch
    data, kl_metrics = ray_trainer.apply_kl_penalty(data, s["kl"], "low_var_kl")
    weights, mask, is_metrics = rollout_corr_helper.compute_rollout_correction_and_rejection_mask(
        b["old_log_probs"], b["rollout_log_probs"], b["response_mask"], rollout_is="token", rollout_is_threshold=2.0)
    metrics = metric_utils.compute_data_metrics(data, use_critic=True)
    return (b["token_level_rewards"], weights.batch["rollout_is_weights"], mask, kl_metrics, is_metrics, metrics)


_RUN = {"score": _run_score, "train": _run_train, "rows": _run_rows, "actor": _run_actor, "ppo": _run_ppo,
        "stats": _run_stats}


def work(case):
    kind = case["kind"]
    if kind == "score":
        n, h, v = case["tokens"], case["hidden"], case["vocab"]
        return {"bytes": 2 * h * (n + v) + 16 * n, "flops": 2 * n * v * h}
    if kind == "train":   # the two gradient products only need the tokens that carry a gradient
        n, h, v = case["tokens"], case["hidden"], case["vocab"]
        active = n - sum(b - a for a, b in _prompt_spans(case))
        return {"bytes": 4 * h * (n + v) + 24 * n, "flops": 2 * n * v * h + 4 * active * v * h}
    if kind == "rows":
        n, v = case["tokens"], case["vocab"]
        return {"bytes": 2 * n * v * getattr(torch, case["dtype"]).itemsize + 24 * n, "flops": 8 * n * v}
    m = MASKS[case["mask"]].itemsize
    BL = case["rows"] * case["cols"]
    if kind == "actor":   # in: rewards, mask, old, new, ref, entropy; out: advantages, two gradients
        return {"bytes": BL * (5 * 4 + m + 3 * 4), "flops": 40 * BL}
    if kind == "ppo":     # in: rewards, values, vpreds, old, new, mask; out: advantages, returns, two gradients
        return {"bytes": BL * (5 * 4 + m + 4 * 4), "flops": 40 * BL}
    # in: scores, old, ref, rollout, advantages, returns, values, both masks; out: rewards, weights
    return {"bytes": BL * (7 * 4 + m + 8 + 2 * 4) + 8 * case["rows"] * case["prompt_cols"], "flops": 40 * BL}


def tolerance(case):
    """About four times what the path differs by from the same mathematics in 64 bits (relative 2-norm error, largest
    error) at sizes up to 2048 tokens and 512 x 4096."""
    kind = case["kind"]
    if kind == "score":    # fp32 outputs: 0.9e-7, 3.5e-7
        return {"rel": 4e-7, "max": 2e-6}
    if kind == "train":    # gradients in bf16, d_logits rounded to bf16 on the way: 2.4e-3, 4.7e-2
        return {"rel": 1e-2, "max": 0.2}
    if kind == "rows":     # outputs in the dtype of the logits: bf16 1.4e-3, 6e-3; fp32 0.7e-7, 1.6e-6
        return {"rel": 6e-3, "max": 2.4e-2} if case["dtype"] == "bfloat16" else {"rel": 4e-7, "max": 6e-6}
    if kind == "actor":    # per token 2e-7; the policy loss is what is left of advantages that cancel: 6e-6
        return {"rel": 3e-5, "max": 3e-5}
    if kind == "ppo":      # per token 2e-7, 1.5e-6; whitened advantages cancel to a policy loss near zero: 3.5e-4
        return {"rel": 1.5e-3, "max": 1.5e-3}
    # per token 1e-7, 4e-7; a difference of perplexities near zero: 2.7e-4
    return {"rel": 1e-3, "max": 1e-3}
