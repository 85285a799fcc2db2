"""The workloads by which the speed of this package is judged.

Each case is one pass through the public entry points the way a trainer calls them: scoring responses with the fused
head, the head as a plain autograd function, the per-micro-batch step from the final hidden states on, the registry
losses and advantage estimators with the sampler correction in front of them, and the log-probabilities of
materialised logits.  Head shapes (hidden x vocabulary) are those of ``bench.py`` and of the workload descriptions in
``axon_amd/workloads.py``, or generic ones; sequence lengths follow the log-normal law of ``workloads.ragged_lengths``
unless a case says otherwise.  All inputs are synthetic and made on the GPU from the seed.
"""

from __future__ import annotations

import math
import random

import numpy as np
import torch

from axon_amd.models.fused_head_loss import fused_head_loss
from axon_amd.protocol import DataProto
from axon_amd.trainer.algos.advantages import compute_advantage
from axon_amd.trainer.algos.loss import compute_loss_fn
from axon_amd.utils.kernel.linear_cross_entropy import linear_cross_entropy
from axon_amd.utils.torch.ops import logprobs_and_entropy_from_logits

# hidden, vocabulary: the three head shapes of bench.py, then generic ones (a power-of-two vocabulary, one that is a
# multiple of 8 only, one that is odd)
HEADS = ((896, 151936), (2880, 201088), (4096, 151936), (2048, 32768), (3072, 128264), (1024, 50257))

# What a case may cost: the work of the largest listed one.
MAX_FLOPS = 6.0 * 32768 * 4096 * 151936
MAX_TOKENS_ELEMENTWISE = 1 << 23


def listed():
    return [
        # One short response scored again by the trainer (old / reference log-probs of a single sequence): the
        # smallest call of the head, forward only.
        dict(name="score_one_sequence", kind="score", tokens=187, hidden=896, vocab=151936, temperature=1.0,
             softcap=0.0, label_bits=64),
        # The old-log-prob pass over one micro-batch of the small head shape, forward only.
        dict(name="score_micro_batch", kind="score", tokens=8192, hidden=896, vocab=151936, temperature=0.7,
             softcap=0.0, label_bits=32),
        # The head as a plain autograd function on a ragged batch whose token count is odd: log-probs and entropy
        # forward, both gradients backward (what a caller with a loss of their own does).
        dict(name="head_autograd_ragged", kind="head", tokens=3001, hidden=2880, vocab=201088, temperature=1.0,
             softcap=0.0, label_bits=64),
        # A gradient-accumulation micro-batch of one prompt's few short responses through the large head: PPO.
        dict(name="step_short", kind="step", loss="ppo", tokens=700, hidden=4096, vocab=151936, side=False,
             correction=False, prompt=0.3, mask_bits=64),
        # The sequence-level loss on a ragged micro-batch of the small head, sampler correction in front.
        dict(name="step_gspo_ragged", kind="step", loss="gspo", tokens=6007, hidden=896, vocab=151936, side=False,
             correction=True, prompt=0.3, mask_bits=64),
        # DAPO (clip-higher) with entropy bonus and KL penalty on the large-vocabulary head; the token count is what
        # the sequences happen to add up to.
        dict(name="step_dapo_side_terms", kind="step", loss="dapo", tokens=16381, hidden=2880, vocab=201088, side=True,
             correction=False, prompt=0.0, mask_bits=32),
        # The headline micro-batch: GRPO advantage, PPO loss, 32768 packed tokens, the largest head.
        dict(name="step_ppo_large", kind="step", loss="ppo", tokens=32768, hidden=4096, vocab=151936, side=False,
             correction=False, prompt=0.0, mask_bits=32),
        # Loss-only GRPO step on the padded layout, 16 groups x 8 samples x 1024 tokens: the smallest elementwise call.
        dict(name="loss_padded", kind="loss", layout="padded", rows=128, length=1024, advantage="grpo", loss="ppo",
             correction="none", mask_bits=64),
        # Sampler-trainer correction with veto and GSPO on one packed micro-batch.
        dict(name="correction_gspo", kind="loss", layout="packed", tokens=65536, advantage="grpo", loss="gspo",
             correction="token_veto", mask_bits=32),
        # A whole global batch at once: sequence-level weights and geometric rejection, all diagnostics, then PPO.
        dict(name="correction_ppo_global_batch", kind="loss", layout="packed", tokens=8388607, advantage="grpo",
             loss="ppo", correction="sequence_geometric", mask_bits=32),
        # Actor-critic: GAE with whitening and the clipped value loss over a batch of responses.
        dict(name="gae_value", kind="value", tokens=2097149, mask_bits=32),
        # Materialised logits (the branch without fused kernels): log-prob and entropy forward, gradient backward.
        dict(name="logits_grad", kind="logits", tokens=2047, vocab=151936, bits=16),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    """One more case of the ranges above; token counts are spread over their logarithm and mostly odd."""
    kind = rng.choice(("score", "score", "head", "step", "step", "step", "loss", "loss", "loss", "value", "logits"))
    if kind in ("score", "head", "step"):
        hidden, vocab = rng.choice(HEADS)
        per_token = (2.0 if kind == "score" else 6.0) * hidden * vocab
        tokens = min(_log_int(rng, 64, 32768), int(0.9 * MAX_FLOPS / per_token))
        if kind == "step":
            return dict(kind=kind, loss=rng.choice(("ppo", "gspo", "dapo", "cispo", "reinforce")), tokens=tokens,
                        hidden=hidden, vocab=vocab, side=rng.random() < 0.4, correction=rng.random() < 0.4,
                        prompt=rng.choice((0.0, 0.3)), mask_bits=rng.choice((32, 64)))
        return dict(kind=kind, tokens=tokens, hidden=hidden, vocab=vocab, temperature=rng.choice((1.0, 0.7, 1.3)),
                    softcap=rng.choice((0.0, 0.0, 0.0, 30.0)), label_bits=rng.choice((32, 64)))
    mask_bits = rng.choice((32, 64))
    if kind == "loss":
        loss = rng.choice(("ppo", "gspo", "dapo", "cispo", "reinforce", "geo_mean"))
        advantage = rng.choice(("grpo", "rloo"))
        correction = rng.choice(("none", "token_veto", "sequence_geometric"))
        if rng.random() < 0.4:
            rows = 8 * rng.randint(2, 64)
            length = _log_int(rng, 100, min(8192, MAX_TOKENS_ELEMENTWISE // rows))
            return dict(kind=kind, layout="padded", rows=rows, length=length, advantage=advantage, loss=loss,
                        correction=correction, mask_bits=mask_bits)
        return dict(kind=kind, layout="packed", tokens=_log_int(rng, 2000, 8000000), advantage=advantage, loss=loss,
                    correction=correction, mask_bits=mask_bits)
    if kind == "value":
        return dict(kind=kind, tokens=_log_int(rng, 2000, 4000000), mask_bits=mask_bits)
    vocab = rng.choice((151936, 201088, 32768, 128264, 50257))
    return dict(kind=kind, tokens=_log_int(rng, 32, 4096), vocab=vocab, bits=rng.choice((16, 16, 32)))


# --------------------------------------------------------------------------------------------------------------
# inputs
# --------------------------------------------------------------------------------------------------------------

def _rand(seed):
    return torch.Generator(device="cuda").manual_seed(seed), random.Random(seed)


def _lengths(total, r, lo=32, hi=8192):
    """Log-normal sequence lengths that add up to ``total``."""
    lens, left = [], total
    while left > 0:
        x = min(max(int(round(math.exp(r.gauss(6.5, 0.8)))), lo), hi)
        if left - x < lo:
            x = left if left <= hi else left // 2
        lens.append(x)
        left -= x
    return lens


def _labels_of(rows, r, group=8):
    """One label per prompt, shared by its samples (the trainer's are random hexadecimal strings)."""
    names = ["%032x" % r.getrandbits(128) for _ in range(-(-rows // group))]
    return np.array([names[i // group] for i in range(rows)], dtype=object)


def _mask(m, bits):
    return m.to(torch.int64) if bits == 64 else m.to(torch.float32)


def _randn(g, *shape):
    return torch.randn(*shape, generator=g, device="cuda")


def _head_weights(g, tokens, hidden, vocab):
    h = _randn(g, tokens, hidden).to(torch.bfloat16)
    w = torch.empty(vocab, hidden, device="cuda", dtype=torch.bfloat16).normal_(0.0, 0.02, generator=g)
    return h, w


def _ids(g, tokens, vocab, bits):
    return torch.randint(0, vocab, (tokens,), generator=g, device="cuda", dtype=torch.int64 if bits == 64 else torch.int32)


def _packed_layout(total, r):
    lens = _lengths(total, r)
    cu = np.zeros(len(lens) + 1, dtype=np.int32)
    np.cumsum(lens, out=cu[1:])
    return lens, torch.from_numpy(cu).cuda()


def _packed_mask(lens, cu, prompt):
    """Response mask of a packed batch: zero on each sequence's first token and on its prompt."""
    n = int(sum(lens))
    mask = torch.ones(n, device="cuda")
    mask[cu[:-1].long()] = 0.0
    if prompt > 0.0:
        lens_t = (cu[1:] - cu[:-1]).long()
        at = torch.arange(n, device="cuda") - torch.repeat_interleave(cu[:-1].long(), lens_t)
        mask[at < torch.repeat_interleave((lens_t * prompt).long(), lens_t)] = 0.0
    return mask


def _prepare_score(c, seed):
    g, _ = _rand(seed)
    h, w = _head_weights(g, c["tokens"], c["hidden"], c["vocab"])
    return dict(c, h=h, w=w, labels=_ids(g, c["tokens"], c["vocab"], c["label_bits"]))


def _prepare_head(c, seed):
    s = _prepare_score(c, seed)
    g, _ = _rand(seed + 7919)
    n = c["tokens"]
    # upstream gradients of a token-mean loss: signed advantages on the log-probs, a small pull on the entropy
    s.update(g_lp=_randn(g, n) / n, g_en=-0.01 / n + 0.001 * _randn(g, n) / n)
    s["h"].requires_grad_(True)
    s["w"].requires_grad_(True)
    return s


def _prepare_step(c, seed):
    g, r = _rand(seed)
    n, hidden, vocab = c["tokens"], c["hidden"], c["vocab"]
    h, w = _head_weights(g, n, hidden, vocab)
    ids = _ids(g, n, vocab, 64)
    lens, cu = _packed_layout(n, r)
    mask = _packed_mask(lens, cu, c["prompt"])
    # the policy that sampled the batch: this head's log-probs (label logit minus the log-sum-exp of Gaussian logits)
    # moved by a little noise
    lp = torch.zeros(n, device="cuda")
    for a in range(0, n - 1, 4096):
        b = min(a + 4096, n - 1)
        logit = (h[a:b].float() * w[ids[a + 1:b + 1]].float()).sum(1)
        lse = math.log(vocab) + 0.5 * (0.02 ** 2) * h[a:b].float().square().sum(1)
        lp[a + 1:b + 1] = logit - lse
    lp[cu[:-1].long()] = 0.0
    old = lp + 0.05 * _randn(g, n)
    tlr = torch.zeros(n, device="cuda")
    tlr[cu[1:].long() - 1] = torch.bernoulli(torch.full((len(lens),), 0.5, device="cuda"), generator=g)
    s = dict(c, h=h.requires_grad_(True), w=w.requires_grad_(True), ids=ids, cu=cu, old=old,
             mask=_mask(mask, c["mask_bits"]), rewards=tlr, uid=_labels_of(len(lens), r),
             sampler=old + 0.01 * _randn(g, n))
    if c["side"]:
        s["ref"] = old + 0.1 * _randn(g, n)
    return s


def _prepare_loss(c, seed):
    g, r = _rand(seed)
    if c["layout"] == "padded":
        b, t = c["rows"], c["length"]
        lens = torch.randint(max(1, t // 16), t + 1, (b,), generator=g, device="cuda")
        mask = (torch.arange(t, device="cuda")[None, :] < lens[:, None]).float()
        last = (torch.arange(b, device="cuda"), lens - 1)
        shape, rows, cu = (b, t), b, None
    else:
        lens, cu = _packed_layout(c["tokens"], r)
        mask = _packed_mask(lens, cu, 0.25)
        last = (cu[1:].long() - 1,)
        shape, rows = (c["tokens"],), len(lens)
    old = -torch.empty(shape, device="cuda").exponential_(1.0, generator=g)
    new = old + 0.05 * _randn(g, *shape)
    # sampler log-probs: tight around the trainer's but for one token in a thousand
    far = torch.rand(shape, generator=g, device="cuda") < 0.001
    samp = old + 0.01 * _randn(g, *shape) + far * 2.0 * _randn(g, *shape)
    tlr = torch.zeros(shape, device="cuda")
    tlr[last] = torch.bernoulli(torch.full((rows,), 0.5, device="cuda"), generator=g)
    return dict(c, cu=cu, old=old, new=new.requires_grad_(True), sampler=samp, rewards=tlr,
                mask=_mask(mask, c["mask_bits"]), uid=_labels_of(rows, r))


def _prepare_value(c, seed):
    g, r = _rand(seed)
    n = c["tokens"]
    lens, cu = _packed_layout(n, r)
    tlr = torch.zeros(n, device="cuda")
    tlr[cu[1:].long() - 1] = torch.bernoulli(torch.full((len(lens),), 0.5, device="cuda"), generator=g)
    values = 0.5 + 0.2 * _randn(g, n)
    return dict(c, cu=cu, rewards=tlr, values=values, vpreds=(values + 0.3 * _randn(g, n)).requires_grad_(True),
                mask=_mask(_packed_mask(lens, cu, 0.25), c["mask_bits"]))


def _prepare_logits(c, seed):
    g, _ = _rand(seed)
    n, v = c["tokens"], c["vocab"]
    z = torch.empty(n, v, device="cuda", dtype=torch.bfloat16 if c["bits"] == 16 else torch.float32)
    z.normal_(0.0, 2.0, generator=g)
    return dict(c, logits=z.requires_grad_(True), labels=torch.randint(0, v, (n,), generator=g, device="cuda"),
                g_lp=_randn(g, n) / n, g_en=-0.01 / n + 0.001 * _randn(g, n) / n)


def prepare(case, seed):
    make = dict(score=_prepare_score, head=_prepare_head, step=_prepare_step, loss=_prepare_loss, value=_prepare_value,
                logits=_prepare_logits)
    return make[case["kind"]](case, seed)


# --------------------------------------------------------------------------------------------------------------
# one pass
# --------------------------------------------------------------------------------------------------------------

# sampler correction settings: token weights with token rejection and the veto; sequence weights with the geometric
# rejection
_CORRECTION = {
    "none": {},
    "token_veto": dict(sampler_is="token", sampler_is_threshold=2.0, sampler_rs="token", sampler_rs_threshold=2.0,
                       sampler_token_veto_threshold=1e-4),
    "sequence_geometric": dict(sampler_is="sequence", sampler_is_threshold=2.0, sampler_rs="geometric",
                               sampler_rs_threshold=1.01),
}
_LOSS_ARGS = {
    "ppo": ("ppo", dict(clip_ratio_low=0.2, clip_ratio_high=0.2)),
    "dapo": ("ppo", dict(clip_ratio_low=0.2, clip_ratio_high=0.28)),
    "gspo": ("gspo", dict(clip_ratio_low=3e-4, clip_ratio_high=4e-4, token_reduce="mean", batch_reduce="step-mean")),
    "cispo": ("cispo", dict(clip_ratio_high=0.28)),
    "reinforce": ("reinforce", {}),
    "geo_mean": ("geo_mean", dict(clip_ratio=0.4)),
}


def _run_score(s):
    with torch.no_grad():
        lp, ent = linear_cross_entropy(s["h"], s["w"], s["labels"], s["temperature"], "none", None, s["softcap"] or None)
    return lp, ent


def _run_head(s):
    s["h"].grad = s["w"].grad = None
    lp, ent = linear_cross_entropy(s["h"], s["w"], s["labels"], s["temperature"], "none", None, s["softcap"] or None)
    torch.autograd.backward([lp, ent], [s["g_lp"], s["g_en"]])
    return lp.detach(), ent.detach(), s["h"].grad, s["w"].grad


def _run_step(s):
    s["h"].grad = s["w"].grad = None
    data = DataProto.from_dict(tensors={"token_level_rewards": s["rewards"], "response_mask": s["mask"]},
                               meta_info={"cu_seqlens": s["cu"]})
    data.non_tensor_batch["uid"] = s["uid"]
    data = compute_advantage(data, {"advantage": "grpo"})
    tensors = {"old_log_probs": s["old"], "advantages": data.batch["advantages"], "response_mask": s["mask"],
               "sampler_log_probs": s["sampler"]}
    name, args = _LOSS_ARGS[s["loss"]]
    args = dict(args)
    if s["side"]:
        tensors["ref_log_prob"] = s["ref"]
        args.update(entropy_coef=0.001, kl_coef=0.01, kl_type="low_var_kl")
    if s["correction"]:
        args.update(_CORRECTION["token_veto"])
    batch = DataProto.from_dict(tensors=tensors)
    loss, metrics = fused_head_loss(s["h"], s["w"], s["ids"], s["cu"], batch,
                                    {"loss_fn": name, "loss_fn_args": args, "temperature": 1.0, "dp_replicas": 1})
    loss.backward()
    return (loss.detach(), metrics["pg_loss"], metrics["entropy"], batch.batch["log_probs"], batch.batch["entropys"],
            s["h"].grad, s["w"].grad)


def _run_loss(s):
    s["new"].grad = None
    data = DataProto.from_dict(tensors={"token_level_rewards": s["rewards"], "response_mask": s["mask"],
                                        "old_log_probs": s["old"], "sampler_log_probs": s["sampler"],
                                        "log_probs": s["new"]},
                               meta_info={} if s["cu"] is None else {"cu_seqlens": s["cu"]})
    # the uid array has one entry per sequence, as the trainer keeps it beside a packed batch
    data.non_tensor_batch["uid"] = s["uid"]
    data = compute_advantage(data, {"advantage": s["advantage"]})
    name, args = _LOSS_ARGS[s["loss"]]
    loss, _ = compute_loss_fn(data, name, dict(args, **_CORRECTION[s["correction"]]))
    loss.backward()
    b = data.batch
    out = [loss.detach(), s["new"].grad, b["advantages"], b["response_mask"]]
    if "sampler_is_weights" in b:
        out.append(b["sampler_is_weights"])
    return out


def _run_value(s):
    s["vpreds"].grad = None
    data = DataProto.from_dict(tensors={"token_level_rewards": s["rewards"], "response_mask": s["mask"],
                                        "values": s["values"], "vpreds": s["vpreds"]},
                               meta_info={"cu_seqlens": s["cu"]})
    data = compute_advantage(data, {"advantage": "gae", "advantage_args": {"gamma": 1.0, "lam": 0.95}})
    loss, _ = compute_loss_fn(data, "value", {"cliprange_value": 0.5})
    loss.backward()
    return loss.detach(), s["vpreds"].grad, data.batch["advantages"], data.batch["returns"]


def _run_logits(s):
    s["logits"].grad = None
    lp, ent = logprobs_and_entropy_from_logits(s["logits"], s["labels"])
    torch.autograd.backward([lp, ent], [s["g_lp"], s["g_en"]])
    return lp.detach(), ent.detach(), s["logits"].grad


def run(state):
    go = dict(score=_run_score, head=_run_head, step=_run_step, loss=_run_loss, value=_run_value, logits=_run_logits)
    return go[state["kind"]](state)


# --------------------------------------------------------------------------------------------------------------
# what a pass cannot do without, and how far two correct implementations may differ
# --------------------------------------------------------------------------------------------------------------

def work(case):
    k, n = case["kind"], case.get("tokens", 0)
    if k in ("score", "head", "step"):
        h, v = case["hidden"], case["vocab"]
        operands = 2 * (n * h + v * h)
        if k == "score":
            return {"bytes": operands + n * (case["label_bits"] // 8 + 8), "flops": 2.0 * n * h * v}
        if k == "head":
            return {"bytes": 2 * operands + n * (case["label_bits"] // 8 + 16), "flops": 6.0 * n * h * v}
        # ids, mask, rewards, old, sampler (and reference) log-probs in; log-probs and entropy out
        token_bytes = 8 + case["mask_bits"] // 8 + 4 * (3 + int(case["side"])) + 8
        return {"bytes": 2 * operands + n * token_bytes, "flops": 6.0 * n * h * v}
    if k == "loss":
        n = case["rows"] * case["length"] if case["layout"] == "padded" else n
        # rewards, mask, old and new log-probs in, advantages and gradient out; with a correction also the sampler's
        # log-probs in, weights and the new mask out
        per = 4 * 3 + case["mask_bits"] // 8 + 4 * 2 + (12 if case["correction"] != "none" else 0)
        return {"bytes": n * per, "flops": 30.0 * n}
    if k == "value":
        # rewards, values, vpreds, mask in; advantages, returns, gradient out
        return {"bytes": n * (4 * 3 + case["mask_bits"] // 8 + 4 * 3), "flops": 30.0 * n}
    v, e = case["vocab"], case["bits"] // 8
    return {"bytes": 2 * n * v * e + n * 24, "flops": 10.0 * n * v}


def tolerance(case):
    # about four times the distance seen from the same path in float64 (head: 2.3e-3 in the gradients, 5e-8 in the
    # outputs; bf16 logits 1.7e-3) or with its rows in another order (losses)
    k = case["kind"]
    if k in ("head", "step"):  # bf16 gradients, formed from bf16 dlogits
        return {"rel": 1e-2}
    if k == "logits" and case["bits"] == 16:  # a gradient rounded to bf16
        return {"rel": 7e-3}
    if k == "loss":  # fp32 sums; the loss itself is what is left of advantages that nearly add up to zero (1.2e-5)
        return {"rel": 5e-5}
    return {"rel": 5e-6}
