"""GPU parity of the step as ONE autograd node that works block of tokens by block (head forward with a
stash -> loss on the block -> head backward from the stash): against the CPU oracle's chain at small sizes
(PPO, DAPO with entropy bonus and KL penalty, GSPO; block borders on and off sequence ends; one block and many),
against the unfused GPU path, and at the full Qwen3-8B shape against an fp32 torch head + the oracle's loss.

Tolerances: loss 1e-4 relative, bf16 gradients 2e-2 relative L2 against the oracle, 5e-3 against the unfused
GPU path (the stash rounds softmax numerators to fp16 where the recompute keeps fp32), metrics 1e-4 relative."""

import numpy as np
import pytest
import torch

from axon_amd import workloads as W
from axon_amd.protocol import DataProto
from axon_amd.trainer.algos.advantages import compute_advantage
from oracle import advantage as OA
from oracle import lmhead as OM
from oracle import loss as OL

pytestmark = pytest.mark.gpu
DEV = "cuda"


def rel_l2(a, b):
    a, b = a.detach().double().cpu(), b.detach().double().cpu()
    return ((a - b).norm() / b.norm().clamp_min(1e-30)).item()


def _inputs(n, h, v, lens, seed, group=3):
    hid, w, ids = W.lmhead_inputs(n, h, v, seed=seed)
    w = (w.float() * 6).bfloat16()
    rl = W.packed_rl_inputs(n, seed=seed + 1, lengths=lens)
    rl["uid"] = W.uids_for(len(lens), group)
    g = torch.Generator().manual_seed(seed + 2)
    labels = torch.roll(ids, -1)
    lp_head, _ = OM.forward(hid, w, labels)
    old = _to_token_positions(lp_head, rl["cu_seqlens"].long()) - 0.05 * torch.randn(n, generator=g)
    ref = old + 0.1 * torch.randn(n, generator=g)
    return hid, w, ids, labels, rl, old, ref


def _to_token_positions(x, cu):
    out = torch.zeros_like(x)
    out[1:] = x[:-1]
    out[cu[:-1][cu[:-1] < x.numel()]] = 0.0
    return out


def _pad(x, cu, tmax):
    return torch.stack([torch.nn.functional.pad(x[a:b], (0, tmax - (b - a))) for a, b in zip(cu[:-1], cu[1:])])


# GRPO advantages add up to zero over a complete group, and GSPO's sequence ratios are within a few 1e-4 of one:
# its loss is then what is left of a cancelling sum, and its relative error is that of the log-probs times the
# cancellation.  The GSPO cases therefore move every advantage by a constant, which makes the loss O(1).
GSPO_ADV_SHIFT = 0.5


def oracle_step(hid, w, labels, rl, old, ref, loss_name, args, dp_replicas=1, n_micro_batches=1, adv_shift=0.0):
    """Head forward -> shift -> GRPO advantage -> actor loss (policy loss, entropy bonus, KL penalty) ->
    backward through the shift -> head backward, all on the CPU oracle."""
    cu = rl["cu_seqlens"].long()
    lens = (cu[1:] - cu[:-1]).tolist()
    tmax = max(lens)
    lp_head, ent_head = OM.forward(hid, w, labels)
    lp_tok, ent_tok = _to_token_positions(lp_head, cu), _to_token_positions(ent_head, cu)
    gidx = torch.tensor(np.unique(rl["uid"], return_inverse=True)[1])
    mask = _pad(rl["response_mask"], cu, tmax)
    adv = OA.grpo_advantage(_pad(rl["token_level_rewards"], cu, tmax), mask, gidx, 1e-6) + adv_shift * mask
    lp_pad = _pad(lp_tok, cu, tmax).requires_grad_(True)
    en_pad = _pad(ent_tok, cu, tmax).requires_grad_(True)
    fn = OL.ppo_loss if loss_name == "ppo" else OL.gspo_loss
    loss, metrics = OL.actor_loss(fn, lp_pad, en_pad, _pad(old, cu, tmax), adv, mask, loss_args=args,
                                  ref_log_prob=_pad(ref, cu, tmax), dp_replicas=dp_replicas,
                                  n_micro_batches=n_micro_batches)
    loss.backward()

    def to_head(g_pad):
        if g_pad is None:
            return None
        g_tok = torch.cat([g_pad[b, :l] for b, l in enumerate(lens)])
        g_head = torch.zeros_like(g_tok)
        g_head[:-1] = g_tok[1:]
        g_head[cu[1:] - 1] = 0.0
        return g_head

    dh, dw = OM.backward(to_head(lp_pad.grad), to_head(en_pad.grad), hid, w, labels)
    return loss.detach(), metrics, lp_tok, ent_tok, dh, dw


def fused_step(hid, w, ids, rl, old, ref, loss_name, args, block_tokens, dp_replicas=1, n_micro_batches=1,
               vocab_chunk=0, extra=None, adv_shift=0.0, dw_group=None):
    from axon_amd.models.fused_head_loss import DEFAULT_DW_GROUP, fused_head_loss
    dw_group = DEFAULT_DW_GROUP if dw_group is None else dw_group
    hd, wd = hid.to(DEV).requires_grad_(True), w.to(DEV).requires_grad_(True)
    cu = rl["cu_seqlens"].to(DEV)
    a_in = DataProto.from_dict(tensors={"token_level_rewards": rl["token_level_rewards"].to(DEV),
                                        "response_mask": rl["response_mask"].to(DEV)}, meta_info={"cu_seqlens": cu})
    a_in.non_tensor_batch["uid"] = rl["uid"]
    adv = compute_advantage(a_in, {"advantage": "grpo", "advantage_args": {"epsilon": 1e-6}}).batch["advantages"]
    adv = adv + adv_shift * rl["response_mask"].to(DEV)
    tensors = {"old_log_probs": old.to(DEV), "advantages": adv, "response_mask": rl["response_mask"].to(DEV),
               "ref_log_prob": ref.to(DEV)}
    tensors.update({k: v.to(DEV) for k, v in (extra or {}).items()})
    data = DataProto.from_dict(tensors=tensors)
    meta = {"loss_fn": loss_name, "loss_fn_args": args, "temperature": 1.0, "dp_replicas": dp_replicas,
            "n_micro_batches": n_micro_batches}
    loss, metrics = fused_head_loss(hd, wd, ids.to(DEV), cu, data, meta, block_tokens=block_tokens,
                                    vocab_chunk=vocab_chunk, dw_group=dw_group)
    loss.backward()
    return loss.detach(), metrics, data, hd.grad, wd.grad


PPO = {"clip_ratio_low": 0.2, "clip_ratio_high": 0.28}
DAPO_SIDE = {"clip_ratio_low": 0.2, "clip_ratio_high": 0.28, "entropy_coef": 0.01, "kl_coef": 0.05,
             "kl_type": "low_var_kl"}
GSPO = {"clip_ratio_low": 3e-4, "clip_ratio_high": 4e-4, "token_reduce": "mean", "batch_reduce": "step-mean"}
GSPO_SIDE = dict(GSPO, entropy_coef=0.01, kl_coef=0.05, kl_type="k2")
RAGGED = [400, 33, 500, 64, 300, 203]          # 1500 tokens; no sequence ends on a multiple of 256
ON_BORDERS = [256, 256, 512, 128, 128, 256]     # 1536 tokens; every sequence ends on a block border
ODD_TOTAL = [400, 33, 500, 64, 300, 205]        # 1502 tokens: a last block of 478 or 222 rows cannot be stashed


@pytest.mark.parametrize("lens", [RAGGED, ON_BORDERS, ODD_TOTAL], ids=["ragged", "on-borders", "odd-total"])
@pytest.mark.parametrize("block_tokens", [256, 512, 4096], ids=["b256", "b512", "one-block"])
@pytest.mark.parametrize("case", ["ppo", "dapo-entropy-kl", "gspo", "gspo-entropy-kl"])
def test_fused_step_vs_oracle(case, block_tokens, lens):
    name, args = {"ppo": ("ppo", PPO), "dapo-entropy-kl": ("ppo", DAPO_SIDE), "gspo": ("gspo", GSPO),
                  "gspo-entropy-kl": ("gspo", GSPO_SIDE)}[case]
    if name == "gspo" and block_tokens < max(lens):
        block_tokens = 512  # blocks hold whole sequences
    n, h, v = sum(lens), 128, 2000
    hid, w, ids, labels, rl, old, ref = _inputs(n, h, v, lens, seed=71)
    shift = GSPO_ADV_SHIFT if name == "gspo" else 0.0
    want = oracle_step(hid, w, labels, rl, old, ref, name, args, dp_replicas=2, n_micro_batches=4, adv_shift=shift)
    got = fused_step(hid, w, ids, rl, old, ref, name, args, block_tokens, dp_replicas=2, n_micro_batches=4,
                     adv_shift=shift)
    data = got[2]
    assert data.meta_info["head_backward"] == "blocked-stash"
    expect_blocks = {256: -(-n // 256), 512: -(-n // 512), 4096: 1}[block_tokens]
    if name == "ppo":
        assert data.meta_info["n_blocks"] == expect_blocks
    else:
        assert data.meta_info["n_blocks"] >= expect_blocks
    assert got[0].item() == pytest.approx(want[0].item(), rel=1e-4, abs=1e-8)
    assert (data.batch["log_probs"].cpu() - want[2]).abs().max() < 1e-3
    assert (data.batch["entropys"].cpu() - want[3]).abs().max() < 1e-3
    assert rel_l2(got[3], want[4]) < 2e-2 and rel_l2(got[4], want[5]) < 2e-2
    keys = ["pg_loss", "entropy", "entropy_token_mean", "pg_clipfrac", "ppo_kl"]
    keys += ["kl_loss", "kl_coef"] if "kl_coef" in args else []
    for k in keys:
        assert got[1][k] == pytest.approx(want[1][k], rel=1e-4, abs=1e-6), k


@pytest.mark.parametrize("lens", [RAGGED, ODD_TOTAL], ids=["ragged", "odd-total"])
@pytest.mark.parametrize("dw_group", [1, 2, 3, 8])
@pytest.mark.parametrize("case", ["dapo-entropy-kl", "gspo-entropy-kl"])
def test_fused_step_with_grouped_weight_gradient_vs_oracle(case, dw_group, lens):
    """Hidden size 256 and a vocabulary that is a multiple of 8: the weight gradient reads the token-major
    dlogits as a K-major GEMM operand (no vocab-major copy), and `dw_group` consecutive blocks share one such
    GEMM (1: every block its own; 8: one GEMM for the step; 2 and 3: groups with a shorter last one, and with
    blocks that are no multiple of 256 rows inside a group)."""
    name, args = {"dapo-entropy-kl": ("ppo", DAPO_SIDE), "gspo-entropy-kl": ("gspo", GSPO_SIDE)}[case]
    n, h, v = sum(lens), 256, 2000
    hid, w, ids, labels, rl, old, ref = _inputs(n, h, v, lens, seed=73)
    shift = GSPO_ADV_SHIFT if name == "gspo" else 0.0
    want = oracle_step(hid, w, labels, rl, old, ref, name, args, adv_shift=shift)
    got = fused_step(hid, w, ids, rl, old, ref, name, args, 256 if name == "ppo" else 512, adv_shift=shift,
                     dw_group=dw_group)
    data = got[2]
    assert data.meta_info["head_backward"] == "blocked-stash" and data.meta_info["n_blocks"] >= 3
    assert got[0].item() == pytest.approx(want[0].item(), rel=1e-4, abs=1e-8)
    assert rel_l2(got[3], want[4]) < 2e-2 and rel_l2(got[4], want[5]) < 2e-2


@pytest.mark.parametrize("vocab_chunk", [0, 1024])
@pytest.mark.parametrize("case", ["ppo", "dapo-entropy-kl", "gspo"])
def test_fused_step_vs_unfused_gpu_path(case, vocab_chunk):
    """The same micro-batch through the node and through head -> loss -> autograd: the loss agrees to fp32
    summation order, the gradients to the rounding of the stash, the metrics and the head outputs as well."""
    from axon_amd.models.fsdp_models import loss_from_outputs
    from axon_amd.utils.fsdp.forward_utils import packed_logprobs
    name, args = {"ppo": ("ppo", PPO), "dapo-entropy-kl": ("ppo", DAPO_SIDE), "gspo": ("gspo", GSPO)}[case]
    g = torch.Generator().manual_seed(5)
    lens = W.uniform_lengths(24, 40, 700, g)
    n, h, v = sum(lens), 256, 8192
    hid, w, ids, labels, rl, old, ref = _inputs(n, h, v, lens, seed=81, group=4)
    samp = old + 0.01 * torch.randn(n, generator=g)
    extra = {"sampler_log_probs": samp}
    got = fused_step(hid, w, ids, rl, old, ref, name, args, 1024, vocab_chunk=vocab_chunk, extra=extra,
                     adv_shift=GSPO_ADV_SHIFT if name == "gspo" else 0.0)
    assert got[2].meta_info["head_backward"] == "blocked-stash" and got[2].meta_info["n_blocks"] >= 3

    hd, wd = hid.to(DEV).requires_grad_(True), w.to(DEV).requires_grad_(True)
    cu = rl["cu_seqlens"].to(DEV)
    lp, ent = packed_logprobs(hd, wd, ids.to(DEV), cu)
    b = got[2].batch
    data = DataProto.from_dict(tensors={"old_log_probs": b["old_log_probs"], "advantages": b["advantages"],
                                        "response_mask": rl["response_mask"].to(DEV), "ref_log_prob": b["ref_log_prob"],
                                        "sampler_log_probs": b["sampler_log_probs"]}, meta_info={"cu_seqlens": cu})
    meta = {"loss_fn": name, "loss_fn_args": args, "temperature": 1.0, "dp_replicas": 1}
    loss, metrics = loss_from_outputs(data, lp, ent, meta)
    loss.backward()
    assert got[0].item() == pytest.approx(loss.item(), rel=2e-6, abs=1e-9)
    assert torch.equal(b["log_probs"], lp.detach()) and torch.equal(b["entropys"], ent.detach())
    assert rel_l2(got[3], hd.grad) < 5e-3 and rel_l2(got[4], wd.grad) < 5e-3
    assert set(got[1]) == set(metrics)
    for k, val in metrics.items():
        assert got[1][k] == pytest.approx(val, rel=1e-4, abs=1e-6), k


def test_fused_step_with_sampler_correction_and_global_counts():
    """The correction hook runs once over the whole batch before the blocks (token IS weights, token rejection,
    per-sequence veto); the loss then uses the corrected mask and the weights, the side terms the original mask;
    a ``valid_token_count`` carried by the batch is the denominator of every block."""
    from axon_amd.models.fsdp_models import loss_from_outputs
    from axon_amd.utils.fsdp.forward_utils import packed_logprobs
    g = torch.Generator().manual_seed(9)
    lens = W.uniform_lengths(20, 30, 500, g)
    n, h, v = sum(lens), 128, 4096
    hid, w, ids, labels, rl, old, ref = _inputs(n, h, v, lens, seed=91, group=4)
    samp = old + 0.01 * torch.randn(n, generator=g)
    samp[::97] += 1.5  # some tokens outside the rejection bounds
    args = dict(DAPO_SIDE, sampler_is="token", sampler_is_threshold=2.0, sampler_rs="token", sampler_rs_threshold=2.0,
                sampler_token_veto_threshold=1e-4)
    count = torch.full((n,), 3.0 * n, dtype=torch.float32)
    extra = {"sampler_log_probs": samp, "valid_token_count": count}
    got = fused_step(hid, w, ids, rl, old, ref, "ppo", args, 512, extra=extra)
    assert got[2].meta_info["head_backward"] == "blocked-stash"
    hd, wd = hid.to(DEV).requires_grad_(True), w.to(DEV).requires_grad_(True)
    cu = rl["cu_seqlens"].to(DEV)
    lp, ent = packed_logprobs(hd, wd, ids.to(DEV), cu)
    b = got[2].batch
    data = DataProto.from_dict(tensors={"old_log_probs": b["old_log_probs"], "advantages": b["advantages"],
                                        "response_mask": rl["response_mask"].to(DEV), "ref_log_prob": b["ref_log_prob"],
                                        "sampler_log_probs": b["sampler_log_probs"], "valid_token_count": count.to(DEV)},
                               meta_info={"cu_seqlens": cu})
    loss, metrics = loss_from_outputs(data, lp, ent, {"loss_fn": "ppo", "loss_fn_args": args, "temperature": 1.0,
                                                     "dp_replicas": 1})
    loss.backward()
    assert torch.equal(b["response_mask"], data.batch["response_mask"])  # the corrected mask, bit for bit
    assert got[0].item() == pytest.approx(loss.item(), rel=2e-6, abs=1e-9)
    assert rel_l2(got[3], hd.grad) < 5e-3 and rel_l2(got[4], wd.grad) < 5e-3
    assert set(got[1]) == set(metrics)
    for k, val in metrics.items():
        assert got[1][k] == pytest.approx(val, rel=1e-4, abs=1e-6), k


@pytest.mark.parametrize("case", ["ppo", "gspo"])
def test_fused_step_odd_shapes_softcap_temperature_and_integer_operands(case):
    """A token count that is no multiple of four (the last block then has no stash and recomputes its logits), a
    vocabulary that is no multiple of the tile, blocks smaller than a tile, soft-capped logits, a temperature,
    int64 token ids and an int64 response mask (the production dtypes): the node against the unfused path."""
    from axon_amd.models.fsdp_models import loss_from_outputs
    from axon_amd.models.fused_head_loss import fused_head_loss
    from axon_amd.utils.fsdp.forward_utils import packed_logprobs
    name, args = {"ppo": ("ppo", DAPO_SIDE), "gspo": ("gspo", GSPO)}[case]
    lens = [130, 7, 251, 64, 301, 90]  # 843 tokens
    n, h, v = sum(lens), 96, 1001
    hid, w, ids, labels, rl, old, ref = _inputs(n, h, v, lens, seed=95)
    cu = rl["cu_seqlens"].to(DEV)
    mask_i64 = rl["response_mask"].to(DEV).long()
    adv = (torch.randn(n, generator=torch.Generator().manual_seed(3)) + (GSPO_ADV_SHIFT if case == "gspo" else 0.0))
    meta = {"loss_fn": name, "loss_fn_args": args, "temperature": 0.7, "dp_replicas": 1}

    def tensors():
        return {"old_log_probs": old.to(DEV), "advantages": adv.to(DEV) * mask_i64, "response_mask": mask_i64.clone(),
                "ref_log_prob": ref.to(DEV)}

    hd, wd = hid.to(DEV).requires_grad_(True), w.to(DEV).requires_grad_(True)
    data = DataProto.from_dict(tensors=tensors())
    loss, metrics = fused_head_loss(hd, wd, ids.to(DEV).long(), cu, data, meta, block_tokens=384 if case == "gspo" else 200,
                                    logit_softcapping=5.0)
    loss.backward()
    assert data.meta_info["head_backward"] == "blocked-stash" and data.meta_info["n_blocks"] >= 3

    h2, w2 = hid.to(DEV).requires_grad_(True), w.to(DEV).requires_grad_(True)
    lp, ent = packed_logprobs(h2, w2, ids.to(DEV).long(), cu, 0.7, 5.0)
    data2 = DataProto.from_dict(tensors=tensors(), meta_info={"cu_seqlens": cu})
    loss2, metrics2 = loss_from_outputs(data2, lp, ent, meta)
    loss2.backward()
    assert loss.item() == pytest.approx(loss2.item(), rel=2e-6, abs=1e-9)
    assert torch.equal(data.batch["log_probs"], lp.detach()) and torch.equal(data.batch["entropys"], ent.detach())
    assert rel_l2(hd.grad, h2.grad) < 5e-3 and rel_l2(wd.grad, w2.grad) < 5e-3
    for k, val in metrics2.items():
        assert metrics[k] == pytest.approx(val, rel=1e-4, abs=1e-6), k


@pytest.mark.parametrize("v", [2000, 1999])
@pytest.mark.parametrize("case", ["ppo", "gspo"])
def test_large_blocks_that_the_stash_is_not_kept_for_recompute_in_fp32(monkeypatch, case, v):
    """Blocks of 256 rows and more whose tokens (the last one's) or vocabulary are no multiple of four recompute
    their logits in fp32: the gradients are bit for bit those of a step that keeps no stash at all.  Where the other
    blocks do keep one, the rows of the last block are."""
    from axon_amd import _ops
    from axon_amd.models.fused_head_loss import fused_head_loss
    lens = [256, 301, 211, 256, 277]  # 1301 tokens; blocks of 512, or whole sequences of 557 and 467: the last has 277 rows
    n, h = sum(lens), 128
    name, args = {"ppo": ("ppo", PPO), "gspo": ("gspo", GSPO)}[case]
    g = torch.Generator().manual_seed(17)
    hid = torch.randn(n, h, generator=g).bfloat16().to(DEV)
    w = (torch.randn(v, h, generator=g) * 0.2).bfloat16().to(DEV)
    ids = torch.randint(0, v, (n,), generator=g).to(DEV)
    old, adv = (-8 + 0.1 * torch.randn(n, generator=g)).to(DEV), torch.randn(n, generator=g).to(DEV)
    cu = torch.tensor([0] + lens).cumsum(0).int().to(DEV)
    real = _ops.HeadBlocks
    kept = []

    class Recording(real):
        def forward(self, k):
            super().forward(k)
            kept.append(self.block_stash_bytes > 0)

    def step(cls):
        monkeypatch.setattr(_ops, "HeadBlocks", cls)
        hd, wd = hid.clone().requires_grad_(True), w.clone().requires_grad_(True)
        data = DataProto.from_dict(tensors={"old_log_probs": old, "advantages": adv,
                                            "response_mask": torch.ones(n, device=DEV)})
        loss, _ = fused_head_loss(hd, wd, ids, cu, data, {"loss_fn": name, "loss_fn_args": args, "temperature": 1.0,
                                                          "dp_replicas": 1}, block_tokens=560 if case == "gspo" else 512)
        loss.backward()
        return hd.grad, wd.grad

    dh, dw = step(Recording)
    dh0, dw0 = step(lambda *a, **k: real(*a, **dict(k, stash=False)))
    assert len(kept) == 3 and not kept[-1] and kept[:-1] == [v % 4 == 0] * 2
    assert torch.equal(dh[1024:], dh0[1024:]) and dh[1024:].float().norm() > 0
    if v % 4:
        assert torch.equal(dh, dh0) and torch.equal(dw, dw0)
    else:
        assert rel_l2(dh, dh0) < 5e-3 and rel_l2(dw, dw0) < 5e-3


def test_fused_step_falls_back_where_blocks_do_not_apply():
    """A loss that selects tokens across the whole batch, and a sequence longer than a block under a
    per-sequence loss, take the unfused path; the node refuses a second backward."""
    lens = RAGGED
    n, h, v = sum(lens), 128, 2000
    hid, w, ids, labels, rl, old, ref = _inputs(n, h, v, lens, seed=71)
    got = fused_step(hid, w, ids, rl, old, ref, "kl_cov", {"kl_cov_ratio": 0.01}, 256)
    assert got[2].meta_info["head_backward"] == "recompute" and torch.isfinite(got[0]).item()
    got = fused_step(hid, w, ids, rl, old, ref, "gspo", GSPO, 256,  # the 400- and 500-token sequences do not fit
                     adv_shift=GSPO_ADV_SHIFT)
    assert got[2].meta_info["head_backward"] == "recompute"
    want = oracle_step(hid, w, labels, rl, old, ref, "gspo", GSPO, adv_shift=GSPO_ADV_SHIFT)
    assert got[0].item() == pytest.approx(want[0].item(), rel=1e-4, abs=1e-8)
    assert rel_l2(got[3], want[4]) < 2e-2 and rel_l2(got[4], want[5]) < 2e-2

    from axon_amd.models.fused_head_loss import fused_head_loss
    hd, wd = hid.to(DEV).requires_grad_(True), w.to(DEV).requires_grad_(True)
    data = DataProto.from_dict(tensors={"old_log_probs": old.to(DEV), "advantages": torch.ones(n, device=DEV),
                                        "response_mask": rl["response_mask"].to(DEV)})
    loss, _ = fused_head_loss(hd, wd, ids.to(DEV), rl["cu_seqlens"].to(DEV), data,
                              {"loss_fn": "ppo", "loss_fn_args": PPO, "temperature": 1.0, "dp_replicas": 1},
                              block_tokens=512)
    loss.backward(retain_graph=True)
    with pytest.raises(RuntimeError, match="second time"):
        loss.backward()


def test_fused_step_scales_the_finished_gradients_by_the_incoming_factor():
    """``dp_replicas`` (and any other factor on the loss) reaches d_hidden and d_weight although they are finished
    before autograd's backward starts."""
    lens = ON_BORDERS
    n, h, v = sum(lens), 128, 2000
    hid, w, ids, labels, rl, old, ref = _inputs(n, h, v, lens, seed=73)
    one = fused_step(hid, w, ids, rl, old, ref, "ppo", PPO, 512, dp_replicas=1)
    four = fused_step(hid, w, ids, rl, old, ref, "ppo", PPO, 512, dp_replicas=4)
    assert four[0].item() == pytest.approx(4 * one[0].item(), rel=1e-6)
    assert rel_l2(four[3], 4 * one[3].float()) < 4e-3 and rel_l2(four[4], 4 * one[4].float()) < 4e-3


def test_qwen3_8b_fused_step_vs_fp32_torch_and_oracle_loss():
    """Config 3 at full size through the node (four blocks of 8192 tokens): log-prob and entropy of every token
    and d_weight on ~120 vocabulary rows against an fp32 torch head on the GPU driven by the CPU oracle's PPO
    loss gradient; d_hidden on a token subset against the CPU oracle; and the loss itself."""
    from head_reference import _fp32_torch_head_reference, _spread_rows
    n, h, v = 32768, 4096, 151936
    hid, w, ids = W.lmhead_inputs(n, h, v, seed=3)
    rl = W.packed_rl_inputs(n, 103, group=8)
    cu = rl["cu_seqlens"].long()
    hd0, wd0, ids_d = hid.to(DEV), w.to(DEV), ids.to(DEV)
    labels_d = torch.roll(ids_d, -1)
    zeros = torch.zeros(n, device=DEV)
    rows = _spread_rows(v)
    ref_lp, ref_ent, _ = _fp32_torch_head_reference(hd0, wd0, labels_d, zeros, None, rows[:1])
    lp_tok = _to_token_positions(ref_lp.cpu(), cu)
    old = lp_tok - 0.05 * torch.randn(n, generator=torch.Generator().manual_seed(7))
    got = fused_step(hid, w, ids, rl, old, old, "ppo", PPO, 8192)
    data = got[2]
    assert data.meta_info["head_backward"] == "blocked-stash" and data.meta_info["n_blocks"] == 4
    assert data.meta_info["stash_bytes"] <= 2 * 8192 * 152064 + (1 << 26)
    assert (data.batch["log_probs"].cpu() - lp_tok).abs().max().item() < 1e-3
    assert (data.batch["entropys"].cpu() - _to_token_positions(ref_ent.cpu(), cu)).abs().max().item() < 1e-3
    # the oracle's loss and its gradient on the reference log-probs, on the padded layout the reference uses
    lens = (cu[1:] - cu[:-1]).tolist()
    tmax = max(lens)
    gidx = torch.tensor(np.unique(rl["uid"], return_inverse=True)[1])
    mask = _pad(rl["response_mask"], cu, tmax)
    adv = OA.grpo_advantage(_pad(rl["token_level_rewards"], cu, tmax), mask, gidx, 1e-6)
    lp_pad = _pad(lp_tok, cu, tmax).requires_grad_(True)
    loss, _ = OL.ppo_loss(lp_pad, _pad(old, cu, tmax), adv, mask, **PPO)
    loss.backward()
    assert got[0].item() == pytest.approx(loss.item(), rel=1e-4, abs=1e-8)
    g_tok = torch.cat([lp_pad.grad[b, :l] for b, l in enumerate(lens)])
    g_head = torch.zeros_like(g_tok)
    g_head[:-1] = g_tok[1:]
    g_head[cu[1:] - 1] = 0.0
    _, _, ref_dw = _fp32_torch_head_reference(hd0, wd0, labels_d, g_head.to(DEV), None, rows)
    got_dw = got[4][rows.to(DEV)].double()
    assert rel_l2(got_dw, ref_dw) < 2e-2
    per_row = (got_dw - ref_dw).norm(dim=1) / ref_dw.norm(dim=1).clamp_min(1e-30)
    assert per_row.max().item() < 5e-2, (per_row.argmax().item(), per_row.max().item())
    idx = torch.cat([torch.arange(0, n, 509), torch.tensor([8191, 8192, 16383, 16384, 24575, 24576, n - 1])])
    o_dh, _ = OM.backward(g_head[idx], None, hid[idx], w, torch.roll(ids, -1)[idx])
    assert rel_l2(got[3][idx.to(DEV)], o_dh) < 2e-2


@pytest.mark.parametrize("nan", [False, True])
@pytest.mark.parametrize("case", ["ppo", "gspo"])
def test_fused_step_with_a_correction_in_flight(case, nan):
    """The step does not wait for the sampler correction: an all-zero mask, known only at the end, leaves the batch as it
    was, without correction metrics and with zero gradients, also where the sampler's log-probs are NaN."""
    from axon_amd.models.fused_head_loss import fused_head_loss
    lens = [40, 25, 63]
    n, h, v = sum(lens), 64, 300
    hid, w, ids, labels, rl, old, ref = _inputs(n, h, v, lens, seed=4)
    name, args = {"ppo": ("ppo", PPO), "gspo": ("gspo", GSPO)}[case]
    args = dict(args, sampler_is="token", sampler_is_threshold=2.0, sampler_token_veto_threshold=1e-4)
    hd, wd = hid.to(DEV).requires_grad_(True), w.to(DEV).requires_grad_(True)
    mask = torch.zeros(n, device=DEV)
    samp = old.to(DEV) * (float("nan") if nan else 1.01)
    data = DataProto.from_dict(tensors={"old_log_probs": old.to(DEV), "advantages": torch.ones(n, device=DEV),
                                        "response_mask": mask, "sampler_log_probs": samp})
    loss, metrics = fused_head_loss(hd, wd, ids.to(DEV), rl["cu_seqlens"].to(DEV), data,
                                    {"loss_fn": name, "loss_fn_args": args, "temperature": 1.0, "dp_replicas": 1})
    loss.backward()
    assert loss.item() == 0.0 and (hd.grad == 0).all() and (wd.grad == 0).all()
    assert data.batch["response_mask"] is mask and "sampler_is_weights" not in data.batch
    assert not any(k.startswith("sampler_corr/") for k in metrics)


def test_fused_step_of_one_block_checks_the_offsets_it_never_reads():
    """A sequence-cut batch of one block does not read its offsets back first; offsets that do not span the batch are refused
    all the same, with the step's one readback."""
    from axon_amd.models.fused_head_loss import fused_head_loss
    lens = [40, 25, 63]
    n, h, v = sum(lens), 64, 300
    hid, w, ids, labels, rl, old, ref = _inputs(n, h, v, lens, seed=4)
    for cu in ([0, 40, 65, n - 1], [1, 40, 65, n], [0, 40, 65, n + 8]):
        for kw in ({}, {"cu_host": cu}):
            data = DataProto.from_dict(tensors={"old_log_probs": old.to(DEV), "advantages": torch.ones(n, device=DEV),
                                                "response_mask": torch.ones(n, device=DEV)})
            with pytest.raises(ValueError, match=f"spans {cu[0]}..{cu[-1]}, the batch has {n} tokens"):
                fused_head_loss(hid.to(DEV).requires_grad_(True), w.to(DEV).requires_grad_(True), ids.to(DEV),
                                torch.tensor(cu, dtype=torch.int32, device=DEV), data,
                                {"loss_fn": "gspo", "loss_fn_args": GSPO, "temperature": 1.0, "dp_replicas": 1}, **kw)


@pytest.mark.parametrize("n,blocks", [(1, 1), (255, 2), (256, 1), (1027, 5)])
@pytest.mark.parametrize("ent,kl", [(0.0, 0.0), (0.01, 0.0), (0.0, 0.2), (0.01, 0.2)])
def test_gradients_and_scalars_between_the_kernels_of_a_step(n, blocks, ent, kl):
    """axon_step_grads / axon_step_scalars against torch, into slices that begin anywhere and leave their neighbours alone."""
    from axon_amd import _ops
    g = torch.Generator().manual_seed(n)
    grad, agg_w, grad_kl = torch.randn(3, n, generator=g).to(DEV)
    accs = torch.randn(blocks, 16, generator=g).to(DEV)
    g_lp, g_en = torch.full((2, n + 7), 9.0, device=DEV)
    _ops.step_grads(grad, accs[0, :8], agg_w, grad_kl if kl else None, accs[0, 8:], ent, kl, g_lp[3:n + 3],
                    g_en[3:n + 3] if ent else None)
    want = grad.double() * accs[0, 5].double() + kl * grad_kl.double() * accs[0, 13].double()
    assert (g_lp[3:n + 3].double() - want).abs().max() < 1e-5
    assert (g_lp[:3] == 9).all() and (g_lp[n + 3:] == 9).all() and (g_en[:3] == 9).all() and (g_en[n + 3:] == 9).all()
    assert not ent or (g_en[3:n + 3].double() + ent * agg_w.double() * accs[0, 13].double()).abs().max() < 1e-6
    out = torch.full((10,), 9.0, device=DEV, dtype=torch.float64)
    cu = torch.tensor([0, 5, n + 11], dtype=torch.int32, device=DEV)
    loss = _ops.step_scalars(accs, ent, kl, cu, out)
    tot = accs.double().sum(0)
    assert loss.shape == () and abs(loss.item() - (tot[0] - ent * tot[8] + kl * tot[9]).item()) < 1e-5
    assert (out[:8].view(torch.float32).double() - tot).abs().max() < 1e-5 and out[8:].tolist() == [0.0, n + 11.0]


@pytest.mark.parametrize("lens", [[1], [3, 0, 0, 1, 1, 1, 2, 9], [0, 0, 5], [4] * 300 + [0] * 700 + [1, 2, 3], [5000, 0]])
def test_sequence_start_flags_and_paired_scaling(lens):
    from axon_amd import _ops
    n = sum(lens)
    cu = torch.tensor([0] + lens).cumsum(0)
    want = torch.zeros((n + 3) // 4 * 4, dtype=torch.uint8)
    want[[int(a) for a, b in zip(cu[:-1], cu[1:]) if b > a]] = 1
    assert torch.equal(_ops.seq_start_flags(cu.int().to(DEV), n).cpu(), want)
    x, y = torch.randn(8 * n, device=DEV).bfloat16(), torch.randn(264, device=DEV).bfloat16()
    for s in (1.0, 0.25, 0.0, 3.0):
        a, b = x.clone(), y.clone()
        _ops.scale_bf16_unless_one(a, b, torch.tensor(s, device=DEV))
        assert torch.equal(a, (x.float() * s).bfloat16()) and torch.equal(b, (y.float() * s).bfloat16())


@pytest.mark.parametrize("offset", [0, 1, 2, 3])
@pytest.mark.parametrize("n", [1, 4, 1027])
def test_sequence_start_flags_at_any_address(n, offset):
    from axon_amd import _lib, _ops
    cu = torch.tensor([0, n // 3, n // 2, n], dtype=torch.int32, device=DEV)
    words = (n + 3) // 4 * 4
    buf = torch.full((words + 8,), 7, dtype=torch.uint8, device=DEV)
    rc = _lib.load().axon_seq_start_flags(cu.data_ptr(), 3, n, buf.data_ptr() + offset, _ops.stream_ptr())
    assert rc == 0 and torch.equal(buf[offset:offset + words], _ops.seq_start_flags(cu, n))
    assert (buf[:offset] == 7).all() and (buf[offset + words:] == 7).all()


@pytest.mark.parametrize("n,at", [(1027, 1027), (1027, 513), (1026, 1), (5, 3)])
def test_sequence_start_flags_of_offsets_padded_with_empty_sequences(n, at):
    """20000 empty sequences at one place: the right flags, and no thread that goes through them one by one (which took
    five hundred times as long as the call without them)."""
    from axon_amd import _ops
    real = torch.arange(0, n + 1, max(n // 40, 1))
    real[-1] = n
    padded = torch.sort(torch.cat([real, torch.full((20000,), at)]))[0]
    want = torch.zeros((n + 3) // 4 * 4, dtype=torch.uint8)
    want[padded[:-1][padded[1:] > padded[:-1]]] = 1

    def timed(cu):
        cu, best = cu.int().to(DEV), float("inf")
        for _ in range(10):
            a, b = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
            a.record()
            for _ in range(5):
                flags = _ops.seq_start_flags(cu, n)
            b.record()
            b.synchronize()
            best = min(best, a.elapsed_time(b))
        return flags, best

    (flags, t), (_, t0) = timed(padded), timed(real)
    assert torch.equal(flags.cpu(), want) and t < 20 * t0


@pytest.mark.parametrize("n,block_tokens,blocks", [(257, 256, 2), (1025, 512, 3)])
@pytest.mark.parametrize("case", ["ppo", "dapo-entropy-kl"])
def test_a_block_that_owns_no_position_adds_nothing(case, n, block_tokens, blocks, monkeypatch):
    """Positions are shifted by one against rows: a last block of one row owns none of them, and no kernel writes its sums.
    With NaN in every new tensor the step is that of one block: loss, metrics, outputs and gradients (the stash rounds
    softmax numerators to fp16 where the odd single block has fp32 logits)."""
    from axon_amd.models.fused_head_loss import token_blocks
    assert token_blocks(n, block_tokens)[-1] == (n - 1, n) and len(token_blocks(n, block_tokens)) == blocks
    lens = [n - 150, 50, 37, 63]
    hid, w, ids, labels, rl, old, ref = _inputs(n, 64, 300, lens, seed=n, group=2)
    args = {"ppo": PPO, "dapo-entropy-kl": DAPO_SIDE}[case]
    want = fused_step(hid, w, ids, rl, old, ref, "ppo", args, 4096, adv_shift=0.5)
    empty, empty_like = torch.empty, torch.empty_like
    as_nan = lambda t: t.fill_(float("nan")) if t.is_cuda and t.is_floating_point() else t  # noqa: E731
    monkeypatch.setattr(torch, "empty", lambda *a, **k: as_nan(empty(*a, **k)))
    monkeypatch.setattr(torch, "empty_like", lambda *a, **k: as_nan(empty_like(*a, **k)))
    got = fused_step(hid, w, ids, rl, old, ref, "ppo", args, block_tokens, adv_shift=0.5)
    assert got[2].meta_info["n_blocks"] == blocks and want[2].meta_info["n_blocks"] == 1
    assert got[0].item() == pytest.approx(want[0].item(), rel=1e-4)
    assert set(got[1]) == set(want[1])
    for k, x in want[1].items():
        assert got[1][k] == pytest.approx(x, rel=1e-4, abs=1e-6), k
    for k in ("log_probs", "entropys"):
        assert (got[2].batch[k] - want[2].batch[k]).abs().max() < 1e-5
    assert rel_l2(got[3], want[3]) < 5e-3 and rel_l2(got[4], want[4]) < 5e-3


@pytest.mark.parametrize("refused", ["later allocations", "the logits", "nothing"])
def test_kept_logits_give_way_to_what_the_step_cannot_do_without(refused, monkeypatch):
    """A step that fits without its blocks' fp32 logits fits with the choice to keep them: the other buffers are there before
    them, and they are not kept where they would leave little room.  The same bits either way."""
    import weakref
    lens = [150, 50, 37, 64]
    n, h, v = sum(lens), 768, 1000
    hid, w, ids, labels, rl, old, ref = _inputs(n, h, v, lens, seed=9, group=2)
    step = lambda: fused_step(hid, w, ids, rl, old, ref, "ppo", DAPO_SIDE, 8192)  # noqa: E731
    want = step()
    need = 4 * 2 * 262144  # four vocabulary tiles, two token tiles
    assert want[2].meta_info["stash_bytes"] == need
    if refused != "later allocations":  # half of the room is what they take, or a byte less
        allocated = torch.cuda.memory_allocated
        monkeypatch.setattr(torch.cuda, "mem_get_info", lambda dev: (need, 4 * need))
        monkeypatch.setattr(torch.cuda, "memory_reserved",
                            lambda dev: allocated(dev) + need - (refused == "the logits"))
    else:
        kept = [None]

        def guard(make):
            def made(*a, **k):
                t = make(*a, **k)
                size = t.numel() * t.element_size()
                if t.is_cuda and size >= 65536 and kept[0] is not None and kept[0]() is not None:
                    raise torch.OutOfMemoryError("no room beside the logits")
                if t.is_cuda and t.dtype == torch.uint8 and size == need:
                    kept[0] = weakref.ref(t)
                return t
            return made

        for name in ("empty", "empty_like", "zeros"):
            monkeypatch.setattr(torch, name, guard(getattr(torch, name)))
    got = step()
    assert got[2].meta_info["stash_bytes"] == (0 if refused == "the logits" else need)
    assert torch.equal(got[0], want[0]) and got[1] == want[1]
    assert torch.equal(got[3], want[3]) and torch.equal(got[4], want[4])


@pytest.mark.parametrize("block_tokens", [8192, 64], ids=["one-block", "blocks"])
def test_refused_offsets_leave_the_batch_as_it_was(block_tokens):
    """Offsets that do not span the batch: no log-probs or entropies of a step that was refused, no mask or weights of its
    sampler correction, whether they are checked before the first launch or with the step's readback."""
    from axon_amd.models.fused_head_loss import fused_head_loss
    lens = [40, 25, 63]
    n, h, v = sum(lens), 64, 300
    hid, w, ids, labels, rl, old, ref = _inputs(n, h, v, lens, seed=4)
    args = dict(GSPO, sampler_is="token", sampler_is_threshold=2.0, sampler_token_veto_threshold=1e-4)
    tensors = {"old_log_probs": old.to(DEV), "advantages": torch.ones(n, device=DEV),
               "response_mask": torch.ones(n, device=DEV), "sampler_log_probs": 1.01 * old.to(DEV)}
    data = DataProto.from_dict(tensors=dict(tensors))
    cu = [0, 40, 65, n - 1]
    with pytest.raises(ValueError, match=f"spans 0..{n - 1}, the batch has {n} tokens"):
        fused_head_loss(hid.to(DEV).requires_grad_(True), w.to(DEV).requires_grad_(True), ids.to(DEV),
                        torch.tensor(cu, dtype=torch.int32, device=DEV), data,
                        {"loss_fn": "gspo", "loss_fn_args": args, "temperature": 1.0, "dp_replicas": 1},
                        block_tokens=block_tokens)
    assert set(data.batch.keys()) == set(tensors) and all(data.batch[k] is t for k, t in tensors.items())
    assert "head_backward" not in data.meta_info
