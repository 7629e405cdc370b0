"""Engine tests on CPU (torch-reference op path): scheduler, KV manager,
end-to-end generation with tiny models, determinism, preemption."""
import pytest
import torch

from inference_gateway_amd.engine.config import (MODEL_PRESETS, EngineConfig,
                                                 SamplingParams)
from inference_gateway_amd.engine.engine import LLMEngine
from inference_gateway_amd.engine.kvcache import BlockManager


def test_block_manager_alloc_free():
    bm = BlockManager(8, 16)  # block 0 is reserved scratch => 7 usable
    a = bm.allocate(33)  # 3 blocks
    assert len(a) == 3 and bm.num_free == 4
    assert 0 not in a
    bm.ensure_capacity(a, 48)
    assert len(a) == 3
    bm.ensure_capacity(a, 49)
    assert len(a) == 4 and bm.num_free == 3
    bm.free(a)
    assert bm.num_free == 7 and a == []


def _engine(**kw):
    torch.manual_seed(0)
    return LLMEngine(EngineConfig.tiny_llama(**kw), device="cpu")


def test_generate_greedy_deterministic():
    eng = _engine()
    rid = eng.add_request(
        list(range(1, 17)),
        SamplingParams(max_new_tokens=8, temperature=0.0),
    )
    while not eng.is_finished():
        eng.step()
    out1 = eng.get_output(rid)
    assert out1.finished and out1.finish_reason == "length"
    assert len(out1.token_ids) == 8

    eng2 = _engine()
    rid2 = eng2.add_request(
        list(range(1, 17)),
        SamplingParams(max_new_tokens=8, temperature=0.0),
    )
    while not eng2.is_finished():
        eng2.step()
    assert eng2.get_output(rid2).token_ids == out1.token_ids


def test_continuous_batching_multiple_requests():
    eng = _engine()
    rids = [
        eng.add_request(
            list(range(1, 5 + i)),
            SamplingParams(max_new_tokens=4 + i, temperature=0.0),
        )
        for i in range(3)
    ]
    steps = 0
    while not eng.is_finished():
        eng.step()
        steps += 1
        assert steps < 64
    for i, rid in enumerate(rids):
        out = eng.get_output(rid)
        assert out.finished
        assert len(out.token_ids) == 4 + i


def test_incremental_batching_matches_isolated():
    """A request decoded inside a batch must produce the same tokens as the
    same request decoded alone (continuous batching must not change
    numerics beyond bf16 noise — greedy on CPU fp32 refs is exact)."""
    eng = _engine()
    ra = eng.add_request(list(range(1, 20)),
                         SamplingParams(max_new_tokens=6, temperature=0.0))
    rb = eng.add_request(list(range(30, 40)),
                         SamplingParams(max_new_tokens=6, temperature=0.0))
    while not eng.is_finished():
        eng.step()
    batched = eng.get_output(ra).token_ids

    eng2 = _engine()
    ra2 = eng2.add_request(list(range(1, 20)),
                          SamplingParams(max_new_tokens=6, temperature=0.0))
    while not eng2.is_finished():
        eng2.step()
    assert eng2.get_output(ra2).token_ids == batched


def test_stop_token():
    eng = _engine()
    # run once to find the first greedy token, then use it as stop token
    rid = eng.add_request(list(range(1, 9)),
                          SamplingParams(max_new_tokens=4, temperature=0.0))
    while not eng.is_finished():
        eng.step()
    first = eng.get_output(rid).token_ids[0]

    eng2 = _engine()
    rid2 = eng2.add_request(
        list(range(1, 9)),
        SamplingParams(max_new_tokens=4, temperature=0.0,
                       stop_token_ids=(first,)),
    )
    while not eng2.is_finished():
        eng2.step()
    out = eng2.get_output(rid2)
    assert out.finish_reason == "stop"
    assert out.token_ids == [first]


def test_preemption_recovers():
    # tiny block pool: force preemption under concurrent decode
    eng = _engine(num_gpu_blocks=10)
    eng.cfg.max_num_seqs = 4
    rids = [
        eng.add_request(list(range(1, 17)),
                        SamplingParams(max_new_tokens=40, temperature=0.0))
        for _ in range(3)
    ]
    steps = 0
    while not eng.is_finished():
        eng.step()
        steps += 1
        assert steps < 500
    for rid in rids:
        out = eng.get_output(rid)
        assert out.finished
        assert len(out.token_ids) == 40


def test_moe_engine_generates():
    torch.manual_seed(0)
    cfg = EngineConfig(
        model=MODEL_PRESETS["tiny-moe"],
        num_gpu_blocks=64,
        max_num_seqs=4,
        max_batched_tokens=512,
        max_model_len=256,
        use_hip_graphs=False,
    )
    eng = LLMEngine(cfg, device="cpu")
    rid = eng.add_request(list(range(1, 12)),
                         SamplingParams(max_new_tokens=5, temperature=0.0))
    while not eng.is_finished():
        eng.step()
    out = eng.get_output(rid)
    assert out.finished and len(out.token_ids) == 5


def test_moe_padded_matches_sorted():
    """The sync-free padded-dispatch MoE path (decode, hipGraph-capturable)
    must agree with the per-expert sorted-GEMM path (prefill)."""
    from inference_gateway_amd.engine.models.mixtral import MixtralMoE

    torch.manual_seed(3)
    cfg = MODEL_PRESETS["tiny-moe"]
    moe = MixtralMoE(cfg, layer=0, device="cpu", dtype=torch.float32)
    x = torch.randn(13, cfg.hidden_size)
    a = moe._forward_padded(x)
    b = moe._forward_sorted(x)
    assert torch.allclose(a, b, atol=1e-5, rtol=1e-4)


def test_moe_without_k_major_copies():
    """Experts that the GPU's kernels take keep one copy of their weights: what
    other calls run then, and state dicts with and without the copies."""
    from inference_gateway_amd.engine.models.mixtral import MixtralMoE

    torch.manual_seed(5)
    cfg = MODEL_PRESETS["tiny-moe"]
    both, one = (MixtralMoE(cfg, layer=i, device="cpu", dtype=torch.float32)
                 for i in range(2))
    assert both.gate_up_t is not None and both.down_t is not None
    one.gate_up_t = one.down_t = None
    one.load_state_dict(both.state_dict())
    x = torch.randn(13, cfg.hidden_size)
    for name in ("_forward_padded", "_forward_sorted"):
        torch.testing.assert_close(getattr(one, name)(x),
                                   getattr(both, name)(x), atol=1e-5,
                                   rtol=1e-4)
    other = MixtralMoE(cfg, layer=2, device="cpu", dtype=torch.float32)
    assert "gate_up_t" not in one.state_dict()
    other.load_state_dict(one.state_dict())
    for name, t in both.state_dict().items():
        assert torch.equal(other.state_dict()[name], t)
    other.gate_up.data.mul_(2)
    other.sync_k_major()
    assert torch.equal(other.gate_up_t, other.gate_up.transpose(1, 2))


def test_moe_padded_every_expert_rank_unique():
    """Dispatch ranks must give every (token, k) pair a unique padded row."""
    from inference_gateway_amd.engine.models.mixtral import MixtralMoE

    torch.manual_seed(4)
    cfg = MODEL_PRESETS["tiny-moe"]
    moe = MixtralMoE(cfg, layer=0, device="cpu", dtype=torch.float32)
    T, E, K = 17, cfg.num_experts, cfg.num_experts_per_tok
    logits = torch.randn(T, E)
    _, topk = torch.topk(logits, K, dim=-1)
    flat = topk.reshape(-1)
    onehot = torch.nn.functional.one_hot(flat, E)
    rank = (torch.cumsum(onehot, 0) - onehot).mul(onehot).sum(-1)
    dst = flat * T + rank
    assert dst.unique().numel() == T * K


def test_moe_route_ref_valid():
    from inference_gateway_amd.ops import torch_ref

    torch.manual_seed(11)
    T, E, K, C = 33, 8, 2, 33
    logits = torch.randn(T, E)
    w, dst, idx, counts = torch_ref.moe_route_ref(logits, K, C)
    # weights are softmax over the top-k logits
    vals, ref_idx = torch.topk(logits, K, dim=-1)
    assert torch.equal(idx.long(), ref_idx)
    assert torch.allclose(w, torch.softmax(vals, -1), atol=1e-6)
    # dst rows are unique and live in the right expert segment with a
    # rank below that expert's count
    assert dst.unique().numel() == T * K
    flat = ref_idx.reshape(-1)
    assert torch.equal(counts.long(), torch.bincount(flat, minlength=E))
    for i in range(T * K):
        e = int(flat[i])
        r = int(dst[i]) - e * C
        assert 0 <= r < int(counts[e])


def test_engine_fuzz_invariants():
    """Randomized add/step/abort interleaving: the engine must never
    wedge, every request must terminate, and the block pool must be fully
    restored (no leaked KV blocks or slots)."""
    import random

    rng = random.Random(1234)
    torch.manual_seed(0)
    eng = _engine(num_gpu_blocks=24, max_model_len=96, max_num_seqs=4)
    bm = eng.block_manager
    free0 = bm.num_free
    slots0 = len(eng.scheduler._free_slots)
    live, done = [], []
    for step in range(300):
        r = rng.random()
        if r < 0.25 and len(live) < 10:
            rid = eng.add_request(
                list(rng.randrange(1, 500) for _ in range(
                    rng.randrange(4, 40))),
                SamplingParams(max_new_tokens=rng.randrange(1, 12),
                               temperature=rng.choice([0.0, 0.8]),
                               top_k=rng.choice([0, 20]),
                               top_p=rng.choice([1.0, 0.9])))
            live.append(rid)
        elif r < 0.32 and live:
            victim = live.pop(rng.randrange(len(live)))
            eng.abort_request(victim)
            done.append(victim)
        outs = eng.step()
        for o in outs:
            if o.finished and o.seq_id in live:
                live.remove(o.seq_id)
                done.append(o.seq_id)
    while not eng.is_finished():
        for o in eng.step():
            if o.finished and o.seq_id in live:
                live.remove(o.seq_id)
    assert eng.is_finished()
    assert bm.num_free == free0, "leaked KV blocks"
    assert len(eng.scheduler._free_slots) == slots0, "leaked slots"


@pytest.mark.parametrize("seed", [77, 1234, 9001])
def test_engine_fuzz_invariants_mixed_mode(seed):
    """The same randomized stress with the FULL r2 feature stack on:
    mixed same-step batches + chunked prefill + prefix caching +
    prefill-first, tiny block pool (preemption pressure), forks and
    aborts.  Invariants: never wedges, pool and slots fully restored."""
    import random

    rng = random.Random(seed)
    torch.manual_seed(0)
    eng = _engine(num_gpu_blocks=28, max_model_len=96, max_num_seqs=4,
                  max_batched_tokens=48, enable_chunked_prefill=True,
                  enable_prefix_caching=True, enable_mixed_batches=True,
                  scheduler_prefill_first=True)
    bm = eng.block_manager
    free0 = bm.num_free
    slots0 = len(eng.scheduler._free_slots)
    shared = list(range(200, 248))       # prefix-cacheable stem
    live, done = [], []
    for step in range(400):
        r = rng.random()
        if r < 0.22 and len(live) < 10:
            prompt = (shared[: rng.choice([16, 32, 48])]
                      + [rng.randrange(1, 500) for _ in range(
                          rng.randrange(1, 20))])
            sp = SamplingParams(max_new_tokens=rng.randrange(1, 10),
                                temperature=rng.choice([0.0, 0.8]),
                                seed=rng.choice([None, 5]),
                                logit_bias=rng.choice(
                                    [None, {7: 50.0}, {3: -40.0}]))
            if r < 0.05 and eng.scheduler.can_adopt():
                rids = eng.add_request_group(prompt, sp, n=2)
                live.extend(rids)
            else:
                live.append(eng.add_request(prompt, sp))
        elif r < 0.30 and live:
            victim = live.pop(rng.randrange(len(live)))
            eng.abort_request(victim)
            done.append(victim)
        outs = eng.step()
        for o in outs:
            if o.finished and o.seq_id in live:
                live.remove(o.seq_id)
                done.append(o.seq_id)
    guard = 0
    while not eng.is_finished():
        guard += 1
        assert guard < 2000, "engine wedged during drain"
        for o in eng.step():
            if o.finished and o.seq_id in live:
                live.remove(o.seq_id)
    assert bm.num_free == free0, "leaked KV blocks"
    assert len(eng.scheduler._free_slots) == slots0, "leaked slots"
    assert eng.scheduler.num_mixed_rounds > 0, "mixed rounds never ran"


def test_prompt_longer_than_token_budget_is_not_starved():
    """A prompt above max_batched_tokens (but under max_model_len) must be
    admitted as its own oversized prefill batch, not starve forever."""
    eng = _engine(max_batched_tokens=64, max_model_len=256,
                  num_gpu_blocks=64)
    rid = eng.add_request(list(range(1, 101)),   # 100 > 64 budget
                          SamplingParams(max_new_tokens=4, temperature=0.0))
    steps = 0
    while not eng.is_finished():
        eng.step()
        steps += 1
        assert steps < 50, "long prompt starved"
    out = eng.get_output(rid)
    assert out.finished and len(out.token_ids) == 4


def test_bucket_ladder_invariants():
    """Bucket ladder: strictly increasing, and from 16 up each step grows
    by <= 1.5x so graph-padding waste is bounded (a 600-seq batch must not
    pad to 1024)."""
    from inference_gateway_amd.engine.graph_runner import _BUCKETS

    assert _BUCKETS == sorted(set(_BUCKETS))
    assert _BUCKETS[0] == 1 and _BUCKETS[-1] == 1024
    for a, b in zip(_BUCKETS, _BUCKETS[1:]):
        if a >= 16:
            assert b <= a * 1.5 + 1e-9, (a, b)


def test_logprobs_eager_greedy():
    """logprobs: greedy sampling must report the argmax as both the
    sampled token's logprob and top-1; alternatives sorted descending;
    sequences that did not ask must get None."""
    eng = _engine()
    rid_lp = eng.add_request(
        list(range(1, 17)),
        SamplingParams(max_new_tokens=4, temperature=0.0, logprobs=3))
    rid_plain = eng.add_request(
        list(range(2, 18)),
        SamplingParams(max_new_tokens=4, temperature=0.0))
    outs = []
    while not eng.is_finished():
        outs.extend(eng.step())
    by_seq = {}
    for o in outs:
        by_seq.setdefault(o.seq_id, []).append(o)
    lp_outs = by_seq[rid_lp]
    assert len(lp_outs) == 4
    for o in lp_outs:
        assert o.logprob is not None and o.logprob <= 0.0
        assert len(o.top_logprobs) == 3
        vals = [v for _, v in o.top_logprobs]
        assert vals == sorted(vals, reverse=True)
        # greedy: the sampled token IS the top-1 alternative
        assert o.top_logprobs[0][0] == o.token_id
        assert abs(o.top_logprobs[0][1] - o.logprob) < 1e-5
    for o in by_seq[rid_plain]:
        assert o.logprob is None and o.top_logprobs is None


def test_logprobs_k_zero_returns_sampled_only():
    eng = _engine()
    rid = eng.add_request(
        list(range(1, 17)),
        SamplingParams(max_new_tokens=3, temperature=0.0, logprobs=0))
    outs = []
    while not eng.is_finished():
        outs.extend(eng.step())
    assert len(outs) == 3
    for o in outs:
        assert o.logprob is not None and o.top_logprobs == []


def test_seeded_sampling_is_request_deterministic():
    """OpenAI `seed`: a seeded request replays the same tokens regardless
    of what else is in the batch; unseeded requests keep engine RNG."""
    def run(extra_load: bool):
        eng = _engine()
        rid = eng.add_request(
            list(range(1, 17)),
            SamplingParams(max_new_tokens=6, temperature=1.0, seed=1234))
        if extra_load:   # batch composition must not matter
            eng.add_request(
                list(range(5, 21)),
                SamplingParams(max_new_tokens=6, temperature=1.0))
        while not eng.is_finished():
            eng.step()
        return eng.get_output(rid).token_ids

    a = run(extra_load=False)
    b = run(extra_load=True)
    assert a == b and len(a) == 6

    eng = _engine()
    rid = eng.add_request(
        list(range(1, 17)),
        SamplingParams(max_new_tokens=6, temperature=1.0, seed=4321))
    while not eng.is_finished():
        eng.step()
    c = eng.get_output(rid).token_ids
    assert c != a    # different seed -> (overwhelmingly) different draw


def test_frequency_penalty_blocks_repetition():
    """A huge frequency penalty must prevent any token from being
    generated twice (greedy, eager path: host counts are exact)."""
    eng = _engine()
    rid = eng.add_request(
        list(range(1, 17)),
        SamplingParams(max_new_tokens=12, temperature=0.0,
                       frequency_penalty=100.0))
    while not eng.is_finished():
        eng.step()
    toks = eng.get_output(rid).token_ids
    assert len(toks) == 12
    assert len(set(toks)) == 12    # all distinct

    # sanity: without the penalty the same model DOES repeat (tiny model,
    # greedy decode converges to a loop)
    eng2 = _engine()
    rid2 = eng2.add_request(
        list(range(1, 17)),
        SamplingParams(max_new_tokens=12, temperature=0.0))
    while not eng2.is_finished():
        eng2.step()
    toks2 = eng2.get_output(rid2).token_ids
    assert len(set(toks2)) < 12


def test_fork_group_matches_independent_requests():
    """n>1 fork: each branch's KV (shared full blocks + copied tail)
    must be bit-equal to a recomputed prefill — greedy branches must
    reproduce an independent request's tokens exactly."""
    prompt = list(range(1, 27))      # 26 tokens: 1 full block + partial
    eng = _engine()
    rid = eng.add_request(
        prompt, SamplingParams(max_new_tokens=8, temperature=0.0))
    while not eng.is_finished():
        eng.step()
    want = eng.get_output(rid).token_ids

    eng2 = _engine()
    rids = eng2.add_request_group(
        prompt, SamplingParams(max_new_tokens=8, temperature=0.0), n=3)
    while not eng2.is_finished():
        eng2.step()
    for r in rids:
        out = eng2.get_output(r)
        assert out.finished
        assert out.token_ids == want


def test_fork_block_accounting():
    """All blocks (shared and private) return to the pool when every
    branch finishes; block-aligned prompts fork with zero copies."""
    for plen in (16, 26, 32):        # aligned and unaligned prompts
        eng = _engine()
        free0 = eng.block_manager.num_free
        rids = eng.add_request_group(
            list(range(1, plen + 1)),
            SamplingParams(max_new_tokens=5, temperature=0.0), n=4)
        while not eng.is_finished():
            eng.step()
        assert all(eng.get_output(r).finished for r in rids)
        assert eng.block_manager.num_free == free0, f"leak at plen={plen}"


def test_fork_seeded_branches_are_identical_and_unseeded_diverge():
    eng = _engine()
    rids = eng.add_request_group(
        list(range(1, 20)),
        SamplingParams(max_new_tokens=6, temperature=1.0, seed=7), n=2)
    while not eng.is_finished():
        eng.step()
    a, b = [eng.get_output(r).token_ids for r in rids]
    assert a == b            # same seed stream -> identical branches

    eng2 = _engine()
    rids2 = eng2.add_request_group(
        list(range(1, 20)),
        SamplingParams(max_new_tokens=8, temperature=1.0), n=4)
    while not eng2.is_finished():
        eng2.step()
    outs = [tuple(eng2.get_output(r).token_ids) for r in rids2]
    assert len(set(outs)) > 1    # engine RNG -> branches diverge


def test_fork_fallback_when_slots_exhausted():
    """More branches than slots: the overflow branches re-prefill as
    ordinary requests and still complete correctly; SEEDED groups stay
    identical even when some branches fall back (the discarded draw's
    seed tick is returned)."""
    eng_s = _engine()
    # an extra occupant forces at least one branch down the fallback path
    eng_s.add_request(list(range(40, 60)),
                      SamplingParams(max_new_tokens=12, temperature=0.0))
    rids_s = eng_s.add_request_group(
        list(range(1, 27)),
        SamplingParams(max_new_tokens=4, temperature=1.0, seed=5), n=8)
    while not eng_s.is_finished():
        eng_s.step()
    outs_s = [tuple(eng_s.get_output(r).token_ids) for r in rids_s]
    assert len(set(outs_s)) == 1, "seeded branches must be identical"

    eng = _engine()                    # max_num_seqs = 8
    rids = eng.add_request_group(
        list(range(1, 27)),
        SamplingParams(max_new_tokens=4, temperature=0.0), n=8)
    # a second independent request for the reference tokens
    ref = eng.add_request(
        list(range(1, 27)), SamplingParams(max_new_tokens=4,
                                           temperature=0.0))
    while not eng.is_finished():
        eng.step()
    want = eng.get_output(ref).token_ids
    for r in rids:
        assert eng.get_output(r).token_ids == want


def test_fork_abort_one_branch_others_complete():
    """Aborting one forked branch mid-decode must not disturb siblings
    or leak blocks (shared refs decremented, not freed)."""
    eng = _engine()
    free0 = eng.block_manager.num_free
    rids = eng.add_request_group(
        list(range(1, 27)),
        SamplingParams(max_new_tokens=10, temperature=0.0), n=3)
    for _ in range(4):
        eng.step()
    eng.abort_request(rids[1])
    while not eng.is_finished():
        eng.step()
    outs = [eng.get_output(r) for r in rids]
    assert outs[1].finish_reason == "abort"
    assert outs[0].finished and outs[2].finished
    assert outs[0].token_ids == outs[2].token_ids   # greedy, undisturbed
    assert len(outs[0].token_ids) == 10
    assert eng.block_manager.num_free == free0


def test_fork_parent_aborted_before_prefill_releases_children():
    """Parent aborted while still WAITING: children must be finished too
    (consumers get a sentinel instead of hanging)."""
    eng = _engine()
    # saturate the prefill queue so nothing runs yet
    rids = eng.add_request_group(
        list(range(1, 20)),
        SamplingParams(max_new_tokens=4, temperature=0.0), n=3)
    eng.abort_request(rids[0])
    for r in rids:
        assert eng.get_output(r).finish_reason == "abort"
    assert not eng.scheduler.has_work


def test_engine_counters():
    eng = _engine()
    rids = eng.add_request_group(
        list(range(1, 27)),
        SamplingParams(max_new_tokens=4, temperature=0.0), n=2)
    while not eng.is_finished():
        eng.step()
    assert all(eng.get_output(r).finished for r in rids)
    assert eng.num_prompt_tokens == 26          # ONE prefill for the group
    assert eng.num_generated_tokens == 8        # 4 tokens x 2 branches
    assert eng.num_forks == 1
    assert eng.scheduler.num_preemptions == 0


def test_fork_under_preemption_pressure():
    """Forks + LIFO preemption interleaved on a tiny block pool: every
    branch still completes with the right token count, no block leaks,
    and greedy branches (re-prefilled or not) agree."""
    eng = _engine(num_gpu_blocks=10, max_num_seqs=8)
    free0 = eng.block_manager.num_free
    groups = []
    for g in range(3):
        groups.append(eng.add_request_group(
            list(range(1 + g, 27 + g)),
            SamplingParams(max_new_tokens=12, temperature=0.0), n=2))
    steps = 0
    while not eng.is_finished():
        eng.step()
        steps += 1
        assert steps < 2000
    for rids in groups:
        outs = [eng.get_output(r) for r in rids]
        for o in outs:
            assert o.finished and len(o.token_ids) == 12
        assert outs[0].token_ids == outs[1].token_ids
    assert eng.block_manager.num_free == free0


def test_preempted_request_respects_max_new_tokens():
    """Regression: preemption folds generated tokens into the rebuilt
    prompt — the resumed request must still stop at max_new_tokens TOTAL
    and report every generated token, matching an unpressured run."""
    eng = _engine()
    rid = eng.add_request(list(range(1, 27)),
                          SamplingParams(max_new_tokens=10,
                                         temperature=0.0))
    while not eng.is_finished():
        eng.step()
    want = eng.get_output(rid).token_ids

    eng2 = _engine(num_gpu_blocks=6, max_num_seqs=4)
    rid2 = eng2.add_request(list(range(1, 27)),
                            SamplingParams(max_new_tokens=10,
                                           temperature=0.0))
    # pressure: a second long-running request forces block contention
    eng2.add_request(list(range(30, 56)),
                     SamplingParams(max_new_tokens=10, temperature=0.0))
    steps = 0
    while not eng2.is_finished():
        eng2.step()
        steps += 1
        assert steps < 2000
    assert eng2.scheduler.num_preemptions > 0
    got = eng2.get_output(rid2).token_ids
    assert len(got) == 10 and got == want


def test_seeded_sampling_survives_preemption():
    """A seeded stochastic request must produce identical tokens with
    and without preemption pressure (the seed stream is indexed by a
    per-seq tick that keeps counting across the rebuild)."""
    sp = SamplingParams(max_new_tokens=10, temperature=1.0, seed=77)
    eng = _engine()
    rid = eng.add_request(list(range(1, 27)), sp)
    while not eng.is_finished():
        eng.step()
    want = eng.get_output(rid).token_ids

    eng2 = _engine(num_gpu_blocks=6, max_num_seqs=4)
    rid2 = eng2.add_request(list(range(1, 27)), sp)
    eng2.add_request(list(range(30, 56)),
                     SamplingParams(max_new_tokens=10, temperature=0.0))
    steps = 0
    while not eng2.is_finished():
        eng2.step()
        steps += 1
        assert steps < 2000
    assert eng2.scheduler.num_preemptions > 0
    assert eng2.get_output(rid2).token_ids == want


def test_prefix_caching_equivalence_and_hits():
    """Prefix caching must be output-invariant: identical and
    prefix-shared prompts produce exactly the tokens a cache-less engine
    produces, while full leading blocks are served from cache."""
    base = list(range(1, 27))                 # 26 tokens: 1 full block
    longer = base + list(range(100, 120))     # 46: shares base's prefix
    sp = lambda: SamplingParams(max_new_tokens=6, temperature=0.0)

    eng0 = _engine()                          # caching OFF
    r_a0 = eng0.add_request(base, sp())
    r_b0 = eng0.add_request(longer, sp())
    while not eng0.is_finished():
        eng0.step()
    want_a = eng0.get_output(r_a0).token_ids
    want_b = eng0.get_output(r_b0).token_ids

    eng = _engine(enable_prefix_caching=True)
    r1 = eng.add_request(base, sp())
    while not eng.is_finished():
        eng.step()
    assert eng.block_manager.prefix_hit_tokens == 0
    assert eng.get_output(r1).token_ids == want_a

    # same prompt again: its 1 full block must come from the pool
    r2 = eng.add_request(base, sp())
    # a longer prompt sharing the 16-token prefix: 1-block hit too
    r3 = eng.add_request(longer, sp())
    while not eng.is_finished():
        eng.step()
    assert eng.get_output(r2).token_ids == want_a
    assert eng.get_output(r3).token_ids == want_b
    assert eng.block_manager.prefix_hit_tokens == 32   # 16 + 16

    # the longer prompt's 2 full blocks are now cached: re-running it
    # must hit both
    r4 = eng.add_request(longer, sp())
    while not eng.is_finished():
        eng.step()
    assert eng.get_output(r4).token_ids == want_b
    assert eng.block_manager.prefix_hit_tokens == 64   # +32


def test_prefix_caching_live_sharing_same_batch():
    """Two identical prompts admitted together: the second shares the
    first's LIVE blocks (KV written earlier in the same forward)."""
    eng = _engine(enable_prefix_caching=True)
    sp = lambda: SamplingParams(max_new_tokens=5, temperature=0.0)
    prompt = list(range(1, 40))               # 2 full blocks + partial
    r1 = eng.add_request(prompt, sp())
    r2 = eng.add_request(prompt, sp())
    while not eng.is_finished():
        eng.step()
    a, b = eng.get_output(r1).token_ids, eng.get_output(r2).token_ids
    assert a == b and len(a) == 5
    assert eng.block_manager.prefix_hit_tokens == 32


def test_prefix_caching_block_aligned_prompt_keeps_query_row():
    """A prompt that is an exact multiple of the block size must keep
    >= 1 uncached token (prefill needs a query row for logits, and the
    suffix's KV writes must stay out of shared blocks)."""
    eng = _engine(enable_prefix_caching=True)
    sp = lambda: SamplingParams(max_new_tokens=4, temperature=0.0)
    prompt = list(range(1, 33))               # exactly 2 blocks
    r1 = eng.add_request(prompt, sp())
    while not eng.is_finished():
        eng.step()
    want = eng.get_output(r1).token_ids
    r2 = eng.add_request(prompt, sp())
    while not eng.is_finished():
        eng.step()
    assert eng.get_output(r2).token_ids == want
    # only ONE of the two full blocks may be served from cache
    assert eng.block_manager.prefix_hit_tokens == 16


def test_prefix_pool_eviction_under_pressure():
    """Retained blocks are reclaimed LRU when the allocator runs dry —
    distinct prompts keep working and match a cache-less engine."""
    prompts = [list(range(1 + 50 * i, 27 + 50 * i)) for i in range(6)]
    sp = lambda: SamplingParams(max_new_tokens=4, temperature=0.0)

    eng0 = _engine()
    want = []
    for p in prompts:
        r = eng0.add_request(p, sp())
        while not eng0.is_finished():
            eng0.step()
        want.append(eng0.get_output(r).token_ids)

    eng = _engine(num_gpu_blocks=8, enable_prefix_caching=True)
    for p, w in zip(prompts, want):
        r = eng.add_request(p, sp())
        while not eng.is_finished():
            eng.step()
        assert eng.get_output(r).token_ids == w


def test_prefix_caching_composes_with_fork_and_preemption():
    """The three block-sharing machineries at once: a cache-hit prompt
    forked n>1 under a pool small enough to preempt — outputs still
    equal the plain engine's, and no blocks leak."""
    prompt = list(range(1, 40))
    sp = lambda n=8: SamplingParams(max_new_tokens=n, temperature=0.0)

    eng0 = _engine()
    r0 = eng0.add_request(prompt, sp())
    while not eng0.is_finished():
        eng0.step()
    want = eng0.get_output(r0).token_ids

    eng = _engine(num_gpu_blocks=12, max_num_seqs=8,
                  enable_prefix_caching=True)
    free0 = eng.block_manager.num_free
    warm = eng.add_request(prompt, sp(2))       # seed the prefix pool
    while not eng.is_finished():
        eng.step()
    assert eng.get_output(warm).token_ids == want[:2]
    rids = eng.add_request_group(prompt, sp(), n=3)
    steps = 0
    while not eng.is_finished():
        eng.step()
        steps += 1
        assert steps < 2000
    for r in rids:
        assert eng.get_output(r).token_ids == want
    assert eng.block_manager.prefix_hit_tokens >= 32
    assert eng.block_manager.num_free == free0


def test_preempted_sequence_reuses_its_own_retained_blocks():
    """After preemption, re-admission hash-hits the victim's own prompt
    blocks instead of recomputing them."""
    eng = _engine(num_gpu_blocks=6, max_num_seqs=4,
                  enable_prefix_caching=True)
    a = eng.add_request(list(range(1, 40)),
                        SamplingParams(max_new_tokens=8, temperature=0.0))
    eng.add_request(list(range(50, 76)),
                    SamplingParams(max_new_tokens=8, temperature=0.0))
    steps = 0
    while not eng.is_finished():
        eng.step()
        steps += 1
        assert steps < 2000
    assert eng.scheduler.num_preemptions > 0
    assert eng.block_manager.prefix_hit_tokens > 0
    assert len(eng.get_output(a).token_ids) == 8


def test_fuzz_block_accounting_invariants():
    """Randomized adds/forks/aborts with prefix caching on a tiny pool:
    after every drain the block accounting must be exactly conservative
    (every block is free, retained, or held by exactly its ref-count
    owners) and at the end everything is reclaimable."""
    import random as rnd

    r = rnd.Random(1234)
    eng = _engine(num_gpu_blocks=16, max_num_seqs=8,
                  enable_prefix_caching=True)
    bm = eng.block_manager
    prompts = [list(range(1 + 10 * i, 24 + 10 * i)) for i in range(4)]
    live = []
    for round_i in range(60):
        act = r.random()
        if act < 0.45 and len(live) < 10:
            p = r.choice(prompts)
            if r.random() < 0.3:
                live.extend(eng.add_request_group(
                    p, SamplingParams(max_new_tokens=r.randint(2, 8),
                                      temperature=0.8), n=2))
            else:
                live.append(eng.add_request(
                    p, SamplingParams(max_new_tokens=r.randint(2, 8),
                                      temperature=0.8)))
        elif act < 0.55 and live:
            eng.abort_request(r.choice(live))
        for _ in range(r.randint(1, 4)):
            if not eng.is_finished():
                eng.step()
        live = [x for x in live
                if not eng.get_output(x).finished]
        # invariant: refs are non-negative and every held ref is owned
        held = {}
        for seq in eng._seqs.values():
            for b in seq.block_ids:
                held[b] = held.get(b, 0) + 1
        for b in range(1, bm.num_blocks):
            assert bm._refs[b] >= 0
            assert bm._refs[b] == held.get(b, 0), (round_i, b)
    while not eng.is_finished():
        eng.step()
    for seq in eng._seqs.values():
        assert seq.state.name == "FINISHED"
    assert bm.num_free == bm.num_blocks - 1   # everything reclaimable


def test_chunked_prefill_equivalence():
    """Chunked prefill must be output-invariant: a prompt much longer
    than max_batched_tokens prefills in several rounds through the
    paged-extend path and produces exactly the unchunked tokens."""
    long_prompt = list(range(3, 200))         # 197 tokens
    short = list(range(7, 30))
    sp = lambda: SamplingParams(max_new_tokens=6, temperature=0.0)

    eng0 = _engine(max_batched_tokens=2048, num_gpu_blocks=64)
    r_l0 = eng0.add_request(long_prompt, sp())
    r_s0 = eng0.add_request(short, sp())
    while not eng0.is_finished():
        eng0.step()
    want_l = eng0.get_output(r_l0).token_ids
    want_s = eng0.get_output(r_s0).token_ids

    eng = _engine(max_batched_tokens=48, num_gpu_blocks=64,
                  enable_chunked_prefill=True)
    r_l = eng.add_request(long_prompt, sp())
    r_s = eng.add_request(short, sp())
    steps = 0
    while not eng.is_finished():
        eng.step()
        steps += 1
        assert steps < 500
    assert eng.get_output(r_l).token_ids == want_l
    assert eng.get_output(r_s).token_ids == want_s
    assert eng.block_manager.num_free == eng.block_manager.num_blocks - 1


def test_chunked_prefill_interleaves_decode():
    """While a long prompt prefills chunk by chunk, an in-flight stream
    must keep producing tokens between the chunks (TTFT fairness — the
    reason chunking exists)."""
    eng = _engine(max_batched_tokens=32, num_gpu_blocks=64,
                  enable_chunked_prefill=True)
    first = eng.add_request(
        list(range(1, 20)),
        SamplingParams(max_new_tokens=40, temperature=0.0))
    # let it prefill and decode a little
    for _ in range(4):
        eng.step()
    long_rid = eng.add_request(
        list(range(3, 160)),                  # ~5 chunks of 32
        SamplingParams(max_new_tokens=4, temperature=0.0))
    produced_during = 0
    for _ in range(8):
        outs = eng.step()
        produced_during += sum(1 for o in outs if o.seq_id == first)
    assert produced_during >= 3               # decode kept flowing
    while not eng.is_finished():
        eng.step()
    assert len(eng.get_output(long_rid).token_ids) == 4
    assert len(eng.get_output(first).token_ids) == 40


def test_chunked_prefill_composes_with_prefix_cache_and_fork():
    long_prompt = list(range(11, 170))
    sp = lambda: SamplingParams(max_new_tokens=5, temperature=0.0)
    eng0 = _engine()
    r0 = eng0.add_request(long_prompt, sp())
    while not eng0.is_finished():
        eng0.step()
    want = eng0.get_output(r0).token_ids

    eng = _engine(max_batched_tokens=64, enable_chunked_prefill=True,
                  enable_prefix_caching=True, num_gpu_blocks=64,
                  max_num_seqs=8)
    r1 = eng.add_request(long_prompt, sp())
    while not eng.is_finished():
        eng.step()
    assert eng.get_output(r1).token_ids == want
    # repeat: leading full blocks hit the cache, remainder chunks
    rids = eng.add_request_group(long_prompt, sp(), n=2)
    while not eng.is_finished():
        eng.step()
    for r in rids:
        assert eng.get_output(r).token_ids == want
    assert eng.block_manager.prefix_hit_tokens > 0


def test_abort_mid_chunk_releases_blocks():
    """Aborting a long prompt between prefill chunks (still WAITING but
    holding its reserved blocks) must release everything."""
    eng = _engine(max_batched_tokens=32, num_gpu_blocks=64,
                  enable_chunked_prefill=True)
    free0 = eng.block_manager.num_free
    rid = eng.add_request(list(range(3, 160)),
                          SamplingParams(max_new_tokens=4,
                                         temperature=0.0))
    eng.step()                                 # first chunk only
    seq = eng._seqs[rid]
    assert 0 < seq.prefilled < seq.prompt_len
    assert seq.block_ids
    eng.abort_request(rid)
    assert eng.get_output(rid).finish_reason == "abort"
    assert eng.block_manager.num_free == free0
    assert not eng.scheduler.has_work


def test_prefill_first_policy_admits_before_decode():
    """scheduler_prefill_first: waiting prompts are admitted in
    consecutive prefill rounds (no decode alternation) until the queue
    drains — the burst-TTFT policy; the default still alternates."""
    from inference_gateway_amd.engine.scheduler import Scheduler, Sequence

    def mk(policy):
        bm = BlockManager(256, 16)
        s = Scheduler(bm, max_num_seqs=16, max_batched_tokens=32,
                      max_model_len=256, prefill_first=policy)
        for i in range(4):
            s.add(Sequence(seq_id=i, prompt_token_ids=list(range(32)),
                           sampling=SamplingParams()))
        return s

    s = mk(True)
    kinds = []
    for _ in range(4):
        b = s.schedule()
        kinds.append("p" if b.is_prefill else "d")
        if b.is_prefill:
            for q, t in zip(b.seqs, b.prefill_takes):
                q.prefilled += t
    assert kinds == ["p", "p", "p", "p"]      # all admissions first

    s = mk(False)
    kinds = []
    for _ in range(4):
        b = s.schedule()
        kinds.append("p" if b.is_prefill else "d")
        if b.is_prefill:
            for q, t in zip(b.seqs, b.prefill_takes):
                q.prefilled += t
    assert kinds == ["p", "d", "p", "d"]      # alternation (default)


def test_abort_mid_chunk_does_not_poison_prefix_cache():
    """with chunked prefill + prefix caching,
    allocate_for_prompt hash-indexes ALL full prompt blocks up front;
    aborting before their KV is computed must un-index the unwritten
    ones, or a later identical prompt would claim garbage KV from the
    retained pool and silently generate wrong tokens."""
    long_prompt = list(range(11, 170))
    sp = lambda: SamplingParams(max_new_tokens=5, temperature=0.0)  # noqa
    eng0 = _engine()
    r0 = eng0.add_request(long_prompt, sp())
    while not eng0.is_finished():
        eng0.step()
    want = eng0.get_output(r0).token_ids

    eng = _engine(max_batched_tokens=32, enable_chunked_prefill=True,
                  enable_prefix_caching=True, num_gpu_blocks=64,
                  max_num_seqs=8)
    rid = eng.add_request(long_prompt, sp())
    eng.step()                                  # first chunk only
    seq = eng._seqs[rid]
    assert 0 < seq.prefilled < seq.prompt_len
    written = seq.prefilled
    eng.abort_request(rid)
    bm = eng.block_manager
    # every surviving hash must belong to a block whose KV was computed
    for (idx, _h, _chunk) in bm._by_hash:
        assert idx < written // bm.block_size
    # a fresh identical prompt must reproduce the reference tokens
    r1 = eng.add_request(long_prompt, sp())
    while not eng.is_finished():
        eng.step()
    assert eng.get_output(r1).token_ids == want


def test_moe_engine_with_chunked_prefix_and_fork():
    """Mixtral path (MoE MLP + shared LlamaAttention): chunked prefill,
    prefix caching and n>1 forks must be output-invariant there too."""
    from inference_gateway_amd.engine.config import EngineConfig as EC

    def run(cfg, prompt, n=1):
        torch.manual_seed(0)
        eng = LLMEngine(cfg, device="cpu")
        sp = SamplingParams(max_new_tokens=4, temperature=0.0)
        rids = (eng.add_request_group(prompt, sp, n=n) if n > 1
                else [eng.add_request(prompt, sp)])
        steps = 0
        while not eng.is_finished():
            eng.step()
            steps += 1
            assert steps < 1000
        return [eng.get_output(r).token_ids for r in rids]

    prompt = list(range(3, 120))
    want = run(EC.tiny_moe(), prompt)[0]
    got = run(EC.tiny_moe(max_batched_tokens=48,
                          enable_chunked_prefill=True,
                          enable_prefix_caching=True), prompt, n=2)
    assert all(g == want for g in got)


@pytest.mark.asyncio
async def test_async_engine_shutdown_unblocks_streams():
    """shutdown() while a stream is mid-generation must deliver the
    sentinel so the consumer ends instead of hanging."""
    import asyncio

    from inference_gateway_amd.engine.async_engine import AsyncEngine
    from inference_gateway_amd.engine.config import EngineConfig

    eng = AsyncEngine(EngineConfig.tiny_llama(), device="cpu")
    got = []

    async def consume():
        async for out in eng.generate(
                list(range(1, 20)),
                SamplingParams(max_new_tokens=10 ** 6, temperature=0.8,
                               ignore_eos=True)):
            got.append(out.token_id)
            if len(got) == 3:
                eng.shutdown()
    await asyncio.wait_for(consume(), timeout=30)
    assert len(got) >= 3


@pytest.mark.asyncio
async def test_async_engine_death_raises_not_clean_stop():
    """a fatal error on the engine thread must not
    look like a successful completion — open streams raise
    EngineDeadError (the gateway turns it into an in-stream error frame)
    and NEW requests fail fast."""
    import asyncio

    from inference_gateway_amd.engine.async_engine import (AsyncEngine,
                                                           EngineDeadError)
    from inference_gateway_amd.engine.config import EngineConfig

    eng = AsyncEngine(EngineConfig.tiny_llama(), device="cpu")

    def boom():
        raise RuntimeError("injected engine fault")

    n = 0
    gen = eng.generate(list(range(1, 20)),
                       SamplingParams(max_new_tokens=10 ** 6,
                                      temperature=0.8, ignore_eos=True))

    async def consume():
        nonlocal n
        async for _ in gen:
            n += 1
            if n == 2:
                eng.engine.step = boom    # next loop iteration dies
    with pytest.raises(EngineDeadError, match="injected engine fault"):
        await asyncio.wait_for(consume(), timeout=30)
    assert n >= 2
    assert isinstance(eng._fatal, RuntimeError)
    # new work is rejected immediately, not queued into a dead engine
    with pytest.raises(EngineDeadError):
        async for _ in eng.generate([1, 2, 3], SamplingParams()):
            pass
    with pytest.raises(EngineDeadError):
        eng.generate_group([1, 2, 3], SamplingParams(), 2)
    eng.shutdown()


@pytest.mark.asyncio
async def test_async_engine_batched_delivery_mode(monkeypatch):
    """IGW_BATCH_DELIVER=1 (the measured-slower opt-in experiment path)
    still delivers every token and the sentinel."""
    import asyncio

    from inference_gateway_amd.engine.async_engine import AsyncEngine
    from inference_gateway_amd.engine.config import EngineConfig

    monkeypatch.setenv("IGW_BATCH_DELIVER", "1")
    eng = AsyncEngine(EngineConfig.tiny_llama(), device="cpu")
    assert eng._batched_delivery
    try:
        toks = []

        async def consume():
            async for out in eng.generate(
                    list(range(1, 20)),
                    SamplingParams(max_new_tokens=6, temperature=0.0)):
                toks.append(out.token_id)
        await asyncio.wait_for(consume(), timeout=30)
        assert len(toks) == 6
    finally:
        eng.shutdown()


def test_mixed_batches_token_equivalence():
    """Same-step mixed prefill+decode rounds must be token-exact vs the
    plain engine: greedy decode of staggered arrivals produces identical
    outputs with enable_mixed_batches on and off."""
    def run(mixed):
        eng = _engine(max_batched_tokens=48, num_gpu_blocks=128,
                      max_num_seqs=8, enable_chunked_prefill=True,
                      enable_mixed_batches=mixed)
        sp = lambda: SamplingParams(max_new_tokens=10, temperature=0.0)  # noqa
        ra = eng.add_request(list(range(1, 40)), sp())
        for _ in range(3):
            eng.step()                  # A decoding (or prefilling)
        rb = eng.add_request(list(range(50, 170)), sp())   # long prompt
        rc = eng.add_request(list(range(7, 30)), sp())
        while not eng.is_finished():
            eng.step()
        return ([eng.get_output(r).token_ids for r in (ra, rb, rc)],
                eng.scheduler.num_mixed_rounds)

    plain, m0 = run(False)
    mixed, m1 = run(True)
    assert m0 == 0 and m1 > 0, (m0, m1)
    assert mixed == plain


def test_mixed_batches_no_itl_bubble():
    """While a long prompt prefills in chunks, running sequences keep
    generating EVERY round (no whole-round decode bubble)."""
    eng = _engine(max_batched_tokens=32, num_gpu_blocks=128,
                  max_num_seqs=8, enable_chunked_prefill=True,
                  enable_mixed_batches=True)
    ra = eng.add_request(list(range(1, 20)),
                         SamplingParams(max_new_tokens=64,
                                        temperature=0.0, ignore_eos=True))
    eng.step()                           # prefill A
    eng.step()                           # A decodes once
    na = len(eng.get_output(ra).token_ids)
    eng.add_request(list(range(50, 170)),
                    SamplingParams(max_new_tokens=4, temperature=0.0))
    # the long prompt needs ~4 chunked rounds at budget 32; A must gain
    # one token in EVERY one of them
    for i in range(4):
        before = len(eng.get_output(ra).token_ids)
        eng.step()
        after = len(eng.get_output(ra).token_ids)
        assert after == before + 1, (i, before, after)
    assert eng.scheduler.num_mixed_rounds >= 3
    assert len(eng.get_output(ra).token_ids) >= na + 4


def test_mixed_batches_with_prefix_cache_and_forks():
    """Mixed rounds compose with the other scheduler features."""
    long_prompt = list(range(11, 150))
    sp = lambda: SamplingParams(max_new_tokens=6, temperature=0.0)  # noqa
    eng0 = _engine()
    r0 = eng0.add_request(long_prompt, sp())
    while not eng0.is_finished():
        eng0.step()
    want = eng0.get_output(r0).token_ids

    eng = _engine(max_batched_tokens=48, num_gpu_blocks=128,
                  max_num_seqs=8, enable_chunked_prefill=True,
                  enable_prefix_caching=True, enable_mixed_batches=True)
    ra = eng.add_request(list(range(200, 230)), sp())
    eng.step()
    rids = eng.add_request_group(long_prompt, sp(), n=2)
    while not eng.is_finished():
        eng.step()
    for r in rids:
        assert eng.get_output(r).token_ids == want
    # repeat the prompt: prefix hits while other seqs decode mixed
    r2 = eng.add_request(long_prompt, sp())
    while not eng.is_finished():
        eng.step()
    assert eng.get_output(r2).token_ids == want
    assert eng.block_manager.prefix_hit_tokens > 0


def test_mixed_batches_moe_token_equivalence():
    """Mixed same-step rounds on the MoE engine (Mixtral path): the
    union forward routes decode rows through the MoE with the prefill
    flag — must stay token-exact vs the plain MoE engine."""
    def run(mixed):
        torch.manual_seed(0)
        cfg = EngineConfig.tiny_moe(
            max_batched_tokens=48, num_gpu_blocks=128, max_num_seqs=8,
            enable_chunked_prefill=True, enable_mixed_batches=mixed)
        eng = LLMEngine(cfg, device="cpu")
        sp = lambda: SamplingParams(max_new_tokens=8, temperature=0.0)  # noqa
        ra = eng.add_request(list(range(1, 30)), sp())
        for _ in range(3):
            eng.step()
        rb = eng.add_request(list(range(40, 150)), sp())
        while not eng.is_finished():
            eng.step()
        return ([eng.get_output(r).token_ids for r in (ra, rb)],
                eng.scheduler.num_mixed_rounds)

    plain, m0 = run(False)
    mixed, m1 = run(True)
    assert m0 == 0 and m1 > 0
    assert mixed == plain


def test_logit_bias_forces_and_bans_tokens():
    """OpenAI logit_bias: +100 forces a token under greedy decoding;
    -100 on the natural argmax bans it."""
    from inference_gateway_amd.engine.config import (EngineConfig,
                                                     SamplingParams)
    from inference_gateway_amd.engine.engine import LLMEngine

    eng = LLMEngine(EngineConfig.tiny_llama(), device="cpu")
    prompt = list(range(1, 17))

    def run(sp):
        rid = eng.add_request(prompt, sp)
        while not eng.is_finished():
            eng.step()
        return eng.get_output(rid).token_ids

    base = run(SamplingParams(max_new_tokens=4, temperature=0))
    forced = run(SamplingParams(max_new_tokens=4, temperature=0,
                                logit_bias={7: 100.0}))
    assert forced == [7, 7, 7, 7]
    banned = run(SamplingParams(max_new_tokens=1, temperature=0,
                                logit_bias={base[0]: -100.0}))
    assert banned[0] != base[0]
    # bias composes with penalties on the same request
    both = run(SamplingParams(max_new_tokens=3, temperature=0,
                              logit_bias={7: 100.0},
                              presence_penalty=0.1))
    assert both[0] == 7


def test_engine_fuzz_qwen2_bias_path():
    """The mixed-mode fuzz on the QKV-BIAS architecture (tiny-qwen2,
    tied embeddings): the bias path must hold the same pool/slot
    invariants under preemption, forks, prefix hits and aborts."""
    import random

    rng = random.Random(4242)
    torch.manual_seed(0)
    eng = LLMEngine(
        EngineConfig(model=MODEL_PRESETS["tiny-qwen2"], num_gpu_blocks=28,
                     max_model_len=96, max_num_seqs=4,
                     max_batched_tokens=48, enable_chunked_prefill=True,
                     enable_prefix_caching=True, enable_mixed_batches=True,
                     scheduler_prefill_first=True),
        device="cpu")
    bm = eng.block_manager
    free0 = bm.num_free
    slots0 = len(eng.scheduler._free_slots)
    shared = list(range(200, 248))
    live = []
    for step in range(250):
        r = rng.random()
        if r < 0.25 and len(live) < 8:
            prompt = (shared[: rng.choice([16, 32])]
                      + [rng.randrange(1, 500) for _ in range(
                          rng.randrange(1, 16))])
            live.append(eng.add_request(
                prompt,
                SamplingParams(max_new_tokens=rng.randrange(1, 8),
                               temperature=rng.choice([0.0, 0.8]),
                               logit_bias=rng.choice([None, {9: 60.0}]))))
        elif r < 0.32 and live:
            eng.abort_request(live.pop(rng.randrange(len(live))))
        for o in eng.step():
            if o.finished and o.seq_id in live:
                live.remove(o.seq_id)
    guard = 0
    while not eng.is_finished():
        guard += 1
        assert guard < 2000, "engine wedged during drain"
        for o in eng.step():
            if o.finished and o.seq_id in live:
                live.remove(o.seq_id)
    assert bm.num_free == free0, "leaked KV blocks"
    assert len(eng.scheduler._free_slots) == slots0, "leaked slots"


def test_step_watchdog_fails_streams_on_wedged_step(monkeypatch):
    """IGW_STEP_WATCHDOG: a step that WEDGES (no exception — e.g. a
    hung GPU queue) must fail waiting clients with EngineDeadError
    instead of hanging them forever."""
    import asyncio
    import threading
    import time

    from inference_gateway_amd.engine.async_engine import (AsyncEngine,
                                                           EngineDeadError)

    monkeypatch.setenv("IGW_STEP_WATCHDOG", "0.4")
    eng = AsyncEngine(EngineConfig.tiny_llama(num_gpu_blocks=16,
                                              max_model_len=64,
                                              max_num_seqs=2),
                      device="cpu")
    release = threading.Event()

    def wedged_step():
        release.wait(timeout=10)      # simulates a hung hipLaunch
        return []

    eng.engine.step = wedged_step
    try:
        async def go():
            with pytest.raises(EngineDeadError, match="watchdog"):
                async for _ in eng.generate(
                        list(range(1, 9)),
                        SamplingParams(max_new_tokens=2)):
                    pass

        t0 = time.monotonic()
        asyncio.run(go())
        assert time.monotonic() - t0 < 5, "watchdog took too long"
    finally:
        release.set()
        eng.shutdown()


def test_unschedulable_prompt_rejected_at_admission():
    """A prompt that can NEVER fit the KV pool is rejected per-request
    at add time (the engine survives; other requests keep serving)."""
    eng = _engine(num_gpu_blocks=6, max_model_len=96)
    with pytest.raises(ValueError, match="KV blocks"):
        eng.add_request(list(range(1, 90)),
                        SamplingParams(max_new_tokens=2, temperature=0))
    # the engine still serves a request that fits
    rid = eng.add_request(list(range(1, 17)),
                          SamplingParams(max_new_tokens=2, temperature=0))
    while not eng.is_finished():
        eng.step()
    assert eng.get_output(rid).finished


def test_generation_outgrowing_pool_fails_loudly():
    """The pathological fold case: a sequence whose PREEMPTION-FOLDED
    prompt can no longer fit must raise (no-progress detection), not
    busy-spin silently.  Requires pool < max_model_len — a
    misconfiguration the startup path cannot always rule out."""
    eng = _engine(num_gpu_blocks=6, max_model_len=96)
    eng.add_request(list(range(1, 41)),
                    SamplingParams(max_new_tokens=50, temperature=0))
    with pytest.raises(RuntimeError, match="no progress"):
        for _ in range(10000):
            eng.step()


def test_differential_plain_vs_full_stack_tie_aware():
    """Randomized differential: staggered greedy request sets through
    the PLAIN engine and the FULL feature stack (chunked + prefix +
    mixed + prefill-first) must match token-for-token — except where
    the two top logits sit within a couple of bf16 ULPs (mixed rounds
    change reduction shapes; a one-quantum argmax tie may flip and is
    NOT a scheduling/attention defect).  Any larger divergence fails."""
    import random

    def run(cfgkw, requests):
        torch.manual_seed(0)
        eng = LLMEngine(EngineConfig.tiny_llama(
            num_gpu_blocks=128, max_model_len=192, max_num_seqs=6,
            **cfgkw), device="cpu")
        rids = []
        added = 0
        while True:
            for _ in range(2):
                if added < len(requests):
                    pr, mnt = requests[added]
                    rids.append(eng.add_request(pr, SamplingParams(
                        max_new_tokens=mnt, temperature=0)))
                    added += 1
            if eng.is_finished() and added == len(requests):
                break
            eng.step()
        while not eng.is_finished():
            eng.step()
        return [eng.get_output(r).token_ids for r in rids]

    def logits_for(prompt):
        torch.manual_seed(0)
        eng = LLMEngine(EngineConfig.tiny_llama(
            num_gpu_blocks=128, max_model_len=192, max_num_seqs=6),
            device="cpu")
        cap = {}
        orig = eng.sampler.sample

        def spy(lg, seqs):
            cap["lg"] = lg.clone()
            return orig(lg, seqs)

        eng.sampler.sample = spy
        eng.add_request(prompt, SamplingParams(max_new_tokens=1,
                                               temperature=0))
        while not eng.is_finished():
            eng.step()
        return cap["lg"][0]

    rng = random.Random(99)
    shared = list(range(300, 348))
    for trial in range(8):
        reqs = []
        for _ in range(rng.randrange(3, 9)):
            stem = shared[: rng.choice([0, 16, 32])]
            pr = stem + [rng.randrange(1, 500)
                         for _ in range(rng.randrange(4, 40))]
            reqs.append((pr, rng.randrange(1, 12)))
        plain = run({}, reqs)
        full = run(dict(enable_chunked_prefill=True,
                        enable_prefix_caching=True,
                        enable_mixed_batches=True,
                        scheduler_prefill_first=True,
                        max_batched_tokens=48), reqs)
        for i, (a, b) in enumerate(zip(plain, full)):
            if a == b:
                continue
            # first divergence must be a near-tie
            j = next(k for k in range(min(len(a), len(b)))
                     if a[k] != b[k])
            prompt = list(reqs[i][0]) + a[:j]
            lg = logits_for(prompt)
            gap = abs((lg[a[j]] - lg[b[j]]).item())
            scale = max(abs(lg[a[j]].item()), 1.0)
            assert gap <= 0.0078125 * 2 * scale, (
                f"trial {trial} seq {i}: real divergence "
                f"{a} vs {b} (logit gap {gap})")


def test_finished_requests_are_evicted_from_bookkeeping(monkeypatch):
    """Serving-lifetime memory: finished Sequence bookkeeping is
    retained for only the last _FINISHED_RETENTION requests — a
    long-running server must not hold every prompt ever served.
    get_output stays valid within the retention window (sync API)."""
    eng = _engine()
    monkeypatch.setattr(type(eng), "_FINISHED_RETENTION", 8)
    rids = []
    for i in range(20):
        rid = eng.add_request(list(range(1, 9)),
                              SamplingParams(max_new_tokens=2,
                                             temperature=0))
        while not eng.is_finished():
            eng.step()
        assert eng.get_output(rid).finished    # valid right after
        rids.append(rid)
    assert len(eng._seqs) <= 8
    assert rids[0] not in eng._seqs            # oldest evicted
    assert rids[-1] in eng._seqs               # recent retained


def _prompt_batch(eng, rows):
    from inference_gateway_amd.engine.models.batch import ForwardBatch

    pos = torch.arange(rows, dtype=torch.int32)
    return ForwardBatch(token_ids=torch.arange(rows) + 1, positions=pos,
                        slot_mapping=pos + 16, is_prefill=True,
                        cu_seqlens=torch.tensor([0, rows], dtype=torch.int32),
                        seq_lens=[rows])


class Negated(torch.nn.Module):
    def __init__(self, m):
        super().__init__()
        self.m = m

    def forward(self, *a, **kw):
        return -self.m(*a, **kw)


@pytest.mark.parametrize("rows", [3, 9])
def test_llama_modules_are_called(rows):
    """A hook on any module of a layer runs, a module put in another's place is
    the one that is used, and what comes out is the same: the layers do without
    calls of their modules only where nobody can tell."""
    eng = _engine()
    model, fb = eng.model, _prompt_batch(eng, rows)
    want = model(fb, eng.kv_caches)
    layer = model.layers[1]
    for m in (layer, layer.attn, layer.attn.o_proj, layer.mlp,
              layer.mlp.down_proj):
        seen = []
        handles = (m.register_forward_hook(lambda *a: seen.append("after")),
                   m.register_forward_pre_hook(lambda *a: seen.append("to")))
        assert torch.equal(model(fb, eng.kv_caches), want)
        assert seen == ["to", "after"]
        for h in handles:
            h.remove()
    seen = []
    handle = torch.nn.modules.module.register_module_forward_hook(
        lambda m, *a: seen.append(m))
    assert torch.equal(model(fb, eng.kv_caches), want)
    handle.remove()
    assert {id(layer.mlp), id(layer.attn.o_proj), id(model.layers[0])} <= {
        id(m) for m in seen}

    for owner, name in ((layer.attn, "o_proj"), (layer, "mlp"),
                        (layer, "attn"), (layer.mlp, "down_proj")):
        m = getattr(owner, name)
        setattr(owner, name, Negated(m))
        other = model(fb, eng.kv_caches)
        setattr(owner, name, Negated(Negated(m)))
        assert torch.equal(model(fb, eng.kv_caches), want)
        setattr(owner, name, m)
        assert not torch.equal(other, want)
    assert torch.equal(model(fb, eng.kv_caches), want)


@pytest.mark.parametrize("preset", ["tiny_llama", "tiny_moe"])
def test_layers_one_by_one(preset):
    """A layer called by itself: what the residual lacks and the residual, its
    input left as it was."""
    from inference_gateway_amd import ops

    eng = LLMEngine(getattr(EngineConfig, preset)(), device="cpu")
    model, fb = eng.model, _prompt_batch(eng, 5)
    want = model(fb, eng.kv_caches)
    x = torch.nn.functional.embedding(fb.token_ids, model.embed)
    kept, first, residual = x.clone(), x, None
    for layer, kv in zip(model.layers, eng.kv_caches):
        x, residual = layer(x, residual, fb, kv, model.cos_sin)
    assert torch.equal(first, kept)
    got, _ = ops.fused_add_rmsnorm(x, residual, model.final_norm_w,
                                   model.cfg.norm_eps)
    assert torch.equal(got, want)


@pytest.mark.parametrize("rows", [3, 9])
def test_mixtral_modules_are_called(rows, monkeypatch):
    """As above; few: the route of a few tokens, which reads the router's weight."""
    from inference_gateway_amd import ops

    eng = LLMEngine(EngineConfig.tiny_moe(), device="cpu")
    model, fb = eng.model, _prompt_batch(eng, rows)
    layer = model.layers[1]

    def few(x, gate_up, down, idx, weights):
        y = torch.zeros_like(x, dtype=torch.float32)
        for t in range(x.shape[0]):
            for e, w in zip(idx[t].tolist(), weights[t]):
                y[t] += w * (ops.linear_silu_mul(x[t:t + 1], gate_up[e])
                             @ down[e].t())[0].float()
        return y.to(x.dtype)

    for fits in (False, True):
        monkeypatch.setattr(ops, "moe_few_fits", lambda *a: fits)
        monkeypatch.setattr(ops, "moe_few", few)
        want = model(fb, eng.kv_caches)
        for m in (layer, layer.attn, layer.attn.o_proj, layer.moe,
                  layer.moe.router):
            seen = []
            handle = m.register_forward_hook(lambda *a: seen.append(1))
            assert torch.equal(model(fb, eng.kv_caches), want)
            handle.remove()
            assert seen == [1]
        for owner, name in ((layer.attn, "o_proj"), (layer, "attn"),
                            (layer.moe, "router")):
            m = getattr(owner, name)
            setattr(owner, name, Negated(m))
            other = model(fb, eng.kv_caches)
            setattr(owner, name, m)
            assert not torch.equal(other, want)


def test_graph_padding_rows_write_nothing():
    """The rows that fill a captured batch all read page 0: none of them is
    written, also where they outnumber the sequences."""
    from inference_gateway_amd.engine.graph_runner import DecodeGraphRunner

    run = object.__new__(DecodeGraphRunner)
    run.cfg, run.pad_slot = EngineConfig.tiny_llama(), 4
    run.in_slot_idx = torch.tensor([2, 0, 4, 4, 4])
    run.slot_token = torch.tensor([11, 12, 13, 14, 0])
    run.slot_pos = torch.tensor([17, 0, 5, 0, 0], dtype=torch.int32)
    run.bt_slots = torch.tensor([[3, 7], [0, 0], [9, 0], [0, 0], [0, 0]],
                                dtype=torch.int32)
    for bucket in (2, 5):
        fb = run._build_fb(bucket)
        assert fb.slot_mapping.dtype == torch.int32
        assert fb.slot_mapping.tolist() == [9 * 16 + 5, 7 * 16 + 1,
                                            -1, -1, -1][:bucket]
        assert fb.ctx_lens.tolist() == [6, 18, 1, 1, 1][:bucket]


@pytest.mark.parametrize("rows,inside", [(1, True), (3, True), (4, False),
                                         (6, False), (7, False)])
def test_llama_rows_that_norm_inside_the_product(rows, inside, monkeypatch):
    """The norm runs inside the product that follows it where that is the faster
    way, up to three rows."""
    from inference_gateway_amd import ops

    eng, seen, real = _engine(), [], ops.norm_linear
    monkeypatch.setattr(ops, "norm_linear",
                        lambda *a, **kw: seen.append(1) or real(*a, **kw))
    eng.model(_prompt_batch(eng, rows), eng.kv_caches)
    assert len(seen) == (2 * len(eng.model.layers) if inside else 0)
