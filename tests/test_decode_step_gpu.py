"""The native decode step (`mlora_decode_step`: one C call per step, LoRA carried inside the GEMV / RoPE / RMSNorm
launches, graph replay) against the per-operator path and against the oracle."""
import numpy as np
import pytest
import torch

import oracle
from conftest import load_pkg
from helpers import check_tokens_against_oracle, oracle_model

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def _prefill(model, kv, prompts, adapter_ids, chunk=4):
    ops = load_pkg("ops")
    B, P = prompts.shape
    first = np.zeros(B, dtype=np.int32)
    for s in range(B):
        kv.add_sequence(s)
    for lo in range(0, B, chunk):
        sids = list(range(lo, min(B, lo + chunk)))
        kv.begin_forward(sids, [P] * len(sids))
        h = model.embed(torch.from_numpy(np.ascontiguousarray(prompts[sids].reshape(-1))))
        ids = np.repeat(adapter_ids[sids], P).astype(np.int32)
        logits = model.forward(h, kv, model._ids(len(ids), {0: (None, ids)}), model._last_rows(kv))
        kv.end_forward()
        first[sids] = ops.argmax(logits).cpu().numpy()
    return first


def _run(model, wl, prompts, ids, kind, steps, synth, run_steps=None):
    dsm = load_pkg("decode_session")
    blocks = -(-(wl.prompt_len + steps + 2) // 16)
    perm = synth.permutation(wl.seed, "pages", wl.batch * blocks)
    kv = model.create_paged_kv_cache(wl.batch, wl.batch * blocks * 16, wl.prompt_len, 16, free_pages=perm, max_seq_len=blocks * 16)
    first = _prefill(model, kv, prompts, ids)
    seqs = list(range(wl.batch))
    if kind == "py":
        s = dsm.DecodeSession(model, kv, seqs, {0: ids}, first)
    else:
        s = dsm.NativeDecodeSession(model, kv, seqs, ids, first, use_graph=(kind == "graph"), dense_lora=(kind == "dense"))
    toks = [first.copy()]
    logits0 = None
    for i in range(steps if run_steps is None else run_steps):
        toks.append(s.step().cpu().numpy().copy())
        if i == 0 and kind != "py":
            logits0 = s.buf["logits"].view(wl.batch, -1).clone()
    return np.stack(toks), kv.k.clone(), logits0


@pytest.mark.parametrize("targets,r,layers,steps", [
    (("q_proj", "k_proj", "v_proj", "o_proj"), 16, 3, 20),        # the benchmark's adapter placement; crosses a page boundary
    (("q_proj", "v_proj"), 8, 2, 6),                                # the reference's placement (compile_tvm.py:180-181)
    (("q_proj", "k_proj", "v_proj", "o_proj", "gate_proj", "up_proj", "down_proj"), 64, 2, 5),
    (("o_proj", "down_proj"), 32, 2, 5),
])
def test_native_step_equals_per_operator_path(targets, r, layers, steps):
    """Llama-7B-shape layers, 32 requests over 16 adapters (two requests without adapter).
    Shrink units riding in the GEMV launch + fused expands: token ids AND the whole K cache are bit-identical to
    the per-operator path, with and without graph replay.  Dense shrink (A tables as extra GEMV rows) changes
    the fp32 summation order of v, so it is compared at rounding-flip tolerance."""
    synth, llama = load_pkg("synth"), load_pkg("llama")
    wl = synth.config3(num_layers=layers, prompt_len=60)
    wl.lora = synth.LoraSpec(r=r, alpha=r / 2, n_adapters=16, targets=targets)
    ids = wl.adapter_ids.copy()
    ids[5] = ids[9] = -1
    model = llama.LlamaForCausalLM.from_synthetic(wl.seed, wl.shape, [wl.lora], DEV)
    prompts = synth.prompts(wl)
    a, ka, _ = _run(model, wl, prompts, ids, "py", steps, synth)
    b, kb, _ = _run(model, wl, prompts, ids, "native", steps, synth)
    c, kc, lg = _run(model, wl, prompts, ids, "graph", steps, synth)
    assert np.array_equal(a, b) and np.array_equal(a, c)
    assert torch.equal(ka, kb) and torch.equal(ka, kc)
    d, kd, ld = _run(model, wl, prompts, ids, "dense", steps, synth, run_steps=1)
    c1, kc1, _ = _run(model, wl, prompts, ids, "native", steps, synth, run_steps=1)
    err = float((ld - lg).abs().max() / lg.std())
    assert err <= 1e-2, err                                   # first step: logits agree to rounding-flip noise
    # cached keys/values: a rounding flip in one layer perturbs every later fp16 rounding at the ulp level, so only
    # the size of the difference is bounded (a few fp16 ulps), not the number of elements that differ
    assert float((kc1.float() - kd.float()).abs().max()) <= 2.0 ** -6        # values are O(1): ulp 2^-10 .. 2^-8
    margin = torch.topk(lg, 2, dim=-1).values
    decided = (margin[:, 0] - margin[:, 1]) >= 2e-2 * lg.std(dim=-1)
    assert np.array_equal(d[1][decided.cpu().numpy()], c[1][decided.cpu().numpy()])


def test_native_step_against_oracle_c3_shape():
    """Llama-7B-shape, 2 layers, 32 requests x 16 rank-16 adapters on q/k/v/o, random page order: prefill +
    greedy decode of the native (dense-shrink, graph) path against the CPU oracle, teacher-forced."""
    synth, llama, dsm = load_pkg("synth"), load_pkg("llama"), load_pkg("decode_session")
    wl = synth.config3(num_layers=2, batch=32, prompt_len=40, gen_len=6)
    model = llama.LlamaForCausalLM.from_synthetic(wl.seed, wl.shape, [wl.lora], DEV)
    prompts = synth.prompts(wl)
    max_gen_len = wl.gen_len + 1
    blocks = -(-(wl.prompt_len + max_gen_len + 1) // 16)
    perm = synth.permutation(wl.seed, "pages.oracle", wl.batch * blocks)
    ref = oracle_model(wl, "mixed")
    exp, margins, scales = oracle.greedy_generate_ref(ref, prompts, {"a0": wl.adapter_ids}, max_gen_len, wl.batch * blocks,
                                                      16, perm, return_logits=True)
    kv = model.create_paged_kv_cache(wl.batch, wl.batch * blocks * 16, wl.prompt_len, 16, free_pages=perm, max_seq_len=blocks * 16)
    # the oracle prefills sequence by sequence, so pages are handed out in the same order with chunk=1
    first = _prefill(model, kv, prompts, wl.adapter_ids, chunk=1)
    got = [[int(first[b])] for b in range(wl.batch)]
    sess = dsm.NativeDecodeSession(model, kv, list(range(wl.batch)), wl.adapter_ids, first, use_graph=True)
    for i in range(1, max_gen_len):
        sess.tokens.copy_(torch.tensor([exp[b][i - 1] for b in range(wl.batch)], dtype=torch.int32))   # teacher forcing
        nxt = sess.step().cpu().numpy()
        for b in range(wl.batch):
            got[b].append(int(nxt[b]))
    ties = check_tokens_against_oracle(got, exp, margins, scales)
    print("near-tie disagreements:", ties)
    assert len(ties) <= 1          # measured: one of the 32 x 7 decisions, request 21 at step 5, a near tie of the oracle


def test_full_depth_benchmark_model_native_equals_per_operator():
    """The benchmark model at full size (32 layers, hidden 4096, 32 requests x 16 rank-16 adapters on q/k/v/o): the
    graph-replayed native step (ids-based shrink) reproduces the per-operator path bit for bit - greedy tokens of
    every step and the whole K cache - which is the size-independent property that ties the benchmarked path to
    the operators checked against the oracle one by one; the dense-shrink variant the benchmark runs agrees on
    every token whose top-2 margin is decided."""
    synth, llama = load_pkg("synth"), load_pkg("llama")
    steps = 4
    wl = synth.config3(num_layers=32, prompt_len=48)
    model = llama.LlamaForCausalLM.from_synthetic(wl.seed, wl.shape, [wl.lora], DEV)
    prompts = synth.prompts(wl)
    ids = wl.adapter_ids
    a, ka, _ = _run(model, wl, prompts, ids, "py", steps, synth)
    c, kc, lg = _run(model, wl, prompts, ids, "graph", steps, synth)
    assert np.array_equal(a, c)
    assert torch.equal(ka, kc)
    del ka, kc
    d, _, ld = _run(model, wl, prompts, ids, "dense", steps, synth, run_steps=1)
    err = float((ld - lg).abs().max() / lg.std())
    print(f"32 layers: dense-shrink vs ids-based first-step logits differ by {err:.2e} of the logit std")
    assert err <= 2e-2
    margin = torch.topk(lg, 2, dim=-1).values
    decided = ((margin[:, 0] - margin[:, 1]) >= 2e-2 * lg.std(dim=-1)).cpu().numpy()
    assert np.array_equal(d[1][decided], c[1][decided])


def test_native_step_between_33_and_64_requests():
    """48 requests (four token tiles: four row tiles per wave in the GEMV with the reduction in two passes, K split,
    the per-unit SiLU kernel at four token tiles): the native step reproduces the per-operator path bit for bit,
    tokens and K cache."""
    synth, llama = load_pkg("synth"), load_pkg("llama")
    wl = synth.config3(num_layers=2, batch=48, prompt_len=30)
    ids = wl.adapter_ids.copy()
    ids[11] = -1
    model = llama.LlamaForCausalLM.from_synthetic(wl.seed, wl.shape, [wl.lora], DEV)
    prompts = synth.prompts(wl)
    a, ka, _ = _run(model, wl, prompts, ids, "py", 5, synth)
    c, kc, lg = _run(model, wl, prompts, ids, "graph", 5, synth)
    assert np.array_equal(a, c)
    assert torch.equal(ka, kc)
    d, _, ld = _run(model, wl, prompts, ids, "dense", 5, synth, run_steps=1)
    err = float((ld - lg).abs().max() / lg.std())
    assert err <= 1e-2, err


@pytest.mark.parametrize("batch,targets,r", [(65, ("q_proj", "k_proj", "v_proj", "o_proj"), 16), (128, ("q_proj", "v_proj"), 8),
                                              (256, ("q_proj", "k_proj", "v_proj", "o_proj", "gate_proj", "up_proj", "down_proj"), 16),
                                              (100, (), 16)])
def test_native_step_for_more_than_64_requests(batch, targets, r):
    """Beyond the 64-token decode tile the native step issues one launch per operator (matrix-core linears on
    fragment-ordered activations, K slices on o_proj and down_proj, grouped matrix-core LoRA): tokens and the whole K
    cache are bit-identical to the per-operator path, eagerly and replayed from a graph, and the first step's logits
    agree with the oracle."""
    synth, llama = load_pkg("synth"), load_pkg("llama")
    wl = synth.config3(num_layers=2, batch=batch, prompt_len=20)
    lora = synth.LoraSpec(r=r, alpha=float(r), n_adapters=24, targets=targets or ("q_proj",))
    ids = synth.randint(wl.seed, f"wide.ids{batch}", (batch,), 24).numpy().astype(np.int32)
    ids[[3, batch - 1]] = -1
    if not targets:
        ids[:] = -1
    wl = synth.Workload("wide", wl.seed, wl.shape, lora, batch=batch, prompt_len=20, gen_len=6, adapter_ids=ids)
    model = llama.LlamaForCausalLM.from_synthetic(wl.seed, wl.shape, [wl.lora], DEV)
    prompts = synth.prompts(wl)
    steps = 5
    a, ka, _ = _run(model, wl, prompts, ids, "py", steps, synth)
    b, kb, lg = _run(model, wl, prompts, ids, "native", steps, synth)
    c, kc, _ = _run(model, wl, prompts, ids, "graph", steps, synth)
    assert np.array_equal(a, b) and np.array_equal(a, c)
    assert torch.equal(ka, kb) and torch.equal(ka, kc)
    with pytest.raises(ValueError, match="dense"):
        _run(model, wl, prompts, ids, "dense", steps, synth, run_steps=1)
    # the first decode step against the oracle, from the oracle's own prefill of the same prompts
    ref = oracle_model(wl, "mixed")
    blocks = -(-(wl.prompt_len + steps + 2) // 16)
    kvr = ref.new_cache(batch * blocks, 16, blocks * 16, synth.permutation(wl.seed, "pages", batch * blocks))
    for q in range(batch):
        kvr.add_sequence(q)
    kvr.begin_forward(list(range(batch)), [wl.prompt_len] * batch)
    ref.forward(prompts.reshape(-1), kvr, {"a0": np.repeat(ids, wl.prompt_len)}, logits_rows=np.arange(batch))
    kvr.end_forward()
    kvr.begin_forward(list(range(batch)), [1] * batch)
    exp = ref.forward(a[0], kvr, {"a0": ids})
    kvr.end_forward()
    err = float(np.abs(lg.float().cpu().numpy() - exp).max() / exp.std())
    print(f"{batch} requests, first native step vs oracle: {err:.2e} of the logit std", flush=True)
    assert err <= 1e-2


def test_native_step_at_most_16_requests():
    """12 requests at the benchmark model's layer shapes (one token tile: the one-tile forms of the per-unit q/k/v and
    SiLU GEMVs, K-range blocks of the appended adapter rows): the native step reproduces the per-operator path bit for
    bit, and the dense-shrink variant agrees with it within rounding."""
    synth, llama = load_pkg("synth"), load_pkg("llama")
    wl = synth.config3(num_layers=2, batch=12, prompt_len=30)
    ids = wl.adapter_ids.copy()
    ids[5] = -1
    model = llama.LlamaForCausalLM.from_synthetic(wl.seed, wl.shape, [wl.lora], DEV)
    prompts = synth.prompts(wl)
    a, ka, _ = _run(model, wl, prompts, ids, "py", 5, synth)
    c, kc, lg = _run(model, wl, prompts, ids, "graph", 5, synth)
    assert np.array_equal(a, c)
    assert torch.equal(ka, kc)
    d, _, ld = _run(model, wl, prompts, ids, "dense", 5, synth, run_steps=1)
    err = float((ld - lg).abs().max() / lg.std())
    assert err <= 1e-2, err


@pytest.mark.parametrize("ranks,dense", [((8, 16), False), ((8, 16), True), ((32, 8, 16), False)])
def test_native_step_over_the_padded_union_of_adapter_types(ranks, dense):
    """Several adapter types of one scaling in one batch, served by the native step from their zero-padded union
    (the reference's padded strategy, `tvm/lora_only/case_study/multiple_ranks.py:66-95`), beside rows without
    adapter.  The padding adds exact zeros: with the ids-based shrink the tokens and the whole K cache equal those of
    the per-operator path on the unpadded tables bit for bit; with the dense shrink (x . A^T by the matrix cores,
    another fp32 summation order) the first step's logits and keys agree with the ids-based ones to rounding noise."""
    synth, llama, dsm = load_pkg("synth"), load_pkg("llama"), load_pkg("decode_session")
    wl = synth.config3(num_layers=2, batch=20, prompt_len=24)
    all7 = ("q_proj", "k_proj", "v_proj", "o_proj", "gate_proj", "up_proj", "down_proj")
    targets = (("q_proj", "k_proj", "v_proj", "o_proj"), ("q_proj", "v_proj", "down_proj"), all7)
    specs = [synth.LoraSpec(r=r, alpha=r / 2, n_adapters=3 + i, targets=targets[i]) for i, r in enumerate(ranks)]
    model = llama.LlamaForCausalLM.from_synthetic(wl.seed, wl.shape, specs, DEV)
    B = wl.batch
    steps = 1 if dense else 10
    tid = np.array([(b % (len(ranks) + 1)) - 1 for b in range(B)])              # -1 = no adapter
    ids = {t: np.where(tid == t, np.arange(B) % specs[t].n_adapters, -1).astype(np.int32) for t in range(len(ranks))}
    prompts = synth.randint(wl.seed, "union.prompts", (B, wl.prompt_len), wl.shape.vocab_size).numpy()
    first = np.arange(B, dtype=np.int32) + 7
    tids = tuple(range(len(ranks)))
    out = {}
    for kind in ("dense", "native") if dense else ("py", "native"):
        blocks = -(-(wl.prompt_len + steps + 2) // 16)
        kv = model.create_paged_kv_cache(B, B * blocks * 16, wl.prompt_len, 16, free_pages=synth.permutation(wl.seed, "union.pages", B * blocks),
                                         max_seq_len=blocks * 16)
        for b in range(B):
            kv.add_sequence(b)
        for b in range(B):           # prefill through the per-operator path, one request at a time
            kv.begin_forward([b], [wl.prompt_len])
            rows = {t: (None, np.full(wl.prompt_len, ids[t][b], dtype=np.int32)) for t in ids}
            model.forward(model.embed(torch.from_numpy(np.ascontiguousarray(prompts[b]))), kv, model._ids(wl.prompt_len, rows),
                          model._last_rows(kv))
            kv.end_forward()
        if kind == "py":
            s = dsm.DecodeSession(model, kv, list(range(B)), ids, first)
        else:
            s = dsm.NativeDecodeSession(model, kv, list(range(B)), model.union_rows(tids, B, {t: (None, ids[t]) for t in ids}), first,
                                        tid=tids, use_graph=not dense, dense_lora=(kind == "dense"))
            assert s.dense_lora == (kind == "dense")
        toks = [s.step().cpu().numpy().copy() for _ in range(steps)]
        out[kind] = (np.stack(toks), kv.k.clone(), None if kind == "py" else s.buf["logits"].view(B, -1).clone())
    if not dense:
        assert np.array_equal(out["py"][0], out["native"][0])
        assert torch.equal(out["py"][1], out["native"][1])
    else:
        for a, b in ((out["dense"][1].float(), out["native"][1].float()), (out["dense"][2], out["native"][2])):
            assert (a - b).abs().max().item() <= 2e-3 * b.abs().max().item()


def test_native_step_where_the_largest_k_needs_the_least_scratch():
    """Hidden size 4096 takes eight K slices, intermediate size 4608 five: every adapted projection finds room for its own, with separate
    shrink units and no dense tables; tokens and keys of the per-operator path."""
    synth, llama = load_pkg("synth"), load_pkg("llama")
    wl = synth.config3(num_layers=1, batch=5, prompt_len=20)
    wl.shape.intermediate_size = 4608
    wl.lora = synth.LoraSpec(r=64, alpha=32, n_adapters=3, targets=("q_proj", "k_proj", "v_proj", "o_proj", "gate_proj", "up_proj", "down_proj"))
    ids = np.array([0, 2, -1, 1, 0], dtype=np.int32)
    model = llama.LlamaForCausalLM.from_synthetic(wl.seed, wl.shape, [wl.lora], DEV)
    prompts = synth.prompts(wl)
    a, ka, _ = _run(model, wl, prompts, ids, "py", 3, synth)
    b, kb, _ = _run(model, wl, prompts, ids, "native", 3, synth)
    assert np.array_equal(a, b) and torch.equal(ka, kb)


@pytest.mark.parametrize("hidden,requests,vocab", [(32, 3, 96), (992, 17, 1004), (4096, 64, 300), (4128, 5, 1024), (8224, 2, 4100)])
def test_native_step_begins_and_ends_as_its_operators(hidden, requests, vocab):
    """Embedding and first norm in one launch with one, two and three of eight columns a thread, argmax with the counters: tokens and the whole
    cache of four steps are the per-operator path's, bit for bit."""
    synth, llama, dsm, ops = (load_pkg(n) for n in ("synth", "llama", "decode_session", "ops"))
    shape = synth.LlamaShape(hidden_size=hidden, intermediate_size=64, num_attention_heads=2, num_key_value_heads=2, num_hidden_layers=1, head_dim=64,
                             vocab_size=vocab)
    model = llama.LlamaForCausalLM.from_synthetic(7, shape, [], DEV)
    first = np.random.default_rng(hidden).integers(0, vocab, requests).astype(np.int32)
    got = []
    for native in (False, True):
        kv = model.create_paged_kv_cache(requests, requests * 32, 16, 16, free_pages=list(range(requests * 2)), max_seq_len=32)
        for s in range(requests):
            kv.add_sequence(s)
        seqs = list(range(requests))
        s = dsm.NativeDecodeSession(model, kv, seqs, np.full(requests, -1, np.int32), first) if native else dsm.DecodeSession(model, kv, seqs, {}, first)
        got.append(([s.step().cpu().numpy().copy() for _ in range(4)], kv.k.clone(), kv.v.clone()))
    for a, b in zip(*[g[0] for g in got]):
        assert np.array_equal(a, b)
    assert torch.equal(got[0][1], got[1][1]) and torch.equal(got[0][2], got[1][2])


ALL = ("q_proj", "k_proj", "v_proj", "o_proj", "gate_proj", "up_proj", "down_proj")


@pytest.mark.parametrize("B,r,targets,dense", [(1, 32, ("q_proj", "v_proj"), False), (6, 16, ALL, False), (17, 8, ALL, False), (33, 64, ALL, False), (64, 32, ("o_proj", "down_proj"), False),
                                               (48, 16, ("q_proj", "up_proj"), False), (20, 16, ALL, True)])
def test_native_step_with_deltas_in_launches_of_their_own(B, r, targets, dense):
    """Steps whose tokens share adapters, on both sides of the rule: tokens and the whole K cache of the per-operator path, bit for bit, and logits that
    agree with the riding forms to rounding; beside appended rows, gate and up alone."""
    synth, llama, dsm = load_pkg("synth"), load_pkg("llama"), load_pkg("decode_session")
    shape = synth.LlamaShape(hidden_size=1024, intermediate_size=1408, num_attention_heads=8, num_key_value_heads=4, num_hidden_layers=2, head_dim=128, vocab_size=600)
    model = llama.LlamaForCausalLM.from_synthetic(9, shape, [synth.LoraSpec(r=r, alpha=r / 2, n_adapters=4, targets=targets)], DEV)
    ids = (np.arange(B) % 7 // 6).astype(np.int32)             # most name adapter 0
    ids[B // 2] = -1 if B > 1 else 0
    most = llama.share_of(B, 4)
    assert most * 4 >= B > (most - 1) * 4 and model.segments_pay(B, most, 0) == (r >= 32 or most * r >= 96)
    got = {}
    for kind in ("py", "native", "graph", "riding"):
        kv = model.create_paged_kv_cache(B, B * 64, 32, 16, max_seq_len=64)
        first = _prefill(model, kv, synth.randint(2, "own", (B, 20), 600).numpy(), ids)
        if kind == "py":
            s = dsm.DecodeSession(model, kv, list(range(B)), {0: ids}, first)
        else:
            s = dsm.NativeDecodeSession(model, kv, list(range(B)), ids, first, use_graph=kind == "graph", dense_lora=dense)
            if kind == "riding":
                s.plan.lora_segments = 0
        toks = [s.step().cpu().numpy().copy()]
        logits = None if kind == "py" else s.buf["logits"].clone()
        toks += [s.step().cpu().numpy().copy() for _ in range(3)]
        got[kind] = (np.stack(toks), kv.k.clone(), logits)
    if not dense:
        assert np.array_equal(got["py"][0], got["native"][0]) and torch.equal(got["py"][1], got["native"][1])
    assert np.array_equal(got["graph"][0], got["native"][0]) and torch.equal(got["graph"][1], got["native"][1])
    a, b = got["native"][2], got["riding"][2]
    assert float((a - b).abs().max() / b.std()) <= 1e-2


@pytest.mark.parametrize("B,r,targets,n_ad,dense", [(6, 16, ALL, 2, False), (12, 8, ("q_proj", "o_proj"), 3, False), (14, 64, ALL, 9, False), (20, 16, ALL, 1, False), (20, 64, ALL, 30, False),
                                                    (41, 32, ALL, 16, False), (8, 16, ALL, 12, True), (24, 8, ALL, 7, True)])
def test_a_request_keeps_its_bits_in_any_row_beside_any_others(B, r, targets, n_ad, dense):
    """Logits and keys of some requests of a step, in three batches of the same size: as they are, the rows in reverse order, and beside requests that name other
    adapters, one or none."""
    synth, llama, dsm = load_pkg("synth"), load_pkg("llama"), load_pkg("decode_session")
    shape = synth.LlamaShape(hidden_size=1024, intermediate_size=1408, num_attention_heads=8, num_key_value_heads=4, num_hidden_layers=2, head_dim=128, vocab_size=600)
    model = llama.LlamaForCausalLM.from_synthetic(9, shape, [synth.LoraSpec(r=r, alpha=r / 2, n_adapters=n_ad, targets=targets)], DEV)
    prompts = synth.randint(2, "bits", (B, 20), 600).numpy()
    ids = (np.arange(B) * 5 % (n_ad + 1) - 1).astype(np.int32)
    kept = [0, B // 2, B - 1]
    got = {}
    for name in ("as is", "reversed", "one", "others", "none"):
        who = {"one": np.full(B, n_ad - 1), "others": (np.arange(B) * 3 + 1) % n_ad, "none": np.full(B, -1)}.get(name, ids).astype(np.int32)
        who[kept] = ids[kept]
        rows = list(range(B))[::-1] if name == "reversed" else list(range(B))
        for native in (True, False) if not dense else (True,):
            kv = model.create_paged_kv_cache(B, B * 64, 32, 16, max_seq_len=64)
            first = _prefill(model, kv, prompts, who, chunk=1)
            if native:
                s = dsm.NativeDecodeSession(model, kv, rows, who[rows], first[rows], use_graph=False, dense_lora=dense)
            else:
                s = dsm.DecodeSession(model, kv, rows, {0: who[rows]}, first[rows])
            logits = []
            for _ in range(3):
                s.step()
                logits += [s.buf["logits"].view(B, -1)[[rows.index(q) for q in kept]]] if native else []
            pages = torch.tensor(np.stack([kv.table_h[kv.slot[q]][:2] for q in kept]), device=DEV).reshape(-1).long()
            got.setdefault(native, []).append((kv.k[:, pages].clone(), s.tokens[[rows.index(q) for q in kept]].clone(), *logits))
    for runs in got.values():
        for other in runs[1:]:
            for a, b in zip(runs[0], other):
                assert torch.equal(a, b)


@pytest.mark.parametrize("r,B", [(16, 5), (32, 5), (64, 24), (16, 30)])
def test_requests_without_adapter_beside_one_type(r, B):
    """One adapter type and rows without: the call per step (`mixed_decode_a0`), the session of the front end and the native step have the same tokens and
    keys, whether a batch's ids are on the host or not."""
    synth, llama, dsm, ops = load_pkg("synth"), load_pkg("llama"), load_pkg("decode_session"), load_pkg("ops")
    shape = synth.LlamaShape(hidden_size=1024, intermediate_size=1408, num_attention_heads=8, num_key_value_heads=4, num_hidden_layers=2, head_dim=128, vocab_size=600)
    model = llama.LlamaForCausalLM.from_synthetic(9, shape, [synth.LoraSpec(r=r, alpha=r / 2, n_adapters=2, targets=ALL)], DEV)
    prompts, ids = synth.randint(2, "bare", (B, 20), 600).numpy(), (np.arange(B) % 4 // 3 * 2 - 1).astype(np.int32) * -1
    ids[1] = -1
    has, got = np.flatnonzero(ids >= 0), []
    for kind in ("steps", "session", "native", "native, of a tuple"):
        kv = model.create_paged_kv_cache(B, B * 64, 32, 16, max_seq_len=64)
        toks = [_prefill(model, kv, prompts, ids)]
        rows = list(range(B))
        if kind == "steps":
            for _ in range(4):
                kv.begin_forward(rows, [1] * B)
                logits, _ = model["mixed_decode_a0"](model.embed(torch.from_numpy(toks[-1])), kv, has, ids[has])
                kv.end_forward()
                toks.append(ops.argmax(logits).cpu().numpy())
        else:
            if kind == "session":
                s = dsm.DecodeSession(model, kv, rows, model._ids(B, {0: (has, ids[has])}), toks[0])
            elif kind == "native":
                s = dsm.NativeDecodeSession(model, kv, rows, ids, toks[0], dense_lora=False)
            else:
                s = dsm.NativeDecodeSession(model, kv, rows, model.union_rows((0,), B, {0: (has, ids[has])}), toks[0], tid=(0,), dense_lora=False)
            toks += [s.step().cpu().numpy().copy() for _ in range(4)]
        got.append((np.stack(toks), kv.k.clone()))
    for toks, k in got[1:]:
        assert np.array_equal(toks, got[0][0]) and torch.equal(k, got[0][1])
