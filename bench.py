"""Benchmark of the speculative-decoding hot path on one MI355X.

Headline (`value`): emitted tokens/s of greedy speculative decoding at batch 1
with k = 4 and paged KV (block size 16); target with SmolLM2-1.7B shapes, draft
with SmolLM2-135M shapes, random-init bf16 weights, a 256-token seeded prompt,
128 new tokens.  One step = one `generate` call.  The line's `e2e` object adds
the request's roofline fraction (algorithmic bytes of every forward of the
request -- weights read as stored, K/V read and written -- over its wall time),
plain greedy decoding on the same GPU, per-round p50/p99 latencies, a
truncated-target draft sweep and a copy draft (acceptance 1).

`roofline`: the verify paged-attention kernel at B = 8, context 4096, 32/32
heads of 64, 5 query tokens, shuffled block table (config 2's largest batch):
algorithmic bytes per launch (K+V of 8 x 4101 positions + Q in + O out + block
tables) over the mean launch time, from HIP events on the launching stream
around graph replays of back-to-back launches.  B = 1 sits beside it.

`cpu_baseline`: the oracle's CPU restatement of the reference loop (gather +
SDPA forward, host accept-reject) on the same weights and prompt, its rounds
interleaved one for one with the GPU loop's rounds, warm-up rounds excluded,
p50/p99 per round.

`batched_sampled`: config 5 -- batches of 8 and 32, T = 0.8, k = 4 and 8,
1024-token prompts with planted repetition decoded to a 4096-token context,
model and n-gram drafters -- with in-loop accept-kernel, verify and attention
times.  `kernels`: per-kernel times for configs 1-3 and 2' (accept-reject at
V = 49152, n-gram lookup at batch 16, cache append and rollback, attention over
the batch x context grid), each with its algorithmic bytes and GB/s.

Usage: python bench.py [--gpus 1] [--steps K] [--warmup W] [--only ...]
"""
from __future__ import annotations

import argparse
import json
import os
import statistics
import subprocess
import sys
import threading
import time
from pathlib import Path

ROOT = Path(__file__).resolve().parent
sys.path.insert(0, str(ROOT / "speculative-decoder_amd"))

import torch  # noqa: E402

HBM_PEAK_GBS = 8000.0
HOST_WAIT = "default"  # how the host waits for the GPU (main() may switch HIP to spinning)
# HBM bytes per launch of the B=8, context-4096 verify attention (one tiled
# launch) from earlier counter runs of the current kernel: rocprofv3
# FETCH_SIZE + WRITE_SIZE of `bench.py --only attention --batch 8`, each
# scaled by what the counter reads for a copy of known size.  The default run
# measures the figure itself (measure_attention_traffic); this one is reported
# only when that measurement fails, and the line says which it is.
ATTN_B8_TRAFFIC = 270_692_966
COPY_BYTES = 256 << 20  # the copy of known size the counters are scaled by
STORED_TRAFFIC_SOURCE = ("rocprofv3 --pmc FETCH_SIZE then WRITE_SIZE runs of `bench.py --only attention --batch 8` "
                         "(x2.0 / x1.0, the factors a 256 MiB copy gives), not counters read during this run")
V = 49152
PROMPT = 256
NEW_TOKENS = 128
K = 4
BLOCK = 16


def log(msg: str) -> None:
    print(f"[bench] {msg}", file=sys.stderr, flush=True)


def pct(xs: list[float], q: float) -> float:
    s = sorted(xs)
    return s[min(len(s) - 1, max(0, round(q / 100 * (len(s) - 1))))]


# ----------------------------------------------------------------- models ---
def build_models(dtype=torch.bfloat16, seed=0):
    from lm.model import SMOLLM2_135M, SMOLLM2_1_7B, Llama, random_state_dict

    dev = torch.device("cuda", 0)
    t_state = random_state_dict(SMOLLM2_1_7B, seed, dev, dtype)
    d_state = random_state_dict(SMOLLM2_135M, seed + 1, dev, dtype)
    return (Llama.from_state_dict(SMOLLM2_1_7B, t_state), Llama.from_state_dict(SMOLLM2_135M, d_state),
            t_state, d_state)


def prompt_ids(seed=0):
    g = torch.Generator().manual_seed(seed)
    return torch.randint(0, V, (PROMPT,), generator=g).tolist()


def caches_for(target, draft, batch=1, context=PROMPT + NEW_TOKENS, k=K):
    """Target and draft caches sized for `batch` rows of `context` tokens
    (+ the verify window); reused across requests, as a server would."""
    from cache.kv import KVCache

    blocks = batch * ((context + 2 * k + 2 * BLOCK) // BLOCK + 2) + 8
    return (KVCache.for_model(target.config, blocks, BLOCK, target.dtype, "cuda", ),
            KVCache.for_model(draft.config, blocks, BLOCK, draft.dtype, "cuda") if draft is not None else None)


def mean_accept_len(stats):
    """Accepted draft tokens per (sequence, round)."""
    return stats.accepted / max(len(stats.emitted_per_round), 1)


# ------------------------------------------------------ algorithmic bytes ---
def weight_bytes(llama) -> int:
    """Bytes of weights one forward reads as stored: every projection of every
    layer and the output head (embedding rows and norm vectors are noise)."""
    n = sum(t.numel() * t.element_size() for layer in llama.layers for t in (layer.wqkv, layer.wo, layer.wgu, layer.wd))
    return n + llama.head_wide.numel() * llama.head_wide.element_size()


def kv_bytes_per_position(llama) -> int:
    """K and V of one token position over every layer."""
    c = llama.config
    return c.num_hidden_layers * c.num_key_value_heads * c.head_dim * 2 * llama.embed.element_size()


def request_bytes(target, draft, prompt_len: int, stats, k: int) -> int:
    """Algorithmic HBM bytes of one batch-1 speculative request: the target's
    and the draft's prefill (weights once, K/V of the prompt written), then per
    round the k draft steps (weights + K/V read up to each step's position +
    its write) and the verify (weights + K/V read + k+1 written).  Contexts
    follow the request's own emitted_per_round."""
    tw, dw = weight_bytes(target), (weight_bytes(draft) if draft is not None else 0)
    tkv, dkv = kv_bytes_per_position(target), (kv_bytes_per_position(draft) if draft is not None else 0)
    total = tw + dw + prompt_len * (tkv + dkv)
    ctx = prompt_len + 1  # the first token comes from the target's prefill
    for emitted in stats.emitted_per_round:
        total += k * dw + sum(ctx + j for j in range(k)) * dkv + k * dkv
        total += tw + (ctx + k) * tkv
        ctx += emitted
    return total


# ------------------------------------------------------------------- e2e ---
def run_e2e(target, draft, prompt, caches, new_tokens=NEW_TOKENS, k=K, drafter=None):
    from spec.draft import ModelDraft
    from spec.loop import generate

    tc, dc = caches
    drafter = drafter if drafter is not None else ModelDraft(draft, dc)
    out, stats = generate(target, tc, drafter, [prompt], new_tokens, k=k, generator=torch.Generator().manual_seed(0))
    return out[0], stats


def bench_e2e(steps, warmup):
    target, draft, t_state, d_state = build_models()
    prompt = prompt_ids()
    caches = caches_for(target, draft)
    log("e2e warmup")
    for _ in range(warmup):
        run_e2e(target, draft, prompt, caches)
    torch.cuda.synchronize()
    t0 = time.perf_counter()
    outs = []
    for _ in range(steps):
        out, stats = run_e2e(target, draft, prompt, caches)
        outs.append(out)
    torch.cuda.synchronize()
    dt = time.perf_counter() - t0
    emitted = sum(len(o) for o in outs)
    nbytes = request_bytes(target, draft, PROMPT, stats, K)
    gbs = nbytes * steps / dt / 1e9
    result = {"tokens_per_s": emitted / dt, "ms_per_step": 1000 * dt / steps, "emitted_per_step": len(outs[0]),
              "rounds": stats.rounds, "mean_accept_len": mean_accept_len(stats),
              "acceptance": stats.accepted / max(stats.drafted, 1),
              "roofline": {"bound": "hbm", "bytes_per_request": nbytes, "achieved": gbs, "peak": HBM_PEAK_GBS,
                           "unit": "GB/s", "frac": gbs / HBM_PEAK_GBS,
                           "bytes": "target + draft weights as stored (bf16 head read as bf16) per forward, K/V read "
                                    "and written per position, over the request's own rounds"}}
    # identity check of this output against plain greedy decoding of the target
    from baselines.cached_autoregressive import generate as plain

    plain_cache = caches_for(target, None)[0]
    plain(target, plain_cache, prompt, NEW_TOKENS)  # warm
    torch.cuda.synchronize()
    t1 = time.perf_counter()
    want = plain(target, plain_cache, prompt, NEW_TOKENS)
    torch.cuda.synchronize()
    result["plain_greedy_tokens_per_s"] = NEW_TOKENS / (time.perf_counter() - t1)
    result["identical_to_plain_greedy"] = want == outs[0]
    result["first_divergence"] = next((i for i, (a, b) in enumerate(zip(want, outs[0])) if a != b), None)
    return result, (target, draft, t_state, d_state, prompt, outs[0])


def bench_e2e_torch_projections(target, draft, prompt, want, steps=2):
    """The same request with every dense projection on torch's GEMMs
    (hipBLASLt; torch matrix-vector products for the draft's single rows)
    instead of specdec_linear: fresh caches, so the graphs are captured
    anew with torch's projections."""
    import lm.forward as fwd

    saved = fwd.LINEAR_KERNEL
    fwd.LINEAR_KERNEL = False
    try:
        caches = caches_for(target, draft)
        run_e2e(target, draft, prompt, caches)  # warm-up, graph capture
        torch.cuda.synchronize()
        t0 = time.perf_counter()
        for _ in range(steps):
            out, stats = run_e2e(target, draft, prompt, caches)
        torch.cuda.synchronize()
        dt = time.perf_counter() - t0
        # the greedy identity holds in this configuration too (its bf16
        # projections round differently, so its tokens may differ from the
        # headline path's on these random weights)
        from baselines.cached_autoregressive import generate as plain

        plain_out = plain(target, caches_for(target, None)[0], prompt, NEW_TOKENS)
    finally:
        fwd.LINEAR_KERNEL = saved
    del caches
    torch.cuda.empty_cache()
    return {"tokens_per_s": len(out) * steps / dt, "ms_per_step": 1000 * dt / steps, "rounds": stats.rounds,
            "identical_to_plain_greedy": out == plain_out, "same_tokens_as_headline_path": out == want}


def bench_truncated_drafts(target, t_state, prompt, depths=(4, 12, 18, 22), noise=0.002):
    """Config 4's second variant: the draft is the target's first n layers
    (embeddings, final norm and head shared) plus N(0, noise^2) on every matrix
    of those layers, swept over the truncation depth."""
    from lm.model import SMOLLM2_1_7B, Llama, perturbed_truncation

    out = {}
    for n in depths:
        state, shape = perturbed_truncation(t_state, SMOLLM2_1_7B, n, noise, seed=7)
        draft = Llama.from_state_dict(shape, state)
        caches = caches_for(target, draft)
        run_e2e(target, draft, prompt, caches)  # warm (graph captures)
        torch.cuda.synchronize()
        t0 = time.perf_counter()
        tokens, stats = run_e2e(target, draft, prompt, caches)
        torch.cuda.synchronize()
        dt = time.perf_counter() - t0
        gbs = request_bytes(target, draft, PROMPT, stats, K) / dt / 1e9
        out[f"layers_{n}"] = {"draft": f"target layers 0..{n - 1} + N(0, {noise}^2)", "tokens_per_s": len(tokens) / dt,
                              "acceptance": stats.accepted / max(stats.drafted, 1),
                              "mean_accept_len": mean_accept_len(stats), "rounds": stats.rounds,
                              "roofline_frac": gbs / HBM_PEAK_GBS}
        log(f"truncated draft {n}: {out[f'layers_{n}']}")
        del draft, caches
        torch.cuda.empty_cache()
    return out


def bench_copy_draft(target, prompt, want):
    """The target as its own draft.  Computing as the verify does
    (ModelDraft(exact=True)), every drafted token is the target's own greedy
    choice: every round accepts all k and emits the bonus token -- the
    accept, bonus and rollback paths at full shapes.  Computing for latency
    (the default draft arithmetic), near-ties of the bf16 forward break the
    other way now and then, and acceptance shows how often."""
    from spec.draft import ModelDraft

    out = {}
    for name, exact in (("exact", True), ("latency", False)):
        caches = caches_for(target, target)
        run_e2e(target, None, prompt, caches, drafter=ModelDraft(target, caches[1], exact=exact))
        torch.cuda.synchronize()
        t0 = time.perf_counter()
        tokens, stats = run_e2e(target, None, prompt, caches, drafter=ModelDraft(target, caches[1], exact=exact))
        torch.cuda.synchronize()
        dt = time.perf_counter() - t0
        gbs = request_bytes(target, target, PROMPT, stats, K) / dt / 1e9
        out[name] = {"tokens_per_s": len(tokens) / dt, "acceptance": stats.accepted / max(stats.drafted, 1),
                     "mean_accept_len": mean_accept_len(stats), "rounds": stats.rounds,
                     "emitted_per_round": sorted(set(stats.emitted_per_round)),
                     "identical_to_plain_greedy": tokens == want, "roofline_frac": gbs / HBM_PEAK_GBS}
        del caches
        torch.cuda.empty_cache()
    return out


# ------------------------------------------------------------ attention -----
def attention_bytes(batch, lengths, t_new=5, h=32, hkv=32, d=64, bs=BLOCK):
    kv = sum((L + t_new) * hkv * d * 2 * 2 for L in lengths)
    qo = batch * t_new * h * d * 2 * 2
    tables = sum(-(-(L + t_new) // bs) * 4 for L in lengths)
    return kv + qo + tables


def setup_attention(batch, length, seed=0, h=32, hkv=32, d=64, t_new=5, num_blocks=4096, layers=1):
    """Config 2: pool of 4096 blocks handed out in a seeded random order,
    `length` cached positions per row, then an append of t_new tokens.
    `layers` pools share the block table, as the layers of a model do."""
    from cache.kv import KVCache

    need = batch * (-(-(length + t_new) // BLOCK))
    num_blocks = max(num_blocks, need + 8)
    cache = KVCache(layers, hkv, d, num_blocks, BLOCK, torch.bfloat16, "cuda", max_seqs=batch + 2)
    perm = torch.randperm(num_blocks, generator=torch.Generator().manual_seed(seed))
    cache.add(-1)
    cache.append([-1], [num_blocks * BLOCK])
    cache.table_tensor[cache.tables[-1].row, :num_blocks] = perm.to(torch.int32).cuda()
    cache.free(-1)
    cache.flush()
    ids = list(range(batch))
    for s in ids:
        cache.add(s)
    g = torch.Generator(device="cuda").manual_seed(seed)
    cache.append(ids, [length] * batch)
    cache.k.normal_(generator=g)
    cache.v.normal_(generator=g)
    step = cache.append(ids, [t_new] * batch)
    q = torch.randn(batch, t_new, h * d, generator=g, device="cuda").to(torch.bfloat16)
    out = torch.empty_like(q)
    return cache, step, q, out


def graph_time_us(launch, per_graph=20, replays=10):
    """Mean GPU time of `launch` (one kernel) from HIP events around replays of
    a graph holding `per_graph` back-to-back launches, so host launch cost
    is not in the measurement."""
    for _ in range(3):
        launch()
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        launch()
    torch.cuda.current_stream().wait_stream(side)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        for _ in range(per_graph):
            launch()
    graph.replay()
    stream = torch.cuda.current_stream()
    start, end = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
    stream.synchronize()
    start.record(stream)
    for _ in range(replays):
        graph.replay()
    end.record(stream)
    end.synchronize()
    return start.elapsed_time(end) * 1000 / (per_graph * replays)


MALL_BYTES = 256 << 20  # MI355X last-level (Infinity) cache


def attention_layers(batch, length, t_new=5, hkv=32, d=64):
    """Layer pools to cycle through so that the K/V read by consecutive
    launches exceed the last-level cache at least threefold: every launch
    then reads HBM, as the layers of a 24-layer model do."""
    touched = batch * (length + t_new) * hkv * d * 2 * 2
    return min(24, max(2, -(-3 * MALL_BYTES // touched)))


def time_attention(batch, length, iters=200, t_new=5, rotate=True):
    """Verify attention over the config-2 setup.  With `rotate`, launches
    cycle over attention_layers() layer pools (K/V from HBM); without, they
    re-read one pool, which at batch 1 (34 MB) stays in the last-level cache."""
    from specdec import ops

    layers = attention_layers(batch, length, t_new) if rotate else 1
    cache, step, q, out = setup_attention(batch, length, t_new=t_new, layers=layers)
    h, hkv, d = 32, 32, 64
    ws = ops.AttentionWorkspace(q.device)
    turn = [0]

    def launch():
        i = turn[0] % layers
        turn[0] += 1
        ops.paged_attention(q, q.stride(1), cache.k[i], cache.v[i], cache.table_tensor, step.meta, batch, t_new, h,
                            hkv, d, BLOCK, 0.125, step.max_total, out, out.stride(1), ws)

    launch()
    per_graph = layers * -(-20 // layers)
    us = graph_time_us(launch, per_graph=per_graph, replays=max(iters // per_graph, 2))
    nbytes = attention_bytes(batch, [length] * batch, t_new=t_new)
    del cache
    torch.cuda.empty_cache()
    return {"batch": batch, "context": length, "us": us, "bytes": nbytes, "gbs": nbytes / us / 1e3,
            "frac_of_peak": nbytes / us / 1e3 / HBM_PEAK_GBS, "layer_pools": layers,
            "kv_source": "HBM (layer pools cycled)" if rotate else "one pool re-read"}


# ------------------------------------------------------- other kernels ------
def time_fn(fn, iters=100, graph=False):
    if graph:
        return graph_time_us(fn, per_graph=10, replays=max(iters // 10, 1))
    for _ in range(5):
        fn()
    stream = torch.cuda.current_stream()
    start, end = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
    stream.synchronize()
    start.record(stream)
    for _ in range(iters):
        fn()
    end.record(stream)
    end.synchronize()
    return start.elapsed_time(end) * 1000 / iters


def bench_head():
    """The output head (49152 x 2048 target, 49152 x 576 draft, bf16) at 1 and
    5 hidden rows: torch's mm with fp32 output, that plus the softmax kernel,
    the head kernel alone, with the row softmax, with the softmax from its own
    statistics (head_softmax: what the forward runs) and as one launch whose
    workgroups meet (head_fused: a library entry).  Launches cycle over copies
    of the head so W is read from HBM."""
    from specdec import ops

    res = {}
    for name, hidden, copies in (("target", 2048, 4), ("draft", 576, 12)):
        g = torch.Generator(device="cuda").manual_seed(3)
        heads = [(torch.randn(V, hidden, generator=g, device="cuda") * 0.02).to(torch.bfloat16) for _ in range(copies)]
        for rows in (1, 5):
            x = torch.randn(rows, hidden, generator=g, device="cuda").to(torch.bfloat16)
            out = torch.empty(rows, V, device="cuda")
            lg = torch.empty(rows, V, device="cuda")
            turn = [0]

            def w():
                turn[0] += 1
                return heads[turn[0] % copies]

            r = {"torch_mm_us": time_fn(lambda: torch.mm(x, w().t(), out_dtype=torch.float32, out=lg), graph=True),
                 "torch_mm_softmax_us": time_fn(
                     lambda: ops.probabilities(torch.mm(x, w().t(), out_dtype=torch.float32, out=lg), 1.0, out=out),
                     graph=True),
                 "head_logits_us": time_fn(lambda: ops.head_logits(x, w(), out=lg), graph=True),
                 "head_logits_softmax_us": time_fn(
                     lambda: ops.probabilities(ops.head_logits(x, w(), out=lg), 1.0, out=out), graph=True),
                 "head_softmax_us": time_fn(lambda: ops.head_softmax(x, w(), 1.0, out=out), graph=True),
                 "head_fused_us": time_fn(lambda: ops.head_probabilities(x, w(), 1.0, out=out), graph=True)}
            nbytes = V * hidden * 2 + rows * hidden * 2 + rows * V * 4
            r["bytes"] = nbytes
            r["head_logits_gbs"] = nbytes / r["head_logits_us"] / 1e3
            r["head_logits_frac_of_peak"] = r["head_logits_gbs"] / HBM_PEAK_GBS
            for kind in ("softmax", "fused"):
                r[f"head_{kind}_gbs"] = nbytes / r[f"head_{kind}_us"] / 1e3
                r[f"head_{kind}_frac_of_peak"] = r[f"head_{kind}_gbs"] / HBM_PEAK_GBS
            res[f"head_{name}_rows{rows}"] = r
            log(f"head {name} rows {rows}: logits {r['head_logits_us']:.2f} us, with the softmax "
                f"{r['head_softmax_us']:.2f} us, one launch {r['head_fused_us']:.2f} us")
        del heads
        torch.cuda.empty_cache()
    return res


def bench_linear():
    """specdec_linear at the decode-sized projections of the e2e models
    (draft SmolLM2-135M: one row; target SmolLM2-1.7B verify: five rows),
    weights cycled over copies so they come from HBM, in the tiled layout the
    forward reads (and row-major beside it), against torch (mv for one row,
    linear otherwise)."""
    from specdec import ops

    res = {}
    shapes = [("draft_qkv", 1, 576, 960), ("draft_o", 1, 576, 576), ("draft_gate_up", 1, 576, 3072),
              ("draft_down", 1, 1536, 576), ("target_qkv", 5, 2048, 6144), ("target_o", 5, 2048, 2048),
              ("target_gate_up", 5, 2048, 16384), ("target_down", 5, 8192, 2048)]
    g = torch.Generator(device="cuda").manual_seed(5)
    for name, rows, k, n in shapes:
        copies = min(24, max(2, -(-3 * MALL_BYTES // (k * n * 2))))
        ws = [(torch.randn(n, k, generator=g, device="cuda") * 0.05).to(torch.bfloat16) for _ in range(copies)]
        wts = [ops.tile_weight(w) for w in ws]
        x = torch.randn(rows, k, generator=g, device="cuda").to(torch.bfloat16)
        out = torch.empty(rows, n, dtype=torch.bfloat16, device="cuda")
        turn = [0]

        def pick(lst):
            turn[0] += 1
            return lst[turn[0] % copies]

        us = time_fn(lambda: ops.linear(x, pick(wts), out=out), graph=True)
        us_rows = time_fn(lambda: ops.linear(x, pick(ws), out=out), graph=True)
        if rows == 1:
            us_torch = time_fn(lambda: torch.mv(pick(ws), x.view(-1)), graph=True)
        else:
            us_torch = time_fn(lambda: torch.nn.functional.linear(x, pick(ws)), graph=True)
        nbytes = n * k * 2 + rows * (k + n) * 2
        res[f"linear_{name}"] = {"rows": rows, "in": k, "out": n, "us": us, "row_major_us": us_rows,
                                 "torch_us": us_torch, "bytes": nbytes, "gbs": nbytes / us / 1e3,
                                 "frac_of_peak": nbytes / us / 1e3 / HBM_PEAK_GBS}
        log(f"linear {name}: {us:.2f} us tiled, {us_rows:.2f} us row-major (torch {us_torch:.2f})")
        del ws, wts
        torch.cuda.empty_cache()
    return res


def bench_prefill_attention():
    """Prompt-sized attention (B=1, 32/32 heads x 64, bf16, block 16, an empty
    cache): RoPE + append + causal attention of T = 256 and 1024 new tokens
    through the paged cache, against torch's scaled_dot_product_attention
    on contiguous q/k/v of the same shape (no RoPE, no paging) for scale.
    Flops are the causal triangle's QK^T and PV: 2 * 2 * H * d * T(T+1)/2."""
    from cache.kv import KVCache
    from lm.model import SMOLLM2_1_7B, rope_tables
    from specdec import ops

    cos, sin = (t.cuda() for t in rope_tables(SMOLLM2_1_7B, 4096))
    res = {}
    for width in (256, 1024):
        cache = KVCache(1, 32, 64, 4096, BLOCK, torch.bfloat16, "cuda", max_seqs=2)
        cache.add(0)
        step = cache.append([0], [width])
        g = torch.Generator(device="cuda").manual_seed(width)
        qkv = torch.randn(1, width, 96 * 64, generator=g, device="cuda").to(torch.bfloat16)
        out = torch.empty(1, width, 32 * 64, device="cuda", dtype=torch.bfloat16)
        ws = ops.AttentionWorkspace(qkv.device)
        us = time_fn(lambda: ops.rope_paged_attention(qkv, cos, sin, cache.k[0], cache.v[0], cache.table_tensor,
                                                      step.meta, 1, width, 32, 32, 64, BLOCK, 0.125, step.max_total,
                                                      out, out.stride(1), ws), graph=True)
        q, k, v = (torch.randn(1, 32, width, 64, generator=g, device="cuda").to(torch.bfloat16) for _ in range(3))
        us_sdpa = time_fn(lambda: torch.nn.functional.scaled_dot_product_attention(q, k, v, is_causal=True),
                          graph=True)
        flops = 2 * 32 * 64 * width * (width + 1)
        res[f"prefill_attention_T{width}"] = {"us": us, "tflops": flops / us / 1e6,
                                              "frac_of_mfma_peak": flops / us / 1e6 / 2500.0,
                                              "torch_sdpa_contiguous_us": us_sdpa}
        del cache
    torch.cuda.empty_cache()
    return res


def bench_kernels(attention_grid=True):
    from specdec import ops
    from workloads import planted_rows

    res = {}
    # config 1: accept-reject, B=1, k=4, V=49152, fp32, T=1
    for b, k in [(1, 4), (8, 4), (32, 8)]:
        g = torch.Generator(device="cuda").manual_seed(1)
        tl = torch.randn(b, k + 1, V, generator=g, device="cuda") * 2
        dl = tl[:, :k] + torch.randn(b, k, V, generator=g, device="cuda") * 0.5
        p = ops.probabilities(tl, 1.0)
        q = ops.probabilities(dl, 1.0)
        draft = torch.randint(0, V, (b, k), device="cuda")
        q.view(-1, V)[torch.arange(b * k, device="cuda"), draft.view(-1)] += 1e-3
        ua = torch.rand(b, k, generator=g, device="cuda")
        ur = torch.rand(b, generator=g, device="cuda")
        both = torch.cat([tl.view(-1, V), dl.view(-1, V)])
        us_soft = time_fn(lambda: ops.probabilities(both, 1.0), graph=True)
        us_acc = time_fn(lambda: ops.accept_reject(p, q, draft, ua, ur), graph=True)
        # one launch from the logits: softmax, accept test, residual, sample
        assert ops.accept_reject_logits(tl, dl, 1.0, draft, ua, ur) is not None
        us_fused = time_fn(lambda: ops.accept_reject_logits(tl, dl, 1.0, draft, ua, ur), graph=True)
        # a round's algorithmic bytes: the 2k+1 logit rows read once
        logit_bytes = (2 * k + 1) * V * 4 * b
        # the same with the logits cycled over copies that together exceed
        # the last-level cache three times, so every launch reads them from
        # HBM (the timing above reuses one set, as a loop whose output head
        # has just written them would find them in the cache)
        copies = min(512, -(-3 * MALL_BYTES // logit_bytes))
        sets = [(tl.clone(), dl.clone()) for _ in range(copies)]
        turn = [0]

        def fused_cycled(temperature):
            t_, d_ = sets[turn[0] % copies]
            turn[0] += 1
            ops.accept_reject_logits(t_, d_, temperature, draft, ua, ur)

        us_fused_hbm, us_fused_hbm_t08 = (
            graph_time_us(lambda: fused_cycled(t), per_graph=copies, replays=max(1, 2000 // copies))
            for t in (1.0, 0.8))
        del sets
        log(f"accept b{b} k{k}: softmax {us_soft:.2f} us + accept {us_acc:.2f} us; fused {us_fused:.2f} us "
            f"({us_fused_hbm:.2f} us with the logits from HBM, {us_fused_hbm_t08:.2f} at T = 0.8)")
        res[f"accept_b{b}_k{k}"] = {
            "round_bytes": logit_bytes,
            "fused_us": us_fused, "fused_gbs": logit_bytes / us_fused / 1e3,
            "fused_frac_of_peak": logit_bytes / us_fused / 1e3 / HBM_PEAK_GBS,
            "fused_hbm_us": us_fused_hbm, "fused_hbm_t08_us": us_fused_hbm_t08,
            "fused_hbm_frac_of_peak": logit_bytes / us_fused_hbm / 1e3 / HBM_PEAK_GBS,
            "softmax_us": us_soft, "accept_us": us_acc, "two_launch_us": us_soft + us_acc,
            "two_launch_frac_of_peak": logit_bytes / (us_soft + us_acc) / 1e3 / HBM_PEAK_GBS,
            # what the two kernels move themselves: the softmax reads the
            # logits and writes p and q; the accept kernel reads the residual
            # position's p and q rows (2 V fp32 per batch entry)
            "softmax_traffic_gbs": 2 * logit_bytes / us_soft / 1e3,
            "accept_traffic_gbs": 2 * V * 4 * b / us_acc / 1e3,
            "what": "fused: specdec_accept_reject_logits (one launch from logits; fused_hbm: the logits "
                    "cycled over copies so each launch reads them from HBM); two-launch: "
                    "specdec_probabilities of the 2k+1 rows, then specdec_accept_reject; "
                    "fractions over the logits read once"}
    # config 3: n-gram, B=16
    for length in (2048, 4096, 8192):
        rows = planted_rows(16, length, V, seed=length)
        hist = torch.tensor(rows, dtype=torch.int32, device="cuda")
        lens = torch.full((16,), length, dtype=torch.int32, device="cuda")
        us = time_fn(lambda: ops.ngram_lookup(hist, lens, 4, 3), graph=True)
        nbytes = 16 * length * 4
        log(f"ngram b16 L{length}: {us:.2f} us")
        res[f"ngram_b16_L{length}"] = {"us": us, "bytes": nbytes, "gbs": nbytes / us / 1e3,
                                       "frac_of_peak": nbytes / us / 1e3 / HBM_PEAK_GBS}
    # config 2': cache append (rope + scatter of 5 tokens) and rollback plan
    cache, step, q, out = setup_attention(1, 4096)
    qkv = torch.randn(1, 5, 96 * 64, device="cuda").to(torch.bfloat16)
    from lm.model import SMOLLM2_1_7B, rope_tables

    cos, sin = (t.cuda() for t in rope_tables(SMOLLM2_1_7B, 8192))
    us_app = time_fn(lambda: ops.rope_append(qkv, 32, 32, 64, cos, sin, step.meta, 1, 5, cache.table_tensor, BLOCK,
                                             cache.k[0], cache.v[0]), graph=True)
    app_bytes = 5 * 96 * 64 * 2 + 5 * 64 * 64 * 2
    res["append_b1_t5"] = {"us": us_app, "bytes": app_bytes, "gbs": app_bytes / us_app / 1e3,
                           "frac_of_peak": app_bytes / us_app / 1e3 / HBM_PEAK_GBS}
    del cache
    res["rollback_grow_b8"] = bench_rollback()
    log("append and rollback done")
    res.update(bench_head())
    log("head done")
    res.update(bench_linear())
    res.update(bench_prefill_attention())
    log("prefill attention done")
    if not attention_grid:
        return res
    # attention over the config-2 grid
    for b in (1, 4, 8):
        for L in (512, 1024, 2048, 4096):
            res[f"attention_b{b}_L{L}"] = time_attention(b, L, iters=50)
    return res


def bench_rollback(batch=8, length=1010, iters=100):
    """Config 2': one round's cache bookkeeping at batch 8 as the device sees
    it -- every row rolls back its rejected tail block (a push) and regrows
    one block for the next verify (a pop) -- i.e. one block-plan launch.
    Timed as graph replays of that launch (its pushes and pops balance, so a
    replay leaves the free stack's depth where it was); plus the host-side
    round trip of truncate + append that the round loop issues."""
    from specdec import ops

    cache, _, _, _ = setup_attention(batch, length - 5)
    ids = list(range(batch))
    lens = [cache.length(s) for s in ids]
    alloc = cache.allocator
    rows = [cache.tables[s].row for s in ids]
    cols = [len(cache.tables[s]) - 1 for s in ids]
    entries = []
    for i, (r, c) in enumerate(zip(rows, cols)):
        entries += [r, c, 1, i]
    for i, (r, c) in enumerate(zip(rows, cols)):
        entries += [r, c, 1, i]
    ent = torch.tensor(entries, dtype=torch.int32, device="cuda")
    top = alloc._dev_top
    us = time_fn(lambda: ops.block_plan(cache.table_tensor, alloc._stack, alloc._used, top, ent, batch, batch),
                 iters=iters, graph=True)
    # entries read + per block: table read, stack write, mark write (push);
    # stack read, table write, mark write (pop)
    nbytes = ent.numel() * 4 + batch * (4 + 4 + 1) * 2

    def host_round():
        for s, n in zip(ids, lens):
            cache.truncate(s, n - 5 + 1)
        cache.append(ids, [4] * batch)

    res = {"us": us, "bytes": nbytes, "gbs": nbytes / us / 1e3, "frac_of_peak": nbytes / us / 1e3 / HBM_PEAK_GBS,
           "host_round_trip_us": time_fn(host_round, iters=50),
           "what": "block-plan launch: 8 rows push their tail block and pop one (rollback + regrowth)"}
    del cache
    return res


# ---------------------------------------------------------- config 5 -------
class LoopTimer:
    """In-loop kernel timing without a synchronisation in the timed region:
    HIP events recorded around each accept-reject launch and each verify
    graph replay on the launching stream, read after the run; and, every
    `every` rounds, the verify attention replayed over that round's cache
    state (the round's row metadata and block tables, every layer's pools,
    read-only: the cache is not changed) as one batch of back-to-back launches
    between two events."""

    def __init__(self, every: int = 32):
        self.every = every
        self.accept, self.verify, self.attention, self.draft = [], [], [], []
        # wall time spent outside the loop's own work: one-time graph
        # captures of new shapes, and the sampled attention replays
        self.excluded = 0.0
        self._round = 0

    def __enter__(self):
        import lm.graphs as graphs
        from specdec import ops

        import spec.draft as sd
        import spec.ngram as sn

        self._ops, self._graphs, self._drafters = ops, graphs, (sd.ModelDraft, sn.NGramDraft)
        self._real_accept = ops.accept_reject
        self._real_run = graphs.VerifyGraph.run
        self._real_capture = graphs._capture
        self._real_propose = {cls: cls.propose for cls in self._drafters}
        timer = self

        def timed_propose(real):
            def propose(drafter, *a, **kw):
                st, en = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
                st.record()
                out = real(drafter, *a, **kw)
                en.record()
                timer.draft.append((st, en))
                return out
            return propose

        for cls in self._drafters:
            cls.propose = timed_propose(self._real_propose[cls])

        def accept(*a, **kw):
            st, en = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
            st.record()
            out = timer._real_accept(*a, **kw)
            en.record()
            timer.accept.append((st, en))
            return out

        def verify_run(runner, ids, meta):
            st, en = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
            st.record()
            out = timer._real_run(runner, ids, meta)
            en.record()
            timer.verify.append((st, en))
            timer._round += 1
            if timer._round % timer.every == 0:
                timer._attention_replay(runner, meta)
            return out

        def capture(run):
            torch.cuda.synchronize()
            t0 = time.perf_counter()
            out = timer._real_capture(run)
            torch.cuda.synchronize()
            timer.excluded += time.perf_counter() - t0
            return out

        ops.accept_reject = accept
        graphs.VerifyGraph.run = verify_run
        graphs._capture = capture
        return self

    def _attention_replay(self, runner, meta):
        torch.cuda.synchronize()
        t0 = time.perf_counter()
        self._replay_layers(runner, meta)
        torch.cuda.synchronize()
        self.excluded += time.perf_counter() - t0

    def _replay_layers(self, runner, meta):
        ops, cache, llama = self._ops, runner.cache, runner.llama
        cfg = llama.config
        b, width = meta.shape[1], runner.ids.shape[1]
        h, hkv, d = cfg.num_attention_heads, cfg.num_key_value_heads, cfg.head_dim
        q = torch.zeros(b, width, h * d, dtype=llama.dtype, device=cache.device)
        out = torch.empty_like(q)
        layers = len(llama.layers)
        ops.paged_attention(q, q.stride(1), cache.k[0], cache.v[0], cache.table_tensor, meta, b, width, h, hkv, d,
                            cache.block_size, llama.scaling, runner.bucket, out, out.stride(1), runner.ws)  # warm
        st, en = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
        st.record()
        for i in range(layers):
            ops.paged_attention(q, q.stride(1), cache.k[i], cache.v[i], cache.table_tensor, meta, b, width, h, hkv,
                                d, cache.block_size, llama.scaling, runner.bucket, out, out.stride(1), runner.ws)
        en.record()
        past = meta[1].tolist()
        self.attention.append((st, en, layers, attention_bytes(b, past, t_new=width, h=h, hkv=hkv, d=d)))

    def __exit__(self, *exc):
        for cls, real in self._real_propose.items():
            cls.propose = real
        self._ops.accept_reject = self._real_accept
        self._graphs.VerifyGraph.run = self._real_run
        self._graphs._capture = self._real_capture
        return False

    def summary(self):
        torch.cuda.synchronize()
        acc = [s.elapsed_time(e) * 1000 for s, e in self.accept]
        ver = [s.elapsed_time(e) * 1000 for s, e in self.verify]
        att = [(s.elapsed_time(e) * 1000 / n, nbytes) for s, e, n, nbytes in self.attention]
        dra = [s.elapsed_time(e) * 1000 for s, e in self.draft]
        out = {"accept_kernel_us_per_round": {"mean": statistics.fmean(acc), "p50": pct(acc, 50), "p99": pct(acc, 99)},
               "verify_us_per_round": {"mean": statistics.fmean(ver), "p50": pct(ver, 50), "p99": pct(ver, 99)},
               # the drafter's k steps (model: two graph replays; n-gram: the
               # lookup launch, its history upload and the one-hot q), GPU
               # time between events around propose()
               "draft_us_per_round": {"mean": statistics.fmean(dra), "p50": pct(dra, 50), "p99": pct(dra, 99)}}
        if att:
            us = statistics.fmean(a for a, _ in att)
            nbytes = statistics.fmean(b for _, b in att)
            out["verify_attention_us_per_layer"] = us
            out["verify_attention_gbs"] = nbytes / us / 1e3
            out["verify_attention_frac_of_peak"] = nbytes / us / 1e3 / HBM_PEAK_GBS
            out["verify_attention_sampled_rounds"] = len(att)
        return out


def bench_batched(target, draft, combos=((8, 4, "model"), (8, 4, "ngram"), (32, 8, "model"), (32, 8, "ngram")),
                  prompt_len=1024, context=4096, temperature=0.8):
    """Config 5: batched sampled speculative decoding on seeded 1024-token
    prompts with ~30% planted repetition, each row decoded to a 4096-token
    context.  Reports emitted tokens/s -- without the one-time HIP graph
    captures of new shapes (new context buckets, the smaller batches left as
    rows finish) and the sampled attention replays, and with them -- mean
    accept length, and in-loop kernel times (LoopTimer)."""
    from spec.draft import ModelDraft
    from spec.loop import generate
    from spec.ngram import NGramDraft
    from workloads import planted_rows

    results = {}
    new_tokens = context - prompt_len
    for batch, k, kind in combos:
        prompts = planted_rows(batch, prompt_len, V, seed=batch * 100 + k)
        tc, dc = caches_for(target, draft if kind == "model" else None, batch, context, k)

        def drafter():
            return ModelDraft(draft, dc) if kind == "model" else NGramDraft(V)

        # warm-up: the first context bucket's graphs at this batch
        generate(target, tc, drafter(), prompts, 16, k=k, temperature=temperature,
                 generator=torch.Generator().manual_seed(1))
        with LoopTimer() as timer:
            torch.cuda.synchronize()
            t0 = time.perf_counter()
            outs, stats = generate(target, tc, drafter(), prompts, new_tokens, k=k, temperature=temperature,
                                   generator=torch.Generator().manual_seed(5))
            torch.cuda.synchronize()
            dt = time.perf_counter() - t0
        emitted = sum(len(o) for o in outs)
        key = f"b{batch}_k{k}_{kind}"
        results[key] = {"tokens_per_s": emitted / (dt - timer.excluded), "tokens_per_s_wall": emitted / dt,
                        "excluded_s": timer.excluded, "seconds": dt, "emitted": emitted,
                        "context": prompt_len + min(len(o) for o in outs),
                        "mean_accept_len": mean_accept_len(stats), "acceptance": stats.accepted / max(stats.drafted, 1),
                        "rounds": stats.rounds, **timer.summary(),
                        "sample": f"{batch} rows, {prompt_len}-token prompts (~30% planted repetition) decoded to "
                                  f"{context} tokens, T={temperature}, k={k}"}
        log(f"batched {key}: {results[key]}")
        del tc, dc
        torch.cuda.empty_cache()
    return results


# ------------------------------------------------- HBM traffic counters ----
def traffic_workload(launches=6):
    """What the counter runs profile (`--only traffic`): a copy of COPY_BYTES
    (three launches), then `launches` launches of the B=8, context-4096 verify
    attention cycling its layer pools, so each reads K/V from HBM."""
    from specdec import ops

    x = torch.ones(COPY_BYTES // 4, dtype=torch.float32, device="cuda")
    y = torch.empty_like(x)
    for _ in range(3):
        y.copy_(x)
    torch.cuda.synchronize()
    del x, y
    layers = attention_layers(8, 4096)
    cache, step, q, out = setup_attention(8, 4096, layers=layers)
    ws = ops.AttentionWorkspace(q.device)
    for i in range(launches):
        ops.paged_attention(q, q.stride(1), cache.k[i % layers], cache.v[i % layers], cache.table_tensor, step.meta,
                            8, 5, 32, 32, 64, BLOCK, 0.125, step.max_total, out, out.stride(1), ws)
    torch.cuda.synchronize()
    return {"copy_bytes_each_way": COPY_BYTES, "attention_launches": launches, "layer_pools": layers}


def _counter_means(csv_path, counter):
    """Mean per-dispatch value (KiB) of `counter` for the copy kernel and for
    the tiled verify attention kernel in a rocprofv3 counter CSV."""
    import csv

    vals = {"copy": [], "attention": []}
    copies = []  # (grid, value) of every copy dispatch: the largest grid is the known copy
    with open(csv_path, newline="") as f:
        for r in csv.DictReader(f):
            if r["Counter_Name"] != counter:
                continue
            name = r["Kernel_Name"]
            if "copyBuffer" in name:
                copies.append((int(r["Grid_Size"]), float(r["Counter_Value"])))
            elif "attention_bf16_kernel<1, 16, true" in name:
                vals["attention"].append(float(r["Counter_Value"]))
    if copies:
        top = max(g for g, _ in copies)
        vals["copy"] = [v for g, v in copies if g == top]
    if not vals["copy"] or not vals["attention"]:
        raise RuntimeError(f"{counter}: no {'copy' if not vals['copy'] else 'attention'} dispatch in {csv_path}")
    return statistics.mean(vals["copy"]), statistics.mean(vals["attention"]), len(vals["attention"])


def measure_attention_traffic(timeout_s=300):
    """HBM bytes per launch of the B=8, context-4096 verify attention, read by
    rocprofv3 in two child runs of `bench.py --only traffic`: FETCH_SIZE, then
    WRITE_SIZE (one pass cannot collect both).  Each counter is scaled by what
    it reads for the copy of COPY_BYTES in the same child run.  Runs before
    this process touches the GPU.  Returns (bytes or None, description)."""
    import shutil
    import signal
    import tempfile

    prof = shutil.which("rocprofv3") or "/opt/rocm/bin/rocprofv3"
    if not os.path.exists(prof):
        return None, "rocprofv3 not found"
    env = dict(os.environ)
    env.setdefault("TMPDIR", "/tmp")
    parts = {}
    with tempfile.TemporaryDirectory(prefix="specdec_traffic_", dir=env["TMPDIR"]) as tmp:
        for counter, tag in (("FETCH_SIZE", "f"), ("WRITE_SIZE", "w")):
            out_dir = os.path.join(tmp, tag)
            cmd = [prof, "--pmc", counter, "--output-format", "csv", "-d", out_dir, "-o", tag, "--",
                   sys.executable, "-u", str(ROOT / "bench.py"), "--only", "traffic"]
            t0 = time.perf_counter()
            proc = subprocess.Popen(cmd, cwd=tmp, env=env, stdout=subprocess.PIPE, stderr=subprocess.STDOUT,
                                    text=True, start_new_session=True)
            try:
                text, _ = proc.communicate(timeout=timeout_s)
            except subprocess.TimeoutExpired:
                os.killpg(proc.pid, signal.SIGKILL)
                proc.communicate()
                return None, f"{counter} counter run exceeded {timeout_s} s"
            csv_path = os.path.join(out_dir, f"{tag}_counter_collection.csv")
            # the profiler can exit non-zero after a complete run; the CSV decides
            if not os.path.exists(csv_path):
                tail = " | ".join(text.strip().splitlines()[-3:])
                return None, f"{counter} counter run (exit {proc.returncode}) wrote no CSV: {tail}"
            try:
                copy_kib, attn_kib, n = _counter_means(csv_path, counter)
            except (RuntimeError, KeyError, ValueError) as e:
                return None, str(e)
            scale = COPY_BYTES / (copy_kib * 1024)
            parts[counter] = {"attention_kib_per_dispatch": attn_kib, "dispatches": n,
                              "copy_kib_per_dispatch": copy_kib, "scale": scale,
                              "bytes": attn_kib * 1024 * scale, "seconds": time.perf_counter() - t0}
            log(f"traffic {counter}: {parts[counter]}")
    total = parts["FETCH_SIZE"]["bytes"] + parts["WRITE_SIZE"]["bytes"]
    desc = ("measured in this run: rocprofv3 --pmc FETCH_SIZE, then WRITE_SIZE, child runs of "
            "`bench.py --only traffic` ({} and {} attention dispatches), each scaled by what the counter reads "
            "for a 256 MiB copy in the same child run (x{:.3f} / x{:.3f})").format(
        parts["FETCH_SIZE"]["dispatches"], parts["WRITE_SIZE"]["dispatches"], parts["FETCH_SIZE"]["scale"],
        parts["WRITE_SIZE"]["scale"])
    return int(round(total)), desc


# ------------------------------------------------------------ CPU side ------
def cpu_model():
    try:
        out = subprocess.run(["lscpu"], capture_output=True, text=True, timeout=10).stdout
        for line in out.splitlines():
            if line.startswith("Model name:"):
                return line.split(":", 1)[1].strip()
    except (OSError, subprocess.SubprocessError):
        pass
    return "unknown"


def oracle_models(t_state, d_state):
    import oracle.forward as of
    from lm.model import SMOLLM2_135M, SMOLLM2_1_7B

    def cfg(s):
        return of.Config(s.vocab_size, s.hidden_size, s.num_hidden_layers, s.num_attention_heads,
                         s.num_key_value_heads, s.intermediate_size, s.head_dim, s.rms_norm_eps, s.rope_theta, True)

    return (of.Model(cfg(SMOLLM2_1_7B), {k: v.cpu() for k, v in t_state.items()}),
            of.Model(cfg(SMOLLM2_135M), {k: v.cpu() for k, v in d_state.items()}))


class _Turns:
    """Strict alternation of two loops' rounds (one thread each): a loop
    hands the turn over at the end of every round (its accept-reject call)
    and waits for it back.  Each side's round time runs from getting the turn
    to its next hand-over, so the other side's rounds are never counted."""

    def __init__(self, sides=("gpu", "cpu")):
        self.cv = threading.Condition()
        self.turn = sides[0]
        self.other = {sides[0]: sides[1], sides[1]: sides[0]}
        self.done = set()
        self.resumed = {s: None for s in sides}
        self.rounds = {s: [] for s in sides}

    def start(self, side):
        with self.cv:
            self.cv.wait_for(lambda: self.turn == side or self.other[side] in self.done, timeout=600)
            self.resumed[side] = time.perf_counter()

    def hand_over(self, side):
        now = time.perf_counter()
        with self.cv:
            self.rounds[side].append(now - self.resumed[side])
            if self.other[side] not in self.done:
                self.turn = self.other[side]
                self.cv.notify_all()
                self.cv.wait_for(lambda: self.turn == side or self.other[side] in self.done, timeout=600)
            self.resumed[side] = time.perf_counter()

    def finish(self, side):
        with self.cv:
            self.done.add(side)
            self.turn = self.other[side]
            self.cv.notify_all()


def cpu_e2e_interleaved(target, draft, t_state, d_state, prompt, warmup_rounds=3, rounds=20):
    """The oracle loop (bf16, host cores) and the GPU loop on the same request,
    their rounds alternating one for one.  The CPU request is a bounded sample
    (prompt + warmup_rounds + rounds + 1 tokens: one token per round at this
    draft's acceptance); the GPU request is the headline's.  Per side: p50 and
    p99 of the measured rounds and emitted tokens/s over them."""
    import oracle.kv as okv
    import oracle.loop as ol
    import spec.loop as loop
    from oracle.draft import ModelDraft as OModelDraft
    from spec.draft import ModelDraft

    threads = len(os.sched_getaffinity(0))
    torch.set_num_threads(threads)
    tm, dm = oracle_models(t_state, d_state)
    cpu_tokens = warmup_rounds + rounds + 1
    blocks = (PROMPT + NEW_TOKENS + 2 * K + 2 * BLOCK) // BLOCK + 4
    turns = _Turns()
    emitted = {"gpu": [], "cpu": []}
    real = {"gpu": loop.accept_reject, "cpu": ol.accept_reject}

    def hooked(side):
        def accept(p, q, draft_ids, generator=None, **kw):
            v = real[side](p, q, draft_ids, generator=generator, **kw)
            emitted[side].append(int(v.n_accepted.sum()) + len(v.n_accepted))
            turns.hand_over(side)
            return v
        return accept

    results, errors = {}, []

    def cpu_side():
        try:
            turns.start("cpu")
            t0 = time.perf_counter()
            out, stats = ol.generate(tm, okv.KVCache.for_model(tm.config, blocks, BLOCK, torch.bfloat16),
                                     OModelDraft(dm, okv.KVCache.for_model(dm.config, blocks, BLOCK, torch.bfloat16)),
                                     [prompt], cpu_tokens, K, generator=torch.Generator().manual_seed(0))
            results["cpu"] = (out[0], stats, time.perf_counter() - t0)
        except BaseException as e:  # surfaced in the main thread
            errors.append(e)
        finally:
            turns.finish("cpu")

    loop.accept_reject, ol.accept_reject = hooked("gpu"), hooked("cpu")
    worker = threading.Thread(target=cpu_side, daemon=True)
    try:
        tc, dc = caches_for(target, draft)
        turns.start("gpu")
        worker.start()
        out, stats = loop.generate(target, tc, ModelDraft(draft, dc), [prompt], NEW_TOKENS, k=K,
                                   generator=torch.Generator().manual_seed(0))
        turns.finish("gpu")
        worker.join(timeout=900)
    finally:
        loop.accept_reject, ol.accept_reject = real["gpu"], real["cpu"]
    if errors:
        raise errors[0]
    cpu_out, cpu_stats, cpu_seconds = results["cpu"]
    summary = {}
    for side in ("gpu", "cpu"):
        measured = turns.rounds[side][warmup_rounds:warmup_rounds + rounds]
        toks = emitted[side][warmup_rounds:warmup_rounds + rounds]
        summary[side] = {"rounds": len(measured), "round_ms_p50": 1000 * pct(measured, 50),
                         "round_ms_p99": 1000 * pct(measured, 99), "tokens_per_s": sum(toks) / sum(measured)}
    first_div = next((i for i, (a, b) in enumerate(zip(cpu_out, out[0])) if a != b), None)
    return summary, {"cpu_request_seconds": cpu_seconds, "cpu_tokens": len(cpu_out), "threads": threads,
                     "bf16_first_divergence_from_gpu": first_div}


def cpu_attention_baseline(length=4096, batch=1, seconds=3.0):
    """Oracle attention step (gather copy + masked SDPA) at context 4096 on the CPU."""
    import oracle.forward as of

    threads = len(os.sched_getaffinity(0))
    torch.set_num_threads(threads)
    g = torch.Generator().manual_seed(0)
    pool = torch.randn(4096 * BLOCK, 32, 64, generator=g).to(torch.bfloat16)
    nblk = -(-(length + 5) // BLOCK)
    perm = torch.randperm(4096, generator=g)[: batch * nblk].view(batch, nblk)
    read = (perm[:, :, None] * BLOCK + torch.arange(BLOCK)).flatten(1)[:, : length + 5]
    q = torch.randn(batch, 32, 5, 64, generator=g).to(torch.bfloat16)
    past, total = torch.full((batch,), length), torch.full((batch,), length + 5)
    n = 0
    t0 = time.perf_counter()
    while time.perf_counter() - t0 < seconds:
        k_all = pool[read].transpose(1, 2)
        v_all = pool[read].transpose(1, 2)
        of.attention(q, k_all, v_all, past, total, 0.125)
        n += 1
    us = (time.perf_counter() - t0) / n * 1e6
    return {"us": us, "gbs": attention_bytes(batch, [length] * batch) / us / 1e3, "cores": threads}


def cpu_kernel_baselines(seconds=1.0):
    """The oracle (the reference's algorithms in torch on the host cores) on
    the kernels' own workloads, each repeated for about `seconds`:
    temperature softmax and accept-reject (config 1 and batch 8), n-gram
    lookup (config 3), and the cache's append + rollback bookkeeping
    (config 2': slot maps and block tables for 8 rows, one layer's write of
    5 tokens)."""
    import oracle.accept as oa
    import oracle.kv as okv
    import oracle.ngram as on
    import oracle.sampling as osamp
    from workloads import planted_rows

    threads = len(os.sched_getaffinity(0))
    torch.set_num_threads(threads)

    def timed(fn):
        fn()
        n, t0 = 0, time.perf_counter()
        while n == 0 or time.perf_counter() - t0 < seconds:
            fn()
            n += 1
        return (time.perf_counter() - t0) / n * 1e6

    res = {"cores": threads}
    for b, k in ((1, 4), (8, 4)):
        g = torch.Generator().manual_seed(1)
        tl = torch.randn(b, k + 1, V, generator=g) * 2
        dl = tl[:, :k] + torch.randn(b, k, V, generator=g) * 0.5
        p, q = osamp.probabilities(tl, 1.0), osamp.probabilities(dl, 1.0)
        draft = torch.randint(0, V, (b, k), generator=g)
        ua, ur = torch.rand(b, k, generator=g), torch.rand(b, generator=g)
        both = torch.cat([tl.reshape(-1, V), dl.reshape(-1, V)])
        res[f"softmax_b{b}_k{k}_us"] = timed(lambda: osamp.probabilities(both, 1.0))
        res[f"accept_b{b}_k{k}_us"] = timed(lambda: oa.accept_reject(p, q, draft, u_accept=ua, u_residual=ur))
    for length in (2048, 4096, 8192):
        rows = planted_rows(16, length, V, seed=length)
        res[f"ngram_b16_L{length}_us"] = timed(lambda: [on.lookup_match(r, 4, 3) for r in rows])
    cache = okv.KVCache(1, 32, 64, 8 * 70, BLOCK, torch.bfloat16)
    ids = list(range(8))
    for s in ids:
        cache.add(s)
    cache.append(ids, [1010] * 8)

    def rollback_and_grow():
        for s in ids:
            cache.truncate(s, 1010 - 5 + 1)
        cache.append(ids, [4] * 8)

    res["rollback_grow_b8_us"] = timed(rollback_and_grow)
    one = okv.KVCache(1, 32, 64, 300, BLOCK, torch.bfloat16)
    one.add(0)
    one.append([0], [4096])
    kv_new = torch.randn(1, 32, 5, 64).to(torch.bfloat16)

    def append_write():
        one.truncate(0, 4096)
        slots = one.append([0], [5])
        one.write(0, slots, kv_new, kv_new)

    res["append_b1_t5_us"] = timed(append_write)
    return res


class _Stop(Exception):
    """Ends a loop once its measured rounds are in."""


def cpu_batched_interleaved(target, draft, tm, dm, batch, k, kind, warmup_rounds=2, rounds=5, prompt_len=1024,
                            temperature=0.8):
    """Config 5 on the host cores at the config's own shapes: the oracle loop
    (bf16, the reference's gather + SDPA forward and host accept-reject) and
    the GPU loop on the same `batch` planted 1024-token prompts, k, T = 0.8,
    the model or n-gram drafter, their rounds alternating one for one
    (_Turns).  Each side stops after `warmup_rounds` + `rounds` rounds.  The
    CPU side skips the prompt's prefill (32 x 1024 prompt tokens through the
    1.7B shapes would take minutes on the host): its caches hold the prompt
    length of zero K/V and its first token comes from seeded random logits,
    so its rounds run the config's shapes -- contexts, batch, k, both
    models' full depth -- on other values.  Per side: p50 / p99 round time
    and emitted tokens/s over the measured rounds."""
    import oracle.draft as od
    import oracle.kv as okv
    import oracle.loop as ol
    import spec.loop as loop
    from spec.draft import ModelDraft
    from spec.ngram import NGramDraft
    from workloads import planted_rows

    threads = len(os.sched_getaffinity(0))
    torch.set_num_threads(threads)
    prompts = planted_rows(batch, prompt_len, V, seed=batch * 100 + k)
    limit = warmup_rounds + rounds
    new_tokens = 4 * limit + 8  # rows outlast the measured rounds (at least one token per round)
    blocks = batch * ((prompt_len + new_tokens + 2 * k + 2 * BLOCK) // BLOCK + 2)
    turns = _Turns()
    emitted = {"gpu": [], "cpu": []}
    real = {"gpu": loop.accept_reject, "cpu": ol.accept_reject}
    real_run = ol.run

    def hooked(side):
        def accept(p, q, draft_ids, generator=None, **kw):
            v = real[side](p, q, draft_ids, generator=generator, **kw)
            emitted[side].append(int(v.n_accepted.sum()) + len(v.n_accepted))
            turns.hand_over(side)
            if len(turns.rounds[side]) >= limit:
                raise _Stop()
            return v
        return accept

    def synthetic_prefill(model, cache, seq_ids, chunks):
        cache.append(seq_ids, [len(c) for c in chunks])  # the pools start zeroed
        return torch.randn(len(seq_ids), V, generator=torch.Generator().manual_seed(batch + k))

    class SyntheticDraft(od.ModelDraft):
        def prefill(self, seq_ids, prompts):
            for s in seq_ids:
                self.cache.add(s)
            self.cache.append(seq_ids, [len(p) for p in prompts])

    errors = []

    def cpu_side():
        try:
            turns.start("cpu")
            tc = okv.KVCache.for_model(tm.config, blocks, BLOCK, torch.bfloat16)
            dr = (SyntheticDraft(dm, okv.KVCache.for_model(dm.config, blocks, BLOCK, torch.bfloat16))
                  if kind == "model" else od.NGramDraft(V))
            ol.generate(tm, tc, dr, prompts, new_tokens, k, temperature=temperature,
                        generator=torch.Generator().manual_seed(5))
        except _Stop:
            pass
        except BaseException as e:  # surfaced in the main thread
            errors.append(e)
        finally:
            turns.finish("cpu")

    loop.accept_reject, ol.accept_reject, ol.run = hooked("gpu"), hooked("cpu"), synthetic_prefill
    worker = threading.Thread(target=cpu_side, daemon=True)
    try:
        tc, dc = caches_for(target, draft if kind == "model" else None, batch, prompt_len + new_tokens + 64, k)
        drafter = ModelDraft(draft, dc) if kind == "model" else NGramDraft(V)
        turns.start("gpu")
        worker.start()
        try:
            loop.generate(target, tc, drafter, prompts, new_tokens, k=k, temperature=temperature,
                          generator=torch.Generator().manual_seed(5))
        except _Stop:
            pass
        turns.finish("gpu")
        worker.join(timeout=900)
    finally:
        loop.accept_reject, ol.accept_reject, ol.run = real["gpu"], real["cpu"], real_run
    if errors:
        raise errors[0]
    del tc, dc
    torch.cuda.empty_cache()
    out = {}
    for side in ("gpu", "cpu"):
        measured = turns.rounds[side][warmup_rounds:limit]
        toks = emitted[side][warmup_rounds:limit]
        out[side] = {"rounds": len(measured), "round_ms_p50": 1000 * pct(measured, 50),
                     "round_ms_p99": 1000 * pct(measured, 99), "tokens_per_s": sum(toks) / sum(measured),
                     "tokens_per_round": sum(toks) / max(len(toks), 1)}
    out["speedup"] = out["gpu"]["tokens_per_s"] / out["cpu"]["tokens_per_s"]
    out["sample"] = (f"{batch} rows, {prompt_len}-token planted prompts, k={k}, T={temperature}, {kind} drafter, "
                     f"bf16; {warmup_rounds} warm-up + {rounds} measured rounds per side, interleaved one for one; "
                     f"CPU side with zero prompt K/V instead of a prefill")
    return out


def kernel_speedups(kernels, ck, attn8, attn1, cpu_attn1, cpu_attn8):
    """Host-oracle time over GPU time for each kernel timed on both sides."""
    pairs = {"attention_b1_L4096": (cpu_attn1["us"], attn1["us"]), "attention_b8_L4096": (cpu_attn8["us"], attn8["us"])}
    for b, k in ((1, 4), (8, 4)):
        g = kernels.get(f"accept_b{b}_k{k}")
        if g:
            pairs[f"softmax_b{b}_k{k}"] = (ck[f"softmax_b{b}_k{k}_us"], g["softmax_us"])
            pairs[f"accept_b{b}_k{k}"] = (ck[f"accept_b{b}_k{k}_us"], g["accept_us"])
    for length in (2048, 4096, 8192):
        g = kernels.get(f"ngram_b16_L{length}")
        if g:
            pairs[f"ngram_b16_L{length}"] = (ck[f"ngram_b16_L{length}_us"], g["us"])
    if "append_b1_t5" in kernels:
        pairs["append_b1_t5"] = (ck["append_b1_t5_us"], kernels["append_b1_t5"]["us"])
    if "rollback_grow_b8" in kernels:
        pairs["rollback_grow_b8_host_round_trip"] = (ck["rollback_grow_b8_us"],
                                                     kernels["rollback_grow_b8"]["host_round_trip_us"])
    return {name: c / g for name, (c, g) in pairs.items()}


def main():
    ap = argparse.ArgumentParser()
    ap.add_argument("--gpus", type=int, default=1)
    ap.add_argument("--steps", type=int, default=3)
    ap.add_argument("--warmup", type=int, default=1)
    ap.add_argument("--only", choices=["all", "e2e", "batched", "batched-cpu", "attention", "kernels", "small", "copy",
                                       "head", "rollback", "traffic"],
                    default="all",
                    help="small: the kernels of configs 1-3 without the attention grid (for counter runs)")
    ap.add_argument("--no-cpu", action="store_true")
    ap.add_argument("--no-batched", action="store_true")
    ap.add_argument("--no-traffic", action="store_true",
                    help="skip the rocprofv3 counter runs of the attention's HBM traffic (the stored figure is reported)")
    ap.add_argument("--batch", type=int, default=8, help="batch of the --only attention run")
    ap.add_argument("--one-pool", action="store_true", help="--only attention: re-read one layer pool")
    ap.add_argument("--context", type=int, default=4096, help="--only batched: context the rows decode to")
    args = ap.parse_args()
    if args.gpus != 1:
        print(f"bench.py runs on one GPU only; --gpus {args.gpus} is not supported (the path is built and "
              "measured on a single GPU; sharding across GPUs is not implemented)", file=sys.stderr)
        sys.exit(2)
    # the roofline's traffic: counter runs in child processes, before this
    # one touches the GPU
    traffic, traffic_source = ATTN_B8_TRAFFIC, "stored (--no-traffic): " + STORED_TRAFFIC_SOURCE
    if args.only == "all" and not args.no_traffic:
        measured, why = measure_attention_traffic()
        if measured is not None:
            traffic, traffic_source = measured, why
        else:
            traffic_source = f"stored (the counter runs failed: {why}): " + STORED_TRAFFIC_SOURCE
        log(f"attention traffic {traffic} B: {traffic_source}")
    # the host spins while it waits for each round's verdict (before anything
    # touches the GPU); SPECDEC_SPIN_WAIT=0 keeps HIP's default wait
    global HOST_WAIT
    if os.environ.get("SPECDEC_SPIN_WAIT", "1") != "0":
        from specdec import spin_wait

        HOST_WAIT = "spin" if spin_wait() else "default (spin refused)"
    if not torch.cuda.is_available():
        print("bench.py needs a GPU", file=sys.stderr)
        sys.exit(2)
    sys.path.insert(0, str(ROOT))

    if args.only == "attention":
        r = time_attention(args.batch, 4096, iters=max(args.steps, 1) * 100, rotate=not args.one_pool)
        print(json.dumps({f"attention_b{args.batch}_L4096": r}))
        return
    if args.only == "head":
        print(json.dumps(bench_head()))
        return
    if args.only in ("kernels", "small"):
        print(json.dumps(bench_kernels(attention_grid=args.only == "kernels")))
        return
    if args.only == "traffic":
        print(json.dumps(traffic_workload()))
        return
    if args.only == "copy":
        # reference copy of a known size for scaling the FETCH_SIZE / WRITE_SIZE counters
        x = torch.ones(64 << 20, dtype=torch.float32, device="cuda")
        y = torch.empty_like(x)
        for _ in range(max(args.steps, 1)):
            y.copy_(x)
        torch.cuda.synchronize()
        print(json.dumps({"copy_bytes_each_way": x.numel() * 4, "launches": max(args.steps, 1)}))
        return
    if args.only == "e2e":
        e2e, _ = bench_e2e(args.steps, args.warmup)
        print(json.dumps({"e2e": e2e}))
        return
    if args.only == "batched":
        target, draft, _, _ = build_models()
        print(json.dumps({"batched_sampled": bench_batched(target, draft, context=args.context)}))
        return
    if args.only == "batched-cpu":
        target, draft, t_state, d_state = build_models()
        tm, dm = oracle_models(t_state, d_state)
        out = {}
        for b, k, kind in ((8, 4, "model"), (32, 8, "model"), (8, 4, "ngram"), (32, 8, "ngram")):
            out[f"batched_b{b}_k{k}_{kind}"] = cpu_batched_interleaved(
                target, draft, tm, dm, b, k, kind, warmup_rounds=2 if b <= 8 else 1, rounds=6 if b <= 8 else 4)
            log(f"b{b} k{k} {kind}: {out[f'batched_b{b}_k{k}_{kind}']}")
        print(json.dumps(out))
        return
    if args.only == "rollback":
        print(json.dumps({"rollback_grow_b8": bench_rollback(iters=max(args.steps, 1) * 100)}))
        return

    e2e, (target, draft, t_state, d_state, prompt, gpu_tokens) = bench_e2e(args.steps, args.warmup)
    log(f"e2e {e2e}")
    e2e["torch_projections"] = bench_e2e_torch_projections(target, draft, prompt, gpu_tokens)
    log(f"torch projections {e2e['torch_projections']}")
    e2e["truncated_drafts"] = bench_truncated_drafts(target, t_state, prompt)
    e2e["copy_draft"] = bench_copy_draft(target, prompt, gpu_tokens)
    log(f"copy draft {e2e['copy_draft']}")
    attn = time_attention(8, 4096, iters=120)
    log(f"attention b8 {attn}")
    attn1 = time_attention(1, 4096, iters=300)
    log(f"attention b1 {attn1}")
    attn1_pool = time_attention(1, 4096, iters=300, rotate=False)
    log(f"attention b1 one pool {attn1_pool}")
    kernels = bench_kernels()
    batched = {} if args.no_batched else bench_batched(target, draft)
    cpu = None
    if not args.no_cpu:
        log("cpu baseline (rounds interleaved with the GPU loop)")
        rounds, extra = cpu_e2e_interleaved(target, draft, t_state, d_state, prompt)
        log(f"cpu rounds {rounds} {extra}")
        tm, dm = oracle_models(t_state, d_state)
        batched_cpu = {}
        for b, k, kind in ((8, 4, "model"), (8, 4, "ngram"), (32, 8, "model"), (32, 8, "ngram")):
            key = f"batched_b{b}_k{k}_{kind}"
            batched_cpu[key] = cpu_batched_interleaved(target, draft, tm, dm, b, k, kind,
                                                       warmup_rounds=2 if b <= 8 else 1, rounds=6 if b <= 8 else 4)
            log(f"cpu {key}: {batched_cpu[key]}")
        del target, draft
        torch.cuda.empty_cache()
        ck = cpu_kernel_baselines()
        log("cpu kernels done")
        cpu_attn1, cpu_attn8 = cpu_attention_baseline(), cpu_attention_baseline(batch=8)
        cpu = {"value": rounds["cpu"]["tokens_per_s"], "unit": "tokens/s", "cores": extra["threads"], "kind": "port",
               "cpu_model": cpu_model(),
               "sample": f"oracle loop (gather+SDPA forward, host accept-reject), bf16, 256-token prompt, "
                         f"{extra['cpu_tokens']} new tokens; rounds interleaved one for one with the GPU loop's, "
                         f"3 warm-up rounds excluded, 20 measured; torch threads={extra['threads']}",
               "rounds": rounds, **extra,
               "steady_state_speedup": rounds["gpu"]["tokens_per_s"] / rounds["cpu"]["tokens_per_s"],
               "attention_b1_L4096": cpu_attn1, "attention_b8_L4096": cpu_attn8, "kernels": ck, **batched_cpu}
        cpu["kernel_speedups"] = kernel_speedups(kernels, ck, attn, attn1, cpu_attn1, cpu_attn8)
        cpu["speedup"] = e2e["tokens_per_s"] / cpu["value"]
    line = {
        "metric": "spec-decode accepted tokens/s, 1.7B/135M k=4 b=1; verify-attn HBM GB/s",
        "value": e2e["tokens_per_s"],
        "unit": "tokens/s",
        "n_gpus": 1,
        "steps": args.steps,
        "warmup": args.warmup,
        "ms_per_step": e2e["ms_per_step"],
        "higher_is_better": True,
        "scaling": "weak",
        "vs_baseline": None,
        "dtype": "bf16",
        "data": "synthetic (random-init weights N(0, 0.02), seeded uniform prompt ids)",
        "config": {"workload": "greedy speculative decode, target SmolLM2-1.7B shapes / draft SmolLM2-135M shapes, "
                               "batch 1, k=4, paged KV block 16, prompt 256, 128 new tokens",
                   "batch": 1, "k": K, "prompt": PROMPT, "new_tokens": NEW_TOKENS, "block_size": BLOCK,
                   "host_wait": HOST_WAIT},
        "roofline": {"bound": "hbm", "achieved": attn["gbs"], "peak": HBM_PEAK_GBS, "unit": "GB/s",
                     "frac": attn["gbs"] / HBM_PEAK_GBS, "traffic": traffic,
                     "traffic_over_algorithmic": traffic / attn["bytes"], "traffic_source": traffic_source,
                     "kernel": "verify paged attention (attention_bf16_kernel<1, 16, true>: one 16-wave workgroup "
                               "per (row, kv head) tile taking its 512-token splits in rounds, no combine launch), "
                               "B=8, context 4096 (+5 appended), 32/32 heads x 64, bf16, block 16, K/V from HBM",
                     "us_per_launch": attn["us"], "bytes_per_launch": attn["bytes"]},
        "cpu_baseline": cpu,
        "e2e": e2e,
        "attention_b1_ctx4096": attn1,
        "attention_b1_ctx4096_one_pool": attn1_pool,
        "batched_sampled": batched,
        "kernels": kernels,
    }
    print(json.dumps(line))


if __name__ == "__main__":
    main()
