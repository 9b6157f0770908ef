"""GPU parity tests of the batched prefill (``prefill``, C ABI ``mk_prefill``) -- the replacement of
the reference's Transformers prefill plus cache copy (/root/reference/model.py:72-87).

Oracles:
  * ``restate.prefill``: the fp32 restatement run over all prompt tokens at once (pinned on the CPU
    against the token-by-token ``restate.decode_step``, tests/test_oracle.py) -- the tight check:
    last logits within 5e-3, the same greedy token, every cache value within one bf16 rounding step
    of the largest values and each layer's relative rms difference below one step;
  * Transformers' own bf16 prefill on the CPU (the reference path): its cache and last logits. The
    kernel is held to the floor of the fp32 restatement measured in the same run: per layer, its
    cache is no further from Transformers' than the restatement's, and its last logits no further.
"""
import time

import pytest
import torch

from oracle import hf, restate
from tests.gpu_common import DEV, Session, stats, write_record

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def mini():
    return Session("mini", 512)


@pytest.fixture(scope="module")
def mini17():
    return Session("mini-1.7b", 512)


@pytest.fixture(scope="module")
def mini_4k():
    return Session("mini", 4096)


@pytest.fixture(scope="module")
def mini17_2k():
    return Session("mini-1.7b", 2048)


def _prefill(sess, ids, kd, vd, position=0):
    tokens = torch.tensor(ids, dtype=torch.int32, device=DEV)
    return sess.kernel.prefill(tokens, sess.embed, sess.lm_head, sess.final_norm, sess.layers, sess.cos, sess.sin,
                               kd, vd, position, sess.max_seq)


def _check_cache(got, want, upto, tag):
    """Rows [0, upto) of the bf16 caches agree to one rounding step of the largest values, and per
    layer their relative rms difference is below one bf16 step (2^-8): where two fp32-accurate
    computations round a value to neighbouring bf16s, the flip propagates to later layers, so the
    share of values off by a step grows with depth (a few percent at 28 layers) while each stays a
    step."""
    g, w = got[:, :, :upto].float().cpu(), want[:, :, :upto].float()
    d = (g - w).abs()
    bound = 2 ** -6 * max(1.0, w.abs().max().item())
    rel = ((g - w).flatten(1).norm(dim=1) / w.flatten(1).norm(dim=1).clamp_min(1e-30))
    print(f"[{tag}] cache rows [0, {upto}): max |d| {d.max().item():.3e} (bound {bound:.3e}), relative rms per layer "
          f"max {rel.max().item():.2e} (bound {2 ** -8:.2e})", flush=True)
    assert d.max().item() <= bound
    assert rel.max().item() <= 2 ** -8


# Prompt lengths by the path that they take from position 0 (mini: the 0.6B width, mini17: 1.7B).
# Skinny products on column blocks of 8 tokens (their number in brackets), the attention straight from their
# sums in the passes of 32 keys that the line names.
SKINNY = [
    *(("mini", n) for n in (1, 9, 24, 32)),                    # [1, 2, 3, 4] 1 pass
    *(("mini17", n) for n in (7, 16, 32)),                     # [1, 2, 4]
    ("mini", 33), ("mini", 64), ("mini17", 33), ("mini17", 64),  # [5, 8] 2
    *(("mini", n) for n in (65, 80, 100, 128)),                # [9, 10, 13, 16] 4
    *(("mini17", n) for n in (41, 49)),                        # [6, 7] 2
    *(("mini17", n) for n in (65, 96, 128)),                   # [9, 12, 16] 4
    *(("mini", n) for n in (131, 160, 161, 192)),              # [17, 20, 21, 24] 6
    *(("mini", n) for n in (193, 225, 256)),                   # [25, 29, 32] 8
]
# 128-row tiles, QKV split over K with qkv_post_kernel, O and down split over K, the attention in key-range
# chunks; gate/up is never split from position 0 (a chunk of 97-128 tokens at 1.7B is: the 104 tokens at 196 of
# test_prefill_in_chunks_and_decode_after_it).
TILES_SPLIT = [("mini", 257), ("mini", 300), ("mini17", 129), ("mini17", 200)]
# 256-row tiles: gate/up (three 128-row tiles in two at 300; 8 row tiles at 1,000), QKV too at 1,100 and at the
# 1.7B 1,500. 656 tokens are the last on 128-row gate/up tiles, 657 the first on 256 rows.
TILES_TALL = [("mini17_2k", 300), ("mini_4k", 656), ("mini_4k", 657), ("mini_4k", 1000), ("mini_4k", 1100)]
# O and down unsplit, two wave groups halving K: 24 row tiles of 8 column tiles, 12 of 16
TILES_LONG = [("mini_4k", 3000), ("mini17_2k", 1500)]


@pytest.mark.parametrize("shape_fixture, P", SKINNY + TILES_SPLIT + TILES_TALL + TILES_LONG)
def test_prefill_matches_oracle(shape_fixture, P, request):
    """Prefill from an empty cache against ``restate.prefill`` on the same prompt: the last token's
    logits and greedy token, every K/V row written, and nothing written past the prompt."""
    sess = request.getfixturevalue(shape_fixture)
    ids = hf.prompt_ids(P, sess.shape.vocab, seed=3)[0].tolist()
    s = sess.shape
    kd = torch.zeros(s.layers, s.kv_heads, sess.max_seq, s.head_dim, dtype=torch.bfloat16, device=DEV)
    vd = torch.zeros_like(kd)
    logits, tok = _prefill(sess, ids, kd, vd)
    want, kw, vw = restate.prefill(sess.W, ids, sess.cos_cpu, sess.sin_cpu, sess.max_seq)
    maxabs, cos = stats(logits.cpu(), want)
    print(f"[prefill {shape_fixture} P={P}] max|kernel - oracle| {maxabs:.3e}, cos {cos:.8f}", flush=True)
    assert maxabs < 5e-3 and cos > 0.999999
    assert int(tok.item()) == restate.argmax_bf16(want)
    assert int(tok.item()) == restate.argmax_bf16(logits.cpu())
    _check_cache(kd, kw, P, f"prefill {shape_fixture} P={P} k")
    _check_cache(vd, vw, P, f"prefill {shape_fixture} P={P} v")
    assert kd[:, :, P:].abs().sum().item() == 0 and vd[:, :, P:].abs().sum().item() == 0
    assert sess.kernel.status() == 0


@pytest.mark.parametrize("shape_fixture, cuts", [("mini", (0, 40, 75, 100)), ("mini_4k", (0, 900, 964, 1000)),
                                                 ("mini17", (0, 100, 196, 300)), ("mini", (0, 3, 250, 510)),
                                                 ("mini_4k", (0, 1801, 2101))],
                         ids=["chunks-40-75", "chunks-900-964", "chunks-100-196-1.7b", "chunks-3-250", "chunks-1801"])
def test_prefill_in_chunks_and_decode_after_it(shape_fixture, cuts, request):
    """A prompt fed in chunks gives the cache and last logits of the one-shot oracle prefill; a decode step
    after it (the decode kernel, reading the prefilled cache) matches the oracle's decode step on the
    oracle's cache. Chunks past position 0 on the skinny products with the general attention: 35 and 25
    tokens (no key-range chunks), 64 at 900 and 36 at 964 (16 key blocks in chunks of two on 64
    workgroups, merged by attn_merge_kernel), 247 at 3, and 96 at 100 at 1.7B. On tiles: 260 at 250, 300 at
    1,801 (key-range chunks of 6 blocks), and 104 at 196 at 1.7B, the case whose gate/up product is split
    over K (silu_post_kernel). The 900 tokens from position 0 take chunks of 5 key blocks (of 4 a few
    short ones would run as a second round)."""
    mini = request.getfixturevalue(shape_fixture)
    P = cuts[-1]
    ids = hf.prompt_ids(P, mini.shape.vocab, seed=4)[0].tolist()
    s = mini.shape
    kd = torch.zeros(s.layers, s.kv_heads, mini.max_seq, s.head_dim, dtype=torch.bfloat16, device=DEV)
    vd = torch.zeros_like(kd)
    for a, b in zip(cuts[:-1], cuts[1:]):
        logits, tok = _prefill(mini, ids[a:b], kd, vd, a)
    want, kw, vw = restate.prefill(mini.W, ids, mini.cos_cpu, mini.sin_cpu, mini.max_seq)
    maxabs, _ = stats(logits.cpu(), want)
    assert maxabs < 5e-3 and int(tok.item()) == restate.argmax_bf16(want)
    _check_cache(kd, kw, P, "chunked k")
    _check_cache(vd, vw, P, "chunked v")
    nxt = int(tok.item())
    got, dev_tok = mini.decode(nxt, kd, vd, P, greedy=True)
    want2 = mini.oracle_step(kw, vw, nxt, P)
    maxabs, _ = stats(got.cpu(), want2)
    print(f"[prefill chunks] decode after prefill: max|d| {maxabs:.3e}", flush=True)
    assert maxabs < 5e-3 and int(dev_tok.item()) == restate.argmax_bf16(want2)


def _layer_dist(a, b, upto):
    """Per layer: mean |a - b| over rows [0, upto) (float64)."""
    d = (a[:, :, :upto].double() - b[:, :, :upto].double()).abs()
    return d.mean(dim=(1, 2, 3))


@pytest.mark.parametrize("shape_name, P, max_seq", [("qwen3-0.6b", 64, 512), ("qwen3-0.6b", 32, 512),
                                                    ("qwen3-0.6b", 3584, 4096), ("qwen3-1.7b", 512, 2048)])
def test_prefill_baseline_prompts_against_transformers(shape_name, P, max_seq):
    """The BASELINE prompts (configs 1, 2, 4 and 5) through the kernel's prefill, the fp32
    restatement's and Transformers' own (the reference path, bf16, CPU).
      * tight: kernel vs restatement -- last logits within 5e-3, the same greedy token, cache values
        within one bf16 rounding step of the largest values, per-layer relative rms below one step;
      * floor: per layer, the kernel's K and V rows are no further from Transformers' cache (mean
        absolute difference) than the restatement's are, within 1%; the kernel's last logits are no
        further from Transformers' (max-abs within 1e-3; cosine within the first-order bound its
        distance r from the restatement allows, r * sqrt(1 - cos^2) + r^2) and pick the same token
        whenever the restatement does.
    Prints the kernel's prefill time (HIP events, second of two runs)."""
    sess = Session(shape_name, max_seq)
    s = sess.shape
    ids_t = hf.prompt_ids(P, s.vocab)
    ids = ids_t[0].tolist()
    kd = torch.zeros(s.layers, s.kv_heads, max_seq, s.head_dim, dtype=torch.bfloat16, device=DEV)
    vd = torch.zeros_like(kd)
    _prefill(sess, ids, kd, vd)  # first run: warm-up
    kd.zero_()
    vd.zero_()
    ev0, ev1 = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
    torch.cuda.synchronize()
    ev0.record()
    logits, tok = _prefill(sess, ids, kd, vd)
    ev1.record()
    torch.cuda.synchronize()
    ms = ev0.elapsed_time(ev1)
    print(f"[prefill {shape_name} P={P}] kernel prefill {ms:.2f} ms ({P / ms * 1e3:.0f} tokens/s)", flush=True)
    got = logits.cpu()
    t0 = time.perf_counter()
    want, kw, vw = restate.prefill(sess.W, ids, sess.cos_cpu, sess.sin_cpu, max_seq)
    t1 = time.perf_counter()
    hf_last, cache = hf.prefill(sess.model, ids_t)
    t2 = time.perf_counter()
    print(f"[prefill {shape_name} P={P}] CPU: restatement {t1 - t0:.1f} s, Transformers {t2 - t1:.1f} s", flush=True)
    kh, vh = hf.cache_to_kernel_layout(cache, s.layers, s.kv_heads, max_seq, s.head_dim)
    del cache
    # tight
    maxabs, _ = stats(got, want)
    assert maxabs < 5e-3, maxabs
    assert int(tok.item()) == restate.argmax_bf16(want)
    _check_cache(kd, kw, P, f"{shape_name} P={P} k")
    _check_cache(vd, vw, P, f"{shape_name} P={P} v")
    # floor against Transformers
    kcpu, vcpu = kd.cpu(), vd.cpu()
    for name, g, w, h in (("k", kcpu, kw, kh), ("v", vcpu, vw, vh)):
        dk, do = _layer_dist(g, h, P), _layer_dist(w, h, P)
        print(f"[{shape_name} P={P} {name}] mean |cache - Transformers| per layer: kernel "
              f"{[round(x, 5) for x in dk[::7].tolist()]} oracle {[round(x, 5) for x in do[::7].tolist()]} "
              f"(layers 0, 7, 14, 21)", flush=True)
        assert bool((dk <= do * 1.01 + 1e-7).all()), (name, dk.tolist(), do.tolist())
    r = hf_last.float()
    km, kc = stats(got, r)
    om, oc = stats(want, r)
    print(f"[{shape_name} P={P}] last logits vs Transformers: kernel max|d| {km:.3e} cos {kc:.8f}, oracle max|d| "
          f"{om:.3e} cos {oc:.8f}; tokens kernel {int(tok.item())} oracle {restate.argmax_bf16(want)} "
          f"Transformers {int(r.argmax())}", flush=True)
    rel = ((got.double() - want.double()).norm() / want.double().norm()).item()
    write_record(f"prefill_{shape_name}_p{P}", {
        "workload": f"{shape_name}, prompt {P}, cache {max_seq}: native prefill", "prefill_ms": ms,
        "tight": {"max_abs": maxabs, "token_kernel": int(tok.item()), "token_oracle": restate.argmax_bf16(want)},
        "last_logits_vs_transformers": {"kernel": {"max_abs": km, "cos": kc}, "oracle": {"max_abs": om, "cos": oc}},
        "tokens": {"kernel": int(tok.item()), "oracle": restate.argmax_bf16(want), "transformers": int(r.argmax())},
        "rel_kernel_vs_oracle": rel,
        "mean_abs_cache_vs_transformers_per_layer": {
            "k": {"kernel": _layer_dist(kcpu, kh, P).tolist(), "oracle": _layer_dist(kw, kh, P).tolist()},
            "v": {"kernel": _layer_dist(vcpu, vh, P).tolist(), "oracle": _layer_dist(vw, vh, P).tolist()}},
    })
    assert km <= om + 1e-3
    assert kc >= oc - (rel * (1.0 - oc * oc) ** 0.5 + rel * rel)  # the per-step bound of the decode tests
    if restate.argmax_bf16(want) == int(r.argmax()):
        assert int(tok.item()) == int(r.argmax())
    assert sess.kernel.status() == 0


def test_prefill_out_of_range_token_is_reported_in_band(mini):
    """A prompt token outside [0, vocab) cannot be checked on the host without a copy: it is embedded
    as token 0 (no read leaves the table) and the call reports NaN logits and token -1."""
    s = mini.shape
    kd = torch.zeros(s.layers, s.kv_heads, mini.max_seq, s.head_dim, dtype=torch.bfloat16, device=DEV)
    vd = torch.zeros_like(kd)
    logits, tok = _prefill(mini, [5, s.vocab + 3, 7], kd, vd)
    assert torch.isnan(logits).all() and int(tok.item()) == -1
    logits, tok = _prefill(mini, [5, 0, 7], kd, vd)  # the next call is healthy again
    assert torch.isfinite(logits).all() and int(tok.item()) >= 0


def _pool(sess, ps, extra, seed):
    """A pool of NaN-filled pages for the session's cache length and a shuffled block table."""
    s = sess.shape
    npl = sess.max_seq // ps
    pool = npl + extra
    table = torch.randperm(pool, generator=torch.Generator().manual_seed(seed))[:npl].to(torch.int32)
    kp = torch.full((s.layers, pool, s.kv_heads, ps, s.head_dim), float("nan"), dtype=torch.bfloat16, device=DEV)
    return table, kp, kp.clone(), pool


@pytest.mark.parametrize("shape_fixture, chunks, ps", [
    ("mini", ((0, 40),), 16),                      # skinny products, pages written by short_attn_kernel<2>
    ("mini", ((0, 7),), 16),                       # ... <1>
    ("mini", ((0, 100),), 16),                     # ... <4>
    ("mini", ((0, 180),), 32),                     # ... <6>
    ("mini", ((0, 250),), 16),                     # ... <8>
    ("mini17", ((0, 100),), 16),                   # ... <4>, 1.7B width
    ("mini", ((0, 3), (3, 250)), 16),              # skinny products past position 0: pages from qkv_post_kernel
    ("mini17", ((0, 100), (100, 204)), 16),        # 1.7B tiles with gate/up split over K
    ("mini", ((0, 300),), 16),                     # 128-row tiles, residual products split over K
    ("mini17", ((0, 200),), 64),
    ("mini", ((0, 40), (40, 75), (75, 100)), 32),  # chunks reading earlier chunks through the table
    ("mini_4k", ((0, 900), (900, 964), (964, 1000)), 64),  # attention as key-range chunks, merged
])
def test_paged_prefill_matches_contiguous(shape_fixture, chunks, ps, request):
    """``prefill_paged`` (C ABI ``mk_prefill_paged``) into a pool of pages in shuffled order, the pool
    filled with NaN, against ``prefill`` into the contiguous cache: the same kernels through another
    address map, so every chunk's logits and token agree bit for bit, the rows gathered back through
    the table equal the contiguous cache's, and no other page is touched. A ``decode_paged`` step after
    it then equals ``decode`` on the contiguous cache (the contiguous prefill and decode are checked
    against the restatement by the tests above)."""
    from tests.paged_layout import from_pages
    sess = request.getfixturevalue(shape_fixture)
    s = sess.shape
    P = chunks[-1][1]
    ids = hf.prompt_ids(P, s.vocab, seed=7)[0].tolist()
    table, kp, vp, pool = _pool(sess, ps, 5, 11)
    table_d = table.to(DEV)
    kd = torch.zeros(s.layers, s.kv_heads, sess.max_seq, s.head_dim, dtype=torch.bfloat16, device=DEV)
    vd = torch.zeros_like(kd)
    for a, b in chunks:
        la, ta = _prefill(sess, ids[a:b], kd, vd, a)
        tokens = torch.tensor(ids[a:b], dtype=torch.int32, device=DEV)
        lb, tb = sess.kernel.prefill_paged(tokens, sess.embed, sess.lm_head, sess.final_norm, sess.layers, sess.cos,
                                           sess.sin, kp, vp, table_d, a, sess.max_seq)
        assert torch.equal(la, lb), f"chunk {a}..{b}: paged prefill logits differ"
        assert int(ta.item()) == int(tb.item())
    kg, vg = from_pages(kp, table.tolist()), from_pages(vp, table.tolist())
    assert torch.equal(kg[:, :, :P], kd[:, :, :P]) and torch.equal(vg[:, :, :P], vd[:, :, :P])
    # rows past the prompt and pages outside the table are untouched (still NaN)
    assert torch.isnan(kg[:, :, P:].float()).all() and torch.isnan(vg[:, :, P:].float()).all()
    unused = sorted(set(range(pool)) - set(table.tolist()))
    assert torch.isnan(kp[:, unused].float()).all() and torch.isnan(vp[:, unused].float()).all()
    tok = int(tb.item())
    l1, t1 = sess.decode(tok, kd, vd, P, greedy=True)
    l2, t2 = sess.kernel.decode_paged(tok, sess.embed, sess.lm_head, sess.final_norm, sess.layers, sess.cos, sess.sin,
                                      kp, vp, table_d, P, sess.max_seq)
    assert torch.equal(l1, l2) and int(t1.item()) == int(t2.item())
    print(f"[paged prefill {shape_fixture} chunks {chunks} page {ps}] identical to the contiguous prefill and "
          f"decode", flush=True)
    assert sess.kernel.status() == 0


@pytest.mark.parametrize("P, bad", [(40, 1), (250, 14), (300, 17)])
def test_paged_prefill_bad_table_entry_is_reported_in_band(mini, P, bad):
    """A block-table entry outside the pool, on a page the prompt writes, cannot be checked on the host
    without a copy: the call reports NaN logits and token -1 and writes nothing through that entry."""
    s = mini.shape
    ps = 16
    table, kp, vp, pool = _pool(mini, ps, 2, 3)
    table[bad] = pool + 5  # positions 16 bad .. 16 bad + 15
    tokens = torch.tensor(hf.prompt_ids(P, s.vocab, seed=2)[0].tolist(), dtype=torch.int32, device=DEV)
    before = kp.clone()  # (vp holds the same)
    logits, tok = mini.kernel.prefill_paged(tokens, mini.embed, mini.lm_head, mini.final_norm, mini.layers, mini.cos,
                                            mini.sin, kp, vp, table.to(DEV), 0, mini.max_seq)
    assert torch.isnan(logits).all() and int(tok.item()) == -1
    good = {int(table[i]) for i in range((P + ps - 1) // ps) if i != bad}  # the prompt's other pages
    for pages in (kp, vp):
        changed = (pages.float().nan_to_num(7.0) != before.float().nan_to_num(7.0)).any(-1).any(-1).any(-1).any(0)
        assert set(changed.nonzero().flatten().tolist()) <= good
    table[bad] = sorted(set(range(pool)) - set(table.tolist()))[0]  # an unused page: the next call is healthy
    logits, tok = mini.kernel.prefill_paged(tokens, mini.embed, mini.lm_head, mini.final_norm, mini.layers, mini.cos,
                                            mini.sin, kp, vp, table.to(DEV), 0, mini.max_seq)
    assert torch.isfinite(logits).all() and int(tok.item()) >= 0
