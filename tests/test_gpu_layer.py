"""GPU parity of the whole hot-expert layer (GEMV and grouped MFMA modes) against the
oracle's `_reference_check` FFN, through the C ABI."""
from dataclasses import replace

import numpy as np
import pytest

from conftest import bf16_bits_of, bf16_tensor, to_dev
from helpers import dequant_w, gemv_layer_oracle
from oracle import gguf_ref as R

pytestmark = pytest.mark.gpu

TOL_REL_L2 = 2e-2  # layer outputs vs the fp64 FFN on the bf16-dequantised weights


def _pkg():
    import kt_prefill_lend_amd._lib as L
    import kt_prefill_lend_amd.kt_gguf_hot as H
    import kt_prefill_lend_amd.synth as S

    return L, H, S


def _case(name, tokens, hidden=None, inter=None, hot=None, experts=None):
    _, _, S = _pkg()
    w = S.WORKLOADS[name]
    w = replace(w, hidden=hidden or w.hidden, inter=inter or w.inter, hot=hot or w.hot, experts=experts or w.experts)
    ids, tw, slot, _ = S.routing(w, tokens)
    xb = S.activations(w, tokens)
    w13, w2 = S.slot_tensors(w)
    return w, xb, tw, slot, w13, w2


def _run(dev, w, xb, tw, slot, w13, w2, mode):
    import torch

    L, H, _ = _pkg()
    W13, W2 = to_dev(w13, dev), to_dev(w2, dev)
    desc = H.layer_desc(W13, W2, w.hidden, w.inter, w.types[0], w.types[2])
    y = H.moe_layer(desc, bf16_tensor(xb, dev), to_dev(tw, dev), to_dev(slot, dev), mode)
    torch.cuda.synchronize()
    return bf16_bits_of(y)


CASES = [
    # (workload, tokens, hidden, inter, hot, experts)
    ("q8_0-h2048-n768-e128-k8-hot16", 40, 512, 256, 6, 24),
    ("q4_k-h2048-n512-e256-k8-hot32-decode", 16, 512, 256, 8, 32),
    ("q4_k+q6_k-h2048-n512-e256-k8-hot40-prefill", 48, 512, 256, 8, 32),
    ("iq3_s-h2048-n512-e512-k10-hot48", 40, 512, 256, 8, 40),
]


@pytest.mark.parametrize("case", CASES, ids=[c[0].split("-")[0] for c in CASES])
@pytest.mark.parametrize("mode", ["gemv", "decode", "grouped"])
def test_layer_vs_ffn_reference(dev, case, mode):
    L, _, S = _pkg()
    if mode == "decode":  # at most 256 routes
        case = (case[0], min(case[1], 256 // S.WORKLOADS[case[0]].top_k)) + tuple(case[2:])
    w, xb, tw, slot, w13, w2 = _case(*case)
    m = {"gemv": L.MODE_GEMV, "decode": L.MODE_DECODE, "grouped": L.MODE_GROUPED}[mode]
    got = R.bf16_to_f32(_run(dev, w, xb, tw, slot, w13, w2, m))
    g, d = dequant_w(w13, w2, w.types, w.hidden, w.inter)
    ref = R.ffn_reference(xb, slot, tw, g, d)
    l2, l1, cos = R.rel_errors(got, ref)
    print(f"{case[0]} {mode}: rel L2 {l2:.2e} rel L1 {l1:.2e} cos {cos:.6f}")
    assert l2 < TOL_REL_L2 and l1 < 0.025 and cos > 0.999, (l2, l1, cos)
    # tokens with no hot route are exactly zero
    cold_tok = (slot < 0).all(axis=1)
    assert np.all(got[cold_tok] == 0)


def test_gemv_mode_matches_reference_kernel_numerics(dev):
    """The decode path reproduces the reference kernels' own sequence (q8_1 GEMV, bf16,
    SiLU*mul, q8_1 GEMV, combine) to bf16 rounding."""
    L, _, _ = _pkg()
    w, xb, tw, slot, w13, w2 = _case("q4_k-h2048-n512-e256-k8-hot32-decode", 4, 512, 256, 8, 32)
    got = R.bf16_to_f32(_run(dev, w, xb, tw, slot, w13, w2, L.MODE_GEMV))
    exp = R.bf16_to_f32(gemv_layer_oracle(xb, tw, slot, w13, w2, w.types, w.hidden, w.inter))
    l2, _, _ = R.rel_errors(got, exp)
    assert l2 < 4e-3, l2


FUSED = [
    # (workload, tokens, top slot must exceed one 16-route pass): at most 256 routes, so GEMV
    # mode runs the two fused decode launches; 3 tokens stage every h row in LDS, the larger
    # windows (240 routes, 138 KB of h) read h from HBM and split the busiest slot's routes
    # over passes of the gate/up block
    ("q8_0-h2048-n768-e128-k8-hot16", 3, False),
    ("q8_0-h2048-n768-e128-k8-hot16", 30, True),
    ("q4_k+q6_k-h2048-n512-e256-k8-hot40-prefill", 3, False),
    ("q4_k+q6_k-h2048-n512-e256-k8-hot40-prefill", 30, True),
    ("iq3_s-h2048-n512-e512-k10-hot48", 3, False),
    ("iq3_s-h2048-n512-e512-k10-hot48", 24, True),
]


@pytest.mark.parametrize("case", FUSED, ids=[f"{c[0].split('-')[0]}-T{c[1]}" for c in FUSED])
def test_fused_decode_every_type(dev, case):
    """The fused decode launches for every weight type (gate/up and down), against the
    oracle's step-by-step restatement of the reference kernels' numerics."""
    L, _, _ = _pkg()
    name, T, multi_pass = case
    w, xb, tw, slot, w13, w2 = _case(name, T, 512, 256, 8, 32)
    assert slot.size <= 256
    per_slot = np.bincount(slot[slot >= 0], minlength=8)
    assert (per_slot.max() > 16) == multi_pass, per_slot
    got = R.bf16_to_f32(_run(dev, w, xb, tw, slot, w13, w2, L.MODE_GEMV))
    exp = R.bf16_to_f32(gemv_layer_oracle(xb, tw, slot, w13, w2, w.types, w.hidden, w.inter))
    l2, _, _ = R.rel_errors(got, exp)
    print(f"{name} T={T}: rel L2 vs the reference-kernel sequence {l2:.2e}")
    assert l2 < 4e-3, l2
    assert np.all(got[(slot < 0).all(axis=1)] == 0)


@pytest.mark.parametrize("T", [32, 33])
def test_decode_at_the_fused_route_limit(dev, T):
    """GEMV mode at 256 routes (32 tokens x 8: the most the fused decode launches take) and at
    264 (33 tokens: the stage-by-stage GEMV sequence), against the oracle's restatement of
    the reference kernels' sequence."""
    L, _, _ = _pkg()
    w, xb, tw, slot, w13, w2 = _case("q4_k-h2048-n512-e256-k8-hot32-decode", T, 512, 256, 8, 32)
    got = R.bf16_to_f32(_run(dev, w, xb, tw, slot, w13, w2, L.MODE_GEMV))
    exp = R.bf16_to_f32(gemv_layer_oracle(xb, tw, slot, w13, w2, w.types, w.hidden, w.inter))
    l2, _, _ = R.rel_errors(got, exp)
    assert l2 < 4e-3, l2
    assert np.all(got[(slot < 0).all(axis=1)] == 0)


@pytest.mark.parametrize("mode", ["gemv", "decode", "grouped"])
def test_layer_deterministic(dev, mode):
    L, _, _ = _pkg()
    T = 24 if mode == "decode" else 300  # the decode mode takes at most 256 routes
    w, xb, tw, slot, w13, w2 = _case("q4_k+q6_k-h2048-n512-e256-k8-hot40-prefill", T, 512, 256, 8, 32)
    m = {"gemv": L.MODE_GEMV, "decode": L.MODE_DECODE, "grouped": L.MODE_GROUPED}[mode]
    a = _run(dev, w, xb, tw, slot, w13, w2, m)
    b = _run(dev, w, xb, tw, slot, w13, w2, m)
    assert np.array_equal(a, b)


@pytest.mark.parametrize("t13,t2", [(R.GGML_Q4_K, R.GGML_Q6_K), (R.GGML_Q8_0, R.GGML_Q8_0), (R.GGML_IQ3_S, R.GGML_IQ3_S)])
def test_decode_mode_column_groups(dev, t13, t2):
    """The decode mode with slots of 64, 33, 17 and 1 routes (4, 3, 2 and 1 groups of 16 MFMA
    columns), 64 tokens x top-4 = 256 routes: against the fp64 FFN, and within the layer
    tolerance of the GEMV mode."""
    L, H, S = _pkg()
    base = S.WORKLOADS["q4_k+q6_k-h2048-n512-e256-k8-hot40-prefill"]
    w = replace(base, hidden=512, inter=256, hot=8, experts=32, top_k=4, types=(t13, t13, t2))
    T = 64
    rng = np.random.default_rng(21)
    slot = np.full((T, 4), -1, np.int32)
    slot[:, 0] = 0                      # slot 0: every token
    slot[:33, 1] = 1                    # slot 1: 33 tokens
    slot[5:22, 2] = 2                   # slot 2: 17 tokens
    slot[40, 2] = 3                     # slot 3: one token
    others = rng.integers(4, w.hot, size=(T, 1))
    slot[:, 3:] = np.where(rng.random((T, 1)) < 0.5, others, -1)
    tw = rng.random((T, 4)).astype(np.float32)
    tw /= tw.sum(axis=1, keepdims=True)
    xb = S.activations(w, T)
    w13, w2 = S.slot_tensors(w)
    got = R.bf16_to_f32(_run(dev, w, xb, tw, slot, w13, w2, L.MODE_DECODE))
    g, d = dequant_w(w13, w2, w.types, w.hidden, w.inter)
    ref = R.ffn_reference(xb, slot, tw, g, d)
    l2, l1, cos = R.rel_errors(got, ref)
    assert l2 < TOL_REL_L2 and cos > 0.999, (l2, l1, cos)
    gemv = R.bf16_to_f32(_run(dev, w, xb, tw, slot, w13, w2, L.MODE_GEMV))
    assert R.rel_errors(got, gemv)[0] < TOL_REL_L2


def test_decode_mode_repeated_slot(dev):
    """A slot listed two or three times by a token (168 routes of 64 tokens on slot 0, 11
    groups of 16 MFMA columns, past the 64 a slot can hold without repeats): every route is
    computed, against the fp64 FFN (which sums the repeats) and the GEMV mode."""
    L, H, S = _pkg()
    base = S.WORKLOADS["q4_k+q6_k-h2048-n512-e256-k8-hot40-prefill"]
    w = replace(base, hidden=512, inter=256, hot=8, experts=32, top_k=4)
    T = 64
    rng = np.random.default_rng(22)
    slot = np.full((T, 4), -1, np.int32)
    slot[:, 0] = 0
    slot[:, 1] = 0
    slot[:40, 2] = 0
    slot[40:, 2] = rng.integers(1, w.hot, size=T - 40)
    slot[:, 3] = np.where(rng.random(T) < 0.5, rng.integers(1, w.hot, size=T), -1)
    assert (slot == 0).sum() == 168
    tw = rng.random((T, 4)).astype(np.float32)
    tw /= tw.sum(axis=1, keepdims=True)
    xb = S.activations(w, T)
    w13, w2 = S.slot_tensors(w)
    got = R.bf16_to_f32(_run(dev, w, xb, tw, slot, w13, w2, L.MODE_DECODE))
    g, d = dequant_w(w13, w2, w.types, w.hidden, w.inter)
    ref = R.ffn_reference(xb, slot, tw, g, d)
    l2, l1, cos = R.rel_errors(got, ref)
    assert l2 < TOL_REL_L2 and cos > 0.999, (l2, l1, cos)
    gemv = R.bf16_to_f32(_run(dev, w, xb, tw, slot, w13, w2, L.MODE_GEMV))
    assert R.rel_errors(got, gemv)[0] < TOL_REL_L2


@pytest.mark.parametrize("seed", range(6))
def test_decode_mode_random_windows(dev, seed):
    """The decode mode on random windows: 1 to 64 tokens, top-1 to top-8 (at most 256 routes),
    slot ids mixing hot slots, -1 and ids past the table, some tokens naming a slot twice;
    against the fp64 FFN."""
    L, H, S = _pkg()
    rng = np.random.default_rng(100 + seed)
    top_k = int(rng.integers(1, 9))
    T = int(rng.integers(1, min(64, 256 // top_k) + 1))
    base = S.WORKLOADS["q4_k+q6_k-h2048-n512-e256-k8-hot40-prefill"]
    w = replace(base, hidden=512, inter=256, hot=8, experts=32, top_k=top_k)
    slot = rng.integers(-2, w.hot + 3, size=(T, top_k)).astype(np.int32)
    slot[slot == -2] = -1
    if T > 2:
        slot[1, :] = slot[1, 0]  # one token naming one slot top_k times
    tw = rng.random((T, top_k)).astype(np.float32)
    tw /= tw.sum(axis=1, keepdims=True)
    xb = S.activations(w, T)
    w13, w2 = S.slot_tensors(w)
    got = R.bf16_to_f32(_run(dev, w, xb, tw, slot, w13, w2, L.MODE_DECODE))
    g, d = dequant_w(w13, w2, w.types, w.hidden, w.inter)
    hot = np.where((slot >= 0) & (slot < w.hot), slot, -1)
    ref = R.ffn_reference(xb, hot, tw, g, d)
    print(f"seed {seed}: T {T} top-{top_k}")
    cold = (hot < 0).all(axis=1)
    assert np.all(got[cold] == 0)
    if (~cold).any():
        l2, l1, cos = R.rel_errors(got[~cold], ref[~cold])
        assert l2 < TOL_REL_L2 and cos > 0.999, (l2, l1, cos)


@pytest.mark.parametrize("top_k", [1, 3, 6, 9, 12, 17])
def test_grouped_mode_any_top_k(dev, top_k):
    """The grouped mode at top-k that are not 8 (the combine reads k's in groups of 8, then of
    2, a group's k's past top_k and its cold routes reading zeros): slot ids mixing hot slots,
    -1 and ids past the table, one token naming one slot top_k times; against the fp64 FFN."""
    L, H, S = _pkg()
    rng = np.random.default_rng(200 + top_k)
    T = 97
    base = S.WORKLOADS["q4_k+q6_k-h2048-n512-e256-k8-hot40-prefill"]
    w = replace(base, hidden=512, inter=256, hot=8, experts=32, top_k=top_k)
    slot = rng.integers(-2, w.hot + 3, size=(T, top_k)).astype(np.int32)
    slot[slot == -2] = -1
    slot[1, :] = slot[1, 0] if slot[1, 0] >= 0 else 0
    tw = rng.random((T, top_k)).astype(np.float32)
    tw /= tw.sum(axis=1, keepdims=True)
    xb = S.activations(w, T)
    w13, w2 = S.slot_tensors(w)
    got = R.bf16_to_f32(_run(dev, w, xb, tw, slot, w13, w2, L.MODE_GROUPED))
    g, d = dequant_w(w13, w2, w.types, w.hidden, w.inter)
    hot = np.where((slot >= 0) & (slot < w.hot), slot, -1)
    ref = R.ffn_reference(xb, hot, tw, g, d)
    cold = (hot < 0).all(axis=1)
    assert np.all(got[cold] == 0)
    l2, l1, cos = R.rel_errors(got[~cold], ref[~cold])
    assert l2 < TOL_REL_L2 and cos > 0.999, (l2, l1, cos)


def test_grouped_edge_cases(dev):
    """Empty slots, a single token, all-cold tokens, slots with one route."""
    L, _, _ = _pkg()
    w, xb, tw, slot, w13, w2 = _case("q4_k+q6_k-h2048-n512-e256-k8-hot40-prefill", 5, 512, 256, 8, 32)
    slot = slot.copy()
    slot[0, :] = -1          # a token with no hot route
    slot[1, :] = -1
    slot[1, 3] = 7           # slot 7 with exactly one route
    for T in (1, 5):
        got = R.bf16_to_f32(_run(dev, w, xb[:T], tw[:T], slot[:T], w13, w2, L.MODE_GROUPED))
        g, d = dequant_w(w13, w2, w.types, w.hidden, w.inter)
        ref = R.ffn_reference(xb[:T], slot[:T], tw[:T], g, d)
        assert np.all(got[0] == 0)
        if T > 1:
            l2, _, _ = R.rel_errors(got, ref)
            assert l2 < TOL_REL_L2


@pytest.mark.parametrize("hot", [400, 512])
def test_grouped_sorts_agree_many_slots(dev, hot):
    """Chunks of up to 4096 routes are sorted by one block (sort_small), longer ones by three
    launches: the first 500 tokens of a 600-token chunk (4800 routes, three launches) equal the
    same 500 tokens alone (4000 routes: one block with 400 slots; three launches with 512,
    whose chunk counts exceed the one block's LDS) bit for bit, at hundreds of slots; both
    against the fp64 FFN."""
    L, _, _ = _pkg()
    w, xb, tw, slot, w13, w2 = _case("q4_k+q6_k-h2048-n512-e256-k8-hot40-prefill", 600, 256, 256, hot, 1024)
    assert len(np.unique(slot[slot >= 0])) > hot // 2
    a = _run(dev, w, xb[:500], tw[:500], slot[:500], w13, w2, L.MODE_GROUPED)
    b = _run(dev, w, xb, tw, slot, w13, w2, L.MODE_GROUPED)
    assert np.array_equal(a, b[:500])
    g, d = dequant_w(w13, w2, w.types, w.hidden, w.inter)
    l2, _, cos = R.rel_errors(R.bf16_to_f32(b), R.ffn_reference(xb, slot, tw, g, d))
    assert l2 < TOL_REL_L2 and cos > 0.999, (l2, cos)


def test_grouped_past_the_combine_grid_limit(dev):
    """70000 tokens (560k routes, hidden 256): the combine runs in slices of 65535 tokens (the
    grid's y limit). Tokens past the first slice equal a call on those tokens alone, bit for
    bit (a token's output depends only on its own routes), and a token sample from both
    slices matches the fp64 FFN."""
    L, _, _ = _pkg()
    T, cut = 70000, 65535
    w, xb, tw, slot, w13, w2 = _case("q4_k+q6_k-h2048-n512-e256-k8-hot40-prefill", T, 256, 256, 8, 32)
    y = _run(dev, w, xb, tw, slot, w13, w2, L.MODE_GROUPED)
    tail = _run(dev, w, xb[cut:], tw[cut:], slot[cut:], w13, w2, L.MODE_GROUPED)
    assert np.array_equal(y[cut:], tail)
    g, d = dequant_w(w13, w2, w.types, w.hidden, w.inter)
    sample = np.concatenate([np.arange(0, cut, 2049), np.arange(cut - 3, T, 157)])
    ref = R.ffn_reference(xb[sample], slot[sample], tw[sample], g, d)
    l2, l1, cos = R.rel_errors(R.bf16_to_f32(y[sample]), ref)
    assert l2 < TOL_REL_L2 and cos > 0.999, (l2, l1, cos)


@pytest.mark.timeout(300)
def test_grouped_past_one_pass(dev):
    """Hidden 7168, top-8: a grouped pass holds 37376 tokens (its Y buffer [R, hidden] bf16
    stays under the kernels' 32-bit offsets), so 37676 tokens run as two passes. The tokens
    of the second pass equal a call on those tokens alone, bit for bit, and a token sample
    from both passes, around the boundary included, matches the fp64 FFN."""
    L, H, _ = _pkg()
    w, xb, tw, slot, w13, w2 = _case("q4_k+q6_k-h2048-n512-e256-k8-hot40-prefill", 37676, 7168, 256, 4, 32)
    desc = L.ktmi_layer(hidden=w.hidden, inter=w.inter, n_slots=w.hot, type13=w.types[0], type2=w.types[2],
                        w13=1 << 20, w2=1 << 21)
    cut = L.lib().ktmi_moe_layer_pass_tokens(desc, w.top_k)
    T = xb.shape[0]
    assert cut == 37376 and T > cut
    print(f"past one pass: {T} tokens, {(slot >= 0).sum()} hot routes", flush=True)
    y = _run(dev, w, xb, tw, slot, w13, w2, L.MODE_GROUPED)
    tail = _run(dev, w, xb[cut:], tw[cut:], slot[cut:], w13, w2, L.MODE_GROUPED)
    assert np.array_equal(y[cut:], tail)
    g, d = dequant_w(w13, w2, w.types, w.hidden, w.inter)
    sample = np.concatenate([np.arange(0, cut - 8, 997), np.arange(cut - 8, T, 31)])
    ref = R.ffn_reference(xb[sample], slot[sample], tw[sample], g, d)
    l2, l1, cos = R.rel_errors(R.bf16_to_f32(y[sample]), ref)
    assert l2 < TOL_REL_L2 and cos > 0.999, (l2, l1, cos)


def test_grouped_short_last_pass(dev):
    """A long call whose last pass is as short as a decode window (top-64, hidden 7168: 4608
    tokens a pass, then 12): the last tokens' outputs are those of one pass over all tokens, bit
    for bit the ones they get at the end of a 300-token call."""
    L, H, S = _pkg()
    base = S.WORKLOADS["q4_k+q6_k-h2048-n512-e256-k8-hot40-prefill"]
    w = replace(base, hidden=7168, inter=256, hot=4, experts=128, top_k=64)
    desc = L.ktmi_layer(hidden=w.hidden, inter=w.inter, n_slots=w.hot, type13=w.types[0], type2=w.types[2],
                        w13=1 << 20, w2=1 << 21)
    cut = L.lib().ktmi_moe_layer_pass_tokens(desc, w.top_k)
    T = cut + 12
    assert cut == 4608
    rng = np.random.default_rng(31)
    slot = np.full((T, w.top_k), -1, np.int32)
    slot[:, 5:9] = rng.integers(-1, w.hot, size=(T, 4))
    tw = rng.random((T, w.top_k)).astype(np.float32)
    xb = S.activations(w, T)
    w13, w2 = S.slot_tensors(w)
    y = _run(dev, w, xb, tw, slot, w13, w2, L.MODE_GROUPED)
    tail = _run(dev, w, xb[-300:], tw[-300:], slot[-300:], w13, w2, L.MODE_GROUPED)
    assert np.array_equal(y[-300:], tail)
    g, d = dequant_w(w13, w2, w.types, w.hidden, w.inter)
    l2, _, cos = R.rel_errors(R.bf16_to_f32(y[cut:]), R.ffn_reference(xb[cut:], slot[cut:], tw[cut:], g, d))
    assert l2 < TOL_REL_L2 and cos > 0.999, (l2, cos)


def test_grouped_at_full_shape(dev):
    """The prefill workload's real layer shape (hidden 2048, inter 512, 40 slots, Q4_K/Q6_K)
    at 1024 tokens, against the fp64 FFN on a sample of tokens."""
    L, _, _ = _pkg()
    w, xb, tw, slot, w13, w2 = _case("q4_k+q6_k-h2048-n512-e256-k8-hot40-prefill", 1024)
    got = R.bf16_to_f32(_run(dev, w, xb, tw, slot, w13, w2, L.MODE_GROUPED))
    g, d = dequant_w(w13, w2, w.types, w.hidden, w.inter)
    sample = np.arange(0, 1024, 8)
    ref = R.ffn_reference(xb[sample], slot[sample], tw[sample], g, d)
    l2, l1, cos = R.rel_errors(got[sample], ref)
    assert l2 < TOL_REL_L2 and cos > 0.999, (l2, l1, cos)


@pytest.mark.parametrize("mode", ["gemv", "decode", "grouped"])
def test_layer_empty_input_and_foreign_ids(dev, mode):
    """T = 0 is a no-op; slot ids >= S or < -1 (experts owned by no slot here) behave exactly
    like -1."""
    import torch

    L, H, _ = _pkg()
    m = {"gemv": L.MODE_GEMV, "decode": L.MODE_DECODE, "grouped": L.MODE_GROUPED}[mode]
    w, xb, tw, slot, w13, w2 = _case("q4_k+q6_k-h2048-n512-e256-k8-hot40-prefill", 24, 512, 256, 8, 32)
    W13, W2 = to_dev(w13, dev), to_dev(w2, dev)
    desc = H.layer_desc(W13, W2, w.hidden, w.inter, w.types[0], w.types[2])
    y0 = H.moe_layer(desc, bf16_tensor(xb[:0], dev), to_dev(tw[:0], dev), to_dev(slot[:0], dev), m)
    torch.cuda.synchronize()
    assert tuple(y0.shape) == (0, w.hidden)
    rng = np.random.default_rng(11)
    pick = rng.random(slot.shape) < 0.3
    foreign = slot.copy()
    foreign[pick] = np.where(rng.random(int(pick.sum())) < 0.5, w.hot + 5, -7).astype(np.int32)
    cold = slot.copy()
    cold[pick] = -1
    a = _run(dev, w, xb, tw, foreign, w13, w2, m)
    b = _run(dev, w, xb, tw, cold, w13, w2, m)
    assert np.array_equal(a, b)


def test_grouped_headline_chunk_properties(dev):
    """The 16384-token prefill chunk at its real shape: a token sample against the fp64 FFN,
    and two size-independent identities that hold bit-exactly because every route's output
    depends only on its own row: permuting the tokens permutes the output, and doubling the
    route weights doubles it."""
    L, _, _ = _pkg()
    T = 16384
    w, xb, tw, slot, w13, w2 = _case("q4_k+q6_k-h2048-n512-e256-k8-hot40-prefill", T)
    y = _run(dev, w, xb, tw, slot, w13, w2, L.MODE_GROUPED)
    g, d = dequant_w(w13, w2, w.types, w.hidden, w.inter)
    sample = np.arange(0, T, 97)
    ref = R.ffn_reference(xb[sample], slot[sample], tw[sample], g, d)
    l2, l1, cos = R.rel_errors(R.bf16_to_f32(y[sample]), ref)
    assert l2 < TOL_REL_L2 and cos > 0.999, (l2, l1, cos)
    perm = np.random.default_rng(12).permutation(T)
    yp = _run(dev, w, xb[perm], tw[perm], slot[perm], w13, w2, L.MODE_GROUPED)
    assert np.array_equal(yp, y[perm])
    y2 = _run(dev, w, xb, tw * np.float32(2), slot, w13, w2, L.MODE_GROUPED)
    assert np.array_equal(R.bf16_to_f32(y2), 2 * R.bf16_to_f32(y))


@pytest.mark.gpu
@pytest.mark.parametrize("mode", ["gemv", "decode", "grouped"])
def test_layer_in_hip_graph(dev, mode):
    """The layer call captured in a HIP graph (no memsets, no host sync inside): every replay,
    with eager layer calls on other inputs between the replays, reproduces the eager output
    bit for bit."""
    import torch

    L, H, _ = _pkg()
    m = {"gemv": L.MODE_GEMV, "decode": L.MODE_DECODE, "grouped": L.MODE_GROUPED}[mode]
    w, xb, tw, slot, w13, w2 = _case("q4_k+q6_k-h2048-n512-e256-k8-hot40-prefill", 12 if mode != "grouped" else 300,
                                     512, 256, 8, 32)
    W13, W2 = to_dev(w13, dev), to_dev(w2, dev)
    desc = H.layer_desc(W13, W2, w.hidden, w.inter, w.types[0], w.types[2])
    T, k = slot.shape
    x, twd, sd = bf16_tensor(xb, dev), to_dev(tw, dev), to_dev(slot, dev)
    lib = L.lib()
    out = torch.empty((T, w.hidden), dtype=torch.bfloat16, device=dev)
    ws = torch.empty((lib.ktmi_moe_layer_workspace(desc, T, k, m),), dtype=torch.uint8, device=dev)
    s = torch.cuda.Stream()
    with torch.cuda.stream(s):
        H.moe_layer(desc, x, twd, sd, m, out, ws)
    torch.cuda.synchronize()
    ref = out.clone()
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g, stream=s):
        H.moe_layer(desc, x, twd, sd, m, out, ws)
    x2 = bf16_tensor(xb[::-1].copy(), dev)
    for r in range(4):
        out.zero_()
        g.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, ref), f"replay {r}"
        H.moe_layer(desc, x2, twd, sd, m)  # eager work between the replays
        torch.cuda.synchronize()


@pytest.mark.parametrize("mode,T", [("grouped", 48), ("grouped", 4096), ("gemv", 8), ("gemv", 64), ("decode", 8),
                                    ("decode", 32)])
def test_slot_address_table_matches_contiguous_slots(dev, mode, T):
    """Slots given as a device table of per-slot addresses (w_is_table, each slot its own
    allocation, in reverse order) give the same bits as the contiguous slot tensors: 128- and
    256-route grouped tiles, the fused decode layer and the stage-by-stage GEMV layer."""
    import torch

    L, H, S = _pkg()
    w = S.WORKLOADS["q4_k+q6_k-h2048-n512-e256-k8-hot40-prefill"]
    _, tw, slot, _ = S.routing(w, T)
    xb = S.activations(w, T)
    w13, w2 = S.slot_tensors(w)
    W13, W2 = to_dev(w13, dev), to_dev(w2, dev)
    m = {"gemv": L.MODE_GEMV, "decode": L.MODE_DECODE, "grouped": L.MODE_GROUPED}[mode]
    x, twd, sd = bf16_tensor(xb, dev), to_dev(tw, dev), to_dev(slot, dev)
    ref = H.moe_layer(H.layer_desc(W13, W2, w.hidden, w.inter, w.types[0], w.types[2]), x, twd, sd, m)
    n = W13.shape[0]
    p13 = [None] * n
    p2 = [None] * n
    for s in reversed(range(n)):
        p13[s], p2[s] = W13[s].clone(), W2[s].clone()
    t13 = torch.tensor([p.data_ptr() for p in p13], dtype=torch.int64, device=dev)
    t2 = torch.tensor([p.data_ptr() for p in p2], dtype=torch.int64, device=dev)
    got = H.moe_layer(H.layer_desc(t13, t2, w.hidden, w.inter, w.types[0], w.types[2], table=True), x, twd, sd, m)
    torch.cuda.synchronize()
    assert np.array_equal(bf16_bits_of(got), bf16_bits_of(ref))


@pytest.mark.parametrize("types", [(R.GGML_Q4_K, R.GGML_Q6_K), (R.GGML_Q6_K, R.GGML_Q4_K), (R.GGML_Q8_0, R.GGML_Q8_0),
                                   (R.GGML_IQ3_S, R.GGML_IQ3_S)])
@pytest.mark.parametrize("hidden,inter,T,mode", [(768, 256, 1, "decode"), (1280, 768, 16, "decode"), (256, 512, 17, "decode"),
                                                 (1280, 256, 32, "grouped"), (512, 1280, 64, "grouped")])
def test_window_columns(dev, types, hidden, inter, T, mode):
    """The decode-sized kernels where the split over super-block columns is ragged (1, 3 and 5
    columns over 4 waves, rings of one column and of more), at 1, 2 and 4 groups of 16 routes a
    pass, past 256 routes and with a slot listed twice (72 routes of one slot: a second pass);
    against the fp64 FFN."""
    L, H, S = _pkg()
    top_k = 9 if mode == "grouped" else 5
    base = S.WORKLOADS["q4_k+q6_k-h2048-n512-e256-k8-hot40-prefill"]
    w = replace(base, hidden=hidden, inter=inter, hot=70, experts=128, top_k=top_k, types=(types[0], types[0], types[1]))
    rng = np.random.default_rng(hidden + inter + T)
    slot = rng.integers(0, 100, size=(T, top_k)).astype(np.int32)
    slot = np.where(slot < w.hot, slot, -1).astype(np.int32)
    slot[:, 0] = 69                 # every token on the last slot
    slot[: T // 8, 1] = 69          # some twice
    if T > 40:
        slot[40:] = np.where(slot[40:] == 69, slot[40:], -1)
    tw = rng.random((T, top_k)).astype(np.float32)
    tw /= tw.sum(axis=1, keepdims=True)
    xb = S.activations(w, T)
    w13, w2 = S.slot_tensors(w)
    got = R.bf16_to_f32(_run(dev, w, xb, tw, slot, w13, w2, L.MODE_DECODE if mode == "decode" else L.MODE_GROUPED))
    g, d = dequant_w(w13, w2, w.types, w.hidden, w.inter)
    l2, l1, cos = R.rel_errors(got, R.ffn_reference(xb, slot, tw, g, d))
    assert l2 < TOL_REL_L2 and cos > 0.999, (l2, l1, cos)


@pytest.mark.parametrize("types,inter", [((R.GGML_Q4_K, R.GGML_Q4_K), 768), ((R.GGML_Q4_K, R.GGML_Q6_K), 768),
                                         ((R.GGML_Q8_0, R.GGML_Q8_0), 288), ((R.GGML_Q8_0, R.GGML_Q8_0), 512),
                                         ((R.GGML_IQ3_S, R.GGML_IQ3_S), 256)])
def test_fused_decode_down_units(dev, types, inter):
    """The fused decode launches where a down row has 8, 9, 12 and 16 weight units: every unit
    is summed (8 lanes a row up to 8 units, 16 past them)."""
    L, _, S = _pkg()
    base = S.WORKLOADS["q4_k+q6_k-h2048-n512-e256-k8-hot40-prefill"]
    w = replace(base, hidden=512, inter=inter, hot=8, experts=32, types=(types[0], types[0], types[1]))
    _, tw, slot, _ = S.routing(w, 3)
    xb = S.activations(w, 3)
    w13, w2 = S.slot_tensors(w)
    got = R.bf16_to_f32(_run(dev, w, xb, tw, slot, w13, w2, L.MODE_GEMV))
    exp = R.bf16_to_f32(gemv_layer_oracle(xb, tw, slot, w13, w2, w.types, w.hidden, w.inter))
    l2, _, _ = R.rel_errors(got, exp)
    assert l2 < 4e-3, l2


@pytest.mark.parametrize("t", [R.GGML_Q8_0, R.GGML_Q4_K, R.GGML_Q6_K, R.GGML_IQ3_S])
@pytest.mark.parametrize("T,mode", [(7, "decode"), (70, "grouped"), (300, "grouped")])
def test_matrix_decoders_over_all_codes(dev, t, T, mode):
    """The matrix kernels' decoders on blocks of random codes and scales with negative, zero and
    the smallest fp16 scales among them, against the fp64 FFN on the exact values."""
    L, _, S = _pkg()
    base = S.WORKLOADS["q4_k+q6_k-h2048-n512-e256-k8-hot40-prefill"]
    w = replace(base, hidden=512, inter=256, hot=5, experts=16, types=(t, t, t))
    rng = np.random.default_rng(t)
    _, tw, slot, _ = S.routing(w, T)
    xb = S.activations(w, T)
    size, at = {R.GGML_Q8_0: (34, (0,)), R.GGML_Q4_K: (144, (0, 2)), R.GGML_Q6_K: (210, (208,)), R.GGML_IQ3_S: (110, (0,))}[t]

    def blocks(a):
        b = rng.integers(0, 256, size=a.shape, dtype=np.uint8).reshape(-1, size)
        for o in at:
            d = (rng.random(b.shape[0]) * 2e-4 * rng.choice([-1.0, 1.0], b.shape[0])).astype(np.float16)
            d[::7], d[3::11] = 0.0, np.float16(6e-8)
            b[:, o:o + 2] = d.view(np.uint8).reshape(-1, 2)
        return b.reshape(a.shape)

    w13, w2 = (blocks(a) for a in S.slot_tensors(w))
    got = R.bf16_to_f32(_run(dev, w, xb, tw, slot, w13, w2, L.MODE_DECODE if mode == "decode" else L.MODE_GROUPED))
    g, d = dequant_w(w13, w2, w.types, w.hidden, w.inter)
    l2, l1, cos = R.rel_errors(got, R.ffn_reference(xb, slot, tw, g, d))
    assert l2 < TOL_REL_L2 and cos > 0.999, (l2, l1, cos)


@pytest.mark.parametrize("types", [(R.GGML_Q4_K, R.GGML_Q6_K), (R.GGML_Q8_0, R.GGML_IQ3_S)])
@pytest.mark.parametrize("T,top_k,hot", [(65, 4, 15), (65, 4, 14), (128, 8, 57), (128, 8, 56), (129, 2, 40)])
def test_window_limits(dev, types, T, top_k, hot):
    """The grouped mode on both sides of the line between the decode-sized kernels and the
    GEMMs (128 tokens, 18 routes a slot, 1024 routes), one slot on every token (several passes
    of 64 routes); against the fp64 FFN."""
    L, _, S = _pkg()
    base = S.WORKLOADS["q4_k+q6_k-h2048-n512-e256-k8-hot40-prefill"]
    w = replace(base, hidden=512, inter=256, hot=hot, experts=128, top_k=top_k, types=(types[0], types[0], types[1]))
    rng = np.random.default_rng(T + hot)
    slot = rng.integers(0, 2 * hot, size=(T, top_k)).astype(np.int32)
    slot = np.where(slot < hot, slot, -1).astype(np.int32)
    slot[:, 0] = 3
    tw = rng.random((T, top_k)).astype(np.float32)
    tw /= tw.sum(axis=1, keepdims=True)
    xb = S.activations(w, T)
    w13, w2 = S.slot_tensors(w)
    got = R.bf16_to_f32(_run(dev, w, xb, tw, slot, w13, w2, L.MODE_GROUPED))
    g, d = dequant_w(w13, w2, w.types, w.hidden, w.inter)
    l2, l1, cos = R.rel_errors(got, R.ffn_reference(xb, slot, tw, g, d))
    assert l2 < TOL_REL_L2 and cos > 0.999, (l2, l1, cos)


def _one_popular_slot(dev, types, hidden, inter, hot, T, top_k, mode):
    """A call whose first slot choice is slot 3 for every token (the others spread over twice the
    slots, half of them cold), against the fp64 FFN."""
    _, _, S = _pkg()
    base = S.WORKLOADS["q4_k+q6_k-h2048-n512-e256-k8-hot40-prefill"]
    w = replace(base, hidden=hidden, inter=inter, hot=hot, experts=2 * hot, top_k=top_k, types=(types[0], types[0], types[1]))
    rng = np.random.default_rng(T + hot)
    slot = rng.integers(0, 2 * hot, size=(T, top_k)).astype(np.int32)
    slot = np.where(slot < hot, slot, -1).astype(np.int32)
    slot[:, 0] = 3
    tw = rng.random((T, top_k)).astype(np.float32)
    tw /= tw.sum(axis=1, keepdims=True)
    xb = S.activations(w, T)
    w13, w2 = S.slot_tensors(w)
    got = R.bf16_to_f32(_run(dev, w, xb, tw, slot, w13, w2, mode))
    g, d = dequant_w(w13, w2, w.types, w.hidden, w.inter)
    l2, l1, cos = R.rel_errors(got, R.ffn_reference(xb, slot, tw, g, d))
    assert l2 < TOL_REL_L2 and cos > 0.999, (l2, l1, cos)


@pytest.mark.parametrize("types", [(R.GGML_Q4_K, R.GGML_Q6_K), (R.GGML_Q6_K, R.GGML_Q4_K), (R.GGML_IQ3_S, R.GGML_Q8_0)])
@pytest.mark.parametrize("T,top_k,hot", [(40, 16, 30), (41, 16, 30), (64, 10, 89), (64, 10, 70), (64, 8, 120), (80, 8, 89)])
def test_window_lines(dev, types, T, top_k, hot):
    """The grouped mode on both sides of the lines between the decode-sized kernels and the GEMMs
    that depend on the weight types: 40 tokens, 640 routes, a chip round of gate/up blocks 0.7
    full (89 slots of 256 rows) and the routes a slot past it."""
    L, _, _ = _pkg()
    _one_popular_slot(dev, types, 512, 256, hot, T, top_k, L.MODE_GROUPED)


@pytest.mark.parametrize("types", [(R.GGML_Q4_K, R.GGML_Q6_K), (R.GGML_Q8_0, R.GGML_IQ3_S)])
@pytest.mark.parametrize("T,top_k,hot,mode", [(48, 2, 70, "decode"), (60, 8, 400, "grouped")])
def test_window_passes_follow_the_mean(dev, types, T, top_k, hot, mode):
    """Many slots with few routes on average take passes of 16 or 32 routes although a slot on
    every token needs several of them."""
    L, _, _ = _pkg()
    _one_popular_slot(dev, types, 256, 256, hot, T, top_k, L.MODE_DECODE if mode == "decode" else L.MODE_GROUPED)


@pytest.mark.parametrize("t", [R.GGML_Q8_0, R.GGML_Q6_K])
@pytest.mark.parametrize("T,mode", [(9, "decode"), (30, "decode"), (60, "decode"), (40, "grouped"), (300, "grouped")])
def test_matrix_decoders_infinite_scale(dev, t, T, mode):
    """A block whose scale is infinite dequantises to +-inf (the codes' signs), also in the matrix
    kernels: activations and all other weights positive, so that a down row with such a block
    gives +-inf, a gate row with one makes its slot's outputs inf, and the rest stays finite."""
    L, _, S = _pkg()
    base = S.WORKLOADS["q4_k+q6_k-h2048-n512-e256-k8-hot40-prefill"]
    w = replace(base, hidden=512, inter=256, hot=3, experts=16, top_k=2, types=(t, t, t))
    rng = np.random.default_rng(t + T)
    size, at = (34, 0) if t == R.GGML_Q8_0 else (210, 208)

    def blocks(shape, neg_row=None, inf_at=()):
        b = np.empty(shape[:2] + (shape[2] // size, size), np.uint8)
        d = rng.uniform(1e-5, 2e-5, b.shape[:3]).astype(np.float16)
        for i in inf_at:
            d[i] = np.inf
        if t == R.GGML_Q8_0:
            q = rng.integers(1, 127, b.shape[:3] + (32,))
            if neg_row is not None:
                q[:, neg_row] *= -1
            b[..., 2:] = q.astype(np.int8).view(np.uint8)
        else:  # codes 33..63, or 1..31 in the negative row
            b[..., :128] = rng.integers(1, 16, b.shape[:3] + (128,)) | rng.integers(1, 16, b.shape[:3] + (128,)) << 4
            hi = rng.integers(0, 256, b.shape[:3] + (64,)) & 0x55
            b[..., 128:192] = hi | 0xAA
            if neg_row is not None:
                b[:, neg_row, :, 128:192] = hi[:, neg_row]
            b[..., 192:208] = rng.integers(1, 128, b.shape[:3] + (16,))
        b[..., at:at + 2] = d.view(np.uint8).reshape(d.shape + (2,))
        return b.reshape(shape)

    s13, s2 = (a.shape for a in S.slot_tensors(w))
    w13 = blocks(s13, inf_at=[(2, 17, 1)])  # gate row 17 of slot 2
    w2 = blocks(s2, neg_row=9, inf_at=[(0, 9, 0), (1, 40, 0)])
    slot = np.stack([np.arange(T) % 3, np.full(T, -1)], 1).astype(np.int32)
    tw = np.full((T, 2), 0.5, np.float32)
    xb = R.bf16_bits(rng.uniform(0.1, 1.0, (T, w.hidden)).astype(np.float32))
    got = R.bf16_to_f32(_run(dev, w, xb, tw, slot, w13, w2, L.MODE_DECODE if mode == "decode" else L.MODE_GROUPED))
    g, d = dequant_w(w13, w2, w.types, w.hidden, w.inter)
    with np.errstate(invalid="ignore"):
        exp = R.ffn_reference(xb, slot, tw, g, d)
    inf = np.isinf(exp)
    assert inf[0::3, 9].all() and inf[1::3, 40].all() and inf[2::3].all() and not inf.all() and not np.isnan(exp).any()
    assert np.array_equal(got[inf], exp[inf].astype(np.float32))
    assert R.rel_errors(got[~inf], exp[~inf])[0] < TOL_REL_L2


def _random_weights(rng, t, shape):
    """Slot weights of random codes with finite scales of both signs, sized as quantised ~N(0, 0.02)
    weights."""
    size, at, mag = {R.GGML_Q8_0: (34, (0,), 3e-4), R.GGML_Q4_K: (144, (0, 2), 1e-4), R.GGML_Q6_K: (210, (208,), 2e-5),
                     R.GGML_IQ3_S: (110, (0,), 2e-4)}[t]
    b = rng.integers(0, 256, size=shape, dtype=np.uint8).reshape(-1, size)
    for o in at:
        d = (rng.uniform(0.5, 1.0, b.shape[0]) * mag * rng.choice([-1.0, 1.0], b.shape[0])).astype(np.float16)
        b[:, o:o + 2] = d.view(np.uint8).reshape(-1, 2)
    return b.reshape(shape)


@pytest.mark.parametrize("types", [(R.GGML_Q8_0, R.GGML_Q8_0), (R.GGML_Q4_K, R.GGML_Q6_K), (R.GGML_Q6_K, R.GGML_Q4_K),
                                   (R.GGML_IQ3_S, R.GGML_IQ3_S)])
@pytest.mark.parametrize("hidden,inter", [(4096, 1024), (7168, 512)])
@pytest.mark.parametrize("T,top_k", [(9, 2), (30, 3), (50, 4), (38, 8)])
def test_window_long_rows(dev, types, hidden, inter, T, top_k):
    """The decode-sized kernels where a wave takes 4 and 7 columns of a gate/up row and 2 and 4 of a
    down row, so that both buffers of its ring are filled again: passes of 16, 32 and 64 routes,
    up to 256 routes and (but for Q6_K gate/up, which the grouped mode's GEMMs take) past them,
    twice with the same bits; against the fp64 FFN."""
    L, _, S = _pkg()
    base = S.WORKLOADS["q4_k+q6_k-h2048-n512-e256-k8-hot40-prefill"]
    w = replace(base, hidden=hidden, inter=inter, hot=3, experts=16, top_k=top_k, types=(types[0], types[0], types[1]))
    rng = np.random.default_rng(types[0] + hidden + T)
    slot = rng.integers(-1, w.hot, size=(T, top_k)).astype(np.int32)
    slot[:, 0] = 1
    tw = rng.random((T, top_k)).astype(np.float32)
    tw /= tw.sum(axis=1, keepdims=True)
    xb = S.activations(w, T)
    w13 = _random_weights(rng, types[0], (w.hot, 2 * inter, R.row_bytes(hidden, types[0])))
    w2 = _random_weights(rng, types[1], (w.hot, hidden, R.row_bytes(inter, types[1])))
    mode = L.MODE_DECODE if T * top_k <= 256 else L.MODE_GROUPED
    y = _run(dev, w, xb, tw, slot, w13, w2, mode)
    assert np.array_equal(y, _run(dev, w, xb, tw, slot, w13, w2, mode))
    g, d = dequant_w(w13, w2, w.types, w.hidden, w.inter)
    l2, l1, cos = R.rel_errors(R.bf16_to_f32(y), R.ffn_reference(xb, slot, tw, g, d))
    assert l2 < TOL_REL_L2 and cos > 0.999, (l2, l1, cos)


@pytest.mark.parametrize("case", CASES, ids=[c[0].split("-")[0] for c in CASES])
def test_gemms_vs_ffn_reference(dev, case):
    """The layer reference test on the sort, the GEMMs and their combine (160 tokens: past the
    chunks that the grouped mode gives to the decode-sized kernels)."""
    test_layer_vs_ffn_reference(dev, (case[0], 160) + tuple(case[2:]), "grouped")


def test_slot_address_table_128_route_tiles(dev):
    """Slot address tables against contiguous slots in the GEMMs of 128-route tiles."""
    test_slot_address_table_matches_contiguous_slots(dev, "grouped", 300)


@pytest.mark.parametrize("top_k", [1, 5])
def test_gemm_edge_cases(dev, top_k):
    """The sort, the GEMMs and their combine on an empty slot, a slot of one route, tokens without a
    hot route (exactly zero) and slot ids of no slot here (the same bits as -1); against the fp64 FFN."""
    L, _, S = _pkg()
    base = S.WORKLOADS["q4_k+q6_k-h2048-n512-e256-k8-hot40-prefill"]
    w = replace(base, hidden=512, inter=256, hot=8, experts=32, top_k=top_k)
    T = 150
    rng = np.random.default_rng(41 + top_k)
    slot = rng.integers(-1, 5, size=(T, top_k)).astype(np.int32)  # slots 5 and 6 empty
    slot[:10] = -1
    slot[77, 0] = 7
    tw = rng.random((T, top_k)).astype(np.float32)
    xb = S.activations(w, T)
    w13, w2 = S.slot_tensors(w)
    y = _run(dev, w, xb, tw, slot, w13, w2, L.MODE_GROUPED)
    foreign = np.where(slot < 0, rng.choice([-7, w.hot, w.hot + 5], size=slot.shape), slot).astype(np.int32)
    assert np.array_equal(y, _run(dev, w, xb, tw, foreign, w13, w2, L.MODE_GROUPED))
    got = R.bf16_to_f32(y)
    cold = (slot < 0).all(axis=1)
    assert cold[:10].all() and np.all(got[cold] == 0)
    g, d = dequant_w(w13, w2, w.types, w.hidden, w.inter)
    l2, l1, cos = R.rel_errors(got[~cold], R.ffn_reference(xb, slot, tw, g, d)[~cold])
    assert l2 < TOL_REL_L2 and cos > 0.999, (l2, l1, cos)
