"""GPU parity of the megakernel (through the C ABI) against the CPU oracle.

Bars: residual stream after every layer within
rel-L2 1e-2, fp32 logits within 2e-2 abs, greedy tokens identical wherever the
oracle's top-1/top-2 margin exceeds 2e-2.  Bit-exact: synthetic generator,
KV-cache bytes (bf16 of the oracle's post-norm, post-RoPE K and V), argmax
tie-break.
"""
from __future__ import annotations

import ctypes
import time

import numpy as np
import pytest
import torch

from megakernel_amd import _lib
from megakernel_amd.bridge import MegakernelEngine
from megakernel_amd.weights import DeviceWeights
from megakernel_amd.config import BASELINE, QWEN3_06B, TINY
from oracle import qwen3_ref, synth

from ._helpers import check_kv_bf16, check_step, check_tokens_teacher_forced, make_pair, rel_l2

pytestmark = pytest.mark.gpu

BASELINE_2L = BASELINE.with_(n_layers=2, vocab=4096)


def _print(*a):
    print(*a, flush=True)


def test_synth_fill_bit_exact(lib):
    """Device generator == numpy restatement (incl. indices past 2^32)."""
    n = 1 << 20
    for std, add_one in [(0.02, 0), (1.0, 0), (0.1, 1)]:
        key = synth.stream_key(123, 7)
        c = float(synth.scale_const(std))
        d = lib.megakernel_device_alloc(2 * n)
        assert d
        _lib.check(lib, lib.megakernel_synth_fill(ctypes.c_void_p(d), n, key, c, add_one), "fill")
        got = np.empty(n, dtype=np.uint16)
        _lib.check(lib, lib.megakernel_memcpy(got.ctypes.data_as(ctypes.c_void_p), ctypes.c_void_p(d),
                                              2 * n, _lib.D2H), "d2h")
        lib.megakernel_device_free(ctypes.c_void_p(d))
        ref = synth.normal_bf16_bits(key, n, std, add_one=bool(add_one))
        assert np.array_equal(got, ref), f"std={std} add_one={add_one}"


def test_tiny_matches_hf_golden_and_oracle():
    """TINY preset against the committed HF fixture (inputs and outputs)."""
    z = np.load("tests/golden/hf_qwen3_tiny.npz")
    eng, orc, dw = make_pair(TINY, int(z["seed"]), 64, gain_std=float(z["gain_std"]))
    try:
        worst_l = worst_g = 0.0
        for i, tok in enumerate(z["tokens_fed"]):
            _print(f"tiny step {i} token {tok}")
            nxt, layers, logits = eng.debug_forward(int(tok))
            ref = orc.step(int(tok), capture=True)
            l2, la = check_step(layers, logits, ref, f"tiny step {i}")
            worst_l, worst_g = max(worst_l, l2), max(worst_g, la)
            # HF fixture (fp32 KV) is within the same bars
            assert rel_l2(layers, z["layers"][i]).max() <= 1e-2
            assert np.abs(logits - z["logits"][i]).max() <= 2e-2
            if nxt != ref["token"]:
                assert qwen3_ref.top2_margin(ref["logits"]) <= 2e-2
        _print(f"tiny worst layer relL2 {worst_l:.2e} logits abs {worst_g:.2e}")
    finally:
        eng.close()
        dw.free()


def test_baseline_2l_matches_hf_golden():
    z = np.load("tests/golden/hf_qwen3_baseline_2l.npz")
    eng, orc, dw = make_pair(BASELINE_2L, int(z["seed"]), 64, gain_std=float(z["gain_std"]))
    try:
        for i, tok in enumerate(z["tokens_fed"]):
            _print(f"baseline_2l step {i} token {tok}")
            nxt, layers, logits = eng.debug_forward(int(tok))
            ref = orc.step(int(tok), capture=True)
            l2, la = check_step(layers, logits, ref, f"step {i}")
            _print(f"  relL2 {l2:.2e} logits {la:.2e}")
            assert rel_l2(layers, z["layers"][i]).max() <= 1e-2
            assert np.abs(logits - z["logits"][i]).max() <= 2e-2
    finally:
        eng.close()
        dw.free()


def test_generate_equals_decode_and_oracle():
    """One resident launch of n tokens == n single-token launches == oracle."""
    eng, orc, dw = make_pair(BASELINE_2L, 5, 256)
    try:
        prompt = synth.prompt_tokens(5, 8, BASELINE_2L.vocab)
        for t in prompt[:-1]:
            eng.decode_token(t)
        a0 = eng.decode_token(prompt[-1])
        gen = eng.decode_many(a0, 40)
        eng.reset()
        for t in prompt[:-1]:
            eng.decode_token(t)
        b = [eng.decode_token(prompt[-1])]
        for _ in range(40):
            b.append(eng.decode_token(b[-1]))
        assert [a0] + gen == b, "generate() and per-token decode disagree"
        assert eng.pos == len(prompt) + 40
        for t in prompt[:-1]:
            orc.step(t)
        same, low = check_tokens_teacher_forced([prompt[-1], a0] + gen[:-1], [a0] + gen, orc)
        _print(f"teacher-forced: {same} identical, {low} low-margin differences")
    finally:
        eng.close()
        dw.free()


def test_kv_cache_bytes_exact():
    """Cache bytes appended by the kernel == bf16 of the oracle's K/V."""
    eng, orc, dw = make_pair(TINY, 3, 64)
    try:
        toks = [5, 77, 901, 13]
        for t in toks:
            eng.decode_token(t)
            orc.step(t)
        kv = eng.get_kv(len(toks))  # [L][2][NKV][len][D]
        ref_k = orc.k_cache[:, :, :len(toks)].contiguous().view(torch.int16).numpy().view(np.uint16)
        ref_v = orc.v_cache[:, :, :len(toks)].contiguous().view(torch.int16).numpy().view(np.uint16)
        # fp32 accumulation order differs, so a value can land on the other
        # side of a bf16 rounding boundary: allow 1 ulp, require >= 99% exact.
        for got, ref, name in [(kv[:, 0], ref_k, "K"), (kv[:, 1], ref_v, "V")]:
            diff = np.abs(got.astype(np.int32) - ref.astype(np.int32))
            assert diff.max() <= 1, f"{name} cache differs by {diff.max()} bf16 ulps"
            assert (diff == 0).mean() >= 0.99, f"{name} exact fraction {(diff == 0).mean()}"
    finally:
        eng.close()
        dw.free()


def test_set_get_kv_roundtrip_and_synthetic_prefill():
    eng, orc, dw = make_pair(TINY, 9, 300)
    try:
        s = TINY
        n = 200
        eng.fill_kv_synthetic(n, 42)
        got = eng.get_kv(n)
        for layer in range(s.n_layers):
            for kv in range(2):
                ref = synth.kv_prefill_bits(42, layer, kv, n, s.n_kv_heads, s.head_dim)
                assert np.array_equal(got[layer, kv], ref), (layer, kv)
        rng = np.random.default_rng(0)
        host = rng.integers(0, 1 << 15, size=got.shape, dtype=np.uint16)
        eng.set_kv(host)
        assert eng.pos == n
        assert np.array_equal(eng.get_kv(n), host)
    finally:
        eng.close()
        dw.free()


@pytest.mark.parametrize("ctx,chunk,merge", [(200, 256, None), (1500, 64, None), (1500, 64, 64), (5000, 256, 4),
                                             (8192, 256, None), (8192, 256, 8), (32768, 256, None)])
def test_long_context_split_attention(ctx, chunk, merge):
    """Prefilled cache + multi-split attention vs the oracle (BASELINE configs[3]
    positions 8192 and 32768 included: 32 splits of up to 32 blocks).  Beyond
    `merge` splits per kv head (default 20) the first split's workgroup merges
    them and the O phase reads one merged partial; at or below it every O
    workgroup merges the splits."""
    shape = BASELINE.with_(n_layers=2, vocab=2048)
    eng, orc, dw = make_pair(shape, 21, ctx + 8)
    try:
        eng.set_attention_chunk(chunk)
        if merge is not None:
            eng.set_attention_merge(merge)
        eng.fill_kv_synthetic(ctx, 77)
        ks = np.stack([synth.kv_prefill_bits(77, l, 0, ctx, shape.n_kv_heads, shape.head_dim)
                       for l in range(shape.n_layers)])
        vs = np.stack([synth.kv_prefill_bits(77, l, 1, ctx, shape.n_kv_heads, shape.head_dim)
                       for l in range(shape.n_layers)])
        orc.set_kv(ks, vs)
        tok = 3
        for i in range(3):
            _print(f"ctx {ctx} chunk {chunk} step {i}")
            nxt, layers, logits = eng.debug_forward(tok)
            ref = orc.step(tok, capture=True)
            check_step(layers, logits, ref, f"ctx {ctx} step {i}")
            tok = ref["token"]
    finally:
        eng.close()
        dw.free()


def test_long_context_class_kernel_chunk():
    """Past eight 512-position splits per kv head the launch widens its
    attention chunk (at most 640 positions) so that eight splits hold the
    context and the class kernel runs: ctx 4,200 takes chunks of 544, then
    launches ending past 4,352 positions take 576 (a new split layout, the
    packed-pair words cleared between them).  Debug steps at the bars, then
    three 60-token launches teacher-forced against the oracle."""
    shape = BASELINE.with_(n_layers=2, vocab=2048)
    ctx = 4200
    eng, orc, dw = make_pair(shape, 23, ctx + 256)
    try:
        eng.fill_kv_synthetic(ctx, 78)
        ks = np.stack([synth.kv_prefill_bits(78, l, 0, ctx, shape.n_kv_heads, shape.head_dim)
                       for l in range(shape.n_layers)])
        vs = np.stack([synth.kv_prefill_bits(78, l, 1, ctx, shape.n_kv_heads, shape.head_dim)
                       for l in range(shape.n_layers)])
        orc.set_kv(ks, vs)
        assert eng.decode_kernel_for(1) == _lib.KERNEL_CLASS
        tok = 3
        for i in range(2):
            _print(f"ctx {ctx} step {i}")
            nxt, layers, logits = eng.debug_forward(tok)
            ref = orc.step(tok, capture=True)
            check_step(layers, logits, ref, f"ctx {ctx} step {i}")
            tok = ref["token"]
        for j in range(3):
            assert eng.decode_kernel_for(60) == _lib.KERNEL_CLASS
            gen = eng.decode_many(tok, 60)
            same, low = check_tokens_teacher_forced([tok] + gen[:-1], gen, orc)
            _print(f"  launch {j} at {eng.pos - 60}: {same} identical, {low} low-margin")
            tok = gen[-1]
    finally:
        eng.close()
        dw.free()


def test_reconfigure_and_rewind_between_launches():
    """The packed-pair hand-off words are not cleared before each launch, only
    when the position moves back or the split / merge configuration changes.
    Toggling the merge off for five tokens (the merged row's 4-bit tag then
    repeats: 5 x 141 phases is a multiple of 15) and back on, then rewinding,
    must still match the oracle and reproduce earlier steps bit for bit; a
    rewound resident launch must equal per-token decoding from the same point."""
    shape = BASELINE.with_(n_layers=2, vocab=2048)
    ctx = 2000
    eng, orc, dw = make_pair(shape, 31, ctx + 64)
    try:
        eng.set_attention_chunk(64)  # 32 splits per kv head at ctx 2000: above merge_min 20
        eng.fill_kv_synthetic(ctx, 5)
        ks = np.stack([synth.kv_prefill_bits(5, l, 0, ctx, shape.n_kv_heads, shape.head_dim)
                       for l in range(shape.n_layers)])
        vs = np.stack([synth.kv_prefill_bits(5, l, 1, ctx, shape.n_kv_heads, shape.head_dim)
                       for l in range(shape.n_layers)])
        orc.set_kv(ks, vs)
        tok, first = 9, []
        for i, merge in enumerate([20, 20, 20, 64, 64, 64, 64, 64, 20, 20]):
            eng.set_attention_merge(merge)
            _print(f"step {i} pos {eng.pos} merge_min {merge}")
            nxt, layers, logits = eng.debug_forward(tok)
            ref = orc.step(tok, capture=True)
            check_step(layers, logits, ref, f"step {i} merge_min {merge}")
            first.append((tok, logits))
            tok = ref["token"]
        # rewind to step 1 (same merge_min as then): bitwise the same step
        eng.set_attention_merge(20)
        eng.set_pos(ctx + 1)
        _, _, again = eng.debug_forward(first[1][0])
        assert np.array_equal(again, first[1][1]), "rewound step differs from the first pass"
        eng.set_pos(ctx)
        gen = eng.decode_many(first[0][0], 8)
        eng.set_pos(ctx)
        b = [eng.decode_token(first[0][0])]
        for _ in range(7):
            b.append(eng.decode_token(b[-1]))
        assert gen == b, "rewound resident launch and per-token decode disagree"
    finally:
        eng.close()
        dw.free()


def test_full_baseline_model_parity():
    """The BASELINE model at full size (28 layers, vocab 151936)."""
    eng, orc, dw = make_pair(BASELINE, 2024, 64, gain_std=0.0, bits_from_device=True)
    try:
        prompt = synth.prompt_tokens(2024, 4, BASELINE.vocab)
        tok = prompt[0]
        for i in range(6):
            tin = prompt[i] if i < len(prompt) else tok
            _print(f"full model step {i} token {tin}")
            nxt, layers, logits = eng.debug_forward(tin)
            ref = orc.step(tin, capture=True)
            l2, la = check_step(layers, logits, ref, f"full step {i}")
            _print(f"  relL2 {l2:.2e} logits abs {la:.2e} margin {qwen3_ref.top2_margin(ref['logits']):.3f}")
            if nxt != ref["token"]:
                assert qwen3_ref.top2_margin(ref["logits"]) <= 2e-2
            tok = nxt
    finally:
        eng.close()
        dw.free()


def test_determinism_bitwise():
    """Two identical runs produce bitwise-identical logits and tokens."""
    eng, _, dw = make_pair(BASELINE_2L, 8, 128)
    try:
        outs = []
        for _ in range(2):
            eng.reset()
            eng.fill_kv_synthetic(60, 1)
            _, layers, logits = eng.debug_forward(17)
            toks = eng.decode_many(5, 20)
            outs.append((layers, logits, toks))
        assert np.array_equal(outs[0][0], outs[1][0])
        assert np.array_equal(outs[0][1], outs[1][1])
        assert outs[0][2] == outs[1][2]
    finally:
        eng.close()
        dw.free()


def test_error_paths():
    """Bad inputs are rejected on the host with an error, not run."""
    eng, _, dw = make_pair(TINY, 1, 16)
    lib = eng.lib
    try:
        assert lib.megakernel_decode(eng._handle, TINY.vocab) == -1
        assert "token id" in _lib.last_error(lib)
        eng.set_pos(16)
        assert lib.megakernel_decode(eng._handle, 1) == -1
        assert "exceeds KV capacity" in _lib.last_error(lib)
        eng.reset()
        assert eng.pos == 0
        assert eng.decode_token(1) >= 0
    finally:
        eng.close()
        dw.free()


@pytest.mark.parametrize("chunk,merge", [(64, None), (32, 4)])
def test_qwen3_preset_head_dim_128(chunk, merge):
    """The reference's own config.cuh shapes (head_dim 128, ffn 3072) in the
    spread kernel, which keeps the chunk it is given (the automatic choice
    would widen it to four splits for the class kernel): chunk 64 gives 5
    splits, chunk 32 gives 10, merged by the first split's workgroup (merge
    threshold 4)."""
    shape = QWEN3_06B.with_(n_layers=2, vocab=2048)
    eng, orc, dw = make_pair(shape, 31, 400)
    try:
        eng.set_decode_kernel(_lib.KERNEL_SPREAD)
        eng.set_attention_chunk(chunk)
        if merge is not None:
            eng.set_attention_merge(merge)
        eng.fill_kv_synthetic(300, 5)
        ks = np.stack([synth.kv_prefill_bits(5, l, 0, 300, shape.n_kv_heads, shape.head_dim) for l in range(2)])
        vs = np.stack([synth.kv_prefill_bits(5, l, 1, 300, shape.n_kv_heads, shape.head_dim) for l in range(2)])
        orc.set_kv(ks, vs)
        tok = 11
        for i in range(3):
            nxt, layers, logits = eng.debug_forward(tok)
            ref = orc.step(tok, capture=True)
            check_step(layers, logits, ref, f"qwen3 step {i}")
            tok = ref["token"]
    finally:
        eng.close()
        dw.free()


@pytest.mark.parametrize("which,prefix,prompt_len", [("tiny", 20, 37), ("baseline_2l", 300, 70), ("tiny", 0, 1)])
def test_batch1_prefill_then_decode(which, prefix, prompt_len):
    """megakernel_prefill on a batch-1 handle (up to 1,024 prompt tokens per weight
    pass, the batched kernels on this handle's own cache), then decode: the
    token after the prompt and the following steps against the oracle stepped
    through the same prompt; the prompt's layer-0 K / V (which depend on each
    token alone) equal bf16 of the oracle's (check_kv_bf16)."""
    shape = TINY if which == "tiny" else BASELINE.with_(n_layers=2, vocab=2048)
    eng, orc, dw = make_pair(shape, 51, prefix + prompt_len + 16)
    try:
        eng.attach_prefill(dw)
        if prefix:
            eng.fill_kv_synthetic(prefix, 9)
            ks = np.stack([synth.kv_prefill_bits(9, l, 0, prefix, shape.n_kv_heads, shape.head_dim)
                           for l in range(shape.n_layers)])
            vs = np.stack([synth.kv_prefill_bits(9, l, 1, prefix, shape.n_kv_heads, shape.head_dim)
                           for l in range(shape.n_layers)])
            orc.set_kv(ks, vs)
        rng = np.random.default_rng(prompt_len)
        prompt = [int(t) for t in rng.integers(0, shape.vocab, size=prompt_len)]
        print(f"batch-1 prefill {which} prefix {prefix} prompt {prompt_len}", flush=True)
        nxt = eng.prefill(prompt)
        assert eng.pos == prefix + prompt_len
        ref = None
        for t in prompt:
            ref = orc.step(t, capture=True)
        if nxt != ref["token"]:
            assert qwen3_ref.top2_margin(ref["logits"]) <= 2e-2, f"prefill token {nxt} != oracle {ref['token']}"
        got = eng.get_kv(prefix + prompt_len)[0, :, :, prefix:, :]  # layer 0: [2][NKV][len][D]
        want = np.stack([orc.k_cache[0, :, prefix:prefix + prompt_len].contiguous().view(torch.int16).numpy(),
                         orc.v_cache[0, :, prefix:prefix + prompt_len].contiguous().view(torch.int16).numpy()]
                        ).view(np.uint16)
        check_kv_bf16(got, want, "layer-0 prompt KV")
        tok = ref["token"]
        for i in range(3):
            _, layers, logits = eng.debug_forward(tok)
            r = orc.step(tok, capture=True)
            check_step(layers, logits, r, f"decode {i} after prefill")
            tok = r["token"]
    finally:
        eng.close()
        dw.free()


def test_batch1_generate_with_prefill_matches_oracle():
    """generate_ids with the prefill context: the prompt in one call, then the
    greedy continuation in one resident launch, against the oracle."""
    shape = TINY
    eng, orc, dw = make_pair(shape, 52, 128, gain_std=0.0)
    try:
        eng.attach_prefill(dw)
        prompt = synth.prompt_tokens(52, 21, shape.vocab)
        gen, _ = eng.generate_ids(prompt, max_tokens=12)
        ref = None
        for t in prompt:
            ref = orc.step(t, capture=True)
        toks = [ref["token"]]
        margins = [qwen3_ref.top2_margin(ref["logits"])]
        for _ in range(11):
            r = orc.step(toks[-1], capture=True)
            toks.append(r["token"])
            margins.append(qwen3_ref.top2_margin(r["logits"]))
        for i, (a, b) in enumerate(zip(gen, toks)):
            if a != b:  # a near-tie may flip; everything after it is a different continuation
                assert margins[i] <= 2e-2, f"token {i}: {a} != oracle {b} (margin {margins[i]:.4f})"
                break
    finally:
        eng.close()
        dw.free()


def test_batch1_prefill_errors():
    shape = TINY
    eng, _, dw = make_pair(shape, 53, 32)
    try:
        with pytest.raises(_lib.MegakernelError, match="attach"):
            eng.prefill([1, 2])
        eng.attach_prefill(dw)
        with pytest.raises(_lib.MegakernelError, match="capacity"):
            eng.prefill([1] * 33)
        with pytest.raises(_lib.MegakernelError, match="token"):
            eng.prefill([shape.vocab])
        assert eng.pos == 0
        eng.prefill([3] * 32)
        assert eng.pos == 32
    finally:
        eng.close()
        dw.free()
    q = QWEN3_06B.with_(n_layers=1, vocab=256)
    eng, _, dw = make_pair(q, 54, 16)
    try:
        with pytest.raises(_lib.MegakernelError, match="BASELINE and TINY"):
            eng.attach_prefill(dw)
    finally:
        eng.close()
        dw.free()


@pytest.mark.parametrize("use_prefill", [False, True])
def test_generate_text_stops_at_eos(use_prefill, capsys):
    """MegakernelEngine.generate (reference host/bridge.py:118-192) with a
    byte tokenizer.  The engine's greedy ids, fed back to the oracle after the
    same prompt, equal the oracle's argmax wherever its top-1/top-2 margin
    exceeds 2e-2.  With EOS set to the engine's k-th token (its first
    occurrence; k >= 2 when the continuation has a new token there) generation
    stops right after it (EOS included), print_stream prints each token as it
    comes, and the returned text is the decoded prompt + generation with
    special tokens skipped."""
    from megakernel_amd.tokenizer import ByteTokenizer
    shape = TINY
    eng, orc, dw = make_pair(shape, 61, 128)
    try:
        if use_prefill:
            eng.attach_prefill(dw)
        prompt = "greedy decode on gfx950"
        ids = ByteTokenizer(shape.vocab).encode(prompt)
        free, _ = eng.generate_ids(ids, max_tokens=12)  # no EOS: 12 tokens
        for t in ids[:-1]:
            orc.step(t)
        check_tokens_teacher_forced([ids[-1]] + free[:-1], free, orc)
        firsts = [i for i in range(len(free)) if free[i] not in free[:i]]
        k = next((i for i in firsts if i >= 2), firsts[-1])
        tok = ByteTokenizer(shape.vocab, eos_token_id=free[k])
        eng.tokenizer = tok
        gen, _ = eng.generate_ids(ids, max_tokens=12, eos_id=tok.eos_token_id)
        assert gen == free[:k + 1], f"with EOS {free[k]}: {gen}, expected {free[:k + 1]}"
        capsys.readouterr()
        text, tps = eng.generate(prompt, max_tokens=12, print_stream=True)
        printed = capsys.readouterr().out
        assert text == tok.decode(ids + free[:k + 1], skip_special_tokens=True)
        assert printed == "".join(tok.decode([t]) for t in free[:k + 1]) + "\n"
        assert k == 0 or tps > 0
    finally:
        eng.close()
        dw.free()


def test_dataflow_handoff_selftest():
    """The hand-off primitive on its own, across every CU and XCD: 20,000
    all-gather rounds of tagged words (full tags and 4-bit packed pairs) with
    the decode kernel's write-through stores and agent-scope polling loads;
    no word may be accepted with the right tag and a wrong value."""
    lib = _lib.load()
    bad, us = ctypes.c_int(-1), ctypes.c_float(0.0)
    rc = lib.megakernel_selftest_dataflow(20000, ctypes.byref(bad), ctypes.byref(us))
    print(f"selftest: mismatches {bad.value}, {us.value:.2f} us per all-gather round", flush=True)
    assert rc == 0, _lib.last_error(lib)
    assert bad.value == 0
    assert 0.0 < us.value < 100.0


def test_bridge_benchmark_and_sweep():
    """MegakernelEngine.benchmark (the reference bridge's per-call loop: five
    warm-up tokens, reset, num_tokens timed calls) and benchmark_sweep (KV
    prefilled to each position, one timed resident launch): positive finite
    rates, the position they leave behind, and bandwidth figures under the
    HBM peak; the per-call loop's tokens are those of one resident launch."""
    eng, orc, dw = make_pair(BASELINE_2L, 83, 640)
    try:
        tps = eng.benchmark(num_tokens=20, prompt_token=3)
        _print(f"benchmark: {tps:.1f} tok/s")
        assert np.isfinite(tps) and tps > 0 and eng.pos == 20
        eng.reset()
        per_call = [eng.decode_token(3)]
        for _ in range(19):
            per_call.append(eng.decode_token(per_call[-1]))
        eng.reset()
        assert eng.decode_many(3, 20) == per_call
        res = eng.benchmark_sweep(positions=[1, 100, 500], bench_tokens=8)
        _print("sweep: " + ", ".join(f"{r['position']}: {r['tok_per_sec']:.0f} tok/s" for r in res))
        assert [r["position"] for r in res] == [1, 100, 500]
        for r in res:
            assert r["tok_per_sec"] > 0 and r["latency_us"] > 0 and 0 < r["bw_util"] < 1.0
        assert eng.pos == 500 + 8
    finally:
        eng.close()
        dw.free()


def test_resident_launch_opens_an_attention_split():
    """A resident launch whose later tokens need one more attention split than
    its first ones: the workgroups of that split have no role before it opens,
    and must not score the LM head from an x word of an earlier layer (4-bit
    tags repeat every 15 phases = 3 layers).  The resident tokens equal the
    per-token path's, whose launches hold exactly their token's splits."""
    shape = BASELINE.with_(n_layers=7, vocab=8192)
    dw = DeviceWeights(shape, 77, gain_std=0.1)
    eng = MegakernelEngine(shape=shape, max_seq=512, device_weights=dw)
    try:
        eng.set_attention_chunk(64)
        for i, start in enumerate([58, 122, 186, 250, 314, 378] * 2):
            eng.fill_kv_synthetic(start, 5 + i)
            n = 10
            assert eng.decode_kernel_for(n) == _lib.KERNEL_CLASS
            got = eng.decode_many(11 + 97 * i, n)
            eng.set_pos(start)
            tok, want = 11 + 97 * i, []
            for _ in range(n):
                tok = eng.decode_token(tok)
                want.append(tok)
            assert got == want, f"start {start}: resident {got}, per token {want}"
    finally:
        eng.close()
        dw.free()


@pytest.mark.parametrize("kv8", [False, True])
@pytest.mark.parametrize("head", [_lib.LMHEAD_BF16, _lib.LMHEAD_FP8, _lib.LMHEAD_SCREENED])
@pytest.mark.parametrize("ctx", [1, 255, 700, 1016, 1300, 1530, 1600])
def test_qwen3_class_kernel_equals_spread(ctx, head, kv8):
    """head_dim 128: the class kernel (two QKV blocks per workgroup, one to
    four splits) against the spread kernel on the same cache, for both cache
    formats and every LM head; resident == per token (1,530 ends in the class
    kernel's range, 1,600 past it).  Up to 1,024 positions both kernels cut
    the context alike and every word is the same.  Past that the class
    kernel's splits are wider (up to 384): the same sums in other groups, equal
    to the packed partials' 2^-20 rounding carried through four layers (1e-4).
    On an FP8 cache the five appended rows may then round to the next code
    (2^-4 of an entry) in every layer; they hold about 5 / 1,300 of the
    attention's weight: 2^-4 * 5 / 1,300 = 2.4e-4 a layer, 1e-3 for four.  The
    screened head scores validation outputs with the bf16 head; its tokens are
    the bf16 head's."""
    shape = QWEN3_06B.with_(n_layers=4, vocab=4096)
    dw = DeviceWeights(shape, 31, gain_std=0.1)
    eng = MegakernelEngine(shape=shape, max_seq=2048, device_weights=dw)
    try:
        eng.set_kv_fp8(kv8)
        eng.fill_kv_synthetic(ctx, 9)
        if head == _lib.LMHEAD_SCREENED:
            bf16_ids = eng.decode_many(5, 5)
            eng.set_pos(ctx)
        eng.set_lmhead_fp8(head)
        assert eng.decode_kernel_for(6) == (_lib.KERNEL_SPREAD if ctx > 1536 else _lib.KERNEL_CLASS)
        got = eng.decode_many(5, 5)
        if head == _lib.LMHEAD_SCREENED:
            assert got == bf16_ids
        nxt, layers, logits = eng.debug_forward(got[-1])
        eng.set_pos(ctx)
        tok, want = 5, []
        for _ in range(5):
            tok = eng.decode_token(tok)
            want.append(tok)
        assert got == want
        eng.set_decode_kernel(_lib.KERNEL_SPREAD)
        eng.set_pos(ctx)
        assert eng.decode_many(5, 5) == got
        nxt_s, layers_s, logits_s = eng.debug_forward(got[-1])
        assert nxt_s == nxt
        err = max(rel_l2(layers, layers_s).max(), rel_l2(logits, logits_s))
        print(f"ctx {ctx} head {head} kv8 {kv8}: class / spread differ by {err:.2e}", flush=True)
        if ctx + 6 <= 1024 or ctx > 1536:
            assert np.array_equal(layers, layers_s) and np.array_equal(logits, logits_s)
        else:
            assert err < (1e-3 if kv8 else 1e-4)
    finally:
        eng.close()
        dw.free()


@pytest.mark.parametrize("kv8", [False, True])
@pytest.mark.parametrize("ctx", [1300, 2500, 5300])
def test_qwen3_context_ranges(ctx, kv8):
    """head_dim 128 at its default splits against the oracle, per layer and
    logit: four widened splits in the class kernel (1,300 positions), ten of
    256 in the spread kernel (merged in batches of four), 21 merged by the
    first split's workgroup; bf16 and FP8 caches."""
    shape = QWEN3_06B.with_(n_layers=2, vocab=2048)
    eng, orc, dw = make_pair(shape, 83, ctx + 16, kv_fp8=kv8)
    try:
        eng.fill_kv_synthetic(ctx, 17)
        ks = np.stack([synth.kv_prefill_bits(17, l, 0, ctx, shape.n_kv_heads, shape.head_dim) for l in range(2)])
        vs = np.stack([synth.kv_prefill_bits(17, l, 1, ctx, shape.n_kv_heads, shape.head_dim) for l in range(2)])
        orc.set_kv(ks, vs)
        assert eng.decode_kernel_for(3) == (_lib.KERNEL_CLASS if ctx == 1300 else _lib.KERNEL_SPREAD)
        tok = 11
        for i in range(3):
            nxt, layers, logits = eng.debug_forward(tok)
            ref = orc.step(tok, capture=True)
            l2, la = check_step(layers, logits, ref, f"qwen3 ctx {ctx} kv8 {kv8} step {i}")
            print(f"qwen3 ctx {ctx} kv8 {kv8} step {i}: layer relL2 {l2:.2e} logits abs {la:.2e}", flush=True)
            tok = ref["token"]
    finally:
        eng.close()
        dw.free()


@pytest.mark.parametrize("kv8", [False, True])
def test_reset_clears_every_written_row(kv8):
    """reset zeroes the cache up to the highest row written since the last
    clear, whichever path wrote it, at block edges and at the capacity; a
    change of format clears what the other format held.  With an FP8 cache what
    is read back is code x scale: that the codes are zero shows, that the
    scales are does not (no call reads them alone)."""
    shape = TINY
    dw = DeviceWeights(shape, 3)
    eng = MegakernelEngine(shape=shape, max_seq=96, device_weights=dw, prefill=True)
    try:
        eng.set_kv_fp8(kv8)

        def fill(n):
            eng.fill_kv_synthetic(n, 4)

        def decode_past(n):
            eng.set_pos(n - 3)
            eng.decode_many(1, 3)
            eng.set_pos(0)

        def prefill_past(n):
            eng.set_pos(n - 5)
            eng.prefill([1, 2, 3, 4, 5])
            eng.set_pos(2)

        def set_kv(n):
            eng.set_kv(np.full((shape.n_layers, 2, shape.n_kv_heads, n, shape.head_dim), 0x3F80, np.uint16))

        for write in (fill, decode_past, prefill_past, set_kv):
            for n in (7, 32, 33, 96):
                write(n)
                assert eng.get_kv(96)[:, :, :, n - 1].any()
                eng.reset()
                assert eng.pos == 0 and not eng.get_kv(96).any()
        fill(96)
        eng.set_kv_fp8(not kv8)
        assert not eng.get_kv(96).any()
    finally:
        eng.close()
        dw.free()


def test_reset_of_a_full_cache_keeps_the_memset_rate():
    """A reset after the whole default capacity was written takes no longer than
    a fill of the whole cache allocation (1.9 GB), give or take a fifth."""
    shape = BASELINE.with_(vocab=4096)
    dw = DeviceWeights(shape, 3)
    eng = MegakernelEngine(shape=shape, max_seq=33024, device_weights=dw)
    dw.free()
    ref = torch.empty(2 * shape.n_layers * shape.n_kv_heads * 33024 * shape.head_dim, dtype=torch.int16, device="cuda")
    try:
        def us(work):
            torch.cuda.synchronize()
            t = time.perf_counter()
            work()
            torch.cuda.synchronize()
            return (time.perf_counter() - t) * 1e6

        fills, resets = [], []
        for _ in range(8):
            eng.fill_kv_synthetic(33024, 7)
            resets.append(us(eng.reset))
            fills.append(us(ref.zero_))
        print(f"reset {min(resets):.0f} us, fill of the allocation {min(fills):.0f} us", flush=True)
        assert min(resets) < 1.2 * min(fills)
        assert not eng.get_kv(64).any()
    finally:
        eng.close()
