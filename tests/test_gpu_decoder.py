"""The batch-1 decode loop against the oracle runner (oracle/qwen3_oracle.py) on
a small Qwen3-architecture model with random LLVQ projections.

Bars: with the oracle's tokens fed to both (teacher forcing) the logits agree to
a few binary16 steps at every position.  Each bar below is at most four times the
largest error observed for that model (printed by the test as OBSERVED ...): a
real regression (a wrong rounding point, a dropped tail column, a mis-scaled
block) moves logits by 1e-2 and more.  Free-running greedy tokens are identical
up to the first position where the oracle's own top-two logits are closer than
twice that logit error plus 1e-4 (ties below 1e-4 are the only ones the
reference's own runner comparison excuses, llvq-llm/src/bin/fusedrun.rs:263-278)."""
import numpy as np
import pytest

from llvq_amd import artifact, decoder, synth

pytestmark = pytest.mark.gpu

# max |dlogit| / max |logit| against the oracle, by model (observed -> bar)
BAR_SMALL = 5e-4    # 1.2e-4: hidden 256, heads of 64
BAR_RAGGED = 2e-3   # 5.3e-4: hidden 200, heads of 32, every projection with tail columns; few logits, so a binary16 step weighs more
BAR_Q8 = 9e-4       # 1.3e-4 position by position, 2.3e-4 after a batched prompt: int8 KV cache
BAR_PARTS = 2.5e-4  # 6.3e-5, before products left parts and after: rows of 1032 and 1024, a prompt of 66 to 200


def _bar(cfg):
    return BAR_RAGGED if cfg.hidden_size == 200 else (BAR_Q8 if cfg.kv_mode == "q8" else BAR_SMALL)


def _near_tie(trace_step, bar):
    """Whether the oracle's own two largest logits at a step are closer than the logit error allows to resolve."""
    l = np.sort(trace_step)[-2:]
    return float(l[1] - l[0]) <= 2 * bar * float(np.abs(trace_step).max()) + 1e-4

SMALL = decoder.Qwen3Config(num_hidden_layers=3, hidden_size=256, num_attention_heads=4, num_key_value_heads=2,
                            head_dim=64, intermediate_size=512, vocab_size=1000, rope_theta=1e6, rms_norm_eps=1e-6,
                            max_positions=96, tie_word_embeddings=True)
# hidden 200 = 8 blocks + 8 tail columns, intermediate 328 = 13 blocks + 16 tail: every projection has a tail
RAGGED = decoder.Qwen3Config(num_hidden_layers=2, hidden_size=200, num_attention_heads=6, num_key_value_heads=2,
                             head_dim=32, intermediate_size=328, vocab_size=517, rope_theta=1e4, rms_norm_eps=1e-5,
                             max_positions=40, tie_word_embeddings=False)


Q8 = decoder.Qwen3Config(num_hidden_layers=2, hidden_size=256, num_attention_heads=10, num_key_value_heads=2,
                         head_dim=64, intermediate_size=384, vocab_size=400, rope_theta=1e6, rms_norm_eps=1e-6,
                         max_positions=80, tie_word_embeddings=True, kv_mode="q8")  # 5 query heads per kv head, as at 14B


def _build(gpu_rt, orc, cfg, seed, rotate=False, prefill_rows=0, shell_cap=12):
    from oracle import qwen3_oracle

    raws = decoder.synthetic_projections(cfg, seed, shell_cap=shell_cap)
    if rotate:
        # stored as W Q^T (format.rs:435-437): q/k/v share a basis, gate/up another, o and down have their own;
        # layer 1 keeps k and v in the natural basis, so one group call spans two bases
        for li, layer in enumerate(raws):
            for m, s in zip(layer, (11, 11, 11, 12, 13, 13, 14)):
                m.rotation_seed = 100 * li + s
            if li == 1:
                layer[1].rotation_seed = layer[2].rotation_seed = None
    weights = decoder.synthetic_weights(cfg, seed)
    dense = [[orc.read_matrix_raw(artifact.write_matrix_raw(m))[0].decode_matrix() for m in layer] for layer in raws]
    ref = qwen3_oracle.Qwen3Oracle(cfg, dense, weights, kv_mode=cfg.kv_mode)
    dec = decoder.Decoder(gpu_rt, cfg, raws, weights, prefill_rows=prefill_rows)
    return dec, ref


@pytest.mark.parametrize("cfg,seed,n", [(SMALL, 1, 24), (RAGGED, 2, 24), (Q8, 6, 70)])
def test_teacher_forced_logits(gpu_rt, orc, cfg, seed, n):
    """Q8: int8 KV cache on both sides; 70 positions also take the cache past one
    range per workgroup (more than 32 positions) in the split attention."""
    dec, ref = _build(gpu_rt, orc, cfg, seed)
    try:
        rng = np.random.default_rng(seed)
        tokens = rng.integers(0, cfg.vocab_size, size=n)
        worst = 0.0
        agree = 0
        for t in tokens:
            want = ref.forward_token(int(t))
            got, best = dec.forward_token(int(t))
            scale = float(np.abs(want).max())
            err = float(np.abs(got - want).max())
            worst = max(worst, err / scale)
            assert best == int(np.argmax(got))  # the device argmax is the argmax of the logits it returns
            top2 = np.sort(want)[-2:]
            if best == int(np.argmax(want)):
                agree += 1
            else:
                assert top2[1] - top2[0] <= 2 * err + 1e-4, "argmax differs where the oracle's top two are well separated"
        print(f"OBSERVED teacher_forced {cfg.hidden_size}/{cfg.kv_mode}: {worst:.3e}")
        assert worst < _bar(cfg), f"max |dlogit| / max|logit| = {worst:.3e}"
        assert agree >= len(tokens) - 2
        assert dec.position == len(tokens)
    finally:
        dec.close()


def test_cap13_projections_in_the_loop(gpu_rt, orc):
    """Every projection a cap-13 matrix (49-bit blocks in a dense stream, llvq-llm/src/fused.rs:1166-1180): the prompt
    through the batched path (a row loop for such matrices), then position by position, against the oracle."""
    dec, ref = _build(gpu_rt, orc, SMALL, 9, prefill_rows=16, shell_cap=13)
    try:
        tokens = np.random.default_rng(9).integers(0, SMALL.vocab_size, size=20)
        for t in tokens[:-1]:
            ref.forward_token(int(t))
        want = ref.forward_token(int(tokens[-1]))
        got, _ = dec.prefill(tokens)
        worst = float(np.abs(got - want).max() / np.abs(want).max())
        for t in np.random.default_rng(109).integers(0, SMALL.vocab_size, size=12):
            want = ref.forward_token(int(t))
            got, _ = dec.forward_token(int(t))
            worst = max(worst, float(np.abs(got - want).max() / np.abs(want).max()))
        print(f"OBSERVED cap13_loop: {worst:.3e}")
        assert worst < BAR_SMALL, f"max |dlogit| / max|logit| = {worst:.3e}"
    finally:
        dec.close()


def test_rotated_projections_in_the_loop(gpu_rt, orc):
    """Every projection stored in a rotated basis, as published artifacts are: the loop
    rotates the activation before each product (fused_cuda.rs:362-384) and must agree with
    the oracle, whose dense weights are un-rotated at decode (format.rs:435-437)."""
    dec, ref = _build(gpu_rt, orc, SMALL, 4, rotate=True)
    try:
        tokens = np.random.default_rng(4).integers(0, SMALL.vocab_size, size=20)
        worst = 0.0
        for t in tokens:
            want = ref.forward_token(int(t))
            got, _ = dec.forward_token(int(t))
            worst = max(worst, float(np.abs(got - want).max() / np.abs(want).max()))
        print(f"OBSERVED rotated_loop: {worst:.3e}")
        assert worst < BAR_SMALL, f"max |dlogit| / max|logit| = {worst:.3e}"
    finally:
        dec.close()


@pytest.mark.parametrize("cfg,seed,rotate", [(SMALL, 5, False), (RAGGED, 6, False), (Q8, 7, False), (SMALL, 8, True)])
def test_batched_prefill_then_decode(gpu_rt, orc, cfg, seed, rotate):
    """The prompt through the batched product, 16 positions a pass (three passes, the last one short),
    then position-by-position decoding over the cache it left: logits against the oracle fed the same
    tokens.  The batched product rounds weights to binary16 once, which is inside the bar the
    token-by-token path is held to."""
    dec, ref = _build(gpu_rt, orc, cfg, seed, rotate=rotate, prefill_rows=16)
    try:
        tokens = np.random.default_rng(seed).integers(0, cfg.vocab_size, size=min(38, cfg.max_positions - 7))
        for t in tokens[:-1]:
            ref.forward_token(int(t))
        want = ref.forward_token(int(tokens[-1]))
        got, best = dec.prefill(tokens)
        assert dec.position == len(tokens)
        worst = float(np.abs(got - want).max() / np.abs(want).max())
        assert best == int(np.argmax(got))
        for t in np.random.default_rng(seed + 100).integers(0, cfg.vocab_size, size=6):
            want = ref.forward_token(int(t))
            got, _ = dec.forward_token(int(t))
            worst = max(worst, float(np.abs(got - want).max() / np.abs(want).max()))
        print(f"OBSERVED batched_prefill {cfg.hidden_size}/{cfg.kv_mode}/rot={rotate}: {worst:.3e}")
        assert worst < _bar(cfg), f"max |dlogit| / max|logit| = {worst:.3e}"
    finally:
        dec.close()


def test_generate_with_batched_prefill_matches_token_by_token(gpu_rt, orc):
    dec, ref = _build(gpu_rt, orc, SMALL, 3, prefill_rows=32)
    try:
        prompt = np.random.default_rng(3).integers(0, SMALL.vocab_size, size=40)
        a = dec.generate(prompt, 24)
        b = dec.generate(prompt, 24, batched_prefill=True)
        same = a == b
        if not same.all():  # a flip needs a near-tie in the oracle's own logits at that step
            first = int(np.argmin(same))
            _, trace = ref.generate(prompt, first + 1)
            assert _near_tie(trace[first], BAR_SMALL), f"first divergence at step {first} without a near-tie"
        with pytest.raises(Exception):
            decoder.Decoder(gpu_rt, SMALL, decoder.synthetic_projections(SMALL, 3), decoder.synthetic_weights(SMALL, 3)).prefill(prompt)
    finally:
        dec.close()


@pytest.mark.parametrize("heads,kv,kv_mode", [(1, 1, "q8"), (3, 1, "f16"), (8, 1, "f16"), (10, 2, "q8")])
def test_decode_attention_at_every_length(gpu_rt, orc, heads, kv, kv_mode):
    """Heads of 128, one to eight of them to a kv head (all columns of a matrix instruction but for those are other heads' again): every
    position of the first tiles, of the second range and of its first tiles, each against the oracle."""
    import dataclasses

    cfg = dataclasses.replace(_wide(heads, kv, kv_mode), num_hidden_layers=1, vocab_size=200)
    cfg.max_positions = 163
    dec, ref = _build(gpu_rt, orc, cfg, 31)
    try:
        for n, t in enumerate(np.random.default_rng(32).integers(0, cfg.vocab_size, size=cfg.max_positions)):
            want, got = ref.forward_token(int(t)), dec.forward_token(int(t))[0]
            # Both round at the same places, and the attention differs by 1e-6 before its result is rounded: a binary16 step of single logits is 1e-3.
            assert np.abs(got - want).max() < 1e-3 * np.abs(want).max(), n
    finally:
        dec.close()


@pytest.mark.parametrize("kv_mode", ["f16", "q8"])
def test_small_attention_weights_keep_their_bits(gpu_rt, orc, kv_mode):
    """Positions with weights of 2^-37 to 2^-25 of the largest, which every sixteen positions have one of, and the only V that is not zero: the context is
    theirs alone, 7e-6 to 0.01.  Every projection is tail columns, so that embeddings, queries, keys and values are exact: rows of 16 columns with a
    single one become 4, heads are of equal magnitudes, and the frequencies of the upper 32 pairs turn nothing.  (Weights in steps of 2^-38 of the
    largest were off by up to 18 %.)"""
    from oracle import qwen3_oracle

    hidden, hd, queries = 16, 128, 6
    cfg = decoder.Qwen3Config(num_hidden_layers=1, hidden_size=hidden, num_attention_heads=1, num_key_value_heads=1, head_dim=hd, intermediate_size=24,
                              vocab_size=16, rope_theta=1e30, rms_norm_eps=1e-6, max_positions=128, tie_word_embeddings=False, kv_mode=kv_mode)
    dense = [np.zeros((do, di), np.float32) for _, do, di in cfg.shapes()]
    slow = np.arange(hd) % 64 >= 32
    dense[0][:] = 0.25
    for c in range(queries):  # query token c differs from the small keys in 4 c of 64 signs less
        dense[0][np.flatnonzero(slow)[: 2 * c], 1 + c] = -0.25
    dense[1][:] = 0.25
    dense[1][:, 0] = -0.25
    dense[2][120:, 0] = 16000.0   # V of the small positions: 64000 in the columns that o_proj has as its tail
    dense[3][15, 120:] = 1e4 / 8
    raws = []
    for m, (site, do, di) in zip(dense, cfg.shapes()):
        r = synth.make_matrix(f"model.layers.0.{site}.weight", do, di, 3)
        r.row_scales = np.full_like(r.row_scales, 1e-30)
        r.tail = np.ascontiguousarray(m[:, di - di % 24:]).ravel()
        raws.append(r)
    one = np.ones((1, hidden), np.float16)
    gains = np.where(slow, 1.0, 0.0).astype(np.float16)[None]
    embed = np.eye(16, hidden, dtype=np.float16)
    weights = decoder.DecoderWeights(one, one, gains, (2.25 * gains).astype(np.float16), one[0], embed, embed)
    ref = qwen3_oracle.Qwen3Oracle(cfg, [[orc.read_matrix_raw(artifact.write_matrix_raw(r))[0].decode_matrix() for r in raws]], weights, kv_mode=kv_mode)
    dec = decoder.Decoder(gpu_rt, cfg, [raws], weights)
    try:
        for i, t in enumerate(([1] + [0] * 15) * 6 + list(range(1, 1 + queries))):
            with np.errstate(all="ignore"):  # (the first small position's result is past binary16, and nobody's but its own)
                want = ref.forward_token(t)
            got = dec.forward_token(t)[0]
            if i < 96:
                continue
            # column 15 of the residual against the token's own, which is one: 10^4 times the context
            ratio, mine = float(want[15]) / float(want[t]), float(got[15]) / float(got[t])
            print(f"OBSERVED small_weights {kv_mode} {ratio / 1e4:.3e}: {mine / ratio - 1.0:.3e}")
            # a binary16 step of the context (2^-24 of those below 2^-14), and of o_proj's result, the residual and two logits
            assert abs(mine / ratio - 1.0) < 2.0 ** -24 / (ratio / 1e4) + 5 * 2.0 ** -11
    finally:
        dec.close()


def _attention_alone(gpu_rt, orc, heads, kv, head_dim, kv_mode, marked, seed):
    """One layer whose logits are the attention's: embeddings are rows of the unit matrix, q, k and v tail columns (a token's 4 times the column, exactly), half
    of every head's columns are ones that no position turns, the MLP is nothing and the head is the unit matrix.  marked: the positions that have a V, and what becomes of a single one of them
    shows in the logits by its share."""
    from oracle import qwen3_oracle

    cfg = decoder.Qwen3Config(num_hidden_layers=1, hidden_size=16, num_attention_heads=heads, num_key_value_heads=kv, head_dim=head_dim, intermediate_size=24,
                              vocab_size=16, rope_theta=1e30, rms_norm_eps=1e-6, max_positions=len(marked), tie_word_embeddings=False, kv_mode=kv_mode)
    rng = np.random.default_rng(seed)
    raws = []
    for i, (site, do, di) in enumerate(cfg.shapes()):
        r = synth.make_matrix(f"model.layers.0.{site}.weight", do, di, seed)
        if i < 2:
            r.tail = rng.choice(np.float32([-0.25, 0.25]), size=r.tail.size)
        elif i == 2:
            r.tail = rng.standard_normal((do, di)).astype(np.float32)
            r.tail[:, 0] = 0.0
            r.tail = r.tail.ravel()
        elif i == 3:
            r.row_scales, r.tail = r.row_scales * 64.0, r.tail * 512.0
        else:
            r.row_scales, r.tail = r.row_scales * 1e-20, r.tail * 0.0
        raws.append(r)
    one, gains = np.ones((1, 16), np.float16), np.where(np.arange(head_dim) % (head_dim // 2) >= head_dim // 4, 1.5, 0.0).astype(np.float16)[None]
    eye = np.eye(16, dtype=np.float16)
    weights = decoder.DecoderWeights(one, one, gains, gains, one[0], eye, eye)
    dense = [[orc.read_matrix_raw(artifact.write_matrix_raw(r))[0].decode_matrix() for r in raws]]
    dec = decoder.Decoder(gpu_rt, cfg, [raws], weights, prefill_rows=512)
    tokens = np.where(marked, rng.integers(1, 16, size=len(marked)), 0)
    return dec, qwen3_oracle.Qwen3Oracle(cfg, dense, weights, kv_mode=kv_mode), tokens


def _worst_of_last(dec, ref, tokens, first):
    """A batched prompt of `first` tokens, then the others one by one: the largest difference of their logits from the oracle's."""
    try:
        ref.prefill_rows(tokens[:first])
        dec.prefill(tokens[:first], want_logits=False)
        worst = 0.0
        for t in tokens[first:]:
            want, (got, _) = ref.forward_token(int(t)), dec.forward_token(int(t))
            worst = max(worst, float(np.abs(got - want).max() / np.abs(want).max()))
        return worst
    finally:
        dec.close()


@pytest.mark.parametrize("heads,kv,kv_mode,first", [(5, 1, "f16", 1018), (4, 2, "f16", 4090), (5, 1, "q8", 4090)])
def test_long_caches_of_heads_of_64(gpu_rt, orc, heads, kv, kv_mode, first):
    """Heads of another width than 128, whose decode attention is attn_decode_kernel: where its ranges go to attn_merge_kernel (past 1024 positions; 17
    ranges, and 64), and past 4096, where a range has a 65th position and its classes a second batch.  The positions that have a V are those, and
    the last twelve (without one of them the logits move by 2 % in the median)."""
    at = np.arange(first + 12)
    worst = _worst_of_last(*_attention_alone(gpu_rt, orc, heads, kv, 64, kv_mode, (at % 65 == 64) | (at >= first), 33), first)
    print(f"OBSERVED heads_of_64 {heads}/{kv}/{kv_mode}/{first}: {worst:.3e}")
    assert worst < 2e-3


@pytest.mark.parametrize("heads,kv,kv_mode,first,last", [(128, 128, "f16", 254, 290), (128, 128, "q8", 254, 290), (160, 32, "f16", 1028, 1042), (160, 32, "q8", 1028, 1042)])
def test_decode_attention_past_a_tile_for_every_wavefront(gpu_rt, orc, heads, kv, kv_mode, first, last):
    """Kv heads enough that the ranges are as many as the CUs take (two, eight) before every wavefront has a tile of sixteen positions: the first ones
    have a second tile, loaded over the first's registers, in which some heads' maxima rise, and the new position is its first row, one in its
    middle, its last (every one of them at two ranges), with the rows behind it past the range.  All positions have a V (without one the logits move by
    7e-3 in the median), or those around the beginning of a second tile and the last (6 %)."""
    at = np.arange(last)
    marked = at >= 0 if kv == 128 else (at % 129 >= 126) | (at >= first)
    worst = _worst_of_last(*_attention_alone(gpu_rt, orc, heads, kv, 128, kv_mode, marked, 33), first)
    print(f"OBSERVED second_tiles {heads}/{kv}/{kv_mode}: {worst:.3e}")
    assert worst < 2e-3


def test_long_cache_takes_the_merge_kernel(gpu_rt, orc):
    """Past 1024 cached positions the attention partials (more than 16 ranges of 64) are merged
    by a kernel of their own; the logits must keep agreeing with the oracle across the switch."""
    import dataclasses

    cfg = dataclasses.replace(Q8, num_hidden_layers=1, max_positions=1080, vocab_size=200)
    dec, ref = _build(gpu_rt, orc, cfg, 9)
    try:
        tokens = np.random.default_rng(9).integers(0, cfg.vocab_size, size=1070)
        worst = 0.0
        for i, t in enumerate(tokens):
            want = ref.forward_token(int(t))
            got, _ = dec.forward_token(int(t), want_logits=i >= 1000)
            if i >= 1000:
                worst = max(worst, float(np.abs(got - want).max() / np.abs(want).max()))
        print(f"OBSERVED long_cache_merge: {worst:.3e}")
        assert worst < BAR_Q8, f"max |dlogit| / max|logit| = {worst:.3e}"
    finally:
        dec.close()


def test_context_of_8192_positions_int8_cache(gpu_rt):
    """BASELINE config 4's regime for the attention: an int8 KV cache filled to 8192 positions, heads of
    128, 5 query heads per kv head (a small model otherwise, so that the oracle can follow).  The cache is
    filled once position by position (split-KV attention over up to 64 ranges, merged in the launch) and once
    by the batched path (matrix-core attention over up to 256 cache tiles, int8 rows rebuilt in LDS); the
    logits of the last prompt position and of six more positions are compared with the oracle's, which are
    a fixture (tests/golden/qwen3_small_q8kv_8192_logits.npz, written by make_long_context_logits.py: the
    oracle takes minutes over the 8192 positions)."""
    import os

    golden = os.path.join(os.path.dirname(os.path.abspath(__file__)), "golden")
    import importlib.util

    spec = importlib.util.spec_from_file_location("make_long_context_logits", os.path.join(golden, "make_long_context_logits.py"))
    gen = importlib.util.module_from_spec(spec)
    spec.loader.exec_module(gen)  # the model description and seeds the fixture was made with (runs nothing)
    with np.load(os.path.join(golden, "qwen3_small_q8kv_8192_logits.npz")) as f:
        want = f["logits"].astype(np.float64)
        assert (int(f["model_seed"]), int(f["prompt_seed"]), int(f["more_seed"]), int(f["n_prompt"])) == \
            (gen.MODEL_SEED, gen.PROMPT_SEED, gen.MORE_SEED, gen.N_PROMPT)
    cfg = gen.CFG
    dec = decoder.Decoder(gpu_rt, cfg, decoder.synthetic_projections(cfg, gen.MODEL_SEED), decoder.synthetic_weights(cfg, gen.MODEL_SEED),
                          prefill_rows=512)
    try:
        tokens = np.random.default_rng(gen.PROMPT_SEED).integers(0, cfg.vocab_size, size=gen.N_PROMPT)
        more = np.random.default_rng(gen.MORE_SEED).integers(0, cfg.vocab_size, size=gen.N_MORE)
        for batched in (False, True):
            dec.reset()
            if batched:
                got = [dec.prefill(tokens)[0]]
            else:
                for t in tokens[:-1]:
                    dec.forward_token(int(t), want_logits=False)
                got = [dec.forward_token(int(tokens[-1]))[0]]
            got += [dec.forward_token(int(t))[0] for t in more]
            assert dec.position == 8192
            worst = max(float(np.abs(g - w).max() / np.abs(w).max()) for g, w in zip(got, want))
            print(f"OBSERVED ctx8192 batched={batched}: {worst:.3e}")
            assert worst < 5e-4, f"batched={batched}: max |dlogit| / max|logit| = {worst:.3e}"  # observed: 1.2e-4, a binary16 ulp
    finally:
        dec.close()


def test_config4_as_stated_14b_int8_cache_8192_positions(gpu_rt):
    """BASELINE config 4 as stated, in one run: the 40-layer model at the Qwen3-14B widths (280 LLVQ
    matrices, 3.3 GB of codes resident), int8 KV cache, batch 1 at 8186+ cached positions, where the decode
    attention has as many ranges as the CUs take (32 of two tiles to every wavefront, merged in its own launch).
    The CPU oracle cannot follow at this size (hours), so
    the checks are properties the reference states for its own cache (llvq-llm/tests/kv_cache.rs:222-262:
    split prefill == whole prefill; llvq-llm/src/bin/run.rs:4-7: cached generation is repeatable):
      * the cache filled by the batched path in passes of 512 rows and in passes of 384 rows gives the same
        next-token logits to 1e-3 of the largest (different row blocks, cache tiles and partial-sum splits);
      * six greedy tokens decoded over that cache are the same both times, and again after a reset;
      * every logit is finite and the position ends at 8192.
    The model's own arithmetic at these widths is pinned against the oracle at 128 positions by the
    fixture test below, and the 8192-position attention against the oracle on a small model above."""
    import dataclasses

    cfg = dataclasses.replace(decoder.QWEN3_14B, max_positions=8192)
    assert (cfg.num_hidden_layers, cfg.hidden_size, cfg.intermediate_size, cfg.kv_mode) == (40, 5120, 17408, "q8")
    n_prompt, n_new = 8186, 6
    weights = decoder.synthetic_weights(cfg, 4)
    projs = []
    for layer in decoder.synthetic_projections(cfg, 4):
        projs.append([gpu_rt.upload(m) for m in layer])
    prompt = np.random.default_rng(4).integers(0, cfg.vocab_size, size=n_prompt)
    runs = []
    try:
        for rows in (512, 384, 512):
            dec = decoder.Decoder(gpu_rt, cfg, projs, weights, prefill_rows=rows)
            try:
                logits, best = dec.prefill(prompt)
                assert dec.position == n_prompt and np.isfinite(logits).all() and best == int(np.argmax(logits))
                toks, tok = [], best
                for _ in range(n_new):
                    step_logits, nxt = dec.forward_token(tok)
                    assert np.isfinite(step_logits).all()
                    toks.append(tok)
                    tok = nxt
                assert dec.position == n_prompt + n_new == 8192
                runs.append((logits.astype(np.float64), toks))
            finally:
                dec.close()
        (l512, t512), (l384, t384), (l512b, t512b) = runs
        diff = float(np.abs(l512 - l384).max() / np.abs(l512).max())
        print(f"OBSERVED config4 prefill 512 vs 384 rows: {diff:.3e}")
        assert diff < 1e-3, f"passes of 512 vs 384 rows: max |dlogit| / max|logit| = {diff:.3e}"
        assert np.array_equal(l512, l512b) and t512 == t512b, "the same run twice must give the same bits"
        assert t512 == t384, (t512, t384)
        assert len(set(t512)) > 1 or n_new == 1
    finally:
        for layer in projs:
            for p in layer:
                gpu_rt.free(p)


def test_greedy_tokens_match_oracle(gpu_rt, orc):
    dec, ref = _build(gpu_rt, orc, SMALL, 3)
    try:
        prompt = np.random.default_rng(3).integers(0, SMALL.vocab_size, size=12)
        want, trace = ref.generate(prompt, 40)
        got = dec.generate(prompt, 40)
        same = want == got
        if not same.all():
            first = int(np.argmin(same))
            assert _near_tie(trace[first], BAR_SMALL), f"first divergence at step {first}: oracle {want[first]}, device {got[first]}"
            assert first >= 8, "diverged almost at once"
        # generation is repeatable and independent of earlier state
        again = dec.generate(prompt, 40)
        assert np.array_equal(got, again)
    finally:
        dec.close()


def test_generate_phased_gives_the_tokens_of_generate(gpu_rt, orc):
    """Qwen3::generate_phased (model.rs:1116-1163): the phased run must yield the tokens of the plain one
    (the reference pins the same), one sample per phase and decoded token, nothing for the prompt."""
    dec, _ = _build(gpu_rt, orc, SMALL, 3)
    try:
        prompt = np.random.default_rng(3).integers(0, SMALL.vocab_size, size=12)
        plain = dec.generate(prompt, 10)
        toks, phases = dec.generate_phased(prompt, 10)
        assert np.array_equal(plain, toks)
        assert phases.shape == (10, 4) and np.isfinite(phases).all()
        assert (phases[:, 0] > 0).all() and (phases[:, 1] > 0).all()       # head, argmax: every token
        assert (phases[:-1, 2] > 0).all() and (phases[:-1, 3] > 0).all()   # embedding, layers: every token fed back
        assert phases[-1, 2] == 0 and phases[-1, 3] == 0
        assert phases[:-1, 3].min() > phases[:-1, 2].max()                  # three layers cost more than a gather
        empty, none = dec.generate_phased(prompt, 0)
        assert empty.size == 0 and none.shape == (0, 4)
    finally:
        dec.close()


def test_full_width_layers_tokens_match_oracle(gpu_rt, orc):
    """Six layers at the Qwen3-4B widths (hidden 2560, 32/8 heads of 128, intermediate 9728, vocabulary
    151 936, untied f16 head): greedy tokens of the device loop, token by token and with the prompt through
    the batched path, against the oracle runner over the same weights decoded on the CPU.  (All 36 layers,
    run by hand the same way, give 40 identical tokens; that takes two minutes and 30 GB of host memory.)"""
    import dataclasses

    from oracle import qwen3_oracle

    cfg = dataclasses.replace(decoder.QWEN3_4B, num_hidden_layers=6, max_positions=96)
    raws = decoder.synthetic_projections(cfg, 0)
    weights = decoder.synthetic_weights(cfg, 0)
    dense = [[orc.read_matrix_raw(artifact.write_matrix_raw(m))[0].decode_matrix() for m in layer] for layer in raws]
    ref = qwen3_oracle.Qwen3Oracle(cfg, dense, weights)
    dec = decoder.Decoder(gpu_rt, cfg, raws, weights, prefill_rows=16)
    try:
        prompt = np.random.default_rng(0).integers(0, cfg.vocab_size, size=24)
        want, trace = ref.generate(prompt, 24)
        for batched in (False, True):
            got = dec.generate(prompt, 24, batched_prefill=batched)
            same = want == got
            if not same.all():  # only a near-tie of the oracle's own logits may flip a token
                first = int(np.argmin(same))
                assert _near_tie(trace[first], BAR_SMALL), (batched, first)
    finally:
        dec.close()


def test_decoder_refusals_are_errors_not_faults(gpu_rt):
    """Positions past the cache, tokens outside the vocabulary, a prompt that cannot fit: a status and a
    message each time (fused_cuda.rs:365-375 convention), and the decoder stays usable afterwards."""
    from llvq_amd import LlvqError

    raws = decoder.synthetic_projections(RAGGED, 1)
    weights = decoder.synthetic_weights(RAGGED, 1)
    dec = decoder.Decoder(gpu_rt, RAGGED, raws, weights, prefill_rows=8)
    try:
        with pytest.raises(LlvqError, match="vocabulary"):
            dec.forward_token(RAGGED.vocab_size)
        with pytest.raises(LlvqError, match="max_positions"):
            dec.generate(np.arange(30), RAGGED.max_positions)  # 30 + 40 - 1 positions
        with pytest.raises(LlvqError, match="empty prompt"):
            dec.generate(np.zeros(0, np.uint32), 3)
        assert dec.generate(np.arange(5), 0).size == 0  # model.rs:1052-1054: nothing asked, nothing done
        with pytest.raises(LlvqError, match="max_positions"):
            dec.prefill(np.arange(RAGGED.max_positions + 1) % RAGGED.vocab_size)
        with pytest.raises(LlvqError, match="vocabulary"):
            dec.prefill([1, 2, RAGGED.vocab_size])
        # exactly to the end of the cache, then one more position is refused
        dec.reset()
        dec.prefill(np.arange(RAGGED.max_positions - 1) % RAGGED.vocab_size)
        dec.forward_token(0)
        assert dec.position == RAGGED.max_positions
        with pytest.raises(LlvqError, match="max_positions"):
            dec.forward_token(0)
        out = dec.generate(np.arange(6), 4)  # still usable
        assert out.shape == (4,)
    finally:
        dec.close()


def test_kv_mode_is_parsed_strictly(gpu_rt):
    """KvMode::parse (kvq.rs:38-49, test :240-249): a typo is an error, never a silent default."""
    import dataclasses

    from llvq_amd import LlvqError

    raws = decoder.synthetic_projections(RAGGED, 1)
    weights = decoder.synthetic_weights(RAGGED, 1)
    for bad in ("Q8", "int8", "q4"):
        with pytest.raises(ValueError):
            decoder.Decoder(gpu_rt, dataclasses.replace(RAGGED, kv_mode=bad), raws, weights)
    with pytest.raises(LlvqError):  # head_dim 32 is not a multiple of the group of 64 (kvq.rs:114-120)
        decoder.Decoder(gpu_rt, dataclasses.replace(RAGGED, kv_mode="q8"), raws, weights)


def test_generate_edge_cases(gpu_rt, orc):
    from llvq_amd import LlvqError

    dec, _ = _build(gpu_rt, orc, RAGGED, 4)
    try:
        assert dec.generate([1, 2, 3], 0).size == 0  # model.rs:1052-1054
        one = dec.generate([5], 1)
        assert one.size == 1 and one[0] < RAGGED.vocab_size
        with pytest.raises(LlvqError):
            dec.generate([RAGGED.vocab_size], 2)  # token outside the vocabulary
        with pytest.raises(LlvqError):
            dec.generate(list(range(30)), 20)  # 49 positions > max_positions 40
        with pytest.raises(LlvqError):
            dec.generate([], 2)
        full = dec.generate(list(range(30)), 11)  # exactly max_positions
        assert full.size == 11
    finally:
        dec.close()


def _wide(heads, kv, kv_mode="f16"):
    return decoder.Qwen3Config(num_hidden_layers=2, hidden_size=256, num_attention_heads=heads, num_key_value_heads=kv,
                               head_dim=128, intermediate_size=384, vocab_size=400, rope_theta=1e6, rms_norm_eps=1e-6,
                               max_positions=128, tie_word_embeddings=True, kv_mode=kv_mode)


@pytest.mark.parametrize("heads,kv,kv_mode,seed", [(4, 2, "f16", 11), (4, 1, "f16", 12), (10, 2, "q8", 13), (8, 1, "q8", 14),
                                                   (6, 2, "f16", 15)])
def test_prompt_attention_on_the_matrix_cores(gpu_rt, orc, heads, kv, kv_mode, seed):
    """Heads of 128 take the matrix-core attention of the batched prompt path: 2, 4, 5 and 8 query heads
    per kv head (3 runs on the instantiation for 4 with a wavefront idle), both caches.  100 positions in
    passes of 48: row blocks of 32 and 16, a last pass of 4, up to four cache tiles per block.  The last
    row's logits and six decoded positions over the cache the passes left, against the oracle and against
    the position-by-position path of the same decoder."""
    cfg = _wide(heads, kv, kv_mode)
    dec, ref = _build(gpu_rt, orc, cfg, seed, prefill_rows=48)
    try:
        tokens = np.random.default_rng(seed).integers(0, cfg.vocab_size, size=100)
        more = np.random.default_rng(seed + 100).integers(0, cfg.vocab_size, size=6)
        want = [ref.forward_token(int(t)) for t in tokens][-1:] + [ref.forward_token(int(t)) for t in more]
        one_by_one = [dec.forward_token(int(t))[0] for t in tokens][-1:] + [dec.forward_token(int(t))[0] for t in more]
        dec.reset()
        got, best = dec.prefill(tokens)
        assert dec.position == len(tokens) and best == int(np.argmax(got))
        batched = [got] + [dec.forward_token(int(t))[0] for t in more]
        for w, o, b in zip(want, one_by_one, batched):
            top = np.abs(w).max()
            # observed: 1e-4 (a binary16 ulp of a logit); a wrong score, mask or V row shows at 1e-2 and more
            assert np.abs(b - w).max() < 2e-3 * top, f"batched vs oracle {np.abs(b - w).max() / top:.3e}"
            assert np.abs(b - o).max() < 2e-3 * top, f"batched vs position by position {np.abs(b - o).max() / top:.3e}"
    finally:
        dec.close()


@pytest.mark.parametrize("heads,kv,kv_mode", [(4, 2, "f16"), (8, 2, "q8"), (10, 2, "f16"), (8, 1, "q8")])
def test_attention_where_its_split_turns(gpu_rt, orc, heads, kv, kv_mode):
    """Prompts that end a row block or a cache tile, one short of it and one past it (an odd count of tiles leaves the second
    set of wavefronts one that is masked whole), from 129 positions on by two heads and four sets of wavefronts; and decoded positions, where
    another range begins every 128: the prompt path against the position-by-position path, whose attention kernels share nothing."""
    cfg = _wide(heads, kv, kv_mode)
    cfg.max_positions = 1040
    dec, _ = _build(gpu_rt, orc, cfg, 21, prefill_rows=512)
    try:
        tokens = np.random.default_rng(22).integers(0, cfg.vocab_size, size=1026)
        one_by_one = [dec.forward_token(int(t))[0] for t in tokens]
        for n in (1, 31, 32, 33, 63, 64, 65, 96, 97, 128, 129, 511, 1023, 1024, 1025, 1026):
            dec.reset()
            got, _best = dec.prefill(tokens[:n])
            want = one_by_one[n - 1]
            assert np.abs(got - want).max() < 2e-3 * np.abs(want).max(), n  # binary16 weights, as above
    finally:
        dec.close()


@pytest.mark.parametrize("fixture_name,cfg,max_positions", [
    ("qwen3_4b_synthetic_greedy.json", decoder.QWEN3_4B, 768),
    ("qwen3_14b_q8kv_synthetic_greedy.json", decoder.QWEN3_14B, 128),
])
def test_full_size_greedy_tokens_match_the_oracle_fixture(gpu_rt, fixture_name, cfg, max_positions):
    """The full-size models.  36 layers at the Qwen3-4B widths, a 512-token prompt, 256
    greedy tokens.  BASELINE config 4's model: 40 layers at the Qwen3-14B widths (5 query heads per kv
    head, 17 408-wide down_proj rows, int8 KV cache), a 96-token prompt and 32 tokens.  The expected tokens
    are the CPU oracle runner's over the same synthetic weights (tests/golden/*.json, written by
    tests/golden/make_full_size_tokens.py; the oracle needs minutes and tens of GB for them, the device
    loop seconds).  The fixtures also hold the gap between the oracle's two largest logits at every step:
    the smallest is one binary16 ulp of a logit (2^-7), no step is a tie, so the tokens must be identical —
    position by position, and with the prompt through the batched path."""
    import dataclasses
    import json
    import os

    with open(os.path.join(os.path.dirname(os.path.abspath(__file__)), "golden", fixture_name)) as f:
        fixture = json.load(f)
    want = np.array(fixture["tokens"], np.uint32)
    assert min(fixture["top_two_gap"]) > 1e-4  # the bar below allows no exception
    cfg = dataclasses.replace(cfg, max_positions=max_positions)
    raws = decoder.synthetic_projections(cfg, fixture["prompt_seed"])
    weights = decoder.synthetic_weights(cfg, fixture["prompt_seed"])
    dec = decoder.Decoder(gpu_rt, cfg, raws, weights, prefill_rows=min(512, fixture["prompt_tokens"]))
    del raws
    try:
        prompt = np.random.default_rng(fixture["prompt_seed"]).integers(0, cfg.vocab_size, size=fixture["prompt_tokens"])
        for batched in (False, True):
            got = dec.generate(prompt, len(want), batched_prefill=batched)
            same = want == got
            assert same.all(), f"batched_prefill={batched}: first divergence at step {int(np.argmin(same))}: " \
                               f"oracle {want[int(np.argmin(same))]}, device {got[int(np.argmin(same))]}, " \
                               f"oracle gap {fixture['top_two_gap'][int(np.argmin(same))]}"
    finally:
        dec.close()


@pytest.mark.parametrize("cfg,seed,cap", [(SMALL, 1, 12), (RAGGED, 2, 12), (Q8, 6, 12), (SMALL, 3, 13)])
def test_sequences_and_separate_launches_give_the_same_bits(gpu_rt, cfg, seed, cap):
    """The three ways a position's projection groups are launched (llvq_launch_mode: single-item sequences, one
    llvq_hip_gemv_group launch per group, chains of ordered items between attention launches): the same arithmetic
    in the same order, so logits and tokens must be identical bit for bit, position after position (30 positions;
    the residual buffers alternate, the counters of the chained sequences count on).  Once with cap-13 matrices
    (the dense 49-bit blocks through the sequence kernel, with the fused prologues of the loop)."""
    from llvq_amd import _ffi

    raws = decoder.synthetic_projections(cfg, seed, shell_cap=cap)
    weights = decoder.synthetic_weights(cfg, seed)
    projs = [[gpu_rt.upload(m) for m in layer] for layer in raws]
    decs = [decoder.Decoder(gpu_rt, cfg, projs, weights, launch_mode=m)
            for m in (_ffi.LAUNCH_PER_GROUP, _ffi.LAUNCH_SINGLE, _ffi.LAUNCH_CHAINED)]
    try:
        tokens = np.random.default_rng(seed).integers(0, cfg.vocab_size, size=30)
        for t in tokens:
            outs = [d.forward_token(int(t)) for d in decs]
            for l, tok in outs[1:]:
                assert tok == outs[0][1] and np.array_equal(l, outs[0][0])
        prompt = tokens[:9]
        gens = [d.generate(prompt, 12) for d in decs]
        assert np.array_equal(gens[0], gens[1]) and np.array_equal(gens[0], gens[2])
    finally:
        for d in decs:
            d.close()
        for layer in projs:
            for p in layer:
                gpu_rt.free(p)


def test_config4_widths_and_context_against_the_oracle(gpu_rt):
    """BASELINE config 4's regime in one piece, against the oracle: the Qwen3-14B widths (hidden 5120, 40 query
    heads over 8 kv heads of 128, 17 408-wide down_proj rows — the lean-image kernel variant), int8 KV cache, 8192
    cached positions; 2 layers and a vocabulary of 2048 so that the oracle can follow (its logits are the fixture
    tests/golden/qwen3_14b_widths_q8kv_8192_logits.npz, written by make_config4_logits.py).  The device fills the
    cache position by position (split-KV attention over up to 32 ranges, merged in the launch) and by the batched path
    (512 rows a pass); the logits of the last prompt position and of six more are compared.  Bar: 1e-3 of the
    largest logit, i.e. one binary16 step: logits are binary16 values on both sides, a step of the largest one is
    between 4.9e-4 and 9.8e-4 of it, and a different summation order can move a logit across one rounding boundary
    (observed position by position: 7.2e-4 — one step of a logit in [1, 2) under a largest logit of 1.36).  Two
    steps fail."""
    import importlib.util
    import os

    golden = os.path.join(os.path.dirname(os.path.abspath(__file__)), "golden")
    spec = importlib.util.spec_from_file_location("make_config4_logits", os.path.join(golden, "make_config4_logits.py"))
    gen = importlib.util.module_from_spec(spec)
    spec.loader.exec_module(gen)  # the model description and seeds the fixture was made with (runs nothing)
    with np.load(os.path.join(golden, "qwen3_14b_widths_q8kv_8192_logits.npz")) as f:
        want = f["logits"].astype(np.float64)
        assert (int(f["model_seed"]), int(f["prompt_seed"]), int(f["more_seed"]), int(f["n_prompt"])) == \
            (gen.MODEL_SEED, gen.PROMPT_SEED, gen.MORE_SEED, gen.N_PROMPT)
    cfg = gen.CFG
    assert (cfg.hidden_size, cfg.intermediate_size, cfg.num_attention_heads, cfg.num_key_value_heads, cfg.kv_mode) == (5120, 17408, 40, 8, "q8")
    dec = decoder.Decoder(gpu_rt, cfg, decoder.synthetic_projections(cfg, gen.MODEL_SEED), decoder.synthetic_weights(cfg, gen.MODEL_SEED),
                          prefill_rows=512)
    try:
        tokens = np.random.default_rng(gen.PROMPT_SEED).integers(0, cfg.vocab_size, size=gen.N_PROMPT)
        more = np.random.default_rng(gen.MORE_SEED).integers(0, cfg.vocab_size, size=gen.N_MORE)
        for batched in (False, True):
            dec.reset()
            if batched:
                got = [dec.prefill(tokens)[0]]
            else:
                for t in tokens[:-1]:
                    dec.forward_token(int(t), want_logits=False)
                got = [dec.forward_token(int(tokens[-1]))[0]]
            got += [dec.forward_token(int(t))[0] for t in more]
            assert dec.position == 8192
            worst = max(float(np.abs(g - w).max() / np.abs(w).max()) for g, w in zip(got, want))
            print(f"OBSERVED config4 widths, 8192 positions, batched={batched}: {worst:.3e}")
            assert worst < 1e-3, f"batched={batched}: max |dlogit| / max|logit| = {worst:.3e}"
    finally:
        dec.close()


@pytest.mark.parametrize("kv_mode,head_dim", [("f16", 64), ("f16", 128), ("q8", 64), ("q8", 128)])
def test_a_decoder_recovers_from_a_non_finite_run(gpu_rt, kv_mode, head_dim):
    """A token with an infinite embedding value leaves NaN in every cache row from its position on.  After a reset the
    same decoder gives the logits of a fresh one, bit for bit: what an earlier run left at positions that are not yet
    written reaches nothing."""
    import dataclasses

    cfg = dataclasses.replace(SMALL, num_hidden_layers=2, head_dim=head_dim, kv_mode=kv_mode, tie_word_embeddings=False)
    weights = decoder.synthetic_weights(cfg, 12)
    weights.embed[7, 3] = np.inf
    tokens = [int(t) for t in np.random.default_rng(12).integers(8, cfg.vocab_size, size=70)]
    projs = [[gpu_rt.upload(m) for m in layer] for layer in decoder.synthetic_projections(cfg, 12)]
    used, fresh = decoder.Decoder(gpu_rt, cfg, projs, weights), decoder.Decoder(gpu_rt, cfg, projs, weights)
    try:
        assert np.isnan(used.forward_token(7)[0]).all()
        for t in tokens:
            used.forward_token(t, want_logits=False)
        used.reset()
        for t in tokens:
            got, want = used.forward_token(t)[0], fresh.forward_token(t)[0]
            assert np.isfinite(want).all() and np.array_equal(got, want)
    finally:
        used.close()
        fresh.close()
        for layer in projs:
            for p in layer:
                gpu_rt.free(p)


@pytest.mark.parametrize("heads,kv_mode", [(4, "f16"), (8, "q8"), (10, "f16"), (12, "q8")])
def test_a_non_finite_row_stays_out_of_earlier_blocks_of_a_prompt(gpu_rt, heads, kv_mode):
    """Prompt attention takes 32 rows at a time.  A token with an infinite embedding value at position 40 (the second
    block, whose first rows and all later ones it spoils) must leave the cache rows of positions 0 to 31 as a prompt
    without it does: the logits of a token decoded behind them are the same bit for bit."""
    import dataclasses

    cfg = dataclasses.replace(SMALL, num_hidden_layers=3, num_attention_heads=heads, head_dim=128, kv_mode=kv_mode, tie_word_embeddings=False)
    weights = decoder.synthetic_weights(cfg, 13)
    weights.embed[7, 3] = -np.inf
    dec = decoder.Decoder(gpu_rt, cfg, decoder.synthetic_projections(cfg, 13), weights, prefill_rows=90)
    try:
        prompt = np.random.default_rng(13).integers(8, cfg.vocab_size, size=90)
        got = []
        for poison in (False, True):
            p = prompt.copy()
            p[40] = 7 if poison else p[40]
            dec.reset()
            last = dec.prefill(p)[0]
            assert np.isnan(last).all() if poison else np.isfinite(last).all()
            dec.seek(32)
            got.append(dec.forward_token(11)[0])
        assert np.isfinite(got[0]).all() and np.array_equal(got[0], got[1])
    finally:
        dec.close()


@pytest.mark.parametrize("hidden,vocab,int8", [
    (64, 3000, False),      # a row of 8 lanes; fewer pairs of rows than wavefronts
    (520, 6143, False),     # one lane into a second chunk; one row short of two a wavefront
    (520, 9300, False),     # a second turn, of one row for some wavefronts
    (1024, 6144, True),     # int8: exactly one chunk, exactly two rows a wavefront
    (1040, 12290, True),    # one lane into a second chunk; a third turn of two rows
])
def test_head_rows_and_chunks(gpu_rt, hidden, vocab, int8):
    """The head at the edges of its rows and chunks against a product in 64 bits.  Its first rows are the unit vectors, so
    the logits carry its input; every other logit then lies within the f32 sum's rounding (n + 3 roundings of at most
    2^-24 of the sum of magnitudes, int8 weights add two) and one binary16 rounding."""
    import dataclasses

    cfg = dataclasses.replace(SMALL, num_hidden_layers=1, hidden_size=hidden, vocab_size=vocab, tie_word_embeddings=False)
    weights = decoder.synthetic_weights(cfg, 31)
    head = weights.lm_head
    head[:hidden] = np.eye(hidden, dtype=np.float16)
    mags = np.abs(head.astype(np.float64))
    if int8:
        rng = np.random.default_rng(31)
        n_groups = (hidden + 63) // 64
        q = rng.integers(0, 256, size=(vocab, hidden), dtype=np.uint8)
        s = (1e-3 * (1 + rng.random((vocab, n_groups)))).astype(np.float16)
        b = (-0.1 * rng.random((vocab, n_groups))).astype(np.float16)
        q[:hidden], s[:hidden], b[:hidden] = np.eye(hidden, dtype=np.uint8), 1, 0
        weights.lm_head = artifact.RawTensor("lm_head.weight", [vocab, hidden], bits=8, group=64, packed=q.reshape(-1),
                                             scales=s.reshape(-1).view(np.uint16), biases=b.reshape(-1).view(np.uint16))
        g = np.arange(hidden) // 64
        head = q * s.astype(np.float64)[:, g] + b.astype(np.float64)[:, g]
        mags = q * s.astype(np.float64)[:, g] - b.astype(np.float64)[:, g]
    dec = decoder.Decoder(gpu_rt, cfg, decoder.synthetic_projections(cfg, 31), weights)
    try:
        for t in (5, 2999):
            got, best = dec.forward_token(t)
            h = got[:hidden].astype(np.float64)
            terms = mags @ np.abs(h)
            want = head.astype(np.float64) @ h
            bound = (hidden + 5) * 2.0 ** -24 * terms + 2.0 ** -11 * np.abs(want) * 1.001 + 2.0 ** -24
            assert np.any(h) and np.all(np.abs(got - want) <= bound)
            assert best == int(np.argmax(got))
    finally:
        dec.close()


# a team of 1, 2, 3 (odd: teams are made even), 5, 7 and 11 wavefronts (one team: rounds are), rows past the last tile, one and two pairs of
# tiles to a workgroup, several batches of rounds
@pytest.mark.parametrize("hidden,inter", [(200, 24), (1032, 4400), (1632, 40), (1632, 4400), (2408, 328), (3600, 328), (5208, 4104), (8192, 72), (200, 24000)])
def test_gate_and_up_as_one_result(gpu_rt, hidden, inter):
    """silu(gate) up formed where gate and up are finished, against the two results taken apart again by down_proj's launch (as sequences of
    one item do): the same bits."""
    from llvq_amd import _ffi

    cfg = decoder.Qwen3Config(num_hidden_layers=1, hidden_size=hidden, num_attention_heads=2, num_key_value_heads=1, head_dim=64, intermediate_size=inter,
                              vocab_size=96, rope_theta=1e6, rms_norm_eps=1e-6, max_positions=8, tie_word_embeddings=True)
    raws = decoder.synthetic_projections(cfg, hidden + inter)
    weights = decoder.synthetic_weights(cfg, 3)
    projs = [[gpu_rt.upload(m) for m in layer] for layer in raws]
    decs = [decoder.Decoder(gpu_rt, cfg, projs, weights, launch_mode=m) for m in (_ffi.LAUNCH_PER_GROUP, _ffi.LAUNCH_SINGLE)]
    try:
        for t in (5, 95, 0):
            (a, ta), (b, tb) = (d.forward_token(t) for d in decs)
            assert ta == tb and np.isfinite(a).all() and np.array_equal(a, b)
    finally:
        for d in decs:
            d.close()
        for p in projs[0]:
            gpu_rt.free(p)


@pytest.mark.parametrize("kv_mode", ["f16", "q8"])
def test_prompt_rows_straight_to_octets(gpu_rt, orc, kv_mode):
    """A pass's rows go to the products' octets where they are made (norm, attention, silu).  Widths with tail columns, of which two have more
    octets than whole units do (208 = 8 blocks + 16, 112 = 4 blocks + 16) and one fewer (256 = 10 blocks + 16); rows around the
    paddings of 16, 64, 128 and 256; what a pass of other rows left in the octets reaches nothing."""
    cfg = decoder.Qwen3Config(num_hidden_layers=2, hidden_size=208, num_attention_heads=2, num_key_value_heads=1, head_dim=128, intermediate_size=112,
                              vocab_size=300, rope_theta=1e6, rms_norm_eps=1e-6, max_positions=160, tie_word_embeddings=True, kv_mode=kv_mode)
    dec, ref = _build(gpu_rt, orc, cfg, 21, prefill_rows=256)
    try:
        tokens = np.random.default_rng(21).integers(0, cfg.vocab_size, size=140)
        want = [ref.forward_token(int(t)) for t in tokens]
        for rows in (130, 1, 2, 16, 17, 64, 65, 128, 129, 33):
            dec.reset()
            got, best = dec.prefill(tokens[:rows])
            after, _ = dec.forward_token(int(tokens[rows]))
            assert best == int(np.argmax(got))
            for g, w in ((got, want[rows - 1]), (after, want[rows])):
                assert np.abs(g - w).max() < 2e-3 * np.abs(w).max(), (rows, np.abs(g - w).max() / np.abs(w).max())
    finally:
        dec.close()


# fewer logits than a 16-byte store has and than a wavefront has lanes, a workgroup's 4096 and one more or less, several with a remainder
@pytest.mark.parametrize("vocab", [2, 63, 4095, 4096, 4097, 8195, 20001])
def test_results_where_the_last_launch_leaves_them(gpu_rt, orc, vocab):
    """Logits of every vocabulary size come whole, with the token or without it, a prompt's as well as a step's, and are those of their own step."""
    cfg = decoder.Qwen3Config(num_hidden_layers=1, hidden_size=64, num_attention_heads=2, num_key_value_heads=1, head_dim=64, intermediate_size=48,
                              vocab_size=vocab, rope_theta=1e6, rms_norm_eps=1e-6, max_positions=16, tie_word_embeddings=True)
    dec, ref = _build(gpu_rt, orc, cfg, 31, prefill_rows=8)
    try:
        tokens = np.random.default_rng(vocab).integers(0, vocab, size=5)
        want = [ref.forward_token(int(t)) for t in tokens]
        first = []
        for t, w in zip(tokens, want):
            got, best = dec.forward_token(int(t))
            first.append(best)
            assert got.shape == (vocab,) and best == int(np.argmax(got))
            assert np.abs(got - w).max() < 2e-3 * np.abs(w).max()
        dec.reset()
        for t, best in zip(tokens, first):
            got, again = dec.forward_token(int(t), want_logits=False)
            assert got is None and again == best
        dec.reset()
        got, best = dec.prefill(tokens)
        assert best == int(np.argmax(got)) and np.abs(got - want[-1]).max() < 2e-3 * np.abs(want[-1]).max()
    finally:
        dec.close()


# Two passes of the launch's quads over the row where it has as many wavefronts as its tiles ask for, one with sixteen (2560: 5 wavefronts to 128
# blocks, 1200: 3 to 64, 5208: 9 to 224), and two whatever it has (8192: 352 blocks)
@pytest.mark.parametrize("hidden,n", [(1200, 60), (2560, 60), (5208, 30), (8192, 60)])
def test_a_norm_does_not_depend_on_what_shares_its_launch(gpu_rt, hidden, n):
    """The f32 sum of a row's squares is formed in one order, however many wavefronts a launch has: the last bit of the norm, and with it binary16
    values of the normed row, would differ between the launch modes for about one row in eight."""
    from llvq_amd import _ffi

    cfg = decoder.Qwen3Config(num_hidden_layers=2, hidden_size=hidden, num_attention_heads=2, num_key_value_heads=1, head_dim=64, intermediate_size=72,
                              vocab_size=96, rope_theta=1e6, rms_norm_eps=1e-6, max_positions=64, tie_word_embeddings=True)
    weights = decoder.synthetic_weights(cfg, hidden)
    projs = [[gpu_rt.upload(m) for m in layer] for layer in decoder.synthetic_projections(cfg, hidden)]
    decs = [decoder.Decoder(gpu_rt, cfg, projs, weights, launch_mode=m) for m in (_ffi.LAUNCH_PER_GROUP, _ffi.LAUNCH_SINGLE, _ffi.LAUNCH_CHAINED)]
    try:
        apart = []
        for i, t in enumerate(np.random.default_rng(hidden).permutation(cfg.vocab_size)[:n]):
            first, *others = [d.forward_token(int(t))[0] for d in decs]
            assert np.isfinite(first).all()
            apart += [i for o in others if not np.array_equal(first, o)]
            for d in decs:  # (each token by itself)
                d.reset()
        assert not apart, f"{len(apart)} of {2 * n} logits differ, first at token {apart[0]}"
    finally:
        for d in decs:
            d.close()
        for layer in projs:
            for p in layer:
                gpu_rt.free(p)


# gate and up rotated, one of them, or of rows without a block; down in the natural basis, narrow and past 512 blocks (the wide form), with tail columns
@pytest.mark.parametrize("hidden,inter,rotated", [(256, 328, (4, 5)), (256, 12328, (4, 5)), (256, 328, (5,)), (256, 12328, (4,)), (16, 328, ()), (16, 12328, ()),
                                                  (8, 72, ())])
def test_silu_formed_by_down_projections_launch(gpu_rt, orc, hidden, inter, rotated):
    """Where gate and up are not one launch, down_proj's forms silu(gate) up from the two results."""
    from oracle import qwen3_oracle

    cfg = decoder.Qwen3Config(num_hidden_layers=2, hidden_size=hidden, num_attention_heads=4, num_key_value_heads=2, head_dim=32, intermediate_size=inter,
                              vocab_size=100, rope_theta=1e6, rms_norm_eps=1e-6, max_positions=16, tie_word_embeddings=True)
    raws = decoder.synthetic_projections(cfg, inter)
    for li, layer in enumerate(raws):
        for i in rotated:
            layer[i].rotation_seed = 100 * li + 7
    weights = decoder.synthetic_weights(cfg, inter)
    dense = [[orc.read_matrix_raw(artifact.write_matrix_raw(m))[0].decode_matrix() for m in layer] for layer in raws]
    ref, dec = qwen3_oracle.Qwen3Oracle(cfg, dense, weights), decoder.Decoder(gpu_rt, cfg, raws, weights)
    try:
        worst = 0.0
        for t in np.random.default_rng(hidden).integers(0, cfg.vocab_size, size=8):
            want = ref.forward_token(int(t))
            got, best = dec.forward_token(int(t))
            assert best == int(np.argmax(got))
            worst = max(worst, float(np.abs(got - want).max() / np.abs(want).max()))
        print(f"OBSERVED silu_by_down {hidden}/{inter}/{rotated}: {worst:.3e}")
        assert worst < BAR_SMALL  # (1.3e-4 observed)
    finally:
        dec.close()


# Gate, up and down in rotated bases: silu(gate) up in their launch (groups of 1 x 256, 5 x 64, 1 x 1024; more pairs of tiles than a workgroup has
# teams), down's activation by rotate_split_kernel (groups of 512, 1024, 2048 and 4096, the most groups and tiles of sizes that are products) and in its
# own launch: fewer columns than that pays for, and 8192 as one group.
@pytest.mark.parametrize("hidden,inter", [(256, 8704), (320, 9216), (256, 10240), (1024, 12288), (256, 20480), (256, 23552), (256, 14848), (320, 4096), (256, 8192)])
def test_rotated_gate_up_and_wide_down(gpu_rt, orc, hidden, inter):
    from oracle import qwen3_oracle

    cfg = decoder.Qwen3Config(num_hidden_layers=2, hidden_size=hidden, num_attention_heads=4, num_key_value_heads=2, head_dim=32, intermediate_size=inter,
                              vocab_size=100, rope_theta=1e6, rms_norm_eps=1e-6, max_positions=16, tie_word_embeddings=True)
    raws = decoder.synthetic_projections(cfg, inter)
    for li, layer in enumerate(raws):
        for i, seed in ((4, 7), (5, 7), (6, 9)):
            layer[i].rotation_seed = 100 * li + seed
    weights = decoder.synthetic_weights(cfg, inter)
    dense = [[orc.read_matrix_raw(artifact.write_matrix_raw(m))[0].decode_matrix() for m in layer] for layer in raws]
    ref, dec = qwen3_oracle.Qwen3Oracle(cfg, dense, weights), decoder.Decoder(gpu_rt, cfg, raws, weights)
    try:
        worst = 0.0
        for t in np.random.default_rng(hidden + inter).integers(0, cfg.vocab_size, size=6):
            want = ref.forward_token(int(t))
            got, best = dec.forward_token(int(t))
            assert best == int(np.argmax(got))
            worst = max(worst, float(np.abs(got - want).max() / np.abs(want).max()))
        print(f"OBSERVED rotated_wide_down {hidden}/{inter}: {worst:.3e}")
        assert worst < BAR_SMALL
    finally:
        dec.close()


# Rows long enough that a prompt's products are split over their columns: 43 and 42 blocks and 16 tail columns, 64 blocks and 8
PARTS = decoder.Qwen3Config(num_hidden_layers=2, hidden_size=1032, num_attention_heads=8, num_key_value_heads=2, head_dim=128, intermediate_size=1544,
                            vocab_size=600, rope_theta=1e6, rms_norm_eps=1e-6, max_positions=210, tie_word_embeddings=True)


@pytest.mark.parametrize("hidden,inter,kv_mode,rotate", [(1032, 1544, "f16", False), (1032, 1544, "q8", False), (1024, 1536, "f16", True)])
@pytest.mark.parametrize("n", [66, 129, 200])
def test_prompt_results_left_in_parts(gpu_rt, orc, hidden, inter, kv_mode, rotate, n):
    """What products of a prompt leave in parts is added up by the launches behind them (norms; heads' norms and rotations, cache rows): one
    pass, and two, of which the last's rows have the head behind them."""
    import dataclasses

    cfg = dataclasses.replace(PARTS, hidden_size=hidden, intermediate_size=inter, kv_mode=kv_mode)
    dec, ref = _build(gpu_rt, orc, cfg, 31, rotate=rotate, prefill_rows=130)
    try:
        tokens = np.random.default_rng(n).integers(0, cfg.vocab_size, size=n)
        for t in tokens[:-1]:
            ref.forward_token(int(t))
        want = ref.forward_token(int(tokens[-1]))
        got, _ = dec.prefill(tokens)
        worst = float(np.abs(got - want).max() / np.abs(want).max())
        for t in (3, 77):  # over the rows that the pass left in the cache
            want = ref.forward_token(t)
            got, _ = dec.forward_token(t)
            worst = max(worst, float(np.abs(got - want).max() / np.abs(want).max()))
        print(f"OBSERVED parts {hidden}/{kv_mode}/{rotate}/{n}: {worst:.3e}")
        assert worst < BAR_PARTS, f"max |dlogit| / max|logit| = {worst:.3e}"
    finally:
        dec.close()


@pytest.mark.parametrize("heads,kv,kv_mode", [(128, 32, "f16"), (160, 32, "q8"), (192, 24, "f16")])
def test_prompt_attention_of_many_heads(gpu_rt, heads, kv, kv_mode):
    """Kv heads and rows enough for every CU: a workgroup takes all query heads of a kv head (four, five, eight), where the small models above
    take them by two.  Against the same tokens position by position."""
    cfg = decoder.Qwen3Config(num_hidden_layers=1, hidden_size=48, num_attention_heads=heads, num_key_value_heads=kv, head_dim=128, intermediate_size=48,
                              vocab_size=300, rope_theta=1e6, rms_norm_eps=1e-6, max_positions=180, tie_word_embeddings=True, kv_mode=kv_mode)
    dec = decoder.Decoder(gpu_rt, cfg, decoder.synthetic_projections(cfg, 41), decoder.synthetic_weights(cfg, 41), prefill_rows=170)
    try:
        tokens = np.random.default_rng(41).integers(0, cfg.vocab_size, size=165)  # six blocks of 32 rows
        want = [dec.forward_token(int(t))[0] for t in tokens][-1]
        dec.reset()
        got, _ = dec.prefill(tokens)
        worst = float(np.abs(got - want).max() / np.abs(want).max())
        print(f"OBSERVED many_heads {heads}/{kv_mode}: {worst:.3e}")
        assert worst < 7e-4  # observed 1.6e-4
    finally:
        dec.close()
