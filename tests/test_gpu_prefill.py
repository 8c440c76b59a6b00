"""Long steps: the prefill matmul tiles and the attention of whole prefill chunks."""
import threading

import numpy as np
import pytest

import jetsonfabric_amd as jf

pytestmark = pytest.mark.gpu

TYPES = [jf.Q4_K, jf.Q6_K, jf.Q2_K, jf.Q8_0]


# Gate/up matrices of 12288 rows (192 sets of 64 rows) and 16896 rows (264): 256 rows make 384 work-groups of 128
# tokens and 1056 of 64, the two large tile shapes. 2304 columns are nine K tiles: a chain of two and seven of one.
@pytest.mark.parametrize("n_ff", [6144, 8448])
@pytest.mark.parametrize("t", TYPES, ids=[jf.TYPE_NAMES[t] for t in TYPES])
def test_long_step_matmul_equals_single_rows(t, n_ff):
    """Rows of a long step (whole and ragged token groups) equal the same rows computed alone, bit for bit."""
    cfg = jf.ModelConfig(n_layer=1, n_embd=2304, n_ff=n_ff, n_head=18, n_head_kv=2, n_vocab=256, n_ctx=256)
    model = jf.Model.synthesize(cfg, type_linear=t, type_embd=t, type_output=t, seed=n_ff + t)
    engine = jf.NativeEngine(model)
    try:
        for name in ("blk.0.ffn_up.weight", "blk.0.ffn_down.weight", "blk.0.attn_k.weight"):
            cols, rows = model.tensor(name)["shape"]
            for n_tok in (47, 241, 256):
                x = np.random.default_rng(n_tok).standard_normal((n_tok, cols)).astype(np.float32)
                wide = engine.matmul(name, x, rows)
                for r in sorted({0, 15, 16, n_tok // 2, n_tok - 2, n_tok - 1}):
                    single = engine.matmul(name, x[r:r + 1], rows)
                    assert np.array_equal(wide[r].view(np.uint32), single[0].view(np.uint32)), f"{name} {n_tok}: row {r}"
    finally:
        engine.close()


# Head dims 64 and 128, an odd query group, a few rows beyond one step, and a prompt of two chunks.
@pytest.mark.parametrize("n_head,n_head_kv,head_dim", [(8, 2, 64), (7, 1, 128), (16, 16, 128)])
@pytest.mark.parametrize("n", [257, 300, 2200])
def test_chunk_attention_matches_short_steps(n_head, n_head_kv, head_dim, n):
    """A prompt run in whole chunks reaches the logits of the same tokens run in steps of 16 rows (split-key
    attention). Float weights: only the attention differs. Its operands are f16 hi + lo pairs (2^-21 of a value),
    scores reach about 10, and two layers add up: 1e-4 of the largest logit is several times that."""
    cfg = jf.ModelConfig(n_layer=2, n_embd=n_head * head_dim, n_ff=256, n_head=n_head, n_head_kv=n_head_kv,
                         n_vocab=512, n_ctx=4096)
    model = jf.Model.synthesize(cfg, type_linear=jf.F32, type_embd=jf.F32, type_output=jf.F32, seed=head_dim + n_head)
    engine = jf.NativeEngine(model)
    try:
        tokens = [int(t) for t in np.random.default_rng(n).integers(0, cfg.n_vocab, n)]
        s = engine.create_session(n + 16)
        _, logits = s.prefill_greedy(tokens, logits=True)
        ref = engine.create_session(n + 16)
        ref.prefill_greedy(tokens[:8])
        at = 8
        while at < n:
            step = tokens[at:at + 16]
            rows = engine.step_batch([ref], [step], logits=True)[2][0]
            at += len(step)
        assert s.position() == ref.position() == n
        assert np.abs(logits - rows[-1]).max() <= 1e-4 * np.abs(rows[-1]).max()
        # the cache it leaves serves the next step
        a = engine.step_batch([s], [[3, 5]], logits=True)[2][0]
        b = engine.step_batch([ref], [[3, 5]], logits=True)[2][0]
        assert np.abs(a - b).max() <= 1e-4 * np.abs(b).max()
    finally:
        engine.close()


def test_step_row_limits_stay():
    """Chunks are longer than a step may be: steps of more than 256 rows are still refused."""
    cfg = jf.ModelConfig(n_layer=1, n_embd=512, n_ff=512, n_head=8, n_head_kv=2, n_vocab=512, n_ctx=1024)
    engine = jf.NativeEngine(jf.Model.synthesize(cfg, type_linear=jf.Q4_K, type_embd=jf.Q4_K, type_output=jf.Q4_K, seed=1))
    try:
        s = engine.create_session(800)
        s.prefill_greedy([1, 2, 3])
        with pytest.raises(jf.JfhError, match="too many token rows"):
            engine.step_batch([s], [[1] * 257])
        assert s.position() == 3
        engine.step_batch([s], [[1] * 256])
        assert s.position() == 259
    finally:
        engine.close()


def test_reused_cache_buffers_start_clean():
    """Sessions opened after others were closed (their buffers are kept, more of them than the engine keeps) give the
    logits of a fresh engine, also with another capacity; a session may be closed after its engine."""
    cfg = jf.ModelConfig(n_layer=2, n_embd=512, n_ff=512, n_head=8, n_head_kv=2, n_vocab=512, n_ctx=2048)
    model = jf.Model.synthesize(cfg, type_linear=jf.Q4_K, type_embd=jf.Q4_K, type_output=jf.Q4_K, seed=9)
    fresh, used = jf.NativeEngine(model), jf.NativeEngine(model)
    tokens = [int(t) for t in np.random.default_rng(2).integers(0, cfg.n_vocab, 40)]
    many = [used.create_session(c) for c in (64, 64, 100, 1500, 1500, 700, 64, 64, 64, 300, 2000, 64)]
    for s in many:
        s.prefill_greedy(tokens[::-1])
    for s in many:
        s.close()
    for capacity in (64, 60, 1500, 2000, 90):
        a, b = fresh.create_session(capacity), used.create_session(capacity)
        la, lb = a.prefill_greedy(tokens, logits=True)[1], b.prefill_greedy(tokens, logits=True)[1]
        assert np.array_equal(la.view(np.uint32), lb.view(np.uint32)), capacity
        a.close()
        b.close()
    late = used.create_session(64)
    used.close()
    late.close()
    fresh.close()


# 8 heads x 64 and 5 x 128; 385 and 769 rows leave a last chunk of one row when cut, 2200 is cut in any case.
@pytest.mark.parametrize("n_head,n_head_kv,head_dim", [(8, 2, 64), (10, 2, 128)])
@pytest.mark.parametrize("n", [385, 769, 1000, 2200])
def test_prompt_cut_for_other_sessions_is_the_same(n_head, n_head_kv, head_dim, n):
    """A prompt run in short chunks because another session steps gives the logits and the cache of the same prompt run
    alone, bit for bit, also while that session goes on stepping on another thread; so do its steps."""
    cfg = jf.ModelConfig(n_layer=2, n_embd=n_head * head_dim, n_ff=768, n_head=n_head, n_head_kv=n_head_kv, n_vocab=512,
                         n_ctx=4096)
    engine = jf.NativeEngine(jf.Model.synthesize(cfg, type_linear=jf.Q4_K, type_embd=jf.Q4_K, type_output=jf.Q6_K, seed=n))
    try:
        tokens = [int(t) for t in np.random.default_rng(n).integers(0, cfg.n_vocab, n)]

        def prefill():
            s = engine.create_session(n + 8)
            logits = s.prefill_greedy(tokens, logits=True)[1]
            k, v = s.read_kv(1, n)
            s.close()
            return logits.view(np.uint32), np.asarray(k), np.asarray(v)

        def greedy(s, count, stop=lambda: False):
            ids = [s.prefill_greedy(tokens[:30])]
            while len(ids) < count and not stop():
                ids.append(s.decode_greedy(ids[-1]))
            return ids

        alone = prefill()
        s = engine.create_session(4000)
        expected = []
        decoder = threading.Thread(target=lambda: expected.extend(greedy(s, 60)))
        decoder.start()
        decoder.join()
        assert all(np.array_equal(a, b) for a, b in zip(alone, prefill()))  # it has just stepped
        s.close()

        s, started, done, got = engine.create_session(4000), threading.Event(), threading.Event(), []

        def stop():  # asked before every step
            started.set()
            return done.is_set()

        decoder = threading.Thread(target=lambda: got.extend(greedy(s, 3900, stop)))
        decoder.start()
        try:
            assert started.wait(60)
            for _ in range(3):
                assert all(np.array_equal(a, b) for a, b in zip(alone, prefill()))
        finally:
            done.set()
            decoder.join()
        assert len(got) > 4 and got[:60] == expected[:len(got)]
        s.close()
    finally:
        engine.close()


# The two-row-group form of the chunk attention (grids of 512 work-groups of 128 query rows or more): a ragged chunk of
# 1900 rows and, after a chunk of 1152, one of 1000. Head dims 128 and 64, one head per kv head.
@pytest.mark.parametrize("n_head,n_head_kv,head_dim,n", [(40, 8, 128, 1900), (40, 8, 64, 1900), (64, 16, 64, 2152), (36, 36, 64, 1900)])
def test_wide_chunk_attention_matches_short_steps(n_head, n_head_kv, head_dim, n):
    """As test_chunk_attention_matches_short_steps (and its bound), and every position's cache rows."""
    cfg = jf.ModelConfig(n_layer=2, n_embd=n_head * head_dim, n_ff=256, n_head=n_head, n_head_kv=n_head_kv, n_vocab=256,
                         n_ctx=4096)
    engine = jf.NativeEngine(jf.Model.synthesize(cfg, type_linear=jf.F32, type_embd=jf.F32, type_output=jf.F32, seed=n_head))
    try:
        tokens = [int(t) for t in np.random.default_rng(n).integers(0, cfg.n_vocab, n)]
        s, ref = engine.create_session(n), engine.create_session(n)
        logits = s.prefill_greedy(tokens, logits=True)[1]
        ref.prefill_greedy(tokens[:16])
        for at in range(16, n, 16):
            rows = engine.step_batch([ref], [tokens[at:at + 16]], logits=True)[2][0]
        assert np.abs(logits - rows[-1]).max() <= 1e-4 * np.abs(rows[-1]).max()
        # the second layer's keys and values follow from every row's attention: f16, so one unit in the last place more
        for got, want in zip(s.read_kv(1, n), ref.read_kv(1, n)):
            got, want = (np.asarray(a).view(np.float16).astype(np.float32) for a in (got, want))
            assert np.abs(got - want).max() <= (1e-4 + 2.0 ** -10) * np.abs(want).max()
    finally:
        engine.close()


@pytest.mark.parametrize("n_head,n_head_kv,head_dim,n", [(40, 8, 128, 230), (64, 8, 64, 128)])
def test_captured_chunk_attention_replays(n_head, n_head_kv, head_dim, n):
    """Prompts of one captured step that run without key splits: captured, then replayed with other work between, each
    equal to the first bit for bit and to 16-row steps (bound as above)."""
    cfg = jf.ModelConfig(n_layer=2, n_embd=n_head * head_dim, n_ff=256, n_head=n_head, n_head_kv=n_head_kv, n_vocab=256,
                         n_ctx=4096)
    engine = jf.NativeEngine(jf.Model.synthesize(cfg, type_linear=jf.F32, type_embd=jf.F32, type_output=jf.F32, seed=3))
    try:
        tokens = [int(t) for t in np.random.default_rng(n).integers(0, cfg.n_vocab, n)]
        ref = engine.create_session(n)
        ref.prefill_greedy(tokens[:16])
        for at in range(16, n, 16):
            rows = engine.step_batch([ref], [tokens[at:at + 16]], logits=True)[2][0]
        runs = []
        for _ in range(4):
            s = engine.create_session(n + 4)
            runs.append(s.prefill_greedy(tokens, logits=True)[1])
            s.decode_greedy(1)
            engine.matmul("blk.0.ffn_up.weight", np.ones((1, cfg.n_embd), np.float32), cfg.n_ff)
            s.close()
        assert np.abs(runs[0] - rows[-1]).max() <= 1e-4 * np.abs(rows[-1]).max()
        assert all(np.array_equal(runs[0].view(np.uint32), r.view(np.uint32)) for r in runs)
    finally:
        engine.close()


# 4096 q|k|v rows x 3072 at 700 rows take the 128-token tiles, their down projection the 64-token ones, 300 rows and the
# 1280-wide model the 32-token ones.
@pytest.mark.parametrize("n_head,n_head_kv,head_dim,n_ff", [(24, 4, 128, 2048), (20, 4, 64, 1536)], ids=["128", "64"])
@pytest.mark.parametrize("t", TYPES, ids=[jf.TYPE_NAMES[t] for t in TYPES])
def test_long_step_epilogues_equal_short_steps(t, n_head, n_head_kv, head_dim, n_ff):
    """Rotated queries and keys, biases, transposed values, SwiGLU and residual adds of long steps: the caches of both
    layers equal those of the same tokens in 8-row steps bit for bit. The first layer's attention output matrix is zero,
    so that the second layer's rows do not depend on the attention's order of keys."""
    cfg = jf.ModelConfig(n_layer=2, n_embd=n_head * head_dim, n_ff=n_ff, n_head=n_head, n_head_kv=n_head_kv, n_vocab=256,
                         n_ctx=1024)
    source = jf.Model.synthesize(cfg, type_linear=t, type_embd=jf.Q8_0, type_output=jf.Q8_0, seed=11)

    def tensors():
        for name in source.tensor_names():
            info, data = source.tensor(name), source.tensor_bytes(name)
            if name.endswith(".bias"):
                data = np.random.default_rng(len(data)).standard_normal(len(data) // 4).astype(np.float32).tobytes()
            yield name, info["type"], info["shape"], bytes(len(data)) if name == "blk.0.attn_output.weight" else data

    engine = jf.NativeEngine(jf.Model.build(cfg, tensors()))
    try:
        for n in (300, 700):
            tokens = [int(v) for v in np.random.default_rng(n).integers(0, cfg.n_vocab, n)]
            s, ref = engine.create_session(n), engine.create_session(n)
            s.prefill_greedy(tokens)
            ref.prefill_greedy(tokens[:8])
            for at in range(8, n, 8):
                engine.step_batch([ref], [tokens[at:at + 8]])
            for layer in (0, 1):
                for what, got, want in zip("kv", s.read_kv(layer, n), ref.read_kv(layer, n)):
                    assert np.array_equal(np.asarray(got), np.asarray(want)), f"{n} rows, layer {layer}: {what}"
            s.close()
            ref.close()
    finally:
        engine.close()
