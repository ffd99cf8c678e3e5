"""Model-level parity through the C ABI: the token loop on the GPU against the oracle
(the reference --stage v2 path restated; bit-identical to the compiled reference).

Bar: identical greedy token streams; logits, per-layer activations and KV cache within
normwise relative error 1e-3 (max|gpu - oracle| / max|oracle|).
"""
import numpy as np
import pytest

from conftest import rel_err
from gpu_util import REGRESS, model_parity

pytestmark = pytest.mark.gpu

SMALL = ["tiny_f32", "tiny_q8", "tiny_mixq4", "tiny_qwen", "tiny_hd128", "small_q8"]
GRAPH, STEP = 0, 1  # HipModel.PATH_GRAPH, PATH_STEP


@pytest.mark.parametrize("path", [GRAPH, STEP], ids=["graph", "step"])
@pytest.mark.parametrize("layout", [0, 1])
@pytest.mark.parametrize("preset", SMALL)
def test_small_models(pkg, gguf, preset, layout, path):
    info = pkg.synth_preset_info(preset)
    prompt = pkg.synth_prompt(info["seed"], 6, info["n_vocab"])
    ids, worst, worst_tap, margin = model_parity(pkg, gguf(preset), prompt, 16, 64, layout, decode_path=path)
    print(f"{preset} layout {layout} path {path}: ids {ids} logits {worst:.2e} taps {worst_tap:.2e} "
          f"margin {margin:.3e}")


@pytest.mark.parametrize("preset,want", [("tiny_q8", STEP), ("tiny_f32", STEP), ("small_q8", STEP),
                                         ("tiny_mixq4", STEP), ("tiny_hd128", STEP)])
def test_decode_path_selection(pkg, gguf, preset, want):
    """The persistent step kernel runs models whose layer matrices share a compiled format
    (Q4_0 layers may have Q4_1 wo / ffn_down, as tiny_mixq4's first and last layer do),
    also with caches longer than 512 positions (attention split over workgroups);
    PATH_GRAPH forces the graph."""
    hip = pkg.HipModel(gguf(preset), max_seq=64)
    assert hip.decode_path() == want
    hip.set_decode_path(GRAPH)
    assert hip.decode_path() == GRAPH
    hip.close()
    big = pkg.HipModel(gguf(preset), max_seq=1024)
    assert big.decode_path() == want
    big.close()


@pytest.mark.parametrize("path", [GRAPH, STEP], ids=["graph", "step"])
@pytest.mark.parametrize("layout", [0, 1])
@pytest.mark.parametrize("preset", ["tiny_q8", "tiny_f32", "tiny_qwen", "small_q8", "tiny_mixq4", "tiny_hd128"])
def test_long_cache_split_attention(pkg, gguf, preset, layout, path):
    """A 600-token prompt in a 1024-position cache: the step kernel's attention splits the
    positions over its trailing workgroups and merges the splits there, the graph path's
    over split workgroups and a combine launch; each against the oracle while decoding
    past it."""
    info = pkg.synth_preset_info(preset)
    prompt = pkg.synth_prompt(info["seed"] + 7, 600, info["n_vocab"])
    ids, worst, worst_tap, margin = model_parity(pkg, gguf(preset), prompt, 12, 1024, layout, decode_path=path)
    print(f"{preset} layout {layout} path {path}: logits {worst:.2e} taps {worst_tap:.2e} margin {margin:.3e}")


# (preset, prompt tokens, cache positions, switch span): the step kernel's splits move from
# its trailing workgroups to every workgroup once the span passes the switch
# (tf_hip_set_split_all_from). The prompts end a few positions short of it, so the
# per-token decodes and the one-launch greedy loop both cross it; with 1024 and 4096 the
# trailing splits hold 64 positions each at the switch (16 and 64 splits per kv head).
# tiny_hd128 runs the head_dim-128 build (6 query heads per kv head, as the Qwen2.5-1.5B
# shape) through both layouts past 1,800 positions.
@pytest.mark.parametrize("layout", [0, 1])
@pytest.mark.parametrize("preset,n_prompt,max_seq,switch", [("tiny_f32", 1018, 2048, 1024),
                                                            ("tiny_q8", 4090, 4200, 4096),
                                                            ("tiny_qwen", 700, 1024, 705),
                                                            ("tiny_hd128", 1800, 2048, 1805)])
def test_long_cache_split_layout_switch(pkg, gguf, preset, n_prompt, max_seq, switch, layout):
    info = pkg.synth_preset_info(preset)
    prompt = pkg.synth_prompt(info["seed"] + 11, n_prompt, info["n_vocab"])

    def setup(hip):
        hip.set_split_all_from(switch)
        cfg = hip.step_config()
        assert cfg["split"] > 0 and cfg["split_all"] > 0 and cfg["split_all_from"] == switch, cfg

    ids, worst, worst_tap, margin = model_parity(pkg, gguf(preset), prompt, 12, max_seq, layout, decode_path=STEP,
                                                 setup=setup)
    print(f"{preset} {n_prompt} layout {layout}: logits {worst:.2e} taps {worst_tap:.2e} margin {margin:.3e}")


# Caches of at most 512 positions: tokens attending up to 64 positions run attention on one
# workgroup per kv head, longer spans split it. Prompts of 60 tokens put the switch inside
# the per-token decodes and inside the one-launch greedy loop, whose later, split tokens
# read the rows the earlier ones stored from other workgroups. tiny_hd128 and the
# full-size Qwen2.5-1.5B shape run the head_dim-128 build on both sides of the switch.
@pytest.mark.parametrize("layout", [0, 1])
@pytest.mark.parametrize("preset", ["tiny_f32", "tiny_q8", "tiny_qwen", "tiny_hd128", "qwen15b_q8"])
def test_short_cache_split_switch(pkg, gguf, preset, layout):
    info = pkg.synth_preset_info(preset)
    prompt = pkg.synth_prompt(info["seed"] + 5, 60, info["n_vocab"])

    def setup(hip):
        assert hip.decode_path() == STEP
        cfg = hip.step_config()
        # the switch really happens inside the decode: a split layout exists and spans
        # 61..72 cross split_from
        assert cfg["split"] > 0 and cfg["split_from"] == 64, cfg

    ids, worst, worst_tap, margin = model_parity(pkg, gguf(preset), prompt, 12, 512, layout, decode_path=STEP,
                                                 setup=setup)
    print(f"{preset} layout {layout}: logits {worst:.2e} taps {worst_tap:.2e} margin {margin:.3e}")


@pytest.mark.parametrize("span", [0, 512])
def test_split_from_knob(pkg, gguf, span):
    """tf_hip_set_split_from: every token split (0) or none below 512 positions (512) gives
    the same function; values above 512 are rejected."""
    preset = "tiny_q8"
    info = pkg.synth_preset_info(preset)
    prompt = pkg.synth_prompt(info["seed"] + 3, 40, info["n_vocab"])

    def setup(hip):
        with pytest.raises(RuntimeError, match="above 512"):
            hip.set_split_from(513)
        hip.set_split_from(span)
        assert hip.step_config()["split_from"] == span

    ids, worst, _, _ = model_parity(pkg, gguf(preset), prompt, 12, 512, 0, decode_path=STEP, setup=setup)
    print(f"split_from {span}: logits {worst:.2e}")


def test_exchange_epoch_wrap(pkg, gguf):
    """A greedy launch that runs the step kernel's 32-bit exchange epoch past 2^32: the
    backend clears the exchange words and restarts the count, and the tokens and logits
    are those of a run far from the wrap."""
    path = gguf("small_q8")
    prompt = np.array([3, 99, 7, 1200, 5, 42, 8], np.int32)
    out = []
    for start in (None, 2**32 - 300):
        hip = pkg.HipModel(path, max_seq=64)
        hip.set_decode_path(STEP)
        hip.prefill(prompt)
        if start is not None:
            hip.set_exchange_epoch(start)  # a few tokens before the wrap (32 epochs per token)
        ids = hip.generate(24)
        ld, _ = hip.decode(int(ids[-1]))
        out.append((ids, ld))
        hip.close()
    assert np.array_equal(out[0][0], out[1][0])
    assert np.array_equal(out[0][1], out[1][1])


@pytest.mark.parametrize("call", ["generate", "decode", "prefill"])
def test_cooperative_refusal_falls_back_to_graph(pkg, gguf, call):
    """A refused cooperative launch (another process holding the GPU's cooperative-launch
    resource, forced here through the test hook) runs the same tokens on the graph path,
    and the context stays there; the greedy stream equals the oracle's."""
    from oracle.bind import OracleModel, greedy_stream

    path = gguf("tiny_q8")
    info = pkg.synth_preset_info("tiny_q8")
    prompt = pkg.synth_prompt(info["seed"], 6, info["n_vocab"])
    ref_ids, _ = greedy_stream(OracleModel(path, max_seq=64, n_threads=4), prompt, 12)
    hip = pkg.HipModel(path, max_seq=64)
    try:
        assert hip.decode_path() == STEP
        if call == "prefill":
            hip.set_prefill_path(pkg.HipModel.PREFILL_TOKENS)  # the prompt runs on the decode path
            hip.test_refuse_cooperative(1)
        _, am = hip.prefill(prompt)
        assert am == ref_ids[0]
        if call == "decode":
            hip.test_refuse_cooperative(1)
            _, am2 = hip.decode(int(ref_ids[0]))
            assert am2 == ref_ids[1]
            assert np.array_equal(hip.generate(10), ref_ids[1:11])
        else:
            if call == "generate":
                hip.test_refuse_cooperative(1)
            ids = hip.generate(11)
            assert np.array_equal(ids, ref_ids[:11])
        assert hip.decode_path() == GRAPH
        hip.set_decode_path(STEP)  # the switch holds for the context's life
        assert hip.decode_path() == GRAPH
    finally:
        hip.close()


TOKENS, MFMA = 0, 1  # HipModel.PREFILL_TOKENS, HipModel.PREFILL_MFMA


@pytest.mark.parametrize("layout", [0, 1])
@pytest.mark.parametrize("preset", ["tiny_q8", "tiny_qwen", "small_q8"])
def test_small_models_token_prefill(pkg, gguf, preset, layout):
    """The per-token prefill path on the models whose prompts otherwise take the matrix cores."""
    info = pkg.synth_preset_info(preset)
    prompt = pkg.synth_prompt(info["seed"], 6, info["n_vocab"])
    ids, worst, worst_tap, margin = model_parity(pkg, gguf(preset), prompt, 8, 64, layout, prefill_path=TOKENS)
    print(f"{preset} layout {layout}: ids {ids} logits {worst:.2e} taps {worst_tap:.2e} margin {margin:.3e}")


@pytest.mark.parametrize("preset,want", [("tiny_q8", MFMA), ("tiny_qwen", MFMA), ("small_q8", MFMA),
                                         ("tiny_f32", TOKENS), ("tiny_mixq4", MFMA), ("tiny_mixfmt", MFMA)])
def test_prefill_path_selection(pkg, gguf, preset, want):
    """Prompts run on the matrix cores when every layer matrix is Q8_0, Q4_0, Q4_1, F16,
    F32 or Q6_K with rows of a multiple of 64 (256 for Q6_K; gate and up in one format);
    tiny_f32's rows of 32 keep the per-token path; PREFILL_TOKENS forces it."""
    hip = pkg.HipModel(gguf(preset), max_seq=64)
    assert hip.prefill_path() == want
    hip.set_prefill_path(TOKENS)
    assert hip.prefill_path() == TOKENS
    hip.close()


def test_prefill_paths_agree(pkg, gguf):
    """A 150-token prompt through the matrix cores and token by token: logits within 1e-4,
    same argmax, same per-layer activations and KV cache within 1e-4, same greedy stream."""
    path = gguf("small_q8")
    info = pkg.synth_preset_info("small_q8")
    prompt = pkg.synth_prompt(info["seed"] + 1, 150, info["n_vocab"])
    res = []
    for pf in (TOKENS, MFMA):
        hip = pkg.HipModel(path, max_seq=256)
        hip.set_prefill_path(pf)
        lg, am = hip.prefill(prompt)
        taps = [hip.layer_act(layer) for layer in range(5)]
        kv = [hip.read_kv(layer, w, 0, 150) for layer in (0, 3) for w in (0, 1)]
        ids = hip.generate(8)
        res.append((lg, am, taps, kv, ids))
        hip.close()
    (l0, a0, t0, k0, i0), (l1, a1, t1, k1, i1) = res
    assert a0 == a1 and np.array_equal(i0, i1)
    assert rel_err(l1, l0) <= 1e-4
    for a, b in zip(t1, t0):
        assert rel_err(a, b) <= 1e-4
    for a, b in zip(k1, k0):
        assert rel_err(a, b) <= 1e-4


@pytest.mark.parametrize("n_prompt", [2, 16, 17, 32, 33, 64, 65, 129, 257, 2700])
def test_prefill_prompt_lengths(pkg, gguf, n_prompt):
    """Prompt lengths on either side of every tile shape the matrix-core prefill picks by
    row count (16-, 32- and 64-row register-streamed tiles, chunks padded to 128-row tiles,
    K split or not; at 2700 rows gate/up's 264 large tiles run as 242 + 22 in two launches):
    logits, per-layer activations and the greedy stream against the oracle."""
    info = pkg.synth_preset_info("small_q8")
    prompt = pkg.synth_prompt(info["seed"] + n_prompt, n_prompt, info["n_vocab"])
    max_seq = max(512, n_prompt + 64)
    ids, worst, worst_tap, margin = model_parity(pkg, gguf("small_q8"), prompt, 2, max_seq, 0)
    print(f"small_q8 {n_prompt}-token prompt: ids {ids} logits {worst:.2e} taps {worst_tap:.2e}")


# head counts, d_model, ffn, layer formats (q, k, v, o, gate / up, down): row lengths that end in half
# a 128-element stage (192, 320, 4160), an odd number of 16-column tiles, head sizes 32 / 64 / 128, q, k
# and v in one to three formats, Q6_K's super-blocks, and ffn_down in K slices (8192 and 4160 long)
SHORT_PROMPT_MODELS = [
    (6, 2, 192, 320, (8, 8, 8, 8, 8, 8)),
    (4, 2, 256, 8192, (2, 2, 2, 3, 2, 2)),
    (2, 1, 256, 4160, (1, 8, 8, 1, 1, 1)),
    (4, 4, 256, 2048, (14, 3, 2, 14, 14, 14)),
    (8, 1, 256, 8192, (14, 14, 14, 8, 3, 3)),
]


class RawModel:
    """A two-layer context built through the C ABI from rows(rng, slot, type, k, n), with the same
    model in float64. fmts: formats of q, k, v, o, gate / up, down. edit(slot, v) changes a norm's weights
    or a bias in place."""

    def __init__(self, pkg, heads, kv, d, ff, fmts, max_seq, rows, edit=lambda slot, v: None):
        import ctypes as C

        from gpu_util import oracle_dequant

        self.C, self.L = C, pkg.hip_lib()
        self.heads, self.kv, self.d, self.hd, self.vocab, self.layers = heads, kv, d, d // heads, 96, 2
        L, rng, hd = self.L, np.random.default_rng(d + ff), self.hd
        hp = pkg.HParams(self.vocab, d, ff, self.layers, heads, kv, hd, max_seq, 1, 1e-5)
        self.ctx, self.w = C.c_void_p(), {}  # slot -> float64
        assert L.tf_hip_create(0, C.cast(C.byref(hp), C.c_void_p), C.byref(self.ctx)) == 0

        def up(slot, t, k, n):
            raw = rows(rng, slot, t, k, n)
            self.w[slot] = oracle_dequant(t, raw, k).astype(np.float64)
            assert L.tf_hip_upload_tensor(self.ctx, slot, t, k, n, raw.ctypes.data, raw.nbytes) == 0

        def vec(slot, n, mean):
            v = (mean + 0.2 * rng.standard_normal(n)).astype(np.float32)
            edit(slot, v)
            self.w[slot] = v.astype(np.float64)
            assert L.tf_hip_upload_tensor(self.ctx, slot, 0, n, 1, v.ctypes.data, v.nbytes) == 0

        up(0, 8, d, self.vocab)
        vec(1, d, 1.0)
        for l in range(self.layers):
            s = 16 + 12 * l
            for slot, t, k, n in ((1, fmts[0], d, d), (2, fmts[1], d, kv * hd), (3, fmts[2], d, kv * hd),
                                  (4, fmts[3], d, d), (9, fmts[4], d, ff), (10, fmts[4], d, ff), (11, fmts[5], ff, d)):
                up(s + slot, t, k, n)
            for slot, n, mean in ((0, d, 1.0), (8, d, 1.0), (5, d, 0.0), (6, kv * hd, 0.0)):
                vec(s + slot, n, mean)
        self.cos, self.sin = pkg.rope_tables(10000.0, hd, max_seq)
        assert L.tf_hip_set_rope_table(self.ctx, self.f(self.cos), self.f(self.sin), max_seq, hd // 2) == 0

    def f(self, a):
        return a.ctypes.data_as(self.C.POINTER(self.C.c_float))

    def i(self, a):
        return a.ctypes.data_as(self.C.POINTER(self.C.c_int32))

    def close(self):
        self.L.tf_hip_destroy(self.ctx)

    def prefill(self, path, tokens):
        """After a call of tokens 1, 2 (the prompt starts past position 0): logits, then each layer's
        last-row tap, K and V rows."""
        L, n, out = self.L, len(tokens), [np.zeros(self.vocab, np.float32)]
        assert L.tf_hip_set_prefill_path(self.ctx, path) == 0 and L.tf_hip_get_prefill_path(self.ctx) == path
        assert L.tf_hip_reset(self.ctx) == 0
        assert L.tf_hip_prefill(self.ctx, self.i(np.array([1, 2], np.int32)), 2, None, None) == 0
        assert L.tf_hip_prefill(self.ctx, self.i(tokens), n, self.f(out[0]), None) == 0
        for l in range(self.layers):
            out.append(np.zeros(self.d, np.float32))
            assert L.tf_hip_get_layer_act(self.ctx, l, self.f(out[-1])) == 0
            for which in (0, 1):
                out.append(np.zeros((n + 2, self.kv, self.hd), np.float32))
                assert L.tf_hip_read_kv(self.ctx, l, which, 0, n + 2, self.f(out[-1])) == 0
        return out

    def exact(self, tokens):
        """prefill's outputs in float64."""
        w, hd, heads, kv = self.w, self.hd, self.heads, self.kv
        kvs, pos = [[[], []] for _ in range(self.layers)], 0
        for part in ([1, 2], tokens):
            x, taps = w[0][np.asarray(part)], []
            m = len(x)
            c, s = (np.float64(t[pos:pos + m])[:, None] for t in (self.cos, self.sin))
            rope = lambda y: np.concatenate((y[..., :hd // 2] * c - y[..., hd // 2:] * s,  # noqa: E731
                                             y[..., :hd // 2] * s + y[..., hd // 2:] * c), -1)
            norm = lambda y, g: y / np.sqrt((y * y).mean(-1, keepdims=True) + np.float32(1e-5)) * g  # noqa: E731
            for l in range(self.layers):
                W = lambda k: w[16 + 12 * l + k]  # noqa: E731
                y = norm(x, W(0))
                q = rope((y @ W(1).T + W(5)).reshape(m, heads, hd))
                k, v = rope((y @ W(2).T + W(6)).reshape(m, kv, hd)), (y @ W(3).T).reshape(m, kv, hd)
                kvs[l][0].append(k)
                kvs[l][1].append(v)
                a = np.zeros((m, heads, hd))
                for h in range(heads):
                    sc = q[:, h] @ k[:, h * kv // heads].T / np.sqrt(hd)
                    sc[np.triu_indices(m, 1)] = -np.inf
                    e = np.exp(sc - sc.max(1, keepdims=True))
                    a[:, h] = e / e.sum(1, keepdims=True) @ v[:, h * kv // heads]
                x = x + a.reshape(m, self.d) @ W(4).T
                y = norm(x, W(8))
                g = y @ W(9).T
                x = x + (g / (1 + np.exp(-g)) * (y @ W(10).T)) @ W(11).T
                taps.append(x[-1])
            pos += m
        out = [w[0] @ norm(x[-1], w[1])]
        for l in range(self.layers):
            out += [taps[l]] + [np.concatenate(r) for r in kvs[l]]
        return out

    def check(self, tokens):
        """The matrix-core prefill no further from float64 than twice what the per-token prefill of
        the same context is, or 4e-6 where that is closer still (random blocks cancel, so fp32 sums
        in any order lose digits: up to 2e-5 here); its second run bit for bit its first."""
        want, got, again = (self.prefill(p, tokens) for p in (TOKENS, MFMA, MFMA))
        for i, (e, a, b, c) in enumerate(zip(self.exact(tokens), want, got, again)):
            assert rel_err(b, e) <= max(2 * rel_err(a, e), 4e-6), (len(tokens), i, rel_err(b, e), rel_err(a, e))
            assert np.array_equal(b.view(np.uint32), c.view(np.uint32)), (len(tokens), i)


@pytest.mark.parametrize("heads,kv,d,ff", [(80, 10, 10240, 64), (4, 2, 256, 16384)])
def test_long_rows_token_by_token(pkg, heads, kv, d, ff):
    """Rows longer than the 9,216 elements that the GEMV's prologue holds in registers, with and without the
    rmsnorm before them: the per-token path against float64 within the 2e-5 of the other model
    tests, and a decode after it."""
    from rows import random_rows

    m = RawModel(pkg, heads, kv, d, ff, (8,) * 6, 48, lambda rng, slot, t, k, n: random_rows(rng, t, k, n))
    try:
        tokens = np.array([5, 9, 3], np.int32)
        for a, e in zip(m.prefill(TOKENS, tokens), m.exact(tokens)):
            assert rel_err(a, e) <= 2e-5, rel_err(a, e)
        logits = np.zeros(m.vocab, np.float32)
        assert m.L.tf_hip_decode(m.ctx, 7, m.f(logits), None) == 0
        # the decode attends to the first call's tokens too: the same three rows and 7 in one prompt
        assert m.L.tf_hip_reset(m.ctx) == 0
        again = np.zeros(m.vocab, np.float32)
        assert m.L.tf_hip_prefill(m.ctx, m.i(np.array([1, 2], np.int32)), 2, None, None) == 0
        assert m.L.tf_hip_prefill(m.ctx, m.i(tokens), 3, None, None) == 0
        assert m.L.tf_hip_decode(m.ctx, 7, m.f(again), None) == 0
        assert np.array_equal(logits.view(np.uint32), again.view(np.uint32)) and np.all(np.isfinite(logits))
    finally:
        m.close()


@pytest.mark.parametrize("shape", SHORT_PROMPT_MODELS)
def test_short_prompt_kernels(pkg, shape):
    """Prompts of 2 to 16 tokens (their own kernels) and of 17."""
    from rows import random_rows

    heads, kv, d, ff, fmts = shape
    m = RawModel(pkg, heads, kv, d, ff, fmts, 48, lambda rng, slot, t, k, n: random_rows(rng, t, k, n))
    rng = np.random.default_rng(ff)
    try:
        for n in (2, 3, 4, 5, 8, 9, 15, 16, 17):
            m.check(rng.integers(0, m.vocab, n).astype(np.int32))
    finally:
        m.close()


@pytest.mark.parametrize("t", [8, 3, 1, 14, 0])
@pytest.mark.parametrize("ff,n", [(512, 70), (4096, 130), (16384, 250)])
def test_hidden_rows_scaled_by_a_bound(pkg, t, ff, n):
    """ffn_down's operand has its row scales from the gate and up rows' norms: rows of 2^-5 to 2^5 times the
    others (one in 16) put that bound up to 2^14 above most hidden values, inside and outside of what
    needs block exponents (test_hidden_rows_of_uneven_models goes further). The K-split reduce, the
    streamed tiles and the large ones (16,384 hidden units at 250 rows: unsplit) write it. Against
    float64 within the 2e-5 of the other model tests: scaled by the rows' largest values, the same
    models measured up to 1.3e-5 (Q4_1 at 512 hidden units, whose two terms cancel) and 8e-6."""
    def rows(rng, slot, t, k, n):
        w = (rng.standard_normal((n, k)) / np.sqrt(k)).astype(np.float32)
        if slot >= 16 and (slot - 16) % 12 in (9, 10):
            w[::16] *= np.exp2(rng.uniform(-5, 5, w[::16].shape[0])).astype(np.float32)[:, None]
        return np.stack([pkg.quantize_row(t, r) for r in w])

    m = RawModel(pkg, 4, 2, 256, ff, (t,) * 6, 256, rows)
    try:
        tokens = np.random.default_rng(n).integers(0, m.vocab, n).astype(np.int32)
        for a, e in zip(m.prefill(MFMA, tokens), m.exact(tokens)):
            assert rel_err(a, e) <= 2e-5
    finally:
        m.close()


# format, d_model, ffn, prompt, kind (not Q4_1's input channel: its two terms cancel there, in gate and up
# themselves)
UNEVEN_MODELS = [(t, d, ff, n, kind)
                 for d, ff, n in ((256, 512, 70), (256, 4096, 130), (256, 8192, 500), (64, 512, 10), (64, 512, 20), (64, 128, 60))
                 for t in ((8, 3, 1, 14, 0) if d == 256 else (8, 3, 1, 0))
                 for kind in ("rows_8", "rows_10", "silu", "channel") if t != 3 or kind != "channel"]


@pytest.mark.parametrize("t,d,ff,n,kind", UNEVEN_MODELS)
def test_hidden_rows_of_uneven_models(pkg, t, d, ff, n, kind):
    """ffn_down's operand keeps its bits where the norms of the gate and up rows say little about the hidden
    values: one gate row and another unit's up row 2^8 or 2^10 times the others, ffn_down reading
    neither; one unit with a gate so far below 0 that its silu is 0, its up row 2^12 times the others;
    an input channel 2^12 times the others that the weights hardly use. The products of the norms
    are 2^25 to 2^33 above the hidden values. The K-split reduce, the streamed tiles (of 16, 32 and 64
    rows, K split or not) and the large ones (500 rows) write and read it; a V matrix in F32 keeps
    prompts of at most 16 tokens on them. The tolerance is check()'s."""
    def rows(rng, slot, t, k, n):
        w = (rng.standard_normal((n, k)) / np.sqrt(k)).astype(np.float32)
        which = (slot - 16) % 12 if slot >= 16 else -1
        if kind.startswith("rows"):
            if which == 9:
                w[5] *= 2.0 ** int(kind[5:])
            if which == 10:
                w[(n // 2 + 40) % n] *= 2.0 ** int(kind[5:])
            if which == 11:
                w[:, [5, (k // 2 + 40) % k]] = 0.0
        if kind == "silu":
            if slot == 0:
                w[:, 0] = 0.25
            if which == 9:
                w[5] = 0.0
                w[5, 0] = -4096.0
            if which == 10:
                w[5] *= 4096.0
            if which in (4, 11):
                w[0] = 0.0  # the residual rows keep their first element
        if kind == "channel" and which in (9, 10):
            w[:, 0] /= 4096.0
        return np.stack([pkg.quantize_row(t, r) for r in w])

    def edit(slot, v):
        if kind == "channel" and slot >= 16 and (slot - 16) % 12 == 8:
            v[0] = 4096.0

    m = RawModel(pkg, d // 32, d // 64, d, ff, (t, t, 0 if n <= 16 else t, t, t, t), 512, rows, edit)
    try:
        m.check(np.random.default_rng(n).integers(0, m.vocab, n).astype(np.int32))
    finally:
        m.close()


@pytest.mark.parametrize("heads,kv,t,n", [(4, 2, 8, 70), (2, 1, 3, 130), (8, 2, 14, 250), (4, 4, 1, 250), (4, 2, 0, 70)])
def test_attention_rows_of_uneven_values(pkg, heads, kv, t, n):
    """wo's operand keeps its bits in the rows that see small values only: the prompt's last token alone has
    a value element some 2^23 times the others'. K and V rows of the second layer (behind the
    first one's attention) of the tokens before it, no further from float64 than twice the per-token
    path's, or 4e-6 where that is closer still."""
    def rows(rng, slot, t, k, n):
        w = (rng.standard_normal((n, k)) / np.sqrt(k)).astype(np.float32)
        if slot == 0:
            w[:, 0] = 0.0
            w[n - 1, 0] = 1.0
        if slot == 16 + 3:
            w[3, 0] = 2.0 ** 20
        return np.stack([pkg.quantize_row(t, r) for r in w])

    m = RawModel(pkg, heads, kv, 256, 512, (t, t, 0, t, t, t), 256, rows)
    try:
        tokens = np.random.default_rng(n).integers(0, m.vocab - 1, n).astype(np.int32)
        tokens[-1] = m.vocab - 1
        want, got, again = (m.prefill(p, tokens) for p in (TOKENS, MFMA, MFMA))
        for i, e in enumerate(m.exact(tokens)):
            assert np.array_equal(got[i].view(np.uint32), again[i].view(np.uint32)), i
            if i in (5, 6):
                b, a, e = got[i][:-1], want[i][:-1], e[:-1]
                assert rel_err(b, e) <= max(2 * rel_err(a, e), 4e-6), (i, rel_err(b, e), rel_err(a, e))
    finally:
        m.close()


# type, query heads, kv heads, d_model, ffn, max_seq, prompt: rows shorter and longer than a tile, rows
# that do not fill one (192, 320), head sizes 32, 64 and 128, odd ffn row counts for the row groups,
# attention on one workgroup per kv head and split over workgroups
STEP_FORMATS = [
    (1, 6, 2, 192, 320, 64, 5), (1, 2, 1, 256, 1056, 1024, 70), (1, 8, 2, 512, 4160, 64, 5), (1, 8, 8, 1024, 64, 600, 90),
    (14, 4, 2, 256, 512, 64, 5), (14, 2, 1, 256, 768, 1024, 70), (14, 8, 1, 256, 8192, 64, 5), (14, 16, 4, 1280, 256, 600, 90),
]


@pytest.mark.parametrize("shape", STEP_FORMATS)
def test_step_kernel_f16_and_q6k(pkg, shape):
    """F16 and Q6_K models decode on the persistent step kernel: 12 greedy tokens as the graph
    path's, logits and K/V rows of the last within 1e-5 of its (the same products summed in another
    order: 4 sqrt(8192) eps, times two layers)."""
    import ctypes as C

    t, heads, kv, d, ff, max_seq, n_prompt = shape
    hd, vocab, layers = d // heads, 96, 2
    L, rng = pkg.hip_lib(), np.random.default_rng(d + ff + t)
    hp = pkg.HParams(vocab, d, ff, layers, heads, kv, hd, max_seq, 0, 1e-5)
    ctx = C.c_void_p()
    assert L.tf_hip_create(0, C.cast(C.byref(hp), C.c_void_p), C.byref(ctx)) == 0
    F = lambda a: a.ctypes.data_as(C.POINTER(C.c_float))  # noqa: E731
    I = lambda a: a.ctypes.data_as(C.POINTER(C.c_int32))  # noqa: E731

    def up(slot, k, n, sigma=0.02):
        raw = np.stack([pkg.quantize_row(t, (sigma * rng.standard_normal(k)).astype(np.float32)) for _ in range(n)])
        assert L.tf_hip_upload_tensor(ctx, slot, t, k, n, raw.ctypes.data, raw.nbytes) == 0

    up(0, d, vocab, 0.5)
    ones = np.ones(d, np.float32)
    assert L.tf_hip_upload_tensor(ctx, 1, 0, d, 1, ones.ctypes.data, ones.nbytes) == 0
    for l in range(layers):
        s = 16 + 12 * l
        for slot, k, n in ((1, d, d), (2, d, kv * hd), (3, d, kv * hd), (4, d, d), (9, d, ff), (10, d, ff), (11, ff, d)):
            up(s + slot, k, n, 2.0 / np.sqrt(k))
        for slot in (0, 8):
            assert L.tf_hip_upload_tensor(ctx, s + slot, 0, d, 1, ones.ctypes.data, ones.nbytes) == 0
    cos, sin = pkg.rope_tables(10000.0, hd, max_seq)
    assert L.tf_hip_set_rope_table(ctx, F(cos), F(sin), max_seq, hd // 2) == 0
    prompt = rng.integers(0, vocab, n_prompt).astype(np.int32)
    res = []
    for path in (GRAPH, STEP):
        assert L.tf_hip_set_decode_path(ctx, path) == 0 and L.tf_hip_get_decode_path(ctx) == path
        assert L.tf_hip_reset(ctx) == 0
        ids, logits = np.zeros(12, np.int32), np.zeros(vocab, np.float32)
        assert L.tf_hip_prefill(ctx, I(prompt), n_prompt, None, None) == 0
        assert L.tf_hip_generate(ctx, 12, I(ids)) == 0
        assert L.tf_hip_decode(ctx, 3, F(logits), None) == 0
        rows = [np.zeros((n_prompt + 13, kv, hd), np.float32) for _ in range(2)]
        for which in (0, 1):
            assert L.tf_hip_read_kv(ctx, layers - 1, which, 0, n_prompt + 13, F(rows[which])) == 0
        res.append((ids, logits, *rows))
    L.tf_hip_destroy(ctx)
    assert np.array_equal(res[0][0], res[1][0])
    for a, b in zip(res[0][1:], res[1][1:]):
        assert rel_err(b, a) <= 1e-5, rel_err(b, a)


@pytest.mark.parametrize("n_prompt", [6, 150])
@pytest.mark.parametrize("preset", ["tiny_mixq4", "tiny_mixfmt"])
def test_mixed_format_prefill(pkg, gguf, preset, n_prompt):
    """Q4_0 / Q4_1 / F16 / F32 / Q6_K / Q8_0 layer matrices on the matrix cores against the
    oracle (tiny_mixfmt: q, k and v in different formats, one launch each; Q4_1 and F16
    gate / up; F32 q and ffn_down; a Q6_K attention output), and against the per-token
    prefill of the same prompt."""
    info = pkg.synth_preset_info(preset)
    prompt = pkg.synth_prompt(info["seed"] + 3, n_prompt, info["n_vocab"])
    hip = pkg.HipModel(gguf(preset), max_seq=256)
    assert hip.prefill_path() == MFMA
    hip.close()
    ids, worst, worst_tap, margin = model_parity(pkg, gguf(preset), prompt, 8, 256, 0)
    print(f"{preset} {n_prompt}-token prompt: ids {ids} logits {worst:.2e} taps {worst_tap:.2e} margin {margin:.3e}")
    res = []
    for pf in (TOKENS, MFMA):
        hip = pkg.HipModel(gguf(preset), max_seq=256)
        hip.set_prefill_path(pf)
        lg, am = hip.prefill(prompt)
        kv = [hip.read_kv(layer, w, 0, n_prompt) for layer in range(hip.n_layer) for w in (0, 1)]
        res.append((lg, am, kv))
        hip.close()
    (l0, a0, k0), (l1, a1, k1) = res
    assert a0 == a1 and rel_err(l1, l0) <= 1e-4
    for a, b in zip(k1, k0):
        assert rel_err(a, b) <= 1e-4


@pytest.mark.parametrize("n_prompt", [4200, 4097])
def test_long_prompt_runs_in_chunks(pkg, gguf, n_prompt):
    """A prompt longer than one prefill chunk (4096 rows): later chunks attend to the earlier
    ones through the cache, as one attn_prefill over the whole prompt does; 4097 tokens leave
    a last chunk of one row."""
    info = pkg.synth_preset_info("tiny_q8")
    prompt = pkg.synth_prompt(info["seed"] + 2, n_prompt, info["n_vocab"])
    ids, worst, worst_tap, margin = model_parity(pkg, gguf("tiny_q8"), prompt, 4, 4352, 1)
    print(f"tiny_q8 {n_prompt}-token prompt: ids {ids} logits {worst:.2e} taps {worst_tap:.2e}")


def test_step_and_graph_agree(pkg, gguf):
    """Both decode paths give the same greedy stream and logits within 1e-5 from the same state."""
    path = gguf("small_q8")
    prompt = np.array([3, 99, 7, 1200, 5, 42, 8], np.int32)
    out = []
    for p in (GRAPH, STEP):
        hip = pkg.HipModel(path, max_seq=64)
        hip.set_decode_path(p)
        lp, _ = hip.prefill(prompt)
        ids = hip.generate(12)
        ld, _ = hip.decode(int(ids[-1]))
        out.append((lp, ids, ld))
        hip.close()
    assert np.array_equal(out[0][1], out[1][1])
    assert rel_err(out[0][0], out[1][0]) <= 1e-5 and rel_err(out[0][2], out[1][2]) <= 1e-5


def test_reference_ci_prompts(pkg, gguf):
    """The reference's correctness gate corpus (test_correctness.cpp:102-109) on its model shape."""
    path = gguf("tiny_f32")
    for i in range(20):
        prompt = np.array([1, 3 + (i % 20), 5 + (i * 3) % 30, 7], np.int32)
        model_parity(pkg, path, prompt, 8, 64, 0, taps=False)


def test_second_prefill_attends_only_to_its_chunk(pkg, gguf):
    """attn_prefill covers only the current call's tokens (attention.cpp:82-111), also when
    n_pos > 0 at entry; the backend reproduces that."""
    from oracle.bind import OracleModel
    path = gguf("tiny_q8")
    orc = OracleModel(path, max_seq=64)
    hip = pkg.HipModel(path, max_seq=64)
    a = np.array([5, 9, 11], np.int32)
    b = np.array([300, 17, 2, 40], np.int32)
    orc.prefill(a)
    hip.prefill(a)
    lo = orc.prefill(b)
    lh, _ = hip.prefill(b)
    assert rel_err(lh, lo) <= 1e-3
    assert hip.n_pos == 7
    hip.close()


def test_errors_and_reset(pkg, gguf):
    path = gguf("tiny_q8")
    hip = pkg.HipModel(path, max_seq=8)
    with pytest.raises(RuntimeError, match="exceeds max_seq"):
        hip.prefill(np.arange(9, dtype=np.int32))
    with pytest.raises(RuntimeError, match="out of range"):
        hip.decode(hip.n_vocab)
    with pytest.raises(RuntimeError, match="out of range"):
        hip.decode(-1)
    with pytest.raises(RuntimeError):
        hip.generate(3)  # nothing decoded yet
    l1, _ = hip.prefill(np.array([1, 2, 3], np.int32))
    g1 = hip.generate(5)
    with pytest.raises(RuntimeError, match="exceeds max_seq"):
        hip.decode(1)  # position 8 == max_seq
    hip.reset()
    assert hip.n_pos == 0
    l2, _ = hip.prefill(np.array([1, 2, 3], np.int32))
    g2 = hip.generate(5)
    assert np.array_equal(l1, l2) and np.array_equal(g1, g2)  # deterministic replays
    hip.close()


@pytest.mark.parametrize("preset,n_prompt,n_gen,max_seq,layout", [
    ("llama1b_q8", 6, 32, 512, 0),      # Llama-3.2-1B shape, Q8_0: the headline workload
    ("qwen05b_q8", 16, 128, 512, 0),    # Qwen2.5-0.5B shape with QKV bias
    ("llama1b_mixq4", 6, 64, 512, 0),   # Q4_0 / Q4_1 / Q6_K mix
    ("qwen15b_q8", 64, 16, 8192, 1),    # Qwen2.5-1.5B shape, head-major cache (short prompt)
    ("llama1b_q8", 512, 16, 1024, 0),   # 512-token prompt on the matrix cores, then 16 decode tokens
    ("llama1b_q8", 513, 8, 1024, 0),    # 513 rows: gate/up's 320 large tiles run as 256 + 64 (K split)
    ("llama1b_mixq4", 512, 16, 1024, 0),  # the same on Q4_0 / Q4_1 layer matrices
])
def test_full_size(pkg, gguf, preset, n_prompt, n_gen, max_seq, layout):
    info = pkg.synth_preset_info(preset)
    prompt = pkg.synth_prompt(info["seed"], n_prompt, info["n_vocab"])
    ids, worst, worst_tap, margin = model_parity(pkg, gguf(preset), prompt, n_gen, max_seq, layout)
    print(f"{preset}: {len(ids)} tokens identical; logits {worst:.2e} taps {worst_tap:.2e} margin {margin:.3e}")


GOLDEN =__import__("pathlib").Path(__file__).resolve().parent / "golden"


def test_long_context_workload_vs_reference_fixture(pkg, gguf):
    """The Qwen2.5-1.5B-shape workload at full size: a 4096-token prompt (matrix-core
    prefill in one chunk), head-major cache of 8192 positions, then 256 greedy tokens,
    against the reference's own run (tests/golden/qwen15b_4096.npz, written by
    make_golden_long.py from the compiled reference; the taps from the oracle run whose
    logits equal the reference's bit for bit). Per step: the device argmax is the
    reference's token, and the device logits at the reference's top-8 tokens are within
    1e-3 of the largest of them; the last step's taps within 1e-3; the one-launch greedy
    loop from a reset gives the same 256 tokens."""
    fx = np.load(GOLDEN / "qwen15b_4096.npz")
    path = gguf("qwen15b_q8")
    import hashlib
    h = hashlib.sha256()
    with open(path, "rb") as f:
        for chunk in iter(lambda: f.read(1 << 20), b""):
            h.update(chunk)
    assert h.digest() == fx["gguf_sha256"].tobytes(), "synthetic writer output changed"
    info = pkg.synth_preset_info("qwen15b_q8")
    prompt = pkg.synth_prompt(int(fx["prompt_seed"]), int(fx["n_prompt"]), info["n_vocab"])
    ids, top_i, top_v = fx["ids"], fx["top_idx"], fx["top_val"]
    hip = pkg.HipModel(path, max_seq=int(fx["max_seq"]), kv_layout=int(fx["layout"]))
    try:
        assert hip.decode_path() == STEP
        worst = 0.0

        def check(step, lg, am):
            nonlocal worst
            want = top_v[step].astype(np.float64)
            e = float(np.max(np.abs(lg[top_i[step]] - want)) / np.max(np.abs(want)))
            assert e <= 1e-3, f"step {step}: top-8 logits rel err {e:.3e}"
            assert am == int(top_i[step][0]), f"step {step}: argmax {am} != reference {top_i[step][0]}"
            worst = max(worst, e)

        lg, am = hip.prefill(prompt)
        check(0, lg, am)
        for i in range(len(ids)):
            lg, am = hip.decode(int(ids[i]))
            check(i + 1, lg, am)
        for layer, want in zip(fx["tap_layers"], fx["taps"]):
            e = rel_err(hip.layer_act(int(layer)), want)
            assert e <= 1e-3, f"tap {layer} rel err {e:.3e}"
            assert e <= REGRESS, f"tap {layer}: numerics regression {e:.2e}"
        hip.reset()
        _, am0 = hip.prefill(prompt, want_logits=False)
        assert am0 == ids[0]
        gen = hip.generate(len(ids))  # its first token is the prefill's argmax
        assert gen.tolist() == ids.tolist()
        assert worst <= REGRESS, f"numerics regression: top-8 logits {worst:.2e}"
        print(f"qwen15b 4096 + {len(ids)}: ids identical, top-8 logits rel err {worst:.2e}")
    finally:
        hip.close()


@pytest.mark.parametrize("preset,layout", [("tiny_q8", "seq"), ("tiny_qwen", "head"), ("tiny_mixq4", "seq")])
def test_reference_cli_with_gpu_backend(pkg, gguf, preset, layout):
    """The reference's own CLI and Model with the backend switch patched in
    (oracle/backend_patch.py): `--backend hip` prints the same greedy tokens as its CPU path.
    (This process holds the cooperative-launch resource, so the child runs the graph path.)"""
    import os
    import pathlib
    import subprocess

    exe = pathlib.Path(__file__).resolve().parents[1] / "oracle" / "_ref" / "tinferno_backend"
    if not exe.exists():
        pytest.skip("oracle/_ref/tinferno_backend not built (needs the reference sources)")
    info = pkg.synth_preset_info(preset)
    toks = ",".join(str(t) for t in pkg.synth_prompt(info["seed"], 6, info["n_vocab"]))
    args = [str(exe), "--model", gguf(preset), "--tokens", toks, "--n-predict", "16", "--max-seq", "64",
            "--kv-layout", layout, "--threads", "4"]
    env = dict(os.environ, TF_HIP_DECODE_PATH="graph")
    cpu = subprocess.run(args, capture_output=True, text=True, timeout=300, env=env)
    gpu = subprocess.run(args + ["--backend", "hip"], capture_output=True, text=True, timeout=300, env=env)
    assert cpu.returncode == 0 and gpu.returncode == 0, cpu.stderr[-500:] + gpu.stderr[-500:]
    assert gpu.stdout == cpu.stdout and cpu.stdout.strip()
