"""The prompt prefill's kernels at the sizes where they can go wrong: the
direct-to-LDS GEMM at tile, slice and pipeline edges (through the planned form
of the exported GEMM), the gate/up GEMM and the attention through whole
prefills of the toy model against the oracle."""
import ctypes as C

import numpy as np
import pytest

import gen
import toy_model
from test_prefill_gpu import GREEDY, TOY, close, dev, gemm_split, gpu_prefill, prompt, read_cache, toy, within_bound  # noqa: F401

pytestmark = pytest.mark.gpu


# rows at each side of every tile's row count and of the planner's lines; K of
# one to three steps (fewer than the pipeline holds), odd step counts, sliced
# deep products; columns that end inside a tile
@pytest.mark.parametrize("m,n,k", [
    (1, 4, 64), (3, 260, 128), (16, 2048, 192), (17, 100, 2048), (32, 2052, 2048), (33, 3072, 2048), (64, 4096, 2048),
    (65, 1028, 320), (128, 2048, 2048), (129, 2048, 2048), (257, 2048, 2048), (385, 4100, 256), (769, 4096, 256),
    (1, 2048, 4096), (17, 2052, 6144), (33, 2048, 6144), (159, 516, 4160), (160, 2048, 6144), (513, 1000, 6144)])
def test_planned_gemm_matches_float64(hip, m, n, k):
    rng = np.random.default_rng(m * 31 + n + k)
    a = gen.activations(rng, m, k)
    b = gen.bf16(0.05 * rng.standard_normal((n, k)).astype(np.float32))
    got = gemm_split(hip, dev(hip, a), dev(hip, b), m, n, k, 0, 0, 0)
    assert within_bound(got, a, b).all()


@pytest.mark.parametrize("m,n,k", [(24, 320, 2048), (130, 256, 2048), (40, 320, 6144)])
def test_planned_gemm_epilogues_match_separate_ops(hip, orc, m, n, k):
    """Residual add and SiLU gate equal the planned GEMM followed by the
    separate op (the same sums: the plan depends on the sizes alone)."""
    rng = np.random.default_rng(m + n)
    a = gen.activations(rng, m, k)
    b = gen.bf16(0.05 * rng.standard_normal((n, k)).astype(np.float32))
    other = gen.activations(rng, m, n)
    da, db = dev(hip, a), dev(hip, b)
    plain = gemm_split(hip, da, db, m, n, k, 0, 0, 0)
    added = gemm_split(hip, da, db, m, n, k, 0, 0, 0, epilogue=1, c_init=other)
    assert np.array_equal(added, orc.add_in_place(other.ravel(), plain.ravel()).reshape(m, n))
    gated = gemm_split(hip, da, db, m, n, k, 0, 0, 0, epilogue=2, c_init=other)
    assert np.array_equal(gated, orc.silu_gate(other.ravel(), plain.ravel()).reshape(m, n))


def hidden_of(hip, s):
    h = np.zeros(TOY["talker_hidden"], np.uint16)
    hip.call("qwen3_tts_session_read_last_hidden_v1", s, h.ctypes.data, h.nbytes)
    return h


# rows at the edges of this model's gate/up tiles (16 and 64 rows; the others
# need production widths, test_prefill_widths_gpu.py) and of the attention's 16
# query rows and 32 keys, with one wave to all four at work
@pytest.mark.parametrize("rows", [1, 15, 16, 17, 31, 33, 63, 65, 97, 128, 129, 193, 257])
def test_prefill_matches_oracle_at_tile_edges(hip, orc, toy, monkeypatch, rows):  # noqa: F811
    monkeypatch.delenv("QWEN3_TTS_PREFILL", raising=False)
    model, om = toy
    text, codec = prompt(np.random.default_rng(rows), max(rows, 2))
    text, codec = text[:rows], codec[:rows]
    s, _ = gpu_prefill(hip, model, 288, text, codec, GREEDY)
    try:
        o = toy_model.OracleSession(om, 288, 7)
        orc.set_threads(8)
        o.prefill_bf16(text, codec, GREEDY)
        orc.set_threads(1)
        kvw = TOY["talker_key_value_heads"] * 128
        for layer in range(TOY["talker_layers"]):
            for which, name in ((0, "tk"), (1, "tv")):
                ref = o.bufs[name].reshape(TOY["talker_layers"], 288, kvw)[layer, :rows]
                close(read_cache(hip, s, layer, which, rows), ref, f"layer {layer} cache {which}")
        close(hidden_of(hip, s), o.bufs["last"], "last hidden")
    finally:
        hip.load().qwen3_tts_session_destroy(s)


@pytest.mark.parametrize("rows", [5, 37])
def test_prefill_ignores_an_earlier_prompt(hip, toy, monkeypatch, rows):  # noqa: F811
    """A prompt on a session whose caches hold a longer one gives the bits of
    a fresh session (the last 8-position value group is partly stale)."""
    monkeypatch.delenv("QWEN3_TTS_PREFILL", raising=False)
    model, _ = toy
    long_text, long_codec = prompt(np.random.default_rng(1), 90)
    text, codec = prompt(np.random.default_rng(2), rows)
    results = []
    for first in (None, (long_text, long_codec)):
        s, _ = gpu_prefill(hip, model, 128, *(first or (text, codec)), GREEDY)
        try:
            if first is not None:
                pre = hip.PrefillResult()
                p = C.POINTER(C.c_int32)
                hip.call("qwen3_tts_session_prefill", s, text.ctypes.data_as(p), codec.ctypes.data_as(p), rows,
                         hip.SamplingConfig(*GREEDY), C.byref(pre))
            results.append([hidden_of(hip, s)] + [read_cache(hip, s, layer, which, rows)
                                                  for layer in range(TOY["talker_layers"]) for which in (0, 1)])
        finally:
            hip.load().qwen3_tts_session_destroy(s)
    for fresh, reused in zip(*results):
        assert np.array_equal(fresh, reused)


def test_longer_prompts_on_one_session_give_a_fresh_ones_bits(hip, toy, monkeypatch):  # noqa: F811
    """Prompt and row buffers that grow from prompt to prompt (the old ones
    are given back first) change nothing."""
    monkeypatch.delenv("QWEN3_TTS_PREFILL", raising=False)
    model, _ = toy
    s = None
    try:
        for rows in (5, 70, 33, 290):
            text, codec = prompt(np.random.default_rng(rows), rows)
            fresh, want = gpu_prefill(hip, model, 300, text, codec, GREEDY)
            try:
                if s is None:
                    s, got = gpu_prefill(hip, model, 300, text, codec, GREEDY)
                else:
                    got = hip.PrefillResult()
                    p = C.POINTER(C.c_int32)
                    hip.call("qwen3_tts_session_reset", s, 7)
                    hip.call("qwen3_tts_session_prefill", s, text.ctypes.data_as(p), codec.ctypes.data_as(p), rows,
                             hip.SamplingConfig(*GREEDY), C.byref(got))
                assert got.first_semantic_token == want.first_semantic_token
                assert np.array_equal(hidden_of(hip, s), hidden_of(hip, fresh))
                for layer in range(TOY["talker_layers"]):
                    for which in (0, 1):
                        assert np.array_equal(read_cache(hip, s, layer, which, rows),
                                              read_cache(hip, fresh, layer, which, rows))
            finally:
                hip.load().qwen3_tts_session_destroy(fresh)
    finally:
        if s is not None:
            hip.load().qwen3_tts_session_destroy(s)
