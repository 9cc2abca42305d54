"""Batched prefill, on the few-row kernels (few_rows.hip: what most prompts here take) and on the tiled GEMMs (prefill.hip:
the longer ones, the `tiled` tests), against the token-by-token decode step.

The reference has no batched prompt path: its semantics for a prompt are the
decode step applied position by position, which is what the oracle does here.
Bars: last-position logits within 1e-3 relative of the oracle (float path and
double shadow), greedy tokens identical, and the decode that continues from
the prefilled KV caches identical to the all-decode run (which checks every
cache row the prefill wrote).  The GEMM itself is compared with a float64
product at 2e-5 of the largest output (int8 weights are exact in bf16; the
two-term bf16 split of an activation leaves 2^-16 relative)."""
import numpy as np
import pytest

from mongoose_amd import configs
from mongoose_amd import engine as E
from oracle import binding as ob
from tests import helpers as H

pytestmark = pytest.mark.gpu
rng = np.random.default_rng(77)


def _up(eng, a):
    return eng.UploadRawBytes(np.ascontiguousarray(a))


@pytest.mark.parametrize("T,N,K,acc,bias", [
    (1, 128, 32, False, False), (5, 100, 64, False, True), (130, 300, 896, True, False),
    (128, 128, 4864, False, False), (257, 1376, 512, True, True), (512, 1024, 4096, False, False),
    # wide matrices: accumulate form, bias form, odd count of 32-wide K steps
    (512, 12288, 64, True, False), (300, 12800, 96, False, True),
])
def test_q8_gemm_against_float64(hip, T, N, K, acc, bias):
    _gemm_against_float64(hip, T, N, K, acc, bias)


@pytest.mark.parametrize("T,N,K,acc,bias,kernel", [
    # past the few-row kernel's line: the small tiles; 256 x 256 tiles with K not a multiple of 128, and through the
    # direct-to-LDS ring (accumulate and bias forms of each; the last row and column tiles partly empty)
    (513, 2925, 32, True, False, "gemm_q8_bf16x2_kernel<0, 64, 128, 256, 1>"), (520, 3001, 96, False, True, "gemm_q8_bf16x2_kernel<0, 64, 128, 256, 0>"),
    (600, 17408, 64, True, False, "gemm_q8_bf16x2_kernel<0, 256, 256, 1024, 1>"), (550, 17300, 96, False, True, "gemm_q8_bf16x2_kernel<0, 256, 256, 1024, 0>"),
    (600, 17400, 128, True, True, "gemm_q8_ring_kernel<1>"), (530, 17408, 384, False, True, "gemm_q8_ring_kernel<0>"),
])
def test_q8_gemm_tiled_against_float64(hip, T, N, K, acc, bias, kernel):
    names = H.launched(lambda: _gemm_against_float64(hip, T, N, K, acc, bias))
    assert any(kernel in n for n in names) and not any("few_rows" in n for n in names), names


def _gemm_against_float64(hip, T, N, K, acc, bias):
    print(f"q8 gemm T={T} N={N} K={K} acc={acc} bias={bias}", flush=True)
    w = E.synth_normal(9, T * 7 + N, 0.02, (N, K))
    q, s = ob.quantize_q8(w)
    a = rng.standard_normal((T, K)).astype(np.float32)
    b = rng.standard_normal(N).astype(np.float32) if bias else None
    y0 = rng.standard_normal((T, N)).astype(np.float32)
    plane = 2 * ((T + 127) // 128 * 128) * ((K + 63) // 64 * 64)
    dq, ds, da, dy = _up(hip, q), _up(hip, s), _up(hip, a), _up(hip, y0)
    db = _up(hip, b) if bias else None
    ws = hip.UploadRawBytes(np.zeros(2 * plane, np.uint8))
    E.KQ8Gemm(da, dq, ds, db, dy, T, N, K, acc, ws, 2 * plane)
    E.KSync()
    assert E.HIPCheck() == 0
    got = hip.DownloadRawBytes(dy, T * N * 4).view(np.float32).reshape(T, N)
    ref = (a.astype(np.float64) @ q.astype(np.float64).T) * s.astype(np.float64)[None, :]
    if bias:
        ref = ref + b.astype(np.float64)[None, :]
    if acc:
        ref = ref + y0.astype(np.float64)
    assert H.rel_err(got, ref) < 2e-5
    # row 0 is also what the decode matvec gives for the same activation
    if not acc and not bias:
        mv = ob.q8_matvec(a[0], q, s, shadow=True, threads=4)
        assert H.rel_err(got[0], mv) < 2e-5
    for t in (dq, ds, da, dy, ws) + ((db,) if bias else ()):
        t.Release()


def test_q8_gemm_rejects_bad_arguments(hip):
    t = hip.Zeros([64])
    E.KQ8Gemm(t, t, t, None, t, 1, 1, 31, False, t, 256)      # K not a multiple of 32
    E.KSync()
    assert E.HIPCheck() != 0
    E.KQ8Gemm(t, t, t, None, t, 1, 1, 32, False, t, 16)       # workspace too small
    E.KSync()
    assert E.HIPCheck() != 0
    assert E.HIPCheck() == 0                                    # the error is reported once
    t.Release()


def _oracle_prompt_logits(m, prompt, shadow):
    m.orc.reset_kv()
    logits = None
    for pos, tok in enumerate(prompt):
        _, logits, _ = m.orc.decode_token(int(tok), pos, shadow=shadow, want_layers=False)
    return logits.copy()


def _prefill_case(hip, s, seed, nPrompt, nDecode, maxSeq, kv_f16=False):
    m = H.Model(s, seed=seed, maxSeq=maxSeq, eng=hip, threads=8, kv_f16=kv_f16)
    prompt = m.prompt(nPrompt)
    lg32 = _oracle_prompt_logits(m, prompt, False)
    lg64 = _oracle_prompt_logits(m, prompt, True)
    assert m.hip.ResetKV() == 0
    rc, nxt, logits, ms = m.hip.Prefill(prompt, 0, wantLogits=True)
    assert rc == 0, E.last_error()
    assert ms > 0
    assert H.rel_err(logits, lg64) < 1e-3 and H.rel_err(logits, lg32) < 1e-3
    assert nxt == int(np.argmax(lg32)) == int(np.argmax(lg64))
    # the token-by-token GPU path gives the same logits to well inside the bar
    assert m.hip.ResetKV() == 0
    lg_dec = np.empty(s.vocab, np.float32)
    for pos, tok in enumerate(prompt):
        rc, _ = m.hip.DecodeToken(int(tok), pos, lg_dec if pos == len(prompt) - 1 else None)
        assert rc == 0, E.last_error()
    assert H.rel_err(logits, lg_dec) < 1e-4
    # decode continues from the prefilled caches exactly as from decoded ones
    toks_ref, _ = H.oracle_generate(m, prompt, nDecode)
    assert m.hip.ResetKV() == 0
    rc, toks_dec = m.hip.Generate(prompt, nDecode, useGraph=True)
    assert rc == 0, E.last_error()
    assert m.hip.ResetKV() == 0
    rc, toks_pf = m.hip.GeneratePrefill(prompt, nDecode)
    assert rc == 0, E.last_error()
    assert toks_pf.tolist() == toks_dec.tolist() == toks_ref.tolist()
    return m, prompt, logits


def test_prefill_toy_matches_decode(hip):
    m, prompt, logits = _prefill_case(hip, configs.TOY, seed=1, nPrompt=37, nDecode=24, maxSeq=72)
    # chunked: 20 positions, then the remaining 17 starting at pos0 = 20
    assert m.hip.ResetKV() == 0
    rc, _, _, _ = m.hip.Prefill(prompt[:20], 0)
    assert rc == 0, E.last_error()
    rc, nxt2, logits2, _ = m.hip.Prefill(prompt[20:], 20, wantLogits=True)
    assert rc == 0, E.last_error()
    assert H.rel_err(logits2, logits) < 1e-5
    # a single-token prefill is a decode step
    assert m.hip.ResetKV() == 0
    rc, n1, l1, _ = m.hip.Prefill(prompt[:1], 0, wantLogits=True)
    assert rc == 0, E.last_error()
    assert m.hip.ResetKV() == 0
    l2 = np.empty(m.s.vocab, np.float32)
    rc, n2 = m.hip.DecodeToken(int(prompt[0]), 0, l2)
    assert rc == 0 and n1 == n2 and H.rel_err(l1, l2) < 1e-5
    m.close()


def test_prefill_qwen_shape_with_bias(hip):
    """Qwen2.5-0.5B shape (GQA 14/2, head 64, QKV bias), 3 layers, 200-token prompt (few-row kernels, 13 row blocks)."""
    s = H.with_layers(configs.QWEN, 3)
    m, _, _ = _prefill_case(hip, s, seed=3, nPrompt=200, nDecode=8, maxSeq=256)
    m.close()


def test_prefill_llama3_shape_one_layer(hip):
    """Llama-3-8B shape (head 128, GQA 32/8), 1 layer, 160-token prompt (tiled GEMMs: past 128 rows)."""
    s = H.with_layers(configs.LLAMA3_8B, 1)
    m, _, _ = _prefill_case(hip, s, seed=4, nPrompt=160, nDecode=4, maxSeq=192)
    m.close()


def test_prefill_llama3_shape_two_row_tiles(hip):
    """Llama-3-8B layer shape with a 300-token prompt (vocab cut to 8192 so the oracle stays fast): two
    256-row tiles, which is where the gate|up GEMM has enough tiles to run unsplit and forms
    silu(gate)*up in its own epilogue, while q|k|v, Wo and down split K and finish in the
    row-wise kernels (RoPE + cache rows; residual + next norm + split)."""
    s = H.with_layers(configs.LLAMA3_8B, 1)._replace(vocab=8192)
    m, _, _ = _prefill_case(hip, s, seed=14, nPrompt=300, nDecode=2, maxSeq=320)
    m.close()


def test_prefill_wide_ffn_with_a_partial_column_tile(hip):
    """An FFN of 80.5 tiles of 128 columns at 300 rows, on the few-row kernels (the tiled GEMMs' partial gate|up tile:
    test_tiled_prefill)."""
    s = configs.Shape("ffn-edge", 1, 256, 4, 2, 64, 10304, 512, 1e-5, 1e4, False, True, "q8")
    m, _, _ = _prefill_case(hip, s, seed=21, nPrompt=300, nDecode=2, maxSeq=320)
    m.close()


def test_prefill_fp16_kv(hip):
    """Prefill writing fp16 KV rows (head sizes 64 and 128) against the oracle with the same rounding."""
    m, _, _ = _prefill_case(hip, H.with_layers(configs.QWEN, 2), seed=7, nPrompt=70, nDecode=6, maxSeq=96, kv_f16=True)
    m.close()
    s = configs.Shape("l3-mini", 2, 512, 4, 1, 128, 1024, 512, 1e-5, 5e5, False, True, "q8")
    m, _, _ = _prefill_case(hip, s, seed=8, nPrompt=45, nDecode=6, maxSeq=64, kv_f16=True)
    m.close()


def test_prefill_buffer_growth_and_sequence_end(hip):
    """Row buffers grow with the prompt (small call first), and a prompt may run to the last position."""
    s = H.with_layers(configs.TOY, 2)
    maxSeq = 200
    m = H.Model(s, seed=12, maxSeq=maxSeq, eng=hip, threads=8)
    prompt = m.prompt(maxSeq)
    rc, n_small, _, _ = m.hip.Prefill(prompt[:5], 0)                  # allocates for 128 rows
    assert rc == 0, E.last_error()
    assert m.hip.ResetKV() == 0
    rc, nxt, logits, _ = m.hip.Prefill(prompt, 0, wantLogits=True)    # 200 rows: buffers are re-made; ends at maxSeq - 1
    assert rc == 0, E.last_error()
    lg64 = _oracle_prompt_logits(m, prompt, True)
    assert H.rel_err(logits, lg64) < 1e-3 and nxt == int(np.argmax(lg64))
    # the position after the last one does not exist
    assert m.hip.Prefill(prompt[:1], maxSeq)[0] == -2
    # prompt + decode may fill the sequence exactly: maxSeq - 3 prompt positions, 4 tokens (the last needs no cache row)
    assert m.hip.ResetKV() == 0
    rc, toks = m.hip.GeneratePrefill(prompt[:maxSeq - 3], 4)
    assert rc == 0, E.last_error()
    assert m.hip.ResetKV() == 0
    rc, toks_dec = m.hip.Generate(prompt[:maxSeq - 3], 4, useGraph=True)
    assert rc == 0 and toks.tolist() == toks_dec.tolist()
    assert m.hip.GeneratePrefill(prompt[:maxSeq - 3], 5)[0] == -2
    m.close()


def test_prefill_errors(hip):
    s = H.with_layers(configs.TOY, 1)
    m = H.Model(s, seed=2, maxSeq=32, eng=hip, oracle=False)
    assert m.hip.Prefill(np.zeros(33, np.int32), 0)[0] == -2          # longer than maxSeq
    assert m.hip.Prefill(np.zeros(4, np.int32), 30)[0] == -2          # runs past maxSeq
    assert m.hip.Prefill(np.array([s.vocab], np.int32), 0)[0] == -2   # token out of range
    assert m.hip.Prefill(np.zeros(4, np.int32), 0)[0] == 0
    m.close()


def test_prefill_qwen_q4_0_shape(hip):
    """Qwen shape with GGUF Q4_0 weights and an fp16 embedding table, 2 layers, 150-token prompt."""
    s = H.with_layers(configs.QWEN_Q4, 2)
    m, _, _ = _prefill_case(hip, s, seed=5, nPrompt=150, nDecode=6, maxSeq=192)
    m.close()


def test_prefill_q4_0_short_prompt_and_k_tail(hip):
    """Toy shape in Q4_0 (ffn 1376: a K of 43 blocks, odd, so the last K step is half empty), 40-token prompt."""
    s = configs.TOY._replace(fmt="q4_0", name="toy-q4")
    m, _, _ = _prefill_case(hip, s, seed=6, nPrompt=40, nDecode=6, maxSeq=64)
    m.close()


EDGE = configs.Shape("ffn-edge", 1, 256, 4, 2, 64, 10304, 512, 1e-5, 1e4, True, True, "q8")
ODD = configs.Shape("odd", 2, 384, 3, 1, 128, 1408, 300, 1e-6, 1e4, True, True, "q8")
MINI = configs.Shape("l3-mini", 2, 512, 4, 1, 128, 1024, 512, 1e-5, 5e5, True, True, "q8")


@pytest.mark.parametrize("s,fmt,kv_f16,pos0,rows,kernels", [
    # an FFN of 80.5 tiles of 128 columns: the gate|up GEMM runs unsplit on the 256 x 256 tiles and forms silu(gate)*up
    # itself.  Whole tiles leave through LDS as 128-byte rows (row blocks past the planes' 896 rows are skipped), the last
    # tile has 64 columns and stores element by element; the down projection then reads both.  Biases without a K split
    (EDGE, "q8", False, 0, 820, ["gemm_q8_ring_kernel<3>", "rope_store_rows"]),
    # ... and in Q4_0, whose gate and up leave the GEMM apart
    (EDGE, "q4_0", False, 7, 820, ["gemm_q8_bf16x2_kernel<1, 128, 256, 512, 0>", "swiglu_split_kernel"]),
    # K split: biases, RoPE and fp16 K/V rows in the kernel that sums the splits
    (H.with_layers(configs.QWEN, 2), "q8", True, 0, 600, ["gemm_q8_bf16x2_kernel<0, 64, 128, 256, 2>", "gemm_reduce_qkv_rope"]),
    # Q4_0 gate|up with the SwiGLU in the epilogue of the tiles in between; an fp16 embedding table
    (H.with_layers(configs.QWEN_Q4, 2), "q4_0", False, 33, 600, ["gemm_q8_bf16x2_kernel<1, 128, 256, 512, 3>", "gemm_reduce_norm_split"]),
    # heads of 128 in groups of 3, widths that end inside a tile: SwiGLU in the small tiles' epilogue, K/V rows of 128
    (ODD, "q8", False, 0, 1505, ["gemm_q8_bf16x2_kernel<0, 64, 128, 256, 3>", "rope_store_rows"]),
    (ODD, "q4_0", True, 3, 1505, ["gemm_q8_bf16x2_kernel<1, 64, 128, 256, 1>", "rope_store_rows"]),
    (MINI, "q8", True, 0, 1510, ["gemm_reduce_swiglu_split", "gemm_reduce_qkv_rope"]),
    # a K of 43 blocks: the last K step is half empty
    (configs.TOY, "q4_0", False, 0, 1390, ["gemm_q8_bf16x2_kernel<1, 64, 128, 256, 2>", "gemm_reduce_swiglu_split"]),
    # large matrices: the ring kernel with K splits; Q4_0 on the large tiles with and without, fp16 K/V rows
    (H.with_layers(configs.TINYLLAMA, 1)._replace(vocab=2000), "q8", False, 0, 350, ["gemm_q8_ring_kernel<2>"]),
    (H.with_layers(configs.LLAMA3_8B, 1)._replace(vocab=2000), "q4_0", True, 0, 170, ["gemm_q8_bf16x2_kernel<1, 128, 256, 512, 2>", "swiglu_split_kernel"]),
    # behind cached rows, three rounds of attention workgroups: a prefill that takes the few-row kernels with nothing cached
    (H.with_layers(configs.TOY, 1), "q8", False, 3000, 1050, ["gemm_q8_bf16x2_kernel"]),
], ids=lambda v: getattr(v, "name", None))
def test_tiled_prefill(hip, s, fmt, kv_f16, pos0, rows, kernels):
    """The tiled GEMMs against the oracle: the last row's logits, and those of a token behind it, which reads every K/V row.
    The bars: a product's two bf16 terms leave 2^-16 of an activation, some 1e-5 of the logits over these layers, ten times
    that is asked for; fp16 rows round at 2^-11 of a value, averaged over the rows, and keep the logit bar."""
    m = H.Model(s, seed=rows, maxSeq=pos0 + rows + 2, eng=hip, threads=16, fmt=fmt, kv_f16=kv_f16)
    toks = m.prompt(pos0 + rows + 1)
    want = []
    m.orc.reset_kv()
    for pos, tok in enumerate(toks):
        _, logits, _ = m.orc.decode_token(int(tok), pos, shadow=True, want_layers=False)
        if pos >= pos0 + rows - 1:
            want.append(logits.copy())
    for p in range(0, pos0, 1000):
        assert m.hip.Prefill(toks[p:min(pos0, p + 1000)], p)[0] == 0, E.last_error()
    got = []
    names = H.launched(lambda: got.append(m.hip.Prefill(toks[pos0:pos0 + rows], pos0, wantLogits=True)))
    rc, nxt, logits, _ = got[0]
    assert rc == 0, E.last_error()
    assert not any("few_" in n for n in names) and all(any(k in n for n in names) for k in kernels), sorted(set(names))
    bar = 1e-3 if kv_f16 else 1e-4
    assert H.rel_err(logits, want[0]) < bar and nxt == int(np.argmax(want[0]))
    after = np.empty(s.vocab, np.float32)
    rc, _ = m.hip.DecodeToken(int(toks[-1]), pos0 + rows, after)
    assert rc == 0 and H.rel_err(after, want[1]) < bar
    m.close()


@pytest.mark.parametrize("s,fmt,kv_f16,pos0,rows,attention", [
    (H.with_layers(configs.TOY, 3), "q8", False, 0, 1, "few_attention_kernel"), (H.with_layers(configs.QWEN, 2), "q8", False, 300, 33, "few_attention_kernel"),
    (H.with_layers(configs.QWEN_Q4, 2), "q4_0", True, 20, 16, "few_attention_kernel"), (MINI, "q8", True, 127, 2, "few_attention_kernel"),
    (ODD, "q8", False, 0, 1505, "prefill_attn_kernel"), (ODD, "q4_0", True, 3, 1505, "prefill_attn_kernel"),
    (H.with_layers(configs.TOY, 1), "q8", False, 0, 18, "few_attention_kernel")], ids=lambda v: getattr(v, "name", None))
def test_last_layer_for_the_last_position(hip, s, fmt, kv_f16, pos0, rows, attention):
    """Behind its cache rows the last of several layers runs for the last position alone, by the decode step's launches: logits, the
    hidden buffer (whose bar is that of the logits: an element is off by what two bf16 terms leave, 2^-16, over the layers) and the
    token behind it, against the same tokens one by one."""
    m = H.Model(s, seed=rows, maxSeq=pos0 + rows + 2, eng=hip, oracle=False, fmt=fmt, kv_f16=kv_f16)
    toks = m.prompt(pos0 + rows + 1)
    ref, after, got = (np.empty(s.vocab, np.float32) for _ in range(3))
    m.hip.SetExecMode(1)                                       # (a token's last row stays in the hidden buffer)
    for pos in range(pos0 + rows):
        rc, nref = m.hip.DecodeToken(int(toks[pos]), pos, ref if pos == pos0 + rows - 1 else None)
        assert rc == 0, E.last_error()
    href = m.hip.ExportHidden().copy()
    assert m.hip.DecodeToken(int(toks[-1]), pos0 + rows, after)[0] == 0
    assert m.hip.ResetKV() == 0
    for pos in range(pos0):
        assert m.hip.DecodeToken(int(toks[pos]), pos)[0] == 0
    out = []
    names = H.launched(lambda: out.append(m.hip.Prefill(toks[pos0:pos0 + rows], pos0, wantLogits=True)))
    rc, nxt, logits, _ = out[0]
    assert rc == 0, E.last_error()
    assert sum(attention in n for n in names) == max(1, s.nLayers - 1) and any("attn_decode" in n for n in names) == (s.nLayers > 1), names
    bar = 1e-3 if kv_f16 else 1e-4
    assert H.rel_err(logits, ref) < bar and nxt == nref
    assert H.rel_err(m.hip.ExportHidden(), href) < bar
    assert m.hip.DecodeToken(int(toks[-1]), pos0 + rows, got)[0] == 0 and H.rel_err(got, after) < bar
    m.close()


@pytest.mark.parametrize("s,rows", [(H.with_layers(configs.TOY, 1), 2), (H.with_layers(configs.TOY, 1), 1100), (MINI, 7)], ids=lambda v: getattr(v, "name", None))
def test_the_last_row_takes_no_copy_of_its_own(hip, s, rows):
    """A call's launches are its kernels, at any number of layers: the row that the lm_head reads reaches the hidden buffer in one of
    them."""
    m = H.Model(s, seed=rows, maxSeq=rows + 2, eng=hip, oracle=False)
    toks = m.prompt(rows)
    assert m.hip.Prefill(toks, 0)[0] == 0                      # (tables and buffers are there afterwards)
    names = H.launched(lambda: m.hip.Prefill(toks, 0))
    assert names and not any("memcpy" in n.lower() or "copybuffer" in n.lower() for n in names), names
    m.close()
