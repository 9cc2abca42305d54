"""The few-row prefill kernels (few_rows.hip) against the token-by-token path, at the edges of their tiles."""
import subprocess
import sys

import numpy as np
import pytest

from mongoose_amd import configs
from mongoose_amd import engine as E
from tests import helpers as H
from tests.conftest import ROOT

pytestmark = pytest.mark.gpu

# heads of 128 with a group of 3, widths that end inside a tile and inside a 64-wide step
ODD = configs.TOY._replace(name="odd", nLayers=2, dim=384, nHeads=3, nKVHeads=1, headDim=128, ffnDim=1376 + 32, vocab=300, bias=True)
SMALL = configs.TOY._replace(name="small", nLayers=2, dim=448, nHeads=7, nKVHeads=1, ffnDim=608, vocab=300, bias=True)


WIDE = configs.TOY._replace(name="wide", nLayers=2, dim=512, ffnDim=9728, vocab=300)
NARROW = SMALL._replace(name="narrow", ffnDim=32)          # the down projection's rows are one half chunk, one Q4_0 block


@pytest.mark.parametrize("shape,fmt,kv_f16,pos0,rows", [
    (WIDE, "q8", False, 9, 37), (WIDE, "q4_0", False, 0, 64), (SMALL, "q8", False, 0, 1), (SMALL, "q8", False, 0, 16), (SMALL, "q8", False, 3, 17), (SMALL, "q8", False, 130, 64),
    (SMALL, "q4_0", False, 5, 33), (SMALL, "q4_0", True, 0, 48), (ODD, "q8", False, 100, 15), (ODD, "q8", True, 17, 63),
    (ODD, "q4_0", False, 250, 31), (NARROW, "q8", False, 0, 17), (NARROW, "q4_0", False, 2, 33)])
def test_few_rows_match_token_by_token(hip, shape, fmt, kv_f16, pos0, rows):
    _prefill_against_tokens(hip, shape, fmt, kv_f16, pos0, rows)


# gate | up through LDS: one chunk of 64 k, two (less than the ring holds) and seven, a last tile of 32 columns, rows one past and one
# short of the tiles of 64 and 128 rows
@pytest.mark.parametrize("heads,ffn,fmt,kv_f16,pos0,rows,bm", [
    (1, 9760, "q8", False, 0, 129, 64), (1, 9760, "q4_0", False, 3, 257, 128), (2, 14304, "q8", False, 0, 193, 128), (2, 14304, "q4_0", True, 0, 129, 64),
    (7, 9760, "q8", False, 5, 65, 128), (7, 9760, "q8", True, 0, 255, 64), (7, 9760, "q4_0", False, 0, 127, 128), (7, 9760, "q4_0", False, 9, 191, 64)])
def test_gate_up_tiles_match_token_by_token(hip, heads, ffn, fmt, kv_f16, pos0, rows, bm):
    shape = configs.TOY._replace(name="swiglu", nLayers=2, dim=64 * heads, nHeads=heads, nKVHeads=1, ffnDim=ffn, vocab=300)
    names = _prefill_against_tokens(hip, shape, fmt, kv_f16, pos0, rows)
    assert any("few_swiglu_kernel<%d, %d>" % (fmt == "q4_0", bm) in n for n in names), sorted(set(names))


def _prefill_against_tokens(hip, shape, fmt, kv_f16, pos0, rows):
    """A prompt in one call against the same tokens one by one; the names of the kernels the call launched."""
    m = H.Model(shape, seed=rows, maxSeq=pos0 + rows + 3, eng=hip, oracle=False, fmt=fmt, kv_f16=kv_f16)
    toks = m.prompt(pos0 + rows + 1)
    ref = np.empty(shape.vocab, np.float32)
    for pos in range(pos0 + rows):
        last = pos == pos0 + rows - 1
        rc, nref = m.hip.DecodeToken(int(toks[pos]), pos, ref if last else None)
        assert rc == 0, E.last_error()
    after = np.empty(shape.vocab, np.float32)               # one more token: reads every K/V row
    rc, _ = m.hip.DecodeToken(int(toks[-1]), pos0 + rows, after)
    assert rc == 0
    assert m.hip.ResetKV() == 0
    for pos in range(pos0):
        rc, _ = m.hip.DecodeToken(int(toks[pos]), pos)
        assert rc == 0
    out = []
    names = H.launched(lambda: out.append(m.hip.Prefill(toks[pos0:pos0 + rows], pos0, wantLogits=True)))
    rc, nxt, logits, _ = out[0]
    assert rc == 0, E.last_error()
    bar = 1e-3 if kv_f16 else 1e-4
    assert H.rel_err(logits, ref) < bar and nxt == nref
    got = np.empty(shape.vocab, np.float32)
    rc, _ = m.hip.DecodeToken(int(toks[-1]), pos0 + rows, got)
    assert rc == 0 and H.rel_err(got, after) < bar
    m.close()
    return names


@pytest.mark.parametrize("shape,fmt,kv_f16,n", [
    (SMALL, "q8", False, 3), (SMALL, "q8", False, 4), (SMALL, "q8", False, 17), (SMALL, "q8", False, 18), (SMALL, "q4_0", True, 34),
    (ODD, "q8", False, 16), (ODD, "q4_0", False, 66), (NARROW, "q8", False, 19), (NARROW, "q4_0", False, 34), (WIDE, "q8", False, 49),
    (SMALL, "q8", False, 130), (ODD, "q8", True, 129), (SMALL, "q4_0", False, 258)])
def test_prompts_of_generate_match_token_by_token(hip, shape, fmt, kv_f16, n):
    """Generate takes a prompt's positions through the layers together (from three on, 128 at a time): the token it chooses and
    the logits of the step after, which reads every cache row, against the same tokens one by one.  Bar: the products are the
    same (three bf16 terms are an fp32 value), so what differs are the roundings of fp32 sums: 2^-24 of a partial sum each,
    some 20 that matter in each of 7 products and 4 norms of 2 layers, at random: 2^-24 sqrt(20 * 11 * 2) = 1.3e-6, and
    4e-6 for the largest of the logits.  Two terms would be off by 2^-17 a value at worst, 2^-18 at random: 1e-5 and more."""
    m = H.Model(shape, seed=n, maxSeq=n + 3, eng=hip, oracle=False, fmt=fmt, kv_f16=kv_f16)
    toks = m.prompt(n)
    for pos in range(n):
        rc, want = m.hip.DecodeToken(int(toks[pos]), pos)
        assert rc == 0, E.last_error()
    ref, got = np.empty((2, shape.vocab), np.float32)
    rc, _ = m.hip.DecodeToken(want, n, ref)
    assert rc == 0
    assert m.hip.ResetKV() == 0
    out = []
    names = H.launched(lambda: out.append(m.hip.Generate(toks, 2)))
    rc, t = out[0]
    assert rc == 0 and int(t[0]) == want, E.last_error()
    assert any("few_rows_kernel" in k for k in names) == (n > 3) and any("flow_layers_kernel" in k for k in names)
    rc, _ = m.hip.DecodeToken(want, n, got)
    assert rc == 0 and H.rel_err(got, ref) < (1e-3 if kv_f16 else 4e-6)
    rc, t = m.hip.Generate(toks[::-1].copy(), 2)            # another prompt into the same buffers, and the first again
    assert rc == 0
    rc, t = m.hip.Generate(toks, 1)
    assert rc == 0 and int(t[0]) == want
    m.close()


def test_prompt_without_room_for_its_rows(tmp_path):
    """Generate where the buffer for a prompt's rows cannot be had: the positions go one by one, as where a prompt is short, and
    once there is room they go together.  A hipMalloc that fails when told to stands before the runtime's own, in a process
    of its own (the buffer is the only allocation of such a call: the context has generated two tokens before)."""
    src = tmp_path / "refuse.c"
    src.write_text("""
#define _GNU_SOURCE
#include <dlfcn.h>
#include <stddef.h>
int refuse, refused;
int hipMalloc(void** p, size_t n) {
    static int (*real)(void**, size_t);
    if (!real) real = (int (*)(void**, size_t))dlsym(RTLD_NEXT, "hipMalloc");
    if (refuse) { refused++; return real(p, (size_t)1 << 50); }      /* the runtime's own refusal */
    return real(p, n);
}
""")
    shim = tmp_path / "refuse.so"
    subprocess.run(["gcc", "-shared", "-fPIC", str(src), "-o", str(shim), "-L/opt/rocm/lib", "-Wl,--no-as-needed", "-lamdhip64", "-ldl",
                    "-Wl,-rpath,/opt/rocm/lib"], check=True)
    out = subprocess.run([sys.executable, "-c", """
import ctypes, sys
shim = ctypes.CDLL(sys.argv[1], mode=ctypes.RTLD_GLOBAL)
import numpy as np
from mongoose_amd import engine as E
from tests import helpers as H
from tests.test_gpu_few_rows import SMALL
refuse, refused = (ctypes.c_int.in_dll(shim, n) for n in ("refuse", "refused"))
m = H.Model(SMALL, seed=5, maxSeq=64, eng=E.NewHIP(), oracle=False)
toks = m.prompt(40)
assert m.hip.Generate(toks[:1], 2)[0] == 0
got = []
for r in (1, 0):
    refuse.value = r
    rc, t = m.hip.Generate(toks, 6)
    assert rc == 0, E.last_error()
    got.append(t.tolist())
    after = np.empty(SMALL.vocab, np.float32)
    assert m.hip.DecodeToken(int(t[-1]), 45, after)[0] == 0
    got.append(after)
assert refused.value == 1, refused.value
assert got[0] == got[2], got
assert H.rel_err(got[1], got[3]) < 4e-6
print("same", flush=True)
""", str(shim)], cwd=ROOT, capture_output=True, text=True, timeout=100)
    assert out.returncode == 0 and "same" in out.stdout, out.stdout + out.stderr


@pytest.mark.parametrize("rows,n,k,accumulate", [(1, 16, 32, 0), (17, 33, 96, 1), (64, 300, 1056, 0), (77, 129, 2080, 1), (130, 1000, 4864, 0),
                                                 (513, 2900, 64, 0), (48, 9000, 64, 0), (300, 5632, 160, 1), (17, 33, 32, 1), (200, 1000, 32, 0)])
def test_few_row_gemm_matches_float64(hip, rows, n, k, accumulate):
    rng = np.random.default_rng(rows)
    a = rng.standard_normal((rows, k), dtype=np.float32)
    w = rng.integers(-127, 128, (n, k), dtype=np.int8)
    sc = (0.01 * (1 + rng.random(n))).astype(np.float32)
    bias = rng.standard_normal(n, dtype=np.float32)
    y0 = rng.standard_normal((rows, n), dtype=np.float32)
    ref = a.astype(np.float64) @ (w.astype(np.float64) * sc[:, None]).T + bias + (y0 if accumulate else 0)
    ts = [hip.FromHost(a, a.shape), hip.UploadRawBytes(w), hip.FromHost(sc, sc.shape), hip.FromHost(bias, bias.shape), hip.FromHost(y0, y0.shape)]
    nbytes = 4 * ((rows + 127) // 128 * 128) * ((k + 63) // 64 * 64)
    ws = hip.UploadRawBytes(np.full(nbytes, 0xff, np.uint8))            # padding rows of the planes read as NaN
    E.KQ8Gemm(ts[0], ts[1], ts[2], ts[3], ts[4], rows, n, k, accumulate, ws, nbytes)
    E.KSync()
    assert E.HIPCheck() == 0
    assert H.rel_err(hip.ToHost(ts[4]).reshape(rows, n), ref) < 3e-5
    for t in ts + [ws]:
        t.Release()


@pytest.mark.parametrize("rows,n,k", [(1, 1, 32), (15, 16, 64), (16, 17, 96), (17, 129, 544), (33, 40, 1056), (64, 128, 1024), (65, 600, 1088),
                                      (5, 48, 8192), (9, 20, 8224), (3, 30, 16384)])
def test_few_row_gemm_digits(hip, rows, n, k):
    """Activations as whole numbers of 24 bits times a scale a row and eighth of K, at edges of the runs and tiles, for rows of
    any magnitude.  A value is off by half a step of its run (2^-23 of the largest value), and by three fp32 roundings of itself,
    so a result by sqrt(sum of (step^2 / 12 + (2^-24 a)^2) weight^2) at random: five times that for the worst of up to 20,000,
    and what fp32 loses in a dozen sums and factors, 2^-21 of its terms' root sum of squares in all.  The rows with one large
    value may hold their values as two bf16 terms instead, off by 2^-18 of themselves at random.  A bit fewer would be ten
    deviations, a step of another run (one is 10,000 times the others, with weights of zero for half of the columns)
    thousands.  A row with a NaN or an infinity is NaN."""
    rng = np.random.default_rng(k)
    a = rng.standard_normal((rows, k), dtype=np.float32)
    for i, scale in enumerate((1e-37, 1e30, 1e-21, 0.0, 2.0 ** -64, 1.0)):
        if i + 2 < rows:
            a[i + 2] *= np.float32(scale)
    if rows > 12:
        a[9, rng.integers(k)] = 3e4
        a[10, k // 2], a[11, k - 1] = np.inf, np.nan
        a[12, 0] = -1e36
    w = rng.integers(-128, 128, (n, k), dtype=np.int8)
    per = ((k + 63) // 64 + 7) // 8 * 64                                # k of a run
    if rows > 1 and k > per:
        a[1, per:2 * per] *= np.float32(1e4)
        w[:(n + 1) // 2, per:2 * per] = 0
    sc = (0.01 * (1 + rng.random(n))).astype(np.float32)
    wd = w.astype(np.float64) * sc[:, None].astype(np.float64)
    with np.errstate(invalid="ignore"):
        ref = a.astype(np.float64) @ wd.T
    ta, tw, ts, to = hip.FromHost(a, a.shape), hip.UploadRawBytes(w), hip.FromHost(sc, sc.shape), hip.Zeros([rows, n])
    nbytes = 4 * ((rows + 127) // 128 * 128) * ((k + 63) // 64 * 64)
    ws = hip.UploadRawBytes(np.full(nbytes, 0xff, np.uint8))
    E.KQ8Gemm(ta, tw, ts, None, to, rows, n, k, 0, ws, nbytes)
    E.KSync()
    assert E.HIPCheck() == 0
    got = hip.ToHost(to).reshape(rows, n)
    for i in range(rows):
        if not np.isfinite(a[i]).all():
            assert np.isnan(got[i]).all()
        else:
            x = a[i].astype(np.float64)
            top = np.concatenate([np.full(len(x[r:r + per]), np.abs(x[r:r + per]).max()) for r in range(0, k, per)])
            each = (top / 8355584) ** 2 / 12 + (2.0 ** -24 * x) ** 2
            if i in (9, 12):
                each = np.maximum(each, (2.0 ** -18 * x) ** 2)
            bar = 5 * np.sqrt((wd ** 2) @ each) + 2.0 ** -21 * np.sqrt((wd ** 2) @ (x ** 2))
            assert (np.abs(got[i] - ref[i]) <= bar + 1e-45).all(), (i, (np.abs(got[i] - ref[i]) / (bar + 1e-45)).max())
    for t in (ta, tw, ts, to, ws):
        t.Release()


@pytest.mark.parametrize("rows,n,k", [(1, 1, 32), (17, 33, 96), (33, 40, 544), (16, 130, 1056), (64, 1000, 1024), (65, 600, 2048), (77, 5632, 2048),
                                      (40, 64, 8224)])
@pytest.mark.parametrize("spread", [100.0, 1e3, 1e5, 1e7, 1e20, "lognormal", "half"])
def test_few_row_gemm_keeps_small_values(hip, rows, n, k, spread):
    """Values far below the largest of their row, seen through weights that are zero at the large ones: each is held to 2^-17 of
    itself at worst (two bf16 terms), so a result is off by 2^-18 of sqrt(sum of squared products) at random, six times that for
    the worst of a call, plus fp32 sums: 2^-24 of a partial sum for each of a wave's k / 16 steps and the eight waves.
    "lognormal": magnitudes over eight decades, weights where |a| is below the median; "half": one half a thousandth of the other."""
    rng = np.random.default_rng(k + rows)
    a = rng.standard_normal((rows, k), dtype=np.float32)
    w = rng.integers(-127, 128, (n, k), dtype=np.int8)
    if spread == "lognormal":
        a *= np.exp(4 * rng.standard_normal(k)).astype(np.float32)
        w[:, np.abs(a).mean(axis=0) > np.median(np.abs(a))] = 0
    elif spread == "half":
        small = rng.permutation(k)[:k // 2]
        a[:, small] *= np.float32(1e-3)
        w[:, np.setdiff1d(np.arange(k), small)] = 0
    else:
        at = rng.integers(k)
        a[:, at] = np.float32(spread) * np.where(rng.random(rows) < 0.5, -1, 1)
        w[:, at] = 0
        if rows > 2:
            a[1] *= np.float32(1e-25)                        # a row of tiny values, and one whose large value is alone
            a[2, np.arange(k) != at] = 0
    sc = (0.01 * (1 + rng.random(n))).astype(np.float32)
    wd = w.astype(np.float64) * sc[:, None].astype(np.float64)
    ref = a.astype(np.float64) @ wd.T
    size = np.sqrt((a.astype(np.float64) ** 2) @ (wd ** 2).T)
    ta, tw, ts, to = hip.FromHost(a, a.shape), hip.UploadRawBytes(w), hip.FromHost(sc, sc.shape), hip.Zeros([rows, n])
    nbytes = 4 * ((rows + 127) // 128 * 128) * ((k + 63) // 64 * 64)
    ws = hip.UploadRawBytes(np.full(nbytes, 0xff, np.uint8))
    E.KQ8Gemm(ta, tw, ts, None, to, rows, n, k, 0, ws, nbytes)
    E.KSync()
    assert E.HIPCheck() == 0
    got = hip.ToHost(to).reshape(rows, n)
    bar = 6 * 2.0 ** -18 * size + 2.0 ** -24 * np.sqrt(k / 16 + 16) * size
    worst = (np.abs(got - ref) / (bar + 1e-300)).max()
    assert worst <= 1, worst
    for t in (ta, tw, ts, to, ws):
        t.Release()


@pytest.mark.parametrize("rows,n,accumulate", [(300, 2048, 0), (16, 2048, 1), (40, 1024, 0)])
def test_gemm_over_its_activations(hip, rows, n, accumulate):
    """out may lie over act: the kernel that reads act again, for its small values beside a large one, does not serve such a call.
    Bar: two bf16 terms."""
    k, rng = 2048, np.random.default_rng(rows)
    a = rng.standard_normal((rows, k), dtype=np.float32)
    a[:, 5] *= 1e4
    w = rng.integers(-127, 128, (n, k), dtype=np.int8)
    sc = (0.01 * (1 + rng.random(n))).astype(np.float32)
    ref = a.astype(np.float64) @ (w.astype(np.float64) * sc[:, None]).T + (a if accumulate else 0)
    ta, tw, ts = hip.FromHost(a, a.shape), hip.UploadRawBytes(w), hip.FromHost(sc, sc.shape)
    nbytes = 4 * ((rows + 127) // 128 * 128) * k
    ws = hip.Zeros([nbytes // 4])
    names = H.launched(lambda: E.KQ8Gemm(ta, tw, ts, None, ta, rows, n, k, accumulate, ws, nbytes))
    assert E.HIPCheck() == 0
    assert not any("few_gemm" in x for x in names) and len(names) > 1, names
    assert H.rel_err(hip.ToHost(ta).reshape(-1)[:rows * n].reshape(rows, n), ref) < 3e-5
    for t in (ta, tw, ts, ws):
        t.Release()


@pytest.mark.parametrize("k,kernel", [(1048064, "few_gemm_kernel"), (1049088, "gemm_q8")])
def test_gemm_at_the_longest_rows(hip, k, kernel):
    """One step below and one above the K up to which 32-bit sums hold: every middle digit is -128 and so is every weight (the
    values are 4161536 = 64 * 65536 - 128 * 256 steps of the run, whose largest value is 8355584 of them), which takes a run's
    sum to the limit.  Bar: fp32 sums of equal terms, every one of k / 16 steps rounded the same way by up to 2^-24 of a sum
    that is half the last one on average; a sum past 32 bits is off by twice the result."""
    a = np.full((1, k), 4161536 * 2.0 ** -23, np.float32)
    a[0, ::((k // 64 + 7) // 8 * 64)] = 8355584 * 2.0 ** -23
    w = np.full((3, k), -128, np.int8)
    w[1, :k // 2] = 127
    sc = np.array([0.01, 0.02, 0.03], np.float32)
    ref = a.astype(np.float64) @ (w.astype(np.float64) * sc[:, None].astype(np.float64)).T
    ta, tw, ts, to = hip.FromHost(a, a.shape), hip.UploadRawBytes(w), hip.FromHost(sc, sc.shape), hip.Zeros([1, 3])
    nbytes = 4 * 128 * ((k + 63) // 64 * 64)
    ws = hip.Zeros([nbytes // 4])
    names = H.launched(lambda: E.KQ8Gemm(ta, tw, ts, None, to, 1, 3, k, 0, ws, nbytes))
    E.KSync()
    assert E.HIPCheck() == 0
    assert any(kernel in n for n in names) and ("few_gemm" in kernel) == any("few_gemm" in n for n in names), names
    got = hip.ToHost(to).reshape(1, 3)
    size = np.abs(a.astype(np.float64)) @ (np.abs(w.astype(np.float64)) * sc[:, None]).T
    assert (np.abs(got - ref) <= k / 16 * 2.0 ** -25 * size).all(), (got, ref)
    for t in (ta, tw, ts, to, ws):
        t.Release()


@pytest.mark.parametrize("rows,dim", [(1, 4), (2, 2048), (3, 2052), (1, 4100), (2, 8192), (1, 8196), (2, 30)])
def test_rmsnorm_rows_kept_in_registers_and_others(hip, rows, dim):
    rng = np.random.default_rng(dim)
    a, b = rng.standard_normal((2, rows, dim), dtype=np.float32)
    w = rng.standard_normal(dim, dtype=np.float32)

    def ref(x):
        return x / np.sqrt((x * x).mean(axis=1, keepdims=True) + 1e-5) * w

    ta, tb, tw, to = (hip.FromHost(v, v.shape) for v in (a, b, w, a))
    E.KRMSNormOutEps(ta, to, tw, rows, dim, 1e-5)
    assert H.rel_err(hip.ToHost(to).reshape(rows, dim), ref(a.astype(np.float64))) < 1e-6
    E.KFusedAddRMSNormEps(ta, tb, tb, tw, rows, dim, 1e-5)                 # out may be an operand
    assert H.rel_err(hip.ToHost(tb).reshape(rows, dim), ref(a.astype(np.float64) + b)) < 1e-6
    for t in (ta, tb, tw, to):
        t.Release()


@pytest.mark.parametrize("vocab", [3, 1023, 1024, 1025, 8190, 8193, 9219, 32767, 32770, 40001])
def test_logits_arrive_whole(hip, vocab):
    """The logits cross to the host in slices of at least 1,024 floats, of which eight workgroups take one each in turn: below,
    at and above a slice, eight slices and the most there can be (32), against the oracle, for a single token and behind a
    prompt.  The page-locked buffer holds the call before's values: a slice copied too early would show those."""
    m = H.Model(SMALL._replace(vocab=vocab, nLayers=1), seed=vocab, maxSeq=16, eng=hip)
    toks, got = m.prompt(8), np.empty(vocab, np.float32)
    want = [m.orc.step(m.orc.embed(int(t)), pos, shadow=True)[1] for pos, t in enumerate(toks)]
    for pos, t in enumerate(toks):
        rc, _ = m.hip.DecodeToken(int(t), pos, got)
        assert rc == 0 and H.rel_err(got, want[pos]) < 1e-4, E.last_error()
    for n in (8, 5):
        rc, nxt, logits, _ = m.hip.Prefill(toks[:n], 0, wantLogits=True)
        assert rc == 0 and H.rel_err(logits, want[n - 1]) < 1e-3 and logits[nxt] == logits.max(), E.last_error()
    m.close()


HEADS8 = configs.TOY._replace(name="heads8", nLayers=2, dim=1024, nHeads=8, nKVHeads=2, headDim=128, ffnDim=608, vocab=300)


@pytest.mark.parametrize("shape,kv_f16,pos0,rows,shares", [
    (SMALL, False, 7, 144, 4), (SMALL, False, 0, 145, 2), (SMALL, True, 3, 288, 2), (SMALL, False, 0, 289, 1), (SMALL, True, 30, 16, 4),
    (HEADS8, False, 5, 128, 4), (HEADS8, True, 0, 129, 2), (HEADS8, False, 0, 256, 2), (HEADS8, False, 2, 257, 1), (HEADS8, True, 200, 1, 4)])
def test_prompt_attention_by_columns(hip, shape, kv_f16, pos0, rows, shares):
    """16 queries of a head are shared by four workgroups up to 64 of them, by two up to 128: both sides of each line, against
    the same positions token by token.  Bar: that of test_few_rows_match_token_by_token (fp16 rows: 1e-3)."""
    m = H.Model(shape, seed=rows, maxSeq=pos0 + rows + 2, eng=hip, oracle=False, kv_f16=kv_f16)
    toks = m.prompt(pos0 + rows)
    ref = np.empty(shape.vocab, np.float32)
    for pos in range(pos0 + rows):
        rc, nref = m.hip.DecodeToken(int(toks[pos]), pos, ref if pos == pos0 + rows - 1 else None)
        assert rc == 0, E.last_error()
    out = []
    names = H.launched(lambda: out.append(m.hip.Prefill(toks[pos0:], pos0, wantLogits=True)))
    rc, nxt, logits, _ = out[0]
    assert rc == 0, E.last_error()
    assert any(f"few_attention_kernel<{shape.headDim}, {str(kv_f16).lower()}, {shares}>" in n for n in names), names
    assert H.rel_err(logits, ref) < (1e-3 if kv_f16 else 1e-4)
    m.close()
