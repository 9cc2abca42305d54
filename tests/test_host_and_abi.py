"""CPU-side checks of the product: the C ABI library loads and exports every
symbol the header declares, and its host-side quantizers / fp16 conversion /
synthetic generator agree bit for bit with the oracle (no GPU needed)."""
import ctypes
import os
import re
import subprocess

import numpy as np
import pytest

from mongoose_amd import engine as E
from mongoose_amd.lib import LIB_PATH, lib
from oracle import binding as ob

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
rng = np.random.default_rng(99)


def test_library_exports_every_declared_symbol():
    hdr = open(os.path.join(ROOT, "include", "mongoose_hip.h")).read()
    hdr = re.sub(r"/\*.*?\*/", "", hdr, flags=re.S)
    declared = set(re.findall(r"\b((?:mg|tw|mongoose)_[a-z0-9_]+)\s*\(", hdr))
    assert len(declared) > 50
    out = subprocess.check_output(["nm", "-D", "--defined-only", LIB_PATH], text=True)
    exported = {l.split()[-1] for l in out.splitlines() if " T " in l}
    missing = sorted(declared - exported)
    assert not missing, missing
    for name in declared:
        assert getattr(lib, name) is not None


def test_host_q8_quantizer_matches_oracle_bit_for_bit():
    w = (rng.standard_normal((64, 896)) * 0.02).astype(np.float32)
    w[0] = 0
    w[1, 5] = 9.0
    for mode in (0, 1):
        q, s = E.quantize_q8(w, mode)
        qo, so = ob.quantize_q8(w, mode)
        assert (q == qo).all() and (s.view(np.uint32) == so.view(np.uint32)).all()


def test_host_q4_0_quantizer_matches_oracle_bit_for_bit():
    w = (rng.standard_normal((32, 4864)) * 0.02).astype(np.float32)
    w[0, :32] = 0
    assert (E.quantize_q4_0(w) == ob.quantize_q4_0(w)).all()


def test_host_fp16_matches_oracle():
    xs = np.concatenate([(rng.standard_normal(5000) * 10.0 ** rng.uniform(-9, 5, 5000)).astype(np.float32),
                         np.array([0, -0.0, 65504, 65520, 1e9, 2.0 ** -24, 2.0 ** -25, 6e-8], np.float32)])
    for x in xs:
        assert lib.mg_f32_to_f16(float(x)) == ob.lib.orc_f32_to_f16(float(x))
    for b in range(0, 65536, 7):
        a, o = lib.mg_f16_to_f32(b), ob.lib.orc_f16_to_f32(b)
        assert (np.isnan(a) and np.isnan(o)) or a == o


def test_synthetic_generator_is_deterministic_and_normal():
    a = E.synth_normal(1, 2, 0.02, (1000, 333))
    b = E.synth_normal(1, 2, 0.02, (1000, 333))
    assert (a == b).all()
    assert not (a == E.synth_normal(1, 3, 0.02, (1000, 333))).all()
    assert abs(float(a.mean())) < 2e-4 and abs(float(a.std()) - 0.02) < 2e-4
    # fraction beyond 2 sigma ~ 4.55 %
    assert abs(float((np.abs(a) > 0.04).mean()) - 0.0455) < 0.003
    # pinned values: the stream must be the same on every machine
    c = E.synth_normal(42, 7, 1.0, (8,))
    assert c.view(np.uint32).tolist() == PINNED_42_7
    t = E.synth_tokens(42, 7, 151936, 6)
    assert t.tolist() == PINNED_TOK_42_7 and t.min() >= 0 and t.max() < 151936


PINNED_42_7 = [3211424173, 1066722117, 1057553308, 3206656046, 3224072043, 3213916856, 1036707676, 1063582405]
PINNED_TOK_42_7 = [27601, 53205, 31491, 35801, 36736, 81368]


def test_context_requires_device_or_fails_cleanly():
    # Without a GPU, NewHIP() is None and so is the context (nil constructor
    # convention, cuda.go:213-217); with one, both exist.
    eng = E.NewHIP()
    f = E.NewHIPFusedInference(eng, 512, 512, 64, 8, 8, 1376, 256, 1, 16, 1e4, 1e-5)
    if eng is None:
        assert f is None
    else:
        assert f is not None and f.NumWeights() == 14
        f.Close()


def test_host_worker_pool_is_safe_under_concurrent_callers():
    """The library's host loops share one set of worker threads, one parallel region at a time.
    Several Python threads (ctypes drops the GIL) quantizing matrices of very different sizes at
    once must each get exactly what a lone caller gets."""
    import threading
    mats = [(rng.standard_normal((r, 256)) * 0.02).astype(np.float32) for r in (1, 3, 17, 64, 300, 1000)]
    want = [(E.quantize_q8(m, 0), E.quantize_q4_0(m)) for m in mats]
    bad = []

    def worker(seed):
        for it in range(60):
            i = (seed + it) % len(mats)
            q, s = E.quantize_q8(mats[i], 0)
            b = E.quantize_q4_0(mats[i])
            if not (np.array_equal(q, want[i][0][0]) and np.array_equal(s, want[i][0][1]) and np.array_equal(b, want[i][1])):
                bad.append((seed, it))

    ths = [threading.Thread(target=worker, args=(k,)) for k in range(6)]
    for t in ths:
        t.start()
    for t in ths:
        t.join()
    assert not bad, bad[:5]


def test_buffers_of_another_type_are_refused():
    """A pointer to ints where the library takes floats is an error of the call, not an address to read from."""
    w, q, sc = np.ones((1, 32), np.float32), np.empty((1, 32), np.int8), np.empty(1, np.float32)
    f, i8 = (lambda a: a.ctypes.data_as(ctypes.POINTER(ctypes.c_float))), (lambda a: a.ctypes.data_as(ctypes.POINTER(ctypes.c_int8)))
    lib.mg_quantize_q8(f(w), 1, 32, 0, i8(q), f(sc))
    assert (q == 127).all()
    for bad in ((i8(q), i8(q), f(sc)), (f(w), f(sc), f(sc)), (w.ctypes.data, i8(q), f(sc))):
        with pytest.raises(ctypes.ArgumentError):
            lib.mg_quantize_q8(bad[0], 1, 32, 0, bad[1], bad[2])


def test_buffers_reach_the_library_whatever_their_kind():
    """Writable, read-only, strided and Fortran-ordered arrays: the same bytes, and the address of a copy only where one has
    to be made."""
    a = np.arange(96, dtype=np.float32).reshape(3, 32) - 40
    want = E.quantize_q8(a)
    ro = a.copy()
    ro.flags.writeable = False
    for v in (ro, np.asfortranarray(a), np.repeat(a, 2, axis=1)[:, ::2]):
        got = E.quantize_q8(v)
        assert (got[0] == want[0]).all() and (got[1] == want[1]).all()

    def read(at, n):
        return bytes((ctypes.c_char * n).from_address(at))

    at, keep = E._addresses([a, None, ro[1:]])
    assert at == [a.ctypes.data, None, ro[1:].ctypes.data] and keep[1] is None
    at, keep = E._addresses([a, None])
    assert at == [a.ctypes.data, None]
    at, keep = E._addresses([a.T, a])
    assert at[1] == a.ctypes.data and read(at[0], a.nbytes) == np.ascontiguousarray(a.T).tobytes()
    assert E._fp(np.empty(0, np.float32)) is not None and E._fp(None) is None


def test_the_benchmark_line_stays_short():
    """A record of every configuration, tables and all, is printed as one line of at most 8,000 characters that still has
    what the line is for."""
    import json
    import bench
    table = [{"launch": "norm2+gate|up+SwiGLU (a launch of the fused path)", "cls": 4, "per_token": 24, "avg_us": 7.123, "share_of_step": 0.2, "bytes": 8755200, "GBps": 1234.5}] * 8
    run = {"start_position": 4000, "steps": 200, "ms_per_step": 0.31234, "tok_per_s": 3201.5, "step_bytes": 8568968192, "step_GBps": 4546.1,
           "step_roofline_frac": 0.5683, "launches": 4, "graph_replay_one_token_a_launch_ms_per_step": 1.89466, "fused_launches_ms_per_step": 2.50344,
           "in_launch_phases": {"phases": table}, "kernels": table, "kernels_fused_launches": table, "tokens_match_fused_launches": True}
    leg = {"tokens": 512, "ms": 15.222, "ms_per_token": 4.303, "host_to_device_GBps": 46.84, "note": "n" * 300}
    conf = {"exec": "e" * 70, "runs": [run, run], "tokens_match": True, "tokens_checked": 48, "tokens_checked_at": "p" * 80, "prefill": leg, "stream": leg}
    out = {"metric": "m", "value": 3201.5, "ms_per_step": 0.31234, "vs_baseline": None, "config": {"workload": "w" * 200}, "roofline": {"kernel": "k" * 700},
           "matvec": {"kernel": "k" * 500}, "kernels": table[:1], "kernels_fused_launches": table, "in_launch_phases": {"phases": table},
           "cpu_baseline": {"sample": "s" * 200}, "prefill": None, "stream": None, "flow_trace": None, "configs": {f"configuration-{i}": conf for i in range(5)}}
    assert len(json.dumps(out)) > 20000
    d = json.loads(json.dumps(bench.digest(out)))
    assert len(json.dumps(d)) < 8000
    assert d["value"] == 3201.5 and d["vs_baseline"] is None and d["roofline"] == out["roofline"]
    assert all(c["runs"][0]["ms_per_step"] == 0.31234 and c["tokens_match"] and c["prefill"]["ms"] == 15.222 for c in d["configs"].values())
