"""The launch-plan cache of flame_sdpa_chunked_bf16 on the GPU: a miss measures both query tiles and stores the
faster, the next call of the shape is a hit, masked problems have one tile and skip the measurement, a forced tile
and a cache file carried from one process to the next behave as the reference documents them
(cuda/src/flame_sdpa_stub.cu:1080-1379).  The output is checked against the oracle whichever tile runs.  The
environment is read once per process, so the cases that set it run in processes of their own."""
import ctypes
import json
import os
import subprocess
import sys

import numpy as np
import pytest
import torch

from flame_amd import workloads as W
from tests.gpu_util import assert_close_bf16, to_dev, to_f32
from tests.test_plan_cache_file import FIELDS, ROOT

pytestmark = pytest.mark.gpu


class Stats(ctypes.Structure):
    _fields_ = [(f, ctypes.c_uint64) for f in FIELDS]


def _stats(lib):
    st = Stats()
    assert lib.flame_sdpa_autotune_get_stats(ctypes.byref(st)) == 0
    return {f: getattr(st, f) for f in FIELDS}


def _p(t):
    return ctypes.c_void_p(0 if t is None else t.data_ptr())


def _chunked(lib, q, k, v, out, scale, causal=0, mask=None, mask_heads=1):
    B, H, Q, D = q.shape
    K = k.shape[2]
    lib.flame_sdpa_chunked_bf16.restype = ctypes.c_int
    rc = lib.flame_sdpa_chunked_bf16(_p(q), _p(k), _p(v), B, H, Q, K, D, D, ctypes.c_float(scale), 64, causal, mask_heads,
                                     _p(mask), _p(out), None, ctypes.c_uint64(0),
                                     ctypes.c_void_p(torch.cuda.current_stream().cuda_stream))
    torch.cuda.synchronize()
    return rc


def test_miss_measures_hit_reuses_mask_skips(oracle):
    from flame_amd import capi
    lib = capi.lib()
    B, H, Q, K, D = 2, 5, 512, 320, 64
    print(f"[plan] {B}x{H} Q={Q} K={K} D={D}", flush=True)
    t = [W.f32_to_bf16_bits(W.normal_f32(911, s, B * H * n * D).reshape(B, H, n, D)) for s, n in enumerate((Q, K, K))]
    q, k, v = (to_dev(x) for x in t)
    out = torch.empty_like(q)
    ro, _, ro32 = oracle.sdpa_fwd(t[0], t[1], t[2], 0.125, want_f32=True)
    lib.flame_sdpa_autotune_reset_stats()
    before = _stats(lib)
    assert _chunked(lib, q, k, v, out, 0.125) == 0
    assert_close_bf16(oracle, "O (first call)", to_f32(out), ro, ro32)
    s1 = _stats(lib)
    assert s1["cache_misses"] == 1 and s1["cache_hits"] == 0 and s1["tuned"] == 1 and s1["errors"] == 0
    assert s1["last_plan_source"] == 2 and s1["last_candidate_count"] == 2 and s1["last_best_time_ns"] > 0
    assert s1["last_q_chunk"] in (128, 256) and s1["last_k_chunk"] == 64
    assert s1["cache_entries"] == before["cache_entries"] + 1
    assert (s1["last_shape_b"], s1["last_shape_h"], s1["last_shape_q"], s1["last_shape_k"], s1["last_shape_dh"],
            s1["last_shape_dv"], s1["last_shape_mask_heads"], s1["last_shape_causal"]) == (B, H, Q, K, D, D, 0, 0)
    out.zero_()
    assert _chunked(lib, q, k, v, out, 0.125) == 0
    assert_close_bf16(oracle, "O (second call)", to_f32(out), ro, ro32)
    s2 = _stats(lib)
    assert s2["cache_hits"] == 1 and s2["cache_misses"] == 1 and s2["tuned"] == 1
    assert s2["last_plan_source"] == 1 and s2["last_q_chunk"] == s1["last_q_chunk"]
    # the causal flag is part of the key: another miss
    assert _chunked(lib, q, k, v, out, 0.125, causal=1) == 0
    roc, _, roc32 = oracle.sdpa_fwd(t[0], t[1], t[2], 0.125, causal=True, want_f32=True)
    assert_close_bf16(oracle, "O (causal)", to_f32(out), roc, roc32)
    s3 = _stats(lib)
    assert s3["cache_misses"] == 2 and s3["tuned"] == 2 and s3["last_shape_causal"] == 1
    # a mask leaves one tile: nothing to measure
    keep = (W.normal_f32(912, 0, B * Q * K).reshape(B, 1, Q, K) > -0.5).astype(np.uint8)
    keep[..., 0] = 1
    mask = torch.from_numpy(keep.astype(np.float32)).to(torch.bfloat16).cuda()
    assert _chunked(lib, q, k, v, out, 0.125, mask=mask, mask_heads=1) == 0
    rom, _, rom32 = oracle.sdpa_fwd(t[0], t[1], t[2], 0.125, mask=keep, want_f32=True)
    assert_close_bf16(oracle, "O (mask)", to_f32(out), rom, rom32)
    s4 = _stats(lib)
    assert s4["skipped"] == 1 and s4["tuned"] == 2 and s4["last_plan_source"] == 3 and s4["last_q_chunk"] == 128
    assert s4["last_shape_mask_heads"] == 1


CHILD = r"""
import ctypes, json, sys
sys.path.insert(0, %r)
import numpy as np, torch
from flame_amd import capi, workloads as W
from oracle import oracle as O
from tests.gpu_util import assert_close_bf16, to_dev, to_f32
from tests.test_gpu_plan_cache import _chunked, _stats
lib = capi.lib()
B, H, Q, K, D = 1, 4, 384, 256, 128
t = [W.f32_to_bf16_bits(W.normal_f32(913, s, B * H * n * D).reshape(B, H, n, D)) for s, n in enumerate((Q, K, K))]
q, k, v = (to_dev(x) for x in t)
out = torch.empty_like(q)
assert _chunked(lib, q, k, v, out, 0.09) == 0
ro, _, ro32 = O.sdpa_fwd(t[0], t[1], t[2], 0.09, want_f32=True)
assert_close_bf16(O, "O", to_f32(out), ro, ro32)
assert lib.flame_sdpa_autotune_flush_cache() == 0
print(json.dumps(_stats(lib)))
""" % ROOT


def _child(env_extra, code=CHILD):
    env = {k: v for k, v in os.environ.items() if not k.startswith("FLAME_SDPA_")}
    env.update(env_extra)
    out = subprocess.run([sys.executable, "-c", code], env=env, capture_output=True, text=True, timeout=300, cwd=ROOT)
    assert out.returncode == 0, out.stdout + out.stderr
    return json.loads(out.stdout.strip().splitlines()[-1])


@pytest.mark.parametrize("forced,ran,clamped", [("256", 256, 0), ("128", 128, 0), ("100", 128, 1), ("4096", 256, 1)])
def test_forced_tile(forced, ran, clamped):
    print(f"[plan] FLAME_SDPA_QCHUNK={forced}", flush=True)
    s = _child({"FLAME_SDPA_QCHUNK": forced})
    assert s["env_forced"] == 1 and s["clamped"] == clamped and s["last_plan_source"] == 4 and s["last_q_chunk"] == ran
    assert s["cache_hits"] == 0 and s["cache_misses"] == 0 and s["tuned"] == 0


def test_switched_off_takes_the_rule_and_counts_nothing():
    s = _child({"FLAME_SDPA_AUTOTUNE": "0"})
    assert s["cache_hits"] == 0 and s["cache_misses"] == 0 and s["tuned"] == 0 and s["cache_entries"] == 0
    assert s["last_plan_source"] == 3 and s["last_q_chunk"] == 128          # 12 workgroups of 128 rows: far from filling the chip


def test_cache_file_carries_a_plan_to_the_next_process(tmp_path):
    path = str(tmp_path / "sub" / "dir" / "plans.json")
    env = {"FLAME_SDPA_AUTOTUNE_CACHE": path, "FLAME_SDPA_AUTOTUNE_PERSIST": "1"}
    s1 = _child(env)
    assert s1["tuned"] == 1 and s1["cache_saved"] == 1 and s1["cache_entries"] == 1 and s1["last_plan_source"] == 2
    lines = open(path).read().splitlines()
    meta = json.loads(lines[0])["meta"]
    assert meta["version"] == 1 and meta["arch"].startswith("gfx950")
    entry = json.loads(lines[1])
    assert entry["key"] == {"B": 1, "H": 4, "Q": 384, "K": 256, "Dh": 128, "Dv": 128, "mask_heads": 0, "causal": 0}
    assert entry["plan"] == {"q": s1["last_q_chunk"], "k": 64}
    s2 = _child(env)
    assert s2["cache_loads"] == 1 and s2["cache_hits"] == 1 and s2["tuned"] == 0 and s2["last_plan_source"] == 1
    assert s2["last_q_chunk"] == s1["last_q_chunk"] and s2["cache_saved"] == 0      # nothing new to write


# O lies between two margins in a buffer of its own: nothing outside it may be written, and every row of it is
CHILD_MARGINS = CHILD.replace("B, H, Q, K, D = 1, 4, 384, 256, 128", "B, H, Q, K, D = %d, %d, %d, %d, %d").replace(
    "out = torch.empty_like(q)",
    "m = 256 * D; buf = torch.full((q.numel() + 2 * m,), 77.0, dtype=q.dtype, device=q.device); out = buf[m:-m].view(q.shape)").replace(
    "assert lib.flame_sdpa_autotune_flush_cache() == 0", "assert (buf[:m] == 77).all() and (buf[-m:] == 77).all()")


@pytest.mark.parametrize("forced", ["", "256"])
@pytest.mark.parametrize("B,H,Q,K,D", [(1, 16, 4224, 64, 64),       # 272 units of 256 queries, 33 tiles of 128 per head
                                       (1, 24, 2944, 128, 128),     # 288 units, 23 tiles of 128
                                       (1, 17, 4096, 64, 64)])      # 272 units, whole: the last 16 run as 32-query ones
def test_256_row_plan_past_one_round(forced, B, H, Q, K, D):
    """A plan of 256 rows where the rule would not take them (an odd count of 128-query tiles), on more workgroups than
    compute units: measured on a miss, and forced."""
    print(f"[plan] {B}x{H} Q={Q} K={K} D={D} forced={forced!r}", flush=True)
    s = _child({"FLAME_SDPA_QCHUNK": forced} if forced else {}, CHILD_MARGINS % (B, H, Q, K, D))
    assert s["errors"] == 0 and s["last_q_chunk"] in ((256,) if forced else (128, 256))
    assert s["tuned"] == (0 if forced else 1)


# what runs is what the plan says: a 256-row workgroup has 8 wavefronts where something is excluded, a 128-row one 4
CHILD_RUNS = CHILD.replace("B, H, Q, K, D = 1, 4, 384, 256, 128", "B, H, Q, K, D, causal = %d, %d, %d, %d, %d, %d").replace(
    "_chunked(lib, q, k, v, out, 0.09)", "_chunked(lib, q, k, v, out, 0.09, causal)").replace("0.09, want_f32", "0.09, causal=bool(causal), want_f32").replace(
    "print(json.dumps(_stats(lib)))", r"""
st = _stats(lib)
from tests.gpu_util import recorded_launches
def call():
    p = lambda t: ctypes.c_void_p(t.data_ptr())
    assert lib.flame_sdpa_chunked_bf16(p(q), p(k), p(v), B, H, Q, K, D, D, ctypes.c_float(0.09), 64, causal, 1, None, p(out), None,
                                       ctypes.c_uint64(0), ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)) == 0
st["launches"] = [x[1:] for x in recorded_launches(call)]
print(json.dumps(st))""")


@pytest.mark.parametrize("B,H,Q,K,D,causal", [(1, 4, 384, 256, 64, 1), (2, 3, 300, 200, 40, 0), (1, 4, 384, 200, 96, 1), (1, 3, 500, 320, 128, 1)])
@pytest.mark.parametrize("forced,lanes", [("256", 512), ("128", 256)])
def test_forced_tile_is_the_one_that_runs(B, H, Q, K, D, causal, forced, lanes):
    print(f"[plan] {B}x{H} Q={Q} K={K} D={D} causal={causal} FLAME_SDPA_QCHUNK={forced}", flush=True)
    s = _child({"FLAME_SDPA_QCHUNK": forced}, CHILD_RUNS % (B, H, Q, K, D, causal))
    assert s["last_q_chunk"] == int(forced) and s["clamped"] == 0
    assert s["launches"] == [[-(-Q // int(forced)) * B * H, lanes]]


def test_a_stored_plan_of_256_rows_is_the_one_that_runs(tmp_path):
    f = tmp_path / "plans.json"
    f.write_text('{"meta":{"version":1}}\n{"key":{"B":1,"H":4,"Q":384,"K":256,"Dh":64,"Dv":64,"mask_heads":0,"causal":1},"plan":{"q":256,"k":64}}\n')
    s = _child({"FLAME_SDPA_AUTOTUNE_CACHE": str(f)}, CHILD_RUNS % (1, 4, 384, 256, 64, 1))
    assert s["last_plan_source"] == 1 and s["last_q_chunk"] == 256 and s["launches"] == [[8, 512]]


@pytest.mark.parametrize("B,H,Q,K,D,causal,rows", [(1, 36, 2048, 256, 128, 1, 128),      # 288 units of 256 queries: a thin last round
                                                   (1, 32, 2048, 256, 128, 1, 256),      # a whole one
                                                   (1, 32, 2048, 256, 64, 1, 128), (1, 32, 2048, 200, 64, 0, 128)])
def test_the_rule_is_that_of_a_call_without_a_plan(B, H, Q, K, D, causal, rows):
    print(f"[plan] rule {B}x{H} Q={Q} K={K} D={D} causal={causal}", flush=True)
    code = (CHILD_RUNS % (B, H, Q, K, D, causal)).replace("print(json.dumps(st))", r"""
st["plain_call"] = [x[1:] for x in recorded_launches(lambda: capi.attn_fwd(q, k, v, 0.09, causal=bool(causal), out=out))]
print(json.dumps(st))""")
    s = _child({"FLAME_SDPA_AUTOTUNE": "0"}, code)
    assert s["last_q_chunk"] == rows and s["launches"] == s["plain_call"] == [[-(-Q // rows) * B * H, 512 if rows == 256 else 256]]
