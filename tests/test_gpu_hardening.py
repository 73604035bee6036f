"""Failure handling of the device path, forced from the host so that every
kernel still runs to completion:

* the split-K linears' XCD placement: a wrong XCD count (``DRT_N_XCC``) makes
  the kernels' own placement check fire; the forward finishes and the host
  raises, and the GPU is then fine for a new runtime;
* the fenced split-K exchange (``DRT_SPLITK_FENCED=1``, what a runtime falls
  back to when its placement probe fails) gives bit-identical results;
* the scores and tokens of a q4 canvas, bit for bit;
* hardware queues that come into being after a runtime and move where its stream's
  work-groups land: the same results as before;
* a placement report of a rotation that the stream has taken (``DRT_PLACEMENT_WORD``) is
  settled, and what a block queued behind it reported meanwhile is not lost;
* the fp16 range of the activations: a first-layer norm weight that pushes the
  normalized activation past 65504 raises the range error, one that keeps it
  near 4e4 (checked on the CPU) does not.
"""
from __future__ import annotations

import os
import subprocess
import sys

import numpy as np
import pytest

from oracle import ops as O

from helpers import tiny_geometry

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu


def _say(*a):
    print("[case]", *a, flush=True)


def _propose(model, env=None):
    from diffusorrt_amd.runtime import Runtime, bd3_session_config

    env = env or {}
    saved = {k: os.environ.get(k) for k in env}
    os.environ.update(env)
    try:
        rt = Runtime(model, max_forward_rows=256, max_positions=512)
    finally:
        for k, v in saved.items():
            if v is None:
                os.environ.pop(k, None)
            else:
                os.environ[k] = v
    g = model.geometry
    x = list(range(64)) + [g.mask_token_id] * 32
    try:
        with rt.session(bd3_session_config(32, 8, len(x))) as s:
            s.start_device(x, prompt_len=0, block_size=32, mask_token_id=g.mask_token_id,
                           exact_kv=False, steps=8)
            return s.propose_device(list(range(64, 96)), window_end=96, frozen_prefix=64)
    finally:
        rt.close()


def test_wrong_xcd_count_raises_and_the_gpu_stays_usable():
    from diffusorrt_amd import synthetic as syn

    _say("placement error path: DRT_N_XCC=4 on an 8-XCD part")
    model = syn.build_model(tiny_geometry(), "q4", seed=51)
    with pytest.raises(RuntimeError, match="unexpected XCD"):
        _propose(model, {"DRT_N_XCC": "4"})
    scores, tokens, _ = _propose(model)  # a fresh runtime on the same GPU works
    assert np.isfinite(scores).all() and len(tokens) == 32


def test_fenced_split_k_exchange_is_bit_identical():
    from diffusorrt_amd import synthetic as syn

    _say("fenced split-K exchange")
    model = syn.build_model(tiny_geometry(), "q4", seed=52)
    s0, t0, f0 = _propose(model)
    s1, t1, f1 = _propose(model, {"DRT_SPLITK_FENCED": "1"})
    assert (t1, f1) == (t0, f0)
    assert np.array_equal(np.asarray(s1), np.asarray(s0))


# Scores and tokens of a q4 canvas, bit for bit as they always were: every fp32 sum of such a
# forward is cut along K where the shape says (big_q4_shape_plan) and its probabilities are
# rounded one way (attn_split_tile), whatever the kernels' tiles and launches. Otherwise a row
# whose two best logits are all but equal takes its other token. 512 rows attend in two key
# ranges (met in one work-group), 257 in four, 100 in more; the gate|up projection stays below
# two work-groups per CU, where nothing depends on the process's hardware queues.
_CANVAS_DIGESTS = {100: "f94f169c64e44037", 257: "bfa80cbd6e0fcbd8", 512: "0738386d73833c8b"}


@pytest.mark.parametrize("n", sorted(_CANVAS_DIGESTS))
def test_canvas_results_are_bit_stable(n):
    import hashlib

    from diffusorrt_amd import synthetic as syn
    from diffusorrt_amd.runtime import Runtime, fixed_quota_session_config

    from helpers import tiny_dream_geometry

    _say("canvas bits", n)
    g = tiny_dream_geometry(hidden_size=1024, intermediate_size=3072, num_heads=14, num_kv_heads=2,
                            vocab_size=4096)
    rt = Runtime(syn.build_model(g, "q4", seed=55), max_forward_rows=512, max_positions=512)
    toks = [(7 * i) % 900 for i in range(n - n // 2)] + [g.mask_token_id] * (n // 2)
    with rt.session(fixed_quota_session_config(64, 64, n)) as s:
        s.start_device(toks, prompt_len=n - n // 2, block_size=64, mask_token_id=g.mask_token_id,
                       exact_kv=False, steps=8)
        scores, tokens, _ = s.propose_device(list(range(n - n // 2, n)), window_end=n,
                                             frozen_prefix=0)
    rt.close()
    h = hashlib.sha256(np.asarray(scores, dtype="<f8").tobytes() +
                       np.asarray(tokens, dtype="<i4").tobytes()).hexdigest()[:16]
    assert h == _CANVAS_DIGESTS[n]


def test_a_settled_rotation_keeps_other_reports():
    from diffusorrt_amd import synthetic as syn

    model = syn.build_model(tiny_geometry(), "q4", seed=56)
    s0, t0, f0 = _propose(model)

    def outcome(word, seen=1, count=0):
        try:
            s, t, f = _propose(model, {"DRT_PLACEMENT_WORD": f"{seen},{word},{count}"})
        except RuntimeError as e:
            return str(e)
        assert (t, f) == (t0, f0) and np.array_equal(np.asarray(s), np.asarray(s0))
        return "settled"

    _say("settled rotation, and other reports")  # 1: a report of the stream's rotation
    assert outcome(1) == "settled"
    for bit, text in ((2, "bounded wait"), (4, "fp16 range")):  # reported after the host looked
        assert text in outcome(1 | bit)
    two = 1 | 1 << 8 | 1 << 9  # two rotations
    assert "unexpected XCD" in outcome(two)
    assert "unexpected XCD" in outcome(two | 4)
    assert "unexpected XCD" in outcome(1, count=1)  # slices of one block counted on two XCDs


_LATER_QUEUES = """
import sys
sys.path[:0] = [%r, %r]
import numpy as np, torch
from diffusorrt_amd import synthetic as syn
from diffusorrt_amd.runtime import Runtime, bd3_session_config
from helpers import tiny_geometry
model = syn.build_model(tiny_geometry(), "q4", seed=54)
g = model.geometry
rt = Runtime(model, max_forward_rows=256, max_positions=512)
x = list(range(64)) + [g.mask_token_id] * 32
with rt.session(bd3_session_config(32, 8, len(x))) as s:
    s.start_device(x, prompt_len=0, block_size=32, mask_token_id=g.mask_token_id,
                   exact_kv=False, steps=8)
    def once():
        return s.propose_device(list(range(64, 96)), window_end=96, frozen_prefix=64)[:2]
    first = [once() for _ in range(3)]  # eager, captured, replayed
    streams = [torch.cuda.Stream() for _ in range(8)]
    for st in streams:
        with torch.cuda.stream(st):
            torch.zeros(1, device="cuda")
    torch.cuda.synchronize()
    later = [once() for _ in range(3)]
assert all(np.array_equal(np.asarray(a[0]), np.asarray(first[0][0])) and a[1] == first[0][1]
           for a in first + later)
rt.close()
print("same")
"""


def test_queues_created_after_the_runtime():
    _say("later hardware queues")
    here = os.path.dirname(os.path.abspath(__file__))
    out = subprocess.run([sys.executable, "-c", _LATER_QUEUES % (os.path.dirname(here), here)],
                         capture_output=True, text=True, timeout=100)
    assert out.returncode == 0 and out.stdout.strip().endswith("same"), out.stdout + out.stderr


def test_fp16_range_flag():
    from diffusorrt_amd import synthetic as syn

    g = tiny_geometry(layer_count=1)
    ids = list(range(64)) + [g.mask_token_id] * 32

    def with_norm_weight(w):
        model = syn.build_model(g, "q4", seed=53)
        model.weights["model.layers.0.input_layernorm.weight"] = torch.full(
            (g.hidden_size,), w, dtype=torch.bfloat16)
        emb = model.weights["model.embed_tokens.weight"].float().numpy()[ids]
        ones = np.ones(g.hidden_size, np.float32)
        peak = np.abs(O.rms_norm(emb, ones, g.rms_norm_eps)).max() * float(
            torch.tensor(w, dtype=torch.bfloat16).float())
        return model, peak

    near, peak = with_norm_weight(1.0e4)
    _say(f"fp16 range: first-layer activation peak {peak:.3g} (in range)")
    assert 2e4 < peak < 6e4  # the CPU check: near, but inside the fp16 range
    scores, _, _ = _propose(near)
    assert np.isfinite(scores).all()
    over, peak = with_norm_weight(1.0e5)
    _say(f"fp16 range: first-layer activation peak {peak:.3g} (beyond 65504)")
    assert peak > 65504
    with pytest.raises(RuntimeError, match="fp16 range"):
        _propose(over)
