"""Float-mode attention of a batched prefill (128 token-heads per workgroup, 32
positions per tile, positions split over workgroups) against one decode step per
token, at the edges of its tiles and splits.

Bound: both paths sum n <= 560 f32 products per score or output in other orders,
each sum off by at most n 2^-24 = 3.3e-5 of its terms' magnitude (in practice a
few 1e-7); the K/V of later layers and the logits inherit it: 1e-4."""
import numpy as np
import pytest

import spkv
from helpers import SMALL, model_files, prompt

pytestmark = pytest.mark.gpu


def close(a, b):
    return np.isfinite(a).all() and np.abs(a.astype(np.float64) - b).max() <= 1e-4 * np.abs(b).max()


# head_dim 64, 128, 256 x 2 and 4 q heads per kv head, full context and windows
SHAPES = ["qwen3-tiny", "gemma3-tiny", "qwen3-hd128", "qwen3-g4", "gemma3-hd256", "gemma3-w200",
          "gemma3-g4w130", "gemma3-g4hd256w150", "gemma3-g4hd64w150", "gemma3-w1"]


@pytest.mark.parametrize("shape", SHAPES)
def test_prefill_equals_decode_steps(tmpdir_models, shape):
    spm, spt = model_files(tmpdir_models, shape, max_context=1024)
    d = SMALL[shape]
    m = spkv.Model(spm, spt)
    s = spkv.Session(m, 1024)
    qm = spkv.l1().sp_session_qwen3_model(s.h)
    V, kvd = d["vocab"], d["n_kv_heads"] * d["head_dim"]
    pr = prompt(561, V, seed=11)
    one = spkv.Backend(qm, 640, batch_prefill=False)
    one.prefill(pr[:560])
    ref = [one.read_kv(l, 0, 560, kvd) for l in range(d["n_layers"])]
    lg0, lg1 = np.zeros(V, np.float32), np.zeros(V, np.float32)
    one.decode(int(pr[560]), lg0)
    # whole passes and ragged ones, each call starting where the last ended
    for cuts in ([560], [1, 31, 32, 33, 63, 400], [129, 431]):
        b = spkv.Backend(qm, 640)
        at = 0
        for n in cuts:
            b.prefill(pr[at:at + n])
            at += n
        for l, (k, v) in enumerate(ref):
            kb, vb = b.read_kv(l, 0, 560, kvd)
            assert close(kb, k) and close(vb, v), (cuts, l)
        b.decode(int(pr[560]), lg1)
        assert close(lg1, lg0) and int(lg1.argmax()) == int(lg0.argmax()), cuts
        b.close()
    one.close(); s.close(); m.close()


def test_rows_outside_the_window_do_not_reach_it(tmpdir_models):
    """A V row that is not finite, in a tile the pass reads but outside every
    window, changes nothing (its weight is zero, not zero times infinity)."""
    spm, spt = model_files(tmpdir_models, "gemma3-tiny")
    m = spkv.Model(spm, spt)
    s = spkv.Session(m, 128)
    qm = spkv.l1().sp_session_qwen3_model(s.h)
    V, kvd = 1000, 128
    pr = prompt(62, V, seed=4)
    out = []
    for batch in (True, False):
        b = spkv.Backend(qm, 128, batch_prefill=batch)
        b.prefill(pr[:21])
        for l in (0, 3):                                # window layers: 16 positions
            k, v = b.read_kv(l, 5, 1, kvd)
            v[:] = np.inf
            b.write_kv(l, 5, k, v)
        b.prefill(pr[21:61])
        lg = np.zeros(V, np.float32)
        b.decode(int(pr[61]), lg)
        out.append(lg)
        b.close()
    assert close(out[0], out[1])
    s.close(); m.close()
