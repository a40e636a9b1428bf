"""Scores of a batched exact prefill where the K magnitudes pick the number of
base-256 digits (three, four, none: the vector units), against one decode step
per token, bit for bit (the score is one integer, whatever the digits)."""
import numpy as np
import pytest

import spkv
from helpers import SMALL, model_files, prompt

pytestmark = pytest.mark.gpu

D3, D4 = 0x7F7F7F, 0x7F7F7F00          # the largest Q16 values of three digits, of four (in f32)


@pytest.mark.parametrize("q16", [D3, D3 + 1, D4, D4 + 256])
@pytest.mark.parametrize("shape", ["qwen3-tiny", "qwen3-hd128", "gemma3-w200", "gemma3-g4hd256w150"])
def test_k_magnitudes_at_the_digits_edges(tmpdir_models, shape, q16):
    spm, spt = model_files(tmpdir_models, shape, max_context=1024)
    d = SMALL[shape]
    m = spkv.Model(spm, spt)
    s = spkv.Session(m, 512)
    qm = spkv.l1().sp_session_qwen3_model(s.h)
    V, kvd = d["vocab"], d["n_kv_heads"] * d["head_dim"]
    pr = prompt(201, V, seed=8)
    out = []
    for batch in (False, True):
        b = spkv.Backend(qm, 512, exact=True, batch_prefill=batch)
        b.prefill(pr[:99])
        for l in range(d["n_layers"]):
            for at, sign in ((3, 1), (70, -1), (98, 1)):
                k, v = b.read_kv(l, at, 1, kvd)
                k[0, (7 * at) % kvd] = sign * q16 / 65536.0
                b.write_kv(l, at, k, v)
        b.prefill(pr[99:200])
        lg = np.zeros(V, np.float32)
        kv = [b.read_kv(l, 99, 101, kvd) for l in range(d["n_layers"])]
        b.decode(int(pr[200]), lg)
        out.append([lg] + [x for p in kv for x in p])
        b.close()
    for x, y in zip(*out):
        assert np.array_equal(x.view(np.uint32), y.view(np.uint32))
    s.close(); m.close()
