"""The token and value beside a step's logits come from a key the output
kernel forms; they must be what a scan of the returned row finds (first value
greater than all before it, from -inf): ties, rows that are NaN or -inf, all
output formats, decode and prefill."""
import ctypes as C

import numpy as np
import pytest

from flarellm_amd import FL_F32, FL_KV_F16, FL_Q4K, FL_Q6K, FL_Q8_0
from flarellm_amd import synth as S
from flarellm_amd._lib import check

pytestmark = pytest.mark.gpu


def _scan(logits):
    bi, bv = 0, -np.inf
    ok = np.where(np.isnan(logits), -np.inf, logits)
    if ok.max() > -np.inf:
        bi = int(np.argmax(ok))
        bv = float(logits[bi])
    return bi, bv


def _step(b, tok, pos):
    out = np.empty(b.spec.vocab, np.float32)
    t, v = C.c_int32(), C.c_float()
    check(b.lib.fl_decode_step(b.ctx, tok, pos, out.ctypes.data, C.byref(t), C.byref(v)), b.ctx)
    return out, t.value, v.value


@pytest.mark.parametrize("layer,embed,output", [(FL_Q8_0, FL_Q8_0, None), (FL_Q8_0, FL_Q8_0, FL_Q8_0),
                                                (FL_Q4K, FL_Q6K, FL_Q6K), (FL_Q4K, FL_Q4K, FL_Q4K),
                                                (FL_Q8_0, FL_F32, FL_F32)])
def test_key_is_the_scan(backend, layer, embed, output):
    print(f"[key] layer={layer} embed={embed} output={output}", flush=True)
    spec = S.tiny_spec(layer, embed_fmt=embed, output_fmt=output, vocab=513)
    model = S.make_model(spec, seed=3)
    w = model.output if model.output is not None else model.embedding
    rows = w.data.reshape(spec.vocab, -1)
    rows[256:] = rows[1:258]  # every logit from 256 on ties with an earlier one
    backend.init_gpu_kv_cache(spec, FL_KV_F16)
    backend.upload_weights_to_gpu(model)
    for pos, tok in enumerate([5, 130, 7]):
        logits, t, v = _step(backend, tok, pos)
        assert (t, v) == _scan(logits)
    logits, t, v = backend.forward_prefill(np.array([5, 130, 7] * 30, np.uint32), 0)
    assert (t, v) == _scan(logits)


def test_key_skips_what_is_not_a_number(backend):
    spec = S.tiny_spec(FL_Q8_0, output_fmt=FL_F32, vocab=300)
    model = S.make_model(spec, seed=4)
    out = model.output.data.view(np.float32).reshape(spec.vocab, -1)
    backend.init_gpu_kv_cache(spec, FL_KV_F16)
    for case in ("some nan", "nan but one", "all nan"):
        if case == "some nan":
            out[::3] = np.nan
        elif case == "nan but one":
            keep = out[100].copy()
            out[:] = np.nan
            out[100] = keep
        else:
            out[:] = np.nan
        backend.upload_weights_to_gpu(model)
        logits, t, v = _step(backend, 9, 0)
        assert np.isnan(logits).any() and (t, v) == _scan(logits), case


def test_replayed_logits_steps_match_the_first(backend):
    """Steps with logits replay a graph after the first 8: every one of 40
    against the same step enqueued directly (FL_OPT_EXACT off and on drops the
    graph), with other work and synchronizations between."""
    from flarellm_amd import _lib as L

    spec = S.tiny_spec(FL_Q8_0, vocab=700)
    backend.init_gpu_kv_cache(spec, FL_KV_F16)
    backend.upload_weights_to_gpu(S.make_model(spec, seed=6))
    toks = S.random_tokens(8, 40, spec.vocab).tolist()
    want = []
    for pos, t in enumerate(toks):
        backend.set_option(L.FL_OPT_EXACT, 1)
        backend.set_option(L.FL_OPT_EXACT, 0)  # drops captured graphs: this step is enqueued
        want.append(_step(backend, t, pos))
    backend.reset()
    for pos, t in enumerate(toks):
        logits, tok, val = _step(backend, t, pos)
        assert np.array_equal(logits.view(np.uint32), want[pos][0].view(np.uint32)) and (tok, val) == want[pos][1:]
        backend.forward_greedy(t, pos)  # the greedy step's own graph, same slot
        backend.sync()
