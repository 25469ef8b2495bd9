"""Many-query attention (k_attw): prefill_attention_gpu at the edges of its
tiles (32 queries per item, 4 items per workgroup, 64 keys per iteration), and
wide prefill passes against the same prompt in short ones."""
import numpy as np
import pytest

from flarellm_amd import FL_KV_F16, FL_KV_F32, FL_KV_Q8, FL_Q4K, FL_Q6K, FL_Q8_0
from flarellm_amd import _lib as L
from flarellm_amd import synth as S
from flarellm_amd._lib import check

pytestmark = pytest.mark.gpu


def _reference(q, k, v, nh, nkv, hd):
    """float64 causal attention and sum_t p_t |v_t| of each output."""
    T, g = q.shape[0], nh // nkv
    q, k, v = (a.astype(np.float64).reshape(T, -1, hd) for a in (q, k, v))
    out, mag = np.empty_like(q), np.empty_like(q)
    top = np.zeros((T, nh, 1))
    for h in range(nh):
        s = q[:, h] @ k[:, h // g].T / np.sqrt(hd)
        s[np.triu_indices(T, 1)] = -np.inf
        p = np.exp(s - s.max(1, keepdims=True))
        p /= p.sum(1, keepdims=True)
        out[:, h], mag[:, h] = p @ v[:, h // g], p @ np.abs(v[:, h // g])
        top[:, h, 0] = np.where(np.isfinite(s), np.abs(s), 0).max(1)
    return out.reshape(T, -1), mag.reshape(T, -1), np.repeat(top, hd, 2).reshape(T, -1)


def _check(backend, nh, nkv, hd, T, edit=None):
    import torch

    print(f"[attw] heads={nh}/{nkv} D={hd} T={T}", flush=True)
    q = S.normal(T + hd, 0, T * nh * hd).reshape(T, -1)
    k = S.normal(T + hd, 1 << 40, T * nkv * hd).reshape(T, -1)
    v = S.normal(T + hd, 2 << 40, T * nkv * hd).reshape(T, -1)
    if edit is not None:
        edit(q, k, v)
    got = backend.prefill_attention_gpu(*(torch.from_numpy(a).cuda() for a in (q, k, v)), T, nh, nkv, hd).cpu().numpy()
    want, mag, top = _reference(q, k, v, nh, nkv, hd)
    # a score's error is at most ~(hd + 16) 2^-24 of |q||k| <= the largest
    # |score| here times sqrt(hd); p's relative error is the same absolute
    # amount, and the sums over T keys add sqrt(T) 2^-24
    sq = np.linalg.norm(q.reshape(T, nh, hd).astype(np.float64), axis=2).max() * \
        np.linalg.norm(k.reshape(T, nkv, hd).astype(np.float64), axis=2).max() / np.sqrt(hd)
    bound = (4 * np.sqrt(hd) * sq + 4 * np.sqrt(T) + 16) * 2.0 ** -24 * mag
    assert (np.abs(got - want) <= bound + 1e-30).all(), float((np.abs(got - want) / (bound + 1e-30)).max())


@pytest.mark.parametrize("nh,nkv,hd", [(1, 1, 64), (6, 3, 128), (9, 3, 64), (16, 4, 128), (16, 2, 64), (8, 1, 128)])
@pytest.mark.parametrize("T", [1, 31, 32, 33, 64, 65, 97, 129, 300])
def test_edges(backend, nh, nkv, hd, T):
    _check(backend, nh, nkv, hd, T)


@pytest.mark.parametrize("hd", [64, 128])
def test_values(backend, hd):
    """Zero queries (a plain mean), large scores (one key takes all), values of
    very different size."""

    def edit(q, k, v):
        q[3] = 0.0
        q[40:50] *= 30.0
        v[::7] *= 1e4
        v[5] *= 1e-6

    _check(backend, 8, 2, hd, 100, edit)


@pytest.fixture
def workspace(backend):
    """Sets the most MiB of workspace; no limit again afterwards."""
    yield lambda mib: backend.set_option(L.FL_OPT_WORKSPACE_MIB, mib)
    backend.set_option(L.FL_OPT_WORKSPACE_MIB, -1)


@pytest.mark.parametrize("mib", [1, 0])
@pytest.mark.parametrize("nh,nkv,hd,T", [(9, 3, 64, 700), (16, 8, 128, 300), (1, 1, 64, 31)])
def test_little_workspace(backend, workspace, mib, nh, nkv, hd, T):
    """Kv heads in pieces (1 MiB holds two or three heads here), and without a
    workspace at all."""
    workspace(mib)
    _check(backend, nh, nkv, hd, T)


def test_workspace_is_bounded(backend, workspace):
    """375 MiB of operand planes: in two pieces (256 MiB are kept at most), the
    same bits as in pieces of 5 heads."""
    import torch

    T, n, hd = 8000, 32, 128
    print(f"[attw] {T} tokens of {n} kv heads", flush=True)
    g = torch.Generator(device="cuda").manual_seed(1)
    q, k, v = (torch.randn(T, n * hd, device="cuda", generator=g) for _ in range(3))
    torch.cuda.synchronize()
    workspace(0)  # (frees what earlier tests left)
    workspace(-1)
    free = torch.cuda.mem_get_info()[0]
    want = backend.prefill_attention_gpu(q, k, v, T, n, n, hd)
    torch.cuda.synchronize()
    assert free - torch.cuda.mem_get_info()[0] <= (256 << 20) + want.numel() * 4 + (32 << 20)
    workspace(64)
    got = backend.prefill_attention_gpu(q, k, v, T, n, n, hd)
    assert torch.equal(got, want)


@pytest.mark.parametrize("hd", [64, 128])
@pytest.mark.parametrize("mib", [-1, 0])  # k_attw, the kernels without a workspace
@pytest.mark.parametrize("j", [0, 40, 70, 99])
@pytest.mark.parametrize("what", ["v nan", "v inf", "k inf", "k nan", "k large", "q inf", "all"])
def test_not_finite(backend, workspace, hd, mib, j, what):
    """Values that are not finite at position j: every earlier token keeps its
    bits, later ones get what the formula gives (an Inf score of -Inf is a key
    of no weight, a visible Inf value an Inf), other channels and heads stay."""
    import torch

    print(f"[attw] D={hd} {what} at {j}, workspace {mib}", flush=True)
    T, nh, nkv = 200, 6, 2
    workspace(mib)
    q = S.normal(hd, 0, T * nh * hd).reshape(T, nh, hd)
    k = S.normal(hd, 1 << 40, T * nkv * hd).reshape(T, nkv, hd)
    v = S.normal(hd, 2 << 40, T * nkv * hd).reshape(T, nkv, hd)

    def run():
        args = (torch.from_numpy(a.reshape(T, -1)).cuda() for a in (q, k, v))
        return backend.prefill_attention_gpu(*args, T, nh, nkv, hd).cpu().numpy().reshape(T, nh, hd)

    clean = run()
    if what in ("v nan", "all"):
        v[j, 0, 3] = np.nan
    if what in ("v inf", "all"):
        v[j, 1, [0, 9, 40]] = np.inf, -np.inf, np.nan
    if what == "k inf":
        k[j, 0, 5], k[j, 1, 6] = np.inf, -np.inf
    if what in ("k nan", "all"):
        k[j, 0, 1] = np.nan
    if what == "k large":  # scores beyond the range of f32, of either sign
        k[j, 0, 5], q[:, :, 5] = 3e38, np.where(np.abs(q[:, :, 5]) < 0.1, 0.1, q[:, :, 5]) * 1000
        k[:j, :, 5], k[j + 1:, :, 5] = 0.0, 0.0
    if what == "q inf":
        q[j, 2, 4] = np.inf
    got = run()
    if what != "k large":  # (its queries differ)
        assert np.array_equal(got[:j].view(np.uint32), clean[:j].view(np.uint32))
    with np.errstate(all="ignore"):
        for t in range(j, T):
            for h in range(nh):
                s = (k[:t + 1, h // 3] * q[t, h]).sum(1, dtype=np.float32).astype(np.float64) / np.sqrt(hd)
                p = np.exp(s - np.fmax.reduce(s)) if not np.isposinf(s).any() else s * np.nan
                # a key of no weight takes no part only if its value is a number
                want = (p[:, None] * v[:t + 1, h // 3]).sum(0) / p.sum()
                mag = (p[:, None] * np.abs(v[:t + 1, h // 3])).sum(0) / p.sum()
                ok = np.isfinite(want)
                assert np.array_equal(got[t, h][~ok], want[~ok].astype(np.float32), equal_nan=True), (t, h)
                # f32 scores here and there: their error is an absolute 2^-24
                # times ~sqrt(hd) max|score|, and the weights' relative error
                big = np.abs(s[np.isfinite(s)]).max(initial=1.0)
                bound = (4 * hd * big + 4 * np.sqrt(T) + 16) * 2.0 ** -24 * mag[ok]
                assert (np.abs(got[t, h][ok] - want[ok]) <= bound).all(), (t, h)


@pytest.mark.parametrize("kv", [FL_KV_F16, FL_KV_F32])
@pytest.mark.parametrize("hd", [64, 128])
@pytest.mark.parametrize("pos0,n", [(40, 50), (2000, 40)])
def test_cache_attention_not_finite(backend, kv, hd, pos0, n):
    """Whole and split key ranges: a value row that is not finite is seen by the
    queries from its position on, in its own channels and kv head; slots behind
    the last query by none.  All else keeps its bits."""
    import torch

    print(f"[attw] cache kv={kv} D={hd} {n} at {pos0}, not finite", flush=True)
    T, nh, nkv = pos0 + n, 4, 2
    spec = S.tiny_spec(FL_Q8_0, heads=nh, kv_heads=nkv, head_dim=hd, max_seq=T + 70)
    backend.init_gpu_kv_cache(spec, kv)
    k, v = (S.normal(T, i << 40, spec.max_seq * nkv * hd).reshape(-1, nkv * hd) for i in (1, 2))
    q = torch.from_numpy(S.normal(T, 0, n * nh * hd).reshape(n, -1)).cuda()

    def run():
        backend.gpu_kv_write_batch(0, 0, k, v)
        out = torch.empty(n, nh * hd, device="cuda")
        torch.cuda.synchronize()
        check(backend.lib.fl_gqa_queries_from_cache(backend.ctx, 0, q.data_ptr(), n, pos0, out.data_ptr(), None),
              backend.ctx)
        return out.cpu().numpy()

    clean = run()
    j = n // 2
    k[T:], v[T:] = np.inf, np.nan
    v[pos0 + j, [3, 40]] = np.nan, np.inf  # kv head 0, query heads 0 and 1
    want = clean.copy()
    for h in (0, 1):
        want[j:, h * hd + 3], want[j:, h * hd + 40] = np.nan, np.inf
    got = run()
    ok = np.isfinite(want)
    assert np.array_equal(got[ok].view(np.uint32), clean[ok].view(np.uint32))
    assert np.array_equal(got[~ok], want[~ok], equal_nan=True)


@pytest.mark.parametrize("kv", [FL_KV_F16, FL_KV_Q8, FL_KV_F32])
@pytest.mark.parametrize("hd", [64, 128])
def test_wide_prefill_over_stale_slots(backend, kv, hd):
    """Slots behind the prompt's last token (an earlier sequence's, rejected
    drafts') that are not finite do not reach a wide pass, nor do rows of the
    prompt's own other layers or tokens: the logits keep their bits."""
    print(f"[wide] stale kv={kv} D={hd}", flush=True)
    n = 101
    spec = S.tiny_spec(FL_Q8_0, heads=4, kv_heads=2, head_dim=hd, hidden=512, max_seq=192)
    backend.init_gpu_kv_cache(spec, kv)
    backend.upload_weights_to_gpu(S.make_model(spec, seed=11))
    toks = S.random_tokens(4, n, spec.vocab)
    want = backend.forward_prefill(toks, 0)[0]
    bad = np.full((64, 2 * hd), np.inf, np.float32)
    bad[::2, ::3] = np.nan
    for l in range(spec.layers):
        backend.gpu_kv_write_batch(l, n, bad, bad)
    got = backend.forward_prefill(toks, 0)[0]
    assert np.isfinite(want).all() and np.array_equal(got.view(np.uint32), want.view(np.uint32))


def _records(raw, n, cols):
    """Packed Q8_0 records (csrc/bgemm_args.h) as codes [n][cols] and scales."""
    rec, steps = 19456, (cols + 255) // 256
    raw = raw.reshape((n + 31) // 32, steps, rec)
    codes = raw[:, :, :16384].copy().view(np.float16)  # [tile][step][block][m][h][token][8]
    codes = codes.reshape(-1, steps, 8, 2, 2, 32, 8)[..., [0, 2, 1, 3, 4, 6, 5, 7]]
    codes = codes.transpose(0, 5, 1, 2, 4, 3, 6).reshape(-1, steps * 256)[:n, :cols]
    scale = raw[:, :, 16384:17408].copy().view(np.float32).reshape(-1, steps, 8, 32)
    return codes, scale.transpose(0, 3, 1, 2).reshape(-1, steps * 8)[:n, :cols // 32]


@pytest.mark.parametrize("kv", [FL_KV_F16, FL_KV_Q8, FL_KV_F32])
@pytest.mark.parametrize("nh,nkv,hd", [(2, 2, 64), (4, 2, 128), (9, 3, 64), (16, 4, 128), (16, 2, 64)])
@pytest.mark.parametrize("pos0,n", [(0, 1), (0, 33), (0, 300), (5, 17), (31, 64), (64, 129), (700, 4), (703, 40),
                                    (704, 64), (950, 161), (3000, 17), (5000, 97)])
def test_cache_attention(backend, oracle, kv, nh, nkv, hd, pos0, n):
    """The attention of wide passes over a model's cache, every query against
    float64 over the values that the cache holds; its packed rows hold the
    codes of the rows it returns."""
    import torch

    print(f"[attw] cache kv={kv} heads={nh}/{nkv} D={hd} {n} at {pos0}", flush=True)
    T, spec = pos0 + n, S.tiny_spec(FL_Q8_0, heads=nh, kv_heads=nkv, head_dim=hd, max_seq=pos0 + n + 70)
    backend.init_gpu_kv_cache(spec, kv)
    q = np.concatenate([np.zeros((pos0, nh * hd), np.float32), S.normal(n + hd, 0, n * nh * hd).reshape(n, -1)])
    k, v = (S.normal(T + hd, i << 40, spec.max_seq * nkv * hd).reshape(-1, nkv * hd) for i in (1, 2))
    v[1::7] *= 100.0
    q[pos0 + n // 2] *= 30.0
    backend.gpu_kv_write_batch(1, 0, k, v)  # slots behind the last query are there as well
    k, v = k[:T], v[:T]
    if kv != FL_KV_F32:
        mode = oracle.OR_KV_F16 if kv == FL_KV_F16 else oracle.OR_KV_Q8
        k, v = (a.reshape(T, -1) for a in oracle.kv_view(mode, k.reshape(T, nkv, hd), v.reshape(T, nkv, hd)))
    got = torch.empty(n, nh * hd, device="cuda")
    packed = torch.zeros((n + 31) // 32 * ((nh * hd + 255) // 256) * 19456, dtype=torch.uint8, device="cuda")
    qd = torch.from_numpy(q[pos0:]).cuda()
    torch.cuda.synchronize()
    check(backend.lib.fl_gqa_queries_from_cache(backend.ctx, 1, qd.data_ptr(), n, pos0, got.data_ptr(),
                                                packed.data_ptr()), backend.ctx)
    got = got.cpu().numpy()
    want, mag, _ = _reference(q, k, v, nh, nkv, hd)
    sq = np.linalg.norm(q.reshape(T, nh, hd).astype(np.float64), axis=2).max() * \
        np.linalg.norm(k.reshape(T, nkv, hd).astype(np.float64), axis=2).max() / np.sqrt(hd)
    # the bound of _check, with 2^-22 for the two-part operands of f16 caches
    eps = 2.0 ** (-22 if kv == FL_KV_F16 else -24)
    bound = (4 * np.sqrt(hd) * sq + 4 * np.sqrt(T) + 16) * eps * mag[pos0:]
    err = np.abs(got - want[pos0:])
    assert (err <= bound + 1e-30).all(), float((err / (bound + 1e-30)).max())
    codes, scale = _records(packed.cpu().numpy(), n, nh * hd)
    for t in range(n):
        c, s = oracle.quantize_q8(got[t])
        assert np.array_equal(codes[t].astype(np.int32), c.reshape(-1)) and np.array_equal(scale[t], s.reshape(-1))


@pytest.mark.parametrize("kv", [FL_KV_F16, FL_KV_Q8, FL_KV_F32])
@pytest.mark.parametrize("fmt,hd,pos0,n", [(FL_Q8_0, 64, 0, 65), (FL_Q4K, 128, 37, 200), (FL_Q8_0, 128, 3, 2150)])
def test_wide_prefill_matches_short_passes(backend, kv, fmt, hd, pos0, n):
    """The last token's logits and the cache a wide prefill leaves (through a
    decode step after it) against the same tokens in 16-token calls.  The two
    round differently, and requantized activations turn a last bit into a code
    step: 1 % of the largest logit, as the prefill tests hold the oracle to."""
    print(f"[wide] kv={kv} fmt={fmt} D={hd} pos0={pos0} n={n}", flush=True)
    spec = S.tiny_spec(fmt, embed_fmt=FL_Q6K if fmt == FL_Q4K else None, output_fmt=FL_Q6K if fmt == FL_Q4K else None,
                       heads=4, kv_heads=2, head_dim=hd, hidden=512, max_seq=pos0 + n + 8)
    model = S.make_model(spec, seed=9)
    toks = S.random_tokens(4, pos0 + n, spec.vocab)
    backend.init_gpu_kv_cache(spec, kv)
    backend.upload_weights_to_gpu(model)
    res = []
    for step in (n, 16):
        backend.reset()
        if pos0:
            backend.forward_prefill(toks[:pos0], 0, logits=False)
        for t in range(pos0, pos0 + n, step):
            logits, tok, val = backend.forward_prefill(toks[t:min(t + step, pos0 + n)], t)
        assert tok == int(np.argmax(logits)) and val == logits[tok]
        res.append((logits, backend.forward_single_token_gpu(1, pos0 + n)))
    for a, b in zip(*res):
        assert np.abs(a - b).max() <= 0.01 * np.abs(b).max()


@pytest.mark.parametrize("fmt", [FL_Q8_0, FL_Q4K])
def test_wide_prefill_buffers_grow(backend, fmt):
    """Prompts that get longer, over buffers that grow with them (and hold more
    than a prompt needs): the bits of a model whose first prompt it is."""
    spec = S.tiny_spec(fmt, embed_fmt=FL_Q6K if fmt == FL_Q4K else None, output_fmt=FL_Q6K if fmt == FL_Q4K else None,
                       hidden=512, inter=1536, max_seq=2304)
    model = S.make_model(spec, seed=12)
    toks = S.random_tokens(7, 2200, spec.vocab)
    sizes = [70, 96, 97, 150, 420, 431, 1000, 2048, 2200, 333]
    runs = []
    for fresh in (False, True):
        rows = []
        for i, n in enumerate(sizes):
            if fresh or i == 0:
                backend.init_gpu_kv_cache(spec, FL_KV_F16)
                backend.upload_weights_to_gpu(model)
            print(f"[wide] grow fmt={fmt} n={n} fresh={fresh}", flush=True)
            rows.append(backend.forward_prefill(toks[:n], 0)[0])
        runs.append(rows)
    for a, b in zip(*runs):
        assert np.array_equal(a.view(np.uint32), b.view(np.uint32))


def test_wide_prefill_greedy_key(backend):
    """Without logits the wide pass returns the fused argmax of the same row."""
    spec = S.tiny_spec(FL_Q8_0, max_seq=256)
    backend.init_gpu_kv_cache(spec, FL_KV_F16)
    backend.upload_weights_to_gpu(S.make_model(spec, seed=2))
    toks = S.random_tokens(5, 130, spec.vocab)
    logits, tok, val = backend.forward_prefill(toks, 0)
    backend.reset()
    none, tok2, val2 = backend.forward_prefill(toks, 0, logits=False)
    assert none is None and tok2 == tok and val2 == val
