"""GPU tests of the attention kernels (k_attn.hip) and the prompt's row-wise
glue through the C ABI, against numpy restatements of candle-transformers
quantized_llama's attention (rope_i, KV cache append, grouped-query heads,
softmax(q.k/sqrt(hd)) with the causal mask, . v) in float64.  f32 sums are
reordered on the GPU: values at 1e-5 relative to the largest output; cache
writes are exact (the rotation is written without FMA contraction, as numpy
computes it in f32).

Decode: the split-context kernels (head_dim 64 / 128, 1..8 query heads per kv
head; a partial record per slice, then a combining launch) at positions on
and around the slice boundaries, up to the longest context, called back to
back on one context (the partial records are reused by every call).
Prefill: prompts at offset 0 and later, lengths that are not a multiple of
the 32-row query tile, q / k / v read with row strides from one merged
buffer."""
import ctypes

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def env():
    import torch

    import arm_ai_amd as A

    if not torch.cuda.is_available():
        pytest.fail("GPU tests need torch to see the GPU (import torch before the library)")
    ctx = A.Context(0)
    yield torch, A._lib, ctx
    ctx.close()


def _dev(torch, a):
    t = torch.from_numpy(np.ascontiguousarray(a)).to("cuda:0")
    torch.cuda.synchronize()
    return t


def _rel(a, b):
    a = np.asarray(a, np.float64)
    b = np.asarray(b, np.float64)
    return float(np.max(np.abs(a - b)) / max(np.max(np.abs(b)), 1e-30))


def _rope(x, c, s):
    """rope_i in f32, as numpy evaluates a*c - b*s (no FMA)."""
    out = np.empty_like(x)
    a, b = x[..., 0::2], x[..., 1::2]
    out[..., 0::2] = a * c - b * s
    out[..., 1::2] = a * s + b * c
    return out


def _tables(hd, max_seq):
    theta = 1.0 / (10000.0 ** (np.arange(0, hd, 2, dtype=np.float32) / hd))
    ang = np.arange(max_seq, dtype=np.float32)[:, None] * theta[None, :]
    return np.cos(ang).astype(np.float32), np.sin(ang).astype(np.float32)


def _attend(q, kc, vc, upto, rep):
    """q [n_head, hd] f32; caches [n_kv, max_seq, hd]; positions 0..upto."""
    n_head, hd = q.shape
    out = np.empty((n_head, hd))
    for h in range(n_head):
        kk = kc[h // rep, :upto + 1].astype(np.float64)
        s = kk @ q[h].astype(np.float64) / np.sqrt(hd)
        p = np.exp(s - s.max())
        p /= p.sum()
        out[h] = p @ vc[h // rep, :upto + 1].astype(np.float64)
    return out


def _decode_call(torch, lib, ctx, n_head, n_kv, hd, max_seq, kc, vc, qk, v, pos, dcos, dsin):
    L = lib.load()
    dqk, dv = _dev(torch, qk), _dev(torch, v)
    dpos = torch.tensor([pos], dtype=torch.int64, device="cuda:0")
    out = torch.empty(n_head * hd, dtype=torch.float32, device="cuda:0")
    torch.cuda.synchronize()
    lib.check(L.aq_llama_attn_decode(ctx.handle, dqk.data_ptr(), dv.data_ptr(), dcos.data_ptr(), dsin.data_ptr(),
                                     dpos.data_ptr(), kc.data_ptr(), vc.data_ptr(), n_head, n_kv, hd, max_seq,
                                     out.data_ptr()))
    ctx.synchronize()
    return out.cpu().numpy().reshape(n_head, hd)


@pytest.mark.parametrize(
    "n_head,n_kv,hd,max_seq,positions",
    [
        # TinyLlama heads: slices of at least 16 positions, 64 slices of 4 kv heads
        (32, 4, 64, 1024, [0, 1, 31, 32, 33, 63, 64, 600, 1023]),
        # max_seq not a multiple of 16: 38 slices can hold positions, the last from 592
        (32, 4, 64, 600, [0, 15, 16, 591, 592, 599]),
        (32, 4, 64, 8192, [8191, 2048, 2049, 4097]),  # slices longer than 16 (8192 / 64 = 128 per slice)
        (32, 8, 128, 2048, [0, 63, 64, 511, 512, 2047]),  # Llama-3-8B heads: 4 per kv head, 32 slices
        (8, 4, 64, 512, [0, 100, 511]),  # 2 per kv head
        (8, 8, 128, 512, [0, 5, 300]),   # one query head per kv head
        (64, 8, 128, 256, [0, 255]),     # 8 per kv head at head_dim 128
        (9, 3, 64, 640, [0, 15, 16, 511, 512, 639]),  # SmolLM-135M heads: 3 per kv head, 85 slices
        (15, 5, 64, 300, [0, 17, 299]),  # 3 per kv head, five kv heads
    ],
)
def test_split_decode_against_numpy_back_to_back(env, n_head, n_kv, hd, max_seq, positions):
    """Several calls on one context in a row, each checked: a record left
    over from a longer context must not enter a shorter one's combine."""
    torch, lib, ctx = env
    rng = np.random.default_rng(n_head * hd + max_seq)
    kc = rng.standard_normal((n_kv, max_seq, hd)).astype(np.float32)
    vc = rng.standard_normal((n_kv, max_seq, hd)).astype(np.float32)
    cos, sin = _tables(hd, max_seq)
    dkc, dvc, dcos, dsin = _dev(torch, kc), _dev(torch, vc), _dev(torch, cos), _dev(torch, sin)
    rep = n_head // n_kv
    for pos in positions:
        qk = (2 * rng.standard_normal((n_head + n_kv) * hd)).astype(np.float32)
        v = rng.standard_normal(n_kv * hd).astype(np.float32)
        got = _decode_call(torch, lib, ctx, n_head, n_kv, hd, max_seq, dkc, dvc, qk, v, pos, dcos, dsin)
        q = _rope(qk[:n_head * hd].reshape(n_head, hd), cos[pos], sin[pos])
        k = _rope(qk[n_head * hd:].reshape(n_kv, hd), cos[pos], sin[pos])
        kc[:, pos], vc[:, pos] = k, v.reshape(n_kv, hd)
        assert _rel(got, _attend(q, kc, vc, pos, rep)) <= 1e-5, f"pos {pos}"
        assert np.array_equal(dkc.cpu().numpy(), kc), f"pos {pos}: k cache"
        assert np.array_equal(dvc.cpu().numpy(), vc), f"pos {pos}: v cache"


def test_split_decode_sharp_softmax(env):
    """Scores 60 apart between slices: the combine's rescaling by e^(m_s - M)
    must take the slice maxima into account (a plain sum of the slices' e^(s -
    m_s) would weight every slice alike)."""
    torch, lib, ctx = env
    n_head, n_kv, hd, max_seq, pos = 32, 4, 64, 1024, 700
    rng = np.random.default_rng(9)
    kc = rng.standard_normal((n_kv, max_seq, hd)).astype(np.float32)
    vc = rng.standard_normal((n_kv, max_seq, hd)).astype(np.float32)
    kc[:, 333] *= 20.0  # one key far above the others
    cos, sin = _tables(hd, max_seq)
    dkc, dvc, dcos, dsin = _dev(torch, kc), _dev(torch, vc), _dev(torch, cos), _dev(torch, sin)
    qk = rng.standard_normal((n_head + n_kv) * hd).astype(np.float32)
    qk[:n_head * hd] *= 3.0
    v = rng.standard_normal(n_kv * hd).astype(np.float32)
    got = _decode_call(torch, lib, ctx, n_head, n_kv, hd, max_seq, dkc, dvc, qk, v, pos, dcos, dsin)
    q = _rope(qk[:n_head * hd].reshape(n_head, hd), cos[pos], sin[pos])
    kc[:, pos] = _rope(qk[n_head * hd:].reshape(n_kv, hd), cos[pos], sin[pos])
    vc[:, pos] = v.reshape(n_kv, hd)
    assert _rel(got, _attend(q, kc, vc, pos, n_head // n_kv)) <= 1e-5


def _prefill_ref(q, k, v, kc, vc, cos, sin, index_pos, n_head, n_kv, hd):
    """Returns (out [m, n_head*hd], kc, vc after the append)."""
    m = q.shape[0]
    rep = n_head // n_kv
    kc, vc = kc.copy(), vc.copy()
    P = np.arange(index_pos, index_pos + m)
    qr = _rope(q.reshape(m, n_head, hd), cos[P][:, None, :], sin[P][:, None, :])
    kr = _rope(k.reshape(m, n_kv, hd), cos[P][:, None, :], sin[P][:, None, :])
    kc[:, P] = kr.transpose(1, 0, 2)
    vc[:, P] = v.reshape(m, n_kv, hd).transpose(1, 0, 2)
    out = np.empty((m, n_head, hd))
    for r in range(m):
        out[r] = _attend(qr[r], kc, vc, index_pos + r, rep)
    return out.reshape(m, n_head * hd), kc, vc


@pytest.mark.parametrize(
    "n_head,n_kv,hd,index_pos,m,max_seq",
    [(4, 2, 64, 0, 7, 64), (32, 4, 64, 0, 512, 640), (32, 4, 64, 0, 100, 128), (8, 8, 128, 5, 70, 128),
     (32, 8, 128, 0, 65, 128), (32, 4, 64, 200, 1, 256), (16, 2, 64, 37, 130, 256),
     (9, 3, 64, 0, 512, 640), (9, 3, 64, 512, 3, 640)],  # SmolLM-135M heads: 3 per kv head
)
def test_prefill_against_numpy(env, n_head, n_kv, hd, index_pos, m, max_seq):
    torch, lib, ctx = env
    L = lib.load()
    rng = np.random.default_rng(m + index_pos + hd)
    width = (n_head + n_kv) * hd
    qk = rng.standard_normal((m, width)).astype(np.float32)  # the merged wq|wk output: strided q and k
    v = rng.standard_normal((m, n_kv * hd)).astype(np.float32)
    kc = rng.standard_normal((n_kv, max_seq, hd)).astype(np.float32)
    vc = rng.standard_normal((n_kv, max_seq, hd)).astype(np.float32)
    cos, sin = _tables(hd, max_seq)
    dqk, dv, dkc, dvc = _dev(torch, qk), _dev(torch, v), _dev(torch, kc), _dev(torch, vc)
    dcos, dsin = _dev(torch, cos), _dev(torch, sin)
    out = torch.empty((m, n_head * hd), dtype=torch.float32, device="cuda:0")
    torch.cuda.synchronize()
    lib.check(L.aq_llama_attn_prefill(ctx.handle, dqk.data_ptr(), width, dqk.data_ptr() + 4 * n_head * hd, width,
                                      dv.data_ptr(), n_kv * hd, dcos.data_ptr(), dsin.data_ptr(), index_pos, m,
                                      dkc.data_ptr(), dvc.data_ptr(), n_head, n_kv, hd, max_seq, out.data_ptr()))
    ctx.synchronize()
    want, kc2, vc2 = _prefill_ref(qk[:, :n_head * hd], qk[:, n_head * hd:], v, kc, vc, cos, sin, index_pos, n_head,
                                  n_kv, hd)
    assert _rel(out.cpu().numpy(), want) <= 1e-5
    assert np.array_equal(dkc.cpu().numpy(), kc2)
    assert np.array_equal(dvc.cpu().numpy(), vc2)


def test_prefill_sharp_softmax(env):
    """One key row twenty times the others and queries three times larger:
    scores far apart across the key blocks of the four wavefronts, so the
    running maxima (base-2 units) and the combine's rescaling decide the
    result."""
    torch, lib, ctx = env
    L = lib.load()
    n_head, n_kv, hd, m, max_seq = 32, 4, 64, 300, 320
    rng = np.random.default_rng(21)
    width = (n_head + n_kv) * hd
    qk = rng.standard_normal((m, width)).astype(np.float32)
    qk[:, :n_head * hd] *= 3.0
    qk[57, n_head * hd:] *= 20.0  # key 57 far above the others for every later query
    v = rng.standard_normal((m, n_kv * hd)).astype(np.float32)
    kc = np.zeros((n_kv, max_seq, hd), np.float32)
    vc = np.zeros((n_kv, max_seq, hd), np.float32)
    cos, sin = _tables(hd, max_seq)
    dqk, dv, dkc, dvc = _dev(torch, qk), _dev(torch, v), _dev(torch, kc), _dev(torch, vc)
    dcos, dsin = _dev(torch, cos), _dev(torch, sin)
    out = torch.empty((m, n_head * hd), dtype=torch.float32, device="cuda:0")
    torch.cuda.synchronize()
    lib.check(L.aq_llama_attn_prefill(ctx.handle, dqk.data_ptr(), width, dqk.data_ptr() + 4 * n_head * hd, width,
                                      dv.data_ptr(), n_kv * hd, dcos.data_ptr(), dsin.data_ptr(), 0, m,
                                      dkc.data_ptr(), dvc.data_ptr(), n_head, n_kv, hd, max_seq, out.data_ptr()))
    ctx.synchronize()
    want, _, _ = _prefill_ref(qk[:, :n_head * hd], qk[:, n_head * hd:], v, kc, vc, cos, sin, 0, n_head, n_kv, hd)
    assert _rel(out.cpu().numpy(), want) <= 1e-5


def test_prefill_then_decode_continue_the_same_cache(env):
    """A prompt through the prefill kernel, then decode steps at the next
    positions read the cache it wrote (the layout both kernels share)."""
    torch, lib, ctx = env
    L = lib.load()
    n_head, n_kv, hd, max_seq, m = 32, 4, 64, 256, 40
    rng = np.random.default_rng(77)
    q = rng.standard_normal((m, n_head * hd)).astype(np.float32)
    k = rng.standard_normal((m, n_kv * hd)).astype(np.float32)
    v = rng.standard_normal((m, n_kv * hd)).astype(np.float32)
    kc = np.zeros((n_kv, max_seq, hd), np.float32)
    vc = np.zeros((n_kv, max_seq, hd), np.float32)
    cos, sin = _tables(hd, max_seq)
    dq, dk, dv = _dev(torch, q), _dev(torch, k), _dev(torch, v)
    dkc, dvc, dcos, dsin = _dev(torch, kc), _dev(torch, vc), _dev(torch, cos), _dev(torch, sin)
    out = torch.empty((m, n_head * hd), dtype=torch.float32, device="cuda:0")
    torch.cuda.synchronize()
    lib.check(L.aq_llama_attn_prefill(ctx.handle, dq.data_ptr(), n_head * hd, dk.data_ptr(), n_kv * hd, dv.data_ptr(),
                                      n_kv * hd, dcos.data_ptr(), dsin.data_ptr(), 0, m, dkc.data_ptr(),
                                      dvc.data_ptr(), n_head, n_kv, hd, max_seq, out.data_ptr()))
    ctx.synchronize()
    _, kc, vc = _prefill_ref(q, k, v, kc, vc, cos, sin, 0, n_head, n_kv, hd)
    for pos in range(m, m + 3):
        qk = rng.standard_normal((n_head + n_kv) * hd).astype(np.float32)
        vv = rng.standard_normal(n_kv * hd).astype(np.float32)
        got = _decode_call(torch, lib, ctx, n_head, n_kv, hd, max_seq, dkc, dvc, qk, vv, pos, dcos, dsin)
        qr = _rope(qk[:n_head * hd].reshape(n_head, hd), cos[pos], sin[pos])
        kc[:, pos] = _rope(qk[n_head * hd:].reshape(n_kv, hd), cos[pos], sin[pos])
        vc[:, pos] = vv.reshape(n_kv, hd)
        assert _rel(got, _attend(qr, kc, vc, pos, n_head // n_kv)) <= 1e-5


def test_prefill_argument_errors(env):
    torch, lib, ctx = env
    L = lib.load()
    buf = torch.zeros(1 << 16, dtype=torch.float32, device="cuda:0")
    p = buf.data_ptr()
    ok = dict(ldq=256, ldk=128, ldv=128, index_pos=0, m=4, n_head=4, n_kv=2, hd=64, max_seq=64)

    def call(**kw):
        a = {**ok, **kw}
        return L.aq_llama_attn_prefill(ctx.handle, p, a["ldq"], p, a["ldk"], p, a["ldv"], p, p, a["index_pos"], a["m"],
                                       p, p, a["n_head"], a["n_kv"], a["hd"], a["max_seq"], p)

    assert call(hd=32) != 0            # head_dim other than 64 / 128
    assert call(index_pos=62) != 0     # past the end of the cache
    assert call(n_kv=3) != 0           # n_head not a multiple of n_kv
    assert call(ldq=128) != 0          # q rows shorter than n_head * head_dim
    assert call(index_pos=-1) != 0
    assert call(m=0) == 0              # nothing to do


def test_embed_rows_and_silu_mul_rows(env):
    torch, lib, ctx = env
    L = lib.load()
    rng = np.random.default_rng(5)
    table = rng.standard_normal((100, 64)).astype(np.float32)
    toks = np.array([3, 99, 100, -5, 42, 3], np.int64)
    dt, dtok = _dev(torch, table), _dev(torch, toks)
    out = torch.empty((len(toks), 64), dtype=torch.float32, device="cuda:0")
    torch.cuda.synchronize()
    lib.check(L.aq_llama_embed_rows(ctx.handle, dt.data_ptr(), 100, dtok.data_ptr(), len(toks), 64, out.data_ptr()))
    ctx.synchronize()
    want = np.stack([table[t] if 0 <= t < 100 else np.zeros(64, np.float32) for t in toks])
    assert np.array_equal(out.cpu().numpy(), want)

    m, n = 5, 700
    gu = (4 * rng.standard_normal((m, 2 * n))).astype(np.float32)
    gu[0, 0], gu[1, 1] = -100.0, 100.0
    dgu = _dev(torch, gu)
    o = torch.empty((m, n), dtype=torch.float32, device="cuda:0")
    torch.cuda.synchronize()
    lib.check(L.aq_llama_silu_mul_rows(ctx.handle, dgu.data_ptr(), dgu.data_ptr() + 4 * n, 2 * n, m, n, o.data_ptr()))
    ctx.synchronize()
    g, u = gu[:, :n].astype(np.float64), gu[:, n:].astype(np.float64)
    got = o.cpu().numpy()
    assert np.all(np.isfinite(got))
    assert _rel(got, g / (1 + np.exp(-g)) * u) <= 1e-5
    # separate g and u buffers (unmerged w1 / w3): ld = n
    dg, du = _dev(torch, gu[:, :n]), _dev(torch, gu[:, n:])
    o2 = torch.empty((m, n), dtype=torch.float32, device="cuda:0")
    torch.cuda.synchronize()
    lib.check(L.aq_llama_silu_mul_rows(ctx.handle, dg.data_ptr(), du.data_ptr(), n, m, n, o2.data_ptr()))
    ctx.synchronize()
    assert np.array_equal(o2.cpu().numpy(), got)


def _prefill_call(torch, lib, ctx, n_head, n_kv, hd, index_pos, m, max_seq, qk, v, kc, vc, cos, sin):
    """(out, kc, vc) after aq_llama_attn_prefill on host arrays."""
    width = (n_head + n_kv) * hd
    dqk, dv, dkc, dvc, dcos, dsin = (_dev(torch, a) for a in (qk, v, kc, vc, cos, sin))
    out = torch.empty((m, n_head * hd), dtype=torch.float32, device="cuda:0")
    torch.cuda.synchronize()
    lib.check(lib.load().aq_llama_attn_prefill(
        ctx.handle, dqk.data_ptr(), width, dqk.data_ptr() + 4 * n_head * hd, width, dv.data_ptr(), n_kv * hd,
        dcos.data_ptr(), dsin.data_ptr(), index_pos, m, dkc.data_ptr(), dvc.data_ptr(), n_head, n_kv, hd, max_seq,
        out.data_ptr()))
    ctx.synchronize()
    return out.cpu().numpy(), dkc.cpu().numpy(), dvc.cpu().numpy()


# The split-operand kernel's forms and edges: each (wavefronts per unit and key
# range), last tiles and blocks of one row and of 31, prompts that begin within a
# block of cached keys, units that do not fill the last workgroup.
@pytest.mark.parametrize(
    "n_head,n_kv,hd,index_pos,m",
    [(4, 1, 64, 0, 321), (3, 3, 64, 650, 1), (9, 3, 64, 95, 1001), (8, 2, 128, 0, 161), (6, 2, 128, 319, 31),
     (32, 32, 64, 0, 321), (32, 4, 64, 33, 450), (32, 8, 128, 95, 330), (33, 11, 128, 0, 1281)],
)
@pytest.mark.parametrize("scaled", [False, True])
def test_prefill_split_operands(env, n_head, n_kv, hd, index_pos, m, scaled):
    torch, lib, ctx = env
    rng = np.random.default_rng(m + hd + scaled)
    max_seq = index_pos + m + 3
    qk = rng.standard_normal((m, (n_head + n_kv) * hd)).astype(np.float32)
    v = rng.standard_normal((m, n_kv * hd)).astype(np.float32)
    kc = rng.standard_normal((n_kv, max_seq, hd)).astype(np.float32)
    vc = rng.standard_normal((n_kv, max_seq, hd)).astype(np.float32)
    if scaled:  # powers of two that change from block to block, and a block of zeros
        pos = np.arange(max_seq)
        ks, vs = 2.0 ** -(pos // 32 % 5), 2.0 ** (9 * (pos // 32 % 4) - 13)
        ks[64:96] = vs[64:96] = 0.0
        kc *= ks[None, :, None].astype(np.float32)
        vc *= vs[None, :, None].astype(np.float32)
        qk[:, n_head * hd:] *= ks[index_pos:index_pos + m, None].astype(np.float32)
        v *= vs[index_pos:index_pos + m, None].astype(np.float32)
        qk[:, :n_head * hd] *= (2.0 ** -(np.arange(m) % 9))[:, None].astype(np.float32)
    cos, sin = _tables(hd, max_seq)
    got, kc1, vc1 = _prefill_call(torch, lib, ctx, n_head, n_kv, hd, index_pos, m, max_seq, qk, v, kc, vc, cos, sin)
    want, kc2, vc2 = _prefill_ref(qk[:, :n_head * hd], qk[:, n_head * hd:], v, kc, vc, cos, sin, index_pos, n_head, n_kv, hd)
    # |score error| <= sum |q k| / sqrt(hd) (2^-22 + hd / 16 2^-24): at most
    # 7.3 * 7.2e-7 = 5.2e-6 for normal values and hd = 128, and as much relative in
    # the output; the sums of the output add 2^-22 + 3 * keys / 16 2^-24
    assert _rel(got, want) <= 1e-5
    assert np.array_equal(kc1, kc2) and np.array_equal(vc1, vc2)


# What the split cannot hold goes through plain f32: values beyond 2^50 or below
# 2^-50, infinities and NaN, in K, V or a query row.
@pytest.mark.parametrize("where,value", [("v", 2.0 ** 70), ("v", 2.0 ** -70), ("k", 2.0 ** -70), ("q", 2.0 ** -70),
                                         ("q", 2.0 ** 70), ("v", np.nan), ("k", np.nan), ("v", np.inf), ("q", np.nan)])
@pytest.mark.parametrize("hd", [64, 128])
def test_prefill_values_beyond_the_split(env, hd, where, value):
    torch, lib, ctx = env
    n_head, n_kv, m, at = 6, 2, 330, 201
    rng = np.random.default_rng(hd)
    qk = rng.standard_normal((m, (n_head + n_kv) * hd)).astype(np.float32)
    v = rng.standard_normal((m, n_kv * hd)).astype(np.float32)
    cos, sin = _tables(hd, m)
    if where == "v":
        v[192:224, hd:] *= value if np.isfinite(value) else 1
        if not np.isfinite(value):
            v[at, hd:] = value  # kv head 1, key 201
    elif where == "k":
        if np.isfinite(value):
            qk[192:224, (n_head + 1) * hd:] *= value
        else:
            qk[at, (n_head + 1) * hd:] = value
    elif np.isfinite(value):
        qk[at, 4 * hd:5 * hd] *= value  # query head 4 (kv head 1), row 201
        if value > 1:  # scores within the f32 range
            qk[:, n_head * hd:] *= 2.0 ** -70
    else:
        qk[at, 4 * hd:5 * hd] = value
    z = np.zeros((n_kv, m, hd), np.float32)
    got, _, _ = _prefill_call(torch, lib, ctx, n_head, n_kv, hd, 0, m, m, qk, v, z, z, cos, sin)
    with np.errstate(all="ignore"):
        want, _, _ = _prefill_ref(qk[:, :n_head * hd], qk[:, n_head * hd:], v, z, z, cos, sin, 0, n_head, n_kv, hd)
    got, want = got.reshape(m, n_head, hd), want.reshape(m, n_head, hd)
    fine = np.isfinite(want)
    assert np.array_equal(np.isfinite(got), fine)
    assert np.array_equal(np.isnan(got), np.isnan(want))
    for r0, r1 in ((0, 192), (192, 224), (224, m)):  # (apart: their sizes differ by 2^70)
        for h in range(n_head):
            f = fine[r0:r1, h]
            if f.any():
                assert _rel(got[r0:r1, h][f], want[r0:r1, h][f]) <= 1e-5


def _prefill_captured(torch, lib, ctx, n_head, n_kv, hd, m, qk, v, cos, sin):
    """out of a prompt at position 0 through the f32 kernel, which a captured call runs."""
    width = (n_head + n_kv) * hd
    z = np.zeros((n_kv, m, hd), np.float32)
    dqk, dv, dkc, dvc, dcos, dsin = (_dev(torch, a) for a in (qk, v, z, z, cos, sin))
    out = torch.empty((m, n_head * hd), dtype=torch.float32, device="cuda:0")
    handle = ctypes.c_void_p()
    lib.check(lib.load().aq_ctx_stream(ctx.handle, ctypes.byref(handle)))
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=torch.cuda.ExternalStream(handle.value)):
        lib.check(lib.load().aq_llama_attn_prefill(
            ctx.handle, dqk.data_ptr(), width, dqk.data_ptr() + 4 * n_head * hd, width, dv.data_ptr(), n_kv * hd,
            dcos.data_ptr(), dsin.data_ptr(), 0, m, dkc.data_ptr(), dvc.data_ptr(), n_head, n_kv, hd, m, out.data_ptr()))
    graph.replay()
    torch.cuda.synchronize()
    return out.cpu().numpy()


def _scores(qk, kc, cos, sin, n_head):
    """[m, n_head, key] of a prompt at position 0 in 64 bits, -inf past the row; kc: the cache after it."""
    n_kv, m, hd = kc.shape
    q = _rope(qk[:, :n_head * hd].reshape(m, n_head, hd), cos[:, None, :], sin[:, None, :]).astype(np.float64)
    s = np.stack([q[:, h] @ kc[h * n_kv // n_head].astype(np.float64).T for h in range(n_head)], 1) / np.sqrt(hd)
    return np.where(np.arange(m)[None, None] <= np.arange(m)[:, None, None], s, -np.inf)


def _row_errors(got, want, m, n_head):
    """Error of each row and head, relative to that row's largest output."""
    got, want = (a.astype(np.float64).reshape(m, n_head, -1) for a in (got, want))
    return np.abs(got - want).max(-1) / np.abs(want).max(-1)


# Scores up to the split's limit and far past it.  A row whose two largest scores
# lie closer than the rounding of a sum of that size (2^-18 of the largest, 64
# roundings) may weigh them otherwise and is left out, but must be finite.
@pytest.mark.parametrize("hd", [64, 128])
@pytest.mark.parametrize("scale", [5, 6, 7, 10, 13, 20, 40])
def test_prefill_large_scores(env, hd, scale):
    torch, lib, ctx = env
    n_head, n_kv, m = 6, 2, 330
    rng = np.random.default_rng(hd + scale)
    qk = (2.0 ** scale * rng.standard_normal((m, (n_head + n_kv) * hd))).astype(np.float32)
    qk[200, :n_head * hd] = 0.0  # a query of zeros: the mean of the values before it
    v = rng.standard_normal((m, n_kv * hd)).astype(np.float32)
    cos, sin = _tables(hd, m)
    z = np.zeros((n_kv, m, hd), np.float32)
    got, kc, _ = _prefill_call(torch, lib, ctx, n_head, n_kv, hd, 0, m, m, qk, v, z, z, cos, sin)
    want, _, _ = _prefill_ref(qk[:, :n_head * hd], qk[:, n_head * hd:], v, z, z, cos, sin, 0, n_head, n_kv, hd)
    assert np.isfinite(got).all()
    s = _scores(qk, kc, cos, sin, n_head)
    top = np.sort(s, -1)[..., -2:]
    # 30: a second key of e^-30 changes nothing
    clear = top[..., 1] - top[..., 0] > 30 + np.abs(s).max(-1, initial=0, where=np.isfinite(s)) * 2.0 ** -18
    clear[200] = clear[0] = True
    assert clear.mean() > (0.7 if scale > 5 else 0.5)
    assert _row_errors(got, want, m, n_head)[clear].max() <= 2e-6


# One key (31: the last of its block, which the rows before it do not see) far
# above the others: every row as exact as the f32 kernel has it.  Left out are the
# rows that weigh key 31 against others: a score of 2^exp is rounded, and one row
# says nothing of how far.
@pytest.mark.parametrize("hd", [64, 128])
@pytest.mark.parametrize("where", ["k", "v"])
@pytest.mark.parametrize("exp", [8, 13, 16, 20, 28, 38])
def test_prefill_one_large_key(env, hd, where, exp):
    torch, lib, ctx = env
    n_head, n_kv, m = 6, 2, 330
    rng = np.random.default_rng(hd + exp)
    qk = rng.standard_normal((m, (n_head + n_kv) * hd)).astype(np.float32)
    v = rng.standard_normal((m, n_kv * hd)).astype(np.float32)
    (qk[:, n_head * hd:] if where == "k" else v)[31] *= 2.0 ** exp
    cos, sin = _tables(hd, m)
    z = np.zeros((n_kv, m, hd), np.float32)
    got, kc, _ = _prefill_call(torch, lib, ctx, n_head, n_kv, hd, 0, m, m, qk, v, z, z, cos, sin)
    f32 = _prefill_captured(torch, lib, ctx, n_head, n_kv, hd, m, qk, v, cos, sin)
    want, _, _ = _prefill_ref(qk[:, :n_head * hd], qk[:, n_head * hd:], v, z, z, cos, sin, 0, n_head, n_kv, hd)
    a, b = (_row_errors(o, want, m, n_head) for o in (got, f32))
    clear = np.ones((m, n_head), bool)
    if where == "k":
        s = _scores(qk, kc, cos, sin, n_head)
        rest = np.where(np.arange(m) == 31, -np.inf, s).max(-1)
        clear[31:] = np.abs(s[31:, :, 31] - rest[31:]) > 30
    for rows in (slice(0, 31), slice(31, m)):
        c = clear[rows]
        assert c.mean() > 0.7
        # (the largest error of a few hundred rows differs by half between two orders of
        # the same f32 sums; its bound is test_prefill_split_operands')
        rms = [np.sqrt((e[rows][c] ** 2).mean()) for e in (a, b)]
        assert rms[0] <= 1.2 * rms[1] and a[rows][c].max() <= 1e-5, (rows, rms, a[rows][c].max())


# The same key within the first of two pieces: the pieces (the second reads the key
# from the cache) give what the whole prompt gives, to the bound of either.
@pytest.mark.parametrize("hd", [64, 128])
@pytest.mark.parametrize("where", ["k", "v"])
@pytest.mark.parametrize("exp", [0, 13, 24])
def test_prefill_in_pieces(env, hd, where, exp):
    torch, lib, ctx = env
    n_head, n_kv, m, cut = 6, 2, 420, 257
    rng = np.random.default_rng(hd + exp)
    qk = rng.standard_normal((m, (n_head + n_kv) * hd)).astype(np.float32)
    v = rng.standard_normal((m, n_kv * hd)).astype(np.float32)
    (qk[:, n_head * hd:] if where == "k" else v)[201] *= 2.0 ** exp
    cos, sin = _tables(hd, m)
    z = np.zeros((n_kv, m, hd), np.float32)
    whole, kw, vw = _prefill_call(torch, lib, ctx, n_head, n_kv, hd, 0, m, m, qk, v, z, z, cos, sin)
    a, k1, v1 = _prefill_call(torch, lib, ctx, n_head, n_kv, hd, 0, cut, m, qk[:cut], v[:cut], z, z, cos, sin)
    b, k2, v2 = _prefill_call(torch, lib, ctx, n_head, n_kv, hd, cut, m - cut, m, qk[cut:], v[cut:], k1, v1, cos, sin)
    assert np.array_equal(kw, k2) and np.array_equal(vw, v2)
    s = _scores(qk, kw, cos, sin, n_head)
    rest = np.where(np.arange(m) == 201, -np.inf, s).max(-1)
    clear = np.ones((m, n_head), bool)
    if where == "k":  # (a score of 2^exp against others: see above)
        clear[201:] = (exp == 0) | (np.abs(s[201:, :, 201] - rest[201:]) > 30)
    assert clear.mean() > 0.7
    assert _row_errors(np.concatenate([a, b]), whole, m, n_head)[clear].max() <= 2e-5


# The range inside a block of V: one key far above the others of its block, at each
# place in it, and dims far below the others.  Each dim of the rows before that key
# as exact as the f32 kernel has it (15: just past the range that the split takes,
# 13: just inside it).
@pytest.mark.parametrize("hd", [64, 128])
@pytest.mark.parametrize("exp", [13, 15, 24])
def test_prefill_range_of_v(env, hd, exp):
    torch, lib, ctx = env
    n_head, n_kv, m = 2, 1, 330
    cos, sin = _tables(hd, m)
    z = np.zeros((n_kv, m, hd), np.float32)
    rng = np.random.default_rng(hd + exp)
    qk = rng.standard_normal((m, (n_head + n_kv) * hd)).astype(np.float32)
    v0 = rng.standard_normal((m, n_kv * hd)).astype(np.float32)
    base, _, _ = _prefill_ref(qk[:, :n_head * hd], qk[:, n_head * hd:], v0, z, z, cos, sin, 0, n_head, n_kv, hd)
    f32 = _prefill_captured(torch, lib, ctx, n_head, n_kv, hd, m, qk, v0, cos, sin)
    err = np.abs(f32 - base).reshape(m, -1)
    for at in range(96, 128):
        v = v0.copy()
        v[at] *= 2.0 ** exp
        got, _, _ = _prefill_call(torch, lib, ctx, n_head, n_kv, hd, 0, m, m, qk, v, z, z, cos, sin)
        # (the rows before key `at` do not see it)
        assert np.abs(got - base)[:at].max() <= 1.5 * err.max(), at
    for d in range(0, hd, 5):
        v = v0.copy()
        v[:, d] *= 2.0 ** -exp
        got, _, _ = _prefill_call(torch, lib, ctx, n_head, n_kv, hd, 0, m, m, qk, v, z, z, cos, sin)
        # (scaling by a power of two is exact: that dim's outputs scale with it)
        own = got.reshape(m, n_head, hd)[..., d] * 2.0 ** exp
        assert np.abs(own - base.reshape(m, n_head, hd)[..., d]).max() <= 1.5 * err.max(), d


def test_prefill_under_capture_is_the_f32_kernel(env):
    """A captured prompt keeps no workspace address: its replays, after larger
    prompts have grown the workspace, give the f32 kernel's result."""
    torch, lib, ctx = env
    L = lib.load()
    n_head, n_kv, hd, m = 8, 2, 64, 400
    rng = np.random.default_rng(3)
    g = [rng.standard_normal(s).astype(np.float32) for s in ((m, (n_head + n_kv) * hd), (m, n_kv * hd))]
    cos, sin = _tables(hd, m)
    z = np.zeros((n_kv, m, hd), np.float32)
    want, _, _ = _prefill_ref(g[0][:, :n_head * hd], g[0][:, n_head * hd:], g[1], z, z, cos, sin, 0, n_head, n_kv, hd)
    dqk, dv, dkc, dvc, dcos, dsin = (_dev(torch, a) for a in (*g, z, z, cos, sin))
    out = torch.empty((m, n_head * hd), dtype=torch.float32, device="cuda:0")
    width = (n_head + n_kv) * hd
    torch.cuda.synchronize()
    handle = ctypes.c_void_p()
    lib.check(L.aq_ctx_stream(ctx.handle, ctypes.byref(handle)))
    stream = torch.cuda.ExternalStream(handle.value)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=stream):
        lib.check(L.aq_llama_attn_prefill(
            ctx.handle, dqk.data_ptr(), width, dqk.data_ptr() + 4 * n_head * hd, width, dv.data_ptr(), n_kv * hd,
            dcos.data_ptr(), dsin.data_ptr(), 0, m, dkc.data_ptr(), dvc.data_ptr(), n_head, n_kv, hd, m, out.data_ptr()))
    for n in (0, 700, 2100):  # eager prompts between the replays
        if n:
            c2, s2 = _tables(hd, n)
            z2 = np.zeros((n_kv, n, hd), np.float32)
            a = rng.standard_normal((n, width)).astype(np.float32)
            _prefill_call(torch, lib, ctx, n_head, n_kv, hd, 0, n, n, a, a[:, :n_kv * hd].copy(), z2, z2, c2, s2)
        out.zero_()
        torch.cuda.synchronize()
        graph.replay()
        torch.cuda.synchronize()
        assert _rel(out.cpu().numpy(), want) <= 1e-5
