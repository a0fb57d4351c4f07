"""A prompt's leading rows taken at once (host/tl_decode.c run_bulk) against
the same decoder fed chunk by chunk (tl_decode_chunk, held against the oracle
in test_decode_gpu.py): rings, last rows, state and the tokens that follow."""
import numpy as np
import pytest

from oracle import StepFns, model

pytestmark = pytest.mark.gpu

KW = dict(V=128, D=96, L=3, H=3, KV=1, F=64, T=64)
# (prompt length, W, mmax): below, at and past the least rows and the ring; a
# prompt of whole chunks; odd chunk widths; a ring that the rest wraps
CUTS = [(15, 64, 8), (16, 64, 8), (17, 64, 8), (24, 64, 8), (63, 64, 8), (64, 64, 8), (65, 64, 8), (150, 64, 8),
        (40, 64, 3), (30, 64, 1), (200, 100, 7), (64, 12, 4), (600, 560, 8)]


@pytest.fixture(scope="module")
def lib():
    import torch
    torch.cuda.init()
    import tlgemm
    L = tlgemm.load()
    L.check(L.tlg_init(0), "tlg_init")
    return L


@pytest.mark.parametrize("kvdt", [0, 1])
@pytest.mark.parametrize("opt", [dict(), dict(win=20, full_every=2), dict(qknorm=1)], ids=str)
@pytest.mark.parametrize("cut", CUTS, ids=str)
def test_prime_is_its_chunks(lib, cut, opt, kvdt):
    import tlgemm
    n, W, mmax = cut
    kw = dict(KW, **opt)
    m = model(**kw)
    r = np.random.default_rng(n)
    P = StepFns("oracle").init_params(m, 3)
    P += (0.05 * r.standard_normal(P.size)).astype(np.float32)
    prompt = r.integers(0, m.V, n).astype(np.int32)
    s = lib.tlg_stream_create()
    made = []
    for whole in (True, False):
        d = tlgemm.host().decode(kw, W, kv_f16=kvdt, exact_exp=1, maxpos=1024, mmax=mmax, pool=1)
        d.upload(P, s)
        if whole:
            d.prime(prompt, s)
        else:
            for i in range(0, n, mmax):
                d.chunk(prompt[i:i + mmax], i, s)
        made.append((d, d.logits((n - 1) % mmax + 1, s), [d.ring(l, s) for l in range(m.L)]))
    (a, la, ra), (b, lb, rb) = made
    # 3 layers of fp32 sums of at most 96 terms in another order, through the
    # softmax: 1e-5 of the mean.  An f16 ring may round such a difference to its
    # neighbouring value, 2^-10 of an element; in the first layer that takes a
    # value within 1e-6 of the middle, 2^-10 apart: a share of about 2e-3.  Later
    # layers see those steps too.
    tol = 2e-3 if kvdt else 1e-5
    assert np.abs(la - lb).max() <= tol * np.abs(lb).mean()
    for l, (x, y) in enumerate(zip(ra, rb)):
        for u, v in zip(x, y):
            u, v = ((t.view(np.float16).astype(np.float64) if kvdt else t) for t in (u, v))
            scale = np.abs(v).mean()
            assert np.abs(u - v).max() <= tol * max(scale, np.abs(v).max())
            assert l > 0 or not kvdt or (u != v).mean() <= 8e-3
    st = a.state(s)
    assert st[0] == n and st[2] == int(np.argmax(la[-1]))
    lib.tlg_stream_destroy(s)


def test_prime_refuses_what_chunks_refuse(lib):
    import tlgemm
    s = lib.tlg_stream_create()
    d = tlgemm.host().decode(KW, 64, kv_f16=0, exact_exp=1, maxpos=48, mmax=8, pool=1)
    d.upload(StepFns("oracle").init_params(model(**KW), 3), s)
    bad = np.full(40, 5, np.int32)
    bad[20] = KW["V"]
    for prompt in (bad, np.full(49, 5, np.int32)):
        with pytest.raises(tlgemm.TlgError):
            d.prime(prompt, s)
    d.prime(np.full(48, 5, np.int32), s)
    assert d.state(s)[0] == 48
    lib.tlg_stream_destroy(s)


def test_a_bad_token_past_the_ring_starts_nothing(lib):
    """Refused before any row of the prompt is copied or run: the rings stay."""
    import tlgemm
    s = lib.tlg_stream_create()
    d = tlgemm.host().decode(KW, 32, kv_f16=0, exact_exp=1, maxpos=128, mmax=8, pool=1)
    d.upload(StepFns("oracle").init_params(model(**KW), 3), s)
    d.prime(np.full(40, 5, np.int32), s)
    rings = [d.ring(l, s) for l in range(KW["L"])]
    bad = np.full(100, 7, np.int32)
    bad[90] = KW["V"]
    with pytest.raises(tlgemm.TlgError):
        d.prime(bad, s)
    for l, ring in enumerate(rings):
        assert all(np.array_equal(x, y) for x, y in zip(ring, d.ring(l, s)))
    lib.tlg_stream_destroy(s)
