"""Batched prefill on the matrix cores (engine/core.cpp:292-294, 353-646).

The reference multiplies FP32 activations by FP32-widened weights
(cblas_sgemm, closed source, summation order unknown: parity unpinned
bitwise, held to tolerance). The GPU GEMM splits each activation exactly into
FP16 hi + lo and accumulates in FP32; it is checked against an FP64 product
with a bound proportional to sum |a||w|, for row independence from the
chunk size (needed for exact canonical prefix reuse), and end to end through
the oracle gate and the reuse-equals-fresh invariant
(tools/check_native_cpu_prefix.py).
"""
import ctypes
import json
import shutil
from pathlib import Path

import numpy as np
import pytest

from oracle_binding import compare_logits

PROMPTS = json.loads((Path(__file__).parent / 'golden' / 'prompts.json').read_text())


@pytest.mark.gpu
@pytest.mark.parametrize('m,n,k', [(1, 1024, 1024), (37, 4096, 1024), (85, 1024, 2048), (512, 6144, 1024),
                                   (129, 1024, 3072), (1000, 4096, 1024), (1100, 6144, 1024),
                                   (1024, 6144, 1024), (2500, 4096, 1024)])
def test_gemm_against_fp64(qpkg, m, n, k):
    """Row counts cover each tile-to-XCD mapping of 128-row tiles: 1000 /
    1024 rows (4 XCDs pool their row tiles), 1100 (2 XCDs pool 2 row tiles
    each), 2500 (2 XCDs pool 3 each), plus the narrower 32 / 64-row tiles."""
    rng = np.random.default_rng(21)
    a = rng.standard_normal((m, k), dtype=np.float32) * 3
    w = (rng.standard_normal((n, k), dtype=np.float32) * 0.02).astype(np.float16)
    got = qpkg.gemm(a, w)
    ref = a.astype(np.float64) @ w.astype(np.float64).T
    bound = 4e-6 * (np.abs(a.astype(np.float64)) @ np.abs(w.astype(np.float64)).T) + 1e-7
    err = np.abs(got - ref)
    assert np.all(err <= bound), float((err / bound).max())
    base = rng.standard_normal((m, n)).astype(np.float32)
    acc = qpkg.gemm(a, w, base)
    assert np.array_equal(acc, (base + got).astype(np.float32))


@pytest.mark.gpu
def test_gemm_range_guard(qpkg):
    """Rows holding values far beyond FP16's range (up to 3e6; FP16 ends at
    65504) are split as a * 2^-e and scaled back (engine/core.cpp:292-294
    multiplies FP32 activations): within the FP64 bound, while rows that fit
    FP16 keep the bits they have in a call where no row is scaled, through
    the allocating and the static entry points."""
    rng = np.random.default_rng(31)
    a = rng.standard_normal((300, 1024), dtype=np.float32)
    big = np.arange(0, 300, 7)
    a[big, 5] = 3e6
    a[big[::2], 900] = -7e4
    a[11, :] *= 40000.0
    w = (rng.standard_normal((1024, 1024), dtype=np.float32) * 0.02).astype(np.float16)
    ref = a.astype(np.float64) @ w.astype(np.float64).T
    bound = 4e-6 * (np.abs(a.astype(np.float64)) @ np.abs(w.astype(np.float64)).T) + 1e-7
    fits = np.setdiff1d(np.arange(300), np.r_[big, 11])
    alone = qpkg.gemm(a[fits], w)
    for got in (qpkg.gemm(a, w), qpkg.gemm_static(a, w)):
        assert np.isfinite(got).all()
        err = np.abs(got - ref)
        assert np.all(err <= bound), float((err / bound).max())
        assert np.array_equal(got[fits].view(np.uint32), alone.view(np.uint32))


@pytest.mark.gpu
@pytest.mark.parametrize('m,amp', [(1024, 1.0), (100, 1.0), (3968, 1.0), (1024, 200.0), (100, 200.0)])
def test_gemm_swiglu_against_fp64(qpkg, m, amp):
    """The gate/up GEMM with its SwiGLU epilogue (engine/core.cpp:630-639 at
    batch > 1). 1024 rows take 128 x 192 tiles (256 workgroups in one round),
    100 rows narrower 32- or 64-row tiles and 3968 rows 128 x 256 tiles, so
    each epilogue's gate/up column mapping is exercised. Against FP64:
    g sigmoid(g) u with g, u the exact products, the GEMM error bound
    propagated through the activation's partial derivatives, plus the FP16
    hi + lo rounding of the stored result. With amp = 200 many activations
    lie beyond FP16's range: their groups of 8 carry exponents (the others
    keep 0, and so does every group at amp = 1)."""
    rng = np.random.default_rng(23 + m)
    a = rng.standard_normal((m, 1024), dtype=np.float32) * np.float32(amp)
    w = (rng.standard_normal((6144, 1024), dtype=np.float32) * 0.02).astype(np.float16)
    # Every column, every third row plus the last (the FP64 products of all
    # 3968 rows would dominate the test's time).
    rows = np.r_[0:m:3, m - 1]
    got, exps = qpkg.gemm_swiglu(a, w, exponents=True)
    got = got.astype(np.float64)[rows]
    if amp == 1.0:
        assert not exps.any()
    else:
        assert 0.005 < (exps > 0).mean() < 0.995, float((exps > 0).mean())
        assert np.isfinite(got).all()
    a64, w64 = a[rows].astype(np.float64), w.astype(np.float64)
    g, u = a64 @ w64[:3072].T, a64 @ w64[3072:].T
    sig = 1.0 / (1.0 + np.exp(-g))
    ref = g * sig * u
    bg = 4e-6 * (np.abs(a64) @ np.abs(w64[:3072]).T) + 1e-7
    bu = 4e-6 * (np.abs(a64) @ np.abs(w64[3072:]).T) + 1e-7
    # The last terms: the FP32 formula's own rounding (2^-23 |g u| also covers
    # the reference's 0.5 + 0.5 tanh(g / 2) for tanh near -1).
    bound = (np.abs(sig * (1.0 + g * (1.0 - sig)) * u) * bg + np.abs(g * sig) * bu
             + 1e-6 * np.abs(ref) + 2.0 ** -23 * np.abs(g * u) + 1e-8)
    # The epilogue itself: the plain GEMM accumulates every element in the
    # same K order, so its g and u are the ones the SwiGLU epilogue saw. The
    # activation must be the reference formula evaluated in FP32 on them, up
    # to what two evaluations of the sigmoid differ by (the reference's form
    # rounds at 2^-24 absolute) and what FP16 hi + lo holds (2^-22 relative,
    # half of FP16's subnormal spacing absolute). A hi / lo pair rounded from
    # two different values misses this by an FP16 ulp.
    plain = qpkg.gemm(a, w)[rows]
    g32, u32 = plain[:, :3072], plain[:, 3072:]
    t32 = np.tanh(np.float32(0.5) * g32).astype(np.float32)
    emu = (g32 * (np.float32(0.5) + np.float32(0.5) * t32) * u32).astype(np.float64)
    tol = (np.abs(g32.astype(np.float64) * u32) * 2.0 ** -23 + 4 * np.spacing(np.abs(emu).astype(np.float32))
           + 2.0 ** -21 * np.abs(emu) + 2.0 ** -24)
    assert np.all(np.abs(got - emu) <= tol), float((np.abs(got - emu) / tol).max())
    err = np.abs(got - ref)
    worst = np.unravel_index(np.argmax(err / bound), err.shape)
    assert np.all(err <= bound), dict(ratio=float((err / bound).max()), row=int(rows[worst[0]]), col=int(worst[1]),
                                      g=float(g[worst]), u=float(u[worst]), got=float(got[worst]),
                                      ref=float(ref[worst]), bound=float(bound[worst]))


@pytest.mark.gpu
@pytest.mark.parametrize('width', [0.5, 4.0, 16.0])
def test_gemm_swiglu_sigmoid(qpkg, width):
    """The sigmoid of the SwiGLU epilogue against FP64, without the GEMM's error:
    one gate per row (A's column 0 times 1, exact), up a power of two. Half of
    the results leave FP16 hi + lo unrounded (|lo| below a quarter of hi's
    spacing); only those count. Relative to the result, in units of 2^-24: the
    quotient and the product with the gate round once each (1), exp2 errs by
    one ulp (2) and its argument by 1.22 |g| (its rounding, and that of
    log2(e)), the last two times 1 - sigmoid. Around 0 the rms of three such
    independent errors is 4.2e-8 (a rounding to nearest has 0.41 x 2^-24, over
    one binade; exp2's ulp counts half); a further one, as of 1 + e, gives 4.9e-8."""
    m, n, k = 8192, 256, 64
    rng = np.random.default_rng(7)
    step = 2.0 ** -19 * width  # 21 bits: hi + lo holds the gate exactly
    gate = np.round(rng.uniform(-width, width, m) / step) * step
    gate[np.abs(gate) < width / 64] = width / 64
    sig = 1.0 / (1.0 + np.exp(-gate))
    up = np.exp2(np.clip(6 - np.floor(np.log2(np.abs(gate * sig))), -14, 15))
    a = np.zeros((m, k), np.float32)
    a[:, 0], a[:, 1] = gate, up
    assert np.array_equal(a[:, 0].astype(np.float64), gate)
    w = np.zeros((n, k), np.float16)
    w[:n // 2, 0] = 1
    w[n // 2:, 1] = 1
    act = qpkg.gemm_swiglu(a, w)
    assert np.array_equal(act, np.repeat(act[:, :1], n // 2, 1))
    act, ref = act[:, 0], gate * sig * up
    lo = act - act.astype(np.float16).astype(np.float32)
    kept = (np.abs(lo) < np.spacing(act.astype(np.float16)).astype(np.float32) / 4) & (np.abs(ref) > 1)
    assert kept.mean() > 0.3
    err = (np.abs(act - ref) / np.abs(ref) * 2.0 ** 24)[kept]
    bound = (1 - sig) * (2 + 1.22 * np.abs(gate)) + 2.1
    assert np.all(err <= bound[kept]), float((err / bound[kept]).max())
    if width <= 0.5:
        assert np.sqrt(np.mean(err ** 2)) * 2.0 ** -24 < 4.25e-8, float(np.sqrt(np.mean(err ** 2)) * 2.0 ** -24)


def causal_attention_fp64(q, keys, values, pos0):
    """softmax(q k^T / sqrt(128)) v per query head over positions 0..pos0 + i,
    query head h reading KV head h // 2 (engine/core.cpp:407-605), in FP64."""
    rows = q.shape[0]
    out = np.empty((rows, 16, 128))
    k64, v64 = keys.astype(np.float64), values.astype(np.float64)
    for i in range(rows):
        n = pos0 + i + 1
        for h in range(16):
            s = k64[h // 2, :n] @ q[i, h].astype(np.float64) / np.sqrt(128.0)
            p = np.exp(s - s.max())
            out[i, h] = (p @ v64[h // 2, :n]) / p.sum()
    return out.reshape(rows, 2048)


@pytest.mark.gpu
@pytest.mark.parametrize('rows,pos0,boost', [(1, 0, False), (45, 0, True), (130, 200, True), (300, 37, False),
                                             (300, 37, True)])
def test_attention_prefill_against_fp64(qpkg, rows, pos0, boost):
    """The prefill attention kernel against an FP64 causal softmax. With
    `boost`, keys at positions 40, 97, 170 and 300 align with a direction
    every query shares, so their scores beat all earlier ones by about 14, 28,
    42 and 56 (natural log units), far past the kernel's lazy-rescale margin.
    Keys 170 and 300 lie in the second and third tiles of key split 1 (tiles
    of 32 keys, split = tile % 4), so the cases past 170 positions rescale a
    running output and sum mid-sequence: a CPU emulation of the kernel's
    order without that rescale misses these two cases by 3.6 and 4.5."""
    rng = np.random.default_rng(rows + pos0)
    context = pos0 + rows + 7
    u = rng.standard_normal(128)
    u *= 4.0 / np.linalg.norm(u)
    q = (u + 0.5 * rng.standard_normal((rows, 16, 128))).astype(np.float32)
    keys = (0.3 * rng.standard_normal((8, context, 128))).astype(np.float16)
    values = rng.standard_normal((8, context, 128)).astype(np.float16)
    if boost:
        for t, alpha in ((40, 10.0), (97, 20.0), (170, 30.0), (300, 40.0)):
            if t < pos0 + rows:
                keys[:, t] = (alpha * u).astype(np.float16)
    qkv = np.zeros((rows, 4096), np.float32)
    qkv[:, :2048] = q.reshape(rows, 2048)
    got = qpkg.attention_prefill(qkv, keys, values, pos0)
    ref = causal_attention_fp64(q, keys, values, pos0)
    err = np.abs(got - ref)
    assert np.all(err <= 1e-4 + 1e-4 * np.abs(ref)), float(err.max())


@pytest.mark.gpu
def test_attention_prefill_range_guard(qpkg):
    """Queries with a channel far beyond FP16's range (4e6 before the
    kernel's scale * log2(e), against keys that are 0 in that channel, so the
    scores stay moderate): the kernel splits such a query as q * 2^-e and
    scales its scores back, within the same FP64 tolerance as plain
    queries."""
    rng = np.random.default_rng(77)
    rows, pos0 = 70, 30
    context = pos0 + rows
    q = rng.standard_normal((rows, 16, 128)).astype(np.float32)
    q[::3, :, 17] = 4e6
    q[1::5, 2, 90] = -9e5
    keys = (0.3 * rng.standard_normal((8, context, 128))).astype(np.float16)
    keys[:, :, 17] = 0
    keys[:, :, 90] = 0
    values = rng.standard_normal((8, context, 128)).astype(np.float16)
    qkv = np.zeros((rows, 4096), np.float32)
    qkv[:, :2048] = q.reshape(rows, 2048)
    got = qpkg.attention_prefill(qkv, keys, values, pos0)
    ref = causal_attention_fp64(q, keys, values, pos0)
    err = np.abs(got - ref)
    assert np.all(err <= 1e-4 + 1e-4 * np.abs(ref)), float(err.max())


@pytest.mark.gpu
def test_gemm_rows_independent_of_chunk(qpkg):
    """Row results do not depend on M, on the row's position in a tile or on
    the tile height chosen for the launch (128-row tiles for 1200 x 4096,
    64-row tiles for the smaller calls)."""
    rng = np.random.default_rng(22)
    a = rng.standard_normal((1200, 1024), dtype=np.float32)
    w = (rng.standard_normal((4096, 1024), dtype=np.float32) * 0.02).astype(np.float16)
    full = qpkg.gemm(a, w)
    for rows in (slice(0, 37), slice(100, 101), slice(300, 512), slice(1100, 1200)):
        part = qpkg.gemm(a[rows], w)
        assert np.array_equal(part.view(np.uint32), full[rows].view(np.uint32))


@pytest.mark.gpu
def test_prefill_1024_matches_oracle(qpkg, pack0, oracle_lib):
    """The 1024-token prompt (seed 2): two full 512-row chunks."""
    prompt = PROMPTS['prefill_1024']
    with qpkg.Model(pack0) as gpu:
        oracle = oracle_lib.model(pack0, 16, 16, 4096)
        try:
            gpu.prefill(prompt)
            oracle.prefill(prompt)
            result = compare_logits(gpu.logits(), oracle.logits())
            print(result)
            assert result['passed'], result
            for _ in range(3):
                token = gpu.greedy()
                gpu.step(token)
                oracle.step(token)
                result = compare_logits(gpu.logits(), oracle.logits())
                assert result['passed'], result
        finally:
            oracle.close()


@pytest.mark.gpu
def test_canonical_prefix_reuse_equals_fresh(qpkg, pack0):
    """Rewind to a 512 boundary and prefill the rest == one fresh prefill
    (chunk shapes match; INTERFACE.md:94-111, tools/check_native_cpu_prefix.py)."""
    prompt = PROMPTS['long_3968'][:1100]
    with qpkg.Model(pack0) as m:
        m.prefill(prompt)
        fresh = (m.logits(), m.hidden())
        m.step(7)
        m.truncate(512)
        m.prefill(prompt[512:])
        assert np.array_equal(m.logits().view(np.uint32), fresh[0].view(np.uint32))
        assert np.array_equal(m.hidden().view(np.uint32), fresh[1].view(np.uint32))
        m.reset()
        m.prefill(prompt[:1024])
        m.truncate(1024)
        m.prefill(prompt[1024:])
        assert np.array_equal(m.logits().view(np.uint32), fresh[0].view(np.uint32))


@pytest.mark.gpu
def test_prefill_rows_independent_of_grouping(qpkg, pack0):
    """A call runs its consecutive 512-row chunks as one batched pass; that is
    only legal because every batched row is computed alone. Any split of a
    prompt into calls of two or more rows must give the same bits, and a
    trailing one-row chunk takes the batch-1 path like a step
    (engine/core.cpp:712)."""
    prompt = PROMPTS['long_3968'][:1025]
    with qpkg.Model(pack0) as m:
        m.prefill(prompt[:700])
        whole = m.logits().view(np.uint32).copy()
        m.reset()
        m.prefill(prompt[:300])
        m.prefill(prompt[300:700])
        assert np.array_equal(m.logits().view(np.uint32), whole)
        m.reset()
        m.prefill(prompt)  # 1024 batched rows + one batch-1 row
        tail = m.logits().view(np.uint32).copy()
        m.reset()
        m.prefill(prompt[:1024])
        m.step(prompt[1024])
        assert np.array_equal(m.logits().view(np.uint32), tail)


@pytest.mark.gpu
@pytest.mark.parametrize('n,k', [(1024, 1024), (4096, 1024), (1024, 3072), (6144, 64)])
def test_gemm_tile_edges(qpkg, n, k):
    """Row counts at the edges of every tile height (16, 32, 48, 64, 96, 128) and
    of the rounds that choose between them: each call's rows must be the bits of
    one 700-row call (whatever tile either takes, every element adds its K
    terms in one order), which in turn meets the FP64 bound. K = 64 is a
    single LDS stage."""
    rng = np.random.default_rng(n + k)
    a = rng.standard_normal((700, k), dtype=np.float32)
    w = (rng.standard_normal((n, k), dtype=np.float32) * 0.02).astype(np.float16)
    full = qpkg.gemm(a, w)
    bound = 4e-6 * (np.abs(a.astype(np.float64)) @ np.abs(w.astype(np.float64)).T) + 1e-7
    assert np.all(np.abs(full - a.astype(np.float64) @ w.astype(np.float64).T) <= bound)
    for m in (1, 15, 16, 17, 31, 32, 33, 47, 48, 49, 63, 64, 65, 95, 96, 97, 127, 128, 129, 143, 144, 145, 191, 192, 193,
              255, 256, 257, 288, 289, 321, 481, 513, 576, 577):
        first = (37 * m) % (700 - m)
        got = qpkg.gemm(a[first:first + m], w)
        assert np.array_equal(got.view(np.uint32), full[first:first + m].view(np.uint32)), m


@pytest.mark.gpu
def test_gemm_swiglu_tile_edges(qpkg):
    """The same for the SwiGLU epilogue (gate and up columns of one tile), with
    rows whose activations carry exponents among them. Tiles of 16 x 32 (up to
    16 rows) to 128 x 192 (641), 128 x 256 (1025) and 96 x 192 (1281 to 1536)."""
    rng = np.random.default_rng(61)
    a = rng.standard_normal((1500, 1024), dtype=np.float32)
    a[::5] *= np.float32(300)
    w = (rng.standard_normal((6144, 1024), dtype=np.float32) * 0.02).astype(np.float16)
    full, exps = qpkg.gemm_swiglu(a, w, exponents=True)
    assert exps.any() and not exps.all() and np.isfinite(full).all()
    for m in (1, 16, 17, 32, 33, 64, 65, 96, 97, 128, 129, 144, 145, 192, 193, 256, 257, 288, 289, 320, 321, 480, 481, 640,
              641, 1024, 1025, 1281, 1344, 1345):
        first = (37 * m) % (1500 - m)
        got, e = qpkg.gemm_swiglu(a[first:first + m], w, exponents=True)
        assert np.array_equal(got.view(np.uint32), full[first:first + m].view(np.uint32)), m
        assert np.array_equal(e, exps[first:first + m]), m


@pytest.mark.gpu
@pytest.mark.parametrize('calls', [(2, 16, 17, 33, 65, 130, 137, 300), (96, 200, 404), (144, 556)])
def test_prefill_rows_independent_of_tile(qpkg, pack0, calls):
    """The QKV epilogue (a head per tile of 16 rows up to 128, of 32 up to 256, 48
    up to 384, 64 up to 512, 96 up to 576, then 128) and the K-split GEMMs (tiles of
    16 x 32 to 128 x 128, each in one of these calls): the logits of one 700-row
    call."""
    prompt = PROMPTS['long_3968'][:700]
    with qpkg.Model(pack0) as m:
        m.prefill(prompt)
        whole = m.logits().view(np.uint32).copy()
        m.reset()
        at = 0
        for rows in calls:
            m.prefill(prompt[at:at + rows])
            at += rows
        assert at == 700
        assert np.array_equal(m.logits().view(np.uint32), whole)


@pytest.mark.gpu
def test_attention_prefill_tile_counts(qpkg):
    """Every residue of the key-tile count modulo the 4 key splits (1 to 9 tiles
    of 32 keys, the last one whole or ragged; with 1 to 3 tiles some splits
    have none), a diagonal inside a tile and on its edge, one to 65 queries:
    against FP64, and bit for bit against the same queries at the end of a
    longer call (a query's key order depends on its position alone)."""
    rng = np.random.default_rng(91)
    context = 300
    keys = (0.3 * rng.standard_normal((8, context, 128))).astype(np.float16)
    values = rng.standard_normal((8, context, 128)).astype(np.float16)
    qkv = np.zeros((context, 4096), np.float32)
    qkv[:, :2048] = 3 * rng.standard_normal((context, 2048)).astype(np.float32)
    whole = qpkg.attention_prefill(qkv, keys, values, 0)
    for end in (1, 31, 32, 33, 64, 65, 96, 97, 128, 129, 160, 192, 200, 255, 256, 257, 288, 300):
        for rows in (1, 2, 31, 32, 33, 65):
            if rows > end:
                continue
            pos0 = end - rows
            got = qpkg.attention_prefill(qkv[pos0:end], keys[:, :end], values[:, :end], pos0)
            assert np.array_equal(got.view(np.uint32), whole[pos0:end].view(np.uint32)), (pos0, rows)
    ref = causal_attention_fp64(qkv[:, :2048].reshape(context, 16, 128), keys, values, 0)
    err = np.abs(whole - ref)
    assert np.all(err <= 1e-4 + 1e-4 * np.abs(ref)), float(err.max())


@pytest.mark.gpu
@pytest.mark.parametrize('rows,end', [(rows, end) for rows in (1, 32, 481, 512, 513)
                                      for end in (1, 33, 97, 512, 1024, 1025) if rows <= end])
def test_attention_prefill_head_split(qpkg, rows, end):
    """Up to 16 query blocks and 1024 keys a workgroup runs one query head,
    beyond that both heads of a KV head: bit for bit the same rows out of a
    call of 1100 rows (a head's key order and arithmetic do not depend on it)."""
    rng = np.random.default_rng(92)
    keys = (0.3 * rng.standard_normal((8, 1100, 128))).astype(np.float16)
    values = rng.standard_normal((8, 1100, 128)).astype(np.float16)
    qkv = np.zeros((1100, 4096), np.float32)
    qkv[:, :2048] = 3 * rng.standard_normal((1100, 2048)).astype(np.float32)
    whole = qpkg.attention_prefill(qkv, keys, values, 0)
    got = qpkg.attention_prefill(qkv[end - rows:end], keys[:, :end], values[:, :end], end - rows)
    assert np.array_equal(got.view(np.uint32), whole[end - rows:end].view(np.uint32))


@pytest.mark.gpu
def test_prefill_fold_order(qpkg, pack0, tmp_path):
    """O and down add their 4 K ranges as (p0 + p1) + (p2 + p3), in the row
    kernels (up to 1024 rows) and in the folding GEMMs (64-, 96- and 128-row
    tiles). Layer 0 is built for exact partials: all queries and keys 0, so
    every score is 0, all values 1, so the attention output is 1, and O rows of
    even channels 1024, 2^-14, 2^-14 and -1024 in the four ranges. In pairs that
    is 2^-14; 1024 + 2^-14 is a tie that rounds to 1024, so one after the other
    it is 0. Nothing else adds to the residual, which starts at 1."""
    path = tmp_path / 'weights.bin'
    shutil.copyfile(pack0, path)
    shutil.copyfile(str(pack0) + '.index', str(path) + '.index')
    blob = np.memmap(path, np.uint8, 'r+')
    tensors = {}
    for line in Path(str(path) + '.index').read_text().splitlines()[1:]:
        name, kind, rows, cols, offset, length = line.split()
        if kind == 'F16':
            tensors[name] = blob[int(offset):int(offset) + int(length)].view('<f2').reshape(int(rows), int(cols))
    for layer in range(28):
        tensors[f'model.layers.{layer}.self_attn.o_proj.weight'][:] = 0
        tensors[f'model.layers.{layer}.mlp.down_proj.weight'][:] = 0
    first = 'model.layers.0.self_attn.'
    for name in ('q', 'k', 'v'):
        tensors[first + name + '_proj.weight'][:] = 0
    tensors[first + 'v_proj.weight'][:, 0] = 1
    tensors[first + 'o_proj.weight'][::2, ::512] = [1024, 2.0 ** -14, 2.0 ** -14, -1024]
    tensors['model.embed_tokens.weight'][0] = 1
    blob.flush()
    del tensors, blob
    with qpkg.Model(path) as m:
        for rows in (2, 85, 1024, 1100, 2100, 3100):
            m.reset()
            m.prefill([0] * rows)
            hidden = m.hidden().astype(np.float64)
            assert np.allclose(hidden[::2] / hidden[1], 1 + 2.0 ** -14, rtol=2.0 ** -22, atol=0), rows
            assert np.all(hidden[1::2] == hidden[1]), rows


@pytest.mark.gpu
@pytest.mark.parametrize('rows', [1100, 2100, 3100])
def test_prefill_folding_gemms(qpkg, pack0, rows):
    """Beyond 1024 rows the O and down GEMMs add their 4 K ranges themselves
    (64-row tiles, 96-row tiles from 2049 rows, 128-row tiles from 3073): the
    bits of calls of at most 1024 rows, whose ranges the row kernels add."""
    prompt = PROMPTS['long_3968'][:rows]
    with qpkg.Model(pack0) as m:
        m.prefill(prompt)
        whole = m.logits().view(np.uint32).copy()
        m.reset()
        for at in range(0, rows, 700):
            m.prefill(prompt[at:at + 700])
        assert np.array_equal(m.logits().view(np.uint32), whole)


@pytest.mark.gpu
def test_prefill_folding_gemms_range_guard(qpkg, tmp_path):
    """The same with activations past FP16's range (norm gains of 32768 in 8
    channels): the folding down GEMM, with tiles of 64, 96 and 128 rows, rescales
    each K range of a flagged row by that range's exponent, as the ranged one
    does."""
    import test_export
    path = test_export.write_full_checkpoint(tmp_path / 'model.safetensors', gains=test_export.LARGE_GAINS)
    out = tmp_path / 'pack' / 'weights.bin'
    test_export.export_pack.write_pack(path, out)
    path.unlink()
    with qpkg.Model(out, context=3200) as m:
        for rows in (1100, 2100, 3100):
            prompt = PROMPTS['long_3968'][:rows]
            m.reset()
            m.prefill(prompt)
            whole = m.logits().view(np.uint32).copy()
            assert np.isfinite(whole.view(np.float32)).all()
            m.reset()
            for at in range(0, rows, 500):
                m.prefill(prompt[at:at + 500])
            assert np.array_equal(m.logits().view(np.uint32), whole), rows


@pytest.mark.gpu
def test_gemm_rows_far_apart(qpkg):
    """W rows of 70 million halves: rows 31, 63, 95 and 127 of W begin 4.34 GB
    behind the first row of their tile, past a 32-bit byte offset. Row n holds
    n + 1 in column K - 1 - n alone and A ones in the last 128 columns, so the
    products are 1 .. 128 exactly."""
    n, k = 128, 70_000_000 // 64 * 64
    a = np.zeros((1, k), np.float32)
    a[0, -n:] = 1
    ad, wd, cd = qpkg.DeviceBuffer.from_array(a), qpkg.DeviceBuffer(n * k * 2), qpkg.DeviceBuffer(n * 4)
    lib, base = qpkg.load_library(), wd.ptr.value
    zeros = np.zeros(1 << 28, np.uint8)
    for at in range(0, n * k * 2, zeros.size):
        qpkg._check(lib.qwen_gpu_memcpy_to_device(base + at, zeros.ctypes.data, min(zeros.size, n * k * 2 - at)))
    for row in range(n):
        value = np.full(1, row + 1, np.float16)
        qpkg._check(lib.qwen_gpu_memcpy_to_device(base + 2 * (row * k + k - 1 - row), value.ctypes.data, 2))
    qpkg._check(lib.qwen_gpu_op_gemm(ad.ptr, wd.ptr, cd.ptr, 1, n, k, 0, None))
    qpkg.synchronize()
    assert np.array_equal(cd.to_array(np.float32, n), np.arange(1, n + 1, dtype=np.float32))


@pytest.mark.gpu
@pytest.mark.parametrize('m,k', [(3, 64), (37, 1024), (5, 4160)])
def test_gemm_operand_alignment(qpkg, m, k):
    """A may begin at any float: the bits of the call whose A begins on 16 bytes,
    through the entry that allocates and the one that does not (rows held in
    registers up to 4096 columns, read twice beyond)."""
    rng = np.random.default_rng(m)
    a = rng.standard_normal((m, k), dtype=np.float32)
    w = (rng.standard_normal((128, k), dtype=np.float32) * 0.02).astype(np.float16)
    expected = qpkg.gemm(a, w).view(np.uint32)
    wd, cd, lib = qpkg.DeviceBuffer.from_array(w), qpkg.DeviceBuffer(m * 128 * 4), qpkg.load_library()
    for shift in (1, 2, 3):
        ad = qpkg.DeviceBuffer.from_array(np.r_[np.full(shift, np.nan, np.float32), a.ravel()])
        for entry in (lib.qwen_gpu_op_gemm, lib.qwen_gpu_op_gemm_static):
            qpkg._check(entry(ad.ptr.value + 4 * shift, wd.ptr, cd.ptr, m, 128, k, 0, None))
            qpkg.synchronize()
            assert np.array_equal(cd.to_array(np.uint32, m * 128).reshape(m, 128), expected), shift


@pytest.mark.gpu
def test_sequence_memory(qpkg, pack0):
    """Device memory of one further sequence at 4096 positions: 448 MiB of K/V and
    44 KiB per prefill row (176 MiB), partial products for 1024 rows only (16
    MiB), and a few MiB of logits and exchange words."""
    def free():
        left, total = ctypes.c_size_t(), ctypes.c_size_t()
        assert qpkg.load_library().hipMemGetInfo(ctypes.byref(left), ctypes.byref(total)) == 0
        return left.value
    # The runtime may hand out memory that it kept from earlier frees: the
    # largest of three.
    with qpkg.Model(pack0, context=16) as owner:
        sequences, used = [], []
        for _ in range(3):
            before = free()
            sequences.append(owner.share(context=4096))
            used.append((before - free()) / 2 ** 20)
        for sequence in sequences:
            sequence.close()
    print(used)
    assert max(used) < 665, used
