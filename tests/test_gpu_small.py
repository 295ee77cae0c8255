"""The few-row GEMMs (gemm_small.hip) at the edges of their tiles and shares.

M covers the 16-, 32- and 64-row tiles and their remainders, N the column tiles
with a ragged last one (and grids that send a mode to its next tile or to the
tiled kernels), K one element, less than one 64-byte step, steps that leave
waves without a share, ragged ends and the deep linears.
"""
import dataclasses

import numpy as np
import pytest

from oracle import oracle as O
from rembed_amd import _lib
from rembed_amd import tensor as T
from rembed_amd.model import Model
from rembed_amd.synthetic import GEMMA3_300M, BertShape, bert_tensors, decoder_tensors

pytestmark = pytest.mark.gpu

SHAPES = [(1, 1, 16), (1, 768, 2304), (15, 30, 48), (16, 64, 256), (17, 65, 272), (28, 768, 768),
          (31, 200, 4112), (32, 129, 1040), (33, 3072, 768), (45, 1024, 6144), (63, 384, 1536),
          (64, 1536, 384), (64, 96, 8208)]
# more rows, int8 only: 64x32 and 64x64 tiles, full and ragged
INT8_SHAPES = [(65, 768, 3072), (200, 320, 2000), (349, 3072, 768), (1213, 768, 768),
               (1024, 80, 1040)]


def say(*a):
    print(*a, flush=True)


def rows(rng, m, k):
    return (rng.standard_normal((m, k)) * np.exp(rng.uniform(-2, 2, (m, 1)))).astype(np.float32)


@pytest.mark.parametrize("shape", SHAPES + INT8_SHAPES)
def test_int8_bit_exact(gpu_ctx, shape):
    m, k, n = shape
    say(f"few-row int8 m={m} k={k} n={n}")
    rng = np.random.default_rng(m + 3 * k + 5 * n)
    a = rows(rng, m, k)
    bT = (rng.standard_normal((n, k)) * 0.05).astype(np.float32)
    bias = rng.standard_normal(n).astype(np.float32)
    pb = T.PackB8VNNI(gpu_ctx, bT, k, n, bias)
    got, (qa, rs) = T.matmul_host(gpu_ctx, a, pb)
    _, q, sc, cs = O.pack_b8_vnni(bT, k, n)
    want, qa_o, _, acc_o = O.matmul_vnni(a, q, cs, sc)
    assert np.array_equal(qa[:, :k], qa_o)
    assert np.array_equal(got, want)
    # the raw accumulators, and bias + GELU in the epilogue
    ldq = T.ldq_for(k)
    dq, dacc = gpu_ctx.upload(qa), gpu_ctx.alloc(m * n * 4)
    T.GemmU8S8I32(gpu_ctx, dacc, dq, ldq, pb, m)
    gpu_ctx.sync()
    assert np.array_equal(dacc.download(np.int32, (m, n)), acc_o)
    got, _ = T.matmul_host(gpu_ctx, a, pb, act=_lib.RH_ACT_GELU)
    assert np.array_equal(got, O.gelu_ref(want + bias))
    # and the row-quantizing epilogues
    st = rng.integers(1, 255, (m, ldq), dtype=np.uint8)
    qo, rso, mx = gpu_ctx.upload(st), gpu_ctx.alloc(m * 4), gpu_ctx.alloc(m * 4)
    ldo = T.ldq_for(n)
    out = gpu_ctx.alloc(m * ldo)
    T.LinearU8(gpu_ctx, dq, ldq, gpu_ctx.upload(rs), pb, m, _lib.RH_ACT_GELU, out, ldo, rso, mx)
    gpu_ctx.sync()
    pairs = [O.quantize_row_u8(r) for r in got]
    assert np.array_equal(out.download(np.uint8, (m, ldo))[:, :n], np.stack([p[0] for p in pairs]))
    assert np.array_equal(rso.download(np.float32, (m,)),
                          np.array([p[1] for p in pairs], np.float32))
    del qo


@pytest.mark.parametrize("mode", ["w8", "fp32"])
@pytest.mark.parametrize("terms", [1, 2])
@pytest.mark.parametrize("shape", SHAPES)
def test_planes_against_float64(gpu_ctx, shape, terms, mode):
    if mode == "fp32" and terms == 1:
        pytest.skip("fp32 always takes two terms")
    m, k, n = shape
    say(f"few-row {mode} terms={terms} m={m} k={k} n={n}")
    rng = np.random.default_rng(m + 3 * k + 5 * n + terms)
    a = rows(rng, m, k)
    bT = (rng.standard_normal((n, k)) * 0.05).astype(np.float32)
    bias = rng.standard_normal(n).astype(np.float32)
    gpu_ctx.set_option(_lib.RH_CTX_W8_TERMS, terms)
    try:
        if mode == "w8":
            pb = T.PackB8(gpu_ctx, bT, k, n, bias)
            q, sc, _ = pb.export()
            w = q.astype(np.float64) * sc.astype(np.float64)[:, None]
        else:
            pb = T.PackB(gpu_ctx, bT, k, n, bias)
            w = bT.astype(np.float64)
        got = T.matmul_host(gpu_ctx, a, pb)
    finally:
        gpu_ctx.set_option(_lib.RH_CTX_W8_TERMS, 1)
    a64 = a.astype(np.float64)
    want = a64 @ w.T
    # |error| <= sum |a||w| · (operand rounding + the fp32 sum's): one bf16 term
    # (8 significant bits) is off by 2^-8 of a value at most, two by 2^-16 (and the
    # dropped lo·lo product, and w's own split); K fp32 additions in any order by K · 2^-24
    eps = 2.0 ** -8 if terms == 1 else 3 * 2.0 ** -16
    bound = (np.abs(a64) @ np.abs(w).T) * (eps + k * 2.0 ** -24) + 1e-30
    assert np.all(np.abs(got - want) <= bound)


@pytest.mark.parametrize("mode", ["w8", "fp32"])
@pytest.mark.parametrize("terms", [1, 2])
@pytest.mark.parametrize("shape", [(1, 768, 768), (17, 40, 48), (33, 3072, 256), (45, 130, 512),
                                   (200, 768, 272)])
def test_planes_rows_equal_the_tiled_kernels(gpu_ctx, shape, terms, mode):
    """A row's result does not depend on the rows computed with it: the same
    bits as a forced tile of the tiled kernel."""
    if mode == "fp32" and terms == 1:
        pytest.skip("fp32 always takes two terms")
    m, k, n = shape
    say(f"few-row vs tiled {mode} terms={terms} m={m} k={k} n={n}")
    rng = np.random.default_rng(m + k + n)
    a = rows(rng, m, k)
    bT = (rng.standard_normal((n, k)) * 0.05).astype(np.float32)
    pb = T.PackedWeight(gpu_ctx, 1 if mode == "w8" else 0, bT, k, n,
                        rng.standard_normal(n).astype(np.float32))
    gpu_ctx.set_option(_lib.RH_CTX_W8_TERMS, terms)
    try:
        got = T.matmul_host(gpu_ctx, a, pb, act=_lib.RH_ACT_GELU)
        gpu_ctx.set_option(_lib.RH_CTX_BF_TILE, 8)
        want = T.matmul_host(gpu_ctx, a, pb, act=_lib.RH_ACT_GELU)
    finally:
        gpu_ctx.set_option(_lib.RH_CTX_BF_TILE, 0)
        gpu_ctx.set_option(_lib.RH_CTX_W8_TERMS, 1)
    assert np.array_equal(got, want)


@pytest.mark.parametrize("act", [_lib.RH_ACT_SWIGLU, _lib.RH_ACT_GEGLU, _lib.RH_ACT_GEGLU_ERF])
@pytest.mark.parametrize("mode", [0, 1, 2])
@pytest.mark.parametrize("shape", [(1, 768, 64), (17, 72, 1040), (45, 1024, 3072), (64, 768, 1152),
                                   (100, 768, 3072)])
def test_gated_equals_the_tiled_kernels(gpu_ctx, shape, mode, act):
    """act(gate)·up in the epilogue: the same bits as a forced tile."""
    m, k, i = shape
    say(f"few-row gated mode={mode} act={act} m={m} k={k} i={i}")
    rng = np.random.default_rng(m + k + i + act)
    pg = T.PackedGated(gpu_ctx, mode, (rng.standard_normal((i, k)) * 0.05).astype(np.float32),
                       (rng.standard_normal((i, k)) * 0.05).astype(np.float32), k, i)
    da, dst = gpu_ctx.upload(rows(rng, m, k)), gpu_ctx.alloc(m * i * 4)
    ldq = T.ldq_for(k)
    qa, rs = gpu_ctx.alloc(m * ldq), gpu_ctx.alloc(m * 4)
    option, tile = (_lib.RH_CTX_I8_TILE, 3) if mode == 2 else (_lib.RH_CTX_BF_TILE, 8)
    out = []
    for t in (0, tile):
        gpu_ctx.set_option(option, t)
        try:
            T.Linear(gpu_ctx, dst, da, pg, m, act, qa if mode == 2 else None,
                     ldq if mode == 2 else 0, rs if mode == 2 else None)
            gpu_ctx.sync()
        finally:
            gpu_ctx.set_option(option, 0)
        out.append(dst.download(np.float32, (m, i)))
    assert np.array_equal(out[0], out[1])


@pytest.mark.parametrize("n", [384, 768, 1024, 1028, 2048])
def test_row_kernels_few_and_many_rows_agree(gpu_ctx, n):
    """LayerNorm and QuantizeRowU8 of the same rows in a call of one row, of the
    most rows that run one per wave (2048) and of one more: the same bits, and
    the quantizer's equal the oracle's."""
    say(f"row kernels n={n}")
    rng = np.random.default_rng(n)
    m = 2049
    x = rows(rng, m, n)
    g = gpu_ctx.upload((1 + 0.1 * rng.standard_normal(n)).astype(np.float32))
    b = gpu_ctx.upload(rng.standard_normal(n).astype(np.float32))
    ln, qs = {}, {}
    for k in (1, 2048, m):
        dx = gpu_ctx.upload(x[:k])
        _lib.check(_lib.lib.rh_layernorm(gpu_ctx.h, dx.ptr, g.ptr, b.ptr, k, n, 1e-12))
        ldq = T.ldq_for(n)
        da, dq, ds = gpu_ctx.upload(x[:k]), gpu_ctx.alloc(k * ldq), gpu_ctx.alloc(k * 4)
        T.QuantizeRowsU8(gpu_ctx, da, k, n, dq, ldq, ds)
        gpu_ctx.sync()
        ln[k] = dx.download(np.float32, (k, n))
        qs[k] = dq.download(np.uint8, (k, ldq))[:, :n]
    assert np.array_equal(ln[2048][:1], ln[1]) and np.array_equal(ln[m][:2048], ln[2048])
    assert np.array_equal(qs[2048][:1], qs[1]) and np.array_equal(qs[m][:2048], qs[2048])
    assert np.array_equal(qs[m], np.stack([O.quantize_row_u8(r)[0] for r in x]))


def in_order(terms, dtype):
    """The rows of `terms` added one after the other in dtype, from zero."""
    return np.cumsum(np.concatenate([np.zeros_like(terms[:1]), terms]), axis=0, dtype=dtype)[-1]


def l2(v):
    s = in_order(np.square(v.astype(np.float64)), np.float64)
    return v if s == 0 else v * np.float32(1.0 / np.sqrt(s))


@pytest.mark.parametrize("pooling", [0, 1, 2])
@pytest.mark.parametrize("lens", [[1], [64, 63, 1], [65, 2], [512, 31, 300], [513, 1, 256, 257, 512],
                                  [1030, 768, 33], [520] + [2] * 300])
def test_pooling_in_row_order(gpu_ctx, lens, pooling):
    """Mean (float32, row after row), CLS and last-token pooling and the L2 scale
    of the longest texts of each kernel and one more, and of a long text whose
    batch is too many for the chunked kernel, bit for bit from the token vectors
    of the same forward."""
    say(f"pooling {pooling} lens={lens}")
    shape = BertShape("pool", layers=1, hidden=192, heads=6, intermediate=320, vocab=500,
                      max_position=1032, pooling=pooling, normalize=1)
    m = Model(gpu_ctx, shape, bert_tensors(shape, seed=3), 0)
    rng = np.random.default_rng(len(lens) + pooling)
    ids = rng.integers(0, shape.vocab, (len(lens), max(lens)))
    lens = np.array(lens, np.int32)
    got, tokens = m.embed(ids, lens), m.embed_tokens(ids, lens)
    for b, t in enumerate(tokens):
        v = {0: lambda: in_order(t, np.float32) * (np.float32(1) / np.float32(len(t))),
             1: lambda: t[0], 2: lambda: t[-1]}[pooling]()
        assert np.array_equal(got[b], l2(v)), b


@pytest.mark.parametrize("hidden", [64, 1024, 1088, 2048])
def test_pooling_widths(gpu_ctx, hidden):
    """One column per thread up to 1024 columns, two above, with the last wave
    part empty: mean of short texts and the L2 scale, bit for bit."""
    say(f"pooling hidden={hidden}")
    shape = BertShape("wide", layers=1, hidden=hidden, heads=hidden // 64, intermediate=64,
                      vocab=100, max_position=64, pooling=0, normalize=1)
    m = Model(gpu_ctx, shape, bert_tensors(shape, seed=3), 0)
    lens = np.array([5, 64, 1], np.int32)
    ids = np.random.default_rng(hidden).integers(0, shape.vocab, (3, 64))
    for v, t in zip(m.embed(ids, lens), m.embed_tokens(ids, lens)):
        assert np.array_equal(v, l2(in_order(t, np.float32)
                                    * (np.float32(1) / np.float32(len(t)))))


@pytest.mark.parametrize("batch", [1, 3, 8, 9, 57, 90])
@pytest.mark.parametrize("dense", [32, 300, 1056])
def test_dense_head_in_order(gpu_ctx, batch, dense):
    """EmbeddingGemma's two head products, each output one float32 sum in
    ascending order, bit for bit from the token vectors; widths that leave
    ragged chunks and column tiles, batches around a workgroup's 8 texts and
    past one round of the chip (for the first product, for both)."""
    say(f"dense head batch={batch} dense={dense}")
    shape = dataclasses.replace(GEMMA3_300M, name="head", layers=1, sliding_pattern=1, vocab=500,
                                dense_hidden=dense)
    t = decoder_tensors(shape, seed=5)
    m = Model(gpu_ctx, shape, t, 0)
    rng = np.random.default_rng(batch + dense)
    lens = rng.integers(1, 40, batch).astype(np.int32)
    ids = rng.integers(0, shape.vocab, (batch, int(lens.max())))
    got, tokens = m.embed(ids, lens), m.embed_tokens(ids, lens)
    w1, w2 = t["2_Dense.linear.weight"], t["3_Dense.linear.weight"]
    for b, x in enumerate(tokens):
        v = in_order(x, np.float32) * (np.float32(1) / np.float32(len(x)))
        v = in_order(w1.T * v[:, None], np.float32)
        v = in_order(w2.T * v[:, None], np.float32)
        assert np.array_equal(got[b], l2(v) if shape.normalize else v), b


@pytest.mark.parametrize("rows", [1, 682, 683, 700, 5461, 5462])
def test_token_vectors_of_every_way_out(gpu_ctx, rows):
    """Token vectors that leave through the pinned buffer in one piece (up to
    1 MiB), in four (up to 8 MiB) and straight to the caller's memory: the same
    bits as the texts in small calls (full int8: a row does not depend on the
    batch it is in), and again on a second call."""
    say(f"token vectors rows={rows}")
    shape = BertShape("out", layers=1, hidden=384, heads=12, intermediate=384, vocab=500,
                      max_position=512)
    m = Model(gpu_ctx, shape, bert_tensors(shape, seed=9), 2)
    lens = np.array([512] * (rows // 512) + ([rows % 512] if rows % 512 else []), np.int32)
    rng = np.random.default_rng(rows)
    ids = rng.integers(0, shape.vocab, (len(lens), 512))
    want = [m.embed_tokens(ids[b:b + 1], lens[b:b + 1])[0] for b in range(len(lens))]
    for _ in range(2):
        for a, b in zip(m.embed_tokens(ids, lens), want):
            assert np.array_equal(a, b)


@pytest.mark.parametrize("act", [_lib.RH_ACT_NONE, _lib.RH_ACT_GELU, _lib.RH_ACT_SWIGLU,
                                 _lib.RH_ACT_GEGLU_ERF])
@pytest.mark.parametrize("shape", [(1213, 768, 3072), (1025, 200, 4128), (700, 3072, 2080),
                                   (16300, 64, 256), (16385, 130, 288)])
def test_int8_one_round_of_the_chip(gpu_ctx, shape, act):
    """Grids of up to 256 64x256 tiles and just past them: integer sums and one
    epilogue, so the bits of a forced 128x128 tile."""
    m, k, n = shape
    say(f"int8 one round m={m} k={k} n={n} act={act}")
    rng = np.random.default_rng(m + k + n + act)
    wt = (rng.standard_normal((n, k)) * 0.05).astype(np.float32)
    gated = act not in (_lib.RH_ACT_NONE, _lib.RH_ACT_GELU)
    if gated:
        pb = T.PackedGated(gpu_ctx, 2, wt[: n // 2].copy(), wt[n // 2:].copy(), k, n // 2)
    else:
        pb = T.PackedWeight(gpu_ctx, 2, wt, k, n, rng.standard_normal(n).astype(np.float32))
    cols, ldq = (n // 2 if gated else n), T.ldq_for(k)
    da, dst = gpu_ctx.upload(rows(rng, m, k)), gpu_ctx.alloc(m * cols * 4)
    qa, rs = gpu_ctx.alloc(m * ldq), gpu_ctx.alloc(m * 4)
    out = []
    for tile in (0, 3):
        gpu_ctx.set_option(_lib.RH_CTX_I8_TILE, tile)
        try:
            T.Linear(gpu_ctx, dst, da, pb, m, act, qa, ldq, rs)
            gpu_ctx.sync()
        finally:
            gpu_ctx.set_option(_lib.RH_CTX_I8_TILE, 0)
        out.append(dst.download(np.float32, (m, cols)))
    assert np.array_equal(out[0], out[1])
