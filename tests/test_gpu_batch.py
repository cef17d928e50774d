"""Batched decode through the C ABI on the GPU: the M <= 64 MFMA GEMM against the oracle's GEMV row
by row, and whole batches of sequences against the oracle's single-sequence decode.

The GEMM splits x into two f16 halves (hi + lo) so its products keep about 22 bits; it accumulates
in f32, so it is held to the GEMV's bar (rel_err < 2e-5 against the f64 oracle). Batched decode is
held to the model tests' bar: logits within 1e-3 of the oracle, identical greedy ids."""
import ctypes

import numpy as np
import pytest
import cpu_oracle as O
import devmem as D
import qne as Q
import weights as W
from test_gpu_kernels import f16_matrix, q4_matrix, rel_err, to_dev

pytestmark = pytest.mark.gpu


def oracle_rows(m, X, G, epi, y0, norm):
    """Row by row with the oracle GEMV (and RMSNorm prologue): the reference's gemm semantics."""
    out = y0.copy()
    for r in range(X.shape[0]):
        x = np.ascontiguousarray(X[r])
        if norm:
            xn = np.empty_like(x)
            O.lib("f64").oc_rmsnorm(O.ptr(x), O.ptr(G), O.ptr(xn), x.size, 1e-6)
            x = xn
        O.lib("f64").oc_gemv(ctypes.byref(m), O.ptr(x), O.ptr(out[r]), {0: O.STORE, 1: O.ACCUMULATE, 2: O.SWIGLU}[epi])
    return out


def run_gemm(kind, group, rows, k, M, epi, norm, seed, x_pad=0, y_pad=0):
    rng = np.random.default_rng(seed)
    m, w, sz = q4_matrix(rows, k, group, rng) if kind == Q.MAT_Q4 else f16_matrix(rows, k, rng)
    X = rng.normal(0, 1, size=(M, k + x_pad)).astype(np.float32)
    G = rng.normal(1, 0.2, size=k).astype(np.float32)
    n_out = rows // 2 if epi == Q.EPI_SWIGLU else rows
    Y0 = rng.normal(size=(M, n_out + y_pad)).astype(np.float32)
    want = Y0.copy()
    want[:, :n_out] = oracle_rows(m, np.ascontiguousarray(X[:, :k]), G, epi, np.ascontiguousarray(Y0[:, :n_out]), norm)
    dw, dx, dy, dg = to_dev(w), to_dev(X), to_dev(Y0), to_dev(G)
    dsz = to_dev(sz) if sz is not None else None
    Q.gemm(kind, dw.data_ptr(), dsz.data_ptr() if dsz is not None else 0, rows, k, group, dx.data_ptr(), k + x_pad, M,
           dy.data_ptr(), n_out + y_pad, epi, norm=dg.data_ptr() if norm else 0)
    D.sync()
    return dy.numpy(), want


@pytest.mark.parametrize("k", [512, 2048, 6144])
@pytest.mark.parametrize("kind,group", [(Q.MAT_Q4, 64), (Q.MAT_Q4, 128), (Q.MAT_F16, 0)])
@pytest.mark.parametrize("epi", [Q.EPI_STORE, Q.EPI_ACCUMULATE, Q.EPI_SWIGLU])
@pytest.mark.parametrize("norm", [False, True])
@pytest.mark.parametrize("M", [1, 7, 64])
def test_gemm_matches_oracle(k, kind, group, epi, norm, M):
    rows = 2 * 150 if epi == Q.EPI_SWIGLU else 300  # ragged last tile of 128 rows
    got, want = run_gemm(kind, group, rows, k, M, epi, norm, seed=k + 7 * epi + 3 * group + norm + 101 * M)
    err = rel_err(got, want)
    assert err < 2e-5, err


@pytest.mark.parametrize("kind,group", [(Q.MAT_Q4, 64), (Q.MAT_F16, 0)])
@pytest.mark.parametrize("epi", [Q.EPI_STORE, Q.EPI_SWIGLU])
@pytest.mark.parametrize("M", [65, 200])
def test_gemm_row_tiles_match_oracle(kind, group, epi, M):
    """More than 64 rows run as tiles of 64 rows (the prefill's passes), each over the same weights;
    a ragged last tile."""
    rows = 2 * 150 if epi == Q.EPI_SWIGLU else 300
    got, want = run_gemm(kind, group, rows, 1024, M, epi, True, seed=41 + M + 5 * epi + group)
    assert rel_err(got, want) < 2e-5


@pytest.mark.parametrize("norm", [False, True])
def test_gemm_swiglu_applied_by_the_gemm(norm):
    """A SwiGLU GEMM with one split over several row tiles (K = 128: two chunks) applies
    silu(gate) * up in the GEMM itself, with no reduce pass; gate and up rows 256 apart, two
    workgroups of 128 output columns, a ragged last row tile."""
    got, want = run_gemm(Q.MAT_Q4, 64, 2 * 256, 128, 200, Q.EPI_SWIGLU, norm, seed=61 + norm)
    assert rel_err(got, want) < 2e-5


@pytest.mark.parametrize("M", [512, 2048])
def test_gemm_full_pass_of_rows(M):
    got, want = run_gemm(Q.MAT_Q4, 64, 256, 512, M, Q.EPI_ACCUMULATE, True, seed=77 + M)
    assert rel_err(got, want) < 2e-5


def gemm_form(rows, k, M, epi):
    """How qne_gemm runs a q4 call, restated from launch_gemm and gemm_wide_pays: "64 rows" (k_gemm), "short"
    (k_gemm_short, of 32 or 64 columns) or "wide" (k_gemm_wide, of 128 rows, of 64 in two halves, or both),
    with its split count and whether the GEMM applies the epilogue itself."""
    def up(a, b):
        return -(-a // b)

    cols, tiles, chunks = up(rows, 256), up(M, 64), k // 64
    if M <= 256:
        return "64 rows"
    splits = up(chunks, up(chunks, max(1, min(256 // (cols * tiles), 24, chunks // 2))))
    splits = up(chunks, up(chunks, max(1, min(splits, chunks // 8))))
    short = up(rows, 64) * up(M, 32) * splits
    own = splits == 1 and short > 512 and (epi != Q.EPI_SWIGLU or (rows % 256 == 0 and k <= 4096))
    if cols * tiles * chunks <= 1344 and not own:
        return "64 rows"
    if short <= 512:
        return f"short {32 if short < 256 else 64}, {splits} splits"
    wide, cost = 0, 1e9
    for n in (cols, cols * up(M, 128) // 256 * 256 // up(M, 128), 0) if splits == 1 else ():
        c = up(n * up(M, 128), 256) + 0.6 * up((cols - n) * tiles, 256)
        if n == cols or c < cost:
            wide, cost = n, c
    rows_of = "128" if wide == cols else "halves" if wide == 0 else "both"
    return f"wide {rows_of}, " + ("own" if own else f"{splits} splits")


@pytest.mark.parametrize("rows,k,group,M,epi,form", [
    # too small a matrix for a pass: the 64-row form over five to eight row tiles
    (256, 64, 64, 257, Q.EPI_STORE, "64 rows"),            # one chunk
    (300, 320, 64, 300, Q.EPI_ACCUMULATE, "64 rows"),      # a ragged column tile
    (520, 128, 128, 333, Q.EPI_STORE, "64 rows"),          # two chunks of one scale group
    (512, 192, 64, 321, Q.EPI_SWIGLU, "64 rows"),          # SwiGLU by the GEMM, one row in the last tile
    (360, 1024, 128, 450, Q.EPI_SWIGLU, "64 rows"),        # SwiGLU by the reduce (180 outputs)
    (4128, 192, 64, 1990, Q.EPI_ACCUMULATE, "wide both, own"),  # 16 column tiles as 128 rows, the ragged 17th as 64
    (4096, 1088, 64, 2048, Q.EPI_SWIGLU, "wide 128, own"),      # 17 chunks: a second batch of the zero points' sums
    (2048, 6144, 64, 333, Q.EPI_ACCUMULATE, "wide halves, 5 splits"),
    (2048, 3520, 64, 333, Q.EPI_STORE, "wide halves, 5 splits"),     # 11 chunks a split: the odd half has one fewer
    (4100, 64, 64, 300, Q.EPI_STORE, "wide halves, own"),            # one chunk: the odd half has none; waves past N
    (4096, 192, 64, 321, Q.EPI_SWIGLU, "wide halves, own"),          # each half one 32-row tile; one row in the last
    (4096, 128, 128, 290, Q.EPI_ACCUMULATE, "wide halves, own"),     # two chunks of one scale group
    (4000, 1024, 128, 450, Q.EPI_SWIGLU, "wide halves, 2 splits"),   # SwiGLU by the reduce (2000 outputs)
    (3841, 4160, 64, 513, Q.EPI_STORE, "wide halves, own"),          # 65 chunks of x^2: two classes
    (64, 4480, 64, 2040, Q.EPI_SWIGLU, "short 64, 8 splits"),
    (40, 17216, 64, 257, Q.EPI_STORE, "short 32, 23 splits"),        # 12 chunks a split; 269 chunks of x^2
])
def test_gemm_wide_forms(rows, k, group, M, epi, form):
    """Calls above 256 rows, at the edges of tiles, chunks, splits and halves. Bar: the two halves of x keep
    22 bits and the f32 sums over up to 24 splits and 64-column chunks round to 2^-24 of a partial sum,
    4e-7 together; five times that for the largest of the outputs."""
    assert gemm_form(rows, k, M, epi) == form
    got, want = run_gemm(Q.MAT_Q4, group, rows, k, M, epi, True, seed=rows + k + M)
    assert rel_err(got, want) < 2e-6


def fused_split(v, g):
    """hi + lo of v g as the operand holds it, lo from the unrounded product, and from the rounded one."""
    exact = v.astype(np.float64) * g.astype(np.float64)
    rounded = exact.astype(np.float32)
    hi = rounded.astype(np.float16).astype(np.float64)
    return [hi + (p - hi).astype(np.float32).astype(np.float16).astype(np.float64) for p in (exact, rounded)]


@pytest.mark.parametrize("kind", [Q.MAT_Q4, Q.MAT_F16])
@pytest.mark.parametrize("k,M", [(64, 3), (2048, 1024)])  # staged a value a lane, and 32 rows of a chunk a wave
def test_gemm_operand_keeps_the_unrounded_product(kind, k, M):
    """x times the norm's gain is split into f16 halves from its unrounded product. x is 1.5 in 3 of 8
    columns and 0.5 in the others (its mean square is 1, so with eps 0 the factor 1 / rms is exactly 1), the
    gains are ones where the two roundings differ, and the matrix picks columns: results are exact."""
    rng = np.random.default_rng(k)
    g = (1 + rng.integers(0, 1 << 23, size=1 << 16) / (1 << 23)).astype(np.float32)
    fused, split = fused_split(np.full(g.size, 1.5, np.float32), g)
    g = g[(fused != split) & (fused.astype(np.float32) == fused)]
    big = np.arange(k) % 8 < 3
    assert g.size >= 64
    G = np.ones(k, np.float32)
    G[big] = g[np.arange(big.sum()) % g.size]
    cols = np.flatnonzero(big)[np.linspace(0, big.sum() - 1, 24).astype(int)]
    X = np.where(big, 1.5, 0.5).astype(np.float32) * np.where(np.arange(M) % 2, -1, 1).astype(np.float32)[:, None]
    want = fused_split(X[:, cols], np.broadcast_to(G[cols], (M, 24)))[0].astype(np.float32)
    one = np.zeros((24, k), np.uint8)
    one[np.arange(24), cols] = 1
    if kind == Q.MAT_Q4:
        w = one[:, 0::2] | (one[:, 1::2] << 4)
        dsz = to_dev(np.tile(np.array([1, 0], np.float16).view(np.uint16), (24, k // 64)))  # scale 1, zero 0
    else:
        w, dsz = one.astype(np.float16).view(np.uint16), None
    dw, dx, dg, dy = to_dev(w), to_dev(X), to_dev(G), D.zeros((M, 24), np.float32)
    Q.gemm(kind, dw.data_ptr(), dsz.data_ptr() if dsz else 0, 24, k, 64, dx.data_ptr(), k, M, dy.data_ptr(), 24,
           norm=dg.data_ptr(), eps=0.0)
    D.sync()
    assert np.array_equal(dy.numpy(), want)


@pytest.mark.parametrize("k,M", [(64, 3), (2048, 1024)])
def test_gemm_operand_adds_a_pairs_squares_with_one_rounding(k, M):
    """The norm's sum of x^2 takes a pair of columns as fma(a, a, b^2), in both staging forms. Rows hold one
    pair and a one; the matrix picks the one, so the result is 1 / rms, and the pairs are ones for which the
    sum's rounding shows in it."""
    f = np.float32
    rng = np.random.default_rng(k)
    a, b = rng.uniform(64, 128, size=(2, 1 << 16)).astype(f)
    low = b * b
    fused, split = ((s + f(1)) / f(k) for s in ((a.astype(np.float64) ** 2 + low).astype(f), a * a + low))
    keep = np.flatnonzero(f(1) / np.sqrt(fused) != f(1) / np.sqrt(split))[:M]
    keep = np.resize(keep, M)
    X = np.zeros((M, k), f)
    X[:, 0], X[:, 1], X[:, 8] = a[keep], b[keep], 1
    w = np.zeros((1, k), np.float16)
    w[0, 8] = 1
    dw, dx, dg, dy = to_dev(w.view(np.uint16)), to_dev(X), to_dev(np.ones(k, f)), D.zeros((M, 1), f)
    Q.gemm(Q.MAT_F16, dw.data_ptr(), 0, 1, k, 0, dx.data_ptr(), k, M, dy.data_ptr(), 1, norm=dg.data_ptr(), eps=0.0)
    D.sync()
    assert np.array_equal(dy.numpy()[:, 0], f(1) / np.sqrt(fused[keep]))


@pytest.mark.parametrize("zero,codes", [(7.5, (0, 15)), (0.0, (0, 1)), (0.0, (0, 3)), (15.0, (14, 15)), (3.49, (0, 7)),
                                        (-20.0, (0, 15)), (40.0, (0, 15))])
@pytest.mark.parametrize("rows,M", [(1024, 1024), (12288, 512)])  # four splits of 8 chunks; one of 32
def test_gemm_wide_zero_points(zero, codes, rows, M):
    """A pass's GEMM over weights that are centred on zero, one-sided, or shifted: the precision does not
    depend on where the zero points lie. Bar: x as two f16 halves keeps 22 bits (2^-23 = 1.2e-7 of a
    product at most), the f32 sums over 64 columns and up to 32 chunks each round to 2^-24 of a partial
    sum, about 1e-7 over a chain; 2.5e-7 in the 2-norm (measured 1.0e-7 to 1.6e-7)."""
    k, group = 2048, 64
    assert gemm_form(rows, k, M, Q.EPI_STORE) == {1024: "wide halves, 4 splits", 12288: "wide 128, own"}[rows]
    rng = np.random.default_rng(rows + M)
    q = rng.integers(codes[0], codes[1] + 1, size=(rows, k), dtype=np.uint8)
    s = rng.uniform(0.002, 0.03, size=(rows, k // group)).astype(np.float16)
    z = np.full((rows, k // group), zero, np.float16)
    X = rng.normal(size=(M, k)).astype(np.float32)
    W = ((q.reshape(rows, -1, group) - z[..., None].astype(np.float64)) * s[..., None].astype(np.float64)).reshape(rows, k)
    want = X.astype(np.float64) @ W.T
    dw, dsz, dx = to_dev(q[:, 0::2] | (q[:, 1::2] << 4)), to_dev(np.stack([s, z], -1).view(np.uint16)), to_dev(X)
    got = D.zeros((M, rows), np.float32)
    Q.gemm(Q.MAT_Q4, dw.data_ptr(), dsz.data_ptr(), rows, k, group, dx.data_ptr(), k, M, got.data_ptr(), rows)
    D.sync()
    err = np.linalg.norm(got.numpy() - want) / np.linalg.norm(want)
    assert err < 2.5e-7, err


@pytest.mark.parametrize("kind,group", [(Q.MAT_Q4, 64), (Q.MAT_F16, 0)])
def test_gemm_one_split_direct_epilogue(kind, group):
    """More than 512 tiles of 128 rows: one split, the GEMM applies 1 / rms and the epilogue itself
    (the LM head's path)."""
    got, want = run_gemm(kind, group, 66000, 512, 3, Q.EPI_ACCUMULATE, True, seed=5)
    assert rel_err(got, want) < 2e-5


def test_gemm_strided_rows_untouched_padding():
    got, want = run_gemm(Q.MAT_Q4, 64, 260, 1024, 5, Q.EPI_STORE, True, seed=9, x_pad=12, y_pad=7)
    assert rel_err(got, want) < 2e-5
    assert np.array_equal(got[:, 260:], want[:, 260:])  # columns past the outputs keep their values


def test_gemm_row_result_does_not_depend_on_other_rows():
    """Each row's sum runs in the same order whatever the other rows hold: bitwise equal."""
    rng = np.random.default_rng(3)
    rows, k = 640, 2048
    _, w, sz = q4_matrix(rows, k, 64, rng)
    X = rng.normal(size=(64, k)).astype(np.float32)
    dw, dsz = to_dev(w), to_dev(sz)
    full = D.zeros((64, rows), np.float32)
    one = D.zeros((1, rows), np.float32)
    dx = to_dev(X)
    Q.gemm(Q.MAT_Q4, dw.data_ptr(), dsz.data_ptr(), rows, k, 64, dx.data_ptr(), k, 64, full.data_ptr(), rows)
    dx1 = to_dev(X[37:38])
    Q.gemm(Q.MAT_Q4, dw.data_ptr(), dsz.data_ptr(), rows, k, 64, dx1.data_ptr(), k, 1, one.data_ptr(), rows)
    # and in the fourth row tile of a 250-row call
    X4 = rng.normal(size=(250, k)).astype(np.float32)
    X4[237] = X[37]
    big = D.zeros((250, rows), np.float32)
    dx4 = to_dev(X4)
    Q.gemm(Q.MAT_Q4, dw.data_ptr(), dsz.data_ptr(), rows, k, 64, dx4.data_ptr(), k, 250, big.data_ptr(), rows)
    D.sync()
    assert np.array_equal(full.numpy()[37], one.numpy()[0])
    assert np.array_equal(big.numpy()[237], one.numpy()[0])


@pytest.mark.parametrize("rows,k,M", [(753, 768, 822), (190, 1024, 1632), (660, 768, 1322), (1989, 1152, 295), (256, 64, 2048)])
def test_gemm_of_a_small_matrix_keeps_its_form_above_256_rows(rows, k, M):
    """Many rows of a matrix that a pass's form would not pay for (it took 1.1 to 1.2 times as long) run as
    few rows do: row by row the same bits as calls of one row."""
    assert gemm_form(rows, k, M, Q.EPI_STORE) == "64 rows"
    rng = np.random.default_rng(M)
    _, w, sz = q4_matrix(rows, k, 64, rng)
    X = rng.normal(size=(M, k)).astype(np.float32)
    dw, dsz, dx = to_dev(w), to_dev(sz), to_dev(X)
    full, one = D.zeros((M, rows), np.float32), D.zeros((3, rows), np.float32)
    Q.gemm(Q.MAT_Q4, dw.data_ptr(), dsz.data_ptr(), rows, k, 64, dx.data_ptr(), k, M, full.data_ptr(), rows)
    picks = [0, 64 * (M // 128) + 3, M - 1]
    for i, r in enumerate(picks):
        Q.gemm(Q.MAT_Q4, dw.data_ptr(), dsz.data_ptr(), rows, k, 64, dx.data_ptr() + 4 * k * r, k, 1,
               one.data_ptr() + 4 * rows * i, rows)
    D.sync()
    assert np.array_equal(full.numpy()[picks], one.numpy())


def test_gemm_rejects_bad_shapes():
    for args in [(Q.MAT_F16, 0, 256, 1000, 4), (Q.MAT_Q4, 32, 256, 1024, 4), (Q.MAT_F16, 0, 256, 1024, 2049),
                 (Q.MAT_F16, 0, 256, 1024, 0)]:
        kind, group, rows, k, M = args
        with pytest.raises(Q.QneError) as e:
            Q.gemm(kind, 1, 1, rows, k, group, 1, k, M, 1, rows)
        assert e.value.code == Q.EINVAL


# ---- whole batches ----

@pytest.fixture(scope="module", params=[("tiny", "q4", "f16"), ("small", "q4", "f16"), ("tiny", "f16", "q4")],
                ids=["tiny-q4body", "small-q4body", "tiny-f16body-q4head"])
def pair(request):
    name, body, head = request.param
    index, buf = W.synth_model(name, seed=11, body=body, head=head, norm_jitter=0.1)
    m = Q.Model.load(index, buf)
    om = O.OracleModel(index, buf, "f64")
    yield m, om
    m.close()


def prompts(vocab, lengths, seed):
    rng = np.random.default_rng(seed)
    return [rng.integers(0, vocab, size=n).astype(np.uint32) for n in lengths]


def test_batch_continues_each_sequence_like_the_oracle(pair):
    m, om = pair
    lengths = [5, 17, 40, 1, 33]
    ps = prompts(m.vocab, lengths, 21)
    steps = 20
    with Q.Batch(m, max_rows=8, max_context=512) as b:
        for r, p in enumerate(ps):
            m.reset()
            m.prefill_batched(p)
            b.admit(r)
        tok, pos = b.row_state(len(ps))
        assert list(pos) == lengths
        picks, logits = b.step(len(ps), logits=True)
        ids = b.decode(len(ps), steps - 1)
        ms, n = b.last_decode_timing()  # the device time of the chained steps
        assert n == steps - 1 and ms > 0.0
    for r, p in enumerate(ps):
        om.reset()
        want_ids, want_logits = om.greedy(p, steps + 1)
        assert tok[r] == want_ids[0]
        assert np.max(np.abs(logits[r] - want_logits[1])) < 1e-3, r
        got = [int(picks[r])] + [int(x) for x in ids[:, r]]
        assert got == want_ids[1:], r


def test_batch_logits_of_many_rows_equal_those_of_few():
    """40 rows of 32768 logits (three slots of the readback's ring, the last one ragged) against the same
    rows four at a time, which are copied straight: a row's bits do not depend on the batch."""
    cfg = dict(layers=1, full_attention_every=2, hidden=512, intermediate=512, vocab=32768, n_q_heads=2, n_kv_heads=1,
               head_dim=256, gdn_heads=4)
    index, buf = W.synth_model(cfg, seed=5, body="q4", head="f16")
    tokens = np.random.default_rng(2).integers(0, cfg["vocab"], 40).astype(np.uint32)
    with Q.Model.load(index, buf) as m, Q.Batch(m, max_rows=40, max_context=16) as b:
        def logits(toks):
            for r, t in enumerate(toks):
                b.reset_row(r, int(t))
            return b.step(len(toks), logits=True)[1]

        few = np.concatenate([logits(tokens[i:i + 4]) for i in range(0, 40, 4)])
        assert np.array_equal(logits(tokens), few)


def test_batch_teacher_forced_logits_and_empty_rows(pair):
    """Rows started empty (reset_row) and fed given tokens: every step's logits against the
    oracle's token-by-token run from position 0."""
    m, om = pair
    R, T = 3, 6
    seqs = prompts(m.vocab, [T] * R, 8)
    with Q.Batch(m, max_rows=R, max_context=64) as b:
        for r in range(R):
            b.reset_row(r, int(seqs[r][0]))
        got = []
        for t in range(T):
            _, lg = b.step(R, tokens=[int(s[t]) for s in seqs], logits=True)
            got.append(lg)
    for r in range(R):
        om.reset()
        for t in range(T):
            want = om.token(int(seqs[r][t]), t)
            assert np.max(np.abs(got[t][r] - want)) < 1e-3, (r, t)


def test_batch_is_bitwise_repeatable(pair):
    m, _ = pair
    ps = prompts(m.vocab, [9, 3, 27], 4)
    runs = []
    for _ in range(2):
        with Q.Batch(m, max_rows=4, max_context=256) as b:
            for r, p in enumerate(ps):
                m.reset()
                m.prefill_batched(p)
                b.admit(r)
            _, lg = b.step(3, logits=True)
            runs.append((lg, b.decode(3, 12)))
    assert np.array_equal(runs[0][0], runs[1][0])
    assert np.array_equal(runs[0][1], runs[1][1])


def test_batch_errors(pair):
    m, _ = pair
    with Q.Batch(m, max_rows=2, max_context=32) as b:
        with pytest.raises(Q.QneError) as e:
            b.admit(2)
        assert e.value.code == Q.EINVAL
        with pytest.raises(Q.QneError) as e:
            b.step(3)
        assert e.value.code == Q.EINVAL
        b.reset_row(0, 1)
        b.reset_row(1, 2)
        with pytest.raises(Q.QneError) as e:
            b.decode(2, 33)  # past the batch context
        assert e.value.code == Q.ECONTEXT
        with pytest.raises(Q.QneError) as e:
            b.step(2, tokens=[1, m.vocab])
        assert e.value.code == Q.EINVAL
        m.reset()
        m.prefill_batched(np.arange(40, dtype=np.uint32))
        with pytest.raises(Q.QneError) as e:
            b.admit(0)  # the model's sequence is longer than the batch context
        assert e.value.code == Q.ECONTEXT
    with pytest.raises(Q.QneError):
        Q.Batch(m, max_rows=65, max_context=32)


def test_batch_row_equals_the_same_row_in_a_one_row_batch(pair):
    """A row's step does not depend on the other rows: every row of a 5-row step is bitwise the step
    of a 1-row batch holding the same sequence (qne_batch_copy_row)."""
    m, _ = pair
    ps = prompts(m.vocab, [12, 1, 30, 7, 19], 31)
    with Q.Batch(m, max_rows=5, max_context=128) as b, Q.Batch(m, max_rows=1, max_context=128) as one:
        for r, p in enumerate(ps):
            m.reset()
            m.prefill_batched(p)
            b.admit(r)
        single = []
        for r in range(5):
            one.copy_row(0, b, r)
            single.append(one.step(1, logits=True))
        picks, lg = b.step(5, logits=True)
    for r in range(5):
        assert int(single[r][0][0]) == int(picks[r]), r
        assert np.array_equal(single[r][1][0].view(np.uint32), lg[r].view(np.uint32)), r


# ---- config 5 at its own workload: 64 rows of the 2B int4 model, contexts U[256, 4096) ----

C5_ROWS = [0, 31, 63]  # where the fixture sequences sit among the synthetic rows


@pytest.fixture(scope="module")
def c5():
    """The c5_rows fixture (three sequences of the 2B int4 model decoded by the oracle) and the model."""
    from test_gpu_golden import fixture, synth
    g = fixture("c5_rows")
    case = __import__("json").loads(str(g["case"]))
    index, buf = synth(case)
    m = Q.Model.load(index, buf)
    yield g, m
    m.close()


def c5_batch(m, g, seed):
    """64 rows: synthetic KV caches and recurrent states at contexts U[256, 4096), with the fixture's
    three sequences (prefilled through the model) admitted at C5_ROWS."""
    b = Q.Batch(m, max_rows=64, max_context=4096)
    ctx = np.random.default_rng(seed).integers(256, 4096 - 32, size=64).astype(np.uint32)
    b.fill_synthetic(ctx, seed=seed)
    b.prompt_logits = {}  # fixture row -> the model's logits after its prompt (logged step 0)
    for i, r in enumerate(C5_ROWS):
        n = int(g["plen"][i])
        p = g["prompt"][i, :n]
        m.reset()
        for s in range(0, n, 512):
            m.prefill_chunk(p[s:s + 512], s, s + 512 >= n)
        b.prompt_logits[i] = m.logits()
        b.admit(r)
    return b, ctx


def test_config5_fixture_rows_decode_like_the_oracle(c5):
    """The three fixture sequences inside a 64-row batch of the 2B model: 16 greedy ids identical to
    the oracle's, and at each of the fixture's logged steps (0, 1, 8, 15) the row's logits within
    1e-2 (the stated bar) of the oracle's sampled logits (kernels/src/model.rs:380-392 per row).
    Step 0 is the prompt's logits from prefill_chunk; steps 1, 8 and 15 come from batched steps
    that return logits, with greedy decode windows between them."""
    g, m = c5
    b, ctx = c5_batch(m, g, seed=17)
    steps = [int(x) for x in g["steps"]]
    assert steps == [0, 1, 8, 15], steps
    lg_at = {}
    with b:
        tok, pos = b.row_state(64)
        for i, r in enumerate(C5_ROWS):
            assert int(pos[r]) == int(g["plen"][i]) and int(tok[r]) == int(g["ids"][i][0]), r
            assert all(int(pos[x]) == int(ctx[x]) for x in range(64) if x not in C5_ROWS)
        p1, lg_at[1] = b.step(64, logits=True)   # feeds ids[0]: logits of step 1, pick ids[1]
        r1 = b.decode(64, 6)                      # picks ids[2..7]
        p8, lg_at[8] = b.step(64, logits=True)   # feeds ids[7]: step 8, pick ids[8]
        r2 = b.decode(64, 6)                      # picks ids[9..14]
        p15, lg_at[15] = b.step(64, logits=True)  # feeds ids[14]: step 15, pick ids[15]
    worst = 0.0
    for i, r in enumerate(C5_ROWS):
        got = ([int(tok[r]), int(p1[r])] + [int(x) for x in r1[:, r]] + [int(p8[r])] + [int(x) for x in r2[:, r]]
               + [int(p15[r])])
        want = [int(x) for x in g["ids"][i]]
        assert got == want, f"row {r}: first divergence at step {next(j for j, (a, c) in enumerate(zip(got, want)) if a != c)}"
        for j, s in enumerate(steps):
            v = b.prompt_logits[i] if s == 0 else lg_at[s][r]
            err = float(np.max(np.abs(v[g["logit_idx"][i, j]] - g["logit_val"][i, j])))
            assert err <= 1e-2, f"row {r} step {s}: max |dlogit| {err:.3e}"
            worst = max(worst, err)
    print(f"config 5: fixture rows identical over 16 steps; max |dlogit| at steps {steps} {worst:.2e}")


def test_config5_each_row_equals_a_one_row_batch(c5):
    """Every one of the 64 rows (synthetic contexts up to 4096, and the fixture rows) steps bitwise
    as it does alone in a 1-row batch: the split-K GEMM reduce, the per-row attention splits and the
    per-row GDN do not depend on the batch."""
    g, m = c5
    b, _ = c5_batch(m, g, seed=23)
    with b, Q.Batch(m, max_rows=1, max_context=4096) as one:
        single = []
        for r in range(64):
            one.copy_row(0, b, r)
            single.append(one.step(1, logits=True))
        picks, lg = b.step(64, logits=True)
    bad = [r for r in range(64) if int(single[r][0][0]) != int(picks[r])
           or not np.array_equal(single[r][1][0].view(np.uint32), lg[r].view(np.uint32))]
    assert not bad, f"rows whose 64-row step differs from their 1-row step: {bad}"
