"""The launch forms a call's sizes choose between, at the sizes where a form
begins, ends or has a remainder, against the CPU oracle or plain numpy."""

import numpy as np
import pytest

pytestmark = pytest.mark.gpu
RNG = np.random.default_rng(77)


@pytest.mark.parametrize("n_ops", [1, 2, 4, 5, 9])
def test_short_graph_replays(ggml, gpu, n_ops):
    """a graph of a few launches, replayed (launch by launch up to four, as
    one HIP graph beyond): every compute is on the inputs of that compute.
    Scaling by a power of two is exact."""
    print(f"short graph of {n_ops}", flush=True)
    G = ggml.Graph()
    X = G.new(ggml.F32, 1000, 3)
    y, f = X, 1.0
    for i in range(n_ops):
        s = 2.0 if i % 2 else -0.25
        y, f = G.lib.ggml_scale(G.ctx, y, s), f * s
    G.build(y)
    G.allocate(gpu.buft)
    for it in range(6):
        x = RNG.standard_normal((3, 1000)).astype(np.float32)
        G.set(X, x)
        assert G.compute(gpu.backend) == 0
        assert np.array_equal(G.get(y).reshape(3, 1000), x * np.float32(f))
    G.free()


# 64 x 64 tiles for 256 CUs: up to 42 (16-row form of four K groups), up to 64
# (32 rows, four groups), up to 192 (two groups), up to 256 (64 x 64 tiles, two
# groups), more (one group); at most two K slices take two groups
@pytest.mark.parametrize("wname,m,k,n", [
    ("q8_0", 16, 544, 65), ("q8_0", 1040, 1184, 97), ("q8_0", 896, 3584, 78), ("q8_0", 2048, 2336, 81),
    ("q8_0", 2064, 320, 127), ("q8_0", 4080, 800, 129), ("q8_0", 6160, 544, 250), ("q8_0", 384, 384, 301),
    ("q4_K", 16, 768, 65), ("q4_K", 1040, 1280, 97), ("q4_K", 2048, 2304, 81), ("q4_K", 4080, 768, 129),
    ("q4_K", 6160, 512, 250),
])
def test_tile_gemm_forms(ggml, gpu, ref, wname, m, k, n):
    """the exact tile GEMM's forms at ragged rows, columns and K slices: the
    oracle's f32 values, but for sums on a rounding boundary"""
    print(f"tile gemm {wname} {m} x {k} x {n}", flush=True)
    wt = ggml.Q8_0 if wname == "q8_0" else ggml.Q4_K
    wq = ggml.quantize(wt, ggml.synth_normal(3, m + k, m * k, 0.0, 0.02).reshape(m, k))
    x = RNG.standard_normal((n, k)).astype(np.float32)
    G = ggml.Graph()
    X = G.new(ggml.F32, k, n)
    W = G.new(wt, k, m, weight=True)
    Y = G.lib.ggml_mul_mat(G.ctx, W, X)
    G.lib.ggml_mul_mat_set_prec(Y, ggml.GGML_PREC_F32)
    G.build(Y)
    G.allocate(gpu.buft)
    G.set(W, wq)
    want = ref.mul_mat(wt, wq, m, k, x)
    for _ in range(3):
        G.set(X, x)
        assert G.compute(gpu.backend) == 0
        y = G.get(Y).reshape(n, m)
        # f64 sums in another order: an f32 result moves only where its sum
        # sits within 2^-50 of a rounding boundary, and then by one step
        assert (y != want).mean() <= 1e-5 and np.abs(y - want).max() <= 2.0 ** -22 * np.abs(want).max()
    G.free()


@pytest.mark.parametrize("wname,m,k,n", [("q8_0", 384, 384, 301), ("q8_0", 64, 1056, 65), ("q4_K", 128, 512, 97)])
@pytest.mark.parametrize("over_columns", [False, True])
def test_products_into_f16_tensors(ggml, gpu, ref, wname, m, k, n, over_columns):
    """products of the same columns copied into f16 tensors (the cross K/V of
    an audio window), a bias on every second one: the bits of f16(product) and
    f16(product + bias). over_columns: the first copy's destination lies over
    the columns, so the later products read what it wrote."""
    print(f"f16 products {wname} {m} x {k} x {n} over {over_columns}", flush=True)
    wt = ggml.Q8_0 if wname == "q8_0" else ggml.Q4_K
    G = ggml.Graph()
    lib, ctx = G.lib, G.ctx
    X = G.new(ggml.F32, k, n, weight=True)
    W = [G.new(wt, k, m, weight=True) for _ in range(5)]
    B = G.new(ggml.F32, m, weight=True)
    C = [G.new(ggml.F16, m, n, weight=True) for _ in range(5)]
    G.gf = lib.ggml_new_graph_custom(ctx, G.graph_size, False)
    for i in range(5):
        y = lib.ggml_mul_mat(ctx, W[i], X)
        if i % 2:
            y = lib.ggml_add(ctx, y, B)
        lib.ggml_build_forward_expand(G.gf, lib.ggml_cpy(ctx, y, C[i]))
    G.allocate(gpu.buft)
    x = RNG.standard_normal((n, k)).astype(np.float32)
    b = RNG.standard_normal(m).astype(np.float32)
    wq = [ggml.quantize(wt, ggml.synth_normal(5, i, m * k, 0.0, 0.02).reshape(m, k)) for i in range(5)]
    for t, q in zip(W, wq):
        G.set(t, q)
    G.set(B, b)
    if over_columns:
        ggml.tensor(C[0]).data = ggml.tensor(X).data
        # the copies' nodes are views of their destinations
        for i in range(lib.ggml_graph_n_nodes(G.gf)):
            node = ggml.tensor(lib.ggml_graph_node(G.gf, i))
            if node.view_src and node.src[1] == C[0]:
                node.data = ggml.tensor(X).data
    for _ in range(3):
        G.set(X, x)
        assert G.compute(gpu.backend) == 0
        cols = x.copy()
        for i in range(5):
            y = ref.mul_mat(wt, wq[i], m, k, cols) + (b if i % 2 else np.float32(0))
            want = y.astype(np.float16)
            if over_columns and i == 0:
                raw = cols.view(np.uint16).reshape(-1)
                raw[:m * n] = want.view(np.uint16).reshape(-1)
                cols = raw.view(np.float32).reshape(n, k)
            else:
                got = G.get(C[i], np.float16).reshape(n, m)
                assert (got.view(np.uint16) != want.view(np.uint16)).mean() <= 1e-5
    G.free()


# heads, kv heads, sequences, queries, span, live: split and combined (one
# sequence), merged in the workgroup (a batch), one split, spans off the tile; a
# sequence of 128 blocks over a long span and one of 266, split alone
@pytest.mark.parametrize("d,hq,hkv,t,span,live", [
    (128, 16, 8, 256, 512, 481), (128, 16, 8, 119, 1024, 1000), (64, 6, 6, 130, 600, 577), (128, 8, 1, 33, 300, 290),
    (128, 16, 8, 512, 4096, 3000), (64, 14, 14, 1216, 1216, 1216),
])
@pytest.mark.parametrize("scale", [None, -0.11])
def test_attention_batched_rows_keep_their_bits(ggml, gpu, d, hq, hkv, t, span, live, scale):
    """a sequence's rows are the same bits in a batch, whose splits merge in
    the workgroup, as alone, where they are written and combined; and f16
    operands' distance from the 64-bit result"""
    print(f"attention {d} {hq}/{hkv} {t} x {span} scale {scale}", flush=True)
    S = 8
    scale = d ** -0.5 if scale is None else scale
    q = RNG.standard_normal((S, hq, t, d)).astype(np.float32)
    k, v = (RNG.standard_normal((S, hkv, span, d)).astype(np.float16) for _ in range(2))
    last = live - t + np.arange(t)
    mask = np.where(np.arange(span)[None, :] <= last[:, None], 0.0, -np.inf).astype(np.float16)
    mask[t // 2, 5:9] = -1.5  # neither open nor closed

    def compute(seqs):
        n = len(seqs)
        G = ggml.Graph()
        Q, K, V = G.new(ggml.F32, d, t, hq, n), G.new(ggml.F16, d, span, hkv, n), G.new(ggml.F16, d, span, hkv, n)
        M = G.new(ggml.F16, span, t, 1, n)
        y = G.lib.ggml_flash_attn_ext(G.ctx, Q, K, V, M, scale, 0.0, 0.0)
        G.build(y)
        G.allocate(gpu.buft)
        for T, a in ((Q, q[seqs]), (K, k[seqs]), (V, v[seqs]), (M, np.broadcast_to(mask, (n, 1, t, span)))):
            G.set(T, a)
        assert G.compute(gpu.backend) == 0
        out = G.get(y).reshape(n, t, hq, d)
        G.free()
        return out

    batch = compute(list(range(S)))
    for s in (0, 5):
        assert np.array_equal(compute([s])[0], batch[s])
    h = hq - 1
    a = q[1, h].astype(np.float64) @ k[1, h // (hq // hkv)].astype(np.float64).T * scale + mask.astype(np.float64)
    a = np.exp(a - a.max(1, keepdims=True))
    want = (a / a.sum(1, keepdims=True)) @ v[1, h // (hq // hkv)].astype(np.float64)
    # f16 queries move a score by at most its size times 2^-11 (|score| < 8
    # here), f16 probabilities the result by 2^-11 of it
    assert np.linalg.norm(batch[1, :, h] - want) <= 4 * 2.0 ** -11 * np.linalg.norm(want)


def test_gelu_erf_against_math_erf(ggml, gpu):
    """GELU_ERF over erf's whole bent range, both ends of it, zeros of either
    sign, subnormals, infinities and NaN: the f32 rounding of math.erf, then the
    op's own f32 steps"""
    from math import erf
    z = np.concatenate([np.linspace(-6.2, 6.2, 30001), np.geomspace(1e-45, 1e-2, 200), [0.0, -0.0, 5.65685, 5.656855,
                        -5.65685, 1e30, np.inf, -np.inf, np.nan]]).astype(np.float32)
    G = ggml.Graph()
    X = G.new(ggml.F32, z.size)
    E = G.lib.ggml_gelu_erf(G.ctx, X)
    G.build(E)
    G.allocate(gpu.buft)
    G.set(X, z)
    assert G.compute(gpu.backend) == 0
    a = z * np.float32(0.70710678118654752440)
    e = np.array([erf(float(v)) if np.isfinite(v) else np.sign(v) for v in a], np.float32)
    with np.errstate(invalid="ignore"):
        want = np.float32(0.5) * z * (np.float32(1) + e)
    got = G.get(E)
    same = (got.view(np.uint32) == want.view(np.uint32)) | (np.isnan(got) & np.isnan(want))
    # math.erf itself is within one double ulp: the f32 roundings of the two
    # differ once in ~2^27 values
    assert same.all(), (z[~same], got[~same], want[~same])
    G.free()


@pytest.mark.parametrize("heads,t,n", [(14, 390, 1), (14, 1170, 1), (3, 97, 1), (2, 64, 2), (1, 2, 3)])
@pytest.mark.parametrize("overwritten", [False, True])
def test_attention_over_f32_keys(ggml, gpu, heads, t, n, overwritten):
    """an encoder's attention over strided f32 K / V head views, its f16 mask cast
    from f32 in the graph: the bits of the same attention over f16 tensors holding
    their roundings. overwritten: the f32 mask changes between the cast and the
    attention, which reads the cast's result"""
    d = 64
    print(f"f32 attention {heads} x {t} x {n} overwritten {overwritten}", flush=True)
    q, k, v = (RNG.standard_normal((n, t, heads, d)).astype(np.float32) for _ in range(3))
    mask = RNG.standard_normal((n, 1, t, t)).astype(np.float32)
    mask[RNG.random(mask.shape) < 0.3] = -np.inf
    mask[..., 0] = 0.0
    for kind in ("zero", "mixed"):
        m = np.zeros_like(mask) if kind == "zero" else mask
        outs = []
        for f32 in (True, False):
            G = ggml.Graph()
            lib, ctx = G.lib, G.ctx
            head = lambda x: lib.ggml_permute(ctx, x, 0, 2, 1, 3)  # noqa: E731
            Q = G.new(ggml.F32, d, heads, t, n)
            G.gf = lib.ggml_new_graph_custom(ctx, G.graph_size, False)
            if f32:
                K, V = (G.new(ggml.F32, d, heads, t, n) for _ in range(2))
                M = G.new(ggml.F32, t, t, 1, n)
                m16 = lib.ggml_cast(ctx, M, ggml.F16)
                lib.ggml_build_forward_expand(G.gf, m16)
                if overwritten:
                    O = G.new(ggml.F32, t, t, 1, n)
                    lib.ggml_build_forward_expand(G.gf, lib.ggml_cpy(ctx, O, M))
                y = lib.ggml_flash_attn_ext(ctx, head(Q), head(K), head(V), m16, d ** -0.5, 0.0, 0.0)
            else:
                K, V = (G.new(ggml.F16, d, t, heads, n) for _ in range(2))
                M = G.new(ggml.F16, t, t, 1, n)
                y = lib.ggml_flash_attn_ext(ctx, head(Q), K, V, M, d ** -0.5, 0.0, 0.0)
            lib.ggml_set_output(y)
            lib.ggml_build_forward_expand(G.gf, y)
            G.allocate(gpu.buft)
            for _ in range(2):
                G.set(Q, q)
                if f32:
                    G.set(K, k), G.set(V, v), G.set(M, m)
                    if overwritten:
                        G.set(O, np.full_like(m, 3.0) * np.arange(t, dtype=np.float32))
                else:
                    G.set(K, k.astype(np.float16).transpose(0, 2, 1, 3)), G.set(V, v.astype(np.float16).transpose(0, 2, 1, 3))
                    G.set(M, m.astype(np.float16))
                assert G.compute(gpu.backend) == 0
            outs.append(G.get(y))
            G.free()
        assert np.array_equal(outs[0], outs[1]) and np.isfinite(outs[0]).all()


# rows of a multiple of eight elements on 16 bytes take eight a thread; others
# (an odd width, an offset view) one
@pytest.mark.parametrize("d,heads,t,n,span,skip", [(128, 8, 256, 8, 300, 0), (64, 3, 7, 2, 9, 0), (8, 1, 1, 1, 3, 0),
                                                   (20, 3, 5, 2, 8, 0), (64, 3, 7, 2, 9, 1)])
@pytest.mark.parametrize("i64", [False, True])
def test_set_rows_widths(ggml, gpu, d, heads, t, n, span, skip, i64):
    """f32 rows [d, t, heads, n] of a strided source into an f16 cache at
    per-sequence rows: f16 roundings at those rows, the other rows untouched"""
    print(f"set_rows {d} x {t} x {heads} x {n} skip {skip}", flush=True)
    G = ggml.Graph()
    lib, ctx = G.lib, G.ctx
    X = G.new(ggml.F32, d + 4 * skip, heads, t, n)
    I = G.new(ggml.I64 if i64 else ggml.I32, t, 1, n)
    C = G.new(ggml.F16, d, span, heads, n, weight=True)
    src = lib.ggml_permute(ctx, X, 0, 2, 1, 3)
    if skip:
        # the last d of d + 4 elements, from 4 bytes past a 16-byte boundary
        src = lib.ggml_permute(ctx, lib.ggml_view_4d(ctx, X, d, heads, t, n, 4 * (d + 4), 4 * (d + 4) * heads,
                                                     4 * (d + 4) * heads * t, 4), 0, 2, 1, 3)
    y = lib.ggml_set_rows(ctx, C, src, I)
    G.gf = lib.ggml_new_graph_custom(ctx, G.graph_size, False)
    lib.ggml_build_forward_expand(G.gf, y)
    G.allocate(gpu.buft)
    x = RNG.standard_normal((n, t, heads, d + 4 * skip)).astype(np.float32) * 3
    rows = np.stack([RNG.permutation(span)[:t] for _ in range(n)])
    want = RNG.standard_normal((n, heads, span, d)).astype(np.float16)
    G.set(C, want)
    G.set(X, x)
    G.set(I, rows.astype(np.int64 if i64 else np.int32))
    assert G.compute(gpu.backend) == 0
    part = x[..., 1:1 + d] if skip else x
    for s in range(n):
        want[s][:, rows[s]] = part[s].transpose(1, 0, 2).astype(np.float16)
    assert np.array_equal(G.get(C, np.uint16).reshape(-1), want.view(np.uint16).reshape(-1))
    G.free()


@pytest.mark.parametrize("heads,kv_heads,t", [(16, 8, 256), (16, 8, 255), (6, 2, 1000), (4, 4, 1024)])
def test_norm_rope_rows(ggml, gpu, heads, kv_heads, t):
    """RMS_NORM, weight and RoPE of the query and key rows: four heads of a
    position a wave (many rows, heads in fours) or one, the same bits as the
    three ops apart"""
    print(f"norm rope {heads}/{kv_heads} x {t}", flush=True)
    d, outs = 128, []
    x = RNG.standard_normal((t, (heads + kv_heads) * d)).astype(np.float32)
    w = RNG.uniform(0.5, 1.5, (2, d)).astype(np.float32)
    for fused in (True, False):
        G = ggml.Graph()
        lib, ctx = G.lib, G.ctx
        X = [G.new(ggml.F32, d, h, t) for h in (heads, kv_heads)]
        W = [G.new(ggml.F32, d, weight=True) for _ in range(2)]
        P = G.new(ggml.I32, t)
        keep, out = [], []
        for a, b in zip(X, W):
            a = lib.ggml_rms_norm(ctx, a, 1e-6)
            b = lib.ggml_mul(ctx, a, b)
            keep += [a, b]
            out.append(lib.ggml_rope_ext(ctx, b, P, None, d, ggml.GGML_ROPE_TYPE_NEOX, 4096, 1e6, 1.0, 0.0, 1.0, 32.0, 1.0))
        G.build(*(out if fused else keep + out))  # intermediate results that are outputs are not folded
        G.allocate(gpu.buft)
        G.set(X[0], x[:, :heads * d]), G.set(X[1], x[:, heads * d:])
        G.set(W[0], w[0]), G.set(W[1], w[1])
        G.set(P, (np.arange(t) * 3 + 5).astype(np.int32))
        assert G.compute(gpu.backend) == 0
        outs.append(np.concatenate([G.get(o).reshape(-1) for o in out]))
        G.free()
    assert np.array_equal(outs[0].view(np.uint32), outs[1].view(np.uint32))


@pytest.mark.parametrize("n", [512, 516, 640, 896, 1020, 1028])
@pytest.mark.parametrize("rows", [1, 390, 1024, 1025])
@pytest.mark.parametrize("layer", [False, True])
def test_norm_row_widths(ggml, gpu, n, rows, layer):
    """RMS_NORM and NORM with weight and bias at the edges of the
    workgroup-a-row form (513 to 1024 elements, a multiple of four; at most 1024
    rows)"""
    f = np.float32
    x = (RNG.standard_normal((rows, n)) * 2 + 0.7).astype(f)
    w, b = RNG.uniform(0.5, 1.5, n).astype(f), RNG.standard_normal(n).astype(f)
    G = ggml.Graph()
    lib, ctx = G.lib, G.ctx
    X, W, B = G.new(ggml.F32, n, rows), G.new(ggml.F32, n, weight=True), G.new(ggml.F32, n, weight=True)
    y = lib.ggml_norm(ctx, X, 1e-5) if layer else lib.ggml_rms_norm(ctx, X, 1e-5)
    y = lib.ggml_mul(ctx, y, W)
    if layer:
        y = lib.ggml_add(ctx, y, B)
    G.build(y)
    G.allocate(gpu.buft)
    G.set(X, x), G.set(W, w), G.set(B, b)
    assert G.compute(gpu.backend) == 0
    mean = (x.astype(np.float64).sum(1, keepdims=True) / n).astype(f) if layer else f(0)
    v = x - mean
    var = ((v * v).astype(np.float64).sum(1, keepdims=True) / n).astype(f)
    want = v * (f(1) / np.sqrt(var + f(1e-5))) * w
    if layer:
        want = want + b
    got = G.get(y).reshape(rows, n)
    # the same f32 steps around f64 sums: a row moves only where its sum lies
    # on an f32 rounding boundary, and then by one step of its mean or scale
    assert (got != want).mean() <= 0.01 and np.abs(got - want).max() <= 4 * 2.0 ** -23 * np.abs(want).max()
    G.free()


def gelu_erf_f32(z):
    from math import erf
    a = z * np.float32(0.70710678118654752440)
    e = np.array([erf(float(v)) for v in a.reshape(-1)], np.float32).reshape(z.shape)
    return np.float32(0.5) * z * (np.float32(1) + e)


@pytest.mark.parametrize("wname,m,k,n", [("q8_0", 64, 352, 97), ("q4_K", 80, 512, 65)])
@pytest.mark.parametrize("bias,res,gelu", [(False, False, True), (False, True, False), (False, True, True),
                                           (True, True, False), (True, True, True)])
def test_product_epilogues_into_f16_tensors(ggml, gpu, ref, wname, m, k, n, bias, res, gelu):
    """a product with a bias, a residual and a GELU_ERF copied into an f16
    tensor: the f16 of the f32 steps (the residual's rows are f32 rows, whatever
    the result's are)"""
    print(f"f16 epilogue {wname} {m} x {k} x {n} bias {bias} res {res} gelu {gelu}", flush=True)
    wt = ggml.Q8_0 if wname == "q8_0" else ggml.Q4_K
    G = ggml.Graph()
    lib, ctx = G.lib, G.ctx
    X, R = G.new(ggml.F32, k, n), G.new(ggml.F32, m, n)
    W, B, C = G.new(wt, k, m, weight=True), G.new(ggml.F32, m, weight=True), G.new(ggml.F16, m, n, weight=True)
    y = lib.ggml_mul_mat(ctx, W, X)
    lib.ggml_mul_mat_set_prec(y, ggml.GGML_PREC_F32)
    if bias:
        y = lib.ggml_add(ctx, y, B)
    if res:
        y = lib.ggml_add(ctx, y, R)
    if gelu:
        y = lib.ggml_gelu_erf(ctx, y)
    G.build(lib.ggml_cpy(ctx, y, C))
    G.allocate(gpu.buft)
    x, r = RNG.standard_normal((n, k)).astype(np.float32), RNG.standard_normal((n, m)).astype(np.float32)
    b = RNG.standard_normal(m).astype(np.float32)
    wq = ggml.quantize(wt, ggml.synth_normal(5, m, m * k, 0.0, 0.02).reshape(m, k))
    G.set(W, wq), G.set(B, b)
    want = ref.mul_mat(wt, wq, m, k, x)
    if bias:
        want = want + b
    if res:
        want = want + r
    if gelu:
        want = gelu_erf_f32(want)
    for _ in range(3):
        G.set(X, x)
        if res:
            G.set(R, r)
        assert G.compute(gpu.backend) == 0
        # an f32 step apart once in ~2^27 values, and an f16 once in ~2^40
        assert np.array_equal(G.get(C, np.uint16).reshape(n, m), want.astype(np.float16).view(np.uint16))
    G.free()


# 80 rows: two launches over one quantization of the columns; 64: a second
# product that could join the first one's launch
@pytest.mark.parametrize("m", [80, 64])
@pytest.mark.parametrize("how", ["pair", "rows", "copy"])
@pytest.mark.parametrize("wname", ["q8_0", "q4_K"])
def test_columns_written_between_products(ggml, gpu, ref, wname, m, how):
    """product, a write over some of its columns (the second of two SET_ROWS of
    the same rows, one SET_ROWS, or a copy), product: the second one sees the
    written columns"""
    print(f"columns written between products {wname} {m} {how}", flush=True)
    k, n, rows = 512, 97, 5
    wt = ggml.Q8_0 if wname == "q8_0" else ggml.Q4_K
    G = ggml.Graph()
    lib, ctx = G.lib, G.ctx
    X, A = G.new(ggml.F32, k, n, weight=True), G.new(ggml.F32, k, n, weight=True)
    W = [G.new(wt, k, m, weight=True) for _ in range(2)]
    V, I = G.new(ggml.F32, k, rows), G.new(ggml.I32, rows)
    G.gf = lib.ggml_new_graph_custom(ctx, G.graph_size, False)
    Y = [lib.ggml_mul_mat(ctx, w, X) for w in W]
    writes = {"pair": lambda: [lib.ggml_set_rows(ctx, A, V, I), lib.ggml_set_rows(ctx, X, V, I)],
              "rows": lambda: [lib.ggml_set_rows(ctx, X, V, I)],
              "copy": lambda: [lib.ggml_cpy(ctx, V, lib.ggml_view_2d(ctx, X, k, rows, 4 * k, 4 * k * 30))]}[how]()
    for t in (Y[0], *writes, Y[1]):
        lib.ggml_build_forward_expand(G.gf, t)
    for y in Y:
        lib.ggml_set_output(y)
    G.allocate(gpu.buft)
    x, v = RNG.standard_normal((n, k)).astype(np.float32), RNG.standard_normal((rows, k)).astype(np.float32)
    at = np.arange(30, 30 + rows) if how == "copy" else np.array([96, 0, 17, 64, 3])
    wq = [ggml.quantize(wt, ggml.synth_normal(6, i, m * k, 0.0, 0.02).reshape(m, k)) for i in range(2)]
    for t, q in zip(W, wq):
        G.set(t, q)
    after = x.copy()
    after[at] = v
    want = [ref.mul_mat(wt, wq[0], m, k, x), ref.mul_mat(wt, wq[1], m, k, after)]
    for _ in range(3):
        G.set(X, x), G.set(V, v)
        if how != "copy":
            G.set(I, at.astype(np.int32))
        assert G.compute(gpu.backend) == 0
        for y, z in zip(Y, want):
            assert np.abs(G.get(y).reshape(n, m) - z).max() <= 2.0 ** -22 * np.abs(z).max()
    G.free()


def test_columns_written_between_gate_and_up(ggml, gpu, ref):
    """the same between the two products of a SwiGLU whose matrix is too tall
    for a launch that quantizes its columns itself"""
    m, k, n = 8224, 256, 4
    G = ggml.Graph()
    lib, ctx = G.lib, G.ctx
    X = G.new(ggml.F32, k, n, weight=True)
    W = [G.new(ggml.Q8_0, k, m, weight=True) for _ in range(2)]
    V, I = G.new(ggml.F32, k, 1), G.new(ggml.I32, 1)
    G.gf = lib.ggml_new_graph_custom(ctx, G.graph_size, False)
    gate, up = (lib.ggml_mul_mat(ctx, w, X) for w in W)
    h = lib.ggml_mul(ctx, lib.ggml_silu(ctx, gate), up)
    for t in (gate, lib.ggml_set_rows(ctx, X, V, I), h):
        lib.ggml_build_forward_expand(G.gf, t)
    lib.ggml_set_output(h)
    G.allocate(gpu.buft)
    x, v = RNG.standard_normal((n, k)).astype(np.float32), RNG.standard_normal((1, k)).astype(np.float32)
    wq = [ggml.quantize(ggml.Q8_0, ggml.synth_normal(6, i, m * k, 0.0, 0.05).reshape(m, k)) for i in range(2)]
    for t, q in zip(W, wq):
        G.set(t, q)
    after = x.copy()
    after[2] = v[0]
    a, b = ref.mul_mat(ggml.Q8_0, wq[0], m, k, x), ref.mul_mat(ggml.Q8_0, wq[1], m, k, after)
    want = a.astype(np.float64) / (1 + np.exp(-a.astype(np.float64))) * b
    for _ in range(3):
        G.set(X, x), G.set(V, v), G.set(I, np.array([2], np.int32))
        assert G.compute(gpu.backend) == 0
        # f32 steps of the SiLU and the product
        assert np.abs(G.get(h).reshape(n, m) - want).max() <= 2.0 ** -20 * np.abs(want).max()
    G.free()


@pytest.mark.parametrize("n", [1, 4, 97])
def test_norm_result_written_between_products(ggml, gpu, ref, n):
    """a norm's result, a product, a SET_ROWS over the result, a product: the
    second one sees the written row (products of few columns normalise for
    themselves where nothing writes between)"""
    print(f"norm result written between products {n}", flush=True)
    k, m, f = 512, 80, np.float32
    G = ggml.Graph()
    lib, ctx = G.lib, G.ctx
    X, V, I = G.new(ggml.F32, k, n), G.new(ggml.F32, k, 1), G.new(ggml.I32, 1)
    N = G.new(ggml.F32, k, weight=True)
    W = [G.new(ggml.Q8_0, k, m, weight=True) for _ in range(2)]
    h = lib.ggml_mul(ctx, lib.ggml_rms_norm(ctx, X, 1e-5), N)
    Y = [lib.ggml_mul_mat(ctx, w, h) for w in W]
    G.gf = lib.ggml_new_graph_custom(ctx, G.graph_size, False)
    for t in (Y[0], lib.ggml_set_rows(ctx, h, V, I), Y[1]):
        lib.ggml_build_forward_expand(G.gf, t)
    for y in Y:
        lib.ggml_set_output(y)
    G.allocate(gpu.buft)
    x, v = RNG.standard_normal((n, k)).astype(f), RNG.standard_normal((1, k)).astype(f)
    w = RNG.uniform(0.5, 1.5, k).astype(f)
    wq = [ggml.quantize(ggml.Q8_0, ggml.synth_normal(8, i, m * k, 0.0, 0.02).reshape(m, k)) for i in range(2)]
    for t, q in zip(W, wq):
        G.set(t, q)
    G.set(N, w)
    var = ((x * x).astype(np.float64).sum(1, keepdims=True) / k).astype(f)
    cols = x * (f(1) / np.sqrt(var + f(1e-5))) * w
    after = cols.copy()
    after[n - 1] = v[0]
    want = [ref.mul_mat(ggml.Q8_0, q, m, k, c) for q, c in zip(wq, (cols, after))]
    for _ in range(3):
        G.set(X, x), G.set(V, v), G.set(I, np.array([n - 1], np.int32))
        assert G.compute(gpu.backend) == 0
        for y, z in zip(Y, want):
            # a norm's f32 rounding may move by a step and take an 8-bit
            # activation over its rounding boundary: a step of one of k terms
            assert np.abs(G.get(y).reshape(n, m) - z).max() <= 0.02 * np.abs(z).max()
    G.free()


@pytest.mark.parametrize("d", [64, 20])
@pytest.mark.parametrize("second", [0, 3])
def test_set_rows_of_no_rows(ggml, gpu, d, second):
    """SET_ROWS of no rows into an f16 cache, alone or before a graph's other
    work: nothing happens to the cache"""
    print(f"set_rows of no rows {d} {second}", flush=True)
    G = ggml.Graph()
    lib, ctx = G.lib, G.ctx
    X, I = G.new(ggml.F32, d, 0), G.new(ggml.I32, 0)
    Y, J = G.new(ggml.F32, d, 3), G.new(ggml.I32, 3)
    C = [G.new(ggml.F16, d, 9, weight=True) for _ in range(2)]
    G.gf = lib.ggml_new_graph_custom(ctx, G.graph_size, False)
    lib.ggml_build_forward_expand(G.gf, lib.ggml_set_rows(ctx, C[0], X, I))
    if second:
        lib.ggml_build_forward_expand(G.gf, lib.ggml_set_rows(ctx, C[1], Y, J))
    G.allocate(gpu.buft)
    c, y = RNG.standard_normal((2, 9, d)).astype(np.float16), RNG.standard_normal((3, d)).astype(np.float32)
    want = c.copy()
    if second:
        want[1][[8, 0, 5]] = y.astype(np.float16)
    for _ in range(3):
        for i in range(2):
            G.set(C[i], c[i])
        if second:
            G.set(Y, y), G.set(J, np.array([8, 0, 5], np.int32))
        assert G.compute(gpu.backend) == 0
        for i in range(2):
            assert np.array_equal(G.get(C[i], np.uint16).reshape(9, d), want[i].view(np.uint16))
    G.free()


def test_attention_reading_f32_keys_takes_no_copy_scratch(ggml, gpu):
    """an attention that reads f32 K and V itself runs in fixed scratch which
    their f16 copies would overflow, with the bits of the arena's"""
    import ctypes
    lib = gpu.cdll
    lib.ggml_backend_mi355x_graph_compute_static.restype = ctypes.c_int
    lib.ggml_backend_mi355x_graph_compute_static.argtypes = [ctypes.c_void_p, ctypes.c_void_p]
    lib.ggml_backend_mi355x_static_scratch_bytes.restype = ctypes.c_size_t
    d, heads, t, kv = 64, 14, 64, 20000
    G = ggml.Graph()
    q, k, v = (G.new(ggml.F32, d, heads, n, 1) for n in (t, kv, kv))
    head = lambda x: G.lib.ggml_permute(G.ctx, x, 0, 2, 1, 3)  # noqa: E731
    y = G.lib.ggml_flash_attn_ext(G.ctx, head(q), head(k), head(v), None, d ** -0.5, 0.0, 0.0)
    G.build(y)
    G.allocate(gpu.buft)
    for x, n in ((q, t), (k, kv), (v, kv)):
        G.set(x, RNG.standard_normal((n, heads, d)).astype(np.float32))
    assert 2 * 2 * d * heads * kv > lib.ggml_backend_mi355x_static_scratch_bytes()
    assert lib.ggml_backend_mi355x_graph_compute_static(gpu.backend, G.gf) == 0
    static = G.get(y).copy()
    assert G.compute(gpu.backend) == 0
    assert np.isfinite(static).all() and np.array_equal(static, G.get(y))
    G.free()


@pytest.mark.parametrize("d,hq,hkv", [(128, 16, 8), (64, 6, 6)])
@pytest.mark.parametrize("seqs,live", [(1, 1000), (8, 1000), (8, 741)])
def test_attention_divides_by_the_row_sum(ggml, gpu, d, hq, hkv, seqs, live):
    """equal scores over splits, combined or merged: the mean of equal values is
    the value, exactly, as every sum is a whole number below 2^24 and the result
    one division"""
    print(f"attention row sums {d} x {seqs} live {live}", flush=True)
    t, span = 256, 1024
    G = ggml.Graph()
    Q, K, V = G.new(ggml.F32, d, t, hq, seqs), G.new(ggml.F16, d, span, hkv, seqs), G.new(ggml.F16, d, span, hkv, seqs)
    M = G.new(ggml.F16, span, t, 1, seqs)
    y = G.lib.ggml_flash_attn_ext(G.ctx, Q, K, V, M, d ** -0.5, 0.0, 0.0)
    G.build(y)
    G.allocate(gpu.buft)
    v = RNG.integers(1, 2048, (seqs, hkv, 1, d)).astype(np.float16)
    mask = np.where(np.arange(span) < live, 0.0, -np.inf).astype(np.float16)
    G.set(Q, RNG.standard_normal((seqs, hq, t, d)).astype(np.float32))
    G.set(K, np.zeros((seqs, hkv, span, d), np.float16))
    G.set(V, np.broadcast_to(v, (seqs, hkv, span, d)))
    G.set(M, np.broadcast_to(mask, (seqs, 1, t, span)))
    assert G.compute(gpu.backend) == 0
    want = np.repeat(v.astype(np.float32), hq // hkv, 1).transpose(0, 2, 1, 3)  # [seqs, 1, hq, d]
    assert np.array_equal(G.get(y).reshape(seqs, t, hq, d), np.broadcast_to(want, (seqs, t, hq, d)))
    G.free()


# bands of eight 64-column tiles: one band, a band and a remainder, several; row
# tiles with a remainder; batches; a K that is split
@pytest.mark.parametrize("m,k,n,b", [(200, 96, 512, 1), (200, 96, 700, 1), (64, 64, 1100, 2), (130, 1024, 600, 1)])
def test_float_gemm_tile_bands(ggml, gpu, m, k, n, b):
    """an f16-weight product over more column tiles than a band: every tile once"""
    print(f"float gemm bands {m} x {k} x {n} x {b}", flush=True)
    G = ggml.Graph()
    W, X = G.new(ggml.F16, k, m, b, weight=True), G.new(ggml.F32, k, n, b)
    y = G.lib.ggml_mul_mat(G.ctx, W, X)
    G.build(y)
    G.allocate(gpu.buft)
    w = RNG.standard_normal((b, m, k)).astype(np.float16)
    x = RNG.standard_normal((b, n, k)).astype(np.float32)
    G.set(W, w), G.set(X, x)
    assert G.compute(gpu.backend) == 0
    want = x.astype(np.float16).astype(np.float64) @ w.astype(np.float64).transpose(0, 2, 1)
    got = G.get(y).reshape(b, n, m)
    # k f32 additions of products of about 1: an error below k 2^-24 each
    assert np.abs(got - want).max() <= k * 2.0 ** -24 * np.sqrt(k) + 1e-6
    G.free()
