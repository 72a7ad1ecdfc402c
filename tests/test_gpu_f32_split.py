"""The fp32 Dense on f16-split operands (qvl_dense_ws) against float64, tile by tile."""
import ctypes as C

import numpy as np
import pytest

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu

DEV = "cuda:0"


@pytest.fixture
def dense(pkg, lib):
    """dense(plan, x, w, b, epi, r) -> y on torch fp32 tensors; w [N rounded up to 64, K]."""
    cp = pkg.capi
    nb = C.c_size_t()
    cp.check(lib.qvl_dense_workspace_size(C.byref(nb)))
    ws = torch.empty(nb.value, dtype=torch.uint8, device=DEV)

    def run(plan, x, w, b, epi=0, r=None):
        (M, K), N = x.shape, b.shape[0]
        y = r.clone() if r is not None else torch.empty((M, N), device=DEV)      # the residual in place
        cp.check(lib.qvl_set_f32_plan(plan))
        cp.check(lib.qvl_dense_ws(torch.cuda.current_stream().cuda_stream, cp.QVL_DTYPE_F32, epi, x.data_ptr(), K,
                                  w.data_ptr(), b.data_ptr(), y.data_ptr() if r is not None else None, N, y.data_ptr(),
                                  N, M, N, K, ws.data_ptr(), nb.value))
        return y
    yield run
    cp.check(lib.qvl_set_f32_plan(0))


def operands(M, N, K, seed):
    g = torch.Generator(device=DEV).manual_seed(seed)
    x = torch.randn((M, K), generator=g, device=DEV)
    w = torch.zeros((-(-N // 64) * 64, K), device=DEV)
    w[:N] = torch.randn((N, K), generator=g, device=DEV) * 0.05
    b = torch.randn(N, generator=g, device=DEV)
    return x, w, b, torch.randn((M, N), generator=g, device=DEV)


def bound(x, w, N, K):
    """|error| per element: the terms an f16 split drops (3 products of 2^-22 of |x w|), then one rounding of the
    running sum, at most sum |x w|, per accumulation step (3 K / 16) and K part."""
    s = x.abs().double() @ w[:N].abs().double().t()
    return s * (3 * 2.0 ** -22 + (3 * K / 16 + 16) * 2.0 ** -24)


# edges of the 64 / 128 / 256 tiles, one k-step pair (K = 64) and split-K (K >= 256), one row, one 4-column group
@pytest.mark.parametrize("plan", [1, 2, 3, 4])
@pytest.mark.parametrize("M,N,K", [(1, 4, 64), (63, 132, 64), (64, 128, 192), (65, 252, 256), (129, 256, 1024),
                                   (257, 260, 320), (300, 1152, 4352), (31, 64, 8192)])
def test_split_dense_vs_fp64(dense, plan, M, N, K):
    x, w, b, r = operands(M, N, K, M + N + K)
    ref = x.double() @ w[:N].double().t() + b.double()
    tol = bound(x, w, N, K) + ref.abs() * 2.0 ** -23
    assert torch.all((dense(plan, x, w, b).double() - ref).abs() <= tol)
    y = dense(plan, x, w, b, 2, r)
    assert torch.all((y.double() - ref - r.double()).abs() <= tol + (ref.abs() + r.abs()) * 2.0 ** -23)
    # GELU: slope at most 1.13; its own fp32 arithmetic (exp2, reciprocal) within 4e-6 of max(|y|, 1)
    y = dense(plan, x, w, b, 1)
    gelu = torch.nn.functional.gelu(ref, approximate="tanh")
    assert torch.all((y.double() - gelu).abs() <= 1.13 * tol + 4e-6 * gelu.abs().clamp(min=1.0))


# edges of the 128x128 tile, with and without K parts; (784, 3072, 1024): the default rule takes it
@pytest.mark.parametrize("M,N,K", [(1, 4, 64), (127, 124, 192), (128, 128, 256), (129, 132, 1024), (300, 1152, 4352),
                                   (784, 3072, 1024)])
def test_split_dense_128x128_tiles(dense, M, N, K):
    x, w, b, r = operands(M, N, K, M + N + K)
    ref = x.double() @ w[:N].double().t() + b.double()
    tol = bound(x, w, N, K) + ref.abs() * 2.0 ** -23
    y = dense(6, x, w, b)
    assert torch.all((y.double() - ref).abs() <= tol)
    assert torch.all((dense(6, x, w, b, 2, r).double() - ref - r.double()).abs() <= tol + (ref.abs() + r.abs()) * 2.0 ** -23)
    if M > 1:
        assert (y.double() - ref).norm() <= (dense(5, x, w, b).double() - ref).norm()
    x[0, 1], w[2, 3] = float("inf"), float("nan")
    y, want = dense(6, x, w, b), dense(5, x, w, b)
    assert torch.equal(torch.isnan(y), torch.isnan(want)) and torch.equal(torch.isinf(y), torch.isinf(want))


@pytest.mark.parametrize("M,N,K", [(784, 1024, 1024), (300, 512, 4096), (2304, 3072, 1024)])
def test_split_dense_is_nearer_to_fp64_than_fp32_mfma(dense, M, N, K):
    x, w, b, _ = operands(M, N, K, K)
    ref = x.double() @ w.double().t() + b.double()
    err = [((dense(p, x, w, b).double() - ref).norm() / ref.norm()).item() for p in (0, 1, 2, 3, 5)]
    assert max(err[:4]) <= err[4], err


def test_split_dense_row_scales(dense):
    """Rows of every magnitude keep their relative error: the split's exponent is per row (of x and of w)."""
    M, N, K = 130, 128, 256
    x, w, b, _ = operands(M, N, K, 3)
    b.zero_()
    x *= (10.0 ** torch.linspace(-30, 18, M, device=DEV))[:, None]
    w *= (10.0 ** torch.linspace(-7, 18, N, device=DEV))[:, None]
    x[5], x[6, 1:], w[7] = 0.0, 0.0, 0.0
    ref = x.double() @ w.double().t()
    for plan in (1, 2, 3, 4):
        y = dense(plan, x, w, b).double()
        assert torch.all((y - ref).abs() <= bound(x, w, N, K))
        assert not y[5].any() and not y[:, 7].any()


@pytest.mark.parametrize("K", [128, 2048])          # without and with split-K
def test_split_dense_infinities_and_nan(dense, K):
    """Rows and weights that hold infinities or NaN give what the fp32 MFMA kernel gives; the others stay exact."""
    M, N = 140, 192
    x, w, b, r = operands(M, N, K, 7)
    inf, nan = float("inf"), float("nan")
    x[3, 7], x[9, 1], x[64, 5], x[64, 6], x[139, K - 1] = inf, nan, inf, -inf, -inf
    w[5, 3], w[100, 2], w[8] = -inf, nan, w[8].bfloat16().float()      # (row 8's lo terms are zeros)
    w[11, 7] = 0.0                                                      # inf * 0
    for epi in (0, 1, 2):
        want = dense(5, x, w, b, epi, r if epi == 2 else None)
        for plan in (1, 2, 3, 4):
            got = dense(plan, x, w, b, epi, r if epi == 2 else None)
            assert torch.equal(torch.isnan(got), torch.isnan(want))
            inf_at = torch.isinf(want)
            assert torch.equal(got[inf_at], want[inf_at]) and torch.equal(torch.isinf(got), inf_at)
            fine = torch.isfinite(want)
            assert torch.allclose(got[fine], want[fine], rtol=1e-4, atol=1e-4)


# ---------------------------------------------------------------------------------------------
# the fp32 tower on weights split when it is bound
# ---------------------------------------------------------------------------------------------
@pytest.mark.parametrize("K,N,groups", [(64, 64, 1), (1024, 192, 3), (1152, 128, 1), (4096, 64, 1), (8192, 128, 2)])
def test_split_weight_values_and_bound(pkg, lib, K, N, groups):
    """hi + lo is the weight to 2^-22 of it (or 2^-39 of the row's largest), and no normalised row's output passes
    the bound: sqrt(K) |gamma w| + |beta . w| + |b|, reached within a factor by the row that points along gamma w."""
    cp = pkg.capi
    g = torch.Generator(device=DEV).manual_seed(K + N)
    w = torch.randn((N, K), generator=g, device=DEV) * 10.0 ** torch.linspace(-20, 5, K, device=DEV)
    w[1] = 0.0
    gamma, beta = (torch.randn(K // 4, generator=g, device=DEV) for _ in range(2))     # repeated 4 times along a row
    b = torch.randn(N, generator=g, device=DEV)
    out = torch.empty((N, K // 32, 2, 32), dtype=torch.float16, device=DEV)
    scale = torch.empty(N, device=DEV)
    bound = torch.empty(groups + N, device=DEV)
    cp.check(lib.qvl_split_dense_weight(torch.cuda.current_stream().cuda_stream, w.data_ptr(), K, N, b.data_ptr(),
                                        gamma.data_ptr(), beta.data_ptr(), K // 4, groups, out.data_ptr(),
                                        scale.data_ptr(), bound.data_ptr()))
    got = (out.double().sum(2) * scale[:, None, None].double()).reshape(N, K)
    big = w.abs().amax(1, keepdim=True).double()
    assert torch.all((got - w.double()).abs() <= w.abs().double() * 2.0 ** -22 + big * 2.0 ** -39)
    ga, be = gamma.double().repeat(4), beta.double().repeat(4)
    gw = ga * w.double()
    want = K ** 0.5 * gw.norm(dim=1) + (w.double() @ be).abs() + b.double().abs()
    assert torch.all(bound[groups:] >= want * 0.9999) and torch.all(bound[groups:] <= want * 1.002)
    assert torch.equal(bound[:groups], bound[groups:].view(groups, -1).amax(1))


def tower_pair(pkg, spec, params):
    """The fp32 tower with its split weights, and without them."""
    a = pkg.Qwen3VisionTransformer(spec).bind(params)
    b = pkg.Qwen3VisionTransformer(spec).bind_packed(a.packed_state())
    assert a._split is not None
    b._split = None
    return a, b


@pytest.mark.parametrize("head_dim", [64, 72, 80])
@pytest.mark.parametrize("grids", [[(1, 2, 2), (1, 6, 4), (2, 10, 14)], [(1, 28, 28)]])
def test_split_tower_large_scores(pkg, head_dim, grids):
    """Scores of some tens (the qkv weights 10 times the usual ones), segments of 4 to 784 keys, whole lists and key
    parts: no further from the fp64 oracle than the fp32 MFMA kernels."""
    from oracle import vision_tower as vt
    spec = pkg.VisionBackboneSpec(hidden_size=16 * head_dim, out_hidden_size=128, depth=1, num_heads=16,
                                  intermediate_size=256)
    params = pkg.random_params(spec, seed=head_dim)
    params["visual"]["blocks_0"]["attn"]["qkv"]["kernel"] *= 10
    n = sum(t * h * w for t, h, w in grids)
    px = np.random.default_rng(1).standard_normal((n, spec.patch_volume), dtype=np.float32)
    ospec = vt.VisionSpec(hidden_size=16 * head_dim, out_hidden_size=128, depth=1, num_heads=16, intermediate_size=256,
                          deepstack_visual_indexes=())
    ref = torch.from_numpy(np.asarray(vt.encode_vision(params, px, grids, ospec, "fp64").tokens, np.float64))
    err = []
    for t in tower_pair(pkg, spec, params):
        tokens, _ = t(px, np.array(grids, np.int32))
        err.append(((tokens.double().cpu() - ref).norm() / ref.norm()).item())
    assert err[0] <= max(err[1], 2e-7), err


def test_split_tower_nan_stays_in_its_segment(pkg):
    spec = pkg.spec_2b()
    spec.depth, spec.deepstack_visual_indexes = 2, (0,)
    a, b = tower_pair(pkg, spec, pkg.random_params(spec, seed=2))
    grids = np.array([[1, 6, 10], [1, 8, 12]], np.int32)
    px = np.random.default_rng(3).standard_normal((156, spec.patch_volume), dtype=np.float32)
    clean = a(px, grids)
    for bad in (np.nan, np.inf):
        px[7, 100] = bad
        (tok, ds), (tok_b, ds_b) = a(px, grids), b(px, grids)
        for x, y, z in ((tok, tok_b, clean[0]), (ds[0], ds_b[0], clean[1][0])):
            assert torch.equal(torch.isnan(x), torch.isnan(y)) and torch.equal(x[15:], z[15:])


def test_weights_that_cannot_be_split_leave_the_tower_unsplit(pkg):
    spec = pkg.spec_2b()
    spec.depth, spec.deepstack_visual_indexes = 1, ()
    params = pkg.random_params(spec, seed=2)
    grids = np.array([[1, 4, 6]], np.int32)
    px = np.random.default_rng(3).standard_normal((24, spec.patch_volume), dtype=np.float32)
    params["visual"]["merger"]["linear_fc2"]["kernel"][3, 5] = np.inf
    t = pkg.Qwen3VisionTransformer(spec).bind(params)
    assert t._split is None
    tokens, _ = t(px, grids)
    assert not torch.isfinite(tokens[:, 5]).any() and torch.isfinite(tokens[:, :5]).all()


def test_split_weights_follow_writes_to_the_bound_buffers(pkg):
    """A weight, a norm's parameter and a bias written in place between two forwards: the second one's outputs are those
    of a tower bound to the written buffers."""
    spec = pkg.spec_2b()
    spec.depth, spec.deepstack_visual_indexes = 1, ()
    grids = np.array([[1, 4, 6]], np.int32)
    px = np.random.default_rng(3).standard_normal((24, spec.patch_volume), dtype=np.float32)
    t = pkg.Qwen3VisionTransformer(spec).bind(pkg.random_params(spec, seed=2))
    before = t(px, grids)[0].clone()
    for name, by in (("blocks.0.fc1.w", 0.01), ("blocks.0.norm1.w", 50.0), ("merger.fc1.b", -2.0)):
        t.packed_state()[name].add_(by)
        got = t(px, grids)[0].clone()
        want = pkg.Qwen3VisionTransformer(spec).bind_packed(t.packed_state())(px, grids)[0]
        assert torch.equal(got, want) and not torch.equal(got, before)
        before = got
    w = t.packed_state()["merger.fc2.w"]
    old = w[5, 3].item()
    w[5, 3] = float("inf")                              # cannot be split: the buffers are read as they are
    tokens = t(px, grids)[0]
    assert not torch.isfinite(tokens[:, 5]).any() and torch.isfinite(tokens[:, :5]).all()
    w[5, 3] = old
    assert torch.equal(t(px, grids)[0], before)


def one_block(pkg):
    spec = pkg.spec_2b()
    spec.depth, spec.deepstack_visual_indexes = 1, (0,)
    grids = np.array([[1, 4, 6]], np.int32)
    px = torch.from_numpy(np.random.default_rng(3).standard_normal((24, spec.patch_volume), dtype=np.float32)).to(DEV)
    return spec, pkg.random_params(spec, seed=2), px, grids


def outputs(tower, px, grids):
    tokens, ds = tower(px, grids)
    return [t.clone() for t in (tokens, *ds)]


def fresh(pkg, tower, px, grids):
    return outputs(pkg.Qwen3VisionTransformer(tower.spec).bind_packed(tower.packed_state()), px, grids)


WRITES = (("blocks.0.fc1.w", 0.01), ("blocks.0.qkv.b", 3.0), ("blocks.0.norm1.w", 50.0), ("deepstack.0.fc1.w", 0.02),
          ("patch_embed.w", 0.01), ("merger.fc2.w", 0.03))


def same(got, want):
    return all(torch.equal(a, b) for a, b in zip(got, want))


@pytest.mark.parametrize("how", ["data", "inference", "dlpack"])
def test_split_tower_follows_writes_that_torch_does_not_count(pkg, how):
    """Writes through .data, to inference tensors and through DLPack leave torch's version counts as they were; the next
    forward reads the written weights all the same."""
    spec, params, px, grids = one_block(pkg)
    with torch.inference_mode(how == "inference"):
        t = pkg.Qwen3VisionTransformer(spec).bind(params)
        assert t._split is not None
        before = outputs(t, px, grids)
        for name, by in WRITES:
            w = t.packed_state()[name]
            (w.data if how == "data" else torch.utils.dlpack.from_dlpack(w) if how == "dlpack" else w).add_(by)
            got = outputs(t, px, grids)
            assert same(got, fresh(pkg, t, px, grids)) and not same(got, before), name
            before = got


def test_captured_split_forward_follows_writes(pkg):
    """A graph captured around a forward, weights written, other forwards and allocations in between: each replay gives
    what a tower bound to the buffers as they are then gives."""
    spec, params, px, grids = one_block(pkg)
    t = pkg.Qwen3VisionTransformer(spec).bind(params)
    before = outputs(t, px, grids)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        tokens, ds = t(px, grids)
    graph.replay()
    torch.cuda.synchronize()
    assert same((tokens, *ds), before)
    for name, by in WRITES:
        t.packed_state()[name].add_(by)
        graph.replay()                                   # no forward since the write
        torch.cuda.synchronize()
        want = fresh(pkg, t, px, grids)
        assert same((tokens, *ds), want) and not same(want, before), name
        assert same(outputs(t, px, grids), want)
        junk = [torch.full((1 << 22,), float("nan"), device=DEV) for _ in range(8)]
        graph.replay()
        torch.cuda.synchronize()
        assert same((tokens, *ds), want), name
        before = want
        del junk


def split_beforehand(pkg, lib, t):
    """qvl_vision_split of a bound tower, made by qvl_split_dense_weight: (struct, what it points to)."""
    cp, st, keep = pkg.capi, t.packed_state(), []

    def split(name, norm=None, groups=1):
        w = st[name + ".w"]
        n, k = w.shape
        g, b = (st[norm + ".w"], st[norm + ".b"]) if norm else (None, None)
        out = [torch.empty(m, device=DEV) for m in (n * k, n, groups + n)]
        cp.check(lib.qvl_split_dense_weight(torch.cuda.current_stream().cuda_stream, w.data_ptr(), k, n,
                                            st[name + ".b"].data_ptr(), g.data_ptr() if norm else None,
                                            b.data_ptr() if norm else None, g.numel() if norm else 0, groups,
                                            *(o.data_ptr() for o in out)))
        keep.extend(out)
        return cp.SplitDense(*(o.data_ptr() for o in out))

    def merger(name):
        return cp.SplitMerger(split(name + ".fc1", name + ".norm"), split(name + ".fc2"))
    s = t.spec
    blocks, ds = (cp.SplitBlock * s.depth)(), (cp.SplitMerger * max(1, len(s.deepstack_visual_indexes)))()
    for i in range(s.depth):
        p = f"blocks.{i}."
        blocks[i] = cp.SplitBlock(split(p + "qkv", p + "norm1", 3), split(p + "proj"), split(p + "fc1", p + "norm2"),
                                  split(p + "fc2"))
    for j in range(len(s.deepstack_visual_indexes)):
        ds[j] = merger(f"deepstack.{j}")
    return cp.VisionSplit(split("patch_embed"), blocks, merger("merger"), ds), (keep, blocks, ds)


@pytest.mark.parametrize("shape", ["spec_2b", "spec_8b"])
def test_weights_split_beforehand_give_the_same_bits(pkg, lib, shape):
    """qvl_encode_vision_split on weights that the caller split against the tower's own forward, two blocks and a tap."""
    cp = pkg.capi
    spec = getattr(pkg, shape)()
    spec.depth, spec.deepstack_visual_indexes = 2, (0,)
    t = pkg.Qwen3VisionTransformer(spec).bind(pkg.random_params(spec, seed=4))
    grids = np.array([[1, 6, 10], [1, 14, 14]], np.int32)
    px = torch.randn((256, spec.patch_volume), device=DEV)
    want = outputs(t, px, grids)
    split, _keep = split_beforehand(pkg, lib, t)
    got = [torch.empty_like(o) for o in want]
    ws, nb = t.workspace(256)
    cp.check(lib.qvl_encode_vision_split(torch.cuda.current_stream().cuda_stream, C.byref(t._cfg), C.byref(t._w),
                                         C.byref(split), C.byref(t.metadata(grids)[2]), px.data_ptr(), got[0].data_ptr(),
                                         (C.c_void_p * 1)(got[1].data_ptr()), ws.data_ptr(), nb))
    assert same(got, want)


@pytest.mark.parametrize("K", [64, 1024, 4352])
def test_split_weight_bound_over_the_fp32_range(pkg, lib, K):
    """Rows from 1e-36 to 1e33 (whose squares fp32 does not hold), no bias: the bound is the row's own."""
    cp = pkg.capi
    N = 128
    g = torch.Generator(device=DEV).manual_seed(K)
    w = torch.randn((N, K), generator=g, device=DEV).double() * 10.0 ** torch.linspace(-36, 33, N, device=DEV).double()[:, None]
    w = w.float()
    gamma, b = 1 + 0.1 * torch.randn(K, generator=g, device=DEV), torch.zeros(N, device=DEV)
    beta = torch.zeros_like(gamma)
    out, scale, bound = (torch.empty(n, device=DEV) for n in (N * K, N, 1 + N))
    cp.check(lib.qvl_split_dense_weight(torch.cuda.current_stream().cuda_stream, w.data_ptr(), K, N, b.data_ptr(),
                                        gamma.data_ptr(), beta.data_ptr(), K, 1, out.data_ptr(), scale.data_ptr(),
                                        bound.data_ptr()))
    want = K ** 0.5 * (gamma.double() * w.double()).norm(dim=1)
    assert torch.all(bound[1:] >= want * 0.9999) and torch.all(bound[1:] <= want * 1.002)


def test_split_tower_with_tiny_hidden_rows(pkg):
    """fc1 weights of 1e-26 and fc2 weights of 1e25, no fc1 bias: the hidden rows keep their values."""
    spec, params, px, grids = one_block(pkg)
    mlp = params["visual"]["blocks_0"]["mlp"]
    mlp["linear_fc1"]["kernel"] *= np.float32(1e-25)
    mlp["linear_fc2"]["kernel"] *= np.float32(1e25)
    a, b = tower_pair(pkg, spec, params)
    for x, y in zip(outputs(a, px, grids), outputs(b, px, grids)):
        assert torch.isfinite(x).all() and (x - y).norm() <= 1e-5 * y.norm()


# One entry far above the rest of its row, a zero against it: what is left of the row decides the output. From 2^17 the
# rows go by the fp32 operands; a third of them are left as they were. K with and without K parts, edges of the tiles.
@pytest.mark.parametrize("M,N,K", [(70, 132, 128), (257, 260, 1024), (33, 64, 4352)])
@pytest.mark.parametrize("side", ["x", "w"])
def test_split_dense_outliers_within_a_row(dense, M, N, K, side):
    for e in (8, 14, 16, 17, 18, 20, 24, 30, 40, 80):
        x, w, b, r = operands(M, N, K, e)
        a, other = (x, w) if side == "x" else (w, x)
        a[:, 3] = torch.where(torch.arange(len(a), device=DEV) % 3 > 0, 2.0 ** e * a.std().item(), 1.0)
        other[:, 3] = 0.0
        b.zero_()
        ref = x.double() @ w[:N].double().t()
        tol = bound(x, w, N, K)
        for plan in (0, 1, 2, 3, 4, 6):
            for epi in (0, 2):
                y = dense(plan, x, w, b, epi, r if epi else None).double() - (r.double() if epi else 0)
                assert torch.all((y - ref).abs() <= tol + epi * (ref.abs() + r.abs().double()) * 2.0 ** -23), (e, plan, epi)
        got, want = dense(0, x, w, b).double(), dense(5, x, w, b).double()
        assert (got - ref).norm() <= 1.1 * (want - ref).norm(), e


def test_split_dense_wide_rows_match_fp32(dense):
    """Rows whose entries are spread over 60 powers of two, in either operand: no further from float64 than the fp32 MFMA
    kernel, whatever the other operand picks out of them."""
    M, N, K = 96, 192, 1024
    for seed, side in ((1, "x"), (2, "w")):
        x, w, b, _ = operands(M, N, K, seed)
        (x if side == "x" else w).mul_(2.0 ** torch.linspace(-60, 0, K, device=DEV))
        b.zero_()
        for k in (200, 600, 1000):                          # the other one reads the first k entries alone
            x1, w1 = x.clone(), w.clone()
            (w1 if side == "x" else x1)[:, k:] = 0.0
            ref = x1.double() @ w1[:N].double().t()
            err = [(dense(plan, x1, w1, b).double() - ref).norm() / ref.norm() for plan in (0, 1, 2, 3, 4, 6, 5)]
            assert max(err[:-1]) <= 1.1 * err[-1] + 1e-8, (side, k, err)


@pytest.mark.parametrize("where", ["fc1", "deepstack"])
def test_split_tower_with_an_outlier_among_the_hidden_rows(pkg, where):
    """One fc1 row 2^16 above the others and a zero fc2 column against it: the others' exponent is not the outlier's. A
    tower bound to such weights is not split; one that they were written to afterwards keeps fp32 hidden rows."""
    spec, params, px, grids = one_block(pkg)
    t = pkg.Qwen3VisionTransformer(spec).bind(params)
    st = t.packed_state()
    pre = "blocks.0." if where == "fc1" else "deepstack.0."
    st[pre + "fc1.w"][5] *= 2.0 ** 16
    st[pre + "fc2.w"][:, 5] = 0.0
    b = pkg.Qwen3VisionTransformer(spec).bind_packed(st)
    assert t._split is not None and b._split is None
    for got, want in zip(outputs(t, px, grids), outputs(b, px, grids)):
        assert torch.isfinite(got).all() and (got - want).norm() <= 3e-6 * want.norm()


@pytest.mark.parametrize("part", [0, 1, 2])
def test_outliers_among_q_k_v_leave_the_tower_unsplit(pkg, part):
    spec, params, px, grids = one_block(pkg)
    w = params["visual"]["blocks_0"]["attn"]["qkv"]["kernel"]
    w[:, part * spec.hidden_size + 7] *= np.float32(2.0 ** 12)
    assert pkg.Qwen3VisionTransformer(spec).bind(params)._split is None
    w[:, part * spec.hidden_size + 7] *= np.float32(2.0 ** -8)          # 2^4 above the others: ordinary
    assert pkg.Qwen3VisionTransformer(spec).bind(params)._split is not None


@pytest.mark.parametrize("cols", [1024, 1152])
def test_split_tower_with_wide_normalised_rows(pkg, lib, cols):
    """Two entries of opposite sign 2^22 above the rest of a token (their sum does not lift the others) and zero weights
    against them: the normalised row goes by fp32. The pixel rows are such tokens through an identity patch embed."""
    spec, params, px, grids = one_block(pkg)
    if cols == 1152:
        spec = pkg.spec_8b()
        spec.depth, spec.deepstack_visual_indexes = 1, (0,)
        params = pkg.random_params(spec, seed=2)
    v = params["visual"]
    v["patch_embed"]["proj"]["kernel"][:] = 0
    for i in range(cols):
        v["patch_embed"]["proj"]["kernel"][i, i] = 1.0
    v["pos_embed"]["embedding"][:] = 0
    px[::2, 3], px[::2, 9] = 2.0 ** 22, -2.0 ** 22
    for k in (v["blocks_0"]["attn"]["qkv"]["kernel"], v["blocks_0"]["mlp"]["linear_fc1"]["kernel"]):
        k[3], k[9] = 0, 0
    a, b = tower_pair(pkg, spec, params)
    for got, want in zip(outputs(a, px, grids), outputs(b, px, grids)):
        assert torch.isfinite(got).all() and (got - want).norm() <= 3e-6 * want.norm()


def test_bind_packed_during_a_capture(pkg):
    """Binding packed buffers launches nothing that a capture refuses; such a tower runs unsplit."""
    spec, params, px, grids = one_block(pkg)
    t = pkg.Qwen3VisionTransformer(spec).bind(params)
    want = outputs(t, px, grids)
    late = pkg.Qwen3VisionTransformer(spec)
    late.metadata(grids), late.workspace(24)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        tokens, ds = late.bind_packed(t.packed_state())(px, grids)
    assert late._split is None
    for _ in range(3):
        graph.replay()
        torch.cuda.synchronize()
        for a, b in zip((tokens, *ds), want):
            assert (a - b).norm() <= 3e-6 * b.norm()
        outputs(t, px, grids)
