"""The GEMM kernel of few-row launches (tile plan 9: 32x128 tiles whose 8 waves share K), epilogue by epilogue, against
float64 and against the 256x128 tiles (plan 3) it stands in for."""
import ctypes as C

import numpy as np
import pytest

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu

DEV = "cuda:0"
BF = torch.bfloat16


def stream():
    return torch.cuda.current_stream().cuda_stream


@pytest.fixture
def plans(pkg, lib):
    """plans(fn) -> fn's result on plan 9 and on plan 3 (no split-K)."""
    def both(fn):
        out = []
        for plan in (9, 3):
            pkg.capi.check(lib.qvl_set_gemm_plan(plan, -1, 0))
            out.append(fn())
        return out
    yield both
    pkg.capi.check(lib.qvl_set_gemm_plan(0, 0, 0))


def operands(M, N, K, seed):
    g = torch.Generator(device=DEV).manual_seed(seed)
    x = torch.randn((M, K), generator=g, device=DEV).to(BF)
    w = torch.zeros((-(-N // 64) * 64, K), device=DEV, dtype=BF)
    w[:N] = (torch.randn((N, K), generator=g, device=DEV) * 0.05).to(BF)
    b = torch.randn(N, generator=g, device=DEV).to(BF).float()
    return x, w, b, torch.randn((M, N), generator=g, device=DEV).to(BF)


def close(a, b, *points):
    """Two summation orders of the same fp32 products, rounded to bf16 at the same points: the norms within 2e-3, and
    each element within one bf16 step (2^-7 of the value, or of 2^-6 where the sum cancels) for every rounding on its way
    (`points`: the values rounded before the last one)."""
    a, b = a.double(), b.double()
    bound = 2 ** -7 * sum(v.double().abs() for v in (*points, b)) + 2 ** -13
    return (a - b).norm() <= 2e-3 * b.norm() and bool(((a - b).abs() <= bound).all())


# K of one 64-wide block (half a step), odd and even counts of blocks, more steps than the ring holds; rows and columns
# at the edges of the 32x128 tile
@pytest.mark.parametrize("M,N,K", [(1, 4, 64), (31, 128, 128), (32, 132, 192), (33, 256, 448), (100, 1024, 1024),
                                   (196, 252, 1152), (257, 192, 4352)])
def test_few_rows_dense(pkg, lib, plans, M, N, K):
    cp = pkg.capi
    x, w, b, r = operands(M, N, K, M + N + K)
    prod = x.double() @ w[:N].double().t()
    ref = prod + b.double()
    for epi in (0, 1, 2):
        def run():
            y = r.clone()
            cp.check(lib.qvl_dense(stream(), cp.QVL_DTYPE_BF16, epi, x.data_ptr(), K, w.data_ptr(), b.data_ptr(),
                                   y.data_ptr() if epi == 2 else None, N, y.data_ptr(), N, M, N, K))
            return y
        y9, y3 = plans(run)
        assert close(y9, y3, prod, ref, ref * 0.13), epi      # (GELU's slope is at most 1.13)
        want = torch.nn.functional.gelu(ref, approximate="tanh") if epi == 1 else ref + (r.double() if epi == 2 else 0)
        assert (y9.double() - want).norm() <= 4e-3 * want.norm()


@pytest.mark.parametrize("M,N,K", [(1, 128, 64), (65, 1024, 1024), (196, 1152, 4352)])
def test_few_rows_row_statistics_and_fold(pkg, lib, plans, M, N, K):
    """The residual epilogue's row partials are the statistics of the bf16 rows it wrote, and the folded LayerNorm of
    the next Dense reads them."""
    cp = pkg.capi
    x, w, b, r = operands(M, N, K, M + K)
    nb = C.c_size_t()
    cp.check(lib.qvl_dense_workspace_size(C.byref(nb)))
    ws = torch.empty(nb.value, dtype=torch.uint8, device=DEV)
    G = N // 128
    parts = torch.empty((M, G, 2), device=DEV)
    gam = (1 + 0.1 * torch.randn(N, device=DEV)).to(BF).float()
    bet = (0.1 * torch.randn(N, device=DEV)).to(BF).float()
    w2, b2 = (torch.randn((256, N), device=DEV) * 0.05).to(BF), torch.randn(256, device=DEV)
    wf, cd = torch.empty_like(w2), torch.empty((256, 2), device=DEV)
    cp.check(lib.qvl_fold_ln_weight(stream(), cp.QVL_DTYPE_BF16, w2.data_ptr(), N, 256, gam.data_ptr(), bet.data_ptr(),
                                    wf.data_ptr(), cd.data_ptr()))

    def run():
        y = r.clone()
        cp.check(lib.qvl_dense_rowstats_ws(stream(), cp.QVL_DTYPE_BF16, x.data_ptr(), K, w.data_ptr(), b.data_ptr(),
                                           y.data_ptr(), N, y.data_ptr(), N, M, N, K, parts.data_ptr(), ws.data_ptr(),
                                           nb.value))
        h = torch.empty((M, 256), device=DEV, dtype=BF)
        cp.check(lib.qvl_dense_ln_parts_ws(stream(), cp.QVL_DTYPE_BF16, 1, y.data_ptr(), N, wf.data_ptr(), cd.data_ptr(),
                                           parts.data_ptr(), G, 1e-6, b2.data_ptr(), h.data_ptr(), 256, M, 256, N,
                                           ws.data_ptr(), nb.value))
        return y, parts.clone(), h
    (y9, p9, h9), (y3, _, h3) = plans(run)
    prod = x.double() @ w[:N].double().t()
    assert close(y9, y3, prod, prod + b.double())
    g = y9.double().view(M, G, 128)
    s, q = g.sum(2), ((g - g.mean(2, keepdim=True)) ** 2).sum(2)
    assert torch.allclose(p9[..., 0].double(), s, rtol=0, atol=1e-5 * 128)
    assert torch.allclose(p9[..., 1].double(), q, rtol=1e-5, atol=1e-5)
    ln = torch.nn.functional.layer_norm(y9.double(), (N,), gam.double(), bet.double(), 1e-6)
    want = torch.nn.functional.gelu(ln @ w2.double().t() + b2.double(), approximate="tanh")
    assert (h9.double() - want).norm() <= 6e-3 * want.norm()
    assert (h9.double() - h3.double()).norm() <= 6e-3 * want.norm()


@pytest.mark.parametrize("table", [False, True])
@pytest.mark.parametrize("grids", [[(1, 2, 2)], [(1, 14, 14)], [(1, 6, 10), (2, 4, 2)]])
def test_few_rows_qkv_rotary(pkg, lib, plans, grids, table):
    """q, k and v^T (their zero rows included) as the other tiles write them."""
    cp = pkg.capi
    H, D = 16, 1024
    m = pkg.grid_metadata(grids, num_heads=H)
    N, Np = m.n_tokens, -(-m.n_tokens // 64) * 64
    x, w, b, _ = operands(N, 3 * D, D, N)
    pos = torch.from_numpy(m.pos_hw).to(DEV)
    cs = torch.empty((N, 32, 2), device=DEV)
    cp.check(lib.qvl_rotary_table(stream(), cp.QVL_DTYPE_BF16, pos.data_ptr(), N, 64, 10000.0, cs.data_ptr()))
    tab = torch.empty((m.n_positions, 16), dtype=torch.int32, device=DEV)
    cp.check(lib.qvl_rotary_pos_table(stream(), 64, 10000.0, m.n_positions, tab.data_ptr()))

    def run():
        q, k, v = (torch.full((H, Np * 64), 7.0, device=DEV, dtype=BF) for _ in range(3))
        if table:
            cp.check(lib.qvl_dense_qkv_rotary_pos(stream(), cp.QVL_DTYPE_BF16, x.data_ptr(), D, w.data_ptr(), b.data_ptr(),
                                                  pos.data_ptr(), tab.data_ptr(), m.n_positions, q.data_ptr(),
                                                  k.data_ptr(), v.data_ptr(), N, D, H, None, 0))
        else:
            cp.check(lib.qvl_dense_qkv_rotary(stream(), cp.QVL_DTYPE_BF16, x.data_ptr(), D, w.data_ptr(), b.data_ptr(),
                                              cs.data_ptr(), q.data_ptr(), k.data_ptr(), v.data_ptr(), N, D, H, None, 0))
        return q.view(H, Np, 64), k.view(H, Np, 64), v.view(H, 64, Np)
    prod = x.double() @ w.double().t()
    rounded = prod.abs() + (prod + b.double()).abs()      # per token and feature; rotary mixes dims d and d + 32 of a head
    rounded = torch.nn.functional.pad(rounded, (0, 0, 0, Np - N)).view(Np, 3, H, 2, 32)
    rounded = (2 * rounded.sum(3, keepdim=True)).expand(-1, -1, -1, 2, -1).reshape(Np, 3, H, 64).permute(1, 2, 0, 3)
    perm = torch.tensor([(t & ~15) | ((0, 2, 1, 3)[(t >> 2) & 3] << 2) | (t & 3) for t in range(Np)], device=DEV)
    vt = torch.empty((H, 64, Np), device=DEV, dtype=torch.double)
    vt[:, :, perm] = rounded[2].transpose(1, 2)
    # (three more roundings of values no larger; q is scaled by less than 1)
    for a, c, r in zip(*plans(run), (2 * rounded[0], 2 * rounded[1], vt)):
        assert close(a, c, r)
        assert torch.equal(a == 0, c == 0) or N % 64 == 0 or not a[:, N:].any()


@pytest.mark.parametrize("grids", [[(1, 2, 2)], [(1, 14, 14)], [(2, 6, 10)]])
def test_few_rows_pos_embed(pkg, lib, plans, grids):
    cp = pkg.capi
    m = pkg.grid_metadata(grids)
    M, N, K = m.n_tokens, 1024, 1536
    x, w, b, _ = operands(M, N, K, M)
    table = torch.randn((2304, N), device=DEV).to(BF)
    idx, tw = torch.from_numpy(m.tap_idx).to(DEV), torch.from_numpy(m.tap_w).to(DEV)
    parts = torch.empty((M, N // 128, 2), device=DEV)

    def run():
        y = torch.empty((M, N), device=DEV, dtype=BF)
        cp.check(lib.qvl_dense_pos_embed_ws(stream(), cp.QVL_DTYPE_BF16, x.data_ptr(), K, w.data_ptr(), b.data_ptr(),
                                            table.data_ptr(), idx.data_ptr(), tw.data_ptr(), y.data_ptr(), N, M, N, K,
                                            parts.data_ptr(), None, 0))
        return y, parts.clone()
    (y9, p9), (y3, _) = plans(run)
    prod = x.double() @ w.double().t()
    assert close(y9, y3, prod, prod + b.double())
    assert torch.allclose(p9[..., 0].double(), y9.double().view(M, -1, 128).sum(2), rtol=0, atol=1e-5 * 128)


# around the row count up to which a launch's idle workgroups read the next GEMM's weights, and the smallest grids
@pytest.mark.parametrize("shape", ["2b", "8b"])
@pytest.mark.parametrize("grids", [[(1, 2, 2)], [(1, 14, 14)], [(1, 28, 32)], [(1, 26, 34), (1, 2, 8)]])
def test_tower_reading_next_weights(pkg, lib, grids, shape):
    """64x128 tiles (whose launches read ahead) against 256x128 tiles (which do not), with a tap and both mergers: the
    same k order, so the same bits (the head_dim-72 qkv GEMM keeps its own tiles on both)."""
    from tests.test_gpu_parity_depth import ckpt_params, pixels, specs
    spec, ospec = specs(pkg, shape, depth=2, ds=(0,))
    tower = pkg.Qwen3VisionTransformer(spec, dtype="bfloat16").bind(ckpt_params(ospec, seed=5))
    px, g = pixels(grids, 5), np.array(grids, np.int32)
    out = []
    for plan in (8, 3):
        pkg.capi.check(lib.qvl_set_gemm_plan(plan, -1, 0))
        try:
            tok, ds = tower(px, g)
            out.append([t.clone() for t in (tok, *ds)])
        finally:
            pkg.capi.check(lib.qvl_set_gemm_plan(0, 0, 0))
    for a, b in zip(*out):
        assert torch.isfinite(a.float()).all() and torch.equal(a, b)
    tok, ds = tower(px, g)                            # the default plans: other K orders, so bf16 steps apart
    for a, b in zip((tok, *ds), out[0]):
        a, b = a.double(), b.double()
        assert (a - b).norm() <= 1e-2 * b.norm()
