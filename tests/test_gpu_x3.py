"""Batches through the tiled matrix-core products (x3gemm.hip), at the sizes where they can go wrong: the
edges of the token tiles (5, 16 and 32 tokens), one and several 512-column groups, K parts that do not
divide the columns evenly, a number of row blocks that is no multiple of anything.

Bar: 1e-6 relative 2-norm against a 64-bit product of the dequantized weights. The products are exact and
a row's sum is at most 48 MFMA roundings per 256 columns and one addition per 32 (int4) or 256 (MXFP4)
columns: rounding errors u = 2^-24 at random signs give u sqrt(n / 6) with n <= 256, about 4e-7.
"""
import numpy as np
import pytest

from helpers import HipGraph, normal, rel_l2
from test_gpu_moe import _small_layer

pytestmark = pytest.mark.gpu


def _matrix(ctx, orc, fmt, rows, cols, seed):
    import torch
    import rabbit_amd as R
    q = orc.synth_mxfp4(rows, cols, seed) if fmt == "mxfp4" else orc.synth_i4g(rows, cols, 32, seed)
    data, scale = torch.from_numpy(q.data).cuda(), torch.from_numpy(q.scale).cuda()
    w = R.QT.mxfp4(data, scale, rows, cols) if fmt == "mxfp4" else R.QT.i4g(data, scale, rows, cols, 32)
    return w, ctx.dequant_rows(w, 0, rows).reshape(rows, cols).double()


# tokens * columns * rows about the line where the tiled products take over, the GEMV below it
@pytest.mark.parametrize("fmt", ["mxfp4", "i4g"])
@pytest.mark.parametrize("cols,rows,tokens", [(7168, 3584, (2, 4, 5, 6, 16, 17, 33)), (512, 16512, (12, 32, 49)),
                                              (2048, 1152, (21, 22, 43, 48, 52, 130)), (4608, 640, (34, 41, 64, 65))])
def test_matmul_batches(ctx, orc, fmt, cols, rows, tokens):
    import torch
    w, dense = _matrix(ctx, orc, fmt, rows, cols, cols + rows)
    for s in tokens:
        x = torch.from_numpy(normal((s, cols), s)).cuda()
        y = torch.full((s + 1, rows), 7.0, device="cuda")
        ctx.matmul_qt(y[:s], x, w, s)
        err = float((y[:s].double() - x.double() @ dense.t()).norm() / (x.double() @ dense.t()).norm())
        assert err < 1e-6, (s, err)
        assert bool((y[s] == 7.0).all()), s  # nothing past the last token


@pytest.mark.parametrize("E,k,S", [(24, 4, 40), (24, 4, 61), (3, 2, 37), (2, 1, 70), (6, 6, 2)])
def test_int4_layer_batches(ctx, orc, E, k, S):
    """Grouped int4 layers whose experts take 1..5, 6..16 and 17..32 tokens, with the shared expert's tiles."""
    import rabbit_amd as R
    H, I = 512, 512
    L = _small_layer(ctx, orc, 1, R.QT_I4_GROUPED, H, I, E, k, seed=E + S)
    x = normal((S, H), S)
    exp, eids, _ = L.forward(x, S)
    out, ids, w = np.empty(S * H, np.float32), np.empty(S * k, np.int32), np.empty(S * k, np.float32)
    ctx.moe_forward(0, x, S, out, ids, w)
    assert np.array_equal(ids.reshape(S, k), eids)
    for t in range(S):
        assert rel_l2(out[t * H:(t + 1) * H], np.asarray(exp).reshape(S, H)[t]) < 1e-5, t


def test_captured_batches(rbt_lib, orc):
    """A batch captured on a context that never ran one (no scratch to be had inside the capture: the GEMV
    path, which needs none) and captured again after an eager call: every replay equals an eager call."""
    import torch
    import rabbit_amd as R
    ctx = R.Context(0)
    rows, cols, s = 3584, 7168, 9
    w, dense = _matrix(ctx, orc, "i4g", rows, cols, 3)
    x = torch.empty(s, cols, device="cuda")
    y = torch.empty(s, rows, device="cuda")
    q = w.c()
    import ctypes as C
    for _ in range(2):
        g = HipGraph(ctx.stream)
        torch.cuda.synchronize()
        g.begin()
        rc = ctx.lib.rbt_matmul_qt_d(ctx.h, y.data_ptr(), x.data_ptr(), C.byref(q), s)
        g.end()
        assert rc == 0
        for i in range(3):
            x.copy_(torch.from_numpy(normal((s, cols), 50 + i)))
            torch.cuda.synchronize()
            g.launch()
            ctx.sync()
            want = x.double() @ dense.t()
            assert float((y.double() - want).norm() / want.norm()) < 1e-6
            ye = torch.empty_like(y)
            ctx.matmul_qt(ye, x, w, s)
            assert float((y - ye).norm() / ye.norm()) < 1e-6
        g.destroy()
    ctx.close()


# 600 experts: the batch selection past 512 (the tiles from 80 tokens on); 24 experts of 1 to 40 tokens: every tile
# form with Situ
@pytest.mark.parametrize("E,k,S", [(600, 4, 2), (600, 4, 40), (600, 4, 80), (24, 4, 11), (24, 4, 16), (24, 4, 60), (6, 4, 66)])
def test_latent_batches(ctx, orc, E, k, S):
    import rabbit_amd as R
    from test_gpu_latent import _latent_case, _run_latent
    H, MH, I = 1024, 512, 512 if E < 600 or S == 80 else 64
    layer = 70 + E % 7
    L, dq, uq, _ = _latent_case(ctx, orc, layer, H, MH, I, E, k, 4000 + E, "i4g", 1.0)
    x = normal((S, H), S, 1.0)
    norm = np.abs(normal(MH, 5, 1.0)) + np.float32(0.5)
    _run_latent(ctx, R, layer, L, dq, uq, x, S, MH, norm, orc.situ(4.0, 25.0), R.situ(4.0, 25.0))


# nobody, one, 5, 6, 16, 17, 33 and 300 of the tokens pick the expert; K parts on both products
@pytest.mark.parametrize("fmt,d,i", [("mxfp4", 8192, 2048), ("i4g", 512, 8704), ("i4g", 512, 512)])
@pytest.mark.parametrize("s,picks", [(9, 0), (5, 1), (7, 5), (20, 6), (16, 16), (47, 17), (49, 33), (300, 300)])
def test_expert_batches(ctx, orc, fmt, d, i, s, picks):
    import torch
    import rabbit_amd as R
    (g, gd), (u, ud), (dn, dd) = (_matrix(ctx, orc, fmt, r, c, 11 + r + n) for n, (r, c) in
                                  enumerate(((i, d), (i, d), (d, i))))
    rng = np.random.default_rng(s)
    k = 3
    ids = rng.integers(1, 50, (s, k)).astype(np.int32)
    who = np.sort(rng.permutation(s)[:picks])
    ids[who, rng.integers(0, k, picks)] = 0
    ids[who[::2], k - 1] = 0  # some pick it twice: the first slot counts
    w = rng.standard_normal((s, k)).astype(np.float32)
    x = torch.from_numpy(normal((s, d), s)).cuda()
    out = torch.full((s, d), 0.5, device="cuda")
    slot = R.Slot(0, dn, gate=g, up=u)
    ctx.apply_single_expert(slot, torch.from_numpy(ids).cuda(), torch.from_numpy(w).cuda(), s, k, x, d, i, out)
    want = torch.full((s, d), 0.5, dtype=torch.float64, device="cuda")
    for t in who:
        h = torch.nn.functional.silu(gd @ x[t].double()) * (ud @ x[t].double())
        want[t] += float(w[t, list(ids[t]).index(0)]) * (dd @ h)
    assert float((out.double() - want).norm() / want.norm()) < 1e-6
    rest = torch.ones(s, dtype=torch.bool)
    rest[torch.from_numpy(who)] = False
    assert bool((out[rest.cuda()] == 0.5).all())


def test_grouping_past_the_lds_bitmaps(ctx, orc):
    """More (expert, 32-token word) bitmap words than one workgroup's LDS holds: the pairs come from their own
    launch. Unused experts on both ends of the ids, and a shared expert."""
    import rabbit_amd as R
    H, I, E, k, S = 512, 1024, 500, 3, 545
    L = _small_layer(ctx, orc, 0, R.QT_MXFP4, H, I, E, k, seed=77, gated=True)
    x = normal((S, H), 9)
    exp, eids, _ = L.forward(x, S)
    out, ids, w = np.empty(S * H, np.float32), np.empty(S * k, np.int32), np.empty(S * k, np.float32)
    ctx.moe_forward(0, x, S, out, ids, w)
    assert np.array_equal(ids.reshape(S, k), eids)
    assert rel_l2(out, exp) < 1e-2  # bf16 activations


def _device_matrix(fmt, n, rows, cols, seed):
    """n matrices on the device, codes and scales uniform, with their 64-bit values on demand."""
    import torch
    import rabbit_amd as R
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    data = torch.randint(0, 256, (n, rows, cols // 2), dtype=torch.uint8, device="cuda", generator=g)
    if fmt == "mxfp4":
        scale = torch.randint(119, 124, (n, rows, cols // 32), dtype=torch.uint8, device="cuda", generator=g)
        return lambda e: R.QT.mxfp4(data[e], scale[e], rows, cols)
    scale = torch.rand(n, rows, cols // 32, device="cuda", generator=g) * 0.015 + 0.005
    return lambda e: R.QT.i4g(data[e], scale[e], rows, cols, 32)


def _device_layer(ctx, fmt, H, I, E, k, shared, seed, layer=0, std=0.05, family=1, gated=False, skip=()):
    """A layer of device-resident experts (but for `skip`): {"gate"/"up"/"down": e -> QT (E: the shared expert), "router"}."""
    import torch
    import rabbit_amd as R
    m = {n: _device_matrix(fmt, E + 1, r, c, seed + i)
         for i, (n, r, c) in enumerate((("gate", I, H), ("up", I, H), ("down", H, I)))}
    slot = lambda e, eid: R.Slot(eid, m["down"](e), gate=m["gate"](e), up=m["up"](e))  # noqa: E731
    for e in set(range(E)) - set(skip):
        ctx.pool_put(layer, slot(e, e))
    router = torch.from_numpy(normal((E, H), seed + 9, std)).cuda()
    gate = torch.from_numpy(normal(H, seed + 8, std)).cuda() if gated else None
    ctx.moe_layer_set(layer, family, H, I, E, k, router, shared=slot(E, 0) if shared else None, shared_gate=gate)
    return m, router


def _ffn64(ctx, m, e, x):
    """down(silu(gate x) * up x) of one expert in 64 bits, the weights dequantized."""
    import torch
    w = {n: ctx.dequant_rows(f(e), 0, f(e).rows).reshape(f(e).rows, f(e).cols).double() for n, f in m.items()}
    return (torch.nn.functional.silu(x @ w["gate"].t()) * (x @ w["up"].t())) @ w["down"].t()


def test_int4_layer_many_tokens_wide_experts(own_ctx):
    """More than 2^32 bytes of the down product's activation parts (6 * tokens * inter): the offsets a lane
    holds in 32 bits reach over one tile there, so the call's size does not bound them. Checked at the first and
    last tokens of the call and of each expert's tiles."""
    import torch
    ctx = own_ctx
    H, I, E, k, S = 512, 65536, 2, 1, 10945
    m, _ = _device_layer(ctx, "i4g", H, I, E, k, True, 300)
    g = torch.Generator(device="cuda")
    g.manual_seed(3)
    x = torch.randn(S, H, device="cuda", generator=g)
    out = torch.empty(S, H, device="cuda")
    ids, w = torch.empty(S, k, dtype=torch.int32, device="cuda"), torch.empty(S, k, device="cuda")
    ctx.moe_forward(0, x, S, out, ids, w)
    picked = set(range(4)) | set(range(S - 4, S))
    for e in range(E):
        t = torch.nonzero(ids[:, 0] == e).flatten().tolist()
        assert len(t) > 100
        picked |= {t[0], t[15], t[16], t[31], t[32], t[-2], t[-1]}
    rows = torch.tensor(sorted(picked), device="cuda")
    xr = x[rows].double()
    want = _ffn64(ctx, m, E, xr)
    for e in range(E):
        at = torch.nonzero(ids[rows, 0] == e).flatten()
        want[at] += w[rows[at], 0].double()[:, None] * _ffn64(ctx, m, e, xr[at])
    err = (out[rows].double() - want).norm(dim=1) / want.norm(dim=1)
    assert float(err.max()) < 1e-5, err


@pytest.mark.parametrize("family", [0, 1])
def test_routing_weights_of_short_prompts(own_ctx, family):
    """The routing weights of 37 tokens (router logits on the matrix cores) are no further from 64 bits than
    those of the same tokens in calls of at most 16 (certified logits), and name the same experts."""
    import torch
    H, I, E, k, S = 4096, 1024, 512, 10, 37
    _, router = _device_layer(own_ctx, "mxfp4", H, I, E, k, True, 500, std=0.03, family=family, gated=family == 0)
    x = torch.from_numpy(normal((S, H), 41)).cuda()

    def call(t):
        n = t.shape[0]
        out = torch.empty(n, H, device="cuda")
        ids, w = torch.empty(n, k, dtype=torch.int32, device="cuda"), torch.empty(n, k, device="cuda")
        own_ctx.moe_forward(0, t, n, out, ids, w)
        return ids, w

    ids, w = call(x)
    small = [call(x[a:a + 16].contiguous()) for a in range(0, S, 16)]
    assert bool((ids == torch.cat([i for i, _ in small])).all())
    logits = torch.gather(x.double() @ router.double().t(), 1, ids.long())
    p = torch.softmax(logits, dim=1) if family == 0 else torch.sigmoid(logits)
    want = p if family == 0 else p / (p.sum(1, keepdim=True) + 1e-20)
    err = [float((v.double() - want).norm() / want.norm()) for v in (w, torch.cat([v for _, v in small]))]
    print("error against 64 bits: one call", err[0], "small calls", err[1])
    assert err[0] <= err[1], err


@pytest.mark.parametrize("H,E,S,cores", [(1024, 16, 63, False), (2048, 160, 62, False), (2048, 160, 63, True),
                                           (512, 16, 17, True), (512, 512, 17, True), (576, 40, 70, True)])
def test_router_of_short_prompts(own_ctx, H, E, S, cores):
    """Few tokens times experts keep the certified logits (the matrix cores' were up to half slower there)."""
    import torch
    I, k = 1024, 4
    _device_layer(own_ctx, "mxfp4", H, I, E, k, False, 600)
    x, out = torch.from_numpy(normal((S, H), 3)).cuda(), torch.empty(S, H, device="cuda")
    own_ctx.profile_kernels()
    own_ctx.moe_forward(0, x, S, out)
    names = " ".join(own_ctx.profile_kernels_read())
    own_ctx.profile_kernels(False)
    assert ("k_rcert" in names) == cores, names
    ids, one = (torch.empty(n, k, dtype=torch.int32, device="cuda") for n in (S, 1))
    own_ctx.moe_forward(0, x, S, out, ids)
    for t in range(0, S, 8):
        own_ctx.moe_forward(0, x[t:t + 1].contiguous(), 1, out, one)
        assert bool((ids[t] == one[0]).all()), t


@pytest.mark.parametrize("E,k,shared,I,S", [(16, 1, False, 1024, 40), (16, 1, True, 512, 40), (4, 4, False, 512, 3),
                                               (4, 4, False, 8704, 3), (6, 6, True, 8704, 2)])
def test_int4_layer_work_area(own_ctx, E, k, shared, I, S):
    """One expert per token, with and without a shared one: what the tiled products keep beside the rows lies
    between the rows and h, and a layer that leaves too little room there takes the GEMVs."""
    import torch
    H = 1024
    m, _ = _device_layer(own_ctx, "i4g", H, I, E, k, shared, 700)
    x, out = torch.from_numpy(normal((S, H), 5)).cuda(), torch.full((S + 1, H), 7.0, device="cuda")
    ids, w = torch.empty(S, k, dtype=torch.int32, device="cuda"), torch.empty(S, k, device="cuda")
    own_ctx.moe_forward(0, x, S, out[:S], ids, w)
    want = _ffn64(own_ctx, m, E, x.double()) if shared else torch.zeros(S, H, dtype=torch.float64, device="cuda")
    for e in range(E):
        t, j = torch.nonzero(ids == e, as_tuple=True)
        want[t] += w[t, j].double()[:, None] * _ffn64(own_ctx, m, e, x[t].double())
    assert float(((out[:S].double() - want).norm(dim=1) / want.norm(dim=1)).max()) < 2e-6
    assert bool((out[S] == 7.0).all())


@pytest.mark.parametrize("H,I,E,k,shared,S,tiled", [(4096, 1024, 16, 1, True, 8, False), (4096, 1024, 16, 1, True, 24, True),
                                                    (1024, 1024, 8, 2, False, 6, False), (1024, 1024, 8, 2, False, 24, True),
                                                    (512, 8704, 4, 1, False, 2, True)])
def test_int4_layer_choice(own_ctx, H, I, E, k, shared, S, tiled):
    """Where the tiles are too few to fill the chip the GEMVs run (the tiled products were up to 1.8 times as
    long there)."""
    import torch
    _device_layer(own_ctx, "i4g", H, I, E, k, shared, 800)
    x, out = torch.from_numpy(normal((S, H), 3)).cuda(), torch.empty(S, H, device="cuda")
    own_ctx.profile_kernels()
    own_ctx.moe_forward(0, x, S, out)
    names = " ".join(own_ctx.profile_kernels_read())
    own_ctx.profile_kernels(False)
    assert ("4k_x3I" in names) == tiled, names


# grouped int4 in one grouping launch and (more bitmap words than its LDS holds) in two, MXFP4 as a decode batch
# and as a prompt (bf16 activations)
@pytest.mark.parametrize("fmt,I,E,k,S,tol", [("i4g", 1024, 8, 2, 40, 2e-6), ("i4g", 512, 520, 2, 520, 2e-6),
                                             ("mxfp4", 1024, 8, 2, 12, 2e-6), ("mxfp4", 1024, 8, 2, 40, 1e-2)])
def test_missing_expert_of_a_batch(own_ctx, fmt, I, E, k, S, tol):
    """A picked expert without weights is an error, and the other experts' rows are what they are: its own count
    as zeros, whatever the work area held."""
    import torch
    import rabbit_amd as R
    H, gone = 1024, 3
    m, _ = _device_layer(own_ctx, fmt, H, I, E, k, True, 900)
    x, out = torch.from_numpy(normal((S, H), 5)).cuda(), torch.empty(S, H, device="cuda")
    ids, w = torch.empty(S, k, dtype=torch.int32, device="cuda"), torch.empty(S, k, device="cuda")
    own_ctx.moe_forward(0, x, S, out, ids, w)  # every expert there: leaves its rows behind
    keep, _ = _device_layer(own_ctx, fmt, H, I, E, k, True, 900, layer=1, skip=(gone,))
    with pytest.raises(R.RbtError) as ei:
        own_ctx.moe_forward(1, x, S, out, ids, w)
    assert ei.value.status == R.abi.RBT_E_NOT_RESIDENT
    assert bool((ids == gone).any())
    want = _ffn64(own_ctx, m, E, x.double())
    for e in range(E):
        if e != gone:
            t, j = torch.nonzero(ids == e, as_tuple=True)
            want[t] += w[t, j].double()[:, None] * _ffn64(own_ctx, m, e, x[t].double())
    assert float(((out.double() - want).norm(dim=1) / want.norm(dim=1)).max()) < tol


@pytest.mark.parametrize("fmt,cols,rows,s,tiled", [
    ("mxfp4", 2048, 2048, 24, False), ("mxfp4", 2048, 2048, 33, True), ("mxfp4", 4096, 4096, 6, False),
    ("mxfp4", 4096, 4096, 7, True), ("mxfp4", 8192, 2048, 2, False), ("mxfp4", 8192, 2048, 3, True),
    ("mxfp4", 16384, 128, 2, True), ("mxfp4", 2048, 8192, 5, True), ("i4g", 2048, 2048, 24, False),
    ("i4g", 2048, 2048, 33, True), ("i4g", 3584, 7168, 2, False), ("i4g", 3584, 7168, 3, True)])
def test_matmul_choice(own_ctx, fmt, cols, rows, s, tiled):
    """Small products keep the GEMV (the tiled ones were up to a sixth slower near the line)."""
    import torch
    q = _device_matrix(fmt, 1, rows, cols, 5)(0)
    x, y = torch.from_numpy(normal((s, cols), 3)).cuda(), torch.empty(s, rows, device="cuda")
    own_ctx.profile_kernels()
    own_ctx.matmul_qt(y, x, q, s)
    names = " ".join(own_ctx.profile_kernels_read())
    own_ctx.profile_kernels(False)
    assert ("4k_x3I" in names) == tiled, names


@pytest.mark.parametrize("fmt", ["mxfp4", "i4g"])
def test_matmul_runs(own_ctx, fmt):
    """A batch whose activations' parts go through in three runs of 672, 672 and 57 tokens."""
    import torch
    cols, rows, s = 65536, 128, 1401
    q = _device_matrix(fmt, 1, rows, cols, 6)(0)
    g = torch.Generator(device="cuda")
    g.manual_seed(4)
    x, y = torch.randn(s, cols, device="cuda", generator=g), torch.full((s + 1, rows), 7.0, device="cuda")
    own_ctx.matmul_qt(y[:s], x, q, s)
    want = x.double() @ own_ctx.dequant_rows(q, 0, rows).reshape(rows, cols).double().t()
    assert float(((y[:s].double() - want).norm(dim=1) / want.norm(dim=1)).max()) < 2e-6
    assert bool((y[s] == 7.0).all())


def test_matmul_scratch_is_bounded(own_ctx):
    """What a large batch through one matrix leaves in the context does not grow with its tokens."""
    import torch
    cols, rows, s = 8192, 2048, 16384
    q = _device_matrix("mxfp4", 1, rows, cols, 7)(0)
    x, y = torch.randn(s, cols, device="cuda"), torch.empty(s, rows, device="cuda")
    torch.cuda.synchronize()
    free = torch.cuda.mem_get_info()[0]
    own_ctx.matmul_qt(y, x, q, s)
    assert free - torch.cuda.mem_get_info()[0] < 400 << 20


def test_captures_outlive_larger_calls(own_ctx):
    """A captured batch through one matrix and a captured decode batch of a layer replay right after larger
    eager calls made the context's scratch grow: the graphs' buffers stay. The memory a growth gives back is
    written over before each replay."""
    import ctypes as C
    import torch
    H, I, E, k, S = 1024, 1024, 8, 2, 12
    m, _ = _device_layer(own_ctx, "mxfp4", H, I, E, k, False, 950)
    q = _device_matrix("i4g", 1, 3584, 7168, 8)(0)
    dense = own_ctx.dequant_rows(q, 0, 3584).reshape(3584, 7168).double()
    x, y = torch.empty(9, 7168, device="cuda"), torch.empty(9, 3584, device="cuda")
    xl, out = torch.empty(S, H, device="cuda"), torch.empty(S, H, device="cuda")
    lib, qc = own_ctx.lib, q.c()
    product = lambda: lib.rbt_matmul_qt_d(own_ctx.h, y.data_ptr(), x.data_ptr(), C.byref(qc), 9)  # noqa: E731
    layer = lambda: lib.rbt_moe_forward_d(own_ctx.h, 0, xl.data_ptr(), S, out.data_ptr(), None, None)  # noqa: E731

    def fill(seed):
        x.copy_(torch.from_numpy(normal((9, 7168), seed)))
        xl.copy_(torch.from_numpy(normal((S, H), seed + 1)))
        torch.cuda.synchronize()

    fill(1)
    graphs = []
    for call in (product, layer):
        assert call() == 0  # eager first: the scratch is there
        own_ctx.sync()
        g = HipGraph(own_ctx.stream)
        g.begin()
        rc = call()
        g.end()
        assert rc == 0
        graphs.append(g)
    for i, s in enumerate((700, 1500, 3000)):
        print("larger calls", s, flush=True)
        own_ctx.matmul_qt(torch.empty(s, 3584, device="cuda"), torch.randn(s, 7168, device="cuda"), q, s)
        own_ctx.moe_forward(0, torch.randn(s, H, device="cuda"), s, torch.empty(s, H, device="cuda"))
        torch.full((64 << 20,), float("nan"), device="cuda")
        fill(10 + i)
        for g in graphs:
            g.launch()
        own_ctx.sync()
        got, want = y.clone(), x.double() @ dense.t()
        assert float((got.double() - want).norm() / want.norm()) < 1e-6
        rows = out.clone()
        assert layer() == 0
        own_ctx.sync()
        assert torch.equal(rows, out)
    for g in graphs:
        g.destroy()


@pytest.mark.parametrize("fmt,d,i,s,tiled", [("mxfp4", 8192, 2048, 5, True), ("mxfp4", 6144, 2048, 4, False),
                                             ("i4g", 2048, 1024, 25, False), ("i4g", 2048, 1024, 26, True),
                                             ("i4g", 512, 512, 200, False), ("i4g", 512, 8704, 2, True)])
def test_expert_choice(own_ctx, fmt, d, i, s, tiled):
    """Small experts keep the GEMVs for longer (the tiled products were up to a fifth slower there)."""
    import torch
    import rabbit_amd as R
    g, u, dn = (_device_matrix(fmt, 1, r, c, 5)(0) for r, c in ((i, d), (i, d), (d, i)))
    ids, w = torch.zeros(s, 2, dtype=torch.int32, device="cuda"), torch.ones(s, 2, device="cuda")
    x, out = torch.from_numpy(normal((s, d), 3)).cuda(), torch.zeros(s, d, device="cuda")
    own_ctx.profile_kernels()
    own_ctx.apply_single_expert(R.Slot(0, dn, gate=g, up=u), ids, w, s, 2, x, d, i, out)
    names = " ".join(own_ctx.profile_kernels_read())
    own_ctx.profile_kernels(False)
    assert ("4k_x3I" in names) == tiled, names


def test_latent_norm_in_the_projection(own_ctx, orc):
    """An up projection that is large enough for the tiled product but of a shape it does not take keeps the norm
    inside its GEMV (no launch of its own for the norm)."""
    import rabbit_amd as R
    from test_gpu_latent import _latent_case, _run_latent
    H, MH, I, E, k, S = 1088, 1024, 64, 4, 2, 96
    L, dq, uq, _ = _latent_case(own_ctx, orc, 0, H, MH, I, E, k, 7000, "i4g", 1.0)
    norm = np.abs(normal(MH, 5, 1.0)) + np.float32(0.5)
    own_ctx.profile_kernels()
    _run_latent(own_ctx, R, 0, L, dq, uq, normal((S, H), 2), S, MH, norm, orc.situ(4.0, 25.0), R.situ(4.0, 25.0))
    names = " ".join(own_ctx.profile_kernels_read())
    own_ctx.profile_kernels(False)
    assert "k_rmsnorm" not in names, names


@pytest.mark.parametrize("s", [9, 20, 36])
def test_extreme_mxfp4_scales(own_ctx, s):
    """Infinite and nearly infinite weights (E8M0 253 and 254; a block of 255 is NaN, as in the GEMVs), the smallest
    scales, infinite and NaN activations: each output is the infinity, the NaN or the number that the 64-bit
    product gives. Activations of 1 to 24
    significant bits meet the infinite weights, so that their lower parts are zero or not. Tiles of up to 5, 16
    and 32 tokens."""
    import torch
    import rabbit_amd as R
    rows, cols = 3584, 3584
    g = torch.Generator(device="cuda")
    g.manual_seed(9)
    data = torch.randint(0, 256, (rows, cols // 2), dtype=torch.uint8, device="cuda", generator=g)
    scale = torch.randint(119, 124, (rows, cols // 32), dtype=torch.uint8, device="cuda", generator=g)
    data[:8, 160:176] = 0                    # block 10 of the first rows: zeros but for one code
    for row, byte, code in ((0, 254, 7), (1, 254, 15), (2, 254, 1), (3, 253, 7), (5, 0, 7), (6, 1, 1)):
        scale[row, 10], data[row, 160] = byte, code
    data[4, 160:176], scale[4, 10] = 0x77, 255
    x = torch.randn(s, cols, device="cuda", generator=g)
    x[:, 320:352] = torch.randn(s, 32, device="cuda", generator=g).abs().bfloat16().float().clamp(0.25, 1.9)
    x[0, 320], x[1, 320], x[2, 320], x[3, 320], x[4, 320] = 1.0, -1.5, 1.0 + 2.0 ** -10, 1.0 + 2.0 ** -23, -0.75
    x[5, 40], x[6, 40], x[7, 40] = float("inf"), -float("inf"), float("nan")
    w = R.QT.mxfp4(data, scale, rows, cols)
    y = torch.empty(s, rows, device="cuda")
    own_ctx.matmul_qt(y, x, w, s)
    dense = own_ctx.dequant_rows(w, 0, rows).reshape(rows, cols).double()
    want = torch.stack([(x[t].double()[None, :] * dense).sum(1) for t in range(s)])
    assert int(torch.isinf(want[:5, [0, 1, 3]]).sum()) == 15
    want[:, 4] = float("nan")
    fin = torch.isfinite(want)
    assert bool((torch.isnan(want) == torch.isnan(y)).all())
    inf = torch.isinf(want)
    assert bool((want[inf] == y[inf].double()).all())
    err = (y[fin].double() - want[fin]).abs() / want.abs().masked_fill(~fin, 0).amax(1, keepdim=True).expand_as(want)[fin]
    assert float(err.max()) < 1e-5
    ordinary = fin.clone()
    ordinary[:, :8] = False
    assert float((y.double() - want)[ordinary].norm() / want[ordinary].norm()) < 1e-6


def test_precision_of_short_activations(own_ctx):
    """Activations that are bf16 values: no further from 64 bits than full ones (the bar of test_matmul_batches)."""
    import torch
    q = _device_matrix("mxfp4", 1, 3584, 7168, 11)(0)
    dense = own_ctx.dequant_rows(q, 0, 3584).reshape(3584, 7168).double()
    for s in (4, 16, 64):
        x = torch.from_numpy(normal((s, 7168), s)).cuda()
        errs = []
        for v in (x.bfloat16().float(), x):
            y = torch.empty(s, 3584, device="cuda")
            own_ctx.matmul_qt(y, v, q, s)
            want = v.double() @ dense.t()
            errs.append(float((y.double() - want).norm() / want.norm()))
        print("error against 64 bits", s, errs)
        assert errs[0] < 1e-6


@pytest.mark.parametrize("fmt", ["mxfp4", "i4g"])
@pytest.mark.parametrize("what", ["x", "y", "data", "scale"])
def test_matmul_unaligned(own_ctx, fmt, what):
    """A batch whose x, y, codes or scales are not 16-byte aligned keeps the kernels that take them."""
    import torch
    import rabbit_amd as R
    cols, rows, s = 2048, 2048, 40
    q = _device_matrix(fmt, 1, rows, cols, 12)(0)

    def off(t, skip):  # the tensor's values, its first byte `skip` bytes past a 16-byte boundary
        n = skip // t.element_size()
        b = torch.empty(t.numel() + 32, dtype=t.dtype, device="cuda")[n:n + t.numel()].view(t.shape)
        b.copy_(t)
        assert b.data_ptr() % 16 == skip
        return b

    x, y = torch.from_numpy(normal((s, cols), 3)).cuda(), torch.empty(s, rows, device="cuda")
    data, scale = q.data, q.scale
    want = x.double() @ own_ctx.dequant_rows(q, 0, rows).reshape(rows, cols).double().t()
    x, y = (off(x, 4) if what == "x" else x), (off(y, 4) if what == "y" else y)
    data, scale = (off(data, 8) if what == "data" else data), (off(scale, 4) if what == "scale" else scale)
    w = R.QT.mxfp4(data, scale, rows, cols) if fmt == "mxfp4" else R.QT.i4g(data, scale, rows, cols, 32)
    own_ctx.profile_kernels()
    own_ctx.matmul_qt(y, x, w, s)
    names = " ".join(own_ctx.profile_kernels_read())
    own_ctx.profile_kernels(False)
    assert "4k_x3I" not in names
    assert float((y.double() - want).norm() / want.norm()) < 1e-6


@pytest.mark.parametrize("latent", [False, True])
def test_captured_layer_batches(own_ctx, orc, latent):
    """An int4 layer's batch and a latent one, captured after an eager call: every replay is the eager call, bit for
    bit, with eager calls in between."""
    import ctypes as C
    import torch
    import rabbit_amd as R
    from rabbit_amd import abi
    from test_gpu_latent import _latent_case
    lib, p = own_ctx.lib, lambda t: t.data_ptr()  # noqa: E731
    k, S = 4, 60
    if latent:
        H, MH, E = 1024, 512, 24
        _, dq, uq, _ = _latent_case(own_ctx, orc, 0, H, MH, 512, E, k, 8000, "i4g", 1.0)
        keep = [torch.from_numpy(a).cuda() for q in (dq, uq) for a in (q.data, q.scale)]
        norm = torch.ones(MH, device="cuda")
        lw = abi.RbtLatentMoeDesc(MH, R.QT.i4g(keep[0], keep[1], MH, H, 32).c(), R.QT.i4g(keep[2], keep[3], H, MH, 32).c(),
                                  p(norm), 1e-5, R.situ(4.0, 25.0))
        call = lambda x, o, i, w: lib.rbt_latent_moe_d(own_ctx.h, 0, C.byref(lw), p(x), S, p(o), p(i), p(w))  # noqa: E731
    else:
        H, E = 1024, 24
        _device_layer(own_ctx, "i4g", H, 1024, E, k, True, 1000)
        call = lambda x, o, i, w: lib.rbt_moe_forward_d(own_ctx.h, 0, p(x), S, p(o), p(i), p(w))  # noqa: E731
    new = lambda: [torch.empty(S, H, device="cuda"), torch.empty(S, k, dtype=torch.int32, device="cuda"),  # noqa: E731
                   torch.empty(S, k, device="cuda")]
    x, got, want = torch.from_numpy(normal((S, H), 1)).cuda(), new(), new()
    torch.cuda.synchronize()
    own_ctx.profile_kernels()
    assert call(x, *got) == 0
    own_ctx.sync()
    assert "4k_x3I" in " ".join(own_ctx.profile_kernels_read())
    own_ctx.profile_kernels(False)
    g = HipGraph(own_ctx.stream)
    g.begin()
    rc = call(x, *got)
    g.end()
    assert rc == 0
    for i in range(3):
        x.copy_(torch.from_numpy(normal((S, H), 20 + i)))
        torch.cuda.synchronize()
        g.launch()
        own_ctx.sync()
        assert call(x, *want) == 0
        own_ctx.sync()
        for a, b in zip(got, want):
            assert torch.equal(a, b)
    g.destroy()
