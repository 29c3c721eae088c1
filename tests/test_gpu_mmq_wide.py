"""The 128 x 128 MMQ tile (65 tokens and more on matrices of more than 64
64 x 256 tiles, rows a multiple of 4) at the edges of its tiles: a last token
tile of at most 64 tokens, ragged rows, one to sixteen K steps, every schedule,
the accumulating and the unaligned store, both weight layouts; several matrices
in one launch, whole and split along K; and the rules that choose between this
tile and 64 x 256. On exact inputs (test_gpu_exact: one d8, one d) every
schedule must give the dequantized product bit for bit; on random inputs, where
each token and sub-block has its own scales, the product is the MMQ oracle's
within 2e-5 * rms (the same terms in another order)."""
import ctypes

import numpy as np
import pytest

import q3q4
from oracle import oracle
from test_gpu_exact import assert_bits, dev, exact_inputs, expected, mmq_stage, nan_out, say, torch  # noqa: F401

pytestmark = pytest.mark.gpu

# (M, N, K): ragged rows (N % 128 != 0) or whole ones
CASES = [(65, 16404, 256), (128, 8452, 512), (129, 5636, 768), (192, 5632, 768), (193, 4356, 256), (321, 3332, 512)]


@pytest.mark.parametrize("M,N,K", CASES)
def test_wide_tile_exact(torch, M, N, K):  # noqa: F811
    L = q3q4.load()
    tiles = -(-M // 128) * -(-N // 128)
    assert L.sera_q4k_mmq_tiles(M, N) == tiles, "not a wide-tile case"
    rng = np.random.default_rng(M * 3 + N + K)
    W, X = exact_inputs(rng, M, N, K)
    ref = expected(W, X, N, K)
    st, nkb = mmq_stage(torch, X), K // 256
    layouts = [(12, dev(torch, W))]
    if N % 16 == 0:
        layouts.append((q3q4.QTYPE_Q4K_TILED, dev(torch, q3q4.q4k_tiled_bytes(W, N, K))))
    for qt, Wd in layouts:
        for s in sorted({1, nkb}):
            say(f"case wide plain qt={qt} M={M} N={N} K={K} splits={s}")
            y = nan_out(torch, M, N)
            part = torch.empty(s * M * N, dtype=torch.float32, device="cuda") if s > 1 else None
            q3q4.mmq(Wd, st, y, M, N, K, splits=s, partial=part, qtype=qt)
            torch.cuda.synchronize()
            assert_bits(y, ref, f"plain splits={s}")
        for dp, pieces in sorted({(tiles, 1), (0, nkb), (tiles - 1, nkb), (tiles // 2, 1)}):
            say(f"case wide tail qt={qt} M={M} N={N} K={K} dp_tiles={dp} pieces={pieces}")
            slots = torch.empty(max(q3q4.mmq_tail_slot_floats(M, N, dp, pieces), 1), dtype=torch.float32, device="cuda")
            counters = torch.zeros(max(tiles - dp, 1), dtype=torch.int32, device="cuda")
            y = nan_out(torch, M, N)
            q3q4.mmq_tail(Wd, st, y, M, N, K, dp, pieces, slots=slots, counters=counters, qtype=qt)
            torch.cuda.synchronize()
            assert int(counters.abs().sum()) == 0, "tile counters not reset"
            assert_bits(y, ref, f"tail dp_tiles={dp} pieces={pieces}")
        say(f"case wide stream-K qt={qt} M={M} N={N} K={K}")
        slots = torch.empty(2 * 8 * L.sera_q4k_mmq_slot_floats(M), dtype=torch.float32, device="cuda")
        counters = torch.zeros(tiles, dtype=torch.int32, device="cuda")
        y = nan_out(torch, M, N)
        q3q4.mmq_streamk(Wd, st, y, M, N, K, slots, counters, wgs=8, qtype=qt)
        torch.cuda.synchronize()
        assert int(counters.abs().sum()) == 0, "tile counters not reset"
        assert_bits(y, ref, "stream-K")
    # Y at a 4-byte aligned address and accumulation: y0 + product, bit for bit
    qt, Wd = layouts[0]
    buf = torch.full((M * N + 2,), -7.0, dtype=torch.float32, device="cuda")
    y = buf[1:1 + M * N].view(M, N)
    say(f"case wide accumulate, unaligned Y M={M} N={N} K={K}")
    base = torch.from_numpy(rng.integers(-4, 5, (M, N)).astype(np.float32)).cuda()
    y.copy_(base)
    q3q4.mmq_tail(Wd, st, y, M, N, K, tiles, 1, accum=True)
    torch.cuda.synchronize()
    assert np.array_equal(y.cpu().numpy(), base.cpu().numpy() + ref.astype(np.float32))
    assert float(buf[0]) == -7.0 and float(buf[-1]) == -7.0, "store past Y"


def random_inputs(rng, M, K, rows):
    """Activations with outlier channels, and Q4_K rows."""
    X = rng.standard_normal((M, K)).astype(np.float32)
    X[:, rng.choice(K, K // 100, replace=False)] *= 20.0
    return X, [oracle.quantize_q4k((rng.standard_normal((n, K)) * 0.02).astype(np.float32)) for n in rows]


def assert_oracle(y, W, q, what):
    """Sampled rows (the first and last tiles' among them) of y, all tokens,
    against the MMQ oracle on the staged activations q = (quants, d8, s8)."""
    N, K = W.shape[0], q[0].shape[1]
    rows = np.unique(np.r_[0:4, N - 20:N, np.linspace(0, N - 1, 60).astype(int)])
    ref = oracle.gemm_mmq(W[rows], *q, len(rows), K)
    err = float(np.max(np.abs(y[:, rows].astype(np.float64) - ref)) / np.sqrt(np.mean(ref * ref)))
    say(f"  {what}: max|err| / rms = {err:.2e}")
    assert np.all(np.isfinite(y)) and err <= 2e-5, what


# M % 128 in 1..64: the 64-token body beside the 128-token one (192: as its only second tile); rows a multiple of 16 that
# do not fill a tile, both layouts; eight and sixteen K steps; whole, all split, one tile split
@pytest.mark.parametrize("M,N,K", [(129, 5648, 2304), (192, 5636, 2048), (577, 2064, 4096)])
def test_wide_tile_scales(torch, M, N, K):  # noqa: F811
    tiles = -(-M // 128) * -(-N // 128)
    assert q3q4.load().sera_q4k_mmq_tiles(M, N) == tiles, "not a wide-tile case"
    X, (W,) = random_inputs(np.random.default_rng(M + N + K), M, K, [N])
    W = W.reshape(N, -1)
    q, st = oracle.q8_1_mmq(X), mmq_stage(torch, X)
    layouts = [(12, dev(torch, W))]
    if N % 16 == 0:
        layouts.append((q3q4.QTYPE_Q4K_TILED, dev(torch, q3q4.q4k_tiled_bytes(W, N, K))))
    for qt, Wd in layouts:
        for dp, pieces in ((tiles, 1), (0, 3), (tiles - 1, K // 256)):
            say(f"case wide scales qt={qt} M={M} N={N} K={K} dp_tiles={dp} pieces={pieces}")
            slots = torch.empty(max(q3q4.mmq_tail_slot_floats(M, N, dp, pieces), 1), dtype=torch.float32, device="cuda")
            counters = torch.zeros(max(tiles - dp, 1), dtype=torch.int32, device="cuda")
            y = nan_out(torch, M, N)
            q3q4.mmq_tail(Wd, st, y, M, N, K, dp, pieces, slots=slots, counters=counters, qtype=qt)
            torch.cuda.synchronize()
            assert int(counters.abs().sum()) == 0, "tile counters not reset"
            assert_oracle(y.cpu().numpy(), W, q, f"dp_tiles={dp} pieces={pieces}")


# all tiles split along K, and whole rounds before a split tail; a matrix whose last row tile is ragged between others
@pytest.mark.parametrize("M,Ns,K", [(129, [4096, 1024, 528], 2560), (193, [4096, 1040, 528, 64], 4096),
                                    (577, [7168, 6400], 2304)])
def test_group_split_along_k(torch, M, Ns, K):  # noqa: F811
    """A grouped launch whose plan has several pieces: every matrix against the
    oracle, plain, with RMSNorm, on tiles, accumulating (product + add bit for
    bit), into outputs that are only 4-byte aligned, replayed from a graph
    between eager calls, and whole where the arena has no room for slots."""
    L = q3q4.load()
    lin = q3q4.Linear(device=0, max_tokens=640, max_features=8192, max_k=4096)
    dp, pieces = ctypes.c_int(), ctypes.c_int()
    cus = torch.cuda.get_device_properties(0).multi_processor_count
    tiles = L.sera_mmq_group_plan(M, len(Ns), (ctypes.c_int * len(Ns))(*Ns), K, cus, ctypes.c_size_t(1 << 25),
                                  ctypes.byref(dp), ctypes.byref(pieces))
    assert tiles == -(-M // 128) * sum(-(-n // 128) for n in Ns) and pieces.value > 1 and (dp.value > 0) == (M == 577)
    rng = np.random.default_rng(M + sum(Ns) + K)
    X, Ws = random_inputs(rng, M, K, Ns)
    Ws = [w.reshape(n, -1) for w, n in zip(Ws, Ns)]
    Xd, Wd, geos = dev(torch, X), [dev(torch, w) for w in Ws], [q3q4.bind_geometry(12, K, n) for n in Ns]
    say(f"case group split M={M} Ns={Ns} K={K} dp_tiles={dp.value} of {tiles} pieces={pieces.value}")

    def run(ys, **kw):
        q3q4.linear_group(kw.pop("geos", geos), kw.pop("W", Wd), ys, Xd, **kw)
        torch.cuda.synchronize()
        assert int(lin.workspace[:256 << 10].to(torch.int32).abs().sum()) == 0, "counters not reset"
        return ys

    q = oracle.q8_1_mmq(X)
    plain = run([nan_out(torch, M, n) for n in Ns])
    for y, w in zip(plain, Ws):
        assert_oracle(y.cpu().numpy(), w, q, "plain")
    gamma = (1.0 + 0.1 * rng.standard_normal(K)).astype(np.float32)
    qn = oracle.q8_1_mmq(oracle.rmsnorm_fused_order(X, gamma, 1e-6))
    for y, w in zip(run([nan_out(torch, M, n) for n in Ns], gamma=dev(torch, gamma), eps=1e-6, flags=q3q4.LIN_RMSNORM), Ws):
        assert_oracle(y.cpu().numpy(), w, qn, "RMSNorm")
    tiled = run([nan_out(torch, M, n) for n in Ns], geos=[q3q4.bind_geometry(q3q4.QTYPE_Q4K_TILED, K, n) for n in Ns],
                W=[dev(torch, q3q4.q4k_tiled_bytes(w, n, K)) for w, n in zip(Ws, Ns)])
    base = [torch.randn((M, n), device="cuda") for n in Ns]
    acc = run([b.clone() for b in base], flags=q3q4.LIN_ACCUMULATE)
    bufs = [torch.full((M * n + 1,), -7.0, device="cuda") for n in Ns]
    odd = run([b[1:].view(M, n) for b, n in zip(bufs, Ns)])
    for i in range(len(Ns)):
        assert torch.equal(tiled[i], plain[i]) and torch.equal(odd[i], plain[i]) and float(bufs[i][0]) == -7.0
        assert torch.equal(acc[i], base[i] + plain[i])
    ys = [torch.zeros((M, n), device="cuda") for n in Ns]
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        q3q4.linear_group(geos, Wd, ys, Xd)
    for _ in range(3):
        for y in ys:
            y.fill_(float("nan"))
        graph.replay()
        torch.cuda.synchronize()
        assert all(torch.equal(a, b) for a, b in zip(ys, plain)), "replay differs"
        run([nan_out(torch, M, n) for n in Ns])
    stage = q3q4.mmq_stage_layout(M, K)["total"]
    small = torch.zeros((256 << 10) + stage, dtype=torch.uint8, device="cuda")
    assert L.sera_q4k_set_arena(ctypes.c_void_p(small.data_ptr()), small.numel()) == 0
    ys = [nan_out(torch, M, n) for n in Ns]
    q3q4.linear_group(geos, Wd, ys, Xd)
    torch.cuda.synchronize()
    for y, w in zip(ys, Ws):
        assert_oracle(y.cpu().numpy(), w, q, "no slots")
    q3q4.Linear(device=0, max_tokens=640, max_features=8192, max_k=4096)


# few enough 128 x 128 tiles for split-K where the 64 x 256 ones would be too many for it
@pytest.mark.parametrize("M,N,K", [(330, 2640, 1024), (1100, 832, 768)])
def test_split_k_on_wide_tiles(torch, M, N, K):  # noqa: F811
    lin = q3q4.Linear(device=0, max_tokens=1152, max_features=2688, max_k=1024)
    assert q3q4.load().sera_q4k_mmq_tiles(M, N) <= 64 and q3q4.load().sera_q4k_mmq_schedule(M, N, K) == 0
    W, X = exact_inputs(np.random.default_rng(M + N), M, N, K)
    say(f"case split-K on wide tiles M={M} N={N} K={K} splits={q3q4.mmq_splits(M, N, K)}")
    y = nan_out(torch, M, N)
    lin(q3q4.bind_geometry(12, K, N), dev(torch, W), dev(torch, X), y)
    torch.cuda.synchronize()
    assert_bits(y, expected(W, X, N, K), "boundary")


@pytest.mark.parametrize("M,Ns,K", [(65, [8192, 512, 260], 512), (200, [4096, 1024, 1024, 132], 768),
                                    (129, [3000, 3000], 256), (300, [1024, 1024], 2048)])
def test_group_in_one_launch(torch, M, Ns, K):  # noqa: F811
    """sera_linear_group over 64 tokens: the matrices' wide tiles in one launch
    (the last case: too few tiles, matrix by matrix), each product bit for bit,
    and twice the same output, which must not share a launch."""
    lin = q3q4.Linear(device=0, max_tokens=512, max_features=8192, max_k=2048)
    rng = np.random.default_rng(M + sum(Ns))
    data = [exact_inputs(rng, M, n, K) for n in Ns]
    X = data[0][1]
    Ws = [dev(torch, w) for w, _ in data]
    geos = [q3q4.bind_geometry(12, K, n) for n in Ns]
    say(f"case group M={M} Ns={Ns} K={K}")
    ys = [nan_out(torch, M, n) for n in Ns]
    q3q4.linear_group(geos, Ws, ys, dev(torch, X))
    torch.cuda.synchronize()
    refs = [expected(w, X, n, K) for (w, _), n in zip(data, Ns)]
    for i, (y, ref) in enumerate(zip(ys, refs)):
        assert_bits(y, ref, f"group[{i}]")
    y = torch.zeros((M, Ns[0]), device="cuda")
    q3q4.linear_group([geos[0]] * 2, [Ws[0]] * 2, [y, y], dev(torch, X), flags=q3q4.LIN_ACCUMULATE)
    torch.cuda.synchronize()
    assert np.array_equal(y.cpu().numpy(), (2 * refs[0]).astype(np.float32)), "accumulating twice into one output"
    assert lin.workspace_bytes > 0


# M * N % 4 != 0: no split-K, so the tail schedule runs them, cut along K where that is modelled faster
@pytest.mark.parametrize("M,N,K", [(203, 1333, 1792), (41, 1333, 1024), (19, 3001, 2048), (13, 1001, 2304), (65, 77, 256)])
def test_odd_products_split_by_the_tail(torch, M, N, K):  # noqa: F811
    L = q3q4.load()
    lin = q3q4.Linear(device=0, max_tokens=512, max_features=8192, max_k=2560)
    assert L.sera_q4k_mmq_schedule(M, N, K) == 2
    rng = np.random.default_rng(M + N + K)
    W, X = exact_inputs(rng, M, N, K)
    say(f"case odd product M={M} N={N} K={K} plan {q3q4.mmq_tail_plan(M, N, K)}")
    y = nan_out(torch, M, N)
    lin(q3q4.bind_geometry(12, K, N), dev(torch, W), dev(torch, X), y)
    torch.cuda.synchronize()
    assert_bits(y, expected(W, X, N, K), "odd product")
    # and Q6_K, against the oracle
    W6 = oracle.q6k_weights(rng, N, K)
    lin(q3q4.bind_geometry(14, K, N), dev(torch, W6), dev(torch, X), y)
    torch.cuda.synchronize()
    ref = oracle.linear_reference_q6k(W6, X, N, K)
    assert float(np.max(np.abs(y.cpu().numpy() - ref))) <= 2e-5 * float(np.sqrt(np.mean(ref * ref)))


# RMSNorm on rows of one to five 1024-value pieces, few and many rows (a
# workgroup takes one piece, several or the whole row): the staged quants are
# those of the quantizer on the normalized row
@pytest.mark.parametrize("M,K", [(9, 5120), (300, 5120), (300, 2304), (1030, 1280), (1100, 256), (520, 4864)])
def test_rmsnorm_quantizer_pieces(torch, M, K):  # noqa: F811
    lin = q3q4.Linear(device=0, max_tokens=1152, max_features=256, max_k=5120)
    rng = np.random.default_rng(M + K)
    H = rng.standard_normal((M, K)).astype(np.float32)
    gamma = (1.0 + 0.1 * rng.standard_normal(K)).astype(np.float32)
    rows = np.unique(np.concatenate([[0, M - 1], rng.integers(0, M, 4)]))
    W = oracle.quantize_q4k((rng.standard_normal((64, K)) * 0.02).astype(np.float32))
    y = nan_out(torch, M, 64)
    say(f"case rmsnorm pieces M={M} K={K}")
    q3q4.linear_group([q3q4.bind_geometry(12, K, 64)], [dev(torch, W)], [y], dev(torch, H), gamma=dev(torch, gamma),
                      eps=1e-6, flags=q3q4.LIN_RMSNORM)
    torch.cuda.synchronize()
    xq, xd, xs = oracle.q8_1_mmq(oracle.rmsnorm_fused_order(H[rows], gamma, 1e-6))
    ref = oracle.gemm_mmq(W, xq, xd, xs, 64, K)
    got = y.cpu().numpy()
    assert np.all(np.isfinite(got))
    # same quants, fp32 sums in another order (2e-5 * rms as for the other schedules)
    assert float(np.max(np.abs(got[rows] - ref))) <= 2e-5 * float(np.sqrt(np.mean(ref * ref)))
    lay = q3q4.mmq_stage_layout(M, K)
    arena = lin.workspace[256 << 10:].cpu().numpy()        # the stage starts after the counters
    qs = arena[lay["qs"]:lay["qs"] + M * K].view(np.int8).reshape(M, K)
    assert np.array_equal(qs[rows], xq)


# the Q6_K stage takes the same pieces
@pytest.mark.parametrize("M,K", [(9, 5120), (300, 2304), (1030, 1280), (1100, 256), (520, 4864)])
def test_rmsnorm_q6k_stage_pieces(torch, M, K):  # noqa: F811
    lin = q3q4.Linear(device=0, max_tokens=1152, max_features=256, max_k=5120)
    rng = np.random.default_rng(M * 2 + K)
    H = rng.standard_normal((M, K)).astype(np.float32)
    gamma = (1.0 + 0.1 * rng.standard_normal(K)).astype(np.float32)
    rows = np.unique(np.concatenate([[0, M - 1], rng.integers(0, M, 4)]))
    y = nan_out(torch, M, 64)
    say(f"case rmsnorm Q6_K pieces M={M} K={K}")
    q3q4.linear_group([q3q4.bind_geometry(14, K, 64)], [dev(torch, oracle.q6k_weights(rng, 64, K))], [y], dev(torch, H),
                      gamma=dev(torch, gamma), eps=1e-6, flags=q3q4.LIN_RMSNORM)
    torch.cuda.synchronize()
    assert np.all(np.isfinite(y.cpu().numpy()))
    xq, xd = oracle.q8_1_mmq_d4(oracle.rmsnorm_fused_order(H[rows], gamma, 1e-6))
    lay = q3q4.q6k_mmq_stage_layout(M, K)
    arena = lin.workspace[256 << 10:].cpu().numpy()        # the stage starts after the counters
    xh = arena[lay["qs"]:lay["qs"] + 2 * M * K].view(np.float16).reshape(M, K)
    assert np.array_equal(xh[rows], 16.0 * xq.astype(np.float32))
    d = arena[lay["d"]:lay["d"] + lay["rows"] * K // 32 * 4].view(np.float32).reshape(K // 32, lay["rows"])
    assert np.array_equal(d[:, rows].T, np.asarray(xd).reshape(len(rows), K // 32))


# 64 x 256 tiles in place of the wide ones: whole tiles and all in three pieces, both layouts, plain and
# accumulating, through the boundary and as a group of one
@pytest.mark.parametrize("M,N,K", [(131, 16532, 256), (129, 5392, 2304)])
def test_narrow_tile_where_it_is_faster(torch, M, N, K):  # noqa: F811
    L = q3q4.load()
    lin = q3q4.Linear(device=0, max_tokens=192, max_features=16640, max_k=2304)
    assert L.sera_q4k_mmq_schedule(M, N, K) == 2 and L.sera_q4k_mmq_on_64x256(M, N, K) == 1
    rng = np.random.default_rng(M + N + K)
    W, X = exact_inputs(rng, M, N, K)
    ref = expected(W, X, N, K)
    base = rng.integers(-4, 5, (M, N)).astype(np.float32)
    layouts = [(12, W)] + ([(q3q4.QTYPE_Q4K_TILED, q3q4.q4k_tiled_bytes(W, N, K))] if N % 16 == 0 else [])
    for qt, w in layouts:
        Wd, Xd, g = dev(torch, w), dev(torch, X), q3q4.bind_geometry(qt, K, N)
        say(f"case 64 x 256 tail qt={qt} M={M} N={N} K={K}")
        y = nan_out(torch, M, N)
        lin(g, Wd, Xd, y)
        torch.cuda.synchronize()
        assert_bits(y, ref, "boundary")
        y.copy_(torch.from_numpy(base))
        q3q4.linear_group([g], [Wd], [y], Xd, flags=q3q4.LIN_ACCUMULATE)
        torch.cuda.synchronize()
        assert np.array_equal(y.cpu().numpy(), base + ref.astype(np.float32))
    assert int(lin.workspace[:256 << 10].to(torch.int32).abs().sum()) == 0, "tile counters not reset"


def test_q6k_odd_products_plan(torch):  # noqa: F811
    """Odd Q6_K products are cut along K only where that is modelled (and was
    measured) faster than whole tiles."""
    q3q4.Linear(device=0, max_tokens=512, max_features=32768, max_k=25600)
    for M, N, K, whole in ((13, 22365, 1280, True), (39, 10343, 1280, True), (11, 1241, 2048, False), (31, 313, 25600, False),
                           (203, 1131, 2048, False), (443, 4369, 1536, True)):
        plan = q3q4.q6k_mmq_tail_plan(M, N, K)
        assert (plan is None) == whole, (M, N, K, plan)


# |x| above 8.3e6 overflows the fp16 token scale: the formula's (I * sw) * inf is +-inf, and NaN only where the dot or the
# scale is zero or infinities of both signs meet. M = 193: both token-tile bodies; the last token's second block overflows too.
@pytest.mark.parametrize("dp,pieces", [(10 ** 6, 1), (0, 2)])
def test_wide_tile_token_scale_overflow(torch, dp, pieces):  # noqa: F811
    M, N, K = 193, 4356, 512
    tiles = q3q4.load().sera_q4k_mmq_tiles(M, N)
    rng = np.random.default_rng(5)
    W, X = exact_inputs(rng, M, N, K)
    signs = np.repeat([1.0, -1.0], 16).astype(np.float32)       # a zero sum keeps the min term finite
    for m, b in ((3, 0), (77, 9), (127, 15), (128, 4), (192, 2), (192, 12)):
        X[m, 32 * b:32 * b + 32] = 1e7 * rng.permutation(signs)
    xq, xd, xs = oracle.q8_1_mmq(X)
    ref = oracle.gemm_mmq(W, xq, xd, xs, N, K)
    lost = np.isinf(ref)
    assert lost.sum() > 2 * N and np.isnan(ref).any() and np.isfinite(ref).sum() == (M - 5) * N
    say(f"case wide scale overflow M={M} N={N} K={K} dp_tiles={min(dp, tiles)} pieces={pieces}")
    slots = torch.empty(max(q3q4.mmq_tail_slot_floats(M, N, min(dp, tiles), pieces), 1), dtype=torch.float32, device="cuda")
    counters = torch.zeros(tiles, dtype=torch.int32, device="cuda")
    y = nan_out(torch, M, N)
    q3q4.mmq_tail(dev(torch, W), mmq_stage(torch, X), y, M, N, K, min(dp, tiles), pieces, slots=slots, counters=counters)
    torch.cuda.synchronize()
    assert np.array_equal(y.cpu().numpy().astype(np.float64), ref, equal_nan=True)
