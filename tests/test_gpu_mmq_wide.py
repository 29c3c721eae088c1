"""The 128 x 128 MMQ tile (65 tokens and more on matrices of more than 64
64 x 256 tiles) at the edges of its tiles: a last token tile of at most 64
tokens, ragged rows, one to three K steps, every schedule, the accumulating
and the unaligned store, both weight layouts. Exact inputs: every schedule
must give the dequantized product bit for bit."""
import numpy as np
import pytest

import q3q4
from oracle import oracle
from test_gpu_exact import assert_bits, dev, exact_inputs, expected, mmq_stage, nan_out, say, torch  # noqa: F401

pytestmark = pytest.mark.gpu

# (M, N, K): ragged rows (N % 128, N % 4 != 0: scalar stores) or whole ones
CASES = [(65, 16401, 256), (128, 8452, 512), (129, 5634, 768), (192, 5632, 768), (193, 4353, 256), (321, 3332, 512)]


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
            if s > 1 and M * N % 4:
                continue
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
