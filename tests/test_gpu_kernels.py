"""Each kernel alone against a plain float64 reference, at sizes other than the engine's."""
import math
import random

import pytest
import torch

import plain_qwen2moe as plain

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def rnd(*shape, dtype=torch.float32, scale=1.0, seed=0):
    g = torch.Generator().manual_seed(seed + sum(shape))
    return (torch.randn(*shape, generator=g) * scale).to(dtype).to(DEV)


def close(got, want, dtype, what, k=1):
    """float32: rounding of sums of k products; bfloat16: inputs are exact, the output is rounded once."""
    got, want = got.double().cpu(), want.double().cpu()
    scale = float(want.abs().max()) + 1e-30
    tol = (1e-5 if dtype == torch.float32 else 1e-2) * scale
    err = float((got - want).abs().max())
    assert err <= tol, f"{what}: max error {err:.3e} > {tol:.3e} (scale {scale:.3e})"


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("M,N,K", [(1, 48, 64), (5, 100, 96), (16, 256, 128), (17, 257, 200), (33, 72, 40),
                                    (64, 64, 64), (130, 300, 520), (257, 129, 1032), (3, 50, 100),
                                    (130, 300, 512), (257, 129, 1024), (300, 520, 64), (513, 72, 128), (65, 16, 192),
                                    (40, 65600, 64), (64, 65536, 128), (128, 2048, 2048), (256, 3584, 512), (200, 96, 264),
                                    (256, 4200, 64)])
def test_gemm_plain_and_epilogues(dtype, M, N, K):
    from ferrox_amd import ops
    a, w = rnd(M, K, dtype=dtype), rnd(N, K, dtype=dtype, seed=1)
    bias = rnd(N, dtype=dtype, seed=2)
    ref = a.double() @ w.double().T
    close(ops.gemm(a, w), ref, dtype, "store")
    close(ops.gemm(a, w, bias=bias), ref + bias.double(), dtype, "store+bias")
    close(ops.gemm(a, w, epilogue=ops.EPI_STORE_F32, bias=bias), ref + bias.double(), torch.float32 if dtype == torch.float32 else dtype, "f32 store")
    h = rnd(M, N, seed=3)
    h0 = h.clone()
    scale = rnd(M, seed=4)
    ops.gemm(a, w, epilogue=ops.EPI_RESID, out=h, row_scale=scale)
    close(h, h0.double() + ref * scale.double()[:, None], dtype, "residual")


@pytest.mark.parametrize("N,K", [(16, 16), (61, 37), (100, 70), (130, 96), (96, 2052), (2048, 264)])
def test_float32_products_have_the_same_bits_in_every_kernel(N, K):
    """The kernel for few rows and the tiles of 32 and 64 rows, at their edges (rows, columns, the last step of K, operands
    that are not 16-byte aligned): each close to float64, and the same bits row for row however many rows there are."""
    from ferrox_amd import debug, ops
    M = 130
    a, w, bias = rnd(M, K), rnd(N, K, seed=1), rnd(N, seed=2)
    w2, scale = rnd(2 * N, K, seed=3, scale=0.3), rnd(M, seed=4)
    ref, ref2 = a.double() @ w.double().T, a.double() @ w2.double().T
    whole = ops.gemm(a, w, bias=bias)
    close(whole, ref + bias.double(), torch.float32, "stored")
    gated = ops.gemm(a, w2, epilogue=ops.EPI_GATED)
    close(gated, plain.silu(ref2[:, :N]) * ref2[:, N:], torch.float32, "silu(gate)*up")
    h0 = rnd(M, N, seed=5)
    for tile in (1, 32, 64, 0):
        with debug.kernel_switch("gemm", "f32_tile", tile):
            for rows in (1, 16, 17, 32, 33, 64, 65, M):
                assert torch.equal(ops.gemm(a[:rows], w, bias=bias), whole[:rows]), (tile, rows)
                assert torch.equal(ops.gemm(a[:rows], w2, epilogue=ops.EPI_GATED), gated[:rows]), (tile, rows)
            h = h0.clone()
            ops.gemm(a, w, epilogue=ops.EPI_RESID, out=h, row_scale=scale)
            close(h, h0.double() + ref * scale.double()[:, None], torch.float32, "residual")
    # rows that begin at an odd multiple of four bytes
    wide = rnd(M, K + 3, seed=6)
    wide[:, 1:K + 1] = a
    assert torch.equal(ops.gemm(wide[:, 1:K + 1], w, bias=bias), whole)


@pytest.mark.parametrize("N,K", [(16, 32), (40, 64), (33, 256), (72, 288), (50, 544), (24, 2080)])
def test_float32_few_rows_in_whole_lines(N, K):
    """Rows of whole 32 k: parts of K with one line, several, an odd number and none (the last parts), columns past the end, one and
    two tiles of rows; against float64 and, bit for bit, against tiles of 32."""
    from ferrox_amd import debug, ops
    for rows in (1, 5, 16, 17, 32):
        a, w, w2 = rnd(rows, K), rnd(N, K, seed=1), rnd(2 * N, K, seed=3, scale=0.3)
        got, gated = ops.gemm(a, w), ops.gemm(a, w2, epilogue=ops.EPI_GATED)
        close(got, a.double() @ w.double().T, torch.float32, f"{rows} rows")
        with debug.kernel_switch("gemm", "f32_tile", 32):
            assert torch.equal(got, ops.gemm(a, w)) and torch.equal(gated, ops.gemm(a, w2, epilogue=ops.EPI_GATED)), rows


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("N,K", [(8, 64), (61, 72), (61, 288), (100, 520), (256, 2048), (40, 4168), (2048, 1024),
                                 (24, 2560), (24, 3072), (24, 3584), (24, 4608), (24, 5120), (40, 5632), (24, 6144)])       # (5, 6, 7, 9, 10, 11 and 12 whole pieces a wave: every remainder of four)
def test_half_sets_of_weight_rows_have_the_bits_of_whole_sets(dtype, N, K):
    """Up to 16 rows: blocks of eight weight rows (of each matrix), with two and with four pieces of K on their way, fewer pieces than that, the piece
    that K ends in, columns past the end; every epilogue, rows and slabs of weights; the sums of whole sets bit for bit."""
    from ferrox_amd import debug, ops
    for M in (1, 4, 5, 16):
        a, w, w2 = (rnd(r, K, dtype=dtype, seed=s, scale=0.3) for r, s in ((M, 0), (N, 1), (2 * N, 2)))
        bias, scale, logits, h0 = rnd(N, seed=3), rnd(M, seed=4), rnd(M, N, seed=5), rnd(M, N, seed=6)
        def outputs():
            h = h0.clone()
            ops.gemm(a, w, epilogue=ops.EPI_RESID, out=h, row_scale=scale)
            got = [h, ops.gemm(a, w, bias=bias), ops.gemm(a, w, epilogue=ops.EPI_STORE_F32, out_gate=(logits, 1)),
                   ops.gemm(a, w, store_activation="relu2"), ops.gemm(a, w2, epilogue=ops.EPI_GATED), ops.gemm(a, w2, epilogue=ops.EPI_GATED, activation="gelu_tanh")]
            if K % 64 == 0 and dtype == torch.bfloat16:
                got += [ops.gemm(a, ops.to_kblocked(w), w_kblocked=True), ops.gemm(a, ops.to_kblocked(w2), epilogue=ops.EPI_GATED, w_kblocked=True)]
            return got
        with debug.kernel_switch("gemm", "skinny_half", 0):
            whole = outputs()
        with debug.kernel_switch("gemm", "skinny_half", 1):
            half = outputs()
        for i, (x, y) in enumerate(zip(half, whole)):
            assert torch.equal(x, y), (M, i)
        close(whole[0], h0.double() + (a.double() @ w.double().T) * scale.double()[:, None], dtype, "residual")


@pytest.mark.parametrize("N,K", [(33, 128), (46, 520), (71, 640), (128, 256)])
@pytest.mark.parametrize("waves", [1, 2, 4, 8])
def test_few_rows_store_runs_of_one_two_and_four_columns(waves, N, K):
    """What a thread finishes of a block's outputs depends on the row tiles, sets and waves of a block: runs that begin and end anywhere, rows and columns past the end, outputs in
    whole rows and in a view that begins and steps at odd places; near float64 whatever the block, the bits of one wave count, and nothing written beside."""
    from ferrox_amd import debug, ops
    for M in (1, 15, 17, 33, 50, 64):
        a, w, w2 = (rnd(r, K, dtype=torch.bfloat16, seed=s, scale=0.3) for r, s in ((M, 0), (N, 1), (2 * N, 2)))
        bias, scale, logits, h0 = rnd(N, seed=3), rnd(M, seed=4), rnd(M, N, seed=5), rnd(M, N, seed=6)
        ref, ref2 = a.double() @ w.double().T, a.double() @ w2.double().T
        cases = [(dict(bias=bias), w, ref + bias.double(), torch.bfloat16), (dict(epilogue=ops.EPI_STORE_F32, out_gate=(logits, 1)), w, ref * torch.sigmoid(logits.double()), torch.float32),
                 (dict(epilogue=ops.EPI_RESID, row_scale=scale, bias=bias), w, h0.double() + (ref + bias.double()) * scale.double()[:, None], torch.float32),
                 (dict(epilogue=ops.EPI_GATED), w2, plain.silu(ref2[:, :N]) * ref2[:, N:], torch.bfloat16)]
        got = {}
        for tiles in (1, 2) if waves == 8 else (1, 2, 4):          # (four tiles of two sets take four waves, whose sums are of other parts)
            for sets in (1, 2):
                with debug.kernel_switch("gemm", "skinny_row_tiles", tiles), debug.kernel_switch("gemm", "skinny_sets", sets), \
                        debug.kernel_switch("gemm", "skinny_waves", waves), debug.kernel_switch("gemm", "skinny_half", 0), debug.kernel_switch("gemm", "plain_rows", 64):
                    for i, (kw, weights, want, dtype) in enumerate(cases):
                        odd = torch.full((M, N + 5), 7.0, device=DEV, dtype=dtype)
                        whole = torch.full((M, -(-N // 8) * 8), 7.0, device=DEV, dtype=dtype)
                        for out in (whole[:, :N], odd[:, 3:3 + N]):
                            if kw.get("epilogue") == ops.EPI_RESID:
                                out.copy_(h0)
                            ops.gemm(a, weights, out=out, **kw)
                            close(out, want, torch.bfloat16, f"{M} rows, {tiles} tiles, {sets} sets, case {i}")
                        assert torch.equal(whole[:, :N], odd[:, 3:3 + N]) and torch.equal(whole[:, :N], got.setdefault(i, whole)[:, :N]), (M, tiles, sets, i)
                        assert bool((whole[:, N:] == 7).all()) and bool((odd[:, :3] == 7).all()) and bool((odd[:, 3 + N:] == 7).all()), (M, tiles, sets, i)


@pytest.mark.parametrize("rows", [1, 16, 17, 32, 33, 48, 49, 64, 65, 81])
def test_float32_tiles_leave_out_row_blocks_that_they_do_not_have(rows):
    """Tiles of 64 and of 32 rows with one to four blocks of 16 rows, steps of K odd and even in number and a partial one: the bits of the product
    for few rows, whose blocks are 16 rows each, plain and sorted by expert."""
    from ferrox_amd import debug, ops
    for K in (64, 96, 104):
        a, w, w2 = rnd(3 * rows, K), rnd(3, 70, K, seed=1), rnd(3, 2 * 70, K, seed=2)
        offsets = torch.tensor([0, rows, rows, 3 * rows], dtype=torch.int32, device=DEV)       # shares of `rows`, none and twice as many
        def outputs(tile):
            with debug.kernel_switch("gemm", "f32_tile", tile):
                return [ops.gemm(a[:rows], w[0]), ops.gemm(a[:rows], w2[0], epilogue=ops.EPI_GATED), ops.gemm(a, w, expert_offsets=offsets, n_rows=3 * rows),
                        ops.gemm(a, w2, epilogue=ops.EPI_GATED, expert_offsets=offsets, n_rows=3 * rows)]
        want = outputs(1)
        close(want[0], a[:rows].double() @ w[0].double().T, torch.float32, "plain")
        for tile in (32, 64):
            for x, y in zip(outputs(tile), want):
                assert torch.equal(x, y), (tile, K)


@pytest.mark.parametrize("N,K", [(33, 32), (40, 96), (130, 64), (70, 1056), (200, 2080), (257, 5632)])
def test_float32_products_from_bfloat16_parts(N, K):
    """Every tile and the kernel for few rows, at the edges of row blocks, with an odd and an even number of steps, plain, sorted by expert and from rows that
    begin at odd multiples of four bytes: the same bits row for row, and an error against float64 of at most a float32 sum's (sqrt(K / 32) roundings of a sum, 2^-24 each, a factor of two on top)."""
    from ferrox_amd import debug, ops
    M = 130
    a, w, w2 = rnd(M, K), rnd(N, K, seed=1), rnd(2 * N, K, seed=3, scale=0.3)
    bias, scale, h0 = rnd(N, seed=2), rnd(M, seed=4), rnd(M, N, seed=5)
    ref, ref2 = a.double() @ w.double().T, a.double() @ w2.double().T
    wide = rnd(M, K + 3, seed=6)
    wide[:, 1:K + 1] = a
    we, we2 = torch.stack([rnd(N, K, seed=7), w]), torch.stack([rnd(2 * N, K, seed=8), w2])
    with debug.kernel_switch("gemm", "f32_split", 1):
        whole, gated = ops.gemm(a, w, bias=bias), ops.gemm(a, w2, epilogue=ops.EPI_GATED)
        err = (whole.double() - ref - bias.double()).norm() / ref.norm()
        assert float(err) <= 2 * (K / 32 + 1) ** 0.5 * 2.0 ** -24 + 2.0 ** -24, float(err)
        close(gated, plain.silu(ref2[:, :N]) * ref2[:, N:], torch.float32, "silu(gate)*up")
        for tile in (1, 32, 48, 64, 128, 144, 160, 0):
            with debug.kernel_switch("gemm", "f32_tile", tile):
                for rows in (1, 16, 17, 31, 33, 47, 48, 49, 63, 64, 65, M):
                    assert torch.equal(ops.gemm(a[:rows], w, bias=bias), whole[:rows]), (tile, rows)
                    assert torch.equal(ops.gemm(a[:rows], w2, epilogue=ops.EPI_GATED), gated[:rows]), (tile, rows)
                h = h0.clone()
                ops.gemm(a, w, epilogue=ops.EPI_RESID, out=h, row_scale=scale)
                close(h, h0.double() + ref * scale.double()[:, None], torch.float32, "residual")
                assert torch.equal(ops.gemm(wide[:, 1:K + 1], w, bias=bias), whole), tile
                for first in (1, 40, 66, 0):                  # (shares of 1 to 130 rows: the second expert's are the plain product's)
                    offsets = torch.tensor([0, first, M], dtype=torch.int32, device=DEV)
                    assert torch.equal(ops.gemm(a, we, expert_offsets=offsets, n_rows=M, bias=None, epilogue=ops.EPI_STORE_F32)[first:], ops.gemm(a[first:], w, epilogue=ops.EPI_STORE_F32)), (tile, first)
                    assert torch.equal(ops.gemm(a, we2, epilogue=ops.EPI_GATED, expert_offsets=offsets, n_rows=M)[first:], gated[first:]), (tile, first)


@pytest.mark.parametrize("tile", [1, 32, 48, 128])
def test_float32_parts_leave_what_is_not_finite_to_the_float32_instruction(tile):
    """Infinities, NaN and values that round to infinity as bfloat16: what has one of them in its four columns is what the float32 instruction gives, and everything else is as without them."""
    from ferrox_amd import debug, ops
    M, N, K = 70, 72, 96
    a, w = rnd(M, K), rnd(N, K, seed=1)
    w2 = torch.cat([w, rnd(N, K, seed=2)])
    bad_a, bad_w2 = a.clone(), w2.clone()
    bad_a[3, 5], bad_a[9, 7], bad_a[20, 3], bad_a[66, 95], bad_w2[17, 90], bad_w2[N + 30, 0] = math.inf, math.nan, 3.4e38, -math.inf, -math.inf, math.nan
    for kw, weights in ((dict(epilogue=ops.EPI_STORE_F32), lambda x: x[:N].contiguous()), (dict(epilogue=ops.EPI_GATED), lambda x: x)):
        clean_w, bad_w = weights(w2), weights(bad_w2)
        with debug.kernel_switch("gemm", "f32_tile", tile):
            with debug.kernel_switch("gemm", "f32_split", 1):
                clean, got = ops.gemm(a, clean_w, **kw), ops.gemm(bad_a, bad_w, **kw)
            with debug.kernel_switch("gemm", "f32_split", 0):
                want = ops.gemm(bad_a, bad_w, **kw)
        sums = bad_a @ bad_w[:N].T, bad_a @ bad_w[-N:].T
        odd = ~(torch.isfinite(sums[0]) & torch.isfinite(sums[1])).view(M, N // 4, 4).all(-1, keepdim=True).expand(M, N // 4, 4).reshape(M, N)
        odd[20] = True                                       # (finite as float32 there, not as bfloat16)
        assert torch.equal(torch.isnan(got[odd]), torch.isnan(want[odd])) and torch.equal(torch.nan_to_num(got[odd], nan=7.0), torch.nan_to_num(want[odd], nan=7.0))
        assert torch.equal(got[~odd], clean[~odd]) and bool(odd.any()) and not bool(odd.all())


@pytest.mark.parametrize("tile", [1, 32, 64, 128])
def test_float32_parts_leave_the_smallest_numbers_to_the_float32_instruction(tile):
    """Rows of numbers whose parts are below what bfloat16 holds, weights and activations, and rows of nothing: the float32 instruction's bits, and those of the
    rows beside them as without them."""
    from ferrox_amd import debug, ops
    M, N, K = 70, 72, 96
    a, w = rnd(M, K), torch.cat([rnd(N, K, seed=1), rnd(N, K, seed=2)])
    small_a, small_w = a.clone(), w.clone()
    rows = {3: 2.0 ** -90, 4: 2.0 ** -108, 17: 2.0 ** -114, 20: 2.0 ** -119, 33: 2.0 ** -123, 66: 0.0}
    for m, scale in rows.items():
        small_a[m] *= scale
    for n, scale in {8: 2.0 ** -90, 9: 2.0 ** -112, 10: 2.0 ** -118, 11: 2.0 ** -121}.items():         # (four columns of their own)
        small_w[n] *= scale
        small_w[N + n] *= scale
    for kw, some in ((dict(epilogue=ops.EPI_STORE_F32), lambda x: x[:N].contiguous()), (dict(epilogue=ops.EPI_GATED, activation="relu"), lambda x: x)):
        with debug.kernel_switch("gemm", "f32_tile", tile):
            with debug.kernel_switch("gemm", "f32_split", 1):
                clean, got = ops.gemm(a, some(w), **kw), ops.gemm(small_a, some(small_w), **kw)
            with debug.kernel_switch("gemm", "f32_split", 0):
                want = ops.gemm(small_a, some(small_w), **kw)
        odd = torch.zeros(M, N, dtype=torch.bool, device=DEV)
        odd[list(rows)] = True
        odd[:, 8:12] = True
        assert torch.equal(got[odd], want[odd]) and torch.equal(got[~odd], clean[~odd]), kw
        assert bool((got[66] == 0).all())


@pytest.mark.parametrize("T,E,k,I,H", [(1, 5, 2, 20, 36), (3, 60, 4, 96, 128), (90, 7, 3, 33, 50), (700, 4, 2, 64, 96)])
def test_float32_grouped_products_have_the_same_bits_in_every_kernel(T, E, k, I, H):
    from ferrox_amd import debug, ops
    x, w = rnd(T, H), rnd(E, 2 * I, H, seed=1, scale=0.3)
    g = torch.Generator().manual_seed(7)
    ids = torch.stack([torch.randperm(E, generator=g)[:k] for _ in range(T)]).to(torch.int32).to(DEV)
    offsets, sorted_token, sorted_pair, inv = ops.moe_align(ids, E)
    got = {}
    for tile in (0, 1, 32, 64):
        with debug.kernel_switch("gemm", "f32_tile", tile):
            got[tile] = ops.gemm(x, w, epilogue=ops.EPI_GATED, a_rows=sorted_token, expert_offsets=offsets, n_rows=T * k)
        assert torch.equal(got[tile], got[0]), tile
    xs, off = x.double()[sorted_token.long()], offsets.cpu().tolist()
    for e in range(E):
        r = slice(off[e], off[e + 1])
        if r.start == r.stop:
            continue
        close(got[0][r], plain.silu(xs[r] @ w[e, :I].double().T) * (xs[r] @ w[e, I:].double().T), torch.float32, f"expert {e}")


@pytest.mark.parametrize("T,H,N,k,S", [(1, 2048, 6144, 4, 4), (8, 2048, 6144, 4, 4), (16, 264, 100, 3, 0), (5, 520, 72, 1, 2)])
def test_combine_that_leaves_the_scale_to_the_product(T, H, N, k, S):
    """combine -> rows times the norm's weight and sums of squares -> product that scales its rows,
    against combine -> norm kernel -> product and against the plain formulas"""
    from ferrox_amd import ops
    h = rnd(T, H, scale=2.0)
    y, wts = rnd(T * k, H, seed=1), torch.rand(T, k, generator=torch.Generator().manual_seed(2)).to(DEV)
    shared = rnd(S, T, H, seed=3) if S else None
    gate = torch.rand(T, generator=torch.Generator().manual_seed(4)).to(DEV) if S else None
    gamma = (1.0 + rnd(H, seed=5, scale=0.2)).to(torch.bfloat16)
    w, bias = rnd(N, H, dtype=torch.bfloat16, seed=6, scale=0.05), rnd(N, dtype=torch.bfloat16, seed=7)
    h1, h2 = h.clone(), h.clone()
    ops.moe_combine(h1, y, None, wts, k, shared=shared, gate=gate)
    two = ops.gemm(ops.rmsnorm(h1, gamma, 1e-6, torch.bfloat16), w, bias=bias)
    later = ops.moe_combine(h2, y, None, wts, k, shared=shared, gate=gate, scale_later=(gamma, 1e-6, torch.bfloat16))
    assert isinstance(later, ops.ScaleLater) and torch.equal(h1, h2)
    close(later.ss.sum(1), (h1.double() ** 2).sum(1), torch.float32, "sums of squares")
    got = ops.gemm(later.x, w, bias=bias, row_ss=(later.ss, later.eps))
    want = plain.rms_norm(h1.double().cpu(), gamma.double().cpu(), 1e-6) @ w.double().cpu().T + bias.double().cpu()
    close(got, want, torch.bfloat16, "product with the scale applied afterwards")
    close(two, want, torch.bfloat16, "norm, then product")


@pytest.mark.parametrize("T,H,k,S,sorted_rows", [(130, 2048, 4, 4, False), (300, 1000, 3, 0, True), (140, 2052, 2, 1, True)])
def test_combine_of_many_rows_equals_that_of_few(T, H, k, S, sorted_rows):
    """Many rows go four columns to a thread, few rows one: the same bits in the residual stream and in the rows
    for the next norm, the same sums of squares up to the order of their terms."""
    from ferrox_amd import ops
    assert T * H >= 1 << 18 and (T // 2 + 1) * H < 1 << 18
    h = rnd(T, H, scale=2.0)
    y, wts = rnd(T * k, H, seed=1), torch.rand(T, k, generator=torch.Generator().manual_seed(2)).to(DEV)
    inv = torch.randperm(T * k, generator=torch.Generator().manual_seed(3)).to(torch.int32).to(DEV) if sorted_rows else None
    shared = rnd(S, T, H, seed=3) if S else None
    gate = torch.rand(T, generator=torch.Generator().manual_seed(4)).to(DEV) if S else None
    gamma = (1.0 + rnd(H, seed=5, scale=0.2)).to(torch.bfloat16)
    h_all = h.clone()
    all_rows = ops.moe_combine(h_all, y, inv, wts, k, shared=shared, gate=gate, scale_later=(gamma, 1e-6, torch.bfloat16))
    cut = T // 2
    for lo, hi in ((0, cut), (cut, T)):
        h_part = h[lo:hi].clone()
        part = ops.moe_combine(h_part, y if inv is not None else y[lo * k:hi * k], inv[lo * k:hi * k] if inv is not None else None,
                               wts[lo:hi].contiguous(), k, shared=shared[:, lo:hi].contiguous() if S else None,
                               gate=gate[lo:hi].contiguous() if S else None, scale_later=(gamma, 1e-6, torch.bfloat16))
        assert torch.equal(h_all[lo:hi], h_part), "residual stream"
        assert torch.equal(all_rows.x[lo:hi], part.x), "rows for the next norm"
        close(all_rows.ss[lo:hi], part.ss, torch.float32, "sums of squares per 256 columns")
    want = h.double().cpu() + (wts.double().cpu()[:, :, None] * (y.double().cpu()[inv.long().cpu()] if inv is not None else y.double().cpu()).view(T, k, H)).sum(1)
    if S:
        want = want + gate.double().cpu()[:, None] * shared.double().cpu().sum(0)
    close(h_all, want, torch.float32, "combined rows")


# 12, 4: tiles of 192 and of 64 rows x 256 weight rows; 464, 4128: 64 x 64 and 64 x 128; 8128: 128 x 128 in two stages
@pytest.mark.parametrize("tile", [256, 192, 128, 64, 12, 4, 464, 4128, 8128])
@pytest.mark.parametrize("M,N,K", [(300, 400, 192), (513, 200, 64), (70, 520, 448)])
def test_gemm_every_wide_tile(tile, M, N, K):
    """The many-row kernel picks its tile by the sizes; here each tile shape is made to run the same products."""
    from ferrox_amd import debug, ops
    dtype = torch.bfloat16
    a, w, bias = rnd(M, K, dtype=dtype), rnd(N, K, dtype=dtype, seed=1), rnd(N, dtype=dtype, seed=2)
    ref = a.double() @ w.double().T
    h = rnd(M, N, seed=3)
    h0 = h.clone()
    with debug.kernel_switch("gemm", "wide", tile):
        got = ops.gemm(a, w, bias=bias)
        ops.gemm(a, w, epilogue=ops.EPI_RESID, out=h)
        w2 = rnd(2 * N, K, dtype=dtype, seed=4, scale=0.5)
        act = ops.gemm(a, w2, epilogue=ops.EPI_GATED)
    close(got, ref + bias.double(), dtype, "store+bias")
    close(h, h0.double() + ref, dtype, "residual")
    close(act, plain.silu(a.double() @ w2[:N].double().T) * (a.double() @ w2[N:].double().T), dtype, "silu(gate)*up")


@pytest.mark.parametrize("tile", [256, 192, 128, 64, 12, 4, 464, 4128, 8128, 8256, 1128, 6128, 6256])
@pytest.mark.parametrize("M,N", [(130, 264), (97, 200), (33, 71), (17, 132), (300, 46)])
def test_wide_tiles_store_the_same_at_any_columns_and_alignment(tile, M, N):
    """A lane stores eight columns (four of float32) at once where they exist and C allows it: every epilogue into rows of whole 16 bytes
    and into a view that begins and steps at odd places, the same bits, and nothing written beside them."""
    from ferrox_amd import debug, ops
    a, w, bias = rnd(M, 128, dtype=torch.bfloat16), rnd(N, 128, dtype=torch.bfloat16, seed=1), rnd(N, seed=2)
    w2, scale, logits = rnd(2 * N, 128, dtype=torch.bfloat16, seed=3, scale=0.1), rnd(M, seed=4), rnd(M, N, seed=5)
    ref, ref2, h0 = a.double() @ w.double().T, a.double() @ w2.double().T, rnd(M, N, seed=6)
    cases = [(dict(epilogue=ops.EPI_STORE, bias=bias), w, ref + bias.double(), torch.bfloat16),
             (dict(epilogue=ops.EPI_STORE_F32, out_gate=(logits, 1)), w, ref * torch.sigmoid(logits.double()), torch.float32),
             (dict(epilogue=ops.EPI_RESID, row_scale=scale), w, h0.double() + ref * scale.double()[:, None], torch.float32)]
    if tile not in (192, 464):
        cases.append((dict(epilogue=ops.EPI_GATED), w2, plain.silu(ref2[:, :N]) * ref2[:, N:], torch.bfloat16))
    with debug.kernel_switch("gemm", "wide", tile), debug.kernel_switch("gemm", "plain_rows", 1):
        for kw, weights, want, dtype in cases:
            whole = torch.zeros(M, -(-N // 8) * 8, device=DEV, dtype=dtype)
            odd = torch.full((M, N + 5), 7.0, device=DEV, dtype=dtype)
            for out in (whole[:, :N], odd[:, 3:3 + N]):
                if kw["epilogue"] == ops.EPI_RESID:
                    out.copy_(h0)
                ops.gemm(a, weights, out=out, **kw)
                close(out, want, torch.bfloat16, f"{kw['epilogue']}")
            assert torch.equal(whole[:, :N], odd[:, 3:3 + N]), kw["epilogue"]
            assert bool((whole[:, N:] == 0).all()) and bool((odd[:, :3] == 7).all()) and bool((odd[:, 3 + N:] == 7).all()), kw["epilogue"]


def test_tiled_silu_at_the_ends_of_its_range():
    """Gates that reach the activation exactly (one product of each sum is not zero), on both sides of where the quotient is scaled, and
    beyond what the exponential holds: what 32-bit division gives, rounded to bfloat16.  Operands that are no finite numbers stay in their rows (an
    infinite gate beside a finite up is `test_a_gate_that_overflows_stays_infinite`)."""
    from ferrox_amd import debug, ops
    x = torch.tensor([0.0, -0.0, 1e-3, -1e-3, 1.0, -1.0, 20.0, -20.0, 79.5, -79.5, 80.0, -80.0, 80.5, -80.5, 87.0, -87.0, -88.5, 89.0, -103.0, 1e4, -1e4,
                      3e38, -3e38, math.inf, math.nan] * 8, dtype=torch.bfloat16, device=DEV)[:, None]
    a = torch.zeros(len(x), 64, dtype=torch.bfloat16, device=DEV)
    a[:, :1], a[:, 1] = torch.nan_to_num(x, nan=0.0, posinf=0.0), 1.0
    w = torch.zeros(32, 64, dtype=torch.bfloat16, device=DEV)
    w[:16, 0], w[16:, 1] = 1.0, 1.0
    f = a[:, :1].float()
    want = (f / (1.0 + torch.exp(-f))).to(torch.bfloat16).expand(-1, 16)
    with debug.kernel_switch("gemm", "wide", 8128):
        assert torch.equal(ops.gemm(a, w, epilogue=ops.EPI_GATED), want)
        a[:, :1] = x                                    # (0 * inf in the up column: NaN, whatever the gate becomes)
        got = ops.gemm(a, w, epilogue=ops.EPI_GATED)
    finite = torch.isfinite(x[:, 0])
    assert torch.equal(got[finite], want[finite]) and bool(torch.isnan(got[~finite]).all())


@pytest.mark.parametrize("tile", [256, 128, 64, 12, 4, 4128, 8128, 8256, 1128, 6128, 6256])
@pytest.mark.parametrize("N", [48, 200, 61])
def test_a_gate_that_overflows_stays_infinite(tile, N):
    """Two finite numbers whose product float32 does not hold, in the gates of every third column and the first row of every four, negative ones in
    the second: an infinite gate times up is infinite with the sign of up (and NaN for minus infinity, whose quotient is inf / inf), in every tile as in
    the kernel for few rows; the columns and rows beside it stay what they are."""
    from ferrox_amd import debug, ops
    a = torch.zeros(40, 64, dtype=torch.bfloat16)
    a[:, 0] = torch.tensor([3e38, -3e38, 1e38, 0.0]).repeat(10)
    a[:, 1] = torch.tensor([1.0, -1.0, 0.5, -2.0, 1.5]).repeat(8)
    w = torch.zeros(2 * N, 64, dtype=torch.bfloat16)
    w[:N, 0] = torch.tensor([2.0, 2.0 ** -125, 2.0 ** -126])[torch.arange(N) % 3]
    w[N:, 1] = torch.tensor([1.0, -1.0])[torch.arange(N) % 2]
    gate = a[:, :1].float() * w[:N, 0].float()          # (one product of each sum is not zero)
    up = a[:, 1:2].float() * w[N:, 1].float()
    want = (gate / (1.0 + torch.exp(-gate)) * up).to(torch.bfloat16)
    assert bool((want == math.inf).any()) and bool((want == -math.inf).any()) and bool(torch.isnan(want).any())
    a, w, want = a.to(DEV), w.to(DEV), want.to(DEV)
    few = ops.gemm(a[:16], w, epilogue=ops.EPI_GATED)
    with debug.kernel_switch("gemm", "wide", tile), debug.kernel_switch("gemm", "plain_rows", 1):
        got = ops.gemm(a, w, epilogue=ops.EPI_GATED)
    assert torch.equal(torch.isnan(got), torch.isnan(want)) and torch.equal(torch.nan_to_num(got, nan=0.0, posinf=1e38, neginf=-1e38)[:16],
                                                                            torch.nan_to_num(few, nan=0.0, posinf=1e38, neginf=-1e38))
    infinite = torch.isinf(want)
    assert torch.equal(got[infinite], want[infinite])
    finite = torch.isfinite(want)
    assert torch.allclose(got[finite].float(), want[finite].float(), rtol=2.0 ** -7, atol=1e-30)      # (a rounding to bfloat16 either way)


@pytest.mark.parametrize("M,N", [(33, 4096), (64, 8200), (129, 64), (257, 1000), (513, 2048), (700, 3000)])
def test_plain_products_have_the_same_bits_in_every_tile(M, N):
    """The tile that the sizes choose (64 x 64 to 256 x 256, edges inside tiles) against one that is forced: every tile adds an
    element's products in ascending order."""
    from ferrox_amd import debug, ops
    K, dtype = 192, torch.bfloat16
    a, w, bias = rnd(M, K, dtype=dtype), rnd(N, K, dtype=dtype, seed=1), rnd(N, dtype=dtype, seed=2)
    chosen = ops.gemm(a, w, bias=bias)
    close(chosen, a.double() @ w.double().T + bias.double(), dtype, "chosen tile")
    with debug.kernel_switch("gemm", "plain_rows", 32):      # (no product for few rows beyond 32 rows)
        gated = ops.gemm(a, w[:N // 2 * 2], epilogue=ops.EPI_GATED)
        chosen = ops.gemm(a, w, bias=bias)
        for tile in (464, 4128, 8128, 64, 256):
            with debug.kernel_switch("gemm", "wide", tile):
                assert torch.equal(ops.gemm(a, w, bias=bias), chosen), tile
                assert torch.equal(ops.gemm(a, w[:N // 2 * 2], epilogue=ops.EPI_GATED), gated), tile


@pytest.mark.parametrize("K", [64, 128, 192, 256, 320, 384, 576])      # steps of 64 k: fewer than stages, as many, one and more beyond
@pytest.mark.parametrize("M,N", [(129, 264), (500, 392)])
def test_tiles_in_quarters_have_the_bits_of_the_ring(M, N, K):
    """Every shape of tile that is worked on in quarters, rows and columns that end inside a tile, every epilogue."""
    from ferrox_amd import debug, ops
    dtype = torch.bfloat16
    a, w, bias, w2 = rnd(M, K + 8, dtype=dtype)[:, :K], rnd(N, K, dtype=dtype, seed=1), rnd(N, dtype=dtype, seed=2), rnd(2 * N, K, dtype=dtype, seed=4, scale=0.5)
    h, scale, blocked = rnd(M, N, seed=3), rnd(M, seed=5).abs(), ops.to_kblocked(w)

    def products():
        return (ops.gemm(a, w, bias=bias), ops.gemm(a, w, epilogue=ops.EPI_STORE_F32), ops.gemm(a, w, epilogue=ops.EPI_RESID, out=h.clone(), row_scale=scale),
                ops.gemm(a, w2, epilogue=ops.EPI_GATED))

    with debug.kernel_switch("gemm", "wide", 4):          # 64 x 256, whose stages go round in a ring
        want = products()
    close(want[1], a.double() @ w.double().T, dtype, "product")
    for tile in (256, 192, 128, 12, 8256, 8128, 6256, 6128):
        with debug.kernel_switch("gemm", "wide", tile):
            for x, y, what in zip(products(), want, ("store + bias", "store float32", "residual", "gated")):
                assert torch.equal(x, y), (tile, what)
            assert torch.equal(ops.gemm(a, blocked, epilogue=ops.EPI_STORE_F32, w_kblocked=True), want[1]), (tile, "slabs")


@pytest.mark.parametrize("blocked", [False, True])
def test_grouped_tiles_in_quarters_at_every_number_of_row_blocks(blocked):
    """Experts with 1 to 260 rows, so that tiles have every number of blocks of 16 rows, none included."""
    from ferrox_amd import debug, ops
    dtype, K, N = torch.bfloat16, 192, 136
    sizes = [0, 1, 16, 17, 33, 64, 65, 96, 0, 97, 128, 129, 160, 161, 192, 193, 224, 225, 256, 260, 0]
    E, n = len(sizes), sum(sizes)
    offsets = torch.tensor([sum(sizes[:i]) for i in range(E + 1)], dtype=torch.int32, device=DEV)
    g = torch.Generator().manual_seed(3)
    x, w, w2 = rnd(300, K, dtype=dtype), rnd(E, N, K, dtype=dtype, seed=1), rnd(E, 2 * N, K, dtype=dtype, seed=2, scale=0.5)
    rows = torch.randint(0, 300, (n,), generator=g).to(torch.int32).to(DEV)
    to = torch.randperm(n, generator=g).to(torch.int32).to(DEV)
    kb = dict(w_kblocked=True) if blocked else {}
    wb, w2b = (ops.to_kblocked(w), ops.to_kblocked(w2)) if blocked else (w, w2)
    want = torch.zeros(n, N, dtype=torch.float64, device=DEV)
    xs = x.double()[rows.long()]
    for e in range(E):
        r = slice(sum(sizes[:e]), sum(sizes[:e + 1]))
        want[to[r].long()] = xs[r] @ w[e].double().T
    first = None
    for tile in (4, 256, 192, 128, 12, 8256, 8128):       # (4: the ring)
        with debug.kernel_switch("gemm", "wide_grouped", tile), debug.kernel_switch("gemm", "stream_w", 0):
            got = ops.gemm(x, wb, epilogue=ops.EPI_STORE_F32, a_rows=rows, c_rows=to, expert_offsets=offsets, n_rows=n, **kb)
            act = ops.gemm(x, w2b, epilogue=ops.EPI_GATED, a_rows=rows, expert_offsets=offsets, n_rows=n, **kb)
        first = first or (got, act)
        close(got, want, dtype, f"tile {tile}")
        assert torch.equal(got, first[0]) and torch.equal(act, first[1]), tile


@pytest.mark.parametrize("K", [16320, 16384, 20480])        # both sides of the line
def test_long_sums_have_the_bits_of_the_tiles_in_quarters(K):
    from ferrox_amd import debug, ops
    M, N = 1025, 2056
    a, w = rnd(M, K, dtype=torch.bfloat16), rnd(N, K, dtype=torch.bfloat16, seed=1, scale=0.05)
    got = ops.gemm(a, w, epilogue=ops.EPI_STORE_F32)
    close(got, a.double() @ w.double().T, torch.bfloat16, "product")
    for tile in (1128, 64, 6128):
        with debug.kernel_switch("gemm", "wide", tile):
            assert torch.equal(ops.gemm(a, w, epilogue=ops.EPI_STORE_F32), got), tile


def grouped_products(sizes, N, K, seed):
    """Rows sorted by expert with shares `sizes`: a stored product to scattered rows, in float64 too, and a gated one, as a call."""
    from ferrox_amd import ops
    E, n, dtype = len(sizes), sum(sizes), torch.bfloat16
    offsets = torch.tensor([sum(sizes[:i]) for i in range(E + 1)], dtype=torch.int32, device=DEV)
    g = torch.Generator().manual_seed(seed)
    x, w, w2 = rnd(300, K, dtype=dtype, seed=seed), rnd(E, N, K, dtype=dtype, seed=seed + 1), rnd(E, 2 * N, K, dtype=dtype, seed=seed + 2, scale=0.5)
    rows, to = torch.randint(0, 300, (n,), generator=g).to(torch.int32).to(DEV), torch.randperm(n, generator=g).to(torch.int32).to(DEV)
    want, xs = torch.zeros(n, N, dtype=torch.float64, device=DEV), x.double()[rows.long()]
    for e in range(E):
        r = slice(sum(sizes[:e]), sum(sizes[:e + 1]))
        want[to[r].long()] = xs[r] @ w[e].double().T
    wb, w2b = ops.to_kblocked(w), ops.to_kblocked(w2)
    kb = dict(expert_offsets=offsets, n_rows=n, w_kblocked=True)
    return want, lambda most=0: (ops.gemm(x, wb, epilogue=ops.EPI_STORE_F32, a_rows=rows, c_rows=to, max_share=most, **kb),
                                 ops.gemm(x, w2b, epilogue=ops.EPI_GATED, a_rows=rows, max_share=most, **kb))


@pytest.mark.parametrize("most", [64, 65, 128, 129, 300])       # up to a tile of 64 and of 128 rows, one more, and beyond tiles of 256
@pytest.mark.parametrize("E", [40, 72, 130])                    # tiles are found 64 experts at a time: one, two and three times
def test_grouped_tiles_at_any_number_of_experts(E, most):
    """Blocks find their tile among shares of 0 to `most` rows, the largest one in the first, a middle and the last expert, whether an XCD takes every
    eighth row tile or an eighth of the tiles (the largest share known, too small a number and unknown); with the hint on the weights that the shares call for and without."""
    from ferrox_amd import debug
    g = torch.Generator().manual_seed(E + most)
    sizes = [int(s) for s in torch.randint(0, 24, (E,), generator=g)]
    sizes[0] = sizes[E // 2 + 1] = sizes[E - 1] = most
    sizes[1] = sizes[E // 2] = sizes[E - 3] = 0
    want, products = grouped_products(sizes, 136, 192, E)
    with debug.kernel_switch("gemm", "wide_grouped", 256), debug.kernel_switch("gemm", "stream_w", 0):
        first = products()
    close(first[0], want, torch.bfloat16, "256 x 256")
    for tile in (4, 12, 64, 8128, 8256, 1256):
        for hint in (-1, 0):
            for known in (0, 1, most):
                with debug.kernel_switch("gemm", "wide_grouped", tile), debug.kernel_switch("gemm", "stream_w", hint):
                    got = products(known)
                assert torch.equal(got[0], first[0]) and torch.equal(got[1], first[1]), (tile, hint, known)


@pytest.mark.parametrize("average", [4, 5, 20, 21, 36, 37, 104, 105, 128, 129])
@pytest.mark.parametrize("crowded", [False, True])
def test_sorted_rows_as_the_sizes_choose(average, crowded):
    """Both sides of every average share where the tiles change: even shares, and one expert with most of the rows."""
    from ferrox_amd import debug
    sizes = [average + d for d in (0, 3, -3, 2, -2, 1, -1, 0)]
    if crowded:
        sizes = [1, 0, average, 8 * average - 3 - 3 * (average // 2) - average, 2, average // 2, average // 2, average // 2]
    assert sum(sizes) == 8 * average
    want, products = grouped_products(sizes, 264, 320, average)
    got = products()
    close(got[0], want, torch.bfloat16, "chosen")
    with debug.kernel_switch("gemm", "wide_grouped", 256), debug.kernel_switch("gemm", "stream_w", 0):
        other = products()
    assert torch.equal(got[0], other[0]) and torch.equal(got[1], other[1])


@pytest.mark.parametrize("T,E", [(2048, 65), (4096, 65), (4096, 128), (8065, 65)])
def test_a_routers_logits_keep_their_order_of_sums(T, E):
    """Up to 524,288 logits come from the product for few rows, whose bits decide between experts that stand close."""
    from ferrox_amd import debug, ops
    a, w = rnd(T, 1024, dtype=torch.bfloat16), rnd(E, 1024, dtype=torch.bfloat16, seed=1)
    got = ops.gemm(a, w, epilogue=ops.EPI_STORE_F32)
    with debug.kernel_switch("gemm", "plain_rows", T):
        assert torch.equal(got, ops.gemm(a, w, epilogue=ops.EPI_STORE_F32))
    close(got, a.double() @ w.double().T, torch.bfloat16, "logits")


@pytest.mark.parametrize("tile", [12, 256, 4])
def test_grouped_gemm_tiles_agree(tile):
    """An expert's rows in tiles of 192 (weights three steps deep), of 256 and of 64 (weights four steps deep) give
    the same sums."""
    from ferrox_amd import debug, ops
    T, E, k, I, H = 900, 6, 2, 64, 256
    x = rnd(T, H, dtype=torch.bfloat16)
    w_gu = rnd(E, 2 * I, H, dtype=torch.bfloat16, seed=1, scale=0.3)
    g = torch.Generator().manual_seed(7)
    # uneven shares: expert 0 gets a third of all pairs, more than one tile of either kind
    first = torch.where(torch.rand(T, generator=g) < 0.66, 0, 1)
    ids = torch.stack([first, 2 + torch.randint(0, E - 2, (T,), generator=g)], dim=1).to(torch.int32).to(DEV)
    offsets, sorted_token, sorted_pair, inv = ops.moe_align(ids, E)
    with debug.kernel_switch("gemm", "wide", tile):
        act = ops.gemm(x, w_gu, epilogue=ops.EPI_GATED, a_rows=sorted_token, expert_offsets=offsets, n_rows=T * k)
    xs = x.double()[sorted_token.long()]
    off = offsets.cpu().tolist()
    assert off[1] - off[0] > 256
    for e in range(E):
        r = slice(off[e], off[e + 1])
        want = plain.silu(xs[r] @ w_gu[e, :I].double().T) * (xs[r] @ w_gu[e, I:].double().T)
        close(act[r], want, torch.bfloat16, f"expert {e}")


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("M,I,K", [(1, 32, 64), (7, 48, 96), (40, 100, 72), (200, 176, 256), (300, 100, 128),
                                    (257, 129, 64)])
def test_gemm_gate_up(dtype, M, I, K):
    from ferrox_amd import ops
    a, w = rnd(M, K, dtype=dtype), rnd(2 * I, K, dtype=dtype, seed=1, scale=0.5)
    g, u = a.double() @ w[:I].double().T, a.double() @ w[I:].double().T
    close(ops.gemm(a, w, epilogue=ops.EPI_GATED), plain.silu(g) * u, dtype, "silu(gate)*up")
    # the gate's activation is a parameter of the call: every kernel that has the epilogue takes every activation
    others = {"gelu_tanh": lambda z: 0.5 * z * (1.0 + torch.tanh(math.sqrt(2.0 / math.pi) * (z + 0.044715 * z ** 3))),
              "gelu": lambda z: 0.5 * z * (1.0 + torch.erf(z / math.sqrt(2.0))), "relu": lambda z: z.clamp(min=0.0),
              "silu": plain.silu}
    assert set(others) | {"swiglu_clamped"} == set(ops.ACTIVATIONS)
    for name, f in others.items():
        close(ops.gemm(a, w, epilogue=ops.EPI_GATED, activation=name), f(g) * u, dtype, f"{name}(gate)*up")
    # the clamped gate bounds both factors, and a scale in front of the activation stands for a scaled row of `a`
    limit, slope = 0.8, 1.702
    scale = torch.rand(M, generator=torch.Generator().manual_seed(3)).to(DEV) + 0.5
    gs, us = g * scale.double()[:, None], u * scale.double()[:, None]
    gc, uc = gs.clamp(max=limit), us.clamp(-limit, limit)
    close(ops.gemm(a, w, epilogue=ops.EPI_GATED, activation="swiglu_clamped", activation_params=(limit, slope), pre_scale=scale),
          gc * torch.sigmoid(slope * gc) * (uc + 1.0), dtype, "clamped gate behind a row scale")
    with pytest.raises(ops.KernelError, match="activation"):
        ops.gemm(a, w, epilogue=ops.EPI_GATED, activation="swish2")


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("T,E,k,I,H", [(1, 4, 2, 32, 64), (9, 6, 3, 48, 96), (70, 5, 1, 40, 120), (300, 8, 2, 64, 128),
                                        (64, 3, 2, 24, 72), (520, 4, 3, 128, 256), (700, 3, 2, 200, 192),
                                        (330, 4, 2, 128, 320), (1300, 16, 2, 64, 192)])
def test_grouped_gemm_and_routing_buffers(dtype, T, E, k, I, H):
    """router ids -> align -> grouped gate/up -> grouped down -> combine, against per-token loops."""
    from ferrox_amd import ops
    x = rnd(T, H, dtype=dtype)
    w_gu, w_dn = rnd(E, 2 * I, H, dtype=dtype, seed=1, scale=0.3), rnd(E, H, I, dtype=dtype, seed=2, scale=0.3)
    g = torch.Generator().manual_seed(5)
    ids = torch.stack([torch.randperm(E, generator=g)[:k] for _ in range(T)]).to(torch.int32).to(DEV)
    wts = torch.rand(T, k, generator=g).to(DEV)
    offsets, sorted_token, sorted_pair, inv = ops.moe_align(ids, E)
    # the sort: offsets are the counts' prefix sums; every pair sits in its expert's range; order is stable
    counts = torch.bincount(ids.flatten().long().cpu(), minlength=E)
    assert offsets.cpu().tolist() == [0] + torch.cumsum(counts, 0).tolist()
    inv_c, st_c, ids_c = inv.cpu(), sorted_token.cpu(), ids.cpu()
    assert sorted(inv_c.tolist()) == list(range(T * k))
    for i in range(T * k):
        e = int(ids_c.flatten()[i])
        assert offsets[e] <= inv_c[i] < offsets[e + 1] and st_c[inv_c[i]] == i // k and sorted_pair[inv_c[i]] == i
    for e in range(E):
        seg = [i for i in range(T * k) if int(ids_c.flatten()[i]) == e]
        assert [int(inv_c[i]) for i in seg] == list(range(int(offsets[e]), int(offsets[e + 1])))
    act = ops.gemm(x, w_gu, epilogue=ops.EPI_GATED, a_rows=sorted_token, expert_offsets=offsets, n_rows=T * k)
    y = ops.gemm(act, w_dn, epilogue=ops.EPI_STORE_F32, expert_offsets=offsets)
    h = torch.zeros(T, H, device=DEV)
    ops.moe_combine(h, y, inv, wts, k)
    # the same with the second product scattering its rows back into pair order
    y2 = ops.gemm(act, w_dn, epilogue=ops.EPI_STORE_F32, expert_offsets=offsets, c_rows=sorted_pair)
    h2 = torch.zeros(T, H, device=DEV)
    ops.moe_combine(h2, y2, None, wts, k)
    assert torch.equal(h, h2)
    ref = torch.zeros(T, H, dtype=torch.float64)
    xd, gud, dnd = x.double().cpu(), w_gu.double().cpu(), w_dn.double().cpu()
    for t in range(T):
        for j in range(k):
            e = int(ids_c[t, j])
            a = plain.silu(xd[t] @ gud[e, :I].T) * (xd[t] @ gud[e, I:].T)
            if dtype == torch.bfloat16:
                a = a.to(torch.bfloat16).double()       # the engine stores the activation in bfloat16
            ref[t] += float(wts[t, j]) * (a @ dnd[e].T)
    close(h, ref, dtype, "moe")


@pytest.mark.parametrize("T,E,k,I,H", [(1, 4, 2, 32, 64), (8, 60, 4, 1408, 2048), (16, 60, 4, 176, 256), (16, 5, 4, 48, 96),
                                        (3, 700, 8, 64, 128), (7, 1, 1, 40, 72)])
def test_grouped_gemm_from_unsorted_pairs(T, E, k, I, H):
    """few rows: the products group the (token, slot) pairs by expert themselves; same numbers as
    the sorted layout gives, row for row"""
    from ferrox_amd import ops
    dtype = torch.bfloat16
    x = rnd(T, H, dtype=dtype)
    w_gu, w_dn = rnd(E, 2 * I, H, dtype=dtype, seed=1, scale=0.3), rnd(E, H, I, dtype=dtype, seed=2, scale=0.3)
    g = torch.Generator().manual_seed(11)
    ids = torch.stack([torch.randperm(E, generator=g)[:k] for _ in range(T)]).to(torch.int32).to(DEV)
    if T >= 8 and E >= 8:
        ids[:, 0] = 5            # one expert with a row of every token
    offsets, sorted_token, sorted_pair, inv = ops.moe_align(ids, E)
    act_s = ops.gemm(x, w_gu, epilogue=ops.EPI_GATED, a_rows=sorted_token, expert_offsets=offsets, n_rows=T * k)
    y_s = ops.gemm(act_s, w_dn, epilogue=ops.EPI_STORE_F32, expert_offsets=offsets, c_rows=sorted_pair)
    act_p = ops.gemm(x, w_gu, epilogue=ops.EPI_GATED, pair_ids=ids, pair_div=k)
    y_p = ops.gemm(act_p, w_dn, epilogue=ops.EPI_STORE_F32, pair_ids=ids)
    assert torch.equal(act_p, act_s[inv.long()])
    assert torch.equal(y_p, y_s)
    xd, gud, dnd = x.double().cpu(), w_gu.double().cpu(), w_dn.double().cpu()
    for t in range(T):
        for j in range(k):
            e = int(ids[t, j])
            a = (plain.silu(xd[t] @ gud[e, :I].T) * (xd[t] @ gud[e, I:].T)).to(torch.bfloat16).double()
            close(y_p[t * k + j], a @ dnd[e].T, dtype, f"pair ({t}, {j})")


@pytest.mark.parametrize("T,E,k,I,H,S", [(1, 4, 2, 32, 64, 1), (8, 60, 4, 1408, 2048, 4), (16, 6, 3, 48, 96, 2), (5, 3, 1, 40, 72, 3)])
def test_shared_expert_as_pieces_beside_unsorted_pairs(T, E, k, I, H, S):
    """a shared expert of width S*I cut into S pieces that every token takes, in the same two launches
    as the routed experts: the combine gives routed + gate * shared"""
    from ferrox_amd import ops
    dtype = torch.bfloat16
    x = rnd(T, H, dtype=dtype)
    w_gu, w_dn = rnd(E, 2 * I, H, dtype=dtype, seed=1, scale=0.3), rnd(E, H, I, dtype=dtype, seed=2, scale=0.3)
    sg, su = rnd(S * I, H, dtype=dtype, seed=3, scale=0.3), rnd(S * I, H, dtype=dtype, seed=4, scale=0.3)
    sd = rnd(H, S * I, dtype=dtype, seed=5, scale=0.3)
    gu_all = torch.cat([w_gu] + [torch.cat([sg[s * I:(s + 1) * I], su[s * I:(s + 1) * I]])[None] for s in range(S)]).contiguous()
    dn_all = torch.cat([w_dn] + [sd[:, s * I:(s + 1) * I][None] for s in range(S)]).contiguous()
    g = torch.Generator().manual_seed(13)
    ids = torch.stack([torch.randperm(E, generator=g)[:k] for _ in range(T)]).to(torch.int32).to(DEV)
    wts, gate = torch.rand(T, k, generator=g).to(DEV), torch.rand(T, generator=g).to(DEV)
    n = T * k
    act = ops.gemm(x, gu_all, epilogue=ops.EPI_GATED, pair_ids=ids, pair_div=k, always=(S, T, True))
    y = ops.gemm(act, dn_all, epilogue=ops.EPI_STORE_F32, pair_ids=ids, always=(S, T, False))
    assert act.shape == (n + S * T, I) and y.shape == (n + S * T, H)
    # the routed rows are what the products without the pieces give
    assert torch.equal(act[:n], ops.gemm(x, w_gu, epilogue=ops.EPI_GATED, pair_ids=ids, pair_div=k))
    h = torch.zeros(T, H, device=DEV)
    ops.moe_combine(h, y[:n], None, wts, k, shared=y[n:].view(S, T, H), gate=gate)
    xd = x.double().cpu()
    ref = torch.zeros(T, H, dtype=torch.float64)
    for t in range(T):
        for j in range(k):
            e = int(ids[t, j])
            a = (plain.silu(xd[t] @ w_gu[e, :I].double().cpu().T) * (xd[t] @ w_gu[e, I:].double().cpu().T)).to(dtype).double()
            ref[t] += float(wts[t, j]) * (a @ w_dn[e].double().cpu().T)
        a = (plain.silu(xd[t] @ sg.double().cpu().T) * (xd[t] @ su.double().cpu().T)).to(dtype).double()
        ref[t] += float(gate[t]) * (a @ sd.double().cpu().T)
    close(h, ref, dtype, "routed + gated shared")


@pytest.mark.parametrize("T,E,k,I,H", [(1, 4, 2, 64, 64), (8, 60, 4, 1408, 2048), (40, 6, 3, 128, 192), (300, 8, 2, 64, 128),
                                        (520, 4, 3, 128, 256), (2048, 60, 4, 192, 256)])
def test_weights_in_slabs_of_64_k(T, E, k, I, H):
    """the same products from weights stored [K/64][rows][64]: bit for bit what plain rows give, for
    few rows, many rows, sorted and unsorted pairs, and a plain (not grouped) matrix"""
    from ferrox_amd import ops
    dtype = torch.bfloat16
    x = rnd(T, H, dtype=dtype)
    w_gu, w_dn = rnd(E, 2 * I, H, dtype=dtype, seed=1, scale=0.3), rnd(E, H, I, dtype=dtype, seed=2, scale=0.3)
    kb_gu, kb_dn = ops.to_kblocked(w_gu), ops.to_kblocked(w_dn)
    assert kb_gu.shape == (E, H // 64, 2 * I, 64) and torch.equal(kb_gu[1, 0, 5], w_gu[1, 5, :64])
    g = torch.Generator().manual_seed(17)
    ids = torch.stack([torch.randperm(E, generator=g)[:k] for _ in range(T)]).to(torch.int32).to(DEV)
    offsets, sorted_token, sorted_pair, inv = ops.moe_align(ids, E)
    act = ops.gemm(x, w_gu, epilogue=ops.EPI_GATED, a_rows=sorted_token, expert_offsets=offsets, n_rows=T * k)
    act_kb = ops.gemm(x, kb_gu, epilogue=ops.EPI_GATED, a_rows=sorted_token, expert_offsets=offsets, n_rows=T * k,
                      w_kblocked=True)
    assert torch.equal(act, act_kb)
    y = ops.gemm(act, w_dn, epilogue=ops.EPI_STORE_F32, expert_offsets=offsets, c_rows=sorted_pair)
    y_kb = ops.gemm(act, kb_dn, epilogue=ops.EPI_STORE_F32, expert_offsets=offsets, c_rows=sorted_pair, w_kblocked=True)
    assert torch.equal(y, y_kb)
    if T * k <= 64:
        assert torch.equal(ops.gemm(x, kb_gu, epilogue=ops.EPI_GATED, pair_ids=ids, pair_div=k, w_kblocked=True),
                           ops.gemm(x, w_gu, epilogue=ops.EPI_GATED, pair_ids=ids, pair_div=k))
    # a plain matrix with bias, stored, and added into a residual
    bias = rnd(2 * I, dtype=dtype, seed=3)
    assert torch.equal(ops.gemm(x, kb_gu[0], bias=bias, w_kblocked=True), ops.gemm(x, w_gu[0], bias=bias))
    h1, h2 = rnd(T, 2 * I, seed=4), rnd(T, 2 * I, seed=4)
    ops.gemm(x, w_gu[0], epilogue=ops.EPI_RESID, out=h1)
    ops.gemm(x, kb_gu[0], epilogue=ops.EPI_RESID, out=h2, w_kblocked=True)
    assert torch.equal(h1, h2)


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_rmsnorm_and_embed(dtype):
    from ferrox_amd import ops
    for T, H, eps in [(1, 64, 1e-6), (5, 96, 1e-5), (3, 1000, 1e-3), (2, 4100, 1e-6)]:
        h = rnd(T, H, scale=3.0)
        w = rnd(H, dtype=dtype, seed=1)
        ref = plain.rms_norm(h.double().cpu(), w.double().cpu(), eps)
        close(ops.rmsnorm(h, w, eps, dtype), ref, dtype, f"rmsnorm {T}x{H}")
        rows = torch.tensor([T - 1, 0], dtype=torch.int32, device=DEV)
        close(ops.rmsnorm(h, w, eps, dtype, rows=rows), ref[[T - 1, 0]], dtype, "rmsnorm rows")
    table = rnd(50, 72, dtype=dtype)
    ids = torch.tensor([3, 49, 0, 3], dtype=torch.int32, device=DEV)
    assert torch.equal(ops.embed(table, ids), table[ids.long()].float())


def paged_setup(dtype, nh, nkv, hd, bs, seq_lens, theta, rot, n_pages, seed=0):
    """Random q, k, v for whole sequences; pages filled through rope_kv_write with a shuffled page order."""
    from ferrox_amd import ops
    rng = random.Random(seed)
    free = list(range(n_pages))
    rng.shuffle(free)
    max_blocks = max(-(-L // bs) for L in seq_lens)
    table = torch.zeros(len(seq_lens), max_blocks, dtype=torch.int32)
    toks = []
    for s, L in enumerate(seq_lens):
        for b in range(-(-L // bs)):
            table[s, b] = free.pop()
        toks += [(s, p) for p in range(L)]
    T = len(toks)
    q, k, v = rnd(T, nh * hd, dtype=dtype), rnd(T, nkv * hd, dtype=dtype, seed=1), rnd(T, nkv * hd, dtype=dtype, seed=2)
    # slots that no token is written to hold NaN: nothing may depend on what lies past a sequence's end
    k_pages = torch.full((n_pages, nkv, bs, hd), float("nan"), dtype=dtype, device=DEV)
    v_pages = torch.full((n_pages, nkv, hd, bs), float("nan"), dtype=dtype, device=DEV)
    pos = torch.tensor([p for _, p in toks], dtype=torch.int32, device=DEV)
    seq = torch.tensor([s for s, _ in toks], dtype=torch.int32, device=DEV)
    q_rot = q.clone()
    ops.rope_kv_write(q_rot, k, v, pos, seq, table.to(DEV), k_pages, v_pages, nh, nkv, hd, bs, rot, theta)
    return q, k, v, q_rot, k_pages, v_pages, table.to(DEV), pos, seq, toks


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("nh,nkv,hd,bs,rot,theta", [(4, 4, 16, 16, 16, 1e4), (3, 1, 32, 8, 32, 1e6), (6, 3, 48, 4, 24, 5e4),
                                                    (2, 2, 128, 64, 128, 1e6), (8, 2, 80, 16, 80, 1e4)])
def test_rope_and_cache_write(dtype, nh, nkv, hd, bs, rot, theta):
    seq_lens = [5, 2 * bs + 3, 1]
    q, k, v, q_rot, k_pages, v_pages, table, pos, seq, toks = paged_setup(dtype, nh, nkv, hd, bs, seq_lens, theta, rot, 12)
    qd, kd = q.double().cpu().reshape(-1, nh, hd), k.double().cpu().reshape(-1, nkv, hd)
    for t, (s, p) in enumerate(toks):
        want_q = torch.cat([plain.rope_neox(qd[t][:, :rot], p, theta), qd[t][:, rot:]], dim=-1)
        close(q_rot[t].reshape(nh, hd), want_q, dtype, f"q rope token {t}")
        want_k = torch.cat([plain.rope_neox(kd[t][:, :rot], p, theta), kd[t][:, rot:]], dim=-1)
        page = int(table[s, p // bs])
        close(k_pages[page, :, p % bs, :], want_k, dtype, f"k page token {t}")
        assert torch.equal(v_pages[page, :, :, p % bs].reshape(-1), v[t]), f"v page token {t}"


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("nh,nkv,hd,bs,rot,seq_lens", [(4, 2, 128, 64, 128, [300, 7, 330]), (3, 1, 80, 64, 48, [640, 5]),
                                                       (2, 2, 64, 16, 64, [530, 40]), (2, 1, 96, 128, 96, [520])])
def test_rope_and_cache_write_of_long_prompts(dtype, nh, nkv, hd, bs, rot, seq_lens):
    """Many tokens, eight pairs to a thread: pages that begin or end inside a sequence, page sizes other than 64,
    tokens of another sequence between."""
    theta = 1e6
    n_pages = sum(-(-L // bs) for L in seq_lens) + 2
    q, k, v, q_rot, k_pages, v_pages, table, pos, seq, toks = paged_setup(dtype, nh, nkv, hd, bs, seq_lens, theta, rot, n_pages)
    assert len(toks) >= 512
    T = len(toks)
    p = pos.double().cpu()
    freq = 1.0 / theta ** (torch.arange(0, rot, 2, dtype=torch.float64) / rot)
    # plain.rope_neox(..., "float32"), all tokens at once: the float32 product of position and float32 frequency
    ang = (p.float()[:, None] * freq.float()[None, :]).double()
    def rotated(x, heads):
        x = x.double().cpu().reshape(T, heads, hd)
        a, b = x[..., :rot // 2], x[..., rot // 2:rot]
        c, s_ = torch.cos(ang)[:, None, :], torch.sin(ang)[:, None, :]
        return torch.cat([a * c - b * s_, a * s_ + b * c, x[..., rot:]], dim=-1)
    for t in (5, T - 1):
        assert torch.allclose(plain.rope_neox(q[t].double().cpu().reshape(nh, hd)[:, :rot], int(pos[t]), theta, "float32"),
                              rotated(q, nh)[t, :, :rot], atol=1e-12)  # the formula above is the plain one
    near = lambda got, want, what: close(got, want, dtype, what)
    near(q_rot.reshape(T, nh, hd), rotated(q, nh), "rotated queries")
    page_of = table.cpu()[seq.cpu().long(), (pos.cpu() // bs).long()].long()
    slot = (pos.cpu() % bs).long()
    near(k_pages.cpu()[page_of, :, slot, :], rotated(k, nkv), "key pages")
    assert torch.equal(v_pages.cpu()[page_of, :, :, slot], v.cpu().reshape(T, nkv, hd)), "value pages"
    used = torch.zeros(n_pages, bs, dtype=torch.bool)
    used[page_of, slot] = True
    assert bool(torch.isnan(v_pages.cpu().float().permute(0, 3, 1, 2)[~used]).all()), "slots past the sequences stay untouched"


DEEP_POSITIONS = [0, 1, 511, 2047, 2048, 4097, 8191, 16384, 20000, 32766, 32767]


def rotated_by_float32_angles(x, positions, rot, theta, angles="float32"):
    """x [T, heads, hd] in float64 with its first `rot` dimensions turned, split halves, by the plain model's angles"""
    out = x.clone()
    for t, p in enumerate(positions):
        out[t, :, :rot] = plain.rope_neox(x[t, :, :rot], int(p), theta, angles)
    return out


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("nh,nkv,hd,bs,rot,theta", [(2, 1, 128, 64, 128, 1e6), (3, 3, 64, 16, 32, 1e4), (2, 2, 16, 16, 16, 1e6)])
def test_rope_deep_in_a_sequence(dtype, nh, nkv, hd, bs, rot, theta):
    """Rotation and cache write at positions up to 32,767.  The angle is the float32 product of the position and
    the float32 frequency (ferrox-core/src/attention.rs:26-27); against float64 sines and cosines of exactly that
    angle the float32 kernel is right to rounding, and would be off by a thousand times that against exact angles."""
    from ferrox_amd import ops
    T = len(DEEP_POSITIONS)
    blocks = -(-32768 // bs)
    table = torch.zeros(1, blocks, dtype=torch.int32)
    used = sorted({p // bs for p in DEEP_POSITIONS})
    order = torch.randperm(len(used), generator=torch.Generator().manual_seed(bs)).tolist()
    for b, page in zip(used, order):
        table[0, b] = page + 1                             # page 0 stays empty
    q, k, v = rnd(T, nh * hd, dtype=dtype), rnd(T, nkv * hd, dtype=dtype, seed=1), rnd(T, nkv * hd, dtype=dtype, seed=2)
    k_pages = torch.full((len(used) + 1, nkv, bs, hd), float("nan"), dtype=dtype, device=DEV)
    v_pages = torch.full((len(used) + 1, nkv, hd, bs), float("nan"), dtype=dtype, device=DEV)
    pos = torch.tensor(DEEP_POSITIONS, dtype=torch.int32, device=DEV)
    seq = torch.zeros(T, dtype=torch.int32, device=DEV)
    q_rot = q.clone()
    ops.rope_kv_write(q_rot, k, v, pos, seq, table.to(DEV), k_pages, v_pages, nh, nkv, hd, bs, rot, theta)
    want_q = rotated_by_float32_angles(q.double().cpu().reshape(T, nh, hd), DEEP_POSITIONS, rot, theta)
    want_k = rotated_by_float32_angles(k.double().cpu().reshape(T, nkv, hd), DEEP_POSITIONS, rot, theta)
    page_of = table[0, (pos.cpu() // bs).long()].long()
    slot = (pos.cpu() % bs).long()
    got_q, got_k = q_rot.reshape(T, nh, hd), k_pages.cpu()[page_of, :, slot, :]
    close(got_q, want_q, dtype, "rotated queries")
    close(got_k, want_k, dtype, "key pages")
    assert torch.equal(v_pages.cpu()[page_of, :, :, slot], v.cpu().reshape(T, nkv, hd)), "value pages"
    assert bool(torch.isnan(k_pages[0].float()).all()), "a page that no position maps to was written"
    if dtype == torch.float32:
        exact = rotated_by_float32_angles(q.double().cpu().reshape(T, nh, hd), DEEP_POSITIONS, rot, theta, "exact")
        off = float((got_q.double().cpu() - exact).abs().max()) / float(exact.abs().max())
        assert off > 1e-4, f"exact angles are only {off:.2e} away: the test does not tell the two apart"


def test_qkv_product_that_rotates_deep_in_a_sequence():
    """the rotating product's epilogue at positions up to 32,767: the bits of the product followed by rope_kv_write,
    which the test above holds against the plain rotation"""
    from ferrox_amd import ops
    T, H, nh, nkv, hd, bs, rot, theta = len(DEEP_POSITIONS), 264, 4, 2, 64, 64, 64, 1e6
    N = (nh + 2 * nkv) * hd
    w = rnd(N, H, dtype=torch.bfloat16, seed=1, scale=0.05)
    b = rnd(N, dtype=torch.bfloat16, seed=2)
    x = rnd(T, H, dtype=torch.bfloat16, seed=3)
    blocks = 32768 // bs
    used = sorted({p // bs for p in DEEP_POSITIONS})
    table = torch.zeros(1, blocks, dtype=torch.int32)
    for i, blk in enumerate(used):
        table[0, blk] = len(used) - i
    table = table.to(DEV)
    pos = torch.tensor(DEEP_POSITIONS, dtype=torch.int32, device=DEV)
    seq = torch.zeros(T, dtype=torch.int32, device=DEV)
    pages = lambda: (torch.zeros(len(used) + 1, nkv, bs, hd, dtype=torch.bfloat16, device=DEV),
                     torch.zeros(len(used) + 1, nkv, hd, bs, dtype=torch.bfloat16, device=DEV))
    assert ops.can_qkv_rope(x, w, T, hd, rot, False)
    k1, v1 = pages()
    got = ops.qkv_rope(x, w, b, pos, seq, table, k1, v1, nh, nkv, hd, bs, rot, theta)
    k2, v2 = pages()
    ref = ops.gemm(x, w, bias=b)
    qw, kvw = nh * hd, nkv * hd
    ops.rope_kv_write(ref[:, :qw], ref[:, qw:qw + kvw], ref[:, qw + kvw:], pos, seq, table, k2, v2, nh, nkv, hd, bs, rot, theta)
    assert torch.equal(got[:, :qw], ref[:, :qw]), "rotated queries"
    assert torch.equal(k1, k2) and float(k1.abs().sum()) > 0, "key pages"
    assert torch.equal(v1, v2), "value pages"


@pytest.mark.parametrize("later", [False, True])
@pytest.mark.parametrize("T,H,nh,nkv,hd,bs,rot,bias", [(1, 2048, 16, 16, 128, 64, 128, True), (8, 2048, 16, 16, 128, 64, 128, True),
                                                       (16, 264, 6, 2, 64, 16, 32, True), (5, 520, 3, 1, 32, 8, 0, False),
                                                       (7, 128, 4, 2, 96, 32, 64, True), (30, 264, 6, 2, 64, 16, 64, True),
                                                       (64, 2048, 16, 16, 128, 64, 128, True), (50, 128, 4, 2, 96, 32, 64, False)])
def test_qkv_product_that_rotates_and_writes_the_cache(later, T, H, nh, nkv, hd, bs, rot, bias):
    """The q/k/v product with rotation and cache write in its epilogue gives the bits of the product followed
    by rope_kv_write: rotated queries, key pages and value pages; also from rows whose norm's scale is applied
    by the product."""
    from ferrox_amd import ops
    N = (nh + 2 * nkv) * hd
    w = rnd(N, H, dtype=torch.bfloat16, seed=1, scale=0.05)
    b = rnd(N, dtype=torch.bfloat16, seed=2) if bias else None
    x = rnd(T, H, dtype=torch.bfloat16, seed=3)
    if later:
        ss = (torch.rand(T, (H + 255) // 256, generator=torch.Generator().manual_seed(4)) * 40 + 1).to(DEV)
        x = ops.ScaleLater(x, ss, 1e-6)
    g = torch.Generator().manual_seed(5)
    n_seq = 3
    seq = torch.randint(0, n_seq, (T,), generator=g)
    pos = torch.zeros(T, dtype=torch.long)
    for s_ in range(n_seq):                       # distinct positions inside a sequence
        idx = (seq == s_).nonzero().flatten()
        pos[idx] = torch.randperm(5 * bs, generator=g)[:idx.numel()]
    table = torch.randperm(n_seq * 5, generator=g).reshape(n_seq, 5).to(torch.int32).to(DEV)
    pos_d, seq_d = pos.to(torch.int32).to(DEV), seq.to(torch.int32).to(DEV)
    pages = lambda: (torch.zeros(n_seq * 5, nkv, bs, hd, dtype=torch.bfloat16, device=DEV),
                     torch.zeros(n_seq * 5, nkv, hd, bs, dtype=torch.bfloat16, device=DEV))
    assert ops.can_qkv_rope(x, w, T, hd, rot, False)
    k1, v1 = pages()
    got = ops.qkv_rope(x, w, b, pos_d, seq_d, table, k1, v1, nh, nkv, hd, bs, rot, 1e6)
    k2, v2 = pages()
    ref = ops.gemm(x.x, w, bias=b, row_ss=(x.ss, x.eps)) if later else ops.gemm(x, w, bias=b)
    qw, kvw = nh * hd, nkv * hd
    ops.rope_kv_write(ref[:, :qw], ref[:, qw:qw + kvw], ref[:, qw + kvw:], pos_d, seq_d, table, k2, v2, nh, nkv, hd, bs, rot, 1e6)
    assert torch.equal(got[:, :qw], ref[:, :qw]), "rotated queries"
    assert torch.equal(k1, k2), "key pages"
    assert torch.equal(v1, v2), "value pages"
    got2 = ops.qkv_rope(x, w, b, pos_d, seq_d, table, None, None, nh, nkv, hd, bs, rot, 1e6)     # no pages: queries only
    assert torch.equal(got2[:, :qw], ref[:, :qw])
    assert not ops.can_qkv_rope(x, w, 65, hd, rot, False) and not ops.can_qkv_rope(x, w, T, hd, rot, True)


@pytest.mark.parametrize("later", [False, True])
@pytest.mark.parametrize("T", [33, 47, 48, 49, 63])
@pytest.mark.parametrize("H,nh,tiles", [(264, 32, (3, 4)), (2312, 32, (3, 4)), (520, 4, (1, 1))])
def test_rotating_product_of_several_row_tiles_a_block(later, T, H, nh, tiles):
    """One, three and four row tiles a block, with rows of the last tile missing, K that ends in a piece, sums of up to eight and of ten numbers."""
    from ferrox_amd import ops
    from ferrox_amd.csrc.build import load_library
    cus = torch.cuda.get_device_properties(0).multi_processor_count
    groups = (nh + 4) * 4
    assert load_library("gemm").fx_qkv_rope_row_tiles(T, groups, cus) == tiles[T > 48] or cus != 256
    test_qkv_product_that_rotates_and_writes_the_cache(later, T, H, nh, 2, 128, 16, 64, True)


@pytest.mark.parametrize("T,H", [(16, 1032), (13, 1384), (9, 2000), (16, 2048), (1, 1032), (3, 2000), (16, 1024)])
def test_rotating_product_whose_weights_leave_before_the_sums(T, H):
    """Sums of one batch and rows enough for it, K with and without a last part of a piece: the bits of the product and the rotation."""
    from ferrox_amd.csrc.build import load_library
    assert load_library("gemm").fx_qkv_rope_weights_first(T, H, -(-H // 256))
    test_qkv_product_that_rotates_and_writes_the_cache(True, T, H, 6, 2, 64, 16, 32, True)


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("nh,nkv,hd,bs,rot,interleaved", [(3, 1, 32, 8, 32, False), (2, 2, 64, 16, 32, False),
                                                          (2, 1, 48, 8, 24, True), (4, 2, 128, 64, 128, False)])
def test_rope_with_frequency_factors(dtype, nh, nkv, hd, bs, rot, interleaved):
    """A table of per-pair factors divides the angles (ferrox-core/src/attention.rs:319-333): the rotating
    kernel, and for bfloat16 split halves also the q/k/v product that rotates in its epilogue, against the
    formula; a table of ones gives the bits of no table."""
    from ferrox_amd import ops
    theta, T = 1e4, 20
    g = torch.Generator().manual_seed(rot)
    factors = (1.0 + 7.0 * torch.rand(rot // 2, generator=g)).to(DEV)
    q, k, v = rnd(T, nh * hd, dtype=dtype), rnd(T, nkv * hd, dtype=dtype, seed=1), rnd(T, nkv * hd, dtype=dtype, seed=2)
    pos = torch.arange(3, 3 + T, dtype=torch.int32, device=DEV)
    seq = torch.zeros(T, dtype=torch.int32, device=DEV)
    n_blocks = -(-(3 + T) // bs)
    table = torch.arange(n_blocks, dtype=torch.int32, device=DEV).flip(0)[None].contiguous()
    pages = lambda: (torch.zeros(n_blocks, nkv, bs, hd, dtype=dtype, device=DEV), torch.zeros(n_blocks, nkv, hd, bs, dtype=dtype, device=DEV))

    def want(x, heads):
        x = x.double().cpu().reshape(T, heads, hd)
        i = torch.arange(rot // 2, dtype=torch.float64)
        ang = pos.double().cpu()[:, None] * (1.0 / theta ** (2 * i / rot))[None, :] / factors.double().cpu()[None, :]
        c, s_ = torch.cos(ang)[:, None, :], torch.sin(ang)[:, None, :]
        out = x.clone()
        ia, ib = (2 * i.long(), 2 * i.long() + 1) if interleaved else (i.long(), i.long() + rot // 2)
        out[..., ia], out[..., ib] = x[..., ia] * c - x[..., ib] * s_, x[..., ia] * s_ + x[..., ib] * c
        return out

    kp, vp = pages()
    q1 = q.clone()
    ops.rope_kv_write(q1, k, v, pos, seq, table, kp, vp, nh, nkv, hd, bs, rot, theta, interleaved, freq_factors=factors)
    close(q1.reshape(T, nh, hd), want(q, nh), dtype, "rotated queries")
    page_of, slot = table[0].cpu()[(pos.cpu() // bs).long()].long(), (pos.cpu() % bs).long()
    close(kp.cpu()[page_of, :, slot, :], want(k, nkv), dtype, "key pages")
    # a table of ones is no table
    ones = torch.ones(rot // 2, device=DEV)
    kp1, vp1 = pages()
    kp0, vp0 = pages()
    qa, qb = q.clone(), q.clone()
    ops.rope_kv_write(qa, k, v, pos, seq, table, kp1, vp1, nh, nkv, hd, bs, rot, theta, interleaved, freq_factors=ones)
    ops.rope_kv_write(qb, k, v, pos, seq, table, kp0, vp0, nh, nkv, hd, bs, rot, theta, interleaved)
    assert torch.equal(qa, qb) and torch.equal(kp1, kp0)
    with pytest.raises(ops.KernelError):
        ops.rope_kv_write(qa, k, v, pos, seq, table, kp1, vp1, nh, nkv, hd, bs, rot, theta, interleaved, freq_factors=ones[:-1])
    if dtype == torch.bfloat16 and not interleaved and rot % 32 == 0 and hd % 32 == 0:
        H = 96
        w = rnd((nh + 2 * nkv) * hd, H, dtype=dtype, seed=5, scale=0.1)
        x = rnd(T, H, dtype=dtype, seed=6)
        assert ops.can_qkv_rope(x, w, T, hd, rot, False)
        k1, v1 = pages()
        got = ops.qkv_rope(x, w, None, pos, seq, table, k1, v1, nh, nkv, hd, bs, rot, theta, freq_factors=factors)
        ref = ops.gemm(x, w)
        qw, kvw = nh * hd, nkv * hd
        k2, v2 = pages()
        ops.rope_kv_write(ref[:, :qw], ref[:, qw:qw + kvw], ref[:, qw + kvw:], pos, seq, table, k2, v2, nh, nkv, hd, bs, rot,
                          theta, freq_factors=factors)
        assert torch.equal(got[:, :qw], ref[:, :qw]) and torch.equal(k1, k2) and torch.equal(v1, v2)


@pytest.mark.parametrize("form", ["plain", "window", "window_keep", "chunked", "gated", "odd_out"])
@pytest.mark.parametrize("bs", [64, 128])
def test_waves_of_32_queries(form, bs):
    """Items of up to 128 queries of 128-wide heads on waves of 32 queries, one group and two, whatever their number, against float64 over what the pages
    hold: sequences that end on both sides of a wave, an item and a tile, NaN past their ends, no other output touched."""
    from ferrox_amd import debug, ops
    nh, nkv, hd = 4, 2, 128
    seq_lens = [1, 31, 33, 64, 129, 200, 450]
    q, k, v, q_rot, k_pages, v_pages, table, pos, seq, toks = paged_setup(torch.bfloat16, nh, nkv, hd, bs, seq_lens, 1e4, hd, 64)
    T, scale = len(toks), hd ** -0.5
    window = 70 if "window" in form else 0
    mask_chunk, keep = 48 if form == "chunked" else 0, 20 if form == "window_keep" else 0
    kw = dict(mask_chunk=mask_chunk, keep_first=keep, sinks=rnd(nh, seed=3) if form == "window_keep" else None,
              gate=rnd(T, nh * hd, dtype=torch.bfloat16, seed=4) if form == "gated" else None)
    kp, vp, tab = k_pages.double().cpu(), v_pages.double().cpu(), table.cpu()
    want, start, items = torch.zeros(T, nh, hd, dtype=torch.float64), 0, []
    for s, L in enumerate(seq_lens):
        ks = torch.stack([kp[int(tab[s, p // bs]), :, p % bs, :] for p in range(L)]).repeat_interleave(nh // nkv, 1)
        vs = torch.stack([vp[int(tab[s, p // bs]), :, :, p % bs] for p in range(L)]).repeat_interleave(nh // nkv, 1)
        qs = q_rot[start:start + L].double().cpu().reshape(L, nh, hd)
        t = torch.arange(L)
        seen = t[None, :] <= t[:, None]
        if window:
            seen &= (t[:, None] - t[None, :] < window) | (t[None, :] < keep)
        if mask_chunk:
            seen &= t[None, :] >= t[:, None] // mask_chunk * mask_chunk
        sc = (torch.einsum("qhd,khd->hqk", qs, ks) * scale).masked_fill(~seen, -math.inf)
        if kw["sinks"] is not None:
            sc = torch.cat([sc, kw["sinks"].double().cpu().view(nh, 1, 1).expand(nh, L, 1)], -1)
        want[start:start + L] = torch.einsum("hqk,khd->qhd", torch.softmax(sc, -1)[..., :L], vs)
        items += [(s, start + t0, min(128, L - t0)) for t0 in range(0, L, 128)]
        start += L
    want = want.reshape(T, nh * hd)
    if kw["gate"] is not None:
        want = want * torch.sigmoid(kw["gate"].double().cpu())
    i32 = lambda x: torch.tensor(x, dtype=torch.int32, device=DEV)
    cols = [i32([it[c] for it in items]) for c in range(3)]
    odd = 3 if form == "odd_out" else 0              # rows of the output not on 8 bytes
    for groups in (1, 2):
        room = torch.full((T + 1, nh * hd + odd), 7.0, dtype=torch.bfloat16, device=DEV)
        out = room[:T, odd:]
        with debug.kernel_switch("attention", "rows32", 2), debug.kernel_switch("attention", "direct_groups", groups):
            ops.attention_tiles(q_rot, out, k_pages, v_pages, table, pos, *cols, nh, nkv, hd, bs, window, scale, tile_q=128, **kw)
        close(out, want, torch.bfloat16, f"{form}, {groups} group(s)")
        assert bool((room[T] == 7).all()) and bool((room[:, :odd] == 7).all())


@pytest.mark.parametrize("window,keep,broken,clean", [(0, 0, 100, [(0, 64)]), (0, 0, 200, [(0, 192)]), (0, 0, 300, [(0, 256)]),
                                                      (64, 0, 70, [(0, 64), (192, 330)]), (64, 10, 70, [(0, 64), (192, 330)]), (64, 10, 5, [])])
def test_a_value_that_is_not_a_number_reaches_no_wave_of_queries_that_sees_none_of_its_tile(window, keep, broken, clean):
    """Infinite values of one key (a later one, one before the window, a kept one): queries in waves of 32 that see no key of its 64 have the bits that they have
    without it, whatever the other waves of their item see; the queries that do see the key are not finite."""
    from ferrox_amd import debug, ops
    nh, nkv, hd, bs, n = 4, 2, 128, 64, 330
    q, k, v, q_rot, k_pages, v_pages, table, pos, seq, toks = paged_setup(torch.bfloat16, nh, nkv, hd, bs, [n], 1e4, hd, 64)
    i32 = lambda x: torch.tensor(x, dtype=torch.int32, device=DEV)
    cols = [i32([0, 0, 0]), i32([0, 128, 256]), i32([128, 128, n - 256])]
    bad = v_pages.clone()
    bad[int(table[0, broken // bs]), :, :, broken % bs] = math.inf
    sees = torch.arange(n)
    sees = (sees >= broken) & ((sees - broken < window) | (broken < keep) if window else True)
    for groups in (1, 2):
        out = [torch.zeros(n, nh * hd, dtype=torch.bfloat16, device=DEV) for _ in range(2)]
        with debug.kernel_switch("attention", "rows32", 2), debug.kernel_switch("attention", "direct_groups", groups):
            for y, vp in zip(out, (v_pages, bad)):
                ops.attention_tiles(q_rot, y, k_pages, vp, table, pos, *cols, nh, nkv, hd, bs, window, hd ** -0.5, tile_q=128, keep_first=keep)
        for b, e in clean:
            assert torch.equal(out[0][b:e], out[1][b:e]), (groups, b, e)
        assert not bool(torch.isfinite(out[1][sees.to(DEV)]).any()) and bool(torch.isfinite(out[0]).all())


@pytest.mark.parametrize("form", ["plain", "window", "window_keep", "shaped", "chunked"])
@pytest.mark.parametrize("vd,bs", [(192, 64), (256, 64), (16, 128)])
def test_attention_of_the_widest_heads_in_blocks_of_64_queries(vd, bs, form):
    """Items of 128 queries on eight waves, items of 64 on four or on the kernel that stages through registers: the same bits from all, near the plain
    attention; sequences that end on both sides of a wave, half an item, an item and a tile, NaN past their ends."""
    from ferrox_amd import debug, ops
    nh, nkv, hd = 4, 2, 256
    seq_lens = [1, 15, 17, 63, 64, 65, 127, 128, 129, 193, 320]
    q, k, v, q_rot, k_pages, v_pages, table, pos, seq, toks = paged_setup(torch.bfloat16, nh, nkv, hd, bs, seq_lens, 1e4, hd, 64)
    v_pages = v_pages[:, :, :vd].contiguous()
    T, scale = len(toks), hd ** -0.5
    window = 70 if "window" in form else 0
    mask_chunk, keep = 48 if form == "chunked" else 0, 20 if form == "window_keep" else 0
    kw = dict(v_dim=vd, mask_chunk=mask_chunk, keep_first=keep, sinks=rnd(nh, seed=3) if form == "window_keep" else None)
    if form == "shaped":
        kw.update(softcap=5.0, slopes=torch.tensor([0.5, 0.25, 0.125, 0.0625], device=DEV))
    kp, vp, tab = k_pages.double().cpu(), v_pages.double().cpu(), table.cpu()
    want, start = torch.zeros(T, nh, vd, dtype=torch.float64), 0
    items = {64: [], 128: []}
    for s, L in enumerate(seq_lens):
        ks = torch.stack([kp[int(tab[s, p // bs]), :, p % bs, :] for p in range(L)]).repeat_interleave(nh // nkv, 1)
        vs = torch.stack([vp[int(tab[s, p // bs]), :, :, p % bs] for p in range(L)]).repeat_interleave(nh // nkv, 1)
        qs = q_rot[start:start + L].double().cpu().reshape(L, nh, hd)
        t = torch.arange(L)
        back = t[:, None] - t[None, :]
        seen = back >= 0
        if window:
            seen &= (back < window) | (t[None, :] < keep)
        if mask_chunk:
            seen &= t[None, :] >= t[:, None] // mask_chunk * mask_chunk
        sc = torch.einsum("qhd,khd->hqk", qs, ks) * scale
        if form == "shaped":
            sc = 5.0 * torch.tanh(sc / 5.0) - kw["slopes"].double().cpu().view(nh, 1, 1) * back
        sc = sc.masked_fill(~seen, -math.inf)
        if kw["sinks"] is not None:
            sc = torch.cat([sc, kw["sinks"].double().cpu().view(nh, 1, 1).expand(nh, L, 1)], -1)
        want[start:start + L] = torch.einsum("hqk,khd->qhd", torch.softmax(sc, -1)[..., :L], vs)
        for n in items:
            items[n] += [(s, start + t0, min(n, L - t0)) for t0 in range(0, L, n)]
        start += L
    i32 = lambda x: torch.tensor(x, dtype=torch.int32, device=DEV)
    got = {}
    for n, stages in ((128, 2), (64, 2), (64, 0)):
        cols = [i32([it[c] for it in items[n]]) for c in range(3)]
        out = torch.full((T + 1, nh * vd), 7.0, dtype=torch.bfloat16, device=DEV)
        with debug.kernel_switch("attention", "direct_stages", stages):
            ops.attention_tiles(q_rot, out[:T], k_pages, v_pages, table, pos, *cols, nh, nkv, hd, bs, window, scale, tile_q=n, **kw)
        assert bool((out[T] == 7).all())
        close(out[:T], want.reshape(T, nh * vd), torch.bfloat16, f"{form}, items of {n}, {stages} stages")
        got[n, stages] = out
    for key, out in got.items():
        assert torch.equal(out, got[128, 2]), key


@pytest.mark.parametrize("form", ["plain", "window", "window_keep", "chunked"])
@pytest.mark.parametrize("nh,nkv,hd,vd", [(16, 1, 256, 192), (32, 1, 256, 256), (8, 4, 256, 256), (28, 4, 192, 192), (4, 1, 320, 320), (3, 3, 200, 136)])
def test_single_queries_of_wide_heads_far_into_a_sequence(nh, nkv, hd, vd, form):
    """Chunks as the sizes and the mask choose them: sequences deep behind a mask's first key, at both ends of a tile and shorter than the mask, beside each other."""
    from ferrox_amd import ops
    bs, seq_lens = 64, [2100, 1, 64, 65, 700, 2047]
    q, k, v, q_rot, k_pages, v_pages, table, pos, seq, toks = paged_setup(torch.bfloat16, nh, nkv, hd, bs, seq_lens, 1e4, min(hd, 256), 96)
    v_pages = v_pages[:, :, :vd].contiguous()
    window, mask_chunk = 130 if "window" in form else 0, 200 if form == "chunked" else 0
    keep, scale = 20 if form == "window_keep" else 0, hd ** -0.5
    kp, vp, tab = k_pages.double().cpu(), v_pages.double().cpu(), table.cpu().long()
    last = [sum(seq_lens[:i + 1]) - 1 for i in range(len(seq_lens))]
    want = torch.zeros(len(seq_lens), nh, vd, dtype=torch.float64)
    for s, L in enumerate(seq_lens):
        pages = tab[s, :-(-L // bs)]
        ks = kp[pages].permute(0, 2, 1, 3).reshape(-1, nkv, hd)[:L].repeat_interleave(nh // nkv, 1)
        vs = vp[pages].permute(0, 3, 1, 2).reshape(-1, nkv, vd)[:L].repeat_interleave(nh // nkv, 1)
        t = torch.arange(L)
        seen = (L - 1 - t < window) | (t < keep) if window else t >= ((L - 1) // mask_chunk * mask_chunk if mask_chunk else 0)
        sc = (torch.einsum("hd,khd->hk", q_rot[last[s]].double().cpu().view(nh, hd), ks) * scale).masked_fill(~seen, -math.inf)
        want[s] = torch.einsum("hk,khd->hd", torch.softmax(sc, -1), vs)
    i32 = lambda x: torch.tensor(x, dtype=torch.int32, device=DEV)
    for bound in (max(seq_lens), 30000):        # (what a recorded step is told is more than the sequences have)
        out = torch.full((len(toks), nh * vd), 7.0, dtype=torch.bfloat16, device=DEV)
        ops.attention_decode(q_rot, out, k_pages, v_pages, table, pos, i32(range(len(seq_lens))), i32(last), nh, nkv, hd, bs, window, scale,
                             max_kv_len=bound, v_dim=vd, mask_chunk=mask_chunk, keep_first=keep)
        close(out[last], want.reshape(len(seq_lens), nh * vd), torch.bfloat16, f"{form}, {bound} keys at most")
        assert bool((out[:last[0]] == 7).all())


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("nh,nkv,hd,bs,window", [(4, 4, 16, 16, 0), (3, 1, 32, 8, 16), (6, 3, 48, 4, 40), (2, 2, 128, 64, 0),
                                                 (8, 2, 80, 16, 7), (4, 1, 256, 32, 100), (4, 2, 64, 64, 50), (3, 1, 128, 128, 90),
                                                 (2, 1, 64, 64, 0), (2, 2, 128, 64, 70)])
def test_attention_kernels(dtype, nh, nkv, hd, bs, window):
    """Whole sequences through the tiled kernel, and their last tokens again through the decode
    kernel, against the plain attention on the same rotated, rounded q/k/v."""
    from ferrox_amd import ops
    seq_lens = [70, 1, 33, 150]
    theta = 1e4
    q, k, v, q_rot, k_pages, v_pages, table, pos, seq, toks = paged_setup(dtype, nh, nkv, hd, bs, seq_lens, theta, hd, 128)
    T = len(toks)
    scale = 1.0 / math.sqrt(hd)
    # reference from what the pages hold
    ref = torch.zeros(T, nh, hd, dtype=torch.float64)
    starts = [0]
    for L in seq_lens:
        starts.append(starts[-1] + L)
    kp, vp, tab = k_pages.double().cpu(), v_pages.double().cpu(), table.cpu()
    for s, L in enumerate(seq_lens):
        ks = torch.stack([kp[int(tab[s, p // bs]), :, p % bs, :] for p in range(L)])
        vs = torch.stack([vp[int(tab[s, p // bs]), :, :, p % bs] for p in range(L)])
        qs = q_rot[starts[s]:starts[s + 1]].double().cpu().reshape(L, nh, hd)
        ref[starts[s]:starts[s + 1]] = plain.causal_attention(qs, ks, vs, nh, nkv, window or None)
    ref = ref.reshape(T, nh * hd)
    # blocks of up to 64 queries
    t_seq, t_tok, t_n = [], [], []
    for s, L in enumerate(seq_lens):
        for t0 in range(0, L, 64):
            t_seq.append(s); t_tok.append(starts[s] + t0); t_n.append(min(64, L - t0))
    i32 = lambda x: torch.tensor(x, dtype=torch.int32, device=DEV)
    from ferrox_amd import debug
    for groups in (1, 2):      # of waves per block of the kernel for pages of 64 keys (it takes two where blocks are few)
        out = torch.zeros(T, nh * hd, dtype=dtype, device=DEV)
        with debug.kernel_switch("attention", "direct_groups", groups):
            ops.attention_tiles(q_rot, out, k_pages, v_pages, table, pos, i32(t_seq), i32(t_tok), i32(t_n), nh, nkv, hd, bs, window, scale)
        close(out, ref, dtype, f"tiled attention, {groups} group(s) of waves")
    tq = ops.attention_tile_queries(dtype, hd, bs)
    assert tq == (128 if dtype == torch.bfloat16 and bs % 64 == 0 and hd in (64, 128) else 64)
    if tq > 64:       # larger items where the kernel takes them: blocks of eight waves
        t_seq, t_tok, t_n = [], [], []
        for s, L in enumerate(seq_lens):
            for t0 in range(0, L, tq):
                t_seq.append(s); t_tok.append(starts[s] + t0); t_n.append(min(tq, L - t0))
        for groups in (1, 2):
            wide = torch.zeros(T, nh * hd, dtype=dtype, device=DEV)
            with debug.kernel_switch("attention", "direct_groups", groups):
                ops.attention_tiles(q_rot, wide, k_pages, v_pages, table, pos, i32(t_seq), i32(t_tok), i32(t_n), nh, nkv, hd, bs, window,
                                    scale, tile_q=tq)
            close(wide, ref, dtype, f"tiled attention, items of {tq}, {groups} group(s) of waves")
    else:
        with pytest.raises(ops.KernelError):
            ops.attention_tiles(q_rot, out, k_pages, v_pages, table, pos, i32(t_seq), i32(t_tok), i32(t_n), nh, nkv, hd, bs, window,
                                scale, tile_q=128)
    # the last token of every sequence as a single query
    out2 = torch.zeros(T, nh * hd, dtype=dtype, device=DEV)
    last = [starts[s + 1] - 1 for s in range(len(seq_lens))]
    for chunk in (64, 256):
        ops.attention_decode(q_rot, out2, k_pages, v_pages, table, pos, i32(list(range(len(seq_lens)))), i32(last),
                             nh, nkv, hd, bs, window, scale, max_kv_len=max(seq_lens), chunk=chunk)
        close(out2[last], ref[last], dtype, f"decode attention chunk {chunk}")


@pytest.mark.parametrize("nh,nkv,hd,vd", [(2, 1, 4, 4), (34, 2, 20, 36), (4, 2, 64, 64), (3, 3, 68, 48), (16, 4, 128, 128),
                                          (2, 2, 132, 96), (2, 1, 192, 256)])
@pytest.mark.parametrize("form", ["plain", "window", "window_keep", "chunk", "shaped", "gated", "turned"])
def test_float32_attention_on_the_matrix_units_against_the_kernels_for_any_shape(nh, nkv, hd, vd, form):
    """The same sequences in pages of 8 keys (the matrix-unit kernels) and of 7 (the kernels for any shape): every form of
    mask and score, group sizes on both sides of 16, edge tiles beside slots that hold NaN.  Both sum float32 products in
    orders of their own: they differ by roundings of sums of up to a few hundred terms."""
    from ferrox_amd import ops
    lens = [1, 70, 197]
    T = sum(lens)
    q, k, v = rnd(T, nh * hd), rnd(T, nkv, hd, seed=1), rnd(T, nkv, vd, seed=2)
    starts = [0, 1, 71, 268]
    pos = torch.cat([torch.arange(n) for n in lens]).to(torch.int32).to(DEV)
    i32 = lambda x: torch.tensor(x, dtype=torch.int32, device=DEV)
    kw = dict(v_dim=vd)
    window = 0
    if form.startswith("window"):
        window = 50
        kw.update(keep_first=20 if form == "window_keep" else 0, sinks=rnd(nh, seed=3))
    elif form == "chunk":
        kw.update(mask_chunk=48)
    elif form == "shaped":
        kw.update(softcap=3.0, slopes=torch.rand(nh, device=DEV) * 0.2, distance_bias=ops.distance_bias_rows(rnd(nh, 30, seed=4)))
    elif form == "gated":
        kw.update(gate=rnd(T, nh * vd, seed=5))
    elif form == "turned":
        angle = torch.rand(T, vd // 2, device=DEV) * 6.0
        kw.update(turns=torch.stack([angle.cos(), angle.sin()], -1).contiguous())
    got = {}
    for bs in (8, 7):
        blocks = [-(-n // bs) for n in lens]
        table = torch.zeros(3, max(blocks), dtype=torch.int32)
        kp = torch.full((sum(blocks), nkv, bs, hd), float("nan"), device=DEV)
        vp = torch.full((sum(blocks), nkv, vd, bs), float("nan"), device=DEV)
        page = 0
        for s, n in enumerate(lens):
            for b in range(blocks[s]):
                table[s, b] = page
                rows = slice(starts[s] + b * bs, min(starts[s] + (b + 1) * bs, starts[s + 1]))
                kp[page, :, :rows.stop - rows.start] = k[rows].transpose(0, 1)
                vp[page, :, :, :rows.stop - rows.start] = v[rows].permute(1, 2, 0)
                page += 1
        items = [(s, starts[s] + o, min(64, n - o)) for s, n in enumerate(lens) for o in range(0, n, 64)]
        out, single = torch.zeros(T, nh * vd, device=DEV), torch.zeros(T, nh * vd, device=DEV)
        args = (nh, nkv, hd, bs, window, 0.7 * hd ** -0.5)
        ops.attention_tiles(q, out, kp, vp, table.to(DEV), pos, *(i32(list(x)) for x in zip(*items)), *args, **kw)
        last = [x - 1 for x in starts[1:]] + [starts[2] + 100]
        ops.attention_decode(q, single, kp, vp, table.to(DEV), pos, i32([0, 1, 2, 2]), i32(last), *args, max_kv_len=max(lens), **kw)
        got[bs] = out, single[last]
        # (rounding errors of a decode row: another order than the tiles', the same numbers)
        assert torch.allclose(single[last], out[last], rtol=2e-5, atol=2e-5)
    assert torch.isfinite(got[8][0]).all()
    for a, b in zip(got[8], got[7]):
        assert torch.allclose(a, b, rtol=2e-5, atol=2e-5), float((a - b).abs().max())


@pytest.mark.parametrize("hd", [64, 128])
@pytest.mark.parametrize("window,keep", [(0, 0), (50, 0), (130, 20), (300, 70)])
def test_float32_prompt_queries_have_the_same_bits_wherever_items_start(hd, window, keep):
    """Items that start at multiples of 64 and items that start anywhere give a query the same bits: tiles of 64 keys that all of a wave's rows
    see whole, which go without masks, beside tiles that some rows see in part or not at all, and tiles left out between kept keys and the
    window.  Against 64 bits: errors of sums of float32 products of up to `hd` and 512 terms."""
    from ferrox_amd import ops
    nh, nkv, n, bs = 4, 2, 512, 16
    q, k, v = rnd(n, nh * hd), rnd(n, nkv, hd, seed=1), rnd(n, nkv, hd, seed=2)
    i32 = lambda x: torch.tensor(x, dtype=torch.int32, device=DEV)
    kp = k.view(n // bs, bs, nkv, hd).transpose(1, 2).contiguous()
    vp = v.view(n // bs, bs, nkv, hd).permute(0, 2, 3, 1).contiguous()
    pos, table = torch.arange(n, dtype=torch.int32, device=DEV), i32([list(range(n // bs))])
    got = []
    for edges in (list(range(0, n + 1, 64)), [0, 1, 6, 63, 66, 128, 145, 209, 257, 321, 380, 444, 508, 512]):
        out = torch.zeros(n, nh * hd, device=DEV)
        starts, sizes = edges[:-1], [b - a for a, b in zip(edges, edges[1:])]
        ops.attention_tiles(q, out, kp, vp, table, pos, i32([0] * len(starts)), i32(starts), i32(sizes), nh, nkv, hd, bs, window,
                            hd ** -0.5, keep_first=keep)
        got.append(out)
    assert torch.equal(got[0], got[1])
    t = torch.arange(n, device=DEV)
    sees = t[None] <= t[:, None]
    if window:
        sees &= (t[:, None] - t[None] < window) | (t[None] < keep)
    qd, kd, vd = q.double().view(n, nh, hd), k.double().repeat_interleave(nh // nkv, 1), v.double().repeat_interleave(nh // nkv, 1)
    for h in range(nh):
        scores = (qd[:, h] @ kd[:, h].T * hd ** -0.5).masked_fill(~sees, -float("inf"))
        want = torch.softmax(scores, -1) @ vd[:, h]
        # a score's error, at most 2^-24 times a few of its roundings times |q||k| / sqrt(hd) < 2 sqrt(hd): 5e-6 of a probability, and
        # as much again for the sums, times values below 6
        assert float((got[0].view(n, nh, hd)[:, h].double() - want).abs().max()) < 6 * 1e-5


@pytest.mark.parametrize("hd", [20, 64, 80, 132])
def test_a_float32_key_at_minus_infinity_is_not_attended_to(hd):
    """A key whose last four numbers (the ones that stand in for numbers that a narrow head does not have) are minus infinity scores
    minus infinity with positive queries: weight 0 beside finite scores, as in the kernels for any shape (pages of 7 keys)."""
    from ferrox_amd import ops
    nh, n, at = 2, 150, 40
    q, k, v = rnd(n, nh * hd).abs() + 0.1, rnd(n, 1, hd, seed=1), rnd(n, 1, hd, seed=2)
    k[at, 0, hd - 4:] = -float("inf")
    i32 = lambda x: torch.tensor(x, dtype=torch.int32, device=DEV)
    pos, got = torch.arange(n, dtype=torch.int32, device=DEV), {}
    for bs in (8, 7):
        blocks = -(-n // bs)
        kp, vp = torch.zeros(blocks, 1, bs, hd, device=DEV), torch.zeros(blocks, 1, hd, bs, device=DEV)
        for t in range(blocks):
            rows = slice(t * bs, min((t + 1) * bs, n))
            kp[t, 0, :rows.stop - rows.start], vp[t, 0, :, :rows.stop - rows.start] = k[rows, 0], v[rows, 0].T
        table, args = i32([list(range(blocks))]), (nh, 1, hd, bs, 0, hd ** -0.5)
        out, single = torch.zeros(n, nh * hd, device=DEV), torch.zeros(n, nh * hd, device=DEV)
        ops.attention_tiles(q, out, kp, vp, table, pos, i32([0, 0, 0]), i32([0, 64, 128]), i32([64, 64, 22]), *args)
        ops.attention_decode(q, single, kp, vp, table, pos, i32([0]), i32([n - 1]), *args, max_kv_len=n)
        got[bs] = out, single[n - 1]
    for a, b in zip(got[8], got[7]):
        assert torch.isfinite(a).all() and torch.allclose(a, b, rtol=2e-5, atol=2e-5)


@pytest.mark.parametrize("nh,nkv,hd,vd", [(3, 3, 16, 16), (4, 1, 64, 64), (34, 2, 80, 48), (8, 4, 128, 128), (17, 1, 192, 256)])
def test_float32_single_queries_at_the_first_positions(nh, nkv, hd, vd):
    """Queries below position 24 (heads of 65 to 128) or 32 go a wave per head, the same bits as the kernel for any shape (pages of 7
    keys), whatever the step holds beside them and under whatever bound; from there on 16 heads of a group in a wave, equal up to roundings."""
    from ferrox_amd import ops
    n, at, few = 140, [0, 7, 23, 24, 31, 32, 127, 128, 139], 24 if 64 < max(hd, vd) <= 128 else 32
    q, k, v = rnd(n, nh * hd), rnd(n, nkv, hd, seed=1), rnd(n, nkv, vd, seed=2)
    i32 = lambda x: torch.tensor(x, dtype=torch.int32, device=DEV)
    pos = torch.arange(n, dtype=torch.int32, device=DEV)

    def run(bs, toks, bound):
        blocks = -(-n // bs)
        kp, vp = torch.zeros(blocks, nkv, bs, hd, device=DEV), torch.zeros(blocks, nkv, vd, bs, device=DEV)
        for t in range(blocks):
            rows = slice(t * bs, min((t + 1) * bs, n))
            kp[t, :, :rows.stop - rows.start], vp[t, :, :, :rows.stop - rows.start] = k[rows].transpose(0, 1), v[rows].permute(1, 2, 0)
        y = torch.full((n, nh * vd), float("nan"), device=DEV)
        ops.attention_decode(q, y, kp, vp, i32([list(range(blocks))]), pos, i32([0] * len(toks)), i32(toks), nh, nkv, hd, bs, 0, hd ** -0.5,
                             max_kv_len=bound, v_dim=vd)
        return y

    both, any_shape = run(8, at, n), run(7, at, n)
    for t in at:
        alone = run(8, [t], 1000)
        assert torch.equal(alone[t], both[t]), t
        assert torch.equal(both[t], any_shape[t]) if t < few else torch.allclose(both[t], any_shape[t], rtol=2e-5, atol=2e-5), t


@pytest.mark.parametrize("bs", [8, 7])
@pytest.mark.parametrize("longest", [128 * 7936, 128 * 7936 + 1, 128 * 8192, 128 * 8192 + 1, 128 * 16384])
def test_float32_single_queries_beside_a_very_long_sequence(bs, longest):
    """The chunks of a float32 sequence, hence its bits, do not depend on the longest sequence that a launch is told of: up to
    the most chunks that are merged, of which LDS holds the weights and sums of 7,936.  (bs 8: the matrix units; 7: any shape)"""
    from ferrox_amd import ops
    nh, hd, n = 2, 16, 700
    q, k, v = rnd(1, nh * hd), rnd(n, 1, hd, seed=1), rnd(n, 1, hd, seed=2)
    blocks = -(-n // bs)
    kp, vp = torch.zeros(blocks, 1, bs, hd, device=DEV), torch.zeros(blocks, 1, hd, bs, device=DEV)
    for t in range(blocks):
        rows = slice(t * bs, min((t + 1) * bs, n))
        kp[t, 0, :rows.stop - rows.start], vp[t, 0, :, :rows.stop - rows.start] = k[rows, 0], v[rows, 0].T
    i32 = lambda x: torch.tensor(x, dtype=torch.int32, device=DEV)
    table, out = i32([list(range(blocks))]), []
    for bound in (n, longest):
        y = torch.zeros(1, nh * hd, device=DEV)
        ops.attention_decode(q, y, kp, vp, table, i32([n - 1]), i32([0]), i32([0]), nh, 1, hd, bs, 0, hd ** -0.5, max_kv_len=bound)
        out.append(y)
    assert torch.equal(out[0], out[1])
    with pytest.raises(ops.KernelError):
        ops.attention_decode(q, y, kp, vp, table, i32([n - 1]), i32([0]), i32([0]), nh, 1, hd, bs, 0, hd ** -0.5, max_kv_len=128 * 16384 + 1)


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("chunks", [7921, 7936, 7937, 7960])
def test_merge_of_more_chunks_than_lds_holds(dtype, chunks):
    """A sequence of that many chunks of 64 keys, every one of them with a weight: the first, the last and one in the middle of those that LDS holds
    with the largest, so that chunks on both sides of what it holds decide the result."""
    from ferrox_amd import ops
    nh, hd, bs = 2, 16, 64
    n = 64 * chunks - 5
    q, k, v = rnd(1, hd, dtype=dtype).repeat(1, nh), rnd(chunks * bs, hd, dtype=dtype, seed=1), rnd(chunks * bs, hd, dtype=dtype, seed=2)
    for at, score in ((3, 15.0), (64 * 4000 + 7, 16.0), (n - 70, 15.5), (n - 10, 14.5), (n - 1, 16.0)):      # (the others' weights: the size of one of e^13.5)
        k[at] = (q[0, :hd].float() * (score * hd ** 0.5 / float((q[0, :hd].float() ** 2).sum()))).to(dtype)
    q[0, hd:] *= 0.95
    kp, vp = k.view(chunks, bs, hd)[:, None].contiguous(), v.view(chunks, bs, hd).transpose(1, 2)[:, None].contiguous()
    i32 = lambda x: torch.tensor(x, dtype=torch.int32, device=DEV)
    y = torch.zeros(1, nh * hd, dtype=dtype, device=DEV)
    ops.attention_decode(q, y, kp, vp, i32([list(range(chunks))]), i32([n - 1]), i32([0]), i32([0]), nh, 1, hd, bs, 0, hd ** -0.5, max_kv_len=n, chunk=64)
    sc = q.double().view(nh, hd) @ k[:n].double().T.contiguous() * hd ** -0.5
    p = torch.softmax(sc, -1)
    inside, beyond = p[:, :64 * 7900].sum(-1), p[:, n - 64:].sum(-1)
    assert bool((inside > 0.05).all()) and bool((beyond > 0.05).all())
    close(y.view(nh, hd), p @ v[:n].double(), dtype, f"{chunks} chunks")


@pytest.mark.parametrize("hd,bs,window", [(64, 16, 0), (64, 64, 0), (128, 64, 40000), (32, 16, 9000)])
def test_attention_over_more_pages_than_a_block_copies(hd, bs, window):
    """A sequence of more than 1024 pages (the kernels copy that many page ids into LDS and read the rest of
    the table from memory): its last 64 tokens as a block of queries, and its last token alone."""
    from ferrox_amd import ops
    nh, nkv, dtype = 2, 1, torch.bfloat16
    L = bs * 1030 + 5
    q, k, v, q_rot, k_pages, v_pages, table, pos, seq, toks = paged_setup(dtype, nh, nkv, hd, bs, [L], 1e6, hd, 1040)
    scale = 1.0 / math.sqrt(hd)
    kp, vp, tab = k_pages.double().cpu(), v_pages.double().cpu(), table.cpu()[0].long()
    ks = kp[tab].permute(0, 2, 1, 3).reshape(-1, nkv, hd)[:L]                  # [L, nkv, hd]
    vs = vp[tab].permute(0, 3, 1, 2).reshape(-1, nkv, hd)[:L]
    qs = q_rot[L - 64:].double().cpu().reshape(64, nh, hd)
    ref = torch.zeros(64, nh, hd, dtype=torch.float64)
    for i in range(64):
        p = L - 64 + i
        lo = max(0, p - window + 1) if window else 0
        for h in range(nh):
            sc = (ks[lo:p + 1, 0] @ qs[i, h]) * scale
            ref[i, h] = torch.softmax(sc, 0) @ vs[lo:p + 1, 0]
    ref = ref.reshape(64, nh * hd)
    i32 = lambda x: torch.tensor(x, dtype=torch.int32, device=DEV)
    out = torch.zeros(L, nh * hd, dtype=dtype, device=DEV)
    ops.attention_tiles(q_rot, out, k_pages, v_pages, table, pos, i32([0]), i32([L - 64]), i32([64]), nh, nkv, hd, bs, window, scale)
    close(out[L - 64:], ref, dtype, "tiled attention, last block")
    out2 = torch.zeros(L, nh * hd, dtype=dtype, device=DEV)
    for chunk in (None, 4096):
        ops.attention_decode(q_rot, out2, k_pages, v_pages, table, pos, i32([0]), i32([L - 1]), nh, nkv, hd, bs, window, scale,
                             max_kv_len=L, chunk=chunk)
        close(out2[L - 1], ref[63], dtype, f"decode attention chunk {chunk}")


@pytest.mark.parametrize("window", [0, 64 * 1027])
def test_waves_of_32_queries_over_more_pages_than_a_block_copies(window):
    """The last 131 tokens of a sequence of more than 1024 pages, in items of 128 on waves of 32 queries: the first pages' ids come from LDS, the last ones' from the table."""
    from ferrox_amd import debug, ops
    nh, nkv, hd, bs, n = 2, 1, 128, 64, 131
    L = bs * 1030 + 5
    q, k, v, q_rot, k_pages, v_pages, table, pos, seq, toks = paged_setup(torch.bfloat16, nh, nkv, hd, bs, [L], 1e6, hd, 1040)
    pages = table[0].long()
    ks, vs = k_pages[pages].permute(0, 2, 1, 3).reshape(-1, hd)[:L].double(), v_pages[pages].permute(0, 3, 1, 2).reshape(-1, hd)[:L].double()
    back = pos[L - n:, None] - pos[None]
    seen = (back >= 0) & (back < window) if window else back >= 0
    want = torch.zeros(n, nh, hd, dtype=torch.float64, device=DEV)
    for h in range(nh):
        sc = q_rot[L - n:, h * hd:(h + 1) * hd].double() @ ks.T.contiguous() * hd ** -0.5
        want[:, h] = torch.softmax(sc.masked_fill(~seen, -math.inf), -1) @ vs
    i32 = lambda x: torch.tensor(x, dtype=torch.int32, device=DEV)
    for groups in (1, 2):
        out = torch.zeros(L, nh * hd, dtype=torch.bfloat16, device=DEV)
        with debug.kernel_switch("attention", "rows32", 2), debug.kernel_switch("attention", "direct_groups", groups):
            ops.attention_tiles(q_rot, out, k_pages, v_pages, table, pos, i32([0, 0]), i32([L - n, L - 3]), i32([128, 3]), nh, nkv, hd, bs, window, hd ** -0.5, tile_q=128)
        close(out[L - n:], want.reshape(n, nh * hd), torch.bfloat16, f"{groups} group(s)")


def test_decode_attention_of_a_short_sequence_beside_a_very_long_one():
    """One launch, no window, two chunks: a sequence of 2,500 pages, whose chunks span more pages than a block
    copies into LDS (1024), beside one of 300 keys.  The short sequence's chunks lie far below the range of page
    ids that its blocks copy (the range is laid out for the launch's longest chunk before the position is known),
    so every one of its lookups goes to the table in memory; both against the plain attention."""
    from ferrox_amd import ops
    nh, nkv, hd, bs, dtype = 4, 2, 64, 16, torch.bfloat16
    lens = [40005, 300]
    n_pages = sum(-(-L // bs) for L in lens) + 3
    q, k, v, q_rot, k_pages, v_pages, table, pos, seq, toks = paged_setup(dtype, nh, nkv, hd, bs, lens, 1e6, hd, n_pages)
    scale = 1.0 / math.sqrt(hd)
    kp, vp = k_pages.double().cpu(), v_pages.double().cpu()
    last = [lens[0] - 1, lens[0] + lens[1] - 1]                               # token numbers of the two last positions
    out = torch.zeros(len(toks), nh * hd, dtype=dtype, device=DEV)
    i32 = lambda x: torch.tensor(x, dtype=torch.int32, device=DEV)
    chunk = 20032                                                             # 1,252 pages a chunk
    assert chunk // bs > 1024
    ops.attention_decode(q_rot, out, k_pages, v_pages, table, pos, i32([0, 1]), i32(last), nh, nkv, hd, bs, 0, scale,
                         max_kv_len=lens[0], chunk=chunk)
    for s_, L in enumerate(lens):
        tab = table.cpu()[s_].long()[: -(-L // bs)]
        ks = kp[tab].permute(0, 2, 1, 3).reshape(-1, nkv, hd)[:L]
        vs = vp[tab].permute(0, 3, 1, 2).reshape(-1, nkv, hd)[:L]
        qs = q_rot[last[s_]].double().cpu().reshape(nh, hd)
        ref = torch.stack([torch.softmax((ks[:, h // (nh // nkv)] @ qs[h]) * scale, 0) @ vs[:, h // (nh // nkv)] for h in range(nh)])
        close(out[last[s_]].reshape(nh, hd), ref, dtype, f"sequence of {L} keys")


def test_decode_attention_of_more_sequences_than_fill_the_cus_once():
    """20 sequences of 16 kv heads are 320 blocks for 256 CUs: the chunks are then chosen by how full the blocks' last
    round would be (eight a sequence here, one with 16 sequences), and sequences of every length, down to one key and
    up to the bound, must come out as plain attention gives them, with the chunks chosen and with one."""
    from ferrox_amd import ops
    nh, nkv, hd, bs, dtype = 16, 16, 64, 64, torch.bfloat16
    lens = [1100, 1, 64, 65, 1087, 1088, 1089, 700, 513, 128] * 2
    n_pages = sum(-(-L // bs) for L in lens) + 3
    q, k, v, q_rot, k_pages, v_pages, table, pos, seq, toks = paged_setup(dtype, nh, nkv, hd, bs, lens, 1e6, hd, n_pages)
    scale = 1.0 / math.sqrt(hd)
    kp, vp = k_pages.double().cpu(), v_pages.double().cpu()
    ends, last = 0, []
    for L in lens:
        ends += L
        last.append(ends - 1)
    i32 = lambda x: torch.tensor(x, dtype=torch.int32, device=DEV)
    outs = []
    for chunk in (None, 1152):
        out = torch.zeros(len(toks), nh * hd, dtype=dtype, device=DEV)
        ops.attention_decode(q_rot, out, k_pages, v_pages, table, pos, i32(list(range(len(lens)))), i32(last), nh, nkv, hd, bs, 0,
                             scale, max_kv_len=1152, chunk=chunk)
        outs.append(out)
    for s_, L in enumerate(lens):
        tab = table.cpu()[s_].long()[: -(-L // bs)]
        ks = kp[tab].permute(0, 2, 1, 3).reshape(-1, nkv, hd)[:L]
        vs = vp[tab].permute(0, 3, 1, 2).reshape(-1, nkv, hd)[:L]
        qs = q_rot[last[s_]].double().cpu().reshape(nh, hd)
        ref = torch.stack([torch.softmax((ks[:, h] @ qs[h]) * scale, 0) @ vs[:, h] for h in range(nh)])
        for out, what in zip(outs, ("chunks as chosen", "one chunk")):
            close(out[last[s_]].reshape(nh, hd), ref, dtype, f"sequence {s_} of {L} keys, {what}")


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("T,H,E,k,renorm", [(1, 64, 8, 2, False), (7, 96, 6, 3, True), (33, 200, 60, 4, False),
                                             (5, 128, 130, 8, True), (4, 72, 5, 5, False)])
def test_router(dtype, T, H, E, k, renorm):
    """router matrix product + selection, with the shared expert's gate as an extra row"""
    from ferrox_amd import ops
    x, wr, sg = rnd(T, H, dtype=dtype), rnd(E, H, dtype=dtype, seed=1, scale=0.3), rnd(H, dtype=dtype, seed=2, scale=0.2)
    logits = ops.gemm(x, torch.cat([wr, sg[None]]).contiguous(), epilogue=ops.EPI_STORE_F32)
    ids, w, gate = ops.router_select(logits, E, k, renorm, has_gate=True)
    xd, wd = x.double().cpu(), wr.double().cpu()
    for t in range(T):
        want_ids, want_w = plain.route_top_k(wd @ xd[t], k, renorm)
        assert ids[t].tolist() == want_ids, f"token {t}: experts {ids[t].tolist()} != {want_ids}"
        close(w[t], want_w, torch.float32, f"router weights token {t}")
    close(gate, torch.sigmoid(xd @ sg.double().cpu()), torch.float32, "shared gate")
    # the product the other way round (router rows as the short side), read through its transpose
    logits_t = ops.gemm(torch.cat([wr, sg[None]]).contiguous(), x, epilogue=ops.EPI_STORE_F32).t()
    assert logits_t.shape == logits.shape and logits_t.stride(1) != 1 or T == 1
    ids_t, w_t, gate_t = ops.router_select(logits_t, E, k, renorm, has_gate=True)
    assert torch.equal(ids_t, ids)
    close(w_t, w, torch.float32, "router weights from transposed logits")
    close(gate_t, gate, torch.float32, "shared gate from transposed logits")


def test_router_golden_vector():
    """logits 1..8, k=3, no renormalisation -> experts [7, 6, 5], weights [0.6323223, 0.2326232,
    0.0855683] (the vector of the reference's own test, ferrox-moe/src/lib.rs:863-893)."""
    from ferrox_amd import ops
    logits = torch.arange(1, 9, dtype=torch.float32, device=DEV)[None].contiguous()
    ids, w, _ = ops.router_select(logits, 8, 3, False)
    assert ids[0].tolist() == [7, 6, 5]
    assert torch.allclose(w[0].cpu(), torch.tensor([0.6323223, 0.2326232, 0.0855683]), atol=1e-4)   # its tolerance
    assert abs(float(w[0].sum()) - 0.9505138) < 1e-4
    exact = torch.softmax(torch.arange(1, 9, dtype=torch.float64), 0).flip(0)[:3]
    assert torch.allclose(w[0].cpu().double(), exact, atol=1e-6)
    ids, w, _ = ops.router_select(logits, 8, 3, True)              # renormalised: the same experts, sum 1
    assert ids[0].tolist() == [7, 6, 5] and abs(float(w[0].sum()) - 1.0) < 1e-6
    ids, w, _ = ops.router_select(torch.zeros(1, 8, device=DEV), 8, 3, True)     # all equal: lowest indices
    assert ids[0].tolist() == [0, 1, 2] and torch.allclose(w[0].cpu(), torch.full((3,), 1 / 3))
    ids, w, _ = ops.router_select(torch.tensor([[0.1, 5.0, 0.2, 3.0, -1.0]], device=DEV), 5, 2, False)
    assert ids[0].tolist() == [1, 3]                               # ferrox-moe/src/lib.rs:834-841


# xorshift64 started from a small number returns small numbers at first (the first uniform draw is 0, which picks
# the first token that has any probability whatever the logits say); the sampling tests start it high
SEED = 0x2545F4914F6CDD1D


def test_sampling_kernel():
    from ferrox_amd import ops
    V = 1000
    logits = rnd(6, V, scale=3.0)
    assert ops.sample(logits).tolist() == logits.argmax(-1).tolist()
    tie = torch.zeros(1, V, device=DEV)
    tie[0, [17, 400]] = 5.0
    assert ops.sample(tie).tolist() == [17]
    # seeded sampling against the plain sampler, option by option
    cases = [dict(temperature=0.8), dict(temperature=1.3, top_k=5), dict(temperature=0.7, top_p=0.6),
             dict(temperature=1.0, top_k=50, top_p=0.9, repetition_penalty=1.3),
             dict(temperature=0.0, repetition_penalty=2.0, presence_penalty=0.5, frequency_penalty=0.25),
             dict(temperature=0.9, top_k=1)]
    hist = [int(logits[0].argmax()), 3, 3, 999, int(logits[0].argmax())]
    draws = []
    for case in cases:
        picked = set()
        for trial in range(12):
            seed = SEED + (trial << 45)
            want = plain.sample(logits[0].double().cpu().tolist(), plain.XorShift64(seed), history=hist, **case)
            u = plain.XorShift64(seed).next_f32()
            draws.append(u)
            f = lambda v: torch.tensor([v], dtype=torch.float32, device=DEV)
            got = ops.sample(logits[:1], temperature=f(case.get("temperature", 0.0)), draw=f(u),
                             top_k=torch.tensor([case.get("top_k", 0)], dtype=torch.int32, device=DEV),
                             top_p=f(case.get("top_p", 1.0)), rep_penalty=f(case.get("repetition_penalty", 1.0)),
                             presence=f(case.get("presence_penalty", 0.0)), frequency=f(case.get("frequency_penalty", 0.0)),
                             hist=torch.tensor(hist, dtype=torch.int32, device=DEV),
                             hist_start=torch.tensor([0, len(hist)], dtype=torch.int32, device=DEV)).tolist()[0]
            assert got == want, f"{case} trial {trial}: kernel {got}, plain {want}"
            picked.add(got)
        if case["temperature"] > 0 and case.get("top_k", 0) != 1:
            assert len(picked) >= 3, f"{case}: twelve draws picked {sorted(picked)} only"
    assert min(draws) > 0.0 and max(draws) - min(draws) > 0.5, "the draws do not spread over (0, 1)"


def test_sampling_kernel_at_the_real_vocabulary():
    """V = 151,936, three rows in one call, eight draws each: the command line's defaults (top-k 40, top-p 0.95,
    repetition penalty 1.1: ferrox-cli/src/run.rs:52-64) and temperature alone, against the plain sampler
    (ferrox-models/src/sampling.rs:93-189).  A few dozen tokens stand out of the noise, as in a trained model, so
    that the most likely token has a probability near 0.2 and top-p cuts inside the top-k."""
    from ferrox_amd import ops
    V, R = 151936, 3
    g = torch.Generator().manual_seed(11)
    logits = torch.randn(R, V, generator=g) * 2.0
    for r in range(R):
        idx = torch.randperm(V, generator=g)[:30]
        logits[r, idx] += 5.0 + 3.0 * torch.rand(30, generator=g)
    rows = logits.double().tolist()
    dev = logits.to(DEV)
    assert ops.sample(dev).tolist() == logits.argmax(-1).tolist()
    hists = [[int(logits[0].argmax()), 7, 7, V - 1], [], [int(logits[2].argmax())] * 3 + [int(logits[2].topk(2).indices[1])]]
    flat = [t for h in hists for t in h]
    starts = [0]
    for h in hists:
        starts.append(starts[-1] + len(h))
    f = lambda v: torch.tensor(v, dtype=torch.float32, device=DEV)
    i32 = lambda v: torch.tensor(v, dtype=torch.int32, device=DEV)
    for case in (dict(temperature=0.8, top_k=40, top_p=0.95, repetition_penalty=1.1), dict(temperature=0.8)):
        gens = [plain.XorShift64(SEED + ((r + 1) << 45)) for r in range(R)]
        mirrors = [plain.XorShift64(SEED + ((r + 1) << 45)) for r in range(R)]
        picked = [set() for _ in range(R)]
        for draw in range(8):
            want = [plain.sample(rows[r], gens[r], history=hists[r], **case) for r in range(R)]
            u = [m.next_f32() for m in mirrors]
            got = ops.sample(dev, temperature=f([case["temperature"]] * R), draw=f(u), top_k=i32([case.get("top_k", 0)] * R),
                             top_p=f([case.get("top_p", 1.0)] * R), rep_penalty=f([case.get("repetition_penalty", 1.0)] * R),
                             presence=f([0.0] * R), frequency=f([0.0] * R), hist=i32(flat), hist_start=i32(starts)).tolist()
            assert got == want, f"{case} draw {draw}: kernel {got}, plain {want}"
            for r in range(R):
                picked[r].add(got[r])
        assert all(len(p) >= 3 for p in picked), f"{case}: eight draws picked {picked}"


@pytest.mark.parametrize("M,N,K", [(1, 6144, 2048), (8, 6144, 2048), (5, 100, 96), (16, 48, 264), (31, 257, 520),
                                    (32, 2560, 1792)])
@pytest.mark.parametrize("gamma_dtype", [torch.bfloat16, torch.float32])
def test_gemm_with_fused_norm(M, N, K, gamma_dtype):
    """RMSNorm applied inside the product against norm kernel + product and against the plain norm"""
    from ferrox_amd import ops
    h = rnd(M, K, scale=2.0)
    gamma = (1.0 + rnd(K, seed=3, scale=0.2)).to(gamma_dtype)
    w, bias = rnd(N, K, dtype=torch.bfloat16, seed=1, scale=0.05), rnd(N, dtype=torch.bfloat16, seed=2)
    eps = 1e-6
    assert ops.can_fuse_norm(h, w, M)
    got = ops.gemm(h, w, bias=bias, norm=(gamma, eps))
    two = ops.gemm(ops.rmsnorm(h, gamma, eps, torch.bfloat16), w, bias=bias)
    want = plain.rms_norm(h.double().cpu(), gamma.double().cpu(), eps) @ w.double().cpu().T + bias.double().cpu()
    close(got, want, torch.bfloat16, "fused norm product")
    close(two, want, torch.bfloat16, "norm, then product")
    assert not ops.can_fuse_norm(rnd(33, K), w, 33)


@pytest.mark.parametrize("T,H,E,k,renorm,has_gate", [(1, 2048, 60, 4, False, True), (8, 2048, 60, 4, False, True),
                                                      (16, 264, 7, 3, True, False), (5, 1792, 130, 8, True, True), (16, 2048, 60, 4, False, True),
                                                      (64, 2048, 60, 4, False, True), (33, 96, 6, 3, True, True),
                                                      (3, 64, 4, 4, False, True), (130, 1792, 60, 4, False, True),
                                                      (256, 264, 64, 8, True, True)])
def test_moe_front(T, H, E, k, renorm, has_gate):
    """norm + router products + selection + sort in one launch, twice in a row (the kernel's counter
    must be back at zero), against the plain norm and router on the rounded activations"""
    from ferrox_amd import ops
    h = rnd(T + 2, H, scale=1.5)[1:T + 1]                                    # a view that starts past row 0
    gamma = (1.0 + rnd(H, seed=3, scale=0.2)).to(torch.bfloat16)
    router = rnd(E + (1 if has_gate else 0), H, dtype=torch.bfloat16, seed=4, scale=0.3)
    eps = 1e-5
    x_sep = ops.rmsnorm(h.contiguous(), gamma, eps, torch.bfloat16)
    for rep in range(3):
        # the third time with the sort by expert in the same launch, and two pieces behind the experts
        got = ops.moe_front(h, gamma, eps, router, E, k, renorm, has_gate=has_gate, align=2 if rep == 2 else None)
        assert got is not None
        x, ids, w, gate, sort = got
        assert (sort is None) == (rep < 2)
        if sort is not None:
            for i, (mine, theirs) in enumerate(zip(sort, ops.moe_align(ids, E, always=2))):
                n_set = T * k if i == 3 else mine.numel()           # the inverse map covers the pairs only
                assert torch.equal(mine[:n_set], theirs[:n_set]), "the launch's own sort is that of moe_align"
        # the same formula as the norm kernel: at most the last float32 bit differs, which moves a
        # bfloat16 result only where it stands on a rounding boundary
        differ = x != x_sep
        assert int(differ.sum()) <= max(1, x.numel() // 10000), "the fused norm rounds like the norm kernel"
        assert bool(((x.float() - x_sep.float()).abs() <= x_sep.float().abs() * 2.0 ** -7).all())
        want_x = plain.rms_norm(h.double().cpu(), gamma.double().cpu(), eps)
        close(x, want_x, torch.bfloat16, "normed rows")
        logits = router.double().cpu() @ x.double().cpu().T                  # [E(+1), T]
        for t in range(T):
            want_ids, want_w = plain.route_top_k(logits[:E, t], k, renorm)
            assert ids[t].tolist() == want_ids, f"rep {rep} token {t}: experts {ids[t].tolist()} != {want_ids}"
            close(w[t], want_w, torch.float32, f"router weights token {t}")
        if has_gate:
            close(gate, torch.sigmoid(logits[E]), torch.float32, "shared gate")
    assert int(ops._counter(DEV).abs().sum()) == 0
    assert ops.moe_front(rnd(257, H), gamma, eps, router, E, k, renorm, has_gate=has_gate) is None     # too many rows


@pytest.mark.parametrize("T,E,k", [(5000, 60, 4), (3000, 700, 2), (1, 3, 1), (130, 1, 1), (2048, 60, 4), (701, 7, 3), (683, 5, 3)])
def test_sort_by_expert_at_large_sizes(T, E, k):
    """more pairs than one round of counters holds: rows of several groups; against a stable sort"""
    from ferrox_amd import ops
    g = torch.Generator().manual_seed(T + E)
    ids = torch.stack([torch.randperm(E, generator=g)[:k] for _ in range(T)]).to(torch.int32).to(DEV)
    offsets, sorted_token, sorted_pair, inv = ops.moe_align(ids, E)
    flat = ids.flatten().long().cpu()
    order = torch.sort(flat, stable=True).indices
    assert sorted_pair.cpu().tolist() == order.tolist()
    assert sorted_token.cpu().tolist() == (order // k).tolist()
    assert offsets.cpu().tolist() == [0] + torch.cumsum(torch.bincount(flat, minlength=E), 0).tolist()
    assert inv.cpu()[order].tolist() == list(range(T * k))


@pytest.mark.parametrize("T,E,k,S", [(24, 60, 4, 4), (64, 8, 2, 3), (17, 5, 1, 1), (40, 6, 3, 2)])
def test_sort_by_expert_with_experts_that_every_token_takes(T, E, k, S):
    """S further experts behind the sorted pairs, each with all T tokens as its rows (a shared expert cut into
    pieces), and the grouped products over that layout against one product per expert"""
    from ferrox_amd import ops
    g = torch.Generator().manual_seed(T + E)
    ids = torch.stack([torch.randperm(E, generator=g)[:k] for _ in range(T)]).to(torch.int32).to(DEV)
    plain_sort = ops.moe_align(ids, E)
    offsets, sorted_token, sorted_pair, _ = ops.moe_align(ids, E, always=S)
    n = T * k
    assert offsets.cpu().tolist() == plain_sort[0].cpu().tolist() + [n + (s + 1) * T for s in range(S)]
    assert sorted_token.cpu().tolist() == plain_sort[1].cpu().tolist() + list(range(T)) * S
    assert sorted_pair.cpu().tolist() == plain_sort[2].cpu().tolist() + list(range(n, n + S * T))
    H, I = 64, 32
    x = rnd(T, H, dtype=torch.bfloat16)
    w_gu, w_dn = rnd(E + S, 2 * I, H, dtype=torch.bfloat16, seed=1, scale=0.3), rnd(E + S, H, I, dtype=torch.bfloat16, seed=2, scale=0.3)
    act = ops.gemm(x, w_gu, epilogue=ops.EPI_GATED, a_rows=sorted_token, expert_offsets=offsets, n_rows=n + S * T)
    y = ops.gemm(act, w_dn, epilogue=ops.EPI_STORE_F32, expert_offsets=offsets, c_rows=sorted_pair)
    assert y.shape == (n + S * T, H)
    xd = x.double().cpu()
    for s_ in range(S):                      # piece s: every token through expert E + s
        e = E + s_
        a = (plain.silu(xd @ w_gu[e, :I].double().cpu().T) * (xd @ w_gu[e, I:].double().cpu().T)).to(torch.bfloat16).double()
        close(y[n + s_ * T:n + (s_ + 1) * T], a @ w_dn[e].double().cpu().T, torch.bfloat16, f"piece {s_}")
    t, j = 3 % T, k - 1                      # and a routed pair
    e = int(ids[t, j])
    a = (plain.silu(xd[t] @ w_gu[e, :I].double().cpu().T) * (xd[t] @ w_gu[e, I:].double().cpu().T)).to(torch.bfloat16).double()
    close(y[t * k + j], a @ w_dn[e].double().cpu().T, torch.bfloat16, "a routed pair")


@pytest.mark.parametrize("T,E,k", [(1, 8, 2), (8, 60, 4), (64, 60, 4), (33, 130, 8), (65, 6, 3), (300, 60, 4)])
def test_route_in_one_launch_equals_two(T, E, k):
    """selection and sort fused for small batches give what the two kernels give"""
    from ferrox_amd import ops
    logits = rnd(T, E + 1, scale=2.0)
    fused = ops.route(logits, E, k, True, has_gate=True)
    ids, w, gate = ops.router_select(logits, E, k, True, has_gate=True)
    two = (ids, w, gate) + ops.moe_align(ids, E)
    for a, b in zip(fused, two):
        assert torch.equal(a, b)


def test_tokens_fed_from_sampled_ids():
    """tokens[place] = ids[row] for the pairs given, everything else untouched; buffers of the wrong kind are refused"""
    from ferrox_amd import ops
    g = torch.Generator().manual_seed(3)
    tokens = torch.randint(0, 1000, (777,), generator=g, dtype=torch.int32)
    ids = torch.randint(0, 1000, (300,), generator=g, dtype=torch.int32)
    places = torch.randperm(777, generator=g)[:300]
    rows = torch.randint(0, 300, (300,), generator=g)
    expect = tokens.clone()
    expect[places] = ids[rows]
    d_tokens, pairs = tokens.cuda(), torch.stack([places, rows], 1).to(torch.int32).cuda()
    ops.feed_tokens(d_tokens, ids.cuda(), pairs, 777, 300)
    assert torch.equal(d_tokens.cpu(), expect)
    with pytest.raises(ops.KernelError):
        ops.feed_tokens(d_tokens, ids.cuda().long(), pairs, 777, 300)
    with pytest.raises(ops.KernelError):
        ops.feed_tokens(d_tokens, ids.cuda(), pairs, 778, 300)


@pytest.mark.parametrize("T,E,k,I,H", [(40, 4, 2, 64, 128), (100, 4, 2, 128, 192), (24, 6, 3, 64, 64)])
def test_sorted_experts_through_either_product(T, E, k, I, H):
    """rows sorted by expert, more than three an expert: the tiled product takes them by itself; the product for few
    rows, told to (it takes up to 64 rows an expert), gives the same activations and outputs up to rounding, and
    both agree with per-token loops"""
    from ferrox_amd import debug, ops
    dtype = torch.bfloat16
    x = rnd(T, H, dtype=dtype)
    w_gu, w_dn = rnd(E, 2 * I, H, dtype=dtype, seed=1, scale=0.3), rnd(E, H, I, dtype=dtype, seed=2, scale=0.3)
    g = torch.Generator().manual_seed(7)
    ids = torch.stack([torch.randperm(E, generator=g)[:k] for _ in range(T)]).to(torch.int32).to(DEV)
    offsets, sorted_token, sorted_pair, inv = ops.moe_align(ids, E)
    xd, gud, dnd = x.double().cpu(), w_gu.double().cpu(), w_dn.double().cpu()
    ref = torch.zeros(T * k, H, dtype=torch.float64)
    for t in range(T):
        for j in range(k):
            e = int(ids[t, j])
            a = (plain.silu(xd[t] @ gud[e, :I].T) * (xd[t] @ gud[e, I:].T)).to(torch.bfloat16).double()
            ref[t * k + j] = a @ dnd[e].T
    outs = []
    for few in (3, 64):
        with debug.kernel_switch("gemm", "few_rows", few):
            act = ops.gemm(x, w_gu, epilogue=ops.EPI_GATED, a_rows=sorted_token, expert_offsets=offsets, n_rows=T * k)
            y = ops.gemm(act, w_dn, epilogue=ops.EPI_STORE_F32, expert_offsets=offsets, c_rows=sorted_pair)
        close(y, ref, dtype, f"sorted experts, few_rows {few}", k=I)
        outs.append(y)
    assert float((outs[0] - outs[1]).abs().max()) <= 2e-2 * float(ref.abs().max())


@pytest.mark.parametrize("D", [33, 64, 100, 128, 129, 256])
def test_delta_rule_adds_a_column_in_one_order(D):
    """One number per lane, queries of ones and nothing written: the output is the sum over a column's lanes alone.  Its bits are
    those of the tree: four exchanges inside each row of 16 lanes, 8, 4, 2 and 1 apart, then the two rows of 32."""
    from ferrox_amd import ops
    V, lanes, per_lane = 40, 16 if D <= 64 else 32, 4 if D <= 128 else 8
    one = lambda *s: torch.ones(s, device=DEV)
    held = torch.zeros(1, 1, V, D, device=DEV)
    held[..., ::per_lane] = rnd(1, 1, V, -(-D // per_lane), seed=6) * torch.exp(4 * rnd(1, 1, V, -(-D // per_lane), seed=7))
    tree = torch.zeros(V, lanes)
    tree[:, :-(-D // per_lane)] = held[0, 0, :, ::per_lane].cpu()
    tree = tree.view(V, lanes // 16, 16)
    for apart in (8, 4, 2, 1):
        tree = tree[..., :apart] + tree[..., apart:2 * apart]
    want = tree.sum(1)[:, 0] if lanes == 16 else tree[:, 0, 0] + tree[:, 1, 0]
    state = held.clone()
    out = ops.channel_delta(one(1, D), one(1, D), one(1, D), 0 * one(1, 1), 0 * one(1, 1), 0 * one(1, V), state,
                            torch.tensor([0, 1], dtype=torch.int32, device=DEV), torch.zeros(1, dtype=torch.int32, device=DEV), 1, 1, 1, D, V)
    assert torch.equal(out.cpu().view(V), want) and torch.equal(state, held)


# one case per instance of the kernel: 16 and 32 lanes a column, whole pieces of four rows and single ones, columns and rows past the end
@pytest.mark.parametrize("D,V,H,G", [(64, 32, 2, 1), (64, 48, 2, 2), (33, 20, 2, 1), (30, 70, 1, 1), (128, 128, 4, 2), (100, 30, 2, 2), (66, 9, 2, 2),
                                     (256, 24, 2, 1), (129, 17, 1, 1)])
def test_delta_rule_at_every_length_of_a_group(D, V, H, G):
    """Tokens travel in groups of eight, two groups ahead: lengths that end inside the first, second and third group, side by
    side, and the same sequences cut in two.  Sums of up to 256 terms in float32: 1e-6 of a result's norm is ten times what is seen."""
    from ferrox_amd import ops
    lengths = [1, 7, 8, 9, 16, 17, 24, 31]
    T, n = sum(lengths), len(lengths)
    q, k = rnd(T, G, D), rnd(T, G, D, seed=1)
    q, k = q / q.norm(dim=-1, keepdim=True), k / k.norm(dim=-1, keepdim=True)
    decay, beta, v = torch.exp(-0.2 * rnd(T, H, D, seed=2).abs()), torch.sigmoid(rnd(T, H, seed=3)), rnd(T, H * V + 3, seed=4)[:, :H * V]
    kq, before = (k * q).sum(-1), rnd(n, H, V, D, seed=5)
    flat = lambda x, lo, hi: x[lo:hi].reshape(hi - lo, -1).contiguous()

    def run(lo, hi, starts, slots, state):
        return ops.channel_delta(flat(q, lo, hi), flat(k, lo, hi), flat(decay, lo, hi), flat(beta, lo, hi), flat(kq, lo, hi), v[lo:hi], state,
                                 torch.tensor(starts, dtype=torch.int32, device=DEV), torch.tensor(slots, dtype=torch.int32, device=DEV), len(slots), H, G, D, V)

    at = [sum(lengths[:i]) for i in range(n + 1)]
    state = before.clone()
    out = run(0, T, at, list(range(n)), state)
    for i in range(n):
        S = before[i].double().transpose(1, 2)
        want = torch.empty(lengths[i], H, V, dtype=torch.float64, device=DEV)
        for t in range(at[i], at[i + 1]):
            kt, qt = (x[t].double().repeat_interleave(H // G, 0)[..., None] for x in (k, q))
            S = decay[t].double()[..., None] * S
            u = beta[t].double()[:, None] * (v[t].double().view(H, V) - (S * kt).sum(1))
            S = S + kt * u[:, None]
            want[t - at[i]] = (S * qt).sum(1)
        got = out[at[i]:at[i + 1]].double().view(-1, H, V)
        assert (got - want).norm() < 1e-6 * want.norm() and (state[i].double().transpose(1, 2) - S).norm() < 1e-6 * S.norm(), lengths[i]
        # in two portions: the same bits
        cut, part = lengths[i] // 2, before.clone()
        halves = [run(lo, hi, [0, hi - lo], [i], part) for lo, hi in ((at[i], at[i] + cut), (at[i] + cut, at[i + 1])) if hi > lo]
        assert torch.equal(torch.cat(halves), out[at[i]:at[i + 1]]) and torch.equal(part[i], state[i]), lengths[i]


@pytest.mark.parametrize("M", [1, 4, 5, 16])
@pytest.mark.parametrize("N2,K2,epi2", [(256, 128, 0), (1024, 2048, 1), (4096, 512, 0), (5120, 512, 1), (24, 64, 0)])
def test_pairs_of_few_row_products_have_the_bits_of_two_launches(M, N2, K2, epi2):
    """Gate/up and a product stored in float32, each beside a stored one in half sets, whole sets and two of them, with the pairs of its heads turned and without; and
    what adds the second one's rows behind its own: the bits of two additions."""
    from ferrox_amd import ops
    x, w_gu, w_down = rnd(M, 2048, dtype=torch.bfloat16), rnd(2 * 5632, 2048, dtype=torch.bfloat16, seed=1, scale=0.02), rnd(2048, 5632, dtype=torch.bfloat16, seed=2, scale=0.02)
    y, w2 = rnd(M, K2, dtype=torch.bfloat16, seed=3), rnd(N2, K2, dtype=torch.bfloat16, seed=4, scale=0.1)
    h0, scale = rnd(M, 2048, seed=5), rnd(M, seed=6)
    heads = 4
    width = N2 // heads
    first_dim = width // 4 * 2
    n_dims = min(first_dim, 64)             # (the rotation by itself takes up to 256)
    positions, inv_freq = torch.randint(0, 30000, (M,), device=DEV, dtype=torch.int32), torch.rand(n_dims // 2, device=DEV)
    def stored():
        return torch.full((M, N2 + 8), 7.0, dtype=torch.bfloat16 if epi2 == 0 else torch.float32, device=DEV)
    act, h = ops.gemm(x, w_gu, epilogue=ops.EPI_GATED, activation="gelu_tanh"), h0.clone()
    w_out = rnd(2048, 2048, dtype=torch.bfloat16, seed=7, scale=0.02)
    for row_scale in (None, scale):
        h, both = h0.clone(), h0.clone()
        ops.gemm(x, w_out, epilogue=ops.EPI_RESID, out=h, row_scale=row_scale)
        ops.gemm(act, w_down, epilogue=ops.EPI_RESID, out=h)
        ops.gemm(x, w_out, epilogue=ops.EPI_RESID, out=both, row_scale=row_scale, then_add=ops.gemm(act, w_down, epilogue=ops.EPI_STORE_F32))
        assert torch.equal(both, h)
    down = ops.gemm(act, w_down, epilogue=ops.EPI_STORE_F32)
    for bad in (dict(epilogue=ops.EPI_STORE_F32, then_add=down), dict(epilogue=ops.EPI_RESID, out=h, then_add=down[:, :2047]), dict(epilogue=ops.EPI_RESID, out=h, then_add=down.bfloat16()),
                dict(epilogue=ops.EPI_RESID, out=h, then_add=down.cpu()), dict(epilogue=ops.EPI_RESID, out=h, then_add=down[:M - 1])):
        with pytest.raises(ops.KernelError):
            ops.gemm(x, w_out, **bad)
    with pytest.raises(ops.KernelError):
        ops.gemm(rnd(17, 2048, dtype=torch.bfloat16), w_out, epilogue=ops.EPI_RESID, out=rnd(17, 2048), then_add=rnd(17, 2048))
    plain2 = ops.gemm(y, w2, epilogue=epi2)
    for turn in (None, (positions, inv_freq, width, first_dim, n_dims, 1.25)) if epi2 == 0 else (None,):
        want = plain2.clone()
        if turn is not None:
            ops.latent_q_rot(want, want, positions, heads, first_dim, width - first_dim, n_dims, first_dim, inv_freq, 1.25)
        got_act, got_down, one, two = torch.full((M, 5632), 7.0, dtype=torch.bfloat16, device=DEV), torch.empty_like(down), stored(), stored()
        first = ops.Product(x, w_gu, got_act, ops.EPI_GATED, "gelu_tanh")
        ops.gemm_pair(first, ops.Product(y, w2, one[:, :N2], epi2, turn=turn))
        ops.gemm_pair(ops.Product(got_act, w_down, got_down, ops.EPI_STORE_F32), ops.Product(y, w2, two[:, :N2], epi2, turn=turn))
        assert torch.equal(got_act, act) and torch.equal(got_down, down)
        for out in (one, two):
            assert torch.equal(out[:, :N2], want) and bool((out[:, N2:] == 7).all()), turn is not None
    assert not ops.can_pair(first, ops.Product(y[:, 1:], w2[:, 1:], one, epi2)) and not ops.can_pair(first, ops.Product(y.float(), w2.float(), one, epi2))
    with pytest.raises(ops.KernelError):
        ops.gemm_pair(first, ops.Product(y, w2, h0, ops.EPI_RESID))


@pytest.mark.parametrize("nh,nkv,hd,vd", [(5, 1, 64, 64), (16, 1, 256, 192), (34, 2, 64, 40), (7, 7, 128, 72), (28, 4, 128, 128), (16, 1, 256, 200)])
@pytest.mark.parametrize("bs", [64, 16, 128, 96])
def test_single_queries_of_one_wave_write_their_rows_and_columns_only(nh, nkv, hd, vd, bs):
    """Blocks of one wave store through a buffer whose end drops what a block does not have: heads beyond the group, columns beyond the
    value head, in outputs and in parts of several chunks.  Whatever stands around the outputs stays.  Probabilities and values are
    rounded to bfloat16, and so is the output: 3 x 2^-9 of the largest value."""
    from ferrox_amd import ops
    lens = [1, 40, 64, 150]
    blocks = [-(-n // bs) for n in lens]
    g = torch.Generator().manual_seed(3)
    ids = torch.randperm(sum(blocks) + 2, generator=g)
    kp = rnd(len(ids), nkv, bs, hd, dtype=torch.bfloat16)
    vp = rnd(len(ids), nkv, vd, bs, dtype=torch.bfloat16, seed=1)
    table, used = torch.zeros(len(lens), max(blocks), dtype=torch.int32), 0
    for s, n in enumerate(blocks):
        table[s, :n] = ids[used:used + n].to(torch.int32)
        used += n
    q = rnd(len(lens), nh * hd, dtype=torch.bfloat16, seed=2)
    i32 = lambda x: torch.tensor(x, dtype=torch.int32, device=DEV)
    for most in (64, 150):      # keys: one chunk of 64, whose block writes the output, and three, whose blocks write parts
        around = torch.full((len(lens) + 2, nh * vd + 16), 7.0, dtype=torch.bfloat16, device=DEV)
        out = around[1:-1, 8:-8]
        ops.attention_decode(q, out, kp, vp, table.to(DEV), i32([min(n, most) - 1 for n in lens]), i32([0, 1, 2, 3]), i32([0, 1, 2, 3]), nh, nkv, hd,
                             bs, 0, hd ** -0.5, max_kv_len=most, chunk=64, v_dim=vd)
        edge = around.clone()
        edge[1:-1, 8:-8] = 7.0
        assert bool((edge == 7.0).all())
        for s, n in enumerate(lens):
            n = min(n, most)
            k = kp[table[s].long().to(DEV)].transpose(1, 2).reshape(-1, nkv, hd)[:n].double().repeat_interleave(nh // nkv, 1)
            v = vp[table[s].long().to(DEV)].permute(0, 3, 1, 2).reshape(-1, nkv, vd)[:n].double().repeat_interleave(nh // nkv, 1)
            p = torch.softmax((q[s].double().view(nh, 1, hd) * k.transpose(0, 1)).sum(-1) * hd ** -0.5, -1)
            want = (p[..., None] * v.transpose(0, 1)).sum(1)
            assert float((out[s].reshape(nh, vd).double() - want).abs().max()) <= 3 * 2 ** -9 * float(v.abs().max()), (s, most)


@pytest.mark.parametrize("waves", [2, 3, 4])
@pytest.mark.parametrize("nh,nkv,hd", [(16, 16, 128), (28, 4, 128), (16, 4, 64), (8, 1, 256)])
def test_an_infinite_value_stays_infinite_in_the_merge_of_a_blocks_waves(nh, nkv, hd, waves):
    """A value of infinity in the keys of the first, a middle and the last of a block's waves, of which there are two and more: the outputs that take
    it are infinite, and all others are as without it."""
    from ferrox_amd import ops
    bs, lens = 64, [129, 200, 300, 500]
    per = 8
    i32 = lambda x: torch.tensor(x, dtype=torch.int32, device=DEV)
    table = torch.randperm(len(lens) * per, generator=torch.Generator().manual_seed(2)).to(torch.int32).view(len(lens), per).to(DEV)
    kp = rnd(len(lens) * per, nkv, bs, hd, dtype=torch.bfloat16)
    vp = rnd(len(lens) * per, nkv, hd, bs, dtype=torch.bfloat16, seed=1)
    q = rnd(len(lens), nh * hd, dtype=torch.bfloat16, seed=2, scale=0.05)          # (no probability is near nothing)
    def run(values):
        out = torch.zeros(len(lens), nh * hd, dtype=torch.bfloat16, device=DEV)
        ops.attention_decode(q, out, kp, values, table, i32([n - 1 for n in lens]), i32([0, 1, 2, 3]), i32([0, 1, 2, 3]), nh, nkv, hd, bs, 0,
                             hd ** -0.5, max_kv_len=512, chunk=512, waves=waves)
        return out.view(len(lens), nkv, nh // nkv, hd)
    clean = run(vp)
    assert torch.isfinite(clean).all()
    for place in (lambda n: 0, lambda n: 70, lambda n: n // 2, lambda n: n - 1):
        bad = vp.clone()
        for s, n in enumerate(lens):
            t = place(n)
            bad[table[s, t // bs].long(), nkv - 1, 5, t % bs] = math.inf
        got, want = run(bad), clean.clone()
        want[:, nkv - 1, :, 5] = math.inf
        assert torch.equal(got, want)


@pytest.mark.parametrize("dtype,decoded,prompts", [(torch.bfloat16, 0, [1030]), (torch.bfloat16, 13, [700, 0, 345]), (torch.bfloat16, 1024, []),
                                                   (torch.float32, 0, [260]), (torch.float32, 6, [131, 3, 140])])
@pytest.mark.parametrize("nkv,vd,bs", [(16, 128, 64), (11, 192, 16), (16, 136, 20), (8, 264, 24)])
def test_values_of_many_tokens_go_to_their_places(dtype, decoded, prompts, nkv, vd, bs):
    """A step whose values go out in windows of 64 tokens: prompts that start at any token and any slot of a page, sequences of single
    tokens, pages that hold a whole number of 16-byte pieces and (20) such that do not.  Every value is where its position says, and nothing else is written."""
    from ferrox_amd import ops
    starts = [5 * i % 61 for i in range(decoded)] + [37 * i for i in range(len(prompts))]
    lens = [1] * decoded + prompts
    seqs = [s for s, n in enumerate(lens) for _ in range(n)]
    poss = [starts[s] + i for s, n in enumerate(lens) for i in range(n)]
    T, per = len(seqs), max(poss) // bs + 1
    assert T * nkv * vd >= (1 << 21 if dtype == torch.bfloat16 else 1 << 19)
    i32 = lambda x: torch.tensor(x, dtype=torch.int32, device=DEV)
    table = torch.randperm(len(lens) * per, generator=torch.Generator().manual_seed(1)).to(torch.int32).view(len(lens), per).to(DEV)
    hd = 32
    buf = rnd(T, 2 * nkv * hd + nkv * vd, dtype=dtype)
    q, k, v = buf[:, :nkv * hd], buf[:, nkv * hd:2 * nkv * hd], buf[:, 2 * nkv * hd:]
    k_pages = torch.zeros(len(lens) * per, nkv, bs, hd, dtype=dtype, device=DEV)
    v_pages = torch.full((len(lens) * per, nkv, vd, bs), 9.0, dtype=dtype, device=DEV)
    want = v_pages.clone()
    at, slot = table[seqs, [p // bs for p in poss]].long(), torch.tensor([p % bs for p in poss], device=DEV)
    want[at, :, :, slot] = v.reshape(T, nkv, vd)
    ops.rope_kv_write(q, k, v, i32(poss), i32(seqs), table, k_pages, v_pages, nkv, nkv, hd, bs, hd, 1e4, v_dim=vd)
    assert torch.equal(v_pages, want)


@pytest.mark.parametrize("M", [33, 49, 64])
@pytest.mark.parametrize("N,K,epi", [(6144, 2048, 0), (5184, 200, 0), (5200, 1192, 1), (5120, 640, 2), (12288, 128, 1), (2560, 1416, 3)])
def test_products_of_four_row_tiles_have_the_bits_of_one(M, N, K, epi):
    """33 to 64 rows in blocks of four row tiles and two sets of weight rows, with one piece of K a wave, several, a last part of one and waves
    without any: the bits of the same rows sixteen at a time."""
    from ferrox_amd import ops
    a = rnd(M, K, dtype=torch.bfloat16)
    w = rnd(N * (2 if epi == ops.EPI_GATED else 1), K, dtype=torch.bfloat16, seed=1, scale=0.05)
    dtype = torch.bfloat16 if epi in (ops.EPI_STORE, ops.EPI_GATED) else torch.float32
    whole = rnd(M, N, dtype=dtype, seed=2)
    parts = whole.clone()
    ops.gemm(a, w, epilogue=epi, out=whole)
    for m in range(0, M, 16):
        ops.gemm(a[m:m + 16], w, epilogue=epi, out=parts[m:m + 16])
    assert torch.equal(whole, parts)


@pytest.mark.parametrize("K", [96, 1056, 2112])
@pytest.mark.parametrize("N", [8, 264, 2056])
def test_few_float32_rows_from_parts_in_whole_lines_and_in_half(N, K):
    """The product for few rows fetches up to eight rows of a tile with one load of whole lines and more with two: at 7, 8, 9, 15, 16, 17 and 25 rows, plain
    and of experts with so many, the bits of tiles."""
    from ferrox_amd import debug, ops
    a, w = rnd(34, K), torch.stack([rnd(2 * N, K, seed=1), rnd(2 * N, K, seed=2)])
    with debug.kernel_switch("gemm", "f32_split", 1):
        for kw, some in ((dict(epilogue=ops.EPI_STORE_F32), lambda x: x[..., :N, :].contiguous()), (dict(epilogue=ops.EPI_GATED), lambda x: x)):
            one, both = some(w[0]), some(w)
            with debug.kernel_switch("gemm", "f32_tile", 32):
                want, other = ops.gemm(a, one, **kw), ops.gemm(a, some(w[1]), **kw)
            for rows in (1, 7, 8, 9, 15, 16, 17, 25, 32):
                offsets = torch.tensor([0, rows, 34], dtype=torch.int32, device=DEV)
                for half in (-1, 0, 1) if rows <= 16 else (-1,):
                    with debug.kernel_switch("gemm", "f32_tile", 1), debug.kernel_switch("gemm", "skinny_half", half):
                        assert torch.equal(ops.gemm(a[:rows], one, **kw), want[:rows]), (rows, half)
                with debug.kernel_switch("gemm", "f32_tile", 1):
                    got = ops.gemm(a, both, expert_offsets=offsets, n_rows=34, **kw)
                assert torch.equal(got[:rows], want[:rows]) and torch.equal(got[rows:], other[rows:]), rows


@pytest.mark.parametrize("K", [96, 128, 160, 192])
@pytest.mark.parametrize("shares,stream", [((0, 1, 17, 8, 0, 12, 5, 3), 2), ((0, 1, 49, 0, 3, 17, 0, 26), 2), ((0, 1, 17, 49, 64, 3, 5, 30), 1), ((65, 0, 1, 17, 0, 49, 3, 50), 1),
                                            ((130, 65, 64, 63, 0, 1, 17, 49), 0)])
def test_float32_experts_from_parts_with_their_weights_in_whole_lines(K, shares, stream):
    """Rows sorted by expert in tiles of 64: up to 12 rows an expert on average with whole lines two stages ahead, up to 24 one stage, beyond without; shares at the edges of row blocks
    and tiles, none at all, every number of steps beside the stages.  The bits of the product for few rows, also beside operands that are not finite."""
    from ferrox_amd import debug, ops
    E, N, M = len(shares), 136, sum(shares)
    average = -(-M // E)
    assert (2 if average <= 12 else 1 if average <= 24 else 0) == stream
    a, w = rnd(M, K), rnd(E, 2 * N, K, seed=1)
    bad_a, bad_w = a.clone(), w.clone()
    bad_a[M // 2, 5], bad_a[M - 1, K - 1], bad_w[2, 17, 3], bad_w[5, N + 30, 0] = math.inf, math.nan, -math.inf, math.nan
    offsets = torch.tensor([sum(shares[:e]) for e in range(E + 1)], dtype=torch.int32, device=DEV)
    for x, weights in ((a, w), (bad_a, bad_w)):
        for kw, some in ((dict(epilogue=ops.EPI_STORE_F32), lambda t: t[:, :N].contiguous()), (dict(epilogue=ops.EPI_GATED), lambda t: t)):
            got = {}
            for split, tile in ((1, 1), (1, 0), (1, 64), (1, 128), (0, 0)):
                with debug.kernel_switch("gemm", "f32_split", split), debug.kernel_switch("gemm", "f32_tile", tile):
                    got[split, tile] = torch.nan_to_num(ops.gemm(x, some(weights), expert_offsets=offsets, n_rows=M, **kw), nan=7e30, posinf=8e30, neginf=-8e30)
            for tile in (0, 64, 128):
                assert torch.equal(got[1, tile], got[1, 1]), (tile, kw)
            odd = got[0, 0].abs() > 1e30
            assert torch.equal(got[1, 1][odd], got[0, 0][odd])
            close(got[1, 1][~odd], got[0, 0][~odd], torch.float32, "float32 instruction")


@pytest.mark.parametrize("nh,nkv,hd", [(16, 16, 64), (16, 16, 128), (28, 4, 128), (12, 12, 48), (8, 1, 256)])
@pytest.mark.parametrize("S,longest", [(3, 1300), (72, 1300), (70, 150)])
@pytest.mark.parametrize("window,keep,softcap", [(0, 0, 0.0), (300, 0, 0.0), (200, 70, 0.0), (0, 0, 20.0)])
def test_single_queries_on_pages_that_hold_whole_tiles(nh, nkv, hd, S, longest, window, keep, softcap):
    """Pages of 64 and 128 positions, where a tile of keys has one page, against pages of 16, where every key has its own: the same bits, in waves that walk
    one tile and many.  What no query may see, the other positions of a sequence's pages, is not a number."""
    from ferrox_amd import ops
    lens = [max(1, longest - (53 * i) % longest) for i in range(S)]
    i32 = lambda x: torch.tensor(x, dtype=torch.int32, device=DEV)
    width = -(-longest // 128) * 128
    t = torch.arange(width, device=DEV)[None]
    n = torch.tensor(lens, device=DEV)[:, None]
    sees = (t < n) & ((t >= n - window) | (t < keep) if window else t >= 0)
    k, v = rnd(S, width, nkv, hd, dtype=torch.bfloat16), rnd(S, width, nkv, hd, dtype=torch.bfloat16, seed=1)
    k[~sees], v[~sees] = math.nan, math.nan
    q = rnd(S, nh * hd, dtype=torch.bfloat16, seed=2)
    got = []
    for bs in (16, 64, 128):
        per = width // bs
        table = torch.randperm(S * per, generator=torch.Generator().manual_seed(bs)).to(DEV)
        kp = torch.empty(S * per, nkv, bs, hd, dtype=torch.bfloat16, device=DEV)
        vp = torch.empty(S * per, nkv, hd, bs, dtype=torch.bfloat16, device=DEV)
        kp[table] = k.view(S * per, bs, nkv, hd).transpose(1, 2)
        vp[table] = v.view(S * per, bs, nkv, hd).permute(0, 2, 3, 1)
        out = torch.zeros(S, nh * hd, dtype=torch.bfloat16, device=DEV)
        seqs = i32(list(range(S)))
        ops.attention_decode(q, out, kp, vp, table.to(torch.int32).view(S, per), i32([m - 1 for m in lens]), seqs, seqs, nh, nkv, hd, bs, window, hd ** -0.5,
                             max_kv_len=longest, keep_first=keep, softcap=softcap)
        got.append(out)
    assert torch.isfinite(got[0]).all() and torch.equal(got[0], got[1]) and torch.equal(got[0], got[2])
