"""The wide matrix-core kernels (batches and expert groups): every cell is the
matvec's, bit for bit, in every launch shape, at the edges of its tiles, token columns and K parts."""
import numpy as np
import pytest

import oracle
from camelid_amd import binding as B
from camelid_amd.binding import DeviceBuffer, Weight, check, lib
from tests import gpu_util as G
from tests.test_gpu_moe import gpu_moe, gpu_route

pytestmark = pytest.mark.gpu

K_FORMATS = [("Q4_K", B.CML_Q4_K, "q4k"), ("Q6_K", B.CML_Q6_K, "q6k")]
SHAPES = [(g, waves) for g in (1, 2, 3, 4, 5, 6, 7, 8) for waves in (4, 8)]


def activations(n: int, cols: int, seed: int):
    x = np.random.default_rng(seed).standard_normal((n, cols)).astype(np.float32)
    x[0] = 0.0
    x[-1, :256] = -np.abs(x[-1, :256]).max() * 4  # a super-block at the negative extreme
    return oracle.quantize_activation(B.CML_Q4_K, x)


# rows below a tile, a tile, past one; one super-block per row; K cut two ways (even and uneven parts), four ways (even and uneven)
@pytest.mark.parametrize("rows,cols", [(1, 256), (16, 768), (130, 1280), (300, 2048), (145, 13 * 256), (300, 4096), (100, 18 * 256)])
@pytest.mark.parametrize("name,fmt,tag", K_FORMATS)
def test_wide_cells_are_bitwise_the_gemv(name, fmt, tag, rows, cols):
    wire = G.synth_weight(fmt, rows, cols, seed=rows + cols)
    w = Weight.upload(fmt, rows, cols, wire)
    cut = {1: 1, 3: 1, 5: 1, 8: 2, 13: 2, 16: 4, 18: 4}[cols // 256]  # the matvec's K cut of these rows
    for n in (3, 16, 17, 47, 130):
        s, q = activations(n, cols, seed=n)
        with G.env(CAMELID_HIP_MFMA_WIDE=0), G.engaged(none=(r"\.wide\.",)):
            ref = G.gpu_gemm(w, s, q)
        for g, waves in SHAPES:
            if n < 16 * (g - 1) and n != 3:
                continue
            for parts in (1, 2):
                if (name, g, waves, parts) == ("Q4_K", 8, 8, 2):
                    continue  # does not fit a compute unit's LDS
                two = parts == 2 and cut > 1
                walk = (r"\.ksplit2" if two else "") + (r"\.serial_split" if cut > (2 if two else 1) else "")
                G.say(f"wide {name} {rows}x{cols} n={n} groups={g} waves={waves} parts={parts}")
                with G.env(CAMELID_HIP_MFMA_WIDE=2, CAMELID_HIP_WIDE_GROUPS=g, CAMELID_HIP_WIDE_WAVES=waves, CAMELID_HIP_WIDE_PARTS=parts,
                           CAMELID_HIP_Q4K_MFMA_MIN_TOKENS=1, CAMELID_HIP_Q6K_MFMA_MIN_TOKENS=1), \
                        G.engaged(rf"^{tag}\.mfma\.wide\.g{g}w{waves}{walk}$", none=(r"\.dot\.",)):
                    assert G.same_bits(G.gpu_gemm(w, s, q), ref)
        with G.env(CAMELID_HIP_MFMA_WIDE=2, CAMELID_HIP_EXACT_ORDER=1, CAMELID_HIP_Q6K_MFMA_MIN_TOKENS=1), G.engaged(rf"^{tag}\.mfma\.wide\."):
            got = G.gpu_gemm(w, s, q)
        order = oracle.ORDER_PRIMARY if fmt == B.CML_Q4_K else oracle.ORDER_ALT  # the fused chains of the reference
        assert G.same_bits(got, oracle.matmul_q(fmt, wire, cols, s, q, order=order, threads=8))


# d (and dmin) subnormal, zero of either sign, negative, infinite, no number; activation scales the same.  Cells are the narrow kernel's, and without a K cut the
# oracle's, the ones that are no number among them (an infinite scale times a zero one, a difference of infinities).
@pytest.mark.parametrize("rows,cols", [(70, 768), (145, 13 * 256)])  # without and with a K cut
@pytest.mark.parametrize("name,fmt,tag", K_FORMATS)
def test_wide_cells_of_extreme_scales(name, fmt, tag, rows, cols):
    blocks = G.synth_weight(fmt, rows, cols, seed=rows).reshape(-1, 144 if fmt == B.CML_Q4_K else 210)
    at = [0, 2] if fmt == B.CML_Q4_K else [208]
    odd = np.array([0x0001, 0x83FF, 0x0000, 0x8000, 0x7C00, 0xFC00, 0x7E01, 0x7BFF, 0xFBFF], np.uint16).view(np.uint8).reshape(-1, 2)
    rng = np.random.default_rng(rows)
    for i, v in enumerate(odd):
        for a in at:
            hit = rng.choice(len(blocks), rows // 20 if 4 <= i <= 6 else len(blocks) // 12, replace=False)  # (most cells stay finite)
            blocks[hit, a:a + 2] = v
    w = Weight.upload(fmt, rows, cols, blocks.reshape(-1))
    for n in (3, 17, 130):
        s, q = activations(n, cols, seed=n)
        s = s.reshape(n, -1).copy()
        s[0], s[1] = 1e-39, -3e-42  # subnormal: products with d round among the subnormal numbers
        s[2] = 2e-36                # products that become subnormal
        if n > 16:
            s[5, 0], s[6, -1], s[7, 0], s[8] = np.inf, -np.inf, np.nan, 3e38
            s[9], s[16] = -0.0, 1e-38
        with G.env(CAMELID_HIP_MFMA_WIDE=0, CAMELID_HIP_Q4K_MFMA_MIN_TOKENS=1, CAMELID_HIP_Q6K_MFMA_MIN_TOKENS=1), G.engaged(r"\.mfma\.", none=(r"\.wide\.",)):
            ref = G.gpu_gemm(w, s, q)
        assert np.isfinite(ref).mean() > 0.3 and not np.isfinite(ref).all() and (np.abs(ref[:3]) < 1e-37).any() and ref[:3].any()
        if cols == 768:
            order = oracle.ORDER_PRIMARY if fmt == B.CML_Q4_K else oracle.ORDER_ALT
            assert np.array_equal(oracle.matmul_q(fmt, blocks.reshape(-1), cols, s, q, order=order, threads=8), ref, equal_nan=True)
        for g, waves, parts in [(g, v, p) for g in (1, 2, 3, 8) for v in (4, 8) for p in (1, 2)]:
            if n < 16 * (g - 1) and n != 3 or (name, g, waves, parts) == ("Q4_K", 8, 8, 2):
                continue
            G.say(f"wide {name} extreme scales {rows}x{cols} n={n} groups={g} waves={waves} parts={parts}")
            with G.env(CAMELID_HIP_MFMA_WIDE=2, CAMELID_HIP_WIDE_GROUPS=g, CAMELID_HIP_WIDE_WAVES=waves, CAMELID_HIP_WIDE_PARTS=parts,
                       CAMELID_HIP_Q4K_MFMA_MIN_TOKENS=1, CAMELID_HIP_Q6K_MFMA_MIN_TOKENS=1), G.engaged(rf"^{tag}\.mfma\.wide\.g{g}w{waves}", none=(r"\.dot\.",)):
                assert np.array_equal(G.gpu_gemm(w, s, q), ref, equal_nan=True)


@pytest.mark.parametrize("name,fmt,tag", K_FORMATS)
def test_wide_on_a_row_band(name, fmt, tag):
    """A view that starts and ends inside a tile, of rows with an odd number of super-blocks (Q6_K: block scales at odd halves of a word)."""
    rows, cols, n = 200, 5 * 256, 70
    w = Weight.upload(fmt, rows, cols, G.synth_weight(fmt, rows, cols, seed=5))
    s, q = activations(n, cols, seed=1)
    G.say(f"wide {name} row band")
    with G.env(CAMELID_HIP_MFMA_WIDE=2), G.engaged(rf"^{tag}\.mfma\.wide\."):
        whole, band = G.gpu_gemm(w, s, q), G.gpu_gemm(w.slice(7, 150), s, q)
    assert G.same_bits(band, whole[:, 7:157])


@pytest.mark.parametrize("name,fmt,tag", K_FORMATS)
def test_batches_of_more_than_32_tokens_take_the_wide_kernel(name, fmt, tag):
    rows, cols, n = 2048, 1024, 65
    w = Weight.upload(fmt, rows, cols, G.synth_weight(fmt, rows, cols, seed=6))
    x = np.random.default_rng(2).standard_normal((n, cols)).astype(np.float32)
    G.say(f"wide {name} default dispatch")
    with G.engaged(rf"^{tag}\.mfma\.wide\."):
        got = G.gpu_matmul_f32(w, x)
    with G.env(CAMELID_HIP_MFMA_WIDE=0), G.engaged(none=(r"\.wide\.",)):
        assert G.same_bits(got, G.gpu_matmul_f32(w, x))


def experts(E, hidden, ff, seed):
    return [Weight.upload(B.CML_Q4_K, E * r, c, G.synth_weight(B.CML_Q4_K, E * r, c, seed=seed + i)) for i, (r, c) in enumerate([(ff, hidden), (ff, hidden), (hidden, ff)])]


# gate and up in one launch, gathered rows, a group without assignments, one past a column, K cut inside the lane (down)
@pytest.mark.parametrize("E,k,hidden,ff,T", [(8, 2, 1024, 4096, 100), (4, 1, 256, 768, 5), (3, 3, 512, 512, 17), (6, 2, 4096, 1280, 130)])
def test_wide_expert_groups_are_bitwise_the_narrow_ones(E, k, hidden, ff, T):
    w = experts(E, hidden, ff, E + T)
    rng = np.random.default_rng(T)
    x = rng.standard_normal((T, hidden)).astype(np.float32)
    logits = rng.standard_normal((T, E)).astype(np.float32)
    logits[:, 0] += 1.0  # a crowded expert, one without assignments
    logits[:, E - 1] -= 50.0 * (E > k)
    idx, weight, _, _ = gpu_route(logits, k)
    run = lambda: gpu_moe(*w, E, k, idx, weight, x)
    with G.env(CAMELID_HIP_MFMA_WIDE=0), G.engaged(none=(r"\.wide\.",)):
        ref = run()
    for g in (1, 3, 4, 8):
        G.say(f"wide experts E={E} k={k} {hidden}/{ff} T={T} groups={g}")
        with G.env(CAMELID_HIP_MFMA_WIDE=2, CAMELID_HIP_WIDE_GROUPS=g), G.engaged(r"^q4k\.mfma\.wide\..*grouped"):
            assert G.same_bits(run(), ref)


B32_FORMATS = [("Q8_0", B.CML_Q8_0, "q8_0"), ("Q4_0", B.CML_Q4_0, "q4_0")]


# rows below a tile, past one, past a workgroup's; one slab, two, an odd number of them, rows long enough for two slabs ahead
@pytest.mark.parametrize("rows,cols", [(1, 256), (16, 512), (70, 1280), (300, 2048), (130, 25 * 256)])
@pytest.mark.parametrize("name,fmt,tag", B32_FORMATS)
def test_wide_b32_cells_are_bitwise_the_gemv(name, fmt, tag, rows, cols):
    wire = G.synth_weight(fmt, rows, cols, seed=rows + cols)
    blocks = wire.reshape(-1, 34 if fmt == B.CML_Q8_0 else 18)
    for special in (False, True):
        if special:  # scales that are no finite numbers, a zero one, a negative one
            blocks[:: 37, :2] = np.frombuffer(np.float16(np.inf).tobytes(), np.uint8)
            blocks[5:: 41, :2] = np.frombuffer(np.float16(-0.0).tobytes(), np.uint8)
            blocks[7:: 43, 1] ^= 0x80
        w = Weight.upload(fmt, rows, cols, wire)
        for n in (3, 16, 17, 70):
            x = np.random.default_rng(n).standard_normal((n, cols)).astype(np.float32)
            x[0] = 0.0
            s, q = oracle.quantize_activation(fmt, x)
            with G.env(CAMELID_HIP_MFMA_WIDE=0), G.engaged(none=(r"\.wide\.",)):
                ref = G.gpu_gemm(w, s, q)
            for g, tiles, ahead in [(g, t, 1) for g in (1, 2, 3, 4) for t in (1, 2)] + [(1, 1, 2)]:
                G.say(f"wide {name} {rows}x{cols} n={n} groups={g} tiles={tiles} ahead={ahead} special={special}")
                with G.env(CAMELID_HIP_MFMA_WIDE=2, CAMELID_HIP_WIDE_GROUPS=g, CAMELID_HIP_WIDE_TILES=tiles, CAMELID_HIP_WIDE_AHEAD=ahead,
                           CAMELID_HIP_B32_MFMA_MIN_TOKENS=1), G.engaged(rf"^{tag}\.mfma\.wide\.g{g}r{tiles}d{ahead}$", none=(r"\.dot\.",)):
                    got = G.gpu_gemm(w, s, q)
                assert np.array_equal(got, ref, equal_nan=True) if special else G.same_bits(got, ref)


# token columns that differ by a group, on enough row blocks that they change places between the workgroups of a compute unit
@pytest.mark.parametrize("n,groups", [(200, 4), (135, 3), (70, 4), (33, 2)])
@pytest.mark.parametrize("name,fmt,tag", B32_FORMATS)
def test_wide_b32_columns_of_unequal_width(name, fmt, tag, n, groups):
    rows, cols = 9300, 512
    w = Weight.upload(fmt, rows, cols, G.synth_weight(fmt, rows, cols, seed=n))
    s, q = oracle.quantize_activation(fmt, np.random.default_rng(n).standard_normal((n, cols)).astype(np.float32))
    with G.env(CAMELID_HIP_MFMA_WIDE=0), G.engaged(none=(r"\.wide\.",)):
        ref = G.gpu_gemm(w, s, q)
    for tiles in (1, 2):
        G.say(f"wide {name} unequal columns n={n} groups={groups} tiles={tiles}")
        with G.env(CAMELID_HIP_MFMA_WIDE=2, CAMELID_HIP_WIDE_GROUPS=groups, CAMELID_HIP_WIDE_TILES=tiles, CAMELID_HIP_WIDE_AHEAD=1), G.engaged(rf"^{tag}\.mfma\.wide\.g{groups}r{tiles}d1$"):
            assert G.same_bits(G.gpu_gemm(w, s, q), ref)


# a last slab of one, two, seven blocks; scale rows that start at odd halves of a word (an odd number of blocks), also where a band starts
@pytest.mark.parametrize("rows,cols", [(1, 288), (70, 320), (300, 736), (131, 4128)])
@pytest.mark.parametrize("name,fmt,tag", B32_FORMATS)
def test_wide_b32_rows_of_no_whole_slabs(name, fmt, tag, rows, cols):
    wire = G.synth_weight(fmt, rows, cols, seed=rows + cols)
    blocks = wire.reshape(-1, 34 if fmt == B.CML_Q8_0 else 18)
    for special in (False, True):
        if special:
            blocks[:: 37, :2] = np.frombuffer(np.float16(np.inf).tobytes(), np.uint8)
            blocks[7:: 43, 1] ^= 0x80
        w = Weight.upload(fmt, rows, cols, wire)
        for n in (5, 17, 70):
            s, q = oracle.quantize_activation(fmt, np.random.default_rng(n).standard_normal((n, cols)).astype(np.float32))
            s = s.reshape(n, -1).copy()
            if special:
                s[1, -1] = np.inf  # the scale that a short slab's requests repeat
            views = [w] + ([w.slice(3, rows - 5)] if rows > 16 else [])
            for v in views:
                with G.env(CAMELID_HIP_MFMA_WIDE=0), G.engaged(r"\.dot\.", none=(r"\.mfma\.",)):
                    ref = G.gpu_gemm(v, s, q)
                for g, tiles, ahead in [(g, t, 1) for g in (1, 2, 3, 4) for t in (1, 2) if (g, t) != (4, 2)] + [(1, 1, 2)]:
                    G.say(f"ragged {name} {rows}x{cols} n={n} groups={g} tiles={tiles} ahead={ahead} special={special}")
                    with G.env(CAMELID_HIP_WIDE_GROUPS=g, CAMELID_HIP_WIDE_TILES=tiles, CAMELID_HIP_WIDE_AHEAD=ahead, CAMELID_HIP_B32_MFMA_MIN_TOKENS=1), \
                            G.engaged(rf"^{tag}\.mfma\.wide\.g{g}r{tiles}d{ahead}\.ragged$", none=(r"\.dot\.",)):
                        got = G.gpu_gemm(v, s, q)
                    assert np.array_equal(got, ref, equal_nan=True) if special else G.same_bits(got, ref)


# 1637 blocks, and 1641: three more than a row of the packed dot holds
@pytest.mark.parametrize("name,fmt,tag", B32_FORMATS)
def test_rows_of_no_whole_slabs_are_refused_where_the_matvec_refuses_them(name, fmt, tag):
    rows, n = 20, 9
    for blocks, served in ((1637, True), (1641, False)):
        cols = 32 * blocks
        wire = G.synth_weight(fmt, rows, cols, seed=blocks)
        w = Weight.upload(fmt, rows, cols, wire)
        s, q = oracle.quantize_activation(fmt, np.random.default_rng(n).standard_normal((n, cols)).astype(np.float32))
        qd, sd, od = DeviceBuffer.from_numpy(q), DeviceBuffer.from_numpy(s), DeviceBuffer(n * rows * 4)
        G.say(f"ragged {name} rows of {blocks} blocks")
        for tokens in (1, 2, n):
            rc = lib().cml_gemm(w.handle, qd.ptr, sd.ptr, tokens, od.ptr, None)
            assert rc == (0 if served else 6), (blocks, tokens, rc)
        check(lib().cml_stream_sync(None))
        if served:
            assert G.same_bits(od.to_numpy(np.float32, (n, rows)), oracle.matmul_q(fmt, wire, cols, s, q, order=oracle.ORDER_PRIMARY, threads=8))


@pytest.mark.parametrize("name,fmt,tag", B32_FORMATS)
def test_wide_b32_on_a_row_band(name, fmt, tag):
    rows, cols, n = 200, 5 * 256, 40
    w = Weight.upload(fmt, rows, cols, G.synth_weight(fmt, rows, cols, seed=5))
    s, q = oracle.quantize_activation(fmt, np.random.default_rng(1).standard_normal((n, cols)).astype(np.float32))
    G.say(f"wide {name} row band")
    with G.engaged(rf"^{tag}\.mfma\.wide\."):
        whole, band = G.gpu_gemm(w, s, q), G.gpu_gemm(w.slice(7, 150), s, q)
    assert G.same_bits(band, whole[:, 7:157])
    with G.env(CAMELID_HIP_MFMA_WIDE=0):
        assert G.same_bits(whole, G.gpu_gemm(w, s, q))


# rows of no whole slabs (down, then both)
@pytest.mark.parametrize("E,k,hidden,ff,T", [(6, 3, 512, 352, 20), (4, 2, 1088, 704, 35)])
@pytest.mark.parametrize("name,fmt,tag", B32_FORMATS)
def test_wide_b32_expert_groups_on_rows_of_no_whole_slabs(name, fmt, tag, E, k, hidden, ff, T):
    gate_up = Weight.upload(fmt, E * 2 * ff, hidden, G.synth_weight(fmt, E * 2 * ff, hidden, seed=E))
    down = Weight.upload(fmt, E * hidden, ff, G.synth_weight(fmt, E * hidden, ff, seed=E + 1))
    rng = np.random.default_rng(T)
    x = rng.standard_normal((T, hidden)).astype(np.float32)
    idx, weight, _, _ = gpu_route(rng.standard_normal((T, E)).astype(np.float32), k)
    run = lambda: gpu_moe(gate_up, None, down, E, k, idx, weight, x, glu=1)
    with G.env(CAMELID_HIP_MFMA_WIDE=0), G.engaged(none=(r"\.wide\.",)):
        ref = run()
    for g in (1, 2):
        G.say(f"ragged {name} experts E={E} k={k} {hidden}/{ff} T={T} groups={g}")
        with G.env(CAMELID_HIP_MFMA_WIDE=2, CAMELID_HIP_WIDE_GROUPS=g), G.engaged(rf"^{tag}\.mfma\.wide\.g{g}r1d1\.ragged\.grouped$", none=(r"\.dot\.",)):
            assert G.same_bits(run(), ref)


# gate | up fused (gathered rows), down on rows of whole slabs; groups of none, one, past a column; a band that ends inside a workgroup
@pytest.mark.parametrize("E,k,hidden,ff,T", [(16, 4, 768, 512, 40), (8, 3, 256, 256, 1), (5, 2, 1280, 768, 33)])
@pytest.mark.parametrize("name,fmt,tag", B32_FORMATS)
def test_wide_b32_expert_groups_are_bitwise_the_gemv(name, fmt, tag, E, k, hidden, ff, T):
    gate_up = Weight.upload(fmt, E * 2 * ff, hidden, G.synth_weight(fmt, E * 2 * ff, hidden, seed=E))
    down = Weight.upload(fmt, E * hidden, ff, G.synth_weight(fmt, E * hidden, ff, seed=E + 1))
    rng = np.random.default_rng(T)
    x = rng.standard_normal((T + 1, hidden)).astype(np.float32)  # (a batch: a single token has a path of its own)
    logits = rng.standard_normal((T + 1, E)).astype(np.float32)
    logits[:, 0] += 1.0
    logits[:, E - 1] -= 50.0
    idx, weight, _, _ = gpu_route(logits, k)
    run = lambda: gpu_moe(gate_up, None, down, E, k, idx, weight, x, glu=1)
    with G.env(CAMELID_HIP_MFMA_WIDE=0), G.engaged(none=(r"\.wide\.",)):
        ref = run()
    for g in (1, 2):
        G.say(f"wide {name} experts E={E} k={k} {hidden}/{ff} T={T + 1} groups={g}")
        with G.env(CAMELID_HIP_MFMA_WIDE=2, CAMELID_HIP_WIDE_GROUPS=g), G.engaged(rf"^{tag}\.mfma\.wide\.g{g}r1d1\.grouped$", none=(r"\.dot\.",)):
            assert G.same_bits(run(), ref)


# Kernels that request the weight past the caches, on weights that small calls can afford: plain calls of one column, never of two; rows of no whole slabs only in
# Q8_0 and where they are whole 128-byte lines (44 blocks, not 41)
@pytest.mark.parametrize("rows,cols", [(70, 1280), (300, 512), (70, 1312), (70, 1408)])
@pytest.mark.parametrize("name,fmt,tag", B32_FORMATS)
def test_wide_b32_weights_requested_past_the_caches(name, fmt, tag, rows, cols):
    w = Weight.upload(fmt, rows, cols, G.synth_weight(fmt, rows, cols, seed=rows))
    for n in (3, 16, 17):
        s, q = oracle.quantize_activation(fmt, np.random.default_rng(n).standard_normal((n, cols)).astype(np.float32))
        with G.env(CAMELID_HIP_MFMA_WIDE=0), G.engaged(none=(r"\.wide\.",)):
            ref = G.gpu_gemm(w, s, q)
        for g, tiles, ahead in ((1, 1, 1), (1, 2, 1), (1, 1, 2), (2, 1, 1)):
            once = g == 1 and n <= 16 and (cols % 256 == 0 or (name == "Q8_0" and cols % 128 == 0))
            form = (r"\.ragged" if cols % 256 else "") + (r"\.once" if once else "")
            G.say(f"past the caches {name} {rows}x{cols} n={n} groups={g} tiles={tiles} ahead={ahead}")
            with G.env(CAMELID_HIP_MFMA_WIDE=2, CAMELID_HIP_WIDE_ONCE=1, CAMELID_HIP_WIDE_GROUPS=g, CAMELID_HIP_WIDE_TILES=tiles, CAMELID_HIP_WIDE_AHEAD=ahead,
                       CAMELID_HIP_B32_MFMA_MIN_TOKENS=1), G.engaged(rf"^{tag}\.mfma\.wide\.g{g}r{tiles}d{ahead}{form}$", none=(r"\.dot\.",)):
                assert G.same_bits(G.gpu_gemm(w, s, q), ref)


# groups of none, of one column and of several in one launch
@pytest.mark.parametrize("hidden,ff", [(768, 512), (512, 352), (512, 384)])
@pytest.mark.parametrize("name,fmt,tag", B32_FORMATS)
def test_wide_b32_expert_groups_requested_past_the_caches(name, fmt, tag, hidden, ff):
    E, k, T = 6, 2, 70
    gate_up = Weight.upload(fmt, E * 2 * ff, hidden, G.synth_weight(fmt, E * 2 * ff, hidden, seed=E))
    down = Weight.upload(fmt, E * hidden, ff, G.synth_weight(fmt, E * hidden, ff, seed=E + 1))
    rng = np.random.default_rng(T)
    x = rng.standard_normal((T, hidden)).astype(np.float32)
    logits = rng.standard_normal((T, E)).astype(np.float32)
    logits[:, 0] += 2.0
    logits[:, E - 2] -= 1.5
    logits[:, E - 1] -= 50.0
    idx, weight, chosen, _ = gpu_route(logits, k)
    held = np.bincount(chosen.reshape(-1), minlength=E)
    assert held.min() == 0 and (held[held > 0].min() <= 16) and held.max() > 32
    run = lambda: gpu_moe(gate_up, None, down, E, k, idx, weight, x, glu=1)
    with G.env(CAMELID_HIP_MFMA_WIDE=0), G.engaged(none=(r"\.wide\.",)):
        ref = run()
    for g in (1, 2):
        G.say(f"past the caches {name} experts {hidden}/{ff} groups={g}")
        past = ff % 256 == 0 or (name == "Q8_0" and ff % 128 == 0)
        down_form = (r"\.ragged" if ff % 256 else "") + r"\.grouped" + (r"\.once$" if past else "$")
        with G.env(CAMELID_HIP_MFMA_WIDE=2, CAMELID_HIP_WIDE_ONCE=1, CAMELID_HIP_WIDE_GROUPS=g), \
                G.engaged(rf"^{tag}\.mfma\.wide\.g{g}r1d1\.grouped\.once$", rf"^{tag}\.mfma\.wide\.g{g}r1d1{down_form}", none=(r"\.dot\.",) if past else (r"\.dot\.", r"ragged.*once")):
            assert G.same_bits(run(), ref)


@pytest.mark.parametrize("hidden,ff", [(1024, 4096), (512, 768)])  # down with a K cut, without
def test_wide_k_quant_expert_groups_requested_past_the_caches(hidden, ff):
    E, k, T = 4, 2, 100
    w = experts(E, hidden, ff, 9)
    rng = np.random.default_rng(T)
    x = rng.standard_normal((T, hidden)).astype(np.float32)
    logits = rng.standard_normal((T, E)).astype(np.float32)
    logits[:, 0] += 1.0
    logits[:, E - 1] -= 50.0
    idx, weight, _, _ = gpu_route(logits, k)
    run = lambda: gpu_moe(*w, E, k, idx, weight, x)
    with G.env(CAMELID_HIP_MFMA_WIDE=0), G.engaged(none=(r"\.wide\.",)):
        ref = run()
    for g, shape in ((2, "g2w4"), (3, "g3w4"), (4, "g4w4"), (8, "g8w8")):
        G.say(f"past the caches Q4_K experts {hidden}/{ff} groups={g}")
        down = r"\.serial_split" if ff == 4096 else ""
        with G.env(CAMELID_HIP_MFMA_WIDE=2, CAMELID_HIP_WIDE_ONCE=1, CAMELID_HIP_WIDE_GROUPS=g), \
                G.engaged(rf"^q4k\.mfma\.wide\.{shape}.*\.grouped\.once$", rf"^q4k\.mfma\.wide\.{shape}{down}\.grouped\.once$", none=(r"grouped$",)):
            assert G.same_bits(run(), ref)


# a row tile below 96 MB and one above; the two tensors of a layer, 102 and 51 MB
def test_which_weights_are_requested_past_the_caches():
    cols, n = 4096, 16
    some = G.synth_weight(B.CML_Q4_0, 128, cols, seed=1).reshape(128, -1)
    s, q = oracle.quantize_activation(B.CML_Q4_0, np.random.default_rng(n).standard_normal((n, cols)).astype(np.float32))
    want = G.gpu_gemm(Weight.upload(B.CML_Q4_0, 128, cols, some), s, q)
    for rows, past in ((43680, False), (43696, True)):
        w = Weight.upload(B.CML_Q4_0, rows, cols, np.tile(some, ((rows + 127) // 128, 1))[:rows])
        G.say(f"past the caches, {rows} rows")
        with G.engaged(r"^q4_0\.mfma\.wide\.g1r\dd\d" + (r"\.once$" if past else "$")):
            got = G.gpu_gemm(w, s, q)
        assert G.same_bits(got, np.tile(want, (1, rows // 128 + 1))[:, :rows])  # (the weight repeats its first 128 rows)
    E, k, T, hidden, ff = 4, 2, 8, 2048, 5888
    row = G.synth_weight(B.CML_Q8_0, 256, hidden, seed=2).reshape(256, -1)
    gate_up = Weight.upload(B.CML_Q8_0, E * 2 * ff, hidden, np.tile(row, (E * 2 * ff // 256, 1)))
    down = Weight.upload(B.CML_Q8_0, E * hidden, ff, np.tile(G.synth_weight(B.CML_Q8_0, 256, ff, seed=3).reshape(256, -1), (E * hidden // 256, 1)))
    rng = np.random.default_rng(T)
    x = rng.standard_normal((T, hidden)).astype(np.float32)
    idx, weight, _, _ = gpu_route(rng.standard_normal((T, E)).astype(np.float32), k)
    G.say("past the caches, the tensors of a layer")
    with G.engaged(r"^q8_0\.mfma\.wide\.g1r1d1\.grouped\.once$", r"^q8_0\.mfma\.wide\.g1r1d1\.grouped$"):
        got = gpu_moe(gate_up, None, down, E, k, idx, weight, x, glu=1)
    with G.env(CAMELID_HIP_MFMA_WIDE=0), G.engaged(none=(r"\.wide\.",)):
        assert G.same_bits(got, gpu_moe(gate_up, None, down, E, k, idx, weight, x, glu=1))


@pytest.mark.parametrize("name,fmt,tag", B32_FORMATS)
def test_scales_that_cannot_be_read_16_bytes_at_a_time_stay_off_the_wide_kernel(name, fmt, tag):
    rows, cols, n = 70, 768, 40
    w = Weight.upload(fmt, rows, cols, G.synth_weight(fmt, rows, cols, seed=8))
    s, q = oracle.quantize_activation(fmt, np.random.default_rng(3).standard_normal((n, cols)).astype(np.float32))
    want = G.gpu_gemm(w, s, q)
    qd, od = DeviceBuffer.from_numpy(q), DeviceBuffer(n * rows * 4)
    sd = DeviceBuffer.from_numpy(np.concatenate([[0.0], s.reshape(-1)]).astype(np.float32))
    G.say(f"wide {name} scales at 4 bytes past a 16-byte boundary")
    with G.engaged(rf"^{tag}\.mfma\.tile\.", none=(r"\.wide\.",)):
        check(lib().cml_gemm(w.handle, qd.ptr, sd.ptr + 4, n, od.ptr, None), "cml_gemm")
        check(lib().cml_stream_sync(None))
    assert G.same_bits(od.to_numpy(np.float32, (n, rows)), want)


# Which kernel a call without knobs takes, on either side of each line of the rules
ROUTES = [
    ("Q4_K", 2560, 4096, 33, r"^q4k\.mfma\.wide\.g1w4\.ksplit2\.serial_split$"),  # the smallest workgroups, where they alone have a compute unit each
    ("Q4_K", 1024, 4096, 48, r"^q4k\.mfma\.ksplit4"),  # K cut four ways, a workgroup of the narrow kernel per compute unit at most
    ("Q4_K", 4096, 4096, 33, r"^q4k\.mfma\.ksplit4"),  # up to two, the wide kernel's come to more than one as well
    ("Q4_K", 2048, 5120, 80, r"^q4k\.mfma\.wide\."),  # K parts of five super-blocks
    ("Q4_K", 2048, 2048, 100, r"^q4k\.mfma\.ksplit2"),  # cut two ways, parts of four
    ("Q4_K", 2056, 2048, 129, r"^q4k\.mfma\.wide\."),  # a third workgroup per compute unit
    ("Q4_K", 2048, 1024, 33, r"^q4k\.mfma\.wide\."),  # no cut
    ("Q6_K", 8200, 1024, 8, r"^q6k\.mfma\.tile\."),  # at most one wave per SIMD
    ("Q6_K", 16400, 1024, 8, r"^q6k\.mfma\.wide\."),  # more
    ("Q6_K", 33000, 512, 16, r"^q6k\.mfma\.tile\."),  # short rows of a tall weight
    ("Q6_K", 8192, 1024, 32, r"^q6k\.mfma\.tile\."),  # rows of four super-blocks
    ("Q6_K", 8192, 1024, 33, r"^q6k\.mfma\.wide\."),  # more tokens
    ("Q6_K", 8192, 1280, 17, r"^q6k\.mfma\.wide\."),  # longer rows
    ("Q8_0", 8320, 5120, 8, r"^q8_0\.mfma\.wide\.g1r1d2$"),  # two slabs ahead where a workgroup has a compute unit
    ("Q4_0", 8320, 4096, 16, r"^q4_0\.mfma\.wide\.g1r1d2$"),  # the same
    ("Q4_0", 33000, 1024, 16, r"^q4_0\.mfma\.wide\.g1r1d1$"),  # two share one
    ("Q8_0", 10000, 768, 8, r"^q8_0\.mfma\.wide\.g1r1d2$"),  # two slabs ahead on rows of three, too
    ("Q8_0", 8832, 1280, 128, r"^q8_0\.mfma\.wide\.g3r1d1$"),  # three workgroups of three token groups on some compute units (14 of 12.3 us for four of two)
    ("Q8_0", 39536, 768, 64, r"^q8_0\.mfma\.wide\.g2r1d1$"),  # two row tiles per wave double the slowest compute unit's work
    ("Q4_0", 21888, 1280, 128, r"^q4_0\.mfma\.wide\.g2r1d1$"),  # the same
    ("Q4_0", 8320, 1024, 16, r"^q4_0\.mfma\.kpar\."),  # up to 768 tiles of short rows
    ("Q4_0", 8320, 2048, 16, r"^q4_0\.mfma\.wide\."),  # longer rows
    ("Q8_0", 8320, 1024, 16, r"^q8_0\.mfma\.wide\."),  # Q8_0: up to 512
    ("Q4_0", 41000, 1024, 12, r"^q4_0\.mfma\.tile\."),  # rows of four to seven slabs of tall weights
    ("Q4_0", 40960, 1024, 12, r"^q4_0\.mfma\.wide\."),  # less tall
    ("Q8_0", 41000, 512, 32, r"^q8_0\.mfma\.tile\."),  # rows of two slabs of tall weights
    ("Q8_0", 41000, 512, 33, r"^q8_0\.mfma\.wide\."),  # more tokens
    ("Q4_0", 4096, 5120, 8, r"^q4_0\.dot\."),  # eight tokens on rows of 17 to 24 slabs, up to 256 tiles
    ("Q4_0", 4100, 5120, 8, r"^q4_0\.mfma\.wide\."),  # more
    ("Q8_0", 7000, 768, 8, r"^q8_0\.dot\."),  # rows of three slabs
    ("Q4_0", 2048, 1024, 8, r"^q4_0\.mfma\.kpar\."),  # four
    ("Q8_0", 4096, 2912, 8, r"^q8_0\.dot\."),  # rows of no whole slabs: one pass of the packed dot on small weights
    ("Q8_0", 4096, 2912, 9, r"^q8_0\.mfma\.wide\..*ragged$"),  # two
    ("Q4_0", 2048, 1056, 5, r"^q4_0\.mfma\.wide\..*ragged$"),  # up to four slabs and a part
    ("Q4_0", 8192, 2912, 5, r"^q4_0\.dot\."),
    ("Q4_0", 8192, 2912, 6, r"^q4_0\.mfma\.wide\..*ragged$"),
    ("Q8_0", 14336, 1056, 3, r"^q8_0\.mfma\.wide\..*ragged$"),  # more than 767 tiles
    ("Q4_0", 12288, 1312, 3, r"^q4_0\.mfma\.wide\..*ragged$"),
    ("Q8_0", 736, 704, 200, r"^q8_0\.mfma\.wide\.g1r1d1\.ragged$"),  # rows of two slabs and a part are over before a second slab ahead pays
    ("Q8_0", 736, 1056, 200, r"^q8_0\.mfma\.wide\.g1r1d2\.ragged$"),
    ("Q8_0", 14336, 1056, 4, r"^q8_0\.dot\."),  # four tokens are one pass of the packed dot
    ("Q4_0", 23984, 800, 4, r"^q4_0\.dot\."),
    ("Q4_0", 24000, 800, 4, r"^q4_0\.mfma\.wide\..*ragged$"),  # more than 1499 tiles
    ("Q8_0", 1024, 928, 5, r"^q8_0\.dot\."),  # rows of 24 to 31 blocks
    ("Q8_0", 1024, 928, 6, r"^q8_0\.mfma\.wide\..*ragged$"),
    ("Q8_0", 768, 1152, 8, r"^q8_0\.mfma\.wide\..*ragged$"),  # eight on rows of four slabs and a part
    ("Q4_0", 992, 1248, 8, r"^q4_0\.mfma\.wide\..*ragged$"),
    ("Q8_0", 4096, 544, 8, r"^q8_0\.dot\."),  # but of up to 31 blocks
    ("Q4_0", 4096, 832, 8, r"^q4_0\.dot\."),
    ("Q4_0", 8192, 832, 8, r"^q4_0\.dot\."),
    ("Q4_0", 8208, 832, 8, r"^q4_0\.mfma\.wide\..*ragged$"),  # more than 512 tiles
    ("Q8_0", 24000, 800, 4, r"^q8_0\.mfma\.wide\..*ragged$"),
    ("Q4_0", 8208, 2912, 5, r"^q4_0\.mfma\.wide\..*ragged$"),  # five on more than 512
    ("Q4_0", 8192, 1056, 5, r"^q4_0\.mfma\.wide\..*ragged$"),  # on less with short rows
]


@pytest.mark.parametrize("name,rows,cols,n,kernel", ROUTES)
def test_calls_take_the_kernel_that_is_ahead(name, rows, cols, n, kernel):
    fmt = {"Q4_K": B.CML_Q4_K, "Q6_K": B.CML_Q6_K, "Q8_0": B.CML_Q8_0, "Q4_0": B.CML_Q4_0}[name]
    w = Weight.upload(fmt, rows, cols, G.synth_weight(fmt, rows, cols, seed=rows + n))
    x = np.random.default_rng(n).standard_normal((n, cols)).astype(np.float32)
    G.say(f"route {name} {rows}x{cols} n={n}")
    with G.engaged(kernel, none=(r"\.mfma\.",) if ".dot" in kernel else (r"\.dot\.",)):
        got = G.gpu_matmul_f32(w, x)
    # the packed-dot kernel on the same inputs
    with G.env(CAMELID_HIP_Q4K_MFMA_MIN_TOKENS=1 << 30, CAMELID_HIP_Q6K_MFMA_MIN_TOKENS=1 << 30, CAMELID_HIP_B32_MFMA_MIN_TOKENS=1 << 30, CAMELID_HIP_FUSED_QUANT=0), \
            G.engaged(r"\.dot\.", none=(r"\.mfma\.",)):
        assert G.same_bits(got, G.gpu_matmul_f32(w, x))


# 10, 18 and 25 assignments per expert on average: both launches narrow; down (K cut, 1024 tiles) wide; both, two token groups per column
@pytest.mark.parametrize("T,expect,none", [(40, (r"^q4k\.mfma\.(tile|serial_split)\..*grouped",), (r"\.wide\.",)),
                                           (72, (r"^q4k\.mfma\.wide\.g2w4\.serial_split\.grouped$", r"^q4k\.mfma\.(tile|serial_split)\..*grouped"), ()),
                                           (100, (r"^q4k\.mfma\.wide\.g2w4\.serial_split\.grouped$",), ())])
def test_expert_groups_take_the_kernel_that_is_ahead(T, expect, none):
    E, k, hidden, ff = 8, 2, 2048, 2048
    w = experts(E, hidden, ff, 3)
    rng = np.random.default_rng(T)
    x = rng.standard_normal((T, hidden)).astype(np.float32)
    idx, weight, _, _ = gpu_route(rng.standard_normal((T, E)).astype(np.float32), k)
    G.say(f"expert groups, default dispatch, T={T}")
    with G.engaged(*expect, none=none):
        got = gpu_moe(*w, E, k, idx, weight, x)
    with G.env(CAMELID_HIP_MFMA_WIDE=0), G.engaged(none=(r"\.wide\.",)):
        assert G.same_bits(got, gpu_moe(*w, E, k, idx, weight, x))
