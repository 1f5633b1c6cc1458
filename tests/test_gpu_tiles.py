"""The batched kernels at the edges of their tiles, bit for bit against the
CPU oracle (the reference's order of every f32 sum, so no tolerance)."""
import ctypes
import time

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

F32, F16, BF16, Q4_0, Q5_0, Q8_0, Q4_K, Q5_K, Q6_K = range(9)


def same_bits(got, ref):
    return np.array_equal(np.asarray(got).view(np.uint32), np.asarray(ref).view(np.uint32))


@pytest.mark.parametrize("kind,cols,rows,m", [
    (F16, 8, 1, 2), (F16, 120, 63, 15), (F16, 128, 64, 16), (F16, 136, 65, 17), (F16, 2568, 130, 37), (F16, 264, 9000, 64),
    (BF16, 24, 65, 3), (BF16, 1024, 131, 64), (BF16, 1160, 17, 100), (BF16, 256, 8200, 33),
    (F32, 8, 17, 2), (F32, 248, 64, 31), (F32, 512, 129, 65), (F32, 136, 8256, 48)])
def test_float_matmul_tiles(aotk, oracle, kind, cols, rows, m):
    """Rows of whole 8-value groups: remainders of the 16-group stages (odd
    and even stage counts), of the 64-row blocks and of one and two token
    tiles, with exponents down to the subnormals."""
    rng = np.random.default_rng(cols + rows + m)
    w = (rng.standard_normal((rows, cols)) * 0.02).astype(np.float32)
    w[:, ::7] *= np.float32(2.0 ** -18)  # f16 subnormals
    xs = (rng.standard_normal((m, cols)) * np.exp2(rng.integers(-70, 20, (m, cols)))).astype(np.float32)
    xs[0] = np.float32(-1e-42) * np.sign(xs[0])  # products that underflow to signed zeros
    raw = oracle.quantize_rows(kind, w)
    h = aotk.Weight(kind, raw, rows, cols)
    got = aotk.matmul(h, xs, m)
    h.free()
    ref = oracle.matmul(kind, raw, np.ascontiguousarray(xs).view(np.uint8).reshape(-1), m, rows, cols,
                        pool=oracle.Pool(8)).reshape(m, rows)
    assert same_bits(got, ref)


@pytest.mark.parametrize("kind", [F16, F32])
def test_float_matmul_two_matrices(aotk, oracle, kind):
    """The gate / up pair: a 64-row block over the boundary of the two."""
    rng = np.random.default_rng(4 + kind)
    rows, cols, m = 83, 384, 21
    raws = [oracle.quantize_rows(kind, (rng.standard_normal((rows, cols)) * 0.02).astype(np.float32)) for _ in range(2)]
    xs = rng.standard_normal((m, cols)).astype(np.float32)
    ws = [aotk.Weight(kind, r, rows, cols) for r in raws]
    got = aotk.matmul2(ws[0], ws[1], xs, m)
    for g, r in zip(got, raws):
        assert same_bits(g, oracle.matmul(kind, r, xs.view(np.uint8).reshape(-1), m, rows, cols).reshape(m, rows))


@pytest.mark.parametrize("kind", [Q8_0, Q4_0, Q5_0])
@pytest.mark.parametrize("cols,rows,m", [
    (32, 1, 2), (96, 17, 15), (256, 16, 16), (288, 33, 17), (480, 47, 32), (512, 48, 33), (544, 15, 48),
    (2048, 131, 49), (2080, 64, 64), (352, 20, 65), (736, 49, 100), (1024, 9, 130)])
def test_q80_family_matmul_tiles(aotk, oracle, kind, cols, rows, m):
    """Remainders of the 4- and 8-block stages (odd and even stage counts),
    the 16-row blocks, and one to four token tiles on one or two waves each."""
    rng = np.random.default_rng(cols + rows + m + kind)
    raw = oracle.quantize_rows(kind, (rng.standard_normal((rows, cols)) * 0.02).astype(np.float32))
    xs = (rng.standard_normal((m, cols)) * np.exp2(rng.integers(-6, 6, (m, 1)))).astype(np.float32)
    acts = np.concatenate([oracle.quantize_act(kind, x) for x in xs])
    h = aotk.Weight(kind, raw, rows, cols)
    got = aotk.matmul(h, acts, m)
    h.free()
    ref = oracle.matmul(kind, raw, acts, m, rows, cols, pool=oracle.Pool(8)).reshape(m, rows)
    assert same_bits(got, ref)


@pytest.mark.parametrize("kind,cols,m", [(Q8_0, 204800, 2), (Q4_0, 65536, 17), (Q5_0, 28672, 45), (Q8_0, 12288, 105)])
def test_noalloc_without_room_for_the_tiled_copy(aotk, oracle, kind, cols, m):
    """Two inputs of 204800 columns and other batches whose staging fits the
    fixed memory, but not with the copy's last 16-vector tile padded: one, two,
    three and four tiles per block."""
    rows = 19
    rng = np.random.default_rng(12)
    raw = oracle.quantize_rows(kind, (rng.standard_normal((rows, cols)) * 0.02).astype(np.float32))
    acts = np.concatenate([oracle.quantize_act(kind, rng.standard_normal(cols).astype(np.float32)) for _ in range(m)])
    h = aotk.Weight(kind, raw, rows, cols)
    got = aotk.matmul_noalloc(h, acts, m)
    h.free()
    assert same_bits(got, oracle.matmul(kind, raw, acts, m, rows, cols, pool=oracle.Pool(8)).reshape(m, rows))


@pytest.mark.parametrize("cols,m", [(12288, 105), (4096, 327)])
def test_noalloc_batch_at_the_limit_of_its_memory(aotk, cols, m):
    """A last tile of a few vectors at the fixed memory's limit: the product is
    the allocating call's, bits and speed. Reading the weights once per vector
    instead of once per tile takes over three times as long here, the allowance
    is 1.6."""
    rows = 4096
    rng = np.random.default_rng(m)
    raw = rng.integers(0, 256, (rows * cols // 32, 34), dtype=np.uint8)
    raw[:, :2] = np.float16(2.7e-4).view(np.uint16).reshape(1).view(np.uint8)
    acts = rng.integers(0, 256, (m * cols // 32, 36), dtype=np.uint8)
    acts[:, :4] = np.float32(0.01).reshape(1).view(np.uint8)
    h = aotk.Weight(Q8_0, raw.reshape(-1), rows, cols)
    lib = aotk.runtime._lib()
    x, y = aotk.DeviceBuffer.from_numpy(acts.reshape(-1)), [aotk.DeviceBuffer(4 * m * rows) for _ in range(2)]
    best = [1e9, 1e9]
    for _ in range(12):  # (the first ones warm up)
        for i, call in enumerate((lib.aotk_matmul, lib.aotk_matmul_noalloc)):
            t = time.perf_counter()
            assert call(h.h, x.ptr, m, y[i].ptr) == 0
            best[i] = min(best[i], time.perf_counter() - t)
    assert same_bits(y[1].to_numpy(np.float32, m * rows), y[0].to_numpy(np.float32, m * rows))
    assert best[1] < 1.6 * best[0]
    h.free()


def attention_ref(oracle, q, kc, vc, nh, nkv, hd, ctx, pos0, m, window):
    ref = np.zeros(m * nh * hd, np.float32)
    p = oracle.Pool(8)
    oracle.load().or_attention(p.p, oracle.ptr(ref), oracle.ptr(q), oracle.ptr(kc), oracle.ptr(vc), nh, nkv, hd, ctx, 0,
                               pos0, m, window)
    return ref


@pytest.mark.parametrize("nh,nkv,hd,pos0,m,window", [
    # one, two and four items per wave; groups of 16 positions cut at either
    # end; every ratio of query to kv heads
    (4, 4, 64, 0, 2, 0), (4, 4, 64, 14, 3, 0), (32, 4, 64, 0, 6, 0), (32, 4, 64, 505, 64, 0), (6, 2, 64, 31, 33, 20),
    (32, 8, 128, 0, 64, 0), (32, 8, 128, 447, 64, 0), (10, 2, 128, 100, 17, 0), (12, 2, 128, 63, 40, 50),
    (14, 2, 128, 5, 30, 0), (16, 2, 128, 130, 64, 100), (32, 8, 128, 985, 39, 0), (32, 8, 128, 1500, 33, 1024),
    (8, 4, 256, 200, 64, 1024), (8, 4, 256, 3001, 50, 1024), (8, 4, 256, 1000, 40, 1024), (4, 4, 256, 70, 5, 64),
    # the softmax's classes: many pairs at 512, 1024, 2048, 4096, 8192
    # positions, few pairs likewise, past 8192
    (32, 8, 128, 448, 64, 0), (32, 8, 128, 449, 64, 0), (32, 4, 64, 960, 64, 0), (32, 4, 64, 961, 64, 0),
    (32, 4, 64, 1984, 64, 0), (32, 4, 64, 1985, 64, 0), (32, 4, 64, 4032, 64, 0), (32, 4, 64, 4033, 64, 0),
    (32, 4, 64, 8128, 64, 0), (32, 4, 64, 8129, 64, 0),
    (8, 4, 64, 508, 4, 0), (8, 4, 64, 509, 4, 0), (8, 4, 64, 1020, 4, 0), (8, 4, 64, 1021, 4, 0),
    (8, 4, 64, 2044, 4, 0), (8, 4, 64, 2045, 4, 0), (8, 4, 64, 8188, 4, 0), (8, 4, 64, 8189, 4, 0), (4, 2, 64, 16379, 2, 0)])
def test_prompt_attention_tiles(aotk, oracle, nh, nkv, hd, pos0, m, window):
    rng = np.random.default_rng(nh * 7 + hd + pos0 + m)
    ctx = pos0 + m + 3  # (at most the longest context, 16384)
    q = (rng.standard_normal(m * nh * hd) * 2).astype(np.float32)
    kc, vc = (rng.standard_normal(ctx * nkv * hd).astype(np.float32) for _ in range(2))
    vc[::5] *= np.float32(1e-39)  # products in the subnormals
    got = aotk.attention(q, kc, vc, nh, nkv, hd, ctx, 0, pos0, m, window)
    assert same_bits(got, attention_ref(oracle, q, kc, vc, nh, nkv, hd, ctx, pos0, m, window))


@pytest.mark.parametrize("nh,nkv,ctx,m", [(0, 4, 16, 2), (0, 4, 16, 1), (4, 0, 16, 2), (5, 2, 16, 2), (18, 2, 16, 2), (4, 2, 16, 0),
                                          (4, 2, 16385, 1), (4, 2, 16385, 2)])
def test_attention_refuses_bad_head_counts_no_rows_and_long_contexts(aotk, nh, nkv, ctx, m):
    """No query head used to reach a division by the group size."""
    z = np.zeros(64 * 64, np.float32)
    with pytest.raises(aotk.abi.AotkError, match="attention: "):
        aotk.attention(z, z, z, nh, nkv, 64, ctx, 0, 4, m, 0)


@pytest.mark.parametrize("nh,nkv,hd,pos0,m,window", [(8, 4, 128, 200, 9, 0), (32, 8, 128, 70, 64, 40), (8, 4, 256, 90, 21, 32)])
def test_prompt_attention_masks_positions(aotk, oracle, nh, nkv, hd, pos0, m, window):
    """Infinities and NaN in cache rows that a query row does not hold (later
    positions, positions before its window) leave it untouched."""
    rng = np.random.default_rng(3 + pos0)
    ctx = pos0 + m + 3
    q = rng.standard_normal(m * nh * hd).astype(np.float32)
    kc, vc = (rng.standard_normal((ctx, nkv * hd)).astype(np.float32) for _ in range(2))
    want = attention_ref(oracle, q, kc.reshape(-1), vc.reshape(-1), nh, nkv, hd, ctx, pos0, m, window)
    clean = [i for i in range(m - 2)]
    if window:
        vc[:pos0 + 4 - window + 1] = np.inf  # before the windows of rows 4 and on
        kc[:pos0 + 4 - window + 1] = np.nan
        clean = clean[4:]
    vc[pos0 + m - 2:] = np.nan  # held by the last two rows only
    kc[pos0 + m - 1:] = np.inf
    got = aotk.attention(q, kc.reshape(-1), vc.reshape(-1), nh, nkv, hd, ctx, 0, pos0, m, window)
    assert same_bits(got.reshape(m, -1)[clean], want.reshape(m, -1)[clean])


@pytest.mark.parametrize("kind,cols", [(Q4_K, 256), (Q4_K, 2048), (Q4_K, 4096), (Q4_K, 16384), (Q4_K, 16640), (Q5_K, 2560), (Q5_K, 5632),
                                       (Q6_K, 768), (Q6_K, 10240), (Q6_K, 12288), (Q6_K, 14336), (Q6_K, 11008),
                                       (Q8_0, 32), (Q8_0, 4128), (Q8_0, 16384), (Q8_0, 16416), (Q4_0, 96), (Q4_0, 16384),
                                       (Q5_0, 2080)])
def test_matvec_from_blocks(aotk, oracle, kind, cols):
    """One token in the reference's blocks, single and as three matrices: the
    widths where the matvec reads the blocks itself, and the first past them."""
    rng = np.random.default_rng(cols + kind)
    rows = (37, 5, 70)
    x = oracle.quantize_act(kind, (rng.standard_normal(cols) * 3).astype(np.float32))
    raws = [oracle.quantize_rows(kind, (rng.standard_normal((r, cols)) * 0.02).astype(np.float32)) for r in rows]
    refs = [oracle.matvec(kind, w, x, r, cols) for w, r in zip(raws, rows)]
    ws = [aotk.Weight(kind, w, r, cols) for w, r in zip(raws, rows)]
    assert same_bits(aotk.matvec(ws[0], x), refs[0])
    for got, ref in zip(aotk.matvec3(ws, x), refs):
        assert same_bits(got, ref)


@pytest.mark.parametrize("kind", [Q4_K, Q8_0])
def test_matvec_output_over_its_input(aotk, oracle, kind):
    rng = np.random.default_rng(kind)
    rows, cols = 700, 4096
    x = oracle.quantize_act(kind, rng.standard_normal(cols).astype(np.float32))
    raw = oracle.quantize_rows(kind, (rng.standard_normal((rows, cols)) * 0.02).astype(np.float32))
    w = aotk.Weight(kind, raw, rows, cols)
    buf = aotk.DeviceBuffer.from_numpy(np.ascontiguousarray(x).view(np.uint8).reshape(-1))
    lib = aotk.runtime._lib()
    assert lib.aotk_matvec(w.h, buf.ptr, buf.ptr) == 0
    assert same_bits(buf.to_numpy(np.float32, rows), oracle.matvec(kind, raw, x, rows, cols))


@pytest.mark.parametrize("kind", [Q4_K, Q8_0])
@pytest.mark.parametrize("n,at", [(1, 0), (1, 256), (3, 0), (3, 1024)])
def test_matvec_outputs_over_the_input_in_many_rounds(aotk, oracle, kind, n, at):
    """40000 rows, 5000 blocks: more than are resident, so that later blocks
    start after earlier ones have stored. The only or the last of three outputs
    starts `at` bytes into the input."""
    rng = np.random.default_rng(kind + at)
    cols, rows = 4096, [8, 24, 40000][3 - n:]
    bs, ts = (256, 144) if kind == Q4_K else (32, 34)
    x = np.ascontiguousarray(oracle.quantize_act(kind, rng.standard_normal(cols).astype(np.float32))).view(np.uint8).reshape(-1)
    assert at < x.size
    raws = []
    for r in rows:
        raw = rng.integers(0, 256, (r * cols // bs, ts), dtype=np.uint8)
        raw[:, :2] = np.float16([1e-3]).view(np.uint8)
        if kind == Q4_K:
            raw[:, 2:4] = np.float16([2e-3]).view(np.uint8)
        raws.append(raw.reshape(-1))
    ws = [aotk.Weight(kind, raw, r, cols) for raw, r in zip(raws, rows)]
    buf = aotk.DeviceBuffer(4 * rows[-1] + at)
    buf.upload(x)
    outs = [aotk.DeviceBuffer(4 * r) for r in rows[:-1]]
    ptrs = [o.ptr for o in outs] + [buf.ptr + at]
    lib = aotk.runtime._lib()
    if n == 1:
        assert lib.aotk_matvec(ws[0].h, buf.ptr, ptrs[0]) == 0
    else:
        assert lib.aotk_matvec3((ctypes.c_void_p * 3)(*[w.h for w in ws]), buf.ptr, (ctypes.c_void_p * 3)(*ptrs)) == 0
    got = [o.to_numpy(np.float32) for o in outs] + [buf.to_numpy(np.uint8)[at:].view(np.float32)]
    for g, raw, r, w in zip(got, raws, rows, ws):
        assert same_bits(g, oracle.matvec(kind, raw, x, r, cols))
        w.free()


@pytest.mark.parametrize("kind,rows,cols,m", [(Q4_K, 2048, 256, 2), (Q6_K, 2050, 768, 17), (Q5_K, 100, 2304, 33), (Q4_K, 33, 512, 16)])
def test_kquant_staging_tiles(aotk, oracle, kind, rows, cols, m):
    """The staged copies of the input's blocks (tiled and plain) around whole
    and partial 16-vector tiles."""
    rng = np.random.default_rng(rows + m)
    xs = np.concatenate([np.ascontiguousarray(oracle.quantize_act(kind, rng.standard_normal(cols).astype(np.float32))).view(np.uint8).reshape(-1)
                         for _ in range(m)])
    raw = oracle.quantize_rows(kind, (rng.standard_normal((rows, cols)) * 0.02).astype(np.float32))
    got = aotk.matmul(aotk.Weight(kind, raw, rows, cols), xs, m)
    assert same_bits(got, oracle.matmul(kind, raw, xs, m, rows, cols, pool=oracle.Pool(8)).reshape(m, rows))


@pytest.mark.parametrize("hd", [64, 128, 256])
@pytest.mark.parametrize("span", [1, 64, 65, 320, 321, 384, 385, 448, 768, 769, 1023, 1152, 1537, 4609, 16384])
def test_decode_attention_chunks(aotk, oracle, hd, span):
    """One row over spans around the 64-value runs and the 384-position chunks
    of its ordered sums, signed zeros and subnormal products among them."""
    rng = np.random.default_rng(span + hd)
    q = rng.standard_normal(4 * hd).astype(np.float32)
    kc, vc = (rng.standard_normal(span * 2 * hd).astype(np.float32) for _ in range(2))
    vc[::3] = np.float32(-0.0)
    vc[1::5] *= np.float32(1e-39)
    got = aotk.attention(q, kc, vc, 4, 2, hd, span, 0, span - 1, 1, 0)
    assert same_bits(got, attention_ref(oracle, q, kc, vc, 4, 2, hd, span, span - 1, 1, 0))


def test_exp_at_its_ends(aotk, oracle):
    """SiLU and softmax where exp leaves its common path: over- and underflow
    and the values beside them, infinities, subnormal results and the inputs
    that are compared one by one."""
    ends = np.array([0x42b17217, 0x42b17218, 0x42b17219, 0x42b00000, 0xc2cff1b4, 0xc2cff1b5, 0xc2cff1b6, 0xc2aeac50, 0xc2b00000,
                     0x4202422f, 0x4202422e, 0xc27c65d9, 0xc27c65da, 0x7f800000, 0xff800000, 0x7f7fffff, 0xff7fffff,
                     0x00000001, 0x80000001], np.uint32).view(np.float32)
    h = np.concatenate([ends, -ends])
    up = np.ones_like(h)
    ref = h.copy()
    oracle.load().or_silu_mul(oracle.ptr(ref), oracle.ptr(up), ref.size)
    got = aotk.silu_mul(h, up)
    nan = np.isnan(ref)
    assert np.array_equal(np.isnan(got), nan) and same_bits(got[~nan], ref[~nan])
    s = np.concatenate([[0.0], np.minimum(ends, 0)]).astype(np.float32)
    ref = s.copy()
    oracle.load().or_softmax(oracle.ptr(ref), ref.size)
    assert same_bits(aotk.softmax(s), ref)


def same_or_nan(got, ref):
    """Equal bits, and NaN exactly where the reference has one (which NaN is
    not part of the contract)."""
    got, ref = np.asarray(got).reshape(-1), np.asarray(ref).reshape(-1)
    nan = np.isnan(ref)
    return np.array_equal(np.isnan(got), nan) and same_bits(got[~nan], ref[~nan])


@pytest.mark.parametrize("kind", [F16, BF16, F32])
@pytest.mark.parametrize("cols,m", [(136, 20), (256, 37)])
def test_float_matmul_not_finite(aotk, oracle, kind, cols, m):
    """Infinities and NaN in weights and inputs, in whole and partial stages,
    and sums that overflow: the fused multiply-add's results, NaN payloads and
    signs among them, and other rows and tokens keep their bits."""
    rng = np.random.default_rng(cols + kind)
    rows = 70
    w = (rng.standard_normal((rows, cols)) * 0.02).astype(np.float32)
    w[3, 0], w[17, cols - 1], w[40, 5], w[41, 9], w[64] = np.inf, np.nan, -np.inf, 60000.0, 0.0
    w.view(np.uint32)[17, cols - 1] = 0xFFC12000  # payload bits that bf16 keeps
    xs = rng.standard_normal((m, cols)).astype(np.float32)
    xs[2, 7], xs[9, cols - 3], xs[15, 1], xs[11, ::2] = np.inf, np.nan, -np.inf, 3e38
    xs.view(np.uint32)[9, cols - 3] = 0x7FC34567
    raw = oracle.quantize_rows(kind, w)
    h = aotk.Weight(kind, raw, rows, cols)
    got = aotk.matmul(h, xs, m)
    h.free()
    ref = oracle.matmul(kind, raw, xs.view(np.uint8).reshape(-1), m, rows, cols, pool=oracle.Pool(8))
    assert np.isnan(ref).any() and np.isinf(ref).any() and np.isfinite(ref).mean() > 0.5
    assert same_bits(got.reshape(-1), ref.reshape(-1))


@pytest.mark.parametrize("kind", [Q8_0, Q4_0, Q5_0])
@pytest.mark.parametrize("cols,m", [(288, 13), (256, 20), (288, 37), (544, 64)])
def test_q80_family_matmul_not_finite(aotk, oracle, kind, cols, m):
    """Infinite and NaN block scales of weights and inputs (the last block's,
    which the blocks past the end repeat, among them), scale products that
    overflow, and an infinite scale times a zero quant."""
    rng = np.random.default_rng(cols + kind + m)
    rows, nb = 40, cols // 32
    w = (rng.standard_normal((rows, cols)) * 0.02).astype(np.float32)
    w[3, 0:4] = 0.0
    raw = np.array(oracle.quantize_rows(kind, w)).view(np.uint8).reshape(rows, nb, -1)

    def put(row, blk, v):
        raw[row, blk, :2] = np.float16([v]).view(np.uint8)
    put(3, 0, np.inf), put(17, nb - 1, np.nan), put(18, nb - 1, -np.inf), put(20, 2, 60000.0)
    acts = np.stack([np.ascontiguousarray(oracle.quantize_act(kind, x.astype(np.float32))).view(np.uint8).reshape(nb, 36)
                     for x in rng.standard_normal((m, cols))])
    for tok, blk, v in ((2, 1, np.inf), (9, nb - 1, np.nan), (10, nb - 1, np.inf), (11, 2, 1e38)):
        acts[tok, blk, :4] = np.float32([v]).view(np.uint8)
    h = aotk.Weight(kind, raw.reshape(-1), rows, cols)
    got = aotk.matmul(h, acts.reshape(-1), m)
    h.free()
    ref = oracle.matmul(kind, raw.reshape(-1), acts.reshape(-1), m, rows, cols, pool=oracle.Pool(8))
    assert np.isnan(ref).any() and np.isinf(ref).any() and np.isfinite(ref).mean() > 0.5
    assert same_or_nan(got, ref)


@pytest.mark.parametrize("m", [2, 20, 64])
def test_q8_0_matmul_extreme_quants(aotk, m):
    """Stored bytes of -128 on both sides, whole groups of them among others.
    Scales of 1: every partial sum is an integer below 2^24, so the result is
    the integers' own. (The reference's sign trick wraps on inputs of -128,
    which its quantizer never makes.)"""
    rng = np.random.default_rng(m)
    rows, cols = 33, 288
    w, x = (rng.integers(-128, 128, s, dtype=np.int8) for s in ((rows, cols), (m, cols)))
    w[::3], x[1::2], w[1, ::2], x[0, :40] = -128, -128, 127, 127
    raw = np.concatenate([np.full((rows, cols // 32, 1), 1, np.float16).view(np.uint8), w.view(np.uint8).reshape(rows, -1, 32)], 2)
    acts = np.concatenate([np.full((m, cols // 32, 1), 1, np.float32).view(np.uint8), x.view(np.uint8).reshape(m, -1, 32)], 2)
    h = aotk.Weight(Q8_0, raw.reshape(-1), rows, cols)
    want = x.astype(np.int64) @ w.astype(np.int64).T
    assert np.abs(want).max() == cols * 128 * 128
    assert same_bits(aotk.matmul(h, acts.reshape(-1), m), want.astype(np.float32))
    assert same_bits(aotk.matvec(h, acts[1].reshape(-1)), want[1].astype(np.float32))
    h.free()


@pytest.mark.parametrize("nh,nkv,hd,pos0,m,window", [
    (4, 4, 64, 30, 3, 0), (32, 4, 64, 400, 64, 0), (32, 8, 128, 900, 40, 0), (8, 4, 64, 700, 4, 0), (8, 4, 64, 1500, 4, 0),
    (8, 4, 64, 3000, 4, 0), (8, 2, 128, 200, 20, 64), (8, 4, 256, 90, 21, 0)])
def test_prompt_attention_scores_not_finite(aotk, oracle, nh, nkv, hd, pos0, m, window):
    """Infinite and NaN scores at positions that the rows hold: +inf and NaN
    make a row NaN, -inf leaves the position out, and a kv head of nothing but
    infinities is NaN."""
    rng = np.random.default_rng(pos0 + m)
    ctx = pos0 + m + 3
    q = rng.standard_normal((m, nh, hd)).astype(np.float32)
    kc, vc = (rng.standard_normal((ctx, nkv, hd)).astype(np.float32) for _ in range(2))
    kc[pos0 - 3, 0, 0] = np.inf   # scores of either sign by q's
    kc[pos0 + m - 2, 1, 1] = np.nan  # held by the last two rows
    kc[:, nkv - 1, 2] = -np.inf
    got = aotk.attention(q.reshape(-1), kc.reshape(-1), vc.reshape(-1), nh, nkv, hd, ctx, 0, pos0, m, window)
    ref = attention_ref(oracle, q.reshape(-1), kc.reshape(-1), vc.reshape(-1), nh, nkv, hd, ctx, pos0, m, window)
    assert np.isnan(ref).any() and (np.isfinite(ref.reshape(m, nh, hd)).all(2).any() or nkv == 1)
    assert same_or_nan(got, ref)
