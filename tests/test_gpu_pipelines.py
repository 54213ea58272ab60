"""The reference pipelines' matvec, router matvec and attention kernels at
the edges of their dispatch rules (styx_amd/csrc/kernels_ref.hip): row
lengths around the lane groups, rows past the last pass, head groups that do
not fill 16 rows, contexts around the split.  Against the oracle's f64
results; matvecs within the f32 forward-error bound for any summation order
(cols 2^-24 sum |w x|), attention within 2e-6 relative L2 (the bound the
paged attention tests use)."""
from __future__ import annotations

import struct

import numpy as np
import pytest

from helpers import clamp_f16_exponents, rel_l2
from oracle import oracle as O
from test_gpu_dispatch import BLK, F16_AT, NAME, f32buf, mmv_id_push, run, sum_bound

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def gpu():
    from styx_amd import Gpu
    g = Gpu(0)
    yield g
    g.close()


def weights(t, rows, cols, seed):
    be, bb = BLK[t]
    a = np.random.default_rng(seed).integers(0, 256, rows * (cols // be) * bb).astype(np.uint8)
    clamp_f16_exponents(a, bb, F16_AT[t])
    return a


# lanes per row 1..64, one and two units per lane, rows longer than 128 units
@pytest.mark.parametrize("t,rows,cols", [(8, 7, 32), (8, 130, 96), (8, 513, 2080), (8, 66, 6176),
                                         (12, 9, 256), (12, 5001, 768), (12, 70, 4608),
                                         (13, 33, 2304), (13, 259, 4096), (14, 65, 1280),
                                         (14, 1030, 2048), (14, 35, 8192)])
def test_matvec_rows(gpu, t, rows, cols):
    be, _ = BLK[t]
    a = weights(t, rows, cols, rows + cols)
    x = np.random.default_rng(1).standard_normal(cols).astype(np.float32)
    guard = 5
    bd = f32buf(gpu, np.full(rows + guard, 9.0))
    push = struct.pack("<13I", cols, cols // be, cols, rows, rows * cols, cols, rows, 0, 0, 1, 1, 1, 1)
    run(gpu, f"mul_mat_vec_{NAME[t]}_f32_f32", [gpu.from_numpy(a), f32buf(gpu, x), bd, gpu.zeros(16),
                                               gpu.zeros(16)], push, (rows, 1, 1), [(1, 1)])
    got = bd.download(np.float32)
    y = O.matvec_f64(t, a, rows, cols, x)
    assert (np.abs(got[:rows] - y) <= sum_bound(t, a, rows, cols, x)).all()
    assert (got[rows:] == 9.0).all()


def matvec(gpu, t, a, rows, cols, x):
    be, _ = BLK[t]
    bd = gpu.zeros(rows * 4)
    push = struct.pack("<13I", cols, cols // be, cols, rows, rows * cols, cols, rows, 0, 0, 1, 1, 1, 1)
    run(gpu, f"mul_mat_vec_{NAME[t]}_f32_f32", [gpu.from_numpy(a), f32buf(gpu, x), bd, gpu.zeros(16),
                                               gpu.zeros(16)], push, (rows, 1, 1), [(1, 1)])
    return bd.download(np.float32)


@pytest.mark.parametrize("t", [8, 12, 13, 14])
@pytest.mark.parametrize("cols", [256, 2048, 8192])
def test_matvec_of_activations_around_one(gpu, t, cols):
    """Nothing cancels but what the weights themselves cancel: a lane adds
    its values in a tree of 4 levels, its units in turn, the lanes in 6
    levels, about 16 roundings of random sign in a row: sqrt(16) 2^-24 of the
    result's norm at most.  (With 32 taken off q6_K's sums instead of its
    values the error was 5e-7.)"""
    rows = 512
    a = weights(t, rows, cols, cols + t)
    x = (1 + 0.1 * np.random.default_rng(t).standard_normal(cols)).astype(np.float32)
    assert rel_l2(matvec(gpu, t, a, rows, cols, x), O.matvec_f64(t, a, rows, cols, x)) < 4 * 2.0 ** -24


@pytest.mark.parametrize("t", [8, 12, 13, 14])
@pytest.mark.parametrize("big", [np.inf, -np.inf, 3e38])
def test_matvec_of_an_infinite_or_huge_activation(gpu, t, big):
    """As the products of the dequantized weights: an infinity where the
    weight is not zero, NaN where it is; a value that fits f32 where the
    product does."""
    rows, cols = 512, 768
    a = weights(t, rows, cols, 5 + t)
    x = np.random.default_rng(3).standard_normal(cols).astype(np.float32)
    x[77] = big
    got = matvec(gpu, t, a, rows, cols, x)
    w = O.dequant(t, a, rows * cols).reshape(rows, cols)[:, 77].astype(np.float64)
    if np.isinf(big):
        assert (np.isnan(got) == (w == 0)).all()
        assert (got[w != 0] == np.sign(w[w != 0]) * big).all()
    else:
        y, top = w * float(np.float32(big)), float(np.finfo(np.float32).max)
        fits, over = np.abs(y) < 0.999 * top, np.abs(y) > 1.001 * top
        assert fits.any() and over.any() and np.isfinite(got[fits]).all()
        assert (got[over] == np.sign(y[over]) * np.inf).all()
        assert (np.abs(got[fits] - y[fits]) <= 1e-6 * np.abs(y[fits]) + 1e30).all()


# two passes of rows per lane group and a ragged last one: one, two and more
# units per lane
@pytest.mark.parametrize("t,rows,cols", [(8, 4099, 2048), (12, 4100, 4096), (13, 4104, 4608), (14, 4101, 4608),
                                         (14, 4099, 2048), (12, 8209, 1024)])
def test_matvec_several_passes(gpu, t, rows, cols):
    test_matvec_rows(gpu, t, rows, cols)


def test_matvec_id_several_passes(gpu):
    """8 slots x 2049 rows of 16 lanes: two passes, the last of one row."""
    t, E, rows, cols, k = 14, 3, 2049, 512, 8
    be, bb = BLK[t]
    a = weights(t, E * rows, cols, 21)
    x = np.random.default_rng(4).standard_normal(cols).astype(np.float32)
    ids = np.array([2, 0, 1, 1, 0, 2, 2, 1], np.int32)
    bd = f32buf(gpu, np.full(k * rows + 5, 9.0))
    run(gpu, f"mul_mat_vec_id_{NAME[t]}_f32_f32",
        [gpu.from_numpy(a), f32buf(gpu, x), bd, gpu.zeros(16), gpu.zeros(16), gpu.from_numpy(ids)],
        mmv_id_push(cols, rows, be, k), (rows, k, 1))
    got = bd.download(np.float32)
    n = rows * (cols // be) * bb
    for s, e in enumerate(ids):
        w = a[e * n:(e + 1) * n]
        assert (np.abs(got[s * rows:(s + 1) * rows] - O.matvec_f64(t, w, rows, cols, x))
                <= sum_bound(t, w, rows, cols, x)).all()
    assert (got[k * rows:] == 9.0).all()


def test_matvec_grid_covers_part_of_the_rows(gpu):
    """NUM_ROWS rows per workgroup of the reference grid, and no row past it."""
    t, rows, cols = 12, 64, 512
    a = weights(t, rows, cols, 3)
    x = np.random.default_rng(2).standard_normal(cols).astype(np.float32)
    bd = f32buf(gpu, np.full(rows, 9.0))
    push = struct.pack("<13I", cols, 2, cols, rows, rows * cols, cols, rows, 0, 0, 1, 1, 1, 1)
    run(gpu, "mul_mat_vec_q4_k_f32_f32", [gpu.from_numpy(a), f32buf(gpu, x), bd, gpu.zeros(16),
                                          gpu.zeros(16)], push, (10, 1, 1), [(1, 4)])
    got = bd.download(np.float32)
    y = O.matvec_f64(t, a, rows, cols, x)
    assert (np.abs(got - y)[:40] <= sum_bound(t, a, rows, cols, x)[:40]).all()
    assert (got[40:] == 9.0).all()


@pytest.mark.parametrize("t", [8, 12, 13, 14])
def test_matvec_id_odd_stride(gpu, t):
    """Activations a whole odd number of floats apart (4-byte aligned rows)."""
    be, bb = BLK[t]
    E, rows, cols, k, stride = 5, 37, 512, 3, 515
    a = weights(t, E * rows, cols, 9 + t)
    x = np.random.default_rng(4).standard_normal(k * stride).astype(np.float32)
    bd = gpu.zeros(k * rows * 4)
    ids = gpu.from_numpy(np.array([4, 0, 2], np.int32))
    push = struct.pack("<12I", cols, cols // be, stride, rows, rows * cols, 0, k * rows, 0, k, k, 0, 1)
    run(gpu, f"mul_mat_vec_id_{NAME[t]}_f32_f32", [gpu.from_numpy(a), f32buf(gpu, x), bd, gpu.zeros(16),
                                                  gpu.zeros(16), ids], push, (rows, k, 1))
    got = bd.download(np.float32).reshape(k, rows)
    n = rows * (cols // be) * bb
    for s, e in enumerate([4, 0, 2]):
        xs = x[s * stride:s * stride + cols]
        w = a[e * n:(e + 1) * n]
        assert (np.abs(got[s] - O.matvec_f64(t, w, rows, cols, xs)) <= sum_bound(t, w, rows, cols, xs)).all()


@pytest.mark.parametrize("E,H,stride", [(1, 3, 3), (17, 259, 261), (16, 2048, 2048), (33, 2563, 2567),
                                        (8, 4352, 4352)])
def test_matvec_strided_shapes(gpu, E, H, stride):
    rng = np.random.default_rng(H)
    W = rng.standard_normal(E * stride).astype(np.float32)
    x = rng.standard_normal(H).astype(np.float32)
    bd = gpu.zeros(E * 4)
    run(gpu, "matvec_strided_f32", [f32buf(gpu, W), f32buf(gpu, x), bd], struct.pack("<2I", H, stride),
        (E, 1, 1))
    Wd = W.reshape(E, stride)[:, :H].astype(np.float64)
    bound = H * 2.0 ** -24 * (np.abs(Wd) @ np.abs(x.astype(np.float64)))
    assert (np.abs(bd.download(np.float32, E) - Wd @ x.astype(np.float64)) <= bound).all()


# contexts around a key block (32), a workgroup's pass (128), the split (256)
# and past one chunk per workgroup; 1..20 heads per kv head, and a head count
# that leaves the last kv head's group short; rows of an odd stride
@pytest.mark.parametrize("n_t,hd,nh,gqa,pad", [
    (1, 64, 4, 1, 0), (31, 128, 8, 8, 0), (33, 256, 6, 3, 0), (129, 64, 20, 20, 0), (256, 128, 32, 8, 0),
    (257, 128, 32, 8, 0), (300, 256, 16, 16, 0), (1000, 64, 7, 4, 0), (1023, 128, 10, 5, 1),
    (9000, 64, 2, 1, 0), (700, 96, 8, 4, 0),
    # the longest contexts of the general kernel and one key more
    (2, 64, 8, 4, 1), (3, 64, 8, 4, 1), (4, 128, 32, 8, 0), (5, 128, 32, 8, 0), (8, 256, 6, 3, 0), (9, 256, 6, 3, 0)])
def test_attn_decode_shapes(gpu, n_t, hd, nh, gqa, pad):
    rng = np.random.default_rng(n_t + hd)
    nkv = -(-nh // gqa)
    kvd = nkv * hd + pad
    q = rng.standard_normal(nh * hd).astype(np.float32)
    K = rng.standard_normal(n_t * kvd).astype(np.float32)
    V = rng.standard_normal(n_t * kvd).astype(np.float32)
    scale = np.float32(1 / np.sqrt(hd))
    bo = f32buf(gpu, np.full(nh * hd + 8, 3.0))
    run(gpu, "attn_decode_f32", [f32buf(gpu, q), f32buf(gpu, K), f32buf(gpu, V), bo],
        struct.pack("<4If", n_t, hd, kvd, gqa, scale), (nh, 1, 1))
    got = bo.download(np.float32)
    ref = O.attn_decode_f64(q, K, V, n_t, hd, kvd, gqa, nh, float(scale))
    assert rel_l2(got[:nh * hd], ref) < 2e-6
    assert (got[nh * hd:] == 3.0).all()


def test_attn_decode_overlapping_rows_and_the_largest_context(gpu):
    """kv_dim 0: every key is the same row, whatever n_t says, up to 2^32 - 1
    (key positions in 64 bits; counted in 32 the last blocks never ended)."""
    hd, nh = 64, 4
    rng = np.random.default_rng(0)
    q, K, V = (rng.standard_normal(n).astype(np.float32) for n in (nh * hd, hd, hd))
    for n_t in (5, 300, 70001, 2 ** 32 - 1):
        bo = gpu.zeros(nh * hd * 4)
        run(gpu, "attn_decode_f32", [f32buf(gpu, q), f32buf(gpu, K), f32buf(gpu, V), bo],
            struct.pack("<4If", n_t, hd, 0, nh, 0.125), (nh, 1, 1))
        # every key adds the same value, so roundings do not average: a wave
        # adds up its blocks in turn (at most 512 chunks, 4 waves, 32 keys),
        # then come 32 keys within a block, 4 waves and the chunks
        adds = n_t / (512 * 4 * 32) + 32 + 4 + 512
        assert rel_l2(bo.download(np.float32).reshape(nh, hd), np.tile(V, (nh, 1))) < adds * 2.0 ** -24, n_t


# contexts that end inside a key block, one and several chunks
@pytest.mark.parametrize("n_t,hd,gqa", [(1, 64, 1), (31, 128, 4), (32, 128, 4), (33, 256, 2), (257, 64, 8),
                                        (600, 128, 4)])
@pytest.mark.parametrize("at", [0, -1])
def test_attn_decode_infinite_value(gpu, n_t, hd, gqa, at):
    """An infinity in the first or last V row: an infinity in that dimension
    of the heads that read it, every other output as without."""
    rng = np.random.default_rng(n_t)
    nh, kvd, scale = 2 * gqa, 2 * hd, np.float32(1 / np.sqrt(hd))
    q, K, V = (rng.standard_normal(n).astype(np.float32) for n in (nh * hd, n_t * kvd, n_t * kvd))
    ref = O.attn_decode_f64(q, K, V, n_t, hd, kvd, gqa, nh, float(scale)).reshape(nh, hd)
    V.reshape(n_t, kvd)[at, 3] = -np.inf
    bo = gpu.zeros(nh * hd * 4)
    run(gpu, "attn_decode_f32", [f32buf(gpu, q), f32buf(gpu, K), f32buf(gpu, V), bo],
        struct.pack("<4If", n_t, hd, kvd, gqa, scale), (nh, 1, 1))
    got = bo.download(np.float32).reshape(nh, hd)
    assert (got[:gqa, 3] == -np.inf).all()
    got[:gqa, 3] = ref[:gqa, 3] = 0
    assert rel_l2(got, ref) < 2e-6


def test_attn_in_async_and_plain_batches(gpu):
    """Split contexts on two streams at once: each batch has its own partials."""
    from styx_amd.runtime import Batch, Kernel, Timeline
    rng = np.random.default_rng(8)
    n_t, hd, nh, nkv = 2000, 128, 8, 2
    kvd, scale = nkv * hd, np.float32(1 / np.sqrt(hd))
    push = struct.pack("<4If", n_t, hd, kvd, nh // nkv, scale)
    k = Kernel(gpu, "attn_decode_f32", [])
    t, ab, mb = Timeline(gpu), Batch(gpu, is_async=True), Batch(gpu)
    sets = []
    for _ in range(2):
        q, K, V = (rng.standard_normal(n).astype(np.float32) for n in (nh * hd, n_t * kvd, n_t * kvd))
        ref = O.attn_decode_f64(q, K, V, n_t, hd, kvd, nh // nkv, nh, float(scale))
        sets.append(([f32buf(gpu, q), f32buf(gpu, K), f32buf(gpu, V), gpu.zeros(nh * hd * 4)], ref))
    for rnd in range(4):
        ab.begin()
        mb.begin()
        for _ in range(4):
            ab.dispatch(k, sets[0][0], push, (nh, 1, 1))
            mb.dispatch(k, sets[1][0], push, (nh, 1, 1))
        ab.submit_async(t, rnd + 1)
        mb.submit()
        ab.wait_idle()
        for binds, ref in sets:
            assert rel_l2(binds[3].download(np.float32), ref) < 2e-6
    for o in (ab, mb, k, t):
        o.free()


def test_freeing_an_async_batch_waits_for_its_own_stream_only(gpu):
    """A batch that ran attention is freed while another batch's work runs on
    (freeing its partials to the device would wait for that)."""
    import time
    from styx_amd.runtime import Batch, Kernel, Timeline
    rows, cols, n_t, hd = 16384, 8192, 2000, 128
    a = [gpu.zeros(rows * cols // 32 * 34), f32buf(gpu, np.ones(cols)), gpu.zeros(rows * 4), gpu.zeros(16),
         gpu.zeros(16)]
    mv, at, t = Kernel(gpu, "mul_mat_vec_q8_0_f32_f32", [(1, 1)]), Kernel(gpu, "attn_decode_f32", []), Timeline(gpu)
    push = struct.pack("<13I", cols, cols // 32, cols, rows, rows * cols, cols, rows, 0, 0, 1, 1, 1, 1)
    kv = [gpu.zeros(hd * 4), gpu.zeros(n_t * hd * 4), gpu.zeros(n_t * hd * 4), gpu.zeros(hd * 4)]
    work, b = Batch(gpu, is_async=True), Batch(gpu, is_async=True)
    b.begin()
    b.dispatch(at, kv, struct.pack("<4If", n_t, hd, hd, 1, 0.1), (1, 1, 1))
    b.submit_async(t, 1)
    b.wait_idle()
    work.begin()
    for _ in range(600):  # about 45 ms
        work.dispatch(mv, a, push, (rows, 1, 1))
    work.submit_async(t, 2)
    t0 = time.perf_counter()
    b.free()
    t1 = time.perf_counter()
    work.wait_idle()
    t2 = time.perf_counter()
    for o in (work, mv, at, t):
        o.free()
    assert t1 - t0 < 0.5 * (t2 - t1), (t1 - t0, t2 - t1)


# op matvec: limbs built by the workgroups (up to 2048 columns, or few rows)
# or by a launch in front (long rows of many rows, outputs over the input)
@pytest.mark.parametrize("t,rows,cols", [(8, 40, 32), (8, 33, 2048), (8, 16, 2112), (12, 64, 4096),
                                         (14, 4096, 3072), (14, 4098, 3072), (13, 24, 8192),
                                         (12, 2048, 4352), (12, 2050, 4352), (12, 2050, 4096)])
@pytest.mark.parametrize("norm", [False, True])
def test_op_matvec_against_f64(gpu, t, rows, cols, norm):
    import ctypes as C
    from styx_amd import _lib as L
    from styx_amd.runtime import to_split
    a = weights(t, rows, cols, rows)
    rng = np.random.default_rng(cols)
    x = rng.standard_normal(cols).astype(np.float32)
    nw = (1 + 0.1 * rng.standard_normal(cols)).astype(np.float32)
    w = to_split(gpu, t, gpu.from_numpy(a), rows, cols)
    bx, bn, by = f32buf(gpu, x), f32buf(gpu, nw), gpu.zeros(rows * 4)
    L.check(gpu.lib.styx_op_matvec(gpu.h, t, w.ptr, rows, cols, bx.ptr, bn.ptr if norm else None,
                                   C.c_float(1e-6), by.ptr, 0))
    gpu.sync()
    xd = x.astype(np.float64)
    xn = (xd / np.sqrt((xd ** 2).mean() + 1e-6) * nw) if norm else xd
    y = O.matvec_f64(t, a, rows, cols, xn.astype(np.float32))
    bound = sum_bound(t, a, rows, cols, xn.astype(np.float32)) + 1e-6 * np.abs(y).max()
    assert (np.abs(by.download(np.float32, rows) - y) <= bound).all()


# limbs built by the workgroups, or by a launch in front: past 4096 rows of
# more than 4096 columns, and past 3 2^25 q4_K weights of more than 2048
@pytest.mark.parametrize("t,H,F,k", [(14, 8192, 512, 4), (14, 8192, 768, 4), (8, 4352, 512, 4), (8, 4352, 544, 4),
                                     (12, 4096, 768, 16), (12, 4096, 776, 16), (12, 2048, 1600, 16)])
def test_op_gate_up_against_f64(gpu, t, H, F, k):
    import ctypes as C
    from styx_amd import _lib as L
    from styx_amd.runtime import to_split
    E = 2
    be, bb = BLK[t]
    w = [weights(t, E * F, H, t + H + i) for i in (0, 1)]
    split = [to_split(gpu, t, gpu.from_numpy(a), F, H, E) for a in w]
    slab = F * (H // be) * bb
    src = [L.ExpertSrc(hot=s.ptr, hot_slab=slab) for s in split]
    x = np.random.default_rng(H).standard_normal(H).astype(np.float32)
    sel = np.random.default_rng(F).integers(0, E, k)
    ids = np.full(64, -1, np.int32)
    ids[:k] = ids[16:16 + k] = sel
    bx, bi, gu = f32buf(gpu, x), gpu.from_numpy(ids), gpu.zeros(2 * k * F * 4)
    L.check(gpu.lib.styx_op_moe_gate_up(gpu.h, t, t, C.byref(src[0]), C.byref(src[1]), bi.ptr, bx.ptr, gu.ptr,
                                        H, F, k))
    gpu.sync()
    got = gu.download(np.float32).reshape(2, k, F)
    for m in (0, 1):
        y = [O.matvec_f64(t, w[m][e * slab:(e + 1) * slab], F, H, x) for e in range(E)]
        bound = [sum_bound(t, w[m][e * slab:(e + 1) * slab], F, H, x) + 1e-6 * np.abs(y[e]).max() for e in range(E)]
        for s, e in enumerate(sel):
            assert (np.abs(got[m, s] - y[e]) <= bound[e]).all(), (m, s)


def test_op_matvec_in_place(gpu):
    """y over x: the product of the old x, as with the limbs formed first."""
    import ctypes as C
    from styx_amd import _lib as L
    from styx_amd.runtime import to_split
    t, n = 8, 2048
    a = weights(t, n, n, 77)
    x = np.random.default_rng(6).standard_normal(n).astype(np.float32)
    w = to_split(gpu, t, gpu.from_numpy(a), n, n)
    apart, inplace, by = f32buf(gpu, x), f32buf(gpu, x), gpu.zeros(n * 4)
    f = gpu.lib.styx_op_matvec
    L.check(f(gpu.h, t, w.ptr, n, n, apart.ptr, None, C.c_float(0.0), by.ptr, 0))
    L.check(f(gpu.h, t, w.ptr, n, n, inplace.ptr, None, C.c_float(0.0), inplace.ptr, 0))
    gpu.sync()
    assert np.array_equal(by.download(np.float32), inplace.download(np.float32))


@pytest.mark.parametrize("E,k", [(16, 4), (64, 16), (65, 8), (200, 10), (512, 10)])
def test_topk_ties_and_unordered_entries(gpu, E, k):
    """Ties keep the lower index; -inf and NaN entries are never picked."""
    lg = np.random.default_rng(E).integers(-3, 4, E).astype(np.float32)
    lg[1], lg[5] = -np.inf, -0.0
    bw, bi = gpu.zeros(64), gpu.from_numpy(np.full(64, -7, np.int32))
    ident = gpu.from_numpy(np.arange(E, dtype=np.uint32))
    skip = gpu.from_numpy(np.full(E, SKIP, np.uint32))

    def go(v):
        run(gpu, "topk_softmax_f32", [f32buf(gpu, v), bw, bi, ident, skip], struct.pack("<3I", E, k, 1),
            (1, 1, 1))
        return bi.download(np.int32, 16 + k), bw.download(np.float32, k)
    ids, w = go(lg)
    w_ref, ids_ref = O.topk_softmax(lg, k, True, None, None)
    assert np.array_equal(ids[:k], ids_ref[:k]) and np.array_equal(ids[16:16 + k], ids_ref[:k])
    assert rel_l2(w, w_ref) < 1e-6
    nan = lg.copy()
    nan[ids[0]] = np.nan
    got, _ = go(nan)
    order = [e for e in sorted(range(E), key=lambda e: (-lg[e], e)) if e != ids[0]][:k]
    assert got[:k].tolist() == order


SKIP = 0xFFFFFFFF
