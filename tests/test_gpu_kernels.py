"""GPU kernels at the sizes where their launch shapes change, word for word against the oracle."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

import oracle as O  # noqa: E402
import stwo_hip as S  # noqa: E402


@pytest.mark.parametrize("log_n", [0, 1, 2, 3, 4, 9, 10, 11, 12, 13, 14, 17, 20, 21, 22])
@pytest.mark.parametrize("start", [1, 3, 0x155])
def test_twiddle_tree_levels(log_n, start):
    """One block writes 2^12 values of level 0 and every level above them: sizes below, at and past
    one block, with starting points other than the canonic one."""
    c = S.Coset((start << (29 - log_n)) & 0x7FFFFFFF, (1 << (31 - log_n)) & 0x7FFFFFFF, log_n)
    tree = S.precompute_twiddles(c)
    tw, itw = O.precompute_twiddles(c.initial_index, c.step_size, c.log_size)
    assert (tree.twiddles.to_numpy() == tw).all()
    assert (tree.itwiddles.to_numpy() == itw).all()


def _m31(rng, n):
    """Uniform values with the extremes among them."""
    v = rng.integers(0, S.P, n, dtype=np.uint32)
    v[:: max(1, n // 7)] = S.P - 1
    v[1 :: max(1, n // 5)] = 0
    return v


@pytest.mark.parametrize("log_n,n_cols,blowup", [(10, (1 << 14) + 1, 0), (10, (1 << 12) + 3, 2), (10, 8197, 1),
                                                 (11, 8193, 0), (11, 4099, 1), (12, 4097, 0), (9, 4098, 3),
                                                 (9, 16387, 1), (8, 16385, 2), (10, 16386, 3)])
def test_small_columns_on_matrix_cores(log_n, n_cols, blowup):
    """Batches of small columns large enough for the matrix cores: the number of columns leaves the
    last group partly empty, and columns of the extreme values lie at both ends."""
    rng = np.random.default_rng(log_n * 1000 + n_cols)
    m = log_n + blowup
    picks = [0, 1, 2, 3, n_cols // 2, n_cols - 2, n_cols - 1]
    host = rng.integers(0, S.P, (n_cols, 1 << log_n), dtype=np.uint32)
    host[1][:] = S.P - 1
    host[2][:] = 0
    host[n_cols - 1][::2] = S.P - 1
    src = S.BaseFieldVec.from_numpy(host.reshape(-1))
    dst = S.BaseFieldVec.uninitialized(n_cols << m)
    coset = S.canonic_half_coset(m)
    tw, itw = S.cached_twiddles(coset)
    sp = S._ptr_array([src.ptr + (c << (log_n + 2)) for c in range(n_cols)])
    dp = S._ptr_array([dst.ptr + (c << (m + 2)) for c in range(n_cols)])
    lo, lm = np.full(n_cols, log_n, np.uint32), np.full(n_cols, m, np.uint32)
    L = S.lib()
    S.check(L.stwo_hip_evaluate_columns_async(sp, lo.ctypes.data_as(S.u32p), dp, lm.ctypes.data_as(S.u32p), n_cols,
                                              tw, 1 << coset.log_size))
    S.check(L.stwo_hip_interpolate_columns_async(sp, lo.ctypes.data_as(S.u32p), n_cols, itw, 1 << coset.log_size))
    out, back = dst.to_numpy().reshape(n_cols, -1), src.to_numpy().reshape(n_cols, -1)
    otw, oitw = O.precompute_twiddles(coset.initial_index, coset.step_size, coset.log_size)
    half = S.canonic_half_coset(log_n).initial_index
    for c in picks:
        ext = np.zeros(1 << m, np.uint32)
        ext[: 1 << log_n] = host[c]
        assert (out[c] == O.evaluate(ext, coset.initial_index, otw)).all(), c
        assert (back[c] == O.interpolate(host[c], half, oitw)).all(), c


@pytest.mark.parametrize("log_n,n_cols,blowup", [(17, 385, 1), (18, 193, 1), (19, 97, 1), (20, 49, 1), (18, 193, 2),
                                                 (17, 384, 3)])
def test_extension_on_matrix_cores(log_n, n_cols, blowup):
    """Every number of strided layers (5 .. 8) of the matrix-core extension, at the fewest columns
    that take it and one more than a whole group."""
    rng = np.random.default_rng(log_n + n_cols)
    m = log_n + blowup
    host = {c: rng.integers(0, S.P, 1 << log_n, dtype=np.uint32) for c in (0, 1, n_cols // 2, n_cols - 1)}
    host[1][:] = S.P - 1
    cols = [S.BaseFieldVec.from_numpy(host[c]) if c in host else S.BaseFieldVec.zeros(1 << log_n) for c in range(n_cols)]
    coset = S.canonic_half_coset(m)
    tw, itw = S.cached_twiddles(coset)
    out = [S.BaseFieldVec.uninitialized(1 << m) for _ in range(n_cols)]
    S.lde_columns_async(cols, cols, out, [log_n] * n_cols, blowup, tw, itw, 1 << coset.log_size)
    S.synchronize()
    otw, oitw = O.precompute_twiddles(coset.initial_index, coset.step_size, coset.log_size)
    ocoef, olde = O.lde_columns([host[c] for c in sorted(host)], blowup, otw, oitw)
    for i, c in enumerate(sorted(host)):
        assert (cols[c].to_numpy() == ocoef[i]).all(), c
        assert (out[c].to_numpy() == olde[i]).all(), c


@pytest.mark.parametrize("log_n,n_cols,n_points", [(11, 3, 2), (12, 1, 1), (12, 33, 3), (13, 5, 2), (14, 700, 1),
                                                   (15, 3, 5), (17, 2, 2), (18, 9, 2), (20, 1, 3), (23, 1, 2)])
def test_oods_values(log_n, n_cols, n_points):
    """Batched evaluation at points: one block per column up to the shapes with several ranges per
    column and one, two or more points (the last of an odd number alone); both entry points."""
    rng = np.random.default_rng(log_n * 100 + n_cols)
    host = rng.integers(0, S.P, (n_cols, 1 << log_n), dtype=np.uint32)
    host[0][:] = S.P - 1
    cols = [S.BaseFieldVec.from_numpy(h) for h in host]
    pts = [S.random_circle_point_qm31(rng) for _ in range(n_points)]
    got = S.eval_at_points_columns(cols, pts)
    assert got == S.eval_at_points_columns(cols, pts, noalloc=True)
    for c in {0, n_cols // 2, n_cols - 1}:
        for k in range(n_points):
            assert got[k][c] == tuple(int(v) for v in O.eval_at_point(host[c], *pts[k])), (c, k)


@pytest.mark.parametrize("log_n,n_cols,n_batches", [(1, 200, 1), (2, 17, 3), (5, 30, 2), (6, 13, 4), (7, 250, 1), (8, 16, 3),
                                                    (9, 33, 4), (11, 70, 2), (12, 5, 3), (10, 700, 1),
                                                    (9, 188, 1), (9, 190, 1), (4, 12400, 1)])
def test_quotients_on_matrix_cores(log_n, n_cols, n_batches):
    """Domains smaller than a wave's rows and larger than a block's, column counts that leave the
    last step partly empty, one and two operand tiles, the sample counts at which the form
    changes; extreme column values; a column sampled twice at one point."""
    rng = np.random.default_rng(log_n * 1000 + n_cols)
    host = [rng.integers(0, S.P, 1 << log_n, dtype=np.uint32) for _ in range(n_cols)]
    host[0][:] = S.P - 1
    cols = [S.BaseFieldVec.from_numpy(h) for h in host]
    batches = []
    for b in range(n_batches):
        cs = [c for c in range(n_cols) if (c + b) % 3 != 1 or c == 0]
        batches.append((S.random_circle_point_qm31(rng), [(c, S.random_qm31(rng)) for c in cs]))
    batches[0][1].append((0, S.random_qm31(rng)))
    rc = S.random_qm31(rng)
    dom = S.canonic_half_coset(log_n)
    out = S.SecureColumn.uninitialized(1 << log_n)
    S.accumulate_quotients_async(dom, cols, rc, S.QuotientSamples(batches), out)
    want = O.accumulate_quotients(dom.initial_index, dom.step_size, log_n, host, rc, batches)
    assert (out.to_numpy() == want).all()
    assert (S.accumulate_quotients(dom, cols, rc, batches).to_numpy() == want).all()


@pytest.mark.parametrize("log_n", [13, 14, 15, 18])
@pytest.mark.parametrize("offset", [1, 2, 3])
def test_bit_reverse_at_word_aligned_columns(log_n, offset):
    """Columns that start at any word: 16-byte accesses off their alignment, and nothing beyond the
    column's ends touched."""
    data = np.arange((1 << log_n) + 8, dtype=np.uint32)
    col = S.BaseFieldVec.from_numpy(data)
    S.lib().bit_reverse_base_field(col.ptr + 4 * offset, 1 << log_n)
    S.check()
    want = data.copy()
    want[offset:offset + (1 << log_n)] = O.bit_reverse(data[offset:offset + (1 << log_n)].copy())
    assert (col.to_numpy() == want).all()


@pytest.mark.parametrize("sizes", [[k] * 4 for k in range(15)] + [[16] * 20 + [15, 7], [17] * 4 + [16, 8, 7, 7, 6],
                                                                  [12] * 4 + [7] * 3 + [5] + [4] * 2, [9] * 17 + [8, 0]])
def test_merkle_subtree_launches(sizes):
    """Trees of every height that one or two subtree launches build: launches whose last block goes on
    above the other blocks' roots, and launches that start from another launch's nodes, with columns
    injected at their first level and above.  Twice: the arrival counters are left as they were."""
    rng = np.random.default_rng(sum(sizes) + len(sizes))
    host = [rng.integers(0, S.P, 1 << k, dtype=np.uint32) for k in sizes]
    cols = [S.BaseFieldVec.from_numpy(h) for h in host]
    want = O.merkle_commit(host)
    for _ in range(2):
        tree = S.MerkleTree(cols).commit_async()
        for k, layer in enumerate(tree.layers):
            assert (layer.to_numpy().reshape(-1) == want[k].reshape(-1)).all(), k


@pytest.mark.parametrize("n", [1, 255, 2049, 1 << 20, (1 << 24) - 3, (1 << 24) + 1])
def test_batch_inverse_secure_field_sizes(n):
    """Sizes at which the kernel changes and blocks end; extreme values and zeros among the inputs."""
    rng = np.random.default_rng(n)
    data = rng.integers(0, S.P, (n, 4), dtype=np.uint32)
    for k, row in enumerate([(0, 0, 0, 0), (S.P - 1,) * 4, (0, 0, S.P - 1, 1), (0, S.P - 1, 0, 0), (1, 0, 0, 0)]):
        data[(k * 37) % n] = row
    dst = S.SecureFieldVec.uninitialized(n)
    S.batch_inverse(S.SecureFieldVec.from_numpy(data), dst)
    got = dst.to_numpy().reshape(-1, 4)
    # x * (1 / x) = 1, in 64 bits: (a + b u)(c + d u) with u^2 = R = 2 + i over CM31
    P = np.uint64(S.P)

    def cm(x, y):
        return ((x[0] * y[0] % P + (P - x[1] * y[1] % P)) % P, (x[0] * y[1] % P + x[1] * y[0] % P) % P)

    x, y = data.astype(np.uint64).T, got.astype(np.uint64).T
    xx, yy = cm(x[:2], y[:2]), cm(x[2:], y[2:])
    xy, yx = cm(x[:2], y[2:]), cm(x[2:], y[:2])
    r = ((P + P + yy[0] + yy[0] - yy[1]) % P, (yy[0] + yy[1] + yy[1]) % P)
    prod = [(xx[0] + r[0]) % P, (xx[1] + r[1]) % P, (xy[0] + yx[0]) % P, (xy[1] + yx[1]) % P]
    zero = (data == 0).all(axis=1)
    assert (prod[0] == np.where(zero, 0, 1)).all()
    assert all((p == 0).all() for p in prod[1:])
    assert (got[zero] == 0).all()


@pytest.mark.parametrize("words,offset", [(1, 0), (1, 3), (255, 1), (257, 0), (1 << 14, 0), ((1 << 14) + 1, 2), (1 << 16, 1)])
def test_copies_to_host_memory(words, offset):
    """Either side of the size up to which a kernel copies, at any word of a buffer, right behind the
    work that wrote it; and copies whose ends are other kinds of memory."""
    data = np.arange(words + offset, dtype=np.uint32) * np.uint32(2654435761)
    col = S.BaseFieldVec.from_numpy(data)
    out = np.zeros(words + 1, np.uint32)
    S.lib().copy_uint32_t_vec_from_device_to_host(col.ptr + 4 * offset, out.ctypes.data, words)
    S.check()
    assert (out[:words] == data[offset:]).all() and out[words] == 0
    other = S.BaseFieldVec.uninitialized(words)
    S.check(S.lib().stwo_hip_memcpy(other.ptr, col.ptr + 4 * offset, 4 * words))
    back = np.zeros(words, np.uint32)
    S.check(S.lib().stwo_hip_memcpy(back.ctypes.data, other.ptr, 4 * words))
    assert (back == data[offset:]).all()
    S.check(S.lib().stwo_hip_memcpy(other.ptr, data.ctypes.data, 4 * words))
    assert (other.to_numpy() == data[:words]).all()
    S.check(S.lib().stwo_hip_memcpy(back.ctypes.data, data.ctypes.data, 4 * words))
    assert (back == data[:words]).all()
