"""Which kernels a call runs, and its results at the sizes where that changes: the results of both forms
are the same words, so the launches are counted too."""
import contextlib

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

import oracle as O  # noqa: E402
import refmath as R  # noqa: E402
import stwo_hip as S  # noqa: E402


@contextlib.contextmanager
def launches(*names):
    """Counts of the named launches inside the block, filled in at its end."""
    got = {}
    S.kernel_stats_reset()
    S.kernel_timing(True)
    try:
        yield got
        S.synchronize()
        got.update({k: S.kernel_stats(k)[0] for k in names})
    finally:
        S.kernel_timing(False)


def _filled(words, seed, column):
    """A buffer of uniform values; the second column of `column` words holds the largest value throughout,
    the last every other one."""
    v = S.BaseFieldVec.uninitialized(words)
    S.fill_uniform(v, seed)
    most = np.full(column, S.P - 1, np.uint32)
    S.check(S.lib().stwo_hip_memcpy(v.ptr + 4 * column, most.ctypes.data, 4 * column))
    most[::2] = 0
    S.check(S.lib().stwo_hip_memcpy(v.ptr + 4 * (words - column), most.ctypes.data, 4 * column))
    return v


def _part(v, first, n):
    return S.BaseFieldVec.view(v.ptr + 4 * first, n).to_numpy()


def _pointers(v, n_cols, words):
    return S._ptr_array([v.ptr + 4 * words * c for c in range(n_cols)])


# whole small columns: values from which the matrix cores take them, in millions (2^20)
FORWARD = {(log, b): (32, 36, 48, 80)[b] for log in (10, 11, 12) for b in range(4)}
FORWARD[10, 3] = 64


@pytest.mark.parametrize("log_m,blowup", sorted(FORWARD))
def test_evaluation_either_side_of_the_line(log_m, blowup):
    """The fewest columns that take the matrix cores plus a remainder of a group, and one column less
    than the line, into other columns."""
    line = (FORWARD[log_m, blowup] << 20) >> log_m
    log_n = log_m - blowup
    coset = S.canonic_half_coset(log_m)
    tw, _ = S.cached_twiddles(coset)
    otw, _ = O.precompute_twiddles(coset.initial_index, coset.step_size, coset.log_size)
    for n_cols, on_matrices in ((line + 1, 1), (line - 1, 0)):
        src, dst = _filled(n_cols << log_n, 3 * log_m + blowup, 1 << log_n), S.BaseFieldVec.uninitialized(n_cols << log_m)
        logs = np.full(n_cols, log_n, np.uint32), np.full(n_cols, log_m, np.uint32)
        with launches("fft_matrices", "fft_fwd_tile") as got:
            S.check(S.lib().stwo_hip_evaluate_columns_async(
                _pointers(src, n_cols, 1 << log_n), logs[0].ctypes.data_as(S.u32p), _pointers(dst, n_cols, 1 << log_m),
                logs[1].ctypes.data_as(S.u32p), n_cols, tw, 1 << coset.log_size))
        assert got["fft_matrices"] == on_matrices
        for c in (0, 1, n_cols // 2, n_cols - 2, n_cols - 1):
            ext = np.zeros(1 << log_m, np.uint32)
            ext[: 1 << log_n] = _part(src, c << log_n, 1 << log_n)
            assert (_part(dst, c << log_m, 1 << log_m) == O.evaluate(ext, coset.initial_index, otw)).all(), c


@pytest.mark.parametrize("log_n", [10, 11, 12])
@pytest.mark.parametrize("in_place", [True, False])
def test_interpolation_either_side_of_the_line(log_n, in_place):
    line = ((24 if in_place else 36) << 20) >> log_n
    coset = S.canonic_half_coset(log_n)
    _, itw = S.cached_twiddles(coset)
    _, oitw = O.precompute_twiddles(coset.initial_index, coset.step_size, coset.log_size)
    for n_cols, on_matrices in ((line + 1, 1), (line - 1, 0)):
        src = _filled(n_cols << log_n, log_n, 1 << log_n)
        dst = src if in_place else S.BaseFieldVec.uninitialized(n_cols << log_n)
        picks = (0, 1, n_cols // 2, n_cols - 2, n_cols - 1)
        before = [_part(src, c << log_n, 1 << log_n) for c in picks]
        logs = np.full(n_cols, log_n, np.uint32).ctypes.data_as(S.u32p)
        sp, dp = _pointers(src, n_cols, 1 << log_n), _pointers(dst, n_cols, 1 << log_n)
        with launches("fft_matrices") as got:
            if in_place:
                S.check(S.lib().stwo_hip_interpolate_columns_async(sp, logs, n_cols, itw, 1 << coset.log_size))
            else:
                S.check(S.lib().stwo_hip_interpolate_columns_oop_async(sp, dp, logs, n_cols, itw, 1 << coset.log_size))
        assert got["fft_matrices"] == on_matrices
        for c, v in zip(picks, before):
            assert (_part(dst, c << log_n, 1 << log_n) == O.interpolate(v, coset.initial_index, oitw)).all(), c


@pytest.mark.parametrize("log_n,blowup", [(10, 1), (11, 1), (12, 0), (9, 2)])
def test_extension_of_small_columns(log_n, blowup):
    """Extensions whose two halves take different forms: the inverse on butterflies, the forward half on
    matrices or both on matrices."""
    log_m = log_n + blowup
    n_cols = max((FORWARD[log_m, blowup] << 20) >> log_m, 1) + 1
    src, dst = _filled(n_cols << log_n, log_n, 1 << log_n), S.BaseFieldVec.uninitialized(n_cols << log_m)
    picks = (0, n_cols // 2, n_cols - 1)
    before = [_part(src, c << log_n, 1 << log_n) for c in picks]
    coset = S.canonic_half_coset(log_m)
    tw, itw = S.cached_twiddles(coset)
    sp, dp = _pointers(src, n_cols, 1 << log_n), _pointers(dst, n_cols, 1 << log_m)
    logs = np.full(n_cols, log_n, np.uint32).ctypes.data_as(S.u32p)
    with launches("fft_matrices") as got:
        S.check(S.lib().stwo_hip_lde_columns_async(sp, sp, dp, logs, n_cols, blowup, tw, itw, 1 << coset.log_size))
    inverse = 10 <= log_n and (n_cols << log_n) >= 36 << 20
    assert got["fft_matrices"] == 1 + inverse
    otw, oitw = O.precompute_twiddles(coset.initial_index, coset.step_size, coset.log_size)
    ocoef, olde = O.lde_columns(before, blowup, otw, oitw)
    for i, c in enumerate(picks):
        assert (_part(src, c << log_n, 1 << log_n) == ocoef[i]).all(), c
        assert (_part(dst, c << log_m, 1 << log_m) == olde[i]).all(), c


def _quotients(log_n, n_cols, n_points, dense):
    """Quotients of n_cols columns sampled at every point or at one point each: launches that expand
    weights, and whether the result is the oracle's."""
    rng = np.random.default_rng(100 * log_n + n_cols)
    host = [rng.integers(0, S.P, 1 << log_n, dtype=np.uint32) for _ in range(n_cols)]
    host[0][:] = S.P - 1
    cols = [S.BaseFieldVec.from_numpy(h) for h in host]
    batches = [(S.random_circle_point_qm31(rng), [(c, S.random_qm31(rng)) for c in range(n_cols) if dense or c % n_points == k])
               for k in range(n_points)]
    rc, dom = S.random_qm31(rng), S.canonic_half_coset(log_n)
    out = S.SecureColumn.uninitialized(1 << log_n)
    with launches("quotient_constants") as got:
        S.accumulate_quotients_async(dom, cols, rc, S.QuotientSamples(batches), out)
    want = O.accumulate_quotients(dom.initial_index, dom.step_size, log_n, host, rc, batches)
    assert (out.to_numpy() == want).all()
    return got["quotient_constants"]


# columns sampled at every point (or at one each): whether the matrix form is the faster one, as timed
@pytest.mark.parametrize("log_n,n_cols,n_points,dense,matrix", [
    (11, 112, 1, True, 0), (11, 128, 1, True, 1), (11, 16, 2, True, 0), (11, 17, 2, True, 1), (11, 16, 3, True, 0),
    (11, 22, 3, True, 1), (11, 32, 3, False, 0), (11, 40, 3, False, 1), (11, 11, 4, True, 0), (11, 12, 4, True, 1),
    (11, 32, 4, False, 1), (17, 16, 2, True, 1), (17, 8, 4, True, 1), (17, 16, 3, True, 0)])
def test_quotients_take_the_faster_form(log_n, n_cols, n_points, dense, matrix):
    assert _quotients(log_n, n_cols, n_points, dense) == matrix


@pytest.mark.parametrize("log_n", [14, 15, 16, 21, 22])
@pytest.mark.parametrize("offset", [0, 1, 2, 3])
def test_bit_reverse_at_the_tile_sizes(log_n, offset):
    """Columns at any word either side of the sizes at which the tile changes, nothing beyond their ends
    touched."""
    data = np.random.default_rng(log_n).integers(0, S.P, (1 << log_n) + 8, dtype=np.uint32)
    col = S.BaseFieldVec.from_numpy(data)
    S.lib().bit_reverse_base_field(col.ptr + 4 * offset, 1 << log_n)
    S.check()
    want = data.copy()
    want[offset:offset + (1 << log_n)] = O.bit_reverse(data[offset:offset + (1 << log_n)].copy())
    assert (col.to_numpy() == want).all()


@pytest.mark.parametrize("log_n,n_cols,blowup", [
    (17, 385, 1), (17, 1024, 1), (17, 1024, 2), (17, 390, 4), (18, 200, 1), (18, 513, 2), (19, 101, 1), (19, 256, 2), (19, 97, 3),
    (20, 67, 1), (20, 128, 1), (20, 128, 2), (20, 72, 3)])
def test_extension_passes(log_n, n_cols, blowup):
    """Every number of strided layers on the matrix cores, two and more blocks of the evaluation domain,
    below and above the size from which accesses stream (2^27 values), uneven groups of columns."""
    log_m = log_n + blowup
    src, dst = _filled(n_cols << log_n, log_n + n_cols, 1 << log_n), S.BaseFieldVec.uninitialized(n_cols << log_m)
    picks = (0, 1, n_cols // 2, n_cols - 1)
    before = [_part(src, c << log_n, 1 << log_n) for c in picks]
    coset = S.canonic_half_coset(log_m)
    tw, itw = S.cached_twiddles(coset)
    sp, dp = _pointers(src, n_cols, 1 << log_n), _pointers(dst, n_cols, 1 << log_m)
    logs = np.full(n_cols, log_n, np.uint32).ctypes.data_as(S.u32p)
    with launches("fft_matrices", "fft_lde_strided") as got:
        S.check(S.lib().stwo_hip_lde_columns_async(sp, sp, dp, logs, n_cols, blowup, tw, itw, 1 << coset.log_size))
    assert got == {"fft_matrices": 1, "fft_lde_strided": 1}
    otw, oitw = O.precompute_twiddles(coset.initial_index, coset.step_size, coset.log_size)
    ocoef, olde = O.lde_columns(before, blowup, otw, oitw)
    for i, c in enumerate(picks):
        assert (_part(src, c << log_n, 1 << log_n) == ocoef[i]).all(), c
        assert (_part(dst, c << log_m, 1 << log_m) == olde[i]).all(), c


@pytest.mark.parametrize("log_n,n_cols,n_points", [(20, 128, 1), (20, 131, 2), (20, 129, 3), (21, 64, 4), (21, 72, 2)])
def test_quotients_of_streamed_columns(log_n, n_cols, n_points):
    """The matrix form with one to four points where the columns are read past the caches; rows at the
    domain's ends and inside against the formula."""
    src = _filled(n_cols << log_n, n_cols, 1 << log_n)
    cols = [S.BaseFieldVec.view(src.ptr + (c << (log_n + 2)), 1 << log_n) for c in range(n_cols)]
    rng = np.random.default_rng(n_cols)
    batches = [(S.random_circle_point_qm31(rng), [(c, S.random_qm31(rng)) for c in range(n_cols) if n_points == 1 or (c + k) % 3])
               for k in range(n_points)]
    rc, dom = S.random_qm31(rng), S.canonic_half_coset(log_n)
    out = S.SecureColumn.uninitialized(1 << log_n)
    with launches("quotient_constants") as got:
        S.accumulate_quotients_async(dom, cols, rc, S.QuotientSamples(batches), out)
    assert got["quotient_constants"] == 1
    result = out.to_numpy()
    rows = [0, 1, 63, 64, 511, 512, (1 << log_n) // 3, (1 << log_n) - 2, (1 << log_n) - 1]
    values = {c: [int(_part(col, r, 1)[0]) for r in rows] for c, col in enumerate(cols)}
    for i, r in enumerate(rows):
        want = R.quotient_at_row(dom, log_n, r, {c: v[i] for c, v in values.items()}, rc, batches)
        assert tuple(int(result[k][r]) for k in range(4)) == want, r


@pytest.mark.parametrize("n_cols,matrix", [(8192, 1), (8193, 0)])
def test_quotients_at_the_most_columns(n_cols, matrix):
    """The matrix form's sums are bounded for 8192 columns; one more takes the other form."""
    assert _quotients(4, n_cols, 1, True) == matrix


@pytest.mark.parametrize("log_n", [10, 12])
def test_evaluation_in_place_either_side_of_the_line(log_n):
    line = (24 << 20) >> log_n
    coset = S.canonic_half_coset(log_n)
    tw, _ = S.cached_twiddles(coset)
    otw, _ = O.precompute_twiddles(coset.initial_index, coset.step_size, coset.log_size)
    for n_cols, on_matrices in ((line + 1, 1), (line - 1, 0)):
        cols = _filled(n_cols << log_n, log_n, 1 << log_n)
        picks = (0, 1, n_cols // 2, n_cols - 2, n_cols - 1)
        before = [_part(cols, c << log_n, 1 << log_n) for c in picks]
        logs = np.full(n_cols, log_n, np.uint32).ctypes.data_as(S.u32p)
        p = _pointers(cols, n_cols, 1 << log_n)
        with launches("fft_matrices") as got:
            S.check(S.lib().stwo_hip_evaluate_columns_async(p, logs, p, logs, n_cols, tw, 1 << coset.log_size))
        assert got["fft_matrices"] == on_matrices
        for c, v in zip(picks, before):
            assert (_part(cols, c << log_n, 1 << log_n) == O.evaluate(v, coset.initial_index, otw)).all(), c
