"""GPU parity of the fit kernels (through the C ABI) against the FP64 oracle.

* absmax: exact; non-finite sources flagged.
* Gram: exactly symmetric; within the fp32 summation bound of the FP64 Gram of the exact values.
* projection: the fp32 rounding of the FP64 dot product -- equal to the oracle except for
  elements within ~1e-13 relative of an fp32 rounding boundary (at most one ulp); the fused
  per-column extrema are exactly the min / max of the returned coefficients.
* energies: FP64, relative 1e-12 of the oracle.
* quantizer: codes bit-exact with the oracle on the same coefficients and affine.
* Cholesky factor and inverse (CholeskyQR): relative 1e-12 of numpy's FP64 factorization;
  LAPACK's info convention for indefinite members.
"""

import functools

import numpy as np
import pytest
import torch

from oracle import fit as of
from oracle import quantize as oq
from reelcache_amd import fit_kernels as fk
from reelcache_amd import quantize as pq

pytestmark = pytest.mark.gpu

DTYPES = {"bfloat16": torch.bfloat16, "float16": torch.float16, "float32": torch.float32}


def _source(rng, rows, channels, dtype, device, spectrum=False):
    if spectrum:
        x = of.decaying_spectrum(rng, rows, channels)
    else:
        x = (rng.standard_normal((rows, channels)) * rng.lognormal(0, 1, channels)).astype(np.float32)
    tensor = torch.from_numpy(x).to(DTYPES[dtype]).to(device)
    return tensor, tensor.float().cpu().numpy()


def _basis(rng, rank, channels, device):
    q, _ = np.linalg.qr(rng.standard_normal((channels, rank)))
    basis = of.stored_basis(q.T)
    return torch.from_numpy(basis).to(device), basis


@pytest.mark.parametrize("dtype", ["bfloat16", "float16", "float32"])
def test_absmax_exact_and_nonfinite(device, dtype):
    rng = np.random.default_rng(10)
    a, a_host = _source(rng, 300, 136, dtype, device)
    b, b_host = _source(rng, 65, 136, dtype, device)
    c, _ = _source(rng, 64, 136, dtype, device)
    c[17, 99] = float("inf")
    keys = fk.absmax([a, b, c]).cpu().numpy().astype(np.uint32)
    assert keys[0].view(np.float32) == np.abs(a_host).max()
    assert keys[1].view(np.float32) == np.abs(b_host).max()
    assert keys[2] >= fk.NONFINITE_BITS


@pytest.mark.parametrize("dtype,rows,channels", [("bfloat16", 300, 136), ("float16", 257, 256),
                                                 ("float32", 129, 200), ("bfloat16", 4680, 1536),
                                                 ("float16", 97, 520), ("float32", 70, 392), ("bfloat16", 33, 768)])
def test_gram_symmetric_and_within_fp32_bound(device, dtype, rows, channels):
    rng = np.random.default_rng(11)
    sources, hosts = zip(*[_source(rng, rows - 7 * i, channels, dtype, device) for i in range(2)])
    grams = fk.gram(list(sources)).cpu().numpy()
    for gram, host in zip(grams, hosts):
        np.testing.assert_array_equal(gram, gram.T)  # exactly symmetric
        expected = of.gram(host)
        bound = (host.shape[0] + 2) * 2.0 ** -24 * (np.abs(host).T.astype(np.float64) @ np.abs(host))
        assert np.all(np.abs(gram - expected) <= bound + 1e-30)


def test_gram_pads_unaligned_channels(device):
    rng = np.random.default_rng(12)
    x, host = _source(rng, 50, 13, "float32", device)
    gram = fk.gram([x]).cpu().numpy()
    assert gram.shape == (1, 13, 13)
    np.testing.assert_allclose(gram[0], of.gram(host), rtol=1e-5, atol=1e-5)


@pytest.mark.parametrize("dtype,rows,channels,rank", [("bfloat16", 300, 136, 40), ("float16", 129, 256, 64),
                                                      ("float32", 100, 64, 7), ("bfloat16", 4680, 1536, 128)])
def test_projection_rounds_the_fp64_product(device, dtype, rows, channels, rank):
    rng = np.random.default_rng(13)
    x, host = _source(rng, rows, channels, dtype, device)
    q, q_host = _basis(rng, rank + 3, channels, device)
    (p,), keys = fk.project([x], [q], [rank], extrema=True)
    p = p.cpu().numpy()
    expected = of.project(host, q_host, rank)
    differ = p != expected
    assert differ.mean() <= 1e-4
    if differ.any():
        ulp = np.abs(p[differ].view(np.int32).astype(np.int64) - expected[differ].view(np.int32).astype(np.int64))
        assert ulp.max() <= 1
    low, high = fk.split_keys(keys[0].cpu().numpy(), rank)
    np.testing.assert_array_equal(low, p.min(0))
    np.testing.assert_array_equal(high, p.max(0))


def test_projection_batch_of_ragged_ranks(device):
    rng = np.random.default_rng(14)
    xs, hosts, qs, q_hosts = [], [], [], []
    ranks = [5, 32, 61]
    for i, rank in enumerate(ranks):
        x, host = _source(rng, 90 + 31 * i, 64, "bfloat16", device)
        q, q_host = _basis(rng, rank, 64, device)
        xs.append(x), hosts.append(host), qs.append(q), q_hosts.append(q_host)
    coefficients, _ = fk.project(xs, qs, ranks)
    for p, host, q_host, rank in zip(coefficients, hosts, q_hosts, ranks):
        expected = of.project(host, q_host, rank)
        assert p.shape == expected.shape
        assert (p.cpu().numpy() == expected).mean() >= 0.999


def test_basis_layouts_read_in_place_or_repadded_give_the_same_values(device):
    """A stored basis is read in place when its rows are unit-stride, 16-byte aligned and 16-byte
    pitched, else through a zero-padded copy.  Row-major, column-major (a transposed view), a row
    block at an odd element offset and a wider pitch must all give the same coefficients and
    energies, bit for bit."""
    rng = np.random.default_rng(41)
    channels, rank = 128, 24
    x, _ = _source(rng, 300, channels, "bfloat16", device, spectrum=True)
    q, _ = _basis(rng, rank, channels, device)
    column_major = q.T.contiguous().T                      # strides (1, rank)
    wide = torch.zeros((rank, channels + 8), dtype=q.dtype, device=device)
    wide[:, :channels] = q
    pitched = wide[:, :channels]                            # row pitch 136 elements (272 bytes)
    shifted_storage = torch.zeros(rank * channels + 1, dtype=q.dtype, device=device)
    shifted = shifted_storage[1:].view(rank, channels)      # address 2 bytes past a 16-byte boundary
    shifted.copy_(q)
    layouts = [q, column_major, pitched, shifted]
    assert column_major.stride() == (1, rank) and shifted.data_ptr() % 16 == 2
    keys = fk.absmax([x] * len(layouts))
    coefficients, extrema = fk.project([x] * len(layouts), layouts, [rank] * len(layouts), extrema=True)
    totals = fk.energies([x] * len(layouts), keys, bases=layouts, ranks=[rank] * len(layouts),
                         coefficients=coefficients).cpu().numpy()
    for p, total, row in zip(coefficients[1:], totals[1:], extrema[1:]):
        assert torch.equal(p, coefficients[0])
        assert np.array_equal(total, totals[0])
        assert torch.equal(row, extrema[0])


@pytest.mark.parametrize("dtype", ["bfloat16", "float32"])
def test_energies_match_fp64(device, dtype):
    rng = np.random.default_rng(15)
    x, host = _source(rng, 1000, 256, dtype, device, spectrum=True)
    y, y_host = _source(rng, 77, 256, dtype, device)
    q, q_host = _basis(rng, 24, 256, device)
    r, r_host = _basis(rng, 3, 256, device)
    keys = fk.absmax([x, y])
    coefficients, _ = fk.project([x, y], [q, r], [24, 3])
    totals = fk.energies([x, y], keys, bases=[q, r], ranks=[24, 3], coefficients=coefficients).cpu().numpy()
    for total, host_x, basis, p, rank in zip(totals, (host, y_host), (q_host, r_host), coefficients, (24, 3)):
        _, source, error = of.energies(host_x, basis, p.cpu().numpy(), rank)
        assert total[0] == pytest.approx(source, rel=1e-12)
        assert total[1] == pytest.approx(error, rel=1e-12)
    source_only = fk.energies([x], fk.absmax([x])).cpu().numpy()
    assert source_only[0, 0] == pytest.approx(of.energies(host)[1], rel=1e-12)


@pytest.mark.parametrize("copies", [1, 12])
def test_energies_and_residual_matrices_of_ragged_ranks(device, copies):
    """Ranks beside the 16-rank steps (and one that is not a multiple of 4) in one batch, in 16-token
    workgroups and, with the batch repeated, in the 128-token ones that share their basis operands: the
    energies match the FP64 oracle, and so does the fp32 residual matrix X - P Q (rounded once from its
    FP64 value)."""
    rng = np.random.default_rng(21)
    ranks = [13, 48, 64, 65, 130]
    sources, hosts, bases, host_bases = [], [], [], []
    for index, rank in enumerate(ranks):
        x, host = _source(rng, 200 + 37 * index, 192, "bfloat16", device, spectrum=True)
        q, q_host = _basis(rng, rank, 192, device)
        sources.append(x)
        hosts.append(host)
        bases.append(q)
        host_bases.append(q_host)
    sources, hosts, bases, host_bases, ranks = (copies * values for values in (sources, hosts, bases, host_bases, ranks))
    keys = fk.absmax(sources)
    coefficients, _ = fk.project(sources, bases, ranks)
    totals, residuals = fk.energies(sources, keys, bases=bases, ranks=ranks, coefficients=coefficients,
                                    residuals=True)
    totals = totals.cpu().numpy()
    for total, residual, host, basis, p, rank in zip(totals, residuals, hosts, host_bases, coefficients, ranks):
        p_host = p.cpu().numpy()
        _, source, error = of.energies(host, basis, p_host, rank)
        assert total[0] == pytest.approx(source, rel=1e-12), rank
        assert total[1] == pytest.approx(error, rel=1e-12), rank
        exact = of.as_float(host) - p_host.astype(np.float64) @ np.asarray(basis, np.float16).astype(np.float64)[:rank]
        got = residual.cpu().numpy()
        # FP64 sums in another order: the fp32 rounding agrees except next to a rounding boundary.
        assert (got == exact.astype(np.float32)).mean() >= 0.999, rank
        assert np.abs(got - exact).max() <= 2 ** -23 * np.abs(exact).max(), rank


def test_zero_matrix_energies(device):
    x = torch.zeros((70, 64), dtype=torch.bfloat16, device=device)
    keys = fk.absmax([x])
    assert int(keys.cpu()[0]) == 0
    assert fk.energies([x], keys).cpu().numpy().tolist() == [[0.0, 0.0]]


@functools.lru_cache(maxsize=1)
def _causvid_spectrum():
    rng = np.random.default_rng(16)
    return of.decaying_spectrum(rng, 4680, 1536), np.linalg.qr(rng.standard_normal((1536, 32)))[0].T


@pytest.mark.parametrize("normalization,fraction", [("per_channel", 1.0), ("global", 0.0), ("leading_columns", 0.25)])
def test_quantizer_bit_exact(device, normalization, fraction):
    x_host, rows = _causvid_spectrum()
    x = torch.from_numpy(x_host).to(torch.bfloat16).to(device)
    q = torch.from_numpy(of.stored_basis(rows)).to(device)
    (p,), keys = fk.project([x], [q], [32], extrema=True)
    values = p.contiguous()
    layout = pq.normalization_layout(32, normalization, fraction)
    low, high = fk.split_keys(keys[0].cpu().numpy(), 32)
    affine = pq.affine_from_extrema(low, high, layout)
    scale, offset = pq.expanded_affine(affine, layout, 32)
    codes = fk.quantize(values, torch.from_numpy(np.asarray(scale, np.float64)).to(device),
                        torch.from_numpy(np.asarray(offset, np.float64)).to(device)).cpu().numpy()
    host_p = values.cpu().numpy()
    o_codes, o_affine, _ = oq.quantize(host_p, normalization, fraction)
    np.testing.assert_array_equal(affine, o_affine)
    np.testing.assert_array_equal(codes, o_codes)
    # The standalone extrema kernel agrees with the fused ones.
    low2, high2 = fk.split_keys(fk.column_extrema(values).cpu().numpy(), 32)
    np.testing.assert_array_equal(low2, low)
    np.testing.assert_array_equal(high2, high)


def test_batched_quantizer_matches_single_launches(device):
    rng = np.random.default_rng(17)
    values, affines = [], []
    for rows, cols in ((4680, 32), (700, 64), (1, 5), (129, 96)):
        v = torch.from_numpy((rng.standard_normal((rows, cols)) * 3).astype(np.float32)).to(device)
        lo, hi = v.amin(0).cpu().numpy(), v.amax(0).cpu().numpy()
        affine = pq.covering_affine(lo, hi).astype(np.float64)
        affine[0, 1] = 0.0  # a zero scale maps the column to code 0
        values.append(v)
        affines.append(affine)
    batched = fk.quantize_batched(values, affines)
    for v, affine, codes in zip(values, affines, batched):
        single = fk.quantize(v, torch.from_numpy(affine[0].copy()).to(device), torch.from_numpy(affine[1].copy()).to(device))
        np.testing.assert_array_equal(codes.cpu().numpy(), single.cpu().numpy())
        np.testing.assert_array_equal(codes.cpu().numpy(), oq.quantize_with_affine(v.cpu().numpy(), affine[0], affine[1]))


@pytest.mark.parametrize("k", [2, 15, 16, 17, 31, 33, 64, 65, 80, 81, 112, 127])
def test_cholesky_inverse_block_edges(device, k):
    """Orders around the kernel's 16-row blocks and 48-column panel waves: A = R^T R and X = R^-1 as
    numpy computes them (relative 1e-12, condition <= 900), zeros below the diagonal; a member whose
    leading minor of order k, or just past the first block, is negative is flagged there."""
    from scipy.linalg import solve_triangular

    rng = np.random.default_rng(57 + k)
    q, _ = np.linalg.qr(rng.standard_normal((k, k)))
    good = (q * rng.uniform(1.0, 30.0, k)) @ q.T
    last = good.copy()
    last[k - 1, k - 1] = -1.0
    early = np.diag(np.arange(1.0, k + 1.0))
    at = min(k, 17)
    early[at - 1, at - 1] = -2.0
    # The matrix's lower triangle is never read.
    stored = np.stack([np.triu(member) + np.tril(np.full((k, k), np.nan), -1) for member in (good, last, early)])
    inverse, info = fk.cholesky_inverse(torch.from_numpy(stored).to(device))
    inverse = inverse.cpu().numpy()
    assert info.cpu().tolist() == [0, k, at]
    r = np.linalg.cholesky(good).T
    want = solve_triangular(r, np.eye(k), lower=False)
    assert np.abs(inverse[0] - want).max() <= 1e-12 * np.abs(want).max()
    assert (np.tril(inverse[0], -1) == 0).all()
    assert (inverse[1] == np.eye(k)).all() and (inverse[2] == np.eye(k)).all()


@pytest.mark.parametrize("k", [1, 7, 96, 128])
def test_cholesky_inverse_matches_fp64_factorization(device, k):
    """The batched factor-and-inverse launch of the planner's CholeskyQR steps against numpy's
    FP64 Cholesky (A = R^T R, R = L^T) and the exact triangular inverse: relative 1e-12 on
    well-conditioned matrices; R^-1 R = I; the lower triangle is zero."""
    from scipy.linalg import solve_triangular

    rng = np.random.default_rng(31 + k)
    batch = []
    for _ in range(5):
        q, _ = np.linalg.qr(rng.standard_normal((k, k)))
        batch.append((q * rng.uniform(1.0, 30.0, k)) @ q.T)  # condition <= 900
    a = np.stack(batch)
    inverse, info = fk.cholesky_inverse(torch.from_numpy(a).to(device))
    inverse, info = inverse.cpu().numpy(), info.cpu().numpy()
    assert (info == 0).all()
    for member, got in zip(a, inverse):
        r = np.linalg.cholesky(member).T
        want = solve_triangular(r, np.eye(k), lower=False)
        assert np.abs(got - want).max() <= 1e-12 * np.abs(want).max()
        assert np.abs(got @ r - np.eye(k)).max() <= 1e-12
        assert (np.tril(got, -1) == 0).all()


@pytest.mark.parametrize("k", [100, 129, 144, 192, 256, 257, 300, 512])
def test_factor_inverse_of_any_order(device, k):
    """Orders beyond one launch go in block rows: the triangular inverse against numpy's FP64 factorization
    (relative 1e-11: condition 900, up to four blocks), zeros below the diagonal, LAPACK's info in the first,
    a later and the last block, NaN at order 1; the same bits again with other work queued behind it."""
    from scipy.linalg import solve_triangular

    rng = np.random.default_rng(61 + k)
    batch = []
    for _ in range(3):
        q, _ = np.linalg.qr(rng.standard_normal((k, k)))
        batch.append((q * rng.uniform(1.0, 30.0, k)) @ q.T)
    early, late, nan = batch[0].copy(), batch[1].copy(), batch[2].copy()
    early[4, 4], late[k - 1, k - 1], nan[0, 0] = -1.0, -1.0, np.nan
    a = torch.from_numpy(np.stack(batch + [early, late, nan])).to(device)
    inverse, info = fk.factor_inverse(a)
    behind = [torch.full((1 << 20,), 1.0, dtype=torch.float64, device=device) * 2 for _ in range(4)]
    again, _ = fk.factor_inverse(a)
    assert info.cpu().tolist() == [0, 0, 0, 5, k, 1] and torch.equal(inverse, again) and len(behind) == 4
    inverse = inverse.cpu().numpy()
    for member, got in zip(batch, inverse):
        want = solve_triangular(np.linalg.cholesky(member).T, np.eye(k), lower=False)
        assert np.abs(got - want).max() <= 1e-11 * np.abs(want).max()
        assert (np.tril(got, -1) == 0).all()
    assert (inverse[3:] == np.eye(k)).all()


def test_cholesky_inverse_flags_indefinite_members(device):
    """LAPACK's info convention: j + 1 for the first leading minor that is not positive definite
    (a negative pivot at order 4, a NaN at order 1); such members come back as the identity and
    do not disturb the others."""
    k = 6
    good = np.diag(np.arange(1.0, k + 1.0))
    indefinite = np.diag([1.0, 2.0, 3.0, -1.0, 5.0, 6.0])
    nan = good.copy()
    nan[0, 0] = np.nan
    inverse, info = fk.cholesky_inverse(torch.from_numpy(np.stack([good, indefinite, nan])).to(device))
    assert info.cpu().tolist() == [0, 4, 1]
    inverse = inverse.cpu().numpy()
    np.testing.assert_allclose(inverse[0], np.diag(1.0 / np.sqrt(np.arange(1.0, k + 1.0))), rtol=1e-15)
    assert (inverse[1] == np.eye(k)).all() and (inverse[2] == np.eye(k)).all()
    with pytest.raises(Exception):
        fk.cholesky_inverse(torch.zeros((1, 129, 129), dtype=torch.float64, device=device))


@pytest.mark.parametrize("dtype", ["bfloat16", "float16", "float32"])
@pytest.mark.parametrize("count,rows,channels,ranks", [
    (1, 17, 72, [1]),                   # one 16-token tile and a row of the next; channels below one step of each wave
    (1, 4680, 264, [96]),               # 32-token projection, 16-token residual; several channel parts
    (3, 31, 136, [16, 33, 130]),        # ragged ranks over several 16-rank chunks
    (70, 2000, 64, [49]),               # 128-token workgroups of both; one residual part, one step a half
    (160, 1664, 40, [32]),              # 128-token workgroups; a second half of one 8-channel group
    (350, 700, 72, [1, 33, 64]),        # 128-token workgroups: a last wave of 28 rows, one to four rank blocks
    (18, 1000, 200, [16, 130, 75]),     # 32-rank chunks beside 128-token residual workgroups, ranks past a step
    (500, 33, 72, [20, 5, 48]),         # 128-token workgroups: waves of 32 rows, one row and none
])
def test_fit_launch_shapes_match_fp64(device, dtype, count, rows, channels, ranks):
    """absmax, projection and residual energies on both sides of their launch-shape rules: maxima
    exact, P within an ulp of the rounded FP64 product (equal on 99.99 %), energies within 1e-12, the
    first, last and middle matrices of a batch against numpy."""
    rng = np.random.default_rng(83)
    x, _ = _source(rng, rows, channels, dtype, device)
    sources = [x * (1 + i % 3) if i % 2 else -x for i in range(count)]
    ranks = [min(ranks[i % len(ranks)], rows, channels) for i in range(count)]
    bases = [_basis(rng, rank, channels, device) for rank in ranks[:3]]
    chosen = [bases[i % len(bases)] for i in range(count)]
    ranks = [int(q.shape[0]) for q, _ in chosen]
    keys = fk.absmax(sources)
    coefficients, extrema = fk.project(sources, [q for q, _ in chosen], ranks, extrema=True)
    totals = fk.energies(sources, keys, bases=[q for q, _ in chosen], ranks=ranks, coefficients=coefficients).cpu().numpy()
    alone = fk.energies(sources, keys).cpu().numpy()
    for i in sorted({0, count // 2, count - 1}):
        host = sources[i].double().cpu().numpy()
        q = np.asarray(chosen[i][1], dtype=np.float16).astype(np.float64)[:ranks[i]]
        bits = np.abs(host).max().astype(np.float32).view(np.int32)
        assert int(keys[i]) == int(bits)
        p, want = coefficients[i].cpu().numpy(), (host @ q.T).astype(np.float32)
        assert (p != want).mean() <= 1e-4
        assert np.abs(p.view(np.int32).astype(np.int64) - want.view(np.int32).astype(np.int64)).max() <= 1
        low, high = fk.split_keys(extrema[i].cpu().numpy(), ranks[i])
        np.testing.assert_array_equal(low, p.min(0))
        np.testing.assert_array_equal(high, p.max(0))
        scale = np.abs(host).max()
        source = np.square(host / scale).sum()
        error = np.square((host - p.astype(np.float64) @ q) / scale).sum()
        assert totals[i, 0] == pytest.approx(source, rel=1e-12) and alone[i, 0] == pytest.approx(source, rel=1e-12)
        assert totals[i, 1] == pytest.approx(error, rel=1e-12)


@pytest.mark.parametrize("dtype,count,rows,channels,rank", [
    ("bfloat16", 400, 700, 264, 49),    # 128-token projection workgroups, shared residual operands
    ("float16", 60, 4680, 136, 96),     # several channel parts, span ranges of more than one stage
    ("float32", 300, 129, 520, 128),    # a last tile of one row, channels beside four equal parts
    ("bfloat16", 24, 333, 1536, 17),    # channel-split projection, shared residual operands
    ("float32", 600, 33, 8, 5),         # one 64-channel group, most waves without rows
])
def test_measurements_do_not_depend_on_the_batch(device, dtype, count, rows, channels, rank):
    """P, its extrema, both energies, the residual matrix and the span terms of a matrix are the same
    bits alone and in a batch, whatever shapes the batch's launches take and whatever rows and ranks
    its other members have: a planned rank is verified in small rounds and finalized in the chunk."""
    rng = np.random.default_rng(131)
    x, _ = _source(rng, rows, channels, dtype, device)
    basis, _ = _basis(rng, rank, channels, device)
    low, _ = _basis(rng, max(1, rank // 2), channels, device)
    # Members of other row counts and ranks between copies of one scaled matrix.
    sources = [x * (1 + i % 3) if i % 4 else x[: 1 + (7 * i) % rows] for i in range(count)]
    bases = [basis if i % 3 else low for i in range(count)]
    ranks = [int(q.shape[0]) for q in bases]

    def measure(members):
        xs, qs, rs = ([values[i] for i in members] for values in (sources, bases, ranks))
        keys = fk.absmax(xs)
        coefficients, extrema = fk.project(xs, qs, rs, extrema=True)
        totals, residuals = fk.energies(xs, keys, bases=qs, ranks=rs, coefficients=coefficients, residuals=True)
        return coefficients, extrema, totals, residuals, fk.energies(xs, keys), fk.span_terms(qs, rs, coefficients)

    together = measure(range(count))
    for i in sorted({0, 1, 4, count // 2, count - 2, count - 1}):
        for members in ([i], [i, (i + 1) % count, (i + 5) % count]):
            part = measure(members)
            assert torch.equal(part[0][0], together[0][i])
            assert torch.equal(part[1][0, :2 * ranks[i]], together[1][i, :2 * ranks[i]])
            assert torch.equal(part[2][0], together[2][i]) and torch.equal(part[3][0], together[3][i])
            assert torch.equal(part[4][0], together[4][i]) and torch.equal(part[5][0], together[5][i])


@pytest.mark.parametrize("dtype", ["bfloat16", "float16", "float32"])
def test_absmax_flags_nonfinite_values(device, dtype):
    """An infinity or a NaN anywhere (first and last element, either sign) puts the key at or above
    the infinity's bits; the other matrices of the batch keep their exact maxima."""
    values = torch.zeros((37, 48), dtype=DTYPES[dtype], device=device)
    values[5, 7] = -3.5
    bad = []
    for value, at in ((float("inf"), (0, 0)), (float("-inf"), (36, 47)), (float("nan"), (36, 40)), (-float("nan"), (0, 7))):
        member = values.clone()
        member[at] = value
        bad.append(member)
    keys = fk.absmax([values] + bad + [torch.zeros_like(values)]).cpu().numpy()
    assert keys[0] == np.float32(3.5).view(np.int32) and keys[-1] == 0
    assert (keys[1:-1] >= fk.NONFINITE_BITS).all()


@pytest.mark.parametrize("channels,rows,ranks", [(136, 500, [1, 15, 16, 17, 33, 64, 65, 127, 128]), (40, 1, [3]),
                                                 (1536, 33, [32, 96]), (264, 4680, [128])])
def test_span_terms_match_fp64(device, channels, rows, ranks):
    """Span trace, Cholesky status and norms of a ragged batch of basis views against numpy in FP64
    (relative 1e-11: the condition of these rows is below 4), and without coefficients."""
    rng = np.random.default_rng(97)
    bases, coefficients = [], []
    for rank in ranks:
        q, _ = np.linalg.qr(rng.standard_normal((channels, rank)))
        bases.append(torch.from_numpy((q * rng.uniform(0.7, 1.3, rank)).T.copy()).to(torch.float16).to(device))
        padded = torch.zeros((rows, -(-rank // 4) * 4), device=device)
        padded[:, :rank] = torch.from_numpy(rng.standard_normal((rows, rank)).astype(np.float32)).to(device)
        coefficients.append(padded[:, :rank])
    terms = fk.span_terms(bases, ranks, coefficients).cpu().numpy()
    plain = fk.span_terms(bases, ranks).cpu().numpy()
    assert (plain[:, 0] == 0).all() and np.array_equal(plain[:, 1:], terms[:, 1:])
    for basis, p, row in zip(bases, coefficients, terms):
        q, c = basis.double().cpu().numpy(), p.double().cpu().numpy()
        gram = q @ q.T
        inverse = np.linalg.inv(gram)
        want = [np.trace(inverse @ (c.T @ c)), 0.0, np.abs(gram - np.eye(len(q))).sum(1).max(), np.abs(np.diag(gram)).max(),
                np.abs(gram).sum(1).max(), np.abs(inverse).sum(1).max()]
        np.testing.assert_allclose(row, want, rtol=1e-11)


def test_span_terms_flag_singular_views(device):
    """A repeated row is not positive definite at its order (the exact FP64 factor's pivot is zero or
    negative); a NaN at the first; the other views of the batch are unaffected."""
    rng = np.random.default_rng(98)
    q, _ = np.linalg.qr(rng.standard_normal((64, 20)))
    good = torch.from_numpy(q.T.copy()).to(torch.float16).to(device)
    zero = good.clone()
    zero[17] = 0.0
    nan = good.clone()
    nan[0, 5] = float("nan")
    terms = fk.span_terms([zero, good, nan], [20, 20, 20]).cpu().numpy()
    assert terms[:, 1].tolist() == [18.0, 0.0, 1.0]
    assert np.isinf(terms[0, 5]) and np.isinf(terms[2, 5]) and np.isfinite(terms[1]).all()


@pytest.mark.parametrize("rank", [12, 33, 128])
def test_span_terms_of_ill_conditioned_views(device, rank):
    """Rows near one direction (condition of G about 1e6): the trace and both norms against extended
    precision, within the forward error of a Cholesky solve, 8 k eps cond(G)."""
    rng = np.random.default_rng(103)
    channels, tokens = 512, 300
    common = rng.standard_normal(channels) / channels ** 0.5
    rows = (common + 0.02 * rng.standard_normal((rank, channels)) / channels ** 0.5).astype(np.float16)
    p = rng.standard_normal((tokens, rank)).astype(np.float32)
    got = fk.span_terms([torch.from_numpy(rows).to(device)], [rank], [torch.from_numpy(p).to(device)]).cpu().numpy()[0]
    q = rows.astype(np.longdouble)
    gram, c = q @ q.T, p.astype(np.longdouble).T @ p.astype(np.longdouble)
    work = np.concatenate([gram, c, np.eye(rank, dtype=np.longdouble)], axis=1)
    for j in range(rank):  # Gauss-Jordan without pivoting (G is positive definite)
        work[j] /= work[j, j]
        others = np.arange(rank) != j
        work[others] -= work[others, j][:, None] * work[j]
    solved, inverse = work[:, rank:2 * rank], work[:, 2 * rank:]
    condition = float(np.linalg.cond(gram.astype(np.float64)))
    assert 1e4 < condition < 1e8 and got[1] == 0
    bound = 8 * rank * 2.0 ** -52 * condition
    assert got[0] == pytest.approx(float(np.trace(solved)), rel=bound)
    assert got[4] == pytest.approx(float(np.abs(gram).sum(1).max()), rel=1e-12)
    assert got[5] == pytest.approx(float(np.abs(inverse).sum(1).max()), rel=bound)


@pytest.mark.parametrize("rank", [129, 192])
def test_projection_above_the_native_order(device, rank):
    """Ranks above the span kernels' order read and check the basis and its condition first, then project:
    coefficients, residual and condition against FP64, and the faults in their order."""
    from reelcache_amd import factorization as fa
    from reelcache_amd.errors import ConfigurationError

    rng = np.random.default_rng(107)
    x, host = _source(rng, 300, 256, "bfloat16", device)
    q, q_host = _basis(rng, rank + 3, 256, device)
    projection = fa.project_onto_basis(x, q, rank=rank)
    p = projection.coefficients.cpu().numpy()
    assert p.shape == (300, rank) and (p == of.project(host, q_host, rank)).mean() >= 0.999
    _, source, error = of.energies(host, q_host, p, rank)
    assert projection.relative_residual == pytest.approx((error / source) ** 0.5, rel=1e-12)
    wide = np.asarray(q_host, dtype=np.float16).astype(np.float64)[:rank]
    gram = wide @ wide.T
    want = np.abs(gram).sum(1).max() * np.abs(np.linalg.inv(gram)).sum(1).max()
    assert projection.condition_bound == pytest.approx(want, rel=1e-9)
    given = fa.project_onto_basis(x, q, rank=rank, _condition_bound=1.25)
    assert given.condition_bound == 1.25 and torch.equal(given.coefficients, projection.coefficients)
    assert projection.condition_seconds > 0 and projection.coefficient_seconds > 0
    bad = q.clone()
    bad[rank + 2, 3] = float("nan")
    infinite = x.clone()
    infinite[0, 0] = float("inf")
    with pytest.raises(ConfigurationError, match="stored basis must be finite"):
        fa.project_onto_basis(infinite, bad, rank=rank)
    singular = q.clone()
    singular[4] = 0.0
    with pytest.raises(ConfigurationError, match="singular or ill-conditioned"):
        fa.project_onto_basis(infinite, singular, rank=rank)
    with pytest.raises(ConfigurationError, match="nonempty finite"):
        fa.project_onto_basis(infinite, q, rank=rank)


def test_projection_reports_its_first_fault(device):
    """project_onto_basis checks the basis before the matrix: a basis that is not finite (also past
    the rank, also with a bad argument), a singular one, an ill-conditioned one, then the matrix."""
    from reelcache_amd import factorization as fa
    from reelcache_amd.errors import ConfigurationError

    rng = np.random.default_rng(99)
    x, _ = _source(rng, 100, 64, "bfloat16", device)
    q, _ = np.linalg.qr(rng.standard_normal((64, 12)))
    basis = torch.from_numpy(q.T.copy()).to(torch.float16).to(device)
    projection = fa.project_onto_basis(x, basis, rank=10)
    gram = basis[:10].double().cpu().numpy() @ basis[:10].double().cpu().numpy().T
    want = np.abs(gram).sum(1).max() * np.abs(np.linalg.inv(gram)).sum(1).max()
    assert projection.condition_bound == pytest.approx(want, rel=1e-12)
    assert fa.basis_condition_bound(basis[:10]) == projection.condition_bound
    bad = basis.clone()
    bad[11, 3] = float("inf")
    for arguments in ({"rank": 10}, {"rank": 99}):
        with pytest.raises(ConfigurationError, match="stored basis must be finite"):
            fa.project_onto_basis(x, bad, **arguments)
    with pytest.raises(ConfigurationError, match="rank"):
        fa.project_onto_basis(x, basis, rank=13)
    singular = basis.clone()
    singular[4] = 0.0
    with pytest.raises(ConfigurationError, match="singular or ill-conditioned"):
        fa.project_onto_basis(x, singular)
    with pytest.raises(ConfigurationError, match="singular or ill-conditioned"):
        fa.project_onto_basis(x, basis, max_condition=1.0)
    infinite = x.clone()
    infinite[99, 63] = float("inf")
    with pytest.raises(ConfigurationError, match="nonempty finite"):
        fa.project_onto_basis(infinite, basis)
    with pytest.raises(ConfigurationError, match="singular or ill-conditioned"):
        fa.project_onto_basis(infinite, singular)


def test_condition_bound_beyond_the_native_addressing(device):
    """basis_condition_bound takes what it took before it had a native path: rows 2 GiB apart in all (the
    kernels' 32-bit offsets end there, so they are read through a copy), also through the projection and
    as a source, and more channels than the fit kernels take."""
    from reelcache_amd import factorization as fa

    rank, channels, pitch = 128, 256, 9 << 20
    generator = torch.Generator(device=device).manual_seed(8)
    rows = torch.linalg.qr(torch.randn(channels, rank, device=device, generator=generator)).Q.T.contiguous().to(torch.float16)
    storage = torch.empty((rank - 1) * pitch + channels, dtype=torch.float16, device=device)
    apart = storage.as_strided((rank, channels), (pitch, 1))
    apart.copy_(rows)
    assert fa.basis_condition_bound(apart) == fa.basis_condition_bound(rows) < 1.5
    x, _ = _source(np.random.default_rng(3), rank, channels, "bfloat16", device)
    assert torch.equal(fk.project([x], [apart], [rank])[0][0], fk.project([x], [rows], [rank])[0][0])
    far = storage.as_strided((32, channels), (4 * pitch, 1))
    assert torch.equal(fk.project([far], [rows], [rank])[0][0], fk.project([far.contiguous()], [rows], [rank])[0][0])
    wide = torch.randn(2, (1 << 20) + 8, device=device, generator=generator).to(torch.float16)
    gram = wide.double() @ wide.double().T
    want = float(gram.abs().sum(1).max() * torch.linalg.inv(gram).abs().sum(1).max())
    assert fa.basis_condition_bound(wide) == pytest.approx(want, rel=1e-9)


def test_projection_times_its_condition(device):
    """condition_seconds covers the condition's device work, though the wait for it comes with the read
    that ends the coefficients; the parts of the time do not exceed the whole."""
    from reelcache_amd import factorization as fa

    channels, rank = 1 << 17, 128  # the basis Gram alone takes about a millisecond
    generator = torch.Generator(device=device).manual_seed(7)
    basis = (torch.randn(rank, channels, device=device, generator=generator) / channels ** 0.5).to(torch.float16)
    x = torch.randn(rank, channels, device=device, generator=generator).to(torch.bfloat16)
    fa.project_onto_basis(x, basis)
    marks = [torch.cuda.Event(enable_timing=True) for _ in range(2)]
    torch.cuda.synchronize(device)
    marks[0].record()
    for _ in range(4):
        fk.span_terms([basis], [rank])
    marks[1].record()
    marks[1].synchronize()
    terms = marks[0].elapsed_time(marks[1]) * 1e-3 / 4
    projection = fa.project_onto_basis(x, basis)
    assert terms > 5e-4 and projection.condition_seconds >= 0.5 * terms
    assert projection.coefficient_seconds > 0
    assert projection.condition_seconds + projection.coefficient_seconds + projection.guard_seconds <= projection.seconds


@pytest.mark.parametrize("rows,cols,stride", [(1, 1, 1), (17, 3, 5), (64, 96, 96), (65, 130, 132), (130, 63, 64)])
def test_extrema_and_codes_at_tile_edges(device, rows, cols, stride):
    """Column extrema and codes of strided matrices around the kernels' row tiles, column lanes and
    four-column groups: exact extrema, codes equal to the oracle's, also through the batched launch."""
    rng = np.random.default_rng(101)
    storage = torch.from_numpy(rng.standard_normal((rows, stride)).astype(np.float32)).to(device)
    values = storage[:, :cols]
    host = values.cpu().numpy()
    low, high = fk.split_keys(fk.column_extrema(values).cpu().numpy(), cols)
    np.testing.assert_array_equal(low, host.min(0))
    np.testing.assert_array_equal(high, host.max(0))
    affine = np.asarray(oq.covering_affine(low, high), dtype=np.float64)
    affine[0, 0] = 0.0  # a zero scale gives code 0
    want = oq.quantize_with_affine(host, affine[0], affine[1])
    scale, offset = (torch.from_numpy(v.copy()).to(device) for v in affine)
    np.testing.assert_array_equal(fk.quantize(values, scale, offset).cpu().numpy(), want)
    for codes in fk.quantize_batched([values, values], [affine, affine]):
        np.testing.assert_array_equal(codes.cpu().numpy(), want)
