"""GPU parity of the exact-SVD boundary initializer
(exact_svd_boundary_launch_v1; the reference runtime's exact_svd initializer,
src/gdn_state_codec/runtime.py:335-389, which calls torch.linalg.svd) through
the C-ABI, against the float64 LAPACK SVD of oracle/svd.py.

The reference's result is its library's fp32 SVD, so no bit pattern is fixed;
the tests hold the fp32 rank-4 product to 4e-7 of the largest singular value,
the singular values likewise, the fp16 compensators to their own rounding of
that product, and the codes bit-exact to the oracle's quant stage applied to
the residual the kernel wrote.  The kernel iterates in double, so what remains
is the fp32 rounding of its outputs: keys and values rounded to fp32 and a
four-term fp32 product, a few units of 2^-24 of the largest singular value
(the bench measures 7.3e-8 on C1 heads).  4e-7 leaves that a margin of about
five, so an accumulation that loses ten times the precision fails; torch's
fp32 SVD, the reference's own call, lands at 3e-7..3e-6 on Gaussian heads."""

import numpy as np
import pytest
import torch

import datagen
import oracle
from gdn_state_codec import codec
from oracle import svd as S

pytestmark = pytest.mark.gpu
FIT_TOLERANCE = 4e-7  # of the largest singular value


def host(t):
    torch.cuda.synchronize()
    return t.cpu().numpy()


def planted_head(seed, spectrum):
    g = np.random.default_rng(seed)
    q1, _ = np.linalg.qr(g.standard_normal((128, 128)))
    q2, _ = np.linalg.qr(g.standard_normal((128, 128)))
    return ((q1 * spectrum) @ q2.T).astype(np.float32)


def dense_heads():
    g = datagen.rng(71)
    spread = np.concatenate([[40.0, 20.0, 10.0, 5.0], np.linspace(1.0, 0.01, 124)])
    return {
        "c1": datagen.c1_heads(4, 72),
        "student_t": datagen.student_t_heads(4, 73),
        "planted": np.stack([planted_head(74, spread), planted_head(75, spread * 1e-3)]),
        "special": np.stack([
            datagen.wide_range_head(76),
            datagen.tiny_head(77),
            datagen.zero_rows_cols_head(78),
            np.outer(g.standard_normal(128), g.standard_normal(128)).astype(np.float32),
            datagen.constant_head(0.25),
            np.zeros((128, 128), np.float32),
        ]),
    }


def run(dense):
    provider = torch.from_numpy(np.ascontiguousarray(dense.transpose(0, 2, 1))).cuda()
    out = codec.exact_svd_boundary(provider)
    return provider, [host(t) for t in out]


def check_heads(dense, got, rank_deficient=()):
    codes, s, sc, keys16, values16, residual, status = got
    assert (status == 0).all()
    provider = dense.transpose(0, 2, 1)
    left, right, singular, product = S.svd_fit_heads(provider)
    keys = keys16.view(np.float16).astype(np.float64)
    values = values16.view(np.float16).astype(np.float64)
    for h in range(len(dense)):
        top = max(singular[h, 0], 1e-30)
        # The fp32 fit the residual was formed with, [key][value].
        fit = (provider[h].astype(np.float64) - residual[h].astype(np.float64)).T
        assert np.abs(fit - product[h]).max() <= FIT_TOLERANCE * top, h
        # fp16 compensators: their product is the fit, to fp16 rounding.
        pair = keys[h] @ values[h].T
        bound = 2.0 ** -10 * (np.abs(keys[h]) @ np.abs(values[h]).T) + 2.0 ** -23 * top
        assert (np.abs(pair - fit) <= bound + FIT_TOLERANCE * top).all(), h
        norms = np.linalg.norm(keys[h], axis=0)
        assert np.abs(norms - singular[h, :4]).max() <= 2.0 ** -10 * top + FIT_TOLERANCE * top, h
        if h not in rank_deficient:
            gram = values[h].T @ values[h]
            assert np.abs(gram - np.eye(4)).max() <= 4e-3, h
    # The quant stage: the oracle's encode of the residual the kernel wrote.
    e_codes, e_s, e_sc = oracle.encode_heads(residual, oracle.LAYOUT_VALUE_KEY, threads=8)
    assert codes.tobytes() == e_codes.tobytes()
    assert s.tobytes() == e_s.tobytes()
    assert sc.tobytes() == e_sc.tobytes()


@pytest.mark.parametrize("family", ["c1", "student_t", "planted"])
def test_exact_svd_matches_float64_svd(device, family):
    dense = dense_heads()[family]
    print(f"exact SVD initializer, {family}, heads={len(dense)}", flush=True)
    provider, got = run(dense)
    check_heads(dense, got)


def test_planted_vectors_are_recovered_up_to_sign(device):
    """Heads with well separated singular values: each compensator pair is the
    planted (sigma u, v) up to one sign per pair, to fp16 rounding."""
    dense = dense_heads()["planted"]
    print("exact SVD initializer, planted vectors", flush=True)
    _, got = run(dense)
    keys = got[3].view(np.float16).astype(np.float64)
    values = got[4].view(np.float16).astype(np.float64)
    left, right, singular, _ = S.svd_fit_heads(dense.transpose(0, 2, 1))
    for h in range(len(dense)):
        for r in range(4):
            sign = np.sign(values[h, :, r] @ right[h, :, r])
            assert np.abs(sign * values[h, :, r] - right[h, :, r]).max() <= 2e-3
            assert (np.abs(sign * keys[h, :, r] - left[h, :, r]).max()
                    <= 2e-3 * singular[h, r] + FIT_TOLERANCE * singular[h, 0])


def test_special_heads(device):
    """Wide exponent range, subnormals, zero rows and columns, rank 1, a
    constant head and an all-zero head (zero compensators, residual = input)."""
    dense = dense_heads()["special"]
    print(f"exact SVD initializer, special heads={len(dense)}", flush=True)
    provider, got = run(dense)
    check_heads(dense, got, rank_deficient=(3, 4, 5))
    keys16, values16, residual = got[3], got[4], got[5]
    assert not keys16[5].any() and not values16[5].any()
    assert residual[5].tobytes() == host(provider)[5].tobytes()


def test_non_finite_heads_are_rejected(device):
    dense = datagen.c1_heads(4, 79)
    dense[1, 5, 9] = np.nan
    dense[2, 0, 127] = -np.inf
    print("exact SVD initializer, rejections", flush=True)
    provider = torch.from_numpy(np.ascontiguousarray(dense.transpose(0, 2, 1))).cuda()
    got = codec.exact_svd_boundary(provider, check=False)
    assert host(got[6]).tolist() == [0, 1, 1, 0]
    with pytest.raises(ValueError, match="head 1 holds a non-finite value"):
        codec.exact_svd_boundary(provider)


def test_many_heads(device):
    """1,024 heads (four rounds of one workgroup per CU): every status 0, and
    every 61st head checked against the float64 SVD."""
    dense = np.concatenate([datagen.c1_heads(512, 81), datagen.student_t_heads(512, 82)])
    print(f"exact SVD initializer, heads={len(dense)}", flush=True)
    _, got = run(dense)
    sample = list(range(0, len(dense), 61))
    check_heads(dense[sample], [g[sample] for g in got])


def test_sweep_limit_flags_unconverged_heads(device):
    """exact_svd_boundary_sweeps_launch_v1: after one sweep no C1 head has
    converged (status 2, and exact_svd_boundary raises), while an all-zero
    head, which never rotates, has (status 0); at the full limit of 30 sweeps
    every output equals the default entry point's bit for bit."""
    print("exact SVD sweep limit", flush=True)
    dense = np.concatenate([datagen.c1_heads(3, 79), np.zeros((1, 128, 128), np.float32)])
    provider = torch.from_numpy(np.ascontiguousarray(dense.transpose(0, 2, 1))).cuda()
    *_, status = codec.exact_svd_boundary(provider, check=False, max_sweeps=1)
    assert host(status).tolist() == [2, 2, 2, 0]
    with pytest.raises(ValueError, match="did not converge"):
        codec.exact_svd_boundary(provider, max_sweeps=1)
    full = [host(t) for t in codec.exact_svd_boundary(provider, max_sweeps=30)]
    default = [host(t) for t in codec.exact_svd_boundary(provider)]
    for a, b in zip(full, default):
        assert a.tobytes() == b.tobytes()
    assert (full[-1] == 0).all()


def mixed_heads(count, seed):
    """Heads of one and of several passes in one batch: plain heads, a fourth
    singular value just above and just below 2^-10 of the first (a pass's
    limit), ranks 1 to 5, and four leading singular values equal but for the
    rounding to fp32."""
    g = np.random.default_rng(seed)
    rest = np.linspace(0.9, 0.01, 124)
    out = []
    for i in range(count):
        kind = i % 8
        if kind < 2:
            out.append(datagen.c1_heads(1, seed + i)[0])
        elif kind < 4:
            ratio = 2.0 ** -10 * (1.25 if kind == 2 else 0.8)
            out.append(planted_head(seed + i, np.concatenate(
                [[1.0, 0.5, 0.1, ratio], ratio * rest])))
        elif kind < 7:
            rank = 1 + (i // 8) % 5
            out.append((g.standard_normal((128, rank))
                        @ g.standard_normal((rank, 128))).astype(np.float32))
        else:
            out.append(planted_head(seed + i, np.concatenate([[3.0, 3.0, 3.0, 3.0], rest])))
    return np.stack(out).astype(np.float32)


@pytest.mark.parametrize("count", [1, 3, 40, 521])
def test_direct_and_jacobi_forms_share_a_batch(device, count):
    """Every head of a mixed batch, whatever passes it took, holds the rank-4
    product to the tolerance of the other tests, and agrees with the Jacobi
    form's."""
    dense = mixed_heads(count, 500)
    print(f"exact SVD initializer, mixed batch of {count}", flush=True)
    _, got = run(dense)
    assert (got[6] == 0).all()
    sample = sorted({*range(min(count, 40)), *range(0, count, 53), count - 1})
    check_heads(dense[sample], [g[sample] for g in got],
                rank_deficient=[n for n, h in enumerate(sample) if h % 8 in (4, 5, 6)])
    # The sweep-limited entry point is Jacobi throughout: same product.
    provider = torch.from_numpy(np.ascontiguousarray(dense.transpose(0, 2, 1))).cuda()
    jacobi = [host(t) for t in codec.exact_svd_boundary(provider, max_sweeps=29)]
    largest = np.abs(dense).max(axis=(1, 2)) * 128  # at least sigma_1
    apart = np.abs(got[5].astype(np.float64) - jacobi[5]).max(axis=(1, 2))
    assert (apart <= 2 * FIT_TOLERANCE * largest).all()


def test_a_later_pass_keeps_double(device):
    """A fourth singular value below 2^-10 of the first, so that a second pass
    finds it, and a fifth 1e-5 below the fourth: how much of the fifth triplet
    the fit holds shows what that pass worked with.  Weighted with the two
    singular vectors, the fp32 roundings of the outputs (about 3e-10 of sigma_1
    a cell in rms) come to about 3e-10; what is left of the head rounded to
    fp32 before the pass gives 5e-8 and more."""
    ratio = 2.0 ** -10.5
    spectrum = np.concatenate([[1.0, 0.5, 0.25, ratio, ratio * (1 - 1e-5)],
                               ratio * np.linspace(0.9, 0.01, 123)])
    dense = np.stack([planted_head(seed, spectrum) for seed in range(910, 914)])
    print("exact SVD initializer, close singular values behind the limit", flush=True)
    provider, got = run(dense)
    assert (got[6] == 0).all()
    for p, residual in zip(host(provider).astype(np.float64), got[5].astype(np.float64)):
        u, s, vt = np.linalg.svd(p)
        fit = p - residual
        assert abs(u[:, 4] @ fit @ vt[3]) <= 3e-9 * s[0]
        assert abs(u[:, 3] @ fit @ vt[4]) <= 3e-9 * s[0]


def repeated_heads(seed):
    """Heads whose leading singular values are exactly equal, which the
    rounding of a planted spectrum to fp32 does not give: equal blocks on the
    diagonal, a block times a Hadamard matrix, a scaled permutation, equal
    unit cells with a smaller rest."""
    g = np.random.default_rng(seed)
    sylvester = np.array([[1.0]])
    while len(sylvester) < 128:
        sylvester = np.block([[sylvester, sylvester], [sylvester, -sylvester]])
    heads = [np.kron(np.eye(128 // n), g.standard_normal((n, n))) for n in (64, 43, 32, 16, 4)]
    heads = [np.pad(h, (0, 128 - len(h))) for h in heads]
    heads += [np.kron(sylvester[:128 // n, :128 // n], g.standard_normal((n, n))) for n in (64, 32)]
    heads += [sylvester, 0.25 * np.eye(128)[g.permutation(128)]]
    cells = np.zeros((128, 128))
    cells[np.arange(6), np.arange(6)] = 2.0
    cells[6:, 6:] = 0.01 * g.standard_normal((122, 122))
    return np.stack(heads + [cells]).astype(np.float32)


def test_exactly_repeated_singular_values(device):
    """Where the fourth singular value is above the fifth the product is
    unique and checked; where it is not, the fit is a rank-4 part of the head
    that holds its four largest singular values."""
    dense = repeated_heads(920)
    print(f"exact SVD initializer, repeated singular values, heads={len(dense)}", flush=True)
    provider, got = run(dense)
    assert (got[6] == 0).all()
    unique = []
    for h, p in enumerate(host(provider).astype(np.float64)):
        s = np.linalg.svd(p, compute_uv=False)
        if s[3] - s[4] > 1e-3 * s[0]:
            unique.append(h)
        fit = p - got[5][h].astype(np.float64)
        left = np.linalg.svd(p - fit, compute_uv=False)
        # The best rank-4 approximation, and what it leaves.
        assert abs(np.linalg.norm(p - fit) - np.linalg.norm(s[4:])) <= 1e-6 * s[0], h
        assert abs(left[0] - s[4]) <= 1e-6 * s[0], h
    assert len(unique) >= 2
    check_heads(dense[unique], [g[unique] for g in got])


def few_line_heads(seed):
    """Provider heads ([value][key]) with one to three nonzero value rows or
    key columns, side by side and scattered, and with equal rows: what is left
    behind the triplets found is rounding noise inside their own span."""
    g = np.random.default_rng(seed)
    heads = []
    for lines in ([0], [0, 1], [0, 1, 2], [127], [125, 126, 127], [5, 60], [5, 60, 101]):
        head = np.zeros((128, 128))
        head[lines] = g.standard_normal((len(lines), 128))
        heads += [head, head.T, 0.01 * head]
    for lines in ([3, 90], [3, 90, 100], [40, 41, 42, 43]):  # equal rows
        head = np.zeros((128, 128))
        head[lines] = g.standard_normal(128)
        heads += [head, head.T]
        other = head.copy()
        other[7] = g.standard_normal(128)
        heads += [other, other.T]
    return np.stack(heads).astype(np.float32)


def test_heads_of_few_rows_or_columns(device):
    """Triplets beyond a head's rank are zero or at rounding level, never the
    earlier ones once more: the fit, the fp16 pair and the residual against the
    float64 SVD, everything finite."""
    provider = few_line_heads(900)
    dense = np.ascontiguousarray(provider.transpose(0, 2, 1))
    print(f"exact SVD initializer, few rows, heads={len(dense)}", flush=True)
    _, got = run(dense)
    for a in got:
        assert np.isfinite(a.view(np.float16) if a.dtype == np.uint16 else a).all()
    check_heads(dense, got, rank_deficient=range(len(dense)))


@pytest.mark.parametrize("count", [2, 97, 700])
def test_heads_left_to_jacobi_share_a_batch(device, count):
    """Every second head a scaled permutation matrix, which the direct form
    leaves to the Jacobi kernel (350 of 700 heads, more than its 256
    workgroups): each keeps four of the 128 equal triplets, and the heads
    between come out with the bytes they have alone."""
    g = np.random.default_rng(930)
    dense = datagen.c1_heads(count, 931)
    for h in range(1, count, 2):
        dense[h] = np.float32(2.0 ** (h % 7 - 3)) * np.eye(128, dtype=np.float32)[g.permutation(128)]
    print(f"exact SVD initializer, heads left to Jacobi, heads={count}", flush=True)
    provider, got = run(dense)
    assert (got[6] == 0).all()
    p = host(provider)
    for h in range(1, count, 2):
        size = np.abs(p[h]).max()
        left = np.sort(np.linalg.svd(got[5][h].astype(np.float64), compute_uv=False)) / size
        assert np.abs(left[:4]).max() <= 1e-6 and np.abs(left[4:] - 1.0).max() <= 1e-6, h
    _, alone = run(dense[::2])
    for a, b in zip(got, alone):
        assert np.ascontiguousarray(a[::2]).tobytes() == b.tobytes()


def test_residual_may_overwrite_the_provider_state(device):
    """residual naming the provider buffer itself: each cell is read for the
    last time by the thread that writes it."""
    dense = mixed_heads(9, 700)
    provider = torch.from_numpy(np.ascontiguousarray(dense.transpose(0, 2, 1))).cuda()
    apart = [host(t) for t in codec.exact_svd_boundary(provider)]
    inside = [host(t) for t in codec.exact_svd_boundary(provider, residual=provider)]
    print("exact SVD initializer in place", flush=True)
    for a, b in zip(apart, inside):
        assert a.tobytes() == b.tobytes()


def test_the_same_bytes_on_every_run(device):
    """The four wavefronts of a head orthogonalize the same four vectors, each
    keeping one: 1,040 heads, two per CU at once and a last round of a few,
    come out with the same bytes every time."""
    dense = np.concatenate([mixed_heads(24, 800)] * 40 + [datagen.c1_heads(80, 801)])
    provider = torch.from_numpy(np.ascontiguousarray(dense.transpose(0, 2, 1))).cuda()
    print(f"exact SVD initializer, repeated, heads={len(dense)}", flush=True)
    first = [host(t) for t in codec.exact_svd_boundary(provider)]
    for a in first[:-1]:  # equal heads, equal bytes
        for copy in range(1, 40):
            assert a[24 * copy:24 * copy + 24].tobytes() == a[:24].tobytes()
    for _ in range(6):
        again = [host(t) for t in codec.exact_svd_boundary(provider)]
        for a, b in zip(first, again):
            assert a.tobytes() == b.tobytes()
