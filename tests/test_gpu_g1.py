"""GPU parity: G1 tensor kernels, Pedersen commitment (fixed-base windowed MSM) and its opening, compared
with the CPU oracle as group elements (both sides normalised to z = ONE, which makes them byte-equal)."""
import random
from operator import mul

import numpy as np
import pytest

from zkhelp import (G1_X, G1_Y, P_MOD, R_MOD, affine_to_jac, ec_add, ec_mul, fr_array, fr_ints, jac_to_affine, load_oracle,
                    mt_random_vec, orc_check)

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def pv():
    from gpuhelp import Prover
    return Prover()


@pytest.fixture(scope="module")
def orc():
    return load_oracle()


def norm(orc, pts):
    pts = np.ascontiguousarray(pts, dtype=np.uint32).reshape(-1, 36)
    out = np.zeros_like(pts)
    orc_check(orc.orc_g1_op(3, pts, pts, out, pts.shape[0]))
    return out


def oracle_gens(orc, seed, n):
    orc.orc_seed(seed)
    g = np.zeros((n, 36), np.uint32)
    orc_check(orc.orc_commitment_random(n, g))
    return g


def test_generators_match_oracle_stream(pv, orc):
    pv.seed(321)
    g = pv.commitment_random(8)
    exp = oracle_gens(orc, 321, 8)
    assert (norm(orc, g.host()) == norm(orc, exp)).all()
    assert jac_to_affine(g.host()[0]) == ec_mul(fr_ints(mt_random_vec(np.random.RandomState(321), 1))[0], (G1_X, G1_Y))


@pytest.mark.parametrize("n", [1, 65, (1 << 17) - 1, (1 << 17) + 130])
def test_normalisation_at_the_edges_of_its_lane_counts(pv, orc, n):
    """one point a lane up to 2^17, four above, infinities among them; a few points tiled, since normalisation takes each alone"""
    few = oracle_gens(orc, 17, 5)
    doubled = np.zeros_like(few)
    orc_check(orc.orc_g1_op(0, few, few, doubled, 5))           # z != 1
    few = np.concatenate([few, doubled, np.zeros((1, 36), np.uint32)])
    at = np.arange(n) % 11
    got = pv.g1_binop(3, pv.g1_from_host(few[at])).host()
    assert (got == norm(orc, few)[at]).all()


def test_elementwise_and_special_cases(pv, orc):
    gens = oracle_gens(orc, 11, 16)
    inf = np.zeros(36, np.uint32)
    A = gens.copy()
    B = gens[::-1].copy()
    B[0] = A[0]                      # equal points -> doubling branch
    neg = np.zeros_like(A[:1])
    orc_check(orc.orc_g1_op(4, A[1:2].copy(), A[1:2].copy(), neg, 1))
    B[1] = neg[0]                    # opposite points -> infinity
    A[2] = inf                       # infinity + Q
    B[3] = inf                       # P + infinity
    hA, hB = pv.g1_from_host(A), pv.g1_from_host(B)
    exp = np.zeros_like(A)
    orc_check(orc.orc_g1_op(0, A, B, exp, 16))
    got = pv.g1_binop(0, hA, hB).host()
    assert (norm(orc, got) == norm(orc, exp)).all()
    assert not norm(orc, got)[1].any()          # canonical infinity = all-zero limbs
    # subtraction and negation
    nb = np.zeros_like(B)
    orc_check(orc.orc_g1_op(4, B, B, nb, 16))
    orc_check(orc.orc_g1_op(0, A, nb, exp, 16))
    assert (norm(orc, pv.g1_binop(1, hA, hB).host()) == norm(orc, exp)).all()
    assert (norm(orc, pv.g1_binop(2, hB).host()) == norm(orc, nb)).all()
    # device-side normalisation equals the oracle's
    assert (pv.g1_binop(3, hA).host() == norm(orc, A)).all()
    # broadcast add / mixed add of one point
    P = gens[5]
    Pb = np.tile(P, (16, 1))
    orc_check(orc.orc_g1_op(0, A, Pb, exp, 16))
    assert (norm(orc, pv.g1_pointop(0, hA, P).host()) == norm(orc, exp)).all()
    Pn = norm(orc, P)[0]
    assert (norm(orc, pv.g1_pointop(2, hA, Pn).host()) == norm(orc, exp)).all()


def test_affine_tensor_ops(pv, orc, tmp_path):
    """G1TensorAffine against the Jacobian arithmetic of the oracle: mixed additions and subtractions (also in place,
    with an equal point -> doubling, an opposite point -> infinity and an infinite left operand), negation, the
    conversion, the file round trip and the element read."""
    n = 70                                         # more than one workgroup
    gens = oracle_gens(orc, 12, n)
    A = gens.copy()
    B = norm(orc, gens[::-1].copy())
    B[0] = norm(orc, A[:1])[0]                     # equal
    neg = np.zeros_like(A[:1])
    orc_check(orc.orc_g1_op(4, A[1:2].copy(), A[1:2].copy(), neg, 1))
    B[1] = norm(orc, neg)[0]                       # opposite
    A[2] = np.zeros(36, np.uint32)                 # infinity + Q
    aff = np.ascontiguousarray(B[:, :24])
    hA = pv.g1_from_host(A)
    exp, nb = np.zeros_like(A), np.zeros_like(B)
    orc_check(orc.orc_g1_op(2, A, B, exp, n))
    for op in (0, 2):
        got = norm(orc, pv.g1_affineop(op, hA, aff).host())
        assert (got == norm(orc, exp)).all() and not got[1].any()
    orc_check(orc.orc_g1_op(4, B, B, nb, n))
    orc_check(orc.orc_g1_op(2, A, nb, exp, n))
    for op in (1, 3):
        assert (norm(orc, pv.g1_affineop(op, hA, aff).host()) == norm(orc, exp)).all()
    assert (pv.g1_affineop(4, hA, aff).host() == B).all()                          # z = one in Montgomery form
    assert (pv.g1_affineop(5, hA, aff).host() == norm(orc, nb)).all()
    assert (pv.g1_affineop(6, hA, aff, str(tmp_path / "aff.bin")).host() == B).all()
    assert (tmp_path / "aff.bin").stat().st_size == n * 96
    assert (pv.g1_affineop(7, hA, aff).host() == B[-1:]).all()
    with pytest.raises(RuntimeError):
        pv.g1_affineop(0, hA, aff[:5])


def test_scalar_mul_sum_rowsum_me(pv, orc):
    gens = oracle_gens(orc, 12, 8)
    rng = random.Random(3)
    ks = [0, 1, 2, R_MOD - 1, 2 ** 31 - 1] + [rng.randrange(R_MOD) for _ in range(19)]   # 24 = 3 x 8 scalars, broadcast over the generators
    S = fr_array(ks)
    exp = np.zeros((24, 36), np.uint32)
    orc_check(orc.orc_g1_mul(gens, 8, S, exp, 24, 0))
    hG, hS = pv.g1_from_host(gens), pv.from_fr(S)
    got = pv.g1_scalar_mul(hG, hS)
    assert (norm(orc, got.host()) == norm(orc, exp)).all()
    tot = np.zeros(36, np.uint32)
    orc_check(orc.orc_g1_sum(exp, 24, tot))
    assert (norm(orc, pv.g1_sum(got)) == norm(orc, tot)).all()
    rows = np.zeros((3, 36), np.uint32)
    for r in range(3):
        orc_check(orc.orc_g1_sum(exp[8 * r:8 * r + 8].copy(), 8, rows[r]))
    assert (norm(orc, pv.g1_rowwise_sum(got, 3, 8).host()) == norm(orc, rows)).all()
    u = mt_random_vec(np.random.RandomState(4), 3)
    me = np.zeros(36, np.uint32)
    orc_check(orc.orc_g1_me(gens, 8, u, 3, me))
    assert (norm(orc, pv.g1_me(hG, u)) == norm(orc, me)).all()
    # larger sum exercising the segmented reduction
    big = np.tile(gens, (200, 1))[:1500]
    orc_check(orc.orc_g1_sum(big, 1500, tot))
    assert (norm(orc, pv.g1_sum(pv.g1_from_host(big))) == norm(orc, tot)).all()


@pytest.mark.parametrize("m,n,lim", [(1, 1, 100), (3, 4, 2 ** 15), (16, 64, 2 ** 14), (5, 64, 2 ** 31 - 1), (300, 32, 2 ** 13)])
def test_commit_int_matches_oracle(pv, orc, m, n, lim):
    print("case", m, n, lim, flush=True)
    gens = oracle_gens(orc, 13 + n, n)
    rng = np.random.default_rng(m * n)
    t = rng.integers(-lim, lim, m * n, endpoint=True).astype(np.int64)
    t[0] = 0
    if m * n > 2:
        t[1], t[2] = lim, -lim
    T = fr_array([int(x) % R_MOD for x in t])
    exp = np.zeros((m, 36), np.uint32)
    orc_check(orc.orc_commit_int(gens, n, T, m * n, exp))
    got = pv.commit_int(pv.g1_from_host(gens), pv.from_fr(T)).host()
    assert (norm(orc, got) == norm(orc, exp)).all()


@pytest.mark.parametrize("m,n,lim", [(40, 100, 1), (5, 64, 7), (3, 520, 9), (2060, 260, 5), (2, 8192, 3), (1, 5000, 2 ** 31 - 1), (3, 129, 9), (200, 300, 2 ** 12), (9, 33, 2 ** 20)])
def test_commit_int_tables_of_every_shape_match_the_oracle(pv, orc, m, n, lim):
    """Tables whose first entries (k_msm_table_first) are all of a window, none, or as many as two waves a SIMD have lanes for, and rows of
    one to 256 parts; one generator is infinity, two are equal."""
    gens = oracle_gens(orc, 90 + n, n)
    gens[1] = 0
    gens[2] = gens[3]
    rng = np.random.default_rng(m * n)
    t = rng.integers(-lim, lim, m * n, endpoint=True).astype(np.int64)
    t[0], t[5], t[n - 1] = -lim, -2 ** 31 if lim > 2 ** 30 else lim, lim
    T = fr_array([int(x) % R_MOD for x in t])
    exp = np.zeros((m, 36), np.uint32)
    orc_check(orc.orc_commit_int(gens, n, T, m * n, exp))
    assert (norm(orc, pv.commit_int(pv.g1_from_host(gens), pv.from_fr(T)).host()) == norm(orc, exp)).all()


@pytest.mark.parametrize("m,n,lim", [(3000, 40, 4000), (4, 2048, 700), (2, 8192, 2 ** 30), (300, 7, 2 ** 20)])
def test_commit_int_of_generators_of_small_order_matches_the_oracle(pv, orc, m, n, lim):
    """(0, 2) has order 3: every pair of entries of its windows that k_msm_table_grow adds and subtracts is equal, opposite or holds infinity."""
    gens = oracle_gens(orc, 70 + n, n)
    for i, p in ((1, (0, 2)), (3, (0, P_MOD - 2)), (n - 2, (0, 2))):
        gens[i] = affine_to_jac(p)
    rng = np.random.default_rng(m + n)
    t = rng.integers(-lim, lim, (m, n), endpoint=True).astype(np.int64)
    t[0] = 0
    t[0, 1], t[1, 1], t[2 % m, 3] = 2, lim, -lim
    T = fr_array([int(x) % R_MOD for x in t.reshape(-1)])
    exp = np.zeros((m, 36), np.uint32)
    orc_check(orc.orc_commit_int(gens, n, T, m * n, exp))
    assert (norm(orc, pv.commit_int(pv.g1_from_host(gens), pv.from_fr(T)).host()) == norm(orc, exp)).all()


@pytest.mark.parametrize("bad", [2 ** 31, R_MOD - 2 ** 31 - 1, 2 ** 32, 2 ** 64, R_MOD - 2 ** 64, 1 << 224, (R_MOD >> 64) << 64, R_MOD - (1 << 224)])
def test_commit_int_refuses_what_is_no_int32(pv, orc, bad):
    gens = pv.g1_from_host(oracle_gens(orc, 14, 8))
    ok = [0, 1, 2 ** 31 - 1, R_MOD - 1, R_MOD - 2 ** 31, 5, 6, 7]
    pv.commit_int(gens, pv.from_fr(fr_array(ok)))
    with pytest.raises(RuntimeError, match="int32"):
        pv.commit_int(gens, pv.from_fr(fr_array(ok[:7] + [bad])))


def test_commit_int_rejects_non_integer_scalars_and_is_linear(pv, orc):
    gens = oracle_gens(orc, 14, 8)
    hG = pv.g1_from_host(gens)
    bad = fr_array([R_MOD >> 1] * 8)
    with pytest.raises(RuntimeError, match="int32"):
        pv.commit_int(hG, pv.from_fr(bad))
    rng = np.random.default_rng(9)
    a, b = rng.integers(-1000, 1000, 8), rng.integers(-1000, 1000, 8)
    ca = jac_to_affine(pv.commit_int(hG, pv.from_i32(a)).host()[0])
    cb = jac_to_affine(pv.commit_int(hG, pv.from_i32(b)).host()[0])
    cab = jac_to_affine(pv.commit_int(hG, pv.from_i32(a + b)).host()[0])
    assert ec_add(ca, cb) == cab
    # the general-scalar commit agrees with commit_int on integers
    assert jac_to_affine(pv.commit(hG, pv.from_i32(a)).host()[0]) == ca


# 300 x 1: raw small integers, whose negative embeddings share their high bytes (one bucket receives whole chunks);
# up to 9001 x 1: all rounds in one batch of sums over the generators, 4500 x 2 with more than one chunk of the bucket kernel and
# odd sizes on the way; 20000 x 2 and 70000 x 1: three rounds as one fold beside the batch of their sums, then the batched rest
@pytest.mark.parametrize("n,m", [(4, 2), (8, 1), (16, 4), (5, 3), (1, 2), (300, 1), (4500, 2), (9001, 1), (20000, 2), (70000, 1)])
def test_open_value_and_g1_transcript(pv, orc, n, m):
    gens = oracle_gens(orc, 15 + n, n)
    rng = np.random.default_rng(n * m)
    t = rng.integers(-2 ** 15, 2 ** 15, m * n).astype(np.int64)
    T = fr_array([int(x) % R_MOD for x in t])
    k = (n - 1).bit_length() + (m - 1).bit_length()
    u = mt_random_vec(np.random.RandomState(16), k)
    exp_proof = np.zeros((3 * (n - 1).bit_length() + 1, 36), np.uint32)
    exp_val = np.zeros(8, np.uint32)
    # rows are padded to a power of two exactly as verifyWeightClaim pads the weight
    mp = 1 << (m - 1).bit_length()
    Tp = np.concatenate([T, np.zeros(((mp - m) * n, 8), np.uint32)])
    orc_check(orc.orc_open(gens, n, Tp, mp * n, mp, u, k, exp_proof, exp_val))
    hG, hT = pv.g1_from_host(gens), pv.from_fr(Tp)
    com = pv.commit_int(hG, hT)
    val, proof = pv.open(hG, hT, com, u)
    assert (val == exp_val).all()
    assert proof.shape == exp_proof.shape
    assert (norm(orc, proof) == norm(orc, exp_proof)).all()


# up to 256: k_msm_few, with eight windows a wave (up to 64 elements), four (128) or two; 257: sorted lists
@pytest.mark.parametrize("n,val", [(64, 7), (65, -3), (128, 70000), (129, -3), (200, 2 ** 31 - 1), (256, 70000), (257, 70000), (300, 70000), (5000, -3), (5000, 0)])
def test_open_with_equal_scalars(pv, orc, n, val):
    """Every scalar in the same bucket of every window (norm weights share their high bytes; here all bytes): the
    bucket sums must not depend on how the elements spread over the buckets."""
    gens = oracle_gens(orc, 40 + n, n)
    T = fr_array([val % R_MOD] * n)
    k = (n - 1).bit_length()
    u = mt_random_vec(np.random.RandomState(17), k)
    exp_proof = np.zeros((3 * k + 1, 36), np.uint32)
    exp_val = np.zeros(8, np.uint32)
    orc_check(orc.orc_open(gens, n, T, n, 1, u, k, exp_proof, exp_val))
    hG, hT = pv.g1_from_host(gens), pv.from_fr(T)
    com = pv.commit_int(hG, hT)
    val_got, proof = pv.open(hG, hT, com, u)
    assert (val_got == exp_val).all()
    assert (norm(orc, proof) == norm(orc, exp_proof)).all()


@pytest.mark.parametrize("counts", [[1, 64], [32] * 3, [127, 1], [97, 32], [200, 55], [97, 97, 62], [1, 255], [128] * 2, [256, 1], [200, 57], [96, 97, 107], [400, 113], [97, 97, 97, 97, 97, 27], [150, 600, 97, 1200, 98, 255, 96, 400], [97] * 42, [2048, 2048], [128] * 20 + [64] * 16])
def test_open_with_several_digits_shared_by_many_scalars(pv, orc, counts):
    """Few scalars (256 at most, a path of its own with eight, four or two windows a wave) and many: buckets that span one lane's share to all of them, whose ends fall
    inside and at the ends of the shares; buckets about the size from which a list is cut into pieces."""
    n = sum(counts)
    gens = oracle_gens(orc, 41 + n, n)
    t = np.repeat(np.arange(1, len(counts) + 1), counts)
    t[::3] *= -1
    T = fr_array([int(x) % R_MOD for x in np.random.default_rng(n).permutation(t)])
    k = (n - 1).bit_length()
    u = mt_random_vec(np.random.RandomState(18), k)
    exp_proof = np.zeros((3 * k + 1, 36), np.uint32)
    exp_val = np.zeros(8, np.uint32)
    orc_check(orc.orc_open(gens, n, T, n, 1, u, k, exp_proof, exp_val))
    hG, hT = pv.g1_from_host(gens), pv.from_fr(T)
    com = pv.commit_int(hG, hT)
    val_got, proof = pv.open(hG, hT, com, u)
    assert (val_got == exp_val).all()
    assert (norm(orc, proof) == norm(orc, exp_proof)).all()


def test_open_with_equal_opposite_and_infinite_generators_in_the_first_round(pv, orc):
    """Pairs of equal generators (their sum is a doubling), of opposite ones (their sum is infinity), with an infinite
    member, and an infinite pair, in the bucket sums: 8200 generators take all their rounds as one batch.  The folds meet such
    generators in test_open_follows_the_logarithms_of_its_generators and its batched counterpart."""
    n = 8200
    gens = oracle_gens(orc, 77, n)
    neg = np.zeros((1, 36), np.uint32)
    gens[1] = gens[0]
    orc_check(orc.orc_g1_op(4, gens[2:3].copy(), gens[2:3].copy(), neg, 1))
    gens[3] = neg[0]
    gens[5] = 0
    gens[6] = 0
    gens[7] = 0
    gens[8] = 0
    T = mt_random_vec(np.random.RandomState(3), n)
    k = (n - 1).bit_length()
    u = mt_random_vec(np.random.RandomState(18), k)
    exp_proof = np.zeros((3 * k + 1, 36), np.uint32)
    exp_val = np.zeros(8, np.uint32)
    orc_check(orc.orc_open(gens, n, T, n, 1, u, k, exp_proof, exp_val))
    hG, hT = pv.g1_from_host(gens), pv.from_fr(T)
    com = pv.g1_from_host(np.zeros((1, 36), np.uint32))
    val_got, proof = pv.open(hG, hT, com, u)
    assert (val_got == exp_val).all()
    assert (norm(orc, proof) == norm(orc, exp_proof)).all()


def test_open_begin_end_matches_open_through_the_c_abi(orc):
    """zk_g1_open_begin/_end (openings on the library's own streams, several in flight, results fetched in another
    order) deliver exactly what zk_g1_open delivers: the proof points are normalised, so even the bytes agree."""
    import ctypes
    from gpuhelp import Hip, c_void_p, c_size_t, c_int
    hip = Hip()
    cases = []
    for n, seed in ((37, 3), (9000, 4), (1, 5)):
        gens = oracle_gens(orc, 60 + n, n)
        S = mt_random_vec(np.random.RandomState(seed), n)
        k = max(1, (n - 1).bit_length())
        u = mt_random_vec(np.random.RandomState(seed + 10), k)
        dG, dS = hip.upload(gens), hip.upload(S)
        proof = np.zeros((3 * k + 1, 36), np.uint32)
        val = np.zeros(8, np.uint32)
        hip.call("zk_g1_open", proof, val, c_void_p(dS), c_void_p(dG), c_size_t(n), u, c_int(k), None)
        cases.append((n, k, u, dG, dS, proof, val))
    handles = []
    for n, k, u, dG, dS, _, _ in cases:
        h = c_void_p()
        hip.call("zk_g1_open_begin", ctypes.byref(h), c_void_p(dS), c_void_p(dG), c_size_t(n), u, c_int(k), None)
        handles.append(h)
    for (n, k, u, dG, dS, proof, val), h in reversed(list(zip(cases, handles))):
        p2 = np.zeros_like(proof)
        v2 = np.zeros(8, np.uint32)
        hip.call("zk_g1_open_end", h, p2, v2)
        assert (v2 == val).all(), n
        assert (p2 == proof).all(), n
    for _, _, _, dG, dS, _, _ in cases:
        hip.free(dG)
        hip.free(dS)


def test_open_batch_over_prepared_generators_matches_single_openings(orc):
    """zk_g1_open_begin_batch (openings of one size as ONE job: every round's kernels launched once for all of them) over
    generators prepared with zk_g1_open_prepare delivers, opening by opening, the bytes of zk_g1_open.  Jobs on both
    sides of the 16384 generators (all openings together) from which on every round is in one batch: above, the first round runs on the
    prepared tables.  Special generators (equal, opposite, infinite) in one member of the batch, and zk_g1_open_begin_prepared
    alone.  (A second round on its tables: test_open_batches_follow_the_logarithms_of_their_generators.)"""
    import ctypes
    from gpuhelp import Hip, c_void_p, c_size_t, c_int
    hip = Hip()
    for n, count in ((9001, 3), (600, 2), (4096, 8), (2049, 2)):
        k = (n - 1).bit_length()
        npts = 3 * k + 1
        gens, dG, dS, us, preps = [], [], [], [], []
        exp_p = np.zeros((count, npts, 36), np.uint32)
        exp_v = np.zeros((count, 8), np.uint32)
        for i in range(count):
            g = oracle_gens(orc, 300 + 7 * i + n, n)
            if i == 1 and n > 20:
                neg = np.zeros((1, 36), np.uint32)
                g[1] = g[0]
                orc_check(orc.orc_g1_op(4, g[2:3].copy(), g[2:3].copy(), neg, 1))
                g[3] = neg[0]
                g[6] = 0
                g[7] = 0
                g[9] = 0
                # special among the points of the second round's tables (pairs of pairs g_4j .. g_4j+3): equal odd members
                # (their difference is infinity), equal pair differences (infinity again), opposite odd members (a doubling)
                g[15] = g[13]
                g[18] = g[16]
                g[19] = g[17]
                orc_check(orc.orc_g1_op(4, g[21:22].copy(), g[21:22].copy(), neg, 1))
                g[23] = neg[0]
            S = mt_random_vec(np.random.RandomState(50 + i), n)
            u = mt_random_vec(np.random.RandomState(70 + i), k)
            gens.append(g); us.append(u)
            dG.append(hip.upload(g)); dS.append(hip.upload(S))
            print(f"open n={n} item={i}: zk_g1_open", flush=True)
            hip.call("zk_g1_open", exp_p[i], exp_v[i], c_void_p(dS[i]), c_void_p(dG[i]), c_size_t(n), u, c_int(k), None)
            pr = c_void_p()
            print(f"open n={n} item={i}: zk_g1_open_prepare", flush=True)
            hip.call("zk_g1_open_prepare", ctypes.byref(pr), c_void_p(dG[i]), c_size_t(n), None)
            preps.append(pr)
        h = c_void_p()
        sc = (c_void_p * count)(*[c_void_p(x) for x in dS])
        pp = (c_void_p * count)(*preps)
        uall = np.ascontiguousarray(np.concatenate(us), dtype=np.uint32)
        print(f"open n={n}: zk_g1_open_begin_batch of {count}", flush=True)
        hip.call("zk_g1_open_begin_batch", ctypes.byref(h), c_int(count), sc, pp, uall, c_int(k), None)
        got_p = np.zeros_like(exp_p)
        got_v = np.zeros_like(exp_v)
        hip.call("zk_g1_open_end_batch", h, got_p, got_v)
        assert (got_v == exp_v).all(), n
        assert (got_p == exp_p).all(), n
        # one prepared opening on its own
        h1 = c_void_p()
        print(f"open n={n}: zk_g1_open_begin_prepared", flush=True)
        hip.call("zk_g1_open_begin_prepared", ctypes.byref(h1), c_void_p(dS[0]), preps[0], us[0], c_int(k), None)
        p1 = np.zeros((npts, 36), np.uint32)
        v1 = np.zeros(8, np.uint32)
        hip.call("zk_g1_open_end", h1, p1, v1)
        assert (v1 == exp_v[0]).all() and (p1 == exp_p[0]).all(), n
        for pr in preps:
            hip.call("zk_g1_open_prepared_free", pr)
        for x in dG + dS:
            hip.free(x)


# two openings a job: 5000: all rounds in one batch; 9000: one round on the prepared table, or three in a span; 50000: two rounds on the tables
# and a span, or one round without tables and a span
@pytest.mark.parametrize("n,tables", [(5000, 2), (9000, 2), (9000, 0), (50000, 2), (50000, 0)])
def test_open_batch_with_row_commitments_delivers_the_points_of_the_plain_opening(pv, n, tables):
    """zk_g1_open_begin_batch_rows takes the first round's T from the tensors' row commitments (sum_r eq(u_rows, r) C_r)
    instead of summing over all generators: for commitments made by commit_int of the same tensors every point of the
    proof, T of the first round included, equals zk_g1_open's on the row-folded vector.  One tensor with a number of
    rows that is no power of two, one with a single row (no row challenge); and with another tensor's commitments only the
    T of the rounds over more than 1024 generators change."""
    import ctypes
    from gpuhelp import Hip, c_void_p, c_size_t, c_int
    hip = Hip()
    pv.lib.zkp_g1_devptr.restype = ctypes.c_void_p
    k = (n - 1).bit_length()
    npts = 3 * k + 1
    pv.seed(77)
    gens = pv.commitment_random(n)
    dG = pv.lib.zkp_g1_devptr(c_void_p(gens.h))
    prep = c_void_p()
    hip.call("zk_g1_open_prepare_tables", ctypes.byref(prep), c_void_p(dG), c_size_t(n), c_int(tables), None)
    rng = np.random.default_rng(5)
    keep, folded, coms, urows, us = [], [], [], [], []
    exp_p = np.zeros((2, npts, 36), np.uint32)
    exp_v = np.zeros((2, 8), np.uint32)
    for i, nrows in enumerate((5, 1)):
        W = pv.from_i32(rng.integers(-30000, 30000, nrows * n).astype(np.int32))
        com = pv.commit_int(gens, W)
        assert com.size == nrows
        kr = (nrows - 1).bit_length()
        ur = mt_random_vec(np.random.RandomState(40 + i), max(kr, 1))[:kr]
        f = pv.partial_me_window(W, ur, n) if kr else W
        assert f.size == n
        u = mt_random_vec(np.random.RandomState(60 + i), k)
        print(f"rows={nrows}: zk_g1_open", flush=True)
        hip.call("zk_g1_open", exp_p[i], exp_v[i], c_void_p(f.devptr), c_void_p(dG), c_size_t(n), u, c_int(k), None)
        keep += [W, com, f]
        folded.append(f); coms.append(com); urows.append(np.ascontiguousarray(ur, dtype=np.uint32)); us.append(u)

    def run(com_order):
        h = c_void_p()
        sc = (c_void_p * 2)(*[c_void_p(f.devptr) for f in folded])
        pp = (c_void_p * 2)(prep, prep)
        rows = (c_void_p * 2)(*[c_void_p(pv.lib.zkp_g1_devptr(c_void_p(coms[j].h))) for j in com_order])
        nr = np.array([coms[j].size for j in com_order], np.uint32)
        ur = (c_void_p * 2)(*[c_void_p(urows[j].ctypes.data if urows[j].size else None) for j in com_order])
        kr = np.array([urows[j].shape[0] for j in com_order], np.int32)
        uall = np.ascontiguousarray(np.concatenate(us), dtype=np.uint32)
        print(f"zk_g1_open_begin_batch_rows, commitments {com_order}", flush=True)
        hip.call("zk_g1_open_begin_batch_rows", ctypes.byref(h), c_int(2), sc, pp, uall, c_int(k), rows, nr, ur, kr, c_int(0), None)
        got_p = np.zeros_like(exp_p)
        got_v = np.zeros_like(exp_v)
        hip.call("zk_g1_open_end_batch", h, got_p, got_v)
        return got_p, got_v

    got_p, got_v = run((0, 1))
    assert (got_v == exp_v).all()
    assert (got_p == exp_p).all()
    # the statement "these are the tensor's row commitments" is the caller's: with the other tensor's, T of the first round
    # is what those commitments give, and with it T of the later rounds over more than 1024 generators, which follow from the earlier
    # rounds' points (the rest are sums over the generators); T0, T1 of every round, the folded generator and the value do not
    # depend on them
    got_p, got_v = run((1, 0))
    assert (got_v == exp_v).all()
    sizes = [n]
    while sizes[-1] > 1:
        sizes.append((sizes[-1] + 1) // 2)
    unrolled = [3 * r for r, size in enumerate(sizes) if size > 1024]
    same = np.ones(npts, bool)
    same[unrolled] = False
    assert (got_p[:, same] == exp_p[:, same]).all()
    for i in range(2):
        assert not any((got_p[i, j] == exp_p[i, j]).all() for j in unrolled)
    hip.call("zk_g1_open_prepared_free", prep)


# two openings a job.  8192: all rounds in one batch of sums over the generators, which needs no commitments; 16384: one round before that batch, or three as one fold; 32768: two rounds, or that fold
@pytest.mark.parametrize("n,R,tables", [(8192, 2, 2), (16384, 3, 3), (16384, 2, 2), (32768, 3, 3), (32768, 2, 2), (32768, 3, 2), (32768, 3, 0)])
def test_open_batch_with_cross_commitments_needs_no_sum_over_the_generators(pv, orc, n, R, tables):
    """With the cross commitments of its first R rounds -- commitments of every 2nd / 4th / 8th column of the tensor's rows
    under every 2nd / 4th / 8th generator, made here with commit_int on slices -- zk_g1_open_begin_batch_rows forms T, T0 and
    T1 of those rounds from rows x patterns points, for the rounds that come before the batch which takes all the rest (16384 generators
    of the whole job).  With three rounds of them the three rounds are one fold, from the tables of zk_g1_open_prepare_tables(.., 3)
    or, with other tables or none, as a span.  Every point of the proof equals zk_g1_open's on the row-folded vector, and at 16384 generators also the
    oracle's own opening of the padded tensor (Commitment::open, commitment.cu:133-141: row fold, then me_open), point by
    point after normalisation, so the batched path is compared with the reference's algorithm directly."""
    import ctypes
    from gpuhelp import Hip, c_void_p, c_size_t, c_int
    hip = Hip()
    pv.lib.zkp_g1_devptr.restype = ctypes.c_void_p
    k = (n - 1).bit_length()
    npts = 3 * k + 1
    pv.seed(78)
    gens = pv.commitment_random(n)
    gens_host = gens.host()
    dG = pv.lib.zkp_g1_devptr(c_void_p(gens.h))
    prep = c_void_p()
    hip.call("zk_g1_open_prepare_tables", ctypes.byref(prep), c_void_p(dG), c_size_t(n), c_int(tables), None)
    rng = np.random.default_rng(6)
    keep, folded, cross, urows, us = [], [], [], [], []
    exp_p = np.zeros((2, npts, 36), np.uint32)
    exp_v = np.zeros((2, 8), np.uint32)
    for i, nrows in enumerate((3, 4)):
        Wi = rng.integers(-30000, 30000, (nrows, n)).astype(np.int32)
        W = pv.from_i32(Wi.ravel())
        pats = [pv.commit_int(gens, W).host()]
        for q in range(R):
            half, L = 1 << q, 2 << q
            for side in (0, 1):
                for a in range(half):
                    for b in range(half):
                        s_off, g_off = (half if side else 0) + a, (0 if side else half) + b
                        sub_g = pv.g1_from_host(np.ascontiguousarray(gens_host[g_off::L]))
                        sub_w = pv.from_i32(np.ascontiguousarray(Wi[:, s_off::L]).ravel())
                        pats.append(pv.commit_int(sub_g, sub_w).host())
        assert len(pats) == 1 + 2 * (4 ** R - 1) // 3 and all(x.shape == (nrows, 36) for x in pats)
        cross.append(hip.upload(np.ascontiguousarray(np.concatenate(pats))))
        kr = (nrows - 1).bit_length()
        ur = mt_random_vec(np.random.RandomState(45 + i), kr)
        f = pv.partial_me_window(W, ur, n)
        u = mt_random_vec(np.random.RandomState(65 + i), k)
        print(f"rows={nrows}: zk_g1_open", flush=True)
        hip.call("zk_g1_open", exp_p[i], exp_v[i], c_void_p(f.devptr), c_void_p(dG), c_size_t(n), u, c_int(k), None)
        keep += [W, f]
        folded.append(f); urows.append(np.ascontiguousarray(ur, dtype=np.uint32)); us.append(u)
        if n == 16384 and R == 3:
            rows_p = 1 << kr
            Tp = np.zeros((rows_p * n, 8), np.uint32)
            Tp[:nrows * n] = fr_array([int(x) % R_MOD for x in Wi.ravel()])
            o_p, o_v = np.zeros((npts, 36), np.uint32), np.zeros(8, np.uint32)
            print(f"rows={nrows}: oracle opening over {n} generators", flush=True)
            orc_check(orc.orc_open(np.ascontiguousarray(gens_host), n, Tp, rows_p * n, rows_p, np.ascontiguousarray(np.concatenate([u, ur]), dtype=np.uint32), k + kr, o_p, o_v))
            assert (o_v == exp_v[i]).all()
            assert (norm(orc, o_p) == exp_p[i]).all()          # the product delivers its points normalised
    for cr in (R, 1):
        h = c_void_p()
        sc = (c_void_p * 2)(*[c_void_p(f.devptr) for f in folded])
        pp = (c_void_p * 2)(prep, prep)
        rows = (c_void_p * 2)(*[c_void_p(x) for x in cross])
        nr = np.array([3, 4], np.uint32)
        ur = (c_void_p * 2)(*[c_void_p(x.ctypes.data) for x in urows])
        kr = np.array([x.shape[0] for x in urows], np.int32)
        uall = np.ascontiguousarray(np.concatenate(us), dtype=np.uint32)
        print(f"zk_g1_open_begin_batch_rows with {cr} rounds of cross commitments", flush=True)
        hip.call("zk_g1_open_begin_batch_rows", ctypes.byref(h), c_int(2), sc, pp, uall, c_int(k), rows, nr, ur, kr, c_int(cr), None)
        got_p = np.zeros_like(exp_p)
        got_v = np.zeros_like(exp_v)
        hip.call("zk_g1_open_end_batch", h, got_p, got_v)
        assert (got_v == exp_v).all(), cr
        assert (got_p == exp_p).all(), cr
    hip.call("zk_g1_open_prepared_free", prep)
    for x in cross:
        hip.free(x)


def opening_logarithms(a, s, u):
    """The opening of the scalars s over the generators [a_i] G with the challenges u (Commitment::me_open, commitment.cu:109-129) in the
    exponent: the logarithms of T, T0, T1 of every round and of the folded generator, and the folded scalar."""
    out = []
    for x in u:
        if len(a) % 2:
            a, s = a + [0], s + [0]
        a0, a1, s0, s1 = a[0::2], a[1::2], s[0::2], s[1::2]
        t0, t1 = sum(map(mul, s0, a1)) % R_MOD, sum(map(mul, s1, a0)) % R_MOD
        out += [(sum(map(mul, s0, a0)) + sum(map(mul, s1, a1))) % R_MOD, t0, t1]
        a = [(q + x * (p - q)) % R_MOD for p, q in zip(a0, a1)]
        s = [(p + x * (q - p)) % R_MOD for p, q in zip(s0, s1)]
    return out + a, s[0]


def special_logarithms(seed, n, shift=0):
    """n random logarithms, among them equal, opposite and infinite generators in pairs, in pairs of pairs and in eights, also eights that
    are one generator throughout, that cancel, that hold one generator alone and, a wave's worth and more, none at all"""
    a = fr_ints(mt_random_vec(np.random.RandomState(seed), n))
    b = a[:]
    b[1], b[3], b[5], b[6], b[7] = b[0], -b[2], 0, 0, 0
    b[15], b[18], b[19], b[23] = b[13], b[16], b[17], -b[21]         # special only in the second round
    b[24:32] = [b[24]] * 8
    b[32:40] = [b[32], -b[32]] * 4
    b[40:48] = [0] * 8
    b[48:56] = [0] * 5 + [b[53]] + [0] * 2
    b[64:72] = [b[64], 0, 0, 0, -b[64], 0, 0, 0]
    b[1024:2048] = [0] * 1024
    if n % 2:
        b[n - 1] = 0 if shift else b[n - 2]
    b[:2048] = b[shift:2048] + b[:shift]
    return [x % R_MOD for x in b]


def known_generators(hip, a):
    from gpuhelp import c_size_t, c_void_p
    dA, dG = hip.upload(fr_array(a)), hip.malloc(144 * len(a))
    hip.call("zk_g1_fixed_base_mul", c_void_p(dG), np.ascontiguousarray(affine_to_jac((G1_X, G1_Y)), dtype=np.uint32), c_void_p(dA), c_size_t(len(a)), None)
    hip.sync()
    hip.free(dA)
    return dG


def assert_points_are(points, logarithms):
    assert len(points) == len(logarithms)
    for i, (p, l) in enumerate(zip(points, logarithms)):
        assert jac_to_affine(p) == (ec_mul(l, (G1_X, G1_Y)) if l else None), i


# 16385 .. 131072: three rounds in a span, then the batched rest (70001 with odd sizes throughout, 98305 with a last generator that has no
# partner); above: one round alone (2^18 + 3: two), then a span
@pytest.mark.parametrize("n", [16385, 20000, 70001, 98304, 98305, 131072, 140001, (1 << 18) + 3])
def test_open_follows_the_logarithms_of_its_generators(n):
    """An unprepared opening over generators of known logarithm, special ones among them, point by point in big-integer arithmetic."""
    from gpuhelp import Hip, c_int, c_size_t, c_void_p
    hip = Hip()
    k = (n - 1).bit_length()
    a = special_logarithms(90, n)
    S, u = mt_random_vec(np.random.RandomState(91), n), mt_random_vec(np.random.RandomState(92), k)
    dG, dS = known_generators(hip, a), hip.upload(S)
    points, value = np.zeros((3 * k + 1, 36), np.uint32), np.zeros(8, np.uint32)
    print(f"zk_g1_open n={n}", flush=True)
    hip.call("zk_g1_open", points, value, c_void_p(dS), c_void_p(dG), c_size_t(n), u, c_int(k), None)
    logs, exp_value = opening_logarithms(a, fr_ints(S), fr_ints(u))
    assert fr_ints(value)[0] == exp_value
    assert_points_are(points, logs)
    hip.free(dG)
    hip.free(dS)


@pytest.mark.parametrize("slice_bits,sign,first", [(b, s, None) for b in (15, 16, 17) for s in (1, -1)] + [(0, 1, f) for f in ((0, 0, 0), (1, 1, 1), (1, 0, 1), (R_MOD - 1, 2, 1))])
def test_span_of_rounds_whose_slices_meet_themselves(slice_bits, sign, first):
    """The slices of a span's combination added to one another as equal and as opposite points: with u = 2/3, 2/3 and 9/4 * 2^slice the
    first generator's coefficient is 2^slice, one digit in the second slice, and those of the next two are 2^(slice - 1), in the first: the
    first slice's point, +-2^slice times the generator, meets the second slice's after its doublings.  Which width a slice has follows from
    the longest of all coefficients: one of the three.  Then challenges that leave single or short coefficients."""
    from gpuhelp import Hip, c_int, c_size_t, c_void_p
    hip = Hip()
    n = 16400
    k = (n - 1).bit_length()
    u = fr_ints(mt_random_vec(np.random.RandomState(93), k))
    inv = lambda x: pow(x, -1, R_MOD)
    u[:3] = first if first is not None else (2 * inv(3) % R_MOD, 2 * inv(3) % R_MOD, 9 * inv(4) * (1 << slice_bits) % R_MOD)
    a = special_logarithms(94, n)
    for m in range(512, 600):
        a[8 * m:8 * m + 8] = [a[8 * m], sign * a[8 * m] % R_MOD, sign * a[8 * m] % R_MOD, 0, 0, 0, 0, 0]
    S = mt_random_vec(np.random.RandomState(95), n)
    dG, dS = known_generators(hip, a), hip.upload(S)
    points, value = np.zeros((3 * k + 1, 36), np.uint32), np.zeros(8, np.uint32)
    print(f"zk_g1_open n={n} slice {slice_bits} sign {sign} first {first}", flush=True)
    hip.call("zk_g1_open", points, value, c_void_p(dS), c_void_p(dG), c_size_t(n), fr_array(u), c_int(k), None)
    logs, exp_value = opening_logarithms(a, fr_ints(S), u)
    assert fr_ints(value)[0] == exp_value
    assert_points_are(points, logs)
    hip.free(dG)
    hip.free(dS)


# one batch of sums of 2^13 to 2^14 generators, whose T all follow from the final generator and scalar, unless a challenge is 0 or 1
@pytest.mark.parametrize("n", [8193, 16384])
@pytest.mark.parametrize("at,to", [(0, None), (0, 0), (12, 1), (5, R_MOD - 1)])
def test_open_whose_sums_follow_from_its_last_round(n, at, to):
    from gpuhelp import Hip, c_int, c_size_t, c_void_p
    hip = Hip()
    k = (n - 1).bit_length()
    a, S, u = special_logarithms(96, n), mt_random_vec(np.random.RandomState(97), n), fr_ints(mt_random_vec(np.random.RandomState(98), k))
    if to is not None:
        u[at] = to
    dG, dS = known_generators(hip, a), hip.upload(S)
    points, value = np.zeros((3 * k + 1, 36), np.uint32), np.zeros(8, np.uint32)
    print(f"zk_g1_open n={n} u[{at}] = {to}", flush=True)
    hip.call("zk_g1_open", points, value, c_void_p(dS), c_void_p(dG), c_size_t(n), fr_array(u), c_int(k), None)
    logs, exp_value = opening_logarithms(a, fr_ints(S), u)
    assert fr_ints(value)[0] == exp_value
    assert_points_are(points, logs)
    hip.free(dG)
    hip.free(dS)


def test_open_round_whose_lists_are_sorted_a_few_windows_at_a_time():
    """One round over so many generators that the lists of all windows of its three sums do not fit the sorting's space: small and large scalars, every eighth of them zero."""
    from gpuhelp import Hip, c_int, c_size_t, c_void_p
    hip = Hip()
    n, period = 1600000, 1 << 12
    a = special_logarithms(130, period)
    S = np.random.RandomState(131).randint(0, 1 << 32, (n, 8), dtype=np.uint64).astype(np.uint32)
    S[:, 7] %= 1944954707
    S[::8] = 0
    S[::3, 1:] = 0
    reps = -(-n // period)
    dA, dG = hip.upload(np.tile(fr_array(a), (reps, 1))[:n]), hip.malloc(144 * n)
    hip.call("zk_g1_fixed_base_mul", c_void_p(dG), np.ascontiguousarray(affine_to_jac((G1_X, G1_Y)), dtype=np.uint32), c_void_p(dA), c_size_t(n), None)
    hip.sync()
    dS, u = hip.upload(S), mt_random_vec(np.random.RandomState(132), 1)
    points, value = np.zeros((4, 36), np.uint32), np.zeros(8, np.uint32)
    print(f"zk_g1_open n={n}, one round", flush=True)
    hip.call("zk_g1_open", points, value, c_void_p(dS), c_void_p(dG), c_size_t(n), u, c_int(1), None)
    # the generators repeat with the period: the sum of all scalars that meet one of them
    tot = np.zeros((period, 8), np.int64)
    pad = np.concatenate([S, np.zeros((reps * period - n, 8), np.uint32)]).reshape(reps, period, 8)
    tot = pad.astype(np.int64).sum(axis=0)
    s = [sum(int(v) << (32 * l) for l, v in enumerate(row)) for row in tot]
    exp = [sum(map(mul, s, a)) % R_MOD, sum(map(mul, s[0::2], a[1::2])) % R_MOD, sum(map(mul, s[1::2], a[0::2])) % R_MOD]
    assert_points_are(points[:3], exp)
    for p in (dA, dG, dS):
        hip.free(p)


# 4099 x 8 and 33001: the first and the second round on their tables (odd halves); 12300 x 8: the first alone without tables, or on its table;
# 40000 x 3: three, the third without a table; 2051 x 8: the first on its table and no table for the second; 2049: sums of
# windows of 128 buckets over all the generators, in a wave a window for two members and with a lane for eight buckets for eight
@pytest.mark.parametrize("n,count,tables", [(4099, 8, 2), (33001, 1, 2), (12300, 8, 0), (12300, 8, 1), (12300, 8, 2), (40000, 3, 2), (2051, 8, 2), (2049, 2, 0), (2049, 8, 0)])
def test_open_batches_follow_the_logarithms_of_their_generators(n, count, tables):
    """zk_g1_open_begin_batch over prepared generators of known logarithm, special ones at another place in each member."""
    import ctypes
    from gpuhelp import Hip, c_int, c_size_t, c_void_p
    hip = Hip()
    k = (n - 1).bit_length()
    a, S, u, preps, keep = [], [], [], [], []
    for i in range(count):
        a.append(special_logarithms(100 + i, n, i % 3))
        S.append(mt_random_vec(np.random.RandomState(110 + i), n))
        u.append(mt_random_vec(np.random.RandomState(120 + i), k))
        dG = known_generators(hip, a[i])
        preps.append(c_void_p())
        hip.call("zk_g1_open_prepare_tables", ctypes.byref(preps[i]), c_void_p(dG), c_size_t(n), c_int(tables), None)
        hip.free(dG)
        keep.append(hip.upload(S[i]))
    h = c_void_p()
    print(f"zk_g1_open_begin_batch n={n} count={count} tables={tables}", flush=True)
    hip.call("zk_g1_open_begin_batch", ctypes.byref(h), c_int(count), (c_void_p * count)(*[c_void_p(x) for x in keep]), (c_void_p * count)(*preps),
             np.ascontiguousarray(np.concatenate(u), dtype=np.uint32), c_int(k), None)
    points, values = np.zeros((count, 3 * k + 1, 36), np.uint32), np.zeros((count, 8), np.uint32)
    hip.call("zk_g1_open_end_batch", h, points, values)
    for i in range(count):
        logs, exp_value = opening_logarithms(a[i], fr_ints(S[i]), fr_ints(u[i]))
        assert fr_ints(values[i])[0] == exp_value
        assert_points_are(points[i], logs)
    for pr, p in zip(preps, keep):
        hip.call("zk_g1_open_prepared_free", pr)
        hip.free(p)


def test_fixed_base_multiplication_equals_the_generic_one_and_big_integer_arithmetic(orc):
    """zk_g1_fixed_base_mul (what Commitment::random runs on) against zk_g1_scalar_mul on the same base and, for the
    small cases, against affine big-integer arithmetic: digits at the signed-window boundaries (127, 128, 129, bytes of
    0x80 and 0xff that carry all the way up), zero, r - 1 and integers above r up to 2^256 - 1; a second base replaces the
    table kept on the device and the first base builds it again."""
    from gpuhelp import Hip, c_void_p, c_size_t
    hip = Hip()
    edge = [0, 1, 2, 127, 128, 129, 255, 256, 0x8080, 0x80 << 248, (1 << 255) - 1, R_MOD - 1, R_MOD, R_MOD + 5,
            (1 << 256) - 1, int("80" * 32, 16), int("7f" * 32, 16), int("81" * 32, 16), 1 << 255]
    S = np.concatenate([fr_array(edge), mt_random_vec(np.random.RandomState(77), 300)])
    n = S.shape[0]
    G = affine_to_jac((G1_X, G1_Y))
    other = oracle_gens(orc, 91, 1)[0]
    dS, dF, dM, dB = hip.upload(S), hip.malloc(144 * n), hip.malloc(144 * n), hip.malloc(144)
    for base in (G, other, G):
        base = np.ascontiguousarray(base, dtype=np.uint32)
        hip.call("zk_memcpy_h2d", c_void_p(dB), base, c_size_t(144), None)
        hip.call("zk_g1_fixed_base_mul", c_void_p(dF), base, c_void_p(dS), c_size_t(n), None)
        hip.call("zk_g1_scalar_mul", c_void_p(dM), c_void_p(dB), c_void_p(dS), c_size_t(1), c_size_t(n), None)
        fixed, generic = hip.download(dF, (n, 36), np.uint32), hip.download(dM, (n, 36), np.uint32)
        assert (norm(orc, fixed) == norm(orc, generic)).all()
        assert not norm(orc, fixed)[0].any()                     # [0] B is the point at infinity
    for i in (1, 3, 4, 5, 11, 14):
        assert jac_to_affine(fixed[i]) == ec_mul(edge[i] % R_MOD, (G1_X, G1_Y)), i
    for p in (dS, dF, dM, dB):
        hip.free(p)


def test_config3_full_size_commitment_and_opening_pass_the_verifier(pv, orc):
    """A 11008 x 4096 fixed-point weight (scale 2^16, N(0, 0.02)) over 4096 generators, far beyond what the oracle can
    follow: the 11008 commitments and the opening at a random point are checked the way a verifier would, in big-integer
    affine arithmetic.  The first T of the opening is the commitments' own multilinear extension at the row challenges
    (this ties commit_int to the opening), every round satisfies T' = u(1-u) T + (1-u)^2 T0 + u^2 T1, the last one
    against [value] g_final, and the value is the tensor's multilinear extension computed apart from the opening."""
    m, n = 11008, 4096
    rng = np.random.default_rng(2024)
    W = np.round(rng.normal(0, 0.02, m * n) * 65536).astype(np.int32)
    pv.seed(33)
    hG = pv.commitment_random(n)
    hW = pv.from_i32(W)
    com = pv.commit_int(hG, hW)
    assert com.size == m
    k_in, k_out = 12, 14
    u = mt_random_vec(np.random.RandomState(34), k_in + k_out)
    val, proof = pv.open(hG, hW, com, u)
    assert proof.shape[0] == 3 * k_in + 1
    ui = fr_ints(u)
    # value = W(u_out, u_in), rows by the last 14 challenges
    assert (pv.multi_dim_me(hW, [u[k_in:], u[:k_in]], (m, n)) == val).all()
    # T of the first round = sum_rows eq(u_out, row) com_row; G1TensorJacobian::operator()(u) reads its challenges as u / R
    u_me = fr_array([x * (1 << 256) % R_MOD for x in ui[k_in:]])
    pts = [jac_to_affine(p) for p in proof]
    assert pts[0] == jac_to_affine(pv.g1_me(com, u_me))
    for r in range(k_in):
        x = ui[r]
        T, T0, T1 = pts[3 * r:3 * r + 3]
        nxt = ec_add(ec_add(ec_mul(x * (1 - x) % R_MOD, T), ec_mul((1 - x) * (1 - x) % R_MOD, T0)), ec_mul(x * x % R_MOD, T1))
        expect = pts[3 * r + 3] if r + 1 < k_in else ec_mul(fr_ints(val)[0], pts[3 * k_in])
        assert nxt == expect, r
    # linearity of the commitment on a few rows: com(a) + com(b) = com(a + b)
    rows = [0, 1, 5503, 11007]
    A = np.concatenate([W[r * n:(r + 1) * n] for r in rows])
    B = np.concatenate([W[((r + 7) % m) * n:((r + 7) % m + 1) * n] for r in rows])
    ca, cb, cab = (pv.commit_int(hG, pv.from_i32(x)).host() for x in (A, B, A + B))
    exp = np.zeros_like(ca)
    orc_check(orc.orc_g1_op(0, ca, cb, exp, len(rows)))
    assert (norm(orc, cab) == norm(orc, exp)).all()
    assert (norm(orc, ca) == norm(orc, com.host()[rows])).all()
