"""ModUp and ModDown where the conversion runs on the matrix cores, fused with the targets' column pass:
source counts on both sides of every operand size (2, 3, 8, 9, 12, 13, 16), partly filled last digits,
target counts that do and do not fill the groups of four, and extreme inputs; against the oracle."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


# (logN, Q towers, special primes, dnum, first / scaling / special bits): alpha = ceil(L1 / dnum)
SHAPES = [
    (12, 5, 2, 2, (60, 50, 60)),     # alpha 3, K 2: ModUp fused, ModDown not
    (12, 16, 8, 2, (60, 50, 60)),    # 8 and 8 sources
    (13, 18, 9, 2, (60, 50, 60)),    # 9 and 9
    (13, 23, 12, 2, (60, 59, 60)),   # 12 and 12, every target on the integer path
    (14, 26, 13, 2, (60, 50, 60)),   # 13 and 13
    (12, 31, 16, 2, (60, 50, 60)),   # 16 and 16, the last digit of 15
    (15, 7, 3, 3, (60, 50, 60)),     # 3 and 3
    (16, 10, 4, 3, (60, 50, 60)),    # 4 and 4, the last digit of 2
    (12, 9, 5, 2, (56, 49, 58)),     # primes down to 49 bits
    (12, 9, 5, 2, (55, 46, 55)),     # below the fused range: the general path
    (12, 9, 5, 2, (61, 55, 61)),     # above it
    (11, 8, 4, 2, (60, 50, 60)),     # a ring below its sizes
]


@pytest.mark.parametrize("shape", SHAPES, ids=lambda s: f"n{s[0]}-q{s[1]}-p{s[2]}-d{s[3]}-{s[4][1]}bit")
def test_modup_moddown(fh, oracle_mod, shape):
    logN, L1, K, dnum, bits = shape
    g = fh.Context(logN, L1, K, dnum, first_bits=bits[0], scale_bits=bits[1], aux_bits=bits[2])
    try:
        o = oracle_mod.Ctx(logN, [int(q) for q in g.moduli], L1, K, dnum)
        qs = np.array([int(m) for m in g.moduli], dtype=np.uint64)
        alpha = -(-L1 // dnum)
        for l in sorted({L1 - 1, alpha, alpha - 1, 0, L1 // 2}):
            ids, ext = list(range(l + 1)), l + 1 + K
            eids = o.ext_pids(l)
            beta = o.num_digits(l)
            # coefficients of every extreme: the transforms of all q-1, of 0, and of an impulse
            top = np.ascontiguousarray(np.broadcast_to(qs[ids][:, None] - np.uint64(1), (l + 1, o.N)))
            etop = np.ascontiguousarray(np.broadcast_to(qs[eids][:, None] - np.uint64(1), (ext, o.N)))
            inputs = [(o.random_poly(50 + l, ids), o.random_poly(70 + l, eids)), (o.ntt(top, ids), o.ntt(etop, eids)), (top, etop),
                      (np.zeros_like(top), np.zeros_like(etop))]
            for i, (x, xe) in enumerate(inputs):
                print(f"[conv cols] {shape} level {l} input {i}", flush=True)
                d, dig = g.to_device(x), g.array((beta * ext, o.N))
                g.modup(d, l, dig)
                assert np.array_equal(dig.download(), o.modup(x, l)), (l, i)
                two = np.concatenate([xe, o.random_poly(90 + l, eids)])
                de, out = g.to_device(two), g.array((2 * (l + 1), o.N))
                g.moddown(de, l, 2, out)
                assert np.array_equal(out.download(), np.concatenate([o.moddown(two[:ext], l), o.moddown(two[ext:], l)])), (l, i)
                for a in (d, dig, de, out):
                    a.free()
    finally:
        g.close()


# the operand sizes at the rings that the shapes above leave out (at N=2^14 and more the largest keeps
# some of its operands in scratch memory)
@pytest.mark.parametrize("shape", [(13, 26, 13, 2), (14, 18, 9, 2), (15, 18, 9, 2), (15, 29, 15, 2), (16, 24, 12, 2), (16, 31, 16, 2)],
                         ids=lambda s: f"n{s[0]}-q{s[1]}-p{s[2]}-d{s[3]}")
def test_modup_moddown_at_the_top_level(fh, oracle_mod, shape):
    logN, L1, K, dnum = shape
    g = fh.Context(logN, L1, K, dnum)
    try:
        o = oracle_mod.Ctx(logN, [int(q) for q in g.moduli], L1, K, dnum)
        qs, l = np.array([int(m) for m in g.moduli], dtype=np.uint64), L1 - 1
        ids, eids, ext = list(range(L1)), o.ext_pids(l), L1 + K
        top = lambda pids: np.ascontiguousarray(np.broadcast_to(qs[pids][:, None] - np.uint64(1), (len(pids), o.N)))
        for i, (x, xe) in enumerate([(o.random_poly(50, ids), o.random_poly(70, eids)), (o.ntt(top(ids), ids), o.ntt(top(eids), eids))]):
            print(f"[conv cols] {shape} input {i}", flush=True)
            d, dig = g.to_device(x), g.array((o.num_digits(l) * ext, o.N))
            g.modup(d, l, dig)
            assert np.array_equal(dig.download(), o.modup(x, l)), i
            de, out = g.to_device(xe), g.array((L1, o.N))
            g.moddown(de, l, 1, out)
            assert np.array_equal(out.download(), o.moddown(xe, l)), i
            for a in (d, dig, de, out):
                a.free()
    finally:
        g.close()


def test_many_polynomials(fh, oracle_mod):
    """Launches of one chunk of targets per workgroup and of several, and the job tables of a mixed-level
    batch, give the same rotation."""
    logN, L1, K, dnum = 13, 12, 6, 2
    g = fh.Context(logN, L1, K, dnum)
    try:
        o = oracle_mod.Ctx(logN, [int(q) for q in g.moduli], L1, K, dnum)
        key = np.concatenate([o.random_poly(10 + i, list(range(L1 + K))) for i in range(2 * dnum)])
        kk, gal, l = g.key(key), g.galois_index(3), L1 - 1
        n = 70
        cts = np.concatenate([o.random_poly(200 + (i % 5), list(range(l + 1))) for i in range(2 * n)])
        d, out = g.to_device(cts), g.array((2 * n * (l + 1), o.N))
        g.rotate_batch(d, n, l, [kk] * n, [gal] * n, out)
        got = out.download().reshape(n, 2 * (l + 1), o.N)
        src = cts.reshape(n, 2 * (l + 1), o.N)
        for i in (0, 1, 34, n - 1):
            assert np.array_equal(got[i], o.eval_rotate(src[i], l, key, gal)), i
        b, out2 = fh.Batch(g), g.array((2 * n * (l + 1), o.N))
        for i in range(n):
            b.rotate(d.addr(i * 2 * (l + 1) * o.N), l, kk, gal, out2.addr(i * 2 * (l + 1) * o.N))
        b.run()
        assert np.array_equal(out2.download().reshape(got.shape), got)
        b.free()
        kk.free()
    finally:
        g.close()


@pytest.mark.parametrize("logN,L1,K,splits", [(13, 6, 3, 0), (12, 6, 1, 0), (12, 2, 3, 0), (13, 4, 2, 1), (11, 6, 3, 1)])
def test_autotuned_context_keeps_the_fused_conversions(fh, oracle_mod, logN, L1, K, splits):
    """The autotuner times transforms alone, so it may not choose a split that the fused conversions are not
    built for: it tries other splits only where no conversion of the context is fused."""
    g = fh.Context(logN, L1, K, 2)
    try:
        o = oracle_mod.Ctx(logN, [int(q) for q in g.moduli], L1, K, 2)
        r = g.autotune(2)
        assert r["candidates"] == 1 + splits + 4, r     # the default, other splits, four workgroup sizes
        key = np.concatenate([o.random_poly(10 + i, list(range(L1 + K))) for i in range(4)])
        ct = np.concatenate([o.random_poly(30 + i, list(range(L1))) for i in range(2)])
        kk, gal, d, out = g.key(key), g.galois_index(1), g.to_device(ct), g.array((2 * L1, o.N))
        g.profile()
        g.profile_reset()
        g.eval_rotate(d, L1 - 1, kk, gal, out)
        assert np.array_equal(out.download(), o.eval_rotate(ct, L1 - 1, key, gal))
        assert g.profile_read("modup_conv_cols")[0] == (logN >= 12 and L1 // 2 > 2)
        assert g.profile_read("moddown_conv_cols")[0] == (logN >= 12 and K > 2)
    finally:
        g.close()
