"""Limbs formed in the forward transform's first launch, against the oracle and Python integers: the
Rescale correction between primes of every pair of sizes, raised towers, residues of signed
coefficients up to the ends of the 64-bit range."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


# (first, scaling, special bits): fp64 to fp64 and to 60-bit primes, integers below 2^60, wide integers,
# a dropped prime far above the others (50 against 30 bits) and below them
@pytest.mark.parametrize("bits", [(60, 50, 60), (60, 59, 60), (61, 61, 61), (50, 30, 50), (30, 50, 50), (52, 48, 56)])
@pytest.mark.parametrize("logN", [10, 13])
def test_rescale_and_mod_raise(fh, oracle_mod, logN, bits):
    L1, K = 4, 1
    g = fh.Context(logN, L1, K, 2, first_bits=bits[0], scale_bits=bits[1], aux_bits=bits[2])
    try:
        o = oracle_mod.Ctx(logN, [int(q) for q in g.moduli], L1, K, 2)
        for l in range(1, L1):
            ids = list(range(l + 1))
            q = np.array([int(g.moduli[i]) for i in ids], dtype=np.uint64)[:, None]
            # the dropped limb at the ends of its range and on both sides of its half
            edge = np.zeros((l + 1, o.N), dtype=np.uint64)
            edge[:, :5] = np.concatenate([q - np.uint64(1), q >> np.uint64(1), (q >> np.uint64(1)) + np.uint64(1), np.ones_like(q), q - np.uint64(2)], axis=1)
            for x in (np.concatenate([o.random_poly(20 + l, ids), o.random_poly(30 + l, ids)]), np.concatenate([o.ntt(edge, ids), o.random_poly(40 + l, ids)])):
                print(f"[first pass] rescale logN={logN} bits={bits} level {l}", flush=True)
                d, out = g.to_device(x), g.array((2 * l, o.N))
                g.rescale(d, l, 2, out)
                assert np.array_equal(out.download(), o.rescale_ct(x, l, 2)), l
                up = g.array((2 * L1, o.N))
                g.mod_raise(d, l, 2, L1 - 1, up)
                assert np.array_equal(up.download(), o.mod_raise(x, l, L1 - 1, 2)), l
                for a in (d, out, up):
                    a.free()
    finally:
        g.close()


@pytest.mark.parametrize("bits", [(60, 50, 60), (61, 61, 61), (50, 30, 36), (35, 34, 33), (52, 51, 59)])
def test_signed_coefficients(fh, oracle_mod, bits):
    logN, L1, K = 11, 3, 1
    g = fh.Context(logN, L1, K, 1, first_bits=bits[0], scale_bits=bits[1], aux_bits=bits[2])
    try:
        o = oracle_mod.Ctx(logN, [int(q) for q in g.moduli], L1, K, 1)
        rng = np.random.default_rng(5)
        m = rng.integers(-(1 << 62), 1 << 62, (3, o.N))
        m[1] = rng.integers(-3, 4, o.N)
        ends = [-(1 << 63), (1 << 63) - 1, -1, 0, 1, 1 << 32, -(1 << 32), (1 << 31) - 1, -(1 << 31)]
        ends += [s * int(q) + d for q in g.moduli for s in (-1, 1) for d in (-1, 0, 1)]
        m[2, :len(ends)] = ends
        ids = list(range(L1 + K))
        out = g.array((3 * len(ids), o.N))
        g.encode_coeffs(m, ids, out)
        res = np.array([[[int(v) % int(q) for v in row] for q in g.moduli] for row in m], dtype=np.uint64)
        assert np.array_equal(out.download().reshape(res.shape), np.stack([o.ntt(r, ids) for r in res]))
        out.free()
    finally:
        g.close()
