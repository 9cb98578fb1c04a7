"""Rotations that are summed or multiplied where they are formed, against the oracle: one digit up to
eight, primes below 2^60 and above, folds and flat transforms of more rotations than one launch takes."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _poly(o, seed, ids, n):
    return np.concatenate([o.random_poly(seed + i, ids) for i in range(n)])


# (towers, special primes, digits, levels): the digits of a level run from 1 to 8
@pytest.mark.parametrize("L1,K,dnum,levels", [(4, 4, 1, (0, 3)), (8, 1, 8, (3, 4, 7)), (5, 2, 3, (1, 4))])
@pytest.mark.parametrize("bits", [(60, 50, 60), (61, 61, 61)])
def test_hoisted_sums(fh, oracle_mod, L1, K, dnum, levels, bits):
    logN = 10
    g = fh.Context(logN, L1, K, dnum, first_bits=bits[0], scale_bits=bits[1], aux_bits=bits[2])
    try:
        o = oracle_mod.Ctx(logN, [int(q) for q in g.moduli], L1, K, dnum)
        s = o.gen_secret(3)
        for l in levels:
            ids = list(range(l + 1))
            x = _poly(o, 50 + l, ids, 2)
            d, out = g.to_device(x), g.array(x.shape)
            # 31 and 1 rotations a level
            radix, size = 32, 64
            idx = o.accumulate_indices(radix, 1, size)
            ks = [o.rot_index(r) for r in idx]
            hk = [o.gen_rot_key(s, k, 200 + i) for i, k in enumerate(ks)]
            dk = [g.key(k) for k in hk]
            print(f"[hoisted sums] L1={L1} dnum={dnum} bits={bits} level {l}: folds", flush=True)
            g.accumulate_sum(d, l, radix, 1, size, dk, ks, out)
            assert np.array_equal(out.download(), o.accumulate_sum(x, l, radix, 1, size, hk, ks))
            g.accumulate_sum_from(d, l, radix, 1, size, 1, dk, ks, out)
            assert np.array_equal(out.download(), o.accumulate_sum_from(x, l, radix, 1, size, hk, ks, 1))
            # bStep 1 (no baby rotation), 2 with 19 giant rotations, 9 over two launches with one left over
            ext = ids + [L1 + k for k in range(K)]
            for rows, baby in ((3, 1), (40, 2), (20, 9)):
                print(f"[hoisted sums] level {l}: {rows} diagonals, {baby} baby steps", flush=True)
                diags = _poly(o, 400, ext, rows)
                giant = [o.rot_index(j * baby) for j in range(1, (rows + baby - 1) // baby)]
                bk = [None] + [o.gen_rot_key(s, o.rot_index(i), 300 + i) for i in range(1, baby)]
                bkk = [1] + [o.rot_index(i) for i in range(1, baby)]
                gk = [o.gen_rot_key(s, k, 600 + j) for j, k in enumerate(giant)]
                dd, dbk, dgk = g.to_device(diags), [None] + [g.key(k) for k in bk[1:]], [g.key(k) for k in gk]
                g.linear_transform_flat(d, l, rows, baby, 1, dd, dbk, bkk, out, giant_keys=dgk, giant_galois=giant)
                assert np.array_equal(out.download(), o.linear_transform_flat(x, l, diags, baby, 1, bk, bkk, gk, giant, None, 1, 0)), (rows, baby)
                for a in [dd] + dbk[1:] + dgk:
                    a.free()
            for a in dk + [d, out]:
                a.free()
    finally:
        g.close()
