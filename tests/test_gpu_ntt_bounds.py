"""NTT / INTT against the oracle where the lazy integer ranges are fullest: extreme inputs at primes on
both sides of 2^60 and at every ring size, through both passes' arithmetics (fp64, below 2^60, wide)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


# (first, scaling, special prime bits): the fp64 class with 60-bit primes, all primes below 2^60 on the
# integer path, primes above 2^60 (wide integers), primes just above the fp64 bound
@pytest.mark.parametrize("bits", [(60, 50, 60), (60, 59, 60), (61, 61, 61), (52, 51, 53)])
@pytest.mark.parametrize("logN", [10, 11, 12, 13, 14, 15, 16])
def test_extreme_inputs(fh, oracle_mod, logN, bits):
    g = fh.Context(logN, 3, 1, 1, first_bits=bits[0], scale_bits=bits[1], aux_bits=bits[2])
    try:
        o = oracle_mod.Ctx(logN, [int(q) for q in g.moduli], 3, 1, 1)
        pids = [0, 1, 2, 3]
        q = np.array([int(m) for m in g.moduli], dtype=np.uint64)[:, None]
        idx = np.arange(o.N, dtype=np.uint64)[None, :]
        inputs = {
            "all q-1": np.broadcast_to(q - np.uint64(1), (4, o.N)),
            "alternating 0, q-1": (q - np.uint64(1)) * (idx & np.uint64(1)),
            "half q": np.broadcast_to(q >> np.uint64(1), (4, o.N)),
            "last only": (q - np.uint64(1)) * (idx == np.uint64(o.N - 1)).astype(np.uint64),
            "random": o.random_poly(40 + logN, pids),
        }
        for name, x in inputs.items():
            x = np.ascontiguousarray(x, dtype=np.uint64)
            print(f"[ntt bounds] logN={logN} bits={bits} {name}", flush=True)
            d = g.to_device(x)
            g.ntt_forward(d, pids)
            assert np.array_equal(d.download(), o.ntt(x, pids)), name
            d.upload(x)
            g.ntt_inverse(d, pids)
            assert np.array_equal(d.download(), o.intt(x, pids)), name
            d.free()
    finally:
        g.close()
