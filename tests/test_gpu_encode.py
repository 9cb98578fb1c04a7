"""Device CKKS encoding (fh_encode_slots / fh_encode_coeffs) against the oracle's encoder, bit for
bit: the special inverse FFT in fp64 with the host encoder's rounding sequence, the gap scatter,
the residues and the forward NTT; batched plaintexts; Q and Q-and-P prime sets."""
import ctypes

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _values(n, seed, count=1, mag=1.0):
    rng = np.random.default_rng(seed)
    return mag * (rng.uniform(-1, 1, (count, n)) + 1j * rng.uniform(-1, 1, (count, n)))


@pytest.mark.parametrize("slots,level,scale_bits,count", [(32768, 24, 50, 1), (8, 3, 50, 2), (4096, 12, 40, 3), (1, 0, 50, 1), (2048, 24, 59, 2)])
def test_encode_slots_matches_oracle(slots, level, scale_bits, count, gctx2, octx2):
    g, o = gctx2, octx2
    z = _values(slots, slots + level, count)
    scale = 2.0 ** scale_bits
    pids = list(range(level + 1))
    out = g.array((count * (level + 1), o.N))
    print(f"[encode_slots] slots={slots} level={level} count={count}", flush=True)
    g.encode_slots(z, scale, pids, out)
    got = out.download()
    for b in range(count):
        assert np.array_equal(got[b * (level + 1):(b + 1) * (level + 1)], o.encode(z[b], scale, level)), b
    out.free()


def test_encode_slots_extended_strided(gctx2, octx2):
    """Q_l and P limbs (the LinearTransform diagonal layout), outputs strided in one buffer."""
    g, o = gctx2, octx2
    level, slots, count = 20, 32768, 2
    pids = list(range(level + 1)) + [o.L1 + k for k in range(o.K)]
    ext = len(pids)
    z = _values(slots, 77, count, mag=2.0)
    stride = (ext + 1) * o.N
    out = g.array((count * (ext + 1), o.N))
    g.encode_slots(z, 2.0 ** 50, pids, out, out_stride=stride)
    got = out.download()
    for b in range(count):
        assert np.array_equal(got[b * (ext + 1):b * (ext + 1) + ext], o.encode_ext(z[b], 2.0 ** 50, level)), b
    out.free()


def test_encode_coeffs_matches_oracle(gctx2, octx2):
    g, o = gctx2, octx2
    rng = np.random.default_rng(5)
    count, pids = 2, [0, 3, 24, o.L1, o.L1 + 8]
    m = rng.integers(-(2 ** 62), 2 ** 62, (count, o.N), dtype=np.int64)
    m[0, :4] = [0, -1, 2 ** 62 - 1, -(2 ** 62)]
    out = g.array((count * len(pids), o.N))
    g.encode_coeffs(m, pids, out)
    got = out.download()
    for b in range(count):
        res = np.stack([np.array([int(v) % int(o.primes[p]) for v in m[b]], dtype=np.uint64) for p in pids])
        assert np.array_equal(got[b * len(pids):(b + 1) * len(pids)], o.ntt(res, pids)), b
    out.free()


def test_encode_rejects_bad_input(gctx1, fh):
    g = gctx1
    out = g.array((2, g.N))
    with pytest.raises(fh.FHError):
        g.encode_slots(np.ones(6), 2.0 ** 40, [0, 1], out)             # slots not a power of two
    with pytest.raises(fh.FHError):
        g.encode_slots(np.full(4, 4.0), 2.0 ** 62, [0, 1], out)         # |value| * scale beyond 2^63
    with pytest.raises(fh.FHError, match="2\\^61"):
        g.encode_slots(np.array([8.0, 0.0]), 2.0 ** 58, [0, 1], out)    # coefficient 2^61: OpenFHE's approximate path
    with pytest.raises(fh.FHError):
        g.encode_slots(np.array([np.nan, 1.0]), 2.0 ** 40, [0, 1], out)
    out.free()


def test_encode_at_the_2_61_boundary(gctx2, octx2):
    """Coefficients just below 2^61 (OpenFHE's MAX_BITS_IN_WORD) still encode exactly, bit for bit
    with the oracle; 2^61 itself is rejected by both encoders."""
    g, o = gctx2, octx2
    pids = [0, 1, 2]
    z = np.array([5.0 - 2.999j])                                        # one slot: coefficients z * 2^58
    out = g.array((3, o.N))
    g.encode_slots(z, 2.0 ** 58, pids, out)
    assert np.array_equal(out.download(), o.encode(z, 2.0 ** 58, 2))
    with pytest.raises(ValueError):
        o.encode(np.array([8.0 + 0j]), 2.0 ** 58, 2)
    out.free()


@pytest.mark.parametrize("form", ["slots", "coeffs"])
def test_input_is_read_when_the_call_returns(form, gctx2, fh):
    """The caller's array is the caller's again on return, page-locked memory (which a copy engine reads
    after the call is queued) included: here the upload is queued behind transforms on the stream."""
    g = gctx2
    pids, count = [0, 1, g.L1], 20          # more than one chunk of slot values
    if form == "slots":
        src = _values(g.N // 2, 12, count)
        encode = lambda v, out: g.encode_slots(v, 2.0 ** 50, pids, out)
    else:
        src = np.random.default_rng(11).integers(-(1 << 50), 1 << 50, (count, g.N), dtype=np.int64)
        encode = lambda v, out: g.encode_coeffs(v, pids, out)
    hip, p = fh.load(), ctypes.c_void_p()   # the runtime's symbols are found through the library's dependencies
    assert hip.hipHostMalloc(ctypes.byref(p), ctypes.c_size_t(src.nbytes), ctypes.c_uint(0)) == 0
    pinned = np.frombuffer((ctypes.c_char * src.nbytes).from_address(p.value), dtype=src.dtype).reshape(src.shape)
    ids = list(range(g.L1 + g.K))
    ref, got, busy = g.array((count * len(pids), g.N)), g.array((count * len(pids), g.N)), g.array((32 * len(ids), g.N))
    g.fill_uniform(busy, ids, num_polys=32)
    encode(src, ref)
    g.sync()
    for _ in range(2):
        pinned[...] = src
        for _ in range(8):
            g.ntt_forward(busy, ids, num_polys=32)
        encode(pinned, got)
        pinned[...] = 0
        assert np.array_equal(got.download(), ref.download())
    for a in (ref, got, busy):
        a.free()
    assert hip.hipHostFree(p) == 0


def test_encode_scratch(fh, oracle_mod):
    """Full-slot values take two buffers of N words a plaintext: the values, where their coefficients follow,
    and the transform's."""
    logN, count = 13, 512
    g = fh.Context(logN, 1, 1, 1)

    def free():
        a, b = ctypes.c_size_t(), ctypes.c_size_t()
        assert fh.load().hipMemGetInfo(ctypes.byref(a), ctypes.byref(b)) == 0
        return a.value

    try:
        o = oracle_mod.Ctx(logN, [int(q) for q in g.moduli], 1, 1, 1)
        z = _values(g.N // 2, 3, count)
        out = g.array((count, g.N))
        g.encode_slots(z[:1], 2.0 ** 40, [0], out)      # tables and code of the encoder
        g.sync()
        before = free()
        g.encode_slots(z, 2.0 ** 40, [0], out)
        got = out.download()
        assert before - free() <= 2 * 8 * g.N * count + (4 << 20)
        for b in (0, 63, 64, count - 1):
            assert np.array_equal(got[b:b + 1], o.encode(z[b], 2.0 ** 40, 0)), b
    finally:
        g.close()
