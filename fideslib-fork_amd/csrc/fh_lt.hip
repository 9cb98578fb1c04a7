// Hoisted BSGS linear transform (plaintext-diagonal matrix-vector product) in the
// extended-basis formulation of the reference: baby-step rotations share one ModUp and
// stay in Q_l ∪ P, one multiply-accumulate kernel forms every giant-step partial sum, and
// the giant steps are folded by Horner's rule with only c1 brought back to Q_l before each
// giant rotation (the extended c0 enters the key-switch product directly).
// Reference: src/CKKS/LinearTransform.cu:65-254 (FUSED branch, ONLY_C1), MAC kernel
// dotProductLtBatchedPt2___ (src/CKKS/ElemenwiseBatchKernels.cu:785-835) via
// LTdotProductPtBatch (src/CKKS/LimbPartitionBatch.cu:266-524), Ciphertext::extend
// (src/CKKS/Ciphertext.cpp:1087-1100), contract api/CryptoContext.hpp:460-517.
#include <algorithm>
#include <type_traits>

#include "fh_keyswitch.hpp"

namespace fh {

namespace {

constexpr int kT = 256;
constexpr int kMaxBaby = 16;

// One group of rotations whose results are consumed where they are formed. Source t holds its
// switched polynomial (EVAL, lq limbs) at own + t * own_stride, the other limbs of its digits at
// dig + t * dig_stride ([beta][ext][N]) and its c0 at c0 + t * c0_stride.
struct Hoist {
  uint32_t N, lq, ext, L1, E, beta, alpha, logN;   // E = L1 + K limbs of a key polynomial
  const PrimeConst* prime;
  const uint64_t* pmod;
  const uint64_t* pmod_sh;
  const uint64_t* dig;
  const uint64_t* own;
  const uint64_t* c0;
  uint64_t dig_stride, own_stride, c0_stride;
  int c0_ext;                     // 1: c0 is given over Q_l ∪ P; 0: over Q_l, folded as P c0
  const uint64_t* key[kMaxBaby];  // [dnum][2][E][N], Montgomery form; null: no rotation (P c0, P c1)
  uint32_t gal[kMaxBaby];
};

// The limb a workgroup works on
struct HoistLimb {
  uint32_t pos, p, own_d;
  uint64_t pm, pmsh;
  PrimeConst P;
  __device__ __forceinline__ HoistLimb(const Hoist& h, uint32_t pos_) : pos(pos_) {
    const bool isq = pos < h.lq;
    p = isq ? pos : h.L1 + (pos - h.lq);
    own_d = isq ? pos / h.alpha : ~0u;
    pm = isq ? h.pmod[pos] : 0;
    pmsh = isq ? h.pmod_sh[pos] : 0;
    P = h.prime[p];
  }
};

// Word n of both components of source t rotated by (key, gal), over Q_l ∪ P: the key inner product
// and c0 at the word that the automorphism brings to n. In the bit-reversed order of the transforms
// an automorphism takes every aligned block of 2^k words to an aligned block, so the 64 words that
// a wave gathers fill whole cache lines. Every load is issued before the first product.
// DM bounds the digits. Memory-bound: the keys are read once; writing the rotations and reading them
// back was a third of the traffic. N = 2^16, 50-bit primes, three digits, against key product, sum
// and extension in launches of their own: the radix-4 fold of 256 slots 1325 -> 1022 us, 63 diagonals
// in 16 baby steps 1495 -> 1270 us.
template <class M, int DM>
__device__ __forceinline__ void hoist_rot(const Hoist& h, const HoistLimb& L, const uint64_t* key, uint32_t gal, uint32_t t, uint32_t n,
                                          uint64_t& r0, uint64_t& r1) {
  const size_t N = h.N;
  const uint32_t s = gal != 1 ? auto_src(n, gal, h.logN) : n;
  const uint64_t* dg = h.dig + t * h.dig_stride + L.pos * N;
  const uint64_t* ow = h.own + t * h.own_stride + L.pos * N;
  const uint64_t* kp = key + L.p * N;
  uint64_t x[DM], kb[DM], ka[DM], c = 0;
#pragma unroll
  for (int d = 0; d < DM; ++d) {
    x[d] = kb[d] = ka[d] = 0;
    if (d < (int)h.beta) {
      x[d] = (d == (int)L.own_d ? ow : dg + (size_t)d * h.ext * N)[s];
      kb[d] = kp[(size_t)(2 * d) * h.E * N + s];
      ka[d] = kp[(size_t)(2 * d + 1) * h.E * N + s];
    }
  }
  if (h.c0_ext || L.pos < h.lq) c = h.c0[t * h.c0_stride + L.pos * N + s];
  M a0, a1;
  a0.zero();
  a1.zero();
#pragma unroll
  for (int d = 0; d < DM; ++d)
    if (d < (int)h.beta) {
      const auto xd = M::prep(x[d]);
      a0.mac(xd, M::prep(kb[d]));
      a1.mac(xd, M::prep(ka[d]));
    }
  uint64_t hi, lo;
  a0.get(hi, lo);
  r0 = redc(hi, lo, L.P);  // keys are in Montgomery form
  a1.get(hi, lo);
  r1 = redc(hi, lo, L.P);
  r0 = add_mod(r0, h.c0_ext ? c : shoup(c, L.pm, L.pmsh, L.P.q), L.P.q);
}

// The same for a rotation by nothing: P times source t, zero on the special limbs.
__device__ __forceinline__ void hoist_ident(const Hoist& h, const HoistLimb& L, uint32_t t, uint32_t n, uint64_t& r0, uint64_t& r1) {
  r0 = r1 = 0;
  if (L.pos < h.lq) {
    r0 = shoup(h.c0[t * h.c0_stride + (size_t)L.pos * h.N + n], L.pm, L.pmsh, L.P.q);
    r1 = shoup(h.own[t * h.own_stride + (size_t)L.pos * h.N + n], L.pm, L.pmsh, L.P.q);
  }
}

struct MacParams {
  uint32_t rowSize, bStep, gStep;
  uint32_t i0 = 0;   // first baby step of this launch (a launch covers baby steps i0 .. i0 + BB - 1)
  uint32_t acc = 0;  // 1: add into R (a later launch over the next baby steps)
};

// R[j][comp][pos] = sum_{i: bStep j + i < rowSize} rot_i[comp][pos] (.) diag[bStep j + i][pos]
// One lane forms the bStep rotated words of both components for its (position, coefficient)
// and streams the diagonals once; each sum (at most 16 products) is accumulated exactly under the
// multiply policy M and reduced once. The rotations never reach memory.
// Up to four digits four waves a SIMD are asked for: left alone the compiler takes 133 registers for
// eight baby steps, which is three waves (28 bytes spilled; 63 diagonals in 16 baby steps 1319 -> 1270
// us). With more digits that would spill 156 bytes, and the compiler's own choice is the faster one: 32
// diagonals in 16 baby steps, N = 2^16, 24 limbs, six digits 1094 us (four waves: 1445), eight digits 1230
// (1685).
template <int BB, class M, int DM>
__global__ __launch_bounds__(kT, DM <= 4 ? 4 : 1) void k_lt_mac(Hoist h, const uint64_t* __restrict__ diags, uint64_t* __restrict__ R, MacParams mp) {
  using Op = typename M::Op;
  const HoistLimb L(h, blockIdx.y);
  const size_t N = h.N, E = (size_t)h.ext * N;
  for (uint32_t n = blockIdx.x * blockDim.x + threadIdx.x; n < h.N; n += gridDim.x * blockDim.x) {
    Op f0[BB], f1[BB];
#pragma unroll
    for (int i = 0; i < BB; ++i) {
      if (mp.i0 + i < mp.bStep) {
        uint64_t r0, r1;
        if (h.key[i]) hoist_rot<M, DM>(h, L, h.key[i], h.gal[i], 0, n, r0, r1);
        else hoist_ident(h, L, 0, n, r0, r1);
        f0[i] = M::prep(r0);
        f1[i] = M::prep(r1);
      }
    }
    for (uint32_t j = 0; j < mp.gStep; ++j) {
      M a0, a1;
      a0.zero();
      a1.zero();
#pragma unroll
      for (int i = 0; i < BB; ++i) {
        const uint32_t k = j * mp.bStep + mp.i0 + i;
        if (mp.i0 + i < mp.bStep && k < mp.rowSize) {
          const Op d = M::prep(diags[(size_t)k * E + (size_t)L.pos * N + n]);
          a0.mac(f0[i], d);
          a1.mac(f1[i], d);
        }
      }
      uint64_t hi, lo;
      uint64_t* r0 = R + ((size_t)j * 2 + 0) * E + (size_t)L.pos * N + n;
      uint64_t* r1 = R + ((size_t)j * 2 + 1) * E + (size_t)L.pos * N + n;
      a0.get(hi, lo);
      const uint64_t v0 = mod128(hi, lo, L.P);
      a1.get(hi, lo);
      const uint64_t v1 = mod128(hi, lo, L.P);
      *r0 = mp.acc ? add_mod(*r0, v0, L.P.q) : v0;
      *r1 = mp.acc ? add_mod(*r1, v1, L.P.q) : v1;
    }
  }
}

inline dim3 grid_n(uint32_t N, uint32_t y) { return dim3(std::max(1u, std::min((N + kT - 1) / kT, 256u)), y); }

// base + sum of n rotations, over the extended basis of both components, written to out ([2][ext][N]).
// base: 0 P times the source, 1 what out holds, 2 the extended c0 of the source and P times its c1.
// per_item: rotation t reads source t (base 1 only), else all read source 0. blockIdx.y = pos.
template <class M, int DM>
__global__ __launch_bounds__(kT) void k_hoist_sum(Hoist h, int n_rot, int base, int per_item, uint64_t* __restrict__ out) {
  const HoistLimb L(h, blockIdx.y);
  uint64_t* o0 = out + (size_t)L.pos * h.N;
  uint64_t* o1 = o0 + (size_t)h.ext * h.N;
  for (uint32_t n = blockIdx.x * blockDim.x + threadIdx.x; n < h.N; n += gridDim.x * blockDim.x) {
    uint64_t s0 = 0, s1 = 0;
    if (base == 1) {
      s0 = o0[n];
      s1 = o1[n];
    } else {
      if (L.pos < h.lq) s1 = shoup(h.own[(size_t)L.pos * h.N + n], L.pm, L.pmsh, L.P.q);
      if (base == 2 || L.pos < h.lq) s0 = h.c0[(size_t)L.pos * h.N + n];
      if (base == 0) s0 = shoup(s0, L.pm, L.pmsh, L.P.q);
    }
    for (int t = 0; t < n_rot; ++t) {
      uint64_t r0, r1;
      hoist_rot<M, DM>(h, L, as_global(h.key[t]), h.gal[t], per_item ? t : 0, n, r0, r1);
      s0 = add_mod(s0, r0, L.P.q);
      s1 = add_mod(s1, r1, L.P.q);
    }
    o0[n] = s0;
    o1[n] = s1;
  }
}

// The parameters that every rotation of a group shares.
Hoist hoist_group(const Context& c, int l, const uint64_t* dig, uint64_t dig_stride, const uint64_t* own, uint64_t own_stride,
                  const uint64_t* c0, uint64_t c0_stride, bool c0_ext) {
  const uint32_t lq = l + 1, beta = c.num_digits(l);
  return Hoist{c.N, lq, lq + c.K, (uint32_t)c.L1, (uint32_t)(c.L1 + c.K), beta, (uint32_t)c.alpha, (uint32_t)c.logN, c.d_prime, c.d_pmod,
               c.d_pmod_sh, dig, own, c0, dig_stride, own_stride, c0_stride, c0_ext ? 1 : 0, {}, {}};
}

void hoist_check(const Context& c, const Hoist& h, const uint64_t* key, uint32_t gal) {
  if (h.beta > (uint32_t)kMaxDnum) throw Error(-3, "dnum above kernel limit");
  if (!key) throw Error(-1, "null key");
  if ((gal & 1) == 0 || gal >= 2 * c.N) throw Error(-1, "galois index must be odd and < 2N");
}

// f(M, DM): the kernel for this context's multiply policy and this level's digits
template <class F>
void with_hoist(const Context& c, uint32_t beta, F f) {
  if (c.split_mac_ok) beta <= 4 ? f(Mac30{}, std::integral_constant<int, 4>{}) : f(Mac30{}, std::integral_constant<int, kMaxDnum>{});
  else beta <= 4 ? f(MacWide{}, std::integral_constant<int, 4>{}) : f(MacWide{}, std::integral_constant<int, kMaxDnum>{});
}

// out = base + the n rotations of the group (base, per_item: as in k_hoist_sum), in launches of at most
// kMaxBaby rotations, the later ones adding to out. out is none of the group's sources.
void hoist_sum(Context& c, Hoist h, int n, const uint64_t* const* keys, const uint32_t* gals, int base, bool per_item, uint64_t* out,
               hipStream_t st) {
  for (int t = 0; t < n; ++t) hoist_check(c, h, keys[t], gals[t]);
  ProfScope ps_(c, "hoist_sum", st);
  for (int t0 = 0; t0 < n; t0 += kMaxBaby, base = 1) {
    const int nt = std::min(n - t0, kMaxBaby);
    for (int t = 0; t < nt; ++t) {
      h.key[t] = keys[t0 + t];
      h.gal[t] = gals[t0 + t];
    }
    with_hoist(c, h.beta, [&](auto m, auto dm) {
      k_hoist_sum<decltype(m), decltype(dm)::value><<<grid_n(c.N, h.ext), kT, 0, st>>>(h, nt, base, per_item ? 1 : 0, out);
    });
    FH_HIP(hipGetLastError());
    if (per_item) {
      h.dig += nt * h.dig_stride;
      h.own += nt * h.own_stride;
      h.c0 += nt * h.c0_stride;
    }
  }
}

// [P]_{q_pos} x for Q limbs, 0 for the special limbs (the P-scaled extended form of ciphertexts over
// Q_l): blockIdx.y = (b, comp, pos)
__global__ __launch_bounds__(kT) void k_extend_p_b(const uint64_t* __restrict__ x, uint64_t x_stride, uint64_t* __restrict__ out,
                                                    uint64_t out_stride, uint32_t N, uint32_t lq, uint32_t ext, const PrimeConst* prime,
                                                    const uint64_t* pmod, const uint64_t* pmod_sh) {
  const uint32_t b = blockIdx.y / (2 * ext), r = blockIdx.y % (2 * ext);
  const uint32_t comp = r / ext, pos = r % ext;
  uint64_t* o = out + b * out_stride + ((size_t)comp * ext + pos) * N;
  if (pos >= lq) {
    for (uint32_t n = blockIdx.x * blockDim.x + threadIdx.x; n < N; n += gridDim.x * blockDim.x) o[n] = 0;
    return;
  }
  const uint64_t q = prime[pos].q, w = pmod[pos], wsh = pmod_sh[pos];
  const uint64_t* xi = x + b * x_stride + ((size_t)comp * lq + pos) * N;
  for (uint32_t n = blockIdx.x * blockDim.x + threadIdx.x; n < N; n += gridDim.x * blockDim.x) o[n] = shoup(xi[n], w, wsh, q);
}

constexpr int kMacTile = 64;   // coefficients per workgroup of the batched MAC
constexpr int kMacLanes = kT / kMacTile;

struct MacBatchParams {
  uint32_t N, lq, ext, L1, rowSize, bStep, gStep, B, nrot;
  const PrimeConst* prime;
  int8_t slot[kMaxBaby];   // baby step i: rotation slot (>= 0) or the P-scaled identity (-1)
};

// Giant-step partial sums for B ciphertexts sharing one diagonal set, from the rotations that
// k_ksk_batch wrote. Forming them here, as k_lt_mac does, was measured slower for a batch: 16
// ciphertexts, N = 2^16, 30 limbs, 8 x 8 steps, 20.5 (two waves a SIMD) and 18.9 ms (four, with spills)
// against 16.7 for the transform. There the key
// product reads its keys once for the whole batch, here once per ciphertext and wave. blockIdx.y = extended
// position, blockIdx.x = a 64-coefficient tile: the tile of every diagonal is staged in LDS once
// (as multiply operands, split into 30-bit halves under Mac30) and applied to all B ciphertexts
// (four ciphertexts in flight per workgroup), so the diagonals are read once per batch.
// R[b][j][comp][pos] = sum_i fast_b[i][comp][pos] (.) diag[bStep j + i][pos], each sum of at most
// 16 products accumulated exactly and reduced once.
template <int BB, class M>
__global__ __launch_bounds__(kT) void k_lt_mac_b(const uint64_t* __restrict__ rot, const uint64_t* __restrict__ ident,
                                                  const uint64_t* __restrict__ diags, uint64_t* __restrict__ R, MacBatchParams mp) {
  using Op = typename M::Op;
  static_assert(sizeof(Op) == 8, "one LDS word per diagonal coefficient");
  extern __shared__ uint64_t sd_raw[];   // rowSize x kMacTile
  Op* sd = reinterpret_cast<Op*>(sd_raw);
  const uint32_t pos = blockIdx.y;
  const PrimeConst P = mp.prime[pos < mp.lq ? pos : mp.L1 + (pos - mp.lq)];
  const size_t N = mp.N, E = (size_t)mp.ext * N;
  const uint32_t lane = threadIdx.x % kMacTile, cl = threadIdx.x / kMacTile;
  const uint32_t n = blockIdx.x * kMacTile + lane;
  for (uint32_t k = cl; k < mp.rowSize; k += kMacLanes) sd[k * kMacTile + lane] = M::prep(diags[k * E + (size_t)pos * N + n]);
  __syncthreads();
  for (uint32_t b = cl; b < mp.B; b += kMacLanes) {
    Op f0[BB], f1[BB];
#pragma unroll
    for (int i = 0; i < BB; ++i) {
      if (i < (int)mp.bStep) {
        const uint64_t* src = mp.slot[i] >= 0 ? rot + ((size_t)b * mp.nrot + mp.slot[i]) * 2 * E : ident + (size_t)b * 2 * E;
        f0[i] = M::prep(src[(size_t)pos * N + n]);
        f1[i] = M::prep(src[E + (size_t)pos * N + n]);
      }
    }
    uint64_t* Rb = R + (size_t)b * mp.gStep * 2 * E;
    for (uint32_t j = 0; j < mp.gStep; ++j) {
      M a0, a1;
      a0.zero();
      a1.zero();
#pragma unroll
      for (int i = 0; i < BB; ++i) {
        const uint32_t k = j * mp.bStep + i;
        if (i < (int)mp.bStep && k < mp.rowSize) {
          const Op d = sd[k * kMacTile + lane];
          a0.mac(f0[i], d);
          a1.mac(f1[i], d);
        }
      }
      uint64_t hi, lo;
      a0.get(hi, lo);
      Rb[((size_t)j * 2 + 0) * E + (size_t)pos * N + n] = mod128(hi, lo, P);
      a1.get(hi, lo);
      Rb[((size_t)j * 2 + 1) * E + (size_t)pos * N + n] = mod128(hi, lo, P);
    }
  }
}

// The keys of the baby steps i0 .. i0 + n - 1 (null for a rotation by nothing). Returns whether one of them rotates.
bool hoist_baby(const Context& c, Hoist& h, int i0, int n, int stride, int slots, const uint64_t* const* baby_keys,
                const uint32_t* baby_gal) {
  bool any = false;
  for (int i = 0; i < n; ++i) {
    h.key[i] = nullptr;
    if (((long long)(i0 + i) * stride) % slots == 0) continue;
    if (!baby_keys[i0 + i]) throw Error(-1, "baby-step key missing");
    hoist_check(c, h, baby_keys[i0 + i], baby_gal[i0 + i]);
    h.key[i] = baby_keys[i0 + i];
    h.gal[i] = baby_gal[i0 + i];
    any = true;
  }
  return any;
}

// Every giant-step partial sum from the baby steps, which share one ModUp: R_j, 2 x (l+1+K) limbs
// each, j < gStep.
DBuf lt_partials(Context& c, const uint64_t* ct, int l, int rowSize, int bStep, int stride, int slots, const uint64_t* diags,
                 const uint64_t* const* baby_keys, const uint32_t* baby_gal, hipStream_t st) {
  const uint32_t lq = l + 1, ext = lq + c.K, beta = c.num_digits(l);
  const size_t E = (size_t)ext * c.N;
  const uint64_t* c1 = ct + (size_t)lq * c.N;
  const int gStep = (rowSize + bStep - 1) / bStep;
  DBuf dig, R(c.pool, (size_t)gStep * 2 * E);
  Hoist h = hoist_group(c, l, nullptr, 0, c1, 0, ct, 0, false);
  if (hoist_baby(c, h, 0, bStep, stride, slots, baby_keys, baby_gal)) {
    dig = DBuf(c.pool, (size_t)beta * E);
    h.dig = dig.p;
    modup_batch(c, c1, l, 1, 0, dig.p, st, false);
  }
  MacParams mp{(uint32_t)rowSize, (uint32_t)bStep, (uint32_t)gStep};
  ProfScope ps_(c, "lt_mac", st);
  const dim3 g = grid_n(c.N, ext);
  with_hoist(c, beta, [&](auto m, auto dm) {
    using M = decltype(m);
    constexpr int DM = decltype(dm)::value;
    if (bStep <= 4) {
      k_lt_mac<4, M, DM><<<g, kT, 0, st>>>(h, diags, R.p, mp);
      return;
    }
    // more than 8 baby steps: launches of 8 each, the later ones adding into R (the sums are
    // exact residues, so the split result is the same word). 16 rotations a lane keep too few waves in
    // flight: 63 diagonals, 16 baby steps, N = 2^16, 30 limbs: 1463 us for the transform against 1319 (1270 with the bound above)
    for (mp.i0 = 0; mp.i0 < (uint32_t)bStep; mp.i0 += 8, mp.acc = 1) {
      hoist_baby(c, h, mp.i0, std::min(8, bStep - (int)mp.i0), stride, slots, baby_keys, baby_gal);
      k_lt_mac<8, M, DM><<<g, kT, 0, st>>>(h, diags, R.p, mp);
    }
  });
  FH_HIP(hipGetLastError());
  return R;
}

// The last step of both forms on the combined extended sum: the offset rotation (ModDown of c1,
// the extended c0 folded directly) and ModDown of both, or the ModDown of both.
void lt_finish(Context& c, uint64_t* acc, int l, int offset, const uint64_t* off_key, uint32_t off_gal, uint64_t* out, hipStream_t st) {
  const uint32_t lq = l + 1, ext = lq + c.K, beta = c.num_digits(l);
  const size_t N = c.N, E = (size_t)ext * N;
  if (offset != 0) {
    DBuf c1q(c.pool, (size_t)lq * N), dig(c.pool, (size_t)beta * E), t(c.pool, 2 * E);
    moddown(c, acc + E, l, c1q.p, 1, 0, 0, st);
    modup_batch(c, c1q.p, l, 1, 0, dig.p, st, false);
    ksk_inner(c, dig.p, l, off_key, t.p, t.p + E, acc, off_gal, st, true, c1q.p);
    moddown(c, t.p, l, out, 2, 0, 0, st);
  } else {
    moddown(c, acc, l, out, 2, 0, 0, st);
  }
}

}  // namespace

void linear_transform(Context& c, const uint64_t* ct, int l, int rowSize, int bStep, int stride, int offset, int slots,
                      const uint64_t* diags, const uint64_t* const* baby_keys, const uint32_t* baby_gal, const uint64_t* giant_key,
                      uint32_t giant_gal, const uint64_t* off_key, uint32_t off_gal, uint64_t* out, hipStream_t st) {
  if (bStep < 1 || bStep > kMaxBaby) throw Error(-1, "bStep must be in [1, 16]");
  if (rowSize < 1) throw Error(-1, "rowSize must be >= 1");
  if (slots < 1 || slots > (int)c.N / 2) throw Error(-1, "slots out of range");
  const uint32_t lq = l + 1, ext = lq + c.K, beta = c.num_digits(l);
  const size_t N = c.N, E = (size_t)ext * N;
  const int gStep = (rowSize + bStep - 1) / bStep;
  const bool giant = ((long long)bStep * stride) % slots != 0;
  if (gStep > 1 && giant && !giant_key) throw Error(-1, "giant-step key required");
  if (offset != 0 && !off_key) throw Error(-1, "offset key required");
  DBuf R = lt_partials(c, ct, l, rowSize, bStep, stride, slots, diags, baby_keys, baby_gal, st);

  // ---- Horner over the giant steps ----
  std::vector<int> epids(ext);
  for (uint32_t p = 0; p < ext; ++p) epids[p] = c.ext_prime(l, p);
  // R_{j-1} += rot_giant(R_j) for j = gStep-1 .. 1: the key switch adds its result into R_{j-1}.
  DBuf c1q(c.pool, (size_t)lq * N), dig(c.pool, (size_t)beta * E);
  for (int j = gStep - 1; j > 0; --j) {
    uint64_t* Rj = R.p + (size_t)j * 2 * E;
    uint64_t* Rp = Rj - 2 * E;
    if (giant) {
      moddown(c, Rj + E, l, c1q.p, 1, 0, 0, st);
      modup_batch(c, c1q.p, l, 1, 0, dig.p, st, false);
      ksk_inner(c, dig.p, l, giant_key, Rp, Rp + E, Rj, giant_gal, st, true, c1q.p, true);
    } else {
      LimbSet a = make_set(Rp, ext, epids.data(), 2, E), b = make_set(Rj, ext, epids.data(), 2, E);
      ew_binary(c, 0, a, b, a, st);
    }
  }
  lt_finish(c, R.p, l, offset, off_key, off_gal, out, st);
}

void linear_transform_flat(Context& c, const uint64_t* ct, int l, int rowSize, int bStep, int stride, int offset, int slots,
                           const uint64_t* diags, const uint64_t* const* baby_keys, const uint32_t* baby_gal,
                           const uint64_t* const* giant_keys, const uint32_t* giant_gal, const uint64_t* off_key, uint32_t off_gal,
                           uint64_t* out, hipStream_t st) {
  if (bStep < 1 || bStep > kMaxBaby) throw Error(-1, "bStep must be in [1, 16]");
  if (rowSize < 1) throw Error(-1, "rowSize must be >= 1");
  if (slots < 1 || slots > (int)c.N / 2) throw Error(-1, "slots out of range");
  const uint32_t lq = l + 1, ext = lq + c.K, beta = c.num_digits(l);
  const size_t N = c.N, E = (size_t)ext * N;
  const int gStep = (rowSize + bStep - 1) / bStep;
  if (offset != 0 && !off_key) throw Error(-1, "offset key required");
  // the partial sums rotated by a nonzero multiple of the giant step, and their keys
  std::vector<int> rot;
  std::vector<const uint64_t*> keys;
  std::vector<uint32_t> gals;
  for (int j = 1; j < gStep; ++j) {
    if (((long long)j * bStep * stride) % slots == 0) continue;
    if (!giant_keys || !giant_keys[j - 1]) throw Error(-1, "giant-step key required");
    rot.push_back(j);
    keys.push_back(giant_keys[j - 1]);
    gals.push_back(giant_gal[j - 1]);
  }
  DBuf R = lt_partials(c, ct, l, rowSize, bStep, stride, slots, diags, baby_keys, baby_gal, st);
  std::vector<int> epids(ext);
  for (uint32_t p = 0; p < ext; ++p) epids[p] = c.ext_prime(l, p);
  const LimbSet acc = make_set(R.p, ext, epids.data(), 2, E);
  if (!rot.empty()) {
    // the rotated partial sums side by side: one ModDown of their c1, one ModUp, and one launch that
    // adds every item's key inner product (the extended c0 folded directly, as a Horner step does)
    const int nr = (int)rot.size();
    bool contiguous = true;
    for (int t = 1; t < nr; ++t) contiguous &= rot[t] == rot[0] + t;
    DBuf gathered, c1q(c.pool, (size_t)nr * lq * N), dig(c.pool, (size_t)nr * beta * E);
    const uint64_t* src = R.p + (size_t)rot[0] * 2 * E;
    if (!contiguous) {
      gathered = DBuf(c.pool, (size_t)nr * 2 * E);
      for (int t = 0; t < nr; ++t)
        FH_HIP(hipMemcpyAsync(gathered.p + (size_t)t * 2 * E, R.p + (size_t)rot[t] * 2 * E, 2 * E * 8, hipMemcpyDeviceToDevice, st));
      src = gathered.p;
    }
    moddown(c, src + E, l, c1q.p, nr, 2 * E, (uint64_t)lq * N, st);
    modup_batch(c, c1q.p, l, nr, (uint64_t)lq * N, dig.p, st, false);
    hoist_sum(c, hoist_group(c, l, dig.p, (uint64_t)beta * E, c1q.p, (uint64_t)lq * N, src, 2 * E, true), nr, keys.data(), gals.data(), 1,
              true, R.p, st);
  }
  for (int j = 1; j < gStep; ++j)
    if (((long long)j * bStep * stride) % slots == 0) ew_binary(c, 0, acc, make_set(R.p + (size_t)j * 2 * E, ext, epids.data(), 2, E), acc, st);
  lt_finish(c, R.p, l, offset, off_key, off_gal, out, st);
}

// The same transform for count ciphertexts sharing the diagonal set and keys: the baby-step
// rotations of all ciphertexts form one key-switch batch (each baby key read once for all of
// them), one multiply-accumulate launch reads the diagonals once for the whole batch, and every
// giant step key-switches all ciphertexts with one read of the giant key. Results are bit-identical
// to count calls of linear_transform.
void linear_transform_batch(Context& c, int count, const uint64_t* cts, uint64_t ct_stride, int l, int rowSize, int bStep, int stride,
                            int offset, int slots, const uint64_t* diags, const uint64_t* const* baby_keys, const uint32_t* baby_gal,
                            const uint64_t* giant_key, uint32_t giant_gal, const uint64_t* off_key, uint32_t off_gal, uint64_t* out,
                            hipStream_t st) {
  if (count < 1) return;
  if (bStep < 1 || bStep > kMaxBaby) throw Error(-1, "bStep must be in [1, 16]");
  if (rowSize < 1) throw Error(-1, "rowSize must be >= 1");
  if ((size_t)rowSize * kMacTile * 8 > 64 * 1024) throw Error(-3, "batched linear transform takes at most 128 diagonals");
  if (slots < 1 || slots > (int)c.N / 2) throw Error(-1, "slots out of range");
  const uint32_t lq = l + 1, ext = lq + c.K, beta = c.num_digits(l);
  const size_t N = c.N, E = (size_t)ext * N;
  if (!ct_stride) ct_stride = 2ull * lq * N;
  const int gStep = (rowSize + bStep - 1) / bStep;
  const bool giant = ((long long)bStep * stride) % slots != 0;
  if (gStep > 1 && giant && !giant_key) throw Error(-1, "giant-step key required");
  if (offset != 0 && !off_key) throw Error(-1, "offset key required");
  const uint32_t B = (uint32_t)count;

  // ---- baby steps ----
  MacBatchParams mp{c.N, lq, ext, (uint32_t)c.L1, (uint32_t)rowSize, (uint32_t)bStep, (uint32_t)gStep, B, 0, c.d_prime, {}};
  std::vector<int> rot_idx;
  bool has_ident = false;
  for (int i = 0; i < bStep; ++i) {
    if (((long long)i * stride) % slots == 0) {
      mp.slot[i] = -1;
      has_ident = true;
    } else {
      if (!baby_keys[i]) throw Error(-1, "baby-step key missing");
      mp.slot[i] = (int8_t)rot_idx.size();
      rot_idx.push_back(i);
    }
  }
  const uint32_t nrot = (uint32_t)rot_idx.size();
  mp.nrot = nrot;
  DBuf ident, rot, dig(c.pool, (size_t)B * beta * E);
  if (has_ident) {
    ident = DBuf(c.pool, (size_t)B * 2 * E);
    ProfScope ps_(c, "lt_extend", st);
    k_extend_p_b<<<grid_n(c.N, B * 2 * ext), kT, 0, st>>>(cts, ct_stride, ident.p, 2 * E, c.N, lq, ext, c.d_prime, c.d_pmod, c.d_pmod_sh);
    FH_HIP(hipGetLastError());
  }
  if (nrot) {
    rot = DBuf(c.pool, (size_t)B * nrot * 2 * E);
    modup_batch(c, cts + (size_t)lq * N, l, (int)B, ct_stride, dig.p, st, false);
    std::vector<const uint64_t*> ks((size_t)B * nrot);
    std::vector<uint32_t> gs((size_t)B * nrot);
    for (uint32_t b = 0; b < B; ++b)
      for (uint32_t r = 0; r < nrot; ++r) {
        ks[(size_t)b * nrot + r] = baby_keys[rot_idx[r]];
        gs[(size_t)b * nrot + r] = baby_gal[rot_idx[r]];
      }
    ksk_items(c, (int)(B * nrot), (int)nrot, dig.p, (uint64_t)beta * E, cts, ct_stride, true, false, l, ks.data(), gs.data(), rot.p, 2 * E,
              st, cts + (size_t)lq * N, ct_stride);
  }

  // ---- giant-step partial sums: diagonals read once for the batch ----
  DBuf R(c.pool, (size_t)B * gStep * 2 * E);
  {
    ProfScope ps_(c, "lt_mac", st);
    const dim3 g(c.N / kMacTile, ext);
    const size_t lds = (size_t)rowSize * kMacTile * 8;
    // 30-bit split products when every prime is below 2^60 (sums of at most bStep <= 16 terms)
    if (c.split_mac_ok) {
      if (bStep <= 4) k_lt_mac_b<4, Mac30><<<g, kT, lds, st>>>(rot.p, ident.p, diags, R.p, mp);
      else if (bStep <= 8) k_lt_mac_b<8, Mac30><<<g, kT, lds, st>>>(rot.p, ident.p, diags, R.p, mp);
      else k_lt_mac_b<16, Mac30><<<g, kT, lds, st>>>(rot.p, ident.p, diags, R.p, mp);
    } else {
      if (bStep <= 4) k_lt_mac_b<4, MacWide><<<g, kT, lds, st>>>(rot.p, ident.p, diags, R.p, mp);
      else if (bStep <= 8) k_lt_mac_b<8, MacWide><<<g, kT, lds, st>>>(rot.p, ident.p, diags, R.p, mp);
      else k_lt_mac_b<16, MacWide><<<g, kT, lds, st>>>(rot.p, ident.p, diags, R.p, mp);
    }
    FH_HIP(hipGetLastError());
  }

  // ---- Horner over the giant steps, all ciphertexts together ----
  std::vector<int> epids(ext);
  for (uint32_t p = 0; p < ext; ++p) epids[p] = c.ext_prime(l, p);
  const uint64_t rstride = (uint64_t)gStep * 2 * E;  // between ciphertexts in R
  DBuf c1q(c.pool, (size_t)B * lq * N);
  std::vector<const uint64_t*> gk(B, giant_key), okv(B, off_key);
  std::vector<uint32_t> gg(B, giant_gal), og(B, off_gal);
  for (int j = gStep - 1; j >= 0; --j) {
    uint64_t* Rj = R.p + (size_t)j * 2 * E;
    if (j > 0) {
      uint64_t* Rp = Rj - 2 * E;  // every ciphertext's R_{j-1} += rot_giant(R_j)
      if (giant) {
        moddown(c, Rj + E, l, c1q.p, (int)B, rstride, (uint64_t)lq * N, st);
        modup_batch(c, c1q.p, l, (int)B, (uint64_t)lq * N, dig.p, st, false);
        ksk_items(c, (int)B, 1, dig.p, (uint64_t)beta * E, Rj, rstride, true, true, l, gk.data(), gg.data(), Rp, rstride, st,
                  c1q.p, (uint64_t)lq * N, true);
      } else {
        for (int comp = 0; comp < 2; ++comp) {
          LimbSet a = make_set(Rp + comp * E, ext, epids.data(), B, rstride), b = make_set(Rj + comp * E, ext, epids.data(), B, rstride);
          ew_binary(c, 0, a, b, a, st);
        }
      }
    } else if (offset != 0) {
      moddown(c, Rj + E, l, c1q.p, (int)B, rstride, (uint64_t)lq * N, st);
      modup_batch(c, c1q.p, l, (int)B, (uint64_t)lq * N, dig.p, st, false);
      DBuf t(c.pool, (size_t)B * 2 * E);
      ksk_items(c, (int)B, 1, dig.p, (uint64_t)beta * E, Rj, rstride, true, true, l, okv.data(), og.data(), t.p, 2 * E, st, c1q.p,
                (uint64_t)lq * N);
      moddown(c, t.p, l, out, (int)(2 * B), E, (uint64_t)lq * N, st);
    } else {
      moddown(c, Rj, l, out, (int)B, rstride, 2ull * lq * N, st);
      moddown(c, Rj + E, l, out + (size_t)lq * N, (int)B, rstride, 2ull * lq * N, st);
    }
  }
}

// Rotation-fold sum from a start factor (the cascade: CKKS::Accumulate(ct, bStep, stride, size,
// startFactor), src/CKKS/AccumulateBroadcast.cu:42-84): per fold level s = start, start*radix, ...
// < size, the rotations by i*stride*s (0 < i < radix, i*s < size) share one ModUp and stay in the
// extended basis with P*c0 folded in, are added to P*ct, and both components take a ModDown at
// every level. keys / galois: one per rotation in fold order.
void accumulate_cascade(Context& c, const uint64_t* ct, int l, int radix, int size, int start, const uint64_t* const* keys,
                    const uint32_t* galois, uint64_t* out, hipStream_t st) {
  const uint32_t N = c.N, lq = l + 1, ext = lq + c.K;
  const size_t E = (size_t)ext * N, Q = (size_t)lq * N;
  if (out != ct) FH_HIP(hipMemcpyAsync(out, ct, 2 * Q * 8, hipMemcpyDeviceToDevice, st));
  if (start <= 0 || size <= 0 || start >= size) return;
  DBuf sum(c.pool, 2 * E), dig(c.pool, (size_t)c.num_digits(l) * E);
  int used = 0;
  for (long long s = start; s < size; s *= radix) {
    int n = 0;
    while (n + 1 < radix && (long long)(n + 1) * s < size) ++n;
    modup_batch(c, out + Q, l, 1, 0, dig.p, st, false);
    hoist_sum(c, hoist_group(c, l, dig.p, 0, out + Q, 0, out, 0, false), n, keys + used, galois + used, 0, false, sum.p, st);
    moddown(c, sum.p, l, out, 2, 0, 0, st);
    used += n;
  }
}

// The lazy rotation-fold sum (CKKS::Accumulate(ct, bStep, stride, size),
// src/CKKS/AccumulateBroadcast.cu:122-160). Per fold level s = 1, radix, ... < size: one ModUp of c1
// shared by the level's rotations (by i*stride*s, 0 < i < radix, i*s < size), each kept in Q_l ∪ P;
// c0 is folded as P*c0 on the first level and afterwards stays in Q_l ∪ P, where it is added on
// every limb before the automorphism (the c0_modup branch of hoistedRotateDotKSK_2_,
// src/CKKS/ElemenwiseBatchKernels.cu:302-307). The rotations are summed into (c0, P*c1); c1 takes a
// ModDown at the end of each level and c0 one ModDown after the last. The levels' sums alternate
// between two buffers, since a level's rotations gather from the last level's c0.
void accumulate_sum(Context& c, const uint64_t* ct, int l, int radix, int size, const uint64_t* const* keys, const uint32_t* galois,
                    uint64_t* out, hipStream_t st) {
  const uint32_t N = c.N, lq = l + 1, ext = lq + c.K, beta = c.num_digits(l);
  const size_t E = (size_t)ext * N, Q = (size_t)lq * N;
  if (out != ct) FH_HIP(hipMemcpyAsync(out, ct, 2 * Q * 8, hipMemcpyDeviceToDevice, st));
  if (size <= 1 || radix < 2) return;
  DBuf sum(c.pool, 4 * E), dig(c.pool, (size_t)beta * E);
  uint64_t* cur = nullptr;   // the last level's sums: extended c0, extended c1
  uint64_t* next = sum.p;
  int used = 0;
  for (long long s = 1; s < size; s *= radix) {
    int n = 0;
    while (n + 1 < radix && (long long)(n + 1) * s < size) ++n;
    // the level's rotations, all from the level's input (c0 or its extension, and c1)
    modup_batch(c, out + Q, l, 1, 0, dig.p, st, false);
    hoist_sum(c, hoist_group(c, l, dig.p, 0, out + Q, 0, cur ? cur : out, 0, cur != nullptr), n, keys + used, galois + used, cur ? 2 : 0,
              false, next, st);
    moddown(c, next + E, l, out + Q, 1, 0, 0, st);
    cur = next;
    next = cur == sum.p ? sum.p + 2 * E : sum.p;
    used += n;
  }
  moddown(c, cur, l, out, 1, 0, 0, st);
}

}  // namespace fh
