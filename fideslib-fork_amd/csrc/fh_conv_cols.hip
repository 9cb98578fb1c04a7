// Basis conversion fused with the column pass of the targets' forward NTT, on the matrix cores.
//
// ModUp and ModDown convert residues of n sources (n <= 16) to residues of m targets,
// out_j = sum_i y_i f_ij mod p_j with y_i the prescaled sources, and transform every target forward
// (src/CKKS/Conv.cu:27-430, src/NTTfusions.cuh:150-212). Here one launch does the conversion and
// the first half of the transform:
//
//  * The sum is a contraction. y_i = sum_a 2^8a y_ia (bytes), so out_j = sum_(i,a) y_ia [2^8a f_ij]_p,
//    and with each constant in signed base-256 digits, [..]_p = sum_b 2^8b d_(i,a),j,b, the eight sums
//    s_b = sum_(i,a) (y_ia - 128) d_(i,a),j,b are int8 products over 8 n terms, exact in int32: rows
//    (target, b), columns coefficients, v_mfma_i32_16x16x64_i8 (three 16x16x32 where 64 < 8 n <= 96). The
//    value sum_b 2^8b s_b + c_j (c_j: the 128s and 2^14 p, so that it is positive) is below 2^15.1 p:
//    its quotient fits fp32, and one small multiply-subtract leaves it in [0, 2p). About 20 vector
//    instructions per output against 85 for 128-bit sums of 30-bit products with a Montgomery
//    reduction.
//  * Row m = 4 t + r of the two 16-row products of a group of four targets holds digit r (r + 4) of
//    target t, so every lane receives all eight digit sums of one (target, coefficient); the operand
//    columns of a wave are chosen so that its 16 products give each lane 16 rows of one column of one
//    target: the register layout of the column pass, whose stages follow with no exchange in between.
//  * A workgroup holds one tile of columns of every source as matrix operands in registers (24 bytes
//    per lane and 16 coefficients) and runs over the target groups: conversion, four stages, one LDS
//    exchange, the remaining stages, store. The converted coefficients are never written or re-read.
//    One workgroup of 8 waves per CU: the loop is bound by vector instructions and stores, has eight
//    independent butterflies in flight per lane and two barriers per group.
//
// Measured at N=2^16, 9 sources: 64 rotations (4928 ModUp and 3200 ModDown targets) 2.69 ms (1671 and
// 1017 us); two conversions and two column passes took 3.77 ms before the column passes' present 60-bit
// arithmetic. 5.7 GB move instead of 14.2: 1.1 ms at the copy rate. Vector instructions issue in 61% of
// the cycles (113 and 100 per target word, the column stages among them), matrix instructions in 15%.
// Each spilled register or wait for an earlier store in the loop showed (3.3 ms at first). With 13 to 16
// sources 35 registers spill at N=2^16 (11 at 2^14, 9 at 2^15, none below).
//
// Against the separate launches by number of sources (both in one build, N = 2^12 .. 2^16, two digits,
// 50-bit targets): one rotation, and 16 in one batch, are faster by the factors
//   2: 0.86-0.92, 0.88-1.02    5: 1.00-1.09, 1.03-1.09    9: 1.06-1.13, 1.05-1.11    13: 1.12-1.27, 1.16-1.30
//   3: 0.91-0.99, 0.92-1.02    6: 1.02-1.07, 1.04-1.10   12: 1.08-1.27, 1.08-1.19    16: 1.12-1.39, 1.16-1.33
//   4: 0.93-1.01, 0.98-1.05    8: 1.08-1.15, 1.07-1.12
// (59-bit targets, 2 .. 4 sources: 0.93-0.98 and 0.97-1.10, 0.98-1.04 and 0.97-1.06, 1.00-1.07 and 1.04-1.10.)
#include "fh_keyswitch.hpp"
#include "fh_ntt_impl.hpp"

namespace fh {

namespace {

typedef int v4i __attribute__((ext_vector_type(4)));
typedef int v2i __attribute__((ext_vector_type(2)));

constexpr int kCcThreads = 512;

struct ConvItem {
  const uint64_t* src;       // first source limb (coefficient form), limbs N words apart
  uint64_t* out;             // target position 0
  uint32_t lq, nsrc, pid0;   // Q towers of the level, sources, prime of the first source
  const uint64_t *inv, *invsh;
  const int8_t* mat;
  const ConvTarget* tgt;
  const uint8_t* ord;
};

// job y of a launch: ModUp: (polynomial, digit) of equally strided polynomials or of a job table;
// ModDown: a polynomial, likewise
struct ConvJobs {
  uint32_t N, L1, K, alpha, dnum, np, kb;
  int down;
  const uint64_t *inv, *invsh;
  const int8_t* mat;
  const ConvTarget* tgt;
  const uint8_t* ord;
  // strided form
  const uint64_t* src;
  uint64_t* out;
  uint64_t src_stride, out_stride;
  uint32_t beta, l;
  // table form
  const ModUpJob* up_jobs;
  const MdJob* md_jobs;

  __device__ __forceinline__ ConvItem at(uint32_t y) const {
    ConvItem it;
    if (down) {
      if (md_jobs) {
        const MdJob j = md_jobs[y];
        it.src = j.pc;
        it.out = j.conv;
        it.lq = j.lq;
      } else {
        it.src = src + y * src_stride;
        it.out = out + y * out_stride;
        it.lq = l + 1;
      }
      it.nsrc = K;
      it.pid0 = L1;
      it.inv = inv;
      it.invsh = invsh;
      it.mat = mat;
      it.tgt = tgt;
      it.ord = ord + (size_t)(it.lq - 1) * kConvOrd;
      return it;
    }
    uint32_t lv, d;
    if (up_jobs) {
      const ModUpJob j = up_jobs[y];
      it.src = j.coef;
      it.out = j.out;
      lv = j.l;
      d = j.d;
    } else {
      const uint32_t b = y / beta;
      d = y - b * beta;
      lv = l;
      it.src = src + b * src_stride;
      it.out = out + b * out_stride + (size_t)d * (l + 1 + K) * N;
    }
    const uint32_t start = d * alpha, last = min(start + alpha, lv + 1) - 1;
    it.src += (size_t)start * N;
    it.lq = lv + 1;
    it.nsrc = last - start + 1;
    it.pid0 = start;
    const size_t o = (size_t)lv * dnum + d;
    it.inv = inv + o * alpha;
    it.invsh = invsh + o * alpha;
    it.mat = mat + (size_t)last * np * 8 * kb;
    it.tgt = tgt + (size_t)last * np;
    it.ord = ord + o * kConvOrd;
    return it;
  }
};

// constants of one target slot
struct SlotConst {
  uint64_t q, lo;
  double qinv;
  float tq, q32, q32l;    // the constant's quotient, 2^32 / p, and that rounded down
  uint32_t pid;           // bit 31: padding, not written
};

// LDS layout of the exchange: [4 targets][C columns][S rows], skewed so that both access patterns of a
// half-wave (16 lanes of 2 targets) meet 32 distinct 8-byte banks
template <int LS>
struct Exch {
  static constexpr int S = 1 << LS, T = S / 16, C = 128 / T;
  static constexpr int kCol = LS == 8 ? S + S / 16 + 18 : S + 1;
  static constexpr int kSlot = C * kCol + ((16 - C * kCol % 32 + 32) % 32);
  // row r0 + T k and row 16 r0 + k of a column (LS = 8: row e at word e + e / 16)
  __device__ __forceinline__ static int lo(int r0, int k) { return r0 + (LS == 8 ? 17 : T) * k; }
  __device__ __forceinline__ static int hi(int r0, int k) { return (LS == 8 ? 17 : 16) * r0 + k; }
};

// x y + c mod 2^64 with signed 32-bit factors: one instruction, which the compiler builds from three
__device__ __forceinline__ uint64_t mad_i32(int x, int y, uint64_t c) {
  uint64_t r;
  asm("v_mad_i64_i32 %0, vcc, %1, %2, %3" : "=v"(r) : "v"(x), "s"(y), "v"(c) : "vcc");
  return r;
}

// sum of the eight digit sums and the target's constant, reduced to [0, 2p). np = -p mod 2^64.
__device__ __forceinline__ uint64_t digits_value(v4i a, v4i b, uint64_t lo, float tq, float q32, uint64_t np) {
  const int t0 = a.x + a.y * 256, t1 = a.z + a.w * 256, t2 = b.x + b.y * 256, t3 = b.z + b.w * 256;
  const uint64_t u = mad_i32(t1, 65536, mad_i32(t0, 1, lo));
  // |t0 + 2^16 t1| < 2^45.1 < p / 4 is left out of the quotient; with the 0.375 taken off the
  // constant it is the true one or one below
  const uint32_t h = (uint32_t)__builtin_fmaf((float)t3, q32 * 65536.f, __builtin_fmaf((float)t2, q32, tq));
  const uint64_t r = (uint64_t)h * (uint32_t)np + u;
  const uint32_t hi = (uint32_t)(r >> 32) + ((uint32_t)t2 + ((uint32_t)t3 << 16)) + h * (uint32_t)(np >> 32);
  return (uint64_t)hi << 32 | (uint32_t)r;
}

// 8-bit operands of one row or column for lane group g: sources 2g, 2g + 1, and 8 + g (96 bytes) or
// 8 + 2g, 9 + 2g (128 bytes)
template <int KB>
struct Operand {
  v4i a;
};
template <>
struct Operand<96> {
  v2i a0, a1, b;
};
template <>
struct Operand<128> {
  v4i a, b;
};

// Chains of one shape only: a 16x16x64 product accumulating onto a 16x16x32 one (and the reverse) gave
// sums read before they were complete.
template <int KB>
__device__ __forceinline__ v4i dot(const Operand<KB>& x, const Operand<KB>& y) {
  v4i c = {0, 0, 0, 0};
  if constexpr (KB == 96) {
    c = __builtin_amdgcn_mfma_i32_16x16x32_i8(__builtin_bit_cast(long, x.a0), __builtin_bit_cast(long, y.a0), c, 0, 0, 0);
    c = __builtin_amdgcn_mfma_i32_16x16x32_i8(__builtin_bit_cast(long, x.a1), __builtin_bit_cast(long, y.a1), c, 0, 0, 0);
    c = __builtin_amdgcn_mfma_i32_16x16x32_i8(__builtin_bit_cast(long, x.b), __builtin_bit_cast(long, y.b), c, 0, 0, 0);
  } else {
    c = __builtin_amdgcn_mfma_i32_16x16x64_i8(x.a, y.a, c, 0, 0, 0);
    if constexpr (KB == 128) c = __builtin_amdgcn_mfma_i32_16x16x64_i8(x.b, y.b, c, 0, 0, 0);
  }
  return c;
}

// put source s of the lane group (0, 1: the first two, then the rest) into a column's operand
template <int KB, int s>
__device__ __forceinline__ void put_source(Operand<KB>& y, uint64_t v) {
  const int lo = (int)(uint32_t)v, hi = (int)(uint32_t)(v >> 32);
  if constexpr (KB == 96) {
    v2i& d = s == 0 ? y.a0 : s == 1 ? y.a1 : y.b;
    d.x = lo;
    d.y = hi;
  } else if constexpr (s == 0) {
    y.a.x = lo;
    y.a.y = hi;
  } else if constexpr (s == 1) {
    y.a.z = lo;
    y.a.w = hi;
  } else if constexpr (KB == 128 && s == 2) {
    y.b.x = lo;
    y.b.y = hi;
  } else if constexpr (KB == 128) {
    y.b.z = lo;
    y.b.w = hi;
  }
}

template <int KB>
__device__ __forceinline__ Operand<KB> load_rows(const int8_t* row, int g) {
  Operand<KB> o;
  const v4i a = *reinterpret_cast<const v4i*>(row + 16 * g);
  if constexpr (KB == 96) {
    o.a0 = v2i{a.x, a.y};
    o.a1 = v2i{a.z, a.w};
    o.b = *reinterpret_cast<const v2i*>(row + 64 + 8 * g);
  } else {
    o.a = a;
    if constexpr (KB == 128) o.b = *reinterpret_cast<const v4i*>(row + 64 + 16 * g);
  }
  return o;
}

struct ConvGrid {
  uint32_t ntiles, nchunks, swz;
};

template <int LOGN, int LS, int KB>
__global__ __launch_bounds__(kCcThreads) __attribute__((amdgpu_waves_per_eu(2, 2))) void k_conv_cols(ConvJobs jobs, ConvGrid cg, NttTables tb) {
  using X = Exch<LS>;
  constexpr int S = X::S, T = X::T, C = X::C;
  __shared__ uint64_t ex[4 * X::kSlot];
  // twiddle slots an odd number of words apart, matrix rows 16 bytes: the four targets (16 rows) a wave
  // reads at a time start in different banks
  constexpr int kTw = 2 * S + 1, kRow = KB + 16;
  __shared__ uint64_t tws[2][4][kTw];
  __shared__ __align__(16) int8_t mats[2][32 * kRow];
  __shared__ SlotConst sc[kConvSlots];
  uint32_t L = blockIdx.x;
  if (cg.swz) {   // blocks b and b + 8 (one XCD) take neighbouring tiles: their 64-byte row pieces share L2 lines
    const uint32_t j = L >> 3;
    L = ((j >> 1) << 4) | ((L & 7) << 1) | (j & 1);
  }
  const uint32_t tile = L % cg.ntiles, rest = L / cg.ntiles;
  const uint32_t chunk = rest % cg.nchunks, y = rest / cg.nchunks;
  ConvItem it = jobs.at(y);
  it.src = as_global(it.src);
  it.out = as_global(it.out);
  it.inv = as_global(it.inv);
  it.invsh = as_global(it.invsh);
  it.mat = as_global(it.mat);
  it.tgt = as_global(it.tgt);
  it.ord = as_global(it.ord);
  const uint32_t ngroups = it.ord[0], nfp = it.ord[1];
  const uint32_t per = (ngroups + cg.nchunks - 1) / cg.nchunks;
  const uint32_t g0 = chunk * per, g1 = min(g0 + per, ngroups);
  if (g0 >= g1) return;   // the whole workgroup
  const int tid = threadIdx.x, lane = tid & 63, n = lane & 15, kg = lane >> 4;
  const int idx = (tid >> 6) * 16 + n;
  const int col = idx % C, r0 = idx / C;
  constexpr size_t N = (size_t)1 << LOGN, N2 = N >> LS;
  const size_t gcol = (size_t)tile * C + col;

  for (uint32_t i = tid; i < 4 * (g1 - g0); i += kCcThreads) {
    const uint32_t slot = it.ord[4 + 4 * g0 + i], pid = slot & 0x7F;
    const PrimeConst& P = tb.prime[pid];
    const ConvTarget t = it.tgt[pid];
    sc[i] = SlotConst{P.q, t.lo, P.qinv, t.q, (float)(4294967296.0 * P.qinv), P.q32inv, pid | (slot >> 7) << 31};
  }

  __syncthreads();

  // ---- the tile of every source as matrix operands: prescaled, bytes offset by 128 to be signed
  Operand<KB> y8[16];
  constexpr int NS = KB == 64 ? 2 : KB == 96 ? 3 : 4;   // sources per lane group
  uint64_t v0[16], v1[16], v2[NS > 2 ? 16 : 1], v3[NS > 3 ? 16 : 1];
  auto index = [&](int s) { return KB == 96 && s == 2 ? 8 + kg : (s & 1) + 2 * kg + 8 * (s >> 1); };
  auto load = [&](int i, uint64_t* v) {   // beyond the last source: the first one, taken times zero
    const uint64_t* p = it.src + (size_t)(i < (int)it.nsrc ? i : 0) * N + (size_t)r0 * N2 + gcol;
#pragma unroll
    for (int k = 0; k < 16; ++k) v[k] = p[(size_t)(T * k) * N2];
  };
  load(index(0), v0);
  load(index(1), v1);
  if constexpr (NS > 2) load(index(2), v2);
  if constexpr (NS > 3) load(index(3), v3);
  auto convert = [&](int i, const uint64_t* v, auto slot) {
    const bool on = i < (int)it.nsrc;
    i = on ? i : 0;
    const uint64_t w = on ? it.inv[i] : 0, wsh = on ? it.invsh[i] : 0, q = tb.prime[it.pid0 + i].q;
    const uint64_t q2 = 2 * q, nq = 0 - q;
#pragma unroll
    for (int k = 0; k < 16; ++k) {
      put_source<KB, decltype(slot)::value>(y8[k], reduce2(reduce2(shoup_lazy4(v[k], w, wsh, nq), q2), q) ^ 0x8080808080808080ull);
      if (k % 4 == 3) __builtin_amdgcn_sched_barrier(0);
    }
  };
  convert(index(0), v0, std::integral_constant<int, 0>{});
  convert(index(1), v1, std::integral_constant<int, 1>{});
  if constexpr (NS > 2) convert(index(2), v2, std::integral_constant<int, 2>{});
  if constexpr (NS > 3) convert(index(3), v3, std::integral_constant<int, 3>{});

  // ---- a group's tables, fetched into registers while an earlier group is worked on and put into LDS
  // ahead of its own barrier. Thread (slot, j) moves NW words of its slot's twiddles (and companions,
  // which the fp64 groups have none of: their words twice), thread (row, j) one word of a matrix row;
  // row m is digit m % 4 (+ 4 from row 16 on) of target m % 16 / 4. The fetch is issued after the
  // products, by when the stores of the group before (which the wait for it includes) are mostly done.
  // (Indices from an opaque thread number: hoisted out of the loop their addresses would cost registers.)
  constexpr int NW = S == 256 ? 2 : 1;
  uint64_t ta0, ta1 = 0, tb0, tb1 = 0, md = 0;
  auto fetch = [&](uint32_t g) {
    const int t_ = OpaqueTid::get(), ts = t_ >> 7, tj = (t_ & 127) * NW & (S - 1), mrow = t_ >> 4, mj = t_ & 15;
    const SlotConst* gs = sc + 4 * (g - g0);
    const size_t o = (size_t)(gs[ts].pid & 0x7F) * N + tj;
    const bool fp = g < nfp;
    const uint64_t* t = (fp ? reinterpret_cast<const uint64_t*>(tb.twd) : tb.tw) + o;
    const uint64_t* h = (fp ? reinterpret_cast<const uint64_t*>(tb.twd) : tb.tw_sh) + o;
    if constexpr (NW == 2) {
      const ulonglong2 x = *reinterpret_cast<const ulonglong2*>(t), y = *reinterpret_cast<const ulonglong2*>(h);
      ta0 = x.x;
      ta1 = x.y;
      tb0 = y.x;
      tb1 = y.y;
    } else {
      ta0 = *t;
      tb0 = *h;
    }
    if (mj < KB / 8)
      md = reinterpret_cast<const uint64_t*>(it.mat + ((size_t)(gs[(mrow & 15) >> 2].pid & 0x7F) * 8 + (mrow & 3) + (mrow >> 4) * 4) * KB)[mj];
  };
  auto put = [&](uint32_t g) {
    const int t_ = OpaqueTid::get(), ts = t_ >> 7, tj = (t_ & 127) * NW & (S - 1), mrow = t_ >> 4, mj = t_ & 15;
    const int buf = (int)(g - g0) & 1;
    uint64_t* t = tws[buf][ts] + tj;
    t[0] = ta0;
    t[S] = tb0;
    if constexpr (NW == 2) {
      t[1] = ta1;
      t[S + 1] = tb1;
    }
    if (mj < KB / 8) *reinterpret_cast<uint64_t*>(mats[buf] + mrow * kRow + 8 * mj) = md;
  };
  fetch(g0);
  put(g0);
  __syncthreads();

  uint64_t* xt = ex + kg * X::kSlot + col * X::kCol;
  for (uint32_t g = g0; g < g1; ++g) {
    const int buf = (int)(g - g0) & 1;
    const bool more = g + 1 < g1;
    const SlotConst& c = sc[4 * (g - g0) + kg];
    const uint64_t lo = c.lo, np = 0 - c.q;
    const float tq = c.tq, q32 = c.q32;
    const Operand<KB> m0 = load_rows<KB>(mats[buf] + n * kRow, kg), m1 = load_rows<KB>(mats[buf] + (16 + n) * kRow, kg);
    uint64_t v[16];
#pragma unroll
    for (int k = 0; k < 16; ++k) {
      const v4i a = dot<KB>(m0, y8[k]), b = dot<KB>(m1, y8[k]);
      v[k] = digits_value(a, b, lo, tq, q32, np);
      // a few products in flight at a time: all of them ahead of their sums (which the compiler would
      // move down into the branches below) would take 128 registers
      asm volatile("" : "+v"(v[k]));
      if (k % 4 == 3) __builtin_amdgcn_sched_barrier(0);
    }
    if (more) fetch(g + 1);
    const uint32_t pid = c.pid & 0x7F, pos = pid < jobs.L1 ? pid : it.lq + (pid - jobs.L1);
    uint64_t* po = it.out + (size_t)pos * N + (size_t)(16 * r0) * N2 + gcol;
    const bool write = (int)c.pid >= 0;
    auto stages = [&](const auto& ar, auto from, const auto* sw, const auto* swp) {
      typename std::decay_t<decltype(ar)>::T x[16];
      int b[16];
#pragma unroll
      for (int k = 0; k < 16; ++k) {
        x[k] = from(v[k]);
        b[k] = 2;
      }
      fwd_cols_lo<LS>(ar, x, b, sw, swp);
      __syncthreads();   // the previous group's exchange has been read
#pragma unroll
      for (int k = 0; k < 16; ++k) xt[X::lo(r0, k)] = ar.to_mid(x[k]);
      if (more) put(g + 1);
      __syncthreads();
#pragma unroll
      for (int k = 0; k < 16; ++k) x[k] = ar.from_mid(xt[X::hi(r0, k)]);
      fwd_cols_hi<LS>(ar, x, b, sw, swp, r0);
      if (write) {
#pragma unroll
        for (int k = 0; k < 16; ++k) po[(size_t)k * N2] = ar.to_mid(x[k]);
      }
    };
    if (g < nfp) {
      const double q = (double)c.q;
      const FpA ar{q, c.qinv, 0.5 * q};
      const double* sw = reinterpret_cast<const double*>(tws[buf][kg]);
      stages(ar, [&](uint64_t r) { double x = (double)r; ar.recenter(x); return x; }, sw, sw);
    } else {
      const IntL ar{c.q, np, c.q32l};
      stages(ar, [](uint64_t r) { return r; }, (const uint64_t*)tws[buf][kg], (const uint64_t*)tws[buf][kg] + S);
    }
  }
}

// Workgroups: tiles x chunks of the target groups x jobs, one per CU at a time. Chunks of the groups
// (each reads the sources again, about one group's time) are taken where the jobs alone leave CUs
// idle: the number with the fewest group times in sequence.
uint32_t conv_chunks(const Context& c, uint32_t wgs, uint32_t groups) {
  const uint32_t cus = (uint32_t)std::max(1, c.cu_count);
  uint32_t best = 1;
  uint64_t cost = ~0ull;
  for (uint32_t n = 1; n <= groups; ++n) {
    const uint64_t t = (uint64_t)((wgs * n + cus - 1) / cus) * (1 + (groups + n - 1) / n);
    if (t < cost) {
      cost = t;
      best = n;
    }
  }
  return best;
}

template <int LOGN, int LS>
void conv_launch(const Context& c, const ConvJobs& j, uint32_t njobs, uint32_t groups, hipStream_t st) {
  const NttTables tb = ntt_tables(c);
  const uint32_t ntiles = (c.N >> LS) / Exch<LS>::C;
  ConvGrid cg{ntiles, 1, 0};
  cg.nchunks = conv_chunks(c, ntiles * njobs, groups);
  const uint64_t total = (uint64_t)ntiles * njobs * cg.nchunks;
  if (total > 0x7fffffffull) throw Error(-3, "too many conversions in one launch");
  cg.swz = LS == 8 && total % 16 == 0 ? 1u : 0u;
  const dim3 g((uint32_t)total), b(kCcThreads);
  switch (j.kb) {
    case 64: k_conv_cols<LOGN, LS, 64><<<g, b, 0, st>>>(j, cg, tb); break;
    case 96: k_conv_cols<LOGN, LS, 96><<<g, b, 0, st>>>(j, cg, tb); break;
    default: k_conv_cols<LOGN, LS, 128><<<g, b, 0, st>>>(j, cg, tb); break;
  }
  FH_HIP(hipGetLastError());
}

void conv_dispatch(const Context& c, const ConvJobs& j, uint32_t njobs, uint32_t targets, hipStream_t st) {
  if (!njobs) return;
  const uint32_t groups = (targets + 3) / 4;
  switch (c.logN) {   // at the default radix split
    case 12: conv_launch<12, 6>(c, j, njobs, groups, st); break;
    case 13: conv_launch<13, 6>(c, j, njobs, groups, st); break;
    case 14: conv_launch<14, 7>(c, j, njobs, groups, st); break;
    case 15: conv_launch<15, 7>(c, j, njobs, groups, st); break;
    case 16: conv_launch<16, 8>(c, j, njobs, groups, st); break;
    default: throw Error(-1, "fused conversion: unsupported ring dimension");
  }
}

ConvJobs conv_jobs(const Context& c, bool down) {
  ConvJobs j{};
  j.N = c.N;
  j.L1 = c.L1;
  j.K = c.K;
  j.alpha = c.alpha;
  j.dnum = c.dnum;
  j.np = c.np;
  j.kb = down ? c.conv_kb_dn : c.conv_kb_up;
  j.down = down ? 1 : 0;
  j.inv = down ? c.d_md_phinv : c.d_modup_qhinv;
  j.invsh = down ? c.d_md_phinv_sh : c.d_modup_qhinv_sh;
  j.mat = down ? c.d_cv_dn : c.d_cv_up;
  j.tgt = down ? c.d_cv_dn_t : c.d_cv_up_t;
  j.ord = down ? c.d_cv_dn_ord : c.d_cv_up_ord;
  return j;
}

}  // namespace

bool conv_cols_usable(const Context& c, int sources) {
  // Two sources cost the plain conversion four products per output, and a rotation is up to 14% faster
  // with its two launches (N=2^13: 64 us against 75). Five and more gain. At three and four it depends on
  // the launch: a single call loses up to 9% (N=2^13, three sources: 68 us against 74), most batches and
  // all of 59-bit targets gain up to 6%; they run fused. Figures above.
  return sources > 2 && c.conv_cols_ok && !c.reduced_noise && !c.tune.ntt_team && (!c.tune.ntt_split || c.tune.ntt_split == ntt_default_split(c.logN));
}

void conv_cols_modup(const Context& c, const uint64_t* coef, int l, int npolys, uint64_t* digits, hipStream_t st) {
  ConvJobs j = conv_jobs(c, false);
  j.l = (uint32_t)l;
  j.beta = (uint32_t)c.num_digits(l);
  j.src = coef;
  j.src_stride = (uint64_t)(l + 1) * c.N;
  j.out = digits;
  j.out_stride = (uint64_t)j.beta * (l + 1 + c.K) * c.N;
  ProfScope ps_(c, "modup_conv_cols", st);
  conv_dispatch(c, j, (uint32_t)npolys * j.beta, (uint32_t)(l + 1 + c.K), st);
}

void conv_cols_moddown(const Context& c, const uint64_t* pcoef, int l, int npolys, uint64_t* conv, hipStream_t st) {
  ConvJobs j = conv_jobs(c, true);
  j.l = (uint32_t)l;
  j.src = pcoef;
  j.src_stride = (uint64_t)c.K * c.N;
  j.out = conv;
  j.out_stride = (uint64_t)(l + 1) * c.N;
  ProfScope ps_(c, "moddown_conv_cols", st);
  conv_dispatch(c, j, (uint32_t)npolys, (uint32_t)(l + 1), st);
}

void conv_cols_modup_jobs(const Context& c, const ModUpJob* jobs, uint32_t n, hipStream_t st) {
  ConvJobs j = conv_jobs(c, false);
  j.up_jobs = jobs;
  ProfScope ps_(c, "modup_conv_cols", st);
  conv_dispatch(c, j, n, (uint32_t)c.np, st);
}

void conv_cols_moddown_jobs(const Context& c, const MdJob* jobs, uint32_t n, hipStream_t st) {
  ConvJobs j = conv_jobs(c, true);
  j.md_jobs = jobs;
  ProfScope ps_(c, "moddown_conv_cols", st);
  conv_dispatch(c, j, n, (uint32_t)c.L1, st);
}

}  // namespace fh
