// NTT / INTT entry points over limb sets (in place and out of place, with the ModDown
// epilogue), and the NTT launch-shape autotuner. The kernels are in fh_ntt_impl.hpp.
#include "fh_keyswitch.hpp"
#include "fh_ntt_impl.hpp"
#include "fh_ops.hpp"

namespace fh {

void ntt_load() { load_unit(); }

void ntt_fwd(const Context& c, const LimbSet& s, hipStream_t st) { dispatch_fwd(c, SetAddr{s}, SetAddr{s}, s.nlimbs * s.npolys, st); }
void ntt_inv(const Context& c, const LimbSet& s, hipStream_t st) { dispatch_inv(c, SetAddr{s}, SetAddr{s}, s.nlimbs * s.npolys, st); }
void ntt_fwd(const Context& c, const LimbSet& in, const LimbSet& out, hipStream_t st) {
  if (in.nlimbs * in.npolys != out.nlimbs * out.npolys) throw Error(-1, "NTT in/out shapes differ");
  dispatch_fwd(c, SetAddr{in}, SetAddr{out}, in.nlimbs * in.npolys, st);
}
void ntt_inv(const Context& c, const LimbSet& in, const LimbSet& out, hipStream_t st) {
  if (in.nlimbs * in.npolys != out.nlimbs * out.npolys) throw Error(-1, "NTT in/out shapes differ");
  dispatch_inv(c, SetAddr{in}, SetAddr{out}, in.nlimbs * in.npolys, st);
}
void ntt_fwd_moddown(const Context& c, const LimbSet& conv, const uint64_t* x, uint64_t x_stride, uint64_t* out, uint64_t out_stride,
                     hipStream_t st, bool cols, const uint64_t* add, uint64_t add_pair) {
  EpiModDown e{x, x_stride, out, out_stride, add, add_pair, c.d_md_pinv, c.d_md_pinv_sh, conv.npolys, conv.nlimbs, nullptr, nullptr, nullptr, 0, 0, 0};
  dispatch_fwd(c, SetAddr{conv}, SetAddr{conv}, conv.nlimbs * conv.npolys, st, e, "ntt_fwd_rows_moddown", cols);
}

// ------------------------------------------------------------------------------- autotuner
namespace {

// forward + inverse over s, best of `reps` timed runs (ms)
double time_fwd_inv(Context& c, const LimbSet& s, int reps) {
  hipEvent_t e0, e1;
  FH_HIP(hipEventCreate(&e0));
  FH_HIP(hipEventCreate(&e1));
  ntt_fwd(c, s, c.stream);
  ntt_inv(c, s, c.stream);
  double best = 1e30;
  for (int r = 0; r < reps; ++r) {
    FH_HIP(hipEventRecord(e0, c.stream));
    ntt_fwd(c, s, c.stream);
    ntt_inv(c, s, c.stream);
    FH_HIP(hipEventRecord(e1, c.stream));
    FH_HIP(hipEventSynchronize(e1));
    float ms = 0;
    FH_HIP(hipEventElapsedTime(&ms, e0, e1));
    best = std::min(best, (double)ms);
  }
  FH_HIP(hipEventDestroy(e0));
  FH_HIP(hipEventDestroy(e1));
  return best;
}

}  // namespace

AutotuneResult autotune_ntt(Context& c, int polys) {
  if (polys < 1) throw Error(-1, "autotune needs at least one polynomial");
  // synthetic polynomials over every prime of the context (both arithmetic paths, in the
  // proportions of an extended basis), resident in HBM
  std::vector<int> ids(c.np);
  for (int i = 0; i < c.np; ++i) ids[i] = i;
  DBuf buf(c.pool, (size_t)polys * c.np * c.N);
  const LimbSet s = make_set(buf.p, (uint32_t)c.np, ids.data(), (uint32_t)polys, (uint64_t)c.np * c.N);
  fill_uniform(c, s, 0x7u, c.stream);
  const bool prof = c.prof.on;
  c.prof.on = false;
  const Tune saved = c.tune;
  AutotuneResult r{};
  const int reps = 3;
  auto measure = [&]() {
    ++r.candidates;
    return time_fwd_inv(c, s, reps);
  };
  try {
    // 1. radix split (all passes at the default workgroup size)
    c.tune.ntt_chunk_mb = saved.ntt_chunk_mb;
    for (int& t : c.tune.ntt_threads) t = kNttThreads;
    const int l1d = ntt_default_split(c.logN);
    c.tune.ntt_split = 0;
    r.ms_default = measure();
    double best = r.ms_default;
    int best_split = 0;
    // a candidate replaces the current choice only when it is clearly faster: timing noise and the
    // difference between this synthetic set and a workload's launches are a few percent
    constexpr double kGain = 0.95;
    // The conversions fused with the column pass (conv_cols) are built for the default split: another
    // one would turn them off in every ModUp and ModDown, which the transforms timed here do not show
    // (16 rotations at N = 2^15, 24 limbs: 882 us, at split 8 1037). Where they run the split stays.
    const bool fixed = conv_cols_usable(c, std::max(c.alpha, c.K));
    for (int l1 = 4; l1 <= 8 && !fixed; ++l1) {
      if (l1 == l1d || !ntt_split_ok(c.logN, l1)) continue;
      c.tune.ntt_split = l1;
      const double t = measure();
      if (t < best * kGain) best = t, best_split = l1;
    }
    c.tune.ntt_split = best_split;
    // 2. workgroup size per pass (wide tiles exist for the default split)
    if (best_split == 0) {
      for (int pass = 0; pass < 4; ++pass) {
        c.tune.ntt_threads[pass] = kNttWide;
        const double t = measure();
        if (t < best * kGain) best = t;
        else c.tune.ntt_threads[pass] = kNttThreads;
      }
    }
    // 3. limbs per launch pair: the whole set, or chunks of 256 / 128 MB (sized for the MALL) when
    // the set holds at least two of them; chunking adds launch tails, so it must win by 5%
    const size_t set_mb = ((size_t)polys * c.np * c.N * 8) >> 20;
    int best_chunk = c.tune.ntt_chunk_mb;
    for (int mb : {256, 128}) {
      if (set_mb < 2 * (size_t)mb || ((size_t)mb << 20) < (size_t)c.N * 8 * c.np) continue;
      c.tune.ntt_chunk_mb = mb;
      const double t = measure();
      if (t < best * 0.95) best = t, best_chunk = mb;
    }
    c.tune.ntt_chunk_mb = best_chunk;
    r.ms_best = best;
  } catch (...) {
    c.tune = saved;
    c.prof.on = prof;
    throw;
  }
  c.prof.on = prof;
  r.split = c.tune.ntt_split ? c.tune.ntt_split : ntt_default_split(c.logN);
  for (int i = 0; i < 4; ++i) r.threads[i] = c.tune.ntt_threads[i];
  r.chunk_mb = c.tune.ntt_chunk_mb;
  r.limbs = polys * c.np;
  return r;
}

}  // namespace fh
