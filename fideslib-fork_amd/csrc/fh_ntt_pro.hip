// Forward NTTs whose inputs are formed in their first launch: the Rescale correction, raised limbs,
// residues of integer coefficients. The kernels are in fh_ntt_impl.hpp.
#include "fh_ntt_impl.hpp"

namespace fh {

void ntt_pro_load() { load_unit(); }

void ntt_fwd_rescale(const Context& c, const LimbSet& e, const uint64_t* top, const uint64_t* x, uint32_t l, uint64_t* out, hipStream_t st) {
  const size_t o = (size_t)l * c.L1;
  EpiRescale ep{x, out, c.d_rs_qlinv + o, c.d_rs_qlinv_sh + o, l, e.npolys, nullptr, nullptr, 0, 0, 0};
  ProRescale pr{top, c.d_rs_QlQl + o, c.d_rs_QlQl_sh + o, l, e.npolys, {}};
  dispatch_fwd(c, SetAddr{e}, SetAddr{e}, e.nlimbs * e.npolys, st, ep, "ntt_fwd_rows_rescale", true, pr);
}

void ntt_fwd_mod_raise(const Context& c, const uint64_t* x0, const LimbSet& out, hipStream_t st) {
  ProModRaise pr{};
  pr.x0 = x0;
  pr.npolys = out.npolys;
  dispatch_fwd(c, SetAddr{out}, SetAddr{out}, out.nlimbs * out.npolys, st, EpiStore{}, "ntt_fwd_rows", true, pr);
}

void ntt_fwd_signed(const Context& c, const int64_t* m, const LimbSet& out, hipStream_t st) {
  ProSigned pr{};
  pr.m = m;
  pr.npolys = out.npolys;
  dispatch_fwd(c, SetAddr{out}, SetAddr{out}, out.nlimbs * out.npolys, st, EpiStore{}, "ntt_fwd_rows", true, pr);
}

}  // namespace fh
