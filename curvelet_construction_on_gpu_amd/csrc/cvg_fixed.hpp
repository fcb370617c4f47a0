// The fixed-point comparisons of the fused curvelet kernel (plain C++, so that
// a host compiler can check them).
#ifndef CVG_FIXED_HPP
#define CVG_FIXED_HPP

namespace cvg {

// Fixed point: max_k is 2^30; conversions and differences saturate.  Two
// approximate bounds whose difference is beyond kFixTol compare as the exact
// ones do: each is off by at most 8 units from the formulas (fused_limits
// keeps the denominators where that holds) and 1 from the conversion.
constexpr int kFixOne = 1 << 30;
constexpr int kFixTol = 18;

// A difference t of two bounds is open, |t| <= kFixTol, exactly where this is
// at most 2 kFixTol.  Formed in unsigned: t is saturated, and two bounds
// beyond the fixed-point range reach INT_MAX.
constexpr unsigned open_key(int t) { return static_cast<unsigned>(t) + static_cast<unsigned>(kFixTol); }

}  // namespace cvg

#endif
