// What the prefill GEMMs (gemm.hip, gemm_rows.hip) share.
#pragma once

namespace wg {

// The weight form of a launch: the three zero-point kinds of 4-bit row
// groups, or Q8 for WG_LAYOUT_Q8 (signed bytes, no zero point).
constexpr int Q8 = 3;

}  // namespace wg
