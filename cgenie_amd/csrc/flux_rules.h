// flux_rules.h -- what a block of the flux kernel stages, as plain constexpr
// functions: the kernel takes them as they are, and a CPU program can go
// through them over their whole range.
#pragma once

namespace cgo {

// A block's level planes have LB slots for its tracers l0 .. l0 + nl - 1
// (fewer than LB in the last block of a count that LB does not divide) and,
// where it forms the isoneutral coefficients itself (im 0), two more for T and
// S, unless those are its own first two tracers (l0 = 0).
constexpr bool flux_staged(int q, int l0, int nl, int LB, int im) { return q < LB ? q < nl : im == 0 && l0 != 0; }
// the tracer of a staged slot
constexpr int flux_slot_tracer(int q, int l0, int LB) { return q < LB ? l0 + q : q - LB; }

}  // namespace cgo
