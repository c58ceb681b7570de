// flux_rules.h -- what a block of the flux kernel stages and which shape an
// engine's launches take, as plain constexpr functions: the engine takes them
// as they are, and a CPU program can go through them over their whole range.
#pragma once

namespace cgo {

// A block's level planes have LB slots for its tracers l0 .. l0 + nl - 1
// (fewer than LB in the last block of a count that LB does not divide) and,
// where it forms the isoneutral coefficients itself (im 0), two more for T and
// S, unless those are its own first two tracers (l0 = 0).
constexpr bool flux_staged(int q, int l0, int nl, int LB, int im) { return q < LB ? q < nl : im == 0 && l0 != 0; }
// the tracer of a staged slot
constexpr int flux_slot_tracer(int q, int l0, int LB) { return q < LB ? l0 + q : q - LB; }

// The shape of a launch: tracers and wet columns per block, level planes
// resident in LDS, isoneutral coefficients from a pre-pass.
struct FluxTile {
    int lb, nt, nbuf, iso;
};
// What an engine starts with (FP64, FP32C).  FP32C: what the tuner picks for a
// large ensemble.  FP64: what it picked while the flux had a branch per face;
// for the flux as it is it picks 6, 256, 2, 0 (us per coupled step of
// 36x36x16x24, this one / that one: 32 members 214 / 175, 64 350 / 341, 256
// 1,307 / 1,255; 24 members of 72x72x32x24 1,048 / 953).
constexpr FluxTile FLUX_TILE[2] = {{8, 256, 2, 1}, {6, 256, 2, 1}};
// With this shape, untouched or set again, a batch too small to fill the chip
// may take the flux split by levels; any other shape was asked for and holds
// for every batch.
constexpr bool flux_auto(const FluxTile& t, int p) {
    return t.lb == FLUX_TILE[p].lb && t.nt == FLUX_TILE[p].nt && t.nbuf == FLUX_TILE[p].nbuf && t.iso == FLUX_TILE[p].iso;
}

}  // namespace cgo
