// flux_rules.h -- what a block of the flux kernel stages and which shape an
// engine's launches take, as plain constexpr functions: the engine takes them
// as they are, and a CPU program can go through them over their whole range.
#pragma once
#include <cstddef>

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

// Levels per block of the flux split by levels, 0: whole columns.  nb: a
// batch's blocks of two tracers and whole columns, cols its wet columns, maxk
// its deepest grid's levels, p its precision (0 FP64, 1 FP32C), mix: some
// member mixes along isoneutrals, bgc: some member has BIOGEM, nv: doubles of
// workspace the split needs (FP32C members with BIOGEM: their new values).
// Up to 768 such blocks the levels are cut into as many chunks (of two levels
// at least) as fill the chip.  The split's price is the convection, which then
// walks every column; what bounds it from above is, for FP64 members, that two
// of its blocks fit a CU (512 in all; a few columns past that still gain), and
// for FP32C members, three of whose blocks fit, that walk, the dearer where it
// also forms BIOGEM's column sums.  us per step, whole columns with their
// pre-pass / split, coupled steps unless said: FP64 36x36x16x24 1 member (nb
// 48) 129 / 76, 10 (480) 154 / 117, 16 (768, 14,500 columns) 167 / 161, 18
// (864) 160 / 191, 24 (1,152) 188 / 219; 36x36x16x8 30 (480) 171 / 145, 41
// (656, 37,200 columns) 166 / 184; 18x18x8x8 120 (480) 109 / 98, 144 (576,
// 32,700) 112 / 120, 256 (1,024) 131 / 160; 72x72x32x8 12 (816, 43,500) 425 /
// 410, 14 (952) 453 / 476.  FP32C 36x36x16x24 1 113 / 77, 8 (384) 120 / 108, 10
// (480) 123 / 124, 16 (768) 130 / 138; 36x36x16x8 14 (224, 12,700) 118 / 103,
// 20 (320, 18,100) 129 / 137; 18x18x8x8 57 (228, 12,900) 73 / 69, 96 (384,
// 21,800) 86 / 98; transport of 48 members of 36x36x16x8 (768) 76 / 74.
// Without isoneutral mixing whole columns need no pre-pass and read no
// corners, so that they take over earlier: on shallow grids, where there is
// little to split, and on deep ones, where the convection that then walks
// every column costs the most.  us per step of transport, whole columns /
// split: FP64 36x36x16x24 8 members (nb 384) 58 / 54, 10 (480) 59 / 53, 12
// (576) 59 / 75; 36x36x8x24 4 (192) 33 / 30, 8 (384) 32 / 36; 72x72x32x8 4
// (272) 102 / 88, 6 (408) 103 / 100, 8 (544) 103 / 148; FP32C 36x36x16x24 8 42
// / 39, 10 45 / 46; 72x72x32x8 4 76 / 73, 6 78 / 86.
constexpr size_t FLUX_NV_MAX = (size_t)64 << 20;  // 512 MiB; a third of it is a full chip on 48 levels
constexpr int flux_split_levels(long long nb, long long cols, int maxk, int p, bool mix, bool bgc, size_t nv) {
    constexpr int FULL = 768;
    const int plain = 30 * maxk < 13056 / maxk ? 30 * maxk : 13056 / maxk;
    const bool split = !mix     ? nb <= (p == 0 ? plain : plain * 17 / 20)
                       : p == 0 ? nb <= 512 || (nb <= 832 && cols <= 1400 * maxk)
                       : bgc    ? nb <= 448 && cols <= 15000
                                : nb <= FULL;
    if (!split || nv > FLUX_NV_MAX) return 0;
    const long long fill = FULL / nb > 1 ? FULL / nb : 1, deep = (maxk + 1) / 2;
    const int chunks = (int)(fill < deep ? fill : deep);
    return (maxk + chunks - 1) / chunks;
}

}  // namespace cgo
