// tstep_impl.h -- GOLDSTEIN tracer step kernels (tstepo_flux + eos, co).
//
// Included by k_tstep_f64.hip (built with -ffp-contract=off: every operation
// rounds as the reference writes it, so the FP64 path reproduces the CPU
// restatement bit for bit) and by k_tstep_f32.hip (the FP32 form).
//
// k_flux: one thread per (member, water column, tracer block).  The thread
// marches k upward like goldstein.f90:2466-2641 and carries the bottom face
// flux fb from the level below (2635), so every vertical face flux is
// computed once.  Horizontal face fluxes are evaluated by both neighbours
// with the same expression and operands (the east flux of cell i is the
// west flux of cell i+1, 2633), so both sides see the same bits and the
// scheme stays conservative.  Level k+1 values are loaded once and carried
// down to level k of the next iteration.
#pragma once
#include "cgocn_dev.h"
#include "flux_rules.h"

#include <type_traits>

namespace cgo {


template <typename R> struct Met;
template <> struct Met<double> {
    static __device__ __forceinline__ const double* j(const GridDev& g) { return g.mj; }
    static __device__ __forceinline__ const double* k(const GridDev& g) { return g.mk; }
};
template <> struct Met<float> {
    static __device__ __forceinline__ const float* j(const GridDev& g) { return g.mjf; }
    static __device__ __forceinline__ const float* k(const GridDev& g) { return g.mkf; }
};

// 2^e for e within a double's normal exponents
__device__ __forceinline__ double pow2(int e) { return __hiloint2double((1023 + e) << 20, 0); }

// weight of one unit of the int16 carry of a float value x: 2^-16 ulp(x)
__device__ __forceinline__ double carry_unit(float x) { return pow2(carry_exp(x) - 23 - 16); }

// the carry of a value x stored as the float h: x - h in those units, rounded
// to nearest (x - h is exact, scaling it by a power of two too, and adding
// 1.5 2^52 leaves the rounded integer in the low word: one instruction in
// place of ldexp, rint and a conversion, each of a quarter of the rate).  It
// lies within +-2^15; the clamp is taken on the integer.
__device__ __forceinline__ int carry_of(double x, float h) {
    const double r = __builtin_fma(x - (double)h, pow2(23 + 16 - carry_exp(h)), 0x1.8p52);
    const int ri = __double2loint(r);
    return ri < -32767 ? -32767 : (ri > 32767 ? 32767 : ri);
}

// state access as double (FP32 form: hi + carry)
// a / b: the IEEE quotient in FP64; in the FP32 form the hardware reciprocal
// (1 ulp), for the per-cell isoneutral coefficients
__device__ __forceinline__ double fdiv(double a, double b) { return a / b; }
__device__ __forceinline__ float fdiv(float a, float b) { return a * __builtin_amdgcn_rcpf(b); }

template <typename R> struct StateIO;
// (all state pointers are global memory: the casts keep the accesses off
// the flat path, whose loads also count against the LDS wait counter)
// ldr/val split a load from its conversion so that a thread can issue the
// loads of many cells before it waits for any of them.
template <> struct StateIO<double> {
    struct Raw {
        double v;
    };
    static __device__ __forceinline__ Raw ldr(const void* s, const int16_t*, uint32_t i) {
        return Raw{at((const AS_GLOBAL double*)s, i)};
    }
    static __device__ __forceinline__ double val(Raw r, bool) { return r.v; }
    static __device__ __forceinline__ double ld(const void* s, const int16_t*, uint32_t i) {
        return at((const AS_GLOBAL double*)s, i);
    }
    static __device__ __forceinline__ void st(void* s, int16_t*, uint32_t i, double x) {
        at((AS_GLOBAL double*)s, i) = x;
    }
    // the value a later ld returns after st(x)
    static __device__ __forceinline__ double rt(double x, bool) { return x; }
};
template <> struct StateIO<float> {
    struct Raw {
        float h;
        int16_t c;
    };
    static __device__ __forceinline__ Raw ldr(const void* s, const int16_t* lo, uint32_t i) {
        Raw r;
        r.h = at((const AS_GLOBAL float*)s, i);
        r.c = lo ? at((const AS_GLOBAL int16_t*)lo, i) : (int16_t)0;
        return r;
    }
    static __device__ __forceinline__ double val(Raw r, bool carry) {
        double x = (double)r.h;
        if (carry) x += (double)r.c * carry_unit(r.h);
        return x;
    }
    static __device__ __forceinline__ double ld(const void* s, const int16_t* lo, uint32_t i) {
        float h = at((const AS_GLOBAL float*)s, i);
        double x = (double)h;
        if (lo) x += (double)at((const AS_GLOBAL int16_t*)lo, i) * carry_unit(h);
        return x;
    }
    static __device__ __forceinline__ void st(void* s, int16_t* lo, uint32_t i, double x) {
        float h = (float)x;
        at((AS_GLOBAL float*)s, i) = h;
        if (lo) at((AS_GLOBAL int16_t*)lo, i) = (int16_t)carry_of(x, h);
    }
    // the value a later ld returns after st(x): the float, plus the carry
    // split and clamped as st stores it
    static __device__ __forceinline__ double rt(double x, bool carry) {
        const float h = (float)x;
        double v = (double)h;
        if (carry) v += (double)carry_of(x, h) * carry_unit(h);
        return v;
    }
};

__device__ __forceinline__ void atomic_max_pos(double* p, double v) {
    // non-negative doubles order like their bit patterns
    atomicMax(reinterpret_cast<unsigned long long*>(p), (unsigned long long)__double_as_longlong(v));
}

// Work of k_flux: a block takes up to FLUX_THREADS consecutive wet columns
// (ascending column order; land columns get no thread) and the tracer block
// [l0, l0 + LB).  LDS layout: the k1 tile, a ring of NBUF level planes of LB
// tracer slots plus T and S, each covering the block's flattened column range
// [t0, t1) -- every east/west (periodic wrap included, offsets below maxi)
// and north/south neighbour of its columns -- and the carried bottom-face
// flux.  With NBUF = 3 the planes k, k+1 and the prefetched k+2 are
// resident; with NBUF = 2 the prefetched plane replaces plane k after a
// second barrier per level (less LDS, more workgroups per CU).  The host cuts
// blocks so that t1 - t0 <= flux_tw(FLUX_THREADS).
// The FP32 form also stages the carry of every value, as a float residual,
// so differences of neighbours are taken at the stored (~40-bit) precision.
// ns level-plane slots (lb tracers, plus T and S when the block computes the
// isoneutral coefficients itself), lb carried bottom fluxes.  Every slot
// holds flux_tw(nt) positions, a compile-time stride, so each slot's offset
// is an immediate of the LDS instruction.
__host__ __device__ constexpr size_t flux_lds_bytes(int ns, int lb, int es, int nt, int nbuf) {
    return (size_t)flux_tw(nt) * 4 + (size_t)nbuf * ns * flux_tw(nt) * es + (size_t)lb * nt * es +
           (es == 4 ? (size_t)nbuf * ns * flux_tw(nt) * 4 : 0);
}

// the carry c of a float h as a float: c * 2^-16 ulp(h) (exact unless |h| < 2^-87)
// (c 2^-39 is exact; times 2^e, the exponent bits of h, it rounds once, as
// ldexpf(c, e - 39) does; zero and subnormal h give 0, as ldexpf(c, -165) does)
__device__ __forceinline__ float carry_residual(float h, int16_t c) {
    return ((float)c * 0x1p-39f) * __uint_as_float(__float_as_uint(h) & 0x7f800000u);
}

// IM selects where the isoneutral coefficients come from: 0 computed in every
// tracer block from T and S staged beside its tracers; 1 the pre-pass (one
// block per column block, T and S only, LB = 2) that computes them once per
// cell into the member's isoc planes; 2 the tracer blocks after that pre-pass,
// which load them and stage only their own tracers.
// MODE 3 is mode 0 for a batch too small to fill the chip with blocks that
// march whole columns: blockIdx.x also runs over chunks of sp.kc levels.  A
// block first forms the level under its chunk without storing it, for the
// flux through its own bottom face.  What a march carries up a whole column,
// the stability of the new density and the coupling's column sums, is left
// to co, which then takes every column (FP32 members hand it their new values
// unrounded, as the march sums them).
template <typename R, int LB, int FLUX_THREADS, int FLUX_NBUF, int MODE>
__global__ __launch_bounds__(FLUX_THREADS, 2) void k_flux(const MemberDev* __restrict__ mems,
                                                       const int32_t* __restrict__ list, FluxSplit sp_) {
    constexpr bool SPLIT = MODE == 3;
    constexpr int IM = SPLIT ? 0 : MODE;
    constexpr int NS = IM == 0 ? LB + 2 : LB;  // slots per staged level plane
    constexpr int TWS = flux_tw(FLUX_THREADS);  // positions per slot (>= every block's t1 - t0)
    extern __shared__ __align__(16) unsigned char smem[];
    const BlockXYZ B = xcd_blk();
    const MemberDev& M = mems[list[B.z]];
    const GridDev& g = M.g;
    const int maxi = g.maxi, maxj = g.maxj, maxk = g.maxk, L = M.L;
    constexpr int V = FLUX_THREADS == 256 ? 1 : 0;
    const int l0 = B.y * LB;
    const int bx = SPLIT ? B.x % sp_.nbx : B.x;
    if (bx >= g.nfblk[V] || l0 >= L) return;  // uniform for the block
    // every wet column's sums are formed below
    if (!SPLIT && IM != 1 && M.bgc && B.x == 0 && B.y == 0 && threadIdx.x == 0) *gp(M.sfresh) = 1;
    const int nl = (L - l0) < LB ? (L - l0) : LB;
    const AS_GLOBAL FluxBlk* blk = gp(g.fblk[V]) + bx;
    const int w0 = blk->w0, t0 = blk->t0, TW = blk->t1 - t0, nw = blk->w1 - w0;
    int* sk1 = reinterpret_cast<int*>(smem);
    R* sp = reinterpret_cast<R*>(smem + (size_t)TWS * 4);
    R* sfb = sp + FLUX_NBUF * NS * TWS;
    float* sr = reinterpret_cast<float*>(sfb + LB * FLUX_THREADS);  // FP32 form: residual ring
    // slot q < LB: tracer l0+q; T and S sit in slots 0/1 when l0 == 0, else
    // (coefficients computed here) LB/LB+1
    const int qT = (l0 == 0 || IM != 0) ? 0 : LB, qS = (l0 == 0 || IM != 0) ? 1 : LB + 1;
    // (a slot past the block's last tracer is not loaded: the member's state ends there)
    auto staged = [&](int q) { return flux_staged(q, l0, nl, LB, IM); };
    __shared__ int s_kmin;
    const int tid = threadIdx.x;
    if (tid == 0) s_kmin = maxk + 1;
    for (int pp = tid; pp < TW; pp += FLUX_THREADS) {
        const int c = t0 + pp;
        sk1[pp] = k1at(g, c % maxi + 1, c / maxi + 1);
    }
    __syncthreads();
    const bool active = tid < nw;
    const int col = active ? gp(g.wetsorted)[w0 + tid] : t0;
    const int i0 = col % maxi, j0 = col / maxi;
    const int I = i0 + 1, J = j0 + 1;
    const int k1c = active ? k1at(g, I, J) : maxk + 1;
    const int k1e = k1at(g, I + 1, J), k1w = k1at(g, I - 1, J);
    const int k1n = k1at(g, I, J + 1), k1s = k1at(g, I, J - 1);
    if (k1c <= maxk) atomicMin(&s_kmin, k1c);
    __syncthreads();
    // the block's levels [klo, khi], entered at kmin: the level under klo where it has one
    const int klo = SPLIT ? 1 + (B.x / sp_.nbx) * sp_.kc : 1, khi = SPLIT ? min(maxk, klo + sp_.kc - 1) : maxk;
    const int kmin = SPLIT ? max(s_kmin, klo - 1) : s_kmin;
    if (kmin > khi) return;  // no wet cell in the block's levels

    constexpr bool ANOM = sizeof(R) == 4;  // FP32 form: fluxes of q - q_cell plus q_cell * div(u)
    const int par = *gp(M.parity);
    const AS_GLOBAL R* __restrict__ src = gp(static_cast<const R*>(M.st[par]));
    AS_GLOBAL R* __restrict__ dst = gp(static_cast<R*>(M.st[par ^ 1]));
    const AS_GLOBAL int16_t* __restrict__ lo_src = M.lo[par] ? gp(M.lo[par]) : nullptr;
    int16_t* __restrict__ lo_dst = M.lo[par ^ 1];
    const AS_GLOBAL R* __restrict__ u = gp(static_cast<const R*>(M.u));
    AS_GLOBAL double* __restrict__ rhop = gp(M.rho);
    const int plane = g.ncol, tstride = maxk * g.ncol, ncell = g.ncell;
    // neighbour positions in the tile
    const int p = col - t0;
    const int pe = p + (i0 + 1 == maxi ? 1 - maxi : 1);
    const int pw = p + (i0 == 0 ? maxi - 1 : -1);
    const int pn = p + (j0 + 1 < maxj ? maxi : 0);
    const int ps = p - (j0 > 0 ? maxi : 0);
    const int cw = j0 * maxi + (i0 == 0 ? maxi - 1 : i0 - 1);
    const int cs = (j0 > 0 ? j0 - 1 : 0) * maxi + i0;
    const AS_GLOBAL R* mj = gp(Met<R>::j(g));
    const AS_GLOBAL R* mk = gp(Met<R>::k(g));
    const int JS = maxj + 2, KS = maxk + 2;
    const R rc = mj[MJ_RC * JS + J], rc2 = mj[MJ_RC2 * JS + J];
    // (the walls' northward metrics are the caller's to leave undefined; their
    // faces are closed, and zero keeps a product with a closed face's zero)
    const bool wallN = J == maxj, wallS = J == 1;
    const R cvn = mj[MJ_CV * JS + J], cv2n = wallN ? (R)0 : mj[MJ_CV2 * JS + J];
    const R cvs = mj[MJ_CV * JS + J - 1], cv2s = wallS ? (R)0 : mj[MJ_CV2 * JS + J - 1];
    const R dsvn = mj[MJ_DSVM * JS + J], dsvs = wallS ? (R)0 : mj[MJ_DSVM * JS + J - 1];
    const R rds = mj[MJ_RDS * JS + J];
    const R rdsvn = wallN ? (R)0 : mj[MJ_RDSV * JS + J], rdsvs = wallS ? (R)0 : mj[MJ_RDSV * JS + J - 1];
    const R dphi = (R)g.dphi, rdphi = (R)g.rdphi;
    const R diff1 = sizeof(R) == 8 ? (R)M.diff1 : (R)M.diff1f;
    const R diffv = sizeof(R) == 8 ? (R)M.diff2 : (R)M.diff2f;
    const R e0 = (R)g.ec[0], e1 = (R)g.ec[1], e2 = (R)g.ec[2], e3 = (R)g.ec[3];
    const bool mixes = __builtin_amdgcn_readfirstlane(M.diso) != 0;
    const uint32_t has_mix = (uint32_t)__builtin_amdgcn_readfirstlane(M.diso ? ~0 : 0);
    const R scc = mixes ? e1 : (R)0;

    auto SP = [&](int buf, int q, int pp) -> R& { return sp[(buf * NS + q) * TWS + pp]; };
    auto SR = [&](int buf, int q, int pp) -> float& { return sr[(buf * NS + q) * TWS + pp]; };
    // difference of two staged values; the FP32 form adds the residuals
    auto D = [&](int buf, int q, int pa, int pb) -> R {
        if (ANOM) return (SP(buf, q, pa) - SP(buf, q, pb)) + (R)(SR(buf, q, pa) - SR(buf, q, pb));
        return SP(buf, q, pa) - SP(buf, q, pb);
    };
    // difference across levels (same column)
    auto DK = [&](int bu, int bc, int q, int pp) -> R {
        if (ANOM) return (SP(bu, q, pp) - SP(bc, q, pp)) + (R)(SR(bu, q, pp) - SR(bc, q, pp));
        return SP(bu, q, pp) - SP(bc, q, pp);
    };
    auto FB = [&](int q) -> R& { return sfb[q * FLUX_THREADS + tid]; };
    // prefetch of one plane into registers, then into the LDS ring
    constexpr int FLUX_PF = flux_pf(FLUX_THREADS);
    R pf[NS][FLUX_PF];
    int16_t pc[ANOM ? NS : 1][FLUX_PF];
    auto fetch = [&](int kz) {
        const int o = kz * plane + t0;
#pragma unroll
        for (int r = 0; r < FLUX_PF; r++) {
            const int pp = tid + r * FLUX_THREADS;
            const bool ok = pp < TW && kz + 1 >= sk1[pp < TW ? pp : 0];
#pragma unroll
            for (int q = 0; q < NS; q++)
                if (staged(q)) {
                    const uint32_t i = (uint32_t)(flux_slot_tracer(q, l0, LB) * tstride + o + pp);
                    pf[q][r] = ok ? at(src, i) : (R)0;
                    if (ANOM) pc[ANOM ? q : 0][r] = (ok && lo_src) ? at(lo_src, i) : (int16_t)0;
                }
        }
    };
    auto commit = [&](int buf) {
#pragma unroll
        for (int r = 0; r < FLUX_PF; r++) {
            const int pp = tid + r * FLUX_THREADS;
            if (pp < TW) {
#pragma unroll
                for (int q = 0; q < NS; q++)
                    if (staged(q)) {
                        SP(buf, q, pp) = pf[q][r];
                        if (ANOM) SR(buf, q, pp) = carry_residual((float)pf[q][r], pc[ANOM ? q : 0][r]);
                    }
            }
        }
    };

    for (int q = 0; q < LB; q++) FB(q) = (R)0;
    // the idle slots of the last block hold zeros
    for (int q = nl; q < LB; q++)
        for (int pp = tid; pp < TW; pp += FLUX_THREADS)
#pragma unroll
            for (int b = 0; b < FLUX_NBUF; b++) {
                SP(b, q, pp) = (R)0;
                if (ANOM) SR(b, q, pp) = 0.0f;
            }
    double rlow = 0.0;     // the new density of the level below, and whether
    bool falls = true;     // it falls strictly from k1 up (co leaves such a column as it is)
    int32_t limps = 0;
    double dmaxv = 0.0;
    // The isoneutral slope terms are formed in FP64 in both forms.  The
    // density gradients they divide by are differences of nearly equal
    // terms, so the FP32 form takes its staged values with their residuals
    // and the FP64 metrics, and rounds the finished coefficients to float
    // once; in float they lose up to 1e-4 of their value where the
    // stratification is weak.  The FP64 form evaluates the restatement's
    // expressions on the same values, bit for bit.
    const double rcD = gp(g.mj)[MJ_RC * JS + J], cvnD = gp(g.mj)[MJ_CV * JS + J];
    const double cvsD = gp(g.mj)[MJ_CV * JS + J - 1];
    const double rdsvnD = wallN ? 0.0 : gp(g.mj)[MJ_RDSV * JS + J], rdsvsD = wallS ? 0.0 : gp(g.mj)[MJ_RDSV * JS + J - 1];
    const double rdphiD = g.rdphi, diff1D = M.diff1;
    const double e0D = g.ec[0], e1D = g.ec[1], e2D = g.ec[2], e3D = g.ec[3];
    const double sccD = mixes ? e1D : 0.0;
    auto SPD = [&](int buf, int q, int pp) -> double {
        if (ANOM) return (double)SP(buf, q, pp) + (double)SR(buf, q, pp);
        return (double)SP(buf, q, pp);
    };
    auto DD = [&](int buf, int q, int pa, int pb) -> double {
        if (ANOM)
            return ((double)SP(buf, q, pa) - (double)SP(buf, q, pb)) + ((double)SR(buf, q, pa) - (double)SR(buf, q, pb));
        return (double)(SP(buf, q, pa) - SP(buf, q, pb));
    };
    auto DKD = [&](int bu, int bc, int q, int pp) -> double {
        if (ANOM)
            return ((double)SP(bu, q, pp) - (double)SP(bc, q, pp)) + ((double)SR(bu, q, pp) - (double)SR(bc, q, pp));
        return (double)(SP(bu, q, pp) - SP(bc, q, pp));
    };
    // The tile positions of a cell's neighbours at a level: its own where the
    // face between them is closed, so that every difference across a closed
    // face is zero without a test.  A test per face and tracer was a branch
    // each, with an LDS read waited for behind it: twenty a tracer, the largest
    // part of the 20,000 cycles a level of eight FP64 tracers took.  Without
    // them the flux alone takes, 64 FP64 members of 36x36x16x24, 250 -> 201 us
    // a launch, 256 FP32C members 512 -> 461 us, six of 72x72x32x40 209 -> 154.
    // (Loading a level's coefficients while the one below it is formed hid no
    // more and cost a wave per SIMD: 483 us for the 256.)
    struct Nbr {
        int e, w, n, s;
    };
    auto nbrs = [&](int k) {
        return Nbr{k >= k1e ? pe : p, k >= k1w ? pw : p, k >= k1n ? pn : p, k >= k1s ? ps : p};
    };
    // the isoneutral slope terms of a cell at level k < maxk from the staged
    // T and S (2489-2501, 2561-2605): dzrho, the four corner gradients, the
    // slope limiter; counts limps and the diffusive stability number
    auto iso_coeffs = [&](int k, int cb, int ub, bool& iso, double& dzrho, double& rdzrho, double& slim,
                          double* dxr, double* dyr) {
        const AS_GLOBAL double* mkD = gp(g.mk);
        const double rdza = mkD[MK_RDZA * KS + k], dt = mkD[MK_DT * KS + k];
        const double Tc = SPD(cb, qT, p), Tu = SPD(ub, qT, p);
        const double tatw = 0.5 * (Tc + Tu);
        const double tec = -e0D - e2D * tatw * 2 - e3D * tatw * tatw * 3;
        dzrho = (e1D * DKD(ub, cb, qS, p) - tec * DKD(ub, cb, qT, p)) * rdza;
        if (mixes && dzrho < -1.0E-12) {
            const Nbr nc = nbrs(k), nu = nbrs(k + 1);
            iso = true;
            rdzrho = fdiv(1.0, dzrho);
            double tv1 = 0;
            // ina order (knp, nnp) = (0,0), (0,1), (1,0), (1,1)
#pragma unroll
            for (int n = 0; n < 4; n++) {
                const int b = n < 2 ? cb : ub;
                const bool east = n & 1;
                const Nbr& m = n < 2 ? nc : nu;
                const double dxT = (east ? DD(b, qT, m.e, p) : DD(b, qT, p, m.w)) * rcD * rdphiD;
                const double dxS = (east ? DD(b, qS, m.e, p) : DD(b, qS, p, m.w)) * rcD * rdphiD;
                const double dyT = east ? DD(b, qT, m.n, p) * cvnD * rdsvnD : DD(b, qT, p, m.s) * cvsD * rdsvsD;
                const double dyS = east ? DD(b, qS, m.n, p) * cvnD * rdsvnD : DD(b, qS, p, m.s) * cvsD * rdsvsD;
                dxr[n] = sccD * dxS - tec * dxT;
                dyr[n] = sccD * dyS - tec * dyT;
                tv1 = tv1 + dxr[n] * dxr[n] + dyr[n] * dyr[n];
            }
            tv1 = 0.25 * tv1 * rdzrho * rdzrho;
            const double ssmax = mkD[MK_SSMAX * KS + k];
            if (tv1 > ssmax) {
                slim = fdiv(ssmax * ssmax, tv1 * tv1);
                if (!SPLIT || k >= klo) limps++;
            } else {
                slim = 1;
            }
            tv1 = tv1 * slim * diff1D * rdza;
            const double tvd = tv1 * dt * rdza;
            if (tvd > dmaxv && (!SPLIT || k >= klo)) dmaxv = tvd;
        }
    };
    // the FP32 form's isoneutral coefficients: corner differences times ax, ay
    // (the sign of the west/south corners folded in) and the vertical qq,
    // formed in FP64 and rounded once
    auto fp32_iso = [&](int k, bool iso, double slim, double rdzrho, const double* dxr, const double* dyr, R* ax,
                        R* ay, R& qq) {
#pragma unroll
        for (int n = 0; n < 4; n++) ax[n] = ay[n] = (R)0;
        qq = (R)0;
        if (iso) {
            const double rdza = gp(g.mk)[MK_RDZA * KS + k];
            const double isoc = 0.25 * slim * diff1D;
            const double f = 2 * isoc * rdzrho;
            double s2 = 0;
#pragma unroll
            for (int n = 0; n < 4; n++) {
                const bool east = n & 1;
                ax[n] = (R)(f * dxr[n] * rcD * rdphiD * (east ? 1.0 : -1.0));
                ay[n] = (R)(f * dyr[n] * (east ? cvnD * rdsvnD : -(cvsD * rdsvsD)));
                s2 = s2 + dxr[n] * dxr[n] + dyr[n] * dyr[n];
            }
            qq = (R)(isoc * s2 * (rdzrho * rdzrho) * rdza);
        }
    };
    // Members with BIOGEM: the coupling's column sums of the new state
    // (biogem.f90:1984-1997, 2016-2025), accumulated up the column in the
    // order the coupling adds them; co redoes the columns it mixes.
    const bool sums = !SPLIT && IM != 1 && M.bgc != 0;
    AS_GLOBAL double* const nvs =
        SPLIT && ANOM && M.bgc ? gp(sp_.nv) + (size_t)B.z * sp_.stride : nullptr;  // [L][ncell]: co's sums
    const double rSold = sums ? 1.0 / gp(M.scal)[SC_SMEAN] : 0.0;
    double accs[LB], accS = 0.0;
#pragma unroll
    for (int q = 0; q < LB; q++) accs[q] = 0.0;
    fetch(kmin - 1);
    commit(kmin % FLUX_NBUF);
    if (kmin < maxk) {
        fetch(kmin);
        commit((kmin + 1) % FLUX_NBUF);
    }
    __syncthreads();
    for (int k = kmin; k <= khi; k++) {
        const int kz = k - 1;
        const int cb = k % FLUX_NBUF, ub = (k + 1) % FLUX_NBUF;
        const bool top = (k == maxk);
        const bool more = k + 2 <= (SPLIT ? min(khi + 1, maxk) : maxk);
        const bool own = !SPLIT || k >= klo;
        if (more) fetch(kz + 2);
        if (IM == 1 && active && k >= k1c && !top && mixes) {
            // the pre-pass: the cell's isoneutral coefficients, once
            const uint32_t oc = (uint32_t)(kz * plane + col);
            bool iso = false;
            double dzrho = 0, rdzrho = 0, slim = 1, dxr[4] = {0, 0, 0, 0}, dyr[4] = {0, 0, 0, 0};
            iso_coeffs(k, cb, ub, iso, dzrho, rdzrho, slim, dxr, dyr);
            if constexpr (ANOM) {
                R ax[4], ay[4], qq;
                fp32_iso(k, iso, slim, rdzrho, dxr, dyr, ax, ay, qq);
                AS_GLOBAL float* ic = reinterpret_cast<AS_GLOBAL float*>(gp(M.isoc));
#pragma unroll
                for (int n = 0; n < 4; n++) {
                    at(ic, (uint32_t)(n * ncell) + oc) = ax[n];
                    at(ic, (uint32_t)((4 + n) * ncell) + oc) = ay[n];
                }
                at(ic, (uint32_t)(8 * ncell) + oc) = qq;
            } else {
                AS_GLOBAL double* ic = gp(M.isoc);
                at(ic, oc) = iso ? (double)dzrho : 1.0;  // +1: no isoneutral flux in this cell
#pragma unroll
                for (int n = 0; n < 4; n++) {
                    at(ic, (uint32_t)((1 + n) * ncell) + oc) = dxr[n];
                    at(ic, (uint32_t)((5 + n) * ncell) + oc) = dyr[n];
                }
                at(ic, (uint32_t)(9 * ncell) + oc) = slim;
            }
        }
        if (IM != 1 && active && k >= k1c) {
            const int o = kz * plane;
            // face velocities and Peclet-weighted upwinding (goldstein.f90:2489-2523);
            // the FP32 form reads its face coefficients instead (below)
            const uint32_t oc = (uint32_t)(o + col);
            const R dza = mk[MK_DZA * KS + k], rdza = mk[MK_RDZA * KS + k];
            const R dt = mk[MK_DT * KS + k], rdz = mk[MK_RDZ * KS + k];
            R ue_ = 0, uw_ = 0, un_ = 0, us_ = 0, ua_ = 0;
            R upe = 0, upw = 0, upn = 0, ups = 0, upa = 0;
            if constexpr (!ANOM) {
                // (closed faces carry nothing)
                ue_ = k >= k1e ? at(u, oc) : (R)0;
                uw_ = k >= k1w ? at(u, (uint32_t)(o + cw)) : (R)0;
                un_ = k >= k1n ? at(u, ncell + oc) : (R)0;
                us_ = k >= k1s ? at(u, (uint32_t)(ncell + o + cs)) : (R)0;
                ua_ = at(u, 2 * ncell + oc);
                R pec;
                pec = ue_ * dphi / diff1; upe = pec / ((R)2.0 + fabs(pec));
                pec = uw_ * dphi / diff1; upw = pec / ((R)2.0 + fabs(pec));
                pec = un_ * dsvn / diff1; upn = pec / ((R)2.0 + fabs(pec));
                pec = us_ * dsvs / diff1; ups = pec / ((R)2.0 + fabs(pec));
                pec = ua_ * dza / diffv; upa = pec / ((R)2.0 + fabs(pec));
            }
            const Nbr nc = nbrs(k), nu = nbrs(k + 1);
            // isoneutral coefficients from T and S (2489-2501, 2561-2605)
            bool iso = false;
            double dzrho = 0, rdzrho = 0, slim = 1, dxr[4] = {0, 0, 0, 0}, dyr[4] = {0, 0, 0, 0};
            R ax[4] = {0, 0, 0, 0}, ay[4] = {0, 0, 0, 0}, qq = 0;  // the FP32 form's coefficients
            if (!top) {
                if constexpr (IM == 2) {
                    if (ANOM ? M.diso != 0 : mixes) {
                        if constexpr (ANOM) {
                            // zero coefficients give the flux without the isoneutral term exactly
                            const AS_GLOBAL float* ic = reinterpret_cast<const AS_GLOBAL float*>(gp(M.isoc));
#pragma unroll
                            for (int n = 0; n < 4; n++) {
                                ax[n] = at(ic, (uint32_t)(n * ncell) + oc);
                                ay[n] = at(ic, (uint32_t)((4 + n) * ncell) + oc);
                            }
                            qq = at(ic, (uint32_t)(8 * ncell) + oc);
                        } else {
                            const AS_GLOBAL double* ic = gp(M.isoc);
                            dzrho = at(ic, oc);
                            iso = dzrho < 0.0;
                            if (iso) {
#pragma unroll
                                for (int n = 0; n < 4; n++) {
                                    dxr[n] = at(ic, (uint32_t)((1 + n) * ncell) + oc);
                                    dyr[n] = at(ic, (uint32_t)((5 + n) * ncell) + oc);
                                }
                                slim = at(ic, (uint32_t)(9 * ncell) + oc);
                            }
                        }
                    }
                } else {
                    iso_coeffs(k, cb, ub, iso, dzrho, rdzrho, slim, dxr, dyr);
                    if constexpr (ANOM) fp32_iso(k, iso, slim, rdzrho, dxr, dyr, ax, ay, qq);
                }
            }
            // discrete divergence of the open faces (FP32 form only)
            // (evaluated in FP64 from the FP64 velocities when they are set)
            const R divu = ANOM ? at(u, 6 * ncell + oc) : (R)0;
            const R isoc = (R)0.25 * slim * diff1;
            // A cell without the isoneutral flux has zero gradients (the FP32
            // form: coefficients), and its flux is masked as well: an infinity at
            // a corner stays out of it.  (Hidden from the compiler, which makes a
            // branch per tracer of a select: 256 FP64 members of 36x36x16x24 729
            // us a launch, 612 so.)
            uint32_t has_iso = iso ? ~0u : 0u;
            if (!ANOM) asm("" : "+v"(has_iso));
            double newT = 0, newS = 0;
            double s_os = 0.0, s_mm = 0.0, s_vv = 0.0;
            if (sums) {
                s_os = at(gp(M.ocn), ncell + oc);
                s_mm = at(gp(M.M), oc);
                if (l0 == 0) s_vv = at(gp(g.V), oc);
            }
            if (!sums || l0 != 0) s_vv = 0.0;
            // a tracer's new value joins the sums of its column (S in slot 1 of
            // the first block; without BIOGEM the factors are zero)
            auto add_sum = [&](int q, double nv) {
                if (q == 0) newT = nv;
                if (q == 1) {
                    newS = nv;
                    accS = ANOM ? __builtin_fma(nv + SALN0 + 0.0, s_vv, accS) : accS + (nv + SALN0 + 0.0) * s_vv;
                }
                const double lv = nv * s_os * rSold;
                accs[q] = ANOM ? __builtin_fma(lv, s_mm, accs[q]) : accs[q] + lv * s_mm;
            };
            // the level's tracers: every value of the cell above is in, so a
            // tracer is one run of instructions with no test but the store's
            auto tracers = [&](auto top_) {
                constexpr bool TOP = decltype(top_)::value;
                if constexpr (ANOM) {
#pragma clang fp contract(off)
                    // (the contractions are written out, so that every tile and
                    // mode rounds alike whatever else its blocks hold)
                    // FP32 form in coefficient form: each face flux is the
                    // neighbour difference times a coefficient of the cell, and the
                    // isoneutral flux a sum of corner differences times
                    // coefficients.  The face coefficients depend on the velocity,
                    // the diffusivities and the mask only: cgo_set_velocity forms
                    // them in FP64 and rounds each once (closed faces are zero)
                    auto fma_ = [](R a, R b, R c) -> R { return __builtin_fmaf(a, b, c); };
                    const R ce = at(u, oc), cw = at(u, ncell + oc);
                    const R cn = at(u, 2 * ncell + oc), cs = at(u, 3 * ncell + oc);
                    const R ca = at(u, 4 * ncell + oc), cbn = at(u, 5 * ncell + oc);
#pragma unroll
                    for (int q = 0; q < LB; q++) {
                        const R Tc = SP(cb, q, p);
                        const R dE = D(cb, q, pe, p), dW = D(cb, q, pw, p), dN = D(cb, q, pn, p), dS = D(cb, q, ps, p);
                        R fa = 0, fbn = 0;
                        // the top cell's surface flux enters in FP64: rounded to
                        // float it would bias every step's forcing alike
                        double incs = 0.0;
                        if constexpr (TOP) {
                            if (M.sflux && q < nl) {
                                const double fsurf = at(gp(M.sflux), (uint32_t)((l0 + q) * plane + col));
                                if (fsurf != 0.0) incs = -(gp(g.mk)[MK_DT * KS + k] * (fsurf * gp(g.mk)[MK_RDZ * KS + k]));
                            }
                        } else {
                            const R dU = DK(ub, cb, q, p);
                            // corner differences with the sign of the west/south
                            // corners folded into ax[0], ax[2], ay[0], ay[2]
                            R tv = fma_(ax[1], dE, ax[0] * dW);
                            tv = fma_(ay[0], dS, tv);
                            tv = fma_(ay[1], dN, tv);
                            tv = fma_(ax[2], D(ub, q, pw, p), tv);
                            tv = fma_(ax[3], D(ub, q, pe, p), tv);
                            tv = fma_(ay[2], D(ub, q, ps, p), tv);
                            tv = fma_(ay[3], D(ub, q, pn, p), tv);
                            tv = __uint_as_float(__float_as_uint(fma_(-qq, dU, tv)) & has_mix);
                            fa = fma_(dU, ca, tv);
                            fbn = fma_(dU, cbn, tv);
                        }
                        const R lat = fma_(ce, dE, -(cw * dW)) + fma_(cn, dN, -(cs * dS));
                        const R div = fma_(Tc, divu, fma_(fa - FB(q), rdz, lat));
                        const int idx = (l0 + q) * tstride + o + col;
                        const R inc = -(dt * div);
                        double nv;
                        if (lo_src) {
                            // compensated accumulation: the rounding residual of every
                            // update is carried to the next step in the int16 plane
                            nv = ((double)Tc + (double)SR(cb, q, p)) + (double)inc + incs;
                            if (own && q < nl) StateIO<R>::st((R*)dst, lo_dst, idx, nv);
                        } else {
                            const R v = Tc + (inc + (R)incs);
                            if (own && q < nl) at(dst, (uint32_t)idx) = v;
                            nv = (double)v;
                        }
                        if (SPLIT && own && nvs && q < nl) at(nvs, (uint32_t)idx) = nv;
                        FB(q) = fbn;
                        add_sum(q, nv);
                    }
                } else {
                    // a cell without the isoneutral flux has zero gradients here
                    const R dzr = iso ? (R)dzrho : (R)1, dz2 = dzr * dzr;
#pragma unroll
                    for (int q = 0; q < LB; q++) {
                        const R Tc = SP(cb, q, p), Te = SP(cb, q, nc.e), Tw = SP(cb, q, nc.w);
                        const R Tn = SP(cb, q, nc.n), Ts = SP(cb, q, nc.s);
                        const R fe = ue_ * rc * (((R)1.0 - upe) * Te + ((R)1.0 + upe) * Tc) * (R)0.5 - (Te - Tc) * rc2 * diff1;
                        const R fw = uw_ * rc * (((R)1.0 - upw) * Tc + ((R)1.0 + upw) * Tw) * (R)0.5 - (Tc - Tw) * rc2 * diff1;
                        const R fn = cvn * un_ * (((R)1.0 - upn) * Tn + ((R)1.0 + upn) * Tc) * (R)0.5 - cv2n * (Tn - Tc) * diff1;
                        const R fs = cvs * us_ * (((R)1.0 - ups) * Tc + ((R)1.0 + ups) * Ts) * (R)0.5 - cv2s * (Tc - Ts) * diff1;
                        R fa = 0;
                        if constexpr (TOP) {
                            if (M.sflux && q < nl) fa = (R)at(gp(M.sflux), (uint32_t)((l0 + q) * plane + col));
                        } else {
                            const R Tu = SP(ub, q, p);
                            fa = ua_ * (((R)1.0 - upa) * Tu + ((R)1.0 + upa) * Tc) * (R)0.5;
                            fa = fa - (Tu - Tc) * rdza * diffv;
                            const R dzts = (Tu - Tc) * rdza;
                            R tv = 0;
#pragma unroll
                            for (int n = 0; n < 4; n++) {
                                const int b = n < 2 ? cb : ub;
                                const bool east = n & 1;
                                const Nbr& m = n < 2 ? nc : nu;
                                const R dx = (east ? D(b, q, m.e, p) : D(b, q, p, m.w)) * rc * rdphi;
                                const R dy = east ? D(b, q, m.n, p) * cvn * rdsvn : D(b, q, p, m.s) * cvs * rdsvs;
                                tv = tv + ((R)2 * dzr * dx - dxr[n] * dzts) * dxr[n] + ((R)2 * dzr * dy - dyr[n] * dzts) * dyr[n];
                            }
                            // divided, not multiplied by a corrected reciprocal: that
                            // rounds alike only while its remainders are normal
                            // numbers (256 FP64 members 610 us a launch, 616 so)
                            const R fi = isoc * tv / dz2;
                            fa = fa + __hiloint2double(__double2hiint(fi) & has_iso, __double2loint(fi) & has_iso);
                        }
                        const R div = ((fe - fw) * rdphi + (fn - fs) * rds) + (fa - FB(q)) * rdz;
                        const int idx = (l0 + q) * tstride + o + col;
                        const R v = Tc - dt * div;
                        if (own && q < nl) at(dst, (uint32_t)idx) = v;
                        FB(q) = fa;
                        add_sum(q, (double)v);
                    }
                }
            };
            if (top)
                tracers(std::true_type{});
            else
                tracers(std::false_type{});
            if (l0 == 0 && own) {
                const double rn = eos<double>(g.ec[0], g.ec[1], g.ec[2], g.ec[3], newT, newS);
                at(rhop, oc) = rn;
                falls = falls & (k == k1c || rn < rlow);
                rlow = rn;
            }
        }
        if (FLUX_NBUF == 2) __syncthreads();  // plane k is read by every thread before it is replaced
        if (more) commit((k + 2) % FLUX_NBUF);
        __syncthreads();
    }
    if (!SPLIT && IM != 1 && l0 == 0) {
        // co's columns: this block's segment [w0, w1) of the member's list,
        // its unstable columns first, in column order
        constexpr int NW = FLUX_THREADS / 64;
        __shared__ int s_uns[NW];
        const int wv = tid >> 6;
        const uint64_t mu = __ballot(active && !falls), before = ((uint64_t)1 << (tid & 63)) - 1;
        if ((tid & 63) == 0) s_uns[wv] = __popcll(mu);
        __syncthreads();
        int pu = __popcll(mu & before), nu = 0;
#pragma unroll
        for (int q = 0; q < NW; q++) {
            if (q < wv) pu += s_uns[q];
            nu += s_uns[q];
        }
        if (active) gp(M.ulist)[w0 + (falls ? nu + tid - pu : pu)] = col;
        if (tid == 0) {
            gp(M.useg)[1 + 2 * B.x] = w0;
            gp(M.useg)[2 + 2 * B.x] = nu;
            if (B.x == 0) gp(M.useg)[0] = g.nfblk[V];
        }
    }
    if (IM != 2 && l0 == 0 && M.diso) {
        limps = wave_sum(limps);
        dmaxv = wave_max(dmaxv);
        if ((tid & 63) == 0) {
            if (limps) atomicAdd(&M.diag[0], limps);
            if (dmaxv > 0.0) atomic_max_pos(M.dmax, dmaxv);
        }
    }
    if (sums && active && k1c <= maxk) {
        const int slot = gp(g.cslot)[col];
        AS_GLOBAL double* cs = gp(M.colsum);
#pragma unroll
        for (int q = 0; q < LB; q++) {
            const int l = l0 + q;
            if (q >= nl) break;
            if (l == 1) cs[slot] = accS;
            else if (l >= 2) cs[(size_t)l * g.nwet + slot] = accs[q];
        }
    }
}

// Launch of k_flux over a batch: nt threads per block (128 or 256), lb
// tracers per block, nbuf level planes; with iso_split the isoneutral
// coefficients come from a pre-pass launch (IM 1) and the tracer blocks (IM 2)
// stage only their tracers.  part: 1 the pre-pass, 2 the tracer blocks, 3 both.  The tracer block, then the block width, then the
// ring shrink until the workgroup fits the LDS the device grants one block.
template <typename R>
void launch_flux_t(const MemberDev* t, const int32_t* l, int n, const FluxShape& fs, int maxL,
                   const FluxTile& tile, const FluxSplit& sp, int part, size_t lds_cap, hipStream_t s) {
    constexpr int es = sizeof(R);
    int lb = tile.lb, nt = tile.nt, nbuf = tile.nbuf;
    const int iso_split = tile.iso;
    if (sp.kc > 0) {
        if (!(part & 2) || fs.nblk[1] == 0) return;
        const dim3 grid(sp.nbx * ((fs.maxk + sp.kc - 1) / sp.kc), (maxL + 1) / 2, n);
        hipLaunchKernelGGL((k_flux<R, 2, 256, 2, 3>), grid, dim3(256), flux_lds_bytes(4, 2, es, 256, 2), s, t, l, sp);
        return;
    }
    if (nt != 256) nt = 128;
    if (nbuf != 2) nbuf = 3;
    auto bytes = [&](int ns, int b) { return flux_lds_bytes(ns, b, es, nt, nbuf); };
    auto slots = [&]() { return iso_split ? lb : lb + 2; };
    while (lb > 2 && bytes(slots(), lb) > lds_cap) lb = lb == 8 ? 6 : (lb == 6 ? 4 : 2);
    if (nt == 256 && bytes(slots(), lb) > lds_cap) nt = 128;
    if (nbuf == 3 && bytes(slots(), lb) > lds_cap) nbuf = 2;
    const int v = nt == 256;
    if (fs.nblk[v] == 0) return;
    const dim3 grid(fs.nblk[v], (maxL + lb - 1) / lb, n);
    const size_t lds = bytes(slots(), lb);
#define CGO_FLUX(LB_, NT_, NB_, IM_) \
    hipLaunchKernelGGL((k_flux<R, LB_, NT_, NB_, IM_>), grid, dim3(NT_), lds, s, t, l, sp)
#define CGO_FLUX_LB(NT_, NB_, IM_)                    \
    do {                                              \
        if (lb == 2) CGO_FLUX(2, NT_, NB_, IM_);      \
        else if (lb == 8) CGO_FLUX(8, NT_, NB_, IM_); \
        else if (lb == 6) CGO_FLUX(6, NT_, NB_, IM_); \
        else CGO_FLUX(4, NT_, NB_, IM_);              \
    } while (0)
    if (iso_split) {
        // the pre-pass: one block per column block, T and S staged
        const dim3 g1(fs.nblk[v], 1, n);
        if (part & 1) {
        const size_t lds1 = bytes(2, 2);
        if (nt == 256) {
            if (nbuf == 2) hipLaunchKernelGGL((k_flux<R, 2, 256, 2, 1>), g1, dim3(256), lds1, s, t, l, sp);
            else hipLaunchKernelGGL((k_flux<R, 2, 256, 3, 1>), g1, dim3(256), lds1, s, t, l, sp);
        } else {
            if (nbuf == 2) hipLaunchKernelGGL((k_flux<R, 2, 128, 2, 1>), g1, dim3(128), lds1, s, t, l, sp);
            else hipLaunchKernelGGL((k_flux<R, 2, 128, 3, 1>), g1, dim3(128), lds1, s, t, l, sp);
        }
        }
        if (!(part & 2)) {
        } else if (nt == 256) {
            if (nbuf == 2) CGO_FLUX_LB(256, 2, 2); else CGO_FLUX_LB(256, 3, 2);
        } else {
            if (nbuf == 2) CGO_FLUX_LB(128, 2, 2); else CGO_FLUX_LB(128, 3, 2);
        }
    } else if (!(part & 2)) {
        // no pre-pass: the tracer blocks compute their own coefficients
    } else if (nt == 256) {
        if (nbuf == 2) CGO_FLUX_LB(256, 2, 0); else CGO_FLUX_LB(256, 3, 0);
    } else {
        if (nbuf == 2) CGO_FLUX_LB(128, 2, 0); else CGO_FLUX_LB(128, 3, 0);
    }
#undef CGO_FLUX_LB
#undef CGO_FLUX
}

// co, goldstein.f90:2657-2777 (iconv = 0, ieos = 0): FP64 arithmetic on the
// new state in place.  Which levels mix depends on T and S alone, so the
// walk and the mixing of the other tracers are taken apart:
//
//   A  a thread per unstable column walks the reference's mixing loop on T, S
//      and density in LDS and writes down what it mixed: the list of
//      (level, thickness) terms of every mean, in the order they are added.
//      The segments are a bit mask of their top levels (the reference's kk
//      map holds the same tops, top to bottom), so a step of the walk reads
//      one density.
//   B  a thread per (unstable column, tracer) loads the tracer's column, all
//      its levels at once, replays the list on its own LDS copy, writes the
//      levels that changed and adds up the coupling's column sum.
//
// Every tracer's means are formed in the reference's order from the values
// the state would hold in between, so FP64 members keep the reference's bits.
// The columns come from the flux, which sees every column's new density and
// leaves them sorted into unstable and stable: a launch finds its work packed,
// and a stable ensemble's blocks read one count and end.
//
// Walking and mixing a column by four lanes together, each mean read from
// and written back to memory, was bound by that chain of round trips.  In a
// convecting state, per launch: 256 members of 36x36x16x24 FP32C 466 ->
// 116 us, six of 72x72x32x40 1,078 -> 100 us, one FP64 member 124 -> 18 us;
// every column stable (256 members): 11.9 -> 4.2 us.
constexpr int CO_NT = 256;
constexpr int CO_CB = 8;  // columns a block takes at a time: their walks share one wave
// LDS of a block: nt private tracer columns of KM levels (before that A's T,
// S, density and thickness of CO_CB <= nt / 4 columns), then the lists of up
// to 2 (KM - 1) terms of the columns
__host__ __device__ constexpr size_t co_lds_bytes(int nt, int KM) {
    return (size_t)nt * KM * 8 + (size_t)CO_CB * 2 * KM * (8 + 1) + (size_t)CO_CB * (8 + 3 * 4);
}
template <typename R>
__device__ __forceinline__ void co_columns(const MemberDev& M, const BlockXYZ& B, int total, int nseg, int KM,
                                           const FluxSplit& sp_) {
    constexpr int CB = CO_CB;
    extern __shared__ double co_lds[];
    const GridDev& g = M.g;
    const int nt = (int)blockDim.x, tid = (int)threadIdx.x;
    const int maxi = g.maxi, maxk = g.maxk, L = M.L;
    const bool every = sp_.kc > 0;  // after a flux split by levels: every wet column
    const AS_GLOBAL int32_t* useg = gp(M.useg);
    if (every && M.bgc && B.x == 0 && tid == 0) *gp(M.sfresh) = 1;
    const int par = *gp(M.parity);
    void* st = M.st[par ^ 1];
    int16_t* lo = M.lo[par ^ 1];
    const bool carry = lo != nullptr;
    const uint32_t plane = (uint32_t)g.ncol, tstride = (uint32_t)g.ncell;
    AS_GLOBAL double* rho = gp(M.rho);
    const int E = 2 * KM;                                   // terms a column's list holds
    double* const r = co_lds;                               // A: [level - 1][CB]
    double* const tp = r + (size_t)KM * CB;
    double* const sp = tp + (size_t)KM * CB;
    double* const dzm = sp + (size_t)KM * CB;
    double* const lw = co_lds + (size_t)nt * KM;            // the lists: thickness [E][CB],
    uint64_t* const ltops = reinterpret_cast<uint64_t*>(lw + (size_t)E * CB);  // the tops left
    int* const lcol = reinterpret_cast<int*>(ltops + CB);   // column, bottom level, terms
    int* const lk1 = lcol + CB;
    int* const lne = lk1 + CB;
    uint8_t* const llev = reinterpret_cast<uint8_t*>(lne + CB);  // level [E][CB], bit 7: last term of a mean
    // members with surface fluxes keep the top level's T and S as tstepo
    // leaves them (tsval_ocn, ssval_ocn of step_goldstein 427-430): the
    // next call of the fluxes reads them, whatever the coupling does after
    auto snap = [&](int f, int col, double x) {
        if (M.sw) gp(M.sw)[(size_t)f * plane + col] = x;
    };
    // the column at place p of the segments' unstable or stable parts
    auto place = [&](int p, bool stable) -> int {
        if (every) return gp(g.wetsorted)[p];
        for (int q = 0; q < nseg; q++) {
            const int w0 = useg[1 + 2 * q], nu = useg[2 + 2 * q];
            const int w1 = q + 1 < nseg ? useg[3 + 2 * q] : g.nwet;
            const int m = stable ? w1 - w0 - nu : nu;
            if (p < m) return gp(M.ulist)[w0 + (stable ? nu : 0) + p];
            p -= m;
        }
        return 0;
    };
    if (M.sw)
        for (int p = B.x * nt + tid; p < g.nwet - total; p += gridDim.x * nt) {
            const int col = place(p, true);
            const uint32_t top = (uint32_t)(maxk - 1) * plane + col;
            snap(SW_TSTAR, col, StateIO<R>::ld(st, lo, top));
            snap(SW_SSTAR, col, StateIO<R>::ld(st, lo, tstride + top));
        }
    for (int i0 = B.x * CB; i0 < total; i0 += gridDim.x * CB) {
        const int n = min(CB, total - i0);
        if (tid < n) {
            const int col = place(i0 + tid, false);
            lcol[tid] = col;
            lk1[tid] = k1at(g, col % maxi + 1, col / maxi + 1);
        }
        __syncthreads();
        for (int x = tid; x < n * maxk; x += nt) {
            const int i = x % n, k = x / n;
            if (k + 1 >= lk1[i]) {
                const uint32_t o = (uint32_t)k * plane + lcol[i];
                const auto a = StateIO<R>::ldr(st, lo, o), b = StateIO<R>::ldr(st, lo, tstride + o);
                r[k * CB + i] = at(rho, o);
                tp[k * CB + i] = StateIO<R>::val(a, carry);
                sp[k * CB + i] = StateIO<R>::val(b, carry);
                dzm[k * CB + i] = gp(g.mk)[MK_DZ * (maxk + 2) + k + 1];
            }
        }
        __syncthreads();
        // ---- A
        if (tid < n) {
            const int i = tid, k1 = lk1[i], col = lcol[i];
            const double e0 = g.ec[0], e1 = g.ec[1], e2 = g.ec[2], e3 = g.ec[3];
            auto R_ = [&](int k) -> double& { return r[(k - 1) * CB + i]; };
            auto T_ = [&](int k) -> double& { return tp[(k - 1) * CB + i]; };
            auto S_ = [&](int k) -> double& { return sp[(k - 1) * CB + i]; };
            auto W_ = [&](int k) -> double& { return dzm[(k - 1) * CB + i]; };
            auto below = [](uint64_t m, int k) -> int {  // the highest top under level k, 0 if none
                const uint64_t b = m & (((uint64_t)1 << k) - 1);
                return b ? 63 - __clzll((long long)b) : 0;
            };
            const uint64_t all = (((uint64_t)2 << maxk) - 1) & ~(((uint64_t)1 << k1) - 1);  // bits k1..maxk
            uint64_t tops = all;
            int km = maxk, lastmix = 0, ne = 0;
            double rk = R_(km);
            // every pass either moves or merges two segments, and it moves up
            // only once after a merge, so the loop ends within O(maxk^2) passes;
            // the cap only guards non-finite densities
            int guard = 4 * maxk * maxk + 64;
            for (int low = below(tops, km); (low > 0 || (lastmix != 0 && km != maxk)) && --guard > 0; low = below(tops, km)) {
                if (low == 0 || rk < R_(low)) {
                    if (lastmix == 0 || km == maxk)
                        km = low;
                    else
                        km = km + 1 + __builtin_ctzll(tops >> (km + 1));
                    lastmix = 0;
                    rk = R_(km);
                } else {
                    lastmix = 1;
                    // the thickness-weighted mean of the segments from km down
                    // through every one that is unstable against the next
                    double dsum = W_(km), tm = T_(km) * dsum, sm = S_(km) * dsum;
                    llev[ne * CB + i] = (uint8_t)km;
                    lw[ne * CB + i] = dsum;
                    ne++;
                    for (int q = low, nx;; q = nx) {
                        const double wq = W_(q);
                        dsum = dsum + wq;
                        tm = tm + T_(q) * wq;
                        sm = sm + S_(q) * wq;
                        tops &= ~((uint64_t)1 << q);
                        nx = below(tops, q);
                        const bool last = nx == 0 || !(R_(q) >= R_(nx));
                        llev[ne * CB + i] = (uint8_t)(q | (last ? 128 : 0));
                        lw[ne * CB + i] = wq;
                        ne++;
                        if (last) break;
                    }
                    tm = StateIO<R>::rt(tm / dsum, carry);
                    sm = StateIO<R>::rt(sm / dsum, carry);
                    T_(km) = tm;
                    S_(km) = sm;
                    W_(km) = dsum;
                    rk = eos<double>(e0, e1, e2, e3, tm, sm);
                    R_(km) = rk;
                }
            }
            if (guard <= 0) atomicAdd(&M.diag[3], 1);
            lne[i] = ne;
            ltops[i] = tops;
            // every level that is no segment's top takes its segment's density
            // (and, in B, its tracers); each such level counts as one convection
            const uint64_t fill = all & ~tops;
            double v = 0.0;
            for (int k = maxk; k >= k1; k--) {
                if ((tops >> k) & 1) v = R_(k);
                if (((fill | (fill << 1)) >> k) & 1) at(rho, (uint32_t)(k - 1) * plane + col) = v;
            }
            if (fill) gp(M.cost)[col] += (double)__popcll(fill);
        }
        __syncthreads();
        // ---- B
        double* const v = co_lds + tid;  // level k at v[(k - 1) * nt]
        const double rSold = M.bgc ? 1.0 / gp(M.scal)[SC_SMEAN] : 0.0;
        for (int x = tid; x < n * L; x += nt) {
            const int i = x % n, l = x / n;
            const int k1 = lk1[i], col = lcol[i], ne = lne[i];
            const uint64_t tops = ltops[i];
            if (ne == 0 && !(l >= 1 && M.bgc) && !(l < 2 && M.sw)) continue;
            const uint32_t base = (uint32_t)l * tstride + col;
            for (int k0 = k1; k0 <= maxk; k0 += 8) {
                typename StateIO<R>::Raw q[8];
#pragma unroll
                for (int u = 0; u < 8; u++)
                    if (k0 + u <= maxk) q[u] = StateIO<R>::ldr(st, lo, base + (uint32_t)(k0 + u - 1) * plane);
#pragma unroll
                for (int u = 0; u < 8; u++)
                    if (k0 + u <= maxk) v[(k0 + u - 1) * nt] = StateIO<R>::val(q[u], carry);
            }
            {
                double sum = 0.0, dsum = 0.0;
                int km = 0;  // the level a mean is written to, 0 before its first term
                for (int e = 0; e < ne; e++) {
                    const int lev = llev[e * CB + i], k = lev & 127;
                    const double wt = lw[e * CB + i], xv = v[(k - 1) * nt];
                    if (km == 0) {
                        km = k;
                        dsum = wt;
                        sum = xv * wt;
                    } else {
                        dsum = dsum + wt;
                        sum = sum + xv * wt;
                        if (lev & 128) {
                            v[(km - 1) * nt] = StateIO<R>::rt(sum / dsum, carry);
                            km = 0;
                        }
                    }
                }
            }
            const uint64_t all = (((uint64_t)2 << maxk) - 1) & ~(((uint64_t)1 << k1) - 1);
            const uint64_t fill = all & ~tops, chg = fill | (fill << 1);
            double sv = 0.0;
            for (int k = maxk; k >= k1; k--) {
                if ((tops >> k) & 1)
                    sv = v[(k - 1) * nt];
                else
                    v[(k - 1) * nt] = sv;
                if ((chg >> k) & 1) StateIO<R>::st(st, lo, base + (uint32_t)(k - 1) * plane, sv);
            }
            if (l < 2) snap(l == 0 ? SW_TSTAR : SW_SSTAR, col, v[(maxk - 1) * nt]);
            if (M.bgc && l >= 1) {
                // the coupling's column sums of this column after mixing and
                // fill-in, or those the flux leaves to this kernel: the FP32
                // form sums its new values before they are rounded, each
                // product added in one rounding
                const bool unr = sizeof(R) == 4 && ne == 0;
                const AS_GLOBAL double* nvs =
                    unr ? gp(sp_.nv) + (size_t)B.y * sp_.stride + base : nullptr;
                const uint32_t ncl = (uint32_t)g.ncell;
                double a = 0.0;
                for (int k0 = k1; k0 <= maxk; k0 += 4) {
                    double f0[4], f1[4], xv[4];
#pragma unroll
                    for (int u = 0; u < 4; u++)
                        if (k0 + u <= maxk) {
                            const uint32_t o = (uint32_t)(k0 + u - 1) * plane, c = o + col;
                            f0[u] = l == 1 ? at(gp(g.V), c) : at(gp(M.ocn), ncl + c);
                            f1[u] = l == 1 ? 0.0 : at(gp(M.M), c);
                            xv[u] = unr ? at(nvs, o) : v[(k0 + u - 1) * nt];
                        }
#pragma unroll
                    for (int u = 0; u < 4; u++)
                        if (k0 + u <= maxk) {
                            const double x1 = l == 1 ? xv[u] + SALN0 + 0.0 : xv[u] * f0[u] * rSold;
                            const double x2 = l == 1 ? f0[u] : f1[u];
                            a = unr ? __builtin_fma(x1, x2, a) : a + x1 * x2;
                        }
                }
                gp(M.colsum)[(size_t)(l == 1 ? 0 : l) * g.nwet + gp(g.cslot)[col]] = a;
            }
        }
        __syncthreads();  // the next columns' T, S and density take B's place
    }
}

// The step ends here: with `flip` the last of a member's blocks to finish turns
// its ping-pong parity, which the others have read by then, and counts the
// step.  As a launch of its own behind this one the flip took 5 us: 24 steps
// of sixteen 31x27x13x11 FP64 members 3,493 -> 3,432 us, 96 of 64 members of
// 36x36x16x24 44.1 -> 43.5 ms.
template <typename R>
__global__ __launch_bounds__(CO_NT) void k_co(const MemberDev* __restrict__ mems, const int32_t* __restrict__ list,
                                               int KM, FluxSplit sp, int flip) {
    const BlockXYZ B = xcd_blk();
    const MemberDev& M = mems[list[B.y]];
    const bool every = sp.kc > 0;
    const AS_GLOBAL int32_t* useg = gp(M.useg);
    const int nseg = every ? 0 : useg[0];
    int total = every ? M.g.nwet : 0;  // the member's columns
    for (int q = 0; q < nseg; q++) total += useg[2 + 2 * q];
    // the blocks that have columns (or, with surface fluxes, all); the first in any case
    const int nb = M.sw ? (int)gridDim.x : max(1, min((int)gridDim.x, (total + CO_CB - 1) / CO_CB));
    if (B.x >= nb) return;  // uniform for the block
    if (total > 0 || M.sw) co_columns<R>(M, B, total, nseg, KM, sp);
    __syncthreads();  // every wave of the block has read the parity
    if (!flip || threadIdx.x != 0) return;
    if (nb > 1) {
        if (atomicAdd(M.cofin, 1) != nb - 1) return;
        *gp(M.cofin) = 0;
    }
    *gp(M.parity) ^= 1;
    *gp(M.steps) += 1;
}

}  // namespace cgo
