// k_tstep_f64.hip -- FP64 instantiations of the GOLDSTEIN tracer-step
// kernels, the inventory reduction and the downloads' packing.  Built with
// -ffp-contract=off (see tstep_impl.h).
#include "tstep_impl.h"

namespace cgo {

void launch_flux64(const MemberDev* t, const int32_t* l, int n, const FluxShape& fs, int maxL,
                   const FluxTile& tile, const FluxSplit& sp, int part, size_t lds_cap, hipStream_t s) {
    launch_flux_t<double>(t, l, n, fs, maxL, tile, sp, part, lds_cap, s);
}

void launch_co(const MemberDev* t, const int32_t* l, int n, int nwetmax, int maxkmax, int prec, const FluxSplit& sp,
               bool flip, hipStream_t s) {
    // A large batch (more chunks of CO_CB columns than the chip holds blocks:
    // 4,096) runs one wave per block and up to four chunks per block, so that
    // blocks that find no unstable column are few; a small one runs every
    // chunk in a block of its own with more threads, so that a chunk's tracers
    // are mixed in fewer rounds.  256 members of 36x36x16x24 FP32C per step:
    // 1,175 us against 1,253 with 256 threads and one chunk per block (3.2
    // against 14.7 us for the launch where every column is stable); eight
    // members 201 against 206, one FP64 member 209 against 213.
    const int KM = maxkmax, chunks = (nwetmax + CO_CB - 1) / CO_CB;
    const bool large = (long long)chunks * n > 4096;
    int nt = large ? 64 : CO_NT;
    while (nt > 64 && co_lds_bytes(nt, KM) > 65536) nt /= 2;
    const dim3 grid(large ? (chunks + 3) / 4 : chunks, n);
    const size_t lds = co_lds_bytes(nt, KM);
    if (prec == 0)
        hipLaunchKernelGGL(k_co<double>, grid, dim3(nt), lds, s, t, l, KM, sp, (int)flip);
    else
        hipLaunchKernelGGL(k_co<float>, grid, dim3(nt), lds, s, t, l, KM, sp, (int)flip);
}

// Per-tracer volume-weighted sum over the member's current state, one block
// per tracer.  A thread adds every 256th cell, one chain in order; the loads of
// INV_U cells are issued before any of them is added, where each add waited for
// its own.  One call (the sums in pinned memory, out, in place of a device
// buffer copied back): 256 members of 36x36x16x24 FP32C in turn 84 -> 30 us
// each, 64 FP64 members 53 -> 27, 72x72x32x40 333 -> 89.
constexpr int INV_U = 16;
template <typename R>
__global__ __launch_bounds__(256) void k_inventory(const MemberDev* __restrict__ mems, int32_t m, double* out,
                                                   const double* __restrict__ w) {
    const MemberDev& M = mems[m];
    const int l = blockIdx.x;
    const int par = *gp(M.parity);
    const uint32_t ncell = M.g.ncell, base = (uint32_t)l * ncell;
    const AS_GLOBAL R* st = gp((const R*)M.st[par]);
    const AS_GLOBAL int16_t* lo = sizeof(R) == 4 && M.lo[par] ? gp(M.lo[par]) : nullptr;
    double s = 0.0;
    for (uint32_t c0 = threadIdx.x; c0 < ncell; c0 += 256 * INV_U) {
        R h[INV_U];
        int16_t cy[INV_U];
        double wc[INV_U];
#pragma unroll
        for (int q = 0; q < INV_U; q++) {
            const uint32_t c = c0 + 256 * q;
            const bool in = c < ncell;
            wc[q] = in ? at(gp(w), c) : 0.0;
            h[q] = at(st, base + (in ? c : c0));
        }
        if (lo) {  // one test for all, so that the carries' loads stay together
#pragma unroll
            for (int q = 0; q < INV_U; q++) cy[q] = at(lo, base + (c0 + 256 * q < ncell ? c0 + 256 * q : c0));
        }
#pragma unroll
        for (int q = 0; q < INV_U; q++) {
            double v = (double)h[q];
            if constexpr (sizeof(R) == 4)
                if (lo) v += (double)cy[q] * carry_unit(h[q]);
            s = wc[q] != 0.0 ? s + v * wc[q] : s;
        }
    }
    __shared__ double red[256];
    red[threadIdx.x] = s;
    __syncthreads();
    for (int h = 128; h > 0; h >>= 1) {
        if (threadIdx.x < h) red[threadIdx.x] += red[threadIdx.x + h];
        __syncthreads();
    }
    if (threadIdx.x == 0) out[l] = red[0];
}

void launch_inventory(const MemberDev* t, int32_t m, int L, double* out, const double* w, int prec, hipStream_t s) {
    // one block per tracer
    if (prec == 0)
        hipLaunchKernelGGL(k_inventory<double>, dim3(L), dim3(256), 0, s, t, m, out, w);
    else
        hipLaunchKernelGGL(k_inventory<float>, dim3(L), dim3(256), 0, s, t, m, out, w);
}

// Cells [c0, c0 + nc) of planes [L][ncell] as rows of L doubles, the order the
// host takes them in (go_ts(maxl, ...)), into pinned host memory: a block
// turns CT cells around in LDS (an odd stride, so that neither side
// meets a bank twice), reads whole lines of every plane and writes one
// contiguous range.  A piece of 1 MiB takes 28 us (37 GB/s into host memory);
// the host's copy of it out of the staging, ~35 us, bounds a download.  FP32
// states are decoded as the host did it: float plus carry times 2^-16 ulp, the
// ulp of an infinity infinite (an infinite value comes out NaN where its carry
// is zero).
template <typename R, uint32_t CT>
__global__ __launch_bounds__(256) void k_pack(PackSrc p, uint32_t c0, uint32_t nc, double* __restrict__ out) {
    extern __shared__ __align__(16) double tile[];  // [L][CT + 1]
    const int q = p.parity ? *gp(p.parity) : 0;
    const AS_GLOBAL R* st = gp((const R*)p.st[q]);
    const AS_GLOBAL int16_t* lo = p.lo[q] ? gp(p.lo[q]) : nullptr;
    const uint32_t b0 = blockIdx.x * CT, n = min(CT, nc - b0), L = p.L;
    for (uint32_t i = threadIdx.x; i < L * CT; i += 256) {
        const uint32_t l = i / CT, c = i % CT;
        if (c >= n) continue;
        const uint32_t s = l * p.ncell + c0 + b0 + c;
        double v;
        if constexpr (sizeof(R) == 8) {
            v = at(st, s);
        } else {
            const float h = at(st, s);
            const double unit = (__float_as_uint(h) << 1) == 0xff000000u ? (double)INFINITY : carry_unit(h);
            v = (double)h + (lo ? (double)at(lo, s) : 0.0) * unit;
        }
        tile[l * (CT + 1) + c] = v;
    }
    __syncthreads();
    AS_GLOBAL double* o = gp(out) + (size_t)b0 * L;
    for (uint32_t i = threadIdx.x; i < n * L; i += 256) o[i] = tile[(i % L) * (CT + 1) + i / L];
}

template <typename R, uint32_t CT>
static void launch_pack_ct(const PackSrc& p, uint32_t c0, uint32_t nc, double* out, hipStream_t s) {
    hipLaunchKernelGGL((k_pack<R, CT>), dim3((nc + CT - 1) / CT), dim3(256), (size_t)p.L * (CT + 1) * 8, s, p, c0, nc, out);
}

void launch_pack(const PackSrc& p, int prec, uint32_t c0, uint32_t nc, double* out, hipStream_t s) {
    // 64 cells a block while their rows fit 64 KiB of LDS, else 16 (35 KB for 256 tracers)
    const bool wide = p.L <= 126;
    if (prec == 0)
        (wide ? launch_pack_ct<double, 64> : launch_pack_ct<double, 16>)(p, c0, nc, out, s);
    else
        (wide ? launch_pack_ct<float, 64> : launch_pack_ct<float, 16>)(p, c0, nc, out, s);
}

}  // namespace cgo
