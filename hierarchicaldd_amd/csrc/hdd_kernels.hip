// HIP kernels for gfx950: matrix-free V-cycle on paged SPGrid levels and the
// outer PCG vector operations.
//
// Launch shapes: the smoothing sweep and the residual take one 64-lane
// wavefront per 4x8x8 page, four cells per lane with 16-byte accesses (see
// Stencil4); the other page kernels one 256-thread workgroup per page, thread
// t owning cell t (t = x*64 + y*8 + z), so every channel access of a wavefront
// is a contiguous, coalesced segment. Face neighbours inside a page are at
// cell offsets +-64, +-8, +-1; across the page face they come from the page's
// 6-entry neighbour table (the zero page `np` stands in for unallocated pages).
//
// Floating-point order reproduces the reference kernels operation by
// operation (the library is compiled with -ffp-contract=off):
//   residual   r = b - sum_f -(u_n - u_c)   LIB/SPGrid_Residual_Legacy.h:52-61
//   correction u += (omega/fc) * r          LIB/SPGrid_Correction_Legacy.h:60-77
//   restriction / prolongation weights      LIB/SPGrid_Restriction_Legacy.h:50-181,
//                                           LIB/SPGrid_Prolongation_Legacy.h:48-123
//   PCG Laplace (double accumulation)       DDS/SPGrid_Gemini_Arithmetic_Helpers.h:240-262
#include <hip/hip_runtime.h>
#include <hip/hip_fp16.h>
#include <algorithm>
#include <atomic>
#include <cstdint>
#include <mutex>
#include "hdd_device.h"

namespace hdd {

__constant__ float c_omega_fc[8];   // (float)(2/3) / (float)fc, fc = 0..6
__constant__ float c_rweights[64];  // restriction weights, [i][j][k] with w = {1,3,3,1}/8
__constant__ float c_pweights[8];   // prolongation weights 4 * {3/4,1/4}^3, [i][j][k]

// Workgroups are dealt to the 8 XCDs round-robin (workgroup i runs on XCD
// i mod 8), and each XCD has its own L2. Giving XCD x the contiguous page range
// [x*chunk, (x+1)*chunk) keeps Morton neighbours, whose halo cells a stencil
// re-reads, in the same L2. Launch with kXcds * chunk workgroups; ids past np
// return.
constexpr int kXcds = 8;
__host__ __device__ inline int xcd_chunk(int np) { return (np + kXcds - 1) / kXcds; }
__device__ __forceinline__ int xcd_page(int np) {
    return (int)(blockIdx.x % kXcds) * xcd_chunk(np) + (int)(blockIdx.x / kXcds);
}

__device__ __forceinline__ bool page_stopped(const DevLevel& L, int p) { return L.active && !L.active[L.prob[p]]; }

__device__ __forceinline__ int nb_index(const int* __restrict__ nbr, int p, int c, int f) {
    switch (f) {
        case 0: return (c >= 64) ? p * 256 + c - 64 : nbr[p * 6 + 0] * 256 + c + 192;
        case 1: return (c < 192) ? p * 256 + c + 64 : nbr[p * 6 + 1] * 256 + c - 192;
        case 2: return ((c & 56) != 0) ? p * 256 + c - 8 : nbr[p * 6 + 2] * 256 + c + 56;
        case 3: return ((c & 56) != 56) ? p * 256 + c + 8 : nbr[p * 6 + 3] * 256 + c - 56;
        case 4: return ((c & 7) != 0) ? p * 256 + c - 1 : nbr[p * 6 + 4] * 256 + c + 7;
        default: return ((c & 7) != 7) ? p * 256 + c + 1 : nbr[p * 6 + 5] * 256 + c - 7;
    }
}

// V-cycle storage: float, or half (FP16 storage, FP32 arithmetic: values are
// widened on load and rounded to nearest on store).
__device__ __forceinline__ float ld(const float* __restrict__ p, size_t i) { return p[i]; }
__device__ __forceinline__ float ld(const __half* __restrict__ p, size_t i) { return __half2float(p[i]); }
__device__ __forceinline__ void st(float* __restrict__ p, size_t i, float v) { p[i] = v; }
__device__ __forceinline__ void st(__half* __restrict__ p, size_t i, float v) { p[i] = __float2half_rn(v); }
// v as a store and load through the storage type would give it
__device__ __forceinline__ float stored(const float*, float v) { return v; }
__device__ __forceinline__ float stored(const __half*, float v) { return __half2float(__float2half_rn(v)); }

// Stencil sweeps: one 64-lane wavefront per page, lane l owns the four cells
// 4l .. 4l+3 (z = 4(l&1) .. +3 of row x = l>>4, y = (l>>1)&7) and moves them
// with one 16-byte access per channel (8 bytes with FP16 storage). Face
// neighbours inside the page are the vectors of lanes l+-16 (x) and l+-2 (y)
// and the neighbouring elements (z); across a page face they come from the
// page's 6-entry neighbour table (the zero page `np` stands in for unallocated
// pages). Four pages per 256-thread workgroup (the sweep: eight per 512).
struct V4 { float v[4]; };
__device__ __forceinline__ V4 ld4(const float* __restrict__ p, size_t i4) {
    const float4 t = reinterpret_cast<const float4*>(p)[i4];
    return {{t.x, t.y, t.z, t.w}};
}
__device__ __forceinline__ V4 ld4(const __half* __restrict__ p, size_t i4) {
    const uint2 t = reinterpret_cast<const uint2*>(p)[i4];
    __half2 a, b;
    __builtin_memcpy(&a, &t.x, 4);
    __builtin_memcpy(&b, &t.y, 4);
    const float2 fa = __half22float2(a), fb = __half22float2(b);
    return {{fa.x, fa.y, fb.x, fb.y}};
}
__device__ __forceinline__ void st4(float* __restrict__ p, size_t i4, const V4& v) {
    reinterpret_cast<float4*>(p)[i4] = make_float4(v.v[0], v.v[1], v.v[2], v.v[3]);
}
__device__ __forceinline__ void st4(__half* __restrict__ p, size_t i4, const V4& v) {
    const __half2 a = __floats2half2_rn(v.v[0], v.v[1]), b = __floats2half2_rn(v.v[2], v.v[3]);
    uint2 t;
    __builtin_memcpy(&t.x, &a, 4);
    __builtin_memcpy(&t.y, &b, 4);
    reinterpret_cast<uint2*>(p)[i4] = t;
}

// The four cells of lane l of page p with their six face neighbours, and the
// float residual of each, in the reference operation order
// (r = b - sum over set face bits (-x,+x,-y,+y,-z,+z) of -(u_n - u_c),
// LIB/SPGrid_Residual_Legacy.h:52-61). Neighbour values are loaded whether or
// not their face bit is set (every address is valid) and selected afterwards.
template <class S>
struct Stencil4 {
    V4 uc, r;
    uint32_t f[4];  // DevLevel::kinds
    __device__ __forceinline__ Stencil4(const DevLevel& L, int p, int l, const S* __restrict__ u, const S* __restrict__ b) {
        const int x = l >> 4, y = (l >> 1) & 7, zh = l & 1;
        const int* nb = L.nbr + p * 6;
        const size_t base = (size_t)p * 64;
        const uint32_t fv = reinterpret_cast<const uint32_t*>(L.kinds)[base + l];
#pragma unroll
        for (int k = 0; k < 4; ++k) f[k] = fv >> (8 * k) & 0xffu;
        uc = ld4(u, base + l);
        const V4 xm = ld4(u, x > 0 ? base + l - 16 : (size_t)nb[0] * 64 + l + 48);
        const V4 xp = ld4(u, x < 3 ? base + l + 16 : (size_t)nb[1] * 64 + l - 48);
        const V4 ym = ld4(u, y > 0 ? base + l - 2 : (size_t)nb[2] * 64 + l + 14);
        const V4 yp = ld4(u, y < 7 ? base + l + 2 : (size_t)nb[3] * 64 + l - 14);
        const float zm = ld(u, zh ? (size_t)p * 256 + 4 * l - 1 : (size_t)nb[4] * 256 + 4 * l + 7);
        const float zp = ld(u, zh ? (size_t)nb[5] * 256 + 4 * l - 4 : (size_t)p * 256 + 4 * l + 4);
        const V4 bv = ld4(b, base + l);
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            const float cv = uc.v[k];
            const float nv[6] = {xm.v[k], xp.v[k], ym.v[k], yp.v[k], k > 0 ? uc.v[k - 1] : zm, k < 3 ? uc.v[k + 1] : zp};
            float result = 0.f;
#pragma unroll
            for (int q = 0; q < 6; ++q)
                if (f[k] >> q & 1u) result -= (nv[q] - cv);
            r.v[k] = bv.v[k] - result;
        }
    }
};

__host__ __device__ inline int page_groups(int np) { return (np + 3) >> 2; }
// the sweep takes eight pages per 512-thread workgroup (measured 1.7% faster than four at 256^3)
constexpr int kSweepPages = 8;
__host__ __device__ inline int sweep_groups(int np) { return (np + kSweepPages - 1) / kSweepPages; }

// One damped-Jacobi sweep (residual + correction fused, ping-pong buffers);
// u += (omega / face count) r on the selected cells
// (LIB/SPGrid_Correction_Legacy.h:60-77), other cells copied unchanged.
// kAgain: u_out already holds the cells that this kind of sweep leaves alone (it is
// the iterate before u_in), so lanes without a cell to write are done: at 32^3
// subdomains a third of the lines. Bound by memory: 13 bytes a cell, of which one is
// the kinds (the flags' four made it 16). 256^3: 55 us a sweep with flags, 46 with
// kinds, 37 again (the same card).
template <class S, bool kAgain>
__global__ void __launch_bounds__(64 * kSweepPages) k_smooth(DevLevel L, const S* __restrict__ u_in, S* __restrict__ u_out,
                                                             const S* __restrict__ b, uint32_t interior, uint32_t boundary) {
    const int ng = sweep_groups(L.np), gi = xcd_page(ng), l = threadIdx.x & 63;
    const int p = gi * kSweepPages + (int)(threadIdx.x >> 6);
    if (gi >= ng || p >= L.np || page_stopped(L, p)) return;
    // a kind is written when its Active and Boundary bits are `interior` or `boundary` (0: none)
    auto written = [&](uint32_t f) {
        const uint32_t sel = f & (kKindActive | kKindBoundary);
        return sel && (sel == interior || sel == boundary);
    };
    if (kAgain) {
        const uint32_t fv = reinterpret_cast<const uint32_t*>(L.kinds)[(size_t)p * 64 + l];
        if (!written(fv & 0xffu) && !written(fv >> 8 & 0xffu) && !written(fv >> 16 & 0xffu) && !written(fv >> 24)) return;
    }
    const Stencil4<S> st(L, p, l, u_in, b);
    V4 out;
#pragma unroll
    for (int k = 0; k < 4; ++k) {
        const uint32_t f = st.f[k];
        float u = st.uc.v[k];
        if (written(f)) u += c_omega_fc[__popc(f & kKindFaces)] * st.r.v[k];
        out.v[k] = u;
    }
    st4(u_out, (size_t)p * 64 + l, out);
}

// Several sweeps of a level in one launch, and the residual after them, where
// its Active cells couple only within small clusters (the coarse levels: a
// cluster is the part of a subdomain, or of a few that meet inside an obstacle).
// A workgroup holds whole clusters in LDS, C cells per thread (cell i of thread
// t: slot i * blockDim + t), and sweeps them with the operations of Stencil4 and
// k_smooth, keeping every iterate in the level's storage type, so the result is
// bit-identical to one launch per sweep. nbr gives each cell's face neighbours as
// LDS values; a neighbour outside the workgroup is a cell no sweep writes, held
// in the halo behind the slots. Where a face bit is not set it names the cell
// itself, whose difference is an exact zero while the cell is finite (an infinite
// one becomes NaN, as the next sweep of it makes of it in any case: its set faces
// give inf - inf). The cells ping-pong between two
// copies (the halo is in both), one barrier per sweep. u is updated in place: no
// other workgroup reads the Active cells of this one's clusters.
//
// Bound by instruction issue and the barrier: a sweep is 6 LDS reads, about 25
// operations and one write per cell, against a launch of 3.3-5 us per sweep of a
// small level. The seven sweeps and the residual of a level take 4.7 us at 343 cells
// a cluster, 13 us at 3375 to 4096 (eight launches: 35-46 us); 200 sweeps of clusters
// of up to 343 cells 28 us. Cells, not pages, make up a cluster: by pages, the 16^3
// clusters of a 100^3 domain's level 1 lie in 46 pages and did not fit, and its
// bottom clusters filled 2048 slots (76 us for the 200 sweeps).
template <class S, int C>
__global__ void __launch_bounds__(1024) k_cluster_sweeps(DevLevel L, DevClusters W, S* u, const S* __restrict__ b, S* __restrict__ r,
                                                         SweepPhases ph, int u_zero) {
    extern __shared__ __align__(16) unsigned char cluster_lds[];
    S* us = reinterpret_cast<S*>(cluster_lds);
    const int wg = blockIdx.x, nt = blockDim.x, cells = W.slots;
    float cur[C], bv[C], wgt[C];
    unsigned nb[C][3];    // LDS values of the six face neighbours, two per register
    unsigned kind = 0;    // two bits per cell: kSweepInterior, kSweepBoundary, 0 (never swept)
    // cell i's place in the level, -1 in an empty slot or a stopped problem's page
    auto place = [&](int i) {
        const int e = W.cell[wg * cells + i * nt + (int)threadIdx.x];
        return e >= 0 && !page_stopped(L, e >> 8) ? e : -1;
    };
#pragma unroll
    for (int i = 0; i < C; ++i) {
        const int ci = i * nt + (int)threadIdx.x, e = place(i);
        const uint16_t* q = W.nbr + (size_t)wg * 6 * cells + ci;
#pragma unroll
        for (int f = 0; f < 3; ++f) nb[i][f] = (unsigned)q[(size_t)(2 * f) * cells] | (unsigned)q[(size_t)(2 * f + 1) * cells] << 16;
        cur[i] = bv[i] = wgt[i] = 0.f;
        if (e >= 0) {
            const uint32_t fl = L.flags[e], sel = fl & (kActive | kBoundary);
            if (sel == kActive) kind |= (unsigned)kSweepInterior << (2 * i);
            if (sel == (kActive | kBoundary)) kind |= (unsigned)kSweepBoundary << (2 * i);
            wgt[i] = c_omega_fc[__popc(fl & (0x3fu * kFaceMX))];
            bv[i] = ld(b, e);
            if (!u_zero) cur[i] = ld(u, e);
        }
        st(us, ci, cur[i]);
        st(us, W.entries + ci, cur[i]);
    }
    if (r && W.rest) {  // a share of the level's cells
        const int n = L.np * kPageCells, share = (n + W.nwg - 1) / W.nwg, end = min(n, (wg + 1) * share);
#pragma unroll 8
        for (int c = wg * share + (int)threadIdx.x; c < end; c += nt)
            if (!(L.flags[c] & kActive) && !page_stopped(L, c >> 8)) st(r, c, 0.f);
    }
    const int h0 = W.halo_ptr[wg], nh = W.halo_ptr[wg + 1] - h0;
    for (int h = threadIdx.x; h < nh; h += nt) {
        const float v = u_zero ? 0.f : ld(u, W.halo_cell[h0 + h]);
        st(us, cells + h, v);
        st(us, W.entries + cells + h, v);
    }
    __syncthreads();
    int from = 0;  // the copy that holds the current iterate: 0, or W.entries
    auto residual = [&](int i, int at) {
        float result = 0.f;
        const S* v = us + at;
#pragma unroll
        for (int f = 0; f < 3; ++f) {
            result -= (ld(v, nb[i][f] & 0xffffu) - cur[i]);
            result -= (ld(v, nb[i][f] >> 16) - cur[i]);
        }
        return bv[i] - result;
    };
    const bool any = __ballot(kind != 0) != 0;  // a wavefront without Active cells only keeps the barriers
    for (int k = 0; k < ph.n; ++k) {
        const unsigned sel = kind & ((unsigned)ph.cells[k] * 0x55555555u);
        for (int it = 0; it < ph.count[k]; ++it) {
            const int to = W.entries - from;
            if (any) {
#pragma unroll
                for (int i = 0; i < C; ++i) {
                    // many cells per thread: the neighbours stay packed (unpacked ahead of the loop they would spill)
                    if (C > 4) asm volatile("" : "+v"(nb[i][0]), "+v"(nb[i][1]), "+v"(nb[i][2]));
                    const float v = stored(us, cur[i] + wgt[i] * residual(i, from));
                    cur[i] = (sel >> (2 * i)) & 3u ? v : cur[i];
                    st(us, to + i * nt + (int)threadIdx.x, cur[i]);
                }
            }
            __syncthreads();
            from = to;
        }
    }
#pragma unroll
    for (int i = 0; i < C; ++i) {
        const int e = place(i);
        if (e < 0) continue;
        st(u, e, cur[i]);
        if (r) st(r, e, residual(i, from));
    }
}

// k_cluster_sweeps where a workgroup is one wavefront with a cell per lane (clusters of up to 64 cells:
// the bottom levels) and the cells around it hold zero: the neighbours come from the lanes' registers
// (ds_bpermute), so a sweep has no LDS write and no barrier in its chain. The 200 sweeps of a bottom
// level take 18 us instead of 28 (21 with a mask on every neighbour and a branch per sweep).
template <class S>
__global__ void __launch_bounds__(64) k_cluster_wave(DevLevel L, DevClusters W, S* u, const S* __restrict__ b, S* __restrict__ r, SweepPhases ph,
                                                     int u_zero) {
    const int wg = blockIdx.x, lane = threadIdx.x;
    int e = W.cell[wg * 64 + lane];
    int from[6], keep[6];  // the neighbour's lane as ds_bpermute wants it; 0 for a cell outside, whose value is zero
#pragma unroll
    for (int f = 0; f < 6; ++f) {
        const int v = W.nbr[(size_t)wg * 6 * 64 + f * 64 + lane];
        from[f] = (v & 63) * 4;
        keep[f] = v < 64 ? -1 : 0;
    }
    if (e >= 0 && page_stopped(L, e >> 8)) e = -1;
    float cur = 0.f, bv = 0.f, wgt = 0.f;
    int kind = 0;
    if (e >= 0) {
        const uint32_t fl = L.flags[e];
        kind = fl & kBoundary ? kSweepBoundary : kSweepInterior;
        wgt = c_omega_fc[__popc(fl & (0x3fu * kFaceMX))];
        bv = ld(b, e);
        if (!u_zero) cur = ld(u, e);
    }
    // a lane without a cell holds zero: where there is one, it stands for the cells outside
    const unsigned long long empty = __ballot(e < 0);
    const int zero = empty ? __ffsll((long long)empty) - 1 : 0;
    if (empty) {
#pragma unroll
        for (int f = 0; f < 6; ++f) {
            if (!keep[f]) from[f] = zero * 4;
            keep[f] = -1;
        }
    }
    auto residual = [&](bool masked) {
        float n[6], result = 0.f;
#pragma unroll
        for (int f = 0; f < 6; ++f) {
            const int v = __builtin_amdgcn_ds_bpermute(from[f], __float_as_int(cur));
            n[f] = __int_as_float(masked ? v & keep[f] : v);
        }
#pragma unroll
        for (int f = 0; f < 6; ++f) result -= (n[f] - cur);
        return bv - result;
    };
    auto sweeps = [&](bool masked) {
        for (int k = 0; k < ph.n; ++k) {
            const bool sel = (kind & ph.cells[k]) != 0;
#pragma unroll 4
            for (int it = 0; it < ph.count[k]; ++it) {
                const float v = stored(u, cur + wgt * residual(masked));
                cur = sel ? v : cur;
            }
        }
    };
    if (empty) sweeps(false);
    else sweeps(true);
    const float res = residual(true);
    if (e < 0) return;
    st(u, e, cur);
    if (r) st(r, e, res);
}

// residual at Active cells; other cells of r are written 0 (the value they
// always hold: only this kernel writes r, and the reference clears it before
// each V-cycle, DDS/SPGrid_Domain_Decomposition_Preconditioner.h:93,120)
template <class S>
__global__ void __launch_bounds__(256) k_residual(DevLevel L, const S* __restrict__ u, const S* __restrict__ b,
                                                  S* __restrict__ r) {
    const int ng = page_groups(L.np), gi = xcd_page(ng), l = threadIdx.x & 63;
    const int p = gi * 4 + (int)(threadIdx.x >> 6);
    if (gi >= ng || p >= L.np || page_stopped(L, p)) return;
    const Stencil4<S> st(L, p, l, u, b);
    V4 out;
#pragma unroll
    for (int k = 0; k < 4; ++k) out.v[k] = (st.f[k] & kKindActive) ? st.r.v[k] : 0.f;
    st4(r, (size_t)p * 64 + l, out);
}

template <class S>
__global__ void k_fill(S* __restrict__ a, float v, size_t n) {
    size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    for (; i < n; i += (size_t)gridDim.x * blockDim.x) st(a, i, v);
}
__global__ void k_copy(float* __restrict__ d, const float* __restrict__ s, size_t n) {
    size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    for (; i < n; i += (size_t)gridDim.x * blockDim.x) d[i] = s[i];
}

// page of block (bx, by, bz) of a level (the zero page outside the block box or where none is allocated)
__device__ __forceinline__ int lut_block(const DevLevel& L, int bx, int by, int bz) {
    if (bx < 0 || by < 0 || bz < 0 || bx >= L.nbx || by >= L.nby || bz >= L.nbz) return L.np;
    const int q = L.lut[(bx * L.nby + by) * L.nbz + bz];
    return q < 0 ? L.np : q;
}

// coarse b = sum_{4x4x4} w r_fine over fine cells 2c-2 .. 2c+1 (Active coarse cells only).
// The stencils of a coarse page (origin o) reach the fine region 2o-2 .. 2o+7
// in x and 2o-2 .. 2o+15 in y and z (10 x 18 x 18 cells in 3 x 3 x 3 fine
// blocks): its pages are looked up once and the region is staged in LDS
// once, so each fine value is read from memory once instead of by up to 8
// stencils; every stencil then sums the same values in the same order.
template <class S>
__global__ void __launch_bounds__(256) k_restrict(DevLevel F, DevLevel C, const S* __restrict__ r_f, S* __restrict__ b_c) {
    constexpr int RX = 10, RY = 18, RZ = 18;
    __shared__ int tab[27];
    __shared__ float sr[RX * RY * RZ];
    const int p = xcd_page(C.np), c = threadIdx.x, e = p * 256 + c;
    if (p >= C.np || page_stopped(C, p)) return;  // uniform over the workgroup
    const uint32_t fl = C.flags[e];  // the cell's own load goes out before the staging's
    const int ox = C.base[p * 3 + 0], oy = C.base[p * 3 + 1], oz = C.base[p * 3 + 2];
    const int X0 = 2 * ox - 2, Y0 = 2 * oy - 2, Z0 = 2 * oz - 2;
    const int bx0 = X0 >> 2, by0 = Y0 >> 3, bz0 = Z0 >> 3;
    if (c < 27) tab[c] = lut_block(F, bx0 + c / 9, by0 + (c / 3) % 3, bz0 + c % 3);
    __syncthreads();
    constexpr int N = (RX * RY * RZ + 255) / 256;
    float v[N];
#pragma unroll
    for (int i = 0; i < N; ++i) {  // all of a thread's loads in flight (one at a time: 7.7 us at 64^3, now 4.9)
        const int t = min(c + i * 256, RX * RY * RZ - 1);
        const int X = X0 + t / (RY * RZ), Y = Y0 + (t / RZ) % RY, Z = Z0 + t % RZ;
        const int q = tab[((X >> 2) - bx0) * 9 + ((Y >> 3) - by0) * 3 + ((Z >> 3) - bz0)];
        v[i] = ld(r_f, q * 256 + ((X & 3) << 6 | (Y & 7) << 3 | (Z & 7)));
    }
#pragma unroll
    for (int i = 0; i < N; ++i)
        if (c + i * 256 < RX * RY * RZ) sr[c + i * 256] = v[i];
    __syncthreads();
    if (!(fl & kActive)) return;
    const int lx = 2 * (c >> 6), ly = 2 * ((c >> 3) & 7), lz = 2 * (c & 7);  // stencil origin in the region
    float acc = 0.f;
    for (int i = 0; i < 4; ++i)
        for (int j = 0; j < 4; ++j)
            for (int k = 0; k < 4; ++k)
                acc += c_rweights[i * 16 + j * 4 + k] * sr[((lx + i) * RY + (ly + j)) * RZ + (lz + k)];
    st(b_c, e, acc);
}

// fine u += sum_{2x2x2} w u_coarse (Active fine cells only). The coarse cells
// a fine page (origin o) reads form the region o/2 .. o/2+2 (x) and
// o/2 .. o/2+4 (y, z), 3 x 5 x 5 cells in 2 x 2 x 2 coarse blocks: its pages
// are looked up once and the region is staged in LDS once per page. A wavefront
// per page, four cells per lane as in the sweeps, and no workgroup barrier:
// bound by the chain origin, page, coarse value, so by the pages in flight (a
// workgroup per page, a cell per thread: 85 us at 256^3, now 47).
template <class S>
__global__ void __launch_bounds__(256) k_prolong(DevLevel F, DevLevel C, S* __restrict__ u_f, const S* __restrict__ u_c) {
    constexpr int RX = 3, RY = 5, RZ = 5;
    __shared__ float staged[4][RX * RY * RZ + 1];
    const int ng = page_groups(F.np), gi = xcd_page(ng), l = threadIdx.x & 63;
    const int p = gi * 4 + (int)(threadIdx.x >> 6);
    if (gi >= ng || p >= F.np || page_stopped(F, p)) return;
    float* su = staged[threadIdx.x >> 6];
    const size_t at = (size_t)p * 64 + l;
    const uint32_t fl = reinterpret_cast<const uint32_t*>(F.kinds)[at];  // the cells' own loads go out before the staging's
    V4 u = ld4(u_f, at);
    const int ox = F.base[p * 3 + 0], oy = F.base[p * 3 + 1], oz = F.base[p * 3 + 2];
    const int X0 = ox >> 1, Y0 = oy >> 1, Z0 = oz >> 1;
    const int bx0 = X0 >> 2, by0 = Y0 >> 3, bz0 = Z0 >> 3;
    const int block = lut_block(C, bx0 + (l >> 2 & 1), by0 + (l >> 1 & 1), bz0 + (l & 1));  // lane q (and q + 8, ..): block q
#pragma unroll
    for (int i = 0; i < 2; ++i) {
        const int t = min(l + 64 * i, RX * RY * RZ - 1);
        const int X = X0 + t / (RY * RZ), Y = Y0 + (t / RZ) % RY, Z = Z0 + t % RZ;
        const int q = __shfl(block, ((X >> 2) - bx0) * 4 + ((Y >> 3) - by0) * 2 + ((Z >> 3) - bz0));
        su[t] = ld(u_c, q * 256 + ((X & 3) << 6 | (Y & 7) << 3 | (Z & 7)));
    }
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    const int x = ox + (l >> 4), y = oy + (l >> 1 & 7);
    const int cx = (x + 1) >> 1, cy = (y + 1) >> 1;
    const int px = 1 - (x - (2 * cx - 1)), py = 1 - (y - (2 * cy - 1));
#pragma unroll
    for (int n = 0; n < 4; ++n) {
        if (!(fl >> (8 * n) & kKindActive)) continue;
        const int z = oz + 4 * (l & 1) + n;
        const int cz = (z + 1) >> 1, pz = 1 - (z - (2 * cz - 1));
        float v = u.v[n];
        for (int i = 0; i < 2; ++i)
            for (int j = 0; j < 2; ++j)
                for (int k = 0; k < 2; ++k) {
                    const int X = cx + i - px, Y = cy + j - py, Z = cz + k - pz;
                    v += c_pweights[((i ^ px) << 2) | ((j ^ py) << 1) | (k ^ pz)] * su[((X - X0) * RY + (Y - Y0)) * RZ + (Z - Z0)];
                }
        u.v[n] = v;
    }
    st4(u_f, at, u);
}

// PCG operator: out = L v on Active|Interface cells (double accumulation); kZero: 0 elsewhere
// (the PCG's Multiply fused with Project), else other cells are left as they are (SPGrid_Laplace)
template <bool kZero>
__global__ void __launch_bounds__(256) k_laplace_pcg(DevLevel L, const float* __restrict__ v, float* __restrict__ out) {
    const int p = xcd_page(L.np), c = threadIdx.x, e = p * 256 + c;
    if (p >= L.np || page_stopped(L, p)) return;
    const uint32_t f = L.flags[e];
    float res = 0.f;
    if (f & (kActive | kInterface)) {
        const double cv = (double)v[e];
        double acc = 0.0;
#pragma unroll
        for (int k = 0; k < 6; ++k)
            if (f & (kFaceMX << k)) acc -= ((double)v[nb_index(L.nbr, p, c, k)] - cv);
        res = (float)acc;
    } else if (!kZero) {
        return;
    }
    out[e] = res;
}

// CG_VECTOR operations over the cells of the real pages (SPGrid_Gemini_Arithmetic_Helpers.h):
// 0 Copy out = a*c, 1 Copy2 out = a*c + b, 2 Plus_Equal out += a, 3 Minus_Equal out -= a, 4 Scale out *= c
__global__ void __launch_bounds__(256) k_vector_op(int op, float* __restrict__ out, const float* __restrict__ a, const float* __restrict__ b,
                                                   float c, size_t n) {
    size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    for (; i < n; i += (size_t)gridDim.x * blockDim.x) {
        switch (op) {
            case 0: out[i] = a[i] * c; break;
            case 1: out[i] = a[i] * c + b[i]; break;
            case 2: out[i] += a[i]; break;
            case 3: out[i] -= a[i]; break;
            default: out[i] *= c; break;
        }
    }
}

// Project: zero values outside Active|Interface
__global__ void __launch_bounds__(256) k_project(DevLevel L, float* __restrict__ v) {
    const int e = blockIdx.x * 256 + threadIdx.x;
    if (!(L.flags[e] & (kActive | kInterface))) v[e] = 0.f;
}

// r = b - q, then Project
__global__ void __launch_bounds__(256) k_sub_project(DevLevel L, const float* __restrict__ b, const float* __restrict__ q, float* __restrict__ r) {
    const int e = blockIdx.x * 256 + threadIdx.x;
    r[e] = (L.flags[e] & (kActive | kInterface)) ? b[e] - q[e] : 0.f;
}

// ---------------------------------------------------------------------------
// PCG vector operations, per problem. Problem p of a batch owns the level-0
// pages [pg0[p], pg0[p+1]); page_prob maps a page to its problem (-1 for the
// zero page, which is never written). Each problem's reductions are laid out
// exactly as a one-problem reduction over its own (pages + 1) * 256 cells
// (parts[p] blocks striding over them; the zero page adds nothing), so a
// problem's sums and scalars do not depend on the batch it is solved in.
// Scalars: 8 floats per problem (rho, alpha, beta, rho_old, max|r|), 4 doubles.

// out = in1 * scal[slot] + in2 (SPGrid_Copy2 with the problem's scalar), active problems only
__global__ void __launch_bounds__(256) k_seg_copy2(float* __restrict__ out, const float* __restrict__ in1, const float* __restrict__ in2,
                                                   const float* __restrict__ scal, int slot, const int* __restrict__ page_prob,
                                                   const int* __restrict__ active, size_t n) {
    size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    for (; i < n; i += (size_t)gridDim.x * blockDim.x) {
        const int pr = page_prob[i >> 8];
        if (pr < 0 || !active[pr]) continue;
        out[i] = in1[i] * scal[pr * 8 + slot] + in2[i];
    }
}

// x = s*alpha + x ; r = q*(-alpha) + r  (two SPGrid_Copy2 calls fused), active problems only
__global__ void __launch_bounds__(256) k_seg_xr_update(float* __restrict__ x, float* __restrict__ r, const float* __restrict__ s,
                                                       const float* __restrict__ q, const float* __restrict__ scal,
                                                       const int* __restrict__ page_prob, const int* __restrict__ active, size_t n) {
    size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    for (; i < n; i += (size_t)gridDim.x * blockDim.x) {
        const int pr = page_prob[i >> 8];
        if (pr < 0 || !active[pr]) continue;
        const float a = scal[pr * 8 + 1], na = -a;
        x[i] = s[i] * a + x[i];
        r[i] = q[i] * na + r[i];
    }
}

// FP64 outer variant of k_seg_copy2: out = (float)(in1 * dscal[slot] + in2) in double
__global__ void __launch_bounds__(256) k_seg_copy2_d(float* __restrict__ out, const float* __restrict__ in1, const float* __restrict__ in2,
                                                     const double* __restrict__ dscal, int slot, const int* __restrict__ page_prob,
                                                     const int* __restrict__ active, size_t n) {
    size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    for (; i < n; i += (size_t)gridDim.x * blockDim.x) {
        const int pr = page_prob[i >> 8];
        if (pr < 0 || !active[pr]) continue;
        out[i] = (float)((double)in1[i] * dscal[pr * 8 + slot] + (double)in2[i]);
    }
}

// FP64 outer variant of k_seg_xr_update: x (double) += alpha s; r = (float)(r - alpha q), alpha double
__global__ void __launch_bounds__(256) k_seg_xr_update_d(double* __restrict__ x, float* __restrict__ r, const float* __restrict__ s,
                                                         const float* __restrict__ q, const double* __restrict__ dscal,
                                                         const int* __restrict__ page_prob, const int* __restrict__ active, size_t n) {
    size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    for (; i < n; i += (size_t)gridDim.x * blockDim.x) {
        const int pr = page_prob[i >> 8];
        if (pr < 0 || !active[pr]) continue;
        const double a = dscal[pr * 8 + 3];
        x[i] += a * (double)s[i];
        r[i] = (float)((double)r[i] - a * (double)q[i]);
    }
}

// True residual r = b - L x from the FP64 iterate (double accumulation), 0 off Active|Interface
__global__ void __launch_bounds__(256) k_true_residual(DevLevel L, const double* __restrict__ x, const float* __restrict__ b,
                                                       float* __restrict__ r) {
    const int p = xcd_page(L.np), c = threadIdx.x, e = p * 256 + c;
    if (p >= L.np || page_stopped(L, p)) return;
    const uint32_t f = L.flags[e];
    float res = 0.f;
    if (f & (kActive | kInterface)) {
        const double cv = x[e];
        double acc = (double)b[e];
#pragma unroll
        for (int k = 0; k < 6; ++k)
            if (f & (kFaceMX << k)) acc += (x[nb_index(L.nbr, p, c, k)] - cv);
        res = (float)acc;
    }
    r[e] = res;
}

__global__ void k_cast_to_float(const double* __restrict__ x, float* __restrict__ y, size_t n) {
    size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    for (; i < n; i += (size_t)gridDim.x * blockDim.x) y[i] = (float)x[i];
}

constexpr int kDotThreads = 1024;
// Sum of a thread's share of float products (a*b rounded to float, then summed in double): every
// g*kDotThreads-th group of four cells from group c*kDotThreads + thread on, four groups in flight, one sum per place
// in a group: 127 MB at 256^3 at 6.1 TB/s (21 us, with the second launch it saves 24.6), one cell at a time
// and in two launches 32 us and 4.
template <bool kWide>
__device__ __forceinline__ double dot_share(const float* __restrict__ a, const float* __restrict__ b, size_t groups, int c, int g) {
    auto four = [](const float* __restrict__ p, size_t i) {
        if (kWide) return reinterpret_cast<const float4*>(p)[i];
        return make_float4(p[4 * i], p[4 * i + 1], p[4 * i + 2], p[4 * i + 3]);
    };
    double s0 = 0.0, s1 = 0.0, s2 = 0.0, s3 = 0.0;
    auto add = [&](const float4& u, const float4& v) {
        s0 += (double)(u.x * v.x); s1 += (double)(u.y * v.y); s2 += (double)(u.z * v.z); s3 += (double)(u.w * v.w);
    };
    const size_t step = (size_t)g * kDotThreads;
    size_t i = (size_t)c * kDotThreads + threadIdx.x;
    for (; i + 3 * step < groups; i += 4 * step) {
        const float4 u0 = four(a, i), u1 = four(a, i + step), u2 = four(a, i + 2 * step), u3 = four(a, i + 3 * step);
        const float4 v0 = four(b, i), v1 = four(b, i + step), v2 = four(b, i + 2 * step), v3 = four(b, i + 3 * step);
        add(u0, v0); add(u1, v1); add(u2, v2); add(u3, v3);
    }
    for (; i < groups; i += step) add(four(a, i), four(b, i));
    return (s0 + s1) + (s2 + s3);
}

// total of one value per thread of a workgroup (the same in every thread)
template <class V, class Add>
__device__ __forceinline__ V block_total(V v, Add add) {
    constexpr int NW = kDotThreads / 64;
    __shared__ V sh[NW];
    for (int o = 32; o > 0; o >>= 1) v = add(v, __shfl_down(v, o, 64));
    if ((threadIdx.x & 63) == 0) sh[threadIdx.x >> 6] = v;
    __syncthreads();
    V t = sh[0];
#pragma unroll
    for (int k = 1; k < NW; ++k) t = add(t, sh[k]);
    return t;
}
__device__ __forceinline__ double block_sum(double s) {
    return block_total(s, [](double x, double y) { return x + y; });
}
__device__ __forceinline__ float block_max(float m) {
    return block_total(m, [](float x, float y) { return fmaxf(x, y); });
}

// Reductions end in their own launch: every block leaves its partial, and the block that draws the last
// ticket adds them, in the order a second launch would (which cost 3-4 us more for each of the three
// reductions of an iteration). The ticket is zero between launches. Partials are exchanged and loaded past
// the caches, and a block draws its ticket when its exchange has returned, so no cache is written back or
// invalidated: with a release and acquire of the device's scope instead, 1024 blocks took 45 us longer, and
// the 256 of a 256^3 domain's inner product, releasing on the ticket with the acquire left to the last of them,
// 26.9 us for 24.8.
template <class V>
__device__ __forceinline__ void leave_partial(V* p, V v) {
    const V old = __hip_atomic_exchange(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    asm volatile("" ::"v"(old) : "memory");  // the exchange is complete
}
__device__ __forceinline__ bool last_block(unsigned* ticket, int g) {
    __shared__ bool last;
    if (threadIdx.x == 0) {
        last = __hip_atomic_fetch_add(ticket, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) == (unsigned)g - 1u;
        if (last) __hip_atomic_store(ticket, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
    __syncthreads();
    return last;
}
template <class V>
__device__ __forceinline__ V partial(const V* p) { return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT); }

// Scalar logic of CONJUGATE_GRADIENT_DUMPING::Solve (:193-205) in float, on a problem's inner product:
//   mode 0: rho = (float)dot -> scal[0]; beta = rho/rho_old -> scal[2]
//   mode 1: s_dot_q = (float)dot; alpha = rho/s_dot_q -> scal[1]; rho_old = rho -> scal[3]
//   mode 3: the plain sum -> dscal[2], no PCG scalar touched
//   modes 5 / 6: as 0 / 1 with the scalars in double (dscal: 0 rho, 1 s_dot_q,
//   3 alpha, 4 beta, 5 rho_old)
// Mode 3 is for every problem, the others for those that iterate.
__device__ __forceinline__ bool dot_skipped(int mode, const int* __restrict__ active, int p) { return mode != 3 && !active[p]; }
__device__ __forceinline__ void dot_scalars(int mode, double s, float* __restrict__ scal, double* __restrict__ dscal) {
    if (mode == 0) {
        const float rho = (float)s;
        scal[0] = rho;
        scal[2] = rho / scal[3];
        dscal[0] = s;
    } else if (mode == 3) {
        dscal[2] = s;
    } else if (mode == 5) {
        dscal[0] = s;
        dscal[4] = s / dscal[5];
    } else if (mode == 6) {
        dscal[1] = s;
        dscal[3] = s != 0.0 ? dscal[0] / s : 3.40282347e+38;
        dscal[5] = dscal[0];
    } else {
        const float sdq = (float)s;
        const float rho = scal[0];
        scal[1] = sdq != 0.f ? rho / sdq : 3.40282347e+38f;
        scal[3] = rho;
        dscal[1] = s;
    }
}

// block (c, p) = partial dot product c of problem p
__global__ void __launch_bounds__(kDotThreads) k_seg_dot(const float* __restrict__ a, const float* __restrict__ b, double* part,
                                                 unsigned* ticket, const int* __restrict__ pg0, const int* __restrict__ parts,
                                                 int max_parts, int mode, const int* __restrict__ active, float* __restrict__ scal,
                                                 double* __restrict__ dscal) {
    const int p = blockIdx.y, c = blockIdx.x, g = parts[p];
    if (c >= g || dot_skipped(mode, active, p)) return;
    const size_t base = (size_t)pg0[p] * 256, groups = (size_t)(pg0[p + 1] - pg0[p]) * 64;
    double s = block_sum(dot_share<true>(a + base, b + base, groups, c, g));
    double* pp = part + (size_t)p * max_parts;
    if (threadIdx.x == 0) leave_partial(pp + c, s);
    if (!last_block(ticket + p, g)) return;
    s = 0.0;
    for (int i = threadIdx.x; i < g; i += kDotThreads) s += partial(pp + i);
    s = block_sum(s);
    if (threadIdx.x == 0) dot_scalars(mode, s, scal + p * 8, dscal + p * 8);
}

// The reference's order of CG_SYSTEM::Inner_Product (DDS/CG_SYSTEM.cpp:62-72): one
// running double sum over the problem's pages in page order and their cells in
// cell order, each term the float product. One workgroup per problem stages 1024
// products at a time in LDS and one lane adds them in sequence. For checking
// against the reference's rounding, not speed.
__global__ void __launch_bounds__(256) k_seg_dot_serial(const float* __restrict__ a, const float* __restrict__ b, const int* __restrict__ pg0,
                                                        int mode, const int* __restrict__ active, float* __restrict__ scal,
                                                        double* __restrict__ dscal) {
    const int p = blockIdx.x;
    if (dot_skipped(mode, active, p)) return;
    const size_t base = (size_t)pg0[p] * 256, n = (size_t)(pg0[p + 1] - pg0[p]) * 256;
    __shared__ double buf[1024];
    double s = 0.0;
    for (size_t c0 = 0; c0 < n; c0 += 1024) {
        const size_t cnt = n - c0 < 1024 ? n - c0 : 1024;
        for (size_t t = threadIdx.x; t < cnt; t += 256) buf[t] = (double)(a[base + c0 + t] * b[base + c0 + t]);
        __syncthreads();
        if (threadIdx.x == 0)
            for (size_t t = 0; t < cnt; ++t) s += buf[t];
        __syncthreads();
    }
    if (threadIdx.x == 0) dot_scalars(mode, s, scal + p * 8, dscal + p * 8);
}

// max |a| of every problem -> scal[4]
__global__ void __launch_bounds__(kDotThreads) k_seg_maxabs(const float* __restrict__ a, float* part, unsigned* ticket,
                                                    const int* __restrict__ pg0, const int* __restrict__ parts, int max_parts,
                                                    float* __restrict__ scal) {
    const int p = blockIdx.y, c = blockIdx.x, g = parts[p];
    if (c >= g) return;
    const size_t groups = (size_t)(pg0[p + 1] - pg0[p]) * 64;
    const float4* a4 = reinterpret_cast<const float4*>(a + (size_t)pg0[p] * 256);
    float m = 0.f;
#pragma unroll 4
    for (size_t i = (size_t)c * kDotThreads + threadIdx.x; i < groups; i += (size_t)g * kDotThreads) {
        const float4 v = a4[i];
        m = fmaxf(m, fmaxf(fmaxf(fabsf(v.x), fabsf(v.y)), fmaxf(fabsf(v.z), fabsf(v.w))));
    }
    m = block_max(m);
    float* pp = part + (size_t)p * max_parts;
    if (threadIdx.x == 0) leave_partial(pp + c, m);
    if (!last_block(ticket + p, g)) return;
    m = 0.f;
    for (int i = threadIdx.x; i < g; i += kDotThreads) m = fmaxf(m, partial(pp + i));
    m = block_max(m);
    if (threadIdx.x == 0) scal[p * 8 + 4] = m;
}

// FP16 storage: the preconditioner is linear, so it runs on r / a and its
// result is scaled back by a, with a = max|r| of the cell's problem (slot 4 of
// its scalars; 1 where r = 0). Values then stay O(1), inside half's normal range.
__global__ void __launch_bounds__(256) k_scale_to_half(const float* __restrict__ r, __half* __restrict__ hb, const int* __restrict__ page_prob,
                                                       const float* __restrict__ scal, size_t n) {
    size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    for (; i < n; i += (size_t)gridDim.x * blockDim.x) {
        const int pr = page_prob[i >> 8];
        if (pr < 0) continue;
        const float a = scal[pr * 8 + 4];
        hb[i] = __float2half_rn(a > 0.f ? r[i] / a : 0.f);
    }
}
// z = a * z16 on Active|Interface cells, 0 elsewhere (Project)
__global__ void __launch_bounds__(256) k_unscale_project(DevLevel L, const __half* __restrict__ hz, float* __restrict__ z,
                                                         const int* __restrict__ page_prob, const float* __restrict__ scal) {
    const int e = blockIdx.x * 256 + threadIdx.x;
    const int pr = page_prob[e >> 8];
    const float a = pr >= 0 ? scal[pr * 8 + 4] : 0.f;
    z[e] = (pr >= 0 && (L.flags[e] & (kActive | kInterface))) ? a * __half2float(hz[e]) : 0.f;
}

// ---------------------------------------------------------------------------
// Inner product that allocates nothing (hdd_inner_product_noalloc): the block
// partials of k_seg_dot for one problem of n_pages pages go to the file-scope
// array `scratch` (one copy per device, held until the process ends), and their
// sum to the caller's device double. The blocks stride over the cells, and both
// reductions add, exactly as k_seg_dot does for a one-problem context, so the
// value has the bits of hdd_inner_product on a context holding the same pages.
// Calls take the tickets in turn and clear the one half a round away: calls that
// overlapped (they may not) spoil no later call's ticket for more than a round. A
// captured call keeps its ticket over all replays, so it clears it by itself first.
constexpr int kNoAllocParts = 1024, kNoAllocTickets = 64;  // reduce_parts never exceeds the first
struct NoAllocScratch {
    double part[kNoAllocParts];
    unsigned ticket[kNoAllocTickets];
};
static __device__ __align__(256) NoAllocScratch scratch;

__global__ void k_clear_ticket(NoAllocScratch* w, int ticket) { w->ticket[ticket] = 0; }

template <bool kWide>
__global__ void __launch_bounds__(kDotThreads) k_dot_flat(const float* __restrict__ a, const float* __restrict__ b, size_t groups, int g,
                                                  NoAllocScratch* w, int ticket, double* __restrict__ out) {
    double s = block_sum(dot_share<kWide>(a, b, groups, blockIdx.x, g));
    if (threadIdx.x == 0) {
        leave_partial(w->part + blockIdx.x, s);
        if (blockIdx.x == 0) __hip_atomic_store(w->ticket + (ticket + kNoAllocTickets / 2) % kNoAllocTickets, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
    if (!last_block(w->ticket + ticket, g)) return;
    s = 0.0;
    for (int i = threadIdx.x; i < g; i += kDotThreads) s += partial(w->part + i);
    s = block_sum(s);
    if (threadIdx.x == 0) *out = s;
}

// ---------------------------------------------------------------------------
// host launchers
static inline int grid_for(size_t n) { size_t g = (n + 255) / 256; return (int)(g > 4096 ? 4096 : (g == 0 ? 1 : g)); }

static void upload_constants_once() {
    float om[8];
    const float omega = (float)(2. / 3.);
    om[0] = 0.f;
    for (int k = 1; k < 8; ++k) om[k] = omega / (float)k;
    float s1[4] = {(float)(1. / 8.), (float)(3. / 8.), (float)(3. / 8.), (float)(1. / 8.)};
    float rw[64];
    for (int i = 0; i < 4; ++i) for (int j = 0; j < 4; ++j) for (int k = 0; k < 4; ++k) rw[i * 16 + j * 4 + k] = s1[i] * s1[j] * s1[k];
    float s2[2] = {0.75f, 0.25f};
    float pw[8];
    for (int i = 0; i < 2; ++i) for (int j = 0; j < 2; ++j) for (int k = 0; k < 2; ++k) pw[i * 4 + j * 2 + k] = s2[i] * s2[j] * s2[k] * 4.0f;
    hdd_check(hipMemcpyToSymbol(HIP_SYMBOL(c_omega_fc), om, sizeof(om)));
    hdd_check(hipMemcpyToSymbol(HIP_SYMBOL(c_rweights), rw, sizeof(rw)));
    hdd_check(hipMemcpyToSymbol(HIP_SYMBOL(c_pweights), pw, sizeof(pw)));
}

// the stencil constants are the same for every context: uploaded once per process
void upload_constants() {
    static std::once_flag once;
    std::call_once(once, upload_constants_once);
}

template <class S>
static void smooth_t(const DevLevel& L, const S* u_in, S* u_out, const S* b, bool interior, bool boundary, bool again, hipStream_t s) {
    if (!L.np) return;
    hipLaunchKernelGGL((again ? k_smooth<S, true> : k_smooth<S, false>), dim3(kXcds * xcd_chunk(sweep_groups(L.np))), dim3(64 * kSweepPages), 0, s,
                       L, u_in, u_out, b, interior ? kKindActive : 0u, boundary ? kKindActive | kKindBoundary : 0u);
}
template <class S, int C>
static void cluster_sweeps_c(const DevLevel& L, const DevClusters& W, S* u, const S* b, S* r, const SweepPhases& ph, bool u_zero, hipStream_t s) {
    hipLaunchKernelGGL((k_cluster_sweeps<S, C>), dim3(W.nwg), dim3(W.threads), 2 * (size_t)W.entries * sizeof(S), s, L, W, u, b, r, ph, (int)u_zero);
}
template <class S>
static void cluster_sweeps_t(const DevLevel& L, const DevClusters& W, S* u, const S* b, S* r, const SweepPhases& ph, bool u_zero, hipStream_t s) {
    if (!W.nwg) return;
    if (W.slots == 64 && W.threads == 64 && !W.rest) {
        hipLaunchKernelGGL(k_cluster_wave<S>, dim3(W.nwg), dim3(64), 0, s, L, W, u, b, r, ph, (int)u_zero);
        return;
    }
    switch (W.slots / W.threads) {  // cells per thread
        case 1: cluster_sweeps_c<S, 1>(L, W, u, b, r, ph, u_zero, s); break;
        case 2: cluster_sweeps_c<S, 2>(L, W, u, b, r, ph, u_zero, s); break;
        case 4: cluster_sweeps_c<S, 4>(L, W, u, b, r, ph, u_zero, s); break;
        case 8: cluster_sweeps_c<S, 8>(L, W, u, b, r, ph, u_zero, s); break;
        default: throw std::runtime_error("cluster sweeps: cells per thread");
    }
}
template <class S, int C>
static void allow_cluster_lds() {
    hdd_check(hipFuncSetAttribute(reinterpret_cast<const void*>(&k_cluster_sweeps<S, C>), hipFuncAttributeMaxDynamicSharedMemorySize,
                                  (int)kClusterLdsBytes),
              "cluster sweeps' LDS");
}
void prepare_cluster_sweeps(const DevClusters& W) {
    if (!W.nwg || 2 * (size_t)W.entries * sizeof(float) <= 48 * 1024) return;
    switch (W.slots / W.threads) {
        case 1: allow_cluster_lds<float, 1>(); allow_cluster_lds<__half, 1>(); break;
        case 2: allow_cluster_lds<float, 2>(); allow_cluster_lds<__half, 2>(); break;
        case 4: allow_cluster_lds<float, 4>(); allow_cluster_lds<__half, 4>(); break;
        case 8: allow_cluster_lds<float, 8>(); allow_cluster_lds<__half, 8>(); break;
        default: throw std::runtime_error("cluster sweeps: cells per thread");
    }
}
template <class S>
static void residual_t(const DevLevel& L, const S* u, const S* b, S* r, hipStream_t s) {
    if (L.np) hipLaunchKernelGGL(k_residual<S>, dim3(kXcds * xcd_chunk(page_groups(L.np))), dim3(256), 0, s, L, u, b, r);
}
template <class S>
static void fill_t(S* a, float v, size_t n, hipStream_t s) {
    if (n) hipLaunchKernelGGL(k_fill<S>, dim3(grid_for(n)), dim3(256), 0, s, a, v, n);
}
template <class S>
static void restrict_t(const DevLevel& F, const DevLevel& C, const S* r_f, S* b_c, hipStream_t s) {
    if (C.np) hipLaunchKernelGGL(k_restrict<S>, dim3(kXcds * xcd_chunk(C.np)), dim3(256), 0, s, F, C, r_f, b_c);
}
template <class S>
static void prolong_t(const DevLevel& F, const DevLevel& C, S* u_f, const S* u_c, hipStream_t s) {
    if (F.np) hipLaunchKernelGGL(k_prolong<S>, dim3(kXcds * xcd_chunk(page_groups(F.np))), dim3(256), 0, s, F, C, u_f, u_c);
}
void launch_smooth(const DevLevel& L, const float* u_in, float* u_out, const float* b, bool interior, bool boundary, bool again, hipStream_t s) {
    smooth_t(L, u_in, u_out, b, interior, boundary, again, s);
}
void launch_smooth(const DevLevel& L, const __half* u_in, __half* u_out, const __half* b, bool interior, bool boundary, bool again, hipStream_t s) {
    smooth_t(L, u_in, u_out, b, interior, boundary, again, s);
}
void launch_cluster_sweeps(const DevLevel& L, const DevClusters& C, float* u, const float* b, float* r, const SweepPhases& ph, bool u_zero,
                           hipStream_t s) {
    cluster_sweeps_t(L, C, u, b, r, ph, u_zero, s);
}
void launch_cluster_sweeps(const DevLevel& L, const DevClusters& C, __half* u, const __half* b, __half* r, const SweepPhases& ph,
                           bool u_zero, hipStream_t s) {
    cluster_sweeps_t(L, C, u, b, r, ph, u_zero, s);
}
void launch_residual(const DevLevel& L, const float* u, const float* b, float* r, hipStream_t s) { residual_t(L, u, b, r, s); }
void launch_residual(const DevLevel& L, const __half* u, const __half* b, __half* r, hipStream_t s) { residual_t(L, u, b, r, s); }
void launch_fill(float* a, float v, size_t n, hipStream_t s) { fill_t(a, v, n, s); }
void launch_fill(__half* a, float v, size_t n, hipStream_t s) { fill_t(a, v, n, s); }
void launch_copy(float* d, const float* src, size_t n, hipStream_t s) {
    if (n) hipLaunchKernelGGL(k_copy, dim3(grid_for(n)), dim3(256), 0, s, d, src, n);
}
void launch_restrict(const DevLevel& F, const DevLevel& C, const float* r_f, float* b_c, hipStream_t s) { restrict_t(F, C, r_f, b_c, s); }
void launch_restrict(const DevLevel& F, const DevLevel& C, const __half* r_f, __half* b_c, hipStream_t s) { restrict_t(F, C, r_f, b_c, s); }
void launch_prolong(const DevLevel& F, const DevLevel& C, float* u_f, const float* u_c, hipStream_t s) { prolong_t(F, C, u_f, u_c, s); }
void launch_prolong(const DevLevel& F, const DevLevel& C, __half* u_f, const __half* u_c, hipStream_t s) { prolong_t(F, C, u_f, u_c, s); }
void launch_scale_to_half(const float* r, __half* hb, const int* page_prob, const float* scal, size_t n, hipStream_t s) {
    if (n) hipLaunchKernelGGL(k_scale_to_half, dim3(grid_for(n)), dim3(256), 0, s, r, hb, page_prob, scal, n);
}
void launch_unscale_project(const DevLevel& L, const __half* hz, float* z, const int* page_prob, const float* scal, hipStream_t s) {
    if (L.np) hipLaunchKernelGGL(k_unscale_project, dim3(L.np + 1), dim3(256), 0, s, L, hz, z, page_prob, scal);
}
void launch_laplace_pcg(const DevLevel& L, const float* v, float* out, hipStream_t s) {
    if (L.np) hipLaunchKernelGGL(k_laplace_pcg<true>, dim3(kXcds * xcd_chunk(L.np)), dim3(256), 0, s, L, v, out);
}
void launch_laplace(const DevLevel& L, const float* v, float* out, hipStream_t s) {
    if (L.np) hipLaunchKernelGGL(k_laplace_pcg<false>, dim3(kXcds * xcd_chunk(L.np)), dim3(256), 0, s, L, v, out);
}
void launch_vector_op(int op, float* out, const float* a, const float* b, float c, size_t n, hipStream_t s) {
    if (n) hipLaunchKernelGGL(k_vector_op, dim3(grid_for(n)), dim3(256), 0, s, op, out, a, b, c, n);
}
void launch_project(const DevLevel& L, float* v, hipStream_t s) {
    if (L.np) hipLaunchKernelGGL(k_project, dim3(L.np), dim3(256), 0, s, L, v);
}
void launch_sub_project(const DevLevel& L, const float* b, const float* q, float* r, hipStream_t s) {
    if (L.np) hipLaunchKernelGGL(k_sub_project, dim3(L.np), dim3(256), 0, s, L, b, q, r);
}
// Blocks of a reduction over n cells: four cells per thread, and one block per CU at most (the blocks draw
// their tickets one after the other, about 12 ns each)
int reduce_parts(size_t n) { return (int)std::max<size_t>(1, std::min<size_t>(256, (n + 4 * kDotThreads - 1) / (4 * kDotThreads))); }

// Device address of `scratch` on the current device: hipGetSymbolAddress once
// per device, with that device current, kept for later calls (each device
// holds its own copy of the array at its own address; the array's name in
// host code is not a device address).
static NoAllocScratch* noalloc_scratch() {
    constexpr int kMaxDevices = 64;
    static std::mutex mu;
    static NoAllocScratch* ptr[kMaxDevices] = {};
    int dev = 0;
    hdd_check(hipGetDevice(&dev), "hipGetDevice");
    if (dev < 0 || dev >= kMaxDevices) throw std::runtime_error("inner product (no allocation): device index out of range");
    std::lock_guard<std::mutex> lk(mu);
    if (!ptr[dev]) {
        void* p = nullptr;
        hdd_check(hipGetSymbolAddress(&p, HIP_SYMBOL(scratch)), "hipGetSymbolAddress(scratch)");
        ptr[dev] = static_cast<NoAllocScratch*>(p);
    }
    return ptr[dev];
}

void launch_inner_product_noalloc(const float* a, const float* b, int64_t n_pages, double* out, hipStream_t s) {
    const size_t n = (size_t)n_pages * kPageCells;
    const int g = reduce_parts((size_t)(n_pages + 1) * kPageCells);  // the partition of a context of n_pages pages
    if (g > kNoAllocParts) throw std::runtime_error("inner product (no allocation): more partial sums than the scratch holds");
    static std::atomic<unsigned> calls{0};
    const int ticket = (int)(calls.fetch_add(1, std::memory_order_relaxed) % kNoAllocTickets);
    if (s) {
        hipStreamCaptureStatus capture = hipStreamCaptureStatusNone;
        if (hipStreamIsCapturing(s, &capture) != hipSuccess) (void)hipGetLastError();
        if (capture == hipStreamCaptureStatusActive) hipLaunchKernelGGL(k_clear_ticket, dim3(1), dim3(1), 0, s, noalloc_scratch(), ticket);
    }
    // the caller's arrays may start anywhere
    const bool wide = ((reinterpret_cast<uintptr_t>(a) | reinterpret_cast<uintptr_t>(b)) & 15) == 0;
    hipLaunchKernelGGL((wide ? k_dot_flat<true> : k_dot_flat<false>), dim3(g), dim3(kDotThreads), 0, s, a, b, n / 4, g, noalloc_scratch(), ticket, out);
    hdd_check(hipGetLastError(), "inner product (no allocation)");
}
void launch_seg_copy2(const DevSegments& S, float* out, const float* in1, const float* in2, int slot, hipStream_t s) {
    hipLaunchKernelGGL(k_seg_copy2, dim3(grid_for(S.ncells)), dim3(256), 0, s, out, in1, in2, (const float*)S.scal, slot, S.page_prob,
                       S.active, S.ncells);
}
void launch_seg_xr_update(const DevSegments& S, float* x, float* r, const float* sv, const float* q, hipStream_t s) {
    hipLaunchKernelGGL(k_seg_xr_update, dim3(grid_for(S.ncells)), dim3(256), 0, s, x, r, sv, q, (const float*)S.scal, S.page_prob,
                       S.active, S.ncells);
}
void launch_seg_dot(const DevSegments& S, const float* a, const float* b, int mode, hipStream_t s) {
    if (S.serial_dots)
        hipLaunchKernelGGL(k_seg_dot_serial, dim3(S.nprob), dim3(256), 0, s, a, b, S.pg0, mode, S.active, S.scal, S.dscal);
    else
        hipLaunchKernelGGL(k_seg_dot, dim3(S.max_parts, S.nprob), dim3(kDotThreads), 0, s, a, b, S.dpart, S.ticket, S.pg0, S.parts, S.max_parts, mode,
                           S.active, S.scal, S.dscal);
}
void launch_seg_copy2_d(const DevSegments& S, float* out, const float* in1, const float* in2, int slot, hipStream_t s) {
    hipLaunchKernelGGL(k_seg_copy2_d, dim3(grid_for(S.ncells)), dim3(256), 0, s, out, in1, in2, (const double*)S.dscal, slot, S.page_prob,
                       S.active, S.ncells);
}
void launch_seg_xr_update_d(const DevSegments& S, double* x, float* r, const float* sv, const float* q, hipStream_t s) {
    hipLaunchKernelGGL(k_seg_xr_update_d, dim3(grid_for(S.ncells)), dim3(256), 0, s, x, r, sv, q, (const double*)S.dscal, S.page_prob,
                       S.active, S.ncells);
}
void launch_true_residual(const DevLevel& L, const double* x, const float* b, float* r, hipStream_t s) {
    if (L.np) hipLaunchKernelGGL(k_true_residual, dim3(kXcds * xcd_chunk(L.np)), dim3(256), 0, s, L, x, b, r);
}
void launch_cast_to_float(const double* x, float* y, size_t n, hipStream_t s) {
    if (n) hipLaunchKernelGGL(k_cast_to_float, dim3(grid_for(n)), dim3(256), 0, s, x, y, n);
}
void launch_seg_maxabs(const DevSegments& S, const float* a, hipStream_t s) {
    hipLaunchKernelGGL(k_seg_maxabs, dim3(S.max_parts, S.nprob), dim3(kDotThreads), 0, s, a, S.fpart, S.ticket, S.pg0, S.parts, S.max_parts, S.scal);
}

}  // namespace hdd

namespace hdd {

// b0[i] = r_e - (float)(-sum over Active face neighbours of z, double accumulation)
// for each interface dof i at level-0 cell e (Laplace_ri + Copy_To_Eigen_Array,
// LIB/SPGrid_Laplace_Legacy.h:95-116, IFS/EIGEN_INTERFACE.cpp:18-30)
template <class S>
__global__ void k_if_gather(DevLevel L, const int* __restrict__ if_index, int n, const S* __restrict__ z,
                            const S* __restrict__ r, float* __restrict__ b0) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const int e = if_index[i];
    if (e < 0) { b0[i] = 0.f; return; }
    const int p = e >> 8, c = e & 255;
    const uint32_t f = L.flags[e];
    double res = 0.0;
#pragma unroll
    for (int k = 0; k < 6; ++k)
        if (f & (kFaceMX << k)) {
            const int q = nb_index(L.nbr, p, c, k);
            if (L.flags[q] & kActive) res -= (double)ld(z, q);
        }
    b0[i] = ld(r, e) - (float)res;
}

template <class S>
__global__ void k_if_scatter(const int* __restrict__ if_index, int n, const float* __restrict__ u0, S* __restrict__ z) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const int e = if_index[i];
    if (e >= 0) st(z, e, u0[i]);
}

void launch_if_gather(const DevLevel& L0, const int* if_index, int n, const float* z, const float* r, float* b0, hipStream_t s) {
    if (n) hipLaunchKernelGGL(k_if_gather<float>, dim3((n + 255) / 256), dim3(256), 0, s, L0, if_index, n, z, r, b0);
}
void launch_if_gather(const DevLevel& L0, const int* if_index, int n, const __half* z, const __half* r, float* b0, hipStream_t s) {
    if (n) hipLaunchKernelGGL(k_if_gather<__half>, dim3((n + 255) / 256), dim3(256), 0, s, L0, if_index, n, z, r, b0);
}
void launch_if_scatter(const int* if_index, int n, const float* u0, float* z, hipStream_t s) {
    if (n) hipLaunchKernelGGL(k_if_scatter<float>, dim3((n + 255) / 256), dim3(256), 0, s, if_index, n, u0, z);
}
void launch_if_scatter(const int* if_index, int n, const float* u0, __half* z, hipStream_t s) {
    if (n) hipLaunchKernelGGL(k_if_scatter<__half>, dim3((n + 255) / 256), dim3(256), 0, s, if_index, n, u0, z);
}

}  // namespace hdd

