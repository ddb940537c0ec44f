// Dense-node form of the interface solver's exact solves (hdd_nodeplan.h): the
// blocks' operators formed in double at set-up, and the two passes of a solve.
//
// An operator is kept in 16x16 tiles of 1 KiB in the lane order of the FP32
// MFMA: lane l holds row l%16, columns 4(l/16) .. +3, so a wavefront loads a
// tile with one contiguous 16-byte access per lane and uses it as the A
// operand of four v_mfma_f32_16x16x4_f32 (instruction s takes the columns
// 4q + s of the lanes' groups q; A and B agree on that order, so it only
// permutes the summands). The B operand is the run's vectors, one node per
// column, in LDS. Blocks of a single node, most of them above the first level,
// would fill one of the sixteen columns: they take the same tiles through vector
// FMAs (16 instead of 128 cycles a tile) and add across the lanes at the end of
// a row (96^3 interfaces: 72.8 -> 67.5 us a solve; with such sums for runs of two
// to four as well the registers cost more than the matrix unit's idle columns).
// The rest of a launch is latency, so a kernel is kept short: the wave's number
// and all loop control are scalars, a pass's first loads go out before its first
// tiles and everything a row tile needs at its end beside them, and no load
// waits at the end of a branch (67.5 -> 57.3 us).
// (The matrix unit consumes tiles at about 20 TB/s over the chip, HBM
// delivers 8.) Forward tiles of a block: row tile rt < nk (Linv) has rt + 1 of
// them, row tile nk + a (W) has nk. Backward: row tile rt has nk - rt (Linv^T)
// and nrk (-W^T). A closed block (nrk = 0): every row tile of its inverse has nk.
#include <hip/hip_runtime.h>
#include <algorithm>
#include <stdexcept>
#include "hdd_nodeplan_device.h"

namespace hdd {

namespace {

typedef float f32x4 __attribute__((ext_vector_type(4)));
constexpr int T = NodePlanHost::kTile;

__device__ __forceinline__ long long fwd_row(int rt, int nk) {
    return rt < nk ? (long long)rt * (rt + 1) / 2 : (long long)nk * (nk + 1) / 2 + (long long)(rt - nk) * nk;
}
__device__ __forceinline__ long long bwd_row(int rt, int nk, int nrk) { return (long long)rt * (nk + nrk) - (long long)rt * (rt - 1) / 2; }

__device__ __forceinline__ bool run_stopped(const int* __restrict__ active, const int* __restrict__ prob, int i0, int cnt) {
    if (!active) return false;
    for (int j = 0; j < cnt; ++j)
        if (active[prob[i0 + j]]) return false;
    return true;
}

// Children's sums of a level, one thread per row: t = b - sum at its columns,
// the sum itself at its boundary rows (in c, where the forward product adds to it).
// On its own because a node's row tiles go to several workgroups, which all need every t of the node:
// with the sums inside the forward kernel, its gather was 3 times its product on the 256^3 level-0
// interiors (171 us against 49 us for the backward pass of the same level); and where the gather is
// small beside the tiles (a tenth of their bytes), no faster: 96^3 level-0 interface 74.6 us with,
// 71.8 us without it.
__global__ void __launch_bounds__(256) k_node_children(int y0, int y1, int c0, int c1, const NodePos* __restrict__ pos_y,
                                                       const NodePos* __restrict__ pos_c, const int* __restrict__ more,
                                                       const int* __restrict__ orig, const float* __restrict__ b,
                                                       float* __restrict__ t, float* __restrict__ c) {
    const int i = blockIdx.x * 256 + threadIdx.x, ny = y1 - y0;
    if (i >= ny + c1 - c0) return;
    const bool col = i < ny;
    const NodePos p = col ? pos_y[y0 + i] : pos_c[c0 + i - ny];
    float bv = 0.f;
    if (col) {
        const int o = orig[y0 + i];
        if (o >= 0) bv = b[o];
    }
    float s = c[p.p0];
    if (p.p1 >= 0) {
        s += c[p.p1];
    } else {
        const int* m = more + ~p.p1;
        const int cnt = m[0];
#pragma unroll 4
        for (int e = 1; e <= cnt; ++e) s += c[m[e]];
    }
    if (col) t[y0 + i] = bv - s;
    else c[c0 + i - ny] = s;
}

// D (16 rows x 16 nodes, or x 1 with ONE, in the matrix unit's layout) of one row tile: tiles [0, nt) at A against the operand vectors from tp on,
// every KS-th tile from kw. The tiles are loaded kAhead at a time, a group ahead of the products
// (`a` holds the first group on entry); four independent sums (one per tile column mod 4) keep the
// chains short.
constexpr int kAhead = 4;
template <int KS>
__device__ __forceinline__ void load_group(const f32x4* __restrict__ A, int k, int nt, f32x4 (&a)[kAhead]) {
#pragma unroll
    for (int u = 0; u < kAhead; ++u)
        if (k + u * KS < nt) a[u] = A[(size_t)(k + u * KS) * 64];
}
template <int KS, bool ONE>
__device__ __forceinline__ f32x4 row_tile(const f32x4* __restrict__ A, const f32x4* tp, int nt, int kw, f32x4 (&a)[kAhead]) {
    if (ONE) {
        f32x4 s = {0.f, 0.f, 0.f, 0.f};
        for (int k = kw; k < nt; k += kAhead * KS) {
            f32x4 nx[kAhead];
            load_group<KS>(A, k + kAhead * KS, nt, nx);
#pragma unroll
            for (int u = 0; u < kAhead; ++u)
                if (k + u * KS < nt) s = __builtin_elementwise_fma(a[u], tp[(k + u * KS) * 4], s);
#pragma unroll
            for (int u = 0; u < kAhead; ++u) a[u] = nx[u];
        }
        float v = (s[0] + s[1]) + (s[2] + s[3]);  // the lane's columns of its row; then all columns
        v += __shfl_xor(v, 16);
        v += __shfl_xor(v, 32);
        const int r = (threadIdx.x & 48) >> 2;  // rows 4q .. 4q + 3, as the matrix unit leaves them
        return f32x4{__shfl(v, r), __shfl(v, r + 1), __shfl(v, r + 2), __shfl(v, r + 3)};
    }
    f32x4 s0 = {0.f, 0.f, 0.f, 0.f}, s1 = s0, s2 = s0, s3 = s0;
    for (int k = kw; k < nt; k += kAhead * KS) {
        f32x4 nx[kAhead];
        load_group<KS>(A, k + kAhead * KS, nt, nx);
#pragma unroll
        for (int u = 0; u < kAhead; ++u)
            if (k + u * KS < nt) {
                const f32x4 t = tp[(k + u * KS) * 4];
                s0 = __builtin_amdgcn_mfma_f32_16x16x4f32(a[u][0], t[0], s0, 0, 0, 0);
                s1 = __builtin_amdgcn_mfma_f32_16x16x4f32(a[u][1], t[1], s1, 0, 0, 0);
                s2 = __builtin_amdgcn_mfma_f32_16x16x4f32(a[u][2], t[2], s2, 0, 0, 0);
                s3 = __builtin_amdgcn_mfma_f32_16x16x4f32(a[u][3], t[3], s3, 0, 0, 0);
            }
#pragma unroll
        for (int u = 0; u < kAhead; ++u) a[u] = nx[u];
    }
    return (s0 + s1) + (s2 + s3);
}

// adds the partial sums of the KS waves that share a row tile (the first of them returns the total);
// every wave of the workgroup takes part
template <int KS>
__device__ __forceinline__ f32x4 join(f32x4 d, f32x4 (*red)[64], int w, int lane) {
    if (KS == 1) return d;
    __syncthreads();  // the previous row tile's sums have been read
    red[w][lane] = d;
    __syncthreads();
    if (w % KS == 0)
        for (int s = 1; s < KS; ++s) d += red[w + s][lane];
    return d;
}

// The row tiles [rt0, rt1) of a workgroup of NW waves, KS of them per row tile: gather fills the
// operand vectors in LDS, its first loads ahead of the first tiles (a wait for a load is a wait for all
// before it), the dependent ones beside them; where(rt, &A, &tp, &nt) gives a row tile's
// tiles and operand, ahead(rt) loads beside the first tiles what out(rt, d, it) needs for the 16x16 result in
// the lanes that hold it.
struct Ahead { f32x4 v; int4 o; };
template <int NW, int KS, bool ONE, class Where, class Gather, class Load, class Out>
__device__ __forceinline__ void row_tiles(int rt0, int rt1, f32x4 (*red)[64], Where where, Gather gather, Load ahead, Out out) {
    // the wave's number as a scalar: its row tiles and their loops stay on the scalar unit
    const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
    constexpr int step = NW / KS;
    int rt = rt0 + w / KS, nt;
    const f32x4 *A, *tp;
    f32x4 a[kAhead];
    const f32x4 g = gather.first();
    {   // (a wave without a row tile loads the last one: no wait at a branch's end)
        const int rf = min(rt, rt1 - 1);
        where(rf, A, tp, nt);
        load_group<KS>(A, w % KS, nt, a);
    }
    Ahead add = ahead(min(rt, rt1 - 1));
    if (!gather.fill(g)) return;
    __syncthreads();
    for (int r0 = rt0; r0 < rt1; r0 += step) {
        const bool live = rt < rt1;
        f32x4 d = {0.f, 0.f, 0.f, 0.f};
        if (live) d = row_tile<KS, ONE>(A, tp, nt, w % KS, a);
        const int rc = rt;
        const Ahead ac = add;
        rt += step;
        if (rt < rt1) {  // the next row tile's first tiles load beside this one's results
            where(rt, A, tp, nt);
            load_group<KS>(A, w % KS, nt, a);
            add = ahead(rt);
        }
        d = join<KS>(d, red, w, lane);
        if (live && w % KS == 0) out(rc, d, ac);
    }
}
template <int NW, bool ONE, class Where, class Gather, class Load, class Out>
__device__ __forceinline__ void row_tiles(int split, int rt0, int rt1, f32x4 (*red)[64], Where where, Gather gather, Load ahead, Out out) {
    if (NW == 16) return row_tiles<NW, 16, ONE>(rt0, rt1, red, where, gather, ahead, out);
    if (split == 1) return row_tiles<NW, 1, ONE>(rt0, rt1, red, where, gather, ahead, out);
    if (split == 2) return row_tiles<NW, 2, ONE>(rt0, rt1, red, where, gather, ahead, out);
    row_tiles<NW, 4, ONE>(rt0, rt1, red, where, gather, ahead, out);
}

template <int NW, class Where, class Gather, class Load, class Out>
__device__ __forceinline__ void run_tiles(const NodeItem& it, f32x4 (*red)[64], Where where, Gather gather, Load ahead, Out out) {
    if (it.one) return row_tiles<NW, true>(it.split, it.rt0, it.rt1, red, where, gather, ahead, out);
    row_tiles<NW, false>(it.split, it.rt0, it.rt1, red, where, gather, ahead, out);
}

// 16 bytes, of floats or of indices (through HIP's int4 instead, the compiler put the LDS address of the
// operand's store into one of its data registers)
__device__ __forceinline__ f32x4 load4(const void* p) { return *reinterpret_cast<const f32x4*>(p); }

// Operand vectors of a run, `rows` of each node: four rows from load(i, j, k) (row k of node j, i in all),
// whose values (a vector, or where to find it) go through value(v, k) to LDS. fill() is false for a run
// of stopped problems.
template <int NW, class Load, class Value>
struct Operands {
    const NodeItem& it;
    int rows;
    const int *active, *prob;
    f32x4* lds;
    Load load;
    Value value;
    __device__ __forceinline__ f32x4 at(int idx) const {
        const int j = it.cnt == 1 ? 0 : idx / (rows / 4);
        return load(4 * idx, j, 4 * idx - j * rows);
    }
    __device__ __forceinline__ f32x4 first() const { return at(min((int)threadIdx.x, it.cnt * rows / 4 - 1)); }
    __device__ __forceinline__ bool fill(f32x4 v) const {
        if (run_stopped(active, prob, it.inst0, it.cnt)) return false;
        const int n = it.cnt * rows / 4;
        for (int idx = threadIdx.x; idx < n;) {
            const int j = it.cnt == 1 ? 0 : idx / (rows / 4);
            lds[idx + j] = value(v, 4 * idx - j * rows);
            idx += NW * 64;
            if (idx < n) v = at(idx);
        }
        return true;
    }
};
template <int NW, class Load, class Value>
__device__ __forceinline__ Operands<NW, Load, Value> operands(const NodeItem& it, int rows, const int* active, const int* prob, f32x4* lds,
                                                              Load load, Value value) {
    return {it, rows, active, prob, lds, load, value};
}

__device__ __forceinline__ void store_rows(int4 o, f32x4 d, float* __restrict__ x) {
    if (o.x >= 0) x[o.x] = d[0];
    if (o.y >= 0) x[o.y] = d[1];
    if (o.z >= 0) x[o.z] = d[2];
    if (o.w >= 0) x[o.w] = d[3];
}

// Forward pass of a level: t into LDS, then the row tiles of [I + S; W] t, or of a closed node's whole
// result (the inverse's diagonal apart as well: its row's largest term is added once, after the others).
// NW waves per workgroup; INC: the nodes have children (t and the boundary rows' sums from k_node_children).
template <int NW, bool INC>
__global__ void __launch_bounds__(NW * 64) k_node_fwd(const NodeItem* __restrict__ items, const int* __restrict__ inst_prob,
                                                      const int* __restrict__ active, const int* __restrict__ orig,
                                                      const float* __restrict__ t, const float* __restrict__ tiles,
                                                      const float* __restrict__ scale, const float* __restrict__ b,
                                                      float* __restrict__ y, float* __restrict__ c, float* __restrict__ z,
                                                      float* __restrict__ x) {
    extern __shared__ f32x4 lds[];
    __shared__ f32x4 red[NW][64];
    const NodeItem it = items[blockIdx.x];
    const int lane = threadIdx.x & 63, col = lane & 15, q = lane >> 4;
    const int np = it.nk * T, ld = np + 4, my_col = min(col, it.cnt - 1);
    const int yb = it.y0 + my_col * np, cb = it.c0 + my_col * it.nrk * T;
    const f32x4* base = reinterpret_cast<const f32x4*>(tiles) + (size_t)it.tile * 64 + lane;
    const f32x4* tcol = lds + (my_col * ld) / 4 + q;
    auto where = [&](int rt, const f32x4*& A, const f32x4*& tp, int& nt) {
        A = base + (size_t)(it.nrk ? fwd_row(rt, it.nk) : (long long)rt * it.nk) * 64;
        tp = tcol;
        nt = it.nrk && rt < it.nk ? rt + 1 : it.nk;
    };
    auto gather = operands<NW>(
        it, np, active, inst_prob, lds,
        [&](int i, int, int) { return INC ? load4(t + it.y0 + i) : load4(orig + it.y0 + i); },
        [&](f32x4 v, int) {
            if (INC) return v;
            f32x4 r;
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const int o = __float_as_int(v[e]);
                r[e] = o >= 0 ? b[o] : 0.f;
            }
            return r;
        });
    auto ahead = [&](int rt) {  // the row tile's D^-2 or inverse diagonal, or its children's sums; rows of x
        // (lanes beyond the run load the last node's, so that no load waits behind a branch)
        Ahead h;
        const int r = INC && rt >= it.nk ? cb + (rt - it.nk) * T : it.scale + min(rt, it.nk - 1) * T;
        h.v = *reinterpret_cast<const f32x4*>((INC && rt >= it.nk ? c : scale) + r + 4 * q);
        h.o = *reinterpret_cast<const int4*>(orig + yb + min(rt, it.nk - 1) * T + 4 * q);
        return h;
    };
    auto out = [&](int rt, f32x4 d, const Ahead& h) {
        if (col >= it.cnt) return;
        if (!it.nrk) {
            d += tcol[rt * 4] * h.v;
            *reinterpret_cast<f32x4*>(z + yb + rt * T + 4 * q) = d;
            store_rows(h.o, d, x);
        } else if (rt < it.nk) {
            d += tcol[rt * 4];  // the unit diagonal
            d *= h.v;
            *reinterpret_cast<f32x4*>(y + yb + rt * T + 4 * q) = d;
        } else {
            if (INC) d += h.v;
            *reinterpret_cast<f32x4*>(c + cb + (rt - it.nk) * T + 4 * q) = d;
        }
    };
    run_tiles<NW>(it, red, where, gather, ahead, out);
}

// Backward pass of a level: [D^-2 y; z of the boundary rows] into LDS, then the row tiles of
// [I + S^T | -W^T]; the result goes to z and, in the original numbering, to x.
template <int NW>
__global__ void __launch_bounds__(NW * 64) k_node_bwd(const NodeItem* __restrict__ items, const int* __restrict__ inst_prob,
                                                      const int* __restrict__ active, const int* __restrict__ orig,
                                                      const int* __restrict__ zidx, const float* __restrict__ tiles,
                                                      const float* __restrict__ y, float* __restrict__ z, float* __restrict__ x) {
    extern __shared__ f32x4 lds[];
    __shared__ f32x4 red[NW][64];
    const NodeItem it = items[blockIdx.x];
    const int lane = threadIdx.x & 63, col = lane & 15, q = lane >> 4;
    const int np = it.nk * T, nz = np + it.nrk * T, ld = nz + 4, my_col = min(col, it.cnt - 1);
    const int yb = it.y0 + my_col * np;
    const f32x4* base = reinterpret_cast<const f32x4*>(tiles) + (size_t)it.tile * 64 + lane;
    const f32x4* tcol = lds + (my_col * ld) / 4 + q;
    auto where = [&](int rt, const f32x4*& A, const f32x4*& tp, int& nt) {
        A = base + (size_t)bwd_row(rt, it.nk, it.nrk) * 64;
        tp = tcol + rt * 4;
        nt = it.nk + it.nrk - rt;
    };
    auto gather = operands<NW>(
        it, nz, active, inst_prob, lds,
        [&](int, int j, int k) {
            return load4(k < np ? reinterpret_cast<const int*>(y) + it.y0 + j * np + k : zidx + it.c0 + j * (nz - np) + k - np);
        },
        [&](f32x4 v, int k) {
            if (k >= np) {
#pragma unroll
                for (int e = 0; e < 4; ++e) v[e] = z[__float_as_int(v[e])];
            }
            return v;
        });
    auto ahead = [&](int rt) { return Ahead{{}, *reinterpret_cast<const int4*>(orig + yb + rt * T + 4 * q)}; };
    auto out = [&](int rt, f32x4 d, const Ahead& h) {
        if (col >= it.cnt) return;
        d += tcol[rt * 4];
        *reinterpret_cast<f32x4*>(z + yb + rt * T + 4 * q) = d;
        store_rows(h.o, d, x);
    };
    run_tiles<NW>(it, red, where, gather, ahead, out);
}

// ---- set-up: the operators from the factor columns, in double -----------------------------------

struct SetupBlock {
    long long l, x;   // first double of the block's columns ((nk + nrk) T x nk T, row-major) and of Linv
    int nk, nrk, fwd, bwd, scale, pad;
};

// A supernode's factor columns on their way into its block: L11 (n x n) and L21 (nr x n), column-major
struct SetupSupernode {
    long long src, l;      // first double of L11 (L21 follows), first of the block's columns
    int np, col, n, nr;    // row length of the block, first column of the supernode
    int rows;              // first of its block rows in the row lists
    int pad0, pad1;        // padding columns [pad0, pad1) of the block, set by its first supernode
    int unused;
};

// One workgroup per supernode: its columns into the zeroed block, one on the padding's diagonal
__global__ void __launch_bounds__(256) k_node_columns(const SetupSupernode* __restrict__ sn, const int* __restrict__ rows,
                                                      const double* __restrict__ src, double* __restrict__ L) {
    const SetupSupernode S = sn[blockIdx.x];
    double* Lb = L + S.l;
    const double* a = src + S.src;
    const long long n11 = (long long)S.n * S.n, n21 = (long long)S.nr * S.n;
    for (long long e = threadIdx.x; e < n11; e += 256) {
        const int j = (int)(e / S.n), r = (int)(e - (long long)j * S.n);
        if (r >= j) Lb[(long long)(S.col + r) * S.np + S.col + j] = a[e];
    }
    for (long long e = threadIdx.x; e < n21; e += 256) {
        const int j = (int)(e / S.nr), r = (int)(e - (long long)j * S.nr);
        Lb[(long long)rows[S.rows + r] * S.np + S.col + j] = a[n11 + e];
    }
    for (int i = S.pad0 + (int)threadIdx.x; i < S.pad1; i += 256) Lb[(long long)i * S.np + i] = 1.0;
}

// s += sign * sum over the tiles k in [k0, k1) of A(., k) B(k, .), element (r, c) of a 16x16 tile, with
// A's tiles along a row at a + 16 k and B's down a column at b + 16 k * ld. Four tile pairs go through
// LDS at a time and the next four load meanwhile: one at a time, the wait for each pair made the
// inverse of a 2080-row block take 30 ms.
// With kAT, A is the transpose of what `a` points to: its tiles go down a column at a + 16 k * ld.
constexpr int kPairs = 4;
template <bool kAT = false>
__device__ __forceinline__ double tile_products(double s, double sign, const double* __restrict__ a, const double* b, long long ld, int k0,
                                                int k1, double (*as)[T][T + 1], double (*bs)[T][T + 1]) {
    const int r = threadIdx.x >> 4, c = threadIdx.x & 15;
    double an[kPairs], bn[kPairs];
    auto fetch = [&](int k) {
#pragma unroll
        for (int u = 0; u < kPairs; ++u) {
            const bool in = k + u < k1;
            an[u] = in ? (kAT ? a[((long long)(k + u) * T + r) * ld + c] : a[r * ld + (long long)(k + u) * T + c]) : 0.0;
            bn[u] = in ? b[((long long)(k + u) * T + r) * ld + c] : 0.0;
        }
    };
    if (k0 < k1) fetch(k0);
    for (int k = k0; k < k1; k += kPairs) {
#pragma unroll
        for (int u = 0; u < kPairs; ++u) { (kAT ? as[u][c][r] : as[u][r][c]) = sign * an[u]; bs[u][r][c] = bn[u]; }
        __syncthreads();
        if (k + kPairs < k1) fetch(k + kPairs);
#pragma unroll
        for (int u = 0; u < kPairs; ++u)
#pragma unroll
            for (int q = 0; q < T; ++q) s = __builtin_fma(as[u][r][q], bs[u][q][c], s);
        __syncthreads();
    }
    return s;
}

// X = L11^{-1}, one workgroup per 16-column strip: X_i = L_ii^{-1} (E_i - sum_{k < i} L_ik X_k) down the
// row tiles; thread (r, c) owns one element of the tile
__global__ void __launch_bounds__(256) k_node_inverse(const SetupBlock* __restrict__ blocks, const int2* __restrict__ strips,
                                                      const double* __restrict__ L, double* X) {
    __shared__ double ls[kPairs][T][T + 1], xs[kPairs][T][T + 1];
    const int2 st = strips[blockIdx.x];
    const SetupBlock B = blocks[st.x];
    const int r = threadIdx.x >> 4, c = threadIdx.x & 15, ct = st.y;
    const long long np = (long long)B.nk * T;
    const double* Lb = L + B.l;
    double* Xb = X + B.x + ct * T;  // the strip's columns
    for (int it = 0; it < ct; ++it) Xb[(it * T + r) * np + c] = 0.0;
    for (int it = ct; it < B.nk; ++it) {
        const double diag = Lb[(it * T + r) * np + it * T + c];
        double s = tile_products(it == ct && r == c ? 1.0 : 0.0, -1.0, Lb + it * T * np, Xb, np, ct, it, ls, xs);
        ls[0][r][c] = diag;
        __syncthreads();
        // forward substitution with the 16x16 diagonal tile, a row at a time
        for (int k = 0; k < T; ++k) {
            if (r == k) { s /= ls[0][k][k]; xs[0][k][c] = s; }
            __syncthreads();
            if (r > k) s = __builtin_fma(-ls[0][r][k], xs[0][k][c], s);
        }
        Xb[(it * T + r) * np + c] = s;
        __syncthreads();  // the next row tile reads it (and the LDS is reused)
    }
}

// forward operator, one workgroup per row tile: S = D Linv - I rounded to float (and D^-2), or W = L21 Linv (double sums);
// of a closed block the inverse Linv^T Linv (double sums), a tile and its mirror image from the same sums
__global__ void __launch_bounds__(256) k_node_forward_tiles(const SetupBlock* __restrict__ blocks, const int2* __restrict__ rows,
                                                            const double* __restrict__ L, const double* __restrict__ X,
                                                            float* __restrict__ tiles, float* __restrict__ scale) {
    __shared__ double ls[kPairs][T][T + 1], xs[kPairs][T][T + 1];
    const int2 rw = rows[blockIdx.x];
    const SetupBlock B = blocks[rw.x];
    const int r = threadIdx.x >> 4, c = threadIdx.x & 15, rt = rw.y;
    const long long np = (long long)B.nk * T;
    const double* Xb = X + B.x;
    if (!B.nrk) {
        const int at = ((c >> 2) * 16 + r) * 4 + (c & 3), mirror = ((r >> 2) * 16 + c) * 4 + (r & 3);
        float* M = tiles + (size_t)B.fwd * 256;
        for (int j = 0; j <= rt; ++j) {
            const double v = tile_products<true>(0.0, 1.0, Xb + rt * T, Xb + j * T, np, rt, B.nk, ls, xs);
            const bool diag = j == rt && r == c;
            const float f = diag ? 0.f : (float)v;
            if (diag) scale[B.scale + rt * T + r] = (float)v;
            M[((size_t)rt * B.nk + j) * 256 + at] = f;
            if (j < rt) M[((size_t)j * B.nk + rt) * 256 + mirror] = f;
        }
        return;
    }
    float* out = tiles + ((size_t)B.fwd + fwd_row(rt, B.nk)) * 256 + ((c >> 2) * 16 + r) * 4 + (c & 3);
    if (rt < B.nk) {
        const double d = L[B.l + (rt * T + r) * np + rt * T + r];
        for (int j = 0; j <= rt; ++j) {
            const double v = Xb[(rt * T + r) * np + j * T + c];
            out[(size_t)j * 256] = j == rt && r == c ? 0.f : (float)(d * v);
        }
        if (c == 0) scale[B.scale + rt * T + r] = (float)(1.0 / (d * d));
        return;
    }
    const double* Lr = L + B.l + (long long)rt * T * np;
    for (int j = 0; j < B.nk; ++j)
        out[(size_t)j * 256] = (float)tile_products(0.0, 1.0, Lr, Xb + j * T, np, j, B.nk, ls, xs);
}

// backward operator from the forward one: row tile rt holds the transposes of the forward tiles
// (kt, rt), kt >= rt, and the negated transposes of the W tiles (a, rt)
__global__ void __launch_bounds__(256) k_node_backward_tiles(const SetupBlock* __restrict__ blocks, const int2* __restrict__ rows,
                                                             float* __restrict__ tiles) {
    const int2 rw = rows[blockIdx.x];
    const SetupBlock B = blocks[rw.x];
    const int r = threadIdx.x >> 4, c = threadIdx.x & 15, rt = rw.y;
    const int to = ((c >> 2) * 16 + r) * 4 + (c & 3), from = ((r >> 2) * 16 + c) * 4 + (r & 3);  // element (r, c) from (c, r)
    float* out = tiles + ((size_t)B.bwd + bwd_row(rt, B.nk, B.nrk)) * 256 + to;
    const float* in = tiles + (size_t)B.fwd * 256 + from;
    for (int kt = rt; kt < B.nk + B.nrk; ++kt) {
        const float v = in[(size_t)(fwd_row(kt, B.nk) + rt) * 256];
        out[(size_t)(kt - rt) * 256] = kt < B.nk ? v : -v;
    }
}

template <class K, class... A>
void launch(K kernel, int grid, int waves, size_t lds, hipStream_t s, A... a) {
    hipLaunchKernelGGL(kernel, dim3((unsigned)grid), dim3((unsigned)(waves * 64)), lds, s, a...);
}

// the kernels may use the whole LDS of a CU for their operand vectors (a default launch stops at 64 KiB)
template <class K>
void allow_lds(K kernel) {
    hdd_check(hipFuncSetAttribute(reinterpret_cast<const void*>(kernel), hipFuncAttributeMaxDynamicSharedMemorySize,
                                  (int)(NodePlanHost::kMaxLdsFloats * sizeof(float))),
              "dense-node kernels' LDS");
}

}  // namespace

bool NodePlan::build(const std::vector<const SupernodalFactor*>& F, const std::vector<int>& offsets, const std::vector<int>& prob_of) {
    NodePlanHost P;
    if (!build_nodeplan(F, offsets, prob_of, P)) return false;
    bool wide = false;
    for (const auto& L : P.levels) wide = wide || std::max(L.fwd_lds, L.bwd_lds) * sizeof(float) > 48 * 1024;
    if (wide) {
        allow_lds(k_node_fwd<4, false>); allow_lds(k_node_fwd<16, false>);
        allow_lds(k_node_fwd<4, true>); allow_lds(k_node_fwd<16, true>);
        allow_lds(k_node_bwd<4>); allow_lds(k_node_bwd<16>);
    }
    n = P.n;
    levels = P.levels;
    fwd.upload(P.fwd); bwd.upload(P.bwd);
    inst_prob.upload(P.inst_prob);
    orig.upload(P.orig);
    P.zidx.resize(std::max<size_t>(1, P.zidx.size()), P.ysize); zidx.upload(P.zidx);
    P.more.resize(std::max<size_t>(1, P.more.size()), 0); more.upload(P.more);
    P.pos_c.resize(std::max<size_t>(1, P.pos_c.size()), NodePos{P.csize, P.csize});
    pos_y.upload(P.pos_y); pos_c.upload(P.pos_c);
    tiles.alloc((size_t)P.tiles * 256); scale.alloc(P.scales);
    t.alloc(P.ysize); y.alloc(P.ysize); z.alloc((size_t)P.ysize + 1); c.alloc((size_t)P.csize + 1);
    // the blocks in chunks: their supernodes' columns uploaded and put in place, inverted and packed
    auto doubles = [](const NodePlanHost::Block& B) { return (size_t)(B.nk + B.nrk) * T * B.nk * T; };
    size_t largest = 0, total = 0;
    for (const auto& B : P.blocks) { largest = std::max(largest, doubles(B)); total += doubles(B); }
    const size_t cap = std::min(total, std::max(largest, NodePlanHost::kSetupChunk));
    DBuf<double> dL, dX;
    hdd_check(hipMalloc(&dL.p, cap * sizeof(double)), "hipMalloc"); dL.n = cap;
    size_t xcap = 0;
    std::vector<std::pair<size_t, size_t>> chunks;
    for (size_t i = 0; i < P.blocks.size();) {
        size_t used = 0, xs = 0, k = i;
        while (k < P.blocks.size() && (k == i || used + doubles(P.blocks[k]) <= cap)) {
            used += doubles(P.blocks[k]);
            xs += (size_t)P.blocks[k].nk * T * P.blocks[k].nk * T;
            ++k;
        }
        xcap = std::max(xcap, xs);
        chunks.push_back({i, k});
        i = k;
    }
    hdd_check(hipMalloc(&dX.p, xcap * sizeof(double)), "hipMalloc"); dX.n = xcap;
    for (auto& ch : chunks) {
        std::vector<SetupBlock> sb;
        std::vector<int2> strips, rows, brows;
        long long l = 0, xo = 0;
        for (size_t k = ch.first; k < ch.second; ++k) {
            const NodePlanHost::Block& B = P.blocks[k];
            const int id = (int)sb.size();
            sb.push_back({l, xo, B.nk, B.nrk, B.fwd, B.bwd, B.scale, 0});
            l += (long long)doubles(B);
            xo += (long long)B.nk * T * B.nk * T;
            for (int r = 0; r < B.nk; ++r) {
                strips.push_back(make_int2(id, r));
                if (B.nrk) brows.push_back(make_int2(id, r));
            }
            for (int r = 0; r < B.nk + B.nrk; ++r) rows.push_back(make_int2(id, r));
        }
        std::vector<SetupSupernode> ss;
        std::vector<std::pair<const SupernodalFactor*, int>> from;
        std::vector<int> list, at;
        long long packed = 0;
        for (size_t k = ch.first; k < ch.second; ++k) {
            const NodePlanHost::Block& B = P.blocks[k];
            node_block_rows(B, at);
            int col = 0, first = (int)list.size();
            list.insert(list.end(), at.begin(), at.end());
            for (int g : B.sns) {
                const int n = B.f->sn[g].n, nr = (int)B.f->sn[g].rows.size(), np = B.nk * T;
                ss.push_back({packed, sb[k - ch.first].l, np, col, n, nr, first, col ? np : B.n, np, 0});
                from.push_back({B.f, g});
                packed += (long long)n * n + (long long)nr * n;
                col += n;
                first += nr;
            }
        }
        std::vector<double> host(packed);
#pragma omp parallel for schedule(dynamic, 16)
        for (size_t k = 0; k < ss.size(); ++k) {
            const std::vector<double>&a = from[k].first->L11[from[k].second], &b = from[k].first->L21[from[k].second];
            std::copy(a.begin(), a.end(), host.begin() + ss[k].src);
            std::copy(b.begin(), b.end(), host.begin() + ss[k].src + (long long)a.size());
        }
        DBuf<SetupBlock> dsb; dsb.upload(sb);
        DBuf<int2> dst, drw, dbr;
        dst.upload(strips); drw.upload(rows);
        if (!brows.empty()) dbr.upload(brows);
        DBuf<SetupSupernode> dss; dss.upload(ss);
        DBuf<int> dlist; dlist.upload(list.empty() ? std::vector<int>(1, 0) : list);
        DBuf<double> dsrc; dsrc.upload(host);
        hdd_check(hipMemset(dL.p, 0, (size_t)l * sizeof(double)), "node blocks");
        launch(k_node_columns, (int)ss.size(), 4, 0, nullptr, (const SetupSupernode*)dss.p, (const int*)dlist.p, (const double*)dsrc.p, dL.p);
        launch(k_node_inverse, (int)strips.size(), 4, 0, nullptr, (const SetupBlock*)dsb.p, (const int2*)dst.p, (const double*)dL.p, dX.p);
        launch(k_node_forward_tiles, (int)rows.size(), 4, 0, nullptr, (const SetupBlock*)dsb.p, (const int2*)drw.p, (const double*)dL.p,
               (const double*)dX.p, tiles.p, scale.p);
        if (!brows.empty())
            launch(k_node_backward_tiles, (int)brows.size(), 4, 0, nullptr, (const SetupBlock*)dsb.p, (const int2*)dbr.p, tiles.p);
        hdd_check(hipGetLastError(), "node blocks");
        hdd_check(hipStreamSynchronize(nullptr), "node blocks");
    }
    return true;
}

size_t NodePlan::bytes() const {
    return (fwd.n + bwd.n) * sizeof(NodeItem) + (inst_prob.n + orig.n + zidx.n + more.n) * 4 +
           (pos_y.n + pos_c.n) * 8 + (tiles.n + scale.n + t.n + y.n + z.n + c.n) * 4;
}

void NodePlan::solve(const float* b, float* x, const int* active, hipStream_t s) {
    auto fwd_level = [&](const NodePlanHost::Level& L) {
        if (L.children)
            hipLaunchKernelGGL(k_node_children, dim3((unsigned)((L.y1 - L.y0 + L.c1 - L.c0 + 255) / 256)), dim3(256), 0, s, L.y0, L.y1, L.c0, L.c1,
                               (const NodePos*)pos_y.p, (const NodePos*)pos_c.p, (const int*)more.p, (const int*)orig.p, b, t.p, c.p);
        auto go = [&](auto kernel) {
            launch(kernel, L.fwd1 - L.fwd0, L.fwd_waves, L.fwd_lds * sizeof(float), s, (const NodeItem*)fwd.p + L.fwd0, (const int*)inst_prob.p,
                   active, (const int*)orig.p, (const float*)t.p,
                   (const float*)tiles.p, (const float*)scale.p, b, y.p, c.p, z.p, x);
        };
        if (L.fwd_waves == 4) { if (L.children) go(k_node_fwd<4, true>); else go(k_node_fwd<4, false>); }
        else { if (L.children) go(k_node_fwd<16, true>); else go(k_node_fwd<16, false>); }
    };
    auto bwd_level = [&](const NodePlanHost::Level& L) {
        auto go = [&](auto kernel) {
            launch(kernel, L.bwd1 - L.bwd0, L.bwd_waves, L.bwd_lds * sizeof(float), s, (const NodeItem*)bwd.p + L.bwd0, (const int*)inst_prob.p,
                   active, (const int*)orig.p, (const int*)zidx.p, (const float*)tiles.p,
                   (const float*)y.p, z.p, x);
        };
        if (L.bwd_waves == 4) go(k_node_bwd<4>);
        else go(k_node_bwd<16>);
    };
    for (const auto& L : levels) if (L.fwd1 > L.fwd0) fwd_level(L);
    for (auto L = levels.rbegin(); L != levels.rend(); ++L) if (L->bwd1 > L->bwd0) bwd_level(*L);
}

}  // namespace hdd
