// emst_kernels.hip -- gfx950 kernels of the EMST engine.
//
// Stages (reference rows they implement, paths relative to the reference root):
//   bbox / params / rescale ..... InputRW.h:541-559, SolutionEMST.cu:305-379
//   curve keys + radix sort ..... the cell-grid build (count, wave-level scan,
//                                 scatter); cells are key prefixes
//   gather / tree ............... leaf cells of <= bucket points with tight boxes
//   cone search ................. NodeComputeOctantMD::computeOctants
//                                 (NodeEMST.h:1018-1296): per point, the nearest
//                                 point of each of the 2D x 2^(D-1) cones
//   round kernels ............... search (NodeEMST.h:1303-1384), component list +
//                                 min pair (NodeEMST.h:817-955), hooking
//                                 (EMSTOperators.h:1267-1303), flatten
//                                 (EMSTOperators.h:412-433)
//   weight ...................... K_EMST_evaluate_ST (EMSTOperators.h:262-292)
//   cell grid ................... ViewGridQuadMD::findCell (ViewGrid.h:339-359)
//
// Squared distances are fl(fl(dx*dx) + dy*dy) [+ dz*dz] with each "+ a*a"
// fused (__builtin_fmaf); the file is built with -ffp-contract=off so no other
// operation is contracted.
#include "emst_internal.h"

namespace emst {

namespace {

constexpr int kBlock = 256;

__device__ __forceinline__ float d2_of(float dx, float dy) { return __builtin_fmaf(dy, dy, dx * dx); }
__device__ __forceinline__ float d2_of(float dx, float dy, float dz)
{
    return __builtin_fmaf(dz, dz, __builtin_fmaf(dy, dy, dx * dx));
}

// Order-preserving float <-> uint maps for atomic min/max of floats.
__device__ __forceinline__ uint32_t f2ord(float f)
{
    uint32_t u = __float_as_uint(f);
    return (u & 0x80000000u) ? ~u : (u | 0x80000000u);
}
__device__ __forceinline__ float ord2f(uint32_t u)
{
    return __uint_as_float((u & 0x80000000u) ? (u & 0x7fffffffu) : ~u);
}

__device__ __forceinline__ uint64_t lanemask_lt()
{
    const int lane = __lane_id();
    return lane == 0 ? 0ull : (~0ull >> (64 - lane));
}

// maximum over each aligned group of 8 lanes, by DPP moves within rows (no
// LDS round trip): swap neighbours, swap pairs, then mirror the half row
// (lane i of the 8 reads lane 7 - i)
__device__ __forceinline__ uint32_t group8_max_u32(uint32_t v)
{
    v = max(v, (uint32_t)__builtin_amdgcn_mov_dpp((int)v, 0xB1, 0xF, 0xF, false));     // quad_perm [1,0,3,2]
    v = max(v, (uint32_t)__builtin_amdgcn_mov_dpp((int)v, 0x4E, 0xF, 0xF, false));     // quad_perm [2,3,0,1]
    v = max(v, (uint32_t)__builtin_amdgcn_mov_dpp((int)v, 0x141, 0xF, 0xF, false));    // row_half_mirror
    return v;
}

// ------------------------------------------------------------ clouds
// largest c with cl[c].pos <= p (the cloud holding global point p)
__device__ __forceinline__ int find_cloud(const Cloud* cl, int ncl, int64_t p)
{
    int lo = 0, hi = ncl - 1;
    while (lo < hi) {
        const int mid = (lo + hi + 1) >> 1;
        if (cl[mid].pos <= p) lo = mid;
        else hi = mid - 1;
    }
    return lo;
}

// largest c with cl[c].lbase <= g (the cloud holding global leaf g)
// This file is built with -fno-honor-nans (the kernels then skip the
// canonicalising moves the compiler puts before fminf / fmaxf inputs): every
// coordinate is checked finite before any search runs, and the tests for NaN
// and infinity look at the bits, passed through an empty asm statement so
// that the compiler cannot turn them back into floating-point class tests
// (which it would then fold under the no-NaN assumption).
__device__ __forceinline__ uint32_t opaque_bits(float x)
{
    uint32_t b = __float_as_uint(x);
    asm("" : "+v"(b));
    return b;
}
__device__ __forceinline__ bool finite_bits(float x)
{
    return (opaque_bits(x) & 0x7f800000u) != 0x7f800000u;
}
// x > 0 and finite
__device__ __forceinline__ bool positive_finite(float x)
{
    return opaque_bits(x) - 1u < 0x7f7fffffu;
}

__device__ __forceinline__ int find_cloud_leaf(const Cloud* cl, int ncl, int64_t g)
{
    int lo = 0, hi = ncl - 1;
    while (lo < hi) {
        const int mid = (lo + hi + 1) >> 1;
        if (cl[mid].lbase <= g) lo = mid;
        else hi = mid - 1;
    }
    return lo;
}

// the cloud whose tree block b is (k_tree_low)
__device__ __forceinline__ int find_cloud_block(const Cloud* cl, int ncl, int64_t b)
{
    int lo = 0, hi = ncl - 1;
    while (lo < hi) {
        const int mid = (lo + hi + 1) >> 1;
        if (cl[mid].tbase <= b) lo = mid;
        else hi = mid - 1;
    }
    return lo;
}

// sorted positions [s0, s1) of leaf slot j of a cloud (empty past its leaves)
__device__ __forceinline__ void leaf_range(const LeafTable& lt, int64_t lfirst, int64_t nl, int64_t cend, int64_t j,
                                           int64_t& s0, int64_t& s1)
{
    if (j < nl) {
        s0 = lt.start[lfirst + j];
        s1 = lt.start[lfirst + j + 1];
    } else {
        s0 = s1 = cend;
    }
}

// ------------------------------------------------------------ bbox (A1)
// Params.pmin/pmax hold order-mapped uints during the reduction.
__global__ void k_bbox_init(Params* P, int ncl)
{
    const int c = blockIdx.x * blockDim.x + threadIdx.x;
    if (c >= ncl) return;
    uint32_t* lo = reinterpret_cast<uint32_t*>(P[c].pmin);
    uint32_t* hi = reinterpret_cast<uint32_t*>(P[c].pmax);
    for (int k = 0; k < 3; ++k) { lo[k] = 0xffffffffu; hi[k] = 0u; }
    P[c].nonfinite = 0;
}

// Each wave walks a contiguous chunk of global points with per-lane
// accumulators for the chunk's current cloud, merged into P[cloud] (wave
// reduction, then order-mapped atomics) whenever the cloud changes.
template <int D>
__global__ __launch_bounds__(kBlock) void k_bbox(const float* __restrict__ xyz, const Cloud* __restrict__ cl,
                                                int ncl, int64_t N, Params* __restrict__ P)
{
    const int lane = __lane_id();
    const int64_t wave = ((int64_t)blockIdx.x * blockDim.x + threadIdx.x) / 64;
    const int64_t nwaves = (int64_t)gridDim.x * blockDim.x / 64;
    const int64_t chunk = ((N + nwaves - 1) / nwaves + 63) / 64 * 64;
    const int64_t a = wave * chunk, b = min(N, a + chunk);
    uint32_t lo[D], hi[D];
    for (int k = 0; k < D; ++k) { lo[k] = 0xffffffffu; hi[k] = 0u; }
    uint32_t bad = 0;
    int cur = -1;
    auto flush = [&]() {
        for (int k = 0; k < D; ++k)
            for (int off = 32; off > 0; off >>= 1) {
                lo[k] = min(lo[k], (uint32_t)__shfl_xor((int)lo[k], off));
                hi[k] = max(hi[k], (uint32_t)__shfl_xor((int)hi[k], off));
            }
        const bool any_bad = __any(bad);
        if (lane == 0) {
            // the extremes only move outwards: a value already at least as far
            // out makes the atomic redundant (so for most waves once a few have run)
            uint32_t* plo = reinterpret_cast<uint32_t*>(P[cur].pmin);
            uint32_t* phi = reinterpret_cast<uint32_t*>(P[cur].pmax);
            for (int k = 0; k < D; ++k) {
                if (__atomic_load_n(&plo[k], __ATOMIC_RELAXED) > lo[k]) atomicMin(&plo[k], lo[k]);
                if (__atomic_load_n(&phi[k], __ATOMIC_RELAXED) < hi[k]) atomicMax(&phi[k], hi[k]);
            }
            if (any_bad) atomicOr(&P[cur].nonfinite, 1u);
        }
        for (int k = 0; k < D; ++k) { lo[k] = 0xffffffffu; hi[k] = 0u; }
        bad = 0;
    };
    for (int64_t i0 = a; i0 < b; i0 += 64) {
        const int64_t i = i0 + lane;
        const int c = i < b ? find_cloud(cl, ncl, i) : -1;
        uint64_t todo = __ballot(c >= 0);
        while (todo) {
            const int cc = __builtin_amdgcn_readfirstlane(__shfl(c, (int)__builtin_ctzll(todo)));
            if (cc != cur) {
                if (cur >= 0) flush();
                cur = cc;
            }
            const bool mine = c == cc;
            todo &= ~__ballot(mine);
            if (mine) {
                const float* q = xyz + i * D;
                for (int k = 0; k < D; ++k) {
                    const float v = q[k];
                    bad |= !finite_bits(v);
                    const uint32_t o = f2ord(v);
                    lo[k] = min(lo[k], o);
                    hi[k] = max(hi[k], o);
                }
            }
        }
    }
    if (cur >= 0) flush();
}

// One cloud: each thread takes points a grid apart, and a block merges its
// waves before it touches the cloud's extremes, so that a launch has as many
// atomics on them as blocks.  (With k_bbox's one per wave, of 8192, they
// queued on one cache line: 70 us at 1.3*10^5 points and 182 at 4*10^6, here
// 6 and 21.)  Four points in flight per thread: 10^7 3D points are read in
// 35 us (3.5 TB/s), with one at a time in 54.
constexpr int kBoxBlocks = 512;
constexpr int kBoxAhead = 4;  // points in flight per thread

template <int D>
__global__ __launch_bounds__(kBlock) void k_bbox_one(const float* __restrict__ xyz, int64_t N, Params* __restrict__ P)
{
    __shared__ uint32_t sh[2 * D + 1][kBlock / 64];
    uint32_t lo[D], hi[D];
    for (int k = 0; k < D; ++k) { lo[k] = 0xffffffffu; hi[k] = 0u; }
    uint32_t bad = 0;
    const int64_t stride = (int64_t)gridDim.x * kBlock;
    for (int64_t i0 = (int64_t)blockIdx.x * kBlock + threadIdx.x; i0 < N; i0 += kBoxAhead * stride) {
        float v[kBoxAhead][D];
#pragma unroll
        for (int u = 0; u < kBoxAhead; ++u) {
            // (past the end: the last point again, which changes nothing)
            const int64_t i = min(i0 + u * stride, N - 1);
#pragma unroll
            for (int k = 0; k < D; ++k) v[u][k] = xyz[i * D + k];
        }
#pragma unroll
        for (int u = 0; u < kBoxAhead; ++u)
#pragma unroll
            for (int k = 0; k < D; ++k) {
                bad |= !finite_bits(v[u][k]);
                const uint32_t o = f2ord(v[u][k]);
                lo[k] = min(lo[k], o);
                hi[k] = max(hi[k], o);
            }
    }
    const int w = threadIdx.x / 64, lane = __lane_id();
#pragma unroll
    for (int k = 0; k < D; ++k) {
        for (int off = 32; off > 0; off >>= 1) {
            lo[k] = min(lo[k], (uint32_t)__shfl_xor((int)lo[k], off));
            hi[k] = max(hi[k], (uint32_t)__shfl_xor((int)hi[k], off));
        }
        if (lane == 0) {
            sh[2 * k][w] = lo[k];
            sh[2 * k + 1][w] = hi[k];
        }
    }
    const bool any_bad = __any(bad);
    if (lane == 0) sh[2 * D][w] = any_bad ? 1u : 0u;
    __syncthreads();
    const int t = threadIdx.x;
    if (t > 2 * D) return;
    uint32_t v = sh[t][0];
    for (int ww = 1; ww < kBlock / 64; ++ww)
        v = t == 2 * D ? (v | sh[t][ww]) : ((t & 1) ? max(v, sh[t][ww]) : min(v, sh[t][ww]));
    if (t == 2 * D) {
        if (v) atomicOr(&P->nonfinite, 1u);
    } else if (t & 1) {
        atomicMax(reinterpret_cast<uint32_t*>(P->pmax) + t / 2, v);
    } else {
        atomicMin(reinterpret_cast<uint32_t*>(P->pmin) + t / 2, v);
    }
}

// ---------------------------------------------------------- params (A2)
// wg = (double)(pMax.x - pMin.x) etc. are float subtractions widened to double,
// _wnd / unitX in double (SolutionEMST.cu:305-342).  The rescaled extremes are
// the rescaled box corners: the map p -> (p - pMin) * unitXf is monotone.
// One thread per cloud; key quantisation uses mbits bits per axis.
__global__ void k_params(Params* Pa, const Cloud* __restrict__ cl, int ncl, int dim, int mbits)
{
    const int c = blockIdx.x * blockDim.x + threadIdx.x;
    if (c >= ncl) return;
    Params* P = Pa + c;
    uint32_t* plo = reinterpret_cast<uint32_t*>(P->pmin);
    uint32_t* phi = reinterpret_cast<uint32_t*>(P->pmax);
    const int64_t n = cl[c].n;
    for (int k = 0; k < 3; ++k) {
        if (k < dim && n > 0) {
            P->pmin[k] = ord2f(plo[k]);
            P->pmax[k] = ord2f(phi[k]);
        } else {
            P->pmin[k] = 0.f;
            P->pmax[k] = 0.f;
        }
    }
    double wg = (double)(P->pmax[0] - P->pmin[0]);
    double hg = (double)(P->pmax[1] - P->pmin[1]);
    double dg = dim >= 3 ? (double)(P->pmax[2] - P->pmin[2]) : 0.0;
    if (wg == 0) wg = 1;
    if (hg == 0) hg = 1;
    const double nn = (double)n;
    double wnd = sqrt(nn * wg / hg) * 2;
    if (dim >= 3 && dg != 0) wnd = pow((nn * wg * wg) / (hg * dg), 0.333);
    const double unit = (ceil(wnd) + 1) / wg;
    P->unit_x = unit;
    const float fu = (float)unit;
    P->unit_xf = fu;
    float mx = 0.f;
    for (int k = 0; k < 3; ++k) {
        P->newmax[k] = k < dim ? (P->pmax[k] - P->pmin[k]) * fu : 0.f;
        mx = fmaxf(mx, P->newmax[k]);
    }
    const double maxq = (double)((1ull << mbits) - 1);
    P->qscale = mx > 0 ? (float)(maxq / (double)mx) : 0.f;
}

// ------------------------------------------- rescale + curve keys (A2, A5)
__device__ __forceinline__ uint64_t spread3(uint64_t x)
{
    x &= 0x1fffff;
    x = (x | (x << 32)) & 0x1f00000000ffffull;
    x = (x | (x << 16)) & 0x1f0000ff0000ffull;
    x = (x | (x << 8)) & 0x100f00f00f00f00full;
    x = (x | (x << 4)) & 0x10c30c30c30c30c3ull;
    x = (x | (x << 2)) & 0x1249249249249249ull;
    return x;
}
__device__ __forceinline__ uint64_t spread2(uint64_t x)
{
    x &= 0xffffffffull;
    x = (x | (x << 16)) & 0x0000ffff0000ffffull;
    x = (x | (x << 8)) & 0x00ff00ff00ff00ffull;
    x = (x | (x << 4)) & 0x0f0f0f0f0f0f0f0full;
    x = (x | (x << 2)) & 0x3333333333333333ull;
    x = (x | (x << 1)) & 0x5555555555555555ull;
    return x;
}

// Hilbert index of D coordinates of `bits` bits (Skilling, "Programming the
// Hilbert curve", 2004: undo the rotations from the top bit down, Gray-code,
// interleave).  Like a Morton key its prefixes are boxes, halved one bit at a
// time, but consecutive cells share a face: the points of a run of sorted
// positions (a packet of 64 queries, its groups of 8, a leaf) lie in one
// compact piece of space, where a Morton run jumps at every cell boundary.
// Measured against Morton keys of the same bits: cone search 5.9 -> 4.5 ms at
// 10^6 uniform 3D points, 6.1 -> 4.4 at 3*10^6 in the 2.5D mode, 23.3 -> 18.5
// at 4*10^6 clustered ones; neighbour lists of 10^7 clustered points 5.2 ->
// 4.2 ms.  The key itself takes 0.05 ms more at 10^7 points.
template <int D>
__device__ __forceinline__ uint64_t hilbert_key(uint32_t x[D], int bits)
{
    for (int q = bits - 1; q > 0; --q) {
        const uint32_t low = (1u << q) - 1u;
#pragma unroll
        for (int i = 0; i < D; ++i) {
            // bit q set: invert x[0]'s low bits; clear: exchange them with x[i]'s
            const uint32_t inv = (uint32_t)((int32_t)(x[i] << (31 - q)) >> 31) & low;
            const uint32_t t = (x[0] ^ x[i]) & (low ^ inv);
            x[0] ^= t | inv;
            if (i > 0) x[i] ^= t;
        }
    }
#pragma unroll
    for (int i = 1; i < D; ++i) x[i] ^= x[i - 1];
    uint32_t t = x[D - 1];          // then bit j of t: the parity of x[D - 1]'s bits above j
    t ^= t >> 1;
    t ^= t >> 2;
    t ^= t >> 4;
    t ^= t >> 8;
    t ^= t >> 16;
    t >>= 1;
    uint64_t code = 0;
#pragma unroll
    for (int i = 0; i < D; ++i)
        code |= (D == 3 ? spread3(x[i] ^ t) : spread2(x[i] ^ t)) << (D - 1 - i);
    return code;
}

template <int D>
__global__ __launch_bounds__(kBlock) void k_rescale_keys(const float* __restrict__ xyz,
                                                           const Cloud* __restrict__ cl, int ncl,
                                                           int64_t N, int mbits,
                                                           const Params* __restrict__ Pa,
                                                           float* __restrict__ resc,
                                                           uint64_t* __restrict__ keys, int hilbert)
{
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= N) return;
    const int c = find_cloud(cl, ncl, i);
    const Params* P = Pa + c;
    const float* q = xyz + i * D;
    const float fu = P->unit_xf;
    const float qs = P->qscale;
    const uint32_t maxq = (uint32_t)((1ull << mbits) - 1);
    uint32_t cell[D];
    for (int k = 0; k < D; ++k) {
        float d = q[k] - P->pmin[k];                // PointE::operator- (Node.h:574-580)
        float v = d * fu;                           // PointE::operator*(float) (Node.h:588-593)
        resc[i * D + k] = v;
        float qf = v * qs;
        cell[k] = qf >= (float)maxq ? maxq : (uint32_t)qf;
    }
    uint64_t code = 0;
    if (hilbert)
        code = hilbert_key<D>(cell, mbits);
    else
        for (int k = 0; k < D; ++k) code |= (D == 3 ? spread3(cell[k]) : spread2(cell[k])) << k;
    if (ncl > 1) code |= (uint64_t)c << (mbits * D);
    keys[i] = code;
}

// the first active lane's v in every lane.  A load of one address by the
// whole wave is served in parts, so while other waves change the word its
// lanes can read different values; a value that steers the wave's control
// flow must then be one lane's (a partly active wave would also read zeros
// from the idle lanes in the shuffles of wave_min_u64).
__device__ __forceinline__ uint64_t wave_first_u64(uint64_t v)
{
    const uint32_t lo = (uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)v);
    const uint32_t hi = (uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)(v >> 32));
    return ((uint64_t)hi << 32) | lo;
}

// ------------------------------------------------------------------ scan
// Exclusive scan of uint32 in three passes: per-block scan of 1024 elements,
// scan of block totals (one block, chunked), add-back.
constexpr int kScanItems = 4;
constexpr int kScanTile = kBlock * kScanItems;

__device__ __forceinline__ uint32_t wave_incl_scan(uint32_t v)
{
    const int lane = __lane_id();
    for (int off = 1; off < 64; off <<= 1) {
        uint32_t t = (uint32_t)__shfl_up((int)v, off);
        if (lane >= off) v += t;
    }
    return v;
}

// Block-wide exclusive scan of one value per thread; returns the block total.
__device__ __forceinline__ uint32_t block_excl_scan(uint32_t v, uint32_t* sh, uint32_t& total)
{
    const int lane = __lane_id(), w = threadIdx.x / 64, nw = blockDim.x / 64;
    uint32_t inc = wave_incl_scan(v);
    if (lane == 63) sh[w] = inc;
    __syncthreads();
    if (threadIdx.x == 0) {
        uint32_t run = 0;
        for (int i = 0; i < nw; ++i) { uint32_t t = sh[i]; sh[i] = run; run += t; }
        sh[nw] = run;
    }
    __syncthreads();
    uint32_t r = sh[w] + inc - v;
    total = sh[nw];
    __syncthreads();
    return r;
}

__global__ __launch_bounds__(kBlock) void k_scan_local(const uint32_t* __restrict__ in,
                                                      uint32_t* __restrict__ out, int64_t n,
                                                      uint32_t* __restrict__ sums)
{
    __shared__ uint32_t sh[16];
    const int64_t base = (int64_t)blockIdx.x * kScanTile + (int64_t)threadIdx.x * kScanItems;
    uint32_t v[kScanItems];
    uint32_t s = 0;
    for (int j = 0; j < kScanItems; ++j) {
        v[j] = (base + j < n) ? in[base + j] : 0u;
        s += v[j];
    }
    uint32_t total;
    uint32_t run = block_excl_scan(s, sh, total);
    for (int j = 0; j < kScanItems; ++j) {
        if (base + j < n) out[base + j] = run;
        run += v[j];
    }
    if (threadIdx.x == 0) sums[blockIdx.x] = total;
}

__global__ __launch_bounds__(1024) void k_scan_top(uint32_t* sums, int64_t nb)
{
    __shared__ uint32_t sh[17];
    uint32_t carry = 0;
    for (int64_t base = 0; base < nb; base += 1024) {
        const int64_t i = base + threadIdx.x;
        uint32_t v = i < nb ? sums[i] : 0u;
        uint32_t total;
        uint32_t r = block_excl_scan(v, sh, total);
        if (i < nb) sums[i] = r + carry;
        carry += total;
        __syncthreads();
    }
}

__global__ __launch_bounds__(kBlock) void k_scan_add(uint32_t* __restrict__ out, int64_t n,
                                                    const uint32_t* __restrict__ sums)
{
    const int64_t base = (int64_t)blockIdx.x * kScanTile;
    const uint32_t add = sums[blockIdx.x];
    for (int j = threadIdx.x; j < kScanTile; j += kBlock)
        if (base + j < n) out[base + j] += add;
}

// few values: one block, each thread a run of them
constexpr int kScanOne = 4096;
__global__ __launch_bounds__(1024) void k_scan_one(const uint32_t* __restrict__ in, uint32_t* __restrict__ out, int n)
{
    __shared__ uint32_t sh[17];
    const int per = (n + 1023) / 1024;
    const int a = min(n, (int)threadIdx.x * per), b = min(n, a + per);
    uint32_t sum = 0;
    for (int i = a; i < b; ++i) sum += in[i];
    uint32_t total;
    uint32_t run = block_excl_scan(sum, sh, total);
    for (int i = a; i < b; ++i) {
        const uint32_t v = in[i];
        out[i] = run;
        run += v;
    }
}

// ------------------------------------------------------------ radix sort
// LSD by 8-bit digits, stable, (u64 key, u32 value) pairs.
//
// Many pairs: one pass over the keys counts every digit's values
// (k_rs_hist), then one launch per digit (k_rs_pass): a tile ranks its keys,
// publishes its digit counts, and finds the start of its runs by looking back
// over the counts of the tiles before it.  Tiles take their number from a
// ticket, so every tile looked at has already begun, and it publishes its
// counts before it looks back itself: each wait ends.
// Per tile of 4096 keys on 512 threads: each wave owns 512 consecutive keys
// and ranks equal digits with 8 ballots; the tile is put in digit order in
// LDS (keys, then values, in the same 32 KB) and written out in that order, so
// that consecutive threads store to consecutive addresses of a digit's run.
//
// A separate count and three scan launches per digit read every key twice and
// launched five times: 10^7 pairs of 48 bits 0.69 ms, now 0.58 (87 us a digit,
// 2.8 TB/s: runs of 16 keys a digit and tile write 128-byte pieces; with 256
// threads of 16 keys 94 us), 10^6 0.19 -> 0.15.
constexpr int kRsThreads = 512;
constexpr int kRsWaves = kRsThreads / 64;
constexpr int kRsItems = 8;
constexpr int kRsTile = kRsThreads * kRsItems;
constexpr int kRsMaxPasses = 8;
constexpr int kRsHistItems = 32;

// scratch words: tile states (u64, [pass][tile][256]), digit counts
// [pass][256], tickets [pass]
__host__ __device__ inline int64_t rs_tiles(int64_t n) { return (n + kRsTile - 1) / kRsTile; }

// lanes of the wave with the same digit (among valid ones)
__device__ __forceinline__ uint64_t digit_peers(uint32_t d, bool valid)
{
    uint64_t peers = __ballot(valid);
#pragma unroll
    for (int b = 0; b < 8; ++b) {
        const bool bit = (d >> b) & 1u;
        const uint64_t bb = __ballot(valid && bit);
        peers &= bit ? bb : ~bb;
    }
    return peers;
}

__global__ __launch_bounds__(kBlock) void k_rs_hist(const uint64_t* __restrict__ keys, int64_t n, int passes,
                                                   uint32_t* __restrict__ hist)
{
    __shared__ uint32_t h[kRsMaxPasses][256];
    for (int i = threadIdx.x; i < passes * 256; i += kBlock) (&h[0][0])[i] = 0;
    __syncthreads();
    const int64_t base = (int64_t)blockIdx.x * (kBlock * kRsHistItems);
    for (int j = 0; j < kRsHistItems; ++j) {
        const int64_t i = base + j * kBlock + threadIdx.x;
        if (i < n) {
            const uint64_t k = keys[i];
            for (int ps = 0; ps < passes; ++ps) atomicAdd(&h[ps][(k >> (8 * ps)) & 255u], 1u);
        }
    }
    __syncthreads();
    for (int i = threadIdx.x; i < passes * 256; i += kBlock) {
        const uint32_t v = (&h[0][0])[i];
        if (v) atomicAdd(&hist[i], v);
    }
}

constexpr uint64_t kRsCounts = 1ull << 62;      // a tile's own digit counts
constexpr uint64_t kRsPrefix = 2ull << 62;      // the counts of it and all tiles before it
constexpr uint64_t kRsValue = kRsCounts - 1;

__global__ __launch_bounds__(kRsThreads) void k_rs_pass(const uint64_t* __restrict__ kin, const uint32_t* __restrict__ vin,
                                                   uint64_t* __restrict__ kout, uint32_t* __restrict__ vout,
                                                   int64_t n, int pass, const uint32_t* __restrict__ hist,
                                                   unsigned long long* __restrict__ state,
                                                   uint32_t* __restrict__ ticket, int identity)
{
    __shared__ uint32_t cnt[kRsWaves][256];        // per wave and digit: counts, then the wave's first tile slot
    __shared__ uint32_t gstart[256];        // per digit: output position minus tile slot (modulo 2^32)
    __shared__ uint32_t wsum[8];
    __shared__ uint32_t tile_sh;
    __shared__ uint64_t stage[kRsTile];
    const int w = threadIdx.x / 64, lane = __lane_id(), d = threadIdx.x;
    if (threadIdx.x == 0) tile_sh = atomicAdd(ticket, 1u);
    for (int k = threadIdx.x; k < kRsWaves * 256; k += kRsThreads) (&cnt[0][0])[k] = 0;
    const uint32_t hd = d < 256 ? hist[d] : 0u;
    __syncthreads();
    const int64_t tile = tile_sh;
    const int64_t tbase = tile * kRsTile;
    const int64_t wbase = tbase + (int64_t)w * (kRsTile / kRsWaves);
    const int shift = 8 * pass;
    uint64_t key[kRsItems];
    uint32_t val[kRsItems], rank[kRsItems];
#pragma unroll
    for (int c = 0; c < kRsItems; ++c) {
        const int64_t i = wbase + c * 64 + lane;
        key[c] = i < n ? kin[i] : 0ull;
        val[c] = identity ? (uint32_t)i : (i < n ? vin[i] : 0u);
    }
    const uint64_t below = lanemask_lt();
#pragma unroll
    for (int c = 0; c < kRsItems; ++c) {
        const bool valid = wbase + c * 64 + lane < n;
        const uint32_t dg = (uint32_t)(key[c] >> shift) & 255u;
        const uint64_t peers = digit_peers(dg, valid);
        const uint32_t before = (uint32_t)__popcll(peers & below);
        rank[c] = valid ? cnt[w][dg] + before : 0u;
        __builtin_amdgcn_wave_barrier();
        if (valid && before == 0u) cnt[w][dg] += (uint32_t)__popcll(peers);
        __builtin_amdgcn_wave_barrier();
    }
    __syncthreads();
    // thread d < 256: the tile's count of digit d, published at once, and the
    // exclusive scans over the digits of the tile's counts and of all keys'
    uint32_t tot = 0, ls = 0, gs = 0;
    unsigned long long* mine = state + tile * 256 + d;
    if (d < 256) {
#pragma unroll
        for (int ww = 0; ww < kRsWaves; ++ww) {
            const uint32_t v = cnt[ww][d];
            cnt[ww][d] = tot;
            tot += v;
        }
        __hip_atomic_store(mine, (tile == 0 ? kRsPrefix : kRsCounts) | tot, __ATOMIC_RELAXED,
                           __HIP_MEMORY_SCOPE_AGENT);
        const uint32_t inc = wave_incl_scan(tot), ginc = wave_incl_scan(hd);
        if (lane == 63) {
            wsum[w] = inc;
            wsum[4 + w] = ginc;
        }
        ls = inc - tot;
        gs = ginc - hd;
    }
    __syncthreads();
    if (d < 256) {
        for (int ww = 0; ww < w; ++ww) {
            ls += wsum[ww];
            gs += wsum[4 + ww];
        }
#pragma unroll
        for (int ww = 0; ww < kRsWaves; ++ww) cnt[ww][d] += ls;
    }
    __syncthreads();
    // the keys in digit order, while the earlier tiles publish
#pragma unroll
    for (int c = 0; c < kRsItems; ++c) {
        if (wbase + c * 64 + lane < n) {
            rank[c] += cnt[w][(uint32_t)(key[c] >> shift) & 255u];
            stage[rank[c]] = key[c];
        }
    }
    if (d < 256) {
        uint32_t prev = 0;              // (fewer than 2^31 pairs)
        for (int64_t t = tile - 1; t >= 0; --t) {
            unsigned long long st;
            do {
                st = __hip_atomic_load(state + t * 256 + d, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            } while (st == 0ull);
            prev += (uint32_t)(st & kRsValue);
            if (st & kRsPrefix) break;
        }
        if (tile > 0)
            __hip_atomic_store(mine, kRsPrefix | (unsigned long long)(prev + tot), __ATOMIC_RELAXED,
                               __HIP_MEMORY_SCOPE_AGENT);
        gstart[d] = gs + prev - ls;
    }
    __syncthreads();
    const int tn = (int)min<int64_t>(kRsTile, n - tbase);
    uint32_t at[kRsItems];
#pragma unroll
    for (int j = 0; j < kRsItems; ++j) {
        const int sl = j * kRsThreads + threadIdx.x;
        if (sl < tn) {
            const uint64_t k = stage[sl];
            at[j] = gstart[(uint32_t)(k >> shift) & 255u] + (uint32_t)sl;
            kout[at[j]] = k;
        }
    }
    __syncthreads();
    uint32_t* sval = reinterpret_cast<uint32_t*>(stage);
#pragma unroll
    for (int c = 0; c < kRsItems; ++c)
        if (wbase + c * 64 + lane < n) sval[rank[c]] = val[c];
    __syncthreads();
#pragma unroll
    for (int j = 0; j < kRsItems; ++j) {
        const int sl = j * kRsThreads + threadIdx.x;
        if (sl < tn) vout[at[j]] = sval[sl];
    }
}

// Few pairs: every pass in one launch of one block, pairs in registers, put in
// order through LDS (key halves and values in turn).  Pairs past n are keys of
// all ones, which the stable order leaves at the end.  One pass of 8192 pairs
// takes 6 us, of 2048 3 us; a pass by k_rs_pass of one tile takes 9 and its
// launch.
constexpr int kRsSmallBlock = 1024;
constexpr int kRsSmallMax = 8192;

template <int ITEMS>
__global__ __launch_bounds__(kRsSmallBlock) void k_rs_small(uint64_t* __restrict__ keys, uint32_t* __restrict__ vals,
                                                           int n, int passes, int identity)
{
    constexpr int kWaves = kRsSmallBlock / 64;
    __shared__ uint32_t cnt[kWaves][256];
    __shared__ uint32_t wsum[4];
    __shared__ uint32_t ex[kRsSmallBlock * ITEMS];
    const int w = threadIdx.x / 64, lane = __lane_id();
    const int base = w * 64 * ITEMS + lane;
    uint64_t key[ITEMS];
    uint32_t val[ITEMS], slot[ITEMS];
#pragma unroll
    for (int c = 0; c < ITEMS; ++c) {
        const int i = base + c * 64;
        key[c] = i < n ? keys[i] : ~0ull;
        val[c] = identity ? (uint32_t)i : (i < n ? vals[i] : 0u);
    }
    const uint64_t below = lanemask_lt();
    for (int ps = 0; ps < passes; ++ps) {
        const int shift = 8 * ps;
        for (int k = threadIdx.x; k < kWaves * 256; k += kRsSmallBlock) (&cnt[0][0])[k] = 0;
        __syncthreads();
#pragma unroll
        for (int c = 0; c < ITEMS; ++c) {
            const uint32_t dg = (uint32_t)(key[c] >> shift) & 255u;
            const uint64_t peers = digit_peers(dg, true);
            const uint32_t before = (uint32_t)__popcll(peers & below);
            slot[c] = cnt[w][dg] + before;
            __builtin_amdgcn_wave_barrier();
            if (before == 0u) cnt[w][dg] += (uint32_t)__popcll(peers);
            __builtin_amdgcn_wave_barrier();
        }
        __syncthreads();
        // first slot of every wave's run of digit d: over the waves, then the digits
        uint32_t tot = 0, inc = 0;
        if (threadIdx.x < 256) {
            const int d = threadIdx.x;
            for (int ww = 0; ww < kWaves; ++ww) {
                const uint32_t v = cnt[ww][d];
                cnt[ww][d] = tot;
                tot += v;
            }
            inc = wave_incl_scan(tot);
            if (lane == 63) wsum[w] = inc;
        }
        __syncthreads();
        if (threadIdx.x < 256) {
            uint32_t start = inc - tot;
            for (int ww = 0; ww < w; ++ww) start += wsum[ww];
            for (int ww = 0; ww < kWaves; ++ww) cnt[ww][threadIdx.x] += start;
        }
        __syncthreads();
#pragma unroll
        for (int c = 0; c < ITEMS; ++c) slot[c] += cnt[w][(uint32_t)(key[c] >> shift) & 255u];
        // exchange: the halves of the keys, then the values
        uint32_t lo[ITEMS], hi[ITEMS];
#pragma unroll
        for (int c = 0; c < ITEMS; ++c) ex[slot[c]] = (uint32_t)key[c];
        __syncthreads();
#pragma unroll
        for (int c = 0; c < ITEMS; ++c) lo[c] = ex[base + c * 64];
        __syncthreads();
#pragma unroll
        for (int c = 0; c < ITEMS; ++c) ex[slot[c]] = (uint32_t)(key[c] >> 32);
        __syncthreads();
#pragma unroll
        for (int c = 0; c < ITEMS; ++c) hi[c] = ex[base + c * 64];
        __syncthreads();
#pragma unroll
        for (int c = 0; c < ITEMS; ++c) ex[slot[c]] = val[c];
        __syncthreads();
#pragma unroll
        for (int c = 0; c < ITEMS; ++c) {
            val[c] = ex[base + c * 64];
            key[c] = ((uint64_t)hi[c] << 32) | lo[c];
        }
        __syncthreads();
    }
#pragma unroll
    for (int c = 0; c < ITEMS; ++c) {
        const int i = base + c * 64;
        if (i < n) {
            keys[i] = key[c];
            vals[i] = val[c];
        }
    }
}

// -------------------------------------------------- gather sorted points
template <int D>
__global__ __launch_bounds__(kBlock) void k_gather_sorted(const float* __restrict__ resc,
                                                         const uint32_t* __restrict__ perm,
                                                         int64_t n, float4* __restrict__ pts,
                                                         int32_t* __restrict__ inv, uint32_t* __restrict__ ids)
{
    const int64_t s = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (s >= n) return;
    const uint32_t o = perm[s];
    ids[s] = o;
    float4 p;
    p.x = resc[(int64_t)o * D + 0];
    p.y = resc[(int64_t)o * D + 1];
    p.z = D == 3 ? resc[(int64_t)o * D + 2] : 0.f;
    p.w = __uint_as_float(o);
    pts[s] = p;
    inv[o] = (int32_t)s;
}

// ------------------------------------------------ coincident-point groups
// Identical points share a key, so each group lies inside one run of
// equal keys; the sort is stable over input order, so within a run positions
// ascend with input id and a group's first position holds its smallest id.
constexpr int kMixedRunMax = 1024;   // longest run holding >= 2 locations that is split
constexpr int kBigRun = 4096;        // longer runs are filled by the whole grid (k_dup_big)

__device__ __forceinline__ bool same_xyz(const float4& a, const float4& b)
{
    return a.x == b.x && a.y == b.y && a.z == b.z;
}

// append the lanes holding `take` to list, one atomic per wave
__device__ __forceinline__ void wave_append_u64(bool take, uint64_t v, uint64_t* list, uint32_t* counter)
{
    const uint64_t m = __ballot(take);
    if (m == 0ull) return;
    const int leader = __builtin_ctzll(m);
    uint32_t base = 0;
    if (__lane_id() == leader) base = atomicAdd(counter, (uint32_t)__popcll(m));
    base = (uint32_t)__shfl((int)base, leader);
    if (take) list[base + (uint32_t)__popcll(m & lanemask_lt())] = v;
}

// wave_append_u64 into a list of cap entries: one atomic per wave reserves
// the slots, and the lanes whose slot lies past the end are left out (the
// count may pass cap; its readers take min(count, cap), and every slot below
// cap is written by the lane that reserved it).  Returns this lane's taking
// part.  (A compare-and-swap loop that reserved only when all fitted queued
// the thousands of waves of one round on the count: 48 ms a round.)
__device__ __forceinline__ bool wave_append_capped_u64(bool take, uint64_t v, uint64_t* list, uint32_t* counter,
                                                       uint32_t cap)
{
    const uint64_t m = __ballot(take);
    if (m == 0ull) return false;
    const int leader = __builtin_ctzll(m);
    uint32_t base = 0;
    if (__lane_id() == leader) base = atomicAdd(counter, (uint32_t)__popcll(m));
    base = (uint32_t)__shfl((int)base, leader);
    const uint32_t slot = base + (uint32_t)__popcll(m & lanemask_lt());
    const bool in = take && slot < cap;
    if (in) list[slot] = v;
    return in;
}

// append the lanes holding `take` to list, one atomic per wave
__device__ __forceinline__ void wave_append(bool take, int32_t v, int32_t* list, uint32_t* counter)
{
    const uint64_t m = __ballot(take);
    if (m == 0ull) return;
    const int leader = __builtin_ctzll(m);
    uint32_t base = 0;
    if (__lane_id() == leader) base = atomicAdd(counter, (uint32_t)__popcll(m));
    base = (uint32_t)__shfl((int)base, leader);
    if (take) list[base + (uint32_t)__popcll(m & lanemask_lt())] = v;
}


// ------------------------------------------------------------ leaves
// Position i starts a leaf when it starts its cloud, or when the smallest
// prefix cell of the sorted keys that holds both i - 1 and i (the cell above
// their highest differing bit) has more than `bucket` points: its two halves
// then lie in different leaves.  The cell is contiguous around i, so two
// binary searches within `bucket` positions of i decide it.  Inside a run of
// equal keys longer than `bucket` a leaf starts every `bucket` points from
// the run's start.
__global__ __launch_bounds__(kBlock) void k_leaf_marks(const uint64_t* __restrict__ keys, int64_t n,
                                                      const Cloud* __restrict__ cl, int ncl, int bucket,
                                                      uint32_t* __restrict__ mark)
{
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const int c = find_cloud(cl, ncl, i);
    const int64_t c0 = cl[c].pos, c1 = cl[c].pos + cl[c].n;
    uint32_t m = 1u;
    if (i > c0) {
        const uint64_t a = keys[i - 1], b = keys[i];
        if (a != b) {
            const int h = 63 - __clzll(a ^ b);
            const uint64_t mask = h >= 63 ? 0ull : ~((2ull << h) - 1ull);
            const uint64_t pre = b & mask;
            int64_t lo = max(c0, i - bucket), hi = i - 1;
            while (lo < hi) {
                const int64_t mid = (lo + hi) >> 1;
                if ((keys[mid] & mask) == pre) hi = mid;
                else lo = mid + 1;
            }
            int64_t lo2 = i, hi2 = min(c1, i + bucket) - 1;
            while (lo2 < hi2) {
                const int64_t mid = (lo2 + hi2 + 1) >> 1;
                if ((keys[mid] & mask) == pre) lo2 = mid;
                else hi2 = mid - 1;
            }
            m = lo2 - lo + 1 > bucket ? 1u : 0u;
        } else {
            int64_t lo = i - 1, step = 1;
            while (lo - step >= c0 && keys[lo - step] == b) {
                lo -= step;
                step <<= 1;
            }
            int64_t a0 = max(c0, lo - step), b0 = lo;
            while (a0 < b0) {
                const int64_t mid = (a0 + b0) >> 1;
                if (keys[mid] == b) b0 = mid;
                else a0 = mid + 1;
            }
            const bool long_run = a0 + bucket < c1 && keys[a0 + bucket] == b;
            m = long_run && (i - a0) % bucket == 0 ? 1u : 0u;
        }
    }
    mark[i] = m;
}

// idx: exclusive scan of mark.  start[leaf] = its first position, of[p] =
// the leaf of p, start[leaves] = n.
__global__ __launch_bounds__(kBlock) void k_leaf_fill(const uint32_t* __restrict__ mark,
                                                     const uint32_t* __restrict__ idx, int64_t n,
                                                     int32_t* __restrict__ start, int32_t* __restrict__ of)
{
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const uint32_t g = idx[i] + mark[i] - 1u;
    of[i] = (int32_t)g;
    if (mark[i]) start[idx[i]] = (int32_t)i;
    if (i == n - 1) start[g + 1] = (int32_t)n;
}

// First leaf of every cloud (every non-empty cloud starts a leaf), and the
// count.  layout: also lay the clouds' hierarchies out in the cloud table as
// the host does after reading the counts (L = the power of two at or above
// the cloud's leaf count, lbase = the sum of the earlier clouds' L), inside
// slot counts the host fixed beforehand (the table's L on entry);
// C->invalid flags a cloud with more leaves than those slots, or with a NaN
// or Inf coordinate.  One block.
__global__ __launch_bounds__(1024) void k_cloud_leaves(Cloud* __restrict__ cl, int ncl,
                                                      const uint32_t* __restrict__ mark,
                                                      const uint32_t* __restrict__ idx, int64_t n,
                                                      int32_t* __restrict__ out, const Params* __restrict__ P,
                                                      Counters* C, int layout)
{
    __shared__ int64_t part[1024];
    if (threadIdx.x == 0) C->invalid = 0u;
    const int32_t total = n > 0 ? (int32_t)(idx[n - 1] + mark[n - 1]) : 0;
    for (int c = threadIdx.x; c <= ncl; c += blockDim.x)
        out[c] = (c < ncl && cl[c].pos < n) ? (int32_t)idx[cl[c].pos] : total;
    __syncthreads();
    if (!layout) return;
    // each thread a run of consecutive clouds
    const int per = (ncl + (int)blockDim.x - 1) / (int)blockDim.x;
    const int c0 = min(ncl, (int)threadIdx.x * per), c1 = min(ncl, c0 + per);
    int64_t sum = 0;
    for (int c = c0; c < c1; ++c) {
        const int64_t nl = (int64_t)out[c + 1] - out[c];
        if (nl > cl[c].L || P[c].nonfinite) atomicOr(&C->invalid, 1u);
        int64_t L = 1;
        while (L < nl) L <<= 1;
        cl[c].lfirst = out[c];
        cl[c].nl = nl;
        cl[c].L = L;
        sum += L;
    }
    part[threadIdx.x] = sum;
    __syncthreads();
    if (threadIdx.x == 0) {
        int64_t run = 0;
        for (int t = 0; t < (int)blockDim.x; ++t) {
            const int64_t v = part[t];
            part[t] = run;
            run += v;
        }
    }
    __syncthreads();
    int64_t run = part[threadIdx.x];
    for (int c = c0; c < c1; ++c) {
        cl[c].lbase = run;
        run += cl[c].L;
    }
}

__global__ __launch_bounds__(kBlock) void k_zero_u32(uint32_t* __restrict__ p, int64_t n)
{
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) p[i] = 0u;
}

// rep[] = -1 everywhere; the first position of every run of >= 2 equal keys is queued
__global__ __launch_bounds__(kBlock) void k_dup_runs(const uint64_t* __restrict__ keys, int64_t n,
                                                    int32_t* __restrict__ rep, int32_t* __restrict__ runs,
                                                    Counters* __restrict__ C)
{
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i == 0) C->dup_big = 0;
    if (i >= n) return;
    rep[i] = -1;
    const uint64_t k = keys[i];
    const bool head = i == 0 || keys[i - 1] != k;
    if (head && i + 1 < n && keys[i + 1] == k) runs[atomicAdd(&C->dup_runs, 1u)] = (int32_t)i;
}

// One wave per run (grid-stride over the queued runs).  A run at one location
// is one group; a run over several locations (distinct points closer than a
// key cell) of at most kMixedRunMax points is split by pairwise
// comparison; a longer one sets dup_overflow, which turns grouping off.
// A run of more than kBigRun points (a heavily repeated location: one wave
// would walk it alone while the grid idles) gets its group slot and list
// range here and is checked and filled by k_dup_big; its (start, end, list
// base) go to the back of `runs`, entry k at runs[n - 3k - 3 ..]: the front
// holds at most n / 2 run heads and the back at most 3n / (kBigRun + 1).
__global__ __launch_bounds__(kBlock) void k_dup_group(const uint64_t* __restrict__ keys,
                                                     const float4* __restrict__ pts, int64_t n,
                                                     int32_t* __restrict__ rep,
                                                     int32_t* __restrict__ runs,
                                                     int32_t* __restrict__ list, int32_t* __restrict__ gslot,
                                                     Counters* __restrict__ C)
{
    const int lane = __lane_id();
    const int64_t nwaves = (int64_t)gridDim.x * (kBlock / 64);
    const int64_t nruns = C->dup_runs;
    for (int64_t w = (int64_t)blockIdx.x * (kBlock / 64) + threadIdx.x / 64; w < nruns; w += nwaves) {
        const int64_t s = runs[w];
        const uint64_t key = keys[s];
        // run end: the first larger key (the keys are sorted)
        int64_t lo = s + 1, hi = n;
        while (lo < hi) {
            const int64_t mid = lo + (hi - lo) / 2;
            if (keys[mid] == key) lo = mid + 1;
            else hi = mid;
        }
        const int64_t e = lo;
        if (e - s > kBigRun) {
            if (lane == 0) {
                gslot[s] = (int32_t)atomicAdd(&C->dup_groups, 1u);
                const uint32_t base = atomicAdd(&C->dup_points, (uint32_t)(e - s));
                const int64_t k = (int64_t)atomicAdd(&C->dup_big, 1u);
                runs[n - 3 * k - 3] = (int32_t)s;
                runs[n - 3 * k - 2] = (int32_t)e;
                runs[n - 3 * k - 1] = (int32_t)base;
            }
            continue;
        }
        const float4 head = pts[s];
        bool mixed = false;
        // four independent loads per lane per trip
        for (int64_t b = s; b < e; b += 256) {
#pragma unroll
            for (int u = 0; u < 4; ++u) {
                const int64_t i = b + 64 * u + lane;
                if (i < e) mixed |= !same_xyz(pts[i], head);
            }
        }
        if (__ballot(mixed) == 0ull) {
            // one group: its list entries are reserved in one step
            uint32_t base = 0;
            if (lane == 0) {
                gslot[s] = (int32_t)atomicAdd(&C->dup_groups, 1u);
                base = atomicAdd(&C->dup_points, (uint32_t)(e - s));
            }
            base = (uint32_t)__shfl((int)base, 0);
            for (int64_t i = s + lane; i < e; i += 64) {
                rep[i] = (int32_t)s;
                list[base + (uint32_t)(i - s)] = (int32_t)i;
            }
        } else if (e - s <= kMixedRunMax) {
            for (int64_t b = s; b < e; b += 64) {
                const int64_t i = b + lane;
                const float4 me = i < e ? pts[i] : head;
                int64_t first = -1;
                int twins = 0;
                for (int64_t j = s; j < e; ++j) {
                    if (same_xyz(pts[j], me)) {
                        if (first < 0) first = j;
                        ++twins;
                    }
                }
                const bool grp = i < e && twins >= 2;
                if (grp) rep[i] = (int32_t)first;
                if (grp && first == i) gslot[i] = (int32_t)atomicAdd(&C->dup_groups, 1u);
                wave_append(grp, (int32_t)i, list, &C->dup_points);
            }
        } else if (lane == 0) {
            atomicOr(&C->dup_overflow, 1u);
        }
    }
}

// The long runs queued by k_dup_group, each spread over the whole grid: one
// group when every point sits at the run head's location, else a mixed run
// too long to split (grouping off).
__global__ __launch_bounds__(kBlock) void k_dup_big(const float4* __restrict__ pts, int64_t n,
                                                   int32_t* __restrict__ rep, const int32_t* __restrict__ runs,
                                                   int32_t* __restrict__ list, Counters* __restrict__ C)
{
    const uint32_t nb = C->dup_big;
    const int64_t stride = (int64_t)gridDim.x * blockDim.x;
    for (uint32_t k = 0; k < nb; ++k) {
        const int64_t s = runs[n - 3 * (int64_t)k - 3], e = runs[n - 3 * (int64_t)k - 2];
        const uint32_t base = (uint32_t)runs[n - 3 * (int64_t)k - 1];
        const float4 head = pts[s];
        bool mixed = false;
        for (int64_t i = s + (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < e; i += stride) {
            mixed |= !same_xyz(pts[i], head);
            rep[i] = (int32_t)s;
            list[base + (uint32_t)(i - s)] = (int32_t)i;
        }
        if (__ballot(mixed) != 0ull && __lane_id() == 0) atomicOr(&C->dup_overflow, 1u);
    }
}

__global__ void k_dup_finish(Counters* C)
{
    C->grouped = (C->dup_points > 0u && C->dup_overflow == 0u) ? 1u : 0u;
}

// ---------------------------------------------------------------- tree
// A leaf box covers the leaf's candidates: while coincident-point grouping is
// on, group members are never candidates (their representative, the group's
// smallest id, wins every tie at their common location), so they are left out
// and a leaf of members only keeps the empty box (+inf, -inf), which no node
// test accepts.
//
// One block per kTreeLeaves leaf slots of a cloud, an aligned subtree of it
// (Cloud::tbase: the cloud's first block): four lanes read a leaf's points,
// and the subtree's levels are combined in LDS.  The levels above, of clouds
// with more slots, follow in one launch (k_tree_top).  With each node goes the
// smallest point id under it (pad[0]): with ties on d2 broken by id, a node
// at the bound can only matter when it holds a smaller id than the best so
// far (runs of coincident points).  (A launch per level, a leaf to a lane and
// the ids by a climb of atomics took 14 launches and 72 us at 131072 points, 20
// and 296 us at 10^7; now 2, and 14 and 66 us.)
constexpr int kTreeBlock = 4 * kTreeLeaves;

__global__ __launch_bounds__(kTreeBlock) void k_tree_low(const float4* __restrict__ pts,
                                                        const Cloud* __restrict__ cl, int ncl, LeafTable lt,
                                                        Node* __restrict__ nodes, const int32_t* __restrict__ rep)
{
    __shared__ float lo[3][kTreeLeaves], hi[3][kTreeLeaves];
    __shared__ uint32_t mid[kTreeLeaves];
    const int c = find_cloud_block(cl, ncl, (int64_t)blockIdx.x);
    const int64_t L = cl[c].L, j0 = ((int64_t)blockIdx.x - cl[c].tbase) * kTreeLeaves;
    if (j0 >= L) return;                    // past the cloud's slots (one-launch capacity)
    Node* base = nodes + 2 * cl[c].lbase;
    const int w = (int)(L < kTreeLeaves ? L : kTreeLeaves);
    const int t = (int)threadIdx.x, slot = t >> 2;
    auto put = [&](int64_t i, const float* l, const float* h, uint32_t m) {
        Node nd;
        for (int k = 0; k < 3; ++k) { nd.lo[k] = l[k]; nd.hi[k] = h[k]; }
        nd.pad[0] = __uint_as_float(m);
        nd.pad[1] = 0.f;
        base[i] = nd;
    };
    float l[3] = {INFINITY, INFINITY, INFINITY}, h[3] = {-INFINITY, -INFINITY, -INFINITY};
    uint32_t m = 0xffffffffu;
    if (slot < w) {
        int64_t s0, s1;
        leaf_range(lt, cl[c].lfirst, cl[c].nl, cl[c].pos + cl[c].n, j0 + slot, s0, s1);
        for (int64_t s = s0 + (t & 3); s < s1; s += 4) {
            if (rep != nullptr) {
                const int32_t r = rep[s];
                if (r >= 0 && r != (int32_t)s) continue;
            }
            const float4 p = pts[s];
            l[0] = fminf(l[0], p.x); h[0] = fmaxf(h[0], p.x);
            l[1] = fminf(l[1], p.y); h[1] = fmaxf(h[1], p.y);
            l[2] = fminf(l[2], p.z); h[2] = fmaxf(h[2], p.z);
            m = min(m, __float_as_uint(p.w));
        }
    }
#pragma unroll
    for (int off = 1; off < 4; off <<= 1) {
        for (int k = 0; k < 3; ++k) {
            l[k] = fminf(l[k], __shfl_xor(l[k], off));
            h[k] = fmaxf(h[k], __shfl_xor(h[k], off));
        }
        m = min(m, (uint32_t)__shfl_xor((int)m, off));
    }
    if ((t & 3) == 0 && slot < w) {
        for (int k = 0; k < 3; ++k) { lo[k][slot] = l[k]; hi[k][slot] = h[k]; }
        mid[slot] = m;
        put(L + j0 + slot, l, h, m);
    }
    // thread t < ww holds node ((L + j0) >> lev) + t of the level
    for (int lev = 1, ww = w / 2; ww >= 1; ++lev, ww >>= 1) {
        __syncthreads();
        if (t < ww) {
            for (int k = 0; k < 3; ++k) {
                l[k] = fminf(lo[k][2 * t], lo[k][2 * t + 1]);
                h[k] = fmaxf(hi[k][2 * t], hi[k][2 * t + 1]);
            }
            m = min(mid[2 * t], mid[2 * t + 1]);
        }
        __syncthreads();
        if (t < ww) {
            for (int k = 0; k < 3; ++k) { lo[k][t] = l[k]; hi[k][t] = h[k]; }
            mid[t] = m;
            put(((L + j0) >> lev) + t, l, h, m);
        }
    }
}

// the levels above the blocks' subtrees: one block per cloud
__global__ __launch_bounds__(1024) void k_tree_top(const Cloud* __restrict__ cl, Node* __restrict__ nodes)
{
    const int c = (int)blockIdx.x;
    Node* base = nodes + 2 * cl[c].lbase;
    for (int64_t w = cl[c].L / kTreeLeaves / 2; w >= 1; w >>= 1) {
        for (int64_t i = w + threadIdx.x; i < 2 * w; i += blockDim.x) {
            const Node a = base[2 * i], b = base[2 * i + 1];
            Node nd;
            for (int k = 0; k < 3; ++k) {
                nd.lo[k] = fminf(a.lo[k], b.lo[k]);
                nd.hi[k] = fmaxf(a.hi[k], b.hi[k]);
            }
            nd.pad[0] = __uint_as_float(min(__float_as_uint(a.pad[0]), __float_as_uint(b.pad[0])));
            nd.pad[1] = 0.f;
            base[i] = nd;
        }
        __syncthreads();
    }
}

// --------------------------------------------------------- cone search
// One wave = 64 query points (consecutive in sorted order, or a query list).
// The wave walks the binary hierarchy together (packet traversal): a node is
// entered when any lane may still improve a cone from it; leaf points are
// read with wave-uniform (scalar) loads and every lane tests them against its
// own query.  Per lane, the best key (d2 bits << 32 | input id) of each cone
// sits in LDS; the key order is (d2, id), which for a fixed query equals
// EMST_isInf's (d2, min id, max id) order (macros_cuda.h:37).
//
// Cone membership follows NodeEMST.h:1204-1233 on the float difference
// q - p: face (axis, sign) for every axis whose |d| equals the max (sign from
// d >= 0, so -0 is '+'), and every slab of that face whose non-axis signs
// agree, where a zero coordinate is in both halves.
//
// Node test: for each face, the smallest float d2 any point of the box can
// have inside the face's pyramid (|d_axis| >= |d_other|), computed with the
// same rounded operations on the box corners, so it never exceeds a point's
// own d2; the face is kept while that bound is <= the face's worst cone best
// (empty cone = +inf).  Equality is kept because a tie can still win on id.
template <int D>
struct ConeCfg {
    static constexpr int NF = 2 * D;
    static constexpr int NS = 1 << (D - 1);
    static constexpr int K = NF * NS;
};

// allowed halves of one non-axis coordinate: bit0 = '+' half, bit1 = '-' half
__device__ __forceinline__ uint32_t halves(float d)
{
    return d > 0.f ? 1u : (d < 0.f ? 2u : 3u);
}

template <int D>
__device__ __forceinline__ uint32_t cone_mask(float dx, float dy, float dz)
{
    const float ax = fabsf(dx), ay = fabsf(dy), az = fabsf(dz);
    const uint32_t hx = halves(dx), hy = halves(dy);
    uint32_t mask = 0;
    if (D == 2) {
        const float m = fmaxf(ax, ay);
        if (ax >= m) mask |= hy << (2 * (dx < 0.f ? 1 : 0));
        if (ay >= m) mask |= hx << (2 * (dy < 0.f ? 3 : 2));
    } else {
        const uint32_t hz = halves(dz);
        const float m = fmaxf(ax, fmaxf(ay, az));
        // slab s = bit0 (first non-axis), bit1 (second); half code b -> bit value
        // expand(h1, h2): slabs {s : (h1 >> (s&1)) & 1 && (h2 >> (s>>1)) & 1}
        auto expand = [](uint32_t h1, uint32_t h2) -> uint32_t {
            return ((h2 & 1u) ? h1 : 0u) | ((h2 & 2u) ? (h1 << 2) : 0u);
        };
        if (ax >= m) mask |= expand(hy, hz) << (4 * (dx < 0.f ? 1 : 0));
        if (ay >= m) mask |= expand(hx, hz) << (4 * (dy < 0.f ? 3 : 2));
        if (az >= m) mask |= expand(hx, hy) << (4 * (dz < 0.f ? 5 : 4));
    }
    return mask;
}

// Node test.  For every point q of the box, |d_k| >= m_k on each axis, m_k the
// smallest |d_k| over the box; a half-axis (d_k >= 0 or d_k <= 0) that the box
// reaches always has that same minimum (0 when the box straddles p's
// coordinate, else the one reachable half).  So inside face (axis a, sign) the
// box's points satisfy |d_a| >= max(smallest |d_a| on the face's side, m_o1,
// m_o2) and |d_oi| >= m_oi, one bound shared by all the face's slabs the box
// reaches.  The float d2 formula is monotone in each |d|, so the same rounded
// operations on these bounds never exceed any q's own d2.  The box is needed
// when, for some face, that bound is <= the largest bound among the face's
// reachable open slabs, and its farthest point lies beyond `inner` (points
// with d2 <= inner were examined in an earlier pass).  Bounds are int32 d2
// bit patterns: -1 = cone closed, INT_MAX = open without candidate.
//
// Faces are strict where the cone is: a '-' face holds d_a < 0 only, so the
// box must reach below the query on that axis; a '+' face holds d_a > 0 or
// the zero vector, and with strict_plus (coincident points never candidates)
// d_a > 0 only.
//
// D = distance dimension, DC = cone dimension.  DC = 2 with D = 3 (the 2.5D
// mode) classifies by the xy offset only, and every face bound also carries
// the box's smallest |dz|.
template <int D, int DC>
__device__ __forceinline__ bool node_needed(const Node& nd, float px, float py, float pz,
                                            const int32_t* bound, int32_t maxb, int32_t inner,
                                            bool strict_plus)
{
    float l[3], h[3], m[3], u[3];
    bool fp[3], fn[3];
    l[0] = nd.lo[0] - px; h[0] = nd.hi[0] - px;
    l[1] = nd.lo[1] - py; h[1] = nd.hi[1] - py;
    if (D == 3) { l[2] = nd.lo[2] - pz; h[2] = nd.hi[2] - pz; }
#pragma unroll
    for (int k = 0; k < D; ++k) {
        m[k] = fmaxf(fmaxf(l[k], -h[k]), 0.f);
        u[k] = fmaxf(-l[k], h[k]);
        fp[k] = h[k] >= 0.f;
        fn[k] = l[k] <= 0.f;
    }
    {
        const float lb = D == 3 ? d2_of(m[0], m[1], m[2]) : d2_of(m[0], m[1]);
        if ((int32_t)__float_as_uint(lb) > maxb) return false;
        const float far = D == 3 ? d2_of(u[0], u[1], u[2]) : d2_of(u[0], u[1]);
        if ((int32_t)__float_as_uint(far) <= inner) return false;
    }
    bool need = false;
#pragma unroll
    for (int f = 0; f < 2 * DC; ++f) {
        const int a = f / 2;
        const bool neg = f & 1;
        const int o1 = a == 0 ? 1 : 0;
        const int o2 = a == 2 ? 1 : 2;
        const float o = DC == 3 ? fmaxf(m[o1], m[o2]) : m[o1];
        const float reach = neg ? -l[a] : h[a];
        const float am = fmaxf(neg ? -h[a] : l[a], o);
        float v[3];
        v[a] = am;
        v[o1] = m[o1];
        if (D == 3) v[o2] = m[o2];      // DC = 2: o2 is the z axis, outside the cone
        const float lb = D == 3 ? d2_of(v[0], v[1], v[2]) : d2_of(v[0], v[1]);
        const int32_t* b = bound + f * (1 << (DC - 1));
        int32_t bm;
        if (DC == 3) {
            bm = max(max((fp[o1] && fp[o2]) ? b[0] : -1, (fn[o1] && fp[o2]) ? b[1] : -1),
                     max((fp[o1] && fn[o2]) ? b[2] : -1, (fn[o1] && fn[o2]) ? b[3] : -1));
        } else {
            bm = max(fp[o1] ? b[0] : -1, fn[o1] ? b[1] : -1);
        }
        const bool open_side = (neg || strict_plus) ? reach > 0.f : true;
        need |= open_side && (reach >= o) && ((int32_t)__float_as_uint(lb) <= bm);
    }
    return need;
}

// best key -> int32 bound pattern (empty cone = INT_MAX)
__device__ __forceinline__ int32_t key_bound(unsigned long long k)
{
    const uint32_t hi = (uint32_t)(k >> 32);
    return hi == 0xffffffffu ? 0x7fffffff : (int32_t)hi;
}

constexpr int kMaxCappedPasses = 6;
// packets of a cone search, at least (launch_cone_search), and the resumed
// queries up to which their packets take kConeFewPacket each
constexpr int64_t kConePackets = 2500;
constexpr int64_t kConeFewLeft = 65536;
constexpr int kConeFewPacket = 16;

// a packet's work counters (slots: the adds of all packets do not queue on
// one address)
__device__ __forceinline__ void cone_work(Counters* ctr, uint32_t nodes, uint32_t leaves, uint32_t points,
                                          unsigned long long pairs)
{
    const int slot = (int)(blockIdx.x % kWorkSlots);
    atomicAdd(&ctr->work[kWorkConePackets][slot], 1ull);
    atomicAdd(&ctr->work[kWorkConeNodes][slot], (unsigned long long)nodes);
    atomicAdd(&ctr->work[kWorkConeLeaves][slot], (unsigned long long)leaves);
    atomicAdd(&ctr->work[kWorkConePoints][slot], (unsigned long long)points);
    atomicAdd(&ctr->work[kWorkConePairs][slot], pairs);
}

// Cone search, exact, by iterative deepening (the tree form of the Elias ring
// expansion).  Pass k caps every open cone's bound at R_k^2 (R_0 = the seed,
// R_{k+1} = 2 R_k); after the pass a cone whose best d2 is <= R_k^2 is exact
// and closes; the pass after kMaxCappedPasses has no cap, so every cone ends
// exact.  The seed only decides how much work each pass does, never the result.
//
// Seeds: seed_r (per sorted point) when given, else seed_scale times the mean
// spacing of the point's own leaf cell ((box volume / points)^(1/D)).
//
// Passes [pass_lo, pass_hi] run here.  With open_out, a query still holding
// an open cone after pass_hi stores its cone bests so far (cand_key) and its
// lane bit in open_out[packet]; a later launch (pass_lo = pass_hi + 1, nq_dev
// = the number of such queries, counted on the device) reloads them and goes
// on, in one of two forms chosen on the device: when at most compact_max
// queries are open, packets of the compacted list qlist (after pass 0 most
// queries are done, so the later passes then run on full waves instead of
// dragging a few live lanes through whole traversals); otherwise each packet
// resumes its own open lanes (resume_mask).  Resuming after pass k rebuilds
// the state exactly: R_k by the same float products, and a cone is open after
// pass k iff its best bound exceeds R_k^2.
// Occupancy: the search waits on dependent box and point loads, so it pays;
// with 8 cones the kernel fits 5 waves per SIMD in 96 VGPRs without spills
// (+8% on the 2D power-law cloud, +9% in the 2.5D mode).  With 24 cones the
// cone bests take 12 KB of LDS per 64-query block, which allows 12 blocks per
// CU, 3 waves per SIMD, whatever the registers; the attribute asks for that
// (160 VGPRs, no VGPR spills).
template <int D, int DC>
__global__ __launch_bounds__(64) __attribute__((amdgpu_waves_per_eu(DC == 3 ? 3 : 5))) void k_cone_search(const float4* __restrict__ pts,
                                                   const Node* __restrict__ nodes,
                                                   const Cloud* __restrict__ clouds, int ncl,
                                                   int bucket, LeafTable lt, int64_t n,
                                                   const int32_t* __restrict__ qlist, int64_t nq,
                                                   const int32_t* __restrict__ label,
                                                   int check_labels,
                                                   const int32_t* __restrict__ inv,
                                                   const float* __restrict__ seed_r,
                                                   float seed_scale,
                                                   uint64_t* __restrict__ cand_key,
                                                   int32_t* __restrict__ cand_pos,
                                                   int32_t* __restrict__ revive,
                                                   int32_t* __restrict__ first_corr,
                                                   uint64_t* __restrict__ first_key,
                                                   Counters* __restrict__ ctr, int collect_stats,
                                                   DupState dup, int pass_lo, int pass_hi,
                                                   uint64_t* __restrict__ open_out,
                                                   const uint32_t* __restrict__ nq_dev,
                                                   const uint64_t* __restrict__ resume_mask,
                                                   int64_t compact_max, int qpp)
{
    using C = ConeCfg<DC>;
    bool compacted = true;
    if (nq_dev) {
        nq = *nq_dev;
        compacted = nq <= compact_max;
        // few queries left: narrower packets (the grid covers 64 to a packet
        // of every query; 41213 left of 200003 1.23 -> 0.97 ms for the search,
        // while 145434 left of 10^6 lose 0.3)
        if (compacted && nq <= kConeFewLeft && nq <= (int64_t)gridDim.x * kConeFewPacket) qpp = kConeFewPacket;
        if (compacted ? (int64_t)blockIdx.x * qpp >= nq : resume_mask[blockIdx.x] == 0ull)
            return;     // nothing to resume in this packet
    }
    __shared__ unsigned long long best[C::K][64];
    __shared__ int32_t stk_id[64];
    __shared__ int32_t stk_ver[64];
    __shared__ unsigned long long stk_mask[64];
    const int lane = __lane_id();
    const int64_t qi = (int64_t)blockIdx.x * (compacted ? qpp : 64) + lane;
    bool active;
    int64_t p;
    if (compacted) {
        active = lane < qpp && qi < nq;
        p = active ? (qlist ? (int64_t)qlist[qi] : qi) : 0;
    } else {
        active = (resume_mask[blockIdx.x] >> lane) & 1ull;     // set bits are points of this packet
        p = active ? qi : 0;
    }
    // grouping on: group members do not search (k_dup_fill gives them their
    // representative's cones) and no point takes a candidate at its own
    // location; otherwise only the point itself is skipped
    const bool grouped = dup.rep != nullptr;
    // strict '+' faces need the '+' cones to hold no point but the query's
    // own location; with xy wedges over 3D points they also hold the points
    // straight above and below it
    const bool strict_plus = grouped && DC == D;
    bool is_rep = false;
    if (grouped && active) {
        const int32_t r = dup.rep[p];
        active = r < 0 || r == (int32_t)p;
        is_rep = r == (int32_t)p;
    }
    bool underflow = false;
    const float4 me = pts[p];
    const float px = me.x, py = me.y, pz = me.z;
    const int32_t mylab = (check_labels && active) ? label[p] : 0;
#pragma unroll
    for (int c = 0; c < C::K; ++c) best[c][lane] = (pass_lo > 0 && active) ? cand_key[(int64_t)c * n + p] : kEmptyKey;

    uint32_t st_nodes = 0, st_leaves = 0, st_pts = 0, st_pairs = 0;
    // one traversal per cloud among the wave's queries (a packet of a single
    // cloud, the usual case, makes one)
    const int my_cl = active ? find_cloud(clouds, ncl, p) : -1;
    uint32_t open_final = 0;
    uint64_t pending = __ballot(active);
    while (pending) {
        const int cl = __builtin_amdgcn_readfirstlane(__shfl(my_cl, (int)__builtin_ctzll(pending)));
        const bool mine = my_cl == cl;
        pending &= ~__ballot(mine);
        const int64_t cend = clouds[cl].pos + clouds[cl].n;
        const int64_t L = clouds[cl].L, lfirst = clouds[cl].lfirst, nl = clouds[cl].nl;
        const Node* __restrict__ tree = nodes + 2 * clouds[cl].lbase;

        // seed radius
        float r = 1.f;
        if (!mine) {
            // not this traversal's query
        } else if (seed_r) {
            r = seed_r[p];
            if (!positive_finite(r)) r = 1e-6f;
        } else {
            const int64_t lf = lt.of[p];
            const Node own = tree[L + (lf - lfirst)];
            const float cnt = (float)(lt.start[lf + 1] - lt.start[lf]);
            float vol = 1.f, ext = 0.f;
            for (int k = 0; k < D; ++k) {
                const float e = own.hi[k] - own.lo[k];
                vol *= e;
                ext = fmaxf(ext, e);
            }
            float sp = vol > 0.f ? powf(vol / cnt, 1.f / D) : ext / cnt;
            if (!positive_finite(sp)) sp = 1e-6f;
            r = seed_scale * sp;
        }
        float r2 = r * r;
        uint32_t open = mine ? (uint32_t)((1ull << C::K) - 1) : 0u;
        int32_t inner = -1;
        for (int k = 0; k < pass_lo; ++k) {
            inner = (int32_t)__float_as_uint(r2);
            r2 *= 4.f;
        }
        if (pass_lo > 0) {
            open = 0u;
#pragma unroll
            for (int c = 0; c < C::K; ++c)
                if (mine && key_bound(best[c][lane]) > inner) open |= 1u << c;
            // no point found so far: the passes before pass_lo saw an empty
            // ball, or left the query out (k_cone_first); it starts over
            bool none = true;
#pragma unroll
            for (int c = 0; c < C::K; ++c) none = none && best[c][lane] == kEmptyKey;
            if (none) {
                inner = -1;
                r2 = r * r;
            }
        }
        int32_t bound[C::K];
        int32_t maxb = -1;

        // packet centre (for near-first child order)
        float cx = mine ? px : 0.f, cy = mine ? py : 0.f, cz = mine ? pz : 0.f;
        float na = mine ? 1.f : 0.f;
        for (int off = 32; off > 0; off >>= 1) {
            cx += __shfl_xor(cx, off);
            cy += __shfl_xor(cy, off);
            cz += __shfl_xor(cz, off);
            na += __shfl_xor(na, off);
        }
        cx /= na; cy /= na; cz /= na;
        auto cdist = [&](const Node& x) {
            const float dxx = fmaxf(fmaxf(x.lo[0] - cx, cx - x.hi[0]), 0.f);
            const float dyy = fmaxf(fmaxf(x.lo[1] - cy, cy - x.hi[1]), 0.f);
            const float dzz = fmaxf(fmaxf(x.lo[2] - cz, cz - x.hi[2]), 0.f);
            return dxx * dxx + dyy * dyy + dzz * dzz;
        };

        for (int pass = pass_lo; pass <= pass_hi; ++pass) {
            if (__ballot(open != 0u) == 0ull) break;
            const bool last = pass == kMaxCappedPasses;
            const int32_t cap = last ? 0x7fffffff : (int32_t)__float_as_uint(r2);
            auto refresh = [&]() {
                maxb = -1;
#pragma unroll
                for (int c = 0; c < C::K; ++c) {
                    const int32_t b = ((open >> c) & 1u) ? min(key_bound(best[c][lane]), cap) : -1;
                    bound[c] = b;
                    maxb = max(maxb, b);
                }
            };
            refresh();
            int sp = 0;
            int ver = 0;        // bumps whenever a leaf tightened the bounds
            if (lane == 0) { stk_id[0] = 1; stk_ver[0] = -1; }
            sp = 1;
            __builtin_amdgcn_wave_barrier();
            while (sp > 0) {
                --sp;
                const int node = __builtin_amdgcn_readfirstlane(stk_id[sp]);
                const int pver = __builtin_amdgcn_readfirstlane(stk_ver[sp]);
                // a node tested against the current bounds when pushed keeps its
                // lane mask; after a leaf tightened the bounds it is tested again
                bool need;
                if (pver == ver) {
                    need = (stk_mask[sp] >> lane) & 1ull;
                } else {
                    const Node nd = tree[node];
                    need = open != 0u && node_needed<D, DC>(nd, px, py, pz, bound, maxb, inner, strict_plus);
                    ++st_nodes;
                }
                const uint64_t needm = __ballot(need);
                if (needm == 0ull) continue;
                if (node >= L) {
                    int64_t s0, s1;
                    leaf_range(lt, lfirst, nl, cend, node - L, s0, s1);
                    const int cnt = (int)(s1 - s0);
                    ++st_leaves;
                    st_pts += (uint32_t)cnt;
                    st_pairs += (uint32_t)cnt * (uint32_t)__popcll(needm);
                    // pair-parallel: lane = (query slot, leaf point); a chunk covers
                    // 64 / bucket needed queries x the leaf's points
                    const int j = lane & (bucket - 1);
                    const int qslot = lane / bucket;
                    const int qpc = 64 / bucket;
                    float4 v = make_float4(0.f, 0.f, 0.f, 0.f);
                    if (j < cnt) v = pts[s0 + j];
                    const int64_t s = s0 + j;
                    // one (query, leaf point) pair per lane: distance, cone, and
                    // an LDS atomic into the query's cone best
                    auto pair = [&](int myq, float qx, float qy, float qz, int32_t qmaxb, int32_t qinner,
                                    uint32_t qopen, int32_t qpos, int32_t qlab) {
                        const float dx = v.x - qx, dy = v.y - qy, dz = v.z - qz;
                        const float d2 = D == 3 ? d2_of(dx, dy, dz) : d2_of(dx, dy);
                        const int32_t db = (int32_t)__float_as_uint(d2);
                        const bool here = dx == 0.f && dy == 0.f && dz == 0.f;
                        bool take = myq >= 0 && j < cnt && (grouped ? !here : s != (int64_t)qpos) &&
                                    db <= qmaxb && db > qinner;
                        // distinct points at float distance 0 (underflow) break the
                        // grouping's premise; the caller then searches ungrouped
                        if (grouped && take && d2 == 0.f) underflow = true;
                        if (check_labels && take && d2 == 0.f) take = label[s] != qlab;
                        if (take) {
                            uint32_t mask = cone_mask<DC>(dx, dy, dz) & qopen;
                            const unsigned long long key =
                                ((unsigned long long)__float_as_uint(d2) << 32) | __float_as_uint(v.w);
                            while (mask) {
                                const int c = __builtin_ctz(mask);
                                mask &= mask - 1;
                                atomicMin(&best[c][myq], key);
                            }
                        }
                    };
                    uint64_t rem = needm;
                    if (qpc == 1) {
                        // every lane works on the same query: broadcast its state with
                        // v_readlane (a scalar register) instead of an LDS permute
                        while (rem) {
                            const int q = (int)__builtin_ctzll(rem);
                            rem &= rem - 1;
                            auto rl = [&](int x) { return __builtin_amdgcn_readlane(x, q); };
                            pair(q, __int_as_float(rl(__float_as_int(px))), __int_as_float(rl(__float_as_int(py))),
                                 __int_as_float(rl(__float_as_int(pz))), rl(maxb), rl(inner), (uint32_t)rl((int)open),
                                 rl((int32_t)p), check_labels ? rl(mylab) : 0);
                        }
                    } else {
                        while (rem) {
                            // the qslot-th remaining needed lane is this lane's query
                            int myq = -1;
                            for (int k = 0; k < qpc; ++k) {
                                const int l = rem ? (int)__builtin_ctzll(rem) : -1;
                                if (rem) rem &= rem - 1;
                                if (k == qslot) myq = l;
                            }
                            const int src = myq >= 0 ? myq : 0;
                            pair(myq, __shfl(px, src), __shfl(py, src), __shfl(pz, src), __shfl(maxb, src),
                                 __shfl(inner, src), (uint32_t)__shfl((int)open, src), __shfl((int32_t)p, src),
                                 check_labels ? __shfl(mylab, src) : 0);
                        }
                    }
                    if (need) refresh();
                    ++ver;
                } else {
                    // the next boxes down: the children when they are leaves, else
                    // the four grandchildren (a descent then waits on half as many
                    // dependent loads; the four loads are independent)
                    const bool leafkids = 2 * (int64_t)node >= L;
                    const int first = leafkids ? 2 * node : 4 * node;
                    const int nk = leafkids ? 2 : 4;
                    Node bx[4];
#pragma unroll
                    for (int i = 0; i < 4; ++i)
                        if (i < nk) bx[i] = tree[first + i];
                    uint64_t mk[4];
                    float dk[4];
                    int id[4];
#pragma unroll
                    for (int i = 0; i < 4; ++i) {
                        mk[i] = i < nk ? __ballot(open != 0u && node_needed<D, DC>(bx[i], px, py, pz, bound,
                                                                                     maxb, inner, strict_plus))
                                       : 0ull;
                        dk[i] = mk[i] ? cdist(bx[i]) : -1.f;
                        id[i] = first + i;
                    }
                    st_nodes += (uint32_t)nk;
                    // farthest pushed first, so the nearest is popped next
                    auto ce = [&](int a, int b) {
                        if (dk[a] < dk[b]) {
                            const float td = dk[a]; dk[a] = dk[b]; dk[b] = td;
                            const uint64_t tm = mk[a]; mk[a] = mk[b]; mk[b] = tm;
                            const int ti = id[a]; id[a] = id[b]; id[b] = ti;
                        }
                    };
                    ce(0, 1); ce(2, 3); ce(0, 2); ce(1, 3); ce(1, 2);
                    if (lane == 0) {
                        int t = sp;
#pragma unroll
                        for (int i = 0; i < 4; ++i)
                            if (mk[i]) { stk_id[t] = id[i]; stk_ver[t] = ver; stk_mask[t] = mk[i]; ++t; }
                    }
#pragma unroll
                    for (int i = 0; i < 4; ++i) sp += mk[i] != 0ull ? 1 : 0;
                    __builtin_amdgcn_wave_barrier();
                }
            }
            // close the cones whose best lies within this pass's radius
#pragma unroll
            for (int c = 0; c < C::K; ++c)
                if (((open >> c) & 1u) && key_bound(best[c][lane]) <= cap) open &= ~(1u << c);
            inner = cap;
            r2 *= 4.f;
        }
        if (mine) open_final = open;
    }
    if (collect_stats && lane == 0) {
        cone_work(ctr, st_nodes, st_leaves, st_pts, st_pairs);
    }
    if (__ballot(underflow) != 0ull && lane == 0) atomicOr(&ctr->underflow, 1u);
    if (open_out) {
        const bool unfinished = active && open_final != 0u;
        const uint64_t om = __ballot(unfinished);
        if (lane == 0) open_out[blockIdx.x] = om;
        if (unfinished) {
            // the bests so far, for the launch that resumes this query
            for (int c = 0; c < C::K; ++c) cand_key[(int64_t)c * n + p] = best[c][lane];
            return;
        }
    }
    if (!active) return;
    if (revive && revive[p] == -2) revive[p] = -1;
    const int64_t gs = is_rep ? (int64_t)dup.gslot[p] : 0;
    // cone-major layout [K][n]: lanes write consecutive words
    uint64_t kmin = kEmptyKey;
    int32_t pmin = -1;
    for (int c = 0; c < C::K; ++c) {
        const uint64_t k = best[c][lane];
        const int32_t q = (k == kEmptyKey) ? -1 : inv[(uint32_t)k];
        cand_key[(int64_t)c * n + p] = k;
        cand_pos[(int64_t)c * n + p] = q;
        if (k < kmin) { kmin = k; pmin = q; }
        // a representative keeps its '+' cones for the rounds in which its
        // group has become one component (k_dup_fill)
        if (is_rep && ((c / C::NS) & 1) == 0) {
            const int64_t b = (int64_t)((c / C::NS / 2) * C::NS + c % C::NS) * dup.ngroups + gs;
            dup.bkey[b] = k;
            dup.bpos[b] = q;
        }
    }
    // first search (all points singletons): the round-1 target is the overall
    // cone minimum (NodeEMST.h:1338-1381 with every label distinct)
    if (first_corr) {
        first_corr[p] = pmin >= 0 ? pmin : -2;
        first_key[p] = kmin;
    }
}

// minimum over the wave, the same in every lane
__device__ __forceinline__ uint32_t wave_min_u32(uint32_t v)
{
    v = min(v, (uint32_t)__builtin_amdgcn_mov_dpp((int)v, 0xB1, 0xF, 0xF, false));     // quad_perm [1,0,3,2]
    v = min(v, (uint32_t)__builtin_amdgcn_mov_dpp((int)v, 0x4E, 0xF, 0xF, false));     // quad_perm [2,3,0,1]
    v = min(v, (uint32_t)__builtin_amdgcn_mov_dpp((int)v, 0x141, 0xF, 0xF, false));    // row_half_mirror
    v = min(v, (uint32_t)__builtin_amdgcn_mov_dpp((int)v, 0x140, 0xF, 0xF, false));    // row_mirror
    // one value per row of 16
    const uint32_t a = (uint32_t)__builtin_amdgcn_readlane((int)v, 0), b = (uint32_t)__builtin_amdgcn_readlane((int)v, 16);
    const uint32_t c = (uint32_t)__builtin_amdgcn_readlane((int)v, 32), d = (uint32_t)__builtin_amdgcn_readlane((int)v, 48);
    return min(min(a, b), min(c, d));
}

__device__ __forceinline__ uint64_t shfl_xor_u64(uint64_t v, int m)
{
    const uint32_t lo = (uint32_t)__shfl_xor((int)(uint32_t)v, m);
    const uint32_t hi = (uint32_t)__shfl_xor((int)(uint32_t)(v >> 32), m);
    return ((uint64_t)hi << 32) | lo;
}

// A gathering starts from every node of depth min(6, leaf depth), 64 at most,
// one per lane: the levels above would each take a dependent step for a few
// nodes.  Returns the count written to work[].
__device__ __forceinline__ int gather_start(int64_t L, int32_t* work)
{
    int d0 = 0;
    while (d0 < 6 && ((int64_t)2 << d0) <= L) ++d0;
    const int cnt = 1 << d0;
    const int lane = __lane_id();
    if (lane < cnt) work[lane] = cnt + lane;
    __builtin_amdgcn_wave_barrier();
    return cnt;
}

// The gathering's next nodes from the inner nodes that passed: each hands on
// its 4 grandchildren (one 128-byte line of the heap), or its 2 children when
// those are leaves.  Every gathering test (box distance, far side, component
// label, empty) is monotone under box inclusion, so a grandchild whose parent
// would have failed fails too: the same nodes pass as level by level, in half
// the dependent steps.  Writes the entries at work[tail ..] and their count to
// add; false (nothing written) when they would pass cap.
__device__ __forceinline__ bool push_inner(bool pass, int nd, int64_t L, int32_t* work, int tail, int cap,
                                           int& add)
{
    const bool deep = pass && 2 * (int64_t)nd < L;     // its children are inner nodes
    const uint64_t m4 = __ballot(deep), m2 = __ballot(pass && !deep);
    add = 4 * __popcll(m4) + 2 * __popcll(m2);
    if (tail + add > cap) return false;
    const uint64_t lt = lanemask_lt();
    const int r = tail + 4 * __popcll(m4 & lt) + 2 * __popcll(m2 & lt);
    if (deep) {
#pragma unroll
        for (int k = 0; k < 4; ++k) work[r + k] = 4 * nd + k;
    } else if (pass) {
        work[r] = 2 * nd;
        work[r + 1] = 2 * nd + 1;
    }
    return true;
}

// ascending bitonic sort of one 64-bit key per lane across the wave
__device__ __forceinline__ uint64_t wave_sort_u64(uint64_t e)
{
    const int lane = __lane_id();
#pragma unroll
    for (int k = 2; k <= 64; k <<= 1) {
#pragma unroll
        for (int j = k >> 1; j > 0; j >>= 1) {
            const uint64_t o = shfl_xor_u64(e, j);
            const bool keep_min = ((lane & j) == 0) == ((lane & k) == 0);
            e = keep_min ? (o < e ? o : e) : (o > e ? o : e);
        }
    }
    return e;
}

// ---- first pass of the cone search over every query (k_cone_first) ----
//
// One wave per 64 consecutive positions; each lane is one query with its cone
// bests in its own column of LDS.  The wave gathers the leaves within the
// lanes' first radius R_0 of the packet's box (64 node tests a step), keeps
// per leaf the 8-lane groups whose box it can matter to, and then takes the
// leaf points one at a time, at one address for the whole wave: every lane
// pairs the point with its own query.  A point enters only when it lies
// within the largest radius of a needed group from that group's box.
//
// Against one query at a time per leaf (k_cone_search), where 64 lanes pair a
// leaf's 25-50 points with each query that needs the leaf: the pairs that lie
// beyond every radius are dropped 64 at a time, no query state is broadcast,
// and a lane's minimum goes to its own column, where no other lane's atomic
// waits on the same address.
//
// Cones are kept as axis * 2^D + octant (the signs of the offset): that
// index comes from three sign bits and two compares.  An offset on a boundary
// between cones (a zero coordinate, or equal largest coordinates) lies in
// several and takes cone_octants.
//
// A query with a cone whose best lies beyond R_0 stores its bests and is left
// open (open_out) for k_cone_search, which goes on from pass 1.  A packet
// whose gathering outgrows the LDS lists (a thin point's radius over a dense
// cluster) is left open without a best, and k_cone_search starts it over: a
// wave that took all those points one by one was the kernel's tail.  (The
// search of 4*10^6 clustered points, seed 3.5: lists of 256 leaves 15.0 ms,
// of 128 11.0; trying halves of such a packet again, down to 32 or 8 lanes,
// 11.0 and 12.7.)
//
// Bound by VALU issue: 32000 instructions a packet of uniform 3D points (60
// leaves, 930 points a lane, 24 instructions a pair; seed 3.5), 71% of the
// cycles busy; 12.5 KB of bests and lists and 1 KB of batch allow 11 waves per
// CU.  Points through scalar loads instead of LDS waited on the scalar cache
// (1.25 times as long); four streams of 16 lanes with a list of points each
// took 18% fewer steps and as long.  The whole search against k_cone_search
// alone: 10^6 uniform points 4.4 -> 2.9 ms in 3D, 0.95 -> 0.79 in 2D; 4*10^6
// clustered ones 18.2 -> 12.4 (with the seed model 17.3 -> 12.8), power-law
// ones in 2D 4.2 -> 3.6.
constexpr int kFirstWork = 1024;
constexpr int kFirstLeaves = 128;
constexpr int kFirstChunks = kFirstLeaves / 64;

// the cones of an offset as bits axis * 2^D + octant: the face of every
// axis whose |d| is the largest, with both signs of each zero coordinate off
// that axis (cone_mask in the other numbering)
template <int D>
__device__ __forceinline__ uint32_t cone_octants(float dx, float dy, float dz)
{
    const float ax = fabsf(dx), ay = fabsf(dy), az = D == 3 ? fabsf(dz) : 0.f;
    const float m = fmaxf(fmaxf(ax, ay), az);
    constexpr uint32_t all = D == 3 ? 0xffu : 0xfu;
    const uint32_t px = 0x55u & all, py = 0x33u & all, pz = 0x0fu;      // octants of '+' signs
    const uint32_t sx = dx < 0.f ? all ^ px : px, sy = dy < 0.f ? all ^ py : py;
    const uint32_t sz = D == 3 ? (dz < 0.f ? all ^ pz : pz) : all;
    const uint32_t ex = dx == 0.f ? all : sx, ey = dy == 0.f ? all : sy;
    const uint32_t ez = D == 3 && dz == 0.f ? all : sz;
    uint32_t r = 0;
    if (ax >= m) r |= sx & ey & ez;
    if (ay >= m) r |= (ex & sy & ez) << (1 << D);
    if (D == 3 && az >= m) r |= (ex & ey & sz) << (2 << D);
    return r;
}

// the row of cone c (face * 2^(D-1) + slab) in that numbering
template <int D>
__device__ __forceinline__ constexpr int cone_row(int c)
{
    const int face = c / ConeCfg<D>::NS, slab = c % ConeCfg<D>::NS;
    const int axis = face / 2;
    int oct = (face & 1) << axis, bit = 0;
    for (int k = 0; k < D; ++k)
        if (k != axis) oct |= ((slab >> bit++) & 1) << k;
    return axis * (1 << D) + oct;
}

template <int D>
__global__ __launch_bounds__(64) __attribute__((amdgpu_waves_per_eu(D == 3 ? 3 : 4))) void k_cone_first(
    const float4* __restrict__ pts, const Node* __restrict__ nodes, const Cloud* __restrict__ clouds, int ncl,
    int bucket, LeafTable lt, int64_t n, const int32_t* __restrict__ inv, const float* __restrict__ seed_r,
    float seed_scale, float seed_mul, uint64_t* __restrict__ cand_key, int32_t* __restrict__ cand_pos,
    int32_t* __restrict__ first_corr, uint64_t* __restrict__ first_key, Counters* __restrict__ ctr,
    int collect_stats, DupState dup, uint64_t* __restrict__ open_out, int32_t* __restrict__ reach)
{
    using C = ConeCfg<D>;
    static_assert(C::K == D * (1 << D), "one row per axis and octant");
    // the gathering's lists and the cone bests take turns in the same LDS
    constexpr int kListWords = kFirstLeaves + kFirstWork / 2;
    constexpr int kBestWords = C::K * 64;
    __shared__ unsigned long long lds[kBestWords > kListWords ? kBestWords : kListWords];
    __shared__ float4 gbox[16];             // per 8-lane group: lo (xyz), hi (xyz)
    __shared__ float4 batch[64];            // leaf points waiting to be paired
    unsigned long long* best = lds;         // [row][lane]
    unsigned long long* gathered = lds;
    int32_t* work = reinterpret_cast<int32_t*>(lds + kFirstLeaves);
    const int lane = __lane_id();
    const int64_t p = (int64_t)blockIdx.x * 64 + lane;
    bool active = p < n;
    // grouping on: as in k_cone_search, members do not search and no point
    // takes a candidate at its own location
    const bool grouped = dup.rep != nullptr;
    bool is_rep = false;
    if (grouped && active) {
        const int32_t r = dup.rep[p];
        active = r < 0 || r == (int32_t)p;
        is_rep = r == (int32_t)p;
    }
    const float4 me = pts[p < n ? p : n - 1];
    const float px = me.x, py = me.y, pz = me.z;
    const int my_cl = active ? find_cloud(clouds, ncl, p) : -1;
    const int lb = 31 - __builtin_clz(bucket);      // log2
    const int per_step = 64 >> lb;                  // leaves per step of 64 lanes
    uint32_t st_nodes = 0, st_leaves = 0, st_pts = 0, st_pairs = 0;
    bool underflow = false;
    uint64_t open_lanes = 0;
    uint64_t pending = __ballot(active);
    while (pending) {
        const int cl = __builtin_amdgcn_readfirstlane(__shfl(my_cl, (int)__builtin_ctzll(pending)));
        const bool mine = my_cl == cl;
        pending &= ~__ballot(mine);
        const int64_t L = clouds[cl].L, lfirst = clouds[cl].lfirst;
        const Node* __restrict__ tree = nodes + 2 * clouds[cl].lbase;
        float r = 1.f;
        if (!mine) {
            // not this traversal's query
        } else if (seed_r) {
            r = seed_r[p];
            if (!positive_finite(r)) r = 1e-6f;
        } else {
            const int64_t lf = lt.of[p];
            const Node own = tree[L + (lf - lfirst)];
            const float cnt = (float)(lt.start[lf + 1] - lt.start[lf]);
            float vol = 1.f, ext = 0.f, area = 0.f;
            for (int k = 0; k < D; ++k) {
                const float e = own.hi[k] - own.lo[k];
                area = fmaxf(area, e * ext);
                vol *= e;
                ext = fmaxf(ext, e);
            }
            float sp = vol > 0.f ? powf(vol / cnt, 1.f / D) : ext / cnt;
            // (late cones: most points of a flat leaf would see no other, and
            // the rounds would ask for all of them; ms a run without / with: a
            // plane of 5*10^5 points along the axes 7.7 / 2.1, a voxel floor
            // of 1.8*10^5 4.4 / 1.25)
            if (reach && !(vol > 0.f) && area > 0.f) sp = sqrtf(area / cnt);
            if (!positive_finite(sp)) sp = 1e-6f;
            r = seed_scale * sp;
        }
        r *= seed_mul;
        const float r2 = r * r;
        // boxes of the lanes and of each 8-lane group
        float qlo[3] = {mine ? px : INFINITY, mine ? py : INFINITY, mine ? pz : INFINITY};
        float qhi[3] = {mine ? px : -INFINITY, mine ? py : -INFINITY, mine ? pz : -INFINITY};
        __builtin_amdgcn_wave_barrier();
#pragma unroll
        for (int off = 1; off < 64; off <<= 1) {
#pragma unroll
            for (int k = 0; k < 3; ++k) {
                qlo[k] = fminf(qlo[k], __shfl_xor(qlo[k], off));
                qhi[k] = fmaxf(qhi[k], __shfl_xor(qhi[k], off));
            }
            if (off == 4 && (lane & 7) == 0) {
                gbox[2 * (lane >> 3)] = make_float4(qlo[0], qlo[1], qlo[2], 0.f);
                gbox[2 * (lane >> 3) + 1] = make_float4(qhi[0], qhi[1], qhi[2], 0.f);
            }
        }
        // the bound per lane, the groups' largest (a group without lanes:
        // its box is empty), and the largest of all
        float cap = mine ? r2 : -1.f;
        uint32_t t8 = group8_max_u32(mine ? __float_as_uint(r2) : 0u);
        uint32_t B = t8;
#pragma unroll
        for (int off = 8; off < 64; off <<= 1) B = max(B, (uint32_t)__shfl_xor((int)B, off));
        B = (uint32_t)__builtin_amdgcn_readfirstlane((int)B);
        __builtin_amdgcn_wave_barrier();
        auto group_d2 = [&](int g, float x0, float y0, float z0, float x1, float y1, float z1) {
            const float4 a = gbox[2 * g], b = gbox[2 * g + 1];
            const float m0 = fmaxf(fmaxf(x0 - b.x, a.x - x1), 0.f);
            const float m1 = fmaxf(fmaxf(y0 - b.y, a.y - y1), 0.f);
            const float m2 = fmaxf(fmaxf(z0 - b.z, a.z - z1), 0.f);
            return __float_as_uint(D == 3 ? d2_of(m0, m1, m2) : d2_of(m0, m1));
        };
        // gather: key = (box d2 bits without the low 8 | group mask) << 32 | node
        int head = 0, tail = gather_start(L, work), ngl = 0;
        bool over = B >= 0x7f800000u;       // (an unbounded first radius: not a capped pass)
        __builtin_amdgcn_wave_barrier();
        while (head < tail && !over) {
            const int take = min(64, tail - head);
            const int nd = lane < take ? work[head + lane] : 0;
            head += take;
            ++st_nodes;
            bool pass = false, leaf = false;
            uint32_t bd = 0, gm = 0;
            if (lane < take) {
                const Node x = tree[nd];
                float m[3];
#pragma unroll
                for (int k = 0; k < 3; ++k) m[k] = fmaxf(fmaxf(x.lo[k] - qhi[k], qlo[k] - x.hi[k]), 0.f);
                bd = __float_as_uint(D == 3 ? d2_of(m[0], m[1], m[2]) : d2_of(m[0], m[1]));
                leaf = nd >= L;
                pass = bd <= B && bd < 0x7f800000u;     // (an empty box lies at infinity)
                if (pass && leaf) {
#pragma unroll
                    for (int g = 0; g < 8; ++g) {
                        const uint32_t tg = (uint32_t)__builtin_amdgcn_readlane((int)t8, 8 * g);
                        const uint32_t d = group_d2(g, x.lo[0], x.lo[1], x.lo[2], x.hi[0], x.hi[1], x.hi[2]);
                        gm |= d <= tg ? 1u << g : 0u;
                    }
                    pass = gm != 0u;
                }
            }
            const uint64_t ml = __ballot(pass && leaf);
            const int nlf = __popcll(ml);
            int add;
            if (!push_inner(pass && !leaf, nd, L, work, tail, kFirstWork, add) || ngl + nlf > kFirstLeaves) {
                over = true;
                break;
            }
            if (pass && leaf)
                gathered[ngl + __popcll(ml & lanemask_lt())] =
                    ((uint64_t)((bd & 0xffffff00u) | gm) << 32) | (uint32_t)nd;
            tail += add;
            ngl += nlf;
            __builtin_amdgcn_wave_barrier();
        }
        if (over) {
            // too far for the lists: left open without a best
            if (mine) {
                for (int c = 0; c < C::K; ++c) cand_key[(int64_t)c * n + p] = kEmptyKey;
                if (reach) {
                    reach[p] = -1;
                    first_corr[p] = -2;
                    first_key[p] = kEmptyKey;
                }
            }
            open_lanes |= __ballot(mine);
            continue;
        }
        // the leaves, nearest first 64 at a time, now in registers
        uint64_t ent[kFirstChunks];
#pragma unroll
        for (int k = 0; k < kFirstChunks; ++k) {
            ent[k] = kEmptyKey;
            if (64 * k < ngl) {
                const uint64_t e = 64 * k + lane < ngl ? gathered[64 * k + lane] : kEmptyKey;
                ent[k] = wave_sort_u64(e);
            }
        }
        __builtin_amdgcn_wave_barrier();
#pragma unroll
        for (int c = 0; c < C::K; ++c) best[c * 64 + lane] = kEmptyKey;
        __builtin_amdgcn_wave_barrier();
        st_leaves += (uint32_t)ngl;
        const uint32_t nin = (uint32_t)__popcll(__ballot(mine));
        // one leaf point against every lane's query; true where it lies
        // on a boundary between cones (lower_all)
        auto pair = [&](const float4 q) {
            const float dx = q.x - px, dy = q.y - py, dz = q.z - pz;
            const float d2 = D == 3 ? d2_of(dx, dy, dz) : d2_of(dx, dy);
            const float ax = fabsf(dx), ay = fabsf(dy), az = fabsf(dz);
            float m, second, least;
            if (D == 3) {
                m = fmaxf(fmaxf(ax, ay), az);
                second = __builtin_amdgcn_fmed3f(ax, ay, az);
                least = fminf(fminf(ax, ay), az);
            } else {
                m = fmaxf(ax, ay);
                second = least = fminf(ax, ay);
            }
            uint32_t row = D == 3 ? __float_as_uint(dz) >> 31 : 0u;
            row = (row << 1) | (__float_as_uint(dy) >> 31);
            row = (row << 1) | (__float_as_uint(dx) >> 31);
            if (D == 3) row |= ax == m ? 0u : (ay == m ? 8u : 16u);
            else row |= ax == m ? 0u : 4u;
            const bool near = d2 <= cap;
            const bool plain = least > 0.f && second < m;
            if (near && plain)
                atomicMin(&best[row * 64 + lane],
                          ((unsigned long long)__float_as_uint(d2) << 32) | __float_as_uint(q.w));
            return near && !plain;
        };
        auto lower_all = [&](const float4 q) {
            const float dx = q.x - px, dy = q.y - py, dz = q.z - pz;
            const float d2 = D == 3 ? d2_of(dx, dy, dz) : d2_of(dx, dy);
            const bool self = __float_as_uint(q.w) == __float_as_uint(me.w);
            const bool here = dx == 0.f && dy == 0.f && dz == 0.f;
            if (d2 <= cap && !(grouped ? here : self)) {
                uint32_t rows = cone_octants<D>(dx, dy, dz);
                while (rows) {
                    const int row = __builtin_ctz(rows);
                    rows &= rows - 1;
                    atomicMin(&best[row * 64 + lane],
                              ((unsigned long long)__float_as_uint(d2) << 32) | __float_as_uint(q.w));
                }
            }
        };
        // the points kept so far, padded to a multiple of 4 with points
        // beyond every bound
        int held = 0;
        auto drain = [&]() {
            if (lane < 3 && held + lane < 64) batch[held + lane] = make_float4(INFINITY, INFINITY, INFINITY, me.w);
            __builtin_amdgcn_wave_barrier();
            for (int j = 0; j < held; j += 4) {
                float4 q[4];
#pragma unroll
                for (int u = 0; u < 4; ++u) q[u] = batch[j + u];
                bool tie = false;
#pragma unroll
                for (int u = 0; u < 4; ++u) tie |= pair(q[u]);
                // (every query meets itself here once, a zero offset)
                if (__ballot(tie) != 0ull) {
#pragma unroll 1
                    for (int u = 0; u < 4; ++u) if (tie) lower_all(batch[j + u]);
                }
            }
            __builtin_amdgcn_wave_barrier();
            held = 0;
        };
        for (int c0 = 0; c0 < ngl; c0 += 64) {
            const int cn = min(64, ngl - c0);
            const int ck = c0 >> 6;
            uint64_t e = ent[0];
#pragma unroll
            for (int k = 1; k < kFirstChunks; ++k) e = ck == k ? ent[k] : e;
            const int e_node = (int)(uint32_t)e;
            const uint32_t e_gm = (uint32_t)(e >> 32) & 0xffu;
            // this lane's leaf point of the step's leaves
            auto fetch = [&](int i, bool& has, float4& w) {
                const int idx = i + (lane >> lb);
                const int node = __shfl(e_node, idx & 63);
                has = false;
                w = make_float4(0.f, 0.f, 0.f, 0.f);
                if (idx < cn) {
                    const int64_t lf = lfirst + (node - L);
                    const int32_t s0 = lt.start[lf] + (lane & (bucket - 1));
                    has = s0 < lt.start[lf + 1];
                    if (has) w = pts[s0];
                }
            };
            bool has, nhas;
            float4 w, nw;
            fetch(0, nhas, nw);
            for (int i = 0; i < cn; i += per_step) {
                has = nhas;
                w = nw;
                if (i + per_step < cn) fetch(i + per_step, nhas, nw);
                uint32_t gm = 0;
                for (int k = i; k < min(cn, i + per_step); ++k) gm |= (uint32_t)__builtin_amdgcn_readlane((int)e_gm, k);
                // the points within reach of a needed group
                bool keep = false;
                while (gm) {
                    const int g = __builtin_ctz(gm);
                    gm &= gm - 1;
                    const uint32_t tg = (uint32_t)__builtin_amdgcn_readlane((int)t8, 8 * g);
                    keep = keep || group_d2(g, w.x, w.y, w.z, w.x, w.y, w.z) <= tg;
                }
                keep = keep && has;
                const uint64_t cand = __ballot(keep);
                const int steps = __popcll(cand);
                st_pts += (uint32_t)__popcll(__ballot(has));
                st_pairs += (uint32_t)steps * nin;
                if (held + steps > 64) {
                    drain();
                    // a lane whose cones all hold a point searches no
                    // farther than the farthest of them
                    uint32_t far = 0;
#pragma unroll
                    for (int c = 0; c < C::K; ++c) far = max(far, (uint32_t)(best[c * 64 + lane] >> 32));
                    if (mine && far < __float_as_uint(cap)) cap = __uint_as_float(far);
                    t8 = group8_max_u32(mine ? __float_as_uint(cap) : 0u);
                }
                if (keep) batch[held + __popcll(cand & lanemask_lt())] = w;
                held += steps;
            }
        }
        if (held > 0) drain();
        __builtin_amdgcn_wave_barrier();
        // results of these lanes: open when a cone's best lies beyond R_0
        bool open = false;
        uint64_t kmin = kEmptyKey;
#pragma unroll
        for (int c = 0; c < C::K; ++c) {
            const uint64_t k = best[cone_row<D>(c) * 64 + lane];
            open = open || key_bound(k) > (int32_t)__float_as_uint(r2);
            kmin = k < kmin ? k : kmin;
        }
        open = open && mine;
        if (reach) {
            // late cones (k_late_mark): nothing is left open here
            if (mine) reach[p] = open ? (int32_t)__float_as_uint(r2) : kReachAll;
            open = false;
        }
        open_lanes |= __ballot(open);
        // distinct points at float distance 0 break the grouping's
        // premise; the caller then searches ungrouped
        if (grouped && mine && (kmin >> 32) == 0u) underflow = true;
        if (mine) {
            const int64_t gs = is_rep ? (int64_t)dup.gslot[p] : 0;
            int32_t pmin = -1;
            for (int c = 0; c < C::K; ++c) {
                const uint64_t k = best[cone_row<D>(c) * 64 + lane];
                cand_key[(int64_t)c * n + p] = k;
                if (open) continue;
                const int32_t q = k == kEmptyKey ? -1 : inv[(uint32_t)k];
                cand_pos[(int64_t)c * n + p] = q;
                if (k == kmin) pmin = q;
                if (is_rep && ((c / C::NS) & 1) == 0) {
                    const int64_t b = (int64_t)((c / C::NS / 2) * C::NS + c % C::NS) * dup.ngroups + gs;
                    dup.bkey[b] = k;
                    dup.bpos[b] = q;
                }
            }
            if (!open && first_corr) {
                // (bests lie within R_0, so the smallest is exact)
                first_corr[p] = pmin >= 0 ? pmin : -2;
                first_key[p] = kmin;
            }
        }
        __builtin_amdgcn_wave_barrier();
    }
    if (lane == 0 && open_out) open_out[blockIdx.x] = open_lanes;
    if (collect_stats && lane == 0) cone_work(ctr, st_nodes, st_leaves, st_pts, st_pairs);
    if (__ballot(underflow) != 0ull && lane == 0) atomicOr(&ctr->underflow, 1u);
}

// Queries left open by a split cone search, in position order: per-packet
// counts (entry P = 0, so that the exclusive scan's entry P is the total),
// then each packet's open lanes at its scanned offset.
__global__ __launch_bounds__(kBlock) void k_open_count(const uint64_t* __restrict__ open_mask, int64_t P,
                                                      uint32_t* __restrict__ cnt)
{
    const int64_t b = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (b <= P) cnt[b] = b < P ? (uint32_t)__popcll(open_mask[b]) : 0u;
}

__global__ __launch_bounds__(64) void k_open_fill(const uint64_t* __restrict__ open_mask,
                                                 const uint32_t* __restrict__ off, int32_t* __restrict__ list)
{
    const int64_t b = blockIdx.x;
    const uint64_t m = open_mask[b];
    const int lane = __lane_id();
    if ((m >> lane) & 1ull) list[off[b] + (uint32_t)__popcll(m & lanemask_lt())] = (int32_t)(b * 64 + lane);
}

// The same compaction in three launches: per-tile exclusive scan of the
// packets' open counts (entry P = 0), the tile sums, then each packet's
// lanes at its offset (src: entries of a query list, else positions); the
// total lands in off[P].
__global__ __launch_bounds__(kBlock) void k_open_scan_local(const uint64_t* __restrict__ open_mask, int64_t P,
                                                           uint32_t* __restrict__ off, uint32_t* __restrict__ sums)
{
    __shared__ uint32_t sh[16];
    const int64_t base = (int64_t)blockIdx.x * kScanTile + (int64_t)threadIdx.x * kScanItems;
    uint32_t v[kScanItems];
    uint32_t t = 0;
    for (int j = 0; j < kScanItems; ++j) {
        v[j] = base + j < P ? (uint32_t)__popcll(open_mask[base + j]) : 0u;
        t += v[j];
    }
    uint32_t total;
    uint32_t run = block_excl_scan(t, sh, total);
    for (int j = 0; j < kScanItems; ++j) {
        if (base + j <= P) off[base + j] = run;
        run += v[j];
    }
    if (threadIdx.x == 0) sums[blockIdx.x] = total;
}

// the tile totals of tiles [0, t) summed by the whole wave (a few hundred
// tiles at most for 10^8 points: cheaper than a launch that scans them)
__device__ __forceinline__ uint32_t tiles_before(const uint32_t* __restrict__ sums, int64_t t)
{
    uint32_t a = 0;
    for (int64_t j = __lane_id(); j < t; j += 64) a += sums[j];
    for (int o = 32; o > 0; o >>= 1) a += (uint32_t)__shfl_xor((int)a, o);
    return a;
}

// (each wave takes a run of consecutive packets, the grid at most 2048
// blocks: the lists are built every round, and a launch of one block per
// packet costs more than its work when few are open; sums holds the tile
// totals of k_open_scan_local: each wave adds up the ones before its run's
// first tile, then the tiles it crosses)
__global__ __launch_bounds__(kBlock) void k_open_fill_scan(uint64_t* __restrict__ open_mask, int64_t P,
                                                          uint32_t* __restrict__ off,
                                                          const uint32_t* __restrict__ sums,
                                                          const int32_t* __restrict__ src, int32_t* __restrict__ dst)
{
    const int lane = __lane_id();
    const int64_t waves = (int64_t)gridDim.x * (kBlock / 64);
    const int64_t w0 = (int64_t)blockIdx.x * (kBlock / 64) + threadIdx.x / 64;
    if (w0 == 0) {
        const uint32_t pre = tiles_before(sums, P / kScanTile);
        if (lane == 0) off[P] += pre;
    }
    const int64_t per = (P + waves - 1) / waves;
    const int64_t b0 = w0 * per, b1 = min(P, b0 + per);
    if (b0 >= b1) return;
    int64_t t = b0 / kScanTile;
    uint32_t pre = tiles_before(sums, t);
    for (int64_t b = b0; b < b1; ++b) {
        if (b / kScanTile != t) {
            pre += sums[t];
            ++t;
        }
        const uint64_t m = wave_first_u64(open_mask[b]);
        if (m == 0ull) continue;
        // read once: cleared, so that the search that writes the next mask
        // need only write the words of its packets
        if (lane == 0) open_mask[b] = 0ull;
        if (!((m >> lane) & 1ull)) continue;
        const uint32_t o = off[b] + pre + (uint32_t)__popcll(m & lanemask_lt());
        dst[o] = src != nullptr ? src[b * 64 + lane] : (int32_t)(b * 64 + lane);
    }
}

void open_compact(uint64_t* open_mask, int64_t P, uint32_t* off, uint32_t* sums, const int32_t* src,
                  int32_t* dst, hipStream_t s)
{
    const int64_t nb = (P + 1 + kScanTile - 1) / kScanTile;
    hipLaunchKernelGGL(k_open_scan_local, dim3((unsigned)nb), dim3(kBlock), 0, s, open_mask, P, off, sums);
    const unsigned gf = (unsigned)std::min<int64_t>((P + kBlock / 64 - 1) / (kBlock / 64), 2048);
    hipLaunchKernelGGL(k_open_fill_scan, dim3(gf), dim3(kBlock), 0, s, open_mask, P, off, (const uint32_t*)sums,
                       src, dst);
}

// Start of a group refresh: m2 = ~0 for every group, dup_split = 0.
__global__ __launch_bounds__(kBlock) void k_dup_reset(Counters* __restrict__ C, DupState dup)
{
    if (C->done || C->dup_settled) return;
    const int64_t stride = (int64_t)gridDim.x * blockDim.x;
    const int64_t t0 = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (t0 == 0) C->dup_split = 0;
    for (int64_t g = t0; g < dup.ngroups; g += stride) dup.m2[g] = 0xffffffffu;
}

// Per group, the smallest member id whose component differs from the
// representative's (labels are distinct before round 1); dup_split is set
// when any group spans >= 2 components.  m2 holds ~0 on entry.
__global__ __launch_bounds__(kBlock) void k_dup_m2(const int32_t* __restrict__ label,
                                                  const float4* __restrict__ pts,
                                                  Counters* __restrict__ C, DupState dup)
{
    if (C->done || C->dup_settled) return;
    bool split = false;
    // every lane walks the same number of trips, so the wave-wide steps below
    // see all 64 lanes
    const int64_t stride = (int64_t)gridDim.x * blockDim.x;
    for (int64_t t0 = (int64_t)blockIdx.x * blockDim.x; t0 < dup.npoints; t0 += stride) {
        const int64_t t = t0 + threadIdx.x;
        bool valid = false;
        int32_t g = 0;
        uint32_t id = 0xffffffffu;
        if (t < dup.npoints) {
            const int32_t p = dup.list[t];
            const int32_t r = dup.rep[p];
            if (label[p] != label[r]) {
                valid = true;
                g = dup.gslot[r];
                id = __float_as_uint(pts[p].w);
            }
        }
        split |= valid;
        // lanes of one group (list entries of a group are mostly adjacent)
        // merge into one atomic; a lower value already there skips it
        const uint64_t vm = __ballot(valid);
        if (vm == 0ull) continue;
        const int32_t lg = __shfl(g, (int)__builtin_ctzll(vm));
        const bool grp = valid && g == lg;
        uint32_t v = grp ? id : 0xffffffffu;
        for (int off = 32; off > 0; off >>= 1) v = min(v, (uint32_t)__shfl_xor((int)v, off));
        if (__lane_id() == (int)__builtin_ctzll(vm) && __atomic_load_n(&dup.m2[lg], __ATOMIC_RELAXED) > v)
            atomicMin(&dup.m2[lg], v);
        if (valid && !grp && __atomic_load_n(&dup.m2[g], __ATOMIC_RELAXED) > id) atomicMin(&dup.m2[g], id);
    }
    if (__ballot(split) != 0ull && __lane_id() == 0 && __atomic_load_n(&C->dup_split, __ATOMIC_RELAXED) == 0u)
        atomicOr(&C->dup_split, 1u);
}

// Cones of the group points.  A point whose location is shared with another
// component (before round 1: with any other point) has d2 = 0 to it; the zero
// vector lies in exactly the '+'-face cones, where (0, smallest such id)
// beats every other key.  The smallest group id of another component is the
// representative's id when p's component differs from the representative's,
// else m2.  Otherwise the '+' cones are the representative's own (kept at its
// search; no point at the shared location is a candidate).  The '-' cones are
// always the representative's: the zero vector is in no '-' cone.  first_corr
// / first_key (round 1) take the smallest key over the point's cones.
template <int D>
__global__ __launch_bounds__(kBlock) void k_dup_fill(int64_t n, const int32_t* __restrict__ label,
                                                    const float4* __restrict__ pts,
                                                    const int32_t* __restrict__ inv,
                                                    uint64_t* __restrict__ cand_key,
                                                    int32_t* __restrict__ cand_pos,
                                                    int32_t* __restrict__ revive,
                                                    int32_t* __restrict__ first_corr,
                                                    uint64_t* __restrict__ first_key,
                                                    const Counters* __restrict__ C, DupState dup)
{
    using CC = ConeCfg<D>;
    if (C->done || C->dup_settled) return;
    for (int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; t < dup.npoints;
         t += (int64_t)gridDim.x * blockDim.x) {
        const int32_t p = dup.list[t];
        const int32_t r = dup.rep[p];
        const int64_t g = dup.gslot[r];
        const uint32_t m2 = dup.m2[g];
        const bool zero = m2 != 0xffffffffu;
        uint32_t z = 0;
        int32_t zpos = -1;
        if (zero) {
            z = label[p] != label[r] ? __float_as_uint(pts[r].w) : m2;
            zpos = inv[z];
        }
        uint64_t kmin = kEmptyKey;
        int32_t pmin = -1;
        // the representative's '-' cones are read, never written, here
        for (int c = 0; c < CC::K; ++c) {
            const int64_t o = (int64_t)c * n;
            uint64_t k;
            int32_t q;
            if (((c / CC::NS) & 1) == 0) {
                const int64_t b = (int64_t)((c / CC::NS / 2) * CC::NS + c % CC::NS) * dup.ngroups + g;
                k = zero ? (uint64_t)z : dup.bkey[b];
                q = zero ? zpos : dup.bpos[b];
                cand_key[o + p] = k;
                cand_pos[o + p] = q;
            } else {
                k = cand_key[o + r];
                q = cand_pos[o + r];
                if (p != r) {
                    cand_key[o + p] = k;
                    cand_pos[o + p] = q;
                }
            }
            if (k < kmin) { kmin = k; pmin = q; }
        }
        if (first_corr) {
            first_corr[p] = pmin >= 0 ? pmin : -2;
            first_key[p] = kmin;
        }
        if (revive && revive[p] == -2) revive[p] = -1;
    }
}

// ------------------------------------------------------- Boruvka rounds
__global__ __launch_bounds__(kBlock) void k_round_init(int64_t n, int32_t* __restrict__ label,
                                                      int32_t* __restrict__ label2,
                                                      int32_t* __restrict__ eu,
                                                      int32_t* __restrict__ corr,
                                                      uint64_t* __restrict__ corr_key,
                                                      uint64_t* __restrict__ comp1,
                                                      uint32_t* __restrict__ comp2, Counters* C,
                                                      uint32_t target, uint32_t max_rounds)
{
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i == 0) {
        C->edges = 0; C->research = 0; C->zero_or_empty = 0; C->unflat = 0;
        C->round = 0; C->done = C->invalid ? 1u : 0u; C->edges_prev = 0; C->dup_settled = 0; C->nsamples = 0;
        C->comp_queries = 0;
        C->deferred = 0;
        C->knn_round1 = 0;
        C->target = target; C->max_rounds = max_rounds;
    }
    if (i < kWorkKinds * kWorkSlots) C->work[i / kWorkSlots][i % kWorkSlots] = 0;
    if (i >= n) return;
    label[i] = (int32_t)i;          // K_EMST_initDisjointSet (EMSTOperators.h:330-343)
    label2[i] = (int32_t)i;
    eu[i] = -1;                     // no edge absorbed this root yet
    corr[i] = -1;                   // correspondenceMap reset (SolutionEMST.cu:464-466)
    corr_key[i] = kEmptyKey;
    comp1[i] = kEmptyKey;
    comp2[i] = 0xffffffffu;
}

// round 1 with its targets from k_knn_first (Counters::knn_round1)
__device__ __forceinline__ bool knn_round1(const Counters* C) { return C->round == 1u && C->knn_round1 != 0u; }

// Termination is tested before a round (SolutionEMSTOperators.cu:194-227 and
// the 100-round cap): the tree is complete or the cap is reached.  While
// done != 0 every round kernel returns at once, so rounds can be issued
// ahead (a captured graph of several rounds) and stop by themselves.
__global__ void k_round_begin(Counters* C)
{
    if (C->done) return;
    if (C->edges >= C->target || C->round >= C->max_rounds) {
        C->done = 1;
        return;
    }
    C->round += 1;
    C->edges_prev = C->edges;
    C->nroots = 0;
    C->walk_left = 0;
    C->late = 0;
    C->late_checks = 0;
    C->deferred = 0;
}

// A round that added no edge leaves a forest with no outgoing candidate: done.
// A flatten that hit its step cap pauses the rounds until the host has
// finished it.  Coincident groups stop being refreshed once none spans two
// components (components only merge).  stamps (one-launch runs): the
// device's constant-rate clock at the end of each round that ran, at
// stamps[round].
__global__ void k_round_end(Counters* C, int grouped, unsigned long long* stamps, uint32_t cap)
{
    if (C->done) return;
    if (stamps != nullptr && C->round <= cap) stamps[C->round] = wall_clock64();
    if (C->unflat) {
        C->done = 2;
        return;
    }
    if (grouped && !C->dup_settled && C->dup_split == 0u) C->dup_settled = 1;
    // (the next round's own test, made here, so that the host need not issue
    // another batch of rounds to learn it)
    if (C->edges == C->edges_prev || C->edges >= C->target || C->round >= C->max_rounds) C->done = 1;
}

__global__ void k_stamp(unsigned long long* at)
{
    *at = wall_clock64();
}

// Points that must search again next round: a zero-distance cone or no cone
// at all (NodeEMST.h:1051-1077).
__global__ __launch_bounds__(kBlock) void k_flag_research(int K, int64_t n,
                                                         const uint64_t* __restrict__ cand_key,
                                                         int32_t* __restrict__ list,
                                                         const int32_t* __restrict__ reach, Counters* C)
{
    const int64_t p = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    bool zero = false, any = p >= n;
    for (int k = 0; k < K && p < n; ++k) {
        const uint64_t key = cand_key[(int64_t)k * n + p];
        if (key == kEmptyKey) continue;
        any = true;
        zero |= (key >> 32) == 0u;
    }
    if (reach) {
        // (late cones: not known to be empty)
        const bool blind = !any && reach[p] != kReachAll;
        any = any || blind;
        const uint64_t m = __ballot(blind);
        if (m != 0ull && __lane_id() == 0)
            atomicAdd(&C->work[kWorkBlind][blockIdx.x % kWorkSlots], (unsigned long long)__popcll(m));
    }
    if (zero || !any) {
        atomicAdd(&C->zero_or_empty, 1u);
        list[atomicAdd(&C->research, 1u)] = (int32_t)p;
    }
}

// Component minima: one atomic per run of equal labels in a wave
// (atomic_min_grouped).  In round 2 of the clustered 10^7 cloud, with
// components of about 3 points, per-lane atomics took 0.15 of the keep pass's
// 0.35 ms.
// The minima only decrease, so a value read (even a stale one) that is
// already <= the key makes the atomic redundant: late rounds, whose few large
// components would otherwise take one atomic per wave on the same address,
// mostly skip it.
__device__ __forceinline__ void atomic_min_if_lower(uint64_t* a, uint64_t key)
{
    if (__atomic_load_n(a, __ATOMIC_RELAXED) > key) atomicMin((unsigned long long*)a, (unsigned long long)key);
}

__device__ __forceinline__ void atomic_min_grouped(uint64_t* arr, int32_t lab, uint64_t key, bool valid)
{
    if (__ballot(valid) == 0ull) return;
    // runs of equal labels across consecutive lanes (the lanes hold
    // consecutive positions or queries, and a component's points lie close
    // together in position order): a segmented minimum from the right leaves
    // each run's minimum in its first lane, which alone updates the entry;
    // a lane past the run reads its own label, so runs never merge
    const int lane = __lane_id();
    const int32_t prev = __shfl_up(lab, 1);
    const uint64_t heads = __ballot(lane == 0 || prev != lab) | 1ull;
    const int seg = 63 - __builtin_clzll(heads & (~0ull >> (63 - lane)));
    uint64_t v = valid ? key : kEmptyKey;
#pragma unroll
    for (int d = 1; d < 64; d <<= 1) {
        const int src = lane + d < 64 ? lane + d : lane;
        const uint32_t lo = (uint32_t)__shfl((int)(uint32_t)v, src);
        const uint32_t hi = (uint32_t)__shfl((int)(uint32_t)(v >> 32), src);
        const int oseg = __shfl(seg, src);
        const uint64_t o = ((uint64_t)hi << 32) | lo;
        if (oseg == seg && o < v) v = o;
    }
    if (seg == lane && v != kEmptyKey) atomic_min_if_lower(&arr[lab], v);
}

// The same with one group, the first valid lane's label: lanes holding it
// merge into one atomic, the rest issue their own.  Fewer live registers than
// the segmented form: in the component search (80 VGPRs at 6 waves per SIMD)
// the segmented form spilled 48 instead of 20 bytes a lane, doubled the
// search's writes (0.50 -> 0.99 GB per EMST) and cost 0.12 ms.
__device__ __forceinline__ void atomic_min_leader(uint64_t* arr, int32_t lab, uint64_t key, bool valid)
{
    const uint64_t vm = __ballot(valid);
    if (vm == 0ull) return;
    const int leader = __builtin_ctzll(vm);
    const int32_t llab = __shfl(lab, leader);
    const bool grp = valid && lab == llab;
    const uint64_t gm = __ballot(grp);
    uint64_t v = grp ? key : kEmptyKey;
    if (__popcll(gm) > 1) {
        for (int off = 32; off > 0; off >>= 1) {
            const uint64_t o = (uint64_t)__shfl_xor((long long)v, off);
            v = o < v ? o : v;
        }
        if (__lane_id() == leader) atomic_min_if_lower(&arr[llab], v);
        if (valid && !grp) atomic_min_if_lower(&arr[lab], key);
    } else if (valid) {
        atomic_min_if_lower(&arr[lab], key);
    }
}

// Each point's cone candidates in key order, for the rounds (bitonic network
// over K padded to a power of two, all indices static so the keys stay in
// registers): rkey[p*K + r], rpos[p*K + r] = key and sorted position of the
// candidate of rank r; cursor[p] = 0.  Equal keys carry equal positions (a
// key holds the candidate's id; empty cones and the padding are (~0, -1)),
// so the position rides along as payload and ranks 0..K-1 are exactly the K
// cones.  Point-major rows keep a point's next ranks in one cache line for
// k_round_min; each row is written with 16-byte stores.  Points: [0, n) or
// qlist[0..nq); with C the kernel does nothing once the rounds are done or
// the groups have settled (it follows a group refresh in a replayed round).
template <int D>
__global__ __launch_bounds__(kBlock) void k_rank_cones(int64_t n, const uint64_t* __restrict__ cand_key,
                                                      const int32_t* __restrict__ cand_pos,
                                                      const int32_t* __restrict__ qlist, int64_t nq,
                                                      uint64_t* __restrict__ rkey, int32_t* __restrict__ rpos,
                                                      uint8_t* __restrict__ cursor,
                                                      const int32_t* __restrict__ reach,
                                                      const Counters* __restrict__ C)
{
    using CC = ConeCfg<D>;
    constexpr int P = CC::K <= 8 ? 8 : 32;
    static_assert(CC::K % 4 == 0, "rows are written in 16-byte pieces");
    if (C && (C->done || C->dup_settled)) return;
    const int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= nq) return;
    const int64_t p = qlist ? (int64_t)qlist[t] : t;
    const int32_t upto = reach ? reach[p] : kReachAll;
    uint64_t key[P];
    int32_t pos[P];
#pragma unroll
    for (int c = 0; c < P; ++c) {
        key[c] = c < CC::K ? cand_key[(int64_t)c * n + p] : kEmptyKey;
        pos[c] = c < CC::K ? cand_pos[(int64_t)c * n + p] : -1;
    }
    // a late point's cones past its first radius are not exact yet
    if (upto != kReachAll)
#pragma unroll
        for (int c = 0; c < P; ++c)
            if (key_bound(key[c]) > upto) {
                key[c] = kEmptyKey;
                pos[c] = -1;
            }
#pragma unroll
    for (int k = 2; k <= P; k <<= 1)
#pragma unroll
        for (int j = k >> 1; j > 0; j >>= 1)
#pragma unroll
            for (int i = 0; i < P; ++i) {
                const int l = i ^ j;
                if (l > i) {
                    const bool up = (i & k) == 0;
                    if ((key[i] > key[l]) == up && key[i] != key[l]) {
                        const uint64_t tk = key[i]; key[i] = key[l]; key[l] = tk;
                        const int32_t tp = pos[i]; pos[i] = pos[l]; pos[l] = tp;
                    }
                }
            }
    uint4* __restrict__ ko = reinterpret_cast<uint4*>(rkey + p * CC::K);
    uint4* __restrict__ po = reinterpret_cast<uint4*>(rpos + p * CC::K);
#pragma unroll
    for (int r = 0; r < CC::K; r += 2)
        ko[r / 2] = make_uint4((uint32_t)key[r], (uint32_t)(key[r] >> 32), (uint32_t)key[r + 1],
                               (uint32_t)(key[r + 1] >> 32));
#pragma unroll
    for (int r = 0; r < CC::K; r += 4)
        po[r / 4] = make_uint4((uint32_t)pos[r], (uint32_t)pos[r + 1], (uint32_t)pos[r + 2], (uint32_t)pos[r + 3]);
    cursor[p] = 0;
}

// find min 1 (NodeEMST.h:1303-1384) + first phase of the component minimum:
// per point, keep the previous target while it is outside the component,
// else the (d2, id)-smallest cone candidate with another label; then
// atomicMin of (d2 bits, min id) on the component root.
//
// The smallest outgoing candidate is the first, in key order, whose label
// differs: the cones are ranked once (k_rank_cones) and cursor[p] skips the
// ones already found inside the component, which never leave it (components
// only merge), so each candidate is looked at about once over all rounds.
__device__ __forceinline__ void round_min_point(bool inb, int64_t p, int K, const uint32_t* __restrict__ ids,
                                                const uint64_t* __restrict__ rkey,
                                                const int32_t* __restrict__ rpos, uint8_t* __restrict__ cursor,
                                                const int32_t* __restrict__ label, int32_t* __restrict__ corr,
                                                uint64_t* __restrict__ corr_key, uint64_t* __restrict__ comp1)
{
    int32_t lp = 0;
    uint64_t key1 = kEmptyKey;
    bool valid = false, held = false;
    if (inb) {
        lp = label[p];
        int32_t c = corr[p];
        uint64_t ck = corr_key[p];
        // corr == -2: every cone candidate already inside the component;
        // since components only merge, the point never has an outgoing
        // candidate again (until a repeated cone search or a group
        // refresh gives it new candidates)
        if (c <= late_held(0)) {
            // (late cones) it bounds the component's edge while it is outside;
            // its key stays as the point's lower bound
            held = label[late_held(c)] != lp;
            if (!held) corr[p] = -2;
        } else if (c != -2 && !(c >= 0 && label[c] != lp)) {
            c = -1;
            ck = kEmptyKey;
            // kStep ranks per step, their loads independent of each other,
            // so a long run of candidates inside the component costs few
            // round trips to memory
            constexpr int kStep = 4;
            int r = cursor[p];
            bool more = r < K;
            const uint64_t* __restrict__ kr = rkey + p * (int64_t)K;
            const int32_t* __restrict__ pr = rpos + p * (int64_t)K;
            while (more) {
                uint64_t key[kStep];
                int32_t q[kStep], lq[kStep];
#pragma unroll
                for (int i = 0; i < kStep; ++i) {
                    key[i] = kEmptyKey;
                    q[i] = -1;
                    if (r + i < K) {
                        key[i] = kr[r + i];
                        q[i] = pr[r + i];
                    }
                }
#pragma unroll
                for (int i = 0; i < kStep; ++i) lq[i] = key[i] != kEmptyKey ? label[q[i]] : lp;
#pragma unroll
                for (int i = 0; i < kStep; ++i) {
                    if (!more) continue;
                    if (key[i] == kEmptyKey) {      // ranked last: no outgoing candidate left
                        r = K;
                        more = false;
                    } else if (lq[i] != lp) {
                        ck = key[i];
                        c = q[i];
                        more = false;
                    } else {
                        ++r;
                    }
                }
                more = more && r < K;
            }
            cursor[p] = (uint8_t)r;
            corr[p] = c == -1 ? -2 : c;
            if (c != -1) corr_key[p] = ck;
        }
        if (c >= 0 || held) {
            const uint32_t pid = ids[p];
            const uint32_t qid = (uint32_t)ck;
            key1 = (ck & 0xffffffff00000000ull) | (uint64_t)min(pid, qid);
            valid = true;
        }
    }
    atomic_min_grouped(comp1, lp, key1, valid);
}

__global__ __launch_bounds__(kBlock) void k_round_min(int K, int64_t n, const uint32_t* __restrict__ ids,
                                                     const uint64_t* __restrict__ rkey,
                                                     const int32_t* __restrict__ rpos,
                                                     uint8_t* __restrict__ cursor,
                                                     const int32_t* __restrict__ label,
                                                     int32_t* __restrict__ corr,
                                                     uint64_t* __restrict__ corr_key,
                                                     uint64_t* __restrict__ comp1, const Counters* C)
{
    if (C->done) return;
    const int64_t p = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    round_min_point(p < n, p, K, ids, rkey, rpos, cursor, label, corr, corr_key, comp1);
}

// a member's edge key, high part: (d2, min id); the max id completes it
__device__ __forceinline__ uint64_t edge_key1(uint64_t ck, uint32_t pid)
{
    return (ck & 0xffffffff00000000ull) | (uint64_t)min(pid, (uint32_t)ck);
}

// Late cones.  A first pass of the cone search leaves a point late when a cone
// of it has no point within R_0: its cones are exact up to reach[p] (the bits
// of R_0^2; -1: none is known; kReachAll: all are exact), and only the exact
// ones are ranked.  The rounds go on without the rest: a late point matters
// only in a round in which every exact candidate of its has joined its
// component while an unknown one could be its component's smallest edge
// (late_first, from its reach and the nearest outside point beyond it that an
// earlier round found, corr_key).  Those points are listed here, after the
// round's minima.  Few of them get their cones searched to the end
// (k_cone_rest).  More of them pause the round, and their nearest points
// outside the component are searched instead (launch_late_search).
//
// A nearest outside point so found that was not its component's edge is held
// (late_held).  While it stays outside, it takes part in the minima, so that
// few points of isolated clusters are asked again, and its owner is asked only
// when its edge is the smallest.  Without it every point of a component with
// no other edge was: solid blocks of 64 voxels apart from each other
// (110592 points, whose every gap ties) 587000 points searched in 8 rounds and
// 3.25 ms a run, now 207000 and 2.39.
constexpr int kLateChunk = 2048;        // points per block: one list reservation each
constexpr int kLatePer = kLateChunk / kBlock;

__global__ __launch_bounds__(kBlock) void k_late_mark(int64_t n, const uint32_t* __restrict__ ids,
                                                     const int32_t* __restrict__ label,
                                                     const int32_t* __restrict__ corr,
                                                     uint64_t* __restrict__ corr_key,
                                                     const uint64_t* __restrict__ comp1,
                                                     const int32_t* __restrict__ reach,
                                                     int32_t* __restrict__ list, Counters* C)
{
    if (C->done) return;
    __shared__ uint32_t wsum[kBlock / 64];
    __shared__ uint32_t base;
    const int64_t c0 = (int64_t)blockIdx.x * kLateChunk + (int64_t)(threadIdx.x / 64) * 64 * kLatePer + __lane_id();
    uint32_t bits = 0, tot = 0;
    uint32_t at[kLatePer];
#pragma unroll
    for (int i = 0; i < kLatePer; ++i) {
        const int64_t p = c0 + i * 64;
        bool need = false;
        const int32_t c = p < n ? corr[p] : 0;
        if (c == -2) {
            const int32_t r = reach[p];
            if (r != kReachAll) {
                const uint64_t ck = corr_key[p], edge = comp1[label[p]];
                uint64_t first = late_first(r, ck, 0u);
                // (its id matters where the d2 ties)
                if (first >> 32 == edge >> 32) first = late_first(r, ck, ids[p]);
                need = first <= edge;
                // (the paused search starts there)
                if (need && first >> 32 != 0u) corr_key[p] = first | 0xffffffffull;
            }
        } else if (c <= late_held(0)) {
            need = edge_key1(corr_key[p], ids[p]) == comp1[label[p]];
        }
        const uint64_t m = __ballot(need);
        at[i] = tot + (uint32_t)__popcll(m & lanemask_lt());
        tot += (uint32_t)__popcll(m);
        if (need) bits |= 1u << i;
    }
    const int w = threadIdx.x / 64;
    if (__lane_id() == 0) wsum[w] = tot;
    __syncthreads();
    if (threadIdx.x == 0) {
        uint32_t t = 0;
        for (int j = 0; j < kBlock / 64; ++j) {
            const uint32_t x = wsum[j];
            wsum[j] = t;
            t += x;
        }
        base = t ? atomicAdd(&C->late, t) : 0u;
    }
    __syncthreads();
#pragma unroll
    for (int i = 0; i < kLatePer; ++i)
        if ((bits >> i) & 1u) list[base + wsum[w] + at[i]] = (int32_t)(c0 + i * 64);
}

// points without a candidate left look again (their cones are exact now)
__global__ __launch_bounds__(kBlock) void k_revive(int64_t n, int32_t* __restrict__ corr)
{
    const int64_t p = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (p < n && corr[p] <= -2) corr[p] = -1;
}

// After the search of the listed points' nearest points outside their
// components: a point whose edge is its component's smallest keeps it as its
// target and is listed for k_cone_rest's check (not in round 1, where every
// point is a component and its nearest point is the smallest cone candidate);
// the others wait (late_held, or the d2 where their search stopped as a lower
// bound).  A pair at distance zero is left to the exact cones (done = 4), with
// its rule of repeated searches.
__global__ __launch_bounds__(kBlock) void k_late_settle(const int32_t* __restrict__ list,
                                                       const uint32_t* __restrict__ ids,
                                                       const int32_t* __restrict__ label,
                                                       int32_t* __restrict__ corr,
                                                       const uint64_t* __restrict__ corr_key,
                                                       const uint64_t* __restrict__ comp1,
                                                       int32_t* __restrict__ check, Counters* C)
{
    if (C->done) return;
    const int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    const bool on = t < (int64_t)C->late;
    bool keep = false;
    int32_t p = 0;
    if (on) {
        p = list[t];
        if (corr[p] >= 0) {
            const uint64_t ck = corr_key[p];
            keep = edge_key1(ck, ids[p]) == comp1[label[p]];
            if ((ck >> 32) == 0u) C->done = 4u;
        }
        if (!keep) corr[p] = corr[p] >= 0 ? late_held(corr[p]) : -2;
    }
    const bool add = keep && C->round > 1u;
    const uint64_t m = __ballot(add);
    if (m == 0ull) return;
    uint32_t base = 0;
    if (__lane_id() == (int)__builtin_ctzll(m)) base = atomicAdd(&C->late_checks, (uint32_t)__popcll(m));
    base = (uint32_t)__shfl((int)base, (int)__builtin_ctzll(m));
    if (add) check[base + (uint32_t)__popcll(m & lanemask_lt())] = p;
}

// The open cones of listed points, searched to the end: one wave per point,
// one tree node per lane.  A step takes the 32 nearest-first nodes on top of
// the stack, tests their 64 children against the cones' bounds, sorts the
// needed ones by distance, reads the leaves among them (64 points at a time)
// and pushes the rest, nearest on top.  Lane c keeps cone c; cones exact to
// reach[p] are closed, the bests found beyond it are bounds.
//
// Against packets of 64 queries (k_cone_search from pass 1), whose wave walks
// the union of their trees one node at a time: a few listed points lie apart,
// and a packet of 25 took 8 ms; here each takes some 100 us, 20 ns in a full
// launch.  Packets of neighbouring queries share their walk and are the faster
// ones for many (400000 points of 10^6: 1.8 against 6.4 ms).
//
// kRestCheck: whether a late point's target is its cone's nearest point (the
// target's cones, up to its distance); if not, done = 4.
constexpr int kRestStack = 1024;
constexpr int kRestBlocks = 5120;       // 20 waves a CU
constexpr int kRestReserve = 64;        // left for a plain descent (one node a step)

__global__ __launch_bounds__(64) void k_cone_rest(ConeRest a, const uint32_t* __restrict__ nq_dev, int64_t few,
                                                  int mode)
{
    using CC = ConeCfg<3>;
    const int64_t nq = (int64_t)*nq_dev;
    if ((int64_t)blockIdx.x >= nq || a.C->done) return;
    if (nq > few) {
        // too many for one wave each: packets (k_cone_search); a round waits
        if (mode == kRestRound && blockIdx.x == 0 && threadIdx.x == 0) a.C->done = 3u;
        return;
    }
    __shared__ unsigned long long stk[kRestStack];
    __shared__ unsigned long long best[CC::K];
    const int lane = __lane_id();
    const int64_t n = a.n;
    const int lb = 31 - __builtin_clz(a.bucket);
    const int per_step = 64 >> lb;
    uint32_t st_nodes = 0, st_leaves = 0;
    for (int64_t qi = blockIdx.x; qi < nq; qi += gridDim.x) {
        const int32_t p = __builtin_amdgcn_readfirstlane(a.list[qi]);
        const int cl = find_cloud(a.clouds, a.ncl, p);
        const int64_t cend = a.clouds[cl].pos + a.clouds[cl].n;
        const int64_t L = a.clouds[cl].L, lfirst = a.clouds[cl].lfirst, nl = a.clouds[cl].nl;
        const Node* __restrict__ tree = a.nodes + 2 * a.clouds[cl].lbase;
        const float4 me = a.pts[p];
        const float px = me.x, py = me.y, pz = me.z;
        int32_t inner = -1;
        unsigned long long mine = kEmptyKey;
        uint64_t open = 0;
        if (mode == kRestCheck) {
            const float4 q = a.pts[a.corr[p]];
            open = cone_mask<3>(q.x - px, q.y - py, q.z - pz);
            mine = a.corr_key[p];
        } else {
            inner = a.reach[p];
            if (lane < CC::K) mine = a.cand_key[(int64_t)lane * n + p];
            open = __ballot(lane < CC::K && key_bound(mine) > inner);
        }
        __builtin_amdgcn_wave_barrier();
        if (lane < CC::K) best[lane] = mine;
        __builtin_amdgcn_wave_barrier();
        // in a round the cones need be exact only up to the component's edge,
        // so up to any outside point met (k_late_seen)
        const int32_t lp = a.label[p];
        int32_t cap = mode == kRestRound ? key_bound(a.comp1[lp]) : kReachAll;
        cap = __builtin_amdgcn_readfirstlane(cap);
        int32_t bound[CC::K];
        int32_t maxb = -1;
        auto refresh = [&]() {
            maxb = -1;
#pragma unroll
            for (int c = 0; c < CC::K; ++c) {
                const int32_t b = (open >> c) & 1ull
                                      ? min(cap, __builtin_amdgcn_readfirstlane(key_bound(best[c]))) : -1;
                bound[c] = b;
                maxb = max(maxb, b);
            }
        };
        refresh();
        // one step's leaves, in the order of their lanes
        auto leaves = [&](uint64_t lm, uint64_t key) {
            while (lm) {
                // the next per_step leaves; lane -> its leaf's lane
                int src = -1, got = 0;
                while (got < per_step && lm) {
                    const int l = (int)__builtin_ctzll(lm);
                    lm &= lm - 1;
                    if ((int32_t)__builtin_amdgcn_readlane((int)(key >> 32), l) > maxb) continue;
                    if (got == (lane >> lb)) src = l;
                    ++got;
                }
                if (got == 0) break;
                st_leaves += (uint32_t)got;
                const int node = __shfl((int)(uint32_t)key, src < 0 ? 0 : src);
                bool low = false;
                uint32_t out = 0xffffffffu;
                if (src >= 0) {
                    int64_t s0, s1;
                    leaf_range(a.lt, lfirst, nl, cend, node - L, s0, s1);
                    s0 += lane & (a.bucket - 1);
                    if (s0 < s1) {
                        const float4 v = a.pts[s0];
                        const float dx = v.x - px, dy = v.y - py, dz = v.z - pz;
                        const float d2 = d2_of(dx, dy, dz);
                        const int32_t db = (int32_t)__float_as_uint(d2);
                        if (s0 != (int64_t)p && db <= maxb && db > inner) {
                            if (mode == kRestRound && a.label[s0] != lp) out = (uint32_t)db;
                            uint32_t cm = cone_mask<3>(dx, dy, dz) & (uint32_t)open;
                            const unsigned long long kk =
                                ((unsigned long long)__float_as_uint(d2) << 32) | __float_as_uint(v.w);
                            while (cm) {
                                const int c = __builtin_ctz(cm);
                                cm &= cm - 1;
                                if (kk < best[c]) {
                                    atomicMin(&best[c], kk);
                                    low = true;
                                }
                            }
                        }
                    }
                }
                __builtin_amdgcn_wave_barrier();
                if (__ballot(out < (uint32_t)cap) != 0ull) cap = min(cap, (int32_t)wave_min_u32(out));
                if (__ballot(low) != 0ull) refresh();
            }
        };
        int sp;
        if (L == 1) {
            sp = 0;
            if (open) leaves(1ull, (uint64_t)1);
        } else {
            sp = (int)(L / 2 < 32 ? L / 2 : 32);
            if (lane < sp) stk[lane] = (unsigned long long)(sp + lane);
        }
        if (!open) sp = 0;
        __builtin_amdgcn_wave_barrier();
        while (sp > 0) {
            const int room = kRestStack - kRestReserve - sp;
            const int take = min(min(sp, 32), max(1, room));
            const bool on = (lane >> 1) < take;
            const unsigned long long e = on ? stk[sp - 1 - (lane >> 1)] : kEmptyKey;
            sp -= take;
            uint64_t key = kEmptyKey;
            if (on && (int32_t)(e >> 32) <= maxb) {
                const int child = 2 * (int)(uint32_t)e + (lane & 1);
                const Node x = tree[child];
                if (node_needed<3, 3>(x, px, py, pz, bound, maxb, inner, false)) {
                    const float m0 = fmaxf(fmaxf(x.lo[0] - px, px - x.hi[0]), 0.f);
                    const float m1 = fmaxf(fmaxf(x.lo[1] - py, py - x.hi[1]), 0.f);
                    const float m2 = fmaxf(fmaxf(x.lo[2] - pz, pz - x.hi[2]), 0.f);
                    const float m = d2_of(m0, m1, m2);
                    key = (uint64_t)__float_as_uint(m) << 32 | (uint32_t)child;
                }
            }
            ++st_nodes;
            if (__ballot(key != kEmptyKey) == 0ull) continue;
            key = wave_sort_u64(key);
            leaves(__ballot(key != kEmptyKey && (int64_t)(uint32_t)key >= L), key);
            const bool go = key != kEmptyKey && (int64_t)(uint32_t)key < L && (int32_t)(key >> 32) <= maxb;
            const uint64_t gm = __ballot(go);
            const int cnt = __popcll(gm);
            if (go) stk[sp + cnt - 1 - __popcll(gm & lanemask_lt())] = key;
            sp += cnt;
            __builtin_amdgcn_wave_barrier();
        }
        __builtin_amdgcn_wave_barrier();
        if (mode == kRestCheck) {
            if (__ballot(((open >> lane) & 1ull) && best[lane < CC::K ? lane : 0] == mine) == 0ull && lane == 0)
                a.C->done = 4u;
            continue;
        }
        // results
        const bool held = a.corr[p] <= late_held(0);
        const uint64_t was = edge_key1(a.corr_key[p], a.ids[p]);
        uint64_t key = kEmptyKey;
        int32_t pos = -1;
        if (lane < CC::K) {
            key = best[lane];
            pos = key == kEmptyKey ? -1 : a.inv[(uint32_t)key];
            a.cand_key[(int64_t)lane * n + p] = key;
            a.cand_pos[(int64_t)lane * n + p] = pos;
        }
        if (lane == 0) a.reach[p] = cap;        // (kReachAll without one)
        key = wave_sort_u64(key_bound(key) <= cap ? key : kEmptyKey);
        pos = key == kEmptyKey ? -1 : a.inv[(uint32_t)key];
        if (lane < CC::K) {
            a.rkey[(int64_t)p * CC::K + lane] = key;
            a.rpos[(int64_t)p * CC::K + lane] = pos;
        }
        // (a pair at distance zero: its rule of repeated searches, as in k_late_settle)
        if (lane == 0 && (key >> 32) == 0u) a.C->done = 4u;
        const uint64_t outm = __ballot(pos >= 0 && a.label[pos >= 0 ? pos : 0] != lp);
        const int first = outm ? (int)__builtin_ctzll(outm) : CC::K;
        if (lane == (outm ? first : 0)) {
            a.cursor[p] = (uint8_t)first;
            const uint64_t k1 = outm ? edge_key1(key, a.ids[p]) : kEmptyKey;
            // (a held edge that no cone has stays held, for k_late_seen; a
            // target that is still outside was the smallest candidate, and
            // stays it)
            if (!held || k1 == was) {
                a.corr[p] = outm ? pos : -2;
                a.corr_key[p] = outm ? key : kEmptyKey;
                if (outm) atomic_min_if_lower(&a.comp1[lp], k1);
            }
        }
    }
    if (lane == 0) {
        const int slot = (int)(blockIdx.x % kWorkSlots);
        atomicAdd(&a.C->work[kWorkConeNodes][slot], (unsigned long long)st_nodes);
        atomicAdd(&a.C->work[kWorkConeLeaves][slot], (unsigned long long)st_leaves);
        atomicAdd(&a.C->work[kWorkConePairs][slot], (unsigned long long)st_leaves * (unsigned long long)a.bucket);
    }
}

// A listed point searched up to its nearest outside point without finding a
// candidate there: a cone's nearest point is one of its component, which lies
// nearer to that outside point and so has the smaller edge.  The component's
// edge is then within what the point has seen; if not (in floats), the run
// needs exact cones.  So it does where the edge is one held until now that is
// no cone's; another such point takes its ranked candidates from here on.
__global__ __launch_bounds__(kBlock) void k_late_seen(const int32_t* __restrict__ list,
                                                     const uint32_t* __restrict__ ids,
                                                     const int32_t* __restrict__ label,
                                                     int32_t* __restrict__ corr,
                                                     const uint64_t* __restrict__ corr_key,
                                                     const uint64_t* __restrict__ comp1,
                                                     const int32_t* __restrict__ reach, Counters* C)
{
    if (C->done) return;
    const uint32_t t = blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= C->late) return;
    const int32_t p = list[t], c = corr[p], r = reach[p];
    if (c >= 0) return;
    const uint64_t edge = comp1[label[p]];
    if (c <= late_held(0)) {
        if (edge_key1(corr_key[p], ids[p]) == edge) C->done = 4u;
        corr[p] = -1;
    } else if (r != kReachAll && (r < 0 || (uint32_t)(edge >> 32) > (uint32_t)r)) {
        C->done = 4u;
    }
}

// second phase: among members matching (d2, min id), the smallest max id.
__global__ __launch_bounds__(kBlock) void k_round_comp2(int64_t n, const uint32_t* __restrict__ ids,
                                                       const int32_t* __restrict__ label,
                                                       const int32_t* __restrict__ corr,
                                                       const uint64_t* __restrict__ corr_key,
                                                       const uint64_t* __restrict__ comp1,
                                                       uint32_t* __restrict__ comp2, const Counters* C)
{
    if (C->done || knn_round1(C)) return;       // one member per component (see k_round_hook)
    const int64_t p = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (p >= n || corr[p] < 0) return;
    const int32_t lp = label[p];
    const uint64_t ck = corr_key[p];
    const uint32_t pid = ids[p];
    if (edge_key1(ck, pid) == comp1[lp]) atomicMin(&comp2[lp], max(pid, (uint32_t)ck));
}

// hook/union (EMSTOperators.h:1267-1303): roots read from the flattened
// labels, written into label2.  label2 is a parent forest whose chase from
// any point ends at its component root (k_round_init starts it as the
// identity; only roots are written here and the flatten only halves paths),
// so it needs no copy of the labels between rounds.
// The winner of a component (fixedMap, NodeEMST.h:947-949) is the member
// whose edge key (d2, min id, max id) equals the component's comp1 / comp2;
// the pair of ids makes it unique, so the test is made here, for p and for
// its target q, with no per-point flag between passes.
// In round 1 every component is one point, whose edge is its own: with the
// targets from k_knn_first, every point with a target wins, and a pair is
// mutual when the target's target is the point; the component minima are
// then not needed (k_comp_keep and k_round_comp2 skip that round).
// Non-mutual: root(p) -> root(q).  Mutual pair (q won its component with an
// edge back to p): the endpoint with the smaller id keeps its root.  Each
// hook absorbs exactly one root and a root is absorbed at most once over the
// run, so the edge is stored at the absorbed root's index (eu = -1 marks an
// empty slot); the edge count is reduced per block.
constexpr int kHookBlock = 1024;

__global__ __launch_bounds__(kHookBlock) void k_round_hook(int64_t n, const uint32_t* __restrict__ ids,
                                                          const int32_t* __restrict__ label,
                                                          int32_t* __restrict__ label2,
                                                          const int32_t* __restrict__ corr,
                                                          const uint64_t* __restrict__ corr_key,
                                                          const uint64_t* __restrict__ comp1,
                                                          const uint32_t* __restrict__ comp2,
                                                          Counters* C, int32_t* __restrict__ eu,
                                                          int32_t* __restrict__ ev,
                                                          float* __restrict__ ed2,
                                                          int32_t* __restrict__ eround,
                                                          const uint8_t* __restrict__ cut)
{
    if (C->done) return;
    const int round = (int)C->round;
    const bool first = knn_round1(C);
    __shared__ uint32_t cnt;
    if (threadIdx.x == 0) cnt = 0;
    __syncthreads();
    uint32_t added = 0;
    const int64_t p = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    const int32_t q = p < n ? corr[p] : -1;
    if (q >= 0) {
        const int32_t rp = first ? (int32_t)p : label[p];
        const uint64_t ck = corr_key[p];
        const uint32_t pid = ids[p], qid = (uint32_t)ck;
        const uint64_t key1 = edge_key1(ck, pid);
        if (first || (key1 == comp1[rp] && max(pid, qid) == comp2[rp] && !(cut && round > 1 && cut[rp]))) {
            const int32_t rq = first ? q : label[q];
            bool mutual = false;            // q won its component with the edge back to p
            if (corr[q] == (int32_t)p) {
                mutual = true;
                if (!first) {
                    const uint64_t cq = corr_key[q];
                    const uint32_t qq = ids[q];
                    mutual = edge_key1(cq, qq) == comp1[rq] && max(qq, (uint32_t)cq) == comp2[rq];
                }
            }
            int32_t absorbed = -1;
            if (!mutual) {
                label2[rp] = rq;
                absorbed = rp;
            } else if (pid < qid) {
                label2[rq] = rp;
                absorbed = rq;
            }
            if (absorbed >= 0) {
                ++added;
                eu[absorbed] = (int32_t)min(pid, qid);
                ev[absorbed] = (int32_t)max(pid, qid);
                ed2[absorbed] = __uint_as_float((uint32_t)(key1 >> 32));
                eround[absorbed] = round;
            }
        }
    }
    for (int off = 32; off > 0; off >>= 1) added += (uint32_t)__shfl_xor((int)added, off);
    if (__lane_id() == 0 && added) atomicAdd(&cnt, added);
    __syncthreads();
    if (threadIdx.x == 0 && cnt) atomicAdd(&C->edges, cnt);
}

// ---- per-round component search (NodeSpiralSearchMD::search,
// emst_coalition/include/NodeEMST.h:67-509; the reference's alternative to
// the round-1 cone search, SolutionEMST.h:55-56,187-194).  Every round, each
// point whose previous target has joined its component looks for its nearest
// point in another component, under (d2, id); a point whose target is still
// outside keeps it (:160-169).  The search is exact per point, so a
// component's smallest member result is its shortest outgoing edge, and the
// rounds build the same forests as the cone search.  Subtrees that lie in
// the point's own component are skipped (node component labels, rebuilt
// every round), which plays the part of the reference's permanent slab
// closures against same-component points (:293-318).

constexpr int32_t kNlabEmpty = -3;      // a node without points
constexpr int32_t kNlabMixed = -1;      // a node holding several components

// Node values of the hierarchy, bottom-up in one launch: one thread per leaf
// climbs from its leaf; at each parent the first child to arrive leaves its
// value and stops, the second combines both and goes on.  The arrival count
// and the first value share one 64-bit word per node (`visit`, updated only
// by compare-and-swap, so no fence is needed between them); every launch
// brings exactly two arrivals to every inner node, so the count's parity
// tells first from second without a reset between launches.
template <class Op, class Store>
__device__ __forceinline__ void climb(typename Op::T v, Store store, unsigned long long* __restrict__ vbase,
                                      int64_t i)
{
    while (i > 1) {
        const int64_t par = i >> 1;
        unsigned long long old = vbase[par];
        bool first;
        for (;;) {
            const uint32_t cnt = (uint32_t)(old >> 32);
            first = (cnt & 1u) == 0u;
            const typename Op::T nv = first ? v : Op::combine((typename Op::T)(uint32_t)old, v);
            const unsigned long long nw = ((unsigned long long)(cnt + 1u) << 32) | (uint32_t)nv;
            const unsigned long long got = atomicCAS(&vbase[par], old, nw);
            if (got == old) {
                v = nv;
                break;
            }
            old = got;
        }
        if (first) return;
        i = par;
        store(i, v);
    }
}

struct LabelOp {
    typedef int32_t T;
    __device__ static int32_t combine(int32_t a, int32_t b)
    {
        return a == kNlabEmpty ? b : (b == kNlabEmpty ? a : (a == b ? a : kNlabMixed));
    }
};
// component label of every node: the common label of its points.  A block
// whose kBlock leaf slots are one aligned subtree of a cloud (every block of a
// cloud with at least kBlock slots) combines the subtree's 8 lower levels in
// LDS, and only the subtree's root climbs with atomics: the climb of every
// leaf through those levels was a chain of dependent atomics per level.  The
// arrival counts of the nodes inside such a subtree are then left alone,
// which keeps their parity.
__global__ __launch_bounds__(kBlock) void k_nlab_tree(const int32_t* __restrict__ label,
                                                     const Cloud* __restrict__ cl, int ncl, int64_t nleaves,
                                                     LeafTable lt, Node* __restrict__ nodes,
                                                     unsigned long long* __restrict__ visit, const Counters* C)
{
    if (C->done || knn_round1(C)) return;       // round 1 searches nothing
    __shared__ int32_t sub_lab[kBlock];
    const int64_t g0 = (int64_t)blockIdx.x * kBlock;
    const int cb = find_cloud_leaf(cl, ncl, g0);
    const int64_t jb = g0 - cl[cb].lbase;
    const bool subtree = (jb & (kBlock - 1)) == 0 && jb + kBlock <= cl[cb].L;
    const int64_t g = g0 + threadIdx.x;
    if (!subtree && g >= nleaves) return;
    const int c = subtree ? cb : find_cloud_leaf(cl, ncl, g);
    const int64_t j = g - cl[c].lbase;
    if (!subtree && j >= cl[c].L) return;   // past the cloud's slots (one-launch capacity)
    int64_t s0, s1;
    leaf_range(lt, cl[c].lfirst, cl[c].nl, cl[c].pos + cl[c].n, j, s0, s1);
    // the leaf's common label (kNlabMixed when two differ), its loads
    // independent of each other (a serial combine waited on each load: the
    // kernel took 0.12 ms per round at 10^7 points)
    int32_t lab = kNlabEmpty;
    if (s1 > s0) {
        lab = label[s0];
        bool diff = false;
        int64_t s = s0 + 1;
        for (; s + 8 <= s1; s += 8) {
            int32_t v[8];
#pragma unroll
            for (int k = 0; k < 8; ++k) v[k] = label[s + k];
#pragma unroll
            for (int k = 0; k < 8; ++k) diff |= v[k] != lab;
        }
        for (; s < s1; ++s) diff |= label[s] != lab;
        if (diff) lab = kNlabMixed;
    }
    Node* base = nodes + 2 * cl[c].lbase;
    auto store = [&](int64_t i, int32_t v) { base[i].pad[1] = __int_as_float(v); };
    const int64_t L = cl[c].L;
    store(L + j, lab);
    if (!subtree) {
        climb<LabelOp>(lab, store, visit + 2 * cl[c].lbase, L + j);
        return;
    }
    // the subtree's levels: at level k (leaves at 0), thread t < kBlock >> k
    // holds node ((L + jb) >> k) + t
    const int t = (int)threadIdx.x;
    sub_lab[t] = lab;
    int32_t v = lab;
    for (int k = 1, w = kBlock / 2; w >= 1; ++k, w >>= 1) {
        __syncthreads();
        if (t < w) v = LabelOp::combine(sub_lab[2 * t], sub_lab[2 * t + 1]);
        __syncthreads();
        if (t < w) {
            sub_lab[t] = v;
            store(((L + jb) >> k) + t, v);
        }
    }
    if (t == 0) climb<LabelOp>(v, store, visit + 2 * cl[c].lbase, (L + jb) / kBlock);
}

// Per point, corr / corr_key between rounds:
//   corr >= 0   the exact nearest point outside the component at its last
//               search, key (d2, id); kept while it stays outside
//               (NodeEMST.h:160-169);
//   corr == -1  no exact result; the high word of corr_key is a lower bound
//               on the d2 of the nearest outside point (all ones: none);
//   corr == -2  nothing outside the component in its cloud (final).
// Keep-previous: the component minimum of the kept targets.
template <int K>
__global__ __launch_bounds__(kBlock) void k_comp_keep(int64_t n, const uint32_t* __restrict__ ids,
                                                     const int32_t* __restrict__ label,
                                                     int32_t* __restrict__ corr,
                                                     uint64_t* __restrict__ corr_key,
                                                     uint64_t* __restrict__ comp1, NbrList nb, const Counters* C)
{
    if (C->done || knn_round1(C)) return;       // every target is outside and kept
    const int64_t p = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    bool valid = false;
    int32_t lp = 0;
    uint64_t key1 = kEmptyKey;
    if (p < n) {
        lp = label[p];
        int32_t c = corr[p];
        const int j0 = nb.pos != nullptr ? (int)nb.cur[p] : K;
        bool outside = c >= 0 && label[c] != lp;
        uint64_t ck = 0;
        bool have_ck = false;
        // a target that joined the component: the next listed point outside
        // it (components only grow, so the listed points before it are inside
        // for good); the list used up, its last key bounds the search.  The
        // remaining entries, then their labels, load at once: a scan entry by
        // entry waited on two dependent loads per entry (the kernel took up to
        // 0.36 ms per round at 10^7 points, when every target has just joined).
        if (c >= 0 && !outside && j0 < K) {
            int32_t e[K], le[K];
#pragma unroll
            for (int k = 1; k < K; ++k) e[k] = k > j0 ? nb.pos[(int64_t)k * n + p] : -1;
            // (unconditional loads, an absent entry reading p's own label, so
            // that they issue together rather than one branch and wait each)
#pragma unroll
            for (int k = 1; k < K; ++k) le[k] = label[e[k] >= 0 ? e[k] : (int32_t)p];
            int j = K;
            int32_t f = -1;
#pragma unroll
            for (int k = K - 1; k >= 1; --k)
                if (k > j0 && (e[k] < 0 || le[k] != lp)) {
                    j = k;
                    f = e[k];
                }
            if (j == K) {
                c = -1;
                ck = (nb.key[(int64_t)(K - 1) * n + p] & 0xffffffff00000000ull) | 0xffffffffull;
            } else if (f < 0) {
                c = -2;             // the cloud's other points are all listed, all inside
                ck = kEmptyKey;
            } else {
                c = f;
                ck = nb.key[(int64_t)j * n + p];
                have_ck = true;
                outside = true;
            }
            nb.cur[p] = (uint8_t)j;
            corr[p] = c;
            corr_key[p] = ck;
        }
        if (outside) {
            if (!have_ck) ck = corr_key[p];
            const uint32_t pid = ids[p], qid = (uint32_t)ck;
            key1 = (ck & 0xffffffff00000000ull) | (uint64_t)min(pid, qid);
            valid = true;
        }
    }
    atomic_min_grouped(comp1, lp, key1, valid);
}

// The points that must search, flagged per 64-position packet: those without
// a kept target whose lower bound does not already exceed the component's
// kept minimum (such a point cannot hold the component's shortest edge this
// round; it keeps its bound for the next), and that do not sit at the same
// location as the position before them in the same component.  Such a point
// is dominated: equal keys sort stably, so the point before it has a smaller
// id, the same nearest outside point at the same d2, and so a key (d2, min
// id, max id) at least as small; the first of the run searches for both (the
// coincident corners of a clamped cloud are runs of 10^4-10^5 points).
__global__ __launch_bounds__(kBlock) void k_comp_prep(int64_t n, const float4* __restrict__ pts,
                                                     const int32_t* __restrict__ label,
                                                     int32_t* __restrict__ corr,
                                                     uint64_t* __restrict__ corr_key,
                                                     const uint64_t* __restrict__ comp1,
                                                     const Node* __restrict__ nodes, const Cloud* __restrict__ cl,
                                                     int ncl, uint64_t* __restrict__ open_mask, const Counters* C)
{
    if (C->done) return;
    const int64_t p = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    bool need = false;
    if (p < n && !knn_round1(C)) {          // else every point holds its nearest neighbour
        const int32_t lp = label[p];
        const int32_t c = corr[p];
        if (c == -1 || (c >= 0 && label[c] == lp)) {
            const uint32_t lb = (uint32_t)(corr_key[p] >> 32);
            const int32_t lbb = lb == 0xffffffffu ? -1 : (int32_t)lb;
            need = lbb <= key_bound(comp1[lp]);
            if (need && p > 0 && label[p - 1] == lp && same_xyz(pts[p - 1], pts[p])) need = false;
            if (!need) corr[p] = -1;    // the absorbed target's d2 stays as the bound
            // a cloud that is one component holds nothing outside it (in a
            // batch, clouds finish rounds apart: each one's points searched
            // once more through every pass, 1.45 of 2.19 ms per run of 256
            // clouds of 10^2-10^4 points went to the searches, now 0.97)
            if (need && __float_as_int(nodes[2 * cl[find_cloud(cl, ncl, p)].lbase + 1].pad[1]) == lp) {
                need = false;
                corr[p] = -2;
                corr_key[p] = kEmptyKey;
            }
        }
    }
    const uint64_t m = __ballot(need);
    if (__lane_id() == 0 && p < n) open_mask[p / 64] = m;
}

// ---- learned seed of the component search.  A component's size and box
// live at its root: single points at the start, and after every round each
// root absorbed in it adds its own to its new root (one atomic per merged
// component and box side).
__global__ __launch_bounds__(kBlock) void k_comp_seed_init(int64_t n, const float4* __restrict__ pts,
                                                          int32_t* __restrict__ csize, uint32_t* __restrict__ cbox)
{
    const int64_t p = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (p >= n) return;
    const float4 v = pts[p];
    csize[p] = 1;
    uint32_t* b = cbox + 6 * p;
    b[0] = b[3] = f2ord(v.x);
    b[1] = b[4] = f2ord(v.y);
    b[2] = b[5] = f2ord(v.z);
}

__global__ __launch_bounds__(kBlock) void k_comp_merge(int64_t n, const int32_t* __restrict__ label,
                                                      const int32_t* __restrict__ eu,
                                                      const int32_t* __restrict__ eround,
                                                      int32_t* __restrict__ csize, uint32_t* __restrict__ cbox,
                                                      const Counters* C)
{
    if (C->done) return;
    const int64_t p = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (p >= n) return;
    const int prev = (int)C->round - 1;
    if (prev < 1 || eu[p] < 0 || eround[p] != prev) return;
    const int64_t r = label[p];
    atomicAdd(&csize[r], csize[p]);
    for (int k = 0; k < 3; ++k) {
        atomicMin(&cbox[6 * r + k], cbox[6 * p + k]);
        atomicMax(&cbox[6 * r + 3 + k], cbox[6 * p + 3 + k]);
    }
}

// Features of every searching point (list order), free of the cloud's scale:
// lengths are taken relative to s0, the mean spacing of the point's leaf cell
// (LS = log s0).  The round, the component's size, the point's lower bound,
// the component's box extent and mean spacing, the component's kept minimum
// (an upper bound on its edge), and the density one and three levels up.
// The model seeds rounds from kLearnedFrom on: the first rounds' searches are
// nearest-neighbour searches of single points and tiny components, for which
// the plain seed is as good and the model's cost would not pay.
// nq_keep[0]: the count of points with features (every round when logging,
// else from kLearnedFrom on), for the sample log; nq_keep[1]: the count the
// model runs on (0 before kLearnedFrom or without a model).
constexpr uint32_t kLearnedFrom = 3;

__global__ __launch_bounds__(kBlock) void k_comp_features(int log_all, int has_model, int dim, const float4* __restrict__ pts,
                                                         const Node* __restrict__ nodes,
                                                         const Cloud* __restrict__ clouds, int ncl, LeafTable lt,
                                                         const int32_t* __restrict__ qlist,
                                                         const uint32_t* __restrict__ nq_dev,
                                                         const int32_t* __restrict__ label,
                                                         const uint64_t* __restrict__ corr_key,
                                                         const uint64_t* __restrict__ comp1,
                                                         const int32_t* __restrict__ csize,
                                                         const uint32_t* __restrict__ cbox, const Counters* C,
                                                         float* __restrict__ X, float* __restrict__ LS,
                                                         uint32_t* __restrict__ nq_keep)
{
    if (C->done) return;
    const int64_t qi = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    const bool learned_round = has_model && C->round >= kLearnedFrom;
    const uint32_t nq = (log_all || learned_round) ? *nq_dev : 0u;
    if (qi == 0) {
        nq_keep[0] = log_all ? nq : 0u;
        nq_keep[1] = learned_round ? nq : 0u;
    }
    if (qi >= (int64_t)nq) return;
    const int64_t p = qlist[qi];
    const int c = find_cloud(clouds, ncl, p);
    const int64_t L = clouds[c].L, lfirst = clouds[c].lfirst, nl = clouds[c].nl;
    const int64_t cend = clouds[c].pos + clouds[c].n;
    const Node* __restrict__ tree = nodes + 2 * clouds[c].lbase;
    int64_t node = L + (lt.of[p] - lfirst);
    float sp[4];
    for (int k = 0; k < 4; ++k) {
        const Node nd = tree[node];
        int64_t first = node, last = node;
        while (first < L) { first = 2 * first; last = 2 * last + 1; }
        int64_t a0, a1, b0, b1;
        leaf_range(lt, lfirst, nl, cend, first - L, a0, a1);
        leaf_range(lt, lfirst, nl, cend, last - L, b0, b1);
        const float cnt = (float)max<int64_t>(b1 - a0, 1);
        float vol = 1.f, ext = 0.f;
        for (int d = 0; d < dim; ++d) {
            const float e = fmaxf(nd.hi[d] - nd.lo[d], 0.f);
            vol *= e;
            ext = fmaxf(ext, e);
        }
        const float sv = vol > 0.f ? powf(vol / cnt, 1.f / dim) : ext / cnt;
        sp[k] = fmaxf(sv, 1e-6f);
        if (node > 1) node >>= 1;
    }
    const float s0 = sp[0], lo = 1e-3f * s0;
    const int32_t lab = label[p];
    const uint32_t lbh = (uint32_t)(corr_key[p] >> 32);
    const float lb = lbh == 0xffffffffu ? 0.f : sqrtf(__uint_as_float(lbh));
    const uint64_t kept = comp1[lab];
    const float kd = kept == kEmptyKey ? 1e3f * s0 : sqrtf(__uint_as_float((uint32_t)(kept >> 32)));
    const uint32_t* b = cbox + 6 * (int64_t)lab;
    float ext = 0.f, vol = 1.f;
    for (int d = 0; d < dim; ++d) {
        const float e = fmaxf(ord2f(b[3 + d]) - ord2f(b[d]), 0.f);
        ext = fmaxf(ext, e);
        vol *= e;
    }
    const float size = (float)max(csize[lab], 1);
    const float spc = vol > 0.f ? powf(vol / size, 1.f / dim) : ext / size;
    float* x = X + qi * 8;
    x[0] = logf((float)max(C->round, 1u));
    x[1] = logf(size);
    x[2] = logf(fmaxf(lb, lo) / s0);
    x[3] = logf(fmaxf(ext, lo) / s0);
    x[4] = logf(fmaxf(spc, lo) / s0);
    x[5] = logf(fmaxf(kd, lo) / s0);
    x[6] = logf(sp[1] / sp[0]);
    x[7] = logf(sp[3] / sp[0]);
    LS[qi] = logf(s0);
}

// seed radius per sorted position: s0 * exp(model output + offset)
__global__ __launch_bounds__(kBlock) void k_comp_seed(const int32_t* __restrict__ qlist,
                                                     const uint32_t* __restrict__ nq_dev,
                                                     const float* __restrict__ LS, const float* __restrict__ Y,
                                                     float* __restrict__ R, const Counters* C)
{
    if (C->done) return;
    const int64_t qi = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (qi >= (int64_t)*nq_dev) return;
    R[qlist[qi]] = expf(LS[qi] + fminf(Y[qi], 20.f));
}

// (features, target) of every stride-th searching point, stride chosen per
// round so that every round logs about `per_round` pairs (the late rounds,
// with few searching points, weigh as much as the first), logged from the
// plain method's rounds to train the model.  Target: log over s0 of the
// radius the point had to search, min(D, d): D = its component's edge length,
// d = its nearest outside point's distance when the search found it exactly
// (beyond D the component's edge stops the point).  Components without an
// outgoing edge are skipped.
__global__ __launch_bounds__(kBlock) void k_comp_samples(const int32_t* __restrict__ qlist,
                                                        const uint32_t* __restrict__ nq_dev,
                                                        const float* __restrict__ X, const float* __restrict__ LS,
                                                        const int32_t* __restrict__ label,
                                                        const int32_t* __restrict__ corr,
                                                        const uint64_t* __restrict__ corr_key,
                                                        const uint64_t* __restrict__ comp1, int64_t per_round,
                                                        int64_t cap, float* __restrict__ samples, Counters* C)
{
    if (C->done) return;
    const int64_t qi = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    const int64_t nq = *nq_dev;
    const int64_t stride = max<int64_t>(1, (nq + per_round - 1) / per_round);
    if (qi >= nq || qi % stride != 0) return;
    const int64_t p = qlist[qi];
    const uint64_t k = comp1[label[p]];
    if (k == kEmptyKey) return;
    uint32_t db = (uint32_t)(k >> 32);
    if (corr[p] >= 0) db = min(db, (uint32_t)(corr_key[p] >> 32));
    const uint32_t slot = atomicAdd(&C->nsamples, 1u);
    if ((int64_t)slot >= cap) return;
    float* o = samples + 9 * (int64_t)slot;
    for (int f = 0; f < 8; ++f) o[f] = X[qi * 8 + f];
    const float s0 = expf(LS[qi]);
    const float d = sqrtf(__uint_as_float(db));
    o[8] = logf(fmaxf(d, 1e-3f * s0)) - LS[qi];
}

// LDS lists of the leaf gatherings (k_comp_search, k_knn_first): node ids of
// the work list, and gathered leaves as (box d2 bits << 32) | leaf
constexpr int kGatherWork = 512;
constexpr int kGatherLeaves = 128;
// Packets whose gathering outgrows the LDS lists hand their open queries to
// the per-query pass (k_comp_search_deferred) rather than walk the tree with
// all of them: in 3D up to kDeferCap queries a round (a walk over the union
// of 64 neighbourhoods is the tail of the large dispatches, and the per-query
// pass takes about as long for 64k queries as one such walk), in 2D only in
// dispatches of at most kDeferQueries queries (1024 packets, one per SIMD of
// the chip; in the large 2D dispatches the walks cost less than the pass)
constexpr int64_t kDeferQueries = 65536;
constexpr uint32_t kDeferCap = 65536;
// the resumed dispatch of the component search runs on at most this many
// one-packet blocks, looping over its packets: its queries are few (most
// close in the first pass), and a grid of one block per packet of the whole
// query list cost 34 us per round at 10^7 points while idle
constexpr int64_t kResumeBlocks = 4096;
// the first dispatch: at most this many blocks (far more than the chip holds,
// so the hardware still balances the packets); the compaction clears the
// mask, so a block need only write the words of the packets it searched
constexpr int64_t kSearchBlocks = 65536;
// Before the first dispatch, a sample of the queries is searched through every
// pass, for the components that have no edge yet: what it finds bounds all
// their other points, which then end in one pass instead of a capped one that
// sees nothing, a compaction and a second dispatch.  512 clouds of eight
// Gaussians (rounds of isolated clusters of some 2000 points): 6.6 -> 2.8 ms
// of searches a run, 19.5 -> 15.3 in all; 64 clusters of 2000: 2.37 -> 2.31.
// kSampleLanes queries of every kSampleStep-th packet: few to a wave, since
// the first finds are slow ones (lanes x step, ms a run: 64 x 16 18.0, 16 x 16
// 16.5, 8 x 16 15.6, 4 x 16 15.5, 4 x 8 15.2), where components have
// kSampleComp points to search on average (in smaller ones the rest has
// little to gain).  In 3D: 2D searches end soon without (10^7 power-law points
// 15.4 ms, with 15.6).
constexpr int kSampleLanes = 4;
constexpr int kSampleStep = 8;
constexpr uint64_t kSampleComp = 512;
constexpr int64_t kSampleBlocks = 4096;
constexpr int64_t kSampleMin = 1 << 16;
// Queries per packet.  A dispatch of few queries (rounds where the searching
// points are scattered) has fewer 64-query packets than the chip holds waves,
// and each packet walks the union of its queries' neighbourhoods: it takes
// kSmallPacket queries per packet instead, so that more, narrower packets run
// at once.
constexpr int64_t kSmallDispatch = 786432;
constexpr int kSmallPacket = 8;
// the neighbour lists' gatherings (k_knn_first): their radius is the packet's
// largest K-th distance after its own leaves, so they reach further
constexpr int kKnnGatherWork = 1024;
constexpr int kKnnGatherLeaves = 256;
// Packets of the neighbour lists, at least: few points take fewer queries to a
// packet, 8 at least.  2048 packets of 64 (131071 points of eight Gaussians)
// are two waves a SIMD, and the launch takes as long as its longest packet; of
// 32 queries each reads fewer leaves.  Runs, ms, 64 to a packet / at least
// 2000, 4000, 8000, 16000 packets: those points 1.751 / 1.751, 1.676, 1.655,
// 1.690; 131071 uniform ones 1.288 / 1.295, 1.273, 1.295, 1.322; 30000 of eight
// Gaussians 1.491 / 1.420, 1.412, 1.417, 1.417; 400000 of 64 1.948 / 1.963,
// 1.950, 1.992, 2.026; 131071 in the plane 1.203 / 1.206, 1.200, 1.213, 1.238.
constexpr int64_t kKnnPackets = 4000;

// d2 (bits) to which a component's edge lets its points search.  Late points go
// some 0.01% further: where distances tie but for rounding (voxels), those just
// beyond the edge are then found, and held for the next rounds, instead of
// searched in each (the blocks at k_late_mark: 332000 points searched and 2.62
// ms a run without).
constexpr int32_t kLateSlack = 1 << 10;

template <bool LATE>
__device__ __forceinline__ int32_t edge_limit(uint64_t k)
{
    const int32_t b = key_bound(k);
    return LATE && b < 0x7f000000 ? b + kLateSlack : b;
}

// nearest point in another component, for the points of qlist (count in
// nq_dev): packet traversal as in the cone search, one best per query, by
// iterative deepening from the seed radius R_0 (capped passes R_k = 8^(k/2) R_0,
// then one uncapped).  Points below the point's lower bound (its previous
// target's d2) were in the component at that search and still are, so they
// are skipped.  The component's shortest edge found so far (comp1, read at
// each pass) also bounds the search: a point whose nearest outside point lies
// beyond it cannot hold the component's edge, and it stops with that d2 as
// its lower bound (corr = -1).  Exact results enter comp1 as they close.
//
// LATE: the queries are late points of the cone form (launch_late_search).
// Their first lower bound is that of their unknown candidates (late_least):
// points outside their component do lie within it, hidden from their cones.
template <int D, int BK, bool SAMPLE, bool LATE>
__global__ __launch_bounds__(64) __attribute__((amdgpu_waves_per_eu(6))) void k_comp_search(
    const float4* __restrict__ pts, const Node* __restrict__ nodes,
    const Cloud* __restrict__ clouds, int ncl, int bucket_rt, LeafTable lt, const int32_t* __restrict__ qlist,
    const uint32_t* __restrict__ nq_dev, const int32_t* __restrict__ label, const int32_t* __restrict__ inv,
    float seed_scale, int32_t* __restrict__ corr, uint64_t* __restrict__ corr_key,
    uint64_t* __restrict__ comp1, int pass_lo, int pass_hi,
    uint64_t* __restrict__ open_out, const float* __restrict__ seed_r, uint64_t* __restrict__ defer, Counters* C,
    int collect)
{
    // the leaf size: a compile-time constant for the default sizes
    const int bucket = BK ? BK : bucket_rt;
    if (C->done) return;
    const int64_t nq = *nq_dev;
    if (SAMPLE) {
        // (small components: a sampled point has hardly more to bound)
        if ((uint64_t)(C->target - C->edges) * kSampleComp > (uint64_t)nq) return;
    } else if (blockIdx.x == 0 && threadIdx.x == 0) {
        atomicAdd(&C->comp_queries, (unsigned long long)nq);
    }
    __shared__ unsigned long long best[64];
    __shared__ int32_t stk_id[64];
    __shared__ int32_t stk_ver[64];
    __shared__ unsigned long long stk_mask[64];
    __shared__ int32_t work[kGatherWork];
    __shared__ unsigned long long gathered[kGatherLeaves];
    // one packet per block; a grid smaller than the packets (the resumed
    // dispatch, whose queries are few but unknown to the host) loops
    const int qpp = nq <= kSmallDispatch ? kSmallPacket : 64;
    // The resumed dispatch (no open_out) gives every block a run of
    // consecutive packets, so that the packets in flight are spread over all
    // components: the first ones find their components' edges, which bound the
    // packets after them (7.2*10^6 points in 512 clouds of eight Gaussians:
    // 17.9 -> 15.9 ms per run).  The first dispatch keeps one packet per block
    // in list order: runs there left the chip with a tail (10^7 clustered
    // points 13.4 -> 14.5 ms), and parts spread out by a stride lost their
    // neighbours' cache lines (13.8 ms).
    const int64_t npk = (nq + qpp - 1) / qpp;
    const bool runs = open_out == nullptr && !SAMPLE;
    const int64_t run = SAMPLE ? kSampleStep : runs ? (npk + gridDim.x - 1) / gridDim.x : 1;
    const int64_t pk0 = (int64_t)blockIdx.x * run, pk1 = runs ? min(npk, pk0 + run) : npk;
    for (int64_t pk = pk0;; pk += runs ? 1 : (int64_t)gridDim.x * (SAMPLE ? kSampleStep : 1)) {
        if (pk >= pk1) {
            if (open_out != nullptr && threadIdx.x == 0 && pk == pk0) open_out[pk] = 0ull;
            break;
        }
        const int lane = __lane_id();
        const int64_t qi = pk * qpp + lane;
        bool active = lane < (SAMPLE ? kSampleLanes : qpp) && qi < nq;
        const int64_t p = active ? (int64_t)qlist[qi] : 0;
        const float4 me = pts[p];
        const float px = me.x, py = me.y, pz = me.z;
        const int32_t mylab = active ? label[p] : -1;
        if (SAMPLE) {
            active = active && comp1[mylab] == kEmptyKey;
            if (__ballot(active) == 0ull) continue;
        }
        const uint64_t prev = active ? corr_key[p] : kEmptyKey;
        best[lane] = kEmptyKey;
        const int my_cl = active ? find_cloud(clouds, ncl, p) : -1;
        const uint32_t pid = __float_as_uint(me.w);
        bool bounded = false, left_open = false, deferred = false;
        int32_t lbnd = 0;
        uint32_t st_nodes = 0, st_leaves = 0, st_walks = 0;   // work counters of this packet
        uint64_t st_pairs = 0;
        uint64_t pending = __ballot(active);
        while (pending) {
            const int cl = __builtin_amdgcn_readfirstlane(__shfl(my_cl, (int)__builtin_ctzll(pending)));
            const bool mine = my_cl == cl;
            pending &= ~__ballot(mine);
            const int64_t cend = clouds[cl].pos + clouds[cl].n;
            const int64_t L = clouds[cl].L, lfirst = clouds[cl].lfirst, nl = clouds[cl].nl;
            const Node* __restrict__ tree = nodes + 2 * clouds[cl].lbase;
            // seed: twice the previous target's distance, at least seed_scale
            // times the mean spacing of the point's leaf cell
            float r = 1.f;
            int32_t inner = -1;
            if (mine) {
                const int64_t lf = lt.of[p];
                const Node own = tree[L + (lf - lfirst)];
                const float cnt = (float)(lt.start[lf + 1] - lt.start[lf]);
                float vol = 1.f, ext = 0.f;
                for (int k = 0; k < D; ++k) {
                    const float e = own.hi[k] - own.lo[k];
                    vol *= e;
                    ext = fmaxf(ext, e);
                }
                float sp = vol > 0.f ? powf(vol / cnt, 1.f / D) : ext / cnt;
                if (!positive_finite(sp)) sp = 1e-6f;
                const bool has_lb = (uint32_t)(prev >> 32) != 0xffffffffu;
                const uint32_t dbits = (uint32_t)(prev >> 32);
                if (has_lb) inner = (int32_t)dbits - 1;
                r = seed_scale * sp;
                if (has_lb) r = fmaxf(r, 2.f * sqrtf(__uint_as_float(dbits)));
                // learned: the predicted length of the component's edge, so
                // that the first pass can already find it
                if (seed_r != nullptr && C->round >= kLearnedFrom) {
                    r = seed_r[p];
                    if (has_lb) r = fmaxf(r, sqrtf(__uint_as_float(dbits)));
                }
                if (!positive_finite(r)) r = 1e-6f;
            }
            const int32_t from = inner;
            float r2 = r * r;
            // a launch that resumes at pass_lo: the state the earlier passes left
            for (int k = 0; k < pass_lo; ++k) {
                inner = max(inner, (int32_t)__float_as_uint(r2));
                r2 *= 8.f;
            }
            bool open = mine;
            float cx = mine ? px : 0.f, cy = mine ? py : 0.f, cz = mine ? pz : 0.f;
            float na = mine ? 1.f : 0.f;
            for (int off = 32; off > 0; off >>= 1) {
                cx += __shfl_xor(cx, off);
                cy += __shfl_xor(cy, off);
                cz += __shfl_xor(cz, off);
                na += __shfl_xor(na, off);
            }
            cx /= na; cy /= na; cz /= na;
            auto cdist = [&](const Node& x) {
                const float dxx = fmaxf(fmaxf(x.lo[0] - cx, cx - x.hi[0]), 0.f);
                const float dyy = fmaxf(fmaxf(x.lo[1] - cy, cy - x.hi[1]), 0.f);
                const float dzz = fmaxf(fmaxf(x.lo[2] - cz, cz - x.hi[2]), 0.f);
                return dxx * dxx + dyy * dyy + dzz * dzz;
            };
            // a box is needed when it holds another component, its nearest point
            // is within the limit and may beat the best so far under (d2, id)
            // (at equal d2 only with a smaller id), and its farthest point lies
            // beyond `inner`
            auto needed = [&](const Node& nd, int32_t nl, uint32_t nm, int32_t lim, uint64_t bk) {
                if (!open || nl == mylab || nl == kNlabEmpty) return false;
                float m[3], u[3];
                const float lo[3] = {nd.lo[0] - px, nd.lo[1] - py, nd.lo[2] - pz};
                const float hi[3] = {nd.hi[0] - px, nd.hi[1] - py, nd.hi[2] - pz};
    #pragma unroll
                for (int k = 0; k < 3; ++k) {
                    m[k] = fmaxf(fmaxf(lo[k], -hi[k]), 0.f);
                    u[k] = fmaxf(-lo[k], hi[k]);
                }
                const float lb = D == 3 ? d2_of(m[0], m[1], m[2]) : d2_of(m[0], m[1]);
                const float far = D == 3 ? d2_of(u[0], u[1], u[2]) : d2_of(u[0], u[1]);
                const uint32_t lbb = __float_as_uint(lb);
                return (int32_t)lbb <= lim && (((uint64_t)lbb << 32) | nm) < bk &&
                       (int32_t)__float_as_uint(far) > inner;
            };
            for (int pass = pass_lo; pass <= pass_hi; ++pass) {
                const bool last = pass == kMaxCappedPasses;
                const int32_t cbb = open ? edge_limit<LATE>(comp1[mylab]) : 0x7fffffff;
                // a point whose component already has an edge (a kept target, or
                // a member's result) searches straight out to it in one pass
                // instead of deepening by 4x per pass
                const int32_t cap = last || cbb != 0x7fffffff ? 0x7fffffff : (int32_t)__float_as_uint(r2);
                // nothing outside the component lies within `inner`: with the
                // component's edge at most that long, the point cannot hold it
                if (open && cbb <= inner) {
                    open = false;
                    bounded = true;
                    lbnd = inner;
                }
                if (__ballot(open) == 0ull) break;
                const int32_t lim = min(cap, cbb);
                uint64_t bk = best[lane];
                int32_t bnd = min(key_bound(bk), lim);
                int sp = 0;
                int ver = 0;
                // first pass (3D): the leaf of the first open lane goes first, so
                // that the packet's lanes enter the tree with bounds from their
                // own neighbourhood; the traversal skips it when it comes again
                // (clustered 3D -3.4%; in 2D +1%, so not there)
                int pre = -1;
                bool pre_done = false;
                if (D == 3 && pass == 0) {
                    const int fl = (int)__builtin_ctzll(__ballot(open));
                    const int myleaf = (int)(L + (mine ? lt.of[p] - lfirst : 0));
                    pre = __builtin_amdgcn_readfirstlane(__shfl(myleaf, fl));
                }
                // a leaf: one (query, leaf point) pair per lane; the query's state by
                // LDS permute (a v_readlane broadcast when 64 / bucket = 1, as in
                // the cone search, measured 7% slower here, and four packets per
                // block 6% slower)
                auto visit_leaf = [&](int node, bool need, uint64_t needm) {
                    int64_t s0, s1;
                    leaf_range(lt, lfirst, nl, cend, node - L, s0, s1);
                    const int cnt = (int)(s1 - s0);
                    ++st_leaves;
                    st_pairs += (uint64_t)cnt * (uint64_t)__popcll(needm);
                    const int j = lane & (bucket - 1);
                    const int qslot = lane / bucket;
                    const int qpc = 64 / bucket;
                    float4 v = make_float4(0.f, 0.f, 0.f, 0.f);
                    int32_t vlab = -1;
                    if (j < cnt) {
                        v = pts[s0 + j];
                        vlab = label[s0 + j];
                    }
                    uint64_t rem = needm;
                    while (rem) {
                        int myq = -1;
                        for (int k = 0; k < qpc; ++k) {
                            const int l = rem ? (int)__builtin_ctzll(rem) : -1;
                            if (rem) rem &= rem - 1;
                            if (k == qslot) myq = l;
                        }
                        const int src = myq >= 0 ? myq : 0;
                        const float qx = __shfl(px, src), qy = __shfl(py, src), qz = __shfl(pz, src);
                        const int32_t qb = __shfl(bnd, src), qin = __shfl(inner, src), ql = __shfl(mylab, src);
                        const float dx = v.x - qx, dy = v.y - qy, dz = v.z - qz;
                        const float d2 = D == 3 ? d2_of(dx, dy, dz) : d2_of(dx, dy);
                        const int32_t db = (int32_t)__float_as_uint(d2);
                        if (myq >= 0 && j < cnt && vlab != ql && db <= qb && db > qin)
                            atomicMin(&best[myq],
                                      ((unsigned long long)__float_as_uint(d2) << 32) | __float_as_uint(v.w));
                    }
                    if (need) {
                        bk = best[lane];
                        bnd = min(key_bound(bk), lim);
                    }
                };
                // The gathering (a finite bound): every leaf whose box lies within
                // the largest bound of the open queries from their box, of another
                // component than all of them, and not inside all of their lower
                // bounds, by box-to-box tests of 64 nodes a step; then those
                // leaves nearest first, each tested per query.  A gathering that
                // outgrows the LDS lists leaves the pass to the per-query walk.
                bool done_by_gather = false;
                uint32_t B = open ? (uint32_t)bnd : 0u;
                for (int off = 32; off > 0; off >>= 1) B = max(B, (uint32_t)__shfl_xor((int)B, off));
                {
                    float qlo[3] = {open ? px : INFINITY, open ? py : INFINITY, open ? pz : INFINITY};
                    float qhi[3] = {open ? px : -INFINITY, open ? py : -INFINITY, open ? pz : -INFINITY};
                    int32_t imin = open ? inner : 0x7fffffff;
                    int32_t fmost = open ? from : -1;
                    for (int off = 32; off > 0; off >>= 1) {
    #pragma unroll
                        for (int k = 0; k < 3; ++k) {
                            qlo[k] = fminf(qlo[k], __shfl_xor(qlo[k], off));
                            qhi[k] = fmaxf(qhi[k], __shfl_xor(qhi[k], off));
                        }
                        imin = min(imin, __shfl_xor(imin, off));
                        if (LATE) fmost = max(fmost, __shfl_xor(fmost, off));
                    }
                    const int fo = (int)__builtin_ctzll(__ballot(open));
                    const int32_t lab0 = __builtin_amdgcn_readfirstlane(__shfl(mylab, fo));
                    const bool one_lab = __ballot(open && mylab != lab0) == 0ull;
                    const int32_t skip_lab = one_lab ? lab0 : (int32_t)0x80000000;
                    int head = 0, tail = gather_start(L, work), ngl = 0;
                    bool over = false;
                    __builtin_amdgcn_wave_barrier();
                    while (head < tail) {
                        const int take = min(64, tail - head);
                        const int nd = lane < take ? work[head + lane] : 0;
                        head += take;
                        st_nodes += (uint32_t)take;
                        bool pass_ = false, leaf = false;
                        uint32_t bd = 0, ub = 0xffffffffu;
                        if (lane < take) {
                            const Node x = tree[nd];
                            const int32_t xl = __float_as_int(x.pad[1]);
                            float m[3], u[3];
    #pragma unroll
                            for (int k = 0; k < 3; ++k) {
                                m[k] = fmaxf(fmaxf(x.lo[k] - qhi[k], qlo[k] - x.hi[k]), 0.f);
                                u[k] = fmaxf(x.hi[k] - qlo[k], qhi[k] - x.lo[k]);
                            }
                            bd = __float_as_uint(D == 3 ? d2_of(m[0], m[1], m[2]) : d2_of(m[0], m[1]));
                            const float far = D == 3 ? d2_of(u[0], u[1], u[2]) : d2_of(u[0], u[1]);
                            leaf = nd >= L;
                            pass_ = xl != kNlabEmpty && xl != skip_lab && bd <= B &&
                                    (int32_t)__float_as_uint(far) > imin && !(leaf && nd == pre);
                            // it holds a point outside every query's component
                            // (it holds two components, or the queries lie in
                            // one, which is another): none needs more than
                            // its far corner, which then bounds the gathering.
                            // Without it a pass whose radius first reaches a far
                            // cluster gathered most of that cluster, outgrew its
                            // lists and walked (512 clouds of eight Gaussians:
                            // 153000 -> 34000 walks per run).  (Late points:
                            // a node beyond all of their first bounds, so that
                            // its points are not hidden ones)
                            if (pass_ && (xl == kNlabMixed || one_lab) && (!LATE || (int32_t)bd > fmost))
                                ub = __float_as_uint(far);
                        }
                        B = min(B, wave_min_u32(ub));
                        pass_ = pass_ && bd <= B;
                        const uint64_t ml = __ballot(pass_ && leaf);
                        const int nlf = __popcll(ml);
                        int add;
                        if (!push_inner(pass_ && !leaf, nd, L, work, tail, kGatherWork, add) ||
                            ngl + nlf > kGatherLeaves) {
                            over = true;
                            break;
                        }
                        if (pass_ && leaf)
                            gathered[ngl + __popcll(ml & lanemask_lt())] = ((uint64_t)bd << 32) | (uint32_t)nd;
                        tail += add;
                        ngl += nlf;
                        __builtin_amdgcn_wave_barrier();
                    }
                    if (!over) {
                        done_by_gather = true;
                        auto try_leaf = [&](int node) {
                            const Node x = tree[node];
                            ++st_nodes;
                            const bool need = needed(x, __float_as_int(x.pad[1]), __float_as_uint(x.pad[0]), lim, bk);
                            const uint64_t needm = __ballot(need);
                            if (needm != 0ull) visit_leaf(node, need, needm);
                        };
                        if (pre >= 0) try_leaf(pre);
                        for (int c0 = 0; c0 < ngl; c0 += 64) {
                            const int cn = min(64, ngl - c0);
                            const uint64_t e = wave_sort_u64(lane < cn ? gathered[c0 + lane] : kEmptyKey);
                            for (int i = 0; i < cn; ++i) {
                                // (gathered before B shrank to less than its distance)
                                if ((uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)(e >> 32), i) > B) break;
                                try_leaf(__builtin_amdgcn_readlane((int)(uint32_t)e, i));
                            }
                        }
                    }
                }
                // a gathering that outgrew its lists: the dispatch takes as long
                // as its slowest packet, and this packet's walk would visit the
                // union of its queries' neighbourhoods in one wave; the open
                // queries go to the per-query pass instead, one wave each, from
                // this pass on (no leaf has been visited in it yet, so their
                // bests are empty), while the round's list has room
                bool handed = false;        // this lane's query went to the per-query pass
                if (!done_by_gather && defer != nullptr) {
                    const uint64_t entry = ((uint64_t)(uint32_t)pass << 32) | (uint32_t)p;
                    if (D == 3) {
                        handed = wave_append_capped_u64(open, entry, defer, &C->deferred, kDeferCap);
                    } else if (nq <= kDeferQueries) {
                        wave_append_u64(open, entry, defer, &C->deferred);
                        handed = open;
                    }
                    if (handed) {
                        open = false;
                        deferred = true;
                    }
                }
                if (SAMPLE && !done_by_gather) break;
                const bool walk = !done_by_gather && __ballot(open) != 0ull;
                if (!done_by_gather && !walk) {
                    ++st_walks;
                } else if (walk) {
                    ++st_walks;
                    if (lane == 0) {
                        stk_id[0] = 1;
                        stk_ver[0] = -1;
                        if (pre >= 0) { stk_id[1] = pre; stk_ver[1] = -1; }
                    }
                    sp = pre >= 0 ? 2 : 1;
                    __builtin_amdgcn_wave_barrier();
                    while (sp > 0) {
                        --sp;
                        const int node = __builtin_amdgcn_readfirstlane(stk_id[sp]);
                        const int pver = __builtin_amdgcn_readfirstlane(stk_ver[sp]);
                        if (node == pre) {
                            if (pre_done) continue;
                            pre_done = true;
                        }
                        bool need;
                        if (pver == ver) {
                            need = (stk_mask[sp] >> lane) & 1ull;
                        } else {
                            {
                                const Node nd = tree[node];
                                need = needed(nd, __float_as_int(nd.pad[1]), __float_as_uint(nd.pad[0]), lim, bk);
                            }
                            ++st_nodes;
                        }
                        const uint64_t needm = __ballot(need);
                        if (needm == 0ull) continue;
                        if (node >= L) {
                            visit_leaf(node, need, needm);
                            ++ver;
                        } else {
                            // (rare: an unbounded pass, or a gathering that
                            // outgrew its lists) both children, the nearer last
                            // on the stack
                            const int first = 2 * node;
                            st_nodes += 2u;
                            const Node b0 = tree[first], b1 = tree[first + 1];
                            const uint64_t m0 =
                                __ballot(needed(b0, __float_as_int(b0.pad[1]), __float_as_uint(b0.pad[0]), lim, bk));
                            const uint64_t m1 =
                                __ballot(needed(b1, __float_as_int(b1.pad[1]), __float_as_uint(b1.pad[0]), lim, bk));
                            const float d0 = m0 ? cdist(b0) : -1.f, d1 = m1 ? cdist(b1) : -1.f;
                            // pushed farthest first, so the nearest pops first; at
                            // equal distance the lower node (smaller ids in a run
                            // of coincident points) pops first
                            const bool swap = d1 > d0;
                            const int ia = swap ? first + 1 : first, ib = swap ? first : first + 1;
                            const uint64_t ma = swap ? m1 : m0, mb = swap ? m0 : m1;
                            if (lane == 0) {
                                int t = sp;
                                if (ma) { stk_id[t] = ia; stk_ver[t] = ver; stk_mask[t] = ma; ++t; }
                                if (mb) { stk_id[t] = ib; stk_ver[t] = ver; stk_mask[t] = mb; ++t; }
                            }
                            sp += (ma != 0ull ? 1 : 0) + (mb != 0ull ? 1 : 0);
                            __builtin_amdgcn_wave_barrier();
                        }
                    }
                }
                // everything outside the component up to min(best, lim) has been
                // seen: best is exact when within lim; else nothing lies within
                // lim, and with lim = cbb the point stops on its lower bound
                bool fresh = false;
                uint64_t key1 = kEmptyKey;
                if (open) {
                    const uint64_t kb = best[lane];
                    if (key_bound(kb) <= lim) {
                        open = false;
                        if (kb != kEmptyKey) {
                            fresh = true;
                            key1 = (kb & 0xffffffff00000000ull) | (uint64_t)min(pid, (uint32_t)kb);
                        }
                    } else if (cbb <= cap) {
                        open = false;
                        bounded = true;
                        lbnd = cbb;
                    }
                }
                atomic_min_leader(comp1, mylab, key1, fresh);
                inner = max(inner, cap);
                r2 *= 8.f;
            }
            if (mine) left_open = open;
        }
        if (SAMPLE) continue;           // only comp1 is kept
        if (open_out != nullptr) {
            const uint64_t m = __ballot(left_open);
            if (qpp == 64) {
                if (lane == 0) open_out[pk] = m;
            } else if (lane == 0 && m != 0ull) {
                // several packets share a mask word (the compaction cleared it)
                atomicOr((unsigned long long*)&open_out[(pk * qpp) >> 6], (unsigned long long)(m << ((pk * qpp) & 63)));
            }
        }
        if (collect && lane == 0) {
            const int slot = (int)(pk % kWorkSlots);
            atomicAdd(&C->work[kWorkCompNodes][slot], (unsigned long long)st_nodes);
            atomicAdd(&C->work[kWorkCompLeaves][slot], (unsigned long long)st_leaves);
            atomicAdd(&C->work[kWorkCompPairs][slot], (unsigned long long)st_pairs);
            atomicAdd(&C->work[kWorkCompWalks][slot], (unsigned long long)st_walks);
        }
        if (active && !left_open && !deferred) {
            const uint64_t k = best[lane];
            if (bounded) {
                corr[p] = -1;
                corr_key[p] = ((uint64_t)(uint32_t)lbnd << 32) | 0xffffffffull;
            } else {
                corr[p] = k == kEmptyKey ? -2 : inv[(uint32_t)k];
                corr_key[p] = k;
            }
        }
    }
}

// The per-query pass of the component search: the queries a packet handed
// over (defer: position | pass << 32, count in C->deferred), one wave per
// query, from the pass it reached to the last.  The same search as
// k_comp_search's, for one query: the wave gathers the candidate leaves
// around the query point by box tests of 64 nodes a step, then visits them
// nearest first with one leaf point per lane and a wave minimum of the keys;
// a gathering that outgrows its lists walks the tree, nearest child first.
constexpr int kDeferWaves = 4;          // waves per block
constexpr int kDeferBlocks = 2048;      // a grid that fills the chip once; waves loop over the queries


__device__ __forceinline__ uint64_t wave_min_u64(uint64_t v)
{
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) {
        const uint64_t o = shfl_xor_u64(v, off);
        v = o < v ? o : v;
    }
    return v;
}

template <int D, bool LATE>
__global__ __launch_bounds__(64 * kDeferWaves) void k_comp_search_deferred(
    const float4* __restrict__ pts, const Node* __restrict__ nodes, const Cloud* __restrict__ clouds, int ncl,
    LeafTable lt, const uint64_t* __restrict__ defer, const int32_t* __restrict__ label,
    const int32_t* __restrict__ inv, float seed_scale, int32_t* __restrict__ corr,
    uint64_t* __restrict__ corr_key, uint64_t* __restrict__ comp1, const float* __restrict__ seed_r, Counters* C,
    int collect)
{
    if (C->done) return;
    // (in 3D the count may pass the list's cap: the lanes past it walked)
    const uint32_t cnt = D == 3 ? min(C->deferred, kDeferCap) : C->deferred;
    __shared__ int32_t work_w[kDeferWaves][kGatherWork];
    __shared__ unsigned long long gathered_w[kDeferWaves][kGatherLeaves];
    __shared__ int32_t stk_w[kDeferWaves][64];
    const int w = (int)threadIdx.x / 64;
    const int lane = __lane_id();
    int32_t* work = work_w[w];
    unsigned long long* gathered = gathered_w[w];
    int32_t* stk = stk_w[w];
    uint32_t st_nodes = 0, st_leaves = 0;
    uint64_t st_pairs = 0;
    for (uint32_t qi = blockIdx.x * kDeferWaves + w; qi < cnt; qi += gridDim.x * kDeferWaves) {
        const uint64_t e = defer[qi];
        const int64_t p = (int64_t)(uint32_t)e;
        const int pass0 = (int)(e >> 32);
        const float4 me = pts[p];
        const float px = me.x, py = me.y, pz = me.z;
        const uint32_t pid = __float_as_uint(me.w);
        const int32_t mylab = label[p];
        const uint64_t prev = corr_key[p];
        const int c = find_cloud(clouds, ncl, p);
        const int64_t cend = clouds[c].pos + clouds[c].n;
        const int64_t L = clouds[c].L, lfirst = clouds[c].lfirst, nl = clouds[c].nl;
        const Node* __restrict__ tree = nodes + 2 * clouds[c].lbase;
        // the seed and the state the earlier passes left, as in k_comp_search
        int32_t inner = -1;
        float r;
        {
            const int64_t lf = lt.of[p];
            const Node own = tree[L + (lf - lfirst)];
            const float cntl = (float)(lt.start[lf + 1] - lt.start[lf]);
            float vol = 1.f, ext = 0.f;
            for (int k = 0; k < D; ++k) {
                const float ee = own.hi[k] - own.lo[k];
                vol *= ee;
                ext = fmaxf(ext, ee);
            }
            float sp = vol > 0.f ? powf(vol / cntl, 1.f / D) : ext / cntl;
            if (!positive_finite(sp)) sp = 1e-6f;
            const bool has_lb = (uint32_t)(prev >> 32) != 0xffffffffu;
            const uint32_t dbits = (uint32_t)(prev >> 32);
            if (has_lb) inner = (int32_t)dbits - 1;
            r = seed_scale * sp;
            if (has_lb) r = fmaxf(r, 2.f * sqrtf(__uint_as_float(dbits)));
            if (seed_r != nullptr && C->round >= kLearnedFrom) {
                r = seed_r[p];
                if (has_lb) r = fmaxf(r, sqrtf(__uint_as_float(dbits)));
            }
            if (!positive_finite(r)) r = 1e-6f;
        }
        const int32_t from = inner;
        float r2 = r * r;
        for (int k = 0; k < pass0; ++k) {
            inner = max(inner, (int32_t)__float_as_uint(r2));
            r2 *= 8.f;
        }
        bool open = true, bounded = false;
        int32_t lbnd = 0;
        uint64_t bk = kEmptyKey;
        auto box_d2 = [&](const Node& x, float& far) {
            float m[3], u[3];
            const float lo[3] = {x.lo[0] - px, x.lo[1] - py, x.lo[2] - pz};
            const float hi[3] = {x.hi[0] - px, x.hi[1] - py, x.hi[2] - pz};
#pragma unroll
            for (int k = 0; k < 3; ++k) {
                m[k] = fmaxf(fmaxf(lo[k], -hi[k]), 0.f);
                u[k] = fmaxf(-lo[k], hi[k]);
            }
            far = D == 3 ? d2_of(u[0], u[1], u[2]) : d2_of(u[0], u[1]);
            return D == 3 ? d2_of(m[0], m[1], m[2]) : d2_of(m[0], m[1]);
        };
        for (int pass = pass0; pass <= kMaxCappedPasses && open; ++pass) {
            const bool last = pass == kMaxCappedPasses;
            // (other waves lower comp1[mylab] meanwhile, and the lanes of one
            // load can see different values: one lane's steers the wave)
            const int32_t cbb = edge_limit<LATE>(wave_first_u64(comp1[mylab]));
            const int32_t cap = last || cbb != 0x7fffffff ? 0x7fffffff : (int32_t)__float_as_uint(r2);
            if (cbb <= inner) {
                open = false;
                bounded = true;
                lbnd = inner;
                break;
            }
            const int32_t lim = min(cap, cbb);
            int32_t bnd = min(key_bound(bk), lim);
            // a node is needed when it holds another component, its nearest
            // point is within the limit and may beat the best so far under
            // (d2, id), and its farthest point lies beyond `inner`
            auto needed = [&](const Node& x) {
                const int32_t xl = __float_as_int(x.pad[1]);
                if (xl == mylab || xl == kNlabEmpty) return false;
                float far;
                const uint32_t lbb = __float_as_uint(box_d2(x, far));
                return (int32_t)lbb <= lim && (((uint64_t)lbb << 32) | __float_as_uint(x.pad[0])) < bk &&
                       (int32_t)__float_as_uint(far) > inner;
            };
            // one leaf point per lane, the wave's minimum key
            auto visit_leaf = [&](int node) {
                int64_t s0, s1;
                leaf_range(lt, lfirst, nl, cend, node - L, s0, s1);
                const int cn = (int)(s1 - s0);
                ++st_leaves;
                st_pairs += (uint64_t)cn;
                uint64_t key = kEmptyKey;
                if (lane < cn) {
                    const float4 v = pts[s0 + lane];
                    const float dx = v.x - px, dy = v.y - py, dz = v.z - pz;
                    const float d2 = D == 3 ? d2_of(dx, dy, dz) : d2_of(dx, dy);
                    const int32_t db = (int32_t)__float_as_uint(d2);
                    if (label[s0 + lane] != mylab && db <= bnd && db > inner)
                        key = ((uint64_t)__float_as_uint(d2) << 32) | __float_as_uint(v.w);
                }
                const uint64_t km = wave_min_u64(key);
                if (km < bk) {
                    bk = km;
                    bnd = min(key_bound(bk), lim);
                }
            };
            bool done_by_gather = false;
            {
                uint32_t B = (uint32_t)bnd;
                int head = 0, tail = gather_start(L, work), ngl = 0;
                bool over = false;
                while (head < tail) {
                    const int take = min(64, tail - head);
                    const int nd = lane < take ? work[head + lane] : 0;
                    head += take;
                    st_nodes += (uint32_t)take;
                    bool pass_ = false, leaf = false;
                    uint32_t bd = 0, ub = 0xffffffffu;
                    if (lane < take) {
                        const Node x = tree[nd];
                        const int32_t xl = __float_as_int(x.pad[1]);
                        float far;
                        bd = __float_as_uint(box_d2(x, far));
                        leaf = nd >= L;
                        pass_ = xl != kNlabEmpty && xl != mylab && bd <= B && (int32_t)__float_as_uint(far) > inner;
                        // it holds a point outside (late points: none of the hidden ones)
                        if (pass_ && (!LATE || (int32_t)bd > from)) ub = __float_as_uint(far);
                    }
                    B = min(B, wave_min_u32(ub));
                    pass_ = pass_ && bd <= B;
                    const uint64_t ml = __ballot(pass_ && leaf);
                    const int nlf = __popcll(ml);
                    int add;
                    if (!push_inner(pass_ && !leaf, nd, L, work, tail, kGatherWork, add) ||
                        ngl + nlf > kGatherLeaves) {
                        over = true;
                        break;
                    }
                    if (pass_ && leaf)
                        gathered[ngl + __popcll(ml & lanemask_lt())] = ((uint64_t)bd << 32) | (uint32_t)nd;
                    tail += add;
                    ngl += nlf;
                    __builtin_amdgcn_wave_barrier();
                }
                if (!over) {
                    done_by_gather = true;
                    for (int c0 = 0; c0 < ngl; c0 += 64) {
                        const int cn = min(64, ngl - c0);
                        const uint64_t ge = wave_sort_u64(lane < cn ? gathered[c0 + lane] : kEmptyKey);
                        for (int i = 0; i < cn; ++i) {
                            const int node = __builtin_amdgcn_readlane((int)(uint32_t)ge, i);
                            const Node x = tree[node];
                            ++st_nodes;
                            if (needed(x)) visit_leaf(node);
                        }
                    }
                }
                __builtin_amdgcn_wave_barrier();
            }
            if (!done_by_gather) {
                // the walk: a wave-uniform stack, nearest child popped first
                int sp = 1;
                if (lane == 0) stk[0] = 1;
                __builtin_amdgcn_wave_barrier();
                while (sp > 0) {
                    --sp;
                    const int node = __builtin_amdgcn_readfirstlane(stk[sp]);
                    __builtin_amdgcn_wave_barrier();
                    const Node x = tree[node];
                    ++st_nodes;
                    if (!needed(x)) continue;
                    if (node >= L) {
                        visit_leaf(node);
                        continue;
                    }
                    const int first = 2 * node;
                    const Node b0 = tree[first], b1 = tree[first + 1];
                    float f0, f1;
                    const float d0 = box_d2(b0, f0), d1 = box_d2(b1, f1);
                    // pushed farther first; at equal distance the lower node pops first
                    const bool swap = d1 >= d0;
                    if (lane == 0) {
                        stk[sp] = swap ? first + 1 : first;
                        stk[sp + 1] = swap ? first : first + 1;
                    }
                    sp += 2;
                    __builtin_amdgcn_wave_barrier();
                }
            }
            // as in k_comp_search: exact when the best is within lim, else
            // nothing lies within lim, and with lim = cbb the point stops on
            // its lower bound
            if (key_bound(bk) <= lim) {
                open = false;
                if (bk != kEmptyKey && lane == 0)
                    atomic_min_if_lower(&comp1[mylab],
                                        (bk & 0xffffffff00000000ull) | (uint64_t)min(pid, (uint32_t)bk));
            } else if (cbb <= cap) {
                open = false;
                bounded = true;
                lbnd = cbb;
            }
            inner = max(inner, cap);
            r2 *= 8.f;
        }
        if (lane == 0) {
            if (bounded) {
                corr[p] = -1;
                corr_key[p] = ((uint64_t)(uint32_t)lbnd << 32) | 0xffffffffull;
            } else {
                corr[p] = bk == kEmptyKey ? -2 : inv[(uint32_t)bk];
                corr_key[p] = bk;
            }
        }
    }
    if (collect && lane == 0) {
        const int slot = (blockIdx.x * kDeferWaves + w) % kWorkSlots;
        atomicAdd(&C->work[kWorkCompNodes][slot], (unsigned long long)st_nodes);
        atomicAdd(&C->work[kWorkCompLeaves][slot], (unsigned long long)st_leaves);
        atomicAdd(&C->work[kWorkCompPairs][slot], st_pairs);
    }
}

// Round 1 of the component search and its neighbour lists.  Every component
// is one point, so a point's nearest outside point is its nearest neighbour.
// One wave per 64 consecutive positions keeps each lane's K smallest keys
// (d2, id) in registers.  The leaves holding the packet's own points come
// first; then every lane's K-th key bounds its search.  The packet
// gathers, 64 nodes per step (one box-to-box test per lane), every other leaf
// whose box lies within the largest of those bounds of the packet's box, and
// visits them nearest first.  At a leaf, a lane takes part only while the
// leaf box may still beat its K-th key, and a leaf point enters the pair
// loop only when it lies within the bound of an 8-lane group of the packet
// that takes part (the group's box and its largest bound).  A packet whose
// gathering outgrows the LDS lists walks the hierarchy per lane instead,
// nearest child first.  In the pair loop each lane is one query and the
// leaf's points are read in turn at one address for the whole wave.
//
// The list holds keys only, biased by 2^52: (d2 bits << 32 | id) + 2^52 with
// d2 bits <= 0x7f800000 is a positive normal double whose order is the key's,
// so an insertion is a min/max network of K FP64 min/max pairs without
// branches or selects (the empty key is the largest finite double).  The
// positions come from inv at the end.
constexpr uint64_t kKnnBias = 1ull << 52;
constexpr uint64_t kKnnEmpty = 0x7fefffffffffffffull;
constexpr uint32_t kKnnBiasHi = (uint32_t)(kKnnBias >> 32);

// returns min(a, x) and leaves max(a, x) in x, for doubles that are never NaN:
// v_min_f64 / v_max_f64 without the canonicalising v_max_f64 the compiler
// puts before each input of fmin / fmax.  The minimum is written over a's
// register, so a network kd[i] = minmax_f64(kd[i], x) needs no copies.
__device__ __forceinline__ double minmax_f64(double a, double& x)
{
    double hi;
    asm("v_max_f64 %1, %0, %2\n\tv_min_f64 %0, %0, %2" : "+v"(a), "=&v"(hi) : "v"(x));
    x = hi;
    return a;
}
template <int D>
__global__ __launch_bounds__(64) void k_knn_first(int64_t n, const float4* __restrict__ pts,
                                                 const Node* __restrict__ nodes, const Cloud* __restrict__ clouds,
                                                 int ncl, int bucket, LeafTable lt, const int32_t* __restrict__ inv,
                                                 int32_t* __restrict__ corr, uint64_t* __restrict__ corr_key,
                                                 NbrList nb, Counters* C, int collect, int qpp)
{
    __shared__ int32_t stk_id[64];
    __shared__ int32_t stk_ver[64];
    __shared__ unsigned long long stk_mask[64];
    __shared__ int32_t work[kKnnGatherWork];
    __shared__ unsigned long long gathered[kKnnGatherLeaves];
    __shared__ float4 gbox[16];             // per 8-lane group: lo (xyz), hi (xyz)
    if (C->done) return;                    // a build whose input was refused on the device
    const int lane = __lane_id();
    if (blockIdx.x == 0 && lane == 0) C->knn_round1 = 1u;
    const int64_t p0 = (int64_t)blockIdx.x * qpp, p = p0 + lane;
    const bool active = lane < qpp && p < n;
    const float4 me = pts[active ? p : 0];
    const float px = me.x, py = me.y, pz = me.z;
    const int my_cl = active ? find_cloud(clouds, ncl, p) : -1;
    constexpr int K = knn_len(D);   // list length
    double kd[K];                   // biased keys as doubles, ascending
#pragma unroll
    for (int i = 0; i < K; ++i) kd[i] = __longlong_as_double((long long)kKnnEmpty);
    auto last = [&]() { return (uint64_t)__double_as_longlong(kd[K - 1]); };
    // sorted insertion of a biased key (keys are distinct: the id is in the
    // low word)
    auto insert = [&](uint64_t key) {
        double x = __longlong_as_double((long long)key);
#pragma unroll
        for (int i = 0; i < K; ++i) kd[i] = minmax_f64(kd[i], x);
    };
    // the K-th d2 bits (an empty list: above every finite d2)
    auto bound = [&]() { return (uint32_t)(last() >> 32) - kKnnBiasHi; };
    uint32_t st_nodes = 0, st_leaves = 0, st_steps = 0, st_walks = 0;   // work counters of this packet
    uint64_t pending = __ballot(active);
    while (pending) {
        const int cl = __builtin_amdgcn_readfirstlane(__shfl(my_cl, (int)__builtin_ctzll(pending)));
        const uint64_t minem = __ballot(my_cl == cl);
        const bool mine = my_cl == cl;
        pending &= ~minem;
        const int64_t cend = clouds[cl].pos + clouds[cl].n;
        const int64_t L = clouds[cl].L, lfirst = clouds[cl].lfirst, nl = clouds[cl].nl;
        const Node* __restrict__ tree = nodes + 2 * clouds[cl].lbase;
        // the box of the group's points, and of each 8-lane group's
        float qlo[3] = {mine ? px : INFINITY, mine ? py : INFINITY, mine ? pz : INFINITY};
        float qhi[3] = {mine ? px : -INFINITY, mine ? py : -INFINITY, mine ? pz : -INFINITY};
        for (int off = 1; off < 64; off <<= 1) {
#pragma unroll
            for (int k = 0; k < 3; ++k) {
                qlo[k] = fminf(qlo[k], __shfl_xor(qlo[k], off));
                qhi[k] = fmaxf(qhi[k], __shfl_xor(qhi[k], off));
            }
            if (off == 4 && (lane & 7) == 0) {
                gbox[2 * (lane >> 3)] = make_float4(qlo[0], qlo[1], qlo[2], 0.f);
                gbox[2 * (lane >> 3) + 1] = make_float4(qhi[0], qhi[1], qhi[2], 0.f);
            }
        }
        __builtin_amdgcn_wave_barrier();
        auto needed = [&](const Node& nd, uint32_t nm) {
            if (!mine) return false;
            const float q[3] = {px, py, pz};
            float m[3];
#pragma unroll
            for (int k = 0; k < 3; ++k) m[k] = fmaxf(fmaxf(nd.lo[k] - q[k], q[k] - nd.hi[k]), 0.f);
            const float lb = D == 3 ? d2_of(m[0], m[1], m[2]) : d2_of(m[0], m[1]);
            return (((uint64_t)(__float_as_uint(lb) + kKnnBiasHi) << 32) | nm) < last();
        };
        // one leaf point per candidate step, at one address for the wave
        auto pairs = [&](int64_t s0, uint64_t cand, bool own) {
            ++st_leaves;
            st_steps += (uint32_t)__popcll(cand);
            while (cand) {
                const int j = (int)__builtin_ctzll(cand);
                cand &= cand - 1;
                const float4 v = pts[s0 + j];
                const float dx = v.x - px, dy = v.y - py, dz = v.z - pz;
                const float d2 = D == 3 ? d2_of(dx, dy, dz) : d2_of(dx, dy);
                const uint32_t db = __float_as_uint(d2);
                const uint64_t key = ((uint64_t)(db + kKnnBiasHi) << 32) | __float_as_uint(v.w);
                if (mine && key < last() && (!own || s0 + j != p)) insert(key);
            }
        };
        // the packet's own leaves: a leaf point farther from the packet's box
        // than every lane's K-th d2 cannot enter a list
        auto scan_own = [&](int node) {
            int64_t s0, s1;
            leaf_range(lt, lfirst, nl, cend, node - L, s0, s1);
            const int cnt = (int)(s1 - s0);
            uint32_t t = mine ? bound() : 0u;
            for (int off = 32; off > 0; off >>= 1) t = max(t, (uint32_t)__shfl_xor((int)t, off));
            bool keep = false;
            if (lane < cnt) {
                const float4 w = pts[s0 + lane];
                const float wq[3] = {w.x, w.y, w.z};
                float m[3];
#pragma unroll
                for (int k = 0; k < 3; ++k) m[k] = fmaxf(fmaxf(qlo[k] - wq[k], wq[k] - qhi[k]), 0.f);
                const float lb = D == 3 ? d2_of(m[0], m[1], m[2]) : d2_of(m[0], m[1]);
                keep = __float_as_uint(lb) <= t;
            }
            pairs(s0, __ballot(keep), true);
        };
        // another leaf, for the lanes of needm: a leaf point is paired when it
        // lies within the largest K-th d2 of a taking-part group's lanes
        // from that group's box
        auto scan_other = [&](int node, bool need, uint64_t needm) {
            int64_t s0, s1;
            leaf_range(lt, lfirst, nl, cend, node - L, s0, s1);
            const int cnt = (int)(s1 - s0);
            const uint32_t t = group8_max_u32(need ? bound() : 0u);
            float4 w = make_float4(0.f, 0.f, 0.f, 0.f);
            if (lane < cnt) w = pts[s0 + lane];
            bool keep = false;
#pragma unroll 1
            for (int g = 0; g < 8; ++g) {
                if (((needm >> (8 * g)) & 0xffull) == 0ull) continue;
                const uint32_t tg = (uint32_t)__builtin_amdgcn_readlane((int)t, 8 * g);
                const float4 lo = gbox[2 * g], hi = gbox[2 * g + 1];
                const float m0 = fmaxf(fmaxf(lo.x - w.x, w.x - hi.x), 0.f);
                const float m1 = fmaxf(fmaxf(lo.y - w.y, w.y - hi.y), 0.f);
                const float m2 = fmaxf(fmaxf(lo.z - w.z, w.z - hi.z), 0.f);
                const float lb = D == 3 ? d2_of(m0, m1, m2) : d2_of(m0, m1);
                keep = keep || __float_as_uint(lb) <= tg;
            }
            pairs(s0, __ballot(keep && lane < cnt), false);
        };
        // the leaves holding the packet's points of this cloud
        const int first = (int)__builtin_ctzll(minem), last = 63 - (int)__builtin_clzll(minem);
        const int64_t pf = p0 + first, pl = p0 + last;
        const int leaf_lo = (int)(L + (lt.of[pf] - lfirst)), leaf_hi = (int)(L + (lt.of[pl] - lfirst));
        for (int lf = leaf_lo; lf <= leaf_hi; ++lf) scan_own(lf);
        // gather the other leaves within the largest K-th d2 of the packet's box
        uint32_t R = mine ? bound() : 0u;
        for (int off = 32; off > 0; off >>= 1) R = max(R, (uint32_t)__shfl_xor((int)R, off));
        int head = 0, tail = gather_start(L, work), ngl = 0;
        bool over = false;
        __builtin_amdgcn_wave_barrier();
        while (head < tail) {
            const int take = min(64, tail - head);
            const int nd = lane < take ? work[head + lane] : 0;
            head += take;
            st_nodes += (uint32_t)take;
            bool pass = false, leaf = false;
            uint32_t bd = 0;
            if (lane < take) {
                const Node x = tree[nd];
                float m[3];
#pragma unroll
                for (int k = 0; k < 3; ++k) m[k] = fmaxf(fmaxf(x.lo[k] - qhi[k], qlo[k] - x.hi[k]), 0.f);
                bd = __float_as_uint(D == 3 ? d2_of(m[0], m[1], m[2]) : d2_of(m[0], m[1]));
                leaf = nd >= L;
                pass = bd <= R && !(leaf && nd >= leaf_lo && nd <= leaf_hi);
            }
            const uint64_t ml = __ballot(pass && leaf);
            const int nl = __popcll(ml);
            int add;
            if (!push_inner(pass && !leaf, nd, L, work, tail, kKnnGatherWork, add) || ngl + nl > kKnnGatherLeaves) {
                over = true;
                break;
            }
            if (pass && leaf) gathered[ngl + __popcll(ml & lanemask_lt())] = ((uint64_t)bd << 32) | (uint32_t)nd;
            tail += add;
            ngl += nl;
            __builtin_amdgcn_wave_barrier();
        }
        if (!over) {
            // nearest first, 64 leaves at a time
            for (int c0 = 0; c0 < ngl; c0 += 64) {
                const int cn = min(64, ngl - c0);
                const uint64_t e = wave_sort_u64(lane < cn ? gathered[c0 + lane] : kEmptyKey);
                for (int i = 0; i < cn; ++i) {
                    const int node = __builtin_amdgcn_readlane((int)(uint32_t)e, i);
                    const Node x = tree[node];
                    ++st_nodes;
                    const bool need = needed(x, __float_as_uint(x.pad[0]));
                    const uint64_t needm = __ballot(need);
                    if (needm != 0ull) scan_other(node, need, needm);
                }
            }
            continue;
        }
        // the per-lane walk: from the root, nearest child first (from the
        // packet's centroid), the own leaves skipped
        ++st_walks;
        float cx = mine ? px : 0.f, cy = mine ? py : 0.f, cz = mine ? pz : 0.f;
        float na = mine ? 1.f : 0.f;
        for (int off = 32; off > 0; off >>= 1) {
            cx += __shfl_xor(cx, off);
            cy += __shfl_xor(cy, off);
            cz += __shfl_xor(cz, off);
            na += __shfl_xor(na, off);
        }
        cx /= na; cy /= na; cz /= na;
        auto cdist = [&](const Node& x) {
            const float dxx = fmaxf(fmaxf(x.lo[0] - cx, cx - x.hi[0]), 0.f);
            const float dyy = fmaxf(fmaxf(x.lo[1] - cy, cy - x.hi[1]), 0.f);
            const float dzz = fmaxf(fmaxf(x.lo[2] - cz, cz - x.hi[2]), 0.f);
            return dxx * dxx + dyy * dyy + dzz * dzz;
        };
        int sp = 1;
        int ver = 0;
        if (lane == 0) {
            stk_id[0] = 1;
            stk_ver[0] = -1;
        }
        __builtin_amdgcn_wave_barrier();
        while (sp > 0) {
            --sp;
            const int node = __builtin_amdgcn_readfirstlane(stk_id[sp]);
            const int pver = __builtin_amdgcn_readfirstlane(stk_ver[sp]);
            bool need;
            if (pver == ver) {
                need = (stk_mask[sp] >> lane) & 1ull;
            } else {
                const Node nd = tree[node];
                need = needed(nd, __float_as_uint(nd.pad[0]));
                ++st_nodes;
            }
            const uint64_t needm = __ballot(need);
            if (needm == 0ull) continue;
            if (node >= L) {
                if (node >= leaf_lo && node <= leaf_hi) continue;
                scan_other(node, need, needm);
                ++ver;
            } else {
                const bool leafkids = 2 * (int64_t)node >= L;
                const int fc = leafkids ? 2 * node : 4 * node;
                const int nk = leafkids ? 2 : 4;
                st_nodes += (uint32_t)nk;
                uint64_t mk[4];
                float dk[4];
                int id[4];
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    mk[i] = 0ull;
                    dk[i] = -1.f;
                    id[i] = fc + i;
                    if (i < nk) {
                        const Node bx = tree[fc + i];
                        mk[i] = __ballot(needed(bx, __float_as_uint(bx.pad[0])));
                        if (mk[i]) dk[i] = cdist(bx);
                    }
                }
                // pushed farthest first, so the nearest pops first
                auto ce = [&](int a, int b) {
                    if (dk[a] < dk[b] || (dk[a] == dk[b] && id[a] < id[b])) {
                        const float td = dk[a]; dk[a] = dk[b]; dk[b] = td;
                        const uint64_t tm = mk[a]; mk[a] = mk[b]; mk[b] = tm;
                        const int ti = id[a]; id[a] = id[b]; id[b] = ti;
                    }
                };
                ce(0, 1); ce(2, 3); ce(0, 2); ce(1, 3); ce(1, 2);
                if (lane == 0) {
                    int t = sp;
#pragma unroll
                    for (int i = 0; i < 4; ++i)
                        if (mk[i]) { stk_id[t] = id[i]; stk_ver[t] = ver; stk_mask[t] = mk[i]; ++t; }
                }
#pragma unroll
                for (int i = 0; i < 4; ++i) sp += mk[i] != 0ull ? 1 : 0;
                __builtin_amdgcn_wave_barrier();
            }
        }
    }
    if (collect && lane == 0) {
        const int slot = blockIdx.x % kWorkSlots;
        atomicAdd(&C->work[kWorkKnnNodes][slot], (unsigned long long)st_nodes);
        atomicAdd(&C->work[kWorkKnnLeaves][slot], (unsigned long long)st_leaves);
        atomicAdd(&C->work[kWorkKnnPairs][slot], (unsigned long long)qpp * st_steps);
        atomicAdd(&C->work[kWorkKnnWalks][slot], (unsigned long long)st_walks);
    }
    if (!active) return;
    int32_t pos0 = -2;
    uint64_t key0 = kEmptyKey;
#pragma unroll
    for (int i = 0; i < K; ++i) {
        const uint64_t b = (uint64_t)__double_as_longlong(kd[i]);
        const bool has = b != kKnnEmpty;
        const uint64_t key = has ? b - kKnnBias : kEmptyKey;
        const int32_t pos = has ? inv[(uint32_t)key] : -1;
        if (i == 0 && has) {
            pos0 = pos;
            key0 = key;
        }
        nb.pos[(int64_t)i * n + p] = pos;
        nb.key[(int64_t)i * n + p] = key;
    }
    corr[p] = pos0;
    corr_key[p] = key0;
    nb.cur[p] = 0;
}

// ---- cycle rule of the 2.5D mode (CycleState).  Roots are the points whose
// flattened label is their own position.  In round 1 every component is one
// point and its chosen edge is its nearest neighbour, whose choices close
// only mutual pairs (the edges along a cycle of choices could not increase),
// so the rule starts at round 2.
//
// k_cycle_init: per root, its target j0 (itself when it has no outgoing
// candidate or is in a mutual pair) and cut = 0; the roots with another target are listed (cy.roots, C->nroots), one
// block-wide reservation per chunk of kCyChunk points.
constexpr int kCyChunk = 2048;                 // (8192: 315 us over those rounds, 2048: 193)
constexpr int kCyPer = kCyChunk / kBlock;      // points per thread, one bit each

__global__ __launch_bounds__(kBlock) void k_cycle_init(int64_t n, const int32_t* __restrict__ label,
                                                      const uint64_t* __restrict__ comp1,
                                                      const uint32_t* __restrict__ comp2, CycleState cy,
                                                      Counters* C)
{
    if (C->done || C->round <= 1u) return;
    __shared__ uint32_t wsum[kBlock / 64];
    __shared__ uint32_t base;
    const int64_t c0 = (int64_t)blockIdx.x * kCyChunk;
    uint32_t bits = 0;
    for (int i = 0; i < kCyPer; ++i) {
        const int64_t r = c0 + (int64_t)i * kBlock + threadIdx.x;
        if (r >= n || label[r] != (int32_t)r) continue;
        int32_t t = (int32_t)r;
        const uint64_t k1 = comp1[r];
        const uint32_t k2 = comp2[r];
        if (k1 != kEmptyKey) {
            // the chosen edge (d2, min id, max id): its end outside the component
            const int32_t la = label[cy.inv[(uint32_t)k1]], lb = label[cy.inv[k2]];
            const int32_t o = la == (int32_t)r ? lb : la;
            if (!(comp1[o] == k1 && comp2[o] == k2)) t = o;     // else a mutual pair
        }
        cy.j0[r] = t;
        cy.cut[r] = 0;
        if (t != (int32_t)r) bits |= 1u << i;
    }
    // block-exclusive offsets of the listed roots, in thread order
    const uint32_t cnt = (uint32_t)__popc(bits);
    uint32_t incl = cnt;
    for (int off = 1; off < 64; off <<= 1) {
        const uint32_t o = (uint32_t)__shfl_up((int)incl, off);
        if (__lane_id() >= off) incl += o;
    }
    const int w = threadIdx.x / 64;
    if (__lane_id() == 63) wsum[w] = incl;
    __syncthreads();
    if (threadIdx.x == 0) {
        uint32_t tot = 0;
        for (int k = 0; k < kBlock / 64; ++k) {
            const uint32_t x = wsum[k];
            wsum[k] = tot;
            tot += x;
        }
        base = tot ? atomicAdd(&C->nroots, tot) : 0u;
    }
    __syncthreads();
    uint32_t at = base + wsum[w] + incl - cnt;
    for (int i = 0; i < kCyPer; ++i)
        if ((bits >> i) & 1u) cy.roots[at++] = (int32_t)(c0 + (int64_t)i * kBlock + threadIdx.x);
}

// the chosen edge of root a is larger than that of root b
__device__ __forceinline__ bool cycle_above(const uint64_t* comp1, const uint32_t* comp2, int32_t a, int32_t b)
{
    const uint64_t ka = comp1[a], kb = comp1[b];
    return ka > kb || (ka == kb && comp2[a] > comp2[b]);
}

// A listed root is cut when its choices lead back to it past smaller edges
// only, so each walks along them until an edge larger than its own, a root
// with no target, itself, or a root met before (a cycle without it: the last
// power-of-two hop is remembered).  Edges mostly shrink along the choices, so
// walks are short: over the 12 rounds of a 3*10^6-point terrain they take
// 171 us in all, and the launches behind them, idle, 245.  (Pointer doubling
// alone took 22 launches a round there, 1.57 ms.)
__global__ __launch_bounds__(kBlock) void k_cycle_walk(const uint64_t* __restrict__ comp1,
                                                      const uint32_t* __restrict__ comp2, CycleState cy,
                                                      Counters* C)
{
    if (C->done || C->round <= 1u) return;
    const uint32_t R = C->nroots;
    for (int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; t < (int64_t)R;
         t += (int64_t)gridDim.x * blockDim.x) {
        const int32_t r = cy.roots[t];
        int32_t x = cy.j0[r], met = r;
        int hops = 0, next = 1;
        bool cut = false, left = false;
        for (;;) {
            if (x == r) {
                cut = true;
                break;
            }
            if (x == met || cycle_above(comp1, comp2, x, r)) break;
            if (++hops == kCyWalk) {
                left = true;
                break;
            }
            if (hops == next) {
                met = x;
                next *= 2;
            }
            const int32_t y = cy.j0[x];
            if (y == x) break;
            x = y;
        }
        if (cut) {
            cy.cut[r] = 1;
            atomicAdd(&C->cycles_cut, 1u);
        }
        if (left) C->walk_left = 1u;
    }
}

// Pointer jumping over the listed roots, when a walk was too long: launch k
// goes kCyHops hops of the last launch's states (launch 0: of the choices
// themselves) and keeps the root on the way whose edge is largest.
__global__ __launch_bounds__(kBlock) void k_cycle_step(const uint64_t* __restrict__ comp1,
                                                      const uint32_t* __restrict__ comp2, CycleState cy, int k,
                                                      const Counters* C)
{
    if (C->done || C->round <= 1u || !C->walk_left) return;
    const uint32_t R = C->nroots;
    if (k >= cycle_steps(R)) return;
    const uint64_t* src = cy.st[k & 1];
    uint64_t* dst = cy.st[(k & 1) ^ 1];
    for (int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; t < (int64_t)R;
         t += (int64_t)gridDim.x * blockDim.x) {
        const int32_t r = cy.roots[t];
        int32_t j = r, top = r;
        for (int hop = 0; hop < kCyHops; ++hop) {
            const int32_t y = cy.j0[j];
            if (y == j) break;
            int32_t to = y, on = j;
            if (k > 0) {
                const uint64_t st = src[j];
                to = (int32_t)(st >> 32);
                on = (int32_t)(uint32_t)st;
            }
            if (on != top && cycle_above(comp1, comp2, on, top)) top = on;
            j = to;
        }
        dst[r] = (uint64_t)(uint32_t)j << 32 | (uint32_t)top;
        if (k == 0) cy.onc[r] = 0;
    }
}

// after the steps, every listed root's hop target lies on a cycle (or is a
// root with no target), and every root of a cycle is such a target
__global__ __launch_bounds__(kBlock) void k_cycle_mark(CycleState cy, const Counters* C)
{
    if (C->done || C->round <= 1u || !C->walk_left) return;
    const uint32_t R = C->nroots;
    const uint64_t* fin = cy.st[cycle_steps(R) & 1];
    for (int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; t < (int64_t)R;
         t += (int64_t)gridDim.x * blockDim.x)
        cy.onc[fin[cy.roots[t]] >> 32] = 1;
}

// (those that their walk has cut are cut here again, and not counted twice)
__global__ __launch_bounds__(kBlock) void k_cycle_cut(CycleState cy, Counters* C)
{
    if (C->done || C->round <= 1u || !C->walk_left) return;
    const uint32_t R = C->nroots;
    const uint64_t* fin = cy.st[cycle_steps(R) & 1];
    for (int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; t < (int64_t)R;
         t += (int64_t)gridDim.x * blockDim.x) {
        const int32_t r = cy.roots[t];
        if (!cy.onc[r] || (int32_t)(uint32_t)fin[r] != r || cy.cut[r]) continue;
        cy.cut[r] = 1;
        atomicAdd(&C->cycles_cut, 1u);
    }
}

// flatten (EMSTOperators.h:412-433): chase label2 to the root, with path
// halving on label2 (every write stores an ancestor, so concurrent chases stay
// valid and label2 stays a parent forest); reset the component minima for the
// next round.  Only this round's roots (label[p] == p) can hold minima (every
// update goes to a point's root), and a label that stays is not rewritten:
// later rounds absorb few roots, and the stores of unchanged values took most
// of the pass.
// Each launch takes at most kFlattenSteps steps per point; a point still off
// its root raises C->unflat and the host launches the kernel again, so every
// wave ends even if the hook forest were malformed.
constexpr int kFlattenSteps = 4096;

__global__ __launch_bounds__(kBlock) void k_round_flatten(int64_t n, int32_t* __restrict__ label,
                                                         int32_t* label2,
                                                         uint64_t* __restrict__ comp1,
                                                         uint32_t* __restrict__ comp2, Counters* C)
{
    if (C->done & 1u || C->done == 4u) return;      // a round paused here (done == 2) still flattens
    const int64_t p = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (p >= n) return;
    const int32_t was = label[p];
    int32_t r = label2[p];
    int32_t nx = label2[r];
    int steps = 0;
    while (nx != r && steps < kFlattenSteps) {
        const int32_t nn = label2[nx];
        label2[r] = nn;
        r = nn;
        nx = label2[r];
        ++steps;
    }
    if (nx != r) atomicOr(&C->unflat, 1u);
    // p itself now points at the root (or the farthest ancestor reached), so
    // the next round's chase from p starts there
    if (steps > 0) label2[p] = r;
    if (r != was) label[p] = r;
    if (was == (int32_t)p) {
        comp1[p] = kEmptyKey;
        comp2[p] = 0xffffffffu;
    }
}

// ------------------------------------------------------------- weight
template <int D>
__global__ __launch_bounds__(kBlock) void k_weight(const float* __restrict__ xyz,
                                                  const int32_t* __restrict__ eu,
                                                  const int32_t* __restrict__ ev, int64_t m,
                                                  double* __restrict__ partial)
{
    __shared__ double sh[kBlock / 64];
    double s = 0;
    const int64_t stride = (int64_t)gridDim.x * blockDim.x;
    for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < m; i += stride) {
        if (eu[i] < 0) continue;
        const float* a = xyz + (int64_t)eu[i] * D;
        const float* b = xyz + (int64_t)ev[i] * D;
        const float dx = a[0] - b[0], dy = a[1] - b[1];
        const float d2 = D == 3 ? d2_of(dx, dy, a[2] - b[2]) : d2_of(dx, dy);
        s += sqrt((double)d2);
    }
    for (int off = 32; off > 0; off >>= 1) s += __shfl_xor(s, off);
    if (__lane_id() == 0) sh[threadIdx.x / 64] = s;
    __syncthreads();
    if (threadIdx.x == 0) {
        double t = 0;
        for (int w = 0; w < kBlock / 64; ++w) t += sh[w];
        partial[blockIdx.x] = t;
    }
}

// Per cloud (one block each): FP64 weight of its edges in input coordinates,
// edge count, last round that added an edge.  Edges sit at the sorted
// position of the root they absorbed, inside the cloud's range.
template <int D>
__global__ __launch_bounds__(kBlock) void k_cloud_results(const float* __restrict__ xyz,
                                                         const Cloud* __restrict__ cl,
                                                         const int32_t* __restrict__ eu,
                                                         const int32_t* __restrict__ ev,
                                                         const int32_t* __restrict__ eround,
                                                         double* __restrict__ weight,
                                                         int32_t* __restrict__ edges,
                                                         int32_t* __restrict__ last_round)
{
    __shared__ double shw[kBlock / 64];
    __shared__ int32_t shc[kBlock / 64], shr[kBlock / 64];
    const int c = blockIdx.x;
    const int64_t a = cl[c].pos, b = a + cl[c].n;
    double s = 0;
    int32_t cnt = 0, lr = 0;
    for (int64_t i = a + threadIdx.x; i < b; i += blockDim.x) {
        if (eu[i] < 0) continue;
        const float* p = xyz + (int64_t)eu[i] * D;
        const float* q = xyz + (int64_t)ev[i] * D;
        const float dx = p[0] - q[0], dy = p[1] - q[1];
        const float d2 = D == 3 ? d2_of(dx, dy, p[2] - q[2]) : d2_of(dx, dy);
        s += sqrt((double)d2);
        ++cnt;
        lr = max(lr, eround[i]);
    }
    for (int off = 32; off > 0; off >>= 1) {
        s += __shfl_xor(s, off);
        cnt += __shfl_xor(cnt, off);
        lr = max(lr, __shfl_xor(lr, off));
    }
    if (__lane_id() == 0) {
        shw[threadIdx.x / 64] = s;
        shc[threadIdx.x / 64] = cnt;
        shr[threadIdx.x / 64] = lr;
    }
    __syncthreads();
    if (threadIdx.x == 0) {
        double t = 0;
        int32_t tc = 0, tr = 0;
        for (int w = 0; w < kBlock / 64; ++w) {
            t += shw[w];
            tc += shc[w];
            tr = max(tr, shr[w]);
        }
        weight[c] = t;
        edges[c] = tc;
        last_round[c] = tr;
    }
}

// ------------------------------------------------------------ outputs
__global__ __launch_bounds__(kBlock) void k_labels_out(int64_t n, const int32_t* __restrict__ label,
                                                      const float4* __restrict__ pts,
                                                      const int32_t* __restrict__ inv,
                                                      int32_t* __restrict__ out)
{
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    out[i] = (int32_t)__float_as_uint(pts[label[inv[i]]].w);
}

__global__ __launch_bounds__(kBlock) void k_cands_out(int K, int64_t n, const uint64_t* __restrict__ ck,
                                                     const int32_t* __restrict__ inv,
                                                     int32_t* __restrict__ cand, float* __restrict__ cd2)
{
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const int64_t s = inv[i];
    for (int k = 0; k < K; ++k) {
        const uint64_t key = ck[(int64_t)k * n + s];
        cand[i * K + k] = key == kEmptyKey ? -1 : (int32_t)(uint32_t)key;
        cd2[i * K + k] = key == kEmptyKey ? INFINITY : __uint_as_float((uint32_t)(key >> 32));
    }
}

// sort key of an edge: its ids, `bits` bits each (u < v, so no edge has the
// empty slots' key of all ones)
__global__ __launch_bounds__(kBlock) void k_edge_keys(const int32_t* __restrict__ eu,
                                                     const int32_t* __restrict__ ev, int64_t m, int bits,
                                                     uint64_t* __restrict__ keys)
{
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= m) return;
    keys[i] = eu[i] < 0 ? (1ull << (2 * bits)) - 1ull : (((uint64_t)(uint32_t)eu[i] << bits) | (uint32_t)ev[i]);
}

__global__ __launch_bounds__(kBlock) void k_edges_out(const uint64_t* __restrict__ keys,
                                                     const uint32_t* __restrict__ idx,
                                                     const float* __restrict__ ed2, int64_t m, int bits,
                                                     int32_t* __restrict__ u, int32_t* __restrict__ v,
                                                     float* __restrict__ d2)
{
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= m) return;
    const uint64_t k = keys[i];
    u[i] = (int32_t)(k >> bits);
    v[i] = (int32_t)(k & ((1ull << bits) - 1ull));
    d2[i] = ed2[idx[i]];
}

// ------------------------------------------------ reference cell grid
// findCell (ViewGrid.h:339-359): p1 = FEuclid(FDual(0)), size_slab = 2R;
// li = (float)(p - p1) + R in double; cell = floor(li / 2R).
__global__ __launch_bounds__(kBlock) void k_cell_grid(const float* __restrict__ resc, int64_t n, int dim,
                                                     int pstride, const int32_t* __restrict__ geo,
                                                     int32_t* __restrict__ cell_of,
                                                     uint64_t* __restrict__ keys,
                                                     uint32_t* __restrict__ cell_count)
{
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const int R = geo[9];
    bool ok = true;
    int32_t c[3] = {0, 0, 0};
    for (int k = 0; k < dim; ++k) {
        const int32_t PC = geo[3 + k], pc = geo[6 + k];
        const float p1 = (float)((PC % 2) * R - PC * R + pc);
        const float p2 = (float)((2 + PC % 2) * R - PC * R + pc);
        const double size_slab = (double)(p2 - p1);
        const float dif = resc[i * pstride + k] - p1;
        const double li = (double)dif + size_slab / 2;
        c[k] = (int32_t)floor(li / size_slab);
        ok = ok && c[k] >= 0 && c[k] < geo[k];
    }
    for (int k = 0; k < 3; ++k) cell_of[i * 3 + k] = ok ? c[k] : -1;
    const int64_t ncell = (int64_t)geo[0] * geo[1] * geo[2];
    const int64_t lin = ok ? (int64_t)c[0] + (int64_t)geo[0] * ((int64_t)c[1] + (int64_t)geo[1] * c[2]) : ncell;
    keys[i] = (uint64_t)lin;
    if (ok) atomicAdd(&cell_count[lin], 1u);
}

inline unsigned nblocks(int64_t n, int b = kBlock) { return (unsigned)((n + b - 1) / b); }

}  // namespace

// ================================================================ launchers
void launch_bbox(const float* xyz, const Cloud* cl, int ncl, int64_t N, int dim, Params* P, hipStream_t s)
{
    hipLaunchKernelGGL(k_bbox_init, dim3(nblocks(ncl)), dim3(kBlock), 0, s, P, ncl);
    if (N <= 0) return;
    if (ncl == 1) {
        const unsigned g1 = (unsigned)std::min<int64_t>(nblocks((N + kBoxAhead - 1) / kBoxAhead), kBoxBlocks);
        hipLaunchKernelGGL(dim == 3 ? k_bbox_one<3> : k_bbox_one<2>, dim3(g1), dim3(kBlock), 0, s, xyz, N, P);
        return;
    }
    const unsigned g = (unsigned)std::min<int64_t>(nblocks(N), 2048);
    if (dim == 3) hipLaunchKernelGGL(k_bbox<3>, dim3(g), dim3(kBlock), 0, s, xyz, cl, ncl, N, P);
    else hipLaunchKernelGGL(k_bbox<2>, dim3(g), dim3(kBlock), 0, s, xyz, cl, ncl, N, P);
}

void launch_params(Params* P, const Cloud* cl, int ncl, int dim, int mbits, hipStream_t s)
{
    hipLaunchKernelGGL(k_params, dim3(nblocks(ncl)), dim3(kBlock), 0, s, P, cl, ncl, dim, mbits);
}

void launch_rescale_keys(const float* xyz, const Cloud* cl, int ncl, int64_t N, int dim, int mbits,
                           const Params* P, float* resc, uint64_t* keys, bool hilbert, hipStream_t s)
{
    if (N <= 0) return;
    if (dim == 3)
        hipLaunchKernelGGL(k_rescale_keys<3>, dim3(nblocks(N)), dim3(kBlock), 0, s, xyz, cl, ncl, N, mbits, P,
                           resc, keys, hilbert ? 1 : 0);
    else
        hipLaunchKernelGGL(k_rescale_keys<2>, dim3(nblocks(N)), dim3(kBlock), 0, s, xyz, cl, ncl, N, mbits, P,
                           resc, keys, hilbert ? 1 : 0);
}

size_t scan_tmp_words(int64_t n) { return (size_t)((n + kScanTile - 1) / kScanTile) + 1; }

void exclusive_scan_u32(const uint32_t* in, uint32_t* out, int64_t n, uint32_t* tmp, hipStream_t s)
{
    if (n <= 0) return;
    if (n <= kScanOne) {
        hipLaunchKernelGGL(k_scan_one, dim3(1), dim3(1024), 0, s, in, out, (int)n);
        return;
    }
    const int64_t nb = (n + kScanTile - 1) / kScanTile;
    hipLaunchKernelGGL(k_scan_local, dim3((unsigned)nb), dim3(kBlock), 0, s, in, out, n, tmp);
    hipLaunchKernelGGL(k_scan_top, dim3(1), dim3(1024), 0, s, tmp, nb);
    hipLaunchKernelGGL(k_scan_add, dim3((unsigned)nb), dim3(kBlock), 0, s, out, n, tmp);
}

// tile states and counts of every pass (k_rs_pass)
size_t radix_hist_words(int64_t n) { return (size_t)(kRsMaxPasses * (rs_tiles(std::max<int64_t>(n, 1)) * 512 + 257)); }

bool radix_sort(uint64_t* k0, uint32_t* v0, uint64_t* k1, uint32_t* v1, int64_t n, int bits, bool vals_identity,
                uint32_t* hist, hipStream_t s)
{
    const int passes = std::max(1, (bits + 7) / 8);
    if (n <= 0) return false;
    if (n <= kRsSmallMax) {
        auto kern = n <= 2 * kRsSmallBlock ? k_rs_small<2> : (n <= 4 * kRsSmallBlock ? k_rs_small<4> : k_rs_small<8>);
        hipLaunchKernelGGL(kern, dim3(1), dim3(kRsSmallBlock), 0, s, k0, v0, (int)n, passes, vals_identity ? 1 : 0);
        return false;
    }
    const int64_t tiles = rs_tiles(n);
    unsigned long long* state = reinterpret_cast<unsigned long long*>(hist);
    uint32_t* counts = hist + passes * tiles * 512;
    uint32_t* ticket = counts + passes * 256;
    launch_zero_u32(hist, passes * (tiles * 512 + 257), s);
    hipLaunchKernelGGL(k_rs_hist, dim3(nblocks(n, kBlock * kRsHistItems)), dim3(kBlock), 0, s, (const uint64_t*)k0, n,
                       passes, counts);
    for (int p = 0; p < passes; ++p) {
        hipLaunchKernelGGL(k_rs_pass, dim3((unsigned)tiles), dim3(kRsThreads), 0, s, (const uint64_t*)k0,
                           (const uint32_t*)v0, k1, v1, n, p, (const uint32_t*)(counts + 256 * p),
                           state + (int64_t)p * tiles * 256, ticket + p, p == 0 && vals_identity ? 1 : 0);
        std::swap(k0, k1);
        std::swap(v0, v1);
    }
    return (passes & 1) != 0;
}

void launch_gather_sorted(const float* resc, const uint32_t* perm, int64_t n, int dim, float4* pts,
                          int32_t* inv, uint32_t* ids, hipStream_t s)
{
    if (n <= 0) return;
    if (dim == 3)
        hipLaunchKernelGGL(k_gather_sorted<3>, dim3(nblocks(n)), dim3(kBlock), 0, s, resc, perm, n, pts, inv, ids);
    else
        hipLaunchKernelGGL(k_gather_sorted<2>, dim3(nblocks(n)), dim3(kBlock), 0, s, resc, perm, n, pts, inv, ids);
}

void launch_dup_groups(const uint64_t* keys, const float4* pts, int64_t n, int32_t* rep,
                       int32_t* runs, int32_t* list, int32_t* gslot, Counters* C, hipStream_t s)
{
    if (n <= 0) return;
    hipLaunchKernelGGL(k_dup_runs, dim3(nblocks(n)), dim3(kBlock), 0, s, keys, n, rep, runs, C);
    const unsigned g = (unsigned)std::min<int64_t>(nblocks(n), 1024);
    hipLaunchKernelGGL(k_dup_group, dim3(g), dim3(kBlock), 0, s, keys, pts, n, rep, runs, list, gslot, C);
    hipLaunchKernelGGL(k_dup_big, dim3((unsigned)std::min<int64_t>(nblocks(n), 512)), dim3(kBlock), 0, s, pts, n,
                       rep, runs, list, C);
    hipLaunchKernelGGL(k_dup_finish, dim3(1), dim3(1), 0, s, C);
}

void launch_build_tree(const float4* pts, const Cloud* cl, int ncl, int64_t blocks, int64_t Lmax, LeafTable lt,
                       Node* nodes, const int32_t* rep, hipStream_t s)
{
    hipLaunchKernelGGL(k_tree_low, dim3((unsigned)blocks), dim3(kTreeBlock), 0, s, pts, cl, ncl, lt, nodes, rep);
    if (Lmax > kTreeLeaves) hipLaunchKernelGGL(k_tree_top, dim3((unsigned)ncl), dim3(1024), 0, s, cl, nodes);
}

void launch_cone_search(int dim, int cdim, const float4* pts, const Node* nodes, const Cloud* cl, int ncl,
                        int bucket, LeafTable lt, int64_t n, const int32_t* qlist, int64_t nq, const int32_t* label,
                        bool check_labels, const int32_t* inv, const float* seed_r, float seed_scale, float seed_mul,
                        uint64_t* cand_key, int32_t* cand_pos, int32_t* revive, int32_t* first_corr,
                        uint64_t* first_key, Counters* C, bool collect_stats, DupState dup,
                        const SplitScratch* split, int32_t* reach, hipStream_t s)
{
    if (nq <= 0) return;
    const unsigned g = nblocks(nq, 64);
    const int cs = collect_stats ? 1 : 0;
    auto kern = dim == 3 ? (cdim == 2 ? k_cone_search<3, 2> : k_cone_search<3, 3>) : k_cone_search<2, 2>;
    if (!split || qlist) {
        // Few queries: fewer to a packet, so that there are some 2500 packets
        // at least (ten waves a CU) and each is shorter: a launch of few
        // packets takes as long as one of them (2D / 3D, ms, 64 to a packet
        // against this rule: 1379 points 0.20 / 0.47 and 0.07 / 0.14, 10^4
        // 0.21 / 0.68 and 0.12 / 0.29, 3*10^4 0.23 / 0.75 and 0.16 / 0.51;
        // 10^5 points take 64).
        int qpp = 1;
        while (qpp < 64 && (int64_t)qpp * kConePackets < nq) qpp <<= 1;
        hipLaunchKernelGGL(kern, dim3(nblocks(nq, qpp)), dim3(64), 0, s, pts, nodes, cl, ncl, bucket, lt, n, qlist,
                           nq, label, check_labels ? 1 : 0, inv, seed_r, seed_scale, cand_key, cand_pos, revive, first_corr,
                           first_key, C, cs, dup, 0, kMaxCappedPasses, (uint64_t*)nullptr,
                           (const uint32_t*)nullptr, (const uint64_t*)nullptr, (int64_t)0, qpp);
        return;
    }
    // pass 0 over every query, then the open ones compacted into full waves.
    // The wedges of the 2.5D mode are unbounded in z, so their bests tighten
    // early and the per-face node test drops most of what a radius would keep:
    // k_cone_search stays faster there (4.3 against 6.2 ms, 3*10^6 points).
    const int64_t P = (int64_t)g;
    if (cdim == dim)
        hipLaunchKernelGGL(dim == 3 ? (k_cone_first<3>) : (k_cone_first<2>), dim3(g), dim3(64), 0, s, pts, nodes, cl,
                           ncl, bucket, lt, n, inv, seed_r, seed_scale, seed_mul, cand_key, cand_pos, first_corr, first_key, C,
                           cs, dup, split->open_mask, reach);
    else
        hipLaunchKernelGGL(kern, dim3(g), dim3(64), 0, s, pts, nodes, cl, ncl, bucket, lt, n, qlist, nq, label,
                           check_labels ? 1 : 0, inv, seed_r, seed_scale, cand_key, cand_pos, revive, first_corr,
                           first_key, C, cs, dup, 0, 0, split->open_mask, (const uint32_t*)nullptr,
                           (const uint64_t*)nullptr, (int64_t)0, 64);
    if (reach) return;          // late cones: the rounds ask for the rest
    hipLaunchKernelGGL(k_open_count, dim3(nblocks(P + 1)), dim3(kBlock), 0, s, split->open_mask, P, split->cnt);
    exclusive_scan_u32(split->cnt, split->off, P + 1, split->tmp, s);
    hipLaunchKernelGGL(k_open_fill, dim3((unsigned)P), dim3(64), 0, s, split->open_mask, split->off, split->list);
    hipLaunchKernelGGL(kern, dim3(g), dim3(64), 0, s, pts, nodes, cl, ncl, bucket, lt, n,
                       (const int32_t*)split->list, nq, label, check_labels ? 1 : 0, inv, seed_r, seed_scale,
                       cand_key, cand_pos, revive, first_corr, first_key, C, cs, dup, 1, kMaxCappedPasses,
                       (uint64_t*)nullptr, (const uint32_t*)(split->off + P), (const uint64_t*)split->open_mask,
                       split->in_place ? (int64_t)-1 : nq, 64);
}

// Points that k_cone_rest takes at most in a round; a round with more pauses.
// (4096 / 16384, ms per run: clustered 10^4 points 1.50 / 1.06, 2*10^5 2.70 /
// 2.18, 4*10^6 10.6 / 10.1.)
constexpr int64_t kRestFew = 16384;

// listed points one wave each: nq_dev of them; none when they are more than
// `few`
static void cone_rest(const ConeRest& a, const uint32_t* nq_dev, int64_t few, int mode, hipStream_t s)
{
    hipLaunchKernelGGL(k_cone_rest, dim3((unsigned)std::min<int64_t>(a.n, kRestBlocks)), dim3(64), 0, s, a, nq_dev,
                       few, mode);
}

// Late cones in a round, after its minima (k_late_mark).
void launch_late_cones(const ConeRest& a, hipStream_t s)
{
    if (a.n <= 0) return;
    hipLaunchKernelGGL(k_late_mark, dim3((unsigned)((a.n + kLateChunk - 1) / kLateChunk)), dim3(kBlock), 0, s, a.n,
                       a.ids, a.label, (const int32_t*)a.corr, a.corr_key, (const uint64_t*)a.comp1,
                       (const int32_t*)a.reach, a.list, a.C);
    cone_rest(a, &a.C->late, kRestFew, kRestRound, s);
    hipLaunchKernelGGL(k_late_seen, dim3((unsigned)(kRestFew / kBlock)), dim3(kBlock), 0, s, (const int32_t*)a.list,
                       a.ids, a.label, a.corr, (const uint64_t*)a.corr_key, (const uint64_t*)a.comp1,
                       (const int32_t*)a.reach, a.C);
}

void launch_revive(int64_t n, int32_t* corr, hipStream_t s)
{
    if (n > 0) hipLaunchKernelGGL(k_revive, dim3(nblocks(n)), dim3(kBlock), 0, s, n, corr);
}

void launch_leaves(const uint64_t* keys, int64_t n, Cloud* cl, int ncl, int bucket, uint32_t* mark,
                   uint32_t* idx, uint32_t* tmp, int32_t* start, int32_t* of, int32_t* cloud_lf, const Params* P,
                   Counters* C, bool layout, hipStream_t s)
{
    if (n > 0) {
        hipLaunchKernelGGL(k_leaf_marks, dim3(nblocks(n)), dim3(kBlock), 0, s, keys, n, (const Cloud*)cl, ncl,
                           bucket, mark);
        exclusive_scan_u32(mark, idx, n, tmp, s);
        hipLaunchKernelGGL(k_leaf_fill, dim3(nblocks(n)), dim3(kBlock), 0, s, (const uint32_t*)mark,
                           (const uint32_t*)idx, n, start, of);
    }
    hipLaunchKernelGGL(k_cloud_leaves, dim3(1), dim3(1024), 0, s, cl, ncl, (const uint32_t*)mark,
                       (const uint32_t*)idx, n, cloud_lf, P, C, layout ? 1 : 0);
}

void launch_zero_u32(uint32_t* p, int64_t n, hipStream_t s)
{
    if (n > 0) hipLaunchKernelGGL(k_zero_u32, dim3(nblocks(n)), dim3(kBlock), 0, s, p, n);
}

void launch_comp_seed_init(int64_t n, const float4* pts, int32_t* csize, uint32_t* cbox, hipStream_t s)
{
    if (n <= 0) return;
    hipLaunchKernelGGL(k_comp_seed_init, dim3(nblocks(n)), dim3(kBlock), 0, s, n, pts, csize, cbox);
}

// the component search's dispatches over a list of points (nq of them); LATE:
// late points of the cone form (3D)
template <bool LATE>
static void comp_dispatches(int dim, int64_t n, const float4* pts, const Node* nodes, const Cloud* cl, int ncl,
                            int bucket, LeafTable lt, const SplitScratch& sc, const int32_t* list,
                            const uint32_t* nq, const int32_t* label, int32_t* corr, uint64_t* corr_key,
                            uint64_t* comp1, const int32_t* inv, float seed_scale, const float* seed_r, Counters* C,
                            hipStream_t s, hipEvent_t* ev)
{
    const int64_t P = (n + 63) / 64;
    auto kern = dim == 3 ? (bucket == 64 ? k_comp_search<3, 64, false, LATE> : k_comp_search<3, 0, false, LATE>)
                         : (bucket == 16 ? k_comp_search<2, 16, false, false> : k_comp_search<2, 0, false, false>);
    // (2D at its default 64-point leaves runs the runtime-size instance: a
    // <2, 64> instance measured 7% slower on the 2D power-law cloud)
    // pass 0 over the searching points; their open packets' lanes into open_mask
    if (ev) (void)hipEventRecord(ev[0], s);
    if (dim == 3 && n >= kSampleMin) {
        const int64_t gs = std::min<int64_t>((P + kSampleStep - 1) / kSampleStep, kSampleBlocks);
        hipLaunchKernelGGL((k_comp_search<3, 0, true, LATE>), dim3((unsigned)gs), dim3(64), 0, s, pts, nodes, cl, ncl, bucket,
                           lt, list, nq, label, inv, seed_scale, corr, corr_key, comp1, 0, kMaxCappedPasses,
                           (uint64_t*)nullptr, seed_r, (uint64_t*)nullptr, C, 0);
    }
    hipLaunchKernelGGL(kern, dim3((unsigned)std::min<int64_t>(P, kSearchBlocks)), dim3(64), 0, s, pts,
                       nodes, cl, ncl, bucket, lt,
                       list, nq, label, inv, seed_scale, corr, corr_key, comp1, 0, 0,
                       sc.open_mask, seed_r, sc.defer, C, ev != nullptr ? 1 : 0);
    if (ev) (void)hipEventRecord(ev[1], s);
    open_compact(sc.open_mask, P, sc.off, sc.tmp, list, sc.list2, s);
    if (ev) (void)hipEventRecord(ev[2], s);
    hipLaunchKernelGGL(kern, dim3((unsigned)std::min<int64_t>(P, kResumeBlocks)), dim3(64), 0, s, pts,
                       nodes, cl, ncl, bucket, lt,
                       (const int32_t*)sc.list2, (const uint32_t*)(sc.off + P), label, inv, seed_scale, corr,
                       corr_key, comp1, 1, kMaxCappedPasses, (uint64_t*)nullptr, seed_r, sc.defer, C,
                       ev != nullptr ? 1 : 0);
    // the queries the packets handed over, one wave each
    if (sc.defer != nullptr) {
        auto dk = dim == 3 ? k_comp_search_deferred<3, LATE> : k_comp_search_deferred<2, false>;
        hipLaunchKernelGGL(dk, dim3(kDeferBlocks), dim3(64 * kDeferWaves), 0, s, pts, nodes, cl, ncl, lt,
                           (const uint64_t*)sc.defer, label, inv, seed_scale, corr, corr_key, comp1, seed_r, C,
                           ev != nullptr ? 1 : 0);
    }
    if (ev) (void)hipEventRecord(ev[3], s);
}

// A round that too many late points pause (done == 3): their nearest points
// outside their components, by the component search.  It finds the smallest
// edge of every component whose exact candidates may not hold it.  The cones
// would choose the same edge: a point nearer to p within the cone of p's edge
// (p, q) is one of p's component and nearer to q than p is.  In floats that
// last step could fail, so every edge chosen here is checked against its cone
// (k_cone_rest), and one that fails restarts the run with exact cones
// (done == 4).
void launch_late_search(const ConeRest& a, Node* nodes, unsigned long long* visit, int64_t nleaves,
                        bool first, float seed_scale, const SplitScratch& sc, hipStream_t s)
{
    const int64_t n = a.n, P = (n + 63) / 64;
    hipLaunchKernelGGL(k_zero_u32, dim3(1), dim3(kBlock), 0, s, &a.C->done, (int64_t)1);
    hipLaunchKernelGGL(k_zero_u32, dim3(nblocks(2 * P)), dim3(kBlock), 0, s, reinterpret_cast<uint32_t*>(sc.open_mask),
                       2 * P);
    if (first)
        hipLaunchKernelGGL(k_zero_u32, dim3(nblocks(4 * nleaves)), dim3(kBlock), 0, s,
                           reinterpret_cast<uint32_t*>(visit), 4 * nleaves);
    hipLaunchKernelGGL(k_nlab_tree, dim3(nblocks(nleaves)), dim3(kBlock), 0, s, a.label, a.clouds, a.ncl, nleaves,
                       a.lt, nodes, visit, (const Counters*)a.C);
    comp_dispatches<true>(3, n, a.pts, nodes, a.clouds, a.ncl, a.bucket, a.lt, sc, (const int32_t*)a.list, &a.C->late,
                    a.label, a.corr, a.corr_key, a.comp1, a.inv, seed_scale, nullptr, a.C, s, nullptr);
    hipLaunchKernelGGL(k_late_settle, dim3(nblocks(n)), dim3(kBlock), 0, s, (const int32_t*)a.list, a.ids, a.label,
                       a.corr, (const uint64_t*)a.corr_key, (const uint64_t*)a.comp1, sc.list2, a.C);
    ConeRest chk = a;
    chk.list = sc.list2;
    cone_rest(chk, &a.C->late_checks, n, kRestCheck, s);
}

void launch_comp_round(int dim, int64_t n, const float4* pts, const uint32_t* ids, Node* nodes,
                       unsigned long long* visit,
                       const Cloud* cl, int ncl, int64_t nleaves,
                       int bucket, LeafTable lt,
                       const int32_t* label, int32_t* corr, uint64_t* corr_key, uint64_t* comp1, const int32_t* inv,
                       float seed_scale, const SplitScratch& sc, const CompSeed& cs, const NbrList& nb,
                       const int32_t* eu, const int32_t* eround, Counters* C, hipStream_t s, hipEvent_t* ev)
{
    if (n <= 0) return;
    const unsigned g = nblocks(n);
    if (cs.features_on)
        hipLaunchKernelGGL(k_comp_merge, dim3(g), dim3(kBlock), 0, s, n, label, eu, eround, cs.csize, cs.cbox,
                           (const Counters*)C);
    hipLaunchKernelGGL(k_nlab_tree, dim3(nblocks(nleaves)), dim3(kBlock), 0, s, label, cl, ncl, nleaves, lt,
                       nodes, visit, (const Counters*)C);
    const int64_t P = (n + 63) / 64;
    hipLaunchKernelGGL(dim == 3 ? k_comp_keep<kKnn3> : k_comp_keep<kKnn2>, dim3(g), dim3(kBlock), 0, s, n, ids,
                       label, corr, corr_key, comp1, nb,
                       (const Counters*)C);
    hipLaunchKernelGGL(k_comp_prep, dim3(g), dim3(kBlock), 0, s, n, pts, label, corr, corr_key,
                       (const uint64_t*)comp1, (const Node*)nodes, cl, ncl, sc.open_mask, (const Counters*)C);
    open_compact(sc.open_mask, P, sc.off, sc.tmp, nullptr, sc.list, s);
    const uint32_t* nq = sc.off + P;
    const float* seed_r = nullptr;
    if (cs.features_on) {
        hipLaunchKernelGGL(k_comp_features, dim3(g), dim3(kBlock), 0, s, cs.samples != nullptr ? 1 : 0,
                           cs.model != nullptr ? 1 : 0, dim, pts, nodes, cl, ncl, lt,
                           (const int32_t*)sc.list, nq, label, (const uint64_t*)corr_key, (const uint64_t*)comp1,
                           (const int32_t*)cs.csize, (const uint32_t*)cs.cbox, (const Counters*)C, cs.X, cs.LS,
                           cs.nq_keep);
        if (cs.model != nullptr) {
            launch_mlp_infer_dev(cs.model, cs.X, cs.nq_keep + 1, n, cs.Y, s);
            hipLaunchKernelGGL(k_comp_seed, dim3(g), dim3(kBlock), 0, s, (const int32_t*)sc.list,
                               (const uint32_t*)(cs.nq_keep + 1), (const float*)cs.LS, (const float*)cs.Y, cs.R,
                               (const Counters*)C);
            seed_r = cs.R;
        }
    }
    comp_dispatches<false>(dim, n, pts, nodes, cl, ncl, bucket, lt, sc, (const int32_t*)sc.list, nq, label, corr, corr_key,
                    comp1, inv, seed_scale, seed_r, C, s, ev);
    // comp1 now holds every component's edge: the sample log of this round
    if (cs.features_on && cs.samples != nullptr)
        hipLaunchKernelGGL(k_comp_samples, dim3(g), dim3(kBlock), 0, s, (const int32_t*)sc.list,
                           (const uint32_t*)cs.nq_keep, (const float*)cs.X, (const float*)cs.LS, label,
                           (const int32_t*)corr, (const uint64_t*)corr_key, (const uint64_t*)comp1, cs.per_round,
                           cs.cap, cs.samples, C);
}

void launch_knn_first(int dim, int64_t n, const float4* pts, const Node* nodes, const Cloud* cl, int ncl,
                      int bucket, LeafTable lt, const int32_t* inv, int32_t* corr, uint64_t* corr_key,
                      const NbrList& nb, Counters* C, bool collect, hipStream_t s)
{
    if (n <= 0) return;
    int qpp = 64;
    while (qpp > 8 && n < kKnnPackets * qpp) qpp >>= 1;
    const unsigned P = nblocks(n, qpp);
    const int cs = collect ? 1 : 0;
    if (dim == 3)
        hipLaunchKernelGGL(k_knn_first<3>, dim3(P), dim3(64), 0, s, n, pts, nodes, cl, ncl, bucket, lt, inv, corr,
                           corr_key, nb, C, cs, qpp);
    else
        hipLaunchKernelGGL(k_knn_first<2>, dim3(P), dim3(64), 0, s, n, pts, nodes, cl, ncl, bucket, lt, inv, corr,
                           corr_key, nb, C, cs, qpp);
}

void launch_dup_fill(int dim, int64_t n, const int32_t* label, const float4* pts, const int32_t* inv,
                     uint64_t* cand_key, int32_t* cand_pos, int32_t* revive, int32_t* first_corr,
                     uint64_t* first_key, Counters* C, DupState dup, hipStream_t s)
{
    if (n <= 0 || dup.rep == nullptr || dup.npoints <= 0) return;
    hipLaunchKernelGGL(k_dup_reset, dim3((unsigned)std::min<int64_t>(nblocks(dup.ngroups), 256)), dim3(kBlock), 0,
                       s, C, dup);
    const unsigned g = (unsigned)std::min<int64_t>(nblocks(dup.npoints), 1024);
    hipLaunchKernelGGL(k_dup_m2, dim3(g), dim3(kBlock), 0, s, label, pts, C, dup);
    if (dim == 3)
        hipLaunchKernelGGL(k_dup_fill<3>, dim3(g), dim3(kBlock), 0, s, n, label, pts, inv, cand_key, cand_pos,
                           revive, first_corr, first_key, C, dup);
    else
        hipLaunchKernelGGL(k_dup_fill<2>, dim3(g), dim3(kBlock), 0, s, n, label, pts, inv, cand_key, cand_pos,
                           revive, first_corr, first_key, C, dup);
}

void launch_round_init(int64_t n, int32_t* label, int32_t* label2, int32_t* eu, int32_t* corr,
                       uint64_t* corr_key, uint64_t* comp1, uint32_t* comp2, Counters* C, uint32_t target,
                       uint32_t max_rounds, hipStream_t s)
{
    hipLaunchKernelGGL(k_round_init, dim3(nblocks(std::max<int64_t>(n, kWorkKinds * kWorkSlots))), dim3(kBlock), 0, s, n, label,
                       label2, eu, corr, corr_key, comp1, comp2, C, target, max_rounds);
}

void launch_round_begin(Counters* C, hipStream_t s)
{
    hipLaunchKernelGGL(k_round_begin, dim3(1), dim3(1), 0, s, C);
}

void launch_round_end(Counters* C, bool grouped, hipStream_t s, unsigned long long* stamps, uint32_t cap)
{
    hipLaunchKernelGGL(k_round_end, dim3(1), dim3(1), 0, s, C, grouped ? 1 : 0, stamps, cap);
}

void launch_stamp(unsigned long long* at, hipStream_t s)
{
    hipLaunchKernelGGL(k_stamp, dim3(1), dim3(1), 0, s, at);
}

void launch_flag_research(int K, int64_t n, const uint64_t* cand_key, int32_t* list, const int32_t* reach,
                          Counters* C, hipStream_t s)
{
    if (n <= 0) return;
    hipLaunchKernelGGL(k_flag_research, dim3(nblocks(n)), dim3(kBlock), 0, s, K, n, cand_key, list, reach, C);
}

void launch_rank_cones(int dim, int64_t n, const uint64_t* cand_key, const int32_t* cand_pos,
                       const int32_t* qlist, int64_t nq, uint64_t* rkey, int32_t* rpos, uint8_t* cursor,
                       const int32_t* reach, const Counters* C, hipStream_t s)
{
    if (nq <= 0) return;
    hipLaunchKernelGGL(dim == 3 ? k_rank_cones<3> : k_rank_cones<2>, dim3(nblocks(nq)), dim3(kBlock), 0, s, n,
                       cand_key, cand_pos, qlist, nq, rkey, rpos, cursor, reach, C);
}

void launch_round_phase(int phase, int K, int64_t n, const uint32_t* ids, const uint64_t* rkey,
                        const int32_t* rpos, uint8_t* cursor, int32_t* label,
                        int32_t* label2, int32_t* corr,
                        uint64_t* corr_key, uint64_t* comp1, uint32_t* comp2,
                        Counters* C, int32_t* eu, int32_t* ev, float* ed2, int32_t* eround,
                        const CycleState& cy, hipStream_t s)
{
    if (n <= 0) return;
    const unsigned g = nblocks(n);
    switch (phase) {
    case 0:
        hipLaunchKernelGGL(k_round_min, dim3(g), dim3(kBlock), 0, s, K, n, ids, rkey, rpos, cursor,
                           label, corr, corr_key, comp1, C);
        break;
    case 1:
        hipLaunchKernelGGL(k_round_comp2, dim3(g), dim3(kBlock), 0, s, n, ids, label, corr, corr_key, comp1,
                           comp2, C);
        break;
    case 2:
        if (cy.j0) {
            const unsigned gc = (unsigned)std::min<int64_t>(g, 1024);
            hipLaunchKernelGGL(k_cycle_init, dim3((unsigned)((n + kCyChunk - 1) / kCyChunk)), dim3(kBlock), 0, s, n,
                               label, comp1, comp2, cy, C);
            hipLaunchKernelGGL(k_cycle_walk, dim3(gc), dim3(kBlock), 0, s, comp1, comp2, cy, C);
            if (n > kCyWalk) {
                for (int k = 0; k < cy.steps; ++k)
                    hipLaunchKernelGGL(k_cycle_step, dim3(gc), dim3(kBlock), 0, s, comp1, comp2, cy, k, C);
                hipLaunchKernelGGL(k_cycle_mark, dim3(gc), dim3(kBlock), 0, s, cy, C);
                hipLaunchKernelGGL(k_cycle_cut, dim3(gc), dim3(kBlock), 0, s, cy, C);
            }
        }
        hipLaunchKernelGGL(k_round_hook, dim3(nblocks(n, kHookBlock)), dim3(kHookBlock), 0, s, n, ids, label,
                           label2, corr, corr_key, comp1, comp2, C, eu, ev, ed2, eround, cy.j0 ? cy.cut : nullptr);
        break;
    case 3:
        hipLaunchKernelGGL(k_round_flatten, dim3(g), dim3(kBlock), 0, s, n, label, label2, comp1, comp2, C);
        break;
    }
}

void launch_weight(const float* xyz, int dim, const int32_t* eu, const int32_t* ev, int64_t m,
                   double* partial, int nblk, hipStream_t s)
{
    if (dim == 3) hipLaunchKernelGGL(k_weight<3>, dim3(nblk), dim3(kBlock), 0, s, xyz, eu, ev, m, partial);
    else hipLaunchKernelGGL(k_weight<2>, dim3(nblk), dim3(kBlock), 0, s, xyz, eu, ev, m, partial);
}

void launch_cloud_results(const float* xyz, int dim, const Cloud* cl, int ncl, const int32_t* eu,
                          const int32_t* ev, const int32_t* eround, double* weight, int32_t* edges,
                          int32_t* last_round, hipStream_t s)
{
    if (ncl <= 0) return;
    if (dim == 3)
        hipLaunchKernelGGL(k_cloud_results<3>, dim3(ncl), dim3(kBlock), 0, s, xyz, cl, eu, ev, eround, weight,
                           edges, last_round);
    else
        hipLaunchKernelGGL(k_cloud_results<2>, dim3(ncl), dim3(kBlock), 0, s, xyz, cl, eu, ev, eround, weight,
                           edges, last_round);
}

void launch_labels_out(int64_t n, const int32_t* label, const float4* pts, const int32_t* inv,
                       int32_t* out, hipStream_t s)
{
    if (n <= 0) return;
    hipLaunchKernelGGL(k_labels_out, dim3(nblocks(n)), dim3(kBlock), 0, s, n, label, pts, inv, out);
}

void launch_cands_out(int K, int64_t n, const uint64_t* cand_key, const int32_t* inv, int32_t* cand,
                      float* cd2, hipStream_t s)
{
    if (n <= 0) return;
    hipLaunchKernelGGL(k_cands_out, dim3(nblocks(n)), dim3(kBlock), 0, s, K, n, cand_key, inv, cand, cd2);
}

void launch_edge_keys(const int32_t* eu, const int32_t* ev, int64_t m, int bits, uint64_t* keys, hipStream_t s)
{
    if (m <= 0) return;
    hipLaunchKernelGGL(k_edge_keys, dim3(nblocks(m)), dim3(kBlock), 0, s, eu, ev, m, bits, keys);
}

void launch_edges_out(const uint64_t* keys, const uint32_t* idx, const float* ed2, int64_t m, int bits, int32_t* u,
                      int32_t* v, float* d2, hipStream_t s)
{
    if (m <= 0) return;
    hipLaunchKernelGGL(k_edges_out, dim3(nblocks(m)), dim3(kBlock), 0, s, keys, idx, ed2, m, bits, u, v, d2);
}

void launch_cell_grid(const float* resc, int64_t n, int dim, int pstride, const int32_t* geo, int32_t* cell_of,
                      uint64_t* keys, uint32_t* cell_count, hipStream_t s)
{
    if (n <= 0) return;
    hipLaunchKernelGGL(k_cell_grid, dim3(nblocks(n)), dim3(kBlock), 0, s, resc, n, dim, pstride, geo, cell_of,
                       keys, cell_count);
}

}  // namespace emst
