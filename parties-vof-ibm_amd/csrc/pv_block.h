// pv_block.h -- block-level helpers of the fused solver kernels (pv_pcg.hip,
// pv_cg.hip): 256-thread blocks that each own a band of rows.
//
// Scalars of a Krylov iteration (alpha, beta, stop tests) are never written
// by one block and read by another inside one kernel.  Each block stores one
// partial sum per reduction; the next kernel's blocks all re-add those few
// hundred partials in the same order, so every block holds bit-identical
// scalars and no one-block scalar kernel sits between the sweeps.
#ifndef PV_BLOCK_H
#define PV_BLOCK_H
#include <hip/hip_runtime.h>

#define NTH 256

// A barrier that orders LDS alone: loads from memory stay in flight across it.
__device__ __forceinline__ void lds_barrier()
{
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
}

// This thread's shares of up to three partial sums: sa = sum of pa[b] over
// b = t, t + NTH, ... < na in increasing b (likewise sb, sc).  The partials
// are loaded in batches of PVB per array, all loads of a batch in flight
// before its first add (one memory latency per batch, not one per partial);
// an array with n = 0 is not read.
#define PVB 4
__device__ __forceinline__ void thread_sums(const double *pa, int na, const double *pb, int nb, const double *pc,
                                            int nc, double &sa, double &sb, double &sc)
{
    const int t = threadIdx.x, n = max(na, max(nb, nc));
    sa = sb = sc = 0.0;
    for (int b0 = t; b0 < n; b0 += PVB * NTH) {
        double va[PVB], vb[PVB], vc[PVB];
#pragma unroll
        for (int k = 0; k < PVB; k++) {
            const int b = b0 + k * NTH;
            va[k] = vb[k] = vc[k] = 0.0;
            if (na > 0) va[k] = pa[min(b, na - 1)];
            if (nb > 0) vb[k] = pb[min(b, nb - 1)];
            if (nc > 0) vc[k] = pc[min(b, nc - 1)];
        }
#pragma unroll
        for (int k = 0; k < PVB; k++) {
            const int b = b0 + k * NTH;
            if (b < na) sa += va[k];
            if (b < nb) sb += vb[k];
            if (b < nc) sc += vc[k];
        }
    }
}

// v of lane t + W, for the lanes t < W of the first 2 W lanes (others: any
// value).  Lane moves in the vector unit: two for a double, where a shuffle
// through LDS costs an LDS round trip.
template <int W> __device__ __forceinline__ unsigned lane_down32(unsigned v)
{
    if constexpr (W == 32) return __builtin_amdgcn_permlane32_swap(v, v, false, false)[1];
    else if constexpr (W == 16) return __builtin_amdgcn_permlane16_swap(v, v, false, false)[1];
    else return __builtin_amdgcn_mov_dpp(v, 0x100 | W, 0xf, 0xf, true);     // row_shl:W
}
template <int W> __device__ __forceinline__ double lane_down(double v)
{
    const unsigned long long b = __builtin_bit_cast(unsigned long long, v);
    const unsigned lo = lane_down32<W>((unsigned)b), hi = lane_down32<W>((unsigned)(b >> 32));
    return __builtin_bit_cast(double, ((unsigned long long)hi << 32) | lo);
}
__device__ __forceinline__ double lane_first(double v)
{
    const unsigned long long b = __builtin_bit_cast(unsigned long long, v);
    const unsigned lo = __builtin_amdgcn_readfirstlane((unsigned)b), hi = __builtin_amdgcn_readfirstlane((unsigned)(b >> 32));
    return __builtin_bit_cast(double, ((unsigned long long)hi << 32) | lo);
}
// lane 0: the sum over the wavefront, halving (v_t + v_{t + 32}, + 16, ... + 1)
__device__ __forceinline__ double wave_sum(double v)
{
    v += lane_down<32>(v);
    v += lane_down<16>(v);
    v += lane_down<8>(v);
    v += lane_down<4>(v);
    v += lane_down<2>(v);
    v += lane_down<1>(v);
    return v;
}
// the block's sum of the NTH values in sh, halving (s_t + s_{t + 128}, + 64,
// ... + 1); every wavefront forms it for itself, so one barrier (before, by
// the caller) is all it takes.  Every CG kernel starts with such a sum and on
// small grids little else is on its critical path: with a barrier a halving
// (ten in all) and shuffles through LDS a ten-step run at 96 x 96 took
// 30.1 ms, with these 27.8.
__device__ __forceinline__ double tree_sum(const double *sh)
{
    static_assert(NTH == 256, "four values a lane");
    const int l = threadIdx.x & 63;
    return lane_first(wave_sum((sh[l] + sh[l + 128]) + (sh[l + 64] + sh[l + 192])));
}

// Sum of n partials, same order in every block; all threads get the result.
__device__ __forceinline__ double block_sum(const double *part, int n, double *sh)
{
    const int t = threadIdx.x;
    double s, u0, u1;
    thread_sums(part, n, nullptr, 0, nullptr, 0, s, u0, u1);
    sh[t] = s;
    __syncthreads();
    const double r = tree_sum(sh);
    __syncthreads();
    return r;
}

// The same in a workgroup of more than NTH threads: the first NTH add.
__device__ __forceinline__ double block_sum_wide(const double *part, int n, double *sh)
{
    if (threadIdx.x < NTH) {
        double s, u0, u1;
        thread_sums(part, n, nullptr, 0, nullptr, 0, s, u0, u1);
        sh[threadIdx.x] = s;
    }
    __syncthreads();
    const double r = tree_sum(sh);
    __syncthreads();
    return r;
}

// Two sums of partials in one pass, each added in exactly block_sum's order;
// sh holds 2 * NTH doubles.
__device__ __forceinline__ void block_sum2(const double *pa, int na, const double *pb, int nb, double *sh,
                                           double &ra, double &rb)
{
    const int t = threadIdx.x;
    double sa, sb, u;
    thread_sums(pa, na, pb, nb, nullptr, 0, sa, sb, u);
    sh[t] = sa;
    sh[NTH + t] = sb;
    __syncthreads();
    ra = tree_sum(sh);
    rb = tree_sum(sh + NTH);
    __syncthreads();
}

// Three sums of partials in one pass (the loads of all three in flight
// together), each added in exactly block_sum's order; sh holds 3 * NTH
// doubles.
__device__ __forceinline__ void block_sum3(const double *pa, int na, const double *pb, int nb, const double *pc,
                                           int nc, double *sh, double &ra, double &rb, double &rc)
{
    const int t = threadIdx.x;
    double sa, sb, s3;
    thread_sums(pa, na, pb, nb, pc, nc, sa, sb, s3);
    sh[t] = sa;
    sh[NTH + t] = sb;
    sh[2 * NTH + t] = s3;
    __syncthreads();
    ra = tree_sum(sh);
    rb = tree_sum(sh + NTH);
    rc = tree_sum(sh + 2 * NTH);
    __syncthreads();
}

// Block total of v (within each wavefront, then the 4 wave sums in order) -> part[slot].
__device__ __forceinline__ void block_store_partial(double v, double *part, int slot, double *sh)
{
    const int t = threadIdx.x;
    v = wave_sum(v);
    if ((t & 63) == 0) sh[t >> 6] = v;
    __syncthreads();
    if (t == 0) {
        double s = sh[0];
        for (int w = 1; w < NTH / 64; w++) s += sh[w];
        part[slot] = s;
    }
    __syncthreads();
}

// Workgroups are dealt to the 8 XCDs round robin (block b runs on XCD b % 8).
// Give each XCD a contiguous run of bands (or tiles, in row-major order) so
// the data a band's stencil shares with its neighbours stays in that XCD's
// L2: XCD x owns q + (x < rem) consecutive indices from x q + min(x, rem),
// q = nblocks / 8, rem = nblocks % 8 (a bijection on [0, nblocks)).
__device__ __forceinline__ int xcd_band(int b, int nblocks)
{
    const int x = b & 7, q = nblocks >> 3, rem = nblocks & 7;
    return x * q + (x < rem ? x : rem) + (b >> 3);
}
#endif
