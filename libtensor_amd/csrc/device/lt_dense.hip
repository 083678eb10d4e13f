// Dense contractions (tod_contract2) on FP64 MFMA with every operand read and
// C written at its own strides: no aligned copies.  A tile of up to 16 FM rows
// x 64 columns per workgroup, as in lt_tile.hip (the same staging, products
// and summation order); row, column and k offsets come from dividing the
// composite indices: rows and columns once per tile, the 16 k of a chunk by 16
// threads one chunk ahead, so the loop adds two offsets per element.
// What bounds it at the sizes such calls have (k of some hundreds to
// thousands): the chunk loop's latency and the launch; k ranges are cut into
// parts where the tiles leave CUs idle.  o = 15, v = 45 ring (675 x 675 x
// 675, all three tensors permuted): 27 us, 40 a call, where three copies, a
// product of 64 x 64 tiles and the lists and temporaries of all took 0.43 ms.
#include <hip/hip_runtime.h>
#include <type_traits>
#include "lt_device.h"

namespace lta {
namespace dev {

typedef double double4_t __attribute__((ext_vector_type(4)));
typedef double double2_t __attribute__((ext_vector_type(2)));
typedef const double __attribute__((address_space(1))) gdouble;
typedef double __attribute__((address_space(1))) gout;

namespace {

//! Element offsets of composite index e in the axis' two tensors.
__device__ __forceinline__ void axis_offsets(const dense_axis &x, uint32_t e, uint32_t &o0, uint32_t &o1) {
    o0 = o1 = 0;
#pragma unroll
    for(int i = kDenseMaxOrder - 1; i >= 0; i--) {
        if(i < (int)x.n) {
            const uint32_t q = (__umulhi(e, x.div[i].mul) + e) >> x.div[i].shift;
            const uint32_t r = e - q * x.div[i].d;
            o0 += r * x.s0[i];
            o1 += r * x.s1[i];
            e = q;
        }
    }
}

const int kRow = 18;            // doubles per staged row of 16 k

template<int FM, int KG>
struct dense_smem {
    static constexpr int BM = 16 * FM, BN = 64;
    static constexpr int CH = (BM + BN) * kRow;
    static constexpr int NST = KG * 2 * CH, NRED = KG == 1 ? 0 : KG * BM * BN;
    alignas(16) double ch[NST > NRED ? NST : NRED];
    uint32_t ko[KG][2][2][16];      // byte offsets of a chunk's 16 k in A and B, two chunks per group
    uint32_t mo[2][BM], no[2][BN];  // byte offsets in A (B), element offsets in C of the tile's rows (columns)
};

//! Adds x to (or puts it at) the element of C at `off`.
__device__ __forceinline__ void dense_write(const dense_args &A, uint32_t off, double x) {
    gout *p = (gout *)A.c + size_t(off);
    *p = A.zero ? x : x + *p;
}

template<int FM, int KG>
__device__ __forceinline__ void dense_body(const dense_args &A, uint32_t m0, uint32_t n0, uint32_t c0,
    uint32_t nchunk, gout *part, dense_smem<FM, KG> &sm) {

    typedef dense_smem<FM, KG> S;
    constexpr int BM = S::BM, BN = S::BN, E = FM + 4;
    const int g = __builtin_amdgcn_readfirstlane(threadIdx.x >> 8);
    const int wave = __builtin_amdgcn_readfirstlane((threadIdx.x >> 6) & 3);
    const int tid = threadIdx.x & 255, lane = tid & 63;
    const int lr = lane & 15, lg = lane >> 4;
    const int hi = tid >> 4, lo = tid & 15;
    const uint32_t mrem = A.m.ext - m0, nrem = A.n.ext - n0, K = A.k.ext;
    const bool arf = A.rows_fast & 1, brf = A.rows_fast & 2;
    const int ra = arf ? lo : hi, ka = arf ? hi : lo, rb = brf ? lo : hi, kb = brf ? hi : lo;

    // offsets of the tile's rows and columns (past the extents: the first's)
    if(threadIdx.x < 64 && threadIdx.x < BM) {
        uint32_t o, p;
        axis_offsets(A.m, m0 + (threadIdx.x < mrem ? threadIdx.x : 0), o, p);
        sm.mo[0][threadIdx.x] = 8u * o;
        sm.mo[1][threadIdx.x] = p;
    } else if(threadIdx.x >= 64 && threadIdx.x < 128) {
        const uint32_t c = threadIdx.x - 64;
        uint32_t o, p;
        axis_offsets(A.n, n0 + (c < nrem ? c : 0), o, p);
        sm.no[0][c] = 8u * o;
        sm.no[1][c] = p;
    }
    // k offsets of chunk c (relative to the part; past its end: its last one)
    auto offsets = [&](uint32_t c, int slot) {
        if(tid < 16) {
            uint32_t oa, ob;
            axis_offsets(A.k, min(16 * (c0 + min(c, nchunk - 1)) + tid, K - 1), oa, ob);
            sm.ko[g][slot][0][tid] = 8u * oa;
            sm.ko[g][slot][1][tid] = 8u * ob;
        }
    };
    double4_t acc[FM];
#pragma unroll
    for(int i = 0; i < FM; i++) acc[i] = double4_t{0.0, 0.0, 0.0, 0.0};

    double v[E];
    double *base = sm.ch + g * 2 * S::CH;
    uint32_t c = g;                        // the chunk to load
    int slot = 0;
    offsets(c, 0);
    __syncthreads();
    uint32_t off[E];                       // of this thread's rows of A and columns of B
#pragma unroll
    for(int e = 0; e < E; e++) off[e] = e < FM ? sm.mo[0][ra + 16 * e] : sm.no[0][rb + 16 * (e - FM)];
    const __attribute__((address_space(1))) char *pa = (const __attribute__((address_space(1))) char *)A.a;
    const __attribute__((address_space(1))) char *pb = (const __attribute__((address_space(1))) char *)A.b;
    // As the step of the stacked kernels: products of the staged chunk, the
    // next chunk's loads and LDS writes between them.
    auto step = [&](auto mc, int rtog, int wtog) {
        constexpr bool mult = decltype(mc)::value;
        const uint32_t xa = sm.ko[g][slot][0][ka], xb = sm.ko[g][slot][1][kb];
        double *wa = base + wtog + ra * kRow + ka, *wb = base + wtog + rb * kRow + kb;
        const double *bp = base + rtog + (BM + 16 * wave + lr) * kRow + 4 * lg;
        const double *ap = base + rtog + lr * kRow + 4 * lg;
        double2_t b0, b1, x0, x1, y0, y1;
        if constexpr(mult) {
            b0 = *(const double2_t *)bp; b1 = *(const double2_t *)(bp + 2);
            x0 = *(const double2_t *)ap; x1 = *(const double2_t *)(ap + 2);
        }
        offsets(c + KG, slot ^ 1);
        auto product = [&](int h) {
            if(h % 2 == 0 && h / 2 + 1 < FM) {
                y0 = *(const double2_t *)(ap + 16 * (h / 2 + 1) * kRow);
                y1 = *(const double2_t *)(ap + 16 * (h / 2 + 1) * kRow + 2);
            }
            const int i = h / 2;
            const double2_t x = h % 2 ? x1 : x0, b = h % 2 ? b1 : b0;
            acc[i] = __builtin_amdgcn_mfma_f64_16x16x4f64(x.x, b.x, acc[i], 0, 0, 0);
            acc[i] = __builtin_amdgcn_mfma_f64_16x16x4f64(x.y, b.y, acc[i], 0, 0, 0);
            if(h % 2) { x0 = y0; x1 = y1; }
        };
#pragma unroll
        for(int h = 0; h < FM; h++) {
#pragma unroll
            for(int e = 2 * h * E / FM; e < 2 * (h + 1) * E / FM; e++)
                if(e < E) v[e] = *(gdouble *)(e < FM ? pa + size_t(off[e] + xa) : pb + size_t(off[e] + xb));
            if constexpr(mult) { product(h); __builtin_amdgcn_sched_barrier(0); }
        }
        // past the extent, and past the part, both operands are zero
        if(16 * (c0 + c) + 16 > K || c >= nchunk) {
            const bool la = c < nchunk && 16 * (c0 + c) + ka < K, lb = c < nchunk && 16 * (c0 + c) + kb < K;
#pragma unroll
            for(int e = 0; e < E; e++) v[e] = (e < FM ? la : lb) ? v[e] : 0.0;
        }
#pragma unroll
        for(int h = FM; h < 2 * FM; h++) {
            if constexpr(mult) product(h);
#pragma unroll
            for(int e = (h - FM) * E / FM; e < (h - FM + 1) * E / FM; e++) {
                if(e < FM) wa[16 * e * kRow] = v[e] * A.d;
                else wb[16 * e * kRow] = v[e];
            }
            if constexpr(mult) __builtin_amdgcn_sched_barrier(0);
        }
        c += KG;
        slot ^= 1;
        __syncthreads();
    };
    step(std::false_type(), 0, 0);
    const uint32_t nstep = (nchunk + KG - 1) / KG;
    int tog = 0;
    if(uint32_t(16 * wave) < nrem) {
        for(uint32_t it = 0; it < nstep; it++, tog = S::CH - tog) step(std::true_type(), tog, S::CH - tog);
    } else {
        for(uint32_t it = 0; it < nstep; it++, tog = S::CH - tog) step(std::false_type(), tog, S::CH - tog);
    }

    if(KG == 1) {
#pragma unroll
        for(int i = 0; i < FM; i++)
#pragma unroll
            for(int q = 0; q < 4; q++) {
                const uint32_t row = 16 * i + lg + 4 * q, col = 16 * wave + lr;
                if(part) part[((i * 4 + q) * 4 + wave) * 64 + lane] = acc[i][q];
                else if(row < mrem && col < nrem) dense_write(A, sm.mo[1][row] + sm.no[1][col], acc[i][q]);
            }
        return;
    }
    double *red = sm.ch;
#pragma unroll
    for(int i = 0; i < FM; i++)
#pragma unroll
        for(int q = 0; q < 4; q++)
            red[g * BM * BN + ((i * 4 + q) * 4 + wave) * 64 + lane] = acc[i][q];
    __syncthreads();
    for(int e = threadIdx.x; e < BM * BN; e += 256 * KG) {
        double x = red[e];
#pragma unroll
        for(int q = 1; q < KG; q++) x += red[q * BM * BN + e];
        const int l = e & 63, w = (e >> 6) & 3, q = (e >> 8) & 3, i = e >> 10;
        const uint32_t row = 16 * i + (l >> 4) + 4 * q, col = 16 * w + (l & 15);
        if(part) part[e] = x;
        else if(row < mrem && col < nrem) dense_write(A, sm.mo[1][row] + sm.no[1][col], x);
    }
}

template<int FM, int KG, int FA>
__device__ __forceinline__ void dense_height(const dense_args &A, uint32_t m0, uint32_t n0, uint32_t c0,
    uint32_t nchunk, gout *part, char *smem) {
    if(FA == 1 || A.m.ext - m0 > 16 * (FA - 1))
        dense_body<FA, KG>(A, m0, n0, c0, nchunk, part, *(dense_smem<FA, KG> *)smem);
    else dense_height<FM, KG, (FA > 1 ? FA - 1 : 1)>(A, m0, n0, c0, nchunk, part, smem);
}

} // unnamed namespace

//! Workgroup (x, y): tile x of C (column tiles of a row together), part y of k.
template<int FM, int KG, int OCC>
__global__ void __launch_bounds__(256 * KG) __attribute__((amdgpu_waves_per_eu(OCC)))
gemm_dense_kernel(dense_args A, uint32_t ntn, double *parts) {
    __shared__ __attribute__((aligned(16))) char smem[sizeof(dense_smem<FM, KG>)];
    const uint32_t tm = blockIdx.x / ntn, tn = blockIdx.x - tm * ntn;
    const uint32_t nch = (A.k.ext + 15) / 16, np = gridDim.y;
    const uint32_t c0 = uint32_t(uint64_t(nch) * blockIdx.y / np);
    const uint32_t c1 = uint32_t(uint64_t(nch) * (blockIdx.y + 1) / np);
    gout *part = np > 1 ? (gout *)parts + (size_t(blockIdx.x) * np + blockIdx.y) * (1024 * FM) : (gout *)0;
    dense_height<FM, KG, FM>(A, tm * (16 * FM), tn * 64, c0, c1 - c0, part, smem);
}

//! C of the tiles whose k range was cut: the parts added in order.
__global__ void __launch_bounds__(256)
dense_sum_kernel(dense_args A, uint32_t ntn, const double *__restrict__ parts, uint32_t np, uint32_t fm) {
    const uint32_t tm = blockIdx.x / ntn, tn = blockIdx.x - tm * ntn;
    const uint32_t e = blockIdx.y * 256 + threadIdx.x;
    const uint32_t l = e & 63, w = (e >> 6) & 3, v = (e >> 8) & 3, i = e >> 10;
    const uint32_t row = tm * (16 * fm) + 16 * i + (l >> 4) + 4 * v, col = tn * 64 + 16 * w + (l & 15);
    if(row >= A.m.ext || col >= A.n.ext) return;
    const double *p = parts + size_t(blockIdx.x) * np * (1024 * fm) + e;
    double x = p[0];
    for(uint32_t q = 1; q < np; q++) x += p[size_t(q) * (1024 * fm)];
    uint32_t t, ro, co;
    axis_offsets(A.m, row, t, ro);
    axis_offsets(A.n, col, t, co);
    dense_write(A, ro + co, x);
}

void dense_tile_shape(int cfg, uint32_t &bm, uint32_t &bn) {
    bm = cfg == DENSE_16x64_G4 ? 16 : cfg == DENSE_32x64_G4 ? 32 : 64;
    bn = 64;
}

hipError_t launch_gemm_dense(int cfg, const dense_args &a, uint32_t nparts, double *parts,
    hipStream_t s) {
    uint32_t bm, bn;
    dense_tile_shape(cfg, bm, bn);
    const uint32_t ntm = (a.m.ext + bm - 1) / bm, ntn = (a.n.ext + bn - 1) / bn;
    if(uint64_t(ntm) * ntn >= (uint64_t(1) << 31) || nparts < 1 || nparts > 65535) return hipErrorInvalidValue;
    const dim3 grid(ntm * ntn, nparts);
    switch(cfg) {
    case DENSE_16x64_G4:
        hipLaunchKernelGGL((gemm_dense_kernel<1, 4, 4>), grid, dim3(1024), 0, s, a, ntn, parts); break;
    case DENSE_32x64_G4:
        hipLaunchKernelGGL((gemm_dense_kernel<2, 4, 4>), grid, dim3(1024), 0, s, a, ntn, parts); break;
    case DENSE_64x64_G1:
        hipLaunchKernelGGL((gemm_dense_kernel<4, 1, 4>), grid, dim3(256), 0, s, a, ntn, parts); break;
    case DENSE_64x64_G2:
        hipLaunchKernelGGL((gemm_dense_kernel<4, 2, 4>), grid, dim3(512), 0, s, a, ntn, parts); break;
    default: return hipErrorInvalidValue;
    }
    hipError_t e = hipGetLastError();
    if(e != hipSuccess || nparts == 1) return e;
    hipLaunchKernelGGL(dense_sum_kernel, dim3(ntm * ntn, bm / 4), dim3(256), 0, s, a, ntn, parts,
        nparts, bm / 16);
    return hipGetLastError();
}

} // namespace dev
} // namespace lta
