// Workgroup-tiled FP64 MFMA GEMM over stacks (C blocks that share their B
// operands, rows concatenated; lt_device.h: tile_stack).
//
// A workgroup computes a tile of up to 16 FM rows x 16 NW columns: KG groups of
// NW waves take the 16-k chunks of the stack's pair list in turn, each wave
// multiplies one 16-column strip against all rows of the tile, and the groups'
// partial tiles are added in LDS in group order (fixed summation order, one
// writer per C element).  A group stages its chunk in two LDS buffers, rows of
// 16 k.
//
// What bounds it: on gfx950 a v_mfma_f64_16x16x4f64 keeps its SIMD for 64
// cycles, and no vector instruction of any wave issues meanwhile (measured:
// products alone 77 TFLOP/s whatever the waves per SIMD; every vector
// instruction between them adds its 4 cycles).  So the loop holds as few of
// them as it can: addresses move on in scalar registers, the accumulators stay
// in place (in architectural registers: kernels whose accumulators the compiler
// copied to and from the accumulation registers in every step reached 48), and
// loads and LDS writes are spread between the products.  The rows and columns
// a chunk brings in are loaded once per workgroup in runs of 128 bytes, in
// either operand layout.  Measured against the kernels that load
// fragments straight from memory (o, v: one ring contraction): o = 29, v = 131
// in one block 3.48 to 2.16 ms a call, o = 48, v = 240 in uneven blocks 85.6 to
// 58.1 ms (53 TFLOP/s).
//
// What is left is loading: a wave's load of 64 x 8 bytes takes 17 to 19 cycles
// of its CU, and rows that are not whole cache lines come twice from the L2
// cache.  Eight waves over 128 columns share the rows of A (7 loads a thread
// and chunk for 24 products instead of 10): 96 x 128 instead of 96 x 64 tiles,
// the same rings 2.13 to 1.98 and 58.9 to 56.7 ms.
//
// Where the tiles of a launch are too few to keep 256 CUs evenly busy, their
// chunk sequences are cut into parts and a second kernel adds the parts'
// partial tiles in order: pp-ladder o = 40, v = 200 (335 tiles of 64 rows)
// 201 to 160 us, the first product of the quadratic CCD term (72 tiles)
// 63 to 20 us.
#include <hip/hip_runtime.h>
#include <type_traits>
#include "lt_device.h"

namespace lta {
namespace dev {

typedef double double4_t __attribute__((ext_vector_type(4)));
typedef double double2_t __attribute__((ext_vector_type(2)));
typedef const double __attribute__((address_space(1))) gdouble;

namespace {

// The lists are reached through pointers read from memory, which the compiler
// takes for generic ones: their address spaces are stated, so that the pair
// descriptors come by scalar loads and all bookkeeping stays in scalar
// registers (FP64 matrix instructions and vector instructions share the SIMD:
// every vector instruction takes its cycles from the products).
typedef const stack_pair __attribute__((address_space(4))) cpair;
typedef const tile_stack __attribute__((address_space(4))) cstack;
typedef const stack_arow __attribute__((address_space(1))) garow;
typedef const stack_crow __attribute__((address_space(1))) gcrow;
typedef double __attribute__((address_space(1))) gout;
typedef const int32_t __attribute__((address_space(1))) gint;
typedef const char __attribute__((address_space(1))) gchar;

//! n / d of a fastdiv (mul, shift).
__device__ __forceinline__ uint32_t tdiv(uint32_t n, uint32_t mul, uint32_t shift) {
    return (__umulhi(n, mul) + n) >> shift;
}

__device__ __forceinline__ uint32_t uniform(uint32_t x) { return __builtin_amdgcn_readfirstlane(x); }

//! B read through offset tables that are not linear in two index groups.
__device__ __forceinline__ bool tabled(cpair *sp) {
    return sp->noff && !(sp->flags & kPairOffArith);
}

struct row_src {
    double d;
    uint32_t off, lda;
};

//! Position in a stack's chunk sequence (16 k each): chunk c of pair p, of
//! extent k, whose tables are in ring slot `slot`; `left` chunks of the
//! tile's part of the sequence from here on.
struct chunk_pos {
    uint32_t p, c, k, slot, left;
    bool valid;
};

//! Moves `by` chunks on; past the part's last chunk the position stays and
//! valid becomes false, so that a load issued from it stays in bounds.
__device__ __forceinline__ chunk_pos chunk_advance(cpair *pairs, const chunk_pos &u, uint32_t by) {
    chunk_pos r = u;
    r.valid = u.valid && by < u.left;
    if(!r.valid) return r;
    r.left -= by;
    r.c += by;
    while(16 * r.c >= r.k) {
        r.c -= (r.k + 15) >> 4;
        r.k = pairs[++r.p].k;
    }
    if(r.p != u.p) r.slot = u.slot ^ 1;
    return r;
}

//! Where a tile's rows come from and go to: the row tables of a stack.
struct stack_rows {
    cpair *pairs;
    garow *arow;
    gcrow *crow;
    uint32_t astride;
    __device__ __forceinline__ row_src row(uint32_t p, uint32_t r) const {
        garow *e = arow + (size_t(p) * astride + r);
        row_src s;
        s.d = e->d; s.off = e->off; s.lda = e->lda;
        return s;
    }
    __device__ __forceinline__ void write(uint32_t r, uint32_t col, double x) const {
        gcrow *cr = crow + r;
        gout *cp = (gout *)(uintptr_t)cr->c + col;
        *cp = cr->zero ? x : x + *cp;
    }
};

//! A tile and its part of the chunk sequence: `count` chunks from chunk c of
//! pair p on.  part: where the tile's partial sums go (fragment order), or
//! null: they are all there is and go to C.
struct tile_part {
    uint32_t m0, n0, mrem, nrem;
    uint32_t p, c, count;
    gout *part;
};

} // unnamed namespace

static const int kTileRow = 18;     // doubles per staged row of 16 k (144 bytes: b128 reads of 16 rows use every bank once)

//! NW: waves to a group, 16 columns each.  16 NW / 4 rows are staged at a time:
//! PA passes over the rows of A (the last one may go past them), four over B's.
template<int FM, int KG, int NW>
struct tile_smem {
    static constexpr int BM = 16 * FM, BN = 16 * NW, RP = 4 * NW;
    static constexpr int PA = (BM + RP - 1) / RP, RA = PA * RP;
    static constexpr int CH = (RA + BN) * kTileRow;      // one staged chunk: A rows, then B columns
    static constexpr int NST = KG * 2 * CH, NRED = KG == 1 ? 0 : KG * BM * BN;
    alignas(16) double ch[NST > NRED ? NST : NRED];
    // tables of two pairs per group: scales, offsets and strides of
    // the rows of A, offsets of the columns of B
    double rd[KG][2][RA];
    uint32_t ro[KG][2][RA];
    uint32_t rl[KG][2][RA];
    uint32_t cn[KG][2][BN];
};

template<int FM, int KG, int NW>
__device__ __forceinline__ void tile_body(const stack_rows &src, const tile_part &tp, tile_smem<FM, KG, NW> &sm) {

    typedef tile_smem<FM, KG, NW> S;
    constexpr int BM = S::BM, BN = S::BN, RP = S::RP, PA = S::PA, GT = 64 * NW;
    const int g = __builtin_amdgcn_readfirstlane(threadIdx.x / GT);
    const int wave = __builtin_amdgcn_readfirstlane((threadIdx.x >> 6) % NW);
    const int tid = threadIdx.x % GT, lane = tid & 63;
    const int lr = lane & 15, lg = lane >> 4;
    const int hi = (tid >> 4) & 15, lo = tid & 15, up = (tid >> 4) & 16;
    const int hr = (((hi & 1) << 3) | (hi >> 1)) + up;  // as a row: rows 8 apart side by side (their LDS banks differ)
    const int lw = lo + up;                             // row of the threads along rows

    const uint32_t m0 = tp.m0, n0 = tp.n0, mrem = tp.mrem, nrem = tp.nrem, nchunk = tp.count;
    cpair *pairs = src.pairs;

    double4_t acc[FM];
#pragma unroll
    for(int i = 0; i < FM; i++) acc[i] = double4_t{0.0, 0.0, 0.0, 0.0};

    if(nchunk > 0) {
        // rows / column of the pair tables this thread stages (past the extent: the first one)
        const uint32_t trow = uint32_t(tid) < mrem ? m0 + tid : m0;
        const uint32_t tc = uint32_t(tid) % BN, tcol = tc < nrem ? n0 + tc : n0;
        auto info_load = [&](uint32_t p, row_src &ar, uint32_t &cn) {
            if(tid < S::RA) ar = src.row(p, trow);
            if(tid >= GT - BN) {
                cpair *sp = pairs + p;
                if(tabled(sp)) cn = 8u * uint32_t(((gint *)(uintptr_t)sp->noff)[tcol]);
                else {
                    const uint32_t q = tdiv(tcol, sp->nd.mul, sp->nd.shift);
                    cn = 8u * (q * uint32_t(sp->ns0) + (tcol - q * sp->nd.d) * uint32_t(sp->ns1));
                }
            }
        };
        auto info_store = [&](int slot, const row_src &ar, uint32_t cn) {
            if(tid < S::RA) {
                sm.rd[g][slot][tid] = ar.d;
                sm.ro[g][slot][tid] = ar.off;
                sm.rl[g][slot][tid] = ar.lda;
            }
            if(tid >= GT - BN) sm.cn[g][slot][tc] = cn;
        };

        // The group's next chunks: n1 to be loaded, n2 whose pair's tables
        // come next.  A group without a chunk keeps an in-bounds position on
        // the first one and multiplies zeros.
        chunk_pos first;
        first.p = tp.p; first.c = tp.c; first.k = pairs[tp.p].k; first.slot = 0;
        first.left = nchunk; first.valid = true;
        chunk_pos n1 = chunk_advance(pairs, first, g);
        chunk_pos n2 = chunk_advance(pairs, n1, KG);
        {
            row_src ar; uint32_t cq = 0;
            info_load(n1.p, ar, cq);
            info_store(n1.slot, ar, cq);
        }
        __syncthreads();

        // Addresses of this thread's elements of the last chunk loaded: byte
        // offsets of rows (A) and columns (B) from uniform bases, which move
        // on from chunk to chunk.
        uint32_t ao[PA], bo[4], kr = 0;
        uint32_t abase = 0, bbase = 0;     // bytes from the pair's A and B
        double v[PA + 4];                  // the chunk on its way
        uint32_t cur = 0xffffffffu;        // pair of the addresses
        uint32_t fl = 0, bstep = 0;        // its flags (kTab: B through offset tables), step of B from chunk to chunk
        const gchar *pa = 0, *pb = 0, *qa = 0, *qb = 0;
        const uint32_t kTab = 0x80000000u;
        // places of the thread's elements in an LDS buffer, by mapping: rows
        // (columns) adjacent in memory run along 16 threads, else k does
        const int a0 = hr * kTileRow + lo, a1 = lw * kTileRow + hi;

        // Addresses from the pair tables, k past the extent on its last element.
        auto locate = [&](cpair *sp, const chunk_pos &n) {
            const uint32_t K = n.k;
            const bool akm = (fl & kPairAKMajor) != 0, bnf = (fl & kPairBNFast) != 0;
            const int ra = akm ? lw : hr, rb = bnf ? lw : hr;
            const uint32_t kac = min(16 * n.c + (akm ? hi : lo), K - 1), kbc = min(16 * n.c + (bnf ? hi : lo), K - 1);
#pragma unroll
            for(int j = 0; j < PA; j++)
                ao[j] = sm.ro[g][n.slot][ra + RP * j] + 8u * (akm ? kac * sm.rl[g][n.slot][ra + RP * j] : kac);
            uint32_t ko;
            if(fl & kTab) ko = 8u * uint32_t(((gint *)(uintptr_t)sp->koff)[kbc]);
            else {
                const uint32_t q = tdiv(kbc, sp->kd.mul, sp->kd.shift);
                kr = kbc - q * sp->kd.d;
                ko = 8u * (q * uint32_t(sp->ks0) + kr * uint32_t(sp->ks1));
            }
#pragma unroll
            for(int j = 0; j < 4; j++) bo[j] = ko + sm.cn[g][n.slot][rb + RP * j];
            abase = bbase = 0;
        };
        // Addresses of chunk n.  Within a pair only the uniform bases move on
        // (by KG chunks); a pair's first and last chunk (and a pair read
        // through offset tables) locate the addresses anew.
        auto seek = [&](const chunk_pos &n) {
            cpair *sp = pairs + n.p;
            if(n.p != cur) {
                cur = n.p;
                fl = sp->flags | (tabled(sp) ? kTab : 0u);
                bstep = uint32_t(128 * KG) * uint32_t(sp->ks1);
                pa = (const gchar *)(uintptr_t)sp->a;
                pb = (const gchar *)(uintptr_t)sp->b;
                locate(sp, n);
            } else if(16 * n.c + 16 > n.k || (fl & kTab)) {
                locate(sp, n);
            } else if(n.valid) {
                if(fl & kPairAKMajor) {
#pragma unroll
                    for(int j = 0; j < PA; j++) ao[j] += 128u * KG * sm.rl[g][n.slot][lw + RP * j];
                }
                abase += (fl & kPairAKMajor) ? 0u : 128u * KG;
                bbase += (fl & kPairOffArith) ? 0u : bstep;
                if(fl & kPairOffArith) {
                    // k = q kd + kr moves on by 16 KG = dq kd + dr
                    const uint32_t dq = tdiv(16u * KG, sp->kd.mul, sp->kd.shift), dr = 16u * KG - dq * sp->kd.d;
                    uint32_t d = 8u * (dq * uint32_t(sp->ks0) + dr * uint32_t(sp->ks1));
                    kr += dr;
                    const bool wrap = kr >= sp->kd.d;
                    kr = wrap ? kr - sp->kd.d : kr;
                    d = wrap ? d + 8u * uint32_t(sp->ks0) - 8u * sp->kd.d * uint32_t(sp->ks1) : d;
#pragma unroll
                    for(int j = 0; j < 4; j++) bo[j] += d;
                }
            }
            qa = pa + uniform(abase);
            qb = pb + uniform(bbase);
        };
        // Element e of the thread (rows of A, then columns of B): its load,
        // and its way into an LDS buffer (A scaled).
        constexpr int E = PA + 4;
        double sc[PA];
        auto load = [&](int e) {
            if(e < PA) v[e] = *(gdouble *)(qa + ao[e < PA ? e : 0]);
            else v[e] = *(gdouble *)(qb + bo[e < PA ? 0 : e - PA]);
        };
        auto put = [&](int e, double *wa, double *wb) {
            if(e < PA) wa[RP * e * kTileRow] = v[e] * sc[e < PA ? e : 0];
            else wb[RP * (e - PA) * kTileRow] = v[e];
        };
        // Past a pair's extent both operands are zero, and everywhere in a
        // chunk past the group's last one.
        auto clip = [&](const chunk_pos &n) {
            const bool la = n.valid && 16 * n.c + ((fl & kPairAKMajor) ? hi : lo) < n.k;
            const bool lb = n.valid && 16 * n.c + ((fl & kPairBNFast) ? hi : lo) < n.k;
#pragma unroll
            for(int e = 0; e < E; e++) v[e] = (e < PA ? la : lb) ? v[e] : 0.0;
        };

        // One step: products of the staged chunk; between them, the loads of
        // the next chunk and its way into the other buffer, so that a wave
        // keeps issuing products (waves that first multiplied and then moved
        // data fell into step with each other and left the matrix cores idle
        // a third of the time).
        double *base = sm.ch + g * 2 * S::CH;
        auto step = [&](auto mc, int rtog, int wtog) {
            constexpr bool mult = decltype(mc)::value;
            const bool info = n2.p != n1.p;
            row_src ar; uint32_t cq = 0;
            seek(n1);
            const bool akm = (fl & kPairAKMajor) != 0, bnf = (fl & kPairBNFast) != 0;
            const double *rd = &sm.rd[g][n1.slot][akm ? lw : hr];
            double *wa = base + wtog + (akm ? a1 : a0), *wb = base + wtog + S::RA * kTileRow + (bnf ? a1 : a0);
            double2_t b0, b1, x0, x1, y0, y1;
            const double *bp = base + rtog + (S::RA + 16 * wave + lr) * kTileRow + 4 * lg;
            const double *ap = base + rtog + lr * kTileRow + 4 * lg;
            if constexpr(mult) {
                b0 = *(const double2_t *)bp; b1 = *(const double2_t *)(bp + 2);
                x0 = *(const double2_t *)ap; x1 = *(const double2_t *)(ap + 2);
            }
            if(info) info_load(n2.p, ar, cq);
            const bool edge = 16 * n1.c + 16 > n1.k || !n1.valid;
            // 2 FM slots of two products each
            constexpr int H = FM;
#pragma unroll
            for(int h = 0; h < H; h++) {
                if constexpr(mult) {
                    if(h % 2 == 0 && h / 2 + 1 < FM) {
                        y0 = *(const double2_t *)(ap + 16 * (h / 2 + 1) * kTileRow);
                        y1 = *(const double2_t *)(ap + 16 * (h / 2 + 1) * kTileRow + 2);
                    }
                }
                // loads in the first FM / 2 slots
#pragma unroll
                for(int e = 2 * h * E / H; e < 2 * (h + 1) * E / H; e++) if(e < E) load(e);
                if constexpr(mult) {
                    const int i = h / 2;
                    const double2_t x = h % 2 ? x1 : x0, b = h % 2 ? b1 : b0;
                    acc[i] = __builtin_amdgcn_mfma_f64_16x16x4f64(x.x, b.x, acc[i], 0, 0, 0);
                    acc[i] = __builtin_amdgcn_mfma_f64_16x16x4f64(x.y, b.y, acc[i], 0, 0, 0);
                    if(h % 2) { x0 = y0; x1 = y1; }
                    __builtin_amdgcn_sched_barrier(0);
                }
            }
#pragma unroll
            for(int e = 0; e < PA; e++) sc[e] = rd[RP * e];
            if(edge) clip(n1);
#pragma unroll
            for(int h = H; h < 2 * FM; h++) {
                if constexpr(mult) {
                    if(h % 2 == 0 && h / 2 + 1 < FM) {
                        y0 = *(const double2_t *)(ap + 16 * (h / 2 + 1) * kTileRow);
                        y1 = *(const double2_t *)(ap + 16 * (h / 2 + 1) * kTileRow + 2);
                    }
                    const int i = h / 2;
                    const double2_t x = h % 2 ? x1 : x0, b = h % 2 ? b1 : b0;
                    acc[i] = __builtin_amdgcn_mfma_f64_16x16x4f64(x.x, b.x, acc[i], 0, 0, 0);
                    acc[i] = __builtin_amdgcn_mfma_f64_16x16x4f64(x.y, b.y, acc[i], 0, 0, 0);
                    if(h % 2) { x0 = y0; x1 = y1; }
                }
                // LDS writes in the last FM slots
#pragma unroll
                for(int e = (h - H) * E / H; e < (h - H + 1) * E / H; e++) put(e, wa, wb);
                if constexpr(mult) __builtin_amdgcn_sched_barrier(0);
            }
            if(info) info_store(n2.slot, ar, cq);
            n1 = n2;
            n2 = chunk_advance(pairs, n2, KG);
            __syncthreads();
        };
        // the first chunk into buffer 0, then a step for every chunk; a wave
        // whose 16 columns are all past the extent only moves data
        step(std::false_type(), 0, 0);
        const uint32_t nstep = (nchunk + KG - 1) / KG;
        int tog = 0;
        if(uint32_t(16 * wave) < nrem) {
            for(uint32_t it = 0; it < nstep; it++, tog = S::CH - tog) step(std::true_type(), tog, S::CH - tog);
        } else {
            for(uint32_t it = 0; it < nstep; it++, tog = S::CH - tog) step(std::false_type(), tog, S::CH - tog);
        }
    }

    if(KG == 1) {
#pragma unroll
        for(int i = 0; i < FM; i++)
#pragma unroll
            for(int v = 0; v < 4; v++) {
                const uint32_t row = 16 * i + lg + 4 * v, col = 16 * wave + lr;
                if(tp.part) tp.part[((i * 4 + v) * NW + wave) * 64 + lane] = acc[i][v];
                else if(row < mrem && col < nrem) src.write(m0 + row, n0 + col, acc[i][v]);
            }
        return;
    }
    // the groups' partial tiles, added in group order
    double *red = sm.ch;
#pragma unroll
    for(int i = 0; i < FM; i++)
#pragma unroll
        for(int v = 0; v < 4; v++)
            red[g * BM * BN + ((i * 4 + v) * NW + wave) * 64 + lane] = acc[i][v];
    __syncthreads();
    for(int e = threadIdx.x; e < BM * BN; e += GT * KG) {
        double x = red[e];
#pragma unroll
        for(int q = 1; q < KG; q++) x += red[q * BM * BN + e];
        const int l = e & 63, w = (e >> 6) % NW, v = (e / GT) & 3, i = e / (4 * GT);
        const uint32_t row = 16 * i + (l >> 4) + 4 * v, col = 16 * w + (l & 15);
        if(tp.part) tp.part[e] = x;
        else if(row < mrem && col < nrem) src.write(m0 + row, n0 + col, x);
    }
}

//! A tile of height up to 16 FM: the loop compiled for its number of 16-row
//! fragments (a condition per fragment inside one loop would make the
//! compiler copy the accumulators).
template<int FM, int KG, int NW, int FA>
__device__ __forceinline__ void tile_height(const stack_rows &src, const tile_part &tp, char *smem) {
    if(FA == 1 || tp.mrem > 16 * (FA - 1)) tile_body<FA, KG, NW>(src, tp, *(tile_smem<FA, KG, NW> *)smem);
    else tile_height<FM, KG, NW, (FA > 1 ? FA - 1 : 1)>(src, tp, smem);
}

//! Workgroups that share a CU get different priorities, the same on its four
//! SIMDs: a workgroup's waves then pass their barriers together instead of
//! each waiting for another workgroup (4 % on large products).
__device__ __forceinline__ void rank_workgroup() {
    switch((blockIdx.x >> 8) & 3) {
    case 0: __builtin_amdgcn_s_setprio(3); break;
    case 1: __builtin_amdgcn_s_setprio(2); break;
    case 2: __builtin_amdgcn_s_setprio(1); break;
    default: __builtin_amdgcn_s_setprio(0); break;
    }
}

template<int FM, int KG, int OCC, int NW>
__global__ void __launch_bounds__(64 * NW * KG) __attribute__((amdgpu_waves_per_eu(OCC)))
gemm_tile_kernel(const tile_stack *__restrict__ stacks, const tile_item *__restrict__ items,
    double *__restrict__ parts) {
    __shared__ __attribute__((aligned(16))) char smem[sizeof(tile_smem<FM, KG, NW>)];
    const tile_item it = items[blockIdx.x];
    cstack *st = (cstack *)(uintptr_t)(stacks + it.stack);
    if(st->rows == 0) return;                    // padding tile (whole workgroup)
    rank_workgroup();
    stack_rows src;
    src.pairs = (cpair *)(uintptr_t)st->pairs;
    src.arow = (garow *)(uintptr_t)st->arow;
    src.crow = (gcrow *)(uintptr_t)st->crow;
    src.astride = st->astride;
    tile_part tp;
    tp.m0 = uint32_t(it.tm) * (16 * FM);
    tp.n0 = uint32_t(it.tn) * (16 * NW);
    tp.mrem = st->rows - tp.m0;
    tp.nrem = st->n - tp.n0;
    tp.p = it.p; tp.c = it.c; tp.count = it.count;
    tp.part = it.part < 0 ? (gout *)0 : (gout *)(uintptr_t)parts + size_t(it.part) * (256 * NW * FM);
    tile_height<FM, KG, NW, FM>(src, tp, smem);
}

//! C of the tiles whose chunks were cut into parts: their partial sums added
//! in the order of the parts.
__global__ void __launch_bounds__(256)
tile_sum_kernel(const tile_stack *__restrict__ stacks, const tile_item *__restrict__ items,
    const double *__restrict__ parts, uint32_t fm, uint32_t lnw) {
    const tile_item it = items[blockIdx.x];      // part: the first part's place, count: parts
    cstack *st = (cstack *)(uintptr_t)(stacks + it.stack);
    const uint32_t m0 = uint32_t(it.tm) * (16 * fm), n0 = uint32_t(it.tn) * (16u << lnw);
    const uint32_t mrem = st->rows - m0, nrem = st->n - n0;
    stack_rows src;
    src.crow = (gcrow *)(uintptr_t)st->crow;
    const uint32_t e = blockIdx.y * 256 + threadIdx.x;
    const uint32_t l = e & 63, w = (e >> 6) & ((1u << lnw) - 1), v = (e >> (6 + lnw)) & 3, i = e >> (8 + lnw);
    const uint32_t row = 16 * i + (l >> 4) + 4 * v, col = 16 * w + (l & 15);
    if(row >= mrem || col >= nrem) return;
    gdouble *p = (gdouble *)(uintptr_t)parts + size_t(it.part) * (256u * fm << lnw) + e;
    double x = p[0];
    for(uint32_t q = 1; q < it.count; q++) x += p[size_t(q) * (256u * fm << lnw)];
    src.write(m0 + row, n0 + col, x);
}

hipError_t launch_tile_sum(int cfg, const tile_stack *st, const tile_item *items, uint32_t n,
    const double *parts, hipStream_t s) {
    if(n == 0) return hipSuccess;
    uint32_t bm, bn;
    tile_shape(cfg, bm, bn);
    hipLaunchKernelGGL(tile_sum_kernel, dim3(n, bm * bn / 256), dim3(256), 0, s, st, items, parts, bm / 16,
        bn == 128 ? 3u : 2u);
    return hipGetLastError();
}

hipError_t launch_gemm_tile(int cfg, const tile_stack *st, const tile_item *items,
    uint32_t nitems, double *parts, hipStream_t s) {
    if(nitems == 0) return hipSuccess;
#define LT_TILE(FM, KG, OCC, NW) \
    hipLaunchKernelGGL((gemm_tile_kernel<FM, KG, OCC, NW>), dim3(nitems), dim3(64 * NW * KG), 0, s, st, items, parts)
    switch(cfg) {
    case WG_16x64_G4: LT_TILE(1, 4, 4, 4); break;
    case WG_32x64_G4: LT_TILE(2, 4, 4, 4); break;
    case WG_96x128_G1: LT_TILE(6, 1, 4, 8); break;
    case WG_48x64_G4: LT_TILE(3, 4, 4, 4); break;
    case WG_64x64_G4: LT_TILE(4, 4, 4, 4); break;
    case WG_64x64_G1: LT_TILE(4, 1, 4, 4); break;
    case WG_80x64_G2: LT_TILE(5, 2, 2, 4); break;
    case WG_96x64_G1: LT_TILE(6, 1, 3, 4); break;
    case WG_112x64_G1: LT_TILE(7, 1, 2, 4); break;
    default: return hipErrorInvalidValue;
    }
#undef LT_TILE
    return hipGetLastError();
}

} // namespace dev
} // namespace lta
