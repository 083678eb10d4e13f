// Dense operations on device arrays: tod_copy, tod_add, tod_contract2
// (libtensor/dense_tensor/tod_copy.h, tod_add.h, tod_contract2.h;
// impl/tod_contract2_impl.h:124-135 for the alignment the reference makes).
//
// A contraction runs as one kernel over C's tiles that reads A and B and
// writes C at their own strides; an operand is copied into another order first
// only where its contiguous dimension cannot be the fastest one of the row (or
// column) or k index it is read along.
#include "lt_runtime.h"

#include <algorithm>
#include <string>

namespace lta {

namespace {

//! Runs of fewer elements than this are copied into a contiguous order: the
//! kernel reads 16 elements of an operand's fast index at a time, so shorter
//! runs touch two and more times the cache lines.
const size_t kMinRun = 8;
//! C whose contiguous dimension is fastest in neither the row nor the column
//! index is written in place up to this size (it stays in the caches, where
//! partial lines meet), beyond it through a contiguous copy.
const size_t kScatterBytes = size_t(32) << 20;
//! Workgroups a contraction is cut into (tiles, or parts of tiles) at most
//! when its tiles alone leave CUs idle.
const size_t kSplitGroups = 256;
static_assert(kSplitGroups * 2048 * sizeof(double) <= dev::kNoallocPartBytes,
    "partial sums of a split contraction in the scratch region");

//! One dimension of an axis: its positions in the two tensors it belongs to.
struct axdim { size_t ext, p0, p1; };
typedef std::vector<axdim> axis;

axis ordered(const axis &x, bool second) {
    axis r(x);
    std::sort(r.begin(), r.end(), [second](const axdim &a, const axdim &b) {
        return second ? a.p1 < b.p1 : a.p0 < b.p0;
    });
    return r;
}

size_t extent(const axis &x) {
    size_t e = 1;
    for(size_t i = 0; i < x.size(); i++) e *= x[i].ext;
    return e;
}

//! Contiguous elements of a tensor (dimensions d) along the fast end of axis x.
size_t run(const dims_t &d, const axis &x, bool second) {
    size_t r = 1, i = x.size();
    for(size_t p = d.n; p-- > 0 && i > 0;) {
        if(d[p] == 1) continue;
        if((second ? x[i - 1].p1 : x[i - 1].p0) != p) break;
        r *= d[p];
        i--;
    }
    return r;
}

bool reads_well(size_t r, const axis &x) { return r >= kMinRun || (r > 1 && r == extent(x)); }

size_t last_dim(const dims_t &d) {
    size_t p = d.n;
    while(p > 0 && d[p - 1] == 1) p--;
    return p;                     // one past it; 0: a single element
}

bool has_last(const dims_t &d, const axis &x, bool second) {
    const size_t l = last_dim(d);
    for(size_t i = 0; i < x.size(); i++) if((second ? x[i].p1 : x[i].p0) + 1 == l) return true;
    return false;
}

size_t round256(size_t b) { return (std::max<size_t>(b, 8) + 255) & ~size_t(255); }

//! Bytes that the entry point without allocations reckons for a permuted copy
//! of a tensor: its elements and 8 bytes of list per 32 x 32 tile (or 2048
//! elements).
size_t aligned_bytes(const dims_t &d, const tensor_tr &tr) {
    dev::perm_desc p = make_perm_desc_public(0, d, tr, 0, false);
    size_t n = 1;
    if(p.tile_p < 0) n = (p.total + dev::kPermChunk - 1) / dev::kPermChunk;
    else for(uint32_t i = 0; i < p.n; i++)
        n *= int32_t(i) == p.tile_p || i + 1 == p.n ? (p.div[i].d + 31) / 32 : p.div[i].d;
    return round256(d.size() * 8) + round256(256 + ((4 * n + 255) & ~size_t(255)) + 4 * n);
}

//! The aligned form's temporaries (permuted copies of the operands that are
//! not in matrix order, lists): the size the entry point without allocations
//! accepts or refuses a call by.
size_t region_bytes(const contraction2 &contr, const dims_t &da, const dims_t &db, const dims_t &dc) {
    contraction2_align al(contr);
    dims_t dc2(dc);
    dc2.permute(al.permc);
    size_t m = 1, n = 1, b = 0;
    for(size_t i = 0; i < contr.NC(); i++)
        (contr.conn[i] < contr.NC() + contr.NA() ? m : n) *= dc[i];
    if(!al.perma.is_identity()) b += aligned_bytes(da, tensor_tr(al.perma, scalar_tr()));
    if(!al.permb.is_identity()) b += aligned_bytes(db, tensor_tr(al.permb, scalar_tr()));
    if(!al.permc.is_identity()) {
        b += aligned_bytes(dc2, tensor_tr(al.permc.inverse(), scalar_tr()));
    }
    return b + round256(1024 + 8 * ((m + 63) / 64) * ((n + 63) / 64));
}

//! One contraction laid out on the host.
struct dense_job {
    bool skip, fill;              //!< d == 0 (or no terms): C kept, C := 0
    size_t cn;
    dev::dense_args g;
    int cfg;
    uint32_t nparts;
    size_t part_bytes;            //!< partial sums
    bool copy_a, copy_b, copy_c;  //!< operands (C) read (written) through a copy
    dev::perm_desc pa, pb, pc;
    size_t na, nb;
    //! Bytes of the copies.
    size_t bytes() const {
        return (copy_a ? round256(8 * na) : 0) + (copy_b ? round256(8 * nb) : 0) +
            (copy_c ? round256(8 * cn) : 0);
    }
};

dev::dense_axis make_axis(const axis &x, const size_t *s0, const size_t *s1) {
    // dimensions next to one another in both tensors count as one
    std::vector<size_t> e, a, b;
    for(size_t i = 0; i < x.size(); i++) {
        const size_t t0 = s0[x[i].p0], t1 = s1[x[i].p1];
        if(!e.empty() && a.back() == t0 * x[i].ext && b.back() == t1 * x[i].ext) {
            e.back() *= x[i].ext;
            a.back() = t0;
            b.back() = t1;
        } else {
            e.push_back(x[i].ext);
            a.push_back(t0);
            b.push_back(t1);
        }
    }
    dev::dense_axis r;
    std::memset(&r, 0, sizeof(r));
    r.n = (uint32_t)e.size();
    r.ext = (uint32_t)extent(x);
    for(size_t i = 0; i < (size_t)dev::kDenseMaxOrder; i++) {
        r.div[i] = dev::make_fastdiv(i < e.size() ? (uint32_t)e[i] : 1);
        r.s0[i] = i < e.size() ? (uint32_t)a[i] : 0;
        r.s1[i] = i < e.size() ? (uint32_t)b[i] : 0;
    }
    return r;
}

void strides(const dims_t &d, size_t *s) { for(size_t i = 0; i < d.n; i++) s[i] = d.inc(i); }

//! The permutation of a tensor into the order (dimensions of one element,
//! outer, inner), and the strides its dimensions have there.
perm_t copy_order(const dims_t &d, const axis &outer, bool outer1,
    const axis &inner, bool inner1, size_t *s) {

    perm_t p(d.n);
    size_t k = d.n, stride = 1;
    std::vector<bool> used(d.n, false);
    auto put = [&](size_t dim) {
        p.p[--k] = (uint8_t)dim;
        used[dim] = true;
        s[dim] = stride;
        stride *= d[dim];
    };
    for(size_t i = inner.size(); i-- > 0;) put(inner1 ? inner[i].p1 : inner[i].p0);
    for(size_t i = outer.size(); i-- > 0;) put(outer1 ? outer[i].p1 : outer[i].p0);
    for(size_t i = d.n; i-- > 0;) if(!used[i]) put(i);
    return p;
}

//! Whether n doubles at p and m at q share memory.
bool overlap(const double *p, size_t n, const double *q, size_t m) {
    return uintptr_t(p) < uintptr_t(q + m) && uintptr_t(q) < uintptr_t(p + n);
}

//! stage_c: C may go through a contiguous copy.
void prepare(const contraction2 &contr, dims_t da, const double *a, dims_t db, const double *b,
    double d, bool zero, double *c, bool stage_c, dense_job &j) {

    const dims_t dc = contract2_dims(contr, da, db);
    // the kernels address operands with 32-bit byte offsets
    const size_t lim = size_t(1) << 29;
    lt_require(da.size() < lim && db.size() < lim && dc.size() < lim, LT_ERR_PARAM,
        "tod_contract2: a tensor of 2^29 or more elements (32-bit byte offsets in the "
        "GEMM kernels)");
    j.skip = j.fill = j.copy_a = j.copy_b = j.copy_c = false;
    j.cn = dc.size();
    j.g.c = c;
    if(d == 0.0 || da.size() == 0 || db.size() == 0) {
        j.fill = zero;
        j.skip = !zero;
        return;
    }
    // axes m (A and C), n (B and C), k (A and B); dimensions of one element
    // take no part
    const size_t NC = contr.NC(), NA = contr.NA();
    axis m, n, k;
    for(size_t i = 0; i < NC; i++) {
        const size_t q = contr.conn[i];
        if(dc[i] == 1) continue;
        if(q < NC + NA) m.push_back(axdim{dc[i], q - NC, i});
        else n.push_back(axdim{dc[i], q - NC - NA, i});
    }
    for(size_t i = 0; i < NA; i++) {
        const size_t q = contr.conn[NC + i];
        if(q >= NC + NA && da[i] != 1) k.push_back(axdim{da[i], i, q - NC - NA});
    }
    // Columns (64 to a tile): the index with C's contiguous dimension, so
    // that C is written in rows; the other one where that leaves half again
    // as much of the tiles empty.
    const auto padded = [](size_t r, size_t q) { return (r + 15) / 16 * ((q + 63) / 64); };
    const size_t em = extent(m), en = extent(n);
    bool swap = has_last(dc, m, true);
    const size_t w = swap ? padded(en, em) : padded(em, en), wo = swap ? padded(em, en) : padded(en, em);
    if(3 * wo < 2 * w) swap = !swap;
    if(swap) {
        std::swap(da, db);
        std::swap(a, b);
        std::swap(m, n);
        for(size_t i = 0; i < k.size(); i++) std::swap(k[i].p0, k[i].p1);
    }
    // order of each index: that of the operand whose contiguous dimension is
    // in it, else C's; of k, that of the operand for which less is copied
    m = ordered(m, !has_last(da, m, false));
    n = ordered(n, !has_last(db, n, false));
    axis ks[2] = { ordered(k, false), ordered(k, true) };
    bool ca[2], cb[2];
    size_t cost[2];
    for(int i = 0; i < 2; i++) {
        ca[i] = da.size() > 1 && !reads_well(run(da, m, false), m) && !reads_well(run(da, ks[i], false), ks[i]);
        cb[i] = db.size() > 1 && !reads_well(run(db, n, false), n) && !reads_well(run(db, ks[i], true), ks[i]);
        cost[i] = (ca[i] ? da.size() : 0) + (cb[i] ? db.size() : 0);
    }
    const int o = cost[1] < cost[0] ? 1 : 0;
    k = ks[o];
    // (an operand that C overlaps is read before C is written)
    j.copy_a = ca[o] || overlap(a, da.size(), c, dc.size());
    j.copy_b = cb[o] || overlap(b, db.size(), c, dc.size());
    j.na = da.size();
    j.nb = db.size();
    size_t sa[kMaxOrder], sb[kMaxOrder], sc[kMaxOrder];
    strides(da, sa);
    strides(db, sb);
    strides(dc, sc);
    bool arf = run(da, m, false) > run(da, k, false), brf = run(db, n, false) > run(db, k, true);
    if(j.copy_a) {
        m = ordered(m, true);
        arf = false;
        j.pa = make_perm_desc_public(a, da, tensor_tr(copy_order(da, m, false, k, false, sa),
            scalar_tr()), 0, false);
    }
    if(j.copy_b) {
        n = ordered(n, true);
        brf = false;
        j.pb = make_perm_desc_public(b, db, tensor_tr(copy_order(db, n, false, k, true, sb),
            scalar_tr()), 0, false);
    }
    if(stage_c && 8 * dc.size() > kScatterBytes && !reads_well(run(dc, n, true), n) &&
        run(dc, m, true) < std::min(kMinRun, extent(m))) {
        j.copy_c = true;
        dims_t dt(dc);
        const perm_t p = copy_order(dc, m, true, n, true, sc);
        dt.permute(p);
        j.pc = make_perm_desc_public(0, dt, tensor_tr(p.inverse(), scalar_tr()), c, !zero);
    }
    j.g.a = a;
    j.g.b = b;
    j.g.d = d;
    j.g.m = make_axis(m, sa, sc);
    j.g.n = make_axis(n, sb, sc);
    j.g.k = make_axis(k, sa, sb);
    j.g.zero = zero ? 1 : 0;
    j.g.rows_fast = (arf ? 1 : 0) | (brf ? 2 : 0);

    // Tiles: 64 x 64 where they keep the CUs busy, the k range in two groups
    // of waves below 1.5 to a CU; 32 x 64 in four groups from half the CUs on,
    // else 16 x 64 in four, both cut along k into parts (of 16 chunks of k and
    // more) that come to a workgroup per CU.  us a call, with each shape in
    // this order: 2000 x 1500 x 600 86, 91, 130, 184; 1000 x 1000 x 500 47,
    // 43, 52, 65; 675 x 675 x 675 54, 49, 40, 48; 500 x 500 x 2000 115, 98, 50
    // (68 uncut), 56; 300 x 300 x 300 34, 33, 27, 23; 128 x 128 x 4000 28 with
    // the last cut, 79 uncut.
    const size_t mm = j.g.m.ext, nn = j.g.n.ext, nch = (size_t(j.g.k.ext) + 15) / 16;
    const size_t tn = (nn + 63) / 64;
    j.nparts = 1;
    const size_t t64 = (mm + 63) / 64 * tn;
    j.cfg = t64 >= 384 ? dev::DENSE_64x64_G1 : t64 >= 200 ? dev::DENSE_64x64_G2 :
        (mm + 31) / 32 * tn >= 128 ? dev::DENSE_32x64_G4 : dev::DENSE_16x64_G4;
    uint32_t bm = 0, bn = 0;
    dev::dense_tile_shape(j.cfg, bm, bn);
    const size_t t = (mm + bm - 1) / bm * tn;
    if(bm < 64 && t < kSplitGroups)
        j.nparts = (uint32_t)std::max<size_t>(1, std::min(kSplitGroups / t, nch / 16));
    j.part_bytes = j.nparts == 1 ? 0 : (mm + bm - 1) / bm * tn * j.nparts * bm * bn * sizeof(double);
}

//! The launches, in stream order (no synchronization); copies at mem, partial
//! sums at parts.
void launch(context &cx, dense_job &j, char *mem, double *parts) {
    if(j.skip) return;
    if(j.fill) {
        hip_check(dev::launch_fill(j.g.c, j.cn, 0.0, cx.stream()), "fill");
        return;
    }
    if(j.copy_a) {
        widen_tiles(&j.pa, 1);
        j.g.a = j.pa.dst = (double*)mem;
        mem += round256(8 * j.na);
        hip_check(dev::launch_permute_one(j.pa, cx.stream()), "permute");
    }
    if(j.copy_b) {
        widen_tiles(&j.pb, 1);
        j.g.b = j.pb.dst = (double*)mem;
        mem += round256(8 * j.nb);
        hip_check(dev::launch_permute_one(j.pb, cx.stream()), "permute");
    }
    if(j.copy_c) {
        widen_tiles(&j.pc, 1);
        j.pc.src = j.g.c = (double*)mem;
        j.g.zero = 1;
    }
    hip_check(dev::launch_gemm_dense(j.cfg, j.g, j.nparts, parts, cx.stream()), "gemm");
    if(j.copy_c) hip_check(dev::launch_permute_one(j.pc, cx.stream()), "permute");
}

//! A device buffer for one call, from the context's allocator.
struct call_buffer {
    context &ctx;
    char *p;
    call_buffer(context &c, size_t bytes) : ctx(c), p(bytes ? (char*)c.alloc(bytes) : 0) { }
    ~call_buffer() { if(p) ctx.free(p); }
    call_buffer(const call_buffer&) = delete;
    call_buffer &operator=(const call_buffer&) = delete;
};

//! Runs jobs in order, their partial sums in the context's staging area and
//! their copies in one buffer (each job's after the one before has read it).
void run_jobs(context &cx, std::vector<dense_job> &jobs) {
    size_t bytes = 0, parts = 0;
    bool any = false;
    for(size_t i = 0; i < jobs.size(); i++) {
        if(jobs[i].skip) continue;
        any = true;
        if(jobs[i].fill) continue;
        bytes = std::max(bytes, jobs[i].bytes());
        parts = std::max(parts, jobs[i].part_bytes);
    }
    if(!any) return;
    call_buffer mem(cx, bytes);
    std::unique_lock<std::mutex> lk(cx.staging_lock(), std::defer_lock);
    double *pp = 0;
    if(parts) {
        lk.lock();
        try {
            pp = (double*)cx.staging(parts);
        } catch(const lt_error &e) {
            // no room for partial sums: every k range whole
            if(e.code != LT_ERR_NOMEM) throw;
            for(size_t i = 0; i < jobs.size(); i++) jobs[i].nparts = 1;
        }
    }
    cx.activate();
    try {
        for(size_t i = 0; i < jobs.size(); i++) launch(cx, jobs[i], mem.p, pp);
    } catch(...) {
        cx.sync();
        throw;
    }
    cx.sync();
}

} // unnamed namespace

void dense_permute(context &cx, const double *src, const dims_t &dsrc,
    const tensor_tr &tr, double *dst, bool accumulate) {
    dev::perm_desc d = make_perm_desc_public(src, dsrc, tr, dst, accumulate);
    widen_tiles(&d, 1);
    if(!d.total) return;
    cx.activate();
    hip_check(dev::launch_permute_one(d, cx.stream()), "permute");
    cx.sync();
}

void dense_add(context &cx, const double *const *a, const dims_t &da,
    const std::vector<tensor_tr> &trs, double *b, bool zero) {
    std::vector<dev::perm_desc> ds;
    for(size_t i = 0; i < trs.size(); i++)
        ds.push_back(make_perm_desc_public(a[i], da, trs[i], b, !(zero && i == 0)));
    if(!ds[0].total) return;
    // the first two terms in one pass where one of them keeps its order
    if(zero && ds.size() > 1 && !overlap(a[0], da.size(), b, da.size()) &&
        !overlap(a[1], da.size(), b, da.size())) fuse_terms(ds[0], ds[1]);
    cx.activate();
    for(size_t i = 0; i < ds.size(); i++) widen_tiles(&ds[i], 1);
    for(size_t i = 0; i < ds.size(); i++)
        if(ds[i].total) hip_check(dev::launch_permute_one(ds[i], cx.stream()), "permute");
    cx.sync();
}

void dense_contract2(context &cx, const contraction2 &contr, const dims_t &da, const double *a,
    const dims_t &db, const double *b, double d, bool zero, double *c) {
    std::vector<dense_job> j(1);
    prepare(contr, da, a, db, b, d, zero, c, true, j[0]);
    run_jobs(cx, j);
}

void dense_contract2_noalloc(context &cx, const contraction2 &contr, const dims_t &da,
    const double *a, const dims_t &db, const double *b, double d, bool zero, double *c) {
    dense_job j;
    prepare(contr, da, a, db, b, d, zero, c, false, j);
    if(j.skip) return;
    cx.activate();
    void *region = 0;
    hip_check(dev::noalloc_scratch(cx.device(), &region), "scratch region address");
    if(!j.fill && (region_bytes(contr, da, db, contract2_dims(contr, da, db)) > dev::kNoallocScratchBytes ||
        j.bytes() > dev::kNoallocScratchBytes)) {
        throw lt_error(LT_ERR_PARAM, "temporaries exceed the fixed scratch region of " +
            std::to_string(dev::kNoallocScratchBytes) + " bytes");
    }
    launch(cx, j, (char*)region, (double*)((char*)region + dev::kNoallocScratchBytes));
    cx.sync();
}

void dense_contract2_many(context &cx, const std::vector<dense_contract_item> &items,
    double *c) {
    std::vector<dense_job> jobs(items.size());
    for(size_t i = 0; i < items.size(); i++)
        prepare(items[i].contr, items[i].da, items[i].a, items[i].db, items[i].b,
            items[i].d, items[i].zero, c, true, jobs[i]);
    run_jobs(cx, jobs);
}

} // namespace lta
