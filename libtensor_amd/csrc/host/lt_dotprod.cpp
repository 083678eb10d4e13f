// btod_dotprod on HBM-resident block tensors: sum over all elements of
// tra(A) * trb(B) (libtensor/block_tensor/btod_dotprod.h:24-70,
// gen_block_tensor/impl/gen_bto_dotprod_impl.h:60-95).
//
// Every block X of the (permuted) index space contributes
// dot(A'[X], B'[X]) with A'[X] = tr_a(Ya) and B'[X] = tr_b(Yb) built from
// the stored canonical blocks Ya, Yb.  The block product is evaluated in
// Ya's index space, dot(tr_a(Ya), tr_b(Yb)) = c_a^2 dot(Ya, tr_a^-1 tr_b (Yb))
// (c_a the scalar of tr_a), so each block is one descriptor of the device
// dot kernel reading both canonical blocks in place.  Blocks forbidden by
// either symmetry or zero in either tensor contribute nothing.  All
// partial sums are added in a fixed order.
#include "lt_runtime.h"

#include <algorithm>
#include <cstring>

namespace lta {

namespace {

//! A transposing descriptor is read by tiles only where a tile is well filled
//! and reading element by element, in the destination's order, would not find
//! its source lines in the caches (0.4 M elements: 5 to 6 us by elements in every
//! order, 5 to 10 by tiles).  4 M elements, us by elements and by tiles
//! (p: extent contiguous in the source, q: in the destination): p = q = 4, 8,
//! 12, 16 and 32 at the ends of a three-dimensional tensor 27, 44, 61, 76, 77;
//! 303, 83, 42, 28, 15.  Matrices with p = 5, 8, 12 and 16: 30, 43, 61, 80; 40,
//! 28, 22, 18; with q = 5, 8, 16 and 24: 15, 15, 15, 14; 42, 28, 18, 16.  Last
//! two dimensions swapped, p = q = 16, 32, 40, 48 and 64: 17, 16, 16, 16, 18; 27,
//! 16, 18, 15, 15.  fill: elements that a tile must hold on the average, least: in
//! all; 144 and 2^19 where the list is kept, 512 and 2^22 where it is made and
//! uploaded for one product (7 ns an item and about 35 us, where a product by
//! elements passes its descriptor with the launch).
void choose_tiles(dev::perm_desc &d, uint64_t fill, uint32_t least) {
    if(d.tile_p < 0) return;
    const uint64_t p = d.tdp.d, q = d.tdq.d;
    const uint64_t s = d.tile_s = std::min(p, q) > dev::kPermTile ? dev::kPermTileMax : dev::kPermTile;
    const uint64_t tiles = ((p + s - 1) / s) * ((q + s - 1) / s);
    if(d.total < least || std::min(p, q) < 8 || p * q < fill * tiles || (q <= 24 && d.dps.d == q) ||
        8 * uint64_t(d.tsq) * q <= 16384) d.tile_p = -1;
}

//! Partial sums of n work items, and the product behind them.
size_t dot_bytes(size_t n) { return (std::min<size_t>(n, dev::kDotGroups) + 1) * sizeof(double); }

//! The product of lists in device memory, partial sums at `part`.
double run_dot(context &ctx, const char *base, const context::cached_launch::segment &g, double *part) {
    double *out = part + std::min<size_t>(g.nchunks, dev::kDotGroups);
    double r = 0.0;
    hip_check(dev::launch_dot((dev::perm_desc*)(base + g.o_d), (uint32_t*)(base + g.o_cd),
        (uint32_t*)(base + g.o_co), (uint32_t)g.nchunks, g.tiles, part, out, ctx.stream()), "dot");
    ctx.download(&r, out, sizeof(double));
    return r;
}

//! Scalar product of the (single) list of a cached entry: sum over its
//! descriptors of dst * alpha P(src).
double run_dot(context &ctx, const context::cached_launch &l) {
    if(l.segs.empty()) return 0.0;
    std::lock_guard<std::mutex> lk(ctx.staging_lock());
    double *part = (double*)ctx.staging(dot_bytes(l.segs[0].nchunks));
    ctx.activate();
    return run_dot(ctx, (const char*)l.mem, l.segs[0], part);
}

} // unnamed namespace

double dense_dotprod(context &ctx, dev::perm_desc d) {
    if(!d.total) return 0.0;
    choose_tiles(d, 512, 1u << 22);
    if(d.tile_p < 0) {
        const size_t n = (d.total + dev::kPermChunk - 1) / dev::kPermChunk;
        double *out, r = 0.0;
        std::lock_guard<std::mutex> lk(ctx.staging_lock());
        double *part = (double*)ctx.staging(dot_bytes(n));
        out = part + std::min<size_t>(n, dev::kDotGroups);
        ctx.activate();
        hip_check(dev::launch_dot_one(d, part, out, ctx.stream()), "dot");
        ctx.download(&r, out, sizeof(double));
        return r;
    }
    std::vector<uint32_t> cd, co;
    make_chunks(std::vector<dev::perm_desc>(1, d), cd, co);
    // descriptor and work items in the staging area, partial sums behind them
    context::cached_launch::segment g;
    g.o_d = 0;
    g.o_cd = (sizeof(d) + 255) & ~size_t(255);
    g.o_co = g.o_cd + ((4 * cd.size() + 255) & ~size_t(255));
    g.nchunks = cd.size();
    g.tiles = true;
    const size_t bytes = g.o_co + ((4 * co.size() + 255) & ~size_t(255));
    std::vector<char> host(bytes, 0);
    std::memcpy(&host[0], &d, sizeof(d));
    std::memcpy(&host[g.o_cd], cd.data(), 4 * cd.size());
    std::memcpy(&host[g.o_co], co.data(), 4 * co.size());
    std::lock_guard<std::mutex> lk(ctx.staging_lock());
    char *mem = (char*)ctx.staging(bytes + dot_bytes(g.nchunks));
    ctx.upload(mem, host.data(), bytes);
    ctx.activate();
    return run_dot(ctx, mem, g, (double*)(mem + bytes));
}

double btod_dotprod(btensor &a, const tensor_tr &tra0, btensor &b, const tensor_tr &trb0) {
    context &ctx = a.ctx();
    ctx.require_device("btod_dotprod");
    lt_require(&b.ctx() == &ctx, LT_ERR_PARAM, "tensors of different contexts");
    bis_t bisa2 = a.bis(), bisb2 = b.bis();
    bisa2.permute(tra0.perm);
    bisb2.permute(trb0.perm);
    lt_require(bisa2 == bisb2, LT_ERR_DIMS, "btod_dotprod: block index spaces differ");
    const dims_t bid2 = bisa2.block_index_dims(), bida = a.bidims(), bidb = b.bidims();
    const perm_t pai = tra0.perm.inverse(), pbi = trb0.perm.inverse();

    const double scale = tra0.st.c * trb0.st.c;

    // descriptors and work items, kept per structure versions of A and B
    const std::string key = "dot" + key_tensor(a, true) + key_tensor(b, true) + "|" +
        key_part(tra0) + "|" + key_part(trb0);
    std::shared_ptr<context::cached_launch> l = ctx.find_launch(key, context::DOT_PRODUCTS);
    if(l) return run_dot(ctx, *l) * scale;
    std::vector<std::vector<dev::perm_desc> > lists(1);
    std::vector<dev::perm_desc> &descs = lists[0];
    for(size_t x = 0; x < bid2.size(); x++) {
        index_t ix = get_index(x, bid2);
        index_t ia = ix, ib = ix;
        pai.apply(ia);
        pbi.apply(ib);
        size_t xa = abs_index(ia, bida), xb = abs_index(ib, bidb);
        short_orbit sa(a.sym(), xa, true);
        if(!sa.allowed || !a.is_nonzero(sa.acidx)) continue;
        short_orbit sb(b.sym(), xb, true);
        if(!sb.allowed || !b.is_nonzero(sb.acidx)) continue;
        orbit oa(a.sym(), xa, false), ob(b.sym(), xb, false);
        tensor_tr ta = oa.get_transf(xa);
        ta.transform(tensor_tr(tra0.perm, scalar_tr()));
        tensor_tr tb = ob.get_transf(xb);
        tb.transform(tensor_tr(trb0.perm, scalar_tr()));
        tensor_tr t(tb);
        t.transform(ta.inverse());
        dims_t dyb = b.bis().block_dims(get_index(sb.acidx, bidb));
        dev::perm_desc d = make_perm_desc_public(b.block_ptr(sb.acidx), dyb, t,
            a.block_ptr(sa.acidx), false);
        d.alpha *= ta.st.c * ta.st.c;
        choose_tiles(d, 144, 1u << 19);
        descs.push_back(d);
    }
    l = upload_launches(ctx, lists);
    ctx.keep_launch(key, l, context::DOT_PRODUCTS);
    return run_dot(ctx, *l) * scale;
}

} // namespace lta
