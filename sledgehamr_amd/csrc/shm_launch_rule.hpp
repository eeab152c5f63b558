// The rule that picks the launch shape of a level nobody tuned.  Host code
// without HIP, so it can be checked where there is no GPU.
#pragma once

#include <algorithm>
#include <vector>

namespace shm {

struct Box3 {
    int lo[3], hi[3];  // inclusive, global index space of the level
    int n(int d) const { return hi[d] - lo[d] + 1; }
    long long vol() const { return (long long)n(0) * n(1) * n(2); }
};

/** Tile shape variants: NW wavefronts per workgroup, RY rows per thread, TX
 *  cells in x (tile = TX x (NW * 64 / TX) * RY cells in x/y).  The 32-wide
 *  tile serves boxes narrower than 64 cells.  The autotuner picks one per
 *  level. */
struct TileVariant {
    int nw, ry, tx;
};
constexpr int kNVar = 5;
constexpr TileVariant kVariants[kNVar] = {
    {4, 1, 64}, {8, 1, 64}, {16, 1, 64}, {4, 1, 32}, {4, 2, 64}};
constexpr int kDefaultVariant = 1;

/** Launch shape of the stage kernels.  A field of -1 (tz: 0) is not set: the
 *  level's tuned value, else the size rule (LaunchRule) applies. */
struct LaunchCfg {
    int variant = -1;     // tile shape index into kVariants
    int tz = 0;           // z-chunk length of a tile (0: automatic)
    int xcd_split = -1;   // each XCD walks one contiguous range of tiles
    int persistent = -1;  // grid = resident capacity (1) or one tile per workgroup (0)
    int zc_minor = -1;    // tile order: z-chunk outermost (0) or innermost (1)
    int fused = -1;       // SSPRK3 stages one and two in one launch (0/1)
    int fused_variant = -1;  // tile shape of that launch
};

/** z-chunk length for which nothing is set: enough tiles to fill every CU
 *  several times, long z runs otherwise. */
inline int auto_chunk(const std::vector<Box3> &boxes, int tx, int ty, int ncu) {
    int maxn = 1;
    long long xy = 0;
    for (const Box3 &b : boxes) {
        maxn = std::max(maxn, b.n(2));
        xy += (long long)((b.n(0) + tx - 1) / tx) * ((b.n(1) + ty - 1) / ty);
    }
    int z = maxn;
    while (z > 16 && xy * ((maxn + z - 1) / z) < 8LL * ncu) z = (z + 1) / 2;
    return z;
}

/** What the rule looks at: the stored boxes of a level and what is built for
 *  its project, precision, radius and integrator. */
struct LaunchRule {
    const std::vector<Box3> &boxes;
    int integrator;          // 10 SSPRK3, 11 leapfrog, 20.. RKN
    int nfields;
    int R;                   // stencil radius
    bool f64;                // states are stored in FP64
    bool tile_lo;            // FP64 tiles of stored pairs
    bool gw, gw_groups, ko;
    int ncu;
    bool can_fuse;           // the first two stages may run in one launch
    bool stage_built[kNVar]; // tile shapes of the first stage's kernel
    int fused_ty[kNVar];     // rows of the fused kernel's tile (0: not built)

    LaunchCfg pick(int fused) const;
};

/** The launch shape the box sizes ask for.  A stage kernel's time is modelled
 *  as the planes a resident workgroup walks one after the other (rounds of
 *  the grid times the chunk with its R extra queue planes), plus a small
 *  share for the wavefront planes of the whole grid; constants fitted to a
 *  sweep of every shape over levels of one and two fields in three
 *  precisions.  It serves levels that leave CUs idle: two fields at 32^3 take
 *  25 us per RKN4 step (63 on the default 64 x 8 tiles of 16 planes, where 8
 *  workgroups walk 16 planes each), 128^3 80 us (95); levels from 130^3 up
 *  have a rule of their own below. */
inline LaunchCfg LaunchRule::pick(int fused) const {
    LaunchCfg c;
    c.variant = kDefaultVariant;
    c.fused = 0;
    // Dissipation is built for one tile shape.
    if (ko || boxes.empty()) return c;
    int maxn = 1;
    for (const Box3 &b : boxes) maxn = std::max(maxn, b.n(2));
    const bool one_field = nfields == 1 && !tile_lo;
    // A thread of a 16-wavefront group has 128 registers: not enough for the
    // queues of several stencil components in FP64 (RKN at 128^3: 208 us
    // against 102 on 8 wavefronts).
    const bool usable16 = nfields == 1 || !(tile_lo || f64);
    auto usable = [&](int v) {
        if (!stage_built[v] || (kVariants[v].nw > 8 && !usable16)) return false;
        // Two rows per thread pay where a thread holds one short queue (one
        // stencil component read as stored: 255 against 315 us at 256^3)
        // and cost registers elsewhere (519 against 470 us with two).
        if (kVariants[v].ry > 1) return one_field;
        if (one_field && kVariants[v].tx == 64 && kVariants[v].nw > 4) return false;
        // At radius 3 a 32 x 8 tile's ring has more cells than the tile.
        return kVariants[v].tx == 64 || R < 3;
    };
    auto tiles = [&](int tx, int ty, int z, double &planes) {
        long long n = 0;
        planes = 0;
        for (const Box3 &b : boxes) {
            const long long xy = (long long)((b.n(0) + tx - 1) / tx) * ((b.n(1) + ty - 1) / ty);
            const int k = (b.n(2) + z - 1) / z;
            n += xy * k;
            planes += (double)xy * (b.n(2) + k * R);
        }
        return n;
    };
    if (gw) {
        // GW levels run as three component groups per stage; a group's time is
        // rounds of its resident workgroups times the chunk with its extra
        // planes.  FP64 tiles: the groups are built with 4 wavefronts and hold
        // three workgroups per CU.  FP32: one, three and four, and the three
        // groups weigh as fitted; the default stays where nothing is 3 %
        // better.  Over 27 sizes from 32^3 to 256^3, SSPRK3, RKN4 and RKN5,
        // the pick is within 1 % (FP64) and 2 % of the fastest of 20 shapes on
        // average and never more than 3 % behind automatic chunks on 64 x 8
        // tiles (7 % over 40 other sizes).  Those take 2.2 to 3.4 times as
        // long at 32^3, 1.1 to 1.3 at 96^3, and are the fastest at 110^3 to
        // 120^3 (chunks of 4 or 8 planes there: up to 1.27 times as long).
        const int n = boxes[0].n(2);
        if (!gw_groups || integrator == 11 || boxes.size() > 1 || n > 256) return c;
        const bool wide = tile_lo || f64;
        auto group_cost = [&](int v, int z) {
            double planes;
            const TileVariant &t = kVariants[v];
            const long long nt = tiles(t.tx, t.nw * 64 / t.tx * t.ry, z, planes);
            auto rounds = [&](int per_cu) {
                return (double)((nt + (long long)per_cu * ncu - 1) / ((long long)per_cu * ncu));
            };
            if (wide) return rounds(3) * (z + 5) + 0.03 * planes * t.nw / ncu;
            return (v == 3 ? 2.25 * rounds(1) + 1.05 * rounds(3) + 2.8 * rounds(4)
                           : 4.8 * rounds(1) + 1.8 * rounds(3) + 0.9 * rounds(4)) * (z + 3);
        };
        auto chunk = [&](int v, int z) {
            const TileVariant &t = kVariants[v];
            return std::min(n, z > 0 ? z : auto_chunk(boxes, t.tx, t.nw * 64 / t.tx * t.ry, ncu));
        };
        c.variant = wide ? 0 : kDefaultVariant;
        const double keep = group_cost(c.variant, chunk(c.variant, 0)) * (wide ? 1. : 0.97);
        double bc = keep;
        for (int v : {wide ? 0 : kDefaultVariant, 3})
            for (int z : {0, 4, 8, 16, 32})
                if (const double m = group_cost(v, chunk(v, z)); m < bc) {
                    bc = m;
                    c.variant = v;
                    c.tz = chunk(v, z);
                }
        if (bc == keep) c.variant = kDefaultVariant;
        return c;
    }
    auto cost = [&](int v, int z) {
        double planes;
        const TileVariant &t = kVariants[v];
        const long long n = tiles(t.tx, t.nw * 64 / t.tx * t.ry, z, planes);
        const long long slots = (long long)ncu * std::max(1, 12 / t.nw);
        return (double)((n + slots - 1) / slots) * (z + R) +
               0.03 * planes * t.nw * t.ry / ncu;
    };
    // -1: no shape the rule would take is built.  Eight stencil components in
    // FP64 at radius 3 leave the 32 x 8 tile alone; such levels keep the
    // default, for which the launch takes the nearest built shape.
    auto best_variant = [&](int z) {
        int bv = -1;
        for (int v = 0; v < kNVar; ++v)
            if (usable(v) && (bv < 0 || cost(v, z) < cost(bv, z))) bv = v;
        return bv;
    };
    // Fused first two stages: one workgroup per CU, a chunk costs 3R + 2
    // extra planes.  Against separate stages on the default shape: SSPRK3 on
    // tiles of the stored type, two fields, 342 against 492 us at 256^3 (FP32
    // + bf16), 563 against 899 us (FP64), 65 against 89 and 89 against 120 at
    // 128^3.  RKN up to radius 2 only: FP64 (one field at 256^3 326 against
    // 394 us, two fields 662 against 826), and FP32 on large levels, for two
    // fields (415 against 493 us at 256^3, equal at 200^3) or one at radius 1
    // (214 against 243; at radius 2 equal at 256^3 and slower below).  FP64
    // tiles of stored pairs, and ensembles (1.57 against 1.42 ms for 64
    // boxes): slower.
    const bool pays = boxes.size() == 1 && maxn >= 64 && !tile_lo &&
                      (integrator == 10 ||
                       (R <= 2 &&
                        (f64 || (maxn >= 224 && (nfields > 1 || R == 1)))));
    if (fused != 0 && can_fuse && (fused > 0 || pays)) {
        double bc = 1e30;
        int bv = -1, bz = maxn;
        // The widest tile that still gives half the CUs work at 8 planes.
        for (int v = kNVar - 1; v >= 0; --v) {
            double p;
            if (fused_ty[v] == 0) continue;
            if (bv < 0 || tiles(64, fused_ty[bv], std::min(8, maxn), p) < ncu / 2) bv = v;
        }
        for (int k = 1; k <= maxn; ++k) {
            const int z = (maxn + k - 1) / k;
            if (z < 4 && k > 1) break;
            double p;
            const long long n = tiles(64, fused_ty[bv], z, p);
            const double m = (double)((n + ncu - 1) / ncu) * (z + 3 * R + 2);
            if (m < bc) {
                bc = m;
                bz = z;
            }
        }
        c.fused = 1;
        c.fused_variant = bv;
        c.tz = bz;
        // The remaining stages take the chunk of the fused pass.  Several
        // components in FP64: eight rows unless it is the shortest (RKN4 of
        // two fields 306 us unfused, 324 with the model's 64 x 4 and 298 with
        // 64 x 8 at 176^3; 743 to 662 at 256^3, 53 to 50 at 80^3).
        const int v = best_variant(bz);
        if (v >= 0 && (usable16 || bz <= 4)) c.variant = v;
        return c;
    }
    double planes;
    const long long ntile32 =
        boxes.size() == 1 ? tiles(64, 8, std::min(32, maxn), planes) : 0;
    bool fills = ntile32 >= ncu;
    if (!fills && 8 * ntile32 >= 7LL * ncu) {
        // One tile short of that (129^3 to 136^3, 255 tiles): on the model's
        // 16-plane chunks of 32 x 8 tiles one field takes up to 1.27 times as
        // long as on automatic chunks (RKN4 at radius 3 in FP64 108 against 85
        // us at 134^3), and so do two fields as long as the automatic chunks
        // are resident at once (FP32 + bf16 RKN4 128 against 109 us at 134^3;
        // 130 against 134 at 136^3, where they are not; FP64 leapfrog 79
        // against 82 at 134^3).
        const int z = auto_chunk(boxes, 64, 8, ncu);
        fills = nfields == 1 || (!f64 && tiles(64, 8, z, planes) <= 3LL * ncu);
    }
    if (fills) {
        // A level that gives every CU a tile of 32 planes (138^3 and up): the
        // model below counts rounds of an occupancy it guesses, and a wrong
        // guess costs a last round that is nearly empty (one field at radius
        // 3: 144 us against 116 at 160^3, 575 against 492 at 300^3).
        // Automatic chunks give every kernel four rounds or more.  Two rows
        // per thread for one field at radius 1 or in leapfrog from 200^3 up
        // (138 against 156 us, 104 against 112, equal from 256^3), else 8
        // wavefronts.
        c.tz = 0;
        const bool two = nfields == 1 && (R == 1 || integrator == 11) &&
                         2 * ntile32 >= 5LL * ncu;
        c.variant = two && stage_built[4] ? 4 : kDefaultVariant;
        return c;
    }
    if (boxes.size() == 1) {
        double bc = 1e30;
        for (int z = 4; z < 2 * maxn; z *= 2) {
            const int zz = std::min(z, maxn), v = best_variant(zz);
            if (v >= 0 && cost(v, zz) < bc) {
                bc = cost(v, zz);
                c.variant = v;
                c.tz = zz;
            }
        }
        // The model counts a plane of a 64 x 4 tile like one of 64 x 8, but
        // with its ring the first loads 2.1 cells per cell (radius 2), the
        // second 1.6: on 16 planes, where that is most of the work, several
        // components in FP64 are faster on the default (112^3 two fields in
        // FP32CS: RKN4 104 against 90 us, SSPRK3 107 against 93; 128^3 108
        // against 102 and 108 against 99).  Shorter chunks are not (104^3 82
        // against 85 us).
        if (!usable16 && c.variant == 0 && c.tz >= 16) {
            c.variant = kDefaultVariant;
            c.tz = 0;
        }
        return c;
    }
    // Many boxes: the chunk by the cells a CU gets, the shape with the least
    // padding.  From a sweep of 48 shapes over 220 layouts of 2 to 64 boxes of
    // 12^3 to 150^3 cells, six of all projects, integrators and precisions
    // each (1320 levels): the pick is 3 % behind the fastest of the 48 on
    // average and 15 % faster than 64 x 8 tiles on automatic chunks (41 levels
    // are 3 to 13 % slower, near the cuts).  A thread with short queues (one
    // field at radius 1, or in stored FP32 but for SSPRK3) takes two rows, and
    // chunks of 4 planes up to 3.1 M cells (from 2.0 to 2.7 M 1.02 of the
    // fastest on average, 8 planes 1.05).  The others keep automatic chunks of
    // 64 x 8 tiles from 2.1 to 3.1 M cells, where 4, 8 and those are within
    // 3 % on average and single levels up to 1.17 behind, but FP64, where 8
    // planes of 32 x 8 are ahead from 1.6 M cells on (1.03 of the fastest,
    // 64 x 8 1.06).  Weights per padded cell: what 64 x 8 tiles may pad more
    // and still be as fast.  Large levels of two fields in stored FP32 run
    // without the XCD ranges (39.5 M cells in boxes 16..64 wide: 2.38 against
    // 2.45 ms for three SSPRK3 stages), all others with them (FP64: up to 1.36
    // times as long without).
    long long cells = 0;
    for (const Box3 &b : boxes) cells += b.vol();
    const long long k = cells / (1024LL * ncu);
    const bool light = nfields == 1 && (R == 1 || (!f64 && !tile_lo && integrator != 10));
    c.persistent = k < 24 ? 1 : 0;
    c.xcd_split = nfields > 1 && !f64 && !tile_lo && k >= 56 ? 0 : 1;
    if (!light && !f64 && k >= 8 && k < 12) return c;
    c.tz = k < (light ? 12 : f64 ? 6 : 8) ? 4 : k >= 56 && nfields == 1 && R > 1 ? 16 : 8;
    c.tz = std::min(c.tz, maxn);
    const double weight[kNVar] = {light ? 1. : 1.08, 1., 0.,
                                  light ? (f64 ? 1.05 : 1.2) : !f64 ? 1.3 : R < 3 ? 1. : 1.15,
                                  light ? 0.9 : 1.};
    double bw = 1e30;
    for (int v = 0; v < kNVar; ++v) {
        const TileVariant &t = kVariants[v];
        if (!stage_built[v] || weight[v] == 0.) continue;
        (void)tiles(t.tx, t.nw * 64 / t.tx * t.ry, c.tz, planes);
        const double w = planes * t.nw * t.ry * weight[v];
        if (w < bw) {
            bw = w;
            c.variant = v;
        }
    }
    if (bw == 1e30) c = LaunchCfg{kDefaultVariant, 0, -1, -1, -1, 0, -1};
    return c;
}

}  // namespace shm
