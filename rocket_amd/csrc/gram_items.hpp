// Work items of the Gram kernels over 256 x 256 partial tiles (the pattern
// store's in store.hip, the pointer table's in ncc.hip): which patterns an
// item loads, which 128 x 64 block each of its 8 waves multiplies, and where
// its partial goes.
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>

namespace prnu {

constexpr int kGramTile = 256;  // patterns per side of a partial tile

// Linear index over the upper triangle (row-major, I <= J) -> (I, J).
__host__ __device__ inline int2 tri_tile(int t, int nt) {
    int I = 0;
    while (t >= nt - I) {
        t -= nt - I;
        ++I;
    }
    return make_int2(I, I + t);
}

// Work items.  The LDS stage holds four quarters of 128 pattern rows; a
// wave multiplies the 128 rows of one quarter by 64 rows of another (a
// 128 x 64 block of the output), and waves 2k, 2k+1 together cover the
// 128 x 128 sub-tile of one quarter pair (unit k of the item).  The triangle
// of Q = ceil(count / 128) quarters has Q (Q + 1) / 2 units (quarter pairs
// qa <= qb); an item holds at most 4 units over at most 4 quarters, so a
// slab needs at least ceil(Q (Q + 1) / 8) items.  With m = floor(Q / 2)
// full 256-row tiles, per slab:
//  - m (m - 1) / 2 off-diagonal tiles (I, J): quarters 2I, 2I+1, 2J, 2J+1,
//    all four units of the pair;
//  - Q even: ceil(6 m / 8) diagonal packs.  A diagonal tile needs 3 units,
//    the 6 wave blocks (wr, wc) = (0,0) (0,1) (0,2) (0,3) (1,2) (1,3); the
//    6m such blocks are numbered e = 6 d + l and pack p gives block 8p + w
//    to wave w.  Eight consecutive blocks span at most two diagonal tiles
//    d0 = 8p / 6 and d0 + 1, whose quarters fill the LDS.
//  - Q odd (last quarter L = 2m alone in tile m): m "edge" items d with
//    quarters 2d, 2d+1, L and units (2d,2d) (2d,2d+1) (2d,L) (2d+1,L), then
//    ceil((m + 1) / 4) items of the remaining one-quarter units
//    (2j+1, 2j+1), j < m, and (L, L), four per item.
// A last item of one or two one-quarter units would leave six or four waves
// idle.  It takes the same unit(s) of ks = 4 or 2 consecutive slabs instead:
// LDS quarter k holds unit k % (4 / ks) at slab k / (4 / ks) of the group, so
// every wave pair multiplies one unit of one slab, adds it up in that slab's
// own order and writes that slab's own partial (the same bits as one slab at
// a time), and the item runs once per ks slabs (slab_split, ItemIndex), where
// that shortens the launch (choose_slab).  A set
// of at most 128 patterns then multiplies with all eight waves instead of two,
// and 300 patterns take 1.5 items per slab instead of 2 (whole 256-row tiles:
// 3; 300 of 640x480 over a pointer table in FP32: 1,056 -> 585 us).
// Both reach the bound: m(m-1)/2 + ceil(6m/8) = ceil(Q(Q+1)/8) for even Q,
// m(m-1)/2 + m + ceil((m+1)/4) = ceil(Q(Q+1)/8) for odd Q.  The output of
// unit (qa, qb) is the sub-tile at rows 128 (qa & 1), columns 128 (qb & 1)
// of partial tile (qa / 2, qb / 2).
struct ItemWaves {
    int q[4];             // first pattern (relative to the range) of LDS rows [128 k, 128 k + 128)
    int nq;               // quarters loaded: LDS rows [0, 128 nq)
    int a_off, b_off;     // this wave's first A row / first B row in LDS
    int out_tile;         // triangle index of the tile this wave writes, -1: idle wave
    int out_off;          // offset of the wave's 128 x 64 block inside that tile
    int ks;               // slabs of this item (1, 2 or 4)
    int kq[4];            // slab of LDS quarter k within them
    int kw;               // slab of this wave within them
};

// First pattern of LDS row `row` (a multiple of 64); no indexed private array.
__host__ __device__ __forceinline__ int row_pattern(const ItemWaves &w, int row) {
    const int k = row >> 7;
    const int q0 = w.q[0], q1 = w.q[1], q2 = w.q[2], q3 = w.q[3];
    return (k < 2 ? (k == 0 ? q0 : q1) : (k == 2 ? q2 : q3)) + (row & 127);
}

__host__ __device__ __forceinline__ int tri_index(int I, int J, int nt) { return I * nt - I * (I - 1) / 2 + (J - I); }

__host__ __device__ __forceinline__ void item_tiles(ItemWaves &r, int x, int y) {
    r.q[0] = x * kGramTile;
    r.q[1] = x * kGramTile + 128;
    r.q[2] = y * kGramTile;
    r.q[3] = y * kGramTile + 128;
}

// Slabs the last item of a slab of the triangle can take at once: 4 or 2 where it
// holds one or two one-quarter units (odd Q, (m + 1) mod 4 = 1 or 2), else 1.
__host__ __device__ inline int slab_split(int count) {
    const int Q = (count + 127) >> 7, m = Q >> 1;
    if (!(Q & 1)) return 1;
    const int rest = (m + 1) & 3;
    return rest == 1 ? 4 : rest == 2 ? 2 : 1;
}

// Item u of a slab of the triangle of `count` patterns, the last one taking ks
// slabs (1 or slab_split(count)) (nt = ceil(count /
// 256) partial tiles), for wave `wave`.
__host__ __device__ __forceinline__ ItemWaves item_waves(int u, int count, int wave, int ks) {
    ItemWaves r;
    r.ks = 1;
    r.kq[0] = r.kq[1] = r.kq[2] = r.kq[3] = r.kw = 0;
    const int Q = (count + 127) >> 7, m = Q >> 1, nt = (count + kGramTile - 1) / kGramTile;
    const int wr = wave >> 2, wc = wave & 3;
    const int toff = m * (m - 1) / 2;
    if (u < toff) {
        int I = 0, t = u;
        while (t >= m - 1 - I) {
            t -= m - 1 - I;
            ++I;
        }
        const int J = I + 1 + t;
        item_tiles(r, I, J);
        r.nq = 4;
        r.a_off = wr * 128;
        r.b_off = kGramTile + wc * 64;
        r.out_tile = tri_index(I, J, nt);
        r.out_off = wr * 128 * kGramTile + wc * 64;
        return r;
    }
    const int p = u - toff;
    r.out_tile = -1;
    r.a_off = r.b_off = r.out_off = 0;
    if (!(Q & 1)) {
        const int d0 = (8 * p) / 6;
        const int dl = min(m - 1, (8 * p + 7) / 6);
        item_tiles(r, d0, dl > d0 ? d0 + 1 : d0);
        r.nq = dl > d0 ? 4 : 2;
        const int e = 8 * p + wave;
        if (e >= 6 * m) return r;
        const int d = e / 6, l = e - 6 * (e / 6);
        const int bwr = l < 4 ? 0 : 1;
        const int bwc = l < 4 ? l : l - 2;
        const int base = (d - d0) * kGramTile;
        r.a_off = base + bwr * 128;
        r.b_off = base + bwc * 64;
        r.out_tile = tri_index(d, d, nt);
        r.out_off = bwr * 128 * kGramTile + bwc * 64;
        return r;
    }
    const int k = wave >> 1, h = wave & 1;
    if (p < m) {  // edge item of tile d = p: quarters 2d, 2d+1, L
        const int d = p;
        r.q[0] = d * kGramTile;
        r.q[1] = d * kGramTile + 128;
        r.q[2] = r.q[3] = m * kGramTile;
        r.nq = 3;
        const int sa = k == 3 ? 1 : 0;           // A quarter: 2d for units 0..2, 2d+1 for unit 3
        const int sb = k == 0 ? 0 : k == 1 ? 1 : 2;
        r.a_off = sa * 128;
        r.b_off = sb * 128 + h * 64;
        r.out_tile = tri_index(d, k < 2 ? d : m, nt);
        r.out_off = sa * 128 * kGramTile + (k == 1 ? 128 : 0) + h * 64;
        return r;
    }
    // one-quarter units 4j' .. 4j'+3 of the list (2j+1, 2j+1) j < m, then (L, L)
    const int j0 = 4 * (p - m);
    const int units = 4 / ks;
    const bool split = ks > 1 && m + 1 - j0 <= units;  // the last item
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const int j = min(j0 + (split ? i % units : i), m);
        r.q[i] = j * kGramTile + (j < m ? 128 : 0);
        r.kq[i] = split ? i / units : 0;
    }
    r.ks = split ? ks : 1;
    r.kw = split ? k / units : 0;
    r.nq = split ? 4 : min(4, m + 1 - j0);
    const int j = j0 + (split ? k % units : k);
    if (j > m) return r;
    r.a_off = k * 128;
    r.b_off = k * 128 + h * 64;
    r.out_tile = tri_index(j, j, nt);
    r.out_off = (j < m ? 128 * kGramTile + 128 : 0) + h * 64;
    return r;
}

// Items per slab of the triangle of `count` patterns (item_waves).
__host__ __device__ inline int tri_items_per_slab(int count) {
    const int Q = (count + 127) >> 7, m = Q >> 1;
    return m * (m - 1) / 2 + ((Q & 1) ? m + (m + 4) / 4 : (6 * m + 7) / 8);
}


// Items of a triangle (ntb == 0) or of a rectangle of nt x ntb tiles over S
// slabs.  The Tn items that take one slab at a time come first, slab by slab,
// the slabs of a round of 8 to ids that differ mod 8 (workgroup ids go to the
// XCDs round-robin), so the items of a slab share one XCD's L2; then the
// split item, one per ks slabs.
struct ItemIndex {
    int Tn, ks, S;   // ks = 1: no split item
    __host__ __device__ ItemIndex(int items, int ks_, int S_) : Tn(items - (ks_ > 1 ? 1 : 0)), ks(ks_), S(S_) {}
    __host__ __device__ int64_t groups() const { return ks > 1 ? (S + ks - 1) / ks : 0; }
    // ids handed out (a multiple of 8 with `remap`), padding included
    __host__ __device__ int64_t ids(bool remap) const {
        const int64_t S8 = remap ? (S + 7) / 8 * 8 : S;
        return Tn * S8 + (remap ? (groups() + 7) / 8 * 8 : groups());
    }
    __host__ __device__ int64_t items() const { return (int64_t)Tn * S + groups(); }
    // items of the XCD that gets the most (ids mod 8 = 0)
    __host__ __device__ int64_t xcd_items() const { return (int64_t)Tn * ((S + 7) / 8) + (groups() + 7) / 8; }
    // id -> item u and its first slab s; false: padding
    __host__ __device__ bool at(int64_t id, bool remap, int &u, int &s) const {
        const int64_t S8 = remap ? (S + 7) / 8 * 8 : S, normal = Tn * S8;
        if (id >= normal) {
            u = Tn;
            s = (int)(id - normal) * ks;
        } else if (remap) {
            const int local = (int)(id >> 3);
            u = local % Tn;
            s = (local / Tn) * 8 + (int)(id & 7);
        } else {
            u = (int)(id % Tn);
            s = (int)(id / Tn);
        }
        return s < S;
    }
};

// A rectangle of nt x ntb tiles: item u = tile (u / ntb, u % ntb).
__host__ __device__ __forceinline__ ItemWaves rect_waves(int u, int ntb, int wave) {
    ItemWaves r;
    r.ks = 1;
    r.kq[0] = r.kq[1] = r.kq[2] = r.kq[3] = r.kw = 0;
    const int wr = wave >> 2, wc = wave & 3;
    item_tiles(r, u / ntb, u - (u / ntb) * ntb);
    r.nq = 4;
    r.a_off = wr * 128;
    r.b_off = kGramTile + wc * 64;
    r.out_tile = u;
    r.out_off = wr * 128 * kGramTile + wc * 64;
    return r;
}


// Blocks of K per slab, at most `longest` (0: no limit), and per set g the
// slabs splits[g] (in: slab_split, out: that or 1) its last item takes, for
// products of format `precision`: store.hip.
int64_t choose_slab(const int *items, int *splits, const int *tiles, const int64_t *nkb, int ngroups, int precision,
                    int cus, size_t max_bytes, int64_t longest);
int device_cus(int device);
// FP64 sum of the S partials of every element and the NCC epilogue: store.hip.
int launch_tri_reduce(const float *partials, int S, int nt, int count, const double *sum, const double *sumsq,
                      const float *scale, double *out, int64_t ld, hipStream_t st);

}  // namespace prnu
