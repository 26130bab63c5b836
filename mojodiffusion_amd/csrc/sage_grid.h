// sage_grid.h — which block of its launch's work a workgroup takes.  Plain arithmetic without any include, so that a
// host compiler can be asked for the same mapping (tests/test_grid_mapping.py).
#pragma once

namespace sage {

// Workgroup `id` of n -> item: consecutive ids go to the 8 XCDs in turn, and each XCD takes a contiguous range of items,
// so that those of a head, which all walk the same rows, share one L2.
__host__ __device__ inline int xcd_item(int id, int n) {
    const int per = n >> 3, extra = n & 7, xcd = id & 7;
    return xcd * per + (xcd < extra ? xcd : extra) + (id >> 3);
}

// The backward's grid: `heads` heads, each with tq blocks of query rows (dQ) and tk blocks of keys (dK, dV), the first lq
// and lk of which hold rows that count.  Those come first, dQ in front of dK/dV, each kind in even ranges over the XCDs;
// blocks of padding, which only store zeros, come last.  In ranges over all blocks, padding included, an XCD that does not
// get whole heads has up to twice another's blocks that count.  Launch 1 + 2 at 128 channels, rows / rows that count, us, so
// -> now:  12 heads  2304/1612 94.5 -> 75.8   4608/2304 149.8 -> 136.1   4608/3225 263.7 -> 230.9   4608/3916 373.5 -> 346.5
//          30 heads  1248/624 45.2 -> 38.8    1248/873 65.6 -> 61.1      4608/3225 580.8 -> 565.8
// Whole heads per XCD are even as they are and keep their order: the padding last measured 5 % behind that to 5 % ahead
// there (16 heads 4608/2304 158.1 -> 166.3, 24 heads 1248/873 57.1 -> 59.0, 24 heads 4608/3225 455.8 -> 432.2).
struct BwdBlock { bool dkdv; int head, tile; };
__host__ __device__ inline BwdBlock bwd_block(int id, int heads, int tq, int lq, int tk, int lk) {
    if ((heads & 7) == 0) lq = tq, lk = tk;
    const int nq = heads * lq, nk = heads * lk;
    if (id < nq) {
        const int i = xcd_item(id, nq);
        return BwdBlock{false, i / lq, i % lq};
    }
    if (id < nq + nk) {
        const int i = xcd_item(id - nq, nk);
        return BwdBlock{true, i / lk, i % lk};
    }
    const int j = id - nq - nk, pq = heads * (tq - lq);
    return j < pq ? BwdBlock{false, j / (tq - lq), lq + j % (tq - lq)} : BwdBlock{true, (j - pq) / (tk - lk), lk + (j - pq) % (tk - lk)};
}

// The encoders' grid where rows are rotated by tables.  What reads the same table rows — the Q and K blocks of one run of
// rows of one head, in every batch that shares the tables — is a set; its `members` go to one XCD, one soon after the other,
// so that the rows come from its L2 after the first.  Sets run over the heads first and are taken 32 at a time, member by
// member: consecutive ids read neighbours in memory, as everywhere in the quantizers.
constexpr int kSetGroup = 32;                    // (a multiple of the XCDs)
struct SetMember { int set, member; };
__host__ __device__ inline SetMember set_member(int id, int members) {
    const int at = id % (kSetGroup * members);
    return SetMember{id / (kSetGroup * members) * kSetGroup + at % kSetGroup, at / kSetGroup};
}
__host__ __device__ inline long long set_grid(long long sets, int members) {
    return (sets + kSetGroup - 1) / kSetGroup * kSetGroup * members;
}

}  // namespace sage
