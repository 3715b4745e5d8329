// Which tile a workgroup takes, so that tiles which read the same weights meet in one XCD's L2 and every XCD has its share of
// them.  Plain C++, for the device and for the host.
#pragma once
#ifdef __HIPCC__
#define OJK_HD __host__ __device__ __forceinline__
#else
#define OJK_HD inline
#endif

// Row tiles x token tiles x K slices of a product, grid [8 ceil(row_tiles / 8) x token_tiles, slices]; workgroups are dealt to
// the eight XCDs in turn by their linear number.  Whole groups of eight row tiles: one of each group per XCD, its token
// tiles one after another.  The row tiles left over (all of them, where they are fewer than eight): the slices' tiles in a
// row, cut into eight runs whose lengths differ by one at most, a run per XCD.  Left to one XCD per row tile as well, 256
// rows would run on two XCDs (256 x 4096 at 2048 tokens 45 us, 31 dealt out) and 17 row tiles on one at 1.5 times the
// others' load (2176 x 4096 at 333 tokens 37, now 31); all tiles in eight runs cost 2 - 3 us where there are whole groups
// (6914 x 2816 at 333 tokens 38 against 35).
// Workgroups without a tile come last on their XCD, which deals its workgroups to its shader engines in turn, whatever they
// do: where every slice ended in some that return at once, one engine got more tiles than it has CUs and ran a second round
// beside idle ones (5312 x 9984 at 333 tokens, 252 tiles: 112 us, 83 with them last; 3090 x 14336 at 513: 139, 98).
// `i`: the workgroup's place among its XCD's.
OJK_HD bool ojk_spread(unsigned xcd, unsigned i, unsigned row_tiles, unsigned token_tiles, unsigned slices, unsigned& row,
                       unsigned& token, unsigned& slice) {
    const unsigned group = (row_tiles >> 3) * token_tiles, whole = group * slices;   // one slice's tiles in whole groups, and all
    if (i < whole) {
        slice = i / group;
        i -= slice * group;
        row = xcd + 8u * (i / token_tiles);
        token = i % token_tiles;
        return true;
    }
    const unsigned total = (row_tiles & 7u) * token_tiles * slices, base = total >> 3, more = total & 7u;
    i -= whole;
    if (i >= base + (xcd < more ? 1u : 0u)) return false;
    const unsigned piece = xcd * base + (xcd < more ? xcd : more) + i, run = piece / token_tiles;
    token = piece - run * token_tiles;
    slice = run % slices;
    row = (row_tiles & ~7u) + run / slices;
    return true;
}
