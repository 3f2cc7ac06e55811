// The order in which the workgroups of a prefill GEMM take its tiles. No device
// code: the launcher and the kernel share it, and a host program can check it.
#pragma once

namespace qwen_hip {

// Tile order. Workgroup w runs on XCD w % 8 (round-robin dispatch). The XCDs
// form 8 / f groups of f: group i takes the row tiles i, i + 8 / f, ... and its
// XCDs split the column tiles by residue mod f, so each W tile is fetched by
// 8 / f XCDs and each A row by f. Short prompts (few row tiles, bound by the
// weights) send every W tile to one XCD (f = 8); with 4 or more row tiles per
// XCD its 32 CUs share rows and columns within the L2 at f = 1 (gate/up of 3968
// rows 93 us, 107 at f = 8). Another f is taken only where it saves a round: 5 row
// tiles of 64 in gate/up at f = 4 give half of the XCDs 36 workgroups for their
// 32 CUs, 23 us instead of 13.
struct GemmMap {
    int mtiles, ntiles, splits, f, per;  // per: row tiles of a group
    unsigned magic;                      // 2^32 / per rounded up (per > 1)
    GemmMap(int M, int N, int BM, int BN, int k_splits) {
        mtiles = (M + BM - 1) / BM;
        ntiles = N / BN;
        splits = k_splits;
        f = mtiles <= 4 ? 8 : mtiles <= 8 ? 4 : mtiles < 25 ? 2 : 1;
        for (int g : {8, 4, 2, 1})
            if (rounds(g) < rounds(f)) f = g;
        per = rows(f);
        magic = unsigned(((1ull << 32) + per - 1) / per);
    }
    int rows(int g) const { return (mtiles + 8 / g - 1) / (8 / g); }
    long tiles(int g) const { return long(rows(g)) * ((ntiles + g - 1) / g); }  // of the fullest XCD, per K split
    long rounds(int g) const { return (tiles(g) * splits + 31) / 32; }
    long rounds() const { return rounds(f); }
    unsigned groups() const { return unsigned(8 * tiles(f)); }
};

// Row tile and column tile of workgroup w; the grid is rounded up, so either
// may lie past the last.
struct MapTile {
    int mt, nt;
};
constexpr MapTile map_tile(unsigned w, int f, int per, unsigned magic) {
    const unsigned xcd = w % 8, slot = w / 8;
    // slot / per and the rest: the product's upper half is the quotient or,
    // where slot x per passes 2^32, at most one more.
    int cc = int(slot), rr = 0;
    if (per > 1) {
        cc = int((static_cast<unsigned long long>(slot) * magic) >> 32);
        rr = int(slot) - cc * per;
        if (rr < 0) --cc, rr += per;
    }
    const int shift = 31 - __builtin_clz(unsigned(f));
    return {int(xcd >> shift) + (8 >> shift) * rr, int(xcd & unsigned(f - 1)) + f * cc};
}

}  // namespace qwen_hip
