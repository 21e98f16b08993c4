// Which kernels a key switch takes, by the shape of the call: host arithmetic
// alone, so that the rules can be checked without a GPU.  `tiles` counts the
// 4096-residue limb tiles of a launch, all its ciphertexts and rotations; n2 is
// log2 of the row length (7: N <= 2^14, 8: N <= 2^16, 9: N = 2^17).
#pragma once
#include <cstddef>

namespace ck {

inline size_t limb_tiles(size_t limbs, size_t n_cts, unsigned logn) { return (limbs * n_cts) << (logn - 12); }

// The fused row kernel (k_row_mac) transforms a tile's digits one after another
// in one workgroup, the separate kernels spread them over the chip: with many
// digits and few tiles the chain is what the call waits for.  Measured, one
// launch's key switch with separate kernels / fused, us: 34 digits, N = 2^13, 16
// tiles 117 / 161, 32 tiles 144 / 169, 64 tiles 188 / 182; 11 digits, 10 tiles
// 61.7 / 70.0, 20 tiles 69.1 / 74.5, 32 tiles 87.8 / 81.8; 23 digits, 30 tiles
// 141 / 148, 60 tiles 173 / 159; 6 digits never behind.
inline bool row_mac_pays(size_t dnum, size_t tiles) { return dnum <= 8 || tiles >= 2 * dnum; }

// Rotations of hoisted digits: the fused kernel (k_row_rotate) reads a tile's
// digits and keys one after another, in runs that shorten with the row length;
// the separate MAC streams them over the whole chip and reads each digit once
// for four exponents.  Few digits, or several exponents that find the digits in
// L2, and enough tiles are what the fused one needs.  Separate / fused, us:
//   N = 2^13: 11 digits, 16 tiles 29.4 / 33.6, 32 tiles 36.6 / 34.8; 23 digits, 30
//   tiles 42.9 / 53.0, 120 tiles 65.8 / 57.3;
//   N = 2^15: 11 digits, 64 tiles 42.0 / 46.7, 128 tiles 55.7 / 49.4; 16 digits, 264
//   tiles of three exponents 131 / 151, 704 of two 214 / 205; 25 digits, 800 tiles
//   of one exponent 353 / 384, 1600 of two 701 / 595;
//   N = 2^17: 3 digits, 352 tiles 82.9 / 91.2, 704 tiles 131 / 116; 5 digits and 16
//   ciphertexts, three exponents 2597 / 2756, four 3680 / 3623; 8 digits, four
//   exponents 2715 / 3015; 16 digits, 4 ciphertexts, one exponent 697 / 798, four 2861
//   / 2496.
// `rotations` counts ciphertexts times exponents.
inline bool row_rotate_pays(size_t dnum, size_t limbs, size_t rotations, size_t exponents, unsigned logn) {
    const size_t tiles = limb_tiles(limbs, rotations, logn);
    if (logn >= 17) {
        if (dnum <= 3) return dnum <= 2 || tiles > 512 || exponents >= 4;
        return dnum <= 6 ? exponents >= 4 : dnum >= 9 && exponents > 1 && rotations >= 16;
    }
    if (dnum <= 4) return true;
    if (logn >= 15) return dnum <= 12 ? tiles > 8 * dnum : exponents > 1 && tiles > 20 * dnum;
    return tiles > (dnum <= 12 || exponents > 1 ? 2 : 3) * dnum;
}

// Row tiles halve where whole ones would not give every CU more than one: a lone
// tile's eight waves compete for issue slots that idle CUs have.  4 ciphertexts
// at N = 2^13: tensor (72 whole tiles) 29.3 -> 23.0 us, key products of 2 digits
// (104) 19.4 -> 15.4 us.  Above, whole tiles read keys in longer runs.
constexpr size_t kHalfTiles = 256;
// Half tiles of a row of 512 read keys in runs of 32 bytes.  Whole / half, us: 11
// digits, 160 tiles 160 / 176; 4 digits, 128 tiles 72 / 67.
inline size_t row_mac_half_tiles(unsigned n2) { return n2 <= 8 ? kHalfTiles : 128; }
// k_row_rotate reads its digits so as well.  N = 2^13, 23 digits, 120 tiles 68.8 /
// 57.3; N = 2^14, 25 digits, 200 tiles 136 / 151; N = 2^15, 11 digits, 128 tiles
// 49.4 / 56.9, 6 digits, 40 tiles 36.8 / 35.1; N = 2^16, 10 digits, 160 tiles 60.2 /
// 86.1; N = 2^17, 6 digits, 160 tiles 66.2 / 98.1.
// Up to 4 digits the latency of the first loads weighs more: 4 digits, 256 tiles
// at N = 2^13 47.3 / 44.2.
inline size_t row_rotate_half_tiles(size_t dnum, unsigned n2) {
    return n2 <= 7 ? (dnum <= 4 ? 256 : 160) : n2 == 8 ? 96 : 0;
}

// ModDown of several jobs of one shape in one launch, or each in its own
// (workgroups of the smallest job).  One launch saves the tails of small ones.
// Where the jobs add their permuted b components it spreads the XCDs over every
// job's gathers, which large jobs feel.  In one / each its own, us: four exponents
// at N = 2^16, 32 limbs, 4 ciphertexts (2048 workgroups) 1070 / 1185, 16 ciphertexts
// (8192) 3980 / 3870, without b components 3617 / 3707; three at 12 limbs, 16
// ciphertexts 1236 / 1178; two at N = 2^17, 12 limbs, 8 ciphertexts (8192) 890 / 896.
inline bool moddown_together(size_t jobs, size_t workgroups, bool permuted) {
    return jobs < 3 || workgroups < 8192 || !permuted;
}

}  // namespace ck
