// The route rules of the key switch (routes.hpp) for the CPU tests.
#include "../../ccmm-rs_amd/csrc/routes.hpp"

extern "C" {
int emu_row_mac_pays(size_t dnum, size_t tiles) { return ck::row_mac_pays(dnum, tiles); }
int emu_row_rotate_pays(size_t dnum, size_t limbs, size_t n_cts, size_t exponents, unsigned logn) {
    return ck::row_rotate_pays(dnum, limbs, n_cts * exponents, exponents, logn);
}
size_t emu_limb_tiles(size_t limbs, size_t n_cts, unsigned logn) { return ck::limb_tiles(limbs, n_cts, logn); }
size_t emu_half_tiles(int rotate, size_t dnum, unsigned n2) {
    return rotate ? ck::row_rotate_half_tiles(dnum, n2) : ck::row_mac_half_tiles(n2);
}
int emu_moddown_together(size_t jobs, size_t workgroups, int permuted) {
    return ck::moddown_together(jobs, workgroups, permuted != 0);
}
}
