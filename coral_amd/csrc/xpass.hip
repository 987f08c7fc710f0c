// Dispatch of the wavefront x passes over the line length, and its shortest
// lengths (xpass_impl.hpp holds the kernels and the radix plans).
#include "xpass_impl.hpp"

namespace coral {

XLENGTHS_B(XEXTERN)
XLENGTHS_C(XEXTERN)
XLENGTHS_D(XEXTERN)
XLENGTHS_E(XEXTERN)
XLENGTHS_A(XINSTANCE)

bool launch_xbwd_wave(hipStream_t st, const FFTPlan &px, const double2 *G, double *phys, int nbatch, long long nlines,
                      int nkx) {
    if (nbatch < 1 || nlines < 1 || 3 * nkx != px.N || !px.tw) return false;
    switch (px.N) {
#define XCASE(n) \
    case n: return xbwd_n<n>(st, px.tw, G, phys, nbatch, nlines);
        XLENGTHS(XCASE)
#undef XCASE
    default: return false;
    }
}

bool launch_xfwd_wave(hipStream_t st, const FFTPlan &px, const double *phys, double2 *H, int nbatch, long long nlines,
                      int nkx) {
    if (nbatch < 1 || nlines < 1 || 3 * nkx != px.N || !px.tw) return false;
    switch (px.N) {
#define XCASE(n) \
    case n: return xfwd_n<n>(st, px.tw, phys, H, nbatch, nlines);
        XLENGTHS(XCASE)
#undef XCASE
    default: return false;
    }
}

bool launch_xpass_wave(hipStream_t st, const FFTPlan &px, const XPassArgs &a) {
    if (a.nfull < 1) return false;
    switch (px.N) {
#define XCASE(n) \
    case n: return xpass_len<n>(st, px, a);
        XLENGTHS(XCASE)
#undef XCASE
    default: return false;
    }
}

}  // namespace coral
