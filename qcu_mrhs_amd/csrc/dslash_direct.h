// dslash_direct.h -- the operator applied to the caller's per-RHS vectors.
#pragma once

#include "dslash.h"
#include "layout.h"

namespace qcu {

struct OperatorArgs {
    PtrTable out, in;      // R vectors [parity][Vh][4][Nc] (full) or [Vh][4][Nc], stored in `prec`
    const void *gauge;     // [4][2][Vh][Nc][Nc] in `prec`
    const void *clover;    // null, or the term's blocks of both parities in `prec` (full only)
    double coef;           // full: out_p = A_pp x_p + coef D_p x_{1-p}; else out = coef D x
    Geom g;
    int Nc, R;
    bool full;
    int parity;            // output parity of a half vector
    int dagger;
    int prec;              // kSingle or kDouble
};

// The lane kernel is the one chosen for the shape and the vectors allow reading them in place (16-byte
// aligned; no output overlaps an input or another output)
bool operator_direct_supported(const OperatorArgs &a);
hipError_t launch_operator_direct(const OperatorArgs &a, hipStream_t stream);

}  // namespace qcu
