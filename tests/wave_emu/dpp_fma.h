// dpp_fma.h of the kernels for the emulated workgroup: the same operations
// without the machine's instructions.
#pragma once

#include "kernels.h"

namespace magma_amd {

template <int K0, int K1, int N, class T>
inline void fmac_row(T (&a)[N], T x0, T x1, T l)
{
    struct Rows { T x0, x1; };
    const emu::Slot *s = emu::exchange(Rows{x0, x1});
    const int row = emu::cur & 48;
    for (int k = K0; k < K1; ++k) {
        const Rows r = emu::lane<Rows>(s, row + (k & 15));
        a[k] = std::fma(k < 16 ? r.x0 : r.x1, l, a[k]);
    }
}

inline GDoublePtr opaque(GDoublePtr p) { return p; }
inline LDoublePtr opaque(LDoublePtr p) { return p; }
inline int opaque(int x) { return x; }

}  // namespace magma_amd
