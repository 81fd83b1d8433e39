// memrule.hpp -- when an optional copy of a context's arrays may take device memory (host only).
#pragma once
#include <cstddef>

namespace dndsr
{
// A copy may take a quarter of the free memory, and must leave what the context may still allocate on
// first use: at most about 14 KB a cell (p3 hexahedra: 7.6 for the viscous adjoint at 9 face points, 1.8
// for the LU-SGS blocks in both precisions, 2 for 50 Krylov vectors, 1.5 for two reconstructions, 0.8 for
// the scalar solve's rows).  Without the bound a copy that took the last memory made those allocations
// fail where they fit before.
inline bool roomForCopy(size_t freeBytes, size_t copyBytes, size_t nCell)
{
    constexpr size_t kLater = 16384;
    return copyBytes <= freeBytes / 4 && freeBytes - copyBytes >= kLater * nCell;
}
} // namespace dndsr
