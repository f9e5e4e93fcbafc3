// Host-side choice of the widths a contraction adds its weights in (no GPU code,
// so it is also built and tested on the CPU).
#pragma once
#include <cstdint>

namespace pggc {

constexpr int64_t C_TOP = 8192;  // largest bound of a coarse row merged in LDS

struct ContractWidths {
    bool small;   // coarse weights staged as int32: all weights sum to less than 2^31
    bool packed;  // big rows' tables with key and 32-bit sum in one word: they sum to less than 2^32
    bool sum32;   // 32-bit sums in LDS: C_TOP of the largest weight sum to less than 2^32
};

// nnz weights of at most wmax as unsigned values (a negative weight is huge; 1
// for unit weights); wsmall: they are known to sum to less than 2^31.
inline ContractWidths contract_widths(int64_t nnz, uint64_t wmax, bool wsmall) {
    const uint64_t m = nnz > 0 ? (uint64_t)nnz : 1;
    ContractWidths r;
    r.small = wsmall || wmax <= 0x7fffffffull / m;
    r.packed = r.small || wmax <= 0xffffffffull / m;
    r.sum32 = r.small || wmax <= 0xffffffffull / C_TOP;
    return r;
}

}  // namespace pggc
