// qs_digits.hpp -- mixed-radix digits of an index on the device.
#ifndef QPP_AMD_QS_DIGITS_HPP_
#define QPP_AMD_QS_DIGITS_HPP_

#include <hip/hip_runtime.h>

#include <cstdint>
#include <utility>
#include <vector>

namespace qs_digits {

// Mixed-radix digits, the last one fastest.  mag[k] = 2^32 / dim[k] rounded
// up makes umulhi(v, mag) = v / dim exact while v * dim < 2^32, which the
// host checks (digits_fit); dimensions of 1 are left out.
constexpr int kMaxDigits = 40;
struct Digits {
    using Index = uint32_t;
    uint32_t n;
    uint32_t dim[kMaxDigits], mag[kMaxDigits];
    uint64_t str[kMaxDigits];
};
// the same for any dimensions, by 64-bit division
struct WideDigits {
    using Index = uint64_t;
    uint32_t n;
    uint64_t dim[kMaxDigits], str[kMaxDigits];
};

// qubits whose digits stay where they are: the set bits of the mask
struct BitDigits {
    using Index = uint64_t;
    uint64_t mask;
};

__device__ __forceinline__ uint64_t offset_of(const BitDigits& g, uint64_t v) { return v & g.mask; }

__device__ __forceinline__ uint64_t offset_of(const Digits& g, uint32_t v) {
    uint64_t off = 0;
    for (int k = int(g.n) - 1; k >= 0; --k) {
        const uint32_t q = __umulhi(v, g.mag[k]);
        off += uint64_t(v - q * g.dim[k]) * g.str[k];
        v = q;
    }
    return off;
}

__device__ __forceinline__ uint64_t offset_of(const WideDigits& g, uint64_t v) {
    uint64_t off = 0;
    for (int k = int(g.n) - 1; k >= 0; --k) {
        off += (v % g.dim[k]) * g.str[k];
        v /= g.dim[k];
    }
    return off;
}

using DigitList = std::vector<std::pair<uint64_t, uint64_t>>;  // (dim, stride)

// false where a digit, their number or their product is out of reach of the
// 32-bit quotients
inline bool digits_fit(const DigitList& list, Digits* g) {
    g->n = 0;
    uint64_t count = 1;
    for (const auto& [dim, str] : list) {
        if (dim == 1) continue;
        if (g->n == kMaxDigits || dim >= (uint64_t{1} << 32) || count >= (uint64_t{1} << 32) / dim)
            return false;
        count *= dim;
        g->dim[g->n] = static_cast<uint32_t>(dim);
        g->mag[g->n] = static_cast<uint32_t>(((uint64_t{1} << 32) + dim - 1) / dim);
        g->str[g->n++] = str;
    }
    for (uint32_t k = 0; k < g->n; ++k)
        if (count * g->dim[k] > (uint64_t{1} << 32)) return false;
    return true;
}

inline WideDigits wide_digits(const DigitList& list) {
    WideDigits g{};  // (at most 40 dimensions above 1 in an index below 2^40)
    for (const auto& [dim, str] : list) {
        if (dim == 1) continue;
        g.dim[g.n] = dim;
        g.str[g.n++] = str;
    }
    return g;
}

}  // namespace qs_digits

#endif  // QPP_AMD_QS_DIGITS_HPP_
