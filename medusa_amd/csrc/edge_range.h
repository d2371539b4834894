// Walking ranges of the edge arrays by 32-bit positions.  An array may end anywhere below 2^32, so a
// position past the end of a range is never formed: it could wrap round to one before the end.
#pragma once

#include <cstdint>

namespace medusa {

#if defined(__HIPCC__)
#define MDS_HD __host__ __device__
#else
#define MDS_HD
#endif

// Whether at + off lies before `end` (at <= end).
MDS_HD inline bool lies_before(uint32_t at, uint32_t off, uint32_t end) { return off < end - at; }

// at + off, or `end` where that does not lie before it (at <= end).
MDS_HD inline uint32_t advance_to(uint32_t at, uint32_t off, uint32_t end) {
    return lies_before(at, off, end) ? at + off : end;
}

// Bounds of part `part` of [begin, begin + count) cut into `parts` (at most 65535) parts of equal length but
// for the last ones, which may be shorter or empty.  No product of these passes 2^32.
struct EdgePart {
    uint32_t lo, hi;
};
MDS_HD inline EdgePart edge_part(uint32_t begin, uint32_t count, uint32_t part, uint32_t parts) {
    if (!count) return {begin, begin};
    const uint32_t per = (count - 1) / parts + 1, at = part * per;
    const uint32_t lo = at < count ? at : count, left = count - lo;
    return {begin + lo, begin + lo + (left < per ? left : per)};
}

}  // namespace medusa
