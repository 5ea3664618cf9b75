// mpmw_readback_plan.hpp -- the host side of the read-back: how arrays are cut
// into chunks, and the staging memory these take.  Needs no GPU.
#pragma once

#include <stddef.h>
#include <stdint.h>

#include <algorithm>
#include <vector>

namespace mpmw_internal {

enum : int32_t { kReadF32 = 0, kReadF64 = 1, kReadI32 = 2, kReadZero = 3 };

// One host array of n x comp values: component c from device array src[c]
// (float or double, widened to double; int32 as it is, comp 1), plus 1 where
// bit c of `ones` is set; kReadZero: zeros.
struct ReadArray {
    void *dst = nullptr;
    int32_t comp = 1, kind = kReadF64;
    uint32_t ones = 0;
    const void *src[9] = {};
};

// A part of one array on its way out: `count` rows from row i0 on, at byte
// `at` of the chunk.
struct ReadPiece {
    const void *src[9];
    int64_t i0;
    uint64_t at;
    int32_t count, comp, kind;
    uint32_t ones;
};
constexpr int kReadPieces = 24;
struct ReadTable {
    ReadPiece p[kReadPieces];
};

// (dst, src, bytes), src null for zeros.
struct HostMove {
    char *dst;
    const char *src;
    size_t bytes;
};

struct ReadChunk {
    ReadTable t{};
    int np = 0;
    size_t bytes = 0;
    std::vector<HostMove> moves;   // src: the offset in the chunk
};

struct ReadPlan {
    std::vector<ReadChunk> chunks;
    std::vector<HostMove> zeros;
    // a staging area for the chunk under way and one for the chunk before it
    size_t areas = 0, area = 0;
};

// The arrays cut into chunks of whole rows, at most `most` bytes each.
inline ReadPlan plan_read_back(const std::vector<ReadArray> &arrays, int64_t n, size_t most) {
    ReadPlan r;
    for (const ReadArray &a : arrays) {
        if (!a.dst || n <= 0) continue;
        const size_t row = a.kind == kReadI32 ? sizeof(int32_t) : sizeof(double) * (size_t)a.comp;
        if (a.kind == kReadZero) {
            r.zeros.push_back({(char *)a.dst, nullptr, row * (size_t)n});
            continue;
        }
        for (int64_t i = 0; i < n;) {
            if (r.chunks.empty() || r.chunks.back().np == kReadPieces || r.chunks.back().bytes + row > most)
                r.chunks.emplace_back();
            ReadChunk &c = r.chunks.back();
            const int64_t k = std::min<int64_t>(n - i, (int64_t)((most - c.bytes) / row));
            ReadPiece &p = c.t.p[c.np++];
            for (int q = 0; q < a.comp; ++q) p.src[q] = a.src[q];
            p.i0 = i;
            p.at = c.bytes;
            p.count = (int32_t)k;
            p.comp = a.comp;
            p.kind = a.kind;
            p.ones = a.ones;
            c.moves.push_back({(char *)a.dst + row * (size_t)i, (const char *)c.bytes, row * (size_t)k});
            c.bytes += (row * (size_t)k + 255) & ~(size_t)255;
            i += k;
        }
    }
    for (const ReadChunk &c : r.chunks) {
        size_t pow2 = 1u << 20;
        while (pow2 < c.bytes) pow2 *= 2;
        r.area = std::max(r.area, pow2);
    }
    r.areas = std::min<size_t>(r.chunks.size(), 2);
    return r;
}

// The plan and its staging memory, get(bytes) true when it is there: chunks of
// 32 MB, of 1 MB when there is no pinned memory for those.  The caller finds
// out from `get` that there was none at all.
template <typename Get> ReadPlan stage_read_back(const std::vector<ReadArray> &arrays, int64_t n, Get get) {
    ReadPlan r = plan_read_back(arrays, n, 32u << 20);
    if (r.chunks.empty() || get(r.areas * r.area)) return r;
    r = plan_read_back(arrays, n, 1u << 20);
    (void)get(r.areas * r.area);
    return r;
}

}  // namespace mpmw_internal
