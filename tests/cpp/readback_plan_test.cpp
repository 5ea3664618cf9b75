// The read-back's plan on the host: the chunks are filled as the kernel fills
// them and moved out as the host moves them, for row counts around a chunk, and
// with staging memory that is refused at first or altogether.
#include <cstdio>
#include <cstdlib>
#include <cstring>

#include "mpmw_readback_plan.hpp"

using namespace mpmw_internal;

static int fails = 0;
#define EXPECT(c)                                                      \
    do {                                                               \
        if (!(c)) {                                                    \
            std::printf("line %d: %s\n", __LINE__, #c);                \
            ++fails;                                                   \
        }                                                              \
    } while (0)

static double value(int array, int c, int64_t i) { return 1000.0 * array + c + 0.25 * (double)i; }

static void run(int64_t n, int refuse) {
    // a vector of doubles, a matrix of floats with the identity, ints, zeros,
    // an array without a destination
    std::vector<std::vector<double>> f64(3, std::vector<double>(n));
    std::vector<std::vector<float>> f32(9, std::vector<float>(n));
    std::vector<int32_t> ids(n);
    for (int64_t i = 0; i < n; ++i) {
        for (int c = 0; c < 3; ++c) f64[c][i] = value(1, c, i);
        for (int c = 0; c < 9; ++c) f32[c][i] = (float)c + (float)(i % 64);
        ids[i] = (int32_t)(n - i);
    }
    std::vector<double> pos(3 * n, 7.0), F(9 * n, 7.0), none(6 * n, 7.0);
    std::vector<int32_t> id(n, 7);
    std::vector<ReadArray> arrays(5);
    arrays[0].dst = pos.data(); arrays[0].comp = 3;
    for (int c = 0; c < 3; ++c) arrays[0].src[c] = f64[c].data();
    arrays[1].dst = F.data(); arrays[1].comp = 9; arrays[1].kind = kReadF32; arrays[1].ones = 0x111u;
    for (int c = 0; c < 9; ++c) arrays[1].src[c] = f32[c].data();
    arrays[2].dst = id.data(); arrays[2].kind = kReadI32; arrays[2].src[0] = ids.data();
    arrays[3].dst = none.data(); arrays[3].comp = 6; arrays[3].kind = kReadZero;
    arrays[4].comp = 3;

    std::vector<size_t> asked;
    std::vector<char> stage;
    bool have = false;
    const ReadPlan p = stage_read_back(arrays, n, [&](size_t bytes) {
        asked.push_back(bytes);
        have = (int)asked.size() > refuse;
        if (have) stage.resize(bytes);
        return have;
    });
    EXPECT(asked.size() == (refuse ? 2u : 1u));
    EXPECT(asked[0] <= (64u << 20) && (!refuse || asked[1] <= (2u << 20)));
    if (refuse > 1) {
        EXPECT(!have);
        return;
    }
    EXPECT(have && p.areas * p.area == stage.size());
    for (size_t k = 0; k < p.chunks.size(); ++k) {
        const ReadChunk &c = p.chunks[k];
        char *const out = stage.data() + (k % p.areas) * p.area;
        EXPECT(c.np >= 1 && c.np <= kReadPieces && c.bytes <= p.area);
        for (int q = 0; q < c.np; ++q) {
            const ReadPiece &r = c.t.p[q];
            EXPECT(r.count >= 1 && r.at % 256 == 0);
            for (int64_t e = 0; e < (int64_t)r.count * r.comp; ++e) {
                if (r.kind == kReadI32) {
                    EXPECT(r.at + 4 * e + 4 <= p.area);
                    ((int32_t *)(out + r.at))[e] = ((const int32_t *)r.src[0])[r.i0 + e];
                    continue;
                }
                const int64_t i = e / r.comp;
                const int cc = (int)(e - i * r.comp);
                double v = r.kind == kReadF64 ? ((const double *)r.src[cc])[r.i0 + i]
                                              : (double)((const float *)r.src[cc])[r.i0 + i];
                if (r.ones >> cc & 1u) v += 1.0;
                EXPECT(r.at + 8 * e + 8 <= p.area);
                ((double *)(out + r.at))[e] = v;
            }
        }
        for (const HostMove &m : c.moves) std::memcpy(m.dst, out + (size_t)m.src, m.bytes);
    }
    for (const HostMove &m : p.zeros) std::memset(m.dst, 0, m.bytes);
    bool same = true;
    for (int64_t i = 0; i < n; ++i) {
        for (int c = 0; c < 3; ++c) same &= pos[3 * i + c] == value(1, c, i);
        for (int c = 0; c < 9; ++c) same &= F[9 * i + c] == (double)c + (double)(i % 64) + (c % 4 == 0 ? 1.0 : 0.0);
        for (int c = 0; c < 6; ++c) same &= none[6 * i + c] == 0.0;
        same &= id[i] == ids[i];
    }
    EXPECT(same);
}

int main() {
    // 1 MB holds 43,690 rows of a vector and 14,563 of a matrix, 32 MB 1,398,101 and 466,033
    for (int64_t n : {(int64_t)1, (int64_t)255, (int64_t)14563, (int64_t)14564, (int64_t)43690, (int64_t)43691,
                      (int64_t)466033, (int64_t)500009, (int64_t)1400003})
        for (int refuse : {0, 1, 2}) run(n, refuse);
    // nothing to read asks for nothing
    int calls = 0;
    std::vector<ReadArray> empty(2);
    (void)stage_read_back(empty, 10, [&](size_t) { ++calls; return false; });
    (void)stage_read_back({}, 0, [&](size_t) { ++calls; return false; });
    EXPECT(calls == 0);
    if (!fails) std::printf("ok\n");
    return fails ? 1 : 0;
}
