// The whole-ray walk (march.hpp, walk) against the reference's loop body taken
// step by step (ray_step with exact std::min and NaN handling) on the host:
// outcome, t (bits), leaf index and word must agree for every finite ray,
// with and without a level-of-detail cut-off and in both address widths.
// Usage: walk_test WORDS.bin LEVELS RAYS_PER_CLASS [loose]
// (loose: a tree with far words in one-word slots, for the 64-bit walk alone)
#include <cmath>
#include <cstdint>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <fstream>
#include <random>
#include <vector>

#include "march.hpp"

using namespace svo::march;

namespace {

long compared = 0, leaves = 0, lods = 0;

template <bool Lod, typename Addr>
bool same(const std::vector<uint32_t> &w, int levels, const float o[3], const float d[3], float rs) {
    Ray<uint32_t> r;
    ray_init(r, w.data(), o[0], o[1], o[2], d[0], d[1], d[2], rs);
    std::vector<uint64_t> mem(24, ~uint64_t(0));
    const Stack<uint32_t> stk(mem.data(), 1, 22, 0);
    uint32_t normal = 0, leaf = 0;
    float t = 0, t2 = 0;
    int code;
    do {
        code = ray_step<true, false, uint32_t, true, 1>(r, w.data(), stk, normal, t, leaf);
    } while (code == kRunning);
    Ray<Addr> q;
    ray_init(q, w.data(), o[0], o[1], o[2], d[0], d[1], d[2], rs);
    std::vector<unsigned char> lds(size_t(levels) * (sizeof(Addr) + 2));  // exactly the walk's entries
    const PathStack<Addr> path(lds.data(), 1, levels, 0);
    WalkEnd<Addr> end;
    const int code2 = walk<Lod, false, Addr>(q, w.data(), path, t2, end);
    compared++;
    leaves += code == kLeaf;
    lods += code == kLod;
    if (code == code2 && (code == kMiss || std::memcmp(&t, &t2, 4) == 0) &&
        (code != kLeaf || (uint64_t(end.leaf()) == leaf && w[size_t(end.leaf())] == normal)))
        return true;
    std::printf("differ: o %a %a %a d %a %a %a rs %a: %d %a %u / %d %a\n", o[0], o[1], o[2], d[0], d[1], d[2], rs, code, t,
                leaf, code2, t2);
    return false;
}

}  // namespace

int main(int argc, char **argv) {
    if (argc < 4) return 2;
    std::ifstream f(argv[1], std::ios::binary);
    std::vector<uint32_t> w;
    f.seekg(0, std::ios::end);
    const size_t bytes = size_t(f.tellg());
    w.resize(bytes / 4 + 1, 0xFFFFFFFFu);  // the spare word of device arrays
    f.seekg(0);
    f.read(reinterpret_cast<char *>(w.data()), std::streamsize(bytes));
    const int levels = std::atoi(argv[2]);
    const long n = std::atol(argv[3]);
    const bool loose = argc > 4;
    std::mt19937 g(7);
    std::uniform_real_distribution<float> U(0, 1);
    std::normal_distribution<float> N;
    for (long i = 0; i < 5 * n; ++i) {
        float o[3], d[3];
        for (int k = 0; k < 3; ++k) {
            switch (i % 5) {
                case 0:  // from outside toward the middle
                    o[k] = 1.5f + (U(g) - 0.5f) * 1.8f;
                    d[k] = 1.5f + (U(g) - 0.5f) * 0.9f - o[k];
                    break;
                case 1:  // from inside, any direction
                    o[k] = 1.0f + U(g);
                    d[k] = N(g);
                    break;
                case 2:  // origins on cell corners, axis-aligned and diagonal directions: ties
                    o[k] = 1.0f + float(int(U(g) * 64)) / 64;
                    d[k] = float(int(U(g) * 5) - 2);
                    break;
                case 3:  // huge and tiny components
                    o[k] = std::fmin(std::fmax(N(g) * std::pow(10.0f, U(g) * 40 - 20), -1.2e30f), 1.2e30f);
                    d[k] = N(g) * std::pow(10.0f, U(g) * 60 - 30);
                    break;
                default:  // nearly parallel rays just above a cell plane
                    o[k] = k == 1 ? 1.0f + float(int(U(g) * 256)) / 256 + N(g) * 1e-6f : 0.9f;
                    d[k] = k == 1 ? N(g) * 1e-4f : U(g) + 0.1f;
            }
        }
        if (!ray_finite(o[0], o[1], o[2], d[0], d[1], d[2])) continue;
        const float rs = i % 3 == 0 ? 0.0f : (i % 3 == 1 ? U(g) * 0.02f : U(g) * 0.5f);
        if (!same<true, uint64_t>(w, levels, o, d, rs) || (rs == 0.0f && !same<false, uint64_t>(w, levels, o, d, rs)))
            return 1;
        if (loose) continue;
        if (!same<true, uint32_t>(w, levels, o, d, rs) || (rs == 0.0f && !same<false, uint32_t>(w, levels, o, d, rs)))
            return 1;
    }
    std::printf("ok %ld walks, %ld leaf hits, %ld cut-offs\n", compared, leaves, lods);
    return 0;
}
