// CPU-only check of the dispatch rules (tr-infer_amd/csrc/geometry.hpp) at sizes where both forms were
// timed on an MI355X: the rule takes the faster one.  Built with g++ by tests/test_geometry.py; the
// argument names the rule.  Prints "ok" and the number of cases, or the first failing one and exits 1.
#include <cstdio>
#include <cstring>
#include <initializer_list>

#include "geometry.hpp"

using namespace trk::geo;

static int n = 0, bad = 0;
static void expect(bool got, bool want, const char* what, unsigned a, unsigned b, unsigned c) {
    n++;
    if (got == want) return;
    bad++;
    std::printf("FAIL %s (%u, %u, %u): %d\n", what, a, b, c, (int)got);
}

// (m, E, H): few experts leave the matrix-core tiles without workgroups, whatever the rows
static void router() {
    const unsigned valu[][3] = {{160, 16, 2048}, {200, 64, 2048}, {200, 128, 2560}, {300, 128, 2048}, {400, 128, 2048},
                                {200, 256, 2048}, {176, 256, 1024}, {160, 384, 2048}, {500, 64, 2048}, {1023, 32, 2048},
                                {800, 16, 2560}, {300, 16, 256}, {500, 64, 320}, {200, 128, 192}, {200, 128, 640},
                                {159, 512, 2048}, {500, 512, 2000}};
    const unsigned mfma[][3] = {{160, 512, 2048}, {176, 384, 2048}, {300, 256, 2048}, {500, 128, 2048}, {500, 256, 2560},
                                {500, 512, 2560}, {512, 512, 2048}, {1500, 16, 2048}, {3072, 512, 2048}, {300, 128, 320},
                                {300, 256, 192}, {800, 64, 640}};
    for (auto& c : valu) expect(router_on_mfma(c[0], c[1], c[2]), false, "router_on_mfma", c[0], c[1], c[2]);
    for (auto& c : mfma) expect(router_on_mfma(c[0], c[1], c[2]), true, "router_on_mfma", c[0], c[1], c[2]);
}

// (tiles, quantising workgroups beside them): 256-wide chunks where both find CUs
static void chunks() {
    const unsigned wide[][2] = {{256, 0}, {160, 1}, {208, 1}, {224, 1}, {1, 1}};
    const unsigned narrow[][2] = {{257, 0}, {256, 1}, {240, 1}, {320, 0}};
    for (auto& c : wide) expect(router_wide_chunks(c[0], c[1] != 0), true, "router_wide_chunks", c[0], c[1], 0);
    for (auto& c : narrow) expect(router_wide_chunks(c[0], c[1] != 0), false, "router_wide_chunks", c[0], c[1], 0);
}

// n workgroups of t threads as rows of a grid: none lost, under 2^32 threads a row
static void grids() {
    const unsigned long long ns[] = {1, 255, 256, 8388600, 8388607, 8388608, 8392609, 16777216, 100000000};
    for (unsigned t : {256u, 512u})
        for (unsigned long long v : ns) {
            const Grid2 g = grid_run(v, t);
            expect((unsigned long long)g.x * t <= 0xffffffffull && (unsigned long long)g.x * g.y >= v &&
                           (g.y == 1 ? g.x == v : g.x % 8 == 0 && (unsigned long long)g.x * (g.y - 1) < v),
                   true, "grid_run", (unsigned)v, t, g.x);
        }
}

// (blocks of 128 weight rows, of 32 activation rows): the 32-row form up to three workgroups per CU and where
// the 64-row one would run empty halves
static void gemm() {
    const unsigned narrow[][3] = {{96, 1, 32}, {96, 8, 32}, {192, 4, 32}, {768, 1, 32}, {782, 1, 32}, {1172, 1, 16},
                                  {1940, 1, 32}, {192, 5, 32}, {192, 5, 16}, {32, 24, 16}, {1024, 3, 32}};
    const unsigned wide[][3] = {{96, 16, 32}, {192, 8, 32}, {192, 8, 16}, {768, 2, 32}, {1940, 2, 16}, {16, 64, 32}, {1024, 3, 16}};
    for (auto& c : narrow) expect(gemm_narrow(c[0], c[1], c[2]), true, "gemm_narrow", c[0], c[1], c[2]);
    for (auto& c : wide) expect(gemm_narrow(c[0], c[1], c[2]), false, "gemm_narrow", c[0], c[1], c[2]);
}

// (GEMV workgroups, TQ codec or 0, k): the tiles from the GEMV's third round of 1024, before it on GGUF formats
// and short columns
static void tiles() {
    const unsigned gemv[][3] = {{1791, 0, 4096}, {1791, 0x410, 80}, {1792, 0x420, 3072}, {1792, 0x420, 1536}, {1792, 0x520, 1024},
                                {2048, 0x520, 2560}, {1920, 0x520, 2560}, {2048, 0x820, 4096}, {1800, 0x820, 10240},
                                {1792, 0x810, 768}, {1920, 0x420, 10240}, {2060, 0x820, 10240}};
    const unsigned mfma[][3] = {{1792, 0, 256}, {1792, 0, 10240}, {1792, 0x420, 1024}, {1792, 0x510, 768}, {1792, 0x810, 512},
                                {1792, 0x820, 768}, {2048, 0x420, 3072}, {2064, 0x520, 2560}, {2064, 0x820, 2048},
                                {2320, 0x820, 10240}, {2080, 0x420, 10240}, {98304, 0x520, 2560}};
    for (auto& c : gemv) expect(gemv_tiles(c[0], c[1], c[2]), false, "gemv_tiles", c[0], c[1], c[2]);
    for (auto& c : mfma) expect(gemv_tiles(c[0], c[1], c[2]), true, "gemv_tiles", c[0], c[1], c[2]);
}

// (rows x passes, activation rows a pass, bits, blocks a row): row quads from enough blocks
static void quads() {
    const unsigned strips[][4] = {{1024, 1, 4, 10}, {64, 2, 5, 16}, {1024, 1, 8, 32}, {1024, 2, 8, 20}, {320, 4, 8, 16}, {2048, 1, 5, 48},
                                  {2048, 1, 8, 64}, {2048, 2, 8, 48}, {2048, 4, 4, 20}, {2064, 4, 4, 320}, {12288, 1, 5, 80}};
    const unsigned quad[][4] = {{1024, 1, 4, 40}, {64, 2, 5, 40}, {1024, 1, 8, 48}, {1024, 2, 8, 40}, {320, 4, 8, 20}, {2048, 1, 5, 128},
                                {2048, 1, 8, 128}, {2048, 2, 4, 80}, {2048, 4, 4, 40}, {320, 1, 8, 320}, {640, 2, 8, 320}};
    for (auto& c : strips) expect(gemv_quads(c[0], c[1], c[2], c[3]), false, "gemv_quads", c[0], c[1], c[3]);
    for (auto& c : quad) expect(gemv_quads(c[0], c[1], c[2], c[3]), true, "gemv_quads", c[0], c[1], c[3]);
}

int main(int argc, char** argv) {
    const char* what = argc > 1 ? argv[1] : "";
    if (!std::strcmp(what, "router")) router();
    if (!std::strcmp(what, "chunks")) chunks();
    if (!std::strcmp(what, "grids")) grids();
    if (!std::strcmp(what, "gemm")) gemm();
    if (!std::strcmp(what, "tiles")) tiles();
    if (!std::strcmp(what, "quads")) quads();
    if (!n || bad) return 1;
    std::printf("ok %d\n", n);
    return 0;
}
