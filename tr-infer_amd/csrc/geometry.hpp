// Launch geometry and workspace extents of the MoE kernels, as plain host arithmetic (no HIP
// types), shared by the launchers, the workspace sizing of trk_create and a CPU-only check that
// sweeps shapes (tests/geometry_check.cpp).  Every grid a launcher builds and every workspace
// extent a kernel indexes is computed here, so a grid that addresses strips past F or a buffer
// sized below what a dispatch writes shows up on the host, without a GPU.  The rules that choose between
// two kernels by size are here too (tests/dispatch_rules_check.cpp: at sizes where both were timed).
#pragma once

#include <stdint.h>

namespace trk {
namespace geo {

constexpr uint32_t KMAX = 32;      // router.rs:6 MOE_K_MAX: stride of the per-token id / weight rows
constexpr uint32_t ITEM_ROWS = 16; // rows of a grouped work item (one 16-row MFMA tile)
constexpr uint32_t CHUNK = 64;     // tokens per dispatch chunk (one wave's lane mask)
constexpr uint32_t DN_R = 4;       // output rows per decode down workgroup

struct Caps {  // what trk_create sizes for (m_max rows, k_cap selections per token)
    uint32_t H, E, F, m_max, k_cap;
};

inline uint64_t ent_cap(const Caps& c) { return (uint64_t)c.m_max * c.k_cap; }
// work items: every non-empty expert's entries in items of <= 16 rows (at most E + entries / 16 of
// them), then the shared expert's tokens in items of <= 16
inline uint64_t item_cap(const Caps& c) {
    return c.E + (ent_cap(c) + ITEM_ROWS - 1) / ITEM_ROWS + (c.m_max + ITEM_ROWS - 1) / ITEM_ROWS + 1;
}
inline uint64_t items_max(uint32_t E, uint32_t m, uint32_t kcap) {
    const uint64_t ent = (uint64_t)m * kcap;
    const uint64_t nonempty = ent < E ? ent : E;
    return nonempty + ent / ITEM_ROWS + (m + ITEM_ROWS - 1) / ITEM_ROWS;
}
// activation rows of the down input: one per entry and one per token (shared), the decode slots
// (K_MAX routed + the shared one, two levels each), and a TQ batch of up to 16 tokens run as
// per-token decodes (k_cap + 1 slots of two rows per token)
inline uint64_t act_rows(const Caps& c) {
    const uint64_t a = ent_cap(c) + c.m_max, d = (uint64_t)(KMAX + 1) * 2;
    const uint64_t t = 2ull * (c.m_max < 16 ? c.m_max : 16) * (c.k_cap + 1);
    const uint64_t ad = a > d ? a : d;
    return ad > t ? ad : t;
}
inline uint64_t yent_rows(const Caps& c) { return ent_cap(c) + c.m_max; }
// dispatch chunks of 64 tokens, and the per-(chunk, expert) offsets the split dispatch writes
inline uint32_t chunks(uint32_t m) { return (m + CHUNK - 1) / CHUNK; }
inline uint64_t doff_elems(uint32_t m, uint32_t E) { return (uint64_t)chunks(m) * E; }
inline bool dispatch_split(uint32_t m) { return m >= 256; }

// MFMA gate/up: grid.x column blocks of F / 16 / grid.x strips, four waves taking every fourth.
// A wave's strips run one after another, so with few items (one or two rounds of workgroups on
// the GPU) the kernel time is a wave's chain of strips: 128-wide blocks below 2048 rows (M = 512:
// gate/up 210 -> 197 us), 256-wide from 2048 (config 4: 507 against 512 us with 128), 64-wide for
// small batches.
inline uint32_t mfma_gateup_cols(uint32_t m, uint32_t F) {
    return m >= 2048 && F % 256 == 0 ? F / 256 : m >= 64 && F % 128 == 0 ? F / 128 : F / 64;
}
inline uint32_t mfma_gateup_strips(uint32_t m, uint32_t F) { return F / 16 / mfma_gateup_cols(m, F); }
// MFMA gate/up over item pairs from 2048 rows: two items of one expert run as one 32-row tile
// (v_mfma_i32_32x32x32_i8) in a workgroup of eight waves, each taking every eighth strip of the
// column block.  The pair's activations and scales take 40 H bytes of LDS, which leaves room for
// two workgroups per CU up to H = 2048.
inline bool gateup_pairs(uint32_t m, uint32_t H) { return m >= 2048 && H <= 2048; }
inline uint64_t gateup_pair_lds(uint32_t H) { return (uint64_t)H * 40; }
// a pair's workgroup takes 32 strips (four per wave) where F allows: the 80 KB of staged
// activations then serve twice the weights (config 4 gate/up 500 -> 483 us against 16 strips)
inline uint32_t gateup_pair_cols(uint32_t m, uint32_t F) { return F % 512 == 0 ? F / 512 : mfma_gateup_cols(m, F); }
inline uint32_t gateup_pair_strips(uint32_t m, uint32_t F) { return F / 16 / gateup_pair_cols(m, F); }
// MFMA down: grid.x blocks of 256 or 64 output rows, four waves of 16-row strips
inline uint32_t mfma_down_cols(uint32_t m, uint32_t H) { return m >= 64 ? H / 256 : H / 64; }
inline uint32_t mfma_down_rows(uint32_t m, uint32_t H) { return H / mfma_down_cols(m, H); }
// MFMA down over item pairs (two items of one expert share each weight load, unpack and scale
// decode) from 256 rows: config 4's Q6_K down 457 -> 416 us, M = 512's Q4_K down 123 -> 120 us
inline bool down_pairs(uint32_t m) { return m >= 256; }
// streaming down: 4 waves of 64 / (2 NSB) units of 2 NSB lanes (half a superblock each)
inline uint32_t stream_down_rows_per_wg(uint32_t F) { return 4 * (64 / (2 * (F / 256))); }
inline uint32_t stream_down_cols(uint32_t H, uint32_t F) {
    const uint32_t r = stream_down_rows_per_wg(F);
    return (H + r - 1) / r;
}
// decode: gate/up (F / 16 strips, kcap + 1 slots), down H / 4 workgroups
inline uint32_t decode_gateup_strips(uint32_t F) { return F / 16; }
inline uint32_t decode_down_wgs(uint32_t H) { return H / DN_R; }

// TQ layer (k_tq.hip): gate/up strips of 16 over F twice (gate, up), down strips of 16 over H;
// grid.y: the decode slots (kcap + 1) or the work items
inline uint32_t tq_gateup_tiles(uint32_t F) { return 2 * F / 16; }
inline uint32_t tq_down_tiles(uint32_t H) { return H / 16; }

// A launch's workgroups over x and y: a launch holds less than 2^32 threads in x, and a kernel that numbers its
// workgroups in one run takes the rest as rows of y (x * y >= n; multiples of 8 in x keep id % 8 the XCD).
struct Grid2 {
    uint32_t x, y;
};
inline Grid2 grid_run(uint64_t n, uint32_t threads) {
    const uint64_t most = 0xffffffffull / threads / 8 * 8;
    if (n <= most) return Grid2{(uint32_t)n, 1};
    return Grid2{(uint32_t)most, (uint32_t)((n + most - 1) / most)};
}

// Router logits in gemm order (k_router.hip) from 64 rows: VALU tiles of 16 rows x 8 experts (x 2 where
// H is no multiple of 256), or matrix-core tiles of 32 x 32.
inline uint64_t router_valu_wgs(uint32_t m, uint32_t E, uint32_t H) {
    const uint64_t te = H % 256 == 0 ? 8 : 2;
    return (E + te - 1) / te * ((m + 15) / 16);
}
// A matrix-core tile takes as long however few they are (the walk of one workgroup: 16 us at H = 2048),
// while the VALU tiles' time goes with their workgroups per CU.  us, VALU / matrix cores, the kernel alone
// and in a layer (x quantised beside it), H = 2048:
//   up to a workgroup per CU: E = 64 x 200 rows 11.6 / 16.0 and 12.6 / 16.1, E = 16 x 800 11.7 / 16.0
//   and 15 / 18, E = 64 x 500 13.2 / 16.0 and 15.2 / 18.2;
//   up to two, from a few hundred rows on beside as many quantising workgroups: E = 128 x 400 (400 of
//   them) 14.3 / 15.9 and 16.9 / 17.8, E = 384 x 160 (480) 14.3 / 16.0 and 15.0 / 16.0, but E = 128 x 500
//   (512) 15.4 / 16.0 and 19.5 / 18.0, E = 256 x 256 (512) 14.6 / 16.0 and 18.5 / 16.8;
//   beyond: E = 512 x 160 (640) 18.2 / 15.9, x 300 27.7 / 18.5.
// H = 640, 320 and 192 (K-split slices): E = 64 x 500 (1024) 7.3 / 7.6, 5.1 / 5.8 and 4.1 / 4.7, E = 128 x
// 300 (1216) 9.6 / 7.6, 6.9 / 5.9 and 5.3 / 4.7.
inline bool router_on_mfma(uint32_t m, uint32_t E, uint32_t H) {
    if (m < 160 || H % 64) return false;
    const uint64_t valu = router_valu_wgs(m, E, H);
    if (H % 256) return valu > 1024;
    return valu > (m <= 400 ? 480u : m <= 1024 ? 256u : 0u);
}

// The matrix-core tiles walk 256-wide chunks (133 KB of LDS: a CU each) while they and what runs beside them
// have CUs of their own, else 128-wide ones (two tiles per CU).  In a layer the quantising workgroups carry
// the tiles' LDS too, in a few turns on the CUs that the tiles leave: an eighth of the GPU is enough, none
// is not.  us in a layer, 256 / 128 wide: E = 512, H = 2048 x 300 rows (160 tiles) 19.1 / 21.9, x 400
// (208) 18.9 / 22.1, x 500 (256) 26.4 / 21.9; the tiles alone x 500 18.9 / 21.9, x 640 (320) 33.7 / 29.2.
inline bool router_wide_chunks(uint64_t tiles, bool aux) { return tiles + (aux ? 32 : 0) <= 256; }

// trk_gemv tiles (k_gemm.hip) of 128 weight rows (rb blocks of them) x 32 activation rows (t32 blocks) or x 64.
// A 64-row workgroup serves two tiles from one unpacking and takes half as long again as a 32-row one (a
// third at kb 16); up to three per CU the 32-row form is ahead however they divide, beyond it where the
// 64-row form has empty halves.  us, 32 / 64 rows a workgroup:
//   2 and 1 per CU: [12288][2560] TQ5_32 x 128 rows 40 / 53; 3 and 2: x 256 53 / 65, [4096][4096] TQ5_16 x 768
//   147 / 154 and Q6_K 167 / 166 (kb 16: two resident, the third a second round, as dear as the 64-row form);
//   6 and 3: [12288][2560] TQ5_32 x 512 93 / 82, [24576][2048] Q4_K x 256 79 / 63, TQ5_16 x 256 137 / 105;
//   4 and 3: [24576][2048] Q4_K x 160 55 / 60, TQ5_16 x 160 95 / 103; 12 and 8: [131072][768] Q6_K x 96 125 / 112;
//   one block: [150016][2048] Q4_K x 8 (5 and 5) 62 / 93, [248320][2560] TQ8_32 x 8 (8 and 8) 162 / 233.
inline bool gemm_narrow(uint64_t rb, uint64_t t32, uint32_t kb) {
    const uint64_t c32 = (rb * t32 + 255) / 256, c64 = (rb * ((t32 + 1) / 2) + 255) / 256;
    return c32 <= 3 || (kb == 16 ? 3 * c32 <= 4 * c64 : 2 * c32 <= 3 * c64);
}

// trk_gemv on TQ strips of few rows: four rows a workgroup (gemv_quad_kernel) or a strip's sixteen.  Row quads put
// four times the workgroups on the GPU, two per CU at 2048 (row, pass) pairs, for staging that a strip does once:
// they are ahead where a row has enough blocks, earlier while each has a CU of its own and with more activation
// rows (more chains to share), later with 8 bits (the bytes summed besides).  us, strips / quads, at blocks:
//   a CU each, 1024 rows x 1: TQ4_32 10 3.2 / 3.4, 20 3.6 / 3.6, 40 4.1 / 3.8, 80 5.8 / 4.5; TQ8_32 20 3.6 / 3.8, 40
//   4.2 / 4.2, 64 5.0 / 4.6; 320 x 4: TQ8_32 10 4.1 / 4.7, 20 5.3 / 5.0, 40 6.6 / 5.3;
//   two per CU, 2048 rows x 1: TQ5_32 20 3.7 / 4.4, 64 5.3 / 5.2, 128 8.1 / 6.7; TQ8_32 64 5.1 / 5.5, 128 7.9 / 7.3;
//   x 4: TQ4_32 20 5.2 / 5.3, 40 6.5 / 5.7.  [320][10240] TQ8_32 at 1 / 2 / 4 rows 18.3 / 22.9 / 31.8 strips, 11.2 / 12.7
//   / 15.5 quads; beyond 2048, [12288][2560] TQ5_32 x 2 11.3 / 28.5.
// na: activation rows a pass (1, 2, 4).
inline bool gemv_quads(uint64_t row_passes, uint32_t na, uint32_t bits, uint32_t blocks) {
    if (row_passes > 2048) return false;
    if (row_passes <= 1024) return blocks >= (bits == 8 && na < 4 ? 40u : 20u);
    return blocks >= (na == 4 ? 40u : bits != 8 ? 64u : na == 2 ? 80u : 96u);
}

// trk_gemv of many activation rows: its passes of four rows x strips are so many GEMV workgroups, four resident
// per CU, so that it takes whole rounds of 1024; the tiles take as long for one row as for thirty-two.  The
// tiles take over in the third round, before it where they beat two rounds: GGUF formats, whose GEMV decodes
// more, and short columns, where the tiles' unpacking (dearer with more bits) is a smaller part.  us, GEMV /
// tiles, at workgroups:
//   GGUF from 1792: [4096][4096] Q6_K x 28 rows (1792) 89 / 76, [2560][2560] Q4_K x 48 (1920) 41 / 26;
//   TQ [4096][3072] 1792 / 2048 / 2304: TQ4_32 26.5 / 28.8, 29.1 / 28.7, 33.7 / 29.0; TQ5_32 28.1 / 33.3, 30.5 /
//   33.2, 35.1 / 33.3; TQ8_32 27.3 / 33.8, 30.1 / 33.6, 34.9 / 33.9; TQ5_16 48.7 / 52.9, 53.7 / 53.1, 61.0 / 53.0;
//   [256][k] at 1792: TQ4_32 k = 1024 11.6 / 11.5, 1536 15.4 / 15.9; TQ5_32 768 10.8 / 10.4, 1024 12.1 / 13.0;
//   TQ8_32 768 10.8 / 10.5, TQ8_16 512 11.3 / 11.5, 768 14.5 / 15.7;
//   longer ones: [320][10240] TQ4_32 1920 82 / 89, 2080 101 / 89; TQ5_32 1920 87 / 104, 2320 113 / 104; TQ8_32 2060
//   100 / 107, 2320 111 / 106.
inline bool gemv_tiles(uint64_t workgroups, uint32_t tq, uint32_t k) {  // tq: 0 for GGUF, else bits << 8 | kb
    const uint32_t bits = tq >> 8;
    if (tq == 0 || k <= (bits == 4 ? 1024u : tq == 0x810 ? 512u : 768u)) return workgroups >= 1792;
    if (bits == 4 && k <= 3072) return workgroups >= 1920;
    return workgroups > (bits == 8 && k > 3072 ? 2303u : 2048u);
}

// Every invariant a call of m rows with kcap selections per token relies on; returns nullptr when
// they hold, else what failed.  tq: the experts are TQ strips (k_tq.hip), not GGUF superblocks.
inline const char* check_call(const Caps& c, uint32_t m, uint32_t kcap, bool tq = false) {
    if (c.H == 0 || c.H % 256) return "H must be a multiple of 256";
    if (c.F == 0 || c.F % (tq ? 16 : 256)) return tq ? "F must be a multiple of 16" : "F must be a multiple of 256";
    if (m == 0 || m > c.m_max) return "m outside 1..m_max";
    if (kcap == 0 || kcap > c.k_cap || kcap > KMAX) return "kcap outside 1..k_cap";
    if ((uint64_t)m * kcap > ent_cap(c)) return "entries above the entry capacity";
    if (items_max(c.E, m, kcap) > item_cap(c)) return "work items above the item capacity";
    if ((uint64_t)m * kcap + m > act_rows(c) || (uint64_t)m * kcap + m > yent_rows(c))
        return "activation rows above capacity";
    if (doff_elems(m, c.E) > doff_elems(c.m_max, c.E)) return "dispatch offsets above capacity";
    if (tq) {
        if (tq_gateup_tiles(c.F) * 16 != 2 * c.F || tq_down_tiles(c.H) * 16 != c.H) return "TQ strips do not tile F / H";
        // decode: slots 0..kcap (the shared one last) in h / yent rows and in the [33][2] act rows
        if (m == 1 && ((uint64_t)kcap + 1 > yent_rows(c) || (uint64_t)(KMAX + 1) * 2 > act_rows(c)))
            return "decode slots above capacity";
        return nullptr;
    }
    {  // MFMA gate/up: the column blocks tile F's strips exactly, four waves each
        const uint32_t cols = mfma_gateup_cols(m, c.F), s = mfma_gateup_strips(m, c.F);
        if (cols == 0 || cols * s * 16 != c.F || s % 4) return "MFMA gate/up grid does not tile F";
        // the pairs' workgroups: eight waves over the block's strips (the launcher runs every item
        // on the 16-row path otherwise), and two workgroups' LDS per CU
        if (gateup_pairs(m, c.H) && gateup_pair_strips(m, c.F) % 8 == 0 && 2 * gateup_pair_lds(c.H) > 160 * 1024)
            return "MFMA gate/up pair LDS above 80 KiB";
    }
    {  // MFMA down: the row blocks tile H exactly, 16-row strips over four waves
        const uint32_t cols = mfma_down_cols(m, c.H), r = mfma_down_rows(m, c.H);
        if (cols == 0 || cols * r != c.H || r % 64) return "MFMA down grid does not tile H";
    }
    {  // streaming down: the row blocks cover H (the kernel guards rows past H)
        const uint32_t r = stream_down_rows_per_wg(c.F);
        if (r == 0 || (uint64_t)stream_down_cols(c.H, c.F) * r < c.H) return "stream down grid does not cover H";
    }
    if (m == 1) {  // decode: slots 0..kcap-1 and the shared slot, strips of F, rows of H
        if (decode_gateup_strips(c.F) * 16 != c.F) return "decode gate/up strips do not tile F";
        if (decode_down_wgs(c.H) * DN_R != c.H) return "decode down workgroups do not tile H";
        if ((uint64_t)(KMAX + 1) * 2 > act_rows(c)) return "decode activation slots above capacity";
    }
    return nullptr;
}

}  // namespace geo
}  // namespace trk
