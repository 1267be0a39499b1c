// The kernel-level GEMV of many activation rows: y[i][r] (+)= W[r] . x_i (gemm_tq_rows, gemv.rs:43-78)
// as int8 MFMA tiles, on TQ strips (codec.rs:1-46) or GGUF superblocks.
//
// A workgroup owns 128 weight rows x TOK activation rows and walks K in slices of 128 values.  Each
// slice's weights are unpacked once into an int8 operand image in LDS, beside the activations, and
// every wave runs 32 x 32 tiles from there: one v_mfma_i32_32x32x32_i8 (32x32x16 at kb 16) gives a
// block's exact dots; the reference's f32 chain
//     acc = fma(m, sx * sum, acc); acc = fma(float(dot), d * sx, acc)          (gemv.rs:141-148)
// then runs block by block, fma(m, u, acc) on the matrix cores (rank1).  The next slice's global
// loads are in flight during a slice.
// [12288][2560] TQ5_32 x 512 rows: 983 us as GEMV passes of 4 rows (each decoding the weights
// again) -> 82 us.  Of these about 60 are the tiles (without the staging) and 40 the staging alone.
// The staging counts its load instructions: row pairs' d and m and the whole plane chunk as wide loads
// instead of 2-byte ones took [12288][2560] TQ4_32 x 16 / 512 from 30 / 75 to 25 / 72 us and [24000][2560]
// TQ8_32 x 512 from 190 to 170.
#include "tq.hpp"

namespace trk {

typedef int v4i __attribute__((ext_vector_type(4)));
typedef int v16i __attribute__((ext_vector_type(16)));
typedef uint32_t u4v __attribute__((ext_vector_type(4)));
typedef u4v u4v_a2 __attribute__((aligned(2)));  // 16 bytes at a 2-byte aligned address

constexpr uint32_t GM_ROWS = 128;  // weight rows per workgroup
constexpr uint32_t GM_KS = 128;    // K values per slice

struct GemmArgs {
    const uint8_t* w;     // the matrix (item applied)
    uint64_t pitch;       // GGUF: bytes per row; TQ: bytes per 16-row strip
    uint32_t k, nb;       // k and blocks per row (k / KB)
    uint32_t r_lo, r_hi;  // output rows [r_lo, r_hi)
    const int8_t* q;      // [m][k], 16-byte aligned
    const float* s;       // [m][nb]
    const int32_t* su;    // [m][nb]
    uint32_t m;           // physical activation rows
    uint32_t tb, n;       // blocks of TOK activation rows; tiles
    int pair;
    float* y;
    uint32_t ldy;
    int accumulate;
};

// One thread's share of a slice's weights: loaded into registers, then unpacked into the operand
// image wb[piece][row] (piece p: values 16p .. 16p + 15 of the slice) and (d, m) per (block, row).
template <int GK, int KB>
struct GmW {
    static constexpr bool TQ = GK >= GK_TQ4;
    static constexpr uint32_t NBLK = GM_KS / KB;
    static constexpr uint32_t PW = GM_ROWS * 16 + 16;  // bytes per piece, padded off the banks' period
    using T = GvTQ<GK_TQ4 <= GK ? GK : GK_TQ4, KB>;
    // TQ: a unit is 16 bytes of a block's q chunk (4 rows x 4 values, two nibbles each at 4/5 bits)
    static constexpr uint32_t UPB = T::NCH * 4, NU = TQ ? 8 * NBLK * UPB / 256 : 0, ND = GM_ROWS / 2 * NBLK / 256;
    static constexpr uint32_t NW = GK == GK_Q4K ? 3 : GK == GK_Q6K ? 3 : GK == GK_Q51 ? 3 : 4;
    u4v v[TQ ? NU : NW];
    u4v pl[GK == GK_TQ5 ? NU : 1];   // the 5-bit plane's chunk
    uint32_t hd[TQ ? 2 * ND : 4];    // TQ: row pairs' d and m; GGUF: the rest

    __device__ __forceinline__ void load(const GemmArgs& g, uint32_t row0, uint32_t b0, uint32_t nblk) {
        const uint32_t tid = threadIdx.x;
        if constexpr (TQ) {
            const uint32_t ns = g.r_hi / 16, s0 = row0 / 16;
#pragma unroll
            for (uint32_t i = 0; i < NU; i++) {
                const uint32_t u = tid + 256 * i, e = u % UPB, j = u / UPB % NBLK, st = s0 + u / UPB / NBLK;
                const uint8_t* blk = g.w + (size_t)(st < ns ? st : ns - 1) * g.pitch +
                                     (size_t)(b0 + (j < nblk ? j : nblk - 1)) * T::BB;
                v[i] = *reinterpret_cast<const u4v*>(blk + 64 + 16 * e);
                if constexpr (GK == GK_TQ5) pl[i] = *reinterpret_cast<const u4v*>(blk + 64 + 64 * T::NCH + 16 * (e / 4));
            }
#pragma unroll
            for (uint32_t i = 0; i < ND; i++) {
                const uint32_t u = tid + 256 * i, r2 = u % 8, j = u / 8 % NBLK, st = s0 + u / 8 / NBLK;
                const uint8_t* blk = g.w + (size_t)(st < ns ? st : ns - 1) * g.pitch +
                                     (size_t)(b0 + (j < nblk ? j : nblk - 1)) * T::BB;
                hd[2 * i] = reinterpret_cast<const uint32_t*>(blk)[r2];
                hd[2 * i + 1] = reinterpret_cast<const uint32_t*>(blk)[8 + r2];
            }
        } else {  // a thread per (row, 64 of the slice's 128 values); k is a multiple of 256
            const uint32_t r = row0 + tid / 2, c = tid % 2, sl = b0 / NBLK;
            const uint8_t* row = g.w + (size_t)(r < g.r_hi ? r : g.r_hi - 1) * g.pitch;
            if constexpr (GK == GK_Q4K) {
                const uint8_t* p = row + (size_t)(sl / 2) * 144;
                v[0] = *reinterpret_cast<const u4v*>(p);
                v[1] = *reinterpret_cast<const u4v*>(p + 16 + 64 * (sl % 2) + 32 * c);
                v[2] = *reinterpret_cast<const u4v*>(p + 32 + 64 * (sl % 2) + 32 * c);
            } else if constexpr (GK == GK_Q6K) {  // values 32 g + 16 c + i, g = 0..3, of half n = sl % 2
                const uint8_t* p = row + (size_t)(sl / 2) * 210;
                const uint32_t n = sl % 2;
                v[0] = *reinterpret_cast<const u4v_a2*>(p + 64 * n + 16 * c);
                v[1] = *reinterpret_cast<const u4v_a2*>(p + 64 * n + 32 + 16 * c);
                v[2] = *reinterpret_cast<const u4v_a2*>(p + 128 + 32 * n + 16 * c);
                const uint16_t* q = reinterpret_cast<const uint16_t*>(p + 192 + 8 * n);
                hd[0] = (uint32_t)q[0] | (uint32_t)q[1] << 16;
                hd[1] = (uint32_t)q[2] | (uint32_t)q[3] << 16;
                hd[2] = *reinterpret_cast<const uint16_t*>(p + 208);
            } else if constexpr (GK == GK_Q51) {  // two 24-byte blocks
                const u4v* p = reinterpret_cast<const u4v*>(row + (size_t)sl * 96 + 48 * c);
                v[0] = p[0], v[1] = p[1], v[2] = p[2];
            } else {  // Q8_0: two 34-byte blocks, 4-byte aligned
                typedef u4v u4v_a4 __attribute__((aligned(4)));
                const uint8_t* p = row + (size_t)sl * 136 + 68 * c;
#pragma unroll
                for (int i = 0; i < 4; i++) v[i] = *reinterpret_cast<const u4v_a4*>(p + 16 * i);
                hd[0] = *reinterpret_cast<const uint32_t*>(p + 64);
            }
        }
    }

    __device__ __forceinline__ void store(uint8_t* wb, float2 (*dm)[GM_ROWS], uint32_t b0) const {
        const uint32_t tid = threadIdx.x;
        if constexpr (TQ) {
#pragma unroll
            for (uint32_t i = 0; i < NU; i++) {
                const uint32_t u = tid + 256 * i, e = u % UPB, j = u / UPB % NBLK, st = u / UPB / NBLK;
                const uint32_t c = e / 4, rq = e % 4, row = 16 * st + 4 * rq;
                uint32_t ql = 0, qh = 0;  // the fifth bits of the four rows' low and high halves
                if constexpr (GK == GK_TQ5) {
                    ql = (rq < 2 ? pl[i].x : pl[i].y) >> (16 * (rq % 2));
                    qh = (rq < 2 ? pl[i].z : pl[i].w) >> (16 * (rq % 2));
                }
                // words c (low nibbles) and NCH + c (high) of the block's KB / 4; 8 bits: word c
                const uint32_t lo = KB / 4 * j + c, hi = lo + T::NCH;
                uint32_t* pl0 = reinterpret_cast<uint32_t*>(wb + lo / 4 * PW + row * 16) + lo % 4;
                uint32_t* ph0 = reinterpret_cast<uint32_t*>(wb + hi / 4 * PW + row * 16) + hi % 4;
#pragma unroll
                for (int rr = 0; rr < 4; rr++) {
                    const uint32_t w = v[i][rr];
                    if constexpr (GK == GK_TQ8) {
                        pl0[4 * rr] = w ^ 0x80808080u;  // q - 128
                    } else {
                        uint32_t a = w & 0x0f0f0f0fu, b = (w >> 4) & 0x0f0f0f0fu;
                        if constexpr (GK == GK_TQ5) {
                            a |= q5_hi4((ql >> (4 * rr)) & 0xfu);
                            b |= q5_hi4((qh >> (4 * rr)) & 0xfu);
                        }
                        pl0[4 * rr] = a;
                        ph0[4 * rr] = b;
                    }
                }
            }
#pragma unroll
            for (uint32_t i = 0; i < ND; i++) {
                const uint32_t u = tid + 256 * i, r2 = u % 8, j = u / 8 % NBLK, st = u / 8 / NBLK;
                const uint32_t d = hd[2 * i], m = hd[2 * i + 1];
                *reinterpret_cast<float4*>(&dm[j][16 * st + 2 * r2]) =
                    make_float4(h2f((uint16_t)(d & 0xffffu)), h2f((uint16_t)(m & 0xffffu)), h2f((uint16_t)(d >> 16)), h2f((uint16_t)(m >> 16)));
            }
        } else {
            const uint32_t r = tid / 2, c = tid % 2, n = b0 / NBLK % 2;
            auto put = [&](uint32_t piece, u4v x) { *reinterpret_cast<u4v*>(wb + piece * PW + r * 16) = x; };
            // (d, m) of the slice's 32-block jb (or, at kb 16, of both its 16-blocks)
            auto put_dm = [&](uint32_t jb, float d, float m) {
#pragma unroll
                for (uint32_t i = 0; i < 32 / KB; i++) dm[32 / KB * jb + i][r] = make_float2(d, m);
            };
            if constexpr (GK == GK_Q4K) {
                const float d = h2f((uint16_t)(v[0].x & 0xffffu)), dmin = h2f((uint16_t)(v[0].x >> 16));
#pragma unroll
                for (int h = 0; h < 2; h++) {
                    put(4 * c + 2 * h, (v[1] >> (4 * h)) & 0x0f0f0f0fu);
                    put(4 * c + 2 * h + 1, (v[2] >> (4 * h)) & 0x0f0f0f0fu);
                    // sub-block 4 n + 2 c + h
                    int sc[4], mn[4];
#pragma unroll
                    for (int t = 0; t < 4; t++) q4k_scale_min_w(v[0].y, v[0].z, v[0].w, 2 * t + h, sc[t], mn[t]);
                    const int s0 = c ? sc[1] : sc[0], s1 = c ? sc[3] : sc[2], m0 = c ? mn[1] : mn[0], m1 = c ? mn[3] : mn[2];
                    float dd, mm;
                    q4k_dm(d, dmin, n ? s1 : s0, n ? m1 : m0, dd, mm);
                    put_dm(2 * c + h, dd, mm);
                }
            } else if constexpr (GK == GK_Q6K) {
                const float d = h2f((uint16_t)hd[2]);
#pragma unroll
                for (int gq = 0; gq < 4; gq++) {
                    const u4v lo = gq < 2 ? (v[gq & 1] & 0x0f0f0f0fu) : ((v[gq & 1] >> 4) & 0x0f0f0f0fu);
                    put(2 * gq + c, lo | (((v[2] >> (2 * gq)) & 0x03030303u) << 4));
                    const int8_t sc = (int8_t)((hd[gq / 2] >> (16 * (gq % 2) + 8 * c)) & 0xffu);
                    const float dd = f16_round(d * (float)sc);
                    dm[2 * gq + c][r] = make_float2(dd, f16_round(-32.0f * dd));
                }
            } else if constexpr (GK == GK_Q51) {
                auto w = [&](int i) -> uint32_t { return v[i / 4][i % 4]; };
#pragma unroll
                for (int jb = 0; jb < 2; jb++) {
                    const uint32_t qh = w(6 * jb + 1);
#pragma unroll
                    for (int hf = 0; hf < 2; hf++) {
                        u4v x;
#pragma unroll
                        for (int t = 0; t < 4; t++)
                            x[t] = ((w(6 * jb + 2 + t) >> (4 * hf)) & 0x0f0f0f0fu) | q5_hi4((qh >> (16 * hf + 4 * t)) & 0xfu);
                        put(4 * c + 2 * jb + hf, x);
                    }
                    put_dm(2 * c + jb, h2f((uint16_t)(w(6 * jb) & 0xffffu)), h2f((uint16_t)(w(6 * jb) >> 16)));
                }
            } else {  // Q8_0: bytes 2 .. 33 of each 34-byte block, kept signed
                const uint32_t w[17] = {v[0].x, v[0].y, v[0].z, v[0].w, v[1].x, v[1].y, v[1].z, v[1].w, v[2].x,
                                        v[2].y, v[2].z, v[2].w, v[3].x, v[3].y, v[3].z, v[3].w, hd[0]};
#pragma unroll
                for (int jb = 0; jb < 2; jb++) {
                    u4v x, z;
#pragma unroll
                    for (int t = 0; t < 4; t++) {
                        x[t] = jb ? w[9 + t] : __builtin_amdgcn_alignbyte(w[t + 1], w[t], 2);
                        z[t] = jb ? w[13 + t] : __builtin_amdgcn_alignbyte(w[t + 5], w[t + 4], 2);
                    }
                    put(4 * c + 2 * jb, x);
                    put(4 * c + 2 * jb + 1, z);
                    const float d = h2f((uint16_t)(jb ? w[8] >> 16 : w[0] & 0xffffu));
                    put_dm(2 * c + jb, d, f16_round(-128.0f * d));
                }
            }
        }
    }
};

// WR x (4 / WR) waves over 128 weight rows x TOK activation rows (a wave: 4 / WR tiles of 32 weight
// rows at 32 activation rows), slices of SL x 128 values.  Three workgroups per CU are resident at kb 32 and
// in the 64-row form at kb 16, two in the 32-row form at kb 16 (62 to 64 KB of LDS) and in the 64-row form of
// 8-bit TQ (186 and 195 registers); a wave's per-block cost is its VALU and rank1 issue (about 48 VALU
// instructions, an int8 MFMA and four rank1 a tile), not the LDS reads (prefetching them: no change).
template <int GK, int KB, int WR, int SL>
__global__ __launch_bounds__(256, 2) void gemm_rows_kernel(GemmArgs g) {
    using W = GmW<GK, KB>;
    constexpr uint32_t NB1 = W::NBLK, NBLK = SL * NB1, RT = 4 / WR, TOK = 4 / WR * 32, PA = TOK * 16 + 16;
    constexpr bool XSUM = GK == GK_TQ8 || GK == GK_Q80;  // signed weights: + 128 x the activations' sum
    constexpr uint32_t NA = SL * TOK / 32;              // 16-byte activation pieces per thread
    constexpr uint32_t NSC = (TOK * NBLK + 255) / 256;   // activation scales per thread
    __shared__ __align__(16) uint8_t xa[8 * SL * PA];
    __shared__ __align__(16) uint8_t wb[8 * SL * W::PW];
    __shared__ __align__(16) float xsc[NBLK][2][TOK];  // sx, u = sx * sum in rank1's lane order
    __shared__ __align__(16) int xsum[XSUM ? NBLK : 1][XSUM ? TOK : 4];
    __shared__ __align__(16) float2 dm[NBLK][GM_ROWS];
    const uint32_t tid = threadIdx.x, lane = tid % 64, wv = tid / 64, h = lane / 32, c32 = lane % 32;
    uint32_t idx = 0;
    if (!xcd_order_1d(g.n, idx, run_id())) return;
    const uint32_t t0 = idx % g.tb * TOK, row0 = g.r_lo + idx / g.tb * GM_ROWS;
    const uint32_t wr = wv % WR * (RT * 32), wt = wv / WR * 32;

    W w[SL];
    u4v xv[NA];
    float sv[NSC];
    int uv[NSC];
    auto load = [&](uint32_t b0, uint32_t nblk) {
#pragma unroll
        for (uint32_t i = 0; i < SL; i++)
            if (i == 0 || i * NB1 < nblk) w[i].load(g, row0, b0 + i * NB1, nblk - i * NB1 < NB1 ? nblk - i * NB1 : NB1);
#pragma unroll
        for (uint32_t i = 0; i < NA; i++) {
            const uint32_t t = t0 + tid / (8 * SL) + 32 / SL * i, p = tid % (8 * SL), pc = 16 * p < nblk * KB ? p : 0;
            xv[i] = *reinterpret_cast<const u4v*>(g.q + (size_t)(t < g.m ? t : g.m - 1) * g.k + (size_t)b0 * KB + 16 * pc);
        }
#pragma unroll
        for (uint32_t i = 0; i < NSC; i++) {
            const uint32_t u = tid + 256 * i, t = t0 + u / NBLK, j = u % NBLK;
            const size_t o = (size_t)(t < g.m ? t : g.m - 1) * g.nb + b0 + (j < nblk ? j : 0);
            sv[i] = g.s[o];
            uv[i] = g.su[o];
        }
    };
    v4f acc[RT][4];
#pragma unroll
    for (uint32_t i = 0; i < RT; i++)
#pragma unroll
        for (int j = 0; j < 4; j++) acc[i][j] = v4f{0.0f, 0.0f, 0.0f, 0.0f};

    uint32_t nblk = g.nb < NBLK ? g.nb : NBLK;
    load(0, nblk);
    for (uint32_t b0 = 0; b0 < g.nb;) {
        __syncthreads();  // the previous slice's readers are done
#pragma unroll
        for (uint32_t i = 0; i < SL; i++)
            if (i == 0 || i * NB1 < nblk) w[i].store(wb + 8 * i * W::PW, dm + i * NB1, b0 + i * NB1);
#pragma unroll
        for (uint32_t i = 0; i < NA; i++) {
            const uint32_t t = tid / (8 * SL) + 32 / SL * i, p = tid % (8 * SL);
            *reinterpret_cast<u4v*>(xa + p * PA + t * 16) = xv[i];
            if constexpr (XSUM) {
                int s = 0;
#pragma unroll
                for (int e = 0; e < 4; e++) s = sdot4((int)xv[i][e], 0x01010101, s);
                if constexpr (KB == 32) s += __builtin_amdgcn_mov_dpp(s, 0xB1, 0xf, 0xf, false);  // the block's other piece
                if (KB == 16 || p % 2 == 0) xsum[p * 16 / KB][t] = 128 * s;
            }
        }
#pragma unroll
        for (uint32_t i = 0; i < NSC; i++) {
            const uint32_t u = tid + 256 * i, t = u / NBLK, j = u % NBLK, e = t % 32;
            if (TOK * NBLK % 256 == 0 || u < TOK * NBLK) {
                const uint32_t o = t / 32 * 32 + e / 4 % 2 * 16 + e % 4 * 4 + e / 8;
                xsc[j][0][t] = sv[i];
                xsc[j][1][o] = sv[i] * (float)uv[i];  // gemv.rs:143
            }
        }
        const uint32_t b1 = b0 + nblk, n1 = g.nb - b1 < NBLK ? g.nb - b1 : NBLK;
        if (b1 < g.nb) load(b1, n1);
        __syncthreads();
        // d * sx on the VALU and fma(m, u, acc) as rank1: both as rank1 or both on the VALU were no faster
#pragma unroll 2
        for (uint32_t b = 0; b < nblk; b++) {
            v4i A, B[RT];
            v4f sx[4];
            float2 d[RT];
            auto operand = [&](const uint8_t* p, uint32_t pitch, uint32_t r) -> v4i {
                if constexpr (KB == 32) return *reinterpret_cast<const v4i*>(p + (2 * b + h) * pitch + r * 16);
                const int2 v = *reinterpret_cast<const int2*>(p + b * pitch + r * 16 + 8 * h);
                return v4i{v.x, v.y, 0, 0};
            };
#pragma unroll
            for (uint32_t i = 0; i < RT; i++) {
                B[i] = operand(wb, W::PW, wr + 32 * i + c32);
                d[i] = dm[b][wr + 32 * i + c32];
            }
            A = operand(xa, PA, wt + c32);
            const v4f u = *reinterpret_cast<const v4f*>(&xsc[b][1][wt + 16 * h + 4 * (lane % 4)]);
#pragma unroll
            for (int q = 0; q < 4; q++) sx[q] = *reinterpret_cast<const v4f*>(&xsc[b][0][wt + 8 * q + 4 * h]);
            v16i z;
#pragma unroll
            for (int q = 0; q < 4; q++) {
                v4i x = v4i{0, 0, 0, 0};
                if constexpr (XSUM) x = *reinterpret_cast<const v4i*>(&xsum[b][wt + 8 * q + 4 * h]);
#pragma unroll
                for (int e = 0; e < 4; e++) z[4 * q + e] = x[e];
            }
#pragma unroll
            for (uint32_t i = 0; i < RT; i++) {
                v16i dot;
                if constexpr (KB == 32)
                    dot = __builtin_amdgcn_mfma_i32_32x32x32_i8(A, B[i], z, 0, 0, 0);
                else
                    dot = __builtin_amdgcn_mfma_i32_32x32x16_i8(__builtin_bit_cast(long, make_int2(A.x, A.y)),
                                                               __builtin_bit_cast(long, make_int2(B[i].x, B[i].y)), z, 0, 0, 0);
#pragma unroll
                for (int q = 0; q < 4; q++) {
                    acc[i][q] = rank1(u[q], d[i].y, acc[i][q]);
#pragma unroll
                    for (int e = 0; e < 4; e++)
                        acc[i][q][e] = __builtin_fmaf((float)dot[4 * q + e], d[i].x * sx[q][e], acc[i][q][e]);
                }
            }
        }
        b0 = b1;
        nblk = n1;
    }
    // lane (h, c32): rows 8 q + 4 h + e of the activation tile, weight row c32 of the row tile
#pragma unroll
    for (uint32_t i = 0; i < RT; i++) {
        const uint32_t row = row0 + wr + 32 * i + c32;
        if (row >= g.r_hi) continue;
#pragma unroll
        for (int q = 0; q < 4; q++) {
            const uint32_t tk = t0 + wt + 8 * q + 4 * h;
#pragma unroll
            for (int e = 0; e < 4; e++) {
                if (tk + e >= g.m || (g.pair && e % 2)) continue;  // a pair's rows sit side by side: e and e + 1
                float* yp = g.y + (size_t)(g.pair ? (tk + e) / 2 : tk + e) * g.ldy + row;
                const float v = g.pair ? acc[i][q][e] + acc[i][q][e | 1] : acc[i][q][e];
                *yp = g.accumulate ? *yp + v : v;
            }
        }
    }
}

template <int GK, int KB>
static hipError_t gemm_go(GemmArgs g, hipStream_t st) {
    const uint32_t rb = (g.r_hi - g.r_lo + GM_ROWS - 1) / GM_ROWS, t32 = (g.m + 31) / 32, t64 = (g.m + 63) / 64;
    // 32 activation rows a workgroup (a tile per wave, 256-value slices) or 64 (two tiles per wave, the
    // unpacked weights serving both, 128-value slices): geo::gemm_narrow
    const bool narrow = geo::gemm_narrow(rb, t32, KB);
    g.tb = narrow ? t32 : t64;
    g.n = rb * g.tb;
    const geo::Grid2 gr = geo::grid_run(g.n, 256);
    if (narrow)
        gemm_rows_kernel<GK, KB, 4, 2><<<dim3(gr.x, gr.y), 256, 0, st>>>(g);
    else
        gemm_rows_kernel<GK, KB, 2, 1><<<dim3(gr.x, gr.y), 256, 0, st>>>(g);
    return hipGetLastError();
}

hipError_t launch_gemm(const Mat& w, uint32_t item, uint32_t s0, uint32_t s1, uint32_t kb, const int8_t* q, const float* s,
                       const int32_t* su, uint32_t m, int pair, float* y, uint32_t ldy, int accumulate, hipStream_t st) {
    GemmArgs g;
    g.w = w.ptr + (size_t)item * w.stride;
    g.pitch = w.row_bytes;
    g.k = w.k;
    g.nb = w.k / kb;
    g.r_lo = 16 * s0;
    g.r_hi = fmt_is_tq(w.fmt) ? 16 * s1 : (16 * s1 < w.rows ? 16 * s1 : w.rows);
    g.q = q;
    g.s = s;
    g.su = su;
    g.m = m;
    g.tb = g.n = 0;
    g.pair = pair;
    g.y = y;
    g.ldy = ldy;
    g.accumulate = accumulate;
    switch (w.fmt) {
        case TRK_FMT_Q4_K: return kb == 32 ? gemm_go<GK_Q4K, 32>(g, st) : gemm_go<GK_Q4K, 16>(g, st);
        case TRK_FMT_Q6_K: return gemm_go<GK_Q6K, 16>(g, st);
        case TRK_FMT_Q8_0: return kb == 32 ? gemm_go<GK_Q80, 32>(g, st) : gemm_go<GK_Q80, 16>(g, st);
        case TRK_FMT_Q5_1: return kb == 32 ? gemm_go<GK_Q51, 32>(g, st) : gemm_go<GK_Q51, 16>(g, st);
        case TRK_FMT_TQ4_32: return gemm_go<GK_TQ4, 32>(g, st);
        case TRK_FMT_TQ4_16: return gemm_go<GK_TQ4, 16>(g, st);
        case TRK_FMT_TQ5_32: return gemm_go<GK_TQ5, 32>(g, st);
        case TRK_FMT_TQ5_16: return gemm_go<GK_TQ5, 16>(g, st);
        case TRK_FMT_TQ8_32: return gemm_go<GK_TQ8, 32>(g, st);
        case TRK_FMT_TQ8_16: return gemm_go<GK_TQ8, 16>(g, st);
        default: return hipErrorInvalidValue;
    }
}

}  // namespace trk
