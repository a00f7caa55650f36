// The prefill's projections for prompts above the row kernels' sizes (rows.h): Y = X W^T with the
// operands streamed from L2 straight into registers, K split over the waves of a block, and the sums
// of the row kernels bit for bit.
//
// A row kernel's output is a sum of runs: K is cut into 8 runs (q|k|v, gate|up: 4 steps of 32 each) or
// 16 (o 4 steps, down 6), a run's products (hi, then lo of each step) are chained in the matrix unit from
// zero, and the runs are added in order. Here each of a block's NW waves takes CH of the runs for the
// block's whole output tile (16 MT rows x 16 NT columns), so an operand byte enters the CU once, with no
// LDS staging and no barrier in the loop; then the runs' tiles meet in LDS, MX 16-row tiles at a time, and
// a wave adds up one 16 x 16 subtile. The tile is computed transposed (D = W X^T: lane l holds row l %
// 16 of X and output columns 4 (l / 16) .. + 3), which changes no product and no sum, so a lane's four
// values are neighbours in every layout the epilogues write.
//
// q|k|v and gate|up read the residual rows in f32 (rows.h pk_a), multiply them by the RMSNorm weight,
// split them into f16 hi + lo and sum their squares on the way, each in the row kernels' order; o and
// down read what the attention and gate|up store already split (pk_s). W is in rows.h's tile layout
// (pk_w).
//
// What bounds them: the operand bytes into a CU (about 70 GB/s from L2), then the exchange and the waits of
// the end. Against the row kernels (16-row blocks, which read every weight once per 16 rows): a prefill of
// 65 rows 1.22 -> 1.06 ms, 130 1.85 -> 1.34, 300 3.01 -> 1.64, 768 6.66 -> 3.26, 1001 9.24 -> 3.92.
// Four waves of longer runs, whose sums start from zero at every step, exchange half as much and take the
// norm's sums from the previous launch (256 rows 1.44 ms, with the attention on the matrix cores; 768 2.80, 1001 3.32).
// They are no further from 64 bits, but have other bits than the row kernels: a row's results then depend on
// the length of its prompt.
#pragma once

#include "rows.h"

namespace navi_amd {
namespace gm {

// Element (m, k) of an f16-pair matrix of width K, MFMA fragment order: per 16-row tile and 32-column
// step 1 KB of hi, then 1 KB of lo (the bytes of the f32 value). Index of the hi half; lo is 512 further on.
__host__ __device__ inline size_t pk_s(int m, int k, int K) {
    return (static_cast<size_t>(m >> 4) * (K >> 5) + (k >> 5)) * 1024 + static_cast<size_t>((m & 15) + 16 * ((k >> 3) & 3)) * 8 + (k & 7);
}

enum { G_QKV = 0, G_SWIGLU = 1, G_RESID = 2 };

struct GemmArgs {
    const void *x;                    // QKV, SWIGLU: the residual rows (rows.h pk_a, width K); RESID: split layout
    const uint16_t *w;                // tile layout [N][K] (SWIGLU: gate [F] | up [F])
    uint32_t *flag;                   // set when a value for the next projection is outside the f16 range
    int M, K, N;                      // N: output columns (SWIGLU: F)
    float eps, q_scale;
    float *res;                       // RESID: the residual stream (rows.h pk_a, width N), added to
    const float *ln;                  // QKV, SWIGLU: the RMSNorm's weight [K]; RESID: the next one's [N] or null (flag only)
    uint16_t *y;                      // SWIGLU [M][N]: split layout
    // QKV: heads of 128 columns, one per block: q (nq heads) | k (nkv) | v (nkv)
    const float *qn, *kn, *cs;        // head norm weights [128]; cs: cos | sin of position p, dim d < 64 at cs[p][2][64]
    float *qf;                        // the normed, rotated queries: f32 rows [M][nq 128], or (null) times q_scale in qs
    uint16_t *qs;                     // split layout [M][nq 128]
    uint16_t *kc, *vc;                // the cache rows [pos][nkv 128] f16
    uint16_t *kf, *vf;                // the keys and values in k_attn_prompt's fragment order, or null
    int nq, nkv;
};

// Keys and values of one prefill as the attention's MFMA operands, per kv group and 32-key step 16
// KB: keys as two 16-key tiles x four 32-dim steps of 64 lanes x 8 halves; values transposed, eight
// 16-dim tiles of 64 lanes x 8 halves.
__host__ __device__ inline size_t kf_at(int g, int key, int d, int steps) {
    return ((static_cast<size_t>(g) * steps + (key >> 5)) * 8 + ((key >> 4) & 1) * 4 + (d >> 5)) * 512 +
           static_cast<size_t>((key & 15) + 16 * ((d >> 3) & 3)) * 8 + (d & 7);
}
__host__ __device__ inline size_t vf_at(int g, int key, int d, int steps) {
    return ((static_cast<size_t>(g) * steps + (key >> 5)) * 8 + (d >> 4)) * 512 +
           static_cast<size_t>((d & 15) + 16 * ((key >> 3) & 3)) * 8 + (key & 7);
}

namespace {

typedef _Float16 ghalf8 __attribute__((ext_vector_type(8)));
typedef _Float16 ghalf4 __attribute__((ext_vector_type(4)));

__device__ __forceinline__ bool outside_f16(float v) { return !(fabsf(v) < 65504.f); }

// One value of an f16-pair row.
__device__ __forceinline__ void split_store(uint16_t *dst, float v, bool &bad) {
    bad |= outside_f16(v);
    _Float16 h, o;
    f16_pair(v, h, o);
    uint16_t u[2];
    __builtin_memcpy(&u[0], &h, 2);
    __builtin_memcpy(&u[1], &o, 2);
    gst(dst, u[0]);
    gst(dst + 512, u[1]);
}

// Four neighbouring columns of an f16-pair row as one 8-byte store each.
__device__ __forceinline__ void split_store4(uint16_t *dst, f32x4_t v, bool &bad) {
    ghalf4 h, o;
#pragma unroll
    for (int r = 0; r < 4; ++r) {
        bad |= outside_f16(v[r]);
        _Float16 hr, lr;
        f16_pair(v[r], hr, lr);
        h[r] = hr;
        o[r] = lr;
    }
    *(NAVI_GLOBAL ghalf4 *) dst = h;
    *(NAVI_GLOBAL ghalf4 *) (dst + 512) = o;
}

// The block's (column block, row tile). Dispatch is round-robin over the 8 XCDs: XCD k's blocks take
// a run of the tiles in column-major order, so a column block's weights and a few row tiles share
// its L2.
__device__ __forceinline__ void tile_of(int nrow, int &col, int &row) {
    const int n = gridDim.x, id = blockIdx.x, k = id & 7, slot = id >> 3, q = n >> 3, r = n & 7;
    const int t = k * q + min(k, r) + slot;
    col = t / nrow;
    row = t % nrow;
}

// The end of a q|k|v block: head `col` of 16 MT rows in hs (times the row scale), one wave per row,
// lane l holding dims l and l + 64 (the values 0 + x, so a -0 sum is stored as +0): q and k heads
// RMSNorm'd and rotated (rotate-half RoPE), k and v rounded to f16 into the cache rows
// (talker.hip:46-82's k_qk_norm_rope).
template <int ROWS>
struct Heads {
    float cs[ROWS], sn[ROWS], n0, n1;

    __device__ __forceinline__ void load(const GemmArgs &a, int col, int m0, int l) {
        if (col >= a.nq + a.nkv) return;
        const float *nw = col < a.nq ? a.qn : a.kn;
        n0 = gld(nw + l);
        n1 = gld(nw + l + 64);
#pragma unroll
        for (int k = 0; k < ROWS; ++k) {
            const float *p = a.cs + static_cast<size_t>(min(m0 + k, a.M - 1)) * 128;
            cs[k] = gld(p + l);
            sn[k] = gld(p + l + 64);
        }
    }
    __device__ __forceinline__ void store(const GemmArgs &a, int col, int m0, int l, const float (*hs)[132], bool &bad) const {
        const int mtiles = (a.M + 15) >> 4, ks = (mtiles + 1) >> 1, QD = a.nq * 128, KVD = a.nkv * 128;
#pragma unroll
        for (int k = 0; k < ROWS; ++k) {
            const int m = m0 + k;
            const float a0 = 0.f + hs[k][l], a1 = 0.f + hs[k][l + 64];
            if (col >= a.nq + a.nkv) {
                const int g = col - a.nq - a.nkv;
                const uint16_t v0 = m < a.M ? f2h(a0) : static_cast<uint16_t>(0), v1 = m < a.M ? f2h(a1) : static_cast<uint16_t>(0);
                if (a.vf && m < 16 * mtiles) {               // zeros for the keys of the last 32-key step past the prompt
                    gst(a.vf + vf_at(g, m, l, ks), v0);
                    gst(a.vf + vf_at(g, m, l + 64, ks), v1);
                    if ((mtiles & 1) && (m >> 4) == mtiles - 1) {
                        gst(a.vf + vf_at(g, m + 16, l, ks), static_cast<uint16_t>(0));
                        gst(a.vf + vf_at(g, m + 16, l + 64, ks), static_cast<uint16_t>(0));
                    }
                }
                if (m < a.M) {
                    uint16_t *vd = a.vc + static_cast<size_t>(m) * KVD + g * 128;
                    gst(vd + l, v0);
                    gst(vd + l + 64, v1);
                }
                continue;
            }
            if (m >= a.M) break;
            const float sc = rsqrtf(wave_sum(fmaf(a0, a0, a1 * a1)) / 128.f + a.eps);
            const float x0 = a0 * sc * n0, x1 = a1 * sc * n1;
            const float y0 = x0 * cs[k] - x1 * sn[k];
            const float y1 = x1 * cs[k] + x0 * sn[k];
            if (col >= a.nq) {
                const int g = col - a.nq;
                const uint16_t k0 = f2h(y0), k1 = f2h(y1);
                uint16_t *kd = a.kc + static_cast<size_t>(m) * KVD + g * 128;
                gst(kd + l, k0);
                gst(kd + l + 64, k1);
                if (a.kf) {
                    gst(a.kf + kf_at(g, m, l, ks), k0);
                    gst(a.kf + kf_at(g, m, l + 64, ks), k1);
                }
            } else if (a.qf) {
                float *qd = a.qf + static_cast<size_t>(m) * QD + col * 128;
                gst(qd + l, y0);
                gst(qd + l + 64, y1);
            } else {
                split_store(a.qs + pk_s(m, col * 128 + l, QD), y0 * a.q_scale, bad);
                split_store(a.qs + pk_s(m, col * 128 + l + 64, QD), y1 * a.q_scale, bad);
            }
        }
    }
};

// NW waves of CH runs of PER steps (K = 32 NW CH PER), ST load slots (ST - 1 steps in flight). ST = 1: every
// fragment is asked for again as soon as its last product is out.
template <int MT, int NT, int EPI, int NW, int CH, int PER, int ST, int WPS, int MX>
__global__ void __launch_bounds__(NW * WAVE, WPS) k_gemm(GemmArgs a) {
    constexpr bool NORM = EPI != G_RESID;
    constexpr int S = CH * PER, STEPS = NW * S, RUNS = NW * CH;
    constexpr int UN = EPI == G_SWIGLU ? NT / 2 : NT, ROUNDS = MT / MX, UPW = (MX * UN + NW - 1) / NW;
    static_assert(EPI != G_QKV || (NT == 8 && MT * 16 % NW == 0), "a block of the q|k|v projection owns one head, a wave whole rows");
    static_assert(EPI != G_SWIGLU || NT % 2 == 0, "as many up columns as gate columns");
    static_assert(MT % MX == 0 && (!NORM || (CH == 1 && MT * 16 <= NW * WAVE)), "whole rounds; one run per wave, one thread per row scale");
    __shared__ f32x4_t red[RUNS][MX * NT][WAVE];
    __shared__ float ssq[NORM ? NW : 1][NORM ? MT : 1][WAVE], rscale[NORM ? MT * 16 : 1];
    __shared__ __align__(16) float lns[NORM ? STEPS * 32 : 4];
    __shared__ __align__(16) float hs[EPI == G_QKV ? MT * 16 : 1][132];
    const int w = __builtin_amdgcn_readfirstlane(static_cast<int>(threadIdx.x) >> 6), l = static_cast<int>(threadIdx.x) & 63;
    const int c = l & 15, g = l >> 4, mtiles = (a.M + 15) >> 4, nrow = (mtiles + MT - 1) / MT;
    int col, row;
    tile_of(nrow, col, row);
    const uint16_t *xb[MT], *wb[NT];                        // wave-uniform; lane l adds 8 l. A step of X is 2 KB either way
    // X tiles past the last one re-read it: their products are never stored
#pragma unroll
    for (int i = 0; i < MT; ++i)
        xb[i] = static_cast<const uint16_t *>(a.x) + (static_cast<size_t>(min(row * MT + i, mtiles - 1)) * STEPS + w * S) * 1024;
#pragma unroll
    for (int t = 0; t < NT; ++t) {
        const int nt = EPI == G_SWIGLU ? (t < NT / 2 ? col * (NT / 2) + t : (a.N >> 4) + col * (NT / 2) + t - NT / 2) : col * NT + t;
        wb[t] = a.w + (static_cast<size_t>(nt) * STEPS + w * S) * 512;
    }
    f32x4_t acc[CH][MT][NT];
    float ss[MT];
#pragma unroll
    for (int i = 0; i < MT; ++i) {
        ss[i] = 0.f;
#pragma unroll
        for (int h = 0; h < CH; ++h)
#pragma unroll
            for (int t = 0; t < NT; ++t) acc[h][i][t] = f32x4_t{0.f, 0.f, 0.f, 0.f};
    }
    u32x4_t fx[ST][MT][2], fw[ST][NT];
    const uint32_t lo8 = static_cast<uint32_t>(l) * 8;
    if constexpr (NORM) {                                   // the norm weights of the wave's own steps
        static_assert(!NORM || S == 4, "two weights per lane");
        const uint32_t i = w * (32 * S) + 2 * l;
        lns[i] = gld(a.ln + i);
        lns[i + 1] = gld(a.ln + i + 1);
    }
    auto load_w = [&](int slot, int t, int s) { fw[slot][t] = *(const NAVI_GLOBAL u32x4_t *) (wb[t] + s * 512 + lo8); };
    auto load_x = [&](int slot, int i, int s) {
#pragma unroll
        for (int p = 0; p < 2; ++p) fx[slot][i][p] = *(const NAVI_GLOBAL u32x4_t *) (xb[i] + s * 1024 + p * 512 + lo8);
    };
    auto load = [&](int slot, int s) {
#pragma unroll
        for (int i = 0; i < MT; ++i) load_x(slot, i, s);
#pragma unroll
        for (int t = 0; t < NT; ++t) load_w(slot, t, s);
    };
    // the f16 pair of a tile's fragment at step s
    auto operand = [&](int slot, int i, int s, ghalf8 &hi, ghalf8 &lo) {
        if constexpr (NORM) {
            float v[8];
            __builtin_memcpy(&v, &fx[slot][i][0], 16);
            __builtin_memcpy(&v[4], &fx[slot][i][1], 16);
            const float *q = lns + w * (32 * S) + 32 * s + 8 * g;
            const f32x4_t l0 = *reinterpret_cast<const f32x4_t *>(q), l1 = *reinterpret_cast<const f32x4_t *>(q + 4);
#pragma unroll
            for (int j = 0; j < 8; ++j) {
                ss[i] = fmaf(v[j], v[j], ss[i]);
                _Float16 h, o;
                f16_pair(v[j] * (j < 4 ? l0[j & 3] : l1[j & 3]), h, o);
                hi[j] = h;
                lo[j] = o;
            }
        } else {
            __builtin_memcpy(&hi, &fx[slot][i][0], 16);
            __builtin_memcpy(&lo, &fx[slot][i][1], 16);
        }
    };
    auto mma = [&](f32x4_t &sum, const u32x4_t &wv, const ghalf8 &xv) {
        ghalf8 v;
        __builtin_memcpy(&v, &wv, 16);
        sum = __builtin_amdgcn_mfma_f32_16x16x32_f16(v, xv, sum, 0, 0, 0);
    };
    const int m0 = row * MT * 16;
    if constexpr (ST == 1) {
        load(0, 0);
#pragma unroll
        for (int s = 0; s < S; ++s)
#pragma unroll
            for (int i = 0; i < MT; ++i) {
                ghalf8 hi, lo;
                operand(0, i, s, hi, lo);
                if (s + 1 < S) load_x(0, i, s + 1);
                constexpr int TB = 4;
#pragma unroll
                for (int t0 = 0; t0 < NT; t0 += TB) {
#pragma unroll
                    for (int t = t0; t < NT && t < t0 + TB; ++t) mma(acc[s / PER][i][t], fw[0][t], hi);
#pragma unroll
                    for (int t = t0; t < NT && t < t0 + TB; ++t) mma(acc[s / PER][i][t], fw[0][t], lo);
                    if (i == MT - 1 && s + 1 < S)
#pragma unroll
                        for (int t = t0; t < NT && t < t0 + TB; ++t) load_w(0, t, s + 1);
                    __builtin_amdgcn_sched_barrier(0);
                }
            }
    } else {
#pragma unroll
        for (int u = 0; u < ST - 1; ++u) load(u, u);
#pragma unroll
        for (int s = 0; s < S; ++s) {
            if (s + ST - 1 < S) load((s + ST - 1) % ST, s + ST - 1);
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int i = 0; i < MT; ++i) {
                ghalf8 hi, lo;
                operand(s % ST, i, s, hi, lo);
#pragma unroll
                for (int t = 0; t < NT; ++t) mma(acc[s / PER][i][t], fw[s % ST][t], hi);
#pragma unroll
                for (int t = 0; t < NT; ++t) mma(acc[s / PER][i][t], fw[s % ST][t], lo);
            }
            __builtin_amdgcn_sched_barrier(0);
        }
    }
    // what the end reads, asked for before the exchange: each residual element by the wave that writes it
    constexpr int RPW = EPI == G_QKV ? MT * 16 / NW : 1;
    Heads<RPW> heads;
    f32x4_t old[ROUNDS][UPW], lw[UPW];
    if constexpr (EPI == G_RESID) {
#pragma unroll
        for (int k = 0; k < UPW; ++k) {
            const int u = w + k * NW, n = (col * NT + u % UN) * 16 + 4 * g;
            lw[k] = f32x4_t{0.f, 0.f, 0.f, 0.f};
            if (a.ln && u < MX * UN) lw[k] = ld4(a.ln + n);
#pragma unroll
            for (int j = 0; j < ROUNDS; ++j) {
                const int m = m0 + (j * MX + u / UN) * 16 + c;
                f32x4_t v = {0.f, 0.f, 0.f, 0.f};
                if (u < MX * UN && m < a.M) v = ld4(a.res + rows::pk_a(m, n, a.N));
                old[j][k] = v;
            }
        }
    }
    bool bad = false;
#pragma unroll
    for (int j = 0; j < ROUNDS; ++j) {
        if (j) __syncthreads();                             // the previous tiles' readers are done
#pragma unroll
        for (int i = 0; i < MX; ++i)
#pragma unroll
            for (int t = 0; t < NT; ++t)
#pragma unroll
                for (int h = 0; h < CH; ++h) red[w * CH + h][i * NT + t][l] = acc[h][j * MX + i][t];
        if constexpr (EPI == G_QKV)
            if (j == ROUNDS - 1) heads.load(a, col, m0 + w * RPW, l);   // the last sums' registers are free now
        if constexpr (NORM)
            if (j == 0)
#pragma unroll
                for (int i = 0; i < MT; ++i) ssq[w][i][l] = ss[i];
        __syncthreads();
        if constexpr (NORM)
            if (j == 0) {
                // row r of a tile: lanes r % 16 + 16 q of every wave hold its sums of squares
                if (threadIdx.x < MT * 16) {
                    const int i = threadIdx.x / 16, r = threadIdx.x % 16;
                    float t = 0.f;
#pragma unroll
                    for (int ww = 0; ww < NW; ++ww)
#pragma unroll
                        for (int q = 0; q < 4; ++q) t += ssq[ww][i][r + 16 * q];
                    rscale[threadIdx.x] = rsqrtf(t / static_cast<float>(a.K) + a.eps);
                }
                __syncthreads();
            }
#pragma unroll
        for (int k = 0; k < UPW; ++k) {
            const int u = w + k * NW, i = u / UN, t = u % UN;
            if (u >= MX * UN) break;
            auto total = [&](int sub) {
                f32x4_t v = red[0][sub][l];
#pragma unroll
                for (int r = 1; r < RUNS; ++r) v += red[r][sub][l];
                return v;
            };
            const f32x4_t v = total(i * NT + t);
            const int mr = (j * MX + i) * 16 + c, m = m0 + mr;
            const bool in = m < a.M;
            if constexpr (EPI == G_RESID) {
                const f32x4_t x = old[j][k] + v;
                if (in) {
                    st4(a.res + rows::pk_a(m, (col * NT + t) * 16 + 4 * g, a.N), x);
#pragma unroll
                    for (int r = 0; r < 4; ++r) bad |= outside_f16(x[r] * lw[k][r]);
                }
            } else if constexpr (EPI == G_SWIGLU) {
                const f32x4_t up = total(i * NT + NT / 2 + t);
                const float sc = rscale[mr];
                f32x4_t h;
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    const float gt = v[r] * sc, u1 = up[r] * sc;
                    h[r] = gt / (1.f + expf(-gt)) * u1;
                }
                if (in) split_store4(a.y + pk_s(m, (col * UN + t) * 16 + 4 * g, a.N), h, bad);
            } else {
                *reinterpret_cast<f32x4_t *>(&hs[mr][16 * t + 4 * g]) = v * rscale[mr];
            }
        }
    }
    if constexpr (EPI == G_QKV) {
        __syncthreads();
        heads.store(a, col, m0 + w * RPW, l, &hs[w * RPW], bad);
    }
    if (bad) gst(a.flag, 1u);
}

// x = the rows src [.][H = 1024] in the layers' layout (rows.h pk_a), the flag set when a value times the
// first norm's weight is outside the f16 range; one block per row.
__global__ void __launch_bounds__(256) k_rows_in(const float *src, const float *ln, float *x, uint32_t *flag) {
    const int m = blockIdx.x, k = 4 * static_cast<int>(threadIdx.x);
    constexpr int H = 1024;
    const f32x4_t v = ld4(src + static_cast<size_t>(m) * H + k), w = ld4(ln + k);
    st4(x + rows::pk_a(m, k, H), v);
    bool bad = false;
#pragma unroll
    for (int r = 0; r < 4; ++r) bad |= outside_f16(v[r] * w[r]);
    if (bad) gst(flag, 1u);
}

// Causal attention of prompts of more than 256 rows from position 0 on the matrix cores: block (16-row tile
// qt, q head h) over keys 0..min(T, 16 qt + 16) - 1 of its kv group, in chunks of 256 keys with a
// running softmax. Queries (f16 pairs), keys and values come in fragment order (GemmArgs::qs, kf, vf), so
// every operand is a 1 KB load straight into registers. Per chunk: S = Q K^T (hi, then lo products of each
// 32-dim step; wave w takes the chunk's key tiles w, w + 4, ...), scaled and causally masked into LDS; per
// row (16 lanes) the chunk's max m_c, the new running max m = max(m_run, m_c), corr = e^(m_run - m), p =
// e^(s - m) as f16 pairs in LDS, l_run = l_run corr + sum p; the output rows scaled by corr, then O +=
// P V, wave w taking dims 32w .. 32w + 31. Finally O / l_run, stored split. Key 0 is in the first chunk of
// every row, so m_run is finite from the first chunk on. Grid (q heads, row tiles), the tiles with the most
// keys first; the two heads of kv group g run on XCD g, whose L2 holds its keys and values.
// With V staged transposed through LDS (84 KB, one block per CU) and K and V from the cache rows the same sums took
// 124 us a layer at 1001 rows, this 25.6 (8.2 at 300). What bounds it: the chunk's chain of scores, softmax and
// products with two barriers, on two blocks per CU (224 registers; at 168 or 128 it spills: 47.7, 79 us).
constexpr int LONG_CHUNK = 256;
struct AttnArgs {
    const uint16_t *q, *kf, *vf;
    uint16_t *att;                    // split layout [T][nq 128]
    uint32_t *flag;
    int T, nq;
    float scale;                      // of the scores (the queries carry q_scale)
};

__global__ void __launch_bounds__(4 * WAVE, 2) k_attn_prompt(AttnArgs a) {
    constexpr int KT = LONG_CHUNK / 16 / 4, KS = LONG_CHUNK / 32, SUB = LONG_CHUNK / 16;
    __shared__ float sS[16][LONG_CHUNK + 4];
    __shared__ __align__(16) _Float16 ph[16][LONG_CHUNK + 8], pl[16][LONG_CHUNK + 8];
    __shared__ float corr[16], lrow[16];
    const int w = __builtin_amdgcn_readfirstlane(static_cast<int>(threadIdx.x) >> 6), l = static_cast<int>(threadIdx.x) & 63;
    const int c = l & 15, kq = l >> 4, qt = static_cast<int>(gridDim.y) - 1 - static_cast<int>(blockIdx.y), r0 = 16 * qt;
    const int nkv = a.nq / 2, kv = static_cast<int>(blockIdx.x) % nkv, h = 2 * kv + static_cast<int>(blockIdx.x) / nkv;
    const int steps = (static_cast<int>(gridDim.y) + 1) >> 1, nk = min(a.T, r0 + 16);
    const uint32_t lo8 = static_cast<uint32_t>(l) * 8;
    const uint16_t *kb = a.kf + static_cast<size_t>(kv) * steps * 4096, *vb = a.vf + static_cast<size_t>(kv) * steps * 4096;
    ghalf8 qf[4][2];
    {
        const uint16_t *qb = a.q + (static_cast<size_t>(qt) * (a.nq * 4) + h * 4) * 1024;
#pragma unroll
        for (int s = 0; s < 4; ++s)
#pragma unroll
            for (int p = 0; p < 2; ++p) qf[s][p] = *(const NAVI_GLOBAL ghalf8 *) (qb + s * 1024 + p * 512 + lo8);
    }
    f32x4_t o[2] = {{0.f, 0.f, 0.f, 0.f}, {0.f, 0.f, 0.f, 0.f}};
    const int prow = threadIdx.x >> 4, j0 = threadIdx.x & 15;   // softmax: this thread's row and keys j0 + 16 m
    float mrun = -INFINITY, lrun = 0.f;                     // of prow, the same in its 16 lanes
    for (int k0 = 0; k0 < nk; k0 += LONG_CHUNK) {
        const int nkc = min(LONG_CHUNK, nk - k0), nkt = (nkc + 15) / 16, nks = (nkc + 31) / 32;
        const uint16_t *kc = kb + static_cast<size_t>(k0 >> 5) * 4096, *vc = vb + static_cast<size_t>(k0 >> 5) * 4096;
        ghalf8 kf[KT][4], vf[KS][2];
#pragma unroll
        for (int i = 0; i < KT; ++i)
            if (w + 4 * i < nkt)
#pragma unroll
                for (int s = 0; s < 4; ++s) kf[i][s] = *(const NAVI_GLOBAL ghalf8 *) (kc + ((w + 4 * i) * 4 + s) * 512 + lo8);
#pragma unroll
        for (int t = 0; t < KS; ++t)
            if (t < nks)
#pragma unroll
                for (int u = 0; u < 2; ++u) vf[t][u] = *(const NAVI_GLOBAL ghalf8 *) (vc + (t * 8 + 2 * w + u) * 512 + lo8);
#pragma unroll
        for (int i = 0; i < KT; ++i) {
            if (w + 4 * i >= nkt) break;
            f32x4_t acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int s = 0; s < 4; ++s)
#pragma unroll
                for (int p = 0; p < 2; ++p) acc = __builtin_amdgcn_mfma_f32_16x16x32_f16(qf[s][p], kf[i][s], acc, 0, 0, 0);
            const int key = 16 * (w + 4 * i) + c;
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const int row = 4 * kq + r;
                sS[row][key] = key < nkc && k0 + key <= r0 + row ? acc[r] * a.scale : -INFINITY;
            }
        }
        __syncthreads();
        {
            float v[SUB], mc = -INFINITY;
#pragma unroll
            for (int m = 0; m < SUB; ++m) {
                v[m] = m < nkt ? sS[prow][j0 + 16 * m] : -INFINITY;
                mc = fmaxf(mc, v[m]);
            }
            mc = fmaxf(mc, dpp_red<0xB1>(mc));
            mc = fmaxf(mc, dpp_red<0x4E>(mc));
            mc = fmaxf(mc, dpp_red<0x141>(mc));
            mc = fmaxf(mc, dpp_red<0x140>(mc));
            const float m1 = fmaxf(mrun, mc), cr = expf(mrun - m1);
            float sum = 0.f;
#pragma unroll
            for (int m = 0; m < SUB; ++m) {
                if (m >= 2 * nks) break;
                const float e = m < nkt ? expf(v[m] - m1) : 0.f;   // masked: e^-inf = 0
                const _Float16 hv = static_cast<_Float16>(e);
                ph[prow][j0 + 16 * m] = hv;
                pl[prow][j0 + 16 * m] = static_cast<_Float16>(e - static_cast<float>(hv));
                sum += e;
            }
            sum += dpp_red<0xB1>(sum);
            sum += dpp_red<0x4E>(sum);
            sum += dpp_red<0x141>(sum);
            sum += dpp_red<0x140>(sum);
            mrun = m1;
            lrun = lrun * cr + sum;
            if (j0 == 0) {
                corr[prow] = cr;
                lrow[prow] = lrun;
            }
        }
        __syncthreads();
#pragma unroll
        for (int u = 0; u < 2; ++u)
#pragma unroll
            for (int r = 0; r < 4; ++r) o[u][r] *= corr[4 * kq + r];
#pragma unroll
        for (int t = 0; t < KS; ++t) {
            if (t >= nks) break;
            const ghalf8 p0 = *reinterpret_cast<const ghalf8 *>(&ph[c][32 * t + 8 * kq]), p1 = *reinterpret_cast<const ghalf8 *>(&pl[c][32 * t + 8 * kq]);
#pragma unroll
            for (int u = 0; u < 2; ++u) o[u] = __builtin_amdgcn_mfma_f32_16x16x32_f16(p0, vf[t][u], o[u], 0, 0, 0);
#pragma unroll
            for (int u = 0; u < 2; ++u) o[u] = __builtin_amdgcn_mfma_f32_16x16x32_f16(p1, vf[t][u], o[u], 0, 0, 0);
        }
        // the next chunk's scores go to sS, which every thread has read; its probabilities wait for its own
        // barrier, which no wave passes before all have read these
    }
    bool bad = false;
#pragma unroll
    for (int u = 0; u < 2; ++u)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const int row = 4 * kq + r;
            if (r0 + row < a.T) split_store(a.att + pk_s(r0 + row, h * 128 + 32 * w + 16 * u + c, a.nq * 128), o[u][r] / lrow[row], bad);
        }
    if (bad) gst(a.flag, 1u);
}

template <int MT, int NT, int EPI, int NW, int CH, int PER, int ST, int WPS, int MX>
void launch_gemm(const GemmArgs &a, hipStream_t s) {
    const int ncol = EPI == G_SWIGLU ? a.N / (8 * NT) : a.N / (16 * NT), nrow = ((a.M + 15) / 16 + MT - 1) / MT;
    hipLaunchKernelGGL((k_gemm<MT, NT, EPI, NW, CH, PER, ST, WPS, MX>), dim3(ncol * nrow), dim3(NW * WAVE), 0, s, a);
}

// The talker's shapes (K 1024 into q|k|v and gate|up, 2048 into o, 3072 into down; N 4096, 2 x 3072,
// 1024, 1024). A block's time is its operand bytes (about 70 GB/s from L2 into one CU, whatever the other
// CUs do) and its end, a block fills a CU, and a block more than CUs is a second round: the tile is the one
// whose rounds take least.
int rounds(int ncol, int mtiles, int MT) { return (ncol * ((mtiles + MT - 1) / MT) + 255) / 256; }

// 16 MT x 128 tiles take 6.6, 9, 12.3 and 15.3 us a round for MT = 1 .. 4, as MT + 1. 640 rows: two rounds of
// MT = 3 23.6 us, three of MT = 2 25.1, two of MT = 4 27.9; 1001: two of MT = 4 30.8, three of MT = 3 36.3.
void launch_qkv(const GemmArgs &a, hipStream_t s) {
    const int mt = (a.M + 15) / 16, ncol = a.N / 128;
    int best = 1;
    for (int MT = 2; MT <= 4; ++MT)
        if (rounds(ncol, mt, MT) * (MT + 1) < rounds(ncol, mt, best) * (best + 1)) best = MT;
    if (best == 1) launch_gemm<1, 8, G_QKV, 8, 1, 4, 4, 2, 1>(a, s);
    else if (best == 2) launch_gemm<2, 8, G_QKV, 8, 1, 4, 1, 2, 1>(a, s);
    else if (best == 3) launch_gemm<3, 8, G_QKV, 8, 1, 4, 1, 2, 1>(a, s);
    else launch_gemm<4, 8, G_QKV, 8, 1, 4, 1, 2, 1>(a, s);
}
// One round: 16 x 128 tiles up to 5 row tiles (7.7 us), 32 x 96 up to 8 (8.4; 16 x 128 would be a second round, 12.3),
// 32 x 128 up to 10 (9.1). Above, 32 x 192 tiles (12.2 us a round of 256 rows) or 64 x 128 (13.5 a round of 340),
// whichever takes fewer rounds: 320 rows 19.6 and 13.6 us, 512 22.5 and 24.7, 640 30.5 and 25.2, 1001 47.5 and 38.0.
void launch_gate_up(const GemmArgs &a, hipStream_t s) {
    const int mt = (a.M + 15) / 16;
    if (mt <= 5) launch_gemm<1, 8, G_SWIGLU, 8, 1, 4, 4, 2, 1>(a, s);
    else if (mt <= 8) launch_gemm<2, 6, G_SWIGLU, 8, 1, 4, 2, 2, 2>(a, s);
    else if (mt <= 10) launch_gemm<2, 8, G_SWIGLU, 8, 1, 4, 2, 2, 2>(a, s);
    else if (rounds(a.N / 96, mt, 2) <= rounds(a.N / 64, mt, 4)) launch_gemm<2, 12, G_SWIGLU, 8, 1, 4, 1, 2, 1>(a, s);
    else launch_gemm<4, 8, G_SWIGLU, 8, 1, 4, 1, 2, 2>(a, s);
}
// PER = K / 512. The smallest tile that gives at most one round, up to 64 x 64. Down at 128 rows: 16 x 32 tiles 5.8
// us, 32 x 32 7.3; 256: 32 x 32 7.6, 32 x 64 9.3, 16 x 32 in two rounds 9.6; 512: 32 x 64 11.9, 64 x 64 16.4; 513:
// 16.5 in one round of 64 x 64, 18.9 in two of 32 x 64; 1001: 20.0 and 31.2.
template <int PER>
void launch_resid(const GemmArgs &a, hipStream_t s) {
    const int mt = (a.M + 15) / 16;
    if (mt <= 8) launch_gemm<1, 2, G_RESID, 16, 1, PER, 4, 4, 1>(a, s);
    else if (mt <= 16) launch_gemm<2, 2, G_RESID, 16, 1, PER, 2, 4, 2>(a, s);
    else if (mt <= 32) launch_gemm<2, 4, G_RESID, 16, 1, PER, 2, 4, 2>(a, s);
    else launch_gemm<4, 4, G_RESID, 8, 2, PER, 2, 2, 2>(a, s);
}

} // namespace
} // namespace gm
} // namespace navi_amd
