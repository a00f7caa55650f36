// The prefill's projections for prompts above the row kernels' sizes (rows.h): Y = X W^T with the
// operands streamed from L2 straight into registers, K split over the four waves of a block.
//
// X is held as f16 pairs x = hi + lo in MFMA fragment order ("split" layout, pk_s: per 16-row tile
// and 32-column step 1 KB of hi, then 1 KB of lo: the bytes of the f32 value), written by the
// kernel that produces it, so an operand is one contiguous 1 KB load per wave and nothing is
// converted on the way in. W is in rows.h's tile layout (pk_w).
//
// Each of a block's NW waves takes its share of K for the block's whole output tile (16 MT rows x 16
// NT columns), with the next step's fragments loading while this step's products run: an operand
// byte enters the CU once, there is no LDS staging and no barrier in the loop. The tile is
// computed transposed (D = W X^T: lane l holds row l % 16 of X and output columns 4 (l / 16) ..
// + 3), so a lane's four values are neighbours in every layout the epilogues write. At the end
// the waves' tiles are summed through LDS in wave order, wave w finishing 16-row tile w.
//
// What bounds them: the operand bytes into a CU (about 70 GB/s from L2, with the products switched
// off as with them on), then the waits of the epilogue, which is why what it reads goes out before
// the loop. 1001 rows, per layer: q|k|v 54.8 -> 32 us, gate|up 71.8 -> 30, o 26.7 -> 16.4, down 50.5 ->
// 21.2, attention 124 -> 17.0; the prefill 9.23 -> 3.31 ms. 130 rows: 15.3 -> 10.6, 16.1 -> 10.7, 8.4
// -> 8.4, 14.5 -> 10.6, 10.8 -> 8.1; 1.85 -> 1.34 ms. Sixteen-row blocks over whole-K (what these
// replaced) read every weight once per 16 rows. Measured and left out: the same tiles staged in LDS by
// eight waves (q|k|v at 1001 rows 25 us, but 21 us at 80 rows and gate|up 35), the loop unrolled over
// all of K (half as fast again: its code does not stay in the instruction cache), three and more steps
// in flight (no faster), hi and lo products in accumulators of their own (+3 %).
#pragma once

#include "rows.h"

namespace navi_amd {
namespace gm {

// Element (m, k) of an f16-pair matrix of width K: index of the hi half; the lo half is 512 further on.
__host__ __device__ inline size_t pk_s(int m, int k, int K) {
    return (static_cast<size_t>(m >> 4) * (K >> 5) + (k >> 5)) * 1024 + static_cast<size_t>((m & 15) + 16 * ((k >> 3) & 3)) * 8 + (k & 7);
}

enum { G_QKV = 0, G_SWIGLU = 1, G_RESID = 2 };
constexpr int SSQ = 32;               // partial sums of squares per residual row (32 columns each)

struct GemmArgs {
    const uint16_t *x;                // split layout [M][K]
    const uint16_t *w;                // tile layout [N][K] (SWIGLU: gate [F] | up [F])
    uint32_t *flag;                   // set when a value written for the next projection is outside the f16 range
    int M, K, N;                      // N: output columns (SWIGLU: F)
    float eps, q_scale;
    const float *ssq_in;              // QKV, SWIGLU: [SSQ][ldq] partial sums of squares of the residual rows
    float *ssq_out;                   // RESID: the same for the rows it writes
    float *res;                       // RESID: the residual stream (rows.h pk_a, width N), added to
    const float *ln;                  // RESID: the next RMSNorm's weight; y = split(res * ln); null: res only
    uint16_t *y;                      // SWIGLU [M][N], RESID [M][N]: split layout
    // QKV: heads of 128 columns, one per block: q (nq heads) | k (nkv) | v (nkv)
    const float *qn, *kn, *cs;        // head norm weights [128]; cs: cos | sin of position p, dim d < 64 at cs[p][2][64]
    uint16_t *q;                      // split layout [M][nq 128], normed, rotated and times q_scale
    uint16_t *kc, *vc;                // the cache rows [pos][nkv 128] f16
    uint16_t *kf, *vf;                // the keys and values in the attention's fragment order (attn.h)
    int nq, nkv, ldq;                 // ldq: row length of ssq
};

// Keys and values of one prefill as the attention's MFMA operands, per kv group and 32-key step 16
// KB: keys as two 16-key tiles x four 32-dim steps of 64 lanes x 8 halves; values transposed, eight
// 16-dim tiles of 64 lanes x 8 halves. Within a 32-key step the value fragments hold the keys in
// the order in which a lane of the transposed score tiles holds them (lane group g, element j: key
// 4 g + j of the first tile for j < 4, of the second above), so probabilities are used where they
// are computed.
__host__ __device__ inline size_t kf_at(int g, int key, int d, int steps) {
    return ((static_cast<size_t>(g) * steps + (key >> 5)) * 8 + ((key >> 4) & 1) * 4 + (d >> 5)) * 512 +
           static_cast<size_t>((key & 15) + 16 * ((d >> 3) & 3)) * 8 + (d & 7);
}
__host__ __device__ inline size_t vf_at(int g, int key, int d, int steps) {
    return ((static_cast<size_t>(g) * steps + (key >> 5)) * 8 + (d >> 4)) * 512 +
           static_cast<size_t>((d & 15) + 16 * ((key & 15) >> 2)) * 8 + ((key >> 4) & 1) * 4 + (key & 3);
}

namespace {

typedef _Float16 ghalf8 __attribute__((ext_vector_type(8)));
typedef _Float16 ghalf4 __attribute__((ext_vector_type(4)));

// Sum over the four 16-lane groups (lanes l, l ^ 16, l ^ 32, l ^ 48).
__device__ __forceinline__ float group_sum(float v) {
    v += __shfl_xor(v, 16);
    v += __shfl_xor(v, 32);
    return v;
}

// Four neighbouring columns of an f16-pair row as one 8-byte store each.
__device__ __forceinline__ void split_store4(uint16_t *dst, f32x4_t v, bool &bad) {
    ghalf4 h, o;
#pragma unroll
    for (int r = 0; r < 4; ++r) {
        bad |= !(fabsf(v[r]) < 65504.f);
        h[r] = static_cast<_Float16>(v[r]);
        o[r] = static_cast<_Float16>(v[r] - static_cast<float>(h[r]));
    }
    *(NAVI_GLOBAL ghalf4 *) dst = h;
    *(NAVI_GLOBAL ghalf4 *) (dst + 512) = o;
}

__device__ __forceinline__ void half_store4(uint16_t *dst, f32x4_t v) {
    ghalf4 h;
#pragma unroll
    for (int r = 0; r < 4; ++r) h[r] = static_cast<_Float16>(v[r]);
    *(NAVI_GLOBAL ghalf4 *) dst = h;
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

// One wave's end of a projection: v[t] = its 16 rows' products with column tiles t (lane l: row m,
// columns 16 t + 4 g .. + 3 of the wave's columns). load() asks for what the end needs besides the
// products, early enough to arrive during the loop: the partial sums of squares of the rows; the
// residual rows and the next norm's weight; the head's norm weights and the rotation.
// col: the wave's column block, 16 NT columns wide (SWIGLU: 8 NT gate and as many up columns).
template <int NT, int EPI>
struct Epilogue {
    float sq[EPI == G_RESID ? 1 : SSQ / 4];
    f32x4_t old[EPI == G_RESID ? NT : 1], lw[EPI == G_RESID ? NT : 1];
    f32x4_t hw[EPI == G_QKV ? 8 : 1], ct[EPI == G_QKV ? 4 : 1], st[EPI == G_QKV ? 4 : 1];

    __device__ __forceinline__ void load(const GemmArgs &a, int col, int m, int g) {
        m = min(m, a.M - 1);
        if constexpr (EPI == G_RESID) {
#pragma unroll
            for (int t = 0; t < NT; ++t) {
                const int n = col * (16 * NT) + 16 * t + 4 * g;
                old[t] = ld4(a.res + rows::pk_a(m, n, a.N));
                lw[t] = a.ln ? ld4(a.ln + n) : f32x4_t{0.f, 0.f, 0.f, 0.f};
            }
        } else {
#pragma unroll
            for (int k = 0; k < SSQ / 4; ++k) sq[k] = gld(a.ssq_in + (SSQ / 4 * g + k) * a.ldq + m);
        }
    }
    // q|k|v; of larger tiles behind the loop, whose registers they would take
    __device__ __forceinline__ void load_head(const GemmArgs &a, int col, int m, int g) {
        m = min(m, a.M - 1);
        if constexpr (EPI == G_QKV) {
            const float *nw = col < a.nq ? a.qn : a.kn, *cs = a.cs + static_cast<size_t>(m) * 128 + 4 * g;
#pragma unroll
            for (int t = 0; t < 8; ++t) hw[t] = ld4(nw + 16 * t + 4 * g);
#pragma unroll
            for (int t = 0; t < 4; ++t) {
                ct[t] = ld4(cs + 16 * t);
                st[t] = ld4(cs + 16 * t + 64);
            }
        }
    }

    // Every row of the tile's 16 comes through here (the sums over lanes need them all); rows past the
    // last are not stored.
    __device__ __forceinline__ void finish(const GemmArgs &a, int col, int m, int mtiles, int g, f32x4_t (&v)[NT], bool &bad) const {
        const bool in = m < a.M;
        float sc = 1.f;
        if constexpr (EPI != G_RESID) {
            float t = 0.f;
#pragma unroll
            for (int k = 0; k < SSQ / 4; ++k) t += sq[k];
            sc = rsqrtf(group_sum(t) / static_cast<float>(a.K) + a.eps);
        }
        if constexpr (EPI == G_RESID) {
            float ss[NT / 2];
#pragma unroll
            for (int t = 0; t < NT; ++t) {
                const int n = col * (16 * NT) + 16 * t + 4 * g;
                const f32x4_t x = old[t] + v[t];
                if (t % 2 == 0) ss[t / 2] = 0.f;
#pragma unroll
                for (int r = 0; r < 4; ++r) ss[t / 2] = fmaf(x[r], x[r], ss[t / 2]);
                if (in) {
                    st4(a.res + rows::pk_a(m, n, a.N), x);
                    if (a.ln) split_store4(a.y + pk_s(m, n, a.N), x * lw[t], bad);
                }
            }
            if (a.ln)
#pragma unroll
                for (int t = 0; t < NT / 2; ++t) {
                    const float q = group_sum(ss[t]);
                    if (g == 0 && in) gst(a.ssq_out + (col * (NT / 2) + t) * a.ldq + m, q);
                }
        } else if constexpr (EPI == G_SWIGLU) {
#pragma unroll
            for (int t = 0; t < NT / 2; ++t) {
                f32x4_t h;
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    const float gt = v[t][r] * sc, up = v[t + NT / 2][r] * sc;
                    h[r] = gt / (1.f + expf(-gt)) * up;
                }
                if (in) split_store4(a.y + pk_s(m, (col * (NT / 2) + t) * 16 + 4 * g, a.N), h, bad);
            }
        } else {
            const int ks = (mtiles + 1) >> 1, KVD = a.nkv * 128;
#pragma unroll
            for (int t = 0; t < NT; ++t) v[t] *= sc;
            if (col >= a.nq + a.nkv) {
                const int kv = col - a.nq - a.nkv;
#pragma unroll
                for (int t = 0; t < NT; ++t) {
                    const int d = 16 * t + 4 * g;
                    if (in) half_store4(a.vc + static_cast<size_t>(m) * KVD + kv * 128 + d, v[t]);
                    // fragments: zeros for the keys of the last 32-key step past the prompt
                    if (m < 16 * mtiles)
#pragma unroll
                        for (int r = 0; r < 4; ++r) {
                            uint16_t *p = a.vf + vf_at(kv, m, d + r, ks);
                            gst(p, in ? f2h(v[t][r]) : static_cast<uint16_t>(0));
                            if ((mtiles & 1) && (m >> 4) == mtiles - 1) gst(p + 4, static_cast<uint16_t>(0));
                        }
                }
            } else {
                float ss = 0.f;
#pragma unroll
                for (int t = 0; t < NT; ++t)
#pragma unroll
                    for (int r = 0; r < 4; ++r) ss = fmaf(v[t][r], v[t][r], ss);
                const float hs = rsqrtf(group_sum(ss) / 128.f + a.eps);
#pragma unroll
                for (int t = 0; t < 4; ++t) {
                    const int d = 16 * t + 4 * g;
                    const f32x4_t x0 = v[t] * hs * hw[t], x1 = v[t + 4] * hs * hw[t + 4];
                    f32x4_t y0 = x0 * ct[t] - x1 * st[t], y1 = x1 * ct[t] + x0 * st[t];
                    if (!in) continue;
                    if (col < a.nq) {
#pragma unroll
                        for (int r = 0; r < 4; ++r) {
                            y0[r] *= a.q_scale;
                            y1[r] *= a.q_scale;
                        }
                        split_store4(a.q + pk_s(m, col * 128 + d, a.nq * 128), y0, bad);
                        split_store4(a.q + pk_s(m, col * 128 + d + 64, a.nq * 128), y1, bad);
                    } else {
                        const int kv = col - a.nq;
                        half_store4(a.kc + static_cast<size_t>(m) * KVD + kv * 128 + d, y0);
                        half_store4(a.kc + static_cast<size_t>(m) * KVD + kv * 128 + d + 64, y1);
                        half_store4(a.kf + kf_at(kv, m, d, ks), y0);
                        half_store4(a.kf + kf_at(kv, m, d + 64, ks), y1);
                    }
                }
            }
        }
    }
};

// NW waves, each PER steps of 32 of K = 32 NW PER, with ST load slots (ST - 1 steps in flight). ST = 1: two
// slots for X and one for W, whose fragments are asked for again as soon as their products are out,
// half a step's registers less than ST = 2: two blocks share a CU, and one's epilogue runs under the
// other's loop. The waves' tiles are exchanged MX 16-row tiles at a time.
//
// A step's products start from zero (lo, then hi) and are added to the tile's sums by the vector units.
// Chained on the sums in the matrix unit, every product is cut to the last bit of a sum that grows with
// K: mean over twelve prompts of 100 rows, the first layer's keys and values then lie 9.1e-6 and 8.5e-6 from
// 64 bits, like this 7.4e-6 and 7.2e-6 (the row kernels' half as long chains: 7.3e-6 and 8.8e-6), the final
// hidden state 1.16e-4 and 9.9e-5 (1.25e-4). It costs nothing up to 300 rows and 4 % of the prefill at 1001. The
// two largest gate|up tiles have no registers left for it and chain (CHAIN): their error reaches the keys and values
// only through the residual stream (without it 768 rows take 2.98 ms instead of 2.79, the second
// layer's keys and values at the same distance).
template <int MT, int NT, int EPI, int NW, int PER, int ST, int WPS, int MX = MT>
__global__ void __launch_bounds__(NW * WAVE, WPS) k_gemm(GemmArgs a) {
    static_assert(EPI != G_QKV || NT == 8, "a block of the q|k|v projection owns one head");
    static_assert(NT % 2 == 0, "as many up columns as gate columns; 32 columns per partial sum of squares");
    static_assert(MT <= NW && PER % ST == 0 && MT % MX == 0, "a wave finishes one 16-row tile; whole rounds of the load slots");
    constexpr int STEPS = NW * PER;
    constexpr bool CHAIN = MT * NT * (ST == 1 ? 2 : 1) >= 48;   // 64 x 192, and 64 x 96 at half the registers: they would spill
    __shared__ f32x4_t red[MX][NW - 1][NT][WAVE];
    const int w = __builtin_amdgcn_readfirstlane(static_cast<int>(threadIdx.x) >> 6), l = static_cast<int>(threadIdx.x) & 63;
    const int g = l >> 4, mtiles = (a.M + 15) >> 4, nrow = (mtiles + MT - 1) / MT;
    int col, row;
    tile_of(nrow, col, row);
    const uint16_t *xb[MT], *wb[NT];                        // wave-uniform; lane l adds 8 l
    // X tiles past the last one re-read it: their products are never stored
#pragma unroll
    for (int i = 0; i < MT; ++i) xb[i] = a.x + (static_cast<size_t>(min(row * MT + i, mtiles - 1)) * STEPS + w * PER) * 1024;
#pragma unroll
    for (int t = 0; t < NT; ++t) {
        const int nt = EPI == G_SWIGLU ? (t < NT / 2 ? col * (NT / 2) + t : (a.N >> 4) + col * (NT / 2) + t - NT / 2) : col * NT + t;
        wb[t] = a.w + (static_cast<size_t>(nt) * STEPS + w * PER) * 512;
    }
    f32x4_t acc[MT][NT];
#pragma unroll
    for (int i = 0; i < MT; ++i)
#pragma unroll
        for (int t = 0; t < NT; ++t) acc[i][t] = f32x4_t{0.f, 0.f, 0.f, 0.f};
    u32x4_t fx[ST > 1 ? ST : 2][MT][2], fw[ST][NT];
    const uint32_t lo = static_cast<uint32_t>(l) * 8;
    auto load_w = [&](int slot, int t, int s) { fw[slot][t] = *(const NAVI_GLOBAL u32x4_t *) (wb[t] + s * 512 + lo); };
    auto load_x = [&](int slot, int s) {
#pragma unroll
        for (int i = 0; i < MT; ++i)
#pragma unroll
            for (int p = 0; p < 2; ++p) fx[slot][i][p] = *(const NAVI_GLOBAL u32x4_t *) (xb[i] + s * 1024 + p * 512 + lo);
    };
    auto load = [&](int slot, int s) {
#pragma unroll
        for (int t = 0; t < NT; ++t) load_w(slot, t, s);
        load_x(slot, s);
    };
    // a step's lo (p = 1), then hi products: from zero into part, which add() adds to the tile's sums, or (CHAIN)
    // straight onto them
    auto product = [&](f32x4_t &part, f32x4_t &sum, const ghalf8 &wv, const ghalf8 &xv, int p) {
        if constexpr (CHAIN) sum = __builtin_amdgcn_mfma_f32_16x16x32_f16(wv, xv, sum, 0, 0, 0);
        else part = __builtin_amdgcn_mfma_f32_16x16x32_f16(wv, xv, p ? f32x4_t{0.f, 0.f, 0.f, 0.f} : part, 0, 0, 0);
    };
    auto add = [&](f32x4_t &sum, const f32x4_t &part) {
        if constexpr (!CHAIN) sum += part;
    };
    auto mma = [&](int slot) {
#pragma unroll
        for (int i = 0; i < MT; ++i) {
            f32x4_t part[NT];
#pragma unroll
            for (int p = 1; p >= 0; --p) {
                ghalf8 xv;
                __builtin_memcpy(&xv, &fx[slot][i][p], 16);
#pragma unroll
                for (int t = 0; t < NT; ++t) {
                    ghalf8 wv;
                    __builtin_memcpy(&wv, &fw[slot][t], 16);
                    product(part[t], acc[i][t], wv, xv, p);
                }
            }
#pragma unroll
            for (int t = 0; t < NT; ++t) add(acc[i][t], part[t]);
        }
    };
#pragma unroll
    for (int u = 0; u < ST - 1; ++u) load(u, u);
    if constexpr (ST == 1) load(0, 0);
    const int m = (row * MT + w) * 16 + (l & 15);           // the row this lane finishes (w < MT)
    Epilogue<NT, EPI> end;
    end.load(a, col, m, g);
    if constexpr (MT == 1) end.load_head(a, col, m, g);
    __builtin_amdgcn_sched_barrier(0);
    if constexpr (ST == 1) {
        auto step = [&](int xs, int s, bool more) {
            if (more) load_x(xs ^ 1, s + 1);
#pragma unroll
            for (int t = 0; t < NT; ++t) {
                ghalf8 wv;
                __builtin_memcpy(&wv, &fw[0][t], 16);
                f32x4_t part[MT];
#pragma unroll
                for (int p = 1; p >= 0; --p)
#pragma unroll
                    for (int i = 0; i < MT; ++i) {
                        ghalf8 xv;
                        __builtin_memcpy(&xv, &fx[xs][i][p], 16);
                        product(part[i], acc[i][t], wv, xv, p);
                    }
#pragma unroll
                for (int i = 0; i < MT; ++i) add(acc[i][t], part[i]);
                if (more) load_w(0, t, s + 1);
                __builtin_amdgcn_sched_barrier(0);
            }
        };
        static_assert(ST > 1 || PER % 2 == 0, "two X slots");
#pragma unroll 1
        for (int s = 0; s < PER - 2; s += 2) {
            step(0, s, true);
            step(1, s + 1, true);
        }
        step(0, PER - 2, true);
        step(1, PER - 1, false);
    } else {
        int s = 0;
#pragma unroll 1
        for (; s < PER - ST; s += ST)
#pragma unroll
            for (int u = 0; u < ST; ++u) {
                load((u + ST - 1) % ST, s + u + ST - 1);
                __builtin_amdgcn_sched_barrier(0);
                mma(u);
                __builtin_amdgcn_sched_barrier(0);
            }
#pragma unroll
        for (int u = 0; u < ST; ++u) {
            if (u == 0) load(ST - 1, PER - 1);
            mma(u);
        }
    }
    if constexpr (MT > 1 && ST > 1) end.load_head(a, col, m, g);
    // wave o finishes 16-row tile o; sums in wave order whichever wave it is; uniform branches and constant
    // indices (an indexed register array would go to memory)
    f32x4_t v[NT];
#pragma unroll
    for (int j = 0; j < MT; j += MX) {
        if (j) __syncthreads();                             // the previous tiles' readers are done
#pragma unroll
        for (int o = j; o < j + MX; ++o)
            if (o != w) {
                const int src = w < o ? w : w - 1;
#pragma unroll
                for (int t = 0; t < NT; ++t) red[o - j][src][t][l] = acc[o][t];
            }
        __syncthreads();
#pragma unroll
        for (int o = j; o < j + MX; ++o)
            if (o == w)
#pragma unroll
                for (int t = 0; t < NT; ++t) {
                    f32x4_t sum = o == 0 ? acc[o][t] : red[o - j][0][t][l];
#pragma unroll
                    for (int u = 1; u < NW; ++u) sum += u == o ? acc[o][t] : red[o - j][u < o ? u : u - 1][t][l];
                    v[t] = sum;
                }
    }
    if (w >= MT) return;
    if constexpr (MT > 1 && ST == 1) end.load_head(a, col, m, g);
    bool bad = false;
    end.finish(a, col, m, mtiles, g, v, bad);
    if (bad) gst(a.flag, 1u);
}

// xs = split(rows * ln), x = rows (rows.h pk_a) and their partial sums of squares: the first norm's
// half of the layers' hand-over, one block per row of H = 1024.
__global__ void __launch_bounds__(256) k_split_rows(const float *src, const float *ln, float *x, uint16_t *xs, float *ssq, int ldq,
                                                    uint32_t *flag) {
    const int m = blockIdx.x, k = 4 * static_cast<int>(threadIdx.x);
    constexpr int H = 1024;
    const f32x4_t v = ld4(src + static_cast<size_t>(m) * H + k), w = ld4(ln + k);
    st4(x + rows::pk_a(m, k, H), v);
    bool bad = false;
    split_store4(xs + pk_s(m, k, H), v * w, bad);
    float s = 0.f;
#pragma unroll
    for (int r = 0; r < 4; ++r) s = fmaf(v[r], v[r], s);
    s += dpp_red<0xB1>(s);                                   // eight lanes hold a group of 32 columns
    s += dpp_red<0x4E>(s);
    s += dpp_red<0x141>(s);
    if ((threadIdx.x & 7) == 0) gst(ssq + (threadIdx.x >> 3) * ldq + m, s);
    if (bad) gst(flag, 1u);
}

// Causal attention of a prompt from position 0 on the matrix cores, both q heads of a kv group and 16
// query rows per block. Queries, keys and values come in fragment order (GemmArgs::q, kf, vf), so every
// operand is a 1 KB load straight into registers; wave w takes the 32-key steps w, w + 4, ... with a
// running softmax of its own. Scores are computed transposed (K Q^T: lane l holds query row l % 16 and
// keys 4 (l / 16) .. + 3 of each 16-key tile): the probabilities of a lane are its own MFMA operand for
// V^T P^T (vf holds the keys in that order), split into f16 hi + lo as the queries are. The four
// waves' sums meet in LDS at the end. The exponentials are the hardware's 2^x of the unscaled scores'
// distance from the maximum (one rounding of the difference, one of its product with the scale): expf
// took more instructions than everything else here. Grid (kv groups, row tiles), the tiles with the most keys first; kv group g's blocks run
// on XCD g, whose L2 holds its keys and values.
struct AttnArgs {
    const uint16_t *q, *kf, *vf;
    uint16_t *att;                    // split layout [T][nq 128]
    uint32_t *flag;
    int T, nq;
    float scale;                      // of the scores, times log2(e): the softmax is taken in powers of two
};

__global__ void __launch_bounds__(4 * WAVE, 2) k_attn_prompt(AttnArgs a) {
    __shared__ f32x4_t ob[4][2][8][WAVE];
    __shared__ float mb[4][2][16], lb[4][2][16];
    const int w = __builtin_amdgcn_readfirstlane(static_cast<int>(threadIdx.x) >> 6), l = static_cast<int>(threadIdx.x) & 63;
    const int c = l & 15, g = l >> 4, kv = blockIdx.x, qt = static_cast<int>(gridDim.y) - 1 - static_cast<int>(blockIdx.y);
    const int row = 16 * qt + c, steps = (static_cast<int>(gridDim.y) + 1) >> 1, mine = (qt >> 1) + 1;
    const uint32_t lo = static_cast<uint32_t>(l) * 8;
    const uint16_t *kb = a.kf + static_cast<size_t>(kv) * steps * 4096, *vb = a.vf + static_cast<size_t>(kv) * steps * 4096;
    ghalf8 qf[2][4][2];
    {
        const uint16_t *qb = a.q + (static_cast<size_t>(qt) * (a.nq * 4) + kv * 8) * 1024;
#pragma unroll
        for (int h = 0; h < 2; ++h)
#pragma unroll
            for (int s = 0; s < 4; ++s)
#pragma unroll
                for (int p = 0; p < 2; ++p) qf[h][s][p] = *(const NAVI_GLOBAL ghalf8 *) (qb + (h * 4 + s) * 1024 + p * 512 + lo);
    }
    f32x4_t o[2][8];
    float mx[2] = {-INFINITY, -INFINITY}, sum[2] = {0.f, 0.f};
#pragma unroll
    for (int h = 0; h < 2; ++h)
#pragma unroll
        for (int t = 0; t < 8; ++t) o[h][t] = f32x4_t{0.f, 0.f, 0.f, 0.f};
    ghalf8 kf[8], vf[8];
    auto load_k = [&](int s) {
#pragma unroll
        for (int i = 0; i < 8; ++i) kf[i] = *(const NAVI_GLOBAL ghalf8 *) (kb + static_cast<size_t>(s) * 4096 + i * 512 + lo);
    };
    if (w < mine) load_k(w);
    for (int s = w; s < mine; s += 4) {
#pragma unroll
        for (int i = 0; i < 8; ++i) vf[i] = *(const NAVI_GLOBAL ghalf8 *) (vb + static_cast<size_t>(s) * 4096 + i * 512 + lo);
        f32x4_t sc[2][2];
#pragma unroll
        for (int h = 0; h < 2; ++h)
#pragma unroll
            for (int t = 0; t < 2; ++t) sc[h][t] = f32x4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int p = 1; p >= 0; --p)                         // the small products first
#pragma unroll
            for (int st = 0; st < 4; ++st)
#pragma unroll
                for (int h = 0; h < 2; ++h)
#pragma unroll
                    for (int t = 0; t < 2; ++t)
                        sc[h][t] = __builtin_amdgcn_mfma_f32_16x16x32_f16(kf[4 * t + st], qf[h][st][p], sc[h][t], 0, 0, 0);
        if (s + 4 < mine) load_k(s + 4);
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            ghalf8 ph, pl;
            float m = mx[h];
#pragma unroll
            for (int t = 0; t < 2; ++t)
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    const int key = 32 * s + 16 * t + 4 * g + r;
                    sc[h][t][r] = key <= row ? sc[h][t][r] : -INFINITY;
                    m = fmaxf(m, sc[h][t][r]);
                }
            m = fmaxf(m, __shfl_xor(m, 16));
            m = fmaxf(m, __shfl_xor(m, 32));                 // finite: a step's first key is no later than any row
            const float corr = __builtin_amdgcn_exp2f((mx[h] - m) * a.scale);
            mx[h] = m;
            float ls = 0.f;
#pragma unroll
            for (int t = 0; t < 2; ++t)
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    const float e = __builtin_amdgcn_exp2f((sc[h][t][r] - m) * a.scale);
                    ls += e;
                    const _Float16 hi = static_cast<_Float16>(e);
                    ph[4 * t + r] = hi;
                    pl[4 * t + r] = static_cast<_Float16>(e - static_cast<float>(hi));
                }
            sum[h] = sum[h] * corr + ls;
#pragma unroll
            for (int t = 0; t < 8; ++t) {
                f32x4_t p = __builtin_amdgcn_mfma_f32_16x16x32_f16(vf[t], pl, f32x4_t{0.f, 0.f, 0.f, 0.f}, 0, 0, 0);
                p = __builtin_amdgcn_mfma_f32_16x16x32_f16(vf[t], ph, p, 0, 0, 0);
#pragma unroll
                for (int r = 0; r < 4; ++r) o[h][t][r] = fmaf(o[h][t][r], corr, p[r]);
            }
        }
    }
#pragma unroll
    for (int h = 0; h < 2; ++h) {
        const float t = group_sum(sum[h]);
        if (g == 0) {
            mb[w][h][c] = mx[h];
            lb[w][h][c] = t;
        }
#pragma unroll
        for (int i = 0; i < 8; ++i) ob[w][h][i][l] = o[h][i];
    }
    __syncthreads();
    // wave w: head w % 2, dims 64 (w / 2) .. + 63; the waves' parts in wave order
    const int h = w & 1, t0 = 4 * (w >> 1);
    const float m = fmaxf(fmaxf(mb[0][h][c], mb[1][h][c]), fmaxf(mb[2][h][c], mb[3][h][c]));
    float f[4], total = 0.f;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        f[i] = __builtin_amdgcn_exp2f((mb[i][h][c] - m) * a.scale);   // 0 for a wave without keys
        total += f[i] * lb[i][h][c];
    }
    bool bad = false;
#pragma unroll
    for (int t = 0; t < 4; ++t) {
        f32x4_t v = f[0] * ob[0][h][t0 + t][l];
#pragma unroll
        for (int i = 1; i < 4; ++i) v += f[i] * ob[i][h][t0 + t][l];
        v /= total;
        if (row < a.T) split_store4(a.att + pk_s(row, (2 * kv + h) * 128 + 16 * (t0 + t) + 4 * g, a.nq * 128), v, bad);
    }
    if (bad) gst(a.flag, 1u);
}

template <int MT, int NT, int EPI, int NW, int PER, int ST, int WPS, int MX = MT>
void launch_gemm(const GemmArgs &a, hipStream_t s) {
    const int ncol = EPI == G_SWIGLU ? a.N / (8 * NT) : a.N / (16 * NT), nrow = ((a.M + 15) / 16 + MT - 1) / MT;
    hipLaunchKernelGGL((k_gemm<MT, NT, EPI, NW, PER, ST, WPS, MX>), dim3(ncol * nrow), dim3(NW * WAVE), 0, s, a);
}

// The talker's shapes (K 1024 into q|k|v and gate|up, 2048 into o, 3072 into down; N 4096, 2 x 3072,
// 1024, 1024). A launch takes about as long as its longest block as long as every block has a CU of
// its own, so the tile is the smallest that still gives at most 256 blocks: a block's time is its
// operand bytes (about 70 GB/s from L2 into one CU, whatever the other CUs do), and a block more
// than CUs is a second round. Above 512 rows no tile gives that: there the one-slot form, two blocks to a
// CU (768 rows: gate|up 30 -> 25 us, with chained sums q|k|v 26 -> 23; its 32 x 128 tiles that add each step's
// products 26.7), except q|k|v above 768 rows, whose 64 x 128 tiles do not fit half the registers with
// a step's products beside the sums (1001 rows 32 us; chained in half the registers 26.5).
void launch_qkv(const GemmArgs &a, hipStream_t s) {
    const int mt = (a.M + 15) / 16;
    if (mt <= 8) launch_gemm<1, 8, G_QKV, 4, 8, 2, 2>(a, s);
    else if (mt <= 16) launch_gemm<2, 8, G_QKV, 4, 8, 2, 1>(a, s);
    else if (mt <= 24) launch_gemm<3, 8, G_QKV, 4, 8, 2, 1>(a, s);
    else if (mt <= 32) launch_gemm<4, 8, G_QKV, 4, 8, 2, 1>(a, s);
    else if (mt <= 48) launch_gemm<2, 8, G_QKV, 4, 8, 1, 2>(a, s);
    else launch_gemm<4, 8, G_QKV, 4, 8, 2, 1>(a, s);
}
void launch_gate_up(const GemmArgs &a, hipStream_t s) {
    const int mt = (a.M + 15) / 16;
    if (mt <= 5) launch_gemm<1, 8, G_SWIGLU, 4, 8, 2, 2>(a, s);
    else if (mt <= 8) launch_gemm<2, 6, G_SWIGLU, 4, 8, 2, 2>(a, s);
    else if (mt <= 10) launch_gemm<2, 8, G_SWIGLU, 4, 8, 2, 1>(a, s);
    else if (mt <= 16) launch_gemm<4, 6, G_SWIGLU, 4, 8, 2, 1>(a, s);
    else if (mt <= 32) launch_gemm<4, 12, G_SWIGLU, 4, 8, 2, 1>(a, s);
    else launch_gemm<4, 6, G_SWIGLU, 4, 8, 1, 2, 2>(a, s);
}
// STEPS = K / 32
template <int STEPS>
void launch_resid(const GemmArgs &a, hipStream_t s) {
    const int mt = (a.M + 15) / 16;
    if (mt <= 8) launch_gemm<1, 2, G_RESID, 8, STEPS / 8, 4, 2>(a, s);
    else if (mt <= 16) launch_gemm<2, 2, G_RESID, 8, STEPS / 8, 2, 2>(a, s);
    else if (mt <= 32) launch_gemm<2, 4, G_RESID, 8, STEPS / 8, 2, 2>(a, s);
    else launch_gemm<4, 4, G_RESID, 8, STEPS / 8, 1, 2>(a, s);
}

} // namespace
} // namespace gm
} // namespace navi_amd
