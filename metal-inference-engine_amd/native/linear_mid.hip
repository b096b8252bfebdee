// Linears of a full decode batch or a short prompt (33 to a few hundred rows), gfx950; semantics in linear_gemm.hip.
//
// What bounds them is reading W (2048 x 6144 INT4: 7.9 MB, 1.5 us at a copy's rate) and the latency of a chain of
// launches, so W is read once, as stored, straight into MFMA operands, and the whole chip shares it: a workgroup takes
// 16 NT weight rows and one K-split, its eight waves an eighth of the split each, and every wave multiplies its blocks
// with all the activation rows of a row block (48 or 64). The activations come as operand-ready pieces from memory
// (the L2s hold them: 6 bytes per value, 0.8 MB for 64 x 2048), written once by split_operands; they pass through no
// LDS, since no two waves of a workgroup use the same ones. Operands are linear_operands.h's: three bf16 pieces of every
// activation and the weights, all exact. A block's scale multiplies its sums on the VALU; an INT4 weight is
// s (q - 8) + (8 s + min), whose second term, times the block's activation sum, is one more MFMA per 4 blocks. The
// waves' sums meet in LDS; K-splits meet in memory, added in order by mid_finish.
//
// Measured (64 rows, INT4, all launches): 12288 x 2048 with silu * up 26 us, 2048 x 6144 28 us (gemm_rows 48 and 37, the
// fp32 GEMM on the expanded weight 100 and 110; two fp16 pieces of x 23 and 23).
#include "linear_operands.h"

namespace rk {
namespace {

constexpr int kWaves = 8;
constexpr int P = 3;               // pieces of an activation

struct MidArgs {
    float* y;
    const uint16_t* a;             // [row block][K / 32][piece][MT][64 lanes][8]: MFMA operands
    const uint16_t* sums;          // INT4: [row block][K / 32][MT][16 rows][8] block sums (split_operands)
    const void* w;
    const uint16_t* scales;
    const uint16_t* mins;
    const float* bias;
    const float* res;
    f32x4* part;                   // S > 1: [row block][row group][split][item]
    int M, N, K;                   // N: weight rows (glu: both halves)
    int S, SB, WB;                 // splits; blocks per split and per wave
    int MB, G, glu;                // row blocks; groups of 16 NT weight rows
};

// Row m of x as operands of the row block m / (16 MT): lane (r, g) of tile i takes row 16 i + r's values 8g .. 8g + 7
// of a block, in three pieces (INT4: in the order of int4_bf16). INT4: also each block's sum, in pieces b1 b2 b3 as
// (b1, b1, b1, b2, b2, b2, b3, b3), against the pieces of 8 s + min as (c1, c2, c3, c1, c2, c3, c1, c2): all products but
// the last, 2^-32 of the whole.
template <int WT, int MT>
__global__ __launch_bounds__(256) void split_operands(uint16_t* a, uint16_t* sums, const float* x, long long x_ld, int K) {
    const int m = blockIdx.x, tid = threadIdx.x;
    const int mb = m / (16 * MT), i = m % (16 * MT) / 16, r = m % 16, nblk = K / kQB;
    const float* xr = x + (size_t)m * x_ld;
    // a thread's first kHeld groups of 8 values are requested together
    constexpr int kHeld = 4;
    f32x4 held[kHeld][2];
#pragma unroll
    for (int j = 0; j < kHeld; ++j) {
        const float* p = xr + 8 * min(tid + 256 * j, K / 8 - 1);
        held[j][0] = *reinterpret_cast<const f32x4*>(p);
        held[j][1] = *reinterpret_cast<const f32x4*>(p + 4);
    }
    auto put = [&](int c, f32x4 v0, f32x4 v1) __attribute__((always_inline)) {
        const float v[8] = {v0[0], v0[1], v0[2], v0[3], v1[0], v1[1], v1[2], v1[3]};
        u32x4 pc[P];
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            const Split3 s0 = split3_any(v[WT == RK_W_INT4 ? kInt4Order[q][0] : 2 * q]);
            const Split3 s1 = split3_any(v[WT == RK_W_INT4 ? kInt4Order[q][1] : 2 * q + 1]);
            pc[0][q] = pack_hi2(s0.hi, s1.hi);
            pc[1][q] = pack_hi2(s0.mid, s1.mid);
            pc[2][q] = pack_hi2(s0.lo, s1.lo);
        }
        const size_t blk = (size_t)mb * nblk + (c >> 2);
#pragma unroll
        for (int p = 0; p < P; ++p)
            *reinterpret_cast<u32x4*>(a + (((blk * P + p) * MT + i) * 64 + 16 * (c & 3) + r) * 8) = pc[p];
        if constexpr (WT == RK_W_INT4) {           // the four threads of a block are neighbours in one wave
            float sum = 0.0f;
#pragma unroll
            for (int e = 0; e < 8; ++e) sum += v[e];
            sum += dpp_f32<0xb1>(sum);             // lane ^ 1
            sum += dpp_f32<0x4e>(sum);             // lane ^ 2
            if ((c & 3) == 0) {
                const Split3 b = split3_any(sum);
                *reinterpret_cast<u32x4*>(sums + ((blk * MT + i) * 16 + r) * 8) =
                    (u32x4){pack_hi2(b.hi, b.hi), pack_hi2(b.hi, b.mid), pack_hi2(b.mid, b.mid), pack_hi2(b.lo, b.lo)};
            }
        }
    };
#pragma unroll
    for (int j = 0; j < kHeld; ++j)
        if (tid + 256 * j < K / 8) put(tid + 256 * j, held[j][0], held[j][1]);
    for (int c = tid + 256 * kHeld; c < K / 8; c += 256)
        put(c, *reinterpret_cast<const f32x4*>(xr + 8 * c), *reinterpret_cast<const f32x4*>(xr + 8 * c + 4));
}

// weight row behind row lr of the tiles: lr, or with glu gate rows 8T .. 8T + 7 then their up rows in tile T
__device__ __forceinline__ size_t mid_row(const MidArgs& a, int lr) {
    if (!a.glu) return (size_t)min(lr, a.N - 1);
    const int F = a.N >> 1, f = min(8 * (lr >> 4) + (lr & 7), F - 1);
    return (size_t)((lr & 8) ? F + f : f);
}

// rows 4g .. 4g + 3 of tile i, column c of tile t (lane l = 16 g + c of item (i, t)): bias, residual or silu * up, store;
// whole waves enter
template <int MT, int NT>
__device__ __forceinline__ void mid_store(const MidArgs& a, f32x4 v, int mb, int rg, int item) {
    const int i = item / (64 * NT), t = item / 64 % NT, l = item & 63, c = l & 15;
    const int m0 = 16 * MT * mb + 16 * i + 4 * (l >> 4);
    if (a.glu) {                                   // uniform
        f32x4 u;
#pragma unroll
        for (int e = 0; e < 4; ++e) u[e] = dpp_f32<0x128>(v[e]);   // row_ror:8 (lane ^ 8)
        const int F = a.N >> 1, n = 8 * (rg * NT + t) + (c & 7);
        if (c < 8 && n < F) {
#pragma unroll
            for (int e = 0; e < 4; ++e)
                if (m0 + e < a.M) a.y[(size_t)(m0 + e) * F + n] = silu_times(v[e], u[e]);
        }
        return;
    }
    const int n = 16 * (rg * NT + t) + c;
    if (n >= a.N) return;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
        if (m0 + e >= a.M) continue;
        float o = v[e];
        if (a.bias) o = __fadd_rn(o, a.bias[n]);
        if (a.res) o = __fadd_rn(o, a.res[(size_t)(m0 + e) * a.N + n]);
        a.y[(size_t)(m0 + e) * a.N + n] = o;
    }
}

// One workgroup per (row group, K-split, row block). A wave walks its blocks four at a time (a chunk: 16-byte weight
// loads of whole blocks, transposed over the lane groups as in linear.hip), the next chunk's weights and scales and the
// next block's activations requested ahead. Chunks past the wave's range repeat loaded addresses and enter with
// weight 0, so the loop body has no branch.
template <int WT, int MT, int NT>
__global__ __launch_bounds__(64 * kWaves) void mid_rows(MidArgs a) {
    constexpr int CH = WT == RK_W_INT4 ? 1 : WT == RK_W_INT8 ? 2 : 4;   // 16-byte loads per tile and chunk
    constexpr bool QUANT = WT != RK_W_BF16;
    extern __shared__ __attribute__((aligned(16))) char smem[];
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int r = lane & 15, grp = lane >> 4;
    const int nblk = a.K / kQB;
    // row blocks of one (row group, split) are 8 workgroups apart: on one XCD, whose L2 keeps the weights for them
    const int oct = blockIdx.x / (8 * a.MB), in8 = blockIdx.x % (8 * a.MB);
    const int t_id = 8 * oct + in8 % 8, mb = in8 / 8;
    if (t_id >= a.G * a.S) return;
    const int rg = t_id / a.S, sp = t_id % a.S;
    const int k0 = sp * a.SB + wave * a.WB;
    const int k1 = min(min(nblk, (sp + 1) * a.SB), k0 + a.WB);

    const uint8_t* wrow[NT];
    const uint16_t* srow[NT];
    const uint16_t* mrow[NT];
#pragma unroll
    for (int t = 0; t < NT; ++t) {
        const size_t n = mid_row(a, 16 * (rg * NT + t) + r);
        wrow[t] = static_cast<const uint8_t*>(a.w) + n * ((size_t)nblk * (WT == RK_W_BF16 ? 64 : WT == RK_W_INT8 ? 32 : 16));
        if constexpr (QUANT) srow[t] = a.scales + n * nblk;
        if constexpr (WT == RK_W_INT4) mrow[t] = a.mins + n * nblk;
    }
    constexpr int DEPTH = WT == RK_W_INT4 && MT * NT < 12 ? 2 : 1;   // chunks of weights in flight (as registers allow)
    u32x4 wn[DEPTH][NT][CH];
    uint32_t sn[DEPTH][QUANT ? NT : 1][2];
    uint16_t mn[DEPTH][WT == RK_W_INT4 ? NT : 1];  // min of the lane group's own block of the chunk
    auto load_w = [&](int kb, int set) __attribute__((always_inline)) {
#pragma unroll
        for (int t = 0; t < NT; ++t) {
#pragma unroll
            for (int c = 0; c < CH; ++c) {
                size_t off;
                if constexpr (WT == RK_W_BF16) off = (size_t)min(kb + c, nblk - 1) * 64 + 16 * grp;
                else if constexpr (WT == RK_W_INT8) off = (size_t)min(kb + grp, nblk - 1) * 32 + 16 * c;
                else off = (size_t)min(kb + grp, nblk - 1) * 16;
                wn[set][t][c] = *reinterpret_cast<const u32x4*>(wrow[t] + off);
            }
            if constexpr (QUANT) {                 // nblk and kb are even
#pragma unroll
                for (int h = 0; h < 2; ++h) {
                    sn[set][t][h] = *reinterpret_cast<const uint32_t*>(srow[t] + min(kb + 2 * h, nblk - 2));
                }
            }
            if constexpr (WT == RK_W_INT4) mn[set][t] = mrow[t][min(kb + grp, nblk - 1)];
        }
    };
    u32x4 xa[2][P][MT];
    auto load_x = [&](int kb, int slot) {
        const size_t blk = (size_t)mb * nblk + min(kb, nblk - 1);
#pragma unroll
        for (int p = 0; p < P; ++p)
#pragma unroll
            for (int i = 0; i < MT; ++i)
                xa[slot][p][i] = *reinterpret_cast<const u32x4*>(a.a + (((blk * P + p) * MT + i) * 64 + lane) * 8);
    };
    f32x4 acc[MT][NT];
#pragma unroll
    for (int i = 0; i < MT; ++i)
#pragma unroll
        for (int t = 0; t < NT; ++t) acc[i][t] = (f32x4){0.f, 0.f, 0.f, 0.f};

    const int k_last = k0 + (k1 - 1 - k0) / 4 * 4;   // the wave's last chunk
    if (k0 < k1) {
#pragma unroll
        for (int i = 0; i < DEPTH; ++i) load_w(min(k0 + 4 * i, k_last), i);
        load_x(k0, 0);
    }
    for (int kc = k0; kc < k1; kc += 4) {
        u32x4 wc[NT][CH];
        uint32_t sc[QUANT ? NT : 1][2];
        uint16_t mc[WT == RK_W_INT4 ? NT : 1];
#pragma unroll
        for (int t = 0; t < NT; ++t) {
            if constexpr (WT == RK_W_INT4) wc[t][0] = xpose4(wn[0][t][0][0], wn[0][t][0][1], wn[0][t][0][2], wn[0][t][0][3]);
            else if constexpr (WT == RK_W_INT8) {
                const u32x4 lo = xpose4(wn[0][t][0][0], wn[0][t][0][2], wn[0][t][1][0], wn[0][t][1][2]);
                const u32x4 hi = xpose4(wn[0][t][0][1], wn[0][t][0][3], wn[0][t][1][1], wn[0][t][1][3]);
                wc[t][0] = (u32x4){lo[0], hi[0], lo[1], hi[1]};
                wc[t][1] = (u32x4){lo[2], hi[2], lo[3], hi[3]};
            } else {
#pragma unroll
                for (int c = 0; c < CH; ++c) wc[t][c] = wn[0][t][c];
            }
            if constexpr (QUANT) {
#pragma unroll
                for (int h = 0; h < 2; ++h) sc[t][h] = sn[0][t][h];
            }
            if constexpr (WT == RK_W_INT4) mc[t] = mn[0][t];
            if constexpr (DEPTH == 2) {
#pragma unroll
                for (int c = 0; c < CH; ++c) wn[0][t][c] = wn[1][t][c];
                if constexpr (QUANT) {
#pragma unroll
                    for (int h = 0; h < 2; ++h) sn[0][t][h] = sn[1][t][h];
                }
                if constexpr (WT == RK_W_INT4) mn[0][t] = mn[1][t];
            }
        }
        load_w(min(kc + 4 * DEPTH, k_last), DEPTH - 1);
        u32x4 bs[WT == RK_W_INT4 ? MT : 1];
        if constexpr (WT == RK_W_INT4) {
#pragma unroll
            for (int i = 0; i < MT; ++i)
                bs[i] = *reinterpret_cast<const u32x4*>(
                    a.sums + ((((size_t)mb * nblk + min(kc + grp, nblk - 1)) * MT + i) * 16 + r) * 8);
        }
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int d = 0; d < 4; ++d) {
            const int s = d & 1;
            // past the wave's range: zero scales, zero bf16 weights (a mask; a condition becomes a branch)
            const uint32_t in = kc + d < k1 ? 0xffffffffu : 0u;
            load_x(min(kc + d + 1, k1 - 1), s ^ 1);
#pragma unroll
            for (int t = 0; t < NT; ++t) {
                u32x4 b;
                if constexpr (WT == RK_W_INT4) b = int4_bf16_centred(wc[t][0][d]);
                else if constexpr (WT == RK_W_INT8) b = int8_bf16(wc[t][d >> 1][2 * (d & 1)], wc[t][d >> 1][2 * (d & 1) + 1]);
                else b = wc[t][d] & (u32x4){in, in, in, in};
                float f = 0.0f;
                if constexpr (QUANT) f = half_to_f32((uint16_t)((sc[t][d >> 1] & in) >> (16 * (d & 1))));
#pragma unroll
                for (int i = 0; i < MT; ++i) {
                    f32x4 p = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
                    for (int q = P - 1; q >= 0; --q) p = mfma16x16x32(xa[s][q][i], b, p);
#pragma unroll
                    for (int e = 0; e < 4; ++e) {
                        if constexpr (QUANT) acc[i][t][e] = fmaf(f, p[e], acc[i][t][e]);
                        else acc[i][t][e] += p[e];
                    }
                }
            }
            __builtin_amdgcn_sched_barrier(0);     // one block ahead: more in flight does not fit the registers
        }
        if constexpr (WT == RK_W_INT4) {           // 8 s + min of the lane group's block, in the pieces that meet its sum's
            const uint32_t in = kc + grp < k1 ? 0xffffffffu : 0u;
#pragma unroll
            for (int t = 0; t < NT; ++t) {
                const uint64_t s4 = (uint64_t)sc[t][1] << 32 | sc[t][0];
                const float c = fmaf(8.0f, half_to_f32((uint16_t)(s4 >> (16 * grp))), half_to_f32(mc[t]));
                const Split3 p = split3(__uint_as_float(__float_as_uint(c) & in));
                const u32x4 b = {pack_hi2(p.hi, p.mid), pack_hi2(p.lo, p.hi), pack_hi2(p.mid, p.lo), pack_hi2(p.hi, p.mid)};
#pragma unroll
                for (int i = 0; i < MT; ++i) acc[i][t] = mfma16x16x32(bs[i], b, acc[i][t]);
                __builtin_amdgcn_sched_barrier(0);
            }
        }
    }

    // the waves' sums, in wave order
    constexpr int ITEMS = 64 * MT * NT;
    f32x4* red = reinterpret_cast<f32x4*>(smem);
#pragma unroll
    for (int i = 0; i < MT; ++i)
#pragma unroll
        for (int t = 0; t < NT; ++t) red[wave * ITEMS + (i * NT + t) * 64 + lane] = acc[i][t];
    __syncthreads();
    for (int item = threadIdx.x; item < ITEMS; item += 64 * kWaves) {
        f32x4 v = red[item];
#pragma unroll
        for (int w = 1; w < kWaves; ++w) {
            const f32x4 o = red[w * ITEMS + item];
#pragma unroll
            for (int e = 0; e < 4; ++e) v[e] += o[e];
        }
        if (a.S == 1) mid_store<MT, NT>(a, v, mb, rg, item);
        else a.part[((size_t)(mb * a.G + rg) * a.S + sp) * ITEMS + item] = v;
    }
}

// The splits of one (row block, row group, wave of items), in order.
template <int MT, int NT>
__global__ __launch_bounds__(256) void mid_finish(MidArgs a) {
    constexpr int ITEMS = 64 * MT * NT;
    const int item = 256 * blockIdx.y + threadIdx.x;
    if (item >= ITEMS) return;                     // whole waves
    const f32x4* p = a.part + (size_t)blockIdx.x * a.S * ITEMS + item;
    f32x4 v = p[0];
    for (int s = 1; s < a.S; ++s) {
        const f32x4 o = p[(size_t)s * ITEMS];
#pragma unroll
        for (int e = 0; e < 4; ++e) v[e] += o[e];
    }
    mid_store<MT, NT>(a, v, blockIdx.x / a.G, blockIdx.x % a.G, item);
}

// What the time is made of, in us: the launches and x's pieces; a round of one workgroup per CU: its start, and for each
// chunk of four blocks a wave walks a constant, the activations from the L2 (per row tile, more when every CU asks) and
// the MFMAs (per row and weight tile); mid_finish and the partial sums it reads. Fitted to 14 weights of 1024 x 1024 to
// 12288 x 2048, 33 to 384 rows, x the NT and S there are: 10 % of root mean square error; NT and S chosen by it cost on
// average 0.5 % more than the best measured, 9 % at worst.
struct MidCost {
    double launch, split, start, item, chunk, x, x_full, mfma, finish, part;
};
constexpr MidCost kCost[3] = {{6.7, 5.9e-6, 0.0, 0.37, 1.51, 0.24, 0.17, 0.294, 1.8, 0.0},         // bf16
                              {6.9, 5.7e-6, 0.0, 0.34, 1.77, 0.08, 0.21, 0.309, 1.8, 0.046e-3},    // INT8
                              {7.1, 5.3e-6, 1.2, 0.31, 2.35, 0.0, 0.20, 0.320, 1.9, 0.070e-3}};    // INT4

}  // namespace

// kMost: the estimates end there; no weight measured was faster here at 512 rows. Scales and mins are read two blocks at
// a time.
MidPlan mid_plan(int M, int N, int K, int w_type, int glu) {
    constexpr int kMost = 384;
    MidPlan p{};
    if (M > kMost || K % (2 * kQB)) return p;
    const int nblk = K / kQB;
    const int tiles = glu ? (N / 2 + 7) / 8 : (N + 15) / 16;
    p.MB = (M + 63) / 64;
    p.MT = (M + 16 * p.MB - 1) / (16 * p.MB) <= 3 ? 3 : 4;
    int cus = device_cus();
    if (cus <= 0) cus = 256;
    const MidCost& c = kCost[w_type == RK_W_BF16 ? 0 : w_type == RK_W_INT8 ? 1 : 2];
    for (int nt = 1; nt <= (w_type == RK_W_BF16 ? 2 : p.MT == 4 ? 3 : 4); ++nt)   // as the registers hold
        for (int s = 1; s <= 16 && s <= (nblk + 31) / 32 * 2; ++s) {
            const int sb = ((nblk + s - 1) / s + 1) / 2 * 2;
            const int wb = ((sb + kWaves - 1) / kWaves + 1) / 2 * 2;
            const int g = (tiles + nt - 1) / nt, used = (nblk + sb - 1) / sb;
            const long long groups = (long long)g * used * p.MB, rounds = (groups + cus - 1) / cus;
            const double full = (double)groups / (double)(rounds * cus);
            double us = c.launch + c.split * (double)M * K +
                        (double)rounds * (c.start + c.item * p.MT * nt +
                                          (wb + 3) / 4 * (c.chunk + p.MT * (c.x + c.x_full * full + c.mfma * nt)));
            if (used > 1) us += c.finish + c.part * (double)groups * nt * p.MT;
            if (p.us == 0.0 || us < p.us) {
                p.us = us;
                p.NT = nt; p.G = g; p.S = used; p.SB = sb; p.WB = wb;
            }
        }
    const size_t rows = (size_t)p.MB * 16 * p.MT;
    auto up = [](size_t n) { return (n + 255) / 256 * 256; };
    p.sums = up(rows * K * 2 * P);
    p.part = p.sums + (w_type == RK_W_INT4 ? up(rows * nblk * 16) : 0);
    p.total = p.part + (p.S > 1 ? (size_t)p.MB * p.G * p.S * 64 * p.MT * p.NT * sizeof(f32x4) : 0);
    return p;
}

bool mid_reads(const void* scales, const void* mins) {
    return reinterpret_cast<uintptr_t>(scales) % 4 == 0 && reinterpret_cast<uintptr_t>(mins) % 4 == 0;
}

int mid_linear(const MidPlan& p, float* y, const float* x, long long x_ld, int M, int N, int K, const void* w, int w_type,
               const void* scales, const void* mins, const float* bias, const float* residual, int glu,
               void* workspace, hipStream_t stream) {
    char* ws = static_cast<char*>(workspace);
    uint16_t* ops = reinterpret_cast<uint16_t*>(ws);
    uint16_t* sums = reinterpret_cast<uint16_t*>(ws + p.sums);
    MidArgs a{};
    a.y = y; a.a = ops; a.sums = sums; a.w = w;
    a.scales = static_cast<const uint16_t*>(scales); a.mins = static_cast<const uint16_t*>(mins);
    a.bias = bias; a.res = residual; a.part = reinterpret_cast<f32x4*>(ws + p.part);
    a.M = M; a.N = N; a.K = K; a.S = p.S; a.SB = p.SB; a.WB = p.WB; a.MB = p.MB; a.G = p.G; a.glu = glu ? 1 : 0;
    using Split = void (*)(uint16_t*, uint16_t*, const float*, long long, int);
    using Fn = void (*)(MidArgs);
    Split split = nullptr;
    Fn rows = nullptr, fin = nullptr;
#define RK_MID(W, T, C)                                                                                        \
    if (w_type == W && p.MT == T && p.NT == C) {                                                               \
        split = split_operands<W, T>;                                                                          \
        rows = mid_rows<W, T, C>;                                                                              \
        fin = mid_finish<T, C>;                                                                                \
    }
#define RK_MIDS(T)                                                                                             \
    RK_MID(RK_W_INT4, T, 1) RK_MID(RK_W_INT4, T, 2) RK_MID(RK_W_INT4, T, 3)                                    \
    RK_MID(RK_W_INT8, T, 1) RK_MID(RK_W_INT8, T, 2) RK_MID(RK_W_INT8, T, 3)                                    \
    RK_MID(RK_W_BF16, T, 1) RK_MID(RK_W_BF16, T, 2)
    RK_MIDS(3) RK_MIDS(4) RK_MID(RK_W_INT4, 3, 4) RK_MID(RK_W_INT8, 3, 4)
#undef RK_MIDS
#undef RK_MID
    if (!rows) return fail(RK_ERR_ARG, "rk_linear_gemm: no kernel for %d x %d tiles", p.MT, p.NT);
    hipLaunchKernelGGL(split, dim3((unsigned)M), dim3(256), 0, stream, ops, sums, x, x_ld, K);
    if (int rc = check_launch("split_operands")) return rc;
    const size_t lds = (size_t)kWaves * 64 * p.MT * p.NT * sizeof(f32x4);
    if (int rc = allow_dynamic_lds((const void*)rows, lds)) return rc;
    const long long ids = ((long long)p.G * p.S + 7) / 8 * 8 * p.MB;
    if (ids >= (1ll << 31)) return fail(RK_ERR_ARG, "rk_linear_gemm: N %d too large", N);
    hipLaunchKernelGGL(rows, dim3((unsigned)ids), dim3(64 * kWaves), lds, stream, a);
    if (int rc = check_launch("mid_rows")) return rc;
    if (p.S == 1) return RK_OK;
    hipLaunchKernelGGL(fin, dim3((unsigned)(p.MB * p.G), (unsigned)((64 * p.MT * p.NT + 255) / 256)), dim3(256), 0, stream, a);
    return check_launch("mid_finish");
}

}  // namespace rk
