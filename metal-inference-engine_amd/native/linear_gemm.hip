// Linears of many rows (prefill tokens, decode batches past the row kernels' 32), gfx950.
//
// Semantics (reference): MetalBackend.linear / _qlinear for M > 32 rows (src/backend/metal.py:55-133), which expands
// the weight to fp32 and runs an fp32 GEMM: y [M, N] = x [M, K] @ dequant(W)^T (+ bias) (+ residual), fp32, W bf16 or
// block-quantized (src/quant.py:1-10, 45-56); and Backend.swiglu (src/backend/base.py:40-41) over a stacked
// [gate; up] weight.
//
// Design: the fp32 matrix rate of gfx950 is 1/16 of its 16-bit rate, so an fp32 product is worth three 16-bit ones, and
// three carry all its bits: operands are linear_operands.h's, three bf16 pieces of every activation and the weights, all
// exact (as in linear.hip, so a row is computed alike however many there are). Products accumulate in fp32. A
// quantization block is one MFMA's k-extent (32), so its scale multiplies the block's sums on the VALU.
//
// The product runs on LDS tiles of both operands. split_rows writes the pieces of x. bf16 weights are read as stored;
// INT8 / INT4 ones are expanded to bf16 rows, a slab at a time (slab_weights). An INT4 weight is s (q - 8) + (8 s + min):
// the codes enter as q - 8 (small partial sums), and 8 s + min, in its three pieces, as K / 8 more columns against the
// block's activation sum. Then gemm_rows (and with K-splits gemm_finish). Up to a few hundred rows linear_mid.hip reads
// quantized weights as stored instead.
//
// Measured, an MLP of 1777 rows, bf16 weights (12288 x 2048 with silu * up, then 2048 x 6144): 1188 us as an fp32 GEMM on
// the expanded weight, 362 on two fp16 pieces of x (23 bits in a range of 2^40 below the row's largest value), 377 so.
// What bounds gemm_rows: matrix-core issue and the fp32 joins beside it, and whole tiles.
#include "linear_operands.h"

#include <type_traits>

namespace rk {
namespace {

constexpr int kBK = 32;                            // k per step
constexpr int P = 3;                               // pieces of an activation
constexpr long long kSlabElems = 1ll << 25;        // quantized weights expanded at a time (64 MiB)
constexpr long long kPieceBytes = 192ll << 20;     // activation pieces made at a time
constexpr long long kPartBytes = 64ll << 20;       // partial sums of K-splits

// 16 bytes per lane from src into LDS at dst (wave-uniform) + 16 * lane
__device__ __forceinline__ void load_to_lds(const void* src, char* dst) {
    __builtin_amdgcn_global_load_lds(src, (__attribute__((address_space(3))) void*)dst, 16, 0, 0);
}

__device__ __forceinline__ void load4_to_lds(const void* src, char* dst) {   // the same, 4 bytes per lane
    __builtin_amdgcn_global_load_lds(src, (__attribute__((address_space(3))) void*)dst, 4, 0, 0);
}

// Rows of 32 bf16 (64 bytes) in LDS: the 16-byte unit u of row R sits at u ^ swizzle(R). A read of lane l: row l % 16,
// unit l / 16, is served 16 lanes at a time, rows 0-3 and 12-15 of one unit with rows 4-11 of the next, and these then
// lie on all 16 units of the 256-byte bank line.
__device__ __forceinline__ int swizzle(int R) { return (0x78 >> (2 * ((R >> 2) & 3))) & 3; }

// Operands of gemm_rows in memory: rows cut into steps of 32 values, x [step][piece][rows][32], an expanded weight slab
// [step][rows][32], so that a stage of a tile is one contiguous run per operand, in the LDS order.
// Rows past the matrix (up to whole tiles) are not written: their products are never stored.
__device__ __forceinline__ size_t unit_at(size_t slice, int rows, int R, int u) {
    return (slice * rows + R) * kBK + 8 * (u ^ swizzle(R));
}

// One workgroup per row m of x: the row's pieces. With SUMS, columns K + 4 b .. + 2 are block b's sum, and zeros to the
// end of the last step.
template <bool SUMS>
__global__ __launch_bounds__(256) void split_rows(uint16_t* a, const float* x, long long x_ld, int Mp, int K, int steps) {
    const int m = blockIdx.x, tid = threadIdx.x;
    const float* xr = x + (size_t)m * x_ld;
    auto put_sum = [&](int b, const Split3& p) {   // eight blocks to a step
        const uint32_t v[P] = {p.hi, p.mid, p.lo};
#pragma unroll
        for (int q = 0; q < P; ++q)
            *reinterpret_cast<u32x2*>(a + unit_at(P * (size_t)(K / kBK + (b >> 3)) + q, Mp, m, (b & 7) >> 1) + 4 * (b & 1)) =
                (u32x2){pack_hi2(v[q], v[q]), v[q] >> 16};
    };
    for (int c = tid; c < K / 8; c += 256) {
        const f32x4 v0 = *reinterpret_cast<const f32x4*>(xr + 8 * c), v1 = *reinterpret_cast<const f32x4*>(xr + 8 * c + 4);
        const float v[8] = {v0[0], v0[1], v0[2], v0[3], v1[0], v1[1], v1[2], v1[3]};
        u32x4 pc[P];
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            const Split3 s0 = split3_any(v[2 * e]), s1 = split3_any(v[2 * e + 1]);
            pc[0][e] = pack_hi2(s0.hi, s1.hi);
            pc[1][e] = pack_hi2(s0.mid, s1.mid);
            pc[2][e] = pack_hi2(s0.lo, s1.lo);
        }
#pragma unroll
        for (int q = 0; q < P; ++q) *reinterpret_cast<u32x4*>(a + unit_at(P * (size_t)(c >> 2) + q, Mp, m, c & 3)) = pc[q];
        if constexpr (SUMS) {                      // the four threads of a block are neighbours in one wave
            float sum = 0.0f;
#pragma unroll
            for (int e = 0; e < 8; ++e) sum += v[e];
            sum += dpp_f32<0xb1>(sum);             // lane ^ 1
            sum += dpp_f32<0x4e>(sum);             // lane ^ 2
            if ((c & 3) == 0) put_sum(c >> 2, split3_any(sum));
        }
    }
    if constexpr (SUMS)
        for (int b = K / kBK + tid; b < 8 * (steps - K / kBK); b += 256) put_sum(b, {0u, 0u, 0u});
}

struct SlabArgs {
    uint16_t* out;                 // [steps][Np][32] bf16
    float* sc;                     // [steps][Np] scales
    const void* w;
    const uint16_t* scales;
    const uint16_t* mins;
    int Np, row0, K, steps;        // padded slab rows; the slab's first weight row (glu: its first gate row)
    int F;                         // glu: rows of each half; 0: plain
};

// the weight row behind tile row j from row0 on: row0 + j, or with glu (F rows in each half) sixteen gate rows, then the
// sixteen up rows of the same outputs, in turn, so that an output's gate and up sums meet in one lane (rows past F, in
// the last pair of sixteens, repeat row F - 1: their outputs are not stored)
__device__ __forceinline__ size_t weight_row(int row0, int F, int j) {
    if (!F) return (size_t)(row0 + j);
    const int f = min(row0 + 16 * (j >> 5) + (j & 15), F - 1);
    return (size_t)((j & 16) ? F + f : f);
}

// One workgroup per slab row: the row's codes and scales; INT4: codes minus 8, then the pieces of 8 s + min.
template <int WT>
__global__ __launch_bounds__(256) void slab_weights(SlabArgs a) {
    const int j = blockIdx.x, tid = threadIdx.x;
    const size_t n = weight_row(a.row0, a.F, j);
    const int nblk = a.K / kQB;
    for (int c = tid; c < a.K / 8; c += 256) {
        u32x4 o;
        if constexpr (WT == RK_W_INT8) {
            const u32x2 q = *reinterpret_cast<const u32x2*>(static_cast<const int8_t*>(a.w) + n * a.K + 8 * c);
            o = int8_bf16(q[0], q[1]);
        } else {
            const uint32_t q = *reinterpret_cast<const uint32_t*>(static_cast<const uint8_t*>(a.w) + n * (a.K / 2) + 4 * c);
#pragma unroll
            for (int e = 0; e < 4; ++e)
                o[e] = pack_hi2(__float_as_uint((float)__builtin_amdgcn_ubfe(q, 8 * e, 4) - 8.0f),
                                __float_as_uint((float)__builtin_amdgcn_ubfe(q, 8 * e + 4, 4) - 8.0f));
        }
        *reinterpret_cast<u32x4*>(a.out + unit_at(c >> 2, a.Np, j, c & 3)) = o;
    }
    const uint16_t* s = a.scales + n * nblk;
    for (int t = tid; t < a.steps; t += 256) a.sc[(size_t)t * a.Np + j] = t < nblk ? half_to_f32(s[t]) : 1.0f;
    if constexpr (WT == RK_W_INT4) {
        const uint16_t* mn = a.mins + n * nblk;
        for (int b = tid; b < 8 * (a.steps - nblk); b += 256) {
            const Split3 p = split3(b < nblk ? fmaf(8.0f, half_to_f32(s[b]), half_to_f32(mn[b])) : 0.0f);
            *reinterpret_cast<u32x2*>(a.out + unit_at(nblk + (b >> 3), a.Np, j, (b & 7) >> 1) + 4 * (b & 1)) =
                (u32x2){pack_hi2(p.hi, p.mid), p.lo >> 16};
        }
    }
}

struct GemmArgs {
    float* y;
    const uint16_t* a;             // [steps][3][Mp][32]
    const uint16_t* w;             // SCALED: [steps][Np][32], the slab; else [N][K] as stored
    const float* sc;               // [steps][Np]
    const float* bias;             // [columns of y] or null
    const float* res;              // as y, or null
    long long y_ld;
    int M, N, Mp, Np, steps;       // N: weight rows of this slab
    int F;                         // bf16 glu: rows of each half; 0: plain
    int col0, cols;                // first column of y this slab gives; columns of y
    int tm, tn;                    // tiles
    int S;                         // K-splits
    float* part;                   // S > 1: [S][M][Np] sums, to be finished by gemm_finish
};

// weight columns 32 q + r and 32 q + 16 + r (v, u) of row m: bias and residual or silu * up
template <bool GLU>
__device__ __forceinline__ void gemm_store(const GemmArgs& g, int m, int n, float v, float u) {
    if constexpr (GLU) {
        const int c = g.col0 + ((n & ~31) >> 1) + (n & 15);
        if (c < g.cols && n < g.N) g.y[(size_t)m * g.y_ld + c] = silu_times(v, u);
    } else {
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            if (n + 16 * h >= g.N) continue;
            const int c = g.col0 + n + 16 * h;
            float o = h ? u : v;
            if (g.bias) o = __fadd_rn(o, g.bias[c]);
            if (g.res) o = __fadd_rn(o, g.res[(size_t)m * g.y_ld + c]);
            g.y[(size_t)m * g.y_ld + c] = o;
        }
    }
}

// Workgroup of WM x WN waves, each a 16 TI x 64 tile of y. A stage is one step of 32: 3 BM piece rows and BN
// weight rows of 64 bytes (and each wave's 64 scales), straight from memory into LDS by global_load_lds, 1 KB per
// instruction, kStages buffers in turn. Per stage and wave 16 operand reads feed 48 MFMAs (TI = 4), each read one group
// of sixteen rows ahead, across the stages' barriers too. The loop has no other memory reads, and a wave's loads complete
// in order, so waiting for all but the newest (kStages - 3) x loads-per-stage leaves this stage and the next in LDS.
template <int WM, int WN, int TI, bool SCALED>
struct Tile {
    static constexpr int NW = WM * WN, BM = 16 * TI * WM, BN = 64 * WN, ROWS = P * BM + BN, NI = ROWS / 16 / NW;
    static constexpr int kLoads = NI + (SCALED ? 1 : 0);
    static constexpr int kBytes = ROWS * 2 * kBK + (SCALED ? 256 * NW : 0);
    static constexpr int kStages = 160 * 1024 / kBytes < 6 ? 160 * 1024 / kBytes : 6;
    static_assert(NI * 16 * NW == ROWS, "whole load instructions");
    static_assert(kStages * kBytes <= 160 * 1024, "LDS");
};

template <int WM, int WN, int TI, bool SCALED, bool GLU>
__global__ __launch_bounds__(64 * WM * WN) void gemm_rows(GemmArgs g) {
    using TL = Tile<WM, WN, TI, SCALED>;
    constexpr int BM = TL::BM, BN = TL::BN, NI = TL::NI, ST = TL::kStages;
    extern __shared__ __attribute__((aligned(16))) char smem[];
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int r = lane & 15, grp = lane >> 4;
    const int wm = wave / WN, wn = wave % WN;

    // tile order: workgroups go to the 8 XCDs in turn, so XCD x takes a contiguous run of tiles, walked in groups of
    // 8 row tiles by all column tiles: the run's weight rows and pieces stay in the XCD's L2
    const int T = g.tm * g.tn, per = T / 8, rem = T % 8, xcd = blockIdx.x % 8;
    const int id = xcd * per + min(xcd, rem) + blockIdx.x / 8;
    const int group = 8 * g.tn, gi = id / group, first = 8 * gi, height = min(8, g.tm - first);
    const int m0 = BM * (first + (id % group) % height), n0 = BN * ((id % group) / height);

    // this split's steps
    const int s0 = (int)((long long)g.steps * blockIdx.y / g.S), S = (int)((long long)g.steps * (blockIdx.y + 1) / g.S) - s0;
    // load instruction i of this wave: stage rows 16 (NI wave + i) .. + 15 (hi, mid, lo piece rows, weight rows);
    // lane l brings unit (l % 4) ^ swizzle of row l / 4 of the sixteen (operands laid out in the LDS order: 16 l on)
    const char* src[NI];
    size_t hop[NI];
#pragma unroll
    for (int i = 0; i < NI; ++i) {
        const int R = 16 * (NI * wave + i);
        const bool pc = R < P * BM;
        if (pc || SCALED) {
            const size_t row = pc ? (size_t)(R / BM) * g.Mp + m0 + R % BM : (size_t)(n0 + R - P * BM);
            src[i] = reinterpret_cast<const char*>((pc ? g.a : g.w) + row * kBK) + 16 * lane;
            hop[i] = (size_t)(pc ? P * g.Mp : g.Np) * kBK * 2;
        } else {
            const int j = n0 + R - P * BM + (lane >> 2);
            const size_t row = weight_row(g.col0, g.F, min(j, g.N - 1));
            src[i] = reinterpret_cast<const char*>(g.w + row * (size_t)(g.steps * kBK)) + 16 * ((lane & 3) ^ swizzle(lane >> 2));
            hop[i] = kBK * 2;
        }
        src[i] += s0 * hop[i];
    }
    const char* scp = reinterpret_cast<const char*>(g.sc + n0 + 64 * wn) + (size_t)s0 * g.Np * 4;
    int ahead = 0;                                 // the next stage to request; past the last, the last again
    auto request = [&](int buf) {
        char* dst = smem + buf * TL::kBytes;
#pragma unroll
        for (int i = 0; i < NI; ++i) load_to_lds(src[i], dst + 1024 * (NI * wave + i));
        if constexpr (SCALED) load4_to_lds(scp + 4 * lane, dst + TL::ROWS * 2 * kBK + 256 * wave);
        if (++ahead < S) {                         // uniform
#pragma unroll
            for (int i = 0; i < NI; ++i) src[i] += hop[i];
            if constexpr (SCALED) scp += (size_t)g.Np * 4;
        }
    };
#pragma unroll
    for (int b = 0; b < ST - 1; ++b) request(b);

    // operand reads: lane (r, grp) takes unit grp of row R0 + r; R0 is a multiple of 16, so the unit's place is the
    // lane's alone
    const int at = 64 * r + 16 * (grp ^ swizzle(r));
    const int at_a = at + 64 * 16 * TI * wm, at_b = at + 64 * (P * BM + 64 * wn);
    const int at_s = TL::ROWS * 2 * kBK + 256 * wave + 4 * r;
    auto rd = [&](const char* p) { return *reinterpret_cast<const u32x4*>(p); };
    // the sums in the making: of one group of sixteen rows and the one before (SCALED), or of every group (two stages)
    constexpr int ND = SCALED ? 2 : TI;
    f32x4 acc[TI][4], d[ND][4];
    u32x4 b[4], bn[4], x[2][P];
    float f[4], fn[4], fd[4];                      // scales: of this stage, of the next, of d[1]'s stage
#pragma unroll
    for (int t = 0; t < 4; ++t) {
        d[ND - 1][t] = (f32x4){0.f, 0.f, 0.f, 0.f};
        f[t] = fn[t] = fd[t] = 0.0f;
#pragma unroll
        for (int i = 0; i < TI; ++i) acc[i][t] = (f32x4){0.f, 0.f, 0.f, 0.f};
    }
    // a stage's sums (a pair of stages' where no scales stand between them) start from zero and join the running ones by
    // an fp32 addition (or fma): a third of the error of MFMAs on the running sums
    auto join = [&](f32x4 (&to)[4], const f32x4 (&from)[4], const float (&by)[4]) {
#pragma unroll
        for (int t = 0; t < 4; ++t)
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                if constexpr (SCALED) to[t][e] = fmaf(by[t], from[t][e], to[t][e]);
                else to[t][e] += from[t][e];
            }
    };
    auto landed = [&] {
        asm volatile("s_waitcnt vmcnt(%0)\n\ts_barrier" ::"n"((ST - 3) * TL::kLoads) : "memory");
    };
    landed();
#pragma unroll
    for (int t = 0; t < 4; ++t) {
        b[t] = rd(smem + at_b + 1024 * t);
        if constexpr (SCALED) f[t] = *reinterpret_cast<const float*>(smem + at_s + 64 * t);
    }
#pragma unroll
    for (int q = 0; q < P; ++q) x[0][q] = rd(smem + at_a + 64 * BM * q);

    int buf = 0;
    auto stage = [&](int s, auto odd_c) __attribute__((always_inline)) {
        constexpr bool kOdd = decltype(odd_c)::value;           // the second stage of a pair: goes on from the first
        // behind this barrier stages s and s + 1 are in LDS, and stage s - 1, whose buffer the request fills, is done
        // with (its last operands were taken before it)
        if (s) landed();
        request(buf == 0 ? ST - 1 : buf - 1);
        const char* cur = smem + buf * TL::kBytes;
        buf = buf == ST - 1 ? 0 : buf + 1;
        const char* nxt = smem + buf * TL::kBytes;
        // rows 16 i: their MFMAs, while the operands of the next sixteen (at the end the next stage's) are read and
        // the sums of the sixteen before are joined
#pragma unroll
        for (int i = 0; i < TI; ++i) {
            const int c = i & 1, o = c ^ 1, di = SCALED ? c : i;
#pragma unroll
            for (int q = 0; q < P; ++q) x[o][q] = rd((i < TI - 1 ? cur + 1024 * (i + 1) : nxt) + at_a + 64 * BM * q);
            if (i >= TI - 2) {
#pragma unroll
                for (int t = 2 * (i - TI + 2); t < 2 * (i - TI + 3); ++t) {
                    bn[t] = rd(nxt + at_b + 1024 * t);
                    if constexpr (SCALED) fn[t] = *reinterpret_cast<const float*>(nxt + at_s + 64 * t);
                }
            }
            // the last group of the stage (pair) before, whose sums this one's overwrite
            if (i == 0 && (SCALED || !kOdd)) join(acc[TI - 1], d[ND - 1], fd);
#pragma unroll
            for (int t = 0; t < 4; ++t)
                d[di][t] = mfma16x16x32(x[c][P - 1], b[t], kOdd ? d[di][t] : (f32x4){0.f, 0.f, 0.f, 0.f});
#pragma unroll
            for (int q = P - 2; q >= 0; --q)
#pragma unroll
                for (int t = 0; t < 4; ++t) d[di][t] = mfma16x16x32(x[c][q], b[t], d[di][t]);
            if (i && (SCALED || kOdd)) join(acc[i - 1], d[SCALED ? o : i - 1], f);
            if (i < TI - 2) __builtin_amdgcn_sched_group_barrier(0x100, P, 0);
            else __builtin_amdgcn_sched_group_barrier(0x100, P + (SCALED ? 4 : 2), 0);
#pragma unroll
            for (int q = 0; q < 4 * P; ++q) {
                __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
                __builtin_amdgcn_sched_group_barrier(0x002, 2, 0);
            }
            __builtin_amdgcn_sched_barrier(0);
        }
#pragma unroll
        for (int t = 0; t < 4; ++t) {
            b[t] = bn[t];
            if constexpr (SCALED) {
                fd[t] = f[t];
                f[t] = fn[t];
            }
        }
    };
    int s = 0;
    if constexpr (SCALED) {
        for (; s < S; ++s) stage(s, std::false_type{});
    } else {
        for (; s + 1 < S; s += 2) {
            stage(s, std::false_type{});
            stage(s + 1, std::true_type{});
        }
        if (s < S) {                               // an odd last stage: no group of it is joined yet
            stage(s, std::false_type{});
#pragma unroll
            for (int i = 0; i < TI - 1; ++i) join(acc[i], d[i], fd);
        }
    }
    join(acc[TI - 1], d[ND - 1], fd);
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");   // the requests past the last stage

    // lane (r, grp) holds rows 4 grp + e, column r of each 16 x 16 tile
#pragma unroll
    for (int i = 0; i < TI; ++i) {
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            const int m = m0 + 16 * TI * wm + 16 * i + 4 * grp + e, n = n0 + 64 * wn + r;
            if (m >= g.M) continue;
            if (g.S > 1) {                         // uniform; the part rows hold whole tiles
#pragma unroll
                for (int t = 0; t < 4; ++t) g.part[((size_t)blockIdx.y * g.M + m) * g.Np + n + 16 * t] = acc[i][t][e];
            } else {
                gemm_store<GLU>(g, m, n, acc[i][0][e], acc[i][1][e]);
                gemm_store<GLU>(g, m, n + 32, acc[i][2][e], acc[i][3][e]);
            }
        }
    }
}

// The splits' sums of row blockIdx.y, in order; a thread per pair of columns 16 apart.
template <bool GLU>
__global__ __launch_bounds__(256) void gemm_finish(GemmArgs g) {
    const int q = 256 * blockIdx.x + threadIdx.x, m = blockIdx.y;
    const int n = 32 * (q >> 4) + (q & 15);
    if (n >= g.N) return;
    const float* p = g.part + (size_t)m * g.Np + n;
    float v = p[0], u = p[16];                     // Np is a multiple of 32
    for (int s = 1; s < g.S; ++s) {
        p += (size_t)g.M * g.Np;
        v += p[0];
        u += p[16];
    }
    gemm_store<GLU>(g, m, n, v, u);
}

struct Layout {
    int Mc, Mp, Np, steps, slab;   // rows of x at a time, and in whole tiles; slab: output columns at a time; Np: its
                                   // weight rows, in whole tiles
    int form, S;                   // gemm_rows' tile (kTiles); K-splits
    double us;                     // the estimated time
    size_t slab_w, slab_sc, part, total;
};

size_t up256(size_t n) { return (n + 255) / 256 * 256; }

// rows of W behind `cols` output columns (glu: whole pairs of sixteens)
int slab_rows(int cols, bool glu) { return glu ? (cols + 15) / 16 * 32 : cols; }

// gemm_rows' tiles, and what its time is made of, in us: a round of one workgroup per CU costs `start`, and for each of
// its steps `step` and up to `full` more when every CU has one ([1]: with scales). Fitted, with the constants of layout(),
// to 168 sizes (seven weights of 1024 x 3584 to 12288 x 2048, 64 to 4096 rows, bf16, INT8, INT4) x up to 10 of these
// forms, 12 to 1200 us: 4.8 % of root mean square error; the form it names is the fastest measured, or within 4 % of it,
// at all but 9 of them (the worst 13 %).
constexpr int kTiles[3][2] = {{128, 256}, {128, 128}, {64, 128}};
struct RoundCost {
    double start, step, full;
};
constexpr RoundCost kRound[2][3] = {{{2.7, 0.88, 0.28}, {2.5, 0.50, 0.17}, {2.2, 0.36, 0.05}},
                                    {{0.6, 1.10, 0.24}, {1.4, 0.69, 0.12}, {1.6, 0.47, 0.03}}};

Layout layout(int M, int N, int K, int w_type, bool glu) {
    Layout l;
    l.steps = K / kBK + (w_type == RK_W_INT4 ? (K / kQB + 7) / 8 : 0);
    // rows in pieces of about the same size whose operands fit kPieceBytes
    const long long row_bytes = (long long)l.steps * P * kBK * 2;
    long long most = kPieceBytes / row_bytes / 128 * 128;
    if (most < 128) most = 128;
    const long long runs = (M + most - 1) / most;
    l.Mc = runs == 1 ? M : (int)((M + 128 * runs - 1) / (128 * runs) * 128);
    l.Mp = (l.Mc + 127) / 128 * 128;
    const int cols = glu ? N / 2 : N;
    l.slab = cols;
    if (w_type != RK_W_BF16) {
        long long s = kSlabElems / (l.steps * kBK) / (glu ? 2 : 1) / 256 * 256;
        if (s < 256) s = 256;
        if (s < cols) l.slab = (int)s;
    }
    const size_t rows = (size_t)slab_rows(l.slab, glu);
    l.Np = (int)up256(rows);
    l.slab_w = (size_t)l.Mp * row_bytes;
    l.slab_sc = l.slab_w + (w_type == RK_W_BF16 ? 0 : (size_t)l.steps * l.Np * kBK * 2);
    l.part = l.slab_sc + (w_type == RK_W_BF16 ? 0 : (size_t)l.steps * l.Np * 4);
    // the tile and the K-splits of the least estimated time
    int cus = device_cus();
    if (cus <= 0) cus = 256;
    const bool quant = w_type != RK_W_BF16;
    l.us = 0.0;
    for (int f = 0; f < 3; ++f) {
        const long long t = (long long)((l.Mc + kTiles[f][0] - 1) / kTiles[f][0]) * (((long long)rows + kTiles[f][1] - 1) / kTiles[f][1]);
        const RoundCost& c = kRound[quant][f];
        for (int sp = 1; sp <= 16; ++sp) {
            // splits of at least 8 steps, for at most two rounds of workgroups, their sums within kPartBytes
            if (sp > 1 && (l.steps < 8 * sp || t * sp > 2 * cus || (long long)sp * l.Mc * l.Np * 4 > kPartBytes)) break;
            const long long rounds = (t * sp + cus - 1) / cus;
            const double full = (double)(t * sp) / (double)(rounds * cus);
            double us = (double)rounds * (c.start + (c.step + c.full * full) * ((l.steps + sp - 1) / sp));
            if (sp > 1) us += 1.5 + 1.05e-6 * sp * l.Mc * (double)rows;       // gemm_finish
            if (l.us == 0.0 || us < l.us) {
                l.us = us;
                l.form = f;
                l.S = sp;
            }
        }
    }
    const double slabs = (cols + l.slab - 1) / l.slab;
    if (quant) l.us += 4.8 + 0.75e-6 * (double)rows * K;                     // slab_weights
    l.us = (double)runs * (slabs * l.us + 6.6 + 1.5e-6 * (double)l.Mc * K);  // split_rows
    l.total = l.part + (l.S > 1 ? (size_t)l.S * l.Mc * l.Np * 4 : 0);
    return l;
}

// Which form takes a call, and the workspace for it (scales or mins at an odd address send a call to the tiles)
struct Choice {
    Layout l;
    MidPlan p;
    bool mid;
    size_t total;
};

Choice choose(int M, int N, int K, int w_type, int glu) {
    Choice c;
    c.l = layout(M, N, K, w_type, glu != 0);
    c.p = mid_plan(M, N, K, w_type, glu);
    c.mid = c.p.us > 0.0 && c.p.us < c.l.us;
    c.total = c.mid && c.p.total > c.l.total ? c.p.total : c.l.total;
    return c;
}

template <int WM, int WN, int TI>
int launch_gemm(const GemmArgs& in, bool scaled, bool glu, hipStream_t s) {
    GemmArgs g = in;
    constexpr int BM = 16 * TI * WM, BN = 64 * WN;
    const size_t lds = scaled ? Tile<WM, WN, TI, true>::kStages * Tile<WM, WN, TI, true>::kBytes
                              : Tile<WM, WN, TI, false>::kStages * Tile<WM, WN, TI, false>::kBytes;
    g.tm = (g.M + BM - 1) / BM;
    g.tn = (g.N + BN - 1) / BN;
    const auto fn = scaled ? (glu ? gemm_rows<WM, WN, TI, true, true> : gemm_rows<WM, WN, TI, true, false>)
                           : (glu ? gemm_rows<WM, WN, TI, false, true> : gemm_rows<WM, WN, TI, false, false>);
    if (int rc = allow_dynamic_lds((const void*)fn, lds)) return rc;
    if ((long long)g.tm * g.tn >= (1ll << 31)) return fail(RK_ERR_ARG, "rk_linear_gemm: M %d too large", g.M);
    hipLaunchKernelGGL(fn, dim3((unsigned)(g.tm * g.tn), (unsigned)g.S), dim3(64 * WM * WN), lds, s, g);
    if (int rc = check_launch("gemm_rows")) return rc;
    if (g.S == 1) return RK_OK;
    const auto fin = glu ? gemm_finish<true> : gemm_finish<false>;
    hipLaunchKernelGGL(fin, dim3((unsigned)((g.Np / 2 + 255) / 256), (unsigned)g.M), dim3(256), 0, s, g);
    return check_launch("gemm_finish");
}

}  // namespace
}  // namespace rk

using namespace rk;

extern "C" {

size_t rk_linear_gemm_workspace_bytes(int M, int N, int K, int w_type, int glu) {
    if (M < 1 || N < 1 || K < kQB || K % kQB) return 0;
    return choose(M, N, K, w_type, glu).total;
}

int rk_linear_gemm_plan(int M, int N, int K, int w_type, int glu, int* plan) {
    if (M < 1 || N < 1 || K < kQB || K % kQB || (glu && N % 2) || !plan)
        return fail(RK_ERR_ARG, "rk_linear_gemm_plan: M %d, N %d, K %d", M, N, K);
    const Choice c = choose(M, N, K, w_type, glu);
    const int cols = glu ? N / 2 : N;
    plan[0] = c.mid ? 0 : 1 + c.l.form;
    plan[1] = c.mid ? c.p.S : c.l.S;
    plan[2] = c.mid ? 1 : (cols + c.l.slab - 1) / c.l.slab;
    plan[3] = c.mid ? 1 : (M + c.l.Mc - 1) / c.l.Mc;
    return RK_OK;
}

int rk_linear_gemm(float* y, const float* x, long long x_ld, int M, int N, int K, const void* w, int w_type,
                   const void* scales, const void* mins, const float* bias, const float* residual, int glu,
                   void* workspace, size_t workspace_bytes, void* stream) {
    if (M == 0 || N == 0) return RK_OK;
    const bool quant = w_type == RK_W_INT8 || w_type == RK_W_INT4;
    if (!y || !x || !w || (quant && !scales) || (w_type == RK_W_INT4 && !mins))
        return fail(RK_ERR_ARG, "rk_linear_gemm: null pointer");
    if (w_type != RK_W_BF16 && !quant) return fail(RK_ERR_UNSUPPORTED, "rk_linear_gemm: weight type %d", w_type);
    if (M < 0 || N < 0 || K < kQB || K % kQB || K > (1 << 24) || (glu && N % 2))
        return fail(RK_ERR_ARG, "rk_linear_gemm: M %d, N %d, K %d (a multiple of %d)", M, N, K, kQB);
    if (glu && (bias || residual)) return fail(RK_ERR_ARG, "rk_linear_gemm: no bias or residual with glu");
    if (reinterpret_cast<uintptr_t>(x) % 16 || reinterpret_cast<uintptr_t>(w) % 16 || x_ld < K || x_ld % 4)
        return fail(RK_ERR_ARG, "rk_linear_gemm: x and w must be 16-byte aligned, x rows at a stride >= K of 4n");
    const Choice c = choose(M, N, K, w_type, glu);
    if (!workspace || workspace_bytes < c.total)
        return fail(RK_ERR_WORKSPACE, "rk_linear_gemm: workspace %zu bytes (need %zu)", workspace_bytes, c.total);
    if (c.mid && mid_reads(scales, mins))
        return mid_linear(c.p, y, x, x_ld, M, N, K, w, w_type, scales, mins, bias, residual, glu, workspace,
                          static_cast<hipStream_t>(stream));
    const Layout& l = c.l;
    char* ws = static_cast<char*>(workspace);
    hipStream_t st = static_cast<hipStream_t>(stream);
    uint16_t* pieces = reinterpret_cast<uint16_t*>(ws);
    const auto split = w_type == RK_W_INT4 ? split_rows<true> : split_rows<false>;
    const int cols = glu ? N / 2 : N;
    for (int m0 = 0; m0 < M; m0 += l.Mc) {
        const int rows_x = l.Mc < M - m0 ? l.Mc : M - m0;
        hipLaunchKernelGGL(split, dim3((unsigned)rows_x), dim3(256), 0, st, pieces, x + (size_t)m0 * x_ld, x_ld, l.Mp, K,
                           l.steps);
        if (int rc = check_launch("split_rows")) return rc;
        for (int c0 = 0; c0 < cols; c0 += l.slab) {
            const int nc = l.slab < cols - c0 ? l.slab : cols - c0;
            const int rows = slab_rows(nc, glu != 0);
            GemmArgs g{};
            g.w = static_cast<const uint16_t*>(w);
            g.F = glu ? cols : 0;
            if (quant) {
                SlabArgs sa{};
                sa.out = reinterpret_cast<uint16_t*>(ws + l.slab_w);
                sa.sc = reinterpret_cast<float*>(ws + l.slab_sc);
                sa.w = w; sa.scales = static_cast<const uint16_t*>(scales); sa.mins = static_cast<const uint16_t*>(mins);
                sa.Np = l.Np; sa.row0 = c0; sa.K = K; sa.steps = l.steps; sa.F = g.F;
                const auto expand = w_type == RK_W_INT8 ? slab_weights<RK_W_INT8> : slab_weights<RK_W_INT4>;
                hipLaunchKernelGGL(expand, dim3((unsigned)rows), dim3(256), 0, st, sa);
                if (int rc = check_launch("slab_weights")) return rc;
                g.w = sa.out; g.sc = sa.sc;
            }
            g.y = y + (size_t)m0 * cols; g.a = pieces; g.bias = bias; g.res = residual ? residual + (size_t)m0 * cols : nullptr;
            g.y_ld = cols; g.M = rows_x; g.N = rows; g.Mp = l.Mp; g.Np = l.Np; g.steps = l.steps; g.col0 = c0; g.cols = cols;
            g.S = l.S;
            g.part = reinterpret_cast<float*>(ws + l.part);
            int rc;
            if (l.form == 0) rc = launch_gemm<2, 4, 4>(g, quant, glu != 0, st);
            else if (l.form == 1) rc = launch_gemm<4, 2, 2>(g, quant, glu != 0, st);
            else rc = launch_gemm<2, 2, 2>(g, quant, glu != 0, st);
            if (rc) return rc;
        }
    }
    return RK_OK;
}

}  // extern "C"
