// mvh_gemm_f32.hip -- batched fp32-activation products on the f32 matrix pipe.
//
// The reference's fp32 dots are fma chains in a fixed order.  On gfx950
// v_mfma_f32_16x16x4_f32 is such a chain: each of its 16 x 16 results is
//   fma(A[3], B[3], fma(A[2], B[2], fma(A[1], B[1], fma(A[0], B[0], C))))
// with every fma rounded to nearest even and subnormals kept (checked bit for
// bit against sequential fmaf over 50 million results: normal, widely scaled,
// subnormal and arbitrary finite operands).  A lane of the operand holds row
// (or token) l % 16 of k-slot l / 16, so giving slot m the elements 8m .. 8m+7
// of a 32-element block makes eight MFMAs, one per e = 0..7, exactly the
// reference's eight lane accumulators t_e over elements e, e+8, e+16, e+24 of
// the block.  Both numerics of the batched path are built on that:
//   batch_chain_kernel  q4_row_batch4_fp32 / q8_row_batch4_fp32
//       (src/gguf_kernels.cpp:191-216): t_e runs over all blocks without
//       reset, term = fma(float(q)*d, x, t_e) with float(q)*d rounded first,
//       result t0+t1+..+t7;
//   batch_blocksum_kernel  dot_q4_0_fp32 / dot_q8_0_fp32 (:93-120): per block
//       t_e from zero, s = 0+t0+..+t7, then sum = fma(d, s, sum) over the blocks.
#include "mvh_kernels.hpp"
#define MVH_STAGE_QUAL __device__ __forceinline__
#include "mvh_stage.h"

#include <cstdlib>
#include <type_traits>

namespace mvh {
namespace {

typedef float v4f __attribute__((ext_vector_type(4)));

// Bytes of a block: a 2-byte scale, then the quants.
template <uint32_t TYPE>
struct Fmt;
template <>
struct Fmt<kQ4_0> {
    static constexpr int kB = 18;
};
template <>
struct Fmt<kQ8_0> {
    static constexpr int kB = 34;
};

// The four weights of one operand dword, times the block's scale.  Q4_0 (v: four
// codes q, one per byte's low nibble, bit 3 flipped, so a nibble is q - 8 in
// two's complement): v_cvt_off_f32_i4 gives (q - 8) / 16, and dq = 16 d makes
// the product float(q - 8) * d with the reference's one rounding (both factors
// are scaled by powers of two).  Q8_0: float(q) * d.
template <uint32_t TYPE, int NE>
__device__ __forceinline__ void weights(uint32_t v, float dq, float (&a)[NE]) {
#pragma unroll
    for (int i = 0; i < NE; ++i) {
        if constexpr (TYPE == kQ4_0) a[i] = __builtin_amdgcn_cvt_off_f32_i4(static_cast<int>(v >> (8 * i))) * dq;
        else a[i] = static_cast<float>(static_cast<int>(static_cast<int8_t>(v >> (8 * i)))) * dq;
    }
}

constexpr int kUnitBlocks = 8;
constexpr int kT = 256;  // threads: four waves

// base + off with a uniform base: one load with the base in SGPRs.
template <typename T>
__device__ __forceinline__ T ld_at(const void* base, uint32_t off) {
    typedef uint32_t V __attribute__((ext_vector_type(sizeof(T) >= 4 ? sizeof(T) / 4 : 1)));
    typedef const __attribute__((address_space(1))) uint8_t* P;
    const P p = (P)(reinterpret_cast<uintptr_t>(base)) + off;
    if constexpr (sizeof(T) == 2) return *(const __attribute__((address_space(1))) T*)p;
    else return __builtin_bit_cast(T, *(const __attribute__((address_space(1))) V*)p);
}

// Bytes of blocks [c*8, c*8+8) of 16*R rows into registers, and from there to
// an LDS copy of pitch kUB bytes per row.  ALIGNED (K % 256 == 0: a row's unit
// starts 16-byte aligned): 16-byte pieces.  Otherwise 2-byte pieces, those past
// the row's last block read from its start (mvh_stage.h).
template <uint32_t TYPE, int R, bool ALIGNED>
struct WStage {
    static constexpr int kUB = kUnitBlocks * Fmt<TYPE>::kB;
    static constexpr int kRows = 16 * R;
    static constexpr int kBytes = kRows * kUB + 16;  // + a spare piece for stores without a use
    static constexpr int kP = kUB / (ALIGNED ? 16 : 2);
    static constexpr int kN = (kRows * kP + kT - 1) / kT;
    typedef std::conditional_t<ALIGNED, uint4, uint16_t> Piece;
    const uint8_t* base;       // the tile's first row (uniform)
    MvhStagePiece src[kN];
    int dst[kN];
    __device__ __forceinline__ void init(const uint8_t* W, int row0, int N, int row_bytes) {
        base = W + static_cast<size_t>(row0) * row_bytes;
#pragma unroll
        for (int i = 0; i < kN; ++i) {
            const int p = static_cast<int>(threadIdx.x) + kT * i;
            src[i] = mvh_stage_piece(p, kRows * kP, kP, sizeof(Piece), N - row0, row_bytes);
            dst[i] = p < kRows * kP ? (p / kP) * kUB + src[i].off : kRows * kUB;
        }
    }
    __device__ __forceinline__ void load(int i, int c, int row_bytes, Piece (&reg)[kN]) const {
        const int at = c * kUB;
        if constexpr (ALIGNED) reg[i] = ld_at<uint4>(base + at, src[i].src);
        else reg[i] = ld_at<uint16_t>(base, mvh_stage_at(src[i], at, row_bytes));
    }
    __device__ __forceinline__ void store(int i, uint8_t* s, const Piece (&reg)[kN]) const {
        *reinterpret_cast<Piece*>(s + dst[i]) = reg[i];
    }
};

// ---- chains over all blocks (default batched numerics) -------------------------
//
// A workgroup of four waves owns 16*R*RW weight rows x 16*TG tokens.  The eight
// accumulators of an output are independent until the last sum, so they are
// split too: wave w owns E consecutive ones (part w % (8/E)) of 16*R rows (set
// w / (8/E)), and the parts meet through LDS at the end.  Per 8-block unit the
// raw weight bytes and the activations go through double-buffered LDS copies,
// fetched D units ahead into registers; the activations lie in lane order
// ([block][part][token group][lane][E]), so an operand read is one contiguous
// 8- or 16-byte piece per lane, and a weight operand is E adjacent quant bytes
// and the row's scale.
// What bounds it: the f32 matrix pipe runs at VALU rate and not beside it (a
// timing copy without the conversions ran 1.7x faster, one without the MFMAs as
// long as those alone), so the conversions (~2.4 VALU per weight operand,
// shared by TG MFMAs) add to the 32 cycles of each MFMA; and a CU takes only
// about 27 bytes per clock from L2, so a unit's loads are spread over its
// blocks (4096x4096 at 32 tokens: 22.7 us with the loads in one burst, 17.5 so).
// Measured against the VALU kernels it replaces (us, default numerics): Q4_0
// 4096x4096 at 32 / 512 tokens 50.1 -> 17.5 / 342 -> 176, 4096 -> 11008 at 32
// tokens 70.4 -> 40.0, 11008 -> 4096 131 -> 42; Q8_0 2048 -> 5632 at 72 tokens
// 75 -> 27.  At 512 tokens 97 of the 142-155 TFLOP/s the pipe reaches alone.
constexpr int kRedPad = 4;

template <uint32_t TYPE, int E, int R, int TG, int D, bool ALIGNED>
__global__ __launch_bounds__(kT) void batch_chain_kernel(const uint8_t* __restrict__ W, const float* __restrict__ x,
                                                          float* __restrict__ y, int N, int nb, int B) {
    constexpr int NS = 8 / E, RW = 4 / NS;  // waves over the accumulators, waves over the rows
    using S = WStage<TYPE, R * RW, ALIGNED>;
    constexpr int kTok = 16 * TG, kRows = 16 * R * RW;
    // floats per part of a block (token groups x 4 m x 16 tokens x E; the
    // padding spreads the stores of a token's blocks and parts over the banks)
    constexpr int kXP = kTok * 4 * E + E;
    constexpr int kXB = NS * kXP;
    constexpr int kX = kUnitBlocks * kXB;
    constexpr int kRP = kRows + kRedPad;
    constexpr int kRed = 8 * kTok * kRP;                 // the last sums, in the activation buffers
    __shared__ __align__(16) uint8_t s_w[2][S::kBytes];
    __shared__ __align__(16) float s_x[2 * kX > kRed ? 2 * kX : kRed];
    const int t = threadIdx.x, l = t & 63, w = __builtin_amdgcn_readfirstlane(t >> 6), li = l & 15, m = l >> 4;
    const int part = w % NS, rw = w / NS;
    const int row0 = blockIdx.x * kRows, tok0 = blockIdx.y * kTok;
    const int units = (nb + kUnitBlocks - 1) / kUnitBlocks;
    const int K = nb * 32, row_bytes = nb * Fmt<TYPE>::kB;

    S ws;
    ws.init(W, row0, N, row_bytes);
    // activations: float4 f = t + 256 k of the unit: token f / 64, elements 4 (f % 64) ..
    constexpr int kXs = kTok * 64 / kT;
    struct Set {
        typename S::Piece w[S::kN];
        float4 x[kXs];
    };
    const int xc = t & 63;
    const float* xbase = x + static_cast<size_t>(tok0) * K;
    uint32_t xoff[kXs];
#pragma unroll
    for (int k = 0; k < kXs; ++k)  // tokens past B read token B - 1 (not stored)
        xoff[k] = 4u * (static_cast<uint32_t>(min((t >> 6) + 4 * k, B - 1 - tok0)) * static_cast<uint32_t>(K) + 4 * xc);
    auto load_x = [&](int k, int c, Set& q) __attribute__((always_inline)) {
        if constexpr (ALIGNED) {
            q.x[k] = ld_at<float4>(xbase + c * 256, xoff[k]);
        } else {  // past the row: its first elements, unused
            q.x[k] = ld_at<float4>(xbase, xoff[k] + (c * 256 + 4 * xc < K ? c * 1024 : -16 * xc));
        }
    };
    auto store_x = [&](int k, int buf, const Set& q) __attribute__((always_inline)) {
        float* d = s_x + buf * kX + (xc >> 3) * kXB + (xc & 1) * (4 / E) * kXP + ((xc & 7) >> 1) * (16 * E);
        const int tk = (t >> 6) + 4 * k, o = (tk >> 4) * (64 * E) + (tk & 15) * E;
        if constexpr (E == 4) {
            *reinterpret_cast<float4*>(d + o) = q.x[k];
        } else {
            *reinterpret_cast<float2*>(d + o) = make_float2(q.x[k].x, q.x[k].y);
            *reinterpret_cast<float2*>(d + kXP + o) = make_float2(q.x[k].z, q.x[k].w);
        }
    };
    // share j of 8 of set q: its unit's pieces to LDS, then the pieces of unit
    // c in their place (spread over the unit's blocks: a CU takes about 27
    // bytes per clock from L2, and a wave whose loads queue up cannot issue MFMAs)
    auto turn = [&](int j, int buf, int c, Set& q) __attribute__((always_inline)) {
#pragma unroll
        for (int k = 0; k < kXs; ++k)
            if (k * 8 / kXs == j) {
                if (buf >= 0) store_x(k, buf, q);
                load_x(k, c, q);
            }
#pragma unroll
        for (int i = 0; i < S::kN; ++i)
            if (i * 8 / S::kN == j) {
                if (buf >= 0) ws.store(i, s_w[buf], q.w);
                ws.load(i, c, row_bytes, q.w);
            }
    };

    v4f acc[R][TG][E];
#pragma unroll
    for (int r = 0; r < R; ++r)
#pragma unroll
        for (int g = 0; g < TG; ++g)
#pragma unroll
            for (int e = 0; e < E; ++e) acc[r][g][e] = v4f{0.f, 0.f, 0.f, 0.f};

    // operand bytes of this lane in a block: Q4_0 elements 8m + E*part .. are
    // nibbles m >> 1 of bytes 8(m&1) + E*part ..; Q8_0 bytes 8m + E*part ..
    const int rowo = (rw * R * 16 + li) * S::kUB;
    const int qo = rowo + (TYPE == kQ4_0 ? 8 * (m & 1) : 8 * m) + E * part;
    const int nib_sh = 4 * (m >> 1);
    const int xo = part * kXP + l * E;

    Set ring[D];
    auto compute = [&](int c, Set& q) __attribute__((always_inline)) {
        const int buf = c & 1;
        const int blocks = ALIGNED ? kUnitBlocks : min(kUnitBlocks, nb - c * kUnitBlocks);
        // three stages, so an MFMA never waits for LDS or for a conversion:
        // LDS reads of block j + 1's activations and j + 2's weights, the
        // conversion of j + 1's weights, the MFMAs of block j
        float xb[2][TG][E], a[2][R][E];
        uint32_t rv[2][R][2], rd[2][R];
        auto read_x = [&](int j, float (&d)[TG][E]) __attribute__((always_inline)) {
#pragma unroll
            for (int g = 0; g < TG; ++g) {
                const float* px = s_x + buf * kX + j * kXB + xo + g * (64 * E);
                if constexpr (E == 4) {
                    const float4 v = *reinterpret_cast<const float4*>(px);
                    d[g][0] = v.x, d[g][1] = v.y, d[g][E - 2] = v.z, d[g][E - 1] = v.w;
                } else {
                    const float2 v = *reinterpret_cast<const float2*>(px);
                    d[g][0] = v.x, d[g][1] = v.y;
                }
            }
        };
        auto read_w = [&](int j, uint32_t (&v)[R][2], uint32_t (&d)[R]) __attribute__((always_inline)) {
#pragma unroll
            for (int r = 0; r < R; ++r) {
                const uint8_t* wr = s_w[buf] + r * 16 * S::kUB + j * Fmt<TYPE>::kB;
                d[r] = *reinterpret_cast<const uint16_t*>(wr + rowo);
                if constexpr (E == 2) {
                    v[r][0] = *reinterpret_cast<const uint16_t*>(wr + qo + 2);
                } else if ((j * Fmt<TYPE>::kB) & 2) {  // the quants are dword aligned
                    v[r][0] = *reinterpret_cast<const uint32_t*>(wr + qo + 2);
                } else {
                    const uint32_t* p = reinterpret_cast<const uint32_t*>(wr + qo);
                    v[r][0] = p[0], v[r][1] = p[1];
                }
            }
        };
        auto convert = [&](int j, const uint32_t (&v)[R][2], const uint32_t (&d)[R], float (&o)[R][E]) __attribute__((always_inline)) {
#pragma unroll
            for (int r = 0; r < R; ++r) {
                float dq = h2f(d[r]);
                uint32_t q = E == 2 || ((j * Fmt<TYPE>::kB) & 2) ? v[r][0] : align16(v[r][1], v[r][0]);
                if constexpr (TYPE == kQ4_0) {
                    q = (q ^ 0x88888888u) >> nib_sh;
                    dq = dq * 16.0f;
                }
                weights<TYPE, E>(q, dq, o[r]);
            }
        };
        read_w(0, rv[0], rd[0]);
        read_x(0, xb[0]);
        read_w(1, rv[1], rd[1]);
        __builtin_amdgcn_sched_barrier(0);
        convert(0, rv[0], rd[0], a[0]);
#pragma unroll
        for (int j = 0; j < kUnitBlocks; ++j) {
            if (j + 1 < kUnitBlocks) read_x(j + 1, xb[(j + 1) & 1]);
            if (j + 2 < kUnitBlocks) read_w(j + 2, rv[j & 1], rd[j & 1]);
            __builtin_amdgcn_sched_barrier(0);
            turn(j, buf ^ 1, min(c + 1 + D, units - 1), q);
            __builtin_amdgcn_sched_barrier(0);
            if (ALIGNED || j < blocks)
#pragma unroll
            for (int r = 0; r < R; ++r)
#pragma unroll
                for (int g = 0; g < TG; ++g)
#pragma unroll
                    for (int e = 0; e < E; ++e)
                        acc[r][g][e] = __builtin_amdgcn_mfma_f32_16x16x4f32(a[j & 1][r][e], xb[j & 1][g][e], acc[r][g][e], 0, 0, 0);
            if (j + 1 < kUnitBlocks) convert(j + 1, rv[(j + 1) & 1], rd[(j + 1) & 1], a[(j + 1) & 1]);
            __builtin_amdgcn_sched_barrier(0);
        }
    };
#pragma unroll
    for (int d = 0; d < D; ++d)
#pragma unroll
        for (int j = 0; j < 8; ++j) turn(j, -1, min(d, units - 1), ring[d]);
#pragma unroll
    for (int j = 0; j < 8; ++j) turn(j, 0, min(D, units - 1), ring[0]);
    __syncthreads();
    for (int c = 0; c < units; c += D) {
#pragma unroll
        for (int d = 0; d < D; ++d) {
            if (c + d >= units) break;
            compute(c + d, ring[(d + 1) % D]);  // the other LDS copy was last read in unit c + d - 1
            __syncthreads();
        }
    }
    // t0 + t1 + .. + t7 in order, through LDS: [e][token][row]
#pragma unroll
    for (int r = 0; r < R; ++r)
#pragma unroll
        for (int g = 0; g < TG; ++g)
#pragma unroll
            for (int e = 0; e < E; ++e)
                *reinterpret_cast<v4f*>(s_x + ((part * E + e) * kTok + 16 * g + li) * kRP + (rw * R + r) * 16 + 4 * m) =
                    acc[r][g][e];
    __syncthreads();
#pragma unroll
    for (int i = 0; i < kRows * kTok / kT; ++i) {
        const int o = t + kT * i, row = o % kRows, tk = o / kRows;
        const float* p = s_x + tk * kRP + row;
        float sum = p[0];
#pragma unroll
        for (int e = 1; e < 8; ++e) sum = sum + p[e * kTok * kRP];
        if (row0 + row < N && tok0 + tk < B) y[static_cast<size_t>(tok0 + tk) * N + row0 + row] = sum;
    }
}

template <uint32_t TYPE, int E, int R, int TG, int D, bool ALIGNED>
void chain_one(const uint8_t* W, const float* x, float* y, int N, int nb, int B, hipStream_t st) {
    constexpr int rows = 16 * R * (4 * E / 8);
    const dim3 grid(static_cast<unsigned>((N + rows - 1) / rows), static_cast<unsigned>((B + 16 * TG - 1) / (16 * TG)));
    batch_chain_kernel<TYPE, E, R, TG, D, ALIGNED><<<grid, kT, 0, st>>>(W, x, y, N, nb, B);
}

// The same chains of rows of up to 3 blocks, a thread per (row, token): a
// unit of the matrix-pipe kernel is 8 blocks of work however few a row has.
// That kernel / this one at 512 tokens of 11008 rows (us): Q4_0 K = 32 / 64 /
// 96 75 / 28, 75 / 44, 76 / 66, Q8_0 95 / 33, 98 / 61, 96 / 103, at 11 tokens
// Q8_0 K = 96 9.9 / 8.6; even at 128.
constexpr int kShortK = 96;
template <uint32_t TYPE>
__global__ __launch_bounds__(kT) void batch_short_kernel(const uint8_t* __restrict__ W, const float* __restrict__ x,
                                                          float* __restrict__ y, int N, int nb) {
    constexpr int kQ = TYPE == kQ4_0 ? 4 : 8;  // dwords of quants in a block
    __shared__ float s_x[kShortK];
    const int K = nb * 32;
    const float* xt = x + static_cast<size_t>(blockIdx.y) * K;
    if (static_cast<int>(threadIdx.x) < K) s_x[threadIdx.x] = xt[threadIdx.x];
    __syncthreads();
    const int r = blockIdx.x * kT + threadIdx.x;
    if (r >= N) return;
    const uint16_t* src = reinterpret_cast<const uint16_t*>(W + static_cast<size_t>(r) * nb * Fmt<TYPE>::kB);
    float t[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
    for (int b = 0; b < nb; ++b, src += Fmt<TYPE>::kB / 2) {
        uint32_t q[kQ];
#pragma unroll
        for (int k = 0; k < kQ; ++k) q[k] = src[1 + 2 * k] | static_cast<uint32_t>(src[2 + 2 * k]) << 16;
        const float d = h2f(src[0]);
#pragma unroll
        for (int k = 0; k < 8; ++k) {  // elements 4k .. 4k + 3
            float a[4];
            if constexpr (TYPE == kQ4_0) weights<TYPE, 4>((q[k & 3] ^ 0x88888888u) >> (k < 4 ? 0 : 4), d * 16.0f, a);
            else weights<TYPE, 4>(q[k], d, a);
#pragma unroll
            for (int i = 0; i < 4; ++i) t[4 * (k & 1) + i] = fmaf(a[i], s_x[32 * b + 4 * k + i], t[4 * (k & 1) + i]);
        }
    }
    float s = t[0];
#pragma unroll
    for (int e = 1; e < 8; ++e) s = s + t[e];
    y[static_cast<size_t>(blockIdx.y) * N + r] = s;
}

template <uint32_t TYPE>
hipError_t launch_chain(const uint8_t* W, const float* x, float* y, size_t rows, size_t cols, size_t batch,
                        hipStream_t st) {
    const int N = static_cast<int>(rows), nb = static_cast<int>(cols / 32), B = static_cast<int>(batch);
    if (cols <= kShortK && batch <= 65535) {  // grid y: tokens
        const dim3 grid(static_cast<unsigned>((rows + kT - 1) / kT), static_cast<unsigned>(batch));
        batch_short_kernel<TYPE><<<grid, kT, 0, st>>>(W, x, y, N, nb);
        return hipGetLastError();
    }
    const bool aligned = cols % 256 == 0 && (reinterpret_cast<uintptr_t>(W) & 15) == 0;
    if (!aligned) {
        chain_one<TYPE, 2, 1, 1, 2, false>(W, x, y, N, nb, B, st);
        return hipGetLastError();
    }
    // The tile with the least estimated time.  A workgroup's time per 8-block
    // unit, measured (us): alone on its CU (4096x4096 at 8 and 32 tokens) and
    // as one of several there (4096 -> 11008 / 22016 at 32 tokens, 4096x4096
    // at 512); the workgroups of the busiest of the 256 CUs count.  Small tiles
    // keep every CU busy where there are few rows (4096x4096 at 32 tokens:
    // 16x32 17.5 us, 32x32 28 us), larger ones read the activations less often
    // (at 512 tokens: 32x32 176 us, 16x32 208 us, 16x16 220 us).  All of it is
    // Q4_0's: a Q8_0 workgroup takes 83 KB of LDS at 32x32 and 92 at 48x32, so
    // a CU has one of them and not two.
    struct Tile {
        int rows, toks;
        float alone, shared;
    };
    static constexpr Tile kTiles[] = {
        {16, 16, 0.83f, 0.49f}, {16, 32, 1.09f, 0.88f}, {32, 16, 1.13f, 0.83f}, {32, 32, 1.75f, 1.42f}, {48, 32, 2.57f, 2.15f}};
    int best = 0;
    float best_us = 0.0f;
    for (int i = 0; i < 5; ++i) {
        const Tile& c = kTiles[i];
        const size_t wgs = (rows + c.rows - 1) / c.rows * ((batch + c.toks - 1) / c.toks), n = (wgs + 255) / 256;
        const float us = n == 1 ? c.alone : static_cast<float>(n) * c.shared;
        if (i == 0 || us < best_us) best = i, best_us = us;
    }
    switch (best) {
    case 0: chain_one<TYPE, 2, 1, 1, 2, true>(W, x, y, N, nb, B, st); break;
    case 1: chain_one<TYPE, 2, 1, 2, 2, true>(W, x, y, N, nb, B, st); break;
    case 2: chain_one<TYPE, 4, 1, 1, 2, true>(W, x, y, N, nb, B, st); break;
    case 3: chain_one<TYPE, 4, 1, 2, 2, true>(W, x, y, N, nb, B, st); break;
    default: chain_one<TYPE, 2, 3, 2, 2, true>(W, x, y, N, nb, B, st); break;
    }
    return hipGetLastError();
}

// ---- per-block sums (the per-token fp32 dots over several tokens) --------------
//
// A workgroup owns 16*R rows x 16 tokens.  The block sums are independent of
// each other, so its four waves take them in turn, four blocks (a step) each;
// the sums and the scales meet in LDS, and per round of 16 blocks every thread
// runs the in-order fma chain of its R outputs over them.  A wave's weight
// bytes of a step pass through an LDS copy of its own; the activations are the
// other operand as they lie in memory (8 floats per lane and block).  Both are
// fetched one round ahead.
// What bounds it: eight f32 MFMAs (256 cycles) and the 28 adds of their lane
// sums per 16 x 16 outputs and block, which exclude each other; with a
// workgroup or less per CU, the latency of a round (about 2 us).
// Against the VALU kernels before (us): Q8_0 2048->5632 at 5 / 16 / 64 / 256
// tokens 22.6 / 25.2 / 51.9 / 161 -> 13.0 / 15.7 / 30.8 / 96; Q4_0 4096->11008
// 55 / 58 / 167 / 604 -> 28.5 / 33.1 / 102 / 346.
template <uint32_t TYPE, int R>
__global__ __launch_bounds__(kT) void batch_blocksum_kernel(const uint8_t* __restrict__ W, const float* __restrict__ x,
                                                            float* __restrict__ y, int N, int nb, int B) {
    constexpr int kS = 4, kRound = 4 * kS;        // blocks per step, per round
    constexpr int kB = Fmt<TYPE>::kB, kUB = kS * kB, kPitch = kUB + 4;  // an odd number of dwords
    constexpr int kRows = 16 * R, kPieces = kRows * (kUB / 8), kN = (kPieces + 63) / 64;
    static_assert(kUB % 8 == 0);
    __shared__ __align__(16) uint8_t s_w[4][kRows * kPitch + 8];  // + a spare slot for unused stores
    __shared__ float s_s[kRound][R][4][64];                       // [block][row group][token v of lane][lane]
    __shared__ float s_d[kRound][kRows];
    const int t = threadIdx.x, l = t & 63, w = __builtin_amdgcn_readfirstlane(t >> 6), li = l & 15, m = l >> 4;
    const int row0 = blockIdx.x * kRows, tok0 = blockIdx.y * 16;
    const int steps = nb / kS, K = nb * 32, row_bytes = nb * kB;

    const uint8_t* wbase = W + static_cast<size_t>(row0) * row_bytes;
    uint32_t src[kN];
    int dst[kN];
#pragma unroll
    for (int i = 0; i < kN; ++i) {
        const int p = l + 64 * i, pc = min(p, kPieces - 1), row = pc / (kUB / 8), k = pc % (kUB / 8);
        // rows past N read row N - 1, tokens past B token B - 1 (not stored)
        src[i] = static_cast<uint32_t>(min(row, N - 1 - row0)) * static_cast<uint32_t>(row_bytes) + 8 * k;
        dst[i] = p < kPieces ? row * kPitch + 8 * k : kRows * kPitch;
    }
    const float* xbase = x + static_cast<size_t>(tok0) * K;
    const uint32_t xoff = 4u * (static_cast<uint32_t>(min(li, B - 1 - tok0)) * static_cast<uint32_t>(K) + 8 * m);
    uint2 wreg[kN];
    float4 xreg[kS][2];
    auto load = [&](int step) __attribute__((always_inline)) {
        const uint8_t* p = wbase + step * kUB;
#pragma unroll
        for (int i = 0; i < kN; ++i) wreg[i] = ld_at<uint2>(p, src[i]);
#pragma unroll
        for (int j = 0; j < kS; ++j) {
            xreg[j][0] = ld_at<float4>(xbase + (step * kS + j) * 32, xoff);
            xreg[j][1] = ld_at<float4>(xbase + (step * kS + j) * 32 + 4, xoff);
        }
    };
    // the lane's operand bytes of a block: Q4_0 elements 8m .. are nibbles m >> 1 of bytes 8 (m & 1) ..
    const int rowo = li * kPitch, qo = rowo + (TYPE == kQ4_0 ? 8 * (m & 1) : 8 * m);
    const int nib_sh = 4 * (m >> 1);
    float sum[R];
#pragma unroll
    for (int r = 0; r < R; ++r) sum[r] = 0.f;

    load(min(w, steps - 1));
    for (int r0 = 0; r0 < steps; r0 += 4) {
        float4 xc[kS][2];
#pragma unroll
        for (int j = 0; j < kS; ++j) xc[j][0] = xreg[j][0], xc[j][1] = xreg[j][1];
#pragma unroll
        for (int i = 0; i < kN; ++i) {
            uint32_t* p = reinterpret_cast<uint32_t*>(s_w[w] + dst[i]);
            p[0] = wreg[i].x, p[1] = wreg[i].y;
        }
        load(min(r0 + 4 + w, steps - 1));
        __builtin_amdgcn_wave_barrier();
        if (r0 + w < steps) {
#pragma unroll
            for (int j = 0; j < kS; ++j) {
                const float xv[8] = {xc[j][0].x, xc[j][0].y, xc[j][0].z, xc[j][0].w,
                                     xc[j][1].x, xc[j][1].y, xc[j][1].z, xc[j][1].w};
#pragma unroll
                for (int r = 0; r < R; ++r) {
                    const uint8_t* wr = s_w[w] + r * 16 * kPitch + j * kB;
                    uint32_t q[2];
                    if ((j * kB) & 2) {  // the quants are dword aligned
                        const uint32_t* p = reinterpret_cast<const uint32_t*>(wr + qo + 2);
                        q[0] = p[0], q[1] = p[1];
                    } else {
                        const uint32_t* p = reinterpret_cast<const uint32_t*>(wr + qo);
                        q[0] = align16(p[1], p[0]), q[1] = align16(p[2], p[1]);
                    }
                    if (m == 0)
                        s_d[w * kS + j][16 * r + li] = h2f(*reinterpret_cast<const uint16_t*>(wr + rowo));
                    float a[2][4];
#pragma unroll
                    for (int e = 0; e < 2; ++e) {
                        if constexpr (TYPE == kQ4_0)
                            weights<TYPE, 4>((q[e] ^ 0x88888888u) >> nib_sh, 16.0f, a[e]);
                        else
                            weights<TYPE, 4>(q[e], 1.0f, a[e]);
                    }
                    v4f te[8];
#pragma unroll
                    for (int e = 0; e < 8; ++e)
                        te[e] = __builtin_amdgcn_mfma_f32_16x16x4f32(xv[e], a[e >> 2][e & 3], v4f{0.f, 0.f, 0.f, 0.f}, 0, 0, 0);
                    v4f s = te[0];
#pragma unroll
                    for (int e = 1; e < 8; ++e)
#pragma unroll
                        for (int v = 0; v < 4; ++v) s[v] = s[v] + te[e][v];
#pragma unroll
                    for (int v = 0; v < 4; ++v) s_s[w * kS + j][r][v][l] = s[v];
                }
            }
        }
        __syncthreads();
        for (int b0 = 0; b0 < min(kRound, nb - r0 * kS); b0 += 8)  // whole halves of a round: nb % 8 == 0
#pragma unroll
            for (int b = 0; b < 8; ++b)
#pragma unroll
                for (int r = 0; r < R; ++r) sum[r] = fmaf(s_d[b0 + b][16 * r + li], s_s[b0 + b][r][w][l], sum[r]);
        __syncthreads();
    }
    // wave w, lane l: token 4m + w, row li of each row group
    const int tk = tok0 + 4 * m + w;
#pragma unroll
    for (int r = 0; r < R; ++r) {
        const int row = row0 + 16 * r + li;
        if (row < N && tk < B) y[static_cast<size_t>(tk) * N + row] = sum[r];
    }
}

template <uint32_t TYPE, int R>
void blocksum_one(const uint8_t* W, const float* x, float* y, int N, int nb, int B, hipStream_t st) {
    const dim3 grid(static_cast<unsigned>((N + 16 * R - 1) / (16 * R)), static_cast<unsigned>((B + 15) / 16));
    batch_blocksum_kernel<TYPE, R><<<grid, kT, 0, st>>>(W, x, y, N, nb, B);
}

}  // namespace

hipError_t launch_batch4_f32act(uint32_t type, const uint8_t* W, const float* x, float* y, size_t rows, size_t cols,
                                size_t batch, hipStream_t st) {
    if (!rows || !batch) return hipSuccess;
    return type == kQ4_0 ? launch_chain<kQ4_0>(W, x, y, rows, cols, batch, st)
                         : launch_chain<kQ8_0>(W, x, y, rows, cols, batch, st);
}

bool batch_blocksum_ok(uint32_t type, const uint8_t* W, size_t cols) {
    return (type == kQ4_0 || type == kQ8_0) && cols % 256 == 0 && (reinterpret_cast<uintptr_t>(W) & 15) == 0;
}

hipError_t launch_batch_blocksum(uint32_t type, const uint8_t* W, const float* x, float* y, size_t rows, size_t cols,
                                 size_t batch, hipStream_t st) {
    if (!rows || !batch) return hipSuccess;
    if (!batch_blocksum_ok(type, W, cols)) return hipErrorInvalidValue;
    const int N = static_cast<int>(rows), nb = static_cast<int>(cols / 32), B = static_cast<int>(batch);
    // 32-row tiles read the activations half as often; 16-row ones where those
    // would be fewer than two workgroups per CU (2048->5632 Q8_0 at 32 / 64
    // tokens: 16 rows 19.9 / 35.9 us, 32 rows 23.4 / 30.8)
    const int R = (rows + 31) / 32 * ((batch + 15) / 16) >= 512 ? 2 : 1;
    if (type == kQ4_0) {
        if (R == 2) blocksum_one<kQ4_0, 2>(W, x, y, N, nb, B, st);
        else blocksum_one<kQ4_0, 1>(W, x, y, N, nb, B, st);
    } else {
        if (R == 2) blocksum_one<kQ8_0, 2>(W, x, y, N, nb, B, st);
        else blocksum_one<kQ8_0, 1>(W, x, y, N, nb, B, st);
    }
    return hipGetLastError();
}

}  // namespace mvh
