// mvh_gemm_q4.hip -- batched-prefill Q4_0 x Q8 GEMM on int8 MFMA.
//
// Numerics: tensor_matmul_batch_v06 with MEMVANTA_FORCE_Q8_ACT=1
// (src/gguf_kernels.cpp:265-267): every token's activation row is quantized
// with quantize_q8, and every (row, token) output is dot_q4_q8 (:189):
//   sum = fma(f16(d_w[b]) * d_a[b], float(isum_b), sum)   over blocks b in order,
// with isum_b the exact integer dot of block b.  One v_mfma_i32_16x16x32_i8
// has K = 32 = one block, so it yields isum_b for a 16 x 16 (token x row)
// tile exactly (int8 x int8 -> int32, no rounding); each lane then applies
// the reference's fma for its 4 outputs, block after block, so every output
// is the reference's chain bit for bit.  No split-K, no reassociation.
//
// Work split: one wave per tile of 16 weight rows x 16*TG tokens, independent
// of every other wave (wave-private LDS, no workgroup barriers); the
// activation operands come in the MFMA operand order (q8_op_offset), so one
// block's A operand is one fully used 512-byte load.  Per K-chunk of 8 blocks
// (256 elements):
//   1. the tile's raw Q4_0 bytes (16 rows x 144 B; a row's chunk is 16-byte
//      aligned when K % 256 == 0) come in with 16-byte loads, D chunks ahead;
//   2. they are staged in a wave-private LDS copy and each lane reads back
//      its own MFMA operand bytes and the row's f16 scale;
//   3. per block and token group two MFMAs give the exact block sum (the
//      nibbles as they are, the -8 through the accumulator); each lane then
//      applies the reference's fma to its 4 outputs.
#include "mvh_kernels.hpp"

#include <cstdlib>

namespace mvh {
namespace {

typedef int v4i __attribute__((ext_vector_type(4)));

constexpr int kRows = 16;   // weight rows per wave
constexpr int kChunk = 8;   // blocks per K-chunk
constexpr int kUnit = 144;  // bytes of 8 Q4_0 blocks of one row
constexpr int kWPieces = kRows * kUnit / 16;  // 144 16-byte pieces of raw weights per chunk

// bytes (q - 8) of four nibbles held one per byte (0..15) are not formed:
// the MFMA takes the nibbles as they are (0..15 is a valid int8) and the
// -8 offset comes in through the accumulator, C = A x (-8), an exact int32.
constexpr long kMinus8 = static_cast<long>(0xF8F8F8F8F8F8F8F8ull);

template <int TG>
struct ChunkRegs {
    uint4 w[3];           // raw weight pieces l, l+64, l+128 (16 rows x 144 B)
    long a[TG][kChunk];   // A operands: token group g, block j
    float da[2 * TG];     // activation scales: token l / (4/TG), blocks 2*TG*(l % (4/TG)) ..
};

// One wave per tile of 16 weight rows x 16*TG tokens, independent of every
// other wave.  The tile's K-chunks (8 blocks, 144 bytes per row) stream
// through a ring of D register sets, D chunks ahead of the chunk being
// computed; every load is issued unconditionally (clamped addresses), so the
// compiler's wait counts stay exact and never wait for the ring's later
// chunks.  Per chunk:
//   1. the raw bytes go to a wave-private LDS copy, the scales next to it;
//   2. each lane reads back the 8 quant bytes of its MFMA operand (row li,
//      elements 8h .. 8h+7 of the block: low nibbles of qs[8(h&1) ..] for
//      h < 2, high nibbles for h >= 2) and the row's scale, in registers;
//   3. per block and token group: C = A x (-8), D = A x nibbles + C -- the
//      exact block sum -- then the reference's fma for the lane's 4 outputs.
template <int TG, int D>
__global__ __launch_bounds__(64) void gemm_q4_0_q8_mfma_kernel(const uint8_t* __restrict__ W,
                                                               const int8_t* __restrict__ aq,
                                                               const float* __restrict__ ad,
                                                               float* __restrict__ y, int N, int nb, int B) {
    constexpr int kToks = 16 * TG;
    constexpr int kDaL = 4 / TG;  // lanes per token in the scale load
    __shared__ __align__(16) uint8_t s_raw[kRows * kUnit];
    __shared__ __align__(16) float s_da[kChunk * kToks];  // [block][token]

    const int l = threadIdx.x, li = l & 15, h = l >> 4;
    const int r0 = blockIdx.x * kRows, t0 = blockIdx.y * kToks;
    const size_t row_bytes = static_cast<size_t>(nb) * 18, K = static_cast<size_t>(nb) * 32;
    const int nchunks = nb / kChunk;
    // raw piece p of the chunk: row p / 9, bytes 16 (p % 9); lanes past 143 reload piece 0
    const uint8_t* wp[3];
    int wo[3];
#pragma unroll
    for (int i = 0; i < 3; ++i) {
        const int p = l + 64 * i, pc = p < kWPieces ? p : 0;
        wp[i] = W + static_cast<size_t>(min(r0 + pc / 9, N - 1)) * row_bytes + (pc % 9) * 16;
        wo[i] = p < kWPieces ? (p / 9) * kUnit + (p % 9) * 16 : -1;
    }
    // A operands in operand order: slab of 16 tokens, then 4 KB per chunk,
    // 512 B per block (lane l's 8 bytes at 8l); a partial group past the last
    // slab reads the last slab again (its outputs are not stored)
    const int8_t* ap[TG];
#pragma unroll
    for (int g = 0; g < TG; ++g)
        ap[g] = aq + static_cast<size_t>(min(blockIdx.y * TG + g, (B - 1) / 16)) * 16 * K + 8 * l;
    const int da_t = l / kDaL, da_b = (l % kDaL) * 2 * TG;
    const float* dp = ad + static_cast<size_t>(min(t0 + da_t, B - 1)) * nb + da_b;

    // the scheduling barriers keep every chunk's loads in ring order: loads
    // reordered across chunks would make the wait for the oldest chunk also
    // wait for the newer ones
    auto fetch = [&](ChunkRegs<TG>& r, int c) {
        __builtin_amdgcn_sched_barrier(0);
        c = min(c, nchunks - 1);
        const size_t wc = static_cast<size_t>(c) * kUnit;
#pragma unroll
        for (int i = 0; i < 3; ++i) r.w[i] = ld_global16(wp[i] + wc);
#pragma unroll
        for (int g = 0; g < TG; ++g)
#pragma unroll
            for (int j = 0; j < kChunk; ++j)
                r.a[g][j] = *reinterpret_cast<const long*>(ap[g] + static_cast<size_t>(c) * 4096 + 512 * j);
        if constexpr (TG == 2) {
            const float4 v = *reinterpret_cast<const float4*>(dp + c * kChunk);
            r.da[0] = v.x; r.da[1] = v.y; r.da[2] = v.z; r.da[3] = v.w;
        } else {
            const float2 v = *reinterpret_cast<const float2*>(dp + c * kChunk);
            r.da[0] = v.x; r.da[1] = v.y;
        }
        __builtin_amdgcn_sched_barrier(0);
    };

    float acc[TG][4];
#pragma unroll
    for (int g = 0; g < TG; ++g) acc[g][0] = acc[g][1] = acc[g][2] = acc[g][3] = 0.f;

    // the lane's operand bytes: row li, qs[8(h&1) .. +8) of each block, nibble half h >> 1
    const uint8_t* my_q = s_raw + li * kUnit + 2 + 8 * (h & 1);
    const uint32_t nib_shift = 4u * static_cast<uint32_t>(h >> 1);

    auto compute = [&](const ChunkRegs<TG>& r) {
        // LDS operations of one wave are performed in order, so the reads
        // below see these writes and the next chunk's writes come after them
#pragma unroll
        for (int i = 0; i < 3; ++i) {
            // pieces past the tile's 144 go to piece 0's place with piece 0's bytes
            *reinterpret_cast<uint4*>(s_raw + (wo[i] < 0 ? 0 : wo[i])) = r.w[i];
        }
#pragma unroll
        for (int e = 0; e < 2 * TG; ++e) s_da[(da_b + e) * kToks + da_t] = r.da[e];
        __builtin_amdgcn_wave_barrier();
#pragma unroll
        for (int j = 0; j < kChunk; ++j) {
            uint32_t q0, q1;
            if ((j & 1) == 0) {  // 18j + 2 + 8(h&1) is 2 mod 4: three dwords, shifted by 2 bytes
                const uint32_t* p = reinterpret_cast<const uint32_t*>(my_q + 18 * j - 2);
                const uint32_t w0 = p[0], w1 = p[1], w2 = p[2];
                q0 = align16(w1, w0);
                q1 = align16(w2, w1);
            } else {
                const uint32_t* p = reinterpret_cast<const uint32_t*>(my_q + 18 * j);
                q0 = p[0];
                q1 = p[1];
            }
            const uint32_t n0 = (q0 >> nib_shift) & 0x0f0f0f0fu, n1 = (q1 >> nib_shift) & 0x0f0f0f0fu;
            const long bop = static_cast<long>((static_cast<unsigned long>(n1) << 32) | n0);
            const float dw = h2f(*reinterpret_cast<const uint16_t*>(s_raw + li * kUnit + 18 * j));
#pragma unroll
            for (int g = 0; g < TG; ++g) {
                const v4i c8 = __builtin_amdgcn_mfma_i32_16x16x32_i8(r.a[g][j], kMinus8, v4i{0, 0, 0, 0}, 0, 0, 0);
                const v4i is = __builtin_amdgcn_mfma_i32_16x16x32_i8(r.a[g][j], bop, c8, 0, 0, 0);
                const float4 da = *reinterpret_cast<const float4*>(s_da + j * kToks + 16 * g + 4 * h);
                acc[g][0] = fmaf(dw * da.x, static_cast<float>(is[0]), acc[g][0]);
                acc[g][1] = fmaf(dw * da.y, static_cast<float>(is[1]), acc[g][1]);
                acc[g][2] = fmaf(dw * da.z, static_cast<float>(is[2]), acc[g][2]);
                acc[g][3] = fmaf(dw * da.w, static_cast<float>(is[3]), acc[g][3]);
            }
        }
        __builtin_amdgcn_wave_barrier();
    };

    ChunkRegs<TG> ring[D];
#pragma unroll
    for (int d = 0; d < D; ++d) fetch(ring[d], d);
    for (int c = 0; c < nchunks; c += D) {
#pragma unroll
        for (int d = 0; d < D; ++d) {
            if (c + d < nchunks) compute(ring[d]);
            fetch(ring[d], c + d + D);
        }
    }

    // lane holds (token 16g + 4h + v, row li) of each token group g
    const int orow = r0 + li;
    if (orow < N) {
#pragma unroll
        for (int g = 0; g < TG; ++g)
#pragma unroll
            for (int v = 0; v < 4; ++v) {
                const int tk = t0 + 16 * g + 4 * h + v;
                if (tk < B) y[static_cast<size_t>(tk) * N + orow] = acc[g][v];
            }
    }
}

typedef int v16i __attribute__((ext_vector_type(16)));
typedef float v16f __attribute__((ext_vector_type(16)));
typedef float v32f __attribute__((ext_vector_type(32)));

// 12582912 = 1.5 * 2^23: an int32 sum s (|s| < 2^22) added to this float's bits
// gives the float 12582912 + s.
constexpr int kMagic = 0x4B400000;

// The same numerics for large batches: a workgroup of 4 waves shares one LDS
// copy of each K-step of 4 blocks, and a wave computes 32 tokens x 32 rows
// (WT waves over the tokens, 4 / WT over the rows).  Per block and 32 x 32
// outputs:
//   * one v_mfma_i32_32x32x32_i8 (twice the rate of the 16x16x32 form) of the
//     activations and 16 (q - 8), a nibble in a byte's upper half with its top
//     bit flipped; no extra product for the -8;
//   * its accumulator starts at kMagic, so the result is the float 12582912 +
//     16 isum, and fma(that, 1/16, -12582912/16) = float(isum) exactly: a
//     v_cvt_f32_i32 issues at half the rate of an fma;
//   * f16(d_w) * d_a for two blocks and all 32 x 32 outputs is one rank-one
//     v_mfma_f32_32x32x1_2b_f32, each product rounded once as the reference's.
// The fmas of a block run while its successor's operands are read, and the
// successor's products then take their registers.
// What bounds it: VALU and f32-MFMA issue, which exclude each other (per 16 x
// 16 outputs and block about 20 cycles of fma, 8 + 8 of MFMA, 7 of unpacking),
// at two waves per SIMD.  Masks and constants are held in VGPRs: an operand in
// an SGPR halves a VALU instruction's rate (4.4 against 2.5 cycles measured).
// Against the four-wave 16x16x32 kernel it replaces, both with the quantizer:
// 512 tokens 4096x4096 61 -> 43 us, 4096->11008 138 -> 97, 11008->4096 140 ->
// 97, 4096->22016 260 -> 176 (525 TOP/s).
template <int WT>
__global__ __launch_bounds__(256, 2) void gemm_q4_0_q8_tile_kernel(const uint8_t* __restrict__ W,
                                                                const int8_t* __restrict__ aq,
                                                                const float* __restrict__ ad,
                                                                float* __restrict__ y, int N, int nb, int B) {
    constexpr int kStep = 4;              // blocks per K-step
    constexpr int kBytes = 18 * kStep;    // a row's bytes of a step
    constexpr int kPitch = kBytes + 4;    // an odd number of dwords: 32 rows on 32 banks
    constexpr int WR = 4 / WT;            // waves over the rows
    constexpr int kToks = 32 * WT, kWgRows = 32 * WR;
    constexpr int kPieces = kWgRows * 9;
    constexpr int kWLd = (kPieces + 255) / 256;  // 8-byte weight loads per thread
    constexpr int kAu = WT;                      // activation units per thread
    constexpr int kDl = (kToks * kStep + 255) / 256;
    __shared__ __align__(16) uint8_t s_w[2][kWgRows * kPitch + 16];     // + a spare slot for unused stores
    __shared__ __align__(16) int8_t s_a[2][kStep * 2 * kToks * 16];     // [block][half][token][16]
    __shared__ __align__(16) float s_da[2][kStep * kToks];              // [block][token]

    const int t = threadIdx.x, l = t & 63, wv = __builtin_amdgcn_readfirstlane(t >> 6), li = l & 31, h = l >> 5;
    const int wt = wv % WT, wr = wv / WT;
    const int r0 = blockIdx.x * kWgRows, t0 = blockIdx.y * kToks;
    const size_t row_bytes = static_cast<size_t>(nb) * 18, K = static_cast<size_t>(nb) * 32;
    const int steps = nb / kStep;

    const uint8_t* wbase = W + static_cast<size_t>(r0) * row_bytes;
    uint32_t wsrc[kWLd];
    int wdst[kWLd];
#pragma unroll
    for (int i = 0; i < kWLd; ++i) {
        const int p = t + 256 * i, pc = min(p, kPieces - 1), row = pc / 9, k = pc % 9;
        wsrc[i] = static_cast<uint32_t>(min(row, N - 1 - r0)) * static_cast<uint32_t>(row_bytes) + k * 8;
        wdst[i] = p < kPieces ? row * kPitch + k * 8 : kWgRows * kPitch;
    }
    // activation unit u = t + 256 i: token u % 16 of 16-token slab u / 128, half u / 16 % 2 (its
    // quarters q and q + 2, as a weight byte's two nibbles) of block u / 32 % 4; slabs past the
    // last read the last one (not stored)
    const int slab0 = static_cast<int>(blockIdx.y) * 2 * WT, slabs = (B + 15) / 16;
    const int8_t* const abase = aq + static_cast<size_t>(slab0) * 16 * K;
    uint32_t asrc[kAu];
#pragma unroll
    for (int i = 0; i < kAu; ++i)
        asrc[i] = static_cast<uint32_t>(min(2 * i + (t >> 7), slabs - 1 - slab0)) * static_cast<uint32_t>(16 * K) +
                  (t >> 5 & 3) * 512 + (t >> 4 & 1) * 128 + (t & 15) * 8;
    const int adst = (t >> 4 & 7) * (kToks * 16) + ((t >> 7) * 16 + (t & 15)) * 16;
    // scale e = t + 256 i: token e / 4, block e % 4
    const float* const dbase = ad + static_cast<size_t>(t0) * nb;
    uint32_t dsrc[kDl];
    int ddst[kDl];
#pragma unroll
    for (int i = 0; i < kDl; ++i) {
        const int e = (t + 256 * i) % (kToks * kStep);
        dsrc[i] = static_cast<uint32_t>(min(e / 4, B - 1 - t0)) * static_cast<uint32_t>(nb) + e % 4;
        ddst[i] = e % 4 * kToks + e / 4;
    }

    struct Regs {
        uint2 w[kWLd], a[kAu][2];
        float d[kDl];
    } q;
    auto load = [&](int c) __attribute__((always_inline)) {
        const uint8_t* wc = wbase + static_cast<size_t>(c) * kBytes;
#pragma unroll
        for (int i = 0; i < kWLd; ++i) q.w[i] = ld_global8(wc + wsrc[i]);
#pragma unroll
        for (int i = 0; i < kAu; ++i) {
            q.a[i][0] = ld_global8(abase + static_cast<size_t>(c) * 2048 + asrc[i]);
            q.a[i][1] = ld_global8(abase + static_cast<size_t>(c) * 2048 + 256 + asrc[i]);
        }
#pragma unroll
        for (int i = 0; i < kDl; ++i) q.d[i] = (dbase + c * kStep)[dsrc[i]];
    };
    auto store = [&](int buf) __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < kWLd; ++i) {
            uint32_t* p = reinterpret_cast<uint32_t*>(s_w[buf] + wdst[i]);
            p[0] = q.w[i].x, p[1] = q.w[i].y;
        }
#pragma unroll
        for (int i = 0; i < kAu; ++i)
            *reinterpret_cast<uint4*>(s_a[buf] + adst + i * 512) = make_uint4(q.a[i][0].x, q.a[i][0].y, q.a[i][1].x, q.a[i][1].y);
#pragma unroll
        for (int i = 0; i < kDl; ++i) s_da[buf][ddst[i]] = q.d[i];
    };

    v16f acc = {};
    v16i is[2];
    v32f p = {};
    v16i magic;
#pragma unroll
    for (int i = 0; i < 16; ++i) magic[i] = kMagic;
    is[0] = is[1] = magic;
    // in VGPRs: see above
    uint32_t mask = 0xf0f0f0f0u, bias = 0x80808080u;
    float sixteenth = 0.0625f, off = -12582912.0f / 16.0f;
    asm volatile("" : "+v"(mask), "+v"(bias), "+v"(sixteenth), "+v"(off));
    const int my_w = (32 * wr + li) * kPitch, my_a = (h * kToks + 32 * wt + li) * 16, my_d = 32 * wt + li;

    struct Ops {
        v4i a[2];
        uint32_t q[2][3], d;
        float da;
    };
    auto read = [&](int buf, int j, Ops& o) __attribute__((always_inline)) {  // blocks j and j + 1, j even: 18j is a whole dword
        const uint8_t* w = s_w[buf] + my_w + 18 * j;
        o.d = *reinterpret_cast<const uint16_t*>(w + 18 * h);
        o.da = s_da[buf][(j + h) * kToks + my_d];
        const uint32_t* p0 = reinterpret_cast<const uint32_t*>(w + 8 * h);
        o.q[0][0] = p0[0], o.q[0][1] = p0[1], o.q[0][2] = p0[2];
        const uint32_t* p1 = reinterpret_cast<const uint32_t*>(w + 20 + 8 * h);
        o.q[1][0] = p1[0], o.q[1][1] = p1[1];
#pragma unroll
        for (int b = 0; b < 2; ++b)
            o.a[b] = *reinterpret_cast<const v4i*>(s_a[buf] + (j + b) * (2 * kToks * 16) + my_a);
    };
    auto chain = [&](int b) __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < 16; ++i) {
            const float s = fmaf(__int_as_float(is[b][i]), sixteenth, off);
            acc[i] = fmaf(p[16 * b + i], s, acc[i]);
        }
    };
    auto operand = [&](uint32_t q0, uint32_t q1) __attribute__((always_inline)) {
        return v4i{static_cast<int>((q0 << 4 & mask) ^ bias), static_cast<int>((q1 << 4 & mask) ^ bias),
                   static_cast<int>((q0 & mask) ^ bias), static_cast<int>((q1 & mask) ^ bias)};
    };
    auto pair = [&](const Ops& o) __attribute__((always_inline)) {
        const v4i w0 = operand(align16(o.q[0][1], o.q[0][0]), align16(o.q[0][2], o.q[0][1]));
        const float dw = h2f(o.d);
        chain(0);
        __builtin_amdgcn_sched_barrier(0);
        is[0] = __builtin_amdgcn_mfma_i32_32x32x32_i8(o.a[0], w0, magic, 0, 0, 0);
        const v4i w1 = operand(o.q[1][0], o.q[1][1]);
        chain(1);
        __builtin_amdgcn_sched_barrier(0);
        is[1] = __builtin_amdgcn_mfma_i32_32x32x32_i8(o.a[1], w1, magic, 0, 0, 0);
        p = __builtin_amdgcn_mfma_f32_32x32x1f32(o.da, dw, v32f{}, 0, 0, 0);
        __builtin_amdgcn_sched_barrier(0);
    };

    load(0);
    store(0);
    load(min(1, steps - 1));
    for (int c = 0; c < steps; c += 2) {
#pragma unroll
        for (int d = 0; d < 2; ++d) {
            __syncthreads();
            Ops o;
            read(d, 0, o);
            __builtin_amdgcn_sched_barrier(0);
            pair(o);
            read(d, 2, o);
            store(d ^ 1);  // the idle buffer was last read in step c + d - 1
            load(min(c + d + 2, steps - 1));  // unconditional: past the end the last step again
            __builtin_amdgcn_sched_barrier(0);
            pair(o);
        }
    }
    chain(0);
    chain(1);

    // lane holds row 32 wr + li, tokens 8 (i / 4) + 4 h + i % 4
    const int orow = r0 + 32 * wr + li;
    if (orow < N) {
#pragma unroll
        for (int i = 0; i < 16; ++i) {
            const int tk = t0 + 32 * wt + 8 * (i / 4) + 4 * h + i % 4;
            if (tk < B) y[static_cast<size_t>(tk) * N + orow] = acc[i];
        }
    }
}

}  // namespace

bool gemm_q4_0_mfma_ok(size_t cols) { return cols >= 256 && cols % 256 == 0; }

hipError_t launch_gemm_q4_0_q8_mfma(const uint8_t* W, const int8_t* aq, const float* ad, float* y, size_t rows,
                                    size_t cols, size_t batch, hipStream_t st) {
    if (!rows || !batch) return hipSuccess;
    if (!gemm_q4_0_mfma_ok(cols)) return hipErrorInvalidValue;
    const unsigned gx = static_cast<unsigned>((rows + kRows - 1) / kRows);
    const int N = static_cast<int>(rows), nb = static_cast<int>(cols / 32), Bn = static_cast<int>(batch);
    const size_t g16 = (batch + 15) / 16, g32 = (batch + 31) / 32;
    // 16-token tiles while the grid is small (more waves, shorter chains);
    // 32-token tiles share each weight operand when there are waves to spare.
    // The deeper ring pays where few waves each stream a long K.
    // From 512 row tiles (N >= 8192: the fused q|k|v and gate|up) 32-token
    // tiles pay even at M <= 32: the raw-weight staging and unpack is shared
    // by two token groups (pp512 +1.5%); below it the 16-token tiles keep
    // the wave count up.  Tuning override: MVH_GEMM_TG2_ROWTILES.
    static const size_t tg2_min = [] {
        const char* e = getenv("MVH_GEMM_TG2_ROWTILES");
        return e ? static_cast<size_t>(atoll(e)) : static_cast<size_t>(512);
    }();
    // The workgroup kernel from rows x tokens = 768 K on: below, its 64 x 64
    // tiles leave CUs idle and a lone wave's chain sets the time (4096x4096 at
    // 128 tokens 27 against 21 us, 4096->11008 at 64 even at 27.5; 4096x4096 at
    // 256 29 against 37, 4096->11008 at 128 35 against 42, 4096->22016 at 64 34
    // against 42).  128-row x 32-token tiles where 64 would leave half of the
    // last ones empty.  Tuning override: MVH_GEMM_WG=0 never, 1 at every batch
    // size.
    static const int wg_mode = [] {
        const char* e = getenv("MVH_GEMM_WG");
        return e ? atoi(e) : -1;
    }();
    if (wg_mode == 1 || (wg_mode != 0 && rows * batch >= size_t{768} * 1024)) {
        if (g32 % 2) {
            const dim3 grid(static_cast<unsigned>((rows + 127) / 128), static_cast<unsigned>(g32));
            gemm_q4_0_q8_tile_kernel<1><<<grid, 256, 0, st>>>(W, aq, ad, y, N, nb, Bn);
        } else {
            const dim3 grid(static_cast<unsigned>((rows + 63) / 64), static_cast<unsigned>(g32 / 2));
            gemm_q4_0_q8_tile_kernel<2><<<grid, 256, 0, st>>>(W, aq, ad, y, N, nb, Bn);
        }
        return hipGetLastError();
    }
    // (17..32 tokens: the row-tile count alone decides -- the fused q|k|v's
    // 768 row tiles on 32-token tiles, pp512 11.84 -> 11.95-12.03 K tok/s;
    // up to 16 tokens a 32-token tile would be half empty)
    if (batch <= 32 ? batch <= 16 || gx < tg2_min : gx * g32 <= 1024) {
        if (gx * g16 <= 1024)
            gemm_q4_0_q8_mfma_kernel<1, 4><<<dim3(gx, static_cast<unsigned>(g16)), 64, 0, st>>>(W, aq, ad, y, N, nb, Bn);
        else
            gemm_q4_0_q8_mfma_kernel<1, 2><<<dim3(gx, static_cast<unsigned>(g16)), 64, 0, st>>>(W, aq, ad, y, N, nb, Bn);
    } else {
        gemm_q4_0_q8_mfma_kernel<2, 2><<<dim3(gx, static_cast<unsigned>(g32)), 64, 0, st>>>(W, aq, ad, y, N, nb, Bn);
    }
    return hipGetLastError();
}

}  // namespace mvh
