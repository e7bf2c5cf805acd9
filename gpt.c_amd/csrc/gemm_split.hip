// The Linear layers' products on gfx950: fp32 in, fp32 out, formed on the bf16
// matrix cores.  No counterpart in gpt.c, whose GEMMs are cuBLAS calls
// (kernels/src/cuda/Linear.cu:40-95).
//
// A float (from 2^-110 on) is the exact sum of three bf16 values (8 + 8 + 8
// significant bits, each part the rest rounded to nearest).  Of the nine products of two such
// sums, the six of relative order 2^0, 2^-8 and 2^-16 are formed; what is left
// out is at most 3 x 2^-26 of a product, under half a rounding of the fp32
// product.  A bf16 product is exact in the matrix core's fp32 sum, and
// v_mfma_f32_32x32x16_bf16 runs 16 times the rate of the fp32 instructions, so
// six of them take 6/16 of the time.
//
// Sums.  The matrix core drops bits below its accumulator towards minus
// infinity: chained over a long reduction that is a shift of every output, which
// a column sum over 8192 rows then shows 90 times larger (a bias gradient
// 1.5e-5 off, relative, against 1.6e-6 with fp32 instructions).  So each step of
// 32 terms sums its twelve products into a fresh accumulator, smallest first,
// and the step's sum is added to the tile with a rounded fp32 add; every
// second step forms -A B and is subtracted, which cancels what shift is
// left over pairs of steps; and odd rows and odd columns are formed negated (for
// free: the scale below takes their sign), so that what an odd last step leaves
// cancels in sums over the rows or the columns.  4096 x 1024 outputs, error of the
// column sums: K = 16 5.7e-7 without the rows' signs, K = 96 2.6e-7.
//
// Range.  bf16 ends at 2^-133, so the parts of a float below 2^-110 would lose its
// last bits.  Both operands are therefore split times 2^24 (exact: the last bit of
// the smallest normal float is 2^-149), and a step's sum comes back times 2^-48 in
// the add that takes it into the tile.  Floats of 2^104 and more, and sums of a step
// past 2^80, overflow on the way: those blocks are formed again in fp32.
//
// Relative error against 64 bits (2-norm, normal inputs), this kernel
// and rocBLAS's fp32 one: K = 768 1.0e-7 and 5.0e-7, 3072 1.9e-7 and 9.7e-7,
// 8192 3e-7 and 1.6e-6; mean error under 2e-9 at K = 768 and 3072.
//
// What bounds it: in a 128 x 128 tile's step a wave issues 48 matrix
// instructions (1536 cycles) and about 280 vector ones (1120 cycles: 6.5 a float
// for the scale and the split, 64 for the sums); counters at 2000 x 4000 x 1000 read the
// matrix cores 47 % busy (of their cycles, at the 2.1 GHz it runs at), the vector units 43 %,
// with no bank conflicts.  Moving the next step's split between this step's matrix
// instructions measured no faster (108.0 against 105.0 us there, before the scale), nor did
// 256 x 128 tiles (their accumulators spill); forming the parts' rests with
// v_dot2_f32_bf16 (exact, 215 vector instructions a step) is slower (block of 8 x 1024
// tokens, step 2.98 against 2.89 ms).  Times in us (GPT-2 small,
// 8192 rows; rocBLAS's own pick as its caller gets it, this): x W^T to 2304
// 229 / 202, to 3072 313 / 231, from 3072 to 768 276 / 251, lm_head 4300 / 3870;
// g W from 2304 225 / 197, from 50257 5800 / 4460; g^T x to 3072 x 768 450 / 250,
// to 768 x 768 116 / 77.  Without the scale these are 0 to 5 % less (lm_head 3780, g W from
// 50257 4240): a multiply of each float of the second operand.
#include <hip/hip_runtime.h>
#include <algorithm>
#include <cmath>
#include <cstdint>
#include <type_traits>
#include "gemm_split.hpp"
#include "gpu_kernels.h"
#include "hip_check.hpp"

namespace gptc {

namespace {

typedef float f32x2 __attribute__((ext_vector_type(2)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));

constexpr int kBK = 32;      // reduction terms per step
constexpr int kPlanes = 3;   // bf16 parts of a float
constexpr int kPad = 2;      // 16-byte chunks of padding per row of chunks
constexpr int kThreads = 256;
constexpr float kScale = 0x1p24f;      // of either operand as it is split
constexpr float kUnscale = 0x1p-48f;   // of a step's sum

template <int N>
using IntC = std::integral_constant<int, N>;

// The six products of bf16 parts of order 2^-16 and larger, the smallest first.
constexpr int kProd[6][2] = {{2, 0}, {0, 2}, {1, 1}, {1, 0}, {0, 1}, {0, 0}};

struct Args {
    const float *A, *B, *bias, *add;
    float *C;
    int M, N, K, lda, ldb, ldc;
    int tiles_m, tiles_n, slice_k;
    int64_t slice_c;  // floats between the slices' outputs
};

__device__ __forceinline__ uint32_t pack_bf16(float x, float y) {
    const f32x2 v = {x, y};
    return __builtin_bit_cast(uint32_t, __builtin_convertvector(v, bf16x2));
}
__device__ __forceinline__ float low_bf16(uint32_t p) { return __builtin_bit_cast(float, p << 16); }
__device__ __forceinline__ float high_bf16(uint32_t p) { return __builtin_bit_cast(float, p & 0xffff0000u); }

// x, y = sum of their three bf16 parts, exactly where their last bits are 2^-133 or more.
__device__ __forceinline__ void split2(float x, float y, uint32_t (&p)[kPlanes]) {
    p[0] = pack_bf16(x, y);
    const float x1 = x - low_bf16(p[0]), y1 = y - high_bf16(p[0]);
    p[1] = pack_bf16(x1, y1);
    p[2] = pack_bf16(x1 - low_bf16(p[1]), y1 - high_bf16(p[1]));
}

// A tile in LDS: 16-byte chunks of eight consecutive terms of one row, as a lane of
// the 32x32x16 instruction takes them, at [part][terms / 8][slot of the row].
// Reads take 32 consecutive slots; the slots' order and the padding of the
// chunk rows keep the stores, which run along the rows or across them, free of
// bank conflicts as well.
__device__ __forceinline__ int row_slot(int m) { return m ^ ((m >> 3) & 3); }

// Buffer loads: what lies past `floats` reads as zero, so a tile's ragged edge
// never reads outside its operand.  They need 4-byte alignment only.
using Rsrc = __amdgpu_buffer_rsrc_t;
__device__ __forceinline__ Rsrc make_rsrc(const float *p, int64_t floats) {
    int64_t bytes = floats * 4;
    if (bytes < 0) bytes = 0;
    if (bytes > 0xfffffffcll) bytes = 0xfffffffcll;
    const uint64_t a = reinterpret_cast<uint64_t>(p);
    const uint32_t lo = __builtin_amdgcn_readfirstlane(static_cast<uint32_t>(a));
    const uint32_t hi = __builtin_amdgcn_readfirstlane(static_cast<uint32_t>(a >> 32));
    const float *q = reinterpret_cast<const float *>((static_cast<uint64_t>(hi) << 32) | lo);
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<float *>(q), 0,
                                             __builtin_amdgcn_readfirstlane(static_cast<uint32_t>(bytes)), 0x00020000);
}
__device__ __forceinline__ f32x4 load4(Rsrc r, uint32_t off) {
    return __builtin_bit_cast(f32x4, __builtin_amdgcn_raw_buffer_load_b128(r, off * 4, 0, 0));
}
__device__ __forceinline__ f32x2 load2(Rsrc r, uint32_t off) {
    return __builtin_bit_cast(f32x2, __builtin_amdgcn_raw_buffer_load_b64(r, off * 4, 0, 0));
}

// One operand's tile: R rows (of M or N) x 32 reduction terms, from memory into
// registers and, a step later, in parts into LDS.  KC: the terms of a row lie
// together in memory (a thread takes eight of one row); else the rows of a term do
// (a thread takes four terms of MV rows, which makes the transposition a matter of
// register names).
template <int R, bool KC>
struct Operand {
    static constexpr int kRowChunks = R + kPad;
    static constexpr int kChunks = kPlanes * 4 * kRowChunks;  // 16-byte chunks of LDS
    static constexpr int MV = R >= 128 ? 4 : 2;
    static constexpr int kItems = KC ? R / 64 : (R >= 128 ? R / 128 : 1);
    static constexpr int kFloats = R * kBK / kThreads;
    float v[kFloats];

    // rows: rows of the operand from this tile's first on (a tile's rows past them
    // repeat the last one, or read on in memory: no output takes them); k0: first term.
    __device__ __forceinline__ void load(const float *base, int ld, int rows, int k0, int k_end, int tid) {
        if (KC) {
            const Rsrc r = make_rsrc(base + k0, static_cast<int64_t>(min(rows, R) - 1) * ld + (k_end - k0));
            const int kg = tid & 3;
#pragma unroll
            for (int i = 0; i < kItems; ++i) {
                const int row = min((tid >> 2) + 64 * i, rows - 1);
                const uint32_t off = static_cast<uint32_t>(row) * ld + 8 * kg;
#pragma unroll
                for (int j = 0; j < 2; ++j) {
                    const f32x4 x = load4(r, off + 4 * j);
#pragma unroll
                    for (int e = 0; e < 4; ++e) v[8 * i + 4 * j + e] = x[e];
                }
            }
        } else {
            const Rsrc r = make_rsrc(base + static_cast<int64_t>(k0) * ld,
                                     static_cast<int64_t>(min(k_end - k0, kBK) - 1) * ld + rows);
            const int lane = tid & 63, w = tid >> 6;
            const int k4 = 8 * w + 4 * (lane & 1);
#pragma unroll
            for (int i = 0; i < kItems; ++i) {
                const int m = MV * ((lane >> 1) + 32 * i);
#pragma unroll
                for (int k = 0; k < 4; ++k) {
                    const uint32_t off = static_cast<uint32_t>(k4 + k) * ld + m;
                    if (MV == 4) {
                        const f32x4 x = load4(r, off);
#pragma unroll
                        for (int e = 0; e < 4; ++e) v[16 * i + 4 * k + e] = x[e];
                    } else {
                        const f32x2 x = load2(r, off);
                        v[2 * k] = x[0];
                        v[2 * k + 1] = x[1];
                    }
                }
            }
        }
    }
    // Zeroes the terms at or past `left` (the last step of a ragged reduction).
    __device__ __forceinline__ void mask(int left, int tid) {
        if (KC) {
            const int kg = tid & 3;
#pragma unroll
            for (int i = 0; i < kItems; ++i)
#pragma unroll
                for (int e = 0; e < 8; ++e)
                    if (8 * kg + e >= left) v[8 * i + e] = 0.0f;
        } else {
            const int k4 = 8 * (tid >> 6) + 4 * (tid & 1);
#pragma unroll
            for (int i = 0; i < kItems; ++i)
#pragma unroll
                for (int k = 0; k < 4; ++k)
                    if (k4 + k >= left) {
#pragma unroll
                        for (int e = 0; e < MV; ++e) v[4 * MV * i + MV * k + e] = 0.0f;
                    }
        }
    }
    // scale: +-kScale, the step's sign in one operand; odd rows are stored negated
    __device__ __forceinline__ void store(u32x4 *lds, int tid, float scale) const {
        if (KC) {
            const int kg = tid & 3;
            if ((tid >> 2) & 1) scale = -scale;
#pragma unroll
            for (int i = 0; i < kItems; ++i) {
                const int row = (tid >> 2) + 64 * i;
                u32x4 c[kPlanes];
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    uint32_t p[kPlanes];
                    split2(scale * v[8 * i + 2 * e], scale * v[8 * i + 2 * e + 1], p);
#pragma unroll
                    for (int q = 0; q < kPlanes; ++q) c[q][e] = p[q];
                }
#pragma unroll
                for (int q = 0; q < kPlanes; ++q) lds[(4 * q + kg) * kRowChunks + row_slot(row)] = c[q];
            }
        } else {
            const int lane = tid & 63, kg = tid >> 6;
            u32x2 *half = reinterpret_cast<u32x2 *>(lds);
#pragma unroll
            for (int i = 0; i < kItems; ++i)
#pragma unroll
                for (int e = 0; e < MV; ++e) {
                    const int m = MV * ((lane >> 1) + 32 * i) + e;
                    const float *x = v + 4 * MV * i + e;
                    const float f = e & 1 ? -scale : scale;
                    uint32_t a[kPlanes], b[kPlanes];
                    split2(f * x[0], f * x[MV], a);
                    split2(f * x[2 * MV], f * x[3 * MV], b);
#pragma unroll
                    for (int q = 0; q < kPlanes; ++q)
                        half[2 * ((4 * q + kg) * kRowChunks + row_slot(m)) + (lane & 1)] = u32x2{a[q], b[q]};
                }
        }
    }
};

__device__ __forceinline__ f32x16 zero16() {
    f32x16 z;
#pragma unroll
    for (int r = 0; r < 16; ++r) z[r] = 0.0f;
    return z;
}
__device__ __forceinline__ f32x16 mfma(u32x4 a, u32x4 b, f32x16 c) {
    return __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, a), __builtin_bit_cast(bf16x8, b), c, 0,
                                                   0, 0);
}

// An infinity (or a float or a step's sum that the scale takes past the largest)
// splits into inf - inf: a block that is not finite is formed again from the
// floats themselves.  Ab, Bb: the operands from the tile's first row
// on; m, n: the block's first row and column in the tile.
template <bool TA, bool TB>
__device__ __forceinline__ void redo_if_not_finite(const Args &a, const float *Ab, const float *Bb, int m, int n,
                                                   int rows_a, int rows_b, int k_begin, int k_end, f32x16 &acc) {
    float z = 0.0f;
#pragma unroll
    for (int r = 0; r < 16; ++r) z = fmaf(acc[r], 0.0f, z);
    if (__builtin_amdgcn_ballot_w64(z != 0.0f) == 0) return;  // NaN compares unequal
    const int l32 = threadIdx.x & 31, hf = (threadIdx.x >> 5) & 1;
    const int row = min(m + l32, rows_a - 1), col = min(n + l32, rows_b - 1);
    const float *ap = Ab + (TA ? row : static_cast<int64_t>(row) * a.lda);
    const float *bp = Bb + (TB ? static_cast<int64_t>(col) * a.ldb : col);
    const int64_t sa = TA ? a.lda : 1, sb = TB ? 1 : a.ldb;
#pragma unroll
    for (int r = 0; r < 16; ++r) acc[r] = 0.0f;
    for (int k = k_begin; k < k_end; k += 2) {
        const bool ok = k + hf < k_end;
        const float x = ok ? ap[(k + hf) * sa] : 0.0f, y = ok ? bp[(k + hf) * sb] : 0.0f;
        acc = __builtin_amdgcn_mfma_f32_32x32x2f32(x, y, acc, 0, 0, 0);
    }
}

// C = block (+ bias) (+ add); m, n: its first row and column of C.
__device__ __forceinline__ void store_block(const Args &a, float *C, int m, int n, const f32x16 &acc) {
    const int l32 = threadIdx.x & 31, hf = (threadIdx.x >> 5) & 1;
    n += l32;
    if (n >= a.N) return;
    const float bias = a.bias != nullptr ? a.bias[n] : 0.0f;
    float old[16];
    if (a.add != nullptr) {
#pragma unroll
        for (int r = 0; r < 16; ++r) {
            const int row = min(m + 8 * (r >> 2) + 4 * hf + (r & 3), a.M - 1);
            old[r] = a.add[static_cast<int64_t>(row) * a.ldc + n];
        }
    }
#pragma unroll
    for (int r = 0; r < 16; ++r) {
        const int row = m + 8 * (r >> 2) + 4 * hf + (r & 3);
        float v = acc[r] + bias;
        if (a.add != nullptr) v += old[r];
        if (row < a.M) C[static_cast<int64_t>(row) * a.ldc + n] = v;
    }
}

// One BM x BN tile of C per workgroup (blockIdx.y: one slice of the reduction),
// four waves in a 2 x 2 grid on its quarters.  DEPTH: steps the loads run
// ahead; the other workgroups of a CU work while one waits at a barrier.
template <int BM, int BN, bool TA, bool TB, int WAVES, int DEPTH>
__global__ __launch_bounds__(kThreads) __attribute__((amdgpu_waves_per_eu(WAVES, WAVES))) void
split_gemm_kernel(const Args a) {
    using OpA = Operand<BM, !TA>;
    using OpB = Operand<BN, TB>;
    constexpr int NM = BM / 64, NN = BN / 64;  // 32 x 32 blocks of a wave's tile
    __shared__ u32x4 lds[OpA::kChunks + OpB::kChunks];
    u32x4 *a_lds = lds, *b_lds = lds + OpA::kChunks;
    const int tid = threadIdx.x, lane = tid & 63;
    const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int l32 = lane & 31, hf = lane >> 5;

    const int n_tiles = a.tiles_m * a.tiles_n;
    const int slice = blockIdx.y;
    // Tiles in 8 contiguous ranges, one per XCD (workgroup i runs on XCD i % 8).
    int t = blockIdx.x;
    {
        const int x = t & 7, q = n_tiles >> 3, r = n_tiles & 7;
        t = (t >> 3) + x * q + min(x, r);
    }
    // Columns of 8 row tiles: the tiles that run together share rows and columns.
    int tm, tn;
    {
        const int G = 8, per = G * a.tiles_n;
        const int g = t / per, first = g * G, h = min(G, a.tiles_m - first);
        const int in = t - g * per;
        tm = first + in % h;
        tn = in / h;
    }
    const int m0 = tm * BM, n0 = tn * BN;
    const int k_begin = slice * a.slice_k, k_end = min(a.K, k_begin + a.slice_k);

    const float *Ab = a.A + (TA ? static_cast<int64_t>(m0) : static_cast<int64_t>(m0) * a.lda);
    const float *Bb = a.B + (TB ? static_cast<int64_t>(n0) * a.ldb : static_cast<int64_t>(n0));
    const int rows_a = a.M - m0, rows_b = a.N - n0;

    OpA pa[DEPTH];
    OpB pb[DEPTH];
    f32x16 acc[NM][NN];
#pragma unroll
    for (int i = 0; i < NM; ++i)
#pragma unroll
        for (int j = 0; j < NN; ++j)
#pragma unroll
            for (int r = 0; r < 16; ++r) acc[i][j][r] = 0.0f;

#pragma unroll
    for (int d = 0; d < DEPTH; ++d) {
        pa[d].load(Ab, a.lda, rows_a, k_begin + d * kBK, k_end, tid);
        pb[d].load(Bb, a.ldb, rows_b, k_begin + d * kBK, k_end, tid);
    }
    const int wm = (w >> 1) * (BM / 2), wn = (w & 1) * (BN / 2);
    const float col_unscale = lane & 1 ? -kUnscale : kUnscale;  // a block's column l32, rows of the parity of r
    const int slot = l32 ^ ((l32 >> 3) & 3);
    float sign = 1.0f;
    for (int k0 = k_begin; k0 < k_end; k0 += DEPTH * kBK) {
#pragma unroll
        for (int d = 0; d < DEPTH; ++d) {
            const int kd = k0 + d * kBK;
            if (d > 0 && kd >= k_end) break;
            if (k_end - kd < kBK) {
                pa[d].mask(k_end - kd, tid);
                pb[d].mask(k_end - kd, tid);
            }
            __syncthreads();
            pa[d].store(a_lds, tid, sign * kScale);
            pb[d].store(b_lds, tid, kScale);
            __syncthreads();
            // Past the end these read nothing (or terms that no step uses).
            pa[d].load(Ab, a.lda, rows_a, kd + DEPTH * kBK, k_end, tid);
            pb[d].load(Bb, a.ldb, rows_b, kd + DEPTH * kBK, k_end, tid);
            const float back = sign * col_unscale;
            u32x4 fb[NN][2][kPlanes];
#pragma unroll
            for (int j = 0; j < NN; ++j)
#pragma unroll
                for (int s = 0; s < 2; ++s)
#pragma unroll
                    for (int q = 0; q < kPlanes; ++q)
                        fb[j][s][q] = b_lds[(4 * q + 2 * s + hf) * OpB::kRowChunks + wn + 32 * j + slot];
#pragma unroll
            for (int i = 0; i < NM; ++i) {
                u32x4 fa[2][kPlanes];
#pragma unroll
                for (int s = 0; s < 2; ++s)
#pragma unroll
                    for (int q = 0; q < kPlanes; ++q)
                        fa[s][q] = a_lds[(4 * q + 2 * s + hf) * OpA::kRowChunks + wm + 32 * i + slot];
                f32x16 t[NN];
#pragma unroll
                for (int j = 0; j < NN; ++j) t[j] = zero16();
#pragma unroll
                for (int p = 0; p < 6; ++p)
#pragma unroll
                    for (int s = 0; s < 2; ++s)
#pragma unroll
                        for (int j = 0; j < NN; ++j) t[j] = mfma(fa[s][kProd[p][0]], fb[j][s][kProd[p][1]], t[j]);
#pragma unroll
                for (int j = 0; j < NN; ++j)
#pragma unroll
                    for (int r = 0; r < 16; ++r) acc[i][j][r] = fmaf(r & 1 ? -back : back, t[j][r], acc[i][j][r]);
            }
            sign = -sign;
        }
    }

#pragma unroll
    for (int i = 0; i < NM; ++i)
#pragma unroll
        for (int j = 0; j < NN; ++j) {
            redo_if_not_finite<TA, TB>(a, Ab, Bb, wm + 32 * i, wn + 32 * j, rows_a, rows_b, k_begin, k_end, acc[i][j]);
            store_block(a, a.C + slice * a.slice_c, m0 + wm + 32 * i, n0 + wn + 32 * j, acc[i][j]);
        }
}

// Small products: one 64 x 64 tile per workgroup, the reduction dealt to its
// eight waves in steps of 16 terms.  Each wave forms the whole tile over its
// terms from its own part of LDS, so the loop has no barriers; the waves'
// sums meet in LDS at the end, in wave order.
constexpr int NW = 8;            // waves
constexpr int kWK = 16;           // terms per step of a wave
constexpr int kWRows = 64 + 4;    // 16-byte chunks per row of chunks, padded
constexpr int kWChunks = kPlanes * 2 * kWRows;

template <bool KC>
struct WaveOperand {
    float v[16];

    __device__ __forceinline__ void load(const float *base, int ld, int rows, int k0, int k_end, int lane) {
        if (KC) {  // rows lane / 4 + 16 i, terms 4 (lane % 4) ..
            const Rsrc r = make_rsrc(base + k0, static_cast<int64_t>(min(rows, 64) - 1) * ld + (k_end - k0));
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const f32x4 x = load4(r, static_cast<uint32_t>(min((lane >> 2) + 16 * i, rows - 1)) * ld + 4 * (lane & 3));
#pragma unroll
                for (int e = 0; e < 4; ++e) v[4 * i + e] = x[e];
            }
        } else {  // terms 8 (lane / 32) + 4 (lane % 2) + i, rows 4 (lane / 2 % 16) ..
            const Rsrc r = make_rsrc(base + static_cast<int64_t>(k0) * ld,
                                     static_cast<int64_t>(min(k_end - k0, kWK) - 1) * ld + rows);
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const f32x4 x = load4(r, static_cast<uint32_t>(8 * (lane >> 5) + 4 * (lane & 1) + i) * ld +
                                             4 * ((lane >> 1) & 15));
#pragma unroll
                for (int e = 0; e < 4; ++e) v[4 * i + e] = x[e];
            }
        }
    }
    __device__ __forceinline__ void mask(int left, int lane) {
#pragma unroll
        for (int i = 0; i < 4; ++i)
#pragma unroll
            for (int e = 0; e < 4; ++e)
                if ((KC ? 4 * (lane & 3) + e : 8 * (lane >> 5) + 4 * (lane & 1) + i) >= left) v[4 * i + e] = 0.0f;
    }
    __device__ __forceinline__ void store(u32x2 *lds, int lane, float scale) const {
        const int kg = KC ? (lane >> 1) & 1 : lane >> 5, half = lane & 1;
        if (KC && ((lane >> 2) & 1)) scale = -scale;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const int m = KC ? (lane >> 2) + 16 * i : 4 * ((lane >> 1) & 15) + i;
            const float f = !KC && (i & 1) ? -scale : scale;
            uint32_t a[kPlanes], b[kPlanes];
            split2(f * (KC ? v[4 * i] : v[i]), f * (KC ? v[4 * i + 1] : v[4 + i]), a);
            split2(f * (KC ? v[4 * i + 2] : v[8 + i]), f * (KC ? v[4 * i + 3] : v[12 + i]), b);
#pragma unroll
            for (int q = 0; q < kPlanes; ++q)
                lds[2 * ((2 * q + kg) * kWRows + row_slot(m)) + half] = u32x2{a[q], b[q]};
        }
    }
};

template <bool TA, bool TB>
__global__ __launch_bounds__(64 * NW) __attribute__((amdgpu_waves_per_eu(2, 2))) void split_gemm_small_kernel(
    const Args a) {
    constexpr int kStage = NW * 2 * kWChunks, kSums = 4 * 4 * 4 * 64;  // 16-byte chunks
    __shared__ u32x4 lds[kStage > kSums ? kStage : kSums];
    const int lane = threadIdx.x & 63, l32 = lane & 31, hf = lane >> 5;
    const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int tm = blockIdx.x % a.tiles_m, tn = blockIdx.x / a.tiles_m;
    const int slice = blockIdx.y;
    const int m0 = tm * 64, n0 = tn * 64;
    const int k_begin = slice * a.slice_k, k_end = min(a.K, k_begin + a.slice_k);
    const float *Ab = a.A + (TA ? static_cast<int64_t>(m0) : static_cast<int64_t>(m0) * a.lda);
    const float *Bb = a.B + (TB ? static_cast<int64_t>(n0) * a.ldb : static_cast<int64_t>(n0));
    const int rows_a = a.M - m0, rows_b = a.N - n0;
    u32x4 *a_lds = lds + w * 2 * kWChunks, *b_lds = a_lds + kWChunks;
    float sign = (w & 1) != 0 ? -1.0f : 1.0f;
    const float col_unscale = lane & 1 ? -kUnscale : kUnscale;

    f32x16 acc[2][2];
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int r = 0; r < 16; ++r) acc[i >> 1][i & 1][r] = 0.0f;
    constexpr int kDepth = 2;
    WaveOperand<!TA> pa[kDepth];
    WaveOperand<TB> pb[kDepth];
    const int k_first = k_begin + kWK * w;
#pragma unroll
    for (int d = 0; d < kDepth; ++d) {
        // Past the end these read nothing (or terms that no step uses).
        const int k = min(k_first + d * NW * kWK, k_end);
        pa[d].load(Ab, a.lda, rows_a, k, k_end, lane);
        pb[d].load(Bb, a.ldb, rows_b, k, k_end, lane);
    }
    const int slot = l32 ^ ((l32 >> 3) & 3);
    for (int k0 = k_first; k0 < k_end; k0 += kDepth * NW * kWK) {
#pragma unroll
        for (int d = 0; d < kDepth; ++d) {
            const int kd = k0 + d * NW * kWK;
            if (d > 0 && kd >= k_end) break;
            if (k_end - kd < kWK) {
                pa[d].mask(k_end - kd, lane);
                pb[d].mask(k_end - kd, lane);
            }
            pa[d].store(reinterpret_cast<u32x2 *>(a_lds), lane, sign * kScale);
            pb[d].store(reinterpret_cast<u32x2 *>(b_lds), lane, kScale);
            const int next = min(kd + kDepth * NW * kWK, k_end);
            pa[d].load(Ab, a.lda, rows_a, next, k_end, lane);
            pb[d].load(Bb, a.ldb, rows_b, next, k_end, lane);
            // The wave's own LDS accesses stay in order; the fences keep the compiler's.
            __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
            __builtin_amdgcn_wave_barrier();
            __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
            const float back = sign * col_unscale;
            u32x4 fa[2][kPlanes], fb[2][kPlanes];
#pragma unroll
            for (int i = 0; i < 2; ++i)
#pragma unroll
                for (int q = 0; q < kPlanes; ++q) {
                    fa[i][q] = a_lds[(2 * q + hf) * kWRows + 32 * i + slot];
                    fb[i][q] = b_lds[(2 * q + hf) * kWRows + 32 * i + slot];
                }
            __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
            __builtin_amdgcn_wave_barrier();
            __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
#pragma unroll
            for (int i = 0; i < 2; ++i) {
                f32x16 t[2] = {zero16(), zero16()};
#pragma unroll
                for (int p = 0; p < 6; ++p)
#pragma unroll
                    for (int j = 0; j < 2; ++j) t[j] = mfma(fa[i][kProd[p][0]], fb[j][kProd[p][1]], t[j]);
#pragma unroll
                for (int j = 0; j < 2; ++j)
#pragma unroll
                    for (int r = 0; r < 16; ++r) acc[i][j][r] = fmaf(r & 1 ? -back : back, t[j][r], acc[i][j][r]);
            }
            sign = -sign;
        }
    }
    // The upper half of the waves hands its sums to the lower half, then wave
    // w < 4 adds up block w.
    auto at = [&](int wave, int b, int r) -> f32x4 & {
        return reinterpret_cast<f32x4 *>(lds)[((wave * 4 + b) * 4 + r) * 64 + lane];
    };
    auto put = [&](int wave) {
#pragma unroll
        for (int b = 0; b < 4; ++b)
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const f32x16 &s = acc[b >> 1][b & 1];
                at(wave, b, r) = f32x4{s[4 * r], s[4 * r + 1], s[4 * r + 2], s[4 * r + 3]};
            }
    };
    __syncthreads();
    if (w >= 4) put(w - 4);
    __syncthreads();
    if (w >= 4) return;
#pragma unroll
    for (int b = 0; b < 4; ++b)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const f32x4 v = at(w, b, r);
#pragma unroll
            for (int e = 0; e < 4; ++e) acc[b >> 1][b & 1][4 * r + e] += v[e];
        }
    put(w);  // over what this wave alone has read
    __syncthreads();
    f32x16 sum;
#pragma unroll
    for (int r = 0; r < 4; ++r) {
        f32x4 v = at(0, w, r);
#pragma unroll
        for (int k = 1; k < 4; ++k) v += at(k, w, r);
#pragma unroll
        for (int e = 0; e < 4; ++e) sum[4 * r + e] = v[e];
    }
    const int m = 32 * (w >> 1), n = 32 * (w & 1);
    if (m >= rows_a || n >= rows_b) return;
    redo_if_not_finite<TA, TB>(a, Ab, Bb, m, n, rows_a, rows_b, k_begin, k_end, sum);
    store_block(a, a.C + slice * a.slice_c, m0 + m, n0 + n, sum);
}

// C = the slices' sums in slice order (+ bias) (+ add); the slices are (M x N)
// without gaps, C and add have rows of ldc.
template <typename V>
__global__ __launch_bounds__(kThreads) void split_reduce_kernel(const float *part, const float *bias, const float *add,
                                                                float *C, int64_t n, int cols, int ldc, int S) {
    constexpr int W = sizeof(V) / sizeof(float);
    const int64_t stride = static_cast<int64_t>(gridDim.x) * kThreads;
    const int cw = cols / W;
    for (int64_t i = blockIdx.x * kThreads + threadIdx.x; i < n / W; i += stride) {
        const int64_t m = i / cw;
        const int c = static_cast<int>(i - m * cw);
        V v = reinterpret_cast<const V *>(part)[i];
        for (int s = 1; s < S; ++s) v += reinterpret_cast<const V *>(part + s * n)[i];
        if (bias != nullptr) v += reinterpret_cast<const V *>(bias)[c];
        const int64_t at = (m * ldc) / W + c;
        if (add != nullptr) v += reinterpret_cast<const V *>(add)[at];
        reinterpret_cast<V *>(C)[at] = v;
    }
}

// The tiles the kernels are built for, with their measured cost per step of 32
// terms (us): alone on a CU, each of several on one CU, and each with every CU
// full; tn: the factor on these when both operands lie along M and N.  The plan
// with the smallest estimate runs: at the sizes above and 24 others, 4 x 1000 x 500
// to 8192 x 50257 x 768, it is within 10 % of the best of all tiles and slice
// counts (small ones under 20 us: within 1.5 us).
struct Tile {
    int bm, bn, resident;
    float alone, shared, full, tn;
};
constexpr Tile kTiles[] = {
    {128, 128, 2, 1.75f, 1.28f, 1.45f, 1.00f},
    {128, 64, 3, 1.20f, 0.79f, 0.79f, 1.05f},
    {64, 64, 4, 0.80f, 0.45f, 0.42f, 1.35f},
};
// Products of fewer multiply-adds without a bias or residual stay with rocBLAS, whose small
// fp32 tiles start up faster (us, here / rocBLAS: x W^T 300 x 512 x 512 11 / 8.5, 512 x 768 x 768
// 14.6 / 8.8; both gradients of the latter 28 / 21).  From here on to about 2e9
// rocBLAS is still up to 1.4 times as fast (1024 x 768 x 768 18 / 14, 2496 x 768 x 768 31 / 24; level at
// 3328 x 768 x 768, 1.96e9), but its chained sums are five times as far off (5e-7 against
// 1e-7, relative), so the line is not drawn there.  With a bias its second launch costs
// about what the start gains (x W^T + b: 512 x 768 x 768 14.5 / 12.4, 64 x 768 x 2304 11.8 / 16.9,
// 8192 x 64 x 64 5.9 / 8.8), so those run here at any size.
constexpr double kLibraryMacs = 6e8;
// rocBLAS does not split the reduction of an A without transposition: from 4096 terms on its
// chain is the time, whatever the outputs (g W, 8 x 64 outputs, here / rocBLAS: 4096 terms 14 / 25,
// 8192 17 / 451, 50257 33 / 2726; 128 x 256: 18 / 20, 21 / 444; at 2304 terms 8 x 768 12 / 12).
constexpr int kLibraryTerms = 4096;
constexpr int kSmallTile = 3;  // the 64 x 64 tile of eight independent waves

constexpr int kMaxSlices = 32;

struct Plan {
    int tile, slices, slice_k;
};

// Estimated time of a plan in us.
float plan_us(int tile, const SplitGemm &g, int S) {
    const int bm = tile < kSmallTile ? kTiles[tile].bm : 64, bn = tile < kSmallTile ? kTiles[tile].bn : 64;
    const int64_t units = static_cast<int64_t>((g.M + bm - 1) / bm) * ((g.N + bn - 1) / bn) * S;
    const int64_t per_cu = (units + 255) / 256;
    const int steps = (g.K + kBK - 1) / kBK, mine = (steps + S - 1) / S;
    float us;
    if (tile == kSmallTile) {  // one workgroup per CU; a round is four steps
        us = 2.5f + per_cu * (5.0f + 1.65f * ((mine + 3) / 4));
    } else {
        const Tile &t = kTiles[tile];
        const float step = std::max({t.alone * ((per_cu + t.resident - 1) / t.resident), t.shared * per_cu,
                                     t.full * (units / 256.0f)});
        us = 2.5f + (mine + 2.5f) * step * (g.trans_a ? t.tn : 1.0f);
    }
    // The slices' sums go out and come back: bytes at 4.5 TB/s and a launch.
    return S == 1 ? us : us + 4.0f + 0.1f * S + (S + 2) * (static_cast<float>(g.M) * g.N * 4e-6f / 4.5f);
}

Plan choose(const SplitGemm &g, int max_slices) {
    const int steps = (g.K + kBK - 1) / kBK;
    Plan best{0, 1, 0};
    float best_us = INFINITY;
    for (int t = 0; t <= kSmallTile; ++t)
        for (int S = 1; S <= max_slices && S <= steps; ++S) {
            const float us = plan_us(t, g, S);
            if (us < best_us) {
                best_us = us;
                best.tile = t;
                best.slices = S;
            }
        }
    best.slice_k = (steps + best.slices - 1) / best.slices * kBK;
    best.slices = (g.K + best.slice_k - 1) / best.slice_k;
    return best;
}

template <int BM, int BN, int WAVES, int DEPTH>
void run_tile(const SplitGemm &g, Args a, int slices, hipStream_t stream) {
    a.tiles_m = (g.M + BM - 1) / BM;
    a.tiles_n = (g.N + BN - 1) / BN;
    const dim3 grid(a.tiles_m * a.tiles_n, slices);
    if (!g.trans_a && g.trans_b)
        split_gemm_kernel<BM, BN, false, true, WAVES, DEPTH><<<grid, dim3(kThreads), 0, stream>>>(a);
    else if (!g.trans_a)
        split_gemm_kernel<BM, BN, false, false, WAVES, DEPTH><<<grid, dim3(kThreads), 0, stream>>>(a);
    else
        split_gemm_kernel<BM, BN, true, false, WAVES, DEPTH><<<grid, dim3(kThreads), 0, stream>>>(a);
    hipCheck(hipGetLastError());
}

void run_small(const SplitGemm &g, Args a, int slices, hipStream_t stream) {
    a.tiles_m = (g.M + 63) / 64;
    a.tiles_n = (g.N + 63) / 64;
    const dim3 grid(a.tiles_m * a.tiles_n, slices), block(64 * NW);
    if (!g.trans_a && g.trans_b)
        split_gemm_small_kernel<false, true><<<grid, block, 0, stream>>>(a);
    else if (!g.trans_a)
        split_gemm_small_kernel<false, false><<<grid, block, 0, stream>>>(a);
    else
        split_gemm_small_kernel<true, false><<<grid, block, 0, stream>>>(a);
    hipCheck(hipGetLastError());
}

bool aligned16(const void *p) { return (reinterpret_cast<uintptr_t>(p) & 15) == 0; }

}  // namespace

void launch_sum_slices(const float *part, const float *bias, const float *add, float *C, int M, int N, int ldc, int S,
                       hipStream_t stream) {
    const int64_t n = static_cast<int64_t>(M) * N;
    const bool vec = N % 4 == 0 && ldc % 4 == 0 && aligned16(C) && aligned16(add) && aligned16(bias);
    const int64_t items = vec ? n / 4 : n;
    const int blocks = static_cast<int>(std::min<int64_t>((items + kThreads - 1) / kThreads, 256 * 8));
    if (vec)
        split_reduce_kernel<f32x4><<<dim3(blocks), dim3(kThreads), 0, stream>>>(part, bias, add, C, n, N, ldc, S);
    else
        split_reduce_kernel<float><<<dim3(blocks), dim3(kThreads), 0, stream>>>(part, bias, add, C, n, N, ldc, S);
    hipCheck(hipGetLastError());
}

namespace {

void run_plan(const SplitGemm &g, const Plan &p, hipStream_t s) {
    const int64_t n = static_cast<int64_t>(g.M) * g.N;
    float *part = nullptr;
    Args a{g.A, g.B, g.bias, g.add, g.C, g.M, g.N, g.K, g.lda, g.ldb, g.ldc, 0, 0, p.slice_k, 0};
    if (p.slices > 1) {
        part = static_cast<float *>(alloc_cuda(static_cast<size_t>(n) * p.slices * sizeof(float)));
        a.bias = a.add = nullptr;
        a.C = part;
        a.ldc = g.N;
        a.slice_c = n;
    }
    switch (p.tile) {
        case 0: run_tile<128, 128, 2, 1>(g, a, p.slices, s); break;
        case 1: run_tile<128, 64, 3, 1>(g, a, p.slices, s); break;
        case 2: run_tile<64, 64, 4, 2>(g, a, p.slices, s); break;
        default: run_small(g, a, p.slices, s); break;
    }
    if (p.slices == 1) return;
    launch_sum_slices(part, g.bias, g.add, g.C, g.M, g.N, g.ldc, p.slices, s);
    free_cuda(part);
}

}  // namespace

bool split_gemm_serves(const SplitGemm &g) {
    constexpr int kMaxLd = 1 << 22;  // a tile's offsets (128 rows) fit 32 bits
    if (g.M <= 0 || g.N <= 0 || g.K <= 0 || (g.trans_a && g.trans_b) || g.lda >= kMaxLd || g.ldb >= kMaxLd) return false;
    const double macs = static_cast<double>(g.M) * g.N * g.K;
    return g.bias != nullptr || (g.add != nullptr && g.add != g.C) || macs >= kLibraryMacs ||
           (!g.trans_a && g.K >= kLibraryTerms);
}

void launch_split_gemm(const SplitGemm &g, hipStream_t stream) {
    Plan p = choose(g, kMaxSlices);
    if (p.slices > 1 && gptc_stream_capturing()) p = choose(g, 1);
    run_plan(g, p, stream);
}

}  // namespace gptc
