// Slab kernels of the causal attention: forward and backward for problems whose
// work is too small, or whose heads are too few, for the kernels on 64- and
// 128-row blocks (the same mathematics, kernels/src/cpu/Attention.c:46-301; head
// sizes up to 128, multiples of 4, 16-byte rows).
//
// Those kernels walk a block's key tiles one after the other; with few heads
// that chain is the time while most of the chip idles (15 heads of T = 333: forward
// 24 us, dk/dv 28, for 4 us of matrix work).  Here a slab of 16 or 32 rows is a
// workgroup, and its four waves deal the row blocks on the other side among
// themselves, each from its own loads straight into registers (no staging, no
// barrier in the loop), and join their partial results in LDS at the end, in wave
// order: results do not depend on scheduling.
//
// The backward is one launch.  Half of its workgroups form dQ of a slab of queries,
// half dK and dV of a slab of keys; both recompute P from the log-sum-exp and
// delta = rowsum(dO o O) from the rows at hand: seven products instead of four,
// but no chain of three launches and no P' or dS through memory.  The longest slabs
// come first.  (The forward still writes P' and its maxima: a backward that
// these kernels do not serve reads them.)
//
// fp32 on v_mfma_f32_16x16x4_f32 throughout, operand layouts as in
// attn_common.hpp.  What bounds them: in the backward a wave loads 20 rows of 1 KB
// for 128 matrix instructions (4096 cycles) at 64 dims, and the row loads (16
// rows x 64 bytes an instruction) keep the CU's load unit about as busy as the matrix
// cores are; two row blocks per wave halve that (12 heads T = 1024: 89 -> 72 us).
// Times (us, whole steps, before / here): B = 2 H = 4 T = 100 38.4 / 13.6, B = 3 H = 5
// T = 333 64.7 / 32.6, B = 2 H = 8 T = 1024 D = 128 486 / 290, B = 1 H = 12 T = 1024
// forward 56.1 / 31.2.
#include <algorithm>

#include "attn_common.hpp"
#include "attn_kernels.hpp"
#include "hip_check.hpp"

namespace gptc {

namespace {

constexpr int kBlock = 16;     // rows of a block
constexpr int kSlabWaves = 4;  // waves of a workgroup
constexpr uint32_t kNoDim = 0x80000000u;  // an offset past every head's rows: reads as zero

// Rows [0, T) of one head; rows past them and dims at or past D read as zeros.
// A block is 16 rows; DP: the padded head size.
template <int DP>
struct HeadRows {
    static constexpr int NC = DP / 16, NE = DP / 64;
    __amdgpu_buffer_rsrc_t rsrc;
    uint32_t st;
    int D;

    __device__ __forceinline__ HeadRows(const float *base, int T, uint32_t stride, int dims) : st(stride), D(dims) {
        const int bytes = static_cast<int>(uniform(((T - 1) * stride + dims) * 4u));
        rsrc = __builtin_amdgcn_make_buffer_rsrc(const_cast<float *>(uniform(base)), 0, bytes, kBufferConfig);
    }
    // x[c] = row r0 + i16, dims 16c + 4g ..: an operand that reduces over dims.
    __device__ __forceinline__ void by_row(int r0, int g, int i16, f32x4 (&x)[NC]) const {
        const uint32_t row = static_cast<uint32_t>(r0 + i16) * st;
#pragma unroll
        for (int c = 0; c < NC; ++c) {
            const int dim = 16 * c + 4 * g;
            x[c] = buffer_load4(rsrc, dim < D ? row + dim : kNoDim / 4);
        }
    }
    // x[r][e] = row r0 + 4g + r, dims 64e + 4 i16 ..: an operand that reduces over rows.
    __device__ __forceinline__ void by_dim(int r0, int g, int i16, f32x4 (&x)[4][NE]) const {
#pragma unroll
        for (int r = 0; r < 4; ++r)
#pragma unroll
            for (int e = 0; e < NE; ++e) {
                const int dim = 64 * e + 4 * i16;
                x[r][e] = buffer_load4(rsrc, dim < D ? static_cast<uint32_t>(r0 + 4 * g + r) * st + dim : kNoDim / 4);
            }
    }
};

__device__ __forceinline__ f32x4 at4(const float *p) { return *reinterpret_cast<const f32x4 *>(p); }

// The wave's accumulators of a slab, X^T in 16 x 16 blocks (acc[i][b][r] = X[row 16i + i16]
// [64 (b / 4) + 16g + 4r + b % 4]), to LDS, [wave][i][block][lane].
template <int R, int NB>
__device__ __forceinline__ void put_sums(f32x4 (*lds)[R][NB][64], int w, int lane, const f32x4 (&acc)[R][NB]) {
#pragma unroll
    for (int i = 0; i < R; ++i)
#pragma unroll
        for (int b = 0; b < NB; ++b) lds[w][i][b][lane] = acc[i][b];
}
// X[row 16i + i16][64e + 16g + 4r ..]: the waves' sums in wave order, times f[wave].
template <int R, int NB>
__device__ __forceinline__ f32x4 take_sums(const f32x4 (*lds)[R][NB][64], int i, int e, int r, int lane,
                                           const f32x4 &f) {
    f32x4 v = zero4();
#pragma unroll
    for (int k = 0; k < kSlabWaves; ++k)
#pragma unroll
        for (int b = 0; b < 4; ++b) v[b] += f[k] * lds[k][i][4 * e + b][lane][r];
    return v;
}

// x . b of row i16 of a block (b: the head's values of one bias), on every lane of the row's
// column; D = 64 NC / 4 only.
template <int NC>
__device__ __forceinline__ float dot_bias(const f32x4 (&x)[NC], const float *b, int g) {
    float s = 0.0f;
#pragma unroll
    for (int c = 0; c < NC; ++c) {
        const f32x4 v = at4(b + 16 * c + 4 * g);
#pragma unroll
        for (int e = 0; e < 4; ++e) s = fmaf(x[c][e], v[e], s);
    }
    return sum4_rows(s);
}

// y, the log-sum-exp, P' and m of R blocks of queries; wave w takes the 64-key tiles
// w, w + 4, ...  DP: the padded head size; BIAS: the qkv bias is added here.  It joins the
// slab's own rows only: (q + qb) . (k + kb) starts from the row's (q + qb) . kb, and the
// probabilities' sum of v + vb is that of v, and vb.
template <int DP, int R, bool BIAS>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(DP == 64 ? 2 : 1, DP == 64 ? 2 : 1))) void
attn_fwd_slab_kernel(const FwdParams a) {
    constexpr int NC = DP / 16, NB = DP / 16, NE = DP / 64;
    __shared__ __attribute__((aligned(16))) f32x4 sums[kSlabWaves][R][NB][64];
    __shared__ float stat[2][kSlabWaves][R][kBlock];
    const int tid = threadIdx.x, lane = tid & 63, g = lane >> 4, i16 = lane & 15;
    const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int BH = a.B * a.H, T = a.T, D = a.D;
    const int rank = static_cast<int>(blockIdx.x) / BH, bh = static_cast<int>(blockIdx.x) - rank * BH;
    const int b = bh / a.H, h = bh - b * a.H;
    const int q0 = ((T + R * kBlock - 1) / (R * kBlock) - 1 - rank) * R * kBlock;  // the longest slabs first
    const int jq = q0 >> 6;  // the slab's own 64-key tile
    // The backward on 128-key blocks reads P' in halves of 32 queries that start before T, rows
    // past T included: a last slab that ends in the middle of a half writes zeros to the rest of it.
    const bool fill_half = ((q0 + R * kBlock) & 31) != 0 && q0 + R * kBlock >= T;

    const HeadRows<DP> q_rows(a.q.p + b * a.q.sb + h * a.q.sh, T, a.q.st, D);
    const HeadRows<DP> k_rows(a.k.p + b * a.k.sb + h * a.k.sh, T, a.k.st, D);
    const HeadRows<DP> v_rows(a.v.p + b * a.v.sb + h * a.v.sh, T, a.v.st, D);
    f32x4 qr[R][NC], acc[R][NB];
    float m_run[R], l_run[R], s0[R];
#pragma unroll
    for (int i = 0; i < R; ++i) {
        q_rows.by_row(q0 + kBlock * i, g, i16, qr[i]);
        if (BIAS) {
#pragma unroll
            for (int c = 0; c < NC; ++c) qr[i][c] += at4(a.qb + h * D + 16 * c + 4 * g);
        }
        s0[i] = BIAS ? dot_bias(qr[i], a.kb + h * D, g) : 0.0f;
#pragma unroll
        for (int n = 0; n < NB; ++n) acc[i][n] = zero4();
        m_run[i] = -INFINITY;
        l_run[i] = 0.0f;
    }
    const float c2 = a.scale_log2;

    for (int kt = w; kt <= jq; kt += kSlabWaves) {
        f32x4 kr[4][NC], vr[4][4][NE];
#pragma unroll
        for (int kb = 0; kb < 4; ++kb) k_rows.by_row(64 * kt + kBlock * kb, g, i16, kr[kb]);
#pragma unroll
        for (int kb = 0; kb < 4; ++kb) v_rows.by_dim(64 * kt + kBlock * kb, g, i16, vr[kb]);
        f32x4 sc[R][4];
#pragma unroll
        for (int i = 0; i < R; ++i)
#pragma unroll
            for (int kb = 0; kb < 4; ++kb) sc[i][kb] = f32x4{s0[i], s0[i], s0[i], s0[i]};
#pragma unroll
        for (int c = 0; c < NC; ++c)
#pragma unroll
            for (int e = 0; e < 4; ++e)
#pragma unroll
                for (int i = 0; i < R; ++i)
#pragma unroll
                    for (int kb = 0; kb < 4; ++kb) sc[i][kb] = mfma16(kr[kb][c][e], qr[i][c][e], sc[i][kb]);
#pragma unroll
        for (int i = 0; i < R; ++i) {
            const int my_q = q0 + kBlock * i + i16;
            if (kt == jq) {
#pragma unroll
                for (int kb = 0; kb < 4; ++kb)
#pragma unroll
                    for (int r = 0; r < 4; ++r)
                        if (64 * kt + kBlock * kb + 4 * g + r > my_q) sc[i][kb][r] = -INFINITY;
            }
            float mx = -INFINITY;
#pragma unroll
            for (int kb = 0; kb < 4; ++kb)
                mx = fmaxf(mx, fmaxf(fmaxf(sc[i][kb][0], sc[i][kb][1]), fmaxf(sc[i][kb][2], sc[i][kb][3])));
            const float m_new = fmaxf(m_run[i], max4_rows(mx) * c2);
            const float m_use = (m_new == -INFINITY) ? 0.0f : m_new;
            const float alpha = fast_exp2(m_run[i] - m_use);
            l_run[i] *= alpha;
#pragma unroll
            for (int n = 0; n < NB; ++n) acc[i][n] *= alpha;
            m_run[i] = m_new;
            float ls[2] = {0.0f, 0.0f};
#pragma unroll
            for (int kb = 0; kb < 4; ++kb)
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    const float p = fast_exp2(fmaf(sc[i][kb][r], c2, -m_use));
                    sc[i][kb][r] = p;
                    ls[r & 1] += p;
                }
            l_run[i] += ls[0] + ls[1];
            if (a.pp != nullptr) {
                float *ptile = a.pp + ds_block_offset(bh, a.nqt, jq, 2 * kt);  // uniform
                const uint32_t prow = ((q0 & 63) + kBlock * i + i16) * 32 + 4 * g;
#pragma unroll
                for (int kb = 0; kb < 4; ++kb)
                    stream_store(reinterpret_cast<f32x4 *>(ptile + (kb >> 1) * kDsBlock + prow + 16 * (kb & 1)),
                                 sc[i][kb]);
                if (i == R - 1 && fill_half) {
#pragma unroll
                    for (int kb = 0; kb < 4; ++kb)
                        stream_store(reinterpret_cast<f32x4 *>(ptile + (kb >> 1) * kDsBlock + prow + kBlock * 32 +
                                                               16 * (kb & 1)),
                                     zero4());
                }
                if (g == 0 && my_q < T) a.pm[(static_cast<uint32_t>(bh) * a.nqt + kt) * T + my_q] = m_use;
            }
        }
#pragma unroll
        for (int kb = 0; kb < 4; ++kb)
#pragma unroll
            for (int r = 0; r < 4; ++r)
#pragma unroll
                for (int e = 0; e < NE; ++e)
#pragma unroll
                    for (int i = 0; i < R; ++i)
#pragma unroll
                        for (int n = 0; n < 4; ++n)
                            acc[i][4 * e + n] = mfma16(vr[kb][r][e][n], sc[i][kb][r], acc[i][4 * e + n]);
    }

    put_sums<R, NB>(sums, w, lane, acc);
#pragma unroll
    for (int i = 0; i < R; ++i) {
        const float l_tot = sum4_rows(l_run[i]);
        if (g == 0) {
            stat[0][w][i][i16] = m_run[i];
            stat[1][w][i][i16] = l_tot;
        }
    }
    __syncthreads();
#pragma unroll
    for (int i = 0; i < R; ++i) {
        const int my_q = q0 + kBlock * i + i16;
        if (my_q >= T) return;
        // Wave 0 always has a key of the row, so m is finite.
        float m = stat[0][0][i][i16], l = 0.0f;
#pragma unroll
        for (int k = 1; k < kSlabWaves; ++k) m = fmaxf(m, stat[0][k][i][i16]);
        f32x4 f;
#pragma unroll
        for (int k = 0; k < kSlabWaves; ++k) {
            f[k] = fast_exp2(stat[0][k][i][i16] - m);
            l += stat[1][k][i][i16] * f[k];
        }
        const float inv = 1.0f / l;
#pragma unroll
        for (int e = 0; e < NE; ++e) {
            const int dim = 64 * e + 16 * g + 4 * w;
            if (dim >= D) continue;
            f32x4 v = take_sums<R, NB>(sums, i, e, w, lane, f) * inv;
            if (BIAS) v += at4(a.vb + h * D + dim);
            const size_t at = b * a.o.sb + static_cast<size_t>(my_q) * a.o.st + h * a.o.sh + dim;
            *reinterpret_cast<f32x4 *>(a.o.p + at) = v;
            if (a.o2 != nullptr) *reinterpret_cast<f32x4 *>(a.o2 + at) = v;
        }
        if (w == 0 && g == 0) a.lse[static_cast<uint32_t>(bh) * T + my_q] = (m + log2f(l)) * kLn2;
    }
}

// One output slab (rows row0 .. of dQ, dK or dV): the waves' sums times scale into
// rows of `out`, and with `part` their column sums.
template <int DP, int R>
__device__ __forceinline__ void store_slab(const f32x4 (*sums)[R][DP / 16][64], int w, int lane, float scale,
                                           const HeadViewW &out, int b, int h, int row0, int T, int D, float *part) {
    const int g = lane >> 4, i16 = lane & 15;
#pragma unroll
    for (int e = 0; e < DP / 64; ++e) {
        const int dim = 64 * e + 16 * g + 4 * w;
        if (dim >= D) continue;  // D < DP only without `part`, whose sums need every lane
        f32x4 cs = zero4();
#pragma unroll
        for (int i = 0; i < R; ++i) {
            const f32x4 v = take_sums<R, DP / 16>(sums, i, e, w, lane, f32x4{scale, scale, scale, scale});
            const int row = row0 + kBlock * i + i16;
            if (row < T) {
                *reinterpret_cast<f32x4 *>(out.p + b * out.sb + static_cast<size_t>(row) * out.st + h * out.sh + dim) =
                    v;
                cs += v;
            }
        }
        if (part != nullptr) {
#pragma unroll
            for (int off = 1; off < 16; off <<= 1)
#pragma unroll
                for (int n = 0; n < 4; ++n) cs[n] += __shfl_xor(cs[n], off, 64);
            if (i16 == 0) *reinterpret_cast<f32x4 *>(part + dim) = cs;
        }
    }
}

// BIAS: the qkv bias joins the slab's own rows only.  The products with the rows that stream by
// start from the slab rows' products with their bias; dQ needs no k bias (a row of dS sums to
// zero), and dK takes the q bias times the key's sum of dS at the end.  So the form with
// the bias keeps the other's registers (adding the bias to the rows as they came spilled 14 of
// them; us with its column sums' launch, then / now / without bias: 12 heads T = 1024 89 / 78 / 72, 3 heads
// T = 2048 147 / 118 / 111; forward of the same 36.6 / 32.7 / 32.5, 42 / 36 / 36).
template <int DP, int R, bool BIAS>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(DP == 64 ? 2 : 1, DP == 64 ? 2 : 1))) void
attn_bwd_slab_kernel(const BwdParams a) {
    constexpr int NC = DP / 16, NB = DP / 16, NE = DP / 64;
    __shared__ __attribute__((aligned(16))) f32x4 sums[kSlabWaves][R][NB][64];
    const int tid = threadIdx.x, lane = tid & 63, g = lane >> 4, i16 = lane & 15;
    const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int BH = a.B * a.H, T = a.T, D = a.D;
    const int n_slabs = (T + R * kBlock - 1) / (R * kBlock), n_blocks = (T + kBlock - 1) / kBlock;
    const int rank = static_cast<int>(blockIdx.x) / BH, bh = static_cast<int>(blockIdx.x) - rank * BH;
    const int b = bh / a.H, h = bh - b * a.H;
    const HeadRows<DP> q_rows(a.q.p + b * a.q.sb + h * a.q.sh, T, a.q.st, D);
    const HeadRows<DP> k_rows(a.k.p + b * a.k.sb + h * a.k.sh, T, a.k.st, D);
    const HeadRows<DP> v_rows(a.v.p + b * a.v.sb + h * a.v.sh, T, a.v.st, D);
    const HeadRows<DP> o_rows(a.o.p + b * a.o.sb + h * a.o.sh, T, a.o.st, D);
    const HeadRows<DP> do_rows(a.dout.p + b * a.dout.sb + h * a.dout.sh, T, a.dout.st, D);
    const float *lse_h = a.lse + static_cast<uint32_t>(bh) * T;
    const float c2 = a.scale * kLog2e;
    auto bias1 = [&](const float *p, f32x4 (&x)[NC]) {
        if (BIAS) {
#pragma unroll
            for (int c = 0; c < NC; ++c) x[c] += at4(p + h * D + 16 * c + 4 * g);
        }
    };
    // rowsum(dO o O) of row i16 of a block, on every lane of the row's column.
    auto delta_of = [&](const f32x4 (&x)[NC], const f32x4 (&y)[NC]) {
        float s = 0.0f;
#pragma unroll
        for (int c = 0; c < NC; ++c)
#pragma unroll
            for (int e = 0; e < 4; ++e) s = fmaf(x[c][e], y[c][e], s);
        return sum4_rows(s);
    };
    float *part = nullptr;

    if ((rank & 1) != 0) {
        // dQ of the slab's queries (lane: query i16 of each block); the waves
        // deal the key blocks up to the slab's last among themselves.
        const int slab = n_slabs - 1 - (rank >> 1), q0 = R * kBlock * slab;
        const int last = min(R * slab + R, n_blocks) - 1;
        f32x4 qr[R][NC], dor[R][NC], acc[R][NB];
        float dl[R], lse2[R], s0[R];
#pragma unroll
        for (int i = 0; i < R; ++i) {
            const int row = q0 + kBlock * i;
            q_rows.by_row(row, g, i16, qr[i]);
            do_rows.by_row(row, g, i16, dor[i]);
            f32x4 orow[NC];
            o_rows.by_row(row, g, i16, orow);
            dl[i] = delta_of(orow, dor[i]);
            bias1(a.qb, qr[i]);
            s0[i] = 0.0f;
            if (BIAS) {
                s0[i] = dot_bias(qr[i], a.kb + h * D, g);
                dl[i] -= dot_bias(dor[i], a.vb + h * D, g);
            }
            // Rows past T: P = 0 (their dO rows are zero too).
            lse2[i] = row + i16 < T ? lse_h[min(row + i16, T - 1)] * kLog2e : INFINITY;
#pragma unroll
            for (int n = 0; n < NB; ++n) acc[i][n] = zero4();
        }
        f32x4 k1[NC], v1[NC];
        if (w <= last) {
            k_rows.by_row(kBlock * w, g, i16, k1);
            v_rows.by_row(kBlock * w, g, i16, v1);
        }
        for (int kb = w; kb <= last; kb += kSlabWaves) {
            f32x4 k2[4][NE];
            k_rows.by_dim(kBlock * kb, g, i16, k2);
            f32x4 sc[R], dp[R];
#pragma unroll
            for (int i = 0; i < R; ++i) {
                sc[i] = f32x4{s0[i], s0[i], s0[i], s0[i]};
                dp[i] = zero4();
            }
#pragma unroll
            for (int c = 0; c < NC; ++c)
#pragma unroll
                for (int e = 0; e < 4; ++e)
#pragma unroll
                    for (int i = 0; i < R; ++i) {
                        sc[i] = mfma16(k1[c][e], qr[i][c][e], sc[i]);
                        dp[i] = mfma16(v1[c][e], dor[i][c][e], dp[i]);
                    }
            // The next block's rows (past the slab: rows that no step uses).
            k_rows.by_row(kBlock * (kb + kSlabWaves), g, i16, k1);
            v_rows.by_row(kBlock * (kb + kSlabWaves), g, i16, v1);
#pragma unroll
            for (int i = 0; i < R; ++i)
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    float p = fast_exp2(fmaf(sc[i][r], c2, -lse2[i]));
                    if (kBlock * kb + 4 * g + r > q0 + kBlock * i + i16) p = 0.0f;
                    sc[i][r] = p * (dp[i][r] - dl[i]);
                }
#pragma unroll
            for (int r = 0; r < 4; ++r)
#pragma unroll
                for (int i = 0; i < R; ++i)
#pragma unroll
                    for (int n = 0; n < NB; ++n) acc[i][n] = mfma16(k2[r][n >> 2][n & 3], sc[i][r], acc[i][n]);
        }
        put_sums<R, NB>(sums, w, lane, acc);
        __syncthreads();
        if (a.db != nullptr) part = a.dbq_part + (static_cast<size_t>(b) * n_slabs + slab) * 3 * a.C + h * D;
        store_slab<DP, R>(sums, w, lane, a.scale, a.dq, b, h, q0, T, D, part);
        return;
    }
    // dK, dV of the slab's keys (lane: key i16 of each block) over the query
    // blocks from the slab's first on.
    const int slab = rank >> 1, k0 = R * kBlock * slab;
    f32x4 kr[R][NC], vr[R][NC], acc_k[R][NB], acc_v[R][NB];
    float s0[R], ds_sum[R];  // BIAS: the keys' (k + kb) . qb, and this lane's part of their sums of dS
#pragma unroll
    for (int i = 0; i < R; ++i) {
        k_rows.by_row(k0 + kBlock * i, g, i16, kr[i]);
        v_rows.by_row(k0 + kBlock * i, g, i16, vr[i]);
        bias1(a.kb, kr[i]);
        bias1(a.vb, vr[i]);
        s0[i] = BIAS ? dot_bias(kr[i], a.qb + h * D, g) : 0.0f;
        ds_sum[i] = 0.0f;
#pragma unroll
        for (int n = 0; n < NB; ++n) acc_k[i][n] = acc_v[i][n] = zero4();
    }
    f32x4 q1[NC], do1[NC];
    const int first = R * slab + w;
    if (first < n_blocks) {
        q_rows.by_row(kBlock * first, g, i16, q1);
        do_rows.by_row(kBlock * first, g, i16, do1);
    }
    for (int qb = first; qb < n_blocks; qb += kSlabWaves) {
        const int q0 = kBlock * qb;
        f32x4 q2[4][NE], do2[4][NE], o1[NC];
        o_rows.by_row(q0, g, i16, o1);
        float lse2[4], dl[4];
#pragma unroll
        for (int r = 0; r < 4; ++r) lse2[r] = lse_h[min(q0 + 4 * g + r, T - 1)];
        do_rows.by_dim(q0, g, i16, do2);
        q_rows.by_dim(q0, g, i16, q2);
        f32x4 sc[R], dp[R];
#pragma unroll
        for (int i = 0; i < R; ++i) {
            sc[i] = f32x4{s0[i], s0[i], s0[i], s0[i]};
            dp[i] = zero4();
        }
#pragma unroll
        for (int c = 0; c < NC; ++c)
#pragma unroll
            for (int e = 0; e < 4; ++e)
#pragma unroll
                for (int i = 0; i < R; ++i) {
                    sc[i] = mfma16(q1[c][e], kr[i][c][e], sc[i]);
                    dp[i] = mfma16(do1[c][e], vr[i][c][e], dp[i]);
                }
        const float d1 = delta_of(o1, do1);
        q_rows.by_row(kBlock * (qb + kSlabWaves), g, i16, q1);
        do_rows.by_row(kBlock * (qb + kSlabWaves), g, i16, do1);
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            dl[r] = __shfl(d1, 4 * g + r, 64);
            lse2[r] = q0 + 4 * g + r < T ? lse2[r] * kLog2e : INFINITY;  // rows past T: P = 0
        }
#pragma unroll
        for (int i = 0; i < R; ++i)
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                float p = fast_exp2(fmaf(sc[i][r], c2, -lse2[r]));
                if (k0 + kBlock * i + i16 > q0 + 4 * g + r) p = 0.0f;
                sc[i][r] = p;
                dp[i][r] = p * (dp[i][r] - dl[r]);
                if (BIAS) ds_sum[i] += dp[i][r];
            }
#pragma unroll
        for (int r = 0; r < 4; ++r)
#pragma unroll
            for (int i = 0; i < R; ++i)
#pragma unroll
                for (int n = 0; n < NB; ++n) {
                    acc_v[i][n] = mfma16(do2[r][n >> 2][n & 3], sc[i][r], acc_v[i][n]);
                    acc_k[i][n] = mfma16(q2[r][n >> 2][n & 3], dp[i][r], acc_k[i][n]);
                }
    }
    if (a.db != nullptr) part = a.dbq_part + (static_cast<size_t>(b) * n_slabs + slab) * 3 * a.C + a.C + h * D;
    if (BIAS) {
#pragma unroll
        for (int i = 0; i < R; ++i) {
            const float s = sum4_rows(ds_sum[i]);
#pragma unroll
            for (int e = 0; e < NE; ++e)
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    const f32x4 qb4 = at4(a.qb + h * D + 64 * e + 16 * g + 4 * r);
#pragma unroll
                    for (int n = 0; n < 4; ++n) acc_k[i][4 * e + n][r] = fmaf(s, qb4[n], acc_k[i][4 * e + n][r]);
                }
        }
    }
    put_sums<R, NB>(sums, w, lane, acc_k);
    __syncthreads();
    store_slab<DP, R>(sums, w, lane, a.scale, a.dk, b, h, k0, T, D, part);
    __syncthreads();
    put_sums<R, NB>(sums, w, lane, acc_v);
    __syncthreads();
    store_slab<DP, R>(sums, w, lane, 1.0f, a.dv, b, h, k0, T, D, part != nullptr ? part + a.C : nullptr);
}

// Every head's rows within the 31 bits of a buffer's offsets.
bool rows_fit(int T, int D, std::initializer_list<uint32_t> strides) {
    for (uint32_t st : strides)
        if ((static_cast<int64_t>(T + 6 * kBlock) * st + D) * 4 >= (1LL << 31)) return false;
    return true;
}

}  // namespace

namespace {

// The rule that picks the slab kernels, from times measured on the MI355X (us).
// tiles = B H nqt (nqt + 1) / 2, the 64 x 64 tiles below the diagonals.  The
// slabs' time is fixed + per tile (their waves are many and short, so the sum of the
// work sets it), with one or two blocks of rows per wave: two load half as much
// per product, one makes twice the workgroups (r2_from: the tiles from which
// two are faster).  The kernels on work lists and 128-row blocks take their
// longest chain, chain0 + chain nqt, or the sum of the work, sum0 + sum tiles.
struct SlabTimes {
    float fixed, one, two, r2_from;
    float chain0, chain, sum0, sum;
};
// Forward, head sizes up to 64: 64 itself, and the others against the 32-row kernel.
// Slab / other at 12 heads of 64: B = 1 T = 1024 31.2 / 56.1, B = 2 50 / 56, B = 8
// T = 256 24 / 17; 48 dims B = 2 T = 1024 47.6 / 95.6, 32 dims 64 heads T = 1024 110 / 107.
constexpr SlabTimes kFwd64{9, 12.5e-3f, 12.5e-3f, 1e9f, 2, 3.4f, 4, 9.4e-3f};
constexpr SlabTimes kFwd32{9, 12.0e-3f, 12.0e-3f, 1e9f, 4, 5.8f, 4, 12.0e-3f};
// Up to 128 dims: 16 heads of 128, T = 1024 62 / 155, 32 heads 124 / 156, 64 heads 245 / 183.
constexpr SlabTimes kFwd128{6, 33e-3f, 26.5e-3f, 1000, 3, 9.6f, 4, 20.6e-3f};
// Backward: 12 heads of 64, T = 1024 72 / 98, 24 heads 130 / 100; T = 600, 24 heads 58 / 66;
// T = 200, 48 heads 28 / 33; 15 heads T = 333 20 / 41; T = 256, 96 heads 54 / 49.
constexpr SlabTimes kBwd64{8, 52e-3f, 41e-3f, 350, 18, 5.0f, 10, 19.5e-3f};
// 48 dims, 24 heads T = 1024 125 / 184; 32 dims, 96 heads T = 200 39 / 49, 64 heads T = 1024 290 / 235.
constexpr SlabTimes kBwd32{8, 42e-3f, 38e-3f, 350, 8, 10.5f, 10, 26e-3f};
// 16 heads of 128, T = 1024 230 / 330, 32 heads 409 / 339; 80 dims, 32 heads T = 300 59 / 107.
constexpr SlabTimes kBwd128{12, 110e-3f, 96e-3f, 250, 8, 20.0f, 10, 46e-3f};

double tiles_of(int B, int H, int nqt) { return 0.5 * B * H * nqt * (nqt + 1); }

bool slab_wins(const SlabTimes &t, double tiles, int nqt) {
    const double slab = t.fixed + tiles * (tiles < t.r2_from ? t.one : t.two);
    return slab < std::max<double>(t.chain0 + t.chain * nqt, t.sum0 + t.sum * tiles);
}

int blocks_per_slab(const BwdParams &p) {
    const SlabTimes &t = p.D > kDPad ? kBwd128 : p.D == kDPad ? kBwd64 : kBwd32;
    return tiles_of(p.B, p.H, p.nqt) < t.r2_from ? 1 : 2;
}

template <int R>
void run_fwd(const FwdParams &p, hipStream_t stream) {
    const dim3 grid((p.T + R * kBlock - 1) / (R * kBlock) * p.B * p.H), block(64 * kSlabWaves);
    if (p.D > kDPad)
        attn_fwd_slab_kernel<2 * kDPad, R, false><<<grid, block, 0, stream>>>(p);
    else if constexpr (R == 1) {
        if (p.kb != nullptr)
            attn_fwd_slab_kernel<kDPad, R, true><<<grid, block, 0, stream>>>(p);
        else
            attn_fwd_slab_kernel<kDPad, R, false><<<grid, block, 0, stream>>>(p);
    }
    hipCheck(hipGetLastError());
}

template <int R>
void run_bwd(const BwdParams &p, hipStream_t stream) {
    const dim3 grid(2 * ((p.T + R * kBlock - 1) / (R * kBlock)) * p.B * p.H), block(64 * kSlabWaves);
    if (p.D > kDPad)
        attn_bwd_slab_kernel<2 * kDPad, R, false><<<grid, block, 0, stream>>>(p);
    else if (p.kb != nullptr)
        attn_bwd_slab_kernel<kDPad, R, true><<<grid, block, 0, stream>>>(p);
    else
        attn_bwd_slab_kernel<kDPad, R, false><<<grid, block, 0, stream>>>(p);
    hipCheck(hipGetLastError());
}

}  // namespace

bool fwd_slab(const FwdParams &p) {
    if (!p.vec || p.qp != nullptr || p.D > 2 * kDPad || !rows_fit(p.T, p.D, {p.q.st, p.k.st, p.v.st})) return false;
    if (p.D == kDPad && p.nqt <= kShortHeadTiles) return false;  // the short-head kernels
    return slab_wins(p.D > kDPad ? kFwd128 : p.D == kDPad ? kFwd64 : kFwd32, tiles_of(p.B, p.H, p.nqt), p.nqt);
}

bool bwd_slab(const BwdParams &p) {
    if (!p.vec || p.D > 2 * kDPad || !rows_fit(p.T, p.D, {p.q.st, p.k.st, p.v.st, p.o.st, p.dout.st})) return false;
    const double tiles = tiles_of(p.B, p.H, p.nqt);
    // Short heads of 64: the recomputing dk/dv kernel runs a workgroup per head, about 30 us a round of 256
    // (96 heads: T = 128 26 / 36, T = 60 14 / 25; 8 heads T = 100 8 / 32; 200 heads T = 128 56 / 45).
    if (p.D == kDPad && p.nqt <= kShortHeadTiles) return 8 + 62.5e-3 * tiles < 30.0 * ((p.B * p.H + 255) / 256);
    return slab_wins(p.D > kDPad ? kBwd128 : p.D == kDPad ? kBwd64 : kBwd32, tiles, p.nqt);
}

int slab_count(const BwdParams &p) {
    const int rows = blocks_per_slab(p) * kBlock;
    return (p.T + rows - 1) / rows;
}

void launch_attn_fwd_slab(const FwdParams &p, hipStream_t stream) {
    if (p.D > kDPad && tiles_of(p.B, p.H, p.nqt) >= kFwd128.r2_from)
        run_fwd<2>(p, stream);
    else
        run_fwd<1>(p, stream);
}

void launch_attn_bwd_slab(const BwdParams &p, hipStream_t stream) {
    if (blocks_per_slab(p) == 1)
        run_bwd<1>(p, stream);
    else
        run_bwd<2>(p, stream);
}

}  // namespace gptc
