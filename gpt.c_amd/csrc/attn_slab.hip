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
// come first.  (The forward still writes P' and its maxima, up to the last slab's
// end: a backward that these kernels do not serve reads them.)
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
#include <cmath>

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

// The rule that picks the slab kernels, from times measured on the MI355X (us; 1128 cases
// of each direction, up to 22000 tiles, head sizes 32, 48, 64, 96 and 128, T = 16 to 2048, both sides
// forced, heads of 64 with and without the bias).
// tiles = B H nqt (nqt + 1) / 2, the 64 x 64 tiles below the diagonals.
//
// The slabs' workgroups come in rounds of 256 times the resident ones; a last round that
// is partly empty costs `tail` of what is missing in it.  A workgroup takes as many steps of its four
// waves as it has blocks on the other side, on average (blocks + 4) / 8: `one` us a step with
// one block of rows per wave, start2 + `two` with two, which load half as much per product where
// one makes twice the workgroups (r2_from: the tiles from which two are faster).  The
// kernels on work lists and 128-row blocks take their longest chain, chain0 + chain nqt, or the
// sum of the work, sum0 + sum tiles.
//
// Against the faster of the two at each shape the rule loses 0.4 % on average in the forward and 0.1 % in
// the backward; a rule on tiles alone lost 1.3 and 0.8 %, and up to 55 % where the last round of
// workgroups is nearly empty (130 heads of 128 T = 256 78 / 51).  Where it picks the slabs they are at most
// 3 % slower but for 48 dims: forward 95 to 114 heads T = 333 to 384 5 and 6 %, backward 256 heads T = 64 24.9 / 22.6; and
// 128 dims, backward 57 heads T = 333 134 / 128 us.
struct SlabTimes {
    float fixed, one, start2, two, tail;
    int resident;
    float r2_from;
    float per_tile;  // with every CU busy to the end: no less than fixed + this a tile
    float chain0, chain, sum0, sum;
};
// Slab / other: 12 heads of 64 B = 1 T = 1024 32 / 56, 24 heads 52 / 57, 33 heads 84 / 62, 20 heads T = 640 24 / 36,
// 48 heads T = 256 17 / 17.
constexpr SlabTimes kFwd64{4.4f, 6.8f, 0, 0, 0.45f, 2, 1e9f, 15.0e-3f, 1.55f, 3.71f, 6.2f, 10.8e-3f};
// 48 dims 24 heads T = 1024 51 / 96, 66 heads 166 / 127; 120 heads T = 200 24 / 26, 220 heads 39 / 35.
constexpr SlabTimes kFwd32{2.07f, 6.0f, 0, 0, 0.634f, 2, 1e9f, 14.0e-3f, 3.0f, 5.85f, 8.18f, 12.8e-3f};
// 16 heads of 128, T = 1024 65 / 155, 33 heads 156 / 158, 48 heads 191 / 166; 120 heads T = 200 55 / 44.
constexpr SlabTimes kFwd128{3.23f, 8.29f, 0.545f, 13.0f, 0.729f, 1, 1000, 28.5e-3f, 4.61f, 9.49f, 13.8f, 27.0e-3f};
// 9 heads of 64 T = 1024 70 / 97, 16 heads 104 / 98; 22 heads T = 640 60 / 66; 57 heads T = 333 56 / 48; with the bias
// 16 heads T = 1024 109 / 111.
constexpr SlabTimes kBwd64{11.2f, 3.56f, 4.1f, 4.74f, 0.502f, 2, 350, 35.0e-3f, 21.4f, 4.83f, 27.3f, 21.2e-3f};
// 48 dims 33 heads T = 1024 163 / 212, 48 heads 247 / 230; 57 heads T = 333 47 / 71, 152 heads 122 / 102.
constexpr SlabTimes kBwd32{4.41f, 4.15f, 3.87f, 3.91f, 0.573f, 2, 350, 32.0e-3f, 6.31f, 12.2f, 14.6f, 25.2e-3f};
// 16 heads of 128 T = 1024 229 / 330, 33 heads 445 / 340; 40 heads T = 640 239 / 218.
constexpr SlabTimes kBwd128{4.18f, 5.71f, 5.63f, 5.8f, 0.714f, 1, 250, 89.0e-3f, 0.04f, 20.4f, 30.0f, 59.7e-3f};
// Heads of 64 up to 128 rows, against the recomputing dk/dv kernel (short_heads_us):
// 96 heads T = 128 26 / 36, 160 heads 39 / 38; 240 heads T = 64 27 / 25; 270 heads T = 65 39 / 52.
constexpr SlabTimes kBwdShort{4.0f, 5.7f, 6.5f, 4.4f, 0.5f, 2, 350, 0, 0, 0, 0, 0};

double tiles_of(int B, int H, int nqt) { return 0.5 * B * H * nqt * (nqt + 1); }

const SlabTimes &fwd_times(int D) { return D > kDPad ? kFwd128 : D == kDPad ? kFwd64 : kFwd32; }
const SlabTimes &bwd_times(int D) { return D > kDPad ? kBwd128 : D == kDPad ? kBwd64 : kBwd32; }

int blocks_per_slab(const SlabTimes &t, int B, int H, int nqt) { return tiles_of(B, H, nqt) < t.r2_from ? 1 : 2; }

// slabs: of one head (and kind); wg: workgroups a slab, one in the forward, two in the backward;
// blocks: on the other side of the last slab (64 keys in the forward, 16 rows in the backward).
double slab_us(const SlabTimes &t, int R, double slabs, int wg, int heads, int blocks, double tiles) {
    const double rounds = wg * slabs * heads / (256.0 * t.resident);
    const double steps = std::max(1.0, blocks / 8.0 + 0.5);
    const double round = R == 1 ? t.one * steps : t.start2 + t.two * steps;
    return t.fixed + std::max((rounds + t.tail * (std::ceil(rounds) - rounds)) * round, t.per_tile * tiles);
}

double tiled_us(const SlabTimes &t, double tiles, int nqt) {
    return std::max<double>(t.chain0 + t.chain * nqt, t.sum0 + t.sum * tiles);
}

// The recomputing dk/dv kernel runs a workgroup per head, in rounds of 256: T = 16 17, 40 22, 64 24, 65 28, 100 35,
// 128 36 us, two rounds 25 to 67.
double short_heads_us(int T, int heads) {
    return (14.5 + 2.75 * ((T + kBlock - 1) / kBlock)) * (0.25 + 0.75 * ((heads + 255) / 256));
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
    const SlabTimes &t = fwd_times(p.D);
    const int R = blocks_per_slab(t, p.B, p.H, p.nqt), slabs = (p.T + R * kBlock - 1) / (R * kBlock);
    const double tiles = tiles_of(p.B, p.H, p.nqt);
    return slab_us(t, R, slabs, 1, p.B * p.H, p.nqt, tiles) < tiled_us(t, tiles, p.nqt);
}

bool bwd_slab(const BwdParams &p) {
    if (!p.vec || p.D > 2 * kDPad || !rows_fit(p.T, p.D, {p.q.st, p.k.st, p.v.st, p.o.st, p.dout.st})) return false;
    const SlabTimes &t = bwd_times(p.D);
    const int R = blocks_per_slab(t, p.B, p.H, p.nqt), heads = p.B * p.H, blocks = (p.T + kBlock - 1) / kBlock;
    const double tiles = tiles_of(p.B, p.H, p.nqt);
    if (p.D == kDPad && p.nqt <= kShortHeadTiles)  // few blocks: the last slab's empty half counts
        return slab_us(kBwdShort, R, static_cast<double>(blocks) / R, 2, heads, blocks, tiles) <
               short_heads_us(p.T, heads);
    return slab_us(t, R, (blocks + R - 1) / R, 2, heads, blocks, tiles) < tiled_us(t, tiles, p.nqt);
}

int slab_count(const BwdParams &p) {
    const int rows = blocks_per_slab(bwd_times(p.D), p.B, p.H, p.nqt) * kBlock;
    return (p.T + rows - 1) / rows;
}

void launch_attn_fwd_slab(const FwdParams &p, hipStream_t stream) {
    if (p.D > kDPad && blocks_per_slab(fwd_times(p.D), p.B, p.H, p.nqt) == 2)
        run_fwd<2>(p, stream);
    else
        run_fwd<1>(p, stream);
}

void launch_attn_bwd_slab(const BwdParams &p, hipStream_t stream) {
    if (blocks_per_slab(bwd_times(p.D), p.B, p.H, p.nqt) == 1)
        run_bwd<1>(p, stream);
    else
        run_bwd<2>(p, stream);
}

}  // namespace gptc
