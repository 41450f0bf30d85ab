// norm.hip -- the LayerNorm that precedes the MoE block in TMT, as part of
// the block (tmt-cuda/src/norm.cu:8-106; caller tmt-cuda/src/model.cu:509-514,
// 678-680).
//
//   ln_fwd      H = bf16(((x - mean) * rstd) * gamma + beta), one wave per row,
//               in the canonical order of ln_row.hpp, which the CPU oracle
//               restates (the reference's block tree and rsqrtf are not
//               reproducible, this order is). H is therefore bit-identical to
//               the oracle's, and so are the router logits computed from it.
//               For routed batches the router computes the same rows itself
//               (router.hip) and this kernel is not launched.
//   ln_bwd      dS = rstd * ((g - mean(g)) - xh * mean(g * xh)) with g = dH * gamma,
//               xh = (x - mean) * rstd, one wave per row; and, from workgroups
//               of the same launch, dgamma = sum_r dH * xh, dbeta = sum_r dH
//               over 512-row chunks in a fixed order.
//   colsum      the fixed-order sum over chunks -- no atomics (the reference
//               uses atomicAdd, norm.cu:68-69).
// For d <= kLnFusedMaxD the block's backward runs the rows and the partials
// inside the dX scatter instead (pointwise.hip) and only colsum runs from
// here; ln_bwd is the path for wider rows, for widths that are not a multiple
// of 64 and for the standalone entry points. Any d >= 1 is accepted: rows
// whose width, strides or base are not multiples of 8 elements are accessed
// without the alignment, their last piece element by element, with the same
// summation order (missing elements of the last 8-element piece count as
// zeros, which leave every sum unchanged).
#include "device_util.hpp"
#include "ln_row.hpp"
#include "moe_internal.hpp"

// Every float operation below is rounded on its own: no contraction into
// fused multiply-adds except the explicit one in ln_row.hpp. Division and
// sqrtf are correctly rounded (hipcc's default for fp32).
#pragma clang fp contract(off)

namespace tmt {
namespace {

// 16 bytes at any element's address (the load and store instructions take
// unaligned global addresses).
typedef unsigned u32x4_any __attribute__((ext_vector_type(4), aligned(2)));
typedef unsigned u32x2_any __attribute__((ext_vector_type(2), aligned(2)));

// The 8 elements k0 .. k0 + 7 of a row: one 16-byte load, 16-byte aligned
// when VEC (d, the row strides and the base pointers are multiples of 8
// elements / 16 bytes), else at any element; elements from column d on are
// zeros (a piece that crosses column d is loaded where the row ends and
// shifted: no load sits under a branch, so a lane's loads stay in flight
// together). PAST: k0 may be d or more (H's padded columns). Zeros leave the
// row sums unchanged (x + 0 = x, fma(0, 0, s) = s), so both forms give the
// same statistics.
template <bool VEC, bool PAST = false>
__device__ __forceinline__ void load_row8(const uint16_t* row, int k0, int d, float (&v)[8]) {
    if constexpr (VEC) {
        unpack8(*reinterpret_cast<const uint4*>(row + k0), v);
    } else if (d >= 8) {  // uniform
        const int c0 = min(k0, d - 8);
        if constexpr (!PAST) __builtin_assume(k0 - c0 < 8);  // one case of the shift less
        const u32x4_any w = *reinterpret_cast<const u32x4_any*>(row + c0);
        uint64_t lo = ((uint64_t)w[1] << 32) | w[0], hi = ((uint64_t)w[3] << 32) | w[2];
        shift_piece(lo, hi, (k0 - c0) * 16);
        unpack8(make_uint4((uint32_t)lo, (uint32_t)(lo >> 32), (uint32_t)hi, (uint32_t)(hi >> 32)), v);
    } else {
#pragma unroll
        for (int t = 0; t < 8; ++t) v[t] = k0 + t < d ? bf1(row[k0 + t]) : 0.0f;
    }
}
// gamma or beta of columns k0 .. k0 + 7 (16-byte aligned; zeros from column d on).
template <bool VEC>
__device__ __forceinline__ void load_col8(const float* q, int k0, int d, float (&v)[8]) {
    if (VEC || k0 + 8 <= d) {
        const f32x4 a = *reinterpret_cast<const f32x4*>(q + k0), b = *reinterpret_cast<const f32x4*>(q + k0 + 4);
#pragma unroll
        for (int t = 0; t < 4; ++t) {
            v[t] = a[t];
            v[t + 4] = b[t];
        }
    } else {
#pragma unroll
        for (int t = 0; t < 8; ++t) v[t] = k0 + t < d ? q[k0 + t] : 0.0f;
    }
}
// 16-byte aligned store; NT: non-temporal (ln_streams). A template argument:
// the compiler merges the two stores of a branch into a plain one.
template <bool NT>
__device__ __forceinline__ void store16(uint16_t* q, const uint4& w) {
    if constexpr (NT) st16_nt(q, w);
    else *reinterpret_cast<uint4*>(q) = w;
}
template <bool VEC, bool NT>
__device__ __forceinline__ void store_row8(uint16_t* row, int k0, int d, const float (&v)[8]) {
    const uint4 w = pack8(v);
    if constexpr (VEC) {
        store16<NT>(row + k0, w);
    } else if (k0 + 8 <= d) {
        *reinterpret_cast<u32x4_any*>(row + k0) = u32x4_any{w.x, w.y, w.z, w.w};
    } else {
#pragma unroll
        for (int t = 0; t < 8; ++t)
            if (k0 + t < d) row[k0 + t] = f2bf(v[t]);
    }
}

template <bool VEC>
__device__ __forceinline__ void row_stats(const uint16_t* x, int d, int lane, float& mean, float& rstd) {
    float ls = 0.0f, lq = 0.0f;
    for (int k0 = lane * 8; k0 < d; k0 += 512) {
        float v[8];
        load_row8<VEC>(x, k0, d, v);
        ln_accumulate(v, ls, lq);
    }
    ln_finish(ls, lq, d, mean, rstd);
}

template <bool VEC, bool NT>
__global__ __launch_bounds__(kThreads) void ln_fwd_kernel(LayerNormParams p) {
    const int lane = threadIdx.x & 63;
    const int r = blockIdx.x * 4 + (threadIdx.x >> 6);
    if (r >= p.T) return;
    const int d = p.d;
    const uint16_t* x = p.S + (int64_t)r * p.lds;
    uint16_t* hrow = p.H + (int64_t)r * p.ldh;
    float mean, rstd;
    row_stats<VEC>(x, d, lane, mean, rstd);
    for (int k0 = lane * 8; k0 < p.ldh; k0 += 512) {
        if constexpr (VEC) {
            uint4 hv = make_uint4(0, 0, 0, 0);  // columns [d, ldh): zeros
            if (k0 < d) {
                float v[8];
                unpack8(*reinterpret_cast<const uint4*>(x + k0), v);
                hv = ln_apply8(v, mean, rstd, p.gamma, p.beta, k0);
            }
            store16<NT>(hrow + k0, hv);
        } else {
            float v[8], g[8], b[8], y[8];
            load_row8<false, true>(x, k0, d, v);
            load_col8<false>(p.gamma, k0, d, g);
            load_col8<false>(p.beta, k0, d, b);
#pragma unroll
            for (int t = 0; t < 8; ++t) {
                const float xh = (v[t] - mean) * rstd;
                y[t] = k0 + t < d ? xh * g[t] + b[t] : 0.0f;  // columns [d, ldh): zeros
            }
            store_row8<false, false>(hrow, k0, p.ldh, y);
        }
    }
    if (lane == 0) {
        p.mean[r] = mean;
        p.rstd[r] = rstd;
    }
}

// Rows of at most NP * 512 elements (16-byte pieces): each lane loads its
// pieces once into registers, so the normalisation does not read the row a
// second time after the statistics (one memory round trip per row instead
// of two). The sums run over the same pieces in the same order as
// row_stats, so mean, 1/std and H are bit-identical to ln_fwd_kernel<true>.
template <int NP, bool NT>
__global__ __launch_bounds__(kThreads) void ln_fwd_reg_kernel(LayerNormParams p) {
    const int lane = threadIdx.x & 63;
    const int r = blockIdx.x * 4 + (threadIdx.x >> 6);
    if (r >= p.T) return;
    const int d = p.d;
    const uint16_t* x = p.S + (int64_t)r * p.lds;
    uint16_t* hrow = p.H + (int64_t)r * p.ldh;
    uint4 raw[NP];
#pragma unroll
    for (int i = 0; i < NP; ++i) {
        const int k0 = lane * 8 + 512 * i;
        raw[i] = k0 < d ? *reinterpret_cast<const uint4*>(x + k0) : make_uint4(0, 0, 0, 0);
    }
    float ls = 0.0f, lq = 0.0f;
#pragma unroll
    for (int i = 0; i < NP; ++i) {
        if (lane * 8 + 512 * i < d) {
            float v[8];
            unpack8(raw[i], v);
            ln_accumulate(v, ls, lq);
        }
    }
    float mean, rstd;
    ln_finish(ls, lq, d, mean, rstd);
#pragma unroll
    for (int i = 0; i < NP; ++i) {
        const int k0 = lane * 8 + 512 * i;
        if (k0 >= p.ldh) break;
        uint4 hv = make_uint4(0, 0, 0, 0);  // columns [d, ldh): zeros
        if (k0 < d) {
            float v[8];
            unpack8(raw[i], v);
            hv = ln_apply8(v, mean, rstd, p.gamma, p.beta, k0);
        }
        store16<NT>(hrow + k0, hv);
    }
    if (lane == 0) {
        p.mean[r] = mean;
        p.rstd[r] = rstd;
    }
}

// Backward, one launch of two kinds of workgroups, chunk by chunk of kLnRows
// rows: first ceil(d / kLnCols) workgroups that each sum dgamma / dbeta of
// kLnCols columns over the chunk, then the chunk's kLnRows / 4 row groups
// (one wave per row). The two read the same rows at about the same time, so
// the second reading comes from the caches, and the column workgroups' chain
// of row loads runs beside the rows' streaming instead of after it.
// Bound by HBM (S and dH in, dS out: 157 MB at T = 20480, d = 1280). There
// rows and column sums as two launches (36.6 + 43.2 us, the column sums on
// 200 workgroups of 256 columns) became one of 47.3 us, 42.5 us with
// non-temporal dS stores. Unaligned rows (T = 1000, d = 1250, forward and
// backward): 180 -> 35 us with loads of 16 bytes instead of 2.
constexpr int kLnRows = 512;
constexpr int kLnCols = 64;

// dS of row r. NP > 0: rows of at most NP * 512 elements, whose S and dH
// pieces stay in registers between the sums and the output; NP == 0: read
// twice. The sums run over the same pieces in the same order in both.
template <bool VEC, int NP, bool NT>
__device__ __forceinline__ void ln_bwd_row(const LayerNormParams& p, int r, int lane) {
    const int d = p.d;
    const uint16_t* x = p.S + (int64_t)r * p.lds;
    const uint16_t* dh = p.dH + (int64_t)r * p.ldh;
    uint16_t* ds = p.dS + (int64_t)r * p.lds;
    const float mean = p.mean[r], rstd = p.rstd[r];
    constexpr int NR = NP > 0 ? NP : 1;
    float v[NR][8], gy[NR][8];
    float s1 = 0.0f, s2 = 0.0f;
    auto sums = [&](int k0, const float (&vv)[8], const float (&gg)[8]) {
        float gam[8];
        load_col8<VEC>(p.gamma, k0, d, gam);
#pragma unroll
        for (int t = 0; t < 8; ++t) {
            if (!VEC && k0 + t >= d) continue;
            const float g = gg[t] * gam[t];
            const float xh = (vv[t] - mean) * rstd;
            s1 = s1 + g;
            s2 = s2 + g * xh;
        }
    };
    if constexpr (NP > 0) {
#pragma unroll
        for (int i = 0; i < NP; ++i) {
            const int k0 = lane * 8 + 512 * i;
            if (k0 < d) {
                load_row8<VEC>(x, k0, d, v[i]);
                load_row8<VEC>(dh, k0, d, gy[i]);
            }
        }
#pragma unroll
        for (int i = 0; i < NP; ++i) {
            const int k0 = lane * 8 + 512 * i;
            if (k0 < d) sums(k0, v[i], gy[i]);
        }
    } else {
        for (int k0 = lane * 8; k0 < d; k0 += 512) {
            load_row8<VEC>(x, k0, d, v[0]);
            load_row8<VEC>(dh, k0, d, gy[0]);
            sums(k0, v[0], gy[0]);
        }
    }
    s1 = wave_sum(s1);
    s2 = wave_sum(s2);
    const float a = s1 / (float)d, b = s2 / (float)d;
    auto out8 = [&](int k0, const float (&vv)[8], const float (&gg)[8]) {
        float out[8], gam[8];
        load_col8<VEC>(p.gamma, k0, d, gam);
#pragma unroll
        for (int t = 0; t < 8; ++t) {
            const float g = gg[t] * gam[t];  // columns from d on are not stored
            const float xh = (vv[t] - mean) * rstd;
            out[t] = rstd * ((g - a) - xh * b);
        }
        store_row8<VEC, NT>(ds, k0, d, out);
    };
    if constexpr (NP > 0) {
#pragma unroll
        for (int i = 0; i < NP; ++i) {
            const int k0 = lane * 8 + 512 * i;
            if (k0 < d) out8(k0, v[i], gy[i]);
        }
    } else {
        for (int k0 = lane * 8; k0 < d; k0 += 512) {
            load_row8<VEC>(x, k0, d, v[0]);
            load_row8<VEC>(dh, k0, d, gy[0]);
            out8(k0, v[0], gy[0]);
        }
    }
}

// dgamma / dbeta of kLnCols columns over one chunk: lane l owns columns
// 4 (l % 16) .. + 3 of row phase 4 wave + l / 16; a phase adds the chunk's
// rows phase, phase + 16, ... in ascending order (8 rows' loads in flight),
// the four phases of a wave are added by a butterfly and the waves in order.
// Partials are rows of ln_width4(d) floats; columns [d, ln_width4(d)) hold zeros.
template <bool VEC>
__device__ __forceinline__ void ln_dgb_block(const LayerNormParams& p, int chunk, int cblk) {
    __shared__ f32x4 s_part[3][2][16];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int col = cblk * kLnCols + (lane & 15) * 4;
    const int d = p.d, pw = ln_width4(d);
    const int r0 = chunk * kLnRows, r1 = min(p.T, r0 + kLnRows);
    const bool cok = col < d;
    const int ccol = cok ? col : 0;
    // four columns of row r of a bf16 matrix with row stride ld (zeros from column d on)
    auto load4 = [&](const uint16_t* base, int ld, int r, float (&v)[4]) {
        const uint16_t* q = base + (int64_t)r * ld + ccol;
        if constexpr (VEC) {
            const uint2 w = *reinterpret_cast<const uint2*>(q);
            v[0] = bf_lo(w.x); v[1] = bf_hi(w.x); v[2] = bf_lo(w.y); v[3] = bf_hi(w.y);
        } else if (d >= 4) {  // uniform; columns past d dropped by the shift, as in load_row8
            const int over = max(ccol + 4 - d, 0);
            const u32x2_any w = *reinterpret_cast<const u32x2_any*>(q - over);
            const uint64_t x = (((uint64_t)w[1] << 32) | w[0]) >> (16 * over);
            const uint32_t x0 = (uint32_t)x, x1 = (uint32_t)(x >> 32);
            v[0] = bf_lo(x0); v[1] = bf_hi(x0); v[2] = bf_lo(x1); v[3] = bf_hi(x1);
        } else {
#pragma unroll
            for (int t = 0; t < 4; ++t) v[t] = ccol + t < d ? bf1(q[t]) : 0.0f;
        }
    };
    f32x4 ag = f32x4{0.f, 0.f, 0.f, 0.f}, ab = f32x4{0.f, 0.f, 0.f, 0.f};
    constexpr int U = 8;
    const int ph = 4 * wave + (lane >> 4);
    for (int rb = r0 + ph; rb < r1; rb += 16 * U) {
        float xv[U][4], gv[U][4], mean[U], rstd[U];
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const int r = min(rb + 16 * u, r1 - 1);
            load4(p.S, p.lds, r, xv[u]);
            load4(p.dH, p.ldh, r, gv[u]);
            mean[u] = p.mean[r];
            rstd[u] = p.rstd[r];
        }
#pragma unroll
        for (int u = 0; u < U; ++u) {
            if (rb + 16 * u < r1) {
#pragma unroll
                for (int t = 0; t < 4; ++t) {
                    const float xh = (xv[u][t] - mean[u]) * rstd[u];
                    ag[t] = ag[t] + gv[u][t] * xh;
                    ab[t] = ab[t] + gv[u][t];
                }
            }
        }
    }
#pragma unroll
    for (int t = 0; t < 4; ++t) {
        ag[t] = ag[t] + xor_lane<16>(ag[t]);
        ab[t] = ab[t] + xor_lane<16>(ab[t]);
        ag[t] = ag[t] + xor_lane<32>(ag[t]);
        ab[t] = ab[t] + xor_lane<32>(ab[t]);
    }
    if (wave > 0 && lane < 16) {
        s_part[wave - 1][0][lane] = ag;
        s_part[wave - 1][1][lane] = ab;
    }
    __syncthreads();
    if (wave == 0 && lane < 16 && cok) {
        for (int w = 0; w < 3; ++w) {
            ag += s_part[w][0][lane];
            ab += s_part[w][1][lane];
        }
        *reinterpret_cast<f32x4*>(p.partial + ((int64_t)chunk * 2) * pw + col) = ag;
        *reinterpret_cast<f32x4*>(p.partial + ((int64_t)chunk * 2 + 1) * pw + col) = ab;
    }
}

template <bool VEC, int NP, bool NT>
__global__ __launch_bounds__(kThreads) void ln_bwd_kernel(LayerNormParams p, int ncol) {
    const int per = ncol + kLnRows / 4;  // workgroups of one chunk
    const int chunk = blockIdx.x / per, b = blockIdx.x % per;
    if (b < ncol) {
        ln_dgb_block<VEC>(p, chunk, b);
        return;
    }
    const int r = chunk * kLnRows + (b - ncol) * 4 + (threadIdx.x >> 6);
    if (r < p.T) ln_bwd_row<VEC, NP, NT>(p, r, threadIdx.x & 63);
}

// Fixed-order column sums of a [nrows][ncols] fp32 matrix (ncols a multiple
// of 4): a workgroup of 16 waves owns 32 columns, thread t columns
// 4 (t % 8) .. + 3 of the rows t / 8, t / 8 + 128, ... in ascending order;
// the 8 row phases of a wave are added by a butterfly, the waves in order.
// Columns [0, split) go to out_lo, the rest to out_hi. One launch: in two
// (64-row groups, then the groups) the sums of 40 rows of 2560 columns took
// 9.3 us, of 16 rows of 512 columns 6.2 us, nearly all of it launch and
// round trips; now 4.9 and 3.7 us.
constexpr int kColThreads = 1024;
constexpr int kColCols = 32;
__global__ __launch_bounds__(kColThreads) void colsum_kernel(const float* in, int nrows, int ncols, int split,
                                                             int width, float* out_lo, float* out_hi) {
    __shared__ f32x4 s_part[kColThreads / 64][8];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int cl = threadIdx.x & 7;
    const int col = blockIdx.x * kColCols + cl * 4;
    const bool cok = col < ncols;
    const float* src = in + (cok ? col : 0);
    f32x4 acc = f32x4{0.f, 0.f, 0.f, 0.f};
    constexpr int P = kColThreads / 8, U = 8;
    for (int r0 = threadIdx.x >> 3; r0 < nrows; r0 += P * U) {
        f32x4 v[U];
#pragma unroll
        for (int u = 0; u < U; ++u)
            v[u] = *reinterpret_cast<const f32x4*>(src + (int64_t)min(r0 + P * u, nrows - 1) * ncols);
#pragma unroll
        for (int u = 0; u < U; ++u)
            if (r0 + P * u < nrows) acc += v[u];
    }
#pragma unroll
    for (int t = 0; t < 4; ++t) {
        acc[t] = acc[t] + xor_lane<8>(acc[t]);
        acc[t] = acc[t] + xor_lane<16>(acc[t]);
        acc[t] = acc[t] + xor_lane<32>(acc[t]);
    }
    if (lane < 8) s_part[wave][cl] = acc;
    __syncthreads();
    if (threadIdx.x >= 8 || !cok) return;
    for (int w = 1; w < kColThreads / 64; ++w) acc += s_part[w][cl];
    const int c = col < split ? col : col - split;
    float* dst = (col < split ? out_lo : out_hi) + c;
    if (c + 4 <= width) {
        *reinterpret_cast<f32x4*>(dst) = acc;
    } else {
        for (int t = 0; t < 4 && c + t < width; ++t) dst[t] = acc[t];
    }
}

}  // namespace

int ln_chunks(int T) {
    const int c = (T + kLnRows - 1) / kLnRows;
    return c < 1 ? 1 : c;
}

hipError_t launch_colsum(const float* in, int nrows, int ncols, int split, int width, float* out_lo,
                         float* out_hi, hipStream_t s) {
    if (ncols % 4 != 0 || split % 4 != 0 || width > split || width > ncols - split) return hipErrorInvalidValue;
    colsum_kernel<<<(ncols + kColCols - 1) / kColCols, kColThreads, 0, s>>>(in, nrows, ncols, split, width, out_lo,
                                                                          out_hi);
    return hipGetLastError();
}

namespace {
bool al16(const void* q) { return (reinterpret_cast<uintptr_t>(q) & 15u) == 0; }
// 16-byte row accesses when d and both row strides are multiples of 8
// elements and every row base is 16-byte aligned; element accesses otherwise.
bool ln_vec(const LayerNormParams& p, bool fwd) {
    if (p.d % 8 != 0 || p.lds % 8 != 0 || p.ldh % 8 != 0 || !al16(p.S)) return false;
    return fwd ? al16(p.H) : (al16(p.dH) && al16(p.dS));
}
// Outputs larger than the L2s hold together (8 x 4 MiB, with the inputs) are
// stored non-temporally: T = 20480, d = 1280 forward + backward 74.5 -> 69.9
// us, T = 32768, d = 512 51.6 -> 46.1 us. Smaller ones stay in L2 for the
// kernel that reads them next, and so does the block's H, which its router
// reads next (14283 x 1216: 2 us less here, 2.4 us more there).
bool ln_streams(int T, int ld) { return (int64_t)T * ld * 2 > (int64_t)16 << 20; }
}  // namespace

hipError_t launch_ln_fwd(const LayerNormParams& p, hipStream_t s) {
    if (p.T <= 0) return hipSuccess;
    if (p.d < 1 || p.lds < p.d || p.ldh < p.d) return hipErrorInvalidValue;
    const unsigned grid = (unsigned)((p.T + 3) / 4);
    if (!ln_vec(p, true)) {
        ln_fwd_kernel<false, false><<<grid, kThreads, 0, s>>>(p);
    } else {
        // 16-byte pieces per lane, H's padded columns included
        const int np = (p.ldh + 511) / 512;
        switch ((np > 4 ? 0 : np) * 2 + (!p.reread && ln_streams(p.T, p.ldh) ? 1 : 0)) {
#define TMT_LN_FWD(NP)                                                               \
    case 2 * NP: ln_fwd_reg_kernel<NP, false><<<grid, kThreads, 0, s>>>(p); break;   \
    case 2 * NP + 1: ln_fwd_reg_kernel<NP, true><<<grid, kThreads, 0, s>>>(p); break;
            TMT_LN_FWD(1)
            TMT_LN_FWD(2)
            TMT_LN_FWD(3)
            TMT_LN_FWD(4)
#undef TMT_LN_FWD
            case 0: ln_fwd_kernel<true, false><<<grid, kThreads, 0, s>>>(p); break;
            case 1: ln_fwd_kernel<true, true><<<grid, kThreads, 0, s>>>(p); break;
        }
    }
    return hipGetLastError();
}

hipError_t launch_ln_bwd(const LayerNormParams& p, hipStream_t s) {
    if (p.d < 1 || p.lds < p.d || p.ldh < p.d) return hipErrorInvalidValue;
    const bool vec = ln_vec(p, false);
    const int nch = ln_chunks(p.T), pw = ln_width4(p.d), ncol = (p.d + kLnCols - 1) / kLnCols;
    const int64_t blocks = (int64_t)nch * (ncol + kLnRows / 4);
    if (blocks > 0x7fffffff) return hipErrorInvalidValue;
    const unsigned grid = (unsigned)blocks;
    const int np = (p.d + 511) / 512;
    // unaligned rows (row form 0), aligned (1), aligned and streamed out (2)
    switch ((np > 4 ? 0 : np) * 3 + (!vec ? 0 : ln_streams(p.T, p.lds) ? 2 : 1)) {
#define TMT_LN_BWD(NP)                                                                        \
    case 3 * NP: ln_bwd_kernel<false, NP, false><<<grid, kThreads, 0, s>>>(p, ncol); break;   \
    case 3 * NP + 1: ln_bwd_kernel<true, NP, false><<<grid, kThreads, 0, s>>>(p, ncol); break; \
    case 3 * NP + 2: ln_bwd_kernel<true, NP, true><<<grid, kThreads, 0, s>>>(p, ncol); break;
        TMT_LN_BWD(0)
        TMT_LN_BWD(1)
        TMT_LN_BWD(2)
        TMT_LN_BWD(3)
        TMT_LN_BWD(4)
#undef TMT_LN_BWD
    }
    return launch_colsum(p.partial, nch, 2 * pw, pw, p.d, p.dgamma, p.dbeta, s);
}

}  // namespace tmt
