// codec.hip - elementwise fp8 kernels: encode / decode over arrays,
// dequantize, the per-row error statistics, and the self-check of the
// hardware conversion the quantizer's fast path relies on.
#include "codec.h"

#include <algorithm>

#include "common.h"

namespace reng {

typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
typedef float f32x2 __attribute__((ext_vector_type(2)));
typedef unsigned short u16x2 __attribute__((ext_vector_type(2)));

namespace {

// Grid of at most ~8 blocks per CU for a grid-stride loop over n items.
dim3 stride_grid(uint64_t n, int threads) {
    uint64_t blocks = (n + threads - 1) / threads;
    const uint64_t cap = (uint64_t)device_props().cus * 8;
    if (blocks > cap) blocks = cap;
    if (blocks < 1) blocks = 1;
    return dim3((unsigned)blocks);
}

}  // namespace

// encode (lib.rs:154-201) over an array.
template <int F>
__global__ void encode_kernel(const float *__restrict__ x, uint64_t n, uint8_t *__restrict__ out) {
    for (uint64_t i = blockIdx.x * (uint64_t)blockDim.x + threadIdx.x; i < n;
         i += (uint64_t)gridDim.x * blockDim.x)
        out[i] = (uint8_t)encode_exact<F>(x[i]);
}

// decode (lib.rs:206-225) over an array.
template <int F>
__global__ void decode_kernel(const uint8_t *__restrict__ c, uint64_t n, float *__restrict__ out) {
    for (uint64_t i = blockIdx.x * (uint64_t)blockDim.x + threadIdx.x; i < n;
         i += (uint64_t)gridDim.x * blockDim.x)
        out[i] = decode_exact<F>(c[i]);
}

// Quantized::dequantize (lib.rs:328-337): decode(code) * scale, one f32
// multiply; dequantize_bf16 (lib.rs:342-344) rounds that to bf16. Any shape and
// alignment, one value per thread and step: small matrices, and what
// dequant_units does not take (codes or output off a unit's alignment).
template <int F, bool BF16>
__global__ void dequant_kernel(const uint8_t *__restrict__ c, const float *__restrict__ scales,
                               uint64_t rows, uint64_t cols, void *__restrict__ out) {
    const uint64_t n = rows * cols;
    for (uint64_t i = blockIdx.x * (uint64_t)blockDim.x + threadIdx.x; i < n;
         i += (uint64_t)gridDim.x * blockDim.x) {
        const float v = decode_exact<F>(c[i]) * scales[i / cols];
        if constexpr (BF16)
            static_cast<uint16_t *>(out)[i] = (uint16_t)f32_to_bf16_bits(v);
        else
            static_cast<float *>(out)[i] = v;
    }
}

// Some byte of w has its top exponent field set: reng-fp8 reads such a code as
// +-inf or NaN, the OCP conversion below (E4M3) as a finite value.
template <int F>
__device__ __forceinline__ bool top_field(uint32_t w) {
    if constexpr (F == RENG_HIP_E4M3) return (((w & 0x78787878u) + 0x08080808u) & 0x80808080u) != 0;
    else return (((w & 0x7c7c7c7cu) + 0x04040404u) & 0x80808080u) != 0;
}

// Four finite codes, exactly (the hardware's OCP conversion).
template <int F>
__device__ __forceinline__ void decode4_finite(uint32_t w, float *v) {
    f32x2 lo, hi;
    if constexpr (F == RENG_HIP_E4M3) {
        lo = __builtin_amdgcn_cvt_pk_f32_fp8(w, false);
        hi = __builtin_amdgcn_cvt_pk_f32_fp8(w, true);
    } else {
        lo = __builtin_amdgcn_cvt_pk_f32_bf8(w, false);
        hi = __builtin_amdgcn_cvt_pk_f32_bf8(w, true);
    }
    v[0] = lo.x;
    v[1] = lo.y;
    v[2] = hi.x;
    v[3] = hi.y;
}

template <int F>
__device__ __forceinline__ void decode4(uint32_t w, float *v) {
    if (top_field<F>(w)) {
#pragma unroll
        for (int i = 0; i < 4; ++i) v[i] = decode_exact<F>((w >> (8 * i)) & 0xffu);
    } else {
        decode4_finite<F>(w, v);
    }
}

// Bound: HBM (1 byte in, 2 or 4 out per value). The codes are one flat array
// cut into units of U codes (8 for bf16, 4 for f32 out: one 16-byte store a
// unit), UNITS units per thread, requested together, the units of a wave
// side by side in each; so any row width divides evenly over the chip. A
// unit's row comes from its chunk's start (one f64 multiply: the quotient is
// off by at most one, corrected) plus an f32 division inside the chunk, and a
// unit that crosses a row's end (cols % U != 0; cols >= U, so it meets two rows
// at most) takes each value's own scale. Needs n < 2^52, rows < 2^31, codes
// aligned to U and out to 16 bytes.
// [4096, 14336] to bf16: 95 -> 28 us (a byte load, a 64-bit division and a 2-byte
// store per value before; 176 MB at the 6.1 TB/s of a mixed stream take 29); 2 or 8
// units per thread within 2%, 4 workgroups per CU in place of 16 20% slower.
constexpr int DQ_THREADS = 256;

template <int F, bool BF16, int UNITS>
__global__ __launch_bounds__(DQ_THREADS) void dequant_units(const uint8_t *__restrict__ c,
                                                            const float *__restrict__ scales, uint32_t rows,
                                                            uint64_t cols, double inv_cols, void *__restrict__ out) {
    constexpr int U = BF16 ? 8 : 4;
    constexpr uint32_t CHUNK = U * UNITS * DQ_THREADS;   // values per workgroup and step
    const uint64_t n = (uint64_t)rows * cols;
    const uint32_t tid = threadIdx.x;
    // Below CHUNK columns a chunk may meet many rows; cols then fits an f32 exactly.
    const bool narrow = cols < CHUNK;
    const float inv32 = narrow ? 1.0f / (float)cols : 0.0f;
    for (uint64_t e0 = (uint64_t)blockIdx.x * CHUNK; e0 < n; e0 += (uint64_t)gridDim.x * CHUNK) {
        uint32_t q[UNITS][U / 4];
#pragma unroll
        for (int j = 0; j < UNITS; ++j) {
            const uint64_t e = e0 + (uint64_t)(j * DQ_THREADS + tid) * U;
            if (e + U <= n) {
                if constexpr (U == 8) {
                    const u32x2 v = __builtin_nontemporal_load(reinterpret_cast<const u32x2 *>(c + e));
                    q[j][0] = v.x;
                    q[j][1] = v.y;
                } else {
                    q[j][0] = __builtin_nontemporal_load(reinterpret_cast<const uint32_t *>(c + e));
                }
            }
        }
        // The chunk's first row and column.
        uint32_t r0 = (uint32_t)((double)e0 * inv_cols);
        int64_t k0 = (int64_t)(e0 - (uint64_t)r0 * cols);
        if (k0 < 0) {
            --r0;
            k0 += (int64_t)cols;
        } else if (k0 >= (int64_t)cols) {
            ++r0;
            k0 -= (int64_t)cols;
        }
#pragma unroll
        for (int j = 0; j < UNITS; ++j) {
            const uint32_t l = (j * DQ_THREADS + tid) * U;
            const uint64_t e = e0 + l;
            if (e + U > n) continue;
            uint32_t r = r0;
            uint32_t left;   // values of the unit in row r, U at most
            if (narrow) {
                const int32_t k = (int32_t)k0 + (int32_t)l, w = (int32_t)cols;   // < 2 CHUNK
                int32_t d = (int32_t)((float)k * inv32), m = k - d * w;
                if (m < 0) {
                    --d;
                    m += w;
                } else if (m >= w) {
                    ++d;
                    m -= w;
                }
                r += (uint32_t)d;
                left = (uint32_t)min(w - m, U);
            } else {
                const uint64_t k = (uint64_t)k0 + l;
                const bool next = k >= cols;   // CHUNK <= cols: one row's end at most
                r += next;
                left = (uint32_t)min((next ? 2 * cols : cols) - k, (uint64_t)U);
            }
            const float s0 = scales[r], s1 = left < U ? scales[r + 1 < rows ? r + 1 : r] : s0;
            float v[U];
#pragma unroll
            for (int i = 0; i < U / 4; ++i) decode4<F>(q[j][i], v + 4 * i);
#pragma unroll
            for (int i = 0; i < U; ++i) v[i] *= (uint32_t)i < left ? s0 : s1;
            u32x4 o;
            if constexpr (BF16) {
#pragma unroll
                for (int i = 0; i < 4; ++i) o[i] = f32_to_bf16_bits(v[2 * i]) | (f32_to_bf16_bits(v[2 * i + 1]) << 16);
                __builtin_nontemporal_store(o, reinterpret_cast<u32x4 *>(static_cast<uint16_t *>(out) + e));
            } else {
#pragma unroll
                for (int i = 0; i < 4; ++i) o[i] = __float_as_uint(v[i]);
                __builtin_nontemporal_store(o, reinterpret_cast<u32x4 *>(static_cast<float *>(out) + e));
            }
        }
    }
    // The last n % U values, all in the last row.
    const uint64_t i = n - n % U + tid;
    if (blockIdx.x == 0 && i < n) {
        const float v = decode_exact<F>(c[i]) * scales[rows - 1];
        if constexpr (BF16) static_cast<uint16_t *>(out)[i] = (uint16_t)f32_to_bf16_bits(v);
        else static_cast<float *>(out)[i] = v;
    }
}

// row_errors / sample_row_errors (lib.rs:364-431): WPR waves per sampled row;
// the f64 sum is reduced in a different order than the host's, which moves
// the mean in its last bits only.
//
// Bound: HBM (3 bytes per weight) and, close behind, the vector ALU. A thread
// takes eight weights (16 bytes) and their codes (8 bytes) at a time with
// loads of any alignment, so odd widths run the same path. |(got - want) / want|
// is a correctly rounded f32 division in the reference; here q0 = a * rcp(b) and
// q = q0 + (a - b q0) * rcp(b) with fused multiply-adds gives the same bits where
// nothing over- or underflows: v_rcp_f32 is within 1 ulp, so q0 is within 2 ulp
// of a / b, a - b q0 is exact, and the corrected value is within 2^-20 ulp of
// the quotient before its one rounding; no quotient is a rounding edge (an edge's
// 25 significant bits times b do not fit a's 24), and b has 8 significant bits, so
// every quotient lies at least 2^-9 ulp from one. Units with a non-zero weight
// outside 2^-60 .. 2^60 or a reserved code, and rows whose scale passes 2^43, take
// the IEEE division and the exact decoder. [4096, 14336]: 127 -> 36 us (a 2-byte
// and a 1-byte load and an IEEE division per weight before; 176 MB take 24.5 us to
// read). Narrow rows take a weight per lane with the IEEE division (no UNITS).
typedef u32x4 u32x4_any __attribute__((aligned(2)));
typedef u32x2 u32x2_any __attribute__((aligned(1)));

struct RowErr {
    double sum;
    float mx;
    uint64_t cnt;
};

template <int F>
__device__ __forceinline__ void row_err_exact(uint32_t wbits, uint32_t code, float s, RowErr &e) {
    const float want = __uint_as_float(wbits << 16);
    if (want == 0.0f) return;
    const float rel = __builtin_fabsf((decode_exact<F>(code) * s - want) / want);
    e.sum += (double)rel;
    e.mx = __builtin_fmaxf(e.mx, rel);   // IEEE maxNum: a NaN loses, as f32::max
    ++e.cnt;
}

// Eight weights of magnitude 0 or ERR_LO .. ERR_HI (bf16 bits: 2^-60 .. just below
// 2^60) and their finite codes; ZEROS: some weight may be 0, which counts for nothing.
constexpr uint32_t ERR_LO = (127 - 60) << 7, ERR_HI = ((127 + 60) << 7) - 1;

template <int F, bool ZEROS>
__device__ __forceinline__ void row_err_unit(const u32x4 &wq, const u32x2 &cq, float s, RowErr &e) {
    float got[8];
    decode4_finite<F>(cq.x, got);
    decode4_finite<F>(cq.y, got + 4);
    uint32_t cnt = 8;
#pragma unroll
    for (int i = 0; i < 8; ++i) {
        const uint32_t b = (i & 1) ? wq[i / 2] & 0xffff0000u : wq[i / 2] << 16;
        const float want = __uint_as_float(b), a = got[i] * s - want;
        const float rc = __builtin_amdgcn_rcpf(want), q0 = a * rc;
        float rel = __builtin_fabsf(__builtin_fmaf(__builtin_fmaf(-want, q0, a), rc, q0));
        if constexpr (ZEROS) {
            const bool zero = (b & 0x7fffffffu) == 0;
            rel = zero ? 0.0f : rel;
            cnt -= zero;
        }
        e.sum += (double)rel;
        e.mx = __builtin_fmaxf(e.mx, rel);
    }
    e.cnt += cnt;
}

template <int F, int WPR, bool UNITS>
__global__ __launch_bounds__(256) void row_errors_kernel(const uint16_t *__restrict__ w,
                                                         const uint8_t *__restrict__ c,
                                                         const float *__restrict__ scales,
                                                         uint64_t cols, uint64_t step,
                                                         uint64_t nsampled,
                                                         float *__restrict__ mean_rel,
                                                         float *__restrict__ max_rel) {
    static_assert(WPR == 1 || WPR == 4, "a row per wave or per workgroup");
    constexpr uint32_t T = 64 * WPR;
    __shared__ RowErr part[4];
    const uint32_t lane = threadIdx.x & 63, wv = threadIdx.x >> 6, t = WPR == 1 ? lane : threadIdx.x;
    const uint64_t rows_per_block = 4 / WPR;
    for (uint64_t k0 = blockIdx.x * rows_per_block; k0 < nsampled; k0 += gridDim.x * rows_per_block) {
        const uint64_t k = WPR == 1 ? k0 + wv : k0;
        RowErr e{0.0, 0.0f, 0};
        if (k < nsampled) {
            const uint64_t r = k * step;
            const float s = scales[r];
            const bool wild = !(__builtin_fabsf(s) <= 0x1p43f);   // |got| may pass 2^59
            const uint16_t *wr = w + r * cols;
            const uint8_t *cr = c + r * cols;
            const uint64_t units = UNITS ? cols / 8 : 0;
            // The next unit is requested before this one's arithmetic (past the
            // row's last unit: that one again).
            u32x4 wn;
            u32x2 cn;
            auto request = [&](uint64_t u) {
                wn = *reinterpret_cast<const u32x4_any *>(wr + 8 * u);
                cn = *reinterpret_cast<const u32x2_any *>(cr + 8 * u);
            };
            if (t < units) request(t);
            for (uint64_t u = t; u < units; u += T) {
                const u32x4 wq = wn;
                const u32x2 cq = cn;
                request(u + T < units ? u + T : u);
                u16x2 lo = {0xffff, 0xffff}, hi = {0, 0}, lo_nz = lo;   // magnitude bits; lo_nz: minus one, zeros on top
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    const u16x2 m = __builtin_bit_cast(u16x2, wq[i] & 0x7fff7fffu);
                    lo = __builtin_elementwise_min(lo, m);
                    lo_nz = __builtin_elementwise_min(lo_nz, (u16x2)(m - (u16x2){1, 1}));
                    hi = __builtin_elementwise_max(hi, m);
                }
                const bool odd = wild || min(lo_nz.x, lo_nz.y) < ERR_LO - 1 || max(hi.x, hi.y) > ERR_HI ||
                                 top_field<F>(cq.x) || top_field<F>(cq.y);
                if (odd) {
#pragma unroll 1
                    for (int i = 0; i < 8; ++i) {
                        const uint32_t wi = i < 2 ? wq.x : i < 4 ? wq.y : i < 6 ? wq.z : wq.w, ci = i < 4 ? cq.x : cq.y;
                        row_err_exact<F>((wi >> (16 * (i & 1))) & 0xffffu, (ci >> (8 * (i & 3))) & 0xffu, s, e);
                    }
                } else if (__ballot(min(lo.x, lo.y) == 0) == 0) {
                    row_err_unit<F, false>(wq, cq, s, e);
                } else {
                    row_err_unit<F, true>(wq, cq, s, e);
                }
            }
            if constexpr (UNITS) {
                if (const uint64_t i = units * 8 + t; i < cols) row_err_exact<F>(wr[i], cr[i], s, e);
            } else {
                for (uint64_t i = t; i < cols; i += T) row_err_exact<F>(wr[i], cr[i], s, e);
            }
        }
#pragma unroll
        for (int o = 32; o > 0; o >>= 1) {
            e.sum += __shfl_xor(e.sum, o, 64);
            e.mx = __builtin_fmaxf(e.mx, __shfl_xor(e.mx, o, 64));
            e.cnt += __shfl_xor(e.cnt, o, 64);
        }
        if constexpr (WPR == 4) {
            if (lane == 0) part[wv] = e;
            __syncthreads();
            e.sum = ((part[0].sum + part[1].sum) + part[2].sum) + part[3].sum;
            e.mx = __builtin_fmaxf(__builtin_fmaxf(part[0].mx, part[1].mx), __builtin_fmaxf(part[2].mx, part[3].mx));
            e.cnt = part[0].cnt + part[1].cnt + part[2].cnt + part[3].cnt;
            __syncthreads();
        }
        if (t == 0 && k < nsampled) {
            mean_rel[k] = e.cnt == 0 ? 0.0f : (float)(e.sum / (double)e.cnt);
            max_rel[k] = e.mx;
        }
    }
}

// Every non-NaN f32 pattern: the conversion as the fast path uses it (clamped
// into +-max finite, then v_cvt_pk_*) against the exact integer encoder; and,
// below the first midpoint past the largest finite value (248 / 61440), the
// unclamped conversion too.
template <int F>
__global__ void verify_hw_kernel(unsigned long long *__restrict__ count, uint32_t *__restrict__ first) {
    constexpr float UNCLAMPED = F == RENG_HIP_E4M3 ? 248.0f : 61440.0f;
    unsigned long long bad = 0;
    uint32_t fbad = 0xffffffffu;
    const uint64_t total = 1ull << 32;
    for (uint64_t i = blockIdx.x * (uint64_t)blockDim.x + threadIdx.x; i < total;
         i += (uint64_t)gridDim.x * blockDim.x) {
        const uint32_t u = (uint32_t)i;
        const float x = __uint_as_float(u);
        if (__builtin_isnan(x)) continue;
        const uint32_t ex = encode_exact<F>(x);
        bool ok = (cvt_pk_lo<F>(prep<F, true>(x), 0.0f, 0u) & 0xffu) == ex;
        // Unclamped, below the first midpoint past the largest finite value.
        if (__builtin_fabsf(x) < UNCLAMPED) ok = ok && (cvt_pk_lo<F>(x, 0.0f, 0u) & 0xffu) == ex;
        if (!ok) {
            ++bad;
            fbad = u < fbad ? u : fbad;
        }
    }
    if (bad) {
        atomicAdd(count, bad);
        atomicMin(first, fbad);
    }
}

int launch_encode(const float *x, uint64_t n, int format, uint8_t *out, hipStream_t st) {
    const dim3 g = stride_grid(n, 256);
    if (format == RENG_HIP_E4M3)
        hipLaunchKernelGGL(encode_kernel<RENG_HIP_E4M3>, g, dim3(256), 0, st, x, n, out);
    else
        hipLaunchKernelGGL(encode_kernel<RENG_HIP_E5M2>, g, dim3(256), 0, st, x, n, out);
    return check_launch("encode");
}

int launch_decode(const uint8_t *c, uint64_t n, int format, float *out, hipStream_t st) {
    const dim3 g = stride_grid(n, 256);
    if (format == RENG_HIP_E4M3)
        hipLaunchKernelGGL(decode_kernel<RENG_HIP_E4M3>, g, dim3(256), 0, st, c, n, out);
    else
        hipLaunchKernelGGL(decode_kernel<RENG_HIP_E5M2>, g, dim3(256), 0, st, c, n, out);
    return check_launch("decode");
}

namespace {

// Four units a thread, or one where four would leave the chip few workgroups (fewer
// than 4 per CU of 8-code units, 2 of 4-code ones): bf16 [265, 5198] 4.9 -> 3.7 us,
// [1024, 4096] 6.4 -> 5.3, f32 [1000, 300] 3.9 -> 3.1, while bf16 [4096, 4096] takes
// 11.8 with one and 10.9 with four, f32 [1024, 4096] 6.4 and 5.5. Below 2^19 values
// a thread per value is faster still (its chain is shorter: bf16 [2700, 180] 3.0 us
// against 3.2 with one unit and 5.0 with four; [64, 8192] 3.3 against 3.2).
constexpr uint64_t DQ_SMALL = 1ull << 19;

template <int F, bool BF16>
int launch_dequantize_t(const uint8_t *c, const float *scales, uint64_t rows, uint64_t cols, void *out,
                        hipStream_t st) {
    constexpr uint64_t U = BF16 ? 8 : 4, CHUNK = U * DQ_THREADS;
    const uint64_t n = rows * cols, cus = (uint64_t)device_props().cus;
    const bool units = n >= DQ_SMALL && cols >= U && rows < (1ull << 31) && n < (1ull << 52) &&
                       (reinterpret_cast<uintptr_t>(c) & (U - 1)) == 0 && (reinterpret_cast<uintptr_t>(out) & 15) == 0;
    if (units) {
        const uint64_t many = BF16 ? 4 : 2;
        const bool four = n >= many * cus * 4 * CHUNK;
        const uint64_t chunk = four ? 4 * CHUNK : CHUNK;
        const dim3 grid((unsigned)std::min((n + chunk - 1) / chunk, cus * 16));
        if (four)
            hipLaunchKernelGGL((dequant_units<F, BF16, 4>), grid, dim3(DQ_THREADS), 0, st, c, scales, (uint32_t)rows,
                               cols, 1.0 / (double)cols, out);
        else
            hipLaunchKernelGGL((dequant_units<F, BF16, 1>), grid, dim3(DQ_THREADS), 0, st, c, scales, (uint32_t)rows,
                               cols, 1.0 / (double)cols, out);
    } else {
        hipLaunchKernelGGL((dequant_kernel<F, BF16>), stride_grid(n, 256), dim3(256), 0, st, c, scales, rows, cols, out);
    }
    return check_launch("dequantize");
}

}  // namespace

int launch_dequantize(const uint8_t *c, const float *scales, uint64_t rows, uint64_t cols,
                      int format, bool bf16, void *out, hipStream_t st) {
    if (format == RENG_HIP_E4M3)
        return bf16 ? launch_dequantize_t<RENG_HIP_E4M3, true>(c, scales, rows, cols, out, st)
                    : launch_dequantize_t<RENG_HIP_E4M3, false>(c, scales, rows, cols, out, st);
    return bf16 ? launch_dequantize_t<RENG_HIP_E5M2, true>(c, scales, rows, cols, out, st)
                : launch_dequantize_t<RENG_HIP_E5M2, false>(c, scales, rows, cols, out, st);
}

int launch_row_errors(const uint16_t *w, const uint8_t *c, const float *scales, uint64_t cols,
                      uint64_t step, uint64_t nsampled, int format, float *mean_rel,
                      float *max_rel, hipStream_t st) {
    const uint64_t cus = (uint64_t)device_props().cus;
    // A wave per row where a workgroup's other waves would idle and the rows fill the
    // chip without them; units of eight where a row has enough of them: the IEEE
    // division of one weight per lane is a shorter chain than a unit and the row's
    // last weights after it ([244, 12] 4.2 -> 3.4 us, [100, 100] 4.0 -> 3.4, [60000,
    // 33] 30.7 -> 22.2; the thread-per-weight workgroup that was here first 3.4, 3.4
    // and 93.3).
    const bool few = nsampled <= cus;
    const bool units = cols > 64 && (few ? cols > 256 : cols >= 128);
    const bool wave = cols <= 64 || (cols <= 1024 && !few);
    uint64_t blocks = wave ? (nsampled + 3) / 4 : nsampled;
    const uint64_t cap = cus * 64;
    if (blocks > cap) blocks = cap;
#define RENG_ERR(F, WPR, UNITS)                                                                                     \
    hipLaunchKernelGGL((row_errors_kernel<F, WPR, UNITS>), dim3((unsigned)blocks), dim3(256), 0, st, w, c, scales, cols, \
                       step, nsampled, mean_rel, max_rel)
#define RENG_ERR_F(F)                                          \
    if (wave && units) RENG_ERR(F, 1, true);                   \
    else if (wave) RENG_ERR(F, 1, false);                      \
    else if (units) RENG_ERR(F, 4, true);                      \
    else RENG_ERR(F, 4, false)
    if (format == RENG_HIP_E4M3) {
        RENG_ERR_F(RENG_HIP_E4M3);
    } else {
        RENG_ERR_F(RENG_HIP_E5M2);
    }
#undef RENG_ERR_F
#undef RENG_ERR
    return check_launch("row_errors");
}

int run_verify_hw(int format, unsigned long long *d_count, uint32_t *d_first, hipStream_t st) {
    const dim3 g((unsigned)device_props().cus * 8);
    if (format == RENG_HIP_E4M3)
        hipLaunchKernelGGL(verify_hw_kernel<RENG_HIP_E4M3>, g, dim3(256), 0, st, d_count, d_first);
    else
        hipLaunchKernelGGL(verify_hw_kernel<RENG_HIP_E5M2>, g, dim3(256), 0, st, d_count, d_first);
    return check_launch("verify_hw_convert");
}

}  // namespace reng
