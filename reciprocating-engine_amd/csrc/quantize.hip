// quantize.hip - the fp8 weight quantizer on CDNA4 (gfx950).
//
// Semantics: reng_fp8::quantize_with (crates/reng-fp8/src/lib.rs:519-563),
// bit-exact on codes and scales. The reference makes two passes over the
// weights (row absmax, then encode with an IEEE divide per element); here one
// workgroup owns a row at a time, holds it in registers between the two
// phases and so reads HBM once: rows*cols*(in_bytes + 1) + 4*rows bytes.
//
// Fast path (a row with no NaN and a finite normal scale s): q = RN32(x * RN64(1/s))
// computed in f64 IS the IEEE f32 quotient
// RN32(x / s) that the reference encodes, for every finite x:
//   * x * RN64(1/s) is within |z| * 2^-52 of z = x / s (two f64 roundings);
//   * the quotient of two 24-bit floats is never an f32 midpoint, and when it
//     is not one it lies more than ulp(z) * 2^-25 >= |z| * 2^-49 away from
//     every midpoint (z - t = (X * 2^a - T * S * 2^b) / (S * 2^c) with integer
//     significands X, S < 2^24 and a 25-bit midpoint significand T), so the f64
//     value rounds to the same f32 as z does.
// The f32 quotient then goes through v_cvt_pk_fp8_f32 / v_cvt_pk_bf8_f32 (OCP
// e4m3 / e5m2, round to nearest even), which agree with reng-fp8's encoder on
// every input of magnitude below the first out-of-range midpoint (248 /
// 61440): checked on all 2^32 patterns by reng_hip_verify_hw_convert. Inputs
// that could reach that range (HW and UNIT scales, or a backoff above 1) are
// clamped first with v_med3 (saturation is monotone). A per-channel scale
// s = RN32(m / (max * backoff)) that is normal is within 2^-24 of the exact
// ratio, so with backoff <= 1 no |x / s| passes max * (1 + 2^-23) and no clamp
// is needed; a subnormal s carries fewer significant bits (s = 4 * 2^-149 for
// m = 1000 * 2^-149, E4M3: x / s = 250), so those rows take the slow path.
// Slow rows (a NaN present, s = inf, 0 or subnormal) use the IEEE divide and
// the exact integer encoder for every element, with x86's NaN semantics.
#include <algorithm>
#include <type_traits>

#include "common.h"
#include "quantize.h"

namespace reng {

typedef unsigned short u16x2 __attribute__((ext_vector_type(2)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));

template <int F>
__device__ __forceinline__ uint32_t exact4(float x0, float x1, float x2, float x3, float s) {
    return encode_div<F>(x0, s) | (encode_div<F>(x1, s) << 8) | (encode_div<F>(x2, s) << 16) |
           (encode_div<F>(x3, s) << 24);
}

// Block-wide max of a u32; every thread gets the result. red has one slot per wave.
template <int WAVES>
__device__ __forceinline__ uint32_t block_max(uint32_t v, uint32_t *red) {
    v = wave_max_u32(v);
    if constexpr (WAVES == 1) {
        return v;
    } else {
        const int w = threadIdx.x >> 6;
        if ((threadIdx.x & 63) == 0) red[w] = v;
        __syncthreads();
        uint32_t m = red[0];
#pragma unroll
        for (int i = 1; i < WAVES; ++i) m = m > red[i] ? m : red[i];
        __syncthreads();
        return m;
    }
}

// RN32(x * R) through f64: R = RN64(1/s), the product and the narrowing are
// each rounded to nearest even.
__device__ __forceinline__ float quot(float x, double R) { return (float)((double)x * R); }

__device__ __forceinline__ float bf_lo(uint32_t d) { return __uint_as_float(d << 16); }
__device__ __forceinline__ float bf_hi(uint32_t d) { return __uint_as_float(d & 0xffff0000u); }

template <typename InT>
struct InTraits;
template <>
struct InTraits<uint16_t> {   // bf16 bits
    static constexpr int EPV = 8;
    typedef uint16_t bits;
    static constexpr uint32_t INF = 0x7f80u;
    typedef u32x4 vec_any __attribute__((aligned(2)));    // 16 bytes at any element
    typedef u32x2 codes, codes_any __attribute__((aligned(1)));   // their codes; at any byte
    __device__ static uint32_t mag(uint16_t b) { return b & 0x7fffu; }
    __device__ static float f(uint32_t b) { return __uint_as_float(b << 16); }
};
template <>
struct InTraits<float> {
    static constexpr int EPV = 4;
    typedef uint32_t bits;
    static constexpr uint32_t INF = 0x7f800000u;
    typedef u32x4 vec_any __attribute__((aligned(4)));
    typedef uint32_t codes, codes_any __attribute__((aligned(1)));
    __device__ static uint32_t mag(uint32_t b) { return b & 0x7fffffffu; }
    __device__ static float f(uint32_t b) { return __uint_as_float(b); }
};

// Magnitude bits of the largest non-NaN value of one 16-byte vector.
template <typename InT>
__device__ __forceinline__ uint32_t vec_absmax_no_nan(const u32x4 &v) {
    using IT = InTraits<InT>;
    uint32_t mx = 0;
#pragma unroll
    for (int k = 0; k < 4; ++k) {
        if constexpr (sizeof(InT) == 2) {
            const uint32_t lo = v[k] & 0x7fffu, hi = (v[k] >> 16) & 0x7fffu;
            if (lo <= IT::INF && lo > mx) mx = lo;
            if (hi <= IT::INF && hi > mx) mx = hi;
        } else {
            const uint32_t a = v[k] & 0x7fffffffu;
            if (a <= IT::INF && a > mx) mx = a;
        }
    }
    return mx;
}

// Magnitude bits of the largest value of VPT vectors, NaN patterns included (they sort above inf).
template <typename InT, int VPT>
__device__ __forceinline__ uint32_t vecs_absmax(const u32x4 (&v)[VPT]) {
    uint32_t mx = 0;
    if constexpr (sizeof(InT) == 2) {
        u16x2 m2 = {0, 0};
#pragma unroll
        for (int j = 0; j < VPT; ++j)
#pragma unroll
            for (int k = 0; k < 4; ++k)
                m2 = __builtin_elementwise_max(m2, __builtin_bit_cast(u16x2, v[j][k] & 0x7fff7fffu));
        mx = m2.x > m2.y ? m2.x : m2.y;
    } else {
#pragma unroll
        for (int j = 0; j < VPT; ++j) {
            const uint32_t a0 = v[j].x & 0x7fffffffu, a1 = v[j].y & 0x7fffffffu;
            const uint32_t a2 = v[j].z & 0x7fffffffu, a3 = v[j].w & 0x7fffffffu;
            mx = max(max(mx, max(a0, a1)), max(a2, a3));
        }
    }
    return mx;
}

// Scale of one row from its absmax bits under the per-channel scheme (lib.rs:537-544).
template <typename InT>
__device__ __forceinline__ float pcs_scale(uint32_t mbits, float full) {
    const float m = sizeof(InT) == 2 ? __uint_as_float(mbits << 16) : __uint_as_float(mbits);
    return m > 0.0f ? m / full : 1.0f;
}

// Row `row`'s scale, and with row 0 the matrix's exponent bias: under the
// hardware-bias scheme hw_bias_kernel has written row 0's and the bias (other
// workgroups read it there).
template <int F>
__device__ __forceinline__ void store_scale(const QMat &M, uint64_t row, float s, int scheme) {
    if (row != 0 || scheme != RENG_HIP_HW) M.scales[row] = s;
    if (row == 0 && scheme != RENG_HIP_HW && M.exp_bias) *M.exp_bias = (uint32_t)Fp8<F>::BIAS;
}

// How a row's vectors lie: every lane full (no tail predication), any count, or
// any count, width and alignment (elements past the last whole vector one per
// thread; 16-byte loads and code stores at whatever address). ROWS_SHARED is
// ROWS_ANY for rows of up to 64 vectors that end inside a line: most of a row's
// code lines are shared with the rows beside it, in other workgroups, and a
// non-temporal store sends each part of a line out by itself; plain stores meet
// in L2 (bf16 [605, 10] 4.5 -> 3.4 us, where quantize_rows_generic takes 3.5;
// [4096, 33] 5.1 -> 4.5, [65536, 9] 26.1 -> 24.1). Whole lines and wider rows
// keep the non-temporal ones ([16000, 512] off its input's alignment 9.1 us
// against 9.5, [4096, 4001] 12.4 against 13.1).
enum { ROWS_TAIL = 0, ROWS_FULL = 1, ROWS_ANY = 2, ROWS_SHARED = 3 };

// One row per workgroup (WAVES waves) at a time, VPT 16-byte vectors per thread
// held in registers between the absmax and the encode. Below ROWS_ANY it requires
// 16-byte aligned rows, cols a multiple of EPV and codes rows aligned to the store
// width. ROWS_ANY against the element-at-a-time kernel it replaced (2-byte loads,
// 1-byte stores, an IEEE division per element): bf16 [16000, 4001] 142 -> 46 us,
// [8000, 8567] 149 -> 52, f32 [16000, 3001] 113 -> 48 (an aligned row of the next
// narrower width 36, 41 and 46: a wave's 16-byte loads then cover no extra line).
template <typename InT, int F, int VPT, int WAVES, bool CLAMP, int MODE>
__global__ __launch_bounds__(64 * WAVES) void quantize_rows_fast(QBatch B, int scheme, float full) {
    constexpr bool FULL = MODE == ROWS_FULL, ANY = MODE >= ROWS_ANY;
    using IT = InTraits<InT>;
    constexpr int EPV = IT::EPV;
    constexpr int CPV = EPV / 4;                 // code dwords per vector: 2 (bf16), 1 (f32)
    constexpr int T = 64 * WAVES;
    __shared__ uint32_t red[WAVES];
    const int tid = threadIdx.x;
    const uint64_t G = gridDim.x;
    uint64_t g = blockIdx.x;
    if (g >= B.total_rows) return;

    // Row g lives in matrix mi; rows only grow, so the lookup only moves forward.
    auto locate = [&](uint64_t gg, int &mi) {
        while (mi + 1 < B.n && gg >= B.m[mi + 1].row_begin) ++mi;
    };
    auto row_src = [&](uint64_t gg, int mi) {
        const QMat &M = B.m[mi];
        return static_cast<const InT *>(M.w) + (gg - M.row_begin) * M.ld;
    };
    auto load = [&](const InT *src, uint64_t cols, u32x4 (&v)[VPT], InT &last) {
        const int nvec = (int)(cols / EPV);
#pragma unroll
        for (int j = 0; j < VPT; ++j) {
            const int i = j * T + tid;
            if (!FULL && i >= nvec) v[j] = u32x4{0u, 0u, 0u, 0u};
            else if constexpr (ANY) v[j] = *(reinterpret_cast<const typename IT::vec_any *>(src) + i);
            else v[j] = __builtin_nontemporal_load(reinterpret_cast<const u32x4 *>(src) + i);
        }
        if constexpr (ANY) last = nvec * EPV + tid < cols ? src[nvec * EPV + tid] : InT(0);
    };

    int mi = 0;
    locate(g, mi);
    u32x4 v[VPT];
    InT last{};   // ROWS_ANY: element tid past the row's whole vectors
    load(row_src(g, mi), B.m[mi].cols, v, last);
    int hw_mi = -1;
    float hw_s = 1.0f;
    for (; g < B.total_rows; g += G) {
        const QMat &M = B.m[mi];
        const uint64_t row = g - M.row_begin;
        const int nvec = (int)(M.cols / EPV);

        // Phase 1: row absmax on the magnitude bits (NaN patterns sort above inf).
        uint32_t mx = vecs_absmax<InT>(v);
        if constexpr (ANY) mx = max(mx, IT::mag(__builtin_bit_cast(typename IT::bits, last)));
        mx = block_max<WAVES>(mx, red);
        const bool has_nan = mx > IT::INF;
        if (has_nan) {   // uniform: recompute ignoring NaN (lib.rs:451-454, `v > m`)
            mx = 0;
#pragma unroll
            for (int j = 0; j < VPT; ++j) mx = max(mx, vec_absmax_no_nan<InT>(v[j]));
            if constexpr (ANY) {
                const uint32_t m = IT::mag(__builtin_bit_cast(typename IT::bits, last));
                if (m <= IT::INF) mx = max(mx, m);
            }
            mx = block_max<WAVES>(mx, red);
        }
        float s;
        if constexpr (CLAMP) {
            if (scheme == RENG_HIP_HW && mi != hw_mi) {
                hw_mi = mi;
                // hw_bias_kernel's, for every row of the matrix; in a scalar register (in a
                // vector one it cost the 16-wave form, which spills, 8-16%: bf16 [2000,
                // 40960] unit 51 -> 59 us).
                hw_s = __uint_as_float(__builtin_amdgcn_readfirstlane(__float_as_uint(M.scales[0])));
            }
            s = scheme == RENG_HIP_PCS ? pcs_scale<InT>(mx, full) : hw_s;
        } else {
            s = pcs_scale<InT>(mx, full);   // the clamp is left out for this scheme alone
        }
        if (tid == 0) store_scale<F>(M, row, s, scheme);
        // The next row's loads go out before this row's encode and stores.
        u32x4 vn[VPT];
        InT last_n{};
        const bool more = g + G < B.total_rows;
        if (more) {
            locate(g + G, mi);
            load(row_src(g + G, mi), B.m[mi].cols, vn, last_n);
        }

        // Phase 2: codes from registers. q = RN32(x * RN64(1/s)) equals the
        // IEEE f32 quotient RN32(x / s) for every finite x and every finite
        // non-zero s (see the top of this file), so each code is one f64
        // multiply and one hardware conversion; rows whose s is subnormal
        // (fewer significant bits: |x / s| may pass the clamp-free range) or
        // not finite and positive take the exact path.
        uint32_t c[VPT][CPV];
        const bool fast = !has_nan && s >= 1.17549435e-38f && s < __builtin_inff();
        double fast_r = 0.0;
        if (fast) {
            const double R = fast_r = 1.0 / (double)s;
#pragma unroll
            for (int j = 0; j < VPT; ++j) {
                const uint32_t d[4] = {v[j].x, v[j].y, v[j].z, v[j].w};
                if constexpr (sizeof(InT) == 2) {
                    c[j][0] = cvt4<F, CLAMP>(quot(bf_lo(d[0]), R), quot(bf_hi(d[0]), R),
                                             quot(bf_lo(d[1]), R), quot(bf_hi(d[1]), R));
                    c[j][1] = cvt4<F, CLAMP>(quot(bf_lo(d[2]), R), quot(bf_hi(d[2]), R),
                                             quot(bf_lo(d[3]), R), quot(bf_hi(d[3]), R));
                } else {
                    c[j][0] = cvt4<F, CLAMP>(quot(__uint_as_float(d[0]), R), quot(__uint_as_float(d[1]), R),
                                             quot(__uint_as_float(d[2]), R), quot(__uint_as_float(d[3]), R));
                }
            }
        } else {
            // Slow row: a NaN is present, or s is infinite or zero; the IEEE
            // divide with x86's NaN semantics for every element.
#pragma unroll
            for (int j = 0; j < VPT; ++j) {
                const uint32_t d[4] = {v[j].x, v[j].y, v[j].z, v[j].w};
                if constexpr (sizeof(InT) == 2) {
                    c[j][0] = exact4<F>(bf_lo(d[0]), bf_hi(d[0]), bf_lo(d[1]), bf_hi(d[1]), s);
                    c[j][1] = exact4<F>(bf_lo(d[2]), bf_hi(d[2]), bf_lo(d[3]), bf_hi(d[3]), s);
                } else {
                    c[j][0] = exact4<F>(__uint_as_float(d[0]), __uint_as_float(d[1]),
                                        __uint_as_float(d[2]), __uint_as_float(d[3]), s);
                }
            }
        }
        uint8_t *dst = M.codes + row * M.cols;
#pragma unroll
        for (int j = 0; j < VPT; ++j) {
            const int i = j * T + tid;
            if (FULL || i < nvec) {
                using Codes = std::conditional_t<ANY, typename IT::codes_any, typename IT::codes>;
                Codes q;
                if constexpr (CPV == 2) q = u32x2{c[j][0], c[j][1]};
                else q = c[j][0];
                if constexpr (MODE == ROWS_SHARED) *(reinterpret_cast<Codes *>(dst) + i) = q;
                else __builtin_nontemporal_store(q, reinterpret_cast<Codes *>(dst) + i);
            }
        }

        if constexpr (ANY) {
            const uint64_t i = (uint64_t)nvec * EPV + tid;
            if (i < M.cols) {
                const float x = IT::f(__builtin_bit_cast(typename IT::bits, last));
                dst[i] = (uint8_t)(fast ? cvt4<F, CLAMP>(quot(x, fast_r), 0.0f, 0.0f, 0.0f) : encode_div<F>(x, s));
            }
        }

        if (more) {
#pragma unroll
            for (int j = 0; j < VPT; ++j) v[j] = vn[j];
            last = last_n;
        }
    }
}

// Rows too wide for the register-resident kernel: 256 threads per row, absmax
// then the exact divide-and-encode for every element (the row is read twice,
// from L2).
template <typename InT, int F>
__global__ __launch_bounds__(256) void quantize_rows_generic(QBatch B, int scheme, float full) {
    using IT = InTraits<InT>;
    __shared__ uint32_t red[4];
    const int tid = threadIdx.x;
    int mi = 0, hw_mi = -1;
    float hw_s = 1.0f;
    for (uint64_t g = blockIdx.x; g < B.total_rows; g += gridDim.x) {
        while (mi + 1 < B.n && g >= B.m[mi + 1].row_begin) ++mi;
        const QMat &M = B.m[mi];
        const uint64_t row = g - M.row_begin;
        const InT *src = static_cast<const InT *>(M.w) + row * M.ld;
        uint32_t mx = 0;
        for (uint64_t c = tid; c < M.cols; c += 256) {
            const uint32_t b = IT::mag(__builtin_bit_cast(typename IT::bits, src[c]));
            if (b <= IT::INF && b > mx) mx = b;
        }
        mx = block_max<4>(mx, red);
        if (scheme == RENG_HIP_HW && mi != hw_mi) {
            hw_mi = mi;
            hw_s = M.scales[0];
        }
        const float s = scheme == RENG_HIP_PCS ? pcs_scale<InT>(mx, full) : hw_s;
        if (tid == 0) store_scale<F>(M, row, s, scheme);
        uint8_t *dst = M.codes + row * M.cols;
        for (uint64_t c = tid; c < M.cols; c += 256)
            dst[c] = (uint8_t)encode_div<F>(IT::f(__builtin_bit_cast(typename IT::bits, src[c])), s);
    }
}

// Row absmax (NaN ignored, inf counted) for reng_hip_row_absmax.
template <typename InT>
__global__ __launch_bounds__(256) void row_absmax_kernel(QBatch B, float *__restrict__ out) {
    using IT = InTraits<InT>;
    __shared__ uint32_t red[4];
    const int tid = threadIdx.x;
    for (uint64_t g = blockIdx.x; g < B.total_rows; g += gridDim.x) {
        int mi = 0;
        while (mi + 1 < B.n && g >= B.m[mi + 1].row_begin) ++mi;
        const QMat &M = B.m[mi];
        const uint64_t row = g - M.row_begin;
        const InT *src = static_cast<const InT *>(M.w) + row * M.ld;
        const uint64_t nvec = M.cols / IT::EPV;
        uint32_t mx = 0;
        for (uint64_t i = tid; i < nvec; i += 256) {
            const u32x4 v = *(reinterpret_cast<const typename IT::vec_any *>(src) + i);
            mx = max(mx, vec_absmax_no_nan<InT>(v));
        }
        for (uint64_t c = nvec * IT::EPV + tid; c < M.cols; c += 256) {
            const uint32_t b = IT::mag(__builtin_bit_cast(typename IT::bits, src[c]));
            if (b <= IT::INF && b > mx) mx = b;
        }
        mx = block_max<4>(mx, red);
        if (tid == 0) out[g] = sizeof(InT) == 2 ? __uint_as_float(mx << 16) : __uint_as_float(mx);
    }
}

// The tensor maxima of a batch for the hardware-bias scheme: workgroup b leaves
// what it saw of a matrix, as magnitude bits, in the matrix's scales[b] (its first
// min(rows, gridDim.x) workgroups take a matrix), where hw_bias_kernel reads it, so
// the scheme needs no workspace (a hipMallocAsync / hipFreeAsync pair cost the
// caller 14 us a call), no atomics and nothing cleared first. Bound: HBM, the
// weights read once. A wave takes ABSMAX_VPT 16-byte vectors per lane of one row
// at a time, whatever their alignment (the row's elements past its last whole
// vector one per lane, with its last piece), the pieces of all rows strided over
// the waves of as many workgroups as the matrix has rows, 512 at most. bf16 [4099,
// 4001]: 7.6 us (32.8 MB out of the Infinity Cache) against 54 with 2-byte loads
// and a barrier per row; 1 or 4 workgroups per CU the same.
constexpr int ABSMAX_VPT = 8, ABSMAX_WAVES = 8, ABSMAX_BLOCKS_PER_CU = 2, ABSMAX_SLOTS = 512;

__host__ __device__ __forceinline__ uint64_t batch_rows(const QBatch &B, int mi) {
    return (mi + 1 < B.n ? B.m[mi + 1].row_begin : B.total_rows) - B.m[mi].row_begin;
}

template <typename InT>
__global__ __launch_bounds__(64 * ABSMAX_WAVES) void tensor_absmax(QBatch B) {
    using IT = InTraits<InT>;
    __shared__ uint32_t smax[QBATCH];
    const uint32_t tid = threadIdx.x, lane = tid & 63;
    if (tid < QBATCH) smax[tid] = 0;
    __syncthreads();
    constexpr uint32_t PIECE = 64 * ABSMAX_VPT;
    for (int mi = 0; mi < B.n; ++mi) {
        const QMat &M = B.m[mi];
        const uint64_t rows = batch_rows(B, mi), blocks = rows < gridDim.x ? rows : gridDim.x, waves = blocks * ABSMAX_WAVES;
        if (blockIdx.x >= blocks) continue;
        const uint64_t nvec = M.cols / IT::EPV, per_row = nvec < PIECE ? 1 : (nvec + PIECE - 1) / PIECE;
        const uint64_t pieces = rows * per_row;
        uint32_t mx = 0;
        for (uint64_t p = blockIdx.x * ABSMAX_WAVES + __builtin_amdgcn_readfirstlane(tid >> 6); p < pieces; p += waves) {
            const uint64_t row = per_row == 1 ? p : p / per_row, at = p - row * per_row;
            const InT *src = static_cast<const InT *>(M.w) + row * M.ld;
            u32x4 v[ABSMAX_VPT];
#pragma unroll
            for (int j = 0; j < ABSMAX_VPT; ++j) {
                const uint64_t i = at * PIECE + j * 64 + lane;
                v[j] = i < nvec ? *(reinterpret_cast<const typename IT::vec_any *>(src) + i) : u32x4{0u, 0u, 0u, 0u};
            }
            const uint64_t c = nvec * IT::EPV + lane;
            if (at + 1 == per_row && c < M.cols) {
                const uint32_t b = IT::mag(__builtin_bit_cast(typename IT::bits, src[c]));
                if (b <= IT::INF) mx = max(mx, b);
            }
            uint32_t m = vecs_absmax<InT>(v);
            if (m > IT::INF) {   // a NaN among them: without it (lib.rs:451-454, `v > m`)
                m = 0;
#pragma unroll
                for (int j = 0; j < ABSMAX_VPT; ++j) m = max(m, vec_absmax_no_nan<InT>(v[j]));
            }
            mx = max(mx, m);
        }
        mx = wave_max_u32(mx);
        if (lane == 0) atomicMax(&smax[mi], mx);
    }
    __syncthreads();
    if (tid < (uint32_t)B.n && blockIdx.x < batch_rows(B, tid))
        B.m[tid].scales[blockIdx.x] = __uint_as_float(smax[tid]);
}

// Per matrix (a workgroup each): the maximum of tensor_absmax's `slots` values,
// b = choose_exp_bias(tensor_absmax / backoff), s = 2^(bias - b) (lib.rs:545-549)
// into the matrix's exp_bias and scales[0].
template <typename InT, int F>
__global__ __launch_bounds__(ABSMAX_SLOTS) void hw_bias_kernel(QBatch B, uint32_t slots, float backoff) {
    __shared__ uint32_t red[ABSMAX_SLOTS / 64];
    const int mi = blockIdx.x;
    const QMat &M = B.m[mi];
    const uint64_t rows = batch_rows(B, mi);
    const bool mine = threadIdx.x < slots && threadIdx.x < rows;
    const uint32_t mb = block_max<ABSMAX_SLOTS / 64>(mine ? __float_as_uint(M.scales[threadIdx.x]) : 0u, red);
    if (threadIdx.x != 0) return;   // every slot has been read (block_max's barriers)
    const float tm = sizeof(InT) == 2 ? __uint_as_float(mb << 16) : __uint_as_float(mb);
    const uint32_t b = choose_exp_bias_t<F>(tm / backoff);
    M.scales[0] = pow2f(Fp8<F>::BIAS - (int)b);
    if (M.exp_bias) *M.exp_bias = b;
}

// ------------------------------------------------------------ host launchers

namespace {

struct FastCfg {
    int vpt, waves, mode;
};

// Exact fits (no tail predication) for the row widths of the Llama / Qwen
// shapes: bf16 1024, 2048, 3584, 4096, 5120, 8192, 14336, 16384, 27648 and
// f32 2048, 8192 columns. Rows of 14336 run as 4 waves of 7 vectors (5.86
// TB/s on the Llama-3.1-8B set against 5.66-5.68 for 7 waves of 4), rows of
// 27648 as 9 waves of 6 (5.74-5.76 TB/s on the Qwen2.5-32B set against 5.69
// for 6 waves of 9).
constexpr FastCfg FULL_CFGS[] = {{8, 1, ROWS_FULL}, {7, 1, ROWS_FULL}, {7, 4, ROWS_FULL}, {5, 2, ROWS_FULL}, {8, 2, ROWS_FULL},
                                 {8, 4, ROWS_FULL}, {6, 9, ROWS_FULL}, {2, 1, ROWS_FULL}, {4, 1, ROWS_FULL}};

FastCfg pick_cfg(uint64_t nvec, bool aligned) {
    const int mode = aligned ? ROWS_TAIL : ROWS_ANY;
    if (aligned)
        for (const FastCfg &c : FULL_CFGS)
            if ((uint64_t)c.vpt * 64 * c.waves == nvec) return c;
    if (nvec <= 512) {
        int vpt = 1;
        while ((uint64_t)vpt * 64 < nvec) vpt <<= 1;
        return FastCfg{vpt, 1, mode};
    }
    for (const int waves : {2, 4, 8, 16})
        if ((uint64_t)waves * 512 >= nvec) return FastCfg{8, waves, mode};
    return FastCfg{0, 0, mode};
}

int encode_key(const FastCfg &c) { return c.vpt * 1000 + c.waves * 10 + c.mode; }

// Waves per CU for the register-resident kernel: enough rows in flight to keep
// HBM busy, few enough that the rows being read and written at one time stay
// close together (measured on MI355X: 8 waves per CU beat full occupancy; 6
// for one-wave rows of 8 vectors per lane, i.e. 4096 bf16 or 2048 f32 values:
// rows of 4096 on the Llama-3.1-8B set 5.74-5.75 -> 5.97-5.98 TB/s; 10 for
// two-wave rows of 5 vectors, i.e. 5120 bf16: 5.43-5.59 -> 5.79 TB/s on the
// Qwen2.5-32B shapes). Rows that leave lanes idle keep fewer bytes in flight per
// wave and take more: one pass at 8 (6 for 8 x 1) against 12 waves of 8 vectors,
// 16 of fewer, bf16 [12000, 5632] 39.3 -> 37.2 us, [8000, 8568] 43.8 -> 40.8,
// [60000, 1000] 45.8 -> 36.1, f32 [6000, 8568] 56.9 -> 48.3; rows of 8 and 16
// waves stay at 8 ([3584, 18944] 41.4 against 43.1 us with 16).
constexpr int QUANT_WAVES_PER_CU = 8;
template <int VPT, int WAVES, int MODE>
constexpr int quant_waves_per_cu() {
    if constexpr (MODE != ROWS_FULL) return VPT < 8 ? 16 : WAVES < 8 ? 12 : 8;
    else if constexpr (WAVES == 1 && VPT == 8) return 6;
    else if constexpr (WAVES == 2 && VPT == 5) return 10;
    else return QUANT_WAVES_PER_CU;
}

template <typename InT, int F, int VPT, int WAVES, bool CLAMP, int MODE>
int launch_fast_t(const QBatch &b, int scheme, float full, hipStream_t st) {
    auto kern = quantize_rows_fast<InT, F, VPT, WAVES, CLAMP, MODE>;
    const uint64_t cus = (uint64_t)device_props().cus;
    constexpr int WPC = quant_waves_per_cu<VPT, WAVES, MODE>();
    uint64_t grid = cus * ((WPC + WAVES - 1) / WAVES);
    // A launch of at most 8 waves' worth of rows per CU (the f32 [2048, 2048]
    // matrix) is latency-bound: every row in flight at once.
    if (b.total_rows <= cus * ((QUANT_WAVES_PER_CU + WAVES - 1) / WAVES) || grid > b.total_rows) grid = b.total_rows;
    hipLaunchKernelGGL(kern, dim3((unsigned)grid), dim3(64 * WAVES), 0, st, b, scheme, full);
    return check_launch("quantize_rows_fast");
}

template <typename InT, int F, bool CLAMP>
int launch_fast(int key, const QBatch &b, int scheme, float full, hipStream_t st) {
#define RENG_Q(V, W, MODE)         \
    case V * 1000 + W * 10 + MODE: \
        return launch_fast_t<InT, F, V, W, CLAMP, MODE>(b, scheme, full, st);
// Any alignment: always with the clamp (the same codes where it is not needed, half the kernels).
#define RENG_QA(V, W)                  \
    case V * 1000 + W * 10 + ROWS_ANY: \
        return launch_fast_t<InT, F, V, W, true, ROWS_ANY>(b, scheme, full, st);
    switch (key) {
        case 1010 + ROWS_SHARED: return launch_fast_t<InT, F, 1, 1, true, ROWS_SHARED>(b, scheme, full, st);
        RENG_Q(8, 1, 1) RENG_Q(7, 1, 1) RENG_Q(7, 4, 1) RENG_Q(5, 2, 1) RENG_Q(8, 2, 1)
        RENG_Q(8, 4, 1) RENG_Q(6, 9, 1) RENG_Q(2, 1, 1) RENG_Q(4, 1, 1)
        RENG_Q(1, 1, 0) RENG_Q(2, 1, 0) RENG_Q(4, 1, 0) RENG_Q(8, 1, 0) RENG_Q(8, 2, 0)
        RENG_Q(8, 4, 0) RENG_Q(8, 8, 0) RENG_Q(8, 16, 0)
        RENG_QA(1, 1) RENG_QA(2, 1) RENG_QA(4, 1) RENG_QA(8, 1) RENG_QA(8, 2) RENG_QA(8, 4) RENG_QA(8, 8)
        RENG_QA(8, 16)
    }
#undef RENG_QA
#undef RENG_Q
    set_error("internal: no quantize kernel for configuration %d", key);
    return RENG_HIP_EUNSUPPORTED;
}

template <typename InT, int F>
int launch_group(const QBatch &b, int key, int scheme, float full, bool clamp, hipStream_t st) {
    if (key >= 0) {
        return clamp ? launch_fast<InT, F, true>(key, b, scheme, full, st)
                     : launch_fast<InT, F, false>(key, b, scheme, full, st);
    }
    uint64_t grid = (uint64_t)device_props().cus * 8;
    if (grid > b.total_rows) grid = b.total_rows;
    hipLaunchKernelGGL((quantize_rows_generic<InT, F>), dim3((unsigned)grid), dim3(256), 0, st, b,
                       scheme, full);
    return check_launch("quantize_rows_generic");
}

// tensor_absmax's workgroups: every piece of the batch in flight, or
// ABSMAX_BLOCKS_PER_CU per CU (128 KB of loads requested per CU).
uint32_t absmax_blocks(const QBatch &b, uint64_t epv) {
    uint64_t pieces = 0;
    for (int i = 0; i < b.n; ++i) pieces += batch_rows(b, i) * (b.m[i].cols / epv / (64 * ABSMAX_VPT) + 1);
    const uint64_t cap = std::min(device_props().cus * ABSMAX_BLOCKS_PER_CU, ABSMAX_SLOTS);
    return (uint32_t)std::min((pieces + ABSMAX_WAVES - 1) / ABSMAX_WAVES, cap);
}

template <typename InT>
int launch_hw_bias(const QBatch &b, float backoff, hipStream_t st) {
    const uint32_t blocks = absmax_blocks(b, InTraits<InT>::EPV);
    hipLaunchKernelGGL(tensor_absmax<InT>, dim3(blocks), dim3(64 * ABSMAX_WAVES), 0, st, b);
    if (const int rc = check_launch("tensor_absmax")) return rc;
    hipLaunchKernelGGL((hw_bias_kernel<InT, RENG_HIP_E4M3>), dim3((unsigned)b.n), dim3(ABSMAX_SLOTS), 0, st, b, blocks,
                       backoff);
    return check_launch("hw_bias");
}

}  // namespace

// The register-resident kernel configuration of a matrix (encode_key), or -1 when
// it must take the generic kernel (rows wider than 16 waves x 8 vectors).
int fast_key(const QMat &m, int dtype) {
    const size_t eb = dtype == RENG_HIP_BF16 ? 2 : 4;
    const size_t epv = 16 / eb;
    const size_t store = dtype == RENG_HIP_BF16 ? 8 : 4;
    const bool aligned = m.cols % epv == 0 && (reinterpret_cast<uintptr_t>(m.w) & 15) == 0 && (m.ld * eb) % 16 == 0 &&
                         (reinterpret_cast<uintptr_t>(m.codes) & (store - 1)) == 0;
    FastCfg c = pick_cfg((m.cols + epv - 1) / epv, aligned);
    if (c.mode == ROWS_ANY && c.vpt == 1 && m.cols % 64 != 0) c.mode = ROWS_SHARED;
    return c.vpt > 0 ? encode_key(c) : -1;
}

int launch_quantize_group(const QBatch &b, int dtype, int format, int scheme, float backoff,
                          int key, hipStream_t st) {
    // Scale inputs: PCS needs full = max_finite * backoff (lib.rs:535); HW needs
    // the per-matrix tensor absmax first (lib.rs:536, 545-549); UNIT is s = 1.
    const float maxf = format == RENG_HIP_E4M3 ? 240.0f : 57344.0f;
    const float full = maxf * backoff;
    // E5M2 offers one bias, its own (choose_exp_bias), so its HW scheme is s = 1
    // whatever the maximum.
    if (scheme == RENG_HIP_HW && format == RENG_HIP_E5M2) scheme = RENG_HIP_UNIT;
    if (scheme == RENG_HIP_HW) {
        const int rc = dtype == RENG_HIP_BF16 ? launch_hw_bias<uint16_t>(b, backoff, st)
                                              : launch_hw_bias<float>(b, backoff, st);
        if (rc) return rc;
    }
    // The conversions are only exact up to the format's largest finite value;
    // per-channel scales with backoff <= 1 keep |x / s| <= max_finite * (1 + 2^-23)
    // for a normal s, which rounds to the largest code without a clamp (the
    // kernel sends rows with a subnormal s to its exact path).
    const bool clamp = !(scheme == RENG_HIP_PCS && backoff <= 1.0f);
    if (dtype == RENG_HIP_BF16)
        return format == RENG_HIP_E4M3 ? launch_group<uint16_t, RENG_HIP_E4M3>(b, key, scheme, full, clamp, st)
                                       : launch_group<uint16_t, RENG_HIP_E5M2>(b, key, scheme, full, clamp, st);
    return format == RENG_HIP_E4M3 ? launch_group<float, RENG_HIP_E4M3>(b, key, scheme, full, clamp, st)
                                   : launch_group<float, RENG_HIP_E5M2>(b, key, scheme, full, clamp, st);
}

// ------------------------------------------------------------------ stream yardstick

// The quantizer's memory stream with no arithmetic: elems bf16 values in (2
// bytes each), one byte out per value (its high byte). The pattern of the
// quantizer without its arithmetic, the fastest of those measured for this
// stream: a wave takes 8 KB chunks of input (lane l: 16-byte vectors
// 64 j + l, j < 8) grid-strided over 8 waves per CU, requests the next chunk
// before it stores this one (8-byte non-temporal stores); block 0 takes the
// vectors past the last whole chunk.
__device__ __forceinline__ u32x2 high_bytes(const u32x4 &v) {
    // bytes 1 and 3 of x, y and of z, w: the high bytes of eight bf16 values
    return u32x2{__builtin_amdgcn_perm(v.y, v.x, 0x07050301u), __builtin_amdgcn_perm(v.w, v.z, 0x07050301u)};
}

__global__ __launch_bounds__(64) void stream_narrow_kernel(const u32x4 *__restrict__ src, uint64_t vecs,
                                                           u32x2 *__restrict__ dst) {
    constexpr int V = 8;
    constexpr uint64_t C = 64 * V;   // vectors per chunk
    const uint64_t chunks = vecs / C, G = gridDim.x;
    const uint32_t l = threadIdx.x;
    if (blockIdx.x == 0)
        for (uint64_t i = chunks * C + l; i < vecs; i += 64)
            __builtin_nontemporal_store(high_bytes(__builtin_nontemporal_load(src + i)), dst + i);
    uint64_t c = blockIdx.x;
    if (c >= chunks) return;
    u32x4 v[V];
#pragma unroll
    for (int j = 0; j < V; ++j) v[j] = __builtin_nontemporal_load(src + c * C + j * 64 + l);
    for (; c < chunks; c += G) {
        const bool more = c + G < chunks;
        u32x4 n[V];
        if (more) {
#pragma unroll
            for (int j = 0; j < V; ++j) n[j] = __builtin_nontemporal_load(src + (c + G) * C + j * 64 + l);
        }
#pragma unroll
        for (int j = 0; j < V; ++j) __builtin_nontemporal_store(high_bytes(v[j]), dst + c * C + j * 64 + l);
        if (more) {
#pragma unroll
            for (int j = 0; j < V; ++j) v[j] = n[j];
        }
    }
}

int launch_stream_narrow(const void *src, uint64_t elems, void *dst, hipStream_t st) {
    const uint32_t blocks = (uint32_t)device_props().cus * 8;   // 8 waves per CU
    hipLaunchKernelGGL(stream_narrow_kernel, dim3(blocks), dim3(64), 0, st, static_cast<const u32x4 *>(src),
                       elems / 8, static_cast<u32x2 *>(dst));
    return check_launch("stream_narrow");
}

int launch_row_absmax(const QBatch &b, int dtype, float *out, hipStream_t st) {
    uint64_t grid = (uint64_t)device_props().cus * 8;
    if (grid > b.total_rows) grid = b.total_rows;
    if (dtype == RENG_HIP_BF16)
        hipLaunchKernelGGL(row_absmax_kernel<uint16_t>, dim3((unsigned)grid), dim3(256), 0, st, b, out);
    else
        hipLaunchKernelGGL(row_absmax_kernel<float>, dim3((unsigned)grid), dim3(256), 0, st, b, out);
    return check_launch("row_absmax");
}

}  // namespace reng
