// gemm_tiles.hip - the w8a16 product for more than 64 activation rows:
//   y[m, n] = bf16(scales[n] * sum_k x[m, k] * dec(codes[n, k]))
// with x bf16 [M, K] and the quantizer's codes [N, K] (the consumer contract
// of crates/reng-synapse/src/fp8.rs:295-331 at prefill sizes, and the m = 256
// rows crates/reng-model/src/bin/fp8_probe.rs:359-431 times).
//
// Output tiles of BM x BN on v_mfma_f32_32x32x16_bf16: a block of WGM x WGN
// waves, each owning WM x WN tiles of 32 x 32. Per stage of BK k (64 or 128)
// the activation rows (2 BK bytes each) and the code rows (BK bytes each) go global -> LDS
// through global_load_lds_dwordx4 into an S-slot ring with the XOR-swizzled
// 16-byte chunks of mfma_pipe.h. A wave reads its activation fragments as
// bf16 (one ds_read_b128 per 32-row tile and 16-k step) and its code
// fragments as fp8 bytes (one ds_read_b128 per two k-steps), decodes the codes
// to bf16 in registers with v_cvt_scalef32_pk_bf16_fp8/bf8 (exact), and feeds both to the
// MFMA with f32 accumulation; the per-channel scale is applied once per output
// in the epilogue. The codes cross HBM once per tile row of the grid; tiles
// run in XCD-major order with m fastest, so the blocks on one XCD that share
// a code tile read it through that XCD's L2.
#include <type_traits>

#include "common.h"
#include "gemm.h"
#include "mfma_pipe.h"
#include "tile_forms.h"

namespace reng {

namespace tiles {

using namespace pipe;

typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));

// What a copy past a row's end reads (TAIL).
static __device__ const uint32_t zero_chunk[4] __attribute__((aligned(16))) = {0, 0, 0, 0};

// BK codes of k per pipeline stage (64 or 128).
template <int WGM, int WGN, int WM, int WN, int BK>
struct Tile {
    static_assert(BK == 64 || BK == 128, "stage widths");
    static constexpr int W = WGM * WGN;
    static constexpr int BM = 32 * WM * WGM, BN = 32 * WN * WGN;
    static constexpr int A_ROW = 2 * BK, B_ROW = BK;            // bytes of one activation / code row per stage
    static constexpr int CHA = A_ROW / 16, CHB = B_ROW / 16;    // 16-byte chunks of a row
    static constexpr int RA = 1024 / A_ROW, RB = 1024 / B_ROW;  // rows of a 1 KB copy
    static constexpr int PAIRS = BK / 32;                       // pairs of 16-k MFMA k-steps per stage
    static constexpr int A_BYTES = BM * A_ROW, B_BYTES = BN * B_ROW, STAGE = A_BYTES + B_BYTES;
    static constexpr int LA = BM / RA / W, LB = BN / RB / W;    // copies per wave per stage
    static constexpr int LOADS = LA + LB;
    static_assert(LA * RA * W == BM && LB * RB * W == BN, "copies split evenly over the waves");
};

// Chunk slots: chunk c of tile row r sits in slot c ^ swz(r). Activation rows
// (8 or 16 chunks) XOR the low three bits of c; code rows use the 4-chunk
// permutation of mfma_pipe.h for 4 chunks, else the 8-chunk one.
__device__ __forceinline__ uint32_t swz_a(uint32_t r) { return swz<8>(r); }
template <int CHB>
__device__ __forceinline__ uint32_t swz_b(uint32_t r) { return swz<CHB == 4 ? 4 : 8>(r); }

// Two fp8 codes of each 16-bit half of w -> bf16 pairs (exact).
template <int F>
__device__ __forceinline__ uint32_t dec_pair(uint32_t w, bool hi);
template <>
__device__ __forceinline__ uint32_t dec_pair<RENG_HIP_E4M3>(uint32_t w, bool hi) {
    return __builtin_bit_cast(uint32_t, hi ? __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(w, 1.0f, true)
                                           : __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(w, 1.0f, false));
}
template <>
__device__ __forceinline__ uint32_t dec_pair<RENG_HIP_E5M2>(uint32_t w, bool hi) {
    return __builtin_bit_cast(uint32_t, hi ? __builtin_amdgcn_cvt_scalef32_pk_bf16_bf8(w, 1.0f, true)
                                           : __builtin_amdgcn_cvt_scalef32_pk_bf16_bf8(w, 1.0f, false));
}

// Work units are (tile, stage) pairs, unit u = tile * n + stage with n = K / BK
// stages per tile. Without SK a block takes one tile's n units, tiles in
// XCD-major order with m fastest. With SK (stream-K) the grid is persistent
// and block b takes units [b U / G, (b + 1) U / G) of all U = tiles * n, so
// every CU gets the same number of stages whatever the tile count; the copy
// pipeline runs straight across tile boundaries. A tile whose units span
// several blocks is finished by the last of them to arrive: each writes its
// partial sums to part (slot b + tile), releases them and increments
// cnt[tile]; the block that sees the
// count reach the segment count adds the partials in block order (the same
// order whichever block arrives last, so the sum is deterministic), writes the
// tile and resets the counter to zero for the next launch. No block waits for
// another.
//
// With TAIL (no SK), K is any multiple of 16 and the last stage is short: a
// lane whose 16-byte chunk lies past its row's end copies zeros instead, in
// both operands, so the chunk adds exact zeros to the sums. The check costs a
// compare and two selects per copy, so whole stages take the form without it.
template <int F, int WGM, int WGN, int WM, int WN, int BK, int S, bool SK, bool TAIL>
__global__ __launch_bounds__(64 * WGM * WGN) void w8a16_tiles(const uint16_t *__restrict__ x,
                                                              const uint8_t *__restrict__ codes,
                                                              const float *__restrict__ scales, uint32_t M,
                                                              uint32_t N, uint32_t K, uint32_t tiles_m,
                                                              uint32_t tiles, uint16_t *__restrict__ y,
                                                              uint32_t vec_out, float *__restrict__ part,
                                                              uint32_t *__restrict__ cnt) {
    using T = Tile<WGM, WGN, WM, WN, BK>;
    constexpr int BM = T::BM, BN = T::BN, NQ = WM * WN;
    constexpr int A_ROW = T::A_ROW, B_ROW = T::B_ROW, CHA = T::CHA, CHB = T::CHB, PAIRS = T::PAIRS;
    static_assert(S >= 2, "at least double-buffered");
    static_assert((S - 1) * T::LOADS < 64, "vmcnt range");
    static_assert(!(SK && TAIL), "stream-K stages are whole");
    __shared__ __attribute__((aligned(1024))) uint8_t lds[S * T::STAGE];
    __shared__ uint32_t last_flag;
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wm = wave / WGN, wn = wave % WGN;
    const uint32_t n = TAIL ? (K + BK - 1) / BK : K / BK;   // stages per tile
    const uint64_t U = (uint64_t)tiles * n, G = gridDim.x;

    uint64_t ub, ue;   // this block's units
    if constexpr (SK) {
        ub = (uint64_t)blockIdx.x * U / G;
        ue = (uint64_t)(blockIdx.x + 1) * U / G;
    } else {
        const uint32_t xcd = blockIdx.x % XCDS, l = blockIdx.x / XCDS;
        const uint32_t per = tiles / XCDS, rem = tiles % XCDS;
        ub = (uint64_t)(xcd * per + (xcd < rem ? xcd : rem) + l) * n;
        ue = ub + n;
    }
    if (ub >= ue) return;   // (SK) more blocks than units: nothing for this one
    const uint32_t L = (uint32_t)(ue - ub);
    // Under SK: the block holding unit u.
    auto block_of = [&](uint64_t u) { return (uint32_t)(((u + 1) * G - 1) / U); };

    // Copy sources: lane l of activation copy c brings tile row RA c + l / CHA
    // and the chunk stored in slot l % CHA of it; of code copy c, row
    // RB c + l / CHB, slot l % CHB. Rows past M / N are clamped (never stored).
    uint32_t tra[T::LA], ofa[T::LA], trb[T::LB], ofb[T::LB];
#pragma unroll
    for (int q = 0; q < T::LA; ++q) {
        tra[q] = (wave * T::LA + q) * T::RA + lane / CHA;
        ofa[q] = ((lane % CHA) ^ swz_a(tra[q])) * 16;
    }
#pragma unroll
    for (int q = 0; q < T::LB; ++q) {
        trb[q] = (wave * T::LB + q) * T::RB + lane / CHB;
        ofb[q] = ((lane % CHB) ^ swz_b<CHB>(trb[q])) * 16;
    }
    // Copies come in unit order; past the block's last unit they repeat it
    // (surplus copies, never read). Without SK the block's rows are fixed:
    // per-lane pointers plus a stage offset. Under SK a cursor (tile row-block
    // tm, column-block tn, stage ks) follows the copies across tiles.
    const uint32_t t_first = (uint32_t)(ub / n), s_first = (uint32_t)(ub % n);
    uint32_t c_tm = t_first % tiles_m, c_tn = t_first / tiles_m, c_ks = s_first, issued = 0;
    const uint8_t *ga[T::LA];
    const uint8_t *gb[T::LB];
    if constexpr (!SK) {
#pragma unroll
        for (int q = 0; q < T::LA; ++q) {
            const uint32_t r = c_tm * BM + tra[q] < M ? c_tm * BM + tra[q] : M - 1;
            ga[q] = reinterpret_cast<const uint8_t *>(x) + (size_t)r * K * 2 + ofa[q];
        }
#pragma unroll
        for (int q = 0; q < T::LB; ++q) {
            const uint32_t r = c_tn * BN + trb[q] < N ? c_tn * BN + trb[q] : N - 1;
            gb[q] = codes + (size_t)r * K + ofb[q];
        }
    }
    auto issue = [&](int slot) __attribute__((always_inline)) {
        uint8_t *base = lds + slot * T::STAGE;
        if constexpr (!SK) {
            const uint32_t st = issued < L ? issued : L - 1;
            ++issued;
            const uint8_t *zero = reinterpret_cast<const uint8_t *>(zero_chunk);
#pragma unroll
            for (int q = 0; q < T::LA; ++q) {
                const uint8_t *src = ga[q] + (size_t)st * A_ROW;
                if constexpr (TAIL) src = st * A_ROW + ofa[q] < 2 * K ? src : zero;
                copy16_to_lds(src, base + (wave * T::LA + q) * 1024);
            }
#pragma unroll
            for (int q = 0; q < T::LB; ++q) {
                const uint8_t *src = gb[q] + (size_t)st * B_ROW;
                if constexpr (TAIL) src = st * B_ROW + ofb[q] < K ? src : zero;
                copy16_to_lds(src, base + T::A_BYTES + (wave * T::LB + q) * 1024);
            }
            return;
        }
        const uint32_t m0 = c_tm * BM, n0 = c_tn * BN, st = c_ks;
        // Advance without branches (selects on wave-uniform values), so the
        // copies stay in the scheduling region of the MFMAs around them.
        const uint32_t adv = ++issued < L ? 1u : 0u;
        const uint32_t ks1 = c_ks + adv, wrap = ks1 == n ? 1u : 0u;
        const uint32_t tm1 = c_tm + wrap, wrap2 = tm1 == tiles_m ? 1u : 0u;
        c_ks = wrap ? 0u : ks1;
        c_tm = wrap2 ? 0u : tm1;
        c_tn += wrap2;
#pragma unroll
        for (int q = 0; q < T::LA; ++q) {
            const uint32_t r = m0 + tra[q] < M ? m0 + tra[q] : M - 1;
            copy16_to_lds(reinterpret_cast<const uint8_t *>(x) + (size_t)r * K * 2 + (size_t)st * A_ROW + ofa[q],
                          base + (wave * T::LA + q) * 1024);
        }
#pragma unroll
        for (int q = 0; q < T::LB; ++q) {
            const uint32_t r = n0 + trb[q] < N ? n0 + trb[q] : N - 1;
            copy16_to_lds(codes + (size_t)r * K + (size_t)st * B_ROW + ofb[q],
                          base + T::A_BYTES + (wave * T::LB + q) * 1024);
        }
    };

    // Fragments come in pairs of k-steps (32 k). Lane l holds row l % 32 of a
    // 32-row tile; half h = l / 32 has the 16 codes of chunk 2 p + h of pair p,
    // the first 8 for its first k-step and the last 8 for its second, and the
    // activations of the same k (chunks 4 p + 2 h and 4 p + 2 h + 1). Every read
    // is a ds_read_b128 (8-byte code reads of one half of each chunk use half
    // the banks), and a pair's reads have 2 WM WN MFMAs to land behind: with
    // one k-step per fragment set the LDS latency (two waves per SIMD, one or
    // two MFMAs each) showed in every k-step. One k-step -> pairs, same box:
    // M = 256 [4096, 4096] 21.4 -> 18.2 us, [14336, 4096] 36.2 -> 33.8,
    // [4096, 14336] 66.0 -> 60.1, M = 512 [5120, 5120] 40.0 -> 35.1, M = 1024
    // [14336, 4096] 108 -> 105, [27648, 5120] 260 -> 249. (128 x 128 on four
    // waves of 64 x 64, half the LDS reads: 39.0 against 37.6 us on M = 256
    // [14336, 4096] past the Infinity Cache.)
    const uint32_t rl = lane & 31, h = lane >> 5, swa = swz_a(rl), swb = swz_b<CHB>(rl);
    auto read_pair = [&](int slot, int p, u32x4 (&fa)[2][WM], u32x4 (&fb)[WN]) __attribute__((always_inline)) {
        const uint8_t *base = lds + slot * T::STAGE;
        const uint32_t ob = ((2 * p + h) ^ swb) * 16;
#pragma unroll
        for (int j = 0; j < WN; ++j)
            fb[j] = *reinterpret_cast<const u32x4 *>(base + T::A_BYTES + (wn * (32 * WN) + j * 32 + rl) * B_ROW + ob);
#pragma unroll
        for (int ks = 0; ks < 2; ++ks) {
            const uint32_t oa = ((4 * p + 2 * h + ks) ^ swa) * 16;
#pragma unroll
            for (int i = 0; i < WM; ++i)
                fa[ks][i] = *reinterpret_cast<const u32x4 *>(base + (wm * (32 * WM) + i * 32 + rl) * A_ROW + oa);
        }
    };

    f32x16 acc[WM][WN];
    auto zero_acc = [&]() __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < WM; ++i)
#pragma unroll
            for (int j = 0; j < WN; ++j)
#pragma unroll
                for (int e = 0; e < 16; ++e) acc[i][j][e] = 0.0f;
    };
    zero_acc();

    // The MFMAs of a pair of k-steps; the code fragments are decoded as they
    // are used. D = codes x^T: rows n, columns m.
    auto mfma_pair = [&](const u32x4 (&fa)[2][WM], const u32x4 (&fb)[WN]) __attribute__((always_inline)) {
#pragma unroll
        for (int ks = 0; ks < 2; ++ks) {
            u32x4 wb[WN];
#pragma unroll
            for (int j = 0; j < WN; ++j) {
                const uint32_t lo = ks ? fb[j].z : fb[j].x, hi = ks ? fb[j].w : fb[j].y;
                wb[j] = u32x4{dec_pair<F>(lo, false), dec_pair<F>(lo, true), dec_pair<F>(hi, false),
                              dec_pair<F>(hi, true)};
            }
#pragma unroll
            for (int q = 0; q < NQ; ++q) {
                const int i = q / WN, j = q % WN;
                acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, wb[j]),
                                                                    __builtin_bit_cast(bf16x8, fa[ks][i]), acc[i][j],
                                                                    0, 0, 0);
            }
        }
    };

    // Lane l holds output row m = ... + l % 32 and, per group g of four
    // accumulators, the four consecutive columns n = ... + 8 g + 4 h + e.
    const float *sp = scales ? scales : &one_f32;   // (pointer, stride): no branch per scale
    const uint32_t ss = scales != nullptr;
    auto store_tile = [&](uint32_t t) __attribute__((always_inline)) {
        const uint32_t m0 = (t % tiles_m) * BM, n0 = (t / tiles_m) * BN;
#pragma unroll
        for (int i = 0; i < WM; ++i) {
            const uint32_t m = m0 + wm * (32 * WM) + i * 32 + rl;
            if (m >= M) continue;
            uint16_t *orow = y + (size_t)m * N;
#pragma unroll
            for (int j = 0; j < WN; ++j)
#pragma unroll
                for (int g = 0; g < 4; ++g) {
                    const uint32_t nb = n0 + wn * (32 * WN) + j * 32 + 8 * g + 4 * h;
                    float o[4];
#pragma unroll
                    for (int e = 0; e < 4; ++e) {
                        const uint32_t nn = nb + e < N ? nb + e : N - 1;
                        o[e] = acc[i][j][4 * g + e] * sp[nn * ss];
                    }
                    if (vec_out && nb + 3 < N) {
                        const uint32_t lo = f32_to_bf16_bits(o[0]) | (f32_to_bf16_bits(o[1]) << 16);
                        const uint32_t hi = f32_to_bf16_bits(o[2]) | (f32_to_bf16_bits(o[3]) << 16);
                        *reinterpret_cast<u32x2 *>(orow + nb) = u32x2{lo, hi};
                    } else {
#pragma unroll
                        for (int e = 0; e < 4; ++e)
                            if (nb + e < N) orow[nb + e] = (uint16_t)f32_to_bf16_bits(o[e]);
                    }
                }
        }
    };
    // The block's only tile (without SK), once no copy into the ring is in
    // flight: the scaled bf16 values go to a row-major BM x BN tile in LDS
    // (16-byte chunk c of row r in slot slot(r, c): c ^ (r % CC) for a
    // power-of-two CC, else (c + r) % CC), then the block stores whole tile
    // rows, 16 bytes per lane, rather than 8 bytes of each of 32 rows per
    // store instruction.
    auto store_tile_lds = [&](uint32_t t) __attribute__((always_inline)) {
        constexpr int CC = BN / 8, RB = BN * 2, NT = 64 * T::W;   // chunks, bytes of a tile row; threads
        static_assert(S * T::STAGE >= BM * RB, "the output tile fits the operand ring");
        static_assert((BM * CC) % NT == 0, "whole passes");
        auto slot = [](uint32_t r, uint32_t c) -> uint32_t {
            if constexpr ((CC & (CC - 1)) == 0) return c ^ (r % CC);
            else return (c + r) % CC;
        };
        const uint32_t m0 = (t % tiles_m) * BM, n0 = (t / tiles_m) * BN;
        wait_vmcnt<0>();
        __syncthreads();
        // The lane index through an empty asm: the epilogue's addresses are
        // computed here rather than hoisted before the main loop (where they
        // would hold registers through it).
        uint32_t te = tid;
        asm volatile("" : "+v"(te));
        const uint32_t rle = te & 31, he = (te >> 5) & 1;
#pragma unroll
        for (int i = 0; i < WM; ++i) {
            const uint32_t r = wm * (32 * WM) + i * 32 + rle;
#pragma unroll
            for (int j = 0; j < WN; ++j)
#pragma unroll
                for (int g = 0; g < 4; ++g) {
                    const uint32_t c = wn * (4 * WN) + 4 * j + g;   // columns 8 c .. 8 c + 7 of the tile
                    const uint32_t nb = n0 + 8 * c + 4 * he;
                    float o[4];
#pragma unroll
                    for (int e = 0; e < 4; ++e) {
                        const uint32_t nn = nb + e < N ? nb + e : N - 1;
                        o[e] = acc[i][j][4 * g + e] * sp[nn * ss];
                    }
                    const uint32_t lo = f32_to_bf16_bits(o[0]) | (f32_to_bf16_bits(o[1]) << 16);
                    const uint32_t hi = f32_to_bf16_bits(o[2]) | (f32_to_bf16_bits(o[3]) << 16);
                    *reinterpret_cast<u32x2 *>(lds + r * RB + slot(r, c) * 16 + 8 * he) = u32x2{lo, hi};
                }
        }
        __syncthreads();
#pragma unroll
        for (int p = 0; p < BM * CC / NT; ++p) {
            const uint32_t ix = p * NT + te, r = ix / CC, c = ix % CC, m = m0 + r, nc = n0 + 8 * c;
            if (m >= M || nc >= N) continue;
            const u32x4 v = *reinterpret_cast<const u32x4 *>(lds + r * RB + slot(r, c) * 16);
            uint16_t *dst = y + (size_t)m * N + nc;
            if (vec_out && nc + 8 <= N) {
                // Non-temporal, as the fp8 GEMM's epilogue (same-box A/B: equal or
                // 0.5-2.5% faster on every tile form's product, M = 256 [14336,
                // 4096] 39.5 -> 38.9 us).
                __builtin_nontemporal_store(v, reinterpret_cast<u32x4 *>(dst));
            } else {
                const uint32_t w[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
                for (int e = 0; e < 8; ++e)
                    if (nc + e < N) dst[e] = (uint16_t)(w[e / 2] >> (16 * (e % 2)));
            }
        }
    };
    // A partial slot holds BM x BN floats: wave w's WM WN 16 accumulators,
    // each as 64 consecutive floats (one per lane). Block b's segment of tile
    // t uses slot b + t: distinct for every (block, tile) pair that meets,
    // since a block only moves to later tiles than the block before it.
    constexpr uint32_t SLOT = BM * BN, WAVE_PART = NQ * 16 * 64;
    auto slot_ptr = [&](uint32_t b, uint32_t t) __attribute__((always_inline)) -> float * {
        return part + ((size_t)b + t) * SLOT + (size_t)wave * WAVE_PART + lane;
    };
    // The end of the block's run on tile t (its last unit u).
    auto finish = [&](uint32_t t) __attribute__((always_inline)) {
        if constexpr (SK) {
            const uint64_t t0 = (uint64_t)t * n;
            if (!(ub <= t0 && ue >= t0 + n)) {
                const uint32_t b0 = block_of(t0), b1 = block_of(t0 + n - 1);
                // Partials and counter go through agent-scope (device-coherent)
                // accesses, which bypass the per-XCD L2s' non-coherent copies;
                // the stores have completed (vmcnt 0) before the count moves.
                // The count is an acquire-release: the block's stores (ordered
                // before it by the barrier) happen before the last block's
                // reads (ordered after its own count by the next barrier).
                float *mine = slot_ptr(blockIdx.x, t);
#pragma unroll
                for (int q = 0; q < NQ; ++q)
#pragma unroll
                    for (int e = 0; e < 16; ++e)
                        __hip_atomic_store(mine + (q * 16 + e) * 64, acc[q / WN][q % WN][e], __ATOMIC_RELAXED,
                                           __HIP_MEMORY_SCOPE_AGENT);
                wait_vmcnt<0>();
                __syncthreads();
                if (tid == 0) {
                    const uint32_t seen = __hip_atomic_fetch_add(cnt + t, 1u, __ATOMIC_ACQ_REL,
                                                                 __HIP_MEMORY_SCOPE_AGENT);
                    last_flag = seen + 1 == b1 - b0 + 1;
                }
                __syncthreads();
                const bool last = last_flag != 0;
                if (last) {
                    zero_acc();
                    for (uint32_t b = b0; b <= b1; ++b) {
                        float *p = slot_ptr(b, t);
#pragma unroll
                        for (int q = 0; q < NQ; ++q)
#pragma unroll
                            for (int e = 0; e < 16; ++e)
                                acc[q / WN][q % WN][e] += __hip_atomic_load(p + (q * 16 + e) * 64, __ATOMIC_RELAXED,
                                                                            __HIP_MEMORY_SCOPE_AGENT);
                    }
                    store_tile(t);
                    if (tid == 0) __hip_atomic_store(cnt + t, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                }
                __syncthreads();   // last_flag is rewritten at the next tile's end
                zero_acc();
                return;
            }
        }
        if constexpr (SK) store_tile(t);
        else store_tile_lds(t);
        zero_acc();
    };

    // The pipeline of gemm_fp8_mfma: S stages in flight from the prologue;
    // per stage one barrier once each wave's own copies of the next stage
    // have landed, then the copy of stage i + S into the slot stage i used.
#pragma unroll
    for (int s = 0; s < S; ++s) issue(s);
    wait_vmcnt<(S - 1) * T::LOADS>();
    lds_barrier();
    u32x4 fa[2][2][WM], fb[2][WN];
    read_pair(0, 0, fa[0], fb[0]);
    // Pair PI of stage i on fragment set PI & 1, the next pair's fragments
    // going into the other set. The stage's last pair starts with the barrier
    // that publishes stage i + 1 and frees stage i's slot.
    auto pair = [&](auto pi_c, uint32_t i) __attribute__((always_inline)) {
        constexpr int PI = decltype(pi_c)::value, CUR = PI & 1, NXT = CUR ^ 1;
        if constexpr (PI + 1 < PAIRS) {
            read_pair((int)(i % S), PI + 1, fa[NXT], fb[NXT]);
            mfma_pair(fa[CUR], fb[CUR]);
            interleave<2 * NQ, 2 * WM + WN, 0>();
            __builtin_amdgcn_sched_barrier(0);
        } else {
            wait_lgkm0();   // the stage's last fragments are in registers
            wait_vmcnt<(S - 2) * T::LOADS>();
            lds_barrier();
            issue((int)(i % S));
            read_pair((int)((i + 1) % S), 0, fa[NXT], fb[NXT]);
            mfma_pair(fa[CUR], fb[CUR]);
            interleave<2 * NQ, 2 * WM + WN, T::LOADS>();
            __builtin_amdgcn_sched_barrier(0);
        }
    };
    static_assert(PAIRS % 2 == 0, "the fragment sets alternate within a stage");
    auto stage = [&](auto self, auto pi_c, uint32_t i) __attribute__((always_inline)) {
        constexpr int PI = decltype(pi_c)::value;
        pair(pi_c, i);
        if constexpr (PI + 1 < PAIRS) self(self, std::integral_constant<int, PI + 1>{}, i);
    };
    // The block's units tile by tile: a run of stages, then the tile's end.
    uint32_t i = 0, f_t = t_first, f_ks = s_first;
    while (i < L) {
        const uint32_t run = n - f_ks < L - i ? n - f_ks : L - i;
        for (uint32_t r = 0; r < run; ++r, ++i) stage(stage, std::integral_constant<int, 0>{}, i);
        finish(f_t);
        f_ks = 0;
        ++f_t;
    }
    wait_vmcnt<0>();   // the clamped surplus copies land before LDS is released
}

// One launch; under SK, `part` holds (G + tiles - 1) BM BN floats and `cnt`
// one zeroed counter per tile (left zeroed by the launch) for a grid of G
// blocks.
template <int F, int WGM, int WGN, int WM, int WN, int BK, int S, bool SK, bool TAIL = false>
int launch_tiles_cfg(const uint16_t *x, const uint8_t *codes, const float *scales, uint32_t M, uint32_t N,
                     uint32_t K, uint16_t *y, hipStream_t st, uint32_t grid, float *part, uint32_t *cnt) {
    using T = Tile<WGM, WGN, WM, WN, BK>;
    const uint32_t tiles_m = (M + T::BM - 1) / T::BM, tiles_n = (N + T::BN - 1) / T::BN;
    const uint32_t tiles = tiles_m * tiles_n;
    // Whole 16-byte chunks of output rows (the LDS-staged store; under SK the
    // direct store of 8-byte groups, which this implies).
    const uint32_t vec_out = N % 8 == 0 && reinterpret_cast<uintptr_t>(y) % 16 == 0;
    if (!SK) grid = tiles;
    hipLaunchKernelGGL((w8a16_tiles<F, WGM, WGN, WM, WN, BK, S, SK, TAIL>), dim3(grid), dim3(64 * T::W), 0, st, x, codes,
                       scales, M, N, K, tiles_m, tiles, y, vec_out, part, cnt);
    return check_launch("w8a16_tiles");
}

template <int F>
int launch_tiles_f(const uint16_t *x, const uint8_t *codes, const float *scales, uint32_t M, uint32_t N,
                   uint32_t K, uint16_t *y, hipStream_t st, const SplitScratch *fixed) {
    const uint64_t cus = (uint64_t)device_props().cus;
    const uint64_t t128 = tile_count(M, N, 128, 128);
    if (streamk_suits(M, N, K, cus)) {
        using T = Tile<2, 4, 2, 1, 128>;
        const uint64_t units = t128 * (K / 128);
        const uint32_t grid = (uint32_t)(units < cus ? units : cus);
        const size_t floats = ((size_t)grid + t128 - 1) * T::BM * T::BN;
        int rc = RENG_HIP_OK;
        float *part = split_partials(floats, st, fixed, &rc);
        if (rc) return rc;
        uint32_t *cnt = fixed ? static_tile_counters(&rc) : tile_counters((uint32_t)t128, st, &rc);
        if (rc) return rc;
        return launch_tiles_cfg<F, 2, 4, 2, 1, 128, 3, true>(x, codes, scales, M, N, K, y, st, grid, part, cnt);
    }
    const bool tail = K % 64 != 0;   // a short last stage: every form takes it
#define RENG_TILES(...)                                                                                          \
    return tail ? launch_tiles_cfg<F, __VA_ARGS__, false, true>(x, codes, scales, M, N, K, y, st, 0, nullptr, nullptr) \
                : launch_tiles_cfg<F, __VA_ARGS__, false>(x, codes, scales, M, N, K, y, st, 0, nullptr, nullptr)
    // Whole 128-code stages copy the codes in 128-byte pieces rather than 64
    // (of L2-resident rows a CU takes in 125 GB/s of the former, 69-93 of the
    // latter). Same box, 64- against 128-code stages: 128 x 256 M = 512 [14336,
    // 4096] 60.8 -> 58.0 us, 64 x 128 M = 128 [14336, 4096] 27.2 -> 24.9, 64 x 64
    // M = 256 [4096, 4096] 18.2 -> 17.3 (three slots: two blocks fit a CU; six:
    // 18.0). The 128 x 128 form needs the six slots (M = 512 [5120, 5120] 34.6
    // against 37.8 us), and 256 x 256 of 128-code stages does not fit.
    const bool wide = K % 128 == 0;
#define RENG_TILES_128(...)                                                                                      \
    return launch_tiles_cfg<F, __VA_ARGS__, false>(x, codes, scales, M, N, K, y, st, 0, nullptr, nullptr)
    switch (tile_pick(M, N, K, cus).form) {
    case TILES_256x256: RENG_TILES(2, 4, 4, 2, 64, 3);
    case TILES_128x256: if (wide) RENG_TILES_128(2, 4, 2, 2, 128, 2); RENG_TILES(2, 4, 2, 2, 64, 3);
    case TILES_128x160: RENG_TILES(4, 1, 1, 5, 128, 2);
    case TILES_128x128: RENG_TILES(2, 4, 2, 1, 64, 6);
    case TILES_64x128: if (wide) RENG_TILES_128(2, 4, 1, 1, 128, 4); RENG_TILES(2, 4, 1, 1, 64, 6);
    default: if (wide) RENG_TILES_128(2, 2, 1, 1, 128, 3); RENG_TILES(2, 2, 1, 1, 64, 6);
    }
#undef RENG_TILES_128
#undef RENG_TILES
}

}  // namespace tiles

bool w8a16_tiles_take(uint32_t M, uint32_t N, uint32_t K) {
    return tiles::tiles_take(M, N, K, (uint64_t)device_props().cus);
}

int launch_w8a16_tiles(const uint16_t *x, const uint8_t *codes, const float *scales, uint32_t M, uint32_t N,
                       uint32_t K, int format, uint16_t *y, hipStream_t st, const SplitScratch *fixed) {
    if (format == RENG_HIP_E4M3) return tiles::launch_tiles_f<RENG_HIP_E4M3>(x, codes, scales, M, N, K, y, st, fixed);
    return tiles::launch_tiles_f<RENG_HIP_E5M2>(x, codes, scales, M, N, K, y, st, fixed);
}

}  // namespace reng
