// SANA ReLU linear attention on the matrix cores for the head dims and types
// the one-launch kernel (linear_attn.hip) does not cover: D = 16, 64 and 128
// in any type, and fp32 input at D = 32.
//
// Three launches: the split states (linattn_wide_state_kernel), the
// fixed-order split reduction (linattn_reduce_kernel) and the output
// (linattn_wide_out_kernel).  Bound by HBM up to D = 64; fp16 and fp32 at
// D = 128 also by the fp32 matrix rate (157 TFLOP/s).  Measured on MI355X,
// whole call, against the VALU kernels (one LDS read per multiply-add), which
// stay for buffers that are not 16-byte aligned:
//   B=2, N=3001, H=18, D=64, bf16 -> fp32    293 -> 25 us (2.8 TB/s)
//   B=2, N=4096, H=35, D=64, bf16 -> fp32    44 us (4.2 TB/s; state kernel 16,
//                                            output kernel 26)
//   B=2, N=4096, H=70, D=32, fp32            61 us (4.8 TB/s)
//   B=2, N=4096, H=17, D=128, fp32           125 us (2.3 TB/s)
//
// Arithmetic.  Products and sums are fp32 as on the VALU path:
//   state   16-bit k and v multiply exactly on the 16-bit MFMA (fp32 sums);
//           fp32 k and v use the fp32 MFMA.  Where all of k or v is subnormal
//           in its 16-bit type the unit keeps fewer bits of the sums than the
//           VALU does (relative 2-norm, N=150: fp16 values near 1e-6 6e-7
//           against 1e-7; bf16 values near 1e-39 5e-3 against 5e-6 and less).
//   output  the fp32 state is never rounded: with bf16 q it is cut into three
//           bf16 parts (8 + 8 + 8 bits, which hold an fp32 value exactly) for
//           three 16-bit MFMAs; fp16 and fp32 q use the fp32 MFMA (fp16 parts
//           would not span fp32's exponents).  The denominator is an fp32 VALU
//           dot product made while q is staged.
// ReLU is fmaxf(x, 0) in fp32, as on the VALU path.
//
// Work split.  A workgroup (8 wavefronts) owns W = 64 channels (64 / D
// adjacent heads; one head of 128 at D = 128), so that every token row it
// reads or writes is a whole 128-byte line or more, and a run of tokens.
// Tiles go global -> registers (two tiles in flight) -> LDS.
#pragma once

#include <type_traits>

#include "kf_common.h"

namespace kf {
namespace {

constexpr int kWideThreads = 512;

// LOADS: 16-byte loads per thread and tile of one qkv part.
template <typename T, int D, int LOADS> struct WideTile {
    static constexpr int HG = D >= 64 ? 1 : 64 / D;       // heads per workgroup
    static constexpr int W = HG * D;                      // channels per workgroup
    static constexpr int EPC = 16 / (int)sizeof(T);       // elements per 16-byte chunk
    static constexpr int CPR = W / EPC;                   // chunks per token row
    static constexpr int TPL = kWideThreads / CPR;        // tokens per load of the workgroup
    static constexpr int TT = LOADS * TPL;                // tokens per tile
};

// One chunk as fp32 with ReLU, and back (relu(x) is representable, so the
// conversions are exact).
template <typename T> __device__ __forceinline__ void unpack_relu(u32x4 raw, float (&f)[16 / sizeof(T)]) {
    const T* e = reinterpret_cast<const T*>(&raw);
#pragma unroll
    for (int i = 0; i < 16 / (int)sizeof(T); ++i) f[i] = fmaxf(to_f32(e[i]), 0.f);
}
template <typename T> __device__ __forceinline__ u32x4 pack_chunk(const float (&f)[16 / sizeof(T)]) {
    u32x4 r;
    if constexpr (sizeof(T) == 4) {
#pragma unroll
        for (int i = 0; i < 4; ++i) r[i] = __float_as_uint(f[i]);
    } else if constexpr (__is_same(T, bf16)) {
#pragma unroll
        for (int i = 0; i < 4; ++i)
            r[i] = __builtin_amdgcn_perm(__float_as_uint(f[2 * i + 1]), __float_as_uint(f[2 * i]), 0x07060302u);
    } else {
        T* e = reinterpret_cast<T*>(&r);
#pragma unroll
        for (int i = 0; i < 8; ++i) e[i] = from_f32<T>(f[i]);
    }
    return r;
}

// Workgroup barrier that leaves global loads in flight (LDS traffic only).
__device__ __forceinline__ void wide_barrier() {
    __builtin_amdgcn_s_waitcnt(0xC07F);  // lgkmcnt(0); vmcnt and expcnt untouched
    asm volatile("" ::: "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
}

__device__ __forceinline__ f32x4 mfma16x16x16(V<bf16>::x4 a, V<bf16>::x4 b, f32x4 c) {
    typedef short s16x4 __attribute__((ext_vector_type(4)));
    return __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(__builtin_bit_cast(s16x4, a), __builtin_bit_cast(s16x4, b), c,
                                                     0, 0, 0);
}

// ---------------------------------------------------------------------------
// State: partial[b][h][s] = (V^T relu(K), sum relu(K)) over the split's tokens.
// ---------------------------------------------------------------------------
// LDS tiles [TT][W] of K and of V.  16-bit tiles are read column-wise
// (ds_read_b64_tr_b16: rows 8i..8i+3 of two or four i, 64 or 32 bytes each);
// the chunk xor sends those rows to distinct 64-byte (W = 64: 32-byte) slots.
// fp32 tiles are read 32 consecutive floats of two rows at a time and need
// none.
template <typename T, int W> __device__ __forceinline__ int wide_swz(int row) {
    if constexpr (sizeof(T) == 4) return 0;
    else if constexpr (W == 64) return ((((row >> 1) ^ (row >> 3)) & 1) << 2) | (((row >> 4) & 1) << 1);
    else return (((row ^ (row >> 3)) & 1) << 2) | (((row >> 1) & 1) << 3);
}

template <typename T, int D>
__global__ __launch_bounds__(kWideThreads) void linattn_wide_state_kernel(const T* __restrict__ qkv,
                                                                          float* __restrict__ partial, int N,
                                                                          int H, int ngroups, int split_len,
                                                                          int splits) {
    typedef WideTile<T, D, 2> Cf;
    constexpr int W = Cf::W, EPC = Cf::EPC, CPR = Cf::CPR, TPL = Cf::TPL, TT = Cf::TT, HG = Cf::HG;
    constexpr int MB = D < 32 ? 16 : 32;                    // MFMA block edge
    constexpr int NBR = D / MB;                             // MFMA blocks per side of a head's state
    constexpr int NBLK = HG * NBR * NBR;
    constexpr int WPB = NBLK >= 8 ? 1 : 8 / NBLK;           // wavefronts (token slices) per block
    constexpr int BPW = NBLK > 8 ? NBLK / 8 : 1;            // blocks per wavefront (one row of blocks)
    constexpr int TS = TT / WPB;                            // tokens per slice
    constexpr int KST = sizeof(T) == 4 ? (MB == 32 ? 2 : 4) : (MB == 32 ? 16 : 32);  // tokens per MFMA
    constexpr int NACC = MB == 32 ? 16 : 4;
    static_assert(TS % KST == 0 && BPW <= NBR, "slices are whole MFMA steps");
    constexpr int TILE = TT * W;                            // elements
    typedef float accv __attribute__((ext_vector_type(NACC)));
    __shared__ __attribute__((aligned(16))) T lds[4 * TILE];  // [buffer][K, V][TT][W]
    constexpr int COMB = NBLK * (WPB - 1) * 64 * NACC;      // floats: the slices' accumulators, then z
    static_assert((COMB + TPL * W) * 4 <= 4 * TILE * (int)sizeof(T), "combine buffer fits");

    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int g = blockIdx.x, s = blockIdx.y;
    const int b = g / ngroups, h0 = (g - b * ngroups) * HG;
    const int64_t C = (int64_t)H * D;
    const int t_begin = s * split_len, t_end = min(N, t_begin + split_len);
    const int ntile = (t_end - t_begin + TT - 1) / TT;
    const int ltok = tid / CPR, lch = tid % CPR;
    // A chunk past the last head re-reads channel 0 of the group and is zeroed.
    const bool ch_ok = (int64_t)h0 * D + lch * EPC < C;
    const T* base = qkv + (int64_t)b * N * 3 * C + C + (int64_t)h0 * D + (ch_ok ? lch * EPC : 0);

    auto gload = [&](u32x4 (&kr)[2], u32x4 (&vr)[2], int t0) {
#pragma unroll
        for (int i = 0; i < 2; ++i) {
            const T* src = base + (int64_t)min(t0 + i * TPL + ltok, t_end - 1) * 3 * C;
            kr[i] = __builtin_nontemporal_load(reinterpret_cast<const u32x4*>(src));
            vr[i] = __builtin_nontemporal_load(reinterpret_cast<const u32x4*>(src + C));
        }
    };
    float zacc[EPC];
#pragma unroll
    for (int e = 0; e < EPC; ++e) zacc[e] = 0.f;
    auto stage = [&](const u32x4 (&kr)[2], const u32x4 (&vr)[2], T* buf, int t0) {
#pragma unroll
        for (int i = 0; i < 2; ++i) {
            const int tok = i * TPL + ltok;
            const bool ok = ch_ok && t0 + tok < t_end;
            float f[EPC];
            unpack_relu<T>(kr[i], f);
#pragma unroll
            for (int e = 0; e < EPC; ++e) {
                f[e] = ok ? f[e] : 0.f;
                zacc[e] += f[e];
            }
            const int off = tok * W + ((lch ^ wide_swz<T, W>(tok)) * EPC);
            *reinterpret_cast<u32x4*>(buf + off) = pack_chunk<T>(f);
            *reinterpret_cast<u32x4*>(buf + TILE + off) = ok ? vr[i] : u32x4{0u, 0u, 0u, 0u};
        }
    };

    // This wavefront's block(s): head hh, block row rb, block columns cb0..,
    // tokens TS * slice.. of every tile.
    const int blk0 = BPW > 1 ? wave * BPW : wave % NBLK;
    const int slice = BPW > 1 ? 0 : wave / NBLK;
    const int hh = blk0 / (NBR * NBR), rb = blk0 / NBR % NBR, cb0 = blk0 % NBR;
    accv acc[BPW];
#pragma unroll
    for (int i = 0; i < BPW; ++i)
#pragma unroll
        for (int e = 0; e < NACC; ++e) acc[i][e] = 0.f;

    auto accumulate = [&](const T* buf) {
        const T* ks = buf;
        const T* vs = buf + TILE;
#pragma unroll
        for (int st = 0; st < TS / KST; ++st) {
            const int t0 = slice * TS + st * KST;
            if constexpr (sizeof(T) == 4) {
                const int row = t0 + lane / MB, col = lane % MB;
                const float a = to_f32(vs[row * W + hh * D + rb * MB + col]);
#pragma unroll
                for (int i = 0; i < BPW; ++i) {
                    const float k = to_f32(ks[row * W + hh * D + (cb0 + i) * MB + col]);
                    if constexpr (MB == 32) acc[i] = __builtin_amdgcn_mfma_f32_32x32x2f32(a, k, acc[i], 0, 0, 0);
                    else acc[i] = __builtin_amdgcn_mfma_f32_16x16x4f32(a, k, acc[i], 0, 0, 0);
                }
            } else {
                // Lane l of an MB-wide operand holds channel l % MB and 8
                // tokens 8 (l / MB)..: two transposing reads of 4 tokens.
                const int G = lane >> 4, j16 = lane & 15;
                const int row = t0 + 8 * (MB == 32 ? G >> 1 : G) + (j16 >> 2);
                const int sub = (MB == 32 ? 16 * (G & 1) : 0) + 4 * (j16 & 3);
                auto operand = [&](const T* tile, int col) {
                    const int ch = col >> 3, in = col & 7;
                    const typename V<T>::x4 lo = lds_read_tr(tile + row * W + ((ch ^ wide_swz<T, W>(row)) << 3) + in);
                    const typename V<T>::x4 hi =
                        lds_read_tr(tile + (row + 4) * W + ((ch ^ wide_swz<T, W>(row + 4)) << 3) + in);
                    typename V<T>::x8 r;
#pragma unroll
                    for (int j = 0; j < 4; ++j) {
                        r[j] = lo[j];
                        r[j + 4] = hi[j];
                    }
                    return r;
                };
                const typename V<T>::x8 a = operand(vs, hh * D + rb * MB + sub);
#pragma unroll
                for (int i = 0; i < BPW; ++i) {
                    const typename V<T>::x8 k = operand(ks, hh * D + (cb0 + i) * MB + sub);
                    if constexpr (MB == 32) acc[i] = mfma32x32x16(a, k, acc[i]);
                    else acc[i] = mfma16x16x32(a, k, acc[i]);
                }
            }
        }
    };

    // Tile it: staged to LDS buffer it & 1 from register set it & 1, whose
    // next loads (tile it + 2) start at once; one barrier per tile, since a
    // buffer is rewritten only after the barrier of the step in between.
    u32x4 k0[2], v0[2], k1[2], v1[2];
    gload(k0, v0, t_begin);
    gload(k1, v1, t_begin + TT);
    auto step = [&](int it, u32x4 (&kr)[2], u32x4 (&vr)[2]) {
        T* buf = lds + (it & 1) * 2 * TILE;
        stage(kr, vr, buf, t_begin + it * TT);
        gload(kr, vr, t_begin + (it + 2) * TT);
        wide_barrier();
        accumulate(buf);
    };
    int it = 0;
    for (; it + 2 <= ntile; it += 2) {
        step(it, k0, v0);
        step(it + 1, k1, v1);
    }
    if (it < ntile) step(it, k0, v0);

    // Slices added in slice order, z in token-row order.
    __syncthreads();
    float* comb = reinterpret_cast<float*>(lds);
    float* zl = comb + COMB;
    if constexpr (WPB > 1) {
        if (slice > 0)
            *reinterpret_cast<accv*>(comb + (((slice - 1) * NBLK + blk0) * 64 + lane) * NACC) = acc[0];
    }
#pragma unroll
    for (int e = 0; e < EPC; ++e) zl[ltok * W + lch * EPC + e] = zacc[e];
    __syncthreads();
    constexpr int SS = (D + 1) * D;
    if (slice == 0 && h0 + hh < H) {
        float* P = partial + ((int64_t)(b * H + h0 + hh) * splits + s) * SS;
        if constexpr (WPB > 1) {
#pragma unroll
            for (int q = 0; q < WPB - 1; ++q)
                acc[0] += *reinterpret_cast<const accv*>(comb + ((q * NBLK + blk0) * 64 + lane) * NACC);
        }
#pragma unroll
        for (int i = 0; i < BPW; ++i)
#pragma unroll
            for (int e = 0; e < NACC; ++e) {
                const int r = MB == 32 ? 8 * (e >> 2) + 4 * (lane >> 5) + (e & 3) : 4 * (lane >> 4) + e;
                P[(rb * MB + r) * D + (cb0 + i) * MB + lane % MB] = acc[i][e];
            }
    }
    if (tid < W && h0 + tid / D < H) {
        float z = 0.f;
        for (int r = 0; r < TPL; ++r) z += zl[r * W + tid];
        partial[((int64_t)(b * H + h0 + tid / D) * splits + s) * SS + D * D + tid % D] = z;
    }
}

// ---------------------------------------------------------------------------
// Output: out = S relu(q) / (z . relu(q) + eps).
// ---------------------------------------------------------------------------
// The wavefront (row block rb of W / MB, token group tg) keeps its MB state
// rows as A operands in registers for the whole run of tokens.  OT writes
// out[b][h*D + r][t] (fp32 only), else out[b][t][h*D + r] through an LDS tile
// so that whole token rows leave in 16-byte chunks.
template <typename T, typename TO, int D, bool OT>
__global__ __launch_bounds__(kWideThreads) __attribute__((amdgpu_waves_per_eu(4)))
void linattn_wide_out_kernel(const T* __restrict__ qkv, const float* __restrict__ state, TO* __restrict__ out,
                             int N, int H, int ngroups, int run_len, float eps) {
    static_assert(!OT || sizeof(TO) == 4, "the transposed output is fp32");
    constexpr bool SPLIT3 = __is_same(T, bf16);
    constexpr int LOADS = sizeof(T) == 4 ? 4 : 2;
    typedef WideTile<T, D, LOADS> Cf;
    typedef typename std::conditional<SPLIT3, T, float>::type TQ;   // q as staged
    constexpr int W = Cf::W, EPC = Cf::EPC, CPR = Cf::CPR, TPL = Cf::TPL, TT = Cf::TT, HG = Cf::HG;
    constexpr int MB = 16;  // state rows per wavefront (32 took twice the registers and was 5-10% slower)
    constexpr int NRB = W / MB, NTG = 8 / NRB, TPG = TT / NTG, SUB = TPG / MB;
    static_assert(SUB >= 1 && TPG % MB == 0, "token groups are whole MFMA blocks");
    constexpr int QC = W * (int)sizeof(TQ) / 16;        // chunks per staged q row
    constexpr int OC = W * (int)sizeof(TO) / 16;        // chunks per output row
    constexpr int QM = QC < 16 ? QC - 1 : 15, OM = OC < 16 ? OC - 1 : 15;
    __shared__ __attribute__((aligned(16))) unsigned char qt[TT * QC * 16];
    __shared__ __attribute__((aligned(16))) unsigned char ot[OT ? 16 : TT * OC * 16];
    __shared__ float2 inv_den[TT * HG];

    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int g = blockIdx.x;
    const int b = g / ngroups, h0 = (g - b * ngroups) * HG;
    const int64_t C = (int64_t)H * D;
    const int t_begin = blockIdx.y * run_len, t_end = min(N, t_begin + run_len);
    const int ltok = tid / CPR, lch = tid % CPR;
    const bool ch_ok = (int64_t)h0 * D + lch * EPC < C;
    const T* base = qkv + (int64_t)b * N * 3 * C + (int64_t)h0 * D + (ch_ok ? lch * EPC : 0);
    constexpr int SS = (D + 1) * D;
    const float* st0 = state + (int64_t)(b * H + h0) * SS;

    auto gload = [&](u32x4 (&qr)[LOADS], int t0) {
#pragma unroll
        for (int i = 0; i < LOADS; ++i)
            qr[i] = __builtin_nontemporal_load(reinterpret_cast<const u32x4*>(
                base + (int64_t)min(t0 + i * TPL + ltok, t_end - 1) * 3 * C));
    };
    u32x4 q0[LOADS];
    gload(q0, t_begin);

    // This thread's z values (its q chunk's channels, which lie in one head).
    // Vector loads from clamped addresses, as below: conditional scalar loads
    // wait for one another.
    float zr[EPC];
    {
        const int ch = ch_ok ? lch * EPC : 0;
        const float* zp = st0 + (int64_t)(ch / D) * SS + D * D + ch % D;
#pragma unroll
        for (int v = 0; v < EPC / 4; ++v) {
            const f32x4 z4 = *reinterpret_cast<const f32x4*>(zp + 4 * v);
#pragma unroll
            for (int e = 0; e < 4; ++e) zr[4 * v + e] = ch_ok ? z4[e] : 0.f;
        }
    }
    // State rows of this wavefront's block as A operands.
    const int rb = wave % NRB, tg = wave / NRB;
    const int hh = rb * MB / D, r0 = rb * MB % D;
    const bool head_ok = h0 + hh < H;
    const float* S = st0 + (head_ok ? (int64_t)hh * SS : 0) + (r0 + lane % MB) * D;
    constexpr int KE = SPLIT3 && D > 16 ? 8 : 4;  // elements per operand chunk and lane
    constexpr int KS = D * MB / (64 * KE);        // operand chunks
    typedef T partv __attribute__((ext_vector_type(KE)));
    partv sp[SPLIT3 ? KS : 1][3];
    f32x4 sf[SPLIT3 ? 1 : KS];
#pragma unroll
    for (int k = 0; k < KS; ++k) {
        float v[KE];
#pragma unroll
        for (int h4 = 0; h4 < KE / 4; ++h4) {
            const f32x4 s4 = *reinterpret_cast<const f32x4*>(S + (64 / MB * k + lane / MB) * KE + 4 * h4);
#pragma unroll
            for (int e = 0; e < 4; ++e) v[4 * h4 + e] = head_ok ? s4[e] : 0.f;
        }
        if constexpr (SPLIT3) {
            // Three truncated bf16 parts hold the 24 bits exactly; an infinite
            // or NaN value stays whole in the first.
#pragma unroll
            for (int e = 0; e < KE; ++e) {
                float rest = v[e];
#pragma unroll
                for (int p = 0; p < 3; ++p) {
                    const float part = __uint_as_float(__float_as_uint(rest) & 0xffff0000u);
                    const bool nan_lost = p == 0 && rest != rest;
                    sp[k][p][e] = (T)(nan_lost ? rest : part);
                    rest = p == 0 && !__builtin_isfinite(rest) ? 0.f : rest - part;
                }
            }
        } else {
            sf[k] = f32x4{v[0], v[1], v[2], v[3]};
        }
    }

    constexpr int LPH = D / EPC;  // threads per (token, head)
    auto stage = [&](const u32x4 (&qr)[LOADS]) {
#pragma unroll
        for (int i = 0; i < LOADS; ++i) {
            const int tok = i * TPL + ltok;
            float f[EPC];
            unpack_relu<T>(qr[i], f);
            float d = 0.f;
#pragma unroll
            for (int e = 0; e < EPC; ++e) {
                f[e] = ch_ok ? f[e] : 0.f;
                d = fmaf(zr[e], f[e], d);
            }
            if constexpr (sizeof(TQ) == sizeof(T)) {
                *reinterpret_cast<u32x4*>(qt + (tok * QC + (lch ^ (tok & QM))) * 16) = pack_chunk<T>(f);
            } else {
#pragma unroll
                for (int hf = 0; hf < 2; ++hf)
                    *reinterpret_cast<f32x4*>(qt + (tok * QC + ((2 * lch + hf) ^ (tok & QM))) * 16) =
                        f32x4{f[4 * hf], f[4 * hf + 1], f[4 * hf + 2], f[4 * hf + 3]};
            }
#pragma unroll
            for (int off = 1; off < LPH; off <<= 1) d += __shfl_xor(d, off, 64);
            if (lch % LPH == 0) {
                // 1 / den as a product of two factors, the second 1 unless den
                // is under 2^-124 or over 2^124: its reciprocal alone could be
                // infinite or subnormal where the quotient is neither.
                const float den = d + eps;
                const float mag = fabsf(den);
                const float up = mag < 0x1p-124f ? 0x1p64f : mag > 0x1p124f ? 0x1p-64f : 1.f;
                inv_den[tok * HG + lch / LPH] = make_float2(1.0f / (den * up), up);
            }
        }
    };
    auto contract = [&](int t0) {
#pragma unroll
        for (int u = 0; u < SUB; ++u) {
            const int tok = tg * TPG + u * MB + lane % MB;
            f32x4 acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int k = 0; k < KS; ++k) {
                // Elements (64 / MB k + l / MB) KE.. of the head's channels.
                const int el = hh * D + (64 / MB * k + lane / MB) * KE;
                const int ch = el * (int)sizeof(TQ) / 16, in = el * (int)sizeof(TQ) % 16;
                const unsigned char* p = qt + (tok * QC + (ch ^ (tok & QM))) * 16 + in;
                if constexpr (SPLIT3) {
                    const partv q = *reinterpret_cast<const partv*>(p);
#pragma unroll
                    for (int part = 2; part >= 0; --part) {
                        if constexpr (KE == 8) acc = mfma16x16x32(sp[k][part], q, acc);
                        else acc = mfma16x16x16(sp[k][part], q, acc);
                    }
                } else {
                    const f32x4 q = *reinterpret_cast<const f32x4*>(p);
#pragma unroll
                    for (int e = 0; e < 4; ++e)
                        acc = __builtin_amdgcn_mfma_f32_16x16x4f32(sf[k][e], q[e], acc, 0, 0, 0);
                }
            }
            const float2 inv = inv_den[tok * HG + hh];
            const int r = r0 + 4 * (lane >> 4);  // this lane's rows r..r+3
            if constexpr (OT) {
                if (head_ok && t0 + tok < t_end) {
                    float* dst = reinterpret_cast<float*>(out) + ((int64_t)b * C + (int64_t)(h0 + hh) * D + r) * N +
                                 t0 + tok;
#pragma unroll
                    for (int e = 0; e < 4; ++e) __builtin_nontemporal_store(acc[e] * inv.x * inv.y, dst + (int64_t)e * N);
                }
            } else {
                typedef TO out4 __attribute__((ext_vector_type(4)));
                out4 o;
#pragma unroll
                for (int e = 0; e < 4; ++e) o[e] = from_f32<TO>(acc[e] * inv.x * inv.y);
                const int off = (hh * D + r) * (int)sizeof(TO);
                *reinterpret_cast<out4*>(ot + (tok * OC + ((off >> 4) ^ (tok & OM))) * 16 + (off & 15)) = o;
            }
        }
    };
    auto store_rows = [&](int t0) {
        if constexpr (!OT) {
#pragma unroll
            for (int i = 0; i < TT * OC / kWideThreads; ++i) {
                const int c = i * kWideThreads + tid;
                const int tok = c / OC, ch = c % OC;
                const int64_t chan = (int64_t)h0 * D + ch * (16 / (int)sizeof(TO));
                if (t0 + tok < t_end && chan < C)
                    *reinterpret_cast<u32x4*>(out + ((int64_t)b * N + t0 + tok) * C + chan) =
                        *reinterpret_cast<const u32x4*>(ot + (tok * OC + (ch ^ (tok & OM))) * 16);
            }
        }
    };
    // Per tile: stage q, barrier, contract into the output tile, barrier,
    // store its rows.  The next stage() writes the q tile, which every
    // wavefront has read by then; the next contract() writes the output tile
    // after the barrier that follows these stores' LDS reads.
    for (int t0 = t_begin; t0 < t_end; t0 += TT) {
        stage(q0);
        gload(q0, t0 + TT);
        wide_barrier();
        contract(t0);
        wide_barrier();
        store_rows(t0);
    }
}

}  // namespace
}  // namespace kf
