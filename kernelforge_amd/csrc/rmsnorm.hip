// RMSNorm forward and backward for gfx950: one HBM read of x, one write of y.
//
// Semantics follow RMSNorm.forward (rmsnorm/original.py:38, 51-52) and the
// compiled rms_norm kernel (rmsnorm/custom.py:25-73):
//   inv = 1 / sqrt(sum(x^2) / dim + eps)          (fp32 accumulation)
//   y   = ty( float(tx(x * inv)) * float(w) )     (two rounding points)
// where tx is x's storage type and ty = promote(tx, tw) is the output type:
// bf16 x with the module's default fp32 weight gives an fp32 y, as torch's
// type promotion does in `output * self.weight` (original.py:52).
// `inv` is a correctly rounded 1/sqrt (not v_rsq_f32) so that the first
// rounding point lands where the host oracle puts it.
//
// Layout: the row is split into 16-byte vectors of x; vector j of a row lives
// in lane (j % 64) of wave-slice (j / 64) % WPR at register slot j / (64*WPR),
// so every load/store instruction of a wave covers a contiguous 1 KiB span of
// x.  A row is owned by WPR waves (WPR = 1 needs no LDS and no barrier).  Rows
// of 4-16 KiB are spread over 2-8 waves with 2 vectors per lane: short-lived
// waves with few loads each kept the HBM queues fuller than long-lived ones
// in sweeps of (VPT, WPR, block size) on MI355X.  Blocks holding two rows
// stage the weight in LDS once per block: re-reading it from L2 for every row
// cost 2-3% of the HBM rate at 2048-4096 channels; with one row per block
// (8192) the staging costs more than it saves.
#include <initializer_list>
#include <type_traits>

#include "kf_common.h"

namespace kf {
namespace {

constexpr int kBlock = 256;  // 4 waves (generic kernels)

// N elements of T as one aligned register value: the slice of a row that
// matches one 16-byte vector of x.
template <typename T, int N>
struct alignas(sizeof(T) * N < 16 ? sizeof(T) * N : 16) Pack {
    T v[N];
};

// Non-temporal store of a Pack of 8, 16 or 32 bytes.
template <typename T, int N>
__device__ __forceinline__ void store_nt(Pack<T, N>* dst, const Pack<T, N>& p) {
    constexpr int BYTES = sizeof(T) * N;
    if constexpr (BYTES % 16 == 0) {
        const u32x4* s = reinterpret_cast<const u32x4*>(&p);
        u32x4* d = reinterpret_cast<u32x4*>(dst);
#pragma unroll
        for (int i = 0; i < BYTES / 16; ++i) __builtin_nontemporal_store(s[i], d + i);
    } else {
        static_assert(BYTES == 8, "packs are 8, 16 or 32 bytes");
        __builtin_nontemporal_store(*reinterpret_cast<const u32x2*>(&p), reinterpret_cast<u32x2*>(dst));
    }
}

// Non-temporal load of a Pack of 8, 16 or 32 bytes.
template <typename T, int N>
__device__ __forceinline__ Pack<T, N> load_nt(const Pack<T, N>* src) {
    constexpr int BYTES = sizeof(T) * N;
    Pack<T, N> p;
    if constexpr (BYTES % 16 == 0) {
        u32x4* d = reinterpret_cast<u32x4*>(&p);
#pragma unroll
        for (int i = 0; i < BYTES / 16; ++i) d[i] = __builtin_nontemporal_load(reinterpret_cast<const u32x4*>(src) + i);
    } else {
        static_assert(BYTES == 8, "packs are 8, 16 or 32 bytes");
        *reinterpret_cast<u32x2*>(&p) = __builtin_nontemporal_load(reinterpret_cast<const u32x2*>(src));
    }
    return p;
}

// Workgroup barrier that waits for LDS traffic only and leaves global loads
// in flight.
__device__ __forceinline__ void barrier_lds_only() {
    __builtin_amdgcn_s_waitcnt(0xC07F);  // lgkmcnt(0); vmcnt and expcnt untouched
    asm volatile("" ::: "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
}

// x and y rows start every ld_x / ld_y elements (ld >= dim); the vector path
// needs those strides, like the base pointers, aligned to the vector slices.
// y may alias x (in place, same stride and type): every row is read whole
// into registers before any of it is written.
template <typename TX, typename TW, typename TY, int VPT, int WPR, int WAVES, bool HAS_W>
__global__ __launch_bounds__(64 * WAVES) void rmsnorm_vec_kernel(const TX* x, const TW* __restrict__ w,
                                                                 TY* y, int64_t rows, int dim,
                                                                 int64_t ld_x, int64_t ld_y, float eps) {
    constexpr int VEC = 16 / sizeof(TX);
    typedef Pack<TW, VEC> WPack;
    typedef Pack<TY, VEC> YPack;
    constexpr int ROWS_PER_BLOCK = WAVES / WPR;
    const int wave = threadIdx.x >> 6;
    const int lane = threadIdx.x & 63;
    const int row_in_block = wave / WPR;
    const int slice = wave % WPR;
    const int64_t row = (int64_t)blockIdx.x * ROWS_PER_BLOCK + row_in_block;
    const bool row_ok = row < rows;
    const int nvec = dim / VEC;

    // Blocks of two or more rows read the weight once per block into LDS
    // instead of once per row (an 8 KiB L2 read per row at dim 4096).
    constexpr bool kStageW = HAS_W && WPR > 1 && ROWS_PER_BLOCK > 1;
    __shared__ WPack wl[kStageW ? VPT * WPR * 64 : 1];
    const WPack* wr = reinterpret_cast<const WPack*>(w);

    const u32x4* xr = reinterpret_cast<const u32x4*>(x + row * ld_x);
    u32x4 xv[VPT];
    float ss = 0.f;
#pragma unroll
    for (int i = 0; i < VPT; ++i) {
        const int j = (i * WPR + slice) * 64 + lane;
        if (row_ok && j < nvec) {
            xv[i] = __builtin_nontemporal_load(xr + j);
        } else {
            xv[i] = u32x4{0u, 0u, 0u, 0u};
        }
    }
    if constexpr (kStageW) {
        for (int j = threadIdx.x; j < nvec; j += 64 * WAVES) wl[j] = wr[j];
    }
#pragma unroll
    for (int i = 0; i < VPT; ++i) {
        const TX* e = reinterpret_cast<const TX*>(&xv[i]);
#pragma unroll
        for (int k = 0; k < VEC; ++k) {
            const float f = to_f32(e[k]);
            ss = fmaf(f, f, ss);
        }
    }
    ss = wave_sum(ss);
    if constexpr (WPR > 1) {
        __shared__ float part[WAVES];
        if (lane == 0) part[wave] = ss;
        __syncthreads();  // also publishes the staged weight
        float t = 0.f;
#pragma unroll
        for (int s = 0; s < WPR; ++s) t += part[row_in_block * WPR + s];
        ss = t;
    }
    if (!row_ok) return;
    const float inv = 1.0f / sqrtf(ss / (float)dim + eps);

    YPack* yr = reinterpret_cast<YPack*>(y + row * ld_y);
#pragma unroll
    for (int i = 0; i < VPT; ++i) {
        const int j = (i * WPR + slice) * 64 + lane;
        if (j < nvec) {
            const TX* e = reinterpret_cast<const TX*>(&xv[i]);
            WPack wv;
            if constexpr (kStageW)
                wv = wl[j];
            else if constexpr (HAS_W)
                wv = wr[j];
            YPack ov;
#pragma unroll
            for (int k = 0; k < VEC; ++k) {
                const TX n = from_f32<TX>(to_f32(e[k]) * inv);
                if constexpr (HAS_W)
                    ov.v[k] = from_f32<TY>(to_f32(n) * to_f32(wv.v[k]));
                else
                    ov.v[k] = from_f32<TY>(to_f32(n));
            }
            store_nt(yr + j, ov);
        }
    }
}

// LiteLA's q/k norm and rotary embedding in one pass, in place on the packed
// qkv[token][q, k, v][dim]: the arithmetic of
// rmsnorm_vec_kernel, with its layout and so its bits, then that of
// rope_packed_kernel on the rounded result (channel pairs lie within a
// 16-byte vector, a vector within a head).  HBM bound: it reads and writes q
// and k once, where two norm launches and a rotary one did so twice.  Measured
// on MI355X at 8192 tokens of 2240 channels, bf16 (147 MB): 40 us with the
// rotary embedding against 62 for the three launches, 37 without it against 36
// for two (which a small call pays for twice: 7 against 20 us at 1024 x 1152).
// Staging the weight in LDS, or q rows and k rows in separate halves of the
// grid, was no faster; requesting the weight and table values with the row,
// per vector, was slower (53 us).
// ROPE: 0 = norm only, 1 = a head divides the 64 vectors of a load (D = 8..512,
// powers of two), so that a lane meets the same table values in every vector and
// loads them once, 2 = any D.
template <typename T, int VPT, int WPR, int WAVES, int ROPE>
__global__ __launch_bounds__(64 * WAVES) void rmsnorm_qk_kernel(T* qkv, const T* __restrict__ qw,
                                                                const T* __restrict__ kw,
                                                                const float* __restrict__ cs,
                                                                const float* __restrict__ sn, int64_t row0,
                                                                int64_t tokens, int64_t N, int dim, int D,
                                                                float eps) {
    // The rotary products and their sum are rounded one by one (rope.hip).
#pragma clang fp contract(off)
    constexpr int VEC = 16 / sizeof(T);
    typedef Pack<T, VEC> P;
    constexpr int RPB = WAVES / WPR;
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
    const int slot = wave / WPR, slice = wave % WPR;
    const int64_t r = row0 + (int64_t)blockIdx.x * RPB + slot;  // a token's q row, then its k row
    const int64_t tok = r >> 1;
    const int part_k = (int)(r & 1);
    const bool ok = tok < tokens;
    const int nvec = dim / VEC;
    const P* wr = reinterpret_cast<const P*>(part_k ? kw : qw);
    P* row = reinterpret_cast<P*>(qkv + (tok * 3 + part_k) * (int64_t)dim);

    typedef Pack<float, VEC> F;
    P xv[VPT];
    float ss = 0.f;
#pragma unroll
    for (int i = 0; i < VPT; ++i) {
        const int j = (i * WPR + slice) * 64 + lane;
        xv[i] = ok && j < nvec ? load_nt(row + j) : P{};
    }
    const int64_t trow = tok % N * D;
    F cv, sv;
    if constexpr (ROPE == 1) {
        cv = *reinterpret_cast<const F*>(cs + trow + lane * VEC % D);
        sv = *reinterpret_cast<const F*>(sn + trow + lane * VEC % D);
    }
#pragma unroll
    for (int i = 0; i < VPT; ++i)
#pragma unroll
        for (int k = 0; k < VEC; ++k) {
            const float f = to_f32(xv[i].v[k]);
            ss = fmaf(f, f, ss);
        }
    ss = wave_sum(ss);
    if constexpr (WPR > 1) {
        __shared__ float part[WAVES];
        if (lane == 0) part[wave] = ss;
        __syncthreads();
        float t = 0.f;
#pragma unroll
        for (int s = 0; s < WPR; ++s) t += part[slot * WPR + s];
        ss = t;
    }
    if (!ok) return;
    const float inv = 1.0f / sqrtf(ss / (float)dim + eps);
#pragma unroll
    for (int i = 0; i < VPT; ++i) {
        const int j = (i * WPR + slice) * 64 + lane;
        if (j < nvec) {
            const P wv = wr[j];
            P ov;
#pragma unroll
            for (int k = 0; k < VEC; ++k) {
                // The product is rounded to fp32 first, as rmsnorm_vec_kernel
                // does; left to itself the compiler forms v_fma_mixlo_f16 for
                // some of them, which rounds once.
                float t = to_f32(xv[i].v[k]) * inv;
                if constexpr (__is_same(T, f16)) asm("" : "+v"(t));
                ov.v[k] = from_f32<T>(to_f32(from_f32<T>(t)) * to_f32(wv.v[k]));
            }
            if constexpr (ROPE == 2) {
                cv = *reinterpret_cast<const F*>(cs + trow + j * VEC % D);
                sv = *reinterpret_cast<const F*>(sn + trow + j * VEC % D);
            }
            if constexpr (ROPE != 0) {
#pragma unroll
                for (int k = 0; k < VEC; k += 2) {
                    const float re = to_f32(ov.v[k]), im = to_f32(ov.v[k + 1]);
                    const float a0 = re * cv.v[k], b0 = -im * sv.v[k];
                    const float a1 = im * cv.v[k + 1], b1 = re * sv.v[k + 1];
                    ov.v[k] = from_f32<T>(a0 + b0);
                    ov.v[k + 1] = from_f32<T>(a1 + b1);
                }
            }
            store_nt(row + j, ov);
        }
    }
}

template <typename T, int VPT, int WPR, int WAVES>
int launch_qk(void* qkv, const void* qw, const void* kw, const float* cs, const float* sn, int64_t tokens, int64_t N,
              int64_t dim, int64_t D, float eps, hipStream_t stream) {
    // Rows per launch: HIP limits a grid to 2^32 - 1 threads.  The two row
    // norms this stands for took twice the tokens in one launch each.
    constexpr int RPB = WAVES / WPR;
    constexpr int64_t kMaxBlocks = 0xffffffffLL / (64 * WAVES);
    for (int64_t row0 = 0; row0 < 2 * tokens; row0 += kMaxBlocks * RPB) {
        const int64_t left = (2 * tokens - row0 + RPB - 1) / RPB;
        const dim3 grid((unsigned)(left < kMaxBlocks ? left : kMaxBlocks));
        auto launch = [&](auto ropec) {
            hipLaunchKernelGGL((rmsnorm_qk_kernel<T, VPT, WPR, WAVES, decltype(ropec)::value>), grid,
                               dim3(64 * WAVES), 0, stream, static_cast<T*>(qkv), static_cast<const T*>(qw),
                               static_cast<const T*>(kw), cs, sn, row0, tokens, N, (int)dim, (int)D, eps);
        };
        if (!cs) launch(std::integral_constant<int, 0>{});
        else if (64 * (16 / (int)sizeof(T)) % D == 0) launch(std::integral_constant<int, 1>{});
        else launch(std::integral_constant<int, 2>{});
        if (int rc = check_launch("rmsnorm_qk_kernel launch")) return rc;
    }
    return KF_OK;
}

template <typename T>
int dispatch_qk(void* qkv, const void* qw, const void* kw, const float* cs, const float* sn, int64_t tokens,
                int64_t N, int64_t dim, int64_t D, float eps, hipStream_t stream) {
    const int64_t nvec = dim / (16 / (int64_t)sizeof(T));
#define KF_RMS_QK(VPT, WPR, WAVES) \
    return launch_qk<T, VPT, WPR, WAVES>(qkv, qw, kw, cs, sn, tokens, N, dim, D, eps, stream)
    // The shapes of dispatch() above, whose sums these must equal.
    if (nvec <= 64) KF_RMS_QK(1, 1, 4);
    if (nvec <= 128) KF_RMS_QK(2, 1, 4);
    if (nvec <= 256) KF_RMS_QK(2, 2, 4);
    if (nvec <= 512) KF_RMS_QK(2, 4, 8);
    KF_RMS_QK(2, 8, 8);
#undef KF_RMS_QK
}

// Any dim / alignment: one block per row, two passes over the row.
template <typename TX, typename TW, typename TY, bool HAS_W>
__global__ __launch_bounds__(kBlock) void rmsnorm_generic_kernel(const TX* x, const TW* __restrict__ w,
                                                                 TY* y, int64_t rows, int64_t dim,
                                                                 int64_t ld_x, int64_t ld_y, float eps) {
    const int64_t row = blockIdx.x;
    if (row >= rows) return;
    const TX* xr = x + row * ld_x;
    float ss = 0.f;
    for (int64_t c = threadIdx.x; c < dim; c += kBlock) {
        const float f = to_f32(xr[c]);
        ss = fmaf(f, f, ss);
    }
    ss = wave_sum(ss);
    __shared__ float part[4];
    if ((threadIdx.x & 63) == 0) part[threadIdx.x >> 6] = ss;
    __syncthreads();
    ss = part[0] + part[1] + part[2] + part[3];
    const float inv = 1.0f / sqrtf(ss / (float)dim + eps);
    TY* yr = y + row * ld_y;
    for (int64_t c = threadIdx.x; c < dim; c += kBlock) {
        const TX n = from_f32<TX>(to_f32(xr[c]) * inv);
        if constexpr (HAS_W)
            yr[c] = from_f32<TY>(to_f32(n) * to_f32(w[c]));
        else
            yr[c] = from_f32<TY>(to_f32(n));
    }
}

template <typename TX, typename TW, typename TY, int VPT, int WPR, int WAVES, bool HAS_W>
int launch_vec(const void* x, const void* w, void* y, int64_t rows, int64_t dim, int64_t ld_x,
               int64_t ld_y, float eps, hipStream_t stream) {
    static_assert(WAVES % WPR == 0, "a block holds whole rows");
    constexpr int ROWS_PER_BLOCK = WAVES / WPR;
    const int64_t blocks = (rows + ROWS_PER_BLOCK - 1) / ROWS_PER_BLOCK;
    KF_REQUIRE(blocks <= 0x7fffffff, KF_E_UNSUPPORTED, "rmsnorm: %lld rows exceed the grid limit",
               (long long)rows);
    hipLaunchKernelGGL((rmsnorm_vec_kernel<TX, TW, TY, VPT, WPR, WAVES, HAS_W>), dim3((unsigned)blocks),
                       dim3(64 * WAVES), 0, stream, static_cast<const TX*>(x),
                       static_cast<const TW*>(w), static_cast<TY*>(y), rows, (int)dim, ld_x, ld_y, eps);
    return check_launch("rmsnorm_vec_kernel launch");
}

bool aligned_to(const void* p, size_t a) { return (uintptr_t)p % a == 0; }

template <typename TX, typename TW, typename TY, bool HAS_W>
int dispatch(const void* x, const void* w, void* y, int64_t rows, int64_t dim, int64_t ld_x,
             int64_t ld_y, float eps, hipStream_t stream) {
    if (rows == 0) return KF_OK;
    constexpr int VEC = 16 / sizeof(TX);
    // Byte alignment of the weight and output slices of one x vector.
    constexpr size_t WA = sizeof(Pack<TW, VEC>) < 16 ? sizeof(Pack<TW, VEC>) : 16;
    constexpr size_t YA = sizeof(Pack<TY, VEC>) < 16 ? sizeof(Pack<TY, VEC>) : 16;
    const bool aligned = aligned_to(x, 16) && aligned_to(y, YA) && (!HAS_W || aligned_to(w, WA)) &&
                         (dim % VEC == 0) && (ld_x % VEC == 0) && (ld_y * sizeof(TY)) % YA == 0;
    const int64_t nvec = dim / VEC;
    if (aligned) {
#define KF_RMS_VEC(VPT, WPR, WAVES) \
    return launch_vec<TX, TW, TY, VPT, WPR, WAVES, HAS_W>(x, w, y, rows, dim, ld_x, ld_y, eps, stream)
        // (vectors per lane, waves per row, waves per block).
        if (nvec <= 64) KF_RMS_VEC(1, 1, 4);
        if (nvec <= 128) KF_RMS_VEC(2, 1, 4);
        if (nvec <= 256) KF_RMS_VEC(2, 2, 4);
        if (nvec <= 512) KF_RMS_VEC(2, 4, 8);
        if (nvec <= 1024) KF_RMS_VEC(2, 8, 8);
        if (nvec <= 2048) KF_RMS_VEC(4, 8, 8);
        if (nvec <= 4096) KF_RMS_VEC(8, 8, 8);
#undef KF_RMS_VEC
    }
    KF_REQUIRE(rows <= 0x7fffffff, KF_E_UNSUPPORTED, "rmsnorm: %lld rows exceed the grid limit",
               (long long)rows);
    hipLaunchKernelGGL((rmsnorm_generic_kernel<TX, TW, TY, HAS_W>), dim3((unsigned)rows), dim3(kBlock), 0,
                       stream, static_cast<const TX*>(x), static_cast<const TW*>(w),
                       static_cast<TY*>(y), rows, dim, ld_x, ld_y, eps);
    return check_launch("rmsnorm_generic_kernel launch");
}

// --------------------------------------------------------------------------
// Backward.
// --------------------------------------------------------------------------
// Gradient of y = ty(float(tx(x * inv)) * float(w)) with the rounding points
// taken as identities (as torch's autograd treats the casts of
// original.py:51-52):
//   n   = tx(x * inv)                          (the saved normalised value)
//   g   = float(tx(float(dy) * float(w)))      (gradient at n: torch forms
//                                               `grad * weight` and casts it to
//                                               n's type tx)
//   dx  = inv * g - x * inv^3 * sum(g * x) / dim
//   dw  = tw(sum over rows of float(dy) * float(n))   (fp32 sum of unrounded
//                                               products)
// Each block owns a contiguous run of rows and writes its dw partial sums in
// fp32 to `partial[block][dim]` (its own row of the workspace, so no two
// blocks touch the same partial); rmsnorm_dw_reduce_kernel then adds the
// block partials in a fixed order (deterministic, no atomics).

// Rows of whole 16-byte vectors, laid out over the lanes as in
// rmsnorm_vec_kernel (RPB = WAVES / WPR rows at a time).  x and dy are read
// once, dx written once: HBM bound.  Every lane owns the same columns of all
// its rows, so the weight and the dw sums stay in registers; the next row's
// loads run while this row is reduced.  Measured on MI355X at rows 8192, dim
// 2240, bf16 x, fp32 weight (147 MB): 38 us, 3.9 TB/s;
// one scalar load at a time, with the dw sums read and written in memory for
// every row, took 87.
template <typename TX, typename TW, typename TY, int VPT, int WPR, int WAVES>
__global__ __launch_bounds__(64 * WAVES) void rmsnorm_bwd_vec_kernel(const TX* __restrict__ x,
                                                                     const TW* __restrict__ w,
                                                                     const TY* __restrict__ dy,
                                                                     TX* __restrict__ dx,
                                                                     float* __restrict__ partial, int64_t rows,
                                                                     int dim, int64_t rows_per_block, float eps) {
    constexpr int VEC = 16 / sizeof(TX);
    typedef Pack<TW, VEC> WPack;
    typedef Pack<TY, VEC> YPack;
    constexpr int RPB = WAVES / WPR;
    constexpr int SLOTS = VPT * WPR * 64;
    constexpr bool kAhead = VPT <= 2;  // registers for a second row
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
    const int slot = wave / WPR, slice = wave % WPR;
    const int nvec = dim / VEC;
    const int64_t r0 = (int64_t)blockIdx.x * rows_per_block;
    const int64_t r1 = r0 + rows_per_block < rows ? r0 + rows_per_block : rows;

    WPack wv[VPT];
    float acc[VPT][VEC];
#pragma unroll
    for (int i = 0; i < VPT; ++i) {
        const int j = (i * WPR + slice) * 64 + lane;
        // Zero past the row's end, as x and dy are (another column's weight
        // may be infinite, and its product with zero would be NaN).
        wv[i] = j < nvec ? reinterpret_cast<const WPack*>(w)[j] : WPack{};
#pragma unroll
        for (int k = 0; k < VEC; ++k) acc[i][k] = 0.f;
    }
    // One row of x and dy; a row past the run re-reads its last row, and a
    // vector past the row's end is left zero.
    auto load = [&](int64_t row, u32x4 (&xv)[VPT], YPack (&gv)[VPT]) {
        if (row >= r1) row = r1 - 1;
        const u32x4* xr = reinterpret_cast<const u32x4*>(x + row * dim);
        const YPack* gr = reinterpret_cast<const YPack*>(dy + row * dim);
#pragma unroll
        for (int i = 0; i < VPT; ++i) {
            const int j = (i * WPR + slice) * 64 + lane;
            if (j < nvec) {
                xv[i] = __builtin_nontemporal_load(xr + j);
                gv[i] = load_nt(gr + j);
            } else {
                xv[i] = u32x4{0u, 0u, 0u, 0u};
                gv[i] = YPack{};
            }
        }
    };
    u32x4 xv[VPT], xn[VPT];
    YPack gv[VPT], gn[VPT];
    load(r0 + slot, xv, gv);
    __shared__ float part[2][WAVES][2];
    const int64_t steps = (r1 - r0 + RPB - 1) / RPB;
    for (int64_t it = 0; it < steps; ++it) {
        const int64_t row = r0 + it * RPB + slot;
        if constexpr (kAhead) load(row + RPB, xn, gn);
        float ss = 0.f, dot = 0.f;
#pragma unroll
        for (int i = 0; i < VPT; ++i) {
            const TX* e = reinterpret_cast<const TX*>(&xv[i]);
#pragma unroll
            for (int k = 0; k < VEC; ++k) {
                const float f = to_f32(e[k]);
                const float g = to_f32(from_f32<TX>(to_f32(gv[i].v[k]) * to_f32(wv[i].v[k])));
                ss = fmaf(f, f, ss);
                dot = fmaf(g, f, dot);
            }
        }
        ss = wave_sum(ss);
        dot = wave_sum(dot);
        if constexpr (WPR > 1) {
            // Two sets of slots in turn: one barrier per row, which leaves the
            // next row's loads in flight.
            float (*pt)[2] = part[it & 1];
            if (lane == 0) {
                pt[wave][0] = ss;
                pt[wave][1] = dot;
            }
            barrier_lds_only();
            ss = dot = 0.f;
#pragma unroll
            for (int q = 0; q < WPR; ++q) {
                ss += pt[slot * WPR + q][0];
                dot += pt[slot * WPR + q][1];
            }
        }
        const float inv = 1.0f / sqrtf(ss / (float)dim + eps);
        const float kk = inv * inv * inv * dot / (float)dim;
        if (row < r1) {
            u32x4* dr = reinterpret_cast<u32x4*>(dx + row * dim);
#pragma unroll
            for (int i = 0; i < VPT; ++i) {
                const int j = (i * WPR + slice) * 64 + lane;
                const TX* e = reinterpret_cast<const TX*>(&xv[i]);
                u32x4 ov;
                TX* o = reinterpret_cast<TX*>(&ov);
#pragma unroll
                for (int k = 0; k < VEC; ++k) {
                    const float f = to_f32(e[k]);
                    const float gy = to_f32(gv[i].v[k]);
                    const float g = to_f32(from_f32<TX>(gy * to_f32(wv[i].v[k])));
                    o[k] = from_f32<TX>(inv * g - f * kk);
                    if (j < nvec) acc[i][k] += gy * to_f32(from_f32<TX>(f * inv));
                }
                if (j < nvec) __builtin_nontemporal_store(ov, dr + j);
            }
        }
        if constexpr (kAhead) {
#pragma unroll
            for (int i = 0; i < VPT; ++i) {
                xv[i] = xn[i];
                gv[i] = gn[i];
            }
        } else {
            load(row + RPB, xv, gv);
        }
    }
    // The row slots' sums in slot order.
    if constexpr (RPB > 1) {
        __shared__ float comb[(RPB - 1) * SLOTS * VEC];
        if (slot > 0) {
#pragma unroll
            for (int i = 0; i < VPT; ++i)
#pragma unroll
                for (int k = 0; k < VEC; ++k)
                    comb[((slot - 1) * VEC + k) * SLOTS + (i * WPR + slice) * 64 + lane] = acc[i][k];
        }
        __syncthreads();
        if (slot > 0) return;
#pragma unroll
        for (int q = 0; q < RPB - 1; ++q)
#pragma unroll
            for (int i = 0; i < VPT; ++i)
#pragma unroll
                for (int k = 0; k < VEC; ++k)
                    acc[i][k] += comb[(q * VEC + k) * SLOTS + (i * WPR + slice) * 64 + lane];
    }
    f32x4* pw = reinterpret_cast<f32x4*>(partial + (int64_t)blockIdx.x * dim);
#pragma unroll
    for (int i = 0; i < VPT; ++i) {
        const int j = (i * WPR + slice) * 64 + lane;
        if (j < nvec) {
#pragma unroll
            for (int k = 0; k < VEC; k += 4)
                pw[(j * VEC + k) / 4] = f32x4{acc[i][k], acc[i][k + 1], acc[i][k + 2], acc[i][k + 3]};
        }
    }
}

// Any dim / alignment: a block's rows one after another, two passes over each.
template <typename TX, typename TW, typename TY>
__global__ __launch_bounds__(kBlock) void rmsnorm_bwd_kernel(const TX* __restrict__ x,
                                                             const TW* __restrict__ w,
                                                             const TY* __restrict__ dy,
                                                             TX* __restrict__ dx,
                                                             float* __restrict__ partial, int64_t rows,
                                                             int64_t dim, int64_t rows_per_block,
                                                             float eps) {
    __shared__ float part[2][4];
    float* pw = partial + (int64_t)blockIdx.x * dim;
    for (int64_t c = threadIdx.x; c < dim; c += kBlock) pw[c] = 0.f;
    const int64_t r0 = (int64_t)blockIdx.x * rows_per_block;
    const int64_t r1 = r0 + rows_per_block < rows ? r0 + rows_per_block : rows;
    for (int64_t row = r0; row < r1; ++row) {
        const TX* xr = x + row * dim;
        const TY* gr = dy + row * dim;
        float ss = 0.f, dot = 0.f;
        for (int64_t c = threadIdx.x; c < dim; c += kBlock) {
            const float f = to_f32(xr[c]);
            const float g = to_f32(from_f32<TX>(to_f32(gr[c]) * to_f32(w[c])));
            ss = fmaf(f, f, ss);
            dot = fmaf(g, f, dot);
        }
        ss = wave_sum(ss);
        dot = wave_sum(dot);
        const int wave = threadIdx.x >> 6;
        if ((threadIdx.x & 63) == 0) {
            part[0][wave] = ss;
            part[1][wave] = dot;
        }
        __syncthreads();
        ss = part[0][0] + part[0][1] + part[0][2] + part[0][3];
        dot = part[1][0] + part[1][1] + part[1][2] + part[1][3];
        __syncthreads();  // part is rewritten by the next row
        const float inv = 1.0f / sqrtf(ss / (float)dim + eps);
        const float k = inv * inv * inv * dot / (float)dim;
        TX* dr = dx + row * dim;
        for (int64_t c = threadIdx.x; c < dim; c += kBlock) {
            const float f = to_f32(xr[c]);
            const float gy = to_f32(gr[c]);
            const float g = to_f32(from_f32<TX>(gy * to_f32(w[c])));
            dr[c] = from_f32<TX>(inv * g - f * k);
            const float n = to_f32(from_f32<TX>(f * inv));
            pw[c] += gy * n;  // the same thread owns column c for every row
        }
    }
}

// dw = the block partials' sums: 32 columns per block, 16 slices of the
// partials each (slice s adds partials s, s + 16, ..., eight loads in flight),
// then the slices in order.  One thread per column over all partials was a
// chain of up to 1024 load latencies (227 us at 1024 partials of 2240 columns
// on MI355X; now 4.8).
constexpr int kDwCols = 32, kDwSlices = 16;
template <typename TW>
__global__ __launch_bounds__(kDwCols * kDwSlices) void rmsnorm_dw_reduce_kernel(const float* __restrict__ partial,
                                                                                 TW* __restrict__ dw, int64_t c0,
                                                                                 int64_t dim, int nblocks) {
    __shared__ float sums[kDwSlices][kDwCols];
    const int col = threadIdx.x % kDwCols, slice = threadIdx.x / kDwCols;
    const int64_t c = c0 + (int64_t)blockIdx.x * kDwCols + col;
    float acc = 0.f;
    if (c < dim) {
        for (int b0 = slice; b0 < nblocks; b0 += 8 * kDwSlices) {
            float v[8];
#pragma unroll
            for (int i = 0; i < 8; ++i) {
                const int b = b0 + i * kDwSlices;
                const float p = partial[(int64_t)(b < nblocks ? b : b0) * dim + c];
                v[i] = b < nblocks ? p : 0.f;
            }
#pragma unroll
            for (int i = 0; i < 8; ++i) acc += v[i];
        }
    }
    sums[slice][col] = acc;
    __syncthreads();
    if (slice == 0 && c < dim) {
#pragma unroll
        for (int q = 1; q < kDwSlices; ++q) acc += sums[q][col];
        dw[c] = from_f32<TW>(acc);
    }
}

constexpr int64_t kBwdMaxBlocks = 1024;  // partials of the workspace

int64_t bwd_blocks(int64_t rows) { return rows < kBwdMaxBlocks ? rows : kBwdMaxBlocks; }

template <typename TX, typename TW, typename TY, int VPT, int WPR, int WAVES>
int launch_bwd_vec(const TX* x, const TW* w, const TY* dy, TX* dx, float* partial, int64_t rows, int64_t dim,
                   float eps, hipStream_t stream, int64_t* used) {
    // As many blocks as stay resident: 16 wavefronts per CU for fp32 x, 8 for
    // 16-bit x, whose kernels take 120-140 registers (rows 16384, dim 4096 on
    // MI355X: bf16 x, fp32 weight 116 us at 16, 102 at 8; fp32 150 and 167),
    // each with at least four rounds of rows where the rows allow it (a
    // block's partial costs two extra passes over a row's width).
    constexpr int RPB = WAVES / WPR;
    constexpr int kWavesPerCu = sizeof(TX) == 4 ? 16 : 8;
    int64_t nb = (int64_t)device_cu_count() * (kWavesPerCu / WAVES);
    const int64_t by_rows = (rows + 4 * RPB - 1) / (4 * RPB);
    if (nb > by_rows) nb = by_rows;
    if (nb > bwd_blocks(rows)) nb = bwd_blocks(rows);
    const int64_t per = (rows + nb - 1) / nb;
    *used = (rows + per - 1) / per;
    hipLaunchKernelGGL((rmsnorm_bwd_vec_kernel<TX, TW, TY, VPT, WPR, WAVES>), dim3((unsigned)*used),
                       dim3(64 * WAVES), 0, stream, x, w, dy, dx, partial, rows, (int)dim, per, eps);
    return check_launch("rmsnorm_bwd_vec_kernel launch");
}

template <typename TX, typename TW, typename TY>
int run_bwd_rows(const TX* x, const TW* w, const TY* dy, TX* dx, float* partial, int64_t rows, int64_t dim,
                 float eps, hipStream_t stream, int64_t* used) {
    constexpr int VEC = 16 / sizeof(TX);
    constexpr size_t WA = sizeof(Pack<TW, VEC>) < 16 ? sizeof(Pack<TW, VEC>) : 16;
    constexpr size_t YA = sizeof(Pack<TY, VEC>) < 16 ? sizeof(Pack<TY, VEC>) : 16;
    const bool aligned = aligned_to(x, 16) && aligned_to(dx, 16) && aligned_to(dy, YA) && aligned_to(w, WA) &&
                         aligned_to(partial, 16) && dim % VEC == 0;
    const int64_t nvec = dim / VEC;
    if (aligned) {
#define KF_RMS_BWD(VPT, WPR, WAVES) \
    return launch_bwd_vec<TX, TW, TY, VPT, WPR, WAVES>(x, w, dy, dx, partial, rows, dim, eps, stream, used)
        // (vectors per lane, waves per row, waves per block).
        if (nvec <= 64) KF_RMS_BWD(1, 1, 4);
        if (nvec <= 128) KF_RMS_BWD(2, 1, 4);
        if (nvec <= 256) KF_RMS_BWD(2, 2, 4);
        if (nvec <= 512) KF_RMS_BWD(2, 4, 4);
        if (nvec <= 1024) KF_RMS_BWD(2, 8, 8);
        if (nvec <= 2048) KF_RMS_BWD(4, 8, 8);
#undef KF_RMS_BWD
    }
    const int64_t nb = bwd_blocks(rows);
    const int64_t per = (rows + nb - 1) / nb;
    *used = (rows + per - 1) / per;  // blocks that own at least one row
    hipLaunchKernelGGL((rmsnorm_bwd_kernel<TX, TW, TY>), dim3((unsigned)*used), dim3(kBlock), 0, stream, x, w, dy,
                       dx, partial, rows, dim, per, eps);
    return check_launch("rmsnorm_bwd_kernel launch");
}

template <typename TX, typename TW, typename TY>
int run_bwd(const void* x, const void* w, const void* dy, void* dx, void* dw, float* partial,
            int64_t rows, int64_t dim, float eps, hipStream_t stream) {
    int64_t used = 0;
    if (rows > 0) {
        if (int rc = run_bwd_rows(static_cast<const TX*>(x), static_cast<const TW*>(w), static_cast<const TY*>(dy),
                                  static_cast<TX*>(dx), partial, rows, dim, eps, stream, &used))
            return rc;
    }
    // With no rows the reduction adds nothing and writes a zero weight gradient.
    // Sixteen threads a column: HIP's limit of 2^32 - 1 threads in a grid is
    // passed at 2^28 columns.
    constexpr int64_t kMaxBlocks = 0xffffffffLL / (kDwCols * kDwSlices);
    for (int64_t c0 = 0; c0 < dim; c0 += kMaxBlocks * kDwCols) {
        const int64_t left = (dim - c0 + kDwCols - 1) / kDwCols;
        hipLaunchKernelGGL((rmsnorm_dw_reduce_kernel<TW>), dim3((unsigned)(left < kMaxBlocks ? left : kMaxBlocks)),
                           dim3(kDwCols * kDwSlices), 0, stream, partial, static_cast<TW*>(dw), c0, dim, (int)used);
        if (int rc = check_launch("rmsnorm_dw_reduce_kernel launch")) return rc;
    }
    return KF_OK;
}

bool valid_dt(int d) { return d == KF_F32 || d == KF_F16 || d == KF_BF16; }

// torch.promote_types over {fp32, fp16, bf16}: equal types stay, any mix
// gives fp32.
int promote(int a, int b) { return a == b ? a : KF_F32; }

// Calls F<TX, TW, TY>::run(args...) for the (x, weight) dtype pair; TY is
// their promotion.
template <template <typename, typename, typename> class F, typename... A>
int by_types(int xd, int wd, A... args) {
    switch (xd * 3 + wd) {
        case KF_F32 * 3 + KF_F32: return F<float, float, float>::run(args...);
        case KF_F32 * 3 + KF_F16: return F<float, f16, float>::run(args...);
        case KF_F32 * 3 + KF_BF16: return F<float, bf16, float>::run(args...);
        case KF_F16 * 3 + KF_F32: return F<f16, float, float>::run(args...);
        case KF_F16 * 3 + KF_F16: return F<f16, f16, f16>::run(args...);
        case KF_F16 * 3 + KF_BF16: return F<f16, bf16, float>::run(args...);
        case KF_BF16 * 3 + KF_F32: return F<bf16, float, float>::run(args...);
        case KF_BF16 * 3 + KF_F16: return F<bf16, f16, float>::run(args...);
        case KF_BF16 * 3 + KF_BF16: return F<bf16, bf16, bf16>::run(args...);
    }
    set_error("rmsnorm: unknown dtype pair (%d, %d)", xd, wd);
    return KF_E_INVALID;
}

template <typename TX, typename TW, typename TY> struct FwdOp {
    static int run(const void* x, const void* w, void* y, int64_t rows, int64_t dim, int64_t ld_x,
                   int64_t ld_y, float eps, hipStream_t s) {
        return dispatch<TX, TW, TY, true>(x, w, y, rows, dim, ld_x, ld_y, eps, s);
    }
};

template <typename TX, typename TW, typename TY> struct BwdOp {
    static int run(const void* x, const void* w, const void* dy, void* dx, void* dw, float* partial,
                   int64_t rows, int64_t dim, float eps, hipStream_t s) {
        return run_bwd<TX, TW, TY>(x, w, dy, dx, dw, partial, rows, dim, eps, s);
    }
};

}  // namespace
}  // namespace kf

extern "C" int kf_rmsnorm_fwd_strided(const void* x, const void* weight, void* y, int64_t rows,
                                      int64_t dim, int64_t ld_x, int64_t ld_y, float eps, int dtype,
                                      kf_stream_t stream) {
    using namespace kf;
    KF_REQUIRE(rows >= 0 && dim >= 1, KF_E_INVALID, "rmsnorm: bad shape rows=%lld dim=%lld",
               (long long)rows, (long long)dim);
    KF_REQUIRE(ld_x >= dim && ld_y >= dim, KF_E_INVALID,
               "rmsnorm: row strides ld_x=%lld ld_y=%lld must be >= dim=%lld", (long long)ld_x,
               (long long)ld_y, (long long)dim);
    KF_REQUIRE(rows == 0 || (x && y && weight), KF_E_INVALID, "rmsnorm: null pointer");
    KF_REQUIRE(dim <= 0x7fffffff, KF_E_UNSUPPORTED, "rmsnorm: dim %lld too large", (long long)dim);
    KF_REQUIRE(valid_dt(dtype), KF_E_INVALID, "rmsnorm: unknown dtype %d", dtype);
    return by_types<FwdOp>(dtype, dtype, x, weight, y, rows, dim, ld_x, ld_y, eps,
                           static_cast<hipStream_t>(stream));
}

extern "C" int kf_qk_norm_rope(void* qkv, const void* q_weight, const void* k_weight, const float* cos,
                               const float* sin, int64_t batch, int64_t seq_len, int64_t heads, int64_t dim,
                               float eps, int dtype, kf_stream_t stream) {
    using namespace kf;
    KF_REQUIRE(batch >= 0 && seq_len >= 0 && heads > 0 && dim > 0, KF_E_INVALID, "qk_norm: bad shape");
    KF_REQUIRE(valid_dt(dtype), KF_E_INVALID, "qk_norm: unknown dtype %d", dtype);
    KF_REQUIRE(heads <= (1 << 20) && dim <= 4096 && batch <= (1 << 20) && seq_len <= ((int64_t)1 << 31), KF_E_INVALID,
               "qk_norm: shape out of range");
    const int64_t C = heads * dim, es = dtype == KF_F32 ? 4 : 2;
    KF_REQUIRE((cos == nullptr) == (sin == nullptr), KF_E_INVALID, "qk_norm: cos and sin come together");
    KF_REQUIRE(C * es % 16 == 0 && C * es <= 16384 && (!cos || dim % 8 == 0), KF_E_UNSUPPORTED,
               "qk_norm: rows must be whole 16-byte vectors, at most 16 KiB, and rotated heads whole multiples of 8");
    if (batch == 0 || seq_len == 0) return KF_OK;
    KF_REQUIRE(qkv && q_weight && k_weight, KF_E_INVALID, "qk_norm: null pointer");
    for (const void* p : {(const void*)qkv, q_weight, k_weight, (const void*)cos, (const void*)sin})
        KF_REQUIRE(aligned_to(p, 16), KF_E_INVALID, "qk_norm: buffers must be 16-byte aligned");
    const int64_t tokens = batch * seq_len;
    const hipStream_t s = static_cast<hipStream_t>(stream);
    switch (dtype) {
        case KF_F32: return dispatch_qk<float>(qkv, q_weight, k_weight, cos, sin, tokens, seq_len, C, dim, eps, s);
        case KF_F16: return dispatch_qk<f16>(qkv, q_weight, k_weight, cos, sin, tokens, seq_len, C, dim, eps, s);
        default: return dispatch_qk<bf16>(qkv, q_weight, k_weight, cos, sin, tokens, seq_len, C, dim, eps, s);
    }
}

extern "C" int kf_rmsnorm_fwd(const void* x, const void* weight, void* y, int64_t rows,
                              int64_t dim, float eps, int dtype, kf_stream_t stream) {
    return kf_rmsnorm_fwd_strided(x, weight, y, rows, dim, dim, dim, eps, dtype, stream);
}

extern "C" int kf_rmsnorm_fwd_mixed(const void* x, const void* weight, void* y, int64_t rows,
                                    int64_t dim, float eps, int x_dtype, int w_dtype, int y_dtype,
                                    kf_stream_t stream) {
    using namespace kf;
    KF_REQUIRE(rows >= 0 && dim >= 1, KF_E_INVALID, "rmsnorm: bad shape rows=%lld dim=%lld",
               (long long)rows, (long long)dim);
    KF_REQUIRE(valid_dt(x_dtype) && valid_dt(w_dtype), KF_E_INVALID, "rmsnorm: unknown dtype (%d, %d)",
               x_dtype, w_dtype);
    KF_REQUIRE(y_dtype == promote(x_dtype, w_dtype), KF_E_INVALID,
               "rmsnorm: output dtype %d is not the promotion of x dtype %d and weight dtype %d", y_dtype,
               x_dtype, w_dtype);
    KF_REQUIRE(rows == 0 || (x && y && weight), KF_E_INVALID, "rmsnorm: null pointer");
    KF_REQUIRE(dim <= 0x7fffffff, KF_E_UNSUPPORTED, "rmsnorm: dim %lld too large", (long long)dim);
    return by_types<FwdOp>(x_dtype, w_dtype, x, weight, y, rows, dim, dim, dim, eps,
                           static_cast<hipStream_t>(stream));
}

extern "C" int64_t kf_rmsnorm_bwd_workspace_bytes(int64_t rows, int64_t dim) {
    if (rows < 0 || dim < 1) return -1;
    return (int64_t)sizeof(float) * kf::bwd_blocks(rows) * dim;
}

extern "C" int kf_rmsnorm_bwd(const void* x, const void* weight, const void* dy, void* dx, void* dweight,
                              void* workspace, int64_t workspace_bytes, int64_t rows, int64_t dim,
                              float eps, int x_dtype, int w_dtype, kf_stream_t stream) {
    using namespace kf;
    KF_REQUIRE(rows >= 0 && dim >= 1, KF_E_INVALID, "rmsnorm: bad shape rows=%lld dim=%lld",
               (long long)rows, (long long)dim);
    KF_REQUIRE(valid_dt(x_dtype) && valid_dt(w_dtype), KF_E_INVALID, "rmsnorm: unknown dtype (%d, %d)",
               x_dtype, w_dtype);
    KF_REQUIRE(dim <= 0x7fffffff, KF_E_UNSUPPORTED, "rmsnorm: dim %lld too large", (long long)dim);
    KF_REQUIRE(x || rows == 0, KF_E_INVALID, "rmsnorm: null pointer");
    KF_REQUIRE(weight && dweight, KF_E_INVALID, "rmsnorm: null weight or weight gradient");
    const int64_t need = kf_rmsnorm_bwd_workspace_bytes(rows, dim);
    KF_REQUIRE(rows == 0 || (workspace && workspace_bytes >= need), KF_E_WORKSPACE,
               "rmsnorm: workspace of %lld bytes needed, %lld given", (long long)need,
               (long long)workspace_bytes);
    KF_REQUIRE(rows == 0 || (dy && dx), KF_E_INVALID, "rmsnorm: null pointer");
    hipStream_t s = static_cast<hipStream_t>(stream);
    return by_types<BwdOp>(x_dtype, w_dtype, x, weight, dy, dx, dweight, static_cast<float*>(workspace),
                           rows, dim, eps, s);
}

extern "C" int kf_rmsnorm_noweight_f32(const float* a, float* b, int64_t rows, int64_t n,
                                       float eps, kf_stream_t stream) {
    using namespace kf;
    KF_REQUIRE(rows >= 0 && n >= 1, KF_E_INVALID, "rmsnorm: bad shape rows=%lld n=%lld",
               (long long)rows, (long long)n);
    KF_REQUIRE(rows == 0 || (a && b), KF_E_INVALID, "rmsnorm: null pointer");
    KF_REQUIRE(n <= 0x7fffffff, KF_E_UNSUPPORTED, "rmsnorm: n %lld too large", (long long)n);
    return dispatch<float, float, float, false>(a, nullptr, b, rows, n, n, n, eps,
                                                static_cast<hipStream_t>(stream));
}
