// Fused 2D-RoPE split and merge for gfx950 (C ABI: include/ebr_rope.h).
//
// Both are HBM-bound elementwise passes. A thread moves VW consecutive elements of one row: the quarter swap maps a
// VW-aligned chunk of a quarter onto a VW-aligned chunk of the partner quarter when VW divides D / 4, so a thread
// reads its chunk and its partner chunk with two vector loads (the partner's bytes are the neighbouring lanes' own,
// so they come from the cache). Work is flattened in the projection's order, [B, N, H, D], in both: its side of each
// thread's accesses is then contiguous over the heads, and only the other side jumps by a head dim's row. In the order
// of its outputs the split read 128 bytes of every 3 KB row: 77 against 67 us at [640, 100, 1536] bf16 (5.1, 5.8 TB/s),
// 37 against 30 at [384, 81, 1536].
//
// Arithmetic is fp32 with contraction off: every product and sum is rounded as the dense formula's separate
// operations are (reference models/fused_attn/rope_split.py:40-44, 58-61), then rounded once to the tensor dtype.
//
// The graded variants (FULL) also carry the learned temperature, which was a broadcast product of its own around the
// split and another around the merge, each with a product and a reduction for the temperature's gradient: the split
// sums w * (R q) per head as it writes t * (R q), and the merge adds a second set of gradients and sums its total dq
// times the rotated q, which it rotates again from qkv. Each extra operand is one read of a third of the projection
// where the products and reductions moved five. Per-head sums go to one row of partial sums per workgroup and are
// added in a fixed order by k_head_sums, so they are the same on every run; each product, and the sum of them all, is
// rounded to the dtype, as the separate ops round them. bf16, [384, 81] tokens, 8 heads of 64, a graded step with its
// second derivative: the products, reductions and sums took 245 us; folded in they add 47 (split 31 -> 45 with its sum,
// merge 32 -> 53 with the second set and its sum, two k_head_sums of 6).
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "../../include/ebr_rope.h"

namespace ebr_rope {

template <typename T, int VW> using Vec = T __attribute__((ext_vector_type(VW)));  // aligned to its size

template <typename T> __device__ __forceinline__ float f32(T x) { return (float)x; }

template <typename T> __device__ __forceinline__ T narrow(float x) { return (T)x; }  // round to nearest even

// An fp32 product kept opaque, so that narrowing it rounds twice (to fp32, then to T) as the dense formula does; for
// fp16 the compiler would otherwise fuse multiply and narrowing into one mixed-precision op that rounds once.
__device__ __forceinline__ float mul_f32(float a, float b) {
    float p = a * b;
    asm volatile("" : "+v"(p));
    return p;
}

// round(a + b) of two values of T.
template <typename T> __device__ __forceinline__ T sum_rounded(T a, T b) {
    float s = f32(a) + f32(b);
    asm volatile("" : "+v"(s));
    return narrow<T>(s);
}

struct SplitArgs {
    const void* qkv;
    int64_t sb, sn;
    const float* cos;
    const float* sin;
    const float* qs;
    void *q, *k, *v;
    int B, N, H, D;
    int64_t total;  // B * H * N * (D / VW) threads
    const void* w;  // FULL: [B, H, N, D] contiguous, multiplied with the rotated q and summed per head, or NULL
    float* part;    // FULL: [workgroups][H] sums
};

struct MergeArgs {
    const void *dq, *dk, *dv;
    int64_t sq[3], sk[3], sv[3];
    const float* cos;
    const float* sin;
    const float* qs;
    void* g;
    int B, H, N, D;
    int64_t total;  // B * N * H * (D / VW) threads
    const void *aq, *ak, *av;  // FULL: gradients to add, [B, H, N, D] contiguous, or NULL
    const void* qkv;           // FULL: the projection (contiguous), whose rotated q multiplies dq per head, or NULL
    float* part;
};

// Partner chunk start of the quarter swap: quarter (d / Q) ^ 1, same offset inside the quarter.
__device__ __forceinline__ int swap_start(int d0, int Q) { return ((d0 / Q) ^ 1) * Q + d0 % Q; }

// Sums ``s`` of the workgroup's threads per head into part[blockIdx.x][H]: over the ``cpr`` lanes of a row (a power of
// two, at most 64) by shuffles, then over the rows in order by one thread per head. Holds a workgroup barrier: every
// thread of the workgroup calls it, those past the last row with head -1.
__device__ __forceinline__ void head_partials(float s, int h, int cpr, int H, float* part) {
    __shared__ float rs[256];
    __shared__ int rh[256];
    for (int m = cpr >> 1; m >= 1; m >>= 1) s += __shfl_xor(s, m, 64);
    const int rows = 256 / cpr;
    if (threadIdx.x % cpr == 0) {
        rs[threadIdx.x / cpr] = s;
        rh[threadIdx.x / cpr] = h;
    }
    __syncthreads();
    for (int k = threadIdx.x; k < H; k += 256) {
        float sum = 0.f;
#pragma unroll 8
        for (int i = 0; i < rows; ++i) {
            const float v = rs[i];
            sum += rh[i] == k ? v : 0.f;
        }
        part[(int64_t)blockIdx.x * H + k] = sum;
    }
}

// out[h] = sum over the workgroups of part[.][h]; one workgroup per head, a fixed order. Bound by the latency of its
// loads: four in flight per thread, 1,024 threads (7,776 rows: 11.8 us with 256 threads and one load in flight).
constexpr int SUM_THREADS = 1024;
template <typename T> __global__ __launch_bounds__(SUM_THREADS) void k_head_sums(const float* part, int64_t n, int H, float* out) {
    __shared__ float ws[SUM_THREADS / 64];
    const int h = blockIdx.x;
    float s[4] = {0.f, 0.f, 0.f, 0.f};
    for (int64_t i = threadIdx.x; i < n; i += 4 * SUM_THREADS) {
        float v[4];
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const int64_t x = i + j * SUM_THREADS;
            v[j] = part[(x < n ? x : n - 1) * H + h];
        }
#pragma unroll
        for (int j = 0; j < 4; ++j) s[j] += i + j * SUM_THREADS < n ? v[j] : 0.f;
    }
    float t = (s[0] + s[1]) + (s[2] + s[3]);
    for (int m = 32; m >= 1; m >>= 1) t += __shfl_xor(t, m, 64);
    if ((threadIdx.x & 63) == 0) ws[threadIdx.x >> 6] = t;
    __syncthreads();
    if (threadIdx.x == 0) {
        float sum = 0.f;
        for (int w = 0; w < SUM_THREADS / 64; ++w) sum += ws[w];
        out[h] = f32(narrow<T>(sum));
    }
}

template <typename T, int VW, bool FULL> __global__ __launch_bounds__(256) void k_rope_split(SplitArgs a) {
#pragma clang fp contract(off)
    const int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    const int cpr = a.D / VW;
    const bool in = t < a.total;
    if (!FULL && !in) return;
    const int64_t tc = FULL && !in ? a.total - 1 : t;  // past the last row: its values, neither summed nor stored
    int64_t r = tc / cpr;
    const int c = (int)(tc - r * cpr);
    const int h = (int)(r % a.H);
    r /= a.H;
    const int n = (int)(r % a.N);
    const int b = (int)(r / a.N);
    const int d0 = c * VW;
    const int p0 = swap_start(d0, a.D >> 2);
    using V = Vec<T, VW>;
    using F = Vec<float, VW>;
    const int64_t hd = (int64_t)a.H * a.D;
    const T* row = reinterpret_cast<const T*>(a.qkv) + (int64_t)b * a.sb + (int64_t)n * a.sn + (int64_t)h * a.D;
    const V xq = *reinterpret_cast<const V*>(row + d0);
    const V xqs = *reinterpret_cast<const V*>(row + p0);
    const V xk = *reinterpret_cast<const V*>(row + hd + d0);
    const V xks = *reinterpret_cast<const V*>(row + hd + p0);
    const V xv = *reinterpret_cast<const V*>(row + 2 * hd + d0);
    const F cs = *reinterpret_cast<const F*>(a.cos + (int64_t)n * a.D + d0);
    const F sn = *reinterpret_cast<const F*>(a.sin + (int64_t)n * a.D + d0);
    V oq, ok;
#pragma unroll
    for (int e = 0; e < VW; ++e) {
        oq[e] = narrow<T>(f32(xq[e]) * cs[e] + f32(xqs[e]) * sn[e]);
        ok[e] = narrow<T>(f32(xk[e]) * cs[e] + f32(xks[e]) * sn[e]);
    }
    const int64_t out = (((int64_t)b * a.H + h) * a.N + n) * a.D + d0;
    float dot = 0.f;
    if constexpr (FULL) {
        if (a.w) {
            const V xw = *reinterpret_cast<const V*>(reinterpret_cast<const T*>(a.w) + out);
#pragma unroll
            for (int e = 0; e < VW; ++e) dot += f32(narrow<T>(mul_f32(f32(xw[e]), f32(oq[e]))));
        }
    }
    if (a.qs) {  // per-head temperature after the rotation: round(round(R q) * t)
        const float tq = FULL ? f32(narrow<T>(a.qs[h])) : a.qs[h];
#pragma unroll
        for (int e = 0; e < VW; ++e) oq[e] = narrow<T>(mul_f32(f32(oq[e]), tq));
    }
    if (in) {
        *reinterpret_cast<V*>(reinterpret_cast<T*>(a.q) + out) = oq;
        *reinterpret_cast<V*>(reinterpret_cast<T*>(a.k) + out) = ok;
        *reinterpret_cast<V*>(reinterpret_cast<T*>(a.v) + out) = xv;
    }
    if constexpr (FULL) {
        if (a.w) head_partials(in ? dot : 0.f, in ? h : -1, cpr, a.H, a.part);  // a.w: the same for the whole grid
    }
}

template <typename T, int VW, bool FULL> __global__ __launch_bounds__(256) void k_rope_merge(MergeArgs a) {
#pragma clang fp contract(off)
    const int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    const int cpr = a.D / VW;
    const bool in = t < a.total;
    if (!FULL && !in) return;
    const int64_t tc = FULL && !in ? a.total - 1 : t;  // past the last row: its values, neither summed nor stored
    int64_t r = tc / cpr;
    const int c = (int)(tc - r * cpr);
    const int h = (int)(r % a.H);
    r /= a.H;
    const int n = (int)(r % a.N);
    const int b = (int)(r / a.N);
    const int d0 = c * VW;
    const int p0 = swap_start(d0, a.D >> 2);
    using V = Vec<T, VW>;
    using F = Vec<float, VW>;
    const T* qr = reinterpret_cast<const T*>(a.dq) + (int64_t)b * a.sq[0] + (int64_t)h * a.sq[1] + (int64_t)n * a.sq[2];
    const T* kr = reinterpret_cast<const T*>(a.dk) + (int64_t)b * a.sk[0] + (int64_t)h * a.sk[1] + (int64_t)n * a.sk[2];
    const T* vr = reinterpret_cast<const T*>(a.dv) + (int64_t)b * a.sv[0] + (int64_t)h * a.sv[1] + (int64_t)n * a.sv[2];
    V gq = *reinterpret_cast<const V*>(qr + d0);
    V gqs = *reinterpret_cast<const V*>(qr + p0);
    V gk = *reinterpret_cast<const V*>(kr + d0);
    V gks = *reinterpret_cast<const V*>(kr + p0);
    V gv = *reinterpret_cast<const V*>(vr + d0);
    const int64_t hd = (int64_t)a.H * a.D;
    float dot = 0.f;
    if constexpr (FULL) {
        if (a.aq) {  // the sum of two gradients, rounded as a sum of its own
            const int64_t r0 = (((int64_t)b * a.H + h) * a.N + n) * a.D;
            const T* aq = reinterpret_cast<const T*>(a.aq) + r0;
            const T* ak = reinterpret_cast<const T*>(a.ak) + r0;
            const V x0 = *reinterpret_cast<const V*>(aq + d0), x1 = *reinterpret_cast<const V*>(aq + p0);
            const V x2 = *reinterpret_cast<const V*>(ak + d0), x3 = *reinterpret_cast<const V*>(ak + p0);
            const V x4 = *reinterpret_cast<const V*>(reinterpret_cast<const T*>(a.av) + r0 + d0);
#pragma unroll
            for (int e = 0; e < VW; ++e) {
                gq[e] = sum_rounded<T>(gq[e], x0[e]);
                gqs[e] = sum_rounded<T>(gqs[e], x1[e]);
                gk[e] = sum_rounded<T>(gk[e], x2[e]);
                gks[e] = sum_rounded<T>(gks[e], x3[e]);
                gv[e] = sum_rounded<T>(gv[e], x4[e]);
            }
        }
    }
    const F cs = *reinterpret_cast<const F*>(a.cos + (int64_t)n * a.D + d0);
    const F sp = *reinterpret_cast<const F*>(a.sin + (int64_t)n * a.D + p0);
    if constexpr (FULL) {
        if (a.qkv) {
            const T* row = reinterpret_cast<const T*>(a.qkv) + ((int64_t)b * a.N + n) * 3 * hd + (int64_t)h * a.D;
            const V xq = *reinterpret_cast<const V*>(row + d0), xqs = *reinterpret_cast<const V*>(row + p0);
            const F sn = *reinterpret_cast<const F*>(a.sin + (int64_t)n * a.D + d0);
#pragma unroll
            for (int e = 0; e < VW; ++e)
                dot += f32(narrow<T>(mul_f32(f32(gq[e]), f32(narrow<T>(f32(xq[e]) * cs[e] + f32(xqs[e]) * sn[e])))));
        }
    }
    float fq[VW], fqs[VW];
#pragma unroll
    for (int e = 0; e < VW; ++e) {
        fq[e] = f32(gq[e]);
        fqs[e] = f32(gqs[e]);
    }
    if (a.qs) {  // adjoint of the temperature first, rounded as the dtype's multiply is
        const float tq = FULL ? f32(narrow<T>(a.qs[h])) : a.qs[h];
#pragma unroll
        for (int e = 0; e < VW; ++e) {
            fq[e] = f32(narrow<T>(mul_f32(fq[e], tq)));
            fqs[e] = f32(narrow<T>(mul_f32(fqs[e], tq)));
        }
    }
    V oq, ok;
#pragma unroll
    for (int e = 0; e < VW; ++e) {
        oq[e] = narrow<T>(fq[e] * cs[e] + fqs[e] * sp[e]);
        ok[e] = narrow<T>(f32(gk[e]) * cs[e] + f32(gks[e]) * sp[e]);
    }
    T* out = reinterpret_cast<T*>(a.g) + ((int64_t)b * a.N + n) * 3 * hd + (int64_t)h * a.D + d0;
    if (in) {
        *reinterpret_cast<V*>(out) = oq;
        *reinterpret_cast<V*>(out + hd) = ok;
        *reinterpret_cast<V*>(out + 2 * hd) = gv;
    }
    if constexpr (FULL) {
        if (a.qkv) head_partials(in ? dot : 0.f, in ? h : -1, cpr, a.H, a.part);
    }
}

// ---------------------------------------------------------------------------------------------------------------------
// Host side
// ---------------------------------------------------------------------------------------------------------------------

constexpr int THREADS = 256;

static int es_of(int dtype) { return dtype == EBR_DTYPE_F32 ? 4 : 2; }

static int check_common(int dtype, int B, int N, int H, int D) {
    if (dtype != EBR_DTYPE_F32 && dtype != EBR_DTYPE_BF16 && dtype != EBR_DTYPE_F16) return EBR_ERR_DTYPE;
    if (B < 1 || N < 1 || H < 1 || D < 4 || D > 256 || D % 4) return EBR_ERR_SHAPE;
    if ((int64_t)B * N * H * D >= ((int64_t)1 << 40)) return EBR_ERR_SHAPE;
    return EBR_OK;
}

static bool aligned(const void* p, int bytes) { return ((uintptr_t)p % (uintptr_t)bytes) == 0; }

// Widest vector (elements) such that it divides D / 4, fits 16 bytes, and every row start and table row is aligned.
static int pick_vw(int es, int D, const void* const* ptrs, int nptr, const int64_t* strides, int nstr,
                   const float* cos, const float* sin) {
    for (int vw = 16 / es; vw > 1; vw >>= 1) {
        if ((D / 4) % vw) continue;
        const int vb = vw * es;
        bool ok = aligned(cos, vw * 4) && aligned(sin, vw * 4) && (D * 4) % (vw * 4) == 0;
        for (int i = 0; i < nptr && ok; ++i) ok = aligned(ptrs[i], vb);
        for (int i = 0; i < nstr && ok; ++i) ok = (strides[i] * es) % vb == 0;
        if (ok) return vw;
    }
    return 1;
}

static int rc_launch() {
    const hipError_t e = hipGetLastError();
    return e == hipSuccess ? EBR_OK : EBR_ERR_HIP_BASE + (int)e;
}

template <typename T, int VW, bool FULL = false> static int launch_split(SplitArgs a, hipStream_t s) {
    a.total = (int64_t)a.B * a.H * a.N * (a.D / VW);
    const int64_t blocks = (a.total + THREADS - 1) / THREADS;
    if (blocks >= ((int64_t)1 << 31)) return EBR_ERR_SHAPE;
    hipLaunchKernelGGL((k_rope_split<T, VW, FULL>), dim3((unsigned)blocks), dim3(THREADS), 0, s, a);
    return rc_launch();
}

template <typename T, int VW, bool FULL = false> static int launch_merge(MergeArgs a, hipStream_t s) {
    a.total = (int64_t)a.B * a.N * a.H * (a.D / VW);
    const int64_t blocks = (a.total + THREADS - 1) / THREADS;
    if (blocks >= ((int64_t)1 << 31)) return EBR_ERR_SHAPE;
    hipLaunchKernelGGL((k_rope_merge<T, VW, FULL>), dim3((unsigned)blocks), dim3(THREADS), 0, s, a);
    return rc_launch();
}

template <typename T> static int split_vw(int vw, SplitArgs a, hipStream_t s) {
    if constexpr (sizeof(T) == 2) {
        if (vw == 8) return launch_split<T, 8>(a, s);
    }
    if (vw == 4) return launch_split<T, 4>(a, s);
    if (vw == 2) return launch_split<T, 2>(a, s);
    return launch_split<T, 1>(a, s);
}

template <typename T> static int merge_vw(int vw, MergeArgs a, hipStream_t s) {
    if constexpr (sizeof(T) == 2) {
        if (vw == 8) return launch_merge<T, 8>(a, s);
    }
    if (vw == 4) return launch_merge<T, 4>(a, s);
    if (vw == 2) return launch_merge<T, 2>(a, s);
    return launch_merge<T, 1>(a, s);
}

// The graded entries take whole 16-byte vectors and a power of two of them per row.
static bool full_width(int es, int D) {
    const int vw = 16 / es, cpr = D / vw;
    return D % (4 * vw) == 0 && cpr <= 64 && (cpr & (cpr - 1)) == 0;
}

static int64_t full_blocks(int es, int B, int N, int H, int D) {
    return ((int64_t)B * N * H * (D / (16 / es)) + THREADS - 1) / THREADS;
}

template <typename T> static int head_sums(const float* part, int64_t n, int H, float* dt, hipStream_t s) {
    hipLaunchKernelGGL((k_head_sums<T>), dim3((unsigned)H), dim3(SUM_THREADS), 0, s, part, n, H, dt);
    return rc_launch();
}

static int head_sums_of(int dtype, const float* part, int64_t n, int H, float* dt, hipStream_t s) {
    if (dtype == EBR_DTYPE_F32) return head_sums<float>(part, n, H, dt, s);
    if (dtype == EBR_DTYPE_BF16) return head_sums<__bf16>(part, n, H, dt, s);
    return head_sums<_Float16>(part, n, H, dt, s);
}

}  // namespace ebr_rope

using namespace ebr_rope;

extern "C" {

int ebr_rope_split(int dtype, int B, int N, int H, int D, const void* qkv, int64_t qkv_sb, int64_t qkv_sn,
                   const float* cos, const float* sin, const float* qscale, void* q, void* k, void* v,
                   void* stream) {
    int rc = check_common(dtype, B, N, H, D);
    if (rc) return rc;
    if (!qkv || !cos || !sin || !q || !k || !v) return EBR_ERR_NULL;
    if (qkv_sb < 0 || qkv_sn < 0) return EBR_ERR_SHAPE;
    const int es = es_of(dtype);
    SplitArgs a = {};
    a.qkv = qkv;
    a.sb = qkv_sb;
    a.sn = qkv_sn;
    a.cos = cos;
    a.sin = sin;
    a.qs = qscale;
    a.q = q;
    a.k = k;
    a.v = v;
    a.B = B;
    a.N = N;
    a.H = H;
    a.D = D;
    const void* ptrs[4] = {qkv, q, k, v};
    const int64_t strides[2] = {qkv_sb, qkv_sn};
    const int vw = pick_vw(es, D, ptrs, 4, strides, 2, cos, sin);
    hipStream_t s = reinterpret_cast<hipStream_t>(stream);
    if (dtype == EBR_DTYPE_F32) return split_vw<float>(vw, a, s);
    if (dtype == EBR_DTYPE_BF16) return split_vw<__bf16>(vw, a, s);
    return split_vw<_Float16>(vw, a, s);
}

int ebr_rope_merge(int dtype, int B, int H, int N, int D, const void* dq, const int64_t dq_str[3], const void* dk,
                   const int64_t dk_str[3], const void* dv, const int64_t dv_str[3], const float* cos,
                   const float* sin, const float* qscale, void* g, void* stream) {
    int rc = check_common(dtype, B, N, H, D);
    if (rc) return rc;
    if (!dq || !dk || !dv || !dq_str || !dk_str || !dv_str || !cos || !sin || !g) return EBR_ERR_NULL;
    MergeArgs a = {};
    for (int i = 0; i < 3; ++i) {
        if (dq_str[i] < 0 || dk_str[i] < 0 || dv_str[i] < 0) return EBR_ERR_SHAPE;
        a.sq[i] = dq_str[i];
        a.sk[i] = dk_str[i];
        a.sv[i] = dv_str[i];
    }
    const int es = es_of(dtype);
    a.dq = dq;
    a.dk = dk;
    a.dv = dv;
    a.cos = cos;
    a.sin = sin;
    a.qs = qscale;
    a.g = g;
    a.B = B;
    a.H = H;
    a.N = N;
    a.D = D;
    const void* ptrs[4] = {dq, dk, dv, g};
    const int64_t strides[9] = {dq_str[0], dq_str[1], dq_str[2], dk_str[0], dk_str[1],
                                dk_str[2], dv_str[0], dv_str[1], dv_str[2]};
    const int vw = pick_vw(es, D, ptrs, 4, strides, 9, cos, sin);
    hipStream_t s = reinterpret_cast<hipStream_t>(stream);
    if (dtype == EBR_DTYPE_F32) return merge_vw<float>(vw, a, s);
    if (dtype == EBR_DTYPE_BF16) return merge_vw<__bf16>(vw, a, s);
    return merge_vw<_Float16>(vw, a, s);
}

int64_t ebr_rope_graded_scratch(int dtype, int B, int N, int H, int D) {
    if (check_common(dtype, B, N, H, D) || !full_width(es_of(dtype), D)) return 0;
    return full_blocks(es_of(dtype), B, N, H, D) * H * 4;
}

int ebr_rope_split_graded(int dtype, int B, int N, int H, int D, const void* qkv, int64_t qkv_sb, int64_t qkv_sn,
                          const float* cos, const float* sin, const float* t, void* q, void* k, void* v,
                          const void* w, float* dt, float* scratch, void* stream) {
    int rc = check_common(dtype, B, N, H, D);
    if (rc) return rc;
    const int es = es_of(dtype);
    if (!full_width(es, D)) return EBR_ERR_SHAPE;
    if (!qkv || !cos || !sin || !t || !q || !k || !v) return EBR_ERR_NULL;
    if (w && (!dt || !scratch)) return EBR_ERR_SCRATCH;
    if (qkv_sb < 0 || qkv_sn < 0) return EBR_ERR_SHAPE;
    SplitArgs a = {};
    a.qkv = qkv;
    a.sb = qkv_sb;
    a.sn = qkv_sn;
    a.cos = cos;
    a.sin = sin;
    a.qs = t;
    a.q = q;
    a.k = k;
    a.v = v;
    a.B = B;
    a.N = N;
    a.H = H;
    a.D = D;
    a.w = w;
    a.part = scratch;
    const void* ptrs[5] = {qkv, q, k, v, w};
    const int64_t strides[2] = {qkv_sb, qkv_sn};
    if (pick_vw(es, D, ptrs, 5, strides, 2, cos, sin) != 16 / es) return EBR_ERR_ALIGN;
    hipStream_t s = reinterpret_cast<hipStream_t>(stream);
    if (dtype == EBR_DTYPE_F32) rc = launch_split<float, 4, true>(a, s);
    else if (dtype == EBR_DTYPE_BF16) rc = launch_split<__bf16, 8, true>(a, s);
    else rc = launch_split<_Float16, 8, true>(a, s);
    if (rc || !w) return rc;
    return head_sums_of(dtype, scratch, full_blocks(es, B, N, H, D), H, dt, s);
}

int ebr_rope_merge_graded(int dtype, int B, int H, int N, int D, const void* dq, const int64_t dq_str[3],
                          const void* dk, const int64_t dk_str[3], const void* dv, const int64_t dv_str[3],
                          const void* aq, const void* ak, const void* av, const float* cos, const float* sin,
                          const float* t, void* g, const void* qkv, float* dt, float* scratch, void* stream) {
    int rc = check_common(dtype, B, N, H, D);
    if (rc) return rc;
    const int es = es_of(dtype);
    if (!full_width(es, D)) return EBR_ERR_SHAPE;
    if (!dq || !dk || !dv || !dq_str || !dk_str || !dv_str || !cos || !sin || !t || !g) return EBR_ERR_NULL;
    if ((!aq != !ak) || (!aq != !av)) return EBR_ERR_NULL;
    if (qkv && (!dt || !scratch)) return EBR_ERR_SCRATCH;
    MergeArgs a = {};
    for (int i = 0; i < 3; ++i) {
        if (dq_str[i] < 0 || dk_str[i] < 0 || dv_str[i] < 0) return EBR_ERR_SHAPE;
        a.sq[i] = dq_str[i];
        a.sk[i] = dk_str[i];
        a.sv[i] = dv_str[i];
    }
    a.dq = dq;
    a.dk = dk;
    a.dv = dv;
    a.aq = aq;
    a.ak = ak;
    a.av = av;
    a.cos = cos;
    a.sin = sin;
    a.qs = t;
    a.g = g;
    a.qkv = qkv;
    a.part = scratch;
    a.B = B;
    a.H = H;
    a.N = N;
    a.D = D;
    const void* ptrs[8] = {dq, dk, dv, g, aq, ak, av, qkv};
    const int64_t strides[9] = {dq_str[0], dq_str[1], dq_str[2], dk_str[0], dk_str[1],
                                dk_str[2], dv_str[0], dv_str[1], dv_str[2]};
    if (pick_vw(es, D, ptrs, 8, strides, 9, cos, sin) != 16 / es) return EBR_ERR_ALIGN;
    hipStream_t s = reinterpret_cast<hipStream_t>(stream);
    if (dtype == EBR_DTYPE_F32) rc = launch_merge<float, 4, true>(a, s);
    else if (dtype == EBR_DTYPE_BF16) rc = launch_merge<__bf16, 8, true>(a, s);
    else rc = launch_merge<_Float16, 8, true>(a, s);
    if (rc || !qkv) return rc;
    return head_sums_of(dtype, scratch, full_blocks(es, B, N, H, D), H, dt, s);
}

}  // extern "C"
