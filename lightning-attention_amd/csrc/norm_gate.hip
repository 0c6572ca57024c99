// Gated output norm of the TNL attention block for gfx950:
//     y = LayerNorm(o; weight, bias, eps) * sigmoid(g)
// forward and backward as row kernels (examples/module/tnl_attn.py:66-69 of the reference, where it
// is three separate PyTorch operators: LayerNorm, sigmoid and a product - seven passes over
// (tokens, embed_dim) tensors forward and eleven backward; here three and five).
//
// Same data movement as the SimpleRMSNorm kernels: a row of o, g (and dy) is read once with 16-byte
// non-temporal loads into registers, reduced, and the results written once.  TPR threads share a row:
// 8, 16, 32, 64, 128, 256, 512 or 1024, with as many rows side by side as the workgroup has room for.  The
// forward kernel takes one group of rows per workgroup and fetches weight and bias from the caches; it is bound by memory, once
// nothing waits between its reductions: us, before weight and bias came along with the row and before short rows shared a
// wavefront / now, bf16: [16384,2048] 38.3 / 33.0 (6.1 TB/s), [4096,8192] 39.6 / 36.0, [16384,1024] 19.0 / 17.1, [700,2048] 6.0 / 4.6,
// [131072,64] 49.3 / 10.1, [40000,200] 19.1 / 11.7; float32 [16384,1024] 37.6 / 31.9, [131072,64] 41.1 / 16.9.  The backward kernel walks the rows with a grid stride and gives every thread one
// 16-byte chunk of the row: a thread always holds the same columns, so weight and bias stay in registers
// as floats and the column sums (d weight, d bias) are accumulated in registers over all rows a thread
// sees (117 registers: four waves per SIMD; with more chunks per thread it ran at two).  Those partial
// sums go to a scratch buffer, one row per workgroup, and a second small kernel adds them up in a fixed
// order: deterministic, no atomics.
// The backward kernel is bound by what it keeps in flight, not by its arithmetic: with 16-bit elements the next group of
// rows is requested before the reduction of this one (float32 runs five waves per SIMD and gains nothing), weight and
// bias come in one 16-byte load each, and a CU holds one workgroup of 1024 threads and so writes one row of partial sums
// (rows of up to 2048 elements: of four, up to 4096 of two; wider rows had such workgroups already).  Few short rows take
// workgroups of 256 threads, a pass and a CU each: us with 1024 / with 256, bf16: [16,64] 7.2 / 6.0, [512,256] 8.0 / 6.4,
// [1024,512] 8.3 / 7.1, [512,1024] 8.2 / 7.8.
// Backward pass with its reduction, bf16, us before / after: [16384,2048] 87.2 / 62.9 (5.3 TB/s), [8192,1024] 33.9 / 22.6,
// [32768,4096] 259 / 225 (6.0 TB/s), [32768,512] 42.0 / 34.7, [4096,8192] 85.5 / 65.1, [700,2048] 22.7 / 9.8.  float32 has the
// vector loads alone: [16384,4096] 252 / 236, [1024,1024] 17.4 / 14.7, [16,64] the same.
//
// Per element, float32 throughout:
//   forward   xh = (o - mean) rstd ; ln = xh w + b ; sg = 1 / (1 + exp(-g)) ; y = ln sg
//   backward  dln = dy sg ; dg = dy ln sg (1 - sg) ; dxh = dln w ;
//             do = rstd (dxh - mean_c(dxh) - xh mean_c(dxh xh)) ; dw += dln xh ; db += dln
#include "la_rows.h"
#include "lightning_attn_hip.h"

namespace la {

// Threads of a workgroup: TPR threads share a row; rows of up to two wavefronts travel 256 / TPR to a
// workgroup of 256, wider rows take a workgroup of 256, 512 or 1024 threads to themselves.
constexpr int ng_threads(int tpr) { return tpr >= 256 ? tpr : 256; }
// The backward kernel with 16-bit elements: 1024 threads (its registers leave a CU 16 wavefronts either way), so that a CU
// leaves one row of partial column sums, not one per workgroup.  `few`: rows of one or two wavefronts, so few that workgroups of 256
// threads get a CU and one pass each (ng_few): there is nothing to add up over passes then, and the rows of a 1024-thread
// workgroup, added up one after the other, are what it waits for.
constexpr int ng_bwd_threads(int tpr, int elt, bool few) { return elt == 2 && !few ? 1024 : ng_threads(tpr); }

// both sums over the TPR threads of a row at once (every thread of the workgroup takes part)
// ONCE: the caller hands over another 32 floats of LDS on every other call, so that the next call's writes cannot meet
// this one's reads and one barrier will do
template <int TPR, bool ONCE = false>
__device__ __forceinline__ void row_sum2(float& a, float& b, float* red) {
    if (TPR >= 128) {
        constexpr int NWV = TPR / 64;  // wavefronts per row
        a = wave_sum(a);
        b = wave_sum(b);
        const int w = threadIdx.x >> 6, w0 = w / NWV * NWV;
        if ((threadIdx.x & 63) == 0) {
            red[w] = a;
            red[16 + w] = b;
        }
        __syncthreads();
        a = b = 0.f;
#pragma unroll
        for (int i = 0; i < NWV; ++i) {
            a += red[w0 + i];
            b += red[16 + w0 + i];
        }
        if (!ONCE) __syncthreads();
        return;
    }
#pragma unroll
    for (int m = TPR / 2; m >= 1; m >>= 1) {
        a += __shfl_xor(a, m, 64);
        b += __shfl_xor(b, m, 64);
    }
}

// 1 / (1 + exp(-x)) with the hardware's exp2 and reciprocal (about 1 ulp each); an IEEE division
// would cost more instructions than the rest of the element's arithmetic
__device__ __forceinline__ float sigmoidf(float x) {
    return __builtin_amdgcn_rcpf(1.0f + __builtin_amdgcn_exp2f(x * -1.44269504088896340736f));
}

template <typename T, int NV, int TPR>
__global__ __launch_bounds__(ng_threads(TPR)) void norm_gate_fwd_kernel(const T* __restrict__ o, const T* __restrict__ g,
                                                                  const T* __restrict__ w, const T* __restrict__ b,
                                                                  T* __restrict__ y, float* __restrict__ mean,
                                                                  float* __restrict__ rstd, int64_t rows, int cols, float eps) {
    constexpr int E = Pack16<T>::N;
    constexpr int RPG = ng_threads(TPR) / TPR;  // rows a workgroup holds
    __shared__ float red[32];
    const int l = threadIdx.x % TPR;
    const float inv = 1.0f / (float)cols;
    const int64_t row = (int64_t)blockIdx.x * RPG + threadIdx.x / TPR;
    const bool row_ok = row < rows;
    const T* orow = o + row * (int64_t)cols;
    const T* grow = g + row * (int64_t)cols;
    T* yrow = y + row * (int64_t)cols;
    // weight and bias come from the caches (every row reads the same cols elements).  Requested along with the row, so that
    // the last pass does not wait for them - but for float32 rows of several wavefronts, where the registers cost more
    // ([32768,4096] 259 / 268 us).
    constexpr bool EARLY = sizeof(T) == 2 || TPR <= 64;
    Pack16<T> po[NV], pg[NV], pw[NV], pb[NV];
    auto affine = [&]() __attribute__((always_inline)) {
#pragma unroll
        for (int u = 0; u < NV; ++u) {
            const int c = (u * TPR + l) * E;
            if (row_ok && c < cols) {
                pw[u] = *reinterpret_cast<const Pack16<T>*>(w + c);
                pb[u] = *reinterpret_cast<const Pack16<T>*>(b + c);
            }
        }
    };
#pragma unroll
    for (int u = 0; u < NV; ++u) {
        const int c = (u * TPR + l) * E;
        if (row_ok && c < cols) {
            po[u] = load16(orow + c);
            pg[u] = load16(grow + c);
        }
    }
    if (EARLY) affine();
    float s = 0.f, dummy = 0.f;
#pragma unroll
    for (int u = 0; u < NV; ++u) {
        const int c = (u * TPR + l) * E;
        if (row_ok && c < cols) {
#pragma unroll
            for (int t = 0; t < E; ++t) s += (float)po[u].v[t];
        }
    }
    row_sum2<TPR>(s, dummy, red);
    const float mu = s * inv;
    // only the packed inputs live across the reductions: the passes convert them again
#pragma unroll
    for (int u = 0; u < NV; ++u) forget(po[u]);
    float ss = 0.f;
#pragma unroll
    for (int u = 0; u < NV; ++u) {
        const int c = (u * TPR + l) * E;
        if (row_ok && c < cols) {
#pragma unroll
            for (int t = 0; t < E; ++t) {
                const float dlt = (float)po[u].v[t] - mu;
                ss += dlt * dlt;
            }
        }
    }
    row_sum2<TPR>(ss, dummy, red);
    const float rs = 1.0f / sqrtf(ss * inv + eps);
#pragma unroll
    for (int u = 0; u < NV; ++u) {
        forget(po[u]);
        forget(pg[u]);
        if (EARLY) {
            forget(pw[u]);
            forget(pb[u]);
        }
    }
    if (!EARLY) affine();
    if (l == 0 && row_ok) {
        mean[row] = mu;
        rstd[row] = rs;
    }
#pragma unroll
    for (int u = 0; u < NV; ++u) {
        const int c = (u * TPR + l) * E;
        if (row_ok && c < cols) {
            Pack16<T> out;
#pragma unroll
            for (int t = 0; t < E; ++t) {
                const float ln = ((float)po[u].v[t] - mu) * rs * (float)pw[u].v[t] + (float)pb[u].v[t];
                out.v[t] = (T)(ln * sigmoidf((float)pg[u].v[t]));
            }
            store16(yrow + c, out);
        }
    }
}

typedef float Quad __attribute__((ext_vector_type(4), aligned(4)));  // (the workspace need not be 16-byte aligned)

// `part`: gridDim.x rows of [d weight | d bias] partial column sums, 2 * cols floats each.
template <typename T, int NV, int TPR, bool FEW = false>
__global__ __launch_bounds__(ng_bwd_threads(TPR, sizeof(T), FEW)) void norm_gate_bwd_kernel(const T* __restrict__ o, const T* __restrict__ g,
                                                                  const T* __restrict__ w, const T* __restrict__ b,
                                                                  const float* __restrict__ mean, const float* __restrict__ rstd,
                                                                  const T* __restrict__ dy, T* __restrict__ d_o,
                                                                  T* __restrict__ d_g, float* __restrict__ part,
                                                                  int64_t rows, int cols) {
    constexpr int E = Pack16<T>::N;
    constexpr int RPG = ng_bwd_threads(TPR, sizeof(T), FEW) / TPR;
    constexpr bool AHEAD = sizeof(T) == 2;
    constexpr int SIDE = TPR < 64 ? RPG * TPR / 64 : RPG;  // column sums to add up once the rows of a wavefront are
    __shared__ float red[64];
    __shared__ float comb[SIDE > 1 ? (SIDE - 1) * TPR * NV * E * 2 : 1];  // column sums of the rows beside the first
    const int l = threadIdx.x % TPR;
    float wf[NV][E], bf[NV][E];  // this thread's columns of weight and bias
    float aw[NV][E], ab[NV][E];  // ... and of the column sums
#pragma unroll
    for (int u = 0; u < NV; ++u) {
        // (one 16-byte load each: element by element every load waited for the one before it, 10 us per workgroup)
        const int c = (u * TPR + l) * E;
        Pack16<T> pw, pb;
        if (c < cols) {
            pw = *reinterpret_cast<const Pack16<T>*>(w + c);
            pb = *reinterpret_cast<const Pack16<T>*>(b + c);
        }
#pragma unroll
        for (int t = 0; t < E; ++t) {
            wf[u][t] = c < cols ? (float)pw.v[t] : 0.f;
            bf[u][t] = c < cols ? (float)pb.v[t] : 0.f;
            aw[u][t] = ab[u][t] = 0.f;
        }
    }
    const float inv = 1.0f / (float)cols;
    // The next group of rows is requested as soon as the first pass has used up the packed registers of this one, so
    // that its memory latency runs beside the reduction, the second pass and the stores.
    const int64_t step = (int64_t)gridDim.x * RPG;
    Pack16<T> po[NV], pg[NV], py[NV];
    float mu_next = 0.f, rs_next = 0.f;
    auto fetch = [&](int64_t row) __attribute__((always_inline)) {
        if (row < rows) {
            const int64_t at = row * (int64_t)cols;
#pragma unroll
            for (int u = 0; u < NV; ++u) {
                const int c = (u * TPR + l) * E;
                if (c < cols) {
                    po[u] = load16(o + at + c);
                    pg[u] = load16(g + at + c);
                    py[u] = load16(dy + at + c);
                }
            }
            mu_next = mean[row];
            rs_next = rstd[row];
        }
    };
    if (AHEAD) fetch((int64_t)blockIdx.x * RPG + threadIdx.x / TPR);
    int turn = 0;
    for (int64_t row0 = (int64_t)blockIdx.x * RPG; row0 < rows; row0 += step, turn ^= 1) {
        const int64_t row = row0 + threadIdx.x / TPR;
        const bool row_ok = row < rows;
        if (!AHEAD) fetch(row);
        const float mu = mu_next, rs = rs_next;
        // Kept from the first pass for the second: xh, dln and 1 - sigmoid(g) (one exp and one
        // reciprocal per element in all; the kernel is close to its VALU budget, not only to HBM's).
        float xh[NV][E], dln[NV][E], cs[NV][E];
        float s1 = 0.f, s2 = 0.f;
        const float shift = -mu * rs;
#pragma unroll
        for (int u = 0; u < NV; ++u) {
            const int c = (u * TPR + l) * E;
            if (row_ok && c < cols) {
#pragma unroll
                for (int t = 0; t < E; ++t) {
                    xh[u][t] = (float)po[u].v[t] * rs + shift;
                    const float sv = sigmoidf((float)pg[u].v[t]);
                    cs[u][t] = 1.0f - sv;
                    dln[u][t] = (float)py[u].v[t] * sv;
                    const float dxh = dln[u][t] * wf[u][t];
                    s1 += dxh;
                    s2 += dxh * xh[u][t];
                    aw[u][t] += dln[u][t] * xh[u][t];
                    ab[u][t] += dln[u][t];
                }
            }
        }
        if (AHEAD) fetch(row + step);
        row_sum2<TPR, true>(s1, s2, red + 32 * turn);
        const float k1 = s1 * inv * rs, k2 = s2 * inv * rs;
#pragma unroll
        for (int u = 0; u < NV; ++u) {
            const int c = (u * TPR + l) * E;
            if (row_ok && c < cols) {
                Pack16<T> out_o, out_g;
#pragma unroll
                for (int t = 0; t < E; ++t) {
                    // do = rstd (dxh - mean(dxh) - xh mean(dxh xh)) ; dg = dy ln sg (1 - sg) = dln ln (1 - sg)
                    out_o.v[t] = (T)(dln[u][t] * wf[u][t] * rs - k1 - xh[u][t] * k2);
                    const float ln = xh[u][t] * wf[u][t] + bf[u][t];
                    out_g.v[t] = (T)(dln[u][t] * ln * cs[u][t]);
                }
                store16(d_o + row * (int64_t)cols + c, out_o);
                store16(d_g + row * (int64_t)cols + c, out_g);
            }
        }
    }
    // column sums of this workgroup: the thread groups of its rows hold the same columns and are
    // added up in a fixed order first, those of a wavefront by shuffles (after which its first TPR lanes, `owner`, speak for it)
    const bool owner = TPR >= 64 || (threadIdx.x & 63) < TPR;
    const int grp = threadIdx.x / (TPR < 64 ? 64 : TPR);
    if (TPR < 64) {
#pragma unroll
        for (int u = 0; u < NV; ++u)
#pragma unroll
            for (int t = 0; t < E; ++t)
#pragma unroll
                for (int m = TPR; m < 64; m *= 2) {
                    aw[u][t] += __shfl_xor(aw[u][t], m, 64);
                    ab[u][t] += __shfl_xor(ab[u][t], m, 64);
                }
    }
    if (SIDE > 1) {
        if (owner && grp > 0) {
#pragma unroll
            for (int u = 0; u < NV; ++u)
#pragma unroll
                for (int t = 0; t < E; ++t) {
                    comb[((((grp - 1) * NV + u) * E + t) * 2 + 0) * TPR + l] = aw[u][t];
                    comb[((((grp - 1) * NV + u) * E + t) * 2 + 1) * TPR + l] = ab[u][t];
                }
        }
        __syncthreads();  // (every thread of the workgroup comes by here)
    }
    if (!owner || grp > 0) return;
    if (SIDE > 1) {
#pragma unroll
        for (int k = 0; k < SIDE - 1; ++k)
#pragma unroll
            for (int u = 0; u < NV; ++u)
#pragma unroll
                for (int t = 0; t < E; ++t) {
                    aw[u][t] += comb[(((k * NV + u) * E + t) * 2 + 0) * TPR + l];
                    ab[u][t] += comb[(((k * NV + u) * E + t) * 2 + 1) * TPR + l];
                }
    }
    float* prow = part + (size_t)blockIdx.x * 2 * cols;
#pragma unroll
    for (int u = 0; u < NV; ++u) {
        const int c = (u * TPR + l) * E;
        if (c < cols) {
#pragma unroll
            for (int t = 0; t < E; t += 4) {
                *reinterpret_cast<Quad*>(prow + c + t) = Quad{aw[u][t], aw[u][t + 1], aw[u][t + 2], aw[u][t + 3]};
                *reinterpret_cast<Quad*>(prow + cols + c + t) = Quad{ab[u][t], ab[u][t + 1], ab[u][t + 2], ab[u][t + 3]};
            }
        }
    }
}

// d weight[c] = sum over the partial rows, in a fixed order: 32 columns per workgroup, 32 interleaved
// partial sums per column (eight independent loads in flight each) combined through LDS.
constexpr int kRedCols = 32, kRedGroups = 32;
template <typename T>
__global__ __launch_bounds__(kRedCols * kRedGroups) void norm_gate_reduce_kernel(const float* __restrict__ part, int nparts,
                                                                                 int cols, T* __restrict__ dweight,
                                                                                 T* __restrict__ dbias) {
    __shared__ float acc[kRedGroups][2 * kRedCols];
    const int lane = threadIdx.x % kRedCols, grp = threadIdx.x / kRedCols;
    const int c = blockIdx.x * kRedCols + lane;
    float sw = 0.f, sb = 0.f;
    if (c < cols) {
        constexpr int U = 8;
        for (int p0 = grp; p0 < nparts; p0 += kRedGroups * U) {
            float vw[U], vb[U];
#pragma unroll
            for (int i = 0; i < U; ++i) {
                const int p = p0 + i * kRedGroups;
                vw[i] = p < nparts ? part[(size_t)p * 2 * cols + c] : 0.f;
                vb[i] = p < nparts ? part[(size_t)p * 2 * cols + cols + c] : 0.f;
            }
#pragma unroll
            for (int i = 0; i < U; ++i) {
                sw += vw[i];
                sb += vb[i];
            }
        }
    }
    acc[grp][lane] = sw;
    acc[grp][kRedCols + lane] = sb;
    __syncthreads();
    if (grp == 0 && c < cols) {
        float tw = 0.f, tb = 0.f;
#pragma unroll
        for (int k = 0; k < kRedGroups; ++k) {
            tw += acc[k][lane];
            tb += acc[k][kRedCols + lane];
        }
        dweight[c] = (T)tw;
        dbias[c] = (T)tb;
    }
}

// Threads per row and 16-byte chunks per thread for rows of `chunks` chunks (nv = 0: too wide).  The
// forward kernel holds little per column and gives a wavefront rows of up to 256 chunks, or several short ones; the backward
// kernel carries weight, bias and two column sums per column and spreads rows over the workgroup earlier.
static void ng_shape(int64_t rows, int64_t chunks, bool backward, int* tpr, int* nv) {
    *nv = 0;
    if (backward) {
        // one chunk per thread: the kernel keeps ~7 floats per element of a thread's columns
        if (chunks > 1024) return;
        *nv = 1;
        // short rows share a wavefront where a row to a wavefront would take more than one pass (us, bf16, a row to a wavefront / shared:
        // [131072,64] 63.6 / 20.8, [16384,64] 14.0 / 9.8, [40000,200] 27.4 / 21.0; but [1,64] 4.9 / 5.7, [512,256] 6.0 / 6.5)
        const bool many = rows > 16 * (int64_t)num_cus();
        *tpr = many && chunks <= 8 ? 8 : many && chunks <= 16 ? 16 : many && chunks <= 32 ? 32 : chunks <= 64 ? 64 : chunks <= 128 ? 128 : chunks <= 256 ? 256 : chunks <= 512 ? 512 : 1024;
        return;
    }
    if (chunks <= 64 * 4) {
        *tpr = chunks <= 8 ? 8 : chunks <= 16 ? 16 : chunks <= 32 ? 32 : 64;
        *nv = 1;
        while (64 * *nv < chunks) *nv *= 2;
    } else if (chunks <= 256 * 4) {
        *tpr = 256;
        *nv = chunks <= 256 ? 1 : chunks <= 512 ? 2 : 4;
    }
}

// backward, 16-bit rows of up to 1024 elements: at most one group of rows of a 256-thread workgroup per CU (with 16 or 32 threads to
// a row, that is 16 or 8 rows per CU, never: ng_shape gives rows so few a wavefront each)
static bool ng_few(int64_t rows, int tpr, int elt) {
    const int64_t rpg = ng_threads(tpr) / tpr;
    return elt == 2 && tpr <= 128 && (rows + rpg - 1) / rpg <= num_cus();
}

// workgroups of a launch: enough to keep every CU's memory pipeline full, never more than row groups
static int64_t ng_grid(int64_t rows, int tpr, bool backward, int elt) {
    const int64_t threads = backward ? ng_bwd_threads(tpr, elt, ng_few(rows, tpr, elt)) : ng_threads(tpr), rpg = threads / tpr, groups = (rows + rpg - 1) / rpg;
    if (!backward) return groups;  // nothing is carried from row to row: one group of rows per workgroup
    const int64_t cap = 4 * (int64_t)num_cus() * 256 / threads;  // ~16 wavefronts per CU
    return groups < cap ? groups : cap;
}

// Bytes that the column sums (d weight, d bias) of a backward launch take, a row of them per workgroup.  Rows that share a wavefront
// are asked for in as many bytes as if they did not (`asked`): the same from 16 rows per CU on, so that memory which is enough for many
// of them is enough for the few that get a wavefront each.
static size_t ng_part_bytes(int64_t rows, int64_t cols, int elt, bool asked) {
    int tpr = 0, nv = 0;
    ng_shape(rows, cols * elt / 16, true, &tpr, &nv);
    return (size_t)ng_grid(rows, asked && tpr < 64 ? 64 : tpr, true, elt) * 2 * (size_t)cols * sizeof(float);
}

#define LA_NG_GO(KERNEL, NV, TPR, THREADS, ...) hipLaunchKernelGGL((KERNEL<T, NV, TPR>), grid, dim3(THREADS), 0, st, __VA_ARGS__)
#define LA_NG_DISPATCH_FWD(KERNEL, ...)                               \
    do {                                                              \
        if (tpr == 8) LA_NG_GO(KERNEL, 1, 8, ng_threads(8), __VA_ARGS__);                     \
        else if (tpr == 16) LA_NG_GO(KERNEL, 1, 16, ng_threads(16), __VA_ARGS__);             \
        else if (tpr == 32) LA_NG_GO(KERNEL, 1, 32, ng_threads(32), __VA_ARGS__);             \
        else if (tpr == 64 && nv == 1) LA_NG_GO(KERNEL, 1, 64, ng_threads(64), __VA_ARGS__);  \
        else if (tpr == 64 && nv == 2) LA_NG_GO(KERNEL, 2, 64, ng_threads(64), __VA_ARGS__);  \
        else if (tpr == 64) LA_NG_GO(KERNEL, 4, 64, ng_threads(64), __VA_ARGS__);             \
        else if (nv == 1) LA_NG_GO(KERNEL, 1, 256, ng_threads(256), __VA_ARGS__);              \
        else if (nv == 2) LA_NG_GO(KERNEL, 2, 256, ng_threads(256), __VA_ARGS__);              \
        else LA_NG_GO(KERNEL, 4, 256, ng_threads(256), __VA_ARGS__);                           \
    } while (0)
#define LA_NG_BWD(TPR, FEW, ...) hipLaunchKernelGGL((norm_gate_bwd_kernel<T, 1, TPR, FEW>), grid, dim3(ng_bwd_threads(TPR, sizeof(T), FEW)), 0, st, __VA_ARGS__)
#define LA_NG_DISPATCH_BWD(...)                                       \
    do {                                                              \
        constexpr bool kFew = sizeof(T) == 2;                         \
        const bool few = ng_few(rows, tpr, sizeof(T));                \
        if (tpr == 8 && few) LA_NG_BWD(8, kFew, __VA_ARGS__);         \
        else if (tpr == 64 && few) LA_NG_BWD(64, kFew, __VA_ARGS__);  \
        else if (tpr == 128 && few) LA_NG_BWD(128, kFew, __VA_ARGS__); \
        else if (tpr == 8) LA_NG_BWD(8, false, __VA_ARGS__);          \
        else if (tpr == 16) LA_NG_BWD(16, false, __VA_ARGS__);        \
        else if (tpr == 32) LA_NG_BWD(32, false, __VA_ARGS__);        \
        else if (tpr == 64) LA_NG_BWD(64, false, __VA_ARGS__);        \
        else if (tpr == 128) LA_NG_BWD(128, false, __VA_ARGS__);      \
        else if (tpr == 256) LA_NG_BWD(256, false, __VA_ARGS__);      \
        else if (tpr == 512) LA_NG_BWD(512, false, __VA_ARGS__);      \
        else LA_NG_BWD(1024, false, __VA_ARGS__);                     \
    } while (0)

template <typename T>
static int ng_fwd(const void* o, const void* g, const void* w, const void* b, void* y, float* mean, float* rstd, int64_t rows,
                  int64_t cols, float eps, hipStream_t st) {
    int tpr = 0, nv = 0;
    ng_shape(rows, cols / (16 / (int64_t)sizeof(T)), false, &tpr, &nv);
    if (!nv) return LA_E_UNSUPPORTED;
    const dim3 grid((unsigned)ng_grid(rows, tpr, false, sizeof(T)));
    LA_NG_DISPATCH_FWD(norm_gate_fwd_kernel, static_cast<const T*>(o), static_cast<const T*>(g), static_cast<const T*>(w),
                   static_cast<const T*>(b), static_cast<T*>(y), mean, rstd, rows, (int)cols, eps);
    return (int)hipGetLastError();
}

template <typename T>
static int ng_bwd(const void* o, const void* g, const void* w, const void* b, const float* mean, const float* rstd,
                  const void* dy, void* d_o, void* d_g, void* dweight, void* dbias, float* part, int64_t rows, int64_t cols,
                  hipStream_t st) {
    int tpr = 0, nv = 0;
    ng_shape(rows, cols / (16 / (int64_t)sizeof(T)), true, &tpr, &nv);
    if (!nv) return LA_E_UNSUPPORTED;
    const dim3 grid((unsigned)ng_grid(rows, tpr, true, sizeof(T)));
    LA_NG_DISPATCH_BWD(static_cast<const T*>(o), static_cast<const T*>(g), static_cast<const T*>(w),
                   static_cast<const T*>(b), mean, rstd, static_cast<const T*>(dy), static_cast<T*>(d_o), static_cast<T*>(d_g),
                   part, rows, (int)cols);
    int rc = (int)hipGetLastError();
    if (rc != 0) return rc;
    hipLaunchKernelGGL((norm_gate_reduce_kernel<T>), dim3((unsigned)((cols + kRedCols - 1) / kRedCols)),
                       dim3(kRedCols * kRedGroups), 0, st, part, (int)grid.x, (int)cols, static_cast<T*>(dweight),
                       static_cast<T*>(dbias));
    return (int)hipGetLastError();
}
#undef LA_NG_DISPATCH_FWD
#undef LA_NG_DISPATCH_BWD
#undef LA_NG_BWD
#undef LA_NG_GO

static int ng_check(int64_t rows, int64_t cols, int dtype) {
    if (rows < 0 || cols <= 0 || rows > 0x7fffffffLL) return LA_E_SHAPE;
    if (dtype != LA_BF16 && dtype != LA_FP16 && dtype != LA_FP32) return LA_E_UNSUPPORTED;
    return norm_gate_supported(cols, dtype) ? LA_OK : LA_E_UNSUPPORTED;
}

}  // namespace la

// Makes the runtime load this file's code object now (it otherwise does at the first launch from it).
namespace la {
int prepare_norm_gate() {
    hipFuncAttributes attr;
    return (int)hipFuncGetAttributes(&attr, reinterpret_cast<const void*>(&norm_gate_reduce_kernel<float>));
}
}  // namespace la

extern "C" int norm_gate_supported(int64_t cols, int dtype) {
    if (dtype != LA_BF16 && dtype != LA_FP16 && dtype != LA_FP32) return 0;
    const int64_t e = dtype == LA_FP32 ? 4 : 8;
    return cols > 0 && cols % e == 0 && cols / e <= 1024;
}

extern "C" size_t norm_gate_workspace_bytes(int64_t rows, int64_t cols, int dtype) {
    if (rows <= 0 || !norm_gate_supported(cols, dtype)) return 0;
    return la::ng_part_bytes(rows, cols, dtype == LA_FP32 ? 4 : 2, true);
}

extern "C" int norm_gate_fwd(const void* o, const void* g, const void* weight, const void* bias, void* y, float* mean,
                             float* rstd, int64_t rows, int64_t cols, float eps, int dtype, void* stream) {
    int rc = la::ng_check(rows, cols, dtype);
    if (rc != LA_OK) return rc;
    if (rows == 0) return LA_OK;
    if (!o || !g || !weight || !bias || !y || !mean || !rstd) return LA_E_NULLPTR;
    for (const void* p : {o, g, weight, bias, (const void*)y})
        if (!la::aligned16(p)) return LA_E_ALIGN;
    hipStream_t st = static_cast<hipStream_t>(stream);
    switch (dtype) {
        case LA_BF16: return la::ng_fwd<__bf16>(o, g, weight, bias, y, mean, rstd, rows, cols, eps, st);
        case LA_FP16: return la::ng_fwd<_Float16>(o, g, weight, bias, y, mean, rstd, rows, cols, eps, st);
        default: return la::ng_fwd<float>(o, g, weight, bias, y, mean, rstd, rows, cols, eps, st);
    }
}

extern "C" int norm_gate_bwd(const void* o, const void* g, const void* weight, const void* bias, const float* mean,
                             const float* rstd, const void* dy, void* d_o, void* d_g, void* dweight, void* dbias,
                             void* workspace, size_t ws_bytes, int64_t rows, int64_t cols, int dtype, void* stream) {
    int rc = la::ng_check(rows, cols, dtype);
    if (rc != LA_OK) return rc;
    if (!dweight || !dbias) return LA_E_NULLPTR;
    hipStream_t st = static_cast<hipStream_t>(stream);
    if (rows == 0) {
        // no rows: the column sums are zero (the reduction over zero partial rows writes them)
        const dim3 grid((unsigned)((cols + la::kRedCols - 1) / la::kRedCols)), block(la::kRedCols * la::kRedGroups);
        if (dtype == LA_BF16) hipLaunchKernelGGL((la::norm_gate_reduce_kernel<__bf16>), grid, block, 0, st, nullptr, 0, (int)cols, static_cast<__bf16*>(dweight), static_cast<__bf16*>(dbias));
        else if (dtype == LA_FP16) hipLaunchKernelGGL((la::norm_gate_reduce_kernel<_Float16>), grid, block, 0, st, nullptr, 0, (int)cols, static_cast<_Float16*>(dweight), static_cast<_Float16*>(dbias));
        else hipLaunchKernelGGL((la::norm_gate_reduce_kernel<float>), grid, block, 0, st, nullptr, 0, (int)cols, static_cast<float*>(dweight), static_cast<float*>(dbias));
        return (int)hipGetLastError();
    }
    if (!o || !g || !weight || !bias || !mean || !rstd || !dy || !d_o || !d_g) return LA_E_NULLPTR;
    for (const void* p : {o, g, weight, bias, dy, (const void*)d_o, (const void*)d_g})
        if (!la::aligned16(p)) return LA_E_ALIGN;
    if (!workspace || ws_bytes < la::ng_part_bytes(rows, cols, dtype == LA_FP32 ? 4 : 2, false) || (reinterpret_cast<uintptr_t>(workspace) & 3u))
        return LA_E_WORKSPACE;
    float* part = static_cast<float*>(workspace);
    switch (dtype) {
        case LA_BF16: return la::ng_bwd<__bf16>(o, g, weight, bias, mean, rstd, dy, d_o, d_g, dweight, dbias, part, rows, cols, st);
        case LA_FP16: return la::ng_bwd<_Float16>(o, g, weight, bias, mean, rstd, dy, d_o, d_g, dweight, dbias, part, rows, cols, st);
        default: return la::ng_bwd<float>(o, g, weight, bias, mean, rstd, dy, d_o, d_g, dweight, dbias, part, rows, cols, st);
    }
}
