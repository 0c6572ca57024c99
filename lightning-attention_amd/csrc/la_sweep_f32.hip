// float32 variant of the sweep (see la_sweep.hip for the algorithm): the same
// block recurrence and work split, with every product on the fp32 matrix
// instruction v_mfma_f32_16x16x4_f32 (one A and one B element per lane:
// row/column = lane % 16, contraction slot = lane / 16).  Nothing is rounded
// below float32, so the result is within float32 accumulation error of the
// exact value.  This is the accuracy path, not the throughput path.
//
// Every operand but z comes out of LDS in 16-byte reads.  A contraction may visit its index in any
// order as long as both operands agree, and the rows of a state tile may stand for any 16 features
// as long as the products that write and read the state agree:
//   scores        step (kt, v) of slot g contracts feature 16kt + 4g + v: x and y rows read 4 floats at a time;
//   state tiles   come in groups of four (kt = 4K + q); row rho of tile kt is feature
//                 64K + 4 pi(rho) + q with pi(rho) = 4 (rho % 4) + rho / 4, so that one 16-byte read of a
//                 y row (state update) or an x row (inter-block term) feeds the four tiles of a group.
//
// What bounds it: the fp32 matrix instruction (32 cycles each, 256 FLOP per cycle and CU).  A block costs the busiest
// wave 48 of them for its score tiles, 64 + 40 for the output and 64 for the state (feature dim 64): 2.9 us at 2.4 GHz,
// measured 4.2 (4.8 before fragments were requested a step ahead of their use and the global accesses went through
// bounds-checked buffers without branches; 5.4 with four score tiles on the last wave).  Few sequences: the walk is cut
// into chunks, whose warm-up blocks cost 1.5 us (0.9 for the matrix instructions) with their tiles double-buffered.
// b1 h8 n1024 d64: forward 49.5 -> 30.8 us, backward 53 -> 36; b4 h32 n2048 d128: 325 -> 259 and 984 -> 764.
#include "la_sweep_common.h"
#include "lightning_attn_hip.h"

namespace la {

#ifndef LA_F32_XPAD
#define LA_F32_XPAD 8  // floats of padding per x / y row
#endif

struct SweepArgsF32 {
    const float* x;
    const float* y;
    const float* z;
    float* out;
    const float* s;
    int64_t n;
    int dk, dv, h, bh, nslice;
    // sequence chunks (few sequences): the workgroup of chunk c produces the blocks chunk_start[c] ..
    // chunk_start[c + 1] - 1 of the walk, after running over the blocks before them with the state
    // update alone (no workspace, same results bit for bit)
    int nchunk;
    int chunk_start[9];
};


__device__ __forceinline__ f32x4 mma4(float a, float b, f32x4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
}

// `bid`: number of the workgroup within its part of the launch.
template <int DKP, bool REVERSE, bool DECAY>
__device__ __forceinline__ void sweep_f32_body(const SweepArgsF32& a, const unsigned bid) {
    constexpr int XS = DKP + LA_F32_XPAD;  // row stride (floats) of the x / y tiles
    constexpr int ZS = 64 + 4;    // row stride of the z slice and the P tile
    constexpr int KT = DKP / 16;  // 16-row state tiles
    constexpr int KG = DKP / 64;  // groups of four state tiles
    constexpr int XC = DKP / 16;  // 16-byte chunks per thread for an x / y tile
    extern __shared__ __align__(16) unsigned char smem[];
    float* Xs = reinterpret_cast<float*>(smem);
    float* Ys = Xs + 64 * XS;
    float* Zs = Ys + 64 * XS;
    float* Ps = Zs + 64 * ZS;

    const int xcd = bid & 7, local = bid >> 3;
    const int per_unit = a.nslice * a.nchunk;
    const int unit = xcd + 8 * (local / per_unit);
    const int slice = (local % per_unit) % a.nslice;
    const int chunk = (local % per_unit) / a.nslice;
    if (unit >= a.bh) return;

    const int tid = threadIdx.x;
    const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int lane = tid & 63, r = lane & 15, g = lane >> 4;
    const int64_t n = a.n;
    const int dk = a.dk, dv = a.dv;
    const float* xg = a.x + (int64_t)unit * n * dk;
    const float* yg = a.y + (int64_t)unit * n * dk;
    const float* zg = a.z + (int64_t)unit * n * dv;
    float* og = a.out + (int64_t)unit * n * dv;
    const int col0 = slice * 64;
    const bool wave_active = (col0 + 16 * w) < dv;

    float rate = 0.f;
    if (DECAY) rate = a.s[unit % a.h];

    // the 16 x 16 score tiles of this wave (at most three: 48 instead of 64 matrix instructions for the busiest wave)
    TileDeal deal = kDeal[w];
    if (REVERSE) {
        deal.itA = 3 - deal.itA; deal.jt0 = 3 - deal.jt0;
        if (deal.itB >= 0) { deal.itB = 3 - deal.itB; deal.jt1 = 3 - deal.jt1; deal.jt2 = 3 - deal.jt2; }
    }
    const int itA = __builtin_amdgcn_readfirstlane(deal.itA), jt0 = __builtin_amdgcn_readfirstlane(deal.jt0);
    const int itB = __builtin_amdgcn_readfirstlane(deal.itB), jt1 = __builtin_amdgcn_readfirstlane(deal.jt1);
    const int jt2 = __builtin_amdgcn_readfirstlane(deal.jt2);
    float dfac[3][4], ofac[4], zfac[4][4], lamB = 1.f;
    {
        const int its[3] = {itA, itB, itB}, jts[3] = {jt0, jt1, jt2};
#pragma unroll
        for (int sl = 0; sl < 3; ++sl)
#pragma unroll
            for (int v = 0; v < 4; ++v) {
                const int i = 16 * its[sl] + r, j = 16 * jts[sl] + 4 * g + v;
                const int diff = REVERSE ? (j - i) : (i - j);
                dfac[sl][v] = diff >= 0 ? (DECAY ? expf(-rate * (float)diff) : 1.f) : 0.f;
            }
    }
#pragma unroll
    for (int jt = 0; jt < 4; ++jt)
#pragma unroll
        for (int v = 0; v < 4; ++v) {
            const int j = 16 * jt + 4 * g + v;
            zfac[jt][v] = DECAY ? expf(-rate * (float)(REVERSE ? j : 64 - j)) : 1.f;
        }
#pragma unroll
    for (int it = 0; it < 4; ++it) {
        const int i = 16 * it + r;
        ofac[it] = DECAY ? expf(-rate * (float)(REVERSE ? 64 - i : i)) : 1.f;
    }
    if (DECAY) lamB = expf(-rate * 64.f);

    f32x4 st[KT];
#pragma unroll
    for (int kt = 0; kt < KT; ++kt) st[kt] = (f32x4){0.f, 0.f, 0.f, 0.f};

    const int64_t nblk = (n + 63) / 64;
    const int64_t it_first = a.chunk_start[chunk], it_end = a.chunk_start[chunk + 1];
    u32x4 xr[XC], yr[XC], zr[4];

    // Block number `it` of the walk; x is not needed for a warm-up block.  One bounds-checked buffer per tensor and
    // block (tokens beyond n and features beyond dk / dv read as zero): no branches, and 32-bit offsets however long
    // the sequence.
    const int lrow = tid / (DKP / 4), lcol = (tid % (DKP / 4)) * 4;
    const int zrow = tid / 16, zcol = col0 + (tid % 16) * 4;
    const unsigned xoff = lcol < dk ? (unsigned)(lrow * dk + lcol) * 4u : kOob;
    const unsigned zoff = zcol < dv ? (unsigned)(zrow * dv + zcol) * 4u : kOob;
    auto load_block = [&](int64_t it) {
        const int64_t tok0 = (REVERSE ? nblk - 1 - it : it) * 64;
        const unsigned rows = (unsigned)min((int64_t)64, n - tok0);
        const __amdgpu_buffer_rsrc_t xb = make_rsrc(xg + tok0 * dk, it >= it_first ? rows * dk * 4u : 0u);
        const __amdgpu_buffer_rsrc_t yb = make_rsrc(yg + tok0 * dk, rows * dk * 4u);
        const __amdgpu_buffer_rsrc_t zb = make_rsrc(zg + tok0 * dv, rows * dv * 4u);
#pragma unroll
        for (int u = 0; u < XC; ++u) {
            const unsigned off = xoff + (unsigned)(u * (1024 / DKP) * dk) * 4u;
            xr[u] = buf_load16(xb, off);
            yr[u] = buf_load16(yb, off);
        }
#pragma unroll
        for (int u = 0; u < 4; ++u) zr[u] = buf_load16(zb, zoff + (unsigned)(u * 16 * dv) * 4u);
    };
    auto stage_x = [&]() {
#pragma unroll
        for (int u = 0; u < XC; ++u) {
            const int c = tid + 256 * u;
            const int row = c / (DKP / 4), col = (c % (DKP / 4)) * 4;
            *reinterpret_cast<u32x4*>(Xs + row * XS + col) = xr[u];
        }
    };
    auto stage_yz = [&](float* Y, float* Z) {
#pragma unroll
        for (int u = 0; u < XC; ++u) {
            const int c = tid + 256 * u;
            const int row = c / (DKP / 4), col = (c % (DKP / 4)) * 4;
            *reinterpret_cast<u32x4*>(Y + row * XS + col) = yr[u];
        }
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            const int c = tid + 256 * u;
            const int row = c / 16, col = (c % 16) * 4;
            *reinterpret_cast<u32x4*>(Z + row * ZS + col) = zr[u];
        }
    };
    // z[j][16w + r] for the 16 tokens j = 16jt + 4g + v this lane contracts over
    float zf[4][4];
    auto read_z = [&](const float* Z) {
#pragma unroll
        for (int jt = 0; jt < 4; ++jt)
#pragma unroll
            for (int v = 0; v < 4; ++v) zf[jt][v] = Z[(16 * jt + 4 * g + v) * ZS + 16 * w + r];
    };
    // state = lam^64 state + y^T (z * Lupd); row r of tile 4K + q is feature 64K + 16 (r % 4) + 4 (r / 4) + q
    auto update = [&](const float* Y) {
        // fragments requested eight at a time, one batch ahead of their use
        f32x4 ay[2][8];
        auto fetch = [&](int bt) {
#pragma unroll
            for (int i = 0; i < 8; ++i) {
                const int K = bt / 2, jt = 2 * (bt % 2) + i / 4, v = i % 4;
                ay[bt % 2][i] = *reinterpret_cast<const f32x4*>(Y + (16 * jt + 4 * g + v) * XS + 64 * K + 16 * (r & 3) + 4 * (r >> 2));
            }
            __builtin_amdgcn_sched_barrier(0);
        };
        fetch(0);
        if (DECAY) {
#pragma unroll
            for (int jt = 0; jt < 4; ++jt)
#pragma unroll
                for (int v = 0; v < 4; ++v) zf[jt][v] *= zfac[jt][v];
#pragma unroll
            for (int kt = 0; kt < KT; ++kt)
#pragma unroll
                for (int v = 0; v < 4; ++v) st[kt][v] *= lamB;
        }
#pragma unroll
        for (int bt = 0; bt < 2 * KG; ++bt) {
            if (bt + 1 < 2 * KG) fetch(bt + 1);
#pragma unroll
            for (int i = 0; i < 8; ++i)
#pragma unroll
                for (int q = 0; q < 4; ++q)
                    st[4 * (bt / 2) + q] = mma4(ay[bt % 2][i][q], zf[2 * (bt % 2) + i / 4][i % 4], st[4 * (bt / 2) + q]);
            __builtin_amdgcn_sched_barrier(0);
        }
    };

    // Warm-up: the blocks before the chunk, state update alone.  They need neither the x nor the P tile, whose LDS
    // serves as the second y / z buffer: one barrier per block, the next block staged and the one after it requested
    // from memory while this one is worked on.
    load_block(0);
    if (it_first > 0) {
        stage_yz(Ys, Zs);
        load_block(1);
        for (int64_t it = 0; it < it_first; ++it) {
            const bool odd = (it & 1) != 0;
            __syncthreads();
            if (wave_active) {
                read_z(odd ? Ps : Zs);
                update(odd ? Xs : Ys);
            }
            if (it + 1 < it_first) {
                stage_yz(odd ? Ys : Xs, odd ? Zs : Ps);
                load_block(it + 2);
            }
        }
        __syncthreads();
    }
    // (tiles of P on the masked side of the diagonal are never written)
    for (int c = tid; c < 64 * ZS / 4; c += 256) reinterpret_cast<uint4*>(Ps)[c] = make_uint4(0, 0, 0, 0);
    stage_x();
    stage_yz(Ys, Zs);
    __syncthreads();

    for (int64_t it = it_first; it < it_end; ++it) {
        const bool have_next = it + 1 < it_end;
        if (have_next) load_block(it + 1);

        // 1. S^T tiles -> masked, decayed P[i][j]
        auto frag = [&](const float* tile, int row16, int kt) { return *reinterpret_cast<const f32x4*>(tile + (16 * row16 + r) * XS + 16 * kt + 4 * g); };
        auto put_p = [&](int sl, int i16, int j16, const f32x4& acc) {
            f32x4 p;
#pragma unroll
            for (int v = 0; v < 4; ++v) p[v] = acc[v] * dfac[sl][v];
            *reinterpret_cast<f32x4*>(Ps + (16 * i16 + r) * ZS + 16 * j16 + 4 * g) = p;
        };
        f32x4 s0 = (f32x4){0.f, 0.f, 0.f, 0.f}, s1 = s0, s2 = s0;
        if (itB >= 0) {
            f32x4 xa[2], xb[2], y0[2], y1[2], y2[2];
            auto fetch = [&](int kt) {
                xa[kt % 2] = frag(Xs, itA, kt);
                y0[kt % 2] = frag(Ys, jt0, kt);
                xb[kt % 2] = frag(Xs, itB, kt);
                y1[kt % 2] = frag(Ys, jt1, kt);
                y2[kt % 2] = frag(Ys, jt2, kt);
                __builtin_amdgcn_sched_barrier(0);
            };
            fetch(0);
#pragma unroll
            for (int kt = 0; kt < KT; ++kt) {
                if (kt + 1 < KT) fetch(kt + 1);
#pragma unroll
                for (int v = 0; v < 4; ++v) {
                    s0 = mma4(y0[kt % 2][v], xa[kt % 2][v], s0);
                    s1 = mma4(y1[kt % 2][v], xb[kt % 2][v], s1);
                    s2 = mma4(y2[kt % 2][v], xb[kt % 2][v], s2);
                }
                __builtin_amdgcn_sched_barrier(0);
            }
            put_p(1, itB, jt1, s1);
            put_p(2, itB, jt2, s2);
        } else {
#pragma unroll
            for (int kt = 0; kt < KT; ++kt) {
                const f32x4 xa = frag(Xs, itA, kt), y0 = frag(Ys, jt0, kt);
#pragma unroll
                for (int v = 0; v < 4; ++v) s0 = mma4(y0[v], xa[v], s0);
            }
        }
        put_p(0, itA, jt0, s0);
        __syncthreads();

        if (wave_active) {
            f32x4 oacc[4];
#pragma unroll
            for (int i4 = 0; i4 < 4; ++i4) oacc[i4] = (f32x4){0.f, 0.f, 0.f, 0.f};
            // 2a. inter-block: st[4K + q][v] holds row 4g + v of its tile, feature 64K + 16v + 4g + q.  Here and in 2b the
            // fragments are requested one step ahead of their use (left to itself the scheduler sinks every read to
            // its first use, and the wave pays an LDS round trip per step).
            f32x4 bx[2][4], bp[2][4];
            auto fetch_x = [&](int step) {
#pragma unroll
                for (int i4 = 0; i4 < 4; ++i4) bx[step % 2][i4] = *reinterpret_cast<const f32x4*>(Xs + (16 * i4 + r) * XS + 16 * step + 4 * g);
                __builtin_amdgcn_sched_barrier(0);
            };
            auto fetch_p = [&](int jt) {
#pragma unroll
                for (int i4 = 0; i4 < 4; ++i4) {
                    const bool need = REVERSE ? (jt >= i4) : (jt <= i4);
                    if (need) bp[jt % 2][i4] = *reinterpret_cast<const f32x4*>(Ps + (16 * i4 + r) * ZS + 16 * jt + 4 * g);
                }
                __builtin_amdgcn_sched_barrier(0);
            };
            fetch_x(0);
#pragma unroll
            for (int step = 0; step < 4 * KG; ++step) {
                if (step + 1 < 4 * KG) fetch_x(step + 1);
                else {
                    read_z(Zs);
                    fetch_p(0);
                }
#pragma unroll
                for (int q = 0; q < 4; ++q)
#pragma unroll
                    for (int i4 = 0; i4 < 4; ++i4) oacc[i4] = mma4(st[4 * (step / 4) + q][step % 4], bx[step % 2][i4][q], oacc[i4]);
                __builtin_amdgcn_sched_barrier(0);
            }
            if (DECAY) {
#pragma unroll
                for (int i4 = 0; i4 < 4; ++i4)
#pragma unroll
                    for (int v = 0; v < 4; ++v) oacc[i4][v] *= ofac[i4];
            }
            // 2b. intra-block: slot g of step (jt, v) is token 16jt + 4g + v
#pragma unroll
            for (int jt = 0; jt < 4; ++jt) {
                if (jt + 1 < 4) fetch_p(jt + 1);
#pragma unroll
                for (int v = 0; v < 4; ++v)
#pragma unroll
                    for (int i4 = 0; i4 < 4; ++i4) {
                        const bool need = REVERSE ? (jt >= i4) : (jt <= i4);
                        if (need) oacc[i4] = mma4(zf[jt][v], bp[jt % 2][i4][v], oacc[i4]);
                    }
                __builtin_amdgcn_sched_barrier(0);
            }
            const int64_t tok0 = (REVERSE ? nblk - 1 - it : it) * 64;
            const __amdgpu_buffer_rsrc_t ob = make_rsrc(og + tok0 * dv, (unsigned)min((int64_t)64, n - tok0) * dv * 4u);
            const int col = col0 + 16 * w + 4 * g;
            const unsigned ooff = col < dv ? (unsigned)(r * dv + col) * 4u : kOob;
#pragma unroll
            for (int i4 = 0; i4 < 4; ++i4) buf_store16(ob, ooff + (unsigned)(16 * i4 * dv) * 4u, 0u, __builtin_bit_cast(u32x4, oacc[i4]));
            if (have_next) update(Ys);
        }
        __syncthreads();
        if (have_next) {
            stage_x();
            stage_yz(Ys, Zs);
            __syncthreads();
        }
    }
}

// (70 KB of LDS at DKP = 64: two workgroups fit a CU when the registers do, which the second bound asks for)
template <int DKP, bool REVERSE, bool DECAY>
__global__ __launch_bounds__(256, DKP <= 64 ? 2 : 1) void la_sweep_f32_kernel(SweepArgsF32 a) {
    sweep_f32_body<DKP, REVERSE, DECAY>(a, blockIdx.x);
}

// The three sweeps of a backward pass with d == e in one launch: part 0 walks forward (dQ), parts 1 and 2
// backward (dK, dV); the parts have the same number of workgroups (a multiple of 8).
struct SweepTrioF32 {
    SweepArgsF32 a[3];
    unsigned per_part;
};
template <int DKP, bool DECAY>
__global__ __launch_bounds__(256, DKP <= 64 ? 2 : 1) void la_sweep_f32_trio_kernel(SweepTrioF32 t) {
    const unsigned part = blockIdx.x / t.per_part, bid = blockIdx.x % t.per_part;
    if (part == 0) sweep_f32_body<DKP, false, DECAY>(t.a[0], bid);
    else sweep_f32_body<DKP, true, DECAY>(t.a[part == 1 ? 1 : 2], bid);
}

template <int DKP, bool DECAY>
static int prep_trio_f32() {
    constexpr size_t lds = (size_t)(2 * 64 * (DKP + LA_F32_XPAD) + 2 * 64 * 68) * sizeof(float);
    static unsigned char lds_allowed[kMaxDevices];
    return allow_lds(la_sweep_f32_trio_kernel<DKP, DECAY>, lds, lds_allowed);
}
template <int DKP, bool REVERSE, bool DECAY>
static int prep_one_f32() {
    constexpr size_t lds = (size_t)(2 * 64 * (DKP + LA_F32_XPAD) + 2 * 64 * 68) * sizeof(float);
    static unsigned char lds_allowed[kMaxDevices];
    return allow_lds(la_sweep_f32_kernel<DKP, REVERSE, DECAY>, lds, lds_allowed);
}
// Every instantiation of this file made ready for its first launch on the current device.
int prepare_f32() {
    int e = 0;
#define LA_P(DKP, D) \
    if (!e) e = prep_trio_f32<DKP, D>(); \
    if (!e) e = prep_one_f32<DKP, false, D>(); \
    if (!e) e = prep_one_f32<DKP, true, D>();
    LA_P(64, false) LA_P(64, true) LA_P(128, false) LA_P(128, true)
#undef LA_P
    return e;
}

template <int DKP, bool DECAY>
static int launch_trio_f32(const SweepTrioF32& t, hipStream_t st) {
    constexpr size_t lds = (size_t)(2 * 64 * (DKP + LA_F32_XPAD) + 2 * 64 * 68) * sizeof(float);
    auto kern = la_sweep_f32_trio_kernel<DKP, DECAY>;
    if (const int e = prep_trio_f32<DKP, DECAY>()) return e;
    hipLaunchKernelGGL(kern, dim3(3 * t.per_part), dim3(256), lds, st, t);
    return (int)hipGetLastError();
}

template <int DKP, bool REVERSE, bool DECAY>
static int launch_one_f32(const SweepArgsF32& a, hipStream_t st) {
    constexpr size_t lds = (size_t)(2 * 64 * (DKP + LA_F32_XPAD) + 2 * 64 * 68) * sizeof(float);
    auto kern = la_sweep_f32_kernel<DKP, REVERSE, DECAY>;
    if (const int e = prep_one_f32<DKP, REVERSE, DECAY>()) return e;
    const int units8 = (a.bh + 7) / 8 * 8;
    hipLaunchKernelGGL(kern, dim3((unsigned)(units8 * a.nslice * a.nchunk)), dim3(256), lds, st, a);
    return (int)hipGetLastError();
}

template <bool REVERSE>
static int launch_dir_f32(const SweepArgsF32& a, hipStream_t st) {
    const bool decay = a.s != nullptr;
#define LA_GO(DKP) (decay ? launch_one_f32<DKP, REVERSE, true>(a, st) : launch_one_f32<DKP, REVERSE, false>(a, st))
    if (a.dk <= 64) return LA_GO(64);
    return LA_GO(128);
#undef LA_GO
}

static SweepArgsF32 make_args_f32(const void* x, const void* y, const void* z, void* out, const float* s, int64_t bh, int64_t h,
                                  int64_t n, int64_t dk, int64_t dv) {
    SweepArgsF32 a;
    a.x = static_cast<const float*>(x); a.y = static_cast<const float*>(y); a.z = static_cast<const float*>(z);
    a.out = static_cast<float*>(out); a.s = s;
    a.n = n; a.dk = (int)dk; a.dv = (int)dv; a.h = (int)h; a.bh = (int)bh;
    a.nslice = (int)((dv + 63) / 64);
    a.nchunk = 1;
    for (int i = 0; i < 9; ++i) a.chunk_start[i] = i == 0 ? 0 : (int)((n + 63) / 64);
    return a;
}

// What a warm-up block costs of a full one (1.5 of 4.2 us), and the fewest blocks a chunk is worth cutting off for.
// b1 h8 d64 forward, us, by number of chunks 1 / 2 / 4 / 8: n = 1024 69.9 / 44.7 / 33.7 / 30.9, n = 4096 268 / 169 / 123 /
// 108: as many as there are CUs for, down to two blocks each.
static const double kWarmCost = 0.36;
static const int64_t kMinBlocks = 2;

int sweep_f32(const void* x, const void* y, const void* z, void* out, const float* s, int64_t bh, int64_t h,
              int64_t n, int64_t dk, int64_t dv, bool reverse, int chunks, hipStream_t st) {
    if (dk > 128) return LA_E_UNSUPPORTED;
    SweepArgsF32 a = make_args_f32(x, y, z, out, s, bh, h, n, dk, dv);
    plan_warm_up_chunks(num_cus(), (bh + 7) / 8 * 8 * a.nslice, (n + 63) / 64, chunks, &a.nchunk, a.chunk_start, kWarmCost, kMinBlocks);
    return reverse ? launch_dir_f32<true>(a, st) : launch_dir_f32<false>(a, st);
}

// float32 backward pass with d == e: dQ = fwd(dO, v, k), dK = rev(v, dO, q), dV = rev(k, q, dO) in one
// launch (the sweeps are independent; with few sequences they run side by side).
int sweep_f32_bwd_once(const void* q, const void* k, const void* v, const void* dout, void* dq, void* dk, void* dv,
                       const float* s, int64_t bh, int64_t h, int64_t n, int64_t d, int chunks, hipStream_t st) {
    if (d > 128) return LA_E_UNSUPPORTED;
    SweepTrioF32 t;
    t.a[0] = make_args_f32(dout, v, k, dq, s, bh, h, n, d, d);
    t.a[1] = make_args_f32(v, dout, q, dk, s, bh, h, n, d, d);
    t.a[2] = make_args_f32(k, q, dout, dv, s, bh, h, n, d, d);
    plan_warm_up_chunks(num_cus(), (bh + 7) / 8 * 8 * t.a[0].nslice * 3, (n + 63) / 64, chunks, &t.a[0].nchunk, t.a[0].chunk_start, kWarmCost, kMinBlocks);
    for (int i = 1; i < 3; ++i) {
        t.a[i].nchunk = t.a[0].nchunk;
        for (int j = 0; j < 9; ++j) t.a[i].chunk_start[j] = t.a[0].chunk_start[j];
    }
    t.per_part = (unsigned)((bh + 7) / 8 * 8 * t.a[0].nslice * t.a[0].nchunk);
    const bool decay = s != nullptr;
    if (d <= 64) return decay ? launch_trio_f32<64, true>(t, st) : launch_trio_f32<64, false>(t, st);
    return decay ? launch_trio_f32<128, true>(t, st) : launch_trio_f32<128, false>(t, st);
}

}  // namespace la
