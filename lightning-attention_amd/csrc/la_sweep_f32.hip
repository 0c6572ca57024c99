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
// What bounds it: the fp32 matrix instruction (32 cycles each, 256 FLOP per cycle and CU).  A block of feature dim 64 and 64
// columns costs the busiest of four wavefronts 48 of them for its score tiles, 64 + 40 for the output and 64 for the state: 2.9 us
// at 2.4 GHz, measured 4.1 with half of the CUs at work, 4.5 with a workgroup on each and 8.0 for two on each (105 of the 154 TFLOP/s that
// a large product reaches: forward of 512 sequences, n1536, 200 us).  Feature dim 128 leaves room in LDS for one
// workgroup only: there two wavefronts share a slab of columns, each with half of the features, so that a SIMD has a second
// one to issue from (b4 h32 n2048: forward 264 -> 230 us, backward 767 -> 668).  Few sequences: 32 columns to a workgroup, the
// halves of the features on a wavefront each (a block 3.05 us, 5.0 at feature dim 128), and the walk cut into chunks whose
// warm-up blocks are fetched from memory in fragment layout, 0.75 us each (1.5 through LDS, a barrier a block).
// Forward + backward, us: b1 h8 d64 n1024 30.7 + 31.9 -> 20.7 + 24.8, n4096 109 + 112 -> 63 + 73; b1 h4 n8192 d128 394 + 428 -> 199 + 327.
#include <type_traits>

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

// The score tiles of eight waves: at most two each, ten to four SIMDs (waves w and w + 4 share one).
__device__ __constant__ const TileDeal kDeal8[8] = {
    {3, 0, 2, 0, -1}, {3, 1, 2, 1, -1}, {3, 2, -1, -1, -1}, {3, 3, -1, -1, -1},
    {2, 2, -1, -1, -1}, {1, 0, -1, -1, -1}, {1, 1, -1, -1, -1}, {0, 0, -1, -1, -1},
};

// How a workgroup is cut up: WC slabs of 16 columns of z / out, times KH parts of the feature dim.  A wavefront (slab, part)
// owns that part of the state under its slab; with KH = 2 the two wavefronts of a slab each sum half of the output
// (half of the features of the inter-block term, half of the tokens of the intra-block one), hand each other half of the
// 64 rows through LDS and write the rest.
template <int DKP, int WC, int KH>
struct F32Form {
    static_assert(KH == 1 || KH == 2, "one or two parts of the feature dim");
    static constexpr int NW = WC * KH, NT = 64 * NW;  // wavefronts, threads
    static constexpr int XS = DKP + LA_F32_XPAD;      // row stride (floats) of the x / y tiles
    static constexpr int ZC = 16 * WC;                // columns of z / out
    static constexpr int ZS = ZC + 4;                 // row stride of the z slice
    static constexpr int PS = 64 + 4;                 // row stride of the P tile
    static constexpr int EX = KH == 2 ? NW * 512 : 0; // floats handed over: two 16 x 16 tiles a wavefront
    static constexpr size_t lds = (size_t)(2 * 64 * XS + 64 * ZS + 64 * PS + EX) * sizeof(float);
    static constexpr int per_cu = lds <= 80 * 1024 ? 2 : 1;  // workgroups that fit a CU's LDS
};

// `bid`: number of the workgroup within its part of the launch.
template <int DKP, int WC, int KH, bool REVERSE, bool DECAY>
__device__ __forceinline__ void sweep_f32_body(const SweepArgsF32& a, const unsigned bid) {
    typedef F32Form<DKP, WC, KH> F;
    constexpr int NT = F::NT, XS = F::XS, ZS = F::ZS, PS = F::PS;
    constexpr int KT = DKP / 16 / KH;           // 16-row state tiles of a wavefront
    constexpr int Q = KT < 4 ? KT : 4;          // ... of one group
    constexpr int KG = KT / Q;                  // groups of a wavefront
    constexpr int XC = 16 * DKP / NT;           // 16-byte chunks per thread for an x / y tile
    constexpr int ZN = 16 * F::ZC / NT;         // ... and for the z slice
    constexpr int SL = F::NW == 8 ? 2 : 3;      // score tiles of a wavefront, at most
    typedef float fq __attribute__((__vector_size__(Q * sizeof(float))));
    extern __shared__ __align__(16) unsigned char smem[];
    float* Xs = reinterpret_cast<float*>(smem);
    float* Ys = Xs + 64 * XS;
    float* Zs = Ys + 64 * XS;
    float* Ps = Zs + 64 * ZS;
    float* Es = Ps + 64 * PS;

    const int xcd = bid & 7, local = bid >> 3;
    const int per_unit = a.nslice * a.nchunk;
    const int unit = xcd + 8 * (local / per_unit);
    const int slice = (local % per_unit) % a.nslice;
    const int chunk = (local % per_unit) / a.nslice;
    if (unit >= a.bh) return;

    const int tid = threadIdx.x;
    const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int slab = w % WC, part = w / WC;
    const int lane = tid & 63, r = lane & 15, g = lane >> 4;
    const int64_t n = a.n;
    const int dk = a.dk, dv = a.dv;
    const float* xg = a.x + (int64_t)unit * n * dk;
    const float* yg = a.y + (int64_t)unit * n * dk;
    const float* zg = a.z + (int64_t)unit * n * dv;
    float* og = a.out + (int64_t)unit * n * dv;
    const int col0 = slice * F::ZC;
    const bool wave_active = (col0 + 16 * slab) < dv;
    const int f0 = 16 * KT * part;  // first feature of this wavefront's part

    float rate = 0.f;
    if (DECAY) rate = a.s[unit % a.h];

    // the 16 x 16 score tiles of this wave (at most three: 48 instead of 64 matrix instructions for the busiest wave)
    TileDeal deal = F::NW == 8 ? kDeal8[w] : kDeal[w & 3];
    if (REVERSE) {
        deal.itA = 3 - deal.itA; deal.jt0 = 3 - deal.jt0;
        if (deal.itB >= 0) { deal.itB = 3 - deal.itB; deal.jt1 = 3 - deal.jt1; deal.jt2 = 3 - deal.jt2; }
    }
    const int itA = __builtin_amdgcn_readfirstlane(deal.itA), jt0 = __builtin_amdgcn_readfirstlane(deal.jt0);
    const int itB = __builtin_amdgcn_readfirstlane(deal.itB), jt1 = __builtin_amdgcn_readfirstlane(deal.jt1);
    const int jt2 = __builtin_amdgcn_readfirstlane(deal.jt2);
    float dfac[SL][4], ofac[4], zfac[4][4], lamB = 1.f;
    {
        const int its[3] = {itA, itB, itB}, jts[3] = {jt0, jt1, jt2};
#pragma unroll
        for (int sl = 0; sl < SL; ++sl)
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
    u32x4 xr[XC], yr[XC], zr[ZN];

    // Block number `it` of the walk.  One bounds-checked buffer per tensor and
    // block (tokens beyond n and features beyond dk / dv read as zero): no branches, and 32-bit offsets however long
    // the sequence.
    const int lrow = tid / (DKP / 4), lcol = (tid % (DKP / 4)) * 4;
    const int zrow = tid / (4 * WC), zcol = col0 + (tid % (4 * WC)) * 4;
    const unsigned xoff = lcol < dk ? (unsigned)(lrow * dk + lcol) * 4u : kOob;
    const unsigned zoff = zcol < dv ? (unsigned)(zrow * dv + zcol) * 4u : kOob;
    auto block_rsrc = [&](const float* base, int cols, int64_t it) {
        const int64_t tok0 = (REVERSE ? nblk - 1 - it : it) * 64;
        return make_rsrc(base + tok0 * cols, (unsigned)min((int64_t)64, n - tok0) * cols * 4u);
    };
    auto load_xy = [&](u32x4 (&to)[XC], const float* base, int64_t it) __attribute__((always_inline)) {
        const __amdgpu_buffer_rsrc_t b = block_rsrc(base, dk, it);
#pragma unroll
        for (int u = 0; u < XC; ++u) to[u] = buf_load16(b, xoff + (unsigned)(u * (NT * 4 / DKP) * dk) * 4u);
    };
    auto load_z = [&](int64_t it) __attribute__((always_inline)) {
        const __amdgpu_buffer_rsrc_t b = block_rsrc(zg, dv, it);
#pragma unroll
        for (int u = 0; u < ZN; ++u) zr[u] = buf_load16(b, zoff + (unsigned)(u * (NT / (4 * WC)) * dv) * 4u);
    };
    auto load_block = [&](int64_t it) __attribute__((always_inline)) {
        load_xy(xr, xg, it);
        load_xy(yr, yg, it);
        load_z(it);
    };
    auto stage = [&]() {
#pragma unroll
        for (int u = 0; u < XC; ++u) {
            const int c = tid + NT * u;
            const int row = c / (DKP / 4), col = (c % (DKP / 4)) * 4;
            *reinterpret_cast<u32x4*>(Xs + row * XS + col) = xr[u];
            *reinterpret_cast<u32x4*>(Ys + row * XS + col) = yr[u];
        }
#pragma unroll
        for (int u = 0; u < ZN; ++u) {
            const int c = tid + NT * u;
            const int row = c / (4 * WC), col = (c % (4 * WC)) * 4;
            *reinterpret_cast<u32x4*>(Zs + row * ZS + col) = zr[u];
        }
    };
    // z[j][16 slab + r] for the 16 tokens j = 16jt + 4g + v this lane contracts over
    float zf[4][4];
    auto read_z = [&]() {
#pragma unroll
        for (int jt = 0; jt < 4; ++jt)
#pragma unroll
            for (int v = 0; v < 4; ++v) zf[jt][v] = Zs[(16 * jt + 4 * g + v) * ZS + 16 * slab + r];
    };
    // state = lam^64 state + y^T (z * Lupd); row r of tile Q K + q is feature f0 + 16 Q K + 4 Q (r % 4) + Q (r / 4) + q
    auto decay_state = [&]() {
        if (DECAY) {
#pragma unroll
            for (int kt = 0; kt < KT; ++kt)
#pragma unroll
                for (int v = 0; v < 4; ++v) st[kt][v] *= lamB;
        }
    };
    const int yfeat = f0 + 4 * Q * (r & 3) + Q * (r >> 2);  // first feature of this lane's fragments of y
    auto update = [&]() {
        // fragments requested eight at a time, one batch ahead of their use
        fq ay[2][8];
        auto fetch = [&](int bt) {
#pragma unroll
            for (int i = 0; i < 8; ++i) {
                const int K = bt / 2, jt = 2 * (bt % 2) + i / 4, v = i % 4;
                ay[bt % 2][i] = *reinterpret_cast<const fq*>(Ys + (16 * jt + 4 * g + v) * XS + yfeat + 16 * Q * K);
            }
            __builtin_amdgcn_sched_barrier(0);
        };
        fetch(0);
        if (DECAY) {
#pragma unroll
            for (int jt = 0; jt < 4; ++jt)
#pragma unroll
                for (int v = 0; v < 4; ++v) zf[jt][v] *= zfac[jt][v];
        }
        decay_state();
#pragma unroll
        for (int bt = 0; bt < 2 * KG; ++bt) {
            if (bt + 1 < 2 * KG) fetch(bt + 1);
#pragma unroll
            for (int i = 0; i < 8; ++i)
#pragma unroll
                for (int q = 0; q < Q; ++q)
                    st[Q * (bt / 2) + q] = mma4(ay[bt % 2][i][q], zf[2 * (bt % 2) + i / 4][i % 4], st[Q * (bt / 2) + q]);
            __builtin_amdgcn_sched_barrier(0);
        }
    };

    // (one part of all the features: the fragments of the warm-up take the registers)
    constexpr bool EARLY = KH == 2;
    if (EARLY || it_first == 0) load_block(it_first);
    // Warm-up: the blocks before the chunk, state update alone.  Here every wavefront fetches its fragments straight from
    // memory: a fragment of y is a whole piece of each of four rows (16 lanes side by side), one of z 64 bytes, so nothing
    // is gained from LDS - and without it there is no barrier between the wavefronts.  Two register sets of WJ 16-token
    // tiles, a block each or half of one where registers are short.
    if (it_first > 0 && wave_active) {
        constexpr int WJ = F::NT * F::per_cu <= 256 || KT == 2 ? 4 : 2;
        fq wy[2][KG][WJ][4];
        float wz[2][WJ][4];
        const int fcol = col0 + 16 * slab + r;
        const unsigned fy = (unsigned)(4 * g * dk + yfeat) * 4u, fz = fcol < dv ? (unsigned)(4 * g * dv + fcol) * 4u : kOob;
        // set S takes its WJ tiles of block `it`: all four, or tokens 32 S .. 32 S + 31
        auto fetch = [&](auto set, int64_t it) __attribute__((always_inline)) {
            constexpr int S = decltype(set)::value, J0 = WJ == 2 ? 2 * S : 0;
            const int64_t tok0 = (REVERSE ? nblk - 1 - it : it) * 64;
            // (a block that is not needed is fetched from an empty buffer: zeros, no memory traffic)
            const unsigned rows = it < it_first ? (unsigned)min((int64_t)64, n - tok0) : 0u;
            const __amdgpu_buffer_rsrc_t yb = make_rsrc(yg + (rows ? tok0 : 0) * dk, rows * dk * 4u);
            const __amdgpu_buffer_rsrc_t zb = make_rsrc(zg + (rows ? tok0 : 0) * dv, rows * dv * 4u);
#pragma unroll
            for (int j = 0; j < WJ; ++j)
#pragma unroll
                for (int v = 0; v < 4; ++v) {
                    const int row = 16 * (J0 + j) + v;
#pragma unroll
                    for (int K = 0; K < KG; ++K) {
                        const unsigned off = yfeat + 16 * Q * K < dk ? fy + (unsigned)(row * dk + 16 * Q * K) * 4u : kOob;
                        if constexpr (Q == 4) wy[S][K][j][v] = __builtin_bit_cast(fq, buf_load16(yb, off));
                        else wy[S][K][j][v] = __builtin_bit_cast(fq, __builtin_amdgcn_raw_buffer_load_b64(yb, off, 0, 0));
                    }
                    wz[S][j][v] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(zb, fz + (unsigned)(row * dv) * 4u, 0, 0));
                }
        };
        auto fold = [&](auto set) __attribute__((always_inline)) {
            constexpr int S = decltype(set)::value, J0 = WJ == 2 ? 2 * S : 0;
            if (J0 == 0) decay_state();
#pragma unroll
            for (int K = 0; K < KG; ++K)
#pragma unroll
                for (int j = 0; j < WJ; ++j)
#pragma unroll
                    for (int v = 0; v < 4; ++v) {
                        const float z = DECAY ? wz[S][j][v] * zfac[J0 + j][v] : wz[S][j][v];
#pragma unroll
                        for (int q = 0; q < Q; ++q) st[Q * K + q] = mma4(wy[S][K][j][v][q], z, st[Q * K + q]);
                    }
        };
        typedef std::integral_constant<int, 0> S0;
        typedef std::integral_constant<int, 1> S1;
        fetch(S0{}, 0);
        fetch(S1{}, WJ == 4 ? 1 : 0);
        for (int64_t it = 0; it < it_first; it += WJ / 2) {
            fold(S0{});
            fetch(S0{}, it + WJ / 2);
            if (WJ == 2 || it + 1 < it_first) {
                fold(S1{});
                fetch(S1{}, it + (WJ == 4 ? 3 : 1));
            }
        }
    }
    if (!EARLY && it_first > 0) load_block(it_first);
    // (tiles of P on the masked side of the diagonal are never written)
    for (int c = tid; c < 64 * PS / 4; c += NT) reinterpret_cast<uint4*>(Ps)[c] = make_uint4(0, 0, 0, 0);
    stage();
    __syncthreads();

    for (int64_t it = it_first; it < it_end; ++it) {
        const bool have_next = it + 1 < it_end;
        // The next block is requested in three parts, spread over this one: all twelve loads at the top hold up the first fragments (us,
        // together / apart: backward of d64 n2048, 96 sequences, 229 / 224, 24 sequences 74.0 / 72.4; forward of 128 sequences of d64 n2048 92.4 /
        // 87.4, n8192 378 / 362; d128 n2048, 64 sequences backward 455 / 446).
        if (have_next) load_xy(xr, xg, it + 1);

        // 1. S^T tiles -> masked, decayed P[i][j]
        auto frag = [&](const float* tile, int row16, int kt) { return *reinterpret_cast<const f32x4*>(tile + (16 * row16 + r) * XS + 16 * kt + 4 * g); };
        auto put_p = [&](int sl, int i16, int j16, const f32x4& acc) {
            f32x4 p;
#pragma unroll
            for (int v = 0; v < 4; ++v) p[v] = acc[v] * dfac[sl][v];
            *reinterpret_cast<f32x4*>(Ps + (16 * i16 + r) * PS + 16 * j16 + 4 * g) = p;
        };
        constexpr int KS = DKP / 16;
        f32x4 s0 = (f32x4){0.f, 0.f, 0.f, 0.f}, s1 = s0, s2 = s0;
        if (itB >= 0) {
            f32x4 xa[2], xb[2], y0[2], y1[2], y2[2];
            auto fetch = [&](int kt) {
                xa[kt % 2] = frag(Xs, itA, kt);
                y0[kt % 2] = frag(Ys, jt0, kt);
                xb[kt % 2] = frag(Xs, itB, kt);
                y1[kt % 2] = frag(Ys, jt1, kt);
                if (SL == 3) y2[kt % 2] = frag(Ys, jt2, kt);
                __builtin_amdgcn_sched_barrier(0);
            };
            fetch(0);
#pragma unroll
            for (int kt = 0; kt < KS; ++kt) {
                if (kt + 1 < KS) fetch(kt + 1);
#pragma unroll
                for (int v = 0; v < 4; ++v) {
                    s0 = mma4(y0[kt % 2][v], xa[kt % 2][v], s0);
                    s1 = mma4(y1[kt % 2][v], xb[kt % 2][v], s1);
                    if (SL == 3) s2 = mma4(y2[kt % 2][v], xb[kt % 2][v], s2);
                }
                __builtin_amdgcn_sched_barrier(0);
            }
            put_p(1, itB, jt1, s1);
            if constexpr (SL == 3) put_p(2, itB, jt2, s2);
        } else {
#pragma unroll
            for (int kt = 0; kt < KS; ++kt) {
                const f32x4 xa = frag(Xs, itA, kt), y0 = frag(Ys, jt0, kt);
#pragma unroll
                for (int v = 0; v < 4; ++v) s0 = mma4(y0[v], xa[v], s0);
            }
        }
        put_p(0, itA, jt0, s0);
        if (have_next) load_z(it + 1);
        __syncthreads();
        if (have_next) load_xy(yr, yg, it + 1);

        f32x4 oacc[4];
        // rows 16 i4 .. 16 i4 + 15 of this wave's slab go to memory
        auto store = [&](auto first, const f32x4 (&o)[4 / KH]) __attribute__((always_inline)) {
            const int64_t tok0 = (REVERSE ? nblk - 1 - it : it) * 64;
            const __amdgpu_buffer_rsrc_t ob = make_rsrc(og + tok0 * dv, (unsigned)min((int64_t)64, n - tok0) * dv * 4u);
            const int col = col0 + 16 * slab + 4 * g;
            const unsigned ooff = col < dv ? (unsigned)(r * dv + col) * 4u : kOob;
#pragma unroll
            for (int i = 0; i < 4 / KH; ++i)
                buf_store16(ob, ooff + (unsigned)(16 * (decltype(first)::value + i) * dv) * 4u, __builtin_bit_cast(u32x4, o[i]));
        };
        if (wave_active) {
#pragma unroll
            for (int i4 = 0; i4 < 4; ++i4) oacc[i4] = (f32x4){0.f, 0.f, 0.f, 0.f};
            // 2a. inter-block: st[Q K + q][v] holds row 4g + v of its tile, feature f0 + 16 Q K + 4 Q v + Q g + q.  Here and in 2b the
            // fragments are requested one step ahead of their use (left to itself the scheduler sinks every read to
            // its first use, and the wave pays an LDS round trip per step).
            fq bx[2][4];
            f32x4 bp[2][4];
            auto fetch_x = [&](int step) {
#pragma unroll
                for (int i4 = 0; i4 < 4; ++i4) bx[step % 2][i4] = *reinterpret_cast<const fq*>(Xs + (16 * i4 + r) * XS + f0 + 4 * Q * step + Q * g);
                __builtin_amdgcn_sched_barrier(0);
            };
            // 2b. intra-block: slot g of step (jt, v) is token 16jt + 4g + v.  KH = 2: tokens 0 .. 15 and 48 .. 63 are one
            // part's, those between the other's (five tiles of P each, whichever way the walk goes).
            auto token_tile = [&](int j) { return KH == 1 ? j : part == 0 ? 3 * j : 1 + j; };
            auto fetch_p = [&](int j) {
                const int jt = token_tile(j);
#pragma unroll
                for (int i4 = 0; i4 < 4; ++i4) {
                    const bool need = KH == 2 || (REVERSE ? (jt >= i4) : (jt <= i4));
                    if (need) bp[j % 2][i4] = *reinterpret_cast<const f32x4*>(Ps + (16 * i4 + r) * PS + 16 * jt + 4 * g);
                }
                __builtin_amdgcn_sched_barrier(0);
            };
            fetch_x(0);
#pragma unroll
            for (int step = 0; step < 4 * KG; ++step) {
                if (step + 1 < 4 * KG) fetch_x(step + 1);
                else {
                    read_z();
                    fetch_p(0);
                }
#pragma unroll
                for (int q = 0; q < Q; ++q)
#pragma unroll
                    for (int i4 = 0; i4 < 4; ++i4) oacc[i4] = mma4(st[Q * (step / 4) + q][step % 4], bx[step % 2][i4][q], oacc[i4]);
                __builtin_amdgcn_sched_barrier(0);
            }
            if (DECAY) {
#pragma unroll
                for (int i4 = 0; i4 < 4; ++i4)
#pragma unroll
                    for (int v = 0; v < 4; ++v) oacc[i4][v] *= ofac[i4];
            }
            auto intra = [&](auto jc, int jt) __attribute__((always_inline)) {
                constexpr int J = decltype(jc)::value;
#pragma unroll
                for (int v = 0; v < 4; ++v)
#pragma unroll
                    for (int i4 = 0; i4 < 4; ++i4) {
                        const bool need = REVERSE ? (jt >= i4) : (jt <= i4);
                        if (need) oacc[i4] = mma4(zf[jt][v], bp[J % 2][i4][v], oacc[i4]);
                    }
            };
            if constexpr (KH == 1) {
                fetch_p(1);
                intra(std::integral_constant<int, 0>{}, 0);
                __builtin_amdgcn_sched_barrier(0);
                fetch_p(2);
                intra(std::integral_constant<int, 1>{}, 1);
                __builtin_amdgcn_sched_barrier(0);
                fetch_p(3);
                intra(std::integral_constant<int, 2>{}, 2);
                __builtin_amdgcn_sched_barrier(0);
                intra(std::integral_constant<int, 3>{}, 3);
                __builtin_amdgcn_sched_barrier(0);
            } else {
                fetch_p(1);
                if (part == 0) {
                    intra(std::integral_constant<int, 0>{}, 0);
                    intra(std::integral_constant<int, 1>{}, 3);
                } else {
                    intra(std::integral_constant<int, 0>{}, 1);
                    intra(std::integral_constant<int, 1>{}, 2);
                }
                __builtin_amdgcn_sched_barrier(0);
            }
            if constexpr (KH == 1) {
                store(std::integral_constant<int, 0>{}, oacc);
            } else {
                // part 0 completes rows 0 .. 31, part 1 rows 32 .. 63
                float* const mine = Es + (size_t)w * 512 + lane * 4;
#pragma unroll
                for (int i = 0; i < 2; ++i) *reinterpret_cast<f32x4*>(mine + 256 * i) = part == 0 ? oacc[2 + i] : oacc[i];
            }
            if (have_next) update();
        }
        __syncthreads();
        if constexpr (KH == 2) {
            if (wave_active) {
                const float* const theirs = Es + (size_t)(w ^ WC) * 512 + lane * 4;
                f32x4 o[2];
#pragma unroll
                for (int i = 0; i < 2; ++i) o[i] = (part == 0 ? oacc[i] : oacc[2 + i]) + *reinterpret_cast<const f32x4*>(theirs + 256 * i);
                if (part == 0) store(std::integral_constant<int, 0>{}, o);
                else store(std::integral_constant<int, 2>{}, o);
            }
        }
        if (have_next) {
            stage();
            __syncthreads();
        }
    }
}

template <int DKP, int WC, int KH, bool REVERSE, bool DECAY>
__global__ __launch_bounds__(64 * WC * KH, (F32Form<DKP, WC, KH>::per_cu)) void la_sweep_f32_kernel(SweepArgsF32 a) {
    sweep_f32_body<DKP, WC, KH, REVERSE, DECAY>(a, blockIdx.x);
}

// The three sweeps of a backward pass with d == e in one launch: part 0 walks forward (dQ), parts 1 and 2
// backward (dK, dV); the parts have the same number of workgroups (a multiple of 8).
struct SweepTrioF32 {
    SweepArgsF32 a[3];
    unsigned per_part;
};
template <int DKP, int WC, int KH, bool DECAY>
__global__ __launch_bounds__(64 * WC * KH, (F32Form<DKP, WC, KH>::per_cu)) void la_sweep_f32_trio_kernel(SweepTrioF32 t) {
    const unsigned part = blockIdx.x / t.per_part, bid = blockIdx.x % t.per_part;
    if (part == 0) sweep_f32_body<DKP, WC, KH, false, DECAY>(t.a[0], bid);
    else sweep_f32_body<DKP, WC, KH, true, DECAY>(t.a[part == 1 ? 1 : 2], bid);
}

template <int DKP, int WC, int KH, bool DECAY>
static int prep_trio_f32() {
    static unsigned char lds_allowed[kMaxDevices];
    return allow_lds(la_sweep_f32_trio_kernel<DKP, WC, KH, DECAY>, F32Form<DKP, WC, KH>::lds, lds_allowed);
}
template <int DKP, int WC, int KH, bool REVERSE, bool DECAY>
static int prep_one_f32() {
    static unsigned char lds_allowed[kMaxDevices];
    return allow_lds(la_sweep_f32_kernel<DKP, WC, KH, REVERSE, DECAY>, F32Form<DKP, WC, KH>::lds, lds_allowed);
}
// Every instantiation of this file made ready for its first launch on the current device.
int prepare_f32() {
    int e = 0;
#define LA_P(DKP, WC, KH, D) \
    if (!e) e = prep_trio_f32<DKP, WC, KH, D>(); \
    if (!e) e = prep_one_f32<DKP, WC, KH, false, D>(); \
    if (!e) e = prep_one_f32<DKP, WC, KH, true, D>();
#define LA_PF(DKP, WC, KH) LA_P(DKP, WC, KH, false) LA_P(DKP, WC, KH, true)
    LA_PF(64, 4, 1) LA_PF(64, 2, 2) LA_PF(128, 4, 2) LA_PF(128, 2, 2)
#undef LA_PF
#undef LA_P
    return e;
}

template <int DKP, int WC, int KH, bool DECAY>
static int launch_trio_f32(const SweepTrioF32& t, hipStream_t st) {
    typedef F32Form<DKP, WC, KH> F;
    auto kern = la_sweep_f32_trio_kernel<DKP, WC, KH, DECAY>;
    if (const int e = prep_trio_f32<DKP, WC, KH, DECAY>()) return e;
    hipLaunchKernelGGL(kern, dim3(3 * t.per_part), dim3(F::NT), F::lds, st, t);
    return (int)hipGetLastError();
}

template <int DKP, int WC, int KH, bool REVERSE, bool DECAY>
static int launch_one_f32(const SweepArgsF32& a, hipStream_t st) {
    typedef F32Form<DKP, WC, KH> F;
    auto kern = la_sweep_f32_kernel<DKP, WC, KH, REVERSE, DECAY>;
    if (const int e = prep_one_f32<DKP, WC, KH, REVERSE, DECAY>()) return e;
    const int units8 = (a.bh + 7) / 8 * 8;
    hipLaunchKernelGGL(kern, dim3((unsigned)(units8 * a.nslice * a.nchunk)), dim3(F::NT), F::lds, st, a);
    return (int)hipGetLastError();
}

static SweepArgsF32 make_args_f32(const void* x, const void* y, const void* z, void* out, const float* s, int64_t bh, int64_t h,
                                  int64_t n, int64_t dk, int64_t dv, int cols) {
    SweepArgsF32 a;
    a.x = static_cast<const float*>(x); a.y = static_cast<const float*>(y); a.z = static_cast<const float*>(z);
    a.out = static_cast<float*>(out); a.s = s;
    a.n = n; a.dk = (int)dk; a.dv = (int)dv; a.h = (int)h; a.bh = (int)bh;
    a.nslice = (int)((dv + cols - 1) / cols);
    a.nchunk = 1;
    for (int i = 0; i < 9; ++i) a.chunk_start[i] = i == 0 ? 0 : (int)((n + 63) / 64);
    return a;
}

// What a warm-up block costs of a full one (0.75 of 3.05 us, 1.1 of 4.1; 1.4 of 5.0, 2.0 of 6.8), and the fewest blocks a
// chunk is worth cutting off for.  b1 h8 n1024 d64 forward, 32 columns, us, by number of chunks 1 / 2 / 4 / 5 / 8: 52 / 33 / 24 /
// 22 / 21: as many as there are CUs for, down to two blocks each.
static const double kWarmCost = 0.27;
static const int64_t kMinBlocks = 2;

// Columns of z / out per workgroup of a launch of nprod sweeps: 32 in place of 64 where that gives no more workgroups than there
// are CUs and a single round of them, in the chunks the CUs left over allow, is estimated faster - and for rows of up to 32 columns, where
// half of a 64-column workgroup's slabs would be idle, on two of a CU's four SIMDs, and there are as many workgroups either way (64 / 32, us:
// backward of 200 sequences n8192 d24 1685 / 1010, 512 n1000 d24 331 / 247, n113 90 sequences 16.9 / 13.8; forward of 300 n2048 d128 e24
// 435 / 333, 264 n2048 d8 160 / 127).  Per block 3.05 against
// 4.2 us (feature dim 64), 5.15 against 6.9 (128); twice the workgroups leave half the chunks.  us of 64 / 32 columns, both taken when the line
// was drawn, with the next block requested in one piece (blocks are 1 - 4 % quicker since, in either form): forward of d64
// n2048: 8 sequences 44.5 / 35.8, 24 48 / 41, 48 59 / 64, 128 90 / 104; backward 8 63 / 46, 16 63 / 66, 24 76 / 100; d128: 8 forward 74 / 57,
// 24 94 / 105, backward 8 93 / 104, 16 144 / 173.
static double f32_walk_us(int64_t cus, int64_t wgs, int64_t nblk, double block_us) {
    int64_t c = cus / wgs < nblk / kMinBlocks ? cus / wgs : nblk / kMinBlocks;
    double sum = 0.0, weight = 1.0;
    for (int64_t i = 0; i < (c < 1 ? 1 : c > 8 ? 8 : c); ++i) { sum += weight; weight *= 1.0 - kWarmCost; }
    return (double)nblk * block_us / sum;
}
static int f32_columns(int64_t cus, int64_t bh, int64_t n, int64_t dk, int64_t dv, int nprod) {
    const int64_t nblk = (n + 63) / 64, units = (bh + 7) / 8 * 8 * nprod;
    const int64_t narrow = units * ((dv + 31) / 32), wide = units * ((dv + 63) / 64);
    if (dv <= 32) return 32;
    if (narrow > cus) return 64;
    return f32_walk_us(cus, narrow, nblk, dk <= 64 ? 3.05 : 5.15) < 1.03 * f32_walk_us(cus, wide, nblk, dk <= 64 ? 4.2 : 6.9) ? 32 : 64;
}

// `nform`: how many such sweeps the form of the workgroups is chosen for (3: those of a backward pass with d == e, launched apart).
int sweep_f32(const void* x, const void* y, const void* z, void* out, const float* s, int64_t bh, int64_t h,
              int64_t n, int64_t dk, int64_t dv, bool reverse, int nform, const Opts& opts, hipStream_t st) {
    if (dk > 128) return LA_E_UNSUPPORTED;
    const int cols = f32_columns(opts.cus, bh, n, dk, dv, nform);
    SweepArgsF32 a = make_args_f32(x, y, z, out, s, bh, h, n, dk, dv, cols);
    plan_warm_up_chunks(opts.cus, (bh + 7) / 8 * 8 * a.nslice, (n + 63) / 64, opts.chunks, &a.nchunk, a.chunk_start, kWarmCost, kMinBlocks);
#define LA_GD(DKP, WC, KH, R) (s ? launch_one_f32<DKP, WC, KH, R, true>(a, st) : launch_one_f32<DKP, WC, KH, R, false>(a, st))
#define LA_GO(DKP, WC, KH) (reverse ? LA_GD(DKP, WC, KH, true) : LA_GD(DKP, WC, KH, false))
    if (dk <= 64) return cols == 32 ? LA_GO(64, 2, 2) : LA_GO(64, 4, 1);
    return cols == 32 ? LA_GO(128, 2, 2) : LA_GO(128, 4, 2);
#undef LA_GO
#undef LA_GD
}

// float32 backward pass with d == e: dQ = fwd(dO, v, k), dK = rev(v, dO, q), dV = rev(k, q, dO) in one
// launch (the sweeps are independent; with few sequences they run side by side).
int sweep_f32_bwd_once(const void* q, const void* k, const void* v, const void* dout, void* dq, void* dk, void* dv,
                       const float* s, int64_t bh, int64_t h, int64_t n, int64_t d, const Opts& opts, hipStream_t st) {
    if (d > 128) return LA_E_UNSUPPORTED;
    const int cols = f32_columns(opts.cus, bh, n, d, d, 3);
    SweepTrioF32 t;
    t.a[0] = make_args_f32(dout, v, k, dq, s, bh, h, n, d, d, cols);
    t.a[1] = make_args_f32(v, dout, q, dk, s, bh, h, n, d, d, cols);
    t.a[2] = make_args_f32(k, q, dout, dv, s, bh, h, n, d, d, cols);
    plan_warm_up_chunks(opts.cus, (bh + 7) / 8 * 8 * t.a[0].nslice * 3, (n + 63) / 64, opts.chunks, &t.a[0].nchunk, t.a[0].chunk_start, kWarmCost, kMinBlocks);
    for (int i = 1; i < 3; ++i) {
        t.a[i].nchunk = t.a[0].nchunk;
        for (int j = 0; j < 9; ++j) t.a[i].chunk_start[j] = t.a[0].chunk_start[j];
    }
    t.per_part = (unsigned)((bh + 7) / 8 * 8 * t.a[0].nslice * t.a[0].nchunk);
#define LA_GO(DKP, WC, KH) (s ? launch_trio_f32<DKP, WC, KH, true>(t, st) : launch_trio_f32<DKP, WC, KH, false>(t, st))
    if (d <= 64) return cols == 32 ? LA_GO(64, 2, 2) : LA_GO(64, 4, 1);
    return cols == 32 ? LA_GO(128, 2, 2) : LA_GO(128, 4, 2);
#undef LA_GO
}

}  // namespace la
