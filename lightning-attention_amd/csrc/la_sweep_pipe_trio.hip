// The three sweeps of a backward pass with d != e (feature dims up to 128) in one launch: dQ walking forward and dK
// backward, both contracting over e, and dV backward, contracting over d.  The two shapes are two instantiations of the
// pipelined body (la_sweep_pipe_body.h) in one kernel.
// (lightning_attn/ops/triton/lightning_attn2.py:88-395 backward.)
#include "la_sweep_pipe_body.h"

namespace la {

// DKA: padded e (dQ, dK), DKB: padded d (dV).  The workgroups of dV come first: with d > e theirs are the longer walks.
template <typename T, int DKA, int DKB, bool DECAY, bool DENSE>
__global__ __launch_bounds__(512, 1) void la_sweep_pipe_trio_kernel(SweepTrio t) {
    const unsigned bid = blockIdx.x;
    if (bid < t.ndv) sweep_pipe_body<T, DKB, 1, 1, true, DECAY, DENSE>(t.dv, bid);
    else if (bid < t.ndv + t.ndq) sweep_pipe_body<T, DKA, 1, 1, false, DECAY, DENSE>(t.dq, bid - t.ndv);
    else sweep_pipe_body<T, DKA, 1, 1, true, DECAY, DENSE>(t.dk, bid - t.ndv - t.ndq);
}

template <int DKA, int DKB>
constexpr size_t trio_lds(size_t elt) {
    constexpr int DK = DKA > DKB ? DKA : DKB;
    return PipeLds<DK, 1, 1>::bytes(elt);
}

template <typename T, int DKA, int DKB, bool DECAY, bool DENSE>
static int prep_trio() {
    static unsigned char lds_allowed[kMaxDevices];
    return allow_lds(la_sweep_pipe_trio_kernel<T, DKA, DKB, DECAY, DENSE>, trio_lds<DKA, DKB>(sizeof(T)), lds_allowed);
}

template <typename T, int DKA, int DKB, bool DECAY, bool DENSE>
static int launch_trio_one(const SweepTrio& t, hipStream_t st) {
    auto kern = la_sweep_pipe_trio_kernel<T, DKA, DKB, DECAY, DENSE>;
    if (const int e = prep_trio<T, DKA, DKB, DECAY, DENSE>()) return e;
    hipLaunchKernelGGL(kern, dim3(t.ndv + t.ndq + part_grid(t.dk)), dim3(512), (trio_lds<DKA, DKB>(sizeof(T))), st, t);
    return (int)hipGetLastError();
}

template <typename T>
static int launch_trio(const SweepTrio& t, hipStream_t st) {
    const bool decay = t.dq.a[0].s != nullptr;
    const bool dense = all_plain(t.dq) && all_plain(t.dk) && all_plain(t.dv);
#define LA_GO2(A, B, DENSE) (decay ? launch_trio_one<T, A, B, true, DENSE>(t, st) : launch_trio_one<T, A, B, false, DENSE>(t, st))
#define LA_GO(A, B) (dense ? LA_GO2(A, B, true) : LA_GO2(A, B, false))
    if (t.dq.a[0].dk <= 64) return t.dv.a[0].dk <= 64 ? LA_GO(64, 64) : LA_GO(64, 128);
    return t.dv.a[0].dk <= 64 ? LA_GO(128, 64) : LA_GO(128, 128);
#undef LA_GO
#undef LA_GO2
}

int sweep_pipe_trio(const SweepTrio& t, int dtype, hipStream_t st) {
    const SweepArgs &q = t.dq.a[0], &k = t.dk.a[0], &v = t.dv.a[0];
    if (q.dk > 128 || v.dk > 128 || q.dk != k.dk || q.dv != k.dv || q.dk != v.dv || q.dv != v.dk || q.n != k.n || q.n != v.n ||
        q.bh != k.bh || q.bh != v.bh || t.ndq != part_grid(t.dq) || t.ndv != part_grid(t.dv))
        return LA_E_UNSUPPORTED;
    for (const SweepPair* p : {&t.dq, &t.dk, &t.dv})
        if (p->wide || p->mode != kWarmUp || p->nprod != 1 || p->a[0].zw != 64) return LA_E_UNSUPPORTED;
    if (dtype == LA_BF16) return launch_trio<__bf16>(t, st);
    if (dtype == LA_FP16) return launch_trio<_Float16>(t, st);
    return LA_E_UNSUPPORTED;
}

// Every instantiation of this file made ready for its first launch on the current device.
int prepare_trio() {
    int e = 0;
#define LA_P(T, A, B) \
    if (!e) e = prep_trio<T, A, B, false, false>(); \
    if (!e) e = prep_trio<T, A, B, false, true>();  \
    if (!e) e = prep_trio<T, A, B, true, false>();  \
    if (!e) e = prep_trio<T, A, B, true, true>();
    LA_P(__bf16, 64, 64) LA_P(__bf16, 64, 128) LA_P(__bf16, 128, 64) LA_P(__bf16, 128, 128)
    LA_P(_Float16, 64, 64) LA_P(_Float16, 64, 128) LA_P(_Float16, 128, 64) LA_P(_Float16, 128, 128)
#undef LA_P
    return e;
}

}  // namespace la
