// Stand-ins for the functions that launch the attention kernels: each writes down what it was asked to launch and
// launches nothing.  Loaded with its symbols global before the library itself, it shows on a machine without a GPU which
// launches a call is mapped onto (tests/launch_routes.py).
#include <cstdio>
#include <string>

#include "la_sweep_common.h"

namespace {
std::string log_;

void note(const char* what, const la::SweepPair& p, bool reverse) {
    static const char* const modes[] = {"warm", "scan", "apply", "resume", "shared"};
    char t[200];
    snprintf(t, sizeof(t), "%s %s%s w%d x%d c%d", what, reverse ? "rev " : "", modes[p.mode], p.wide, p.nprod, p.a[0].nchunk);
    log_ += t;
    if (p.nslot) log_ += p.nprod == 2 ? " shared" : " carried";
    if (p.save) log_ += " saving";
    log_ += ";";
}
}  // namespace

namespace la {
int sweep_pipe(const SweepPair& p, int, bool reverse, hipStream_t) { note("sweep", p, reverse); return 0; }
int sweep_pipe_collect(const SweepPair& p, int, bool reverse, hipStream_t) { note("collect", p, reverse); return 0; }
int sweep_pipe_apply(const SweepPair& p, int, bool reverse, hipStream_t) {
    SweepPair q = p;
    q.mode = kApply;
    note("apply", q, reverse);
    return 0;
}
int sweep_pipe_both(const SweepBoth& b, int, hipStream_t) { note(b.rev.nprod == 2 ? "once" : "dq+dk", b.fwd, false); return 0; }
int sweep_pipe_trio(const SweepTrio& t, int, hipStream_t) { note("trio", t.dq, false); return 0; }
}  // namespace la

// what was recorded since the last call
extern "C" const char* recorded() {
    static std::string out;
    out.swap(log_);
    log_.clear();
    return out.c_str();
}
