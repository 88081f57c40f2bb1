// sw_scaled.hip -- linear-gap soft Smith-Waterman and Needleman-Wunsch in the linear
// domain (scaled.hip.h).
#include "scaled_sweeps.hip.h"
#include "sw_internal.hip.h"

namespace d2p_amd {
namespace sw {

int run_scaled(const float* scores, const int* lengths, int B, int max_L1, int max_L2, float gap,
               float T, const Layout& ws, float* value, float* marginals, float* grad_gap,
               float* grad_T, hipStream_t st, bool global, bool* done,
               sc::Args* args) {
    *done = false;
    if (!sc::takes(max_L1, max_L2, T, gap, 0.0)) return D2P_OK;
    sc::Args& A = *args;
    A = sc::Args{};
    A.m = scores;
    A.lengths = lengths;
    A.out = marginals;
    A.value = value;
    A.grad0 = grad_gap;
    A.gradT = grad_T;
    A.status = ws.status;
    A.redo = ws.redo;
    A.fflag = ws.fflag;
    A.bflag = ws.bflag;
    A.bpart = ws.bpart;
    A.gap = gap;
    A.T = T;
    A.B = B;
    A.L1max = max_L1;
    A.L2max = max_L2;
    A.k = sc::consts(T, gap, 0.0);
    const size_t room = (size_t)((char*)ws.brow - (char*)ws.alpha_sk);
    if (global) return sc::run<sc::NW>(A, ws.alpha_sk, room, done, st, "nw_forward", "nw_backward");
    return sc::run<sc::SW>(A, ws.alpha_sk, room, done, st, "sw_forward", "sw_backward");
}

}  // namespace sw
}  // namespace d2p_amd
