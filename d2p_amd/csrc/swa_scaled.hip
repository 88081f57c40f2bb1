// swa_scaled.hip -- affine-gap soft Smith-Waterman and Needleman-Wunsch in the linear
// domain (scaled.hip.h).
#include "scaled_sweeps.hip.h"
#include "swa_internal.hip.h"

namespace d2p_amd {
namespace swa {

int run_scaled(const float* scores, const int* lengths, int B, int max_L1, int max_L2, float go,
               float ge, float T, const Layout& ws, float* value, float* marginals,
               float* grad_open, float* grad_ext, float* grad_T, hipStream_t st, bool nwa,
               bool* done,
               sc::Args* args) {
    *done = false;
    if (!sc::takes(max_L1, max_L2, T, go, ge)) return D2P_OK;
    sc::Args& A = *args;
    A = sc::Args{};
    A.m = scores;
    A.lengths = lengths;
    A.out = marginals;
    A.value = value;
    A.grad0 = grad_open;
    A.grad1 = grad_ext;
    A.gradT = grad_T;
    A.status = ws.status;
    A.redo = ws.redo;
    A.fflag = ws.fflag;
    A.bflag = ws.bflag;
    A.bpart = ws.bpart;
    A.gap = go;
    A.ext = ge;
    A.T = T;
    A.B = B;
    A.L1max = max_L1;
    A.L2max = max_L2;
    A.k = sc::consts(T, go, ge);
    const size_t room = (size_t)((char*)ws.brow - (char*)ws.alpha_sk);
    if (nwa)
        return sc::run<sc::NWAFF>(A, ws.alpha_sk, room, done, st, "nwa_forward", "nwa_backward");
    return sc::run<sc::AFF>(A, ws.alpha_sk, room, done, st, "swa_forward", "swa_backward");
}

}  // namespace swa
}  // namespace d2p_amd
