// family_impl.hpp -- a mixed signing batch of the fast parameter sets of one
// hash family (128f / 192f / 256f) with its WOTS chains in ONE launch.
//
// Each set's batch keeps its own inputs, outputs and workspace; the prep and
// FORS kernels of all sets run first, then k_sign_family runs every set's
// chains (256f, 192f, 128f; the bulk of the work), so that the batch has one
// tail instead of one per set; then the subtrees, T_k (batches over 256
// requests) and the WOTS gather per set.  Family TUs instantiate it for
// SHA-256 and SHAKE256.  It takes a batch whose sets the split rule runs at 1
// or 2; others run one set after another.  The two are equal but for small
// batches, where a set's own sequence has FORS and chains in one launch: three
// sets, requests each, one launch of chains / one set after another, ms:
// SHA-256 20 1.03 / 0.77, 100 2.18 / 2.17, 600 10.08 / 10.14, SHAKE256 20 1.85
// / 1.40, 100 5.27 / 5.13, 600 26.56 / 27.18, two sets 2048 38.96 / 39.17.  The
// table's split is 1 from 256 to 1024 requests on, by set.
#pragma once
#include "set_impl.hpp"

namespace spx {

struct FamilyWaves {
    uint32_t n[3];  // chain waves per set
};

template <class P0, class P1, class P2>
__global__ void __launch_bounds__(256)
k_sign_family(BatchArgs A0, BatchArgs A1, BatchArgs A2, FamilyWaves W) {
    static_assert(P0::hash == P1::hash && P1::hash == P2::hash, "one hash family");
    uint32_t wave = __builtin_amdgcn_readfirstlane(blockIdx.x * 4 + threadIdx.x / 64);
    if (wave < W.n[2]) {
        chain_wave<P2, 0>(A2, wave);
        return;
    }
    wave -= W.n[2];
    if (wave < W.n[1]) {
        chain_wave<P1, 0>(A1, wave);
        return;
    }
    wave -= W.n[1];
    if (wave < W.n[0]) chain_wave<P0, 0>(A0, wave);
}

template <class P0, int J0, class P1, int J1, class P2, int J2>
struct FamilyImpl {
    static int pid_[3];

    template <class P>
    static void args(const DevBatch& b, BatchArgs& A, int pid) {
        A = BatchArgs{};
        A.sk = b.sk;
        A.sk_stride = b.sk_stride;
        A.msg = b.msg;
        A.moff = b.moff;
        A.mlen = b.mlen;
        A.optrand = b.optrand;
        A.key_idx = b.key_idx;
        A.key_mid = b.key_mid;
        A.sig = b.sig;
        A.sig_stride = b.sig_stride;
        A.n_req = b.n;
        Layout<P>::carve(pid, A, (uint8_t*)b.ws, b.n, kOpSign);
    }
    template <class P, int J>
    static void fors(const BatchArgs& A, uint32_t n, hipStream_t s) {
        if (n) launch_fors<P, J>(A, n, s);
    }
    template <class P>
    static void tail(const BatchArgs& A, uint32_t n, hipStream_t s) {
        if (!n) return;
        launch_ht<P, 0, 1>(A, s);
        prof_mark(s, "k_ht");
        if (!A.fors_count) {
            launch_fors_pk<P>(A, n, s);
            prof_mark(s, "k_fors_pk");
        }
        hipLaunchKernelGGL((k_wots_gather<P>), dim3(cdiv((uint64_t)n * P::d * P::len, 256)),
                           dim3(256), 0, s, A);
        prof_mark(s, "k_wots_gather");
    }

    static int sign(const DevBatch* b, hipStream_t s) {
        const uint32_t n0 = b[0].n, n1 = b[1].n, n2 = b[2].n;
        if (n0 + n1 + n2 == 0) return kOk;
        if ((n0 && Layout<P0>::split(pid_[0], kOpSign, n0 * P0::d) > 2) ||
            (n1 && Layout<P1>::split(pid_[1], kOpSign, n1 * P1::d) > 2) ||
            (n2 && Layout<P2>::split(pid_[2], kOpSign, n2 * P2::d) > 2))
            return kNotFused;
        BatchArgs A0, A1, A2;
        args<P0>(b[0], A0, pid_[0]);
        args<P1>(b[1], A1, pid_[1]);
        args<P2>(b[2], A2, pid_[2]);
        (void)hipGetLastError();  // report only errors of these launches
        prof_begin(s, "family");
        if (n0) launch_prep<P0, false>(A0, n0, b[0].mlen_bound, s);
        if (n1) launch_prep<P1, false>(A1, n1, b[1].mlen_bound, s);
        if (n2) launch_prep<P2, false>(A2, n2, b[2].mlen_bound, s);
        prof_mark(s, "k_prep");
        fors<P0, J0>(A0, n0, s);
        fors<P1, J1>(A1, n1, s);
        fors<P2, J2>(A2, n2, s);
        prof_mark(s, "k_fors");
        // slices of the same share of every set (slices.hpp)
        const uint64_t waves = (uint64_t)chain_waves<P0>(n0 * P0::d) + chain_waves<P1>(n1 * P1::d) +
                               chain_waves<P2>(n2 * P2::d);
        const uint64_t c = 64 * waves / kSliceLanes + 1;
        for (uint64_t i = 0; i < c; i++) {
            const uint32_t a0 = n0 * i / c, a1 = n1 * i / c, a2 = n2 * i / c;
            const BatchArgs B0 = batch_rows<P0, 0>(A0, a0, n0 * (i + 1) / c - a0),
                            B1 = batch_rows<P1, 0>(A1, a1, n1 * (i + 1) / c - a1),
                            B2 = batch_rows<P2, 0>(A2, a2, n2 * (i + 1) / c - a2);
            FamilyWaves W{{chain_waves<P0>(B0.n_req * P0::d), chain_waves<P1>(B1.n_req * P1::d),
                           chain_waves<P2>(B2.n_req * P2::d)}};
            const uint32_t grid = cdiv((uint64_t)W.n[0] + W.n[1] + W.n[2], 4);
            hipLaunchKernelGGL((k_sign_family<P0, P1, P2>), dim3(grid), dim3(256), 0, s, B0, B1, B2,
                               W);
        }
        prof_mark(s, "k_sign_family");
        tail<P0>(A0, n0, s);
        tail<P1>(A1, n1, s);
        tail<P2>(A2, n2, s);
        return hipGetLastError() == hipSuccess ? 0 : kErrHip;
    }

    static FamilyOps ops(int p0, int p1, int p2) {
        pid_[0] = p0;
        pid_[1] = p1;
        pid_[2] = p2;
        FamilyOps o{};
        o.pid[0] = p0;
        o.pid[1] = p1;
        o.pid[2] = p2;
        o.sign = &sign;
        return o;
    }
};

template <class P0, int J0, class P1, int J1, class P2, int J2>
int FamilyImpl<P0, J0, P1, J1, P2, J2>::pid_[3] = {-1, -1, -1};

}  // namespace spx

#define SPX_REGISTER_FAMILY(SYM, P0, J0, PID0, P1, J1, PID1, P2, J2, PID2)              \
    extern "C" const spx::FamilyOps* SYM(void) {                                        \
        static const spx::FamilyOps o =                                                 \
            spx::FamilyImpl<P0, J0, P1, J1, P2, J2>::ops(PID0, PID1, PID2);             \
        return &o;                                                                      \
    }
