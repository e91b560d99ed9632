// spx_kernels.hpp -- batched SPHINCS+ sign / verify / keygen kernels.
//
// One signature is split across many lanes (MI355X needs >> 256 workgroups
// and prefers uniform control flow inside a wave):
//
//   sign:   k_prep       lane group per request: midstate, PRF_msg, H_msg, plan
//           k_fors       L lanes per FORS tree (2^J leaves per lane), LDS reduce
//           k_fors_pk    lane group per request: T_k over the k roots (small
//                        batches: run by the lane storing the last root)
//           k_chains     lane per WOTS chain of every leaf of every hypertree
//                        layer (all d layers at once: every layer's tree/leaf
//                        comes from H_msg alone); the signing leaf's chain
//                        values are captured.  k_sign_fused: k_fors and
//                        k_chains in one launch
//           k_ht         T_len per leaf, LDS reduce, auth path, layer root
//           k_wots_gather lane per (request, layer, chain): picks the
//                        captured chain value for the layer's message
//   verify: k_vprep, k_vfors, k_fors_pk, k_vht (the chains of a workgroup's
//           requests dealt over its lanes, layers in sequence); small
//           batches: k_vspec (FORS trees, every chain from every start) +
//           k_vht_spec (T_k, then T_len and the climb per layer)
//   keygen: k_kprep, k_chains and k_ht in keygen mode (top layer only)
//
// Semantics follow sign.cu:1924-1994 (sign), sign.cu:3048-3121 (verify),
// sign.cu:154-182 (keygen), utils.cu:94-241 (compute_root / treehash),
// wots.cu:27-790 and fors.cu:24-633 of the reference.
#pragma once
#include <type_traits>

#include "sha2_dev.hpp"
#include "shake_dev.hpp"

namespace spx {

__host__ __device__ constexpr int max_int(int a, int b) { return a > b ? a : b; }

template <class P>
using HashT = typename std::conditional<P::hash == kSha2, Sha2<P::n>, Shake<P::n>>::type;
// PH = false: for launches of at most kAloneWaves waves (one per SIMD), where
// SHA-256 does without two-phase rounds.  With -> without them, us: k_chains of
// SHA2-128f key generation, 1 key 48 -> 39, 200 (875 waves) 53 -> 44; k_vspec
// SHA2-128f 1 request 46 -> 40, SHA2-256s 3 92 -> 75; k_sign_fused SHA2-128f 1
// 51 -> 48, SHA2-192f 3 88 -> 81; k_vfors SHA2-192f 300 (155 waves) 55 -> 45,
// but SHA2-128f 1900 (980 waves) 32 -> 38.
template <class P, bool PH>
using HashPh =
    typename std::conditional<P::hash == kSha2, Sha2<P::n, PH>, Shake<P::n>>::type;
constexpr uint32_t kAloneWaves = 1024;

// ------------------------------------------------------------- arguments

struct BatchArgs {
    // inputs
    const uint8_t* sk;        // sign: secret keys, stride sk_stride
    uint32_t sk_stride;
    const uint8_t* pk;        // verify: public keys, stride pk_stride
    uint32_t pk_stride;
    const uint8_t* seed;      // keygen: 3n-byte seeds, stride seed_stride
    uint32_t seed_stride;
    const uint8_t* msg;       // messages: msg + moff[i], mlen[i] bytes, 4-byte aligned
    const uint64_t* moff;
    const uint32_t* mlen;
    const uint8_t* optrand;   // sign: [N][n]
    const uint32_t* key_idx;  // optional: request i uses key row key_idx[i] of sk / pk
    const uint32_t* key_mid;  // optional: precomputed SHA-256 midstate per key row (8 words)
    // outputs
    uint8_t* sig;             // signatures (sign: written, verify: read)
    uint64_t sig_stride;
    int32_t* status;          // verify: 0 ok / -1 fail per request
    uint8_t* pk_out;          // keygen outputs
    uint8_t* sk_out;
    // workspace
    Plan* plan;
    uint8_t* fors_roots;      // [N][k][n]
    uint8_t* fors_pk;         // [N][n]
    uint8_t* roots;           // [N][d][n]
    uint8_t* cap;             // [N][d][len][16][n]
    uint32_t* tl_buf;         // chain ends: [len*nw][leaves]
    uint32_t tl_lanes;
    uint32_t* ht_parts;       // split subtrees (before them, split FORS trees): part roots
                              // [tree][part][nw]
    uint32_t* ht_count;       // split subtrees: parts finished per tree (zeroed by the prep kernel)
    uint32_t* fors_count;     // FORS roots finished per request (zeroed by the prep kernels)
    uint32_t n_req;
    // prep kernels: messages of long_min bytes or more (0: none) are hashed by
    // the first long_wgs workgroups, in their two-wave form
    uint32_t long_wgs;
    uint32_t long_min;
};

// ----------------------------------------------------- message / indices

template <class P>
__device__ __forceinline__ void plan_from_digest(Plan& pl, const uint8_t* dg) {
    // message_to_indices (fors.cu:77-91): LSB-first bits within each byte
#pragma unroll
    for (int t = 0; t < P::k; t++) {
        uint32_t v = 0;
#pragma unroll
        for (int j = 0; j < P::a; j++) {
            const int off = t * P::a + j;
            v |= (uint32_t)((dg[off >> 3] >> (off & 7)) & 1) << j;
        }
        pl.fors_idx[t] = v;
    }
    // tree / leaf (hash_sha256.cu:249-261): big-endian, masked
    uint64_t tree = 0;
#pragma unroll
    for (int i = 0; i < P::tree_bytes; i++)
        tree = (tree << 8) | dg[P::fors_msg_bytes + i];
    if (P::tree_bits < 64) tree &= (~0ull) >> (64 - P::tree_bits);
    uint32_t leaf = 0;
#pragma unroll
    for (int i = 0; i < P::leaf_bytes; i++)
        leaf = (leaf << 8) | dg[P::fors_msg_bytes + P::tree_bytes + i];
    leaf &= (~0u) >> (32 - P::leaf_bits);
    pl.tree = tree;
    pl.leaf = leaf;
}

// The prep kernels (128-lane workgroups).  Workgroups from long_wgs on: every
// request hashes its message on a lane group; all its lanes compute
// everything, the first one stores.  SHA-256: 8 lanes, 16 requests per
// workgroup; the message's blocks run on each pair alike, the HMAC keys, the
// MGF1 blocks and the midstate on a pair each, so that a short message's 9
// dependent blocks are 6 (SHA2-128f, 32 bytes: 30.4 -> 25.0 us at 1 request,
// 45 -> 37 at 4096; k_vprep 19.8 -> 15.5).  SHAKE256: 32 lanes, Keccak32, 4
// requests, and a lane pair in large batches.  SHA-256 messages of at least long_min bytes are left to the
// workgroups before those: each takes long requests in turn and runs one with
// both waves (Sha2::stream_msg_long), the schedules of its message-only blocks
// computed by wave 1 ahead of wave 0's rounds.  They come first so that the
// dispatcher spreads them evenly: placed among thousands of short workgroups
// that end at once, some CUs held several of them to the end (65536 SHA2-128f
// requests of 4 KiB, k_vprep 28-38 ms; 12.5 ms first).
//
// Lanes past the last request repeat it and store nothing, here and in the
// other kernels whose time is one wave's: a wave with less than all its
// lanes active has been slower by up to a third, and four such waves on one CU
// by up to 3.5 times, changing from launch to launch (T_len's rounds on a
// pair: 2.9k cycles a block with all lanes active, 2.9-10k with two of 16).
template <class P>
__host__ __device__ constexpr uint32_t prep_lanes(bool pair) {
    return pair ? 2 : P::hash == kSha2 ? 8 : 32;
}
// SHAKE256 requests up to which a row of 32 lanes hashes a message: beyond,
// the rows' instructions (two requests a wave) last longer than a lane pair's
// serial run.  k_vprep of SHAKE256-128f, rows / pairs, us: 6144 requests of
// 1000 B 57 / 62, of 16 KiB 715 / 734; 8192 68 / 62 and 900 / 734; 16384 of 16
// KiB 1672 / 736; 65536 of 4 KiB 1665 / 385.
constexpr uint32_t kPrepRows = 7168;
constexpr uint32_t kPrepWg = 128;
// the two-wave path from this length: signing one SHA2-128f / 256f request of
// 512 B takes 129 / 233 us against 141 / 240 on the group of 8 lanes, of 2 KiB
// 191 / 295 against 240 / 339, of 64 KiB 2.69 / 2.80 ms against 4.40 / 4.33; 300
// requests of 512 B 0.895 / 2.898 ms against 0.903 / 2.924.  (In batches that
// fill the SIMDs with groups the 512 workgroups are behind: 2000 requests of
// 512 B 5.12 / 17.64 ms against 4.97 / 17.42, of 2 KiB 5.42 / 18.01 against
// 5.10 / 17.59.)
constexpr uint32_t kLongMsgBytes = 512;
constexpr uint32_t kLongWgs = 512;         // at most this many two-wave workgroups

template <class P>
__host__ __device__ constexpr bool prep_has_long() { return P::hash == kSha2; }

__device__ __forceinline__ bool prep_is_long(const BatchArgs& A, uint32_t i) {
    return A.long_min && A.mlen[i] >= A.long_min;
}

// the plan's midstate: the table's where the caller keeps one, else the one
// that h_msg made beside its last blocks
__device__ __forceinline__ void prep_midstate(const BatchArgs& A, uint32_t row,
                                              const uint32_t mid[8], Plan& pl) {
#pragma unroll
    for (int j = 0; j < 8; j++) pl.mid[j] = A.key_mid ? A.key_mid[(size_t)row * 8 + j] : mid[j];
}

// sign, one request: midstate, R = PRF_msg, digest = H_msg, plan; LONG: the
// two-wave form over kw_s (prod: wave 1), else a lane group (SHAKE256: with
// its row's sponge k, or a lane pair)
template <class P, bool LONG, bool PAIR = false>
__device__ __forceinline__ void prep_sign_one(const BatchArgs& A, uint32_t i, bool store,
                                              lds_u32* kw_s, bool prod, Keccak32* k) {
    using Hh = HashT<P>;
    constexpr int NW = P::nw;
    const uint32_t row = A.key_idx ? A.key_idx[i] : i;
    const uint8_t* sk = A.sk + (size_t)row * A.sk_stride;
    uint32_t skseed[NW], skprf[NW], pub[NW], pk[2 * NW], opt[NW], R[NW];
    load_val<P::hash, NW>(sk, skseed);
    load_val<P::hash, NW>(sk + P::n, skprf);
    load_val<P::hash, NW>(sk + 2 * P::n, pub);
    load_val<P::hash, 2 * NW>(sk + 2 * P::n, pk);
    load_val<P::hash, NW>(A.optrand + (size_t)i * P::n, opt);
    const uint8_t* m = A.msg + A.moff[i];
    const uint32_t ml = A.mlen[i];
    Plan pl;
    uint32_t mid[8] = {};
#pragma unroll
    for (int j = 0; j < 8; j++) {
        pl.skseed[j] = j < NW ? skseed[j] : 0u;
        pl.pubseed[j] = j < NW ? pub[j] : 0u;
        pl.root[j] = 0;
    }
    uint8_t dg[P::dgst_bytes];
    if constexpr (LONG) {
        Hh::template prf_msg<true>(skprf, opt, m, ml, R, kw_s, prod);
        Hh::template h_msg<P::dgst_bytes, true>(R, pk, m, ml, dg, mid, kw_s, prod);
    } else if constexpr (P::hash == kShake) {
        Hh::template prf_msg<PAIR>(k, skprf, opt, m, ml, R);
        Hh::template h_msg<P::dgst_bytes, PAIR>(k, R, pk, m, ml, dg);
    } else {
        Hh::prf_msg(skprf, opt, m, ml, R);
        Hh::template h_msg<P::dgst_bytes>(R, pk, m, ml, dg, mid);
    }
    (void)kw_s;
    (void)prod;
    (void)k;
    if (!store) return;
    uint8_t* sig = A.sig + (size_t)i * A.sig_stride;
    store_val<P::hash, NW>(sig, R);
    prep_midstate(A, row, mid, pl);
    plan_from_digest<P>(pl, dg);
    pl.status = 0;
    A.plan[i] = pl;
}

// sign: midstate, R = PRF_msg, digest = H_msg, plan
template <class P, bool PAIR>
__global__ void __launch_bounds__(kPrepWg) k_prep(BatchArgs A) {
    // one serial hash chain per request over the whole message: ask the SIMD
    // arbiter to favour these waves over concurrent bulk hypertree waves
    __builtin_amdgcn_s_setprio(3);
    if (blockIdx.x < A.long_wgs) {
        if constexpr (prep_has_long<P>()) {
            __shared__ __align__(16) uint32_t kw_s[HashT<P>::kLongLdsWords];
            const bool prod = threadIdx.x >= 64;
#pragma unroll 1
            for (uint32_t i = blockIdx.x; i < A.n_req; i += A.long_wgs)
                if (prep_is_long(A, i))
                    prep_sign_one<P, true>(A, i, threadIdx.x == 0, (lds_u32*)kw_s, prod, nullptr);
        }
        return;
    }
    constexpr uint32_t PL = prep_lanes<P>(PAIR);
    const uint32_t lane0 = (blockIdx.x - A.long_wgs) * kPrepWg;
    const uint32_t i0 = (lane0 + threadIdx.x) / PL;
    if ((lane0 + (threadIdx.x & ~63u)) / PL >= A.n_req) return;  // an empty wave
    const uint32_t i = i0 < A.n_req ? i0 : A.n_req - 1;
    const bool first = i0 < A.n_req && threadIdx.x % PL == 0;
    if (A.ht_count && first) {
#pragma unroll 1
        for (int layer = 0; layer < P::d; layer++) A.ht_count[(size_t)i * P::d + layer] = 0;
    }
    if (A.fors_count && first) A.fors_count[i] = 0;
    if (prep_is_long(A, i)) return;
    if constexpr (P::hash == kShake && !PAIR) {
        constexpr int RW = HashT<P>::kRowWords;
        __shared__ __align__(16) uint32_t row_s[kPrepWg / PL * RW];
        Keccak32 k;
        k.init((lds_u32*)row_s + threadIdx.x / PL * RW);
        prep_sign_one<P, false>(A, i, first, nullptr, false, &k);
    } else {
        prep_sign_one<P, false, PAIR>(A, i, first, nullptr, false, nullptr);
    }
}

// verify, one request: midstate, digest = H_msg(R from the signature), plan
// (LONG, PAIR as for prep_sign_one)
template <class P, bool LONG, bool PAIR = false>
__device__ __forceinline__ void prep_verify_one(const BatchArgs& A, uint32_t i, bool store,
                                                lds_u32* kw_s, bool prod, Keccak32* k) {
    using Hh = HashT<P>;
    constexpr int NW = P::nw;
    const uint32_t row = A.key_idx ? A.key_idx[i] : i;
    const uint8_t* pkp = A.pk + (size_t)row * A.pk_stride;
    uint32_t pub[NW], pk[2 * NW], R[NW];
    load_val<P::hash, NW>(pkp, pub);
    load_val<P::hash, 2 * NW>(pkp, pk);
    const uint8_t* sig = A.sig + (size_t)i * A.sig_stride;
    load_val<P::hash, NW>(sig, R);
    Plan pl;
    uint32_t mid[8] = {};
#pragma unroll
    for (int j = 0; j < 8; j++) {
        pl.skseed[j] = 0;
        pl.pubseed[j] = j < NW ? pub[j] : 0u;
        pl.root[j] = j < NW ? pk[NW + j] : 0u;
    }
    uint8_t dg[P::dgst_bytes];
    if constexpr (LONG) {
        Hh::template h_msg<P::dgst_bytes, true>(R, pk, A.msg + A.moff[i], A.mlen[i], dg, mid,
                                                kw_s, prod);
    } else if constexpr (P::hash == kShake) {
        Hh::template h_msg<P::dgst_bytes, PAIR>(k, R, pk, A.msg + A.moff[i], A.mlen[i], dg);
    } else {
        Hh::template h_msg<P::dgst_bytes>(R, pk, A.msg + A.moff[i], A.mlen[i], dg, mid);
    }
    (void)kw_s;
    (void)prod;
    (void)k;
    if (!store) return;
    prep_midstate(A, row, mid, pl);
    plan_from_digest<P>(pl, dg);
    pl.status = 0;
    A.plan[i] = pl;
}

// verify: midstate, digest = H_msg(R from the signature), plan
template <class P, bool PAIR>
__global__ void __launch_bounds__(kPrepWg) k_vprep(BatchArgs A) {
    __builtin_amdgcn_s_setprio(3);  // serial message hash per request, as in k_prep
    if (blockIdx.x < A.long_wgs) {
        if constexpr (prep_has_long<P>()) {
            __shared__ __align__(16) uint32_t kw_s[HashT<P>::kLongLdsWords];
            const bool prod = threadIdx.x >= 64;
#pragma unroll 1
            for (uint32_t i = blockIdx.x; i < A.n_req; i += A.long_wgs)
                if (prep_is_long(A, i))
                    prep_verify_one<P, true>(A, i, threadIdx.x == 0, (lds_u32*)kw_s, prod, nullptr);
        }
        return;
    }
    constexpr uint32_t PL = prep_lanes<P>(PAIR);
    const uint32_t lane0 = (blockIdx.x - A.long_wgs) * kPrepWg;
    const uint32_t i0 = (lane0 + threadIdx.x) / PL;
    if ((lane0 + (threadIdx.x & ~63u)) / PL >= A.n_req) return;  // an empty wave
    const uint32_t i = i0 < A.n_req ? i0 : A.n_req - 1;
    const bool first = i0 < A.n_req && threadIdx.x % PL == 0;
    if (prep_is_long(A, i)) return;
    if constexpr (P::hash == kShake && !PAIR) {
        constexpr int RW = HashT<P>::kRowWords;
        __shared__ __align__(16) uint32_t row_s[kPrepWg / PL * RW];
        Keccak32 k;
        k.init((lds_u32*)row_s + threadIdx.x / PL * RW);
        prep_verify_one<P, false>(A, i, first, nullptr, false, &k);
    } else {
        prep_verify_one<P, false, PAIR>(A, i, first, nullptr, false, nullptr);
    }
}

// grid of the prep kernels for n requests whose messages are at most
// mlen_bound bytes (0: not known); sets A.long_wgs / A.long_min
template <class P, bool PAIR>
inline uint32_t prep_grid(BatchArgs& A, uint32_t n, uint32_t mlen_bound) {
    const bool lng = prep_has_long<P>() && (mlen_bound == 0 || mlen_bound >= kLongMsgBytes);
    A.long_min = lng ? kLongMsgBytes : 0;
    A.long_wgs = !lng ? 0 : n < kLongWgs ? n : kLongWgs;
    return A.long_wgs + (uint32_t)(((uint64_t)n * prep_lanes<P>(PAIR) + kPrepWg - 1) / kPrepWg);
}
// sets fields of A, which later launches then carry along
template <class P, bool VERIFY>
inline void launch_prep(BatchArgs& A, uint32_t n, uint32_t mlen_bound, hipStream_t s) {
    auto go = [&](auto pair) {
        constexpr bool PAIR = decltype(pair)::value;
        const uint32_t wgs = prep_grid<P, PAIR>(A, n, mlen_bound);
        if constexpr (VERIFY)
            hipLaunchKernelGGL((k_vprep<P, PAIR>), dim3(wgs), dim3(kPrepWg), 0, s, A);
        else hipLaunchKernelGGL((k_prep<P, PAIR>), dim3(wgs), dim3(kPrepWg), 0, s, A);
    };
    if constexpr (P::hash == kShake) {
        if (n > kPrepRows) {
            go(std::true_type{});
            return;
        }
    }
    go(std::false_type{});
}

// resident-key midstates: mid[i] = state after pub_seed || 0^(64-n) for the
// public key row i (seed_state, sha256.cu:391-405); zero for SHAKE sets
template <class P>
__global__ void __launch_bounds__(64) k_midstate(const uint8_t* pk, uint32_t pk_stride,
                                                 uint32_t* mid, uint32_t n) {
    using Hh = HashT<P>;
    constexpr int NW = P::nw;
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    uint32_t pub[NW], m[8];
    load_val<P::hash, NW>(pk + (size_t)i * pk_stride, pub);
    Hh::midstate(pub, m);
#pragma unroll
    for (int j = 0; j < 8; j++) mid[(size_t)i * 8 + j] = m[j];
}

// keygen: sk = seed (3n) || root, plan with the key material
template <class P>
__global__ void __launch_bounds__(64) k_kprep(BatchArgs A) {
    using Hh = HashT<P>;
    constexpr int NW = P::nw;
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= A.n_req) return;
    const uint8_t* s = A.seed + (size_t)i * A.seed_stride;
    uint32_t skseed[NW], pub[NW];
    load_val<P::hash, NW>(s, skseed);
    load_val<P::hash, NW>(s + 2 * P::n, pub);
    Plan pl;
    Hh::midstate(pub, pl.mid);
#pragma unroll
    for (int j = 0; j < 8; j++) {
        pl.skseed[j] = j < NW ? skseed[j] : 0u;
        pl.pubseed[j] = j < NW ? pub[j] : 0u;
        pl.root[j] = 0;
    }
    pl.tree = 0;
    pl.leaf = 0;
    pl.status = 0;
    A.plan[i] = pl;
    if (A.ht_count) A.ht_count[i] = 0;
    // sk = SK_SEED || SK_PRF || PUB_SEED (|| root, written by k_ht); pk = PUB_SEED || root
    uint8_t* sko = A.sk_out + (size_t)i * P::sk_bytes;
    uint8_t* pko = A.pk_out + (size_t)i * P::pk_bytes;
    for (int j = 0; j < 3 * P::n; j++) sko[j] = s[j];
    for (int j = 0; j < P::n; j++) pko[j] = s[2 * P::n + j];
}

// ------------------------------------------------------------------ FORS

template <class P>
__device__ __forceinline__ void fors_pk_wave(const BatchArgs& A, uint32_t i, lds_u32* lds);
template <class P>
__host__ __device__ constexpr int fors_pk_wave_words();

// a FORS root of request req is stored: count it; true for the request's last
// root.  The wave that stored it then computes the FORS public key (fors_pk_wave), so T_k overlaps the
// hypertree chains instead of taking a launch of its own (the k roots of one
// request come from several workgroups; every counter was zeroed by the prep
// kernel).  Large batches launch k_fors_pk instead: there the per-tile
// release fences (an L2 write-back each) cost more than the launch.
// (FP: parts of a tree, each counted)
template <class P, int FP>
__device__ __forceinline__ bool fors_root_done(const BatchArgs& A, uint32_t req) {
    __threadfence();  // release this root before counting it
    const bool last = atomicAdd(&A.fors_count[req], 1u) == (uint32_t)(P::k * FP) - 1;
    if (last) __threadfence();  // acquire: every root of the request is visible
    return last;
}

// workgroups of 256 lanes that a FORS tree of 2^J leaves per lane is split over
template <class P, int J>
__host__ __device__ constexpr int fors_parts() {
    return P::a - J > 8 ? 1 << (P::a - J - 8) : 1;
}

// LDS words a FORS tile of set P uses (two levels of 256 nodes)
template <class P>
constexpr int fors_lds_words() {
    return 2 * 256 * P::nw;
}

// The top of request req's split FORS trees (FP parts each, their roots in
// ht_parts) on a whole wave, a lane per tree: node m of 1 .. 2 FP - 1 (1 the
// root) is H(2 m, 2 m + 1).  smem: 2 FP values per lane.  The FORS roots are
// visible to the wave's later loads.
template <class P, int FP, class Hh>
__device__ __forceinline__ void fors_top(const BatchArgs& A, uint32_t req, lds_u32* smem) {
    constexpr int NW = P::nw;
    static_assert(2 * FP * 64 * NW <= fors_lds_words<P>() && P::k <= 64, "");
    const uint32_t lane = threadIdx.x & 63u;
    const uint32_t t = lane < (uint32_t)P::k ? lane : P::k - 1;  // repeated past the last tree
    const Plan& pl = A.plan[req];
    typename Hh::Key key;
    Hh::load_key(pl, key);
    Adr a = adr_make(0, pl.tree, kForsTree);
    adr_keypair<P::th>(a, pl.leaf);
    const uint32_t tg = pl.fors_idx[t];
    uint8_t* rec = A.sig + (size_t)req * A.sig_stride + P::n + (size_t)t * (P::a + 1) * P::n;
    const uint32_t* parts = A.ht_parts + ((size_t)req * P::k + t) * (FP * NW);
    lds_u32* val = smem + lane;  // word w of node m at val[64 (m NW + w)]
#pragma unroll 1
    for (int i = 0; i < FP * NW; i++)
        val[64 * (FP * NW + i)] = __builtin_nontemporal_load(parts + i);
#pragma unroll 1
    for (int m = FP - 1; m >= 1; m--) {
        const uint32_t up = 31 - __builtin_clz((uint32_t)m);  // levels below the root
        const uint32_t hgt = P::a - up, x = m - (1u << up);
        uint32_t l[NW], r[NW], out[NW];
#pragma unroll
        for (int w = 0; w < NW; w++) {
            l[w] = val[64 * (2 * m * NW + w)];
            r[w] = val[64 * ((2 * m + 1) * NW + w)];
        }
        adr_node(a, hgt, ((t << P::a) >> hgt) + x);
        Hh::H(key, a, l, r, out);
#pragma unroll
        for (int w = 0; w < NW; w++) val[64 * (m * NW + w)] = out[w];
        if (lane == t) {
            if (m == 1)
                store_val<P::hash, NW>(A.fors_roots + ((size_t)req * P::k + t) * P::n, out);
            else if (x == ((tg >> hgt) ^ 1u))
                store_val<P::hash, NW>(rec + P::n + (size_t)hgt * P::n, out);
        }
    }
    __threadfence();
}

// sign: FORS trees, L = 2^(a-J) lanes per tree, 2^J leaves per lane; `blk`
// is the workgroup's tile (TPW trees, or one of FP parts of a tree wider than
// a workgroup), so the same body serves the fused signing kernels.  smem: fors_lds_words<P>() words of LDS owned by the kernel
// PK: count the roots and run T_k here (fors_count set)
template <class P, int J, bool PK, bool PH = true>
__device__ __forceinline__ void fors_tile(const BatchArgs& A, uint32_t blk, uint32_t* smem) {
    using Hh = HashPh<P, PH>;
    using Key = typename Hh::Key;
    constexpr int NW = P::nw;
    constexpr int WG = 256;
    constexpr int FP = fors_parts<P, J>();
    static_assert(FP == 1 || PK, "the last part climbs from the others' roots");
    constexpr int LOGL = P::a - J - ilog2(FP);  // levels reduced in the workgroup
    constexpr int L = 1 << LOGL;                // lanes of a tree, or of its part, here
    constexpr int TPW = WG / L;
    auto& lds = *reinterpret_cast<uint32_t (*)[2][WG][NW]>(smem);

    const int tid = threadIdx.x;
    const uint32_t part = FP > 1 ? blk % FP : 0;
    if (FP > 1) blk /= FP;
    const uint32_t g = blk * TPW + tid / L;  // global tree id
    const uint32_t u = part * L + tid % L;
    const bool active = g < A.n_req * P::k;
    const uint32_t req = active ? g / P::k : 0;
    const uint32_t t = active ? g % P::k : 0;
    const Plan& pl = A.plan[req];
    Key key;
    Hh::load_key(pl, key);
    const uint32_t target = pl.fors_idx[t];
    Adr adr = adr_make(0, pl.tree, kForsTree);
    adr_keypair<P::th>(adr, pl.leaf);
    uint8_t* rec = A.sig + (size_t)req * A.sig_stride + P::n + (size_t)t * (P::a + 1) * P::n;

    uint32_t node[NW];
    uint32_t stk[J > 0 ? J : 1][NW];
    const uint32_t base = (t << P::a) + (u << J);  // global leaf index of this lane's first leaf
#pragma unroll 1
    for (uint32_t i = 0; i < (1u << J); i++) {
        const uint32_t li = (u << J) + i;  // leaf index within the tree
        uint32_t sk[NW];
        adr_node(adr, 0, base + i);
        Hh::PRF(key, adr, sk);
        Hh::F(key, adr, sk, node);
        if (active && li == target) store_val<P::hash, NW>(rec, sk);
        if (active && li == (target ^ 1u)) store_val<P::hash, NW>(rec + P::n, node);
        // merge with pending left siblings (i is uniform across the wave)
        uint32_t h = 0;
#pragma unroll 1
        while (h < (uint32_t)J && ((i >> h) & 1u)) {
            uint32_t left[NW];
#pragma unroll
            for (int w = 0; w < NW; w++) {
                uint32_t x = stk[0][w];
#pragma unroll
                for (int s = 1; s < J; s++) x = (h == (uint32_t)s) ? stk[s][w] : x;
                left[w] = x;
            }
            h++;
            const uint32_t idx = li >> h;  // node index at height h within the tree
            adr_node(adr, h, ((t << P::a) >> h) + idx);
            Hh::H(key, adr, left, node, node);
            if (active && idx == ((target >> h) ^ 1u))
                store_val<P::hash, NW>(rec + P::n + (size_t)h * P::n, node);
        }
        if (h < (uint32_t)J) {
#pragma unroll
            for (int s = 0; s < J; s++)
#pragma unroll
                for (int w = 0; w < NW; w++) stk[s][w] = (h == (uint32_t)s) ? node[w] : stk[s][w];
        }
    }
    // cross-lane reduction: level l holds WG >> l nodes, node x = H(2x, 2x+1)
#pragma unroll
    for (int w = 0; w < NW; w++) lds[0][tid][w] = node[w];
#pragma unroll 1
    for (int l = 1; l <= LOGL; l++) {
        __syncthreads();
        const int src = (l - 1) & 1, dst = l & 1;
        // whole waves: lanes past the level's nodes repeat them
        if (tid < max_int(WG >> l, 64)) {
            const int i = tid & ((WG >> l) - 1);
            const uint32_t tau = i >> (LOGL - l);
            const uint32_t x = part * (L >> l) + (i & ((L >> l) - 1));
            const uint32_t g2 = blk * TPW + tau;
            bool last = false;  // this lane stored its request's last root
            const bool act2 = g2 < A.n_req * P::k;
            const uint32_t req2 = act2 ? g2 / P::k : 0, t2 = act2 ? g2 % P::k : 0;
            const Plan& p2 = A.plan[req2];
            Key k2;
            Hh::load_key(p2, k2);
            uint32_t lft[NW], rgt[NW], out[NW];
#pragma unroll
            for (int w = 0; w < NW; w++) {
                lft[w] = lds[src][2 * i][w];
                rgt[w] = lds[src][2 * i + 1][w];
            }
            const uint32_t hgt = J + l;
            Adr a2 = adr_make(0, p2.tree, kForsTree);
            adr_keypair<P::th>(a2, p2.leaf);
            adr_node(a2, hgt, ((t2 << P::a) >> hgt) + x);
            Hh::H(k2, a2, lft, rgt, out);
            if (act2 && tid == i) {
#pragma unroll
                for (int w = 0; w < NW; w++) lds[dst][i][w] = out[w];
                uint8_t* rec2 =
                    A.sig + (size_t)req2 * A.sig_stride + P::n + (size_t)t2 * (P::a + 1) * P::n;
                const uint32_t tg = p2.fors_idx[t2];
                if (hgt < (uint32_t)P::a && x == ((tg >> hgt) ^ 1u))
                    store_val<P::hash, NW>(rec2 + P::n + (size_t)hgt * P::n, out);
                if constexpr (FP > 1) {
                    if (l == LOGL) {
                        uint32_t* pr = A.ht_parts + ((size_t)g2 * FP + part) * NW;
#pragma unroll
                        for (int w = 0; w < NW; w++) pr[w] = out[w];
                        last = fors_root_done<P, FP>(A, req2);
                    }
                } else if (hgt == (uint32_t)P::a) {
                    store_val<P::hash, NW>(A.fors_roots + ((size_t)req2 * P::k + t2) * P::n, out);
                    if constexpr (PK) last = fors_root_done<P, 1>(A, req2);
                }
            }
            if (PK && l == LOGL) {
                // wave 0 alone is here (TPW <= 64): the tile's LDS is free
                static_assert(TPW <= 64 && fors_pk_wave_words<P>() <= fors_lds_words<P>(), "");
#pragma unroll 1
                for (uint64_t m = __ballot(last); m; m &= m - 1) {
                    const uint32_t rq = __shfl((int)req2, __ffsll((unsigned long long)m) - 1);
                    if constexpr (FP > 1) {
                        fors_top<P, FP, Hh>(A, rq, (lds_u32*)smem);
                        Keccak16::order();
                    }
                    fors_pk_wave<P>(A, rq, (lds_u32*)smem);
                }
            }
        }
    }
}

template <class P, int J, bool PK, bool PH = true>
__global__ void __launch_bounds__(256) k_fors(BatchArgs A) {
    __shared__ __align__(16) uint32_t smem[fors_lds_words<P>()];
    fors_tile<P, J, PK, PH>(A, blockIdx.x, smem);
}

// thash (SHA-256) over M payload words after the 22-byte address,
// thash_sha256.cu:16-34: one compression per loop step; rd(i) returns payload
// word i (native order) from LDS or global memory.  The words of a block are
// read together (one memory latency per block), and blocks of payload words
// only cost one v_alignbit per word.
template <int NW, int M, class Rd>
__device__ __forceinline__ void thash_sha2_rd(const uint32_t mid[8], const Adr& a, const Rd& rd,
                                              uint32_t out[NW]) {
    constexpr int B = (6 + M + 2 + 15) / 16;             // compression blocks
    constexpr int FT = (M + 5) / 16;                     // first block that is not payload only
    constexpr uint32_t bits = (64u + 22u + 4u * M) * 8u;
    static_assert(FT >= 1 && FT < B, "a head, payload and tail blocks");
    uint32_t st[8];
#pragma unroll
    for (int i = 0; i < 8; i++) st[i] = mid[i];
#pragma unroll 1
    for (int blk = 0; blk < B; blk++) {
        uint32_t w[16], x[17];
        if (blk == 0) {
#pragma unroll
            for (int j = 0; j < 11; j++) x[j] = rd(j);
#pragma unroll
            for (int i = 0; i < 16; i++)
                w[i] = i < 5 ? a.w[i < 5 ? i : 0]
                     : i == 5 ? (a.w[5] | (x[0] >> 16))
                              : __builtin_amdgcn_alignbit(x[i - 6 > 0 ? i - 6 : 0], x[i - 5], 16);
        } else if (blk < FT) {
            const int base = 16 * blk - 6;
#pragma unroll
            for (int j = 0; j < 17; j++) x[j] = rd(base + j);
#pragma unroll
            for (int i = 0; i < 16; i++) w[i] = __builtin_amdgcn_alignbit(x[i], x[i + 1], 16);
        } else {
#pragma unroll
            for (int tb = FT; tb < B; tb++) {
                if (blk == tb) {
#pragma unroll
                    for (int j = 0; j < 17; j++) {
                        const int k = 16 * tb - 6 + j;
                        x[j] = rd(k < M ? k : M - 1);
                    }
#pragma unroll
                    for (int i = 0; i < 16; i++) {
                        const int g = 16 * tb + i;
                        uint32_t y = 0;
                        if (g < 5 + M) y = __builtin_amdgcn_alignbit(x[i], x[i + 1], 16);
                        else if (g == 5 + M) y = (x[i] << 16) | 0x8000u;
                        else if (g == 16 * B - 1) y = bits;
                        w[i] = y;
                    }
                }
            }
        }
        sha256_compress_ph<0>(st, w);
    }
#pragma unroll
    for (int i = 0; i < NW; i++) out[i] = st[i];
}

// thash_sha2_rd on a lane pair (both lanes active with the same mid, a and
// payload; sha256_compress_pair): rd2(j) returns payload word j + (lane & 1)
// clamped to 0..M-1, so each lane reads the words of its own half of every
// block.  The steps are separate so that a caller can feed the payload-only
// blocks from precomputed K + W (sha256_rounds_pair_kw).
template <int NW, int M>
struct Sha2Pair {
    static constexpr int B = (6 + M + 2 + 15) / 16;  // compression blocks
    static constexpr int FT = (M + 5) / 16;          // first block that is not payload only
    static constexpr uint32_t bits = (64u + 22u + 4u * M) * 8u;

    __device__ static __forceinline__ uint32_t mask() { return (threadIdx.x & 1u) ? ~0u : 0u; }

    // chaining value halves: e..h (even lane), a..d (odd lane)
    __device__ static __forceinline__ void init(const uint32_t mid[8], uint32_t st[4]) {
        const uint32_t m = mask();
#pragma unroll
        for (int i = 0; i < 4; i++) st[i] = lane_sel(m, mid[i], mid[4 + i]);
    }
    // word pairs of block tb (a constant once unrolled): word g = 16 tb + i is
    // address, payload re-aligned by 2 bytes (lo / hi = this lane's payload
    // words g - 6 and g - 5), the 0x80 pad, zero or the bit length
    template <class Rd2>
    __device__ static __forceinline__ void block(int tb, const Adr& a, const Rd2& rd2, uint32_t v[8]) {
        const uint32_t m = mask();
#pragma unroll
        for (int k = 0; k < 8; k++) {
            const uint32_t lo = rd2(16 * tb - 6 + 2 * k), hi = rd2(16 * tb - 5 + 2 * k);
            uint32_t y[2];
#pragma unroll
            for (int p = 0; p < 2; p++) {
                const int g = 16 * tb + 2 * k + p;
                y[p] = g < 5        ? a.w[g < 5 ? g : 0]
                     : g == 5       ? (a.w[5] | (lo >> 16))
                     : g < 5 + M    ? __builtin_amdgcn_alignbit(lo, hi, 16)
                     : g == 5 + M   ? ((lo << 16) | 0x8000u)
                     : g == 16 * B - 1 ? bits : 0u;
            }
            v[k] = lane_sel(m, y[1], y[0]);
        }
    }
    // payload-only block blk (runtime): this lane's word pairs
    template <class Rd2>
    __device__ static __forceinline__ void payload(int blk, const Rd2& rd2, uint32_t v[8]) {
        const int base = 16 * blk - 6;
#pragma unroll
        for (int k = 0; k < 8; k++)
            v[k] = __builtin_amdgcn_alignbit(rd2(base + 2 * k), rd2(base + 2 * k + 1), 16);
    }
    // blocks from..to-1
    template <class Rd2>
    __device__ static __forceinline__ void absorb(uint32_t st[4], int from, int to, const Adr& a,
                                                  const Rd2& rd2) {
#pragma unroll 1
        for (int blk = from; blk < to; blk++) {
            uint32_t v[8];
            if (blk == 0) {
                block(0, a, rd2, v);
            } else if (blk < FT) {
                payload(blk, rd2, v);
            } else {
#pragma unroll
                for (int tb = 1; tb < B; tb++)
                    if (tb >= FT && blk == tb) block(tb, a, rd2, v);
            }
            sha256_compress_pair(st, v);
        }
    }
    // a..d are on the odd lane, e..h on the even one; the output in both
    __device__ static __forceinline__ void output(const uint32_t st[4], uint32_t out[NW]) {
        const uint32_t m = mask();
#pragma unroll
        for (int w = 0; w < NW; w++) {
            const uint32_t own = st[w & 3], other = pair_swap(st[w & 3]);
            out[w] = w < 4 ? lane_sel(m, own, other) : lane_sel(m, other, own);
        }
    }
};

// the whole thash on a lane pair; the output is in both lanes
template <int NW, int M, class Rd2>
__device__ __forceinline__ void thash_sha2_pair(const uint32_t mid[8], const Adr& a, const Rd2& rd2,
                                                uint32_t out[NW]) {
    using SP = Sha2Pair<NW, M>;
    uint32_t st[4];
    SP::init(mid, st);
    SP::absorb(st, 0, SP::B, a, rd2);
    SP::output(st, out);
}

// K[t] + W[t] (t = 0..63) of compression block b (any of Sha2Pair's, b may
// differ from lane to lane) on one lane: a block's message schedule does not
// depend on the chaining value, so lanes that would idle run it ahead of the
// pair that compresses (sha256_rounds_pair_kw).  rd(i): payload word i.
// kw: 16-byte aligned LDS.
template <int NW, int M, class Rd>
__device__ __forceinline__ void sha2_kw_block(const Adr& a, const Rd& rd, int b, lds_u32* kw) {
    using SP = Sha2Pair<NW, M>;
    uint32_t w[16], x[17];
    const int base = 16 * b - 6;
#pragma unroll
    for (int j = 0; j < 17; j++) {
        const int i = base + j;
        x[j] = rd(i < 0 ? 0 : i < M ? i : M - 1);
    }
#pragma unroll
    for (int i = 0; i < 16; i++) {
        uint32_t y = __builtin_amdgcn_alignbit(x[i], x[i + 1], 16);
        if (i < 5) y = b == 0 ? a.w[i < 5 ? i : 0] : y;
        if (i == 5) y = b == 0 ? (a.w[5] | (x[6] >> 16)) : y;
        if (b >= SP::FT) {
            const int g = 16 * b + i;
            y = g < 5 + M ? y : g == 5 + M ? ((x[i] << 16) | 0x8000u) : 0u;
            if (i == 15) y = b == SP::B - 1 ? SP::bits : y;
        }
        w[i] = y;
    }
    lds_u32x4* out = (lds_u32x4*)kw;
#pragma unroll
    for (int q = 0; q < 16; q++) {
        uint32_t o[4];
#pragma unroll
        for (int j = 0; j < 4; j++) {
            const int t = 4 * q + j;
            if (t >= 16)
                w[t & 15] = sha256_s1(w[(t - 2) & 15]) + w[(t - 7) & 15] +
                            sha256_s0(w[(t - 15) & 15]) + w[t & 15];
            o[j] = kSha256K[t] + w[t & 15];
        }
        out[q] = u32x4{o[0], o[1], o[2], o[3]};
    }
}

// SHAKE256 thash over M payload words (thash_shake256.cu:15-25: pub_seed ||
// addr32 || payload), 136 bytes per permutation; rd(i) returns payload word
// i, bit-interleaved, read a block at a time.  The output is a plain value.
template <class P, int M, class Rd>
__device__ __forceinline__ void thash_shake_rd(const typename Shake<P::n>::Key& key, const Adr& a,
                                               const Rd& rd, uint32_t out[P::nw]) {
    using Hh = Shake<P::n>;
    constexpr int NW = P::nw;
    constexpr int T = NW + 8 + M;             // absorbed words
    constexpr int NB = T / 34 + 1;            // permutations (the pad always fits)
    constexpr int TAIL = T - 34 * (NB - 1);   // words in the last block: the 0x1F byte follows
    static_assert(NB >= 2, "at least two blocks");
    typename Hh::ChainIl c;  // pub_seed || address
    Hh::chain_il_begin(key, a, c);
    uint32_t s[50];
#pragma unroll
    for (int i = 0; i < 50; i++) s[i] = 0;
#pragma unroll 1
    for (int blk = 0; blk < NB; blk++) {
        if (blk == 0) {
            uint32_t x[34 - NW - 8];
#pragma unroll
            for (int j = 0; j < 34 - NW - 8; j++) x[j] = rd(j);
#pragma unroll
            for (int i = 0; i < 34; i++) s[i] ^= i < NW + 8 ? c.w[i < NW + 8 ? i : 0] : x[i - NW - 8];
        } else if (blk < NB - 1) {
            const int base = 34 * blk - NW - 8;
            uint32_t x[34];
#pragma unroll
            for (int j = 0; j < 34; j++) x[j] = rd(base + j);
#pragma unroll
            for (int i = 0; i < 34; i++) s[i] ^= x[i];
        } else {
            constexpr int base = 34 * (NB - 1) - NW - 8;
            uint32_t x[TAIL > 0 ? TAIL : 1];
#pragma unroll
            for (int j = 0; j < TAIL; j++) x[j] = rd(base + j);
#pragma unroll
            for (int i = 0; i < TAIL; i++) s[i] ^= x[i];
            if constexpr ((TAIL & 1) == 0) {  // 0x1F at bit 0 of lane TAIL / 2
                s[TAIL] ^= 7u;
                s[TAIL + 1] ^= 3u;
            } else {                                  // 0x1F at bit 32 of lane TAIL / 2
                s[TAIL - 1] ^= 7u << 16;
                s[TAIL] ^= 3u << 16;
            }
            s[33] ^= 0x80000000u;  // 0x80 at byte 135 (lane 16, bit 63: odd, so the same word)
        }
        keccak_f_il<false>(s);
    }
    Hh::from_il(s, out);
}

// SHAKE256 thash on a lane pair in the interleaved domain (both lanes
// active, same key, address and payload; keccak_f_il_pair): rd2(j), j even,
// returns interleaved payload word j + (lane & 1), clamped to 0..M-1, i.e.
// this lane's half of payload lane j / 2.  The output (plain) is in both
// lanes.
template <class P, int M, class Rd2>
__device__ __forceinline__ void thash_shake_pair(const typename Shake<P::n>::Key& key,
                                                 const Adr& a, const Rd2& rd2,
                                                 uint32_t out[P::nw]) {
    using Hh = Shake<P::n>;
    constexpr int NW = P::nw;
    constexpr int PRE = NW + 8;                // pub_seed || address, interleaved words
    constexpr int T = PRE + M;                 // absorbed words
    constexpr int NB = T / 34 + 1;             // permutations (the pad always fits)
    constexpr int TAIL = T - 34 * (NB - 1);    // words in the last block
    static_assert((PRE & 1) == 0, "the prefix fills whole lanes");
    const bool odd = threadIdx.x & 1u;
    const uint32_t m = odd ? ~0u : 0u;
    typename Hh::ChainIl c;
    Hh::chain_il_begin(key, a, c);
    uint32_t s[25];
#pragma unroll
    for (int i = 0; i < 25; i++) s[i] = 0;
    // interleaved word w of the last block: the 0x1F pad (byte 4 TAIL) and
    // 0x80 (byte 135) in their interleaved bits
    auto pad = [](int w) -> uint32_t {
        uint32_t v = 0;
        if ((TAIL & 1) == 0) v ^= w == TAIL ? 7u : w == TAIL + 1 ? 3u : 0u;
        else v ^= w == TAIL - 1 ? 7u << 16 : w == TAIL ? 3u << 16 : 0u;
        return v ^ (w == 33 ? 0x80000000u : 0u);
    };
    // block tb (a constant once unrolled): stream word g = 34 tb + 2 L + half
    // is prefix, payload (this lane's half from rd2), zero, and the pad in
    // the last block
    auto block = [&](int tb) {
#pragma unroll
        for (int L = 0; L < 17; L++) {
            const int g0 = 34 * tb + 2 * L;
            const uint32_t x = (g0 >= PRE && g0 < T) ? rd2(g0 - PRE) : 0u;
            uint32_t y[2];
#pragma unroll
            for (int p = 0; p < 2; p++) {
                const int g = g0 + p;
                uint32_t v = g < PRE ? c.w[g < PRE ? g : 0] : g < T ? x : 0u;
                if (tb == NB - 1) v ^= pad(g - 34 * (NB - 1));
                y[p] = v;
            }
            s[L] ^= lane_sel(m, y[1], y[0]);
        }
    };
#pragma unroll 1
    for (int blk = 0; blk < NB; blk++) {
        if (blk == 0) {
            block(0);
        } else if (blk < NB - 1) {  // payload only
            const int base = 34 * blk - PRE;
#pragma unroll
            for (int L = 0; L < 17; L++) s[L] ^= rd2(base + 2 * L);
        } else {
            block(NB - 1);
        }
        keccak_f_il_pair(s);
    }
    uint32_t il[NW];
#pragma unroll
    for (int L = 0; L < NW / 2; L++) {
        const uint32_t other = pair_swap(s[L]);
        il[2 * L] = lane_sel(m, other, s[L]);
        il[2 * L + 1] = lane_sel(m, s[L], other);
    }
    Hh::from_il(il, out);
}

// SHAKE256 thash on a row of lanes (K: Keccak16, Keccak32) over a stream held
// in LDS as interleaved words: pub_seed || address (PRE words) || M payload words ||
// pad, in whole rate blocks.  The caller fills the payload; every lane of the
// row calls these.
template <class P, int M>
struct ThashRow {
    using Hh = Shake<P::n>;
    static constexpr int NW = P::nw;
    static constexpr int PRE = NW + 8;
    static constexpr int T = PRE + M;
    static constexpr int NB = T / 34 + 1;  // permutations (the pad always fits)
    static constexpr int kWords = 34 * NB;
    static_assert(PRE % 2 == 0 && M % 2 == 0, "whole 64-bit lanes");

    // pub_seed and the pad, which stay for every hash of one key
    template <class K>
    __device__ static __forceinline__ void begin(const K& k, const uint32_t pub[NW],
                                                 lds_u32* buf) {
#pragma unroll
        for (int l = 0; l < NW / 2; l++)
            buf[2 * l + k.half] = k.split(pub[2 * l], pub[2 * l + 1]);
        buf[PRE - 2 + k.half] = 0;  // address bytes 24..31
        // 0x1F at the payload's end, 0x80 at the block's last byte
        for (int i = T + (threadIdx.x & (K::kLanes - 1)); i < kWords; i += K::kLanes)
            buf[i] = (i == T ? 7u : i == T + 1 ? 3u : 0u) ^ (i == kWords - 1 ? 0x80000000u : 0u);
    }
    template <class K>
    __device__ static __forceinline__ void address(const K& k, const Adr& a, lds_u32* buf) {
#pragma unroll
        for (int l = 0; l < 3; l++)
            buf[NW + 2 * l + k.half] = k.split(Hh::aw(a, 2 * l), Hh::aw(a, 2 * l + 1));
    }
};
// the sponge over nb blocks of such a stream
template <class K>
__device__ __forceinline__ void sponge_row(K& k, const lds_u32* buf, int nb) {
    k.clear();
    K::order();
#pragma unroll 1
    for (int b = 0; b < nb; b++) {
        k.absorb(buf, b);
        k.permute();
    }
}

// words of a WOTS public key in LDS: native, or the whole T_len stream
template <class P>
__host__ __device__ constexpr int tlen_words() {
    return P::hash == kSha2 ? P::len * P::nw : ThashRow<P, P::len * P::nw>::kWords;
}

// FORS public key of request i: T_k over its k roots (fors.cu:142); the
// roots are read past the caches, as another workgroup may have stored them.
template <class P>
__device__ __forceinline__ uint32_t fors_root_word(const BatchArgs& A, uint32_t i, int u) {
    return __builtin_nontemporal_load(
        reinterpret_cast<const uint32_t*>(A.fors_roots + (size_t)i * P::k * P::n) + u);
}
template <class P>
__device__ __forceinline__ Adr fors_pk_adr(const Plan& pl) {
    Adr adr = adr_make(0, pl.tree, kForsPk);
    adr_keypair<P::th>(adr, pl.leaf);
    return adr;
}
// SHAKE256 on a row of lanes; row: fors_pk_row words of LDS
template <class P>
__host__ __device__ constexpr int fors_pk_row() {
    return Keccak16::row_words(Keccak16::kLdsWords + ThashRow<P, P::k * P::nw>::kWords);
}
template <class P, class K>
__device__ __forceinline__ void fors_pk_rows(const BatchArgs& A, uint32_t i, lds_u32* row,
                                           uint32_t out[P::nw]) {
    constexpr int NW = P::nw, KW = P::k * NW;
    using T16 = ThashRow<P, KW>;
    const Plan& pl = A.plan[i];
    typename HashT<P>::Key key;
    HashT<P>::load_key(pl, key);
    K k;
    k.init(row);
    lds_u32* buf = row + K::kLdsWords;
    T16::begin(k, key.pub, buf);
    T16::address(k, fors_pk_adr<P>(pl), buf);
    for (int l = threadIdx.x & (K::kLanes - 1); l < KW / 2; l += K::kLanes) {
        uint32_t e, o;
        il_to(fors_root_word<P>(A, i, 2 * l), fors_root_word<P>(A, i, 2 * l + 1), e, o);
        buf[T16::PRE + 2 * l] = e;
        buf[T16::PRE + 2 * l + 1] = o;
    }
    sponge_row(k, buf, T16::NB);
#pragma unroll
    for (int l = 0; l < NW / 2; l++) k.lane(l, out[2 * l], out[2 * l + 1]);
}
// a whole wave on one request, for latency: SHA-256 with the schedules of
// T_k's blocks on one lane each, then their rounds on the pairs (all alike);
// SHAKE256 on the rows of 32 lanes (all alike).  lds: fors_pk_wave_words
// words of the wave's own.  The value is in every lane.
template <class P>
__host__ __device__ constexpr int fors_pk_wave_words() {
    return P::hash == kSha2 ? Sha2Pair<P::nw, P::k * P::nw>::B * 68 + kKwOnes : fors_pk_row<P>();
}
template <class P>
__device__ __forceinline__ void fors_pk_value(const BatchArgs& A, uint32_t i, lds_u32* lds,
                                              uint32_t out[P::nw]) {
    using Hh = HashT<P>;
    constexpr int NW = P::nw, KW = P::k * NW;
    const int lane = threadIdx.x & 63;
    if constexpr (P::hash == kSha2) {
        using SP = Sha2Pair<NW, KW>;
        const Plan& pl = A.plan[i];
        typename Hh::Key key;
        Hh::load_key(pl, key);
        lds_u32* ones = lds + SP::B * 68;
        ones[lane] = 1u;
        if (lane < SP::B)
            sha2_kw_block<NW, KW>(fors_pk_adr<P>(pl),
                                  [&](int u) { return bswap32(fors_root_word<P>(A, i, u)); }, lane,
                                  lds + 68 * lane);
        Keccak16::order();
        uint32_t st[4];
        SP::init(key.mid, st);
#pragma unroll 1
        for (int b = 0; b < SP::B; b++)
            sha256_rounds_pair_kw(st, (lane & 1) ? ones : lds + 68 * b);
        Keccak16::order();
        SP::output(st, out);
    } else {
        fors_pk_rows<P, Keccak32>(A, i, lds, out);
    }
}
template <class P>
__device__ __forceinline__ void fors_pk_wave(const BatchArgs& A, uint32_t i, lds_u32* lds) {
    uint32_t out[P::nw];
    fors_pk_value<P>(A, i, lds, out);
    if ((threadIdx.x & 63) == 0)
        store_val<P::hash, P::nw>(A.fors_pk + (size_t)i * P::n, out);
}

// FORS public keys of a whole batch (large sign batches and verify): a wave
// per request up to kForsPkWaves requests, else a lane group (SHA-256: a
// pair, SHAKE256: 16 lanes).
constexpr uint32_t kForsPkWaves = 1024;  // a wave per SIMD
template <class P>
__host__ __device__ constexpr uint32_t fors_pk_lanes() { return P::hash == kSha2 ? 2 : 16; }
template <class P, bool WAVE>
__global__ void __launch_bounds__(64) k_fors_pk(BatchArgs A) {
    constexpr int NW = P::nw, KW = P::k * NW;
    if constexpr (WAVE) {
        __shared__ __align__(16) uint32_t lds[fors_pk_wave_words<P>()];
        fors_pk_wave<P>(A, blockIdx.x, (lds_u32*)lds);
    } else {
        const uint32_t i0 = (blockIdx.x * blockDim.x + threadIdx.x) / fors_pk_lanes<P>();
        const uint32_t i = i0 < A.n_req ? i0 : A.n_req - 1;
        uint32_t out[NW];
        if constexpr (P::hash == kSha2) {
            const Plan& pl = A.plan[i];
            typename HashT<P>::Key key;
            HashT<P>::load_key(pl, key);
            const int h = threadIdx.x & 1;
            thash_sha2_pair<NW, KW>(key.mid, fors_pk_adr<P>(pl), [&](int j) {
                const int u = j + h;
                return bswap32(fors_root_word<P>(A, i, u < 0 ? 0 : u < KW ? u : KW - 1));
            }, out);
        } else {
            __shared__ __align__(16) uint32_t row_s[4 * fors_pk_row<P>()];
            fors_pk_rows<P, Keccak16>(A, i, (lds_u32*)row_s + threadIdx.x / 16 * fors_pk_row<P>(), out);
        }
        if (i0 == i && threadIdx.x % fors_pk_lanes<P>() == 0)
            store_val<P::hash, NW>(A.fors_pk + (size_t)i * P::n, out);
    }
}
template <class P>
inline void launch_fors_pk(const BatchArgs& A, uint32_t n, hipStream_t s) {
    if (n <= kForsPkWaves)
        hipLaunchKernelGGL((k_fors_pk<P, true>), dim3(n), dim3(64), 0, s, A);
    else
        hipLaunchKernelGGL((k_fors_pk<P, false>),
                           dim3((uint32_t)(((uint64_t)fors_pk_lanes<P>() * n + 63) / 64)),
                           dim3(64), 0, s, A);
}

// verify: one FORS tree per lane: leaf from the revealed sk, climb with the
// auth path (fors_pk_from_sig, fors.cu:596-633; compute_root utils.cu:94-135)
template <class P, bool PH>
__device__ __forceinline__ void vfors_lane(const BatchArgs& A, uint32_t g0) {
    using Hh = HashPh<P, PH>;
    using Key = typename Hh::Key;
    constexpr int NW = P::nw;
    const uint32_t g = g0 < A.n_req * P::k ? g0 : A.n_req * P::k - 1;  // repeated past the end
    const uint32_t req = g / P::k, t = g % P::k;
    const Plan& pl = A.plan[req];
    Key key;
    Hh::load_key(pl, key);
    const uint8_t* rec = A.sig + (size_t)req * A.sig_stride + P::n + (size_t)t * (P::a + 1) * P::n;
    uint32_t li = pl.fors_idx[t];
    uint32_t off = t << P::a;
    Adr adr = adr_make(0, pl.tree, kForsTree);
    adr_keypair<P::th>(adr, pl.leaf);
    adr_node(adr, 0, li + off);
    uint32_t sk[NW], node[NW];
    load_val<P::hash, NW>(rec, sk);
    Hh::F(key, adr, sk, node);
#pragma unroll 1
    for (int h = 0; h < P::a; h++) {
        uint32_t ap[NW];
        load_val<P::hash, NW>(rec + P::n + (size_t)h * P::n, ap);
        const bool odd = li & 1u;
        li >>= 1;
        off >>= 1;
        adr_node(adr, h + 1, li + off);
        uint32_t l[NW], r[NW];
#pragma unroll
        for (int w = 0; w < NW; w++) {
            l[w] = odd ? ap[w] : node[w];
            r[w] = odd ? node[w] : ap[w];
        }
        Hh::H(key, adr, l, r, node);
    }
    store_val<P::hash, NW>(A.fors_roots + (size_t)g * P::n, node);
}
template <class P, bool PH>
__global__ void __launch_bounds__(64) k_vfors(BatchArgs A) {
    vfors_lane<P, PH>(A, blockIdx.x * 64 + threadIdx.x);
}

// ------------------------------------------------------------- hypertree

// WOTS chain lengths of an n-byte message (wots.cu:84-162): nibbles MSB
// first, then the 3-nibble checksum (sum of 15 - d_i, shifted left by 4)
template <class P>
__device__ __forceinline__ uint32_t chain_len(const uint32_t msg[P::nw], int j) {
    if (j < P::len1) {
        const uint32_t byte = val_byte<P::hash>(msg, j >> 1);
        return (j & 1) ? (byte & 15u) : (byte >> 4);
    }
    uint32_t csum = 0;
#pragma unroll
    for (int i = 0; i < P::n; i++) {
        const uint32_t byte = val_byte<P::hash>(msg, i);
        csum += 30u - (byte >> 4) - (byte & 15u);
    }
    const uint32_t v = csum << 4;  // 16-bit field, digits are its top 12 bits
    const int c = j - P::len1;
    return (v >> (12 - 4 * c)) & 15u;
}

// tree index of hypertree layer `layer`: the reference shifts by h' once per
// layer (sign.cu:1987-1988), so a total shift of 64 bits (256f, layer 16)
// yields 0 -- a single 64-bit shift by 64 would be undefined
template <class P>
__device__ __forceinline__ uint64_t layer_tree(uint64_t tree, uint32_t layer) {
    const uint32_t sh = layer * P::th;
    return sh >= 64 ? 0ull : (tree >> sh);
}

// a chain value into the capture, as signature bytes for SHA-256 and
// bit-interleaved for SHAKE256, in 16-byte (n = 24: 8-byte) stores
template <class P>
__device__ __forceinline__ void store_raw(uint8_t* p, const uint32_t v[P::nw]) {
    if constexpr (P::nw % 4 == 0) {
#pragma unroll
        for (int k = 0; k < P::nw / 4; k++)
            reinterpret_cast<uint4*>(p)[k] =
                make_uint4(to_native<P::hash>(v[4 * k]), to_native<P::hash>(v[4 * k + 1]),
                           to_native<P::hash>(v[4 * k + 2]), to_native<P::hash>(v[4 * k + 3]));
    } else {
#pragma unroll
        for (int k = 0; k < P::nw / 2; k++)
            reinterpret_cast<uint2*>(p)[k] =
                make_uint2(to_native<P::hash>(v[2 * k]), to_native<P::hash>(v[2 * k + 1]));
    }
}

// One Merkle node of a hypertree subtree (treehash, utils.cu:189-241): node x
// of level l = H(left, right) under the subtree's HASHTREE address; writes the
// node into the signature's auth path when it is the sibling of the signing
// leaf's ancestor, and the subtree root (sign: roots[], keygen: pk / sk).
template <class P, int MODE>
__device__ __forceinline__ void ht_node(const BatchArgs& A, uint32_t g, uint32_t ntrees, int l,
                                        uint32_t x, const uint32_t lft[P::nw],
                                        const uint32_t rgt[P::nw], uint32_t out[P::nw],
                                        bool store) {
    using Hh = HashT<P>;
    constexpr int NW = P::nw;
    constexpr int L = 1 << P::th;
    const bool act = g < ntrees;
    const uint32_t req = act ? (MODE == 0 ? g / P::d : g) : 0;
    const uint32_t lay = MODE == 0 ? (act ? g % P::d : 0) : P::d - 1;
    const Plan& pl = A.plan[req];
    typename Hh::Key key;
    Hh::load_key(pl, key);
    uint64_t tree = 0;
    uint32_t target = 0;
    if (MODE == 0) {
        tree = layer_tree<P>(pl.tree, lay);
        target = lay == 0 ? pl.leaf : (uint32_t)((pl.tree >> ((lay - 1) * P::th)) & (L - 1));
    }
    Adr ha = adr_make(lay, tree, kHashTree);
    adr_node(ha, l, x);
    Hh::H(key, ha, lft, rgt, out);
    if (!act || !store) return;
    if (MODE == 0) {
        uint8_t* a2 = A.sig + (size_t)req * A.sig_stride + P::n + P::fors_bytes +
                      (size_t)lay * P::layer_bytes + P::wots_bytes;
        if (l < P::th && x == ((target >> l) ^ 1u)) store_val<P::hash, NW>(a2 + (size_t)l * P::n, out);
        if (l == P::th) store_val<P::hash, NW>(A.roots + ((size_t)req * P::d + lay) * P::n, out);
    } else if (l == P::th) {
        store_val<P::hash, NW>(A.sk_out + (size_t)req * P::sk_bytes + 3 * P::n, out);
        store_val<P::hash, NW>(A.pk_out + (size_t)req * P::pk_bytes + P::n, out);
    }
}

// WOTS chains of the hypertree leaves.  MODE 0 = sign: every (request, layer)
// subtree, the chain values of the signing leaf captured.  MODE 1 = keygen:
// the top subtree only.
//
// One lane per chain: wave `wave` runs chain j = wave % len of the 64 leaves
// of block wave / len, PRF and 15 F, and parks the chain's end in tl_buf
// ([word][leaf], coalesced; SHAKE256 values bit-interleaved).  Bound by VALU
// issue.  A lane holds one chain and no T_len state, so SHA-256 runs 8 waves
// per SIMD (64 VGPRs), where the two-phase rounds issue best; and a batch of
// any size splits into len x as many equal items as it has leaves.  (Before:
// S = 1..16 lanes per leaf, each walking len / S chains, T_len streamed in
// registers at S = 1.)
template <class P>
__host__ __device__ constexpr uint32_t leaf_count(uint32_t trees) {
    return trees << P::th;
}
template <class P>
__host__ __device__ constexpr uint32_t chain_waves(uint32_t trees) {
    return (leaf_count<P>(trees) + 63) / 64 * P::len;
}

template <class P, int MODE, bool PH = true>
__device__ __forceinline__ void chain_wave(const BatchArgs& A, uint32_t wave) {
    using Hh = HashPh<P, PH>;
    constexpr int NW = P::nw;
    constexpr int L = 1 << P::th;
    const uint32_t ntrees = MODE == 0 ? A.n_req * P::d : A.n_req;
    const uint32_t j = wave % P::len;
    const uint32_t leaf_0 = wave / P::len * 64 + (threadIdx.x & 63u);
    const uint32_t nleaf = leaf_count<P>(ntrees);
    const bool own = leaf_0 < nleaf;
    const uint32_t leaf_g = own ? leaf_0 : nleaf - 1;  // column in tl_buf
    const uint32_t g = leaf_g / L, u = leaf_g % L;  // subtree; leaf index = keypair address
    const uint32_t req = MODE == 0 ? g / P::d : g;
    const uint32_t layer = MODE == 0 ? g % P::d : P::d - 1;
    const Plan& pl = A.plan[req];
    typename Hh::Key key;
    Hh::load_key(pl, key);
    uint64_t tree = 0;
    uint32_t target = ~0u;
    if (MODE == 0) {
        tree = layer_tree<P>(pl.tree, layer);
        target = layer == 0 ? pl.leaf
                            : (uint32_t)((pl.tree >> ((layer - 1) * P::th)) & (L - 1));
    }
    const bool capture = MODE == 0 && own && u == target;
    uint8_t* cap = A.cap + (((size_t)req * P::d + layer) * P::len + j) * 16 * P::n;
    Adr wa = adr_make(layer, tree, kWots);
    adr_keypair<P::th>(wa, u);
    adr_chain(wa, j);
    uint32_t v[NW];
    Hh::PRF(key, wa, v);  // wots_gen_sk, wots.cu:27-33
    typename Hh::Chain ch;
    Hh::chain_begin(key, wa, ch);
    if constexpr (P::hash == kShake) {
        // the chain runs bit-interleaved; the capture keeps that form
        // (k_wots_gather converts the values it picks)
        uint32_t t[NW];
        Hh::to_il(v, t);
#pragma unroll
        for (int w = 0; w < NW; w++) v[w] = t[w];
    }
    if (capture) store_raw<P>(cap, v);
#pragma unroll 1
    for (int s = 0; s < P::w - 1; s++) {  // gen_chain(0, w-1), wots.cu:51-62
        Hh::chain_step(key, ch, s, v, v);
        if (capture) store_raw<P>(cap + (s + 1) * P::n, v);
    }
    if (own) {
#pragma unroll
        for (int i = 0; i < NW; i++) A.tl_buf[(size_t)(j * NW + i) * A.tl_lanes + leaf_g] = v[i];
    }
}

template <class P, int MODE, bool PH>
__global__ void __launch_bounds__(256) k_chains(BatchArgs A, uint32_t nwaves) {
    const uint32_t wave = __builtin_amdgcn_readfirstlane(blockIdx.x * 4 + threadIdx.x / 64);
    if (wave < nwaves) chain_wave<P, MODE, PH>(A, wave);
}

// Signing: the FORS tiles of a batch (n_fors workgroups, first: a tile is
// longer than a chain) and its WOTS chains in one launch, so that small
// batches have both in flight together
template <class P, int J, bool PH>
__global__ void __launch_bounds__(256) k_sign_fused(BatchArgs A, uint32_t n_fors, uint32_t nwaves) {
    __shared__ __align__(16) uint32_t smem[fors_lds_words<P>()];
    if (blockIdx.x < n_fors) {
        fors_tile<P, J, true, PH>(A, blockIdx.x, smem);
        return;
    }
    const uint32_t wave =
        __builtin_amdgcn_readfirstlane((blockIdx.x - n_fors) * 4 + threadIdx.x / 64);
    if (wave < nwaves) chain_wave<P, 0, PH>(A, wave);
}

// Hypertree subtrees from the parked chain ends: T_len of every leaf, then
// the Merkle levels in LDS, auth paths and roots.  S lanes per leaf: S = 1
// the most leaves per wave (large batches); S = 2 a lane pair per leaf, which
// shares the serial T_len (sha256_compress_pair / keccak_f_il_pair); S = 16
// the shortest T_len (small batches: SHAKE256 on the 16 lanes, Keccak16;
// SHA-256 with the schedules of 16 blocks at a time on the 16 lanes, then
// their rounds on the first two).
//
// At S = 1 a subtree is one workgroup's (512 lanes for 512 leaves).  With
// more lanes per leaf, a subtree whose lanes exceed 256 is split over PARTS
// workgroups, which costs each of them a device-scope fence: at S = 1, two
// workgroups per subtree took longer than one (SHA2-128s, 256 requests, 819 us
// against 378).  Each part reduces its leaves to a part root in LDS; the part
// that finishes last (device-scope counter, release/acquire fences, no
// waiting) climbs the remaining log2(PARTS) levels from the part roots.
template <class P, int S>
struct HtShape {
    static constexpr int L = 1 << P::th;                 // leaves per subtree
    static constexpr int LT = L * S;                     // lanes per subtree
    static constexpr int WG = S == 1 && L > 256 ? L : 256;  // lanes per workgroup
    static constexpr int PARTS = LT > WG ? LT / WG : 1;
    static constexpr int LP = L / PARTS;                 // leaves per part
    static constexpr int LOGP = P::th - ilog2(PARTS);    // levels reduced inside a part
    static constexpr int TPW = PARTS > 1 ? 1 : WG / LT;  // subtrees per workgroup
    static constexpr int NL = WG / S;                    // leaves per workgroup
    static constexpr int NLDS = NL > PARTS ? NL : PARTS; // the last part climbs from PARTS roots
};

template <class P, int MODE, int S>
__global__ void __launch_bounds__((HtShape<P, S>::WG)) k_ht(BatchArgs A) {
    using Hh = HashT<P>;
    using Key = typename Hh::Key;
    using Sh = HtShape<P, S>;
    constexpr int NW = P::nw;
    constexpr int L = Sh::L, TPW = Sh::TPW, NL = Sh::NL;
    constexpr int PARTS = Sh::PARTS, LP = Sh::LP, LOGP = Sh::LOGP;
    constexpr int LPT = LP * S;  // lanes per subtree in this workgroup
    constexpr int TLW = P::len * NW;
    __shared__ uint32_t lds[2][Sh::NLDS][NW];  // two levels of nodes
    // S = 16, per leaf: SHA-256 16 rows of K + W (68 words each and 16 more
    // per leaf: distinct banks for the lanes' writes and the leaves' reads),
    // SHAKE256 the row's sponge and T_len stream
    constexpr int XW = S < 16            ? 0
                       : P::hash == kSha2 ? 16 * 68 + 16
                                          : Keccak16::row_words(Keccak16::kLdsWords + tlen_words<P>());
    __shared__ __align__(16) uint32_t x_s[XW ? NL * XW : 1];
    __shared__ __align__(16) uint32_t ones_s[XW && P::hash == kSha2 ? kKwOnes : 1];

    const int tid = threadIdx.x;
    if (XW && P::hash == kSha2 && tid < kKwOnes) ones_s[tid] = 1u;
    const uint32_t blk = blockIdx.x;
    const uint32_t part = PARTS > 1 ? blk % PARTS : 0;
    const uint32_t u = part * LP + (tid % LPT) / S;  // leaf index = keypair address
    const int q = tid % S;
    const int slot = tid / S;                         // leaf slot in the workgroup
    const uint32_t g = (blk / PARTS) * TPW + tid / LPT;
    const uint32_t ntrees = MODE == 0 ? A.n_req * P::d : A.n_req;
    const bool active = g < ntrees;
    const uint32_t req = active ? (MODE == 0 ? g / P::d : g) : 0;
    const uint32_t layer = MODE == 0 ? (active ? g % P::d : 0) : P::d - 1;
    const uint32_t leaf_g = active ? g * L + u : 0;   // column in tl_buf
    {
        const Plan& pl = A.plan[req];
        Key key;
        Hh::load_key(pl, key);
        uint64_t tree = 0;
        uint32_t target = 0;
        if (MODE == 0) {
            tree = layer_tree<P>(pl.tree, layer);
            target = layer == 0 ? pl.leaf
                                : (uint32_t)((pl.tree >> ((layer - 1) * P::th)) & (L - 1));
        }
        // ---- T_len of leaf u (wots_gen_leaf, sign.cu:87-104)
        Adr pa = adr_make(layer, tree, kWotsPk);
        adr_keypair<P::th>(pa, u);
        auto parked = [&](int w) { return A.tl_buf[(size_t)w * A.tl_lanes + leaf_g]; };
        auto parked2 = [&](int j) {
            const int i = j + q;
            return parked(i < 0 ? 0 : i < TLW ? i : TLW - 1);
        };
        uint32_t node[NW];
        if constexpr (S == 16 && P::hash == kSha2) {
            using SP = Sha2Pair<NW, TLW>;
            uint32_t* kw = x_s + slot * XW;
            uint32_t st[4];
            SP::init(key.mid, st);
#pragma unroll 1
            for (int b0 = 0; b0 < SP::B; b0 += 16) {
                const int nb = SP::B - b0 < 16 ? SP::B - b0 : 16;
                if (q < nb) sha2_kw_block<NW, TLW>(pa, parked, b0 + q, (lds_u32*)kw + 68 * q);
                __syncthreads();
                // every pair of the leaf's lanes, all alike: with two lanes
                // of 16 active the same rounds took 1-3.5 times as long from
                // launch to launch
#pragma unroll 1
                for (int b = 0; b < nb; b++)
                    sha256_rounds_pair_kw(st, (q & 1) ? &ones_s[0] : kw + 68 * b);
                if (b0 + 16 < SP::B) __syncthreads();
            }
            SP::output(st, node);
        } else if constexpr (S == 16) {
            using TL = ThashRow<P, TLW>;
            Keccak16 k;
            k.init((lds_u32*)x_s + slot * XW);
            lds_u32* buf = (lds_u32*)x_s + slot * XW + Keccak16::kLdsWords;
            TL::begin(k, key.pub, buf);
            TL::address(k, pa, buf);
            uint32_t x[(TLW + 15) / 16];  // one load latency for all
#pragma unroll
            for (int i = 0; i < (TLW + 15) / 16; i++) x[i] = parked(16 * i + q < TLW ? 16 * i + q : 0);
#pragma unroll
            for (int i = 0; i < (TLW + 15) / 16; i++)
                if (16 * i + q < TLW) buf[TL::PRE + 16 * i + q] = x[i];
            sponge_row(k, buf, TL::NB);
#pragma unroll
            for (int l = 0; l < NW / 2; l++) k.lane(l, node[2 * l], node[2 * l + 1]);
        } else if constexpr (P::hash == kSha2) {
            if constexpr (S == 2) thash_sha2_pair<NW, TLW>(key.mid, pa, parked2, node);
            else thash_sha2_rd<NW, TLW>(key.mid, pa, parked, node);
        } else {
            if constexpr (S == 2) thash_shake_pair<P, TLW>(key, pa, parked2, node);
            else thash_shake_rd<P, TLW>(key, pa, parked, node);
        }
        if (q == 0) {
            uint8_t* auth = A.sig + (size_t)req * A.sig_stride + P::n + P::fors_bytes +
                            (size_t)layer * P::layer_bytes + P::wots_bytes;
            if (MODE == 0 && active && u == (target ^ 1u)) store_val<P::hash, NW>(auth, node);
#pragma unroll
            for (int w = 0; w < NW; w++) lds[0][slot][w] = node[w];
        }
    }

    // ---- subtree: level l has NL >> l nodes here, node x = H(2x, 2x+1)
#pragma unroll 1
    for (int l = 1; l <= LOGP; l++) {
        __syncthreads();
        const int src = (l - 1) & 1, dst = l & 1;
        // whole waves: lanes past the level's nodes repeat them
        if (tid < max_int(NL >> l, 64)) {
            const int i = tid & ((NL >> l) - 1);
            const uint32_t t2 = i >> (LOGP - l);
            const uint32_t x = part * (LP >> l) + (i & ((LP >> l) - 1));
            uint32_t lft[NW], rgt[NW];
#pragma unroll
            for (int w = 0; w < NW; w++) {
                lft[w] = lds[src][2 * i][w];
                rgt[w] = lds[src][2 * i + 1][w];
            }
            uint32_t out[NW];
            ht_node<P, MODE>(A, (blk / PARTS) * TPW + t2, ntrees, l, x, lft, rgt, out, tid == i);
            if (tid == i) {
#pragma unroll
                for (int w = 0; w < NW; w++) lds[dst][i][w] = out[w];
            }
        }
    }
    if constexpr (PARTS > 1) {
        // part root -> ht_parts; the last part of the subtree climbs the rest
        __shared__ uint32_t last;
        __syncthreads();
        if (tid == 0) {
            uint32_t* dst = A.ht_parts + ((size_t)g * PARTS + part) * NW;
#pragma unroll
            for (int w = 0; w < NW; w++) dst[w] = lds[LOGP & 1][0][w];
            __threadfence();  // release the part root before counting this part
            last = active ? (atomicAdd(&A.ht_count[g], 1u) == (uint32_t)PARTS - 1) : 0u;
        }
        __syncthreads();
        if (last) {
            __threadfence();  // acquire: every part root is visible
            if (tid < PARTS) {
                const uint32_t* srcp = A.ht_parts + ((size_t)g * PARTS + tid) * NW;
#pragma unroll
                for (int w = 0; w < NW; w++)
                    lds[LOGP & 1][tid][w] = __builtin_nontemporal_load(srcp + w);
            }
#pragma unroll 1
            for (int l = LOGP + 1; l <= P::th; l++) {
                __syncthreads();
                const int src = (l - 1) & 1, dst = l & 1;
                if (tid < 64) {  // at most PARTS / 2 = 16 nodes
                    const int i = tid & ((L >> l) - 1);
                    uint32_t lft[NW], rgt[NW], out[NW];
#pragma unroll
                    for (int w = 0; w < NW; w++) {
                        lft[w] = lds[src][2 * i][w];
                        rgt[w] = lds[src][2 * i + 1][w];
                    }
                    ht_node<P, MODE>(A, g, ntrees, l, i, lft, rgt, out, tid == i);
                    if (tid == i) {
#pragma unroll
                        for (int w = 0; w < NW; w++) lds[dst][i][w] = out[w];
                    }
                }
            }
        }
    }
}

// WOTS signatures: lane per (request, layer, chain); the layer signs the FORS
// public key (layer 0) or the root of the layer below (sign.cu:1970-1989)
template <class P>
__global__ void __launch_bounds__(256) k_wots_gather(BatchArgs A) {
    constexpr int NW = P::nw;
    const uint32_t g = blockIdx.x * blockDim.x + threadIdx.x;
    if (g >= A.n_req * P::d * P::len) return;
    const uint32_t j = g % P::len;
    const uint32_t rl = g / P::len;
    const uint32_t layer = rl % P::d, req = rl / P::d;
    const uint8_t* mp = layer == 0 ? A.fors_pk + (size_t)req * P::n
                                   : A.roots + ((size_t)req * P::d + layer - 1) * P::n;
    uint32_t msg[NW];
    load_val<P::hash, NW>(mp, msg);
    const uint32_t len = chain_len<P>(msg, j);
    // the capture holds n-byte values at multiples of n from a 256-byte
    // aligned base: 16-byte loads (8-byte for n = 24), all before the stores
    // (word-by-word load / store pairs could alias and stayed 4-byte
    // accesses)
    const uint8_t* src = A.cap + ((((size_t)req * P::d + layer) * P::len + j) * 16 + len) * P::n;
    uint8_t* dst = A.sig + (size_t)req * A.sig_stride + P::n + P::fors_bytes +
                   (size_t)layer * P::layer_bytes + (size_t)j * P::n;
    uint32_t v[NW];
    if constexpr (NW % 4 == 0) {
#pragma unroll
        for (int k = 0; k < NW / 4; k++) {
            const uint4 x = reinterpret_cast<const uint4*>(src)[k];
            v[4 * k] = x.x;
            v[4 * k + 1] = x.y;
            v[4 * k + 2] = x.z;
            v[4 * k + 3] = x.w;
        }
    } else {
#pragma unroll
        for (int k = 0; k < NW / 2; k++) {
            const uint2 x = reinterpret_cast<const uint2*>(src)[k];
            v[2 * k] = x.x;
            v[2 * k + 1] = x.y;
        }
    }
    if constexpr (P::hash == kShake) {  // SHAKE chains are captured bit-interleaved
        uint32_t vi[NW];
#pragma unroll
        for (int w = 0; w < NW; w++) vi[w] = v[w];
        Shake<P::n>::from_il(vi, v);
    }
#pragma unroll
    for (int w = 0; w < NW; w++) reinterpret_cast<uint32_t*>(dst)[w] = v[w];
}

// The climb of one layer's subtree on a lane pair (SHA-256; compute_root,
// utils.cu:94-135): node (in both lanes) is the WOTS public key's T_len on
// entry and the layer root on exit; the auth path is in LDS (raw words) and
// nd is NW words of LDS for the node.
template <class P>
__device__ __forceinline__ void climb_pair(const typename HashT<P>::Key& key, uint32_t layer,
                                           uint64_t tree, uint32_t leaf, const uint32_t* auth,
                                           uint32_t* nd, uint32_t node[P::nw]) {
    constexpr int NW = P::nw;
    const int half = threadIdx.x & 1;
    uint32_t li = leaf;
    Adr ha = adr_make(layer, tree, kHashTree);
#pragma unroll 1
    for (int h = 0; h < P::th; h++) {
        const bool right = li & 1u;  // node is the right child
        li >>= 1;
        adr_node(ha, h + 1, li);
        // payload node || auth or auth || node from LDS (nd: the node as raw
        // words, like the auth path)
#pragma unroll
        for (int w = 0; w < NW; w++) nd[w] = bswap32(node[w]);
        const uint32_t* ap = auth + h * NW;
        auto word = [&](int i) {  // payload word i (raw)
            const uint32_t* src = (i < NW) == right ? ap : nd;
            return src[i < NW ? i : i - NW];
        };
        thash_sha2_pair<NW, 2 * NW>(key.mid, ha, [&](int j) {
            int i = j + half;
            i = i < 0 ? 0 : i < 2 * NW ? i : 2 * NW - 1;
            return bswap32(word(i));
        }, node);
    }
}

// reader of a WOTS public key held in LDS for the lane-pair thashes
template <class P>
struct PkPair {
    static constexpr int TLW = P::len * P::nw;
    const uint32_t* pk;
    int half;
    __device__ uint32_t operator()(int j) const {
        const int i = j + half;
        return pk[i < 0 ? 0 : i < TLW ? i : TLW - 1];
    }
};

// Verification of one layer's subtree on a lane pair (SHA-256, both lanes
// active): T_len over the WOTS public key in LDS (pk, native words), then
// climb_pair.  node is the layer root, in both lanes.
template <class P>
__device__ __forceinline__ void tlen_climb_pair(const typename HashT<P>::Key& key,
                                                uint32_t layer, uint64_t tree, uint32_t leaf,
                                                const uint32_t* pk, const uint32_t* auth,
                                                uint32_t* nd, uint32_t node[P::nw]) {
    constexpr int NW = P::nw;
    constexpr int TLW = P::len * NW;
    Adr pa = adr_make(layer, tree, kWotsPk);
    adr_keypair<P::th>(pa, leaf);
    const PkPair<P> rpk{pk, (int)(threadIdx.x & 1)};
    thash_sha2_pair<NW, TLW>(key.mid, pa, rpk, node);
    climb_pair<P>(key, layer, tree, leaf, auth, nd, node);
}

// The same for SHAKE256 on a row of lanes (K: Keccak16, Keccak32), one loop
// over T_len and the th nodes.  pk: the T_len stream (ThashRow<P, len * nw>) with the
// chain ends as payload; nd: the stream of one node; begin() of both has run.
// auth: the auth path, interleaved words.  node is the layer root, plain, in
// every lane.
template <class P>
struct LayerRow {
    using TL = ThashRow<P, P::len * P::nw>;
    using TH = ThashRow<P, 2 * P::nw>;
    static constexpr int NW = P::nw;
    static_assert(TH::NB == 1 && NW <= 8, "a node is one block");

    template <class K>
    __device__ static __forceinline__ void run(K& k, uint32_t layer, uint64_t tree,
                                               uint32_t leaf, lds_u32* pk, const lds_u32* auth,
                                               lds_u32* nd, uint32_t node[NW]) {
        const int p = threadIdx.x & (K::kLanes - 1);
        Adr a = adr_make(layer, tree, kWotsPk);
        adr_keypair<P::th>(a, leaf);
        TL::address(k, a, pk);
        Adr ha = adr_make(layer, tree, kHashTree);
        uint32_t li = leaf;
#pragma unroll 1
        for (int h = 0; h <= P::th; h++) {
            if (h > 0) {
                const bool right = li & 1u;  // node is the right child
                li >>= 1;
                adr_node(ha, h, li);
                TH::address(k, ha, nd);
                lds_u32* own = nd + TH::PRE + (right ? NW : 0);
                lds_u32* sib = nd + TH::PRE + (right ? 0 : NW);
                if (k.col < NW / 2 && K::own0()) own[2 * k.col + k.half] = k.s[0];
                if (p < NW) sib[p] = auth[(h - 1) * NW + p];
            }
            sponge_row(k, h == 0 ? pk : nd, h == 0 ? TL::NB : 1);
        }
#pragma unroll
        for (int l = 0; l < NW / 2; l++) k.lane(l, node[2 * l], node[2 * l + 1]);
    }
};

// verify: the d layers of R = 256 / G requests per workgroup in order
// (sign.cu:3077-3113), so G is the mean number of lanes per request.  Per
// layer the R * len WOTS chains of the workgroup (15 - len_j steps each,
// data dependent) are ranked by remaining steps with a counting sort in LDS
// and dealt to the 256 lanes in snake order: a longest-first schedule that
// evens the per-lane F counts across all requests of the workgroup, not per
// request.  Each lane runs its chains in one flattened loop (one F site;
// SHAKE256 chains run bit-interleaved).  The lane pair 2r, 2r + 1 then
// computes T_len of request r block by block from LDS and climbs its subtree
// (compute_root, utils.cu:94-135; tlen_climb_pair, or for SHA-256 with n <=
// 24 the rounds of T_len's blocks on K + W that all waves computed before);
// SHAKE256 does so on 16 lanes per request (LayerRow).  The next layer's WOTS
// signature words and this layer's auth path are fetched into registers while
// the chains run, so the layer loop waits on no global load.
// CH: how a chain step runs.
//  kVhtLane: on one lane.
//  kVhtPhased (SHA-256): in two-phase rounds, for launches that put two or
//    more workgroups on a CU (SHA2-128f, G = 16: 8192 requests 2.70 -> 2.10
//    ms, 16384 5.19 -> 4.15); with one wave per SIMD the compiler's order
//    stays ahead (4096 requests 1.51 against 1.77 ms).
//  kVhtPair: on a lane pair, where a workgroup holds few requests (G >= 64):
//    the chain phase lasts as long as its longest chain, 15 steps, and a step
//    is 4.2k cycles on a pair against 5.6k on a lane (Keccak 12.9k, 19.7k).
//    300 requests, k_vht: SHA2-128f 1281 -> 1084 us, SHA2-192f 1693 -> 1493,
//    SHAKE256-128f 3067 -> 2338, SHAKE256-256f 3109 -> 2403; two workgroups
//    per CU (2000 requests, G = 64): SHA2-128f 1916 -> 1696, SHAKE256-128f
//    3374 -> 3075.
enum { kVhtLane, kVhtPhased, kVhtPair };
template <class P, int G, int CH>
__global__ void __launch_bounds__(256) k_vht(BatchArgs A) {
    constexpr bool PH = CH == kVhtPhased;
    using Hh = HashT<P>;
    using Key = typename Hh::Key;
    constexpr bool SHA2 = P::hash == kSha2;
    constexpr int NW = P::nw;
    constexpr int LEN = P::len;
    constexpr int TH = P::th;
    constexpr int R = 256 / G;                   // requests per workgroup
    constexpr int TLW = LEN * NW;                // WOTS signature / public key words
    constexpr int NCH = R * LEN;                 // chains per workgroup and layer
    constexpr int MAXC = (NCH + 255) / 256;      // chains per lane
    constexpr int MAXP = (NCH + 127) / 128;      // chains per lane pair (kVhtPair)
    constexpr int MAXW = (R * TLW + 255) / 256;  // prefetched WOTS words per lane
    constexpr int AW = TH * NW;                  // auth path words per request
    constexpr int MAXA = (R * AW + 255) / 256;   // prefetched auth words per lane
    static_assert(NCH < 4096, "chain ids take 12 bits of an order entry");
    // SHA-256 with n <= 24: T_len's blocks take their message schedules from
    // all waves (the LDS for n = 32 would not fit)
    constexpr int MB = Sha2Pair<NW, TLW>::B;  // blocks of T_len
    constexpr bool PRE = SHA2 && NW <= 6;
    __builtin_amdgcn_s_setprio(2);  // d dependent layers per request: latency-bound
    __shared__ uint32_t key_s[R][8];    // SHA-256 midstate / SHAKE256 pub_seed
    __shared__ uint32_t root_s[R][NW];  // root of the last finished layer
    __shared__ uint64_t tree_s[R];
    __shared__ uint32_t leaf_s[R];
    __shared__ uint32_t sig_s[R][TLW];  // WOTS signature of the layer, raw words
    // chain ends: native words, for SHAKE256 the payload of a T_len stream
    // (LayerRow), interleaved
    constexpr int PKW = tlen_words<P>(), PKO = SHA2 ? 0 : NW + 8;
    __shared__ uint32_t pk_s[R][PKW];
    __shared__ uint32_t auth_s[R][AW];  // auth path of the layer, raw / interleaved words
    // climb: the node, raw words (SHAKE256: the stream of one node)
    __shared__ uint32_t node_s[R][SHA2 ? NW : 34];
    // SHAKE256: the rows' sponges
    __shared__ __align__(16) uint32_t row_s[SHA2 ? 1 : R][Keccak16::kLdsWords];
    // K + W of T_len's blocks: 64-word rows, row (r, b) skewed by 4 words per
    // request so the pairs' 16-byte reads of one t (one row per request) fall
    // into distinct bank groups
    __shared__ __align__(16) uint32_t kw_s[PRE ? R * MB * 64 + 64 : 1];
    __shared__ __align__(16) uint32_t ones_s[PRE ? kKwOnes : 1];
    if (PRE && threadIdx.x < kKwOnes) ones_s[threadIdx.x] = 1u;
    auto kw_row = [&](int r, int b) { return &kw_s[(r * MB + b) * 64 + 4 * (r & 15)]; };
    __shared__ uint16_t order_s[NCH];   // rank -> chain id | remaining steps << 12
    __shared__ uint32_t hist_s[16];     // chains per remaining-step count

    const int tid = threadIdx.x;
    const uint32_t req0 = blockIdx.x * R;
    const int nact = (int)min((uint32_t)R, A.n_req - req0);  // >= 1 by the grid
    const int nch = nact * LEN;
    auto sig_of = [&](int r) { return A.sig + (size_t)(req0 + r) * A.sig_stride; };
    auto wots_of = [&](int r, int layer) {
        return reinterpret_cast<const uint32_t*>(sig_of(r) + P::n + P::fors_bytes +
                                                 (size_t)layer * P::layer_bytes);
    };

    if (tid < nact) {
        const Plan& pl = A.plan[req0 + tid];
#pragma unroll
        for (int i = 0; i < 8; i++) key_s[tid][i] = SHA2 ? pl.mid[i] : pl.pubseed[i];
        uint32_t fp[NW];
        load_val<P::hash, NW>(A.fors_pk + (size_t)(req0 + tid) * P::n, fp);
#pragma unroll
        for (int w = 0; w < NW; w++) root_s[tid][w] = fp[w];
        tree_s[tid] = pl.tree;
        leaf_s[tid] = pl.leaf;
    }
    if (tid < 16) hist_s[tid] = 0;
#pragma unroll
    for (int k = 0; k < MAXW; k++) {
        const int u = tid + 256 * k;
        if (u < nact * TLW) sig_s[u / TLW][u % TLW] = wots_of(u / TLW, 0)[u % TLW];
    }
    // SHAKE256: request of this row of 16 lanes; rows past the last request
    // repeat their wave's first one (in step with it, on its LDS)
    const int row0 = tid / 64 * 4;
    const int rr = (tid >> 4) < nact ? tid >> 4 : row0;
    Keccak16 sponge;
    if constexpr (!SHA2) {
        if (row0 < nact) {
            const Plan& pl = A.plan[req0 + rr];
            Key k2;
            Hh::load_key(pl, k2);
            sponge.init((lds_u32*)row_s[rr]);
            LayerRow<P>::TL::begin(sponge, k2.pub, (lds_u32*)pk_s[rr]);
            LayerRow<P>::TH::begin(sponge, k2.pub, (lds_u32*)node_s[rr]);
        }
    }

#pragma unroll 1
    for (int layer = 0; layer < P::d; layer++) {
        __syncthreads();  // roots, tree / leaf, signature words and histogram ready
        // remaining steps of every chain and its slot within its step count
        uint32_t cst[MAXC], cslot[MAXC];
#pragma unroll
        for (int k = 0; k < MAXC; k++) {
            const int q = tid + 256 * k;
            cst[k] = 0;
            cslot[k] = 0;
            if (q < nch) {
                uint32_t msg[NW];
#pragma unroll
                for (int w = 0; w < NW; w++) msg[w] = root_s[q / LEN][w];
                cst[k] = P::w - 1 - chain_len<P>(msg, q % LEN);
                cslot[k] = atomicAdd(&hist_s[15 - cst[k]], 1u);
            }
        }
        __syncthreads();
        // rank = chains with more steps + slot (longest first)
        {
            uint32_t h[16];
#pragma unroll
            for (int b = 0; b < 16; b++) h[b] = hist_s[b];
#pragma unroll
            for (int k = 0; k < MAXC; k++) {
                const int q = tid + 256 * k;
                const uint32_t bk = 15 - cst[k];
                uint32_t start = 0;
#pragma unroll
                for (int b = 0; b < 15; b++) start += (uint32_t)b < bk ? h[b] : 0u;
                if (q < nch) order_s[start + cslot[k]] = (uint16_t)(q | (cst[k] << 12));
            }
        }
        __syncthreads();
        // fetch the next layer's WOTS signature and this layer's auth path
        const bool more = layer + 1 < P::d;
        uint32_t nx[MAXW], au[MAXA];
#pragma unroll
        for (int k = 0; k < MAXW; k++) {
            const int u = tid + 256 * k;
            nx[k] = (more && u < nact * TLW) ? wots_of(u / TLW, layer + 1)[u % TLW] : 0u;
        }
#pragma unroll
        for (int k = 0; k < MAXA; k++) {
            const int u = tid + 256 * k;
            au[k] = u < nact * AW ? wots_of(u / AW, layer)[TLW + u % AW] : 0u;
        }
        if constexpr (CH == kVhtPair) {
            // the same with pair tid / 2 in the place of lane tid
            const int p = tid >> 1;
            int nm = 0;
#pragma unroll
            for (int c = 0; c < MAXP; c++) nm += ((c & 1) ? (c + 1) * 128 - 1 - p : c * 128 + p) < nch;
            int c = 0, r = 0, j = 0;
            uint32_t s = P::w - 1;
            Adr wa{};
            typename Hh::PairChain pc{};
            constexpr int VW = Hh::kPairWords;
            uint32_t v[VW];
#pragma unroll
            for (int w = 0; w < VW; w++) v[w] = 0;
            auto take = [&](int cc) {
                const uint32_t e = order_s[(cc & 1) ? (cc + 1) * 128 - 1 - p : cc * 128 + p];
                const int q = e & 0xFFF;
                r = q / LEN;
                j = q % LEN;
                s = P::w - 1 - (e >> 12);
                wa = adr_make(layer, tree_s[r], kWots);
                adr_keypair<TH>(wa, leaf_s[r]);
                adr_chain(wa, j);
                const uint32_t* sg = &sig_s[r][j * NW];
                Key key;
#pragma unroll
                for (int i = 0; i < NW; i++) key.sk[i] = 0;
                if constexpr (SHA2) {
#pragma unroll
                    for (int w = 0; w < NW; w++) v[w] = bswap32(sg[w]);
#pragma unroll
                    for (int i = 0; i < 8; i++) key.mid[i] = key_s[r][i];
                } else {
#pragma unroll
                    for (int l = 0; l < VW; l++) v[l] = il_half(sg[2 * l], sg[2 * l + 1], tid & 1);
#pragma unroll
                    for (int i = 0; i < NW; i++) key.pub[i] = key_s[r][i];
                }
                Hh::pair_begin(key, wa, pc);
            };
            bool run = nm > 0;
            if (run) take(0);
#pragma unroll 1
            while (true) {
                while (run && s >= (uint32_t)P::w - 1) {
                    uint32_t* out = &pk_s[r][PKO + j * NW];
                    if constexpr (SHA2) {
                        if ((tid & 1) == 0) {
#pragma unroll
                            for (int w = 0; w < NW; w++) out[w] = v[w];
                        }
                    } else {
#pragma unroll
                        for (int l = 0; l < VW; l++) out[2 * l + (tid & 1)] = v[l];
                    }
                    c++;
                    run = c < nm;
                    if (run) take(c);
                }
                if (!__any(run)) break;
                Hh::pair_step(pc, wa, s, v);
                s++;
            }
        } else {
            // walk the chains: ranks tid, 511 - tid, 512 + tid, ... (snake order;
            // the ranks grow with c, so the valid ones are a prefix) in one
            // flattened loop, one F site
            int nm = 0;
#pragma unroll
            for (int c = 0; c < MAXC; c++) nm += ((c & 1) ? (c + 1) * 256 - 1 - tid : c * 256 + tid) < nch;
            int c = 0, r = 0, j = 0;
            uint32_t s = P::w - 1;
            Key key{};
            Adr wa{};
            uint32_t v[NW];
            typename std::conditional<SHA2, int, typename Shake<P::n>::ChainIl>::type ch{};
            uint32_t pre[SHA2 ? 8 : 1] = {};  // SHA-256: the chain's rounds 0-4 (Sha2::F_prefix)
            typename Hh::Chain chn{};         // the same for two-phase rounds
#pragma unroll
            for (int w = 0; w < NW; w++) v[w] = 0;
#pragma unroll
            for (int i = 0; i < NW; i++) key.sk[i] = 0;
            auto take = [&](int cc) {  // start chain cc of this lane (everything from LDS)
                const int rank = (cc & 1) ? (cc + 1) * 256 - 1 - tid : cc * 256 + tid;
                const uint32_t e = order_s[rank];
                const int q = e & 0xFFF;
                r = q / LEN;
                j = q % LEN;
                s = P::w - 1 - (e >> 12);
#pragma unroll
                for (int w = 0; w < NW; w++) v[w] = to_native<P::hash>(sig_s[r][j * NW + w]);
                wa = adr_make(layer, tree_s[r], kWots);
                adr_keypair<TH>(wa, leaf_s[r]);
                adr_chain(wa, j);
                if constexpr (SHA2) {
#pragma unroll
                    for (int i = 0; i < 8; i++) key.mid[i] = key_s[r][i];
                    if constexpr (PH) Hh::chain_begin(key, wa, chn);
                    else Hh::F_prefix(key, wa, pre);
                } else {
#pragma unroll
                    for (int i = 0; i < NW; i++) key.pub[i] = key_s[r][i];
                    Hh::chain_il_begin(key, wa, ch);
                    uint32_t t[NW];
                    Hh::to_il(v, t);
#pragma unroll
                    for (int w = 0; w < NW; w++) v[w] = t[w];
                }
            };
            bool run = nm > 0;
            if (run) take(0);
            // all lanes step until every chain of the wave is done (full waves run
            // fastest); a lane without one steps on a value that nothing reads
#pragma unroll 1
            while (true) {
                while (run && s >= (uint32_t)P::w - 1) {  // chain done: park its end, take the next
#pragma unroll
                    for (int w = 0; w < NW; w++) pk_s[r][PKO + j * NW + w] = v[w];
                    c++;
                    run = c < nm;
                    if (run) take(c);
                }
                if (!__any(run)) break;
                if constexpr (SHA2) {
                    if constexpr (PH) {
                        Hh::chain_step(key, chn, s, v, v);
                    } else {
                        adr_hash(wa, s);
                        Hh::F_step(key, pre, wa, v, v);
                    }
                } else {
                    Hh::F_il(ch, s, v, v);
                }
                s++;
            }
        }
#pragma unroll
        for (int k = 0; k < MAXA; k++) {
            const int u = tid + 256 * k;
            if constexpr (!SHA2) {  // adjacent threads hold the words of one 64-bit lane
                const uint32_t other = pair_swap(au[k]);
                const bool odd = tid & 1;
                au[k] = il_half(odd ? other : au[k], odd ? au[k] : other, tid & 1);
            }
            if (u < nact * AW) auth_s[u / AW][u % AW] = au[k];
        }
        __builtin_amdgcn_s_setprio(2);  // two-phase rounds leave 0
        __syncthreads();  // every chain end parked; this layer's sig_s reads done
#pragma unroll
        for (int k = 0; k < MAXW; k++) {
            const int u = tid + 256 * k;
            if (more && u < nact * TLW) sig_s[u / TLW][u % TLW] = nx[k];
        }
        if (tid < 16) hist_s[tid] = 0;
        // T_len and the subtree climb of request rq on the lane pair 2 rq,
        // 2 rq + 1 (sha256_compress_pair / keccak_f_il_pair)
        // (the other pairs of wave 0 repeat a request)
        const int rq = (tid >> 1) < nact ? tid >> 1 : 0;
        if constexpr (PRE) {
            // SHA-256: every wave runs message schedules of T_len's blocks
            // (they depend on the chain ends only); the pairs then take K + W
            // from LDS.  Consecutive lanes take consecutive requests.
            using SP = Sha2Pair<NW, TLW>;
            for (int it = tid; it < nact * MB; it += 256) {
                const int r = it % nact, b = it / nact;
                Adr pa = adr_make(layer, tree_s[r], kWotsPk);
                adr_keypair<TH>(pa, leaf_s[r]);
                const uint32_t* pk = &pk_s[r][0];
                sha2_kw_block<NW, TLW>(pa, [&](int i) { return pk[i]; }, b,
                                      (lds_u32*)kw_row(r, b));
            }
            __syncthreads();  // K + W of every block in LDS
            if (tid < 64) {
                const uint64_t tree = tree_s[rq];
                const uint32_t leaf = leaf_s[rq];
                Key k2;
#pragma unroll
                for (int i = 0; i < NW; i++) k2.sk[i] = 0;
#pragma unroll
                for (int i = 0; i < 8; i++) k2.mid[i] = key_s[rq][i];
                uint32_t st[4], node[NW];
                SP::init(k2.mid, st);
#pragma unroll 1
                for (int b = 0; b < MB; b++)
                    sha256_rounds_pair_kw(st, (tid & 1) ? &ones_s[0] : kw_row(rq, b));
                SP::output(st, node);
                climb_pair<P>(k2, layer, tree, leaf, &auth_s[rq][0], &node_s[rq][0], node);
                if (tid < 2 * nact && (tid & 1) == 0) {
#pragma unroll
                    for (int w = 0; w < NW; w++) root_s[rq][w] = node[w];
                    leaf_s[rq] = (uint32_t)(tree & ((1u << TH) - 1));
                    tree_s[rq] = tree >> TH;
                }
            }
        } else if constexpr (!SHA2) {
            if (row0 < nact) {
                const uint64_t tree = tree_s[rr];
                const uint32_t leaf = leaf_s[rr];
                uint32_t node[NW];
                LayerRow<P>::run(sponge, layer, tree, leaf, (lds_u32*)pk_s[rr],
                                (lds_u32*)auth_s[rr], (lds_u32*)node_s[rr], node);
                if (tid == 16 * rr) {
#pragma unroll
                    for (int w = 0; w < NW; w++) root_s[rr][w] = node[w];
                    leaf_s[rr] = (uint32_t)(tree & ((1u << TH) - 1));
                    tree_s[rr] = tree >> TH;
                }
            }
        } else if (tid < 64) {
            const uint64_t tree = tree_s[rq];
            const uint32_t leaf = leaf_s[rq];
            Key k2;
#pragma unroll
            for (int i = 0; i < NW; i++) k2.sk[i] = 0;
#pragma unroll
            for (int i = 0; i < 8; i++) k2.mid[i] = key_s[rq][i];
            uint32_t node[NW];
            tlen_climb_pair<P>(k2, layer, tree, leaf, &pk_s[rq][0], &auth_s[rq][0], &node_s[rq][0],
                               node);
            if (tid < 2 * nact && (tid & 1) == 0) {
#pragma unroll
                for (int w = 0; w < NW; w++) root_s[rq][w] = node[w];
                leaf_s[rq] = (uint32_t)(tree & ((1u << TH) - 1));
                tree_s[rq] = tree >> TH;
            }
        }
    }
    __syncthreads();
    if (tid < nact) {
        const Plan& pl = A.plan[req0 + tid];
        bool ok = true;
#pragma unroll
        for (int w = 0; w < NW; w++) ok = ok && (root_s[tid][w] == pl.root[w]);
        A.status[req0 + tid] = ok ? 0 : -1;
    }
}

// Speculative verify for small batches, part 1: every WOTS chain of every
// layer from every possible start.  The start of chain j in layer L is the
// digit d_j of layer L-1's root, known only after that layer, so the chains
// of all 16 starts are computed up front: cap[req][L][j][d] = F_14(..F_d(sig_j))
// (wots_pk_from_sig, wots.cu:777-790, with d = 15 the signature value
// itself).  Lane p of a chain walks the starts p and 15 - p, 15 F steps for
// every lane.  The per-layer pass that remains (k_vht_spec) is T_len and the
// climb only.  SHAKE256 values are stored bit-interleaved.
// The first n_fors workgroups are the batch's FORS trees: neither waits for
// the other, and both are serial runs that leave most of the chip idle (one
// SHAKE256-256f signature: 95 us of trees, 123 us of chains).
template <class P, bool PH>
__global__ void __launch_bounds__(256) k_vspec(BatchArgs A, uint32_t n_fors) {
    if (blockIdx.x < n_fors) {
        vfors_lane<P, PH>(A, blockIdx.x * 256 + threadIdx.x);
        return;
    }
    using Hh = HashPh<P, PH>;
    using Key = typename Hh::Key;
    constexpr bool SHA2 = P::hash == kSha2;
    constexpr int NW = P::nw;
    const uint64_t g0 = (uint64_t)(blockIdx.x - n_fors) * 256 + threadIdx.x;
    const uint64_t ng = (uint64_t)A.n_req * P::d * P::len * 8;
    const uint64_t g = g0 < ng ? g0 : ng - 1;  // repeated past the end
    const int p = (int)(g & 7);
    const uint64_t c = g >> 3;                       // (req * d + layer) * len + j
    const int j = (int)(c % P::len);
    const uint32_t layer = (uint32_t)((c / P::len) % P::d);
    const uint32_t req = (uint32_t)(c / ((uint64_t)P::len * P::d));
    const Plan& pl = A.plan[req];
    Key key;
    Hh::load_key(pl, key);
    const uint64_t tree = layer_tree<P>(pl.tree, layer);
    const uint32_t leaf = layer == 0 ? pl.leaf
                                     : (uint32_t)((pl.tree >> ((layer - 1) * P::th)) &
                                                  ((1u << P::th) - 1));
    Adr wa = adr_make(layer, tree, kWots);
    adr_keypair<P::th>(wa, leaf);
    adr_chain(wa, j);
    uint32_t sg[NW], v[NW];
    load_val<P::hash, NW>(A.sig + (size_t)req * A.sig_stride + P::n + P::fors_bytes +
                              (size_t)layer * P::layer_bytes + (size_t)j * P::n,
                          sg);
    typename Hh::Chain ch;
    Hh::chain_begin(key, wa, ch);
    if constexpr (!SHA2) {
        uint32_t t[NW];
        Hh::to_il(sg, t);
#pragma unroll
        for (int w = 0; w < NW; w++) sg[w] = t[w];
    }
    uint32_t* out = reinterpret_cast<uint32_t*>(A.cap) + c * 16 * NW;
    if (p == 0) {  // start 15: no step
#pragma unroll
        for (int w = 0; w < NW; w++) out[15 * NW + w] = sg[w];
    }
#pragma unroll
    for (int w = 0; w < NW; w++) v[w] = sg[w];
    uint32_t s = p;     // chain A: start p, 15 - p steps; then chain B: start 15 - p, p steps
    bool second = false;
#pragma unroll 1
    for (int it = 0; it < 15; it++) {
        Hh::chain_step(key, ch, s, v, v);
        s++;
        if (s == (uint32_t)P::w - 1) {
            const int d = second ? 15 - p : p;
#pragma unroll
            for (int w = 0; w < NW; w++) out[d * NW + w] = v[w];
            second = true;
            s = 15 - p;
#pragma unroll
            for (int w = 0; w < NW; w++) v[w] = sg[w];
        }
    }
}

// Speculative verify, part 2: one wave per request computes T_k and walks the
// d layers (sign.cu:3077-3113): lanes pick each chain's end for the layer's
// message from the candidates of k_vspec and load the auth path, then run
// T_len and compute_root (utils.cu:94-135): SHA-256 on lane pairs with the
// message schedules of T_len's blocks from one lane each, SHAKE256 on rows of
// 32 lanes (LayerRow).  The serial work per layer is T_len + h' nodes instead
// of the longest chain + T_len + h' nodes.  One SHAKE256-256f signature: 958 ->
// 854 us against rows of 16 lanes.
template <class P>
__global__ void __launch_bounds__(64) k_vht_spec(BatchArgs A) {
    using Hh = HashT<P>;
    using Key = typename Hh::Key;
    constexpr int NW = P::nw;
    constexpr int LEN = P::len;
    constexpr int TH = P::th;
    constexpr int TLW = LEN * NW;
    constexpr int AW = TH * NW;
    constexpr bool SHA2 = P::hash == kSha2;
    // as in k_vht
    constexpr int PKO = SHA2 ? 0 : NW + 8;
    __shared__ uint32_t pk_s[tlen_words<P>()];
    __shared__ uint32_t auth_s[AW];
    __shared__ uint32_t root_s[NW];
    __shared__ uint32_t node_s[SHA2 ? NW : 34];
    __shared__ __align__(16) uint32_t row_s[SHA2 ? 1 : Keccak32::kLdsWords];
    // SHA-256: K + W of T_len's blocks, 68-word rows (the lanes' 16-byte
    // writes fall into distinct banks)
    constexpr int MB = SHA2 ? Sha2Pair<NW, TLW>::B : 1;
    static_assert(MB <= 64, "one lane per block");
    __shared__ __align__(16) uint32_t kw_s[SHA2 ? MB : 1][68];
    __shared__ __align__(16) uint32_t ones_s[SHA2 ? kKwOnes : 1];
    __shared__ __align__(16) uint32_t fpk_s[fors_pk_wave_words<P>()];
    if (SHA2) ones_s[threadIdx.x] = 1u;
    const int tid = threadIdx.x;
    const uint32_t req = blockIdx.x;  // grid = n_req
    const Plan& pl = A.plan[req];
    const uint8_t* sig = A.sig + (size_t)req * A.sig_stride;
    const uint32_t* cand = reinterpret_cast<const uint32_t*>(A.cap) + (size_t)req * P::d * LEN * 16 * NW;
    {
        uint32_t fp[NW];
        fors_pk_value<P>(A, req, (lds_u32*)fpk_s, fp);
        if (tid == 0) {
#pragma unroll
            for (int w = 0; w < NW; w++) root_s[w] = fp[w];
        }
    }
    Keccak32 sponge;  // both rows of 32 lanes run the same one in step
    if constexpr (!SHA2) {
        Key key;
        Hh::load_key(pl, key);
        sponge.init((lds_u32*)row_s);
        LayerRow<P>::TL::begin(sponge, key.pub, (lds_u32*)pk_s);
        LayerRow<P>::TH::begin(sponge, key.pub, (lds_u32*)node_s);
    }
    uint64_t tree = pl.tree;
    uint32_t leaf = pl.leaf;
#pragma unroll 1
    for (int layer = 0; layer < P::d; layer++) {
        __syncthreads();
        uint32_t msg[NW];
#pragma unroll
        for (int w = 0; w < NW; w++) msg[w] = root_s[w];
        const uint32_t* lc = cand + (size_t)layer * LEN * 16 * NW;
#pragma unroll 1
        for (int j = tid; j < LEN; j += 64) {
            const uint32_t d = chain_len<P>(msg, j);
#pragma unroll
            for (int w = 0; w < NW; w++) pk_s[PKO + j * NW + w] = lc[((size_t)j * 16 + d) * NW + w];
        }
        const uint32_t* auth = reinterpret_cast<const uint32_t*>(
            sig + P::n + P::fors_bytes + (size_t)layer * P::layer_bytes + P::wots_bytes);
        for (int u = tid; u < AW; u += 64)
            auth_s[u] = SHA2 ? auth[u] : il_half(auth[u & ~1], auth[u | 1], u & 1);
        __syncthreads();
        uint32_t node[NW];
        if constexpr (P::hash == kSha2) {
            // every lane computes K + W of one of T_len's blocks, then the
            // pair 0, 1 runs only their rounds
            Adr pa = adr_make(layer, tree, kWotsPk);
            adr_keypair<TH>(pa, leaf);
            if (tid < MB)
                sha2_kw_block<NW, TLW>(pa, [&](int i) { return pk_s[i]; }, tid, (lds_u32*)kw_s[tid]);
            __syncthreads();
            // T_len and the climb on lane pairs, all alike (k_ht says why)
            using SP = Sha2Pair<NW, TLW>;
            Key key;
            Hh::load_key(pl, key);
            uint32_t st[4];
            SP::init(key.mid, st);
#pragma unroll 1
            for (int b = 0; b < MB; b++)
                sha256_rounds_pair_kw(st, (tid & 1) ? &ones_s[0] : &kw_s[b][0]);
            SP::output(st, node);
            climb_pair<P>(key, layer, tree, leaf, auth_s, node_s, node);
        } else {
            LayerRow<P>::run(sponge, layer, tree, leaf, (lds_u32*)pk_s, (lds_u32*)auth_s,
                            (lds_u32*)node_s, node);
        }
        if (tid == 0) {
#pragma unroll
            for (int w = 0; w < NW; w++) root_s[w] = node[w];
        }
        leaf = (uint32_t)(tree & ((1u << TH) - 1));
        tree >>= TH;
    }
    __syncthreads();
    if (tid == 0) {
        bool ok = true;
#pragma unroll
        for (int w = 0; w < NW; w++) ok = ok && (root_s[w] == pl.root[w]);
        A.status[req] = ok ? 0 : -1;
    }
}

}  // namespace spx
