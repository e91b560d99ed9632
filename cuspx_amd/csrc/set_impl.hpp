// set_impl.hpp -- host-side launch sequences for one parameter set.
// Each set_<name>.hip instantiates SetImpl<P, J> and registers its SetOps.
#pragma once
#include "engine.hpp"
#include "profile.hpp"
#include "slices.hpp"
#include "spx_kernels.hpp"

namespace spx {

static inline uint32_t cdiv(uint64_t a, uint64_t b) { return (uint32_t)((a + b - 1) / b); }

// lanes that fill the chip: 1024 SIMDs x 64 lanes x 4 waves
static constexpr uint64_t kFillLanes = 1024ull * 64 * 4;

// workspace carve-up shared by sign / verify / keygen
template <class P>
struct Layout {
    static constexpr uint64_t al(uint64_t x) { return (x + 255) & ~uint64_t(255); }

    // The split of a sign / keygen batch over `trees` subtrees: a tuned value
    // when the tuning table has one.  k_ht runs a lane per WOTS leaf at 1, a
    // lane pair at 2 and 4 and 16 lanes at 8 and 16 (the chains take a lane
    // each whatever the split); mixed batches go to the family kernel up to 2.
    // Without a table: 16 lanes while their waves are 2 per SIMD or fewer, a
    // pair up to 24576 leaves.  k_ht at 1 / 4 / 16, us: SHA2-128f, 8000 leaves
    // 47 / 50 / 45, 11264 51 / 41 / 67, 35200 51 / 62 / 168; SHA2-128s, 7168
    // 75 / 63 / 73, 57344 79 / 108 / 456; SHAKE256-128f, 11264 80 / 60 / 82,
    // 88000 93 / 121 / 360.
    static int split(int pid, int op, uint32_t trees) {
        const int t = tuned_split(pid, op, trees);
        if (t == 1 || t == 2 || t == 4 || t == 8 || t == 16) return t;
        const uint64_t leaves = (uint64_t)trees << P::th;
        return leaves <= 8192 ? 16 : leaves <= 24576 ? 4 : 1;
    }
    // Verify kernel width: G lanes per request on average (k_vht runs
    // 256 / G requests per workgroup and deals all their chains over its 256
    // lanes).  A tuned value when the table has one, else G = 16 doubled
    // while the launch would fill under an eighth of the chip: wider groups
    // shorten each layer's chain phase down to the longest chain, narrower
    // ones keep more requests per lane.
    // G = 1 selects speculative verification (k_vspec + k_vht_spec): every
    // chain from every start up front, then T_len and the climb per layer;
    // 16x the chain work for half the dependent path, so batches up to
    // kSpecMax requests only (the workspace keeps candidates for that many).
    static constexpr int vmin() { return 16; }
    static constexpr int vmax() { return P::len > 64 ? 128 : 64; }
    static constexpr uint32_t kSpecMax = 256;
    static constexpr uint32_t kSpecDefault = 64;  // built-in choice without a table
    // sign batches up to this size run T_k inside the FORS tiles
    static constexpr uint32_t kForsPkInline = 256;
    static bool vvalid(int g, uint32_t n) {
        if (g == 1) return n <= kSpecMax;
        return g >= vmin() && g <= vmax() && (g & (g - 1)) == 0;
    }
    // candidate chain ends of min(n, kSpecMax) requests: monotone in n, so a
    // workspace sized for a batch also holds every smaller batch's layout
    static uint64_t spec_bytes(uint32_t n) {
        return (uint64_t)(n < kSpecMax ? n : kSpecMax) * P::d * P::len * 16 * P::n;
    }
    static int vsplit(int pid, uint32_t n) {
        const int t = tuned_split(pid, kOpVerify, n);
        if (vvalid(t, n)) return t;
        if (n <= kSpecDefault) return 1;
        int G = vmin();
        while (G < vmax() && (uint64_t)n * G * 8 <= kFillLanes) G *= 2;
        return G;
    }
    static constexpr int L = 1 << P::th;
    template <int S>
    static uint32_t ht_blocks(uint32_t trees) {
        return HtShape<P, S>::PARTS > 1 ? trees * HtShape<P, S>::PARTS
                                        : cdiv(trees, HtShape<P, S>::TPW);
    }
    // workspace room for split subtrees (part roots) and for the
    // chain ends' columns, whole workgroups of leaves: the sizes that callers
    // with a fixed scratch area have had for their batch limits
    static constexpr int max_parts() { return L * 16 > 1024 ? L * 16 / 256 : 1; }
    static uint64_t tl_cols(uint32_t trees) {
        constexpr uint64_t lanes = (uint64_t)L * (P::hash == kShake ? 1 : 2);
        constexpr uint64_t tpw = lanes < 256 ? 256 / lanes : 1;
        return (trees + tpw - 1) / tpw * tpw * L;
    }
    static_assert(max_parts() >= HtShape<P, 16>::PARTS, "part roots fit");
    static uint64_t bytes(int pid, uint32_t n, int op) {
        uint64_t b = al((uint64_t)n * sizeof(Plan));
        b += al((uint64_t)n * P::k * P::n);   // fors roots
        b += al((uint64_t)n * P::n);          // fors pk
        if (op == kOpSign) b += al((uint64_t)n * 4);  // fors root counters
        if (op == kOpVerify) b += al(spec_bytes(n));              // speculative candidates
        if (op == kOpSign) {
            b += al((uint64_t)n * P::d * P::n);                    // layer roots
            b += al((uint64_t)n * P::d * P::len * 16 * P::n);      // chain capture
            b += al(4);                                            // (spare)
        }
        if (op != kOpVerify) {
            const uint32_t trees = op == kOpSign ? n * P::d : n;
            b += al(tl_cols(trees) * P::len * P::nw * 4);
            if (max_parts() > 1) {
                b += al((uint64_t)trees * max_parts() * P::nw * 4);  // part roots
                b += al((uint64_t)trees * 4);                       // part counters
            }
        }
        (void)pid;
        return b + 256;
    }
    static void carve(int pid, BatchArgs& A, uint8_t* ws, uint32_t n, int op) {
        uint8_t* p = (uint8_t*)(((uintptr_t)ws + 255) & ~(uintptr_t)255);
        A.plan = (Plan*)p;
        p += al((uint64_t)n * sizeof(Plan));
        A.fors_roots = p;
        p += al((uint64_t)n * P::k * P::n);
        A.fors_pk = p;
        p += al((uint64_t)n * P::n);
        A.fors_count = nullptr;
        if (op == kOpSign) {
            // T_k in the FORS tiles for small batches only (see fors_root_done)
            if (n <= kForsPkInline) A.fors_count = (uint32_t*)p;
            p += al((uint64_t)n * 4);
        }
        A.roots = nullptr;
        A.cap = nullptr;
        A.tl_buf = nullptr;
        A.tl_lanes = 0;
        A.ht_parts = nullptr;
        A.ht_count = nullptr;
        if (op == kOpVerify) {
            A.cap = p;
            p += al(spec_bytes(n));
        }
        if (op == kOpSign) {
            A.roots = p;
            p += al((uint64_t)n * P::d * P::n);
            A.cap = p;
            p += al((uint64_t)n * P::d * P::len * 16 * P::n);
            p += al(4);
        }
        if (op != kOpVerify) {
            const uint32_t trees = op == kOpSign ? n * P::d : n;
            A.tl_buf = (uint32_t*)p;
            A.tl_lanes = leaf_count<P>(trees);
            p += al(tl_cols(trees) * P::len * P::nw * 4);
            if (max_parts() > 1) {
                A.ht_parts = (uint32_t*)p;
                p += al((uint64_t)trees * max_parts() * P::nw * 4);
                A.ht_count = (uint32_t*)p;
                p += al((uint64_t)trees * 4);
            }
        }
        (void)pid;
    }
};

// Chain waves up to which FORS and chains share a launch (k_sign_fused), so
// that FORS does not run before the chains; larger batches launch k_fors and
// k_chains one after the other.  The fused kernel takes the FORS tile's
// registers (103-152 VGPRs, 4 or 3 waves per SIMD) for the chains too, which
// k_chains alone runs at 8 (SHA-256, 58-61 VGPRs) or 5; what it gains is the
// overlap.  Whole call, separate / fused, us: SHA2-128f 1 request 171 / 105,
// 61 320 / 258, 85 (8190 waves) 364 / 310, 130 487 / 420, 250 (24080) 768 /
// 720; SHAKE256-256f 28 1013 / 867, 60 1773 / 1600; SHA2-128s 8 642 / 497.  So
// the crossover lies beyond 24000 waves, and the line is short of it: 8 waves
// per SIMD, the last size where the chains alone are one round of waves.
static constexpr uint32_t kFuseWaves = 8192;
// Chain waves of a fused launch up to which its FORS tiles are the narrowest
// (JF leaves per lane): with 3.5 chain waves per SIMD or fewer there is room
// for twice the FORS waves and the tile's serial run is what the launch waits
// for; beyond, the extra waves only compete with the chains.  Measured,
// k_sign_fused with J -> JF, us: SHA2-128f 1 request 67 -> 51, 16 93 -> 77,
// 32 (3080 waves) 134 -> 125, 61 (5880) 201 -> 202, 85 260 -> 263;
// SHAKE256-256f 1 278 -> 138, 7 321 -> 245, 14 (3987) 399 -> 436;
// SHA2-256f 14 201 -> 194, 28 315 -> 332.
static constexpr uint32_t kShortForsWaves = 3584;
// Waves of FORS tiles up to which a tree of 2^14 leaves (192s, 256s) is split
// over 4 workgroups, whose last one climbs the top two levels: one workgroup
// per tree is a serial run of 64 leaves and their nodes on every lane, about
// 270 hashes, which nothing else in a small batch hides.  4096 waves are 4 per
// SIMD, about what the kernels hold at once (117-152 VGPRs).  Whole -> split,
// us: k_sign_fused of 1 SHA2-192s request 843 -> 297, of 1 SHAKE256-256s 1784 ->
// 537; k_fors of SHA2-192s 3 requests 826 -> 232, 15 (4080 waves) 853 -> 547,
// SHA2-256s 5 845 -> 316, 20 (7040 waves) 986 -> 877.
static constexpr uint32_t kSplitForsWaves = 4096;

// J: FORS leaves per lane, 2^J (2^(a-J) lanes per tree).  Short tiles at every
// size: a tile is a serial run of 3-4 x 2^J hashes, and with the two-phase
// rounds the longer tiles of before (2^4 to 2^6 leaves) gained 0-4% of k_fors
// at 4096 requests and cost it up to 2.9 times at 128 (SHA2-256f, 2^6 -> 2^3
// leaves: 512 requests 1377 -> 982 us, 4096 7.28 -> 7.15 ms; SHA2-128f 128
// requests, 2^4 -> 2^2: 203 -> 105 us).
template <class P, int J>
inline void launch_fors(const BatchArgs& A, uint32_t n, hipStream_t s) {
    const uint32_t tiles = cdiv((uint64_t)n * P::k, 256u >> (P::a - J));
    if (A.fors_count)
        hipLaunchKernelGGL((k_fors<P, J, true>), dim3(tiles), dim3(256), 0, s, A);
    else
        hipLaunchKernelGGL((k_fors<P, J, false>), dim3(tiles), dim3(256), 0, s, A);
}

// A's requests [a, a + n) as a batch of their own for the chains' and the
// subtrees' kernels, in A's workspace and outputs (MODE as for those kernels)
template <class P, int MODE>
inline BatchArgs batch_rows(const BatchArgs& A, uint32_t a, uint32_t n) {
    BatchArgs B = A;
    const size_t trees = (size_t)a * (MODE == 0 ? P::d : 1);
    B.n_req = n;
    B.plan += a;
    B.tl_buf += trees << P::th;  // columns; tl_lanes stays the whole batch's
    if (B.ht_parts) {
        B.ht_parts += trees * (Layout<P>::max_parts() * P::nw);
        B.ht_count += trees;
    }
    if (MODE == 0) {
        B.sig += a * B.sig_stride;
        B.roots += trees * P::n;
        B.cap += trees * (P::len * 16 * P::n);
    } else {
        B.pk_out += (size_t)a * P::pk_bytes;
        B.sk_out += (size_t)a * P::sk_bytes;
    }
    return B;
}

template <class P, int MODE, bool PH>
inline void launch_chains(const BatchArgs& A, hipStream_t s) {
    constexpr uint32_t trees = MODE == 0 ? P::d : 1;
    for_slices(A.n_req, 64ull * chain_waves<P>(A.n_req * trees), [&](uint32_t a, uint32_t n) {
        const uint32_t nwaves = chain_waves<P>(n * trees);
        hipLaunchKernelGGL((k_chains<P, MODE, PH>), dim3(cdiv(nwaves, 4)), dim3(256), 0, s,
                           batch_rows<P, MODE>(A, a, n), nwaves);
    });
}
template <class P, int MODE, int S>
inline void launch_ht(const BatchArgs& A, hipStream_t s) {
    constexpr uint32_t trees = MODE == 0 ? P::d : 1, WG = HtShape<P, S>::WG;
    for_slices(A.n_req, (uint64_t)WG * Layout<P>::template ht_blocks<S>(A.n_req * trees),
               [&](uint32_t a, uint32_t n) {
                   hipLaunchKernelGGL((k_ht<P, MODE, S>),
                                      dim3(Layout<P>::template ht_blocks<S>(n * trees)), dim3(WG),
                                      0, s, batch_rows<P, MODE>(A, a, n));
               });
}

template <class P, int J>
struct SetImpl {
    using Lay = Layout<P>;

    static int pid_;
    static const char* set_name_;
    static size_t workspace(uint32_t n, int op) { return (size_t)Lay::bytes(pid_, n, op); }

    template <int MODE>
    static void launch_ht(const BatchArgs& A, int S, hipStream_t s) {
        if (S == 1) spx::launch_ht<P, MODE, 1>(A, s);
        else if (S <= 4) spx::launch_ht<P, MODE, 2>(A, s);
        else spx::launch_ht<P, MODE, 16>(A, s);
    }
    // a launch of so many waves leaves each of them a SIMD (HashPh)
    static constexpr bool kSha = P::hash == kSha2;
    static bool alone(uint32_t waves) { return kSha && waves <= kAloneWaves; }
    // FORS leaves per lane in a fused launch of few waves: 2, or as many as 256
    // lanes per tree leave; trees of 2^14 leaves (192s, 256s) are split over
    // FP = 4 workgroups (kSplitForsWaves)
    static constexpr int JF = P::a - 8 > 4 ? P::a - 10 : P::a - 8 > 1 ? P::a - 8 : 1;
    static constexpr int FP = fors_parts<P, JF>();
    static_assert(FP == 1 || P::k * FP <= P::d * Lay::max_parts(), "the parts' roots fit ht_parts");
    template <int FJ>
    static uint32_t fors_tiles(uint32_t n) {
        constexpr int parts = fors_parts<P, FJ>();
        if constexpr (parts > 1) return n * (P::k * parts);
        else return cdiv((uint64_t)n * P::k, 256u >> (P::a - FJ));
    }

    // workgroups of k_vht up to which each has a CU to itself
    static constexpr uint32_t kVhtAlone = 256;
    template <int G>
    static void launch_vht(const BatchArgs& A, uint32_t n, hipStream_t s) {
        const uint32_t wgs = cdiv(n, 256 / G);
        if constexpr (G >= 64) {
            hipLaunchKernelGGL((k_vht<P, G, kVhtPair>), dim3(wgs), dim3(256), 0, s, A);
        } else {
            if constexpr (P::hash == kSha2) {
                if (wgs > kVhtAlone) {
                    hipLaunchKernelGGL((k_vht<P, G, kVhtPhased>), dim3(wgs), dim3(256), 0, s, A);
                    return;
                }
            }
            hipLaunchKernelGGL((k_vht<P, G, kVhtLane>), dim3(wgs), dim3(256), 0, s, A);
        }
    }
    static int sign(const DevBatch& b, hipStream_t s) {
        BatchArgs A{};
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
        const uint32_t n = b.n;
        const int S = Lay::split(pid_, kOpSign, n * P::d);
        Lay::carve(pid_, A, (uint8_t*)b.ws, b.n, kOpSign);
        (void)hipGetLastError();  // report only errors of these launches
        prof_begin(s, set_name_);
        launch_prep<P, false>(A, n, b.mlen_bound, s);
        prof_mark(s, "k_prep");
        // (up to kForsPkInline requests T_k runs on the lane that stores a
        // request's last FORS root, inside the FORS tiles)
        const uint32_t nwaves = chain_waves<P>(n * P::d);
        if (nwaves <= kFuseWaves) {
            if (FP > 1 || nwaves <= kShortForsWaves) {
                const uint32_t nf = fors_tiles<JF>(n);
                const uint32_t wgs = nf + cdiv(nwaves, 4);
                if (alone(4 * wgs))
                    hipLaunchKernelGGL((k_sign_fused<P, JF, !kSha>), dim3(wgs), dim3(256), 0, s, A,
                                       nf, nwaves);
                else
                    hipLaunchKernelGGL((k_sign_fused<P, JF, true>), dim3(wgs), dim3(256), 0, s, A,
                                       nf, nwaves);
            } else if constexpr (FP == 1) {
                const uint32_t nf = fors_tiles<J>(n);
                hipLaunchKernelGGL((k_sign_fused<P, J, true>), dim3(nf + cdiv(nwaves, 4)),
                                   dim3(256), 0, s, A, nf, nwaves);
            }
            prof_mark(s, "k_sign_fused");
        } else {
            if (FP > 1 && 4 * fors_tiles<JF>(n) <= kSplitForsWaves) {
                if constexpr (FP > 1) {
                    const uint32_t nf = fors_tiles<JF>(n);
                    if (alone(4 * nf))
                        hipLaunchKernelGGL((k_fors<P, JF, true, !kSha>), dim3(nf), dim3(256), 0, s, A);
                    else hipLaunchKernelGGL((k_fors<P, JF, true>), dim3(nf), dim3(256), 0, s, A);
                }
            } else {
                launch_fors<P, J>(A, n, s);
            }
            prof_mark(s, "k_fors");
            launch_chains<P, 0, true>(A, s);
            prof_mark(s, "k_chains");
        }
        if (!A.fors_count) {
            launch_fors_pk<P>(A, n, s);
            prof_mark(s, "k_fors_pk");
        }
        launch_ht<0>(A, S, s);
        prof_mark(s, "k_ht");
        hipLaunchKernelGGL((k_wots_gather<P>), dim3(cdiv((uint64_t)n * P::d * P::len, 256)),
                           dim3(256), 0, s, A);
        prof_mark(s, "k_wots_gather");
        return hipGetLastError() == hipSuccess ? 0 : kErrHip;
    }

    static int verify(const DevBatch& b, hipStream_t s) {
        BatchArgs A{};
        A.pk = b.pk;
        A.pk_stride = b.pk_stride;
        A.key_idx = b.key_idx;
        A.key_mid = b.key_mid;
        A.msg = b.msg;
        A.moff = b.moff;
        A.mlen = b.mlen;
        A.sig = b.sig;
        A.sig_stride = b.sig_stride;
        A.status = b.status;
        A.n_req = b.n;
        Lay::carve(pid_, A, (uint8_t*)b.ws, b.n, kOpVerify);
        const uint32_t n = b.n;
        const int G = Lay::vsplit(pid_, n);
        (void)hipGetLastError();  // report only errors of these launches
        prof_begin(s, set_name_);
        launch_prep<P, true>(A, n, b.mlen_bound, s);
        prof_mark(s, "k_vprep");
        if (G == 1) {
            const uint32_t nf = cdiv((uint64_t)n * P::k, 256);
            const uint32_t wgs = nf + cdiv((uint64_t)n * P::d * P::len * 8, 256);
            if (alone(4 * wgs))
                hipLaunchKernelGGL((k_vspec<P, !kSha>), dim3(wgs), dim3(256), 0, s, A, nf);
            else
                hipLaunchKernelGGL((k_vspec<P, true>), dim3(wgs), dim3(256), 0, s, A, nf);
            prof_mark(s, "k_vspec");
            hipLaunchKernelGGL((k_vht_spec<P>), dim3(n), dim3(64), 0, s, A);
            prof_mark(s, "k_vht");
            return hipGetLastError() == hipSuccess ? 0 : kErrHip;
        }
        const uint32_t fw = cdiv((uint64_t)n * P::k, 64);
        // (of one-wave workgroups two can meet on a SIMD well before all have one)
        if (alone(2 * fw)) hipLaunchKernelGGL((k_vfors<P, !kSha>), dim3(fw), dim3(64), 0, s, A);
        else hipLaunchKernelGGL((k_vfors<P, true>), dim3(fw), dim3(64), 0, s, A);
        prof_mark(s, "k_vfors");
        launch_fors_pk<P>(A, n, s);
        prof_mark(s, "k_fors_pk");
        if (G == 16) launch_vht<16>(A, n, s);
        else if (G == 32) launch_vht<32>(A, n, s);
        else if (G == 64) launch_vht<64>(A, n, s);
        else if constexpr (Lay::vmax() >= 128) launch_vht<128>(A, n, s);
        prof_mark(s, "k_vht");
        return hipGetLastError() == hipSuccess ? 0 : kErrHip;
    }

    static int keygen(const DevBatch& b, hipStream_t s) {
        BatchArgs A{};
        A.seed = b.seed;
        A.seed_stride = b.seed_stride;
        A.pk_out = b.pk_out;
        A.sk_out = b.sk_out;
        A.n_req = b.n;
        const uint32_t n = b.n;
        const int S = Lay::split(pid_, kOpKeygen, n);
        Lay::carve(pid_, A, (uint8_t*)b.ws, b.n, kOpKeygen);
        (void)hipGetLastError();  // report only errors of these launches
        prof_begin(s, set_name_);
        hipLaunchKernelGGL((k_kprep<P>), dim3(cdiv(n, 64)), dim3(64), 0, s, A);
        prof_mark(s, "k_kprep");
        if (alone(chain_waves<P>(n))) launch_chains<P, 1, !kSha>(A, s);
        else launch_chains<P, 1, true>(A, s);
        prof_mark(s, "k_chains_keygen");
        launch_ht<1>(A, S, s);
        prof_mark(s, "k_ht_keygen");
        return hipGetLastError() == hipSuccess ? 0 : kErrHip;
    }

    static int midstates(const uint8_t* pk, uint32_t pk_stride, uint32_t* mid, uint32_t n,
                         hipStream_t s) {
        if (n == 0) return 0;
        (void)hipGetLastError();
        hipLaunchKernelGGL((k_midstate<P>), dim3(cdiv(n, 64)), dim3(64), 0, s, pk, pk_stride, mid,
                           n);
        return hipGetLastError() == hipSuccess ? 0 : kErrHip;
    }

    static int split(int op, uint32_t n) {
        if (op == kOpVerify) return Lay::vsplit(pid_, n);
        return Lay::split(pid_, op, op == kOpSign ? n * P::d : n);
    }

    static SetOps ops(const char* name, int pid) {
        pid_ = pid;
        set_name_ = name;
        SetOps o{};
        o.name = name;
        o.pid = pid;
        o.hash = P::hash;
        o.n = P::n;
        o.full_h = P::full_h;
        o.d = P::d;
        o.a = P::a;
        o.k = P::k;
        o.len = P::len;
        o.sig_bytes = P::sig_bytes;
        o.pk_bytes = P::pk_bytes;
        o.sk_bytes = P::sk_bytes;
        o.workspace = &workspace;
        o.sign = &sign;
        o.verify = &verify;
        o.keygen = &keygen;
        o.midstates = &midstates;
        o.split = &split;
        return o;
    }
};

template <class P, int J>
int SetImpl<P, J>::pid_ = -1;
template <class P, int J>
const char* SetImpl<P, J>::set_name_ = "";

}  // namespace spx

#define SPX_REGISTER_SET(SYM, NAME, PID, PARAMS, J)                        \
    extern "C" const spx::SetOps* SYM(void) {                              \
        static const spx::SetOps o = spx::SetImpl<PARAMS, J>::ops(NAME, PID); \
        return &o;                                                         \
    }
