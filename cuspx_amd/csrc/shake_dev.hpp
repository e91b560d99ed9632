// shake_dev.hpp -- SHAKE256 tweakable-hash family for CDNA4 (gfx950).
//
// Semantics follow the reference host path:
//   thash  T_l(x) = SHAKE256(pub_seed || addr[0..32) || x, n)   thash_shake256.cu:15-25
//   PRF(a)        = SHAKE256(sk_seed || addr[0..32), n)         hash_shake256.cu:38-47
//   PRF_msg       = SHAKE256(sk_prf || optrand || m, n)         hash_shake256.cu:64-75
//   H_msg         = SHAKE256(R || pk || m, dgst)                hash_shake256.cu:96-130
// The address uses the SHA-256 byte layout (params.h:148), so bytes 22..31
// are zero.
//
// Keccak-f[1600] runs on 32-bit lane halves: the 200-byte state is 50
// little-endian words s[2i] (low) / s[2i+1] (high), so sponge byte j sits in
// word j/4.  64-bit rotations are two v_alignbit, theta's column parity two
// v_bitop3 (3-way xor) per half, theta application one 3-way xor per word and
// chi one v_bitop3 (a ^ (~b & c)) per word.
#pragma once
#include "spx_common.hpp"

namespace spx {

__constant__ uint32_t kKeccakRC[48] = {
    0x00000001u, 0x00000000u, 0x00008082u, 0x00000000u, 0x0000808au, 0x80000000u,
    0x80008000u, 0x80000000u, 0x0000808bu, 0x00000000u, 0x80000001u, 0x00000000u,
    0x80008081u, 0x80000000u, 0x00008009u, 0x80000000u, 0x0000008au, 0x00000000u,
    0x00000088u, 0x00000000u, 0x80008009u, 0x00000000u, 0x8000000au, 0x00000000u,
    0x8000808bu, 0x00000000u, 0x0000008bu, 0x80000000u, 0x00008089u, 0x80000000u,
    0x00008003u, 0x80000000u, 0x00008002u, 0x80000000u, 0x00000080u, 0x80000000u,
    0x0000800au, 0x00000000u, 0x8000000au, 0x80000000u, 0x80008081u, 0x80000000u,
    0x00008080u, 0x80000000u, 0x80000001u, 0x00000000u, 0x80008008u, 0x80000000u};

// rotation offsets r[x + 5y]
static constexpr int kRho[25] = {0,  1,  62, 28, 27, 36, 44, 6,  55, 20, 3,  10, 43,
                                 25, 39, 41, 45, 15, 21, 8,  18, 2,  61, 56, 14};

template <int R>
__device__ __forceinline__ void rol64(uint32_t lo, uint32_t hi, uint32_t& olo, uint32_t& ohi) {
    if (R == 0) {
        olo = lo;
        ohi = hi;
    } else if (R < 32) {
        ohi = __builtin_amdgcn_alignbit(hi, lo, 32 - R);
        olo = __builtin_amdgcn_alignbit(lo, hi, 32 - R);
    } else if (R == 32) {
        olo = hi;
        ohi = lo;
    } else {
        ohi = __builtin_amdgcn_alignbit(lo, hi, 64 - R);
        olo = __builtin_amdgcn_alignbit(hi, lo, 64 - R);
    }
}

// one round of Keccak-f[1600] on s[50] with round constant (rc_lo, rc_hi)
__device__ __forceinline__ void keccak_round(uint32_t s[50], uint32_t rc_lo, uint32_t rc_hi) {
    uint32_t C[10];
#pragma unroll
    for (int x = 0; x < 5; x++) {
#pragma unroll
        for (int h = 0; h < 2; h++) {
            C[2 * x + h] = xor3(xor3(s[2 * x + h], s[2 * (x + 5) + h], s[2 * (x + 10) + h]),
                                s[2 * (x + 15) + h], s[2 * (x + 20) + h]);
        }
    }
#pragma unroll
    for (int x = 0; x < 5; x++) {
        uint32_t rlo, rhi;
        const int xp = (x + 1) % 5, xm = (x + 4) % 5;
        rol64<1>(C[2 * xp], C[2 * xp + 1], rlo, rhi);
#pragma unroll
        for (int y = 0; y < 5; y++) {
            s[2 * (x + 5 * y)] = xor3(s[2 * (x + 5 * y)], C[2 * xm], rlo);
            s[2 * (x + 5 * y) + 1] = xor3(s[2 * (x + 5 * y) + 1], C[2 * xm + 1], rhi);
        }
    }
    uint32_t B[50];
#pragma unroll
    for (int x = 0; x < 5; x++) {
#pragma unroll
        for (int y = 0; y < 5; y++) {
            // pi: B[y, 2x + 3y] = rol(A[x, y], r[x, y])
            const int src = x + 5 * y;
            const int dst = y + 5 * ((2 * x + 3 * y) % 5);
            uint32_t lo, hi;
            switch (kRho[src]) {
#define SPX_ROT_CASE(R) \
    case R: rol64<R>(s[2 * src], s[2 * src + 1], lo, hi); break;
                SPX_ROT_CASE(0) SPX_ROT_CASE(1) SPX_ROT_CASE(62) SPX_ROT_CASE(28)
                SPX_ROT_CASE(27) SPX_ROT_CASE(36) SPX_ROT_CASE(44) SPX_ROT_CASE(6)
                SPX_ROT_CASE(55) SPX_ROT_CASE(20) SPX_ROT_CASE(3) SPX_ROT_CASE(10)
                SPX_ROT_CASE(43) SPX_ROT_CASE(25) SPX_ROT_CASE(39) SPX_ROT_CASE(41)
                SPX_ROT_CASE(45) SPX_ROT_CASE(15) SPX_ROT_CASE(21) SPX_ROT_CASE(8)
                SPX_ROT_CASE(18) SPX_ROT_CASE(2) SPX_ROT_CASE(61) SPX_ROT_CASE(56)
                SPX_ROT_CASE(14)
#undef SPX_ROT_CASE
                default: lo = s[2 * src]; hi = s[2 * src + 1]; break;
            }
            B[2 * dst] = lo;
            B[2 * dst + 1] = hi;
        }
    }
#pragma unroll
    for (int y = 0; y < 5; y++) {
#pragma unroll
        for (int x = 0; x < 5; x++) {
#pragma unroll
            for (int h = 0; h < 2; h++) {
                s[2 * (x + 5 * y) + h] = bit_chi(B[2 * (x + 5 * y) + h],
                                                 B[2 * ((x + 1) % 5 + 5 * y) + h],
                                                 B[2 * ((x + 2) % 5 + 5 * y) + h]);
            }
        }
    }
    s[0] ^= rc_lo;
    s[1] ^= rc_hi;
}

// ------------------------------------------------------- two-phase rounds
//
// Rotates (v_alignbit) and simple instructions of different waves issue
// together when a wave in its rotates is picked first (sha2_dev.hpp says
// how): theta's rotates by one and rho are asm blocks between s_setprio 3 and
// s_setprio 0, the xors and chi run at priority 0 beside other waves'
// rotates.  The empty asm blocks keep theta's xors before rho's run.  The F
// step of a chain, G permutations/s at 1 / 2 / 4 / 5 waves per SIMD:
// interleaved 7.4 / 9.0 / 10.4 / 10.5 -> 8.4 / 13.1 / 14.4 / 14.6.

#define SPX_AL(d, h, l, n) "v_alignbit_b32 %" #d ", %" #h ", %" #l ", %" #n "\n\t"
#define SPX_AL1(d, h, l) "v_alignbit_b32 %" #d ", %" #h ", %" #l ", 31\n\t"
#define SPX_PIN10(v, i)                                                                  \
    asm volatile(""                                                                      \
                 : "+v"(v[i]), "+v"(v[i + 1]), "+v"(v[i + 2]), "+v"(v[i + 3]),           \
                   "+v"(v[i + 4]), "+v"(v[i + 5]), "+v"(v[i + 6]), "+v"(v[i + 7]),       \
                   "+v"(v[i + 8]), "+v"(v[i + 9]))

// theta's column parities
__device__ __forceinline__ void keccak_parity(const uint32_t s[50], uint32_t C[10]) {
#pragma unroll
    for (int i = 0; i < 10; i++)
        C[i] = xor3(xor3(s[i], s[i + 10], s[i + 20]), s[i + 30], s[i + 40]);
}
// chi and iota on the rotated lanes B
__device__ __forceinline__ void keccak_chi(uint32_t s[50], const uint32_t B[50], uint32_t rc0,
                                           uint32_t rc1) {
#pragma unroll
    for (int y = 0; y < 5; y++)
#pragma unroll
        for (int x = 0; x < 5; x++)
#pragma unroll
            for (int h = 0; h < 2; h++)
                s[2 * (x + 5 * y) + h] = bit_chi(B[2 * (x + 5 * y) + h],
                                                 B[2 * ((x + 1) % 5 + 5 * y) + h],
                                                 B[2 * ((x + 2) % 5 + 5 * y) + h]);
    s[0] ^= rc0;
    s[1] ^= rc1;
}

// v_alignbit count and half order of rho's rotate of lane l: out = (lo, hi)
// by alignbit(hi, lo, n) and alignbit(lo, hi, n), swapped for rotates over 32
constexpr int keccak_rho_count(int l) { return (64 - kRho[l]) & 31; }
constexpr bool keccak_rho_swap(int l) { return kRho[l] > 32; }

// one round on s[50] (low, high words)
__device__ __forceinline__ void keccak_round_ph(uint32_t s[50], uint32_t rc_lo, uint32_t rc_hi) {
    uint32_t C[10], R[10];  // R = C rotated by one
    keccak_parity(s, C);
    asm volatile(SPX_HI SPX_AL1(0, 10, 11) SPX_AL1(1, 11, 10) SPX_AL1(2, 12, 13)
                     SPX_AL1(3, 13, 12) SPX_AL1(4, 14, 15) SPX_AL1(5, 15, 14)
                         SPX_AL1(6, 16, 17) SPX_AL1(7, 17, 16) SPX_AL1(8, 18, 19)
                             SPX_AL1(9, 19, 18) SPX_LO
                 : "=&v"(R[0]), "=&v"(R[1]), "=&v"(R[2]), "=&v"(R[3]), "=&v"(R[4]), "=&v"(R[5]),
                   "=&v"(R[6]), "=&v"(R[7]), "=&v"(R[8]), "=&v"(R[9])
                 : "v"(C[0]), "v"(C[1]), "v"(C[2]), "v"(C[3]), "v"(C[4]), "v"(C[5]), "v"(C[6]),
                   "v"(C[7]), "v"(C[8]), "v"(C[9]));
#pragma unroll
    for (int i = 0; i < 50; i++) {
        const int x = (i % 10) / 2, h = i & 1;
        s[i] = xor3(s[i], C[2 * ((x + 4) % 5) + h], R[2 * ((x + 1) % 5) + h]);
    }
    SPX_PIN10(s, 0);
    SPX_PIN10(s, 10);
    SPX_PIN10(s, 20);
    SPX_PIN10(s, 30);
    SPX_PIN10(s, 40);
    uint32_t B[50];
    // rho of lanes l .. l + 3 into q, then pi
#define SPX_RHO4(pre, post, l)                                                           \
    do {                                                                                 \
        uint32_t q[8];                                                                   \
        asm volatile(pre SPX_AL(0, 9, 8, 16) SPX_AL(1, 8, 9, 16) SPX_AL(2, 11, 10, 17)   \
                         SPX_AL(3, 10, 11, 17) SPX_AL(4, 13, 12, 18) SPX_AL(5, 12, 13, 18) \
                             SPX_AL(6, 15, 14, 19) SPX_AL(7, 14, 15, 19) post            \
                     : "=&v"(q[0]), "=&v"(q[1]), "=&v"(q[2]), "=&v"(q[3]), "=&v"(q[4]),  \
                       "=&v"(q[5]), "=&v"(q[6]), "=&v"(q[7])                             \
                     : "v"(s[2 * (l)]), "v"(s[2 * (l) + 1]), "v"(s[2 * (l) + 2]),        \
                       "v"(s[2 * (l) + 3]), "v"(s[2 * (l) + 4]), "v"(s[2 * (l) + 5]),    \
                       "v"(s[2 * (l) + 6]), "v"(s[2 * (l) + 7]),                         \
                       "i"(keccak_rho_count(l)), "i"(keccak_rho_count((l) + 1)),         \
                       "i"(keccak_rho_count((l) + 2)), "i"(keccak_rho_count((l) + 3)));  \
        _Pragma("unroll") for (int i = 0; i < 4; i++) {                                  \
            const int src = (l) + i, x = src % 5, y = src / 5;                           \
            const int dst = y + 5 * ((2 * x + 3 * y) % 5);                               \
            const int w = keccak_rho_swap(src) ? 0 : 1;                                  \
            B[2 * dst] = q[2 * i + w];                                                   \
            B[2 * dst + 1] = q[2 * i + 1 - w];                                           \
        }                                                                                \
    } while (0)
    B[0] = s[0];
    B[1] = s[1];
    SPX_RHO4(SPX_HI, "", 1);
    SPX_RHO4("", "", 5);
    SPX_RHO4("", "", 9);
    SPX_RHO4("", "", 13);
    SPX_RHO4("", "", 17);
    SPX_RHO4("", SPX_LO, 21);
#undef SPX_RHO4
    keccak_chi(s, B, rc_lo, rc_hi);
}

// Keccak-f[1600] of which only the first words are used: the last round is left
// to the compiler, which drops what those do not need (about 50 of its 180
// instructions stay for a 16-byte output)
__device__ __forceinline__ void keccak_f(uint32_t s[50]) {
    keccak_round_ph(s, 0x00000001u, 0x00000000u);
#pragma unroll 1
    for (int r = 1; r < 23; r += 2) {
        keccak_round_ph(s, kKeccakRC[2 * r], kKeccakRC[2 * r + 1]);
        keccak_round_ph(s, kKeccakRC[2 * r + 2], kKeccakRC[2 * r + 3]);
    }
    keccak_round(s, 0x80008008u, 0x80000000u);
}

// ---------------------------------------------------- bit-interleaved form
//
// A 64-bit lane (lo, hi) can also be held as (E, O): E = its even-numbered
// bits, O = its odd-numbered bits.  A 64-bit rotation by 2k is then a 32-bit
// rotation of both halves by k, and by 2k+1 a swap plus rotations by k+1 and
// k -- theta's rotation by 1 costs one v_alignbit instead of two, and so does
// rho's rotation by 1: 52 instead of 58 rotates per round.  The WOTS chain
// steps of the hypertree kernel run in this form (values stay interleaved
// from step to step); everything else uses the plain form.

// bits 0, 2, 4, ... of x into bits 0..15
__device__ __forceinline__ uint32_t il_even16(uint32_t x) {
    x &= 0x55555555u;
    x = (x | (x >> 1)) & 0x33333333u;
    x = (x | (x >> 2)) & 0x0F0F0F0Fu;
    x = (x | (x >> 4)) & 0x00FF00FFu;
    return (x | (x >> 8)) & 0x0000FFFFu;
}
// bits 0..15 of x into bits 0, 2, 4, ...
__device__ __forceinline__ uint32_t il_spread16(uint32_t x) {
    x &= 0x0000FFFFu;
    x = (x | (x << 8)) & 0x00FF00FFu;
    x = (x | (x << 4)) & 0x0F0F0F0Fu;
    x = (x | (x << 2)) & 0x33333333u;
    return (x | (x << 1)) & 0x55555555u;
}
// (lo, hi) -> (E, O)
__device__ __forceinline__ void il_to(uint32_t lo, uint32_t hi, uint32_t& e, uint32_t& o) {
    e = il_even16(lo) | (il_even16(hi) << 16);
    o = il_even16(lo >> 1) | (il_even16(hi >> 1) << 16);
}
// E (h = 0) or O (h = 1) of (lo, hi)
__device__ __forceinline__ uint32_t il_half(uint32_t lo, uint32_t hi, uint32_t h) {
    return il_even16(lo >> h) | (il_even16(hi >> h) << 16);
}
// (E, O) -> (lo, hi)
__device__ __forceinline__ void il_from(uint32_t e, uint32_t o, uint32_t& lo, uint32_t& hi) {
    lo = il_spread16(e) | (il_spread16(o) << 1);
    hi = il_spread16(e >> 16) | (il_spread16(o >> 16) << 1);
}

// rotl32 by M (M in 0..32)
template <int M>
__device__ __forceinline__ uint32_t rotl32c(uint32_t x) {
    if constexpr (M == 0 || M == 32) return x;
    else return __builtin_amdgcn_alignbit(x, x, 32 - M);
}

// 64-bit rotation by R of an interleaved lane
template <int R>
__device__ __forceinline__ void rol64_il(uint32_t e, uint32_t o, uint32_t& oe, uint32_t& oo) {
    if constexpr ((R & 1) == 0) {
        oe = rotl32c<R / 2>(e);
        oo = rotl32c<R / 2>(o);
    } else {
        oe = rotl32c<(R + 1) / 2>(o);
        oo = rotl32c<(R - 1) / 2>(e);
    }
}

// round constants in interleaved form: (E, O) of each 64-bit constant
struct KeccakRcIl {
    uint32_t w[48];
    constexpr KeccakRcIl() : w{} {
        constexpr uint64_t rc[24] = {
            0x0000000000000001ull, 0x0000000000008082ull, 0x800000000000808aull,
            0x8000000080008000ull, 0x000000000000808bull, 0x0000000080000001ull,
            0x8000000080008081ull, 0x8000000000008009ull, 0x000000000000008aull,
            0x0000000000000088ull, 0x0000000080008009ull, 0x000000008000000aull,
            0x000000008000808bull, 0x800000000000008bull, 0x8000000000008089ull,
            0x8000000000008003ull, 0x8000000000008002ull, 0x8000000000000080ull,
            0x000000000000800aull, 0x800000008000000aull, 0x8000000080008081ull,
            0x8000000000008080ull, 0x0000000080000001ull, 0x8000000080008008ull};
        for (int r = 0; r < 24; r++) {
            uint32_t e = 0, o = 0;
            for (int b = 0; b < 32; b++) {
                e |= (uint32_t)((rc[r] >> (2 * b)) & 1u) << b;
                o |= (uint32_t)((rc[r] >> (2 * b + 1)) & 1u) << b;
            }
            w[2 * r] = e;
            w[2 * r + 1] = o;
        }
    }
};
__constant__ KeccakRcIl kKeccakRcIl = KeccakRcIl();

// one round on the interleaved state (s[2i] = E, s[2i+1] = O of lane i)
__device__ __forceinline__ void keccak_round_il(uint32_t s[50], uint32_t rc_e, uint32_t rc_o) {
    uint32_t C[10];
#pragma unroll
    for (int x = 0; x < 5; x++) {
#pragma unroll
        for (int h = 0; h < 2; h++) {
            C[2 * x + h] = xor3(xor3(s[2 * x + h], s[2 * (x + 5) + h], s[2 * (x + 10) + h]),
                                s[2 * (x + 15) + h], s[2 * (x + 20) + h]);
        }
    }
#pragma unroll
    for (int x = 0; x < 5; x++) {
        const int xp = (x + 1) % 5, xm = (x + 4) % 5;
        const uint32_t re = rotl32c<1>(C[2 * xp + 1]), ro = C[2 * xp];  // rol64 by 1
#pragma unroll
        for (int y = 0; y < 5; y++) {
            s[2 * (x + 5 * y)] = xor3(s[2 * (x + 5 * y)], C[2 * xm], re);
            s[2 * (x + 5 * y) + 1] = xor3(s[2 * (x + 5 * y) + 1], C[2 * xm + 1], ro);
        }
    }
    uint32_t B[50];
#pragma unroll
    for (int x = 0; x < 5; x++) {
#pragma unroll
        for (int y = 0; y < 5; y++) {
            const int src = x + 5 * y;
            const int dst = y + 5 * ((2 * x + 3 * y) % 5);
            uint32_t e, o;
            switch (kRho[src]) {
#define SPX_ROT_CASE(R) \
    case R: rol64_il<R>(s[2 * src], s[2 * src + 1], e, o); break;
                SPX_ROT_CASE(0) SPX_ROT_CASE(1) SPX_ROT_CASE(62) SPX_ROT_CASE(28)
                SPX_ROT_CASE(27) SPX_ROT_CASE(36) SPX_ROT_CASE(44) SPX_ROT_CASE(6)
                SPX_ROT_CASE(55) SPX_ROT_CASE(20) SPX_ROT_CASE(3) SPX_ROT_CASE(10)
                SPX_ROT_CASE(43) SPX_ROT_CASE(25) SPX_ROT_CASE(39) SPX_ROT_CASE(41)
                SPX_ROT_CASE(45) SPX_ROT_CASE(15) SPX_ROT_CASE(21) SPX_ROT_CASE(8)
                SPX_ROT_CASE(18) SPX_ROT_CASE(2) SPX_ROT_CASE(61) SPX_ROT_CASE(56)
                SPX_ROT_CASE(14)
#undef SPX_ROT_CASE
                default: e = s[2 * src]; o = s[2 * src + 1]; break;
            }
            B[2 * dst] = e;
            B[2 * dst + 1] = o;
        }
    }
#pragma unroll
    for (int y = 0; y < 5; y++) {
#pragma unroll
        for (int x = 0; x < 5; x++) {
#pragma unroll
            for (int h = 0; h < 2; h++) {
                s[2 * (x + 5 * y) + h] = bit_chi(B[2 * (x + 5 * y) + h],
                                                 B[2 * ((x + 1) % 5 + 5 * y) + h],
                                                 B[2 * ((x + 2) % 5 + 5 * y) + h]);
            }
        }
    }
    s[0] ^= rc_e;
    s[1] ^= rc_o;
}

// the same round in two phases (keccak_round_ph): 52 rotates, all in place.
// Word j (half j & 1 of lane j / 2) is rotated left by keccak_il_rot(j); odd
// rotations swap the halves, which pi's renaming does.
constexpr int keccak_il_rot(int j) {
    const int r = kRho[j >> 1];
    return (r & 1) == 0 ? r / 2 : (j & 1) ? (r + 1) / 2 : (r - 1) / 2;
}
constexpr int keccak_il_count(int j) { return (32 - keccak_il_rot(j)) & 31; }
static_assert(keccak_il_rot(0) == 0 && keccak_il_rot(1) == 0 && keccak_il_rot(2) == 0,
              "words 3..49 rotate");

__device__ __forceinline__ void keccak_round_il_ph(uint32_t s[50], uint32_t rc_e, uint32_t rc_o) {
    uint32_t C[10], R[5];  // R[x] = odd half of column x rotated by one
    keccak_parity(s, C);
    asm volatile(SPX_HI SPX_AL1(0, 5, 5) SPX_AL1(1, 6, 6) SPX_AL1(2, 7, 7)
                     SPX_AL1(3, 8, 8) SPX_AL1(4, 9, 9) SPX_LO
                 : "=&v"(R[0]), "=&v"(R[1]), "=&v"(R[2]), "=&v"(R[3]), "=&v"(R[4])
                 : "v"(C[1]), "v"(C[3]), "v"(C[5]), "v"(C[7]), "v"(C[9]));
#pragma unroll
    for (int l = 0; l < 25; l++) {
        const int x = l % 5, xp = (x + 1) % 5, xm = (x + 4) % 5;
        s[2 * l] = xor3(s[2 * l], C[2 * xm], R[xp]);
        s[2 * l + 1] = xor3(s[2 * l + 1], C[2 * xm + 1], C[2 * xp]);
    }
    SPX_PIN10(s, 0);
    SPX_PIN10(s, 10);
    SPX_PIN10(s, 20);
    SPX_PIN10(s, 30);
    SPX_PIN10(s, 40);
#define SPX_SV(i) "+v"(s[i])
#define SPX_SN(i) "i"(keccak_il_count(i))
#define SPX_RHO10(pre, i)                                                                \
    asm volatile(pre SPX_AL(0, 0, 0, 10) SPX_AL(1, 1, 1, 11) SPX_AL(2, 2, 2, 12)         \
                     SPX_AL(3, 3, 3, 13) SPX_AL(4, 4, 4, 14) SPX_AL(5, 5, 5, 15)         \
                         SPX_AL(6, 6, 6, 16) SPX_AL(7, 7, 7, 17) SPX_AL(8, 8, 8, 18)     \
                             SPX_AL(9, 9, 9, 19)                                         \
                 : SPX_SV(i), SPX_SV(i + 1), SPX_SV(i + 2), SPX_SV(i + 3), SPX_SV(i + 4), \
                   SPX_SV(i + 5), SPX_SV(i + 6), SPX_SV(i + 7), SPX_SV(i + 8), SPX_SV(i + 9) \
                 : SPX_SN(i), SPX_SN(i + 1), SPX_SN(i + 2), SPX_SN(i + 3), SPX_SN(i + 4), \
                   SPX_SN(i + 5), SPX_SN(i + 6), SPX_SN(i + 7), SPX_SN(i + 8), SPX_SN(i + 9))
    SPX_RHO10(SPX_HI, 3);
    SPX_RHO10("", 13);
    SPX_RHO10("", 23);
    SPX_RHO10("", 33);
    asm volatile(SPX_AL(0, 0, 0, 7) SPX_AL(1, 1, 1, 8) SPX_AL(2, 2, 2, 9) SPX_AL(3, 3, 3, 10)
                     SPX_AL(4, 4, 4, 11) SPX_AL(5, 5, 5, 12) SPX_AL(6, 6, 6, 13) SPX_LO
                 : SPX_SV(43), SPX_SV(44), SPX_SV(45), SPX_SV(46), SPX_SV(47), SPX_SV(48), SPX_SV(49)
                 : SPX_SN(43), SPX_SN(44), SPX_SN(45), SPX_SN(46), SPX_SN(47), SPX_SN(48), SPX_SN(49));
#undef SPX_RHO10
#undef SPX_SV
#undef SPX_SN
    SPX_PIN10(s, 0);
    SPX_PIN10(s, 10);
    SPX_PIN10(s, 20);
    SPX_PIN10(s, 30);
    SPX_PIN10(s, 40);
    uint32_t B[50];
#pragma unroll
    for (int l = 0; l < 25; l++) {
        const int x = l % 5, y = l / 5, dst = y + 5 * ((2 * x + 3 * y) % 5);
        const int w = kRho[l] & 1;
        B[2 * dst] = s[2 * l + w];
        B[2 * dst + 1] = s[2 * l + 1 - w];
    }
    keccak_chi(s, B, rc_e, rc_o);
}

// Keccak-f[1600] on the interleaved state.  HEAD: only the first words of
// the result are used, so the last round is left to the compiler, which drops
// the rest of it (see keccak_f); else all of it is.
template <bool HEAD>
__device__ __forceinline__ void keccak_f_il(uint32_t s[50]) {
    keccak_round_il_ph(s, 1u, 0u);  // RC[0] = 1: bit 0 is even
#pragma unroll 1
    for (int r = 1; r < 23; r += 2) {
        keccak_round_il_ph(s, kKeccakRcIl.w[2 * r], kKeccakRcIl.w[2 * r + 1]);
        keccak_round_il_ph(s, kKeccakRcIl.w[2 * r + 2], kKeccakRcIl.w[2 * r + 3]);
    }
    if constexpr (HEAD) keccak_round_il(s, kKeccakRcIl.w[46], kKeccakRcIl.w[47]);
    else keccak_round_il_ph(s, kKeccakRcIl.w[46], kKeccakRcIl.w[47]);
}

// Keccak-f[1600] on a lane pair in the interleaved form: the even lane holds
// the E halves of the 25 lanes, the odd lane the O halves (s[i] = this
// lane's half of Keccak lane i).  A rotation by 2k rotates both halves by k
// (no exchange); a rotation by 2k + 1 swaps them (one DPP move) and rotates
// by k + 1 (even lane) or k (odd lane), a per-lane count.  Theta's column
// sums, chi and iota stay within a half.  128 instructions per round on
// each lane (in the built ISA) against 174 for the whole state on one lane:
// for serial sponges whose lane would otherwise run alone.
__device__ __forceinline__ void keccak_round_il_pair(uint32_t s[25], uint32_t m, uint32_t rc) {
    uint32_t C[5];
#pragma unroll
    for (int x = 0; x < 5; x++) C[x] = xor3(xor3(s[x], s[x + 5], s[x + 10]), s[x + 15], s[x + 20]);
    const uint32_t sh1 = lane_sel(m, 0u, 31u);  // rotl by 1 (E) or 0 (O) after the swap
#pragma unroll
    for (int x = 0; x < 5; x++) {
        const uint32_t t = pair_swap(C[(x + 1) % 5]);
        const uint32_t r = __builtin_amdgcn_alignbit(t, t, sh1);  // rol64(C[x+1], 1), this half
#pragma unroll
        for (int y = 0; y < 5; y++) s[x + 5 * y] = xor3(s[x + 5 * y], C[(x + 4) % 5], r);
    }
    uint32_t B[25];
#pragma unroll
    for (int x = 0; x < 5; x++) {
#pragma unroll
        for (int y = 0; y < 5; y++) {
            const int src = x + 5 * y;
            const int dst = y + 5 * ((2 * x + 3 * y) % 5);
            const int R = kRho[src];
            uint32_t v;
            if (R == 0) {
                v = s[src];
            } else if ((R & 1) == 0) {
                v = __builtin_amdgcn_alignbit(s[src], s[src], (32 - R / 2) & 31);
            } else {
                const uint32_t t = pair_swap(s[src]);
                const uint32_t sh = lane_sel(m, (uint32_t)((32 - R / 2) & 31),
                                             (uint32_t)((31 - R / 2) & 31));
                v = __builtin_amdgcn_alignbit(t, t, sh);
            }
            B[dst] = v;
        }
    }
#pragma unroll
    for (int y = 0; y < 5; y++)
#pragma unroll
        for (int x = 0; x < 5; x++)
            s[x + 5 * y] = bit_chi(B[x + 5 * y], B[(x + 1) % 5 + 5 * y], B[(x + 2) % 5 + 5 * y]);
    s[0] ^= rc;
}

__device__ __forceinline__ void keccak_f_il_pair(uint32_t s[25]) {
    const uint32_t m = (threadIdx.x & 1u) ? ~0u : 0u;
    keccak_round_il_pair(s, m, lane_sel(m, 0u, 1u));  // RC[0] = 1: bit 0 is even
#pragma unroll 1
    for (int r = 1; r < 24; r++)
        keccak_round_il_pair(s, m, lane_sel(m, kKeccakRcIl.w[2 * r + 1], kKeccakRcIl.w[2 * r]));
}

// ---------------------------------------------------------- sixteen lanes
//
// One Keccak-f[1600] on a row of 16 lanes (all active), for serial sponges:
// a wave alone on its SIMD issues an instruction every 4-5 cycles whatever it
// holds, so a permutation costs what its instruction stream is long.  Lane p
// < 7 holds the even-bit halves of one column, lane p + 8 the odd-bit halves:
// s[y] = lane (x, y) with x = (p + 4) % 5.  Positions 0 and 6 repeat columns
// 4 and 0 so that theta's two neighbours (x - 1, same half; x + 1, other half
// rotated by one) are fixed DPP row moves; 7 and 15 idle.  After rho (a rotate
// count per lane and row) every word goes through LDS to its place under pi,
// and each lane reads its new column and the two after it, which chi needs.
// 35 instructions (21 VALU, 11 LDS) and one LDS round trip per round, against 128
// instructions on a lane pair.
struct Keccak16Tab {
    uint8_t rot[16][5];   // v_alignbit count of row y
    uint8_t wr[16][5];    // word written by row y
    uint8_t rd[16][3];    // first word of columns x, x + 1, x + 2
    constexpr Keccak16Tab() : rot{}, wr{}, rd{} {
        for (int p = 0; p < 16; p++) {
            const int h = p >> 3, q = p & 7, x = (q + 4) % 5;
            const bool owner = q >= 1 && q <= 5;
            for (int y = 0; y < 5; y++) {
                const int r = kRho[x + 5 * y];
                const int n = (r & 1) == 0 ? r / 2 : h ? (r + 1) / 2 : (r - 1) / 2;
                const int h2 = h ^ (r & 1);  // odd rotations swap the halves
                rot[p][y] = (uint8_t)((32 - n) & 31);
                // column y, row 2x + 3y; the repeated columns write aside
                wr[p][y] = (uint8_t)(owner ? (h2 * 5 + y) * 8 + 4 * h2 + (2 * x + 3 * y) % 5 : 84 + p);
            }
            for (int k = 0; k < 3; k++) rd[p][k] = (uint8_t)((h * 5 + (x + k) % 5) * 8 + 4 * h);
        }
    }
};
__constant__ Keccak16Tab kKeccak16 = Keccak16Tab();

struct Keccak16 {
    static constexpr int kLanes = 16;
    // per row of 16 lanes, 16-byte aligned.  Columns are 8 words apart, the odd
    // halves 4 words further, and rows an odd multiple of 16 words, so that
    // the four rows of a wave start in different banks (of 5.6 LDS cycles per
    // access SQ_LDS_BANK_CONFLICT still counts 3.0).
    static constexpr int kLdsWords = 112;
    static constexpr int row_words(int w) { return ((w + 15) / 16 | 1) * 16; }
    typedef uint32_t __attribute__((address_space(3))) lds_word;
    typedef uint32_t v4 __attribute__((ext_vector_type(4)));
    typedef v4 __attribute__((address_space(3))) lds_v4;

    uint32_t s[5];
    uint32_t rot[5];
    lds_word* wr[5];
    lds_word* rd[3];
    lds_word* base;
    uint32_t me, mo;  // iota: all ones where column 0's even / odd half is held
    uint32_t sh1;     // theta's rotate by one (even half)
    uint32_t half;
    int col;

    __device__ __forceinline__ void init(lds_word* row) {
        const int p = threadIdx.x & 15;
        half = p >> 3;
        col = ((p & 7) + 4) % 5;
        base = row;
#pragma unroll
        for (int y = 0; y < 5; y++) {
            rot[y] = kKeccak16.rot[p][y];
            wr[y] = row + kKeccak16.wr[p][y];
        }
#pragma unroll
        for (int k = 0; k < 3; k++) rd[k] = row + kKeccak16.rd[p][k];
        me = (col == 0 && !half) ? ~0u : 0u;
        mo = (col == 0 && half) ? ~0u : 0u;
        sh1 = half ? 0u : 31u;
        clear();
    }
    __device__ __forceinline__ void clear() {
#pragma unroll
        for (int y = 0; y < 5; y++) s[y] = 0;
    }
    // s[0] is lane (col, 0) and not a repeated column
    __device__ static __forceinline__ bool own0() { return (threadIdx.x & 7u) - 1u < 5u; }
    // LDS words written by other lanes of the row are read next: keep the order
    __device__ static __forceinline__ void order() {
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        __builtin_amdgcn_wave_barrier();
    }
    __device__ __forceinline__ void round(uint32_t rc_e, uint32_t rc_o) {
        const uint32_t C = xor3(xor3(s[0], s[1], s[2]), s[3], s[4]);
        // lane p - 1 (row_shr 1): column x - 1; lane p + 9 (row_ror 7): the
        // other half of column x + 1
        const uint32_t cm = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)C, 0x111, 0xF, 0xF, true);
        const uint32_t t = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)C, 0x127, 0xF, 0xF, true);
        const uint32_t cp = __builtin_amdgcn_alignbit(t, t, sh1);
#pragma unroll
        for (int y = 0; y < 5; y++) {
            const uint32_t u = xor3(s[y], cm, cp);
            *wr[y] = __builtin_amdgcn_alignbit(u, u, rot[y]);
        }
        order();
        v4 b[3];
        uint32_t b4[3];
#pragma unroll
        for (int k = 0; k < 3; k++) {
            b[k] = *(const lds_v4*)rd[k];
            b4[k] = rd[k][4];
        }
        order();
        const uint32_t rc = (me & rc_e) | (mo & rc_o);
#pragma unroll
        for (int y = 0; y < 4; y++) s[y] = bit_chi(b[0][y], b[1][y], b[2][y]);
        s[4] = bit_chi(b4[0], b4[1], b4[2]);
        s[0] ^= rc;
    }
    __device__ __forceinline__ void permute() {
        constexpr KeccakRcIl rc;  // as literals: no scalar load waits among the LDS reads
#pragma unroll
        for (int r = 0; r < 24; r++) round(rc.w[2 * r], rc.w[2 * r + 1]);
    }
    // this half of a 64-bit lane (lo, hi)
    __device__ __forceinline__ uint32_t split(uint32_t lo, uint32_t hi) const {
        return il_half(lo, hi, half);
    }
    // Keccak lane l of the state (l < 25), interleaved or plain, in every
    // lane of the row
    __device__ __forceinline__ void lane_il(int l, uint32_t& e, uint32_t& o) const {
        const int at = (threadIdx.x & 48) + 1 + l % 5;
        e = (uint32_t)__builtin_amdgcn_ds_bpermute(4 * at, (int)s[l / 5]);
        o = (uint32_t)__builtin_amdgcn_ds_bpermute(4 * (at + 8), (int)s[l / 5]);
    }
    __device__ __forceinline__ void lane(int l, uint32_t& lo, uint32_t& hi) const {
        uint32_t e, o;
        lane_il(l, e, o);
        il_from(e, o, lo, hi);
    }
    // Absorb rate block b of a stream held in LDS as interleaved words (E, O
    // of 64-bit lane i at buf[2 i], buf[2 i + 1]; whole blocks, padded)
    __device__ __forceinline__ void absorb(const lds_word* buf, int b) {
#pragma unroll
        for (int y = 0; y < 4; y++) {
            const int l = col + 5 * y;
            if (l < 17) s[y] ^= buf[2 * (17 * b + l) + half];
        }
    }
};

// The same on two such rows, 32 lanes: the first holds rows y = 0, 1, 2 of the
// columns in s, the second rows 3 and 4 (and a zero), and the column parities
// are put together by swapping the rows (v_permlane16_swap).  26 instructions
// (17 VALU, 6 LDS) per round.  A permutation alone on its SIMD: 5.5 us on a lane
// pair, 2.50 on 16 lanes, 2.12 on 32; four waves per CU 2.86 and 2.47.
struct Keccak32Tab {
    uint8_t rot[32][3], wr[32][3], rd[32][3];  // as Keccak16Tab
    // column (h, x): 8 words, rows 0-2 in one half and 3, 4 in the other
    static constexpr int at(int h, int x, int y) {
        return (h * 5 + x) * 8 + ((4 * h) ^ (y < 3 ? y : y + 1));
    }
    constexpr Keccak32Tab() : rot{}, wr{}, rd{} {
        for (int p = 0; p < 32; p++) {
            const int g = p >> 4, h = (p >> 3) & 1, q = p & 7, x = (q + 4) % 5;
            const bool owner = q >= 1 && q <= 5;
            for (int i = 0; i < 3; i++) {
                const int y = i + 3 * g;
                const int r = kRho[x + 5 * (y < 5 ? y : 0)];
                const int n = (r & 1) == 0 ? r / 2 : h ? (r + 1) / 2 : (r - 1) / 2;
                const int h2 = h ^ (r & 1);
                rot[p][i] = (uint8_t)((32 - n) & 31);
                wr[p][i] = (uint8_t)(owner && y < 5 ? at(h2, y, (2 * x + 3 * y) % 5) : 80 + p);
            }
            for (int k = 0; k < 3; k++) rd[p][k] = (uint8_t)((h * 5 + (x + k) % 5) * 8 + 4 * (g ^ h));
        }
    }
};
__constant__ Keccak32Tab kKeccak32 = Keccak32Tab();

struct Keccak32 {
    static constexpr int kLanes = 32;
    static constexpr int kLdsWords = 112;  // per 32 lanes, 16-byte aligned; as Keccak16
    static constexpr int row_words(int w) { return Keccak16::row_words(w); }
    typedef Keccak16::lds_word lds_word;
    typedef Keccak16::v4 v4;
    typedef Keccak16::lds_v4 lds_v4;

    uint32_t s[3];    // lanes (col, row + i)
    uint32_t rot[3];
    lds_word* wr[3];
    lds_word* rd[3];
    lds_word* base;
    uint32_t me, mo;  // as Keccak16
    uint32_t sh1, half;
    int col, row;

    __device__ __forceinline__ void init(lds_word* lds) {
        const int p = threadIdx.x & 31;
        half = (p >> 3) & 1;
        col = ((p & 7) + 4) % 5;
        row = 3 * (p >> 4);
        base = lds;
#pragma unroll
        for (int i = 0; i < 3; i++) {
            rot[i] = kKeccak32.rot[p][i];
            wr[i] = lds + kKeccak32.wr[p][i];
            rd[i] = lds + kKeccak32.rd[p][i];
        }
        me = (col == 0 && row == 0 && !half) ? ~0u : 0u;
        mo = (col == 0 && row == 0 && half) ? ~0u : 0u;
        sh1 = half ? 0u : 31u;
        clear();
        // the third words of rows 3, 4 are read, and stay zero
#pragma unroll
        for (int i = 0; i < kLdsWords; i += 16) lds[i + (p & 15)] = 0;
        order();
    }
    __device__ __forceinline__ void clear() {
#pragma unroll
        for (int i = 0; i < 3; i++) s[i] = 0;
    }
    __device__ static __forceinline__ bool own0() {
        return (threadIdx.x & 7u) - 1u < 5u && (threadIdx.x & 16u) == 0;
    }
    __device__ static __forceinline__ void order() { Keccak16::order(); }
    __device__ __forceinline__ void round(uint32_t rc_e, uint32_t rc_o) {
        const uint32_t part = xor3(s[0], s[1], s[2]);
        const auto sw = __builtin_amdgcn_permlane16_swap(part, part, false, false);
        const uint32_t C = sw[0] ^ sw[1];
        const uint32_t cm = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)C, 0x111, 0xF, 0xF, true);
        const uint32_t t = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)C, 0x127, 0xF, 0xF, true);
        const uint32_t cp = __builtin_amdgcn_alignbit(t, t, sh1);
#pragma unroll
        for (int i = 0; i < 3; i++) {
            const uint32_t u = xor3(s[i], cm, cp);
            *wr[i] = __builtin_amdgcn_alignbit(u, u, rot[i]);
        }
        order();
        v4 b[3];
#pragma unroll
        for (int k = 0; k < 3; k++) b[k] = *(const lds_v4*)rd[k];
        order();
        const uint32_t rc = (me & rc_e) | (mo & rc_o);
#pragma unroll
        for (int i = 0; i < 3; i++) s[i] = bit_chi(b[0][i], b[1][i], b[2][i]);
        s[0] ^= rc;
    }
    __device__ __forceinline__ void permute() {
        constexpr KeccakRcIl rc;
#pragma unroll
        for (int r = 0; r < 24; r++) round(rc.w[2 * r], rc.w[2 * r + 1]);
    }
    __device__ __forceinline__ uint32_t split(uint32_t lo, uint32_t hi) const {
        return il_half(lo, hi, half);
    }
    __device__ __forceinline__ void lane(int l, uint32_t& lo, uint32_t& hi) const {
        const int g = l >= 15, i = l / 5 - 3 * g;
        const int at = (threadIdx.x & 32) + 16 * g + 1 + l % 5;
        const uint32_t e = (uint32_t)__builtin_amdgcn_ds_bpermute(4 * at, (int)s[i]);
        const uint32_t o = (uint32_t)__builtin_amdgcn_ds_bpermute(4 * (at + 8), (int)s[i]);
        il_from(e, o, lo, hi);
    }
    __device__ __forceinline__ void absorb(const lds_word* buf, int b) {
#pragma unroll
        for (int i = 0; i < 3; i++) {
            const int l = col + 5 * (row + i);
            if (l < 17) s[i] ^= buf[2 * (17 * b + l) + half];
        }
    }
};

template <int N>
struct Shake {
    static constexpr int hash = kShake;
    static constexpr int NW = N / 4;

    struct Key {
        uint32_t pub[NW];
        uint32_t sk[NW];
    };

    __device__ static __forceinline__ void load_key(const Plan& p, Key& k) {
#pragma unroll
        for (int i = 0; i < NW; i++) {
            k.pub[i] = p.pubseed[i];
            k.sk[i] = p.skseed[i];
        }
    }

    // address byte-words (big-endian) as sponge words (little-endian)
    __device__ static __forceinline__ uint32_t aw(const Adr& a, int i) {
        return i < 6 ? bswap32(a.w[i]) : 0u;
    }

    // single-permutation SHAKE256 over pre(NW) || addr32 || d(M), output n
    template <int M>
    __device__ static __forceinline__ void one_block(const uint32_t pre[NW], const Adr& a,
                                                     const uint32_t* d, uint32_t out[NW]) {
        constexpr int L = NW + 8 + M;  // input words
        static_assert(4 * L <= 135, "input must fit one block");
        uint32_t s[50];
#pragma unroll
        for (int i = 0; i < 50; i++) {
            uint32_t x = 0;
            if (i < NW) x = pre[i];
            else if (i < NW + 8) x = aw(a, i - NW);
            else if (i < L) x = d[i - NW - 8];
            if (i == L) x ^= 0x1Fu;
            if (i == 33) x ^= 0x80000000u;
            s[i] = x;
        }
        keccak_f(s);
#pragma unroll
        for (int i = 0; i < NW; i++) out[i] = s[i];
    }

    __device__ static __forceinline__ void F(const Key& k, const Adr& a, const uint32_t in[NW],
                                             uint32_t out[NW]) {
        one_block<NW>(k.pub, a, in, out);
    }

    // WOTS chain in the interleaved form: pub_seed and the chain's address
    // (hash field 0) are interleaved once; each step adds the hash field --
    // address byte 21, bits 40..43 of sponge lane (n + 21) / 8 -- by xor,
    // which commutes with interleaving.  Values in and out are interleaved.
    static constexpr int kHashLane = (N + 21) / 8;
    static constexpr int kPadLane = (2 * N + 32) / 8;  // the 0x1F byte, at a lane start
    struct ChainIl {
        uint32_t w[NW + 8];  // (E, O) of the pub_seed and address lanes
    };
    __device__ static __forceinline__ void chain_il_begin(const Key& k, const Adr& a,
                                                          ChainIl& c) {
#pragma unroll
        for (int l = 0; l < (NW + 8) / 2; l++) {
            const uint32_t lo = 2 * l < NW ? k.pub[2 * l] : aw(a, 2 * l - NW);
            const uint32_t hi = 2 * l + 1 < NW ? k.pub[2 * l + 1] : aw(a, 2 * l + 1 - NW);
            il_to(lo, hi, c.w[2 * l], c.w[2 * l + 1]);
        }
    }
    // one chain step at hash address h (h < 16), in and out interleaved
    __device__ static __forceinline__ void F_il(const ChainIl& c, uint32_t h,
                                                const uint32_t in[NW], uint32_t out[NW]) {
        uint32_t s[50];
#pragma unroll
        for (int i = 0; i < 50; i++) {
            uint32_t x = 0;
            if (i < NW + 8) x = c.w[i];
            else if (i < 2 * NW + 8) x = in[i - NW - 8];
            if (i == 2 * kPadLane) x ^= 7u;      // 0x1F: even bits 0, 2, 4
            if (i == 2 * kPadLane + 1) x ^= 3u;  //       odd bits 1, 3
            if (i == 33) x ^= 0x80000000u;       // 0x80 at byte 135: lane 16, bit 63
            s[i] = x;
        }
        s[2 * kHashLane] ^= ((h & 1u) << 20) | (((h >> 2) & 1u) << 21);
        s[2 * kHashLane + 1] ^= (((h >> 1) & 1u) << 20) | (((h >> 3) & 1u) << 21);
        keccak_f_il<true>(s);
#pragma unroll
        for (int i = 0; i < NW; i++) out[i] = s[i];
    }
    // the chain form shared with Sha2 (values interleaved)
    using Chain = ChainIl;
    __device__ static __forceinline__ void chain_begin(const Key& k, const Adr& a, Chain& c) {
        chain_il_begin(k, a, c);
    }
    __device__ static __forceinline__ void chain_step(const Key&, const Chain& c, uint32_t h,
                                                      const uint32_t in[NW], uint32_t out[NW]) {
        F_il(c, h, in, out);
    }
    // The same on a lane pair (both lanes active, the same chain): this lane's
    // half of every Keccak lane.
    static constexpr int kPairWords = NW / 2;
    struct PairChain {
        uint32_t w[(NW + 8) / 2];  // pub_seed and address lanes
    };
    __device__ static __forceinline__ void pair_begin(const Key& k, const Adr& a, PairChain& c) {
        const uint32_t h = threadIdx.x & 1u;
#pragma unroll
        for (int l = 0; l < (NW + 8) / 2; l++)
            c.w[l] = il_half(2 * l < NW ? k.pub[2 * l < NW ? 2 * l : 0] : aw(a, 2 * l - NW),
                             2 * l + 1 < NW ? k.pub[2 * l + 1 < NW ? 2 * l + 1 : 0]
                                            : aw(a, 2 * l + 1 - NW), h);
    }
    __device__ static __forceinline__ void pair_step(const PairChain& c, const Adr&, uint32_t h,
                                                     uint32_t v[NW / 2]) {
        constexpr int PL = (NW + 8) / 2, VL = NW / 2;
        const uint32_t half = threadIdx.x & 1u;
        const uint32_t m = half ? ~0u : 0u;
        uint32_t s[25];
#pragma unroll
        for (int l = 0; l < 25; l++) {  // as F_il
            s[l] = l < PL ? c.w[l < PL ? l : 0]
                 : l < PL + VL ? v[l < PL ? 0 : l - PL < VL ? l - PL : 0] : 0u;
            if (l == kPadLane) s[l] ^= lane_sel(m, 3u, 7u);
            if (l == 16) s[l] ^= m & 0x80000000u;
        }
        const uint32_t x = h >> half;
        s[kHashLane] ^= ((x & 1u) << 20) | (((x >> 2) & 1u) << 21);
        keccak_f_il_pair(s);
#pragma unroll
        for (int l = 0; l < VL; l++) v[l] = s[l];
    }
    // NW plain words (NW / 2 lanes) <-> interleaved
    __device__ static __forceinline__ void to_il(const uint32_t in[NW], uint32_t out[NW]) {
#pragma unroll
        for (int l = 0; l < NW / 2; l++) il_to(in[2 * l], in[2 * l + 1], out[2 * l], out[2 * l + 1]);
    }
    __device__ static __forceinline__ void from_il(const uint32_t in[NW], uint32_t out[NW]) {
#pragma unroll
        for (int l = 0; l < NW / 2; l++)
            il_from(in[2 * l], in[2 * l + 1], out[2 * l], out[2 * l + 1]);
    }

    __device__ static __forceinline__ void H(const Key& k, const Adr& a, const uint32_t l[NW],
                                             const uint32_t r[NW], uint32_t out[NW]) {
        uint32_t d[2 * NW];
#pragma unroll
        for (int i = 0; i < NW; i++) {
            d[i] = l[i];
            d[NW + i] = r[i];
        }
        one_block<2 * NW>(k.pub, a, d, out);
    }

    __device__ static __forceinline__ void PRF(const Key& k, const Adr& a, uint32_t out[NW]) {
        one_block<0>(k.sk, a, nullptr, out);
    }

    // ------------------------------------------------ per-request hashing

    // SHAKE256(pre || m) squeezed to OUTB bytes (OUTB <= 136), on 32 lanes
    // holding identical inputs (Keccak32).  m is 4-byte aligned; the word
    // holding the last message byte is the last one read.  Lane p of the row
    // loads words p and p + 32 of a block (the next block's while this one
    // permutes) into LDS, from where every lane takes its halves.  The output
    // is in every lane.
    static constexpr int kStage = 36;  // LDS words of one staged block
    static constexpr int kRowWords = Keccak32::row_words(Keccak32::kLdsWords + kStage);
    template <int NPRE, int OUTB>
    __device__ static __forceinline__ void stream_msg(Keccak32& k, const uint32_t pre[NPRE], const uint8_t* m,
                                      uint32_t mlen, uint8_t out[OUTB]) {
        static_assert(NPRE < 34 && OUTB <= 136, "prefix within one block");
        const gbl_u32* mg = (gbl_u32*)reinterpret_cast<const uint32_t*>(m);  // address-space cast
        Keccak32::lds_word* stage = k.base + Keccak32::kLdsWords;
        const int p = threadIdx.x & 31;
        const uint32_t nb = (uint32_t)((4ull * NPRE + mlen) / 136u) + 1;
        // stream word g (behind the prefix): message bytes, then 0x1F
        auto word = [&](uint32_t g) -> uint32_t {
            const int64_t valid = (int64_t)mlen - 4 * ((int64_t)g - NPRE);
            if (g < (uint32_t)NPRE || valid < 0) return 0u;
            uint32_t x = valid > 0 ? mg[g - NPRE] : 0u;
            if (valid < 4) {
                const uint32_t sh = 8 * (uint32_t)valid;
                x = (x & ((1u << sh) - 1u)) | (0x1Fu << sh);
            }
            return x;
        };
        auto fetch = [&](uint32_t b, uint32_t x[2]) {
            x[0] = word(34 * b + p);
            x[1] = p < 2 ? word(34 * b + p + 32) : 0u;
        };
        uint32_t x[2];
        fetch(0, x);
        k.clear();
#pragma unroll 1
        for (uint32_t b = 0; b < nb; b++) {
            stage[p] = x[0];
            if (p < 2) stage[p + 32] = b + 1 == nb && p == 1 ? x[1] ^ 0x80000000u : x[1];
            Keccak32::order();
            if (b == 0) {  // the same values from every lane
#pragma unroll
                for (int q = 0; q < NPRE; q++) stage[q] = pre[q];
                Keccak32::order();
            }
#pragma unroll
            for (int i = 0; i < 3; i++) {
                const int l = k.col + 5 * (k.row + i);
                if (l < 17) k.s[i] ^= k.split(stage[2 * l], stage[2 * l + 1]);
            }
            Keccak32::order();
            if (b + 1 < nb) fetch(b + 1, x);
            k.permute();
        }
#pragma unroll
        for (int l = 0; l < (OUTB + 7) / 8; l++) {
            uint32_t lo, hi;
            k.lane(l, lo, hi);
#pragma unroll
            for (int o = 0; o < 8; o++)
                if (8 * l + o < OUTB) out[8 * l + o] = (uint8_t)((o < 4 ? lo : hi) >> (8 * (o & 3)));
        }
    }

    // The same on a lane pair holding identical inputs (keccak_f_il_pair): a
    // quarter of the instructions per request, at 2.9 times the latency.  Each
    // lane absorbs its half of every Keccak lane, the next block's words in
    // flight while this one permutes.  The output is in both lanes.
    template <int NPRE, int OUTB>
    __device__ static __forceinline__ void stream_msg_pair(const uint32_t pre[NPRE], const uint8_t* m,
                                                           uint32_t mlen, uint8_t out[OUTB]) {
        static_assert(NPRE < 34 && OUTB <= 136, "prefix within one block");
        const gbl_u32* mg = (gbl_u32*)reinterpret_cast<const uint32_t*>(m);  // address-space cast
        const uint32_t h = threadIdx.x & 1u;
        const uint32_t msk = h ? ~0u : 0u;
        const uint32_t nb = (uint32_t)((4ull * NPRE + mlen) / 136u) + 1;
        uint32_t s[25], x[34];
#pragma unroll
        for (int l = 0; l < 25; l++) s[l] = 0;
        // as above
        auto word = [&](uint32_t g) -> uint32_t {
            const int64_t valid = (int64_t)mlen - 4 * ((int64_t)g - NPRE);
            if (g < (uint32_t)NPRE || valid < 0) return 0u;
            uint32_t x = valid > 0 ? mg[g - NPRE] : 0u;
            if (valid < 4) {
                const uint32_t sh = 8 * (uint32_t)valid;
                x = (x & ((1u << sh) - 1u)) | (0x1Fu << sh);
            }
            return x;
        };
        auto fetch = [&](uint32_t b) {
            const uint32_t g = 34 * b;
            if (g >= (uint32_t)NPRE && 4ull * (g + 34 - NPRE) <= mlen) {  // message words only
#pragma unroll
                for (int l = 0; l < 34; l++) x[l] = mg[g - NPRE + l];
            } else {
#pragma unroll
                for (int l = 0; l < 34; l++) {
                    x[l] = word(g + l);
                    if (l < NPRE) x[l] = b == 0 ? pre[l < NPRE ? l : 0] : x[l];
                }
                if (b + 1 == nb) x[33] ^= 0x80000000u;
            }
        };
        fetch(0);
#pragma unroll 1
        for (uint32_t b = 0; b < nb; b++) {
#pragma unroll
            for (int l = 0; l < 17; l++) s[l] ^= il_half(x[2 * l], x[2 * l + 1], h);
            if (b + 1 < nb) fetch(b + 1);
            keccak_f_il_pair(s);
        }
#pragma unroll
        for (int l = 0; l < (OUTB + 7) / 8; l++) {
            const uint32_t other = pair_swap(s[l]);
            uint32_t lo, hi;
            il_from(lane_sel(msk, other, s[l]), lane_sel(msk, s[l], other), lo, hi);
#pragma unroll
            for (int o = 0; o < 8; o++)
                if (8 * l + o < OUTB) out[8 * l + o] = (uint8_t)((o < 4 ? lo : hi) >> (8 * (o & 3)));
        }
    }

    // R = SHAKE256(sk_prf || optrand || m, n) (hash_shake256.cu:64-75), on 32
    // lanes holding identical inputs (PAIR: 2 lanes, no k)
    template <bool PAIR>
    __device__ static __forceinline__ void prf_msg(Keccak32* k, const uint32_t skprf[NW], const uint32_t opt[NW],
                                   const uint8_t* m, uint32_t mlen, uint32_t R[NW]) {
        uint32_t pre[2 * NW];
        uint8_t o[N];
#pragma unroll
        for (int i = 0; i < NW; i++) {
            pre[i] = skprf[i];
            pre[NW + i] = opt[i];
        }
        if constexpr (PAIR) stream_msg_pair<2 * NW, N>(pre, m, mlen, o);
        else stream_msg<2 * NW, N>(*k, pre, m, mlen, o);
#pragma unroll
        for (int i = 0; i < NW; i++)
            R[i] = (uint32_t)o[4 * i] | (uint32_t)o[4 * i + 1] << 8 |
                   (uint32_t)o[4 * i + 2] << 16 | (uint32_t)o[4 * i + 3] << 24;
    }

    // digest = SHAKE256(R || pk || m, DG) (hash_shake256.cu:96-130), on 32
    // lanes holding identical inputs (PAIR: 2 lanes, no k)
    template <int DG, bool PAIR>
    __device__ static __forceinline__ void h_msg(Keccak32* k, const uint32_t R[NW], const uint32_t pk[2 * NW],
                                 const uint8_t* m, uint32_t mlen, uint8_t dg[DG]) {
        uint32_t pre[3 * NW];
#pragma unroll
        for (int i = 0; i < NW; i++) pre[i] = R[i];
#pragma unroll
        for (int i = 0; i < 2 * NW; i++) pre[NW + i] = pk[i];
        if constexpr (PAIR) stream_msg_pair<3 * NW, DG>(pre, m, mlen, dg);
        else stream_msg<3 * NW, DG>(*k, pre, m, mlen, dg);
    }

    // no midstate for SHAKE256 (zeros)
    __device__ static __forceinline__ void midstate(const uint32_t*, uint32_t mid[8]) {
#pragma unroll
        for (int i = 0; i < 8; i++) mid[i] = 0;
    }
};

}  // namespace spx
