// Exact integer attention for gfx950 and its operand producers, bit-exact with the reference's
// fused attention (src/attn.cu:1-6, whose unfused form is src/kernels.cu:673-722) and its operand
// kernels (src/kernels.cu:611-672,799-805). Heads of 64 values, G = B * heads groups.
//
// Semantics per query row q of group g, over the valid keys k (k < Tk, and k <= q when causal):
//   S = sum_d Q_d K_d (Q, K the int16 values of the planes: 256 hi + lo + 128)
//   s = rshr(S, 19 - eq - ek); mx = max s; E = lutexp(mx - s); sumE = sum E; r = floor(2^62 / sumE)
//   P = min(32767, (E r + 2^46) >> 47); O_d = sum_k P_k V_kd; out = rshr(O, 15 - ev_d)
//
// Design. The row maximum, the sum of E and P need one another in that order over all keys, so a row
// takes three passes over its scores; what the kernel spends is vector instructions per (query, key)
// pair, and its layout is chosen to compute the scores once and to keep every pass in registers.
//   * A wave owns 16 queries and up to 64 NT keys. Scores are 16x16x64 int8 MFMAs of the signed planes
//     with K as the A operand, so a lane holds one query and four consecutive keys of a 16-key subtile;
//     the subtile's rows are the keys 16 fg + 4 ks + j of a 64-key tile, so that the 16 scores a lane
//     holds of a tile are 16 consecutive keys -- the order in which the P.V MFMA wants its B operand.
//     P therefore never crosses lanes: it is packed in place into two signed byte planes.
//   * KW waves share a block's queries and split the keys (KW 64 NT >= Tkp): they exchange row
//     maxima and sums through LDS and add their partial outputs there. More keys than that (MULTI): one
//     wave sees all keys and recomputes the scores in each pass.
//   * Vector instructions bound the kernel, four cycles each when they issue back to back, and the lane permutes of
//     the operands, not memory (leaving the loads out gains 2 %): by the counters of whole calls 29 per pair with the
//     scores kept (80 groups of 1024 x 1024), 41 recomputed in each pass (40 groups of 4096 x 4096), MFMAs among them.
//   * The unsigned-offset terms of the planes ride in the MFMA accumulators' initial values: with q =
//     256 qh + ql + 128 and likewise k, S = 65536 hh + 256 hl + ll where hl starts at 128 qhs + qls / 2
//     and ll at 128 ksum (+ 128 when qls is odd).
//   * P is used as N = -P in signed digits, N = 256 h + l with h = (N + 128) >> 8 in [-128, 0] and l in
//     [-128, 127]: no offset to correct, and N = -32767 still fits. O = 128 sum P - sum N (256 vh + vl).
// Two forms of the per-pair arithmetic, chosen per block, both exact:
//   * integer (FAST), when the block's eq + ek lie in [0, 12], the table falls from at least 2^30 and
//     every entry is in [0, 2^31). Then S / 64 (floor) fits int32, s2 = S >> (18 - eq - ek) is one more
//     shift, rshr(S, 19 - eq - ek) = (s2 + 1) >> 1, and the table index and fraction of mx - s are fields
//     of one word w = (s2 - 2 mx + const) << 5. A table entry is 64 bits of a multiply-add whose high
//     word is E. sum E >= 2^30, so r <= 2^32, and r = 2^32 only when one key has all of it, where 2^32 -
//     1 gives the same P.
//   * general: the reference's formulas in double and 64-bit integers.
#include <algorithm>
#include <climits>

#include "attn.h"
#include "dispatch_rules.h"

namespace vk {

namespace {

typedef short h2 __attribute__((ext_vector_type(2)));

constexpr int AT_K = 64;            // keys per tile
constexpr int LUT_N = 1025;         // LDS table entries: (FAST) a zero entry and 1024 intervals
constexpr int KEY_RANGE = 4096;     // keys whose constants are in LDS at a time (MULTI)
constexpr int O_LD = 20;            // LDS stride of a dimension's 16 queries of partial outputs: the 64
                                    // lanes of an add (dimension 4 fg + j, query fr) hit 64 banks

// 16 bytes at a wave-uniform base plus a lane's 32-bit offset (the scalar-base form of the load)
__device__ __forceinline__ v4i ld16(const int8_t* p, unsigned off) { return *reinterpret_cast<const v4i*>(p + off); }

__device__ __forceinline__ double clampd32(double v) { return fmin(fmax(v, -2147483648.0), 2147483647.0); }

// floor(2^62 / s) for an integer 0 < s < 2^53: a double quotient, off by at most 2^9 for s = 1 and by at
// most one from s = 2^10 on, then exact corrections on the 64-bit remainder
__device__ __forceinline__ u64 recip62(u64 d) {
    u64 q = u64(0x1p62 / double(d));
    i64 rem = i64((u64(1) << 62) - q * d);
    while (rem < 0) { --q; rem += i64(d); }
    while (rem >= i64(d)) { ++q; rem -= i64(d); }
    return q;
}

// hides how a value was made from the optimiser (no instruction)
__device__ __forceinline__ void keep32(int& v) { asm("" : "+v"(v)); }

// table offset 8 * (w >> 16) and fraction (w & 0xffc0) << 16 of a score word, one instruction each
__device__ __forceinline__ unsigned lut_off(unsigned w) {
    unsigned r;
    asm("v_lshlrev_b32_sdwa %0, %1, %2 dst_sel:DWORD dst_unused:UNUSED_PAD src0_sel:DWORD src1_sel:WORD_1" : "=v"(r) : "v"(3), "v"(w));
    return r;
}
__device__ __forceinline__ unsigned lut_frac(unsigned w) {
    unsigned r;   // s_nop: a VALU read of a partly selected destination needs one wait state
    asm("v_and_b32_sdwa %0, %1, %2 dst_sel:WORD_1 dst_unused:UNUSED_PAD src0_sel:DWORD src1_sel:WORD_0\n\ts_nop 0" : "=v"(r) : "v"(0xffc0), "v"(w));
    return r;
}
// y >> (byte J of k)
template <int J>
__device__ __forceinline__ int ashr_byte(int y, unsigned k) {
    int r;
    if constexpr (J == 0) asm("v_ashrrev_i32_sdwa %0, %1, %2 dst_sel:DWORD dst_unused:UNUSED_PAD src0_sel:BYTE_0 src1_sel:DWORD" : "=v"(r) : "v"(k), "v"(y));
    if constexpr (J == 1) asm("v_ashrrev_i32_sdwa %0, %1, %2 dst_sel:DWORD dst_unused:UNUSED_PAD src0_sel:BYTE_1 src1_sel:DWORD" : "=v"(r) : "v"(k), "v"(y));
    if constexpr (J == 2) asm("v_ashrrev_i32_sdwa %0, %1, %2 dst_sel:DWORD dst_unused:UNUSED_PAD src0_sel:BYTE_2 src1_sel:DWORD" : "=v"(r) : "v"(k), "v"(y));
    if constexpr (J == 3) asm("v_ashrrev_i32_sdwa %0, %1, %2 dst_sel:DWORD dst_unused:UNUSED_PAD src0_sel:BYTE_3 src1_sel:DWORD" : "=v"(r) : "v"(k), "v"(y));
    return r;
}

// LDS pointers keep their address space through the structs below (as generic pointers every access
// would be a flat load or store).
#define LDS_AS __attribute__((address_space(3)))
typedef LDS_AS const int8_t* lds_bytes;
typedef unsigned u2 __attribute__((ext_vector_type(2)));
template <class T>
__device__ __forceinline__ T lds_ld(lds_bytes p) { return *(LDS_AS const T*)p; }

// LDS of a block after the table, in this order
struct AttnLds {
    LDS_AS u2* lut;             // LUT_N entries (static: constant LDS addresses)
    LDS_AS int* flag;           // 16: one vote word per wave
    LDS_AS int* mx;             // [wave][16]
    LDS_AS u64* sum;            // [wave][16]
    LDS_AS int* o;              // [query group][64][O_LD] partial outputs (KW > 1)
    LDS_AS int *kc0, *kc1;      // [key]: 128 ksum, and + 128
    LDS_AS uint8_t* ek;         // [key]
};
// byte offsets of the parts and their total
struct AttnLayout { unsigned flag, mx, sum, o, kc0, kc1, ek, bytes; };
__host__ __device__ inline AttnLayout attn_layout(int waves, int qw, int kw, int keys) {
    AttnLayout l;
    unsigned o = 0;
    auto take = [&](unsigned n) { const unsigned p = o; o += (n + 15) / 16 * 16; return p; };
    l.flag = take(64);
    l.mx = take(waves * 64);
    l.sum = take(waves * 128);
    l.o = take(kw > 1 ? qw * 64 * O_LD * 4 : 0);
    l.kc0 = take(keys * 4);
    l.kc1 = take(keys * 4);
    l.ek = take(keys);
    l.bytes = o;
    return l;
}

// One wave's work. lane = (fg, fr): query fr of the wave's 16, keys 16 fg + 4 ks + j of a tile.
template <bool FAST, int NT, bool MULTI>
struct AttnWave {
    const AttnArgs& a;
    const AttnLds& s;
    const int lane, fr, fg, wave, qw, kw, KW, g, q;   // q: this lane's query
    const bool active;                                // some query of the wave is below Tq
    int nT;                                           // key tiles the wave's queries see
    int kt0;                                          // its first tile (0 for MULTI)
    int q_lo;                                         // its first query
    v4i qa_h, qa_l, hl0;
    LDS_AS const int* kc;
    const int8_t *kp_h, *kp_l, *vp_h, *vp_l;          // the group's planes, and this lane's offsets in a tile
    unsigned ko_lane, vo_lane;
    int eq;
    unsigned k4base;

    // whether a key of tile kt can be invalid for one of the wave's queries
    __device__ __forceinline__ bool masked(int kt) const { return kt * AT_K + AT_K > a.Tk || (a.causal && kt * AT_K + AT_K - 1 > q_lo); }
    __device__ __forceinline__ bool valid(int kt, int ks, int j) const {
        const int key = kt * AT_K + 16 * fg + 4 * ks + j;
        return key < a.Tk && !(a.causal && key > q);
    }

    // Operand rows of 64 bytes (a key's values, or a dimension's 64 keys of a tile) are loaded with four
    // lanes to a row, so that 16 neighbouring lanes read 256 contiguous bytes, and reach the MFMA layout
    // (lane = chunk fg of row fr) by lane permutes. Loaded in that layout directly, a quarter of a wave
    // touches 16 rows and the address path takes a cycle for each (1024 x 1024 over 80 groups: 152 us, 119
    // with the permutes, 135 turned through LDS, 137 through a wave's DMA ring).
    struct Frag { v4i h, l; };
    int perm_idx;
    __device__ __forceinline__ Frag spread(const Frag& r) const {
        Frag f;
#pragma unroll
        for (int c = 0; c < 4; ++c) {
            f.h[c] = __builtin_amdgcn_ds_bpermute(perm_idx, r.h[c]);
            f.l[c] = __builtin_amdgcn_ds_bpermute(perm_idx, r.l[c]);
        }
        return f;
    }
    __device__ __forceinline__ Frag load_k(int kt, int ks) const {
        const size_t o = size_t(kt) * (AT_K * 64) + 256 * ks;
        return Frag{ld16(kp_h + o, ko_lane), ld16(kp_l + o, ko_lane)};
    }
    struct Acc { v4i hh, hl, ll; };
    // the MFMAs of a subtile; ko: its tile's first key relative to the LDS key constants
    __device__ __forceinline__ Acc qk(const Frag& k, int ko, int ks) const {
        Acc c;
        const v4i c4 = lds_ld<v4i>((lds_bytes)(kc + ko + 16 * fg + 4 * ks));
        c.hh = __builtin_amdgcn_mfma_i32_16x16x64_i8(k.h, qa_h, v4i{0, 0, 0, 0}, 0, 0, 0);
        c.hl = __builtin_amdgcn_mfma_i32_16x16x64_i8(k.h, qa_l, hl0, 0, 0, 0);
        c.ll = __builtin_amdgcn_mfma_i32_16x16x64_i8(k.l, qa_l, c4, 0, 0, 0);
        c.hl = __builtin_amdgcn_mfma_i32_16x16x64_i8(k.l, qa_h, c.hl, 0, 0, 0);
        return c;
    }
    // the scores of subtile ks of tile kt from its sums (FAST: s2; else s)
    __device__ __forceinline__ void finish(const Acc& c, int kt, int ko, int ks, int (&sv)[4]) const {
        if constexpr (FAST) {
            // |S| <= 2^36: S >> 6 is exact in 32 bits, and 256 hl is a multiple of 64
            int y[4];
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                int t = (c.hl[j] << 2) + (c.ll[j] >> 6);
                keep32(t);   // else the sum is reassociated into two shifts and a three-way add
                y[j] = (c.hh[j] << 10) + t;
            }
            const unsigned k4 = k4base - lds_ld<unsigned>((lds_bytes)(s.ek + ko + 16 * fg + 4 * ks));
            sv[0] = ashr_byte<0>(y[0], k4);
            sv[1] = ashr_byte<1>(y[1], k4);
            sv[2] = ashr_byte<2>(y[2], k4);
            sv[3] = ashr_byte<3>(y[3], k4);
        } else {
            const int32_t* ek = a.ek + size_t(g) * a.Tkp + kt * AT_K + 16 * fg + 4 * ks;
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                const double S = fma(double(c.hh[j]), 65536.0, double((c.hl[j] << 8) + c.ll[j]));
                sv[j] = int(clampd32(floor(ldexp(S, ek[j] + eq - 19) + 0.5)));   // rshr(S, 19 - eq - ek), saturated
            }
        }
    }
    // INT_MIN for the scores of tile kt's invalid keys (FAST)
    __device__ __forceinline__ void mask(int kt, int (&sv)[4][4]) const {
#pragma unroll
        for (int ks = 0; ks < 4; ++ks)
#pragma unroll
            for (int j = 0; j < 4; ++j) sv[ks][j] = valid(kt, ks, j) ? sv[ks][j] : INT_MIN;
    }
    __device__ __forceinline__ void scores(int kt, int ko, int (&sv)[4][4]) const {
#pragma unroll
        for (int ks = 0; ks < 4; ++ks) finish(qk(spread(load_k(kt, ks)), ko, ks), kt, ko, ks, sv[ks]);
        if (FAST && masked(kt)) mask(kt, sv);
    }
    __device__ __forceinline__ void tile_max(int kt, const int (&sv)[4][4], int& m) const {
#pragma unroll
        for (int ks = 0; ks < 4; ++ks)
#pragma unroll
            for (int j = 0; j < 4; ++j)
                if (FAST || valid(kt, ks, j)) m = max(m, sv[ks][j]);
    }

    // E of a score: FAST from s2 with c = 2^21 - 1 - 2 mx + 2048 (w >> 16 = 1024 - ((mx - s) >> 10), the
    // zero entry from 2^20 on); else lutexp(mx - s) (src/attn.cu:85-91) from {L[i], L[i + 1]} pairs
    int mxc;   // FAST: c; else mx
    __device__ __forceinline__ unsigned exp_of(int v) const {
        if constexpr (FAST) {
            const unsigned w = unsigned(max(v, -mxc) + mxc) << 5;
            const u2 en = lds_ld<u2>((lds_bytes)s.lut + lut_off(w));
            const unsigned d = __builtin_amdgcn_alignbit(en.x, en.x, 22);
            return unsigned((u64(d) * lut_frac(w) + ((u64(en.y) << 32) | en.x)) >> 32);
        } else {
            const unsigned z = unsigned(mxc) - unsigned(v);
            if (z >= (1u << 20)) return 0;
            const u2 en = s.lut[z >> 10];
            return unsigned(int(en.x) + int(((i64(int(en.y)) - i64(int(en.x))) * int(z & 1023u)) >> 10));
        }
    }
    __device__ __forceinline__ void tile_exp(int kt, int (&sv)[4][4]) const {
#pragma unroll
        for (int ks = 0; ks < 4; ++ks)
#pragma unroll
            for (int j = 0; j < 4; ++j) sv[ks][j] = FAST || valid(kt, ks, j) ? int(exp_of(sv[ks][j])) : 0;
    }
    __device__ __forceinline__ static u64 tile_sum(const int (&sv)[4][4], u64 sum) {
#pragma unroll
        for (int ks = 0; ks < 4; ++ks)
#pragma unroll
            for (int j = 0; j < 4; ++j) sum += unsigned(sv[ks][j]);
        return sum;
    }

    // P of a tile's E, as the byte planes of -P (pn_h, pn_l: byte 4 ks + j), and their sum
    u64 rr;
    __device__ __forceinline__ void tile_p(const int (&sv)[4][4], v4i& pn_h, v4i& pn_l, int& psum) const {
#pragma unroll
        for (int ks = 0; ks < 4; ++ks) {
            int p[4];
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                int e = sv[ks][j];
                keep32(e);   // else E is widened where it is made and takes a register pair
                const unsigned E = unsigned(e);
                if constexpr (FAST) {
                    p[j] = int(unsigned((u64(E) * unsigned(rr) + (u64(1) << 46)) >> 32) >> 15);
                } else {
                    const u64 pp = (u64(E) * rr + (u64(1) << 46)) >> 47;
                    p[j] = pp > 32767u ? 32767 : int(pp);
                }
            }
            const h2 p01 = __builtin_bit_cast(h2, __builtin_amdgcn_cvt_pk_i16(p[0], p[1]));   // saturates 32768 to 32767
            const h2 p23 = __builtin_bit_cast(h2, __builtin_amdgcn_cvt_pk_i16(p[2], p[3]));
            const h2 one = h2{1, 1}, z = h2{0, 0}, c128 = h2{128, 128};
            psum = __builtin_amdgcn_sdot2(p01, one, psum, false);
            psum = __builtin_amdgcn_sdot2(p23, one, psum, false);
            const unsigned n01 = __builtin_bit_cast(unsigned, h2(z - p01)), n23 = __builtin_bit_cast(unsigned, h2(z - p23));
            const unsigned m01 = __builtin_bit_cast(unsigned, h2(c128 - p01)), m23 = __builtin_bit_cast(unsigned, h2(c128 - p23));
            pn_l[ks] = int(__builtin_amdgcn_perm(n23, n01, 0x06040200));
            pn_h[ks] = int(__builtin_amdgcn_perm(m23, m01, 0x07050301));
        }
    }
    __device__ __forceinline__ Frag load_v(int kt, int ds) const {
        const size_t o = size_t(16 * ds) * a.Tkp + kt * AT_K;
        return Frag{ld16(vp_h + o, vo_lane), ld16(vp_l + o, vo_lane)};
    }
    __device__ __forceinline__ static void pv(const Frag& v, v4i pn_h, v4i pn_l, v4i& hh, v4i& hl, v4i& ll) {
        hh = __builtin_amdgcn_mfma_i32_16x16x64_i8(v.h, pn_h, hh, 0, 0, 0);
        hl = __builtin_amdgcn_mfma_i32_16x16x64_i8(v.h, pn_l, hl, 0, 0, 0);
        ll = __builtin_amdgcn_mfma_i32_16x16x64_i8(v.l, pn_l, ll, 0, 0, 0);
        hl = __builtin_amdgcn_mfma_i32_16x16x64_i8(v.l, pn_h, hl, 0, 0, 0);
    }
};

// rshr(O, 15 - ev), saturated, and its magnitude into am; O below 2^53
__device__ __forceinline__ int attn_out(double O, int ev, uint32_t& am) {
    const int o = int(clampd32(floor(ldexp(O, ev - 15) + 0.5)));
    am = max(am, uabs(o));
    return o;
}

template <bool FAST, int NT, bool MULTI>
__device__ __forceinline__ void attn_body(const AttnArgs& a, const AttnLds& s, int g, int qb, int QW, int KW) {
    typedef AttnWave<FAST, NT, MULTI> W;
    const int tid = threadIdx.x, lane = tid & 63, fr = lane & 15, fg = lane >> 4;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int qw = wave / KW, kw = wave - qw * KW;
    const int q_lo = qb * 16 * QW + 16 * qw, nTall = a.Tkp / AT_K;
    const int nTk = (a.Tk + AT_K - 1) / AT_K;
    const bool active = q_lo < a.Tq;
    W w{a, s, lane, fr, fg, wave, qw, kw, KW, g, q_lo + fr, active};
    w.q_lo = q_lo;
    w.nT = !active ? 0 : a.causal ? min(nTk, (min(q_lo + 15, a.Tq - 1) / AT_K) + 1) : nTk;
    w.kt0 = MULTI ? 0 : kw * NT;
    {
        const size_t r = size_t(g) * a.Tqp + min(w.q, a.Tq - 1);
        w.qa_h = *reinterpret_cast<const v4i*>(a.qh + r * 64 + 16 * fg);
        w.qa_l = *reinterpret_cast<const v4i*>(a.ql + r * 64 + 16 * fg);
        const int hs = int(a.qhs[r]), ls = int(a.qls[r]);
        const int h0 = 128 * hs + (ls >> 1);
        w.hl0 = v4i{h0, h0, h0, h0};
        w.kc = ls & 1 ? s.kc1 : s.kc0;
        w.eq = a.eq[r];
        w.k4base = unsigned(12 - w.eq) * 0x01010101u;
        w.kp_h = a.kh + size_t(g) * a.Tkp * 64;
        w.kp_l = a.kl + size_t(g) * a.Tkp * 64;
        // lane 4 r + c loads chunk c of row r: key 16 (r / 4) + 4 ks + r % 4 of the tile, or dimension 16 ds + r
        const int r4 = lane >> 2, c4 = lane & 3;
        w.perm_idx = 4 * (4 * fr + fg);
        w.ko_lane = (16 * (r4 >> 2) + (r4 & 3)) * 64 + 16 * c4;
        w.vp_h = a.vth + size_t(g) * 64 * a.Tkp;
        w.vp_l = a.vtl + size_t(g) * 64 * a.Tkp;
        w.vo_lane = unsigned(r4) * a.Tkp + 16 * c4;
    }
    // key constants of the keys [base, base + KEY_RANGE) (MULTI; else all of them, staged by the caller)
    auto stage = [&](int base) {
        __syncthreads();
        const int n = min(KEY_RANGE, a.Tkp - base);
        for (int i = tid; i < n; i += blockDim.x) {
            const size_t k = size_t(g) * a.Tkp + base + i;
            const int c = 128 * int(a.ksum[k]);
            s.kc0[i] = c;
            s.kc1[i] = c + 128;
            s.ek[i] = base + i < a.Tk ? uint8_t(a.ek[k]) : 0;
        }
        __syncthreads();
    };
    // f(tile, first key relative to the staged constants) over every tile of the wave (MULTI)
    auto all_tiles = [&](auto&& f) {
        for (int base = 0; base < a.Tkp; base += KEY_RANGE) {
            if (a.Tkp > KEY_RANGE) stage(base);
            const int t1 = min(w.nT, (base + KEY_RANGE) / AT_K);
            for (int kt = base / AT_K; kt < t1; ++kt) f(kt, kt * AT_K - base);
        }
    };

    int sv[MULTI ? 1 : NT][4][4];
    constexpr int PF = 4;
    const bool any = w.kt0 < w.nT;                                     // the wave has a valid key (not MULTI)
    auto tile = [&](int t) { return min(w.kt0 + t, nTall - 1); };      // the tile whose operands tile t reads (its keys past Tk are masked)
    // ---- pass 0: the row maximum
    int m = INT_MIN;
    if constexpr (MULTI) {
        all_tiles([&](int kt, int ko) {
            w.scores(kt, ko, sv[0]);
            w.tile_max(kt, sv[0], m);
        });
    } else {
        if (any) {
            // rows loaded PF subtiles ahead, permuted one ahead, scores finished one behind the MFMAs
            typename W::Frag kb[PF], kn;
            typename W::Acc acc;
#pragma unroll
            for (int i = 0; i < PF; ++i) kb[i] = w.load_k(tile(i / 4), i % 4);
            kn = w.spread(kb[0]);
#pragma unroll
            for (int i = 0; i < 4 * NT; ++i) {
                const typename W::Frag k = kn;
                if (i + PF < 4 * NT) kb[i % PF] = w.load_k(tile((i + PF) / 4), (i + PF) % 4);
                if (i + 1 < 4 * NT) kn = w.spread(kb[(i + 1) % PF]);
                const typename W::Acc cur = w.qk(k, tile(i / 4) * AT_K, i % 4);
                if (i) w.finish(acc, tile((i - 1) / 4), tile((i - 1) / 4) * AT_K, (i - 1) % 4, sv[(i - 1) / 4][(i - 1) % 4]);
                acc = cur;
            }
            w.finish(acc, tile(NT - 1), tile(NT - 1) * AT_K, 3, sv[NT - 1][3]);
            if (FAST && w.masked(w.kt0 + NT - 1)) {
#pragma unroll
                for (int t = 0; t < NT; ++t) w.mask(w.kt0 + t, sv[t]);
            }
#pragma unroll
            for (int t = 0; t < NT; ++t) w.tile_max(w.kt0 + t, sv[t], m);
        }
    }
    m = max(m, __shfl_xor(m, 16));
    m = max(m, __shfl_xor(m, 32));
    if (KW > 1) {
        if (fg == 0) s.mx[wave * 16 + fr] = m;
        __syncthreads();
        for (int k = 0; k < KW; ++k) m = max(m, s.mx[(qw * KW + k) * 16 + fr]);
    }
    // FAST: m is the maximum s2 = 2 s or 2 s - 1 of the score s
    w.mxc = FAST ? (1 << 21) + 2047 - 2 * ((m >> 1) + (m & 1)) : m;

    // ---- pass 1: sum of E, then r = floor(2^62 / sumE) (0 for sumE = 0)
    u64 se = 0;
    if constexpr (MULTI) {
        all_tiles([&](int kt, int ko) {
            w.scores(kt, ko, sv[0]);
            w.tile_exp(kt, sv[0]);
            se = W::tile_sum(sv[0], se);
        });
    } else {
        if (any) {
#pragma unroll
            for (int t = 0; t < NT; ++t) {
                w.tile_exp(w.kt0 + t, sv[t]);
                se = W::tile_sum(sv[t], se);
            }
        }
    }
    se += u64(__shfl_xor((long long)se, 16));
    se += u64(__shfl_xor((long long)se, 32));
    if (KW > 1) {
        if (fg == 0) s.sum[wave * 16 + fr] = se;
        __syncthreads();
        se = 0;
        for (int k = 0; k < KW; ++k) se += s.sum[(qw * KW + k) * 16 + fr];
    }
    w.rr = se ? recip62(se) : 0;
    if (FAST) w.rr = min(w.rr, u64(0xffffffffu));

    // ---- pass 2: P and P.V
    int psum = 0;
    uint32_t am = 0;
    const bool store = w.q < a.Tq;
    const int b = g / a.heads, h = g - b * a.heads;
    int32_t* orow = a.out + (size_t(b) * a.Tq + (store ? w.q : 0)) * a.C + h * 64;
    const int32_t* ev = a.ev + g * 64;
    if constexpr (MULTI) {
        v4i hh[4], hl[4], ll[4];
#pragma unroll
        for (int ds = 0; ds < 4; ++ds) hh[ds] = hl[ds] = ll[ds] = v4i{0, 0, 0, 0};
        all_tiles([&](int kt, int ko) {
            v4i pn_h, pn_l;
            w.scores(kt, ko, sv[0]);
            w.tile_exp(kt, sv[0]);
            w.tile_p(sv[0], pn_h, pn_l, psum);
#pragma unroll
            for (int ds = 0; ds < 4; ++ds) W::pv(w.spread(w.load_v(kt, ds)), pn_h, pn_l, hh[ds], hl[ds], ll[ds]);
        });
        psum += __shfl_xor(psum, 16);
        psum += __shfl_xor(psum, 32);
#pragma unroll
        for (int ds = 0; ds < 4; ++ds) {
            int o4[4];
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                const double N = fma(double(hh[ds][j]), 65536.0, fma(double(hl[ds][j]), 256.0, double(ll[ds][j])));
                o4[j] = attn_out(128.0 * psum - N, ev[16 * ds + 4 * fg + j], am);
            }
            if (store) *reinterpret_cast<int4*>(orow + 16 * ds + 4 * fg) = make_int4(o4[0], o4[1], o4[2], o4[3]);
        }
    } else {
        if (any) {
            v4i pn_h[NT], pn_l[NT];
            typename W::Frag vb[PF], vn;   // V rows loaded PF ahead, dimension by dimension, permuted one ahead
            auto vload = [&](int i) { return w.load_v(tile(i % NT), i / NT); };
#pragma unroll
            for (int i = 0; i < PF; ++i) vb[i] = vload(i);
#pragma unroll
            for (int t = 0; t < NT; ++t) {
                w.tile_p(sv[t], pn_h[t], pn_l[t], psum);
            }
            psum += __shfl_xor(psum, 16);
            psum += __shfl_xor(psum, 32);
            vn = w.spread(vb[0]);
            // |O| < 2^31 (the P of a row sum to at most 32768 + Tk / 2 < 2^16), so partial sums may wrap
#pragma unroll
            for (int ds = 0; ds < 4; ++ds) {
                v4i hh = v4i{0, 0, 0, 0}, hl = hh, ll = hh;
#pragma unroll
                for (int t = 0; t < NT; ++t) {
                    const int i = ds * NT + t;
                    const typename W::Frag v = vn;
                    if (i + PF < 4 * NT) vb[i % PF] = vload(i + PF);
                    if (i + 1 < 4 * NT) vn = w.spread(vb[(i + 1) % PF]);
                    W::pv(v, pn_h[t], pn_l[t], hh, hl, ll);
                }
                unsigned O[4];
#pragma unroll
                for (int j = 0; j < 4; ++j) O[j] = 128u * unsigned(psum) - ((unsigned(hh[j]) << 16) + (unsigned(hl[j]) << 8) + unsigned(ll[j]));
                if (KW > 1) {
#pragma unroll
                    for (int j = 0; j < 4; ++j) __hip_atomic_fetch_add((LDS_AS unsigned*)s.o + (qw * 64 + 16 * ds + 4 * fg + j) * O_LD + fr, O[j], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
                } else {
                    int o4[4];
#pragma unroll
                    for (int j = 0; j < 4; ++j) o4[j] = attn_out(double(int(O[j])), ev[16 * ds + 4 * fg + j], am);
                    if (store) *reinterpret_cast<int4*>(orow + 16 * ds + 4 * fg) = make_int4(o4[0], o4[1], o4[2], o4[3]);
                }
            }
        }
        if (KW > 1) {
            // the summed outputs, four dimensions of a query per thread: 16 lanes share a query
            __syncthreads();
            for (int i = tid; i < QW * 256; i += blockDim.x) {
                const int ql = i >> 4, d = 4 * (i & 15), qq = qb * 16 * QW + ql;
                int o4[4];
                uint32_t mo = 0;
#pragma unroll
                for (int j = 0; j < 4; ++j) o4[j] = attn_out(double(s.o[((ql >> 4) * 64 + d + j) * O_LD + (ql & 15)]), ev[d + j], mo);
#pragma unroll
                for (int x = 8; x; x >>= 1) mo = max(mo, uint32_t(__shfl_xor(int(mo), x)));
                if (qq < a.Tq) {
                    *reinterpret_cast<int4*>(a.out + (size_t(b) * a.Tq + qq) * a.C + h * 64 + d) = make_int4(o4[0], o4[1], o4[2], o4[3]);
                    if (a.rowmax && d == 0 && mo) atomicMax(a.rowmax + size_t(b) * a.Tq + qq, mo);
                }
            }
            return;
        }
    }
    if (a.rowmax) {
        am = max(am, uint32_t(__shfl_xor(int(am), 16)));
        am = max(am, uint32_t(__shfl_xor(int(am), 32)));
        if (fg == 0 && store && am) atomicMax(a.rowmax + size_t(b) * a.Tq + w.q, am);
    }
}

}  // namespace

// grid (query blocks * G), 64 QW KW threads: QW groups of 16 queries, KW waves splitting the keys.
template <int NT, bool MULTI, int THREADS, int WPE>
__global__ void __launch_bounds__(THREADS, WPE) attn_kernel(const AttnArgs a, int QW, int KW, int qblocks) {
    __shared__ __attribute__((aligned(16))) u2 s_lut[LUT_N + 1];
    extern __shared__ __attribute__((aligned(16))) int8_t smem[];
    const int tid = threadIdx.x, nthr = blockDim.x, wave = tid >> 6;
    const AttnLayout l = attn_layout(nthr >> 6, QW, KW, MULTI ? min(a.Tkp, KEY_RANGE) : a.Tkp);
    LDS_AS int8_t* const base = (LDS_AS int8_t*)smem;
    const AttnLds s{(LDS_AS u2*)s_lut,           (LDS_AS int*)(base + l.flag), (LDS_AS int*)(base + l.mx),  (LDS_AS u64*)(base + l.sum), (LDS_AS int*)(base + l.o),
                    (LDS_AS int*)(base + l.kc0),  (LDS_AS int*)(base + l.kc1), (LDS_AS uint8_t*)(base + l.ek)};
    // an XCD takes a contiguous run of blocks, so that few groups' keys and values share its L2
    const int nb = gridDim.x, per = nb >> 3, rem = nb & 7, x = blockIdx.x & 7;
    const int blk = x * per + min(x, rem) + int(blockIdx.x >> 3);
    const int g = blk / qblocks, qb = blk - g * qblocks;

    // the table (src/attn.cu:85-91), key constants, cleared partial outputs, and the test for FAST
    bool ok = true;
    auto lut_build = [&](bool fast) {
        for (int i = tid; i < 1024; i += nthr) {
            const long long l0 = a.Lexp[i], l1 = a.Lexp[i + 1];
            if (fast) {
                ok = ok && l0 < (1ll << 31) && l0 >= l1 && l1 >= 0 && (i != 0 || l0 >= (1ll << 30));
                const unsigned d = unsigned(l0 - l1);
                s.lut[1024 - i] = u2{(d << 22) | (d >> 10), unsigned(l1) + (d >> 10)};
            } else {
                s.lut[i] = u2{unsigned(l0), unsigned(l1)};
            }
        }
    };
    lut_build(true);
    if (tid == 0) s.lut[0] = u2{0, 0};
    const size_t k0 = size_t(g) * a.Tkp;
    int ekmax = 0;
    const int staged = MULTI ? min(a.Tkp, KEY_RANGE) : a.Tkp;
    for (int i = tid; i < a.Tkp; i += nthr) {
        const int e = i < a.Tk ? a.ek[k0 + i] : 0;
        ok = ok && e >= 0;
        ekmax = max(ekmax, e);
        if (i < staged) {
            const int c = 128 * int(a.ksum[k0 + i]);
            s.kc0[i] = c;
            s.kc1[i] = c + 128;
            s.ek[i] = uint8_t(e);
        }
    }
    if (KW > 1)
        for (int i = tid; i < QW * 64 * O_LD; i += nthr) s.o[i] = 0;
    int eqmax = 0;
    for (int i = tid; i < 16 * QW; i += nthr) {
        const int q = qb * 16 * QW + i;
        const int e = q < a.Tq ? a.eq[size_t(g) * a.Tqp + q] : 0;
        ok = ok && e >= 0;
        eqmax = max(eqmax, e);
    }
    // the wave's word: 1 << 16 where a test failed, else the largest ek and eq seen
#pragma unroll
    for (int o = 32; o; o >>= 1) {
        ekmax = max(ekmax, __shfl_xor(ekmax, o));
        eqmax = max(eqmax, __shfl_xor(eqmax, o));
    }
    const bool wok = __ballot(!ok) == 0;
    if ((tid & 63) == 0) s.flag[wave] = wok ? min(ekmax, 127) | (min(eqmax, 127) << 8) : 1 << 16;
    __syncthreads();
    int mk = 0, mq = 0, bad = 0;
    for (int i = 0; i < (nthr >> 6); ++i) {
        const int f = s.flag[i];
        bad |= f >> 16;
        mk = max(mk, f & 255);
        mq = max(mq, (f >> 8) & 255);
    }
    if (!bad && mk + mq <= 12) {
        attn_body<true, NT, MULTI>(a, s, g, qb, QW, KW);
    } else {
        __syncthreads();
        lut_build(false);
        __syncthreads();
        attn_body<false, NT, MULTI>(a, s, g, qb, QW, KW);
    }
}

// ---------------------------------------------------------------- operands

// src/kernels.cu:611-631 (k_quant_heads): one wave per (g, t) row of 64 values, lane d owning value d
__global__ void __launch_bounds__(256) quant_heads_kernel(const int32_t* __restrict__ X, int B, int T, int C, int heads, int Tp, int8_t* __restrict__ hi,
                                                          int8_t* __restrict__ lo, int32_t* __restrict__ e, long long* __restrict__ hs,
                                                          long long* __restrict__ ls, long long* __restrict__ tsum) {
    const int lane = threadIdx.x & 63;
    const long long w = (long long)blockIdx.x * 4 + (threadIdx.x >> 6);
    const int G = B * heads;
    if (w >= (long long)G * Tp) return;
    const int g = int(w / Tp), t = int(w - (long long)g * Tp), b = g / heads, h = g - b * heads;
    const size_t o = size_t(w) * 64 + lane;
    if (t >= T) {
        hi[o] = 0;
        lo[o] = -128;
        if (lane == 0) { e[w] = 0; hs[w] = 0; ls[w] = -128 * 64; tsum[w] = 0; }
        return;
    }
    const int x = X[(size_t(b) * T + t) * C + h * 64 + lane];
    uint32_t m = uabs(x);
#pragma unroll
    for (int s = 32; s; s >>= 1) m = max(m, uint32_t(__shfl_xor(int(m), s)));
    const int ee = rowexp_u32(m);
    const int q = quant16_32(x, ee);
    const int hv = q >> 8, lv = (q & 255) - 128;
    hi[o] = int8_t(hv);
    lo[o] = int8_t(lv);
    int sh = hv, sl = lv, st = q;
#pragma unroll
    for (int s = 32; s; s >>= 1) { sh += __shfl_xor(sh, s); sl += __shfl_xor(sl, s); st += __shfl_xor(st, s); }
    if (lane == 0) { e[w] = ee; hs[w] = sh; ls[w] = sl; tsum[w] = st; }
}

// The same with 16 lanes to a row, four values a lane and R rows of each 16-lane group in flight (rows R n +
// i * 16 of a block): one 16-byte load and two 4-byte stores per lane and row, reductions inside a DPP row,
// where the form above stores single bytes and shuffles through 64 lanes (8 x 1024 x 640 in 10 heads, 31 MB:
// 26.3 -> 7.7 us). Needs a 16-byte aligned X, C % 4 == 0 and 4-byte aligned planes.
template <int CTRL>
__device__ __forceinline__ int dpp(int v) { return __builtin_amdgcn_update_dpp(0, v, CTRL, 0xF, 0xF, false); }
__device__ __forceinline__ uint32_t row16_umax(uint32_t v) {
    v = max(v, uint32_t(dpp<0xB1>(int(v))));
    v = max(v, uint32_t(dpp<0x4E>(int(v))));
    v = max(v, uint32_t(dpp<0x141>(int(v))));
    return max(v, uint32_t(dpp<0x140>(int(v))));
}
__device__ __forceinline__ int row16_sum(int v) {
    v += dpp<0xB1>(v);
    v += dpp<0x4E>(v);
    v += dpp<0x141>(v);
    return v + dpp<0x140>(v);
}
template <int R>
__global__ void __launch_bounds__(256) quant_heads_vec_kernel(const int32_t* __restrict__ X, int B, int T, int C, int heads, int Tp,
                                                              int8_t* __restrict__ hi, int8_t* __restrict__ lo, int32_t* __restrict__ e,
                                                              long long* __restrict__ hs, long long* __restrict__ ls, long long* __restrict__ tsum) {
    const int l16 = threadIdx.x & 15;
    const unsigned w0 = blockIdx.x * (16 * R) + (threadIdx.x >> 4), rows = unsigned(B) * heads * Tp;   // below 2^31
    int4 x[R];
    bool real[R];
#pragma unroll
    for (int i = 0; i < R; ++i) {
        const unsigned w = w0 + 16 * i;
        const int g = int(w / unsigned(Tp)), t = int(w - unsigned(g) * Tp), b = g / heads, h = g - b * heads;
        real[i] = w < rows && t < T;
        x[i] = make_int4(0, 0, 0, 0);
        if (real[i]) x[i] = *reinterpret_cast<const int4*>(X + (size_t(b) * T + t) * C + h * 64 + 4 * l16);
    }
#pragma unroll
    for (int i = 0; i < R; ++i) {
        const unsigned w = w0 + 16 * i;
        const int v[4] = {x[i].x, x[i].y, x[i].z, x[i].w};
        const int ee = rowexp_u32(row16_umax(max(max(uabs(v[0]), uabs(v[1])), max(uabs(v[2]), uabs(v[3])))));
        unsigned h4 = 0, l4 = 0;
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const int q = quant16_32(v[j], ee);
            h4 |= unsigned(q >> 8 & 255) << (8 * j);
            l4 |= unsigned((q & 255) ^ 128) << (8 * j);
        }
        const int sh = row16_sum(__builtin_amdgcn_sdot4(int(h4), 0x01010101, 0, false));
        const int sl = row16_sum(__builtin_amdgcn_sdot4(int(l4), 0x01010101, 0, false));
        if (w < rows) {   // a pad row is the value 0: hi 0, lo -128
            const size_t o = size_t(w) * 16 + l16;
            reinterpret_cast<unsigned*>(hi)[o] = h4;
            reinterpret_cast<unsigned*>(lo)[o] = l4;
            if (l16 == 0) {
                e[w] = ee;
                hs[w] = sh;
                ls[w] = sl;
                tsum[w] = 256 * sh + sl + 128 * 64;
            }
        }
    }
}

// src/kernels.cu:799-805: rows t in [T, Tp) of every group take the value 0
__global__ void __launch_bounds__(256) quant_heads_pad_kernel(int G, int T, int Tp, int8_t* __restrict__ hi, int8_t* __restrict__ lo, int32_t* __restrict__ e,
                                                              long long* __restrict__ hs, long long* __restrict__ ls, long long* __restrict__ tsum) {
    const int lane = threadIdx.x & 63, npad = Tp - T;
    const long long w = (long long)blockIdx.x * 4 + (threadIdx.x >> 6);
    if (w >= (long long)G * npad) return;
    const int g = int(w / npad);
    const size_t row = size_t(g) * Tp + T + (w - (long long)g * npad);
    hi[row * 64 + lane] = 0;
    lo[row * 64 + lane] = -128;
    if (lane == 0) { e[row] = 0; hs[row] = 0; ls[row] = -128 * 64; tsum[row] = 0; }
}

// src/kernels.cu:632-650 (k_quant_v, exponents): ev = row_exp(max |x|) per dimension. row_exp is monotone,
// so blocks of QV_ROWS rows of a group combine their exponents by an atomic maximum on a cleared ev; the
// clear also zeroes vsum for the write pass. One block per group scanning all rows (1 MB a block), four loads deep,
// was most of the operand's time: 4096 rows in 40 groups 286 us with the write pass, 26 in runs of 128 rows (calls
// back to back; 127 and 28 by the kernel trace of an attention layer).
constexpr int QV_ROWS = 128;
constexpr int QV_ONE = 128;    // keys a block quantises on its own, in one launch in place of three
__global__ void __launch_bounds__(256) quant_v_clear_kernel(int n, int32_t* __restrict__ ev, long long* __restrict__ vsum) {
    const int i = blockIdx.x * 256 + threadIdx.x;
    if (i < n) {
        ev[i] = 0;
        vsum[i] = 0;
    }
}
__global__ void __launch_bounds__(256) quant_v_exp_kernel(const int32_t* __restrict__ X, int Tk, int C, int heads, int32_t* __restrict__ ev) {
    __shared__ uint32_t s_m[4][64];
    const int g = blockIdx.y, b = g / heads, h = g - b * heads, d = threadIdx.x & 63, sl = threadIdx.x >> 6;
    const int t0 = blockIdx.x * QV_ROWS + sl;
    const int32_t* x = X + size_t(b) * Tk * C + h * 64 + d;
    uint32_t m = 0;
#pragma unroll 8
    for (int i = 0; i < QV_ROWS; i += 4) m = max(m, uabs(x[size_t(min(t0 + i, Tk - 1)) * C]));
    s_m[sl][d] = m;
    __syncthreads();
    if (sl == 0) {
        m = max(max(s_m[0][d], s_m[1][d]), max(s_m[2][d], s_m[3][d]));
        const int e = rowexp_u32(m);
        if (e) atomicMax(ev + g * 64 + d, e);
    }
}

// src/kernels.cu:651-672 (k_quant_v, transposed write): block per (64-row tile, group): the tile in
// LDS, then thread (d, quarter) quantises 16 consecutive rows of dimension d, writes them as 16
// bytes of each plane of vt[g * 64 + d], and adds its part of vsum
// ONE: the block has all of its group's rows (Tkp <= QV_ONE), finds the exponents itself and writes ev and vsum.
template <bool ONE>
__global__ void __launch_bounds__(256) quant_v_write_kernel(const int32_t* __restrict__ X, int Tk, int C, int heads, int Tkp,
                                                            int32_t* __restrict__ ev, int8_t* __restrict__ vth, int8_t* __restrict__ vtl,
                                                            long long* __restrict__ vsum) {
    constexpr int NT = ONE ? QV_ONE / 64 : 1;   // tiles of the block
    __shared__ int32_t tile[NT * 64][65];
    __shared__ int s_e[4][64];
    const int g = blockIdx.y, t0 = blockIdx.x * 64, b = g / heads, h = g - b * heads;
    const int tx = threadIdx.x & 63, ty = threadIdx.x >> 6;
    const int32_t* x = X + size_t(b) * Tk * C + h * 64 + tx;
    uint32_t m = 0;
#pragma unroll
    for (int r = 0; r < NT * 64; r += 4) {
        const int t = t0 + r + ty;
        const int v = t < Tk ? x[size_t(t) * C] : 0;
        tile[r + ty][tx] = v;
        m = max(m, uabs(v));
    }
    if (ONE) s_e[ty][tx] = rowexp_u32(m);
    __syncthreads();
    const int d = threadIdx.x >> 2, qt = threadIdx.x & 3;
    const int e = ONE ? max(max(s_e[0][d], s_e[1][d]), max(s_e[2][d], s_e[3][d])) : ev[g * 64 + d];
    int s = 0;   // of 16 NT values below 2^15
#pragma unroll
    for (int k = 0; k < NT; ++k) {
        if (ONE && k * 64 >= Tkp) break;
        unsigned hw[4], lw[4];
#pragma unroll
        for (int c = 0; c < 4; ++c) {
            unsigned hv = 0, lv = 0;
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const int q = quant16_32(tile[64 * k + 16 * qt + 4 * c + i][d], e);   // rows past Tk hold 0
                s += q;
                hv |= unsigned(q >> 8 & 255) << (8 * i);
                lv |= unsigned((q & 255) ^ 128) << (8 * i);
            }
            hw[c] = hv;
            lw[c] = lv;
        }
        const size_t o = (size_t(g) * 64 + d) * Tkp + t0 + 64 * k + 16 * qt;
        *reinterpret_cast<v4i*>(vth + o) = v4i{int(hw[0]), int(hw[1]), int(hw[2]), int(hw[3])};
        *reinterpret_cast<v4i*>(vtl + o) = v4i{int(lw[0]), int(lw[1]), int(lw[2]), int(lw[3])};
    }
    s += dpp<0xB1>(s);   // the four quarters of a dimension are a quad of lanes
    s += dpp<0x4E>(s);
    if (qt == 0) {
        if (ONE) {
            ev[g * 64 + d] = e;
            vsum[g * 64 + d] = s;
        } else {
            atomicAdd(reinterpret_cast<unsigned long long*>(vsum + g * 64 + d), (unsigned long long)(long long)s);
        }
    }
}

// ---------------------------------------------------------------- launchers

// Four waves a block, in the form that attn_form gives. The register limits are what measured best of 2, 3 and 4
// waves per SIMD.
hipError_t launch_attention(hipStream_t st, const AttnArgs& a, int G) {
    const AttnForm f = attn_form(a.Tkp);
    const int KW = f.waves, QW = 4 / KW;
    const int qblocks = (a.Tq + 16 * QW - 1) / (16 * QW);
    const unsigned lds = attn_layout(4, QW, KW, f.multi ? std::min(a.Tkp, KEY_RANGE) : a.Tkp).bytes;
    const dim3 grid(unsigned(qblocks * G)), blk(256);
    if (f.multi) hipLaunchKernelGGL((attn_kernel<1, true, 256, 2>), grid, blk, lds, st, a, QW, KW, qblocks);
    else if (f.tiles == 1) hipLaunchKernelGGL((attn_kernel<1, false, 256, 4>), grid, blk, lds, st, a, QW, KW, qblocks);
    else if (f.tiles == 2) hipLaunchKernelGGL((attn_kernel<2, false, 256, 4>), grid, blk, lds, st, a, QW, KW, qblocks);
    else hipLaunchKernelGGL((attn_kernel<4, false, 256, 3>), grid, blk, lds, st, a, QW, KW, qblocks);
    return hipGetLastError();
}

hipError_t launch_quant_heads(hipStream_t st, const int32_t* X, int B, int T, int C, int heads, int Tp, int8_t* hi, int8_t* lo, int32_t* e, long long* hs,
                              long long* ls, long long* tsum) {
    const long long rows = (long long)B * heads * Tp;
    const uintptr_t al = reinterpret_cast<uintptr_t>(X) % 16 | reinterpret_cast<uintptr_t>(hi) % 4 | reinterpret_cast<uintptr_t>(lo) % 4 | unsigned(C % 4);
    if (al || rows > INT_MAX - 64) hipLaunchKernelGGL(quant_heads_kernel, dim3(unsigned((rows + 3) / 4)), dim3(256), 0, st, X, B, T, C, heads, Tp, hi, lo, e, hs, ls, tsum);
    // few rows: one per 16-lane group, so that every CU has a block
    else if (rows < 32768) hipLaunchKernelGGL(quant_heads_vec_kernel<1>, dim3(unsigned((rows + 15) / 16)), dim3(256), 0, st, X, B, T, C, heads, Tp, hi, lo, e, hs, ls, tsum);
    else hipLaunchKernelGGL(quant_heads_vec_kernel<4>, dim3(unsigned((rows + 63) / 64)), dim3(256), 0, st, X, B, T, C, heads, Tp, hi, lo, e, hs, ls, tsum);
    return hipGetLastError();
}

hipError_t launch_quant_heads_pad(hipStream_t st, int G, int T, int Tp, int8_t* hi, int8_t* lo, int32_t* e, long long* hs, long long* ls, long long* tsum) {
    const long long rows = (long long)G * (Tp - T);
    hipLaunchKernelGGL(quant_heads_pad_kernel, dim3(unsigned((rows + 3) / 4)), dim3(256), 0, st, G, T, Tp, hi, lo, e, hs, ls, tsum);
    return hipGetLastError();
}

hipError_t launch_quant_v(hipStream_t st, const int32_t* X, int B, int Tk, int C, int heads, int Tkp, int8_t* vth, int8_t* vtl, int32_t* ev, long long* vsum) {
    const int G = B * heads;
    if (Tkp <= QV_ONE) {
        hipLaunchKernelGGL(quant_v_write_kernel<true>, dim3(1, unsigned(G)), dim3(256), 0, st, X, Tk, C, heads, Tkp, ev, vth, vtl, vsum);
        return hipGetLastError();
    }
    hipLaunchKernelGGL(quant_v_clear_kernel, dim3(unsigned((G * 64 + 255) / 256)), dim3(256), 0, st, G * 64, ev, vsum);
    hipLaunchKernelGGL(quant_v_exp_kernel, dim3(unsigned((Tk + QV_ROWS - 1) / QV_ROWS), unsigned(G)), dim3(256), 0, st, X, Tk, C, heads, ev);
    hipLaunchKernelGGL(quant_v_write_kernel<false>, dim3(unsigned(Tkp / 64), unsigned(G)), dim3(256), 0, st, X, Tk, C, heads, Tkp, ev, vth, vtl, vsum);
    return hipGetLastError();
}

}  // namespace vk
