// aes_dev.h -- AES-128 encryption on CDNA4 with T-tables staged in LDS, and the
// half-tree hashes / dealer PRF built on it.
//
// State: four little-endian 32-bit columns (c_j = byte 4j | byte 4j+1 << 8 | ...).
// One round:  n_j = T0[b0(c_j)] ^ T1[b1(c_j+1)] ^ T2[b2(c_j+2)] ^ T3[b3(c_j+3)] ^ rk_j
// with T0[x] = (2S[x], S[x], S[x], 3S[x]) as bytes 0..3 and T_k = rotl(T0, 8k).
// The last round reads S[x] out of the byte of T_(r+3)%4 that holds it.
//
// LDS layout: NT tables (1 = T0 only, rotations computed; 4 = all four), each
// entry replicated REP times and interleaved so that word address of entry e,
// copy c is e*REP + c.  Lane l reads copy (l % REP), so with REP equal to the
// number of LDS banks the 64 lanes of a wavefront never collide on a bank.
#pragma once
#include <hip/hip_runtime.h>

#include <cstdint>
#include <type_traits>

#include "mpcx_core.h"

namespace mpcx {

struct T0Table {
  uint32_t v[256];
};

constexpr uint8_t xtime_c(uint8_t a) { return uint8_t((a << 1) ^ ((a & 0x80) ? 0x1b : 0)); }
constexpr T0Table make_t0() {
  T0Table t{};
  for (int x = 0; x < 256; x++) {
    uint8_t s = kSboxC[x];
    uint8_t s2 = xtime_c(s);
    uint8_t s3 = uint8_t(s2 ^ s);
    t.v[x] = uint32_t(s2) | (uint32_t(s) << 8) | (uint32_t(s) << 16) | (uint32_t(s3) << 24);
  }
  return t;
}

__device__ __constant__ const T0Table c_T0 = make_t0();

// The fixed keys as compile-time constants: a round key is then an immediate move
// into a scalar register where it is used, and holds none across a DCF level.
constexpr AesRK c_rkH = aes_expand_c(kKeyHc);  // tree hash H
constexpr AesRK c_rkL = aes_expand_c(kKeyLc);  // leaf hash HL

__device__ __forceinline__ uint32_t rotl32(uint32_t v, int k) {
  return k == 0 ? v : ((v << k) | (v >> (32 - k)));
}

// a ^ b ^ c in one v_bitop3_b32 (truth table 0x96 = 0xf0 ^ 0xcc ^ 0xaa).
__device__ __forceinline__ uint32_t xor3(uint32_t a, uint32_t b, uint32_t c) {
  return __builtin_amdgcn_bitop3_b32(a, b, c, 0x96);
}

template <int NT, int REP>
struct AesTab {
  static_assert(NT == 1 || NT == 4, "NT");  // NT == 0: AesPerm
  static_assert(REP >= 1 && REP <= 64 && (REP & (REP - 1)) == 0, "REP");
  static constexpr int kWords = NT * 256 * REP;
  static constexpr int kBytes = kWords * 4;
  static constexpr int kLogRep = REP == 1 ? 0 : REP == 2 ? 1 : REP == 4 ? 2 : REP == 8 ? 3 : REP == 16 ? 4 : REP == 32 ? 5 : 6;

  const char *base;
  uint32_t laneoff;

  // Fill the replicated tables; must be called by every thread of the block.
  __device__ static void fill(uint32_t *lds) {
    for (int w = threadIdx.x; w < kWords; w += blockDim.x) {
      int e = w >> kLogRep;
      int k = e >> 8, x = e & 255;
      lds[w] = rotl32(c_T0.v[x], 8 * k);
    }
    __syncthreads();
  }

  __device__ AesTab(const uint32_t *lds) : base((const char *)lds) {
    laneoff = (threadIdx.x & (REP - 1)) * 4u;
  }

  __device__ __forceinline__ uint32_t T(int k, uint32_t x) const {
    if constexpr (NT == 4) {
      return *(const uint32_t *)(base + k * (256 * REP * 4) + (x << (2 + kLogRep)) + laneoff);
    } else {
      uint32_t v = *(const uint32_t *)(base + (x << (2 + kLogRep)) + laneoff);
      return rotl32(v, 8 * k);
    }
  }

  __device__ __forceinline__ uint4 enc(uint4 in, const AesRK &rk) const {
    uint32_t c0 = in.x ^ rk.w[0], c1 = in.y ^ rk.w[1], c2 = in.z ^ rk.w[2], c3 = in.w ^ rk.w[3];
#pragma unroll
    for (int r = 1; r < 10; r++) {
      uint32_t n0 = xor3(xor3(T(0, c0 & 255u), T(1, (c1 >> 8) & 255u), T(2, (c2 >> 16) & 255u)), T(3, c3 >> 24), rk.w[4 * r + 0]);
      uint32_t n1 = xor3(xor3(T(0, c1 & 255u), T(1, (c2 >> 8) & 255u), T(2, (c3 >> 16) & 255u)), T(3, c0 >> 24), rk.w[4 * r + 1]);
      uint32_t n2 = xor3(xor3(T(0, c2 & 255u), T(1, (c3 >> 8) & 255u), T(2, (c0 >> 16) & 255u)), T(3, c1 >> 24), rk.w[4 * r + 2]);
      uint32_t n3 = xor3(xor3(T(0, c3 & 255u), T(1, (c0 >> 8) & 255u), T(2, (c1 >> 16) & 255u)), T(3, c2 >> 24), rk.w[4 * r + 3]);
      c0 = n0;
      c1 = n1;
      c2 = n2;
      c3 = n3;
    }
    uint4 o;
    o.x = ((T(3, c0 & 255u) & 0xffu) | (T(0, (c1 >> 8) & 255u) & 0xff00u) | (T(1, (c2 >> 16) & 255u) & 0xff0000u) |
           (T(2, c3 >> 24) & 0xff000000u)) ^ rk.w[40];
    o.y = ((T(3, c1 & 255u) & 0xffu) | (T(0, (c2 >> 8) & 255u) & 0xff00u) | (T(1, (c3 >> 16) & 255u) & 0xff0000u) |
           (T(2, c0 >> 24) & 0xff000000u)) ^ rk.w[41];
    o.z = ((T(3, c2 & 255u) & 0xffu) | (T(0, (c3 >> 8) & 255u) & 0xff00u) | (T(1, (c0 >> 16) & 255u) & 0xff0000u) |
           (T(2, c1 >> 24) & 0xff000000u)) ^ rk.w[42];
    o.w = ((T(3, c3 & 255u) & 0xffu) | (T(0, (c0 >> 8) & 255u) & 0xff00u) | (T(1, (c1 >> 16) & 255u) & 0xff0000u) |
           (T(2, c2 >> 24) & 0xff000000u)) ^ rk.w[43];
    return o;
  }

  // H(s) = AES_k(sigma(s)) ^ sigma(s), sigma(xL||xR) = (xL^xR)||xL, xR = words 0,1.
  __device__ __forceinline__ uint4 hash(uint4 s, const AesRK &rk) const {
    uint4 x;
    x.x = s.z;
    x.y = s.w;
    x.z = s.z ^ s.x;
    x.w = s.w ^ s.y;
    uint4 y = enc(x, rk);
    y.x ^= x.x;
    y.y ^= x.y;
    y.z ^= x.z;
    y.w ^= x.w;
    return y;
  }

  // Dealer PRF block AES_kd(idx_lo, idx_hi, field, gate).
  __device__ __forceinline__ uint4 prf(const AesRK &kd, uint32_t gate, uint32_t field, uint64_t idx) const {
    uint4 b;
    b.x = uint32_t(idx);
    b.y = uint32_t(idx >> 32);
    b.z = field;
    b.w = gate;
    return enc(b, kd);
  }
};

// T0 alone, 64 copies per entry: entry x, copy j at byte address 256*x + 4*j.
// Lane l reads copy l mod 64, so a wavefront never has two lanes on one bank,
// and the byte address of "T0[byte k of c]" for this lane is one v_perm_b32 of
// (c, lane word): byte 0 = (lane*4) mod 256, byte 1 = byte k of c, bytes 2..3 = 0.
// T1..T3 are rotations of T0 (v_alignbit_b32), three-input XORs are
// v_bitop3_b32, and the last round gathers the S-box bytes (byte 1 of T0) with
// v_perm_b32.  The hash folds sigma into the first AddRoundKey and the
// feed-forward into the last one.  (Holding T1 as a second 64 KiB table saves
// two rotations per column but leaves room for only one workgroup per CU; it
// measured slower.)
struct AesPerm {
  static constexpr int kWords = 256 * 64;
  static constexpr int kBytes = kWords * 4;

  const char *base;
  uint32_t lane4;  // (lane * 4) mod 256

  // 16-byte stores: 16 per entry (its 64 copies), kWords / 4 in all
  __device__ static void fill(uint32_t *lds) {
    uint4 *l4 = reinterpret_cast<uint4 *>(lds);
    for (int q = threadIdx.x; q < kWords / 4; q += blockDim.x) {
      const uint32_t v = c_T0.v[q >> 4];
      l4[q] = make_uint4(v, v, v, v);
    }
    __syncthreads();
  }

  __device__ AesPerm(const uint32_t *lds) : base((const char *)lds) { lane4 = (threadIdx.x & 63u) * 4u; }

  // T0[byte K of c]
  template <int t, int K>
  __device__ __forceinline__ uint32_t L(uint32_t c) const {
    static_assert(t == 0, "one table");
    const uint32_t addr = __builtin_amdgcn_perm(c, lane4, 0x0c0c0000u | ((4u + K) << 8));
    return *(const uint32_t *)(base + addr);
  }
  // rotl(v, 8k) as a funnel shift
  template <int K>
  __device__ __forceinline__ static uint32_t rot(uint32_t v) {
    return K == 0 ? v : __builtin_amdgcn_alignbit(v, v, 32 - 8 * K);
  }
  __device__ __forceinline__ uint32_t col(uint32_t a, uint32_t b, uint32_t c, uint32_t d, uint32_t k) const {
    return xor3(xor3(L<0, 0>(a), rot<1>(L<0, 1>(b)), rot<2>(L<0, 2>(c))), rot<3>(L<0, 3>(d)), k);
  }
  // S[byte 0 of a] | S[byte 1 of b] << 8 | S[byte 2 of c] << 16 | S[byte 3 of d] << 24
  __device__ __forceinline__ uint32_t last(uint32_t a, uint32_t b, uint32_t c, uint32_t d) const {
    const uint32_t lo = __builtin_amdgcn_perm(L<0, 1>(b), L<0, 0>(a), 0x0c0c0501u);
    const uint32_t hi = __builtin_amdgcn_perm(L<0, 3>(d), L<0, 2>(c), 0x0c0c0501u);
    return (hi << 16) | lo;
  }

  // rounds 1..9 on the whitened state
  __device__ __forceinline__ void rounds(uint32_t &c0, uint32_t &c1, uint32_t &c2, uint32_t &c3,
                                         const AesRK &rk) const {
#pragma unroll
    for (int r = 1; r < 10; r++) {
      const uint32_t n0 = col(c0, c1, c2, c3, rk.w[4 * r + 0]);
      const uint32_t n1 = col(c1, c2, c3, c0, rk.w[4 * r + 1]);
      const uint32_t n2 = col(c2, c3, c0, c1, rk.w[4 * r + 2]);
      const uint32_t n3 = col(c3, c0, c1, c2, rk.w[4 * r + 3]);
      c0 = n0;
      c1 = n1;
      c2 = n2;
      c3 = n3;
    }
  }

  __device__ __forceinline__ uint4 enc(uint4 in, const AesRK &rk) const {
    uint32_t c0 = in.x ^ rk.w[0], c1 = in.y ^ rk.w[1], c2 = in.z ^ rk.w[2], c3 = in.w ^ rk.w[3];
    rounds(c0, c1, c2, c3, rk);
    uint4 o;
    o.x = last(c0, c1, c2, c3) ^ rk.w[40];
    o.y = last(c1, c2, c3, c0) ^ rk.w[41];
    o.z = last(c2, c3, c0, c1) ^ rk.w[42];
    o.w = last(c3, c0, c1, c2) ^ rk.w[43];
    return o;
  }

  // H(s) = AES_k(sigma(s)) ^ sigma(s), sigma(xL||xR) = (xL^xR)||xL, xR = words 0,1
  __device__ __forceinline__ uint4 hash(uint4 s, const AesRK &rk) const {
    uint32_t c0 = s.z ^ rk.w[0], c1 = s.w ^ rk.w[1];
    uint32_t c2 = xor3(s.z, s.x, rk.w[2]), c3 = xor3(s.w, s.y, rk.w[3]);
    rounds(c0, c1, c2, c3, rk);
    uint4 o;
    o.x = xor3(last(c0, c1, c2, c3), rk.w[40], s.z);
    o.y = xor3(last(c1, c2, c3, c0), rk.w[41], s.w);
    o.z = xor3(last(c2, c3, c0, c1), rk.w[42], s.z) ^ s.x;
    o.w = xor3(last(c3, c0, c1, c2), rk.w[43], s.w) ^ s.y;
    return o;
  }

  // Two whitened blocks under one key: a round's 16 reads of one go out while the
  // other's columns are formed, as in AesPerm2 (one after the other, which the
  // scheduler makes of two calls, the dealer's gates take up to 1.7 times as long).
  struct Reads {
    uint32_t v[4][4];  // byte b of column j
  };
  __device__ __forceinline__ void read(Reads &r, uint4 c) const {
    const uint32_t w[4] = {c.x, c.y, c.z, c.w};
#pragma unroll
    for (int j = 0; j < 4; j++) {
      r.v[j][0] = L<0, 0>(w[j]);
      r.v[j][1] = L<0, 1>(w[j]);
      r.v[j][2] = L<0, 2>(w[j]);
      r.v[j][3] = L<0, 3>(w[j]);
    }
    __builtin_amdgcn_sched_barrier(0);
  }
  __device__ __forceinline__ static uint32_t col(const Reads &r, int j, uint32_t k) {
    return xor3(xor3(r.v[j][0], rot<1>(r.v[(j + 1) & 3][1]), rot<2>(r.v[(j + 2) & 3][2])),
                rot<3>(r.v[(j + 3) & 3][3]), k);
  }
  __device__ __forceinline__ static uint4 cols(const Reads &r, const uint32_t *k) {
    return make_uint4(col(r, 0, k[0]), col(r, 1, k[1]), col(r, 2, k[2]), col(r, 3, k[3]));
  }
  __device__ __forceinline__ static uint32_t last(const Reads &r, int j) {
    const uint32_t lo = __builtin_amdgcn_perm(r.v[(j + 1) & 3][1], r.v[j][0], 0x0c0c0501u);
    const uint32_t hi = __builtin_amdgcn_perm(r.v[(j + 3) & 3][3], r.v[(j + 2) & 3][2], 0x0c0c0501u);
    return (hi << 16) | lo;
  }
  __device__ __forceinline__ static uint4 lasts(const Reads &r, const uint32_t *k) {
    return make_uint4(last(r, 0) ^ k[0], last(r, 1) ^ k[1], last(r, 2) ^ k[2], last(r, 3) ^ k[3]);
  }
  __device__ __forceinline__ void rounds2(uint4 &u, uint4 &v, const AesRK &rk) const {
    Reads a, b;
    read(a, u);
    read(b, v);
#pragma unroll
    for (int r = 1; r < 10; r++) {
      read(a, cols(a, rk.w + 4 * r));
      read(b, cols(b, rk.w + 4 * r));
    }
    u = lasts(a, rk.w + 40);
    v = lasts(b, rk.w + 40);
  }
  __device__ __forceinline__ void enc2(uint4 u, uint4 v, const AesRK &rk, uint4 *eu, uint4 *ev) const {
    *eu = make_uint4(u.x ^ rk.w[0], u.y ^ rk.w[1], u.z ^ rk.w[2], u.w ^ rk.w[3]);
    *ev = make_uint4(v.x ^ rk.w[0], v.y ^ rk.w[1], v.z ^ rk.w[2], v.w ^ rk.w[3]);
    rounds2(*eu, *ev, rk);
  }
  __device__ __forceinline__ void hash2(uint4 s, uint4 u, const AesRK &rk, uint4 *hs, uint4 *hu) const {
    enc2(make_uint4(s.z, s.w, s.z ^ s.x, s.w ^ s.y), make_uint4(u.z, u.w, u.z ^ u.x, u.w ^ u.y), rk, hs, hu);
    *hs = make_uint4(hs->x ^ s.z, hs->y ^ s.w, xor3(hs->z, s.z, s.x), xor3(hs->w, s.w, s.y));
    *hu = make_uint4(hu->x ^ u.z, hu->y ^ u.w, xor3(hu->z, u.z, u.x), xor3(hu->w, u.w, u.y));
  }

  // Dealer PRF block AES_kd(idx_lo, idx_hi, field, gate).
  __device__ __forceinline__ uint4 prf(const AesRK &kd, uint32_t gate, uint32_t field, uint64_t idx) const {
    uint4 b;
    b.x = uint32_t(idx);
    b.y = uint32_t(idx >> 32);
    b.z = field;
    b.w = gate;
    return enc(b, kd);
  }
};

// T0 and T1 = rotl(T0, 8) in one 64 KiB table, 32 copies each: entry x holds
// T0[x] at byte address 256*x + 4*j and T1[x] at 256*x + 128 + 4*j, copy j.
// Lane l reads copy l mod 32, so the two half-waves, which the LDS serves in
// turn, never have two lanes on one bank.  One v_perm_b32 gives the address of
// "T0[byte k of c]" (byte 0 = 4 (lane mod 32), byte 1 = byte k of c); T1 is the
// same address plus the read's immediate offset 128.  A column is 4 address
// permutes, one rotation and two three-input XORs (28 VALU per round against 36
// with T0 alone).
struct AesPerm2 {
  static constexpr int kWords = 256 * 64;
  static constexpr int kBytes = kWords * 4;

  const char *base;
  uint32_t lane4;  // (lane * 4) mod 128

  // Entry x is 8 16-byte words of T0[x], then 8 of T1[x]; a thread writes one of
  // the two halves of an entry, starting at word x mod 8, so that 16 lanes' stores
  // cover the 64 banks.  The reads of T0 go out together: a loop of one read per
  // store spends a memory latency per iteration, and this is what a launch of few
  // elements starts with (1024 truncations 33.7 -> 32.6 us, a forward of one
  // sample 501 -> 487 us).
  // fill_words() issues those reads, so that a kernel can put its own behind them
  // before it waits.
  struct FillWords {
    uint32_t w0, w1;
  };
  __device__ static FillWords fill_words() {
    const uint32_t nt = blockDim.x, q0 = threadIdx.x, q1 = q0 + nt;
    return {c_T0.v[(q0 >> 1) & 255u], nt < 512 ? c_T0.v[(q1 >> 1) & 255u] : 0u};
  }
  __device__ static void fill(uint32_t *lds) { fill(lds, fill_words()); }
  __device__ static void fill(uint32_t *lds, const FillWords &w) {
    uint4 *l4 = reinterpret_cast<uint4 *>(lds);
    const uint32_t nt = blockDim.x, q0 = threadIdx.x, q1 = q0 + nt;
    auto half = [&](uint32_t q, uint32_t t) {
      const uint32_t v = (q & 1u) ? rotl32(t, 8) : t;
#pragma unroll
      for (uint32_t k = 0; k < 8; k++) l4[8 * q + ((k + (q >> 1)) & 7u)] = make_uint4(v, v, v, v);
    };
    if (q0 < 512) half(q0, w.w0);
    if (q1 < 512) half(q1, w.w1);
    for (uint32_t q = q1 + nt; q < 512; q += nt) half(q, c_T0.v[q >> 1]);
    __syncthreads();
  }

  __device__ AesPerm2(const uint32_t *lds) : base((const char *)lds) { lane4 = (threadIdx.x & 31u) * 4u; }

  // byte address of entry (byte K of c), copy lane mod 32
  template <int K>
  __device__ __forceinline__ uint32_t adr(uint32_t c) const {
    return __builtin_amdgcn_perm(c, lane4, 0x0c0c0000u | ((4u + K) << 8));
  }
  template <int K>
  __device__ __forceinline__ uint32_t t0(uint32_t c) const {
    return *(const uint32_t *)(base + adr<K>(c));
  }
  template <int K>
  __device__ __forceinline__ uint32_t t1(uint32_t c) const {
    return *(const uint32_t *)(base + adr<K>(c) + 128);
  }
  // The 16 table reads of a round by source column: T0[byte 0], T1[byte 1],
  // T0[byte 2], T1[byte 3] of column j (the last round reads T0 throughout, whose
  // byte 1 is S).
  struct Reads {
    uint32_t v[16];
  };
  template <bool LAST>
  __device__ __forceinline__ void read(Reads &r, int j, uint32_t c) const {
    r.v[4 * j] = t0<0>(c);
    r.v[4 * j + 1] = LAST ? t0<1>(c) : t1<1>(c);
    r.v[4 * j + 2] = t0<2>(c);
    r.v[4 * j + 3] = LAST ? t0<3>(c) : t1<3>(c);
  }
  // Column j of the round whose reads are r: T0[a] ^ T1[b] ^ rotl(T0[c] ^ T1[d] ^
  // rotl(k, 16), 16), the second half being T2[c] ^ T3[d] ^ k; the round key is
  // uniform, so its rotation is scalar work.
  __device__ __forceinline__ static uint32_t col(const Reads &r, int j, uint32_t k) {
    const uint32_t h = xor3(r.v[4 * ((j + 2) & 3) + 2], r.v[4 * ((j + 3) & 3) + 3], (k << 16) | (k >> 16));
    return xor3(r.v[4 * j], r.v[4 * ((j + 1) & 3) + 1], __builtin_amdgcn_alignbit(h, h, 16));
  }
  // Column j of the last round before its key: S of byte i of column j + i
  __device__ __forceinline__ static uint32_t last(const Reads &r, int j) {
    const uint32_t lo = __builtin_amdgcn_perm(r.v[4 * ((j + 1) & 3) + 1], r.v[4 * j], 0x0c0c0501u);
    const uint32_t hi = __builtin_amdgcn_perm(r.v[4 * ((j + 3) & 3) + 3], r.v[4 * ((j + 2) & 3) + 2], 0x0c0c0501u);
    return (hi << 16) | lo;
  }
  // Finishes round k from its reads and issues the reads of round k + 1.
  __device__ __forceinline__ void step(Reads &r, const AesRK &rk, int k) const {
    uint32_t c[4];
#pragma unroll
    for (int j = 0; j < 4; j++) c[j] = col(r, j, rk.w[4 * k + j]);
#pragma unroll
    for (int j = 0; j < 4; j++)
      if (k < 9)
        read<false>(r, j, c[j]);
      else
        read<true>(r, j, c[j]);
  }
  // A round's 16 reads go out together, and the scheduler is held to that order:
  // left to itself it keeps few reads in flight (a wait every 2.6 reads) and takes
  // more registers for addresses formed early.  With two chains, one chain's reads
  // are in flight while the other's columns are formed.  61 registers in the two-
  // chain walk, so that two 1024-thread workgroups fit a CU: 105-106 G AES/s (348
  // clocks per wave and AES, against 341 for its 160 reads) where the scheduler's
  // own order ran 98 G in half the waves and 87-92 with one chain (walks of 25
  // calls over 2^22 elements, both parties, correction words read from HBM).
  __device__ __forceinline__ static void phase() { __builtin_amdgcn_sched_barrier(0); }

  __device__ __forceinline__ void start(Reads &r, uint4 c) const {
    read<false>(r, 0, c.x);
    read<false>(r, 1, c.y);
    read<false>(r, 2, c.z);
    read<false>(r, 3, c.w);
    phase();
  }
  // rounds 1..9 of the block whose first reads are r; then r holds the last round's
  __device__ __forceinline__ void rounds(Reads &r, const AesRK &rk) const {
#pragma unroll
    for (int k = 1; k < 10; k++) {
      step(r, rk, k);
      phase();
    }
  }
  // two blocks, each under its own key
  __device__ __forceinline__ void rounds2(Reads &a, const AesRK &ka, Reads &b, const AesRK &kb) const {
#pragma unroll
    for (int k = 1; k < 10; k++) {
      step(a, ka, k);
      phase();
      step(b, kb, k);
      phase();
    }
  }
  __device__ __forceinline__ static uint4 whiten(uint4 in, const AesRK &rk) {
    return make_uint4(in.x ^ rk.w[0], in.y ^ rk.w[1], in.z ^ rk.w[2], in.w ^ rk.w[3]);
  }
  __device__ __forceinline__ static uint4 enc_out(const Reads &r, const AesRK &rk) {
    return make_uint4(last(r, 0) ^ rk.w[40], last(r, 1) ^ rk.w[41], last(r, 2) ^ rk.w[42], last(r, 3) ^ rk.w[43]);
  }
  // H(s) = AES_k(sigma(s)) ^ sigma(s), sigma(xL||xR) = (xL^xR)||xL, xR = words 0,1
  __device__ __forceinline__ static uint4 hash_in(uint4 s, const AesRK &rk) {
    return make_uint4(s.z ^ rk.w[0], s.w ^ rk.w[1], xor3(s.z, s.x, rk.w[2]), xor3(s.w, s.y, rk.w[3]));
  }
  __device__ __forceinline__ static uint4 hash_out(const Reads &r, const AesRK &rk, uint4 s) {
    return make_uint4(xor3(last(r, 0), rk.w[40], s.z), xor3(last(r, 1), rk.w[41], s.w),
                      xor3(last(r, 2), rk.w[42], s.z) ^ s.x, xor3(last(r, 3), rk.w[43], s.w) ^ s.y);
  }

  __device__ __forceinline__ uint4 enc(uint4 in, const AesRK &rk) const {
    Reads r;
    start(r, whiten(in, rk));
    rounds(r, rk);
    return enc_out(r, rk);
  }
  __device__ __forceinline__ void enc2(uint4 u, uint4 v, const AesRK &rk, uint4 *eu, uint4 *ev) const {
    Reads a, b;
    start(a, whiten(u, rk));
    start(b, whiten(v, rk));
    rounds2(a, rk, b, rk);
    *eu = enc_out(a, rk);
    *ev = enc_out(b, rk);
  }
  __device__ __forceinline__ uint4 hash(uint4 s, const AesRK &rk) const {
    Reads r;
    start(r, hash_in(s, rk));
    rounds(r, rk);
    return hash_out(r, rk, s);
  }
  __device__ __forceinline__ void hash2(uint4 s, uint4 u, const AesRK &rk, uint4 *hs, uint4 *hu) const {
    Reads a, b;
    start(a, hash_in(s, rk));
    start(b, hash_in(u, rk));
    rounds2(a, rk, b, rk);
    *hs = hash_out(a, rk, s);
    *hu = hash_out(b, rk, u);
  }

  // Dealer PRF block AES_kd(idx_lo, idx_hi, field, gate).
  __device__ __forceinline__ uint4 prf(const AesRK &kd, uint32_t gate, uint32_t field, uint64_t idx) const {
    uint4 b;
    b.x = uint32_t(idx);
    b.y = uint32_t(idx >> 32);
    b.z = field;
    b.w = gate;
    return enc(b, kd);
  }
};

// AesPerm2 with single blocks in the scheduler's own order, which starts a column
// while the reads of the next ones are on their way: with a single chain a phase
// forms all four columns and then waits for all reads.  25 hashes one after another
// take 34 against 41 us with one wave per SIMD, 42-45 in both orders with 1.5 and two
// and 72-73 with four; but the order needs more registers, and one held to 64 of them
// keeps few reads in flight (146 against 103 us for 64-bit ReLUs of 160 elements per
// CU).  For gates of few waves and for kernels that draw PRF blocks one by one; the
// others, the gates' dealer among them (1.4 M EXTRELU keys 530 against 535 us), stay
// in phases.
struct AesPerm2Few : AesPerm2 {
  using AesPerm2::AesPerm2;
  __device__ __forceinline__ uint32_t col(uint32_t a, uint32_t b, uint32_t c, uint32_t d, uint32_t k) const {
    const uint32_t h = xor3(t0<2>(c), t1<3>(d), (k << 16) | (k >> 16));
    return xor3(t0<0>(a), t1<1>(b), __builtin_amdgcn_alignbit(h, h, 16));
  }
  __device__ __forceinline__ uint32_t last(uint32_t a, uint32_t b, uint32_t c, uint32_t d) const {
    const uint32_t lo = __builtin_amdgcn_perm(t0<1>(b), t0<0>(a), 0x0c0c0501u);
    const uint32_t hi = __builtin_amdgcn_perm(t0<3>(d), t0<2>(c), 0x0c0c0501u);
    return (hi << 16) | lo;
  }
  // the block from its whitened input to before the last round key
  __device__ __forceinline__ uint4 block(uint4 c, const AesRK &rk) const {
#pragma unroll
    for (int r = 1; r < 10; r++) {
      const uint32_t n0 = col(c.x, c.y, c.z, c.w, rk.w[4 * r + 0]);
      const uint32_t n1 = col(c.y, c.z, c.w, c.x, rk.w[4 * r + 1]);
      const uint32_t n2 = col(c.z, c.w, c.x, c.y, rk.w[4 * r + 2]);
      const uint32_t n3 = col(c.w, c.x, c.y, c.z, rk.w[4 * r + 3]);
      c = make_uint4(n0, n1, n2, n3);
    }
    return make_uint4(last(c.x, c.y, c.z, c.w), last(c.y, c.z, c.w, c.x), last(c.z, c.w, c.x, c.y),
                      last(c.w, c.x, c.y, c.z));
  }
  __device__ __forceinline__ uint4 enc(uint4 in, const AesRK &rk) const {
    const uint4 o = block(whiten(in, rk), rk);
    return make_uint4(o.x ^ rk.w[40], o.y ^ rk.w[41], o.z ^ rk.w[42], o.w ^ rk.w[43]);
  }
  __device__ __forceinline__ uint4 hash(uint4 s, const AesRK &rk) const {
    const uint4 o = block(hash_in(s, rk), rk);
    return make_uint4(xor3(o.x, rk.w[40], s.z), xor3(o.y, rk.w[41], s.w), xor3(o.z, rk.w[42], s.z) ^ s.x,
                      xor3(o.w, rk.w[43], s.w) ^ s.y);
  }
  __device__ __forceinline__ uint4 prf(const AesRK &kd, uint32_t gate, uint32_t field, uint64_t idx) const {
    return enc(make_uint4(uint32_t(idx), uint32_t(idx >> 32), field, gate), kd);
  }
};

// Quad-lane AES on the AesPerm2 table, for latency-bound launches: four
// consecutive lanes (a quad) hold one block, lane j its column c_j.  A round has
// each lane look up its own column's four bytes -- A = T0[b0], B = T1[b1],
// C = T0[b2], D = T1[b3] -- and take the other three terms of its new column from
// the quad's other lanes (DPP quad permutes):
//   n_j = A_j ^ B_(j+1) ^ rotl(C_(j+2) ^ D_(j+3) ^ rotl(k_j, 16), 16),
// 10 VALU instructions and 4 table reads per lane and round instead of 28 and 16
// for one lane per block, so a round's dependent chain is shorter.  Every lane of
// a quad must run the same code (the permutes read the other three lanes).
struct AesQuad {
  const AesPerm2 &t;
  uint32_t j;  // the lane's column (lane mod 4)
  __device__ AesQuad(const AesPerm2 &tab) : t(tab), j(threadIdx.x & 3u) {}

  // DPP quad permutes: the value of lane (j + d) mod 4 of the quad
  __device__ __forceinline__ static uint32_t from1(uint32_t v) { return __builtin_amdgcn_mov_dpp(int(v), 0x39, 0xf, 0xf, false); }
  __device__ __forceinline__ static uint32_t from2(uint32_t v) { return __builtin_amdgcn_mov_dpp(int(v), 0x4e, 0xf, 0xf, false); }
  __device__ __forceinline__ static uint32_t from3(uint32_t v) { return __builtin_amdgcn_mov_dpp(int(v), 0x93, 0xf, 0xf, false); }
  // the value of the quad's lane 0, and the xor over the quad
  __device__ __forceinline__ static uint32_t lane0(uint32_t v) { return __builtin_amdgcn_mov_dpp(int(v), 0x00, 0xf, 0xf, false); }
  __device__ __forceinline__ static uint32_t quad_xor(uint32_t v) {
    v ^= __builtin_amdgcn_mov_dpp(int(v), 0xb1, 0xf, 0xf, false);  // lanes 1,0,3,2
    return v ^ __builtin_amdgcn_mov_dpp(int(v), 0x4e, 0xf, 0xf, false);
  }

  // The lane's round-key words of rk: k[0] and k[10] as they are, k[1..9]
  // rotated by 16 (the rotation the round folds in).
  struct Keys {
    uint32_t k[11];
  };
  __device__ __forceinline__ Keys keys(const AesRK &rk) const {
    Keys o;
#pragma unroll
    for (int r = 0; r < 11; r++) {
      const uint32_t w = rk.w[4 * r + int(j)];
      o.k[r] = (r == 0 || r == 10) ? w : ((w << 16) | (w >> 16));
    }
    return o;
  }

  __device__ __forceinline__ uint32_t enc(uint32_t c, const Keys &k) const {
    c ^= k.k[0];
#pragma unroll
    for (int r = 1; r < 10; r++) {
      const uint32_t a = t.t0<0>(c), b = t.t1<1>(c), cc = t.t0<2>(c), d = t.t1<3>(c);
      const uint32_t h = xor3(from2(cc), from3(d), k.k[r]);
      c = xor3(a, from1(b), __builtin_amdgcn_alignbit(h, h, 16));
    }
    // last round: S[x] is byte 1 of T0[x]; the lane packs the S bytes of its own
    // column, byte i of the new column comes from lane j + i
    const uint32_t lo = __builtin_amdgcn_perm(t.t0<1>(c), t.t0<0>(c), 0x0c0c0501u);
    const uint32_t hi = __builtin_amdgcn_perm(t.t0<3>(c), t.t0<2>(c), 0x0c0c0501u);
    const uint32_t P = (hi << 16) | lo;
    const uint32_t x01 = __builtin_amdgcn_perm(from1(P), P, 0x0c0c0500u);       // bytes 0 (own), 1 (lane j+1)
    const uint32_t x23 = __builtin_amdgcn_perm(from3(P), from2(P), 0x07020c0cu);  // bytes 2 (lane j+2), 3 (j+3)
    return (x01 | x23) ^ k.k[10];
  }

  // H(s) = AES_k(sigma(s)) ^ sigma(s), sigma(xL||xR) = (xL^xR)||xL, xR = words 0,1:
  // sigma_j = s_(j^2), and ^ s_j for j >= 2
  __device__ __forceinline__ uint32_t hash(uint32_t s, const Keys &k) const {
    const uint32_t sg = from2(s) ^ ((j & 2u) ? s : 0u);
    return enc(sg, k) ^ sg;
  }
};

// NT = 0 selects the permute-addressed single table (REP must be 64); NT = 2
// (REP 32) the interleaved pair.
template <int NT, int REP>
struct AesSel {
  using type = AesTab<NT, REP>;
};
template <>
struct AesSel<0, 64> {
  using type = AesPerm;
};
// NT = 2, REP = 32: T0 and T1 interleaved in one table (AesPerm2)
template <>
struct AesSel<2, 32> {
  using type = AesPerm2;
};
template <int NT, int REP>
using AesLds = typename AesSel<NT, REP>::type;

// The table type of kernels that draw PRF blocks one by one.
template <int NT, int REP>
using AesPrf = std::conditional_t<std::is_same<AesLds<NT, REP>, AesPerm2>::value, AesPerm2Few, AesLds<NT, REP>>;

// Table types whose enc2 and hash2 run two blocks side by side
template <class A>
constexpr bool kTwoChains = std::is_base_of<AesPerm2, A>::value || std::is_same<A, AesPerm>::value;

// Two dealer PRF blocks of one key, side by side where the table type can.
template <class A>
__device__ __forceinline__ void enc_pair(const A &aes, const AesRK &k, uint4 u, uint4 v, uint4 *eu, uint4 *ev) {
  if constexpr (kTwoChains<A>) {
    aes.enc2(u, v, k, eu, ev);
  } else {
    *eu = aes.enc(u, k);
    *ev = aes.enc(v, k);
  }
}
__device__ __forceinline__ uint4 prf_block(uint32_t gate, uint32_t field, uint64_t idx) {
  return make_uint4(uint32_t(idx), uint32_t(idx >> 32), field, gate);
}
// fields f0 and f1 of index idx
template <class A>
__device__ __forceinline__ void prf2(const A &aes, const AesRK &k, uint32_t gate, uint32_t f0, uint32_t f1,
                                     uint64_t idx, uint4 *o0, uint4 *o1) {
  enc_pair(aes, k, prf_block(gate, f0, idx), prf_block(gate, f1, idx), o0, o1);
}

// a ^ (b & m) in one v_bitop3_b32 (truth table 0x78 = 0xf0 ^ (0xcc & 0xaa))
__device__ __forceinline__ uint32_t xor_and(uint32_t a, uint32_t b, uint32_t m) {
  return __builtin_amdgcn_bitop3_b32(a, b, m, 0x78);
}
__device__ __forceinline__ uint4 xor_and4(uint4 a, uint4 b, uint32_t m) {
  return make_uint4(xor_and(a.x, b.x, m), xor_and(a.y, b.y, m), xor_and(a.z, b.z, m), xor_and(a.w, b.w, m));
}
__device__ __forceinline__ uint4 xor4(uint4 a, uint4 b) {
  return make_uint4(a.x ^ b.x, a.y ^ b.y, a.z ^ b.z, a.w ^ b.w);
}
__device__ __forceinline__ uint4 and4(uint4 a, uint32_t m) {
  return make_uint4(a.x & m, a.y & m, a.z & m, a.w & m);
}

// parity of the bits of b at positions > pos, pos in [0, 127]
__device__ __forceinline__ uint32_t parity_above(uint4 b, uint32_t pos) {
  uint32_t acc = 0;
  const uint32_t w[4] = {b.x, b.y, b.z, b.w};
#pragma unroll
  for (int k = 0; k < 4; k++) {
    uint32_t lo = 32u * k;
    uint32_t m;
    if (pos < lo)
      m = 0xffffffffu;
    else if (pos >= lo + 31)
      m = 0u;
    else
      m = 0xffffffffu << (pos - lo + 1);
    acc ^= w[k] & m;
  }
  return __popc(acc) & 1u;
}

}  // namespace mpcx
