// dcf_dev.h -- device-side half-tree DPF/DCF walks (evaluation and dealer).
//
// Evaluation of the comparison [x < alpha] (m-bit x): walk the DPF tree of the
// point alpha along the bits of x, MSB first.  At every level where the bit of x
// is 0 the right sibling's control bit is XORed into the output: the two parties'
// control bits differ exactly on the path of alpha, so the XOR of both outputs is
// 1 iff the path of alpha leaves the path of x to the right, i.e. x < alpha.  The
// 128-bit leaf holds the last 7 levels as a one-hot block, and the bits above
// the low 7 bits of x are folded in with a parity.  This is the DPF-based DCF the
// reference builds on (gpu_mpc/dpf_dcf_adapter.h:1-12, gpu_mpc/ddg_orca.h:11-12).
//
// The tree is the half-tree one (Guo et al., EUROCRYPT 2023): one fixed-key AES
// call per level,  sL = H(s) ^ t*CW,  sR = sL ^ s,  t = lsb(s).
#pragma once
#include <type_traits>

#include "aes_dev.h"

namespace mpcx {


// A 16-byte word of a key plane: base is uniform over the workgroup (a scalar
// register pair), off a thread's 32-bit byte offset, so a load carries one
// address register per lane.
__device__ __forceinline__ uint4 ld16(const uint8_t *base, uint32_t off) {
  return *reinterpret_cast<const uint4 *>(base + off);
}

// The planes of a DCF key at a workgroup's tile: pointers to the tile's first
// element, and the distance of two levels' correction words in bytes.
struct DcfTile {
  const uint8_t *cw, *leaf;
  size_t stride;
};

// All ones where bit k of v is set.
__device__ __forceinline__ uint32_t bit_mask(uint32_t v, int k) {
  return uint32_t(__builtin_amdgcn_sbfe(int(v), uint32_t(k), 1u));
}
// The path bits of an m-bit x left-aligned: the sign bit is the next level's, and
// after the levels the low 7 bits of x (all of it for m < 7) are on top.
template <typename X>
struct PathBits {
  X v;
  __device__ __forceinline__ PathBits(X x, int m) : v(X(x << (int(8 * sizeof(X)) - m))) {}
  __device__ __forceinline__ uint32_t next() {  // mask of the level's bit
    const uint32_t r = uint32_t(int32_t(uint32_t(v >> (8 * sizeof(X) - 32))) >> 31);
    v = X(v << 1);
    return r;
  }
  __device__ __forceinline__ uint32_t leaf_pos(int m) const { return uint32_t(v >> (int(8 * sizeof(X)) - (m < 7 ? m : 7))); }
};
// (a ^ b) & ~m and a ^ (b & m) as one v_bitop3_b32 each
__device__ __forceinline__ uint32_t xor_andn(uint32_t a, uint32_t b, uint32_t m) {
  return __builtin_amdgcn_bitop3_b32(a, b, m, 0x14);
}

// One party's walk: s the party's root; t and the path bits are kept as masks.
// A level's correction word is loaded at its start and used after its hash, some
// thousand clocks later, so none is held a level ahead.
template <class A, typename X>
__device__ __forceinline__ uint32_t dcf_eval_walk(const A &aes, uint4 s, int m, int L, const DcfTile &k, uint32_t off,
                                                  X x) {
  uint32_t t = bit_mask(s.x, 0), out = 0;
  PathBits<X> path(x, m);
  const uint8_t *cw = k.cw;
  for (int l = 0; l < L; l++, cw += k.stride) {
    const uint4 c = ld16(cw, off);
    const uint32_t bit = path.next();
    const uint4 sl = xor_and4(aes.hash(s, c_rkH), c, t);
    const uint32_t tl = bit_mask(sl.x, 0);
    out ^= xor_andn(tl, t, bit);
    s = xor_and4(sl, s, bit);
    t = xor_and(tl, t, bit);
  }
  const uint4 leaf = ld16(k.leaf, off);
  const uint4 lb = xor_and4(aes.hash(s, c_rkL), leaf, t);
  return (out & 1u) ^ parity_above(lb, path.leaf_pos(m));
}

// Both parties' hashes of a level: side by side on the T0/T1 table, one after
// the other on the other layouts.
template <class A>
__device__ __forceinline__ void hash_pair(const A &aes, uint4 s, uint4 u, const AesRK &rk, uint4 *hs, uint4 *hu) {
  if constexpr (kTwoChains<A>) {
    aes.hash2(s, u, rk, hs, hu);
  } else {
    *hs = aes.hash(s, rk);
    *hu = aes.hash(u, rk);
  }
}

// Both parties' walks of one element in one thread, from their roots s0 and s1
// (the correction words and the leaf are common to the two keys): the XOR of
// the two parties' outputs, i.e. the reconstructed bit.  Each level hashes the
// two seeds side by side and reads its correction word once.
template <class A, typename X>
__device__ __forceinline__ uint32_t dcf_eval_walk2(const A &aes, uint4 s0, uint4 s1, int m, int L, const DcfTile &k,
                                                   uint32_t off, X x) {
  uint32_t t0 = bit_mask(s0.x, 0), t1 = bit_mask(s1.x, 0), out = 0;
  PathBits<X> path(x, m);
  const uint8_t *cw = k.cw;
  for (int l = 0; l < L; l++, cw += k.stride) {
    const uint4 c = ld16(cw, off);
    const uint32_t bit = path.next();
    uint4 h0, h1;
    hash_pair(aes, s0, s1, c_rkH, &h0, &h1);
    const uint4 sl0 = xor_and4(h0, c, t0), sl1 = xor_and4(h1, c, t1);
    const uint32_t tl0 = bit_mask(sl0.x, 0), tl1 = bit_mask(sl1.x, 0);
    out ^= xor_andn(tl0 ^ tl1, t0 ^ t1, bit);
    s0 = xor_and4(sl0, s0, bit);
    s1 = xor_and4(sl1, s1, bit);
    t0 = xor_and(tl0, t0, bit);
    t1 = xor_and(tl1, t1, bit);
  }
  const uint4 leaf = ld16(k.leaf, off);
  uint4 l0, l1;
  hash_pair(aes, s0, s1, c_rkL, &l0, &l1);
  const uint4 lb = xor4(xor_and4(l0, leaf, t0), xor_and4(l1, leaf, t1));
  return (out & 1u) ^ parity_above(lb, path.leaf_pos(m));
}

// The same walk on the quad-lane AES (latency-bound launches): lane j of a quad
// holds word j of the seed, of every correction word (cw: where the lane's word of
// level 0, cw0, is; levels stride_words apart, each loaded a level ahead) and of
// the leaf; the control bits are bit
// 0 of word 0 (lane 0's), and the leaf's parity above pos is the xor of the four
// lanes' parities of their 32 bits.  Every lane of the quad returns the bit.
template <typename X>
__device__ __forceinline__ uint32_t dcf_eval_walk_quad(const AesQuad &aes, const AesQuad::Keys &kH,
                                                       const AesQuad::Keys &kL, uint32_t s, int m, int L,
                                                       uint32_t cw0, const uint32_t *__restrict__ cw,
                                                       size_t stride_words, uint32_t leaf, X x) {
  uint32_t t = bit_mask(AesQuad::lane0(s), 0), out = 0, cnext = cw0;
  PathBits<X> path(x, m);
  for (int l = 0; l < L; l++) {
    const uint32_t c = cnext;
    cw += stride_words;
    if (l + 1 < L) cnext = *cw;
    const uint32_t bit = path.next();
    const uint32_t sl = xor_and(aes.hash(s, kH), c, t);
    const uint32_t tl = bit_mask(AesQuad::lane0(sl), 0);
    out ^= xor_andn(tl, t, bit);
    s = xor_and(sl, s, bit);
    t = xor_and(tl, t, bit);
  }
  const uint32_t lb = xor_and(aes.hash(s, kL), leaf, t);
  const uint32_t pos = path.leaf_pos(m);
  const uint32_t lo = 32u * aes.j;
  const uint32_t msk = pos < lo ? 0xffffffffu : (pos >= lo + 31 ? 0u : 0xffffffffu << (pos - lo + 1));
  return (out ^ AesQuad::quad_xor(__popc(lb & msk))) & 1u;
}

struct DcfGenOut {
  uint4 s0;      // party 0's final on-path seed
  uint32_t t0;   // party 0's final on-path control bit, as a mask
  uint4 leafcw;  // leaf correction word
};

__device__ __forceinline__ void st16(uint8_t *base, uint32_t off, uint4 v) {
  *reinterpret_cast<uint4 *>(base + off) = v;
}
// a ^ (b & ~m) in one v_bitop3_b32
__device__ __forceinline__ uint32_t xor_not_and(uint32_t a, uint32_t b, uint32_t m) {
  return __builtin_amdgcn_bitop3_b32(a, b, m, 0xb4);
}

// Dealer walk for element base + e from the parties' root seeds s0 (lsb 0) and s1
// (lsb 1), both parties' seeds hashed side by side: writes the roots, the level
// correction words (level-major) and the leaf correction word of both keys.
// base is uniform over the wave.
template <class A, typename X>
__device__ __forceinline__ DcfGenOut dcf_gen_walk(const A &aes, uint4 s0, uint4 s1, const DcfLayout &d, X alpha,
                                                  size_t base, uint32_t e, uint8_t *k0, uint8_t *k1) {
  const uint4 D = xor4(s0, s1);
  const uint32_t off = 16 * e;
  st16(k0 + d.off_root + 16 * base, off, s0);
  st16(k1 + d.off_root + 16 * base, off, s1);
  uint32_t t0 = 0, t1 = ~0u;
  uint8_t *c0 = k0 + d.off_cw + 16 * base, *c1 = k1 + d.off_cw + 16 * base;
  PathBits<X> path(alpha, d.m);
  for (int l = 0; l < d.L; l++, c0 += 16 * d.N, c1 += 16 * d.N) {
    const uint32_t a = path.next();
    uint4 h0, h1;
    hash_pair(aes, s0, s1, c_rkH, &h0, &h1);
    uint4 cw;  // h0 ^ h1 ^ (a ? 0 : D)
    cw.x = xor_not_and(h0.x ^ h1.x, D.x, a);
    cw.y = xor_not_and(h0.y ^ h1.y, D.y, a);
    cw.z = xor_not_and(h0.z ^ h1.z, D.z, a);
    cw.w = xor_not_and(h0.w ^ h1.w, D.w, a);
    st16(c0, off, cw);
    st16(c1, off, cw);
    s0 = xor_and4(xor_and4(h0, cw, t0), s0, a);
    s1 = xor_and4(xor_and4(h1, cw, t1), s1, a);
    t0 = bit_mask(s0.x, 0);
    t1 = bit_mask(s1.x, 0);
  }
  const uint32_t pos = path.leaf_pos(d.m);
  uint4 l0, l1;
  hash_pair(aes, s0, s1, c_rkL, &l0, &l1);
  uint4 lcw = xor4(l0, l1);
  const uint32_t bitv = 1u << (pos & 31u);
  lcw.x ^= (pos >> 5) == 0 ? bitv : 0u;
  lcw.y ^= (pos >> 5) == 1 ? bitv : 0u;
  lcw.z ^= (pos >> 5) == 2 ? bitv : 0u;
  lcw.w ^= (pos >> 5) == 3 ? bitv : 0u;
  st16(k0 + d.off_leaf + 16 * base, off, lcw);
  st16(k1 + d.off_leaf + 16 * base, off, lcw);
  return {s0, t0, lcw};
}

// Roots drawn from the dealer PRF: s0 = PRF(fb) with lsb 0, s1 = s0 ^ D,
// D = PRF(fb + 1) with lsb 1.
template <class A>
__device__ __forceinline__ void dealer_roots(const A &aes, const AesRK &kd, uint32_t gate, uint32_t fb, size_t i,
                                             uint4 *s0, uint4 *s1) {
  uint4 D;
  prf2(aes, kd, gate, fb, fb + 1, i, s0, &D);
  s0->x &= ~1u;
  D.x |= 1u;
  *s1 = xor4(*s0, D);
}

// Root seed of party p for a DCF drawn from the party's own PRF key: lsb = p.
template <class A>
__device__ __forceinline__ uint4 party_root(const A &aes, const AesRK &kp, int p, uint32_t gate, uint32_t fb,
                                            size_t i) {
  uint4 s = aes.prf(kp, gate, fb + 0, i);
  s.x = (s.x & ~1u) | uint32_t(p);
  return s;
}
// The same and the party's output-mask bit (field fb + 2).
template <class A>
__device__ __forceinline__ uint4 party_root_bit(const A &aes, const AesRK &kp, int p, uint32_t gate, uint32_t fb,
                                                size_t i, uint32_t *z) {
  uint4 s, b;
  prf2(aes, kp, gate, fb, fb + 2, i, &s, &b);
  s.x = (s.x & ~1u) | uint32_t(p);
  *z = b.x & 1u;
  return s;
}

}  // namespace mpcx
