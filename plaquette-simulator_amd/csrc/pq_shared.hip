// Shared-X/Z persistent kernels (gfx950).
//
// H, S, CX, CZ and measurements change X and Z in every shot alike, so a
// program without flagged H/S/CX/CZ that starts from |0...0> keeps the X/Z
// words of a 64-shot group all zeros or all ones throughout: one bit instead
// of 64 per entry.  The kernels here run a whole compiled program on that
// packed tableau, in one workgroup per 1, 2 or 4 word groups, and write the
// groups' 64-shot words once at the end.  Per workgroup they keep
//  * X and Z as bits, one column of KW = 2 KH + 1 words per x_q and z_q
//    (KH = ceil(n/64)): KH words of destabilizer rows, KH words of stabilizer
//    rows, so rows i and n+i share a bit position, and one word whose bit 0
//    is the scratch row;
// and per word group
//  * the signs as R[i] = Rv[i] ^ rc[i] ^ <E, P_i>: a 64-shot word per row
//    that only measurements change, a bit per row for what all shots share
//    (gate phases, rowsum phases), and a Pauli frame E (an x and a z word of
//    64 shots per qubit).  A Pauli applied to some shots flips the sign of
//    the rows that anticommute with it, so noise, flagged and plain Paulis
//    cost two words of E; E moves through the gates like a row; the symplectic
//    product <E, .> is additive under rowsums.
//
// What this saves: the per-shot kernel (k_program_t) moves and computes
// R = 2n+1 words of 64 shots per column and gate; here a column is 2 n/64 words
// of rows.  Up to 464 qubits (487 in programs without noise and flags) the packed
// columns (2n (2 n/64 + 1) words) sit in LDS; up to 2048 they sit at the start
// of a group's tableau block, which the run overwrites anyway.
#include "pq_kernels.h"

#include <algorithm>
#include <type_traits>

#include "plaquette_amd.h"

namespace pq {

namespace {

#define PQ_CONST __attribute__((address_space(4)))

// wide states: columns a lane has in flight, in determined chains and in the
// rowsums of random measurements (more spill registers)
constexpr uint32_t kWideCols = 5, kRandCols = 6;
constexpr uint32_t kWindow = 64;       // measurements whose pivots are checked at once

__device__ __forceinline__ uint32_t lane_id() { return threadIdx.x & 63u; }
__device__ __forceinline__ uint32_t rfl(uint32_t v) { return __builtin_amdgcn_readfirstlane(v); }
__device__ __forceinline__ uint64_t rfl64(uint64_t v) {
  return (uint64_t)rfl((uint32_t)v) | ((uint64_t)rfl((uint32_t)(v >> 32)) << 32);
}
__device__ __forceinline__ uint64_t read_lane64(uint64_t v, uint32_t l) {
  const uint32_t lo = __builtin_amdgcn_readlane((uint32_t)v, l);
  const uint32_t hi = __builtin_amdgcn_readlane((uint32_t)(v >> 32), l);
  return (uint64_t)lo | ((uint64_t)hi << 32);
}
__device__ __forceinline__ uint64_t wave_xor(uint64_t v) {
#pragma unroll
  for (uint32_t off = 32; off > 0; off >>= 1) v ^= __shfl_xor(v, off, 64);
  return v;
}
__device__ __forceinline__ void lds_xor(uint64_t *p, uint64_t v) {
  atomicXor(reinterpret_cast<unsigned long long *>(p), (unsigned long long)v);
}
// Bit i of the result: parity of bits 0..i of v.
__device__ __forceinline__ uint64_t prefix_parity(uint64_t v) {
  v ^= v << 1;
  v ^= v << 2;
  v ^= v << 4;
  v ^= v << 8;
  v ^= v << 16;
  v ^= v << 32;
  return v;
}

// Per-wave total of small counts v, mod 4, as its bit 1.
__device__ __forceinline__ uint32_t wave_sum_bit1(uint32_t v) {
  const uint32_t b0 = (uint32_t)__popcll(__ballot(v & 1u));
  const uint32_t b1 = (uint32_t)__popcll(__ballot((v >> 1) & 1u));
  return ((b0 >> 1) ^ b1) & 1u;
}

// One staged op: `cw` = the flags below, and from bit 12 the ops of the layer
// part it opens, or the measurements left in its run; `qq` = qa | qb << 16 (qb
// = qa for one-qubit ops).  Its four masks (per word group) are what the noise after it XORs into the
// frame's x and z words of qa and of qb; a flagged op keeps its flag in the
// third, and with a record as its flag the record in the fourth.  A
// measurement has record | coin threshold << 32 and its sequence number there.
struct SharedOp {
  uint32_t cw, qq;
};
constexpr uint32_t kOpH = 1, kOpS = 2, kOpCX = 4, kOpCZ = 8;
constexpr uint32_t kOpMeas = 1u << 4;
constexpr uint32_t kOpMasks = 1u << 5;    // some mask word may not be zero
constexpr uint32_t kOpNotX = 1u << 6, kOpNotZ = 1u << 7;  // a Pauli on every shot: x, z flip
constexpr uint32_t kOpFlagX = 1u << 10, kOpFlagZ = 1u << 11;  // flagged: the flag goes to x, z
constexpr uint32_t kOpRecord = 1u << 24;  // the flag is a record
constexpr uint32_t kOpDropped = 1u << 8;  // a later measurement writes its record
constexpr uint32_t kOpRandom = 1u << 9;   // a measurement found random (set when it runs)
constexpr uint32_t kOpLenShift = 12, kOpLenMask = 0xFFFu;

constexpr uint32_t kMaxRowWords = 2 * (kSharedMaxQubits / 64) + 2;
struct SharedLds {
  SharedOp ops[kStage + 1];
  uint64_t rc[kMaxRowWords];  // sign bits, laid out like a column
  uint64_t sm[kMaxRowWords];  // row mask of the current random measurement
  uint64_t c0[kMaxRowWords];  // and the low bits of its rows' phase sums
  uint32_t list[512];         // its pivot row's columns (columns in the tableau: in dynamic LDS)
  uint32_t bad;               // a word of the state is not the |0...0> tableau's
  // determined measurements of wide states, two in turn: phase count, XOR of
  // Rv rows
  uint32_t tot[2];
  uint64_t rx[2][kSharedMaxGroups];
  uint32_t nl;                // entries of list
  uint64_t item;
};
constexpr uint64_t kSharedLdsBytes = 159 * 1024 - sizeof(SharedLds);  // dynamic LDS cap

// Dynamic LDS words: Rv and the frame of each of the G word groups, their op
// masks (programs with noise or flags), and the packed columns if they fit.
// (Programs without masks keep only the measurements' two words there.)
__host__ __device__ inline uint64_t mask_words(bool masked, uint32_t gs) {
  return masked ? (4ull * kStage) << gs : 2ull * kStage;
}
__host__ __device__ inline uint64_t groups_words(uint32_t n, bool masked, uint32_t gs) {
  return ((4ull * n + 1) << gs) + mask_words(masked, gs);
}
__host__ __device__ inline uint64_t packed_words(uint32_t n) {
  return 2ull * n * (2ull * ((n + 63) / 64) + 1);
}
__host__ __device__ inline bool packed_in_lds(uint32_t n, bool masked) {
  return (groups_words(n, masked, 0) + packed_words(n)) * 8 <= kSharedLdsBytes;
}

// Runs the program on word groups w0 .. w0 + G - 1 (those below a.W), which
// share the packed X/Z, G = 1 << gs.  Groups whose X/Z are not the |0...0>
// tableau (kSharedVerify: looked at here; kSharedChecked: told by a.done) are
// left untouched.  Returns the groups that ran as a bit mask.  With a.packed
// the 64-shot X/Z words are left to k_shared_expand, which reads the packed
// columns there.
template <bool kLds>
__device__ uint32_t shared_words(const ProgramArgs &a, uint64_t seed, uint64_t mseq0, uint64_t w0,
                                 uint32_t gs, uint64_t *dyn, SharedLds &sh) {
  const uint32_t tid = threadIdx.x, NT = blockDim.x, lane = lane_id();
  const uint32_t wv = rfl(tid >> 6), nw = NT >> 6;
  const uint32_t n = a.n, R = a.R;
  const uint32_t KH = (n + 63) / 64, K2 = 2 * KH, KW = K2 + 1;
  const uint64_t W = a.W;
  const uint32_t G = 1u << gs, g_mask = G - 1;
  const uint64_t blk = (uint64_t)a.C * R;
  uint64_t *const T0 = a.tab + w0 * blk;  // group g's block: T0 + g * blk
  const bool masked = a.masked;
  // per-group arrays: group g's Rv at g * R, its frame at g * 2n, its masks of
  // op t at (t * G + g) * 4
  uint64_t *Rv = dyn;
  uint64_t *E = Rv + R * G;
  uint64_t *msk = E + 2 * n * G;
  const uint32_t mstep = masked ? 4 * G : 2;  // op t's measurement words: msk + t * mstep
  uint64_t *const rc = sh.rc;
  const PQ_CONST DInstr *ins = (const PQ_CONST DInstr *)a.instrs;

  uint32_t live = w0 + G <= W ? (1u << G) - 1 : (1u << (W - w0)) - 1;
  if (a.shared == kSharedChecked) {
    for (uint32_t g = 0; g < G; ++g)
      if (((live >> g) & 1) && !rfl(a.done[w0 + g])) live &= ~(1u << g);
  } else if (a.shared == kSharedVerify) {
    // word t of the X/Z block is all ones iff t is a multiple of R + 1
    if (tid == 0) sh.bad = 0;
    __syncthreads();
    const uint32_t total = 2 * n * R, M = R + 1, step = NT % M;
    for (uint32_t g = 0; g < G; ++g) {
      if (!((live >> g) & 1)) continue;
      const uint64_t *T = T0 + g * blk;
      uint32_t rem = tid % M;
      for (uint32_t base = tid; base < total; base += 8 * NT) {
        uint64_t v[8];
#pragma unroll
        for (uint32_t u = 0; u < 8; ++u) v[u] = T[min(base + u * NT, total - 1)];
        bool bad = false;
#pragma unroll
        for (uint32_t u = 0; u < 8; ++u) {
          bad |= base + u * NT < total && v[u] != (rem == 0 ? ~0ull : 0ull);
          rem += step;
          if (rem >= M) rem -= M;
        }
        if (bad) atomicOr(&sh.bad, 1u << g);
        if (__ballot(bad) || ((*(volatile uint32_t *)&sh.bad >> g) & 1)) break;
      }
    }
    __syncthreads();
    live &= ~rfl(sh.bad);
    if (tid < G && w0 + tid < W) a.done[w0 + tid] = (live >> tid) & 1;
  }
  if (!live) return 0;

  // packed column c (x_c, or z_{c-n}) starts at P + c * KW: one compact block,
  // in LDS, or at the start of a group's tableau block, which the run
  // overwrites anyway
  uint64_t *const past = msk + mask_words(masked, gs);
  uint64_t *P = kLds ? past : T0 + ((uint32_t)__ffs((int)live) - 1) * blk;
  uint32_t *const list = kLds ? sh.list : reinterpret_cast<uint32_t *>(past);

  // ---- |0...0>: destabilizer i = X_i, stabilizer i = Z_i ----
  for (uint32_t u = tid; u < 2 * n * KW; u += NT) {
    const uint32_t c = u / KW, k = u - c * KW;
    const uint32_t q = c < n ? c : c - n;
    const uint32_t kq = (c < n ? 0 : KH) + (q >> 6);
    P[c * KW + k] = k == kq ? 1ull << (q & 63) : 0ull;
  }
  for (uint32_t g = 0; g < G; ++g)
    for (uint32_t i = tid; i < R; i += NT)
      Rv[g * R + i] = (live >> g) & 1 ? T0[g * blk + 2ull * n * R + i] : 0ull;
  for (uint32_t i = tid; i < 2 * n * G; i += NT) E[i] = 0;
  if (tid < KW) rc[tid] = 0;
  if (tid < 2) {
    sh.tot[tid] = 0;
    for (uint32_t g = 0; g < kSharedMaxGroups; ++g) sh.rx[tid][g] = 0;
  }
  __syncthreads();

  // this thread's share of a layer's column work: word my_k of every opp-th op
  const uint32_t opp = NT / KW;
  const uint32_t my_op = tid / KW, my_k = tid - my_op * KW;
  const bool on = my_op < opp;
  // and of a random measurement's: word my_i of every rpp-th of its columns
  const uint32_t rpp = NT / K2;
  const uint32_t my_j = tid / K2, my_i = tid - my_j * K2;

  uint64_t rp = 0;    // sign flips of row word my_k, not yet in rc
  uint32_t slot2 = 0; // which of sh.tot / sh.rx is in use (wide states)
  for (uint32_t base = 0; base < a.ninstr;) {
    const uint32_t wn = min(kStage, a.ninstr - base);
    // instructions [base, base + wn) and their masks, whatever segments they
    // belong to: two dependent loads per window, not per segment
    bool flags = false;
    const uint32_t ss = masked ? gs : 0;  // one thread per op and group, or per op
    for (uint32_t u = tid; u < wn << ss; u += NT) {
      const uint32_t t = u >> ss, g = u & ((1u << ss) - 1);
      const PQ_CONST DInstr *I = ins + base + t;
      const uint32_t code = I->code, qa = I->qa, qb = I->qb, slot = I->slot, na = I->na,
                     nb = I->nb, t0 = I->t0, pad = I->pad;
      SharedOp J;
      if (code == PQ_OP_M) {
        J.cw = kOpMeas | (pad & kMeasSuperseded ? kOpDropped : 0u) |
               (min(pad >> kMeasLeftShift, kStage) << kOpLenShift);
        J.qq = qa;
        if (g == 0) {
          msk[t * mstep] = (uint64_t)slot | ((uint64_t)t0 << 32);
          msk[t * mstep + 1] = (uint64_t)na | ((uint64_t)nb << 32);
        }
      } else {
        const bool two = code == PQ_OP_CX || code == PQ_OP_CZ;
        const bool flg = code >= PQ_OP_H_FLAG && code != PQ_OP_NOISE;
        const bool rec = flg && !(slot & kSlotPlane);
        const bool px = code == PQ_OP_X || code == PQ_OP_Y || code == PQ_OP_X_FLAG ||
                        code == PQ_OP_Y_FLAG;
        const bool pz = code == PQ_OP_Z || code == PQ_OP_Y || code == PQ_OP_Z_FLAG ||
                        code == PQ_OP_Y_FLAG;
        J.cw = (code == PQ_OP_H ? kOpH : code == PQ_OP_S ? kOpS : 0u) |
               (code == PQ_OP_CX ? kOpCX : code == PQ_OP_CZ ? kOpCZ : 0u) |
               (px ? (flg ? kOpFlagX : kOpNotX) : 0u) | (pz ? (flg ? kOpFlagZ : kOpNotZ) : 0u) |
               (rec ? kOpRecord : 0u) | (na != kNone || nb != kNone || flg ? kOpMasks : 0u) |
               (((pad >> kLayerLenShift) & kLayerLenMask) << kOpLenShift);
        J.qq = qa | ((two ? qb : qa) << 16);
        if (J.cw & kOpMasks) {
          const uint64_t w = min(w0 + g, W - 1);
          const PQ_CONST uint64_t *gp = (const PQ_CONST uint64_t *)a.planes + 2ull * a.nk * w;
          uint64_t m0 = 0, m1 = 0, m2 = 0, m3 = 0;
          if (na != kNone) {
            m0 = gp[2ull * na];
            m1 = gp[2ull * na + 1];
          }
          if (nb != kNone) {
            m2 = gp[2ull * nb];
            m3 = gp[2ull * nb + 1];
          } else if (flg) {
            m2 = rec ? a.recs[(2ull * slot) * W + w] : gp[2ull * (slot & ~kSlotPlane)];
            m3 = slot;
          }
          uint64_t *M = msk + 4 * u;
          M[0] = m0;
          M[1] = m1;
          M[2] = m2;
          M[3] = m3;
          flags |= rec;
        }
      }
      if (g == 0) sh.ops[t] = J;
    }
    // flags from records are read again where measurements of this window
    // precede them
    const bool reread = __syncthreads_or(flags);
    bool measured = false;
    uint32_t b = 0;
    uint32_t cw = rfl(sh.ops[0].cw);  // of op b
    while (b < wn) {
      const uint32_t cnt = max(1u, (cw >> kOpLenShift) & kOpLenMask);
      if (!(cw & kOpMeas)) {
        if (b + cnt > wn) break;  // a layer part runs whole: it opens the next window
        if (measured && reread) {
          for (uint32_t u = (b << gs) + tid; u < wn << gs; u += NT)
            if (sh.ops[u >> gs].cw & kOpRecord)
              msk[4 * u + 2] = a.recs[2ull * msk[4 * u + 3] * W + min(w0 + (u & g_mask), W - 1)];
          __syncthreads();
        }
        measured = false;
        // a layer's ops act on distinct qubits: no barrier inside it
        if (on)
          for (uint32_t o = my_op; o < cnt; o += opp) {
            const SharedOp J = sh.ops[b + o];
            uint64_t *xa = P + (__umul24(J.qq & 0xFFFFu, KW) + my_k), *za = xa + n * KW;
            if (J.cw & kOpCX) {
              uint64_t *xb = P + (__umul24(J.qq >> 16, KW) + my_k), *zb = xb + n * KW;
              const uint64_t x = *xa, z = *za, xt = *xb, zt = *zb;
              rp ^= x & zt & ~(xt ^ z);
              *xb = xt ^ x;
              *za = z ^ zt;
            } else if (J.cw & kOpH) {
              const uint64_t x = *xa, z = *za;
              rp ^= x & z;
              *xa = z;
              *za = x;
            } else if (J.cw & kOpS) {
              const uint64_t x = *xa, z = *za;
              rp ^= x & z;
              *za = z ^ x;
            } else if (J.cw & kOpCZ) {
              uint64_t *xb = P + (__umul24(J.qq >> 16, KW) + my_k), *zb = xb + n * KW;
              const uint64_t x = *xa, z = *za, xt = *xb, zt = *zb;
              rp ^= x & xt & (zt ^ z);
              *zb = zt ^ x;
              *za = z ^ xt;
            }
          }
        // The frame moves through a gate as a row does.  Its words are for the
        // last threads: the column work starts at thread 0, and a wave's
        // instruction stream is the bound here, not the SIMD.
        for (uint32_t u = NT - 1 - tid; u < cnt << gs; u += NT) {
          const SharedOp J = sh.ops[b + (u >> gs)];
          const uint32_t qa = J.qq & 0xFFFFu, qb = J.qq >> 16;
          const uint64_t *M = msk + 4 * ((b << gs) + u);
          uint64_t *Ex = E + (u & g_mask) * 2 * n, *Ez = Ex + n;
          uint64_t ex = Ex[qa], ez = Ez[qa];
          if (J.cw & (kOpCX | kOpCZ)) {
            uint64_t fx = Ex[qb], fz = Ez[qb];
            if (J.cw & kOpCX) {
              fx ^= ex;
              ez ^= fz;
            } else {
              fz ^= ex;
              ez ^= fx;
            }
            if (J.cw & kOpMasks) {
              fx ^= M[2];
              fz ^= M[3];
            }
            Ex[qb] = fx;
            Ez[qb] = fz;
          } else if (J.cw & kOpH) {
            const uint64_t t = ex;
            ex = ez;
            ez = t;
          } else if (J.cw & kOpS) {
            ez ^= ex;
          } else {
            if (J.cw & kOpNotX) ex = ~ex;
            if (J.cw & kOpNotZ) ez = ~ez;
            if (J.cw & kOpFlagX) ex ^= M[2];
            if (J.cw & kOpFlagZ) ez ^= M[2];
          }
          if (J.cw & kOpMasks) {
            ex ^= M[0];
            ez ^= M[1];
          }
          Ex[qa] = ex;
          Ez[qa] = ez;
        }
        b += cnt;
        cw = rfl(sh.ops[b].cw);
        __syncthreads();
        continue;
      }

      // ---- measurements [b, b + mn) ----
      if (!measured) {
        if (on && rp) lds_xor(rc + my_k, rp);
        rp = 0;
        __syncthreads();
      }
      measured = true;
      uint32_t scratch_q = kNone;  // wide states: qubit of the last determined one
      const uint32_t mbeg = b, mend = min(wn, b + cnt);
      while (b < mend) {
        // Which of the next measurements have a pivot (a stabilizer row with
        // x_q set)?  Every wave finds out by itself.  A determined one's
        // outcome stays what it is while others are measured, so with the
        // columns in LDS those wait for the end of the run, to share the
        // waves.  Wide states: one measurement at a time, lane i keeping word i
        // of x_q.
        uint32_t nm, jr;
        uint64_t xqv = 0;
        if (kLds) {
          nm = min(mend - b, kWindow);
          uint64_t acc = 0;
          if (lane < nm) {
            const uint64_t *xq = P + __umul24(sh.ops[b + lane].qq, KW) + KH;
            for (uint32_t i = 0; i < KH; i += 4)
              acc |= xq[i] | xq[min(i + 1, KH - 1)] | xq[min(i + 2, KH - 1)] |
                     xq[min(i + 3, KH - 1)];
          }
          const uint64_t piv = __ballot(acc != 0);
          jr = piv ? (uint32_t)__ffsll((long long)piv) - 1 : nm;
        } else {
          nm = 1;
          xqv = lane < K2 ? P[sh.ops[b].qq * KW + lane] : 0ull;
          jr = (__ballot(xqv != 0) >> KH) ? 0u : 1u;
        }

        if (!kLds && jr) {
          // determined: as below, but the whole workgroup runs it, KH
          // lanes per column, so a column's words are one contiguous run
          const uint32_t q = rfl(sh.ops[b].qq), slot = rfl((uint32_t)msk[b * mstep]);
          const uint32_t cpw = 64 / KH, sub = lane / KH, kk = lane - sub * KH;
          const uint64_t below = ((1ull << kk) - 1) << (sub * KH);
          for (uint32_t g = 0; g < G; ++g) {
            uint64_t rx = 0;
            for (uint32_t i = tid; i < n; i += NT)
              if ((read_lane64(xqv, rfl(i >> 6)) >> lane) & 1) rx ^= Rv[g * R + n + i];
            if (__ballot(rx != 0)) {
              rx = wave_xor(rx);
              if (lane == 0) lds_xor(&sh.rx[slot2][g], rx);
            }
          }
          const uint64_t cm = __shfl(xqv, kk, 64);
          const uint64_t c = sub < cpw ? cm : 0ull;
          uint32_t tot = tid < KH ? 2u * (uint32_t)__popcll(c & rc[KH + kk]) : 0u;
          const uint32_t cstep = nw * cpw;
          for (uint32_t j0 = wv * cpw; j0 < n; j0 += kWideCols * cstep) {
            uint64_t xs[kWideCols], zs[kWideCols];
#pragma unroll
            for (uint32_t u = 0; u < kWideCols; ++u) {
              const uint32_t j = j0 + u * cstep + sub;
              const bool use = c != 0 && j < n;
              const uint64_t *xj = P + (use ? j * KW + KH + kk : 0u);
              xs[u] = use ? xj[0] & c : 0ull;
              zs[u] = use ? xj[n * KW] & c : 0ull;
            }
#pragma unroll
            for (uint32_t u = 0; u < kWideCols; ++u) {
              if (__ballot((xs[u] | zs[u]) != 0) == 0) continue;
              const uint64_t inc = prefix_parity(zs[u]);
              const uint64_t odd = __ballot(inc >> 63);
              const uint64_t carry = 0ull - (uint64_t)(__popcll(odd & below) & 1);
              tot += (uint32_t)__popcll(xs[u] & zs[u]) +
                     2u * (uint32_t)__popcll(xs[u] & ((inc << 1) ^ carry));
            }
          }
          // sum mod 4 over the wave: lanes' low bits and twos
          const uint32_t s = ((uint32_t)__popcll(__ballot(tot & 1u)) +
                              2u * (uint32_t)__popcll(__ballot((tot >> 1) & 1u))) & 3u;
          if (lane == 0 && s) atomicAdd(&sh.tot[slot2], s);
          // the other slot is free: it was read before this barrier
          if (tid == 0) {
            sh.tot[slot2 ^ 1] = 0;
            for (uint32_t g = 0; g < G; ++g) sh.rx[slot2 ^ 1][g] = 0;
          }
          __syncthreads();
          scratch_q = q;
          if (tid < G) {
            const uint32_t cst = (sh.tot[slot2] >> 1) & 1u;
            const uint64_t rxa = sh.rx[slot2][tid];
            if (!(sh.ops[b].cw & kOpDropped) && ((live >> tid) & 1)) {
              uint64_t *rec = a.recs + (2ull * slot) * W + w0 + tid;
              rec[0] = rxa ^ (0ull - (uint64_t)cst) ^ E[tid * 2 * n + q];
              rec[W] = ~0ull;
            }
            if (tid == 0) rc[K2] = cst;
            Rv[tid * R + 2 * n] = rxa;
          }
          slot2 ^= 1;
        }
        if (jr == nm) {
          b += nm;
          continue;
        }

        // measurement b + jr is random in every shot, with one pivot p for all
        // of them: rows with x_q set take the stabilizer row n+p, row p
        // becomes row n+p, and row n+p becomes Z_q with the coin as its sign
        {
          const uint32_t q = sh.ops[b + jr].qq;
          const uint64_t M0 = msk[(b + jr) * mstep], m = msk[(b + jr) * mstep + 1];
          if (kLds) xqv = lane < K2 ? P[__umul24(q, KW) + lane] : 0ull;
          const uint32_t kp = (uint32_t)__ffsll((long long)(__ballot(xqv != 0) >> KH)) - 1;
          const uint32_t bp = (uint32_t)__ffsll((long long)read_lane64(xqv, KH + kp)) - 1;
          const uint32_t p = 64 * kp + bp;
          const uint64_t bit = 1ull << bp;
          // group of this thread's Rv rows, and of this wave's coin
          const uint32_t rg = (NT - 1 - tid) & g_mask, cg = nw - 1 - wv;
          const uint64_t Rs = Rv[rg * R + n + p];
          const uint64_t Rc = cg < G ? Rv[cg * R + n + p] : 0ull;
          const uint64_t rck = rc[kp];
          const uint64_t rs = 0ull - ((rc[KH + kp] >> bp) & 1);
          if (lane == kp || lane == KH + kp) xqv &= ~bit;  // the rows to update
          // the sign bits: rows to update take row n+p's (and their phase's), row
          // p takes row n+p's, row n+p's is cleared
          uint64_t dr = xqv & rs;
          if (lane == kp) dr ^= (rs ^ rck) & bit;
          if (lane == KH + kp) dr ^= rs & bit;
          if (tid < K2) {
            sh.sm[tid] = xqv;
            sh.c0[tid] = 0;
          }
          if (tid == 0) {
            sh.ops[b + jr].cw |= kOpRandom;
            sh.nl = 0;
          }
          __syncthreads();
          if (tid < K2 && dr) lds_xor(rc + tid, dr);
          // rows p and n+p, a lane per column; columns where row n+p is not the
          // identity go on the list
          constexpr uint32_t kU = kLds ? 1 : 2;
          for (uint32_t v = wv; v < KH; v += kU * nw) {
            uint64_t wx[kU], wz[kU], dx[kU], dz[kU];
#pragma unroll
            for (uint32_t u = 0; u < kU; ++u) {
              const uint64_t *X = P + __umul24(min(64 * (v + u * nw) + lane, n - 1), KW) + kp;
              wx[u] = X[KH];
              wz[u] = X[n * KW + KH];
              dx[u] = X[0];
              dz[u] = X[n * KW];
            }
#pragma unroll
            for (uint32_t u = 0; u < kU; ++u) {
              const uint32_t j = 64 * (v + u * nw) + lane;
              uint32_t ent = 0;
              if (j < n) {
                uint64_t *X = P + __umul24(j, KW) + kp, *Z = X + n * KW;
                ent = (uint32_t)((wx[u] >> bp) & 1) | ((uint32_t)((wz[u] >> bp) & 1) << 1);
                X[0] = (dx[u] & ~bit) | (wx[u] & bit);
                Z[0] = (dz[u] & ~bit) | (wz[u] & bit);
                X[KH] = wx[u] & ~bit;
                Z[KH] = (wz[u] & ~bit) | (j == q ? bit : 0ull);
              }
              const uint64_t bal = __ballot(ent != 0);
              uint32_t at = 0;
              if (lane == 0 && bal) at = atomicAdd(&sh.nl, (uint32_t)__popcll(bal));
              at = rfl(at) + (uint32_t)__popcll(bal & ((1ull << lane) - 1));
              if (ent) list[at] = j | (ent << 16);
            }
          }
          // (from the last threads down: the columns start at thread 0)
          for (uint32_t u = NT - 1 - tid; u < (2 * n) << gs; u += NT) {
            const uint32_t i = u >> gs, ii = i < n ? i : i - n;
            const uint64_t mk = sh.sm[(i < n ? 0 : KH) + (ii >> 6)];
            if ((mk >> (ii & 63)) & 1) Rv[rg * R + i] ^= Rs;  // never rows p, n+p
          }
          if (cg < G) {
            const uint64_t w = min(w0 + cg, W - 1);
            uint64_t coin;
            if (a.coin_planes) {
              coin = a.coin_planes[m * W + w];
            } else {
              const uint64_t key = stream_key(seed, 2 * (mseq0 + m));
              coin = __ballot((uint32_t)(draw_keyed(key, 64 * w + lane) >> 40) <
                              (uint32_t)(M0 >> 32));
            }
            if (lane == 0) {
              Rv[cg * R + p] = Rc;
              Rv[cg * R + n + p] = coin ^ E[cg * 2 * n + q];
              if (!(sh.ops[b + jr].cw & kOpDropped) && ((live >> cg) & 1)) {
                uint64_t *rec = a.recs + (2ull * (uint32_t)M0) * W + w;
                rec[0] = coin;
                rec[W] = 0ull;
              }
            }
          }
          __syncthreads();
          // phases: per row, the sum mod 4 over columns of the phase exponent
          // of row * (row n+p): each thread's columns in registers, then
          // LDS atomics; the low bits' old value gives the carry, and the high
          // bits go into the signs
          uint64_t c0 = 0, c1 = 0;
          uint32_t ci = my_i;
          if (kLds) {
            const uint64_t mk = my_j < rpp ? sh.sm[my_i] : 0ull;
            const uint32_t nl = sh.nl;
            if (mk)
              for (uint32_t e = my_j; e < nl; e += rpp) {
                const uint32_t ent = list[e];
                uint64_t *X = P + (__umul24(ent & 0xFFFFu, KW) + my_i), *Z = X + n * KW;
                const uint64_t x = *X, z = *Z;
                const uint64_t fx = (ent >> 16) & 1 ? mk : 0ull, fz = ent >> 17 ? mk : 0ull;
                phase_acc(x, z, fx, fz, c0, c1);
                *X = x ^ fx;
                *Z = z ^ fz;
              }
          } else {
            // K2 lanes of one wave per listed column (a column's words are one
            // run), kRandCols columns a lane in flight.  One CU's VALU and its
            // path to the L2 are the bound: the columns where row n+p is the
            // identity, the row's bits by ballots, and the rows p and n+p are not
            // in this pass (n = 1024, 1409 of these in a run: 20 -> 9 us each).
            const uint32_t cpw = 64 / K2, sub = lane / K2, i = lane - sub * K2;
            const uint64_t mk = sub < cpw ? sh.sm[i] : 0ull;
            const uint32_t nl = sh.nl, cstep = nw * cpw;
            for (uint32_t e0 = wv * cpw; e0 < nl; e0 += kRandCols * cstep) {
              uint64_t x[kRandCols], z[kRandCols];
              uint32_t ent[kRandCols];
#pragma unroll
              for (uint32_t u = 0; u < kRandCols; ++u) {
                const uint32_t e = e0 + u * cstep + sub;
                ent[u] = e < nl ? list[e] : 0u;
                const uint64_t *X = P + (__umul24(ent[u] & 0xFFFFu, KW) + i);
                x[u] = X[0];
                z[u] = X[n * KW];
              }
#pragma unroll
              for (uint32_t u = 0; u < kRandCols; ++u) {
                const uint64_t fx = (ent[u] >> 16) & 1 ? mk : 0ull, fz = ent[u] >> 17 ? mk : 0ull;
                phase_acc(x[u], z[u], fx, fz, c0, c1);
                uint64_t *X = P + (__umul24(ent[u] & 0xFFFFu, KW) + i);
                if (fx) X[0] = x[u] ^ fx;
                if (fz) X[n * KW] = z[u] ^ fz;
              }
            }
            ci = i;
          }
          if (c0 | c1) {
            c1 ^= c0 & atomicXor(reinterpret_cast<unsigned long long *>(sh.c0 + ci),
                                 (unsigned long long)c0);
            if (c1) lds_xor(rc + ci, c1);
          }
          __syncthreads();
          b += jr + 1;
        }
      }
      // the run's determined measurements: the outcome is the sign of
      // the product, in ascending order, of the stabilizers whose
      // destabilizer has x_q set, which is Z_q up to that sign.  Writing a
      // Pauli row as i^y X^x Z^z (y the number of Y's), the product's
      // phase is i^(sum y) times -1 for every earlier z that meets a later x:
      // per column, a walk along the chain's rows, or where a word holds
      // several of them a prefix parity.  Rows without x bits (the Z checks of
      // a code) have no phase at all.
      if (kLds) {
        uint32_t last = mend;  // the last determined one
        while (last > mbeg && (rfl(sh.ops[last - 1].cw) & kOpRandom)) --last;
        --last;
        for (uint32_t idx = mbeg + wv; idx < mend; idx += nw) {
          const SharedOp J = sh.ops[idx];
          if (rfl(J.cw) & kOpRandom) continue;
          const uint32_t q = J.qq, slot = (uint32_t)msk[idx * mstep];
          // lane: group lane % G, and the (lane / G)-th slice of long chains
          const uint64_t *Rg = Rv + (lane & g_mask) * R + n;
          const uint64_t cv = lane < KH ? P[__umul24(q, KW) + lane] : 0ull;
          const uint64_t rv = lane < KH ? rc[KH + lane] : 0ull;
          const uint64_t nz = __ballot(cv != 0);
          const bool chain = __ballot((cv & (cv - 1)) != 0) != 0 || (nz & (nz - 1)) != 0;
          const uint32_t par = (uint32_t)__popcll(__ballot(__popcll(cv & rv) & 1));
          uint64_t rx = 0, ry = 0;
          uint32_t tot = 0, carry = 0;  // carry: bit u is column 64 u + lane's
          bool wide = false;
          uint64_t anyx = 0;
          for (uint64_t left = nz; left; left &= left - 1) {
            const uint32_t kk = (uint32_t)__ffsll((long long)left) - 1;
            const uint64_t c = read_lane64(cv, kk);
            const uint32_t cl = (uint32_t)__popcll(c);
            if (cl <= 4) {
              for (uint64_t r = c; r; r &= r - 1)
                rx ^= Rg[64 * kk + (uint32_t)__ffsll((long long)r) - 1];
            } else {
              wide = true;
              for (uint32_t i = lane >> gs; i < 64; i += 64 >> gs)
                if ((c >> i) & 1) ry ^= Rg[64 * kk + i];
            }
            if (chain)
              for (uint32_t j = lane; j < n; j += 64)
                anyx |= P[__umul24(j, KW) + KH + kk] & c;
          }
          if (__ballot(anyx != 0)) {
            for (uint64_t left = nz; left; left &= left - 1) {
              const uint32_t kk = (uint32_t)__ffsll((long long)left) - 1;
              const uint64_t c = read_lane64(cv, kk);
              const bool one = (c & (c - 1)) == 0;
              for (uint32_t u0 = 0; 64 * u0 < n; u0 += 3) {
                uint64_t xs[3], zs[3];
#pragma unroll
                for (uint32_t u = 0; u < 3; ++u) {
                  const uint32_t j = 64 * (u0 + u) + lane;
                  const uint64_t *xj = P + min(j, n - 1) * KW + KH + kk;
                  const uint64_t cm = j < n ? c : 0ull;
                  xs[u] = xj[0] & cm;
                  zs[u] = xj[n * KW] & cm;
                }
#pragma unroll
                for (uint32_t u = 0; u < 3; ++u) {
                  const uint32_t cb = (carry >> (u0 + u)) & 1u;
                  if (one) {
                    const uint32_t xb = xs[u] != 0, zb = zs[u] != 0;
                    tot += xb & zb;
                    tot += 2u * (xb & cb);
                    carry ^= zb << (u0 + u);
                  } else if (__ballot((xs[u] | zs[u]) != 0)) {
                    const uint64_t inc = prefix_parity(zs[u]);
                    tot += (uint32_t)__popcll(xs[u] & zs[u]) +
                           2u * (uint32_t)__popcll(xs[u] & ((inc << 1) ^ (0ull - (uint64_t)cb)));
                    carry ^= (uint32_t)(inc >> 63) << (u0 + u);
                  }
                }
              }
            }
          }
          if (wide) {
            for (uint32_t off = 32; off >= G; off >>= 1) ry ^= __shfl_xor(ry, off, 64);
            rx ^= ry;
          }
          const uint32_t cst = (par ^ wave_sum_bit1(tot)) & 1u;
          if (lane < G && ((live >> lane) & 1) && !(J.cw & kOpDropped)) {
            uint64_t *rec = a.recs + (2ull * slot) * W + w0 + lane;
            rec[0] = rx ^ (0ull - (uint64_t)cst) ^ E[lane * 2 * n + q];
            rec[W] = ~0ull;
          }
          if (idx == last) {  // the scratch row keeps the last product
            for (uint32_t j = lane; j < n; j += 64) {
              P[j * KW + K2] = 0;
              P[(n + j) * KW + K2] = j == q ? 1ull : 0ull;
            }
            if (lane == 0) rc[K2] = cst;
            if (lane < G) Rv[lane * R + 2 * n] = rx;
          }
        }
        __syncthreads();
      }
      if (!kLds && scratch_q != kNone) {  // the scratch row keeps the last product
        for (uint32_t j = tid; j < n; j += NT) {
          P[j * KW + K2] = 0;
          P[(n + j) * KW + K2] = j == scratch_q ? 1ull : 0ull;
        }
        __syncthreads();
      }
      b = mend;
      if (b < wn) cw = rfl(sh.ops[b].cw);
    }
    // every wave has read op b (which the window may end at, behind a
    // measurement): the next window's ops and masks take their place
    __syncthreads();
    base += b;
  }
  if (on && rp) lds_xor(rc + my_k, rp);
  __syncthreads();

  // ---- the 64-shot words ----
  // <E, P_i> of 64 rows at a time, row words times column shares over the
  // waves, gathered in Rv.
  auto add_signs = [&](uint32_t g, uint32_t kk, bool share0, uint64_t acc) {
    if (share0) acc ^= 0ull - ((rc[kk] >> lane) & 1);
    const uint32_t ii = 64 * (kk < KH ? kk : kk - KH) + lane;
    if (kk == K2) {
      if (lane == 0) lds_xor(Rv + g * R + 2 * n, acc);
    } else if (ii < n) {
      lds_xor(Rv + g * R + (kk < KH ? 0 : n) + ii, acc);
    }
  };
  {
    // A lane takes its row's bit of a column as a mask, once for all groups:
    // VALU-bound.  Column words and frames read from lanes as scalars instead
    // stalled on every one: 449 qubits, one group 106 -> 50 us of the run's 1180;
    // 161 qubits, four groups 56 -> 28 us of 337.  Two columns at a time: four
    // took the kernel from 128 to 159 VGPRs, at which no other kernel's wave fits
    // beside it on a CU (d=9, 16384 shots, several states in flight: 266 us a
    // pass with four, 200-240 with two, 255 with one).
    const uint32_t parts = max(1u, 2 * nw / KW), per = (n + parts - 1) / parts;
    for (uint32_t task = wv; task < KW * parts; task += nw) {
      const uint32_t kk = task / parts, pt = task - kk * parts;
      const uint32_t ja = pt * per, jb = min(n, ja + per);
      const int32_t *Px = reinterpret_cast<const int32_t *>(P + kk) + (lane >> 5);
      const int32_t *Pz = Px + 2 * n * KW;
      const uint32_t sh31 = 31 - (lane & 31);
      auto run = [&](auto groups) {
        constexpr uint32_t kG = decltype(groups)::value;
        uint64_t acc[kG] = {};
#pragma unroll 2
        for (uint32_t j = ja; j < jb; ++j) {
          const uint64_t mx = (uint64_t)(int64_t)((Px[2 * j * KW] << sh31) >> 31);
          const uint64_t mz = (uint64_t)(int64_t)((Pz[2 * j * KW] << sh31) >> 31);
#pragma unroll
          for (uint32_t g = 0; g < kG; ++g)
            acc[g] ^= (mx & E[g * 2 * n + n + j]) ^ (mz & E[g * 2 * n + j]);
        }
#pragma unroll
        for (uint32_t g = 0; g < kG; ++g) add_signs(g, kk, pt == 0, acc[g]);
      };
      if (gs == 0)
        run(std::integral_constant<uint32_t, 1>());
      else if (gs == 1)
        run(std::integral_constant<uint32_t, 2>());
      else
        run(std::integral_constant<uint32_t, 4>());
    }
  }
  __syncthreads();
  for (uint32_t g = 0; g < G; ++g)
    if ((live >> g) & 1)
      for (uint32_t i = tid; i < R; i += NT) T0[g * blk + 2ull * n * R + i] = Rv[g * R + i];
  if (a.packed) {
    // one workgroup leaves the columns for k_shared_expand: the first that
    // holds a group that ran
    bool later = false;
    if (a.shared == kSharedChecked)
      for (uint64_t i = tid; i < w0; i += NT) later |= a.done[i] != 0;
    else
      later = w0 != 0;
    if (!__syncthreads_or(later))
      for (uint32_t i = tid; i < 2 * n * KW; i += NT) a.packed[i] = P[i];
    return live;
  }
  __syncthreads();
  // Columns in the tableau: the packed block covers the first KW tableau
  // columns of its group; those are written last, from a copy.
  const uint32_t c0 = kLds ? 0 : KW;
  if (!kLds) {
    for (uint32_t i = tid; i < c0 * KW; i += NT) dyn[i] = P[i];
    __syncthreads();
  }
  // a wave per column
  auto expand = [&](uint64_t *T, uint32_t c, const uint64_t *src) {
    const uint64_t v0 = lane < KW ? src[lane] : 0ull;
    const uint64_t v1 = lane + 64 < KW ? src[lane + 64] : 0ull;
    uint64_t *dst = T + (uint64_t)c * R;
    for (uint32_t kk = 0; kk < K2; ++kk) {
      const uint64_t s = kk < 64 ? read_lane64(v0, kk) : read_lane64(v1, kk - 64);
      const uint32_t ii = 64 * (kk < KH ? kk : kk - KH) + lane;
      if (ii < n)
        dst[(kk < KH ? 0 : n) + ii] = __builtin_amdgcn_inverse_ballot_w64(s) ? ~0ull : 0ull;
    }
    const uint64_t s = K2 < 64 ? read_lane64(v0, K2) : read_lane64(v1, K2 - 64);
    if (lane == 0) dst[2 * n] = 0ull - (s & 1);
  };
  for (uint32_t g = G; g-- > 0;) {  // the group whose block holds the columns last
    if (!((live >> g) & 1)) continue;
    uint64_t *T = T0 + g * blk;
    for (uint32_t c = c0 + wv; c < 2 * n; c += nw) expand(T, c, P + c * KW);
    if (!kLds) {
      __syncthreads();
      for (uint32_t c = wv; c < c0; c += nw) expand(T, c, dyn + c * KW);
    }
  }
  __syncthreads();
  return live;
}

// One workgroup per G = 1 << a.gshift word groups.  With a.done, groups that
// ran are marked there and the per-shot kernel launched behind this one passes
// over them.
template <bool kLds>
__global__ __launch_bounds__(kSharedThreads) void k_program_shared(
    ProgramArgs a, const ProgParams *__restrict__ pp) {
  extern __shared__ uint64_t dyn[];
  __shared__ SharedLds sh;
  const uint64_t seed = pp->seed, mseq0 = pp->mseq0;
  for (uint64_t i = blockIdx.x; i << a.gshift < a.W; i += gridDim.x) {
    shared_words<kLds>(a, seed, mseq0, i << a.gshift, a.gshift, dyn, sh);
    __syncthreads();
  }
}

// done[w] = whether group w's X/Z are the |0...0> tableau; done starts at 1.
// One block per group and share of its words.
__global__ __launch_bounds__(256) void k_shared_verify(const uint64_t *__restrict__ tab,
                                                       uint32_t n, uint32_t R, uint64_t blk,
                                                       uint64_t W, uint32_t *done) {
  const uint32_t total = 2 * n * R, M = R + 1;
  const uint32_t NT = 256 * gridDim.x, first = blockIdx.x * 256 + threadIdx.x, step = NT % M;
  for (uint64_t w = blockIdx.y; w < W; w += gridDim.y) {
    const uint64_t *T = tab + w * blk;
    uint32_t rem = first % M;
    bool bad = false;
    for (uint32_t base = first; base < total && !bad; base += 8 * NT) {
      uint64_t v[8];
#pragma unroll
      for (uint32_t u = 0; u < 8; ++u) v[u] = T[min(base + u * NT, total - 1)];
#pragma unroll
      for (uint32_t u = 0; u < 8; ++u) {
        bad |= base + u * NT < total && v[u] != (rem == 0 ? ~0ull : 0ull);
        rem += step;
        if (rem >= M) rem -= M;
      }
    }
    if (bad) done[w] = 0;
  }
}

__global__ void k_fill_u32(uint32_t *p, uint64_t n, uint32_t v) {
  for (uint64_t i = blockIdx.x * (uint64_t)blockDim.x + threadIdx.x; i < n;
       i += (uint64_t)gridDim.x * blockDim.x)
    p[i] = v;
}

// The packed columns as 64-shot words in every word group (done: those that
// ran).  A block per 256 rows of a column and share of the groups: the word is
// the same in every group, so it is made once.
__global__ __launch_bounds__(256) void k_shared_expand(uint64_t *__restrict__ tab,
                                                       const uint64_t *__restrict__ packed,
                                                       uint32_t n, uint32_t R, uint64_t blk,
                                                       uint64_t W,
                                                       const uint32_t *__restrict__ done) {
  const uint32_t row = blockIdx.x * 256 + threadIdx.x, c = blockIdx.y;
  if (row >= R) return;
  const uint32_t KH = (n + 63) / 64, KW = 2 * KH + 1;
  const uint32_t i = row < n ? row : row - n;
  const uint32_t k = row < n ? i >> 6 : row < 2 * n ? KH + (i >> 6) : 2 * KH;
  const uint32_t bit = row < 2 * n ? i & 63 : 0;
  const uint64_t v = 0ull - ((packed[c * KW + k] >> bit) & 1);
  for (uint64_t w = blockIdx.z; w < W; w += gridDim.z)
    if (!done || done[w]) tab[w * blk + (uint64_t)c * R + row] = v;
}

// The members of a mixed batch that may run packed: work items (circuit << 40 |
// word group), taken from counter[1] (columns in LDS) or counter[3] (in the
// tableau); counter[2] counts the word groups that ran.  k_batch_t runs what is
// left.
template <bool kLds>
__global__ __launch_bounds__(kSharedThreads) void k_batch_shared(
    const BatchCircuit *__restrict__ circ, const uint64_t *__restrict__ items, uint64_t nitems,
    unsigned long long *counter, uint32_t wtile) {
  extern __shared__ uint64_t dyn[];
  __shared__ SharedLds sh;
  for (;;) {
    if (threadIdx.x == 0) sh.item = atomicAdd(counter + (kLds ? 1 : 3), 1ull);
    __syncthreads();
    const uint64_t it = rfl64(sh.item);
    __syncthreads();
    if (it >= nitems) break;
    const uint64_t code = rfl64(items[it]);
    const BatchCircuit &bc = circ[(uint32_t)(code >> 40)];
    if (!bc.a.shared || packed_in_lds(bc.a.n, bc.a.masked) != kLds) continue;
    const uint64_t w = code & ((1ull << 40) - 1);
    const uint64_t wend = min(w + wtile, bc.a.nwords);
    const uint32_t gs = rfl(bc.a.gshift);
    for (uint64_t wi = w; wi < wend; ++wi) {
      if (wi & ((1u << gs) - 1)) continue;  // the item of its first group runs it
      const uint32_t ran = shared_words<kLds>(bc.a, bc.seed, bc.mseq0, wi, gs, dyn, sh);
      if (threadIdx.x == 0 && ran) atomicAdd(counter + 2, (unsigned long long)__popc(ran));
      __syncthreads();
    }
  }
}

}  // namespace

bool shared_fits(uint32_t n) { return n >= 1 && n <= kSharedMaxQubits; }

bool shared_wide(uint32_t n, bool masked) { return !packed_in_lds(n, masked); }

static size_t lds_bytes(uint32_t n, bool masked, uint32_t gshift) {
  // the packed columns, or the list of a random measurement's columns
  return 8 * (groups_words(n, masked, gshift) +
              (packed_in_lds(n, masked) ? packed_words(n) : (n + 1) / 2));
}

size_t shared_lds_bytes(uint32_t n, bool masked, uint32_t gshift) {
  return lds_bytes(n, masked, gshift);
}

// Word groups per workgroup of a batch's member, `groups` of all members on
// `cus` compute units: more of them while a workgroup per unit is left (256
// surface-code circuits, d = 3..25, 3718 groups: 686 -> 358 ms).
uint32_t shared_batch_gshift(uint32_t n, uint64_t W, bool masked, uint64_t groups, uint32_t cus) {
  uint32_t gs = 0;
  while ((2u << gs) <= kSharedMaxGroups && (W >> (gs + 1)) && (groups >> (gs + 1)) >= cus &&
         lds_bytes(n, masked, gs + 1) <= kSharedLdsBytes)
    ++gs;
  return gs;
}

// Word groups per workgroup.  Groups that share a workgroup share the packed
// X/Z work; more workgroups finish sooner on an empty GPU.  Columns in LDS: at
// least 64 workgroups, so that four states' run side by side on 256 compute units
// (d=9, 16384 shots, us for 1, 2, 3, 6 and 12 states in flight: 421, 542, 648, 1285,
// 2552 with 64 workgroups of four groups; 377, 500, 797, 1465, 2643 with 128 of
// two; 64 random qubits, 8192 shots: 375, 384, 391, 756, 1493; 367, 376, 717, 1078,
// 2135; with 32 workgroups one state of 8192 shots takes 383 instead of 337).
// Columns in the tableau, whose work is the L2's: as many groups as fit (n=1024,
// 4096 shots, 1 and 2 states: 3766, 4415 us; one group per workgroup 4120, 6160).
// Up to 16 groups in all one per workgroup would be the faster (n=1024, 1024 shots:
// 3267 against 2892 us).
uint32_t shared_gshift(uint32_t n, uint64_t W, bool masked) {
  uint32_t gs = 0;
  const uint64_t least = packed_in_lds(n, masked) ? 64 : 1;
  while ((2u << gs) <= kSharedMaxGroups && (W >> (gs + 1)) >= least &&
         lds_bytes(n, masked, gs + 1) <= kSharedLdsBytes)
    ++gs;
  return gs;
}

// Whether the tableau check and the 64-shot words are launches of their own,
// over the whole GPU: for a small state the two launches cost more than they
// save.  What they save grows with the tableau words a workgroup would write:
// at 33 MB, alone, checked: 64 qubits 236 us with, 249 without; 161 qubits 377,
// 393; 300 qubits 378, 475; below, at 8 MB: 64 qubits 217, 205 (four states in
// flight 488, 405), 161 qubits 362, 384 (780, 768), 300 qubits 362, 462.
bool shared_split(uint32_t n, uint64_t W, bool masked) {
  return !packed_in_lds(n, masked) || W * (2ull * n + 1) * (2ull * n + 1) * 8 >= (32ull << 20);
}

uint64_t shared_packed_bytes(uint32_t n) { return 8 * packed_words(n); }

hipError_t prepare_shared() {
  hipError_t e = hipSuccess;
  for (const void *fn : {(const void *)k_program_shared<true>, (const void *)k_program_shared<false>,
                         (const void *)k_batch_shared<true>, (const void *)k_batch_shared<false>})
    if (e == hipSuccess)
      e = hipFuncSetAttribute(fn, hipFuncAttributeMaxDynamicSharedMemorySize,
                              (int)kSharedLdsBytes);
  return e;
}

hipError_t launch_batch_shared(hipStream_t s, const BatchCircuit *circ, const uint64_t *items,
                               uint64_t nitems, unsigned long long *counter, uint32_t cus,
                               size_t lds_packed, size_t lds_wide, uint32_t wtile) {
  wtile = std::max<uint32_t>(wtile, 1);
  // as many workgroups per CU as the largest member's LDS allows
  auto blocks = [&](size_t lds) {
    const uint64_t per_cu = std::max<uint64_t>(1, 160 * 1024 / (lds + sizeof(SharedLds)));
    return dim3((uint32_t)std::min<uint64_t>(nitems, cus * std::min<uint64_t>(4, per_cu)));
  };
  if (nitems && lds_packed)
    hipLaunchKernelGGL(k_batch_shared<true>, blocks(lds_packed), dim3(kSharedThreads), lds_packed,
                       s, circ, items, nitems, counter, wtile);
  if (nitems && lds_wide)
    hipLaunchKernelGGL(k_batch_shared<false>, blocks(lds_wide), dim3(kSharedThreads), lds_wide, s,
                       circ, items, nitems, counter, wtile);
  return hipGetLastError();
}

hipError_t launch_shared(hipStream_t s, const ProgramArgs &args, const void *params) {
  ProgramArgs a = args;
  if (!a.W) return hipSuccess;
  const uint64_t blk = (uint64_t)a.C * a.R;
  if (a.packed && a.shared == kSharedVerify) {
    a.shared = kSharedChecked;
    hipLaunchKernelGGL(k_fill_u32, dim3((uint32_t)std::min<uint64_t>((a.W + 255) / 256, 256)),
                       dim3(256), 0, s, a.done, a.W, 1u);
    const uint64_t parts = std::max<uint64_t>(1, std::min<uint64_t>(2048 / a.W + 1,
                                                                    (2ull * a.n * a.R) >> 13));
    hipLaunchKernelGGL(k_shared_verify,
                       dim3((uint32_t)parts, (uint32_t)std::min<uint64_t>(a.W, 65535)), dim3(256),
                       0, s, a.tab, a.n, a.R, blk, a.W, a.done);
  }
  a.gshift = shared_gshift(a.n, a.W, a.masked);
  const size_t lds = lds_bytes(a.n, a.masked, a.gshift);
  const uint64_t wgs = (a.W + (1u << a.gshift) - 1) >> a.gshift;
  const dim3 grid((uint32_t)std::min<uint64_t>(wgs, 1u << 20));
  const uint32_t threads = kSharedThreads;
  if (packed_in_lds(a.n, a.masked))
    hipLaunchKernelGGL(k_program_shared<true>, grid, dim3(threads), lds, s, a,
                       (const ProgParams *)params);
  else
    hipLaunchKernelGGL(k_program_shared<false>, grid, dim3(threads), lds, s, a,
                       (const ProgParams *)params);
  if (a.packed) {
    // about 65536 blocks, each writing its rows in several word groups
    const uint64_t blocks = (uint64_t)((a.R + 255) / 256) * 2 * a.n;
    const uint64_t z = std::max<uint64_t>(1, std::min<uint64_t>(a.W, (65536 + blocks - 1) / blocks));
    hipLaunchKernelGGL(k_shared_expand,
                       dim3((a.R + 255) / 256, 2 * a.n, (uint32_t)std::min<uint64_t>(z, 64)),
                       dim3(256), 0, s, a.tab, a.packed, a.n, a.R, blk, a.W,
                       a.shared == kSharedChecked ? a.done : nullptr);
  }
  return hipGetLastError();
}

}  // namespace pq
