// Shared-X/Z persistent kernels (gfx950).
//
// H, S, CX, CZ and measurements change X and Z in every shot alike, so a
// program without flagged H/S/CX/CZ that starts from |0...0> keeps the X/Z
// words of a 64-shot group all zeros or all ones throughout: one bit instead
// of 64 per entry.  The kernels here run a whole compiled program on that
// packed tableau, in one workgroup per word group, and write the group's 64-shot
// words once at the end.  Per word group they keep
//  * X and Z as bits, one column of KW = 2 KH + 1 words per x_q and z_q
//    (KH = ceil(n/64)): KH words of destabilizer rows, KH words of stabilizer
//    rows, so rows i and n+i share a bit position, and one word whose bit 0
//    is the scratch row;
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
// of rows.  n <= about 460: the packed columns (2n (2 n/64 + 1) words) sit in
// LDS; up to 2048 qubits they sit at the start of their own column of the
// group's tableau block, which the run overwrites anyway (L2-resident).
#include "pq_kernels.h"

#include <algorithm>

#include "plaquette_amd.h"

namespace pq {

namespace {

#define PQ_CONST __attribute__((address_space(4)))

constexpr uint32_t kChunk = 448;       // staged ops; must equal kStage in pq_kernels.hip
constexpr uint32_t kChunkWords = kChunk * 5;
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

struct SharedLds {
  uint32_t bad;     // a word of the state is not the |0...0> tableau's
  uint32_t tot;     // determined measurement (wide states): phase count
  uint64_t piv;     // pivot check: measurements of the window with a pivot
  uint64_t rx;      // determined measurement (wide states): XOR of Rv rows
  uint64_t item;
};

// LDS words besides the packed columns: Rv, E, four KW-word row masks, the
// staged ops.
__host__ __device__ inline uint64_t shared_base_words(uint32_t n) {
  const uint64_t KW = 2ull * ((n + 63) / 64) + 1;
  return (2ull * n + 1) + 2ull * n + 4 * KW + kChunkWords;
}
__host__ __device__ inline uint64_t shared_packed_words(uint32_t n) {
  return 2ull * n * (2ull * ((n + 63) / 64) + 1);
}

__host__ __device__ inline bool packed_in_lds(uint32_t n) {
  return (shared_base_words(n) + shared_packed_words(n)) * 8 <= kSharedLdsBytes;
}

// One staged gate-segment op: `cw` = code (bits 0-7), has noise or a flag
// (bit 8), ops of the layer part it opens inside the chunk (bits 10-20);
// `qq` = qa | qb << 16.
struct SharedOp {
  uint32_t cw, qq;
};

// Runs the program on word group w.  Returns false, with the state untouched,
// if a.shared asks to verify that the group's X/Z are the |0...0> tableau and
// they are not.
template <bool kLds>
__device__ bool shared_word(const ProgramArgs &a, uint64_t seed, uint64_t mseq0, uint64_t w,
                            uint64_t *dyn, SharedLds &sh) {
  const uint32_t tid = threadIdx.x, NT = blockDim.x, lane = lane_id();
  const uint32_t wv = rfl(tid >> 6), nw = NT >> 6;
  const uint32_t n = a.n, R = a.R;
  const uint32_t KH = (n + 63) / 64, KW = 2 * KH + 1;
  const uint64_t W = a.W;
  uint64_t *T = a.tab + w * (uint64_t)a.C * R;
  uint64_t *Tr = T + 2ull * n * R;  // the R column
  uint64_t *Rv = dyn;
  uint64_t *E = Rv + R;             // E.x[0..n), E.z[n..2n)
  uint64_t *rc = E + 2 * n;         // sign bits, laid out like a column
  uint64_t *sm = rc + KW;           // row mask of the current measurement
  uint64_t *s_c0 = sm + KW, *s_c1 = s_c0 + KW;
  uint64_t *s_msk = s_c1 + KW;
  SharedOp *s_ops = reinterpret_cast<SharedOp *>(s_msk + 4 * kChunk);
  // packed column c (x_c, or z_{c-n}) starts at P + c * stride
  uint64_t *P = kLds ? s_msk + kChunkWords : T;
  const uint32_t stride = kLds ? KW : R;
  const PQ_CONST DInstr *ins = (const PQ_CONST DInstr *)a.instrs;
  const PQ_CONST DSegment *segs = (const PQ_CONST DSegment *)a.segs;
  const PQ_CONST uint64_t *gp = (const PQ_CONST uint64_t *)a.planes + 2ull * a.nk * w;

  if (a.shared == kSharedVerify) {
    // word t of the X/Z block is all ones iff t is a multiple of R + 1
    if (tid == 0) sh.bad = 0;
    __syncthreads();
    const uint32_t total = 2 * n * R, M = R + 1, step = NT % M;
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
      if (bad) sh.bad = 1;
      if (__ballot(bad) || *(volatile uint32_t *)&sh.bad) break;
    }
    __syncthreads();
    if (sh.bad) return false;
  }

  // ---- |0...0>: destabilizer i = X_i, stabilizer i = Z_i ----
  for (uint32_t u = tid; u < 2 * n * KW; u += NT) {
    const uint32_t c = u / KW, k = u - c * KW;
    const uint32_t q = c < n ? c : c - n;
    const uint32_t kq = (c < n ? 0 : KH) + (q >> 6);
    P[c * stride + k] = k == kq ? 1ull << (q & 63) : 0ull;
  }
  for (uint32_t i = tid; i < R; i += NT) Rv[i] = Tr[i];
  for (uint32_t i = tid; i < 2 * n; i += NT) E[i] = 0;
  if (tid < KW) rc[tid] = 0;
  __syncthreads();

  // this thread's share of a layer's column work: word my_k of every opp-th op
  const uint32_t opp = NT / KW;
  const uint32_t my_op = tid / KW, my_k = tid - my_op * KW;
  const bool on = my_op < opp;

  for (uint32_t si = 0; si < a.nseg; ++si) {
    const uint32_t kind = segs[si].kind, sbegin = segs[si].begin, scount = segs[si].count;
    const uint32_t send = sbegin + scount;
    if (kind == 0) {
      uint64_t rp = 0;  // sign flips of row word my_k
      for (uint32_t cb = sbegin; cb < send; cb += kChunk) {
        const uint32_t cn = min(kChunk, send - cb);
        for (uint32_t t = tid; t < cn; t += NT) {
          const PQ_CONST DInstr *I = ins + cb + t;
          const uint32_t code = I->code, na = I->na, nb = I->nb, slot = I->slot, pad = I->pad;
          uint64_t m0 = 0, m1 = 0, m2 = 0, m3 = 0;
          if (na != kNone) {
            m0 = gp[2ull * na];
            m1 = gp[2ull * na + 1];
          }
          if (nb != kNone) {
            m2 = gp[2ull * nb];
            m3 = gp[2ull * nb + 1];
          } else if (code >= PQ_OP_H_FLAG && code != PQ_OP_NOISE) {
            m2 = (slot & kSlotPlane) ? gp[2ull * (slot & ~kSlotPlane)]
                                     : a.recs[(2ull * slot) * W + w];
          }
          SharedOp J;
          J.cw = code | ((m0 | m1 | m2 | m3) ? 1u << 8 : 0u) |
                 (((pad >> kLayerLenShift) & kLayerLenMask) << 10);
          J.qq = I->qa | (I->qb << 16);
          s_ops[t] = J;
          s_msk[4 * t + 0] = m0;
          s_msk[4 * t + 1] = m1;
          s_msk[4 * t + 2] = m2;
          s_msk[4 * t + 3] = m3;
        }
        __syncthreads();
        uint32_t b = 0;
        while (b < cn) {
          // a layer's ops act on distinct qubits: no barrier inside it
          const uint32_t cnt = max(1u, (rfl(s_ops[b].cw) >> 10) & kLayerLenMask);
          if (on) {
            for (uint32_t o = my_op; o < cnt; o += opp) {
              const SharedOp J = s_ops[b + o];
              const uint32_t code = J.cw & 0xFFu, qa = J.qq & 0xFFFFu, qb = J.qq >> 16;
              uint64_t *xa = P + (qa * stride + my_k), *za = xa + n * stride;
              if (code == PQ_OP_CX) {
                uint64_t *xb = P + (qb * stride + my_k), *zb = xb + n * stride;
                const uint64_t x = *xa, z = *za, xt = *xb, zt = *zb;
                rp ^= x & zt & ~(xt ^ z);
                *xb = xt ^ x;
                *za = z ^ zt;
              } else if (code == PQ_OP_H) {
                const uint64_t x = *xa, z = *za;
                rp ^= x & z;
                *xa = z;
                *za = x;
              } else if (code == PQ_OP_S) {
                const uint64_t x = *xa, z = *za;
                rp ^= x & z;
                *za = z ^ x;
              } else if (code == PQ_OP_CZ) {
                uint64_t *xb = P + (qb * stride + my_k), *zb = xb + n * stride;
                const uint64_t x = *xa, z = *za, xt = *xb, zt = *zb;
                rp ^= x & xt & (zt ^ z);
                *zb = zt ^ x;
                *za = z ^ xt;
              }
            }
          }
          // the frame words, from the last threads down (the column work
          // starts at thread 0)
          for (uint32_t o = NT - 1 - tid; o < cnt; o += NT) {
            const SharedOp J = s_ops[b + o];
            const uint32_t code = J.cw & 0xFFu, qa = J.qq & 0xFFFFu, qb = J.qq >> 16;
            const uint64_t *M = s_msk + 4 * (b + o);
            uint64_t ex = E[qa], ez = E[n + qa];
            const bool noisy = (J.cw >> 8) & 1u;
            switch (code) {
              case PQ_OP_H: {
                const uint64_t t = ex;
                ex = ez;
                ez = t;
                break;
              }
              case PQ_OP_S: ez ^= ex; break;
              case PQ_OP_X: ex = ~ex; break;
              case PQ_OP_Y: ex = ~ex; ez = ~ez; break;
              case PQ_OP_Z: ez = ~ez; break;
              case PQ_OP_CX:
              case PQ_OP_CZ: {
                uint64_t fx = E[qb], fz = E[n + qb];
                if (code == PQ_OP_CX) {
                  fx ^= ex;
                  ez ^= fz;
                } else {
                  fz ^= ex;
                  ez ^= fx;
                }
                if (noisy) {
                  fx ^= M[2];
                  fz ^= M[3];
                }
                E[qb] = fx;
                E[n + qb] = fz;
                break;
              }
              case PQ_OP_X_FLAG: ex ^= M[2]; break;
              case PQ_OP_Y_FLAG: ex ^= M[2]; ez ^= M[2]; break;
              case PQ_OP_Z_FLAG: ez ^= M[2]; break;
              default: break;  // PQ_OP_NOISE: the masks below
            }
            if (noisy) {
              ex ^= M[0];
              ez ^= M[1];
            }
            E[qa] = ex;
            E[n + qa] = ez;
          }
          b += cnt;
          __syncthreads();
        }
      }
      if (on && rp) lds_xor(rc + my_k, rp);
      __syncthreads();
      continue;
    }

    // ---- measurements ----
    for (uint32_t mb = sbegin; mb < send; mb += kChunk) {
      const uint32_t mn = min(kChunk, send - mb);
      // staged: qubit | record << 32, coin threshold | pad << 32, sequence number
      for (uint32_t t = tid; t < mn; t += NT) {
        const PQ_CONST DInstr *I = ins + mb + t;
        s_msk[4 * t + 0] = (uint64_t)I->qa | ((uint64_t)I->slot << 32);
        s_msk[4 * t + 1] = (uint64_t)I->t0 | ((uint64_t)I->pad << 32);
        s_msk[4 * t + 2] = (uint64_t)I->na | ((uint64_t)I->nb << 32);
      }
      if (!kLds && tid == 0) sh.piv = 0;
      __syncthreads();
      uint32_t k = 0;
      while (k < mn) {
        // which of the next measurements have a pivot (a stabilizer row
        // with x_q set)?
        uint32_t nm = min(mn - k, kWindow);
        uint64_t piv;
        if (kLds) {
          uint64_t acc = 0;
          if (lane < nm) {
            const uint64_t *xq = P + (uint32_t)s_msk[4 * (k + lane)] * stride + KH;
            for (uint32_t i = 0; i < KH; ++i) acc |= xq[i];
          }
          piv = __ballot(acc != 0);
        } else {
          nm = min(nm, NT / KH);
          const uint32_t i = tid / KH, kk = tid - i * KH;
          if (i < nm && P[(uint32_t)s_msk[4 * (k + i)] * stride + KH + kk])
            atomicOr(reinterpret_cast<unsigned long long *>(&sh.piv), 1ull << i);
          __syncthreads();
          piv = rfl64(sh.piv);
          __syncthreads();
          if (tid == 0) sh.piv = 0;
        }
        const uint32_t jr = piv ? (uint32_t)__ffsll((long long)piv) - 1 : nm;

        // measurements [k, k + jr) are determined: the outcome is the sign of
        // the product, in ascending order, of the stabilizers whose
        // destabilizer has x_q set, which is Z_q up to that sign.  Writing a
        // Pauli row as i^y X^x Z^z (y the number of Y's), the product's
        // phase is i^(sum y) times -1 for every earlier z that meets a later x:
        // per column, a prefix parity over the chain's rows.
        if (kLds) {
          for (uint32_t idx = wv; idx < jr; idx += nw) {
            const uint64_t *M = s_msk + 4 * (k + idx);
            const uint32_t q = rfl((uint32_t)M[0]), slot = rfl((uint32_t)(M[0] >> 32));
            const uint64_t *cq = P + q * stride;
            uint32_t len = 0, par = 0;
            uint64_t rx = 0;
            for (uint32_t kk = 0; kk < KH; ++kk) len += (uint32_t)__popcll(cq[kk]);
            len = rfl(len);
            for (uint32_t kk = 0; kk < KH; ++kk) {
              uint64_t c = rfl64(cq[kk]);
              par ^= (uint32_t)__popcll(c & rc[KH + kk]);
              if (len <= 8) {
                while (c) {
                  const uint32_t i = (uint32_t)__ffsll((long long)c) - 1;
                  c &= c - 1;
                  rx ^= Rv[n + 64 * kk + i];
                }
              } else if ((c >> lane) & 1) {
                rx ^= Rv[n + 64 * kk + lane];
              }
            }
            if (len > 8) rx = wave_xor(rx);
            uint32_t ph = 0;
            if (len > 1) {
              uint32_t tot = 0;
              for (uint32_t j0 = 0; j0 < n; j0 += 64) {
                const uint32_t j = min(j0 + lane, n - 1);
                const uint64_t *xj = P + j * stride + KH, *zj = xj + n * stride;
                uint64_t carry = 0;
                uint32_t t = 0;
                for (uint32_t kk = 0; kk < KH; ++kk) {
                  const uint64_t c = rfl64(cq[kk]);
                  if (!c) continue;
                  const uint64_t xs = xj[kk] & c, zs = zj[kk] & c;
                  if (__ballot((xs | zs) != 0) == 0) continue;
                  const uint64_t inc = prefix_parity(zs);
                  t += (uint32_t)__popcll(xs & zs) +
                       2u * (uint32_t)__popcll(xs & ((inc << 1) ^ carry));
                  carry ^= 0ull - (inc >> 63);
                }
                if (j0 + lane < n) tot += t;
              }
              ph = wave_sum_bit1(tot);
            }
            const uint32_t cst = (par ^ ph) & 1u;
            if (lane == 0) {
              if (!((M[1] >> 32) & kMeasSuperseded)) {
                a.recs[(2ull * slot) * W + w] = rx ^ (0ull - (uint64_t)cst) ^ E[q];
                a.recs[(2ull * slot + 1) * W + w] = ~0ull;
              }
            }
            if (idx == jr - 1) {  // the scratch row keeps the last product
              for (uint32_t j = lane; j < n; j += 64) {
                P[j * stride + 2 * KH] = 0;
                P[(n + j) * stride + 2 * KH] = j == q ? 1ull : 0ull;
              }
              if (lane == 0) {
                rc[2 * KH] = cst;
                Rv[2 * n] = rx;
              }
            }
          }
        } else {
          // columns in global memory: the whole workgroup runs each, KH
          // lanes per column, so a column's words are one contiguous run
          const uint32_t cpw = 64 / KH, sub = lane / KH, kk = lane - sub * KH;
          const uint64_t below = ((1ull << kk) - 1) << (sub * KH);
          for (uint32_t idx = 0; idx < jr; ++idx) {
            const uint64_t *M = s_msk + 4 * (k + idx);
            const uint32_t q = rfl((uint32_t)M[0]), slot = rfl((uint32_t)(M[0] >> 32));
            if (tid < KH) sm[tid] = P[q * stride + tid];
            if (tid == 0) {
              sh.tot = 0;
              sh.rx = 0;
            }
            __syncthreads();
            uint64_t rx = 0;
            for (uint32_t i = tid; i < n; i += NT)
              if ((sm[i >> 6] >> (i & 63)) & 1) rx ^= Rv[n + i];
            if (__ballot(rx != 0)) {
              rx = wave_xor(rx);
              if (lane == 0) lds_xor(&sh.rx, rx);
            }
            uint32_t tot = 0;
            const uint64_t c = sub < cpw ? sm[kk] : 0ull;
            if (tid < KH) tot = 2u * (uint32_t)__popcll(c & rc[KH + kk]);
            const uint32_t cstep = nw * cpw;
            for (uint32_t j0 = wv * cpw; j0 < n; j0 += 4 * cstep) {
              uint64_t xs[4], zs[4];
#pragma unroll
              for (uint32_t u = 0; u < 4; ++u) {
                const uint32_t j = j0 + u * cstep + sub;
                const bool use = c != 0 && j < n;
                const uint64_t *xj = P + (use ? j * stride + KH + kk : 0u);
                xs[u] = use ? xj[0] & c : 0ull;
                zs[u] = use ? xj[n * stride] & c : 0ull;
              }
#pragma unroll
              for (uint32_t u = 0; u < 4; ++u) {
                const uint64_t inc = prefix_parity(zs[u]);
                const uint64_t odd = __ballot(inc >> 63);
                const uint64_t carry = 0ull - (uint64_t)(__popcll(odd & below) & 1);
                tot += (uint32_t)__popcll(xs[u] & zs[u]) +
                       2u * (uint32_t)__popcll(xs[u] & ((inc << 1) ^ carry));
              }
            }
            // sum mod 4 over the wave: lanes' low bits and twos
            {
              const uint32_t s = (uint32_t)__popcll(__ballot(tot & 1u)) +
                                 2u * (uint32_t)__popcll(__ballot((tot >> 1) & 1u));
              if (lane == 0 && (s & 3u)) atomicAdd(&sh.tot, s & 3u);
            }
            __syncthreads();
            const uint32_t cst = (sh.tot >> 1) & 1u;
            if (idx == jr - 1) {
              for (uint32_t j = tid; j < n; j += NT) {
                P[j * stride + 2 * KH] = 0;
                P[(n + j) * stride + 2 * KH] = j == q ? 1ull : 0ull;
              }
            }
            if (tid == 0) {
              const uint64_t rxa = sh.rx;
              if (!((M[1] >> 32) & kMeasSuperseded)) {
                a.recs[(2ull * slot) * W + w] = rxa ^ (0ull - (uint64_t)cst) ^ E[q];
                a.recs[(2ull * slot + 1) * W + w] = ~0ull;
              }
              rc[2 * KH] = cst;
              Rv[2 * n] = rxa;
            }
            __syncthreads();
          }
        }
        if (jr == nm) {
          k += nm;
          __syncthreads();
          continue;
        }

        // measurement k + jr is random in every shot, with one pivot p for
        // all of them: rows with x_q set take the stabilizer row n+p, row p
        // becomes row n+p, and row n+p becomes Z_q with the coin as its sign
        {
          const uint64_t *M = s_msk + 4 * (k + jr);
          const uint32_t q = rfl((uint32_t)M[0]), slot = rfl((uint32_t)(M[0] >> 32));
          const uint32_t coin_T = rfl((uint32_t)M[1]);
          const uint64_t m = M[2];
          const uint64_t *xq = P + q * stride;
          const uint64_t sw = lane < KH ? xq[KH + lane] : 0ull;
          const uint64_t hit = __ballot(sw != 0);
          const uint32_t kp = (uint32_t)__ffsll((long long)hit) - 1;
          const uint64_t pw = read_lane64(sw, kp);
          const uint32_t bp = (uint32_t)__ffsll((long long)pw) - 1;
          const uint32_t p = 64 * kp + bp;
          const uint64_t bit = 1ull << bp;
          const uint64_t Rs = Rv[n + p], exq = E[q];
          const uint64_t rs = 0ull - ((rc[KH + kp] >> bp) & 1);  // row n+p's sign bit
          if (tid < KW) {
            uint64_t mk = tid < 2 * KH ? xq[tid] : 0ull;
            if (tid == kp || tid == KH + kp) mk &= ~bit;
            sm[tid] = mk;
            s_c0[tid] = 0;
            s_c1[tid] = 0;
          }
          __syncthreads();
          // phases: per row, the sum mod 4 over columns of the phase
          // exponent of row * (row n+p), gathered with LDS atomics
          // (the returned old value carries)
          if (kLds) {
            for (uint32_t j = tid; j < n; j += NT) {
              uint64_t *X = P + j * stride, *Z = X + n * stride;
              const uint64_t wx = X[KH + kp], wz = Z[KH + kp];
              const uint64_t xp = (wx >> bp) & 1, zp = (wz >> bp) & 1;
              if (xp | zp) {
                const uint64_t fx = 0ull - xp, fz = 0ull - zp;
                for (uint32_t i = 0; i < 2 * KH; ++i) {
                  const uint64_t mk = sm[i];
                  if (!mk) continue;
                  const uint64_t x = X[i], z = Z[i];
                  uint64_t d0 = 0, d1 = 0;
                  phase_acc(x, z, fx, fz, d0, d1);
                  X[i] = x ^ (mk & fx);
                  Z[i] = z ^ (mk & fz);
                  d0 &= mk;
                  if (d0) {
                    d1 &= d0;
                    d1 ^= d0 & atomicXor(reinterpret_cast<unsigned long long *>(s_c0 + i),
                                         (unsigned long long)d0);
                    if (d1) lds_xor(s_c1 + i, d1);
                  }
                }
              }
              X[kp] = (X[kp] & ~bit) | (xp << bp);
              Z[kp] = (Z[kp] & ~bit) | (zp << bp);
              X[KH + kp] &= ~bit;
              Z[KH + kp] = (Z[KH + kp] & ~bit) | (j == q ? bit : 0ull);
            }
          } else {
            // 2 KH lanes of one wave per column (a column's words are one
            // run): its loads come before its stores in program order, so
            // lanes read row n+p's bits before the lane that owns that word
            // clears them
            const uint32_t K2 = 2 * KH, cpw = 64 / K2, sub = lane / K2, i = lane - sub * K2;
            const bool use = sub < cpw;
            const uint64_t mk = use ? sm[i] : 0ull;
            const uint32_t cstep = nw * cpw;
            uint64_t c0 = 0, c1 = 0;
            for (uint32_t j0 = wv * cpw + (use ? sub : 0u); j0 < n; j0 += 4 * cstep) {
              uint64_t x[4], z[4], wx[4], wz[4];
#pragma unroll
              for (uint32_t u = 0; u < 4; ++u) {
                const uint32_t j = min(j0 + u * cstep, n - 1);
                const uint64_t *X = P + j * stride, *Z = X + n * stride;
                x[u] = X[i];
                z[u] = Z[i];
                wx[u] = X[KH + kp];
                wz[u] = Z[KH + kp];
              }
              __builtin_amdgcn_wave_barrier();
#pragma unroll
              for (uint32_t u = 0; u < 4; ++u) {
                const uint32_t j = j0 + u * cstep;
                if (use && j < n) {
                  const uint64_t xp = (wx[u] >> bp) & 1, zp = (wz[u] >> bp) & 1;
                  const uint64_t fx = mk & (0ull - xp), fz = mk & (0ull - zp);
                  phase_acc(x[u], z[u], fx, fz, c0, c1);
                  uint64_t nx = x[u] ^ fx, nz = z[u] ^ fz;
                  if (i == kp) {
                    nx = (nx & ~bit) | (xp << bp);
                    nz = (nz & ~bit) | (zp << bp);
                  } else if (i == KH + kp) {
                    nx &= ~bit;
                    nz = (nz & ~bit) | (j == q ? bit : 0ull);
                  }
                  uint64_t *X = P + j * stride + i;
                  if (nx != x[u]) X[0] = nx;
                  if (nz != z[u]) X[n * stride] = nz;
                }
              }
            }
            if (c0 | c1) {
              c1 ^= c0 & atomicXor(reinterpret_cast<unsigned long long *>(s_c0 + i),
                                   (unsigned long long)c0);
              if (c1) lds_xor(s_c1 + i, c1);
            }
          }
          for (uint32_t i = tid; i < 2 * n; i += NT) {
            const uint32_t ii = i < n ? i : i - n;
            const uint64_t mk = sm[(i < n ? 0 : KH) + (ii >> 6)];
            if ((mk >> (ii & 63)) & 1) Rv[i] ^= Rs;  // never rows p, n+p
          }
          if (wv == nw - 1) {
            uint64_t coin;
            if (a.coin_planes) {
              coin = a.coin_planes[m * W + w];
            } else {
              const uint64_t key = stream_key(seed, 2 * (mseq0 + m));
              coin = __ballot((uint32_t)(draw_keyed(key, 64 * w + lane) >> 40) < coin_T);
            }
            if (lane == 0) {
              Rv[p] = Rs;
              Rv[n + p] = coin ^ exq;
              a.recs[(2ull * slot) * W + w] = coin;
              a.recs[(2ull * slot + 1) * W + w] = 0ull;
            }
          }
          __syncthreads();
          if (tid < 2 * KH) {
            uint64_t v = rc[tid] ^ (sm[tid] & (rs ^ s_c1[tid]));
            if (tid == kp) v = (v & ~bit) | (rs & bit);
            if (tid == KH + kp) v &= ~bit;
            rc[tid] = v;
          }
          __syncthreads();
          k += jr + 1;
        }
      }
    }
  }

  // ---- the 64-shot words ----
  // <E, P_i> of 64 rows at a time: a column's word is the lane mask.  Row
  // words times column shares over the waves, gathered in Rv.
  {
    const uint32_t parts = max(1u, 2 * nw / KW);
    const uint32_t per = (n + parts - 1) / parts;
    for (uint32_t task = wv; task < KW * parts; task += nw) {
      const uint32_t kk = task / parts, pt = task - kk * parts;
      const uint32_t ja = pt * per, jb = min(n, ja + per);
      uint64_t acc = 0;
      for (uint32_t j0 = ja; j0 < jb; j0 += 64) {
        const uint32_t jl = min(j0 + lane, n - 1);
        const uint64_t xw = P[jl * stride + kk], zw = P[(n + jl) * stride + kk];
        const uint32_t cnt = min(64u, jb - j0);
        for (uint32_t t = 0; t < cnt; ++t) {
          const uint64_t sx = read_lane64(xw, t), sz = read_lane64(zw, t);
          if (sx) acc ^= (0ull - ((sx >> lane) & 1)) & E[n + j0 + t];
          if (sz) acc ^= (0ull - ((sz >> lane) & 1)) & E[j0 + t];
        }
      }
      if (pt == 0) acc ^= 0ull - ((rc[kk] >> lane) & 1);
      const uint32_t ii = 64 * (kk < KH ? kk : kk - KH) + lane;
      if (kk == 2 * KH) {
        if (lane == 0) lds_xor(Rv + 2 * n, acc);
      } else if (ii < n) {
        lds_xor(Rv + (kk < KH ? 0 : n) + ii, acc);
      }
    }
  }
  __syncthreads();
  for (uint32_t i = tid; i < R; i += NT) Tr[i] = Rv[i];
  // a wave per column: its packed words are read before the column is written
  // over them
  for (uint32_t c = wv; c < 2 * n; c += nw) {
    const uint64_t *src = P + c * stride;
    const uint64_t v0 = lane < KW ? src[lane] : 0ull;
    const uint64_t v1 = lane + 64 < KW ? src[lane + 64] : 0ull;
    __builtin_amdgcn_wave_barrier();
    uint64_t *dst = T + (uint64_t)c * R;
    for (uint32_t kk = 0; kk < 2 * KH; ++kk) {
      const uint64_t s = kk < 64 ? read_lane64(v0, kk) : read_lane64(v1, kk - 64);
      const uint32_t ii = 64 * (kk < KH ? kk : kk - KH) + lane;
      if (ii < n) dst[(kk < KH ? 0 : n) + ii] = 0ull - ((s >> lane) & 1);
    }
    const uint64_t s = 2 * KH < 64 ? read_lane64(v0, 2 * KH) : read_lane64(v1, 2 * KH - 64);
    if (lane == 0) dst[2 * n] = 0ull - (s & 1);
  }
  __syncthreads();
  return true;
}

struct ProgParams {
  uint64_t seed, mseq0, nseq0;
};

// One workgroup per word group.  With a.done, groups that ran are marked
// there and the per-shot kernel launched behind this one passes over them.
template <bool kLds>
__global__ __launch_bounds__(kSharedThreads) void k_program_shared(
    ProgramArgs a, const ProgParams *__restrict__ pp) {
  extern __shared__ uint64_t dyn[];
  __shared__ SharedLds sh;
  const uint64_t seed = pp->seed, mseq0 = pp->mseq0;
  for (uint64_t wi = blockIdx.x; wi < a.nwords; wi += gridDim.x) {
    const bool ran = shared_word<kLds>(a, seed, mseq0, a.word0 + wi, dyn, sh);
    if (a.done && threadIdx.x == 0) a.done[a.word0 + wi] = ran ? 1u : 0u;
    __syncthreads();
  }
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
    if (!bc.a.shared || packed_in_lds(bc.a.n) != kLds) continue;
    const uint64_t w = code & ((1ull << 40) - 1);
    const uint64_t wend = min(w + wtile, bc.a.nwords);
    for (uint64_t wi = w; wi < wend; ++wi) {
      const bool ran = shared_word<kLds>(bc.a, bc.seed, bc.mseq0, wi, dyn, sh);
      if (threadIdx.x == 0) {
        if (bc.a.done) bc.a.done[wi] = ran ? 1u : 0u;
        if (ran) atomicAdd(counter + 2, 1ull);
      }
    }
  }
}

}  // namespace

bool shared_wide(uint32_t n) { return !packed_in_lds(n); }

bool shared_fits(uint32_t n) { return n >= 1 && n <= kSharedMaxQubits; }

size_t shared_lds_bytes(uint32_t n) {
  return 8 * (shared_base_words(n) + (packed_in_lds(n) ? shared_packed_words(n) : 0));
}

hipError_t prepare_shared(uint32_t n) {
  const size_t lds = shared_lds_bytes(n);
  if (lds <= 65536) return hipSuccess;
  const void *fn = packed_in_lds(n) ? (const void *)k_program_shared<true>
                                    : (const void *)k_program_shared<false>;
  return hipFuncSetAttribute(fn, hipFuncAttributeMaxDynamicSharedMemorySize,
                             (int)kSharedLdsBytes);
}

hipError_t prepare_batch_shared() {
  hipError_t e = hipSuccess;
  for (const void *fn : {(const void *)k_batch_shared<true>, (const void *)k_batch_shared<false>})
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
    return dim3((uint32_t)std::min<uint64_t>(
        nitems, cus * std::min<uint64_t>(4, std::max<uint64_t>(1, 160 * 1024 / (lds + 1024)))));
  };
  if (nitems && lds_packed)
    hipLaunchKernelGGL(k_batch_shared<true>, blocks(lds_packed), dim3(kSharedThreads), lds_packed,
                       s, circ, items, nitems, counter, wtile);
  if (nitems && lds_wide)
    hipLaunchKernelGGL(k_batch_shared<false>, blocks(lds_wide), dim3(kSharedThreads), lds_wide, s,
                       circ, items, nitems, counter, wtile);
  return hipGetLastError();
}

hipError_t launch_shared(hipStream_t s, const ProgramArgs &a, const void *params) {
  if (!a.nwords) return hipSuccess;
  const size_t lds = shared_lds_bytes(a.n);
  const uint32_t threads = kSharedThreads;
  const dim3 grid((uint32_t)std::min<uint64_t>(a.nwords, 1u << 20));
  if (packed_in_lds(a.n))
    hipLaunchKernelGGL(k_program_shared<true>, grid, dim3(threads), lds, s, a,
                       (const ProgParams *)params);
  else
    hipLaunchKernelGGL(k_program_shared<false>, grid, dim3(threads), lds, s, a,
                       (const ProgParams *)params);
  return hipGetLastError();
}

}  // namespace pq
