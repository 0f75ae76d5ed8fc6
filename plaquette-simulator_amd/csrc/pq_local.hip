// Per-shot persistent kernel of small states (gfx950): a word group's whole
// tableau stays in LDS.
//
// Programs with flagged H/S/CX/CZ, and runs that do not start from |0...0>,
// have X/Z of their own in every shot.  Up to kLocalMaxQubits qubits the (2n+1)^2
// words of a 64-shot group fit the LDS (n = 41: 55 KB, n = 64: 133 KB), so a
// run reads and writes the tableau once, where k_program_t moves each gate
// segment's columns in and out and measures in memory.
//
// What bounds it is the chain of barriers and LDS latencies of one workgroup:
//  * a layer's ops act on distinct qubits, and each thread keeps one row: rows
//    x ops in parallel, one barrier per layer;
//  * a measurement takes three barriers.  Shots differ in their pivot, but the
//    row operations of different pivots touch different shots: the source
//    words of all pivots are gathered into one row first, and one pass over the
//    tableau does every shot's rowsums (k_program_t: a pass per distinct
//    pivot, up to min(n, 64) of them);
//  * the shots that are determined run their chain of stabilizer rows beside
//    that, cut into one piece per wave: each wave needs the product of the
//    pieces before it, which is an XOR.
// 41 qubits, 5000 shots, 800 ops (a tenth of them flagged), 40 measurements:
// 1759 -> 195 us alone, 516 -> 71 us a pass with several states in flight.
#include "pq_kernels.h"

#include <algorithm>

#include "plaquette_amd.h"

namespace pq {

namespace {

#define PQ_CONST __attribute__((address_space(4)))

constexpr uint32_t kLocalThreads = 768;
constexpr uint32_t kLocalWaves = kLocalThreads / 64;
constexpr uint32_t kLocalSteps = (kLocalMaxQubits + kLocalWaves - 1) / kLocalWaves;
static_assert(kLocalSteps % 2 == 0, "steps run in pairs");

__device__ __forceinline__ uint32_t rfl(uint32_t v) { return __builtin_amdgcn_readfirstlane(v); }
__device__ __forceinline__ uint64_t read_lane64(uint64_t v, uint32_t l) {
  const uint32_t lo = __builtin_amdgcn_readlane((uint32_t)v, l);
  const uint32_t hi = __builtin_amdgcn_readlane((uint32_t)(v >> 32), l);
  return (uint64_t)lo | ((uint64_t)hi << 32);
}
__device__ __forceinline__ void lds_xor(uint64_t *p, uint64_t v) {
  atomicXor(reinterpret_cast<unsigned long long *>(p), (unsigned long long)v);
}
// v of the lane that the DPP control names, 0 where it names none or the row is
// masked off.
template <int kCtrl, int kRows = 0xF>
__device__ __forceinline__ uint64_t dpp64(uint64_t v) {
  const uint32_t lo = __builtin_amdgcn_update_dpp(0, (int)(uint32_t)v, kCtrl, kRows, 0xF, false);
  const uint32_t hi =
      __builtin_amdgcn_update_dpp(0, (int)(uint32_t)(v >> 32), kCtrl, kRows, 0xF, false);
  return (uint64_t)lo | ((uint64_t)hi << 32);
}
// Inclusive OR over the lanes up to this one.
__device__ __forceinline__ uint64_t or_scan(uint64_t v) {
  v |= dpp64<0x111>(v);       // row_shr:1, 2, 4, 8: within rows of 16 lanes
  v |= dpp64<0x112>(v);
  v |= dpp64<0x114>(v);
  v |= dpp64<0x118>(v);
  v |= dpp64<0x142, 0xA>(v);  // row_bcast:15 into rows 1 and 3
  v |= dpp64<0x143, 0xC>(v);  // row_bcast:31 into rows 2 and 3
  return v;
}
template <int kCtrl>
__device__ __forceinline__ void add_dpp(uint64_t &c0, uint64_t &c1) {
  add_mod4(c0, c1, dpp64<kCtrl>(c0), dpp64<kCtrl>(c1));
}
// Sum mod 4, per shot, over each half wave (all its lanes get it).
__device__ __forceinline__ void half_sum(uint64_t &c0, uint64_t &c1) {
  add_dpp<0xB1>(c0, c1);   // quad_perm [1,0,3,2]
  add_dpp<0x4E>(c0, c1);   // quad_perm [2,3,0,1]
  add_dpp<0x141>(c0, c1);  // row_half_mirror
  add_dpp<0x140>(c0, c1);  // row_mirror
  add_mod4(c0, c1, __shfl_xor(c0, 16, 64), __shfl_xor(c1, 16, 64));
}

// One staged op: `cw` = the flags below and from bit 12 the ops of the layer part
// it opens; `qq` = qa | qb << 16.  Its four mask words: what the noise after it
// adds on qa (X part, Z part) and qb; a flagged op keeps its flag in the third,
// and with a record as its flag the record in the fourth.  A measurement has
// record | coin threshold << 32 and its sequence number there.
struct LocalOp {
  uint32_t cw, qq;
};
constexpr uint32_t kOpH = 1, kOpS = 2, kOpCX = 4, kOpCZ = 8;
constexpr uint32_t kOpMeas = 1u << 4, kOpMasks = 1u << 5, kOpX = 1u << 6, kOpZ = 1u << 7;
constexpr uint32_t kOpFlag = 1u << 8, kOpRecord = 1u << 9;
constexpr uint32_t kOpLenShift = 12, kOpLenMask = 0xFFFu;

// Dynamic LDS words besides the staged ops (5 words each): the tableau, a row of
// source words, the rows' masks and the low bits of their phase sums, and the
// waves' pieces of the determined chain.
__host__ __device__ constexpr uint32_t local_words(uint32_t n) {
  const uint32_t R = 2 * n + 1;
  return R * R + R + 4 * n + kLocalWaves * 128;
}
constexpr uint32_t kLocalLdsBytes = 159 * 1024;
__host__ __device__ constexpr uint32_t local_stage(uint32_t n) {
  const uint32_t room = (kLocalLdsBytes / 8 - local_words(n)) / 5;
  return room < kStage ? room : kStage;
}
// a layer, of at most a qubit's op each, runs whole
static_assert(local_stage(kLocalMaxQubits) >= kLocalMaxQubits, "a layer fits the window");

__global__ __launch_bounds__(kLocalThreads) void k_program_local(ProgramArgs a,
                                                                 const ProgParams *__restrict__ pp) {
  extern __shared__ uint64_t dyn[];
  __shared__ uint64_t s_racc;
  const uint32_t tid = threadIdx.x, lane = tid & 63u, wv = rfl(tid >> 6);
  constexpr uint32_t NT = kLocalThreads, NW = kLocalWaves;
  const uint32_t n = a.n, R = a.R, stage = local_stage(n);
  const uint64_t W = a.W;
  const uint64_t seed = pp->seed, mseq0 = pp->mseq0;
  uint64_t *const T = dyn;              // word (column c, row i) at c * R + i
  uint64_t *const rcol = T + 2 * n * R;
  uint64_t *const s_src = T + R * R;
  uint64_t *const s_m = s_src + R;
  uint64_t *const s_c0 = s_m + 2 * n;
  uint64_t *const s_seg = s_c0 + 2 * n;  // [wave][x, z][column]
  uint64_t *const msk = s_seg + NW * 128;
  LocalOp *const ops = reinterpret_cast<LocalOp *>(msk + 4 * stage);
  const PQ_CONST DInstr *ins = (const PQ_CONST DInstr *)a.instrs;
  const uint32_t words = R * R;
  // this thread's row, and its share of a layer's ops
  const uint32_t my_op = tid / R, my_row = tid - my_op * R, opp = NT / R;
  // and of a rowsum pass: columns my_part, my_part + parts, ... of my_i
  const uint32_t parts = NT / (2 * n), my_part = tid / (2 * n), my_i = tid - my_part * 2 * n;
  const uint32_t coin_wave = (2 * n) >> 6;  // the wave of column 2n

  for (uint64_t w = a.word0 + blockIdx.x; w < a.word0 + a.nwords; w += gridDim.x) {
    if (a.done && rfl(a.done[w])) continue;  // k_program_shared ran it
    uint64_t *tab = a.tab + w * (uint64_t)words;
    __syncthreads();
    if (a.fresh) {  // X/Z are the identity, and not in memory
      for (uint32_t i = tid; i < 2 * n * R; i += NT) T[i] = i % (R + 1) == 0 ? ~0ull : 0ull;
      if (tid < R) rcol[tid] = tab[2 * n * R + tid];
    } else {
      for (uint32_t i = tid; i < words; i += 8 * NT) {
        uint64_t v[8];
#pragma unroll
        for (uint32_t u = 0; u < 8; ++u) v[u] = tab[min(i + u * NT, words - 1)];
#pragma unroll
        for (uint32_t u = 0; u < 8; ++u)
          if (i + u * NT < words) T[i + u * NT] = v[u];
      }
    }

    uint64_t rp = 0;  // sign flips of my_row not yet in rcol
    for (uint32_t base = 0; base < a.ninstr;) {
      // instructions [base, base + wn) and their masks, whatever segments they
      // belong to
      const uint32_t wn = min(stage, a.ninstr - base);
      bool flags = false;
      for (uint32_t t = tid; t < wn; t += NT) {
        const PQ_CONST DInstr *I = ins + base + t;
        const uint32_t code = I->code, qa = I->qa, qb = I->qb, slot = I->slot, na = I->na,
                       nb = I->nb, t0 = I->t0, pad = I->pad;
        uint64_t m0 = 0, m1 = 0, m2 = 0, m3 = 0;
        LocalOp J;
        if (code == PQ_OP_M) {
          J.cw = kOpMeas;
          J.qq = qa;
          m0 = (uint64_t)slot | ((uint64_t)t0 << 32);
          m1 = (uint64_t)na | ((uint64_t)nb << 32);
        } else {
          const bool cx = code == PQ_OP_CX || code == PQ_OP_CX_FLAG;
          const bool cz = code == PQ_OP_CZ || code == PQ_OP_CZ_FLAG;
          const bool flg = code >= PQ_OP_H_FLAG && code != PQ_OP_NOISE;
          const bool rec = flg && !(slot & kSlotPlane);
          const bool y = code == PQ_OP_Y || code == PQ_OP_Y_FLAG;
          J.cw = (code == PQ_OP_H || code == PQ_OP_H_FLAG ? kOpH : 0u) |
                 (code == PQ_OP_S || code == PQ_OP_S_FLAG ? kOpS : 0u) | (cx ? kOpCX : 0u) |
                 (cz ? kOpCZ : 0u) |
                 (y || code == PQ_OP_X || code == PQ_OP_X_FLAG ? kOpX : 0u) |
                 (y || code == PQ_OP_Z || code == PQ_OP_Z_FLAG ? kOpZ : 0u) |
                 (flg ? kOpFlag : 0u) | (rec ? kOpRecord : 0u) |
                 (na != kNone || nb != kNone ? kOpMasks : 0u) |
                 (((pad >> kLayerLenShift) & kLayerLenMask) << kOpLenShift);
          J.qq = qa | ((cx || cz ? qb : qa) << 16);
          const PQ_CONST uint64_t *gp = (const PQ_CONST uint64_t *)a.planes + 2ull * a.nk * w;
          if (na != kNone) {
            m0 = gp[2ull * na];
            m1 = gp[2ull * na + 1];
          }
          if (flg) {
            m2 = rec ? a.recs[(2ull * slot) * W + w] : gp[2ull * (slot & ~kSlotPlane)];
            m3 = slot;
          } else if (nb != kNone) {
            m2 = gp[2ull * nb];
            m3 = gp[2ull * nb + 1];
          }
          flags |= rec;
        }
        uint64_t *M = msk + 4 * t;
        M[0] = m0;
        M[1] = m1;
        M[2] = m2;
        M[3] = m3;
        ops[t] = J;
      }
      // flags from records are read again where measurements of this window
      // precede them
      const bool reread = __syncthreads_or(flags);
      bool measured = false;
      uint32_t b = 0;
      while (b < wn) {
        const uint32_t cw = rfl(ops[b].cw);
        if (!(cw & kOpMeas)) {
          const uint32_t cnt = max(1u, (cw >> kOpLenShift) & kOpLenMask);
          if (b + cnt > wn) break;  // a layer part runs whole: it opens the next window
          if (measured && reread) {
            __syncthreads();  // the records are in
            for (uint32_t t = b + tid; t < wn; t += NT)
              if (ops[t].cw & kOpRecord) msk[4 * t + 2] = a.recs[2ull * msk[4 * t + 3] * W + w];
            __syncthreads();
          }
          measured = false;
          if (my_op < opp)
            for (uint32_t o = my_op; o < cnt; o += opp) {
              const LocalOp J = ops[b + o];
              const uint64_t *M = msk + 4 * (b + o);
              uint64_t *xa = T + (__umul24(J.qq & 0xFFFFu, R) + my_row), *za = xa + n * R;
              uint64_t x = *xa, z = *za;
              const uint64_t f = J.cw & kOpFlag ? M[2] : ~0ull;
              if (J.cw & (kOpCX | kOpCZ)) {
                uint64_t *xb = T + (__umul24(J.qq >> 16, R) + my_row), *zb = xb + n * R;
                uint64_t xt = *xb, zt = *zb;
                if (J.cw & kOpCX) {
                  rp ^= f & x & zt & ~(xt ^ z);
                  xt ^= f & x;
                  z ^= f & zt;
                  *xb = xt;
                } else {
                  rp ^= f & x & xt & (zt ^ z);
                  zt ^= f & x;
                  z ^= f & xt;
                  *zb = zt;
                }
                *za = z;
                if ((J.cw & (kOpMasks | kOpFlag)) == kOpMasks) rp ^= (M[2] & zt) ^ (M[3] & xt);
              } else if (J.cw & kOpH) {
                const uint64_t d = f & (x ^ z);
                rp ^= f & x & z;
                x ^= d;
                z ^= d;
                *xa = x;
                *za = z;
              } else if (J.cw & kOpS) {
                rp ^= f & x & z;
                z ^= f & x;
                *za = z;
              } else {
                if (J.cw & kOpX) rp ^= f & z;
                if (J.cw & kOpZ) rp ^= f & x;
              }
              if (J.cw & kOpMasks) rp ^= (M[0] & z) ^ (M[1] & x);
            }
          b += cnt;
          __syncthreads();
          continue;
        }

        // ---- a measurement (MeasurementFunctors.hpp:225-317) ----
        if (!measured) {
          if (my_op < opp && rp) lds_xor(rcol + my_row, rp);
          rp = 0;
          __syncthreads();
        }
        measured = true;
        const uint32_t q = rfl(ops[b].qq);
        const uint64_t M0 = msk[4 * b], mnum = msk[4 * b + 1];
        // lane p: stabilizer row n+p's x_q, and the shots whose pivot it is
        // (the first such row); every wave finds them by itself
        const uint64_t *xq = T + __umul24(q, R);
        const uint64_t xs = lane < n ? xq[n + lane] : 0ull;
        const uint64_t xd = lane < n ? xq[lane] : 0ull;
        const uint64_t inc = or_scan(xs);
        const uint64_t first = xs & ~dpp64<0x138>(inc);  // wave_shr:1
        const uint64_t rm = read_lane64(inc, 63), D = ~rm;
        __syncthreads();  // every wave has read column q
        // the determined shots' chain: destabilizers with x_q set, in order
        const uint64_t dm = xd & D;
        const uint64_t chain = __ballot(dm != 0);
        uint64_t coin = 0;
        if (wv == coin_wave) {
          if (rm) {
            if (a.coin_planes) {
              coin = a.coin_planes[mnum * W + w];
            } else {
              const uint64_t key = stream_key(seed, 2 * (mseq0 + mnum));
              coin = __ballot((uint32_t)(draw_keyed(key, 64 * w + lane) >> 40) <
                              (uint32_t)(M0 >> 32));
            }
          }
          if (lane == 0) s_racc = 0;
        }
        if (rm) {
          // What follows changes the bits of the random shots alone, so D's
          // bits of every word may be read beside it.
          if (wv == NW - 1 && lane < n) {  // the rows that take the source row
            s_m[lane] = xd & rm & ~first;
            s_m[n + lane] = xs & rm & ~first;
            s_c0[lane] = 0;
            s_c0[n + lane] = 0;
          }
          // per pivot row and its shots: row p takes row n+p, row n+p becomes
          // Z_q with the coin as its sign; the old rows n+p, each in its
          // shots, are the source row.  The next pivot's words are read before
          // this one's are written (they are other rows).
          uint64_t left = __ballot(first != 0), acc = 0;
          if (tid < R) {
            uint64_t *col = T + tid * R;
            const uint64_t set = tid == n + q ? ~0ull : tid == 2 * n ? coin : 0ull;
            uint32_t p = (uint32_t)__ffsll((long long)left) - 1;
            uint64_t va = col[n + p], vb = col[p];
            for (;;) {
              left &= left - 1;
              const uint64_t Mp = read_lane64(first, p);
              const uint32_t here = p;
              const uint64_t ha = va, hb = vb;
              if (left) {
                p = (uint32_t)__ffsll((long long)left) - 1;
                va = col[n + p];
                vb = col[p];
              }
              acc |= ha & Mp;
              col[here] = (hb & ~Mp) | (ha & Mp);
              col[n + here] = (ha & ~Mp) | (set & Mp);
              if (!left) break;
            }
            s_src[tid] = acc;
          }
        }
        // this wave's piece of the chain: steps [k0, k1), a lane per column
        const uint32_t nchain = (uint32_t)__popcll(chain), per = (nchain + NW - 1) / NW;
        const uint32_t k0 = min(nchain, wv * per), k1 = min(nchain, k0 + per);
        uint64_t cx[kLocalSteps], cz[kLocalSteps];
        uint64_t mine = chain;  // the destabilizers from step k0 on
        for (uint32_t k = 0; k < k0; ++k) mine &= mine - 1;
        if (chain) {
          uint64_t left = mine;
          uint64_t sx = 0, sz = 0;
#pragma unroll
          for (uint32_t u = 0; u < kLocalSteps; ++u) {
            cx[u] = cz[u] = 0;
            if (k0 + u < k1) {
              const uint32_t i = (uint32_t)__ffsll((long long)left) - 1;
              left &= left - 1;
              const uint64_t m = read_lane64(dm, i);
              const uint64_t *col = T + min(lane, n - 1) * R + n + i;
              cx[u] = lane < n ? col[0] & m : 0ull;
              cz[u] = lane < n ? col[n * R] & m : 0ull;
              sx ^= cx[u];
              sz ^= cz[u];
            }
          }
          s_seg[wv * 128 + lane] = sx;
          s_seg[wv * 128 + 64 + lane] = sz;
        }
        __syncthreads();
        if (rm && my_part < parts) {
          // rowsum(i <- source row) in every random shot with x_q set in row i:
          // partial phase sums mod 4 gathered by LDS atomics, whose old value
          // carries
          const uint64_t mi = s_m[my_i];
          if (mi) {
            uint64_t c0 = 0, c1 = 0;
            for (uint32_t j = my_part; j < n; j += parts) {
              uint64_t *X = T + (__umul24(j, R) + my_i), *Z = X + n * R;
              const uint64_t x = *X, z = *Z, x2 = s_src[j], z2 = s_src[n + j];
              phase_acc(x, z, x2, z2, c0, c1);
              *X = x ^ (mi & x2);
              *Z = z ^ (mi & z2);
            }
            if (my_part == 0) c1 ^= s_src[2 * n];
            c1 ^= c0 & atomicXor(reinterpret_cast<unsigned long long *>(s_c0 + my_i),
                                 (unsigned long long)c0);
            if (c1 & mi) lds_xor(rcol + my_i, c1 & mi);
          }
        }
        if (D && wv == NW - 1) {
          // the scratch row's D shots hold the chain's product
          uint64_t sx = 0, sz = 0;
          if (chain)
#pragma unroll
            for (uint32_t v = 0; v < NW; ++v) {
              sx ^= s_seg[v * 128 + lane];
              sz ^= s_seg[v * 128 + 64 + lane];
            }
          if (lane < n) {
            uint64_t *col = T + lane * R + 2 * n;
            col[0] = (col[0] & ~D) | sx;
            col[n * R] = (col[n * R] & ~D) | sz;
          }
        }
        if (k0 < k1) {
          uint64_t sx = 0, sz = 0;
          for (uint32_t v = 0; v < wv; ++v) {
            sx ^= s_seg[v * 128 + lane];
            sz ^= s_seg[v * 128 + 64 + lane];
          }
          // two steps at a time: each half wave sums one of them
          const bool hi = lane >= 32;
          uint64_t racc = 0;
#pragma unroll
          for (uint32_t u = 0; u < kLocalSteps; u += 2) {
            if (k0 + u >= k1) break;
            const uint32_t ia = (uint32_t)__ffsll((long long)mine) - 1;
            mine &= mine - 1;
            const bool two = k0 + u + 1 < k1;
            const uint32_t ib = two ? (uint32_t)__ffsll((long long)mine) - 1 : ia;
            mine &= mine - 1;
            const uint64_t ma = read_lane64(dm, ia), mb = two ? read_lane64(dm, ib) : 0ull;
            const uint64_t r = rcol[n + (hi ? ib : ia)];
            uint64_t a0 = 0, a1 = 0, b0 = 0, b1 = 0;
            phase_acc(sx, sz, cx[u], cz[u], a0, a1);
            sx ^= cx[u];
            sz ^= cz[u];
            phase_acc(sx, sz, cx[u + 1], cz[u + 1], b0, b1);
            sx ^= cx[u + 1];
            sz ^= cz[u + 1];
            uint64_t c0 = hi ? b0 : a0, c1 = hi ? b1 : a1;
            add_mod4(c0, c1, __shfl_xor(hi ? a0 : b0, 32, 64), __shfl_xor(hi ? a1 : b1, 32, 64));
            half_sum(c0, c1);
            racc ^= (hi ? mb : ma) & (r ^ c1);
          }
          if ((lane & 31) == 0) lds_xor(&s_racc, racc);
        }
        __syncthreads();
        if (wv == coin_wave && lane == 0) {
          const uint64_t rdet = s_racc;
          uint64_t *rec = a.recs + (2ull * (uint32_t)M0) * W + w;
          rec[0] = (coin & rm) | (rdet & D);
          rec[W] = D;
          rcol[2 * n] = (rcol[2 * n] & ~D) | (rdet & D);
        }
        ++b;
      }
      base += b;
      __syncthreads();
    }
    if (my_op < opp && rp) lds_xor(rcol + my_row, rp);
    __syncthreads();
    for (uint32_t i = tid; i < words; i += NT) tab[i] = T[i];
  }
}

}  // namespace

bool local_fits(uint32_t n) { return n >= 1 && n <= kLocalMaxQubits; }

static size_t local_lds_bytes(uint32_t n) {
  return 8ull * (local_words(n) + 5ull * local_stage(n));
}

hipError_t prepare_local() {
  return hipFuncSetAttribute((const void *)k_program_local,
                             hipFuncAttributeMaxDynamicSharedMemorySize, (int)kLocalLdsBytes);
}

hipError_t launch_local(hipStream_t s, const ProgramArgs &a, const void *params) {
  if (!a.nwords) return hipSuccess;
  hipLaunchKernelGGL(k_program_local, dim3((uint32_t)std::min<uint64_t>(a.nwords, 1u << 20)),
                     dim3(kLocalThreads), local_lds_bytes(a.n), s, a, (const ProgParams *)params);
  return hipGetLastError();
}

}  // namespace pq
