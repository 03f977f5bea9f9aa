// fp32 path of the MoE layer (include/smel_f32.h): the reference's layer on fp32 tensors, whose _gmm falls to a
// per-group matmul loop for any non-bf16 tensor (smel/moe.py:58-72). Grouped GEMMs on v_mfma_f32_16x16x4_f32 (int4 tiles
// also as exact bf16 parts on v_mfma_f32_16x16x32_bf16, Split below) over the same tile lists and group kinds as the bf16
// GEMMs, LoRA weight gradients as row-group reductions on the same MFMA,
// and the fp32 element-wise steps around them (gather, act-gate, combine, dX reduce, router selection and backward,
// the Gemma router input, the shared-expert gate). Everything sums in a fixed order: no atomics.
#include <math.h>

#include <type_traits>

#include "../../include/smel_f32.h"
#include "abi_util.h"
#include "common.h"

namespace {

typedef float f32v4 __attribute__((ext_vector_type(4)));

// v_mfma_f32_16x16x4_f32: lane l supplies A[i = l % 16][k = l / 16] and B[k = l / 16][j = l % 16] and holds
// D[4 (l / 16) + r][j = l % 16], r = 0..3
SMEL_DEV f32v4 mfma4(float a, float b, const f32v4& c) { return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0); }

// ---------------------------------------------------------------------------------------------- weight matrices

// One matrix [R][C] of a weight set: fp32 values, or the reference's int4 format dequantized as w = q s + z in fp32
// (q s is exact in fp32, so this equals the separate product and sum), optionally rounded to bf16. Offsets inside a
// matrix are 32-bit (one matrix is below 2^31 elements); the group index is a shift when the group is a power of two.
struct WMat {
  const float* f;
  const uint8_t* q;
  const uint16_t* s;
  const uint16_t* z;
  int C;
  int gpr;      // groups per row, C / group
  int group;
  int gshift;   // log2(group), or -1
  uint32_t gmul;   // ceil(2^32 / group): col / group as one high product (0: some col group is 2^32 or more)
  int rbf;
};

SMEL_DEV int gidx(const WMat& m, int row, int col) {
  return row * m.gpr +
         (m.gshift >= 0 ? col >> m.gshift : m.gmul ? (int)__umulhi((uint32_t)col, m.gmul) : col / m.group);
}

SMEL_DEV float dq(const WMat& m, uint32_t q, int gi) {
  const float v = fmaf((float)q, bf2f(m.s[gi]), bf2f(m.z[gi]));
  return m.rbf ? bf2f(f2bf(v)) : v;
}

SMEL_DEV float w_at(const WMat& m, int row, int col) {
  if (m.f) return m.f[row * m.C + col];
  const uint32_t b = m.q[row * (m.C >> 1) + (col >> 1)];
  return dq(m, (b >> (4 * (col & 1))) & 0xfu, gidx(m, row, col));
}

// Elements [row][col .. col + 3] (col a multiple of 4, col + 3 < C, C a multiple of 4): one 16-byte load for fp32,
// one 16-bit load of nibbles for int4 (one scale / zero pair when the group is a multiple of 4).
SMEL_DEV void w_quad(const WMat& m, int row, int col, float v[4]) {
  if (m.f) {
    const float4 x = *reinterpret_cast<const float4*>(m.f + row * m.C + col);
    v[0] = x.x, v[1] = x.y, v[2] = x.z, v[3] = x.w;
    return;
  }
  const uint32_t qq = *reinterpret_cast<const uint16_t*>(m.q + row * (m.C >> 1) + (col >> 1));
  if ((m.group & 3) == 0) {
    const int gi = gidx(m, row, col);
    const float sc = bf2f(m.s[gi]), ze = bf2f(m.z[gi]);
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const float x = fmaf((float)((qq >> (4 * i)) & 0xfu), sc, ze);
      v[i] = m.rbf ? bf2f(f2bf(x)) : x;
    }
  } else {
#pragma unroll
    for (int i = 0; i < 4; ++i) v[i] = dq(m, (qq >> (4 * i)) & 0xfu, gidx(m, row, col + i));
  }
}

SMEL_DEV bool resolve(const smel_wset_f32& w, int kind, int idx, WMat& m) {
  m.C = (int)w.C;
  m.group = w.group > 0 ? w.group : 1;
  m.gpr = (int)(w.C / m.group);
  m.gshift = (m.group & (m.group - 1)) == 0 ? __builtin_ctz((unsigned)m.group) : -1;
  m.gmul = (int64_t)m.C * m.group < (1ll << 32) ? 0xffffffffu / (uint32_t)m.group + 1u : 0u;
  m.rbf = w.q4_round_bf16;
  m.f = nullptr;
  m.q = nullptr;
  m.s = m.z = nullptr;
  const int64_t n = w.R * w.C;
  switch (kind) {
    case SMEL_KIND_INT4:
      if (!w.q4) return false;
      m.q = w.q4 + (int64_t)idx * (n >> 1);
      m.s = w.scale + (int64_t)idx * w.R * m.gpr;
      m.z = w.zero + (int64_t)idx * w.R * m.gpr;
      return true;
    case SMEL_KIND_BF16: m.f = w.wf ? w.wf + (int64_t)idx * n : nullptr; break;
    case SMEL_KIND_SEL: m.f = w.wsel ? w.wsel + (int64_t)idx * n : nullptr; break;
    default: m.f = w.wsh ? w.wsh + (int64_t)idx * n : nullptr; break;
  }
  return m.f != nullptr;
}

// Eight consecutive weights from one 32-bit word of nibbles (even column in the low nibble of a byte), one scale / zero.
SMEL_DEV void dq8(uint32_t w, float sc, float ze, int rbf, float* v) {
  const uint32_t e = w & 0x0f0f0f0fu, o = (w >> 4) & 0x0f0f0f0fu;
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    v[2 * j] = fmaf((float)((e >> (8 * j)) & 0xffu), sc, ze);
    v[2 * j + 1] = fmaf((float)((o >> (8 * j)) & 0xffu), sc, ze);
  }
  if (rbf) {
#pragma unroll
    for (int j = 0; j < 8; ++j) v[j] = bf2f(f2bf(v[j]));
  }
}

// ---------------------------------------------------------------------------------------------- grouped GEMM
// What bounds it: the fp32 MFMA rate (64 FLOP per SIMD and clock), then the dequant of the weights beside it (about 3
// VALU instructions per weight and 64-row tile). A block takes RB rows of one tile of the list (the tile in RB-row
// steps) and NT output columns; per k-step of FK the operands go through two LDS stages (the next step's global loads
// in flight during this step's MFMAs, one barrier per step). The rows run in 16-row slices, only as many as the tile
// has: a frozen expert of 32 rows costs 2 slices (the 32x32 MFMA form computed 64 rows for it). A lane takes four
// consecutive k of its row with one 16-byte LDS read and feeds them to four MFMAs (the order inside the sum over k is
// free); a wave's NF column fragments interleave their columns (column = NF i + f), so that for W [K][N] one NF-float
// read gives every fragment its value.
// Two shapes (the rule is in smel_gmm_f32): 64 x 128 with the four waves side by side along the columns, and 32 x 64
// with the four waves each on a quarter of the staged k, summed through LDS in wave order, for launches whose tiles
// would leave most of the 256 CUs idle.
// Measured, 1021 tokens top-8 of 256 experts (12 of them fp32), H 2048, I 512 (about 32 rows per expert): gate_up 991 ->
// 445 us, down 462 -> 240, down backward 528 -> 274, gate_up backward 949 -> 485 (against 64 x 64 blocks of 32x32x2
// MFMAs; int4 tiles on whole k-steps now run as Split below); the 16-row slices computed are 43 GFLOP of gate_up = 97
// TFLOP/s of the 157 nominal. With the loop's barriers
// waiting for global loads, or its load and store code behind branches, the same tiles took 560-620 us.
// One k-step's operands of a thread on their way from global memory to LDS.
struct StageRegs {
  u32x4_t a[2];   // 8 values of A
  u32x4_t b[4];   // 16 weights: fp32 values, or the raw nibbles in b[0] (b[0..1]: pairs)
  uint32_t bs, bz;   // scale and zero of a run of 16
  uint32_t ms[8], mz[8];   // of each quad or pair
};

struct GemmArgs {
  const float* A;
  int64_t lda;
  float alpha;
  int beta1;
  float* C;
  int64_t ldc;
  int c2;   // columns of C in aligned pairs
};

// How a block reads its operands.
//   W_INT4   A in 16-byte loads, runs of 16 nibbles (8 bytes, one scale / zero pair); W_INT4R: rounded to bf16
//   W_F32    A and fp32 weights in 16-byte loads
// and the forms for any alignment and any group, whose threads take neighbouring elements of the stage instead of runs:
//   W_QUAD   A in 16-byte loads, four nibbles with a scale / zero pair of their own (W_QUAD1: A element by element)
//   W_PAIR   A element by element, two nibbles with a pair of their own
//   W_ELEM   A and fp32 weights element by element
// All of them keep their loads two k-steps ahead. Measured (64 experts of 32 rows, 1024 x 2048; quads one step ahead on
// 32x32 MFMAs -> element by element without loads ahead -> here): groups of 8 306 -> 1199 -> 155 us, transposed 230 ->
// 545 -> 147, A of an odd pitch 253 -> 811 -> 147; fp32 matrices of 2046 columns (16 of 64 rows) 167 -> 190 -> 70,
// transposed 93 -> 220 -> 77.
enum { W_INT4 = 0, W_F32 = 1, W_INT4R = 2, W_QUAD = 3, W_QUAD1 = 4, W_PAIR = 5, W_ELEM = 6 };

template <int TRANS, int RB, int NT, int KS, int FK>
struct Gemm {
  static constexpr int NWN = 4 / KS;            // waves along the columns
  static constexpr int NF = NT / NWN / 16;      // 16-column fragments of a wave
  static constexpr int RF = RB / 16;            // 16-row slices
  static constexpr int KW = FK / KS;            // k of a step that one wave takes
  static constexpr int PA = FK + 4;             // pitch of the [row][k] stages: 16-byte reads of 8 lanes on distinct banks
  static constexpr int PB = TRANS ? NT : PA;    // W stage: [k][n] for TRANS, else [n][k]
  static constexpr int SA = RB * PA, SB = TRANS ? FK * NT : NT * PA;
  static constexpr int LDS_FLOATS = 2 * (SA + SB);
  static_assert(RB * FK == 8 * 256 && NT * FK == 16 * 256, "staging split");
  static_assert(KS == 1 || KS * RB * (NT + 4) <= LDS_FLOATS, "reduction buffer");

  // The forms for any alignment: thread t takes units x = 256 e + t of U weights, in the order of the W stage (SW weights a
  // row of it). Matrix row and column of a unit, held inside the matrix, and whether it is inside.
  static constexpr int SW = TRANS ? NT : FK;
  template <int U>
  SMEL_DEV static int wrow(int x, int k0, int n0, int WR) {
    return min((TRANS ? k0 : n0) + x / (SW / U), WR - 1);
  }
  template <int U>
  SMEL_DEV static int wcol(int x, int k0, int n0, int WC) {
    return min((TRANS ? n0 : k0) + x % (SW / U) * U, WC - U);
  }
  template <int U>
  SMEL_DEV static bool wok(int x, int k0, int n0, int WR, int WC) {
    return (TRANS ? k0 : n0) + x / (SW / U) < WR && (TRANS ? n0 : k0) + x % (SW / U) * U < WC;
  }

  // NRF: the 16-row slices computed (those of the tile's rows; the others' rows are zeros in LDS); only: the rows stored
  // (bit r: row mr0 + r)
  template <int MODE, int NRF>
  SMEL_DEV static void tile(float* __restrict__ lds, const GemmArgs& G, const WMat& m, int N, int K, int n0, int mr0,
                            int mr1, uint64_t only = ~0ull) {
    constexpr bool INT4 = MODE == W_INT4 || MODE == W_INT4R, RUNS = INT4 || MODE == W_F32;
    constexpr bool AVEC = RUNS || MODE == W_QUAD;
    int t = threadIdx.x;
    asm volatile("" : "+v"(t));   // the addresses made from it belong to this tile: kept over a loop of tiles they would spill
    const int l = t & 63, wv = t >> 6, i = l & 15, kq = l >> 4;
    const int wn = wv % NWN, wk = wv / NWN;
    const int nk = (K + FK - 1) / FK;
    // load coordinates: A row t / (FK / 8), 8 k; W: a run of 16 along the matrix's rows
    const int am = t / (FK / 8), ak = 8 * (t % (FK / 8));
    const int bo = TRANS ? t / (NT / 16) : t / (FK / 16);           // outer index: k (TRANS) or n
    const int br = TRANS ? 16 * (t % (NT / 16)) : 16 * (t % (FK / 16));
    const int WR = TRANS ? K : N, WC = TRANS ? N : K;
    const float* const ab = G.A + (int64_t)mr0 * G.lda;
    const rsrc_t ra = make_rsrc(ab, ((uint64_t)(mr1 - mr0 - 1) * G.lda + K) * 4);
    const rsrc_t rw = INT4 ? make_rsrc(m.q, (uint64_t)WR * (m.C >> 1)) : make_rsrc(m.f, (uint64_t)WR * m.C * 4);
    const rsrc_t rs = make_rsrc(m.s, INT4 ? (uint64_t)WR * m.gpr * 2 : 0);
    const rsrc_t rz = make_rsrc(m.z, INT4 ? (uint64_t)WR * m.gpr * 2 : 0);
    const uint32_t arow = am < mr1 - mr0 ? (uint32_t)(am * G.lda) : OOB;
    auto load = [&](StageRegs& S, int k0) {
      const int k = k0 + ak;
      const int wr = TRANS ? k0 + bo : n0 + bo;   // matrix row and first column of the run
      const int wc = TRANS ? n0 + br : k0 + br;
      if (AVEC) {
#pragma unroll
        for (int h = 0; h < 2; ++h) S.a[h] = ld16(ra, (arow != OOB && k + 4 * h < K) ? 4 * (arow + k + 4 * h) : OOB);
      } else {
#pragma unroll
        for (int e = 0; e < 8; ++e) {
          const int x = 256 * e + t;
          S.a[e >> 2][e & 3] = __float_as_uint(ab[min(x / FK, mr1 - mr0 - 1) * G.lda + min(k0 + x % FK, K - 1)]);
        }
      }
      // elements past the edges: the last one's value here, zero where it is stored
      if (MODE == W_ELEM) {
#pragma unroll
        for (int e = 0; e < 16; ++e) {
          const int x = 256 * e + t;
          S.b[e >> 2][e & 3] = __float_as_uint(m.f[wrow<1>(x, k0, n0, WR) * (int64_t)m.C + wcol<1>(x, k0, n0, WC)]);
        }
      } else if (!RUNS) {
        constexpr int U = MODE == W_PAIR ? 2 : 4;
#pragma unroll
        for (int e = 0; e < 16 / U; ++e) {
          const int x = 256 * e + t, r = wrow<U>(x, k0, n0, WR), c = wcol<U>(x, k0, n0, WC);
          const uint8_t* const p = m.q + (int64_t)r * (m.C >> 1) + (c >> 1);
          S.b[e >> 2][e & 3] = U == 4 ? *reinterpret_cast<const uint16_t*>(p) : *p;
          const int gi = gidx(m, r, c);
          S.ms[e] = m.s[gi], S.mz[e] = m.z[gi];
        }
      } else if (INT4) {   // C a multiple of 16, so a run is inside the matrix or past it
        const bool ok = wr < WR && wc < WC;
        const u32x2_t q = ld8(rw, ok ? (uint32_t)(wr * (m.C >> 1) + (wc >> 1)) : OOB);
        S.b[0][0] = q[0], S.b[0][1] = q[1];
        // past the matrix: zero nibbles under a zero scale and zero
        const uint32_t go = ok ? 2u * (uint32_t)(wr * m.gpr + (int)__umulhi((uint32_t)wc, m.gmul)) : OOB;
        S.bs = ld2(rs, go), S.bz = ld2(rz, go);
      } else {
#pragma unroll
        for (int j = 0; j < 4; ++j)
          S.b[j] = ld16(rw, (wr < WR && wc + 4 * j < WC) ? 4u * (uint32_t)(wr * m.C + wc + 4 * j) : OOB);
      }
    };
    auto store = [&](StageRegs& S, int buf, int k0) {
      float* const As = lds + buf * (SA + SB);
      float* const Bs = As + SA;
      float* const ap = As + am * PA + ak;
      float* const bp = Bs + bo * PB + br;
      if (!AVEC) {
#pragma unroll
        for (int e = 0; e < 8; ++e) {
          const int x = 256 * e + t;
          const bool ok = x / FK < mr1 - mr0 && k0 + x % FK < K;
          As[x / FK * PA + x % FK] = ok ? __uint_as_float(S.a[e >> 2][e & 3]) : 0.f;
        }
      }
      if (MODE == W_ELEM) {
#pragma unroll
        for (int e = 0; e < 16; ++e) {
          const int x = 256 * e + t;
          Bs[x / SW * PB + x % SW] = wok<1>(x, k0, n0, WR, WC) ? __uint_as_float(S.b[e >> 2][e & 3]) : 0.f;
        }
        return;
      }
      if (!RUNS) {
        constexpr int U = MODE == W_PAIR ? 2 : 4;
#pragma unroll
        for (int e = 0; e < 16 / U; ++e) {
          const int x = 256 * e + t;
          const bool ok = wok<U>(x, k0, n0, WR, WC);
          const uint32_t n4 = S.b[e >> 2][e & 3];
          float v[U];
#pragma unroll
          for (int j = 0; j < U; ++j) {
            v[j] = fmaf((float)(n4 >> (4 * j) & 0xfu), bf2f(S.ms[e]), bf2f(S.mz[e]));
            if (m.rbf) v[j] = bf2f(f2bf(v[j]));
            v[j] = ok ? v[j] : 0.f;
          }
          float* const d = Bs + x / (SW / U) * PB + x % (SW / U) * U;
          if (U == 4) *reinterpret_cast<float4*>(d) = make_float4(v[0], v[1], v[2 % U], v[3 % U]);
          else *reinterpret_cast<float2*>(d) = make_float2(v[0], v[1]);
        }
        if (!AVEC) return;
      }
#pragma unroll
      for (int h = 0; h < 2; ++h) *reinterpret_cast<u32x4_t*>(ap + 4 * h) = S.a[h];
      if (!RUNS) return;
      if (INT4) {
        float v[16];
        const float sc = __uint_as_float(S.bs << 16), ze = __uint_as_float(S.bz << 16);
        dq8(S.b[0][0], sc, ze, MODE == W_INT4R, v);
        dq8(S.b[0][1], sc, ze, MODE == W_INT4R, v + 8);
#pragma unroll
        for (int j = 0; j < 4; ++j)
          *reinterpret_cast<float4*>(bp + 4 * j) = make_float4(v[4 * j], v[4 * j + 1], v[4 * j + 2], v[4 * j + 3]);
      } else {
#pragma unroll
        for (int j = 0; j < 4; ++j) *reinterpret_cast<u32x4_t*>(bp + 4 * j) = S.b[j];
      }
    };
    f32v4 acc[NRF][NF] = {};
    auto compute16 = [&](int buf, int k16) {
      const float* const As = lds + buf * (SA + SB);
      const float* const Bs = As + SA;
      {
        const int kk = wk * KW + k16 + 4 * kq;
        float b[4][NF];   // [k in the quad][fragment]
        if (TRANS) {
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            const float* p = Bs + (kk + e) * PB + 16 * NF * wn + NF * i;
            if (NF == 2) {
              const float2 v = *reinterpret_cast<const float2*>(p);
              b[e][0] = v.x, b[e][1] = v.y;
            } else {
              const float4 v = *reinterpret_cast<const float4*>(p);
              b[e][0] = v.x, b[e][1] = v.y, b[e][2 % NF] = v.z, b[e][3 % NF] = v.w;
            }
          }
        } else {
#pragma unroll
          for (int f = 0; f < NF; ++f) {
            const float4 v = *reinterpret_cast<const float4*>(Bs + (16 * NF * wn + NF * i + f) * PB + kk);
            b[0][f] = v.x, b[1][f] = v.y, b[2][f] = v.z, b[3][f] = v.w;
          }
        }
#pragma unroll
        for (int rf = 0; rf < NRF; ++rf) {
          const float4 a = *reinterpret_cast<const float4*>(As + (16 * rf + i) * PA + kk);
#pragma unroll
          for (int f = 0; f < NF; ++f) acc[rf][f] = mfma4(a.x, b[0][f], acc[rf][f]);
#pragma unroll
          for (int f = 0; f < NF; ++f) acc[rf][f] = mfma4(a.y, b[1][f], acc[rf][f]);
#pragma unroll
          for (int f = 0; f < NF; ++f) acc[rf][f] = mfma4(a.z, b[2][f], acc[rf][f]);
#pragma unroll
          for (int f = 0; f < NF; ++f) acc[rf][f] = mfma4(a.w, b[3][f], acc[rf][f]);
        }
      }
    };
    auto compute = [&](int buf) {
#pragma unroll
      for (int k16 = 0; k16 < KW; k16 += 16) compute16(buf, k16);
    };
    // Global loads run two k-steps ahead of their use, in two register sets; the barriers wait for LDS only. One
    // branch-free block per step, so that the next stage's dequant is issued between the MFMAs (two waves of a SIMD
    // reach their MFMA and VALU phases together: apart, the phases would add up). Steps past K load and add zeros.
    StageRegs S0, S1;
    load(S0, 0);
    load(S1, FK);
    store(S0, 0, 0);
    lds_barrier();
    int kt = 0;
    for (; (kt + 2) * FK <= K; kt += 2) {
      load(S0, (kt + 2) * FK);
      compute(0);
      store(S1, 1, (kt + 1) * FK);
      lds_barrier();
      load(S1, (kt + 3) * FK);
      compute(1);
      store(S0, 0, (kt + 2) * FK);
      lds_barrier();
    }
    // up to two steps left, the last one for the k it has: all of a LoRA factor's rank (12 groups of 600 rows, N 2048: K 16
    // 41 -> 23 us, transposed 42 -> 21; K 48 41 -> 34, 44 -> 32; whole steps of zeros before, results in single columns)
    auto rest = [&](int buf, int step) {
#pragma unroll 1
      for (int k16 = 0; k16 < KW && step * FK + wk * KW + k16 < K; k16 += 16) compute16(buf, k16);
    };
    if (kt < nk) rest(0, kt);
    if (kt + 1 < nk) {
      store(S1, 1, (kt + 1) * FK);
      lds_barrier();
      rest(1, kt + 1);
    }
    if constexpr (KS > 1) lds_barrier();   // the stages become the reduction buffer
    if constexpr (KS == 1) {
#pragma unroll
      for (int rf = 0; rf < NRF; ++rf)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const int row = mr0 + 16 * rf + 4 * kq + r;
          if (row >= mr1 || !(only >> (row - mr0) & 1)) continue;
          float* const p = G.C + (int64_t)row * G.ldc;
          if (NF == 2 && G.c2) {   // a lane's two columns in one access
            const int col = n0 + 16 * NF * wn + NF * i;
            if (col >= N) continue;
            float2* const p2 = reinterpret_cast<float2*>(p + col);
            const float2 o = G.beta1 ? *p2 : make_float2(0.f, 0.f);
            const float v0 = G.alpha * acc[rf][0][r], v1 = G.alpha * acc[rf][NF - 1][r];
            *p2 = G.beta1 ? make_float2(o.x + v0, o.y + v1) : make_float2(v0, v1);
            continue;
          }
#pragma unroll
          for (int f = 0; f < NF; ++f) {
            const int col = n0 + 16 * NF * wn + NF * i + f;
            if (col < N) p[col] = G.beta1 ? p[col] + G.alpha * acc[rf][f][r] : G.alpha * acc[rf][f][r];
          }
        }
    } else {   // the waves' k quarters, summed in wave order
      constexpr int PR = NT + 4;
#pragma unroll
      for (int rf = 0; rf < NRF; ++rf)
#pragma unroll
        for (int r = 0; r < 4; ++r)
#pragma unroll
          for (int f = 0; f < NF; ++f) lds[(wk * RB + 16 * rf + 4 * kq + r) * PR + 16 * NF * wn + NF * i + f] = acc[rf][f][r];
      lds_barrier();
      for (int e = t; e < RB * NT; e += 256) {
        const int rr = e / NT, cc = e % NT;
        const int row = mr0 + rr, col = n0 + cc;
        if (row >= mr1 || col >= N || !(only >> rr & 1)) continue;   // rows past NRF slices are past mr1
        float v = lds[rr * PR + cc];
#pragma unroll
        for (int q = 1; q < KS; ++q) v += lds[(q * RB + rr) * PR + cc];
        float* const p = G.C + (int64_t)row * G.ldc + col;
        *p = G.beta1 ? *p + G.alpha * v : G.alpha * v;
      }
      lds_barrier();
    }
  }
};

// ---------------------------------------------------------------------------------------------- int4 tiles on bf16 MFMAs
// fp32 products of int4 tiles from 16-bit matrix instructions without losing bits: an fp32 value is the sum of three bf16
// values (x0 = bf16(x), x1 = bf16(x - x0), x2 = bf16(x - x0 - x1); the differences are exact and 3 x 8 bits hold all 24),
// a weight q s + z of a group whose scale and zero are of similar size the sum of two (its bits lie in 16 places, see
// splits()), and a bf16 x bf16 product is exact in fp32: x w = x0 w0 + (x0 w1 + x1 w0 + x1 w1 + x2 w0 + x2 w1), all six
// products kept. Weights rounded to bf16 (RBF) are one value: three products. Six v_mfma_f32_16x16x32_bf16 take 96 cycles
// for the 32 k that eight v_mfma_f32_16x16x4_f32 take 256 for.
// The sums: that instruction loses up to a unit in the last place of what it adds to (an fp32 addition half of one), so
// no sum runs through it from step to step: per 32 k the products x0 w0 and the small ones each start from zero, and fp32
// additions bring them together and onto the running sum. Error against 64 bits relative to sum |x w| (1024 to 2048
// columns, all int4; fp32 instruction -> here), largest / rms: one non-zero term 5.96e-8 / 2.51e-8 -> 5.98e-8 / 2.51e-8,
// two terms 1.17e-7 / 2.59e-8 -> 1.17e-7 / 3.05e-8 (each rounded before they meet, as in any sum by parts), eight 2.4e-7
// / 2.7e-8 -> 2.2e-7 / 2.8e-8, 64 3.2e-7 / 2.8e-8 -> 1.3e-7 / 1.5e-8, full rows 3.6e-7 / 2.8e-8 -> 3.4e-8 / 3.7e-9.
// What the parts cannot hold is computed by the fp32 instruction, in rows of their own (a row's bits depend on that row and
// the weights alone): rows with a non-zero value below 2^-72 (the parts of smaller values, or their products with the
// smallest weights, come near the end of the exponent range) and rows with an infinite or NaN sum (infinities, NaN,
// numbers that round up to infinity); all rows where a weight of the block is no sum of two.
// What bounds it: the VALU work of dequant and splitting, about 6 instructions per weight and pass, and 6 per row value
// (48 rows: 888 for 144 MFMAs a step). So no weight is split twice in a pass of up to 48 rows: a wave takes all 128
// columns of the block for its quarter of the k-steps (every fourth step of 32), straight from global memory into
// registers without a barrier, and the waves' sums are added through LDS in wave order. Only the block's scales and
// zeros (packed) wait in LDS. Measured (8168 rows over 256 int4 experts, H 2048, I 512; the six largest of nine products
// of three-part weights, summed in the instruction -> here): gate_up 309 -> 302 us, down 166 -> 166, down backward 158 ->
// 146, gate_up backward 288 -> 272 (the fp32 instruction: 445, 240, 274, 485).
// x and y as three bf16 values each, packed (the differences are exact).
SMEL_DEV void split3(float x, float y, uint32_t& p0, uint32_t& p1, uint32_t& p2) {
  p0 = pack2bf(x, y);
  x -= bf_lo(p0), y -= bf_hi(p0);
  p1 = pack2bf(x, y);
  x -= bf_lo(p1), y -= bf_hi(p1);
  p2 = pack2bf(x, y);
}

SMEL_DEV f32v4 mfma32b(const u32x4_t& a, const u32x4_t& b, const f32v4& c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8_t, a), __builtin_bit_cast(bf16x8_t, b), c, 0,
                                                 0, 0);
}

template <int TRANS>
struct Split {
  using GM = Gemm<TRANS, 64, 128, 1, 32>;
  static constexpr int NF = 8, NT = 128, MAXRF = 3;
  static constexpr int PR = NT + 4;   // pitch of the reduction rows
  static_assert(4 * 16 * PR <= GM::LDS_FLOATS, "reduction buffer");

  // groups of one k row (TRANS) or of one output row that the block's panel of scales holds
  SMEL_DEV static int panel_groups(const WMat& m, int N, int n0) {
    return TRANS ? (min(n0 + NT, N) - 1) / m.group - n0 / m.group + 1 : m.gpr;
  }
  // (vec and qvec hold) whole k-steps, a lane's 8 weights under one scale / zero pair, the panel inside the LDS
  SMEL_DEV static bool fits(const WMat& m, int N, int K, int n0) {
    return K % 32 == 0 && m.group % 32 == 0 && (int64_t)panel_groups(m, N, n0) * (TRANS ? K : NT) <= GM::LDS_FLOATS;
  }

  // A weight q s + z is two bf16 values exactly when all its bits lie in 16 consecutive places: the last bits of s and z
  // are 2^(exponent - 7) each, the weight is below 2^(1 + max(exponent of s + 4, exponent of z)). Zero or exponents of at
  // least -40 (what is left of a weight after cancellation is then a normal bf16 value), finite.
  template <bool RBF>
  SMEL_DEV static bool splits(uint32_t s, uint32_t z) {
    const int es = s >> 7 & 0xff, ez = z >> 7 & 0xff;
    const bool zs = (s & 0x7fffu) == 0, zz = (z & 0x7fffu) == 0;
    const bool in = (zs | ((unsigned)(es - (127 - 40)) < 168u)) & (zz | ((unsigned)(ez - (127 - 40)) < 168u));
    return in & (RBF | zs | zz | ((unsigned)(ez - es + 4) <= 12u));
  }

  // Returns the rows that are still to be computed (bit r: row mr0 + r), the same for the whole block.
  template <int NRF, bool RBF>
  SMEL_DEV static uint64_t tile(float* __restrict__ lds, const GemmArgs& G, const WMat& m, int N, int K, int n0, int mr0,
                                int mr1) {
    __shared__ uint32_t again[2];   // rows to compute again (48 bits)
    int t = threadIdx.x;
    asm volatile("" : "+v"(t));   // as in Gemm
    const int l = t & 63, i = l & 15, kq = l >> 4;
    const int wv = __builtin_amdgcn_readfirstlane(t >> 6);
    const int nk = K / 32, nfw = min(NT, N - n0);
    const int half = m.C >> 1, WR = TRANS ? K : N;
    const rsrc_t ra = make_rsrc(G.A + (int64_t)mr0 * G.lda, ((uint64_t)(mr1 - mr0 - 1) * G.lda + K) * 4);
    const rsrc_t rw = make_rsrc(m.q, (uint64_t)WR * half);
    uint32_t arow[NRF];
#pragma unroll
    for (int rf = 0; rf < NRF; ++rf) {
      const int r = 16 * rf + i;
      arow[rf] = r < mr1 - mr0 ? 4u * (uint32_t)(r * (int)G.lda + 8 * kq) : OOB;
    }
    // column 8 i + f of the block is fragment f of lane i; rows of the matrix past its last read as zeros
    const uint32_t wb = TRANS ? (8 * i < nfw ? (uint32_t)(8 * kq * half + ((n0 + 8 * i) >> 1)) : OOB)
                              : (uint32_t)((n0 + 8 * i) * half + 4 * kq);
    u32x4_t araw[NRF][2];   // 8 k of the lane's row per 16-row slice
    uint32_t q[8], qn[8];   // 64 nibbles
    // OOB plus any offset inside a matrix stays out of range; steps past the last one load it again
    auto load_a = [&](int step) {
      uint32_t at = 128u * min(step, nk - 1);
      asm("" : "+s"(at));
#pragma unroll
      for (int rf = 0; rf < NRF; ++rf)
#pragma unroll
        for (int h = 0; h < 2; ++h) araw[rf][h] = ld16(ra, arow[rf] + at + 16 * h);
    };
    auto load_q = [&](uint32_t* o, int step) {
      const uint32_t at = (uint32_t)min(step, nk - 1) * (TRANS ? 32u * half : 16u);
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        uint32_t aj = at + (uint32_t)(j * half);
        asm("" : "+s"(aj));   // one vector add per load, not eight addresses kept over the loop
        o[j] = ld4(rw, wb + aj);
      }
    };
    load_a(wv);
    load_q(q, wv);
    if (t < 2) again[t] = 0;
    // scale | zero << 16 of the block's weights: [group][column] or, TRANS, [group][k]
    uint32_t* const P = reinterpret_cast<uint32_t*>(lds);
    const int ng = panel_groups(m, N, n0), g0 = TRANS ? n0 / m.group : 0;
    const int outer = TRANS ? K : NT;
    const int gs = ng <= 1 ? 0 : 32 - __builtin_clz((unsigned)(ng - 1));   // consecutive threads: a row's groups
    uint32_t range = 0, apart = 0;
    {
      const rsrc_t rs = make_rsrc(m.s, (uint64_t)WR * m.gpr * 2), rz = make_rsrc(m.z, (uint64_t)WR * m.gpr * 2);
#pragma unroll 8
      for (int e = t; e < outer << gs; e += 256) {
        const int o = e >> gs, g = e & ((1 << gs) - 1);
        const uint32_t off = 2u * (uint32_t)((TRANS ? o : n0 + o) * m.gpr + g0 + g);
        const uint32_t s = ld2(rs, off), z = ld2(rz, off);
        if (g < ng) P[g * outer + o] = s | (z << 16);
        // the common case of splits() without its exceptions: exponents in range and apart by no more than it allows
        const uint32_t s1 = (s & 0x7fffu) - (87u << 7), z1 = (z & 0x7fffu) - (87u << 7);
        range = max(range, max(s1, z1));
        if constexpr (!RBF) apart = max(apart, z1 - s1 + 512u);
      }
    }
    lds_barrier();
    const uint32_t* const pl = P + (TRANS ? ((n0 + min(8 * i, nfw - 1)) / m.group - g0) * K + 8 * kq : 8 * i);
    f32v4 acc[NRF][NF] = {};
    uint32_t least[NRF];   // smallest of 2 |bits| - 1 (zeros wrap to the largest)
#pragma unroll
    for (int rf = 0; rf < NRF; ++rf) least[rf] = ~0u;
    for (int step = wv; step < nk; step += 4) {   // no barrier: each wave its own steps
      u32x4_t a0[NRF], a1[NRF], a2[NRF];
#pragma unroll
      for (int rf = 0; rf < NRF; ++rf)
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          const uint32_t x = araw[rf][j >> 1][2 * (j & 1)], y = araw[rf][j >> 1][2 * (j & 1) + 1];
          least[rf] = min(least[rf], min(2 * x - 1, 2 * y - 1));
          uint32_t p0, p1, p2;
          split3(__uint_as_float(x), __uint_as_float(y), p0, p1, p2);
          a0[rf][j] = p0, a1[rf][j] = p1, a2[rf][j] = p2;
        }
      const uint32_t* const sp = pl + (TRANS ? 32 * step : 32 * step / m.group * NT);
      const u32x4_t z0 = *reinterpret_cast<const u32x4_t*>(sp), z1 = *reinterpret_cast<const u32x4_t*>(sp + 4);
      // TRANS: nibble f of every row's word; the even ones first, then the odd ones shifted into their bytes
      uint32_t nib8[8];
      u32x4_t b[2][2];
      auto weights = [&](int f, u32x4_t* o) {   // fragment f's 8 weights, split
        float w[8];
#pragma unroll
        for (int j = 0; j < 8; ++j) {   // TRANS: row j's nibble f; else row f's nibble j
          const int wd = TRANS ? j : f, nb = TRANS ? f : j;
          if (TRANS ? (f == 0 || f == 1) : j < 2)
            nib8[TRANS ? j : j & 1] = (nb & 1 ? q[wd] >> 4 : q[wd]) & 0x0f0f0f0fu;
          const uint32_t sz = wd < 4 ? z0[wd & 3] : z1[wd & 3];
          const uint32_t n4 = nib8[TRANS ? j : j & 1];
          w[j] = fmaf(nb < 2 ? ub0(n4) : nb < 4 ? ub1(n4) : nb < 6 ? ub2(n4) : ub3(n4), bf_lo(sz), bf_hi(sz));
        }
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          const uint32_t p0 = pack2bf(w[2 * j], w[2 * j + 1]);
          o[0][j] = p0;
          if constexpr (!RBF) o[1][j] = pack2bf(w[2 * j] - bf_lo(p0), w[2 * j + 1] - bf_hi(p0));
        }
      };
      // fragments in the order 0 2 4 6 1 3 5 7; the next one's weights are made between this one's MFMAs, and the fence
      // keeps the later ones out of registers that are not there
      weights(0, b[0]);
#pragma unroll
      for (int o = 0; o < NF; ++o) {
        const int f = o < 4 ? 2 * o : 2 * o - 7, fn = o + 1 < 4 ? 2 * o + 2 : 2 * o - 5;
        __builtin_amdgcn_sched_barrier(0);
        if (o == 4) load_q(qn, step + 4);
        if (o == 5) load_a(step + 4);
        f32v4 big[NRF], small[NRF];   // a0 w0, and the other products, the smallest first
        const u32x4_t* const c = b[o & 1];
        auto mm = [&](f32v4* d, const u32x4_t* a, const u32x4_t& bb, bool first) {
#pragma unroll
          for (int rf = 0; rf < NRF; ++rf) d[rf] = mfma32b(a[rf], bb, first ? f32v4{} : d[rf]);
        };
        if constexpr (!RBF) mm(small, a2, c[1], true);
        mm(small, a2, c[0], RBF);
        if constexpr (!RBF) mm(small, a1, c[1], false);
        mm(small, a1, c[0], false);
        if constexpr (!RBF) mm(small, a0, c[1], false);
        mm(big, a0, c[0], true);
        if (o + 1 < NF) weights(fn, b[(o + 1) & 1]);
#pragma unroll
        for (int rf = 0; rf < NRF; ++rf) acc[rf][f] += big[rf] + small[rf];
      }
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int j = 0; j < 8; ++j) q[j] = qn[j];
    }
    // rows of a value below 2^-72 that is not zero, and rows with an infinite or NaN sum
    constexpr uint32_t LEAST = 2u * ((127u - 72u) << 23) - 1u;
    float bad = 0.f;   // NaN once a sum is infinite or NaN
    uint32_t low = ~0u;
#pragma unroll
    for (int rf = 0; rf < NRF; ++rf) {
      low = min(low, least[rf]);
#pragma unroll
      for (int f = 0; f < NF; ++f)
#pragma unroll
        for (int r = 0; r < 4; ++r) bad = fmaf(acc[rf][f][r], 0.f, bad);
    }
    bool odd = range >= 168u << 7 || apart > 1536u;   // (a group past the block's counts too)
    if (__builtin_amdgcn_ballot_w64(bad != 0.f || low < LEAST || odd)) {
      if (odd) {
        odd = false;
        for (int e = t; e < outer << gs; e += 256) {
          const int o = e >> gs, g = e & ((1 << gs) - 1);
          if (g < ng) odd |= !splits<RBF>(P[g * outer + o] & 0xffffu, P[g * outer + o] >> 16);
        }
        if (odd) atomicOr(&again[0], ~0u), atomicOr(&again[1], ~0u);
      }
#pragma unroll
      for (int rf = 0; rf < NRF; ++rf) {
        if (least[rf] < LEAST) atomicOr(&again[rf >> 1], 1u << (16 * (rf & 1) + i));
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          float v = 0.f;
#pragma unroll
          for (int f = 0; f < NF; ++f) v = fmaf(acc[rf][f][r], 0.f, v);
          if (v != 0.f) atomicOr(&again[rf >> 1], 1u << (16 * (rf & 1) + 4 * kq + r));
        }
      }
    }
    lds_barrier();   // every wave is done with the scales
    const uint32_t redo[2] = {(uint32_t)__builtin_amdgcn_readfirstlane(again[0]),
                              (uint32_t)__builtin_amdgcn_readfirstlane(again[1])};
#pragma unroll
    for (int rf = 0; rf < NRF; ++rf) {
#pragma unroll
      for (int r = 0; r < 4; ++r)
#pragma unroll
        for (int h = 0; h < 2; ++h)
          *reinterpret_cast<f32v4*>(lds + (16 * wv + 4 * kq + r) * PR + 8 * i + 4 * h) =
              f32v4{acc[rf][4 * h][r], acc[rf][4 * h + 1][r], acc[rf][4 * h + 2][r], acc[rf][4 * h + 3][r]};
      lds_barrier();
      const int cc = t & (NT - 1), row0 = mr0 + 16 * rf;
      const uint32_t skip = redo[rf >> 1] >> (16 * (rf & 1) + (t >> 7));
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        const int rr = (t >> 7) + 2 * j;
        float v = lds[rr * PR + cc];
#pragma unroll
        for (int q = 1; q < 4; ++q) v += lds[(16 * q + rr) * PR + cc];
        if (row0 + rr < mr1 && cc < nfw && !(skip >> 2 * j & 1)) {
          float* const p = G.C + (int64_t)(row0 + rr) * G.ldc + n0 + cc;
          *p = G.beta1 ? *p + G.alpha * v : G.alpha * v;
        }
      }
      lds_barrier();
    }
    return redo[0] | (uint64_t)redo[1] << 32;
  }
};

// FORMS: what a launch's kinds need of the forms above, in kernels of their own (the registers of one cost the others a
// block per CU): fp32 weights in 16-byte loads only (dense weights, LoRA factors), those and runs of nibbles, or any
// alignment and group.
enum { FORMS_F32 = 0, FORMS_RUNS = 1, FORMS_ANY = 2 };
template <int TRANS, int RB, int NT, int KS, int FK, int FORMS>
__global__ __launch_bounds__(256, FORMS == FORMS_F32 && TRANS ? 3 : 2) void gmm_f32_kernel(smel_wset_f32 w, const int32_t* __restrict__ gkind,
                                                         const int32_t* __restrict__ tiles,
                                                         const int32_t* __restrict__ n_tiles, int vec, int qvec,
                                                         GemmArgs G) {
  using GM = Gemm<TRANS, RB, NT, KS, FK>;
  __shared__ __align__(16) float lds[GM::LDS_FLOATS];
  const int N = (int)(TRANS ? w.C : w.R), K = (int)(TRANS ? w.R : w.C);
  // the column blocks of a tile run back to back on XCD tile % 8 (blocks go to the XCDs round robin): its A rows are
  // read from that XCD's L2
  const int ncol = (N + NT - 1) / NT, slot = blockIdx.x >> 3;
  const int ti = (slot / ncol) * 8 + (blockIdx.x & 7), n0 = (slot % ncol) * NT;
  if (ti >= n_tiles[0]) return;
  const int g = tiles[4 * ti], r0 = tiles[4 * ti + 1], r1 = tiles[4 * ti + 2];
  const int gk = gkind ? gkind[g] : tiles[4 * ti + 3];
  const int kind = gk >> 16, idx = gk & 0xffff;
  if (!((w.kinds >> kind) & 1)) return;
  WMat m;
  if (!resolve(w, kind, idx, m)) return;
  if constexpr (FORMS == FORMS_RUNS && NT == Split<TRANS>::NT) {
    if (!m.f && Split<TRANS>::fits(m, N, K, n0)) {
      // the tile's 16-row slices in passes of up to three, as even as they go
      const int ns = (r1 - r0 + 15) >> 4, np = (ns + Split<TRANS>::MAXRF - 1) / Split<TRANS>::MAXRF;
      for (int p = blockIdx.z; p < np; p += gridDim.z) {
        const int s0 = p * ns / np, s1 = (p + 1) * ns / np;
        const int mr0 = r0 + 16 * s0, mr1 = min(r1, r0 + 16 * s1);
        uint64_t redo;
        if (m.rbf) redo = Split<TRANS>::template tile<3, true>(lds, G, m, N, K, n0, mr0, mr1);
        else if (s1 - s0 == 1) redo = Split<TRANS>::template tile<1, false>(lds, G, m, N, K, n0, mr0, mr1);
        else if (s1 - s0 == 2) redo = Split<TRANS>::template tile<2, false>(lds, G, m, N, K, n0, mr0, mr1);
        else redo = Split<TRANS>::template tile<3, false>(lds, G, m, N, K, n0, mr0, mr1);
        if (!redo) continue;
        if (m.rbf) GM::template tile<W_INT4R, GM::RF>(lds, G, m, N, K, n0, mr0, mr1, redo);
        else GM::template tile<W_INT4, GM::RF>(lds, G, m, N, K, n0, mr0, mr1, redo);
        lds_barrier();
      }
      return;
    }
  }
  // the tile's rows in RB-row steps; gridDim.z blocks share them
  for (int mr0 = r0 + RB * (int)blockIdx.z; mr0 < r1; mr0 += RB * (int)gridDim.z) {
    const int mr1 = min(r1, mr0 + RB);
    const int nrf = (mr1 - mr0 + 15) >> 4;
    if constexpr (FORMS == FORMS_ANY) {
      auto run = [&](auto mode) {
        if (nrf <= 2) GM::template tile<mode.value, 2>(lds, G, m, N, K, n0, mr0, mr1);
        else if constexpr (GM::RF > 2) GM::template tile<mode.value, GM::RF>(lds, G, m, N, K, n0, mr0, mr1);
      };
      if (m.f) run(std::integral_constant<int, W_ELEM>{});
      else if (qvec == 0) run(std::integral_constant<int, W_PAIR>{});
      else if (vec & 1) run(std::integral_constant<int, W_QUAD>{});
      else run(std::integral_constant<int, W_QUAD1>{});
    } else if (FORMS == FORMS_F32 || m.f) {
      if (nrf == 1) GM::template tile<W_F32, 1>(lds, G, m, N, K, n0, mr0, mr1);
      else if (nrf == 2) GM::template tile<W_F32, 2>(lds, G, m, N, K, n0, mr0, mr1);
      else GM::template tile<W_F32, GM::RF>(lds, G, m, N, K, n0, mr0, mr1);
    } else if (m.rbf) {
      GM::template tile<W_INT4R, GM::RF>(lds, G, m, N, K, n0, mr0, mr1);
    } else {
      if (nrf == 1) GM::template tile<W_INT4, 1>(lds, G, m, N, K, n0, mr0, mr1);
      else if (nrf == 2) GM::template tile<W_INT4, 2>(lds, G, m, N, K, n0, mr0, mr1);
      else if (GM::RF > 2 && nrf == 3) GM::template tile<W_INT4, GM::RF - 1>(lds, G, m, N, K, n0, mr0, mr1);
      else GM::template tile<W_INT4, GM::RF>(lds, G, m, N, K, n0, mr0, mr1);
    }
    lds_barrier();
  }
}

// Few output columns (LoRA factors, the shared gate): one block per 16 rows of a tile, the 8 waves on interleaved
// 16-wide runs of k, straight from global memory into registers (no staging: nothing is used twice), summed through
// LDS in wave order. Bound: memory latency, which a wave meets K / 128 / UNR times. Columns of fragment f: NF i + f.
template <int TRANS, int NF>
__global__ __launch_bounds__(512) void gmm_f32_skinny_kernel(smel_wset_f32 w, const int32_t* __restrict__ gkind,
                                                             const int32_t* __restrict__ tiles,
                                                             const int32_t* __restrict__ n_tiles,
                                                             const float* __restrict__ A, int64_t lda, int vec,
                                                             float alpha, int beta1, float* __restrict__ C,
                                                             int64_t ldc) {
  constexpr int NT = 16 * NF, UNR = 4;
  __shared__ float red[8][16][NT + 1];
  const int ti = blockIdx.x;
  if (ti >= n_tiles[0]) return;
  const int g = tiles[4 * ti], r0 = tiles[4 * ti + 1], r1 = tiles[4 * ti + 2];
  const int gk = gkind ? gkind[g] : tiles[4 * ti + 3];
  const int kind = gk >> 16, idx = gk & 0xffff;
  if (!((w.kinds >> kind) & 1)) return;
  WMat m;
  if (!resolve(w, kind, idx, m)) return;
  const int N = (int)(TRANS ? w.C : w.R), K = (int)(TRANS ? w.R : w.C);
  const int t = threadIdx.x, l = lane_id(), wv = t >> 6, i = l & 15, kq = l >> 4;
  const bool avec = vec & 1, wvec = (m.C & 3) == 0 && (m.f ? (vec & 2) != 0 : true);
  for (int mr0 = r0 + 16 * (int)blockIdx.z; mr0 < r1; mr0 += 16 * (int)gridDim.z) {
    const int row = mr0 + i;
    const bool rok = row < r1;
    const float* const ap = A + (int64_t)(rok ? row : mr0) * lda;
    f32v4 acc[NF] = {};
    for (int k0 = 16 * wv; k0 < K; k0 += 16 * 8 * UNR) {
      float a[UNR][4], b[UNR][4][NF];
#pragma unroll
      for (int u = 0; u < UNR; ++u) {
        const int k = k0 + 128 * u + 4 * kq;
        if (avec && k + 3 < K) {
          const float4 v = *reinterpret_cast<const float4*>(ap + k);
          a[u][0] = v.x, a[u][1] = v.y, a[u][2] = v.z, a[u][3] = v.w;
        } else {
#pragma unroll
          for (int e = 0; e < 4; ++e) a[u][e] = k + e < K ? ap[k + e] : 0.f;
        }
        if (TRANS) {
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            if (NF == 4 && wvec && k + e < K && NF * i + 3 < N) {
              float v[4];
              w_quad(m, k + e, 4 * i, v);
#pragma unroll
              for (int f = 0; f < NF; ++f) b[u][e][f] = v[f % 4];
            } else {
#pragma unroll
              for (int f = 0; f < NF; ++f) b[u][e][f] = (k + e < K && NF * i + f < N) ? w_at(m, k + e, NF * i + f) : 0.f;
            }
          }
        } else {
#pragma unroll
          for (int f = 0; f < NF; ++f) {
            const int n = NF * i + f;
            if (wvec && n < N && k + 3 < K) {
              float v[4];
              w_quad(m, n, k, v);
#pragma unroll
              for (int e = 0; e < 4; ++e) b[u][e][f] = v[e];
            } else {
#pragma unroll
              for (int e = 0; e < 4; ++e) b[u][e][f] = (n < N && k + e < K) ? w_at(m, n, k + e) : 0.f;
            }
          }
        }
      }
#pragma unroll
      for (int u = 0; u < UNR; ++u)
#pragma unroll
        for (int e = 0; e < 4; ++e)
#pragma unroll
          for (int f = 0; f < NF; ++f) acc[f] = mfma4(rok ? a[u][e] : 0.f, b[u][e][f], acc[f]);
    }
#pragma unroll
    for (int f = 0; f < NF; ++f)
#pragma unroll
      for (int r = 0; r < 4; ++r) red[wv][4 * kq + r][NF * i + f] = acc[f][r];
    __syncthreads();
    for (int e = t; e < 16 * NT; e += 512) {
      const int rr = e / NT, cc = e % NT;
      if (mr0 + rr < r1 && cc < N) {
        float v = red[0][rr][cc];
#pragma unroll
        for (int q = 1; q < 8; ++q) v += red[q][rr][cc];
        float* const p = C + (int64_t)(mr0 + rr) * ldc + cc;
        *p = beta1 ? *p + alpha * v : alpha * v;
      }
    }
    __syncthreads();
  }
}

// ---------------------------------------------------------------------------------------------- weight gradients
// Block = (16 columns of the narrower side, 64 of the wider one, job); the job's rows are the contraction. The 8 waves
// take interleaved row quads straight from global memory: lane (kq, i) reads S[row][s0 + i] and the 16 bytes
// B[row][b0 + 4 i ..] of row = quad + kq, which feed four MFMAs (column 4 i + f in fragment f). The waves' sums are
// added through LDS in wave order. Bound: memory latency of the row loop (rows / 32 quads per wave, UNR in flight).
// S is X (SWAP 0: the output is [s][b]) or Y (SWAP 1: [b][s]).
template <int SWAP>
__global__ __launch_bounds__(512) void wgrad_f32_kernel(const float* __restrict__ S, int64_t lds_, int64_t ns,
                                                        const float* __restrict__ B, int64_t ldb, int64_t nb,
                                                        const int32_t* __restrict__ offsets,
                                                        const int32_t* __restrict__ job_group, int vec, int64_t N,
                                                        float alpha, float* __restrict__ C, int64_t c_stride) {
  constexpr int UNR = 8;
  __shared__ float red[8][16][65];
  const int j = blockIdx.y;
  const int nbb = (int)((nb + 63) / 64);
  const int64_t s0 = (int64_t)(blockIdx.x / nbb) * 16, b0 = (int64_t)(blockIdx.x % nbb) * 64;
  const int g = job_group[j];
  const int64_t r0 = offsets[g], r1 = offsets[g + 1];
  const int t = threadIdx.x, l = lane_id(), wv = t >> 6, i = l & 15, kq = l >> 4;
  const int64_t si = s0 + i, bi = b0 + 4 * i;
  f32v4 acc[4] = {};
  for (int64_t q0 = r0 + 4 * wv; q0 < r1; q0 += 32 * UNR) {
    float a[UNR], b[UNR][4];
#pragma unroll
    for (int u = 0; u < UNR; ++u) {
      const int64_t r = q0 + 32 * u + kq;
      const bool ok = r < r1;
      a[u] = (ok && si < ns) ? S[r * lds_ + si] : 0.f;
      if (vec && ok && bi + 3 < nb) {
        const float4 v = *reinterpret_cast<const float4*>(B + r * ldb + bi);
        b[u][0] = v.x, b[u][1] = v.y, b[u][2] = v.z, b[u][3] = v.w;
      } else {
#pragma unroll
        for (int f = 0; f < 4; ++f) b[u][f] = (ok && bi + f < nb) ? B[r * ldb + bi + f] : 0.f;
      }
    }
#pragma unroll
    for (int u = 0; u < UNR; ++u)
#pragma unroll
      for (int f = 0; f < 4; ++f) acc[f] = mfma4(a[u], b[u][f], acc[f]);
  }
#pragma unroll
  for (int f = 0; f < 4; ++f)
#pragma unroll
    for (int r = 0; r < 4; ++r) red[wv][4 * kq + r][4 * i + f] = acc[f][r];
  __syncthreads();
  float* const Cj = C + (int64_t)j * c_stride;
  for (int e = t; e < 16 * 64; e += 512) {
    const int ss = SWAP ? e % 16 : e / 64, bb = SWAP ? e / 16 : e % 64;
    if (s0 + ss >= ns || b0 + bb >= nb) continue;
    float v = red[0][ss][bb];
#pragma unroll
    for (int q = 1; q < 8; ++q) v += red[q][ss][bb];
    if (SWAP)
      Cj[(b0 + bb) * N + s0 + ss] = alpha * v;
    else
      Cj[(s0 + ss) * N + b0 + bb] = alpha * v;
  }
}

// ---------------------------------------------------------------------------------------------- element-wise

// Sum over a 256-thread block, the same order every time (each wave's tree, then the waves in order).
SMEL_DEV float block_sum(float v, float* red) {
  v = wave_sum(v);
  __syncthreads();
  if (lane_id() == 0) red[threadIdx.x >> 6] = v;
  __syncthreads();
  return red[0] + red[1] + red[2] + red[3];
}

SMEL_DEV float sigmoid32(float x) { return 1.0f / (1.0f + expf(-x)); }

// act(g) as torch computes it in fp32 (F.silu: g / (1 + e^-g); F.gelu tanh), and (act, act') as act_and_grad
SMEL_DEV float act32(float g, int act) {
  if (act == 0) return g / (1.0f + expf(-g));
  const float c = 0.7978845608028654f;
  return 0.5f * g * (1.0f + tanhf(c * (g + 0.044715f * g * g * g)));
}
SMEL_DEV void act_grad32(float g, int act, float& a, float& da) {
  if (act == 0) {
    const float s = sigmoid32(g);
    a = g * s;
    da = s * (1.0f + g * (1.0f - s));
    return;
  }
  const float c = 0.7978845608028654f;
  const float th = tanhf(c * (g + 0.044715f * g * g * g));
  a = 0.5f * g * (1.0f + th);
  da = 0.5f * (1.0f + th) + 0.5f * g * (1.0f - th * th) * c * (1.0f + 3.0f * 0.044715f * g * g);
}

// The row kernels below take V = 4 columns per thread and access (16-byte loads and stores) where the row length, the
// pitches and the bases allow it, V = 1 elsewhere; the same sums in the same order either way. They are bound by HBM;
// 1021 tokens (8168 rows of 2048): combine and its backward 32 -> 24 us, dX reduce 37 -> 17 us with V = 4
// against V = 1.
template <int V>
struct FVec {
  float v[V];
};
template <int V>
SMEL_DEV FVec<V> ldv(const float* p) {
  FVec<V> r;
  if constexpr (V == 4) {
    const float4 x = *reinterpret_cast<const float4*>(p);
    r.v[0] = x.x, r.v[1] = x.y, r.v[2] = x.z, r.v[3] = x.w;
  } else {
    r.v[0] = p[0];
  }
  return r;
}
template <int V>
SMEL_DEV void stv(float* p, const FVec<V>& r) {
  if constexpr (V == 4)
    *reinterpret_cast<float4*>(p) = make_float4(r.v[0], r.v[1], r.v[2], r.v[3]);
  else
    p[0] = r.v[0];
}

template <int V>
__global__ __launch_bounds__(256) void gather_rows_f32_kernel(const float* __restrict__ src, int64_t lds,
                                                              const int32_t* __restrict__ idx, int div,
                                                              const int32_t* __restrict__ n_valid, int64_t cols,
                                                              float* __restrict__ out) {
  const int64_t p = blockIdx.x;
  const int i = (n_valid && p >= n_valid[0]) ? -1 : idx[p];
  const float* s = i >= 0 ? src + (int64_t)(i / div) * lds : nullptr;
  float* o = out + p * cols;
  for (int64_t c = V * threadIdx.x; c < cols; c += 256 * V) stv<V>(o + c, s ? ldv<V>(s + c) : FVec<V>{});
}

template <int V>
__global__ __launch_bounds__(256) void act_gate_f32_kernel(const float* __restrict__ h, int64_t ldh, int64_t I, int act,
                                                           float* __restrict__ a, int64_t lda) {
  const int64_t r = blockIdx.x;
  for (int64_t j = V * threadIdx.x; j < I; j += 256 * V) {
    const FVec<V> g = ldv<V>(h + r * ldh + j), u = ldv<V>(h + r * ldh + I + j);
    FVec<V> o;
#pragma unroll
    for (int e = 0; e < V; ++e) o.v[e] = act32(g.v[e], act) * u.v[e];
    stv<V>(a + r * lda + j, o);
  }
}

template <int V>
__global__ __launch_bounds__(256) void act_gate_bwd_f32_kernel(const float* __restrict__ h, int64_t ldh,
                                                               const float* __restrict__ da, int64_t ldda, int64_t I,
                                                               int act, float* __restrict__ dh, int64_t lddh) {
  const int64_t r = blockIdx.x;
  for (int64_t j = V * threadIdx.x; j < I; j += 256 * V) {
    const FVec<V> g = ldv<V>(h + r * ldh + j), u = ldv<V>(h + r * ldh + I + j), d = ldv<V>(da + r * ldda + j);
    FVec<V> og, ou;
#pragma unroll
    for (int e = 0; e < V; ++e) {
      float a, dg;
      act_grad32(g.v[e], act, a, dg);
      og.v[e] = d.v[e] * u.v[e] * dg;
      ou.v[e] = d.v[e] * a;
    }
    stv<V>(dh + r * lddh + j, og);
    stv<V>(dh + r * lddh + I + j, ou);
  }
}

template <int V>
__global__ __launch_bounds__(256) void combine_f32_kernel(const float* __restrict__ ys, const float* __restrict__ topv,
                                                          const int32_t* __restrict__ inv, int K, int64_t H,
                                                          float* __restrict__ out) {
  const int64_t t = blockIdx.x;
  for (int64_t c = V * threadIdx.x; c < H; c += 256 * V) {
    FVec<V> acc = {};
#pragma unroll 8
    for (int k = 0; k < K; ++k) {   // no branch: eight rows' loads in flight
      const int p = inv[t * K + k];
      const FVec<V> y = ldv<V>(ys + (int64_t)max(p, 0) * H + c);
      const float w = topv[t * K + k];
#pragma unroll
      for (int e = 0; e < V; ++e) acc.v[e] = p >= 0 ? acc.v[e] + y.v[e] * w : acc.v[e];
    }
    stv<V>(out + t * H + c, acc);
  }
}

// One block per (token, slot): the row's gradient and its dot product with the row.
template <int V>
__global__ __launch_bounds__(256) void combine_bwd_f32_kernel(const float* __restrict__ ys,
                                                              const float* __restrict__ dout,
                                                              const float* __restrict__ topv,
                                                              const int32_t* __restrict__ inv, int K, int64_t H,
                                                              float* __restrict__ dys, float* __restrict__ dtopv) {
  __shared__ float red[4];
  const int64_t t = blockIdx.x, tk = t * K + blockIdx.y;
  const int p = inv[tk];   // block-uniform
  float dot = 0.f;
  if (p >= 0) {
    const float tv = topv[tk];
    for (int64_t c = V * threadIdx.x; c < H; c += 256 * V) {
      const FVec<V> d = ldv<V>(dout + t * H + c), y = ldv<V>(ys + (int64_t)p * H + c);
      FVec<V> o;
#pragma unroll
      for (int e = 0; e < V; ++e) {
        o.v[e] = tv * d.v[e];
        dot += y.v[e] * d.v[e];
      }
      stv<V>(dys + (int64_t)p * H + c, o);
    }
  }
  dot = block_sum(dot, red);
  if (threadIdx.x == 0) dtopv[tk] = dot;
}

template <int V>
__global__ __launch_bounds__(256) void dx_reduce_f32_kernel(const float* __restrict__ dxs,
                                                            const int32_t* __restrict__ inv, int K, int64_t H,
                                                            float* __restrict__ dx) {
  const int64_t t = blockIdx.x;
  for (int64_t c = V * threadIdx.x; c < H; c += 256 * V) {
    FVec<V> acc = {};
#pragma unroll 8
    for (int k = 0; k < K; ++k) {
      const int p = inv[t * K + k];
      const FVec<V> y = ldv<V>(dxs + (int64_t)max(p, 0) * H + c);
#pragma unroll
      for (int e = 0; e < V; ++e) acc.v[e] = p >= 0 ? acc.v[e] + y.v[e] : acc.v[e];
    }
    stv<V>(dx + t * H + c, acc);
  }
}

// One wave per token. The top-k compares the fp32 probabilities themselves (the reference's torch.topk(probs)):
// 64-bit keys (probability bits, then the complement of the expert id, so equal values take the lower id first).
template <int NPL>
__global__ __launch_bounds__(256) void route_select_f32_kernel(const float* __restrict__ logits, int64_t ldl, int T,
                                                               int E, int K, const float* __restrict__ pes,
                                                               float* __restrict__ probs, float* __restrict__ topv,
                                                               int64_t* __restrict__ topi,
                                                               int32_t* __restrict__ topi32) {
  const int64_t t = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6);
  if (t >= T) return;
  const int l = lane_id();
  float v[NPL];
#pragma unroll
  for (int j = 0; j < NPL; ++j) {
    const int e = l + 64 * j;
    v[j] = e < E ? logits[t * ldl + e] : -INFINITY;
  }
  float mx = v[0];
#pragma unroll
  for (int j = 1; j < NPL; ++j) mx = fmaxf(mx, v[j]);
  mx = wave_max(mx);
  float ex[NPL], s = 0.f;
#pragma unroll
  for (int j = 0; j < NPL; ++j) {
    ex[j] = (l + 64 * j) < E ? expf(v[j] - mx) : 0.f;
    s += ex[j];
  }
  s = wave_sum(s);
  uint64_t key[NPL];
#pragma unroll
  for (int j = 0; j < NPL; ++j) {
    const int e = l + 64 * j;
    const float p = ex[j] / s;
    if (e < E) probs[t * E + e] = p;
    key[j] = e < E ? ((uint64_t)__float_as_uint(p) << 32) | (uint64_t)(0xffffffffu - (uint32_t)e) : 0ull;
  }
  float pk[16];
  int ik[16];
  float psum = 0.f;
  for (int k = 0; k < K; ++k) {
    uint64_t best = key[0];
#pragma unroll
    for (int j = 1; j < NPL; ++j) best = key[j] > best ? key[j] : best;
#pragma unroll
    for (int o = 32; o >= 1; o >>= 1) {
      const uint32_t hi = (uint32_t)__shfl_xor((int)(uint32_t)(best >> 32), o, 64);
      const uint32_t lo = (uint32_t)__shfl_xor((int)(uint32_t)best, o, 64);
      const uint64_t other = ((uint64_t)hi << 32) | lo;
      best = other > best ? other : best;
    }
    const int bi = (int)(0xffffffffu - (uint32_t)best);
#pragma unroll
    for (int j = 0; j < NPL; ++j)
      if (bi == l + 64 * j) key[j] = 0ull;
    ik[k] = bi;
    pk[k] = __uint_as_float((uint32_t)(best >> 32));
    psum += pk[k];
  }
  if (l < K) {
    float p = 0.f;
    int i = 0;
    for (int k = 0; k < K; ++k)
      if (k == l) {
        p = pk[k];
        i = ik[k];
      }
    const float tv = p / psum;
    topv[t * K + l] = pes ? tv * pes[i] : tv;
    topi[t * K + l] = i;
    topi32[t * K + l] = i;
  }
}

// dtopv -> dlogits, one wave per token (the fp32 form of route_bwd in router.hip):
//   per-expert scale: d(renorm)_k = dtopv_k pes[i_k];  renorm: dp_k = (d_k - sum_j d_j tv_j) / S, tv_j = p_j / S;
//   softmax: dlogit_e = p_e (dp_e - sum_k dp_k p_{i_k}),  dp_e = 0 off the top-k.
__global__ __launch_bounds__(256) void route_bwd_f32_kernel(const float* __restrict__ dtopv,
                                                            const float* __restrict__ probs,
                                                            const int32_t* __restrict__ topi32,
                                                            const float* __restrict__ pes, int T, int K, int E,
                                                            float* __restrict__ dlogits) {
  const int64_t t = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6);
  if (t >= T) return;
  const int l = lane_id();
  float d = 0.f, p = 0.f;
  int idx = -1;
  if (l < K) {
    idx = topi32[t * K + l];
    if (idx >= 0 && idx < E) {
      p = probs[t * E + idx];
      d = dtopv[t * K + l];
      if (pes) d *= pes[idx];
    } else {
      idx = -1;
    }
  }
  float S = 0.f, dot = 0.f, pdp = 0.f;
  for (int k = 0; k < K; ++k) S += __shfl(p, k, 64);
  const float tv = (l < K) ? p / S : 0.f;
  for (int k = 0; k < K; ++k) dot += __shfl(d * tv, k, 64);
  const float dp = (l < K) ? (d - dot) / S : 0.f;
  for (int k = 0; k < K; ++k) pdp += __shfl(dp * p, k, 64);
  int ik[16];
  float dk[16];
#pragma unroll
  for (int k = 0; k < 16; ++k) {
    ik[k] = k < K ? __shfl(idx, k, 64) : -1;
    dk[k] = k < K ? __shfl(dp, k, 64) : 0.f;
  }
  for (int e = l; e < E; e += 64) {
    float dpe = 0.f;
#pragma unroll
    for (int k = 0; k < 16; ++k)
      if (ik[k] == e) dpe = dk[k];
    dlogits[t * E + e] = probs[t * E + e] * (dpe - pdp);
  }
}

__global__ __launch_bounds__(256) void route_prenorm_f32_kernel(const float* __restrict__ h,
                                                                const float* __restrict__ scale, int64_t H, float eps,
                                                                float hs, float* __restrict__ xn,
                                                                float* __restrict__ rstd) {
  __shared__ float red[4];
  const int64_t t = blockIdx.x;
  float ss = 0.f;
  for (int64_t j = threadIdx.x; j < H; j += 256) ss += h[t * H + j] * h[t * H + j];
  ss = block_sum(ss, red);
  const float r = 1.0f / sqrtf(ss / (float)H + eps);
  if (threadIdx.x == 0) rstd[t] = r;
  for (int64_t j = threadIdx.x; j < H; j += 256) xn[t * H + j] = ((h[t * H + j] * r) * scale[j]) * hs;
}

__global__ __launch_bounds__(256) void route_prenorm_bwd_f32_kernel(const float* __restrict__ h,
                                                                    const float* __restrict__ scale,
                                                                    const float* __restrict__ rstd,
                                                                    const float* __restrict__ dxn, int64_t H, float hs,
                                                                    float* __restrict__ dh) {
  __shared__ float red[4];
  const int64_t t = blockIdx.x;
  const float r = rstd[t];
  float dot = 0.f;
  for (int64_t j = threadIdx.x; j < H; j += 256) dot += (dxn[t * H + j] * hs) * scale[j] * h[t * H + j];
  dot = block_sum(dot, red);
  const float c = r * r * r * dot / (float)H;
  for (int64_t j = threadIdx.x; j < H; j += 256) {
    const float g = (dxn[t * H + j] * hs) * scale[j];
    dh[t * H + j] = g * r - h[t * H + j] * c;
  }
}

template <int V>
__global__ __launch_bounds__(256) void gate_mul_f32_kernel(const float* __restrict__ y, const float* __restrict__ s,
                                                           const float* __restrict__ base, int64_t H,
                                                           float* __restrict__ out) {
  const int64_t t = blockIdx.x;
  const float sg = sigmoid32(s[t]);
  for (int64_t c = V * threadIdx.x; c < H; c += 256 * V) {
    FVec<V> v = ldv<V>(y + t * H + c);
    const FVec<V> b = base ? ldv<V>(base + t * H + c) : FVec<V>{};
#pragma unroll
    for (int e = 0; e < V; ++e) v.v[e] = base ? b.v[e] + v.v[e] * sg : v.v[e] * sg;
    stv<V>(out + t * H + c, v);
  }
}

template <int V>
__global__ __launch_bounds__(256) void gate_mul_bwd_f32_kernel(const float* __restrict__ y,
                                                               const float* __restrict__ s,
                                                               const float* __restrict__ dout, int64_t H,
                                                               float* __restrict__ dy, float* __restrict__ ds) {
  __shared__ float red[4];
  const int64_t t = blockIdx.x;
  const float sg = sigmoid32(s[t]);
  float dot = 0.f;
  for (int64_t c = V * threadIdx.x; c < H; c += 256 * V) {
    FVec<V> d = ldv<V>(dout + t * H + c);
    const FVec<V> yv = ldv<V>(y + t * H + c);
#pragma unroll
    for (int e = 0; e < V; ++e) {
      dot += d.v[e] * yv.v[e];
      d.v[e] *= sg;
    }
    stv<V>(dy + t * H + c, d);
  }
  dot = block_sum(dot, red);
  if (threadIdx.x == 0) ds[t] = dot * sg * (1.0f - sg);
}

bool aligned16(const void* p) { return ((uintptr_t)p & 15u) == 0; }

}  // namespace

// ---------------------------------------------------------------------------------------------- C-ABI

extern "C" int smel_gmm_f32(const smel_wset_f32* w, int32_t trans, const int32_t* gkind, const int32_t* tiles,
                            const int32_t* n_tiles, int64_t max_tiles, const float* A, int64_t lda, float alpha,
                            float beta, float* C, int64_t ldc, hipStream_t stream) {
  SMEL_REQUIRE(w && tiles && n_tiles && A && C, SMEL_EINVAL, "smel_gmm_f32: null pointer");
  SMEL_REQUIRE(trans == 0 || trans == 1, SMEL_EINVAL, "smel_gmm_f32: trans must be 0 or 1");
  SMEL_REQUIRE(beta == 0.f || beta == 1.f, SMEL_EINVAL, "smel_gmm_f32: beta must be 0 or 1");
  SMEL_REQUIRE(w->R > 0 && w->C > 0 && max_tiles >= 0 && max_tiles < (1 << 30), SMEL_EINVAL,
               "smel_gmm_f32: bad sizes R=%lld C=%lld max_tiles=%lld", (long long)w->R, (long long)w->C,
               (long long)max_tiles);
  SMEL_REQUIRE(w->R * w->C < (1LL << 31), SMEL_EUNSUPPORTED, "smel_gmm_f32: one weight matrix of 2^31 elements or more");
  const int64_t N = trans ? w->C : w->R, K = trans ? w->R : w->C;
  SMEL_REQUIRE(lda >= K && ldc >= N, SMEL_EINVAL, "smel_gmm_f32: lda %lld < K %lld or ldc %lld < N %lld",
               (long long)lda, (long long)K, (long long)ldc, (long long)N);
  const int32_t known = (1 << SMEL_KIND_INT4) | (1 << SMEL_KIND_BF16) | (1 << SMEL_KIND_SEL) | (1 << SMEL_KIND_SHARED);
  SMEL_REQUIRE((w->kinds & ~known) == 0 && w->kinds != 0, SMEL_EINVAL, "smel_gmm_f32: bad kinds mask %d", w->kinds);
  SMEL_REQUIRE(!(w->kinds & (1 << SMEL_KIND_INT4)) ||
                   (w->q4 && w->scale && w->zero && w->group > 0 && w->group % 2 == 0 && w->C % w->group == 0),
               SMEL_EINVAL, "smel_gmm_f32: int4 tiles need q4 / scale / zero and an even group dividing C");
  SMEL_REQUIRE(!(w->kinds & (1 << SMEL_KIND_BF16)) || w->wf, SMEL_EINVAL, "smel_gmm_f32: no dense bank (wf)");
  SMEL_REQUIRE(!(w->kinds & (1 << SMEL_KIND_SEL)) || w->wsel, SMEL_EINVAL, "smel_gmm_f32: no selected weights");
  SMEL_REQUIRE(!(w->kinds & (1 << SMEL_KIND_SHARED)) || w->wsh, SMEL_EINVAL, "smel_gmm_f32: no shared weights");
  if (max_tiles == 0) return 0;
  // bit 0: A rows in 16-byte loads (32-bit offsets inside a tile); bit 1: every fp32 weight matrix too
  const int vec = (aligned16(A) && lda % 4 == 0 && K % 4 == 0 && lda < (1 << 22) ? 1 : 0) |
                  (w->C % 4 == 0 && w->R * w->C < (1 << 29) && (!w->wf || aligned16(w->wf)) && (!w->wsel || aligned16(w->wsel)) &&
                           (!w->wsh || aligned16(w->wsh))
                       ? 2
                       : 0);
  // nibbles under one scale / zero pair in one load: 2: 16 (8 bytes), 1: 4 (2 bytes), 0: 2
  const bool q16 = w->q4 && w->C % 16 == 0 && w->group % 16 == 0 && w->C * w->group < (1LL << 32) &&
                   ((uintptr_t)w->q4 & 7) == 0 && ((uintptr_t)w->scale & 1) == 0 && ((uintptr_t)w->zero & 1) == 0;
  const int qvec = q16 ? 2 : w->C % 4 == 0 && w->group % 4 == 0 && ((uintptr_t)w->q4 & 1) == 0;
  const int b1 = beta != 0.f;
  const unsigned mt = (unsigned)max_tiles;
  if (N <= 64) {   // at most one column block of the staged kernel: the whole K of a row tile in one block is the latency
    const dim3 grid(mt, 1, 4);
#define SKINNY(TR, NF) \
  gmm_f32_skinny_kernel<TR, NF><<<grid, 512, 0, stream>>>(*w, gkind, tiles, n_tiles, A, lda, vec, alpha, b1, C, ldc)
    if (trans == 0) {
      if (N <= 16) SKINNY(0, 1);
      else if (N <= 32) SKINNY(0, 2);
      else SKINNY(0, 4);
    } else {
      if (N <= 16) SKINNY(1, 1);
      else if (N <= 32) SKINNY(1, 2);
      else SKINNY(1, 4);
    }
#undef SKINNY
    return smel::launch_status();
  }
  // two 64 x 128 blocks fit a CU: below that count the quarter tiles (32 x 64) fill more of the chip, where there is more
  // than one of their k-steps of 64 to share among the waves (12 groups of 600 rows, K 16, N 512: 16 us in quarter tiles,
  // 9 in whole ones; 1021 rows, K 16, N 2048: 11 and 8)
  const int64_t wide = max_tiles * ((N + 127) / 128);
  const bool small = wide < 512 && K > 64;
  const int64_t ncol = small ? (N + 63) / 64 : (N + 127) / 128;
  const int64_t blocks = (max_tiles + 7) / 8 * 8 * ncol;
  SMEL_REQUIRE(blocks < (1LL << 31), SMEL_EUNSUPPORTED, "smel_gmm_f32: too many blocks");
  const dim3 grid((unsigned)blocks, 1, small ? 2 : 1);
  const int c2 = N % 2 == 0 && ldc % 2 == 0 && ((uintptr_t)C & 7) == 0;
  const bool q4 = w->kinds & (1 << SMEL_KIND_INT4), f32 = w->kinds & ~(1 << SMEL_KIND_INT4);
  const bool any = !(vec & 1) || (q4 && qvec != 2) || (f32 && !(vec & 2));
  const GemmArgs G{A, lda, alpha, b1, C, ldc, c2};
#define STAGED_F(TR, RB, NT, KS, FK, FORMS) \
  gmm_f32_kernel<TR, RB, NT, KS, FK, FORMS><<<grid, 256, 0, stream>>>(*w, gkind, tiles, n_tiles, vec, qvec, G)
#define STAGED(TR, RB, NT, KS, FK)                            \
  do {                                                        \
    if (any) STAGED_F(TR, RB, NT, KS, FK, FORMS_ANY);         \
    else if (q4) STAGED_F(TR, RB, NT, KS, FK, FORMS_RUNS);    \
    else STAGED_F(TR, RB, NT, KS, FK, FORMS_F32);             \
  } while (0)
  if (trans == 0) {
    if (small) STAGED(0, 32, 64, 4, 64);
    else STAGED(0, 64, 128, 1, 32);
  } else {
    if (small) STAGED(1, 32, 64, 4, 64);
    else STAGED(1, 64, 128, 1, 32);
  }
#undef STAGED
#undef STAGED_F
  return smel::launch_status();
}

extern "C" int smel_wgrad_f32(const float* X, int64_t ldx, const float* Y, int64_t ldy, const int32_t* offsets,
                              const int32_t* job_group, int32_t n_jobs, int64_t M, int64_t N, float alpha, float* C,
                              int64_t c_stride, hipStream_t stream) {
  SMEL_REQUIRE(X && Y && offsets && job_group && C, SMEL_EINVAL, "smel_wgrad_f32: null pointer");
  SMEL_REQUIRE(M > 0 && N > 0 && ldx >= M && ldy >= N && n_jobs >= 0 && n_jobs < 65536 && c_stride >= M * N,
               SMEL_EINVAL, "smel_wgrad_f32: bad sizes");
  if (n_jobs == 0) return 0;
  // the narrower side in 16-column slices, the wider one in 16-byte loads of 64 columns per block
  const bool swap = N < M;
  const int64_t ns = swap ? N : M, nb = swap ? M : N, lds_ = swap ? ldy : ldx, ldb = swap ? ldx : ldy;
  const float *S = swap ? Y : X, *B = swap ? X : Y;
  const int64_t tiles = ((ns + 15) / 16) * ((nb + 63) / 64);
  SMEL_REQUIRE(tiles < (1 << 30), SMEL_EINVAL, "smel_wgrad_f32: output too large");
  const int vec = aligned16(B) && ldb % 4 == 0;
  const dim3 grid((unsigned)tiles, (unsigned)n_jobs);
  if (swap)
    wgrad_f32_kernel<1><<<grid, 512, 0, stream>>>(S, lds_, ns, B, ldb, nb, offsets, job_group, vec, N, alpha, C, c_stride);
  else
    wgrad_f32_kernel<0><<<grid, 512, 0, stream>>>(S, lds_, ns, B, ldb, nb, offsets, job_group, vec, N, alpha, C, c_stride);
  return smel::launch_status();
}

extern "C" int smel_gather_rows_f32(const float* src, int64_t lds, const int32_t* idx, int32_t div,
                                    const int32_t* n_valid, int64_t n, int64_t cols, float* out, hipStream_t stream) {
  SMEL_REQUIRE(src && idx && out && div > 0 && n >= 0 && cols > 0 && lds >= cols && n < (1LL << 31), SMEL_EINVAL,
               "smel_gather_rows_f32: bad arguments");
  if (n == 0) return 0;
  if (cols % 4 == 0 && lds % 4 == 0 && aligned16(src) && aligned16(out))
    gather_rows_f32_kernel<4><<<(unsigned)n, 256, 0, stream>>>(src, lds, idx, div, n_valid, cols, out);
  else
    gather_rows_f32_kernel<1><<<(unsigned)n, 256, 0, stream>>>(src, lds, idx, div, n_valid, cols, out);
  return smel::launch_status();
}

extern "C" int smel_act_gate_f32(const float* h, int64_t ldh, int64_t rows, int64_t I, int32_t act, float* a,
                                 int64_t lda, hipStream_t stream) {
  SMEL_REQUIRE(h && a && rows >= 0 && I > 0 && ldh >= 2 * I && lda >= I && (act == 0 || act == 1) &&
                   rows < (1LL << 31),
               SMEL_EINVAL, "smel_act_gate_f32: bad arguments");
  if (rows == 0) return 0;
  if (I % 4 == 0 && ldh % 4 == 0 && lda % 4 == 0 && aligned16(h) && aligned16(a))
    act_gate_f32_kernel<4><<<(unsigned)rows, 256, 0, stream>>>(h, ldh, I, act, a, lda);
  else
    act_gate_f32_kernel<1><<<(unsigned)rows, 256, 0, stream>>>(h, ldh, I, act, a, lda);
  return smel::launch_status();
}

extern "C" int smel_act_gate_bwd_f32(const float* h, int64_t ldh, const float* da, int64_t ldda, int64_t rows,
                                     int64_t I, int32_t act, float* dh, int64_t lddh, hipStream_t stream) {
  SMEL_REQUIRE(h && da && dh && rows >= 0 && I > 0 && ldh >= 2 * I && ldda >= I && lddh >= 2 * I &&
                   (act == 0 || act == 1) && rows < (1LL << 31),
               SMEL_EINVAL, "smel_act_gate_bwd_f32: bad arguments");
  if (rows == 0) return 0;
  if (I % 4 == 0 && ldh % 4 == 0 && ldda % 4 == 0 && lddh % 4 == 0 && aligned16(h) && aligned16(da) && aligned16(dh))
    act_gate_bwd_f32_kernel<4><<<(unsigned)rows, 256, 0, stream>>>(h, ldh, da, ldda, I, act, dh, lddh);
  else
    act_gate_bwd_f32_kernel<1><<<(unsigned)rows, 256, 0, stream>>>(h, ldh, da, ldda, I, act, dh, lddh);
  return smel::launch_status();
}

extern "C" int smel_combine_f32(const float* ys, const float* topv, const int32_t* inv, int64_t T, int64_t K,
                                int64_t H, float* out, hipStream_t stream) {
  SMEL_REQUIRE(ys && topv && inv && out && T >= 0 && K > 0 && K <= 64 && H > 0 && T < (1LL << 31), SMEL_EINVAL,
               "smel_combine_f32: bad arguments");
  if (T == 0) return 0;
  if (H % 4 == 0 && aligned16(ys) && aligned16(out))
    combine_f32_kernel<4><<<(unsigned)T, 256, 0, stream>>>(ys, topv, inv, (int)K, H, out);
  else
    combine_f32_kernel<1><<<(unsigned)T, 256, 0, stream>>>(ys, topv, inv, (int)K, H, out);
  return smel::launch_status();
}

extern "C" int smel_combine_bwd_f32(const float* ys, const float* dout, const float* topv, const int32_t* inv,
                                    int64_t T, int64_t K, int64_t H, float* dys, float* dtopv, hipStream_t stream) {
  SMEL_REQUIRE(ys && dout && topv && inv && dys && dtopv && T >= 0 && K > 0 && K <= 64 && H > 0 && T < (1LL << 31),
               SMEL_EINVAL, "smel_combine_bwd_f32: bad arguments");
  if (T == 0) return 0;
  if (H % 4 == 0 && aligned16(ys) && aligned16(dout) && aligned16(dys))
    combine_bwd_f32_kernel<4><<<dim3((unsigned)T, (unsigned)K), 256, 0, stream>>>(ys, dout, topv, inv, (int)K, H, dys, dtopv);
  else
    combine_bwd_f32_kernel<1><<<dim3((unsigned)T, (unsigned)K), 256, 0, stream>>>(ys, dout, topv, inv, (int)K, H, dys, dtopv);
  return smel::launch_status();
}

extern "C" int smel_dx_reduce_f32(const float* dxs, const int32_t* inv, int64_t T, int64_t K, int64_t H, float* dx,
                                  hipStream_t stream) {
  SMEL_REQUIRE(dxs && inv && dx && T >= 0 && K > 0 && K <= 64 && H > 0 && T < (1LL << 31), SMEL_EINVAL,
               "smel_dx_reduce_f32: bad arguments");
  if (T == 0) return 0;
  if (H % 4 == 0 && aligned16(dxs) && aligned16(dx))
    dx_reduce_f32_kernel<4><<<(unsigned)T, 256, 0, stream>>>(dxs, inv, (int)K, H, dx);
  else
    dx_reduce_f32_kernel<1><<<(unsigned)T, 256, 0, stream>>>(dxs, inv, (int)K, H, dx);
  return smel::launch_status();
}

extern "C" int smel_route_select_f32(const float* logits, int64_t ldl, int64_t T, int64_t E, int64_t K,
                                     const float* pes, float* probs, float* topv, int64_t* topi, int32_t* topi32,
                                     hipStream_t stream) {
  SMEL_REQUIRE(logits && probs && topv && topi && topi32, SMEL_EINVAL, "smel_route_select_f32: null pointer");
  SMEL_REQUIRE(E > 0 && E <= 512, SMEL_EUNSUPPORTED, "smel_route_select_f32: E=%lld outside 1..512", (long long)E);
  SMEL_REQUIRE(K > 0 && K <= 16 && K <= E, SMEL_EUNSUPPORTED, "smel_route_select_f32: top-k %lld outside 1..16",
               (long long)K);
  SMEL_REQUIRE(T >= 0 && ldl >= E && T < (1LL << 31), SMEL_EINVAL, "smel_route_select_f32: bad sizes");
  if (T == 0) return 0;
  const unsigned grid = (unsigned)((T + 3) / 4);
  if (E <= 256)
    route_select_f32_kernel<4><<<grid, 256, 0, stream>>>(logits, ldl, (int)T, (int)E, (int)K, pes, probs, topv, topi,
                                                         topi32);
  else
    route_select_f32_kernel<8><<<grid, 256, 0, stream>>>(logits, ldl, (int)T, (int)E, (int)K, pes, probs, topv, topi,
                                                         topi32);
  return smel::launch_status();
}

extern "C" int smel_route_bwd_f32(const float* dtopv, const float* probs, const int32_t* topi32, const float* pes,
                                  int64_t T, int64_t K, int64_t E, float* dlogits, hipStream_t stream) {
  SMEL_REQUIRE(dtopv && probs && topi32 && dlogits, SMEL_EINVAL, "smel_route_bwd_f32: null pointer");
  SMEL_REQUIRE(E > 0 && K > 0 && K <= 16 && T >= 0 && T < (1LL << 31), SMEL_EINVAL, "smel_route_bwd_f32: bad sizes");
  if (T == 0) return 0;
  route_bwd_f32_kernel<<<(unsigned)((T + 3) / 4), 256, 0, stream>>>(dtopv, probs, topi32, pes, (int)T, (int)K, (int)E,
                                                                    dlogits);
  return smel::launch_status();
}

extern "C" int smel_route_prenorm_f32(const float* h, const float* scale, int64_t T, int64_t H, float eps, float hs,
                                      float* xn, float* rstd, hipStream_t stream) {
  SMEL_REQUIRE(h && scale && xn && rstd && T >= 0 && H > 0 && T < (1LL << 31), SMEL_EINVAL,
               "smel_route_prenorm_f32: bad arguments");
  if (T == 0) return 0;
  route_prenorm_f32_kernel<<<(unsigned)T, 256, 0, stream>>>(h, scale, H, eps, hs, xn, rstd);
  return smel::launch_status();
}

extern "C" int smel_route_prenorm_bwd_f32(const float* h, const float* scale, const float* rstd, const float* dxn,
                                          int64_t T, int64_t H, float hs, float* dh, hipStream_t stream) {
  SMEL_REQUIRE(h && scale && rstd && dxn && dh && T >= 0 && H > 0 && T < (1LL << 31), SMEL_EINVAL,
               "smel_route_prenorm_bwd_f32: bad arguments");
  if (T == 0) return 0;
  route_prenorm_bwd_f32_kernel<<<(unsigned)T, 256, 0, stream>>>(h, scale, rstd, dxn, H, hs, dh);
  return smel::launch_status();
}

extern "C" int smel_gate_mul_f32(const float* y, const float* s, const float* base, int64_t T, int64_t H, float* out,
                                 hipStream_t stream) {
  SMEL_REQUIRE(y && s && out && T >= 0 && H > 0 && T < (1LL << 31), SMEL_EINVAL, "smel_gate_mul_f32: bad arguments");
  if (T == 0) return 0;
  if (H % 4 == 0 && aligned16(y) && aligned16(out) && aligned16(base))
    gate_mul_f32_kernel<4><<<(unsigned)T, 256, 0, stream>>>(y, s, base, H, out);
  else
    gate_mul_f32_kernel<1><<<(unsigned)T, 256, 0, stream>>>(y, s, base, H, out);
  return smel::launch_status();
}

extern "C" int smel_gate_mul_bwd_f32(const float* y, const float* s, const float* dout, int64_t T, int64_t H,
                                     float* dy, float* ds, hipStream_t stream) {
  SMEL_REQUIRE(y && s && dout && dy && ds && T >= 0 && H > 0 && T < (1LL << 31), SMEL_EINVAL,
               "smel_gate_mul_bwd_f32: bad arguments");
  if (T == 0) return 0;
  if (H % 4 == 0 && aligned16(y) && aligned16(dout) && aligned16(dy))
    gate_mul_bwd_f32_kernel<4><<<(unsigned)T, 256, 0, stream>>>(y, s, dout, H, dy, ds);
  else
    gate_mul_bwd_f32_kernel<1><<<(unsigned)T, 256, 0, stream>>>(y, s, dout, H, dy, ds);
  return smel::launch_status();
}
