// Varlen scaled-dot-product attention over packed sequences: the reference's sparseAttention
// (src/sparse/ops/attention.ts:24-79, which runs B > 1 as a per-sample CPU round trip) and its
// dense scaledDotProductAttention (src/dense/ops/attention.ts:36-110) for B = 1.
//
//   out[n, h, :] = softmax_k(q[n, h, :] . k[m, h, :] * scale) @ v[m, h, :]
//   n in [cu_q[b], cu_q[b+1]),  m in [cu_kv[b], cu_kv[b+1]),  rows (total, H, D) row-major.
//   A sample with no keys gives zeros (attention.ts:57).
//
// A block owns 128 or 256 queries of one (sequence, head), 32 or 64 per wave, and walks the
// sequence's keys in blocks, with an online softmax (running max and sum per query).
// The scores are computed transposed, S^T = K Q^T (M = keys, N = queries), so that in the MFMA
// result layout each lane holds 16 keys of ONE query (lane l: query l % 32): the row max / sum
// need one cross-half exchange (lane l ^ 32) per step, and the output O^T = V^T P^T keeps the
// same "one query per lane" layout, so the rescale by exp(m_old - m_new) is lane-local.  P^T is
// used as the MFMA B operand straight from the score registers; the keys of each MFMA k-step are
// therefore the score layout's rows 8(j/4) + 4(l/32) + j%4.
//   bf16/f16: v_mfma_f32_32x32x16, Q^T fragments in registers, 64-key blocks of K and V row-major
//             in LDS; V^T fragments come from transposed LDS reads.
//   f32:      v_mfma_f32_32x32x2f32 (k-step = 2 dims / 2 keys; K and V row-major in LDS with
//             padded strides, no transpose needed), 32-key blocks.
// Bound: MFMA (4 * D flops per query-key pair) and the softmax's exp per pair.  Two sequences of
// 24.7 k and 39.6 k tokens, 12 x 128 bf16: 12.9-13.3 ms (1010-1040 TFLOP/s; 14.2 with one wave's
// MFMAs and softmax in turn and V transposed on its way into LDS), MFMA busy 49 % at 2.04 GHz
// (hipBLASLt's 8192^3 bf16 product: 1.32 PFLOP/s); 20 k tokens, 24 x 64 f16: 2.95 ms against 3.57;
// cross, 36 k queries x 1.3 k keys, 16 x 64 f16: 268 us against 365.

#include <type_traits>

#include "tsc_internal.h"

namespace tsc {
namespace {

typedef __bf16 bf16x8_t __attribute__((__vector_size__(8 * sizeof(__bf16))));
typedef _Float16 f16x8_t __attribute__((__vector_size__(8 * sizeof(_Float16))));
typedef float f32x16_t __attribute__((__vector_size__(16 * sizeof(float))));
typedef uint32_t u32x4_t __attribute__((ext_vector_type(4)));
typedef float f32x2_t __attribute__((ext_vector_type(2)));
typedef __bf16 bf16x2_t __attribute__((ext_vector_type(2)));
typedef _Float16 f16x2_t __attribute__((ext_vector_type(2)));

constexpr int kThreads = 256;   // f32 kernel: 4 waves
constexpr int kBQ = 128;        // f32 kernel: queries per block, 32 per wave
constexpr float kLazy = 8.f;    // log2 headroom before the running max is raised

template <typename T>
struct Mma;
template <>
struct Mma<__bf16> {
  static __device__ __forceinline__ void run(u32x4_t a, u32x4_t b, f32x16_t& c) {
    c = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8_t, a),
                                                __builtin_bit_cast(bf16x8_t, b), c, 0, 0, 0);
  }
  static __device__ __forceinline__ uint32_t pack(float lo, float hi) {  // RNE, one cvt_pk
    return __builtin_bit_cast(uint32_t, __builtin_convertvector(f32x2_t{lo, hi}, bf16x2_t));
  }
  // acc + the two packed values (v_dot2 with (1, 1)): the softmax denominator is summed over the
  // same rounded P that the second product uses.
  static __device__ __forceinline__ float add2(uint32_t packed, float acc) {
    return __builtin_amdgcn_fdot2_f32_bf16(__builtin_bit_cast(bf16x2_t, packed),
                                          __builtin_bit_cast(bf16x2_t, 0x3f803f80u), acc, false);
  }
};
template <>
struct Mma<_Float16> {
  static __device__ __forceinline__ void run(u32x4_t a, u32x4_t b, f32x16_t& c) {
    c = __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(f16x8_t, a),
                                               __builtin_bit_cast(f16x8_t, b), c, 0, 0, 0);
  }
  static __device__ __forceinline__ uint32_t pack(float lo, float hi) {
    return __builtin_bit_cast(uint32_t, __builtin_convertvector(f32x2_t{lo, hi}, f16x2_t));
  }
  static __device__ __forceinline__ float add2(uint32_t packed, float acc) {
    return __builtin_amdgcn_fdot2(__builtin_bit_cast(f16x2_t, packed),
                                  __builtin_bit_cast(f16x2_t, 0x3c003c00u), acc, false);
  }
};

__device__ __forceinline__ float fast_exp2(float x) { return __builtin_amdgcn_exp2f(x); }

// Max / sum of a value and the one held by lane l ^ 32 (both halves of the wave hold the same
// query): v_permlane32_swap exchanges the wave halves in registers (no LDS round trip).
__device__ __forceinline__ float pair_max(float x) {
  const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(x), false, false);
  return fmaxf(__uint_as_float(r[0]), __uint_as_float(r[1]));
}
__device__ __forceinline__ float pair_sum(float x) {
  const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(x), false, false);
  return __uint_as_float(r[0]) + __uint_as_float(r[1]);
}

// Segment b's [begin, end) clamped into [0, total] (a malformed cu_seqlens cannot index outside).
__device__ __forceinline__ void segment(const int32_t* cu, int b, int64_t total, int* begin,
                                        int* len) {
  const int64_t s = min<int64_t>(max<int64_t>(cu[b], 0), total);
  const int64_t e = min<int64_t>(max<int64_t>(cu[b + 1], s), total);
  *begin = (int)s;
  *len = (int)(e - s);
}

// Block -> (q tile, head, sequence).  Blocks start in the order of their index and go to the 8 XCDs
// round robin.  Every XCD gets the same share of every sequence, whatever the sequences' lengths:
// of each eight heads XCD x takes one, so that a head's K and V come into one L2 only, and the q
// tiles of the heads past a multiple of eight are spread over all XCDs.  (Contiguous runs of
// blocks per XCD left the XCDs of the short sequences idle: 21.1 ms against 14.2 ms for sequences
// of 24.7 k and 39.6 k tokens, 12 x 128 bf16, MFMAs and softmax still in turn.)
// Sequences with more keys go first, so that the launch ends on its shortest blocks; past
// kMaxRanked sequences the ranking would cost more than the tail it saves, and they keep their
// order.
constexpr int kMaxRanked = 8;

__device__ __forceinline__ void block_tile(const int32_t* cu_kv, int* bx, int* bh, int* bb) {
  const int gx = gridDim.x, H = gridDim.y, B = gridDim.z;
  const int per_seq = gx * H;
  const int lin = blockIdx.x + gx * (blockIdx.y + H * blockIdx.z);
  const int slot = blockIdx.z, u = lin - slot * per_seq;
  const int whole = H & ~7;  // heads dealt one per XCD
  if (u < gx * whole) {      // a run of eight blocks holds every XCD once, so (u / 8, lin % 8) is
    const int i = u >> 3;    // another numbering of the same blocks
    *bx = i % gx;
    *bh = (i / gx) * 8 + (lin & 7);
  } else {
    *bx = blockIdx.x;
    *bh = blockIdx.y;
  }
  int seq = slot;
  if (B > 1 && B <= kMaxRanked) {  // lane 8 b + c: does sequence c come before sequence b?
    const int lane = threadIdx.x & 63, b = min(lane >> 3, B - 1), c = min(lane & 7, B - 1);
    const uint32_t len = (uint32_t)cu_kv[b + 1] - (uint32_t)cu_kv[b];
    const uint32_t other = (uint32_t)cu_kv[c + 1] - (uint32_t)cu_kv[c];
    const bool before = (lane & 7) < B && (other > len || (other == len && c < b));
    const uint64_t all = __builtin_amdgcn_ballot_w64(before);
    const bool mine = lane < B && __popc((uint32_t)(all >> (8 * (lane & 7))) & 0xffu) == slot;
    seq = __builtin_ctzll(__builtin_amdgcn_ballot_w64(mine));  // exactly one lane
  }
  *bb = seq;
}

// ---------------------------------------------------------------------------------- bf16 / f16
// LDS tile of 64 rows of K or V, row-major, 16-byte chunks XOR-swizzled by row.  K: the 16 (or 8)
// rows of one read step, one chunk column, fall into distinct bank groups.  V: a transposed read
// (ds_read_b64_tr_b16) takes 32 bytes of each of 4 consecutive rows per 16 lanes; their chunk
// pairs are spread the same way.
template <int D>
__device__ __forceinline__ int kswz(int row) {
  return D == 128 ? (row & 15) : (((row >> 1) & 7) ^ ((row & 1) << 2));
}
template <int D>
__device__ __forceinline__ int vswz(int row) {
  const int r = row & 3;
  return (D == 128 ? (r << 1) ^ (r & 1) ^ ((r >> 1) & 1) : r) << 1;
}

typedef short s16x4_t __attribute__((ext_vector_type(4)));
// Lane i of each 16 gets column i of the 4 rows x 16 columns whose row r the lanes 4r..4r+3
// address (8 bytes each).
__device__ __forceinline__ uint2 lds_read_tr(const unsigned char* p) {
#if defined(__HIP_DEVICE_COMPILE__)
  return __builtin_bit_cast(
      uint2, __builtin_amdgcn_ds_read_tr16_b64_v4i16(
                 (__attribute__((address_space(3))) s16x4_t*)(__attribute__((address_space(3))) void*)p));
#else
  return make_uint2(0, 0);
#endif
}

typedef uint32_t u32x4_t __attribute__((ext_vector_type(4)));
// NW waves of QT 32-query tiles.  The MFMAs and the softmax of one wave overlap: a step multiplies
// the next 32 keys' scores while the current ones are exponentiated (phase A), then adds its V
// while the next row max is taken (phase B), in a fixed interleaving; with one softmax after the
// other the two pipes took turns even with two waves per SIMD.  Two waves per SIMD are kept: one
// wave alone issues an instruction every 5-6 cycles, and 64 queries per wave with 512 registers
// (half the LDS reads) measured the same time.
template <typename T, int D, int QT, int NW>
__global__ void __launch_bounds__(64 * NW, 2)
    attn_mma_kernel(const T* __restrict__ q, const T* __restrict__ k, const T* __restrict__ v,
                    const int32_t* __restrict__ cu_q, const int32_t* __restrict__ cu_kv,
                    int64_t total_q, int64_t total_kv, int32_t H, float scale_log2,
                    T* __restrict__ out) {
  constexpr int BK = 64;                     // keys per staged block: two steps of 32
  constexpr int DC = D / 8;                  // 16-byte chunks per row
  constexpr int KS = D / 16;                 // k-steps of S^T = K Q^T
  constexpr int MT = D / 32;                 // 32-dim tiles of O^T
  constexpr int NT = 64 * NW;
  constexpr int RI = NT / DC;       // rows one load instruction of the block covers
  constexpr int NL = BK / RI;                // K (and V) chunks each thread stages per block
  constexpr int ROWB = D * 2;                // bytes per row
  constexpr int NA = KS * QT, NB = 2 * MT * QT;  // MFMAs of the two phases
  constexpr int BQ = 32 * NW * QT;             // queries per block
  static_assert(NL >= 1 && (D == 64 || D == 128), "tile shape");
  __shared__ __attribute__((aligned(16))) unsigned char kbuf[2][BK * ROWB];
  __shared__ __attribute__((aligned(16))) unsigned char vbuf[2][BK * ROWB];

  int bx, h, bb;
  block_tile(cu_kv, &bx, &h, &bb);
  int q0, q_len, kv0, kv_len;
  segment(cu_q, bb, total_q, &q0, &q_len);
  segment(cu_kv, bb, total_kv, &kv0, &kv_len);
  const int64_t rs = (int64_t)H * D;
  const T* kbase = k + (int64_t)kv0 * rs + (int64_t)h * D;
  const T* vbase = v + (int64_t)kv0 * rs + (int64_t)h * D;

  for (int qt = bx * BQ; qt < q_len; qt += gridDim.x * BQ) {
    int tid = threadIdx.x;
    asm volatile("" : "+v"(tid));  // nothing derived from it is kept across q tiles
    const int lane = tid & 63, w = tid >> 6, l32 = lane & 31, hf = lane >> 5;
    // Staging: thread (srow, sc) copies chunk sc of rows srow + RI * i.
    const int srow = tid / DC, sc = tid % DC;
    const int kdst = srow * ROWB + (sc ^ kswz<D>(srow)) * 16;
    const int vdst = srow * ROWB + (sc ^ vswz<D>(srow)) * 16;
    const uint32_t rsb = (uint32_t)rs * 2u;  // row bytes
    const uint32_t soff = (uint32_t)srow * rsb + 16u * sc, sstep = RI * rsb;
    // Fragment addresses: K chunk 2 st + hf of row l32 is kfrag ^ (st * 32); V^T's 4-row x 16-column
    // piece of dim tile mt is vfrag ^ (mt * 64), rows 16 half + 8 x + 4 hf + (lane % 16) / 4.
    const int kfrag = l32 * ROWB + ((hf ^ kswz<D>(l32)) << 4);
    const int vr = (lane & 15) >> 2;
    const int vfrag = (4 * hf + vr) * ROWB +
                      (((2 * ((lane >> 4) & 1) + ((lane & 3) >> 1)) ^ vswz<D>(vr)) << 4) + (lane & 1) * 8;

    const int qb = qt + w * 32 * QT + l32;  // this lane's query of q tile 0
    if (kv_len == 0) {  // no keys: zeros (uniform over the block)
#pragma unroll
      for (int i = 0; i < QT; ++i)
        if (qb + 32 * i < q_len) {
          T* orow = out + (int64_t)(q0 + qb + 32 * i) * rs + (int64_t)h * D;
          for (int c = hf; c < DC; c += 2) *(uint4*)(orow + 8 * c) = make_uint4(0, 0, 0, 0);
        }
      continue;
    }
    u32x4_t qf[QT][KS];  // Q^T fragments: lane (query l32, half hf) holds dims 16 st + 8 hf .. + 7
#pragma unroll
    for (int i = 0; i < QT; ++i) {
      const T* qrow = q + (int64_t)(q0 + min(qb + 32 * i, q_len - 1)) * rs + (int64_t)h * D + 8 * hf;
#pragma unroll
      for (int st = 0; st < KS; ++st) qf[i][st] = *(const u32x4_t*)(qrow + 16 * st);
    }
    // Block kb's rows; rows past the last key repeat it, a block past the end is block 0.  The scores
    // of such keys are masked, and their V is stored as zeros (P is zero there, but zero times an
    // infinity in a repeated row is not).
    u32x4_t kr[NL], vreg[NL];
    auto load = [&](const T* base, int kb, u32x4_t(&r)[NL]) {
      if (kb >= kv_len) kb = 0;
      const char* p = (const char*)(base + (int64_t)kb * rs);
      const uint32_t lim = (uint32_t)min(kv_len - 1 - kb, BK - 1) * rsb + 16u * sc;
#pragma unroll
      for (int i = 0; i < NL; ++i) r[i] = *(const u32x4_t*)(p + min(soff + i * sstep, lim));
    };
    auto store = [&](int vb, int kb, auto masked, int v0) {  // v0: first key of the V block
#pragma unroll
      for (int i = 0; i < NL; ++i) {
        if (decltype(masked)::value && v0 + srow + RI * i >= kv_len) vreg[i] = u32x4_t{0, 0, 0, 0};
        *(u32x4_t*)(&vbuf[vb][vdst] + i * RI * ROWB) = vreg[i];
      }
#pragma unroll
      for (int i = 0; i < NL; ++i) *(u32x4_t*)(&kbuf[kb][kdst] + i * RI * ROWB) = kr[i];
    };

    constexpr std::true_type Y{};
    constexpr std::false_type N{};
    float m_use[QT], mc[QT], l_run[QT], alpha[QT];  // mc = m_use * scale_log2
    f32x16_t o[QT][MT], sa[QT], sb[QT];
#pragma unroll
    for (int i = 0; i < QT; ++i) {
      m_use[i] = mc[i] = -INFINITY;
      l_run[i] = 0.f;
#pragma unroll
      for (int mt = 0; mt < MT; ++mt)
#pragma unroll
        for (int j = 0; j < 16; ++j) o[i][mt][j] = 0.f;
    }
    u32x4_t kf[KS];       // K fragments of the next score product
    uint2 vf[2][MT][2];   // V^T fragments of the current step
    u32x4_t pf[QT][2];     // P^T of the current step

    auto read_k = [&](int buf, int half, int st) {
      kf[st] = *(const u32x4_t*)(&kbuf[buf][0] + ((kfrag ^ (st * 32)) + half * 32 * ROWB));
    };
    auto read_v = [&](int buf, int half, int n) {  // n-th of 4 MT reads, in the order of use
      const int g = n / (2 * MT), mt = (n / 2) % MT, x = n % 2;
      vf[g][mt][x] = lds_read_tr(&vbuf[buf][0] + ((vfrag ^ (mt * 64)) + (half * 32 + 16 * g + 8 * x) * ROWB));
    };
    // Score j of q tile i of the step from key k0 on; -inf past the last key in masked steps.
    auto score = [&](const f32x16_t(&s)[QT], int i, int j, auto masked, int k0) {
      return decltype(masked)::value && k0 + 8 * (j >> 2) + 4 * hf + (j & 3) >= kv_len ? -INFINITY
                                                                                        : s[i][j];
    };
    float pr[16 * QT];  // probabilities, before rounding
    // e-th of the step's 16 QT scores -> probability.
    auto exp_one = [&](const f32x16_t(&s)[QT], int e, auto masked, int k0) {
      pr[e] = fast_exp2(fmaf(score(s, e / 16, e % 16, masked, k0), scale_log2, -mc[e / 16]));
    };
    // n-th of the step's 8 QT pairs -> rounded P and the denominator.
    auto pack_one = [&](int n) {
      const int i = n / 8, e = 2 * (n % 8);
      const uint32_t p = Mma<T>::pack(pr[2 * n], pr[2 * n + 1]);
      pf[i][e / 8][(e / 2) % 4] = p;
      l_run[i] = Mma<T>::add2(p, l_run[i]);
    };
    auto max_part = [&](const f32x16_t(&s)[QT], int i, int part, float mx, auto masked, int k0) {
#pragma unroll
      for (int j = 4 * part; j < 4 * part + 4; ++j) mx = fmaxf(mx, score(s, i, j, masked, k0));
      return mx;
    };
    // Raises the running maxima of q tile i if a score exceeds one by more than 2^kLazy: alpha is what the
    // accumulators have to be multiplied with.
    auto raise = [&](int i, float mx) {
      const bool up = __builtin_amdgcn_ballot_w64(mx * scale_log2 > mc[i] + kLazy) != 0;
      if (up) {
        const float m_new = fmaxf(m_use[i], mx);
        alpha[i] = fast_exp2((m_use[i] - m_new) * scale_log2);  // 0 while m_use = -inf
        m_use[i] = m_new;
        mc[i] = m_new * scale_log2;
      }
      return up;
    };
    auto rescale = [&](int i) {
      l_run[i] *= alpha[i];
#pragma unroll
      for (int mt = 0; mt < MT; ++mt)
#pragma unroll
        for (int j = 0; j < 16; ++j) o[i][mt][j] *= alpha[i];
    };
    auto pv = [&](int m) {  // m-th of the step's NB products O^T += V^T P^T
      const int g = m / (MT * QT), mt = (m / QT) % MT, i = m % QT;
      Mma<T>::run(u32x4_t{vf[g][mt][0].x, vf[g][mt][0].y, vf[g][mt][1].x, vf[g][mt][1].y}, pf[i][g],
                  o[i][mt]);
    };
    // One step of 32 keys whose scores are in cur, the first half of them already exponentiated.
    //   A  next scores (MFMA) beside the rest of this step's softmax (VALU) and its V^T reads
    //   B  O^T += V^T P^T beside the next step's row max, the first half of its exponentials and
    //      the K reads of the step after
    // The groups are pinned in program order: left to itself the compiler gathers the MFMAs.
    auto step = [&](f32x16_t(&cur)[QT], f32x16_t(&nxt)[QT], int vb, int vhalf, int kb, int khalf,
                    auto masked, int k0, auto stage) {
      constexpr int EA = 8 * QT / NA > 0 ? 8 * QT / NA : 1;      // exponentials per A group
      constexpr int PA = (8 * QT + NA - 1) / NA;                 // pairs packed per A group
      constexpr int VA = (4 * MT + NA - 1) / NA;                 // V reads per A group
#pragma unroll
      for (int m = 0; m < NA; ++m) {
        const int st = m / QT, i = m % QT;
        if (st == 0) {
#pragma unroll
          for (int j = 0; j < 16; ++j) nxt[i][j] = 0.f;
        }
        Mma<T>::run(kf[st], qf[i][st], nxt[i]);
#pragma unroll
        for (int n = 0; n < VA; ++n)
          if (m * VA + n < 4 * MT) read_v(vb, vhalf, m * VA + n);
#pragma unroll
        for (int n = 0; n < EA; ++n)
          if (m * EA + n < 8 * QT) exp_one(cur, 8 * QT + m * EA + n, masked, k0);
#pragma unroll
        for (int n = 0; n < PA; ++n)  // the pairs of the two halves in turn
          if (m * PA + n < 8 * QT) pack_one((m * PA + n) / 2 + (m * PA + n) % 2 * 4 * QT);
        __builtin_amdgcn_sched_barrier(0);
      }
      constexpr int KB = (KS + NB - 1) / NB;      // K reads per B group
      constexpr int M0 = (NB + 7) / 8;               // groups before the row max (MFMA latency)
      constexpr int MG = NB / 4;                  // groups of the row max
      constexpr int E0 = M0 + MG;                 // first group with exponentials
      constexpr int EB = (8 * QT + NB - E0 - 1) / (NB - E0);
      float mx[QT];
      auto b_common = [&](int m) {
        pv(m);
#pragma unroll
        for (int n = 0; n < KB; ++n)
          if (m * KB + n < KS) read_k(kb, khalf, m * KB + n);
      };
#pragma unroll
      for (int m = 0; m < M0; ++m) {
        b_common(m);
        __builtin_amdgcn_sched_barrier(0);
      }
#pragma unroll
      for (int i = 0; i < QT; ++i) mx[i] = score(nxt, i, 0, masked, k0 + 32);
#pragma unroll
      for (int m = M0; m < E0; ++m) {
        b_common(m);
#pragma unroll
        for (int n = (m - M0) * 4 * QT / MG; n < (m - M0 + 1) * 4 * QT / MG; ++n)
          mx[n / 4] = max_part(nxt, n / 4, n % 4, mx[n / 4], masked, k0 + 32);
        __builtin_amdgcn_sched_barrier(0);
      }
#pragma unroll
      for (int i = 0; i < QT; ++i) mx[i] = pair_max(mx[i]);
      bool up[QT];
#pragma unroll
      for (int i = 0; i < QT; ++i) up[i] = raise(i, mx[i]);
#pragma unroll
      for (int m = E0; m < NB; ++m) {
        b_common(m);
#pragma unroll
        for (int n = 0; n < EB; ++n)
          if ((m - E0) * EB + n < 8 * QT) exp_one(nxt, (m - E0) * EB + n, masked, k0 + 32);
        if (decltype(stage)::value && m == NB - NB / 4) store(kb, kb ^ 1, masked, k0 + 32);
        __builtin_amdgcn_sched_barrier(0);
      }
#pragma unroll
      for (int i = 0; i < QT; ++i)
        if (up[i]) rescale(i);
    };
    {
      u32x4_t k1[NL];
      load(kbase, 0, kr);
      load(vbase, 0, vreg);
      load(kbase, BK, k1);
      store(0, 0, Y, 0);
#pragma unroll
      for (int i = 0; i < NL; ++i) kr[i] = k1[i];
      store(0, 1, Y, 0);
    }
    __syncthreads();
#pragma unroll
    for (int st = 0; st < KS; ++st) read_k(0, 0, st);
#pragma unroll
    for (int i = 0; i < QT; ++i) {
#pragma unroll
      for (int j = 0; j < 16; ++j) sa[i][j] = 0.f;
#pragma unroll
      for (int st = 0; st < KS; ++st) Mma<T>::run(kf[st], qf[i][st], sa[i]);
    }
#pragma unroll
    for (int st = 0; st < KS; ++st) read_k(0, 1, st);
#pragma unroll
    for (int i = 0; i < QT; ++i) {
      float mx = -INFINITY;
#pragma unroll
      for (int part = 0; part < 4; ++part) mx = max_part(sa, i, part, mx, Y, 0);
      raise(i, pair_max(mx));  // the accumulators are still zero
    }
#pragma unroll
    for (int e = 0; e < 8 * QT; ++e) exp_one(sa, e, Y, 0);
    __syncthreads();  // block 0's K has been read by every wave: kbuf[0] may be refilled
    // Block jb: its V and the next block's K are in LDS; meanwhile the V of the next block and the
    // K of the one after come in through registers, into the buffers that the block before used.
    int jb = 0;
    auto block = [&](auto masked) {
      const int b = jb & 1, kb = jb * BK;
      load(vbase, kb + BK, vreg);
      load(kbase, kb + 2 * BK, kr);
      step(sa, sb, b, 0, b ^ 1, 0, masked, kb, N);
      step(sb, sa, b, 1, b ^ 1, 1, masked, kb + 32, Y);
      __syncthreads();
    };
    // Blocks all of whose scores, and the next block's first, are of keys that exist; then the
    // others, masked.
    const int nfull = max(0, kv_len / BK - 1), nblk = (kv_len + BK - 1) / BK;
    for (; jb < nfull; ++jb) block(N);
    for (; jb < nblk; ++jb) block(Y);
#pragma unroll
    for (int i = 0; i < QT; ++i) {
      const float inv = 1.f / pair_sum(l_run[i]);
      const int qi = qb + 32 * i;
      if (qi < q_len) {
        T* orow = out + (int64_t)(q0 + qi) * rs + (int64_t)h * D;
#pragma unroll
        for (int mt = 0; mt < MT; ++mt)
#pragma unroll
          for (int g = 0; g < 4; ++g)
            *(uint2*)(orow + 32 * mt + 8 * g + 4 * hf) =
                make_uint2(Mma<T>::pack(o[i][mt][4 * g] * inv, o[i][mt][4 * g + 1] * inv),
                           Mma<T>::pack(o[i][mt][4 * g + 2] * inv, o[i][mt][4 * g + 3] * inv));
      }
    }
    __syncthreads();  // the next q tile of this block stages over these buffers
  }
}

// ---------------------------------------------------------------------------------- f32
// W waves per SIMD.  Two, at D = 128 for 44 spilled registers (180 bytes a lane): one wave's softmax
// then runs beside the other's MFMAs.  5.8 k and 9.3 k tokens, 12 x 128: 6.26 ms (118 TFLOP/s of
// the 154 that a large fp32 product reaches; 6.92 with one wave, 7.47 with it and a rescale and the
// mask in every block).  D = 128 takes one where the spills show and the second wave does not
// (attention_launch).
template <int D, int W>
__global__ void __launch_bounds__(kThreads, W)
    attn_f32_kernel(const float* __restrict__ q, const float* __restrict__ k,
                    const float* __restrict__ v, const int32_t* __restrict__ cu_q,
                    const int32_t* __restrict__ cu_kv, int64_t total_q, int64_t total_kv,
                    int32_t H, float scale_log2, float* __restrict__ out) {
  constexpr int BK = 32;
  constexpr int KST = D + 2;  // K row stride: lanes (key, half) read 64 distinct banks
  constexpr int VST = D + 8;  // V row stride: rows 4 apart land 32 banks apart
  constexpr int MT = D / 32;
  constexpr int NC = BK * D / 4;               // float4 chunks per K (or V) block
  constexpr int CL = NC / kThreads;            // chunks each thread stages
  static_assert(CL >= 1 && (D == 64 || D == 128), "tile shape");
  __shared__ __attribute__((aligned(16))) float ks[2][BK * KST];
  __shared__ __attribute__((aligned(16))) float vs[2][BK * VST];

  int bx, h, bb;
  block_tile(cu_kv, &bx, &h, &bb);
  int q0, q_len, kv0, kv_len;
  segment(cu_q, bb, total_q, &q0, &q_len);
  segment(cu_kv, bb, total_kv, &kv0, &kv_len);
  const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6, l32 = lane & 31, hf = lane >> 5;
  const int64_t rs = (int64_t)H * D;
  const float* kbase = k + (int64_t)kv0 * rs + (int64_t)h * D;
  const float* vbase = v + (int64_t)kv0 * rs + (int64_t)h * D;

  for (int qt = bx * kBQ; qt < q_len; qt += gridDim.x * kBQ) {
    const int qi = qt + w * 32 + l32;
    float* orow = out + (int64_t)(q0 + qi) * rs + (int64_t)h * D;
    if (kv_len == 0) {
      if (qi < q_len)
        for (int c = hf; c < D / 4; c += 2) *(float4*)(orow + 4 * c) = make_float4(0, 0, 0, 0);
      continue;
    }
    float qf[D / 2];  // B operand of step st: dim 2st + hf of this lane's query
    {
      const float* qrow = q + (int64_t)(q0 + min(qi, q_len - 1)) * rs + (int64_t)h * D;
#pragma unroll
      for (int c = 0; c < D / 4; ++c) {
        const float4 x = *(const float4*)(qrow + 4 * c);
        qf[2 * c] = hf ? x.y : x.x;
        qf[2 * c + 1] = hf ? x.w : x.z;
      }
    }
    float4 kr[CL], vr[CL];
    auto load = [&](int kb) {
#pragma unroll
      for (int i = 0; i < CL; ++i) {
        const int id = tid + kThreads * i, row = id / (D / 4), c = id % (D / 4);
        const bool ok = kb + row < kv_len;
        const int64_t off = (int64_t)(kb + row) * rs + 4 * c;
        kr[i] = ok ? *(const float4*)(kbase + off) : make_float4(0, 0, 0, 0);
        vr[i] = ok ? *(const float4*)(vbase + off) : make_float4(0, 0, 0, 0);
      }
    };
    auto store = [&](int buf) {
#pragma unroll
      for (int i = 0; i < CL; ++i) {
        const int id = tid + kThreads * i, row = id / (D / 4), c = id % (D / 4);
        float2* kd = (float2*)&ks[buf][row * KST + 4 * c];
        kd[0] = make_float2(kr[i].x, kr[i].y);
        kd[1] = make_float2(kr[i].z, kr[i].w);
        *(float4*)&vs[buf][row * VST + 4 * c] = vr[i];
      }
    };

    float m_run = -INFINITY, mc = -INFINITY, l_run = 0.f;  // mc = m_run * scale_log2
    f32x16_t o[MT];
#pragma unroll
    for (int mt = 0; mt < MT; ++mt)
#pragma unroll
      for (int j = 0; j < 16; ++j) o[mt][j] = 0.f;
    const int nblk = (kv_len + BK - 1) / BK;
    load(0);
    store(0);
    __syncthreads();
    // Only the last block can hold keys past the end.
    auto block = [&](int jb, auto masked) {
      const int buf = jb & 1, kb = jb * BK;
      const bool more = jb + 1 < nblk;
      if (more) load(kb + BK);
      f32x16_t s0, s1;  // two accumulation chains over the dims
#pragma unroll
      for (int j = 0; j < 16; ++j) s0[j] = s1[j] = 0.f;
      const float* krow = &ks[buf][l32 * KST + hf];
#pragma unroll
      for (int st = 0; st < D / 2; st += 2) {
        s0 = __builtin_amdgcn_mfma_f32_32x32x2f32(krow[2 * st], qf[st], s0, 0, 0, 0);
        s1 = __builtin_amdgcn_mfma_f32_32x32x2f32(krow[2 * st + 2], qf[st + 1], s1, 0, 0, 0);
      }
      float s[16];
#pragma unroll
      for (int j = 0; j < 16; ++j) {
        s[j] = s0[j] + s1[j];
        if (decltype(masked)::value && kb + 8 * (j >> 2) + 4 * hf + (j & 3) >= kv_len)
          s[j] = -INFINITY;
      }
      // What was summed is rescaled only when the maximum of some query of the wave moves.  No
      // headroom as in the 16-bit kernels: a probability stays at most 1, or large values of v
      // (past 2^120) would make a sum infinite that is not.
      float mx = s[0];
#pragma unroll
      for (int j = 1; j < 16; ++j) mx = fmaxf(mx, s[j]);
      mx = pair_max(mx);
      if (__builtin_amdgcn_ballot_w64(mx > m_run) != 0) {
        const float m_new = fmaxf(m_run, mx);
        const float alpha = fast_exp2((m_run - m_new) * scale_log2);  // 0 while m_run = -inf
        m_run = m_new;
        mc = m_new * scale_log2;
        l_run *= alpha;
#pragma unroll
        for (int mt = 0; mt < MT; ++mt)
#pragma unroll
          for (int j = 0; j < 16; ++j) o[mt][j] *= alpha;
      }
#pragma unroll
      for (int j = 0; j < 16; ++j) {
        s[j] = fast_exp2(fmaf(s[j], scale_log2, -mc));
        l_run += s[j];
      }
#pragma unroll
      for (int j = 0; j < 16; ++j) {
        const float* vrow = &vs[buf][(8 * (j >> 2) + 4 * hf + (j & 3)) * VST + l32];
#pragma unroll
        for (int mt = 0; mt < MT; ++mt)
          o[mt] = __builtin_amdgcn_mfma_f32_32x32x2f32(vrow[32 * mt], s[j], o[mt], 0, 0, 0);
      }
      if (more) store(buf ^ 1);
      __syncthreads();
    };
    for (int jb = 0; jb + 1 < nblk; ++jb) block(jb, std::false_type());
    block(nblk - 1, std::true_type());
    l_run = pair_sum(l_run);
    const float inv = 1.f / l_run;
    if (qi < q_len) {
#pragma unroll
      for (int mt = 0; mt < MT; ++mt)
#pragma unroll
        for (int g = 0; g < 4; ++g)
          *(float4*)(orow + 32 * mt + 8 * g + 4 * hf) =
              make_float4(o[mt][4 * g] * inv, o[mt][4 * g + 1] * inv, o[mt][4 * g + 2] * inv,
                          o[mt][4 * g + 3] * inv);
    }
  }
}

}  // namespace

int attention_launch(tsc_ctx* ctx, int32_t dtype, const void* q, const void* k, const void* v,
                     const int32_t* cu_q, const int32_t* cu_kv, int32_t B, int64_t total_q,
                     int64_t total_kv, int32_t H, int32_t D, float scale, int32_t max_seqlen_q,
                     void* out) {
  if (B == 0 || total_q == 0 || max_seqlen_q == 0) return TSC_OK;
  const float sl2 = scale * 1.4426950408889634f;  // scale * log2(e): softmax in base 2
  const int64_t hb = (int64_t)H * B;  // the block index arithmetic is 32-bit
  if (hb > (int64_t)(INT32_MAX / 16))
    return fail(TSC_ERR_UNSUPPORTED, "attention: %lld (head, sequence) pairs", (long long)hb);
  // Queries per block.  fp32: 128.  bf16 / f16: 256 (D = 64: four waves of 64, so that every K and V
  // fragment read from LDS serves two q tiles; D = 128: eight waves of 32, the accumulators of 64
  // would leave one wave per SIMD), or four waves of 32 = 128 where too few blocks of 256 come
  // together.  us, blocks of 256 / 128:
  //   D = 64, whose blocks share a CU in pairs: 256 from 1.5 blocks of it per CU on.  24 heads, two
  //     sequences of 2.5 k queries (264 blocks of 256) 52 / 46, of 4 k (408) 79 / 88.
  //   D = 128: 128 while every one of those has a CU of its own: 12 heads, 2.5 k queries (240 blocks
  //     of 128) 79 / 64, 3 k (288) 91 / 104; 12 heads, four sequences, 3 k queries on 900 keys each
  //     40 / 45.  And, below one block of 256 per CU, self-attention over uneven sequences of 700
  //     and more, whose blocks take as long as their sequence is: the shorter ones fill in.  12
  //     heads, four of 4 k in all 63 / 56, two of 5 k 136 / 120, eight of 3 k 29 / 32; 8 heads,
  //     three of 430 to 1283 47 / 38.  Up to 160
  //     keys a sequence the prologue decides, and half as many waves stage its first blocks in
  //     twice the time: four of 500 in all 14.9 / 15.8.
  const int64_t tiles = std::min<int64_t>(B * (((int64_t)max_seqlen_q + 255) / 256),
                                          (total_q + 255) / 256 + B / 2);
  const bool each_a_cu = (((int64_t)max_seqlen_q + 127) / 128) * hb <= 256;
  const bool uneven = total_kv == total_q && total_q >= 700 * (int64_t)B &&
                      6 * B * (int64_t)max_seqlen_q >= 7 * total_q;
  const bool wide = D == 64 ? tiles * H >= 384
                            : total_kv <= 160 * (int64_t)B ||
                                  (!each_a_cu && (tiles * H >= 256 || !uneven));
  const int bq = dtype == TSC_F32 ? kBQ : wide ? 256 : 128;
  // q tiles beyond the grid's x extent are covered by the kernels' tile loops
  const unsigned gx = (unsigned)std::min<int64_t>(
      std::min<int64_t>((max_seqlen_q + bq - 1) / bq, 65535), (INT32_MAX / 16) / hb);
  const dim3 grid(gx, (unsigned)H, (unsigned)B);
  ProfScope p(ctx, "attention");
  auto mma = [&](auto t, auto d, auto qt, auto nw) {
    constexpr int QT = decltype(qt)::value, NW = decltype(nw)::value;
    attn_mma_kernel<decltype(t), decltype(d)::value, QT, NW><<<grid, 64 * NW, 0, ctx->stream>>>(
        (const decltype(t)*)q, (const decltype(t)*)k, (const decltype(t)*)v, cu_q, cu_kv, total_q,
        total_kv, H, sl2, (decltype(t)*)out);
  };
  constexpr std::integral_constant<int, 1> I1{};
  constexpr std::integral_constant<int, 2> I2{};
  constexpr std::integral_constant<int, 4> I4{};
  constexpr std::integral_constant<int, 8> I8{};
  constexpr std::integral_constant<int, 64> D64{};
  constexpr std::integral_constant<int, 128> D128{};
  auto by_size = [&](auto t) {
    if (D == 64) wide ? mma(t, D64, I2, I4) : mma(t, D64, I1, I4);
    else wide ? mma(t, D128, I1, I8) : mma(t, D128, I1, I4);
  };
  if (dtype == TSC_BF16) {
    by_size(__bf16());
  } else if (dtype == TSC_F16) {
    by_size(_Float16());
  } else {
    auto f32 = [&](auto d, auto w) {
      attn_f32_kernel<decltype(d)::value, decltype(w)::value><<<grid, kThreads, 0, ctx->stream>>>(
          (const float*)q, (const float*)k, (const float*)v, cu_q, cu_kv, total_q, total_kv, H,
          sl2, (float*)out);
    };
    // D = 128, one wave per SIMD and so one block per CU, or two.  us, 12 heads, one / two:
    //   up to 80 keys a sequence the spills are most of it: 8 x 700 queries on 64 keys 69 / 77,
    //     5 k on 77 52.4 / 52.2;
    //   a grid that gives no CU a second block: 2 x 700 on 258 keys 50 / 55, on 500 78 / 84; from
    //     there on they are alike (8 x 50 on 900 165 / 170, 50 on 900 118 / 115);
    //   one of 2.35 to 3 blocks per CU, which the pairs take two rounds for as well, on not many
    //     keys: 8 x 700 on 258 147 / 160, on 320 184 / 200.
    // Else two: 2 x 1.2 k on 258 106 / 98, 4 x 1.2 k on 128 84 / 61, 8 x 1.2 k on 150 153 / 125.
    const int64_t blocks = (int64_t)gx * hb;
    const bool one = total_kv <= 80 * (int64_t)B || (total_kv <= 512 * (int64_t)B && blocks <= 256) ||
                     (total_kv <= 320 * (int64_t)B && blocks >= 600 && blocks <= 768);
    if (D == 64) f32(D64, I2);
    else one ? f32(D128, I1) : f32(D128, I2);
  }
  return check_hip(hipGetLastError(), "attention launch");
}

}  // namespace tsc
