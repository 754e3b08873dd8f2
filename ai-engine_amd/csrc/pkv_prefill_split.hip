// pkv_prefill_split.hip -- chunked-prefill attention of f32 pools on the
// bf16 matrix cores (gfx950).
//
// The f32 MFMA (v_mfma_f32_16x16x4f32) does 64 flops per cycle and SIMD, the
// bf16 one 1,024.  Every f32 operand here is split into three bf16 values,
// x = x0 + x1 + x2 (x0 = bf16(x), x1 = bf16(x - x0), x2 = bf16(x - x0 - x1):
// 24 significant bits, the f32's own, of values above 2^-102; below, x2 falls
// out of bf16's range), and a product is the six bf16 products
// x0 y0, x0 y1, x1 y0, x0 y2, x1 y1, x2 y0 with f32 accumulation: exact
// products, and what is left out (x1 y2, x2 y1, x2 y2) is below 2^-25 of the
// product.  Six bf16 MFMAs take 6/16 of the f32 MFMA's time.  The small
// products go to an accumulator of their own (scores) or are summed per tile
// before they meet the running output, so no more f32 roundings touch the
// large sums than before: 1.6e-7 relative (2-norm) from 64 bits, against
// 2.6e-7 with the f32 MFMA (6 prompts of 200 to 775 tokens, 14 query heads on
// 2 kv heads).
//
// A launch of short prompts is bound by its longest chain of key tiles, so a
// workgroup's eight waves are four groups of 32 rows times two key groups:
// each step covers 64 keys, wave w takes rows 32 (w % 4) .. + 31 and keys
// 32 (w / 4) .. + 31 of it, and the two halves' (m, l, O) are merged through
// LDS at the end.  K and V are split once per workgroup where they are stored
// to LDS (three bf16 planes each), Q once in registers, the weights per lane.
// Against the f32 MFMA kernel (64 rows per workgroup), whole calls on one box:
// the 6 prompts 59.7 -> 36.7 us, one prompt of 775 tokens 43.8 -> 36.1, of
// 2,048 121.7 -> 96.3, 6 of 256 27.7 -> 17.9, 6 of 775 114.8 -> 57.4.  A step
// takes 2.7 us (48 MFMAs a wave, 1,536 cycles; 280 VALU instructions): running
// the key groups one phase apart, matrix against vector work with a barrier
// between (2,300 and 2,800 cycles a phase), placing the split and store among
// the score MFMAs, or 64 rows per workgroup gave the same or longer times.
//
// The split of a value beyond bf16's range (|x| > 3.39e38, infinities) leaves
// NaN in its remainders, so every sum it enters ends as NaN: rows whose sums
// are not all finite are computed again from the f32 values on the f32 MFMA,
// and such inputs give what f32 arithmetic gives.  So are rows that small
// values reach: a query with an element outside [2^-100, 2^64] (other than 0;
// within, a K element below 2^-102 shifts a score by 2^-56 at most), and rows
// with an output below kSmallOut that is not 0 (V elements below 2^-102 are
// off by 2^-126 at most, 2^-46 of any larger output).  What stays: a V column
// of f32 denormals alone may count as 0, and a weight below 2^-102 of the
// row's largest has fewer bits, which only a V element above 2^80 shows.
//
// head_dim 128 and 256 stay on the f32 MFMA (pkv_prefill.hip): two stages of
// the six planes would take 204 and 396 KB of LDS; a step of 32 keys (102 KB at
// 128), which leaves one key group, has not been built.
#include <type_traits>

#include "pkv_prefill_dev.h"

namespace pkv {
namespace {

constexpr int HD = 64;               // head_dim
constexpr int RG = kSplitRows / 32;  // groups of 32 rows; times two key groups: 2 RG waves
constexpr int kSKeys = kSplitKeys;   // keys per step (2 groups of 32)
constexpr float kSmallOut = 0x1p-80f;
constexpr float kQMin = 0x1p-100f, kQMax = 0x1p64f;

struct SCfg {
  static constexpr int ROWS = kSplitRows;
  static constexpr int NT = 128 * RG;           // threads
  static constexpr int RB = HD * 4;             // row bytes in the pool
  static constexpr int CH = RB / 16;            // 16-byte chunks per row
  static constexpr int PASS = kSKeys * CH / NT;  // chunks per thread and step (K, and V)
  static constexpr int PITCH = HD * 2 + 16;     // bf16 row pitch in LDS
  static constexpr int PLANE = 32 * PITCH;      // one plane of a key group's 32 rows
  static constexpr int GRP = 6 * PLANE;         // K planes 0..2, V planes 0..2
  static constexpr int STAGE = 2 * GRP;         // both key groups
  static constexpr int NDT = HD / 32;           // 32-dim tiles of O^T
  static constexpr int NKQ = HD / 16;           // 16-dim steps of Q K^T
  // rows computed again in f32: K and V as they are, the weights of a wave
  static constexpr int KP32 = RB + 16, VP32 = RB + 32;  // row pitches
  static constexpr int STAGE32 = kSKeys * (KP32 + VP32);
  static constexpr int P32 = 32 * 32 * 4;
  static_assert(kSKeys * CH % NT == 0, "");
  static_assert(2 * STAGE32 + 2 * RG * P32 <= 2 * STAGE, "the f32 rows fit the bf16 planes' LDS");
};

// Four floats to three bf16 planes (round to nearest even; remainders are
// exact in f32).
__device__ __forceinline__ void split4(const u32x4& x, uint2 (&p)[3]) {
  float r[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) r[i] = __uint_as_float(x[i]);
#pragma unroll
  for (int q = 0; q < 3; ++q) {
    p[q].x = cvt_pk16<PKV_BF16>(r[0], r[1]);
    p[q].y = cvt_pk16<PKV_BF16>(r[2], r[3]);
    if (q < 2) {
      r[0] -= bf16lo(p[q].x);
      r[1] -= bf16hi(p[q].x);
      r[2] -= bf16lo(p[q].y);
      r[3] -= bf16hi(p[q].y);
    }
  }
}

__device__ __forceinline__ void mfma32b(const u32x4& a, const u32x4& b, f32x16& acc) {
  acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, a),
                                                __builtin_bit_cast(bf16x8, b), acc, 0, 0, 0);
}

__device__ __forceinline__ void mfma32f(float a, float b, f32x16& acc) {
  acc = __builtin_amdgcn_mfma_f32_32x32x2f32(a, b, acc, 0, 0, 0);
}

template <bool FUSED>
__global__ void __launch_bounds__(SCfg::NT) prefill_split_kernel(PrefillKArgs a) {
  using C = SCfg;
  __shared__ __attribute__((aligned(16))) char lds[2 * C::STAGE];
  __shared__ uint32_t again[RG];  // rows to compute again in f32, a bit each

  const int R = a.rq;
  const int tid = threadIdx.x;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int lane = tid & 63;
  const int hh = lane >> 5, c32 = lane & 31;
  const int rw = wave % RG, kg = wave / RG;

  int sg, rb, part, q0, q1, ctx;
  if (!prefill_item(a, blockIdx.x, sg, rb, part, q0, q1, ctx)) return;
  const int g = sg % a.kvh;
  const int s = sg / a.kvh;
  const int q_len_raw = q1 - q0;
  const int q_len = min(q_len_raw, a.max_q_len);
  const bool reporter = tid == 0 && rb == 0 && g == 0;
  if (q_len_raw > a.max_q_len && reporter) atomicOr(a.err, PKV_EBIT_LENGTH);
  const int BS = 1 << a.bs_log2;
  if (ctx > a.max_context_len || ctx > a.mbps * BS || ctx < q_len || q_len < 0) {
    if (reporter) atomicOr(a.err, PKV_EBIT_LENGTH);
    return;
  }
  const int n_rows = q_len * R;
  const int row0 = rb * C::ROWS;
  if (row0 >= n_rows) return;  // uniform over the workgroup
  const int prior = ctx - q_len;
  const int H = a.kvh * R;
  const int tmask = BS - 1;
  const size_t slot_stride = (size_t)a.kvh * C::RB;
  const size_t blk_stride = (size_t)BS * slot_stride;
  const char* kh = a.k_pool + (size_t)g * C::RB;
  const char* vh = a.v_pool + (size_t)g * C::RB;
  const int32_t* table = a.block_tables + (size_t)s * a.mbps;
  const int n_keys = prior + min(row0 + C::ROWS - 1, n_rows - 1) / R + 1;
  const int nparts = n_parts_of(prior, a.part_keys);
  if (part >= nparts) return;  // uniform over the workgroup
  const char* kin = FUSED ? a.k_new + (size_t)g * C::RB : nullptr;
  const char* vin = FUSED ? a.v_new + (size_t)g * C::RB : nullptr;
  if constexpr (FUSED)
    prefill_store_chunk<C::ROWS, C::RB, C::NT>(a, R, rb, n_rows, q_len, prior, q0,
                                                  part == nparts - 1, table, kh, vh, kin, vin);
  if (tid < RG) again[tid] = 0u;

  const int k_hi = part + 1 < nparts ? (part + 1) * a.part_keys : n_keys;
  const int t_lo = part * (a.part_keys / kSKeys);
  const int n_steps = (k_hi + kSKeys - 1) / kSKeys;  // steps t_lo .. n_steps - 1

  const int roww = row0 + 32 * rw;
  const bool has_rows = roww < n_rows;
  const int klim_lo = prior + min(roww, n_rows - 1) / R;
  const int klim_hi = prior + min(roww + 31, n_rows - 1) / R;
  const int rc = min(roww + c32, n_rows - 1);
  const int lim = prior + rc / R;

  // ---- loads: chunk i of a thread is key (tid / CH) + (NT / CH) i of
  //      the step, bytes 16 (tid % CH); keys past n_keys are clamped.  The
  //      block id of each is read one step before its rows. ----
  const int lkey = tid / C::CH;
  const int lbyte = 16 * (tid % C::CH);
  bool bad_block = false;
  const size_t dk = FUSED ? (size_t)(kin - kh) : 0, dv = FUSED ? (size_t)(vin - vh) : 0;
  int id[C::PASS];
  u32x4 kreg[C::PASS], vreg[C::PASS];
  auto key_of = [&](int t, int i) __attribute__((always_inline)) {
    return min(t * kSKeys + lkey + (C::NT / C::CH) * i, n_keys - 1);
  };
  auto ids = [&](int t) __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < C::PASS; ++i) id[i] = table[key_of(t, i) >> a.bs_log2];
  };
  auto loads = [&](int t) __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < C::PASS; ++i) {
      const int key = key_of(t, i);
      const bool fresh = FUSED && key >= prior;
      const bool bad = !fresh && (unsigned)id[i] >= (unsigned)a.num_blocks;
      bad_block |= bad;
      const size_t off =
          fresh ? (size_t)(q0 + key - prior) * slot_stride
                : (size_t)(bad ? 0 : id[i]) * blk_stride + (uint32_t)(key & tmask) * slot_stride;
      kreg[i] = ld16(kh + (off + lbyte + (fresh ? dk : 0)));
      vreg[i] = ld16(vh + (off + lbyte + (fresh ? dv : 0)));
    }
  };
  auto store = [&](int stage) __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < C::PASS; ++i) {
      const int key = lkey + (C::NT / C::CH) * i;  // 0 .. 63
      char* dst = lds + stage * C::STAGE + (key >> 5) * C::GRP + (key & 31) * C::PITCH + lbyte / 2;
      uint2 p[3];
      split4(kreg[i], p);
#pragma unroll
      for (int q = 0; q < 3; ++q) *reinterpret_cast<uint2*>(dst + q * C::PLANE) = p[q];
      split4(vreg[i], p);
#pragma unroll
      for (int q = 0; q < 3; ++q) *reinterpret_cast<uint2*>(dst + (3 + q) * C::PLANE) = p[q];
    }
  };

  ids(t_lo);
  // ---- this wave's rows of Q (B operand), three planes ----
  u32x4 qf[3][C::NKQ];
  float q_lo = INFINITY, q_hi = 0.0f;  // extremes of |q| of this wave's half of the steps
  {
    const char* qrow = a.q + ((size_t)(q0 + rc / R) * H + g * R + rc % R) * C::RB;
#pragma unroll
    for (int ks = 0; ks < C::NKQ; ++ks) {
      uint2 lo[3], hi[3];
      const u32x4 x0 = ld16(qrow + 64 * ks + 32 * hh), x1 = ld16(qrow + 64 * ks + 32 * hh + 16);
      split4(x0, lo);
      split4(x1, hi);
      if ((ks & 1) == kg) {  // (both key groups hold these rows)
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const float y0 = fabsf(__uint_as_float(x0[i])), y1 = fabsf(__uint_as_float(x1[i]));
          q_lo = __builtin_elementwise_minimum(__builtin_elementwise_minimum(q_lo, y0), y1);
          q_hi = __builtin_elementwise_maximum(__builtin_elementwise_maximum(q_hi, y0), y1);
        }
      }
#pragma unroll
      for (int q = 0; q < 3; ++q) qf[q][ks] = u32x4{lo[q].x, lo[q].y, hi[q].x, hi[q].y};
    }
  }

  f32x16 o[C::NDT];
  float m = -INFINITY, l = 0.0f;
#pragma unroll
  for (int dt = 0; dt < C::NDT; ++dt)
#pragma unroll
    for (int r = 0; r < 16; ++r) o[dt][r] = 0.0f;

  // LDS reads of this wave: K rows c32 of its key group, 16-byte pieces; V by
  // ds_read_b64_tr_b16 (lane i of a 16-lane group, element j, gets the
  // (i & 3)-th value at the address of lane 4 j + (i >> 2)).
  const int kofs = kg * C::GRP + c32 * C::PITCH + 16 * hh;
  const int vs = lane & 15;
  const int vofs = kg * C::GRP + 3 * C::PLANE + (4 * hh + (vs >> 2)) * C::PITCH +
                   (4 * (vs & 3) + 16 * ((lane >> 4) & 1)) * 2;
  auto v_frag = [&](const char* b) __attribute__((always_inline)) {
    typedef short s4 __attribute__((ext_vector_type(4)));
    typedef __attribute__((address_space(3))) s4 lds_s4;
    const uint2 x = __builtin_bit_cast(uint2, __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s4*)(b)));
    const uint2 y = __builtin_bit_cast(
        uint2, __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s4*)(b + 8 * C::PITCH)));
    return u32x4{x.x, x.y, y.x, y.y};
  };

  auto compute = [&](int t) __attribute__((always_inline)) {
    const char* base = lds + (t & 1) * C::STAGE;
    const int k0 = t * kSKeys + 32 * kg;
    // ---- S^T = K Q^T: lane (half hh, row c32) gets, in register r, the score
    //      of key 8 (r / 4) + 4 hh + r % 4 ----
    f32x16 sc, sm;  // the large and the small products
#pragma unroll
    for (int r = 0; r < 16; ++r) sc[r] = sm[r] = 0.0f;
#pragma unroll
    for (int ks = 0; ks < C::NKQ; ++ks) {
      u32x4 kf[3];
#pragma unroll
      for (int q = 0; q < 3; ++q) kf[q] = ld16(base + kofs + q * C::PLANE + 32 * ks);
      mfma32b(kf[0], qf[0][ks], sc);
      mfma32b(kf[2], qf[0][ks], sm);
      mfma32b(kf[1], qf[0][ks], sc);
      mfma32b(kf[1], qf[1][ks], sm);
      mfma32b(kf[0], qf[1][ks], sc);
      mfma32b(kf[0], qf[2][ks], sm);
    }
#pragma unroll
    for (int r = 0; r < 16; ++r) sc[r] += sm[r];
    if (k0 + 31 > klim_lo) {  // wave-uniform: causal mask
      const int kk = k0 + 4 * hh - lim;
#pragma unroll
      for (int r = 0; r < 16; ++r)
        if (kk + 8 * (r >> 2) + (r & 3) > 0) sc[r] = -INFINITY;
    }
    // ---- online softmax, lazily raised reference (as prefill_body) ----
    float lmax = sc[0];
#pragma unroll
    for (int r = 1; r < 16; ++r) lmax = fmaxf(lmax, sc[r]);
    if (__builtin_amdgcn_ballot_w64(lmax * a.scale_log2 > m + kTau)) {  // wave-uniform
      const auto w = __builtin_amdgcn_permlane32_swap(__float_as_uint(lmax), __float_as_uint(lmax), false, false);
      const float tmax = fmaxf(__uint_as_float(w[0]), __uint_as_float(w[1])) * a.scale_log2;
      float alpha = 1.0f;
      if (tmax > m + kTau) {
        alpha = fast_exp2(m - tmax);
        m = tmax;
      }
      l *= alpha;
#pragma unroll
      for (int dt = 0; dt < C::NDT; ++dt)
#pragma unroll
        for (int r = 0; r < 16; ++r) o[dt][r] *= alpha;
    }
    // a row that has seen no key yet (this key group starts past it) keeps
    // m = -inf: its weights are exp2(-inf - 0) = 0
    const float nm = m == -INFINITY ? 0.0f : -m;
    u32x4 pf[3][2];  // [plane][16 keys]
#pragma unroll
    for (int r = 0; r < 16; r += 4) {
      u32x4 x;
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const float p = fast_exp2(fmaf(sc[r + i], a.scale_log2, nm));
        l += p;
        x[i] = __float_as_uint(p);
      }
      uint2 p[3];
      split4(x, p);
#pragma unroll
      for (int q = 0; q < 3; ++q) {
        pf[q][r >> 3][(r & 4) / 2] = p[q].x;
        pf[q][r >> 3][(r & 4) / 2 + 1] = p[q].y;
      }
    }
    // ---- O^T += V^T P^T, the tile's sum first, smallest products first ----
    f32x16 d[C::NDT];
#pragma unroll
    for (int dt = 0; dt < C::NDT; ++dt)
#pragma unroll
      for (int r = 0; r < 16; ++r) d[dt][r] = 0.0f;
#pragma unroll
    for (int ks = 0; ks < 2; ++ks) {
      u32x4 vf[C::NDT][3];
#pragma unroll
      for (int dt = 0; dt < C::NDT; ++dt)
#pragma unroll
        for (int q = 0; q < 3; ++q)
          vf[dt][q] = v_frag(base + vofs + q * C::PLANE + 16 * ks * C::PITCH + 64 * dt);
#pragma unroll
      for (int e = 0; e < 6; ++e) {
        constexpr int kv[6] = {2, 1, 0, 1, 0, 0}, kp[6] = {0, 1, 2, 0, 1, 0};
#pragma unroll
        for (int dt = 0; dt < C::NDT; ++dt) mfma32b(vf[dt][kv[e]], pf[kp[e]][ks], d[dt]);
      }
    }
#pragma unroll
    for (int dt = 0; dt < C::NDT; ++dt)
#pragma unroll
      for (int r = 0; r < 16; ++r) o[dt][r] += d[dt][r];
  };

  // ---- pipeline: step t is computed from LDS stage t & 1 while the rows of
  //      t + 1 sit in registers and the block ids of t + 2 are on the way;
  //      rows and ids past the last step are clamped (valid, unused) ----
  loads(t_lo);
  ids(t_lo + 1);
  store(t_lo & 1);
  loads(t_lo + 1);
  ids(t_lo + 2);
  __syncthreads();
  for (int t = t_lo; t < n_steps; ++t) {
    const int k0 = t * kSKeys + 32 * kg;
    if (has_rows && k0 < k_hi && k0 <= klim_hi) compute(t);  // wave-uniform
    if (t + 1 < n_steps) {                                    // workgroup-uniform
      store((t + 1) & 1);
      loads(t + 2);
      ids(t + 3);
    }
    __syncthreads();
  }
  if (bad_block) atomicOr(a.err, PKV_EBIT_BLOCK);

  auto full_sum = [&]() __attribute__((always_inline)) {  // both halves' part of l
    const auto lw = __builtin_amdgcn_permlane32_swap(__float_as_uint(l), __float_as_uint(l), false, false);
    l = __uint_as_float(lw[0]) + __uint_as_float(lw[1]);
  };
  full_sum();
  // rows to compute again, by a lane mask of this wave
  auto mark = [&](unsigned long long lanes) __attribute__((always_inline)) {
    const uint32_t left = max(n_rows - roww, 0);  // rows of this wave
    const uint32_t rows =
        ((uint32_t)lanes | (uint32_t)(lanes >> 32)) & (left < 32u ? (1u << left) - 1u : ~0u);
    if (rows && lane == 0) atomicOr(&again[rw], rows);
  };
  // queries out of the range in which small keys are exact enough; 0 is in it
  // (looked at again, from the first parts, only where there is one)
  if (__builtin_amdgcn_ballot_w64(!(q_lo >= kQMin && q_hi <= kQMax))) {  // wave-uniform
    bool far = false;
#pragma unroll
    for (int ks = 0; ks < C::NKQ; ++ks)
#pragma unroll
      for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int e = 0; e < 2; ++e) {
          const float y = fabsf(e ? bf16hi(qf[0][ks][i]) : bf16lo(qf[0][ks][i]));
          far |= (y < kQMin && y != 0.0f) || y > kQMax;
        }
    mark(__builtin_amdgcn_ballot_w64(far));
  }

  // ---- merge of the two key groups: group 1 hands (m, l, O) over in LDS,
  //      each register 64 lanes wide (no bank conflicts) ----
  constexpr int kXW = (C::NDT * 16 + 2) * 64;  // floats per row group
  static_assert(RG * kXW * 4 <= 2 * C::STAGE, "");
  float* xo = reinterpret_cast<float*>(lds) + rw * kXW;
  const bool partial = nparts > 1;
  float* const out_rows = partial ? a.part_o : reinterpret_cast<float*>(a.out);
  const size_t item = ((size_t)sg * a.row_blocks + rb) * a.max_parts + part;
  auto hand_over = [&]() __attribute__((always_inline)) {
    if (kg == 1) {
#pragma unroll
      for (int dt = 0; dt < C::NDT; ++dt)
#pragma unroll
        for (int r = 0; r < 16; r += 4)
          *reinterpret_cast<f32x4*>(xo + ((dt * 4 + r / 4) * 64 + lane) * 4) =
              f32x4{o[dt][r], o[dt][r + 1], o[dt][r + 2], o[dt][r + 3]};
      xo[C::NDT * 16 * 64 + lane] = m;
      xo[C::NDT * 16 * 64 + 64 + lane] = l;
    }
    __syncthreads();
  };
  // Key group 0 stores the merged rows: all of them, marking those to compute
  // again, or (`check` false) the marked ones, bit c32 of rows for row roww +
  // c32.  Marked are rows with an output that is not finite (a value whose
  // split overflowed, or an infinity or NaN in the inputs), rows without a
  // weight in key group 0, which every row sees (its products all overflowed
  // to -inf), and outputs too small for the split that are not 0.
  auto merge_store = [&](auto check, uint32_t rows) __attribute__((always_inline)) {
    constexpr bool CHECK = decltype(check)::value;
    const float m1 = xo[C::NDT * 16 * 64 + lane], l1 = xo[C::NDT * 16 * 64 + 64 + lane];
    const float M = fmaxf(m, m1);
    // (m = m1 = -inf: no finite score, sums of 0)
    const float w0 = m == M ? 1.0f : fast_exp2(m - M), w1 = m1 == M ? 1.0f : fast_exp2(m1 - M);
    l = l * w0 + l1 * w1;
    const int r = roww + c32;
    const bool live = r < n_rows && (CHECK || ((rows >> c32) & 1u));
    const float f0 = partial ? w0 : w0 / l, f1 = partial ? w1 : w1 / l;
    const size_t pr = item * C::ROWS + (r - row0);
    float* dst = out_rows + (partial ? pr : (size_t)(q0 + r / R) * H + g * R + r % R) * HD;
    auto merged = [&](int dt, int q4) __attribute__((always_inline)) {
      const f32x4 x = *reinterpret_cast<const f32x4*>(xo + ((dt * 4 + q4) * 64 + lane) * 4);
      f32x4 y;
#pragma unroll
      for (int j = 0; j < 4; ++j) y[j] = o[dt][4 * q4 + j] * f0 + x[j] * f1;
      return y;
    };
    float lo = INFINITY, hi = 0.0f;  // extremes of |y|, NaN if one is NaN
#pragma unroll
    for (int dt = 0; dt < C::NDT; ++dt)
#pragma unroll
      for (int q4 = 0; q4 < 4; ++q4) {
        const f32x4 y = merged(dt, q4);
        if (live) *reinterpret_cast<f32x4*>(dst + 32 * dt + 8 * q4 + 4 * hh) = y;
        if constexpr (CHECK) {
#pragma unroll
          for (int j = 0; j < 4; ++j) {
            lo = __builtin_elementwise_minimum(lo, fabsf(y[j]));
            hi = __builtin_elementwise_maximum(hi, fabsf(y[j]));
          }
        }
      }
    if (partial && live && hh == 0) {
      a.part_ml[2 * pr] = M;
      a.part_ml[2 * pr + 1] = l;
    }
    if constexpr (CHECK) {
      const float small = partial ? l * kSmallOut : kSmallOut;
      const bool fine = lo >= small && hi < INFINITY && m != -INFINITY;
      if (__builtin_amdgcn_ballot_w64(!fine)) {  // wave-uniform: a 0 among them, or worse
        bool bad = !(hi < INFINITY) || m == -INFINITY;
#pragma unroll
        for (int dt = 0; dt < C::NDT; ++dt)
#pragma unroll
          for (int q4 = 0; q4 < 4; ++q4) {
            const f32x4 y = merged(dt, q4);
#pragma unroll
            for (int j = 0; j < 4; ++j) bad |= fabsf(y[j]) < small && y[j] != 0.0f;
          }
        mark(__builtin_amdgcn_ballot_w64(bad));
      }
    }
  };
  hand_over();
  if (kg == 0 && has_rows) merge_store(std::true_type{}, ~0u);  // wave-uniform
  __syncthreads();  // the marks are there, and the merge's values have been read
  uint32_t mine = 0, any = 0;
#pragma unroll
  for (int i = 0; i < RG; ++i) {
    const uint32_t w = (uint32_t)__builtin_amdgcn_readfirstlane((int)again[i]);
    any |= w;
    mine = i == rw ? w : mine;
  }
  if (any == 0u) return;  // workgroup-uniform

  // ---- rows `mine` again on the f32 MFMA, with the same split of rows and
  //      keys over the waves: K and V in LDS as they are (double-buffered),
  //      the running maximum exact (a weight above 1 could overflow a large
  //      value).  One prompt of 4,096 tokens (14 query heads on 2) whose first
  //      key holds a NaN: 531 us (205 without it), against 26,200 with a row
  //      per wave and a key at a time on the VALU. ----
  float qs[HD / 2];  // Q[row c32][HD / 2 hh ..], the B operand
  {
    const char* qrow = a.q + ((size_t)(q0 + rc / R) * H + g * R + rc % R) * C::RB + C::RB / 2 * hh;
#pragma unroll
    for (int i = 0; i < HD / 8; ++i) {
      const f32x4 x = *reinterpret_cast<const f32x4*>(qrow + 16 * i);
#pragma unroll
      for (int j = 0; j < 4; ++j) qs[4 * i + j] = x[j];
    }
  }
  m = -INFINITY;
  l = 0.0f;
#pragma unroll
  for (int dt = 0; dt < C::NDT; ++dt)
#pragma unroll
    for (int r = 0; r < 16; ++r) o[dt][r] = 0.0f;
  auto again_step = [&](int t) __attribute__((always_inline)) {
    const char* base = lds + (t & 1) * C::STAGE32;
    const char* kl = base + (32 * kg + c32) * C::KP32 + C::RB / 2 * hh;
    const char* vl = base + kSKeys * C::KP32 + 32 * kg * C::VP32;
    const int k0 = t * kSKeys + 32 * kg;
    f32x16 sc;
#pragma unroll
    for (int r = 0; r < 16; ++r) sc[r] = 0.0f;
#pragma unroll
    for (int i = 0; i < HD / 8; ++i) {
      const f32x4 x = *reinterpret_cast<const f32x4*>(kl + 16 * i);
#pragma unroll
      for (int j = 0; j < 4; ++j) mfma32f(x[j], qs[4 * i + j], sc);
    }
    const int kk = k0 + 4 * hh - lim;
    const bool masked = k0 + 31 > klim_lo;  // wave-uniform
    float tmax = -INFINITY;
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      if (masked && kk + 8 * (r >> 2) + (r & 3) > 0) sc[r] = -INFINITY;
      tmax = fmaxf(tmax, sc[r]);
    }
    tmax = fmaxf(tmax, shfl_xor_f(tmax, 32)) * a.scale_log2;
    const float mn = fmaxf(m, tmax);
    const float alpha = mn == m ? 1.0f : fast_exp2(m - mn);
    const float nm = mn == -INFINITY ? 0.0f : -mn;  // no finite score yet: weights 0
    m = mn;
    l *= alpha;
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      sc[r] = fast_exp2(fmaf(sc[r], a.scale_log2, nm));
      l += sc[r];
    }
#pragma unroll
    for (int dt = 0; dt < C::NDT; ++dt)
#pragma unroll
      for (int r = 0; r < 16; ++r) o[dt][r] *= alpha;
    if (!masked) {  // MFMA r sums the keys of register r of both halves
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        const char* v = vl + (8 * (r >> 2) + 4 * hh + (r & 3)) * C::VP32 + 4 * c32;
#pragma unroll
        for (int dt = 0; dt < C::NDT; ++dt)
          mfma32f(*reinterpret_cast<const float*>(v + 128 * dt), sc[r], o[dt]);
      }
    } else {  // a row's own keys only: 0 times an infinity that it does not see is NaN
      float* pl = reinterpret_cast<float*>(lds + 2 * C::STAGE32 + wave * C::P32);
#pragma unroll
      for (int r = 0; r < 16; ++r) pl[(8 * (r >> 2) + 4 * hh + (r & 3)) * 32 + c32] = sc[r];
      __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
      __builtin_amdgcn_wave_barrier();
#pragma unroll 1
      for (int k = 0; k < 32; ++k) {
        const float p = pl[k * 32 + c32];
        const bool seen = k0 + k <= lim;
#pragma unroll
        for (int dt = 0; dt < C::NDT; ++dt)
#pragma unroll
          for (int q4 = 0; q4 < 4; ++q4) {
            const f32x4 v = *reinterpret_cast<const f32x4*>(
                vl + k * C::VP32 + 4 * (32 * dt + 8 * q4 + 4 * hh));
#pragma unroll
            for (int j = 0; j < 4; ++j)
              o[dt][4 * q4 + j] = seen ? fmaf(p, v[j], o[dt][4 * q4 + j]) : o[dt][4 * q4 + j];
          }
      }
    }
  };
  ids(t_lo);
  loads(t_lo);
  for (int t = t_lo; t < n_steps; ++t) {
    char* base = lds + (t & 1) * C::STAGE32;
#pragma unroll
    for (int i = 0; i < C::PASS; ++i) {
      const int key = lkey + (C::NT / C::CH) * i;
      st16(base + key * C::KP32 + lbyte, kreg[i]);
      st16(base + kSKeys * C::KP32 + key * C::VP32 + lbyte, vreg[i]);
    }
    __syncthreads();
    ids(t + 1);
    loads(t + 1);
    const int k0 = t * kSKeys + 32 * kg;
    if (mine && k0 < k_hi && k0 <= klim_hi) again_step(t);  // wave-uniform
  }
  full_sum();
  __syncthreads();  // every wave has read its tiles
  hand_over();
  if (kg == 0 && mine) merge_store(std::false_type{}, mine);
}

}  // namespace

hipError_t launch_prefill_split(const PrefillKArgs& k0, hipStream_t s) {
  using C = SCfg;
  PrefillKArgs k = k0;
  k.row_blocks = (int)(((long long)k.max_q_len * k.rq + C::ROWS - 1) / C::ROWS);
  const long long grid = (long long)k.n_seqs * k.kvh * k.row_blocks * k.max_parts;
  if (grid <= 0) return hipSuccess;
  if (!grid_fits(grid, C::NT)) return hipErrorInvalidValue;
  // Plain order, longest row blocks of every pair first: the launches this
  // kernel is bound on have few workgroups, and the affinity mapping left
  // XCDs idle (6 prompts x 2 kv heads: 12 pairs on 8 XCDs).
  k.per_xcd = 0;
  if (k.k_new)
    prefill_split_kernel<true><<<(unsigned)grid, C::NT, 0, s>>>(k);
  else
    prefill_split_kernel<false><<<(unsigned)grid, C::NT, 0, s>>>(k);
  return hipGetLastError();
}

}  // namespace pkv
