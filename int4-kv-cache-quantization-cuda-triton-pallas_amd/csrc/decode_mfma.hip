// Fused INT4 flash decoding for grouped query heads on the matrix cores
// (gfx950): key products on the int8 ones, value products on the 16-bit (16-bit
// values) or float32 ones. Same semantics as decode_kernel and decode_gqa_kernel
// (reference src/flash_decode_ref.py:30-139 per (sequence, q-head) stream,
// q-head h reading kv-head h // (Hq/Hkv), src/ops.py:189-192): unscaled logits
// sum_d (q_d*s_d)*nib_d - sum_d q_d*(zp_d*s_d), online softmax, float32 value
// accumulation, split partials or the final output. One workgroup serves HG
// (2, 4 or 8) q-heads of one kv-head.
//
// Lane l: g = l / 16, n = l % 16, head n / CPH, column c = n % CPH of its head
// (CPH = 16 / HG columns per head). A 16-row chunk goes through a wave as
//
//   logits: the products v_d = q_d*s_d (exact in double) are scaled by
//      2^(46-E), E the binary exponent of the head's largest, rounded to
//      integers |v_d| <= 2^46 and written as six balanced base-256 digits (the
//      bytes of v + 0x808080808080, each less 128). v_mfma_i32_16x16x64_i8
//      multiplies the 16 rows' nibbles (A: row n, channels of group g) by
//      digits (B), and the columns of a head hold DIFFERENT digits: all six in
//      one product at HG = 2, in two at HG = 4, in three at HG = 8. The exact
//      int32 sums of a row's digits, which lie in neighbouring lanes, meet by
//      quad permutes (a reduce-scatter over the columns), so each logit is
//      recombined in double and exponentiated in one lane (two lanes at
//      HG = 2), not in every column: lane (g, head, c) ends with row
//      4g + c % 4 (HG = 8: rows 4g + c and 4g + c + 2). Error against double
//      products: 2^(E-47) per product and the double rounding of the sum.
//   probabilities: the lane group g that holds the logits of rows 4g .. 4g+3 is
//      the one that must supply them as the value product's B operand, so they
//      move by quad permutes too and nothing goes through LDS.
//   values, 16-bit: lane (g, n) loads its 8 (4 at D = 64) channels of rows
//      4g .. 4g+3; byte permutes pair the rows, and each 16x16x16 product adds
//      four rows a lane group to the output of 16 channels x 16 columns. A
//      float32 probability is the exact sum of three 8-bit (bfloat16) or
//      11-bit (float16) terms, which sit in different columns of the head
//      (HG = 8: the first term in one column, the others in the second, in two
//      products), so the products are exact, their sums are float32, and one
//      instruction does all terms. Only the final output adds the columns up.
//      float16 has 40 binades for the terms: they are scaled by 2^15 (the first)
//      and 2^25 (the others), which holds every bit of a probability down to
//      2^-26. A chunk with a smaller one (a row 18 below the wave's maximum in
//      the logit) takes the float32 products below, in the first column: with
//      logits of standard deviation 2 none does; where every chunk does (12), a
//      B8 Hkv8 Hq32 T8192 decode takes 41 us in place of 32, B16 Hkv8 Hq64 ragged
//      to 4096 45 in place of 27.
//      A non-finite value times an empty term is NaN where the float32 product
//      is infinite: a wave that ends with a NaN runs its range again with the
//      float32 products below.
//   values, float32: v_mfma_f32_16x16x4_f32, a row of each lane group at a time.
//      Chunk sums come first and are then added to the rescaled accumulators.
//
//      The matrix cores align a product of a subnormal float16 value as if the
//      value were 2^-14: sums of values below that are good to 2^-38.
//
// What bounds it, and why this form: a chunk of 16-bit values at D = 128 is 5 KB,
// 0.66 us of a SIMD's share of HBM; float32 FMAs of every value with every
// head's probability, widening, the LDS round trip of the probabilities and one
// logit recombination per (row, column) cost more vector-unit time than that at
// HG = 4 and twice as much at HG = 8. Measured against that form, per call with
// the merge: B8 Hkv8 Hq32 T8192 bfloat16 37.3 -> 31.6 us (172 MB, read once: 5.7
// TB/s over the kernel's 30.0 us, of which a workgroup's first 6 and last 2 stream
// nothing); D = 256 B4 Hkv4 Hq16 T4095 30.0 -> 16.3 us (against the vector
// kernel); a B16 Hkv8 Hq64 float16 step of ragged lengths to 4096 56.7 -> 34.3 us;
// B8 H32 over one float32 stream of 2048 rows 16.0 -> 12.6 us.

#include "decode_common.hpp"

namespace fdi4 {

typedef int v4i __attribute__((ext_vector_type(4)));
typedef float v4f __attribute__((ext_vector_type(4)));
typedef short v4s __attribute__((ext_vector_type(4)));
typedef _Float16 v4h __attribute__((ext_vector_type(4)));

template <int D, int VDT, int HG>
struct MfmaGeo {
  static constexpr int NB = D / 64;                // 64-channel MFMA blocks
  static constexpr int KW = D / 32;                // packed key words per lane per row
  static constexpr int CPH = 16 / HG;              // result columns per head
  static constexpr int NSET = CPH >= 8 ? 1 : CPH == 4 ? 2 : 3;  // digit products per block
  static constexpr int RN = CPH >= 4 ? 1 : 2;      // logits a lane ends with
  static constexpr int PPL = HG * D / 64;          // channels of q*s a lane turns into digits
  static constexpr int VEB = VDT == kVF32 ? 4 : 2; // bytes per value element
  static constexpr int PB = D * VEB / 16 < 16 ? D * VEB / 16 : 16;  // bytes per value load
  static constexpr int NP = D * VEB / (16 * PB);   // value loads per lane per row
  static constexpr int CPP = PB / VEB;             // channels per value load
  static constexpr int NA = D / 16;                // 16-channel output tiles
  static constexpr int SZI = D / 2;                // 16-byte items in a scale+zp block
  static constexpr int SZL = (SZI + 63) / 64;      // scale+zp loads per lane
  static constexpr int DIGITS = 6;
  // LDS per wave: the staged scale/zero-point block and the digits of a group
  // while the wave streams, its partial output afterwards.
  static constexpr int kDigBytes = DIGITS * HG * D;
  static constexpr int kStreamBytes = kDigBytes + 16 * D;
  static constexpr int kAccBytes = 4 * HG * D;
  static constexpr int kWaveBytes = kStreamBytes > kAccBytes ? kStreamBytes : kAccBytes;
  static_assert(D == 64 || D == 128 || D == 256, "head_dim");
  static_assert(HG == 2 || HG == 4 || HG == 8, "heads per workgroup");
};

// Position of channel d in the operands' order: lane group g holds channels
// [g*D/4, (g+1)*D/4) in 16-channel blocks, of each block the even channels
// (low nibbles of the packed bytes) before the odd ones (high nibbles).
__device__ __forceinline__ int slot_of(int d) {
  return (d & ~15) | ((d & 1) << 3) | ((d & 15) >> 1);
}

template <int CTRL>
__device__ __forceinline__ unsigned dpp(unsigned x) {
  return (unsigned)__builtin_amdgcn_mov_dpp((int)x, CTRL, 0xF, 0xF, false);
}

// Value of lane ^ 4: mirrored within 8 lanes, then within 4.
__device__ __forceinline__ double xchg4_dpp(double x) {
  DU v;
  v.d = x;
  v.u[0] = dpp<0x1B>(dpp<0x141>(v.u[0]));
  v.u[1] = dpp<0x1B>(dpp<0x141>(v.u[1]));
  return v.d;
}

template <int LO, int HI>
__device__ __forceinline__ unsigned allreduce_max_u(unsigned x) {
  if constexpr (LO <= 1 && 1 < HI) x = max(x, xchg_u32<1>(x));
  if constexpr (LO <= 2 && 2 < HI) x = max(x, xchg_u32<2>(x));
  if constexpr (LO <= 4 && 4 < HI) x = max(x, xchg_u32<4>(x));
  if constexpr (LO <= 8 && 8 < HI) x = max(x, xchg_u32<8>(x));
  if constexpr (LO <= 16 && 16 < HI) x = max(x, xchg_u32<16>(x));
  if constexpr (LO <= 32 && 32 < HI) x = max(x, xchg_u32<32>(x));
  return x;
}

// The chunk walk of a wave: logical page, chunk within it, scale group and the
// page's index in its group, advanced by compares.
struct ChunkPos {
  int lp, j, group, pig;
};

__device__ __forceinline__ ChunkPos chunk_pos(const DecodeArgs& a, int c, int cpp) {
  ChunkPos p;
  p.lp = fdiv(c, a.div_cpp);
  p.j = c - p.lp * cpp;
  p.group = fdiv(p.lp, a.div_ppg);
  p.pig = p.lp - p.group * a.pages_per_group;
  return p;
}

__device__ __forceinline__ ChunkPos chunk_next(ChunkPos p, int cpp, int ppg) {
  p.j += 1;
  const bool np = p.j == cpp;
  p.j = np ? 0 : p.j;
  p.lp += np ? 1 : 0;
  p.pig += np ? 1 : 0;
  const bool ng = p.pig == ppg;
  p.pig = ng ? 0 : p.pig;
  p.group += ng ? 1 : 0;
  return p;
}

struct PosMeta {
  unsigned phys;
  int r0, nval, group;
};

// One sequence's page metadata. An absent table (null) is read at element 0 of
// some valid array and the value dropped, which spares the chunk loop a branch
// and its mask arithmetic.
struct PageMeta {
  const int32_t* table;
  const int32_t* lens;
  int table_mul, lens_mul;    // 1, or 0: absent
};

__device__ __forceinline__ PageMeta page_meta(const DecodeArgs& a, int b) {
  PageMeta p;
  const int32_t* any = reinterpret_cast<const int32_t*>(a.k_scale);
  p.table = a.page_table ? a.page_table + (int64_t)b * a.pt_b : any;
  p.lens = a.page_lens ? a.page_lens + (int64_t)b * a.pl_b : any;
  p.table_mul = a.page_table ? 1 : 0;
  p.lens_mul = a.page_lens ? 1 : 0;
  return p;
}

__device__ __forceinline__ PosMeta pos_meta(const DecodeArgs& a, const PageMeta& pm, int T,
                                            const ChunkPos& p) {
  PosMeta m;
  const int pg = ld_ro(pm.table, p.lp * pm.table_mul);
  const int pl = ld_ro(pm.lens, p.lp * pm.lens_mul);
  const int left = T - p.lp * a.page_rows;
  const int rows = min(pm.lens_mul ? max(pl, 0) : left, a.page_rows);
  m.r0 = p.j * 16;
  m.nval = min(16, rows - m.r0);
  m.phys = (unsigned)min(max(pm.table_mul ? pg : p.lp, 0), a.num_pages - 1);
  m.group = p.group;
  return m;
}

// v_max without the quieting moves that fmax puts before operands of unknown
// origin (the instruction quiets them itself).
__device__ __forceinline__ float max_raw(float x, float y) {
  float r;
  asm("v_max_f32 %0, %1, %2" : "=v"(r) : "v"(x), "v"(y));
  return r;
}

__device__ __forceinline__ double max_raw(double x, double y) {
  double r;
  asm("v_max_f64 %0, %1, %2" : "=v"(r) : "v"(x), "v"(y));
  return r;
}

// Maximum over the four 16-lane groups: a swap of a register with its copy
// leaves both groups' values in the two results.
__device__ __forceinline__ float groups_max(float x) {
  auto r = __builtin_amdgcn_permlane16_swap(f2u(x), f2u(x), false, false);
  x = max_raw(u2f(r[0]), u2f(r[1]));
  auto s = __builtin_amdgcn_permlane32_swap(f2u(x), f2u(x), false, false);
  return max_raw(u2f(s[0]), u2f(s[1]));
}

template <int D, int VDT, int WAVES, int HG>
__global__ __launch_bounds__(WAVES * 64) void decode_mfma_kernel(DecodeArgs a) {
  using G = MfmaGeo<D, VDT, HG>;
  constexpr int NT = WAVES * 64, CPH = G::CPH, RN = G::RN;
  // float16 terms of a probability: the first is that of p * 2^15 (p <= 1, so it
  // is finite), the others those of the remainder (below 2^-10 p) times 2^25. The
  // last bit of p is at least 2^-49 from p = 2^-26 up, so every term is a multiple
  // of float16's smallest number.
  constexpr float kPScale = VDT == kVF16 ? 0x1p15f : 1.f;
  constexpr float kRestScale = VDT == kVF16 ? 0x1p10f : 1.f;   // of the others, beyond it
  constexpr float kLeastP = 0x1p-26f * kPScale;

  const int split = blockIdx.x, b = blockIdx.z;
  const int h0 = blockIdx.y * HG;           // first q-head of this workgroup
  const int hk = fdiv(h0, a.div_hpk);         // HG divides hq_per_kv: one kv-head
  const int tid = threadIdx.x, lane = tid & 63;
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int n16 = lane & 15;                // key row (A) and result column
  const int grp = lane >> 4;                // channel group; result rows 4*grp..+3
  const int hh = n16 / CPH;                 // head of this lane's column
  const int col = n16 % CPH;                // column within the head
  const bool odd = (n16 & 1) != 0, hi2 = (n16 & 2) != 0, hi4 = (n16 & 4) != 0;
  const int lrow = 4 * grp + (CPH >= 4 ? (n16 & 3) : (n16 & 1));  // row of logit 0

  __shared__ __align__(16) float q_s[HG][D];                      // slot order
  __shared__ __align__(16) uint8_t wave_s[WAVES][G::kWaveBytes];
  __shared__ double m_s[WAVES][HG];
  __shared__ float l_s[WAVES][HG];
  uint8_t* const dig_w = wave_s[w];
  double* const sz_w = reinterpret_cast<double*>(wave_s[w] + G::kDigBytes);

  // The q rows of the HG heads are loaded first and go to LDS once the first
  // chunk's loads are issued.
  constexpr int QPT = (HG * D + NT - 1) / NT;
  float qv[QPT];
#pragma unroll
  for (int j = 0; j < QPT; ++j) {
    const int idx = tid + j * NT;
    qv[j] = (idx < HG * D)
                ? load_elem(a.q, (int64_t)b * a.q_b + (int64_t)(h0 + idx / D) * a.q_h + idx % D,
                            a.q_dtype)
                : 0.f;
  }

  const int cpp = (a.page_rows + 15) >> 4, ppg = a.pages_per_group;
  const PageMeta pgm = page_meta(a, b);
  const int T = seq_len_of(a, b);
  const int n_chunks = pages_of(a, T) * cpp;
  const int c_begin = split * a.chunks_per_split;
  const int c_end = min(c_begin + a.chunks_per_split, n_chunks);
  const WaveRange wr = wave_chunks(c_begin, c_end, w, WAVES);
  const int wc0 = wr.c0, wc1 = wr.c1;

  // Softmax state of head hh in units of log2 (the same in all its lanes), and
  // the sum of the probabilities of this lane's rows.
  double m_run = -INFINITY;
  float l_run = 0.f;
  // Output tiles: channel 8 (CPP) * m + j of piece u for result row m, column n16.
  v4f acc[G::NA];
  // Digits of head hh's scaled q*s (B operands), and logit = sum * c1 - cg.
  v4i bq[G::NSET][G::NB];
  double c1 = 0.0, cg = 0.0;
  int cur_group = -1;

  const float* sbase = a.k_scale + (int64_t)b * a.s_b + (int64_t)hk * a.s_h;
  const float* zbase = a.k_zp + (int64_t)b * a.s_b + (int64_t)hk * a.s_h;
  // Page bases are wave-uniform (scalar registers); each lane adds a 32-bit
  // byte offset (its channel slice and row), so the loads take the
  // scalar-base + vector-offset form with no 64-bit address arithmetic per
  // lane (row strides are checked on the host: 16 rows fit in 31 bits).
  const uint8_t* kbase_h = a.k_pages + (int64_t)hk * a.k_head;
  const uint8_t* vbase_h = reinterpret_cast<const uint8_t*>(a.v_pages) +
                           (int64_t)hk * a.v_head * G::VEB;
  const unsigned krow_b = (unsigned)a.k_row, vrow_b = (unsigned)(a.v_row * G::VEB);
  // Offsets of this lane's key row and value rows in a full chunk; a partial one
  // takes the smaller of these and the last valid row's.
  const unsigned k_lane = grp * (D / 8), v_lane = n16 * G::PB;
  const unsigned k_full = k_lane + n16 * krow_b;
  unsigned v_full[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) v_full[i] = v_lane + (4 * grp + i) * vrow_b;
  // Scale/zero-point block of a group: items 0..D/4-1 are scale[4e..4e+3], items
  // D/4..D/2-1 are zp. Lanes past the block reload an in-range item.
  const float* sz_src[G::SZL];
#pragma unroll
  for (int i = 0; i < G::SZL; ++i) {
    const int e = (i * 64 + lane) % G::SZI;
    sz_src[i] = e < D / 4 ? sbase + 4 * e : zbase + 4 * (e - D / 4);
  }

  struct Buf {
    unsigned k[G::KW];
    unsigned v[4][G::NP][G::PB / 4];
  };

  auto load_sz = [&](const PosMeta& m, U32x4* sz) __attribute__((always_inline)) {
    const int64_t off = (uint64_t)(unsigned)m.group * (uint64_t)a.s_g +
                        (uint64_t)m.phys * (uint64_t)a.s_p;
#pragma unroll
    for (int i = 0; i < G::SZL; ++i) sz[i] = ld16(sz_src[i] + off);
  };

  // Rows past the valid count are loaded from the last valid row (never out of
  // bounds); their probabilities are 0.
  auto load_chunk = [&](const PosMeta& m, int nval, Buf& f) __attribute__((always_inline)) {
    const unsigned last = (unsigned)max(nval - 1, 0);
    const uint8_t* kb = kbase_h + ((uint64_t)m.phys * (uint64_t)a.k_page +
                                   (uint64_t)(unsigned)m.r0 * krow_b);
    const unsigned ko = min(k_full, k_lane + last * krow_b);
    constexpr int KL = G::KW < 4 ? G::KW : 4;
#pragma unroll
    for (int i = 0; i < G::KW / KL; ++i) {
      const KVec<KL> x = load_k<KL>(kb + (ko + 16 * i));
#pragma unroll
      for (int k = 0; k < KL; ++k) f.k[KL * i + k] = x.w[k];
    }
    const uint8_t* vb = vbase_h + ((uint64_t)m.phys * (uint64_t)(a.v_page * G::VEB) +
                                   (uint64_t)(unsigned)m.r0 * vrow_b);
    const unsigned v_last = v_lane + last * vrow_b;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const unsigned vo = min(v_full[i], v_last);
#pragma unroll
      for (int u = 0; u < G::NP; ++u) {
        const KVec<G::PB / 4> x = load_k<G::PB / 4>(vb + (vo + 16 * G::PB * u));
#pragma unroll
        for (int k = 0; k < G::PB / 4; ++k) f.v[i][u][k] = x.w[k];
      }
    }
  };

  // Rebuild the B operands (digits), scale factors and group constants of the
  // HG heads from the loaded scale/zero-point block. Lane (g, head, c) turns
  // the PPL channels at slots c*PPL of its group into digits; the bytes go
  // through LDS ([digit][head][slot]) to the lanes whose column needs them.
  auto rebuild = [&](const U32x4* sz) __attribute__((always_inline)) {
    // Staged as doubles, in slot order: the conversions are shared by the heads.
#pragma unroll
    for (int i = 0; i < G::SZL; ++i) {
      const int e = i * 64 + lane;
      if (e < G::SZI) {
        double* dst = sz_w + (e < D / 4 ? 0 : D) + slot_of(4 * (e % (D / 4)));
        *reinterpret_cast<double2*>(dst) = make_double2(u2f(sz[i].x), u2f(sz[i].z));
        *reinterpret_cast<double2*>(dst + 8) = make_double2(u2f(sz[i].y), u2f(sz[i].w));
      }
    }
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    constexpr int PPL = G::PPL, PK = PPL < 4 ? PPL : 4;
    const int s0 = grp * (D / 4) + col * PPL;
    const float* qh = q_s[hh] + s0;
    const double* sh = sz_w + s0;
    const double* zh = sz_w + D + s0;
    // The largest |q*s| by its high word (exponent and leading bits), and the
    // group constant.
    unsigned mx = 0;
    double cgp = 0.0;
    DU qs[PPL];
#pragma unroll
    for (int i = 0; i < PPL; ++i) {
      const double qd = (double)qh[i], sd = sh[i];
      qs[i].d = qd * sd;
      mx = max(mx, qs[i].u[1] & 0x7FFFFFFFu);
      cgp = __builtin_fma(qd, zh[i] * sd, cgp);
    }
    mx = allreduce_max_u<16, 64>(allreduce_max_u<1, CPH>(mx));
    cgp = allreduce_sum<16, 64>(allreduce_sum<1, CPH>(cgp));
    // |q*s| < 2^E, E = (mx >> 20) - 1022; all zero, infinite or NaN (then the
    // group constant is too): any scale.
    const int E = mx - 1u < 0x7FEFFFFFu ? (int)(mx >> 20) - 1022 : 0;
    DU up, down;
    up.u[0] = 0;
    up.u[1] = (unsigned)(1023 + 46 - E) << 20;
    down.u[0] = 0;
    down.u[1] = (unsigned)(1023 - 46 + E) << 20;
    c1 = down.d * 1.4426950408889634;
    cg = cgp * 1.4426950408889634;
    // 1.5 * 2^52 + the bias of the balanced digits: the low 48 bits of the sum
    // are rint(q*s * 2^(46-E)) + 0x808080808080.
    constexpr double kMagic = 6755399441055744.0 + 141289400074368.0;
#pragma unroll
    for (int i0 = 0; i0 < PPL; i0 += PK) {
      unsigned lo[4] = {0, 0, 0, 0}, hi[4] = {0, 0, 0, 0};
#pragma unroll
      for (int k = 0; k < PK; ++k) {
        DU v;
        v.d = __builtin_fma(qs[i0 + k].d, up.d, kMagic);
        lo[k] = v.u[0];
        hi[k] = v.u[1];
      }
      const unsigned t0 = __builtin_amdgcn_perm(lo[1], lo[0], 0x05010400u);
      const unsigned t1 = __builtin_amdgcn_perm(lo[1], lo[0], 0x07030602u);
      const unsigned u0 = __builtin_amdgcn_perm(lo[3], lo[2], 0x05010400u);
      const unsigned u1 = __builtin_amdgcn_perm(lo[3], lo[2], 0x07030602u);
      const unsigned h0w = __builtin_amdgcn_perm(hi[1], hi[0], 0x05010400u);
      const unsigned h1w = __builtin_amdgcn_perm(hi[3], hi[2], 0x05010400u);
      // Digit 0 is the most significant.
      const unsigned dg[6] = {
          __builtin_amdgcn_perm(h1w, h0w, 0x07060302u), __builtin_amdgcn_perm(h1w, h0w, 0x05040100u),
          __builtin_amdgcn_perm(u1, t1, 0x07060302u),   __builtin_amdgcn_perm(u1, t1, 0x05040100u),
          __builtin_amdgcn_perm(u0, t0, 0x07060302u),   __builtin_amdgcn_perm(u0, t0, 0x05040100u)};
#pragma unroll
      for (int k = 0; k < G::DIGITS; ++k) {
        uint8_t* dst = dig_w + k * HG * D + hh * D + s0 + i0;
        if constexpr (PK == 4)
          *reinterpret_cast<unsigned*>(dst) = dg[k] ^ 0x80808080u;
        else
          *reinterpret_cast<uint16_t*>(dst) = (uint16_t)(dg[k] ^ 0x8080u);
      }
    }
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
#pragma unroll
    for (int s = 0; s < G::NSET; ++s) {
      // The digit of this lane's column in product s.
      int dg;
      if constexpr (CPH == 2) dg = 2 * s + col;
      else if constexpr (CPH == 4) dg = s == 0 ? col : 4 + (col & 1);
      else dg = hi4 ? 4 + (col & 1) : (col & 3);
#pragma unroll
      for (int kb = 0; kb < G::NB; ++kb)
        bq[s][kb] = *reinterpret_cast<const v4i*>(dig_w + dg * HG * D + hh * D +
                                                  grp * (D / 4) + 16 * kb);
    }
    __builtin_amdgcn_wave_barrier();
  };

  // Column sums of a digit pair: lane pairs (even column: high digit) exchange
  // rows, the even lane keeping rows 0 and 2 of its four, the odd one 1 and 3.
  const int wsh = odd ? 0 : 8;
  // Selects as bit selects under lane masks: a ternary over vector elements
  // becomes an indexed access, five instructions for one.
  const int m_odd = odd ? -1 : 0, m_hi2 = hi2 ? -1 : 0;
  auto sel = [](int m, int x, int y) __attribute__((always_inline)) {
    return (m & x) | (~m & y);
  };
  auto pair_rows = [&](const v4i& d, int* r) __attribute__((always_inline)) {
#pragma unroll
    for (int k = 0; k < 2; ++k) {
      const int keep = sel(m_odd, d[2 * k + 1], d[2 * k]) << wsh;
      const int send = sel(m_odd, d[2 * k], d[2 * k + 1]) << wsh;
      r[k] = keep + (int)dpp<0xB1>((unsigned)send);
    }
  };
  // Weights of the lane's own digit pair and of the pair its partner sends.
  const double w_own = CPH >= 8 && hi4 ? 1.0 : hi2 ? 0x1p16 : 0x1p32;
  const double w_oth = CPH >= 8 && hi4 ? 0.0 : hi2 ? 0x1p32 : 0x1p16;

  // Logits (log2 units) of the lane's RN rows.
  auto logits = [&](const Buf& f, double* lg) __attribute__((always_inline)) {
    v4i ds[G::NSET];
#pragma unroll
    for (int kb = 0; kb < G::NB; ++kb) {
      const unsigned w0 = f.k[2 * kb], w1 = f.k[2 * kb + 1];
      const v4i ak = v4i{(int)(w0 & 0x0F0F0F0Fu), (int)(w1 & 0x0F0F0F0Fu),
                         (int)((w0 >> 4) & 0x0F0F0F0Fu), (int)((w1 >> 4) & 0x0F0F0F0Fu)};
#pragma unroll
      for (int s = 0; s < G::NSET; ++s)
        ds[s] = __builtin_amdgcn_mfma_i32_16x16x64_i8(ak, bq[s][kb],
                                                      kb == 0 ? v4i{0, 0, 0, 0} : ds[s], 0, 0, 0);
    }
    if constexpr (CPH == 2) {
      int p[3][2];
#pragma unroll
      for (int s = 0; s < 3; ++s) pair_rows(ds[s], p[s]);
#pragma unroll
      for (int k = 0; k < 2; ++k) {
        const double s = __builtin_fma((double)p[0][k], 0x1p32,
                                       __builtin_fma((double)p[1][k], 0x1p16, (double)p[2][k]));
        lg[k] = __builtin_fma(s, c1, -cg);
      }
    } else {
      int p[2];
      pair_rows(ds[0], p);
      const int own = sel(m_hi2, p[1], p[0]);
      const int oth = (int)dpp<0x4E>((unsigned)sel(m_hi2, p[0], p[1]));
      double s;
      if constexpr (CPH == 4) {
        int r[2];
        pair_rows(ds[1], r);
        s = __builtin_fma((double)own, w_own,
                          __builtin_fma((double)oth, w_oth, (double)sel(m_hi2, r[1], r[0])));
      } else {
        s = __builtin_fma((double)own, w_own, (double)oth * w_oth);
        s += xchg4_dpp(s);
      }
      lg[0] = __builtin_fma(s, c1, -cg);
    }
  };

  // Float32 products of the values with the four rows' probabilities x, added
  // to the accumulators rescaled by corr. A chunk's rows are summed by
  // themselves first, in two chains of eight: one rounding per chunk reaches
  // the running sum, not one per row (measured against one chain through all
  // rows: 2.3e-7 -> 1.9e-7 of the result at T 15000).
  auto value_f32 = [&](const Buf& f, const float* x, float corr) __attribute__((always_inline)) {
#pragma unroll
    for (int u = 0; u < G::NP; ++u)
#pragma unroll
      for (int j = 0; j < G::CPP; ++j) {
        v4f t[2] = {{0.f, 0.f, 0.f, 0.f}, {0.f, 0.f, 0.f, 0.f}};
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          t[i / 2] = __builtin_amdgcn_mfma_f32_16x16x4f32(u2f(f.v[i][u][j]), x[i], t[i / 2],
                                                          0, 0, 0);
        }
        v4f& o = acc[u * G::CPP + j];
#pragma unroll
        for (int i = 0; i < 4; ++i) o[i] = __builtin_fmaf(o[i], corr, t[0][i] + t[1][i]);
      }
  };

  // The same with 16-bit values, for the rare chunks whose probabilities or
  // values the 16-bit products below would not hold: products added to the
  // accumulators one after the other, which takes no registers for chunk sums
  // (those would cost every chunk a wave of occupancy).
  auto value_wide = [&](const Buf& f, const float* x) __attribute__((always_inline)) {
#pragma unroll
    for (int u = 0; u < G::NP; ++u)
#pragma unroll
      for (int j = 0; j < G::CPP; ++j)
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const unsigned w = f.v[i][u][j / 2];
          float v;
          if constexpr (VDT == kVF16)
            v = (float)__builtin_bit_cast(_Float16, (unsigned short)(w >> (16 * (j & 1))));
          else
            v = u2f(j & 1 ? w & 0xFFFF0000u : w << 16);
          v4f& t = acc[u * G::CPP + j];
          t = __builtin_amdgcn_mfma_f32_16x16x4f32(v, x[i], t, 0, 0, 0);
        }
  };

  // Upper bits of a probability that one 16-bit term holds.
  constexpr unsigned kTerm = VDT == kVF16 ? 0xFFFFE000u : 0xFFFF0000u;
  // Two terms packed as the 16-bit type: the bits below a term's are dropped.
  auto pack2 = [&](float lo, float hi) __attribute__((always_inline)) -> unsigned {
    if constexpr (VDT == kVF16)
      return __builtin_bit_cast(unsigned, __builtin_amdgcn_cvt_pkrtz(lo, hi));
    else
      return __builtin_amdgcn_perm(f2u(hi), f2u(lo), 0x07060302u);
  };
  // Bits of a probability that go to earlier columns, first term and second; at
  // HG = 8 what the second product of column 0 leaves out is everything.
  const unsigned term1 = col >= 1 ? kTerm : 0u;
  const unsigned term2 = CPH == 2 ? (col == 0 ? ~0u : kTerm) : (col >= 2 ? kTerm : 0u);
  const float rest = col >= 1 ? kRestScale : 1.f;

  // 16-bit products of the values with the terms of the probabilities x.
  auto value_16 = [&](const Buf& f, const float* x) __attribute__((always_inline)) {
    unsigned bt[4];
    if constexpr (CPH == 2) {
      // Column 0: first term, then nothing; column 1: second, then third term.
      float ta[4], tb[4];
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        ta[i] = x[i] - u2f(f2u(x[i]) & term1);
        tb[i] = ta[i] - u2f(f2u(ta[i]) & term2);
      }
      bt[0] = pack2(ta[0], ta[1]);
      bt[1] = pack2(ta[2], ta[3]);
      bt[2] = pack2(tb[0], tb[1]);
      bt[3] = pack2(tb[2], tb[3]);
    } else {
      // Column c: term c (columns 3 and beyond repeat term 2 and are dropped).
      // (Masks keep leading bits, so the columns' scale may come before them.)
      float t[4];
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        t[i] = x[i] - u2f(f2u(x[i]) & term1);
        t[i] = t[i] - u2f(f2u(t[i]) & term2);
      }
      bt[0] = pack2(t[0], t[1]);
      bt[1] = pack2(t[2], t[3]);
      bt[2] = bt[3] = 0;
    }
#pragma unroll
    for (int u = 0; u < G::NP; ++u)
#pragma unroll
      for (int j = 0; j < G::CPP; ++j) {
        const unsigned sel = j & 1 ? 0x07060302u : 0x05040100u;
        const unsigned a0 = __builtin_amdgcn_perm(f.v[1][u][j / 2], f.v[0][u][j / 2], sel);
        const unsigned a1 = __builtin_amdgcn_perm(f.v[3][u][j / 2], f.v[2][u][j / 2], sel);
        v4f& t = acc[u * G::CPP + j];
        const uint2 av = make_uint2(a0, a1);
#pragma unroll
        for (int q = 0; q < (CPH == 2 ? 2 : 1); ++q) {
          const uint2 bv = make_uint2(bt[2 * q], bt[2 * q + 1]);
          if constexpr (VDT == kVF16)
            t = __builtin_amdgcn_mfma_f32_16x16x16f16(__builtin_bit_cast(v4h, av),
                                                      __builtin_bit_cast(v4h, bv), t, 0, 0, 0);
          else
            t = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(__builtin_bit_cast(v4s, av),
                                                          __builtin_bit_cast(v4s, bv), t, 0, 0, 0);
        }
      }
  };

  // Consume one chunk of nval > 0 rows. wide: float32 products also for 16-bit
  // values.
  auto consume = [&](Buf& f, int nval, bool wide) __attribute__((always_inline)) {
    double lg[RN];
    logits(f, lg);
    float mc = -INFINITY;
#pragma unroll
    for (int k = 0; k < RN; ++k) {
      lg[k] = lrow + 2 * k < nval ? lg[k] : -INFINITY;
      mc = max_raw(mc, (float)lg[k]);
    }
    mc = max_raw(mc, xchg<1>(mc));
    if constexpr (CPH >= 4) mc = max_raw(mc, xchg<2>(mc));
    mc = groups_max(mc);
    // The shift: the maximum of the rounded logits, brought up to a whole number,
    // so that every factor between shifts (chunks, waves, splits) is an exact
    // power of two -- from 2^20 up, where a float32 logit is off by 1/16 and more,
    // the double maximum. A probability exceeds 1 by a factor 2^(1/16) at most.
    double mx = __builtin_ceil((double)mc);
    if (__builtin_expect(
            __builtin_amdgcn_ballot_w64(!(__builtin_fabsf(mc) < 0x1p20f)) != 0, 0)) {
      mx = lg[0];
      if constexpr (RN > 1) mx = fmax(mx, lg[RN - 1]);
      mx = __builtin_ceil(allreduce_max<16, 64>(allreduce_max<1, (CPH >= 4 ? 4 : 2)>(mx)));
    }
    const double m_new = max_raw(m_run, mx);
    const float corr = __builtin_amdgcn_exp2f((float)(m_run - m_new));
    m_run = m_new;
    float p[RN], psum = 0.f;
#pragma unroll
    for (int k = 0; k < RN; ++k) {
      p[k] = __builtin_amdgcn_exp2f((float)(lg[k] - m_new)) * kPScale;
      psum += p[k];
    }
    l_run = l_run * corr + psum;
    // Most chunks do not move the maximum of any head.
    if (VDT != kVF32 && __builtin_amdgcn_ballot_w64(corr != 1.f)) {
#pragma unroll
      for (int t = 0; t < G::NA; ++t) acc[t] *= corr;
    }
    float x[4];
    if constexpr (CPH >= 4) {
      x[0] = u2f(dpp<0x00>(f2u(p[0])));
      x[1] = u2f(dpp<0x55>(f2u(p[0])));
      x[2] = u2f(dpp<0xAA>(f2u(p[0])));
      x[3] = u2f(dpp<0xFF>(f2u(p[0])));
    } else {
      x[0] = u2f(dpp<0xA0>(f2u(p[0])));
      x[1] = u2f(dpp<0xF5>(f2u(p[0])));
      x[2] = u2f(dpp<0xA0>(f2u(p[RN - 1])));
      x[3] = u2f(dpp<0xF5>(f2u(p[RN - 1])));
    }
    if constexpr (VDT == kVF16) {
#pragma unroll
      for (int i = 0; i < 4; ++i) x[i] *= rest;
    }
    // Rows past the valid ones hold the last valid row: zeros in its place, lest
    // an infinity there times their probability 0 be NaN. (The 16-bit products
    // leave such a NaN to the run with float32 ones.)
    if ((VDT == kVF32 || wide) && nval < 16) {
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const unsigned keep = 4 * grp + i < nval ? ~0u : 0u;
#pragma unroll
        for (int u = 0; u < G::NP; ++u)
#pragma unroll
          for (int k = 0; k < G::PB / 4; ++k) f.v[i][u][k] &= keep;
      }
    }
    if constexpr (VDT == kVF32) {
      value_f32(f, x, corr);
    } else if (wide) {
      value_wide(f, x);
    } else {
      if constexpr (VDT == kVF16) {
        bool small = false;   // 0 < p < kLeastP
#pragma unroll
        for (int k = 0; k < RN; ++k) small |= f2u(p[k]) - 1u < f2u(kLeastP) - 1u;
        if (__builtin_expect(__builtin_amdgcn_ballot_w64(small) != 0, 0)) {
          // The float32 products, in column 0, and then 16-bit products of
          // nothing: with those in the other branch the accumulators would be
          // copied where the branches meet, in every chunk.
          float x0[4];
#pragma unroll
          for (int i = 0; i < 4; ++i) {
            x0[i] = col == 0 ? x[i] : 0.f;
            x[i] = 0.f;
          }
          value_wide(f, x0);
        }
      }
      value_16(f, x);
    }
  };

  // One step: (1) rebuild for a new scale group, (2) load the next chunk and its
  // scale block (past the end one row of the last chunk, so that every step
  // issues the same loads and the wait counts stay exact), (3) read the
  // page-table entry of the chunk after that on the scalar unit, (4) consume
  // chunk c. Called with the two buffers in turn, so no register copy waits on a
  // load.
  int c = wc0;
  ChunkPos np{};
  PosMeta cur, next;          // of chunks c and c + 1
  U32x4 sz[G::SZL];
  auto next_meta = [&](int ci) __attribute__((always_inline)) -> PosMeta {
    if (ci < wc1) np = chunk_next(np, cpp, ppg);
    return pos_meta(a, pgm, T, np);
  };
  auto step = [&](Buf& f, Buf& nf) __attribute__((always_inline)) -> bool {
    if (cur.group != cur_group) {
      rebuild(sz);
      cur_group = cur.group;
    }
    load_sz(next, sz);
    load_chunk(next, c + 1 >= wc1 ? 1 : next.nval, nf);
    const PosMeta ahead = next_meta(c + 2);
    if (cur.nval > 0) consume(f, cur.nval, false);
    cur = next;
    next = ahead;
    c += 1;
    return c >= wc1;
  };

  const bool has_work = wc0 < wc1;
  Buf f[2];
  auto first_loads = [&]() __attribute__((always_inline)) {
    np = chunk_pos(a, wc0, cpp);
    cur = pos_meta(a, pgm, T, np);
    next = next_meta(wc0 + 1);
    load_sz(cur, sz);
    load_chunk(cur, cur.nval, f[0]);
  };
  auto clear = [&]() __attribute__((always_inline)) {
#pragma unroll
    for (int t = 0; t < G::NA; ++t) acc[t] = v4f{0.f, 0.f, 0.f, 0.f};
  };
  if (has_work) first_loads();
#pragma unroll
  for (int j = 0; j < QPT; ++j) {
    const int idx = tid + j * NT;
    if (idx < HG * D) q_s[idx / D][slot_of(idx % D)] = qv[j];
  }
  clear();
  __syncthreads();
  if (has_work) {
    while (true) {
      if (step(f[0], f[1])) break;
      if (step(f[1], f[0])) break;
    }
  }

  if constexpr (VDT != kVF32) {
    // Columns beyond the three terms hold nothing.
    int cols = CPH == 2 ? 2 : 3;
    bool bad = false;
#pragma unroll
    for (int t = 0; t < G::NA; ++t)
#pragma unroll
      for (int i = 0; i < 4; ++i) bad |= !(acc[t][i] == acc[t][i]);
    if (__builtin_amdgcn_ballot_w64(bad)) {
      // Rare (an infinite or NaN value or query): the range again, one chunk at
      // a time, with float32 products, whose columns are all the full sum.
      clear();
      m_run = -INFINITY;
      l_run = 0.f;
      cols = 1;
      ChunkPos p = chunk_pos(a, wc0, cpp);
      for (int ci = wc0; ci < wc1; ++ci) {
        const PosMeta m = pos_meta(a, pgm, T, p);
        load_sz(m, sz);
        load_chunk(m, m.nval, f[0]);
        if (m.group != cur_group) {
          rebuild(sz);
          cur_group = m.group;
        }
        if (m.nval > 0) consume(f[0], m.nval, true);
        p = chunk_next(p, cpp, ppg);
      }
    }
    // The terms' columns add up, each taken back by its scale.
    const float back = col == 0 ? 1.f / kPScale : 1.f / (kPScale * kRestScale);
#pragma unroll
    for (int t = 0; t < G::NA; ++t)
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const float x = col < cols ? acc[t][i] * back : 0.f;
        acc[t][i] = allreduce_sum<1, (CPH >= 4 ? 4 : 2)>(x);
      }
  }

  // Wave totals per head to LDS (over the wave's digits), then the log-sum-exp
  // merge of the waves.
  const float l_tot =
      allreduce_sum<16, 64>(allreduce_sum<1, (CPH >= 4 ? 4 : 2)>(l_run)) * (1.f / kPScale);
  float* acc_w = reinterpret_cast<float*>(wave_s[w]) + hh * D;
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  if (col == 0) {
#pragma unroll
    for (int u = 0; u < G::NP; ++u)
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        float* dst = acc_w + u * 16 * G::CPP + (4 * grp + i) * G::CPP;
#pragma unroll
        for (int j = 0; j < G::CPP; j += 4)
          *reinterpret_cast<float4*>(dst + j) =
              make_float4(acc[u * G::CPP + j][i], acc[u * G::CPP + j + 1][i],
                          acc[u * G::CPP + j + 2][i], acc[u * G::CPP + j + 3][i]);
      }
    if (grp == 0) {
      m_s[w][hh] = m_run;
      l_s[w][hh] = l_tot;
    }
  }
  __syncthreads();

  // Four channels a thread: the waves' weights once, 16-byte reads and stores.
  for (int idx = tid * 4; idx < HG * D; idx += NT * 4) {
    const int h = idx / D, d = idx % D;
    double ms = -INFINITY;
#pragma unroll
    for (int i = 0; i < WAVES; ++i) ms = fmax(ms, m_s[i][h]);
    // Weighted waves, then their sum as a tree (the weights are powers of two, so
    // only its additions round; as one chain they were the larger part of a short
    // sequence's error).
    float l[WAVES], o[WAVES][4];
#pragma unroll
    for (int i = 0; i < WAVES; ++i) {
      const float e =
          (m_s[i][h] == -INFINITY) ? 0.f : __builtin_amdgcn_exp2f((float)(m_s[i][h] - ms));
      const float4 x = *reinterpret_cast<const float4*>(
          reinterpret_cast<const float*>(wave_s[i]) + idx);
      const float xs[4] = {x.x, x.y, x.z, x.w};
      if (i & 1) {
        l[i / 2] = __builtin_fmaf(e, l_s[i][h], l[i / 2]);
#pragma unroll
        for (int k = 0; k < 4; ++k) o[i / 2][k] = __builtin_fmaf(e, xs[k], o[i / 2][k]);
      } else {
        l[i / 2] = e * l_s[i][h];
#pragma unroll
        for (int k = 0; k < 4; ++k) o[i / 2][k] = e * xs[k];
      }
    }
#pragma unroll
    for (int n = WAVES / 4; n > 0; n /= 2)
#pragma unroll
      for (int i = 0; i < n; ++i) {
        l[i] = l[2 * i] + l[2 * i + 1];
#pragma unroll
        for (int k = 0; k < 4; ++k) o[i][k] = o[2 * i][k] + o[2 * i + 1][k];
      }
    const int hq = h0 + h;
    if (a.final_out) {
      const float r = fmaxf(l[0], 1e-10f);
#pragma unroll
      for (int k = 0; k < 4; ++k)
        store_elem(a.out, (int64_t)b * a.o_b + (int64_t)hq * a.o_h + d + k, a.out_dtype,
                   o[0][k] / r);
    } else {
      const int64_t pi = ((int64_t)b * a.num_q_heads + hq) * a.num_splits + split;
      *reinterpret_cast<float4*>(a.ws_acc + pi * D + d) = make_float4(o[0][0], o[0][1], o[0][2], o[0][3]);
      if (d == 0) {
        a.ws_ml[2 * pi] = ms * 0.6931471805599453;   // natural log units
        a.ws_ml[2 * pi + 1] = (double)l[0];
      }
    }
  }
  hand_back_length(a, b);
}

hipError_t launch_decode_mfma(const DecodeArgs& a, int D, int v_dtype, int batch, int hg,
                              hipStream_t st) {
  dim3 grid(a.num_splits, a.num_q_heads / hg, batch);
#define FDI4_MF(DD, VV, WW, HH)                                                            \
  if (D == DD && v_dtype == VV && a.waves == WW && hg == HH) {                             \
    hipLaunchKernelGGL((decode_mfma_kernel<DD, VV, WW, HH>), grid, dim3(WW * 64), 0, st, a); \
    return hipGetLastError();                                                              \
  }
#define FDI4_MF_V(DD, WW, HH) \
  FDI4_MF(DD, kVF32, WW, HH) FDI4_MF(DD, kVF16, WW, HH) FDI4_MF(DD, kVBF16, WW, HH)
#define FDI4_MF_H(WW, HH) FDI4_MF_V(64, WW, HH) FDI4_MF_V(128, WW, HH)
  FDI4_MF_H(4, 2) FDI4_MF_H(8, 2) FDI4_MF_H(4, 4) FDI4_MF_H(8, 4)
  FDI4_MF_H(4, 8) FDI4_MF_H(8, 8)
  FDI4_MF_V(256, 4, 2) FDI4_MF_V(256, 4, 4)   // four waves only, see plan_decode
#undef FDI4_MF_H
#undef FDI4_MF_V
#undef FDI4_MF
  return hipErrorInvalidValue;
}

}  // namespace fdi4
