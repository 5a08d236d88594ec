// HIP kernels for the zeroth-order (ZO) step and the DiZO projection, gfx950.
//
// All arithmetic reproduces PyTorch's elementwise recipe bit for bit: every
// operation is one IEEE fp32 operation on fp32-widened operands followed by a
// round-to-nearest-even conversion to the parameter dtype T (identity for
// fp32). Products are never contracted into FMAs (the file is compiled with
// -ffp-contract=off and the pragma below), and dz_opq() keeps the backend from
// folding an fp32 multiply and its fp16 conversion into one mixed-precision
// FMA (which would round once instead of twice and flip the sign of zeros).
#include <hip/hip_ext.h>
#include <hip/hip_runtime.h>
#include <stdint.h>

#include <type_traits>

#include "dz_common.h"
#include "dz_kernels.h"

#pragma clang fp contract(off)

namespace dz {

template <int DT>
struct DT_;

template <>
struct DT_<DZ_F32> {
  using S = uint32_t;
  static constexpr int kBits = 32;
  __device__ static __forceinline__ float to_f(uint32_t b) { return __uint_as_float(b); }
  __device__ static __forceinline__ uint32_t from_f(float f) { return __float_as_uint(f); }
};

template <>
struct DT_<DZ_F16> {
  using S = uint16_t;
  static constexpr int kBits = 16;
  __device__ static __forceinline__ float to_f(uint32_t b) {
    return dz_opq((float)__builtin_bit_cast(_Float16, (uint16_t)b));
  }
  __device__ static __forceinline__ uint32_t from_f(float f) {
    return (uint32_t)__builtin_bit_cast(uint16_t, (_Float16)dz_opq(f));
  }
};

template <>
struct DT_<DZ_BF16> {
  using S = uint16_t;
  static constexpr int kBits = 16;
  __device__ static __forceinline__ float to_f(uint32_t b) { return __uint_as_float(b << 16); }
  __device__ static __forceinline__ uint32_t from_f(float f) {
    return (uint32_t)__builtin_bit_cast(uint16_t, (__bf16)dz_opq(f));
  }
};

// R_T(x): round an fp32 result to T and widen back.
template <int DT>
__device__ __forceinline__ float rt(float x) {
  if constexpr (DT == DZ_F32) {
    return x;
  } else {
    return DT_<DT>::to_f(DT_<DT>::from_f(x));
  }
}

// ---------------------------------------------------------------------------
// Per-element operations (theta and z are fp32-widened values of T).
// ---------------------------------------------------------------------------

// trainer.py:1442   param.data + scaling_factor * z * eps
template <int DT>
__device__ __forceinline__ uint32_t op_perturb(float th, float z, float s, float eps) {
  const float a = rt<DT>(s * z);
  const float b = rt<DT>(a * eps);
  return DT_<DT>::from_f(th + b);
}

// trainer.py:1608   param.data - lr * (projected_grad * z)
template <int DT>
__device__ __forceinline__ uint32_t op_update(float th, float z, float g, float lr) {
  const float c = rt<DT>(g * z);
  const float d = rt<DT>(lr * c);
  return DT_<DT>::from_f(th - d);
}

template <int DT>
__device__ __forceinline__ float load_scalar_T(const void* p) {
  return DT_<DT>::to_f((uint32_t)(*(const typename DT_<DT>::S*)p));
}

template <int DT>
__device__ __forceinline__ DzScalars resolve_scalars(DzScalars s, const DzScalarPtrs& p) {
  if (p.seed) s.seed = *p.seed;
  if (p.seed2) s.seed2 = *p.seed2;
  if (p.grad) s.grad = load_scalar_T<DT>(p.grad);
  if (p.lr) s.lr = *p.lr;
  return s;
}

__device__ __forceinline__ uint32_t word_of(const DzU4& w, int i) {
  return i == 0 ? w.x : i == 1 ? w.y : i == 2 ? w.z : w.w;
}

// ---------------------------------------------------------------------------
// Per-launch delta tables.
//
// Every z is +-Q_T[i] for a 15-bit index i, and each of the reference's
// per-element expressions adds an odd function of z to theta:
//   perturb  theta' = R(theta + b),     b = R(R(s*z)*eps)      trainer.py:1442
//   update   theta' = R(theta - d),     d = R(lr*R(g*z))       trainer.py:1608
//                   = R(theta + (-d))   (x - y is x + (-y) in IEEE arithmetic,
//                                        signed zeros included)
// RNE rounding is symmetric in sign, so b(-z) = -b(z) and d(-z) = -d(z). A
// launch evaluates b, or -d, once per table index (32768 entries in LDS, with
// exactly the arithmetic above), and each element then costs one lookup, a
// sign flip and the final add. The fused restore+update keeps the pair
// (b, -d) per entry for 16-bit T. For 16-bit T the final add is done in T:
// fp16 adds natively; bf16 adds in fp32 and rounds to bf16 (the reference's
// own recipe). fp32 carries 24 >= 2p+2 significand bits for p = 11, so the
// fp16 sum rounded once equals the fp32 sum rounded to fp16.
// fp32 tables hold the fp32 delta bits, or for restore+update z itself (the
// pair would not fit in LDS) with b and d evaluated per element.
// ---------------------------------------------------------------------------
template <int DT, int MODE>
struct RmwTraits {
  static constexpr bool kWide = (DT == DZ_F32 || rmw_pair_mode(MODE));
  using E = typename std::conditional<kWide, uint32_t, uint16_t>::type;
  static constexpr int kGroups = rmw_groups(DT, MODE);
  static constexpr int kChunk = rmw_chunk_elems(DT, MODE);
  static constexpr bool kPrefetch = rmw_prefetch_mode(DT, MODE);
};
// Waves per SIMD of an RMW launch: one 1024-thread workgroup per CU, 4 waves
// per SIMD (up to 128 VGPRs per lane).
constexpr int kRmwWavesPerEU = 4;

// bf16 pair tables (restore + update, and with the next perturbation) hold
// each entry's 16-bit halves xor-ed with their own index i: a z field
// h = sign << 15 | i then turns entry i into its signed value with one xor
// against h (i ^ i = 0 and the sign lands on bit 15, the value's sign), which
// a word-selecting xor does for one operand of a packed word at a time
// (xor_hi below). It takes the bf16 three-way pass from 171 to 151 VALU
// instructions per 8-element group; for the single-value bf16 tables of
// perturb and update it measured 0.6-1.8 % slower (HBM-bound passes, same
// box, alternating builds), so they keep plain entries. fp16 applies the
// signs as packed FMA factors.
__host__ __device__ constexpr bool rmw_index_xor(int dt, int mode) {
  return dt == DZ_BF16 && rmw_pair_mode(mode);
}
// What of a z field h is xor-ed into its table entry's halves.
template <int DT, int MODE>
__device__ __forceinline__ uint32_t field_xor(uint32_t h) {
  return rmw_index_xor(DT, MODE) ? (h & 0xffffu) : (h & 0x8000u);
}

typedef _Float16 dz_half2 __attribute__((ext_vector_type(2)));
typedef __bf16 dz_bf2 __attribute__((ext_vector_type(2)));

// bf16 lanes of a packed word as fp32 (a bf16 value is the high half of its
// fp32 bit pattern), and two fp32 values rounded to bf16 and packed by one
// v_cvt_pk_bf16_f32 (round to nearest even, as torch converts fp32 to bf16).
__device__ __forceinline__ float bf16_lo_f(uint32_t x) { return __uint_as_float(x << 16); }
__device__ __forceinline__ float bf16_hi_f(uint32_t x) { return __uint_as_float(x & 0xffff0000u); }
__device__ __forceinline__ uint32_t pack_bf16(float lo, float hi) {
  const dz_bf2 r = {(__bf16)lo, (__bf16)hi};
  return __builtin_bit_cast(uint32_t, r);
}
// Low (pack_lo) or high (pack_hi) 16-bit halves of two words, a's in the low
// lane and b's in the high lane: one v_perm_b32.
__device__ __forceinline__ uint32_t pack_lo(uint32_t a, uint32_t b) {
  return __builtin_amdgcn_perm(b, a, 0x05040100u);
}
__device__ __forceinline__ uint32_t pack_hi(uint32_t a, uint32_t b) {
  return __builtin_amdgcn_perm(b, a, 0x07060302u);
}

// The two 16-bit lanes of a packed word as fp32, and two fp32 values rounded
// to T and packed: one conversion instruction each way.
struct F32Pair {
  float lo, hi;
};
template <int DT>
__device__ __forceinline__ F32Pair widen_pair(uint32_t x) {
  return F32Pair{DT_<DT>::to_f(x & 0xffffu), DT_<DT>::to_f(x >> 16)};
}
template <int DT>
__device__ __forceinline__ uint32_t round_pair(float lo, float hi) {
  if constexpr (DT == DZ_F16) {
    const dz_half2 r = {(_Float16)dz_opq(lo), (_Float16)dz_opq(hi)};
    return __builtin_bit_cast(uint32_t, r);
  } else {
    return pack_bf16(dz_opq(lo), dz_opq(hi));
  }
}
// b = R(R(s z) eps) of two packed signed z. kUnit: s is 1 (the fused modes'
// perturbations), so R(s z) is z.
template <int DT, bool kUnit>
__device__ __forceinline__ uint32_t delta_b_pair(uint32_t z, const DzScalars& sc) {
  F32Pair a = widen_pair<DT>(z);
  if constexpr (!kUnit) a = widen_pair<DT>(round_pair<DT>(sc.scale * a.lo, sc.scale * a.hi));
  return round_pair<DT>(a.lo * sc.eps, a.hi * sc.eps);
}
// -d = -R(lr R(g z)) of two packed signed z.
template <int DT>
__device__ __forceinline__ uint32_t delta_nd_pair(uint32_t z, const DzScalars& sc) {
  const F32Pair a = widen_pair<DT>(z);
  const F32Pair c = widen_pair<DT>(round_pair<DT>(sc.grad * a.lo, sc.grad * a.hi));
  return round_pair<DT>(sc.lr * c.lo, sc.lr * c.hi) ^ 0x80008000u;
}
// fp32 table entry for z = +Q_T[i] (qbits = its bits): the launch's delta, or
// for the pair modes z itself.
template <int MODE>
__device__ __forceinline__ uint32_t table_entry_f32(uint32_t qbits, const DzScalars& sc) {
  const float z = __uint_as_float(qbits);
  if constexpr (MODE == kModePerturb) return __float_as_uint((sc.scale * z) * sc.eps);
  if constexpr (MODE == kModeUpdate) return __float_as_uint(sc.lr * (sc.grad * z)) ^ 0x80000000u;
  return qbits;
}

typedef uint32_t dz_u32x4 __attribute__((ext_vector_type(4)));

// The launch's delta table, built by the 1024 threads of a workgroup in two
// steps: each thread loads its 16-byte slices of Q_T (4 fp32 or 8 16-bit
// entries; slice t + v * 1024), all loads in flight at once (load_table), then
// writes the slices' entries to the same indices of the LDS table
// (store_table). A plain loop of one 32-bit load, a wait and one LDS store
// per entry costs 32 memory latencies in a row per launch. 16-bit entries are
// evaluated two at a time (one rounding conversion for both): entry by entry,
// the three-way pass took 1 (fp16) to 2 us (bf16) longer, 40.3 against 38.2 us
// at 2^25.5 bf16 elements.
template <int DT>
struct TableSlices {
  static constexpr int kPer = DT == DZ_F32 ? 4 : 8;  // Q_T entries per 16-byte slice
  static constexpr int kSlices = kDzTabEntries / (kRmwThreads * kPer);
  static_assert(kSlices * kRmwThreads * kPer == kDzTabEntries, "table slices");
  dz_u32x4 q[kSlices];
};

template <int DT>
__device__ __forceinline__ void load_table(TableSlices<DT>& t, const void* qtab) {
#pragma unroll
  for (int v = 0; v < TableSlices<DT>::kSlices; ++v)
    t.q[v] = *(const dz_u32x4*)((const char*)qtab + (size_t)(v * kRmwThreads + threadIdx.x) * 16);
}

template <int DT, int MODE>
__device__ __forceinline__ void store_table(typename RmwTraits<DT, MODE>::E* tab, const TableSlices<DT>& t,
                                            const DzScalars& sc) {
  constexpr int kPer = TableSlices<DT>::kPer;
#pragma unroll
  for (int v = 0; v < TableSlices<DT>::kSlices; ++v) {
    const uint32_t i0 = (uint32_t)(v * kRmwThreads + threadIdx.x) * kPer;
    dz_u32x4* dst = (dz_u32x4*)(tab + i0);
    if constexpr (DT == DZ_F32) {
      dz_u32x4 o;
#pragma unroll
      for (int i = 0; i < 4; ++i) o[i] = table_entry_f32<MODE>(t.q[v][i], sc);
      dst[0] = o;
    } else if constexpr (!rmw_pair_mode(MODE)) {  // two 16-bit entries a word
      dz_u32x4 o;
#pragma unroll
      for (int i = 0; i < 4; ++i)
        o[i] = MODE == kModePerturb ? delta_b_pair<DT, false>(t.q[v][i], sc) : delta_nd_pair<DT>(t.q[v][i], sc);
      dst[0] = o;
    } else {  // entries b | (-d) << 16
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        dz_u32x4 o;
#pragma unroll
        for (int i = 0; i < 2; ++i) {
          const uint32_t q = t.q[v][2 * h + i];
          const uint32_t b = delta_b_pair<DT, true>(q, sc), nd = delta_nd_pair<DT>(q, sc);
          o[2 * i] = pack_lo(b, nd);
          o[2 * i + 1] = pack_hi(b, nd);
          if constexpr (rmw_index_xor(DT, MODE)) {
            const uint32_t at = i0 + 4 * h + 2 * i;
            o[2 * i] ^= at * 0x10001u;
            o[2 * i + 1] ^= (at + 1) * 0x10001u;
          }
        }
        dst[h] = o;
      }
    }
  }
}

// R_bf16(a + b) lane by lane for packed bf16 words, the fp32 sums written out.
__device__ __forceinline__ uint32_t add_pair_bf16(uint32_t a, uint32_t b) {
  return pack_bf16(bf16_lo_f(a) + bf16_lo_f(b), bf16_hi_f(a) + bf16_hi_f(b));
}
// R_bf16(x) as an fp32 value: v_cvt_pk_bf16_f32 with a zero low lane leaves
// the rounded bf16 in the high half and zeros below it, which is the fp32
// bit pattern of the rounded value (no unpacking before the next fp32 add).
// Written as the instruction: from pack_bf16(0.0f, x) the compiler converts
// into the low lane and moves the result up with a v_perm_b32.
__device__ __forceinline__ float round_bf16_f(float x) {
  uint32_t r;
  asm("v_cvt_pk_bf16_f32 %0, 0, %1" : "=v"(r) : "v"(x));
  return __uint_as_float(r);
}

// R_T(a + b) for a pair of 16-bit values packed in one word: fp16 adds
// natively (v_pk_add_f16); bf16 adds in fp32 and rounds both lanes with one
// v_cvt_pk_bf16_f32 (RNE). Either equals the reference's fp32 add rounded
// to T: fp32 holds at least 2p + 2 bits of a p-bit format. (Written out for
// bf16: the compiler's own bf16 vector add issued about 5 conversions per
// three-add chain of a word instead of 3.)
template <int DT>
__device__ __forceinline__ uint32_t add_pair(uint32_t a, uint32_t b) {
  if constexpr (DT == DZ_F16) {
    const dz_half2 x = __builtin_bit_cast(dz_half2, a);
    const dz_half2 y = __builtin_bit_cast(dz_half2, b);
    return __builtin_bit_cast(uint32_t, x + y);
  } else {
    return add_pair_bf16(a, b);
  }
}

// (half EH of e) ^ (half WH of w), placed in the high half over a zero low
// half: the fp32 pattern of the bf16 value it holds. Two high halves are one
// v_bitop3_b32 ((e ^ w) & 0xffff0000); the other forms are one word-selecting
// (SDWA) xor: each source reads bits 0..15 or 16..31 zero-extended, and the
// result's bits 0..15 are written to bits 16..31 with zeros below. (Written
// as the instruction: from the shift-and-xor expression the compiler forms it
// for only some of the uses.)
template <int EH, int WH>
__device__ __forceinline__ float xor_hi(uint32_t e, uint32_t w) {
  uint32_t r;
  if constexpr (EH == 1 && WH == 1)
    r = (e ^ w) & 0xffff0000u;
  else if constexpr (EH == 0 && WH == 0)
    asm("v_xor_b32_sdwa %0, %1, %2 dst_sel:WORD_1 dst_unused:UNUSED_PAD src0_sel:WORD_0 src1_sel:WORD_0"
        : "=v"(r) : "v"(e), "v"(w));
  else if constexpr (EH == 0)
    asm("v_xor_b32_sdwa %0, %1, %2 dst_sel:WORD_1 dst_unused:UNUSED_PAD src0_sel:WORD_0 src1_sel:WORD_1"
        : "=v"(r) : "v"(e), "v"(w));
  else
    asm("v_xor_b32_sdwa %0, %1, %2 dst_sel:WORD_1 dst_unused:UNUSED_PAD src0_sel:WORD_1 src1_sel:WORD_0"
        : "=v"(r) : "v"(e), "v"(w));
  return __uint_as_float(r);
}

// R_T(a + b) for one 16-bit value.
template <int DT>
__device__ __forceinline__ uint32_t add_one(uint32_t a, uint32_t b) {
  if constexpr (DT == DZ_F16) {
    const _Float16 r = __builtin_bit_cast(_Float16, (uint16_t)a) + __builtin_bit_cast(_Float16, (uint16_t)b);
    return (uint32_t)__builtin_bit_cast(uint16_t, r);
  } else {
    return DT_<DT>::from_f(__uint_as_float(a << 16) + __uint_as_float(b << 16));
  }
}

// The two table entries indexed by the 15-bit fields of a z word (bits 0..14
// and 16..30; bits 15 and 31 are the signs). The byte offsets index *
// sizeof(E) take three instructions per word: the sign bits are cleared once,
// then each half is shifted into place by a word-selecting (SDWA) shift, which
// reads bits 0..15 or 16..31 of its operand zero-extended (checked on the
// part against the plain mask-and-shift form). Both offsets are at most
// 0x7fff * sizeof(E), inside the table.
template <typename E>
__device__ __forceinline__ void lookup2(const E* tab, uint32_t w, uint32_t& e0, uint32_t& e1) {
  const uint32_t m = w & 0x7fff7fffu;
  uint32_t a0, a1;
  if constexpr (sizeof(E) == 4) {
    asm("v_lshlrev_b32_sdwa %0, 2, %1 dst_sel:DWORD dst_unused:UNUSED_PAD src0_sel:DWORD src1_sel:WORD_0"
        : "=v"(a0)
        : "v"(m));
    asm("v_lshlrev_b32_sdwa %0, 2, %1 dst_sel:DWORD dst_unused:UNUSED_PAD src0_sel:DWORD src1_sel:WORD_1"
        : "=v"(a1)
        : "v"(m));
  } else {
    asm("v_lshlrev_b32_sdwa %0, 1, %1 dst_sel:DWORD dst_unused:UNUSED_PAD src0_sel:DWORD src1_sel:WORD_0"
        : "=v"(a0)
        : "v"(m));
    asm("v_lshlrev_b32_sdwa %0, 1, %1 dst_sel:DWORD dst_unused:UNUSED_PAD src0_sel:DWORD src1_sel:WORD_1"
        : "=v"(a1)
        : "v"(m));
  }
  e0 = (uint32_t)*(const E*)((const char*)tab + a0);
  e1 = (uint32_t)*(const E*)((const char*)tab + a1);
}

// Table entries of two 16-bit elements whose z fields are the halves of `w`
// (and, for the step-fused mode, whose next-step z fields are the halves of
// w2): the lookups of one packed word.
struct Entries16 {
  uint32_t e0, e1, f0, f1;
};
template <int DT, int MODE>
__device__ __forceinline__ Entries16 lookup_pair16(uint32_t w, uint32_t w2,
                                                   const typename RmwTraits<DT, MODE>::E* tab) {
  Entries16 t;
  lookup2(tab, w, t.e0, t.e1);
  if constexpr (MODE == kModeRestoreUpdatePerturb) {
    lookup2(tab, w2, t.f0, t.f1);
  } else {
    t.f0 = t.f1 = 0u;
  }
  return t;
}

// The two elements' new values from their entries. A field's sign bit (bit
// 15 of its half) negates its table value: for fp16, once the two lanes'
// values are packed, one xor with w & 0x80008000 (or a +-1.0 factor); for
// bf16 the xor_hi that takes each value to its fp32 pattern.
// R(th + sg * v) lane by lane for sg = +-1.0 (fp16): the product is exact, so
// the fused multiply-add rounds th +- v once, as the add of the negated value does.
__device__ __forceinline__ uint32_t fma_sign_pair(uint32_t sg, uint32_t v, uint32_t th) {
  return __builtin_bit_cast(uint32_t, __builtin_elementwise_fma(__builtin_bit_cast(dz_half2, sg),
                                                                __builtin_bit_cast(dz_half2, v),
                                                                __builtin_bit_cast(dz_half2, th)));
}

template <int DT, int MODE>
__device__ __forceinline__ uint32_t combine_pair16(uint32_t th, uint32_t w, uint32_t w2, const Entries16& t) {
  if constexpr (DT == DZ_F16 && rmw_pair_mode(MODE)) {
    // entry = b | (-d) << 16 for a positive z; the signs enter as factors
    // +-1.0 of packed fused multiply-adds (fma_sign_pair), one per add.
    // +-1.0 in each lane: (w & 0x80008000) | 0x3c003c00 as one three-input
    // bitwise op (truth table 0xEA: src0 & src1 | src2)
    const uint32_t sg = __builtin_amdgcn_bitop3_b32(w, 0x80008000u, 0x3c003c00u, 0xEA);
    uint32_t r = fma_sign_pair(sg, pack_hi(t.e0, t.e1), fma_sign_pair(sg, pack_lo(t.e0, t.e1), th));
    if constexpr (MODE == kModeRestoreUpdatePerturb) {
      const uint32_t sg2 = __builtin_amdgcn_bitop3_b32(w2, 0x80008000u, 0x3c003c00u, 0xEA);
      r = fma_sign_pair(sg2, pack_lo(t.f0, t.f1), r);
    }
    return r;
  }
  if constexpr (!rmw_pair_mode(MODE)) {
    return add_pair<DT>(th, (t.e0 | (t.e1 << 16)) ^ (w & 0x80008000u));
  } else {
    // bf16 pairs: entry i = (b ^ i) | ((-d) ^ i) << 16 for a positive z. Each
    // signed value comes out as its fp32 pattern from one xor_hi against the
    // element's z half (element 0: bits 0..15 of w, element 1: bits 16..31).
    // The three adds are the reference's fp32 adds, each rounded to bf16
    // (round_bf16_f for the first two, one packing conversion for the last).
    float lo = round_bf16_f(bf16_lo_f(th) + xor_hi<0, 0>(t.e0, w));
    float hi = round_bf16_f(bf16_hi_f(th) + xor_hi<0, 1>(t.e1, w));
    if constexpr (MODE == kModeRestoreUpdatePerturb) {
      lo = round_bf16_f(lo + xor_hi<1, 0>(t.e0, w));
      hi = round_bf16_f(hi + xor_hi<1, 1>(t.e1, w));
      // the next step's +1 perturbation uses the same b (same scale and eps)
      return pack_bf16(lo + xor_hi<0, 0>(t.f0, w2), hi + xor_hi<0, 1>(t.f1, w2));
    } else {
      return pack_bf16(lo + xor_hi<1, 0>(t.e0, w), hi + xor_hi<1, 1>(t.e1, w));
    }
  }
}

// One element with 16-bit z field h (and next-step field h2).
template <int DT, int MODE>
__device__ __forceinline__ uint32_t apply_one(uint32_t th, uint32_t h, uint32_t h2,
                                              const typename RmwTraits<DT, MODE>::E* tab, const DzScalars& sc) {
  if constexpr (DT == DZ_F32) {
    const uint32_t e = tab[h & 0x7fffu] ^ ((h & 0x8000u) << 16);
    if constexpr (!rmw_pair_mode(MODE)) {
      return __float_as_uint(__uint_as_float(th) + __uint_as_float(e));
    } else {
      const float z = __uint_as_float(e);
      const float th1 = __uint_as_float(op_perturb<DZ_F32>(__uint_as_float(th), z, 1.0f, sc.eps));
      const uint32_t r = op_update<DZ_F32>(th1, z, sc.grad, sc.lr);
      if constexpr (MODE == kModeRestoreUpdatePerturb) {
        const float z2 = __uint_as_float(tab[h2 & 0x7fffu] ^ ((h2 & 0x8000u) << 16));
        return op_perturb<DZ_F32>(__uint_as_float(r), z2, 1.0f, sc.eps);
      }
      return r;
    }
  } else if constexpr (!rmw_pair_mode(MODE)) {
    return add_one<DT>(th, (uint32_t)tab[h & 0x7fffu] ^ field_xor<DT, MODE>(h));
  } else {
    const uint32_t e = tab[h & 0x7fffu] ^ (field_xor<DT, MODE>(h) * 0x10001u);
    uint32_t r = add_one<DT>(add_one<DT>(th, e & 0xffffu), e >> 16);
    if constexpr (MODE == kModeRestoreUpdatePerturb) {
      r = add_one<DT>(r, (tab[h2 & 0x7fffu] ^ field_xor<DT, MODE>(h2)) & 0xffffu);
    }
    return r;
  }
}

// Streaming 16-byte accesses: theta is touched once per pass, so loads and
// stores carry the non-temporal hint. The pointers are global-memory ones
// (address space 1): the accesses then compile to global_load / global_store,
// which count only against the vector-memory wait counter. As generic (FLAT)
// accesses they would also count against the LDS counter, and every wait for
// an LDS table lookup would then wait for the tile loads in flight as well.
//
// The vectors are declared at element alignment: gfx950 takes global accesses
// of every size at any address, and the instruction is the same, so tensors
// that start anywhere (views into a packed buffer) go the same way as aligned
// ones: a bf16 pass over 60 M elements of a packed buffer of odd sizes takes
// 50 us against 96 when its groups went element by element.
typedef dz_u32x4 dz_u32x4_any __attribute__((aligned(2)));
typedef __attribute__((address_space(1))) dz_u32x4_any dz_global_u32x4;
typedef __attribute__((address_space(1))) char dz_global_char;
__device__ __forceinline__ dz_u32x4 ld_stream(const void* p) {
  return __builtin_nontemporal_load((const dz_global_u32x4*)(uintptr_t)p);
}
__device__ __forceinline__ void st_stream(void* p, dz_u32x4 v) {
  __builtin_nontemporal_store(v, (dz_global_u32x4*)(uintptr_t)p);
}
// The same accesses without the hint, for data that the Infinity Cache holds
// from one kernel to the next.
__device__ __forceinline__ dz_u32x4 ld_any(const void* p) { return *(const dz_global_u32x4*)(uintptr_t)p; }
__device__ __forceinline__ void st_any(void* p, dz_u32x4 v) { *(dz_global_u32x4*)(uintptr_t)p = v; }

// Wave-uniform copy of a 32-bit value in a scalar register.
// __builtin_amdgcn_readfirstlane returns a signed int: cast back to uint32_t
// before widening, or values >= 2^31 would sign-extend.
__device__ __forceinline__ uint32_t rfl_u32(uint32_t x) {
  return (uint32_t)__builtin_amdgcn_readfirstlane((int)x);
}
__device__ __forceinline__ uint64_t rfl_u64(uint64_t x) {
  return ((uint64_t)rfl_u32((uint32_t)(x >> 32)) << 32) | (uint64_t)rfl_u32((uint32_t)x);
}

// Workgroup barrier that orders LDS accesses only. __syncthreads() is a
// barrier between release and acquire fences on every address space, so
// before the barrier each wave waits for all of its vector-memory operations
// (s_waitcnt vmcnt(0)), its global stores included. The projection kernel's
// barriers only hand over LDS state (the chunk and descriptor rings, the
// reduction slots), and its chunks' stores need no ordering with the other
// waves (chunks are disjoint and nothing in the launch reads them back), so
// its barriers wait for the LDS counter alone. (Measured at OPT-13B: the
// reverse + norm pass, whose reduction barrier comes after the chunk's
// stores, 1.98 -> 1.91 ms; the other projection passes unchanged. The RMW
// kernel's tile loop measured no faster with the same change, since a tile's
// loads complete behind the previous tile's stores either way, so it keeps
// __syncthreads().)
__device__ __forceinline__ void lds_barrier() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
  __builtin_amdgcn_s_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
}

// Work tickets of the projection kernel's loop: lane 0 takes the next index
// from a work counter with a returning vector atomic add, issued as an
// instruction of its own so that the compiler's wait-counter bookkeeping does
// not track it, and ticket_wait<N> waits for it explicitly once N more
// vector-memory operations have been issued behind it (the chunk's loads and
// stores). Tracked by the compiler, the ticket's result, read where the full
// and partial chunk paths merge, is waited for with a wait for every
// operation in flight (the chunk's stores included). Hidden from the
// compiler, the ticket only ever makes the compiler's own waits wait for one
// operation more than they count, never less: vector-memory operations leave
// the wait counter in issue order.
//
// The register the atomic writes is not ready until that wait, which the
// compiler does not know: nothing between the two statements may read, copy
// or spill it. ticket_wait takes no operands (a wait that took the ticket as
// an operand, one per chunk path, made the compiler copy the register into
// the merged value's register ahead of the wait), and the value is used only
// through ticket_ready, after the waits. tests/test_kernel_asm.py checks the
// library's generated code for any instruction between the atomic and its
// wait that touches the register.
__device__ __forceinline__ uint32_t ticket_take(uint32_t* counter) {
  uint32_t t;
  asm volatile("global_atomic_add %0, %1, %2, off sc0" : "=&v"(t) : "v"(counter), "v"(1u) : "memory");
  return t;
}
// Waits until at most N vector-memory operations are in flight: the ticket,
// issued before at least N operations that follow it, has returned.
template <int N>
__device__ __forceinline__ void ticket_wait() {
  static_assert(N >= 0 && N < 64, "vmcnt range");
  asm volatile("s_waitcnt vmcnt(%0)" ::"n"(N) : "memory");
}
// The ticket as a value the compiler may use: an empty volatile statement
// that redefines it, placed after the waits. Volatile statements keep their
// order, so no use of the returned value is scheduled above a wait (a use of
// the atomic's own output could be: the waits have no operands).
__device__ __forceinline__ uint32_t ticket_ready(uint32_t t) {
  asm volatile("" : "+v"(t));
  return t;
}

// A chunk descriptor read from LDS is the same for every lane: move it to
// scalar registers so tile addresses are formed once per wave.
__device__ __forceinline__ DzChunk uniform_chunk(const DzChunk& c) {
  DzChunk u;
  u.ptr = rfl_u64(c.ptr);
  u.aux = 0;
  u.zgroup = rfl_u64(c.zgroup);
  u.n = rfl_u32(c.n);
  u.meta = rfl_u32(c.meta);
  return u;
}

// The same for a projection chunk, whose anchor address (aux) is used and
// whose element offset (zgroup) only DOT reads.
template <bool kOffset>
__device__ __forceinline__ DzChunk uniform_proj_chunk(const DzChunk& c) {
  DzChunk u;
  u.ptr = rfl_u64(c.ptr);
  u.aux = rfl_u64(c.aux);
  u.zgroup = kOffset ? rfl_u64(c.zgroup) : 0;
  u.n = rfl_u32(c.n);
  u.meta = rfl_u32(c.meta);
  return u;
}

// The group of a full tile whose Philox block the thread draws for its set u.
// 16-bit T: the group the thread holds. fp32: of a wave's 64 groups, lanes 2k
// and 2k + 1 hold the halves of groups k and 32 + k; the even lane draws the
// block of k, the odd one that of 32 + k.
template <int DT>
__device__ __forceinline__ uint32_t tile_group(int u) {
  const uint32_t t = threadIdx.x + (uint32_t)u * kRmwThreads;
  return DT != DZ_F32 ? t : (t & ~63u) + ((t & 1u) << 5) + ((t & 63u) >> 1);
}

// fp32: the z words of the thread's two vectors (x, y: the first; z, w: the
// second) from the block it drew and its neighbour's: even lanes hold the low
// halves of both groups, odd lanes the high ones.
__device__ __forceinline__ DzU4 exchange_halves(const DzU4& b) {
  const bool odd = (threadIdx.x & 1u) != 0u;
  // quad_perm [1, 0, 3, 2]
  const uint32_t r0 = (uint32_t)__builtin_amdgcn_mov_dpp((int)(odd ? b.x : b.z), 0xB1, 0xF, 0xF, true);
  const uint32_t r1 = (uint32_t)__builtin_amdgcn_mov_dpp((int)(odd ? b.y : b.w), 0xB1, 0xF, 0xF, true);
  return DzU4{odd ? r0 : b.x, odd ? r1 : b.y, odd ? b.z : r0, odd ? b.w : r1};
}

// The words of a thread's own elements from the block it drew.
template <int DT>
__device__ __forceinline__ DzU4 thread_words(const DzU4& b) {
  if constexpr (DT == DZ_F32) return exchange_halves(b);
  return b;
}

// Registers of one full tile: kVecs 16-byte vectors per thread.
template <int DT, int MODE>
struct TileRegs {
  static constexpr int kVecs = (DT == DZ_F32 ? 2 : 1) * RmwTraits<DT, MODE>::kGroups;
  dz_u32x4 v[kVecs];
};

template <int DT, int MODE>
__device__ __forceinline__ bool full_tile(const DzChunk& ch) {
  return ch.n == (uint32_t)RmwTraits<DT, MODE>::kChunk;
}

// Lane layout of a full tile: each load instruction of a wave covers contiguous
// memory. 16-bit T: a thread's groups of 8 elements (one vector each) are
// threadIdx.x + u * 1024 for u < G (tile-local group indices). fp32 groups are
// two vectors: a wave's 64 groups of set u are 128 consecutive vectors, of
// which lane l holds l and 64 + l, that is half l mod 2 of groups l / 2 and 32
// + l / 2 (tile_group and exchange_halves hand the Philox words on). With a
// group's two vectors in one thread, each instruction took every other 16
// bytes of its lines, and every fp32 pass ran 7-12 % slower: OPT-125m 121.5
// against 108.5 us, 2^29 elements 702 / 721 against 656 / 653 us (perturb /
// three-way). at(i) is the byte offset of the thread's vector i from the tile's
// start: set u = i (16-bit) or i / 2 (fp32). A tile holds at most 64 KB. The
// offsets are loop-invariant 64-bit values, so each access adds one to the
// tile's base (one v_lshl_add_u64).
//
// kPlain: plain loads and stores, else streaming (non-temporal) ones (see
// kPlainBytes for which launches take which).
template <int DT, int MODE, bool kPlain>
struct TileAccess {
  __device__ __forceinline__ size_t at(int i) const {
    if constexpr (DT != DZ_F32) return ((size_t)threadIdx.x + (size_t)i * kRmwThreads) * 16;
    return ((size_t)(threadIdx.x & ~63u) + (size_t)(i >> 1) * kRmwThreads) * 32 + (size_t)(i & 1) * 1024 +
           (size_t)(threadIdx.x & 63u) * 16;
  }
  __device__ __forceinline__ dz_u32x4 load(const void* p) const { return kPlain ? ld_any(p) : ld_stream(p); }
  __device__ __forceinline__ void store(void* p, dz_u32x4 v) const {
    if constexpr (kPlain)
      st_any(p, v);
    else
      st_stream(p, v);
  }
};

template <int DT, int MODE, class Access>
__device__ __forceinline__ void load_tile_at(uint64_t addr, const Access& to, TileRegs<DT, MODE>& r) {
#pragma unroll
  for (int i = 0; i < TileRegs<DT, MODE>::kVecs; ++i) r.v[i] = to.load((const char*)addr + to.at(i));
}

// Philox block of a thread's group of set u of a tile (tile_group): counter
// zgroup + that group. kUniformHi: the counters' high words agree across the tile (the
// low word does not wrap inside it), so the high word is wave-uniform and the
// counter's other uniform words keep round 0 and a product of rounds 1 and 2
// on the scalar unit.
template <int DT, bool kUniformHi>
__device__ __forceinline__ DzU4 tile_block(const DzChunk& ch, uint64_t seed, int u) {
  const uint32_t g = tile_group<DT>(u);
  if constexpr (kUniformHi) {
    return dz_philox_counter(seed, kDzStreamParam, (uint32_t)ch.zgroup + g, (uint32_t)(ch.zgroup >> 32));
  } else {
    return dz_philox_group(seed, kDzStreamParam, ch.zgroup + g);
  }
}

// Group u of a full fp32 tile with its z words w (and next-step words w2):
// the launch's operation applied and the group stored.
template <int DT, int MODE, class Access>
__device__ __forceinline__ void apply_store_group32(uint64_t base, const Access& to,
                                                    const TileRegs<DT, MODE>& r, int u,
                                                    const DzU4& wb, const DzU4& wb2,
                                                    const typename RmwTraits<DT, MODE>::E* tab, const DzScalars& sc) {
  const DzU4 w = exchange_halves(wb);
  const DzU4 w2 = MODE == kModeRestoreUpdatePerturb ? exchange_halves(wb2) : w;
  const dz_u32x4 a = r.v[2 * u], b = r.v[2 * u + 1];
  dz_u32x4 o0, o1;
  o0.x = apply_one<DT, MODE>(a.x, w.x & 0xffffu, w2.x & 0xffffu, tab, sc);
  o0.y = apply_one<DT, MODE>(a.y, w.x >> 16, w2.x >> 16, tab, sc);
  o0.z = apply_one<DT, MODE>(a.z, w.y & 0xffffu, w2.y & 0xffffu, tab, sc);
  o0.w = apply_one<DT, MODE>(a.w, w.y >> 16, w2.y >> 16, tab, sc);
  o1.x = apply_one<DT, MODE>(b.x, w.z & 0xffffu, w2.z & 0xffffu, tab, sc);
  o1.y = apply_one<DT, MODE>(b.y, w.z >> 16, w2.z >> 16, tab, sc);
  o1.z = apply_one<DT, MODE>(b.z, w.w & 0xffffu, w2.w & 0xffffu, tab, sc);
  o1.w = apply_one<DT, MODE>(b.w, w.w >> 16, w2.w >> 16, tab, sc);
  to.store((char*)base + to.at(2 * u), o0);
  to.store((char*)base + to.at(2 * u + 1), o1);
}

// A thread's share of a full tile as one straight-line block: the Philox
// blocks of all its groups, then the lookups, adds and stores. Keeping both
// in one basic block (the branch on the counters' high word is taken once
// per tile, outside it) lets the scheduler overlap the ALU work of the Philox
// chains with the LDS lookups; with the chains in a block of their own the
// two ran one after the other (three-way pass at OPT-13B: 8.9 -> 8.2 ms at
// equal Philox rounds).
// kLoadNext (the prefetching tile loop): the next tile's loads, from nptr
// into *nxt, go out once the first group is stored (for fp32's one group per
// thread at the tile's end: 2^28 elements 324 us, before the Philox chains 335,
// OPT-125m the same), held there by scheduling barriers.
// Measured at OPT-13B fp16, three-way pass, kernel microbench, same box,
// alternating builds: 7.86-7.90 ms with the loads issued before the Philox
// chains, 7.69-7.70 after them, 7.58-7.59 half-way, 7.59 a quarter in, 7.60
// three quarters in, and 7.89 with one vector loaded after each group's
// store; OPT-30B bf16 20.10-20.16 -> 19.83-19.89 ms half-way. In the ZO step
// (the bench's 20-step command, three alternating runs each), where the pass
// follows the GEMMs at a lower clock, after the first of four groups
// 7.63-7.66 ms, half-way 7.73-7.78, three quarters in 7.68-7.72; with three
// groups (bf16) after the first and after the second measured the same.
// Issued at the start, the next tile's reads meet this tile's first stores in
// the memory system (rocprofv3 counts 18 % fewer reads in flight and 2.7
// times the L2 tag stalls per cycle of the perturb pass).
template <int DT, int MODE, bool kUniformHi, bool kLoadNext = false, class Access>
__device__ __forceinline__ void tile_body(const DzChunk& ch, const Access& to,
                                          const TileRegs<DT, MODE>& r,
                                          const typename RmwTraits<DT, MODE>::E* tab, const DzScalars& sc,
                                          uint64_t nptr = 0, TileRegs<DT, MODE>* nxt = nullptr) {
  constexpr int G = RmwTraits<DT, MODE>::kGroups;
  constexpr bool kTwoSeeds = MODE == kModeRestoreUpdatePerturb;
  const uint64_t base = ch.ptr;
  DzU4 w[G], w2[G];
#pragma unroll
  for (int u = 0; u < G; ++u) {
    w[u] = tile_block<DT, kUniformHi>(ch, sc.seed, u);
    w2[u] = kTwoSeeds ? tile_block<DT, kUniformHi>(ch, sc.seed2, u) : w[u];
  }
#pragma unroll
  for (int u = 0; u < G; ++u) {
    if constexpr (DT == DZ_F32) {
      apply_store_group32<DT, MODE>(base, to, r, u, w[u], w2[u], tab, sc);
    } else {
      dz_u32x4 o;
      o.x = combine_pair16<DT, MODE>(r.v[u].x, w[u].x, w2[u].x, lookup_pair16<DT, MODE>(w[u].x, w2[u].x, tab));
      o.y = combine_pair16<DT, MODE>(r.v[u].y, w[u].y, w2[u].y, lookup_pair16<DT, MODE>(w[u].y, w2[u].y, tab));
      o.z = combine_pair16<DT, MODE>(r.v[u].z, w[u].z, w2[u].z, lookup_pair16<DT, MODE>(w[u].z, w2[u].z, tab));
      o.w = combine_pair16<DT, MODE>(r.v[u].w, w[u].w, w2[u].w, lookup_pair16<DT, MODE>(w[u].w, w2[u].w, tab));
      to.store((char*)base + to.at(u), o);
    }
    if constexpr (kLoadNext) {
      if (u == 0) {
        __builtin_amdgcn_sched_barrier(0);
        load_tile_at<DT, MODE>(nptr, to, *nxt);
        __builtin_amdgcn_sched_barrier(0);
      }
    }
  }
}

// Whether the Philox counters of a full tile's groups share their high word
// (the low word does not wrap inside the tile).
template <int DT, int MODE>
__device__ __forceinline__ bool tile_counters_share_high_word(const DzChunk& ch) {
  constexpr uint32_t kSpan = (uint32_t)(RmwTraits<DT, MODE>::kGroups * kRmwThreads);
  return (uint32_t)ch.zgroup <= 0xffffffffu - (kSpan - 1u);
}

// Whether the prefetching tile loop can take a tile: a full tile whose
// Philox counters share their high word.
template <int DT, int MODE>
__device__ __forceinline__ bool prefetchable_tile(const DzChunk& ch) {
  return full_tile<DT, MODE>(ch) && tile_counters_share_high_word<DT, MODE>(ch);
}

// Take bit of the RMW kernel's LDS descriptor ring: the top bit of a slot's
// Philox group (a group index is an element index / 8, so its top three bits
// are always clear), set when the slot holds a valid tile that
// prefetchable_tile accepts. bf16 launches that run the prefetching loop set
// it (ring_tagged); every reader of their ring clears it.
constexpr uint64_t kRingTake = 1ull << 63;

// Whether the prefetching loop's ring carries take bits: bf16 only, whose
// three-way pass is VALU-bound (1.4-1.9 % faster with them); the fp16 pass,
// which is not, measured 0.1 % slower.
__host__ __device__ constexpr bool ring_tagged(int dtype) { return dtype == DZ_BF16; }

// The next tile's descriptor as the prefetching loop's steps read it from the
// ring: the address and the Philox group with its take bit. n and meta are
// not read (0 here): the loop's body does not use them.
__device__ __forceinline__ DzChunk uniform_next_chunk(const DzChunk& c) {
  DzChunk u;
  u.ptr = rfl_u64(c.ptr);
  u.aux = 0;
  u.zgroup = rfl_u64(c.zgroup);
  u.n = 0;
  u.meta = 0;
  return u;
}

// Applies the launch's operation to a thread's share of a full tile, already
// in registers, and stores it.
template <int DT, int MODE, class Access>
__device__ __forceinline__ void compute_store_tile(const DzChunk& ch, const Access& to,
                                                   const TileRegs<DT, MODE>& r,
                                                   const typename RmwTraits<DT, MODE>::E* tab,
                                                   const DzScalars& sc) {
  if (tile_counters_share_high_word<DT, MODE>(ch)) {
    tile_body<DT, MODE, true>(ch, to, r, tab, sc);
  } else {
    tile_body<DT, MODE, false>(ch, to, r, tab, sc);
  }
}

// Partial tile (a tensor's last), bounds-checked: groups threadIdx.x,
// threadIdx.x + 1024, ... of the tile. A group with all 8 elements inside the
// tile goes through vector loads and stores like a full tile's; the tensor's
// last, incomplete group goes element by element. (A loop over the groups: with
// the loop unrolled and all loads issued first, the compiler scheduled the full
// tiles' code worse, 0.4-1 % in the long passes.)
template <int DT, int MODE, class Access>
__device__ __forceinline__ void rmw_partial(const DzChunk& ch, const Access& to, const typename RmwTraits<DT, MODE>::E* tab,
                                            const DzScalars& sc) {
  using S = typename DT_<DT>::S;
  constexpr bool kTwoSeeds = MODE == kModeRestoreUpdatePerturb;
  char* base = (char*)ch.ptr;
  for (uint32_t g = threadIdx.x; g * 8u < ch.n; g += kRmwThreads) {
    const DzU4 w = dz_philox_group(sc.seed, kDzStreamParam, ch.zgroup + g);
    const DzU4 w2 = kTwoSeeds ? dz_philox_group(sc.seed2, kDzStreamParam, ch.zgroup + g) : w;
    if ((g + 1u) * 8u <= ch.n) {
      if constexpr (DT == DZ_F32) {
        char* p = base + (size_t)g * 32;
        const dz_u32x4 a = to.load(p), b = to.load(p + 16);
        dz_u32x4 o0, o1;
        o0.x = apply_one<DT, MODE>(a.x, w.x & 0xffffu, w2.x & 0xffffu, tab, sc);
        o0.y = apply_one<DT, MODE>(a.y, w.x >> 16, w2.x >> 16, tab, sc);
        o0.z = apply_one<DT, MODE>(a.z, w.y & 0xffffu, w2.y & 0xffffu, tab, sc);
        o0.w = apply_one<DT, MODE>(a.w, w.y >> 16, w2.y >> 16, tab, sc);
        o1.x = apply_one<DT, MODE>(b.x, w.z & 0xffffu, w2.z & 0xffffu, tab, sc);
        o1.y = apply_one<DT, MODE>(b.y, w.z >> 16, w2.z >> 16, tab, sc);
        o1.z = apply_one<DT, MODE>(b.z, w.w & 0xffffu, w2.w & 0xffffu, tab, sc);
        o1.w = apply_one<DT, MODE>(b.w, w.w >> 16, w2.w >> 16, tab, sc);
        to.store(p, o0);
        to.store(p + 16, o1);
      } else {
        char* p = base + (size_t)g * 16;
        const dz_u32x4 v = to.load(p);
        dz_u32x4 o;
        o.x = combine_pair16<DT, MODE>(v.x, w.x, w2.x, lookup_pair16<DT, MODE>(w.x, w2.x, tab));
        o.y = combine_pair16<DT, MODE>(v.y, w.y, w2.y, lookup_pair16<DT, MODE>(w.y, w2.y, tab));
        o.z = combine_pair16<DT, MODE>(v.z, w.z, w2.z, lookup_pair16<DT, MODE>(w.z, w2.z, tab));
        o.w = combine_pair16<DT, MODE>(v.w, w.w, w2.w, lookup_pair16<DT, MODE>(w.w, w2.w, tab));
        to.store(p, o);
      }
      continue;
    }
    const uint32_t m = min(8u, ch.n - g * 8u);
    for (uint32_t j = 0; j < m; ++j) {
      const uint32_t h = (word_of(w, (int)(j >> 1)) >> (16 * (j & 1))) & 0xffffu;
      const uint32_t h2 = (word_of(w2, (int)(j >> 1)) >> (16 * (j & 1))) & 0xffffu;
      S* p = (S*)(base + (size_t)(g * 8u + j) * sizeof(S));
      *p = (S)apply_one<DT, MODE>((uint32_t)*p, h, h2, tab, sc);
    }
  }
}

// ---------------------------------------------------------------------------
// Multi-tensor read-modify-write kernel (perturb / update / restore+update).
// Persistent workgroups (one per CU) build the launch's delta table in LDS,
// then take tiles from the table's counters, handed out dynamically: that
// keeps the work in flight close together in memory and lets fast
// workgroups take more, which a static grid-stride split does not. The
// workgroup takes whole tiles from counters j of K = min(8, grid / 8),
// workgroup b using counter (b / 8) mod K, so every counter serves
// workgroups on every XCD; wave 0 keeps a ring in LDS (while tile k streams,
// the index of tile k+3 is taken and the descriptor of tile k+2 is loaded,
// with scalar loads) and a barrier ends each tile. The chunk list holds its
// full tiles first. The last workgroup to finish resets the
// counters for the next launch.
//
// Two tile loops: the plain loop (rmw_tiles) loads each tile when its turn
// comes; the prefetching loop (rmw_tiles_prefetch, the restore + update +
// next perturb passes; a table can set a minimum launch size,
// dz_table_set_prefetch_min_tiles) issues the next full tile's loads once
// each tile's first group is stored, and hands the workgroup's remaining
// tiles to rmw_tiles at its first tile that is not full.
// ---------------------------------------------------------------------------
template <int DT, int MODE, bool kTagged = false, class Access>
__device__ __forceinline__ void rmw_tiles(uint32_t k0, const DzChunk* __restrict__ chunks, uint32_t nchunks,
                                          const typename RmwTraits<DT, MODE>::E* tab, const DzScalars& sc,
                                          const Access& to, uint32_t* sidx, DzChunk* sdesc,
                                          uint32_t* mine, uint32_t ncnt, uint32_t j) {
  const uint64_t nch = nchunks;
  TileRegs<DT, MODE> cur;
  for (uint32_t k = k0;; ++k) {
    const uint32_t c = sidx[k % 4];
    if (c >= nchunks) break;
    DzChunk ch = uniform_chunk(sdesc[k % 3]);
    if constexpr (kTagged) ch.zgroup &= ~kRingTake;
    // Wave 0 fetches a descriptor with scalar loads (it is uniform, so it
    // costs no vector registers); lane 0 takes an index with a vector
    // atomic. The anchor field is unused by ZO tables.
    uint32_t grabbed = 0;
    uint64_t n_ptr = 0, n_zg = 0;
    uint32_t n_n = 0, n_meta = 0;
    bool have_desc = false;
    if ((rfl_u32(threadIdx.x) >> 6) == 0) {  // wave 0 (uniform branch)
      if (threadIdx.x == 0) grabbed = atomicAdd(mine, 1u);
      const uint32_t cd = rfl_u32(sidx[(k + 2) % 4]);
      if (cd < nchunks) {
        const DzChunk* src = chunks + cd;
        n_ptr = src->ptr;
        n_zg = src->zgroup;
        n_n = src->n;
        n_meta = src->meta;
        have_desc = true;
      }
    }
    if (full_tile<DT, MODE>(ch)) {
      load_tile_at<DT, MODE>(ch.ptr, to, cur);
      compute_store_tile<DT, MODE>(ch, to, cur, tab, sc);
    } else {
      rmw_partial<DT, MODE>(ch, to, tab, sc);
    }
    if (threadIdx.x == 0) {
      sidx[(k + 3) % 4] = (uint32_t)min((uint64_t)grabbed * ncnt + j, nch);
      if (have_desc) {
        DzChunk& d = sdesc[(k + 2) % 3];
        d.ptr = n_ptr;
        d.aux = 0;
        d.zgroup = n_zg;
        d.n = n_n;
        d.meta = n_meta;
      }
    }
    __syncthreads();
  }
}

// A wait for every vector-memory operation in flight that the compiler sees
// (s_waitcnt with vmcnt 0 and the other counters at their maximum, gfx9
// encoding), so its own bookkeeping knows that nothing is pending after it.
__device__ __forceinline__ void wait_vm_all() { __builtin_amdgcn_s_waitcnt(0x0F70); }

// One tile of the prefetching tile loop (see rmw_tiles_prefetch): full tile
// k, whose descriptor `ch` the step before read, is computed from `cur`
// (loaded during tile k - 1) while tile k + 1 is loaded into `nxt` (the loads
// go out after the first group, in tile_body). Tile k + 1's descriptor is
// read into `ch1`. Returns whether tile k + 1 is a full tile (its data is
// then in `nxt`); if it is not, the loads read a stand-in of the same size
// (the quantile table), so that every path issues the same loads.
// Descriptor slot (k + 1) % 3 is next written in step k + 2, so the copy read
// here is the one step k + 1 would read; carrying it saves each wave a
// descriptor's LDS reads and its moves to scalar registers per tile. For
// bf16 (ring_tagged), wave 0, which writes the slot, also stores there
// whether the loop can take the tile (kRingTake), so the other waves read
// only the address and the Philox group (one ds_read2_b64, four lane moves;
// no index, n or meta). With these, the bookkeeping below 64 KB of LDS
// (RmwShared) and the wave test taken once (wave0), a thread's VALU
// instructions per tile of the three-way pass went from 459 to 447 for bf16
// (three groups; 2 more on every other step of the unrolled loop) and from
// 430 to 422 for fp16 (four groups). Loading the next tile with buffer loads
// (a descriptor on the scalar unit, 32-bit offsets: no 64-bit address add per
// vector) took 3-4 more off and measured no faster; it is left out. So is
// reading tile k + 1's descriptor from the table with scalar loads in every
// wave (wave 0 has read the entry a step earlier, so they hit the scalar
// cache): 7 fewer per bf16 tile than without take bits (149 per group
// counted), but each tile's start then waits for the scalar loads, and the
// bf16 pass measured 1.4 % faster on one box and 2-3 % slower on two others,
// also with the next index carried from the step before so that those loads
// go out with no LDS read ahead of them.
template <int DT, int MODE, class Access>
__device__ __forceinline__ bool rmw_prefetch_step(uint32_t k, const DzChunk& ch, DzChunk& ch1,
                                                  const DzChunk* __restrict__ chunks, uint32_t nchunks,
                                                  const typename RmwTraits<DT, MODE>::E* tab, const DzScalars& sc,
                                                  const Access& to, uint32_t* sidx, DzChunk* sdesc,
                                                  uint32_t* mine, uint32_t ncnt, uint32_t j, const void* dummy,
                                                  bool wave0, const TileRegs<DT, MODE>& cur,
                                                  TileRegs<DT, MODE>& nxt) {
  bool nxt_full;
  if constexpr (ring_tagged(DT)) {
    // The slot's offset is opaque to the compiler, so both fields are read
    // through one address register (one ds_read2_b64), and the take bit is
    // tested on the high word (no 64-bit scalar compare).
    uint32_t slot = (k + 1) % 3 * (uint32_t)sizeof(DzChunk);
    asm("" : "+s"(slot));
    ch1 = uniform_next_chunk(*(const DzChunk*)((const char*)sdesc + slot));
    uint32_t zhi = (uint32_t)(ch1.zgroup >> 32);
    asm("" : "+s"(zhi));  // keeps the test on 32 bits (no 64-bit compare folded back)
    nxt_full = (int32_t)zhi < 0;
    ch1.zgroup = (uint64_t)(zhi & 0x7fffffffu) << 32 | (uint32_t)ch1.zgroup;
  } else {
    const uint32_t c1 = rfl_u32(sidx[(k + 1) % 4]);
    ch1 = uniform_chunk(sdesc[(k + 1) % 3]);
    nxt_full = c1 < nchunks && prefetchable_tile<DT, MODE>(ch1);
  }
  const uint64_t nptr = nxt_full ? ch1.ptr : (uint64_t)(uintptr_t)dummy;
  // wave 0: the ticket of tile k + 3 and the descriptor of tile k + 2
  uint32_t grabbed = 0;
  uint64_t n_ptr = 0, n_zg = 0;
  uint32_t n_n = 0, n_meta = 0;
  bool have_desc = false;
  if (wave0) {  // uniform branch
    if (threadIdx.x == 0) grabbed = atomicAdd(mine, 1u);
    const uint32_t cd = rfl_u32(sidx[(k + 2) % 4]);
    if (cd < nchunks) {
      const DzChunk* src = chunks + cd;
      n_ptr = src->ptr;
      n_zg = src->zgroup;
      n_n = src->n;
      n_meta = src->meta;
      have_desc = true;
      if constexpr (ring_tagged(DT))
        if (prefetchable_tile<DT, MODE>(DzChunk{n_ptr, 0, n_zg, n_n, n_meta})) n_zg |= kRingTake;
    }
  }
  tile_body<DT, MODE, true, true>(ch, to, cur, tab, sc, nptr, &nxt);
  // The ticket is first read here, one straight block after the atomic, so
  // the compiler's wait for it counts the tile's stores and the next tile's
  // loads issued behind it (vmcnt(2 * kVecs)) instead of draining them.
  if (threadIdx.x == 0) {
    sidx[(k + 3) % 4] = (uint32_t)min((uint64_t)grabbed * ncnt + j, (uint64_t)nchunks);
    DzChunk& d = sdesc[(k + 2) % 3];
    if (have_desc) {
      d.ptr = n_ptr;
      d.aux = 0;
      if constexpr (!ring_tagged(DT)) d.zgroup = n_zg;
      d.n = n_n;
      d.meta = n_meta;
    }
    // with the take bit step k + 1 reads; 0 (no take bit) past the table's end
    if constexpr (ring_tagged(DT)) d.zgroup = n_zg;
  }
  lds_barrier();
  return nxt_full;
}

// Tile loop with the next tile's loads in flight during each tile's work,
// over the run of full tiles a workgroup takes first (a table lists its full
// tiles first); the rest of its tiles go through rmw_tiles. Two register
// sets are used in turn (the loop unrolled by two, so no pending registers
// are copied); each step is one straight block whose loads go out at a fixed
// point of it; the ticket is first read in the same straight block as its
// atomic; and the barrier orders LDS only. With those, the compiler's waits for a tile's
// data count the operations behind it (the previous tile's stores and the
// next tile's loads) instead of draining everything in flight.
template <int DT, int MODE, class Access>
__device__ __forceinline__ uint32_t rmw_tiles_prefetch(const DzChunk* __restrict__ chunks, uint32_t nchunks,
                                                       const typename RmwTraits<DT, MODE>::E* tab,
                                                       const DzScalars& sc, const Access& to,
                                                       uint32_t* sidx, DzChunk* sdesc, uint32_t* mine, uint32_t ncnt,
                                                       uint32_t j, const void* dummy) {
  const uint32_t c0 = rfl_u32(sidx[0]);
  DzChunk ch0 = uniform_chunk(sdesc[0]);
  if constexpr (ring_tagged(DT)) ch0.zgroup &= ~kRingTake;
  if (!(c0 < nchunks && prefetchable_tile<DT, MODE>(ch0))) return 0;
  // the stand-in must hold a whole tile (a thread's last vector ends at the
  // tile's size)
  static_assert(RmwTraits<DT, MODE>::kChunk <= kDzTabEntries, "the quantile table is a tile's stand-in");
  TileRegs<DT, MODE> a, b;
  DzChunk da = ch0, db;
  const bool wave0 = (rfl_u32(threadIdx.x) >> 6) == 0;
  load_tile_at<DT, MODE>(ch0.ptr, to, a);
  uint32_t k = 0;
  for (;;) {
    if (!rmw_prefetch_step<DT, MODE>(k, da, db, chunks, nchunks, tab, sc, to, sidx, sdesc, mine, ncnt, j, dummy,
                                     wave0, a, b)) {
      k += 1;
      break;
    }
    if (!rmw_prefetch_step<DT, MODE>(k + 1, db, da, chunks, nchunks, tab, sc, to, sidx, sdesc, mine, ncnt, j, dummy,
                                     wave0, b, a)) {
      k += 2;
      break;
    }
    k += 2;
  }
  wait_vm_all();  // the stand-in loads of the last step
  return k;
}

// The RMW kernel's LDS: the tile bookkeeping rings first, so that their
// addresses stay below 64 KB and each wave's reads of them take one address
// register and the DS instructions' 16-bit offset field (with the 128 KB
// table first they took a register per read), then the launch's table.
template <typename E>
struct RmwShared {
  DzChunk sdesc[3];      // descriptors of tiles k .. k + 2
  uint32_t sidx[4];      // indices of tiles k .. k + 3
  E tab[kDzTabEntries];  // the delta table
};

// kPF: run the prefetching tile loop over the workgroup's leading full tiles
// (only where RmwTraits::kPrefetch allows it; the launcher picks it by size).
template <int DT, int MODE, bool kPF, bool kPlain>
__global__ void __launch_bounds__(kRmwThreads, kRmwWavesPerEU) rmw_kernel(const DzChunk* __restrict__ chunks,
                                                                          uint32_t nchunks,
                                                                          const void* __restrict__ qtab,
                                                                          DzScalars sc_in, DzScalarPtrs sp,
                                                                          uint32_t* __restrict__ counters) {
  using Tr = RmwTraits<DT, MODE>;
  using E = typename Tr::E;
  __shared__ __attribute__((aligned(16))) RmwShared<E> sh;
  E* const tab = sh.tab;
  uint32_t* const sidx = sh.sidx;
  DzChunk* const sdesc = sh.sdesc;
  const DzScalars sc = resolve_scalars<DT>(sc_in, sp);
  // Counters in use: every one of them must be served by at least one
  // workgroup, or its tiles would never be taken (a small grid uses fewer).
  const uint32_t ncnt = rfl_u32(max(1u, min((uint32_t)kCounters, gridDim.x >> 3)));
  const uint32_t j = rfl_u32((blockIdx.x >> 3) % ncnt);
  uint32_t* mine = counters + j * kCounterStride;
  const uint64_t nch = nchunks;
  // Start-up: lane 0 takes the first three tickets with one atomic, the
  // table's loads are issued behind it, then the first two descriptors are
  // loaded (clamped to a valid index; only tickets below nchunks are used)
  // and the table is written.
  uint32_t t0 = 0;
  if (threadIdx.x == 0) t0 = atomicAdd(mine, 3u);
  TableSlices<DT> qs;
  load_table<DT>(qs, qtab);
  if (threadIdx.x == 0) {
    uint64_t c[3];
    for (int i = 0; i < 3; ++i) {
      c[i] = (uint64_t)(t0 + i) * ncnt + j;
      sidx[i] = (uint32_t)min(c[i], nch);
    }
    if (nch > 0) {
      const DzChunk d0 = chunks[min(c[0], nch - 1)];
      const DzChunk d1 = chunks[min(c[1], nch - 1)];
      sdesc[0] = d0;
      sdesc[1] = d1;
      if constexpr (Tr::kPrefetch && kPF && ring_tagged(DT)) {  // the take bits (kRingTake)
        if (c[0] < nch && prefetchable_tile<DT, MODE>(d0)) sdesc[0].zgroup |= kRingTake;
        if (c[1] < nch && prefetchable_tile<DT, MODE>(d1)) sdesc[1].zgroup |= kRingTake;
      }
    }
  }
  store_table<DT, MODE>(tab, qs, sc);
  const TileAccess<DT, MODE, kPlain> to{};
  __syncthreads();
  uint32_t k0 = 0;
  if constexpr (Tr::kPrefetch && kPF)
    k0 = rmw_tiles_prefetch<DT, MODE>(chunks, nchunks, tab, sc, to, sidx, sdesc, mine, ncnt, j, qtab);
  constexpr bool kTagged = Tr::kPrefetch && kPF && ring_tagged(DT);  // the ring may hold take bits
  rmw_tiles<DT, MODE, kTagged>(k0, chunks, nchunks, tab, sc, to, sidx, sdesc, mine, ncnt, j);
  if (threadIdx.x == 0) {
    const uint32_t done = atomicAdd(counters + kDoneSlot * kCounterStride, 1u);
    if (done == gridDim.x - 1) {
      for (int i = 0; i <= kDoneSlot; ++i) atomicExch(counters + i * kCounterStride, 0u);
    }
  }
}

// ---------------------------------------------------------------------------
// Read-modify-write launches of short tables. The persistent kernel above pays
// for its work counters, its descriptor ring and its delta table (3 to 10 us),
// which a pass over a few million elements does not earn back. Here workgroups
// of 1024 threads take tiles of 8 elements per thread in a fixed order (tile
// blockIdx.x, then every gridDim.x-th), the quantile table is copied to LDS as
// it is, and the deltas are evaluated for each pair of elements with the same
// operations that the delta tables' entries take. The accesses are plain ones:
// what a short pass writes stays in the 256 MB Infinity Cache for the forward
// and the next pass (with the non-temporal hint, fp32, 2^24 elements: 30.5
// against 22.6 us). Pass times in us (perturb / three-way), this kernel and the
// persistent one with its hints: fp16 2^14 elements 4.0 / 4.1 and 6.8 / 9.0,
// 2^20 4.2 / 4.3 and 10.2 / 14.3, 2^22 6.0 / 7.5 and 13.1 / 19.5, 2^24 12.8 /
// 19.0, 2^25 21.1 / 30.7 and 27.2 / 30.3 (the three-way pass runs the persistent
// kernel there: short_elems); fp32 2^20 4.6 / 5.4 and 9.9 / 10.4, 2^24 21.8 / 22.9
// and 27.6 / 28.2. A launch is bound by its latencies (about 4 us) up to 2^20
// elements, then by the VALU: with one Philox round for seven, fp16 2^25 elements
// take 21.4 / 22.4 us; with lookups free of bank conflicts, the same time.
// ---------------------------------------------------------------------------

// The launch's operation on two packed 16-bit elements with their signed z
// (and next step's z).
template <int DT, int MODE>
__device__ __forceinline__ uint32_t apply_z_pair(uint32_t th, uint32_t z, uint32_t z2, const DzScalars& sc) {
  if constexpr (MODE == kModeUpdate) return add_pair<DT>(th, delta_nd_pair<DT>(z, sc));
  uint32_t r = add_pair<DT>(th, delta_b_pair<DT, MODE != kModePerturb>(z, sc));
  if constexpr (rmw_pair_mode(MODE)) r = add_pair<DT>(r, delta_nd_pair<DT>(z, sc));
  if constexpr (MODE == kModeRestoreUpdatePerturb) r = add_pair<DT>(r, delta_b_pair<DT, true>(z2, sc));
  return r;
}
// The launch's operation on one fp32 element with its signed z.
template <int MODE>
__device__ __forceinline__ uint32_t apply_z_f32(uint32_t th, uint32_t z, uint32_t z2, const DzScalars& sc) {
  const float zf = __uint_as_float(z);
  if constexpr (MODE == kModePerturb) return op_perturb<DZ_F32>(__uint_as_float(th), zf, sc.scale, sc.eps);
  if constexpr (MODE == kModePerturbUnit) return op_perturb<DZ_F32>(__uint_as_float(th), zf, 1.0f, sc.eps);
  if constexpr (MODE == kModeUpdate) return op_update<DZ_F32>(__uint_as_float(th), zf, sc.grad, sc.lr);
  uint32_t r = op_perturb<DZ_F32>(__uint_as_float(th), zf, 1.0f, sc.eps);
  r = op_update<DZ_F32>(__uint_as_float(r), zf, sc.grad, sc.lr);
  if constexpr (MODE == kModeRestoreUpdatePerturb)
    r = op_perturb<DZ_F32>(__uint_as_float(r), __uint_as_float(z2), 1.0f, sc.eps);
  return r;
}

// The eight z of a Philox block in T, from a quantile table `tab` of T (in LDS
// or in memory): 16-bit T packed into one vector, fp32 into two.
template <int DT>
struct ZVec {
  static constexpr int kVecs = DT == DZ_F32 ? 2 : 1;
  dz_u32x4 v[kVecs];
};
template <int DT>
__device__ __forceinline__ ZVec<DT> z_vec(const typename DT_<DT>::S* tab, const DzU4& w) {
  ZVec<DT> r;
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const uint32_t x = word_of(w, i);
    uint32_t e0, e1;
    lookup2(tab, x, e0, e1);
    if constexpr (DT == DZ_F32) {
      r.v[i >> 1][2 * (i & 1)] = e0 | ((x & 0x8000u) << 16);
      r.v[i >> 1][2 * (i & 1) + 1] = e1 | (x & 0x80000000u);
    } else {
      r.v[0][i] = (e0 | (e1 << 16)) | (x & 0x80008000u);
    }
  }
  return r;
}

// A thread's 8 elements of a short table's tile: one vector of 16-bit T, or two
// of fp32 laid out as in TileAccess.
template <int DT>
struct ShortGroup {
  using S = typename DT_<DT>::S;
  static constexpr int kVecs = ZVec<DT>::kVecs;
  static constexpr uint32_t kPer = 16 / (uint32_t)sizeof(S);
  char* base;       // the tile
  uint32_t n;       // its elements
  dz_u32x4 v[kVecs];

  // First element of the thread's vector k.
  static __device__ __forceinline__ uint32_t first(int k) {
    return DT != DZ_F32 ? threadIdx.x * 8u : (threadIdx.x & ~63u) * 8u + (uint32_t)k * 256u + (threadIdx.x & 63u) * 4u;
  }
  __device__ __forceinline__ uint32_t get(int k, int j) const {
    return DT == DZ_F32 ? v[k][j & 3] : v[k][j >> 1] >> (16 * (j & 1));
  }
  __device__ __forceinline__ ShortGroup() {}
  __device__ __forceinline__ explicit ShortGroup(const DzChunk& ch) {
    base = (char*)ch.ptr;
    n = ch.n;
#pragma unroll
    for (int k = 0; k < kVecs; ++k) {
      const uint32_t e = first(k);
      const S* p = (const S*)base + e;
      if (e + kPer <= n) {
        v[k] = ld_any(p);
      } else if (e < n) {  // the tensor's last elements
#pragma unroll
        for (int j = 0; j < (int)kPer; ++j) {
          const uint32_t x = e + (uint32_t)j < n ? (uint32_t)p[j] : 0u;
          if constexpr (DT == DZ_F32)
            v[k][j & 3] = x;
          else
            v[k][j >> 1] = j & 1 ? v[k][j >> 1] | (x << 16) : x;
        }
      }
    }
  }
  __device__ __forceinline__ void store() const {
#pragma unroll
    for (int k = 0; k < kVecs; ++k) {
      const uint32_t e = first(k);
      S* p = (S*)base + e;
      if (e + kPer <= n) {
        st_any(p, v[k]);
      } else if (e < n) {
#pragma unroll
        for (int j = 0; j < (int)kPer; ++j)
          if (e + (uint32_t)j < n) p[j] = (S)get(k, j);
      }
    }
  }
  // Whether any lane of the wave holds elements of the tile (the lanes of an
  // fp32 pair exchange words, so a wave runs whole or not at all).
  __device__ __forceinline__ bool wave_active() const { return (threadIdx.x & ~63u) * 8u < n; }
};

template <int DT, int MODE>
__global__ void __launch_bounds__(kRmwThreads, DT == DZ_F32 ? 4 : 8)
    rmw_short_kernel(const DzChunk* __restrict__ chunks, uint32_t nchunks, const void* __restrict__ qtab,
                     DzScalars sc_in, DzScalarPtrs sp) {
  using S = typename DT_<DT>::S;
  constexpr bool kNext = MODE == kModeRestoreUpdatePerturb;
  constexpr int kSlices = kDzTabEntries * (int)sizeof(S) / (16 * kRmwThreads);
  __shared__ __attribute__((aligned(16))) S tab[kDzTabEntries];
  uint32_t t = blockIdx.x;
  DzChunk ch = chunks[t];
  ShortGroup<DT> cur(ch);  // in flight while the table is copied
  {
    dz_u32x4 q[kSlices];
#pragma unroll
    for (int k = 0; k < kSlices; ++k)
      q[k] = *(const dz_u32x4*)((const char*)qtab + (size_t)(k * kRmwThreads + threadIdx.x) * 16);
#pragma unroll
    for (int k = 0; k < kSlices; ++k) *(dz_u32x4*)((char*)tab + (size_t)(k * kRmwThreads + threadIdx.x) * 16) = q[k];
  }
  const DzScalars sc = resolve_scalars<DT>(sc_in, sp);
  __syncthreads();
  for (;;) {
    // the tile's counters share their high word (build_chunks), which stays on
    // the scalar unit
    const uint32_t q = (uint32_t)ch.zgroup + tile_group<DT>(0), q_hi = (uint32_t)(ch.zgroup >> 32);
    const uint32_t tn = t + gridDim.x;
    const bool more = tn < nchunks;
    ShortGroup<DT> nxt;
    if (more) {
      ch = chunks[tn];
      nxt = ShortGroup<DT>(ch);
    }
    if (cur.wave_active()) {
      const ZVec<DT> z = z_vec<DT>(tab, thread_words<DT>(dz_philox_counter(sc.seed, kDzStreamParam, q, q_hi)));
      const ZVec<DT> z2 =
          kNext ? z_vec<DT>(tab, thread_words<DT>(dz_philox_counter(sc.seed2, kDzStreamParam, q, q_hi))) : z;
#pragma unroll
      for (int k = 0; k < ZVec<DT>::kVecs; ++k) {
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          if constexpr (DT == DZ_F32)
            cur.v[k][i] = apply_z_f32<MODE>(cur.v[k][i], z.v[k][i], z2.v[k][i], sc);
          else
            cur.v[k][i] = apply_z_pair<DT, MODE>(cur.v[k][i], z.v[k][i], z2.v[k][i], sc);
        }
      }
      cur.store();
    }
    if (!more) break;
    t = tn;
    cur = nxt;
  }
}

// ---------------------------------------------------------------------------
// Projection kernels over the projected (k/v) tensors, one group per tensor.
//   SUMSQ          partial[c] = sum over chunk of fp32(R_T(theta - theta0))^2
//   APPLY          theta <- R_T(R_T(R_T(theta - theta0) * alpha) + theta0)   trainer.py:428-436
//   REVERSE        theta <- R_T(R_T(R_T(theta - theta0) / alpha) + theta0)   trainer.py:447-451
//   REVERSE_SUMSQ  REVERSE, then partial[c] of the new theta (next norm, trainer.py:455-457)
//   APPLY_F32      theta <- R_T(fp32(R_T(theta - theta0)) * alpha + theta0) with an fp32 alpha:
//                  the first-order path's apply (trainer.py:428-436 with gamma an fp32
//                  Parameter, so v and temp stay fp32 and copy_ rounds once)
//   DOT            partial[c] = sum over chunk of fp32(other) * fp32(R_T(theta - theta0)), other a third
//                  tensor per group: the gradient of the first-order objective with respect to
//                  alpha (trainer.py:428-429 under autograd). One workgroup per chunk with an
//                  element per load took 615 us over 64 x 6,553,600 fp16 elements, these loops
//                  take 383 (6.6 TB/s)
// Each chunk is processed by one workgroup; squares and sums in fp64 (exact
// squares of the fp32-widened differences) in a fixed reduction order, so the
// per-chunk partials, and the group sums built from them, are deterministic.
// ---------------------------------------------------------------------------
template <int DT>
__device__ __forceinline__ void proj_elem(int mode, uint32_t thb, uint32_t t0b, float alpha,
                                          uint32_t* outb, double* acc) {
  const float th = DT_<DT>::to_f(thb);
  const float t0 = DT_<DT>::to_f(t0b);
  const float d = rt<DT>(th - t0);
  if (mode == kProjSumsq) {
    const double dd = (double)d;
    *acc += dd * dd;
    *outb = thb;
    return;
  }
  float v;
  if (mode == kProjApply) {
    v = rt<DT>(d * alpha);
  } else if (mode == kProjApplyF32) {
    v = d * alpha;
  } else {
    v = rt<DT>(d / alpha);
  }
  const uint32_t nb = DT_<DT>::from_f(v + t0);
  *outb = nb;
  if (mode == kProjReverseSumsq) {
    const double d2 = (double)rt<DT>(DT_<DT>::to_f(nb) - t0);
    *acc += d2 * d2;
  }
}

// R_T(a - b) and R_T(a * b) for two packed 16-bit lanes of T (both operands
// in T: the exact difference or product rounded once, which is the
// reference's fp32 op rounded to T).
template <int DT>
__device__ __forceinline__ uint32_t sub_pair(uint32_t a, uint32_t b) {
  if constexpr (DT == DZ_F16) {
    return __builtin_bit_cast(uint32_t, __builtin_bit_cast(dz_half2, a) - __builtin_bit_cast(dz_half2, b));
  } else {
    return __builtin_bit_cast(uint32_t, __builtin_bit_cast(dz_bf2, a) - __builtin_bit_cast(dz_bf2, b));
  }
}
template <int DT>
__device__ __forceinline__ uint32_t mul_pair(uint32_t a, uint32_t b) {
  if constexpr (DT == DZ_F16) {
    return __builtin_bit_cast(uint32_t, __builtin_bit_cast(dz_half2, a) * __builtin_bit_cast(dz_half2, b));
  } else {
    return __builtin_bit_cast(uint32_t, __builtin_bit_cast(dz_bf2, a) * __builtin_bit_cast(dz_bf2, b));
  }
}

// Sum of squares of the two lanes of a packed 16-bit word, low lane first.
template <int DT>
__device__ __forceinline__ void acc_sq_pair(uint32_t d, double* acc) {
  const double d0 = (double)DT_<DT>::to_f(d & 0xffffu);
  const double d1 = (double)DT_<DT>::to_f(d >> 16);
  *acc += d0 * d0;
  *acc += d1 * d1;
}

// REVERSE's quotient R_T(fp32(d) / alpha) for bf16 T. The reference's fp32
// division rounded to bf16 equals bf16(d * inv), inv = fp32(1 / alpha), for
// every pair of bf16 values d, alpha with inv finite, unless the product is
// nonzero and below the smallest normal fp32 value: checked over all 2^32
// pairs (RN_bf16 of the fp32 quotient is RN_bf16 of the exact quotient, since
// fp32 carries 24 >= 2 * 8 + 2 bits, and for normal operands a bf16 quotient
// is at least 2^-16 of itself away from a bf16 rounding midpoint, where the
// product's error is under 2^-23). Vectors with an element outside that range
// divide. One multiply replaces the IEEE division sequence per element.
struct RecipDiv {
  float inv;  // fp32(1 / alpha)
  bool ok;    // inv is finite (alpha is neither 0, infinite nor below 2^-128)
};
__device__ __forceinline__ RecipDiv recip_div(float alpha) {
  const float inv = 1.0f / alpha;
  return RecipDiv{inv, __builtin_isfinite(inv) != 0};
}
__device__ __forceinline__ bool recip_quotient_subnormal(float q) {
  return __builtin_amdgcn_classf(q, 0x10 | 0x80);  // +- subnormal
}

// proj_elem for the two 16-bit elements of a word, in packed arithmetic where
// the reference's op has both operands in T (SUMSQ, APPLY and the subtract /
// add of REVERSE); alpha2 holds alpha in both lanes. APPLY_F32 is not here
// (its fp32 alpha keeps v and the sum in fp32).
template <int DT, int MODE>
__device__ __forceinline__ uint32_t proj_word16(uint32_t th, uint32_t t0, uint32_t alpha2, float alpha,
                                                double* acc) {
  const uint32_t d = sub_pair<DT>(th, t0);
  if constexpr (MODE == kProjSumsq) {
    acc_sq_pair<DT>(d, acc);
    return th;
  } else {
    uint32_t v;
    if constexpr (MODE == kProjApply) {
      v = mul_pair<DT>(d, alpha2);
    } else {
      const float v0 = DT_<DT>::to_f(d & 0xffffu) / alpha;
      const float v1 = DT_<DT>::to_f(d >> 16) / alpha;
      v = DT_<DT>::from_f(v0) | (DT_<DT>::from_f(v1) << 16);
    }
    const uint32_t nb = add_pair<DT>(v, t0);
    if constexpr (MODE == kProjReverseSumsq) acc_sq_pair<DT>(sub_pair<DT>(nb, t0), acc);
    return nb;
  }
}

__device__ __forceinline__ double block_sum_f64(double x, double* red) {
#pragma unroll
  for (int off = 32; off >= 1; off >>= 1) x += __shfl_xor(x, off, 64);
  const int wid = threadIdx.x >> 6;
  if ((threadIdx.x & 63) == 0) red[wid] = x;
  lds_barrier();
  double t = 0.0;
  if (threadIdx.x == 0) {
    for (int i = 0; i < (int)(blockDim.x >> 6); ++i) t += red[i];
  }
  return t;
}

// A chunk the vector path takes whole.
template <int DT>
__device__ __forceinline__ bool proj_full_chunk(const DzChunk& ch) {
  return ch.n == (uint32_t)proj_chunk_elems(DT);
}

// The operation on one 16-byte vector of theta with its anchor's. What depends
// on the group's alpha is made once per chunk (ProjScalars).
template <int DT, int MODE>
struct ProjScalars {
  float alpha;
  uint32_t alpha2;  // alpha in both 16-bit lanes (the ZO modes' alpha is a value of T)
  RecipDiv rd;
  __device__ __forceinline__ explicit ProjScalars(float a)
      : alpha(a),
        alpha2((DT != DZ_F32 && MODE != kProjApplyF32) ? DT_<DT>::from_f(a) * 0x10001u : 0u),
        rd((DT == DZ_BF16 && (MODE == kProjReverse || MODE == kProjReverseSumsq)) ? recip_div(a)
                                                                                : RecipDiv{0.0f, false}) {}
};
template <int DT, int MODE>
__device__ __forceinline__ dz_u32x4 proj_vec(dz_u32x4 vt, dz_u32x4 va, const ProjScalars<DT, MODE>& ps, double* acc) {
  dz_u32x4 o;
  if constexpr (DT == DZ_BF16 && (MODE == kProjReverse || MODE == kProjReverseSumsq)) {
    // the quotients of the whole vector by the reciprocal, or by division if one
    // of them asks for it: one branch for eight elements (with one for two, the
    // reverse + norm pass over 64 x 26,214,400 elements took 1684 us, 1622 now)
    float q[8];
    bool divide = !ps.rd.ok;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const uint32_t d = sub_pair<DT>(vt[i], va[i]);
      q[2 * i] = bf16_lo_f(d);
      q[2 * i + 1] = bf16_hi_f(d);
      divide |= recip_quotient_subnormal(q[2 * i] * ps.rd.inv);
      divide |= recip_quotient_subnormal(q[2 * i + 1] * ps.rd.inv);
    }
    if (divide) {
#pragma unroll
      for (int j = 0; j < 8; ++j) q[j] /= ps.alpha;
    } else {
#pragma unroll
      for (int j = 0; j < 8; ++j) q[j] *= ps.rd.inv;
    }
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      o[i] = add_pair<DT>(pack_bf16(q[2 * i], q[2 * i + 1]), va[i]);
      if constexpr (MODE == kProjReverseSumsq) acc_sq_pair<DT>(sub_pair<DT>(o[i], va[i]), acc);
    }
  } else {
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      if constexpr (DT != DZ_F32 && MODE != kProjApplyF32) {
        o[i] = proj_word16<DT, MODE>(vt[i], va[i], ps.alpha2, ps.alpha, acc);
      } else if constexpr (DT != DZ_F32) {
        uint32_t r0, r1;
        proj_elem<DT>(MODE, vt[i] & 0xffffu, va[i] & 0xffffu, ps.alpha, &r0, acc);
        proj_elem<DT>(MODE, vt[i] >> 16, va[i] >> 16, ps.alpha, &r1, acc);
        o[i] = (r0 & 0xffffu) | (r1 << 16);
      } else {
        uint32_t r;
        proj_elem<DT>(MODE, vt[i], va[i], ps.alpha, &r, acc);
        o[i] = r;
      }
    }
  }
  return o;
}
// DOT: sum of fp32(other) * fp32(R_T(theta - theta0)) over one vector (fp64:
// products of two fp32 values are exact, so each sum is rounded once).
template <int DT>
__device__ __forceinline__ void dot_vec(dz_u32x4 vt, dz_u32x4 va, dz_u32x4 vo, double* acc) {
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    if constexpr (DT == DZ_F32) {
      const float d = __uint_as_float(vt[i]) - __uint_as_float(va[i]);
      *acc = __builtin_fma((double)__uint_as_float(vo[i]), (double)d, *acc);
    } else {
      const F32Pair d = widen_pair<DT>(sub_pair<DT>(vt[i], va[i])), o = widen_pair<DT>(vo[i]);
      *acc = __builtin_fma((double)o.lo, (double)d.lo, *acc);
      *acc = __builtin_fma((double)o.hi, (double)d.hi, *acc);
    }
  }
}
template <int DT>
__device__ __forceinline__ void dot_tail(const char* tp, const char* ap, const char* op, uint32_t e, uint32_t n,
                                         double* acc) {
  using S = typename DT_<DT>::S;
  for (; e < n; ++e) {
    const float d = rt<DT>(DT_<DT>::to_f((uint32_t)((const S*)tp)[e]) - DT_<DT>::to_f((uint32_t)((const S*)ap)[e]));
    *acc = __builtin_fma((double)DT_<DT>::to_f((uint32_t)((const S*)op)[e]), (double)d, *acc);
  }
}

// Elements e .. n - 1 of a chunk, one by one (its last, incomplete vector; the
// rest of a partial chunk goes vector by vector. With all of it one by one, and
// misaligned groups too, 128 groups of 20,480 fp16 elements took 26 us to apply,
// 12 now).
template <int DT, int MODE>
__device__ __forceinline__ void proj_tail(char* tp, const char* ap, uint32_t e, uint32_t n, float alpha, double* acc) {
  using S = typename DT_<DT>::S;
  for (; e < n; ++e) {
    S* p = (S*)tp + e;
    uint32_t r;
    proj_elem<DT>(MODE, (uint32_t)*p, (uint32_t)((const S*)ap)[e], alpha, &r, acc);
    if constexpr (MODE != kProjSumsq) *p = (S)r;
  }
}

// Vector-memory operations a thread issues for a full chunk: its 16-byte
// loads of theta and theta0, and its stores of theta (none for SUMSQ; for DOT
// the loads of the third tensor).
template <int DT, int MODE>
struct ProjChunkOps {
  static constexpr int kVecs = proj_chunk_elems(DT) / (kProjThreads * (16 / (int)sizeof(typename DT_<DT>::S)));
  static constexpr int kAfterTicket = 2 * kVecs + (MODE == kProjSumsq ? 0 : kVecs);  // DOT: a third load
};

// One chunk of a projection launch: the chunk's elements read (theta and
// theta0), updated and written back, and for the SUMSQ modes the chunk's
// partial sum (fixed reduction order) stored at *partial.
template <int DT, int MODE>
__device__ __forceinline__ void proj_chunk(const DzChunk& ch, float alpha, const char* op, double* partial,
                                           double* red) {
  using S = typename DT_<DT>::S;
  constexpr int kES = (int)sizeof(S);
  char* tp = (char*)ch.ptr;
  const char* ap = (const char*)ch.aux;
  double acc = 0.0;
  if (proj_full_chunk<DT>(ch)) {
    constexpr int kVecsPerThread = ProjChunkOps<DT, MODE>::kVecs;
    const ProjScalars<DT, MODE> ps(alpha);
    dz_u32x4 vt[kVecsPerThread], va[kVecsPerThread], vo[MODE == kProjDot ? kVecsPerThread : 1];
#pragma unroll
    for (int u = 0; u < kVecsPerThread; ++u) {
      const size_t off = (size_t)(threadIdx.x + u * kProjThreads) * 16;
      vt[u] = ld_stream(tp + off);
      va[u] = ld_stream(ap + off);
      if constexpr (MODE == kProjDot) vo[u] = ld_stream(op + off);
    }
#pragma unroll
    for (int u = 0; u < kVecsPerThread; ++u) {
      if constexpr (MODE == kProjDot) {
        dot_vec<DT>(vt[u], va[u], vo[u], &acc);
        continue;
      }
      const dz_u32x4 o = proj_vec<DT, MODE>(vt[u], va[u], ps, &acc);
      if constexpr (proj_stores(MODE)) st_stream(tp + (size_t)(threadIdx.x + u * kProjThreads) * 16, o);
    }
  } else {
    const ProjScalars<DT, MODE> ps(alpha);
    constexpr uint32_t kPer = 16 / kES;
    for (uint32_t e = threadIdx.x * kPer; e < ch.n; e += kProjThreads * kPer) {
      if constexpr (MODE == kProjDot) {
        const size_t off = (size_t)e * kES;
        if (e + kPer <= ch.n)
          dot_vec<DT>(ld_stream(tp + off), ld_stream(ap + off), ld_stream(op + off), &acc);
        else
          dot_tail<DT>(tp, ap, op, e, ch.n, &acc);
      } else if (e + kPer <= ch.n) {
        const dz_u32x4 o = proj_vec<DT, MODE>(ld_stream(tp + (size_t)e * kES), ld_stream(ap + (size_t)e * kES), ps, &acc);
        if constexpr (proj_stores(MODE)) st_stream(tp + (size_t)e * kES, o);
      } else {
        proj_tail<DT, MODE>(tp, ap, e, ch.n, alpha, &acc);
      }
    }
  }
  if constexpr (proj_sums(MODE)) {
    const double t = block_sum_f64(acc, red);
    if (threadIdx.x == 0) *partial = t;
  }
}

// alpha of a group: one value of T, or fp32 for APPLY_F32; none for SUMSQ.
template <int DT, int MODE>
__device__ __forceinline__ float group_alpha(const void* __restrict__ alpha_T, uint32_t grp) {
  if constexpr (!proj_stores(MODE)) {
    return 0.0f;
  } else if constexpr (MODE == kProjApplyF32) {
    return ((const float*)alpha_T)[grp];
  } else {
    return DT_<DT>::to_f((uint32_t)((const typename DT_<DT>::S*)alpha_T)[grp]);
  }
}

struct NoGroups {};  // no per-group arguments: the chunks come from the table's list

// Persistent projection kernel: one 1024-thread workgroup per CU takes chunks
// from the table's work counters, as the RMW kernel does (counter j of the K
// in use hands out chunks j, j + K, ...). The groups' alphas are copied to
// LDS once (up to kProjAlphaLds groups; beyond that each chunk reads its
// group's alpha from memory). Wave 0 keeps a pipeline: while chunk k streams,
// lane 0 takes the index of chunk k + 3 and the wave loads the descriptor of
// chunk k + 2 with scalar loads, so no descriptor latency sits between two
// chunks. The last workgroup to finish resets the counters.
template <int DT, int MODE, class Groups>
__global__ void __launch_bounds__(kProjThreads) proj_kernel(const DzChunk* __restrict__ chunks, uint32_t nchunks,
                                                            uint32_t ngroups, const void* __restrict__ alpha_T,
                                                            double* __restrict__ partials,
                                                            uint32_t* __restrict__ counters, Groups dg) {
  __shared__ double red[kProjThreads / 64];
  __shared__ uint32_t sidx[4];   // chunk indices of k .. k + 3 (ring)
  __shared__ DzChunk sdesc[3];   // descriptors of k .. k + 2
  __shared__ float salpha[proj_stores(MODE) ? kProjAlphaLds : 1];
  const bool alpha_in_lds = proj_stores(MODE) && ngroups <= (uint32_t)kProjAlphaLds;
  if (alpha_in_lds) {
    for (uint32_t g = threadIdx.x; g < ngroups; g += kProjThreads) salpha[g] = group_alpha<DT, MODE>(alpha_T, g);
  }
  const uint32_t ncnt = rfl_u32(max(1u, min((uint32_t)kCounters, gridDim.x >> 3)));
  const uint32_t j = rfl_u32((blockIdx.x >> 3) % ncnt);
  uint32_t* mine = counters + j * kCounterStride;
  const uint64_t nch = nchunks;
  // start-up as in rmw_kernel: three tickets from one atomic, then both
  // descriptors loaded together (clamped to a valid index; only tickets below
  // nchunks are used)
  if (threadIdx.x == 0) {
    const uint32_t t0 = atomicAdd(mine, 3u);
    for (int i = 0; i < 3; ++i) sidx[i] = (uint32_t)min((uint64_t)(t0 + i) * ncnt + j, nch);
    if (nch > 0) {
      const DzChunk d0 = chunks[min((uint64_t)t0 * ncnt + j, nch - 1)];
      const DzChunk d1 = chunks[min((uint64_t)(t0 + 1) * ncnt + j, nch - 1)];
      sdesc[0] = d0;
      sdesc[1] = d1;
    }
  }
  __syncthreads();
  for (uint32_t k = 0;; ++k) {
    const uint32_t c = sidx[k % 4];
    if (c >= nchunks) break;
    const DzChunk ch = uniform_proj_chunk<MODE == kProjDot>(sdesc[k % 3]);
    const uint32_t grp = ch.meta;
    const float alpha = !proj_stores(MODE) ? 0.0f
                        : alpha_in_lds     ? salpha[grp]
                                           : group_alpha<DT, MODE>(alpha_T, grp);
    const char* op = nullptr;
    if constexpr (MODE == kProjDot)
      op = (const char*)dg.other[grp - dg.group_base] + ch.zgroup * sizeof(typename DT_<DT>::S);
    uint32_t grabbed = 0;
    uint64_t n_ptr = 0, n_aux = 0, n_off = 0;
    uint32_t n_n = 0, n_meta = 0;
    bool have_desc = false;
    if ((rfl_u32(threadIdx.x) >> 6) == 0) {  // wave 0 (uniform branch)
      const uint32_t cd = rfl_u32(sidx[(k + 2) % 4]);
      if (threadIdx.x == 0) grabbed = ticket_take(mine);
      if (cd < nchunks) {
        const DzChunk* src = chunks + cd;
        n_ptr = src->ptr;
        n_aux = src->aux;
        if constexpr (MODE == kProjDot) n_off = src->zgroup;
        n_n = src->n;
        n_meta = src->meta;
        have_desc = true;
      }
    }
    // lane 0 waits for its ticket behind the chunk's loads and stores (a full
    // chunk issues at least kAfterTicket of them after the ticket; the
    // partial path waits for everything), and the barrier that ends the chunk
    // waits for LDS alone
    if (proj_full_chunk<DT>(ch)) {
      proj_chunk<DT, MODE>(ch, alpha, op, partials + c, red);
      if (threadIdx.x == 0) ticket_wait<ProjChunkOps<DT, MODE>::kAfterTicket>();
    } else {
      proj_chunk<DT, MODE>(ch, alpha, op, partials + c, red);
      if (threadIdx.x == 0) ticket_wait<0>();
    }
    if (threadIdx.x == 0) {
      const uint32_t t = ticket_ready(grabbed);
      sidx[(k + 3) % 4] = (uint32_t)min((uint64_t)t * ncnt + j, nch);
      if (have_desc) {
        DzChunk& d = sdesc[(k + 2) % 3];
        d.ptr = n_ptr;
        d.aux = n_aux;
        d.zgroup = n_off;
        d.n = n_n;
        d.meta = n_meta;
      }
    }
    lds_barrier();
  }
  if (threadIdx.x == 0) {
    const uint32_t done = atomicAdd(counters + kDoneSlot * kCounterStride, 1u);
    if (done == gridDim.x - 1) {
      for (int i = 0; i <= kDoneSlot; ++i) atomicExch(counters + i * kCounterStride, 0u);
    }
  }
}

// A group's results from the sum t of its chunks' partials.
template <int DT>
__device__ __forceinline__ void write_group(const GroupOutputs& o, uint32_t g, double t, bool take_sqrt) {
  using S = typename DT_<DT>::S;
  // correctly rounded fp32 sqrt of the fp32 sum (a double sqrt rounds once more, exactly)
  const float n = take_sqrt ? (float)sqrt((double)(float)t) : (float)t;
  if (o.sumsq) o.sumsq[g] = t;
  if (o.norm_f32) o.norm_f32[g] = n;
  if (o.norm_T) ((S*)o.norm_T)[g] = (S)DT_<DT>::from_f(n);
}

// Per-group reduction of chunk partials, in chunk order. With take_sqrt:
// norm = R_T(sqrt_f32(fp32(sum)))  (torch.norm: fp32 accumulate, fp32 sqrt, cast to T);
// without: the fp32 / T outputs hold the rounded sum itself.
template <int DT>
__global__ void __launch_bounds__(kProjThreads) finalize_kernel(const double* __restrict__ partials,
                                                                const uint32_t* __restrict__ gbegin,
                                                                double* __restrict__ sumsq,
                                                                float* __restrict__ norm_f32,
                                                                void* __restrict__ norm_T, bool take_sqrt) {
  __shared__ double red[kProjThreads / 64];
  const uint32_t g = blockIdx.x;
  const uint32_t b = gbegin[g], e = gbegin[g + 1];
  double x = 0.0;
  for (uint32_t i = b + threadIdx.x; i < e; i += kProjThreads) x += partials[i];
  const double t = block_sum_f64(x, red);
  if (threadIdx.x == 0) write_group<DT>(GroupOutputs{sumsq, norm_f32, norm_T}, g, t, take_sqrt);
}

// ---------------------------------------------------------------------------
// Projection launches over short tables: one workgroup of 256 threads per chunk
// of short_proj_elems, all of a thread's vectors in flight at once, no work
// counters. The workgroup that ends a group's last chunk sums the group's
// partials (in chunk order) and writes its results, so that a norm pass is one
// launch. Without counts (ProjShort) the launch only writes the partials, and a
// kernel behind it sums them in the same order. Chunks come from the table's
// list, or (StaticGroups) from the group list in the launch's arguments.
// ---------------------------------------------------------------------------

// Counts a finished chunk of group g after publishing its partial sum; true in
// every thread of the workgroup that finished last, which then reads the
// group's other partials with read_partial. The partial is written through to
// where every XCD sees it (agent-scope atomic store) and waited for before the
// count, so the count needs no write-back of the L2 for it.
__device__ __forceinline__ bool publish_partial(double* slot, double t, uint32_t* done, uint32_t chunks, uint32_t* flag) {
  if (threadIdx.x == 0) {
    __hip_atomic_store((uint64_t*)slot, __builtin_bit_cast(uint64_t, t), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    const uint32_t before = __hip_atomic_fetch_add(done, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    const bool last = before + 1u == chunks;
    if (last) __hip_atomic_store(done, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);  // for the next launch
    *flag = last ? 1u : 0u;
  }
  __syncthreads();
  return *flag != 0u;
}
__device__ __forceinline__ double read_partial(const double* slot) {
  return __builtin_bit_cast(double, __hip_atomic_load((const uint64_t*)slot, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT));
}

template <int DT, int MODE, class Groups>
__global__ void __launch_bounds__(kShortProjThreads) proj_short_kernel(ProjShort a, Groups sg) {
  constexpr bool kStatic = std::is_same<Groups, StaticGroups>::value;
  using S = typename DT_<DT>::S;
  constexpr uint32_t kPer = 16 / (uint32_t)sizeof(S);
  constexpr int kVecs = short_proj_elems(DT) / (kShortProjThreads * (int)kPer);
  constexpr bool kSums = proj_sums(MODE);
  __shared__ double red[kShortProjThreads / 64];
  __shared__ uint32_t flag;
  uint32_t c = blockIdx.x, grp, first = 0u, count = 0u;
  char* tp;
  const char *ap, *op = nullptr;
  uint32_t n;
  if constexpr (kStatic) {
    uint32_t lo = 0, hi = sg.ngroups;  // the group whose chunks hold c
    while (hi - lo > 1u) {
      const uint32_t mid = (lo + hi) >> 1;
      if (sg.chunk_begin[mid] <= c)
        lo = mid;
      else
        hi = mid;
    }
    const int64_t s = (int64_t)(c - sg.chunk_begin[lo]) * short_proj_elems(DT);
    const int64_t left = sg.numel[lo] - s;
    tp = (char*)sg.ptr[lo] + s * (int64_t)sizeof(S);
    ap = (const char*)sg.anchor[lo] + s * (int64_t)sizeof(S);
    n = (uint32_t)(left < short_proj_elems(DT) ? left : short_proj_elems(DT));
    grp = lo;
  } else {
    if constexpr (MODE == kProjDot) c += sg.chunk_base;
    const DzChunk ch = a.chunks[c];
    tp = (char*)ch.ptr;
    ap = (const char*)ch.aux;
    n = ch.n;
    grp = ch.meta;
    if constexpr (kSums) {
      first = a.group_begin[grp];
      count = a.group_begin[grp + 1] - first;
    }
    if constexpr (MODE == kProjDot) op = (const char*)sg.other[grp - sg.group_base] + ch.zgroup * sizeof(S);
  }
  dz_u32x4 vt[kVecs], va[kVecs], vo[MODE == kProjDot ? kVecs : 1];
#pragma unroll
  for (int u = 0; u < kVecs; ++u) {
    const uint32_t e = (threadIdx.x + (uint32_t)u * kShortProjThreads) * kPer;
    if (e + kPer <= n) {
      vt[u] = ld_any(tp + (size_t)e * sizeof(S));
      va[u] = ld_any(ap + (size_t)e * sizeof(S));
      if constexpr (MODE == kProjDot) vo[u] = ld_any(op + (size_t)e * sizeof(S));
    }
  }
  const ProjScalars<DT, MODE> ps(group_alpha<DT, MODE>(a.alpha, grp));
  double acc = 0.0;
#pragma unroll
  for (int u = 0; u < kVecs; ++u) {
    const uint32_t e = (threadIdx.x + (uint32_t)u * kShortProjThreads) * kPer;
    if constexpr (MODE == kProjDot) {
      if (e + kPer <= n)
        dot_vec<DT>(vt[u], va[u], vo[u], &acc);
      else if (e < n)
        dot_tail<DT>(tp, ap, op, e, n, &acc);
    } else if (e + kPer <= n) {
      const dz_u32x4 o = proj_vec<DT, MODE>(vt[u], va[u], ps, &acc);
      if constexpr (proj_stores(MODE)) st_any(tp + (size_t)e * sizeof(S), o);
    } else if (e < n) {
      proj_tail<DT, MODE>(tp, ap, e, n, ps.alpha, &acc);
    }
  }
  if constexpr (kSums) {
    const double t = block_sum_f64(acc, red);
    if (kStatic || a.group_done == nullptr) {
      if (threadIdx.x == 0) a.partials[c] = t;
    } else if (publish_partial(a.partials + c, t, a.group_done + (size_t)grp * kDoneStride, count, &flag)) {
      double x = 0.0;
      for (uint32_t i = threadIdx.x; i < count; i += kShortProjThreads) x += read_partial(a.partials + first + i);
      const double sum = block_sum_f64(x, red);
      if (threadIdx.x == 0) write_group<DT>(a.out, grp, sum, MODE != kProjDot);
    }
  }
}

// A table-free norm pass over groups of at most kStaticSmallChunks chunks:
// workgroup g computes group g's chunk sums, a quarter of its threads one chunk
// each, and adds them up, all in proj_short_kernel's order.
template <int DT>
__global__ void __launch_bounds__(4 * kShortProjThreads) static_small_kernel(StaticGroups sg, GroupOutputs out) {
  using S = typename DT_<DT>::S;
  constexpr uint32_t kPer = 16 / (uint32_t)sizeof(S), kElems = short_proj_elems(DT);
  constexpr int kVecs = short_proj_elems(DT) / (kShortProjThreads * (int)kPer);
  constexpr int kRounds = kStaticSmallChunks / 4, kWaves = kShortProjThreads / 64;
  __shared__ double red[kStaticSmallChunks][kWaves];
  const uint32_t t = threadIdx.x % kShortProjThreads, team = threadIdx.x / kShortProjThreads;
  char* tp = (char*)sg.ptr[blockIdx.x];
  const char* ap = (const char*)sg.anchor[blockIdx.x];
  const uint32_t numel = (uint32_t)sg.numel[blockIdx.x];
  dz_u32x4 vt[kRounds][kVecs], va[kRounds][kVecs];
#pragma unroll
  for (int k = 0; k < kRounds; ++k) {
#pragma unroll
    for (int u = 0; u < kVecs; ++u) {
      const uint32_t e = (team + 4u * k) * kElems + (t + (uint32_t)u * kShortProjThreads) * kPer;
      if (e + kPer <= numel) {
        vt[k][u] = ld_any(tp + (size_t)e * sizeof(S));
        va[k][u] = ld_any(ap + (size_t)e * sizeof(S));
      }
    }
  }
  const ProjScalars<DT, kProjSumsq> ps(0.0f);
#pragma unroll
  for (int k = 0; k < kRounds; ++k) {
    double acc = 0.0;
#pragma unroll
    for (int u = 0; u < kVecs; ++u) {
      const uint32_t e = (team + 4u * k) * kElems + (t + (uint32_t)u * kShortProjThreads) * kPer;
      if (e + kPer <= numel)
        (void)proj_vec<DT, kProjSumsq>(vt[k][u], va[k][u], ps, &acc);
      else if (e < numel)
        proj_tail<DT, kProjSumsq>(tp, ap, e, numel, 0.0f, &acc);
    }
#pragma unroll
    for (int off = 32; off >= 1; off >>= 1) acc += __shfl_xor(acc, off, 64);
    if ((t & 63u) == 0u) red[team + 4u * k][t >> 6] = acc;
  }
  __syncthreads();
  if (threadIdx.x >= 64) return;
  double x = 0.0;
  if (threadIdx.x < kStaticSmallChunks) {
#pragma unroll
    for (int w = 0; w < kWaves; ++w) x += red[threadIdx.x][w];
  }
#pragma unroll
  for (int off = 32; off >= 1; off >>= 1) x += __shfl_xor(x, off, 64);
  if (threadIdx.x == 0) write_group<DT>(out, sg.group_base + blockIdx.x, x, true);
}

// The group sums of a launch of proj_short_kernel without counts, workgroup g for
// group g of the launch, in that kernel's order, with kAhead loads of a thread in
// flight (one by one, the norms of one group of 8,192 chunks took 34.9 us, now
// 27.8).
template <int DT, class Sums>
__global__ void __launch_bounds__(kShortProjThreads) short_sums_kernel(const double* __restrict__ partials, Sums ss,
                                                                       GroupOutputs out, bool take_sqrt) {
  constexpr int kAhead = 8;
  __shared__ double red[kShortProjThreads / 64];
  const uint32_t b = ss.chunk_begin[blockIdx.x], e = ss.chunk_begin[blockIdx.x + 1];
  double x = 0.0;
  for (uint32_t i = b + threadIdx.x; i < e; i += kAhead * kShortProjThreads) {
    double v[kAhead];
#pragma unroll
    for (int k = 0; k < kAhead; ++k) {
      const uint32_t at = i + (uint32_t)k * kShortProjThreads;
      v[k] = at < e ? partials[at] : 0.0;
    }
#pragma unroll
    for (int k = 0; k < kAhead; ++k) x += v[k];
  }
  const double t = block_sum_f64(x, red);
  if (threadIdx.x == 0) write_group<DT>(out, ss.group_base + blockIdx.x, t, take_sqrt);
}

// Chunk descriptors of a projection launch planned on the device (the
// table-free norm pass): block g writes group g's chunks, split as
// dz_table_create splits them (proj_chunk_elems(dtype) elements, the last one
// shorter), and its first chunk index; the last batch also writes the end index of the last group. The
// first batch zeroes the work counters the projection kernel takes chunks
// from.
__global__ void __launch_bounds__(256) static_plan_kernel(StaticPlanBatch b, DzChunk* __restrict__ chunks,
                                                          uint32_t* __restrict__ group_begin,
                                                          uint32_t* __restrict__ counters) {
  const uint32_t g = blockIdx.x;
  if (b.first && g == 0) {
    for (int i = threadIdx.x; i < kCounterWords; i += blockDim.x) counters[i] = 0u;
  }
  if (g >= b.ngroups) return;
  const uint32_t gi = b.group_base + g;
  const uint64_t p = b.ptr[g], a = b.anchor[g];
  const int64_t ne = b.numel[g];
  const uint32_t meta = gi;
  const int64_t cn = b.chunk_elems;
  const uint32_t nch = (uint32_t)((ne + cn - 1) / cn);
  for (uint32_t k = threadIdx.x; k < nch; k += blockDim.x) {
    const uint64_t s = (uint64_t)k * (uint64_t)cn;
    DzChunk c;
    c.ptr = p + s * (uint64_t)b.elem_size;
    c.aux = a + s * (uint64_t)b.elem_size;
    c.zgroup = s;
    c.n = (uint32_t)min(cn, ne - (int64_t)s);
    c.meta = meta;
    chunks[b.chunk_begin[g] + k] = c;
  }
  if (threadIdx.x == 0) {
    group_begin[gi] = b.chunk_begin[g];
    if (gi + 1 == b.total_groups) group_begin[b.total_groups] = b.total_chunks;
  }
}

// One vector of z (kPer elements of T) from element e of the launch's groups:
// n elements from element `offset` of the stream make groups of 8 (one Philox
// block each) whose element e is output e - skip, skip = offset mod 8. Element
// indices wrap modulo 2^64.
template <int DT, int kPer>
__device__ __forceinline__ void store_z(dz_u32x4 v, uint64_t e, uint32_t skip, uint64_t n, void* out) {
  using S = typename DT_<DT>::S;
  const int64_t i0 = (int64_t)e - (int64_t)skip;
  S* p = (S*)out + i0;
  if (i0 >= 0 && (uint64_t)i0 + kPer <= n) {
    st_any(p, v);
  } else {
#pragma unroll
    for (int j = 0; j < kPer; ++j) {
      const uint32_t b = DT == DZ_F32 ? v[j & 3] : v[(j >> 1) & 3] >> (16 * (j & 1));
      if (i0 + j >= 0 && (uint64_t)(i0 + j) < n) p[j] = (S)b;
    }
  }
}

// z(seed, stream, offset + i) for i < n, written densely in T: one thread per
// Philox block of 8 elements, looked up in the quantile table in memory. For
// short ranges, which a launch's start and one chain of latencies bound (1.5
// us for a wave's worth, 2.8 at 2^16 fp16 elements).
template <int DT>
__global__ void __launch_bounds__(256) normals_kernel(const void* __restrict__ gtab, uint64_t seed,
                                                      uint32_t stream, uint64_t offset, uint64_t n,
                                                      void* __restrict__ out) {
  const uint32_t skip = (uint32_t)(offset & 7u);
  const uint64_t g = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (g * 8u >= n + skip) return;
  const DzU4 w = dz_philox_group(seed, stream, (offset - skip + g * 8u) >> 3);
  const ZVec<DT> z = z_vec<DT>((const typename DT_<DT>::S*)gtab, w);
#pragma unroll
  for (int k = 0; k < ZVec<DT>::kVecs; ++k)
    store_z<DT, 8 / ZVec<DT>::kVecs>(z.v[k], g * 8u + (uint64_t)k * (8 / ZVec<DT>::kVecs), skip, n, out);
}

// The same for long ranges: persistent workgroups copy the quantile table to
// LDS once (64 KB for 16-bit T, two workgroups per CU; 128 KB for fp32, one),
// then take tiles of 1024 groups in turn. 105 M fp16 elements into buffers
// used in turn take 44 us, 4.8 TB/s of stores (with a thread and a block of
// the generator per element 214 us); 2^27 fp16 elements into one buffer, which
// the Infinity Cache holds, 44 us, where the Philox chain's VALU work is the
// bound; 2^27 fp32 elements 124 us (4.3 TB/s). The stores are plain ones: with
// the non-temporal hint 2^27 elements took 84 us (fp16) and 252 us (fp32), and
// whoever asked for z reads it next.
template <int DT>
__global__ void __launch_bounds__(kNormalsThreads, DT == DZ_F32 ? 4 : 8)
    normals_lds_kernel(const void* __restrict__ gtab, uint64_t seed, uint32_t stream, uint64_t offset, uint64_t n,
                       void* __restrict__ out) {
  using S = typename DT_<DT>::S;
  __shared__ __attribute__((aligned(16))) S tab[kDzTabEntries];
  constexpr int kSlices = kDzTabEntries * (int)sizeof(S) / (16 * kNormalsThreads);
#pragma unroll
  for (int v = 0; v < kSlices; ++v) {
    const uint32_t at = (uint32_t)(v * kNormalsThreads + threadIdx.x) * 16u;
    *(dz_u32x4*)((char*)tab + at) = *(const dz_u32x4*)((const char*)gtab + at);
  }
  __syncthreads();
  const uint32_t skip = (uint32_t)(offset & 7u);
  const uint64_t groups = (n + skip + 7u) >> 3;
  const uint64_t first = offset - skip;
  for (uint64_t t = blockIdx.x; t * kNormalsThreads < groups; t += gridDim.x) {
    const uint64_t g0 = t * kNormalsThreads;  // the tile's first group
    if (g0 + (threadIdx.x & ~63u) >= groups) break;  // whole waves: fp32 lanes exchange words
    const uint32_t g = tile_group<DT>(0);
    const uint64_t q = (first + g0 * 8u) >> 3;
    // the counters' high word is uniform over the tile unless the low word
    // (or the element index) wraps in it
    const DzU4 w = (uint32_t)q <= 0xffffffffu - (kNormalsThreads - 1u)
                       ? dz_philox_counter(seed, stream, (uint32_t)q + g, (uint32_t)(q >> 32))
                       : dz_philox_group(seed, stream, (first + (g0 + g) * 8u) >> 3);
    const ZVec<DT> z = z_vec<DT>(tab, thread_words<DT>(w));
    if constexpr (DT == DZ_F32) {
      const uint64_t e = (g0 + (threadIdx.x & ~63u)) * 8u + (threadIdx.x & 63u) * 4u;
      store_z<DT, 4>(z.v[0], e, skip, n, out);
      store_z<DT, 4>(z.v[1], e + 256u, skip, n, out);
    } else {
      store_z<DT, 8>(z.v[0], (g0 + g) * 8u, skip, n, out);
    }
  }
}

// Raw Philox blocks for counter q = q0 + i (test and KAT use).
__global__ void __launch_bounds__(256) philox_kernel(uint64_t seed, uint32_t stream, uint64_t q0,
                                                     uint64_t n, uint32_t* __restrict__ out) {
  const uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  const DzU4 w = dz_philox_group(seed, stream, q0 + i);
  out[4 * i + 0] = w.x;
  out[4 * i + 1] = w.y;
  out[4 * i + 2] = w.z;
  out[4 * i + 3] = w.w;
}

// ---------------------------------------------------------------------------
// Launchers (host side, C++ linkage; the C ABI validates before calling).
// With timing events given (LaunchEvents), a launch goes through
// hipExtLaunchKernel, which records them when the kernel starts and ends.
// ---------------------------------------------------------------------------
#define DZ_LAUNCH(kernel, grid, block, st, ev, ...)                                              \
  do {                                                                                          \
    if ((ev).start || (ev).stop) {                                                              \
      hipExtLaunchKernelGGL(kernel, grid, block, 0, st, (ev).start, (ev).stop, 0, __VA_ARGS__); \
    } else {                                                                                    \
      hipLaunchKernelGGL(kernel, grid, block, 0, st, __VA_ARGS__);                              \
    }                                                                                           \
  } while (0)

template <int DT, bool kPlain>
static hipError_t launch_rmw_dt(int mode, const DzChunk* chunks, uint32_t nchunks, uint32_t grid,
                                const void* tab, const DzScalars& s, const DzScalarPtrs& p,
                                uint32_t* counters, bool prefetch, hipStream_t st, const LaunchEvents& ev) {
  switch (mode) {
    case kModePerturb:
      DZ_LAUNCH((rmw_kernel<DT, kModePerturb, false, kPlain>), dim3(grid), dim3(kRmwThreads), st, ev,
                         chunks, nchunks, tab, s, p, counters);
      break;
    case kModeUpdate:
      DZ_LAUNCH((rmw_kernel<DT, kModeUpdate, false, kPlain>), dim3(grid), dim3(kRmwThreads), st, ev,
                         chunks, nchunks, tab, s, p, counters);
      break;
    case kModeRestoreUpdate:
      DZ_LAUNCH((rmw_kernel<DT, kModeRestoreUpdate, false, kPlain>), dim3(grid), dim3(kRmwThreads),
                         st, ev, chunks, nchunks, tab, s, p, counters);
      break;
    case kModeRestoreUpdatePerturb:
      // the caller asks for the prefetching loop on long launches (the table's prefetch_min_tiles)
      if (RmwTraits<DT, kModeRestoreUpdatePerturb>::kPrefetch && prefetch) {
        DZ_LAUNCH((rmw_kernel<DT, kModeRestoreUpdatePerturb, true, kPlain>), dim3(grid), dim3(kRmwThreads),
                           st, ev, chunks, nchunks, tab, s, p, counters);
      } else {
        DZ_LAUNCH((rmw_kernel<DT, kModeRestoreUpdatePerturb, false, kPlain>), dim3(grid), dim3(kRmwThreads),
                           st, ev, chunks, nchunks, tab, s, p, counters);
      }
      break;
    default:
      return hipErrorInvalidValue;
  }
  return hipGetLastError();
}

hipError_t launch_rmw(int dtype, int mode, const DzChunk* chunks, uint32_t nchunks, uint32_t grid,
                      const void* tab, const DzScalars& s, const DzScalarPtrs& p, uint32_t* counters,
                      bool prefetch, bool plain, hipStream_t st, const LaunchEvents& ev) {
  const auto go = [&](auto launch) {
    return launch(mode, chunks, nchunks, grid, tab, s, p, counters, prefetch, st, ev);
  };
  switch (dtype) {
    case DZ_F32: return plain ? go(launch_rmw_dt<DZ_F32, true>) : go(launch_rmw_dt<DZ_F32, false>);
    case DZ_F16: return plain ? go(launch_rmw_dt<DZ_F16, true>) : go(launch_rmw_dt<DZ_F16, false>);
    case DZ_BF16: return plain ? go(launch_rmw_dt<DZ_BF16, true>) : go(launch_rmw_dt<DZ_BF16, false>);
    default: return hipErrorInvalidValue;
  }
}

template <int DT>
static hipError_t launch_rmw_short_dt(int mode, const DzChunk* chunks, uint32_t nchunks, uint32_t cus, const void* tab,
                                      const DzScalars& s, const DzScalarPtrs& p, hipStream_t st,
                                      const LaunchEvents& ev) {
  const uint32_t most = cus * (DT == DZ_F32 ? 1u : 2u);  // workgroups that the LDS tables leave room for
  const dim3 grid(nchunks < most ? nchunks : most), block(kRmwThreads);
  switch (mode) {
    case kModePerturb:
      DZ_LAUNCH((rmw_short_kernel<DT, kModePerturb>), grid, block, st, ev, chunks, nchunks, tab, s, p);
      break;
    case kModePerturbUnit:
      DZ_LAUNCH((rmw_short_kernel<DT, kModePerturbUnit>), grid, block, st, ev, chunks, nchunks, tab, s, p);
      break;
    case kModeUpdate:
      DZ_LAUNCH((rmw_short_kernel<DT, kModeUpdate>), grid, block, st, ev, chunks, nchunks, tab, s, p);
      break;
    case kModeRestoreUpdate:
      DZ_LAUNCH((rmw_short_kernel<DT, kModeRestoreUpdate>), grid, block, st, ev, chunks, nchunks, tab, s, p);
      break;
    case kModeRestoreUpdatePerturb:
      DZ_LAUNCH((rmw_short_kernel<DT, kModeRestoreUpdatePerturb>), grid, block, st, ev, chunks, nchunks, tab, s, p);
      break;
    default:
      return hipErrorInvalidValue;
  }
  return hipGetLastError();
}

hipError_t launch_rmw_short(int dtype, int mode, const DzChunk* chunks, uint32_t nchunks, uint32_t cus, const void* tab,
                            const DzScalars& s, const DzScalarPtrs& p, hipStream_t st, const LaunchEvents& ev) {
  switch (dtype) {
    case DZ_F32: return launch_rmw_short_dt<DZ_F32>(mode, chunks, nchunks, cus, tab, s, p, st, ev);
    case DZ_F16: return launch_rmw_short_dt<DZ_F16>(mode, chunks, nchunks, cus, tab, s, p, st, ev);
    case DZ_BF16: return launch_rmw_short_dt<DZ_BF16>(mode, chunks, nchunks, cus, tab, s, p, st, ev);
    default: return hipErrorInvalidValue;
  }
}

template <int DT>
static hipError_t launch_proj_dt(int mode, const DzChunk* chunks, uint32_t nchunks, uint32_t ngroups,
                                 uint32_t grid, const void* alpha, double* partials, uint32_t* counters,
                                 hipStream_t st, const LaunchEvents& ev) {
  switch (mode) {
    case kProjSumsq:
      DZ_LAUNCH((proj_kernel<DT, kProjSumsq, NoGroups>), dim3(grid), dim3(kProjThreads), st, ev, chunks, nchunks,
                         ngroups, alpha, partials, counters, NoGroups{});
      break;
    case kProjApply:
      DZ_LAUNCH((proj_kernel<DT, kProjApply, NoGroups>), dim3(grid), dim3(kProjThreads), st, ev, chunks, nchunks,
                         ngroups, alpha, partials, counters, NoGroups{});
      break;
    case kProjReverse:
      DZ_LAUNCH((proj_kernel<DT, kProjReverse, NoGroups>), dim3(grid), dim3(kProjThreads), st, ev, chunks, nchunks,
                         ngroups, alpha, partials, counters, NoGroups{});
      break;
    case kProjReverseSumsq:
      DZ_LAUNCH((proj_kernel<DT, kProjReverseSumsq, NoGroups>), dim3(grid), dim3(kProjThreads), st, ev, chunks,
                         nchunks, ngroups, alpha, partials, counters, NoGroups{});
      break;
    case kProjApplyF32:
      DZ_LAUNCH((proj_kernel<DT, kProjApplyF32, NoGroups>), dim3(grid), dim3(kProjThreads), st, ev, chunks, nchunks,
                         ngroups, alpha, partials, counters, NoGroups{});
      break;
    default:
      return hipErrorInvalidValue;
  }
  return hipGetLastError();
}

hipError_t launch_proj(int dtype, int mode, const DzChunk* chunks, uint32_t nchunks, uint32_t ngroups,
                       uint32_t grid, const void* alpha, double* partials, uint32_t* counters, hipStream_t st,
                       const LaunchEvents& ev) {
  switch (dtype) {
    case DZ_F32:
      return launch_proj_dt<DZ_F32>(mode, chunks, nchunks, ngroups, grid, alpha, partials, counters, st, ev);
    case DZ_F16:
      return launch_proj_dt<DZ_F16>(mode, chunks, nchunks, ngroups, grid, alpha, partials, counters, st, ev);
    case DZ_BF16:
      return launch_proj_dt<DZ_BF16>(mode, chunks, nchunks, ngroups, grid, alpha, partials, counters, st, ev);
    default: return hipErrorInvalidValue;
  }
}

template <int DT>
static hipError_t launch_proj_short_dt(int mode, uint32_t nchunks, const ProjShort& a, hipStream_t st,
                                       const LaunchEvents& ev) {
  const dim3 grid(nchunks), block(kShortProjThreads);
  const NoGroups none{};
  switch (mode) {
    case kProjSumsq: DZ_LAUNCH((proj_short_kernel<DT, kProjSumsq, NoGroups>), grid, block, st, ev, a, none); break;
    case kProjApply: DZ_LAUNCH((proj_short_kernel<DT, kProjApply, NoGroups>), grid, block, st, ev, a, none); break;
    case kProjReverse: DZ_LAUNCH((proj_short_kernel<DT, kProjReverse, NoGroups>), grid, block, st, ev, a, none); break;
    case kProjReverseSumsq:
      DZ_LAUNCH((proj_short_kernel<DT, kProjReverseSumsq, NoGroups>), grid, block, st, ev, a, none);
      break;
    case kProjApplyF32: DZ_LAUNCH((proj_short_kernel<DT, kProjApplyF32, NoGroups>), grid, block, st, ev, a, none); break;
    default: return hipErrorInvalidValue;
  }
  return hipGetLastError();
}

hipError_t launch_proj_short(int dtype, int mode, uint32_t nchunks, const ProjShort& a, hipStream_t st,
                             const LaunchEvents& ev) {
  switch (dtype) {
    case DZ_F32: return launch_proj_short_dt<DZ_F32>(mode, nchunks, a, st, ev);
    case DZ_F16: return launch_proj_short_dt<DZ_F16>(mode, nchunks, a, st, ev);
    case DZ_BF16: return launch_proj_short_dt<DZ_BF16>(mode, nchunks, a, st, ev);
    default: return hipErrorInvalidValue;
  }
}

hipError_t launch_static_sumsq(int dtype, uint32_t nchunks, double* partials, const StaticGroups& sg, hipStream_t st) {
  const LaunchEvents ev{};
  const ProjShort a{nullptr, nullptr, nullptr, nullptr, partials, {}};
  const dim3 grid(nchunks), block(kShortProjThreads);
  switch (dtype) {
    case DZ_F32: DZ_LAUNCH((proj_short_kernel<DZ_F32, kProjSumsq, StaticGroups>), grid, block, st, ev, a, sg); break;
    case DZ_F16: DZ_LAUNCH((proj_short_kernel<DZ_F16, kProjSumsq, StaticGroups>), grid, block, st, ev, a, sg); break;
    case DZ_BF16: DZ_LAUNCH((proj_short_kernel<DZ_BF16, kProjSumsq, StaticGroups>), grid, block, st, ev, a, sg); break;
    default: return hipErrorInvalidValue;
  }
  return hipGetLastError();
}

hipError_t launch_static_small(int dtype, const StaticGroups& sg, const GroupOutputs& out, hipStream_t st) {
  const LaunchEvents ev{};
  const dim3 grid(sg.ngroups), block(4 * kShortProjThreads);
  switch (dtype) {
    case DZ_F32: DZ_LAUNCH((static_small_kernel<DZ_F32>), grid, block, st, ev, sg, out); break;
    case DZ_F16: DZ_LAUNCH((static_small_kernel<DZ_F16>), grid, block, st, ev, sg, out); break;
    case DZ_BF16: DZ_LAUNCH((static_small_kernel<DZ_BF16>), grid, block, st, ev, sg, out); break;
    default: return hipErrorInvalidValue;
  }
  return hipGetLastError();
}

template <class Sums>
static hipError_t launch_sums(int dtype, uint32_t ngroups, const double* partials, const Sums& ss, const GroupOutputs& out,
                              bool take_sqrt, hipStream_t st, const LaunchEvents& ev) {
  const dim3 grid(ngroups), block(kShortProjThreads);
  switch (dtype) {
    case DZ_F32: DZ_LAUNCH((short_sums_kernel<DZ_F32, Sums>), grid, block, st, ev, partials, ss, out, take_sqrt); break;
    case DZ_F16: DZ_LAUNCH((short_sums_kernel<DZ_F16, Sums>), grid, block, st, ev, partials, ss, out, take_sqrt); break;
    case DZ_BF16: DZ_LAUNCH((short_sums_kernel<DZ_BF16, Sums>), grid, block, st, ev, partials, ss, out, take_sqrt); break;
    default: return hipErrorInvalidValue;
  }
  return hipGetLastError();
}

hipError_t launch_static_sums(int dtype, uint32_t ngroups, const double* partials, const StaticSums& ss,
                              const GroupOutputs& out, hipStream_t st) {
  return launch_sums(dtype, ngroups, partials, ss, out, true, st, {});
}

hipError_t launch_short_sums(int dtype, uint32_t ngroups, const double* partials, const TableSums& ts,
                             const GroupOutputs& out, bool take_sqrt, hipStream_t st, const LaunchEvents& ev) {
  return launch_sums(dtype, ngroups, partials, ts, out, take_sqrt, st, ev);
}

template <int DT>
static void launch_dot_dt(const DzChunk* chunks, uint32_t nchunks, uint32_t grid, const DotGroups& dg, double* partials,
                          uint32_t* counters, hipStream_t st, const LaunchEvents& ev) {
  const void* no_alpha = nullptr;
  DZ_LAUNCH((proj_kernel<DT, kProjDot, DotGroups>), dim3(grid), dim3(kProjThreads), st, ev, chunks, nchunks, 0u, no_alpha,
            partials, counters, dg);
}

hipError_t launch_dot(int dtype, const DzChunk* chunks, uint32_t nchunks, uint32_t grid, const DotGroups& dg,
                      double* partials, uint32_t* counters, hipStream_t st, const LaunchEvents& ev) {
  switch (dtype) {
    case DZ_F32: launch_dot_dt<DZ_F32>(chunks, nchunks, grid, dg, partials, counters, st, ev); break;
    case DZ_F16: launch_dot_dt<DZ_F16>(chunks, nchunks, grid, dg, partials, counters, st, ev); break;
    case DZ_BF16: launch_dot_dt<DZ_BF16>(chunks, nchunks, grid, dg, partials, counters, st, ev); break;
    default: return hipErrorInvalidValue;
  }
  return hipGetLastError();
}

hipError_t launch_dot_short(int dtype, uint32_t nchunks, const ProjShort& a, const DotGroups& dg, hipStream_t st,
                            const LaunchEvents& ev) {
  const dim3 grid(nchunks), block(kShortProjThreads);
  switch (dtype) {
    case DZ_F32: DZ_LAUNCH((proj_short_kernel<DZ_F32, kProjDot, DotGroups>), grid, block, st, ev, a, dg); break;
    case DZ_F16: DZ_LAUNCH((proj_short_kernel<DZ_F16, kProjDot, DotGroups>), grid, block, st, ev, a, dg); break;
    case DZ_BF16: DZ_LAUNCH((proj_short_kernel<DZ_BF16, kProjDot, DotGroups>), grid, block, st, ev, a, dg); break;
    default: return hipErrorInvalidValue;
  }
  return hipGetLastError();
}

hipError_t launch_finalize(int dtype, const double* partials, const uint32_t* gbegin, uint32_t ngroups,
                           double* sumsq, float* norm_f32, void* norm_T, bool take_sqrt, hipStream_t st,
                           const LaunchEvents& ev) {
  switch (dtype) {
    case DZ_F32:
      DZ_LAUNCH((finalize_kernel<DZ_F32>), dim3(ngroups), dim3(kProjThreads), st, ev,
                         partials, gbegin, sumsq, norm_f32, norm_T, take_sqrt);
      break;
    case DZ_F16:
      DZ_LAUNCH((finalize_kernel<DZ_F16>), dim3(ngroups), dim3(kProjThreads), st, ev,
                         partials, gbegin, sumsq, norm_f32, norm_T, take_sqrt);
      break;
    case DZ_BF16:
      DZ_LAUNCH((finalize_kernel<DZ_BF16>), dim3(ngroups), dim3(kProjThreads), st, ev,
                         partials, gbegin, sumsq, norm_f32, norm_T, take_sqrt);
      break;
    default:
      return hipErrorInvalidValue;
  }
  return hipGetLastError();
}

hipError_t launch_static_plan(const StaticPlanBatch& b, DzChunk* chunks, uint32_t* group_begin, uint32_t* counters,
                              hipStream_t st) {
  hipLaunchKernelGGL(static_plan_kernel, dim3(b.ngroups ? b.ngroups : 1), dim3(256), 0, st, b, chunks, group_begin,
                     counters);
  return hipGetLastError();
}

template <int DT>
static void launch_normals_dt(const void* tab, uint64_t seed, uint32_t stream, uint64_t offset, uint64_t n, void* out,
                              uint32_t cus, hipStream_t st) {
  const uint64_t groups = ((offset & 7u) + n + 7u) >> 3;
  if (groups >= kNormalsLdsGroups) {
    const uint32_t grid = cus * (DT == DZ_F32 ? 1u : 2u);
    hipLaunchKernelGGL((normals_lds_kernel<DT>), dim3(grid), dim3(kNormalsThreads), 0, st, tab, seed, stream, offset, n,
                       out);
  } else {
    hipLaunchKernelGGL((normals_kernel<DT>), dim3((uint32_t)((groups + 255) / 256)), dim3(256), 0, st, tab, seed, stream,
                       offset, n, out);
  }
}

hipError_t launch_normals(int dtype, const void* tab, uint64_t seed, uint32_t stream, uint64_t offset,
                          uint64_t n, void* out, uint32_t cus, hipStream_t st) {
  switch (dtype) {
    case DZ_F32: launch_normals_dt<DZ_F32>(tab, seed, stream, offset, n, out, cus, st); break;
    case DZ_F16: launch_normals_dt<DZ_F16>(tab, seed, stream, offset, n, out, cus, st); break;
    case DZ_BF16: launch_normals_dt<DZ_BF16>(tab, seed, stream, offset, n, out, cus, st); break;
    default: return hipErrorInvalidValue;
  }
  return hipGetLastError();
}

hipError_t launch_philox(uint64_t seed, uint32_t stream, uint64_t q0, uint64_t n, uint32_t* out,
                         hipStream_t st) {
  const uint64_t blocks = (n + 255) / 256;
  hipLaunchKernelGGL(philox_kernel, dim3((uint32_t)blocks), dim3(256), 0, st, seed, stream, q0, n, out);
  return hipGetLastError();
}

}  // namespace dz
