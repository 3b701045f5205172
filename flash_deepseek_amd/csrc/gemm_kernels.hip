// gemm_kernels.hip -- the grouped expert GEMMs of batched decode and prefill
// on MFMA: per distinct expert (and the shared one), its tokens' activations
// against the expert's Q4_K rows for gate/up (+ SwiGLU) and its Q4_K or Q6_K
// rows for the down.
//
// Numerics.  Inside one Q4_K block a weight is d*sc*q - dmin*m (quant.c:49-57)
// with 6-bit sc, m and 4-bit q, so
//   sum_k w_k x_k = d * sum_k sc_k q_k x_k - dmin * sum_sb m_sb X_sb
// (X_sb: the sum of the sub-block's 32 activations).  The integer sc*q <= 945
// is exact in fp16 and is built per element pair by one mask-or and one
// packed fma: (0x6400 | q) is the half 1024 + q, and (1024 + q) sc - 1024 sc
// is sc q exactly (one rounding of an exact half).  The MFMA
// (v_mfma_f32_16x16x32_f16, fp32 accumulation) contracts it with the
// activations over a whole block and the scales are applied once per block:
//   y += d * C  -  sum_sb X_sb dmin m_sb
// the second term by 16x16x4 fp32 MFMAs over the block's eight sub-blocks.
// (Weights carried as 1024 + sc q, with 1024 X cancelled afterwards, would
// inflate the accumulator several times over the sum it carries and cost
// the batched path its fp32 grade on SwiGLU activations.)
// A Q6_K weight is d*sc*(q - 32) with an int8 sc per 16 elements: the integer
// sc (q - 32), up to 13 significant bits, enters as two halves (build_b6),
// with no min term.
// Activations enter as P fp16 planes of x' = x * 2^s (a per-row power of
// two: the largest |x'| lies in [2^13, 2^14)): P = 3 carries every fp32
// value exactly (hi + mid + lo, 33 significant bits) -- batched decode and
// every Q6_K down, fp32 grade; P = 1 carries 11 bits -- prefill, whose bar is
// 1e-2.  X_sb is the sum of the planes' values (planes_device.h).
//
// Mapping.  A workgroup of 4 waves owns 64 gate and 64 up rows (wave w:
// rows 16 w .. 16 w + 15 of both, two of gate and the same two of up by turns
// in its two 16-column tiles, as the resident layout holds them) or 128 down
// rows (wave w: two tiles of 16) for one chunk of tokens of one expert.
// Weight rows are the MFMA columns (B operand): lane (c, j)
// holds row c and group j (qs bytes 32 j .. 32 j + 31, sub-blocks 2j, 2j+1)
// of every block, read as two whole 16-byte pieces of the resident expert
// layout: four consecutive lanes, four rows' group j, read one 64-byte run,
// and each lane needs only its own group's two scales and mins.  MFMA step m
// (0..7) of a block takes from lane j the 8 elements 64 j + 8 m .. + 7 (low
// nibbles for m < 4, high nibbles for m >= 4); the token operand (A, from
// LDS) reads the same elements.  Per block the chunk's token planes are
// copied global -> LDS by direct loads into one of two buffers, so block
// b + 1 streams in while block b is contracted.
//
// What bounds it.  A read of the same weight lines with the same tiles and
// no math takes 180-205 us for 71 experts' gate and up (5.7-6.6 TB/s).  The
// vector ALU (three planes: 97, 105 and 117 instructions per 16-row tile and
// block at up to 5, 10 and 16 tokens, of them 64 for the weight operands; one
// plane 93 .. 105) and the matrix cores (8, 16 or 24 16x16x32 of 16 cycles and
// two 16x16x4 of 32) need about as long and overlap only partly, so the kernel
// lives on loads in flight and on few instructions.  What that came to, gate/up
// of a step of 16 tokens unless said otherwise, each before and after on one box
// (boxes differ by 5%):
//  - the three planes of a chunk of few tokens share 16-row operands:
//    up to 5 tokens cost 8 MFMAs per tile and block instead of 24 and a
//    third of the LDS traffic; with that, two tiles per wave and three waves
//    per SIMD beat four tiles and two waves (328 -> 234 us; four tiles 279);
//  - each weight register is refilled with block b + 2 right after its last
//    use, so the stream runs one to two blocks ahead on two register sets; and
//    buffer loads: no address arithmetic on the vector ALU, and a pad row's
//    planes and sub-block sums lie past the buffer's end, so they cost no
//    traffic and the sums no select that waits for the load (234 -> 219);
//  - a block's scales and mins are taken from the header two at a time (220 ->
//    213);
//  - three planes' items lie on the XCDs in contiguous ranges (221 -> 210);
//  - the resident layout's row-fastest pieces halve the L1 cycles of a weight
//    load (210 -> 199; 64 / 256 tokens 468 -> 444, 883 -> 855);
//  - an expert with one chunk is streamed past the L2 (nontemporal).
// On one build and box: gate/up of 71 / 130 / 176 experts (16 / 64 / 256 tokens)
// 213, 459 and 909 us, the down of 16 / 256 tokens 117 and 486 us; one plane, 512
// tokens, gate/up 844, down 474 us.
// The Q6_K down costs 196 .. 208 vector instructions per tile and block (two
// halves per weight, six bits from two places) and 16, 32 or 48 MFMAs: 375 us for
// 130 experts of 64 tokens, where the dot4 kernel, which unpacks every weight
// again for every token, took 922; 538 against 1906 us for 150 prompt tokens.
#include "fdm_internal.h"
#include "planes_device.h"
#include "route_device.h"

#include <type_traits>

namespace fdm {

namespace {

typedef unsigned short u16x2 __attribute__((ext_vector_type(2)));
typedef _Float16 f16x2 __attribute__((ext_vector_type(2)));

constexpr int kQWaves = 4;            // waves per workgroup
constexpr int kQRowB = kQK * 2;       // LDS token row: one block of fp16 (512 B)
constexpr int kQMaxTok = 64;          // tokens of the largest chunk
// Weight tiles of 16 columns per wave: two of gate/up (8 rows of each, gate
// and up by turns of two), or two of down; every token operand read from LDS serves both.
constexpr int kQTiles = 2;
// Waves per SIMD: 3 for three planes (168 VGPRs), 2 for one plane, whose
// 64-token chunks hold four operand blocks of accumulators.
__host__ __device__ constexpr int qgemm_waves(int planes) { return planes == 3 ? 3 : 2; }
__host__ __device__ constexpr int qgemm_rows(bool down) {  // rows per workgroup (of gate for gate/up)
  return (down ? 16 : 8) * kQTiles * kQWaves;
}

// The matrices a grouped GEMM contracts.
enum QMat { kGateUp, kDownQ4, kDownQ6 };

// One lane's share of one block of one weight row (resident expert layout).
// Q4_K: its group's 32 qs bytes (q0, q1) and the 16-byte block header.
// Q6_K: lane j = 2 h + s holds 16 weights of each quarter k of half h: ql
// chunk s (q0: quarters 0 and 2), ql chunk 2 + s (q1: quarters 1 and 3) and qh
// chunk s; hdr = the half's 8 scales and the block's d.
template <QMat M>
struct QLane {
  u32x4 q0, q1, hdr;
};
typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
template <>
struct QLane<kDownQ6> {
  u32x4 q0, q1, qh;
  u32x2 sc;
  uint32_t d;
};

// fp16 halves of sc * q for the two q held in bits 0-3 (MASK 0x000F000F)
// of the halves of w, the rest of w arbitrary: 0x6400 | q is the half
// 1024 + q, and one fused multiply-add per half, (1024 + q) sc - 1024 sc,
// gives sc q exactly (q < 16, sc < 64: the exact result is a half, which the
// single rounding keeps).  For the q in bits 4-7 (MASK 0x00F000F0),
// 0x6400 | 16 q is the half 1024 + 16 q, and (1024 + 16 q) (sc / 16) - 64 sc
// is sc q exactly, with no shift to bring the nibble down.  Both halves of
// the fma read one half of k and of a (op_sel).
template <uint32_t MASK>
__device__ __forceinline__ uint32_t magic2(uint32_t w, _Float16 k, _Float16 a) {
  // one v_and_or_b32 (mask from an SGPR, 0x64006400 from a VGPR: a VOP3
  // takes no literal and one SGPR), which the compiler otherwise splits
  uint32_t m;
  asm("v_and_or_b32 %0, %1, %2, %3" : "=v"(m) : "v"(w), "s"(MASK), "v"(0x64006400u));
  const f16x2 v = __builtin_bit_cast(f16x2, m);
  return __builtin_bit_cast(uint32_t, __builtin_elementwise_fma(v, (f16x2){k, k}, (f16x2){a, a}));
}

// The B operands of MFMA steps m (low nibbles) and m + 4 (high nibbles):
// bytes 8 m' .. 8 m' + 7 of the lane's group, m' = m & 3 (q0 for m' < 2).
// Elements are taken in the order 0 2 1 3 4 6 5 7 of each 8 (the order in
// which k_xplanes stores the activations): a dword of qs holds the low
// nibbles of elements 0 and 2 at bits 0 and 16 and their high nibbles at
// bits 4 and 20, elements 1 and 3 eight bits higher, so one shift per dword
// and per fp16 pair one mask-or and one packed fma suffice.
struct BPair {
  f16x8 lo, hi;
};

__device__ __forceinline__ BPair build_b(uint32_t w0, uint32_t w1, f16x2 k, f16x2 a) {
  const uint32_t v0 = w0 >> 8, v1 = w1 >> 8;
  u32x4 lo, hi;
  lo.x = magic2<0x000F000Fu>(w0, k.x, a.x);
  lo.y = magic2<0x000F000Fu>(v0, k.x, a.x);
  lo.z = magic2<0x000F000Fu>(w1, k.x, a.x);
  lo.w = magic2<0x000F000Fu>(v1, k.x, a.x);
  hi.x = magic2<0x00F000F0u>(w0, k.y, a.y);
  hi.y = magic2<0x00F000F0u>(v0, k.y, a.y);
  hi.z = magic2<0x00F000F0u>(w1, k.y, a.y);
  hi.w = magic2<0x00F000F0u>(v1, k.y, a.y);
  BPair b;
  b.lo = __builtin_bit_cast(f16x8, lo);
  b.hi = __builtin_bit_cast(f16x8, hi);
  return b;
}

// Q6_K: the B operands of MFMA steps m (quarter k = m / 2) and m + 4 (quarter
// k + 2), m = 2 k + u (k, u = 0, 1): bytes 8 u .. 8 u + 7 of the lane's 16 of
// each quarter.  A weight's integer is sc (q - 32), up to 4096 in magnitude
// with 13 significant bits, so two halves carry it exactly: its rounding to
// 11 bits and what that leaves (-1, 0 or 1).  q is put together in place: four
// bits of ql at bits 0-3 (4-7 for the high nibbles) and two of qh above
// them, so (0x6400 | q) - 1056 is q - 32 (and (0x6400 | 16 q) - 1536 is
// 16 (q - 32)) exactly; then one packed multiply and one packed fma for the
// rest.  Element order inside each 8 as for Q4_K.
template <bool HIGH>
__device__ __forceinline__ void q6_pair(uint32_t l, uint32_t h, _Float16 k1, uint32_t& v, uint32_t& r) {
  uint32_t t;
  if (HIGH) {
    asm("v_and_or_b32 %0, %1, %2, %3" : "=v"(t) : "v"(l), "s"(0x00F000F0u), "v"(0x64006400u));
    asm("v_and_or_b32 %0, %1, %2, %3" : "=v"(t) : "v"(h), "s"(0x03000300u), "v"(t));
  } else {
    asm("v_and_or_b32 %0, %1, %2, %3" : "=v"(t) : "v"(l), "s"(0x000F000Fu), "v"(0x64006400u));
    asm("v_and_or_b32 %0, %1, %2, %3" : "=v"(t) : "v"(h), "s"(0x00300030u), "v"(t));
  }
  const _Float16 off = HIGH ? (_Float16)-1536.0f : (_Float16)-1056.0f;
  const f16x2 e = __builtin_bit_cast(f16x2, t) + (f16x2){off, off};
  const f16x2 k = {k1, k1}, a = e * k;
  v = __builtin_bit_cast(uint32_t, a);
  r = __builtin_bit_cast(uint32_t, __builtin_elementwise_fma(e, k, -a));
}

// One nibble's operands: ql dwords w0, w1 and qh dwords h0, h1 of the 8 bytes.
// K = 0: quarters 0 (HIGH: 2), whose two qh bits lie at bits 0 (4) of a byte;
// K = 1: quarters 1 (3), at bits 2 (6).
struct BHalf6 {
  f16x8 v, r;
};
template <int K, bool HIGH>
__device__ __forceinline__ BHalf6 build_b6(uint32_t w0, uint32_t w1, uint32_t h0, uint32_t h1, _Float16 k) {
  u32x4 bv, br;
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    const uint32_t w = i ? w1 : w0, h = i ? h1 : h0;
    uint32_t v, r;
    q6_pair<HIGH>(w, K ? h << 2 : h << 4, k, v, r);
    bv[2 * i] = v, br[2 * i] = r;
    q6_pair<HIGH>(w >> 8, K ? h >> 6 : h >> 4, k, v, r);
    bv[2 * i + 1] = v, br[2 * i + 1] = r;
  }
  return BHalf6{__builtin_bit_cast(f16x8, bv), __builtin_bit_cast(f16x8, br)};
}

// Per-block constants of the lane's row: d and, for each quarter k, the
// lane's 16 weights' scale (its sixteenth for quarters 2 and 3, both in both
// halves).
struct QScale6 {
  float d;
  f16x2 k01, k23;
};

__device__ __forceinline__ QScale6 qscale6(const QLane<kDownQ6>& w, int s) {
  // the half's scales 2 k + s: bytes s and 2 + s of each dword, signed
  auto two = [s](uint32_t d) {
    const uint32_t b = ((d >> (8 * s)) & 0x00FF00FFu) ^ 0x64806480u;  // the halves 1152 + sc
    return __builtin_bit_cast(f16x2, b) + (f16x2){(_Float16)-1152.0f, (_Float16)-1152.0f};
  };
  const f16x2 a = two(w.sc.x), b = two(w.sc.y) * (f16x2){(_Float16)0.0625f, (_Float16)0.0625f};
  return QScale6{half_to_float(w.d), a, b};
}

// Per-block constants of the lane's row and group, halves for sub-blocks 2j
// (low) and 2j + 1 (high).
struct QScale {
  float d;
  f16x2 k;             // {sc, sc / 16}
  f16x2 a;             // {-1024 sc, -64 sc}
  float bc_lo, bc_hi;  // -dmin m
};

// The scale and min bits of a lane's two sub-blocks, taken from the header's
// twelve scale bytes two sub-blocks at a time: v_perm_b32 puts the two bytes
// that hold the low bits (and the two with the top bits of groups 2 and 3)
// into the two halves of a word.  Selectors and masks are constants of the
// lane's group g.
struct QSel {
  uint32_t lo, top;       // byte selectors
  uint32_t msk, mshift;   // low bits kept; shift of a min's low bits
  uint32_t tmsk;          // 0x00300030 where bits 4, 5 come from the top bytes
};
__device__ __forceinline__ QSel qsel(int g) {
  const uint32_t b = 2 * (uint32_t)(g & 1);
  QSel s;
  // v_perm_b32 (a, b): selector 0-3 the bytes of b, 4-7 those of a, 12 zero
  s.top = 0x0C000C00u | (b + 1) << 16 | b;
  s.lo = g < 2 ? s.top : s.top + 0x00040004u;
  s.msk = g < 2 ? 0x003F003Fu : 0x000F000Fu;
  s.mshift = g < 2 ? 0 : 4;
  s.tmsk = g < 2 ? 0 : 0x00300030u;
  return s;
}

__device__ __forceinline__ QScale qscale(const u32x4 hdr, const QSel& sel) {
  const uint32_t s0 = hdr.y, s1 = hdr.z, s2 = hdr.w;
  auto six = [&](uint32_t low, uint32_t top) {  // the halves 1024 + v
    const uint32_t t = __builtin_amdgcn_perm(0u, top, sel.top) >> 2;
    uint32_t v;
    asm("v_and_or_b32 %0, %1, %2, %3" : "=v"(v) : "v"(low), "v"(sel.msk), "v"(0x64006400u));
    asm("v_and_or_b32 %0, %1, %2, %3" : "=v"(v) : "v"(t), "v"(sel.tmsk), "v"(v));
    return __builtin_bit_cast(f16x2, v);
  };
  const f16x2 sc = six(__builtin_amdgcn_perm(s2, s0, sel.lo), s0);
  const f16x2 m = six(__builtin_amdgcn_perm(s2, s1, sel.lo) >> sel.mshift, s1) +
                  (f16x2){(_Float16)-1024.0f, (_Float16)-1024.0f};
  QScale s;
  s.d = half_to_float(hdr.x);
  s.k = __builtin_elementwise_fma(sc, (f16x2){(_Float16)1.0f, (_Float16)0.0625f},
                                  (f16x2){(_Float16)-1024.0f, (_Float16)-64.0f});
  s.a = s.k * (f16x2){(_Float16)-1024.0f, (_Float16)-1024.0f};
  const float dmin = half_to_float(hdr.x >> 16);
  s.bc_lo = fmaf(-dmin, (float)m.x, 0.0f);  // one v_fma_mix_f32 each
  s.bc_hi = fmaf(-dmin, (float)m.y, 0.0f);
  return s;
}

__device__ __forceinline__ f32x4 mfma_h(f16x8 a, f16x8 b, f32x4 c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_f16(a, b, c, 0, 0, 0);
}
__device__ __forceinline__ f32x4 mfma_f(float a, float b, f32x4 c) {
  return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
}

// Buffer accesses: a uniform 128-bit descriptor, a constant 32-bit offset per
// lane and a uniform one per block, so no address arithmetic runs on the
// vector ALU and no lane holds a 64-bit address.
typedef __amdgpu_buffer_rsrc_t rsrc_t;
__device__ __forceinline__ rsrc_t make_rsrc(const void* p, size_t bytes) {
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(p), 0, (int)bytes, 0x00020000);
}
constexpr int kCacheNt = 2;  // the nontemporal policy bit of a buffer access
template <int POLICY>
__device__ __forceinline__ u32x4 buf_load16(rsrc_t r, uint32_t lane_off, uint32_t off) {
  return __builtin_amdgcn_raw_buffer_load_b128(r, (int)lane_off, (int)off, POLICY);
}

// One 16-byte direct global -> LDS load per lane (lane i writes lds_dst + 16 i).
__device__ __forceinline__ void lds_dma16(rsrc_t r, uint32_t lane_off, uint32_t off, void* lds_dst) {
  __builtin_amdgcn_raw_ptr_buffer_load_lds(r, (__attribute__((address_space(3))) void*)lds_dst, 16, (int)lane_off,
                                           (int)off, 0, 0);
}

// LDS shared by the lanes of one wave: what they wrote before is there for the
// reads after.  The hardware runs a wave's LDS operations in order; this keeps
// the compiler, which sees one lane only, from moving them.
__device__ __forceinline__ void wave_lds_fence() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// waits until at most N of the wave's loads are in flight
template <int N>
__device__ __forceinline__ void wait_vm() {
  asm volatile("s_waitcnt vmcnt(%0)" ::"i"(N) : "memory");
}

}  // namespace

// ---- activation planes ---------------------------------------------------------------
// Rows of KD fp32 into the planes (planes_device.h).  One thread per
// 32-element sub-block holds it in registers: the row is read once, its
// largest |x| reduced across the row's threads, then converted.  KD = 2048:
// one wave per row, four rows per workgroup; KD = 7168: one workgroup per
// row (224 of its 256 threads hold a sub-block).
template <int P, int KD>
__device__ __forceinline__ void xplanes_rows(unsigned blk, const float* __restrict__ x, size_t n_rows,
                                             _Float16* __restrict__ xp, float* __restrict__ xs,
                                             float* __restrict__ xe) {
  constexpr int NSB = KD / 32;
  constexpr int TPR = NSB <= 64 ? 64 : 256;  // threads per row
  static_assert(NSB * 32 == KD && NSB <= TPR, "sub-blocks of a row fit its threads");
  constexpr int RPB = 256 / TPR;
  __shared__ float red[4];
  const size_t row = (size_t)blk * RPB + threadIdx.x / TPR;
  const int sb = threadIdx.x % TPR;
  const bool live = row < n_rows && sb < NSB;
  f32x4 v[8];
  float m = 0.0f;
  if (live) {
    const f32x4* src = reinterpret_cast<const f32x4*>(x + row * KD + 32 * sb);
#pragma unroll
    for (int i = 0; i < 8; ++i) v[i] = src[i];
    m = subblock_absmax(v);
  }
#pragma unroll
  for (int o = 32; o >= 1; o >>= 1) m = fmaxf(m, __shfl_xor(m, o));
  if constexpr (TPR == 256) {
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = m;
    __syncthreads();
    m = fmaxf(fmaxf(red[0], red[1]), fmaxf(red[2], red[3]));
  }
  if (!live) return;
  const int s = planes_shift(m);
  if (sb == 0) xe[row] = ldexpf(1.0f, -s);
  xs[row * NSB + sb] = planes_subblock<P>(v, s, xp + row * KD + 32 * sb, n_rows * KD);
}

// The rows of the gate/up activations, for the down.
template <int P>
__global__ __launch_bounds__(256) void k_xplanes(const float* __restrict__ x, size_t n_rows,
                                                 _Float16* __restrict__ xp, float* __restrict__ xs,
                                                 float* __restrict__ xe) {
  xplanes_rows<P, kFfn>(blockIdx.x, x, n_rows, xp, xs, xe);
}

// route() of T tokens (the first (T + 3) / 4 workgroups, one wave per token)
// and the three planes of their rows (one workgroup each).  Neither reads
// what the other writes and both are a chain of latencies, so one launch takes
// little more than the longer: 9.5 us against 8.7 + 5.0 at 5 tokens, 11.6
// against 9.8 + 5.2 at 16, 13.4 / 11.6 + 6.3 at 64, 15.6 / 11.5 + 9.8 at 256.
__global__ __launch_bounds__(256) void k_route_xplanes(const float* __restrict__ logits,
                                                       const float* __restrict__ bias, int T, int K,
                                                       int* __restrict__ idx, float* __restrict__ w,
                                                       const float* __restrict__ x, _Float16* __restrict__ xp,
                                                       float* __restrict__ xs, float* __restrict__ xe) {
  const unsigned n_route = (unsigned)(T + 3) / 4;
  if (blockIdx.x >= n_route) {
    xplanes_rows<3, kHidden>(blockIdx.x - n_route, x, (size_t)T, xp, xs, xe);
    return;
  }
  const int t = blockIdx.x * 4 + (threadIdx.x >> 6);
  if (t >= T) return;
  route_wave(logits + (size_t)t * 256, bias, K, 2.5f, idx + (size_t)t * K, w + (size_t)t * K);
}

// ---- the grouped GEMM ------------------------------------------------------------------
// One chunk (n tokens) of one expert, one row group.  The token operand has
// 16 NB rows in LDS, row r plane r / n of token r % n, so the three planes
// of up to 5 (NB = 1) or 10 (NB = 2) tokens share the 16-row operands that
// padding would otherwise fill.  Every row is summed by itself, in the same
// steps whatever NB and r are, and a token's planes are added up once after
// the last block: a token's bits do not depend on the others of its chunk.
// NT: the expert has one chunk, its weights are read once and streamed past
// the L2.
template <int P, int NB, QMat M, bool NT>
__device__ __forceinline__ void qgemm_body(const QGemmArgs& g, uint8_t* lds0, uint8_t* lds1, int* rows, const int4 ck,
                                           int rg) {
  constexpr int TL = kQTiles;
  constexpr bool DOWN = M != kGateUp, Q6 = M == kDownQ6;
  constexpr int KD = DOWN ? kFfn : kHidden;  // contraction length
  constexpr int NBLK = KD / kQK;             // 8 or 28 (even)
  constexpr int NT16 = 16 * NB;              // operand rows
  constexpr int NTOK = NT16 / P;
  constexpr int NBX = (NTOK + 15) / 16;      // 16-row blocks that hold plane 0 rows
  constexpr int ROUNDS = NT16 / (2 * kQWaves);  // direct loads per wave per block (2 rows each)
  static_assert(ROUNDS * 2 * kQWaves == NT16, "the direct loads tile the buffer");
  // the wave's number as a scalar: as a vector value it kept each LDS
  // destination of the direct loads in a register, and the Q6_K down spilled
  // 18, reloaded in the contraction behind waits for every load in flight
  // (a step of 64 tokens 785 -> 768 us, 150 prompt tokens 1086 -> 1070)
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int c16 = lane & 15, j = lane >> 4;
  const int n = ck.z;
  const bool shared = ck.x < 0;
  const int P0 = g.T * g.K;
  int* rin = rows;              // input row of chunk token t (activation plane row)
  int* rout = rows + kQMaxTok;  // output row
  if (threadIdx.x < n) {
    const int t = threadIdx.x;
    const int orow = shared ? P0 + ck.y + t : ck.y + t;
    rout[t] = orow;
    rin[t] = DOWN ? orow : (shared ? ck.y + t : g.pair_tok[ck.y + t]);
  }
  // weight addresses: a uniform base per block and constant lane offsets
  const uint8_t* blob = shared ? g.shared : g.experts + (size_t)ck.x * g.expert_size;
  const uint8_t* mat = blob + (DOWN ? 2 * (size_t)kGateBytes : 0);
  constexpr int ROWS = qgemm_rows(DOWN);
  // gate/up: column c16 of tile t is row 2 (4 t + c16 / 4) + c16 % 2 of the
  // wave's 16, of gate for c16 % 4 < 2, else of up.  Tile t's rows lie t
  // kTileRows further and its bytes t kTileStep: a scalar offset, so that a lane
  // keeps the addresses of tile 0 only.
  constexpr int kTileRows = DOWN ? 16 : 8;
  constexpr uint32_t kTileStep = Q6 ? kRel6Step : kRelStep * (DOWN ? 4 : 4 * (kHidden / 1024));
  const int row0 = DOWN ? rg * ROWS + 16 * TL * wave + c16
                        : rg * ROWS + 8 * TL * wave + 2 * (c16 >> 2) + (c16 & 1);
  uint32_t qoff, hoff, soff = 0;
  if constexpr (Q6) {
    const uint32_t base = (uint32_t)rel6_step_off(row0, 0), bi = (uint32_t)rel6_block_index(row0, 0);
    qoff = base + 16 * (2 * bi + (j >> 1)) + 2048 * (j & 1);
    soff = base + 16 * bi + 8 * (j >> 1);
    hoff = base + 2 * bi;
  } else {
    const uint32_t base = (uint32_t)rel_step_off<DOWN>(row0, 0), ri = c16 & 3;
    qoff = base + 16 * (uint32_t)rel_piece((int)ri, 0, j);
    hoff = base + kRelHdr + 16 * ri;
  }
  const rsrc_t wr = make_rsrc(mat, M == kGateUp ? 2 * (size_t)kGateBytes : Q6 ? kDownQ6KBytes : kDownQ4KBytes);
  constexpr int NLOADS = (Q6 ? 5 : 3) * TL;  // weight loads per block
  constexpr int kNt = NT ? kCacheNt : 0;
  // header of block b, then its quants in the two parts in which a block's
  // contraction uses them up
  auto load_hdr = [&](QLane<M> (&w)[TL], int b) {
#pragma unroll
    for (int t = 0; t < TL; ++t) {
      if constexpr (Q6) {
        const uint32_t st = (uint32_t)rel6_step_off(0, b) + kTileStep * t, bi = (uint32_t)rel6_block_index(0, b);
        w[t].sc = __builtin_bit_cast(
            u32x2, __builtin_amdgcn_raw_buffer_load_b64(wr, (int)soff, (int)(st + kRel6Sc + 16 * bi), 0));
        w[t].d = __builtin_amdgcn_raw_buffer_load_b16(wr, (int)hoff, (int)(st + kRel6D + 2 * bi), 0);
      } else {
        w[t].hdr = buf_load16<0>(wr, hoff, (uint32_t)rel_step_off<DOWN>(0, b) + 64 * (uint32_t)(b & 3) + kTileStep * t);
      }
    }
  };
  auto load_q = [&](QLane<M> (&w)[TL], int b, int part) {
    const uint32_t st = Q6 ? (uint32_t)rel6_step_off(0, b) + 32 * (uint32_t)rel6_block_index(0, b) + 4096 * part
                           : (uint32_t)rel_step_off<DOWN>(0, b) + 256 * (uint32_t)(b & 3) + kRelQ1 * part;
#pragma unroll
    for (int t = 0; t < TL; ++t) {
      (part ? w[t].q1 : w[t].q0) = buf_load16<kNt>(wr, qoff, st + kTileStep * t);
      if constexpr (Q6) {
        if (part) w[t].qh = buf_load16<kNt>(wr, qoff, st + kTileStep * t - 4096 + kRel6Qh);
      }
    }
  };
  QLane<M> wa[TL], wb[TL];
  load_hdr(wa, 0);
  load_q(wa, 0, 0);
  load_q(wa, 0, 1);
  __syncthreads();  // rin, rout
  // operand row r -> (plane, token); token < 0: a pad row
  auto row_token = [&](int r, int& plane) {
    plane = P == 1 ? 0 : (r >= n) + (r >= 2 * n);
    const int t = r - plane * n;
    return t < n ? t : -1;
  };
  // direct-load sources: round k of wave w fills LDS rows 2 (w + 4 k), +1 of
  // the buffer; lane i: row 2 (w + 4 k) + i / 32,
  // slot i % 32 holds piece (i % 32) ^ (r & 7) of that row's block.  The
  // token operand's 16-byte reads (lane (c16, j): row c16, piece
  // (8 j + m) ^ (c16 & 7)) are then free of bank conflicts; an XOR with all
  // four bits of c16 measured twice the cycles per read (2-way conflicts).
  const rsrc_t pr = make_rsrc(g.xp, 2 * P * g.plane);
  uint32_t src[ROUNDS];
#pragma unroll
  for (int k = 0; k < ROUNDS; ++k) {
    const int r = 2 * (wave + kQWaves * k) + (lane >> 5);
    int plane;
    const int t = row_token(r, plane);
    uint32_t piece = (uint32_t)((lane & 31) ^ (r & 7));
    // the Q6_K lane's step m = 2 k + u takes elements 128 h + 32 k + 16 s + 8 u:
    // kept at piece 8 j + m of the row too
    if (Q6) piece = 16 * (piece >> 4) + 2 * (piece >> 3 & 1) + 4 * (piece >> 1 & 3) + (piece & 1);
    // byte offset; past the buffer's end (no access, zeros) for a pad row
    src[k] = t < 0 ? 0x80000000u : 2u * ((uint32_t)plane * (uint32_t)g.plane + (uint32_t)(rin[t] * KD) + 8u * piece);
  }
  auto dma = [&](int b, int buf) {
    uint8_t* base = buf ? lds1 : lds0;
#pragma unroll
    for (int k = 0; k < ROUNDS; ++k) lds_dma16(pr, src[k], (uint32_t)b * (2 * kQK), base + 2 * (wave + kQWaves * k) * kQRowB);
  };
  [[maybe_unused]] const QSel sel = qsel(j);
  // corr operand A: plane 0 row c16 of block nb, sub-blocks 2j and 2j+1 of
  // block b; past the buffer's end (zeros) for a row of another plane or a pad
  const rsrc_t xr = make_rsrc(g.xs, g.plane / 32 * sizeof(float));
  uint32_t xoff[NBX];
#pragma unroll
  for (int nb = 0; nb < NBX; ++nb) {
    const int t = 16 * nb + c16;
    xoff[nb] = t < n ? 4u * (uint32_t)(rin[t] * (KD / 32) + 2 * j) : 0x80000000u;
  }
  auto load_xs = [&](u32x2 (&v)[NBX], int b) {
    if (Q6) return;  // no min term
#pragma unroll
    for (int nb = 0; nb < NBX; ++nb)
      v[nb] = __builtin_bit_cast(u32x2, __builtin_amdgcn_raw_buffer_load_b64(xr, (int)xoff[nb], 32 * b, 0));
  };
  f32x4 acc[TL][NB];
#pragma unroll
  for (int tt = 0; tt < TL; ++tt)
#pragma unroll
    for (int nb = 0; nb < NB; ++nb) acc[tt][nb] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};

  // One block: the token operands of an MFMA step are read from LDS once and
  // serve every tile, whose B operands are built per step.  With refill, each
  // weight register is loaded with block b + 2 right after its last use: the
  // weight stream runs one to two blocks ahead on two register sets.
  auto block = [&](int buf, QLane<M> (&w)[TL], const u32x2 (&xsv)[NBX], bool refill, int b) {
    const uint8_t* base = buf ? lds1 : lds0;
    // the token operand's row c16, piece 8 j + step at step 0
    uint32_t lane_op = (uint32_t)(c16 * kQRowB + 16 * ((8 * j) ^ (c16 & 7)));
    // the steps' addresses are made from this one in every block: kept, they
    // and the 48 accumulators do not fit 168 registers
    if (P == 3 && NB == 3) asm volatile("" : "+v"(lane_op));
    std::conditional_t<Q6, QScale6, QScale> sc[TL];
#pragma unroll
    for (int t = 0; t < TL; ++t) {
      // every constant is in a register of its own here: the header's are free
      if constexpr (Q6) {
        sc[t] = qscale6(w[t], j & 1);
        asm volatile("" : "+v"(sc[t].d), "+v"(sc[t].k01), "+v"(sc[t].k23));
      } else {
        sc[t] = qscale(w[t].hdr, sel);
        asm volatile("" : "+v"(sc[t].d), "+v"(sc[t].k), "+v"(sc[t].a), "+v"(sc[t].bc_lo), "+v"(sc[t].bc_hi));
      }
    }
    __builtin_amdgcn_sched_barrier(0);
    if (refill) load_hdr(w, b + 2);
    __builtin_amdgcn_sched_barrier(0);
    // Three planes: d C and the min term, which cancels most of its mean, are
    // put together before the running sum, which then holds the result's own
    // partial sums and rounds once per block (6.0e-7 -> 4.2e-7 of 64 bits for
    // 16 .. 256 tokens; 2.9e-7 with the planes' sums in 64 bits and each plane
    // summed by itself; dot4 4.5e-7), at four additions per tile.  Rows without
    // a min term (planes 1 and 2) take the same two steps wherever they lie.
    // One plane: the activations' 11 bits set the error (3.4e-4 either way), and
    // the registers and additions of up to four token blocks cost 5%.
    constexpr bool MIN_FIRST = P == 3 && !Q6;
    auto min_term = [&](int t, int nb, f32x4 a) {
      if constexpr (!Q6) {
        a = mfma_f(__uint_as_float(xsv[nb].x), sc[t].bc_lo, a);
        a = mfma_f(__uint_as_float(xsv[nb].y), sc[t].bc_hi, a);
      }
      return a;
    };
    [[maybe_unused]] f32x4 X[TL][NBX];
    if constexpr (MIN_FIRST) {
#pragma unroll
      for (int t = 0; t < TL; ++t)
#pragma unroll
        for (int nb = 0; nb < NBX; ++nb) X[t][nb] = min_term(t, nb, f32x4{0.0f, 0.0f, 0.0f, 0.0f});
    }
    f32x4 C[TL][NB];
#pragma unroll
    for (int t = 0; t < TL; ++t)
#pragma unroll
      for (int nb = 0; nb < NB; ++nb) C[t][nb] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
    for (int m = 0; m < 4; ++m) {
      const int i0 = 2 * (m & 1);
      auto operand = [&](int nb, int step) {
        return *reinterpret_cast<const f16x8*>(base + 16 * nb * kQRowB + (lane_op ^ (16 * step)));
      };
      if constexpr (Q6) {
        // one nibble of both tiles at a time: the operands are 16 registers
        auto nibble = [&](auto high) {
          constexpr bool HIGH = decltype(high)::value;
          BHalf6 B[TL];
#pragma unroll
          for (int t = 0; t < TL; ++t) {
            const u32x4& q = m < 2 ? w[t].q0 : w[t].q1;
            const f16x2 k = HIGH ? sc[t].k23 : sc[t].k01;
            B[t] = m < 2 ? build_b6<0, HIGH>(q[i0], q[i0 + 1], w[t].qh[i0], w[t].qh[i0 + 1], k.x)
                         : build_b6<1, HIGH>(q[i0], q[i0 + 1], w[t].qh[i0], w[t].qh[i0 + 1], k.y);
          }
#pragma unroll
          for (int nb = 0; nb < NB; ++nb) {
            const f16x8 a = operand(nb, HIGH ? m + 4 : m);
#pragma unroll
            for (int t = 0; t < TL; ++t) C[t][nb] = mfma_h(a, B[t].r, C[t][nb]);
#pragma unroll
            for (int t = 0; t < TL; ++t) C[t][nb] = mfma_h(a, B[t].v, C[t][nb]);
          }
          __builtin_amdgcn_sched_barrier(0);
        };
        nibble(std::false_type{});
        nibble(std::true_type{});
      } else {
        BPair B[TL];
#pragma unroll
        for (int t = 0; t < TL; ++t) {
          const u32x4& q = m < 2 ? w[t].q0 : w[t].q1;
          B[t] = build_b(q[i0], q[i0 + 1], sc[t].k, sc[t].a);
        }
#pragma unroll
        for (int nb = 0; nb < NB; ++nb) {
          const f16x8 a = operand(nb, m);
#pragma unroll
          for (int t = 0; t < TL; ++t) C[t][nb] = mfma_h(a, B[t].lo, C[t][nb]);
        }
#pragma unroll
        for (int nb = 0; nb < NB; ++nb) {
          const f16x8 a = operand(nb, m + 4);
#pragma unroll
          for (int t = 0; t < TL; ++t) C[t][nb] = mfma_h(a, B[t].hi, C[t][nb]);
        }
      }
      if (refill && (m & 1)) {
        __builtin_amdgcn_sched_barrier(0);
        load_q(w, b + 2, m >> 1);
        __builtin_amdgcn_sched_barrier(0);
      }
    }
#pragma unroll
    for (int t = 0; t < TL; ++t)
#pragma unroll
      for (int nb = 0; nb < NB; ++nb) {
        f32x4& a = acc[t][nb];
        if (MIN_FIRST) {
#pragma clang fp contract(off)
#pragma unroll
          for (int i = 0; i < 4; ++i)
            a[i] += nb < NBX ? fmaf(sc[t].d, C[t][nb][i], X[t][nb][i]) : sc[t].d * C[t][nb][i];
        } else {
#pragma unroll
          for (int i = 0; i < 4; ++i) a[i] = fmaf(sc[t].d, C[t][nb][i], a[i]);
          if constexpr (!Q6) {
            if (nb < NBX) a = min_term(t, nb, a);
          }
        }
      }
  };

  dma(0, 0);
  u32x2 xa[NBX], xb[NBX];
  load_xs(xa, 0);
  __builtin_amdgcn_sched_barrier(0);
  load_hdr(wb, 1);
  load_q(wb, 1, 0);
  load_q(wb, 1, 1);
  __builtin_amdgcn_sched_barrier(0);
  // Block b from buffer b & 1 while block b + 1 lands in the other one.  The
  // wait before a block leaves the NLOADS youngest loads in flight (the weights
  // of block b + 1): the loads before them, block b's weights, operands and
  // sub-block sums, have then landed.  That holds only in this order of issue,
  // which the scheduling barriers keep, here and around every refill: a
  // compiler free to move a weight load ahead of a direct load (its max-ilp
  // strategy does) would let a wave past the wait with its part of the buffer
  // still in flight, and the others read the block before.
  auto pair = [&](int b, bool last) {
    wait_vm<NLOADS>();
    __syncthreads();  // block b staged by every wave; buffer 1 read by all (block b - 1)
    dma(b + 1, 1);
    load_xs(xb, b + 1);
    __builtin_amdgcn_sched_barrier(0);
    block(0, wa, xa, !last, b);
    if (last)
      wait_vm<0>();
    else
      wait_vm<NLOADS>();
    __syncthreads();  // block b + 1 staged; buffer 0 read by all (block b)
    if (!last) {
      dma(b + 2, 0);
      load_xs(xa, b + 2);
    }
    __builtin_amdgcn_sched_barrier(0);
    block(1, wb, xb, !last, b + 1);
  };
#pragma nounroll
  for (int b = 0; b < NBLK - 2; b += 2) pair(b, false);
  pair(NBLK - 2, true);
  // D of a 16x16 MFMA: lane (c16, j) holds row (column) c16 of the tile and
  // operand rows 4 j .. 4 j + 3 of the 16-row block
  auto put = [&](int t, int tile, float gate, float up) {
    const float e = g.xe[rin[t]];
    if (DOWN)
      g.out[(size_t)rout[t] * kHidden + row0 + kTileRows * tile] = gate * e;
    else
      g.out[(size_t)rout[t] * kFfn + row0 + kTileRows * tile] = silu_mul(gate * e, up * e);
  };
  // gate/up: the up value of a gate lane's row lies two lanes on
  const bool writer = DOWN || (c16 & 2) == 0;
  auto up_of = [](float v) {
    return DOWN ? 0.0f : __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0xEE, 0xF, 0xF, false));
  };
  if constexpr (P == 1) {
#pragma unroll
    for (int nb = 0; nb < NB; ++nb) {
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int t = 16 * nb + 4 * j + i;
        float up[TL];
#pragma unroll
        for (int tt = 0; tt < TL; ++tt) up[tt] = up_of(acc[tt][nb][i]);
        if (t >= n || !writer) continue;
#pragma unroll
        for (int tt = 0; tt < TL; ++tt) put(t, tt, acc[tt][nb][i], up[tt]);
      }
    }
  } else {
    // the three planes of a token lie in other lanes' rows: through a
    // wave-private piece of buffer 0 (no longer read or written: the last
    // block is in buffer 1), tile by tile
    float* red = reinterpret_cast<float*>(lds0) + wave * NT16 * 16;
#pragma unroll
    for (int tt = 0; tt < TL; ++tt) {
#pragma unroll
      for (int nb = 0; nb < NB; ++nb)
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const int r = 16 * nb + 4 * j + i;
          red[r * 16 + c16] = acc[tt][nb][i];
        }
      wave_lds_fence();  // the values of other lanes are read below
      auto sum = [&](const float* p) { return (p[2 * n * 16] + p[n * 16]) + p[0]; };
      if (writer) {
        for (int t = j; t < n; t += 4) {
          const float* p = red + t * 16 + c16;
          put(t, tt, sum(p), DOWN ? 0.0f : sum(p + 2));
        }
      }
      wave_lds_fence();  // the next tile's values overwrite these
    }
  }
}

// NB: the largest token block count of a chunk (1 for the 16-token chunks
// of batched decode, 4 for the 64-token chunks of prefill); a chunk runs the
// body of the fewest 16-row operand blocks that hold its tokens (three planes:
// 3 n rows), so its weight operands are built once for up to 64 tokens and no
// MFMA runs on an empty block.  (From 11 tokens on three planes fill three
// blocks however they lie, and letting a token's planes share one accumulator
// there needs a third of the registers: a step of 256 tokens 1299 against 1322
// us.  But then a token's bits, and its error, 4.4e-7 against 3.8e-7 of 64
// bits, depend on how many others chose its expert.)
// One-dimensional grid: workgroups are handed to the eight XCDs in turn
// (id % 8), so id -> (xcd = id % 8, k = id / 8).  The items of an expert whose
// chunks are f .. f + c - 1 are ordered row group by row group, its chunks
// back to back, so its weights are read from HBM once per row group and
// served from that XCD's L2 to its other chunks.
// Three planes of Q4_K rows: the items of all experts in one row, cut into eight equal
// ranges, one per XCD.  An expert's token planes (up to 690 KB of 16 tokens)
// are then read by one XCD or two instead of all eight (gate/up of 256 tokens
// fetches 3.85 GB instead of 4.44; 16 / 64 / 256 tokens 221 -> 210, 474 -> 457,
// 873 -> 853 us; the down 121 -> 110 and 458 -> 438 us for 16 and 256).
// One plane, and the Q6_K down: XCD x has row groups x, x + 8, .. of every
// chunk.  Chunks of up to 64 tokens differ fourfold in cost, and equal ranges
// of them left XCDs idle at the end (512 tokens: 829 -> 860 us); the Q6_K down
// reads more weights per token plane (384 -> 387 us, 1080 -> 1090 at 512).
template <int P, int NB, QMat M, bool NT>
__device__ __forceinline__ void qgemm_chunk(const QGemmArgs& g, uint8_t* lds0, uint8_t* lds1, int* rows, const int4 ck,
                                            int rg) {
  const int n = ck.z;
  if constexpr (P == 3) {
    if (n <= 5) return qgemm_body<3, 1, M, NT>(g, lds0, lds1, rows, ck, rg);
    if (n <= 10) return qgemm_body<3, 2, M, NT>(g, lds0, lds1, rows, ck, rg);
    return qgemm_body<3, 3, M, NT>(g, lds0, lds1, rows, ck, rg);
  } else {
    if constexpr (NB == 4) {
      if (n > 48) return qgemm_body<P, 4, M, NT>(g, lds0, lds1, rows, ck, rg);
      if (n > 32) return qgemm_body<P, 3, M, NT>(g, lds0, lds1, rows, ck, rg);
    }
    if constexpr (NB >= 2) {
      if (n > 16) return qgemm_body<P, 2, M, NT>(g, lds0, lds1, rows, ck, rg);
    }
    return qgemm_body<P, 1, M, NT>(g, lds0, lds1, rows, ck, rg);
  }
}

template <int P, int NB, QMat M>
__global__ __launch_bounds__(kQWaves * 64) __attribute__((amdgpu_waves_per_eu(qgemm_waves(P)))) void k_qgemm(QGemmArgs g) {
  constexpr bool DOWN = M != kGateUp;
  constexpr int RG = (DOWN ? kHidden : kFfn) / qgemm_rows(DOWN);
  constexpr int Q = RG / 8;
  static_assert(Q * 8 == RG, "row groups split evenly over the XCDs");
  const int id = blockIdx.x, xcd = id & 7, k = id >> 3, n_chunks = *g.n_chunks;
  int chunk, rg, c;
  if constexpr (P == 3 && M != kDownQ6) {
    const int items = n_chunks * RG, per = (items + 7) >> 3, item = xcd * per + k;
    if (k >= per || item >= items) return;
    const int grp = g.chunks[item / RG].w, f = grp & 0xFFFF, off = item - RG * f;
    c = grp >> 16;
    chunk = f + off % c, rg = off / c;
  } else {
    const int m = k / Q;  // a chunk of the item's expert
    if (m >= n_chunks) return;
    const int grp = g.chunks[m].w, f = grp & 0xFFFF, off = k - Q * f;
    c = grp >> 16;
    chunk = f + off % c, rg = 8 * (off / c) + xcd;
  }
  // two arrays, not one: the compiler then sees that the direct loads into
  // one buffer cannot alias the reads of the other, and does not wait for
  // them (with all outstanding loads) before the contraction
  __shared__ __attribute__((aligned(16))) uint8_t lds0[P * 16 * NB * kQRowB];
  __shared__ __attribute__((aligned(16))) uint8_t lds1[P * 16 * NB * kQRowB];
  __shared__ int rows[2 * kQMaxTok];
  const int4 ck = g.chunks[chunk];
  if (c == 1)
    qgemm_chunk<P, NB, M, true>(g, lds0, lds1, rows, ck, rg);
  else
    qgemm_chunk<P, NB, M, false>(g, lds0, lds1, rows, ck, rg);
}

hipError_t launch_xplanes(const float* x, size_t n_rows, int planes, _Float16* xp, float* xs, float* xe,
                          hipStream_t s) {
  const dim3 grid((unsigned)((n_rows + 3) / 4)), blk(256);
  if (planes == 3)
    hipLaunchKernelGGL(k_xplanes<3>, grid, blk, 0, s, x, n_rows, xp, xs, xe);
  else
    hipLaunchKernelGGL(k_xplanes<1>, grid, blk, 0, s, x, n_rows, xp, xs, xe);
  return hipGetLastError();
}

hipError_t launch_route_xplanes(const float* logits, const float* bias, int T, int K, int* idx, float* w,
                                const float* x, _Float16* xp, float* xs, float* xe, hipStream_t s) {
  hipLaunchKernelGGL(k_route_xplanes, dim3((unsigned)((T + 3) / 4 + T)), dim3(256), 0, s, logits, bias, T, K, idx, w,
                     x, xp, xs, xe);
  return hipGetLastError();
}

int qgemm_chunk_tokens(int planes) { return planes == 3 ? 16 : 64; }

hipError_t launch_qgemm(const QGemmArgs& g, int planes, bool down, bool q6, int max_chunks, hipStream_t s) {
  const dim3 blk(kQWaves * 64);
  const int RG = (down ? kHidden : kFfn) / qgemm_rows(down);
  const dim3 grid((unsigned)(RG * max_chunks));
  if (down && q6) {
    if (planes != 3) return hipErrorInvalidValue;
    hipLaunchKernelGGL((k_qgemm<3, 1, kDownQ6>), grid, blk, 0, s, g);
  } else if (planes == 3) {
    if (down)
      hipLaunchKernelGGL((k_qgemm<3, 1, kDownQ4>), grid, blk, 0, s, g);
    else
      hipLaunchKernelGGL((k_qgemm<3, 1, kGateUp>), grid, blk, 0, s, g);
  } else {
    if (down)
      hipLaunchKernelGGL((k_qgemm<1, 4, kDownQ4>), grid, blk, 0, s, g);
    else
      hipLaunchKernelGGL((k_qgemm<1, 4, kGateUp>), grid, blk, 0, s, g);
  }
  return hipGetLastError();
}

}  // namespace fdm
