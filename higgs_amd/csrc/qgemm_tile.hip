// qgemm_tile.hip -- quantized_matmul over many rows (M > 64) on gfx950 MFMA
// (QLinear::forward, crates/higgs-models/src/qwen3_next.rs:174-221).
//
// Exact products: a code q enters the matrix core as the bf16 number q, so
// every product x q is exact, and per 64-code group acc += s * C with
// C = sum x q in f32. The bias term sum_g b Sx_g, with the row sums Sx_g of
// x (ones against x: every column of that product is one row's own), is one
// more bf16 MFMA per tile and 4 groups: Sx_g is split into three
// bf16 parts (24 bits: nothing is rounded), b is a bf16 number already, and
// the 16 k-slots of the MFMA take 4 groups x 3 such products.
//
// What sets the pace is instruction issue: an MFMA takes 8 cycles of a SIMD's
// vector issue and a VALU instruction 4, beside the matrix core's 16 cycles
// per 16 x 16 x 32 or 32 per 32 x 32 x 16. The f32 update is 4 (16) FMAs per
// 2 (4) MFMAs, so the 32 x 32 form issues half the MFMAs for the same work
// (256 x 256 tiles at M 4096, N 12288, K 2048: 222 -> 211 us), and the FMAs
// of one tile run beside the MFMAs of the next. The two-plane kernel this
// replaced (weights as hi + lo bf16: twice the MFMAs, no update) took 348 us,
// 593 TFLOP/s against 975; the exact 64-row kernel 197 us at 301 x 12288 x
// 4096 and 357 at 301 x 4096 x 12288, now 58 and 82.
//
// A block is WK x WM x WN waves over BM = 32 MT WM rows and BN = 32 NT WN
// columns; with WK > 1 the waves of each k-part walk their own contiguous
// share of the groups and the parts meet in LDS at the end.
//
// Memory: x, codes, scales and biases go straight from global memory to LDS
// (buffer loads with the lds bit: no staging registers), a ring of three
// 64-code stages, and a block meets at one barrier per group. With PRE a stage
// has landed one group before it is computed, so its codes and first row tile
// are read before the barrier (large tiles: a group lasts longer than a load);
// without, two groups of loads are in flight. The DMA writes lanes to
// consecutive addresses, so the order of a row's 16-byte pieces in LDS
// (tg_swizzle) is chosen by which piece a lane reads.
//
// The loads are inline assembly: they have no output register, and the waits
// are counted by hand (a stage is P loads, plus E for the scales and biases
// of 4 groups in every fourth stage), because the compiler would wait for
// every load in flight before any LDS read.
#include "../../include/higgs_hip.h"
#include "hgk_common.h"
#include "hgk_host.h"
#include "qgemm.h"

namespace hgk {

namespace {

typedef __bf16 bf16x8_t __attribute__((ext_vector_type(8)));
typedef float f32x4_t __attribute__((ext_vector_type(4)));
typedef float f32x16_t __attribute__((ext_vector_type(16)));
typedef __bf16 bf16x2_t __attribute__((ext_vector_type(2)));
typedef uint32_t u32x2_t __attribute__((ext_vector_type(2)));

constexpr int kTgRing = 3;

__device__ inline __amdgpu_buffer_rsrc_t tg_rsrc(const void* p, uint32_t bytes) {
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(p), (short)0, (int)bytes, 0x00020000);
}

__device__ inline uint32_t lds_addr(const void* p) {
  return (uint32_t)(uintptr_t)(__attribute__((address_space(3))) const void*)p;
}

// 16 (or 4) bytes per lane from rsrc + voff + soff to LDS at dst + 16 (4) * lane.
// dst and soff are wave-uniform. m0 is a register that the compiler reserves: it never holds a
// value of its own there for long, but may move or merge its writes to it, so it has to know of
// this one (and need not warn that nothing preserves it).
#pragma clang diagnostic push
#pragma clang diagnostic ignored "-Winline-asm"
__device__ inline void dma16(uint32_t dst, __amdgpu_buffer_rsrc_t r, uint32_t voff, uint32_t soff) {
  asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tbuffer_load_dwordx4 %1, %2, %3 offen lds"
               :: "s"(dst), "v"(voff), "s"(r), "s"(soff) : "m0", "memory");
}
__device__ inline void dma4(uint32_t dst, __amdgpu_buffer_rsrc_t r, uint32_t voff, uint32_t soff) {
  asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tbuffer_load_dword %1, %2, %3 offen lds"
               :: "s"(dst), "v"(voff), "s"(r), "s"(soff) : "m0", "memory");
}

#pragma clang diagnostic pop

// all but the newest N loads of this wave have landed, then the block's barrier
template <int N>
__device__ inline void wait_barrier() {
  asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" :: "n"(N) : "memory");
}

// 8 codes of one word (code i at bits 4i) -> their bf16 values in order. A
// byte 0 .. 15 read as fp8 (e4m3) is q * 2^-9 exactly (subnormals up to 7,
// the first binade from 8), so the scaled conversion gives q itself.
__device__ inline bf16x8_t tg_expand(uint32_t c) {
  const uint32_t lo = c & 0x0f0f0f0fu;         // q0 q2 q4 q6
  const uint32_t hi = (c >> 4) & 0x0f0f0f0fu;  // q1 q3 q5 q7
  const uint32_t p = __builtin_amdgcn_perm(hi, lo, 0x05010400u);  // q0 q1 q2 q3
  const uint32_t q = __builtin_amdgcn_perm(hi, lo, 0x07030602u);  // q4 q5 q6 q7
  u32x4 v;
  v[0] = __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(p, 512.0f, false));
  v[1] = __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(p, 512.0f, true));
  v[2] = __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(q, 512.0f, false));
  v[3] = __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(q, 512.0f, true));
  return __builtin_bit_cast(bf16x8_t, v);
}

// Where piece p of x row r sits among the row's 8: at p ^ tg_swizzle(r). Rows
// 0 .. 7 get 8 different values, and so do the even (odd) rows of 0 .. 15, so
// that neither 8 nor 16 consecutive lanes of a fragment read share a bank.
__device__ inline int tg_swizzle(int r) { return ((r >> 1) & 3) | (((r ^ (r >> 3)) & 1) << 2); }

// The Inf and NaN outputs of a wave's tile (rows m0 .., columns n0 ..; at most 64 columns), again
// in plain f32. The group form meets an Inf of x with the zero codes and with b Sx of the other
// sign, an Inf bias with the zero parts of Sx, and products x q may overflow where x w does not:
// NaN where the sum is Inf or finite. So an output of finite scales and biases is sum x (s q + b)
// in f32, as the GEMV has it, and one with others the sum of s C + b Sx per group. Rows that hold a
// NaN are NaN in every column already. The outputs are read past the L1, which a neighbour's read
// of the same line may have filled before this wave's stores.
__device__ inline void tg_redo(const QgemmArgs& a, int64_t m0, int rows, int64_t n0, int cols, int lane) {
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  const int64_t KW = a.K / 8, G = a.K / 64;
  for (int64_t m = m0; m < m0 + rows && m < a.M; ++m) {
    uint32_t v = 0;
    if (lane < cols && n0 + lane < a.N)
      v = __hip_atomic_load(a.y + m * a.ys + n0 + lane, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    uint64_t todo = __ballot((v & 0x7f80u) == 0x7f80u);
    if (!todo) continue;
    const uint16_t* xr = a.x + m * a.xs;
    bool nan = false;
    for (int64_t k = 8 * lane; k < a.K; k += 512) {
      const u32x4 q = *reinterpret_cast<const u32x4*>(xr + k);
#pragma unroll
      for (int i = 0; i < 4; ++i) nan |= (q[i] & 0x7fffu) > 0x7f80u || (q[i] & 0x7fff0000u) > 0x7f800000u;
    }
    if (__ballot(nan)) continue;
    for (; todo; todo &= todo - 1) {
      const int64_t n = n0 + __builtin_ctzll(todo);
      float each = 0.0f, grouped = 0.0f;
      bool finite = true;
      for (int64_t c = lane; c < KW; c += 64) {  // K a multiple of 512: the same count in every lane
        const uint32_t q = a.w[n * KW + c];
        const u32x4 xq = *reinterpret_cast<const u32x4*>(xr + 8 * c);
        const uint32_t su = a.sc[n * G + c / 8], bu = a.bi[n * G + c / 8];
        const float s = BF16::lo(su), b = BF16::lo(bu);
        finite &= (su & 0x7f80u) != 0x7f80u && (bu & 0x7f80u) != 0x7f80u;
        float cq = 0.0f, sx = 0.0f;
#pragma unroll
        for (int i = 0; i < 8; ++i) {
          const float x = i & 1 ? BF16::hi(xq[i / 2]) : BF16::lo(xq[i / 2]), qf = (float)((q >> (4 * i)) & 15u);
          each = __builtin_fmaf(x, __builtin_fmaf(s, qf, b), each);
          cq = __builtin_fmaf(x, qf, cq);
          sx += x;
        }
#pragma unroll
        for (int o = 1; o < 8; o <<= 1) {
          cq += __shfl_xor(cq, o, 64);
          sx += __shfl_xor(sx, o, 64);
        }
        grouped = __builtin_fmaf(s, cq, __builtin_fmaf(b, sx, grouped));
      }
      each = group_sum<64>(each);
#pragma unroll
      for (int o = 8; o < 64; o <<= 1) grouped += __shfl_xor(grouped, o, 64);
      const float r = __ballot(!finite) ? grouped : each;
      if (lane == 0) a.y[m * a.ys + n] = (uint16_t)(BF16::pack(r, 0.0f) & 0xffffu);
    }
  }
}

template <int WK, int WM, int WN, int MT, int NT, bool PRE>
struct TileCfg {
  static constexpr int TP = 64 * WM * WN;       // threads of a k-part
  static constexpr int T = TP * WK;
  static constexpr int BM = 32 * MT * WM, BN = 32 * NT * WN;
  static constexpr int XB = BM * 128, CB = BN * 32, SB = BN * 16;  // bytes of a stage's x, codes; scales + biases
  static constexpr int PX = BM * 8 / TP;
  static constexpr int PC = (BN * 2 + TP - 1) / TP;
  static constexpr int P = PX + PC, E = BN * 4 / TP;
  static constexpr int Q = MT > WN ? MT / WN : 1;  // row tiles whose row sums a wave forms
  static constexpr int PART = kTgRing * (XB + CB) + 2 * SB + 2 * 4 * BM * 4;
  static constexpr int LDS = WK * PART;
  static_assert(!PRE || MT % 2 == 0, "the next stage's first row tile goes where row tile 0's was");
  static_assert(BM * 8 % TP == 0 && BN * 4 % TP == 0 && BN % 32 == 0, "even split of a stage");
  static_assert(BN * 2 % TP == 0 || TP % (BN * 2) == 0, "even split of the codes");
  static_assert(MT % WN == 0 || WN % MT == 0, "row sums split over the column waves");
  // the k-parts' sums, and the output tiles of the waves, meet in the same memory
  static_assert((WK - 1) * WM * WN * MT * NT * 4096 <= LDS, "partial sums");
  static_assert(T / 64 * 32 * (NT * 64 + 16) <= LDS, "output staging");
};

template <int WK, int WM, int WN, int MT, int NT, bool PRE>
__global__ __launch_bounds__(64 * WK * WM * WN, 2) void qgemm_tile_kernel(QgemmArgs a, int mt, int nt) {
  using C = TileCfg<WK, WM, WN, MT, NT, PRE>;
  __shared__ __align__(16) unsigned char lds[C::LDS];

  // tile of this block: the blocks of one XCD (dealt in turn) take consecutive
  // tiles, 8 column tiles wide, so that they share x rows and weight columns in
  // its L2
  const int tiles = mt * nt, per = (tiles + 7) >> 3;
  const int lin = ((int)blockIdx.x & 7) * per + ((int)blockIdx.x >> 3);
  if (((int)blockIdx.x >> 3) >= per || lin >= tiles) return;  // whole block
  const int wide = lin / (8 * mt), rem = lin - wide * 8 * mt;
  const int gw = nt - wide * 8 < 8 ? nt - wide * 8 : 8;
  const int64_t m0 = (int64_t)(rem / gw) * C::BM, n0 = (int64_t)(wide * 8 + rem % gw) * C::BN;

  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wk = wave / (WM * WN), wv = wave % (WM * WN);
  const int wm = wv / WN, wn = wv % WN;
  const int tk = wv * 64 + lane;
  const int l32 = lane & 31, lh = lane >> 5;
  const int G = (int)(a.K / 64), GP = G / WK, g0 = wk * GP;
  const int mrem = a.M - m0 < C::BM ? (int)(a.M - m0) : C::BM;
  const int nrem = a.N - n0 < C::BN ? (int)(a.N - n0) : C::BN;

  unsigned char* const xs = lds + wk * C::PART;
  unsigned char* const cs = xs + kTgRing * C::XB;
  unsigned char* const ss = cs + kTgRing * C::CB;
  float* const sums = reinterpret_cast<float*>(ss + 2 * C::SB);

  const __amdgpu_buffer_rsrc_t rx = tg_rsrc(a.x + m0 * a.xs, (uint32_t)(((int64_t)(mrem - 1) * a.xs + a.K) * 2));
  const __amdgpu_buffer_rsrc_t rw = tg_rsrc(a.w + n0 * (a.K / 8), (uint32_t)((int64_t)nrem * a.K / 2));
  uint32_t xo[C::PX], co[C::PC], so[C::E];
#pragma unroll
  for (int p = 0; p < C::PX; ++p) {
    const int c = tk + C::TP * p, row = c >> 3;
    xo[p] = (uint32_t)((row < mrem ? row : mrem - 1) * a.xs * 2) + (uint32_t)(((c & 7) ^ tg_swizzle(row)) * 16);
  }
#pragma unroll
  for (int p = 0; p < C::PC; ++p) {
    const int c = (tk + C::TP * p) % (C::BN * 2), col = c >> 1;
    co[p] = (uint32_t)((col < nrem ? col : nrem - 1) * (a.K / 2)) + (uint32_t)(((c ^ (col >> 3)) & 1) * 16);
  }
  // scales and biases of 4 groups: 4 words per column (s01, s23, b01, b23), word-major
#pragma unroll
  for (int p = 0; p < C::E; ++p) {
    const int e = tk + C::TP * p, col = e % C::BN, word = e / C::BN;
    so[p] = (uint32_t)((col < nrem ? col : nrem - 1) * G * 2) + (uint32_t)((word & 1) * 4);
  }
  const uint32_t xl = lds_addr(xs) + wv * 1024, cl = lds_addr(cs), sl = lds_addr(ss) + wv * 256;

  auto issue = [&](int i, int slot) {
    const int g = g0 + i;
#pragma unroll
    for (int p = 0; p < C::PX; ++p) dma16(xl + slot * C::XB + p * C::TP * 16, rx, xo[p], (uint32_t)g * 128);
#pragma unroll
    for (int p = 0; p < C::PC; ++p)
      dma16(cl + slot * C::CB + ((wv * 64 + C::TP * p) % (C::BN * 2)) * 16, rw, co[p], (uint32_t)g * 32);
    if ((i & 3) == 0) {
#pragma unroll
      for (int p = 0; p < C::E; ++p) {
        const uint16_t* base = (wv * 64 + C::TP * p) / C::BN < 2 ? a.sc : a.bi;
        const __amdgpu_buffer_rsrc_t rs = tg_rsrc(base + n0 * G, (uint32_t)nrem * G * 2);
        dma4(sl + ((i >> 2) & 1) * C::SB + p * C::TP * 4, rs, so[p], (uint32_t)g * 2);
      }
    }
  };

  f32x16_t acc[MT][NT];
#pragma unroll
  for (int i = 0; i < MT; ++i)
#pragma unroll
    for (int t = 0; t < NT; ++t) acc[i][t] = f32x16_t{};

  // this lane's LDS reads: x pieces 4 lh + f of row l32, code words 4 lh .. 4 lh + 3 of column
  // l32 (f = 0 .. 3: the group's four MFMAs)
  const int arow = wm * 32 * MT + l32;
  int ao[4];
#pragma unroll
  for (int f = 0; f < 4; ++f) ao[f] = arow * 128 + ((4 * lh + f) ^ tg_swizzle(l32)) * 16;
  const int bo = (wn * 32 * NT + l32) * 32 + ((lh ^ (l32 >> 3)) & 1) * 16;
  const int sco = (wn * 32 * NT + l32) * 4;
  // the row sums' B operand of a 16 x 16 x 32 MFMA against ones: rows 0 .. 15 (16 .. 31) of a
  // row tile in its columns, pieces lg and lg + 4 of them in k-group lg = lane / 16. A column
  // holds one row of x only, so that an Inf or NaN stays in its own row's sum.
  const int ro = (wm * 32 * MT + (lane & 15)) * 128 + ((lane >> 4) ^ tg_swizzle(lane & 15)) * 16;
  const bf16x8_t ones = __builtin_bit_cast(bf16x8_t, u32x4{0x3f803f80u, 0x3f803f80u, 0x3f803f80u, 0x3f803f80u});

  u32x4 wr[NT];
  bf16x8_t av[2][4];
  uint32_t sr[NT];
  // a stage's codes, scales and first row tile
  auto preload = [&](int slot, int sbuf, int j) {
    const unsigned char* const xb = xs + slot * C::XB;
    const unsigned char* const cb = cs + slot * C::CB;
    const unsigned char* const sb = ss + sbuf * C::SB + (j >> 1) * (C::BN * 4) + sco;
#pragma unroll
    for (int t = 0; t < NT; ++t) wr[t] = *reinterpret_cast<const u32x4*>(cb + bo + t * 1024);
#pragma unroll
    for (int f = 0; f < 4; ++f) av[0][f] = *reinterpret_cast<const bf16x8_t*>(xb + ao[f]);
#pragma unroll
    for (int t = 0; t < NT; ++t) sr[t] = *reinterpret_cast<const uint32_t*>(sb + t * 128);
  };
  auto compute = [&](int slot, int sbuf, int j, int next) {
    const unsigned char* const xb = xs + slot * C::XB;
    bf16x8_t bw[NT][4];
    float s[NT];
    f32x16_t c[2];
    if constexpr (!PRE) preload(slot, sbuf, j);
#pragma unroll
    for (int t = 0; t < NT; ++t) s[t] = u2f((j & 1) ? (sr[t] & 0xffff0000u) : (sr[t] << 16));
#pragma unroll
    for (int f = 0; f < 4; ++f) bw[0][f] = tg_expand(wr[0][f]);
    // Tile k = (row tile k / NT, column tile k % NT): its four MFMAs run beside tile k - 1's
    // f32 update, the next column tile's code expansion and the next row tile's x reads. (The
    // empty asm holds each update in its place: otherwise every MFMA result of the group is
    // kept until the end.)
#pragma unroll
    for (int k = 0; k <= MT * NT; ++k) {
      const int i = k / NT, t = k % NT;
      if (k < MT * NT) {
        if (t == NT - 1 && i + 1 < MT) {
#pragma unroll
          for (int f = 0; f < 4; ++f) av[(i + 1) & 1][f] = *reinterpret_cast<const bf16x8_t*>(xb + ao[f] + (i + 1) * 4096);
        }
        if constexpr (PRE) {
          if (k == MT * NT - 1) preload(next, j == 3 ? sbuf ^ 1 : sbuf, (j + 1) & 3);
        }
        c[k & 1] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(av[i & 1][0], bw[t][0], f32x16_t{}, 0, 0, 0);
#pragma unroll
        for (int f = 1; f < 4; ++f)
          c[k & 1] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(av[i & 1][f], bw[t][f], c[k & 1], 0, 0, 0);
        if (i == 0 && t + 1 < NT) {
#pragma unroll
          for (int f = 0; f < 4; ++f) {
            bw[t + 1][f] = tg_expand(wr[t + 1][f]);
            asm volatile("" : "+v"(bw[t + 1][f]));
          }
        }
      }
      if (k > 0) {
        f32x16_t& u = acc[(k - 1) / NT][(k - 1) % NT];
#pragma unroll
        for (int r = 0; r < 16; ++r) u[r] = __builtin_fmaf(s[(k - 1) % NT], c[(k - 1) & 1][r], u[r]);
        asm volatile("" : "+v"(u));
      }
      if (k < MT * NT) {
        constexpr int PER = 4;
#pragma unroll
        for (int f = 0; f < 4; ++f) {
          __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
          __builtin_amdgcn_sched_group_barrier(0x002, PER, 0);
        }
      }
      if (k == (MT * NT > 2 ? 2 : 0)) {
        // row sums of this wave's Q row tiles
#pragma unroll
        for (int q = 0; q < C::Q; ++q) {
          const int rt = (wn * C::Q + q) % MT;
          f32x4_t sx[2] = {};
#pragma unroll
          for (int f = 0; f < 2; ++f)
#pragma unroll
            for (int h = 0; h < 2; ++h)
              sx[h] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
                  ones, *reinterpret_cast<const bf16x8_t*>(xb + (ro ^ (64 * f)) + h * 2048 + rt * 4096), sx[h], 0, 0, 0);
          // every row of a result is the same: lanes 0 .. 31 take the sum of row l32
          if (lh == 0) sums[(sbuf * 4 + j) * C::BM + wm * 32 * MT + rt * 32 + l32] = (lane & 16) ? sx[1][0] : sx[0][0];
        }
      }
      __builtin_amdgcn_sched_barrier(0);
    }
  };
  // acc += sum over the 4 groups of b Sx: lane half lh's k-slots are (h, m, l, 0) of Sx of
  // groups 2 lh and 2 lh + 1 against (b, b, b, 0)
  auto apply_bias = [&](int sbuf) {
    bf16x8_t bb[NT];
#pragma unroll
    for (int t = 0; t < NT; ++t) {
      const uint32_t v = *reinterpret_cast<const uint32_t*>(ss + sbuf * C::SB + (2 + lh) * (C::BN * 4) + sco + t * 128);
      const uint32_t b0 = v & 0xffffu, b1 = v >> 16;
      bb[t] = __builtin_bit_cast(bf16x8_t, u32x4{b0 | (b0 << 16), b0, b1 | (b1 << 16), b1});
    }
#pragma unroll
    for (int i = 0; i < MT; ++i) {
      u32x4 av;
#pragma unroll
      for (int h2 = 0; h2 < 2; ++h2) {
        const float v = sums[(sbuf * 4 + 2 * lh + h2) * C::BM + arow + i * 32];
        const float h = u2f(f2u(v) & 0xffff0000u), r = v - h;
        const float m = u2f(f2u(r) & 0xffff0000u), l = r - m;
        av[2 * h2] = __builtin_amdgcn_perm(f2u(m), f2u(h), 0x07060302u);
        av[2 * h2 + 1] = f2u(l) >> 16;
      }
#pragma unroll
      for (int t = 0; t < NT; ++t)
        acc[i][t] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8_t, av), bb[t], acc[i][t], 0, 0, 0);
#pragma unroll
      for (int t = 0; t < NT; ++t) asm volatile("" : "+v"(acc[i][t]));
      __builtin_amdgcn_sched_barrier(0);
    }
  };

  issue(0, 0);
  issue(1, 1);
  int slot = 0;
  for (int i0 = 0; i0 < GP; i0 += 4) {
    const int sbuf = (i0 >> 2) & 1;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const int i = i0 + j;
      // every wave is done with stage i - 1, and stage i (PRE: and i + 1) has landed for all
      if (PRE || i + 1 >= GP) wait_barrier<0>();
      else if (j == 3) wait_barrier<C::P + C::E>();
      else wait_barrier<C::P>();
      const int prev = slot == 0 ? kTgRing - 1 : slot - 1, next = slot == kTgRing - 1 ? 0 : slot + 1;
      if (i + 2 < GP) issue(i + 2, prev);
      if (PRE && i == 0) preload(0, 0, 0);
      if (j == 0 && i0 > 0) apply_bias(sbuf ^ 1);
      compute(slot, sbuf, j, next);
      slot = next;
    }
  }
  wait_barrier<0>();
  apply_bias(((GP >> 2) - 1) & 1);
  wait_barrier<0>();  // the stages' memory is free

  if constexpr (WK > 1) {
    // the k-parts' sums, added in part order
    float* red = reinterpret_cast<float*>(lds);
    if (wk > 0) {
#pragma unroll
      for (int i = 0; i < MT; ++i)
#pragma unroll
        for (int t = 0; t < NT; ++t)
#pragma unroll
          for (int r = 0; r < 16; ++r)
            red[((((wk - 1) * WM * WN + wv) * MT * NT + i * NT + t) * 16 + r) * 64 + lane] = acc[i][t][r];
    }
    wait_barrier<0>();
    if (wk == 0) {
#pragma unroll
      for (int k = 0; k < WK - 1; ++k)
#pragma unroll
        for (int i = 0; i < MT; ++i)
#pragma unroll
          for (int t = 0; t < NT; ++t)
#pragma unroll
            for (int r = 0; r < 16; ++r)
              acc[i][t][r] += red[(((k * WM * WN + wv) * MT * NT + i * NT + t) * 16 + r) * 64 + lane];
    }
    wait_barrier<0>();
    if (wk > 0) return;
  }

  // y: each 32-row tile through the wave's own LDS slice, so that the stores
  // are 16-byte pieces of whole rows. A lane holds, in register r, row
  // 8 (r / 4) + 4 lh + r % 4 of column l32.
  constexpr int PITCH = NT * 64 + 16, PCS = NT * 4;  // bytes and 16-byte pieces per row
  unsigned char* const ob = lds + wv * 32 * PITCH;
  const bool vec = (reinterpret_cast<uintptr_t>(a.y) & 15) == 0 && a.ys % 8 == 0;
  uint32_t bad = 0;  // bit 15 or 31: an Inf or NaN
#pragma unroll
  for (int i = 0; i < MT; ++i) {
#pragma unroll
    for (int t = 0; t < NT; ++t)
#pragma unroll
      for (int r = 0; r < 16; ++r)
        *reinterpret_cast<uint16_t*>(ob + (8 * (r >> 2) + 4 * lh + (r & 3)) * PITCH + (t * 32 + l32) * 2) =
            (uint16_t)(BF16::pack(acc[i][t][r], 0.0f) & 0xffffu);
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
#pragma unroll
    for (int q = 0; q < 32 * PCS / 64; ++q) {
      const int pc = lane + 64 * q, row = pc / PCS, cp = pc % PCS;
      const u32x4 v = *reinterpret_cast<const u32x4*>(ob + row * PITCH + cp * 16);
      const int64_t m = m0 + wm * 32 * MT + i * 32 + row, n = n0 + wn * 32 * NT + cp * 8;
      if (m < a.M) {
#pragma unroll
        for (int k = 0; k < 4; ++k) bad |= (v[k] & 0x7f807f80u) + 0x00800080u;
        uint16_t* const yp = a.y + m * a.ys + n;
        if (vec && n + 8 <= a.N) {
          *reinterpret_cast<u32x4*>(yp) = v;
        } else {
#pragma unroll
          for (int k = 0; k < 8; ++k)
            if (n + k < a.N) yp[k] = (uint16_t)(v[k >> 1] >> (16 * (k & 1)));
        }
      }
    }
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
  }
  if (__ballot(bad & 0x80008000u)) tg_redo(a, m0 + wm * 32 * MT, 32 * MT, n0 + wn * 32 * NT, 32 * NT, lane);
}

template <int WK, int WM, int WN, int MT, int NT, bool PRE>
void tile_launch(const QgemmArgs& a, hipStream_t s) {
  using C = TileCfg<WK, WM, WN, MT, NT, PRE>;
  const int mt = (int)((a.M + C::BM - 1) / C::BM), nt = (int)((a.N + C::BN - 1) / C::BN);
  const int per = (mt * nt + 7) / 8;
  HGK_LAUNCH((qgemm_tile_kernel<WK, WM, WN, MT, NT, PRE>), dim3((unsigned)per * 8), dim3(C::T), 0, s, a, mt, nt);
}

}  // namespace

bool qgemm_tile_fits(const QgemmArgs& a) {
  const int64_t lim = (int64_t)1 << 31;
  return a.K % 512 == 0 && (reinterpret_cast<uintptr_t>(a.w) & 15) == 0 &&
         ((reinterpret_cast<uintptr_t>(a.sc) | reinterpret_cast<uintptr_t>(a.bi)) & 3) == 0 &&
         256 * a.xs * 2 + a.K * 2 < lim && 256 * a.K / 2 < lim &&
         ((a.M + 63) / 64) * ((a.N + 63) / 64) < lim / 256;
}

// 33 to 64 rows over few columns: 32 x 32 tiles whose 8 waves split K, where
// they all run at once. The decode kernel gives a block 16 columns of all rows
// there, and a CU's x traffic and the chain over K set its time. us, decode
// kernel / these tiles (N x K): 64 rows 4096 x 12288 55.0 / 27.7, 2048 x 8192
// 36.5 / 17.3, 4096 x 4096 20.2 / 11.4, 2048 x 2048 10.8 / 7.2; 33 rows 37.9 /
// 26.3, 24.6 / 16.4, 14.3 / 11.0, 7.7 / 7.1. Up to 32 rows the decode kernel is
// as fast or faster (17 rows, 2048 x 2048: 6.0 / 7.0), and so it is with more
// columns where 96-column tiles fill one round of CUs (64 rows, 12288 x 4096:
// 22.6 / 31.8). Past that it is not (64 rows, 14336 x 3584: 39.3, 23.7 in this
// arithmetic): those calls stay on the decode kernel for want of a rule.
bool qgemm_tile_split_fits(const QgemmArgs& a) {
  return a.M > 32 && a.M <= 64 && a.K % 2048 == 0 && 2 * ((a.N + 31) / 32) <= 256 && qgemm_tile_fits(a);
}

void qgemm_tile_split_launch(const QgemmArgs& a, hipStream_t s) { tile_launch<8, 1, 1, 1, 1, false>(a, s); }

// The tile is chosen by the time the launch would take: rounds of resident
// blocks x groups x the measured time of one group (ns) with 1, 2 or 3 blocks
// on a CU (the last round may be partly filled). Measured from K = 2048 ..
// 12288 runs (M, N, K -> us per tile, in the order of the table):
//   4096 x 12288 x 2048   212  252  305  360  410
//   2048 x 4096 x 2048     64   46   59   64   75
//   640 x 14336 x 3584    101  109  113  126  132
//   301 x 12288 x 4096    112   70   58   63   68
//   301 x 4096 x 12288    319  147  117   82   91
//   1024 x 2048 x 2048     58   29   25   19   21
//   128 x 4096 x 4096     109   51   41   30   24
// Large tiles read x and the codes least often and win once they fill the
// chip; below that, more and smaller blocks, and two k-parts per block, do.
struct TileCost {
  int bm, bn, resident;
  int ns[3];
};
constexpr TileCost kTiles[] = {
    {256, 256, 1, {1900, 0, 0}},   {128, 128, 2, {800, 1310, 0}}, {64, 128, 3, {650, 900, 1190}},
    {64, 128, 1, {470, 0, 0}},     {64, 64, 2, {370, 530, 0}},
};

void qgemm_tile_launch(const QgemmArgs& a, hipStream_t s) {
  int best = 0;
  int64_t best_ns = 0;
  for (int i = 0; i < 5; ++i) {
    const TileCost& c = kTiles[i];
    const int64_t blocks = ((a.M + c.bm - 1) / c.bm) * ((a.N + c.bn - 1) / c.bn), full = 256 * c.resident;
    const int64_t rest = blocks % full;
    const int64_t ns = blocks / full * c.ns[c.resident - 1] + (rest ? c.ns[(rest - 1) / 256] : 0);
    if (i == 0 || ns < best_ns) {
      best = i;
      best_ns = ns;
    }
  }
  switch (best) {
    case 0: tile_launch<1, 2, 4, 4, 2, true>(a, s); break;
    case 1: tile_launch<1, 2, 2, 2, 2, true>(a, s); break;
    case 2: tile_launch<1, 2, 2, 1, 2, false>(a, s); break;
    case 3: tile_launch<2, 1, 4, 2, 1, false>(a, s); break;
    default: tile_launch<2, 2, 2, 1, 1, false>(a, s); break;
  }
}

}  // namespace hgk
