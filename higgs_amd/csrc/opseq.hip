// opseq.hip -- a decode step's per-layer op sequence in one launch.
//
// The reference runs each decoder layer as (qwen3_next.rs:1508-1547, for each
// of the 64 sequences of a continuous batch, batch_engine.rs:395-403):
//   normed = input_layernorm(h)                        -- add + RMSNorm
//   r = attention(normed)   gated RMSNorm (linear-attention layers) or
//                           q/k RMSNorm + partial RoPE (full-attention layers)
//   h2 = h + r; normed_post = post_attention_layernorm(h2)  -- add + RMSNorm
//   mlp_out = mlp(normed_post)                         -- SwiGLU of the experts
//   h = h2 + mlp_out
// Every one of those ops is row-wise: token t's outputs depend only on token
// t's inputs, and the residual stream of token t feeds only token t. So one
// workgroup per token walks the whole op list in order, with nothing but
// workgroup barriers between ops; no workgroup ever waits on another, so the
// grid needs no co-residency and no wait can hang.
//
// Most of those ops do not depend on each other: of the 192 ops of a 48-layer
// Qwen3-Next step, 96 form the residual chain and 96 read nothing that the
// list writes. Upload therefore sorts the ops into up to kChains chains (ops
// that share a buffer, one of them writing it, for the same token stay in one
// chain, in list order), and a token gets a workgroup per chain where there are
// few tokens, else fewer that walk several chains each. Within a
// chain an op waits for earlier stores (a wait on every outstanding memory
// operation, then the workgroup barrier) only where it touches what an op
// since the last wait wrote, and a run of residual adds + norms over the same
// rows carries h in registers, with the next residual and weight loaded
// beside the current sum. 64 tokens x 48 layers, every buffer in cache: 411 us
// with every op in one workgroup, waiting; 125 with chains (buffers that change
// between runs: 466 and 159). What the launch then measures is the list's own
// dependences: a model that fills the list's inputs from the list's outputs
// (attention, experts) cannot run the whole step in one launch.
// Every consumer of an op's output inside the launch is the same workgroup,
// so workgroup-scope ordering is all the data needs; other consumers see it
// after the launch. Buffers that only meet for some later token (views with
// different token strides) bound the token count up to which the chains hold
// (`safe`); a run over more tokens walks the whole list in one workgroup per
// token, waiting after every op.
//
// Each op's arithmetic is the standalone kernel's (norm.hip, rope.hip,
// glu.hip) for 16-bit activations and weights of the same type: results are
// the same bits as the separate calls.
//
// The op list is a device array written by hgk_op_list_upload into memory the
// caller owns; this file allocates nothing.
#include <algorithm>
#include <array>
#include <cmath>
#include <iterator>
#include <map>
#include <new>
#include <utility>
#include <vector>

#include "../../include/higgs_hip.h"
#include "hgk_act.h"
#include "hgk_common.h"
#include "hgk_host.h"

namespace hgk {

constexpr uint32_t kOpListMagic = 0x6f70736bu;  // "opsk"
constexpr int kOpMaxHalf = 256;                 // rotated dims / 2
constexpr int kOpThreads = 1024;
constexpr int kChains = 8;                      // chains per token

// One op as the kernel reads it (written by the host from an hgk_op).
struct alignas(16) DevOp {
  int32_t kind, act, rows, n;
  int32_t k_rows, dims, half, lpr;      // rope: k heads, rotated dims, dims / 2, lanes per row
  int32_t g, same_table;                // norms: lanes per row; rope: the cos/sin table of the
                                        // previous rope op (bit 0: of the list, bit 1: of the
                                        // chain) serves (same positions, frequencies)
  int32_t next;                         // the chain's next op (INT32_MAX: none)
  int32_t flags;                        // kOpWait, kOpCarry
  float eps, inv_n, scale, pad1;
  int64_t zg, zgs;                      // gated: z rows per group, group stride
  const void* x; int64_t x_tok, x_row;  // x / gate / q
  const void* r; int64_t r_tok, r_row;  // r / z / up / k
  const void* w; const void* w2;        // norm weight (q), k norm weight
  void* y; int64_t y_tok, y_row;        // y / out / q out
  void* h; int64_t h_tok, h_row;        // residual out / k out
  const int32_t* offsets;
  int32_t offset;
  int32_t first;                        // in op c: the first op of chain c (INT32_MAX: none)
  float inv_freq[kOpMaxHalf];
};

struct alignas(16) DevOpList {  // its first 16 bytes: one load
  uint32_t magic;
  uint16_t dtype, count;  // count <= HGK_OP_LIST_MAX
  int32_t safe;           // tokens up to which the chains are independent
  uint16_t chains, first; // chains in use; the first op of chain 0
  DevOp ops[1];  // count entries
};
static_assert(HGK_OP_LIST_MAX < 65536, "count and first");

constexpr int64_t op_list_bytes(int n) {
  return (int64_t)sizeof(DevOpList) + (int64_t)(n - 1) * (int64_t)sizeof(DevOp);
}

// kOpWait: in its chain, the op waits for the stores before it. kOpCarry: its x
// is the h of the chain's previous op, an add + norm over the same rows (one
// 16-byte unit per thread), so it is taken from registers.
enum { kOpWait = 1, kOpCarry = 2 };
enum { kOpRms = 0, kOpAddRms = 1, kOpGated = 2, kOpRope = 3, kOpGlu = 4 };

// Whether each op brings the next op's descriptor into the scalar cache.
#ifndef HGK_OPSEQ_PREFETCH
#define HGK_OPSEQ_PREFETCH 1
#endif

// Every store of this op has completed before any thread of the workgroup
// issues the next op's loads.
__device__ inline void op_boundary() {
  __builtin_amdgcn_s_waitcnt(0);  // all counters: loads, stores, LDS
  __syncthreads();
}

// f64 sum over the G lanes of a row group; G = 128 or 256 spans waves and
// goes through LDS (`part`, one slot per wave). Every thread calls it (it
// holds a workgroup barrier when G > 64).
template <int G>
__device__ inline double row_sum(double v, double* part) {
  if constexpr (G <= 64) {
    return group_sum<G>(v);
  } else {
    v = group_sum<64>(v);
    const int wave = threadIdx.x >> 6;
    if ((threadIdx.x & 63) == 0) part[wave] = v;
    __syncthreads();
    constexpr int WPG = G / 64;  // waves per group
    const int first = wave / WPG * WPG;
    double s = 0.0;
#pragma unroll
    for (int k = 0; k < WPG; ++k) s += part[first + k];
    __syncthreads();  // the slots are reused by the next row
    return s;
  }
}

// RMSNorm / add + RMSNorm / gated RMSNorm over the token's rows: G lanes per
// row (G a power of two, 4..1024), one 16-byte unit per lane, 1024 / G rows
// per pass (a token's 32 head rows of 128 in one pass). rms_norm_kernel's
// arithmetic, 16-bit X, weights in X.
template <class X, int MODE, int G>
__device__ __forceinline__ void op_norm(const DevOp& op, int64_t t, double* part) {
  constexpr int V = Vec<X>::N;
  constexpr int P = kOpThreads / G;  // rows per pass
  const int slot = threadIdx.x / G, j = threadIdx.x % G;
  const int nch = op.n / V;
  const bool has_w = op.w != nullptr;
  const int chc = j < nch ? j : nch - 1;
  const char* xb = reinterpret_cast<const char*>(op.x) + t * op.x_tok * X::kBytes;
  const char* rb = reinterpret_cast<const char*>(op.r) + t * op.r_tok * X::kBytes;
  char* yb = reinterpret_cast<char*>(op.y) + t * op.y_tok * X::kBytes;
  char* hb = reinterpret_cast<char*>(op.h) + t * op.h_tok * X::kBytes;
  const u32x4 wr = has_w ? ld16<X>(op.w, (int64_t)chc * V) : u32x4{0u, 0u, 0u, 0u};
  for (int pass = 0; pass * P < op.rows; ++pass) {  // uniform over the workgroup
    const int row = pass * P + slot;
    const bool live = row < op.rows;
    const int rr = live ? row : op.rows - 1;
    int64_t zoff = 0;
    if constexpr (MODE == kOpGated) zoff = (rr / op.zg) * op.zgs + (rr % op.zg) * op.r_row;
    if constexpr (MODE == kOpAddRms) zoff = (int64_t)rr * op.r_row;
    u32x4 xr = ld16<X>(xb, (int64_t)rr * op.x_row + (int64_t)chc * V);
    u32x4 zr{0u, 0u, 0u, 0u};
    if constexpr (MODE != kOpRms) zr = ld16<X>(rb, zoff + (int64_t)chc * V);
    const bool own = live && j < nch;
    if constexpr (MODE == kOpAddRms) {
#pragma unroll
      for (int k = 0; k < 4; ++k)
        xr[k] = X::pack(X::lo(xr[k]) + X::lo(zr[k]), X::hi(xr[k]) + X::hi(zr[k]));
      if (op.h && own)
        *reinterpret_cast<u32x4*>(hb + ((int64_t)row * op.h_row + (int64_t)j * V) * X::kBytes) = xr;
    }
    double ss = 0.0;
    if (j < nch) {
#pragma unroll
      for (int e = 0; e < V; ++e) {
        const double d = (double)elem<X>(xr, e);
        ss = __builtin_fma(d, d, ss);
      }
    }
    ss = row_sum<G>(ss, part);
    const float rs = rms_scale(ss, op.inv_n, op.eps);
    if (!own) continue;
    float o[V];
#pragma unroll
    for (int e = 0; e < V; e += 2) {
      float n0 = elem<X>(xr, e) * rs, n1 = elem<X>(xr, e + 1) * rs;
      round2<X>(n0, n1);
      const float w0 = has_w ? elem<X>(wr, e) : 1.0f, w1 = has_w ? elem<X>(wr, e + 1) : 1.0f;
      n0 = n0 * w0;
      n1 = n1 * w1;
      if constexpr (MODE == kOpGated) {
        round2<X>(n0, n1);
        const float z0 = elem<X>(zr, e), z1 = elem<X>(zr, e + 1);
        float s0, s1;
        sigmoid2_rounded<X>(z0, z1, s0, s1);
        float g0 = z0 * s0, g1 = z1 * s1;
        round2<X>(g0, g1);
        n0 = g0 * n0;
        n1 = g1 * n1;
      }
      o[e] = n0;
      o[e + 1] = n1;
    }
    store_elems<X, V, false>(yb, (int64_t)row * op.y_row + (int64_t)j * V, o);
  }
}

// A run of add + norm ops of one chain over the same rows (at most one row per
// lane group): op i and the ops after it that take their x from its h in
// registers. The next op's r and weight are loaded before the current sum, and
// the sum's LDS slots alternate, so an op costs one workgroup barrier.
// (Two ops ahead measured slower: 196 against 123 us for the 96 ops of a
// 48-layer step; finding the op after next stalls on its cold descriptor.)
// Returns the last op's index.
template <class X, int G>
__device__ __forceinline__ int op_add_run(const DevOpList* list, int i, int n_ops, int64_t t, double (*part)[kOpThreads / 64]) {
  constexpr int V = Vec<X>::N;
  const int row = threadIdx.x / G, j = threadIdx.x % G;
  const DevOp* op = &list->ops[i];
  const int nch = op->n / V;
  const bool own = row < op->rows && j < nch;
  const int rr = row < op->rows ? row : op->rows - 1, chc = j < nch ? j : nch - 1;
  auto at = [&](const void* p, int64_t tok, int64_t rs) {
    return reinterpret_cast<const char*>(p) + (t * tok + (int64_t)rr * rs + (int64_t)chc * V) * X::kBytes;
  };
  auto weight = [&](const DevOp* o) {
    return o->w ? ld16<X>(o->w, (int64_t)chc * V) : u32x4{0u, 0u, 0u, 0u};
  };
  u32x4 xr = ld16<X>(at(op->x, op->x_tok, op->x_row), 0);
  u32x4 r = ld16<X>(at(op->r, op->r_tok, op->r_row), 0);
  u32x4 w = weight(op);
  for (int par = 0;; par ^= 1) {
    const int nx = op->next;
    const DevOp* const no = &list->ops[nx < n_ops ? nx : i];
    const bool more = nx < n_ops && (no->flags & kOpCarry);  // uniform
    u32x4 nr = r, nw = w;
    if (more) {
      nr = ld16<X>(at(no->r, no->r_tok, no->r_row), 0);
      nw = weight(no);
    }
#pragma unroll
    for (int k = 0; k < 4; ++k)
      xr[k] = X::pack(X::lo(xr[k]) + X::lo(r[k]), X::hi(xr[k]) + X::hi(r[k]));
    if (op->h && own) *reinterpret_cast<u32x4*>(const_cast<char*>(at(op->h, op->h_tok, op->h_row))) = xr;
    double ss = 0.0;
    if (j < nch) {
#pragma unroll
      for (int e = 0; e < V; ++e) {
        const double d = (double)elem<X>(xr, e);
        ss = __builtin_fma(d, d, ss);
      }
    }
    if constexpr (G <= 64) {
      ss = group_sum<G>(ss);
    } else {
      ss = group_sum<64>(ss);
      const int wave = threadIdx.x >> 6;
      if ((threadIdx.x & 63) == 0) part[par][wave] = ss;
      __syncthreads();
      constexpr int WPG = G / 64;
      ss = 0.0;
#pragma unroll
      for (int k = 0; k < WPG; ++k) ss += part[par][wave / WPG * WPG + k];
    }
    const float rs = rms_scale(ss, op->inv_n, op->eps);
    if (own) {
      float o[V];
#pragma unroll
      for (int e = 0; e < V; e += 2) {
        float n0 = elem<X>(xr, e) * rs, n1 = elem<X>(xr, e + 1) * rs;
        round2<X>(n0, n1);
        o[e] = n0 * (op->w ? elem<X>(w, e) : 1.0f);
        o[e + 1] = n1 * (op->w ? elem<X>(w, e + 1) : 1.0f);
      }
      store_elems<X, V, false>(const_cast<char*>(at(op->y, op->y_tok, op->y_row)), 0, o);
    }
    if (!more) return i;
    op = no;
    i = nx;
    r = nr;
    w = nw;
  }
}

template <class X>
__device__ __forceinline__ int add_run_dispatch(const DevOpList* list, int i, int n_ops, int64_t t,
                                double (*part)[kOpThreads / 64]) {
  switch (list->ops[i].g) {
    case 4: return op_add_run<X, 4>(list, i, n_ops, t, part);
    case 8: return op_add_run<X, 8>(list, i, n_ops, t, part);
    case 16: return op_add_run<X, 16>(list, i, n_ops, t, part);
    case 32: return op_add_run<X, 32>(list, i, n_ops, t, part);
    case 64: return op_add_run<X, 64>(list, i, n_ops, t, part);
    case 128: return op_add_run<X, 128>(list, i, n_ops, t, part);
    case 256: return op_add_run<X, 256>(list, i, n_ops, t, part);
    case 512: return op_add_run<X, 512>(list, i, n_ops, t, part);
    default: return op_add_run<X, 1024>(list, i, n_ops, t, part);
  }
}

// q/k RMSNorm (where a weight is given) + RoPE of the token's q and k heads:
// rope_kernel's two-chunk layout (lane j < R holds the rotation pair j, j + R;
// the others hold two pass-through chunks), LPR lanes per head row, every
// load issued before the cos/sin table is built. The table (cos/sin of the
// token's position from f64 sincos, rounded to X) lives in LDS; an op whose
// positions and frequencies are those of the previous rope op reuses it.
template <class X, int LPR>
__device__ __forceinline__ void op_rope(const DevOp& op, int64_t t, bool same_table, float* cs, float* sn) {
  constexpr int V = Vec<X>::N;
  constexpr int P = kOpThreads / LPR;
  const int R = op.dims / (2 * V);
  const int slot = threadIdx.x / LPR, j = threadIdx.x % LPR;
  const bool rot = j < R;
  const int c0 = rot ? j : 2 * j, c1 = rot ? j + R : 2 * j + 1;
  const int total = op.rows + op.k_rows;
  for (int pass = 0; pass * P < total; ++pass) {  // uniform over the workgroup
    const int row = pass * P + slot;
    const int rc = row < total ? row : total - 1;
    const bool isk = rc >= op.rows;
    const int hh = isk ? rc - op.rows : rc;
    const char* xp = isk ? reinterpret_cast<const char*>(op.r) +
                               (t * op.r_tok + (int64_t)hh * op.r_row) * X::kBytes
                         : reinterpret_cast<const char*>(op.x) +
                               (t * op.x_tok + (int64_t)hh * op.x_row) * X::kBytes;
    char* yp = isk ? reinterpret_cast<char*>(op.h) + (t * op.h_tok + (int64_t)hh * op.h_row) * X::kBytes
                   : reinterpret_cast<char*>(op.y) + (t * op.y_tok + (int64_t)hh * op.y_row) * X::kBytes;
    const void* nw = isk ? op.w2 : op.w;
    const bool has = nw != nullptr;
    const u32x4 d0 = ld16<X>(xp, (int64_t)c0 * V), d1 = ld16<X>(xp, (int64_t)c1 * V);
    const u32x4 wa = has ? ld16<X>(nw, (int64_t)c0 * V) : u32x4{0u, 0u, 0u, 0u};
    const u32x4 wb = has ? ld16<X>(nw, (int64_t)c1 * V) : u32x4{0u, 0u, 0u, 0u};
    if (pass == 0 && !same_table) {  // built while the loads are in flight
      const int32_t off = op.offsets ? op.offsets[t] : op.offset;
      const float pos = (0.0f + (float)off) * op.scale;
      for (int i = threadIdx.x; i < op.half; i += kOpThreads) {
        float c, s;
        cos_sin_f32(pos * op.inv_freq[i], c, s);
        cs[i] = X::round(c);
        sn[i] = X::round(s);
      }
      __syncthreads();
    }
    if (row >= total) continue;  // whole lane groups leave together; no barrier below
    float v0[V], v1[V];
#pragma unroll
    for (int e = 0; e < V; ++e) {
      v0[e] = elem<X>(d0, e);
      v1[e] = elem<X>(d1, e);
    }
    if (has) {  // uniform over the row's lanes
      double ss = 0.0;
#pragma unroll
      for (int e = 0; e < V; ++e) ss = __builtin_fma((double)v0[e], (double)v0[e], ss);
#pragma unroll
      for (int e = 0; e < V; ++e) ss = __builtin_fma((double)v1[e], (double)v1[e], ss);
      ss = group_sum<LPR>(ss);
      const float rs = rms_scale(ss, op.inv_n, op.eps);
#pragma unroll
      for (int e = 0; e < V; e += 2) {
        float p0 = v0[e] * rs, p1 = v0[e + 1] * rs, q0 = v1[e] * rs, q1 = v1[e + 1] * rs;
        round2<X>(p0, p1);
        round2<X>(q0, q1);
        p0 = p0 * elem<X>(wa, e);
        p1 = p1 * elem<X>(wa, e + 1);
        q0 = q0 * elem<X>(wb, e);
        q1 = q1 * elem<X>(wb, e + 1);
        round2<X>(p0, p1);
        round2<X>(q0, q1);
        v0[e] = p0; v0[e + 1] = p1; v1[e] = q0; v1[e + 1] = q1;
      }
    }
    if (rot) {
      const float* cp = cs + j * V;
      const float* sp = sn + j * V;
#pragma unroll
      for (int e = 0; e < V; e += 2) {
        const float ca = cp[e], sa = sp[e], cb = cp[e + 1], sb = sp[e + 1];
        const float x10 = v0[e], x20 = v1[e], x11 = v0[e + 1], x21 = v1[e + 1];
        float a0 = x10 * ca, a1 = x11 * cb, b0 = x20 * sa, b1 = x21 * sb;
        float d0v = x10 * sa, d1v = x11 * sb, f0 = x20 * ca, f1 = x21 * cb;
        round2<X>(a0, a1);
        round2<X>(b0, b1);
        round2<X>(d0v, d1v);
        round2<X>(f0, f1);
        v0[e] = a0 - b0;
        v0[e + 1] = a1 - b1;
        v1[e] = d0v + f0;
        v1[e + 1] = d1v + f1;
      }
    }
    store_elems<X, V, false>(yp, (int64_t)c0 * V, v0);
    store_elems<X, V, false>(yp, (int64_t)c1 * V, v1);
  }
}

// act(gate) * up over the token's rows: one 16-byte unit per thread per pass
// (glu_kernel's arithmetic).
template <class X, int ACT>
__device__ __forceinline__ void op_glu(const DevOp& op, int64_t t) {
  constexpr int V = Vec<X>::N;
  const int cpr = op.n / V;
  const int total = op.rows * cpr;
  const char* gb = reinterpret_cast<const char*>(op.x) + t * op.x_tok * X::kBytes;
  const char* ub = reinterpret_cast<const char*>(op.r) + t * op.r_tok * X::kBytes;
  char* ob = reinterpret_cast<char*>(op.y) + t * op.y_tok * X::kBytes;
  for (int q = threadIdx.x; q < total; q += kOpThreads) {
    const int row = q / cpr, c = q - row * cpr;
    const u32x4 gr = ld16<X>(gb, (int64_t)row * op.x_row + (int64_t)c * V);
    const u32x4 ur = ld16<X>(ub, (int64_t)row * op.r_row + (int64_t)c * V);
    float o[V];
    if constexpr (ACT == HGK_ACT_SILU) {
      float gv[V], uv[V];
#pragma unroll
      for (int e = 0; e < V; ++e) {
        gv[e] = elem<X>(gr, e);
        uv[e] = elem<X>(ur, e);
      }
      swiglu16<X, V>(gv, uv, o);
    } else {
#pragma unroll
      for (int e = 0; e < V; ++e) o[e] = glu1<X, ACT>(elem<X>(gr, e), elem<X>(ur, e));
    }
    store_elems<X, V, false>(ob, (int64_t)row * op.y_row + (int64_t)c * V, o);
  }
}

template <class X, int MODE>
__device__ __forceinline__ void norm_dispatch(const DevOp& op, int64_t t, double* part) {
  switch (op.g) {
    case 4: op_norm<X, MODE, 4>(op, t, part); break;
    case 8: op_norm<X, MODE, 8>(op, t, part); break;
    case 16: op_norm<X, MODE, 16>(op, t, part); break;
    case 32: op_norm<X, MODE, 32>(op, t, part); break;
    case 64: op_norm<X, MODE, 64>(op, t, part); break;
    case 128: op_norm<X, MODE, 128>(op, t, part); break;
    case 256: op_norm<X, MODE, 256>(op, t, part); break;
    case 512: op_norm<X, MODE, 512>(op, t, part); break;
    default: op_norm<X, MODE, 1024>(op, t, part); break;
  }
}

// ONE: a workgroup per token, which walks the chains one after another (its own
// form: the division by `tokens` alone is 5 % of a one-op list). Else `wgs` per
// token, workgroup wg walking chains wg, wg + wgs, ..
template <class X, bool ONE>
__global__ __launch_bounds__(kOpThreads) void opseq_kernel(const DevOpList* __restrict__ list,
                                                           int n_ops, int tokens, int wgs) {
  __shared__ float cs[kOpMaxHalf], sn[kOpMaxHalf];
  __shared__ double part[2][kOpThreads / 64];
  // all tokens of chain 0 (the longest) first
  if constexpr (ONE) wgs = 1;
  const int wg = ONE ? 0 : blockIdx.x / (unsigned)tokens;
  const int64_t t = blockIdx.x - (unsigned)wg * (unsigned)tokens;
  // a list that hgk_op_list_upload did not write for this dtype and length
  // is not walked (no pointer in it is trusted)
  if (list->magic != kOpListMagic || list->dtype != X::kCode || list->count < n_ops) return;
  const bool serial = tokens > list->safe;  // uniform over the grid
  const int chains = serial ? 1 : list->chains;
  // the first op of chain c is in the descriptor of op c, chain 0's in the list's header too
  auto first = [&](int c) { return c < chains ? list->ops[c].first : INT32_MAX; };
  int chain = wg, i = wg > 0 ? first(wg) : serial ? 0 : list->first;
  int after = first(wg + wgs);  // where this workgroup's next chain begins
  while (chain < chains) {
    if (i < n_ops) {
      const DevOp& op = list->ops[i];
      if (!serial && (op.flags & kOpWait)) op_boundary();
      int nx = serial ? i + 1 : op.next;
      const int ahead = nx < n_ops ? nx : after;
      uint32_t pf[4] = {0u, 0u, 0u, 0u};
      if (HGK_OPSEQ_PREFETCH && ahead < n_ops) {
        // one dword of each 64-byte line of the next descriptor's fields
        const uint32_t* nd = reinterpret_cast<const uint32_t*>(&list->ops[ahead]);
        pf[0] = nd[0]; pf[1] = nd[16]; pf[2] = nd[32]; pf[3] = nd[48];
      }
      switch (op.kind) {
        case kOpRms: norm_dispatch<X, kOpRms>(op, t, part[0]); break;
        case kOpAddRms:
          if (!serial && op.rows * op.g <= kOpThreads) {
            nx = list->ops[add_run_dispatch<X>(list, i, n_ops, t, part)].next;
          } else {
            norm_dispatch<X, kOpAddRms>(op, t, part[0]);
          }
          break;
        case kOpGated: norm_dispatch<X, kOpGated>(op, t, part[0]); break;
        case kOpRope: {
          const bool same = op.same_table & (serial ? 1 : 2);
          switch (op.lpr) {
            case 2: op_rope<X, 2>(op, t, same, cs, sn); break;
            case 4: op_rope<X, 4>(op, t, same, cs, sn); break;
            case 8: op_rope<X, 8>(op, t, same, cs, sn); break;
            case 16: op_rope<X, 16>(op, t, same, cs, sn); break;
            default: op_rope<X, 32>(op, t, same, cs, sn); break;
          }
          break;
        }
        default:
          if (op.act == HGK_ACT_SILU) op_glu<X, HGK_ACT_SILU>(op, t);
          else op_glu<X, HGK_ACT_GELU_TANH>(op, t);
          break;
      }
      if (HGK_OPSEQ_PREFETCH) asm volatile("" ::"s"(pf[0]), "s"(pf[1]), "s"(pf[2]), "s"(pf[3]));
      if (serial) op_boundary();
      else __syncthreads();  // the op's LDS is free
      i = nx;
    }
    if (i >= n_ops) {
      i = after;
      chain += wgs;
      after = first(chain + wgs);
    }
  }
}

namespace {

bool a16(const void* p) { return (reinterpret_cast<uintptr_t>(p) & 15u) == 0; }

int next_pow2(int v) {
  int p = 1;
  while (p < v) p <<= 1;
  return p;
}

// Translate and check one host op; returns HGK_OK or an error status.
int translate(const hgk_op& s, int i, DevOp& d) {
  const char* fn = "hgk_op_list_upload";
  const int V = 8;  // 16-bit elements per 16-byte unit
  d = DevOp{};
  d.kind = s.kind;
  d.rows = s.rows;
  d.n = s.n;
  d.eps = s.eps;
  d.x = s.x; d.x_tok = s.x_tok; d.x_row = s.x_row;
  d.r = s.r; d.r_tok = s.r_tok; d.r_row = s.r_row;
  d.w = s.w; d.w2 = s.w2;
  d.y = s.y; d.y_tok = s.y_tok; d.y_row = s.y_row;
  d.h = s.h; d.h_tok = s.h_tok; d.h_row = s.h_row;
  if (s.rows <= 0 || s.n <= 0 || s.n % V)
    return fail(HGK_ERR_ARG, "%s: op %d: rows=%d n=%d (rows > 0, n a positive multiple of 8)", fn,
                i, s.rows, s.n);
  auto strides_ok = [&](const void* p, int64_t tok, int64_t row) {
    return p && a16(p) && tok % V == 0 && row % V == 0 && tok >= 0 && row >= 0;
  };
  if (!strides_ok(s.x, s.x_tok, s.x_row) || !strides_ok(s.y, s.y_tok, s.y_row))
    return fail(HGK_ERR_ARG, "%s: op %d: x and y must be 16-byte aligned with strides in whole "
                "16-byte units", fn, i);
  if (s.w && !a16(s.w)) return fail(HGK_ERR_ARG, "%s: op %d: weight not 16-byte aligned", fn, i);
  const int nch = s.n / V;
  switch (s.kind) {
    case HGK_OP_RMS_NORM:
    case HGK_OP_ADD_RMS_NORM:
    case HGK_OP_GATED_RMS_NORM: {
      if (!(s.eps >= 0.0f)) return fail(HGK_ERR_ARG, "%s: op %d: eps must be >= 0", fn, i);
      if (nch > kOpThreads)
        return fail(HGK_ERR_UNSUPPORTED, "%s: op %d: n=%d (at most %d)", fn, i, s.n, 8 * kOpThreads);
      if (s.kind != HGK_OP_RMS_NORM && !strides_ok(s.r, s.r_tok, s.r_row))
        return fail(HGK_ERR_ARG, "%s: op %d: r/z must be 16-byte aligned with strides in whole "
                    "16-byte units", fn, i);
      if (s.kind == HGK_OP_ADD_RMS_NORM && s.h && !strides_ok(s.h, s.h_tok, s.h_row))
        return fail(HGK_ERR_ARG, "%s: op %d: h must be 16-byte aligned with strides in whole "
                    "16-byte units", fn, i);
      if (s.kind == HGK_OP_GATED_RMS_NORM) {
        if (!s.w) return fail(HGK_ERR_ARG, "%s: op %d: the gated norm needs a weight", fn, i);
        d.zg = s.z_group_rows > 0 ? s.z_group_rows : s.rows;
        d.zgs = s.z_group_rows > 0 ? s.z_group_stride : 0;
        if (d.zgs % V) return fail(HGK_ERR_ARG, "%s: op %d: z group stride not whole units", fn, i);
      } else {
        d.zg = 1;
      }
      d.g = std::min(kOpThreads, std::max(4, next_pow2(nch)));
      d.inv_n = (float)(1.0 / (double)s.n);
      return HGK_OK;
    }
    case HGK_OP_QK_NORM_ROPE: {
      const int D = s.n;
      if (D < 32 || D > 512 || (D & (D - 1)))
        return fail(HGK_ERR_UNSUPPORTED, "%s: op %d: head_dim %d (a power of two, 32..512)", fn,
                    i, D);
      if (s.dims <= 0 || s.dims > D || s.dims % 16)
        return fail(HGK_ERR_UNSUPPORTED, "%s: op %d: rotated dims %d (a multiple of 16 up to "
                    "head_dim)", fn, i, s.dims);
      if (s.k_heads < 0) return fail(HGK_ERR_ARG, "%s: op %d: k_heads < 0", fn, i);
      if (s.k_heads > 0 && (!strides_ok(s.r, s.r_tok, s.r_row) || !strides_ok(s.h, s.h_tok, s.h_row)))
        return fail(HGK_ERR_ARG, "%s: op %d: k and its output must be 16-byte aligned with "
                    "strides in whole 16-byte units", fn, i);
      if (s.w2 && !a16(s.w2)) return fail(HGK_ERR_ARG, "%s: op %d: k weight not aligned", fn, i);
      if (s.w && !(s.eps >= 0.0f)) return fail(HGK_ERR_ARG, "%s: op %d: eps must be >= 0", fn, i);
      if (s.offsets && (reinterpret_cast<uintptr_t>(s.offsets) & 3u))
        return fail(HGK_ERR_ARG, "%s: op %d: offsets not 4-byte aligned", fn, i);
      d.k_rows = s.k_heads;
      d.dims = s.dims;
      d.half = s.dims / 2;
      d.lpr = D / 16;
      d.scale = s.scale;
      d.offsets = s.offsets;
      d.offset = s.offset;
      d.inv_n = (float)(1.0 / (double)D);
      const int st = hgk_rope_inv_freq(s.base, s.dims, s.freqs, d.inv_freq);
      if (st) return st;
      return HGK_OK;
    }
    case HGK_OP_GLU: {
      if (s.act != HGK_ACT_SILU && s.act != HGK_ACT_GELU_TANH)
        return fail(HGK_ERR_ARG, "%s: op %d: activation %d", fn, i, s.act);
      if (!strides_ok(s.r, s.r_tok, s.r_row))
        return fail(HGK_ERR_ARG, "%s: op %d: up must be 16-byte aligned with strides in whole "
                    "16-byte units", fn, i);
      if ((int64_t)s.rows * s.n > ((int64_t)1 << 30))
        return fail(HGK_ERR_UNSUPPORTED, "%s: op %d: rows x n too large", fn, i);
      d.act = s.act;
      return HGK_OK;
    }
    default:
      return fail(HGK_ERR_ARG, "%s: op %d: unknown kind %d", fn, i, s.kind);
  }
}

// Whether rope op d's cos/sin table is p's: same positions and frequencies.
bool same_positions(const DevOp& p, const DevOp& d) {
  return p.offsets == d.offsets && p.offset == d.offset && p.scale == d.scale && p.half == d.half &&
         std::equal(d.inv_freq, d.inv_freq + d.half, p.inv_freq);
}

// The bytes an op reads or writes for token t: [lo + t tok, lo + t tok + span).
// key: who touches them, where one thread holds one 16-byte unit (add + norm
// over at most kOpThreads units): equal keys, the same threads. -1: others.
struct Range {
  int64_t lo, span, tok;
  bool write;
  int op, key;
  int64_t end() const { return lo + span; }
};

// The smallest t >= 0 for which a's and b's bytes of token t overlap.
int64_t first_overlap(Range a, Range b) {
  if (b.tok < a.tok) std::swap(a, b);
  const int64_t d0 = b.lo - a.lo, dt = b.tok - a.tok;  // overlap: -b.span < d0 + t dt < a.span
  if (d0 >= a.span) return INT64_MAX;
  if (d0 > -b.span) return 0;
  if (dt == 0) return INT64_MAX;
  const int64_t t = (-b.span - d0) / dt + 1;  // the first t with d0 + t dt > -b.span
  return d0 + t * dt < a.span ? t : INT64_MAX;
}

// Append an op's ranges to v; x is the first.
void op_ranges(const DevOp& d, int op, std::map<std::array<int64_t, 5>, int>& keys, std::vector<Range>& v) {
  const bool own = d.kind == kOpAddRms && d.rows * d.g <= kOpThreads;
  auto add = [&](const void* p, int64_t tok, int64_t rows, int64_t row, bool write) {
    if (!p || rows <= 0) return;
    const int64_t lo = (int64_t)(intptr_t)p;
    int key = -1;
    if (own) key = keys.try_emplace({lo, tok, row, rows, d.n}, (int)keys.size()).first->second;
    v.push_back({lo, ((rows - 1) * row + d.n) * 2, tok * 2, write, op, key});
  };
  auto other = [&](const void* p, int64_t off, int64_t bytes, int64_t tok) {
    v.push_back({(int64_t)(intptr_t)p + off, bytes, tok, false, op, -1});
  };
  add(d.x, d.x_tok, d.rows, d.x_row, false);
  add(d.y, d.y_tok, d.rows, d.y_row, true);
  if (d.w) other(d.w, 0, d.n * 2, 0);
  if (d.kind == kOpAddRms || d.kind == kOpGlu) add(d.r, d.r_tok, d.rows, d.r_row, false);
  if (d.kind == kOpAddRms) add(d.h, d.h_tok, d.rows, d.h_row, true);
  if (d.kind == kOpGated) {
    const int64_t groups = (d.rows + d.zg - 1) / d.zg, rows = std::min<int64_t>(d.rows, d.zg);
    const int64_t far = (groups - 1) * d.zgs;  // may be negative
    const int64_t lo = std::min<int64_t>(far, 0), hi = std::max<int64_t>(far, 0) + (rows - 1) * d.r_row + d.n;
    other(d.r, lo * 2, (hi - lo) * 2, d.r_tok * 2);
  }
  if (d.kind == kOpRope) {
    add(d.r, d.r_tok, d.k_rows, d.r_row, false);
    add(d.h, d.h_tok, d.k_rows, d.h_row, true);
    if (d.w2) other(d.w2, 0, d.n * 2, 0);
    if (d.offsets) other(d.offsets, 0, 4, 4);
  }
}

struct Groups {
  std::vector<int> root, size;
  explicit Groups(int n) : root(n), size(n, 1) {
    for (int i = 0; i < n; ++i) root[i] = i;
  }
  int find(int i) {
    while (root[i] != i) i = root[i] = root[root[i]];
    return i;
  }
  void join(int i, int j) {
    i = find(i);
    j = find(j);
    if (i == j) return;
    size[j] += size[i];
    root[i] = j;
  }
};

// Join the ops that share bytes of token 0, one of them writing: a sweep over
// the ranges, sorted by address. Of the writes that reach the current address one
// stands for all (they overlap there, so their ops are joined; the one that
// ends last is met by whatever meets any), and so does one of the reads that a
// write has joined.
void join_overlaps(const std::vector<Range>& sorted, Groups& g) {
  Range w{};  // the write that ends last (op -1: none)
  w.op = -1;
  std::vector<Range> reads;  // not joined with each other; some have ended
  for (const Range& r : sorted) {
    if (w.op >= 0 && w.end() > r.lo) g.join(w.op, r.op);
    if (!r.write) {
      reads.push_back(r);
      continue;
    }
    Range last = r;
    for (const Range& q : reads) {
      if (q.end() <= r.lo) continue;
      g.join(q.op, r.op);
      if (q.end() > last.end()) last = q;
    }
    reads.clear();
    if (last.op != r.op || last.end() > r.end()) reads.push_back(last);
    if (w.op < 0 || w.end() <= r.lo || r.end() > w.end()) w = r;
  }
}

// The first token t >= 1 for which ops share bytes, one of them writing, that
// they do not share for token 0 (only ranges with different token strides do),
// or `safe` where that is smaller. Per pair of strides, each range of the
// larger one meets the ranges above it, nearest first, until a range is too far
// to be met before `safe`.
int64_t first_later_overlap(const std::vector<Range>& sorted, int64_t safe) {
  std::map<int64_t, std::array<std::vector<Range>, 2>> by;  // per stride: all ranges, the writes
  for (const Range& r : sorted) {
    auto& lists = by[r.tok];
    lists[0].push_back(r);
    if (r.write) lists[1].push_back(r);
  }
  // (many strides would make many pairs: such a list runs in order)
  if (by.size() > 32) return 0;
  for (const auto& [small, as] : by)
    for (const auto& [large, bs] : by) {
      if (large <= small) continue;
      for (const Range& b : bs[0]) {
        const std::vector<Range>& l = as[b.write ? 0 : 1];
        auto a = std::lower_bound(l.begin(), l.end(), b.end(), [](const Range& r, int64_t end) { return r.lo < end; });
        for (; a != l.end() && (a->lo - b.end()) / (large - small) + 1 < safe; ++a)
          if (a->op != b.op) safe = std::min(safe, first_overlap(*a, b));
      }
    }
  return safe;
}

// The bytes that a chain's ops have read (written) since its last wait, as
// disjoint segments; a segment has the key of its only range, or -1.
struct Touched {
  std::map<int64_t, std::pair<int64_t, int>> seg;  // lo -> end, key
  // whether [r.lo, r.end()) meets a segment, other than one of key `but` (>= 0)
  bool meets(const Range& r, int but) const {
    auto it = seg.upper_bound(r.lo);
    if (it != seg.begin() && std::prev(it)->second.first > r.lo) --it;
    for (; it != seg.end() && it->first < r.end(); ++it)
      if (but < 0 || it->second.second != but) return true;
    return false;
  }
  void add(const Range& r) {
    int64_t lo = r.lo, end = r.end();
    int key = r.key;
    auto it = seg.upper_bound(lo);
    if (it != seg.begin() && std::prev(it)->second.first > lo) --it;
    while (it != seg.end() && it->first < end) {
      if (it->second.second != key) key = -1;
      lo = std::min(lo, it->first);
      end = std::max(end, it->second.first);
      it = seg.erase(it);
    }
    seg.emplace(lo, std::make_pair(end, key));
  }
};

// Sort the list's ops into chains (see the top of the file).
void make_chains(DevOpList* L) {
  const int n = L->count;
  std::map<std::array<int64_t, 5>, int> keys;
  std::vector<Range> all;        // op i's ranges: at[i] .. at[i + 1] - 1
  std::vector<size_t> at(n + 1, 0);
  all.reserve(6 * n);
  for (int i = 0; i < n; ++i) {
    op_ranges(L->ops[i], i, keys, all);
    at[i + 1] = all.size();
  }
  std::vector<Range> sorted = all;
  std::sort(sorted.begin(), sorted.end(), [](const Range& a, const Range& b) { return a.lo < b.lo; });
  Groups groups(n);
  join_overlaps(sorted, groups);
  int64_t safe = first_later_overlap(sorted, INT32_MAX);
  // the largest group of dependent ops is chain 0; each other group goes to
  // the chain with the fewest ops so far
  int big = 0;
  for (int i = 0; i < n; ++i)
    if (groups.size[groups.find(i)] > groups.size[groups.find(big)]) big = i;
  std::vector<int> of(n, -1), chain(n);
  int load[kChains] = {};
  of[groups.find(big)] = 0;
  load[0] = groups.size[groups.find(big)];
  for (int i = 0; i < n; ++i) {
    int& c = of[groups.find(i)];
    if (c < 0) {
      c = (int)(std::min_element(load, load + kChains) - load);
      load[c] += groups.size[groups.find(i)];
    }
    chain[i] = c;
  }
  int last[kChains], rope[kChains];
  Touched reads[kChains], writes[kChains];
  for (int c = 0; c < kChains; ++c) {
    last[c] = rope[c] = -1;
    if (c < n) L->ops[c].first = INT32_MAX;
  }
  for (int i = 0; i < n; ++i) {
    DevOp& d = L->ops[i];
    const int c = chain[i], p = last[c];
    d.next = INT32_MAX;
    d.flags = 0;
    if (p < 0) {
      L->ops[c].first = i;
    } else {
      DevOp& q = L->ops[p];
      q.next = i;
      bool carry = d.kind == kOpAddRms && q.kind == kOpAddRms && q.h && d.x == q.h &&
                   d.x_tok == q.h_tok && d.x_row == q.h_row && d.rows == q.rows && d.n == q.n &&
                   d.rows * d.g <= kOpThreads;
      // where q's y lies on its h, x is y, stored last
      int64_t over = INT64_MAX;
      if (carry)
        for (size_t a = at[p]; a < at[p + 1]; ++a)
          for (size_t b = a + 1; b < at[p + 1]; ++b)
            if (all[a].write && all[b].write) over = std::min(over, first_overlap(all[a], all[b]));
      carry = carry && over > 0;
      // a carried op reads x from registers, and where it writes what the same
      // threads read or wrote before, program order is enough
      bool wait = false;
      for (size_t k = at[i] + carry; k < at[i + 1] && !wait; ++k) {
        const Range& r = all[k];
        const int but = carry && r.write ? r.key : -1;
        wait = writes[c].meets(r, but) || (r.write && reads[c].meets(r, but));
      }
      if (carry && !wait) {
        d.flags = kOpCarry;
        safe = std::min(safe, over);
      }
      if (wait) {
        d.flags |= kOpWait;
        reads[c].seg.clear();
        writes[c].seg.clear();
      }
    }
    for (size_t k = at[i]; k < at[i + 1]; ++k) (all[k].write ? writes : reads)[c].add(all[k]);
    last[c] = i;
    if (d.kind == kOpRope) {
      if (rope[c] >= 0 && same_positions(L->ops[rope[c]], d)) d.same_table |= 2;
      rope[c] = i;
    }
  }
  L->chains = (uint16_t)(1 + *std::max_element(chain.begin(), chain.end()));
  L->first = (uint16_t)L->ops[0].first;
  L->safe = (int32_t)safe;
}

}  // namespace
}  // namespace hgk

using namespace hgk;

extern "C" int64_t hgk_op_list_bytes(int n_ops) {
  if (n_ops <= 0 || n_ops > HGK_OP_LIST_MAX) return -1;
  return op_list_bytes(n_ops);
}

extern "C" int hgk_op_list_upload(int dtype, const hgk_op* ops, int n_ops, void* dev_list,
                                  int64_t dev_bytes, void* stream) try {
  clear_error();
  const char* fn = "hgk_op_list_upload";
  if (dtype != DT_BF16 && dtype != DT_F16)
    return fail(HGK_ERR_UNSUPPORTED, "%s: dtype %s (bf16 or f16)", fn, dtype_name(dtype));
  if (!ops || n_ops <= 0 || n_ops > HGK_OP_LIST_MAX)
    return fail(HGK_ERR_ARG, "%s: %d ops (1..%d)", fn, n_ops, HGK_OP_LIST_MAX);
  if (!dev_list || !a16(dev_list)) return fail(HGK_ERR_ARG, "%s: null or unaligned list", fn);
  const int64_t need = op_list_bytes(n_ops);
  if (dev_bytes < need)
    return fail(HGK_ERR_ARG, "%s: %lld bytes given, %lld needed", fn, (long long)dev_bytes,
                (long long)need);
  std::vector<char> host((size_t)need, 0);
  DevOpList* L = reinterpret_cast<DevOpList*>(host.data());
  L->magic = kOpListMagic;
  L->dtype = (uint16_t)dtype;
  L->count = (uint16_t)n_ops;
  int last_rope = -1;
  for (int i = 0; i < n_ops; ++i) {
    const int st = translate(ops[i], i, L->ops[i]);
    if (st) return st;
    DevOp& d = L->ops[i];
    if (d.kind != kOpRope) continue;
    // the previous rope op's table is still in LDS when this op runs: reuse it
    // when the positions and frequencies are the same
    if (last_rope >= 0) d.same_table = same_positions(L->ops[last_rope], d);
    last_rope = i;
  }
  make_chains(L);
  hipError_t e = hipMemcpyAsync(dev_list, host.data(), (size_t)need, hipMemcpyHostToDevice,
                                as_stream(stream));
  if (e == hipSuccess) e = hipStreamSynchronize(as_stream(stream));
  if (e != hipSuccess) return fail(HGK_ERR_HIP, "%s: copy failed: %s", fn, hipGetErrorString(e));
  return HGK_OK;
} catch (const std::bad_alloc&) {
  return fail(HGK_ERR_HIP, "hgk_op_list_upload: out of host memory");
}

extern "C" int hgk_op_list_run(int dtype, const void* dev_list, int n_ops, int64_t tokens,
                               void* stream) {
  clear_error();
  const char* fn = "hgk_op_list_run";
  if (dtype != DT_BF16 && dtype != DT_F16)
    return fail(HGK_ERR_UNSUPPORTED, "%s: dtype %s (bf16 or f16)", fn, dtype_name(dtype));
  if (!dev_list || !a16(dev_list)) return fail(HGK_ERR_ARG, "%s: null or unaligned list", fn);
  if (n_ops <= 0 || n_ops > HGK_OP_LIST_MAX)
    return fail(HGK_ERR_ARG, "%s: %d ops (1..%d)", fn, n_ops, HGK_OP_LIST_MAX);
  if (tokens < 0 || tokens > ((int64_t)1 << 31) - 1)
    return fail(HGK_ERR_ARG, "%s: tokens=%lld", fn, (long long)tokens);
  if (tokens == 0) return HGK_OK;
  const DevOpList* L = static_cast<const DevOpList*>(dev_list);
  const dim3 b(kOpThreads);
  // Workgroups per token: one per chain while the tokens alone leave CUs idle. A
  // workgroup fills a CU, so with more of them than CUs each costs a start (some
  // 0.5 us), also where its chains are empty. us for the 192 ops of a 48-layer
  // step / 8 independent GLUs / one add + norm, by workgroups per token:
  //   tokens   1                 3                 4                 8
  //   64       348 / 13.8 / 4.8  190 / 7.8 / 4.8   159 / 6.7 / 4.8   125 / 7.8 / 4.8
  //   128      409 / 14.1 / 5.5  238 / 11.2 / 5.5  239 / 10.3 / 5.5  243 / 12.3 / 6.3
  //   192      420 / 14.2 / 5.8  353 / 14.8 / 6.2  355 / 14.1 / 6.7  358 / 16.9 / 8.2
  //   256      435 / 14.7 / 6.0  443 / 17.0 / 7.5  444 / 17.7 / 8.0  455 / 21.8 / 9.9
  // and at 4096 tokens 222 / 52 us for the GLUs / the one norm against 340 / 116
  // (one workgroup that waits after every op: 208 / 47.5; 8 adds + norms in a
  // chain 219, 284 and 316).
  const int wgs = tokens <= 96 ? kChains : tokens <= 128 ? 4 : tokens < 224 ? 3 : 1;
  const dim3 g((unsigned)(tokens * wgs));
  const int nt = (int)tokens;
  const hipStream_t st = as_stream(stream);
  if (dtype == DT_BF16) {
    if (wgs == 1) HGK_LAUNCH((opseq_kernel<BF16, true>), g, b, 0, st, L, n_ops, nt, wgs);
    else HGK_LAUNCH((opseq_kernel<BF16, false>), g, b, 0, st, L, n_ops, nt, wgs);
  } else {
    if (wgs == 1) HGK_LAUNCH((opseq_kernel<F16, true>), g, b, 0, st, L, n_ops, nt, wgs);
    else HGK_LAUNCH((opseq_kernel<F16, false>), g, b, 0, st, L, n_ops, nt, wgs);
  }
  return launch_status(fn);
}
