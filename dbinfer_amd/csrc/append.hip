// Append kernels: one launch writes n consecutive positions of one layer and
// leaves the storage exactly as n sequential KVCache::append calls would
// (model.cpp:357-404). For the dense caches of head dims 64 and 128 the same
// launch also produces the rows from raw projections (bias, rope;
// model.cpp:933-954) and ropes the chunk's queries (rows_f32_kernel,
// rows_i8_kernel); the kernels before them serve rings and other head dims.
//
// The int8 arithmetic (quant.hpp) is bit-exact with the reference; codes are
// stored as signed bytes in the granule layout of kv_internal.hpp.
#include "kv_internal.hpp"
#include "quant.hpp"

namespace dbi {
namespace {

constexpr int kThreads = 256;

// In a batch, a ring row is overwritten by row p + W when that row is in the
// same batch; only the last writer of each slot stores (sequential result).
__device__ __forceinline__ bool ring_row_final(int p, int end, int s, int W) {
  return p < s || p + W >= end;
}

// fp32 copy into dense slot pos or ring slot slot_for(pos) (model.cpp:386-402).
__global__ __launch_bounds__(kThreads) void append_f32_kernel(KvGeom g, float* kst, float* vst,
                                                              int layer, int pos0, int n,
                                                              const float* __restrict__ k,
                                                              const float* __restrict__ v) {
  const int P = g.nkv * g.hd;
  const size_t total = static_cast<size_t>(n) * P;
  for (size_t idx = blockIdx.x * static_cast<size_t>(kThreads) + threadIdx.x; idx < total;
       idx += static_cast<size_t>(gridDim.x) * kThreads) {
    const int r = static_cast<int>(idx / P);
    const int c = static_cast<int>(idx % P);
    const int p = pos0 + r;
    int slot = p;
    if (g.ring) {
      if (!ring_row_final(p, pos0 + n, g.n_sink, g.window)) continue;
      slot = slot_for(p, g.n_sink, g.window);
    }
    const int kh = c / g.hd, i = c % g.hd;
    const size_t hb = (static_cast<size_t>(layer) * g.nkv + kh) * head_elems(g);
    kst[hb + k_off(g, slot, i)] = k[idx];
    vst[hb + v_off(g, slot, i)] = v[idx];
  }
}

// Ring int8: quant_head of K and V per kv head into slot_for(pos)
// (model.cpp:386-396). One lane per element, 32 lanes per block.
__global__ __launch_bounds__(kThreads) void append_i8_ring_kernel(KvGeom g, KvStore s, int layer,
                                                                  int pos0, int n,
                                                                  const float* __restrict__ k,
                                                                  const float* __restrict__ v) {
  const int P = g.nkv * g.hd;
  const size_t blocks = static_cast<size_t>(n) * g.nkv * g.nb;
  const size_t bidx = (blockIdx.x * static_cast<size_t>(kThreads) + threadIdx.x) / kBlock;
  const int t = threadIdx.x % kBlock;
  if (bidx >= blocks) return;  // whole 32-lane groups leave together
  const int b = static_cast<int>(bidx % g.nb);
  const int kh = static_cast<int>((bidx / g.nb) % g.nkv);
  const int r = static_cast<int>(bidx / (static_cast<size_t>(g.nb) * g.nkv));
  const int p = pos0 + r;
  const int i = b * kBlock + t;
  const bool in = i < g.hd;
  const size_t src = static_cast<size_t>(r) * P + kh * g.hd + i;
  const float kx = in ? k[src] : 0.0f;
  const float vx = in ? v[src] : 0.0f;
  float ks, vs;
  const int8_t kc = quant_lane(kx, &ks);
  const int8_t vc = quant_lane(vx, &vs);
  if (!ring_row_final(p, pos0 + n, g.n_sink, g.window)) return;
  const int slot = slot_for(p, g.n_sink, g.window);
  const size_t head = static_cast<size_t>(layer) * g.nkv + kh;
  const size_t row = head * g.capg + slot;
  if (in) {
    s.k8[head * head_elems(g) + k_off(g, slot, i)] = kc;
    s.v8[head * head_elems(g) + v_off(g, slot, i)] = vc;
  }
  if (t == 0) {
    s.k_scale[row * g.nb + b] = ks;
    s.v_scale[row * g.nb + b] = vs;
  }
}

// Dense int8 key side (model.cpp:358-384, requantize_kgroup :329-355) of a
// batch [pos0, pos0 + n): one thread per (32-token group, channel). The
// result is that of n sequential appends: a group ends requantized over its
// raw rows [0, within] that are not sinks, with within the batch's last row
// in the group. Those rows come from the batch, or, before pos0 in the first
// group, from the staging rows k_raw left by earlier appends (which keeps the
// reference's staging-row aliasing after a rollback). Groups are
// independent; the staging rows are rewritten afterwards
// (append_i8_kraw_kernel), so every reader here sees them as they were.
__global__ __launch_bounds__(kThreads) void append_i8_kgroup_kernel(KvGeom g, KvStore s, int layer,
                                                                    int pos0, int n,
                                                                    const float* __restrict__ k) {
  const int P = g.nkv * g.hd;
  const int c = blockIdx.x * kThreads + threadIdx.x;
  if (c >= P) return;
  const int kh = c / g.hd, i = c % g.hd;
  const int grp = pos0 / kKGroup + static_cast<int>(blockIdx.y);
  const int first = grp * kKGroup, end = pos0 + n;
  const int within = min(end - 1, first + kKGroup - 1) - first;
  const float* raw = s.k_raw + static_cast<size_t>(layer) * kKGroup * P + c;
  const size_t head = static_cast<size_t>(layer) * g.nkv + kh;
  float x[kKGroup];
  float mx = 0.0f;
#pragma unroll
  for (int w = 0; w < kKGroup; ++w) {
    const int p = first + w;  // uniform over the block
    x[w] = w > within ? 0.0f
                      : (p >= pos0 ? k[static_cast<size_t>(p - pos0) * P + c]
                                   : raw[static_cast<size_t>(w) * P]);
    if (w <= within && p >= g.n_sink) mx = max_f(mx, fabsf(x[w]));
  }
  const float sc = mx / 127.0f;
  s.k_scale[(head * g.ngroups + grp) * g.hd + i] = sc;
  const float inv = sc > 0.0f ? 1.0f / sc : 0.0f;
#pragma unroll
  for (int w = 0; w < kKGroup; ++w)
    if (w <= within && first + w >= g.n_sink)
      s.k8[head * head_elems(g) + k_off(g, first + w, i)] = quant_code(x[w], inv);
}

// The staging rows after the batch: k_raw[w] holds the batch's last row p
// with p % 32 == w (n sequential appends each copy k into k_raw[p % 32]).
__global__ __launch_bounds__(kThreads) void append_i8_kraw_kernel(KvGeom g, KvStore s, int layer,
                                                                  int pos0, int n,
                                                                  const float* __restrict__ k) {
  const int P = g.nkv * g.hd;
  const size_t idx = blockIdx.x * static_cast<size_t>(kThreads) + threadIdx.x;
  if (idx >= static_cast<size_t>(kKGroup) * P) return;
  const int w = static_cast<int>(idx / P), c = static_cast<int>(idx % P);
  const int last = pos0 + n - 1;
  const int p = last - (((last - w) % kKGroup) + kKGroup) % kKGroup;
  if (p >= pos0)
    s.k_raw[static_cast<size_t>(layer) * kKGroup * P + idx] = k[static_cast<size_t>(p - pos0) * P + c];
}

// Dense int8 value side (model.cpp:366-384), one lane per element, 32 lanes
// per (row, kv head, block): fp32 sink copy of K and V for pos < n_sink, else
// quant_head of V.
__global__ __launch_bounds__(kThreads) void append_i8_dense_v_kernel(KvGeom g, KvStore s, int layer,
                                                                     int pos0, int n,
                                                                     const float* __restrict__ k,
                                                                     const float* __restrict__ v) {
  const int P = g.nkv * g.hd;
  const size_t blocks = static_cast<size_t>(n) * g.nkv * g.nb;
  const size_t bidx = (blockIdx.x * static_cast<size_t>(kThreads) + threadIdx.x) / kBlock;
  const int t = threadIdx.x % kBlock;
  if (bidx >= blocks) return;  // whole 32-lane groups leave together
  const int b = static_cast<int>(bidx % g.nb);
  const int kh = static_cast<int>((bidx / g.nb) % g.nkv);
  const int r = static_cast<int>(bidx / (static_cast<size_t>(g.nb) * g.nkv));
  const int p = pos0 + r;
  const int i = b * kBlock + t;
  const bool in = i < g.hd;
  const size_t src = static_cast<size_t>(r) * P + kh * g.hd + i;
  const size_t head = static_cast<size_t>(layer) * g.nkv + kh;
  const float vx = in ? v[src] : 0.0f;
  if (p < g.n_sink) {  // uniform over the 32-lane group
    if (in) {
      const size_t dst = (head * g.n_sink + p) * g.hd + i;
      s.k_sink[dst] = k[src];
      s.v_sink[dst] = vx;
    }
    return;
  }
  float vs;
  const int8_t vc = quant_lane(vx, &vs);
  if (in) s.v8[head * head_elems(g) + v_off(g, p, i)] = vc;
  if (t == 0) s.v_scale[(head * g.capg + p) * g.nb + b] = vs;
}

int grid_for(size_t work) {
  const size_t blocks = (work + kThreads - 1) / kThreads;
  return static_cast<int>(blocks < 65536 ? (blocks == 0 ? 1 : blocks) : 65536);
}

// [L][len][nkv][hd] <-> the head-major K (is_k) or V store
template <typename T>
__global__ __launch_bounds__(kThreads) void prefix_pack_kernel(KvGeom g, const T* store, T* dst,
                                                               int len, int unpack, int is_k) {
  const size_t P = static_cast<size_t>(g.nkv) * g.hd;
  const size_t total = static_cast<size_t>(g.n_layers) * len * P;
  for (size_t idx = blockIdx.x * static_cast<size_t>(kThreads) + threadIdx.x; idx < total;
       idx += static_cast<size_t>(gridDim.x) * kThreads) {
    const size_t l = idx / (len * P);
    const size_t rem = idx % (len * P);
    const size_t p = rem / P;
    const size_t kh = (rem % P) / g.hd;
    const size_t i = rem % g.hd;
    const size_t st = (l * g.nkv + kh) * head_elems(g) +
                      (is_k ? k_off(g, static_cast<int>(p), static_cast<int>(i))
                            : v_off(g, static_cast<int>(p), static_cast<int>(i)));
    if (unpack)
      const_cast<T*>(store)[st] = dst[idx];
    else
      dst[idx] = store[st];
  }
}

// Row-major per-head arrays: store [L][nkv][dev_rows][inner] <-> file
// [L][rows][nkv][inner], the first `rows` rows of every head.
__global__ __launch_bounds__(kThreads) void rows_pack_kernel(const float* store, float* file,
                                                             int n_layers, int nkv, int dev_rows,
                                                             int rows, int inner, int unpack) {
  const size_t per_layer = static_cast<size_t>(rows) * nkv * inner;
  const size_t total = static_cast<size_t>(n_layers) * per_layer;
  for (size_t idx = blockIdx.x * static_cast<size_t>(kThreads) + threadIdx.x; idx < total;
       idx += static_cast<size_t>(gridDim.x) * kThreads) {
    const size_t l = idx / per_layer;
    const size_t rem = idx % per_layer;
    const size_t r = rem / (static_cast<size_t>(nkv) * inner);
    const size_t kh = (rem / inner) % nkv;
    const size_t i = rem % inner;
    const size_t st = ((l * nkv + kh) * dev_rows + r) * inner + i;
    if (unpack)
      const_cast<float*>(store)[st] = file[idx];
    else
      file[idx] = store[st];
  }
}

// ---------------------------------------------------------------------------
// Rows of a dense cache (head dims 64 and 128) in one launch: the producer's
// bias and rope (produce.hip's arithmetic), the append, and the roped queries.
// A chunk step took up to four launches for this (the producer, then K
// groups, staging rows and V of the int8 cache, each reading back what the
// one before wrote); at a few rows each is a launch and a memory round trip.
//
// Bound: latency at verify rounds, bandwidth at prompts (every row read once
// and written once). 8 values per lane, a K or q piece being two float4 that
// are each other's rope partners (dims 4 c.. and hd/2 + 4 c..: a granule's
// layout), a V piece dims 8 c.. .
// Measured, a layer's whole chunk step: 5 rows at 16 k (32/8 heads, hd 128)
// int8 37.8 -> 27.1 us (0.4 of it V codes in 4-byte stores; twice the threads
// at hd 128 measured no faster), fp32 35.5 -> 33.2; 256 int8 rows at 3840 99.7 -> 88.0;
// 1000 fp32 rows of 28/4 heads 75.5 -> 70.7.
constexpr int kRowThreads = 256;
typedef float f4u __attribute__((ext_vector_type(4), aligned(4)));  // rows of any alignment
typedef float f4a __attribute__((ext_vector_type(4)));

struct RowsArgs {
  AppendRows r;
  int layer, pos0, n;
};

struct Piece {
  f4a lo, hi;
};

__device__ __forceinline__ Piece load_piece(const float* row, int lo, int hi) {
  Piece p;
  p.lo = *reinterpret_cast<const f4u*>(row + lo);
  p.hi = *reinterpret_cast<const f4u*>(row + hi);
  return p;
}

__device__ __forceinline__ void add_bias(Piece& p, const float* bias, int lo, int hi) {
  if (bias == nullptr) return;  // uniform
  const Piece b = load_piece(bias, lo, hi);
  p.lo += b.lo;
  p.hi += b.hi;
}

// (cos, sin) of a piece's four pairs at a position
struct PairTab {
  double2 t[4];
};
__device__ __forceinline__ PairTab load_tab(const double2* cs, int half, int pos, int c) {
  PairTab t;
#pragma unroll
  for (int i = 0; i < 4; ++i) t.t[i] = cs[static_cast<size_t>(pos) * half + 4 * c + i];
  return t;
}
__device__ __forceinline__ void rope_piece(Piece& p, const PairTab& t) {
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const float2 y = rope_rotate(p.lo[i], p.hi[i], t.t[i].x, t.t[i].y);
    p.lo[i] = y.x;
    p.hi[i] = y.y;
  }
}

// query piece idx of the chunk, roped into q_out
template <int HD>
__device__ __forceinline__ void rope_query(const RowsArgs& a, size_t idx) {
  constexpr int LPR = HD / 8, half = HD / 2;
  const int nh = a.r.n_heads;
  const int c = static_cast<int>(idx % LPR);
  const size_t rh = idx / LPR;  // row * nh + head
  if (rh >= static_cast<size_t>(a.n) * nh) return;
  const int h = static_cast<int>(rh % nh), row = static_cast<int>(rh / nh);
  Piece x = load_piece(a.r.q + rh * HD, 4 * c, half + 4 * c);
  PairTab t;
  if (a.r.cs != nullptr) t = load_tab(a.r.cs, half, a.pos0 + row, c);
  add_bias(x, a.r.qb == nullptr ? nullptr : a.r.qb + h * HD, 4 * c, half + 4 * c);
  if (a.r.cs != nullptr) rope_piece(x, t);
  float* dst = a.r.q_out + rh * HD;
  *reinterpret_cast<f4a*>(dst + 4 * c) = x.lo;
  *reinterpret_cast<f4a*>(dst + half + 4 * c) = x.hi;
}

// fp32: pieces of the key heads, the value heads and the query heads of a row
template <int HD>
__global__ __launch_bounds__(kRowThreads) void rows_f32_kernel(KvGeom g, KvStore s, RowsArgs a) {
  constexpr int LPR = HD / 8, half = HD / 2;
  const size_t idx = blockIdx.x * static_cast<size_t>(kRowThreads) + threadIdx.x;
  const size_t kv = static_cast<size_t>(a.n) * 2 * g.nkv * LPR;
  if (idx >= kv) {
    rope_query<HD>(a, idx - kv);
    return;
  }
  const int c = static_cast<int>(idx % LPR);
  const int w = static_cast<int>(idx / LPR % (2 * g.nkv));
  const int row = static_cast<int>(idx / (static_cast<size_t>(LPR) * 2 * g.nkv));
  const bool is_k = w < g.nkv;
  const int kh = is_k ? w : w - g.nkv, pos = a.pos0 + row;
  const size_t head = (static_cast<size_t>(a.layer) * g.nkv + kh) * head_elems(g);
  const float* src = (is_k ? a.r.k : a.r.v) + (static_cast<size_t>(row) * g.nkv + kh) * HD;
  const float* bias = is_k ? a.r.kb : a.r.vb;
  const int lo = is_k ? 4 * c : 8 * c, hi = is_k ? half + 4 * c : 8 * c + 4;
  Piece x = load_piece(src, lo, hi);
  PairTab t;
  const bool rope = is_k && a.r.cs != nullptr;
  if (rope) t = load_tab(a.r.cs, half, pos, c);
  add_bias(x, bias == nullptr ? nullptr : bias + kh * HD, lo, hi);
  if (rope) rope_piece(x, t);
  // (a granule slot holds the pieces' first halves, then their second halves)
  float* dst = (is_k ? s.k + k_off_tiled(HD, false, pos, 4 * c) : s.v + v_off_tiled(HD, false, pos, 8 * c)) + head;
  *reinterpret_cast<f4a*>(dst) = x.lo;
  *reinterpret_cast<f4a*>(dst + 256) = x.hi;
}

// int8: a workgroup per (32-token group, kv head), after n_groups * nkv of
// them the query pieces. The group ends requantized over its raw rows
// [0, within] that are not sinks, within the batch's last row in it: rows from
// the batch, or before pos0 from the staging rows k_raw as earlier appends
// left them. The first group's workgroup is the only one to touch its head's
// staging rows: it reads them, then rewrites k_raw[w] with the batch's last
// row p = w (mod 32). Codes cross LDS so that a whole group goes out in
// 16-byte stores; of a partial one only the rows it holds.
template <int HD>
__global__ __launch_bounds__(kRowThreads) void rows_i8_kernel(KvGeom g, KvStore s, RowsArgs a, int n_groups) {
  constexpr int LPR = HD / 8, half = HD / 2;
  constexpr int RP = kRowThreads / LPR, NP = kKGroup / RP;  // rows per pass, passes
  constexpr int CH = kKGroup * HD;                          // codes of a group
  __shared__ float s_max[kRowThreads / 64][HD];
  __shared__ __align__(16) int8_t s_k[CH];
  __shared__ __align__(16) int8_t s_v[CH];
  const int groups = n_groups * g.nkv;
  if (static_cast<int>(blockIdx.x) >= groups) {
    rope_query<HD>(a, (blockIdx.x - groups) * static_cast<size_t>(kRowThreads) + threadIdx.x);
    return;
  }
  const int kh = static_cast<int>(blockIdx.x) % g.nkv, gi = static_cast<int>(blockIdx.x) / g.nkv;
  const int grp = a.pos0 / kKGroup + gi, first = grp * kKGroup, end = a.pos0 + a.n;
  const int within = min(end - 1, first + kKGroup - 1) - first;
  const int w0 = max(a.pos0 - first, 0);        // the group's first row of the batch
  const int ws = max(g.n_sink - first, 0);      // its first row that is no sink
  const int tid = static_cast<int>(threadIdx.x), c = tid % LPR, r = tid / LPR;
  const int P = g.nkv * HD;
  const size_t head = static_cast<size_t>(a.layer) * g.nkv + kh;
  float* raw = s.k_raw + static_cast<size_t>(a.layer) * kKGroup * P + kh * HD;
  const float* kin = a.r.k + kh * HD;
  const float* kb = a.r.kb == nullptr ? nullptr : a.r.kb + kh * HD;

  // batch row p of the keys, produced
  auto key_row = [&](int p) {
    Piece x = load_piece(kin + static_cast<size_t>(p - a.pos0) * P, 4 * c, half + 4 * c);
    PairTab t;
    if (a.r.cs != nullptr) t = load_tab(a.r.cs, half, p, c);
    add_bias(x, kb, 4 * c, half + 4 * c);
    if (a.r.cs != nullptr) rope_piece(x, t);
    return x;
  };
  // every load of the lane's rows before the first use (a row past `within`
  // repeats it, a V row before the batch its first)
  Piece k[NP], v[NP];
  PairTab t[NP];
#pragma unroll
  for (int i = 0; i < NP; ++i) {
    const int w = min(r + RP * i, within), wb = max(w, w0);
    k[i] = load_piece(w >= w0 ? kin + static_cast<size_t>(first + w - a.pos0) * P : raw + static_cast<size_t>(w) * P,
                      4 * c, half + 4 * c);
    v[i] = load_piece(a.r.v + static_cast<size_t>(first + wb - a.pos0) * P + kh * HD, 8 * c, 8 * c + 4);
    if (a.r.cs != nullptr) t[i] = load_tab(a.r.cs, half, first + wb, c);
  }
#pragma unroll
  for (int i = 0; i < NP; ++i) {
    add_bias(v[i], a.r.vb == nullptr ? nullptr : a.r.vb + kh * HD, 8 * c, 8 * c + 4);
    if (min(r + RP * i, within) >= w0) {  // (a staging row is a produced one)
      add_bias(k[i], kb, 4 * c, half + 4 * c);
      if (a.r.cs != nullptr) rope_piece(k[i], t[i]);
    }
  }
  // ---- K: channel maxima over the group's rows that are not sinks
  float m[8];
#pragma unroll
  for (int e = 0; e < 8; ++e) m[e] = 0.0f;
#pragma unroll
  for (int i = 0; i < NP; ++i)
    if (r + RP * i >= ws && r + RP * i <= within) {
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        m[e] = max_f(m[e], fabsf(k[i].lo[e]));
        m[4 + e] = max_f(m[4 + e], fabsf(k[i].hi[e]));
      }
    }
#pragma unroll
  for (int off = LPR; off < 64; off <<= 1)
#pragma unroll
    for (int e = 0; e < 8; ++e) m[e] = max_f(m[e], __shfl_xor(m[e], off));
  if ((tid & 63) < LPR) {
#pragma unroll
    for (int e = 0; e < 8; ++e) s_max[tid >> 6][e < 4 ? 4 * c + e : half + 4 * c + e - 4] = m[e];
  }
  // ---- V: block scales and codes; sinks as they are
#pragma unroll
  for (int i = 0; i < NP; ++i) {
    const int w = r + RP * i, pos = first + w;
    const bool batch = w >= w0 && w <= within;
    float b = 0.0f;
#pragma unroll
    for (int e = 0; e < 4; ++e) b = max_f(max_f(b, fabsf(v[i].lo[e])), fabsf(v[i].hi[e]));
    b = max_f(b, __shfl_xor(b, 1));  // the 4 lanes of a 32-channel block
    b = max_f(b, __shfl_xor(b, 2));
    if (!batch) continue;
    if (w < ws) {
      const size_t row = (head * g.n_sink + pos) * HD;
      *reinterpret_cast<f4a*>(s.k_sink + row + 4 * c) = k[i].lo;
      *reinterpret_cast<f4a*>(s.k_sink + row + half + 4 * c) = k[i].hi;
      *reinterpret_cast<f4a*>(s.v_sink + row + 8 * c) = v[i].lo;
      *reinterpret_cast<f4a*>(s.v_sink + row + 8 * c + 4) = v[i].hi;
      continue;
    }
    const float sc = b / 127.0f;
    const float inv = sc > 0.0f ? 1.0f / sc : 0.0f;
    if ((c & 3) == 0) s.v_scale[(head * g.capg + pos) * g.nb + (c >> 2)] = sc;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      s_v[v_off_i8d(HD, w, 8 * c + e)] = quant_code(v[i].lo[e], inv);
      s_v[v_off_i8d(HD, w, 8 * c + 4 + e)] = quant_code(v[i].hi[e], inv);
    }
  }
  __syncthreads();  // s_max; the staging rows are read
#pragma unroll
  for (int e = 0; e < 8; ++e) {
    const int ch = e < 4 ? 4 * c + e : half + 4 * c + e - 4;
    float x = s_max[0][ch];
#pragma unroll
    for (int i = 1; i < kRowThreads / 64; ++i) x = max_f(x, s_max[i][ch]);
    m[e] = x / 127.0f;
  }
  if (r == 0) {
    float* ks = s.k_scale + (head * g.ngroups + grp) * HD;
    *reinterpret_cast<f4a*>(ks + 4 * c) = f4a{m[0], m[1], m[2], m[3]};
    *reinterpret_cast<f4a*>(ks + half + 4 * c) = f4a{m[4], m[5], m[6], m[7]};
  }
#pragma unroll
  for (int e = 0; e < 8; ++e) m[e] = m[e] > 0.0f ? 1.0f / m[e] : 0.0f;
#pragma unroll
  for (int i = 0; i < NP; ++i) {
    const int w = r + RP * i;
    char4 lo, hi;
    lo.x = quant_code(k[i].lo[0], m[0]);
    lo.y = quant_code(k[i].lo[1], m[1]);
    lo.z = quant_code(k[i].lo[2], m[2]);
    lo.w = quant_code(k[i].lo[3], m[3]);
    hi.x = quant_code(k[i].hi[0], m[4]);
    hi.y = quant_code(k[i].hi[1], m[5]);
    hi.z = quant_code(k[i].hi[2], m[6]);
    hi.w = quant_code(k[i].hi[3], m[7]);
    *reinterpret_cast<char4*>(s_k + k_off_i8d(HD, w, 4 * c)) = lo;
    *reinterpret_cast<char4*>(s_k + k_off_i8d(HD, w, half + 4 * c)) = hi;
  }
  __syncthreads();
  int8_t* k8 = s.k8 + head * head_elems(g) + static_cast<size_t>(grp) * CH;
  int8_t* v8 = s.v8 + head * head_elems(g) + static_cast<size_t>(grp) * CH;
  const int vlo = max(w0, ws);
  if (within == kKGroup - 1 && ws == 0) {  // every K row of the group
    for (int i = tid; i < CH / 16; i += kRowThreads)
      reinterpret_cast<f4a*>(k8)[i] = reinterpret_cast<const f4a*>(s_k)[i];
  } else {
    // 8 bytes: 8 channels of position 16 (granule) + (lane & 15)
    for (int i = tid; i < CH / 8; i += kRowThreads) {
      const int w = (i >> 7) / (HD / 64) * kGranule + ((i >> 1) & 15);
      if (w >= ws && w <= within) reinterpret_cast<uint2*>(k8)[i] = reinterpret_cast<const uint2*>(s_k)[i];
    }
  }
  if (within == kKGroup - 1 && vlo == 0) {
    for (int i = tid; i < CH / 16; i += kRowThreads)
      reinterpret_cast<f4a*>(v8)[i] = reinterpret_cast<const f4a*>(s_v)[i];
  } else {
    // 4 bytes: a channel of positions w .. w + 3
#pragma unroll
    for (int i = tid; i < CH / 4; i += kRowThreads) {
      const int w = 16 * (i & 1) + 4 * ((i >> 6) & 3);
      if (w + 3 < vlo || w > within) continue;
      const uint32_t x = reinterpret_cast<const uint32_t*>(s_v)[i];
      if (w >= vlo && w + 3 <= within) {
        reinterpret_cast<uint32_t*>(v8)[i] = x;
      } else {
#pragma unroll
        for (int j = 0; j < 4; ++j)
          if (w + j >= vlo && w + j <= within) v8[4 * i + j] = static_cast<int8_t>(x >> (8 * j));
      }
    }
  }
  // ---- the staging rows after the batch
  if (gi != 0) return;
#pragma unroll
  for (int i = 0; i < NP; ++i) {
    const int w = r + RP * i;
    Piece x = k[i];
    if (n_groups > 1) {
      const int last = end - 1, p = last - ((last - w) & (kKGroup - 1));
      if (p < a.pos0) continue;
      x = key_row(p);
    } else if (w < w0 || w > within) {
      continue;
    }
    *reinterpret_cast<f4a*>(raw + static_cast<size_t>(w) * P + 4 * c) = x.lo;
    *reinterpret_cast<f4a*>(raw + static_cast<size_t>(w) * P + half + 4 * c) = x.hi;
  }
}

template <int HD>
hipError_t launch_rows(const KvGeom& g, const KvStore& s, const RowsArgs& a, hipStream_t st) {
  constexpr int LPR = HD / 8;
  const size_t qp = a.r.q == nullptr ? 0 : static_cast<size_t>(a.n) * a.r.n_heads * LPR;
  auto blocks = [](size_t w) { return static_cast<unsigned>((w + kRowThreads - 1) / kRowThreads); };
  if (!g.int8) {
    const size_t kvp = static_cast<size_t>(a.n) * 2 * g.nkv * LPR;
    hipLaunchKernelGGL(rows_f32_kernel<HD>, dim3(blocks(kvp + qp)), dim3(kRowThreads), 0, st, g, s, a);
  } else {
    const int n_groups = (a.pos0 + a.n - 1) / kKGroup - a.pos0 / kKGroup + 1;
    if (n_groups > 65535) return hipErrorInvalidValue;
    hipLaunchKernelGGL(rows_i8_kernel<HD>, dim3(n_groups * g.nkv + blocks(qp)), dim3(kRowThreads), 0, st,
                       g, s, a, n_groups);
  }
  return hipGetLastError();
}

}  // namespace

hipError_t launch_append_rows(const KvGeom& g, const KvStore& s, int layer, int pos0, int n,
                              const AppendRows& r, hipStream_t st) {
  if (g.ring || !g.tiled) return hipErrorNotSupported;
  if (n <= 0) return hipSuccess;
  const RowsArgs a{r, layer, pos0, n};
  return g.hd == 64 ? launch_rows<64>(g, s, a, st) : launch_rows<128>(g, s, a, st);
}

hipError_t launch_append(const KvGeom& g, const KvStore& s, int layer, int pos0, int n,
                         const float* k, const float* v, hipStream_t st) {
  if (n <= 0) return hipSuccess;
  if (!g.ring && g.tiled) {
    AppendRows r{};
    r.k = k;
    r.v = v;
    return launch_append_rows(g, s, layer, pos0, n, r, st);
  }
  const size_t P = static_cast<size_t>(g.nkv) * g.hd;
  if (!g.int8) {
    hipLaunchKernelGGL(append_f32_kernel, dim3(grid_for(n * P)), dim3(kThreads), 0, st, g, s.k,
                       s.v, layer, pos0, n, k, v);
  } else if (g.ring) {
    const size_t lanes = static_cast<size_t>(n) * g.nkv * g.nb * kBlock;
    hipLaunchKernelGGL(append_i8_ring_kernel, dim3((lanes + kThreads - 1) / kThreads),
                       dim3(kThreads), 0, st, g, s, layer, pos0, n, k, v);
  } else {
    const int n_groups = (pos0 + n - 1) / kKGroup - pos0 / kKGroup + 1;
    if (n_groups > 65535) return hipErrorInvalidValue;
    hipLaunchKernelGGL(append_i8_kgroup_kernel,
                       dim3(static_cast<unsigned>((P + kThreads - 1) / kThreads), n_groups),
                       dim3(kThreads), 0, st, g, s, layer, pos0, n, k);
    hipLaunchKernelGGL(append_i8_kraw_kernel, dim3(grid_for(kKGroup * P)), dim3(kThreads), 0, st, g,
                       s, layer, pos0, n, k);
    const size_t vwork = static_cast<size_t>(n) * g.nkv * g.nb * kBlock;
    hipLaunchKernelGGL(append_i8_dense_v_kernel, dim3((vwork + kThreads - 1) / kThreads),
                       dim3(kThreads), 0, st, g, s, layer, pos0, n, k, v);
  }
  return hipGetLastError();
}

hipError_t launch_prefix_pack(const KvGeom& g, const float* src_store, float* dst, int len,
                              bool is_k, hipStream_t st) {
  const size_t total = static_cast<size_t>(g.n_layers) * len * g.nkv * g.hd;
  hipLaunchKernelGGL(prefix_pack_kernel<float>, dim3(grid_for(total)), dim3(kThreads), 0, st, g,
                     src_store, dst, len, 0, is_k ? 1 : 0);
  return hipGetLastError();
}

hipError_t launch_prefix_unpack(const KvGeom& g, const float* src, float* dst_store, int len,
                                bool is_k, hipStream_t st) {
  const size_t total = static_cast<size_t>(g.n_layers) * len * g.nkv * g.hd;
  hipLaunchKernelGGL(prefix_pack_kernel<float>, dim3(grid_for(total)), dim3(kThreads), 0, st, g,
                     dst_store, const_cast<float*>(src), len, 1, is_k ? 1 : 0);
  return hipGetLastError();
}

hipError_t launch_prefix_codes(const KvGeom& g, int8_t* store, int8_t* file, int len, bool is_k,
                               bool unpack, hipStream_t st) {
  const size_t total = static_cast<size_t>(g.n_layers) * len * g.nkv * g.hd;
  if (total == 0) return hipSuccess;
  hipLaunchKernelGGL(prefix_pack_kernel<uint8_t>, dim3(grid_for(total)), dim3(kThreads), 0, st,
                     g, reinterpret_cast<const uint8_t*>(store),
                     reinterpret_cast<uint8_t*>(file), len, unpack ? 1 : 0, is_k ? 1 : 0);
  return hipGetLastError();
}

hipError_t launch_rows_pack(float* store, float* file, int n_layers, int nkv, int dev_rows,
                            int rows, int inner, bool unpack, hipStream_t st) {
  const size_t total = static_cast<size_t>(n_layers) * rows * nkv * inner;
  if (total == 0) return hipSuccess;
  hipLaunchKernelGGL(rows_pack_kernel, dim3(grid_for(total)), dim3(kThreads), 0, st, store, file,
                     n_layers, nkv, dev_rows, rows, inner, unpack ? 1 : 0);
  return hipGetLastError();
}

}  // namespace dbi
