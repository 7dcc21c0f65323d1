// Causal chunk attention of the dense caches on the matrix cores: the
// attention loop of decode_layer_chunk (model.cpp:956-981), rows c of a
// chunk at pos0 attending keys [0, pos0 + c], for chunks long enough to
// make QK^T and PV real matrix products (the prefill chunks of config 2).
//
// Design (CDNA4 v_mfma_f32_32x32x16_bf16 over exact three-part splits of the
// fp32 operands, bf16x3.hpp, so the result stays within the fp32 tolerance
// of the CPU path):
//  - A workgroup of 8 waves (one per CU) owns 256 query vectors of one kv
//    head: each wave 32 columns, 32/G rows x the G query heads sharing the
//    kv head (32 mod G padding columns compute and write nothing of use).
//  - The workgroup walks its keys in stages of 32. Staging: a stage's fp32 K
//    and V are loaded into registers ahead of their use, split once per
//    workgroup into hi, mid and lo bf16 parts and written to LDS in the
//    matrix cores' operand layout: every operand read of the waves is one
//    16-byte LDS load of 8 bf16, and no wave converts K or V itself.
//  - Two groups of four waves (one wave of each per SIMD) work half a stage
//    apart: while one group is in its matrix phase (PV of the stage before,
//    then QK^T of this one), the other is in its vector phase (softmax and
//    the splits of its staging share: waves 0-3 K, waves 4-7 V), with a
//    barrier between the phases. A SIMD's two waves then never want the same
//    unit at once. What bounds a stage is the matrix phase: 48 instructions
//    of 32 cycles at hd 64 (96 at hd 128) against ~270 vector instructions of
//    4 cycles, two waves per SIMD.
//    Measured against 16-column waves in lockstep (v_mfma_f32_16x16x32_bf16,
//    both groups in the same phase): 256 rows of 32 query
//    heads over 8 at 1792 keys 33.8 -> 31.5 us at hd 64, 55.9 -> 51.3 at hd
//    128; at 7936 110 -> 91 and 181 -> 159; 1000 rows of 28 heads over 4 from
//    position 0 (hd 128) 89.9 -> 59.5. In a long run of calls the chip's clock
//    sinks to about 1.5 GHz under the products of hd 128 (the matrix units
//    busy 90 % of the time then), which is what a large bf16 matrix product
//    reaches too (1.3 PFLOP/s).
//  - Dense int8: the staging dequantizes, k = fp32(code * scale) per channel
//    and v = fp32(code * scale) per 32-channel block, and takes the fp32 sinks
//    for positions < n_sink; everything after it is the fp32 kernel. One fp32
//    rounding of code * scale stands where attend_dense_int8 (model.cpp:
//    605-660) rounds q * scale and weight * scale, so the error against 64
//    bits is of the same size (256 rows of 24/8 heads at 3840, hd 128: 5.8e-7,
//    7.0e-7 with the products of codes). Exact products of codes would halve
//    the matrix work, but need the query scaled and split per 32-key group,
//    about 300 vector instructions per stage and 16 vectors, which is what
//    bounds the rows kernel (that chunk 98 us there, 81 here).
//  - Key splits: the row blocks' stages are dealt to workgroups of at most T
//    stages each, T the smallest that needs at most one workgroup per CU
//    (prefill_plan), so a causal chunk's longer row blocks get more of them.
//    A split writes its unnormalized (o, m, l) and prefill_merge combines
//    them.
//  - S^T = K Q^T: A = K (32 keys x 16 dims), B = Q^T (16 dims x 32 vectors),
//    six bf16 products per 16-dim step. In k-step ks, lane half h's k-index
//    e stands for dim 16 ks + 8 h + e. The result holds S[vector l % 32]
//    [key 8 (i / 4) + 4 h + i % 4] in element i of lane l = vector + 32 h.
//  - O^T += V^T P^T over the stage's 32 keys in two k-steps of 16: B = P^T
//    straight from the score registers (elements 8 kk .. 8 kk + 7 of k-step
//    kk), A = V^T in the same key order. Output tile t row 8 q + 4 h + j
//    stands for dim h HD/2 + 16 NU (t / NU) + (4 q + j) NU + t % NU, NU =
//    HD/64: a lane's output is HD/2 contiguous floats of its vector.
//  - Online softmax per vector (= per lane % 32) with a lazy reference
//    maximum; the two lane halves holding one vector combine through one lane
//    swap (the maximum per stage, the sum once at the end).
#include <cmath>

#include "bf16x3.hpp"
#include "kv_internal.hpp"

namespace dbi {
namespace {

using f32x16 = float __attribute__((ext_vector_type(16)));

constexpr int kPWaves = 8;
constexpr int kPThreads = 64 * kPWaves;
constexpr int kPVec = 32 * kPWaves;        // query vectors per workgroup
constexpr float kLog2eP = 1.4426950408889634f;
constexpr float kMinitP = -1.0e30f;  // finite: exp2(kMinit - kMinit) == 1
constexpr float kLazyLog2 = 8.0f;    // weights relative to the running maximum: at most 2^8

// Workgroups of one kv head: item i of a split launch is split (i >> 16) & 255
// of (i >> 24) of row block i & 0xffff; the splits of a block are neighbours,
// longer blocks come first.
constexpr int kMaxItems = kPrefillBlocks;
struct PrefillParams {
  const float* kf;  // this layer's K, V: [nkv][capg * hd], granule layout
  const float* vf;
  // dense int8: codes [nkv][capg * hd] in the matrix-core layout, K channel
  // scales [nkv][ng][hd], V block scales [nkv][capg][hd / 32], sinks
  // [nkv][n_sink][hd]
  const int8_t* k8;
  const int8_t* v8;
  const float* ks;
  const float* vs;
  const float* ksink;
  const float* vsink;
  int ng, n_sink;
  const float* q;   // [rows][n_heads][hd]
  float* out;       // [rows][n_heads][hd]
  float* part;      // split records, one region of record_floats per workgroup
  int capg, nkv, n_heads, rows, pos0;
  int rpv;                 // rows per wave
  int n_blocks, n_items;   // (n_items 0: one item per block)
  float qscale;            // scale * log2(e)
  uint32_t item[kMaxItems];
  uint16_t first[kMaxItems];  // a row block's first item
};

// one workgroup's record: o [256 vectors][HD], then (m, l) [256][2]
template <int HD>
__host__ __device__ constexpr size_t prefill_record() {
  return static_cast<size_t>(kPVec) * (HD + 2);
}

// Workgroup barrier after this wave's LDS accesses have completed.
__device__ __forceinline__ void lds_barrier() {
  asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
}

// Exchange between the lane halves through the gfx950 permlane swap (VALU, no
// LDS round trip like a bpermute). After v_permlane32_swap of (x, x), a lane
// holds its own x and the x of lane ^ 32, one in each register. Emitted
// through asm: the compiler's builtin folds the two results into one when
// both are used. The maximum is taken inside the asm too: fmaxf on asm
// results costs two NaN-quieting v_max of its operands first.
__device__ __forceinline__ float xmax32(float x) {
  float a = x, b = x;
  asm("s_nop 1\n\tv_permlane32_swap_b32 %0, %1\n\ts_nop 0\n\tv_max_f32 %0, %0, %1"
      : "+v"(a), "+v"(b));
  return a;
}
__device__ __forceinline__ float xsum32(float x) {
  float a = x, b = x;
  asm("s_nop 1\n\tv_permlane32_swap_b32 %0, %1" : "+v"(a), "+v"(b));
  return a + b;
}

// One stage in LDS: parts p = 0, 1, 2 (hi, mid, lo) of K or of V, each a
// plane of SK x HD bf16; two buffers of each.
//  - K plane: key k's dims 8 u .. 8 u + 7 are the 16-byte unit
//    k * HD/8 + (u ^ kswz(k)). The swizzle puts the 8 (16) keys of one
//    operand read's 8-lane (16-lane) group on distinct banks of 128 (256)
//    bytes.
//  - V plane: unit (2 kk + h) * HD + s holds keys 16 kk + 4 h + {0..3, 8..11}
//    (k-step kk, lane half h) of the dim of output row s (vdim): lane i of
//    output tile t reads s = 32 t + i, 32 contiguous units.
template <int HD>
struct Stage {
  static constexpr int SK = 32;                   // keys per stage
  static constexpr int UPR = HD / 8;              // 16-byte units per key of a K part
  static constexpr int PLANE = SK * HD * 2;       // bytes of one part of K or V
  static constexpr int BUF = 3 * PLANE;           // K or V of one stage
  static constexpr int STG = kPThreads / 2;       // staging lanes of K (and of V)
  static constexpr int NU = SK * HD / 8 / STG;    // staging lane: K units, or V dims
};

template <int HD>
__host__ __device__ constexpr int kswz(int key) {
  return HD == 64 ? ((key & 7) ^ ((key >> 3) & 1)) : (key & 15);
}

__device__ __forceinline__ f32x16 mfma32(const uint4& a, const uint4& b, const f32x16& c) {
  return __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, a),
                                                 __builtin_bit_cast(bf16x8, b), c, 0, 0, 0);
}

template <int HD, bool I8>
__global__ __launch_bounds__(kPThreads) __attribute__((amdgpu_waves_per_eu(2, 2))) void prefill_kernel(const PrefillParams P) {
  using S = Stage<HD>;
  constexpr int SK = S::SK, UPR = S::UPR, PLANE = S::PLANE, BUF = S::BUF, NU = S::NU;
  constexpr int KS = HD / 16;    // k-steps of QK^T
  constexpr int NT = HD / 32;    // output tiles
  static_assert(NU == 1 || NU == 2, "staging shapes");
  // the split q: hd 64 keeps its three parts in registers; at hd 128 the
  // third part (32 registers, of 256) sits in LDS, each lane's own
  constexpr int QR = HD == 64 ? 3 : 2;
  // K of even, odd stages; V of even, odd. Before and after the stages: a
  // wave's own [32 vectors][64 dims] of q or of the output on the way between
  // global rows (whole lines) and lanes (a vector each); rows padded by 16
  // bytes, so that 16 lanes' pieces of 16 rows fall in distinct banks.
  constexpr int XROW = 64 * 4 + 16, XTILE = 32 * XROW;
  __shared__ __align__(16) char s_stage[4 * BUF > kPWaves * XTILE ? 4 * BUF : kPWaves * XTILE];
  __shared__ uint4 s_qlo[QR == 2 ? KS * kPThreads : 1];
  auto kbuf = [&](int b) { return s_stage + b * BUF; };
  auto vbuf = [&](int b) { return s_stage + (2 + b) * BUF; };

  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int h = lane >> 5;       // lane half
  const int vec = lane & 31;     // query vector of this lane
  // kv heads innermost: workgroups go to the 8 XCDs round-robin by linear id,
  // so with 8 kv heads every row block and split of one head runs on one XCD,
  // and that XCD's L2 serves the head's K/V to all of them
  const int kh = static_cast<int>(blockIdx.x) % P.nkv;
  const int it = static_cast<int>(blockIdx.x) / P.nkv;
  int rb = P.n_blocks - 1 - it, z = 0, nz = 1;  // longest blocks first
  if (P.n_items > 0) {
    const uint32_t w = P.item[it];
    rb = static_cast<int>(w & 0xffffu);
    z = static_cast<int>((w >> 16) & 0xffu);
    nz = static_cast<int>(w >> 24);
  }
  const int G = P.n_heads / P.nkv, RPV = P.rpv;       // rows per wave
  const int rowb = rb * (kPWaves * RPV);              // first row of the workgroup
  const int row0 = rowb + wave * RPV;                 // first row of the wave
  const bool wave_live = row0 < P.rows;               // wave-uniform
  const int vrow = vec / G;
  // (a padding column repeats the wave's last row; it writes nothing)
  const int row = min(row0 + min(vrow, RPV - 1), P.rows - 1);
  const int limit = P.pos0 + row;  // last key of this vector
  // the workgroup's keys [0, last_key], in stages; split z takes its share
  const int last_key = P.pos0 + min(rowb + kPWaves * RPV - 1, P.rows - 1);
  const int n_stages = last_key / SK + 1;
  const int st0 = n_stages * z / nz;
  const int n = n_stages * (z + 1) / nz - st0;        // (>= 1: nz <= n_stages)
  const int wave_last = P.pos0 + min(row0 + RPV - 1, P.rows - 1);  // wave-uniform

  const size_t head_el = static_cast<size_t>(kh) * P.capg * HD;

  // ---- staging. K lanes (the first half of the waves, t < STG): units
  // u = t + STG m, key u / UPR, dims 8 (u % UPR) .. + 7 (two float4 of the
  // granule layout). V lanes (t = STG + 64 kq + c): the 8 keys of (k-step,
  // lane half) kq = 2 kk + h and the NU dims of output rows
  // s = 32 (NU (c / 32) + m) + c % 32, consecutive in memory. The source
  // offsets of stage 0 (stage st adds st * SK * HD: a stage is two whole
  // granules).
  const bool k_stager = wave < kPWaves / 2;  // uniform
  // One source and one destination offset per lane; the rest of a lane's
  // pieces sit at constant distances. K: the second float4 of a unit 16 bytes
  // on, unit m's key 16 m keys on (a granule: 16 HD floats; 16 UPR units in
  // LDS, its swizzle the same). V: key e's dims (e & 3) row pieces of 16
  // bytes x HD/8 and (e >> 2) times 8 keys of a granule (1024 / (HD/64) floats
  // x NU = HD/64: 32 HD bytes) on; output row m 32 units.
  // int8: K: a unit is 8 consecutive bytes, unit m one granule (16 HD bytes)
  // on, its 8 channel scales shared; V: a dim's keys 0..3 are 4 bytes, keys
  // 8..11 512 bytes on, the next dim 16 bytes on; scl the scale of the first
  // key, HD/32 floats apart.
  uint32_t src, dst, scl = 0;
  int vd = 0;  // V: the lane's first dim
  const int kq = (wave - kPWaves / 2) & 3;              // V: k-step and lane half
  const int vkey0 = 16 * (kq >> 1) + 4 * (kq & 1);      // V: keys vkey0 + {0..3, 8..11}
  if (k_stager) {
    const int key = static_cast<int>(threadIdx.x) / UPR, u = static_cast<int>(threadIdx.x) % UPR;
    src = I8 ? static_cast<uint32_t>(k_off_i8d(HD, key, 8 * u))
             : static_cast<uint32_t>(k_off_tiled(HD, false, key, 8 * u)) * 4u;
    scl = 8u * u * 4u;
    dst = static_cast<uint32_t>((key * UPR + (u ^ kswz<HD>(key))) * 16);
  } else {
    const int c = lane, r5 = c & 31;
    const int d = ((r5 >> 2) & 1) * (HD / 2) + (c >> 5) * 16 * NU + (4 * (r5 >> 3) + (r5 & 3)) * NU;
    src = I8 ? static_cast<uint32_t>(v_off_i8d(HD, vkey0, d))
             : static_cast<uint32_t>(v_off_tiled(HD, false, vkey0, d)) * 4u;
    scl = static_cast<uint32_t>(vkey0 * (HD / kBlock) + d / kBlock) * 4u;
    vd = d;
    dst = static_cast<uint32_t>((kq * HD + 32 * NU * (c >> 5) + r5) * 16);
  }
  constexpr int KDST = 16 * UPR * 16, VDST = 32 * 16;
  // the loaded stage: K lanes hold unit m in r[2 m], r[2 m + 1]; V lanes key
  // e's dim in component e % 4 of r[e / 4] (NU = 1) or its two dims in half
  // e % 2 of r[e / 2] (NU = 2). int8: the codes, and 8 scales in r.
  float4 r[I8 ? 2 : 2 * NU];
  uint32_t code[I8 ? 2 * NU : 1];
  auto rsrc = [&](const void* at, int bytes) {
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(at), static_cast<short>(0), bytes,
                                             0x00020000);
  };
  auto load_codes = [&](int st) {
    const auto rc = rsrc((k_stager ? P.k8 : P.v8) + head_el + static_cast<size_t>(st) * SK * HD, SK * HD);
    if (k_stager) {
#pragma unroll
      for (int m = 0; m < NU; ++m) {
        const uint2 w = __builtin_bit_cast(
            uint2, __builtin_amdgcn_raw_buffer_load_b64(rc, src, m * 16 * HD, 0));
        code[2 * m] = w.x;
        code[2 * m + 1] = w.y;
      }
      const auto rs = rsrc(P.ks + (static_cast<size_t>(kh) * P.ng + st) * HD, HD * 4);
#pragma unroll
      for (int i = 0; i < 2; ++i)
        r[i] = __builtin_bit_cast(float4, __builtin_amdgcn_raw_buffer_load_b128(rs, scl + 16 * i, 0, 0));
    } else {
#pragma unroll
      for (int m = 0; m < NU; ++m)
#pragma unroll
        for (int i = 0; i < 2; ++i)
          code[2 * m + i] = __builtin_amdgcn_raw_buffer_load_b32(rc, src + 16 * m + 512 * i, 0, 0);
      constexpr int NBK = HD / kBlock;
      const auto rs = rsrc(P.vs + (static_cast<size_t>(kh) * P.capg + st * SK) * NBK, SK * NBK * 4);
#pragma unroll
      for (int e = 0; e < 8; e += 4) {
        float x[4];
#pragma unroll
        for (int i = 0; i < 4; ++i)
          x[i] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(
                                               rs, scl + (i + 2 * e) * NBK * 4, 0, 0));
        r[e / 4] = make_float4(x[0], x[1], x[2], x[3]);
      }
    }
  };
  auto load_stage = [&](int st) {
    if constexpr (I8) {
      load_codes(st);
      return;
    }
    const auto rs = rsrc((k_stager ? P.kf : P.vf) + head_el + static_cast<size_t>(st) * SK * HD, SK * HD * 4);
    if (k_stager) {
#pragma unroll
      for (int i = 0; i < (I8 ? 0 : 2 * NU); ++i)
        r[i] = __builtin_bit_cast(float4, __builtin_amdgcn_raw_buffer_load_b128(
                                              rs, src + (i & 1) * 16, (i >> 1) * 16 * HD * 4, 0));
    } else {
      constexpr int RP = HD / 8 * 16, GP = 32 * HD;  // bytes to the next key, to 8 keys on
      auto off = [](int e) { return (e & 3) * RP; };
      if constexpr (NU == 1) {
#pragma unroll
        for (int e = 0; e < 8; e += 4) {
          float x[4];
#pragma unroll
          for (int i = 0; i < 4; ++i)
            x[i] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(
                                                 rs, src + off(e + i), (e >> 2) * GP, 0));
          r[e / 4] = make_float4(x[0], x[1], x[2], x[3]);
        }
      } else {
#pragma unroll
        for (int e = 0; e < 8; e += 2) {
          const float2 a = __builtin_bit_cast(
              float2, __builtin_amdgcn_raw_buffer_load_b64(rs, src + off(e), (e >> 2) * GP, 0));
          const float2 b = __builtin_bit_cast(
              float2, __builtin_amdgcn_raw_buffer_load_b64(rs, src + off(e + 1), (e >> 2) * GP, 0));
          r[e / 2] = make_float4(a.x, a.y, b.x, b.y);
        }
      }
    }
  };
  auto at4 = [](const float4& x, int i) { return i == 0 ? x.x : i == 1 ? x.y : i == 2 ? x.z : x.w; };
  // value e of piece m: element e of K unit m, or key e of V dim m
  auto value = [&](int e, int m) -> float {
    if constexpr (I8) {
      // (code + 128) * scale - 128 * scale, rounded once: fp32(code * scale)
      const float sc8 = at4(r[e / 4], e % 4);
      const uint32_t w = code[2 * m + e / 4] ^ 0x80808080u;
      return fmaf(static_cast<float>((w >> (8 * (e % 4))) & 0xFFu), sc8, -128.0f * sc8);
    } else if (k_stager || NU == 1) {
      return at4(r[2 * m + e / 4], e % 4);
    } else {
      return at4(r[e / 2], 2 * (e & 1) + m);
    }
  };
  // int8: the fp32 sinks of stage st (keys < n_sink) over the lane's own
  // stored pieces, one value at a time
  auto put_sinks = [&](int st, int b) {
    auto put = [&](char* at, float x) {
      const uint32_t hi = fbits(x) & 0xFFFF0000u;
      const float e = x - ffrom(hi);
      const uint32_t mid = fbits(e) & 0xFFFF0000u;
      const uint32_t part[3] = {hi, mid, fbits(e - ffrom(mid))};
#pragma unroll
      for (int p = 0; p < 3; ++p)
        *reinterpret_cast<uint16_t*>(at + p * PLANE) = static_cast<uint16_t>(part[p] >> 16);
    };
    const int t = static_cast<int>(threadIdx.x);
#pragma unroll 1
    for (int i = 0; i < 8 * NU; ++i) {
      const int m = i >> 3, e = i & 7;
      const int key = st * SK + (k_stager ? t / UPR + 16 * m : vkey0 + (e & 3) + 8 * (e >> 2));
      if (key >= P.n_sink || key > last_key) continue;
      const float* row = (k_stager ? P.ksink : P.vsink) + (static_cast<size_t>(kh) * P.n_sink + key) * HD;
      put((k_stager ? kbuf(b) + m * KDST : vbuf(b) + m * VDST) + dst + 2 * e,
          row[k_stager ? 8 * (t % UPR) + e : vd + m]);
    }
  };
  // split and store stage st into buffer b; V of keys past the workgroup's
  // last key is stored as 0 (its weight is 0, and the cache past the chunk
  // may hold anything)
  auto store_stage = [&](int st, int b) {
    const int key0 = st * SK;
    if (k_stager) {
      char* sb = kbuf(b);
#pragma unroll
      for (int m = 0; m < NU; ++m) {
        float x[8];
#pragma unroll
        for (int e = 0; e < 8; ++e) x[e] = value(e, m);
        uint4 part[3];
        split3(x, part);
#pragma unroll
        for (int p = 0; p < 3; ++p) *reinterpret_cast<uint4*>(sb + p * PLANE + m * KDST + dst) = part[p];
      }
    } else {
      char* sb = vbuf(b);
      const bool tail = key0 + SK - 1 > last_key;  // uniform
#pragma unroll
      for (int m = 0; m < NU; ++m) {
        float x[8];
#pragma unroll
        for (int e = 0; e < 8; ++e) {
          const float v = value(e, m);
          x[e] = !tail || key0 + vkey0 + (e & 3) + 8 * (e >> 2) <= last_key ? v : 0.0f;
        }
        uint4 part[3];
        split3(x, part);
#pragma unroll
        for (int p = 0; p < 3; ++p) *reinterpret_cast<uint4*>(sb + p * PLANE + m * VDST + dst) = part[p];
      }
    }
    if (I8 && key0 < P.n_sink) put_sinks(st, b);  // uniform; rare
  };

  // ---- Q^T: dims 16 ks + 8 h + e of k-step ks, pre-scaled into the log2
  // domain, in three bf16 parts. A vector's row comes in whole lines through
  // the wave's LDS tile, 64 dims at a time: loaded by each lane from its own
  // vector's row, 16 bytes an instruction, the 128 KB of a workgroup took
  // 12 500 cycles at hd 128 (5 300 at hd 64).
  char* const xt = s_stage + wave * XTILE;
  load_stage(st0);
  uint4 qp[KS][QR];
  {
    float4 qv[HD / 64][8];
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      const int v = 4 * i + (lane >> 4);  // lanes 16 j .. 16 j + 15: vector 4 i + j
      const int vr = v / G;
      const int rv = min(row0 + min(vr, RPV - 1), P.rows - 1);
      const float* qs = P.q + (static_cast<size_t>(rv) * P.n_heads + kh * G + (v - vr * G)) * HD;
#pragma unroll
      for (int c = 0; c < HD / 64; ++c)
        qv[c][i] = *reinterpret_cast<const float4*>(qs + 64 * c + 4 * (lane & 15));
    }
#pragma unroll
    for (int c = 0; c < HD / 64; ++c) {
#pragma unroll
      for (int i = 0; i < 8; ++i)
        *reinterpret_cast<f32x4*>(xt + (4 * i + (lane >> 4)) * XROW + (lane & 15) * 16) =
            __builtin_bit_cast(f32x4, qv[c][i]);
      // (the wave's own tile: its LDS accesses complete in order)
#pragma unroll
      for (int k4 = 0; k4 < 4; ++k4) {
        const int ks = 4 * c + k4;
        const f32x4 a = *reinterpret_cast<const f32x4*>(xt + vec * XROW + (16 * k4 + 8 * h) * 4);
        const f32x4 b = *reinterpret_cast<const f32x4*>(xt + vec * XROW + (16 * k4 + 8 * h) * 4 + 16);
        const float x[8] = {a.x * P.qscale, a.y * P.qscale, a.z * P.qscale, a.w * P.qscale,
                            b.x * P.qscale, b.y * P.qscale, b.z * P.qscale, b.w * P.qscale};
        uint4 part[3];
        split3(x, part);
#pragma unroll
        for (int p = 0; p < QR; ++p) qp[ks][p] = part[p];
        if constexpr (QR == 2) s_qlo[ks * kPThreads + threadIdx.x] = part[2];
      }
    }
    lds_barrier();  // the tiles are done with: stage 0 goes there
  }
  // lane byte offsets of the K reads (k-step 0; k-step ks flips the bits of
  // 2 ks units) and V reads (output tile 0) within a part plane
  const int klo = (vec * UPR + (h ^ kswz<HD>(vec))) * 16;
  const int vlo = (h * HD + vec) * 16;

  f32x16 acc[NT];
#pragma unroll
  for (int t = 0; t < NT; ++t) acc[t] = f32x16{};
  float m_run = kMinitP, l_run = 0.0f;  // (l: this lane half's keys)

  // a b = sum of a_i b_j over the parts; the six terms with i + j <= 2 are
  // kept (the dropped ones are below 2^-23 |a b|, the size of the fp32
  // rounding the reference's own sums carry). hi accumulates a_0 b_0, lo the
  // five small terms. Each part of a is read again, for the next group of
  // six, as soon as its last product is issued: its LDS latency passes under
  // the three to five products (32 cycles each) until its next use, in the
  // same registers. Left to the compiler, the reads sat right before their
  // use: 2.38 us per stage and workgroup at hd 64 (4.56 at hd 128), of which
  // the products are 1.50 (3.00).
  uint4 a3[3];
  auto read3 = [&](const char* at, int p) {
    a3[p] = *reinterpret_cast<const uint4*>(at + p * PLANE);
  };
  auto group = [&](const uint4& b0, const uint4& b1, const uint4& b2, f32x16& hi, f32x16& lo,
                   bool more, const char* next, auto&& after_b2) {
    lo = mfma32(a3[0], b1, lo);
    hi = mfma32(a3[0], b0, hi);
    lo = mfma32(a3[0], b2, lo);
    __builtin_amdgcn_sched_barrier(0);
    if (more) read3(next, 0);
    after_b2();
    __builtin_amdgcn_sched_barrier(0);
    lo = mfma32(a3[1], b1, lo);
    lo = mfma32(a3[1], b0, lo);
    __builtin_amdgcn_sched_barrier(0);
    if (more) read3(next, 1);
    __builtin_amdgcn_sched_barrier(0);
    lo = mfma32(a3[2], b0, lo);
    __builtin_amdgcn_sched_barrier(0);
    if (more) read3(next, 2);
    __builtin_amdgcn_sched_barrier(0);
  };

  // keys every row of the wave attends, and that the workgroup holds
  const int wave_full = min(P.pos0 + row0, last_key);

  f32x16 sc;      // S^T of the stage between the wave's two phases
  uint4 pb[2][3]; // its weights, split
  // (both are entered with a3 holding their first operand; pv leaves K's)
  auto first3 = [&](const char* at) {
#pragma unroll
    for (int p = 0; p < 3; ++p) read3(at, p);
  };
  auto qlo = [&](int ks) { return s_qlo[ks * kPThreads + threadIdx.x]; };
  auto qk = [&](const char* sb) {
    // the small terms sum apart, so the large sum is rounded once per k-step
    // (six times otherwise; the 64-bit error of a C2 chunk 4.8e-7 instead of
    // 6.9e-7)
    sc = f32x16{};
    f32x16 lo = f32x16{};
    uint4 b2{};
    if constexpr (QR == 2) b2 = qlo(0);
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) {
      const bool more = ks + 1 < KS;
      const char* next = sb + (klo ^ (32 * (more ? ks + 1 : 0)));
      if constexpr (QR == 3)
        group(qp[ks][0], qp[ks][1], qp[ks][2], sc, lo, more, next, [] {});
      else
        group(qp[ks][0], qp[ks][1], b2, sc, lo, more, next, [&] {
          if (more) b2 = qlo(ks + 1);
        });
    }
    sc += lo;
  };
  auto pv = [&](const char* sb, const char* kb) {
#pragma unroll
    for (int t = 0; t < NT; ++t)
#pragma unroll
      for (int kk = 0; kk < 2; ++kk) {
        const int u = 2 * t + kk + 1;  // the next group
        const char* next = u < 2 * NT ? sb + (2 * (u & 1) * HD + 32 * (u >> 1)) * 16 + vlo : kb + klo;
        group(pb[kk][0], pb[kk][1], pb[kk][2], acc[t], acc[t], true, next, [] {});
      }
  };
  // Online softmax of a stage's 32 keys.
  auto soft = [&](int st) {
    // past some row's last key (causal diagonal, chunk tail): masked
    if (st * SK + SK - 1 > wave_full) {  // uniform
#pragma unroll
      for (int i = 0; i < 16; ++i)
        sc[i] = st * SK + 8 * (i / 4) + 4 * h + i % 4 <= limit ? sc[i] : -INFINITY;
    }
    float mx = kMinitP;
#pragma unroll
    for (int i = 0; i < 16; ++i) mx = fmaxf(mx, sc[i]);
    mx = xmax32(mx);
    // The reference maximum m_run moves only when a score passes it by more
    // than 2^kLazyLog2 (so every weight is at most 2^kLazyLog2: the splits
    // stay exact and the sums far from fp32's range), and then to the
    // stage's maximum. Otherwise alpha is exactly 1 in every lane and the
    // rescale is skipped (a rare branch, and told so: the compiler otherwise
    // moves every accumulator to other registers around it).
    const float mn = mx > m_run + kLazyLog2 ? mx : m_run;
    const float alpha = __builtin_amdgcn_exp2f(m_run - mn);
    float ls = 0.0f;
#pragma unroll
    for (int kk = 0; kk < 2; ++kk) {
      float w[8];
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        w[e] = __builtin_amdgcn_exp2f(sc[8 * kk + e] - mn);
        ls += w[e];
      }
      split3(w, pb[kk]);
    }
    l_run = l_run * alpha + ls;
    m_run = mn;
    if (__builtin_expect(__builtin_amdgcn_ballot_w64(alpha != 1.0f) != 0, 0)) {
#pragma unroll
      for (int t = 0; t < NT; ++t) acc[t] *= alpha;
    }
  };
  // the stages that reach some row of the wave (the causal tail is only staged)
  const int nl = wave_live ? min(n, max(wave_last / SK + 1 - st0, 0)) : 0;  // uniform
  // stage s + 1 into LDS, stage s + 2 requested
  auto advance = [&](int s) {
    if (s + 1 < n) store_stage(st0 + s + 1, (s & 1) ^ 1);
    if (s + 2 < n) load_stage(st0 + s + 2);
  };

  // Phases, a barrier after each. Matrix phase s: O += P V of stage s - 1, S =
  // K Q of stage s; vector phase s: staging, then the softmax of stage s.
  // Group 0 (the K stagers) runs matrix phase s in phase 2 s and vector phase
  // s in phase 2 s + 1; group 1 (the V stagers) runs one phase later. K of
  // stage s is read in phases 2 s, 2 s + 1 and written by group 0 in phase
  // 2 s - 1, when its buffer was last read two barriers before (stage s - 2:
  // phase 2 s - 3); V of stage s is read in phases 2 s + 2, 2 s + 3 (its first
  // operand at the end of the vector phase before, two barriers after its
  // store) and written by group 1 in phase 2 s, its buffer last read in phase
  // 2 s - 1. Stage 0 is staged here.
  store_stage(st0, 0);
  if (n > 1) load_stage(st0 + 1);
  lds_barrier();
  if (!k_stager) lds_barrier();
  if (nl > 0) {
    first3(kbuf(0) + klo);
    qk(kbuf(0));
  }
  lds_barrier();
#pragma unroll 1
  for (int s = 0; s < nl; ++s) {
    advance(s);
    __builtin_amdgcn_sched_barrier(0);
    soft(st0 + s);
    __builtin_amdgcn_sched_barrier(0);
    first3(vbuf(s & 1) + vlo);
    lds_barrier();
    __builtin_amdgcn_s_setprio(3);
    const char* kb = kbuf((s & 1) ^ 1);
    pv(vbuf(s & 1), kb);
    if (s + 1 < nl) qk(kb);
    __builtin_amdgcn_s_setprio(0);
    lds_barrier();
  }
#pragma unroll 1
  for (int s = nl; s < n; ++s) {
    advance(s);
    lds_barrier();
    lds_barrier();
  }
  if (k_stager) lds_barrier();

  // lane holds O^T[dims HD/2 h .. + HD/2 - 1][vec]; out through the wave's
  // tile (every wave is past its last matrix phase): whole lines of a
  // vector's row at a time
  if (!wave_live) return;
  l_run = xsum32(l_run);
  const float f = nz == 1 ? 1.0f / l_run : 1.0f;
  float* rec = P.part + blockIdx.x * prefill_record<HD>();
  int ol = lane;
  asm volatile("" : "+v"(ol));  // the rows' offsets anew: kept from q's loads they spill
  // (a tile holds dims 32 c .. + 31 of both halves of the head)
#pragma unroll
  for (int c = 0; c < HD / 64; ++c) {
#pragma unroll
    for (int i = 0; i < 32; i += 4) {
      f32x4 x;
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const int d = 32 * c + i + j;  // of the lane's HD/2 dims
        x[j] = acc[NU * (d / (16 * NU)) + d % NU][d % (16 * NU) / NU] * f;
      }
      *reinterpret_cast<f32x4*>(xt + vec * XROW + (32 * h + i) * 4) = x;
    }
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      const int v = 4 * i + (ol >> 4), d4 = ol & 15;
      const f32x4 x = *reinterpret_cast<const f32x4*>(xt + v * XROW + d4 * 16);
      const int vr = v / G, d = (d4 >> 3) * (HD / 2) + 32 * c + 4 * (d4 & 7);
      if (vr < RPV && row0 + vr < P.rows) {
        float* op = nz == 1 ? P.out + (static_cast<size_t>(row0 + vr) * P.n_heads + kh * G + (v - vr * G)) * HD
                            : rec + static_cast<size_t>(wave * 32 + v) * HD;
        *reinterpret_cast<f32x4*>(op + d) = x;
      }
    }
  }
  if (nz > 1 && h == 0)
    *reinterpret_cast<float2*>(rec + static_cast<size_t>(kPVec) * HD + 2 * (wave * 32 + vec)) =
        make_float2(m_run, l_run);
}

// Combines the key splits of every (row, query head) of the row blocks that
// have several: HD / 4 threads per vector, 4 dims each; a workgroup serves
// vectors of one row block and kv head (kv heads innermost, as in the chunk
// kernel, so it runs on the XCD that wrote the records). The records of up to
// 8 splits are requested before any of them is used.
constexpr int kMergeThreads = 256;
template <int HD>
__global__ __launch_bounds__(kMergeThreads) void prefill_merge(const PrefillParams P) {
  constexpr int TPV = HD / 4;                // threads per vector
  constexpr int VPW = kMergeThreads / TPV;   // vectors per workgroup
  constexpr int WPB = kPVec / VPW;           // workgroups per (row block, kv head)
  const int kh = static_cast<int>(blockIdx.x) % P.nkv;
  const int rb = static_cast<int>(blockIdx.x) / P.nkv / WPB;
  const int part = static_cast<int>(blockIdx.x) / P.nkv % WPB;
  const int it = P.first[rb];
  const int nz = static_cast<int>(P.item[it] >> 24);
  if (nz == 1) return;
  const int G = P.n_heads / P.nkv;
  const int j = static_cast<int>(threadIdx.x) / TPV, d4 = static_cast<int>(threadIdx.x) % TPV;
  const int v = part * VPW + j;
  const int vrow = (v & 31) / G;
  const int row = rb * (kPWaves * P.rpv) + (v >> 5) * P.rpv + vrow;
  if (vrow >= P.rpv || row >= P.rows) return;
  const int head = kh * G + ((v & 31) - vrow * G);
  const size_t step = static_cast<size_t>(P.nkv) * prefill_record<HD>();  // split to split
  const float* rec = P.part + (static_cast<size_t>(it) * P.nkv + kh) * prefill_record<HD>();
  float M = kMinitP, L = 0.0f;
  float4 O = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
  for (int z0 = 0; z0 < nz; z0 += 8) {
    float4 o[8];
    float2 ml[8];
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      const float* rz = rec + min(z0 + i, nz - 1) * step;
      o[i] = *reinterpret_cast<const float4*>(rz + static_cast<size_t>(v) * HD + 4 * d4);
      ml[i] = *reinterpret_cast<const float2*>(rz + static_cast<size_t>(kPVec) * HD + 2 * v);
    }
    float Mn = M;
#pragma unroll
    for (int i = 0; i < 8; ++i) Mn = fmaxf(Mn, ml[i].x);
    const float a = __builtin_amdgcn_exp2f(M - Mn);
    M = Mn;
    L *= a;
    O.x *= a;
    O.y *= a;
    O.z *= a;
    O.w *= a;
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      if (z0 + i >= nz) break;
      const float f = __builtin_amdgcn_exp2f(ml[i].x - M);
      L += ml[i].y * f;
      O.x += o[i].x * f;
      O.y += o[i].y * f;
      O.z += o[i].z * f;
      O.w += o[i].w * f;
    }
  }
  *reinterpret_cast<float4*>(P.out + (static_cast<size_t>(row) * P.n_heads + head) * HD + 4 * d4) =
      make_float4(O.x / L, O.y / L, O.z / L, O.w / L);
}

// The workgroups of a launch, per kv head. Every row block takes
// ceil(stages / T) of them, T the smallest number of stages (at least
// kMinStages, at most kPrefillMaxSplits per block) for which the launch fits
// one workgroup per CU; with more row blocks than that, one each.
struct PrefillPlan {
  int rpv, n_blocks, n_items, max_split, T;
};
constexpr int kMinStages = 2;

// (with out: its item table too)
PrefillPlan prefill_plan(const KvGeom& g, const AttnCall& c, PrefillParams* out) {
  PrefillPlan p{};
  p.rpv = 32 / (c.n_heads / g.nkv);
  const int rb = kPWaves * p.rpv;
  p.n_blocks = (c.rows + rb - 1) / rb;
  p.max_split = 1;
  const int room = kPrefillBlocks / g.nkv;  // workgroups per kv head
  auto stages = [&](int i) {
    const int last = c.pos0 + ((i + 1) * rb < c.rows ? (i + 1) * rb : c.rows) - 1;
    return last / Stage<64>::SK + 1;
  };
  const int longest = stages(p.n_blocks - 1);
  if (p.n_blocks >= room) {
    p.T = longest;
    return p;
  }
  auto splits = [&](int i, int T) { return (stages(i) + T - 1) / T; };
  long long total = 0;
  for (int i = 0; i < p.n_blocks; ++i) total += stages(i);
  p.T = static_cast<int>((total + room - 1) / room);
  const int by_splits = (longest + kPrefillMaxSplits - 1) / kPrefillMaxSplits;
  if (p.T < by_splits) p.T = by_splits;
  if (p.T < kMinStages) p.T = kMinStages;
  for (;; ++p.T) {
    int w = 0;
    for (int i = 0; i < p.n_blocks && w <= room; ++i) w += splits(i, p.T);
    if (w <= room) break;
  }
  for (int i = p.n_blocks - 1; i >= 0; --i) {
    const int nz = splits(i, p.T);
    p.max_split = nz > p.max_split ? nz : p.max_split;
    if (out != nullptr) {
      out->first[i] = static_cast<uint16_t>(p.n_items);
      for (int z = 0; z < nz; ++z)
        out->item[p.n_items + z] = static_cast<uint32_t>(i) | static_cast<uint32_t>(z) << 16 |
                                   static_cast<uint32_t>(nz) << 24;
    }
    p.n_items += nz;
  }
  return p;
}

template <int HD, bool I8>
hipError_t launch(const PrefillParams& p, int max_split, hipStream_t st) {
  const int items = p.n_items > 0 ? p.n_items : p.n_blocks;
  hipLaunchKernelGGL((prefill_kernel<HD, I8>), dim3(items * p.nkv), dim3(kPThreads), 0, st, p);
  const hipError_t e = hipGetLastError();
  if (e != hipSuccess || max_split == 1) return e;
  constexpr int wpb = kPVec / (kMergeThreads / (HD / 4));
  hipLaunchKernelGGL(prefill_merge<HD>, dim3(p.n_blocks * p.nkv * wpb), dim3(kMergeThreads), 0, st, p);
  return hipGetLastError();
}

}  // namespace

int prefill_split_count(const KvGeom& g, const AttnCall& c) { return prefill_plan(g, c, nullptr).max_split; }

// The rows kernels stream the keys once per group of 32 vectors with little
// else to pay; this kernel pays for its prologue, pipeline and merge launch
// and then takes a quarter (int8: two thirds) of the time per vector and key.
// Estimates in us of both, from chunks of 16 to 256 rows of 8 kv heads at 0 to
// 8000 keys, G 1, 3 and 4 (rows | here):
//  fp32 hd 64, G 4: 64 rows at 1984 18.7 | 21.7, 100 rows 28.4 | 22.1, 64 rows
//    at 8000 45 | 39, 256 rows at 0 10.0 | 13.5, at 1984 45 | 33;
//  fp32 hd 128, G 4: 64 rows at 1984 30.2 | 32.6, 100 rows 48 | 34, 128 rows at
//    448 25 | 23, 256 rows at 0 16.8 | 18.8;
//  int8 hd 64, G 4: 100 rows at 1984 22.2 | 22.6, at 8000 56 | 46, 256 rows at
//    448 20.9 | 19.6, at 1984 38 | 32;
//  int8 hd 128, G 3: 100 rows at 8000 66 | 68, 256 rows at 448 30 | 26, at 1984
//    59 | 48, at 8000 174 | 135.
bool prefill_supported(const KvGeom& g, const AttnCall& c) {
  if (g.ring || !g.tiled || c.rows < kPrefillMinRows || c.n_heads % g.nkv != 0 ||
      c.n_heads / g.nkv > 8)
    return false;
  struct Cost {
    double base, stage, split, rows, key;
  };
  static constexpr Cost kCost[2][2] = {{{12.0, 2.40, 0.15, 8.5, 70.5e-6}, {14.0, 4.4, 0.3, 14.0, 123e-6}},
                                       {{10.0, 2.35, 0.15, 11.0, 52e-6}, {14.0, 4.2, 0.3, 13.0, 90e-6}}};
  const Cost& k = kCost[g.int8][g.hd != 64];
  const int rpg = 32 / (c.n_heads / g.nkv);
  const double keys = static_cast<double>(g.nkv) * ((c.rows + rpg - 1) / rpg) * (c.pos0 + c.rows / 2 + 16);
  const PrefillPlan p = prefill_plan(g, c, nullptr);
  return k.base + k.stage * p.T + k.split * p.max_split < k.rows + k.key * keys;
}

// (one region per workgroup whatever the split, so one call's workspace
// serves every later one)
size_t prefill_workspace_need(const KvGeom& g, const AttnCall&) {
  return static_cast<size_t>(kPrefillBlocks) *
         (g.hd == 64 ? prefill_record<64>() : prefill_record<128>());
}

hipError_t launch_prefill(const KvGeom& g, const KvStore& s, Workspace& ws, const AttnCall& c,
                          hipStream_t st) {
  PrefillParams p{};
  const PrefillPlan pl = prefill_plan(g, c, &p);
  if (pl.max_split > 1 && ws.part_floats < prefill_workspace_need(g, c))
    return hipErrorInvalidValue;
  const size_t layer_heads = static_cast<size_t>(c.layer) * g.nkv;
  const size_t layer_el = layer_heads * head_elems(g);
  if (g.int8) {
    p.k8 = s.k8 + layer_el;
    p.v8 = s.v8 + layer_el;
    p.ks = s.k_scale + layer_heads * g.ngroups * g.hd;
    p.vs = s.v_scale + layer_heads * g.capg * g.nb;
    p.ng = g.ngroups;
    p.n_sink = g.n_sink;
    if (g.n_sink > 0) {
      p.ksink = s.k_sink + layer_heads * g.n_sink * g.hd;
      p.vsink = s.v_sink + layer_heads * g.n_sink * g.hd;
    }
  } else {
    p.kf = s.k + layer_el;
    p.vf = s.v + layer_el;
  }
  p.q = c.q;
  p.out = c.out;
  p.part = ws.part;
  p.capg = g.capg;
  p.nkv = g.nkv;
  p.n_heads = c.n_heads;
  p.rows = c.rows;
  p.pos0 = c.pos0;
  p.rpv = pl.rpv;
  p.n_blocks = pl.n_blocks;
  p.n_items = pl.n_items;
  p.qscale = c.scale * kLog2eP;
  if (g.int8)
    return g.hd == 64 ? launch<64, true>(p, pl.max_split, st) : launch<128, true>(p, pl.max_split, st);
  return g.hd == 64 ? launch<64, false>(p, pl.max_split, st) : launch<128, false>(p, pl.max_split, st);
}

}  // namespace dbi
