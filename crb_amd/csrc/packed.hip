// Packed low-bit storage of CRB/BRAQ-quantized weights and its GEMV.
//
// The reference stores the quantized layer as fake-quantized fp16/bf16
// weights (bigptq.py:278-280).  Within one 128-column block of one row,
// those weights take at most 2 distinct values in each non-salient group
// (mask1, mask2: order-1 binarization, mu +- alpha) and at most 4 on the
// salient columns (mask3: order 2, mu + a1 s1 + a2 s2); the salient columns
// of a block are whole columns, the same for every row
// (utils/structure.py:8-20).  So the layer is stored exactly as
//   codes [R][nblk * 32] bytes : 2 bits per weight, element j of a block at
//                                byte j / 4, bits 2 (j % 4) .. +1;
//   lut   [R][nblk][8]         : the block row's values in the weight
//                                dtype: mask1 {lo, hi}, mask2 {lo, hi},
//                                mask3 4 values, each ascending;
//   sal   [nblk][16] bytes     : salient-column bitmap of each block;
// with weight = lut[r][b][4 * sal + code], code = (mask2 ? 2 : 0) + rank
// for non-salient weights and rank (0..3) for salient ones: 3 bits per
// weight instead of 16, and unpacking reproduces the weights bit for bit.
#include <algorithm>
#include <type_traits>

#include "common.h"

namespace crbq {

constexpr int PB = 128;   // packing block (columns)

// Order-preserving 16-bit keys: -0 sorts just below +0, so the two zeros
// are distinct values and round-trip exactly.
__device__ __forceinline__ int key16(uint32_t u) {
  return (u & 0x8000u) ? (int)(~u & 0xffffu) : (int)(u | 0x8000u);
}
__device__ __forceinline__ uint16_t unkey16(int k) {
  return (k & 0x8000) ? (uint16_t)(k & 0x7fff) : (uint16_t)(~k & 0xffff);
}
__device__ __forceinline__ int wave_min_i(int v) {
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) v = min(v, __shfl_xor(v, o, CRBQ_WAVE));
  return v;
}
__device__ __forceinline__ int wave_or_i(int v) {
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) v |= __shfl_xor(v, o, CRBQ_WAVE);
  return v;
}

__global__ void k_zero_status(int* status, int* ex_count) {
  *status = 0;
  *ex_count = 0;
}

__device__ __forceinline__ float half_bits_to_float(uint32_t u, bool bf16) {
  return bf16 ? __uint_as_float(u << 16)
              : (float)__builtin_bit_cast(_Float16, (unsigned short)(u & 0xffffu));
}

constexpr int NDV = 8;    // distinct values a group's table is chosen from

// Packs one block row (r, b) with a whole wavefront, exceptions included;
// lane l holds elements l and 64 + l.
// Per group (mask 1 and 2: 2 table entries, mask 3: 4) the table keeps the
// most frequent values among the group's NDV smallest distinct values (ties
// to the smaller key), in ascending order; every other element is an
// exception: code = the group's first entry, and (flat index r * C + c, raw
// value, value - first entry in fp32) appended to the exception list.
__device__ __forceinline__ void pack_block(const uint16_t* __restrict__ Q, int64_t ldq,
                                           const uint8_t* __restrict__ M, int64_t ldm, int r,
                                           int b, int C, int nblk, bool bf16,
                                           uint8_t* __restrict__ codes, int64_t ldc,
                                           uint16_t* __restrict__ lut,
                                           int64_t* __restrict__ ex_idx,
                                           uint16_t* __restrict__ ex_val,
                                           float* __restrict__ ex_delta, int ex_cap,
                                           int* ex_count, int* status) {
  const int lane = threadIdx.x & 63;
  int key[2], grp[2];
  bool inside[2];
#pragma unroll
  for (int s = 0; s < 2; ++s) {
    const int c = b * PB + s * 64 + lane;
    inside[s] = c < C;
    key[s] = inside[s] ? key16(Q[(int64_t)r * ldq + c]) : 0;
    grp[s] = inside[s] ? M[(int64_t)r * ldm + c] : 0;
  }
  int err = 0;
  int code[2] = {0, 0};
  bool exc[2] = {false, false};
  uint32_t lv[8];
#pragma unroll
  for (int G = 1; G <= 3; ++G) {
    const int cap = G == 3 ? 4 : 2, base = G == 1 ? 0 : (G == 2 ? 2 : 4);
    // the group's NDV smallest distinct keys and their counts (uniform)
    int cand[NDV], cnt[NDV], nd = 0, prev = -1;
#pragma unroll
    for (int k = 0; k < NDV; ++k) {
      cand[k] = 0x10000;
      cnt[k] = 0;
    }
#pragma unroll
    for (int k = 0; k < NDV; ++k) {
      int m = 0x10000;
#pragma unroll
      for (int s = 0; s < 2; ++s)
        if (grp[s] == G && key[s] > prev) m = min(m, key[s]);
      m = wave_min_i(m);
      if (__builtin_amdgcn_readfirstlane(m) >= 0x10000) break;
      cand[k] = m;
      cnt[k] = __popcll(__ballot(grp[0] == G && key[0] == m)) +
               __popcll(__ballot(grp[1] == G && key[1] == m));
      nd = k + 1;
      prev = m;
    }
    // keep the cap most frequent (ties: smaller key), in ascending key order
    bool keep[NDV];
#pragma unroll
    for (int k = 0; k < NDV; ++k) {
      int better = 0;
#pragma unroll
      for (int q = 0; q < NDV; ++q)
        better += (q < nd && (cnt[q] > cnt[k] || (cnt[q] == cnt[k] && q < k))) ? 1 : 0;
      keep[k] = k < nd && better < cap;
    }
    int keys[4] = {0, 0, 0, 0}, found = 0;
#pragma unroll
    for (int k = 0; k < NDV; ++k) {
      const bool take = keep[k] && found < 4;
#pragma unroll
      for (int q = 0; q < 4; ++q) keys[q] = take && found == q ? cand[k] : keys[q];
      found += take;
    }
    int last = keys[0];
#pragma unroll
    for (int q = 1; q < 4; ++q) last = q < found ? keys[q] : last;
#pragma unroll
    for (int s = 0; s < 2; ++s) {
      if (grp[s] != G) continue;
      int rk = -1;
#pragma unroll
      for (int k = 0; k < 4; ++k)
        if (k < found && keys[k] == key[s]) rk = k;
      exc[s] = rk < 0;
      code[s] = (G == 2 ? 2 : 0) + (rk < 0 ? 0 : rk);
    }
#pragma unroll
    for (int k = 0; k < cap; ++k)
      lv[base + k] = found ? unkey16(k < found ? keys[k] : last) : 0u;
  }
  // exceptions (rare): append to the list
#pragma unroll
  for (int s = 0; s < 2; ++s) {
    if (!exc[s]) continue;
    const int c = b * PB + s * 64 + lane;
    const uint32_t v = unkey16(key[s]);
    const int at = (grp[s] == 3 ? 4 : 0) + code[s];
    uint32_t t = lv[0];
#pragma unroll
    for (int q = 1; q < 8; ++q) t = at == q ? lv[q] : t;
    const int e = atomicAdd(ex_count, 1);
    if (e < ex_cap) {
      ex_idx[e] = (int64_t)r * C + c;
      ex_val[e] = (uint16_t)v;
      ex_delta[e] = half_bits_to_float(v, bf16) - half_bits_to_float(t, bf16);
    } else {
      err |= 1;
    }
  }
  err = wave_or_i(err);
  if (lane == 0 && err) atomicOr(status, err);
  // byte t (lanes 0..31) packs elements 4t .. 4t+3, all in slot t / 16
  uint32_t byte = 0;
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int src = (4 * lane + i) & 63;
    const int c0 = __shfl(code[0], src, CRBQ_WAVE), c1 = __shfl(code[1], src, CRBQ_WAVE);
    byte |= (uint32_t)((lane < 16 ? c0 : c1) & 3) << (2 * i);
  }
  if (lane < 32) codes[(int64_t)r * ldc + b * 32 + lane] = (uint8_t)byte;
  if (lane < 4) {
    uint32_t v = lv[0] | (lv[1] << 16);
    if (lane == 1) v = lv[2] | (lv[3] << 16);
    if (lane == 2) v = lv[4] | (lv[5] << 16);
    if (lane == 3) v = lv[6] | (lv[7] << 16);
    ((uint32_t*)(lut + ((int64_t)r * nblk + b) * 8))[lane] = v;
  }
}

typedef unsigned short us2_t __attribute__((ext_vector_type(2)));
__device__ __forceinline__ us2_t pk_min(us2_t a, us2_t b) { return __builtin_elementwise_min(a, b); }
// minimum of both halves over each 16-lane row
__device__ __forceinline__ us2_t row_pk_min(us2_t v) {
  auto u = [](us2_t x) { return __builtin_bit_cast(unsigned, x); };
  auto f = [](unsigned x) { return __builtin_bit_cast(us2_t, x); };
  v = pk_min(v, f(dpp_u32<DPP_XOR1>(u(v))));
  v = pk_min(v, f(dpp_u32<DPP_XOR2>(u(v))));
  v = pk_min(v, f(dpp_u32<DPP_HALF_MIRROR>(u(v))));
  return pk_min(v, f(dpp_u32<DPP_MIRROR>(u(v))));
}

// 16 lanes per block row, 8 consecutive elements per lane.  Almost every
// block row has at most 2 distinct values in mask groups 1 and 2 and 4 in
// group 3, so each group's table is its smallest and largest value (kept as
// the minima of key and ~key in the halves of one register) and, for group
// 3, the smallest and largest of what is left; a block row with an element
// outside those goes through pack_block, the workgroup's in turn over its
// wavefronts (768 x 768 with 500 exceptions 96 us, each wavefront its own
// 103, on one card; 16 wavefronts a workgroup: 295 for 4096 x 16384 without
// any).  Bound by issue (753 vector instructions per 4 block rows, 85 % of
// the time busy): with the host's part 85 us for 4096 x 4096, 43 of them the
// kernel, and 189 for 4096 x 16384, against 357 and 1254 with one wavefront
// per block row and eight minimum searches per group.
constexpr int PK_WAVES = 4;
__global__ __launch_bounds__(64 * PK_WAVES) void k_pack(
    const uint16_t* __restrict__ Q, int64_t ldq, const uint8_t* __restrict__ M, int64_t ldm, int R,
    int C, int nblk, bool bf16, uint8_t* __restrict__ codes, int64_t ldc,
    uint16_t* __restrict__ lut, uint8_t* __restrict__ sal, int64_t* __restrict__ ex_idx,
    uint16_t* __restrict__ ex_val, float* __restrict__ ex_delta, int ex_cap, int* ex_count,
    int* status) {
  __shared__ unsigned slow4[PK_WAVES];
  const int64_t w = (int64_t)blockIdx.x * (4 * PK_WAVES) + (threadIdx.x >> 4);
  const bool live = w < (int64_t)R * nblk;
  const int r = live ? (int)(w / nblk) : 0, b = live ? (int)(w - (int64_t)r * nblk) : 0;
  const int l16 = threadIdx.x & 15;
  const int c0 = b * PB + l16 * 8;
  const uint16_t* q = Q + (int64_t)r * ldq + c0;
  const uint8_t* m = M + (int64_t)r * ldm + c0;
  uint32_t v[4];
  uint64_t g8, s8;                 // mask codes of this row and of row 0
  if (live && c0 + 8 <= C) {
    __builtin_memcpy(v, q, 16);
    __builtin_memcpy(&g8, m, 8);
    __builtin_memcpy(&s8, M + c0, 8);
  } else {
    g8 = s8 = 0;
#pragma unroll
    for (int e = 0; e < 4; ++e) v[e] = 0u;
#pragma unroll
    for (int e = 0; e < 8; ++e)
      if (live && c0 + e < C) {
        v[e >> 1] |= (uint32_t)q[e] << (16 * (e & 1));
        g8 |= (uint64_t)m[e] << (8 * e);
        s8 |= (uint64_t)M[c0 + e] << (8 * e);
      }
  }
  int err = 0;
  uint32_t key[8], salb = 0;
  us2_t mn[3];
#pragma unroll
  for (int G = 0; G < 3; ++G) mn[G] = us2_t{0xffff, 0xffff};
#pragma unroll
  for (int e = 0; e < 8; ++e) {
    const uint32_t u = (v[e >> 1] >> (16 * (e & 1))) & 0xffffu;
    const int g = (int)(g8 >> (8 * e)) & 0xff;
    key[e] = (uint32_t)key16(u);
    const uint32_t kk = key[e] | (~key[e] << 16);
#pragma unroll
    for (int G = 0; G < 3; ++G)
      mn[G] = pk_min(mn[G], __builtin_bit_cast(us2_t, g == G + 1 ? kk : 0xffffffffu));
    const bool in = live && c0 + e < C;
    salb |= (uint32_t)(g == 3) << e;
    if (in && (g < 1 || g > 3)) err |= 4;
    if ((g == 3) != (((int)(s8 >> (8 * e)) & 0xff) == 3)) err |= 2;  // row 0 sets the columns
  }
  uint32_t lo[3], hi[3];
  bool some[3];
#pragma unroll
  for (int G = 0; G < 3; ++G) {
    mn[G] = row_pk_min(mn[G]);
    lo[G] = mn[G][0];
    hi[G] = 0xffffu & ~(uint32_t)mn[G][1];
    some[G] = !(mn[G][0] == 0xffff && mn[G][1] == 0xffff);
  }
  us2_t rest = us2_t{0xffff, 0xffff};      // group 3 without its smallest and largest
#pragma unroll
  for (int e = 0; e < 8; ++e) {
    const bool in = ((int)(g8 >> (8 * e)) & 0xff) == 3 && key[e] != lo[2] && key[e] != hi[2];
    rest = pk_min(rest, __builtin_bit_cast(us2_t, in ? key[e] | (~key[e] << 16) : 0xffffffffu));
  }
  rest = row_pk_min(rest);
  const bool has = !(rest[0] == 0xffff && rest[1] == 0xffff);
  const uint32_t b0 = rest[0], b1 = 0xffffu & ~(uint32_t)rest[1];
  const bool two = has && b0 != b1;
  bool slow = false;
  uint32_t word = 0;
#pragma unroll
  for (int e = 0; e < 8; ++e) {
    const int g = (int)(g8 >> (8 * e)) & 0xff;
    const uint32_t k = key[e];
    uint32_t code = 0;
    if (g == 1) {
      code = k != lo[0];
      slow |= k != lo[0] && k != hi[0];
    } else if (g == 2) {
      code = 2u + (k != lo[1]);
      slow |= k != lo[1] && k != hi[1];
    } else if (g == 3) {
      code = (uint32_t)(k > lo[2]) + (uint32_t)(has && k > b0) + (uint32_t)(two && k > b1);
      slow |= k != lo[2] && k != hi[2] && k != b0 && k != b1;
    }
    word |= code << (2 * e);
  }
  const uint64_t sm = __ballot(slow);
  const int lane = threadIdx.x & 63;
  const bool mine = live && ((sm >> (lane & 48)) & 0xffffull) == 0;
  if (mine) {
    const uint16_t wd = (uint16_t)word;
    __builtin_memcpy(codes + (int64_t)r * ldc + b * 32 + 2 * l16, &wd, 2);
    if (l16 < 4) {
      auto pair = [](bool any, uint32_t x, uint32_t y) {
        return any ? (uint32_t)unkey16((int)x) | ((uint32_t)unkey16((int)y) << 16) : 0u;
      };
      // group 3 ascending, padded with its largest value
      const uint32_t e1 = has ? b0 : hi[2], e2 = two ? b1 : hi[2];
      const uint32_t t = l16 == 0 ? pair(some[0], lo[0], hi[0])
                       : l16 == 1 ? pair(some[1], lo[1], hi[1])
                       : l16 == 2 ? pair(some[2], lo[2], e1)
                                  : pair(some[2], e2, hi[2]);
      ((uint32_t*)(lut + ((int64_t)r * nblk + b) * 8))[l16] = t;
    }
  }
  if (live && r == 0) sal[(int64_t)b * 16 + l16] = (uint8_t)salb;
  if (!live) err = 0;
  err = wave_or_i(err);
  if (lane == 0 && err) atomicOr(status, err);
  // block rows with exceptions: the workgroup's, over its wavefronts in turn
  // (a barrier that does not wait for the stores)
  auto any16 = [&](int k) { return (unsigned)(((sm >> (16 * k)) & 0xffffull) != 0) << k; };
  if (lane == 0) slow4[threadIdx.x >> 6] = any16(0) | any16(1) | any16(2) | any16(3);
  asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
  const int wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
  int k = 0;
#pragma unroll 1
  for (int q = 0; q < PK_WAVES; ++q) {
    unsigned todo = __builtin_amdgcn_readfirstlane(slow4[q]);
    for (; todo; todo &= todo - 1, ++k) {
      if (k % PK_WAVES != wave) continue;
      const int64_t wi = (int64_t)blockIdx.x * (4 * PK_WAVES) + 4 * q + __builtin_ctz(todo);
      int rr = (int)(wi / nblk), bb = (int)(wi - (int64_t)rr * nblk);
      // in vector registers: as scalars their addresses would spill others
      asm volatile("" : "+v"(rr), "+v"(bb));
      pack_block(Q, ldq, M, ldm, rr, bb, C, nblk, bf16, codes, ldc, lut, ex_idx, ex_val, ex_delta,
                 ex_cap, ex_count, status);
    }
  }
}

// Decoding four weights at a time.  The eight table entries of a block row
// are split into their low and their high bytes (two registers each, the
// eight byte sources of one v_perm_b32), so a selector of four bytes 4 *
// salient + code picks the low bytes of four weights with one v_perm_b32 and
// the high bytes with another, and two more interleave them: 8 instructions
// per four weights, the selector included.
struct Planes {
  uint32_t l0, l1, h0, h1;     // low / high bytes of entries 0-3 and 4-7
};
__device__ __forceinline__ Planes planes_of(uint4 L) {
  return Planes{__builtin_amdgcn_perm(L.y, L.x, 0x06040200u),
                __builtin_amdgcn_perm(L.w, L.z, 0x06040200u),
                __builtin_amdgcn_perm(L.y, L.x, 0x07050301u),
                __builtin_amdgcn_perm(L.w, L.z, 0x07050301u)};
}
// Bits 0-3 of n, each times 4, into the four bytes of a selector.
__device__ __forceinline__ uint32_t sal_bytes(uint32_t n) {
  return ((n & 15u) * 0x00204081u & 0x01010101u) << 2;
}
// Weights of code byte c (0-255: a bit above would reach code 1) and salient
// selector S as two 32-bit pairs.
__device__ __forceinline__ uint2 decode4(uint32_t c, uint32_t S, const Planes& t) {
  const uint32_t x = (c << 12) | c, y = (x << 6) | x;    // code j at bits 8 j
  const uint32_t sel = (y & 0x03030303u) | S;
  const uint32_t lo = __builtin_amdgcn_perm(t.l1, t.l0, sel);
  const uint32_t hi = __builtin_amdgcn_perm(t.h1, t.h0, sel);
  return make_uint2(__builtin_amdgcn_perm(hi, lo, 0x05010400u),
                    __builtin_amdgcn_perm(hi, lo, 0x07030602u));
}

// One thread per 8 columns (one 16-byte store) of UP_ROWS rows, whose
// salient selectors it builds once; 1 << lg threads along a row's columns
// (as many as it has chunks of 8, up to the workgroup) and the rest down the
// rows, so that narrow matrices fill their wavefronts too.  Bound by the
// stores: 23 us for 14336 x 4096 (6 TB/s written and read), 72 with 4 weights
// per thread and 2-byte stores.  With one row of threads per 4 rows whatever
// the width, 100000 x 64 took 17.6 us against 8.9, 1048576 x 8 147 against 15.
constexpr int UP_ROWS = 4;
__global__ __launch_bounds__(256) void k_unpack(const uint8_t* __restrict__ codes, int64_t ldc,
                                                const uint16_t* __restrict__ lut,
                                                const uint8_t* __restrict__ sal, int R, int C,
                                                int nblk, uint16_t* __restrict__ Q, int64_t ldq,
                                                int lg) {
  const int64_t r0 = ((int64_t)blockIdx.x * (256 >> lg) + (threadIdx.x >> lg)) * UP_ROWS;
  if (r0 >= R) return;
  const int64_t nch = ((int64_t)C + 7) / 8;
  for (int64_t j = ((int64_t)blockIdx.y << lg) + (threadIdx.x & ((1 << lg) - 1)); j < nch;
       j += (int64_t)gridDim.y << lg) {
    const int64_t b = j >> 4, c0 = j * 8;
    const int t = (int)(j & 15);
    const uint32_t sb = sal[b * 16 + t];
    const uint32_t S0 = sal_bytes(sb), S1 = sal_bytes(sb >> 4);
    uint16_t cw[UP_ROWS];
    uint4 L[UP_ROWS];
#pragma unroll
    for (int k = 0; k < UP_ROWS; ++k) {
      const int64_t r = r0 + k < R ? r0 + k : R - 1;
      __builtin_memcpy(&cw[k], codes + r * ldc + b * 32 + 2 * t, 2);
      __builtin_memcpy(&L[k], lut + (r * nblk + b) * 8, 16);
    }
#pragma unroll
    for (int k = 0; k < UP_ROWS; ++k) {
      if (r0 + k >= R) break;
      const Planes p = planes_of(L[k]);
      const uint2 w0 = decode4(cw[k] & 0xffu, S0, p), w1 = decode4((uint32_t)cw[k] >> 8, S1, p);
      const uint4 o = make_uint4(w0.x, w0.y, w1.x, w1.y);
      uint16_t* d = Q + (r0 + k) * ldq + c0;
      if (c0 + 8 <= C) {
        __builtin_memcpy(d, &o, 16);
      } else {
#pragma unroll
        for (int e = 0; e < 8; ++e) {
          const uint32_t h = e < 2 ? o.x : e < 4 ? o.y : e < 6 ? o.z : o.w;
          if (c0 + e < C) d[e] = (uint16_t)(h >> (16 * (e & 1)));
        }
      }
    }
  }
}

// Exceptions of the packed form: the exact values over the unpacked ones.
__global__ __launch_bounds__(256) void k_unpack_ex(const int64_t* __restrict__ ex_idx,
                                                   const uint16_t* __restrict__ ex_val,
                                                   int64_t n_ex, int C, int64_t n,
                                                   uint16_t* __restrict__ Q, int64_t ldq) {
  const int64_t e = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (e >= n_ex) return;
  const int64_t i = ex_idx[e];
  if (i < 0 || i >= n) return;           // indices outside R x C are ignored
  Q[(i / C) * ldq + i % C] = ex_val[e];
}

// y[t][r] += delta_e * x[t][c] for every exception e = (r, c), one thread
// per token, exceptions in list order (deterministic for a given list).
__global__ __launch_bounds__(256) void k_apply_ex(const int64_t* __restrict__ ex_idx,
                                                  const float* __restrict__ ex_delta,
                                                  int64_t n_ex, int C, int64_t n,
                                                  const uint16_t* __restrict__ x, int64_t ldx,
                                                  bool bf16, int T, float* __restrict__ y,
                                                  int64_t ldy) {
  const int t = blockIdx.x * 256 + threadIdx.x;
  if (t >= T) return;
  for (int64_t e = 0; e < n_ex; ++e) {
    const int64_t i = ex_idx[e];
    if (i < 0 || i >= n) continue;       // indices outside R x C are ignored
    const int r = (int)(i / C), c = (int)(i % C);
    y[(int64_t)t * ldy + r] += ex_delta[e] * half_bits_to_float(x[(int64_t)t * ldx + c], bf16);
  }
}

constexpr int GV_MAXVEC = 16;

template <typename T8>
__device__ __forceinline__ f4_t mfma_gv(T8 a, T8 b, f4_t c);
template <>
__device__ __forceinline__ f4_t mfma_gv<h8_t>(h8_t a, h8_t b, f4_t c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_f16(a, b, c, 0, 0, 0);
}
template <>
__device__ __forceinline__ f4_t mfma_gv<b8_t>(b8_t a, b8_t b, f4_t c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0);
}

// What a fused linear layer adds to its fp32 sums before the one rounding to
// the weights' dtype: the exceptions' delta * x (in list order) and the bias.
struct PkEnd {
  const uint16_t* bias;      // [R] in the weights' dtype, or NULL
  const int64_t* ex_idx;
  const float* ex_delta;
  int n_ex;
  bool bf16;
};
__device__ __forceinline__ uint32_t to_half_bits(float v, bool bf16) {
  return bf16 ? (uint32_t)__builtin_bit_cast(unsigned short, (__bf16)v)
              : (uint32_t)__builtin_bit_cast(unsigned short, (_Float16)v);
}
// f(r, c, delta) for the exceptions with a row in [r_lo, r_hi), in list order;
// called by whole wavefronts (64 list entries are tested at a time).
template <typename F>
__device__ __forceinline__ void for_ex(const PkEnd& e, int r_lo, int r_hi, int R, int C, F f) {
  const int lane = threadIdx.x & 63;
  if (r_hi > R) r_hi = R;
  for (int base = 0; base < e.n_ex; base += 64) {
    const bool in = base + lane < e.n_ex;
    const int64_t i = in ? e.ex_idx[base + lane] : -1;
    const float d = in ? e.ex_delta[base + lane] : 0.f;
    const bool hit = i >= (int64_t)r_lo * C && i < (int64_t)r_hi * C;   // outside R x C: ignored
    uint64_t m = __ballot(hit);
    const int r = hit ? (int)(i / C) : 0, c = hit ? (int)(i - (int64_t)r * C) : 0;
    while (m) {
      const int j = __builtin_ctzll(m);
      m &= m - 1;
      f(__builtin_amdgcn_readlane(r, j), __builtin_amdgcn_readlane(c, j),
        __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, d), j)));
    }
  }
}

// y[v][r] = sum_c W[r][c] x[v][c] for up to 16 vectors, W packed, x in the
// weights' 16-bit dtype, fp32 sums, on v_mfma_f32_16x16x32.  A workgroup
// takes 16 rows; its 16 wavefronts split the row's 128-column blocks into
// contiguous ranges.  Per block, lane l takes the 32 contiguous columns
// 32 (l >> 4) .. +31 of row l & 15 (8 bytes of codes and the row-block's
// table) and the same columns of vector l & 15 (64 bytes), and feeds them to
// four MFMAs as 8-column slices: the MFMA sums over k in any order as long
// as A and B agree, so the columns need not be in the instruction's natural
// k order.  The salient selectors are the same for every row: each
// wavefront builds those of two blocks at a time, one per lane, in LDS of its
// own, while the two blocks' loads are in flight (built for the whole
// workgroup behind a barrier before the first load, us at 1 / 8 / 16 vectors:
// 4096 x 16384 16.6 / 21.4 / 25.9, 16384 x 4096 17.0 / 21.7 / 27.6, 768 x 3072
// 4.7 / 5.7 / 6.6, 4100 x 36000 45 / 58 / 76; now 15.3 / 20.0 / 25.1, 16.2 / 20.9 /
// 26.2, 4.6 / 5.4 / 6.5, 41 / 52 / 72).  Bound by latency: four wavefronts per
// SIMD, codes and tables in pieces of lines.  The wavefronts' 16 x 16
// partial products are summed in LDS.  END: the result is rounded to the
// weights' dtype after bias and exceptions, else fp32.
constexpr int GV_WAVES = 16;

// A lane's part of one block: its codes, its row's table and its vector's columns.
struct GvIn {
  uint2 cw;
  uint4 L, xs[4];
};
__device__ __forceinline__ GvIn gv_load(const uint8_t* crow, const uint4* lrow, const uint16_t* xv,
                                        int b, int kq, int C, bool row_ok, bool vec_ok) {
  const int c = b * PB + kq * 32;                // this lane's 32 columns
  GvIn d;
  d.cw = row_ok ? *(const uint2*)(crow + b * 32 + kq * 8) : make_uint2(0u, 0u);
  d.L = row_ok ? lrow[b] : make_uint4(0u, 0u, 0u, 0u);
  if (c + 32 <= C) {                             // all blocks but a ragged last one
    const uint4* xp = (const uint4*)(xv + c);
#pragma unroll
    for (int k = 0; k < 4; ++k) d.xs[k] = vec_ok ? xp[k] : make_uint4(0u, 0u, 0u, 0u);
  } else {
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      uint32_t h[8];
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        const int cc = c + 8 * k + e;
        h[e] = vec_ok && cc < C ? xv[cc] : 0u;
      }
      d.xs[k] = make_uint4(h[0] | (h[1] << 16), h[2] | (h[3] << 16), h[4] | (h[5] << 16),
                           h[6] | (h[7] << 16));
    }
  }
  return d;
}
template <typename T8>
__device__ __forceinline__ void gv_mul(const GvIn& d, const uint32_t* S, int kq, f4_t& acc) {
  const uint4 s0 = *(const uint4*)(S + kq * 8), s1 = *(const uint4*)(S + kq * 8 + 4);
  const Planes p = planes_of(d.L);
#pragma unroll
  for (int k = 0; k < 4; ++k) {
    const uint32_t w = (k < 2 ? d.cw.x : d.cw.y) >> (16 * (k & 1));
    const uint4 sv = k < 2 ? s0 : s1;
    const uint2 a0 = decode4(w & 0xffu, k & 1 ? sv.z : sv.x, p);
    const uint2 a1 = decode4((w >> 8) & 0xffu, k & 1 ? sv.w : sv.y, p);
    acc = mfma_gv<T8>(__builtin_bit_cast(T8, make_uint4(a0.x, a0.y, a1.x, a1.y)),
                      __builtin_bit_cast(T8, d.xs[k]), acc);
  }
}

template <typename T8, bool END>
__global__ __launch_bounds__(64 * GV_WAVES) void k_gemv_packed(
    const uint8_t* __restrict__ codes, int64_t ldc, const uint16_t* __restrict__ lut,
    const uint8_t* __restrict__ sal, int R, int C, int nblk, const uint16_t* __restrict__ x,
    int64_t ldx, int nvec, void* __restrict__ y, int64_t ldy, PkEnd end) {
  __shared__ float red[GV_WAVES][16][17];
  __shared__ __attribute__((aligned(16))) uint32_t Ss[GV_WAVES][64];
  const int r0 = blockIdx.x * 16;
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  const int row = r0 + (lane & 15), kq = lane >> 4, vec = lane & 15;
  const bool row_ok = row < R, vec_ok = vec < nvec;
  const uint8_t* crow = codes + (int64_t)(row_ok ? row : 0) * ldc;
  const uint4* lrow = (const uint4*)(lut + (int64_t)(row_ok ? row : 0) * nblk * 8);
  const uint16_t* xv = x + (int64_t)(vec_ok ? vec : 0) * ldx;
  uint32_t* const Sw = Ss[wave];
  f4_t acc = {0.f, 0.f, 0.f, 0.f};
  const int b_end = (int)((int64_t)nblk * (wave + 1) / GV_WAVES);
  for (int b = (int)((int64_t)nblk * wave / GV_WAVES); b < b_end; b += 2) {
    const bool two = b + 1 < b_end;
    const uint32_t sb = lane < 32 || two ? sal[(int64_t)b * 16 + (lane >> 1)] : 0u;
    const GvIn d0 = gv_load(crow, lrow, xv, b, kq, C, row_ok, vec_ok);
    GvIn d1;
    if (two) d1 = gv_load(crow, lrow, xv, b + 1, kq, C, row_ok, vec_ok);
    // a wavefront's LDS accesses complete in order: no barrier, only the
    // compiler kept from moving accesses
    asm volatile("" ::: "memory");
    Sw[lane] = sal_bytes(sb >> (4 * (lane & 1)));
    asm volatile("" ::: "memory");
    gv_mul<T8>(d0, Sw, kq, acc);
    if (two) gv_mul<T8>(d1, Sw + 32, kq, acc);
  }
  // acc[i] = partial y[vector lane & 15][row r0 + 4 (lane >> 4) + i]
#pragma unroll
  for (int i = 0; i < 4; ++i) red[wave][4 * (lane >> 4) + i][lane & 15] = acc[i];
  __syncthreads();
  const int t = threadIdx.x;
  if (t < 256) {
    const int v = t >> 4, rr = t & 15;           // consecutive rows of one vector
    float s0 = 0.f;
#pragma unroll
    for (int w = 0; w < GV_WAVES; ++w) s0 += red[w][rr][v];
    const bool ok = v < nvec && r0 + rr < R;
    if constexpr (END) {
      for_ex(end, r0, r0 + 16, R, C, [&](int r, int c, float d) {
        if (ok && r == r0 + rr) s0 += d * half_bits_to_float(x[(int64_t)v * ldx + c], end.bf16);
      });
      if (ok) {
        if (end.bias) s0 += half_bits_to_float(end.bias[r0 + rr], end.bf16);
        ((uint16_t*)y)[(int64_t)v * ldy + r0 + rr] = (uint16_t)to_half_bits(s0, end.bf16);
      }
    } else if (ok) {
      ((float*)y)[(int64_t)v * ldy + r0 + rr] = s0;
    }
  }
}

// Y[t][r] = sum_c W[r][c] X[t][c] for many tokens (prefill), W packed: each
// decoded fragment is reused for a tile of up to 16 TG tokens.  A workgroup
// of GM_WAVES wavefronts covers RT 16-row tiles per wavefront x tt tokens
// (a multiple of 16, up to 16 TG: the tokens are split evenly); per
// 128-column block each wavefront decodes its rows' 128 columns (lane l: row
// l & 15 of each tile, columns 32 (l >> 4) .. +31, four 8-column MFMA slices)
// and multiplies them with every 16-token group of the X tile, which the
// whole workgroup stages in LDS (rows padded to 136 halves so a 16-lane
// group's 16-byte reads of 16 tokens fall on disjoint banks) beside the
// block's salient selectors.  With two row tiles an X fragment read from LDS
// feeds two MFMAs, so that LDS and the matrix units are needed for the same
// time; with one they wait for LDS twice as long (80 against 74 us at 4096 x
// 16384 and 300 tokens).  When row and token tiles alone would leave CUs
// idle the block range is split over gridDim.z workgroups, each writing an
// fp32 partial [T][R] slice that k_gemm_packed_sum adds in split order.  END:
// the result is rounded to the weights' dtype after bias and exceptions.
// Counters at 4096 x 16384 and 256 tokens: MFMA busy 32 %, LDS 41 %, 234
// vector instructions per wavefront and block, half of the wavefronts' time
// in waits.  Codes and tables of four blocks at a time through LDS (whole
// lines) measured no faster (85 us at 300 tokens, 34 against 22 at 17).
constexpr int GM_WAVES = 8;
constexpr int GM_XP = PB + 8;                     // LDS pitch of an X tile row (halves)

template <typename T8, int TG, int RT, bool END>
__global__ __launch_bounds__(64 * GM_WAVES) void k_gemm_packed(
    const uint8_t* __restrict__ codes, int64_t ldc, const uint16_t* __restrict__ lut,
    const uint8_t* __restrict__ sal, int R, int C, int nblk, const uint16_t* __restrict__ x,
    int64_t ldx, int T, int tt, int bps, void* __restrict__ y, int64_t ldy, PkEnd end) {
  __shared__ __attribute__((aligned(16))) uint16_t Xs[2][16 * TG][GM_XP];
  __shared__ __attribute__((aligned(16))) uint32_t Ss[2][32];
  const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63;
  const int r0 = (blockIdx.x * GM_WAVES + wave) * 16 * RT, t0 = blockIdx.y * tt;
  const int b_beg = blockIdx.z * bps, b_end = min(nblk, b_beg + bps);
  const int kq = lane >> 4;
  const int nt = min(tt, T - t0), ng = (nt + 15) / 16;
  // rows past R read row 0: an MFMA output row depends only on its own
  // weight row, and those rows are not stored
  const uint8_t* crow[RT];
  const uint4* lrow[RT];
#pragma unroll
  for (int i = 0; i < RT; ++i) {
    const int row = r0 + 16 * i + (lane & 15);
    crow[i] = codes + (int64_t)(row < R ? row : 0) * ldc + kq * 8;
    lrow[i] = (const uint4*)(lut + (int64_t)(row < R ? row : 0) * nblk * 8);
  }
  // X tile loader: thread -> (token xt, XPT 8-column chunks from xc)
  constexpr int XPT = TG * 16 * PB / 8 / (64 * GM_WAVES);   // 16-byte chunks per thread
  constexpr int TPR = PB / 8 / XPT;                         // threads per token row
  const int xt = tid / TPR, xc = (tid % TPR) * XPT * 8;
  const bool tok_ok = xt < nt;
  const uint16_t* xrow = x + (int64_t)(tok_ok ? t0 + xt : 0) * ldx;
  uint4 u[XPT];
  uint2 cw[RT];
  uint4 L[RT];
  uint32_t sb = 0;
  auto load_x = [&](int b) {
    const int c = b * PB + xc;
    if (tok_ok && c + 8 * XPT <= C) {
#pragma unroll
      for (int k = 0; k < XPT; ++k) u[k] = *(const uint4*)(xrow + c + 8 * k);
    } else {
#pragma unroll
      for (int k = 0; k < XPT; ++k) {
        uint32_t h[8];
#pragma unroll
        for (int e = 0; e < 8; ++e) h[e] = tok_ok && c + 8 * k + e < C ? xrow[c + 8 * k + e] : 0u;
        u[k] = make_uint4(h[0] | (h[1] << 16), h[2] | (h[3] << 16), h[4] | (h[5] << 16),
                          h[6] | (h[7] << 16));
      }
    }
  };
  auto load_codes = [&](int b) {                 // and tables and salient bits
#pragma unroll
    for (int i = 0; i < RT; ++i) {
      cw[i] = *(const uint2*)(crow[i] + b * 32);
      L[i] = lrow[i][b];
    }
    if (tid < 32) sb = sal[(int64_t)b * 16 + (tid >> 1)] >> (4 * (tid & 1));
  };
  f4_t acc[RT][TG];
#pragma unroll
  for (int i = 0; i < RT; ++i)
#pragma unroll
    for (int g = 0; g < TG; ++g) acc[i][g] = f4_t{0.f, 0.f, 0.f, 0.f};
  // Fragment a[i][k] of a block from codes c, tables p and selectors s0, s1
  T8 a[RT][4], an[RT][4];
  auto decode = [&](T8& f, int k, uint2 c, const Planes& p, uint4 s0, uint4 s1) {
    const uint32_t w = (k < 2 ? c.x : c.y) >> (16 * (k & 1));
    const uint4 sv = k < 2 ? s0 : s1;
    const uint2 a0 = decode4(w & 0xffu, k & 1 ? sv.z : sv.x, p);
    const uint2 a1 = decode4((w >> 8) & 0xffu, k & 1 ? sv.w : sv.y, p);
    f = __builtin_bit_cast(T8, make_uint4(a0.x, a0.y, a1.x, a1.y));
  };
  if (b_beg < b_end) {
    load_codes(b_beg);
    load_x(b_beg);
    if (tid < 32) Ss[b_beg & 1][tid] = sal_bytes(sb);
    __syncthreads();
    const uint4 s0 = *(const uint4*)&Ss[b_beg & 1][kq * 8];
    const uint4 s1 = *(const uint4*)&Ss[b_beg & 1][kq * 8 + 4];
#pragma unroll
    for (int i = 0; i < RT; ++i) {
      const Planes p = planes_of(L[i]);
#pragma unroll
      for (int k = 0; k < 4; ++k) decode(a[i][k], k, cw[i], p, s0, s1);
    }
    load_codes(min(b_beg + 1, b_end - 1));
  }
  // Block b: multiply its fragments while block b + 1's are decoded, a part
  // with each token group (decoding at the top of a block, where the barrier
  // has just lined the wavefronts up, left the matrix units idle meanwhile);
  // X is loaded one block ahead, codes, tables and salient bits two.  The
  // last block stands by itself, with nothing to load or decode behind it:
  // 64 x 64 at 64 tokens 5.0 us to 4.1, 1000 x 1000 at 300 16.4 to 13.1, 4096 x
  // 4096 at 64 15.1 to 14.0.
  auto block = [&](int b, auto is_last) {
    constexpr bool LAST = decltype(is_last)::value;
    const int buf = b & 1;
#pragma unroll
    for (int k = 0; k < XPT; ++k) *(uint4*)&Xs[buf][xt][xc + 8 * k] = u[k];
    uint2 cn[RT];
    Planes p[RT];
    if constexpr (!LAST) {
      if (tid < 32) Ss[buf ^ 1][tid] = sal_bytes(sb);
#pragma unroll
      for (int i = 0; i < RT; ++i) {
        cn[i] = cw[i];
        p[i] = planes_of(L[i]);
      }
    }
    __syncthreads();
    uint4 s0, s1;
    if constexpr (!LAST) {
      load_x(b + 1);
      load_codes(min(b + 2, b_end - 1));
      s0 = *(const uint4*)&Ss[buf ^ 1][kq * 8];
      s1 = *(const uint4*)&Ss[buf ^ 1][kq * 8 + 4];
    }
    constexpr int PER = RT * 4 / TG > 0 ? RT * 4 / TG : 1;   // fragments decoded per group
    auto part = [&](int g) {
#pragma unroll
      for (int q = 0; q < PER; ++q) {
        const int f = g * PER + q;
        if (f < RT * 4) decode(an[f >> 2][f & 3], f & 3, cn[f >> 2], p[f >> 2], s0, s1);
      }
    };
    // a group's X fragments are read while the group before it is multiplied
    const uint16_t* xr = &Xs[buf][lane & 15][kq * 32];
    T8 xf[2][4];
#pragma unroll
    for (int k = 0; k < 4; ++k) xf[0][k] = *(const T8*)(xr + 8 * k);
#pragma unroll
    for (int g = 0; g < TG; ++g) {
      if (g < ng) {                               // uniform
        if (g + 1 < TG) {
#pragma unroll
          for (int k = 0; k < 4; ++k)
            xf[(g + 1) & 1][k] = *(const T8*)(xr + (g + 1) * 16 * GM_XP + 8 * k);
        }
#pragma unroll
        for (int k = 0; k < 4; ++k)
#pragma unroll
          for (int i = 0; i < RT; ++i) acc[i][g] = mfma_gv<T8>(a[i][k], xf[g & 1][k], acc[i][g]);
      }
      if constexpr (!LAST) part(g);
    }
    if constexpr (!LAST) {
#pragma unroll
      for (int i = 0; i < RT; ++i)
#pragma unroll
        for (int k = 0; k < 4; ++k) a[i][k] = an[i][k];
    }
    // the other X buffer is written next; this one is only read again after
    // the following block's barrier
  };
  for (int b = b_beg; b + 1 < b_end; ++b) block(b, std::false_type{});
  if (b_beg < b_end) block(b_end - 1, std::true_type{});
  // acc[i][g][e] = y[token t0 + 16 g + (lane & 15)][row r0 + 16 i + 4 (lane >> 4) + e]
  if constexpr (END) {
    for_ex(end, r0, r0 + 16 * RT, R, C, [&](int r, int c, float d) {
#pragma unroll
      for (int g = 0; g < TG; ++g) {
        const int t = g * 16 + (lane & 15);
        if (t >= nt) continue;
        const float dx = d * half_bits_to_float(x[(int64_t)(t0 + t) * ldx + c], end.bf16);
#pragma unroll
        for (int i = 0; i < RT; ++i)
#pragma unroll
          for (int e = 0; e < 4; ++e)
            if (r == r0 + 16 * i + 4 * kq + e) acc[i][g][e] += dx;
      }
    });
  }
  float* out = (float*)y + (size_t)blockIdx.z * (size_t)T * (size_t)ldy;
#pragma unroll
  for (int i = 0; i < RT; ++i) {
    const int rb = r0 + 16 * i + 4 * kq;
    float bias[4] = {0.f, 0.f, 0.f, 0.f};
    if constexpr (END) {
#pragma unroll
      for (int e = 0; e < 4; ++e)
        if (end.bias && rb + e < R) bias[e] = half_bits_to_float(end.bias[rb + e], end.bf16);
    }
#pragma unroll
    for (int g = 0; g < TG; ++g) {
      const int t = g * 16 + (lane & 15);
      if (t >= nt) continue;
      if constexpr (END) {
        uint16_t* o = (uint16_t*)y + (int64_t)(t0 + t) * ldy + rb;
        uint32_t h[4];
#pragma unroll
        for (int e = 0; e < 4; ++e) h[e] = to_half_bits(acc[i][g][e] + bias[e], end.bf16);
        if (rb + 3 < R && ((((uintptr_t)o) & 7) == 0)) {
          *(uint2*)o = make_uint2(h[0] | (h[1] << 16), h[2] | (h[3] << 16));
        } else {
#pragma unroll
          for (int e = 0; e < 4; ++e)
            if (rb + e < R) o[e] = (uint16_t)h[e];
        }
      } else {
        float* o = out + (int64_t)(t0 + t) * ldy + rb;
        if (rb + 3 < R && ((((uintptr_t)o) & 15) == 0)) {
          *(float4*)o = make_float4(acc[i][g][0], acc[i][g][1], acc[i][g][2], acc[i][g][3]);
        } else {
#pragma unroll
          for (int e = 0; e < 4; ++e)
            if (rb + e < R) o[e] = acc[i][g][e];
        }
      }
    }
  }
}

// y[t][r] = sum_s P[s][t][r] in split order (P rows of R floats), 4 rows per
// thread: grid (ceil(R / 1024), T).  END as above.
template <bool END>
__global__ __launch_bounds__(256) void k_gemm_packed_sum(const float* __restrict__ P, int ns,
                                                         int T, int R, int C,
                                                         const uint16_t* __restrict__ x,
                                                         int64_t ldx, void* __restrict__ y,
                                                         int64_t ldy, PkEnd end) {
  const int r = (blockIdx.x * 256 + threadIdx.x) * 4;
  const bool vec = (R & 3) == 0 && (((uintptr_t)P) & 15) == 0;   // the caller's workspace
  for (int t = blockIdx.y; t < T; t += gridDim.y) {
    float v[4] = {0.f, 0.f, 0.f, 0.f};
    const float* p = P + (int64_t)t * R + r;
    if (vec && r < R) {
#pragma unroll 4
      for (int s = 0; s < ns; ++s) {
        const float4 q = *(const float4*)(p + (int64_t)s * T * R);
        v[0] += q.x; v[1] += q.y; v[2] += q.z; v[3] += q.w;
      }
    } else {
      for (int s = 0; s < ns; ++s)
#pragma unroll
        for (int e = 0; e < 4; ++e)
          if (r + e < R) v[e] += p[(int64_t)s * T * R + e];
    }
    if constexpr (END) {
      for_ex(end, 0, R, R, C, [&](int er, int c, float d) {
        const float dx = d * half_bits_to_float(x[(int64_t)t * ldx + c], end.bf16);
#pragma unroll
        for (int e = 0; e < 4; ++e)
          if (er == r + e) v[e] += dx;
      });
      uint32_t h[4];
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        if (end.bias && r + e < R) v[e] += half_bits_to_float(end.bias[r + e], end.bf16);
        h[e] = to_half_bits(v[e], end.bf16);
      }
      uint16_t* o = (uint16_t*)y + (int64_t)t * ldy + r;
      if (r + 3 < R && ((((uintptr_t)o) & 7) == 0)) {
        *(uint2*)o = make_uint2(h[0] | (h[1] << 16), h[2] | (h[3] << 16));
      } else {
#pragma unroll
        for (int e = 0; e < 4; ++e)
          if (r + e < R) o[e] = (uint16_t)h[e];
      }
    } else {
      float* o = (float*)y + (int64_t)t * ldy + r;
#pragma unroll
      for (int e = 0; e < 4; ++e)
        if (r + e < R) o[e] = v[e];
    }
  }
}

// Launch shape of a packed product, a function of the shapes only so that
// the workspace size is known without a device: 64-token tiles up to 64
// tokens, else the tokens split evenly over tiles of up to 128; one or two
// row tiles per wavefront and the number of column splits (of at least 2
// blocks) with the least modelled time.  Rounds of one workgroup per CU, each
// 5 us and 0.7 + 2.1 tt / 128 us a block with two row tiles, 3.5 us and 0.5 +
// 1.8 tt / 128 us with one; a sum launch of 3.5 us and the partials written
// and read at 4 TB/s.  Two row tiles share every X fragment, which wins where
// the chip is full; one gives twice the workgroups and a shorter block, which
// wins where they are few, and is taken if modelled 8 % faster.  Whole linear
// calls with one / two, each at its own splits (us): 768 x 768 at 17, 64 and
// 300 tokens 7.1 / 8.2, 8.0 / 9.7, 11.4 / 13.7, 256 x 1024 at 64 11.5 / 16.7,
// 3072 x 768 at 300 14.6 / 18.6, 4096 x 4096 at 64 and 300 14.3 / 18.7, 38.9 /
// 31.1, 4096 x 16384 at 64 27.6 / 26.4.  Against splits to fill the chip once,
// twice: 4096 x 16384 at 300 tokens 74 / 83, at 768 167 / 151, 4096 x 4096 at
// 300 33 / 34, at 768 57 / 65; against no split, 4096 x 1920 at 64 11.1 / 18.4.
// Over 15 shapes at 17 to 768 tokens the plan is within 14 % of the best of
// both and 11 splits, but for 3072 x 768 at 17 (24 %) and the rule below.
// Products of at most 256 rows, one token tile and 8 blocks take no
// workspace, as their callers expect (256 x 1024 at 64 tokens 11.6, with
// splits 7.1).
struct GmPlan {
  int tg, rt, tt, ns, bps;
  int64_t row_tiles, tok_tiles;
};
// room: partial slices there is workspace for.
static inline GmPlan gemm_packed_plan(int64_t R, int64_t C, int64_t T,
                                      int64_t room = (int64_t)1 << 40) {
  GmPlan p;
  const int64_t nblk = (C + PB - 1) / PB;
  p.tg = T > 64 ? 8 : 4;
  p.tok_tiles = (T + 16 * p.tg - 1) / (16 * p.tg);
  p.tt = (int)(((T + p.tok_tiles - 1) / p.tok_tiles + 15) / 16 * 16);
  p.tok_tiles = (T + p.tt - 1) / p.tt;
  const double slice = 8.0 * (double)T * (double)R / 4e6;
  const bool none = R <= 256 && p.tok_tiles == 1 && nblk <= 8;
  const int64_t most = none ? 1 : std::max<int64_t>(1, std::min(nblk / 2, room));
  double best = 0.0;
  p.ns = 0;
  for (int rt = 2; rt >= 1; --rt) {
    const int64_t rows = 16 * GM_WAVES * rt, row_tiles = (R + rows - 1) / rows;
    const int64_t tiles = row_tiles * p.tok_tiles;
    const double wg = rt == 2 ? 5.0 : 3.5;
    const double block = rt == 2 ? 0.7 + 2.1 * p.tt / 128.0 : 0.5 + 1.8 * p.tt / 128.0;
    const double less = rt == 2 ? 1.0 : 1.0 / 0.92;
    int64_t n = 1, per = nblk;
    while (n == 1 || (n <= most && tiles * n <= 1024)) {
      const double t = less * ((double)((tiles * n + 255) / 256) * (wg + block * (double)per) +
                               (n > 1 ? 3.5 + slice * (double)n : 0.0));
      if (p.ns == 0 || t < best) {
        best = t;
        p.rt = rt;
        p.row_tiles = row_tiles;
        p.ns = (int)n;
        p.bps = (int)per;
      }
      if (per == 1) break;
      n = (nblk + per - 2) / (per - 1);        // the fewest splits with fewer blocks each
      per = (nblk + n - 1) / n;
    }
  }
  return p;
}

// Partial slices a crbq_gemm_packed call has to bring (crbq.h): splits of at
// least 8 blocks, as many as keep tiles of 128 rows within 512 workgroups.
static inline int64_t gemm_packed_least(int64_t R, int64_t C, int64_t T) {
  const int64_t nblk = (C + PB - 1) / PB, tt = T > 64 ? 128 : 64;
  const int64_t tiles = ((R + 127) / 128) * ((T + tt - 1) / tt);
  const int64_t ns = std::max<int64_t>(1, std::min<int64_t>(512 / tiles, nblk / 8));
  const int64_t per = (nblk + ns - 1) / ns, n = (nblk + per - 1) / per;
  return n > 1 ? n : 0;
}

}  // namespace crbq

extern "C" int crbq_pack(const void* Q, int dtype, int64_t R, int64_t C, int64_t ldq,
                         const uint8_t* masks, int64_t ldm, uint8_t* codes, int64_t ldc,
                         void* lut, uint8_t* sal, int64_t* ex_idx, void* ex_val,
                         float* ex_delta, int ex_cap, int* ex_count, int* status,
                         void* stream) {
  if (!Q || !masks || !codes || !lut || !sal || !status || !ex_count) return CRBQ_ERR_ARG;
  if (ex_cap < 0 || (ex_cap > 0 && (!ex_idx || !ex_val || !ex_delta))) return CRBQ_ERR_ARG;
  if (dtype != CRBQ_F16 && dtype != CRBQ_BF16) return CRBQ_ERR_ARG;
  if (R <= 0 || C <= 0 || R > 0x7fffffff || C > 0x7fffffff || ldq < C || ldm < C)
    return CRBQ_ERR_ARG;
  const int64_t nblk = (C + crbq::PB - 1) / crbq::PB;
  if (ldc < nblk * 32 || (ldc & 7) || (((uintptr_t)lut) & 15) || (((uintptr_t)sal) & 7) ||
      (((uintptr_t)codes) & 7))
    return CRBQ_ERR_ARG;
  hipStream_t s = (hipStream_t)stream;
  crbq::k_zero_status<<<1, 1, 0, s>>>(status, ex_count);
  CRBQ_LAUNCH_CHECK();
  const int64_t rows = R * nblk;
  crbq::k_pack<<<(unsigned)((rows + 4 * crbq::PK_WAVES - 1) / (4 * crbq::PK_WAVES)),
                 64 * crbq::PK_WAVES, 0, s>>>(
      (const uint16_t*)Q, ldq, masks, ldm, (int)R, (int)C, (int)nblk, dtype == CRBQ_BF16, codes,
      ldc, (uint16_t*)lut, sal, ex_idx, (uint16_t*)ex_val, ex_delta, ex_cap, ex_count, status);
  CRBQ_LAUNCH_CHECK();
  return CRBQ_OK;
}

extern "C" int crbq_unpack(const uint8_t* codes, int64_t ldc, const void* lut, const uint8_t* sal,
                           const int64_t* ex_idx, const void* ex_val, int64_t n_ex, int dtype,
                           int64_t R, int64_t C, void* Q, int64_t ldq, void* stream) {
  if (!codes || !lut || !sal || !Q) return CRBQ_ERR_ARG;
  if (n_ex < 0 || (n_ex > 0 && (!ex_idx || !ex_val))) return CRBQ_ERR_ARG;
  if (dtype != CRBQ_F16 && dtype != CRBQ_BF16) return CRBQ_ERR_ARG;
  if (R <= 0 || C <= 0 || R > 0x7fffffff || C > 0x7fffffff || ldq < C) return CRBQ_ERR_ARG;
  const int64_t nblk = (C + crbq::PB - 1) / crbq::PB;
  if (ldc < nblk * 32) return CRBQ_ERR_ARG;
  const int64_t nch = (C + 7) / 8;
  int lg = 0;
  while (lg < 8 && ((int64_t)1 << lg) < nch) ++lg;
  const int64_t per_wg = (int64_t)(256 >> lg) * crbq::UP_ROWS;
  const int64_t rows = (R + per_wg - 1) / per_wg;
  const int64_t chunks = std::min<int64_t>((nch + ((int64_t)1 << lg) - 1) >> lg, 65535);
  hipStream_t s = (hipStream_t)stream;
  crbq::k_unpack<<<dim3((unsigned)rows, (unsigned)chunks), 256, 0, s>>>(
      codes, ldc, (const uint16_t*)lut, sal, (int)R, (int)C, (int)nblk, (uint16_t*)Q, ldq, lg);
  CRBQ_LAUNCH_CHECK();
  if (n_ex > 0) {
    crbq::k_unpack_ex<<<(unsigned)((n_ex + 255) / 256), 256, 0, s>>>(
        ex_idx, (const uint16_t*)ex_val, n_ex, (int)C, R * C, (uint16_t*)Q, ldq);
    CRBQ_LAUNCH_CHECK();
  }
  return CRBQ_OK;
}

static int apply_ex(const int64_t* ex_idx, const float* ex_delta, int64_t n_ex, int64_t R,
                    int64_t C, const void* x, int64_t ldx, int dtype, int64_t T, float* y,
                    int64_t ldy, hipStream_t s) {
  if (n_ex <= 0) return CRBQ_OK;
  crbq::k_apply_ex<<<(unsigned)((T + 255) / 256), 256, 0, s>>>(
      ex_idx, ex_delta, n_ex, (int)C, R * C, (const uint16_t*)x, ldx, dtype == CRBQ_BF16,
      (int)T, y, ldy);
  CRBQ_LAUNCH_CHECK();
  return CRBQ_OK;
}

// Argument checks the packed products share.
static int packed_check(const uint8_t* codes, int64_t ldc, const void* lut, const uint8_t* sal,
                        const int64_t* ex_idx, const float* ex_delta, int64_t n_ex, int dtype,
                        int64_t R, int64_t C, const void* x, int64_t ldx, int64_t ntok,
                        const void* y, int64_t ldy) {
  if (!codes || !lut || !sal || !x || !y) return CRBQ_ERR_ARG;
  if (n_ex < 0 || (n_ex > 0 && (!ex_idx || !ex_delta))) return CRBQ_ERR_ARG;
  if (dtype != CRBQ_F16 && dtype != CRBQ_BF16) return CRBQ_ERR_ARG;
  if (R <= 0 || C <= 0 || ntok <= 0 || R > 0x7fffffff || C > 0x7fffffff || ntok > 0x7fffffff ||
      ldx < C || ldy < R)
    return CRBQ_ERR_ARG;
  const int64_t nblk = (C + crbq::PB - 1) / crbq::PB;
  if (ldc < nblk * 32 || (ldc & 7) || (ldx & 7) || (((uintptr_t)x) & 15) ||
      (((uintptr_t)lut) & 15) || (((uintptr_t)codes) & 7) || (((uintptr_t)sal) & 3))
    return CRBQ_ERR_ARG;
  return CRBQ_OK;
}

template <bool END>
static int gemv_go(const uint8_t* codes, int64_t ldc, const void* lut, const uint8_t* sal,
                   int dtype, int64_t R, int64_t C, const void* x, int64_t ldx, int nvec, void* y,
                   int64_t ldy, const crbq::PkEnd& end, hipStream_t s) {
  const int nblk = (int)((C + crbq::PB - 1) / crbq::PB);
  const unsigned grid = (unsigned)((R + 15) / 16);
  if (dtype == CRBQ_BF16)
    crbq::k_gemv_packed<b8_t, END><<<grid, 64 * crbq::GV_WAVES, 0, s>>>(
        codes, ldc, (const uint16_t*)lut, sal, (int)R, (int)C, nblk, (const uint16_t*)x, ldx,
        nvec, y, ldy, end);
  else
    crbq::k_gemv_packed<h8_t, END><<<grid, 64 * crbq::GV_WAVES, 0, s>>>(
        codes, ldc, (const uint16_t*)lut, sal, (int)R, (int)C, nblk, (const uint16_t*)x, ldx,
        nvec, y, ldy, end);
  CRBQ_LAUNCH_CHECK();
  return CRBQ_OK;
}

static size_t gemm_ws_bytes(const crbq::GmPlan& p, int64_t R, int64_t T) {
  return p.ns > 1 ? (size_t)p.ns * (size_t)T * (size_t)R * sizeof(float) : 0;
}

// END: y is [ntok][ldy] in the weights' dtype, else fp32.
template <bool END>
static int gemm_go(const uint8_t* codes, int64_t ldc, const void* lut, const uint8_t* sal,
                   int dtype, int64_t R, int64_t C, const void* x, int64_t ldx, int64_t ntok,
                   void* y, int64_t ldy, const crbq::PkEnd& end, void* ws, size_t ws_bytes,
                   hipStream_t s) {
  const int nblk = (int)((C + crbq::PB - 1) / crbq::PB);
  crbq::GmPlan p = crbq::gemm_packed_plan(R, C, ntok);
  const size_t need = gemm_ws_bytes(p, R, ntok);
  if (need && (!ws || ws_bytes < need)) {
    const int64_t room = ws ? (int64_t)(ws_bytes / ((size_t)ntok * (size_t)R * sizeof(float))) : 0;
    if (END || room < crbq::gemm_packed_least(R, C, ntok)) return CRBQ_ERR_WORKSPACE;
    p = crbq::gemm_packed_plan(R, C, ntok, room);
  }
  if (p.tok_tiles > 65535) return CRBQ_ERR_ARG;
  const dim3 grid((unsigned)p.row_tiles, (unsigned)p.tok_tiles, (unsigned)p.ns);
  const bool split = p.ns > 1;
  void* out = split ? ws : y;
  const int64_t ldo = split ? R : ldy;
#define CRBQ_GM_LAUNCH(T8, TG, RT, E)                                                           \
  crbq::k_gemm_packed<T8, TG, RT, E><<<grid, 64 * crbq::GM_WAVES, 0, s>>>(                      \
      codes, ldc, (const uint16_t*)lut, sal, (int)R, (int)C, nblk, (const uint16_t*)x, ldx,     \
      (int)ntok, p.tt, p.bps, out, ldo, end)
#define CRBQ_GM_TILE(T8, E)                                                               \
  do {                                                                                    \
    if (p.rt == 2) {                                                                      \
      if (p.tg == 8) CRBQ_GM_LAUNCH(T8, 8, 2, E); else CRBQ_GM_LAUNCH(T8, 4, 2, E);       \
    } else {                                                                              \
      if (p.tg == 8) CRBQ_GM_LAUNCH(T8, 8, 1, E); else CRBQ_GM_LAUNCH(T8, 4, 1, E);       \
    }                                                                                     \
  } while (0)
  if (END && !split) {
    if (dtype == CRBQ_BF16) CRBQ_GM_TILE(b8_t, true); else CRBQ_GM_TILE(h8_t, true);
  } else {
    if (dtype == CRBQ_BF16) CRBQ_GM_TILE(b8_t, false); else CRBQ_GM_TILE(h8_t, false);
  }
#undef CRBQ_GM_TILE
#undef CRBQ_GM_LAUNCH
  CRBQ_LAUNCH_CHECK();
  if (split) {
    const dim3 sg((unsigned)((R + 1023) / 1024), (unsigned)std::min<int64_t>(ntok, 65535));
    crbq::k_gemm_packed_sum<END><<<sg, 256, 0, s>>>((const float*)ws, p.ns, (int)ntok, (int)R,
                                                    (int)C, (const uint16_t*)x, ldx, y, ldy, end);
    CRBQ_LAUNCH_CHECK();
  }
  return CRBQ_OK;
}

extern "C" int crbq_gemv_packed(const uint8_t* codes, int64_t ldc, const void* lut,
                                const uint8_t* sal, const int64_t* ex_idx,
                                const float* ex_delta, int64_t n_ex, int dtype, int64_t R,
                                int64_t C, const void* x, int64_t ldx, int nvec, float* y,
                                int64_t ldy, void* stream) {
  if (nvec < 1 || nvec > crbq::GV_MAXVEC) return CRBQ_ERR_ARG;
  int st = packed_check(codes, ldc, lut, sal, ex_idx, ex_delta, n_ex, dtype, R, C, x, ldx, nvec,
                        y, ldy);
  if (st) return st;
  hipStream_t s = (hipStream_t)stream;
  st = gemv_go<false>(codes, ldc, lut, sal, dtype, R, C, x, ldx, nvec, y, ldy, crbq::PkEnd{}, s);
  if (st) return st;
  return apply_ex(ex_idx, ex_delta, n_ex, R, C, x, ldx, dtype, nvec, y, ldy, s);
}

extern "C" size_t crbq_gemm_packed_workspace_size(int64_t R, int64_t C, int64_t ntok) {
  if (R <= 0 || C <= 0 || ntok <= 0) return 0;
  return gemm_ws_bytes(crbq::gemm_packed_plan(R, C, ntok), R, ntok);
}

extern "C" int crbq_gemm_packed(const uint8_t* codes, int64_t ldc, const void* lut,
                                const uint8_t* sal, const int64_t* ex_idx,
                                const float* ex_delta, int64_t n_ex, int dtype, int64_t R,
                                int64_t C, const void* x, int64_t ldx, int64_t ntok, float* y,
                                int64_t ldy, void* ws, size_t ws_bytes, void* stream) {
  int st = packed_check(codes, ldc, lut, sal, ex_idx, ex_delta, n_ex, dtype, R, C, x, ldx, ntok,
                        y, ldy);
  if (st) return st;
  hipStream_t s = (hipStream_t)stream;
  st = gemm_go<false>(codes, ldc, lut, sal, dtype, R, C, x, ldx, ntok, y, ldy, crbq::PkEnd{}, ws,
                      ws_bytes, s);
  if (st) return st;
  return apply_ex(ex_idx, ex_delta, n_ex, R, C, x, ldx, dtype, ntok, y, ldy, s);
}

extern "C" int crbq_linear_packed(const uint8_t* codes, int64_t ldc, const void* lut,
                                  const uint8_t* sal, const int64_t* ex_idx,
                                  const float* ex_delta, int64_t n_ex, int dtype, int64_t R,
                                  int64_t C, const void* x, int64_t ldx, int64_t ntok,
                                  const void* bias, void* y, int64_t ldy, void* ws,
                                  size_t ws_bytes, void* stream) {
  const int st = packed_check(codes, ldc, lut, sal, ex_idx, ex_delta, n_ex, dtype, R, C, x, ldx,
                              ntok, y, ldy);
  if (st) return st;
  if (n_ex > CRBQ_LINEAR_MAX_EX) return CRBQ_ERR_ARG;
  const crbq::PkEnd end{(const uint16_t*)bias, ex_idx, ex_delta, (int)n_ex, dtype == CRBQ_BF16};
  hipStream_t s = (hipStream_t)stream;
  if (ntok <= crbq::GV_MAXVEC)
    return gemv_go<true>(codes, ldc, lut, sal, dtype, R, C, x, ldx, (int)ntok, y, ldy, end, s);
  return gemm_go<true>(codes, ldc, lut, sal, dtype, R, C, x, ldx, ntok, y, ldy, end, ws, ws_bytes,
                       s);
}
