// Load-time quantizers and the int8 embedding gather (gfx950): floating
// weights -> quantized values, row-major or already in the compute kernels'
// tile order; table rows -> fp16.  Bound by memory: one read of the input, one
// write of the output.
//
// Quantizer arithmetic (the steps of rhinoforge_amd/quant/_common.py and
// int4.py, bit for bit):
//   step = max(fp16(amax * (1 / top)), 2^-14),  q = clamp(rint(w / step), lo, hi)
// with amax over the fp16-rounded row (per channel) or over the fp32 values of
// a group of 32 / 64 / 128 (group-wise).  The product with the fp32 reciprocal
// of `top` is how the torch division by a scalar is evaluated on a device.
// w / step is a correctly rounded fp32 division: t = w r, t + r (w - t step)
// with r the correctly rounded reciprocal of step (Markstein 1990), three
// operations per value instead of a full division's ten.  A row or group whose
// step is not finite (an infinity or NaN among its values) gets q = 0, which
// is what converting the NaN quotients gives.
#include "w8a16_common.h"
#include "w8a16_internal.h"

namespace rf {

__host__ __device__ inline int i4_nibble_of(int i) { return (i & 1) ? 4 + (i >> 1) : (i >> 1); }

namespace {

enum : int { kDtF16 = RF_W8A16_DTYPE_F16, kDtBf16 = RF_W8A16_DTYPE_BF16, kDtF32 = RF_W8A16_DTYPE_F32 };

struct QuantArgs {
  const void* w;
  int64_t N, K, ldw;      // ldw in elements
  int64_t rows;           // N, padded to 16 for the tile layouts
  int chunks;             // 16-wide chunks per row, K padded to the tile for the tile layouts
  int vec;                // rows are 16-byte aligned: whole chunks are read with 16-byte loads
  int qvec;               // row-major output rows are 16-byte aligned
  int group;              // group size (group-wise kernel)
  float lo, hi, inv_top;
  uint8_t* q;
  _Float16* scale;        // [N], or [K / group][N]
};

// Sixteen consecutive values of a row as fp32; zero past K.
template <int DT>
__device__ __forceinline__ void load_chunk(const QuantArgs& a, const uint8_t* row, int64_t k0,
                                           float (&v)[16]) {
  if (k0 + 16 <= a.K && a.vec) {
    if constexpr (DT == kDtF32) {
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const floatx4 f = *reinterpret_cast<const floatx4*>(row + (k0 + 4 * i) * 4);
#pragma unroll
        for (int j = 0; j < 4; ++j) v[4 * i + j] = f[j];
      }
    } else {
      const uint4 d[2] = {load_u4(row + k0 * 2), load_u4(row + k0 * 2 + 16)};
#pragma unroll
      for (int i = 0; i < 2; ++i) {
        const uint32_t w[4] = {d[i].x, d[i].y, d[i].z, d[i].w};
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          if constexpr (DT == kDtBf16) {
            v[8 * i + 2 * j] = __builtin_bit_cast(float, w[j] << 16);
            v[8 * i + 2 * j + 1] = __builtin_bit_cast(float, w[j] & 0xffff0000u);
          } else {
            const half2v h = __builtin_bit_cast(half2v, w[j]);
            v[8 * i + 2 * j] = (float)h[0];
            v[8 * i + 2 * j + 1] = (float)h[1];
          }
        }
      }
    }
  } else {
#pragma unroll
    for (int i = 0; i < 16; ++i) {
      float f = 0.f;
      if (k0 + i < a.K) {
        if constexpr (DT == kDtF32) f = reinterpret_cast<const float*>(row)[k0 + i];
        else if constexpr (DT == kDtBf16)
          f = __builtin_bit_cast(float, (uint32_t)reinterpret_cast<const uint16_t*>(row)[k0 + i] << 16);
        else f = (float)reinterpret_cast<const _Float16*>(row)[k0 + i];
      }
      v[i] = f;
    }
  }
}

__device__ __forceinline__ _Float16 step_of(float amax, float inv_top) {
  // Rounded to fp32, then to fp16: the empty asm keeps the two from being
  // joined into one multiply that rounds once.
  float t = amax * inv_top;
  asm("" : "+v"(t));
  const _Float16 s = (_Float16)t;
  const _Float16 tiny = (_Float16)6.103515625e-05f;
  return s < tiny ? tiny : s;  // NaN stays NaN
}

// q of sixteen values in one byte each (two's complement).
__device__ __forceinline__ void quantize16(const QuantArgs& a, const float (&v)[16], float s,
                                           uint32_t (&out)[4]) {
  const bool finite = __builtin_fabsf(s) < 65536.f;
  const float r = 1.0f / s;
#pragma unroll
  for (int w = 0; w < 4; ++w) {
    uint32_t p = 0;
#pragma unroll
    for (int b = 0; b < 4; ++b) {
      const float x = v[4 * w + b];
      float t = x * r;
      t = __builtin_fmaf(__builtin_fmaf(-t, s, x), r, t);
      t = __builtin_fminf(__builtin_fmaxf(__builtin_rintf(t), a.lo), a.hi);
      const uint32_t qi = finite ? (uint32_t)(int)t & 0xffu : 0u;
      p |= qi << (8 * b);
    }
    out[w] = p;
  }
}

// Stores the chunk's values: row-major bytes, or their place in the tiles.
template <int LAYOUT>
__device__ __forceinline__ void store_chunk(const QuantArgs& a, int64_t n, int c,
                                            const uint32_t (&qv)[4]) {
  if constexpr (LAYOUT == RF_W8A16_LAYOUT_ROWMAJOR) {
    uint8_t* p = a.q + n * a.K + (int64_t)c * 16;
    if (a.qvec) {
      *reinterpret_cast<uint4*>(p) = make_uint4(qv[0], qv[1], qv[2], qv[3]);
    } else {
#pragma unroll
      for (int i = 0; i < 16; ++i)
        if ((int64_t)c * 16 + i < a.K) p[i] = (uint8_t)(qv[i >> 2] >> (8 * (i & 3)));
    }
  } else if constexpr (LAYOUT == RF_W8A16_LAYOUT_TILE16X64) {
    // tile (n / 16, c / 4), lane 16 (c % 4) + n % 16
    uint8_t* p = a.q + ((n >> 4) * (a.chunks >> 2) + (c >> 2)) * kTileBytes +
                 (16 * (c & 3) + (int)(n & 15)) * 16;
    const uint32_t f = 0x80808080u;
    *reinterpret_cast<uint4*>(p) = make_uint4(qv[0] ^ f, qv[1] ^ f, qv[2] ^ f, qv[3] ^ f);
  } else {
    // tile (n / 16, c / 8), lane 16 ((c % 8) / 2) + n % 16, its dwords 2 (c % 2) and + 1
    uint32_t d[2] = {0, 0};
#pragma unroll
    for (int i = 0; i < 16; ++i) {
      const uint32_t u = ((qv[i >> 2] >> (8 * (i & 3))) + 8u) & 0xFu;
      d[i >> 3] |= u << (4 * i4_nibble_of(i & 7));
    }
    uint8_t* p = a.q + ((n >> 4) * (a.chunks >> 3) + (c >> 3)) * kTileBytes +
                 (16 * ((c & 7) >> 1) + (int)(n & 15)) * 16 + 8 * (c & 1);
    *reinterpret_cast<uint2*>(p) = make_uint2(d[0], d[1]);
  }
}

// Per channel: one wavefront per row, four rows per workgroup.  Lane l holds
// chunks l, l + 64, ... : the first kKeep of them stay in registers between the
// amax and the rounding pass (rows up to 4096 wide are read from memory once),
// the rest are read again, from the caches.  A chunk of a tile layout is one
// 16-byte store; four rows fill 64 contiguous bytes of a tile.
// (12288 x 4096 bf16 -> TILE16X64: 31 us, 4.9 TB/s over the 151 MB it reads and
// writes, the rate of a large device copy; 636 us the call as ten elementwise
// passes, a reduction and the pack kernel.)
constexpr int kKeep = 4;
template <int DT, int LAYOUT>
__global__ __launch_bounds__(256) void quant_rows_kernel(QuantArgs a) {
  const int lane = threadIdx.x & 63;
  const int64_t n = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6);
  if (n >= a.rows) return;
  const bool real = n < a.N;
  const uint8_t* row = static_cast<const uint8_t*>(a.w) +
                       (real ? n : 0) * a.ldw * (DT == kDtF32 ? 4 : 2);
  const int real_chunks = real ? (int)((a.K + 15) / 16) : 0;
  typedef uint16_t ushort2v __attribute__((ext_vector_type(2)));
  half2v keep[kKeep][8];
  ushort2v m = {0, 0};
  // Rounds a chunk to fp16 and folds |value|'s bits into m: as unsigned numbers
  // they order like the magnitudes, with NaN above infinity.
  auto fold = [&](int64_t k0, half2v (&h)[8]) {
    float v[16];
    load_chunk<DT>(a, row, k0, v);
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      h[i] = half2v{(_Float16)v[2 * i], (_Float16)v[2 * i + 1]};
      const ushort2v b = __builtin_bit_cast(ushort2v, __builtin_bit_cast(uint32_t, h[i]) & 0x7fff7fffu);
      m = __builtin_elementwise_max(m, b);
    }
  };
#pragma unroll
  for (int i = 0; i < kKeep; ++i) {
#pragma unroll
    for (int j = 0; j < 8; ++j) keep[i][j] = half2v{(_Float16)0.f, (_Float16)0.f};
    if (i * 64 + lane < real_chunks) fold((int64_t)(i * 64 + lane) * 16, keep[i]);
  }
  for (int c = kKeep * 64 + lane; c < real_chunks; c += 64) {
    half2v h[8];
    fold((int64_t)c * 16, h);
  }
  uint32_t mx = m[0] > m[1] ? m[0] : m[1];
#pragma unroll
  for (int w = 32; w > 0; w >>= 1) {
    const uint32_t o = (uint32_t)__shfl_xor((int)mx, w);
    mx = o > mx ? o : mx;
  }
  const _Float16 s16 = step_of((float)__builtin_bit_cast(_Float16, (uint16_t)mx), a.inv_top);
  if (real && lane == 0) a.scale[n] = s16;
  const float s = (float)s16;
  auto emit = [&](int c, const half2v (&h)[8]) {
    float v[16];
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      v[2 * i] = (float)h[i][0];
      v[2 * i + 1] = (float)h[i][1];
    }
    uint32_t qv[4];
    quantize16(a, v, s, qv);
    store_chunk<LAYOUT>(a, n, c, qv);
  };
#pragma unroll
  for (int i = 0; i < kKeep; ++i)
    if (i * 64 + lane < a.chunks) emit(i * 64 + lane, keep[i]);
  for (int c = kKeep * 64 + lane; c < a.chunks; c += 64) {
    half2v h[8];
#pragma unroll
    for (int j = 0; j < 8; ++j) h[j] = half2v{(_Float16)0.f, (_Float16)0.f};
    if (c < real_chunks) fold((int64_t)c * 16, h);
    emit(c, h);
  }
}

// Group-wise int4: one wavefront per row and run of 64 chunks (1024 values); a
// group is 2, 4 or 8 neighbouring lanes, so everything stays in registers and
// the input is read once (12288 x 4096 bf16, groups of 32: 29 us).
template <int DT, int LAYOUT>
__global__ __launch_bounds__(256) void quant_groups_kernel(QuantArgs a) {
  const int lane = threadIdx.x & 63;
  const int64_t n = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6);
  const int c = blockIdx.y * 64 + lane;
  if (n >= a.rows) return;
  const int64_t k0 = (int64_t)c * 16;
  float v[16];
#pragma unroll
  for (int i = 0; i < 16; ++i) v[i] = 0.f;
  const bool real = n < a.N && k0 < a.K;  // K is a multiple of the group, so of 16
  if (real)
    load_chunk<DT>(a, static_cast<const uint8_t*>(a.w) + n * a.ldw * (DT == kDtF32 ? 4 : 2), k0, v);
  uint32_t mx = 0;
#pragma unroll
  for (int i = 0; i < 16; ++i) {
    const uint32_t b = __builtin_bit_cast(uint32_t, v[i]) & 0x7fffffffu;
    mx = b > mx ? b : mx;
  }
  const int lanes = a.group >> 4;
#pragma unroll
  for (int w = 1; w < 8; w <<= 1) {
    const uint32_t o = (uint32_t)__shfl_xor((int)mx, w);
    if (w < lanes) mx = o > mx ? o : mx;
  }
  const _Float16 s16 = step_of(__builtin_bit_cast(float, mx), a.inv_top);
  if (real && (lane & (lanes - 1)) == 0) a.scale[(k0 / a.group) * a.N + n] = s16;
  if (c >= a.chunks) return;
  uint32_t qv[4];
  quantize16(a, v, (float)s16, qv);
  store_chunk<LAYOUT>(a, n, c, qv);
}

// Row gather of an int8 table: y[m][h] = fp16(f32(q[id][h]) * f32(s[id])), the
// product exact in fp32 and rounded once.  One workgroup per 256 * VEC outputs
// of a row; VEC int8 values per thread (16-byte loads, 32-byte stores).
template <int VEC, typename Id>
__global__ __launch_bounds__(256) void embed_kernel(const int8_t* __restrict__ table, int64_t V,
                                                    int64_t H, const _Float16* __restrict__ scale,
                                                    const Id* __restrict__ ids, int per_row,
                                                    _Float16* __restrict__ y) {
  const int64_t m = blockIdx.x / (uint32_t)per_row;
  const int64_t h = ((int64_t)(blockIdx.x - (uint32_t)m * (uint32_t)per_row) * 256 + threadIdx.x) * VEC;
  int64_t id = (int64_t)ids[m];
  if (id < 0) id += V;  // as torch indexing counts from the end
  // An id outside the table gives a row of NaN (a trap would end the process).
  const bool inside = (uint64_t)id < (uint64_t)V;
  if (!inside) id = 0;
  if (h >= H) return;
  const float s = inside ? (float)scale[id] : __builtin_nanf("");
  const int8_t* q = table + id * H + h;
  _Float16* o = y + m * H + h;
  if constexpr (VEC == 1) {
    *o = (_Float16)((float)*q * s);
  } else {
    uint32_t d[VEC / 4];
    if constexpr (VEC == 16) {
      const uint4 t = load_u4(q);
      d[0] = t.x; d[1] = t.y; d[2] = t.z; d[3] = t.w;
    } else {
      const uint2 t = *reinterpret_cast<const uint2*>(q);
      d[0] = t.x; d[1] = t.y;
    }
    uint32_t r[VEC / 2];
#pragma unroll
    for (int i = 0; i < VEC / 2; ++i) {
      const int b = 2 * i;
      const float f0 = (float)(int8_t)(d[b >> 2] >> (8 * (b & 3))) * s;
      const float f1 = (float)(int8_t)(d[b >> 2] >> (8 * (b & 3) + 8)) * s;
      r[i] = __builtin_bit_cast(uint32_t, half2v{(_Float16)f0, (_Float16)f1});
    }
#pragma unroll
    for (int i = 0; i < VEC / 8; ++i)
      reinterpret_cast<uint4*>(o)[i] = make_uint4(r[4 * i], r[4 * i + 1], r[4 * i + 2], r[4 * i + 3]);
  }
}

template <int DT>
hipError_t launch_quant_t(const QuantArgs& a, int layout, hipStream_t stream) {
  const dim3 block(256);
  const int64_t gx = ceil_div(a.rows, 4);
  if (gx >= (int64_t)1 << 24) return hipErrorInvalidValue;  // (fewer than 2^32 threads along x)
  if (a.group) {
    const int64_t gy = ceil_div(a.chunks, 64);
    if (gy > 65535) return hipErrorInvalidValue;
    const dim3 grid((unsigned)gx, (unsigned)gy);
    if (layout == RF_W8A16_LAYOUT_ROWMAJOR)
      hipLaunchKernelGGL((quant_groups_kernel<DT, RF_W8A16_LAYOUT_ROWMAJOR>), grid, block, 0, stream, a);
    else
      hipLaunchKernelGGL((quant_groups_kernel<DT, RF_W8A16_LAYOUT_TILE16X128_I4>), grid, block, 0, stream, a);
    return hipGetLastError();
  }
  const dim3 grid((unsigned)gx);
  switch (layout) {
    case RF_W8A16_LAYOUT_ROWMAJOR:
      hipLaunchKernelGGL((quant_rows_kernel<DT, RF_W8A16_LAYOUT_ROWMAJOR>), grid, block, 0, stream, a);
      break;
    case RF_W8A16_LAYOUT_TILE16X64:
      hipLaunchKernelGGL((quant_rows_kernel<DT, RF_W8A16_LAYOUT_TILE16X64>), grid, block, 0, stream, a);
      break;
    default:
      hipLaunchKernelGGL((quant_rows_kernel<DT, RF_W8A16_LAYOUT_TILE16X128_I4>), grid, block, 0, stream, a);
  }
  return hipGetLastError();
}

template <int VEC>
hipError_t launch_embed_t(const int8_t* table, int64_t V, int64_t H, const _Float16* scale,
                          const void* ids, bool ids64, int64_t M, _Float16* y, hipStream_t stream) {
  // A launch holds fewer than 2^32 threads along x, so fewer than 2^24
  // workgroups of 256; more rows than that take several launches.
  const int64_t per_row = ceil_div(H, 256 * VEC);
  const int64_t rows = (((int64_t)1 << 24) - 1) / per_row;
  if (rows < 1) return hipErrorInvalidValue;
  for (int64_t m0 = 0; m0 < M; m0 += rows) {
    const dim3 grid((unsigned)((M - m0 < rows ? M - m0 : rows) * per_row));
    if (ids64)
      hipLaunchKernelGGL((embed_kernel<VEC, int64_t>), grid, dim3(256), 0, stream, table, V, H, scale,
                         static_cast<const int64_t*>(ids) + m0, (int)per_row, y + m0 * H);
    else
      hipLaunchKernelGGL((embed_kernel<VEC, int32_t>), grid, dim3(256), 0, stream, table, V, H, scale,
                         static_cast<const int32_t*>(ids) + m0, (int)per_row, y + m0 * H);
    const hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;
  }
  return hipSuccess;
}

bool aligned_to(const void* p, size_t n) { return (uintptr_t)p % n == 0; }

}  // namespace

hipError_t launch_quantize(const void* w, int dtype, int64_t N, int64_t K, int64_t ldw, int bits,
                           int group, int layout, void* q, void* scale, hipStream_t stream) {
  QuantArgs a;
  const int size = dtype == kDtF32 ? 4 : 2;
  const int64_t tk = layout == RF_W8A16_LAYOUT_TILE16X64 ? 64
                     : layout == RF_W8A16_LAYOUT_TILE16X128_I4 ? 128 : 16;
  a.w = w;
  a.N = N;
  a.K = K;
  a.ldw = ldw;
  a.rows = layout == RF_W8A16_LAYOUT_ROWMAJOR ? N : round_up(N, 16);
  const int64_t chunks = round_up(K, tk) / 16;
  if (chunks > 0x3fffffff) return hipErrorInvalidValue;
  a.chunks = (int)chunks;
  a.vec = aligned_to(w, 16) && (ldw * size) % 16 == 0;
  a.qvec = aligned_to(q, 16) && K % 16 == 0;
  a.group = group;
  a.hi = bits == 8 ? 127.f : 7.f;
  a.lo = -a.hi - 1.f;
  a.inv_top = 1.0f / a.hi;
  a.q = static_cast<uint8_t*>(q);
  a.scale = static_cast<_Float16*>(scale);
  switch (dtype) {
    case kDtF16: return launch_quant_t<kDtF16>(a, layout, stream);
    case kDtBf16: return launch_quant_t<kDtBf16>(a, layout, stream);
    default: return launch_quant_t<kDtF32>(a, layout, stream);
  }
}

hipError_t launch_embed(const int8_t* table, int64_t V, int64_t H, const void* scale,
                        const void* ids, bool ids64, int64_t M, void* y, hipStream_t stream) {
  const _Float16* s = static_cast<const _Float16*>(scale);
  _Float16* o = static_cast<_Float16*>(y);
  if (H % 16 == 0 && aligned_to(table, 16) && aligned_to(y, 16))
    return launch_embed_t<16>(table, V, H, s, ids, ids64, M, o, stream);
  if (H % 8 == 0 && aligned_to(table, 8) && aligned_to(y, 16))
    return launch_embed_t<8>(table, V, H, s, ids, ids64, M, o, stream);
  return launch_embed_t<1>(table, V, H, s, ids, ids64, M, o, stream);
}

}  // namespace rf
