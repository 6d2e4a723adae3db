// Signed LEB128 encoding of quantized feature-transformer tensors on the GPU,
// the compression of the .nnue writer (src/scripts/serialize.py:61-93,
// _encode_leb_128_array; used by _write_leb_128_array :254-257 for the FT
// bias, weights and PSQT weights).
//
// Per value: 7-bit groups from the least significant, a continuation bit on
// every byte but the last, stopping once the rest of the value is all sign
// bits and the last group's bit 6 equals the sign.  The byte stream is the
// concatenation in element order, so the encoder is a length pass, a sum of the
// lengths before each tile and a write pass:
//   leb_len_kernel:   per tile of kLebTile values its byte count, per group of
//                     kLebGroup tiles theirs
//   leb_scan_kernel:  exclusive scan of the group counts, only for more groups
//                     than a writing workgroup adds up itself
//   leb_write_kernel: per tile, its start from the counts before it, in-tile
//                     exclusive scan of the value lengths, the codes placed in
//                     LDS and stored in 16-byte pieces
// The values are read twice (the second time from the memory-side cache) and the
// codes written once.  23.4 M int16 values (47 MB, 25 MB of codes): 135 -> 40 us
// against 64-bit loops over the groups of 7 bits, one workgroup scanning every
// tile's count and a byte store per code byte.
#include <algorithm>

#include "common.h"

namespace sft {

namespace {

constexpr int kLebItems = 16;                 // values per thread
constexpr int kLebTile = kBlock * kLebItems;  // values per tile
constexpr int kLebGroup = 4;                  // tiles per length workgroup
// Groups a writing workgroup sums itself, 256 at a time (32 loads a thread at most).
constexpr int64_t kLebDirectGroups = 8192;

// Bytes of v's code: m significant bits and a sign bit in groups of 7.
__device__ __forceinline__ int leb_len(int v) {
  const int m = 32 - __clz(v ^ (v >> 31));  // 0 .. 31
  return ((m + 7) * 37) >> 8;               // (m + 7) / 7
}

// The thread's values base .. base + kLebItems - 1, zero past n (vec: 16-byte
// aligned values, a whole run in range).
template <typename T>
__device__ __forceinline__ void leb_load(const T *__restrict__ values, int64_t base, int64_t n, bool vec,
                                         int (&v)[kLebItems]) {
  constexpr int PER = 16 / sizeof(T);
  if (vec && base + kLebItems <= n) {
    i32x4 raw[kLebItems / PER];
#pragma unroll
    for (int i = 0; i < kLebItems / PER; ++i) raw[i] = reinterpret_cast<const i32x4 *>(values + base)[i];
#pragma unroll
    for (int i = 0; i < kLebItems; ++i) {
      const int w = raw[i / PER][(i % PER) * (int)sizeof(T) / 4];
      if (sizeof(T) == 4) v[i] = w;
      else v[i] = (int)(T)(w >> (8 * ((i * (int)sizeof(T)) & 3)));
    }
    return;
  }
#pragma unroll
  for (int i = 0; i < kLebItems; ++i) v[i] = base + i < n ? (int)values[base + i] : 0;
}

// Bytes of the thread's values in range.
__device__ __forceinline__ int leb_bytes(const int (&v)[kLebItems], int64_t base, int64_t n) {
  int b = 0;
#pragma unroll
  for (int i = 0; i < kLebItems; ++i) b += base + i < n ? leb_len(v[i]) : 0;
  return b;
}

__device__ __forceinline__ int wave_total(int x) {
#pragma unroll
  for (int m = 1; m < kWave; m <<= 1) x += __shfl_xor(x, m);
  return x;
}

template <typename T>
__global__ __launch_bounds__(kBlock) void leb_len_kernel(const T *__restrict__ values, int64_t n, int64_t ntiles,
                                                         int vec, int32_t *__restrict__ tile_bytes,
                                                         int64_t *__restrict__ group_bytes) {
  __shared__ int s[kLebGroup][kWavesPerBlock];
  const int wave = threadIdx.x / kWave;
  int mine[kLebGroup];
#pragma unroll
  for (int g = 0; g < kLebGroup; ++g) {
    const int64_t base = ((int64_t)blockIdx.x * kLebGroup + g) * kLebTile + (int64_t)threadIdx.x * kLebItems;
    int v[kLebItems];
    leb_load(values, base, n, vec, v);
    mine[g] = leb_bytes(v, base, n);
  }
#pragma unroll
  for (int g = 0; g < kLebGroup; ++g) {
    const int t = wave_total(mine[g]);
    if (threadIdx.x % kWave == 0) s[g][wave] = t;
  }
  __syncthreads();
  if (threadIdx.x == 0) {
    int64_t all = 0;
#pragma unroll
    for (int g = 0; g < kLebGroup; ++g) {
      const int t = s[g][0] + s[g][1] + s[g][2] + s[g][3];
      const int64_t tile = (int64_t)blockIdx.x * kLebGroup + g;
      if (tile < ntiles) tile_bytes[tile] = t;
      all += t;
    }
    group_bytes[blockIdx.x] = all;
  }
}

// group_bytes[0 .. n) becomes its exclusive scan (one workgroup).
__global__ __launch_bounds__(kBlock) void leb_scan_kernel(int64_t *__restrict__ group_bytes, int64_t n) {
  __shared__ int64_t s[kBlock];
  const int tid = threadIdx.x;
  const int64_t per = (n + kBlock - 1) / kBlock;
  const int64_t lo = min(n, (int64_t)tid * per), hi = min(n, lo + per);
  int64_t mine = 0;
  for (int64_t i = lo; i < hi; ++i) mine += group_bytes[i];
  s[tid] = mine;
  __syncthreads();
  for (int off = 1; off < kBlock; off <<= 1) {
    const int64_t v = tid >= off ? s[tid - off] : 0;
    __syncthreads();
    s[tid] += v;
    __syncthreads();
  }
  int64_t run = s[tid] - mine;
  for (int64_t i = lo; i < hi; ++i) {
    const int64_t v = group_bytes[i];
    group_bytes[i] = run;
    run += v;
  }
}

template <typename T>
__global__ __launch_bounds__(kBlock) void leb_write_kernel(const T *__restrict__ values, int64_t n, int64_t ntiles,
                                                           int vec, const int32_t *__restrict__ tile_bytes,
                                                           const int64_t *__restrict__ group_bytes, int scanned,
                                                           uint8_t *__restrict__ out, int64_t *__restrict__ out_len) {
  constexpr int kMost = sizeof(T) == 1 ? 2 : sizeof(T) == 2 ? 3 : 5;  // bytes per code
  __shared__ __align__(16) uint8_t s_out[kLebTile * kMost + 16];
  __shared__ int s_wave[kWavesPerBlock];
  __shared__ int64_t s_before[kWavesPerBlock];
  const int tid = threadIdx.x, wave = tid / kWave, lane = tid % kWave;
  const int64_t tile = blockIdx.x, group = tile / kLebGroup;
  const int64_t base = tile * kLebTile + (int64_t)tid * kLebItems;
  int v[kLebItems];
  leb_load(values, base, n, vec, v);
  // bytes before the tile: the groups before its own, then the tiles of its group
  int64_t before = 0;
  if (scanned) before = tid == 0 ? group_bytes[group] : 0;
  else
    for (int64_t g = tid; g < group; g += kBlock) before += group_bytes[g];
  if (tid < (int)(tile - group * kLebGroup)) before += tile_bytes[group * kLebGroup + tid];
#pragma unroll
  for (int m = 1; m < kWave; m <<= 1) before += __shfl_xor(before, m);
  const int mine = leb_bytes(v, base, n);
  int incl = mine;
#pragma unroll
  for (int off = 1; off < kWave; off <<= 1) {
    const int o = __shfl_up(incl, off);
    if (lane >= off) incl += o;
  }
  if (lane == kWave - 1) s_wave[wave] = incl;
  if (lane == 0) s_before[wave] = before;
  __syncthreads();
  const int64_t start = s_before[0] + s_before[1] + s_before[2] + s_before[3];
  int at = incl - mine, total = 0;
#pragma unroll
  for (int w = 0; w < kWavesPerBlock; ++w) {
    at += w < wave ? s_wave[w] : 0;
    total += s_wave[w];
  }
  // The codes in LDS at the phase of their 16-byte pieces in memory.
  uint8_t *dst = out + start;
  const int phase = (int)((uintptr_t)dst & 15);
  uint8_t *code = s_out + phase + at;
#pragma unroll
  for (int i = 0; i < kLebItems; ++i) {
    if (base + i >= n) break;
    const int len = leb_len(v[i]);
#pragma unroll
    for (int k = 0; k < kMost; ++k)
      if (k < len) code[k] = (uint8_t)(((v[i] >> (7 * k)) & 0x7f) | (k + 1 < len ? 0x80 : 0));
    code += len;
  }
  __syncthreads();
  // whole 16-byte pieces, and byte by byte the pieces shared with a neighbour
  uint8_t *piece0 = dst - phase;
  const int end = phase + total;
  for (int i = tid * 16; i < end; i += kBlock * 16) {
    if (i >= phase && i + 16 <= end) {
      *reinterpret_cast<i32x4 *>(piece0 + i) = *reinterpret_cast<const i32x4 *>(s_out + i);
    } else {
      for (int b = max(i, phase); b < min(i + 16, end); ++b) piece0[b] = s_out[b];
    }
  }
  if (tile == ntiles - 1 && tid == 0) *out_len = start + total;
}

int64_t leb_tiles(int64_t n) { return ceil_div(std::max<int64_t>(n, 1), kLebTile); }
// The tiles' counts, padded to 8 bytes, then the groups'.
int64_t leb_tile_count_bytes(int64_t ntiles) { return (ntiles * 4 + 7) / 8 * 8; }

}  // namespace

size_t leb128_workspace(int64_t n) {
  const int64_t ntiles = leb_tiles(n);
  return (size_t)(leb_tile_count_bytes(ntiles) + ceil_div(ntiles, kLebGroup) * 8);
}

int leb128_encode(const void *values, int elem, int64_t n, uint8_t *out, int64_t *out_len, void *ws, hipStream_t s) {
  const int64_t ntiles = leb_tiles(n), ngroups = ceil_div(ntiles, kLebGroup);
  int32_t *tiles = static_cast<int32_t *>(ws);
  int64_t *groups = reinterpret_cast<int64_t *>(static_cast<char *>(ws) + leb_tile_count_bytes(ntiles));
  const int vec = (uintptr_t)values % 16 == 0;
  const int scanned = ngroups > kLebDirectGroups;
  ProfScope prof(kProfLeb128, s);
#define SFT_LEB(T)                                                                                                 \
  do {                                                                                                             \
    const T *v = static_cast<const T *>(values);                                                                   \
    hipLaunchKernelGGL(leb_len_kernel<T>, dim3((unsigned)ngroups), dim3(kBlock), 0, s, v, n, ntiles, vec, tiles,   \
                       groups);                                                                                    \
    if (scanned) hipLaunchKernelGGL(leb_scan_kernel, dim3(1), dim3(kBlock), 0, s, groups, ngroups);                \
    hipLaunchKernelGGL(leb_write_kernel<T>, dim3((unsigned)ntiles), dim3(kBlock), 0, s, v, n, ntiles, vec, tiles,  \
                       groups, scanned, out, out_len);                                                             \
  } while (0)
  if (elem == 1) SFT_LEB(int8_t);
  else if (elem == 2) SFT_LEB(int16_t);
  else SFT_LEB(int32_t);
#undef SFT_LEB
  return check_launch("sft_leb128_encode");
}

}  // namespace sft
