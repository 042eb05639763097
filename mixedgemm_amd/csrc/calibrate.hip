// Calibration step that produces the reorder index: per-channel absolute maximum over the rows of
// a bf16 activation sample, channels sorted by it in ascending order, index as int16 (the commented
// lines main.py:31-33 of the reference: torch.max(torch.abs(X), dim=0) -> torch.sort ascending ->
// .to(torch.int16)).  Ties are broken by channel number (a stable sort; torch.sort leaves the
// order of equal keys open).
//
// Two launches.  Pass 1 (HBM-bound, reads X once): a workgroup reduces a strip of rows for a group of
// kColLanes * 8 columns -- kColLanes lanes wide with 16-byte loads, 256 / kColLanes lanes deep over the
// rows --, folds its row lanes through LDS and writes one row of partial maxima (the bf16 bit patterns with
// the sign cleared order like the values).  The strips are few (kStrips), so that pass 2 can afford to fold
// them in every workgroup: each folds the partials of all K channels into unique 32-bit keys
// (absmax bits << 16 | channel) in LDS and ranks 16 channels against all keys.  Wide layers sort and search instead, in
// two launches (see kRankMost).
#include "mg_common.h"

namespace mg {

namespace {

constexpr int kStrips = 8;                   // row strips of pass 1 = rows of partial maxima
constexpr int kColLanes = 16;                // lanes across the columns of a group
constexpr int kRowLanes = 256 / kColLanes;   // lanes over the rows of a strip
constexpr int kColsPerGroup = kColLanes * 8;
constexpr int kInFlight = 8;                 // loads a lane has outstanding

typedef unsigned short v2h __attribute__((ext_vector_type(2)));

// The larger of both halves, one instruction (as masks, shifts and two maxima seven of them per dword: M = 4096, K = 4096 13.3 us, now 12.8
// with this and the arguments of the absmax pass fetched at once; 300 rows 8.3 -> 8.0; M = 1000, K = 2048 9.25 -> 8.7).
__device__ __forceinline__ unsigned max_halves(unsigned a, unsigned b) {
  return __builtin_bit_cast(unsigned, __builtin_elementwise_max(__builtin_bit_cast(v2h, a), __builtin_bit_cast(v2h, b)));
}

__device__ __forceinline__ void absmax_fold(v4u& m, const v4u& v) {
#pragma unroll
  for (int j = 0; j < 4; ++j) m[j] = max_halves(m[j], v[j] & 0x7fff7fffu);   // |x| of both halves
}

__global__ void __launch_bounds__(256)
column_absmax_kernel(const uint16_t* __restrict__ x, int rows, int K, uint16_t* __restrict__ partial) {
  __shared__ v4u part[kRowLanes][kColLanes];
  asm volatile("" : : "s"(x), "s"(rows), "s"(K), "s"(partial));   // all arguments in one batch of loads
  const int strip = blockIdx.y, nstrips = gridDim.y;
  const int cl = threadIdx.x % kColLanes, rl = threadIdx.x / kColLanes;
  const int c0 = blockIdx.x * kColsPerGroup + cl * 8;
  const int r0 = (int)((long long)rows * strip / nstrips), r1 = (int)((long long)rows * (strip + 1) / nstrips);
  v4u m = {0, 0, 0, 0};
  if (c0 < K) {   // K is a multiple of 32, so a lane's 8 columns are all inside or all outside
    int r = r0 + rl;
    const uint16_t* p = x + (size_t)r * K + c0;
    const size_t step = (size_t)kRowLanes * K;
    for (; r + (kInFlight - 1) * kRowLanes < r1; r += kInFlight * kRowLanes) {
      v4u v[kInFlight];
#pragma unroll
      for (int u = 0; u < kInFlight; ++u) v[u] = *reinterpret_cast<const v4u*>(p + u * step);
      p += kInFlight * step;
#pragma unroll
      for (int u = 0; u < kInFlight; ++u) absmax_fold(m, v[u]);
    }
    for (; r < r1; r += kRowLanes) {
      absmax_fold(m, *reinterpret_cast<const v4u*>(p));
      p += step;
    }
  }
  part[rl][cl] = m;
  __syncthreads();
  if (threadIdx.x < kColLanes && c0 < K) {
    v4u best = part[0][cl];
#pragma unroll
    for (int s = 1; s < kRowLanes; ++s) {
      const v4u v = part[s][cl];
#pragma unroll
      for (int j = 0; j < 4; ++j) best[j] = max_halves(best[j], v[j]);
    }
    *reinterpret_cast<v4u*>(partial + (size_t)strip * K + c0) = best;
  }
}

// The keys are unique, so the position of a channel in the sorted order is the number of smaller keys.
// Every workgroup folds the strips of partial maxima for all K channels (8 channels per lane and pass) into the
// keys, kept in LDS, and ranks 16 channels: a lane counts, for channel lane % 16, the smaller keys in one
// of kRankSlices slices of the K keys (sixteen lanes of a wave read the same 16 bytes of LDS: a broadcast), the counts
// of a channel are added through LDS, and the channel number is scattered to its rank.  K^2 compares in total over
// K/16 workgroups of 8 waves (two per SIMD: one wave's LDS latency under the other's compares).
constexpr int kRankChannels = 16, kRankSlices = 32, kRankThreads = kRankChannels * kRankSlices;

__global__ void __launch_bounds__(kRankThreads)
rank_channels_kernel(const uint16_t* __restrict__ partial, int nstrips, int K, int16_t* __restrict__ idx) {
  extern __shared__ __align__(16) unsigned lds_keys[];   // K keys, then kRankSlices x kRankChannels counts
  int* counts = reinterpret_cast<int*>(lds_keys + K);
  for (int c0 = threadIdx.x * 8; c0 < K; c0 += kRankThreads * 8) {
    // all strips requested at once (a strip past the last one reads the last one again: a maximum does not mind)
    v4u v[kStrips];
    const uint16_t* p = partial + c0;
#pragma unroll
    for (int s = 0; s < kStrips; ++s) v[s] = *reinterpret_cast<const v4u*>(p + (size_t)min(s, nstrips - 1) * K);
    v4u m = v[0];
#pragma unroll
    for (int s = 1; s < kStrips; ++s)
#pragma unroll
      for (int j = 0; j < 4; ++j) m[j] = max_halves(m[j], v[s][j]);
    v4u k0, k1;
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      k0[2 * j] = (m[j] << 16) | (unsigned)(c0 + 2 * j);
      k0[2 * j + 1] = (m[j] & 0xffff0000u) | (unsigned)(c0 + 2 * j + 1);
      k1[2 * j] = (m[2 + j] << 16) | (unsigned)(c0 + 4 + 2 * j);
      k1[2 * j + 1] = (m[2 + j] & 0xffff0000u) | (unsigned)(c0 + 4 + 2 * j + 1);
    }
    *reinterpret_cast<v4u*>(lds_keys + c0) = k0;
    *reinterpret_cast<v4u*>(lds_keys + c0 + 4) = k1;
  }
  __syncthreads();
  const int ch = threadIdx.x % kRankChannels, slice = threadIdx.x / kRankChannels;
  const int c = blockIdx.x * kRankChannels + ch;
  const unsigned mine = c < K ? lds_keys[c] : 0u;
  const int chunk = ceil_div(K / 4, kRankSlices) * 4;
  const int j0 = slice * chunk, j1 = min(K, j0 + chunk);
  int rank = 0;
#pragma unroll 8
  for (int j = j0; j < j1; j += 4) {
    const v4u q = *reinterpret_cast<const v4u*>(lds_keys + j);
#pragma unroll
    for (int e = 0; e < 4; ++e) rank += q[e] < mine ? 1 : 0;
  }
  counts[slice * kRankChannels + ch] = rank;
  __syncthreads();
  if (threadIdx.x < kRankChannels && c < K) {
    int total = 0;
#pragma unroll
    for (int s = 0; s < kRankSlices; ++s) total += counts[s * kRankChannels + ch];
    idx[total] = (int16_t)c;
  }
}

// Wide layers (K > kRankMost): K^2 compares, and K/16 workgroups that each fold all partial maxima, are most of the time.
// So two launches instead: each workgroup of the first folds 256 channels and sorts their keys (every key ranked against
// the 256), one of the second holds all sorted chunks in LDS and ranks 128 keys by binary search in every chunk, four
// threads per key with a quarter of the chunks each: 9 K / 256 steps per key instead of K.  Bound by latency and the
// LDS reads of the searches.  Calibration as a whole, M = 300: K = 6144 11.1 -> 12.3 us (not taken), 8192
// 13.0 -> 12.1, 14336 27.4 -> 15.0, 18944 40.6 -> 17.0, 32736 131 -> 23; M = 4096, K = 14336 46 -> 34.
constexpr int kRankMost = 7168;
constexpr int kChunk = 256, kSearchKeys = 128, kSearchThreads = 4 * kSearchKeys;

__global__ void __launch_bounds__(kChunk)
sort_chunks_kernel(const uint16_t* __restrict__ partial, int nstrips, int K, unsigned* __restrict__ sorted) {
  __shared__ __align__(16) unsigned keys[kChunk];
  const int c0 = blockIdx.x * kChunk, t = threadIdx.x;
  keys[t] = 0xffffffffu;   // past the last channel: larger than every key
  __syncthreads();
  if (t < kChunk / 8 && c0 + t * 8 < K) {   // K is a multiple of 32: a lane's 8 channels are all inside or all outside
    const uint16_t* p = partial + c0 + t * 8;
    v4u m = *reinterpret_cast<const v4u*>(p);
#pragma unroll
    for (int s = 1; s < kStrips; ++s) absmax_fold(m, *reinterpret_cast<const v4u*>(p + (size_t)min(s, nstrips - 1) * K));
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      keys[t * 8 + 2 * j] = (m[j] << 16) | (unsigned)(c0 + t * 8 + 2 * j);
      keys[t * 8 + 2 * j + 1] = (m[j] & 0xffff0000u) | (unsigned)(c0 + t * 8 + 2 * j + 1);
    }
  }
  __syncthreads();
  const unsigned mine = keys[t];
  int rank = 0;
#pragma unroll 8
  for (int j = 0; j < kChunk; j += 4) {
    const v4u q = *reinterpret_cast<const v4u*>(keys + j);
#pragma unroll
    for (int e = 0; e < 4; ++e) rank += q[e] < mine ? 1 : 0;
  }
  // (the keys past the last channel are equal: they keep their places at the end)
  sorted[c0 + (c0 + t < K ? rank : t)] = mine;
}

__global__ void __launch_bounds__(kSearchThreads)
rank_sorted_kernel(const unsigned* __restrict__ sorted, int K, int16_t* __restrict__ idx) {
  extern __shared__ __align__(16) unsigned chunks[];   // all chunks, then four counts per key
  const int nchunks = ceil_div(K, kChunk), total = nchunks * kChunk;
  int* counts = reinterpret_cast<int*>(chunks + total);
#pragma unroll 4
  for (int j = threadIdx.x * 4; j < total; j += kSearchThreads * 4)
    *reinterpret_cast<v4u*>(chunks + j) = *reinterpret_cast<const v4u*>(sorted + j);
  __syncthreads();
  const int key = threadIdx.x % kSearchKeys, part = threadIdx.x / kSearchKeys;
  const unsigned mine = chunks[blockIdx.x * kSearchKeys + key];
  int rank = 0;
  // several chunks at once: the steps of one search wait for each other
  constexpr int kAtOnce = 4;
  for (int c = part; c < nchunks; c += 4 * kAtOnce) {
    const unsigned* at[kAtOnce];
    int pos[kAtOnce];
#pragma unroll
    for (int u = 0; u < kAtOnce; ++u) {
      at[u] = chunks + min(c + 4 * u, nchunks - 1) * kChunk;
      pos[u] = 0;
    }
#pragma unroll
    for (int step = kChunk / 2; step >= 1; step >>= 1)
#pragma unroll
      for (int u = 0; u < kAtOnce; ++u) pos[u] += at[u][pos[u] + step - 1] < mine ? step : 0;
#pragma unroll
    for (int u = 0; u < kAtOnce; ++u)
      if (c + 4 * u < nchunks) rank += pos[u] + (at[u][pos[u]] < mine ? 1 : 0);
  }
  counts[part * kSearchKeys + key] = rank;
  __syncthreads();
  if (threadIdx.x < kSearchKeys && mine != 0xffffffffu)
    idx[counts[key] + counts[kSearchKeys + key] + counts[2 * kSearchKeys + key] + counts[3 * kSearchKeys + key]] = (int16_t)(mine & 0xffffu);
}

}  // namespace

// kStrips rows of partial maxima (K x 2 B each, a multiple of 16), and the sorted chunks of a wide layer
size_t calibrate_workspace_bytes(int K) {
  return (size_t)kStrips * K * sizeof(uint16_t) + (K > kRankMost ? (size_t)ceil_div(K, kChunk) * kChunk * sizeof(unsigned) : 0);
}

hipError_t launch_calibrate(const void* x, int rows, int K, int16_t* idx, void* workspace, hipStream_t stream) {
  uint16_t* partial = static_cast<uint16_t*>(workspace);
  // a strip has at least one row per row lane where the sample has that many rows
  const int nstrips = rows >= kStrips * kRowLanes ? kStrips : (rows + kRowLanes - 1) / kRowLanes;
  hipLaunchKernelGGL(column_absmax_kernel, dim3(ceil_div(K, kColsPerGroup), nstrips), dim3(256), 0, stream,
                     static_cast<const uint16_t*>(x), rows, K, partial);
  hipError_t e = hipGetLastError();
  if (e != hipSuccess) return e;
  if (K > kRankMost) {
    unsigned* sorted = reinterpret_cast<unsigned*>(partial + (size_t)kStrips * K);
    const int nchunks = ceil_div(K, kChunk);
    constexpr int kMostLds = 32768 * (int)sizeof(unsigned) + kSearchThreads * (int)sizeof(int);
    e = allow_dynamic_lds(reinterpret_cast<const void*>(rank_sorted_kernel), kMostLds);
    if (e != hipSuccess) return e;
    hipLaunchKernelGGL(sort_chunks_kernel, dim3(nchunks), dim3(kChunk), 0, stream, partial, nstrips, K, sorted);
    e = hipGetLastError();
    if (e != hipSuccess) return e;
    hipLaunchKernelGGL(rank_sorted_kernel, dim3(nchunks * (kChunk / kSearchKeys)), dim3(kSearchThreads),
                       (size_t)nchunks * kChunk * sizeof(unsigned) + kSearchThreads * sizeof(int), stream, sorted, K, idx);
    return hipGetLastError();
  }
  const size_t lds = (size_t)(K + kRankSlices * kRankChannels) * sizeof(unsigned);
  e = allow_dynamic_lds(reinterpret_cast<const void*>(rank_channels_kernel),
                        (32768 + kRankSlices * kRankChannels) * (int)sizeof(unsigned));
  if (e != hipSuccess) return e;
  hipLaunchKernelGGL(rank_channels_kernel, dim3(ceil_div(K, kRankChannels)), dim3(kRankThreads), lds, stream, partial, nstrips, K, idx);
  return hipGetLastError();
}

}  // namespace mg
