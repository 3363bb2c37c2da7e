// helix_direct.hip -- gfx950 kernels of the exchange between logical ranks of one device.
//
// The cp "transpose" is pure addressing (row e * cp + peer on both sides), so the
// exchange is a copy in rows: what bounds it is the memory system, and from
// where the ranks' memory is in reach the only work is to read every byte once
// and write it once. Against the same exchange through FIFO lines (write, read
// back): cp = 8, T = 256, rows of 2 KiB 24 -> 10 us, rows of 16 KiB at T = 128
// 83 -> 46 us (5.9 TB/s, a plain copy of 1 GiB reaches 6.2), cp = 16, T = 1024,
// rows of 512 bytes 93 -> 43 us.
#include "helix_direct.hpp"

namespace helix {
namespace {

using u32x2 = uint32_t __attribute__((ext_vector_type(2)));
using u32x4 = uint32_t __attribute__((ext_vector_type(4)));

// buffer cache-policy immediates: bit 0 sc0, bit 1 nt, bit 4 sc1
constexpr int kAuxNone = 0;
constexpr int kAuxNt = 2;
constexpr int kAuxNtSc1 = 18;
constexpr uint32_t kRsrcWord3 = 0x00020000u;   // raw buffer, 32-bit data format
constexpr uint32_t kOutOfRange = 0x80000000u;  // beyond any descriptor (extents are < 2 GiB): how a lane opts out
constexpr uint32_t kStatusBrokenWorkspace = 8u;
constexpr int kBlockWaves = 4;
constexpr int kBlockThreads = kBlockWaves * kWaveLanes;

__device__ __forceinline__ __amdgpu_buffer_rsrc_t make_rsrc(const void* base, uint32_t bytes) {
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(base), 0, static_cast<int>(bytes), kRsrcWord3);
}

// Whether the workspace was broken before this launch, read through the scalar cache (empty at every launch).
__device__ __forceinline__ bool broken_at_launch(const DirectArgs& a) {
  using ConstWord = const __attribute__((address_space(4))) uint64_t;
  return *reinterpret_cast<ConstWord*>(reinterpret_cast<uintptr_t>(a.broken)) != 0;
}
__device__ __forceinline__ void report_broken(const DirectArgs& a) {
  if (threadIdx.x % kWaveLanes == 0) atomicOr(a.status, kStatusBrokenWorkspace);
}

using GlobalPiece = __attribute__((address_space(1))) u32x2;

// One workgroup moves kPerThread * 256 consecutive statistics pieces in the order (entry, receiver, sender,
// piece). A statistics row can be as small as 8 bytes and its neighbours go to other ranks, so the pairs are not
// kept apart here as they are for partial_o: with all ranks in one workgroup the lines that rows of different
// pairs share are fetched by one L2 and written from one L2, and every store covers cp consecutive rows of the
// receiver. The rank is a lane's own then; the 2 * cp pointers go through LDS.
template <int kPerThread>
__device__ __forceinline__ void move_statistics(const DirectArgs& a, uint64_t (&from)[kMaxCpSize], uint64_t (&to)[kMaxCpSize]) {
  const int tid = static_cast<int>(threadIdx.x);
  uint64_t mineFrom = 0, mineTo = 0;
  for (int base = 0; base < a.cpSize; base += 8) {
#pragma unroll
    for (int i = 0; i < 8; ++i) {  // eight ranks' pointers in one trip to the scalar cache
      const uint64_t f = reinterpret_cast<uint64_t>(a.rank[base + i].send1), t = reinterpret_cast<uint64_t>(a.rank[base + i].recv1);
      if (tid == base + i) {
        mineFrom = f;
        mineTo = t;
      }
    }
  }
  if (tid < kMaxCpSize) {
    from[tid] = mineFrom;
    to[tid] = mineTo;
  }
  const bool broken = broken_at_launch(a);
  __syncthreads();
  u32x2 v[kPerThread];
  uint64_t dst[kPerThread];
#pragma unroll
  for (int i = 0; i < kPerThread; ++i) {
    const uint32_t j = (blockIdx.x * kPerThread + i) * kBlockThreads + threadIdx.x;
    dst[i] = 0;
    if (j < a.pieces) {
      const uint32_t row = fast_div_by(j, a.byRowPieces);  // (e * cp + r) * cp + s
      const uint32_t off = (j - row * a.rowPieces) * kPieceBytes;
      const uint32_t er = fast_div_by(row, a.byCp);
      const uint32_t s = row - er * a.cpSize;
      const uint32_t e = fast_div_by(er, a.byCp);
      const uint32_t r = er - e * a.cpSize;
      v[i] = *reinterpret_cast<const GlobalPiece*>(from[s] + (er * a.sendStride1 + off));
      dst[i] = to[r] + ((e * a.cpSize + s) * a.recvStride1 + off);
    }
  }
  if (broken) return report_broken(a);
#pragma unroll
  for (int i = 0; i < kPerThread; ++i)
    if (dst[i] != 0) *reinterpret_cast<GlobalPiece*>(dst[i]) = v[i];
}

// A wavefront moves one access, 64 units = 1 KiB, of one (sender s, receiver r) pair: both tensors are
// wave-uniform, and the launch is as many short wavefronts as there are KiB (two or four accesses per wavefront
// measured 0-4 % slower from 64 MB up and the same below). Consecutive wavefronts take consecutive receivers, so a
// workgroup reads neighbouring rows of one tensor and the launch sweeps all tensors in order; where a row is
// shorter than an access, a workgroup takes four consecutive accesses of one pair instead (cp = 16 rows of 512 bytes
// 46.3 -> 43.7 us; rows of 2 KiB stay with the receivers side by side: 512 tokens per rank more 44.9 -> 48.0 us).
template <int kStatsPerThread, int kAuxLoad, int kAuxStore>
__global__ __launch_bounds__(kBlockThreads) void helix_direct_exchange_kernel(DirectArgs a) {
  __shared__ uint64_t from[kMaxCpSize], to[kMaxCpSize];
  if (blockIdx.x < a.statsBlocks) return move_statistics<kStatsPerThread>(a, from, to);
  const int wave = __builtin_amdgcn_readfirstlane(static_cast<int>(threadIdx.x) / kWaveLanes);
  const uint32_t w = (blockIdx.x - a.statsBlocks) * kBlockWaves + wave;
  if (w >= a.waves) return;
  const uint32_t pairs = w >> a.groupShift;
  const uint32_t t = fast_div_by(pairs, a.byCp);
  const uint32_t group = fast_div_by(t, a.byCp);
  const uint32_t r = pairs - t * a.cpSize, s = t - group * a.cpSize;
  const uint32_t chunk = (group << a.groupShift) + (w & ((1u << a.groupShift) - 1u));
  const bool broken = broken_at_launch(a);
  const __amdgpu_buffer_rsrc_t in = make_rsrc(a.rank[s].send0, a.sendBytes0);
  const __amdgpu_buffer_rsrc_t out = make_rsrc(a.rank[r].recv0, a.recvBytes0);
  const uint32_t U = chunk * kWaveLanes + threadIdx.x % kWaveLanes;
  const uint32_t e = fast_div_by(U, a.byRowUnits);
  const uint32_t off = (U - e * a.rowUnits) * kUnitBytes;
  const bool live = U < a.units;
  const u32x4 v = __builtin_amdgcn_raw_buffer_load_b128(in, live ? (e * a.cpSize + r) * a.sendStride0 + off : kOutOfRange, 0, kAuxLoad);
  if (broken) return report_broken(a);
  __builtin_amdgcn_raw_buffer_store_b128(v, out, live ? (e * a.cpSize + s) * a.recvStride0 + off : kOutOfRange, 0, kAuxStore);
}

}  // namespace

// A launch that reads and writes more than this takes its payload past the memory-side cache (256 MB) on the way
// in: what the previous kernels left there is mostly older than the inputs, or is not all of them, and a read that
// does not allocate leaves room for the writes. Measured over inputs that were just written, over rotating sets,
// and over three sets in rotation: 134 MB 20.2 -> 19.4, 25.2 -> 23.6, 19.8 -> 23.6 us; 168 MB 31.2 -> 23.8,
// 29.8 -> 28.5, 27.6 -> 28.4; 201 MB 53.2 -> 28.9, 35.2 -> 33.3, 32.0 -> 33.4; 268 MB 55.4 -> 32.8, 47.0 -> 45.0,
// 46.3 -> 44.9.
constexpr uint64_t kStreamingBytes = 150ull << 20;

// Statistics pieces up to which a thread takes one piece instead of four: below, the launch waits for the chain of
// one thread (pointers, load, store), not for memory (cp = 4, T = 64: 3.4 -> 2.7 us; an empty kernel takes 2.1).
constexpr uint32_t kShortStatsPieces = 65536;

// Wavefronts of a launch, at most: larger exchanges go out as several launches of consecutive entries.
constexpr uint64_t kMaxLaunchWaves = 1ull << 25;

hipError_t launch_direct_exchange(const KernelArgs& a, const uint64_t* broken, hipStream_t stream) {
  DirectArgs d{};
  const uint32_t cp = static_cast<uint32_t>(a.cpSize);
  d.broken = broken;
  d.status = a.status;
  d.cpSize = a.cpSize;
  d.sendStride0 = static_cast<uint32_t>(a.sendStride0);
  d.sendStride1 = static_cast<uint32_t>(a.sendStride1);
  d.recvStride0 = static_cast<uint32_t>(a.recvStride0);
  d.recvStride1 = static_cast<uint32_t>(a.recvStride1);
  d.byCp = fast_div(cp);
  d.rowUnits = static_cast<uint32_t>(a.field0Bytes) / kUnitBytes;
  d.byRowUnits = fast_div(d.rowUnits);
  d.rowPieces = static_cast<uint32_t>(a.field1Bytes) / kPieceBytes;
  d.byRowPieces = fast_div(d.rowPieces);
  d.groupShift = a.field0Bytes < kWaveLanes * kUnitBytes ? 2 : 0;
  const bool streaming = cp * (static_cast<uint64_t>(a.sendBytes0) + a.recvBytes0) > kStreamingBytes;
  // Rows of whole 128-byte lines are written through (their lines are complete with one store: rows of 2 KiB 11.0 ->
  // 10.1 us, of 512 bytes 46.0 -> 43.5); others leave it to the L2 to put the halves of a line together (rows of 480
  // bytes 9.8 us written through, 9.2 left there).
  bool wholeLines = a.field0Bytes % kLineBytes == 0 && a.recvStride0 % kLineBytes == 0;
  for (uint32_t r = 0; r < cp; ++r) wholeLines = wholeLines && reinterpret_cast<uintptr_t>(a.rank[r].recv0) % kLineBytes == 0;

  const uint64_t chunksPerRow = (d.rowUnits + kWaveLanes - 1) / kWaveLanes;
  const uint64_t wavesPerEntry = static_cast<uint64_t>(cp) * cp * (chunksPerRow > d.rowPieces ? chunksPerRow : d.rowPieces);
  const uint64_t entriesPerLaunch = kMaxLaunchWaves / wavesPerEntry > 0 ? kMaxLaunchWaves / wavesPerEntry : 1;
  for (uint64_t begin = 0; begin < static_cast<uint64_t>(a.entryEnd); begin += entriesPerLaunch) {
    const uint64_t left = a.entryEnd - begin;
    const uint32_t entries = static_cast<uint32_t>(left < entriesPerLaunch ? left : entriesPerLaunch);
    for (uint32_t r = 0; r < cp; ++r) {
      d.rank[r].send0 = a.rank[r].send0 + begin * cp * d.sendStride0;
      d.rank[r].send1 = a.rank[r].send1 + begin * cp * d.sendStride1;
      d.rank[r].recv0 = a.rank[r].recv0 + begin * cp * d.recvStride0;
      d.rank[r].recv1 = a.rank[r].recv1 + begin * cp * d.recvStride1;
    }
    d.sendBytes0 = entries * cp * d.sendStride0;
    d.recvBytes0 = entries * cp * d.recvStride0;
    d.units = entries * d.rowUnits;
    d.pieces = entries * cp * cp * d.rowPieces;
    const bool shortStats = !streaming && d.pieces <= kShortStatsPieces;
    const uint32_t piecesPerBlock = (shortStats ? 1 : 4) * kBlockThreads;
    d.statsBlocks = (d.pieces + piecesPerBlock - 1) / piecesPerBlock;
    const uint32_t group = 1u << d.groupShift;
    const uint32_t chunks = (d.units + kWaveLanes - 1) / kWaveLanes;
    d.waves = (chunks + group - 1) / group * group * cp * cp;
    const dim3 blocks(d.statsBlocks + (d.waves + kBlockWaves - 1) / kBlockWaves);
#define HELIX_LAUNCH_DIRECT(P, L, S) hipLaunchKernelGGL((helix_direct_exchange_kernel<P, L, S>), blocks, dim3(kBlockThreads), 0, stream, d)
    if (streaming && wholeLines) HELIX_LAUNCH_DIRECT(4, kAuxNt, kAuxNtSc1);
    else if (streaming) HELIX_LAUNCH_DIRECT(4, kAuxNt, kAuxNt);
    else if (shortStats && wholeLines) HELIX_LAUNCH_DIRECT(1, kAuxNone, kAuxNtSc1);
    else if (shortStats) HELIX_LAUNCH_DIRECT(1, kAuxNone, kAuxNt);
    else if (wholeLines) HELIX_LAUNCH_DIRECT(4, kAuxNone, kAuxNtSc1);
    else HELIX_LAUNCH_DIRECT(4, kAuxNone, kAuxNt);
#undef HELIX_LAUNCH_DIRECT
    const hipError_t err = hipGetLastError();
    if (err != hipSuccess) return err;
  }
  return hipSuccess;
}

}  // namespace helix
