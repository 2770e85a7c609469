// HBM copy and read kernels (memory_bandwidth row).
//
// Copy: every lane moves 16-byte vectors, at any address (global_load_dwordx4 /
// global_store_dwordx4); consecutive lanes touch consecutive vectors, so each
// wave64 instruction covers 1 KiB of contiguous memory. A workgroup step holds
// `vectors_per_thread` independent loads in flight before the stores. The
// cache policy is a template argument: plain, non-temporal (nt loads and
// stores), or streaming (nt loads, device-scope stores that write through the
// XCD's L2 instead of leaving dirty lines to be evicted later) - on MI355X the
// last measures ~1% faster than nt stores for HBM-sized copies.
//
// Read: a wave streams its segments of `block_elements` values with
// non-temporal 16-byte loads and reduces each to a single float (the
// reference's per-program sum): one segment of more than 4 KiB, or several that
// fill 4 KiB. Non-temporal loads stream HBM ~7% faster than plain ones on
// MI355X (88-90% of 8 TB/s against 82-84%, read-only). The summation depth
// stays below the 2*eps*log2(block) bound the reference validates block sums
// with (bench_bandwidth.py:87).
#include "mb_internal.h"

namespace mb {
namespace {

typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
typedef float f32x4 __attribute__((ext_vector_type(4)));

// Copy cache policies.
constexpr int kPlain = 0, kNontemporal = 1, kStream = 2;

// 16 bytes at any address: gfx950 takes a global_load_dwordx4 there.
typedef u32x4 u32x4_unaligned __attribute__((aligned(1)));

template <int POLICY, bool UNALIGNED>
__device__ __forceinline__ u32x4 load_elem(const u32x4* ptr) {
  if constexpr (UNALIGNED) {
    const u32x4_unaligned* at = reinterpret_cast<const u32x4_unaligned*>(ptr);
    if constexpr (POLICY != kPlain) return __builtin_nontemporal_load(at);
    return *at;
  } else {
    if constexpr (POLICY != kPlain) return __builtin_nontemporal_load(ptr);
    return *ptr;
  }
}

// Device-scope (sc1) vector stores; the compiler has no builtin for the scope
// bits. A store of more than 8 bytes needs one wait state before a VALU
// instruction rewrites its data registers, which the compiler cannot see to
// behind inline assembly.
__device__ __forceinline__ void store_sc1(u32x4* ptr, u32x4 value) {
  asm volatile("global_store_dwordx4 %0, %1, off sc1\n\ts_nop 0" ::"v"(ptr), "v"(value) : "memory");
}

template <int POLICY>
__device__ __forceinline__ void store_elem(u32x4* ptr, u32x4 value) {
  if constexpr (POLICY == kStream) {
    store_sc1(ptr, value);
  } else if constexpr (POLICY == kNontemporal) {
    __builtin_nontemporal_store(value, ptr);
  } else {
    *ptr = value;
  }
}

// n 16-byte vectors; dst is 16-byte aligned, src unless UNALIGNED too. The
// kernels pass blockDim.x: read in here, it costs every wave a load (the
// compiler then allows for a partial last workgroup; 1 GiB 330 us, not 316).
template <int VPT, int POLICY, bool UNALIGNED>
__device__ __forceinline__ void copy_vectors(const u32x4* __restrict__ src, u32x4* __restrict__ dst, uint64_t n,
                                             uint32_t block_threads) {
  const uint64_t step = static_cast<uint64_t>(block_threads) * VPT;
  const uint64_t stride = static_cast<uint64_t>(gridDim.x) * step;
  for (uint64_t base = blockIdx.x * step + threadIdx.x; base < n; base += stride) {
    // Opaque per trip: otherwise the grid-stride loop keeps one 64-bit scalar
    // pointer per vector and per operand live across trips, which exceeds the
    // SGPR file at 16 vectors per lane and spills.
    uint32_t threads = block_threads;
    asm("" : "+s"(threads));
    const u32x4* s = src + base;
    u32x4* d = dst + base;
    const uint64_t left = n - base;
    u32x4 values[VPT];
    if (left > static_cast<uint64_t>(VPT - 1) * threads) {
#pragma unroll
      for (int j = 0; j < VPT; ++j) values[j] = load_elem<POLICY, UNALIGNED>(s + j * threads);
#pragma unroll
      for (int j = 0; j < VPT; ++j) store_elem<POLICY>(d + j * threads, values[j]);
    } else {
#pragma unroll
      for (int j = 0; j < VPT; ++j)
        if (j * threads < left) values[j] = load_elem<POLICY, UNALIGNED>(s + j * threads);
#pragma unroll
      for (int j = 0; j < VPT; ++j)
        if (j * threads < left) store_elem<POLICY>(d + j * threads, values[j]);
    }
  }
}

template <int VPT, int POLICY>
__global__ void __launch_bounds__(1024) copy_kernel(const u32x4* __restrict__ src, u32x4* __restrict__ dst,
                                                     uint64_t n) {
  copy_vectors<VPT, POLICY, false>(src, dst, n, blockDim.x);
}

// A copy with `head` bytes before and `tail` bytes after its n whole vectors,
// which the first workgroup moves: dst + head is 16-byte aligned, src + head
// need not be. One launch where the body and its tail took two (8 MiB and a
// tail 6.5 -> 5.2 us), and 16-byte accesses where unaligned pointers took single
// dwords or bytes (1 GiB, one wave a workgroup, streaming: on dwords 888 -> 330
// us, on bytes 3531 -> 331; aligned it takes 317).
template <int VPT, int POLICY>
__global__ void __launch_bounds__(1024)
    copy_edges_kernel(const uint8_t* __restrict__ src, uint8_t* __restrict__ dst, uint64_t n, uint32_t head,
                      uint32_t tail) {
  copy_vectors<VPT, POLICY, true>(reinterpret_cast<const u32x4*>(src + head), reinterpret_cast<u32x4*>(dst + head), n,
                                  blockDim.x);
  if (blockIdx.x == 0) {
    const uint64_t after = head + n * 16;
    for (uint32_t i = threadIdx.x; i < head; i += blockDim.x) dst[i] = src[i];
    if (threadIdx.x < tail) dst[after + threadIdx.x] = src[after + threadIdx.x];
  }
}

// A copy of less than one whole vector.
__global__ void copy_tail_kernel(const uint8_t* __restrict__ src, uint8_t* __restrict__ dst, uint32_t n) {
  for (uint32_t i = threadIdx.x; i < n; i += blockDim.x) dst[i] = src[i];
}

// Write-only stream (the copy's store half): every 32-bit word of dst becomes
// `pattern`, one 16-byte store per lane per trip, grid-stride, with the copy's
// store policies.
// The `tail` bytes after them are the first workgroup's; byte i of the buffer
// is byte (i % 4) of the little-endian pattern (the tail starts 16-aligned).
template <int POLICY>
__global__ void __launch_bounds__(1024)
    fill_kernel(u32x4* __restrict__ dst, uint64_t n, uint32_t pattern, uint32_t tail) {
  const u32x4 value = {pattern, pattern, pattern, pattern};
  const uint64_t stride = static_cast<uint64_t>(gridDim.x) * blockDim.x;
  for (uint64_t i = blockIdx.x * static_cast<uint64_t>(blockDim.x) + threadIdx.x; i < n; i += stride)
    store_elem<POLICY>(dst + i, value);
  if (blockIdx.x == 0 && threadIdx.x < tail)
    reinterpret_cast<uint8_t*>(dst + n)[threadIdx.x] = static_cast<uint8_t>(pattern >> (8 * (threadIdx.x & 3)));
}

// A fill of less than one whole vector.
__global__ void fill_tail_kernel(uint8_t* __restrict__ dst, uint32_t n, uint32_t pattern) {
  for (uint32_t i = threadIdx.x; i < n; i += blockDim.x) dst[i] = static_cast<uint8_t>(pattern >> (8 * (i & 3)));
}

template <typename T>
__device__ __forceinline__ float to_float(T value);
template <>
__device__ __forceinline__ float to_float<float>(float value) { return value; }
template <>
__device__ __forceinline__ float to_float<_Float16>(_Float16 value) { return static_cast<float>(value); }
template <>
__device__ __forceinline__ float to_float<uint16_t>(uint16_t bits) {  // bfloat16 bit pattern
  return __uint_as_float(static_cast<uint32_t>(bits) << 16);
}

// Sum of one 16-byte vector: four floats, or eight halves, as pairwise sums.
template <typename T>
__device__ __forceinline__ float vector_sum(u32x4 raw) {
  if constexpr (sizeof(T) == 4) {
    const f32x4 v = __builtin_bit_cast(f32x4, raw);
    return (v[0] + v[1]) + (v[2] + v[3]);
  } else {
    const T* h = reinterpret_cast<const T*>(&raw);
    return ((to_float(h[0]) + to_float(h[1])) + (to_float(h[2]) + to_float(h[3]))) +
           ((to_float(h[4]) + to_float(h[5])) + (to_float(h[6]) + to_float(h[7])));
  }
}

__device__ __forceinline__ float wave_sum(float value) {
#pragma unroll
  for (int offset = 32; offset > 0; offset >>= 1) value += __shfl_xor(value, offset, 64);
  return value;
}

template <typename T>
__device__ __forceinline__ u32x4 load_vector(const T* ptr) {
  return __builtin_nontemporal_load(reinterpret_cast<const u32x4_unaligned*>(ptr));
}

// value[j] = the sum of the 16 bytes at ptr + j * 64 vectors, for N loads: all
// of them in flight before any is summed, or, `serial`, one after the other.
template <typename T, int N>
__device__ __forceinline__ void load_and_sum(float (&value)[N], const T* ptr, bool serial) {
  constexpr int VEC = 16 / sizeof(T);
  if (serial) {
#pragma unroll
    for (int j = 0; j < N; ++j) {
      value[j] = vector_sum<T>(load_vector(ptr + j * 64 * VEC));
      asm volatile("" : "+v"(ptr) : "v"(value[j]));  // the next address waits for this sum
    }
  } else {
    u32x4 raw[N];
#pragma unroll
    for (int j = 0; j < N; ++j) raw[j] = load_vector(ptr + j * 64 * VEC);
#pragma unroll
    for (int j = 0; j < N; ++j) value[j] = vector_sum<T>(raw[j]);
  }
}

// The sum of `count` elements by one wave, eight bounded loads in flight: the
// buffer's clipped last segment.
template <typename T>
__device__ __forceinline__ float clipped_sum(const T* base, uint32_t count, uint32_t lane) {
  constexpr int VEC = 16 / sizeof(T);
  const uint32_t vectors = count / VEC;
  float acc[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
  for (uint32_t p = lane; p < vectors; p += 512) {
    u32x4 raw[8];
#pragma unroll
    for (uint32_t j = 0; j < 8; ++j)
      raw[j] = p + j * 64 < vectors ? load_vector(base + (p + j * 64) * VEC) : u32x4{0, 0, 0, 0};
#pragma unroll
    for (int j = 0; j < 8; ++j) acc[j] += vector_sum<T>(raw[j]);
  }
  if (lane < count % VEC) acc[0] += to_float(base[vectors * VEC + lane]);
  return wave_sum(((acc[0] + acc[1]) + (acc[2] + acc[3])) + ((acc[4] + acc[5]) + (acc[6] + acc[7])));
}

// 16-byte vectors a wave of the packed read sums.
constexpr uint32_t kPackedVectors = 256;

// Segments of V 16-byte vectors, V from 8 to kPackedVectors: one wave sums the
// segments of 4 KiB.
//
// Bound by HBM: 1 GiB takes 150-160 us (6.7-7.2 TB/s) at every block size.
// One wave per segment, as larger blocks have it, starts and folds a wave for
// 1 KiB at FP32 blocks of 256 (220 us) and reads two bytes per lane where a
// segment is shorter than a wave's load (BF16 blocks of 256: 721 us). Here a
// lane's loads of one segment are summed first; then the values of different
// segments fold over the lanes together: at offset o, two values become one, a
// lane with bit o clear keeping the first and adding its partner's share of it,
// the others the second. That takes half the shuffles of such a step away and
// leaves each sum in the lanes that store it. Adding commutes, so a sum's tree
// is the plain butterfly's.
//
// The four loads go out together where waves are few (FP32 blocks of 1024,
// 8 MiB: 4.9 us, one by one 6.3; 256 MiB, 64-value blocks: 40.6 and 44.8) and
// from unaligned sources (1 GiB of FP32 156 and 162). Past 131072 waves (half a
// GiB here), one load per wave at a time covers the latency (32 waves of 1 KiB
// per CU) and more only disturbs the DRAM pages: 1 GiB takes 146 us one by one
// and 157 together.
template <typename T, int V>
__global__ void __launch_bounds__(1024)
    read_sum_packed_kernel(const T* __restrict__ src, float* __restrict__ sink, uint64_t elements, uint64_t chunks,
                           bool serial) {
  constexpr int VEC = 16 / sizeof(T), LOADS = kPackedVectors / 64;
  constexpr int PER_SEGMENT = V > 64 ? V / 64 : 1;       // loads of one segment
  constexpr int VALUES = LOADS / PER_SEGMENT;            // segments a lane has a share of
  constexpr int LANES = V < 64 ? V : 64;                 // lanes sharing a segment
  constexpr uint32_t SEGMENTS = LOADS * 64 / V;          // of one chunk
  const uint32_t lane = threadIdx.x & 63;
  const uint64_t waves_per_block = blockDim.x >> 6;
  const uint64_t whole = elements / (V * VEC);  // segments that are not clipped
  const uint64_t total_waves = static_cast<uint64_t>(gridDim.x) * waves_per_block;
  for (uint64_t chunk = blockIdx.x * waves_per_block + (threadIdx.x >> 6); chunk <= chunks; chunk += total_waves) {
    if (chunk == chunks) {  // after the last chunk of whole segments: the clipped one
      const uint32_t left = static_cast<uint32_t>(elements - whole * (V * VEC));
      if (left) {
        const float total = clipped_sum(src + whole * (V * VEC), left, lane);
        if (lane == 0) sink[whole] = total;
      }
      break;
    }
    const uint64_t first = chunk * SEGMENTS;
    const T* base = src + chunk * (LOADS * 64 * VEC) + lane * VEC;
    float value[LOADS];
    if (first + SEGMENTS <= whole) {
      load_and_sum(value, base, serial);
    } else {
      const uint32_t vectors = static_cast<uint32_t>(whole - first) * V;
#pragma unroll
      for (int j = 0; j < LOADS; ++j)
        value[j] = j * 64 + lane < vectors ? vector_sum<T>(load_vector(base + j * 64 * VEC)) : 0.f;
    }
    // One value per segment: pairwise over its loads.
#pragma unroll
    for (int width = 1; width < PER_SEGMENT; width *= 2)
#pragma unroll
      for (int j = 0; j < LOADS; j += 2 * width) value[j] += value[j + width];
#pragma unroll
    for (int i = 1; i < VALUES; ++i) value[i] = value[i * PER_SEGMENT];
    int values = VALUES, index = 0;
#pragma unroll
    for (int offset = LANES / 2; offset > 0; offset >>= 1) {
      if (values > 1) {
        const bool second = lane & offset;
#pragma unroll
        for (int i = 0; i < values / 2; ++i) {
          const float keep = second ? value[2 * i + 1] : value[2 * i];
          const float give = second ? value[2 * i] : value[2 * i + 1];
          value[i] = keep + __shfl_xor(give, offset, 64);
        }
        index += second ? VALUES / values : 0;  // bit 0 of the value's number first
        values /= 2;
      } else {
        value[0] += __shfl_xor(value[0], offset, 64);
      }
    }
    // Lanes whose plain-butterfly bits are clear hold one segment each (several
    // values in every lane where the lanes ran out first).
    constexpr int MERGES = VALUES == 4 ? 2 : VALUES == 2 ? 1 : 0;
    constexpr int STEPS = LANES == 64 ? 6 : LANES == 32 ? 5 : LANES == 16 ? 4 : 3;
    static_assert(MERGES <= STEPS, "every value folds away");
    constexpr uint32_t PLAIN = (1u << (STEPS - MERGES)) - 1;
    const uint64_t segment = first + index * (64 / LANES) + lane / LANES;
    if ((lane & PLAIN) == 0 && segment < whole) sink[segment] = value[0] + 0.f;
  }
}

// Segments of more than kPackedVectors 16-byte vectors: one wave per segment; waves stride
// over the segments of the buffer. Bound by HBM. `serial` is worth 2 to 6 % past
// 131072 waves, FP16 (24 waves per CU by its registers) included: 8 KiB segments
// of 4 GiB take 623 us with it and 652 without in FP32, 614 and 640 in FP16, 624
// and 644 in BF16; 32 KiB segments of 8 GiB 1274 and 1296, 1232 and 1305, 1257
// and 1301. Few waves feel their one load in flight (FP16, 128 KiB segments of
// 1 GiB 195 and 169).
template <typename T>
__global__ void __launch_bounds__(1024) read_sum_kernel(const T* __restrict__ src, float* __restrict__ sink,
                                                         uint64_t elements, uint32_t block_elements,
                                                         uint64_t segments, bool serial) {
  constexpr int VEC = 16 / sizeof(T);
  const uint32_t lane = threadIdx.x & 63;
  const uint64_t waves_per_block = blockDim.x >> 6;
  const uint64_t wave = blockIdx.x * waves_per_block + (threadIdx.x >> 6);
  const uint64_t total_waves = static_cast<uint64_t>(gridDim.x) * waves_per_block;
  const uint32_t chunk = 64 * VEC;  // elements one wave covers per load
  for (uint64_t segment = wave; segment < segments; segment += total_waves) {
    const uint64_t first = segment * block_elements;
    const T* base = src + first;
    float total;
    if (elements - first >= block_elements) {
      // Load p feeds acc[p & 7]; block_elements is a multiple of eight loads.
      float acc[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
      const uint32_t loads = block_elements / chunk;
      for (uint32_t p = 0; p < loads; p += 8) {
        float value[8];
        load_and_sum(value, base + p * chunk + lane * VEC, serial);
#pragma unroll
        for (int j = 0; j < 8; ++j) acc[j] += value[j];
      }
      total = wave_sum(((acc[0] + acc[1]) + (acc[2] + acc[3])) + ((acc[4] + acc[5]) + (acc[6] + acc[7])));
    } else {
      total = clipped_sum(base, static_cast<uint32_t>(elements - first), lane);
    }
    if (lane == 0) sink[segment] = total;
  }
}

// Launches the aligned kernel (head = tail = 0 and src aligned) or the one with
// edges over `vectors` whole vectors.
template <int VPT, int POLICY>
void launch_copy_kernel(const char* src, char* dst, uint64_t vectors, uint32_t head, uint32_t tail, dim3 grid,
                        dim3 threads, hipStream_t stream) {
  if (head == 0 && tail == 0 && aligned(src, 16))
    copy_kernel<VPT, POLICY><<<grid, threads, 0, stream>>>(reinterpret_cast<const u32x4*>(src),
                                                           reinterpret_cast<u32x4*>(dst), vectors);
  else
    copy_edges_kernel<VPT, POLICY><<<grid, threads, 0, stream>>>(reinterpret_cast<const uint8_t*>(src),
                                                                 reinterpret_cast<uint8_t*>(dst), vectors, head, tail);
}

template <int POLICY>
int launch_copy(const char* src, char* dst, uint64_t vectors, uint32_t head, uint32_t tail, uint32_t threads,
                uint32_t vpt, uint32_t grid_blocks, hipStream_t stream) {
  const uint64_t step = static_cast<uint64_t>(threads) * vpt;
  const uint64_t steps = (vectors + step - 1) / step;
  const uint64_t grid = grid_blocks ? (grid_blocks < steps ? grid_blocks : steps) : steps;
  if (grid > 0x7fffffffull)
    return fail(MB_ERR_INVALID, "mb_copy: %llu workgroups exceed the grid limit; raise vectors_per_thread",
                static_cast<unsigned long long>(grid));
  dim3 g(static_cast<uint32_t>(grid)), b(threads);
  switch (vpt) {
    case 1: launch_copy_kernel<1, POLICY>(src, dst, vectors, head, tail, g, b, stream); break;
    case 2: launch_copy_kernel<2, POLICY>(src, dst, vectors, head, tail, g, b, stream); break;
    case 4: launch_copy_kernel<4, POLICY>(src, dst, vectors, head, tail, g, b, stream); break;
    case 8: launch_copy_kernel<8, POLICY>(src, dst, vectors, head, tail, g, b, stream); break;
    case 16: launch_copy_kernel<16, POLICY>(src, dst, vectors, head, tail, g, b, stream); break;
    default: return fail(MB_ERR_INVALID, "mb_copy: vectors_per_thread %u not in {1,2,4,8,16}", vpt);
  }
  return launch_status("copy_kernel");
}

#define MB_REGISTER_COPY(P, SUFFIX)                                                         \
  MB_REGISTER_KERNEL("copy_dwordx4_vpt1" SUFFIX, (copy_kernel<1, P>));               \
  MB_REGISTER_KERNEL("copy_dwordx4_vpt2" SUFFIX, (copy_kernel<2, P>));               \
  MB_REGISTER_KERNEL("copy_dwordx4_vpt4" SUFFIX, (copy_kernel<4, P>));               \
  MB_REGISTER_KERNEL("copy_dwordx4_vpt8" SUFFIX, (copy_kernel<8, P>));               \
  MB_REGISTER_KERNEL("copy_dwordx4_vpt16" SUFFIX, (copy_kernel<16, P>));             \
  MB_REGISTER_KERNEL("copy_edges_vpt1" SUFFIX, (copy_edges_kernel<1, P>));                  \
  MB_REGISTER_KERNEL("copy_edges_vpt2" SUFFIX, (copy_edges_kernel<2, P>));                  \
  MB_REGISTER_KERNEL("copy_edges_vpt4" SUFFIX, (copy_edges_kernel<4, P>));                  \
  MB_REGISTER_KERNEL("copy_edges_vpt8" SUFFIX, (copy_edges_kernel<8, P>));                  \
  MB_REGISTER_KERNEL("copy_edges_vpt16" SUFFIX, (copy_edges_kernel<16, P>))

MB_REGISTER_COPY(kPlain, "");
MB_REGISTER_COPY(kNontemporal, "_nt");
MB_REGISTER_COPY(kStream, "_stream");
MB_REGISTER_KERNEL("copy_tail", copy_tail_kernel);
MB_REGISTER_KERNEL("fill_dwordx4", (fill_kernel<kPlain>));
MB_REGISTER_KERNEL("fill_dwordx4_nt", (fill_kernel<kNontemporal>));
MB_REGISTER_KERNEL("fill_dwordx4_stream", (fill_kernel<kStream>));
MB_REGISTER_KERNEL("fill_tail", fill_tail_kernel);
MB_REGISTER_KERNEL("read_sum_f32_vec", (read_sum_kernel<float>));
MB_REGISTER_KERNEL("read_sum_f16_vec", (read_sum_kernel<_Float16>));
MB_REGISTER_KERNEL("read_sum_bf16_vec", (read_sum_kernel<uint16_t>));
#define MB_REGISTER_READ_PACKED(T, TNAME)                                            \
  MB_REGISTER_KERNEL("read_sum_" TNAME "_packed8", (read_sum_packed_kernel<T, 8>));     \
  MB_REGISTER_KERNEL("read_sum_" TNAME "_packed16", (read_sum_packed_kernel<T, 16>));   \
  MB_REGISTER_KERNEL("read_sum_" TNAME "_packed32", (read_sum_packed_kernel<T, 32>));   \
  MB_REGISTER_KERNEL("read_sum_" TNAME "_packed64", (read_sum_packed_kernel<T, 64>));   \
  MB_REGISTER_KERNEL("read_sum_" TNAME "_packed128", (read_sum_packed_kernel<T, 128>)); \
  MB_REGISTER_KERNEL("read_sum_" TNAME "_packed256", (read_sum_packed_kernel<T, 256>))
MB_REGISTER_READ_PACKED(float, "f32");
MB_REGISTER_READ_PACKED(_Float16, "f16");
MB_REGISTER_READ_PACKED(uint16_t, "bf16");

template <typename T>
int launch_read(const void* src, float* sink, uint64_t elements, uint32_t block_elements, uint32_t threads,
                hipStream_t stream) {
  constexpr uint32_t kVec = 16 / sizeof(T);
  const uint64_t segments = elements / block_elements + (elements % block_elements != 0);
  const uint64_t whole = elements / block_elements;
  const uint64_t waves_per_block = threads / 64;
  const uint32_t vectors = block_elements / kVec;
  // Waves: one per 4 KiB of whole segments and one for a clipped segment, or
  // one per segment. They stride, so a bounded grid still covers everything.
  const bool packed = vectors <= kPackedVectors;
  const uint64_t per_chunk = packed ? kPackedVectors / vectors : 1;
  const uint64_t chunks = (whole + per_chunk - 1) / per_chunk;
  const uint64_t waves = packed ? chunks + (segments != whole) : segments;
  uint64_t grid = (waves + waves_per_block - 1) / waves_per_block;
  const bool serial = waves > 131072 && aligned(src, 16);  // see read_sum_packed_kernel
  const uint64_t max_grid = 1ull << 20;
  if (grid > max_grid) grid = max_grid;
  const T* s = static_cast<const T*>(src);
  dim3 g(static_cast<uint32_t>(grid)), b(threads);
  switch (vectors) {
    case 8: read_sum_packed_kernel<T, 8><<<g, b, 0, stream>>>(s, sink, elements, chunks, serial); break;
    case 16: read_sum_packed_kernel<T, 16><<<g, b, 0, stream>>>(s, sink, elements, chunks, serial); break;
    case 32: read_sum_packed_kernel<T, 32><<<g, b, 0, stream>>>(s, sink, elements, chunks, serial); break;
    case 64: read_sum_packed_kernel<T, 64><<<g, b, 0, stream>>>(s, sink, elements, chunks, serial); break;
    case 128: read_sum_packed_kernel<T, 128><<<g, b, 0, stream>>>(s, sink, elements, chunks, serial); break;
    case 256: read_sum_packed_kernel<T, 256><<<g, b, 0, stream>>>(s, sink, elements, chunks, serial); break;
    default: read_sum_kernel<T><<<g, b, 0, stream>>>(s, sink, elements, block_elements, segments, serial);
  }
  return launch_status("read_sum_kernel");
}

}  // namespace
}  // namespace mb

extern "C" {

int mb_copy(const void* src, void* dst, uint64_t bytes, uint32_t block_threads, uint32_t vectors_per_thread,
            uint32_t grid_blocks, uint32_t flags, void* stream) {
  using namespace mb;
  if (bytes == 0) return MB_OK;
  if (src == nullptr || dst == nullptr) return fail(MB_ERR_INVALID, "mb_copy: NULL buffer");
  if (block_threads == 0 || block_threads % 64 || block_threads > 1024)
    return fail(MB_ERR_INVALID, "mb_copy: block_threads %u must be a multiple of 64 up to 1024", block_threads);
  if (!power_of_two(vectors_per_thread) || vectors_per_thread > 16)
    return fail(MB_ERR_INVALID, "mb_copy: vectors_per_thread %u not in {1,2,4,8,16}", vectors_per_thread);
  if (flags & ~(MB_COPY_NONTEMPORAL | MB_COPY_WRITE_THROUGH))
    return fail(MB_ERR_INVALID, "mb_copy: unknown flags 0x%x", flags);
  const char* s = static_cast<const char*>(src);
  char* d = static_cast<char*>(dst);
  if (s < d + bytes && d < s + bytes) return fail(MB_ERR_INVALID, "mb_copy: source and destination overlap");
  // Write-through stores pair with streaming loads; without it, the nt flag
  // makes both loads and stores non-temporal.
  const int policy = (flags & MB_COPY_WRITE_THROUGH) ? kStream : (flags & MB_COPY_NONTEMPORAL) ? kNontemporal : kPlain;
  hipStream_t st = static_cast<hipStream_t>(stream);
  // The head brings unaligned stores to whole 128-byte lines; an aligned dst
  // keeps its vectors where they are.
  const uint32_t head = aligned(dst, 16) ? 0 : static_cast<uint32_t>(-reinterpret_cast<uintptr_t>(dst) & 127);
  const uint64_t vectors = bytes > head ? (bytes - head) / 16 : 0;
  if (vectors == 0) {
    copy_tail_kernel<<<1, 64, 0, st>>>(reinterpret_cast<const uint8_t*>(s), reinterpret_cast<uint8_t*>(d),
                                       static_cast<uint32_t>(bytes));
    return launch_status("copy_tail_kernel");
  }
  const uint32_t tail = static_cast<uint32_t>((bytes - head) % 16);
  switch (policy) {
    case kStream: return launch_copy<kStream>(s, d, vectors, head, tail, block_threads, vectors_per_thread,
                                              grid_blocks, st);
    case kNontemporal: return launch_copy<kNontemporal>(s, d, vectors, head, tail, block_threads, vectors_per_thread,
                                                        grid_blocks, st);
    default: return launch_copy<kPlain>(s, d, vectors, head, tail, block_threads, vectors_per_thread, grid_blocks, st);
  }
}

int mb_fill(void* dst, uint64_t bytes, uint32_t pattern, uint32_t block_threads, uint32_t grid_blocks,
            uint32_t flags, void* stream) {
  using namespace mb;
  if (bytes == 0) return MB_OK;
  if (dst == nullptr) return fail(MB_ERR_INVALID, "mb_fill: NULL buffer");
  if (!aligned(dst, 16)) return fail(MB_ERR_ALIGNMENT, "mb_fill: dst must be 16-byte aligned");
  if (block_threads == 0 || block_threads % 64 || block_threads > 1024)
    return fail(MB_ERR_INVALID, "mb_fill: block_threads %u must be a multiple of 64 up to 1024", block_threads);
  if (flags & ~(MB_COPY_NONTEMPORAL | MB_COPY_WRITE_THROUGH))
    return fail(MB_ERR_INVALID, "mb_fill: unknown flags 0x%x", flags);
  hipStream_t st = static_cast<hipStream_t>(stream);
  const uint64_t vectors = bytes / 16;
  const uint64_t steps = (vectors + block_threads - 1) / block_threads;
  const uint64_t grid = grid_blocks ? (grid_blocks < steps ? grid_blocks : steps) : steps;
  if (grid > 0x7fffffffull)
    return fail(MB_ERR_INVALID, "mb_fill: %llu workgroups exceed the grid limit; pass grid_blocks",
                static_cast<unsigned long long>(grid));
  u32x4* d = static_cast<u32x4*>(dst);
  const uint32_t tail = static_cast<uint32_t>(bytes % 16);
  if (grid == 0) {
    fill_tail_kernel<<<1, 64, 0, st>>>(static_cast<uint8_t*>(dst), tail, pattern);
    return launch_status("fill_tail_kernel");
  }
  dim3 g(static_cast<uint32_t>(grid)), b(block_threads);
  if (flags & MB_COPY_WRITE_THROUGH) fill_kernel<kStream><<<g, b, 0, st>>>(d, vectors, pattern, tail);
  else if (flags & MB_COPY_NONTEMPORAL) fill_kernel<kNontemporal><<<g, b, 0, st>>>(d, vectors, pattern, tail);
  else fill_kernel<kPlain><<<g, b, 0, st>>>(d, vectors, pattern, tail);
  return launch_status("fill_kernel");
}

int mb_read_sum(int dtype, const void* src, float* sink, uint64_t elements, uint32_t block_elements,
                uint32_t block_threads, void* stream) {
  using namespace mb;
  if (elements == 0) return MB_OK;
  if (src == nullptr || sink == nullptr) return fail(MB_ERR_INVALID, "mb_read_sum: NULL buffer");
  if (!power_of_two(block_elements) || block_elements < 64 || block_elements > 65536)
    return fail(MB_ERR_INVALID, "mb_read_sum: block_elements %u must be a power of two in [64, 65536]",
                block_elements);
  if (block_threads == 0 || block_threads % 64 || block_threads > 1024)
    return fail(MB_ERR_INVALID, "mb_read_sum: block_threads %u must be a multiple of 64 up to 1024",
                block_threads);
  if (!aligned(sink, 4)) return fail(MB_ERR_ALIGNMENT, "mb_read_sum: sink must be 4-byte aligned");
  hipStream_t st = static_cast<hipStream_t>(stream);
  switch (dtype) {
    case MB_DTYPE_F32:
      if (!aligned(src, 4)) return fail(MB_ERR_ALIGNMENT, "mb_read_sum: f32 source must be 4-byte aligned");
      return launch_read<float>(src, sink, elements, block_elements, block_threads, st);
    case MB_DTYPE_F16:
      if (!aligned(src, 2)) return fail(MB_ERR_ALIGNMENT, "mb_read_sum: f16 source must be 2-byte aligned");
      return launch_read<_Float16>(src, sink, elements, block_elements, block_threads, st);
    case MB_DTYPE_BF16:
      if (!aligned(src, 2)) return fail(MB_ERR_ALIGNMENT, "mb_read_sum: bf16 source must be 2-byte aligned");
      return launch_read<uint16_t>(src, sink, elements, block_elements, block_threads, st);
    default:
      return fail(MB_ERR_INVALID, "mb_read_sum: unknown dtype %d", dtype);
  }
}

}  // extern "C"
