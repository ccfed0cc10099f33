// Stable sort of a species' particles by cell (no reference counterpart: it
// keeps gathers and deposits of neighbouring particles on the same cache
// lines).  Key = i * (nz-1) + k of the reference's cell index
// (include/geometry.h:44, clamped at 0); dead particles get the next key and
// end up behind the living ones, chunk padding slots after those.  The order
// among equal keys is the input order; the result is written back in the
// chunk-transposed layout.
//
// A sorted species stays nearly sorted between sorts, so the sort works on
// runs rather than particles:
//   runs:    each wavefront's 64 consecutive keys split into runs of equal
//            keys (a run never spans two wavefronts); one record (key,
//            length) per run, in logical order
//   records: stable LSD radix sort of the records by key, digits of up to 10
//            bits (the width that divides the key into the fewest equal parts):
//              hist:    per block of 4096 records, a digit histogram
//              scan:    exclusive scan of the bin-major histogram matrix
//              scatter: per block, stable ranks from wavefront ballots (lanes
//                       holding the same digit are matched with one ballot
//                       per bit), running per-wave digit counters in LDS
//   ranks:   exclusive scan of the run lengths in sorted order: each run's
//            first rank; a particle's rank = its run's + its place in the run
// The grids are sized for the record capacity (the number of records is known
// on the device only); what lies past the records' number returns at once.
// then every particle array is gathered through the resulting permutation in
// one pass (for a particle that stayed in place the gather reads its own
// slot, so a nearly sorted species is moved with coalesced reads).
#include "context.hpp"

namespace pdp3 {

namespace {

// A radix block: each lane holds 16 records of its wave in registers, their
// loads all in flight at once: a scatter launch takes 15 us where there are few
// (1e6 particles of 13 per cell) and 106 us for an ensemble of 1.3e8.  (4096
// per wave, read one at a time in two passes, took 64 us and 290 us: a chain
// of 128 loads.)
constexpr int kThreads = 256;
constexpr int kWaves = kThreads / 64;
constexpr int kPer = 16;  // records per lane
constexpr int kPerBlock = kThreads * kPer;
constexpr int kMaxDigit = 10;
constexpr int kMaxBins = 1 << kMaxDigit;

// the number of records present: the count on the device, or none when it
// exceeds the capacity (that sort is then skipped)
__device__ __forceinline__ long long present(const uint32_t *count, long long cap) {
  const long long m = *count;
  return m <= cap ? m : 0;
}

__host__ __device__ __forceinline__ uint32_t radix_blocks(long long n) {
  return (uint32_t)((n + kPerBlock - 1) / kPerBlock);
}

__device__ __forceinline__ uint64_t lanemask_lt() {
  unsigned lane = __lane_id();
  return lane == 0 ? 0ull : (~0ull >> (64 - lane));
}

// lanes (among `active`) whose digit of `width` bits equals this lane's
__device__ __forceinline__ uint64_t match_digit(uint32_t d, uint64_t active, int width) {
  uint64_t m = active;
  for (int b = 0; b < width; b++) {
    uint64_t bal = __ballot((d >> b) & 1u);
    m &= ((d >> b) & 1u) ? bal : ~bal;
  }
  return m;
}

// hist[digit * blocks + block], blocks = those that hold records
__global__ void __launch_bounds__(kThreads) k_hist(const uint32_t *__restrict__ keys, const uint32_t *count,
                                                   long long cap, int shift, int width, uint32_t *__restrict__ hist) {
  __shared__ uint32_t cnt[kMaxBins];
  const long long n = present(count, cap);
  const uint32_t blocks = radix_blocks(n), bins = 1u << width;
  if (blockIdx.x >= blocks) return;
  const long long base = (long long)blockIdx.x * kPerBlock + threadIdx.x;
  uint32_t key[kPer];
#pragma unroll
  for (int u = 0; u < kPer; u++) key[u] = base + u * kThreads < n ? keys[base + u * kThreads] : 0u;
  for (uint32_t d = threadIdx.x; d < bins; d += kThreads) cnt[d] = 0;
  __syncthreads();
#pragma unroll
  for (int u = 0; u < kPer; u++) {
    const bool valid = base + u * kThreads < n;
    const uint32_t d = (key[u] >> shift) & (bins - 1);
    // records that are nearly in order mostly share their high digits
    const uint64_t active = __ballot(valid);
    if (active == 0) break;
    const uint32_t d0 = __builtin_amdgcn_readfirstlane(d);  // the valid lanes are a prefix
    if (__ballot(valid && d == d0) == active) {
      if (__lane_id() == 0) atomicAdd(&cnt[d0], (uint32_t)__popcll(active));
    } else if (valid) {
      atomicAdd(&cnt[d], 1u);
    }
  }
  __syncthreads();
  for (uint32_t d = threadIdx.x; d < bins; d += kThreads) hist[(size_t)d * blocks + blockIdx.x] = cnt[d];
}

__global__ void __launch_bounds__(kThreads) k_scatter(const uint32_t *__restrict__ kin, const uint32_t *__restrict__ vin,
                                                      uint32_t *__restrict__ kout, uint32_t *__restrict__ vout,
                                                      const uint32_t *count, long long cap, int shift, int width,
                                                      const uint32_t *__restrict__ offs) {
  __shared__ uint32_t run[kWaves][kMaxBins];
  const long long n = present(count, cap);
  const uint32_t blocks = radix_blocks(n), bins = 1u << width;
  if (blockIdx.x >= blocks) return;
  const int wave = threadIdx.x / 64;
  const unsigned lane = __lane_id();
  const long long base = (long long)blockIdx.x * kPerBlock + (long long)wave * (64 * kPer) + lane;
  uint32_t key[kPer], val[kPer], place[kPer], off[kMaxBins / kThreads];
#pragma unroll
  for (int u = 0; u < kPer; u++) {
    const bool valid = base + u * 64 < n;
    key[u] = valid ? kin[base + u * 64] : 0u;
    val[u] = valid ? vin[base + u * 64] : 0u;
  }
#pragma unroll
  for (int u = 0; u < kMaxBins / kThreads; u++) {
    const uint32_t d = u * kThreads + threadIdx.x;
    off[u] = d < bins ? offs[(size_t)d * blocks + blockIdx.x] : 0u;
    for (int w = 0; w < kWaves; w++) run[w][d] = 0;
  }
  __syncthreads();
  // each record's place among its wave's records of the same digit
#pragma unroll
  for (int u = 0; u < kPer; u++) {
    const bool valid = base + u * 64 < n;
    const uint64_t active = __ballot(valid);
    if (active == 0) break;
    const uint32_t d = (key[u] >> shift) & (bins - 1);
    const uint64_t m = match_digit(d, active, width);
    const uint32_t before = run[wave][d];
    place[u] = before + (uint32_t)__popcll(m & lanemask_lt());
    // every lane's read of run[] before the leaders' update
    __builtin_amdgcn_wave_barrier();
    if (valid && (m & lanemask_lt()) == 0) run[wave][d] = before + (uint32_t)__popcll(m);
    __builtin_amdgcn_wave_barrier();
  }
  __syncthreads();
  // the global offset of the block's records of each digit, then of each wave's
#pragma unroll
  for (int u = 0; u < kMaxBins / kThreads; u++) {
    const uint32_t d = u * kThreads + threadIdx.x;
    uint32_t acc = off[u];
    for (int w = 0; w < kWaves; w++) {
      const uint32_t c = run[w][d];
      run[w][d] = acc;
      acc += c;
    }
  }
  __syncthreads();
#pragma unroll
  for (int u = 0; u < kPer; u++)
    if (base + u * 64 < n) {
      const uint32_t pos = run[wave][(key[u] >> shift) & (bins - 1)] + place[u];
      kout[pos] = key[u];
      vout[pos] = val[u];
    }
}

// ---- exclusive scan: the blocks' sums, then each block's scan from the sum
// of those before it (the block adds them up itself).  S: size(), load(j),
// store(j, scanned); one thread loads and stores an element, so that both may
// be the same array. ----
constexpr int kScanThreads = 1024, kScanPer = 4, kScanBlock = kScanThreads * kScanPer;
// a block adding up more sums than this would cost more than scanning them first
constexpr long long kScanSums = 8192;

struct ScanArray {
  uint32_t *p;
  long long n;
  __device__ __forceinline__ long long size() const { return n; }
  __device__ __forceinline__ uint32_t load(long long j) const { return p[j]; }
  __device__ __forceinline__ void store(long long j, uint32_t v) const { p[j] = v; }
};
// the histogram matrix of the records present
struct ScanHist {
  uint32_t *p;
  const uint32_t *count;
  long long cap;
  int width;
  __device__ __forceinline__ long long size() const { return (long long)radix_blocks(present(count, cap)) << width; }
  __device__ __forceinline__ uint32_t load(long long j) const { return p[j]; }
  __device__ __forceinline__ void store(long long j, uint32_t v) const { p[j] = v; }
};
// the run lengths in sorted order; each is replaced by its run's first rank
struct ScanRuns {
  const uint32_t *order;
  uint32_t *len;
  const uint32_t *count;
  long long cap;
  __device__ __forceinline__ long long size() const { return present(count, cap); }
  __device__ __forceinline__ uint32_t load(long long j) const { return len[order[j]]; }
  __device__ __forceinline__ void store(long long j, uint32_t v) const { len[order[j]] = v; }
};

// the exclusive prefix of v over the block and, in total, its sum; w: kScanThreads / 64 words of LDS
__device__ __forceinline__ uint32_t block_prefix(uint32_t v, uint32_t *w, uint32_t &total) {
  const unsigned lane = __lane_id(), wave = threadIdx.x >> 6;
  uint32_t x = v;
#pragma unroll
  for (int o = 1; o < 64; o <<= 1) {
    const uint32_t y = __shfl_up(x, o);
    if (lane >= (unsigned)o) x += y;
  }
  __syncthreads();  // the last use of w
  if (lane == 63) w[wave] = x;
  __syncthreads();
  uint32_t before = 0;
  total = 0;
#pragma unroll
  for (unsigned k = 0; k < kScanThreads / 64; k++) {
    before += k < wave ? w[k] : 0u;
    total += w[k];
  }
  return before + x - v;
}

template <class S>
__global__ void __launch_bounds__(kScanThreads) k_scan_sums(S s, uint32_t *__restrict__ sums) {
  __shared__ uint32_t w[kScanThreads / 64];
  const long long n = s.size(), j0 = (long long)blockIdx.x * kScanBlock + threadIdx.x;
  uint32_t v = 0, total;
  if (j0 - threadIdx.x < n) {
#pragma unroll
    for (int u = 0; u < kScanPer; u++) v += j0 + u * kScanThreads < n ? s.load(j0 + u * kScanThreads) : 0u;
  }
  block_prefix(v, w, total);
  if (threadIdx.x == 0) sums[blockIdx.x] = total;
}
// scanned: sums holds the exclusive prefixes already
template <class S>
__global__ void __launch_bounds__(kScanThreads) k_scan_write(S s, const uint32_t *__restrict__ sums, int scanned) {
  __shared__ uint32_t w[kScanThreads / 64];
  const long long n = s.size(), j0 = (long long)blockIdx.x * kScanBlock + (long long)threadIdx.x * kScanPer;
  if ((long long)blockIdx.x * kScanBlock >= n) return;
  uint32_t v[kScanPer], base = 0, t = 0, total;
#pragma unroll
  for (int u = 0; u < kScanPer; u++) {
    v[u] = j0 + u < n ? s.load(j0 + u) : 0u;
    t += v[u];
  }
  if (scanned) {
    base = sums[blockIdx.x];
  } else if (blockIdx.x > 0) {
    uint32_t b = 0;
    for (unsigned k = threadIdx.x; k < blockIdx.x; k += kScanThreads) b += sums[k];
    block_prefix(b, w, base);
  }
  uint32_t acc = base + block_prefix(t, w, total);
#pragma unroll
  for (int u = 0; u < kScanPer; u++)
    if (j0 + u < n) {
      s.store(j0 + u, acc);
      acc += v[u];
    }
}

// ---- runs of equal keys ----

// the runs of this wavefront's keys (lanes >= the valid prefix are not
// keys): heads = mask of first lanes; head, len = this lane's run
__device__ __forceinline__ uint64_t wave_runs(uint32_t key, bool valid, int &head, int &len) {
  const unsigned lane = __lane_id();
  const uint32_t prev = __shfl_up(key, 1);
  const bool starts = valid && (lane == 0 || prev != key);
  const uint64_t heads = __ballot(starts);
  const uint64_t upto = lane == 63 ? ~0ull : ((2ull << lane) - 1);
  const uint64_t hm = heads & upto;  // heads at or below this lane
  head = hm ? 63 - __clzll(hm) : 0;
  const uint64_t after = heads & ~upto;
  const int nvalid = __popcll(__ballot(valid));  // the valid lanes are a prefix
  const int end = after ? __ffsll((long long)after) - 1 : nvalid;
  len = end - head;
  return heads;
}

// The run kernels take kCPB chunks per block (their loads all in flight
// before the block's one barrier).  A chunk's keys are evaluated in slot order
// (coalesced) and transposed to logical order in LDS (rows padded to 17
// words, so that neither direction has bank conflicts); the block then walks
// them in groups of 256 logical keys, one record count (block_runs /
// block_base entry) per group.  nch: the species' number of chunks.
constexpr int kCPB = 2;
constexpr int kGroups = kChunk / 256;         // groups per chunk
constexpr int kBlockGroups = kCPB * kGroups;  // groups per block
constexpr int kRow = kPPT + 1;
constexpr int kChunkLds = 64 * kRow;

// the number of this block's chunks (the last block may hold fewer)
__device__ __forceinline__ int block_chunks(long long nch) {
  return (int)min((long long)kCPB, nch - (long long)blockIdx.x * kCPB);
}
template <class K>
__device__ __forceinline__ void chunk_keys(const K &keys, int nc, uint32_t *t) {
  const long long c0 = (long long)blockIdx.x * kCPB * kChunk;
  uint32_t v[kCPB * kGroups];
#pragma unroll
  for (int c = 0; c < kCPB; c++) {
    // the key function of this chunk (uniform over the block; a chunk past
    // the species' last takes the block's first, whose keys are not used)
    const auto kc = keys.at_chunk(c < nc ? c0 + (long long)c * kChunk : c0);
#pragma unroll
    for (int m = 0; m < kGroups; m++)
      v[c * kGroups + m] = c < nc ? kc(c0 + (long long)c * kChunk + m * 256 + (int)threadIdx.x) : 0u;
  }
#pragma unroll
  for (int c = 0; c < kCPB; c++)
#pragma unroll
    for (int m = 0; m < kGroups; m++) {
      const int w = m * 256 + (int)threadIdx.x;  // slot offset: iteration w / 64 of lane w % 64
      t[c * kChunkLds + (w % 64) * kRow + w / 64] = v[c * kGroups + m];
    }
  __syncthreads();
}
// logical offset s in the block's chunks: chunk s / kChunk, and in it lane
// (s % kChunk) / kPPT, iteration s % kPPT
__device__ __forceinline__ uint32_t chunk_key(const uint32_t *t, int s) {
  const int c = s / kChunk, l = s % kChunk;
  return t[c * kChunkLds + (l / kPPT) * kRow + l % kPPT];
}

// the runs of the block's groups of 256 logical keys: per lane the key and
// its run (head lane, length) in each group, and per group and wave the
// number of runs in wc[group * 4 + wave] (LDS, read after a barrier)
struct ChunkRuns {
  uint32_t key[kBlockGroups];
  uint64_t heads[kBlockGroups];
  int head[kBlockGroups], len[kBlockGroups];
};
__device__ __forceinline__ void chunk_runs(const uint32_t *t, ChunkRuns &cr, uint32_t *wc) {
#pragma unroll
  for (int m = 0; m < kBlockGroups; m++) {
    cr.key[m] = chunk_key(t, m * 256 + (int)threadIdx.x);
    cr.heads[m] = wave_runs(cr.key[m], true, cr.head[m], cr.len[m]);
    if (__lane_id() == 0) wc[m * 4 + (threadIdx.x >> 6)] = (uint32_t)__popcll(cr.heads[m]);
  }
  __syncthreads();
}
// the record index of this lane's run in group m (base: exclusive scan of the
// group counts at this group)
__device__ __forceinline__ uint32_t run_index(const ChunkRuns &cr, int m, uint32_t base, const uint32_t *wc) {
  const int wave = threadIdx.x >> 6;
  uint32_t r = base;
  for (int w = 0; w < wave; w++) r += wc[m * 4 + w];
  const int head = cr.head[m];
  const uint64_t below = head == 0 ? 0ull : (cr.heads[m] & (~0ull >> (64 - head)));
  return r + (uint32_t)__popcll(below);
}

// runs per group of 256 logical keys, and a zero behind the last group's (where
// the scan leaves the number of runs)
template <class K>
__global__ void __launch_bounds__(256) k_run_count(K keys, long long nch, uint32_t *__restrict__ block_runs) {
  __shared__ uint32_t t[kCPB * kChunkLds];
  __shared__ uint32_t wc[kBlockGroups * 4];
  const int nc = block_chunks(nch);
  chunk_keys(keys, nc, t);
  ChunkRuns cr;
  chunk_runs(t, cr, wc);
  if (threadIdx.x < nc * kGroups) {
    const uint32_t *g = wc + threadIdx.x * 4;
    block_runs[(long long)blockIdx.x * kBlockGroups + threadIdx.x] = g[0] + g[1] + g[2] + g[3];
  }
  if (blockIdx.x == 0 && threadIdx.x == 0) block_runs[nch * kGroups] = 0;
}

// one record (key, index, length) per run
template <class K>
__global__ void __launch_bounds__(256) k_run_emit(K keys, long long nch, const uint32_t *__restrict__ block_base,
                                                  const uint32_t *count, long long cap, uint32_t *__restrict__ rkey,
                                                  uint32_t *__restrict__ ridx, uint32_t *__restrict__ rlen) {
  if (*count > cap) return;  // more runs than record slots: this sort is skipped
  __shared__ uint32_t t[kCPB * kChunkLds];
  __shared__ uint32_t wc[kBlockGroups * 4];
  const int nc = block_chunks(nch);
  chunk_keys(keys, nc, t);
  ChunkRuns cr;
  chunk_runs(t, cr, wc);
#pragma unroll
  for (int m = 0; m < kBlockGroups; m++) {
    if (m >= nc * kGroups) break;
    const uint32_t r = run_index(cr, m, block_base[(long long)blockIdx.x * kBlockGroups + m], wc);
    if (cr.head[m] == (int)__lane_id()) {
      rkey[r] = cr.key[m];
      ridx[r] = r;
      rlen[r] = (uint32_t)cr.len[m];
    }
  }
}

// src[rank] = the slot of the particle of that rank, indexed by logical
// position (consecutive ranks are written by consecutive lanes); a skipped
// sort leaves every particle in its own slot
template <class K>
__global__ void __launch_bounds__(256) k_run_place(K keys, long long nch, const uint32_t *__restrict__ block_base,
                                                   const uint32_t *count, long long cap,
                                                   const uint32_t *__restrict__ rfirst, uint32_t *__restrict__ src) {
  const long long c0 = (long long)blockIdx.x * kCPB * kChunk;
  const int nc = block_chunks(nch);
  if (*count > cap) {
    for (int s = threadIdx.x; s < nc * kChunk; s += 256) src[c0 + s] = (uint32_t)phys_of(c0 + s);
    return;
  }
  __shared__ uint32_t t[kCPB * kChunkLds];
  __shared__ uint32_t wc[kBlockGroups * 4];
  chunk_keys(keys, nc, t);
  ChunkRuns cr;
  chunk_runs(t, cr, wc);
  const unsigned lane = __lane_id();
#pragma unroll
  for (int m = 0; m < kBlockGroups; m++) {
    if (m >= nc * kGroups) break;
    const uint32_t r = run_index(cr, m, block_base[(long long)blockIdx.x * kBlockGroups + m], wc);
    const int head = cr.head[m];
    const uint32_t first = head == (int)lane ? rfirst[r] : 0u;
    const uint32_t rank = __shfl(first, head) + (lane - (unsigned)head);
    src[rank] = (uint32_t)phys_of(c0 + m * 256 + (int)threadIdx.x);
  }
}

// every particle array in one pass, one chunk per block: slot p of the
// output takes the input slot src[logical position of p].  The block reads
// its chunk of src coalesced and transposes it to slot order in LDS (rows
// padded to 17 words); each thread then moves kGatherPer particles (256
// slots apart) so that all their loads are in flight together (non-temporal
// loads were slower: the slots of neighbouring particles share cache lines;
// the stores, each written once, are non-temporal: 5% off the sort).
struct Arrays7 {
  void *a[7];
};
constexpr int kGatherPer = kChunk / 256;
template <class T>
__device__ __forceinline__ void gather_array(const void *in, void *out, const uint32_t (&q)[kGatherPer],
                                             long long p0) {
  T x[kGatherPer];
#pragma unroll
  for (int u = 0; u < kGatherPer; u++) x[u] = static_cast<const T *>(in)[q[u]];
#pragma unroll
  for (int u = 0; u < kGatherPer; u++) __builtin_nontemporal_store(x[u], static_cast<T *>(out) + p0 + u * 256);
}
// the source slots of this thread's kGatherPer output slots c0 + u*256 + tid
__device__ __forceinline__ void gather_sources(const uint32_t *__restrict__ src, long long c0,
                                               uint32_t (&q)[kGatherPer]) {
  __shared__ uint32_t t[kChunkLds];
#pragma unroll
  for (int u = 0; u < kGatherPer; u++) {
    const int s = u * 256 + (int)threadIdx.x;  // logical offset
    t[(s / kPPT) * kRow + s % kPPT] = src[c0 + s];
  }
  __syncthreads();
#pragma unroll
  for (int u = 0; u < kGatherPer; u++) {
    const int w = u * 256 + (int)threadIdx.x;  // slot offset: lane w % 64, iteration w / 64
    q[u] = t[(w % 64) * kRow + w / 64];
  }
}
__global__ void __launch_bounds__(256) k_gather_f32(Arrays7 in, Arrays7 out, const uint32_t *__restrict__ src) {
  const long long c0 = (long long)blockIdx.x * kChunk;
  uint32_t q[kGatherPer];
  gather_sources(src, c0, q);
#pragma unroll
  for (int k = 0; k < 7; k++) gather_array<uint32_t>(in.a[k], out.a[k], q, c0 + threadIdx.x);
}
__global__ void __launch_bounds__(256) k_gather_f64(Arrays7 in, Arrays7 out, const uint32_t *__restrict__ src) {
  const long long c0 = (long long)blockIdx.x * kChunk;
  uint32_t q[kGatherPer];
  gather_sources(src, c0, q);
#pragma unroll
  for (int k = 0; k < 6; k++) gather_array<double>(in.a[k], out.a[k], q, c0 + threadIdx.x);
  gather_array<uint8_t>(in.a[6], out.a[6], q, c0 + threadIdx.x);
}

// the multi-segment gather: one chunk per block, the chunk's segment gives
// the arrays, the permutation holds global slots of the same segment
__global__ void __launch_bounds__(256) k_gather_f32_multi(const MultiSeg *__restrict__ seg,
                                                          const uint32_t *__restrict__ seg_of_chunk,
                                                          const uint32_t *__restrict__ src) {
  const long long c0 = (long long)blockIdx.x * kChunk;
  const MultiSeg &d = seg[seg_of_chunk[blockIdx.x]];
  uint32_t q[kGatherPer];
  gather_sources(src, c0, q);
#pragma unroll
  for (int u = 0; u < kGatherPer; u++) q[u] -= (uint32_t)d.slot_base;
  const long long p0 = c0 - d.slot_base + threadIdx.x;
#pragma unroll
  for (int k = 0; k < 7; k++) gather_array<uint32_t>(d.in[k], d.out[k], q, p0);
}

// the sort key of the particle in slot j, from its state
struct KeysF32 {
  GridDesc g;
  const uint32_t *cell;
  uint32_t dead_key;
  __device__ __forceinline__ uint32_t operator()(long long j) const {
    const uint32_t c = cell[j];
    if (c == kPadCell) return dead_key + 1;
    if (c & 0x80000000u) return dead_key;
    return ((c >> 16) & 0x7FFF) * (uint32_t)(g.nz - 1) + (c & 0xFFFF);
  }
  __device__ __forceinline__ const KeysF32 &at_chunk(long long) const { return *this; }
};
struct KeysF64 {
  GridDesc g;
  const double *r, *z;
  const uint8_t *alive;
  uint32_t dead_key;
  __device__ __forceinline__ uint32_t operator()(long long j) const {
    if (alive[j] == kPadSlot) return dead_key + 1;
    if (alive[j] != 1) return dead_key;
    int i = (int)ceil(r[j] / g.dr) - 1, k = (int)ceil(z[j] / g.dz) - 1;
    i = max(0, min(i, g.nr - 2));
    k = max(0, min(k, g.nz - 2));
    return (uint32_t)i * (uint32_t)(g.nz - 1) + (uint32_t)k;
  }
  __device__ __forceinline__ const KeysF64 &at_chunk(long long) const { return *this; }
};

// several species sorted as one: segment s holds global slots
// [slot_base, slot_base + n_cap) (whole chunks) and keys
// [key_base, key_base + ncell + 2), so the sorted order keeps every
// particle inside its own segment
__device__ __forceinline__ int seg_of(const MultiSeg *seg, const uint32_t *seg_of_chunk, long long j) {
  return (int)seg_of_chunk[j / kChunk];
}
// the keys of one segment (global slot j): row-major cells, or bands of two
// rows ordered column by column (cell (i, k) -> (i / 2) 2 (nz-1) + 2 k + i % 2)
struct KeysSeg {
  const uint32_t *cell;  // shifted so that cell[j] is global slot j
  uint32_t key_base, ncell, nzm1, band;
  __device__ __forceinline__ uint32_t operator()(long long j) const {
    const uint32_t c = cell[j];
    if (c == kPadCell) return key_base + ncell + 1;
    if (c & 0x80000000u) return key_base + ncell;
    const uint32_t i = (c >> 16) & 0x7FFF, k = c & 0xFFFF;
    return key_base + (band ? (i >> 1) * (2 * nzm1) + 2 * k + (i & 1) : i * nzm1 + k);
  }
};
struct KeysMulti {
  const MultiSeg *seg;
  const uint32_t *seg_of_chunk;
  // the segment of the chunk starting at global slot j0
  __device__ __forceinline__ KeysSeg at_chunk(long long j0) const {
    const int s = __builtin_amdgcn_readfirstlane(seg_of(seg, seg_of_chunk, j0));
    const MultiSeg &d = seg[s];
    return KeysSeg{d.cell - d.slot_base, d.key_base, d.ncell, d.nzm1, d.band};
  }
  __device__ __forceinline__ uint32_t operator()(long long j) const { return at_chunk(j - j % kChunk)(j); }
};

// scans at most n elements (S::size() on the device may be fewer); sums:
// scan_scratch(n) words
template <class S>
void exclusive_scan(const S &s, long long n, uint32_t *sums, hipStream_t st) {
  const long long nb = (n + kScanBlock - 1) / kScanBlock;
  const bool two = nb > kScanSums;
  if (nb > 1) hipLaunchKernelGGL(k_scan_sums<S>, dim3((unsigned)nb), dim3(kScanThreads), 0, st, s, sums);
  if (two) exclusive_scan(ScanArray{sums, nb}, nb, sums + nb, st);
  hipLaunchKernelGGL(k_scan_write<S>, dim3((unsigned)nb), dim3(kScanThreads), 0, st, s, sums, two ? 1 : 0);
}
// scratch words exclusive_scan needs for n elements
long long scan_scratch(long long n) {
  long long t = 0;
  while (n > 1) {
    n = (n + kScanBlock - 1) / kScanBlock;
    t += n;
  }
  return t + 1;
}

int digit_width(int bits) {
  const int passes = (bits + kMaxDigit - 1) / kMaxDigit;
  return (bits + passes - 1) / passes;
}
// words of the histogram matrix and its scan
long long hist_words(long long cap, int bits) { return (long long)radix_blocks(cap) << digit_width(bits); }

// stable LSD radix sort of the (key, val) pairs by the low `bits` bits of the
// key; returns the buffers holding the result (a or b).  hist: hist_words and
// their scan's scratch
void radix_pairs(uint32_t *&ka, uint32_t *&va, uint32_t *&kb, uint32_t *&vb, const uint32_t *count, long long cap,
                 int bits, uint32_t *hist, hipStream_t st) {
  const int width = digit_width(bits);
  const uint32_t blocks = radix_blocks(cap);
  const long long words = hist_words(cap, bits);
  for (int shift = 0; shift < bits; shift += width) {
    hipLaunchKernelGGL(k_hist, dim3(blocks), dim3(kThreads), 0, st, ka, count, cap, shift, width, hist);
    exclusive_scan(ScanHist{hist, count, cap, width}, words, hist + words, st);
    hipLaunchKernelGGL(k_scatter, dim3(blocks), dim3(kThreads), 0, st, ka, va, kb, vb, count, cap, shift, width,
                       hist);
    std::swap(ka, kb);
    std::swap(va, vb);
  }
}

bool ensure_alt(void *&alt, size_t bytes) {
  if (alt) return true;
  if (hipMalloc(&alt, bytes) != hipSuccess) {
    alt = nullptr;
    return false;
  }
  return true;
}

// workspace bytes for n slots and cap run records of `bits` bits (u32 words):
// src (n), before it is written the digit histograms with their scan, where
// they fit; group counts (nb + 1); scratch for the scans of the group counts
// and run lengths, and for the histograms that do not fit; the records (5 per
// slot)
struct SortWs {
  long long nb, scratch;
  bool hist_in_src;
  size_t bytes;
};
SortWs sort_ws(long long n, long long cap, int bits) {
  SortWs w;
  w.nb = (n + 255) / 256;
  const long long words = hist_words(cap, bits), hist = words + scan_scratch(words);
  w.hist_in_src = hist <= n;
  w.scratch = std::max(std::max(scan_scratch(w.nb + 1), scan_scratch(cap)), w.hist_in_src ? 0 : hist);
  w.bytes = (size_t)(n + (w.nb + 1) + w.scratch + 5 * cap) * sizeof(uint32_t);
  return w;
}
// bits of the keys 0 .. nkeys - 1 (at least one)
int key_bits(unsigned long long nkeys) {
  int bits = 1;
  while ((1ull << bits) < nkeys) bits++;
  return bits;
}
// the keys of a species: cells, the dead particles' and the padding's
unsigned long long cell_keys(const Ctx &c) {
  return (unsigned long long)(c.g.nr - 1) * (unsigned long long)(c.g.nz - 1) + 2;
}
bool ensure_ws(Ctx &c, size_t need) {
  if (c.sort_ws_bytes >= need) return true;
  if (c.sort_ws) (void)hipFree(c.sort_ws);
  c.sort_ws = nullptr;
  c.sort_ws_bytes = 0;
  if (hipMalloc(&c.sort_ws, need) != hipSuccess) return false;
  c.sort_ws_bytes = need;
  return true;
}
// the pinned run count and its event
bool ensure_runs(Species &sp) {
  if (sp.runs_host) return true;
  if (hipHostMalloc((void **)&sp.runs_host, sizeof(uint32_t), hipHostMallocDefault) != hipSuccess) {
    sp.runs_host = nullptr;
    return false;
  }
  *sp.runs_host = 0;
  if (hipEventCreateWithFlags(&sp.runs_ev, hipEventDisableTiming) != hipSuccess) {
    sp.runs_ev = nullptr;
    return false;
  }
  return true;
}
// the second buffer of every particle array
bool ensure_alts(Ctx &c, Species &sp) {
  const long long n = sp.n_cap;
  if (c.precision == 1) {
    SpeciesF32 &b = sp.f32_alt;
    void **bp[7] = {(void **)&b.cell, (void **)&b.fr, (void **)&b.fz, (void **)&b.vr, (void **)&b.vphi,
                    (void **)&b.vz, (void **)&b.w};
    for (int k = 0; k < 7; k++)
      if (!ensure_alt(*bp[k], (size_t)n * 4)) return false;
  } else {
    SpeciesF64 &b = sp.f64_alt;
    void **bp[7] = {(void **)&b.r, (void **)&b.z, (void **)&b.vr, (void **)&b.vphi, (void **)&b.vz, (void **)&b.w,
                    (void **)&b.alive};
    for (int k = 0; k < 7; k++)
      if (!ensure_alt(*bp[k], (size_t)n * (k < 6 ? 8 : 1))) return false;
  }
  return true;
}
bool sortable(const Ctx &c, const Species &sp) {
  return sp.n_cap > 1 && sp.chunked && !(c.precision == 1 && !sp.f32.cell);
}

}  // namespace

size_t sort_periodic_bytes(const Ctx &c) {
  size_t need = 0;
  for (const Species &sp : c.species) {
    if (sp.kind != 0 || !sortable(c, sp)) continue;
    const long long cap = sp.rec_cap > 0 ? sp.rec_cap : std::min(sp.n_cap, sp.n_cap / 4 + 65536);
    need = std::max(need, sort_ws(sp.n_cap, cap, key_bits(cell_keys(c))).bytes);
  }
  return need;
}

int sort_shrink_ws(Ctx &c, size_t need) {
  if (c.sort_ws_bytes <= need + need / 2) return 0;
  if (hipStreamSynchronize(c.stream) != hipSuccess) return -3;
  (void)hipFree(c.sort_ws);
  c.sort_ws = nullptr;
  c.sort_ws_bytes = 0;
  return need == 0 || ensure_ws(c, need) ? 0 : -3;
}

int sort_prepare(Ctx &c, Species &sp) {
  if (sp.sort_prepared || !sortable(c, sp)) return 0;
  const long long n = sp.n_cap;
  if (sp.rec_cap <= 0) sp.rec_cap = std::min(n, n / 4 + 65536);
  if (!ensure_runs(sp) || !ensure_ws(c, sort_ws(n, sp.rec_cap, key_bits(cell_keys(c))).bytes) || !ensure_alts(c, sp)) return -3;
  sp.sort_prepared = true;
  return 0;
}

void settle_sort(Species &sp) {
  if (sp.unsorted_before >= 0 && sp.runs_host && (long long)*sp.runs_host > sp.sort_cap) sp.steps_unsorted += sp.unsorted_before;
  sp.unsorted_before = -1;
}

void settle_sort_multi(MultiSort &ms, const std::vector<Ctx *> &cs) {
  for (Ctx *c : cs)
    for (Species &sp : c->species) {
      if (sp.unsorted_before >= 0 && (long long)*ms.runs_host > ms.sort_cap) sp.steps_unsorted += sp.unsorted_before;
      sp.unsorted_before = -1;
    }
}

int sort_species(Ctx &c, Species &sp, bool exact) {
  const long long n = sp.n_cap;
  if (!sortable(c, sp)) return 0;
  if (n % kChunk != 0) return -1;  // a chunked species fills whole chunks
  const uint32_t ncell = (uint32_t)(c.g.nr - 1) * (uint32_t)(c.g.nz - 1);
  const uint32_t dead_key = ncell;
  const int bits = key_bits(cell_keys(c));
  // record capacity: grown from the previous sort's run count (read back
  // asynchronously), so that no sort waits for the device
  const bool first = !sp.runs_host;
  if (!ensure_runs(sp)) return -3;
  if (!first && hipEventSynchronize(sp.runs_ev) != hipSuccess) return -3;
  settle_sort(sp);
  const long long last = *sp.runs_host;
  long long cap = sp.rec_cap > 0 ? sp.rec_cap : std::min(n, n / 4 + 65536);
  if (4 * last > 3 * cap) cap = std::min(n, 2 * last + 65536);
  sp.rec_cap = cap;
  if (exact) cap = n;  // room for one run per particle: this sort cannot be skipped
  const SortWs ws = sort_ws(n, cap, bits);
  const long long nb = ws.nb, scratch = ws.scratch;
  if (!ensure_ws(c, ws.bytes) || !ensure_alts(c, sp)) return -3;
  sp.unsorted_before = exact ? -1 : sp.steps_unsorted;
  sp.sort_cap = cap;
  sp.steps_unsorted = 0;
  uint32_t *src = (uint32_t *)c.sort_ws, *block = src + n, *tmp = block + nb + 1;
  uint32_t *rk = tmp + scratch, *ri = rk + cap, *rk2 = ri + cap, *ri2 = rk2 + cap, *rlen = ri2 + cap;
  const uint32_t *count = block + nb;  // the number of runs, after the scan
  const KeysF32 k32{c.g, (const uint32_t *)sp.f32.cell, dead_key};
  const KeysF64 k64{c.g, sp.f64.r, sp.f64.z, sp.f64.alive, dead_key};
  const bool f32 = c.precision == 1;
  // runs per group of 256 logical keys and their scan (block[nb] = the
  // number of runs); n is a whole number of chunks, one per block
  const long long nch = n / kChunk;
  const unsigned chunks = (unsigned)nch, rblocks = (unsigned)((nch + kCPB - 1) / kCPB);
  if (f32)
    hipLaunchKernelGGL(k_run_count<KeysF32>, dim3(rblocks), dim3(256), 0, c.stream, k32, nch, block);
  else
    hipLaunchKernelGGL(k_run_count<KeysF64>, dim3(rblocks), dim3(256), 0, c.stream, k64, nch, block);
  exclusive_scan(ScanArray{block, nb + 1}, nb + 1, tmp, c.stream);
  if (f32)
    hipLaunchKernelGGL(k_run_emit<KeysF32>, dim3(rblocks), dim3(256), 0, c.stream, k32, nch, block, count, cap, rk,
                       ri, rlen);
  else
    hipLaunchKernelGGL(k_run_emit<KeysF64>, dim3(rblocks), dim3(256), 0, c.stream, k64, nch, block, count, cap, rk,
                       ri, rlen);
  // records by key (stable), then each run's first rank
  radix_pairs(rk, ri, rk2, ri2, count, cap, bits, ws.hist_in_src ? src : tmp, c.stream);
  exclusive_scan(ScanRuns{ri, rlen, count, cap}, cap, tmp, c.stream);
  if (f32)
    hipLaunchKernelGGL(k_run_place<KeysF32>, dim3(rblocks), dim3(256), 0, c.stream, k32, nch, block, count, cap, rlen,
                       src);
  else
    hipLaunchKernelGGL(k_run_place<KeysF64>, dim3(rblocks), dim3(256), 0, c.stream, k64, nch, block, count, cap, rlen,
                       src);
  // the run count for the next sort's capacity
  if (hipMemcpyAsync(sp.runs_host, count, sizeof(uint32_t), hipMemcpyDeviceToHost, c.stream) != hipSuccess ||
      hipEventRecord(sp.runs_ev, c.stream) != hipSuccess)
    return -3;
  // all arrays in one gather
  Arrays7 in{}, out{};
  if (c.precision == 1) {
    SpeciesF32 &a = sp.f32, &b = sp.f32_alt;
    void **ap[7] = {(void **)&a.cell, (void **)&a.fr, (void **)&a.fz, (void **)&a.vr, (void **)&a.vphi,
                    (void **)&a.vz, (void **)&a.w};
    void **bp[7] = {(void **)&b.cell, (void **)&b.fr, (void **)&b.fz, (void **)&b.vr, (void **)&b.vphi,
                    (void **)&b.vz, (void **)&b.w};
    for (int k = 0; k < 7; k++) {
      in.a[k] = *ap[k];
      out.a[k] = *bp[k];
    }
    hipLaunchKernelGGL(k_gather_f32, dim3(chunks), dim3(256), 0, c.stream, in, out, src);
    for (int k = 0; k < 7; k++) std::swap(*ap[k], *bp[k]);
  } else {
    SpeciesF64 &a = sp.f64, &b = sp.f64_alt;
    void **ap[7] = {(void **)&a.r, (void **)&a.z, (void **)&a.vr, (void **)&a.vphi, (void **)&a.vz, (void **)&a.w,
                    (void **)&a.alive};
    void **bp[7] = {(void **)&b.r, (void **)&b.z, (void **)&b.vr, (void **)&b.vphi, (void **)&b.vz, (void **)&b.w,
                    (void **)&b.alive};
    for (int k = 0; k < 7; k++) {
      in.a[k] = *ap[k];
      out.a[k] = *bp[k];
    }
    hipLaunchKernelGGL(k_gather_f64, dim3(chunks), dim3(256), 0, c.stream, in, out, src);
    for (int k = 0; k < 7; k++) std::swap(*ap[k], *bp[k]);
  }
  return 0;
}


void sort_multi_free(MultiSort &ms) {
  if (ms.seg) (void)hipFree(ms.seg);
  if (ms.seg_of_chunk) (void)hipFree(ms.seg_of_chunk);
  if (ms.ws) (void)hipFree(ms.ws);
  if (ms.runs_host) (void)hipHostFree(ms.runs_host);
  if (ms.runs_ev) (void)hipEventDestroy(ms.runs_ev);
  ms = MultiSort();
}

int sort_multi(MultiSort &ms, const std::vector<Ctx *> &cs, hipStream_t stream) {
  // the segments: every sortable plasma species of every context, in order
  std::vector<std::pair<Ctx *, Species *>> list;
  for (Ctx *c : cs)
    for (Species &sp : c->species)
      if (sp.kind == 0 && sortable(*c, sp) && c->precision == 1) list.emplace_back(c, &sp);
  if (list.empty()) return 0;
  std::vector<MultiSeg> segs(list.size());
  long long n = 0, keys = 0;
  for (size_t s = 0; s < list.size(); s++) {
    Ctx &c = *list[s].first;
    Species &sp = *list[s].second;
    if (sp.n_cap % kChunk != 0) return -1;
    if (!ensure_alts(c, sp)) return -3;
    MultiSeg &d = segs[s];
    d.cell = (const uint32_t *)sp.f32.cell;
    d.slot_base = n;
    d.key_base = (uint32_t)keys;
    d.nzm1 = (uint32_t)(c.g.nz - 1);
    // A particle tile of 4096 consecutive particles spans 4096 / ppc cells; in
    // row order that overruns the tile's 128-column field box below about 32
    // particles per cell, in bands of two rows only below about 16.  Instances
    // with fewer particles per cell sort in bands.
    const long long rows = c.g.nr - 1;
    d.band = sp.n < 32LL * rows * (long long)d.nzm1 ? 1u : 0u;
    d.ncell = d.band ? (uint32_t)(2 * ((rows + 1) / 2)) * d.nzm1 : (uint32_t)rows * d.nzm1;
    SpeciesF32 &a = sp.f32, &b = sp.f32_alt;
    void *ap[7] = {a.cell, a.fr, a.fz, a.vr, a.vphi, a.vz, a.w};
    void *bp[7] = {b.cell, b.fr, b.fz, b.vr, b.vphi, b.vz, b.w};
    for (int k = 0; k < 7; k++) {
      d.in[k] = ap[k];
      d.out[k] = bp[k];
    }
    n += sp.n_cap;
    keys += (long long)d.ncell + 2;
  }
  if (n >= (1ll << 32) || keys >= (1ll << 32)) return -1;  // slots and keys are 32-bit
  const long long nch = n / kChunk;
  // the tables (rebuilt only when the segments change size)
  if (ms.n != n || ms.nseg != (long long)list.size()) {
    if (ms.seg) (void)hipFree(ms.seg);
    if (ms.seg_of_chunk) (void)hipFree(ms.seg_of_chunk);
    ms.seg = nullptr;
    ms.seg_of_chunk = nullptr;
    if (hipMalloc((void **)&ms.seg, list.size() * sizeof(MultiSeg)) != hipSuccess ||
        hipMalloc((void **)&ms.seg_of_chunk, (size_t)nch * sizeof(uint32_t)) != hipSuccess)
      return -3;
    std::vector<uint32_t> soc((size_t)nch);
    for (size_t s = 0; s < list.size(); s++) {
      const long long c0 = segs[s].slot_base / kChunk, c1 = c0 + list[s].second->n_cap / kChunk;
      for (long long ch = c0; ch < c1; ch++) soc[(size_t)ch] = (uint32_t)s;
    }
    if (hipMemcpy(ms.seg_of_chunk, soc.data(), soc.size() * sizeof(uint32_t), hipMemcpyHostToDevice) != hipSuccess)
      return -3;
    ms.n = n;
    ms.nseg = (long long)list.size();
    ms.rec_cap = 0;
    ms.counted = false;
  }
  // the segment table changes with every sort (the arrays swap); the
  // previous copy from seg_host has completed (the last sort's run-count
  // event, waited for below or above, comes after it on the stream)
  if (ms.counted && hipEventSynchronize(ms.runs_ev) != hipSuccess) return -3;
  if (ms.counted) settle_sort_multi(ms, cs);
  ms.seg_host = segs;
  if (hipMemcpyAsync(ms.seg, ms.seg_host.data(), segs.size() * sizeof(MultiSeg), hipMemcpyHostToDevice, stream) !=
      hipSuccess)
    return -3;
  const int bits = key_bits((unsigned long long)keys);
  // record capacity from the previous sort's run count (read back
  // asynchronously), as sort_species does
  if (!ms.runs_host) {
    if (hipHostMalloc((void **)&ms.runs_host, sizeof(uint32_t), hipHostMallocDefault) != hipSuccess) return -3;
    *ms.runs_host = 0;
    if (hipEventCreateWithFlags(&ms.runs_ev, hipEventDisableTiming) != hipSuccess) return -3;
  }
  const long long last = ms.counted ? (long long)*ms.runs_host : 0;
  long long cap = ms.rec_cap > 0 ? ms.rec_cap : std::min(n, n / 4 + 65536);
  if (4 * last > 3 * cap) cap = std::min(n, 2 * last + 65536);
  ms.rec_cap = ms.sort_cap = cap;
  const SortWs ws = sort_ws(n, cap, bits);
  if (ms.ws_bytes < ws.bytes) {
    if (ms.ws) (void)hipFree(ms.ws);
    ms.ws = nullptr;
    ms.ws_bytes = 0;
    if (hipMalloc(&ms.ws, ws.bytes) != hipSuccess) return -3;
    ms.ws_bytes = ws.bytes;
  }
  const long long nb = ws.nb, scratch = ws.scratch;
  uint32_t *src = (uint32_t *)ms.ws, *block = src + n, *tmp = block + nb + 1;
  uint32_t *rk = tmp + scratch, *ri = rk + cap, *rk2 = ri + cap, *ri2 = rk2 + cap, *rlen = ri2 + cap;
  const uint32_t *count = block + nb;
  const KeysMulti km{ms.seg, ms.seg_of_chunk};
  const unsigned chunks = (unsigned)nch, rblocks = (unsigned)((nch + kCPB - 1) / kCPB);
  hipLaunchKernelGGL(k_run_count<KeysMulti>, dim3(rblocks), dim3(256), 0, stream, km, nch, block);
  exclusive_scan(ScanArray{block, nb + 1}, nb + 1, tmp, stream);
  hipLaunchKernelGGL(k_run_emit<KeysMulti>, dim3(rblocks), dim3(256), 0, stream, km, nch, block, count, cap, rk, ri,
                     rlen);
  radix_pairs(rk, ri, rk2, ri2, count, cap, bits, ws.hist_in_src ? src : tmp, stream);
  exclusive_scan(ScanRuns{ri, rlen, count, cap}, cap, tmp, stream);
  hipLaunchKernelGGL(k_run_place<KeysMulti>, dim3(rblocks), dim3(256), 0, stream, km, nch, block, count, cap, rlen,
                     src);
  if (hipMemcpyAsync(ms.runs_host, count, sizeof(uint32_t), hipMemcpyDeviceToHost, stream) != hipSuccess ||
      hipEventRecord(ms.runs_ev, stream) != hipSuccess)
    return -3;
  ms.counted = true;
  hipLaunchKernelGGL(k_gather_f32_multi, dim3(chunks), dim3(256), 0, stream, ms.seg, ms.seg_of_chunk, src);
  if (hipGetLastError() != hipSuccess) return -3;
  for (auto &e : list) {
    SpeciesF32 &a = e.second->f32, &b = e.second->f32_alt;
    void **ap[7] = {(void **)&a.cell, (void **)&a.fr, (void **)&a.fz, (void **)&a.vr, (void **)&a.vphi,
                    (void **)&a.vz, (void **)&a.w};
    void **bp[7] = {(void **)&b.cell, (void **)&b.fr, (void **)&b.fz, (void **)&b.vr, (void **)&b.vphi,
                    (void **)&b.vz, (void **)&b.w};
    for (int k = 0; k < 7; k++) std::swap(*ap[k], *bp[k]);
    e.second->unsorted_before = e.second->steps_unsorted;
    e.second->steps_unsorted = 0;
  }
  return 0;
}

}  // namespace pdp3
