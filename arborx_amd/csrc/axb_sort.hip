// axb_sort.hip -- stable LSD radix sort (onesweep) and device-wide scans.
//
// Replaces the reference's sortObjects -> sortByKey (misc/ArborX_SortUtils.hpp:
// 26-43, kokkos_ext/ArborX_KokkosExtSort.hpp:79-149: Kokkos BinSort on the
// CPU, rocThrust sort_by_key on HIP) and KokkosExt::exclusive_scan
// (kokkos_ext/ArborX_KokkosExtStdAlgorithms.hpp).
//
// Sort design for gfx950 (wave64):
//  * 8-bit digits; the bucket counts of every pass come from one histogram
//    computed by the key-generation kernel (no per-pass counting sweep);
//  * one kernel per pass: a block takes a 4096-key tile (tile id from an
//    atomic ticket so that every tile it waits on is already running), ranks
//    its keys per wavefront with 8 ballots per key (equal-digit lane masks),
//    publishes its per-digit counts, looks back over predecessor tiles for
//    the digit prefixes (decoupled look-back with bounded waits), stages the
//    tile in LDS in digit order and writes runs of equal digits contiguously;
//  * stability: a key's rank orders (wave, item, lane), which is its order in
//    the input, and tiles are prefixed in tile order.
#include "axb_internal.hpp"

namespace axb
{

namespace
{

constexpr uint32_t FLAG_AGG = 1u << 30;
constexpr uint32_t FLAG_PREFIX = 2u << 30;
constexpr uint32_t VALUE_MASK = (1u << 30) - 1u;

// (gate: given and zero, the kernel does nothing)
__global__ void k_fill_u32(uint32_t *p, uint32_t v, int64_t n,
                           const uint32_t *gate = nullptr)
{
  if (gate && *gate == 0u)
    return;
  int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  int64_t stride = (int64_t)gridDim.x * blockDim.x;
  for (; i < n; i += stride)
    p[i] = v;
}
__global__ void k_iota_u32(uint32_t *p, int64_t n)
{
  int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  int64_t stride = (int64_t)gridDim.x * blockDim.x;
  for (; i < n; i += stride)
    p[i] = (uint32_t)i;
}
__global__ void k_fill_u64(uint64_t *p, uint64_t v, int64_t n)
{
  int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  int64_t stride = (int64_t)gridDim.x * blockDim.x;
  for (; i < n; i += stride)
    p[i] = v;
}

template <class K>
__global__ __launch_bounds__(256) void k_key_hist(const K *__restrict__ keys,
                                                  int64_t n, int passes, int shift0,
                                                  uint32_t *__restrict__ hist,
                                                  const uint32_t *gate)
{
  if (gate && *gate == 0u)
    return;
  __shared__ uint32_t s_h[8 * 256];
  for (int j = threadIdx.x; j < passes * 256; j += blockDim.x)
    s_h[j] = 0;
  __syncthreads();
  int64_t stride = (int64_t)gridDim.x * blockDim.x;
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n;
       i += stride)
  {
    K k = keys[i];
    for (int p = 0; p < passes; ++p)
      atomicAdd(&s_h[p * 256 + (uint32_t)((k >> (shift0 + 8 * p)) & 255)], 1u);
  }
  __syncthreads();
  for (int j = threadIdx.x; j < passes * 256; j += blockDim.x)
    if (s_h[j])
      atomicAdd(&hist[j], s_h[j]);
}

// Wave64 inclusive sum scan.
template <class T>
AXB_D T wave_inclusive_sum(T v)
{
  const int lane = threadIdx.x & 63;
#pragma unroll
  for (int o = 1; o < 64; o <<= 1)
  {
    T u = __shfl_up(v, o, 64);
    if (lane >= o)
      v += u;
  }
  return v;
}

// hist (passes x 256 counts) -> exclusive digit offsets in place, plus a
// per-pass flag telling whether every key has the same digit in that pass.
__global__ __launch_bounds__(256) void k_hist_scan(uint32_t *hist,
                                                   uint32_t *trivial,
                                                   int passes, int64_t n,
                                                   const uint32_t *gate)
{
  if (gate && *gate == 0u)
    return;
  __shared__ uint32_t s_w[4];
  const int d = threadIdx.x, lane = d & 63, wave = d >> 6;
  for (int p = 0; p < passes; ++p)
  {
    uint32_t c = hist[p * 256 + d];
    uint32_t inc = wave_inclusive_sum(c);
    if (lane == 63)
      s_w[wave] = inc;
    __syncthreads();
    uint32_t add = 0;
    for (int w = 0; w < wave; ++w)
      add += s_w[w];
    hist[p * 256 + d] = inc - c + add;
    if ((int64_t)c == n)
      trivial[p] = 1u;
    __syncthreads();
  }
}

template <class K>
__global__ __launch_bounds__(SORT_BLOCK) void k_onesweep(
    const K *__restrict__ kin, const uint32_t *__restrict__ vin,
    K *__restrict__ kout, uint32_t *__restrict__ vout, int64_t n, int shift,
    const uint32_t *__restrict__ digit_offset,
    const uint32_t *__restrict__ trivial, uint32_t *__restrict__ status,
    uint32_t *__restrict__ tile_counter, uint32_t *__restrict__ err,
    const uint32_t *__restrict__ gate, const uint32_t *__restrict__ no_vals)
{
  if (gate && *gate == 0u)
    return;
  // (no_vals: given and not zero, the values are the positions)
  if (no_vals && *no_vals != 0u)
    vin = nullptr;
  constexpr int WAVES = SORT_BLOCK / 64;
  __shared__ uint32_t s_tile;
  __shared__ uint32_t s_whist[WAVES][256];
  __shared__ uint32_t s_bstart[256];
  __shared__ uint32_t s_gbase[256];
  __shared__ uint32_t s_wsum[WAVES];
  __shared__ K s_keys[SORT_TILE];
  __shared__ uint32_t s_vals[SORT_TILE];

  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;

  if (*trivial)
  {
    // Every key has the same digit in this pass: the stable pass is the
    // identity; copy through.
    int64_t base = (int64_t)blockIdx.x * SORT_TILE;
    for (int j = tid; j < SORT_TILE; j += SORT_BLOCK)
    {
      int64_t i = base + j;
      if (i < n)
      {
        kout[i] = kin[i];
        vout[i] = vin ? vin[i] : (uint32_t)i;
      }
    }
    return;
  }

  if (tid == 0)
    s_tile = atomicAdd(tile_counter, 1u);
  for (int j = tid; j < WAVES * 256; j += SORT_BLOCK)
    (&s_whist[0][0])[j] = 0;
  __syncthreads();
  const uint32_t tile = s_tile;
  const int64_t tile_base = (int64_t)tile * SORT_TILE;
  const int tile_count = (int)((n - tile_base) < SORT_TILE ? (n - tile_base)
                                                           : SORT_TILE);

  // ---- load (wave w owns items [w*64*ITEMS, (w+1)*64*ITEMS) of the tile)
  K key[SORT_ITEMS];
  uint32_t val[SORT_ITEMS];
  uint32_t rank[SORT_ITEMS];
  uint32_t dig[SORT_ITEMS];
#pragma unroll
  for (int i = 0; i < SORT_ITEMS; ++i)
  {
    int local = wave * 64 * SORT_ITEMS + i * 64 + lane;
    int64_t gi = tile_base + local;
    if (local < tile_count)
    {
      key[i] = kin[gi];
      val[i] = vin ? vin[gi] : (uint32_t)gi;
      dig[i] = (uint32_t)((key[i] >> shift) & 255);
    }
    else
    {
      key[i] = 0;
      val[i] = 0;
      dig[i] = 256u;
    }
  }

  // ---- per-wave ranking by equal-digit lane masks
  const uint64_t lt_mask = (lane == 0) ? 0ull : (~0ull >> (64 - lane));
#pragma unroll
  for (int i = 0; i < SORT_ITEMS; ++i)
  {
    const uint32_t d = dig[i];
    const bool valid = d < 256u;
    uint64_t m = __ballot(valid);
#pragma unroll
    for (int b = 0; b < 8; ++b)
    {
      const bool bit = (d >> b) & 1u;
      const uint64_t bb = __ballot(bit);
      m &= bit ? bb : ~bb;
    }
    const uint32_t before = (uint32_t)__popcll(m & lt_mask);
    uint32_t old = 0;
    if (valid)
      old = s_whist[wave][d];
    if (valid && before == 0)
      s_whist[wave][d] = old + (uint32_t)__popcll(m);
    rank[i] = old + before;
  }
  __syncthreads();

  // ---- per digit: wave prefixes and tile total; publish the aggregate
  const int d = tid;
  uint32_t total = 0;
#pragma unroll
  for (int w = 0; w < WAVES; ++w)
  {
    uint32_t c = s_whist[w][d];
    s_whist[w][d] = total;
    total += c;
  }
  uint32_t *my_status = status + (size_t)tile * 256 + d;
  if (tile == 0)
    st_agent(my_status, FLAG_PREFIX | total);
  else
    st_agent(my_status, FLAG_AGG | total);

  // ---- block-local digit starts (exclusive scan of totals over digits)
  uint32_t inc = wave_inclusive_sum(total);
  if (lane == 63)
    s_wsum[wave] = inc;
  __syncthreads();
  uint32_t add = 0;
  for (int w = 0; w < wave; ++w)
    add += s_wsum[w];
  const uint32_t bstart = inc - total + add;
  s_bstart[d] = bstart;
  __syncthreads();

  // ---- stage the tile in LDS in digit order
#pragma unroll
  for (int i = 0; i < SORT_ITEMS; ++i)
  {
    if (dig[i] < 256u)
    {
      uint32_t pos = s_bstart[dig[i]] + s_whist[wave][dig[i]] + rank[i];
      if (pos < (uint32_t)SORT_TILE)
      {
        s_keys[pos] = key[i];
        s_vals[pos] = val[i];
      }
    }
  }

  // ---- decoupled look-back for digit d
  uint32_t excl = 0;
  if (tile != 0)
  {
    int64_t j = (int64_t)tile - 1;
    uint32_t spins = 0;
    while (j >= 0)
    {
      uint32_t v = ld_agent(status + (size_t)j * 256 + d);
      uint32_t flag = v & ~VALUE_MASK;
      if (flag == 0u)
      {
        if (++spins >= SPIN_LIMIT)
        {
          raise_error(err, KERR_SPIN);
          break;
        }
        __builtin_amdgcn_s_sleep(1);
        continue;
      }
      excl += v & VALUE_MASK;
      if (flag == FLAG_PREFIX)
        break;
      --j;
    }
    st_agent(my_status, FLAG_PREFIX | (excl + total));
  }
  s_gbase[d] = digit_offset[d] + excl - bstart;
  __syncthreads();

  // ---- write out runs of equal digits
  for (int j = tid; j < tile_count; j += SORT_BLOCK)
  {
    K k = s_keys[j];
    uint32_t dd = (uint32_t)((k >> shift) & 255);
    uint32_t pos = s_gbase[dd] + (uint32_t)j;
    if ((int64_t)pos < n) // only a failed look-back could break this
    {
      kout[pos] = k;
      vout[pos] = s_vals[j];
    }
  }
}

// ------------------------------------------------------------ scans
// Reduce, then scan: (1) the sum of each tile of SCAN_TILE elements,
// (2) one block turns the tile sums into exclusive tile offsets, (3) each
// tile scans itself from its offset.  The input is read twice and no block
// waits on another.  A thread owns SCAN_ITEMS consecutive elements.

// Elements [base, base + SCAN_ITEMS) of a thread, 0 past n; running sums in
// v.  A whole, 16-byte aligned run is read with 16-byte loads.
template <class Tin>
AXB_D int64_t scan_load_items(const Tin *in, int64_t n, int64_t base, int64_t v[SCAN_ITEMS])
{
  static_assert(SCAN_ITEMS * sizeof(Tin) % 16 == 0, "runs of whole 16-byte words");
  Tin x[SCAN_ITEMS];
  if (base + SCAN_ITEMS <= n && ((uintptr_t)(in + base) & 15u) == 0)
  {
#pragma unroll
    for (int i = 0; i < SCAN_ITEMS; i += 16 / (int)sizeof(Tin))
      *(uint4 *)&x[i] = *(const uint4 *)(in + base + i);
  }
  else
  {
#pragma unroll
    for (int i = 0; i < SCAN_ITEMS; ++i)
      x[i] = (base + i < n) ? in[base + i] : Tin(0);
  }
  int64_t run = 0;
#pragma unroll
  for (int i = 0; i < SCAN_ITEMS; ++i)
  {
    run += (int64_t)x[i];
    v[i] = run;
  }
  return run;
}

// Exclusive prefix of x over the block's threads, and the block's total
// (s_wsum: one slot per wavefront).
template <int BLOCK>
AXB_D int64_t block_exclusive_sum(int64_t x, int64_t *s_wsum, int64_t &total)
{
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int64_t inc = wave_inclusive_sum(x);
  if (lane == 63)
    s_wsum[wave] = inc;
  __syncthreads();
  int64_t add = 0;
  total = 0;
#pragma unroll
  for (int w = 0; w < BLOCK / 64; ++w)
  {
    add += w < wave ? s_wsum[w] : 0;
    total += s_wsum[w];
  }
  return inc - x + add;
}

template <class Tin>
__global__ __launch_bounds__(SCAN_BLOCK) void k_scan_tile_sums(const Tin *in, int64_t n,
                                                               int64_t *__restrict__ sums)
{
  __shared__ int64_t s_wsum[SCAN_BLOCK / 64];
  const int64_t base = (int64_t)blockIdx.x * SCAN_TILE + (int64_t)threadIdx.x * SCAN_ITEMS;
  int64_t v[SCAN_ITEMS];
  const int64_t run = scan_load_items(in, n, base, v);
  int64_t total;
  block_exclusive_sum<SCAN_BLOCK>(run, s_wsum, total);
  if (threadIdx.x == 0)
    sums[blockIdx.x] = total;
}

// One block: sums[0, tiles) -> their exclusive prefix, in place.
constexpr int SCAN_OFFSETS_BLOCK = 1024;
__global__ __launch_bounds__(SCAN_OFFSETS_BLOCK) void k_scan_tile_offsets(int64_t *sums,
                                                                          int64_t tiles)
{
  __shared__ int64_t s_wsum[SCAN_OFFSETS_BLOCK / 64];
  int64_t carry = 0;
  for (int64_t c0 = 0; c0 < tiles; c0 += (int64_t)SCAN_OFFSETS_BLOCK * SCAN_ITEMS)
  {
    const int64_t base = c0 + (int64_t)threadIdx.x * SCAN_ITEMS;
    int64_t v[SCAN_ITEMS];
    const int64_t run = scan_load_items(sums, tiles, base, v);
    int64_t total;
    const int64_t pre = carry + block_exclusive_sum<SCAN_OFFSETS_BLOCK>(run, s_wsum, total);
#pragma unroll
    for (int i = 0; i < SCAN_ITEMS; ++i)
      if (base + i < tiles)
        sums[base + i] = pre + (i == 0 ? 0 : v[i - 1]);
    carry += total;
    __syncthreads(); // s_wsum is rewritten by the next chunk
  }
}

// flags (when given): bit i of byte e is set when input e * 8 + i exceeds
// limit (the CRS's rows that overflow their scratch row, read from the
// counts as they are scanned).
template <class Tin, class Tout, bool INCLUSIVE>
__global__ __launch_bounds__(SCAN_BLOCK) void k_scan_tiles(const Tin *in, Tout *out, int64_t n,
                                                           const int64_t *__restrict__ offs,
                                                           uint8_t *__restrict__ flags,
                                                           int64_t limit)
{
  static_assert(SCAN_ITEMS == 8, "one flag byte per thread");
  __shared__ int64_t s_wsum[SCAN_BLOCK / 64];
  const int64_t base = (int64_t)blockIdx.x * SCAN_TILE + (int64_t)threadIdx.x * SCAN_ITEMS;
  int64_t v[SCAN_ITEMS];
  const int64_t run = scan_load_items(in, n, base, v);
  if (flags && base < n)
  {
    uint32_t bits = 0;
#pragma unroll
    for (int i = 0; i < SCAN_ITEMS; ++i)
      bits |= (uint32_t)(base + i < n && v[i] - (i == 0 ? 0 : v[i - 1]) > limit) << i;
    flags[base >> 3] = (uint8_t)bits;
  }
  int64_t total;
  const int64_t pre = offs[blockIdx.x] + block_exclusive_sum<SCAN_BLOCK>(run, s_wsum, total);
  Tout y[SCAN_ITEMS];
#pragma unroll
  for (int i = 0; i < SCAN_ITEMS; ++i)
    y[i] = (Tout)(pre + (INCLUSIVE ? v[i] : (i == 0 ? 0 : v[i - 1])));
  if (base + SCAN_ITEMS <= n && ((uintptr_t)(out + base) & 15u) == 0)
  {
#pragma unroll
    for (int i = 0; i < SCAN_ITEMS; i += 16 / (int)sizeof(Tout))
      *(uint4 *)(out + base + i) = *(const uint4 *)&y[i];
  }
  else
  {
#pragma unroll
    for (int i = 0; i < SCAN_ITEMS; ++i)
      if (base + i < n)
        out[base + i] = y[i];
  }
}

inline int fill_grid(int64_t n)
{
  int64_t g = div_up(n, 256);
  return (int)(g < 4096 ? (g < 1 ? 1 : g) : 4096);
}

// Stable LSD sort by the digits of bits [shift0, shift0 + 8 passes).  vals0
// holds the values when have_vals (and not *no_vals), else they are the
// positions.  gate: as in the kernels.
template <class K>
hipError_t radix_sort_pairs(K *keys0, K *keys1, uint32_t *vals0,
                            uint32_t *vals1, int64_t n, int passes, int shift0, bool have_vals,
                            uint32_t *hist, void *workspace, uint32_t *err,
                            hipStream_t stream, const uint32_t *gate,
                            const uint32_t *no_vals = nullptr)
{
  const int64_t tiles = div_up(n, SORT_TILE);
  // workspace layout: [hist passes*256][trivial passes][counters passes]
  //                   [status passes*tiles*256]
  uint32_t *ws = (uint32_t *)workspace;
  uint32_t *own_hist = ws;
  uint32_t *trivial = ws + passes * 256;
  uint32_t *counters = trivial + passes;
  uint32_t *status = counters + passes;
  const int64_t zero_words =
      (hist ? 0 : passes * 256) + 2 * passes + (int64_t)passes * tiles * 256;
  uint32_t *zero_from = hist ? trivial : own_hist;
  AXB_LAUNCH(k_fill_u32, dim3(fill_grid(zero_words)), dim3(256), 0,
                     stream, zero_from, 0u, zero_words, gate);
  if (!hist)
  {
    hist = own_hist;
    int g = (int)(tiles < 2048 ? tiles : 2048);
    AXB_LAUNCH(k_key_hist<K>, dim3(g), dim3(256), 0, stream, keys0, n,
                       passes, shift0, hist, gate);
  }
  AXB_LAUNCH(k_hist_scan, dim3(1), dim3(256), 0, stream, hist,
                     trivial, passes, n, gate);
  K *kin = keys0, *kout = keys1;
  uint32_t *vin = have_vals ? vals0 : nullptr, *vout = vals1;
  for (int p = 0; p < passes; ++p)
  {
    AXB_LAUNCH(k_onesweep<K>, dim3((unsigned)tiles), dim3(SORT_BLOCK),
                       0, stream, kin, vin, kout, vout, n, shift0 + 8 * p,
                       hist + p * 256, trivial + p,
                       status + (size_t)p * tiles * 256, counters + p, err, gate,
                       p == 0 ? no_vals : (const uint32_t *)nullptr);
    K *kt = kin;
    kin = kout;
    kout = kt;
    vin = vout;
    vout = (vout == vals1) ? vals0 : vals1;
  }
  return hipGetLastError();
}

// ---------------------------------------------- 63-bit keys, top half first
// Keys sorted by their top 32 bits (shift HI_SHIFT) are sorted altogether
// but for runs of equal top halves whose low halves are out of order.  An
// inversion (a neighbour with the same top half and a smaller key) that is
// the first of its run lists the run: up to RUN_TINY keys for a thread, up to
// RUN_SHORT for a wavefront, up to RUN_LONG for a block.  A longer one, or one
// whose first inversion comes after RUN_SHORT keys in order, opens the gate of
// the full sort.  Runs of equal keys hold no inversions.  k_find_runs takes
// 0.031 ms for the keys of 10M uniform points, each of the four passes saved
// 0.12 to 0.15 ms.
constexpr int HI_SHIFT = 31;
constexpr int RUN_TINY = 8;
constexpr int RUN_SHORT = 64;
constexpr int RUN_LONG = 4096;
struct RunWords
{
  uint32_t tinies, shorts, longs; // runs on the lists
  uint32_t gate;                  // the full sort runs
  uint32_t top;                   // the sort by the top halves runs
  uint32_t crowded;               // it does not (no permutation yet)
};
static_assert(sizeof(RunWords) == SORT_RUN_WORDS * 4, "scratch words");

// A look at SAMPLE keys before the sort, for whether the full sort runs at
// once, without the four passes by the top halves.  A sampled key matches when
// an earlier one has its top half but not its low half; where keys crowd into
// cells there are about SAMPLE^2 / 2 times the sum of the squared parts of the
// keys in a cell of them.  From SAMPLE_MATCHES on, putting the runs right
// costs more than the passes saved (1000 clusters of sigma 0.001, 30 to 40
// matches: 10M points 2.35 ms with eight passes, 2.66 with four, 1M 0.58 /
// 0.59; of sigma 0.0001 1M 0.61 / 0.73; of sigma 0.01, no match, 2.23 / 1.80
// and 0.56 / 0.49), and `crowd` matches in one cell stand for a run of 1.5
// RUN_LONG (SAMPLE L / n of a run of L), too long for a block.  Also clears
// the words.
constexpr uint32_t SAMPLE_MATCHES = 24;
constexpr int SAMPLE = 4096, SAMPLE_SLOTS = 8192, SAMPLE_COUNTS = 2048;
inline uint32_t sample_crowd(int64_t n)
{
  const int64_t c = (int64_t)SAMPLE * (RUN_LONG + RUN_LONG / 2) / n;
  return (uint32_t)(c < 3 ? 3 : c);
}
__global__ __launch_bounds__(1024) void k_sample_runs(const uint64_t *__restrict__ keys,
                                                      int64_t n, uint32_t crowd, RunWords *w)
{
  constexpr uint32_t EMPTY = ~0u;
  constexpr int PER = SAMPLE / 1024;
  __shared__ __align__(16) uint32_t s_top[SAMPLE_SLOTS], s_count[SAMPLE_COUNTS];
  __shared__ uint32_t s_low[SAMPLE_SLOTS];
  __shared__ uint32_t s_crowded, s_matches;
  uint64_t k[PER];
#pragma unroll
  for (int j = 0; j < PER; ++j)
  {
    // one key of each part of the input, at a different place in each
    const uint32_t s = (uint32_t)j * 1024u + threadIdx.x;
    const uint64_t at = (uint64_t)s * 65536u + ((s * 40503u) & 65535u);
    k[j] = keys[at * (uint64_t)n / ((uint64_t)SAMPLE * 65536u)];
  }
  for (int j = threadIdx.x; j < SAMPLE_SLOTS / 4; j += 1024)
    ((uint4 *)s_top)[j] = make_uint4(EMPTY, EMPTY, EMPTY, EMPTY);
  for (int j = threadIdx.x; j < SAMPLE_COUNTS / 4; j += 1024)
    ((uint4 *)s_count)[j] = make_uint4(0u, 0u, 0u, 0u);
  if (threadIdx.x == 0)
    s_crowded = 0u, s_matches = 0u;
  __syncthreads();
  uint32_t slot[PER];
#pragma unroll
  for (int j = 0; j < PER; ++j)
  {
    uint32_t top = (uint32_t)(k[j] >> HI_SHIFT);
    top = top == EMPTY ? EMPTY - 1u : top;
    uint32_t h = (top * 2654435761u) >> 19; // half of the slots stay empty
    while (true)
    {
      const uint32_t was = atomicCAS(&s_top[h], EMPTY, top);
      if (was == EMPTY)
        s_low[h] = (uint32_t)k[j]; // the first of its top half
      if (was == EMPTY || was == top)
        break;
      h = (h + 1u) & (SAMPLE_SLOTS - 1u);
    }
    slot[j] = h;
  }
  __syncthreads();
#pragma unroll
  for (int j = 0; j < PER; ++j)
    if (((s_low[slot[j]] ^ (uint32_t)k[j]) & ((1u << HI_SHIFT) - 1u)) != 0u &&
        (atomicAdd(&s_count[slot[j] & (SAMPLE_COUNTS - 1)], 1u) + 1u >= crowd ||
         atomicAdd(&s_matches, 1u) + 1u >= SAMPLE_MATCHES))
      s_crowded = 1u;
  __syncthreads();
  if (threadIdx.x == 0)
    *w = RunWords{0u, 0u, 0u, s_crowded, s_crowded ^ 1u, s_crowded};
}

// The first inversion of a run at i: its run [b, e); e - b > RUN_LONG stands
// for the gate.  False: no inversion at i, or not its run's first.
AXB_D bool run_at(const uint64_t *__restrict__ keys, int64_t n, int64_t i, int64_t &b, int64_t &e)
{
  const uint64_t k = keys[i], next = keys[i + 1];
  const uint64_t top = k >> HI_SHIFT;
  if (next >= k || (next >> HI_SHIFT) != top)
    return false;
  b = i;
  uint64_t at = k;
  while (b > 0)
  {
    const uint64_t before = keys[b - 1];
    if ((before >> HI_SHIFT) != top)
      break;
    if (before > at)
      return false;
    if (i - b >= RUN_SHORT)
    {
      e = b + RUN_LONG + 1;
      return true;
    }
    at = before;
    --b;
  }
  // the run's end, by doubling steps and bisection (the top halves are sorted)
  e = i + 2;
  int64_t step = 1;
  while (e < n && (keys[e] >> HI_SHIFT) == top && e - b <= RUN_LONG)
  {
    int64_t f = e + step < n ? e + step : n;
    while (f - e > 1 && (keys[f - 1] >> HI_SHIFT) != top)
      f = e + (f - e + 1) / 2;
    e = f;
    step *= 2;
  }
  return true;
}
// tinies: starts of the tiny runs; shorts, longs: {start, end} of the others.  A
// block gathers the runs of RUN_TILE keys in LDS and takes its place in the
// lists with one atomic each.  All of them meet in one word, 20 to 27 ns an
// atomic, and bound the kernel where most tiles hold a run: one per run took
// 0.8 ms for the 41k runs of 5M clustered points; one per 4096 keys 0.071 ms
// for 10M uniform points, one per 16384 keys 0.031 ms (loading 8 steps ahead
// in tiles of 4096 left it at 0.071 ms).
constexpr int RUN_TILE = 16384;
constexpr int RUN_BLOCK = 1024;
constexpr int RUN_AHEAD = 8;
static_assert(RUN_TILE % (RUN_BLOCK * RUN_AHEAD) == 0, "whole steps");
__global__ __launch_bounds__(RUN_BLOCK) void k_find_runs(const uint64_t *__restrict__ keys, int64_t n,
                                                   uint32_t *__restrict__ tinies,
                                                   uint2 *__restrict__ shorts,
                                                   uint2 *__restrict__ longs, RunWords *w)
{
  // a run on the list has an inversion, two keys, in the tile, and all but the
  // last of the tile end in it
  __shared__ uint32_t s_tiny[RUN_TILE / 2 + 1];
  __shared__ uint2 s_short[RUN_TILE / RUN_TINY + 2];
  __shared__ uint2 s_long[RUN_TILE / RUN_SHORT + 2];
  __shared__ uint32_t s_n[6];
  if (threadIdx.x < 6)
    s_n[threadIdx.x] = 0u;
  __syncthreads();
  const int64_t base = (int64_t)blockIdx.x * RUN_TILE;
  if (ld_agent(&w->gate) == 0u)
    for (int j = threadIdx.x; j < RUN_TILE && base + j + 1 < n; j += RUN_BLOCK * RUN_AHEAD)
    {
      uint64_t k[RUN_AHEAD], next[RUN_AHEAD];
#pragma unroll
      for (int a = 0; a < RUN_AHEAD; ++a)
      {
        const int64_t i = base + j + RUN_BLOCK * a + 1 < n ? base + j + RUN_BLOCK * a : n - 2;
        k[a] = keys[i];
        next[a] = keys[i + 1];
      }
      uint32_t inversions = 0u;
#pragma unroll
      for (int a = 0; a < RUN_AHEAD; ++a)
        if (base + j + RUN_BLOCK * a + 1 < n && next[a] < k[a] &&
            (next[a] >> HI_SHIFT) == (k[a] >> HI_SHIFT))
          inversions |= 1u << a;
      for (; inversions; inversions &= inversions - 1u)
      {
        int64_t b, e;
        if (!run_at(keys, n, base + j + RUN_BLOCK * (__ffs(inversions) - 1), b, e))
          continue;
        if (e - b <= RUN_TINY)
          s_tiny[atomicAdd(&s_n[0], 1u)] = (uint32_t)b;
        else if (e - b <= RUN_SHORT)
          s_short[atomicAdd(&s_n[1], 1u)] = make_uint2((uint32_t)b, (uint32_t)e);
        else if (e - b <= RUN_LONG)
          s_long[atomicAdd(&s_n[2], 1u)] = make_uint2((uint32_t)b, (uint32_t)e);
        else
          st_agent(&w->gate, 1u);
      }
    }
  __syncthreads();
  if (threadIdx.x == 0)
  {
    s_n[3] = s_n[0] ? atomicAdd(&w->tinies, s_n[0]) : 0u;
    s_n[4] = s_n[1] ? atomicAdd(&w->shorts, s_n[1]) : 0u;
    s_n[5] = s_n[2] ? atomicAdd(&w->longs, s_n[2]) : 0u;
  }
  __syncthreads();
  for (uint32_t j = threadIdx.x; j < s_n[0]; j += RUN_BLOCK)
    tinies[s_n[3] + j] = s_tiny[j];
  for (uint32_t j = threadIdx.x; j < s_n[1]; j += RUN_BLOCK)
    shorts[s_n[4] + j] = s_short[j];
  for (uint32_t j = threadIdx.x; j < s_n[2]; j += RUN_BLOCK)
    longs[s_n[5] + j] = s_long[j];
}

// Stable insertion sort of a tiny run by a thread.
AXB_D void fix_tiny_run(uint64_t *keys, uint32_t *vals, int64_t n, int64_t b)
{
  const uint64_t top = keys[b] >> HI_SHIFT;
  for (int64_t j = b + 1; j < n && j - b < RUN_TINY; ++j)
  {
    const uint64_t k = keys[j];
    if ((k >> HI_SHIFT) != top)
      break;
    const uint32_t v = vals[j];
    int64_t h = j;
    while (h > b && keys[h - 1] > k)
    {
      keys[h] = keys[h - 1], vals[h] = vals[h - 1];
      --h;
    }
    keys[h] = k, vals[h] = v;
  }
}

// A short run by a wavefront: bitonic sort in registers of (low half,
// position), which is the stable order.
AXB_D void fix_short_run(uint64_t *keys, uint32_t *vals, uint2 be)
{
  static_assert(RUN_SHORT == 64, "a key per lane");
  constexpr uint64_t LOW = (1ull << HI_SHIFT) - 1ull;
  const int lane = threadIdx.x & 63;
  const bool in = lane < (int)(be.y - be.x); // at most RUN_SHORT
  unsigned long long k = ~0ull;
  uint64_t top = 0;
  uint32_t v = 0;
  if (in)
  {
    const uint64_t key = keys[be.x + lane];
    v = vals[be.x + lane];
    top = key & ~LOW;
    k = ((key & LOW) << 6) | (uint64_t)lane;
  }
#pragma unroll
  for (int span = 2; span <= 64; span *= 2)
#pragma unroll
    for (int stride = span / 2; stride > 0; stride /= 2)
    {
      const unsigned long long o = __shfl_xor(k, stride, 64);
      const bool smaller = ((lane & stride) == 0) == ((lane & span) == 0);
      k = (o < k) == smaller ? o : k;
    }
  const uint32_t from = (uint32_t)__shfl((int)v, (int)(k & 63ull), 64);
  if (in)
  {
    keys[be.x + lane] = top | (k >> 6);
    vals[be.x + lane] = from;
  }
}

// The tiny runs by the first TINY_BLOCKS blocks, the short ones by the others.
// 10M points in 1000 clusters of sigma 0.001, runs of 10 to 60 keys: 2.9 ms
// with a thread per short run, 0.11 here.
constexpr int TINY_BLOCKS = 256, SHORT_BLOCKS = 1024;
__global__ __launch_bounds__(256) void k_fix_runs(uint64_t *keys, uint32_t *vals, int64_t n,
                                                  const uint32_t *__restrict__ tinies,
                                                  const uint2 *__restrict__ shorts,
                                                  const RunWords *__restrict__ w)
{
  if (w->gate)
    return;
  if (blockIdx.x < TINY_BLOCKS)
  {
    const uint32_t runs = w->tinies;
    for (uint32_t r = blockIdx.x * 256u + threadIdx.x; r < runs; r += TINY_BLOCKS * 256u)
      fix_tiny_run(keys, vals, n, tinies[r]);
  }
  else
  {
    const uint32_t runs = w->shorts;
    for (uint32_t r = (blockIdx.x - TINY_BLOCKS) * 4u + threadIdx.x / 64u; r < runs;
         r += SHORT_BLOCKS * 4u)
      fix_short_run(keys, vals, shorts[r]);
  }
}

// A block per long run: bitonic sort in LDS of (low half, position), which is
// the stable order.
__global__ __launch_bounds__(256) void k_fix_long_runs(uint64_t *keys, uint32_t *vals,
                                                       const uint2 *__restrict__ list,
                                                       const RunWords *__restrict__ w)
{
  __shared__ uint64_t s_key[RUN_LONG];
  __shared__ uint32_t s_val[RUN_LONG];
  constexpr uint64_t LOW = (1ull << HI_SHIFT) - 1ull;
  static_assert(RUN_LONG == 4096, "positions of 12 bits");
  const uint32_t runs = w->gate ? 0u : w->longs;
  for (uint32_t r = blockIdx.x; r < runs; r += gridDim.x)
  {
    const uint2 be = list[r];
    const int m = (int)(be.y - be.x); // at most RUN_LONG
    int size = 128;
    while (size < m)
      size *= 2;
    const uint64_t top = keys[be.x] & ~LOW;
    __syncthreads(); // the run before is written out; every thread has read top
    for (int j = threadIdx.x; j < size; j += 256)
    {
      s_key[j] = j < m ? ((keys[be.x + j] & LOW) << 12) | (uint64_t)j : ~0ull;
      if (j < m)
        s_val[j] = vals[be.x + j];
    }
    __syncthreads();
    for (int span = 2; span <= size; span *= 2)
      for (int stride = span / 2; stride > 0; stride /= 2)
      {
        for (int j = threadIdx.x; j < size / 2; j += 256)
        {
          const int lo = 2 * j - (j & (stride - 1)), hi = lo + stride;
          const uint64_t x = s_key[lo], y = s_key[hi];
          if ((x > y) == ((lo & span) == 0))
            s_key[lo] = y, s_key[hi] = x;
        }
        __syncthreads();
      }
    for (int j = threadIdx.x; j < m; j += 256)
    {
      const uint64_t x = s_key[j];
      keys[be.x + j] = top | (x >> 12);
      vals[be.x + j] = s_val[x & 4095ull];
    }
  }
}

} // namespace

size_t sort_workspace_bytes(int64_t n, int passes, int)
{
  const int64_t tiles = div_up(n, SORT_TILE);
  return sizeof(uint32_t) *
         (size_t)(passes * 256 + 2 * passes + (int64_t)passes * tiles * 256);
}

hipError_t sort_keys63(uint64_t *keys0, uint64_t *keys1, uint32_t *vals0, uint32_t *vals1,
                       int64_t n, uint32_t *hist, void *workspace, uint32_t *words,
                       uint32_t *err, hipStream_t stream)
{
  if (!sort_top_first(n))
    return radix_sort_pairs<uint64_t>(keys0, keys1, vals0, vals1, n, 8, 0, false, hist,
                                      workspace, err, stream, nullptr);
  RunWords *w = (RunWords *)words;
  AXB_LAUNCH(k_sample_runs, dim3(1), dim3(1024), 0, stream, keys0, n, sample_crowd(n), w);
  hipError_t e = radix_sort_pairs<uint64_t>(keys0, keys1, vals0, vals1, n, 4, HI_SHIFT, false,
                                            hist, workspace, err, stream, &w->top);
  if (e != hipSuccess)
    return e;
  // the other buffers hold the lists (a tiny run has at least two keys, a
  // short one 9, a long one 65)
  uint2 *shorts = (uint2 *)keys1, *longs = (uint2 *)keys1 + n / 2;
  AXB_LAUNCH(k_find_runs, dim3((unsigned)div_up(n, RUN_TILE)), dim3(RUN_BLOCK), 0, stream, keys0, n,
             vals1, shorts, longs, w);
  AXB_LAUNCH(k_fix_runs, dim3(TINY_BLOCKS + SHORT_BLOCKS), dim3(256), 0, stream, keys0, vals0, n,
             vals1, shorts, w);
  AXB_LAUNCH(k_fix_long_runs, dim3(512), dim3(256), 0, stream, keys0, vals0, longs, w);
  // nothing to do unless the gate is open
  return radix_sort_pairs<uint64_t>(keys0, keys1, vals0, vals1, n, 8, 0, true, nullptr,
                                    workspace, err, stream, &w->gate, &w->crowded);
}
hipError_t radix_sort_pairs_u32(uint32_t *keys0, uint32_t *keys1,
                                uint32_t *vals0, uint32_t *vals1, int64_t n,
                                int passes, uint32_t *hist, void *workspace,
                                uint32_t *err, hipStream_t stream)
{
  return radix_sort_pairs<uint32_t>(keys0, keys1, vals0, vals1, n, passes, 0, false,
                                    hist, workspace, err, stream, nullptr);
}

size_t scan_workspace_bytes(int64_t n)
{
  return sizeof(int64_t) * (size_t)(div_up(n, SCAN_TILE) + 1);
}

// In place (out == in) is allowed: each element is read and written by the
// same thread.  n < 2^31 * SCAN_TILE (the grid's x limit).
template <class Tin, class Tout, bool INC>
static hipError_t scan_impl(const Tin *in, Tout *out, int64_t n, void *workspace, uint32_t *,
                            hipStream_t stream, uint8_t *flags = nullptr, int64_t limit = 0)
{
  if (n <= 0)
    return hipSuccess;
  const int64_t tiles = div_up(n, SCAN_TILE);
  int64_t *sums = (int64_t *)workspace;
  AXB_LAUNCH(k_scan_tile_sums<Tin>, dim3((unsigned)tiles), dim3(SCAN_BLOCK), 0, stream, in, n,
             sums);
  AXB_LAUNCH(k_scan_tile_offsets, dim3(1), dim3(SCAN_OFFSETS_BLOCK), 0, stream, sums, tiles);
  AXB_LAUNCH((k_scan_tiles<Tin, Tout, INC>), dim3((unsigned)tiles), dim3(SCAN_BLOCK), 0, stream,
             in, out, n, sums, flags, limit);
  return hipGetLastError();
}

hipError_t exclusive_scan_i64(const int64_t *in, int64_t *out, int64_t n, void *workspace,
                              uint32_t *err, hipStream_t stream, uint8_t *over_flags,
                              int64_t over_limit)
{
  return scan_impl<int64_t, int64_t, false>(in, out, n, workspace, err, stream, over_flags,
                                            over_limit);
}
hipError_t inclusive_scan_i32(const int32_t *in, int32_t *out, int64_t n,
                              void *workspace, uint32_t *err,
                              hipStream_t stream)
{
  return scan_impl<int32_t, int32_t, true>(in, out, n, workspace, err, stream);
}

hipError_t fill_u32(uint32_t *p, uint32_t v, int64_t n, hipStream_t stream)
{
  if (n <= 0)
    return hipSuccess;
  AXB_LAUNCH(k_fill_u32, dim3(fill_grid(n)), dim3(256), 0, stream, p,
                     v, n, (const uint32_t *)nullptr);
  return hipGetLastError();
}
hipError_t launch_iota_u32(uint32_t *p, int64_t n, hipStream_t stream)
{
  if (n <= 0)
    return hipSuccess;
  AXB_LAUNCH(k_iota_u32, dim3(fill_grid(n)), dim3(256), 0, stream, p, n);
  return hipGetLastError();
}
hipError_t fill_u64(uint64_t *p, uint64_t v, int64_t n, hipStream_t stream)
{
  if (n <= 0)
    return hipSuccess;
  AXB_LAUNCH(k_fill_u64, dim3(fill_grid(n)), dim3(256), 0, stream, p,
                     v, n);
  return hipGetLastError();
}

} // namespace axb
