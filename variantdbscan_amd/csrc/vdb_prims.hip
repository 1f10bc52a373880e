// Device-wide primitives: scans, stable LSD radix sort, extent reduction.
#include "vdb_prims.h"
#include "vdb_blocksort.h"

namespace vdb {

namespace {

constexpr int kScanBlock = 256;
constexpr int kScanItems = 8;
constexpr int kScanTile = kScanBlock * kScanItems; // 2048

template <typename T> __device__ __forceinline__ T wave_incl_scan(T x)
{
    int lane = lane_id();
#pragma unroll
    for (int o = 1; o < kWave; o <<= 1) {
        T y = __shfl_up(x, o, kWave);
        if (lane >= o) x += y;
    }
    return x;
}

// exclusive scan across the block; sm must hold NW+1 elements
template <typename T, int NW>
__device__ __forceinline__ T block_excl_scan(T v, T *sm, T *block_total)
{
    int lane = lane_id(), w = threadIdx.x / kWave;
    T inc = wave_incl_scan(v);
    if (lane == kWave - 1) sm[w] = inc;
    __syncthreads();
    if (threadIdx.x == 0) {
        T run = 0;
        for (int i = 0; i < NW; i++) {
            T t = sm[i];
            sm[i] = run;
            run += t;
        }
        sm[NW] = run;
    }
    __syncthreads();
    T r = sm[w] + inc - v;
    *block_total = sm[NW];
    __syncthreads();
    return r;
}

// Scan inputs: a plain array, or the population counts of an array of
// 32-bit words (the scan then numbers the set bits).
struct PopcSrc {
    const uint32_t *w;
    __device__ uint32_t operator[](size_t i) const { return (uint32_t)__popc(w[i]); }
};

template <typename Src, typename Out>
__global__ void __launch_bounds__(kScanBlock) k_tile_sums(Src in, size_t n, Out *sums)
{
    __shared__ Out sm[kScanBlock / kWave + 1];
    size_t base = (size_t)blockIdx.x * kScanTile + (size_t)threadIdx.x * kScanItems;
    Out s = 0;
#pragma unroll
    for (int i = 0; i < kScanItems; i++)
        if (base + i < n) s += (Out)in[base + i];
    Out tot;
    block_excl_scan<Out, kScanBlock / kWave>(s, sm, &tot);
    if (threadIdx.x == 0) sums[blockIdx.x] = tot;
}

// tile_off == nullptr: single tile, writes total
template <typename Src, typename Out>
__global__ void __launch_bounds__(kScanBlock)
    k_tile_scan(Src in, Out *out, size_t n, const Out *tile_off, Out *total)
{
    __shared__ Out sm[kScanBlock / kWave + 1];
    size_t base = (size_t)blockIdx.x * kScanTile + (size_t)threadIdx.x * kScanItems;
    Out v[kScanItems];
    Out s = 0;
#pragma unroll
    for (int i = 0; i < kScanItems; i++) {
        v[i] = (base + i < n) ? (Out)in[base + i] : (Out)0;
        s += v[i];
    }
    Out tot;
    Out run = block_excl_scan<Out, kScanBlock / kWave>(s, sm, &tot);
    if (tile_off) run += tile_off[blockIdx.x];
#pragma unroll
    for (int i = 0; i < kScanItems; i++) {
        if (base + i < n) out[base + i] = run;
        run += v[i];
    }
    if (!tile_off && total && threadIdx.x == 0) *total = tot;
}

// Up to kScanOne elements one block takes them all, 4 consecutive ones a
// thread and round: one launch of 5.4 us instead of two of 8.2 (6,252 words).
constexpr int kOneBlock = 1024;
constexpr size_t kScanOne = 16384;
template <typename Src, typename Out>
__global__ void __launch_bounds__(kOneBlock) k_scan_one(Src in, Out *out, uint32_t n, Out *total)
{
    constexpr int W = kOneBlock / kWave, R = (int)(kScanOne / (4 * kOneBlock));
    __shared__ Out sm[W + 1];
    Out v[R][4], s[R];
#pragma unroll
    for (int r = 0; r < R; r++) {
        const uint32_t base = (uint32_t)(r * kOneBlock + (int)threadIdx.x) * 4u;
        s[r] = 0;
#pragma unroll
        for (int i = 0; i < 4; i++) {
            v[r][i] = base + i < n ? (Out)in[base + i] : (Out)0;
            s[r] += v[r][i];
        }
    }
    Out off = 0;
#pragma unroll
    for (int r = 0; r < R; r++) {
        const uint32_t base = (uint32_t)(r * kOneBlock + (int)threadIdx.x) * 4u;
        if ((uint32_t)(r * kOneBlock) * 4u >= n) break; // block-uniform
        Out tot;
        Out run = block_excl_scan<Out, W>(s[r], sm, &tot) + off;
        off += tot;
#pragma unroll
        for (int i = 0; i < 4; i++) {
            if (base + i < n) out[base + i] = run;
            run += v[r][i];
        }
    }
    if (total && threadIdx.x == 0) *total = off;
}

// Up to kScanFewTiles tiles, the second pass needs no scan of the tile sums:
// each block adds up the sums of the tiles before it (at most that many
// loads), and the last block writes the total.
constexpr unsigned kScanFewTiles = 1024;
template <typename Src, typename Out>
__global__ void __launch_bounds__(kScanBlock)
    k_tile_scan_few(Src in, Out *out, size_t n, const Out *sums, Out *total)
{
    __shared__ Out sm[kScanBlock / kWave + 1];
    __shared__ Out red[kScanBlock / kWave];
    Out part = 0;
    for (unsigned t = threadIdx.x; t < blockIdx.x; t += kScanBlock) part += sums[t];
#pragma unroll
    for (int o = kWave / 2; o > 0; o >>= 1) part += __shfl_xor(part, o, kWave);
    if (lane_id() == 0) red[threadIdx.x / kWave] = part;
    __syncthreads();
    Out off = 0;
#pragma unroll
    for (int w = 0; w < kScanBlock / kWave; w++) off += red[w];
    size_t base = (size_t)blockIdx.x * kScanTile + (size_t)threadIdx.x * kScanItems;
    Out v[kScanItems];
    Out s = 0;
#pragma unroll
    for (int i = 0; i < kScanItems; i++) {
        v[i] = (base + i < n) ? (Out)in[base + i] : (Out)0;
        s += v[i];
    }
    Out tot;
    Out run = block_excl_scan<Out, kScanBlock / kWave>(s, sm, &tot) + off;
#pragma unroll
    for (int i = 0; i < kScanItems; i++) {
        if (base + i < n) out[base + i] = run;
        run += v[i];
    }
    if (total && blockIdx.x == gridDim.x - 1 && threadIdx.x == 0) *total = off + tot;
}

template <typename Src, typename Out>
int scan_impl(Context &c, Src in, Out *out, size_t n, Out *total_dev, int level)
{
    if (n == 0) {
        if (total_dev) VDB_HIP(hipMemsetAsync(total_dev, 0, sizeof(Out), c.stream()));
        return kOk;
    }
    if (n <= (size_t)kScanTile) {
        k_tile_scan<Src, Out><<<1, kScanBlock, 0, c.stream()>>>(in, out, n, nullptr, total_dev);
        VDB_HIP(hipGetLastError());
        return kOk;
    }
    if (n <= kScanOne) {
        k_scan_one<Src, Out><<<1, kOneBlock, 0, c.stream()>>>(in, out, (uint32_t)n, total_dev);
        VDB_HIP(hipGetLastError());
        return kOk;
    }
    size_t tiles = (n + kScanTile - 1) / kScanTile;
    char na[32], nb[32];
    snprintf(na, sizeof na, "scan.L%d.a.%d", level, (int)sizeof(Out));
    snprintf(nb, sizeof nb, "scan.L%d.b.%d", level, (int)sizeof(Out));
    Out *sums = nullptr, *offs = nullptr;
    VDB_TRY(c.get(na, tiles, &sums));
    k_tile_sums<Src, Out><<<(unsigned)tiles, kScanBlock, 0, c.stream()>>>(in, n, sums);
    VDB_HIP(hipGetLastError());
    if (tiles <= kScanFewTiles) {
        k_tile_scan_few<Src, Out><<<(unsigned)tiles, kScanBlock, 0, c.stream()>>>(in, out, n, sums,
                                                                                  total_dev);
        VDB_HIP(hipGetLastError());
        return kOk;
    }
    VDB_TRY(c.get(nb, tiles, &offs));
    VDB_TRY((scan_impl<const Out *, Out>(c, sums, offs, tiles, total_dev, level + 1)));
    k_tile_scan<Src, Out><<<(unsigned)tiles, kScanBlock, 0, c.stream()>>>(in, out, n, offs, nullptr);
    VDB_HIP(hipGetLastError());
    return kOk;
}

// ------------------------------------------------------------ radix sort
// Digits of 8 or 9 bits, whichever takes fewer passes; tiles of kSortBlock
// times ITEMS pairs. Up to kFewTiles tiles the scatter adds up the tiles'
// histograms itself (FEW), which saves a pass the two launches of a scan, and
// the tiles are as small as that allows, so that more blocks share the pairs.
// A pass over 50,000 pairs takes 9.5 us in 2 launches (20 in 4), over 100,003
// 10.8 (19).
constexpr int kSortBlock = 512;
constexpr int kSortWaves = kSortBlock / kWave;
constexpr unsigned kFewTiles = 64;

// hist: by digit, then tile, for the scan; FEW: by tile, then digit
template <int BITS, int ITEMS, bool FEW>
__global__ void __launch_bounds__(kSortBlock)
    k_radix_hist(const uint32_t *keys, size_t n, int shift, uint32_t *hist, unsigned tiles)
{
    constexpr int D = 1 << BITS;
    __shared__ uint32_t h[kSortWaves][D];
    for (int i = threadIdx.x; i < kSortWaves * D; i += kSortBlock) (&h[0][0])[i] = 0;
    __syncthreads();
    int w = threadIdx.x / kWave;
    size_t base = (size_t)blockIdx.x * (kSortBlock * ITEMS);
    uint32_t k[ITEMS];
#pragma unroll
    for (int i = 0; i < ITEMS; i++) {
        size_t idx = base + (size_t)i * kSortBlock + threadIdx.x;
        k[i] = idx < n ? keys[idx] : 0u;
    }
#pragma unroll
    for (int i = 0; i < ITEMS; i++)
        if (base + (size_t)i * kSortBlock + threadIdx.x < n)
            atomicAdd(&h[w][(k[i] >> shift) & (D - 1)], 1u);
    __syncthreads();
    for (int d = threadIdx.x; d < D; d += kSortBlock) {
        uint32_t s = 0;
        for (int q = 0; q < kSortWaves; q++) s += h[q][d];
        hist[FEW ? (size_t)blockIdx.x * D + d : (size_t)d * tiles + blockIdx.x] = s;
    }
}

// The block's first slot of every digit from the tiles' histograms: the pairs
// of smaller digits, and those of this digit in the tiles before.
template <int BITS>
__device__ __forceinline__ void few_bases(const uint32_t *hist, unsigned tiles, uint32_t *gbase)
{
    constexpr int D = 1 << BITS, P = kSortBlock / D; // P threads share a digit's tiles
    __shared__ uint32_t part[P][D], mine[P][D], sm[kSortWaves + 1];
    const int d = threadIdx.x % D, q = threadIdx.x / D;
    uint32_t all = 0, before = 0;
#pragma unroll 8
    for (unsigned t = q; t < tiles; t += P) {
        const uint32_t v = hist[(size_t)t * D + d];
        all += v;
        before += t < blockIdx.x ? v : 0u;
    }
    part[q][d] = all;
    mine[q][d] = before;
    __syncthreads();
    uint32_t total = 0, own = 0;
#pragma unroll
    for (int u = 0; u < P; u++) {
        total += part[u][d];
        own += mine[u][d];
    }
    uint32_t sum;
    const uint32_t smaller = block_excl_scan<uint32_t, kSortWaves>(q == 0 ? total : 0u, sm, &sum);
    if (q == 0) gbase[d] = smaller + own;
    __syncthreads();
}

// A tile is ranked, put in digit order in LDS and written out in runs per
// digit: 2M pairs take 9.6 us a pass of 8 bits (21 us with a rank and a store
// per 256 items, four barriers each, straight to the output).
template <int BITS, int ITEMS, bool FEW>
__global__ void __launch_bounds__(kSortBlock)
    k_radix_scatter(const uint32_t *keys, const uint32_t *vals, uint32_t *okeys, uint32_t *ovals,
                    size_t n, int shift, const uint32_t *offs, unsigned tiles)
{
    constexpr int D = 1 << BITS, kTile = kSortBlock * ITEMS;
    __shared__ BlockRank<BITS, kSortWaves> rk;
    __shared__ uint32_t xk[kTile], xv[kTile];
    __shared__ uint32_t gbase[D];
    const size_t base = (size_t)blockIdx.x * kTile;
    const uint32_t cnt = n - base < (size_t)kTile ? (uint32_t)(n - base) : (uint32_t)kTile;
    uint32_t k[ITEMS], v[ITEMS], pos[ITEMS] = {};
#pragma unroll
    for (int i = 0; i < ITEMS; i++) {
        uint32_t t = block_rank_item(i, ITEMS);
        k[i] = t < cnt ? keys[base + t] : 0xffffffffu;
        v[i] = t < cnt ? vals[base + t] : 0u;
    }
    if constexpr (FEW) few_bases<BITS>(offs, tiles, gbase);
    else
        for (int d = threadIdx.x; d < D; d += kSortBlock)
            gbase[d] = offs[(size_t)d * tiles + blockIdx.x];
    // the padding of the last tile ranks behind its real items
    block_rank<ITEMS, BITS, kSortWaves>(k, ITEMS, shift, pos, rk);
#pragma unroll
    for (int i = 0; i < ITEMS; i++) {
        xk[pos[i]] = k[i];
        xv[pos[i]] = v[i];
    }
    __syncthreads();
#pragma unroll
    for (int i = 0; i < ITEMS; i++) {
        uint32_t t = (uint32_t)i * kSortBlock + threadIdx.x;
        if (t < cnt) {
            uint32_t key = xk[t], d = (key >> shift) & (D - 1);
            uint32_t dst = gbase[d] + (t - rk.start[d]);
            okeys[dst] = key;
            ovals[dst] = xv[t];
        }
    }
}

template <int BITS, int ITEMS, bool FEW>
int radix_pass(Context &c, const uint32_t *ka, const uint32_t *va, uint32_t *kb, uint32_t *vb,
               size_t n, int shift, uint32_t *hist, uint32_t *offs)
{
    const unsigned tiles = ceil_div(n, kSortBlock * ITEMS);
    k_radix_hist<BITS, ITEMS, FEW><<<tiles, kSortBlock, 0, c.stream()>>>(ka, n, shift, hist, tiles);
    VDB_HIP(hipGetLastError());
    if (!FEW) VDB_TRY(scan_exclusive_u32(c, hist, offs, (size_t)tiles << BITS, nullptr));
    k_radix_scatter<BITS, ITEMS, FEW><<<tiles, kSortBlock, 0, c.stream()>>>(
        ka, va, kb, vb, n, shift, FEW ? hist : offs, tiles);
    VDB_HIP(hipGetLastError());
    return kOk;
}

template <int BITS>
int radix_pass(Context &c, const uint32_t *ka, const uint32_t *va, uint32_t *kb, uint32_t *vb,
               size_t n, int shift, int items, uint32_t *hist, uint32_t *offs)
{
    if (items == 2) return radix_pass<BITS, 2, true>(c, ka, va, kb, vb, n, shift, hist, offs);
    if (items == 4) return radix_pass<BITS, 4, true>(c, ka, va, kb, vb, n, shift, hist, offs);
    if (items == 8) return radix_pass<BITS, 8, true>(c, ka, va, kb, vb, n, shift, hist, offs);
    return radix_pass<BITS, kSortItems, false>(c, ka, va, kb, vb, n, shift, hist, offs);
}

} // namespace

int bits_for(uint64_t m)
{
    int b = 0;
    while (b < 64 && ((uint64_t)1 << b) < m) b++;
    return b;
}

int scan_exclusive_u32(Context &c, const uint32_t *in, uint32_t *out, size_t n,
                       uint32_t *total_dev)
{
    return scan_impl<const uint32_t *, uint32_t>(c, in, out, n, total_dev, 0);
}

int scan_popc_u32(Context &c, const uint32_t *words, uint32_t *out, size_t n)
{
    return scan_impl<PopcSrc, uint32_t>(c, PopcSrc{words}, out, n, nullptr, 0);
}

int scan_exclusive_u32_u64(Context &c, const uint32_t *in, uint64_t *out, size_t n,
                           uint64_t *total_dev)
{
    return scan_impl<const uint32_t *, uint64_t>(c, in, out, n, total_dev, 0);
}

int compact_count(Context &c, const uint32_t *flags, uint32_t *out, size_t n,
                  uint32_t *total_host)
{
    uint32_t *tot = nullptr;
    VDB_TRY(c.get("compact.total", 1, &tot));
    VDB_TRY(scan_exclusive_u32(c, flags, out, n, tot));
    void *h = nullptr;
    VDB_TRY(c.host_scratch(sizeof(uint32_t), &h));
    VDB_HIP(hipMemcpyAsync(h, tot, sizeof(uint32_t), hipMemcpyDeviceToHost, c.stream()));
    VDB_TRY(c.wait(c.stream()));
    *total_host = *(uint32_t *)h;
    return kOk;
}

int radix_sort_pairs(Context &c, uint32_t *keys, uint32_t *vals, uint32_t *tmp_keys,
                     uint32_t *tmp_vals, size_t n, int key_bits, uint32_t **keys_out,
                     uint32_t **vals_out)
{
    uint32_t *ka = keys, *va = vals, *kb = tmp_keys, *vb = tmp_vals;
    if (n > 1 && key_bits > 0) {
        // (the allocation-free mode keeps its scratch for 8-bit tables)
        const int bits = !c.in_arena() && (key_bits + 8) / 9 < (key_bits + 7) / 8 ? 9 : 8;
        const size_t D = (size_t)1 << bits;
        int items = 0; // of small tiles; 0: tiles of kSortItems, offsets by scan
        for (int i = 8; i >= 2 && !c.in_arena(); i /= 2)
            if (n <= (size_t)kFewTiles * kSortBlock * i) items = i;
        const size_t tiles = ceil_div(n, kSortBlock * (items ? items : kSortItems));
        uint32_t *hist = nullptr, *offs = nullptr;
        VDB_TRY(c.get("radix.hist", tiles * D, &hist));
        if (!items) VDB_TRY(c.get("radix.offs", tiles * D, &offs));
        for (int shift = 0; shift < key_bits; shift += bits) {
            if (bits == 8)
                VDB_TRY(radix_pass<8>(c, ka, va, kb, vb, n, shift, items, hist, offs));
            else
                VDB_TRY(radix_pass<9>(c, ka, va, kb, vb, n, shift, items, hist, offs));
            uint32_t *t = ka; ka = kb; kb = t;
            t = va; va = vb; vb = t;
        }
    }
    *keys_out = ka;
    *vals_out = va;
    return kOk;
}

} // namespace vdb
