// marxs_analysis.hip -- per-order figures of merit of a traced photon list
// on the GPU (MI355X, gfx950).
//
// The reference analyses every tolerancing variant on the host:
// effectivearea_from_photonlist (marxs/analysis/gratings.py:333-363) sums the
// probability of each grating order, resolvingpower_from_photonlist (215-270)
// takes astropy's sigma_clipped_stats of the dispersion coordinate of each
// order (sigma 3, at most 5 rounds, median centre, std with ddof 0: drop
// non-finite values, then repeat {keep values within median -/+ 3 std,
// inclusive} until a round removes nothing).
//
// Here the photon list stays in HBM and nothing is sorted.  The kept set of
// every round is an interval of values, so it is enough to know the values in
// bins (count, mean, squared deviations of each) and to look inside the few
// bins that hold a bound or the median:
//   1. sample  one workgroup per order sorts up to 4096 photons drawn over the
//              list and takes evenly filled bin edges from them;
//   2. split   each workgroup takes one chunk of photons (pieces of 64 from all
//              over the list), orders its counted
//              values by (order, bin) in LDS and writes them back in that order
//              with the offset of every (order, bin) piece, the piece's sums of
//              deviations and squared deviations from an edge of the bin, and
//              the probability sum of each order;
//   3. merge   adds up the pieces' sums, and copies the values of the bins that
//              are likely to be looked into to one place each;
//   4. clip    one workgroup per order: the rounds, from the bins' sums and the
//              values of the bins that hold a bound or the median.
// The bins only decide how fast the answer is found, never what it is: edges
// are compared exactly, the median is selected exactly, and a bound's bin is
// summed value by value.  Every sum has a fixed order for a given photon list.
// The library allocates nothing: all scratch is the caller's workspace.
//
// What it costs: the columns are read once (20 B per photon) and the counted
// values written once (8 B each); a method that keeps no table of values could
// do with the read alone.  The two device-wide radix sorts this replaced
// moved each value nine times.  CaptureResAeff on 8e6 photons in 15 orders:
// 1230 us a call with them, 320 us now, 213 us of it in the kernels (160 MB: 26
// us at the card's read rate); on 5e4 photons 400 us in 44 launches, now 133 us
// in 4, 88 us of it in the kernels.  The split kernel has the vector unit busy
// for 39 % of its time and half of its waves' time waits; the kernels with one
// workgroup per order (sample, clip) wait for loads and barriers for more than
// half of theirs on 15 of the 256 CUs.

#include <hip/hip_runtime.h>
#include <mutex>
#include <stdint.h>
#include <stdio.h>
#include <math.h>

#include "marxs_hip.h"

__attribute__((visibility("hidden"))) void mx_set_error(const char *msg);

#define MX_OS_SAMPLE 4096      // photons looked at for the bin edges
#define MX_OS_SPLIT 512        // work-items per splitting workgroup
#define MX_OS_SPLIT_WAVES (MX_OS_SPLIT / 64)
// Photons per work-item of the splitting kernel.  12 (chunks of 6144, 77 KiB
// of LDS, two workgroups per CU) keeps the number of chunks, and with it the
// piece tables, small; below MX_OS_FEW photons that would leave CUs without a
// chunk (326 chunks at 2e6), so 4 are taken there.
#define MX_OS_ROWS 12
#define MX_OS_ROWS_FEW 4
#define MX_OS_FEW 2000000
#define MX_OS_MERGE 512        // work-items per merging workgroup
#define MX_OS_MERGE_RUN 8      // chunks a work-item of it merges, about
#define MX_OS_NEAR 12          // bins around the middle that are copied to one place,
#define MX_OS_ENDS 4           // and at each end
#define MX_OS_PIECES 8         // pieces in flight per work-item
// Work-items per clipping workgroup: with 1024 each wave would have 128 VGPRs,
// and the kernel needs 174.
#define MX_OS_CLIP 512
#define MX_OS_LIST 15360       // values of a bin the clipping workgroup holds in LDS
#define MX_OS_HIST 2048        // buckets of a selection round
#define MX_OS_CAND 64          // values ranked by counting, one per lane
#define MX_OS_MAX_BINS 512
// An order that holds more than MX_OS_SKEW times its even share of the sample
// has its bins in proportion, at the cost of the others (order_bins): every
// round of the clipping passes over the two bins with the bounds, so bins of
// one large order among many were what a call took (1e7 photons, 97 % of them
// in one of 64 orders: 7028 us a call with 16 bins each, 707 so; one of 15
// orders 1963 us with 64 bins, 676).  Below that line bins are at most four times
// larger than even ones.
#define MX_OS_SKEW 4
#define MX_OS_LEAST_BINS 8
#define MX_OS_LUT 256

static size_t align256(size_t x) { return (x + 255) & ~(size_t)255; }

// Sizes of one call and the byte offsets of its workspace parts.
struct OsPlan {
    int32_t no, bins, keys;           // orders; bins per order; pieces per chunk
    int32_t rows, chunk, groups;      // photons per work-item and per chunk; groups of chunks
    int64_t chunks, stride;           // chunks; length of an offset row (one per piece, an entry per chunk)
    size_t edges, off, piece, grp, place, next, lay, psum, vals, copied, total;
};

// One bin: place of its values when they were copied (-1: in pieces), their
// count, the sums of deviations and of their squares from bin_ref.
struct BinInfo {
    int64_t at;
    double n, s1, s2;
};

// Bins per order (as shared evenly): about 1000 (order, bin) pieces in all, so that the split
// kernel's counters fit beside the values in LDS; each order has one more
// piece for the photons whose value is not counted.
static void os_plan(int64_t n, int no, bool values, OsPlan &L) {
    int bins = 0;
    if (values) {
        bins = 16;
        while (bins * 2 <= MX_OS_MAX_BINS && bins * 2 * no <= 1024) bins *= 2;
    }
    L.no = no;
    L.bins = bins;
    L.keys = no * (bins + 1);
    L.rows = n >= MX_OS_FEW ? MX_OS_ROWS : MX_OS_ROWS_FEW;
    L.chunk = L.rows * MX_OS_SPLIT;
    L.chunks = (n + L.chunk - 1) / L.chunk;
    L.stride = (L.chunks + 63) & ~(int64_t)63;
    const int64_t run = (int64_t)MX_OS_MERGE * MX_OS_MERGE_RUN / (bins > 0 ? bins : 1);   // chunks per group
    const int64_t g = (L.chunks + run - 1) / run;
    L.groups = (int32_t)(g < 1 ? 1 : (g > 256 ? 256 : g));
    size_t o = 0;
    L.edges = o;  o += align256(sizeof(double) * (size_t)no * bins);
    L.off = o;    o += align256(sizeof(uint16_t) * (size_t)L.stride * (L.keys + 1));
    L.piece = o;  o += align256(sizeof(double2) * (size_t)L.chunks * no * bins);
    L.grp = o;    o += align256(sizeof(BinInfo) * (size_t)L.groups * no * bins);
    L.place = o;  o += align256(sizeof(int64_t) * (size_t)no * bins);
    L.next = o;   o += align256(sizeof(unsigned long long));
    L.lay = o;    o += align256(sizeof(int32_t) * (MX_MAX_ORDERS + 2));
    L.psum = o;   o += align256(sizeof(double) * (size_t)L.chunks * no);
    L.vals = o;   o += values ? align256(sizeof(double) * (size_t)L.chunks * L.chunk) : 0;
    L.copied = o; o += values ? align256(sizeof(double) * (size_t)(n > 0 ? n : 1)) : 0;
    L.total = o;
    // The size that callers are told, and that the static workspace is
    // checked against, is that of the limits this library states (27.17 B per
    // photon with values, 32 B per order and 4096 photons): the call itself
    // needs less from some thousand photons on.
    const int64_t nb = n <= 0 ? 1 : (n + 4095) / 4096 > 16384 ? 16384 : (n + 4095) / 4096;
    const size_t stated = (size_t)32 * nb * no + (values ? (size_t)27 * n + (size_t)n * 17 / 100 : 0) + 1024;
    if (L.total < stated) L.total = align256(stated);
}

// ------------------------------------------------------------ order lookup
// index of order o in the list (linear: at most MX_MAX_ORDERS entries), -1
__device__ __forceinline__ int order_index(const int *ords, int no, int o) {
    for (int j = 0; j < no; ++j)
        if (ords[j] == o) return j;
    return -1;
}

// Order number -> index through a table of MX_OS_LUT entries in LDS when the
// orders span fewer values (the usual case), else the linear search.  Built
// by the whole workgroup.
struct OrderLut {
    const int *t;
    const int *ords;
    int lo, no;
    bool ok;
    __device__ __forceinline__ int operator()(int o) const {
        if (!ok) return order_index(ords, no, o);
        const int64_t d = (int64_t)o - lo;
        const int k = (d >= 0 && d < MX_OS_LUT) ? t[d] : MX_MAX_ORDERS;
        return k < MX_MAX_ORDERS ? k : -1;
    }
};

__device__ __forceinline__ OrderLut build_lut(const MxOrderStats &a, int *ords, int *lut) {
    const int no = a.n_orders;
    for (int k = threadIdx.x; k < no; k += blockDim.x) ords[k] = a.orders[k];
    for (int j = threadIdx.x; j < MX_OS_LUT; j += blockDim.x) lut[j] = MX_MAX_ORDERS;
    __syncthreads();
    int mn = 0x7fffffff, mx = INT32_MIN;
    for (int k = 0; k < no; ++k) {
        mn = ords[k] < mn ? ords[k] : mn;
        mx = ords[k] > mx ? ords[k] : mx;
    }
    OrderLut L;
    L.t = lut;
    L.ords = ords;
    L.lo = mn;
    L.no = no;
    L.ok = (int64_t)mx - (int64_t)mn < MX_OS_LUT;
    // the first index of an order number, as the linear search finds it
    if (L.ok)
        for (int k = threadIdx.x; k < no; k += blockDim.x) atomicMin(&lut[(int64_t)ords[k] - mn], k);
    __syncthreads();
    return L;
}

// ---------------------------------------------------------------- 1 sample
// Place of edge j (of bins - 1) among m sorted values: evenly filled bins, the
// outer two half as full (1/512 of the values at least, where the 3 sigma
// bounds of a bell curve still fall): the clipping looks into them every round.
__device__ __forceinline__ int edge_rank(int j, int bins, int m) {
    const double q = 0.5 / (bins - 1) > 1.0 / 512 ? 0.5 / (bins - 1) : 1.0 / 512;
    const int i = (int)((double)m * (q + (double)j * ((1.0 - 2.0 * q) / (bins - 2))));
    return i < m ? i : m - 1;
}

// The bins of an order: the first among those of all orders, and their number.
struct Bins {
    int first, n;
};
// As the sample kernel shared them out: the first bin of each order and, last,
// the end; then whether they are shared evenly.
// (Read by scalar loads: the kernels that read it do not write it.)
typedef const __attribute__((address_space(4))) int32_t *Layout;
__device__ __forceinline__ Layout layout(const OsPlan &L, const unsigned char *ws) { return (Layout)(ws + L.lay); }
__device__ __forceinline__ Bins bins_of(const OsPlan &L, const unsigned char *ws, int k) {
    const Layout lay = layout(L, ws);
    return {lay[k], lay[k + 1] - lay[k]};
}

// Bins of the order of this lane, by every wave for itself, from the photons of
// each order (`count`, of lane's order) among `looked` ones: powers of two, evenly or,
// when one order holds MX_OS_SKEW times its share, in proportion and
// MX_OS_LEAST_BINS at least.
__device__ __forceinline__ Bins order_bins(const OsPlan &L, int count, int looked, bool &even) {
    const int lane = threadIdx.x & 63;
    even = __ballot(count * L.no > MX_OS_SKEW * looked) == 0;
    if (even) return {lane * L.bins, L.bins};
    int total = count;
    for (int o = 32; o > 0; o >>= 1) total += __shfl_xor(total, o);
    int n = 0;
    if (lane < L.no) {
        const int share = count * (L.no * (L.bins - MX_OS_LEAST_BINS)) / total;
        n = MX_OS_LEAST_BINS;
        while (2 * n <= share && 2 * n <= MX_OS_MAX_BINS) n *= 2;
    }
    int end = n;
    for (int d = 1; d < 64; d <<= 1) {
        const int o = __shfl_up(end, d);
        if (lane >= d) end += o;
    }
    return {end - n, n};
}

// Bin edges of one order (one workgroup each): the finite, counted values of
// this order among MX_OS_SAMPLE photons, one from a pseudo-random place of
// each of as many equal parts of the list, sorted; the edges split them
// (edge_rank).  An edge that repeats moves up by one step of the number format, so
// that a value holding many photons has a bin of its own.  Bin of x: the
// number of edges <= x.  Bound by the latency of its loads and of the sort
// (17 us at 15 orders and 8e6 photons).
__global__ __launch_bounds__(1024) void mx_os_sample_kernel(MxOrderStats a, OsPlan L,
                                                             unsigned char *ws) {
    __shared__ double s[MX_OS_SAMPLE];
    __shared__ int cnt, held[256];
    const int k = blockIdx.x, t = threadIdx.x, lane = t & 63, mine = a.orders[k];
    double *edges = (double *)(ws + L.edges);
    if (k == 0 && t == 0) *(unsigned long long *)(ws + L.next) = 0;    // the merge kernel's allocator
    const bool filter = (a.flags & MX_OS_FILTER) != 0;
    if (t == 0) cnt = 0;
    if (t < 256) held[t] = 0;
    __syncthreads();
    const int number = lane < L.no ? a.orders[lane] : 0;
    const int64_t parts = a.n < MX_OS_SAMPLE ? a.n : MX_OS_SAMPLE;
    int64_t at[MX_OS_SAMPLE / 1024];
    int ord[MX_OS_SAMPLE / 1024];
#pragma unroll
    for (int r = 0; r < MX_OS_SAMPLE / 1024; ++r) {
        const int64_t i = t + 1024 * r;
        at[r] = -1;
        if (i < parts) {
            const int64_t b = i * a.n / parts, e = (i + 1) * a.n / parts;
            const uint32_t h = ((uint32_t)i * 2654435761u) >> 7;
            at[r] = b + (int64_t)h % (e - b);
        }
        ord[r] = parts > 0 ? a.order[at[r] >= 0 ? at[r] : 0] : 0;
    }
    double v[MX_OS_SAMPLE / 1024], pr[MX_OS_SAMPLE / 1024];
#pragma unroll
    for (int r = 0; r < MX_OS_SAMPLE / 1024; ++r) {
        if (ord[r] != mine) at[r] = -1;
        v[r] = parts > 0 ? a.value[at[r] >= 0 ? at[r] : 0] : 0.0;
        pr[r] = parts > 0 && filter ? a.prob[at[r] >= 0 ? at[r] : 0] : 1.0;
    }
    // (for order_bins, while the values are on their way; orders that are 256
    // apart are counted together)
#pragma unroll
    for (int r = 0; r < MX_OS_SAMPLE / 1024; ++r)
        if (t % 16 == 0 && t + 1024 * r < parts && ord[r] != INT32_MIN) atomicAdd(&held[ord[r] & 255], 1);
#pragma unroll
    for (int r = 0; r < MX_OS_SAMPLE / 1024; ++r)
        if (at[r] >= 0 && isfinite(v[r]) && (!filter || pr[r] > 0.0)) s[atomicAdd(&cnt, 1)] = v[r];
    __syncthreads();
    const int m = cnt;
    int size = 1;
    while (size < m) size *= 2;
    for (int i = m + t; i < size; i += 1024) s[i] = __builtin_inf();
    __syncthreads();
    bool even;
    // (with few orders none can hold that many times its share)
    const Bins lay = order_bins(L, lane < L.no && L.no > MX_OS_SKEW ? held[number & 255] : 0, (int)(parts + 15) / 16, even);
    const int bins = __builtin_amdgcn_readlane(lay.n, k), first = __builtin_amdgcn_readlane(lay.first, k);
    if (k == 0 && t < L.no) {
        int32_t *all = (int32_t *)(ws + L.lay);
        all[t] = lay.first;
        if (t == L.no - 1) all[L.no] = lay.first + lay.n;
        if (t == 0) all[MX_MAX_ORDERS + 1] = even ? 1 : 0;
    }
    if (m <= 512) {
        // few values: each goes to the place that its rank says, one step
        // instead of up to 45 with a barrier each
        int rank = 0;
        const double x = t < m ? s[t] : 0.0;
        if (t < m)
#pragma unroll 16
            for (int j = 0; j < m; ++j) rank += (s[j] < x || (s[j] == x && j < t)) ? 1 : 0;
        __syncthreads();
        if (t < m) s[rank] = x;
        __syncthreads();
        size = 1;
    }
    for (int w = 2; w <= size; w *= 2)
        for (int d = w / 2; d > 0; d /= 2) {
            for (int i = t; i < size / 2; i += 1024) {
                const int lo = 2 * i - (i & (d - 1)), hi = lo + d;
                const double x = s[lo], y = s[hi];
                if ((x > y) == ((lo & w) == 0)) {
                    s[lo] = y;
                    s[hi] = x;
                }
            }
            __syncthreads();
        }
    for (int j = t; j < bins; j += 1024) {
        // the last entry only fills the row
        double e = __builtin_inf();
        if (m > 0 && j < bins - 1) {
            e = s[edge_rank(j, bins, m)];
            if (j > 0 && s[edge_rank(j - 1, bins, m)] == e) e = nextafter(e, __builtin_inf());
        }
        edges[first + j] = e;
        ((int64_t *)(ws + L.place))[first + j] = -1;
    }
}

// What a bin's sums are taken about: its edge nearer to the middle of the
// order, so that deviations from any point between the bins' middle and that
// edge add up without cancelling; 0 for an order without a photon in the
// sample.
__device__ __forceinline__ double bin_ref(const double *edges, int bins, int b) {
    const double e = edges[b < bins / 2 ? b : b - 1];
    return isfinite(e) ? e : 0.0;
}

__device__ __forceinline__ int bin_of(const double *edges, int bins, double x) {
    int b = 0;
    for (int h = bins >> 1; h > 0; h >>= 1)
        if (edges[b + h - 1] <= x) b += h;
    return b;
}

// Sums over the lanes up to each one, by the cross-lane moves of the vector
// unit (a move through LDS costs ten times the latency).
template <int CTRL, int ROWS> __device__ __forceinline__ double lane_move(double v) {
    return __hiloint2double(__builtin_amdgcn_update_dpp(0, __double2hiint(v), CTRL, ROWS, 0xf, false),
                            __builtin_amdgcn_update_dpp(0, __double2loint(v), CTRL, ROWS, 0xf, false));
}
__device__ __forceinline__ double wave_scan(double v) {
    v += lane_move<0x111, 0xf>(v);    // one lane up within 16
    v += lane_move<0x112, 0xf>(v);
    v += lane_move<0x114, 0xf>(v);
    v += lane_move<0x118, 0xf>(v);
    v += lane_move<0x142, 0xa>(v);    // the last lane of 16 to the next 16
    v += lane_move<0x143, 0xc>(v);    // the last lane of 32 to the next 32
    return v;
}
__device__ __forceinline__ double lane_value(double v, int lane) {
    return __hiloint2double(__builtin_amdgcn_readlane(__double2hiint(v), lane),
                            __builtin_amdgcn_readlane(__double2loint(v), lane));
}
// Sum over the wave in a fixed order; every lane gets it.
__device__ __forceinline__ double wave_add(double v) { return lane_value(wave_scan(v), 63); }

// ----------------------------------------------------------------- 2 split
// LDS of the split kernel: the chunk's values (then its probabilities), the
// edges, one counter (16 bits) per wave and piece, piece starts.
static size_t split_lds(const OsPlan &L) {
    const int kh = (L.keys + 1) & ~1;
    return sizeof(double) * L.chunk + sizeof(double) * (size_t)L.no * L.bins +
           sizeof(uint16_t) * ((size_t)MX_OS_SPLIT_WAVES * kh + kh + 2);
}

// One chunk of photons ordered by (order, bin).  The chunk takes 64 consecutive
// photons for each row of each wave from equal steps over the whole list: in a
// list sorted by value a chunk of consecutive photons is one long piece of one
// bin, whose sums and copies are then one work-item's (1e7 photons sorted in two
// orders 2942 us a call, 456 so; unsorted 600 either way).  A photon's place is
// the start of its piece, plus the photons of the piece in the waves before, plus its
// rank within its wave, which an LDS counter of that wave and piece returns:
// only one wave uses it.  That places and sums are the same in every run assumes
// that the lanes of one LDS instruction are served in a fixed order, which no
// document states (the tests call twice and compare); in another order values
// would change places within a piece, and means their last bits.  Reads
// 20 B per photon and writes 8 B per counted value plus 18 B per piece; bound
// by the LDS work between (edge search 6 reads per value at 64 bins, counter,
// scatter, sums): 77 us for 8e6 photons in 15 orders (247 MB: 48 us at the
// card's copy rate).
template <int ROWS, bool VALUES>
__global__ __launch_bounds__(MX_OS_SPLIT, 4) void mx_os_split_kernel(MxOrderStats a, OsPlan L, unsigned char *ws) {
    extern __shared__ __align__(16) unsigned char sm[];
    __shared__ int ords[MX_MAX_ORDERS], lut[MX_OS_LUT], wtot[MX_OS_SPLIT_WAVES], lay[MX_MAX_ORDERS + 1];
    constexpr int CH = ROWS * MX_OS_SPLIT;
    const int t = threadIdx.x, lane = t & 63, w = t >> 6;
    const int kh = (L.keys + 1) & ~1, bins = VALUES ? L.bins : 0;
    double *buf = (double *)sm;
    double *edges = buf + CH;
    uint16_t *hist = (uint16_t *)(edges + (size_t)L.no * bins);   // [wave][kh]
    uint16_t *start = hist + MX_OS_SPLIT_WAVES * kh;              // [keys + 1]
    uint32_t *mine = (uint32_t *)(hist + w * kh);
    const int64_t c = blockIdx.x, step = (int64_t)MX_OS_SPLIT * L.chunks;
    const int64_t first = ((int64_t)w * L.chunks + c) * 64 + lane;   // photon of row r: first + r * step
    const bool filter = (a.flags & MX_OS_FILTER) != 0;
    const bool even = !VALUES || layout(L, ws)[MX_MAX_ORDERS + 1] != 0;
    // columns first: their latency covers the set-up below
    int ord[ROWS];
    double pr[ROWS], val[ROWS];
#pragma unroll
    for (int r = 0; r < ROWS; ++r) {
        const int64_t i = first + r * step;
        const bool in = i < a.n;
        ord[r] = in ? a.order[i] : INT32_MIN;
        pr[r] = in ? a.prob[i] : 0.0;
        val[r] = (VALUES && in) ? a.value[i] : 0.0;
    }
    for (int j = lane; j < kh / 2; j += 64) mine[j] = 0;
    if (VALUES) {
        const double *ge = (const double *)(ws + L.edges);
        for (int j = t; j < L.no * bins; j += MX_OS_SPLIT) edges[j] = ge[j];
        if (!even && t <= L.no) lay[t] = ((const int32_t *)(ws + L.lay))[t];
    }
    const OrderLut index_of = build_lut(a, ords, lut);
    __shared__ double part[MX_MAX_ORDERS];
    double *psum = (double *)(ws + L.psum);
    uint16_t *off = (uint16_t *)(ws + L.off) + c;
    if (!VALUES && L.no <= MX_OS_SPLIT_WAVES) {
        // sums alone, few orders: in registers (their counters in LDS would
        // be the same few words for all lanes: 1e7 photons of one order
        // 123 us a call, 101 us this way)
        double s[MX_OS_SPLIT_WAVES];
        int m[MX_OS_SPLIT_WAVES];
#pragma unroll
        for (int k = 0; k < MX_OS_SPLIT_WAVES; ++k) {
            s[k] = 0.0;
            m[k] = 0;
        }
#pragma unroll
        for (int r = 0; r < ROWS; ++r) {
            const int k0 = first + r * step < a.n ? index_of(ord[r]) : -1;
#pragma unroll
            for (int k = 0; k < MX_OS_SPLIT_WAVES; ++k) {
                s[k] += k == k0 ? pr[r] : 0.0;
                m[k] += k == k0 ? 1 : 0;
            }
        }
        __shared__ int count[MX_MAX_ORDERS];
#pragma unroll
        for (int k = 0; k < MX_OS_SPLIT_WAVES; ++k) {
            const double sum = wave_scan(s[k]), n = wave_scan((double)m[k]);
            if (lane == 63) {
                part[k * MX_OS_SPLIT_WAVES + w] = sum;
                count[k * MX_OS_SPLIT_WAVES + w] = (int)n;
            }
        }
        __syncthreads();
        if (t == 0) {
            int run = 0;
            for (int k = 0; k < L.no; ++k) {
                double x = 0.0;
                off[(size_t)k * L.stride] = (uint16_t)run;
                for (int q = 0; q < MX_OS_SPLIT_WAVES; ++q) {
                    x += part[k * MX_OS_SPLIT_WAVES + q];
                    run += count[k * MX_OS_SPLIT_WAVES + q];
                }
                psum[(size_t)k * L.chunks + c] = x;
            }
            off[(size_t)L.no * L.stride] = (uint16_t)run;
        }
        return;
    }
    // bins and pieces of order k
    auto first_key = [&](int k) { return even ? k * (bins + 1) : lay[k] + k; };
    const int keys = even ? L.keys : __builtin_amdgcn_readfirstlane(lay[L.no]) + L.no;
    uint32_t place[ROWS];   // piece and rank within the wave
    auto put = [&](int r, int key) {
        const int sh = (key & 1) * 16;
        const uint32_t old = atomicAdd(mine + (key >> 1), 1u << sh);
        place[r] = ((uint32_t)key << 16) | ((old >> sh) & 0xffffu);
    };
    if (even) {
#pragma unroll
        for (int r = 0; r < ROWS; ++r) {
            const bool in = first + r * step < a.n;
            const int k = in ? index_of(ord[r]) : -1;
            place[r] = 0xffffffffu;
            if (k >= 0) {
                int key = k;
                if (VALUES) {
                    const bool counted = isfinite(val[r]) && (!filter || pr[r] > 0.0);
                    key = k * (bins + 1) + (counted ? bin_of(edges + k * bins, bins, val[r]) : bins);
                }
                put(r, key);
            }
        }
    } else {
#pragma unroll
        for (int r = 0; r < ROWS; ++r) {
            const bool in = first + r * step < a.n;
            const int k = in ? index_of(ord[r]) : -1;
            place[r] = 0xffffffffu;
            if (k >= 0) {
                const bool counted = isfinite(val[r]) && (!filter || pr[r] > 0.0);
                const int b0 = lay[k], n = lay[k + 1] - b0;
                put(r, b0 + k + (counted ? bin_of(edges + b0, n, val[r]) : n));
            }
        }
    }
    __syncthreads();
    // piece starts: counts over the waves, then a scan over the pieces
    const int per = (keys + MX_OS_SPLIT - 1) / MX_OS_SPLIT, j0 = t * per;
    int sum = 0;
    for (int j = j0; j < j0 + per && j < keys; ++j) {
        int run = 0;
        for (int q = 0; q < MX_OS_SPLIT_WAVES; ++q) {
            const int x = hist[q * kh + j];
            hist[q * kh + j] = (uint16_t)run;
            run += x;
        }
        start[j] = (uint16_t)run;
        sum += run;
    }
    int inc = sum;
    for (int d = 1; d < 64; d <<= 1) {
        const int o = __shfl_up(inc, d);
        if (lane >= d) inc += o;
    }
    if (lane == 63) wtot[w] = inc;
    __syncthreads();
    int run = inc - sum;
    for (int q = 0; q < w; ++q) run += wtot[q];
    for (int j = j0; j < j0 + per && j < keys; ++j) {
        const int x = start[j];
        start[j] = (uint16_t)run;
        run += x;
    }
    if (t == MX_OS_SPLIT - 1) start[keys] = (uint16_t)run;
    __syncthreads();
    // (a row per piece: who reads a bin's offsets reads consecutive words)
    for (int j = t; j <= keys; j += MX_OS_SPLIT) off[(size_t)j * L.stride] = start[j];
#pragma unroll
    for (int r = 0; r < ROWS; ++r)
        if (place[r] != 0xffffffffu) {
            const int key = place[r] >> 16;
            place[r] = (place[r] & 0xffffu) + start[key] + hist[w * kh + key];
            if (VALUES) buf[place[r]] = val[r];
        }
    if (VALUES) {
        __syncthreads();
        double *out = (double *)(ws + L.vals) + (size_t)c * CH;
        const int all = start[keys];
        for (int j = t; j < all; j += MX_OS_SPLIT) out[j] = buf[j];
        double2 *piece = (double2 *)(ws + L.piece) + (size_t)c * L.no * bins;
        auto sum_up = [&](int j, int k, int b0, int n) {
            const int e = start[j + k + 1];
            const double ref = bin_ref(edges + b0, n, j - b0);
            double2 p = make_double2(0.0, 0.0);
#pragma unroll 4
            for (int q = start[j + k]; q < e; ++q) {
                const double d = buf[q] - ref;
                p.x += d;
                p.y += d * d;
            }
            piece[j] = p;
        };
        if (even) {
            for (int j = t; j < L.no * bins; j += MX_OS_SPLIT) sum_up(j, j / bins, j / bins * bins, bins);
        } else {
            for (int j = t; j < keys - L.no; j += MX_OS_SPLIT) {
                int k = 0;
                while (lay[k + 1] <= j) ++k;
                sum_up(j, k, lay[k], lay[k + 1] - lay[k]);
            }
        }
        __syncthreads();
    }
    // probabilities in the same places; each order's run summed by one wave,
    // or by all of them when there are fewer orders than waves
#pragma unroll
    for (int r = 0; r < ROWS; ++r)
        if (place[r] != 0xffffffffu) buf[place[r]] = pr[r];
    __syncthreads();
    const int parts = L.no < MX_OS_SPLIT_WAVES ? MX_OS_SPLIT_WAVES : 1;
    for (int j = w; j < L.no * parts; j += MX_OS_SPLIT_WAVES) {
        const int k = j / parts, b = start[first_key(k)], e = start[first_key(k + 1)];
        double s = 0.0;
#pragma unroll 4
        for (int q = b + (j % parts) * 64 + lane; q < e; q += 64 * parts) s += buf[q];
        for (int o = 32; o > 0; o >>= 1) s += __shfl_xor(s, o);
        if (lane == 0) part[j] = s;
    }
    __syncthreads();
    for (int k = t; k < L.no; k += MX_OS_SPLIT) {
        double s = 0.0;
        for (int j = 0; j < parts; ++j) s += part[k * parts + j];
        psum[(size_t)k * L.chunks + c] = s;
    }
}

// ----------------------------------------------------------------- 3 merge
// Order-preserving integer of a finite double, and back.
__device__ __forceinline__ uint64_t key_of(double x) {
    const uint64_t u = (uint64_t)__double_as_longlong(x);
    return u >> 63 ? ~u : u | 0x8000000000000000ull;
}
__device__ __forceinline__ double of_key(uint64_t k) {
    return __longlong_as_double((long long)(k >> 63 ? k & 0x7fffffffffffffffull : ~k));
}

// The bin has room for one number only, its lower edge.
__device__ __forceinline__ bool bin_single(const double *edges, int b) {
    return b > 0 && key_of(edges[b]) == key_of(edges[b - 1]) + 1;
}

// The pieces of one bin, or of `span` consecutive ones, in all chunks.
struct BinPieces {
    const uint16_t *off;      // the bin's offset in chunk 0
    const double *vals;
    int64_t chunks, end;      // end: from there to the offset after the last bin
    int chunk;
    // f(x, place) for the values of the pieces of chunks group, group + groups,
    // ..., of every piece those at sub, sub + per, ...; place: among the values
    // of these pieces; MX_OS_PIECES pieces at a time, so that loads overlap
    template <typename F>
    __device__ __forceinline__ void each(int64_t group, int64_t groups, int sub, int per, F f) const {
        int64_t run = 0;
        for (int64_t c = group; c < chunks; c += MX_OS_PIECES * groups) {
            int j[MX_OS_PIECES], m[MX_OS_PIECES], first[MX_OS_PIECES];
            int64_t at[MX_OS_PIECES];
            const double *v[MX_OS_PIECES];
#pragma unroll
            for (int u = 0; u < MX_OS_PIECES; ++u) {
                // (no load under a condition: its wait would stand in the
                // branch, before the next load)
                const int64_t x = c + u * groups < chunks ? c + u * groups : c;
                first[u] = off[x];
                m[u] = off[end + x];
            }
#pragma unroll
            for (int u = 0; u < MX_OS_PIECES; ++u) {
                const int64_t x = c + u * groups;
                m[u] = x < chunks ? m[u] - first[u] : 0;
                v[u] = m[u] ? vals + (size_t)x * chunk + first[u] : vals;
                j[u] = sub;
                at[u] = run;
                run += m[u];
            }
            for (;;) {
                bool more = false;
                double x[MX_OS_PIECES];
#pragma unroll
                for (int u = 0; u < MX_OS_PIECES; ++u) {
                    more |= j[u] < m[u];
                    x[u] = v[u][j[u] < m[u] ? j[u] : 0];
                }
                if (!more) break;
#pragma unroll
                for (int u = 0; u < MX_OS_PIECES; ++u) {
                    if (j[u] < m[u]) f(x[u], at[u] + j[u]);
                    j[u] += per;
                }
            }
        }
    }
};

// (key: number of the piece, its bin's among the orders' bins and the piece
// of uncounted photons behind those of each order)
__device__ __forceinline__ BinPieces pieces_of(const OsPlan &L, const unsigned char *ws, int key, int span) {
    return {(const uint16_t *)(ws + L.off) + key * L.stride, (const double *)(ws + L.vals), L.chunks, span * L.stride,
            L.chunk};
}

// Work-items per piece of m values on average: the power of two above it.
__device__ __forceinline__ int items_per_piece(int64_t values, int64_t chunks, int most) {
    int per = 1;
    while (per < most && values > chunks * per) per *= 2;
    return per;
}

// How a workgroup of NT work-items shares the pieces: `per` of them on a piece,
// this one on the pieces of chunks group, group + NT / per, ..., whose values
// follow those of the groups before (`first` of them; `all` in total).
struct Share {
    int per, sub, group, first, all;
};
template <int NT> __device__ __forceinline__ Share share_pieces(const BinPieces &P, int *s_first, int *s_wave) {
    const int t = threadIdx.x, lane = t & 63, w = t >> 6;
    Share H = {1, 0, t, 0, 0};
    // counted by a work-item per piece, and again when pieces are longer
    for (;;) {
        const int groups = NT / H.per;
        int n = 0;
        if (H.sub == 0)
#pragma unroll 8
            for (int64_t c = H.group; c < P.chunks; c += groups) n += (int)P.off[P.end + c] - (int)P.off[c];
        int inc = n;
        for (int d = 1; d < 64; d <<= 1) {
            const int o = __shfl_up(inc, d);
            if (lane >= d) inc += o;
        }
        __syncthreads();
        if (lane == 63) s_wave[w] = inc;
        __syncthreads();
        int before = inc - n;
        H.all = 0;
        for (int q = 0; q < NT / 64; ++q) {
            if (q < w) before += s_wave[q];
            H.all += s_wave[q];
        }
        if (H.sub == 0) s_first[H.group] = before;
        const int per = items_per_piece(H.all, P.chunks, NT);
        if (H.per > 1 || per == 1) break;
        H.per = per;
        H.sub = t & (per - 1);
        H.group = t / per;
    }
    __syncthreads();
    H.first = s_first[H.group];
    return H;
}

// Workgroups 0 .. groups-1 of an order add up a group of chunks: work-item t
// its share of bin t % bins, the shares joined in LDS in a fixed order.  The
// others copy one bin each to one place: those at the ends, where the bounds of a
// single-peaked order lie, and those around the middle, where its median lies
// (3 % of an order's photons is the error of the middle of 270 samples).  A
// bin's pieces lie in as many places as there are chunks: left there, the
// clipping workgroup needed 22 us for every look into a bin at 8e6 photons.
// Copying all bins took 88 us; this kernel takes 26 us.
__global__ __launch_bounds__(MX_OS_MERGE) void mx_os_merge_kernel(OsPlan L, unsigned char *ws) {
    __shared__ double red[3][MX_OS_MERGE];
    __shared__ int s_first[MX_OS_MERGE], s_wave[MX_OS_MERGE / 64];
    __shared__ long long base;
    const int t = threadIdx.x, k = blockIdx.y, all = L.no * L.bins;
    const Bins B = bins_of(L, ws, k);
    const int bins = B.n;
    if ((int)blockIdx.x < L.groups) {
        const int b = t % bins, sub = t / bins, subs = MX_OS_MERGE / bins;
        const int64_t per = (L.chunks + L.groups - 1) / L.groups;
        const int64_t c0 = blockIdx.x * per, c1 = c0 + per < L.chunks ? c0 + per : L.chunks;
        const BinPieces P = pieces_of(L, ws, B.first + k + b, 1);
        const double2 *piece = (const double2 *)(ws + L.piece) + B.first + b;
        double n = 0.0, s1 = 0.0, s2 = 0.0;
#pragma unroll 4
        for (int64_t c = c0 + sub; c < c1; c += subs) {
            const double2 p = piece[(size_t)c * all];
            n += (double)((int)P.off[P.end + c] - (int)P.off[c]);
            s1 += p.x;
            s2 += p.y;
        }
        red[0][t] = n;
        red[1][t] = s1;
        red[2][t] = s2;
        __syncthreads();
        if (sub == 0) {
            for (int q = t + bins; q < subs * bins; q += bins) {
                n += red[0][q];
                s1 += red[1][q];
                s2 += red[2][q];
            }
            ((BinInfo *)(ws + L.grp))[(size_t)B.first * L.groups + (size_t)blockIdx.x * bins + b] = {0, n, s1, s2};
        }
        return;
    }
    const int j = (int)blockIdx.x - L.groups;
    const int b = j < MX_OS_ENDS ? j : (j < 2 * MX_OS_ENDS ? bins - 1 - (j - MX_OS_ENDS)
                                                           : bins / 2 - MX_OS_NEAR / 2 + (j - 2 * MX_OS_ENDS));
    if (j >= 2 * MX_OS_ENDS && (b < MX_OS_ENDS || b >= bins - MX_OS_ENDS)) return;
    if (bin_single((const double *)(ws + L.edges) + B.first, b)) return;
    const BinPieces P = pieces_of(L, ws, B.first + k + b, 1);
    const Share H = share_pieces<MX_OS_MERGE>(P, s_first, s_wave);
    if (t == 0) {
        base = (long long)atomicAdd((unsigned long long *)(ws + L.next), (unsigned long long)H.all);
        ((int64_t *)(ws + L.place))[B.first + b] = base;
    }
    __syncthreads();
    double *out = (double *)(ws + L.copied) + base + H.first;
    P.each(H.group, MX_OS_MERGE / H.per, H.sub, H.per, [&](double x, int64_t at) { out[at] = x; });
}

// ------------------------------------------------------------------ 4 clip
// What the clipping workgroup of one order works on.
struct ClipOrder {
    const OsPlan &L;
    const unsigned char *ws;
    int key, bins;            // piece of bin 0; bins
    const double *edges;      // LDS
    const BinInfo *info;      // LDS
    // f(x) for every value of bin b, by the `nth` work-items tid = 0, 1, ...
    template <typename F> __device__ __forceinline__ void each(int b, int tid, int nth, F f) const {
        const int64_t n = (int64_t)info[b].n;
        if (info[b].at >= 0) {
            const double *x = (const double *)(ws + L.copied) + info[b].at;
            for (int64_t j = tid; j < n; j += 8 * nth) {
                double v[8];
#pragma unroll
                for (int u = 0; u < 8; ++u) v[u] = x[j + u * nth < n ? j + u * nth : j];
#pragma unroll
                for (int u = 0; u < 8; ++u)
                    if (j + u * nth < n) f(v[u]);
            }
        } else {
            const int per = items_per_piece(n, L.chunks, nth);
            pieces_of(L, ws, key + b, 1).each(tid / per, nth / per, tid & (per - 1), per, [&](double x, int64_t) { f(x); });
        }
    }
    __device__ __forceinline__ bool single(int b) const { return bin_single(edges, b); }
    // bin of x, by the wave: the number of edges <= x
    __device__ __forceinline__ int bin_of(double x) const {
        int n = 0;
        for (int b0 = 0; b0 < bins - 1; b0 += 64) {
            const int b = b0 + (int)(threadIdx.x & 63);
            n += __popcll(__ballot(b < bins - 1 && edges[b] <= x));
        }
        return n;
    }
};

// LDS of the clipping kernel: bins, edges, list.
static size_t clip_lds(const OsPlan &L) {
    return (sizeof(double) + sizeof(BinInfo)) * (size_t)(L.no > MX_OS_SKEW ? MX_OS_MAX_BINS : L.bins) +
           sizeof(double) * MX_OS_LIST;
}

#define MX_OS_CW (MX_OS_CLIP / 64)
#define MX_OS_HALF (MX_OS_CLIP / 2)

// n and the sums of deviations and their squares over the kept values of a
// cut bin.
struct CutSums {
    double n, s1, s2;
};
struct ClipShared {
    double cand[2][MX_OS_CAND];
    CutSums part[2][MX_OS_CW];
    double below[2][MX_OS_CW];
    uint64_t kmin, kmax;
    unsigned pre[MX_OS_HIST + 1];
    int iw[MX_OS_CW], n[2], m, first[MX_OS_CLIP];
};

// The kept interval: bins bl .. bh, of which bl and bh count only their values
// in [lo, hi] when `cut` (bl == bh: all of it in c0); all bins fully otherwise.
struct Kept {
    int bl, bh;
    bool cut;
    double lo, hi;
    CutSums c0, c1;
    __device__ __forceinline__ double count(const ClipOrder &O, int b) const {
        if (b < bl || b > bh) return 0.0;
        if (!cut) return O.info[b].n;
        return b == bl ? c0.n : (b == bh ? c1.n : O.info[b].n);
    }
    __device__ __forceinline__ bool partial(int b) const { return cut && (b == bl || b == bh); }
    __device__ __forceinline__ bool has(double x) const { return !cut || (x >= lo && x <= hi); }
};

// The next three are computed by every wave for itself from the bins in LDS,
// which costs less than a barrier.
__device__ __forceinline__ double kept_count(const ClipOrder &O, const Kept &K) {
    double n = 0.0;
    for (int b = threadIdx.x & 63; b < O.bins; b += 64) n += K.count(O, b);
    return wave_add(n);
}

// Bin of rank r (from 0) of the kept values and the rank of its first value.
__device__ __forceinline__ void find_bin(const ClipOrder &O, const Kept &K, int64_t r, int &bin, int64_t &first) {
    const int lane = threadIdx.x & 63, per = (O.bins + 63) / 64, b0 = lane * per;
    double s = 0.0;
    for (int b = b0; b < b0 + per && b < O.bins; ++b) s += K.count(O, b);
    double run = wave_scan(s) - s, at = 0.0;
    int mine = -1;
    for (int b = b0; b < b0 + per && b < O.bins; ++b) {
        const double x = K.count(O, b);
        if ((double)r >= run && (double)r < run + x) {
            mine = b;
            at = run;
        }
        run += x;
    }
    const int src = __ffsll((unsigned long long)__ballot(mine >= 0)) - 1;
    bin = __builtin_amdgcn_readlane(mine, src);
    first = (int64_t)lane_value(at, src);
}

// Mean and standard deviation of the N kept values: sums of deviations from
// their median c or that of the round before (|mean - median| is at most one
// standard deviation, so nothing cancels); the sums of the cut bins are about
// the same c (all: they are the sums of all kept values).
__device__ __forceinline__ void kept_moments(const ClipOrder &O, const Kept &K, double N, double c, bool all,
                                             double &mean, double &sd) {
    double s1 = 0.0, s2 = 0.0;
    for (int b = threadIdx.x & 63; b < O.bins && !all; b += 64) {
        if (b < K.bl || b > K.bh || K.partial(b) || O.info[b].n == 0.0) continue;
        const BinInfo f = O.info[b];
        const double r = bin_ref(O.edges, O.bins, b) - c;
        s1 += f.s1 + f.n * r;
        s2 += f.s2 + r * (2.0 * f.s1 + f.n * r);
    }
    s1 = wave_add(s1);
    s2 = wave_add(s2);
    if (K.cut || all) {
        s1 += K.c0.s1 + K.c1.s1;
        s2 += K.c0.s2 + K.c1.s2;
    }
    const double m = s1 / N;
    mean = c + m;
    const double sq = s2 / N, var = sq - m * m;
    sd = isinf(sq) ? sq : sqrt(var > 0.0 || var != var ? var : 0.0);   // var: >= 0 up to rounding
}

// Values of ranks r and r + 1 among the cnt <= 64 candidates of S.cand[p],
// whose first has rank `base`; by every wave for itself, one per lane.
__device__ __forceinline__ void rank_candidates(const ClipShared &S, int p, int cnt, int64_t base, int64_t r,
                                                double &x0, double &x1) {
    const int lane = threadIdx.x & 63;
    const double x = S.cand[p][lane < cnt ? lane : 0];
    const uint64_t kx = key_of(x);
    const unsigned lo = (unsigned)kx, hi = (unsigned)(kx >> 32);
    int rank = 0;
    for (int j = 0; j < cnt; ++j) {
        const uint64_t kj = (uint64_t)(unsigned)__builtin_amdgcn_readlane((int)lo, j) |
                            ((uint64_t)(unsigned)__builtin_amdgcn_readlane((int)hi, j) << 32);
        rank += (kj < kx || (kj == kx && j < lane)) ? 1 : 0;
    }
    const unsigned long long m0 = __ballot(lane < cnt && base + rank == r);
    const unsigned long long m1 = __ballot(lane < cnt && base + rank == r + 1);
    if (m0) x0 = lane_value(x, __ffsll(m0) - 1);
    if (m1) x1 = lane_value(x, __ffsll(m1) - 1);
}

// The buckets of S.pre scanned: S.pre[j] becomes the number of values in the
// buckets before j, S.pre[MX_OS_HIST] that of all.
__device__ __forceinline__ void scan_buckets(ClipShared &S) {
    constexpr int PER = MX_OS_HIST / MX_OS_CLIP;
    const int t = threadIdx.x;
    unsigned h[PER], sum = 0;
#pragma unroll
    for (int u = 0; u < PER; ++u) {
        h[u] = S.pre[PER * t + u];
        sum += h[u];
    }
    unsigned inc = sum;
    for (int d = 1; d < 64; d <<= 1) {
        const unsigned o = __shfl_up(inc, d);
        if ((t & 63) >= d) inc += o;
    }
    if ((t & 63) == 63) S.iw[t >> 6] = (int)inc;
    __syncthreads();
    unsigned run = inc - sum;
    for (int q = 0; q < (t >> 6); ++q) run += (unsigned)S.iw[q];
#pragma unroll
    for (int u = 0; u < PER; ++u) {
        S.pre[PER * t + u] = run;
        run += h[u];
    }
    if (t == MX_OS_CLIP - 1) S.pre[MX_OS_HIST] = run;
    __syncthreads();
}

// The workgroup's least and greatest integer into S.kmin and S.kmax, which
// hold ~0 and 0 before.
__device__ __forceinline__ void key_range(ClipShared &S, uint64_t mn, uint64_t mx) {
    for (int o = 32; o > 0; o >>= 1) {
        const uint64_t u = __shfl_xor(mn, o), v = __shfl_xor(mx, o);
        mn = u < mn ? u : mn;
        mx = v > mx ? v : mx;
    }
    if ((threadIdx.x & 63) == 0) {
        atomicMin((unsigned long long *)&S.kmin, (unsigned long long)mn);
        atomicMax((unsigned long long *)&S.kmax, (unsigned long long)mx);
    }
    __syncthreads();
}

// Kept values of bin b into the list (when n of them fit) with their least
// and greatest integers.
__device__ __forceinline__ void load_bin(const ClipOrder &O, const Kept &K, int b, bool part, bool fits, ClipShared &S,
                                         double *list) {
    __syncthreads();
    if (threadIdx.x == 0) {
        S.m = 0;
        S.kmin = ~0ull;
        S.kmax = 0;
    }
    __syncthreads();
    uint64_t mn = ~0ull, mx = 0;
    O.each(b, threadIdx.x, MX_OS_CLIP, [&](double x) {
        if (part && !K.has(x)) return;
        const uint64_t k = key_of(x);
        mn = k < mn ? k : mn;
        mx = k > mx ? k : mx;
        if (fits) list[atomicAdd(&S.m, 1)] = x;
    });
    key_range(S, mn, mx);
}

// Shift that maps [0, span] to the MX_OS_HIST buckets.
__device__ __forceinline__ int bucket_shift(uint64_t span) {
    const int bits = span ? 64 - __clzll((long long)span) : 0;
    return bits > 11 ? bits - 11 : 0;
}

// Bucket of rank r, by the wave: the last j with S.pre[j] <= r.
__device__ __forceinline__ int bucket_of(const ClipShared &S, unsigned r) {
    constexpr int PER = MX_OS_HIST / 64;      // 32: the second look takes half the lanes
    const int lane = threadIdx.x & 63;
    const int g = __popcll(__ballot(S.pre[lane * PER] <= r)) - 1;
    return g * PER + __popcll(__ballot(lane < PER && S.pre[g * PER + (lane & (PER - 1))] <= r)) - 1;
}

#define MX_OS_ALL (-2)

// State of the list between medians: the uncut bin that the list holds (-1:
// none; MX_OS_ALL: every value of the order, n of them), whether S.pre holds
// its buckets, its least and greatest integers, the candidate buffer next to
// use; buckets of a bin are equal steps of 1 / inv from x0.
struct Held {
    int bin;
    bool buckets;
    int p;
    int64_t n;
    uint64_t kmin, kmax;
    double x0, inv;
    __device__ __forceinline__ void steps(double a, double b, int n) {
        x0 = a;
        inv = b > a && !isinf(b - a) ? n / (b - a) : 0.0;
        if (isinf(inv)) inv = 0.0;
    }
    __device__ __forceinline__ int step(double x, int n) const {
        const int j = (int)((x - x0) * inv);
        return j < 0 ? 0 : (j < n ? j : n - 1);
    }
    // of a whole order: equal steps within each bin, so that an order of a
    // narrow line and values far from it still fills them evenly
    __device__ __forceinline__ int bucket(const ClipOrder &O, double x) {
        if (bin != MX_OS_ALL) return step(x, MX_OS_HIST);
        const int b = ::bin_of(O.edges, O.bins, x), per = MX_OS_HIST / O.bins;
        if (b == 0 || b == O.bins - 1) return b * per;
        steps(O.edges[b - 1], O.edges[b], per);
        return b * per + step(x, per);
    }
};

// The kept values of bin b of ranks r and r + 1 (from 0, r + 1 only when
// `two`), exactly.  An uncut bin that fits the list is loaded and counted into
// buckets once; every further median in it takes one pass over the list, for
// the values of one or two buckets, and one barrier.  Otherwise (a cut bin, one
// larger than the list, or one with a crowded bucket) buckets of the values'
// order-preserving integers narrow them down until few are left.
__device__ __forceinline__ void select_in_bin(const ClipOrder &O, const Kept &K, int b, int64_t r, bool two,
                                              ClipShared &S, double *list, Held &H, double &x0, double &x1) {
    const int t = threadIdx.x;
    const bool all = b == MX_OS_ALL;
    if (!all && O.single(b)) {
        x0 = x1 = O.edges[b - 1];
        return;
    }
    const bool part = !all && K.partial(b);
    const int64_t n = all ? H.n : (int64_t)K.count(O, b);
    const bool fits = n <= MX_OS_LIST;
    if (H.bin != b || part) {
        load_bin(O, K, b, part, fits, S, list);
        H.bin = fits && !part ? b : -1;
        H.buckets = false;
        H.kmin = S.kmin;
        H.kmax = S.kmax;
        H.steps(of_key(H.kmin), of_key(H.kmax), MX_OS_HIST);
    }
    uint64_t klo = H.kmin, khi = H.kmax;
    int64_t cnt = n, below = 0;     // values in [klo, khi], and before it
    // mode 0: count into buckets of integers; 1: collect the values of
    // [klo, khi]; 2: the least integer above khi; 3: count into the buckets
    // that are kept; 4: they are there
    int mode = n <= MX_OS_CAND ? 1 : (H.buckets ? 4 : (H.bin == b ? 3 : 0));
    for (;;) {
        const int shift = bucket_shift(khi - klo);
        if (mode != 4) {
            __syncthreads();
            if (mode == 0 || mode == 3) {
                for (int j = t; j < MX_OS_HIST; j += MX_OS_CLIP) S.pre[j] = 0;
                if (t < 2) S.n[t] = 0;
            } else if (t == 0) {
                S.m = 0;
                S.kmin = ~0ull;
            }
            __syncthreads();
            uint64_t mn = ~0ull;
            auto f = [&](double x) {
                const uint64_t k = key_of(x);
                if (mode == 2) {
                    if (k > khi && k < mn) mn = k;
                } else if (mode == 3) {
                    atomicAdd(&S.pre[H.bucket(O, x)], 1u);
                } else if (k >= klo && k <= khi) {
                    if (mode == 0) atomicAdd(&S.pre[(k - klo) >> shift], 1u);
                    else S.cand[0][atomicAdd(&S.m, 1)] = x;
                }
            };
            if (fits) {
                for (int j = t; j < (int)n; j += MX_OS_CLIP) f(list[j]);
            } else {
                O.each(b, t, MX_OS_CLIP, [&](double x) { if (!part || K.has(x)) f(x); });
            }
            if (mode == 2) {
                for (int o = 32; o > 0; o >>= 1) {
                    const uint64_t u = __shfl_xor(mn, o);
                    mn = u < mn ? u : mn;
                }
                if ((t & 63) == 0) atomicMin((unsigned long long *)&S.kmin, (unsigned long long)mn);
            }
            __syncthreads();
            if (mode == 2) {
                x1 = of_key(S.kmin);
                break;
            }
            if (mode == 1) {
                rank_candidates(S, 0, (int)cnt, below, r, x0, x1);
                if (!two || r + 1 < below + cnt) break;
                mode = 2;
                continue;
            }
            scan_buckets(S);
        }
        const int64_t q = r - below;
        const int j0 = bucket_of(S, (unsigned)q);
        if (mode >= 3) {
            H.buckets = true;
            const int j1 = two ? bucket_of(S, (unsigned)q + 1) : j0;
            const int c = (int)(S.pre[j0 + 1] - S.pre[j0]) + (j1 != j0 ? (int)(S.pre[j1 + 1] - S.pre[j1]) : 0);
            if (c <= MX_OS_CAND) {
                const int p = H.p;
                double lo = -__builtin_inf(), hi = __builtin_inf();
                if (all) {
                    const int per = MX_OS_HIST / O.bins, b0 = j0 / per, b1 = j1 / per;
                    if (b0 > 0) lo = O.edges[b0 - 1];
                    if (b1 < O.bins - 1) hi = O.edges[b1];
                }
                for (int j = t; j < (int)n; j += MX_OS_CLIP) {
                    const double x = list[j];
                    if (!(x >= lo && x <= hi)) continue;
                    const int u = H.bucket(O, x);
                    if (u == j0 || u == j1) S.cand[p][atomicAdd(&S.n[p], 1)] = x;
                }
                __syncthreads();
                // the other buffer's last readers passed this barrier
                if (t == 0) S.n[p ^ 1] = 0;
                H.p = p ^ 1;
                rank_candidates(S, p, c, S.pre[j0], r, x0, x1);
                break;
            }
            H.buckets = false;      // the narrowing uses S.pre for its own
            mode = 0;
            continue;
        }
        cnt = (int64_t)(S.pre[j0 + 1] - S.pre[j0]);
        below += S.pre[j0];
        klo += (uint64_t)j0 << shift;
        if (khi - klo > (1ull << shift) - 1) khi = klo + ((1ull << shift) - 1);
        mode = cnt > MX_OS_CAND ? 0 : 1;
        if (klo == khi) {
            x0 = x1 = of_key(klo);
            if (!two || r + 1 < below + cnt) break;
            mode = 2;
        }
    }
}

// Median of the N > 0 kept values (below: the values under them, when the list
// holds all).
__device__ __forceinline__ double kept_median(const ClipOrder &O, const Kept &K, int64_t N, int64_t below,
                                              ClipShared &S, double *list, Held &H) {
    const int64_t r = (N - 1) / 2;
    const bool two = !(N & 1);
    double lower = 0.0;
    // the upper middle value may be the least of a later bin
    for (int u = 0;; ++u) {
        int b = MX_OS_ALL;
        int64_t first = -below;
        if (H.bin != MX_OS_ALL) find_bin(O, K, r + u, b, first);
        const bool both = two && u == 0 && (b == MX_OS_ALL || r + 1 < first + (int64_t)K.count(O, b));
        double x0 = 0.0, x1 = 0.0;
        select_in_bin(O, K, b, r + u - first, both, S, list, H, x0, x1);
        __syncthreads();
        if (!two) return x0;
        if (both) return (x0 + x1) / 2;
        if (u == 1) return (lower + x0) / 2;
        lower = x0;
    }
}

// Count, sum and squares about c of the kept values of the cut bins: the first
// half of the waves takes bin bl, the second bin bh (none when they are the
// same).  With every value in the list (nlist of them, else -1): of all kept values,
// with the number below lo.
__device__ __forceinline__ void cut_bins(const ClipOrder &O, Kept &K, double c, ClipShared &S, int p,
                                         const double *list, int nlist, double &below) {
    const int t = threadIdx.x, half = t / MX_OS_HALF, th = t % MX_OS_HALF;
    const int b = half ? K.bh : K.bl;
    CutSums a = {0.0, 0.0, 0.0};
    auto add = [&](double x) {
        if (!K.has(x)) return;
        const double d = x - c;
        a.n += 1.0;
        a.s1 += d;
        a.s2 += d * d;
    };
    below = 0.0;
    if (nlist >= 0) {
        for (int j = t; j < nlist; j += MX_OS_CLIP) {
            add(list[j]);
            below += list[j] < K.lo ? 1.0 : 0.0;
        }
        below = wave_add(below);
    } else if (half && K.bl == K.bh) {
    } else if (O.single(b)) {
        if (th == 0 && O.info[b].n > 0.0 && K.has(O.edges[b - 1])) {
            const double d = O.edges[b - 1] - c;
            a.n = O.info[b].n;
            a.s1 = a.n * d;
            a.s2 = a.n * (d * d);
        }
    } else {
        O.each(b, th, MX_OS_HALF, add);
    }
    a.n = wave_add(a.n);
    a.s1 = wave_add(a.s1);
    a.s2 = wave_add(a.s2);
    if ((t & 63) == 0) {
        S.part[p][t >> 6] = a;
        S.below[p][t >> 6] = below;
    }
    __syncthreads();
    below = 0.0;
    for (int q = 0; q < MX_OS_CW; ++q) below += S.below[p][q];
    K.c0 = K.c1 = {0.0, 0.0, 0.0};
    for (int q = 0; q < MX_OS_CW; ++q) {
        CutSums &d = q < MX_OS_CW / 2 ? K.c0 : K.c1;
        d.n += S.part[p][q].n;
        d.s1 += S.part[p][q].s1;
        d.s2 += S.part[p][q].s2;
    }
}

// One order: probability sum and count, then the clipping rounds.  Bound by
// the latency of its dependent steps, so everything that can be is done by
// every wave for itself, and a round has two barriers: one after the sums over
// the two cut bins, one after the candidates of the median (94 us for 8e6
// photons in 15 orders; with a workgroup-wide reduction for each sum and a
// selection from the start for each median 179 us).
template <bool VALUES>
__global__ __launch_bounds__(MX_OS_CLIP) void mx_os_clip_kernel(MxOrderStats a, OsPlan L, unsigned char *ws) {
    extern __shared__ __align__(16) unsigned char sm[];
    __shared__ ClipShared S;
    const int k = blockIdx.x, t = threadIdx.x, w = t >> 6;
    const Bins B = VALUES ? bins_of(L, ws, k) : Bins{0, 0};
    const int bins = B.n, key = B.first + k;
    const BinPieces rest = pieces_of(L, ws, key + bins, 1);
    // probability sum; photons outside the bins
    const double *psum = (const double *)(ws + L.psum) + (size_t)k * L.chunks;
    CutSums tot = {0.0, 0.0, 0.0};
    // (a list of 3e8 photons has 95 chunks for each work-item, one latency each
    // unless the loads overlap)
#pragma unroll 8
    for (int64_t c = t; c < L.chunks; c += MX_OS_CLIP) {
        tot.s1 += psum[c];
        tot.n += (double)((int)rest.off[rest.end + c] - (int)rest.off[c]);
    }
    tot.n = wave_add(tot.n);
    tot.s1 = wave_add(tot.s1);
    if ((t & 63) == 0) S.part[1][w] = tot;
    BinInfo *info = (BinInfo *)sm;
    double *edges = (double *)(info + bins), *list = edges + bins;
    if (VALUES) {
        for (int b = t; b < bins; b += MX_OS_CLIP) {
            BinInfo f = {((const int64_t *)(ws + L.place))[B.first + b], 0.0, 0.0, 0.0};
#pragma unroll 4
            for (int g = 0; g < L.groups; ++g) {
                const BinInfo q = ((const BinInfo *)(ws + L.grp))[(size_t)B.first * L.groups + (size_t)g * bins + b];
                f.n += q.n;
                f.s1 += q.s1;
                f.s2 += q.s2;
            }
            info[b] = f;
            edges[b] = ((const double *)(ws + L.edges))[B.first + b];
        }
        if (t < 2) S.n[t] = 0;
    }
    __syncthreads();
    double ps = 0.0, other = 0.0;
    for (int q = 0; q < MX_OS_CW; ++q) {
        ps += S.part[1][q].s1;
        other += S.part[1][q].n;
    }
    if (!VALUES) {
        if (t == 0) {
            a.prob_sum[k] = ps;
            a.count[k] = (int64_t)other;
        }
        return;
    }
    const ClipOrder O = {L, ws, key, bins, edges, info};
    Kept K = {0, bins - 1, false, 0.0, 0.0, {0.0, 0.0, 0.0}, {0.0, 0.0, 0.0}};
    double N = kept_count(O, K);
    if (t == 0) {
        a.prob_sum[k] = ps;
        a.count[k] = (int64_t)(N + ((a.flags & MX_OS_FILTER) ? 0.0 : other));
    }
    const double nan = __builtin_nan("");
    double mean = nan, cen = nan, sd = nan;
    if (N > 0.0) {
        Held H = {-1, false, 0, 0, 0, 0, 0.0, 0.0};
        int nlist = -1;
        double c = 0.0, below = 0.0;
        if (N <= (double)MX_OS_LIST) {
            // the whole order into the list, in the same places every run
            const BinPieces P = pieces_of(L, ws, key, bins);
            const Share R = share_pieces<MX_OS_CLIP>(P, S.first, S.iw);
            if (t == 0) {
                S.kmin = ~0ull;
                S.kmax = 0;
            }
            __syncthreads();
            uint64_t mn = ~0ull, mx = 0;
            P.each(R.group, MX_OS_CLIP / R.per, R.sub, R.per, [&](double x, int64_t at) {
                const uint64_t q = key_of(x);
                mn = q < mn ? q : mn;
                mx = q > mx ? q : mx;
                list[R.first + at] = x;
            });
            key_range(S, mn, mx);
            nlist = (int)N;
            H.bin = MX_OS_ALL;
            H.n = nlist;
            H.kmin = S.kmin;
            H.kmax = S.kmax;
        }
        if (isinf(edges[0])) {
            // no photon of the order in the sample: one bin holds them all,
            // and its values are summed one by one, about their mean
            K.cut = true;
            K.bh = 0;
            K.lo = -__builtin_inf();
            K.hi = __builtin_inf();
            c = info[0].s1 / info[0].n;
        }
        int p = 0;
        for (int it = 0;; ++it) {
            Kept Q = K;
            bool any = true;
            if (it > 0) {
                double lo = cen - sd * a.sigma, hi = cen + sd * a.sigma;
                if (K.cut) {
                    lo = K.lo > lo ? K.lo : lo;
                    hi = K.hi < hi ? K.hi : hi;
                }
                any = lo <= hi;      // false for NaN bounds, which keep nothing
                Q.cut = true;
                Q.lo = lo;
                Q.hi = hi;
                if (nlist < 0) {
                    Q.bl = O.bin_of(lo);
                    Q.bh = O.bin_of(hi);
                }
            }
            double kept = 0.0;
            if (any) {
                if (Q.cut) cut_bins(O, Q, c, S, p, list, nlist, below);
                p ^= 1;
                kept = nlist >= 0 && Q.cut ? Q.c0.n + Q.c1.n : kept_count(O, Q);
            }
            if (it > 0 && kept == N) break;
            N = kept;
            if (N == 0.0) {
                mean = cen = sd = nan;
                break;
            }
            K = Q;
            cen = kept_median(O, K, (int64_t)N, (int64_t)below, S, list, H);
            // few values: summed again about their own median, as they may be
            // a pair one standard deviation from it, which stays or goes with
            // the last bit (more bits are lost in sums about another point)
            const bool few = N <= (double)MX_OS_CAND && (K.cut || nlist >= 0);
            if (few) {
                double unused;
                cut_bins(O, K, cen, S, p, list, nlist, unused);
                p ^= 1;
            }
            kept_moments(O, K, N, few || !K.cut ? cen : c, nlist >= 0 && (K.cut || few), mean, sd);
            c = cen;
            if (it == a.maxiters) break;
        }
    }
    if (t == 0) {
        a.mean[k] = mean;
        a.median[k] = cen;
        a.std[k] = sd;
        a.n_kept[k] = (int64_t)N;
    }
}

extern "C" int64_t mx_order_stats_workspace(int64_t n, int32_t n_orders, int32_t with_values) {
    if (n < 0 || n_orders < 1 || n_orders > MX_MAX_ORDERS) return -1;
    OsPlan L;
    os_plan(n, n_orders, with_values != 0, L);
    return (int64_t)L.total;
}

extern "C" int mx_order_stats(const MxOrderStats *a, void *stream) {
    if (!a) { mx_set_error("order stats: arguments NULL"); return 1; }
    if (a->n < 0 || a->n > 0x7fffffffLL) { mx_set_error("order stats: photon count outside [0, 2^31)"); return 1; }
    if (a->n_orders < 1 || a->n_orders > MX_MAX_ORDERS) { mx_set_error("order stats: n_orders outside [1, 64]"); return 1; }
    if (!a->orders || !a->prob_sum || !a->count || (a->n > 0 && (!a->order || !a->prob))) {
        mx_set_error("order stats: a required pointer is NULL");
        return 1;
    }
    const bool values = a->value != nullptr;
    if (values && (!a->mean || !a->median || !a->std || !a->n_kept || a->maxiters < 0)) {
        mx_set_error("order stats: statistics outputs NULL or maxiters negative");
        return 1;
    }
    if ((a->flags & MX_OS_FILTER) && !values) {
        mx_set_error("order stats: the finite-value filter needs a value column");
        return 1;
    }
    OsPlan L;
    os_plan(a->n, a->n_orders, values, L);
    if (!a->workspace || a->workspace_bytes < (int64_t)L.total) {
        mx_set_error("order stats: workspace missing or smaller than mx_order_stats_workspace()");
        return 1;
    }
    hipStream_t st = (hipStream_t)stream;
    unsigned char *ws = (unsigned char *)a->workspace;
    const dim3 chunks((unsigned)L.chunks), split(MX_OS_SPLIT);
    const size_t lds = split_lds(L);
    if (values) {
        hipLaunchKernelGGL(mx_os_sample_kernel, dim3((unsigned)L.no), dim3(1024), 0, st, *a, L, ws);
        if (L.chunks > 0 && L.rows == MX_OS_ROWS)
            hipLaunchKernelGGL((mx_os_split_kernel<MX_OS_ROWS, true>), chunks, split, lds, st, *a, L, ws);
        else if (L.chunks > 0)
            hipLaunchKernelGGL((mx_os_split_kernel<MX_OS_ROWS_FEW, true>), chunks, split, lds, st, *a, L, ws);
        hipLaunchKernelGGL(mx_os_merge_kernel, dim3((unsigned)(L.groups + 2 * MX_OS_ENDS + MX_OS_NEAR), (unsigned)L.no),
                           dim3(MX_OS_MERGE), 0, st, L, ws);
        hipLaunchKernelGGL(mx_os_clip_kernel<true>, dim3((unsigned)L.no), dim3(MX_OS_CLIP), clip_lds(L), st, *a, L,
                           ws);
    } else {
        if (L.chunks > 0 && L.rows == MX_OS_ROWS)
            hipLaunchKernelGGL((mx_os_split_kernel<MX_OS_ROWS, false>), chunks, split, lds, st, *a, L, ws);
        else if (L.chunks > 0)
            hipLaunchKernelGGL((mx_os_split_kernel<MX_OS_ROWS_FEW, false>), chunks, split, lds, st, *a, L, ws);
        hipLaunchKernelGGL(mx_os_clip_kernel<false>, dim3((unsigned)L.no), dim3(MX_OS_CLIP), 0, st, *a, L, ws);
    }
    hipError_t err = hipGetLastError();
    if (err != hipSuccess) {
        char buf[256];
        snprintf(buf, sizeof(buf), "order stats: launch failed: %s", hipGetErrorString(err));
        mx_set_error(buf);
        return 2;
    }
    return 0;
}

// ------------------------------------------------ allocation-free variant
// mx_order_stats_static: mx_order_stats with its workspace in `scratch`, a
// file-scope device array of MX_OS_STATIC_BYTES, for callers that cannot
// allocate (tight serving loops, harnesses that forbid hipMalloc).  Every GPU
// the library runs on holds its own copy until the process ends.  Host code
// never passes the array's name to a kernel or a copy (in host code it is a
// host-side stand-in): the device address of this GPU's copy comes from
// hipGetSymbolAddress on the entry point's first call on that GPU and is
// kept per device.  Calls on one GPU share the array, so calls that overlap
// on one GPU race; it keeps the last call's contents, and every word a call
// reads it has written first (edges, offsets, sums, values), so nothing needs
// clearing.
static __device__ __align__(256) unsigned char scratch[MX_OS_STATIC_BYTES];

#define MX_OS_MAX_DEVICES 64
static std::mutex g_scratch_mutex;
static void *g_scratch_dev[MX_OS_MAX_DEVICES];

static int scratch_address(void **out) {
    int dev = -1;
    if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= MX_OS_MAX_DEVICES) {
        mx_set_error("order stats (static workspace): no current device or device index too large");
        return 2;
    }
    std::lock_guard<std::mutex> lock(g_scratch_mutex);
    if (!g_scratch_dev[dev]) {
        void *p = nullptr;
        const hipError_t e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
        if (e != hipSuccess || !p) {
            char buf[256];
            snprintf(buf, sizeof(buf), "order stats (static workspace): hipGetSymbolAddress failed: %s",
                     hipGetErrorString(e));
            mx_set_error(buf);
            return 2;
        }
        g_scratch_dev[dev] = p;
    }
    *out = g_scratch_dev[dev];
    return 0;
}

extern "C" int mx_order_stats_static(const MxOrderStats *a, void *stream) {
    if (!a) { mx_set_error("order stats: arguments NULL"); return 1; }
    if (a->n < 0 || a->n > 0x7fffffffLL) { mx_set_error("order stats: photon count outside [0, 2^31)"); return 1; }
    if (a->n_orders < 1 || a->n_orders > MX_MAX_ORDERS) { mx_set_error("order stats: n_orders outside [1, 64]"); return 1; }
    OsPlan L;
    os_plan(a->n, a->n_orders, a->value != nullptr, L);
    // sums alone: the workspace grows with the number of orders, so that many
    // orders of a list of several 1e8 photons take a few calls, one after
    // another on the stream
    int per = a->n_orders;
    while (!a->value && per > 1 && (int64_t)L.total > (int64_t)MX_OS_STATIC_BYTES) {
        per = (per + 1) / 2;
        os_plan(a->n, per, false, L);
    }
    if ((int64_t)L.total > (int64_t)MX_OS_STATIC_BYTES) {
        char buf[256];
        snprintf(buf, sizeof(buf),
                 "order stats (static workspace): %lld photons need %lld bytes of workspace, the static "
                 "workspace holds %lld (use mx_order_stats with a workspace of your own)",
                 (long long)a->n, (long long)L.total, (long long)MX_OS_STATIC_BYTES);
        mx_set_error(buf);
        return 1;
    }
    void *ws = nullptr;
    if (scratch_address(&ws)) return 2;
    MxOrderStats b = *a;
    b.workspace = ws;
    b.workspace_bytes = (int64_t)MX_OS_STATIC_BYTES;
    if (per == a->n_orders || !a->orders || !a->prob_sum || !a->count) return mx_order_stats(&b, stream);
    for (int k = 0; k < a->n_orders; k += per) {
        b.n_orders = a->n_orders - k < per ? a->n_orders - k : per;
        b.orders = a->orders + k;
        b.prob_sum = a->prob_sum + k;
        b.count = a->count + k;
        const int rc = mx_order_stats(&b, stream);
        if (rc) return rc;
    }
    return 0;
}
