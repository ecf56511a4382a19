// call.hip -- reads to calls in one launch: the batched form's site matrix,
// sort, likelihood and posterior for 64 consecutive sites per wave, with no
// record ever written to memory.
//
// A tile is 64 consecutive sites; lane i of a wave owns site i.  The wave
//  A. walks the reads that cover the tile: each lane takes its byte of the
//     read (64 consecutive bytes, one load), makes the observation record
//     and appends it to its own column of an LDS buffer [slot][lane].  Reads
//     that share their strand and anchor (the start on '+', the last base on
//     '-') are exactly the ones whose records share a cycle and strand at
//     every site, so the dependency count t of a record (how many earlier
//     records of its base, in sorted order, repeat its cycle and strand) is
//     settled here, for the few reads that have such a partner, and kept in
//     the record's low byte (a pile of reads on one anchor instead leaves its
//     number there, and is counted in sorted order in B);
//  B. loads its records into registers and sorts them with a Batcher
//     network over registers: two VALU instructions per compare-exchange for
//     64 sites, no lane exchange.  A walk over the sorted registers gives g
//     (first occurrences of the base so far), the adjusted quality (a table
//     in LDS) and the score row, parked in LDS as 16 bits;
//  C. adds the score rows with five lanes per site, two genotypes each, in
//     record order (kernel/likelihood_kernel.cu:168-256), eight rows in
//     flight: an 80-byte row is one line read by five neighbouring lanes;
//  D. calls its site from registers (posterior.h) and stores the site's
//     counters and results.
// Against a build that writes records to memory and sorts them one site per
// lane group this needs no 1 KB row per site, and a padding slot costs a lane
// of one instruction instead of a lane of every network step: on one 24.8 Mb
// chromosome (30x, 150 bp, 7.4e8 records) the launches from reads to calls
// take 5.3 ms a pass, where the site matrix, the depth classes and the fused
// sort + likelihood took 9.4 ms.
//
// What bounds it is C's rows out of the XCDs' L2: the table (2-3 MB) is far
// beyond a CU's 32 KB L1, so every record asks the L2 for one 128-byte line.
// Such random lines come at 263e9 a second and no faster however many are in
// flight (measured alone, 8 to 32 waves a CU); these launches reach 170e9
// while they also sort, about two thirds of it.  Other waves' A, B and D
// hide under it, so waves in flight matter more than instructions there, and
// LDS is what limits them: 8 to 12 waves a CU.
//
// Tiles are classed by the largest number of unique-hit reads over one of
// their sites (the bound on a site's records), one launch per class with
// registers and LDS for that many records: 16, 32, 40, 64, 128.  A third of
// a 30x genome's tiles lie at 33 to 40, and there 12 waves a CU instead of
// the 64-record class's 8 took the launches from 6.1 to 5.3 ms.  Tiles beyond
// 128 records a site, 512 reads or max_unique go through k_site_build and
// k_fused<256>, and spans that lie mostly beyond the 64-record class do not
// come here at all (add_tile_gain).
#include <hip/hip_runtime.h>

#include <utility>

#include "gsnp_common.h"
#include "kernels.h"
#include "posterior.h"

namespace gsnp {

namespace {

constexpr uint32_t kTile = 64;
constexpr uint32_t kPriorBytes = 640u;   // ten log10 priors of the eight reference codes
// Spans of up to this many tiles use the 64- and 128-record classes only: a
// tile alone takes 30 to 40 us, so a launch does however few its tiles, and
// five classes in a row leave most of the device idle.  24 contigs of 0.12 to
// 2.4 Mb (2,000 to 37,000 tiles) took 11.4 ms with the line at 4,096 tiles,
// 10.8 at 20,000 and 10.7 at 60,000, where the 32- and 40-record classes
// begin to win on uniform depth.
constexpr uint32_t kFewTiles = 20000;
// Record of an empty slot: above every record (bits 24:0), and its base,
// quality field, cycle and t are 0, so that it walks to score row 0 (ten
// +0.0) like any record.
constexpr uint32_t kNoRec = 1u << 25;
constexpr uint32_t kDeepClass = kTileClasses;  // after the classes of k_call_tile

// Batcher's odd-even merge exchange for any N, as a list of pairs.
template <int N>
struct Network {
    int n = 0;
    uint8_t lo[16 * N] = {}, hi[16 * N] = {};
    constexpr Network()
    {
        for (int p = 1; p < N; p *= 2)
            for (int k = p; k >= 1; k /= 2)
                for (int j = k % p; j <= N - 1 - k; j += 2 * k)
                    for (int i = 0; i < k && i < N - j - k; i++)
                        if ((i + j) / (2 * p) == (i + j + k) / (2 * p)) {
                            lo[n] = (uint8_t)(i + j);
                            hi[n] = (uint8_t)(i + j + k);
                            n++;
                        }
    }
};
template <int N>
constexpr Network<N> kNetwork{};

template <int I, int J, int D>
__device__ __forceinline__ void exchange(uint32_t (&v)[D])
{
    const uint32_t a = v[I], b = v[J];
    v[I] = a < b ? a : b;
    v[J] = a < b ? b : a;
}

template <int N, int B, int D, size_t... I>
__device__ __forceinline__ void exchange_block(uint32_t (&v)[D], std::index_sequence<I...>)
{
    (exchange<kNetwork<N>.lo[B + I], kNetwork<N>.hi[B + I]>(v), ...);
}

// v[0, N) ascending
template <int N, int B = 0, int D>
__device__ __forceinline__ void sort_regs(uint32_t (&v)[D])
{
    constexpr int left = kNetwork<N>.n - B, m = left < 64 ? left : 64;
    exchange_block<N, B>(v, std::make_index_sequence<m>());
    if constexpr (left > m) sort_regs<N, B + m>(v);
}

__device__ __forceinline__ uint32_t uniform(uint32_t v) { return (uint32_t)__builtin_amdgcn_readfirstlane((int)v); }
__device__ __forceinline__ uint64_t uniform(uint64_t v)
{
    return ((uint64_t)uniform((uint32_t)(v >> 32)) << 32) | uniform((uint32_t)v);
}
__device__ __forceinline__ uint32_t lane_of(uint32_t v, uint32_t l)
{
    return (uint32_t)__builtin_amdgcn_readlane((int)v, (int)l);
}

// One step of a wave scan over lanes, in VALU lane moves: `from` lanes down
// within a row of 16, or (0x142, 0x143) the last lane of the rows before into
// the rows of the mask; lanes without a source take `none`.
template <int CTRL, int ROWS>
__device__ __forceinline__ int scan_move(int v, int none)
{
    return __builtin_amdgcn_update_dpp(none, v, CTRL, ROWS, 0xF, false);
}

// inclusive prefix sum over the lanes
__device__ __forceinline__ int wave_prefix(int v)
{
    v += scan_move<0x111, 0xF>(v, 0);  // row_shr 1, 2, 4, 8
    v += scan_move<0x112, 0xF>(v, 0);
    v += scan_move<0x114, 0xF>(v, 0);
    v += scan_move<0x118, 0xF>(v, 0);
    v += scan_move<0x142, 0xA>(v, 0);  // row_bcast 15 into rows 1 and 3
    v += scan_move<0x143, 0xC>(v, 0);  // row_bcast 31 into rows 2 and 3
    return v;
}

// largest value (at least 0) over the wave, in every lane's scalar copy
__device__ __forceinline__ uint32_t wave_max(uint32_t x)
{
    int v = (int)x;
    v = max(v, scan_move<0x111, 0xF>(v, 0));
    v = max(v, scan_move<0x112, 0xF>(v, 0));
    v = max(v, scan_move<0x114, 0xF>(v, 0));
    v = max(v, scan_move<0x118, 0xF>(v, 0));
    v = max(v, scan_move<0x142, 0xA>(v, 0));
    v = max(v, scan_move<0x143, 0xC>(v, 0));
    return lane_of((uint32_t)v, 63);
}

// The whole wave looks at one site: the unique-hit records of absolute
// position p among reads [b, e) starting at or before `last`, in read order
// and up to 255, summed into q_sum (returned in every lane) and, with row
// set, written to it.
__device__ int4 wave_site_records(const ReadView& r, uint64_t b, uint64_t e, int64_t p, int64_t last, uint32_t* row)
{
    const uint32_t lane = __lane_id();
    const uint64_t below = lane == 0 ? 0ull : (~0ull >> (64 - lane));
    uint32_t have = 0;
    int s0 = 0, s1 = 0, s2 = 0, s3 = 0;
    for (uint64_t c = b; c < e; c += 64) {
        const uint64_t i = c + lane;
        uint32_t byte = 0, m = 0;
        int64_t coord = 0;
        if (i < e) {
            m = r.meta[i];
            const int64_t st = r.pos[i];
            coord = p - st;
            if (rm_hit(m) == 1 && st <= last && coord >= 0 && coord < (int64_t)rm_len(m))
                byte = r.seq[i * (uint64_t)r.pitch + (uint64_t)coord];
        }
        const uint64_t obs = __ballot(byte != 0);
        const uint32_t at = have + (uint32_t)__popcll(obs & below);
        if (byte != 0 && at < kMaxDepUni) {
            const uint32_t o = pb_base(byte), q = pb_q(byte);
            s0 += o == 0 ? (int)q : 0;
            s1 += o == 1 ? (int)q : 0;
            s2 += o == 2 ? (int)q : 0;
            s3 += o == 3 ? (int)q : 0;
            if (row) {
                const uint32_t k = (uint32_t)coord, rev = rm_strand(m);
                row[at] = rec_encode(rev ? rm_len(m) - 1u - k : k, rev, o, q, 1);
            }
        }
        have += (uint32_t)__popcll(obs);
    }
    for (int off = 32; off > 0; off >>= 1) {
        s0 += __shfl_xor(s0, off);
        s1 += __shfl_xor(s1, off);
        s2 += __shfl_xor(s2, off);
        s3 += __shfl_xor(s3, off);
    }
    return make_int4(s0, s1, s2, s3);
}

// bytes of a site's parked rows (16 bits a slot), whose place its ten sums
// take: an odd number of 16-byte units
template <int D>
constexpr uint32_t park_stride()
{
    return D <= 32 ? 80u : ((2u * D + 15u) / 16u | 1u) * 16u;
}

constexpr uint32_t kCountBytes = 4u * kTile * 4u;  // packed counters per base and site
constexpr uint32_t kAnchorWords = 1280u;           // one word per (anchor, strand)

// Chunks of 64 reads a tile of the class may have: the deep class keeps its
// reads' positions and metadata in LDS, the others in two registers each.
template <int D>
constexpr uint32_t tile_chunks()
{
    return D <= 64 ? kShallowReads / 64u : kMaxTileReads / 64u;
}

// the list of reads that share an anchor: a word for any read of the tile
template <int D>
constexpr uint32_t list_bytes()
{
    return 4u * 64u * tile_chunks<D>();
}

// Groups of more than kBigGroup reads on one anchor (amplicons, duplicates)
// are counted after the sort, with a counter per group, base and site beyond
// the parked rows, as far as those hold; smaller ones read by read, which is
// quadratic in the group: a pile of 75 reads took a tile from 40 to 300 us.
constexpr uint32_t kBigGroup = 6;

// LDS of a wave: the record columns, which the parked rows replace once the
// records are in registers, the reads of the deep class, the list and the counters
template <int D>
constexpr uint32_t wave_lds()
{
    constexpr uint32_t rec = D * kTile * 4u, park = kTile * park_stride<D>();
    constexpr uint32_t both = rec > park ? rec : park;
    static_assert(both >= kAnchorWords * 4u, "the anchor table lies in the record columns");
    return both + (tile_chunks<D>() > 2 ? kMaxTileReads * 8u : 0u) + list_bytes<D>() + kCountBytes;
}

// A counter word: sum of 64 - q in bits 12:0, unique-hit records in 20:13,
// observed bases of other reads in 31:21.
constexpr uint32_t kOneRec = 1u << 13, kOneOther = 1u << 21;

// 16 bytes (two genotypes) of each of N parked rows
template <int N>
__device__ __forceinline__ void load_rows(const char* score, const uint8_t* parked, uint32_t cl, double2 (&y)[N])
{
    uint4 w[N / 8];
#pragma unroll
    for (int h = 0; h < N / 8; h++) w[h] = *reinterpret_cast<const uint4*>(parked + 16 * h);
#pragma unroll
    for (int h = 0; h < N / 8; h++) {
        const uint32_t p[4] = {w[h].x, w[h].y, w[h].z, w[h].w};
#pragma unroll
        for (int u = 0; u < 4; u++) {
            y[8 * h + 2 * u] = *reinterpret_cast<const double2*>(score + ((p[u] & 0xFFFFu) * 128u + cl));
            y[8 * h + 2 * u + 1] = *reinterpret_cast<const double2*>(score + ((p[u] >> 16) * 128u + cl));
        }
    }
}

template <int N>
__device__ __forceinline__ void add_rows(const double2 (&y)[N], double& a0, double& a1)
{
#pragma unroll
    for (int u = 0; u < N; u++) {
        a0 += y[u].x;
        a1 += y[u].y;
    }
}

// A read as the record loops take it, in three words that a wave holds one
// read per lane: its row's offset in the tile's bytes less its start, its
// start (bits 9:0), length (18:10) and strand (31), and what the record's
// cycle and strand fields are beyond the site's lane (record_word).
__device__ __forceinline__ uint32_t read_offset(uint32_t idx, uint32_t pitch, int32_t st) { return idx * pitch + 64u - (uint32_t)st; }
__device__ __forceinline__ uint32_t read_shape(int32_t st, uint32_t m)
{
    return ((uint32_t)st & 1023u) | (rm_len(m) << 10) | (m & 0x80000000u);
}
__device__ __forceinline__ int32_t shape_start(uint32_t w) { return __builtin_amdgcn_sbfe((int)w, 0, 10); }
__device__ __forceinline__ uint32_t shape_len(uint32_t w) { return (w >> 10) & 511u; }
// cycle << 9 | strand << 8 of lane l is (l << 9) + field on '+' and ~(l << 9) + field on '-'
__device__ __forceinline__ uint32_t shape_field(uint32_t w)
{
    const uint32_t st9 = (uint32_t)shape_start(w) << 9;
    return (w >> 31) ? st9 + ((shape_len(w) - 1u) << 9) + 257u : 0u - st9;
}

// waves of a block per class: one block takes a CU's LDS (two of 16 records)
constexpr int kWaves16 = 8, kWaves32 = 12, kWaves40 = 12, kWaves64 = 8, kWaves128 = 3;

template <int D, int NW>
__global__ __launch_bounds__(64 * NW) void k_call_tile(TileArgs f, const uint32_t* list, const uint32_t* count_ptr)
{
    extern __shared__ __align__(16) uint8_t lds[];
    const uint32_t count = *count_ptr;
    if (blockIdx.x * NW >= count) return;
    const uint32_t lane = __lane_id(), wib = uniform(threadIdx.x >> 6);
    const uint32_t td = (uint32_t)f.t.td & 511u, gd = (uint32_t)f.t.gd & 511u;
    const ReadView& r = f.reads;
    // the adjusted-quality table and the prior rows of the reference codes, once per block
    const uint32_t qwords = f.qtab_bytes / 4u;  // whole 16-byte units
    double* lprior = reinterpret_cast<double*>(lds);
    uint8_t* qtab = lds + kPriorBytes;
    __shared__ uint32_t block_sum;  // records of the block's sites
    if (threadIdx.x == 0) block_sum = 0;
    for (uint32_t i = threadIdx.x; i < 80u; i += 64u * NW) lprior[i] = f.t.lprior[i];
    for (uint32_t i = threadIdx.x; i < qwords; i += 64u * NW)
        reinterpret_cast<uint32_t*>(qtab)[i] = reinterpret_cast<const uint32_t*>(f.qtab)[i];
    __syncthreads();
    uint8_t* mine = lds + kPriorBytes + f.qtab_bytes + wib * wave_lds<D>();
    uint32_t* rec = reinterpret_cast<uint32_t*>(mine);  // [D][64]
    uint8_t* park = mine;
    uint32_t* cnt = reinterpret_cast<uint32_t*>(mine + wave_lds<D>() - kCountBytes);          // [4][64]
    uint32_t* shared_list = reinterpret_cast<uint32_t*>(mine + wave_lds<D>() - kCountBytes - list_bytes<D>());
    uint2* kept_reads = reinterpret_cast<uint2*>(shared_list) - kMaxTileReads;  // the deep class only
    // counters of big groups, [group][64]: what is left of the columns beside the parked rows
    constexpr uint32_t kColumns = D * kTile * 4u, kParked = kTile * park_stride<D>();
    constexpr uint32_t max_big = kColumns > kParked ? (kColumns - kParked) / (kTile * 4u) : 0u;
    uint32_t* big = reinterpret_cast<uint32_t*>(mine + kParked);
    const uint32_t pitch = r.pitch;
    const uint32_t nwave = gridDim.x * NW;
    const uint64_t below = lane == 0 ? 0ull : (~0ull >> (64 - lane));
    uint32_t records = 0;

    // the next tile's list entry, reads and first chunks are loaded while this
    // tile is worked on: four dependent loads otherwise
    constexpr uint32_t CH = tile_chunks<D>();
    uint32_t item = blockIdx.x * NW + wib;
    uint32_t tile = 0;
    uint64_t b = 0, e = 0;
    int32_t pos0 = 0, pos1 = 0;
    uint32_t m0 = 0, m1 = 0;
    auto load_first = [&](uint64_t rb, uint64_t re) {
        const bool ok0 = rb + lane < re, ok1 = rb + 64u + lane < re;
        pos0 = ok0 ? r.pos[rb + lane] : 0;
        m0 = ok0 ? r.meta[rb + lane] : 0u;
        if constexpr (CH == 2) {
            pos1 = ok1 ? r.pos[rb + 64u + lane] : 0;
            m1 = ok1 ? r.meta[rb + 64u + lane] : 0u;
        }
    };
    if (item < count) {
        tile = uniform(list[item]);
        b = uniform(f.range[2 * tile]), e = uniform(f.range[2 * tile + 1]);
        load_first(b, e);
    }
    while (item < count) {
        const bool more = item + nwave < count;
        const uint32_t next_item = more ? item + nwave : item;
        const uint32_t next_tile = list[next_item];
        const uint32_t R = (uint32_t)(e - b);  // <= 64 CH (k_tile_class)
        const uint32_t s = tile * kTile + lane;
        const int64_t p0 = (int64_t)f.ws + (int64_t)tile * kTile;
        const bool built = s < f.n_built;
        const uint32_t ori = s < f.n_sites ? f.ref.code[p0 + lane] & 0xFu : 0u;
        const int32_t x = built ? (int32_t)lane : 1 << 20;  // a lane beyond the span is covered by no read
        const uint32_t lane9 = lane << 9;

        // ---- A: records -------------------------------------------------
        // a chunk's read of this lane: start relative to the tile, and
        // metadata (0: no read)
        const int32_t st0 = (int32_t)((int64_t)pos0 - p0), st1 = (int32_t)((int64_t)pos1 - p0);
        if constexpr (CH > 2) {
            int32_t ps[CH];
            uint32_t ms[CH];
#pragma unroll
            for (uint32_t c = 0; c < CH; c++) {
                const bool ok = c * 64u + lane < R;
                ps[c] = ok ? r.pos[b + c * 64u + lane] : 0;
                ms[c] = ok ? r.meta[b + c * 64u + lane] : 0u;
            }
#pragma unroll
            for (uint32_t c = 0; c < CH; c++)
                kept_reads[c * 64u + lane] = make_uint2(ms[c] ? (uint32_t)(int32_t)((int64_t)ps[c] - p0) : 0u, ms[c]);
            wave_lds_sync();
        }
        auto load_read = [&](uint32_t c, int32_t& st, uint32_t& m) {
            if constexpr (CH > 2) {
                const uint2 w = kept_reads[c * 64u + lane];
                st = (int32_t)w.x;
                m = w.y;
            } else {
                m = c ? m1 : m0;
                st = m ? (c ? st1 : st0) : 0;
            }
        };
        auto anchor = [&](int32_t st, uint32_t m) -> uint32_t {
            const uint32_t rev = rm_strand(m);
            return ((uint32_t)(st + (rev ? (int32_t)rm_len(m) : 1) - 1 + 256) << 1) | rev;
        };
        const uint32_t nch = (R + 63u) / 64u;
        int32_t st;
        uint32_t m;
        load_read(0, st, m);
        // which reads share their anchor: the lowest read index of each
        // (anchor, strand) by an LDS minimum, then a flag for those with more
        // than one.  Two bits per chunk: 0 alone, 1 first of its group, 2 a
        // later member.
        uint32_t flags = 0;
        {
            uint4* z = reinterpret_cast<uint4*>(mine);
            const uint4 ones = make_uint4(~0u, ~0u, ~0u, ~0u);
#pragma unroll
            for (uint32_t k = 0; k < kAnchorWords / 256u; k++) z[k * 64u + lane] = ones;
            wave_lds_sync();
#pragma unroll 1
            for (uint32_t c = 0; c < nch; c++) {
                load_read(c, st, m);
                if (rm_hit(m) == 1) atomicMin(&rec[anchor(st, m)], c * 64u + lane);
            }
            wave_lds_sync();
#pragma unroll 1
            for (uint32_t c = 0; c < nch; c++) {
                load_read(c, st, m);
                if (rm_hit(m) == 1) {
                    uint32_t* w = &rec[anchor(st, m)];
                    if ((*w & 0xFFFFu) != c * 64u + lane) {
                        flags |= 2u << (2 * c);
                        atomicOr(w, 0x80000000u);
                    }
                }
            }
            wave_lds_sync();
#pragma unroll 1
            for (uint32_t c = 0; c < nch; c++) {
                load_read(c, st, m);
                if (rm_hit(m) == 1 && rec[anchor(st, m)] == (0x80000000u | (c * 64u + lane))) flags |= 1u << (2 * c);
            }
        }
        // the group members' list: first member of the group, then the read's index
        uint32_t n_shared = 0;  // wave-uniform
        if (__ballot(flags != 0)) {
#pragma unroll 1
            for (uint32_t c = 0; c < nch; c++) {
                load_read(c, st, m);
                const bool in = ((flags >> (2 * c)) & 3u) != 0;
                const uint64_t who = __ballot(in);
                if (in) {
                    const uint32_t at = n_shared + (uint32_t)__popcll(who & below);
                    const uint32_t first = rec[anchor(st, m)] & 0xFFFFu;
                    shared_list[at] = (first << 16) | (c * 64u + lane);
                }
                n_shared += (uint32_t)__popcll(who);
            }
        }
        wave_lds_sync();
        {
            uint4* z = reinterpret_cast<uint4*>(mine);
            const uint4 none = make_uint4(kNoRec, kNoRec, kNoRec, kNoRec);
#pragma unroll
            for (uint32_t k = 0; k < (uint32_t)D / 4u; k++) z[k * 64u + lane] = none;
            reinterpret_cast<uint4*>(cnt)[lane] = make_uint4(0, 0, 0, 0);
        }
        wave_lds_sync();
        uint32_t* slot = rec + lane;  // my next free slot
        int depth = 0, other = 0;     // reads over my site; hit counts of its repeat reads beyond one each
        // my byte of a read of the tile: unconditional (the read store is
        // padded on both sides), so that no load waits behind a branch; a read
        // that does not cover my site is told by its start and length
        const uint8_t* seqb = r.seq + b * (uint64_t)pitch - 64;
        auto load_byte = [&](uint32_t offset) -> uint32_t { return (seqb + offset)[lane]; };
        // appends my record of a unique-hit read with its count t
        auto add_record = [&](uint32_t byte, uint32_t shape, uint32_t field, uint32_t t) {
            const uint32_t flip = (uint32_t)((int32_t)shape >> 31);
            *slot = (byte << 17) + (lane9 ^ flip) + field + t;
            atomicAdd(&cnt[(byte & 0xC0u) + lane], (byte & 63u) | kOneRec);
            slot += kTile;
        };
#pragma unroll 1
        for (uint32_t c = 0; c < nch; c++) {
            load_read(c, st, m);
            const uint32_t idx = c * 64u + lane;
            const uint32_t hit = rm_hit(m);
            const bool there = idx < R, lone = hit == 1 && ((flags >> (2 * c)) & 3u) == 0;
            // reads alone on their anchor, moved to the first lanes: their
            // words then come from lanes known in advance.  Eight bytes are
            // in flight while the eight before them are used.
            const uint64_t who = __ballot(lone);
            const uint32_t n_lone = (uint32_t)__popcll(who);
            {
                const uint32_t to = (lone ? (uint32_t)__popcll(who & below)
                                          : n_lone + (uint32_t)__popcll(~who & below)) << 2;
                const uint32_t sh = lone ? read_shape(st, m) : 0u;  // length 0: covers nothing
                const uint32_t off = (uint32_t)__builtin_amdgcn_ds_permute((int)to, (int)read_offset(there ? idx : 0u, pitch, st));
                const uint32_t shape = (uint32_t)__builtin_amdgcn_ds_permute((int)to, (int)sh);
                const uint32_t field = shape_field(shape);
                auto fetch = [&](uint32_t k0, uint32_t (&byte)[8]) {
#pragma unroll
                    for (uint32_t u = 0; u < 8; u++) byte[u] = load_byte(lane_of(off, (k0 + u) & 63u));
                };
                auto use = [&](uint32_t k0, const uint32_t (&byte)[8]) {
#pragma unroll
                    for (uint32_t u = 0; u < 8; u++) {
                        const uint32_t w = lane_of(shape, k0 + u), fd = lane_of(field, k0 + u);
                        const bool in = (uint32_t)(x - shape_start(w)) < shape_len(w);
                        depth += in ? 1 : 0;
                        if (in && byte[u] != 0) add_record(byte[u], w, fd, 0u);
                    }
                };
                if (n_lone) {
                    uint32_t even[8], odd[8];
                    fetch(0, even);
#pragma unroll 1
                    for (uint32_t k = 0; k < n_lone; k += 16) {
                        fetch(k + 8, odd);
                        use(k, even);
                        fetch(k + 16, even);
                        if (k + 8 < n_lone) use(k + 8, odd);
                    }
                }
            }
            // repeat reads count, but leave no record
            uint64_t rep = __ballot(there && hit != 1);
            if (rep) {
                const uint32_t off = read_offset(there ? idx : 0u, pitch, st), shape = read_shape(st, m);
                while (rep) {
                    uint32_t byte[8], w[8], h[8];
#pragma unroll
                    for (uint32_t u = 0; u < 8; u++) {
                        const uint32_t j = rep ? (uint32_t)__builtin_ctzll(rep) : 0u;
                        w[u] = rep ? lane_of(shape, j) : 0u;
                        h[u] = lane_of(hit, j);
                        byte[u] = load_byte(lane_of(off, j));
                        rep &= rep - 1;
                    }
#pragma unroll
                    for (uint32_t u = 0; u < 8; u++) {
                        const bool in = (uint32_t)(x - shape_start(w[u])) < shape_len(w[u]);
                        depth += in ? 1 : 0;
                        other += in ? (int)h[u] - 1 : 0;
                        if (in && byte[u] != 0) atomicAdd(&cnt[(byte[u] & 0xC0u) + lane], kOneOther);
                    }
                }
            }
        }
        // groups that share an anchor, each whole and in read order: the
        // group's earlier records of my site are my last slots, and of two
        // with the same base the one of lower quality (or the later one)
        // counts the other
        auto add_member = [&](uint32_t byte, uint32_t w, uint32_t fd, uint32_t* group, uint32_t earlier,
                              uint32_t id) {
            const bool in = (uint32_t)(x - shape_start(w)) < shape_len(w);
            depth += in ? 1 : 0;
            const bool ok = in && byte != 0;
            uint32_t t = id;
            uint32_t* g = group;
            for (uint32_t k = 0; k < earlier; k++) {
                if (ok && g < slot) {
                    const uint32_t v = *g, vb = v >> 17;
                    if ((vb ^ byte) < 64u) {
                        if (vb <= byte)
                            t++;
                        else
                            *g = v + 1u;
                    }
                }
                g += kTile;
            }
            if (ok) add_record(byte, w, fd, t);
        };
        uint32_t n_big = 0;
        if (n_shared) {
            // ordered by group, then read: an entry's place is the count of
            // smaller words; bit 31 marks the members of a big group
            uint32_t mem[CH], place[CH], size[CH];
#pragma unroll
            for (uint32_t l = 0; l < CH; l++) {
                const uint32_t i = l * 64u + lane;
                mem[l] = i < n_shared ? shared_list[i] : ~0u;
                place[l] = size[l] = 0;
            }
#pragma unroll 1
            for (uint32_t k = 0; k < n_shared; k++) {
                const uint32_t y = uniform(shared_list[k]);
#pragma unroll
                for (uint32_t l = 0; l < CH; l++) {
                    place[l] += y < mem[l] ? 1u : 0u;
                    size[l] += (y ^ mem[l]) < 65536u ? 1u : 0u;
                }
            }
            wave_lds_sync();
#pragma unroll
            for (uint32_t l = 0; l < CH; l++)
                if (l * 64u + lane < n_shared) shared_list[place[l]] = mem[l] | (size[l] > kBigGroup ? 0x80000000u : 0u);
            wave_lds_sync();
            uint32_t* group = slot;
            uint32_t earlier = 0, id = 0;  // id: 128 + the big group's number, 0 in a small one
#pragma unroll 1
            for (uint32_t g0 = 0; g0 < n_shared; g0 += 64u) {
                const uint32_t i = g0 + lane;
                const uint32_t w = i < n_shared ? shared_list[i] : 0u;
                const uint32_t before = i && i < n_shared ? shared_list[i - 1u] : ~0u;
                const uint64_t heads = __ballot((w >> 16) != (before >> 16)), bigs = __ballot(w >> 31);
                const uint32_t idx = w & 0xFFFFu;
                uint32_t shape;
                if constexpr (CH > 2) {
                    const uint2 rd = kept_reads[idx];
                    shape = read_shape((int32_t)rd.x, rd.y);
                } else {
                    const uint32_t a0 = (uint32_t)__shfl((int)read_shape(st0, m0), (int)(idx & 63u));
                    const uint32_t a1 = (uint32_t)__shfl((int)read_shape(st1, m1), (int)(idx & 63u));
                    shape = idx < 64u ? a0 : a1;
                }
                const uint32_t off = read_offset(idx, pitch, shape_start(shape));
                const uint32_t field = shape_field(shape);
                const uint32_t here = n_shared - g0 < 64u ? n_shared - g0 : 64u;
#pragma unroll 1
                for (uint32_t k0 = 0; k0 < here; k0 += 8) {
                    uint32_t byte[8];
#pragma unroll
                    for (uint32_t u = 0; u < 8; u++) byte[u] = load_byte(lane_of(off, k0 + u));
#pragma unroll
                    for (uint32_t u = 0; u < 8; u++) {
                        if (k0 + u < here) {
                            if ((heads >> (k0 + u)) & 1u) {
                                group = slot;
                                earlier = 0;
                                id = ((bigs >> (k0 + u)) & 1u) && n_big < max_big ? 128u + n_big++ : 0u;
                            }
                            add_member(byte[u], lane_of(shape, k0 + u), lane_of(field, k0 + u), group, earlier, id);
                            earlier += id ? 0u : 1u;
                        }
                    }
                }
            }
        }
        wave_lds_sync();
        const uint32_t n = (uint32_t)(slot - rec) / kTile;  // records of my site
        SiteVals v;
        v.depth = depth;
        v.dep_uni = (int)n;
        const uint32_t w0 = cnt[lane], w1 = cnt[64 + lane], w2 = cnt[128 + lane], w3 = cnt[192 + lane];
        const uint32_t M = wave_max(n);
        const uint32_t tile2 = uniform(next_tile);
        const uint64_t b2 = f.range[2 * tile2], e2 = f.range[2 * tile2 + 1];

        // ---- B: sort, adjusted qualities, parked rows --------------------
        {
            uint32_t q[D];
#pragma unroll
            for (int k = 0; k < D; k++) q[k] = rec[k * kTile + lane];
            wave_lds_sync();  // the parked rows take the columns' place
            if constexpr (D == 64) {
                // short spans send every tile up to 64 records here
                if (M <= 32)
                    sort_regs<32>(q);
                else
                    sort_regs<64>(q);
            } else {
                sort_regs<D>(q);
            }
            const uint32_t cycles = pitch & 511u;
            if (n_big) {
                for (uint32_t k = 0; k < n_big; k++) big[k * kTile + lane] = 0;
                wave_lds_sync();
            }
            uint32_t prev = 0, g = ~0u;  // g: first occurrences of the base so far, minus one
#pragma unroll
            for (int k0 = 0; k0 < D; k0 += 8) {
                if ((uint32_t)k0 < M) {
                    uint32_t qa[8], tt[8];
#pragma unroll
                    for (int k = 0; k < 8; k++) tt[k] = q[k0 + k] & 255u;
                    if (n_big) {
                        // a big group's records of one base count themselves, a byte per base
#pragma unroll
                        for (int k = 0; k < 8; k++)
                            if (tt[k] & 128u) {
                                const uint32_t sh = (q[k0 + k] >> 23) << 3;
                                tt[k] = (atomicAdd(&big[(tt[k] & 127u) * kTile + lane], 1u << sh) >> sh) & 255u;
                            }
                    }
#pragma unroll
                    for (int k = 0; k < 8; k++) {
                        const uint32_t w = q[k0 + k];
                        g = (w ^ prev) < (1u << 23) ? g : ~0u;
                        prev = w;
                        const uint32_t t = tt[k];
                        g += t == 0 ? 1u : 0u;
                        const uint32_t tm = t < td ? t : td - 1u, gm = g < gd ? g : gd - 1u;
                        qa[k] = qtab[(((w >> 17) & 63u) * td + tm) * gd + gm];
                    }
                    uint32_t row[8];
#pragma unroll
                    for (int k = 0; k < 8; k++) {
                        const uint32_t w = q[k0 + k];
                        row[k] = ((w >> 23 << 6 & 0xC0u) + qa[k]) * cycles + ((w >> 9) & 0xFFu);
                    }
                    *reinterpret_cast<uint4*>(park + lane * park_stride<D>() + 2u * (uint32_t)k0) =
                        make_uint4(row[0] | (row[1] << 16), row[2] | (row[3] << 16), row[4] | (row[5] << 16),
                                   row[6] | (row[7] << 16));
                }
            }
        }
        wave_lds_sync();

        // ---- C: score rows in record order -------------------------------
        const uint64_t nb = uniform(b2), ne = uniform(e2);
        load_first(nb, ne);
        const char* score = reinterpret_cast<const char*>(f.score);
        // 320 (site, genotype pair) tasks in five rounds.  A site's sums take
        // the place of its parked rows one round late: its tasks lie in at
        // most two consecutive rounds.
        double p_a0 = 0.0, p_a1 = 0.0;
        uint8_t* p_at = nullptr;
#pragma unroll 1
        for (uint32_t k = 0; k < 5; k++) {
            const uint32_t task = k * 64u + lane, site = task / 5u, cl = (task - 5u * site) << 4;
            const uint32_t mm = (uint32_t)__shfl((int)n, (int)site);
            uint8_t* rw = park + site * park_stride<D>();
            double a0 = 0.0, a1 = 0.0;
            // eight rows (slots past the site's records hold row 0, all +0.0),
            // or sixteen while the site has that many left
            for (uint32_t i = 0; i < mm;) {
                if (i + 8u < mm) {
                    double2 y[16];
                    load_rows<16>(score, rw + 2u * i, cl, y);
                    add_rows<16>(y, a0, a1);
                    i += 16;
                } else {
                    double2 y[8];
                    load_rows<8>(score, rw + 2u * i, cl, y);
                    add_rows<8>(y, a0, a1);
                    i += 8;
                }
            }
            wave_lds_sync();
            if (k) *reinterpret_cast<double2*>(p_at) = make_double2(p_a0, p_a1);
            p_a0 = a0;
            p_a1 = a1;
            p_at = rw + cl;
        }
        *reinterpret_cast<double2*>(p_at) = make_double2(p_a0, p_a1);
        wave_lds_sync();

        // ---- D: call ------------------------------------------------------
        double acc[10];
#pragma unroll
        for (int h = 0; h < 5; h++) {
            const double2 y = *reinterpret_cast<const double2*>(park + lane * park_stride<D>() + 16 * h);
            acc[2 * h] = y.x;
            acc[2 * h + 1] = y.y;
        }
        v.cu = make_int4((int)((w0 >> 13) & 255u), (int)((w1 >> 13) & 255u), (int)((w2 >> 13) & 255u),
                         (int)((w3 >> 13) & 255u));
        v.qs = make_int4(64 * v.cu.x - (int)(w0 & 0x1FFFu), 64 * v.cu.y - (int)(w1 & 0x1FFFu),
                         64 * v.cu.z - (int)(w2 & 0x1FFFu), 64 * v.cu.w - (int)(w3 & 0x1FFFu));
        v.ca = make_int4(v.cu.x + (int)(w0 >> 21), v.cu.y + (int)(w1 >> 21), v.cu.z + (int)(w2 >> 21),
                         v.cu.w + (int)(w3 >> 21));
        v.ori = ori;
        const bool in_span = s < f.n_sites;
        SiteCall c = call_site(
            f.t, f.ref, (uint32_t)p0 + lane, v, [&](int g) { return acc[g]; },
            [&](int g) { return lprior[(ori & 7u) * 10u + (uint32_t)g]; });
        c.called = c.called && in_span;
        wave_lds_sync();  // the next tile's records take the sums' place
        if (in_span) {
            records += n;
            if (f.write_lk) {
                double2* out = reinterpret_cast<double2*>(f.out.lk + (size_t)s * 10);
#pragma unroll
                for (int h = 0; h < 5; h++) out[h] = make_double2(acc[2 * h], acc[2 * h + 1]);
            }
        }
        if (built) {
            f.a.depth[s] = depth;
            f.a.repeat[s] = depth + other;
            f.a.nrec[s] = (int)n;
            f.a.cu[s] = v.cu;
            f.a.qs[s] = v.qs;
            f.a.ca[s] = v.ca;
        }
        int4 nq = v.qs;
        const uint64_t ask = __ballot(c.called && c.next);
        if (ask) {  // N references: rare
            nq.x = __shfl_down(v.qs.x, 1);
            nq.y = __shfl_down(v.qs.y, 1);
            nq.z = __shfl_down(v.qs.z, 1);
            nq.w = __shfl_down(v.qs.w, 1);
        }
        // sites whose reads the whole wave looks at: a het of the rank-sum
        // mode (the test reads its records from memory), the next tile's first
        // site where the last lane asks for its q_sum, and the first site of a
        // window for its q_sum before the reads that start on it
        uint64_t rows = __ballot(c.called && job_site(f.t, v, c));
        uint32_t extra = ((ask >> 63) ? 1u : 0u) | (p0 % kWin == 0 ? 2u : 0u);
        while (rows || extra) {
            uint32_t l = kTile, what = 0;  // 0: a row, 1: the next tile's site, 2: the window's first
            if (rows) {
                l = (uint32_t)__builtin_ctzll(rows);
                rows &= rows - 1;
            } else {
                what = extra & 1u ? 1u : 2u;
                extra &= ~what;
                l = what == 1u ? kTile : 0u;
            }
            const uint32_t t = what == 1u ? tile + 1u : tile;
            const int64_t p = p0 + l;
            const uint64_t rb = uniform(f.range[2 * t]), re = uniform(f.range[2 * t + 1]);
            const int4 h = wave_site_records(f.reads, rb, re, p, what && p % kWin == 0 ? p - 1 : p,
                                             what ? nullptr : f.a.rec + ((size_t)tile * kTile + l) * kSlots);
            if (what == 1u && lane == 63) nq = h;
            if (what == 2u && lane == 0) f.head_qs[p0 / kWin - f.ws / kWin] = h;
        }
        if (c.called) finish_site(f.t, v, c, nq, s, f.out, f.jobs, f.job_count);
        item += nwave;
        tile = tile2;
        b = nb;
        e = ne;
    }
    for (int off = 32; off > 0; off >>= 1) records += (uint32_t)__shfl_xor((int)records, off);
    // one global add per block: adds to one address take turns
    if (lane == 0) atomicAdd(&block_sum, records);
    __syncthreads();  // every wave of a block with work comes here
    if (threadIdx.x == 0) atomicAdd(f.n_records, (unsigned long long)block_sum);
}

// What a span's first launch clears.
__global__ __launch_bounds__(256) void k_span_clear(SpanClear clr)
{
    const uint32_t i = blockIdx.x * 256u + threadIdx.x;
    if (i < clr.n_heads) clr.head_qs[i] = make_int4(0, 0, 0, 0);
    if (i < 8) clr.counts[i * kCountStride] = clr.counts[i] = 0;
    if (i == 8) *clr.job_count = 0;
    if (i == 9) *clr.fix_count = 0;
}

// first read that starts at or after v: a search among the reads of v's
// kReadBlock sites.  The index is that of the last reads loaded, which a
// chromosome without reads (n = 0) does not have.
__device__ uint64_t lower_start(const ReadView& r, int64_t v)
{
    if (v <= 0 || r.n == 0) return 0;
    const uint64_t k = (uint64_t)v / kReadBlock;
    uint64_t lo = r.first[k], hi = r.first[k + 1];
    while (lo < hi) {
        const uint64_t m = (lo + hi) >> 1;
        if ((int64_t)r.pos[m] < v)
            lo = m + 1;
        else
            hi = m;
    }
    return lo;
}

// The reads of each tile, its class -- the largest number of unique-hit reads
// over one of its sites, from their starts and ends -- and its place in its
// class list.  A wave takes K tiles: their range searches run side by side
// in its lanes, and their reads' positions and metadata are loaded together,
// so that the pass is a few memory latencies long instead of a few per tile.
template <uint32_t K>
__global__ __launch_bounds__(512) void k_tile_class(ReadView r, uint32_t ws, uint32_t n_tiles, uint32_t min_class,
                                                    uint64_t* range, uint32_t* lists, uint32_t pitch, uint32_t* counts)
{
    __shared__ int hist[8][kTile];
    __shared__ uint32_t in_wave[8][kDeepClass + 1], block_base[kDeepClass + 1];
    const uint32_t lane = __lane_id(), w = uniform(threadIdx.x >> 6);
    const uint32_t t0 = (blockIdx.x * 8u + w) * K;
    // lane 2k / 2k + 1: the range of tile k
    uint64_t rg = 0;
    if (lane < 2u * K && (uint64_t)t0 + lane / 2u < n_tiles) {
        const int64_t p = (int64_t)ws + ((int64_t)t0 + lane / 2u) * kTile;
        rg = lower_start(r, lane & 1u ? p + kTile : p - ((int64_t)r.pitch - 1));
        range[2 * (size_t)t0 + lane] = rg;
    }
    const uint32_t rlo = (uint32_t)rg, rhi = (uint32_t)(rg >> 32);
    int32_t pos[K];
    uint32_t meta[K];
#pragma unroll
    for (uint32_t k = 0; k < K; k++) {
        const uint64_t b = ((uint64_t)lane_of(rhi, 2 * k) << 32) | lane_of(rlo, 2 * k);
        const uint64_t e = ((uint64_t)lane_of(rhi, 2 * k + 1) << 32) | lane_of(rlo, 2 * k + 1);
        const bool ok = b + lane < e;  // a tile beyond the span has no reads
        pos[k] = ok ? r.pos[b + lane] : 0;
        meta[k] = ok ? r.meta[b + lane] : 0u;
    }
    uint32_t cls = ~0u;  // lane k: class of tile k
#pragma unroll
    for (uint32_t k = 0; k < K; k++) {
        const uint32_t tile = t0 + k;
        if (tile >= n_tiles) break;
        const uint64_t b = ((uint64_t)lane_of(rhi, 2 * k) << 32) | lane_of(rlo, 2 * k);
        const uint64_t e = ((uint64_t)lane_of(rhi, 2 * k + 1) << 32) | lane_of(rlo, 2 * k + 1);
        uint32_t c = kDeepClass;
        if (e - b <= kMaxTileReads) {
            const int64_t p0 = (int64_t)ws + (int64_t)tile * kTile;
            hist[w][lane] = 0;
            wave_lds_sync();
            int uniq = 0;  // my unique-hit reads
            auto count = [&](int32_t p, uint32_t m) {
                uniq += rm_hit(m) == 1 ? 1 : 0;
                const int32_t st = (int32_t)((int64_t)p - p0), en = st + (int32_t)rm_len(m);
                if (rm_hit(m) == 1 && en > 0) {
                    atomicAdd(&hist[w][st > 0 ? st : 0], 1);
                    if (en < (int32_t)kTile) atomicAdd(&hist[w][en], -1);
                }
            };
            count(pos[k], meta[k]);
            for (uint64_t i = b + 64u + lane; i < e; i += 64) count(r.pos[i], r.meta[i]);
            wave_lds_sync();
            const uint32_t most = wave_max((uint32_t)wave_prefix(hist[w][lane]));
            c = most <= 16 ? 0u : most <= 32 ? 1u : most <= 40 ? 2u : most <= 64 ? 3u : most <= 128 ? 4u : kDeepClass;
            if (e - b > kShallowReads && c < 4u) c = 4u;
            if (e - b > max_unique(r.pitch) && lane_of((uint32_t)wave_prefix(uniq), 63) > max_unique(r.pitch)) c = kDeepClass;
            if (c < min_class) c = min_class;
        }
        cls = lane == k ? c : cls;
    }
    // places within the block, one global add per class and block (adds to
    // one address take turns, so the classes' counters lie on lines of their own)
    const uint64_t below = lane == 0 ? 0ull : (~0ull >> (64 - lane));
    uint32_t place = 0;
#pragma unroll
    for (uint32_t k = 0; k <= kDeepClass; k++) {
        const uint64_t who = __ballot(cls == k);
        if (lane == 0) in_wave[w][k] = (uint32_t)__popcll(who);
        place = cls == k ? (uint32_t)__popcll(who & below) : place;
    }
    __syncthreads();
    if (threadIdx.x <= kDeepClass) {
        uint32_t sum = 0;
        for (uint32_t j = 0; j < 8; j++) {
            const uint32_t x = in_wave[j][threadIdx.x];
            in_wave[j][threadIdx.x] = sum;
            sum += x;
        }
        block_base[threadIdx.x] = sum ? atomicAdd(&counts[threadIdx.x * kCountStride], sum) : 0u;
    }
    __syncthreads();
    if (cls <= kDeepClass) lists[(size_t)cls * pitch + block_base[cls] + in_wave[w][cls] + place] = t0 + lane;
}

__global__ __launch_bounds__(256) void k_tile_scores(const double* score, double* tscore, uint32_t cycles)
{
    const uint32_t i = blockIdx.x * 256u + threadIdx.x;  // a double of the tile table
    const uint32_t row = i / kScoreRowStride, k = i % kScoreRowStride;
    const uint32_t o = row / (64u * cycles), qa = row / cycles % 64u, cyc = row % cycles;
    tscore[i] = score[(size_t)((qa << 10) | (cyc << 2) | o) * kScoreRowStride + k];
}

// more than 64 KB of dynamic LDS, on the current device
template <int D, int NW>
hipError_t allow_class()
{
    constexpr uint32_t most = kPriorBytes + kTileQtabMax + NW * wave_lds<D>();
    static_assert(most <= 163840u, "a CU's LDS");
    return hipFuncSetAttribute(reinterpret_cast<const void*>(&k_call_tile<D, NW>),
                               hipFuncAttributeMaxDynamicSharedMemorySize, (int)most);
}

template <int D, int NW>
void launch_class(hipStream_t st, const TileArgs& f, const uint32_t* list, const uint32_t* count, uint32_t n_tiles,
                  uint32_t per_cu)
{
    const uint32_t bytes = kPriorBytes + f.qtab_bytes + NW * wave_lds<D>();
    uint32_t blocks = (n_tiles + NW - 1) / NW;
    if (blocks > 256u * per_cu) blocks = 256u * per_cu;
    hipLaunchKernelGGL((k_call_tile<D, NW>), dim3(blocks), dim3(64 * NW), bytes, st, f, list, count);
}

}  // namespace

hipError_t allow_tile_lds()
{
    for (hipError_t (*allow)() : {allow_class<64, kWaves64>, allow_class<40, kWaves40>, allow_class<32, kWaves32>,
                                  allow_class<16, kWaves16>, allow_class<128, kWaves128>})
        if (const hipError_t e = allow()) return e;
    return hipSuccess;
}

uint32_t tile_min_class(uint32_t n_tiles) { return n_tiles <= kFewTiles ? 3u : 0u; }

void launch_span_clear(hipStream_t st, const SpanClear& clr)
{
    const uint32_t n = clr.n_heads < 10u ? 10u : clr.n_heads;
    hipLaunchKernelGGL(k_span_clear, dim3((n + 255) / 256), dim3(256), 0, st, clr);
}

void launch_tile_classes(hipStream_t st, const ReadView& r, uint32_t ws, uint32_t n_tiles, uint64_t* range,
                         uint32_t* lists, uint32_t pitch, const SpanClear& clr)
{
    launch_span_clear(st, clr);
    if (!n_tiles) return;
    const uint32_t mc = tile_min_class(n_tiles);
    constexpr uint32_t K = 8;
    hipLaunchKernelGGL(k_tile_class<K>, dim3((n_tiles + 8 * K - 1) / (8 * K)), dim3(512), 0, st, r, ws, n_tiles, mc, range,
                       lists, pitch, clr.counts);
}

void launch_tile_scores(hipStream_t st, const double* score, double* tscore, uint32_t cycles)
{
    static_assert(4u * 64u * kScoreRowStride % 256u == 0, "whole blocks");
    hipLaunchKernelGGL(k_tile_scores, dim3(4u * 64u * cycles * kScoreRowStride / 256u), dim3(256), 0, st, score, tscore,
                       cycles);
}

void launch_call_tiles(hipStream_t st, const TileArgs& f, const uint32_t* lists, uint32_t pitch, const uint32_t* counts,
                       uint32_t n_tiles)
{
    if (!n_tiles) return;
    const uint32_t C = kCountStride;
    launch_class<64, kWaves64>(st, f, lists + 3 * (size_t)pitch, counts + 3 * C, n_tiles, 1);
    if (tile_min_class(n_tiles)) return;
    launch_class<40, kWaves40>(st, f, lists + 2 * (size_t)pitch, counts + 2 * C, n_tiles, 1);
    launch_class<32, kWaves32>(st, f, lists + 1 * (size_t)pitch, counts + 1 * C, n_tiles, 1);
    launch_class<16, kWaves16>(st, f, lists + 0 * (size_t)pitch, counts + 0 * C, n_tiles, 2);
}

void launch_call_deepest(hipStream_t st, const TileArgs& f, const uint32_t* lists, uint32_t pitch,
                         const uint32_t* counts, uint32_t n_tiles)
{
    if (n_tiles) launch_class<128, kWaves128>(st, f, lists + 4 * (size_t)pitch, counts + 4 * kCountStride, n_tiles, 1);
}

}  // namespace gsnp
