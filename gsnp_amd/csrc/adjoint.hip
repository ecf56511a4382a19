// adjoint.hip -- gradient of the summed per-site log marginal likelihood
//
//   l = sum_s ln sum_g prior_s(g) 10^{lk_s(g)},
//   lk_s(g) = sum_r log10(0.5 p[qa_r, c_r, a1(g), o_r] + 0.5 p[qa_r, c_r, a2(g), o_r])
//
// with respect to ln p[q][c][a][o] (q < 64) and ln het_rate, where the records
// r of a site, their adjusted qualities qa_r and the genotype order are those
// of the calling path (kernel/likelihood_kernel.cu:137-256) and the priors
// those of cpp/prior.cc.  No reference counterpart: the reference has no
// gradient.  With w_s(g) = prior_s(g) 10^{lk_s(g)} / sum_g', the gradient is
//
//   dl/d ln p[q,c,a,o] = sum_{records r with key (q,c,o)} sum_g w_s(g) share_g(a)
//   share_g(a) = p_a ([a == a1] + [a == a2]) / (p_a1 + p_a2)
//   dl/d ln het = sum_s sum_g w_s(g) [prior_s(g) carries one factor of het]
//
// By linearity a key's four entries come from the ten sums W_k(g) of w_s(g)
// over its records, share_g(a) being the key's own.  Accumulation is
// deterministic and in a fixed order: sites are cut into blocks of kSiteBlock,
// the records of each block are sorted by key once (stable LSD radix sort of
// words key << 16 | site in block) and cut into chunks of kChunk, and each
// evaluation sums the weights of every piece -- a chunk's records of one key --
// in that order, then a key's pieces over the blocks in eight parts, then the
// parts.  No
// floating-point atomics.
//
// A block's weights (2 MB, a 128-byte line per site) stay in an XCD's L2 while
// the block's pieces gather them; sorted by key over the whole span, every
// record fetched its 80 bytes from beyond L2, 1.5 lines each, and took its own
// divisions.  2 Mb at 30x (60 million records): the pieces take 0.56 ms instead
// of 1.64, an evaluation 1.38 ms instead of 2.76.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstring>
#include <string>
#include <vector>

#include "../../include/gsnp_abi.h"
#include "engine.h"
#include "gsnp_common.h"
#include "kernels.h"
#include "tables.h"

namespace gsnp {

namespace {

constexpr uint32_t kNoRow = 0xFFFFFFFFu;
constexpr uint32_t kChunk = 64;         // records that one lane group sums at a time
constexpr uint32_t kSiteBlock = 16384;  // sites whose records are sorted together; a power of two, at most 65,536
constexpr uint32_t kWStride = 16;       // doubles per site of the weights: one line
constexpr uint32_t kParts = 8;          // parts of a key's sum over the site blocks
constexpr uint32_t kKeys = 65536;       // score-row keys with q < 64: q<<10 | cycle<<2 | o
constexpr uint32_t kRadixChunk = 4096;  // items per block of a radix pass (16 tiles of 256)

// per site: record count of a called site and its prior row (0..7 reference
// rows, 8+i known SNP i); N rows without coverage are not called
__global__ __launch_bounds__(256) void k_adj_sites(Tables t, RefView ref, uint32_t ws, SiteArrays a, uint32_t n,
                                                   uint32_t* cnt, uint32_t* prow)
{
    const uint32_t s = blockIdx.x * 256u + threadIdx.x;
    if (s >= n) return;
    const uint32_t ori = ref.code[ws + s] & 0xF;
    if ((ori & 4) && a.depth[s] == 0) {
        cnt[s] = 0;
        prow[s] = kNoRow;
        return;
    }
    cnt[s] = (uint32_t)a.nrec[s];
    uint32_t row = ori & 7;
    if ((ori & 8) && t.refine && ref.n_snp) {
        uint32_t lo = 0, hi = ref.n_snp;
        const uint32_t p = ws + s;
        while (lo < hi) {
            const uint32_t m = (lo + hi) >> 1;
            if (ref.snp_pos[m] < p)
                lo = m + 1;
            else
                hi = m;
        }
        if (lo < ref.n_snp && ref.snp_pos[lo] == p) row = 8 + lo;
    }
    prow[s] = row;
}

// exclusive scan of u32 counts into u64 offsets: per-block local scan, block
// sums scanned by k_scan_blocks, then the block offsets added
__global__ __launch_bounds__(256) void k_scan_local(const uint32_t* in, uint32_t n, uint64_t* out, uint64_t* bsum)
{
    __shared__ uint64_t ws[4];
    const uint32_t i = blockIdx.x * 256u + threadIdx.x;
    const uint64_t x = i < n ? in[i] : 0;
    uint64_t incl = x;
    const uint32_t lane = __lane_id(), w = threadIdx.x >> 6;
    for (int off = 1; off < 64; off <<= 1) {
        const uint64_t y = __shfl_up(incl, off);
        if ((int)lane >= off) incl += y;
    }
    if (lane == 63) ws[w] = incl;
    __syncthreads();
    uint64_t before = 0;
    for (uint32_t k = 0; k < w; k++) before += ws[k];
    if (i < n) out[i] = before + incl - x;
    if (threadIdx.x == 255) bsum[blockIdx.x] = before + incl;
}

__global__ __launch_bounds__(256) void k_scan_add(uint64_t* out, uint32_t n, const uint64_t* boff, const uint64_t* total)
{
    const uint32_t i = blockIdx.x * 256u + threadIdx.x;
    if (i < n) out[i] += boff[blockIdx.x];
    if (i == n) out[n] = *total;
}

// ---- stable LSD radix sort of each site block's record words by key --------
// Block y of the grid is a site block: its words are [start[y], start[y + 1]),
// its digit counts lie at hbase[y] + digit * chunks + chunk, so that one scan
// of all counts gives every place.

__global__ __launch_bounds__(256) void k_block_starts(const uint64_t* off, uint32_t n, uint32_t nblk, uint64_t* start)
{
    const uint32_t i = blockIdx.x * 256u + threadIdx.x;
    if (i <= nblk) start[i] = off[(uint64_t)i * kSiteBlock < n ? (uint64_t)i * kSiteBlock : n];
}

__global__ __launch_bounds__(256) void k_radix_hist(const uint32_t* word, const uint64_t* start, const uint32_t* hbase,
                                                    uint32_t shift, uint32_t* hist)
{
    __shared__ uint32_t h[256];
    const uint64_t b = start[blockIdx.y], e = start[blockIdx.y + 1];
    const uint32_t chunks = (uint32_t)((e - b + kRadixChunk - 1) / kRadixChunk);
    if (blockIdx.x >= chunks) return;
    h[threadIdx.x] = 0;
    __syncthreads();
    const uint64_t c0 = b + (uint64_t)blockIdx.x * kRadixChunk;
#pragma unroll 4
    for (uint32_t i = threadIdx.x; i < kRadixChunk; i += 256)
        if (c0 + i < e) atomicAdd(&h[(word[c0 + i] >> shift) & 255u], 1u);
    __syncthreads();
    hist[(size_t)hbase[blockIdx.y] + threadIdx.x * chunks + blockIdx.x] = h[threadIdx.x];
}

// Each block scatters its chunk in input order, one tile of 256 at a time:
// an item's place is its digit's offset for the block, plus the items of the
// same digit in earlier tiles, earlier waves and earlier lanes of its wave.
__global__ __launch_bounds__(256) void k_radix_scatter(const uint32_t* word, const uint64_t* start,
                                                       const uint32_t* hbase, uint32_t shift, const uint64_t* off,
                                                       uint32_t* out)
{
    __shared__ uint32_t wcnt[2][4][256];
    __shared__ uint64_t place[256];  // next place of each digit
    const uint64_t b = start[blockIdx.y], e = start[blockIdx.y + 1];
    const uint32_t chunks = (uint32_t)((e - b + kRadixChunk - 1) / kRadixChunk);
    if (blockIdx.x >= chunks) return;
    const uint32_t lane = __lane_id(), w = threadIdx.x >> 6;
    const uint64_t below = lane == 0 ? 0ull : (~0ull >> (64 - lane));
    place[threadIdx.x] = off[(size_t)hbase[blockIdx.y] + threadIdx.x * chunks + blockIdx.x];
    for (uint32_t k = 0; k < 2; k++)
        for (uint32_t j = 0; j < 4; j++) wcnt[k][j][threadIdx.x] = 0;
    __syncthreads();
    const uint64_t c0 = b + (uint64_t)blockIdx.x * kRadixChunk;
    constexpr uint32_t T = kRadixChunk / 256u;
    uint32_t v[T];
#pragma unroll
    for (uint32_t t = 0; t < T; t++) {
        const uint64_t idx = c0 + t * 256u + threadIdx.x;
        v[t] = idx < e ? word[idx] : 0u;
    }
#pragma unroll
    for (uint32_t t = 0; t < T; t++) {
        const bool valid = c0 + t * 256u + threadIdx.x < e;
        const uint32_t d = (v[t] >> shift) & 255u;
        uint64_t peers = __ballot(valid);
#pragma unroll
        for (int k = 0; k < 8; k++) {
            const uint64_t bal = __ballot((d >> k) & 1u);
            peers &= ((d >> k) & 1u) ? bal : ~bal;
        }
        const uint32_t rank = (uint32_t)__popcll(peers & below);
        const uint32_t cntw = (uint32_t)__popcll(peers);
        uint32_t(*cnt)[256] = wcnt[t & 1u];  // the other buffer is cleared for the next tile
        if (valid && rank == cntw - 1) cnt[w][d] = cntw;
        __syncthreads();
        if (valid) {
            uint64_t pos = place[d] + rank;
            for (uint32_t j = 0; j < w; j++) pos += cnt[j][d];
            out[pos] = v[t];
        }
        __syncthreads();
        place[threadIdx.x] += cnt[0][threadIdx.x] + cnt[1][threadIdx.x] + cnt[2][threadIdx.x] + cnt[3][threadIdx.x];
        for (uint32_t j = 0; j < 4; j++) cnt[j][threadIdx.x] = 0;
    }
}

// piece heads: a new piece starts at every site block, key change and
// kChunk-th word of a block
__global__ __launch_bounds__(256) void k_piece_flags(const uint32_t* word, const uint64_t* start, uint32_t* flag,
                                                     uint32_t* used)
{
    const uint64_t b = start[blockIdx.y], e = start[blockIdx.y + 1];
    for (uint64_t j = b + blockIdx.x * 256u + threadIdx.x; j < e; j += gridDim.x * 256u) {
        const uint32_t k = word[j] >> 16;
        const bool head = (j - b) % kChunk == 0 || k != word[j - 1] >> 16;
        flag[j] = head ? 1u : 0u;
        if (head) used[k] = 1u;
    }
}

__global__ __launch_bounds__(256) void k_piece_starts(const uint32_t* flag, const uint64_t* pidx, uint32_t n,
                                                      const uint64_t* start, uint32_t nblk, uint32_t* pstart,
                                                      uint32_t* pblock)
{
    const uint32_t j = blockIdx.x * 256u + threadIdx.x;
    if (j < n && flag[j]) pstart[pidx[j]] = j;
    if (j == 0) pstart[pidx[n]] = n;
    if (j <= nblk) pblock[j] = (uint32_t)pidx[start[j]];  // pieces before the block: pidx counts the heads before a word
}

__global__ __launch_bounds__(256) void k_chunk_pieces(const uint64_t* pidx, const uint64_t* start, const uint32_t* cbase,
                                                      uint32_t* cpiece)
{
    const uint32_t c = blockIdx.x * 256u + threadIdx.x, chunks = cbase[blockIdx.y + 1] - cbase[blockIdx.y];
    if (c < chunks) cpiece[cbase[blockIdx.y] + c] = (uint32_t)pidx[start[blockIdx.y] + (uint64_t)c * kChunk];
}

// the used keys in order, then each block's first piece of each used key
__global__ __launch_bounds__(256) void k_used_keys(const uint32_t* used, const uint64_t* uidx, uint32_t* ukey)
{
    const uint32_t k = blockIdx.x * 256u + threadIdx.x;
    if (k < kKeys && used[k]) ukey[uidx[k]] = k;
}

__global__ __launch_bounds__(256) void k_key_pieces(const uint32_t* word, const uint32_t* pstart, const uint32_t* pblock,
                                                    const uint32_t* ukey, uint32_t nuk, uint32_t* kpiece)
{
    const uint32_t i = blockIdx.x * 256u + threadIdx.x;
    if (i > nuk) return;
    uint32_t lo = pblock[blockIdx.y], hi = pblock[blockIdx.y + 1];
    const uint32_t k = i < nuk ? ukey[i] : ~0u;
    while (lo < hi) {
        const uint32_t m = (lo + hi) >> 1;
        if (word[pstart[m]] >> 16 < k)
            lo = m + 1;
        else
            hi = m;
    }
    kpiece[(size_t)blockIdx.y * (nuk + 1u) + i] = lo;
}

// ---- evaluation ------------------------------------------------------------

// device score rows for q < 64 from the current p_matrix (device log10; the
// calling path's exact table is host-built)
__global__ __launch_bounds__(256) void k_adj_table(const double* pm, double* T)
{
    const uint32_t r = blockIdx.x * 256u + threadIdx.x;  // q<<10 | c<<2 | o
    if (r >= kKeys) return;
    const uint32_t q = r >> 10, c = (r >> 2) & 255u, o = r & 3u;
    const double* row = pm + ((size_t)q << 12) + ((size_t)c << 4);
    double* out = T + (size_t)r * kScoreRowStride;
    int g = 0;
    for (uint32_t a1 = 0; a1 < 4; a1++)
        for (uint32_t a2 = a1; a2 < 4; a2++) {
            const double h1 = 0.5 * row[(a1 << 2) | o], h2 = 0.5 * row[(a2 << 2) | o];
            out[g++] = log10(h1 + h2);
        }
}

// consecutive words, four to a load at any four-byte alignment; arrays hold
// kWordPad words past their end
constexpr uint32_t kWordPad = 16;
typedef uint32_t Word4 __attribute__((ext_vector_type(4), aligned(4)));

template <uint32_t U>
struct Words {
    uint32_t w[U];
    __device__ __forceinline__ void load(const uint32_t* p)
    {
#pragma unroll
        for (uint32_t i = 0; i < U; i += 4) {
            const Word4 v = *reinterpret_cast<const Word4*>(p + i);
            w[i] = v.x;
            w[i + 1] = v.y;
            w[i + 2] = v.z;
            w[i + 3] = v.w;
        }
    }
};

// per site: log-likelihoods in record order, log marginal, genotype weights
// and the het derivative.  Five lanes per site add its score rows (two
// genotypes each, every genotype in record order, eight records in flight):
// one load instruction reads whole 80-byte rows of twelve sites instead of a
// 16-byte piece of 64 rows, while the next eight words load.  The ten sums meet in LDS; each lane takes the
// exponentials and weights of its own two genotypes (on one lane of the five
// they were most of the kernel's instructions).  2 Mb at 30x: 0.46 ms, was 0.60;
// the row gathers alone take 0.23 at the rate measured for lines out of L2.
constexpr uint32_t kAdjSitesPerWave = 12;

__global__ __launch_bounds__(256) void k_adj_site(const double* T, const uint32_t* word, const uint64_t* off,
                                                  const uint32_t* prow, const double* lp, const uint32_t* hmask,
                                                  uint32_t n, int monoploid, double* ll, double* dh, double* wout)
{
    __shared__ __align__(16) double sums[4][65][2];  // [wave][5 * site + pair]: a site's ten values are contiguous; lanes 60-63 read to row 64
    const uint32_t lane = __lane_id(), wib = threadIdx.x >> 6;
    const uint32_t sl = lane / 5u, cl = lane - 5u * sl;
    const uint32_t s = (blockIdx.x * 4u + wib) * kAdjSitesPerWave + sl;
    const bool on = lane < 60u && s < n;
    const uint64_t r0 = on ? off[s] : 0, r1 = on ? off[s + 1] : 0;
    const uint32_t pr = on ? prow[s] : kNoRow;
    double a0 = 0.0, a1 = 0.0;
    constexpr uint32_t U = 8;
    const uint32_t len = (uint32_t)(r1 - r0);
    const uint32_t* wp = word + r0;
    Words<U> cur, next;
    cur.load(wp);
    for (uint32_t j = 0; j < len; j += U) {
        double2 x[U];  // every 16-bit key has a row, also those of words past the site's
#pragma unroll
        for (uint32_t u = 0; u < U; u++)
            x[u] = *reinterpret_cast<const double2*>(T + (size_t)(cur.w[u] >> 16) * kScoreRowStride + 2u * cl);
        next.load(wp + j + U);
#pragma unroll
        for (uint32_t u = 0; u < U; u++)
            if (j + u < len) {
                a0 += x[u].x;
                a1 += x[u].y;
            }
        cur = next;
    }
    const double* row = lp + (size_t)(pr == kNoRow ? 0u : pr) * 10;
    auto het = [&](uint32_t g) {
        const uint32_t gt = geno_code((int)g);
        return (gt >> 2) != (gt & 3u);
    };
    double2* mine = reinterpret_cast<double2*>(sums[wib][lane]);
    const double* ten = sums[wib][5u * sl];
    const double v0 = monoploid && het(2u * cl) ? -INFINITY : row[2u * cl] + a0;
    const double v1 = monoploid && het(2u * cl + 1u) ? -INFINITY : row[2u * cl + 1u] + a1;
    *mine = make_double2(v0, v1);
    wave_lds_sync();
    double m = -INFINITY;
#pragma unroll
    for (int g = 0; g < 10; g++) m = ten[g] > m ? ten[g] : m;
    wave_lds_sync();
    const double e0 = exp10(v0 - m), e1 = exp10(v1 - m);
    *mine = make_double2(e0, e1);
    wave_lds_sync();
    double z = 0.0;
#pragma unroll
    for (int g = 0; g < 10; g++) z += ten[g];
    wave_lds_sync();
    const bool called = pr != kNoRow;
    const double w0 = called ? e0 / z : 0.0, w1 = called ? e1 / z : 0.0;
    *mine = make_double2(w0, w1);
    wave_lds_sync();
    if (!on) return;
    *reinterpret_cast<double2*>(wout + (size_t)s * kWStride + 2u * cl) = make_double2(w0, w1);
    if (cl != 0) return;
    double d = 0.0;
    if (called) {
        const uint32_t mask = hmask[pr];
#pragma unroll
        for (int g = 0; g < 10; g++)
            if ((mask >> g) & 1u) d += ten[g];
    }
    ll[s] = called ? m * 2.302585092994045684 + log(z) : 0.0;
    dh[s] = d;
}

// The ten weights summed over each piece, in order: five lanes per chunk, two
// genotypes each, twelve chunks per wave, eight records in flight while the
// next eight words load.  A chunk's pieces follow each other in a lane group,
// so every group has the same work whatever the pieces' lengths (with a group
// per piece of up to 256 records, a block took as long as its longest piece:
// 0.89 ms over 60 million records, 0.79 in chunks).  Workgroups are dealt to
// the eight XCDs in turn and start in order, so the list of work gives
// workgroup 8 j + x the j-th share of the site blocks x, x + 8, ...: a block's
// weights are gathered by one XCD, out of its L2, while few blocks are in flight
// (waves that stay for the whole launch drift apart over the blocks, and two in
// three gathers missed: 0.79 ms; this way 0.56).
// Chunks of 32 and blocks of 8,192 sites are as fast here, but their pieces
// cost the next kernel 35 to 75 us more.
constexpr uint32_t kChunksPerGroup = 48;  // of a workgroup

__global__ __launch_bounds__(256) void k_adj_pieces(const uint32_t* word, const double* wsite, const uint64_t* start,
                                                    const uint32_t* cbase, const uint32_t* cpiece, const uint2* work,
                                                    double* psum)
{
    const uint32_t lane = __lane_id(), sl = lane / 5u, cl = lane - 5u * sl;
    const uint2 wk = work[blockIdx.x];  // site block, first chunk
    const uint32_t b = wk.x, c0 = cbase[b], chunks = cbase[b + 1] - c0;
    const uint32_t c = wk.y + (threadIdx.x >> 6) * 12u + sl;
    if (lane >= 60u || c >= chunks) return;
    const double* wb = wsite + (size_t)b * kSiteBlock * kWStride + 2u * cl;
    const uint64_t j0 = start[b] + (uint64_t)c * kChunk;
    const uint64_t left = start[b + 1] - j0;
    const uint32_t len = left < kChunk ? (uint32_t)left : kChunk;
    const uint32_t* wp = word + j0;
    double* dst = psum + (size_t)cpiece[c0 + c] * 10 + 2u * cl;
    double a0 = 0.0, a1 = 0.0;
    constexpr uint32_t U = 8;
    Words<U> cur, next;
    cur.load(wp);
    uint32_t key = cur.w[0] >> 16;
    for (uint32_t j = 0; j < len; j += U) {
        // whatever a word past the chunk's end says, its row lies in the weights' blocks
        double2 x[U];
#pragma unroll
        for (uint32_t u = 0; u < U; u++)
            x[u] = *reinterpret_cast<const double2*>(wb + (size_t)(cur.w[u] & (kSiteBlock - 1u)) * kWStride);
        next.load(wp + j + U);
#pragma unroll
        for (uint32_t u = 0; u < U; u++) {
            if (j + u < len) {
                const uint32_t k = cur.w[u] >> 16;
                if (k != key) {
                    *reinterpret_cast<double2*>(dst) = make_double2(a0, a1);
                    dst += 10;
                    key = k;
                    a0 = a1 = 0.0;
                }
                a0 += x[u].x;
                a1 += x[u].y;
            }
        }
        cur = next;
    }
    *reinterpret_cast<double2*>(dst) = make_double2(a0, a1);
}

// a used key's pieces summed over part blockIdx.y of the site blocks, in order
__global__ __launch_bounds__(256) void k_adj_parts(const double* psum, const uint32_t* kpiece, uint32_t nuk,
                                                   uint32_t nblk, double* part)
{
    const uint32_t lane = __lane_id(), sl = lane / 5u, cl = lane - 5u * sl;
    const uint32_t i = (blockIdx.x * 4u + (threadIdx.x >> 6)) * 12u + sl;
    if (lane >= 60u || i >= nuk) return;
    const uint32_t b0 = (uint32_t)((uint64_t)nblk * blockIdx.y / kParts);
    const uint32_t b1 = (uint32_t)((uint64_t)nblk * (blockIdx.y + 1u) / kParts);
    double a0 = 0.0, a1 = 0.0;
#pragma unroll 4
    for (uint32_t b = b0; b < b1; b++) {
        const uint32_t* kp = kpiece + (size_t)b * (nuk + 1u) + i;
        for (uint32_t p = kp[0]; p < kp[1]; p++) {
            const double2 x = *reinterpret_cast<const double2*>(psum + (size_t)p * 10 + 2u * cl);
            a0 += x.x;
            a1 += x.y;
        }
    }
    *reinterpret_cast<double2*>(part + ((size_t)blockIdx.y * nuk + i) * 10 + 2u * cl) = make_double2(a0, a1);
}

// gradient of a used key's four entries, p_matrix layout q<<12 | c<<4 | a<<2 | o,
// from its ten sums: one division per genotype pair
__global__ __launch_bounds__(256) void k_adj_grad(const double* pm, const double* part, const uint32_t* ukey,
                                                  uint32_t nuk, double* grad)
{
    const uint32_t i = blockIdx.x * 256u + threadIdx.x;
    if (i >= nuk) return;
    double w[10];
#pragma unroll
    for (int g = 0; g < 10; g++) w[g] = 0.0;
    for (uint32_t y = 0; y < kParts; y++)
#pragma unroll
        for (int g = 0; g < 10; g++) w[g] += part[((size_t)y * nuk + i) * 10 + g];
    const uint32_t k = ukey[i], q = k >> 10, cyc = (k >> 2) & 255u, o = k & 3u;
    const size_t at = ((size_t)q << 12) + ((size_t)cyc << 4) + o;
    double pa[4], c[4] = {0.0, 0.0, 0.0, 0.0};
#pragma unroll
    for (int a = 0; a < 4; a++) pa[a] = pm[at + 4 * a];
    int g = 0;
#pragma unroll
    for (int a1 = 0; a1 < 4; a1++)
#pragma unroll
        for (int a2 = a1; a2 < 4; a2++) {
            if (a1 == a2) {
                c[a1] += w[g];
            } else {
                const double inv = 1.0 / (pa[a1] + pa[a2]);
                c[a1] += w[g] * (pa[a1] * inv);
                c[a2] += w[g] * (pa[a2] * inv);
            }
            g++;
        }
#pragma unroll
    for (int a = 0; a < 4; a++) grad[at + 4 * a] = c[a];
}

// fixed-order sums of two per-site arrays: 256-site block partials (fixed
// shuffle tree), then one block summing the partials in order
__global__ __launch_bounds__(256) void k_sum2_blocks(const double* x, const double* y, uint32_t n, double* part)
{
    __shared__ double sx[4], sy[4];
    const uint32_t i = blockIdx.x * 256u + threadIdx.x;
    double a = i < n ? x[i] : 0.0, b = i < n ? y[i] : 0.0;
    for (int off = 32; off > 0; off >>= 1) {
        a += __shfl_xor(a, off);
        b += __shfl_xor(b, off);
    }
    if (__lane_id() == 0) {
        sx[threadIdx.x >> 6] = a;
        sy[threadIdx.x >> 6] = b;
    }
    __syncthreads();
    if (threadIdx.x == 0) {
        part[2 * blockIdx.x] = (sx[0] + sx[1]) + (sx[2] + sx[3]);
        part[2 * blockIdx.x + 1] = (sy[0] + sy[1]) + (sy[2] + sy[3]);
    }
}

__global__ __launch_bounds__(1024) void k_sum2_final(const double* part, uint32_t nb, double* out)
{
    __shared__ double sx[16], sy[16];
    double a = 0.0, b = 0.0;
    for (uint32_t i = threadIdx.x; i < nb; i += 1024) {
        a += part[2 * i];
        b += part[2 * i + 1];
    }
    for (int off = 32; off > 0; off >>= 1) {
        a += __shfl_xor(a, off);
        b += __shfl_xor(b, off);
    }
    if (__lane_id() == 0) {
        sx[threadIdx.x >> 6] = a;
        sy[threadIdx.x >> 6] = b;
    }
    __syncthreads();
    if (threadIdx.x) return;
    for (int w = 1; w < 16; w++) {
        sx[0] += sx[w];
        sy[0] += sy[w];
    }
    out[0] = sx[0];
    out[1] = sy[0];
}

inline uint32_t blocks_for(uint64_t n) { return (uint32_t)((n + 255) / 256); }

}  // namespace

#define HIPCHK(x)                                                                                 \
    do {                                                                                          \
        hipError_t e_ = (x);                                                                      \
        if (e_ != hipSuccess) return fail(GSNP_E_DEVICE, std::string(#x) + ": " + hipGetErrorString(e_)); \
    } while (0)

// exclusive scan of n u32 counts into out[0, n] (out[n] = total)
static int scan_counts(Ctx& c, const uint32_t* in, uint32_t n, uint64_t* out)
{
    const uint32_t nb = blocks_for(n) ? blocks_for(n) : 1;
    if (c.adj_bsum.n < nb + 1) HIPCHK(c.adj_bsum.alloc(nb + 1));
    if (c.total.n < 1) HIPCHK(c.total.alloc(1));
    hipLaunchKernelGGL(k_scan_local, dim3(nb), dim3(256), 0, c.stream, in, n, out, c.adj_bsum.p);
    launch_scan_blocks(c.stream, c.adj_bsum.p, nb, c.total.p);
    hipLaunchKernelGGL(k_scan_add, dim3(blocks_for((uint64_t)n + 1)), dim3(256), 0, c.stream, out, n, c.adj_bsum.p,
                       c.total.p);
    HIPCHK(hipGetLastError());
    return GSNP_OK;
}

// a workspace of at least n elements, kept between spans; one that a much longer
// span left behind is given back
template <class T>
static hipError_t room(DevBuf<T>& b, size_t n)
{
    constexpr size_t kept = (size_t(4) << 20) / sizeof(T);  // 4 MB stay whatever the span
    return b.p && b.n >= n && (b.n <= kept || b.n / 4 <= n) ? hipSuccess : b.alloc(n);
}

}  // namespace gsnp

using namespace gsnp;

extern "C" int gsnp_adjoint_prepare(gsnp_ctx* c, uint32_t start, uint32_t n)
{
    if (!c) return fail(GSNP_E_ARG, "null context");
    if ((uint64_t)start + n > c->chr_len) return fail(GSNP_E_ARG, "span outside the chromosome");
    if (!c->n_reads && n) return fail(GSNP_E_ARG, "no reads loaded");
    int rc = c->alloc_window(n + 2);
    if (rc) return rc;
    c->adj_n = 0;
    hipStream_t st = c->stream;
    SiteArrays a = c->site_view(0);
    // site matrix of the span, and where each called site's words go
    launch_site_build(st, c->read_view(), 0, c->n_reads, start, n + 1, INT64_MIN, (int64_t)start + n, 0, a, nullptr,
                      c->ranges.p);
    HIPCHK(hipGetLastError());
    const uint32_t nblk = (n + kSiteBlock - 1) / kSiteBlock;
    HIPCHK(room(c->adj_cnt, (size_t)n + 1));
    HIPCHK(room(c->adj_prow, (size_t)n + 1));
    HIPCHK(room(c->adj_off, (size_t)n + 1));
    HIPCHK(room(c->adj_start_of, (size_t)nblk + 1));
    if (n)
        hipLaunchKernelGGL(k_adj_sites, dim3(blocks_for(n)), dim3(256), 0, st, c->tables(), c->ref_view(), start, a, n,
                           c->adj_cnt.p, c->adj_prow.p);
    rc = scan_counts(*c, c->adj_cnt.p, n, c->adj_off.p);
    if (rc) return rc;
    hipLaunchKernelGGL(k_block_starts, dim3(blocks_for((uint64_t)nblk + 1)), dim3(256), 0, st, c->adj_off.p, n, nblk,
                       c->adj_start_of.p);
    HIPCHK(hipGetLastError());
    std::vector<uint64_t> starts(nblk + 1);
    HIPCHK(hipMemcpyAsync(starts.data(), c->adj_start_of.p, 8ull * (nblk + 1), hipMemcpyDeviceToHost, st));
    HIPCHK(hipStreamSynchronize(st));
    if (starts[nblk] >= 0xFFFFFFFFull) return fail(GSNP_E_RANGE, "span holds too many records for one adjoint");
    const uint32_t nr = (uint32_t)starts[nblk];
    std::vector<uint32_t> hbase(nblk + 1, 0), cbase(nblk + 1, 0);
    uint32_t most = 0;  // radix chunks of a block
    for (uint32_t b = 0; b < nblk; b++) {
        const uint32_t chunks = (uint32_t)((starts[b + 1] - starts[b] + kRadixChunk - 1) / kRadixChunk);
        most = std::max(most, chunks);
        hbase[b + 1] = hbase[b] + 256u * chunks;
        cbase[b + 1] = cbase[b] + (uint32_t)((starts[b + 1] - starts[b] + kChunk - 1) / kChunk);
    }
    const uint32_t nh = hbase[nblk];
    // record words: every site's records sorted in registers, their adjusted qualities, stored as one word each
    HIPCHK(room(c->adj_word, (size_t)nr + kWordPad));
    HIPCHK(room(c->adj_sword, (size_t)nr + kWordPad));
    HIPCHK(room(c->adj_tmp, (size_t)nr + 1));
    HIPCHK(room(c->adj_hist, (size_t)nh + 1));
    HIPCHK(room(c->adj_hoff, (size_t)nh + 1));
    HIPCHK(room(c->adj_hbase, (size_t)nblk + 1));
    std::vector<uint2> work[8];
    for (uint32_t b = 0; b < nblk; b++)
        for (uint32_t k = 0; k < cbase[b + 1] - cbase[b]; k += kChunksPerGroup) work[b & 7u].push_back(make_uint2(b, k));
    size_t rounds = 0;
    for (const auto& w : work) rounds = std::max(rounds, w.size());
    std::vector<uint2> order(8 * rounds, make_uint2(0, 0xFFFFFF00u));  // no such chunk
    for (uint32_t x = 0; x < 8; x++)
        for (size_t k = 0; k < work[x].size(); k++) order[8 * k + x] = work[x][k];
    HIPCHK(room(c->adj_work, order.size() + 1));
    HIPCHK(hipMemcpyAsync(c->adj_work.p, order.data(), sizeof(uint2) * order.size(), hipMemcpyHostToDevice, st));
    HIPCHK(room(c->adj_cbase, (size_t)nblk + 1));
    HIPCHK(room(c->adj_cpiece, (size_t)cbase[nblk] + 1));
    HIPCHK(hipMemcpyAsync(c->adj_cbase.p, cbase.data(), 4ull * (nblk + 1), hipMemcpyHostToDevice, st));
    HIPCHK(hipMemcpyAsync(c->adj_hbase.p, hbase.data(), 4ull * (nblk + 1), hipMemcpyHostToDevice, st));
    launch_fill_u32(st, c->err.p, 1, 0u);
    if (nr) {
        launch_bucket(st, a.nrec, n, c->lists.p, c->win_cap, c->counts.p, 1, nullptr, (int)c->tune.min_class);
        FusedArgs f = c->fused_args(start);
        f.posterior = 0;
        f.key_words = c->adj_word.p;
        f.key_off = c->adj_off.p;
        f.key_block = kSiteBlock;
        launch_fused(st, f, c->lists.p, c->win_cap, c->counts.p, n, c->tune);
        for (uint32_t shift = 16; shift < 32; shift += 8) {
            const uint32_t* in = shift == 16 ? c->adj_word.p : c->adj_tmp.p;
            uint32_t* out = shift == 16 ? c->adj_tmp.p : c->adj_sword.p;
            hipLaunchKernelGGL(k_radix_hist, dim3(most, nblk), dim3(256), 0, st, in, c->adj_start_of.p, c->adj_hbase.p,
                               shift, c->adj_hist.p);
            rc = scan_counts(*c, c->adj_hist.p, nh, c->adj_hoff.p);
            if (rc) return rc;
            hipLaunchKernelGGL(k_radix_scatter, dim3(most, nblk), dim3(256), 0, st, in, c->adj_start_of.p, c->adj_hbase.p,
                               shift, c->adj_hoff.p, out);
        }
        HIPCHK(hipGetLastError());
    }
    // reduction pieces and the keys in use
    uint32_t* flag = c->adj_tmp.p;
    HIPCHK(room(c->adj_pidx, (size_t)nr + 1));
    HIPCHK(room(c->adj_used, kKeys));
    HIPCHK(room(c->adj_uidx, (size_t)kKeys + 1));
    launch_fill_u32(st, c->adj_used.p, kKeys, 0u);
    if (nr)
        hipLaunchKernelGGL(k_piece_flags, dim3(std::min(most * 16u, 1024u), nblk), dim3(256), 0, st, c->adj_sword.p,
                           c->adj_start_of.p, flag, c->adj_used.p);
    rc = scan_counts(*c, flag, nr, c->adj_pidx.p);
    if (!rc) rc = scan_counts(*c, c->adj_used.p, kKeys, c->adj_uidx.p);
    if (rc) return rc;
    uint64_t np = 0, nu = 0;
    uint32_t e = 0;
    HIPCHK(hipMemcpyAsync(&np, c->adj_pidx.p + nr, 8, hipMemcpyDeviceToHost, st));
    HIPCHK(hipMemcpyAsync(&nu, c->adj_uidx.p + kKeys, 8, hipMemcpyDeviceToHost, st));
    HIPCHK(hipMemcpyAsync(&e, c->err.p, 4, hipMemcpyDeviceToHost, st));
    HIPCHK(hipStreamSynchronize(st));
    if (e & kErrQadjRange) return fail(GSNP_E_RANGE, "adjusted quality exceeds the score table");
    if (e & kErrAdjQ) return fail(GSNP_E_RANGE, "adjusted quality of 64 or more: outside the gradient table");
    const uint32_t npieces = (uint32_t)np, nuk = (uint32_t)nu;
    HIPCHK(room(c->adj_pstart, (size_t)npieces + 1));
    HIPCHK(room(c->adj_pblock, (size_t)nblk + 1));
    HIPCHK(room(c->adj_ukey, (size_t)nuk + 1));
    HIPCHK(room(c->adj_kpiece, (size_t)nblk * (nuk + 1) + 1));
    hipLaunchKernelGGL(k_piece_starts, dim3(blocks_for(std::max<uint64_t>(nr, (uint64_t)nblk + 1))), dim3(256), 0, st, flag,
                       c->adj_pidx.p, nr, c->adj_start_of.p, nblk, c->adj_pstart.p, c->adj_pblock.p);
    hipLaunchKernelGGL(k_used_keys, dim3(blocks_for(kKeys)), dim3(256), 0, st, c->adj_used.p, c->adj_uidx.p, c->adj_ukey.p);
    if (nr)
        hipLaunchKernelGGL(k_chunk_pieces, dim3(blocks_for((uint64_t)most * (kRadixChunk / kChunk)), nblk), dim3(256), 0, st,
                           c->adj_pidx.p, c->adj_start_of.p, c->adj_cbase.p, c->adj_cpiece.p);
    if (nblk)
        hipLaunchKernelGGL(k_key_pieces, dim3(blocks_for((uint64_t)nuk + 1), nblk), dim3(256), 0, st, c->adj_sword.p,
                           c->adj_pstart.p, c->adj_pblock.p, c->adj_ukey.p, nuk, c->adj_kpiece.p);
    HIPCHK(hipGetLastError());
    // evaluation buffers; the entries of keys not in use stay 0
    HIPCHK(room(c->adj_T, (size_t)kKeys * kScoreRowStride));
    HIPCHK(room(c->adj_w, (size_t)nblk * kSiteBlock * kWStride + 1));
    HIPCHK(room(c->adj_ll, (size_t)n + 1));
    HIPCHK(room(c->adj_dh, (size_t)n + 1));
    HIPCHK(room(c->adj_psum, 10 * (size_t)npieces + 10));
    HIPCHK(room(c->adj_sums, 10 * (size_t)kParts * nuk + 10));
    HIPCHK(room(c->adj_part, 2 * (size_t)blocks_for(n) + 2));
    HIPCHK(room(c->adj_out, 2));
    HIPCHK(room(c->adj_pm, (size_t)64 * 256 * 16));
    HIPCHK(room(c->adj_grad, (size_t)64 * 256 * 16));
    launch_fill_u32(st, c->adj_grad.p, 2u * 64u * 256u * 16u, 0u);
    HIPCHK(hipGetLastError());
    HIPCHK(hipStreamSynchronize(st));
    c->adj_snps = c->h_snps;
    c->adj_snp_ref = c->h_snp_ref;
    c->adj_start = start;
    c->adj_n = n;
    c->adj_nrec = nr;
    c->adj_npieces = npieces;
    c->adj_nblk = nblk;
    c->adj_groups = (uint32_t)order.size();
    c->adj_nuk = nuk;
    return GSNP_OK;
}

// Prior rows (log10) at het rate exp(log_het): the 8 reference-code rows
// (cpp/prior.cc:3-43), then one row per known SNP (cpp/prior.cc:45-97); and
// per row the genotypes whose prior carries one factor of het.  The rows of a
// prepared span are those of the chromosome it was prepared on.
static const std::vector<gsnp_snp>& adjoint_snps(const Ctx& c) { return c.adj_n ? c.adj_snps : c.h_snps; }
static void adjoint_priors(const Ctx& c, double log_het, std::vector<double>& lp, std::vector<uint32_t>& mask)
{
    gsnp_params pp = c.p;
    pp.het_novel_r = std::exp(log_het);
    std::vector<double> prior(128);
    prior_gen(pp, prior.data());
    lp = log_prior_rows(prior.data());
    static const int kGenoCodes[10] = {0, 1, 2, 3, 5, 6, 7, 10, 11, 15};
    uint32_t het_bits = 0;
    for (int g = 0; g < 10; g++)
        if ((kGenoCodes[g] >> 2) != (kGenoCodes[g] & 3)) het_bits |= 1u << g;
    mask.assign(8, het_bits);
    const std::vector<gsnp_snp>& snps = adjoint_snps(c);
    const std::vector<uint8_t>& snp_ref = c.adj_n ? c.adj_snp_ref : c.h_snp_ref;
    const size_t nsnp = snps.size();
    lp.resize((8 + nsnp) * 10);
    mask.resize(8 + nsnp);
    for (size_t i = 0; i < nsnp; i++) {
        const gsnp_snp& sn = snps[i];
        snp_log_prior(pp, prior.data(), snp_ref[i], sn, &lp[(8 + i) * 10]);
        uint32_t m = 0;
        for (int g = 0; g < 10; g++) {
            const int a1 = kGenoCodes[g] >> 2, a2 = kGenoCodes[g] & 3;
            const bool replaced = !sn.indel && sn.freq[a1] > 0 && sn.freq[a2] > 0;
            if (a1 != a2 && !replaced) m |= 1u << g;
        }
        mask[8 + i] = m;
    }
}

extern "C" int gsnp_adjoint_eval(gsnp_ctx* c, const double* p_matrix, double log_het, double* loglik,
                                 double* grad_log_p, double* grad_log_het, double* site_loglik)
{
    if (!c || !p_matrix) return fail(GSNP_E_ARG, "null argument");
    if (!c->adj_n) return fail(GSNP_E_ARG, "gsnp_adjoint_prepare has not been called");
    const uint32_t n = c->adj_n;
    std::vector<double> lp;
    std::vector<uint32_t> mask;
    adjoint_priors(*c, log_het, lp, mask);
    if (c->adj_lp.n < lp.size()) HIPCHK(c->adj_lp.alloc(lp.size()));
    if (c->adj_mask.n < mask.size()) HIPCHK(c->adj_mask.alloc(mask.size()));
    hipStream_t st = c->stream;
    HIPCHK(hipMemcpyAsync(c->adj_lp.p, lp.data(), 8 * lp.size(), hipMemcpyHostToDevice, st));
    HIPCHK(hipMemcpyAsync(c->adj_mask.p, mask.data(), 4 * mask.size(), hipMemcpyHostToDevice, st));
    // the rows of qualities below 64: the objective uses no other
    HIPCHK(hipMemcpyAsync(c->adj_pm.p, p_matrix, 8ull * 64 * 256 * 16, hipMemcpyHostToDevice, st));
    c->timer.begin(kStAdjoint, st);
    hipLaunchKernelGGL(k_adj_table, dim3(blocks_for(kKeys)), dim3(256), 0, st, c->adj_pm.p, c->adj_T.p);
    if (n) {
        hipLaunchKernelGGL(k_adj_site, dim3((n + 4 * kAdjSitesPerWave - 1) / (4 * kAdjSitesPerWave)), dim3(256), 0, st,
                           c->adj_T.p, c->adj_word.p, c->adj_off.p,
                           c->adj_prow.p, c->adj_lp.p, c->adj_mask.p, n, c->p.is_monoploid, c->adj_ll.p, c->adj_dh.p,
                           c->adj_w.p);
    }
    if (c->adj_npieces) {
        const uint32_t nuk = c->adj_nuk;
        hipLaunchKernelGGL(k_adj_pieces, dim3(c->adj_groups), dim3(256), 0, st, c->adj_sword.p, c->adj_w.p,
                           c->adj_start_of.p, c->adj_cbase.p, c->adj_cpiece.p, c->adj_work.p, c->adj_psum.p);
        hipLaunchKernelGGL(k_adj_parts, dim3((nuk + 47u) / 48u, kParts), dim3(256), 0, st, c->adj_psum.p, c->adj_kpiece.p,
                           nuk, c->adj_nblk, c->adj_sums.p);
        hipLaunchKernelGGL(k_adj_grad, dim3(blocks_for(nuk)), dim3(256), 0, st, c->adj_pm.p, c->adj_sums.p, c->adj_ukey.p,
                           nuk, c->adj_grad.p);
    }
    const uint32_t nb = blocks_for(n) ? blocks_for(n) : 1;
    hipLaunchKernelGGL(k_sum2_blocks, dim3(nb), dim3(256), 0, st, c->adj_ll.p, c->adj_dh.p, n, c->adj_part.p);
    hipLaunchKernelGGL(k_sum2_final, dim3(1), dim3(1024), 0, st, c->adj_part.p, nb, c->adj_out.p);
    c->timer.end(kStAdjoint, st);
    HIPCHK(hipGetLastError());
    double out2[2];
    HIPCHK(hipMemcpyAsync(out2, c->adj_out.p, 16, hipMemcpyDeviceToHost, st));
    if (grad_log_p) HIPCHK(hipMemcpyAsync(grad_log_p, c->adj_grad.p, 8ull * 64 * 256 * 16, hipMemcpyDeviceToHost, st));
    if (site_loglik && n) HIPCHK(hipMemcpyAsync(site_loglik, c->adj_ll.p, 8ull * n, hipMemcpyDeviceToHost, st));
    HIPCHK(hipStreamSynchronize(st));
    if (loglik) *loglik = out2[0];
    if (grad_log_het) *grad_log_het = out2[1];
    return GSNP_OK;
}

extern "C" int gsnp_adjoint_info(gsnp_ctx* c, uint32_t* n_sites, uint64_t* n_records, uint32_t* n_prior_rows)
{
    if (!c) return fail(GSNP_E_ARG, "null context");
    if (n_sites) *n_sites = c->adj_n;
    if (n_records) *n_records = c->adj_nrec;
    if (n_prior_rows) *n_prior_rows = 8 + (uint32_t)adjoint_snps(*c).size();
    return GSNP_OK;
}

extern "C" int gsnp_adjoint_export(gsnp_ctx* c, uint32_t* keys, uint64_t* offsets, uint32_t* prior_row)
{
    if (!c) return fail(GSNP_E_ARG, "null context");
    if (!c->adj_n) return fail(GSNP_E_ARG, "gsnp_adjoint_prepare has not been called");
    const uint32_t n = c->adj_n;
    if (keys && c->adj_nrec)
        HIPCHK(hipMemcpyAsync(keys, c->adj_word.p, 4ull * c->adj_nrec, hipMemcpyDeviceToHost, c->stream));
    if (offsets) HIPCHK(hipMemcpyAsync(offsets, c->adj_off.p, 8ull * (n + 1), hipMemcpyDeviceToHost, c->stream));
    if (prior_row) HIPCHK(hipMemcpyAsync(prior_row, c->adj_prow.p, 4ull * n, hipMemcpyDeviceToHost, c->stream));
    HIPCHK(hipStreamSynchronize(c->stream));
    if (keys)
        for (uint64_t r = 0; r < c->adj_nrec; r++) keys[r] >>= 16;
    return GSNP_OK;
}

extern "C" int gsnp_adjoint_priors(gsnp_ctx* c, double log_het, double* lp10, uint32_t* het_mask, uint32_t cap_rows)
{
    if (!c) return fail(GSNP_E_ARG, "null context");
    std::vector<double> lp;
    std::vector<uint32_t> mask;
    adjoint_priors(*c, log_het, lp, mask);
    if (cap_rows < mask.size()) return fail(GSNP_E_ARG, "prior row buffer too small");
    if (lp10) std::memcpy(lp10, lp.data(), 8 * lp.size());
    if (het_mask) std::memcpy(het_mask, mask.data(), 4 * mask.size());
    return GSNP_OK;
}
