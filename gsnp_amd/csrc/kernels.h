// kernels.h -- device buffers and launch wrappers of the calling kernels.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

namespace gsnp {

// Per-site counters, structure of arrays over a span of sites.
struct SiteArrays {
    uint32_t* rec = nullptr;  // [n][256] observation records, site-major
    int32_t* nrec = nullptr;  // records per site (== dep_uni)
    int32_t* depth = nullptr;
    int32_t* repeat = nullptr;
    int4* cu = nullptr;  // count_uni per base
    int4* qs = nullptr;  // q_sum per base
    int4* ca = nullptr;  // count_all per base
};

struct Tables {
    const double* score = nullptr;  // [256*256*4][10]
    const uint8_t* qadj = nullptr;  // [64][td][gd]
    int td = 1, gd = 1;
    int qadj_full = 1;  // no entry of q in [1,64) is above 255 (0 in the table)
    const double* lprior = nullptr;  // [8][10]
    const double* prank = nullptr;   // 64*64*2048
    int read_len = 100;
    int q_min = 64;
    int q_max_min = 40;
    int monoploid = 0;
    int refine = 0;
    int rank_mode = 0;
};

struct RefView {
    const uint8_t* code = nullptr;  // chromosome codes
    uint32_t len = 0;
    const uint32_t* snp_pos = nullptr;
    const double* snp_lp = nullptr;  // [n_snp][10]
    uint32_t n_snp = 0;
    const uint32_t* snp_first = nullptr;  // [len/256 + 2]: first known SNP at or after each 256-site block
};

constexpr uint32_t kReadBlock = 1024;  // sites per entry of ReadView::first
struct ReadView {
    uint64_t n = 0;                   // reads of the chromosome; with none, nothing below is read
    const uint64_t* first = nullptr;  // [len / kReadBlock + 3]: first read at or after each block of sites
    const int32_t* pos = nullptr;
    const uint32_t* meta = nullptr;
    const uint8_t* seq = nullptr;
    uint32_t pitch = 0;
};

struct Results {
    uint8_t* base1 = nullptr;
    uint8_t* base2 = nullptr;
    uint8_t* type1 = nullptr;
    int32_t* q_cns = nullptr;
    double* rank = nullptr;
    double* lk = nullptr;  // [n][10]
};

// A het call that needs the rank-sum test (filled by the posterior kernel).
struct RankJob {
    uint32_t site;
    uint8_t type1, het_ok, pad0, pad1;
    int32_t cap;
    double dtp;  // type_prob[type1] - type_prob[type2]
};

// A site whose value depends on a host-libm transcendental (normal tail, or a
// log10 within the guard band of an integer): the host recomputes it.
struct FixJob {
    uint32_t site;
    int32_t n1, n2;
    uint8_t het_ok, normal, pad0, pad1;
    int32_t cap;
    double T1, T2, dtp, table_rank;
};

struct GText;

struct RowCtx {
    const char* name = nullptr;
    int name_len = 0;
    uint32_t pos_base = 0;         // 1-based position of local site 0
    const uint32_t* gidx = nullptr;  // per site: entry of gtext (valid where the fast %#g path fails)
    const GText* gtext = nullptr;
};

// error flags written by kernels
enum : uint32_t { kErrQadjRange = 1u, kErrRecordOverflow = 2u, kErrAdjQ = 4u /* adjusted quality of 64 or more in the adjoint */ };

// Arguments of the fused sort + likelihood + posterior launch (batched form).
struct FusedArgs {
    Tables t;
    RefView ref;
    uint32_t ws = 0;
    SiteArrays a;
    const int4* head_qs = nullptr;
    Results out;
    RankJob* jobs = nullptr;
    uint32_t* job_count = nullptr;
    uint32_t* err = nullptr;
    int write_lk = 0;   // also store the ten log-likelihoods of each site
    int posterior = 1;  // call the sites (0: likelihoods only, for the per-window path)
    // caller-owned records (posterior 0): sorted rows written back, and the
    // list entries of the sites that are scored set to kScored; the others'
    // records are not all plain (k_likelihood's sites)
    int store = 0;
    // the adjoint's record words, each site's from key_off on (key_block: a power of two)
    uint32_t* key_words = nullptr;
    const uint64_t* key_off = nullptr;
    uint32_t key_block = 1;
};

// Launch shape of the fused stage: bucket classes below min_class run on
// min_class's network (the smallest bucket edge), and each class gets its
// waves per block (0: the most that fit 64 KB of LDS) and a grid cap.  The
// defaults are what gsnp_autotune picks on a 100 bp, 30x-mean contig of
// 8 Mb: sites of up to 8 records on the 16-wide network, four waves per
// block for that class and the wide ones, eight for the 32 and 64 classes.
struct FusedTune {
    uint32_t min_class = 1;
    uint32_t max_class = 5;  // no site is deeper
    uint32_t wpb[6] = {0, 4, 8, 8, 4, 4};
    uint32_t max_blocks[6] = {8192, 8192, 8192, 8192, 8192, 8192};
    uint32_t deep_blocks = 1024;  // the same for a span's tiles beyond the tile classes: mostly none, so a small grid
};

// Counters that many blocks add to lie this many words apart.
constexpr uint32_t kCountStride = 64;

// Arguments of the reads-to-calls launch over tiles of 64 sites (call.hip).
constexpr uint32_t kTileClasses = 5;         // at most 16, 32, 40, 64, 128 records a site; then the deep tiles
constexpr uint32_t kTileQtabMax = 17408;     // bytes of the adjusted-quality table that fit beside the waves' LDS
constexpr uint32_t kMaxTileReads = 512;  // eight chunks of 64
constexpr uint32_t kShallowReads = 128;  // the same for the classes up to 64 records
// Unique-hit reads a tile may have: of more, most share their anchor with
// another one, and a wave settles such reads one after the other, so that a few
// tiles of short reads outlast everything beside them.  36 bp reads, us: 16 kb at
// 8x with a thirtieth of it at 100x 319 without the limit, 262 with it; 1 Mb with
// a hundredth so deep 457 and 398, as much at 40x throughout 513 and 514 (with the
// limit at 127 a handful of its tiles went past the class, 581).  100 bp reads: 24
// contigs of 0.12 to 2.4 Mb with piles of repeats 10.4 ms as without it, 11.2 with a
// limit of 256 on all of a tile's reads.
__host__ __device__ inline uint32_t max_unique(uint32_t pitch) { return pitch / 2u + 192u; }
struct TileArgs {
    Tables t;
    RefView ref;
    ReadView reads;
    const uint64_t* range = nullptr;  // reads of each tile
    const uint8_t* qtab = nullptr;    // [64 - q][td][gd], 16-byte aligned; row 0 (empty slots) all 0
    uint32_t qtab_bytes = 0;          // a multiple of 16, at most kTileQtabMax
    const double* score = nullptr;    // [base][adjusted quality < 64][cycle < read length][16]
    uint32_t ws = 0;
    uint32_t n_sites = 0;   // sites called
    uint32_t n_built = 0;   // sites whose counters are stored (one more)
    SiteArrays a;
    int4* head_qs = nullptr;
    Results out;
    RankJob* jobs = nullptr;
    uint32_t* job_count = nullptr;
    unsigned long long* n_records = nullptr;
    int write_lk = 0;
};
// what the first launch of a span clears: window heads, class counters (the tiles' 8, kCountStride words apart, and the
// sites' in the first words), job counters
struct SpanClear {
    int4* head_qs = nullptr;
    uint32_t n_heads = 0;
    uint32_t* counts = nullptr;
    uint32_t *job_count = nullptr, *fix_count = nullptr;
};
void launch_span_clear(hipStream_t s, const SpanClear& clr);
hipError_t allow_tile_lds();  // once for each device, before the first launch there
// reads, class and class list (lists[class * pitch]) of each tile of 64 sites
void launch_tile_classes(hipStream_t s, const ReadView& r, uint32_t ws, uint32_t n_tiles, uint64_t* range,
                         uint32_t* lists, uint32_t pitch, const SpanClear& clr);
// the deepest class, a few long tiles, and the others
void launch_call_deepest(hipStream_t s, const TileArgs& f, const uint32_t* lists, uint32_t pitch,
                         const uint32_t* counts, uint32_t n_tiles);
void launch_call_tiles(hipStream_t s, const TileArgs& f, const uint32_t* lists, uint32_t pitch, const uint32_t* counts,
                       uint32_t n_tiles);
// the tiles beyond those classes: site matrix, then every called site of them
// sorted and called by the 256-record network
void launch_deep_tiles(hipStream_t s, const FusedArgs& f, const ReadView& r, const uint64_t* range, uint32_t n_built,
                       uint32_t n_sites, int4* head_qs, const uint32_t* tiles, const uint32_t* n_deep, uint32_t* sites,
                       uint32_t* site_count, uint32_t n_tiles, unsigned long long* n_records, const FusedTune& tune);

// score rows [base][adjusted quality < 64][cycle] from the table by quality, cycle, base
void launch_tile_scores(hipStream_t s, const double* score, double* tscore, uint32_t cycles);

void launch_fill_u32(hipStream_t s, void* p, uint32_t n_words, uint32_t v);

// range: 2 u64 per 64-site block (read interval of the block)
void launch_site_build(hipStream_t s, const ReadView& r, uint64_t r0, uint64_t r1, uint32_t ws, uint32_t n_sites,
                       int64_t lo_min, int64_t hi_max, uint32_t carry, const SiteArrays& a, int4* head_qs,
                       uint64_t* range);
void launch_bucket(hipStream_t s, const int32_t* nrec, uint32_t n_sites, uint32_t* lists, uint32_t list_pitch,
                   uint32_t* counts, int all, unsigned long long* n_records, int min_class = 0,
                   const uint32_t* skip = nullptr, bool clear = true);
// sort and likelihood of caller-owned records (rows of 256): counts (8 words)
// and lists are working memory; nothing happens when *skip (may be null) is set
void launch_sort_likelihood(hipStream_t s, const Tables& t, const SiteArrays& a, uint32_t n_sites, uint32_t* lists,
                            uint32_t list_pitch, uint32_t* counts, double* lk, uint32_t* err, const FusedTune& tune,
                            const uint32_t* skip);
void launch_posterior(hipStream_t s, const Tables& t, const RefView& ref, uint32_t ws, const SiteArrays& a,
                      uint32_t n_sites, const int4* head_qs, Results& out, RankJob* jobs, uint32_t* job_count);
void launch_fused(hipStream_t s, const FusedArgs& f, const uint32_t* lists, uint32_t list_pitch, const uint32_t* counts,
                  uint32_t max_sites, const FusedTune& tune);
void launch_fused_one(hipStream_t s, const FusedArgs& f, const uint32_t* lists, uint32_t list_pitch,
                      const uint32_t* counts, uint32_t max_sites, uint32_t cls, uint32_t wpb, uint32_t max_blocks);
// normal_count: incremented once per site whose normal approximation the
// device finished
void launch_rank(hipStream_t s, const Tables& t, const SiteArrays& a, const RankJob* jobs, const uint32_t* job_count,
                 uint32_t max_jobs, Results& out, FixJob* fixes, uint32_t* fix_count, unsigned long long* normal_count);
void launch_apply_fix(hipStream_t s, const FixJob* fixes, const double* rank, const int32_t* qcns, uint32_t n,
                      Results& out);
// row lengths and block sums; rows that need the exact %#g routine are listed
// in gtext (gcount must be zero on entry) for launch_gtext
void launch_rowlen(hipStream_t s, const RefView& ref, uint32_t ws, const SiteArrays& a, const Results& res,
                   uint32_t n_sites, RowCtx rc, uint32_t* gidx, GText* gtext, uint32_t* gcount, uint32_t* rowlen,
                   uint64_t* block_sum);
// exact %#g text of the listed rows; their lengths are added to rowlen and block_sum
void launch_gtext(hipStream_t s, const SiteArrays& a, const Results& res, uint32_t n_sites, GText* gtext,
                  const uint32_t* gcount, uint32_t* rowlen, uint64_t* block_sum);
void launch_scan_blocks(hipStream_t s, uint64_t* block_sum, uint32_t n_blocks, uint64_t* total);
void launch_format(hipStream_t s, const RefView& ref, uint32_t ws, const SiteArrays& a, const Results& res,
                   uint32_t n_sites, RowCtx rc, const uint32_t* rowlen, const uint64_t* block_off, char* out);
void launch_recycle(hipStream_t s, const SiteArrays& a, uint32_t win, uint32_t L);

constexpr uint32_t kRowBlock = 256;

}  // namespace gsnp
