// calib.hip -- pass-1 calibration counts on the device (the counting loop of
// Prob_matrix::matrix_gen, cpp/matrix.cc:58-121): every base of a unique-hit
// read that was observed (A, C, G or T at or above the quality floor) and
// lies on a reference base that is neither N nor a known SNP counts once in
// the bin (quality, cycle, reference base, observed base).  The counts are
// exact integers, so the order of the additions does not matter; the matrix
// itself is then derived from them on the host (matrix_from_counts, a few
// thousand rows).
#include <hip/hip_runtime.h>

#include <algorithm>
#include <string>
#include <vector>

#include "../../include/gsnp_abi.h"
#include "engine.h"
#include "gsnp_common.h"

namespace gsnp {

namespace {

// Each workgroup counts one slice of 16 cycles over a range of reads into a
// private histogram in LDS -- 63 qualities x 16 (reference, observed) pairs x
// 16 cycles of 32-bit counters, 64,512 bytes -- and leaves it in its part of a
// workspace; k_calib_sum adds the parts of a bin.  Counting in LDS takes the
// per-base atomics (and their contention on the few bins of high-quality
// matches) off the device memory path.
//
// Bound by the instructions and line look-ups per base, so a lane takes four
// bases with one load from the read and one from the reference, and works on
// the four together until their bins.  With a lane per base, slices of a range
// on different XCDs and each bin added by every workgroup with a 64-bit
// atomic, 3 million reads of 150 bases took 0.81 ms; now 0.35.
constexpr uint32_t kSliceCycles = 16;
constexpr uint32_t kCalibQ = 63;  // q - q_min in [1, 63] on unique-hit bases
constexpr uint32_t kSliceBins = kCalibQ * kSliceCycles * 16;
constexpr uint32_t kCalibThreads = 1024;
constexpr uint32_t kCalibReads = kCalibThreads / 4;  // reads per step of a workgroup, four lanes each
constexpr uint32_t kCalibUnroll = 4;                 // steps whose loads are in flight together

typedef uint32_t Word1 __attribute__((aligned(1)));  // four bases at any address

// Workgroup 8 (slices g + y) + x of the grid counts cycles [16 y, 16 y + 16)
// over range 8 g + x of the reads: the slices of a range go to one XCD together,
// so that a line of reads comes to its L2 once for all of them.  Lane 4 r + k
// of a step takes cycles 16 y + 4 k + {0, 1, 2, 3} of read r.  The read store
// holds base << 6 | (64 - (q - q_min)) per base, 0 where the base was not
// observed.
//
// The LDS word of a bin is (64 - (q - q_min) - 1, pair, cycle in the slice), the
// pair as (ref ^ obs) << 2 | obs, so that the four matches, which take most of
// the counts, are pairs 0-3: with the cycle in the low bits, a wave's counts on
// the matching pairs spread over 64 banks, since its lanes start at different
// ones of their four bases.
__global__ __launch_bounds__(kCalibThreads) void k_calib_count(ReadView r, uint64_t n_reads, const uint8_t* ref,
                                                               uint32_t slices, uint32_t ranges, uint32_t* part)
{
    __shared__ uint32_t bins[kSliceBins];
    for (uint32_t i = threadIdx.x; i < kSliceBins; i += kCalibThreads) bins[i] = 0;
    __syncthreads();
    const uint32_t y = (blockIdx.x >> 3) % slices, range = ((blockIdx.x >> 3) / slices) * 8u + (blockIdx.x & 7u);
    const int32_t cyc = (int32_t)(y * kSliceCycles + 4u * (threadIdx.x & 3u));
    const uint32_t rot = (threadIdx.x >> 2) & 3u;
    uint32_t j[4];
#pragma unroll
    for (uint32_t t = 0; t < 4; t++) j[t] = 4u * (threadIdx.x & 3u) + ((t + rot) & 3u);
    const uint64_t stride = (uint64_t)ranges * kCalibReads * kCalibUnroll;
    for (uint64_t i0 = (uint64_t)range * kCalibReads * kCalibUnroll + (threadIdx.x >> 2); i0 < n_reads; i0 += stride) {
        uint32_t m[kCalibUnroll];
        int32_t p[kCalibUnroll];
#pragma unroll
        for (uint32_t u = 0; u < kCalibUnroll; u++) {
            const uint64_t i = i0 + u * kCalibReads;
            const uint64_t at = i < n_reads ? i : i0;
            m[u] = i < n_reads ? r.meta[at] : 0u;  // hit count 0: skipped
            p[u] = r.pos[at];
        }
        uint32_t b[kCalibUnroll], o[kCalibUnroll];
#pragma unroll
        for (uint32_t u = 0; u < kCalibUnroll; u++) {
            const int32_t len = (int32_t)rm_len(m[u]);
            const bool ok = rm_hit(m[u]) == 1 && cyc < len;
            // read coordinate of the four bases' first; up to three of them lie
            // past the read's end (in the padding of the read store and of the
            // reference), or before the first site
            const int32_t k = rm_strand(m[u]) ? len - 4 - cyc : cyc;
            const int64_t at = (int64_t)p[u] + k;
            b[u] = ok ? *reinterpret_cast<const Word1*>(r.seq + ((int64_t)(i0 + u * kCalibReads) * r.pitch + k)) : 0u;
            o[u] = ok ? *reinterpret_cast<const Word1*>(ref + (at < 0 ? 0 : at)) : 0u;
            o[u] <<= ok && at < 0 ? 8u * (uint32_t)-at : 0u;
        }
#pragma unroll
        for (uint32_t u = 0; u < kCalibUnroll; u++) {
            // in cycle order, those of cycles past the read's last cleared
            const uint32_t order = rm_strand(m[u]) ? 0x00010203u : 0x03020100u;
            const int32_t left = (int32_t)rm_len(m[u]) - cyc;
            uint32_t bw = __builtin_amdgcn_perm(b[u], b[u], order), ow = __builtin_amdgcn_perm(o[u], o[u], order);
            bw &= left >= 4 ? 0xFFFFFFFFu : left > 0 ? 0xFFFFFFFFu >> (32 - 8 * left) : 0u;
            bw = __builtin_amdgcn_alignbit(bw, bw, 8u * rot);
            ow = __builtin_amdgcn_alignbit(ow, ow, 8u * rot);
            const uint32_t obs = (bw >> 6) & 0x03030303u;
            const uint32_t pair = (((ow ^ obs) & 0x03030303u) << 2) | obs;
            // the quality field, above 63 where the reference is N or a known SNP
            const uint32_t qf = (bw & 0x3F3F3F3Fu) | ((ow & 0x0C0C0C0Cu) << 4);
#pragma unroll
            for (uint32_t t = 0; t < 4; t++) {
                const uint32_t q = ((qf >> (8u * t)) & 255u) - 1u;
                if (q < kCalibQ) atomicAdd(&bins[(((q << 4) | ((pair >> (8u * t)) & 15u)) << 4) | j[t]], 1u);
            }
        }
    }
    __syncthreads();
    uint32_t* mine = part + ((size_t)y * ranges + range) * kSliceBins;
    for (uint32_t i = threadIdx.x; i < kSliceBins; i += kCalibThreads) mine[i] = bins[i];
}

// counts[q << 12 | cycle << 4 | reference << 2 | observed] of every bin
__global__ __launch_bounds__(256) void k_calib_sum(const uint32_t* part, uint32_t slices, uint32_t ranges,
                                                   unsigned long long* hist)
{
    const uint32_t i = blockIdx.x * 256u + threadIdx.x;  // LDS word of slice blockIdx.y
    if (i >= 64u * 256u) return;
    const uint32_t y = blockIdx.y, f = i >> 8;  // 64 - (q - q_min) - 1; 63: q = 0, never counted
    const uint32_t pm = (i >> 4) & 15u, obs = pm & 3u, rb = (pm >> 2) ^ obs, cyc = y * kSliceCycles + (i & 15u);
    unsigned long long sum = 0;
    if (y < slices && f < kCalibQ) {
        const uint32_t* p = part + (size_t)y * ranges * kSliceBins + i;
#pragma unroll 8
        for (uint32_t k = 0; k < ranges; k++) sum += p[(size_t)k * kSliceBins];
    }
    hist[((63u - f) << 12) | (cyc << 4) | (rb << 2) | obs] = sum;
}

}  // namespace

#define HIPCHK(x)                                                                                 \
    do {                                                                                          \
        hipError_t e_ = (x);                                                                      \
        if (e_ != hipSuccess) return fail(GSNP_E_DEVICE, std::string(#x) + ": " + hipGetErrorString(e_)); \
    } while (0)

}  // namespace gsnp

extern "C" int gsnp_calib_count(gsnp_ctx* c, uint64_t* counts)
{
    using namespace gsnp;
    if (!c || !counts) return fail(GSNP_E_ARG, "null argument");
    if (!c->n_reads) return GSNP_OK;
    if (c->calib.n < (size_t)kCalibBins) HIPCHK(c->calib.alloc(kCalibBins));
    // two workgroups fit a CU's LDS, so at most 512 of them, which fill the device once
    const uint32_t slices = ((uint32_t)c->p.read_length + kSliceCycles - 1) / kSliceCycles;
    const uint64_t per_step = (uint64_t)kCalibReads * kCalibUnroll;
    const uint32_t steps = (uint32_t)((c->n_reads + per_step - 1) / per_step);
    const uint32_t ranges = std::min((steps + 7u) & ~7u, std::max(8u, 512u / slices & ~7u));
    const size_t words = (size_t)slices * ranges * kSliceBins;
    if (c->calib_part.n < words) HIPCHK(c->calib_part.alloc(words));
    c->timer.begin(kStCalib, c->stream);
    hipLaunchKernelGGL(k_calib_count, dim3(ranges * slices), dim3(kCalibThreads), 0, c->stream, c->read_view(), c->n_reads,
                       c->ref.p, slices, ranges, c->calib_part.p);
    hipLaunchKernelGGL(k_calib_sum, dim3(64, 16), dim3(256), 0, c->stream, c->calib_part.p, slices, ranges, c->calib.p);
    c->timer.end(kStCalib, c->stream);
    HIPCHK(hipGetLastError());
    std::vector<unsigned long long> h(kCalibBins);
    HIPCHK(hipMemcpyAsync(h.data(), c->calib.p, 8ull * kCalibBins, hipMemcpyDeviceToHost, c->stream));
    HIPCHK(hipStreamSynchronize(c->stream));
    for (uint32_t i = 0; i < kCalibBins; i++) counts[i] += h[i];
    return GSNP_OK;
}
