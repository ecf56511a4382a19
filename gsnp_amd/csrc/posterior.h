// posterior.h -- genotype call of one site from its ten log-likelihoods
// (kernel/posterior_kernel.cu:635-786 and the q_cns rules of :833-864).
// Shared by the kernels that hold a site's counters in memory and the ones
// that hold them in registers.
#pragma once

#include <hip/hip_runtime.h>

#include "gsnp_common.h"
#include "kernels.h"

namespace gsnp {

__device__ __forceinline__ int get4(const int4& v, uint32_t i)
{
    return i == 0 ? v.x : i == 1 ? v.y : i == 2 ? v.z : v.w;
}

// The counters of one site.
struct SiteVals {
    uint32_t ori;  // reference code
    int depth, dep_uni;
    int4 qs, cu, ca;
};

// First half of a call: the two bases, the genotype and its margin.
struct SiteCall {
    uint32_t base1, base2, type1;
    int qual1, qual2, qual3;
    double dtp;
    bool called;  // false: an N row without reads
    bool hom;
    bool next;  // the HET cap reads the next site's q_sum (a base code of 4..7)
};

// Priors are host-computed log10 rows: lpv(0..9) is the reference code's, and
// a known SNP at absolute position p has its own.
template <class LK, class LP>
__device__ __forceinline__ SiteCall call_site(const Tables& t, const RefView& ref, uint32_t p, const SiteVals& v, LK lkv,
                                              LP lpv)
{
    SiteCall c;
    const uint32_t ori = v.ori;
    c.called = !((ori & 4) && v.depth == 0);
    // base1/base2 and qual1..3 (>= keeps the later base on ties)
    uint32_t base1 = 0, base2 = 0;
    c.qual1 = -1, c.qual2 = -2, c.qual3 = -3;
    const int4 key = v.dep_uni ? v.qs : v.ca;
    int k1 = v.dep_uni ? -1 : 0, k2 = v.dep_uni ? -2 : 0, k3 = v.dep_uni ? -3 : 0;
#pragma unroll
    for (uint32_t i = 0; i < 4; i++) {
        const int x = get4(key, i);
        if (x >= k1) {
            k3 = k2;
            base2 = base1;
            k2 = k1;
            base1 = i;
            k1 = x;
        } else if (x >= k2) {
            k3 = k2;
            base2 = i;
            k2 = x;
        } else if (x >= k3) {
            k3 = x;
        }
    }
    if (k1 == 0)
        base1 = ori & 7;
    else if (k2 == 0 && base1 != (ori & 7))
        base2 = ori & 7;
    if (v.dep_uni) {
        c.qual1 = k1;
        c.qual2 = k2;
        c.qual3 = k3;
    }
    const double* own = nullptr;
    if ((ori & 8) && t.refine && ref.n_snp) {
        // the known SNPs of the site's 256-site block, then a search among them
        uint32_t lo = ref.snp_first[p >> 8], hi = ref.snp_first[(p >> 8) + 1];
        while (lo < hi) {
            uint32_t m = (lo + hi) >> 1;
            if (ref.snp_pos[m] < p)
                lo = m + 1;
            else
                hi = m;
        }
        if (lo < ref.n_snp && ref.snp_pos[lo] == p) own = ref.snp_lp + (size_t)lo * 10;
    }
    double lp[10];
#pragma unroll
    for (int g = 0; g < 10; g++) lp[g] = lpv(g);
    if (own) {
#pragma unroll
        for (int g = 0; g < 10; g++) lp[g] = own[g];
    }
    uint32_t type1 = 16, type2 = 16;
    double tp1 = 0.0, tp2 = 0.0;
#pragma unroll
    for (int g = 0; g < 10; g++) {
        const uint32_t gt = geno_code(g);
        if (t.monoploid && (gt >> 2) != (gt & 3)) continue;
        const double x = lkv(g) + lp[g];
        if (x >= tp1 || type1 == 16) {
            type2 = type1;
            tp2 = tp1;
            type1 = gt;
            tp1 = x;
        } else if (x >= tp2 || type2 == 16) {
            type2 = gt;
            tp2 = x;
        }
    }
    c.base1 = base1;
    c.base2 = base2;
    c.type1 = type1;
    c.dtp = tp1 - tp2;
    c.hom = (type1 & 3) == ((type1 >> 2) & 3);
    c.next = !c.hom && (base1 >= 4 || base2 >= 4);
    return c;
}

// Whether the site's call goes to k_rank.
__device__ __forceinline__ bool job_site(const Tables& t, const SiteVals& v, const SiteCall& c)
{
    return t.rank_mode && !c.hom && get4(v.cu, c.type1 & 3) != 0 && get4(v.cu, (c.type1 >> 2) & 3) != 0;
}

// Second half, for a called site: consensus quality with its caps, stored to
// the outputs, or (a het under the rank-sum mode) the site's job for k_rank.  nq is the next site's q_sum, read when
// c.next: q_sum is flat over sites, so base codes 4..7 read the next site --
// for the last site of a window, as it stands before the reads that start on
// the window boundary.
__device__ __forceinline__ void finish_site(const Tables& t, const SiteVals& v, const SiteCall& c, const int4& nq,
                                            uint32_t s, const Results& out, RankJob* jobs, uint32_t* job_count)
{
    const uint32_t base1 = c.base1, base2 = c.base2, type1 = c.type1;
    bool het_ok = false;
    if (!c.hom) {
        const uint32_t het = base1 < base2 ? (base1 << 2 | base2) : (base2 << 2 | base1);
        const int q_b1 = base1 < 4 ? get4(v.qs, base1) : get4(nq, base1 & 3);
        const int q_b2 = base2 < 4 ? get4(v.qs, base2) : get4(nq, base2 & 3);
        het_ok = q_b1 > 0 && q_b2 > 0 && type1 == het;
    }
    double rank = 1.0;
    int q_cns;
    if (t.rank_mode && !c.hom) {
        if (!job_site(t, v, c)) {
            rank = 0.0;
        } else {
            const uint32_t j = atomicAdd(job_count, 1u);
            // written as three words (a struct copy with byte fields would go through scratch)
            uint32_t* jw = reinterpret_cast<uint32_t*>(jobs + j);
            jw[0] = s;
            jw[1] = (type1 & 0xffu) | ((het_ok ? 1u : 0u) << 8);
            jw[2] = (uint32_t)(c.qual2 - c.qual3);
            jobs[j].dtp = c.dtp;
            out.base1[s] = (uint8_t)base1;
            out.base2[s] = (uint8_t)base2;
            out.type1[s] = (uint8_t)type1;
            return;  // rank and q_cns come from k_rank
        }
    }
    if (rank == 0.0)
        q_cns = 0;
    else
        q_cns = trunc_int_x86(10 * c.dtp + 0.0);  // 10*log10(1) == 0
    if (c.hom) {
        if (c.qual1 > 0 && base1 != (type1 & 3))
            q_cns = 0;
        else if (q_cns > c.qual1 - c.qual2)
            q_cns = c.qual1 - c.qual2;
    } else {
        if (het_ok) {
            if (q_cns > c.qual2 - c.qual3) q_cns = c.qual2 - c.qual3;
        } else {
            q_cns = 0;
        }
    }
    if (q_cns > 99) q_cns = 99;
    if (q_cns < 0) q_cns = 0;
    out.base1[s] = (uint8_t)base1;
    out.base2[s] = (uint8_t)base2;
    out.type1[s] = (uint8_t)type1;
    out.q_cns[s] = q_cns;
    out.rank[s] = rank;
}

}  // namespace gsnp
