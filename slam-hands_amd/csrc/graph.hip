// Proximity factors of the factor graph: CudaDroid::add_proximity_factors
// (cuda_slam/main.cu:1679-1779) up to the edge-state update. The distances
// of every (i, j) pair of the window come from one frame_distance launch and
// one read-back (the reference launches and synchronises per 1024 pairs,
// compute_frame_distances_batch, main.cu:1655-1676); the selection that
// follows (invalidation, NMS against existing edges, mandatory neighbour
// edges, greedy best-distance edges) is the reference's host logic, step for
// step, over a few hundred values.
#include <algorithm>
#include <cstdint>
#include <cstdlib>
#include <cstring>
#include <vector>

#include "slk_internal.hpp"

namespace slk {
namespace {

// pair k = (i - t0) * jrange + (j - t1): ii[k] = i, jj[k] = j
__global__ __launch_bounds__(256) void k_pairs(int* __restrict__ ii, int* __restrict__ jj, int t0,
                                               int t1, int jrange, int np) {
    const int k = blockIdx.x * blockDim.x + threadIdx.x;
    if (k >= np) return;
    ii[k] = t0 + k / jrange;
    jj[k] = t1 + k % jrange;
}

// The host logic of add_proximity_factors over the window's pairs. Pairs
// that a step invalidates or suppresses (the reference raises their distance
// to 1e6) are marked in a byte map, edges that exist in another, so the part
// that needs no distance (existing edges, mandatory neighbours) runs while the
// distances are computed, and the greedy step sorts only the pairs that are
// still open when it comes to their bucket of distances. For 200 keyframes and
// 2000 edges: 0.16 ms, half of it beside the GPU, against 0.6 ms with a hash
// set of edges and one sort of all candidates (one host core).
struct Selection {
    int t, t0, t1, rad, nms, jrange, np, lo, width;
    std::vector<unsigned char> gone;  // [np]
    // pairs (a, b) with a >= t0: [a - t0][b - lo]; others: after them, [b - t0][a - lo]
    std::vector<unsigned char> have;
    std::vector<int> es;

    Selection(int t_, int t0_, int t1_, int rad_, int nms_)
        : t(t_), t0(t0_), t1(t1_), rad(rad_), nms(nms_), jrange(t_ - t1_),
          np((t_ - t0_) * jrange), lo(std::max(0, std::min({t0_, t1_, t0_ - rad_ - 1}))),
          width(t_ - lo), gone(np, 0), have(2 * (size_t)(t_ - t0_) * width, 0) {}

    // of a pair whose larger index is in [t0, t) and whose other is in [lo, t)
    unsigned char& known(int a, int b) {
        return a >= t0 ? have[(size_t)(a - t0) * width + (b - lo)]
                       : have[(size_t)(t - t0 + b - t0) * width + (a - lo)];
    }
    // NMS around an edge (main.cu:1708-1726)
    void suppress(int i, int j) {
        if (nms < 0) return;
        const int r = std::max(std::min(std::abs(i - j) - 2, nms), 0);
        for (int i1 = std::max(i - r, t0); i1 <= std::min(i + r, t - 1); i1++) {
            const int w = r - std::abs(i1 - i);
            const int a = std::max(j - w, t1), b = std::min(j + w, t - 1);
            if (a <= b) std::memset(&gone[(size_t)(i1 - t0) * jrange + (a - t1)], 1, b - a + 1);
        }
    }
    void add(int i, int j) { es.insert(es.end(), {i, j, j, i}); }
    void existing(const int* ii, const int* jj, int n) {
        for (int e = 0; e < n; e++) {
            const int i = ii[e], j = jj[e];
            suppress(i, j);
            if (std::min(i, j) >= lo && std::max(i, j) >= t0 && std::max(i, j) < t) known(i, j) = 1;
        }
    }
    // mandatory neighbour edges (main.cu:1728-1736); the index is formed
    // without checking j >= t1, as in the reference
    void mandatory() {
        for (int i = t0; i < t; i++)
            for (int j = std::max(i - rad - 1, 0); j < i; j++) {
                if (!known(i, j)) add(i, j);
                const int idx = (i - t0) * jrange + (j - t1);
                if (idx >= 0 && idx < np) gone[idx] = 1;
            }
    }
    // greedy best-distance edges (main.cu:1738-1755). Ascending distance;
    // equal distances in pair order (the reference's std::sort leaves their
    // order unspecified). Pairs above thresh are skipped before the
    // max_factors test and suppression only raises distances, so visiting the
    // open pairs at or below thresh visits the same pairs in the same order;
    // from a thresh of 1e6 on, the value that suppression sets, it closes none.
    void greedy(const float* d, float thresh, int max_factors, int n_edges) {
        const bool closes = thresh < 1e6f;
        // (distance bits, pair): non-negative floats sort as their bits
        std::vector<uint64_t> cand;
        for (int i = t0; i < t; i++)
            for (int j = t1; j < t; j++) {
                const int k = (i - t0) * jrange + (j - t1);
                // too close in time or too far apart (main.cu:1702-1706)
                const float v = gone[k] || i - rad < j || d[k] > 100.0f ? 1e6f : d[k];
                if (!(v <= thresh)) continue;
                uint32_t bits;
                std::memcpy(&bits, &v, 4);
                cand.push_back((uint64_t)bits << 32 | (uint32_t)k);
            }
        constexpr int kBuckets = 1024;
        const float scale = kBuckets / std::max(std::min(thresh, 100.0f), 1e-30f);
        auto bucket = [&](uint64_t c) {
            const uint32_t bits = (uint32_t)(c >> 32);
            float v;
            std::memcpy(&v, &bits, 4);
            return (int)std::min(v * scale, (float)(kBuckets - 1));
        };
        std::vector<int> first(kBuckets + 1, 0);
        for (uint64_t c : cand) first[bucket(c) + 1]++;
        for (int q = 0; q < kBuckets; q++) first[q + 1] += first[q];
        std::vector<uint64_t> open(cand.size());
        {
            std::vector<int> fill(first.begin(), first.end() - 1);
            for (uint64_t c : cand) open[fill[bucket(c)]++] = c;
        }
        for (int q = 0; q < kBuckets; q++) {
            uint64_t* s = open.data() + first[q];
            int n = 0;
            for (int m = 0; m < first[q + 1] - first[q]; m++)
                if (!closes || !gone[(uint32_t)s[m]]) s[n++] = s[m];
            std::sort(s, s + n);
            for (int m = 0; m < n; m++) {
                const int k = (int)(uint32_t)s[m];
                if (closes && gone[k]) continue;
                if (max_factors > 0 && n_edges + (int)es.size() / 2 > max_factors) return;
                const int i = t0 + k / jrange, j = t1 + k % jrange;
                add(i, j);
                suppress(i, j);
            }
        }
    }
};

}  // namespace
}  // namespace slk

using namespace slk;

extern "C" int slk_proximity_factors(slk_ctx* ctx, const float* poses, const float* disps,
                                     const float* intrinsics, int num_keyframes, int t0, int t1,
                                     int rad, int nms, float thresh, float beta,
                                     const int* ii_host, const int* jj_host, int n_edges,
                                     const int* ii_inac_host, const int* jj_inac_host,
                                     int n_inac, int max_factors, int* new_ii_host,
                                     int* new_jj_host, int capacity, int* n_new, int* n_es,
                                     float* dists_host, hipStream_t stream) {
    if (!ctx || !n_new || !n_es) return fail(SLK_E_ARG, "proximity_factors: null argument");
    *n_new = 0;
    *n_es = 0;
    if (n_edges < 0 || n_inac < 0 || (n_edges > 0 && (!ii_host || !jj_host)) ||
        (n_inac > 0 && (!ii_inac_host || !jj_inac_host)))
        return fail(SLK_E_ARG, "proximity_factors: bad edge lists");
    const int t = num_keyframes;
    if (t < 2) return SLK_OK;  // main.cu:1682
    t0 = std::max(0, t0);
    t1 = std::max(0, t1);
    // 1. distances of all pairs i in [t0, t), j in [t1, t) (main.cu:1686-1697)
    const int irange = std::max(0, t - t0), jrange = std::max(0, t - t1);
    const int np = irange * jrange;
    if (np == 0) return SLK_OK;  // main.cu:1694-1695
    if (!poses || !disps || !intrinsics) return fail(SLK_E_ARG, "proximity_factors: null state");
    SLK_TRY(ctx->graph_pairs.ensure((size_t)np * 2 * sizeof(int)));
    SLK_TRY(ctx->graph_dist.ensure((size_t)np * sizeof(float)));
    int* d_ii = ctx->graph_pairs.as<int>();
    int* d_jj = d_ii + np;
    hipLaunchKernelGGL(k_pairs, dim3((np + 255) / 256), dim3(256), 0, stream, d_ii, d_jj, t0, t1,
                       jrange, np);
    SLK_HIP(hipGetLastError());
    SLK_TRY(slk_frame_distance(poses, disps, intrinsics, d_ii, d_jj,
                               ctx->graph_dist.as<float>(), np, ctx->h, ctx->w, beta, stream));
    SLK_TRY(ctx->glue_stage.ensure((size_t)np * sizeof(float)));
    float* d = static_cast<float*>(ctx->glue_stage.ptr);
    SLK_HIP(hipMemcpyAsync(d, ctx->graph_dist.ptr, np * sizeof(float), hipMemcpyDeviceToHost,
                           stream));
    // 2., 3. what the existing edges close, and the mandatory ones
    Selection sel(t, t0, t1, rad, nms);
    sel.existing(ii_host, jj_host, n_edges);
    sel.existing(ii_inac_host, jj_inac_host, n_inac);
    sel.mandatory();
    SLK_HIP(hipStreamSynchronize(stream));
    if (dists_host) std::copy(d, d + np, dists_host);
    // 4. greedy best-distance edges
    sel.greedy(d, thresh, max_factors, n_edges);
    const std::vector<int>& es = sel.es;
    *n_es = (int)es.size() / 2;
    // 6. the edges the update appends: those not present yet, each once
    // (main.cu:1773-1781; the age-based removal in between moves edges from
    // the active to the inactive list, which has_edge treats alike)
    int m = 0;
    for (size_t q = 0; q < es.size(); q += 2) {
        const int i = es[q], j = es[q + 1];
        unsigned char& known = sel.known(i, j);  // has_edge (main.cu:786-792)
        if (known) continue;
        known = 1;
        if (m < capacity && new_ii_host && new_jj_host) {
            new_ii_host[m] = i;
            new_jj_host[m] = j;
        }
        m++;
    }
    *n_new = m;
    if (m > capacity)
        return fail(SLK_E_ARG, "proximity_factors: more new edges than capacity (see n_new)");
    return SLK_OK;
}
