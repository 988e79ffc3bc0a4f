// cuslines_hip.hip -- gfx950 kernels and C ABI of the per-seed tracking hot
// path: bootstrap (OPDT/CSA), probabilistic and PTT direction getters, the
// stepping loop and the two-phase seed protocol of dipy/GPUStreamlines.
//
// Layout in HBM (one tracker):
//   prob/boot data  float [X][Y][Z][T32]   channels padded to a multiple of
//                                          32 so each half-wave gather of 32
//                                          channels is one aligned 128-B line
//   PTT ODF         float [V][X][Y][Z]     vertex-major: the 8 texels of one
//                                          probe tap share z-adjacent lines
//   stop map        float [X][Y][Z]
//   sphere          float [V][3], edges packed (u | v << 16)
//   LUT             uint16 [R][R][R]       nearest sphere vertex
//
// Execution model: wave64, two seed slots per wave (one per 32-lane half).
// The 32 lanes of a slot hold the reference's 32 per-lane random streams and
// reproduce its reduction orders, so the results are bit-identical to the
// CPU oracle (oracle/cuslines_oracle.cpp) on the same inputs.
#include "device_math.h"

#include "../../include/cuslines_hip.h"

#include <rocprofiler-sdk-roctx/roctx.h>

#include <algorithm>
#include <cmath>
#include <cstdio>
#include <cstring>
#include <mutex>
#include <string>
#include <vector>

using namespace cusl;

namespace {

constexpr double PMF_THRESHOLD_P = 0.05;               // _globals.py:4
constexpr float REAL_MAX = 3.40282346638528859812e+38f;
constexpr float REAL_MIN = -REAL_MAX;                  // globals.h:41-42
constexpr float K_SMALL = 0.0001f;                     // ptt.cuh:10
constexpr float PTT_NORM_EPS = 1e-8f;                  // ptt.cuh:12
constexpr float PTT_MIN_NORM2 = 1e-16f;                // (1/PTT_INV_NORM_EPS)^2, ptt.cuh:13
constexpr float CSA_C0 = 0.28209479177387814f;         // boot.cu:363
constexpr int DISC_VERT_CNT = 24;                      // disc.h:20
constexpr int DISC_FACE_CNT = 31;                      // disc.h:21
constexpr int XCDS = 8;
constexpr int SEED_CLASSES = 8;                          // by direction count; the last has none and is not queued
constexpr int QUEUES = XCDS * (SEED_CLASSES - 1);        // persistent-queue counters, one per class and XCD
constexpr int WORK_INTS = QUEUES + SEED_CLASSES;         // counters, then where each class starts in the seed order
constexpr int VPROP_K = 24 * 9;                        // PTT table: curvatures after the 24 propagators
constexpr int VPROP_FLOATS = VPROP_K + 2 * 24;

// PTT disc tables (quality 2): numeric data of cuslines/cuda_c/disc.h:20-84
// (nibrary, BSD-3-Clause, Copyright (c) 2024 Dogu Baran Aydogan).
__constant__ float c_disc_vert[DISC_VERT_CNT * 2] = {
    -0.99680788f, -0.07983759f, -0.94276539f, 0.33345677f, -0.87928469f, -0.47629658f,
    -0.72856617f, 0.68497542f,  -0.60006556f, -0.79995082f, -0.54129995f, -0.02761342f,
    -0.39271207f, 0.37117272f,  -0.39217391f, 0.91989110f,  -0.36362884f, -0.40757367f,
    -0.22391316f, -0.97460910f, -0.00130022f, 0.53966106f,  0.00000000f,  0.00000000f,
    0.00973999f,  0.99995257f,  0.01606516f,  -0.54289908f, 0.21342395f,  -0.97695968f,
    0.38192071f,  -0.38666136f, 0.38897094f,  0.37442837f,  0.40696681f,  0.91344295f,
    0.54387161f,  -0.01477123f, 0.59119367f,  -0.80652963f, 0.73955688f,  0.67309406f,
    0.87601150f,  -0.48229022f, 0.94617928f,  0.32364298f,  0.99585368f,  -0.09096944f};
__constant__ int c_disc_face[DISC_FACE_CNT * 3] = {
    9, 8, 4,    11, 16, 10, 5, 8, 11,   5, 1, 0,    18, 16, 11, 11, 15, 18, 13, 8, 9,  11, 8, 13,
    13, 15, 11, 22, 18, 23, 22, 20, 16, 16, 18, 22, 16, 20, 17, 12, 10, 17, 17, 10, 16, 15, 19, 21,
    23, 18, 21, 21, 18, 15, 2, 4, 8,    2, 5, 0,    8, 5, 2,    7, 10, 12,  6, 7, 3,    10, 7, 6,
    3, 1, 6,    1, 5, 6,    11, 10, 6,  6, 5, 11,   14, 19, 15, 15, 13, 14, 14, 13, 9};

struct DevParams {
    int dimx, dimy, dimz, dimt, t32;
    int nverts, nv32, nedges, sphere_symm, max_sline_len, model;
    int hr, hr32, delta_nr;
    int hr16, dn16, nv16;  // batched bootstrap: hr, delta_nr, nverts rounded up to 16
    uint32_t seed_lo, seed_hi;
    float tc_threshold, rel_peak, cos_max_angle, cos_min_sep, min_signal;
    double step_d;
    // PTT
    int step_frac, probe_quality, lut_res, nx, ny, nz, log2x, log2y;
    float probe_step, max_curv, min_support_f, ptt_seed_thr_f;
    float ptt_sub_step;  // (float)(STEP_SIZE / STEP_FRAC)
    int lut_brick;               // PTT LUT stored as 4x4x4 bricks
    int ptt_nonneg;              // PTT ODF has no negative value: rejection rounds may stop early
    uint32_t rec_thresh;  // record a sub-step when its hash is below this
    int rec_cap;          // capacity of the pair buffer
    int slot_cap;         // bounded chunk: phase 2 skips seeds whose streamlines end past this slot (0: none)
    int rk16;             // batched bootstrap: rank of H rounded up to 16 when H.d = U (U^T d) (0: [H; R] product)
};

struct DevBufs {
    const float *data;
    const float *stop;
    const float *verts;
    const uint32_t *edges;
    const uint16_t *nbr;  // [nverts][8] neighbours, padded with the vertex itself (nullptr: edge path)
    const float *H, *R, *db, *dq, *smat;
    const float *hr_mat, *fit_mat, *odf_mat;  // batched bootstrap: [H;R], [dq|-db], smat, zero padded
    const float *ut_mat, *u_mat, *invlev;      // batched bootstrap, low-rank form: U^T, U, 1/sqrt(1 - H_ii)
    const int *b0;
    const int *dwi_idx;
    const uint32_t *lut;  // PTT LUT entry: vertex | (direction rank << 16)
    const float *blocks;  // PTT corner blocks (nullptr: gather 8 texels)
    const float *fprop;    // learned proposal: per disc vertex, propagator of 4 probe steps [24][9]
    const float *vprop;    // PTT: per disc vertex, propagator of one probe step [24][9], then (k1, k2) [24][2]
    const uint16_t *mlp;   // proposal network, bf16, lane-interleaved (IL_NPARAM)
    float *rec;            // training pairs [rec_cap][PAIR_FLOATS]
    int *rec_count;
    unsigned long long *stats;  // learned sub-steps, fallbacks, plain sub-steps
};

// Queue k of an XCD's order: its counter and its range [lo, hi) of the seed
// order.  The seeds with the most directions come first, each class in
// spatial order and split in one range per XCD: an XCD drains its own range
// (one region of the volume, for its L2), helps with the others', and goes on
// to the next class.  A seed is tracked by one slot, direction after
// direction on one random stream, and most of a run of a few seeds per slot
// is the wait for the seeds that take longest; those now start first
// (25,000 seeds on 6,144 slots of equal speed: 3,284 instead of 4,376 steps;
// the longest seed has 3,284).
struct QueueRange {
    int counter, lo, hi;
};

__device__ __forceinline__ QueueRange queue_range(const int *work, int k) {
    const int cls = k / XCDS, x = ((int)blockIdx.x + k) & (XCDS - 1);
    const int a = work[QUEUES + cls], b = work[QUEUES + cls + 1];
    QueueRange q;
    q.counter = cls * XCDS + x;
    q.lo = a + (int)((long long)(b - a) * x / XCDS);
    q.hi = a + (int)((long long)(b - a) * (x + 1) / XCDS);
    return q;
}

// -------------------------------------------------------------------------
// Sorting, scans and peak extraction (per half-wave)
// -------------------------------------------------------------------------

// warp_sort<32,32,WSORT_DIR_DEC> (cuwsort.cuh:104-168) on (key, value): Knuth's
// merge exchange (TAOCP 5.2.2 Algorithm M) for 32 keys, the network of the
// reference's tables (cuwsort.cuh:37-52; the same comparators in the same
// order on every wire, so ties end where the tables put them).  One pass:
// lanes i with i & P == R compare with i + D.
template <int P, int R, int D>
__device__ __forceinline__ void sort_pass(float &k, int &v) {
    const int g = lane32();
    const bool lo = (g & P) == R && g + D < 32, hi = g >= D && ((g - D) & P) == R;
    const int src = lo ? g + D : hi ? g - D : g;
    const float a = shfl32(k, src);
    const int b = shfl32(v, src);
    if (lo ? (a > k) : (a < k)) { k = a; v = b; }
}

// n keys, the lanes past them at the lowest value: a comparator that reaches a
// lane past the keys finds it in order, so 16 keys need 10 of the 15 passes
// and 8 need 6.
__device__ __forceinline__ void sort_dec(float &k, int &v, int n) {
    const bool n16 = n > 16, n8 = n > 8;
    if (n16) sort_pass<16, 0, 16>(k, v);
    if (n8) sort_pass<8, 0, 8>(k, v);
    if (n16) sort_pass<8, 8, 8>(k, v);
    sort_pass<4, 0, 4>(k, v);
    if (n16) sort_pass<4, 4, 12>(k, v);
    if (n8) sort_pass<4, 4, 4>(k, v);
    sort_pass<2, 0, 2>(k, v);
    if (n16) sort_pass<2, 2, 14>(k, v);
    if (n8) sort_pass<2, 2, 6>(k, v);
    sort_pass<2, 2, 2>(k, v);
    sort_pass<1, 0, 1>(k, v);
    if (n16) sort_pass<1, 1, 15>(k, v);
    if (n8) sort_pass<1, 1, 7>(k, v);
    sort_pass<1, 1, 3>(k, v);
    sort_pass<1, 1, 1>(k, v);
}

// prefix_sum_sh_d (utils.cu:81-120): blocks of 32, lane 0 adds the previous
// block's last value, Hillis-Steele inside the block.
__device__ void prefix_sum(float *a, int len) {
    const int l = lane32();
    float carry = 0.0f;
    for (int j = 0; j < len; j += 32) {
        float v = (j + l < len) ? a[j + l] : 0.0f;
        if (j != 0 && l == 0) v = v + carry;
#pragma unroll
        for (int i = 1; i < 32; i <<= 1) {
            const float o = shfl_up32(v, i);
            if (l >= i && j + l < len) v = v + o;
        }
        if (j + l < len) a[j + l] = v;
        carry = shfl32(v, 31);
    }
    WAVE_SYNC();
}

// peak_directions_d (tracking_helpers.cu:75-245).  odf, marks and cand are
// this slot's LDS arrays; the kept vertex indices end in cand[0..return).
// marks holds 2 bits per vertex, 16 vertices per word: bit 1 "has a strictly
// larger neighbour", bit 0 "has a strictly smaller one"; the reference's
// positive mark is exactly "bit 0 only".
__device__ __forceinline__ uint32_t peak_mark(const uint32_t *marks, int j) {
    return (marks[j >> 4] >> (2 * (j & 15))) & 3u;
}

// What the peak search reads of the parameters and buffers: few enough to be
// passed to its out-of-line forms.
struct SepParams {
    int sphere_symm;
    float cos_min_sep;
};
struct PeakParams {
    int nverts, nedges;
    float rel_peak;
    SepParams sep;
    const uint16_t *nbr;
    const uint32_t *edges;
};

__device__ __forceinline__ SepParams sep_params(const DevParams &P) { return SepParams{P.sphere_symm, P.cos_min_sep}; }
__device__ __forceinline__ PeakParams peak_params(const DevParams &P, const DevBufs &B) {
    return PeakParams{P.nverts, P.nedges, P.rel_peak, sep_params(P), B.nbr, B.edges};
}

__device__ int sort_dedup_peaks(const SepParams &P, const float *odf, uint16_t *cand, const float *sv, int n);
__device__ __noinline__ int bb_tail(SepParams P, const float *odf, uint16_t *cand, const float *verts, int n);

// CALL: the tail out of line.
template <bool CALL = false>
__device__ int peak_directions(const PeakParams &P, const float *odf, uint32_t *marks, uint16_t *cand, const float *sv) {
    const int l = lane32();
    const int nv = P.nverts;
    float mn = REAL_MAX;
    for (int j = l; j < nv; j += 32) mn = (mn < odf[j]) ? mn : odf[j];
    mn = min32(mn);
    mn = (0.0f > mn) ? 0.0f : mn;
    if (P.nbr) {
        // Vertex-centred form of the edge marks below: a vertex is a peak when
        // some neighbour is strictly smaller and none strictly larger, i.e.
        // when the smallest neighbour is below it and the largest not above
        // it (fminf / fmaxf pass over a NaN neighbour as the comparisons do).
        // Bit r of pk: vertex l + 32 r (nverts <= 1024).  Groups of 4
        // vertices per lane: the 4 adjacency rows are loaded before the first
        // is used, so their latencies overlap.
        uint32_t pk = 0u;
        float m = REAL_MIN;
        for (int r0 = 0, j0 = l; j0 < nv; r0 += 4, j0 += 128) {
            uint4 qs[4];
#pragma unroll
            for (int u = 0; u < 4; ++u)
                qs[u] = reinterpret_cast<const uint4 *>(P.nbr)[min(j0 + 32 * u, nv - 1)];  // past the end: dropped
#pragma unroll
            for (int u = 0; u < 4; ++u) {
                const int j = j0 + 32 * u;
                if (j >= nv) break;
                const uint32_t w[4] = {qs[u].x, qs[u].y, qs[u].z, qs[u].w};
                const float x = odf[j];
                float lo = odf[w[0] & 0xffffu], hi = lo;
#pragma unroll
                for (int k = 1; k < 8; ++k) {
                    const float y = odf[(w[k >> 1] >> (16 * (k & 1))) & 0xffffu];
                    lo = fminf(lo, y);
                    hi = fmaxf(hi, y);
                }
                if (lo < x && !(hi > x)) {
                    pk |= 1u << (r0 + u);
                    const float xm = x + (-mn);
                    m = (m > xm) ? m : xm;
                }
            }
        }
        m = max32(m);
        const float comp = (float)((double)P.rel_peak * (double)m);
        int n = 0;
        for (int r = 0, j0 = 0; j0 < nv; ++r, j0 += 32) {
            const int j = j0 + l;
            const bool keep = (j < nv) && ((pk >> r) & 1u) && ((odf[j] - mn) >= comp);
            const uint32_t msk = half_ballot(keep);
            if (keep) cand[n + __popc(msk & ((1u << l) - 1u))] = (uint16_t)j;
            n += __popc(msk);
        }
        WAVE_SYNC();
        return CALL ? bb_tail(P.sep, odf, cand, sv, n) : sort_dedup_peaks(P.sep, odf, cand, sv, n);
    }
    for (int w = l; w < (nv + 15) >> 4; w += 32) marks[w] = 0u;
    WAVE_SYNC();
    for (int e = l; e < P.nedges; e += 32) {
        const uint32_t uv = P.edges[e];
        const int u = (int)(uv & 0xffffu), v = (int)(uv >> 16);
        const float a = odf[u], b = odf[v];
        if (a < b) {
            atomicOr(&marks[u >> 4], 2u << (2 * (u & 15)));
            atomicOr(&marks[v >> 4], 1u << (2 * (v & 15)));
        } else if (b < a) {
            atomicOr(&marks[v >> 4], 2u << (2 * (v & 15)));
            atomicOr(&marks[u >> 4], 1u << (2 * (u & 15)));
        }
    }
    WAVE_SYNC();
    float m = REAL_MIN;
    for (int j = l; j < nv; j += 32)
        if (peak_mark(marks, j) == 1u) { const float x = odf[j] + (-mn); m = (m > x) ? m : x; }
    m = max32(m);
    const float comp = (float)((double)P.rel_peak * (double)m);
    int n = 0;
    for (int j0 = 0; j0 < nv; j0 += 32) {
        const int j = j0 + l;
        const bool keep = (j < nv) && (peak_mark(marks, j) == 1u) && ((odf[j] - mn) >= comp);
        const uint32_t msk = half_ballot(keep);
        if (keep) cand[n + __popc(msk & ((1u << l) - 1u))] = (uint16_t)j;
        n += __popc(msk);
    }
    WAVE_SYNC();
    return CALL ? bb_tail(P.sep, odf, cand, sv, n) : sort_dedup_peaks(P.sep, odf, cand, sv, n);
}

// The tail of peak_directions_d (tracking_helpers.cu:182-245) on the n
// candidates in cand: descending sort when n < 32, then the greedy
// minimum-separation filter.
__device__ int sort_dedup_peaks(const SepParams &P, const float *odf, uint16_t *cand, const float *sv, int n) {
    const int l = lane32();
    if (n == 0) return 0;
    if (n <= 32) {
        int ci = (l < n) ? cand[l] : 0;
        if (n < 32) {
            float k = (l < n) ? odf[ci] : REAL_MIN;
            sort_dec(k, ci, half_ballot(k < REAL_MIN) ? 32 : n);
        }
        // remove_similar_vertices (tracking_helpers.cu:195-223) on 32 lanes:
        // lane i holds candidate i's direction and marks which earlier
        // candidates j lie within the minimum separation (the same dot
        // product and test as the greedy loop below).  Candidate i is kept
        // iff none of its marked candidates is: each round decides those
        // whose marked candidates are all decided, a few rounds instead of
        // one step per candidate.  Four directions are read at a time.
        float ax = 0.0f, ay = 0.0f, az = 0.0f;
        if (l < n) { ax = sv[3 * ci]; ay = sv[3 * ci + 1]; az = sv[3 * ci + 2]; }
        uint32_t conf = 0u;
        for (int j0 = 0; j0 < n - 1; j0 += 4) {
            float bx[4], by[4], bz[4];
#pragma unroll
            for (int u = 0; u < 4; ++u) {  // lanes past n - 2 hold nothing that is marked
                bx[u] = shfl32(ax, (j0 + u) & 31);
                by[u] = shfl32(ay, (j0 + u) & 31);
                bz[u] = shfl32(az, (j0 + u) & 31);
            }
#pragma unroll
            for (int u = 0; u < 4; ++u) {
                float c = dot3(ax, ay, az, bx[u], by[u], bz[u]);
                if (P.sphere_symm) c = fabsf(c);
                if (j0 + u < l && c > P.cos_min_sep) conf |= 1u << ((j0 + u) & 31);
            }
        }
        uint32_t keep = 0u, decided = ~0u << (n & 31);  // lanes n.. count as decided
        if (n == 32) decided = 0u;
        while (decided != 0xffffffffu) {
            const bool open = !((decided >> l) & 1u);
            const bool gone = open && (conf & keep) != 0u;
            const bool kept = open && !gone && (conf & ~decided) == 0u;
            const uint32_t kmask = half_ballot(kept);
            decided |= half_ballot(gone) | kmask;
            keep |= kmask;
        }
        WAVE_SYNC();
        if (l < n && ((keep >> l) & 1u)) cand[__popc(keep & ((1u << l) - 1u))] = (uint16_t)ci;
        WAVE_SYNC();
        return __popc(keep);
    }
    int kept = 1;
    if (l == 0) {
        // remove_similar_vertices, single lane (tracking_helpers.cu:195-223),
        // compacting the kept indices in place.
        for (int i = 1; i < n; ++i) {
            const int ci = cand[i];
            const float ax = sv[3 * ci], ay = sv[3 * ci + 1], az = sv[3 * ci + 2];
            int j = 0;
            for (; j < kept; ++j) {
                const int cj = cand[j];
                float c = dot3(ax, ay, az, sv[3 * cj], sv[3 * cj + 1], sv[3 * cj + 2]);
                if (P.sphere_symm) c = fabsf(c);
                if (c > P.cos_min_sep) break;
            }
            if (j == kept) cand[kept++] = (uint16_t)ci;
        }
    }
    kept = shfl32(kept, 0);
    WAVE_SYNC();
    return kept;
}

// -------------------------------------------------------------------------
// Interpolation and the stop check
// -------------------------------------------------------------------------

// trilinear_interp_d (tracking_helpers.cu:3-61) over `dimt` channels with
// channel stride `ld`; writes out[0..dimt).  UNROLL channel iterations are
// in flight together (8 corner loads each): the probabilistic getter, whose
// step is this 23 KB gather, uses 3.
template <int UNROLL = 1>
__device__ int trilinear(const DevParams &P, const float *__restrict__ data, int ld, int dimt,
                         float px, float py, float pz, float *out) {
    if (px < -0.5f || px + 0.5f >= (float)P.dimx || py < -0.5f || py + 0.5f >= (float)P.dimy ||
        pz < -0.5f || pz + 0.5f >= (float)P.dimz)
        return -1;
    const float fx = floorf(px), fy = floorf(py), fz = floorf(pz);
    const float wx1 = px - fx, wy1 = py - fy, wz1 = pz - fz;
    const float wx0 = 1.0f - wx1, wy0 = 1.0f - wy1, wz0 = 1.0f - wz1;
    const int x0 = (int)((0.0f > fx) ? 0.0f : fx), y0 = (int)((0.0f > fy) ? 0.0f : fy),
              z0 = (int)((0.0f > fz) ? 0.0f : fz);
    const int x1 = min(P.dimx - 1, x0 + 1), y1 = min(P.dimy - 1, y0 + 1), z1 = min(P.dimz - 1, z0 + 1);
    const float w[8] = {(wx0 * wy0) * wz0, (wx0 * wy0) * wz1, (wx0 * wy1) * wz0, (wx0 * wy1) * wz1,
                        (wx1 * wy0) * wz0, (wx1 * wy0) * wz1, (wx1 * wy1) * wz0, (wx1 * wy1) * wz1};
    const size_t DY = (size_t)P.dimy, DZ = (size_t)P.dimz;
    const float *c[8] = {
        data + (((size_t)x0 * DY + y0) * DZ + z0) * ld, data + (((size_t)x0 * DY + y0) * DZ + z1) * ld,
        data + (((size_t)x0 * DY + y1) * DZ + z0) * ld, data + (((size_t)x0 * DY + y1) * DZ + z1) * ld,
        data + (((size_t)x1 * DY + y0) * DZ + z0) * ld, data + (((size_t)x1 * DY + y0) * DZ + z1) * ld,
        data + (((size_t)x1 * DY + y1) * DZ + z0) * ld, data + (((size_t)x1 * DY + y1) * DZ + z1) * ld};
    const int l = lane32();
#pragma unroll UNROLL
    for (int t = l; t < dimt; t += 32) {
        float v[8];
#pragma unroll
        for (int k = 0; k < 8; ++k) v[k] = c[k][t];
        float acc = 0.0f;
#pragma unroll
        for (int k = 0; k < 8; ++k) acc = __builtin_fmaf(w[k], v[k], acc);
        out[t] = acc;
    }
    return 0;
}

// Texture coordinate -> (first texel, 8-bit weight of the second texel),
// after the CUDA guide's linear filtering: xB = x - 0.5, i = floor(xB),
// weight = frac(xB) with 8 fractional bits.
__device__ __forceinline__ float tex_weight(float c, int *i0) {
    const float b = c - 0.5f;
    asm("v_cvt_flr_i32_f32 %0, %1" : "=v"(*i0) : "v"(b));
    // v_fract_f32: b - floor(b), held below 1, which rounds to the same 1/256
    return __builtin_rintf(__builtin_amdgcn_fractf(b) * 256.0f) * 0.00390625f;
}

// check_point_d (tracking_helpers.cu:63-73): linear filter of the stop map,
// border colour -1, texture x = array z (cu_tractography.py:237-241).  In two
// halves, so that a caller can put other loads between the 8 texel reads and
// their use; texels outside the map read a clamped one and are replaced.
struct StopTap {
    float a, b, g;
    float t[8];
    uint32_t in;  // bit k: texel k lies in the map
};

__device__ __forceinline__ StopTap stop_begin(const DevParams &P, const float *__restrict__ stop, float px, float py,
                                              float pz) {
    StopTap s;
    int iz, iy, ix;
    s.a = tex_weight(pz, &iz);
    s.b = tex_weight(py, &iy);
    s.g = tex_weight(px, &ix);
    const int DX = P.dimx, DY = P.dimy, DZ = P.dimz;
    uint32_t xo[2], yo[2], zo[2];
    bool xi[2], yi[2], zi[2];
#pragma unroll
    for (int k = 0; k < 2; ++k) {
        // k + clamp(i) would overflow for a position far outside, so the
        // second texel is clamped from the first's range
        xi[k] = ix >= -k && ix < DX - k;
        yi[k] = iy >= -k && iy < DY - k;
        zi[k] = iz >= -k && iz < DZ - k;
        xo[k] = (uint32_t)min(max(ix, -k), DX - 1 - k) + k;
        yo[k] = (uint32_t)min(max(iy, -k), DY - 1 - k) + k;
        zo[k] = (uint32_t)min(max(iz, -k), DZ - 1 - k) + k;
    }
    s.in = 0u;
#pragma unroll
    for (int k = 0; k < 8; ++k) {
        const int kz = k & 1, ky = (k >> 1) & 1, kx = k >> 2;
        s.t[k] = stop[(size_t)((xo[kx] * (uint32_t)DY + yo[ky]) * (uint32_t)DZ + zo[kz])];
        if (xi[kx] && yi[ky] && zi[kz]) s.in |= 1u << k;
    }
    return s;
}

__device__ __forceinline__ int stop_end(const DevParams &P, const StopTap &s) {
    const float a = s.a, b = s.b, g = s.g;
    const float a0 = 1.0f - a, b0 = 1.0f - b, g0 = 1.0f - g;
    auto t = [&](int k) { return ((s.in >> k) & 1u) ? s.t[k] : -1.0f; };
    float acc = ((a0 * b0) * g0) * t(0);
    acc = __builtin_fmaf((a * b0) * g0, t(1), acc);
    acc = __builtin_fmaf((a0 * b) * g0, t(2), acc);
    acc = __builtin_fmaf((a * b) * g0, t(3), acc);
    acc = __builtin_fmaf((a0 * b0) * g, t(4), acc);
    acc = __builtin_fmaf((a * b0) * g, t(5), acc);
    acc = __builtin_fmaf((a0 * b) * g, t(6), acc);
    acc = __builtin_fmaf((a * b) * g, t(7), acc);
    if (acc == -1.0f) return CUSLINES_OUTSIDEIMAGE;
    return (acc > P.tc_threshold) ? CUSLINES_TRACKPOINT : CUSLINES_ENDPOINT;
}

__device__ __forceinline__ int check_point(const DevParams &P, const float *__restrict__ stop, float px, float py,
                                           float pz) {
    return stop_end(P, stop_begin(P, stop, px, py, pz));
}

// Texel index I of one axis of the vertex-tiled PTT texture -> (tile, local),
// clamp address mode; `hint` is the tile the query was built from.
__device__ __forceinline__ void axis_split(int I, int D, int ntiles, int hint, int *tile, int *loc) {
    I = min(max(I, 0), ntiles * D - 1);
    int t = hint, c = I - hint * D;
    while (c < 0) { --t; c += D; }
    while (c >= D) { ++t; c -= D; }
    *tile = t;
    *loc = c;
}

// Linear-filtered sample of the (nx,ny,nz)-tiled ODF texture at big-texture
// coordinates (xq,yq,zq) built from tile (tx,ty,tz); slots >= nverts read 0.
__device__ float tiled_sample(const DevParams &P, const float *__restrict__ odfv, float xq, float yq,
                              float zq, int tx, int ty, int tz) {
    int i, j, k;
    const float a = tex_weight(xq, &i), b = tex_weight(yq, &j), g = tex_weight(zq, &k);
    const float a0 = 1.0f - a, b0 = 1.0f - b, g0 = 1.0f - g;
    int txa, txb, lxa, lxb, tya, tyb, lya, lyb, tza, tzb, lza, lzb;
    axis_split(i, P.dimx, P.nx, tx, &txa, &lxa);
    axis_split(i + 1, P.dimx, P.nx, tx, &txb, &lxb);
    axis_split(j, P.dimy, P.ny, ty, &tya, &lya);
    axis_split(j + 1, P.dimy, P.ny, ty, &tyb, &lyb);
    axis_split(k, P.dimz, P.nz, tz, &tza, &lza);
    axis_split(k + 1, P.dimz, P.nz, tz, &tzb, &lzb);
    const int DX = P.dimx, DY = P.dimy, DZ = P.dimz, NV = P.nverts, nx = P.nx, ny = P.ny;
    auto fetch = [&](int ti, int li, int tj, int lj, int tk, int lk) -> float {
        const int v = ti + nx * (tj + ny * tk);
        if (v >= NV) return 0.0f;
        return odfv[(((size_t)v * DX + li) * DY + lj) * DZ + lk];
    };
    float acc = ((a0 * b0) * g0) * fetch(txa, lxa, tya, lya, tza, lza);
    acc = __builtin_fmaf((a * b0) * g0, fetch(txb, lxb, tya, lya, tza, lza), acc);
    acc = __builtin_fmaf((a0 * b) * g0, fetch(txa, lxa, tyb, lyb, tza, lza), acc);
    acc = __builtin_fmaf((a * b) * g0, fetch(txb, lxb, tyb, lyb, tza, lza), acc);
    acc = __builtin_fmaf((a0 * b0) * g, fetch(txa, lxa, tya, lya, tzb, lzb), acc);
    acc = __builtin_fmaf((a * b0) * g, fetch(txb, lxb, tya, lya, tzb, lzb), acc);
    acc = __builtin_fmaf((a0 * b) * g, fetch(txa, lxa, tyb, lyb, tzb, lzb), acc);
    acc = __builtin_fmaf((a * b) * g, fetch(txb, lxb, tyb, lyb, tzb, lzb), acc);
    return acc;
}

// interp4_d (ptt.cu:24-42) in two halves, so a caller can issue the LUT
// read of one tap before it consumes the previous tap's block.
// lut_index: linear index of the nearest-vertex LUT cell of the tangent
// (point sampling, normalised coordinates, clamp).  Index products use
// 24-bit multiplies (full rate; every operand is below 2^24: LUT coordinates,
// tile indices, cell coordinates).
// v_cvt_u32_f32 takes negative values and NaN to 0 and truncates, so one
// minimum is left of floor and clamp.
__device__ __forceinline__ uint32_t cvt_u32_sat(float x) {
    uint32_t r;
    asm("v_cvt_u32_f32 %0, %1" : "=v"(r) : "v"(x));
    return r;
}

__device__ __forceinline__ uint32_t lut_index(const DevParams &P, float f0, float f1, float f2) {
    const int res = P.lut_res;
    const float rf = (float)res;
    const uint32_t imax = (uint32_t)res - 1u;
    const float u0 = __builtin_fmaf(f0, 0.5f, 0.5f), u1 = __builtin_fmaf(f1, 0.5f, 0.5f),
                u2 = __builtin_fmaf(f2, 0.5f, 0.5f);
    const uint32_t i0 = min(cvt_u32_sat(u0 * rf), imax), i1 = min(cvt_u32_sat(u1 * rf), imax),
                   i2 = min(cvt_u32_sat(u2 * rf), imax);
    if (P.lut_brick) {
        const uint32_t nb = (uint32_t)res >> 2;
        return (__umul24(__umul24(i0 >> 2, nb) + (i1 >> 2), nb) + (i2 >> 2)) * 64u + ((i0 & 3u) << 4) +
               ((i1 & 3u) << 2) + (i2 & 3u);
    }
    return __umul24(__umul24(i0, (uint32_t)res) + i1, (uint32_t)res) + i2;
}

// The linear-filtered sample of a vertex's tile of the ODF texture at
// (px, py, pz); `lv` is the vertex's LUT entry (vertex | rank << 16).  One
// 32-byte corner block when the cell is inside the volume (its 8 texels, the
// tile's clamp already applied), else the 8-texel gather.  Blocks are stored
// cell-major, the vertices of a cell in the rank order, so one 128-byte line
// holds a cell's blocks for four neighbouring directions.
//
// In two halves, so that a probe loop can issue one tap's block read, do
// other work and blend afterwards: tap_begin computes the weights and issues
// the read (fast = the cell has a corner block), tap_end blends (or gathers
// the 8 texels when there is no block).
struct Tap {
    float a, b, g;
    float4 lo, hi;
    float xq, yq, zq;
    uint32_t lv;
    bool fast;
};

__device__ __forceinline__ Tap tap_begin(const DevParams &P, const DevBufs &B, uint32_t lv, float px, float py,
                                         float pz) {
    Tap t;
    t.lv = lv;
    const int idx = (int)(lv & 0xffffu);
    const int tx = idx & (P.nx - 1);
    const int ty = (idx >> P.log2x) & (P.ny - 1);
    const int tz = idx >> (P.log2x + P.log2y);
    const int ox = (int)__umul24((uint32_t)tx, (uint32_t)P.dimx);
    const int oy = (int)__umul24((uint32_t)ty, (uint32_t)P.dimy);
    const int oz = (int)__umul24((uint32_t)tz, (uint32_t)P.dimz);
    t.xq = (float)ox + px;
    t.yq = (float)oy + py;
    t.zq = (float)oz + pz;
    t.fast = false;
    if (B.blocks) {
        int i, j, k;
        t.a = tex_weight(t.xq, &i);
        t.b = tex_weight(t.yq, &j);
        t.g = tex_weight(t.zq, &k);
        const int cx = i - ox, cy = j - oy, cz = k - oz;
        if ((unsigned)(cx + 1) <= (unsigned)P.dimx && (unsigned)(cy + 1) <= (unsigned)P.dimy &&
            (unsigned)(cz + 1) <= (unsigned)P.dimz) {
            const uint32_t inner =
                __umul24(__umul24((uint32_t)(cx + 1), (uint32_t)(P.dimy + 1)) + (uint32_t)(cy + 1),
                         (uint32_t)(P.dimz + 1)) + (uint32_t)(cz + 1);
            const uint64_t cell = (uint64_t)inner * (uint32_t)P.nverts + (lv >> 16);
            const float4 *blk = reinterpret_cast<const float4 *>(B.blocks + cell * 8);
            t.lo = blk[0];
            t.hi = blk[1];
            t.fast = true;
        }
    }
    return t;
}

// Linear filter of a corner block (texel order x fastest, then y, z).
__device__ __forceinline__ float corner_blend(float a, float b, float g, const float4 &lo, const float4 &hi) {
    const float a0 = 1.0f - a, b0 = 1.0f - b, g0 = 1.0f - g;
    float acc = ((a0 * b0) * g0) * lo.x;
    acc = __builtin_fmaf((a * b0) * g0, lo.y, acc);
    acc = __builtin_fmaf((a0 * b) * g0, lo.z, acc);
    acc = __builtin_fmaf((a * b) * g0, lo.w, acc);
    acc = __builtin_fmaf((a0 * b0) * g, hi.x, acc);
    acc = __builtin_fmaf((a * b0) * g, hi.y, acc);
    acc = __builtin_fmaf((a0 * b) * g, hi.z, acc);
    acc = __builtin_fmaf((a * b) * g, hi.w, acc);
    return acc;
}

__device__ __forceinline__ float tap_end(const DevParams &P, const DevBufs &B, const Tap &t) {
    if (t.fast) return corner_blend(t.a, t.b, t.g, t.lo, t.hi);
    const int idx = (int)(t.lv & 0xffffu);
    return tiled_sample(P, B.data, t.xq, t.yq, t.zq, idx & (P.nx - 1), (idx >> P.log2x) & (P.ny - 1),
                        idx >> (P.log2x + P.log2y));
}

__device__ __forceinline__ float tap_sample(const DevParams &P, const DevBufs &B, uint32_t lv, float px, float py,
                                            float pz) {
    return tap_end(P, B, tap_begin(P, B, lv, px, py, pz));
}

// A tap for loops that hold several in flight: tap_begin's weights and
// block read, with a cell that has no block gathered at once (its value in
// lo.x), so a tap in flight holds no more than its weights and block.
struct TapB {
    float a, b, g;
    float4 lo, hi;
    bool fast;
};

__device__ __forceinline__ TapB tapb_begin(const DevParams &P, const DevBufs &B, uint32_t lv, float px, float py,
                                           float pz) {
    const Tap t = tap_begin(P, B, lv, px, py, pz);
    TapB r;
    r.a = t.a; r.b = t.b; r.g = t.g;
    r.lo = t.lo; r.hi = t.hi;
    r.fast = t.fast;
    if (!t.fast) r.lo.x = tap_end(P, B, t);
    return r;
}

__device__ __forceinline__ float tapb_end(const TapB &t) {
    return t.fast ? corner_blend(t.a, t.b, t.g, t.lo, t.hi) : t.lo.x;
}

__device__ __forceinline__ float interp4(const DevParams &P, const DevBufs &B, float px, float py,
                                         float pz, float f0, float f1, float f2) {
    return tap_sample(P, B, B.lut[lut_index(P, f0, f1, f2)], px, py, pz);
}


// -------------------------------------------------------------------------
// Half-wave matrix-vector products with the reference's per-row summation
// (ndotp_d, boot.cu:195-235): per row, 32 lane partials over j = l, l+32, ...
// (fma, in order), then the 16/8/4/2/1 pair tree.
// XF selects the elementwise transform of the vector: 0 none, 1 OPDT, 2 CSA.
// -------------------------------------------------------------------------
template <int XF>
__device__ __forceinline__ float gemv_xf(float x) {
    if (XF == 1) {
        const float lx = ulog(x);
        return ((-lx) * (1.5f + lx)) * x;
    } else if (XF == 2) {
        const float c = fminf(fmaxf(x, 0.001f), 0.999f);
        return ulog(-ulog(c));
    }
    return x;
}

// One row per lane: lane r of the slot sums row i0 + r itself, keeping the
// 32 partials in registers and adding them with the pair tree, so a row
// costs M fma + 31 adds (a shuffle reduction across lanes costs ~4 VALU per
// row-lane pair more).  When M % 4 == 0 the matrix is stored lane-interleaved
// (mat_offset: the 4-column pieces of 32 consecutive rows side by side), so
// the 16-byte row loads of one instruction are 512 contiguous bytes; else
// row-major.  x comes from LDS as broadcast reads and must be 16-byte
// aligned, already transformed (gemv_xf).
__host__ __device__ inline size_t mat_offset(int M, int i, int j) {
    return (((size_t)(i >> 5) * (size_t)(M >> 2) + (size_t)(j >> 2)) << 7) + (size_t)((i & 31) << 2) + (size_t)(j & 3);
}

__device__ void gemv_lanerow(int N, int M, const float *x, const float *__restrict__ mat, float *out) {
    const int l = lane32();
    const bool vec = (M & 3) == 0;
    for (int i0 = 0; i0 < N; i0 += 32) {
        const int i = i0 + l;
        if (i < N) {
            const float *row = vec ? mat + mat_offset(M, i, 0) : mat + (size_t)i * M;
            float p[32];
#pragma unroll
            for (int q = 0; q < 32; ++q) p[q] = 0.0f;
            for (int j0 = 0; j0 < M; j0 += 32) {
                // All loads of the block are issued before the first use: a
                // column past M re-reads the block's last valid one, and its
                // product is dropped by the select, so no load sits behind a
                // branch (and none leaves the matrix).
                const int nj = min(32, M - j0);
                if (vec) {  // M % 4 == 0: a vector is all in or all out
                    const int nq = nj >> 2;
                    float4 m[8];
#pragma unroll
                    for (int q = 0; q < 8; ++q)
                        m[q] = *reinterpret_cast<const float4 *>(row + ((size_t)(j0 + 4 * min(q, nq - 1)) << 5));
#pragma unroll
                    for (int q = 0; q < 8; ++q) {
                        const float4 v = *reinterpret_cast<const float4 *>(x + j0 + 4 * q);
                        const bool in = q < nq;
                        const float a0 = __builtin_fmaf(v.x, m[q].x, p[4 * q]);
                        const float a1 = __builtin_fmaf(v.y, m[q].y, p[4 * q + 1]);
                        const float a2 = __builtin_fmaf(v.z, m[q].z, p[4 * q + 2]);
                        const float a3 = __builtin_fmaf(v.w, m[q].w, p[4 * q + 3]);
                        p[4 * q] = in ? a0 : p[4 * q];
                        p[4 * q + 1] = in ? a1 : p[4 * q + 1];
                        p[4 * q + 2] = in ? a2 : p[4 * q + 2];
                        p[4 * q + 3] = in ? a3 : p[4 * q + 3];
                    }
                } else {
                    float m[32];
#pragma unroll
                    for (int q = 0; q < 32; ++q) m[q] = row[j0 + min(q, nj - 1)];
#pragma unroll
                    for (int q = 0; q < 32; ++q) {
                        const float a = __builtin_fmaf(x[j0 + q], m[q], p[q]);
                        p[q] = (q < nj) ? a : p[q];
                    }
                }
            }
#pragma unroll
            for (int d = 16; d >= 1; d >>= 1)
#pragma unroll
                for (int q = 0; q < d; ++q) p[q] = p[q] + p[q + d];
            out[i] = p[0];
        }
    }
    WAVE_SYNC();
}

// The same sums for the kernel of 2 waves per SIMD.  Four of these products are
// three quarters of an exact attempt's time (148 k cycles for a lone slot), and
// each waits for its matrix's blocks from L2 (some 1200 cycles) rather than for
// its sums: a step reads 282 KB of matrices.  Here the next block's loads are in
// flight behind the sums, without a branch per column, and with the 256
// registers they take; boot_waves has the rule and its figures.  The kernel
// still spills 80 (CSA) and 92 (OPDT) vector registers around the products.
// Out of line, 3001 seeds are faster still (77 ms), but the kernel has one wave
// per SIMD left (20 000 seeds: 260 ms); two or three blocks ahead spill more
// (20 000 seeds: 213, 233 ms).
__device__ __forceinline__ void gemv_lanerow_wide(int N, int M, const float *x, const float *__restrict__ mat, float *out) {
    const int l = lane32();
    if ((M & 3) == 0) {
        // 32 rows by 32 columns a block; the next block's loads, of the same
        // rows or the next ones, are in flight while a block is summed.
        const int nblk = (M + 31) >> 5, total = nblk * ((N + 31) >> 5);
        auto load = [&](int i0, int j0, float4 (&m)[8]) {
            const int nq = min(8, (M - j0) >> 2);
            const float *row = mat + mat_offset(M, min(i0 + l, N - 1), j0);  // past the last row: re-read, dropped
#pragma unroll
            for (int q = 0; q < 8; ++q)  // past the last column: the last valid one, its product dropped
                m[q] = *reinterpret_cast<const float4 *>(row + ((size_t)(4 * min(q, nq - 1)) << 5));
        };
        float p[32];
#pragma unroll
        for (int q = 0; q < 32; ++q) p[q] = 0.0f;
        float4 m[2][8];
        load(0, 0, m[0]);
        int i0 = 0, j0 = 0;
        auto block = [&](const float4 (&cur)[8], float4 (&nxt)[8], bool more) {
            int i1 = i0, j1 = j0 + 32;
            if (j1 >= M) { j1 = 0; i1 += 32; }
            if (more) load(i1, j1, nxt);
            const int nq = (M - j0) >> 2;
            float4 v[8];
#pragma unroll
            for (int q = 0; q < 8; ++q) v[q] = *reinterpret_cast<const float4 *>(x + j0 + 4 * min(q, nq - 1));
            if (nq >= 8) {
#pragma unroll
                for (int q = 0; q < 8; ++q) {
                    p[4 * q] = __builtin_fmaf(v[q].x, cur[q].x, p[4 * q]);
                    p[4 * q + 1] = __builtin_fmaf(v[q].y, cur[q].y, p[4 * q + 1]);
                    p[4 * q + 2] = __builtin_fmaf(v[q].z, cur[q].z, p[4 * q + 2]);
                    p[4 * q + 3] = __builtin_fmaf(v[q].w, cur[q].w, p[4 * q + 3]);
                }
            } else {
                int nqv = nq;
                asm volatile("" : "+v"(nqv));  // selects: a branch each would wait for each product
#pragma unroll
                for (int q = 0; q < 8; ++q) {
                    const bool in = q < nqv;
                    const float a0 = __builtin_fmaf(v[q].x, cur[q].x, p[4 * q]);
                    const float a1 = __builtin_fmaf(v[q].y, cur[q].y, p[4 * q + 1]);
                    const float a2 = __builtin_fmaf(v[q].z, cur[q].z, p[4 * q + 2]);
                    const float a3 = __builtin_fmaf(v[q].w, cur[q].w, p[4 * q + 3]);
                    p[4 * q] = in ? a0 : p[4 * q];
                    p[4 * q + 1] = in ? a1 : p[4 * q + 1];
                    p[4 * q + 2] = in ? a2 : p[4 * q + 2];
                    p[4 * q + 3] = in ? a3 : p[4 * q + 3];
                }
            }
            if (j1 == 0) {
#pragma unroll
                for (int d = 16; d >= 1; d >>= 1)
#pragma unroll
                    for (int q = 0; q < d; ++q) p[q] = p[q] + p[q + d];
                if (i0 + l < N) out[i0 + l] = p[0];
#pragma unroll
                for (int q = 0; q < 32; ++q) p[q] = 0.0f;
            }
            i0 = i1;
            j0 = j1;
        };
        for (int it = 0; it < total; it += 2) {
            block(m[0], m[1], it + 1 < total);
            if (it + 1 < total) block(m[1], m[0], it + 2 < total);
        }
        WAVE_SYNC();
        return;
    }
    gemv_lanerow(N, M, x, mat, out);
}

// -------------------------------------------------------------------------
// Probabilistic getter (generate_streamlines_cuda.cu:49-275)
// -------------------------------------------------------------------------
struct ProbLds {
    float *pmf;
    uint32_t *marks;
    uint16_t *cand;
};

// Threshold, cone test and running sum of the interpolated pmf (LDS, nverts
// values); returns its last element.
__device__ float prob_sum(int nv, int symm, float cos_max_angle, const float *sv, float *pmf, float dx, float dy,
                          float dz) {
    const int l = lane32();
    float mx = REAL_MIN;
    for (int i = l; i < nv; i += 32) mx = (mx > pmf[i]) ? mx : pmf[i];
    mx = max32(mx);
    const float thr = (float)(PMF_THRESHOLD_P * (double)mx);
    for (int i = l; i < nv; i += 32) {
        float v = pmf[i];
        if (v < thr) v = 0.0f;
        float d = dot3(dx, dy, dz, sv[3 * i], sv[3 * i + 1], sv[3 * i + 2]);
        if (symm) d = fabsf(d);
        if (d < cos_max_angle) v = 0.0f;
        pmf[i] = v;
    }
    WAVE_SYNC();
    prefix_sum(pmf, nv);
    return pmf[nv - 1];
}

// Index of the direction that `sel` falls on in the running sum `pmf`.
__device__ int prob_pick(const float *pmf, int nv, float sel) {
    const int l = lane32();
    int low = 0, high = nv - 1;
    while ((high - low) >= 32) {
        const int mid = (low + high) / 2;
        if (pmf[mid] < sel) low = mid; else high = mid;
    }
    const bool pr = (low + l <= high) ? (sel < pmf[low + l]) : false;
    const uint32_t msk = half_ballot(pr);
    int ind = low + __ffs(msk) - 1;
    if (ind < 0) ind = 0;
    return ind;
}

// The getter draws one uniform a step from lane 0's stream.  The slot's
// lanes (32 or 64) hold consecutive blocks of it, 4 draws each, so a Philox
// evaluation serves 128 or 256 steps.
template <int LANES>
struct ProbStream {
    uint32_t k0, k1, s0, s1;
    uint32_t r0, r1, r2, r3;
    uint32_t k;  // draws taken

    __device__ __forceinline__ void refill() {
        Philox p;
        p.k0 = k0; p.k1 = k1; p.s0 = s0; p.s1 = s1;
        p.c0 = (k >> 2) + (threadIdx.x & (LANES - 1));
        p.c1 = 0u;
        p.refill();
        r0 = p.r0; r1 = p.r1; r2 = p.r2; r3 = p.r3;
    }
    __device__ __forceinline__ void init(uint64_t seed, uint64_t sub) {
        k0 = (uint32_t)seed; k1 = (uint32_t)(seed >> 32);
        s0 = (uint32_t)sub; s1 = (uint32_t)(sub >> 32);
        k = 0u;
        refill();
    }
    // the next draw's uniform; take() moves past it
    __device__ __forceinline__ float peek() const {
        const uint32_t a = (k & 1u) ? r1 : r0, b = (k & 1u) ? r3 : r2;
        const int w = (int)((k & 2u) ? b : a), from = (int)((k >> 2) & (LANES - 1));
        const uint32_t x =
            (uint32_t)((LANES == 64) ? __builtin_amdgcn_readlane(w, __builtin_amdgcn_readfirstlane(from)) : shfl32(w, from));
        return 2.32830644e-10f + (float)x * 2.32830644e-10f;
    }
    __device__ __forceinline__ void take() {
        if ((++k & (4u * LANES - 1u)) == 0u) refill();
    }
};

template <bool IS_START>
__device__ int get_direction_prob(const DevParams &P, const DevBufs &B, const float *sv, ProbLds &S,
                                  ProbStream<32> &rng, float dx, float dy, float dz, float px, float py,
                                  float pz, float *ndx, float *ndy, float *ndz) {
    float *pmf = S.pmf;
    if (trilinear<3>(P, B.data, P.t32, P.dimt, px, py, pz, pmf) != 0) return 0;
    WAVE_SYNC();
    const int l = lane32();
    const int nv = P.nverts;
    if (!IS_START) {
        const float last = prob_sum(nv, P.sphere_symm, P.cos_max_angle, sv, pmf, dx, dy, dz);
        if (last == 0.0f) return 0;
        const int ind = prob_pick(pmf, nv, rng.peek() * last);
        rng.take();
        const float vx = sv[3 * ind], vy = sv[3 * ind + 1], vz = sv[3 * ind + 2];
        if (dot3(dx, dy, dz, vx, vy, vz) > 0.0f) { *ndx = vx; *ndy = vy; *ndz = vz; }
        else { *ndx = -vx; *ndy = -vy; *ndz = -vz; }
        WAVE_SYNC();
        return 1;
    }
    float mx = REAL_MIN;
    for (int i = l; i < nv; i += 32) mx = (mx > pmf[i]) ? mx : pmf[i];
    mx = max32(mx);
    const float thr = (float)(PMF_THRESHOLD_P * (double)mx);
    for (int i = l; i < nv; i += 32)
        if (pmf[i] < thr) pmf[i] = 0.0f;
    WAVE_SYNC();
    return peak_directions(peak_params(P, B), pmf, S.marks, S.cand, sv);
}

// The random streams of a slot: the probabilistic getter's one, the others' 32.
template <int MODEL>
struct SlotRng {
    typedef Philox type;
};
template <>
struct SlotRng<CUSLINES_PROB> {
    typedef ProbStream<32> type;
};
// The exact bootstrap kernels' registers are full: with PAIR, and with the peak
// tail inline, the one of 4 waves per SIMD spills 140 (CSA) and 143 (OPDT)
// vector registers instead of 76.  100,000 seeds on 81x106x76, ms: CSA
// 464 -> 418, OPDT 365 -> 335; 25,000 on this variant: 243 -> 230, 299 -> 286.
template <>
struct SlotRng<CUSLINES_OPDT> {
    typedef PhiloxStream<false> type;
};
template <>
struct SlotRng<CUSLINES_CSA> {
    typedef PhiloxStream<false> type;
};

// trilinear on 16-byte loads: lane l owns channels 128 c + 4 l .. + 3, a
// chunk's 8 corner loads in flight (two chunks' 64 registers spill at 4 waves
// per SIMD: 25,000 seeds 101 instead of 91 ms).  False outside the volume.
__device__ __forceinline__ bool bb_gather(const DevParams &P, const float *__restrict__ data, float px, float py,
                                          float pz, float *out) {
    if ((px < -0.5f) | (px + 0.5f >= (float)P.dimx) | (py < -0.5f) | (py + 0.5f >= (float)P.dimy) | (pz < -0.5f) |
        (pz + 0.5f >= (float)P.dimz))
        return false;
    const int l = lane32();
    const float fx = floorf(px), fy = floorf(py), fz = floorf(pz);
    const float wx1 = px - fx, wy1 = py - fy, wz1 = pz - fz;
    const float wx0 = 1.0f - wx1, wy0 = 1.0f - wy1, wz0 = 1.0f - wz1;
    const int x0 = (int)((0.0f > fx) ? 0.0f : fx), y0 = (int)((0.0f > fy) ? 0.0f : fy),
              z0 = (int)((0.0f > fz) ? 0.0f : fz);
    const float w[8] = {(wx0 * wy0) * wz0, (wx0 * wy0) * wz1, (wx0 * wy1) * wz0, (wx0 * wy1) * wz1,
                        (wx1 * wy0) * wz0, (wx1 * wy0) * wz1, (wx1 * wy1) * wz0, (wx1 * wy1) * wz1};
    const uint32_t dzv = (z0 + 1 < P.dimz) ? 1u : 0u;
    const uint32_t dyv = (y0 + 1 < P.dimy) ? (uint32_t)P.dimz : 0u;
    const uint32_t dxv = (x0 + 1 < P.dimx) ? (uint32_t)P.dimy * (uint32_t)P.dimz : 0u;
    const uint32_t vox = ((uint32_t)x0 * (uint32_t)P.dimy + (uint32_t)y0) * (uint32_t)P.dimz + (uint32_t)z0;
    const float *c[8];
#pragma unroll
    for (int k = 0; k < 8; ++k)
        c[k] = data + (uint64_t)(vox + ((k & 4) ? dxv : 0u) + ((k & 2) ? dyv : 0u) + ((k & 1) ? dzv : 0u)) *
                          (uint32_t)P.t32;
    for (int t0 = 0; t0 < P.t32; t0 += 128) {
        const int ta = t0 + 4 * l;
        const int sa = min(ta, P.t32 - 4);  // past the row: re-read, dropped
        float4 va[8];
#pragma unroll
        for (int k = 0; k < 8; ++k) va[k] = *reinterpret_cast<const float4 *>(c[k] + sa);
        float4 a = float4{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
        for (int k = 0; k < 8; ++k) {
            a.x = __builtin_fmaf(w[k], va[k].x, a.x); a.y = __builtin_fmaf(w[k], va[k].y, a.y);
            a.z = __builtin_fmaf(w[k], va[k].z, a.z); a.w = __builtin_fmaf(w[k], va[k].w, a.w);
        }
        if (ta < P.t32) *reinterpret_cast<float4 *>(out + ta) = a;
    }
    return true;
}

// -------------------------------------------------------------------------
// Bootstrap getter (boot.cu:19-113, 115-193, 330-608)
// -------------------------------------------------------------------------
struct BootLds {
    float *h;          // region C: H.d, then the ODF
    float *vox, *msk;  // region A during the refit: vox [t32], msk [hr32]
    float *r;          // region A: R.d, then the model coefficients
    uint32_t *marks;   // region A once the ODF is computed: peak marks, 2 bits per vertex
    uint16_t *cand;    // region A after the marks: peak candidates
};

// closest_peak_d (boot.cu:115-193): lane-strided best |dot| with strict
// improvement, then an xor tree with the same rule; lane 0's winner counts.
__device__ int closest_peak(const DevParams &P, const float *sv, float dx, float dy, float dz, int npeaks,
                            const uint16_t *peaks, float *ox, float *oy, float *oz) {
    const int l = lane32();
    float cd = 0.0f;
    int ci = -1;
    for (int j = l; j < npeaks; j += 32) {
        const int v = peaks[j];
        const float d = dot3(dx, dy, dz, sv[3 * v], sv[3 * v + 1], sv[3 * v + 2]);
        if (fabsf(d) > fabsf(cd)) { cd = d; ci = j; }
    }
    for (int m = 16; m; m >>= 1) {
        const float od = shfl_xor32(cd, m);
        const int oi = shfl_xor32(ci, m);
        if (fabsf(od) > fabsf(cd)) { cd = od; ci = oi; }
    }
    cd = shfl32(cd, 0);
    ci = shfl32(ci, 0);
    if (ci >= 0) {
        const int v = peaks[ci];
        if (cd >= P.cos_max_angle) { *ox = sv[3 * v]; *oy = sv[3 * v + 1]; *oz = sv[3 * v + 2]; return 1; }
        if (cd <= -P.cos_max_angle) { *ox = -sv[3 * v]; *oy = -sv[3 * v + 1]; *oz = -sv[3 * v + 2]; return 1; }
    }
    return 0;
}

// WIDE: the kernel of 2 waves per SIMD.
template <int MODEL, bool WIDE = false>
__device__ int get_direction_boot(const DevParams &P, const DevBufs &B, const float *sv, BootLds &S,
                                  typename SlotRng<MODEL>::type &rng, int nattempts, float dx, float dy, float dz, float px,
                                  float py, float pz, float *ndx, float *ndy, float *ndz) {
    const int l = lane32();
    const auto gemv = [](int N, int M, const float *x, const float *__restrict__ mat, float *out) {
        if constexpr (WIDE) gemv_lanerow_wide(N, M, x, mat, out);
        else gemv_lanerow(N, M, x, mat, out);
    };
    const int hr = P.hr, dn = P.delta_nr, nv = P.nverts, T = P.dimt;
    for (int att = 0; att < nattempts; ++att) {
        int rv;
        if constexpr (WIDE) rv = bb_gather(P, B.data, px, py, pz, S.vox) ? 0 : -1;
        else rv = trilinear(P, B.data, P.t32, T, px, py, pz, S.vox);
        WAVE_SYNC();
        if (rv == 0) {
            for (int m = l; m < hr; m += 32) S.msk[m] = S.vox[B.dwi_idx[m]];
            WAVE_SYNC();
            gemv(hr, hr, S.msk, B.R, S.r);
            gemv(hr, hr, S.msk, B.H, S.h);
            for (int j = l; j < hr; j += 32) {
                const int src = (int)(rng.next() % (uint32_t)hr);
                S.h[j] = S.h[j] + S.r[src];
            }
            WAVE_SYNC();
            for (int m = l; m < hr; m += 32) S.vox[B.dwi_idx[m]] = S.h[m];
            WAVE_SYNC();
            float part = 0.0f;
            int cnt = 0;
            for (int j = l; j < T; j += 32) {
                float v = S.vox[j];
                v = (P.min_signal > v) ? P.min_signal : v;
                S.vox[j] = v;
                if (B.b0[j]) { ++cnt; part = part + v; }
            }
            const float sum = tree_sum32(part);
            for (int m = 16; m; m >>= 1) cnt += shfl_xor32(cnt, m);
            const float denom = sum / (float)cnt;
            for (int j = l; j < T; j += 32) S.vox[j] = S.vox[j] / denom;
            WAVE_SYNC();
            for (int m = l; m < hr; m += 32) S.msk[m] = S.vox[B.dwi_idx[m]];
            WAVE_SYNC();
            // the model's transform of the signal, staged in h (free here)
            for (int j = l; j < hr; j += 32) S.h[j] = gemv_xf<(MODEL == CUSLINES_OPDT) ? 1 : 2>(S.msk[j]);
            WAVE_SYNC();
            gemv(dn, hr, S.h, B.dq, S.r);
            if (MODEL == CUSLINES_OPDT) {
                gemv(dn, hr, S.msk, B.db, S.h);
                for (int j = l; j < dn; j += 32) S.r[j] = S.r[j] - S.h[j];
            } else {
                if (l == 0) S.r[0] = CSA_C0;
            }
            WAVE_SYNC();
            gemv(nv, dn, S.r, B.smat, S.h);
        } else {
            for (int j = l; j < nv; j += 32) S.h[j] = 0.0f;
            WAVE_SYNC();
        }
        float mx = REAL_MIN;
        for (int j = l; j < nv; j += 32) mx = (mx > S.h[j]) ? mx : S.h[j];
        mx = max32(mx);
        const float thr = (float)(PMF_THRESHOLD_P * (double)mx);
        for (int j = l; j < nv; j += 32)
            if (S.h[j] < thr) S.h[j] = 0.0f;
        WAVE_SYNC();
        const int ndir = peak_directions<!WIDE>(peak_params(P, B), S.h, S.marks, S.cand, sv);
        if (nattempts == 1) return ndir;
        if (ndir > 0 && closest_peak(P, sv, dx, dy, dz, ndir, S.cand, ndx, ndy, ndz)) {
            WAVE_SYNC();
            return 1;
        }
        WAVE_SYNC();
    }
    return 0;
}

// -------------------------------------------------------------------------
// PTT getter (ptt.cu)
// -------------------------------------------------------------------------
// norm3_d (ptt.cu:1-13): scale to unit length when 1/|v| is finite, positive
// and below 1e8 (|v|^2 > 1e-16), else the FAIL axis.
template <int FAIL>
__device__ __forceinline__ void norm3(float &x, float &y, float &z) {
    const float n2 = __builtin_fmaf(z, z, __builtin_fmaf(y, y, x * x));
    if (n2 > PTT_MIN_NORM2 && n2 <= 3.40282347e+38f) {
        const float inv = rsqrt_nr(n2);
        x *= inv; y *= inv; z *= inv;
    } else {
        x = (FAIL == 0) ? 1.0f : 0.0f;
        y = (FAIL == 1) ? 1.0f : 0.0f;
        z = (FAIL == 2) ? 1.0f : 0.0f;
    }
}

template <int FAIL>
__device__ __forceinline__ void crossnorm3(float *d, const float *a, const float *b) {
    d[0] = __builtin_fmaf(a[1], b[2], -(a[2] * b[1]));
    d[1] = __builtin_fmaf(a[2], b[0], -(a[0] * b[2]));
    d[2] = __builtin_fmaf(a[0], b[1], -(a[1] * b[0]));
    norm3<FAIL>(d[0], d[1], d[2]);
}

__device__ __forceinline__ void prepare_propagator(float k1, float k2, float arclen, float *p) {
    if (fabsf(k1) < K_SMALL && fabsf(k2) < K_SMALL) {
        p[0] = arclen; p[1] = 0.0f; p[2] = 0.0f; p[3] = 1.0f; p[4] = 0.0f;
        p[5] = 0.0f; p[6] = 0.0f; p[7] = 0.0f; p[8] = 1.0f;
        return;
    }
    if (fabsf(k1) < K_SMALL) k1 = K_SMALL;
    if (fabsf(k2) < K_SMALL) k2 = K_SMALL;
    const float k = __builtin_sqrtf(__builtin_fmaf(k2, k2, k1 * k1));
    float sinkt, coskt;
    usincos(k * arclen, &sinkt, &coskt);
    const float kk = 1.0f / (k * k);
    p[0] = sinkt / k;
    p[1] = (k1 * (1.0f - coskt)) * kk;
    p[2] = (k2 * (1.0f - coskt)) * kk;
    p[3] = coskt;
    p[4] = (k1 * sinkt) / k;
    p[5] = (k2 * sinkt) / k;
    p[6] = -p[5];
    p[7] = ((k1 * k2) * (coskt - 1.0f)) * kk;
    p[8] = __builtin_fmaf(k2 * k2, coskt, k1 * k1) * kk;
}

__device__ __forceinline__ void propagate_frame(const float *p, float *f, float *direc) {
    float tmp[3];
#pragma unroll
    for (int i = 0; i < 3; ++i) {
        direc[i] = __builtin_fmaf(p[2], f[6 + i], __builtin_fmaf(p[1], f[3 + i], p[0] * f[i]));
        tmp[i] = __builtin_fmaf(p[5], f[6 + i], __builtin_fmaf(p[4], f[3 + i], p[3] * f[i]));
        f[6 + i] = __builtin_fmaf(p[8], f[6 + i], __builtin_fmaf(p[7], f[3 + i], p[6] * f[i]));
    }
    norm3<0>(tmp[0], tmp[1], tmp[2]);
    crossnorm3<1>(f + 3, f + 6, tmp);
    crossnorm3<2>(f + 6, tmp, f + 3);
    f[0] = tmp[0]; f[1] = tmp[1]; f[2] = tmp[2];
}

template <bool INIT>
__device__ __forceinline__ void probing_frame(const float *frame, Philox &rng, float *pf) {
    if (INIT) {
        pf[0] = frame[0]; pf[1] = frame[1]; pf[2] = frame[2];
        norm3<0>(pf[0], pf[1], pf[2]);
        pf[3] = rng.normal();
        pf[4] = rng.normal();
        pf[5] = rng.normal();
        const float dt = __builtin_fmaf(pf[5], pf[2], __builtin_fmaf(pf[4], pf[1], pf[3] * pf[0]));
        pf[3] = __builtin_fmaf(-dt, pf[0], pf[3]);
        pf[4] = __builtin_fmaf(-dt, pf[1], pf[4]);
        pf[5] = __builtin_fmaf(-dt, pf[2], pf[5]);
        const float n2 = __builtin_fmaf(pf[5], pf[5], __builtin_fmaf(pf[4], pf[4], pf[3] * pf[3]));
        if (n2 < PTT_NORM_EPS) {
            const float ax = fabsf(pf[0]), ay = fabsf(pf[1]), az = fabsf(pf[2]);
            if (ax <= ay && ax <= az) { pf[3] = 0.0f; pf[4] = pf[2]; pf[5] = -pf[1]; }
            else if (ay <= az) { pf[3] = -pf[2]; pf[4] = 0.0f; pf[5] = pf[0]; }
            else { pf[3] = pf[1]; pf[4] = -pf[0]; pf[5] = 0.0f; }
        }
        norm3<1>(pf[3], pf[4], pf[5]);
        crossnorm3<2>(pf + 6, pf, pf + 3);
    } else {
#pragma unroll
        for (int i = 0; i < 9; ++i) pf[i] = frame[i];
    }
}

// calculate_data_support_d (ptt.cu:156-192)
// The frames of successive probes do not depend on the sampled values, so
// probe i's block read is issued, then probe i+1's frame is propagated and
// its LUT read issued, and only then is probe i's block blended: each load's
// latency overlaps the other probe's work.
// With ALLOW_WEAK_LINK (ptt.cuh:8) the support is first_val plus the taps,
// all >= 0 (the ODF is clipped at 0 and linear filtering keeps the sign),
// so the running sum never decreases: once it reaches `stop_at` the
// candidate passes whatever the remaining taps add, and the lane stops
// probing.  Callers that need the value itself pass +infinity.  `ntap`
// (instrumented kernels only; nullptr otherwise) counts the taps read.
__device__ __forceinline__ float data_support(const DevParams &P, const DevBufs &B, float support,
                                              float px, float py, float pz, float k1, float k2, float *pf,
                                              float stop_at, uint32_t *ntap = nullptr,
                                              const float *prop_pre = nullptr) {
    // already at the threshold: no tap can change the outcome, and the
    // probe frames are dropped by every caller that passes a finite stop_at
    if (support >= stop_at) return support;
    float prop[9], direc[3];
    if (prop_pre) {
#pragma unroll
        for (int i = 0; i < 9; ++i) prop[i] = prop_pre[i];
    } else {
        prepare_propagator(k1, k2, P.probe_step, prop);
    }
    propagate_frame(prop, pf, direc);
    px += direc[0]; py += direc[1]; pz += direc[2];
    uint32_t idx = B.lut[lut_index(P, pf[0], pf[1], pf[2])];
    for (int i = 0; i < P.probe_quality; ++i) {
        if (support >= stop_at) break;
        if (ntap) ++*ntap;
        const Tap t = tap_begin(P, B, idx, px, py, pz);
        if (i + 1 < P.probe_quality) {
            propagate_frame(prop, pf, direc);
            px += direc[0]; py += direc[1]; pz += direc[2];
            idx = B.lut[lut_index(P, pf[0], pf[1], pf[2])];
        }
        support += tap_end(P, B, t);
    }
    return support;
}

struct PttLds {
    float *frame;     // 18 floats: [0..8] backward frame, [9..17] forward frame
    float *vert_pdf;  // 32
    float *face_cdf;  // 32
    float *act;       // learned proposal: inputs [64], hidden 1 [128], hidden 2 [128], outputs [32]
};

// Face CDF over the 31 disc faces from S.vert_pdf (prefix_sum_sh_d, one
// block of 32); returns the total.
__device__ __forceinline__ float ptt_face_cdf(PttLds &S) {
    const int l = lane32();
    float face = 0.0f;
    if (l < DISC_FACE_CNT) {
#pragma unroll
        for (int jj = 0; jj < 3; ++jj) {
            const float vv = S.vert_pdf[c_disc_face[l * 3 + jj]];
            if (vv == 0.0f) { face = 0.0f; break; }
            face = face + vv;
        }
    }
#pragma unroll
    for (int i = 1; i < 32; i <<= 1) {
        const float o = shfl_up32(face, i);
        if (l >= i && l < DISC_FACE_CNT) face = face + o;
    }
    if (l < DISC_FACE_CNT) S.face_cdf[l] = face;
    const float last = shfl32(face, DISC_FACE_CNT - 1);
    WAVE_SYNC();
    return last;
}

// One PTT sub-step (ptt.cu:194-412) as a single loop over phases: phase 0
// measures the 24 vertex supports (lanes < 24) into S.vert_pdf, phases
// 1..rounds are rejection rounds of 32 candidates drawn from the face CDF.
// Every phase ends in the same data_support call, so the two seeds of a
// wavefront probe together whichever phase each one is in.  first_phase 1
// starts from supports already in S.vert_pdf.  Returns 1 with the new
// direction, 0 when no vertex passes, the CDF is empty or no round has a
// winner.  `wk` (optional) receives the winner's curvature, `raw` (optional,
// LDS [24]) the vertex supports before the 0.4 cut.
template <bool INIT, bool CNT = false>
__device__ int ptt_substep(const DevParams &P, const DevBufs &B, PttLds &S, float *frame, const float *fr,
                           Philox &rng, float first_val, int first_phase, int rounds, float dx, float dy, float dz,
                           float px, float py, float pz, float *ndx, float *ndy, float *ndz, float *wk, float *raw,
                           uint32_t *ntap = nullptr) {
    const int l = lane32();
    const double mc = (double)P.max_curv;
    float last = 0.0f;
    for (int ph = first_phase; ph <= rounds; ++ph) {
        if (ph == 1) {
            last = ptt_face_cdf(S);
            if (last == 0.0f) return 0;
        }
        float k1 = 0.0f, k2 = 0.0f;
        bool active = true;
        if (ph == 0) {
            active = l < DISC_VERT_CNT;
            if (active) {
                if (B.vprop) {
                    k1 = B.vprop[VPROP_K + 2 * l];
                    k2 = B.vprop[VPROP_K + 2 * l + 1];
                } else {
                    k1 = (float)((double)c_disc_vert[2 * l] * mc);
                    k2 = (float)((double)c_disc_vert[2 * l + 1] * mc);
                }
            }
        } else {
            float r1 = rng.uniform(), r2 = rng.uniform();
            if (r1 + r2 > 1.0f) { r1 = 1.0f - r1; r2 = 1.0f - r2; }
            const float tmp = rng.uniform() * last;
            // first face jj < 30 with cdf >= tmp, else the last (the
            // reference's linear scan): the cdf is a prefix sum of values
            // >= 0, so it never decreases and a binary search finds the same
            // face in 5 reads (a NaN tmp fails every test in both)
            int jj = 0, hi = DISC_FACE_CNT - 1;
            while (jj < hi) {
                const int mid = (jj + hi) >> 1;
                if (S.face_cdf[mid] >= tmp) hi = mid; else jj = mid + 1;
            }
            const int f0 = c_disc_face[jj * 3], f1 = c_disc_face[jj * 3 + 1], f2 = c_disc_face[jj * 3 + 2];
            float vx0, vx1, vx2, vy0, vy1, vy2;
            if (B.vprop) {  // the same products, computed once per tracker
                const float *vk = B.vprop + VPROP_K;
                vx0 = vk[2 * f0]; vx1 = vk[2 * f1]; vx2 = vk[2 * f2];
                vy0 = vk[2 * f0 + 1]; vy1 = vk[2 * f1 + 1]; vy2 = vk[2 * f2 + 1];
            } else {
                vx0 = (float)(mc * (double)c_disc_vert[f0 * 2]);
                vx1 = (float)(mc * (double)c_disc_vert[f1 * 2]);
                vx2 = (float)(mc * (double)c_disc_vert[f2 * 2]);
                vy0 = (float)(mc * (double)c_disc_vert[f0 * 2 + 1]);
                vy1 = (float)(mc * (double)c_disc_vert[f1 * 2 + 1]);
                vy2 = (float)(mc * (double)c_disc_vert[f2 * 2 + 1]);
            }
            k1 = __builtin_fmaf(r2, vx2 - vx0, __builtin_fmaf(r1, vx1 - vx0, vx0));
            k2 = __builtin_fmaf(r2, vy2 - vy0, __builtin_fmaf(r1, vy1 - vy0, vy0));
        }
        float pf[9];
        float sup = 0.0f;
        if (active) {
            probing_frame<INIT>(fr, rng, pf);
            // rejection rounds of a non-initial sub-step only test sup >= min_support_f
            const float stop_at = (ph >= 1 && !INIT && P.ptt_nonneg) ? P.min_support_f : __builtin_inff();
            // the vertex phase's curves are the disc vertices: their one-step
            // propagators are the same at every sub-step (computed once by
            // vertex_propagators with the same prepare_propagator)
            sup = data_support(P, B, first_val, px, py, pz, k1, k2, pf, stop_at, CNT ? ntap : nullptr,
                               (ph == 0 && B.vprop) ? B.vprop + 9 * l : nullptr);
        }
        if (ph == 0) {
            const bool ok = active && !(sup < P.min_support_f);
            if (active) {
                S.vert_pdf[l] = ok ? sup : 0.0f;
                if (raw) raw[l] = sup;
            }
            if (half_ballot(ok) == 0u) return 0;
            WAVE_SYNC();
            continue;
        }
        uint32_t msk;
        if (INIT) {
            float mx = sup;
            for (int m = 16; m; m >>= 1) mx = fmaxf(mx, shfl_xor32(mx, m));
            msk = half_ballot(sup == mx && mx >= P.min_support_f);
        } else {
            // >= as ptt.cu:384: a NaN support never wins a round (the vertex
            // phase above keeps the reference's `<` test, which lets it in)
            msk = half_ballot(sup >= P.min_support_f);
        }
        if (msk != 0u) {
            const int win = __ffs(msk) - 1;
            float ox = dx, oy = dy, oz = dz;
            if (l == win) {
                if (!INIT) {
                    float prop[9], d[3];
                    prepare_propagator(k1, k2, P.ptt_sub_step, prop);
#pragma unroll
                    for (int i = 0; i < 9; ++i) pf[i] = fr[i];
                    propagate_frame(prop, pf, d);
                    norm3<0>(d[0], d[1], d[2]);
                    ox = d[0]; oy = d[1]; oz = d[2];
                }
#pragma unroll
                for (int i = 0; i < 9; ++i) frame[i] = pf[i];
            }
            *ndx = shfl32(ox, win);
            *ndy = shfl32(oy, win);
            *ndz = shfl32(oz, win);
            if (wk) { wk[0] = shfl32(k1, win); wk[1] = shfl32(k2, win); }
            WAVE_SYNC();
            return 1;
        }
    }
    return 0;
}

// get_direction_ptt_d (ptt.cu:194-412); `frame` is the 9-float frame in use.
// CNT (instrumented kernels): every tap read is counted in *ntap.
template <bool INIT, bool CNT = false>
__device__ int get_direction_ptt(const DevParams &P, const DevBufs &B, PttLds &S, float *frame,
                                 Philox &rng, float dx, float dy, float dz, float px, float py, float pz,
                                 float *ndx, float *ndy, float *ndz, float *wk = nullptr, float *raw = nullptr,
                                 uint32_t *ntap = nullptr) {
    const int l = lane32();
    if (INIT) {
        if (l == 0) { frame[0] = dx; frame[1] = dy; frame[2] = dz; }
        WAVE_SYNC();
    }
    float fr[9];
#pragma unroll
    for (int i = 0; i < 9; ++i) fr[i] = frame[i];
    const float first_val = interp4(P, B, px, py, pz, fr[0], fr[1], fr[2]);
    if (CNT) ++*ntap;
    return ptt_substep<INIT, CNT>(P, B, S, frame, fr, rng, first_val, 0, 1024 / 32, dx, dy, dz, px, py, pz, ndx, ndy,
                                  ndz, wk, raw, ntap);
}

// init_frame_ptt_d (ptt.cu:415-474); frame[15..17] is set to the binormal.
template <bool CNT = false>
__device__ bool init_frame_ptt(const DevParams &P, const DevBufs &B, PttLds &S, Philox &rng,
                               float fx, float fy, float fz, float sx, float sy, float sz, uint32_t *ntap = nullptr) {
    const int l = lane32();
    float tx, ty, tz;
    int att = 0;
    bool ok = false;
    for (; att < 2; ++att) {  // +dir first, then -dir
        const float sg = att ? -1.0f : 1.0f;
        ok = get_direction_ptt<true, CNT>(P, B, S, S.frame, rng, sg * fx, sg * fy, sg * fz, sx, sy, sz, &tx, &ty, &tz,
                                          nullptr, nullptr, ntap);
        if (ok) break;
    }
    if (!ok) return false;
    if (l == 0) {
        if (att == 0)
            for (int i = 0; i < 6; ++i) S.frame[i] = -S.frame[i];
        for (int i = 0; i < 6; ++i) S.frame[9 + i] = -S.frame[i];
        for (int i = 0; i < 3; ++i) S.frame[15 + i] = S.frame[6 + i];
    }
    WAVE_SYNC();
    return true;
}

// -------------------------------------------------------------------------
// Learned PTT proposal (no counterpart in the reference).
//
// The network predicts the 24 vertex supports that the plain getter measures
// with 8 probe taps each, from two taps per vertex; the reference's face CDF
// and acceptance rule then run on the prediction.  The MLP runs on the 32
// lanes of the seed slot: lane l owns hidden neurons l, l+32, l+64, l+96 and
// output l; each neuron is an fma chain over its inputs in order, starting
// from the bias.  Parameters are bf16, arithmetic fp32.
// -------------------------------------------------------------------------
constexpr int MLP_IN = CUSLINES_MLP_IN, MLP_H = CUSLINES_MLP_HIDDEN, MLP_OUT = CUSLINES_MLP_OUT;
constexpr int MLP_W1 = 0, MLP_B1 = MLP_W1 + MLP_H * MLP_IN, MLP_W2 = MLP_B1 + MLP_H,
              MLP_B2 = MLP_W2 + MLP_H * MLP_H, MLP_W3 = MLP_B2 + MLP_H, MLP_B3 = MLP_W3 + MLP_OUT * MLP_H,
              MLP_NPARAM = MLP_B3 + MLP_OUT;
// The network as the tracking kernel reads it: each weight matrix stored
// lane-interleaved (mlp_il_offset: the 8-weight pieces of 32 consecutive
// rows side by side, rows padded to 32), so lane j's 16-byte row loads of
// one instruction are 512 contiguous bytes; biases after the matrices.
constexpr int MLP_OUT32 = 32;
constexpr int IL_W1 = 0, IL_W2 = IL_W1 + MLP_H * MLP_IN, IL_W3 = IL_W2 + MLP_H * MLP_H,
              IL_B1 = IL_W3 + MLP_OUT32 * MLP_H, IL_B2 = IL_B1 + MLP_H, IL_B3 = IL_B2 + MLP_H,
              IL_NPARAM = IL_B3 + MLP_OUT32;
constexpr int MLP_LDS_FLOATS = ((IL_NPARAM + 1) / 2 + 3) & ~3;  // the network staged in LDS (learned kernels)
__host__ __device__ inline int mlp_il_offset(int K, int j, int k) {
    return (((j >> 5) * (K >> 3) + (k >> 3)) << 8) + ((j & 31) << 3) + (k & 7);
}
static_assert(MLP_NPARAM == CUSLINES_MLP_NPARAM, "MLP layout");
static_assert(MLP_OUT == DISC_VERT_CNT, "one output per disc vertex");
constexpr int ACT_X = 0, ACT_H1 = 64, ACT_H2 = 192, ACT_O = 320, ACT_FLOATS = 352;
constexpr int PTT_SLOT_FLOATS = 96 + ACT_FLOATS;
constexpr int FEAT_STEPS = 4;  // probe steps between the two feature taps

__device__ __forceinline__ float bf16f(uint32_t h) { return __uint_as_float(h << 16); }

// Inputs at the start of a sub-step into x[0..39] (LDS).  Lane v < 24: ODF
// taps after 4 and 8 probe steps along vertex v's curve (one propagator of
// arc length 4 probe steps, applied twice), summed.
__device__ __forceinline__ void mlp_features(const DevParams &P, const DevBufs &B, float px, float py, float pz,
                                             float dx, float dy, float dz, const float *fr, float first_val,
                                             float *x) {
    const int l = lane32();
    if (l < DISC_VERT_CNT) {
        float pf[9], prop[9], d[3];
#pragma unroll
        for (int i = 0; i < 9; ++i) pf[i] = fr[i];
#pragma unroll
        for (int i = 0; i < 9; ++i) prop[i] = B.fprop[9 * l + i];
        // both frames first (they do not depend on the taps), then both LUT
        // reads, then both block reads, so the two taps' loads overlap
        propagate_frame(prop, pf, d);
        const float q1x = px + d[0], q1y = py + d[1], q1z = pz + d[2];
        const uint32_t lv1 = B.lut[lut_index(P, pf[0], pf[1], pf[2])];
        propagate_frame(prop, pf, d);
        const float q2x = q1x + d[0], q2y = q1y + d[1], q2z = q1z + d[2];
        const uint32_t lv2 = B.lut[lut_index(P, pf[0], pf[1], pf[2])];
        const Tap a = tap_begin(P, B, lv1, q1x, q1y, q1z);
        const Tap b = tap_begin(P, B, lv2, q2x, q2y, q2z);
        const float t1 = tap_end(P, B, a);
        const float t2 = tap_end(P, B, b);
        x[l] = t1 + t2;
    } else if (l == DISC_VERT_CNT) {
        x[l] = first_val;
    } else if (l < 28) {
        x[l] = 0.0f;
    } else if (l < 31) {
        x[l] = (l == 28) ? dx : (l == 29) ? dy : dz;
    }
    if (l < 9) x[31 + l] = fr[l];
    WAVE_SYNC();
}

// One neuron: bias + sum_k w[k] in[k] as an fma chain, K a multiple of 8.
// Address-space-qualified pointers for the out-of-line network: its
// arguments arrive as generic pointers, and generic (flat) loads are slower
// than ds loads.  The learned kernels stage the network in LDS
// (stage_network), so weights and activations are both LDS reads.
#define AS_LDS __attribute__((address_space(3)))
typedef const AS_LDS uint16_t GWeight;
typedef AS_LDS float LAct;
typedef float vf4 __attribute__((ext_vector_type(4)));
typedef uint32_t vu4 __attribute__((ext_vector_type(4)));

// Four neurons of one lane (rows j, j + 32, j + 64, j + 96 of the layer),
// each summed in input order like a single neuron; w: row j in the
// lane-interleaved layout (mlp_il_offset(K, j, 0)), the other rows 32 rows
// further, i.e. (K / 8) * 256 weights on.
template <int K>
__device__ __forceinline__ void mlp_neuron4(GWeight *__restrict__ w, GWeight *bias, const LAct *in, float *acc) {
    const AS_LDS vu4 *w8 = reinterpret_cast<const AS_LDS vu4 *>(w);
#pragma unroll
    for (int r = 0; r < 4; ++r) acc[r] = bf16f(bias[32 * r]);
#pragma unroll 2
    for (int k8 = 0; k8 < K / 8; ++k8) {
        const vf4 a = *reinterpret_cast<const AS_LDS vf4 *>(in + 8 * k8);
        const vf4 b = *reinterpret_cast<const AS_LDS vf4 *>(in + 8 * k8 + 4);
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const vu4 q = w8[k8 * 32 + r * (K / 8) * 32];
            float c = acc[r];
            c = __builtin_fmaf(bf16f(q.x & 0xffffu), a.x, c);
            c = __builtin_fmaf(bf16f(q.x >> 16), a.y, c);
            c = __builtin_fmaf(bf16f(q.y & 0xffffu), a.z, c);
            c = __builtin_fmaf(bf16f(q.y >> 16), a.w, c);
            c = __builtin_fmaf(bf16f(q.z & 0xffffu), b.x, c);
            c = __builtin_fmaf(bf16f(q.z >> 16), b.y, c);
            c = __builtin_fmaf(bf16f(q.w & 0xffffu), b.z, c);
            c = __builtin_fmaf(bf16f(q.w >> 16), b.w, c);
            acc[r] = c;
        }
    }
}

// w: the neuron's row in the lane-interleaved layout (mlp_il_offset(K, j, 0)).
template <int K>
__device__ __forceinline__ float mlp_neuron(GWeight *__restrict__ w, uint16_t bias, const LAct *in) {
    float acc = bf16f(bias);
    const AS_LDS vu4 *w8 = reinterpret_cast<const AS_LDS vu4 *>(w);
#pragma unroll 2
    for (int k8 = 0; k8 < K / 8; ++k8) {
        const vu4 q = w8[k8 * 32];
        const vf4 a = *reinterpret_cast<const AS_LDS vf4 *>(in + 8 * k8);
        const vf4 b = *reinterpret_cast<const AS_LDS vf4 *>(in + 8 * k8 + 4);
        acc = __builtin_fmaf(bf16f(q.x & 0xffffu), a.x, acc);
        acc = __builtin_fmaf(bf16f(q.x >> 16), a.y, acc);
        acc = __builtin_fmaf(bf16f(q.y & 0xffffu), a.z, acc);
        acc = __builtin_fmaf(bf16f(q.y >> 16), a.w, acc);
        acc = __builtin_fmaf(bf16f(q.z & 0xffffu), b.x, acc);
        acc = __builtin_fmaf(bf16f(q.z >> 16), b.y, acc);
        acc = __builtin_fmaf(bf16f(q.w & 0xffffu), b.z, acc);
        acc = __builtin_fmaf(bf16f(q.w >> 16), b.w, acc);
    }
    return acc;
}

// Kept out of line so the tracking loop keeps its register budget.  Both
// W_generic (the staged network) and act_generic (the slot's activations)
// point into LDS.
__device__ __noinline__ void mlp_forward(const uint16_t *__restrict__ W_generic, float *act_generic) {
    GWeight *W = (GWeight *)W_generic;
    LAct *act = (LAct *)act_generic;
    const int l = lane32();
    float v[4];
    mlp_neuron4<MLP_IN>(W + IL_W1 + mlp_il_offset(MLP_IN, l, 0), W + IL_B1 + l, act + ACT_X, v);
#pragma unroll
    for (int r = 0; r < 4; ++r) act[ACT_H1 + l + 32 * r] = (v[r] > 0.0f) ? v[r] : 0.0f;
    WAVE_SYNC();
    mlp_neuron4<MLP_H>(W + IL_W2 + mlp_il_offset(MLP_H, l, 0), W + IL_B2 + l, act + ACT_H1, v);
#pragma unroll
    for (int r = 0; r < 4; ++r) act[ACT_H2 + l + 32 * r] = (v[r] > 0.0f) ? v[r] : 0.0f;
    WAVE_SYNC();
    if (l < MLP_OUT)
        act[ACT_O + l] = mlp_neuron<MLP_H>(W + IL_W3 + mlp_il_offset(MLP_H, l, 0), W[IL_B3 + l], act + ACT_H2);
    WAVE_SYNC();
}

// Learned proposal with an exact correction.  The reference draws a face
// with probability proportional to its value F (the sum of its 3 vertex
// supports, 0 when one is below 0.4) and a point uniform in it, then keeps
// the lowest lane whose candidate has support >= 0.4 (ptt.cu:270-410).  Here
// the face is drawn from the network's estimate instead,
//   g(f) = sum of the 3 predicted supports (clipped at 0) + a floor
//          (PROPOSAL_FLOOR x the mean predicted face value),
// and accepted with probability F(f) / (PROPOSAL_M g(f)) before the
// reference's support test; F(f) needs only the exact supports of the drawn
// faces' vertices (8 probes each, measured once per sub-step and shared by
// the lanes).  An accepted candidate is then distributed as F(f) x uniform
// x [support >= 0.4], the reference's sampler, whenever F <= PROPOSAL_M g
// on every face; draws where that bound fails are counted (stats[3]).
// Up to LEARNED_ROUNDS rounds of 32 candidates, then the plain sub-step.
constexpr float PROPOSAL_M = 2.0f;
constexpr float PROPOSAL_FLOOR = 0.5f;
constexpr int LEARNED_ROUNDS = 4;

// Inclusive prefix sum over the 31 faces (lanes >= 31 keep 0), the
// Hillis-Steele order of ptt_face_cdf; returns the total on every lane.
__device__ __forceinline__ float face_scan(float v, float *out) {
    const int l = lane32();
    if (l >= DISC_FACE_CNT) v = 0.0f;
#pragma unroll
    for (int i = 1; i < 32; i <<= 1) {
        const float o = shfl_up32(v, i);
        if (l >= i && l < DISC_FACE_CNT) v = v + o;
    }
    if (out && l < DISC_FACE_CNT) out[l] = v;
    return shfl32(v, DISC_FACE_CNT - 1);
}

__device__ int get_direction_ptt_learned(const DevParams &P, const DevBufs &B, PttLds &S, float *frame, Philox &rng,
                                         bool learned, float dx, float dy, float dz, float px, float py, float pz,
                                         float *ndx, float *ndy, float *ndz, int *fell, uint32_t *misses) {
    const int l = lane32();
    float fr[9];
#pragma unroll
    for (int i = 0; i < 9; ++i) fr[i] = frame[i];
    const float first_val = interp4(P, B, px, py, pz, fr[0], fr[1], fr[2]);
    *fell = 0;
    if (learned) {
        mlp_features(P, B, px, py, pz, dx, dy, dz, fr, first_val, S.act + ACT_X);
        mlp_forward(B.mlp, S.act);
        float *E = S.act + ACT_X;   // exact vertex supports (the inputs are dead now)
        float *G = S.act + ACT_H1;  // proposal face values (so are the hidden activations)
        float gh = 0.0f;
        if (l < DISC_FACE_CNT) {
#pragma unroll
            for (int jj = 0; jj < 3; ++jj) {
                const float sv = S.act[ACT_O + c_disc_face[l * 3 + jj]];
                gh = gh + ((sv > 0.0f) ? sv : 0.0f);
            }
        }
        const float tot = face_scan(gh, nullptr);
        const float g = gh + (PROPOSAL_FLOOR * (tot / (float)DISC_FACE_CNT) + 1e-3f);
        if (l < DISC_FACE_CNT) G[l] = g;
        const float last = face_scan(g, S.face_cdf);
        WAVE_SYNC();
        const double mc = (double)P.max_curv;
        uint32_t known = 0u;
        for (int round = 0; round < LEARNED_ROUNDS; ++round) {
            float r1 = rng.uniform(), r2 = rng.uniform();
            if (r1 + r2 > 1.0f) { r1 = 1.0f - r1; r2 = 1.0f - r2; }
            const float tmp = rng.uniform() * last;
            const float ua = rng.uniform();
            int jj = 0, hi = DISC_FACE_CNT - 1;
            while (jj < hi) {
                const int mid = (jj + hi) >> 1;
                if (S.face_cdf[mid] >= tmp) hi = mid; else jj = mid + 1;
            }
            const int f0 = c_disc_face[jj * 3], f1 = c_disc_face[jj * 3 + 1], f2 = c_disc_face[jj * 3 + 2];
            uint32_t need = (1u << f0) | (1u << f1) | (1u << f2);
#pragma unroll
            for (int m = 16; m; m >>= 1) need |= (uint32_t)shfl_xor32((int)need, m);
            const uint32_t todo = need & ~known;
            if (l < DISC_VERT_CNT && ((todo >> l) & 1u)) {
                float pf[9];
#pragma unroll
                for (int i = 0; i < 9; ++i) pf[i] = fr[i];
                const float k1v = (float)((double)c_disc_vert[2 * l] * mc);
                const float k2v = (float)((double)c_disc_vert[2 * l + 1] * mc);
                E[l] = data_support(P, B, first_val, px, py, pz, k1v, k2v, pf, __builtin_inff(), nullptr,
                                    B.vprop ? B.vprop + 9 * l : nullptr);
            }
            known |= need;
            WAVE_SYNC();
            // the reference's face value from the exact supports (vertex
            // phase test `< 0.4`, ptt_face_cdf's zero rule)
            float F = 0.0f;
#pragma unroll
            for (int q = 0; q < 3; ++q) {
                const float e = E[c_disc_face[jj * 3 + q]];
                const float vv = (e < P.min_support_f) ? 0.0f : e;
                if (vv == 0.0f) { F = 0.0f; break; }
                F = F + vv;
            }
            const float mg = PROPOSAL_M * G[jj];
            const bool acc = ua * mg < F;
            const float vx0 = (float)(mc * (double)c_disc_vert[f0 * 2]);
            const float vx1 = (float)(mc * (double)c_disc_vert[f1 * 2]);
            const float vx2 = (float)(mc * (double)c_disc_vert[f2 * 2]);
            const float vy0 = (float)(mc * (double)c_disc_vert[f0 * 2 + 1]);
            const float vy1 = (float)(mc * (double)c_disc_vert[f1 * 2 + 1]);
            const float vy2 = (float)(mc * (double)c_disc_vert[f2 * 2 + 1]);
            const float k1 = __builtin_fmaf(r2, vx2 - vx0, __builtin_fmaf(r1, vx1 - vx0, vx0));
            const float k2 = __builtin_fmaf(r2, vy2 - vy0, __builtin_fmaf(r1, vy1 - vy0, vy0));
            float sup = 0.0f;
            if (acc) {
                float pf[9];
#pragma unroll
                for (int i = 0; i < 9; ++i) pf[i] = fr[i];
                const float stop_at = P.ptt_nonneg ? P.min_support_f : __builtin_inff();
                sup = data_support(P, B, first_val, px, py, pz, k1, k2, pf, stop_at);
            }
            *misses += (uint32_t)__popc(half_ballot(F > mg));
            const uint32_t msk = half_ballot(acc && sup >= P.min_support_f);
            if (msk != 0u) {
                const int win = __ffs(msk) - 1;
                float ox = dx, oy = dy, oz = dz;
                if (l == win) {
                    float prop[9], d[3], pf[9];
                    prepare_propagator(k1, k2, P.ptt_sub_step, prop);
#pragma unroll
                    for (int i = 0; i < 9; ++i) pf[i] = fr[i];
                    propagate_frame(prop, pf, d);
                    norm3<0>(d[0], d[1], d[2]);
                    ox = d[0]; oy = d[1]; oz = d[2];
#pragma unroll
                    for (int i = 0; i < 9; ++i) frame[i] = pf[i];
                }
                *ndx = shfl32(ox, win);
                *ndy = shfl32(oy, win);
                *ndz = shfl32(oz, win);
                WAVE_SYNC();
                return 1;
            }
        }
        *fell = 1;
    }
    return ptt_substep<false>(P, B, S, frame, fr, rng, first_val, 0, 1024 / 32, dx, dy, dz, px, py, pz, ndx, ndy,
                              ndz, nullptr, nullptr);
}

// Training pair of a plain sub-step: inputs at the sub-step's start and the
// 24 measured vertex supports.
__device__ void record_pair(const DevParams &P, const DevBufs &B, PttLds &S, float px, float py, float pz, float dx,
                            float dy, float dz, const float *fr0, const float *raw) {
    const int l = lane32();
    const float first_val = interp4(P, B, px, py, pz, fr0[0], fr0[1], fr0[2]);
    mlp_features(P, B, px, py, pz, dx, dy, dz, fr0, first_val, S.act + ACT_X);
    int idx = 0;
    if (l == 0) idx = atomicAdd(B.rec_count, 1);
    idx = shfl32(idx, 0);
    if (idx < P.rec_cap) {
        float *o = B.rec + (size_t)idx * CUSLINES_PAIR_FLOATS;
        for (int j = l; j < MLP_IN; j += 32) o[j] = S.act[ACT_X + j];
        if (l < DISC_VERT_CNT) o[MLP_IN + l] = raw[l];
    }
    WAVE_SYNC();
}

__device__ __forceinline__ uint32_t mix32(uint32_t h) {  // murmur3 finaliser
    h ^= h >> 16; h *= 0x85ebca6bu; h ^= h >> 13; h *= 0xc2b2ae35u; h ^= h >> 16;
    return h;
}

// -------------------------------------------------------------------------
// Tracker (generate_streamlines_cuda.cu:277-421, boot.cu:720-824)
// -------------------------------------------------------------------------
struct SlotLds {
    ProbLds prob;
    BootLds boot;
    PttLds ptt;
};

// V (PTT only): 0 plain getter, 1 learned proposal, 2 plain getter recording
// training pairs (tag identifies seed, direction and pass for the hash), 3
// plain getter counting its taps and sub-steps into *ntap and *nsub.
template <int MODEL, int V = 0>
__device__ int tracker(const DevParams &P, const DevBufs &B, const float *sv, SlotLds &S,
                       typename SlotRng<MODEL>::type &rng, float sx, float sy, float sz, float dx, float dy, float dz, float *frame,
                       float *__restrict__ sl, uint32_t tag = 0, uint32_t *ntap = nullptr,
                       uint32_t *nsub = nullptr) {
    const int l = lane32();
    const int step_frac = (MODEL == CUSLINES_PTT) ? P.step_frac : 1;
    const int MAXL = P.max_sline_len;
    const double sub = P.step_d / (double)step_frac;
    float px = sx, py = sy, pz = sz;
    if (l == 0) { sl[0] = px; sl[1] = py; sl[2] = pz; }
    int ltries = 0, lfalls = 0, nplain = 0;
    uint32_t lmiss = 0;
    bool learned = (V == 1);
    int i;
    for (i = 1; i < MAXL * step_frac; ++i) {
        float nx = 0.0f, ny = 0.0f, nz = 0.0f;
        int ndir;
        if constexpr (MODEL == CUSLINES_PROB)
            ndir = get_direction_prob<false>(P, B, sv, S.prob, rng, dx, dy, dz, px, py, pz, &nx, &ny, &nz);
        else if constexpr (MODEL == CUSLINES_PTT && V == 1) {
            int fell = 0;
            ndir = get_direction_ptt_learned(P, B, S.ptt, frame, rng, learned, dx, dy, dz, px, py, pz, &nx, &ny, &nz,
                                             &fell, &lmiss);
            if (learned) {
                ++ltries;
                lfalls += fell;
                if (ltries >= 16 && 4 * lfalls > ltries) learned = false;
            } else {
                ++nplain;
            }
        } else if constexpr (MODEL == CUSLINES_PTT && V == 2) {
            float fr0[9];
#pragma unroll
            for (int q = 0; q < 9; ++q) fr0[q] = frame[q];
            const bool rec = mix32(tag * 0x9E3779B1u + (uint32_t)i) < P.rec_thresh;
            ndir = get_direction_ptt<false>(P, B, S.ptt, frame, rng, dx, dy, dz, px, py, pz, &nx, &ny, &nz, nullptr,
                                            rec ? S.ptt.act + ACT_O : nullptr);
            if (rec) record_pair(P, B, S.ptt, px, py, pz, dx, dy, dz, fr0, S.ptt.act + ACT_O);
        } else if constexpr (MODEL == CUSLINES_PTT && V == 3) {
            ++*nsub;
            ndir = get_direction_ptt<false, true>(P, B, S.ptt, frame, rng, dx, dy, dz, px, py, pz, &nx, &ny, &nz,
                                                  nullptr, nullptr, ntap);
        } else if constexpr (MODEL == CUSLINES_PTT)
            ndir = get_direction_ptt<false>(P, B, S.ptt, frame, rng, dx, dy, dz, px, py, pz, &nx, &ny, &nz);
        else
            ndir = get_direction_boot<MODEL>(P, B, sv, S.boot, rng, 5, dx, dy, dz, px, py, pz, &nx, &ny, &nz);
        if (ndir == 0) break;
        dx = nx; dy = ny; dz = nz;
        px = (float)__builtin_fma((double)(dx / 1.0f), sub, (double)px);
        py = (float)__builtin_fma((double)(dy / 1.0f), sub, (double)py);
        pz = (float)__builtin_fma((double)(dz / 1.0f), sub, (double)pz);
        if (l == 0 && (i % step_frac) == 0) {
            float *o = sl + 3 * (size_t)(i / step_frac);
            o[0] = px; o[1] = py; o[2] = pz;
        }
        const int tissue = check_point(P, B.stop, px, py, pz);
        if (tissue == CUSLINES_ENDPOINT || tissue == CUSLINES_INVALIDPOINT || tissue == CUSLINES_OUTSIDEIMAGE)
            break;
    }
    if (V == 1 && B.stats && l == 0) {
        atomicAdd(B.stats, (unsigned long long)(ltries - lfalls));
        atomicAdd(B.stats + 1, (unsigned long long)lfalls);
        atomicAdd(B.stats + 2, (unsigned long long)nplain);
        atomicAdd(B.stats + 3, (unsigned long long)lmiss);
    }
    int nsteps = i / step_frac;
    if ((i % step_frac) != 0 && i < step_frac * (MAXL - 1)) {
        ++nsteps;
        if (l == 0) {
            float *o = sl + 3 * (size_t)nsteps;
            o[0] = px; o[1] = py; o[2] = pz;
        }
    }
    return nsteps;
}

// -------------------------------------------------------------------------
// PTT with L lanes per seed (L in {8, 16, 32}; 64/L seeds per wave).
//
// The reference gives every seed 32 lanes, each with its own Philox stream
// (subsequence 32*slot + lane + 1).  Here those 32 streams are virtual lanes
// whose state -- the next draw index k and, for a cached Box-Muller value,
// the index c of the draw pair it came from (-1: none) -- lives in LDS, and
// draws are computed from (subsequence, k) directly (counter-based Philox).
// A physical lane p evaluates virtual lanes p, p+L, p+2L, ... in batches.
//  - vertex phase: all 24 candidates (their supports build the face CDF);
//  - INIT rejection: all 32 candidates (the winner is the arg-max);
//  - non-INIT rejection: batches in lane order, stopping at the first batch
//    that holds a candidate with enough support.  The winner is the lowest
//    virtual lane that passes, as in the reference, and every virtual lane's
//    stream still advances by its 3 uniforms per round.
// The vertex propagators depend only on the disc and MAX_CURVATURE and are
// computed once per block.
// -------------------------------------------------------------------------
template <int L>
struct Grp {
    static __device__ __forceinline__ int lane() { return threadIdx.x & (L - 1); }
    static __device__ __forceinline__ uint32_t ballot(bool p) {
        const unsigned long long b = __ballot(p);
        const int base = (threadIdx.x & 63) & ~(L - 1);
        return (uint32_t)((b >> base) & (L == 32 ? 0xffffffffull : ((1ull << L) - 1)));
    }
    static __device__ __forceinline__ float shfl(float v, int src) { return __shfl(v, src, L); }
    static __device__ __forceinline__ int shfl(int v, int src) { return __shfl(v, src, L); }
    static __device__ __forceinline__ float shfl_xor(float v, int m) { return __shfl_xor(v, m, L); }
    static __device__ __forceinline__ int shfl_xor(int v, int m) { return __shfl_xor(v, m, L); }
};

// Philox draw k of subsequence `sub`, with a one-block cache per lane.
struct DrawCache {
    uint32_t sub, blk, r0, r1, r2, r3;
    int valid;
};

__device__ __forceinline__ uint32_t philox_draw(uint32_t key0, uint32_t key1, uint32_t sub, uint32_t k,
                                                DrawCache &dc) {
    const uint32_t blk = k >> 2;
    if (!(dc.valid && dc.sub == sub && dc.blk == blk)) {
        uint32_t x0 = blk, x1 = 0, x2 = sub, x3 = 0;
        uint32_t a = key0, b = key1;
#pragma unroll
        for (int r = 0; r < 10; ++r) {
            const uint32_t lo0 = 0xD2511F53u * x0, hi0 = __umulhi(0xD2511F53u, x0);
            const uint32_t lo1 = 0xCD9E8D57u * x2, hi1 = __umulhi(0xCD9E8D57u, x2);
            const uint32_t n0 = hi1 ^ x1 ^ a, n2 = hi0 ^ x3 ^ b;
            x0 = n0; x1 = lo1; x2 = n2; x3 = lo0;
            a += 0x9E3779B9u;
            b += 0xBB67AE85u;
        }
        dc.r0 = x0; dc.r1 = x1; dc.r2 = x2; dc.r3 = x3;
        dc.sub = sub; dc.blk = blk; dc.valid = 1;
    }
    const int w = k & 3;
    return (w == 0) ? dc.r0 : (w == 1) ? dc.r1 : (w == 2) ? dc.r2 : dc.r3;
}

__device__ __forceinline__ float uniform_of(uint32_t x) { return 2.32830644e-10f + (float)x * 2.32830644e-10f; }

// Box-Muller pair of draws (x, y): the sine term is returned first and the
// cosine term cached, as Philox::normal does.
__device__ __forceinline__ void box_muller(uint32_t x, uint32_t y, float *sn_out, float *cs_out) {
    const float u = 2.32830644e-10f + (float)x * 2.32830644e-10f;
    const float v = 1.46291807e-09f + (float)y * 1.46291807e-09f;
    const float s = __builtin_sqrtf(-2.0f * ulog(u));
    float sn, cs;
    usincos(v, &sn, &cs);
    *sn_out = sn * s;
    *cs_out = cs * s;
}

struct VLane {
    uint32_t key0, key1, sub;  // stream of this virtual lane
    uint32_t k;                // next draw index
    int c;                     // draw pair of the cached normal, -1 if none
    __device__ __forceinline__ float uniform(DrawCache &dc) { return uniform_of(philox_draw(key0, key1, sub, k++, dc)); }
    __device__ __forceinline__ float normal(DrawCache &dc) {
        float sn, cs;
        if (c >= 0) {
            box_muller(philox_draw(key0, key1, sub, (uint32_t)c, dc), philox_draw(key0, key1, sub, (uint32_t)c + 1, dc),
                       &sn, &cs);
            c = -1;
            return cs;
        }
        box_muller(philox_draw(key0, key1, sub, k, dc), philox_draw(key0, key1, sub, k + 1, dc), &sn, &cs);
        c = (int)k;
        k += 2;
        return sn;
    }
};

// LDS of one PTT seed group.
struct PttG {
    float *frame;     // 18
    float *vert_pdf;  // 24
    float *face_cdf;  // 32
    uint32_t *rk;     // 32 virtual-lane draw indices
    int *rc;          // 32 cached-normal pair indices
};
constexpr int PTTG_FLOATS = 160;

// Block-shared constants: 24 vertex propagators (9 each) and the scaled
// disc vertices (MAX_CURVATURE * DISC_VERT, 48).
struct PttConst {
    float *vprop;  // 24 * 9
    float *vk;     // 48
};
constexpr int PTTC_FLOATS = 24 * 9 + 48;

__device__ void ptt_const_init(const DevParams &P, PttConst &C) {
    const double mc = (double)P.max_curv;
    for (int i = threadIdx.x; i < 48; i += blockDim.x) C.vk[i] = (float)(mc * (double)c_disc_vert[i]);
    for (int i = threadIdx.x; i < 24; i += blockDim.x) {
        const float k1 = (float)((double)c_disc_vert[2 * i] * mc);
        const float k2 = (float)((double)c_disc_vert[2 * i + 1] * mc);
        prepare_propagator(k1, k2, P.probe_step, C.vprop + 9 * i);
    }
}

__device__ __forceinline__ void probe_frame_init(const float *frame, VLane &vl, DrawCache &dc, float *pf) {
    pf[0] = frame[0]; pf[1] = frame[1]; pf[2] = frame[2];
    norm3<0>(pf[0], pf[1], pf[2]);
    pf[3] = vl.normal(dc);
    pf[4] = vl.normal(dc);
    pf[5] = vl.normal(dc);
    const float dt = __builtin_fmaf(pf[5], pf[2], __builtin_fmaf(pf[4], pf[1], pf[3] * pf[0]));
    pf[3] = __builtin_fmaf(-dt, pf[0], pf[3]);
    pf[4] = __builtin_fmaf(-dt, pf[1], pf[4]);
    pf[5] = __builtin_fmaf(-dt, pf[2], pf[5]);
    const float n2 = __builtin_fmaf(pf[5], pf[5], __builtin_fmaf(pf[4], pf[4], pf[3] * pf[3]));
    if (n2 < PTT_NORM_EPS) {
        const float ax = fabsf(pf[0]), ay = fabsf(pf[1]), az = fabsf(pf[2]);
        if (ax <= ay && ax <= az) { pf[3] = 0.0f; pf[4] = pf[2]; pf[5] = -pf[1]; }
        else if (ay <= az) { pf[3] = -pf[2]; pf[4] = 0.0f; pf[5] = pf[0]; }
        else { pf[3] = pf[1]; pf[4] = -pf[0]; pf[5] = 0.0f; }
    }
    norm3<1>(pf[3], pf[4], pf[5]);
    crossnorm3<2>(pf + 6, pf, pf + 3);
}

// Support of one candidate with a precomputed propagator; probing stops
// once the running support reaches `stop_at` (see data_support).
__device__ __forceinline__ float support_prop(const DevParams &P, const DevBufs &B, float support, float px,
                                              float py, float pz, const float *prop, float *pf, float stop_at) {
    for (int i = 0; i < P.probe_quality; ++i) {
        if (support >= stop_at) break;
        float direc[3];
        propagate_frame(prop, pf, direc);
        px += direc[0]; py += direc[1]; pz += direc[2];
        support += interp4(P, B, px, py, pz, pf[0], pf[1], pf[2]);
    }
    return support;
}

template <int L, bool INIT>
__device__ int get_direction_ptt_g(const DevParams &P, const DevBufs &B, const PttConst &K, PttG &S, float *frame,
                                   uint32_t key0, uint32_t key1, uint32_t sub0, DrawCache &dc, float dx, float dy,
                                   float dz, float px, float py, float pz, float *ndx, float *ndy, float *ndz) {
    using G = Grp<L>;
    const int p = G::lane();
    if (INIT) {
        if (p == 0) { frame[0] = dx; frame[1] = dy; frame[2] = dz; }
        WAVE_SYNC();
    }
    float fr[9];
#pragma unroll
    for (int i = 0; i < 9; ++i) fr[i] = frame[i];
    const float first_val = interp4(P, B, px, py, pz, fr[0], fr[1], fr[2]);
    // vertex phase: virtual lanes 0..23
    bool found = false;
    constexpr int NC = (DISC_VERT_CNT + L - 1) / L;  // curves per lane
    if (INIT || NC > 2) {
        for (int v = p; v < DISC_VERT_CNT; v += L) {
            float pf[9];
            if (INIT) {
                VLane vl{key0, key1, sub0 + (uint32_t)v, S.rk[v], S.rc[v]};
                probe_frame_init(fr, vl, dc, pf);
                S.rk[v] = vl.k;
                S.rc[v] = vl.c;
            } else {
#pragma unroll
                for (int i = 0; i < 9; ++i) pf[i] = fr[i];
            }
            const float sup = support_prop(P, B, first_val, px, py, pz, K.vprop + 9 * v, pf, __builtin_inff());
            const bool ok = !(sup < P.min_support_f);
            S.vert_pdf[v] = ok ? sup : 0.0f;
            found |= ok;
        }
    } else {
        // this lane's NC <= 2 curves v = p, p + L probed in lockstep: each
        // probe step issues every curve's LUT read, then every curve's block
        // read, then blends, so the curves' load latencies overlap (with 3
        // curves per lane the registers of three taps in flight spill, which
        // costs more than it hides).  Each curve's arithmetic is
        // support_prop's, in its order.
        float pf[NC][9], qx[NC], qy[NC], qz[NC], sup[NC];
#pragma unroll
        for (int c = 0; c < NC; ++c) {
#pragma unroll
            for (int i = 0; i < 9; ++i) pf[c][i] = fr[i];
            qx[c] = px; qy[c] = py; qz[c] = pz;
            sup[c] = first_val;
        }
        for (int i = 0; i < P.probe_quality; ++i) {
            uint32_t lv[NC];
#pragma unroll
            for (int c = 0; c < NC; ++c) {
                if (p + c * L < DISC_VERT_CNT) {
                    float direc[3];
                    propagate_frame(K.vprop + 9 * (p + c * L), pf[c], direc);
                    qx[c] += direc[0]; qy[c] += direc[1]; qz[c] += direc[2];
                    lv[c] = B.lut[lut_index(P, pf[c][0], pf[c][1], pf[c][2])];
                }
            }
            TapB t[NC];
#pragma unroll
            for (int c = 0; c < NC; ++c)
                if (p + c * L < DISC_VERT_CNT) t[c] = tapb_begin(P, B, lv[c], qx[c], qy[c], qz[c]);
#pragma unroll
            for (int c = 0; c < NC; ++c)
                if (p + c * L < DISC_VERT_CNT) sup[c] += tapb_end(t[c]);
        }
#pragma unroll
        for (int c = 0; c < NC; ++c) {
            const int v = p + c * L;
            if (v < DISC_VERT_CNT) {
                const bool ok = !(sup[c] < P.min_support_f);
                S.vert_pdf[v] = ok ? sup[c] : 0.0f;
                found |= ok;
            }
        }
    }
    if (G::ballot(found) == 0u) return 0;
    WAVE_SYNC();
    // faces and the 32-wide Hillis-Steele scan of prefix_sum_sh_d, per lane
    float cdf[DISC_FACE_CNT];
#pragma unroll
    for (int f = 0; f < DISC_FACE_CNT; ++f) {
        float face = 0.0f;
#pragma unroll
        for (int jj = 0; jj < 3; ++jj) {
            const float vv = S.vert_pdf[c_disc_face[f * 3 + jj]];
            if (vv == 0.0f) { face = 0.0f; break; }
            face = face + vv;
        }
        cdf[f] = face;
    }
#pragma unroll
    for (int d = 1; d < 32; d <<= 1) {
#pragma unroll
        for (int f = DISC_FACE_CNT - 1; f >= d; --f) cdf[f] = cdf[f] + cdf[f - d];
    }
    const float last = cdf[DISC_FACE_CNT - 1];
    if (last == 0.0f) return 0;
    for (int round = 0; round < 1024 / 32; ++round) {
        float best = -__builtin_inff();
        int bestv = -1;
        int win = -1;
        float wk1 = 0.0f, wk2 = 0.0f, wpf[9];
        for (int b = 0; b < 32 / L; ++b) {
            const int v = b * L + p;
            VLane vl{key0, key1, sub0 + (uint32_t)v, S.rk[v], INIT ? S.rc[v] : -1};
            float r1 = vl.uniform(dc), r2 = vl.uniform(dc);
            if (r1 + r2 > 1.0f) { r1 = 1.0f - r1; r2 = 1.0f - r2; }
            const float tmp = vl.uniform(dc) * last;
            int jj = DISC_FACE_CNT - 1;
#pragma unroll
            for (int f = DISC_FACE_CNT - 2; f >= 0; --f)
                if (cdf[f] >= tmp) jj = f;
            const int f0 = c_disc_face[jj * 3], f1 = c_disc_face[jj * 3 + 1], f2 = c_disc_face[jj * 3 + 2];
            const float vx0 = K.vk[f0 * 2], vx1 = K.vk[f1 * 2], vx2 = K.vk[f2 * 2];
            const float vy0 = K.vk[f0 * 2 + 1], vy1 = K.vk[f1 * 2 + 1], vy2 = K.vk[f2 * 2 + 1];
            const float k1 = __builtin_fmaf(r2, vx2 - vx0, __builtin_fmaf(r1, vx1 - vx0, vx0));
            const float k2 = __builtin_fmaf(r2, vy2 - vy0, __builtin_fmaf(r1, vy1 - vy0, vy0));
            float pf[9];
            if (INIT) {
                probe_frame_init(fr, vl, dc, pf);
                S.rk[v] = vl.k;
                S.rc[v] = vl.c;
            } else {
#pragma unroll
                for (int i = 0; i < 9; ++i) pf[i] = fr[i];
            }
            float prop[9];
            prepare_propagator(k1, k2, P.probe_step, prop);
            const float sup = support_prop(P, B, first_val, px, py, pz, prop, pf,
                                           (!INIT && P.ptt_nonneg) ? P.min_support_f : __builtin_inff());
            if (INIT) {
                // batches visit this lane's virtual lanes in increasing order, so
                // keeping the first of equal supports keeps the lowest one
                if (bestv < 0 || sup > best) {
                    best = sup;
                    bestv = v;
#pragma unroll
                    for (int i = 0; i < 9; ++i) wpf[i] = pf[i];
                }
            } else {
                const uint32_t m = G::ballot(sup >= P.min_support_f);
                if (m != 0u) {
                    win = b * L + (__ffs(m) - 1);
                    if (v == win) {
                        wk1 = k1; wk2 = k2;
                    }
                    break;
                }
            }
        }
        if (INIT) {
            // arg-max over the 32 virtual lanes, ties to the lowest virtual lane
            float m = best;
            int mv = bestv;
            for (int o = L / 2; o; o >>= 1) {
                const float om = G::shfl_xor(m, o);
                const int ov = G::shfl_xor(mv, o);
                if (om > m || (om == m && ov < mv)) { m = om; mv = ov; }
            }
            WAVE_SYNC();
            if (m >= P.min_support_f) {
                if (bestv == mv) {
#pragma unroll
                    for (int i = 0; i < 9; ++i) frame[i] = wpf[i];
                }
                *ndx = dx; *ndy = dy; *ndz = dz;
                WAVE_SYNC();
                return 1;
            }
        } else {
            // every virtual lane drew its 3 uniforms this round
            for (int v = p; v < 32; v += L) S.rk[v] += 3u;
            WAVE_SYNC();
            if (win >= 0) {
                float ox = 0.0f, oy = 0.0f, oz = 0.0f;
                if ((win & (L - 1)) == p) {
                    float prop[9], d[3], pf[9];
                    prepare_propagator(wk1, wk2, P.ptt_sub_step, prop);
#pragma unroll
                    for (int i = 0; i < 9; ++i) pf[i] = fr[i];
                    propagate_frame(prop, pf, d);
                    norm3<0>(d[0], d[1], d[2]);
                    ox = d[0]; oy = d[1]; oz = d[2];
#pragma unroll
                    for (int i = 0; i < 9; ++i) frame[i] = pf[i];
                }
                const int wl = win & (L - 1);
                *ndx = G::shfl(ox, wl);
                *ndy = G::shfl(oy, wl);
                *ndz = G::shfl(oz, wl);
                WAVE_SYNC();
                return 1;
            }
        }
    }
    return 0;
}

template <int L>
__device__ bool init_frame_ptt_g(const DevParams &P, const DevBufs &B, const PttConst &K, PttG &S, uint32_t key0,
                                 uint32_t key1, uint32_t sub0, DrawCache &dc, float fx, float fy, float fz, float sx,
                                 float sy, float sz) {
    const int p = Grp<L>::lane();
    float tx, ty, tz;
    int att = 0;
    bool ok = false;
    for (; att < 2; ++att) {
        const float sg = att ? -1.0f : 1.0f;
        ok = get_direction_ptt_g<L, true>(P, B, K, S, S.frame, key0, key1, sub0, dc, sg * fx, sg * fy, sg * fz, sx, sy,
                                          sz, &tx, &ty, &tz);
        if (ok) break;
    }
    if (!ok) return false;
    if (p == 0) {
        if (att == 0)
            for (int i = 0; i < 6; ++i) S.frame[i] = -S.frame[i];
        for (int i = 0; i < 6; ++i) S.frame[9 + i] = -S.frame[i];
        for (int i = 0; i < 3; ++i) S.frame[15 + i] = S.frame[6 + i];
    }
    WAVE_SYNC();
    return true;
}

template <int L>
__device__ int tracker_ptt_g(const DevParams &P, const DevBufs &B, const PttConst &K, PttG &S, float *frame,
                             uint32_t key0, uint32_t key1, uint32_t sub0, DrawCache &dc, float sx, float sy, float sz,
                             float dx, float dy, float dz, float *__restrict__ sl) {
    const int p = Grp<L>::lane();
    const int step_frac = P.step_frac;
    const int MAXL = P.max_sline_len;
    const double sub = P.step_d / (double)step_frac;
    float px = sx, py = sy, pz = sz;
    if (p == 0) { sl[0] = px; sl[1] = py; sl[2] = pz; }
    int i;
    for (i = 1; i < MAXL * step_frac; ++i) {
        float nx = 0.0f, ny = 0.0f, nz = 0.0f;
        const int ndir = get_direction_ptt_g<L, false>(P, B, K, S, frame, key0, key1, sub0, dc, dx, dy, dz, px, py, pz,
                                                       &nx, &ny, &nz);
        if (ndir == 0) break;
        dx = nx; dy = ny; dz = nz;
        px = (float)__builtin_fma((double)(dx / 1.0f), sub, (double)px);
        py = (float)__builtin_fma((double)(dy / 1.0f), sub, (double)py);
        pz = (float)__builtin_fma((double)(dz / 1.0f), sub, (double)pz);
        if (p == 0 && (i % step_frac) == 0) {
            float *o = sl + 3 * (size_t)(i / step_frac);
            o[0] = px; o[1] = py; o[2] = pz;
        }
        const int tissue = check_point(P, B.stop, px, py, pz);
        if (tissue == CUSLINES_ENDPOINT || tissue == CUSLINES_INVALIDPOINT || tissue == CUSLINES_OUTSIDEIMAGE) break;
    }
    int nsteps = i / step_frac;
    if ((i % step_frac) != 0 && i < step_frac * (MAXL - 1)) {
        ++nsteps;
        if (p == 0) {
            float *o = sl + 3 * (size_t)nsteps;
            o[0] = px; o[1] = py; o[2] = pz;
        }
    }
    return nsteps;
}

template <int L>
__device__ void track_seed_ptt_g(const DevParams &P, const DevBufs &B, const PttConst &K, PttG &S, int s,
                                 const float *__restrict__ seeds, int rng_chunk, const int *__restrict__ offsets,
                                 const int *__restrict__ dirs, int *__restrict__ sline_seed, int *__restrict__ sline_len,
                                 float *__restrict__ sline) {
    const int p = Grp<L>::lane();
    const float sx = seeds[3 * s], sy = seeds[3 * s + 1], sz = seeds[3 * s + 2];
    const uint32_t key0 = P.seed_lo, key1 = P.seed_hi;
    const uint32_t sub0 = 32u * (uint32_t)(s % rng_chunk) + 1u;
    for (int v = p; v < 32; v += L) { S.rk[v] = 0u; S.rc[v] = -1; }
    WAVE_SYNC();
    DrawCache dc;
    dc.valid = 0;
    const int ndir = (P.slot_cap > 0 && offsets[s + 1] > P.slot_cap) ? 0 : offsets[s + 1] - offsets[s];
    int off = offsets[s];
    const size_t slot_f = (size_t)2 * P.max_sline_len * 3;
    for (int i = 0; i < ndir; ++i, ++off) {
        const int vi = dirs[(size_t)s * P.nverts + i];
        const float fx = B.verts[3 * vi], fy = B.verts[3 * vi + 1], fz = B.verts[3 * vi + 2];
        float *cur = sline + (size_t)off * slot_f;
        if (p == 0) sline_seed[off] = s;
        if (!init_frame_ptt_g<L>(P, B, K, S, key0, key1, sub0, dc, fx, fy, fz, sx, sy, sz)) {
            if (p == 0) {
                sline_len[off] = 1;
                cur[0] = sx; cur[1] = sy; cur[2] = sz;
            }
            continue;
        }
        int nb = 0, nf = 0;
        for (int pass = 0; pass < 2; ++pass) {
            const float sg = pass ? 1.0f : -1.0f;
            float *out = pass ? cur + 3 * (size_t)(nb - 1) : cur;
            const int ns = tracker_ptt_g<L>(P, B, K, S, S.frame + 9 * pass, key0, key1, sub0, dc, sx, sy, sz, sg * fx,
                                            sg * fy, sg * fz, out);
            if (pass == 0) {
                nb = ns;
                MEM_SYNC();
                for (int j = p; j < nb / 2; j += L) {
                    float *a = cur + 3 * (size_t)j, *b = cur + 3 * (size_t)(nb - 1 - j);
                    const float a0 = a[0], a1 = a[1], a2 = a[2];
                    a[0] = b[0]; a[1] = b[1]; a[2] = b[2];
                    b[0] = a0; b[1] = a1; b[2] = a2;
                }
                MEM_SYNC();
            } else {
                nf = ns;
            }
        }
        if (p == 0) sline_len[off] = nb - 1 + nf;
    }
}

// track_seed_ptt_g's work for a stream of seeds with the stepping loop
// flattened, as flat_slot does for 32-lane slots: one loop iteration is one
// sub-step of whichever pass the L-lane group holds, and a group whose pass
// ends finishes it and starts its next pass, direction or seed at once, so
// the 64/L seeds of a wavefront keep sub-stepping together.  Seeds come from
// the XCD-ordered queues over the spatial order.  `st` (16 floats of the
// group's LDS) holds the seed's index, direction count, next direction,
// first slot, current slot, backward length and stream base (ints), its
// seed point and the direction (floats).
template <int L>
__device__ void flat_group_ptt(const DevParams &P, const DevBufs &B, const PttConst &K, PttG &S, float *st,
                               const float *__restrict__ seeds, int nseeds, int rng_chunk,
                               const int *__restrict__ offsets, const int *__restrict__ dirs,
                               int *__restrict__ sline_seed, int *__restrict__ sline_len, float *__restrict__ sline,
                               const int *__restrict__ order, int *__restrict__ work) {
    using G = Grp<L>;
    const int p = G::lane();
    const int step_frac = P.step_frac, MAXL = P.max_sline_len;
    const int nsub_max = MAXL * step_frac;
    const double sub = P.step_d / (double)step_frac;
    const size_t slot_f = (size_t)2 * MAXL * 3;
    const uint32_t key0 = P.seed_lo, key1 = P.seed_hi;
    int *si = reinterpret_cast<int *>(st);  // s, ndir, next direction, offsets[s], slot, nb, sub0
    float *sf = st + 8;                     // seed point [0..2], direction [3..5]
    if (p == 0) { si[1] = 0; si[2] = 0; }
    WAVE_SYNC();
    DrawCache dc;
    dc.valid = 0;
    int qk = 0;
    bool have = false;
    int pass = 0, i = 1, ri = 1, qi = 0;  // sub-step i = qi * step_frac + ri
    float px = 0.0f, py = 0.0f, pz = 0.0f, dx = 0.0f, dy = 0.0f, dz = 0.0f;
    float *sl = sline;
    for (;;) {
        if (!have) {
            while (qk < QUEUES) {
                const int di = si[2];
                if (di >= si[1]) {
                    const QueueRange qr = queue_range(work, qk);
                    const int lo = qr.lo, hi = qr.hi;
                    int q = 0;
                    if (p == 0 && lo < hi) q = atomicAdd(work + qr.counter, 1);
                    q = G::shfl(q, 0);
                    if (lo + q >= hi) { ++qk; continue; }
                    const int s = order[lo + q];
                    const int nd = (P.slot_cap > 0 && offsets[s + 1] > P.slot_cap) ? 0 : offsets[s + 1] - offsets[s];
                    WAVE_SYNC();
                    for (int v = p; v < 32; v += L) { S.rk[v] = 0u; S.rc[v] = -1; }
                    if (p == 0) {
                        si[0] = s; si[1] = nd; si[2] = 0; si[3] = offsets[s];
                        si[6] = (int)(32u * (uint32_t)(s % rng_chunk) + 1u);
                        sf[0] = seeds[3 * s]; sf[1] = seeds[3 * s + 1]; sf[2] = seeds[3 * s + 2];
                    }
                    dc.valid = 0;
                    WAVE_SYNC();
                    continue;
                }
                const int s = si[0], off = si[3] + di;
                const uint32_t sub0 = (uint32_t)si[6];
                const float sx = sf[0], sy = sf[1], sz = sf[2];
                const int vi = dirs[(size_t)s * P.nverts + di];
                const float fx = B.verts[3 * vi], fy = B.verts[3 * vi + 1], fz = B.verts[3 * vi + 2];
                float *cur = sline + (size_t)off * slot_f;
                WAVE_SYNC();
                if (p == 0) {
                    sline_seed[off] = s;
                    si[2] = di + 1; si[4] = off;
                    sf[3] = fx; sf[4] = fy; sf[5] = fz;
                }
                WAVE_SYNC();
                if (!init_frame_ptt_g<L>(P, B, K, S, key0, key1, sub0, dc, fx, fy, fz, sx, sy, sz)) {
                    if (p == 0) {
                        sline_len[off] = 1;
                        cur[0] = sx; cur[1] = sy; cur[2] = sz;
                    }
                    continue;
                }
                pass = 0;
                px = sx; py = sy; pz = sz;
                dx = -fx; dy = -fy; dz = -fz;
                sl = cur;
                if (p == 0) { sl[0] = px; sl[1] = py; sl[2] = pz; }
                i = 1; qi = (step_frac == 1) ? 1 : 0; ri = (step_frac == 1) ? 0 : 1;
                have = true;
                break;
            }
            if (!have) break;  // the queues are empty
        }
        // one sub-step of the pass (tracker_ptt_g's loop body)
        bool end = i >= nsub_max;
        if (!end) {
            float nx = 0.0f, ny = 0.0f, nz = 0.0f;
            const int nd = get_direction_ptt_g<L, false>(P, B, K, S, S.frame + (pass ? 9 : 0), key0, key1,
                                                         (uint32_t)si[6], dc, dx, dy, dz, px, py, pz, &nx, &ny, &nz);
            if (nd == 0) {
                end = true;
            } else {
                dx = nx; dy = ny; dz = nz;
                px = (float)__builtin_fma((double)(dx / 1.0f), sub, (double)px);
                py = (float)__builtin_fma((double)(dy / 1.0f), sub, (double)py);
                pz = (float)__builtin_fma((double)(dz / 1.0f), sub, (double)pz);
                if (p == 0 && ri == 0) {
                    float *o = sl + 3 * (size_t)qi;
                    o[0] = px; o[1] = py; o[2] = pz;
                }
                const int tissue = check_point(P, B.stop, px, py, pz);
                if (tissue == CUSLINES_ENDPOINT || tissue == CUSLINES_INVALIDPOINT || tissue == CUSLINES_OUTSIDEIMAGE) {
                    end = true;
                } else {
                    ++i;
                    if (++ri == step_frac) { ri = 0; ++qi; }
                    end = i >= nsub_max;
                }
            }
        }
        if (!end) continue;
        int nsteps = qi;
        if (ri != 0 && i < step_frac * (MAXL - 1)) {
            ++nsteps;
            if (p == 0) {
                float *o = sl + 3 * (size_t)nsteps;
                o[0] = px; o[1] = py; o[2] = pz;
            }
        }
        const int off = si[4];
        float *cur = sline + (size_t)off * slot_f;
        if (pass == 0) {
            const int nb = nsteps;
            MEM_SYNC();
            for (int j = p; j < nb / 2; j += L) {
                float *a = cur + 3 * (size_t)j, *b = cur + 3 * (size_t)(nb - 1 - j);
                const float a0 = a[0], a1 = a[1], a2 = a[2];
                a[0] = b[0]; a[1] = b[1]; a[2] = b[2];
                b[0] = a0; b[1] = a1; b[2] = a2;
            }
            MEM_SYNC();
            if (p == 0) si[5] = nb;
            pass = 1;
            px = sf[0]; py = sf[1]; pz = sf[2];
            dx = sf[3]; dy = sf[4]; dz = sf[5];
            sl = cur + 3 * (size_t)(nb - 1);
            if (p == 0) { sl[0] = px; sl[1] = py; sl[2] = pz; }
            i = 1; qi = (step_frac == 1) ? 1 : 0; ri = (step_frac == 1) ? 0 : 1;
            WAVE_SYNC();
        } else {
            if (p == 0) sline_len[off] = si[5] - 1 + nsteps;
            have = false;
        }
    }
}

// flat_group_ptt over workgroups of 256 threads (256/L seed groups).
template <int L>
__global__ void __launch_bounds__(256, 3) phase2_ptt_flat_kernel(DevParams P, DevBufs B,
                                                                 const float *__restrict__ seeds, int nseeds,
                                                                 int rng_chunk, const int *__restrict__ offsets,
                                                                 const int *__restrict__ dirs,
                                                                 int *__restrict__ sline_seed,
                                                                 int *__restrict__ sline_len,
                                                                 float *__restrict__ sline,
                                                                 const int *__restrict__ order,
                                                                 int *__restrict__ work) {
    extern __shared__ float smem[];
    PttConst K;
    K.vprop = smem;
    K.vk = smem + 24 * 9;
    ptt_const_init(P, K);
    __syncthreads();
    const int g = threadIdx.x / L;
    float *base = smem + PTTC_FLOATS + g * PTTG_FLOATS;
    PttG S;
    S.frame = base;
    S.vert_pdf = base + 18;
    S.face_cdf = base + 48;
    S.rk = reinterpret_cast<uint32_t *>(base + 80);
    S.rc = reinterpret_cast<int *>(base + 112);
    flat_group_ptt<L>(P, B, K, S, base + 144, seeds, nseeds, rng_chunk, offsets, dirs, sline_seed, sline_len, sline,
                      order, work);
}

// Persistent PTT phase 2 with L lanes per seed.
template <int L>
__global__ void __launch_bounds__(256) phase2_ptt_queue_kernel(DevParams P, DevBufs B, const float *__restrict__ seeds,
                                                               int nseeds, int rng_chunk,
                                                               const int *__restrict__ offsets,
                                                               const int *__restrict__ dirs,
                                                               int *__restrict__ sline_seed,
                                                               int *__restrict__ sline_len, float *__restrict__ sline,
                                                               int *__restrict__ work) {
    extern __shared__ float smem[];
    PttConst K;
    K.vprop = smem;
    K.vk = smem + 24 * 9;
    ptt_const_init(P, K);
    __syncthreads();
    const int g = threadIdx.x / L;
    float *base = smem + PTTC_FLOATS + g * PTTG_FLOATS;
    PttG S;
    S.frame = base;
    S.vert_pdf = base + 18;
    S.face_cdf = base + 48;
    S.rk = reinterpret_cast<uint32_t *>(base + 80);
    S.rc = reinterpret_cast<int *>(base + 112);
    const int p = Grp<L>::lane();
    for (;;) {
        int s = 0;
        if (p == 0) s = atomicAdd(work, 1);
        s = Grp<L>::shfl(s, 0);
        if (s >= nseeds) break;
        track_seed_ptt_g<L>(P, B, K, S, s, seeds, rng_chunk, offsets, dirs, sline_seed, sline_len, sline);
    }
}

// -------------------------------------------------------------------------
// Kernels
// -------------------------------------------------------------------------


// Floats of LDS per seed slot.  Peak marks take nv32/16 words, peak
// candidates nv32/2 floats (uint16 indices).
__host__ __device__ inline int marks_floats(int nv32) { return ((nv32 >> 4) + 3) & ~3; }
__host__ __device__ inline int cand_floats(int nv32) { return ((nv32 >> 1) + 3) & ~3; }

// Bootstrap slot: region C holds H.d and then the ODF; region A holds vox,
// msk and R.d / the model coefficients while the refit runs, and the peak
// marks and candidates once the ODF is computed (A is dead by then).
__host__ __device__ inline int boot_region_a(int nv32, int t32, int hr32) {
    const int refit = t32 + 2 * hr32;
    const int peaks = marks_floats(nv32) + cand_floats(nv32);
    return (refit > peaks) ? refit : peaks;
}

__host__ __device__ inline int slot_floats(int model, bool phase1, int nv32, int t32, int hr32) {
    if (model == CUSLINES_PTT && !phase1) return PTT_SLOT_FLOATS;
    if (model == CUSLINES_PROB && !phase1) return nv32;
    if (model == CUSLINES_PROB || model == CUSLINES_PTT) return nv32 + marks_floats(nv32) + cand_floats(nv32);
    const int c = (nv32 > hr32) ? nv32 : hr32;
    return c + boot_region_a(nv32, t32, hr32);
}

template <int MODEL>
__device__ void bind_slot(const DevParams &P, bool phase1, float *base, SlotLds &S) {
    if (MODEL == CUSLINES_PTT && !phase1) {
        S.ptt.frame = base;
        S.ptt.vert_pdf = base + 32;
        S.ptt.face_cdf = base + 64;
        S.ptt.act = base + 96;
    } else if (MODEL == CUSLINES_PROB || MODEL == CUSLINES_PTT) {
        S.prob.pmf = base;
        S.prob.marks = reinterpret_cast<uint32_t *>(base + P.nv32);
        S.prob.cand = reinterpret_cast<uint16_t *>(base + P.nv32 + marks_floats(P.nv32));
    } else {
        const int c = (P.nv32 > P.hr32) ? P.nv32 : P.hr32;
        float *a = base + c;
        S.boot.h = base;
        S.boot.vox = a;
        S.boot.msk = a + P.t32;
        S.boot.r = a + P.t32 + P.hr32;
        S.boot.marks = reinterpret_cast<uint32_t *>(a);
        S.boot.cand = reinterpret_cast<uint16_t *>(a + marks_floats(P.nv32));
    }
}

// Sphere vertices are staged in LDS for prob and PTT phase 1; bootstrap
// reads them from global memory (L1/L2), leaving its LDS to the seed slots.
template <int MODEL>
__host__ __device__ inline bool verts_in_lds() { return MODEL == CUSLINES_PROB || MODEL == CUSLINES_PTT; }

__device__ __forceinline__ int verts_floats(const DevParams &P) { return (3 * P.nverts + 3) & ~3; }

// getNumStreamlines{Prob,Boot,Ptt}_k (generate_streamlines_cuda.cu:423-462,
// boot.cu:610-718, ptt_init.cu:1-63): initial peak directions per seed.
template <int MODEL>
__global__ void __launch_bounds__(256) phase1_kernel(DevParams P, DevBufs B, const float *__restrict__ seeds,
                                                     int nseeds, int rng_chunk, int *__restrict__ counts,
                                                     int *__restrict__ dirs) {
    extern __shared__ float smem[];
    const float *sv = B.verts;
    int svf = 0;
    if (verts_in_lds<MODEL>()) {
        for (int i = threadIdx.x; i < 3 * P.nverts; i += blockDim.x) smem[i] = B.verts[i];
        sv = smem;
        svf = verts_floats(P);
    }
    __syncthreads();
    const int nslots = blockDim.x >> 5;
    const int slot = threadIdx.x >> 5;
    const int s = blockIdx.x * nslots + slot;
    if (s >= nseeds) return;
    const int l = lane32();
    float *base = smem + svf + slot * slot_floats(MODEL, true, P.nv32, P.t32, P.hr32);
    SlotLds S;
    bind_slot<MODEL>(P, true, base, S);
    const float px = seeds[3 * s], py = seeds[3 * s + 1], pz = seeds[3 * s + 2];
    typename SlotRng<MODEL>::type rng;  // the bootstrap getter draws from it
    if (MODEL == CUSLINES_OPDT || MODEL == CUSLINES_CSA)
        rng.init(((uint64_t)P.seed_hi << 32) | P.seed_lo, (uint64_t)32 * (uint64_t)(s % rng_chunk) + l);
    int n;
    const uint16_t *kept;
    if constexpr (MODEL == CUSLINES_PROB) {
        float a, b, c;
        n = get_direction_prob<true>(P, B, sv, S.prob, rng, 0.0f, 0.0f, 0.0f, px, py, pz, &a, &b, &c);
        kept = S.prob.cand;
    } else if constexpr (MODEL == CUSLINES_PTT) {
        float *pmf = S.prob.pmf;
        for (int i = l; i < P.nverts; i += 32) {
            const int tx = i & (P.nx - 1), ty = (i >> P.log2x) & (P.ny - 1), tz = i >> (P.log2x + P.log2y);
            const float v = tiled_sample(P, B.data, (float)(tx * P.dimx) + px, (float)(ty * P.dimy) + py,
                                         (float)(tz * P.dimz) + pz, tx, ty, tz);
            pmf[i] = (v < P.ptt_seed_thr_f) ? 0.0f : v;
        }
        WAVE_SYNC();
        n = peak_directions(peak_params(P, B), pmf, S.prob.marks, S.prob.cand, sv);
        kept = S.prob.cand;
    } else {
        float a, b, c;
        n = get_direction_boot<MODEL>(P, B, sv, S.boot, rng, 1, 0.0f, 0.0f, 0.0f, px, py, pz, &a, &b, &c);
        kept = S.boot.cand;
    }
    int *out = dirs + (size_t)s * P.nverts;
    for (int k = l; k < n; k += 32) out[k] = kept[k];
    if (l == 0) counts[s] = n;
}

// genStreamlinesMerge{Prob,Boot}_k body for one seed (generate_streamlines_cuda.cu:484-621,
// boot.cu:855-979): per direction, backward track, reverse, forward track.
template <int MODEL, int V = 0>
__device__ void track_seed(const DevParams &P, const DevBufs &B, const float *sv, SlotLds &S, int s,
                           const float *__restrict__ seeds, int rng_chunk, const int *__restrict__ offsets,
                           const int *__restrict__ dirs, int *__restrict__ sline_seed, int *__restrict__ sline_len,
                           float *__restrict__ sline) {
    const int l = lane32();
    const float sx = seeds[3 * s], sy = seeds[3 * s + 1], sz = seeds[3 * s + 2];
    typename SlotRng<MODEL>::type rng;
    rng.init(((uint64_t)P.seed_hi << 32) | P.seed_lo,
             (uint64_t)32 * (uint64_t)(s % rng_chunk) + (MODEL == CUSLINES_PROB ? 0 : l) + 1);
    const int ndir = (P.slot_cap > 0 && offsets[s + 1] > P.slot_cap) ? 0 : offsets[s + 1] - offsets[s];
    int off = offsets[s];
    const size_t slot_f = (size_t)2 * P.max_sline_len * 3;
    uint32_t ntap = 0, nsub = 0;  // V == 3: this lane's taps, the seed's sub-steps
    for (int i = 0; i < ndir; ++i, ++off) {
        const int vi = dirs[(size_t)s * P.nverts + i];
        const float fx = B.verts[3 * vi], fy = B.verts[3 * vi + 1], fz = B.verts[3 * vi + 2];
        float *cur = sline + (size_t)off * slot_f;
        if (l == 0) sline_seed[off] = s;
        if constexpr (MODEL == CUSLINES_PTT) {
            if (!init_frame_ptt<V == 3>(P, B, S.ptt, rng, fx, fy, fz, sx, sy, sz, &ntap)) {
                if (l == 0) {
                    sline_len[off] = 1;
                    cur[0] = sx; cur[1] = sy; cur[2] = sz;
                }
                continue;
            }
        }
        int nb = 0, nf = 0;
        for (int pass = 0; pass < 2; ++pass) {  // backward (-dir), then forward (+dir)
            const float sg = pass ? 1.0f : -1.0f;
            float *frame = (MODEL == CUSLINES_PTT) ? S.ptt.frame + 9 * pass : nullptr;
            float *out = pass ? cur + 3 * (size_t)(nb - 1) : cur;
            const int ns = tracker<MODEL, V>(P, B, sv, S, rng, sx, sy, sz, sg * fx, sg * fy, sg * fz, frame, out,
                                             ((uint32_t)s * 64u + (uint32_t)i) * 2u + (uint32_t)pass, &ntap, &nsub);
            if (pass == 0) {
                nb = ns;
                MEM_SYNC();
                for (int j = l; j < nb / 2; j += 32) {
                    float *a = cur + 3 * (size_t)j, *b = cur + 3 * (size_t)(nb - 1 - j);
                    const float a0 = a[0], a1 = a[1], a2 = a[2];
                    a[0] = b[0]; a[1] = b[1]; a[2] = b[2];
                    b[0] = a0; b[1] = a1; b[2] = a2;
                }
                MEM_SYNC();
            } else {
                nf = ns;
            }
        }
        if (l == 0) sline_len[off] = nb - 1 + nf;
    }
    if (V == 3 && B.stats) {
        unsigned long long taps = ntap;
        for (int m = 16; m; m >>= 1) taps += __shfl_xor(taps, m, 32);
        if (l == 0) {
            atomicAdd(B.stats, taps);
            atomicAdd(B.stats + 1, (unsigned long long)nsub);
        }
    }
}

// The learned kernels (V == 1, 5) copy the proposal network (IL_NPARAM bf16,
// lane-interleaved) into the first MLP_LDS_FLOATS floats of `lds` and point
// Bl.mlp there; every slot of the workgroup reads it from LDS.  Returns the
// floats used.  The caller synchronises the workgroup before use.
template <int V>
__device__ __forceinline__ int stage_network(const DevBufs &B, float *lds, DevBufs &Bl) {
    Bl = B;
    if (V != 1 && V != 5) return 0;
    const uint4 *src = reinterpret_cast<const uint4 *>(B.mlp);
    uint4 *dst = reinterpret_cast<uint4 *>(lds);
    for (int i = threadIdx.x; i < IL_NPARAM / 8; i += blockDim.x) dst[i] = src[i];
    Bl.mlp = reinterpret_cast<const uint16_t *>(lds);
    return MLP_LDS_FLOATS;
}

// Phase 2 of one 32-lane slot with the stepping loop flattened (the queue
// kernel's V == 4: the exact bootstrap getters and spheres too large for the
// probabilistic getter's own kernel; V == 5: the learned proposal; V == 6: the exact bootstrap getters at 2 waves
// per SIMD).  In track_seed a slot whose streamline pass, direction
// or seed ends leaves its loops and waits at their exit until the wave's
// other slot leaves them too; here one iteration of a single loop is one
// step (PTT: sub-step) of whichever pass the slot holds, and a slot whose
// pass ends finishes it (last point, reversal, length) and starts its next
// pass, direction or seed at once, so the wave's two slots keep stepping
// together.  Each seed's work, its order and its random draws are those of
// track_seed (genStreamlinesMerge{Prob,Boot,Ptt}, boot.cu:826-980,
// generate_streamlines_cuda.cu:464-621), so the results are identical.
// `st` (FLAT_STATE_FLOATS of the slot's LDS) holds the seed's index,
// direction count, next direction, first slot, current slot and backward
// length (ints), its seed point and the direction (floats).
constexpr int FLAT_STATE_FLOATS = 16;

template <int MODEL, bool LEARNED = false, bool WIDE = false>
__device__ void flat_slot(const DevParams &P, const DevBufs &B, const float *sv, SlotLds &S, float *st,
                          const float *__restrict__ seeds, int nseeds, int rng_chunk, const int *__restrict__ offsets,
                          const int *__restrict__ dirs, int *__restrict__ sline_seed, int *__restrict__ sline_len,
                          float *__restrict__ sline, const int *__restrict__ order, int *__restrict__ work) {
    constexpr bool PTT = MODEL == CUSLINES_PTT;
    static_assert(PTT == LEARNED, "plain PTT: flat_slot_ptt");
    const int l = lane32();
    const int step_frac = PTT ? P.step_frac : 1, MAXL = P.max_sline_len;
    const int nsub_max = MAXL * step_frac;
    const double sub = P.step_d / (double)step_frac;
    const size_t slot_f = (size_t)2 * MAXL * 3;
    int *si = reinterpret_cast<int *>(st);  // s, ndir, next direction, offsets[s], slot, nb
    float *sf = st + 8;                     // seed point [0..2], direction [3..5]
    if (l == 0) { si[1] = 0; si[2] = 0; }
    WAVE_SYNC();
    typename SlotRng<MODEL>::type rng;
    int qk = 0;
    bool have = false;
    int pass = 0, i = 1, ri = 1, qi = 0;  // step i = qi * step_frac + ri
    float px = 0.0f, py = 0.0f, pz = 0.0f, dx = 0.0f, dy = 0.0f, dz = 0.0f;
    float *sl = sline;
    // learned proposal (tracker's per-pass state): proposal on, its tries,
    // fallbacks to the plain sub-step, plain sub-steps and envelope misses
    bool learned = LEARNED;
    int ltries = 0, lfalls = 0, nplain = 0;
    uint32_t lmiss = 0;
    for (;;) {
        if (!have) {
            // the next direction of this seed, or of the next seeds
            while (qk < QUEUES) {
                const int di = si[2];
                if (di >= si[1]) {
                    const QueueRange qr = queue_range(work, qk);
                    const int lo = qr.lo, hi = qr.hi;
                    int q = 0;
                    if (l == 0 && lo < hi) q = atomicAdd(work + qr.counter, 1);
                    q = shfl32(q, 0);
                    if (lo + q >= hi) { ++qk; continue; }
                    const int s = order[lo + q];
                    const int nd = (P.slot_cap > 0 && offsets[s + 1] > P.slot_cap) ? 0 : offsets[s + 1] - offsets[s];
                    rng.init(((uint64_t)P.seed_hi << 32) | P.seed_lo,
                             (uint64_t)32 * (uint64_t)(s % rng_chunk) + (MODEL == CUSLINES_PROB ? 0 : l) + 1);
                    WAVE_SYNC();
                    if (l == 0) {
                        si[0] = s; si[1] = nd; si[2] = 0; si[3] = offsets[s];
                        sf[0] = seeds[3 * s]; sf[1] = seeds[3 * s + 1]; sf[2] = seeds[3 * s + 2];
                    }
                    WAVE_SYNC();
                    continue;
                }
                const int s = si[0], off = si[3] + di;
                const float sx = sf[0], sy = sf[1], sz = sf[2];
                const int vi = dirs[(size_t)s * P.nverts + di];
                const float fx = B.verts[3 * vi], fy = B.verts[3 * vi + 1], fz = B.verts[3 * vi + 2];
                float *cur = sline + (size_t)off * slot_f;
                WAVE_SYNC();
                if (l == 0) {
                    sline_seed[off] = s;
                    si[2] = di + 1; si[4] = off;
                    sf[3] = fx; sf[4] = fy; sf[5] = fz;
                }
                WAVE_SYNC();
                if constexpr (PTT) {
                    if (!init_frame_ptt(P, B, S.ptt, rng, fx, fy, fz, sx, sy, sz)) {
                        if (l == 0) {
                            sline_len[off] = 1;
                            cur[0] = sx; cur[1] = sy; cur[2] = sz;
                        }
                        continue;
                    }
                }
                // backward pass (-dir; PTT: on the frame at [0..8])
                pass = 0;
                px = sx; py = sy; pz = sz;
                dx = -fx; dy = -fy; dz = -fz;
                sl = cur;
                if (l == 0) { sl[0] = px; sl[1] = py; sl[2] = pz; }
                i = 1; qi = (step_frac == 1) ? 1 : 0; ri = (step_frac == 1) ? 0 : 1;
                if (LEARNED) { learned = true; ltries = lfalls = nplain = 0; lmiss = 0; }
                have = true;
                break;
            }
            if (!have) break;  // the queues are empty
        }
        // one step of the pass (tracker's loop body)
        bool end = i >= nsub_max;
        if (!end) {
            float nx = 0.0f, ny = 0.0f, nz = 0.0f;
            int nd;
            if constexpr (MODEL == CUSLINES_PROB) {
                nd = get_direction_prob<false>(P, B, sv, S.prob, rng, dx, dy, dz, px, py, pz, &nx, &ny, &nz);
            } else if constexpr (LEARNED) {
                int fell = 0;
                nd = get_direction_ptt_learned(P, B, S.ptt, S.ptt.frame + (pass ? 9 : 0), rng, learned, dx, dy, dz, px,
                                               py, pz, &nx, &ny, &nz, &fell, &lmiss);
                if (learned) {
                    ++ltries;
                    lfalls += fell;
                    if (ltries >= 16 && 4 * lfalls > ltries) learned = false;
                } else {
                    ++nplain;
                }
            } else
                nd = get_direction_boot<MODEL, WIDE>(P, B, sv, S.boot, rng, 5, dx, dy, dz, px, py, pz, &nx, &ny, &nz);
            if (nd == 0) {
                end = true;
            } else {
                dx = nx; dy = ny; dz = nz;
                px = (float)__builtin_fma((double)(dx / 1.0f), sub, (double)px);
                py = (float)__builtin_fma((double)(dy / 1.0f), sub, (double)py);
                pz = (float)__builtin_fma((double)(dz / 1.0f), sub, (double)pz);
                if (l == 0 && ri == 0) {
                    float *o = sl + 3 * (size_t)qi;
                    o[0] = px; o[1] = py; o[2] = pz;
                }
                const int tissue = check_point(P, B.stop, px, py, pz);
                if (tissue == CUSLINES_ENDPOINT || tissue == CUSLINES_INVALIDPOINT || tissue == CUSLINES_OUTSIDEIMAGE) {
                    end = true;
                } else {
                    ++i;
                    if (++ri == step_frac) { ri = 0; ++qi; }
                    end = i >= nsub_max;
                }
            }
        }
        if (!end) continue;
        // the pass ends at step i (tracker's tail)
        if (LEARNED && B.stats && l == 0) {
            atomicAdd(B.stats, (unsigned long long)(ltries - lfalls));
            atomicAdd(B.stats + 1, (unsigned long long)lfalls);
            atomicAdd(B.stats + 2, (unsigned long long)nplain);
            atomicAdd(B.stats + 3, (unsigned long long)lmiss);
        }
        int nsteps = qi;
        if (ri != 0 && i < step_frac * (MAXL - 1)) {
            ++nsteps;
            if (l == 0) {
                float *o = sl + 3 * (size_t)nsteps;
                o[0] = px; o[1] = py; o[2] = pz;
            }
        }
        const int off = si[4];
        float *cur = sline + (size_t)off * slot_f;
        if (pass == 0) {
            const int nb = nsteps;
            MEM_SYNC();
            for (int j = l; j < nb / 2; j += 32) {
                float *a = cur + 3 * (size_t)j, *b = cur + 3 * (size_t)(nb - 1 - j);
                const float a0 = a[0], a1 = a[1], a2 = a[2];
                a[0] = b[0]; a[1] = b[1]; a[2] = b[2];
                b[0] = a0; b[1] = a1; b[2] = a2;
            }
            MEM_SYNC();
            if (l == 0) si[5] = nb;
            // forward pass (+dir; PTT: on the frame at [9..17]), from the seed point at index nb - 1
            pass = 1;
            px = sf[0]; py = sf[1]; pz = sf[2];
            dx = sf[3]; dy = sf[4]; dz = sf[5];
            sl = cur + 3 * (size_t)(nb - 1);
            if (l == 0) { sl[0] = px; sl[1] = py; sl[2] = pz; }
            i = 1; qi = (step_frac == 1) ? 1 : 0; ri = (step_frac == 1) ? 0 : 1;
            if (LEARNED) { learned = true; ltries = lfalls = nplain = 0; lmiss = 0; }
            WAVE_SYNC();
        } else {
            if (l == 0) sline_len[off] = si[5] - 1 + nsteps;
            have = false;
        }
    }
}

// -------------------------------------------------------------------------
// Probabilistic phase 2 with the pmf and the cell in registers (rows of up to
// 768 channels), one seed per wavefront.
//
// The step of flat_slot<PROB> reads 8 corners x 724 channels (23 KB) through
// L2 whether or not the seed left its cell, and is a chain of short dependent
// pieces: 8 rounds of loads, 23 blocks of 5 lane shuffles that each wait for
// the block before (the running sum's carry), a 5-level binary search through
// LDS, 8 branchy stop-map reads.  A lone slot took 14 us a step, and 25,000
// seeds, which share few cells, ran at the rate of the fabric.  Here
//  - a lane owns channels 256 c + 4 l .. + 3, and the cell's 8 corners stay
//    in its registers: a step of 1/4 voxel leaves the cell about every third
//    time, usually by one face, and then reads 4 corners (about 1/5 of the
//    bytes; nothing is kept beyond the wave's own last cell);
//  - the threshold, the cone test and the running sum work on registers;
//  - the stop map of the point just stored is read with the next step;
//  - the position, the cell, the search and every branch are the wave's, so
//    addresses and control flow are scalar.
//
// The running sum keeps the additions of prefix_sum (utils.cu:81-120) and
// their order.  In its Hillis-Steele block only values that include element 0
// see the carry: with m the highest power of two <= e,
//     out[e] = W[e] + out[e - m],  out[0] = x[0] + carry,
// W[e] the sum of the m elements ending at e as the first log2(m) rounds form
// it.  So W needs no carry (4 rounds of in-lane adds and row-shift DPP, all
// blocks at once); the block carries are a chain of 6 adds per block over
// W[0], W[1], W[3], W[7], W[15], W[31], one block per lane; and out is only
// formed where it is read: the 31 midpoints that the 5 levels of the binary
// search can visit (one per lane), the last element and the final window.
//
// What bounds it: VALU issue (745 instructions a step; 0.5 a cycle and CU at
// 25,000 seeds, 0.79 at 250,000) and, for the last seeds, the chain of one step
// (2.8 us alone).
// Measured against flat_slot<PROB> (81x106x76, 724 vertices, step 1/4 voxel):
// 64 seeds 9.8 -> 2.6 ms, 25,000 seeds 120 -> 41 ms, 100,000 255 -> 126 ms;
// fetched from memory at 25,000 seeds: 17 GB for 9.6 M steps.  The same
// kernel with 32 lanes a seed and the gather repeated every step: 67 and
// 187 ms.
//
// Fast values only: a NaN or a value of 1e30 or more anywhere in the pmf
// sends the step to prob_sum and prob_pick.  Values left by the threshold are
// never negative (a negative maximum zeroes everything), so masked additions
// of +0 change nothing.
// -------------------------------------------------------------------------
// 2 waves per SIMD: 96 registers hold the cell.  At 3 (168 registers) 82 spill
// and a 25,000-seed chunk takes 59.9 ms instead of 42.8.
constexpr int PROB_WAVES = 2;
constexpr int PROB_W_BLOCK = 36;  // LDS floats per 32-value block: the 4 extra spread the lanes' block reads over banks
constexpr float PROB_FAST_MAX = 1e30f;
constexpr int prob_slot_floats(int nch) { return PROB_W_BLOCK * 8 * nch + 64; }

constexpr int DPP_ROW_SHR = 0x110, DPP_ROW_ROR = 0x120, DPP_WAVE_SHR1 = 0x138;
template <int CTRL>
__device__ __forceinline__ float dpp0(float x) {  // 0 where the shift has no source lane
    return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(x), CTRL, 0xf, 0xf, true));
}

// Maximum over the wave, NaN if any value is.
__device__ __forceinline__ float nan_max64(float v) {
    v = __builtin_elementwise_maximum(v, dpp0<DPP_ROW_ROR + 8>(v));
    v = __builtin_elementwise_maximum(v, dpp0<DPP_ROW_ROR + 4>(v));
    v = __builtin_elementwise_maximum(v, dpp0<DPP_ROW_ROR + 2>(v));
    v = __builtin_elementwise_maximum(v, dpp0<DPP_ROW_ROR + 1>(v));
    const auto s16 = __builtin_amdgcn_permlane16_swap(__float_as_uint(v), __float_as_uint(v), false, false);
    v = __builtin_elementwise_maximum(__uint_as_float(s16[0]), __uint_as_float(s16[1]));
    const auto s32 = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
    return __builtin_elementwise_maximum(__uint_as_float(s32[0]), __uint_as_float(s32[1]));
}

__device__ __forceinline__ float uniform_f(float x) {
    return __int_as_float(__builtin_amdgcn_readfirstlane(__float_as_int(x)));
}
__device__ __forceinline__ float lane_f(float x, int lane) {
    return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(x), lane));
}

// out[i] of the running sum, from the blocks' W and carries.
__device__ __forceinline__ float prob_cdf(const float *W, const float *carry, int i) {
    const int b = i >> 5, e = i & 31;
    const float *w = W + PROB_W_BLOCK * b;
    const float c = carry[b], w0 = w[0], w1 = w[e & 1], w2 = w[e & 3], w3 = w[e & 7], w4 = w[e & 15], w5 = w[e];
    float s = w0 + c;
    s = (e & 1) ? w1 + s : s;
    s = (e & 2) ? w2 + s : s;
    s = (e & 4) ? w3 + s : s;
    s = (e & 8) ? w4 + s : s;
    s = (e & 16) ? w5 + s : s;
    return s;
}

// The midpoint that node k of the binary search's tree compares (root 0, the
// children of k at 2 k + 1 for "below", 2 k + 2 for "not below").
__device__ __forceinline__ int prob_node_mid(int nv, int k) {
    int low = 0, high = nv - 1;
    const int path = k + 1;
    for (int d = 30 - __clz(path); d >= 0; --d) {
        const int mid = (low + high) >> 1;
        if ((path >> d) & 1) high = mid; else low = mid;
    }
    return (low + high) >> 1;
}

// The step's choice by the general routines (out of line: rare); -1: none.
// Both halves of the wave do the same work on the same array.
__device__ __noinline__ int prob_slow(int nv, int symm, float cos_max_angle, const float *verts, float *pmf, float u,
                                      float dx, float dy, float dz) {
    const float last = prob_sum(nv, symm, cos_max_angle, verts, pmf, dx, dy, dz);
    return (last == 0.0f) ? -1 : prob_pick(pmf, nv, u * last);
}

typedef float prob_v4 __attribute__((ext_vector_type(4)));

// A wave's last cell: its corners (bit 2 x, bit 1 y, bit 0 z, as trilinear's).
template <int NCH>
struct ProbCell {
    prob_v4 v[8][NCH];
    int x, y, z;
};

// Move the corners one cell along the axis of corner bit BIT (e: -1, 0, 1);
// returns the corners that hold the new cell's values (bit mask).
template <int NCH, int BIT>
__device__ __forceinline__ uint32_t prob_shift(ProbCell<NCH> &C, int e) {
    constexpr uint32_t LOW = (BIT == 1) ? 0x55u : (BIT == 2) ? 0x33u : 0x0fu;  // corners with the bit clear
    constexpr int U = (BIT == 1) ? 2 : 1, V = (BIT == 4) ? 2 : 4;              // the other two bits
    // The empty asm keeps the two branches apart: merged, their stores would
    // index the register array at run time and send it to scratch.
    if (e > 0) {
#pragma unroll
        for (int c = 0; c < NCH; ++c) {
            C.v[0][c] = C.v[BIT][c];
            C.v[U][c] = C.v[U | BIT][c];
            C.v[V][c] = C.v[V | BIT][c];
            C.v[U | V][c] = C.v[7][c];
        }
        asm volatile("; cell up");
        return LOW;
    }
    if (e < 0) {
#pragma unroll
        for (int c = 0; c < NCH; ++c) {
            C.v[BIT][c] = C.v[0][c];
            C.v[U | BIT][c] = C.v[U][c];
            C.v[V | BIT][c] = C.v[V][c];
            C.v[7][c] = C.v[U | V][c];
        }
        asm volatile("; cell down");
        return 0xffu & ~LOW;
    }
    return 0xffu;
}

// Bring the cell to (x0, y0, z0): corners shared with the last cell move,
// the others are read.
template <int NCH>
__device__ __forceinline__ void prob_move_cell(const DevParams &P, const float *__restrict__ data, ProbCell<NCH> &C,
                                               int x0, int y0, int z0, uint32_t off, uint32_t off_last) {
    const int ex = x0 - C.x, ey = y0 - C.y, ez = z0 - C.z;
    if ((ex | ey | ez) == 0) return;
    C.x = x0; C.y = y0; C.z = z0;
    uint32_t valid = 0u;
    if ((uint32_t)(ex + 1) <= 2u && (uint32_t)(ey + 1) <= 2u && (uint32_t)(ez + 1) <= 2u) {
        valid = 0xffu;
        valid &= prob_shift<NCH, 1>(C, ez);
        valid &= prob_shift<NCH, 2>(C, ey);
        valid &= prob_shift<NCH, 4>(C, ex);
    }
    const uint32_t dzv = (z0 + 1 < P.dimz) ? 1u : 0u;
    const uint32_t dyv = (y0 + 1 < P.dimy) ? (uint32_t)P.dimz : 0u;
    const uint32_t dxv = (x0 + 1 < P.dimx) ? (uint32_t)P.dimy * (uint32_t)P.dimz : 0u;
    const uint32_t vox = ((uint32_t)x0 * (uint32_t)P.dimy + (uint32_t)y0) * (uint32_t)P.dimz + (uint32_t)z0;
#pragma unroll
    for (int k = 0; k < 8; ++k) {
        if ((valid >> k) & 1u) continue;
        const uint32_t vk = vox + ((k & 4) ? dxv : 0u) + ((k & 2) ? dyv : 0u) + ((k & 1) ? dzv : 0u);
        const char *row = reinterpret_cast<const char *>(data + (uint64_t)vk * (uint32_t)P.t32);
#pragma unroll
        for (int c = 0; c < NCH; ++c)
            C.v[k][c] = *reinterpret_cast<const prob_v4 *>(row + ((c == NCH - 1) ? off_last : off + 1024u * c));
    }
}

// check_point for a wave whose lanes share the point: lane k (of every 8)
// reads texel k and forms its weight, and the sum moves along the lanes, one
// fused multiply-add each, in check_point's order.
struct WaveTap {
    float w, t;
};

__device__ __forceinline__ WaveTap wave_stop_begin(const DevParams &P, const float *__restrict__ stop, float px,
                                                   float py, float pz) {
    const int kz = threadIdx.x & 1, ky = (threadIdx.x >> 1) & 1, kx = (threadIdx.x >> 2) & 1;
    int iz, iy, ix;
    const float a = tex_weight(pz, &iz), b = tex_weight(py, &iy), g = tex_weight(px, &ix);
    const float wa = kz ? a : 1.0f - a, wb = ky ? b : 1.0f - b, wg = kx ? g : 1.0f - g;
    // i = -k .. D - 1 - k is inside; outside reads a clamped texel, replaced
    const bool in = (ix >= -kx) & (ix < P.dimx - kx) & (iy >= -ky) & (iy < P.dimy - ky) & (iz >= -kz) &
                    (iz < P.dimz - kz);
    const uint32_t x = (uint32_t)(min(max(ix, -kx), P.dimx - 1 - kx) + kx),
                   y = (uint32_t)(min(max(iy, -ky), P.dimy - 1 - ky) + ky),
                   z = (uint32_t)(min(max(iz, -kz), P.dimz - 1 - kz) + kz);
    WaveTap r;
    const float t = stop[(size_t)((x * (uint32_t)P.dimy + y) * (uint32_t)P.dimz + z)];
    r.t = in ? t : -1.0f;
    r.w = (wa * wb) * wg;
    return r;
}

__device__ __forceinline__ int wave_stop_end(const DevParams &P, const WaveTap &r) {
    float acc = r.w * r.t;
#pragma unroll
    for (int k = 1; k < 8; ++k) acc = __builtin_fmaf(r.w, r.t, dpp0<DPP_ROW_SHR + 1>(acc));
    acc = lane_f(acc, 7);
    if (acc == -1.0f) return CUSLINES_OUTSIDEIMAGE;
    return (acc > P.tc_threshold) ? CUSLINES_TRACKPOINT : CUSLINES_ENDPOINT;
}

// One direction draw at (px, py, pz).  `check`: the point's stop-map check
// is still to do (not at a pass's first point).  Returns 1 with the new
// direction, 0 when there is none, -1 when the stop check ends the pass.
template <int NCH>
__device__ __forceinline__ int prob_step(const DevParams &P, const DevBufs &B, const float *sv, float *W, float *carry,
                                         ProbCell<NCH> &C, int my_mid, float m1, float m2, float m4, bool tail,
                                         uint32_t off, uint32_t off_last, bool check, ProbStream<64> &rng, float dx,
                                         float dy, float dz, float px, float py, float pz, float *ndx, float *ndy,
                                         float *ndz) {
    const int l = threadIdx.x & 63;
    const int nv = P.nverts;
    const WaveTap tap = wave_stop_begin(P, B.stop, px, py, pz);
    // trilinear()'s cell and weights, the cell clamped so that a point
    // outside reads in bounds (its values are dropped)
    const bool outside = (px < -0.5f) | (px + 0.5f >= (float)P.dimx) | (py < -0.5f) | (py + 0.5f >= (float)P.dimy) |
                         (pz < -0.5f) | (pz + 0.5f >= (float)P.dimz);
    const float fx = floorf(px), fy = floorf(py), fz = floorf(pz);
    const float wx1 = px - fx, wy1 = py - fy, wz1 = pz - fz;
    const float wx0 = 1.0f - wx1, wy0 = 1.0f - wy1, wz0 = 1.0f - wz1;
    const float w[8] = {(wx0 * wy0) * wz0, (wx0 * wy0) * wz1, (wx0 * wy1) * wz0, (wx0 * wy1) * wz1,
                        (wx1 * wy0) * wz0, (wx1 * wy0) * wz1, (wx1 * wy1) * wz0, (wx1 * wy1) * wz1};
    const int x0 = min((int)((0.0f > fx) ? 0.0f : fx), P.dimx - 1), y0 = min((int)((0.0f > fy) ? 0.0f : fy), P.dimy - 1),
              z0 = min((int)((0.0f > fz) ? 0.0f : fz), P.dimz - 1);
    prob_move_cell<NCH>(P, B.data, C, __builtin_amdgcn_readfirstlane(x0), __builtin_amdgcn_readfirstlane(y0),
                        __builtin_amdgcn_readfirstlane(z0), off, off_last);
    if (check && wave_stop_end(P, tap) != CUSLINES_TRACKPOINT) return -1;
    if (__builtin_amdgcn_readfirstlane(outside)) return 0;
    prob_v4 acc[NCH];
#pragma unroll
    for (int c = 0; c < NCH; ++c) {
        acc[c] = prob_v4{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
        for (int k = 0; k < 8; ++k) {
            acc[c].x = __builtin_fmaf(w[k], C.v[k][c].x, acc[c].x);
            acc[c].y = __builtin_fmaf(w[k], C.v[k][c].y, acc[c].y);
            acc[c].z = __builtin_fmaf(w[k], C.v[k][c].z, acc[c].z);
            acc[c].w = __builtin_fmaf(w[k], C.v[k][c].w, acc[c].w);
        }
    }
    if (!tail) acc[NCH - 1] = prob_v4{0.0f, 0.0f, 0.0f, 0.0f};
    // channels nverts.. of a row are 0 in memory: they leave a maximum that
    // would be negative at 0, and either way the threshold drops everything
    float mx = __builtin_elementwise_maximum(__builtin_elementwise_maximum(acc[0].x, acc[0].y),
                                             __builtin_elementwise_maximum(acc[0].z, acc[0].w));
#pragma unroll
    for (int c = 1; c < NCH; ++c)
        mx = __builtin_elementwise_maximum(
            mx, __builtin_elementwise_maximum(__builtin_elementwise_maximum(acc[c].x, acc[c].y),
                                              __builtin_elementwise_maximum(acc[c].z, acc[c].w)));
    mx = uniform_f(nan_max64(mx));
    const float u = rng.peek();
    int ind;
    if (!(mx < PROB_FAST_MAX)) {
#pragma unroll
        for (int c = 0; c < NCH; ++c) *reinterpret_cast<prob_v4 *>(W + 256 * c + 4 * l) = acc[c];
        WAVE_SYNC();
        ind = __builtin_amdgcn_readfirstlane(
            prob_slow(nv, P.sphere_symm, P.cos_max_angle, B.verts, W, u, dx, dy, dz));
        if (ind < 0) return 0;
        rng.take();
    } else {
        const float thr = (float)(PMF_THRESHOLD_P * (double)mx);
        const float cosm = P.cos_max_angle;
        const uint32_t dmask = P.sphere_symm ? 0x7fffffffu : 0xffffffffu;
        auto keep = [&](float v, float x, float y, float z) {
            // |d| on a symmetric sphere: the sign bit masked off
            const float d = __uint_as_float(__float_as_uint(dot3(dx, dy, dz, x, y, z)) & dmask);
            return ((v < thr) | (d < cosm)) ? 0.0f : v;
        };
#pragma unroll
        for (int c = 0; c < NCH; ++c) {
            const prob_v4 vx = *reinterpret_cast<const prob_v4 *>(sv + 256 * c + 4 * l);
            const prob_v4 vy = *reinterpret_cast<const prob_v4 *>(sv + 256 * (NCH + c) + 4 * l);
            const prob_v4 vz = *reinterpret_cast<const prob_v4 *>(sv + 256 * (2 * NCH + c) + 4 * l);
            acc[c].x = keep(acc[c].x, vx.x, vy.x, vz.x);
            acc[c].y = keep(acc[c].y, vx.y, vy.y, vz.y);
            acc[c].z = keep(acc[c].z, vx.z, vy.z, vz.z);
            acc[c].w = keep(acc[c].w, vx.w, vy.w, vz.w);
        }
        // rounds 1, 2, 4, 8 for elements >= 2, 4, 8, 16 of a block (8 lanes),
        // round by round over the independent chunks; a factor 0 or 1 masks
        // the addition
#pragma unroll
        for (int c = 0; c < NCH; ++c) {
            const prob_v4 q = acc[c];
            acc[c].w = q.w + q.z;
            acc[c].z = q.z + q.y;
            acc[c].y = __builtin_fmaf(q.x, m1, q.y);
            acc[c].x = __builtin_fmaf(dpp0<DPP_ROW_SHR + 1>(q.w), m1, q.x);
        }
#pragma unroll
        for (int c = 0; c < NCH; ++c) {
            const prob_v4 q = acc[c];
            acc[c].w = __builtin_fmaf(q.y, m1, q.w);
            acc[c].z = __builtin_fmaf(q.x, m1, q.z);
            acc[c].y = __builtin_fmaf(dpp0<DPP_ROW_SHR + 1>(q.w), m1, q.y);
            acc[c].x = __builtin_fmaf(dpp0<DPP_ROW_SHR + 1>(q.z), m1, q.x);
        }
        // v <- v + m * shift(v) in one instruction each; a DPP source must be
        // two instructions old, hence the s_nop at both ends of a round
#define PROB_SHIFT_ADD(SHIFT, MASK)                                                                              \
    _Pragma("unroll") for (int c = 0; c < NCH; ++c) {                                                            \
        float ax = acc[c].x, ay = acc[c].y, az = acc[c].z, aw = acc[c].w;                                        \
        asm volatile("s_nop 1\n\t"                                                                                            \
        "v_fmac_f32_dpp %0, %0, %4 row_shr:" SHIFT " row_mask:0xf bank_mask:0xf bound_ctrl:0\n\t"                 \
        "v_fmac_f32_dpp %1, %1, %4 row_shr:" SHIFT " row_mask:0xf bank_mask:0xf bound_ctrl:0\n\t"                 \
        "v_fmac_f32_dpp %2, %2, %4 row_shr:" SHIFT " row_mask:0xf bank_mask:0xf bound_ctrl:0\n\t"                 \
        "v_fmac_f32_dpp %3, %3, %4 row_shr:" SHIFT " row_mask:0xf bank_mask:0xf bound_ctrl:0\n\t"                 \
        "s_nop 1"                                                                                                \
        : "+v"(ax), "+v"(ay), "+v"(az), "+v"(aw)                                                                 \
        : "v"(MASK));                                                                                            \
        acc[c] = prob_v4{ax, ay, az, aw};                                                                        \
    }
        PROB_SHIFT_ADD("1", m2)
        PROB_SHIFT_ADD("2", m4)
#undef PROB_SHIFT_ADD
#pragma unroll
        for (int c = 0; c < NCH; ++c)
            *reinterpret_cast<prob_v4 *>(W + PROB_W_BLOCK * (8 * c + (l >> 3)) + 4 * (l & 7)) = acc[c];
        WAVE_SYNC();
        // lane b: block b's part of the carry chain
        const int nblk = (nv + 31) >> 5;
        {
            const float *wb = W + PROB_W_BLOCK * min(l, nblk - 1);
            const float4 q = *reinterpret_cast<const float4 *>(wb);
            const float s7 = wb[7], s15 = wb[15], s31 = wb[31];
            float x = 0.0f;
            for (int it = 1; it < nblk; ++it) {
                float t = q.x + dpp0<DPP_WAVE_SHR1>(x);
                t = q.y + t;
                t = q.w + t;
                t = s7 + t;
                t = s15 + t;
                x = s31 + t;
            }
            carry[l] = dpp0<DPP_WAVE_SHR1>(x);
        }
        WAVE_SYNC();
        // lane k < 31: node k of the search tree; lane 31: the last element
        const float node = prob_cdf(W, carry, my_mid);
        const float last = lane_f(node, 31);
        if (last == 0.0f) return 0;
        rng.take();
        const float sel = u * last;
        const uint32_t below = (uint32_t)__ballot(node < sel);
        int low = 0, high = nv - 1, k = 0;
#pragma unroll
        for (int lev = 0; lev < 5; ++lev) {
            const int mid = (low + high) >> 1;
            const bool open = (high - low) >= 32;
            const bool bl = (below >> k) & 1u;
            low = (open && bl) ? mid : low;
            high = (open && !bl) ? mid : high;
            k = 2 * k + (bl ? 1 : 2);
        }
        const float win = prob_cdf(W, carry, min(low + l, nv - 1));
        const unsigned long long msk = __ballot(low + l <= high && sel < win);
        ind = max(low + __ffsll(msk) - 1, 0);
    }
    const float ux = sv[ind], uy = sv[256 * NCH + ind], uz = sv[512 * NCH + ind];
    const bool fwd = dot3(dx, dy, dz, ux, uy, uz) > 0.0f;
    *ndx = fwd ? ux : -ux;
    *ndy = fwd ? uy : -uy;
    *ndz = fwd ? uz : -uz;
    WAVE_SYNC();
    return 1;
}

// flat_slot's loop for one wave.
template <int NCH>
__device__ void flat_wave_prob(const DevParams &P, const DevBufs &B, const float *sv, float *lds,
                               const float *__restrict__ seeds, int nseeds, int rng_chunk,
                               const int *__restrict__ offsets, const int *__restrict__ dirs,
                               int *__restrict__ sline_seed, int *__restrict__ sline_len, float *__restrict__ sline,
                               const int *__restrict__ order, int *__restrict__ work) {
    const int l = threadIdx.x & 63;
    const int MAXL = P.max_sline_len;
    const double sub = P.step_d;
    const size_t slot_f = (size_t)2 * MAXL * 3;
    float *W = lds, *carry = lds + PROB_W_BLOCK * 8 * NCH;
    const int my_mid = (l < 31) ? prob_node_mid(P.nverts, l) : (l == 31) ? P.nverts - 1 : 0;
    const float m1 = ((l & 7) >= 1) ? 1.0f : 0.0f, m2 = ((l & 7) >= 2) ? 1.0f : 0.0f, m4 = ((l & 7) >= 4) ? 1.0f : 0.0f;
    // NCH is the number of chunks of a padded row, so only the last can be
    // partial: its lanes past the row re-read chunk 0 and drop it
    const bool tail = 256 * (NCH - 1) + 4 * l < P.t32;
    const uint32_t off = 16u * l, off_last = off + (tail ? 1024u * (NCH - 1) : 0u);
    ProbCell<NCH> C;
    C.x = C.y = C.z = -4;  // no cell's neighbour
#pragma unroll
    for (int c = 0; c < NCH; ++c) {
#pragma unroll
        for (int k = 0; k < 8; ++k) C.v[k][c] = prob_v4{0.0f, 0.0f, 0.0f, 0.0f};
    }
    ProbStream<64> rng;
    int qk = 0, s = 0, ndir = 0, di = 0, slot = 0, nb = 0;  // seed, its directions, the next, output slot, backward points
    float sx = 0.0f, sy = 0.0f, sz = 0.0f, fx = 0.0f, fy = 0.0f, fz = 0.0f;
    bool have = false, check = false;
    int pass = 0, i = 1;
    float px = 0.0f, py = 0.0f, pz = 0.0f, dx = 0.0f, dy = 0.0f, dz = 0.0f;
    float *sl = sline;
    for (;;) {
        if (!have) {
            // the next direction of this seed, or of the next seeds
            while (di >= ndir && qk < QUEUES) {
                const QueueRange qr = queue_range(work, qk);
                const int lo = qr.lo, hi = qr.hi;
                int q = 0;
                if (l == 0 && lo < hi) q = atomicAdd(work + qr.counter, 1);
                q = __builtin_amdgcn_readfirstlane(q);
                if (lo + q >= hi) { ++qk; continue; }
                s = __builtin_amdgcn_readfirstlane(order[lo + q]);
                const int o0 = __builtin_amdgcn_readfirstlane(offsets[s]),
                          o1 = __builtin_amdgcn_readfirstlane(offsets[s + 1]);
                ndir = (P.slot_cap > 0 && o1 > P.slot_cap) ? 0 : o1 - o0;
                di = 0;
                slot = o0 - 1;
                sx = seeds[3 * (size_t)s]; sy = seeds[3 * (size_t)s + 1]; sz = seeds[3 * (size_t)s + 2];
                rng.init(((uint64_t)P.seed_hi << 32) | P.seed_lo, (uint64_t)32 * (uint64_t)(s % rng_chunk) + 1);
            }
            if (di >= ndir) break;  // the queues are empty
            const int vi = __builtin_amdgcn_readfirstlane(dirs[(size_t)s * P.nverts + di]);
            fx = B.verts[3 * vi]; fy = B.verts[3 * vi + 1]; fz = B.verts[3 * vi + 2];
            ++di;
            ++slot;
            sl = sline + (size_t)slot * slot_f;
            // backward pass (-dir)
            px = sx; py = sy; pz = sz;
            dx = -fx; dy = -fy; dz = -fz;
            if (l == 0) {
                sline_seed[slot] = s;
                sl[0] = px; sl[1] = py; sl[2] = pz;
            }
            pass = 0;
            i = 1;
            check = false;
            have = true;
        }
        // one step of the pass: `i` points are stored; the stop check of the
        // last one, left over from the step that stored it, comes with this
        // step's reads
        float nx = 0.0f, ny = 0.0f, nz = 0.0f;
        int nsteps;
        if (i >= MAXL) {
            const bool bad = check && wave_stop_end(P, wave_stop_begin(P, B.stop, px, py, pz)) != CUSLINES_TRACKPOINT;
            nsteps = bad ? i - 1 : i;
        } else {
            const int nd = prob_step<NCH>(P, B, sv, W, carry, C, my_mid, m1, m2, m4, tail, off, off_last, check, rng, dx,
                                          dy, dz, px, py, pz, &nx, &ny, &nz);
            if (nd > 0) {
                dx = nx; dy = ny; dz = nz;
                px = (float)__builtin_fma((double)(dx / 1.0f), sub, (double)px);
                py = (float)__builtin_fma((double)(dy / 1.0f), sub, (double)py);
                pz = (float)__builtin_fma((double)(dz / 1.0f), sub, (double)pz);
                if (l < 3) sl[3 * (size_t)i + l] = (l == 0) ? px : (l == 1) ? py : pz;
                ++i;
                check = true;
                continue;
            }
            nsteps = (nd < 0) ? i - 1 : i;
        }
        // the pass ends with nsteps points (tracker's tail)
        check = false;
        if (pass == 0) {
            MEM_SYNC();
            for (int j = l; j < nsteps / 2; j += 64) {
                float *a = sl + 3 * (size_t)j, *b = sl + 3 * (size_t)(nsteps - 1 - j);
                const float a0 = a[0], a1 = a[1], a2 = a[2];
                a[0] = b[0]; a[1] = b[1]; a[2] = b[2];
                b[0] = a0; b[1] = a1; b[2] = a2;
            }
            MEM_SYNC();
            nb = nsteps;
            // forward pass (+dir), from the seed point at index nsteps - 1
            pass = 1;
            px = sx; py = sy; pz = sz;
            dx = fx; dy = fy; dz = fz;
            sl += 3 * (size_t)(nsteps - 1);
            if (l == 0) { sl[0] = px; sl[1] = py; sl[2] = pz; }
            i = 1;
        } else {
            if (l == 0) sline_len[slot] = nb - 1 + nsteps;
            have = false;
        }
    }
}

template <int NCH>
__global__ void __launch_bounds__(256, PROB_WAVES)
    phase2_prob_kernel(DevParams P, DevBufs B, const float *__restrict__ seeds, int nseeds, int rng_chunk,
                       const int *__restrict__ offsets, const int *__restrict__ dirs, int *__restrict__ sline_seed,
                       int *__restrict__ sline_len, float *__restrict__ sline, const int *__restrict__ order,
                       int *__restrict__ work) {
    extern __shared__ float4 smem4[];
    float *smem = reinterpret_cast<float *>(smem4);
    // vertices as x[], y[], z[], 0 past the last
    for (int i = threadIdx.x; i < 3 * 256 * NCH; i += blockDim.x) {
        const int a = i / (256 * NCH), v = i - a * (256 * NCH);
        smem[i] = (v < P.nverts) ? B.verts[3 * v + a] : 0.0f;
    }
    __syncthreads();
    flat_wave_prob<NCH>(P, B, smem, smem + 3 * 256 * NCH + (threadIdx.x >> 6) * prob_slot_floats(NCH), seeds, nseeds,
                        rng_chunk, offsets, dirs, sline_seed, sline_len, sline, order, work);
}

// -------------------------------------------------------------------------
// Plain PTT phase 2 (the queue's flat stepping).
//
// Same sub-step as ptt_substep, arranged for the latency of a lone wave and
// for issue slots:
//  - the vertex phase's 24 curves first run all their frames (no load is
//    waited for: each probe's LUT entry arrives while the next frame is
//    propagated and goes to LDS with the probe's position); then the 192
//    taps are shared by the slot's 32 lanes, 6 each instead of 8 on 24
//    lanes, their block reads in flight 3 at a time, and lane v adds its 8
//    values in probe order.  data_support instead waits for a LUT entry and
//    a block per probe;
//  - the tangent's own tap is read under the frames;
//  - frames skip their three norms' range tests one by one (one test of the
//    smallest and largest square; the rare failure redoes the frame), and
//    the last probe's normal and binormal, which nothing reads;
//  - a rejection round ends as soon as lane 0's candidate passes: the lowest
//    passing lane wins, and every lane has taken its three draws already;
//  - the disc's propagators and faces come from LDS, the face search from
//    two LDS reads (levels 1-3, then 4-5) instead of five dependent ones, and
//    the face scan from row shifts; the frame stays in registers.
// Same additions, products and draws in the same order: bit-identical.
//
// What bounds it: a wave's own chain.  A dependent instruction takes 8.4
// cycles, and a lone seed 8 us (19,000 cycles) a sub-step.  At 250,000 seeds
// (1,365 VALU instructions a sub-step, a third of them the 24 x 8 frames;
// data_support's loop took 1,881) the CUs issue 0.66 a cycle, and reads, 6.5 TB/s
// of them past L2, are open for 765 cycles: neither issue nor the fabric is at its
// limit, two waves per SIMD wait.  Against flat_slot<PTT> with the seeds in
// spatial order: 40 seeds 195 -> 151 ms (runs differ by as much), 4,001 352 ->
// 255 ms, 25,000 696 -> 480 ms, 250,000 3.95 -> 3.66 s.
// -------------------------------------------------------------------------
// 2 waves per SIMD and all of a group's taps in flight: at 3 waves (168
// registers, 29 spilled) with 3 taps 25,000 seeds take 714 ms instead of 618
// and 250,000 seeds 4.75 s instead of 4.39.
constexpr int PTT_WAVES = 2;
constexpr int PTT_BATCH = 6;                          // tap rounds in flight
constexpr int PTT_GROUP = 8;                          // probes whose taps are in LDS together
constexpr int PTT_ENTRIES = DISC_VERT_CNT * PTT_GROUP;
constexpr int PTT_TAB_FLOATS = DISC_VERT_CNT * 12 + 32 * 8;  // propagators [24][12], faces [32][8]
// frame 32, vertex pdf 32, face cdf 32, search 40, tap entries, tap values, flat state
constexpr int PTT_FLAT_FLOATS = 32 + 32 + 32 + 40 + 4 * PTT_ENTRIES + PTT_ENTRIES + FLAT_STATE_FLOATS;

struct PttFlatLds {
    PttLds init;       // the initial frame's arrays (init_frame_ptt)
    float *search;     // cdf of faces 0..30 ([30] = inf), then the midpoints of levels 1-3
    float4 *entry;     // probe position and LUT entry
    float *tap;        // tap values
    const float *tab;  // the workgroup's tables
};

constexpr int DPP_ROW_NEWBCAST = 0x150;

// check_point on the slot's lanes: wave_stop_begin's lane-parallel texels.
__device__ __forceinline__ int slot_stop_end(const DevParams &P, const WaveTap &r) {
    float acc = r.w * r.t;
#pragma unroll
    for (int k = 1; k < 8; ++k) acc = __builtin_fmaf(r.w, r.t, dpp0<DPP_ROW_SHR + 1>(acc));
    acc = dpp0<DPP_ROW_NEWBCAST + 7>(acc);
    if (acc == -1.0f) return CUSLINES_OUTSIDEIMAGE;
    return (acc > P.tc_threshold) ? CUSLINES_TRACKPOINT : CUSLINES_ENDPOINT;
}

// Value of the lane I places below in the slot (rows of 16 joined); what the
// lanes below I get is not used.
template <int I>
__device__ __forceinline__ float slot_shr(float v) {
    if (I == 16) return __uint_as_float(__builtin_amdgcn_permlane16_swap(__float_as_uint(v), __float_as_uint(v), false, false)[0]);
    const float r = dpp0<DPP_ROW_ROR + (I & 15)>(v);
    const float x = __uint_as_float(
        __builtin_amdgcn_permlane16_swap(__float_as_uint(r), __float_as_uint(r), false, false)[0]);
    return ((threadIdx.x & 15) < I) ? x : r;
}

// norm3 without its range test (the caller tests the squares).
__device__ __forceinline__ float norm3_raw(float &x, float &y, float &z) {
    const float n2 = __builtin_fmaf(z, z, __builtin_fmaf(y, y, x * x));
    const float inv = rsqrt_nr(n2);
    x *= inv; y *= inv; z *= inv;
    return n2;
}

// propagate_frame; the norms' range tests as one.
__device__ __forceinline__ void propagate_frame_fast(const float *p, float *f, float *direc) {
    float t[3], w[3], u[3], v[3];
#pragma unroll
    for (int i = 0; i < 3; ++i) {
        direc[i] = __builtin_fmaf(p[2], f[6 + i], __builtin_fmaf(p[1], f[3 + i], p[0] * f[i]));
        t[i] = __builtin_fmaf(p[5], f[6 + i], __builtin_fmaf(p[4], f[3 + i], p[3] * f[i]));
        w[i] = __builtin_fmaf(p[8], f[6 + i], __builtin_fmaf(p[7], f[3 + i], p[6] * f[i]));
    }
    const float nt = norm3_raw(t[0], t[1], t[2]);
    u[0] = __builtin_fmaf(w[1], t[2], -(w[2] * t[1]));
    u[1] = __builtin_fmaf(w[2], t[0], -(w[0] * t[2]));
    u[2] = __builtin_fmaf(w[0], t[1], -(w[1] * t[0]));
    const float nu = norm3_raw(u[0], u[1], u[2]);
    v[0] = __builtin_fmaf(t[1], u[2], -(t[2] * u[1]));
    v[1] = __builtin_fmaf(t[2], u[0], -(t[0] * u[2]));
    v[2] = __builtin_fmaf(t[0], u[1], -(t[1] * u[0]));
    const float nv = norm3_raw(v[0], v[1], v[2]);
    const float lo = __builtin_elementwise_minimum(__builtin_elementwise_minimum(nt, nu), nv);
    const float hi = __builtin_elementwise_maximum(__builtin_elementwise_maximum(nt, nu), nv);
    float g[9];
#pragma unroll
    for (int i = 0; i < 9; ++i) g[i] = f[i];
#pragma unroll
    for (int i = 0; i < 3; ++i) {
        f[i] = t[i]; f[3 + i] = u[i]; f[6 + i] = v[i];
        // here, not inside the branch below: no copies at its end
        asm volatile("" : "+v"(f[i]), "+v"(f[3 + i]), "+v"(f[6 + i]), "+v"(direc[i]));
    }
    if (__builtin_expect(!(lo > PTT_MIN_NORM2 && hi <= 3.40282347e+38f), 0)) {
#pragma unroll
        for (int i = 0; i < 9; ++i) f[i] = g[i];
        propagate_frame(p, f, direc);
    }
}

// The tangent alone (the last probe of a curve).
__device__ __forceinline__ void propagate_tangent(const float *p, float *f, float *direc) {
    float t[3];
#pragma unroll
    for (int i = 0; i < 3; ++i) {
        direc[i] = __builtin_fmaf(p[2], f[6 + i], __builtin_fmaf(p[1], f[3 + i], p[0] * f[i]));
        t[i] = __builtin_fmaf(p[5], f[6 + i], __builtin_fmaf(p[4], f[3 + i], p[3] * f[i]));
    }
    norm3<0>(t[0], t[1], t[2]);
    f[0] = t[0]; f[1] = t[1]; f[2] = t[2];
}

// Vertex phase of a sub-step on frame `fr` at (px, py, pz): the 24 supports
// (0 below the cut) into S.init.vert_pdf, the tangent's tap into first_val.
// `check`: the point's stop-map check, left over from the sub-step before,
// is done under the frames.  1, 0 when no vertex passes, -1 when the check
// ends the pass.
__device__ __forceinline__ int ptt_vertices(const DevParams &P, const DevBufs &B, const PttFlatLds &S, const float *fr,
                                            bool check, float px, float py, float pz, float *first_val) {
    const int l = lane32();
    const int Q = P.probe_quality;
    const uint32_t lv0 = B.lut[lut_index(P, fr[0], fr[1], fr[2])];
    const WaveTap stop = wave_stop_begin(P, B.stop, px, py, pz);
    float f[9], p[9];
    float x = px, y = py, z = pz;
    const float4 pa = *reinterpret_cast<const float4 *>(S.tab + 12 * min(l, DISC_VERT_CNT - 1));
    const float4 pb = *reinterpret_cast<const float4 *>(S.tab + 12 * min(l, DISC_VERT_CNT - 1) + 4);
    p[0] = pa.x; p[1] = pa.y; p[2] = pa.z; p[3] = pa.w;
    p[4] = pb.x; p[5] = pb.y; p[6] = pb.z; p[7] = pb.w;
    p[8] = S.tab[12 * min(l, DISC_VERT_CNT - 1) + 8];
#pragma unroll
    for (int i = 0; i < 9; ++i) f[i] = fr[i];
    Tap t0;
    float sup = 0.0f;
    for (int g = 0; g < Q; g += PTT_GROUP) {
        const int cnt = min(PTT_GROUP, Q - g);
        if (l < DISC_VERT_CNT) {
            // LUT entries of the last three probes, on their way
            uint32_t lv1 = 0u, lv2 = 0u, lv3 = 0u;
            for (int i = 0; i < cnt; ++i) {
                float d[3];
                if (g + i + 1 < Q) propagate_frame_fast(p, f, d); else propagate_tangent(p, f, d);
                x += d[0]; y += d[1]; z += d[2];
                const uint32_t nlv = B.lut[lut_index(P, f[0], f[1], f[2])];
                float *e = reinterpret_cast<float *>(S.entry + i * DISC_VERT_CNT + l);
                e[0] = x; e[1] = y; e[2] = z;
                if (i >= 3) e[3 - 3 * 4 * DISC_VERT_CNT] = __uint_as_float(lv3);
                lv3 = lv2; lv2 = lv1; lv1 = nlv;
            }
            float *e = reinterpret_cast<float *>(S.entry + (cnt - 1) * DISC_VERT_CNT + l);
            if (cnt >= 3) e[3 - 2 * 4 * DISC_VERT_CNT] = __uint_as_float(lv3);
            if (cnt >= 2) e[3 - 4 * DISC_VERT_CNT] = __uint_as_float(lv2);
            e[3] = __uint_as_float(lv1);
        }
        if (g == 0) {
            t0 = tap_begin(P, B, lv0, px, py, pz);
            if (check && slot_stop_end(P, stop) != CUSLINES_TRACKPOINT) return -1;
        }
        WAVE_SYNC();
        // the group's taps: entry 32 r + l in round r
        const int ne = cnt * DISC_VERT_CNT;
        uint32_t slow = 0u;  // rounds whose cell has no corner block
        constexpr int BATCH = PTT_BATCH, ROUNDS = (PTT_ENTRIES + 31) / 32;
#pragma unroll
        for (int r0 = 0; r0 < ROUNDS; r0 += BATCH) {
            Tap t[BATCH];
#pragma unroll
            for (int u = 0; u < BATCH; ++u) {
                const int e = 32 * (r0 + u) + l;
                const float4 q = S.entry[min(e, ne - 1)];
                t[u] = tap_begin(P, B, __float_as_uint(q.w), q.x, q.y, q.z);
            }
#pragma unroll
            for (int u = 0; u < BATCH; ++u) {
                const int e = 32 * (r0 + u) + l;
                if (e < ne) S.tap[e] = corner_blend(t[u].a, t[u].b, t[u].g, t[u].lo, t[u].hi);
                if (!t[u].fast) slow |= 1u << (r0 + u);
            }
        }
        if (half_ballot(slow != 0u)) {
            for (int r = 0; r < ROUNDS; ++r) {
                const int e = 32 * r + l;
                if (((slow >> r) & 1u) && e < ne) {
                    const float4 q = S.entry[e];
                    const uint32_t lv = __float_as_uint(q.w);
                    const int idx = (int)(lv & 0xffffu);
                    const int tx = idx & (P.nx - 1), ty = (idx >> P.log2x) & (P.ny - 1), tz = idx >> (P.log2x + P.log2y);
                    S.tap[e] = tiled_sample(P, B.data, (float)(tx * P.dimx) + q.x, (float)(ty * P.dimy) + q.y,
                                            (float)(tz * P.dimz) + q.z, tx, ty, tz);
                }
            }
        }
        WAVE_SYNC();
        if (g == 0) {
            *first_val = tap_end(P, B, t0);
            sup = *first_val;
        }
        if (l < DISC_VERT_CNT) {
            float v[PTT_GROUP];
#pragma unroll
            for (int i = 0; i < PTT_GROUP; ++i) v[i] = S.tap[i * DISC_VERT_CNT + l];  // past cnt: not used
#pragma unroll
            for (int i = 0; i < PTT_GROUP; ++i) sup = (i < cnt) ? sup + v[i] : sup;
        }
        if (g + PTT_GROUP < Q) WAVE_SYNC();
    }
    const bool ok = l < DISC_VERT_CNT && !(sup < P.min_support_f);
    S.init.vert_pdf[l] = ok ? sup : 0.0f;
    const uint32_t any = half_ballot(ok);
    WAVE_SYNC();
    return any != 0u ? 1 : 0;
}

// Support of a rejection candidate, up to stop_at; ends early when lane 0's
// candidate has passed.
__device__ __forceinline__ float ptt_candidate(const DevParams &P, const DevBufs &B, float support, float px, float py,
                                               float pz, float k1, float k2, const float *fr, float stop_at) {
    uint32_t pass = half_ballot(support >= stop_at);
    if (pass & 1u) return support;
    float prop[9], pf[9], direc[3];
#pragma unroll
    for (int i = 0; i < 9; ++i) pf[i] = fr[i];
    prepare_propagator(k1, k2, P.probe_step, prop);
    propagate_frame_fast(prop, pf, direc);
    px += direc[0]; py += direc[1]; pz += direc[2];
    uint32_t idx = B.lut[lut_index(P, pf[0], pf[1], pf[2])];
    for (int i = 0; i < P.probe_quality; ++i) {
        if (!(support >= stop_at)) {
            const Tap t = tap_begin(P, B, idx, px, py, pz);
            if (i + 1 < P.probe_quality) {
                propagate_frame_fast(prop, pf, direc);
                px += direc[0]; py += direc[1]; pz += direc[2];
                idx = B.lut[lut_index(P, pf[0], pf[1], pf[2])];
            }
            support += tap_end(P, B, t);
        }
        pass = half_ballot(support >= stop_at);
        if ((pass & 1u) || pass == 0xffffffffu) break;
    }
    return support;
}

// One sub-step (non-initial): 1 with the frame `fr` moved and the new
// direction, 0 when there is none, -1 when the point's pending stop check
// ends the pass.
__device__ __forceinline__ int ptt_flat_substep(const DevParams &P, const DevBufs &B, const PttFlatLds &S, float *fr,
                                                int face, bool check, Philox &rng, float px, float py, float pz,
                                                float *nx, float *ny, float *nz) {
    const int l = lane32();
    float first_val;
    const int vt = ptt_vertices(P, B, S, fr, check, px, py, pz, &first_val);
    if (vt <= 0) return vt;
    // face CDF (ptt_face_cdf): lane f < 31 holds face f; `face` packs its vertices
    float c = 0.0f;
    {
        const float a = S.init.vert_pdf[face & 0xff], b = S.init.vert_pdf[(face >> 8) & 0xff],
                    d = S.init.vert_pdf[face >> 16];
        c = (a == 0.0f || b == 0.0f || d == 0.0f || l >= DISC_FACE_CNT) ? 0.0f : (a + b) + d;
    }
    {
        float o = slot_shr<1>(c);
        c = (l >= 1 && l < DISC_FACE_CNT) ? c + o : c;
        o = slot_shr<2>(c);
        c = (l >= 2 && l < DISC_FACE_CNT) ? c + o : c;
        o = slot_shr<4>(c);
        c = (l >= 4 && l < DISC_FACE_CNT) ? c + o : c;
        o = slot_shr<8>(c);
        c = (l >= 8 && l < DISC_FACE_CNT) ? c + o : c;
        o = slot_shr<16>(c);
        c = (l >= 16 && l < DISC_FACE_CNT) ? c + o : c;
    }
    // the search's order: 31 values, the last one's test always true, and
    // the midpoints of levels 1-3 (15; 7, 23; 3, 11, 19, 27)
    S.search[l] = (l >= DISC_FACE_CNT - 1) ? __builtin_inff() : c;
    if ((l & 3) == 3 && l < 28) S.search[32 + (l >> 2)] = c;
    const float last = shfl32(c, DISC_FACE_CNT - 1);
    WAVE_SYNC();
    if (last == 0.0f) return 0;
    const float4 ma = *reinterpret_cast<const float4 *>(S.search + 32);      // cdf at 3, 7, 11, 15
    const float4 mb = *reinterpret_cast<const float4 *>(S.search + 32 + 4);  // cdf at 19, 23, 27, -
    const float stop_at = P.ptt_nonneg ? P.min_support_f : __builtin_inff();
    for (int round = 0; round < 1024 / 32; ++round) {
        float r1 = rng.uniform(), r2 = rng.uniform();
        if (r1 + r2 > 1.0f) { r1 = 1.0f - r1; r2 = 1.0f - r2; }
        const float tmp = rng.uniform() * last;
        // ptt_substep's binary search over [0, 30]
        const bool l1 = ma.w >= tmp;
        const bool l2 = (l1 ? ma.y : mb.y) >= tmp;
        const float m3 = l1 ? (l2 ? ma.x : ma.z) : (l2 ? mb.x : mb.z);
        const bool l3 = m3 >= tmp;
        const int base = (l1 ? 0 : 16) + (l2 ? 0 : 8) + (l3 ? 0 : 4);
        const float4 q = *reinterpret_cast<const float4 *>(S.search + base);
        const bool l4 = q.y >= tmp;
        const bool l5 = (l4 ? q.x : q.z) >= tmp;
        const int jj = min(base + (l4 ? 0 : 2) + (l5 ? 0 : 1), DISC_FACE_CNT - 1);
        const float4 fa = *reinterpret_cast<const float4 *>(S.tab + DISC_VERT_CNT * 12 + 8 * jj);
        const float2 fb = *reinterpret_cast<const float2 *>(S.tab + DISC_VERT_CNT * 12 + 8 * jj + 4);
        float k1 = __builtin_fmaf(r2, fa.z, __builtin_fmaf(r1, fa.y, fa.x));
        float k2 = __builtin_fmaf(r2, fb.y, __builtin_fmaf(r1, fb.x, fa.w));
        const float sup = ptt_candidate(P, B, first_val, px, py, pz, k1, k2, fr, stop_at);
        const uint32_t msk = half_ballot(sup >= P.min_support_f);
        if (msk == 0u) continue;
        const int win = __ffs(msk) - 1;
        k1 = shfl32(k1, win);
        k2 = shfl32(k2, win);
        float prop[9], d[3];
        prepare_propagator(k1, k2, P.ptt_sub_step, prop);
        propagate_frame_fast(prop, fr, d);
        norm3<0>(d[0], d[1], d[2]);
        *nx = d[0]; *ny = d[1]; *nz = d[2];
        return 1;
    }
    return 0;
}

// flat_slot's loop for a plain PTT slot.
__device__ void flat_slot_ptt(const DevParams &P, const DevBufs &B, const PttFlatLds &S, float *st,
                              const float *__restrict__ seeds, int nseeds, int rng_chunk,
                              const int *__restrict__ offsets, const int *__restrict__ dirs,
                              int *__restrict__ sline_seed, int *__restrict__ sline_len, float *__restrict__ sline,
                              const int *__restrict__ order, int *__restrict__ work) {
    const int l = lane32();
    const int step_frac = P.step_frac, MAXL = P.max_sline_len;
    const int nsub_max = MAXL * step_frac;
    const double sub = P.step_d / (double)step_frac;
    const size_t slot_f = (size_t)2 * MAXL * 3;
    int *si = reinterpret_cast<int *>(st);  // s, ndir, next direction, offsets[s], slot, nb
    float *sf = st + 8;                     // seed point [0..2], direction [3..5]
    if (l == 0) { si[1] = 0; si[2] = 0; }
    WAVE_SYNC();
    const int fl = min(l, DISC_FACE_CNT - 1);
    const int face = c_disc_face[fl * 3] | (c_disc_face[fl * 3 + 1] << 8) | (c_disc_face[fl * 3 + 2] << 16);
    Philox rng;
    int qk = 0;
    bool have = false, check = false;
    int pass = 0, i = 1, ri = 1, qi = 0;  // step i = qi * step_frac + ri
    float px = 0.0f, py = 0.0f, pz = 0.0f;
    float fr[9];
#pragma unroll
    for (int k = 0; k < 9; ++k) fr[k] = 0.0f;
    float *sl = sline;
    for (;;) {
        if (!have) {
            // the next direction of this seed, or of the next seeds
            while (qk < QUEUES) {
                const int di = si[2];
                if (di >= si[1]) {
                    const QueueRange qr = queue_range(work, qk);
                    const int lo = qr.lo, hi = qr.hi;
                    int q = 0;
                    if (l == 0 && lo < hi) q = atomicAdd(work + qr.counter, 1);
                    q = shfl32(q, 0);
                    if (lo + q >= hi) { ++qk; continue; }
                    const int s = order[lo + q];
                    const int nd = (P.slot_cap > 0 && offsets[s + 1] > P.slot_cap) ? 0 : offsets[s + 1] - offsets[s];
                    rng.init(((uint64_t)P.seed_hi << 32) | P.seed_lo, (uint64_t)32 * (uint64_t)(s % rng_chunk) + l + 1);
                    WAVE_SYNC();
                    if (l == 0) {
                        si[0] = s; si[1] = nd; si[2] = 0; si[3] = offsets[s];
                        sf[0] = seeds[3 * s]; sf[1] = seeds[3 * s + 1]; sf[2] = seeds[3 * s + 2];
                    }
                    WAVE_SYNC();
                    continue;
                }
                const int s = si[0], off = si[3] + di;
                const float sx = sf[0], sy = sf[1], sz = sf[2];
                const int vi = dirs[(size_t)s * P.nverts + di];
                const float fx = B.verts[3 * vi], fy = B.verts[3 * vi + 1], fz = B.verts[3 * vi + 2];
                float *cur = sline + (size_t)off * slot_f;
                WAVE_SYNC();
                if (l == 0) {
                    sline_seed[off] = s;
                    si[2] = di + 1; si[4] = off;
                    sf[3] = fx; sf[4] = fy; sf[5] = fz;
                }
                WAVE_SYNC();
                PttLds in = S.init;
                if (!init_frame_ptt(P, B, in, rng, fx, fy, fz, sx, sy, sz)) {
                    if (l == 0) {
                        sline_len[off] = 1;
                        cur[0] = sx; cur[1] = sy; cur[2] = sz;
                    }
                    continue;
                }
                // backward pass on the frame at [0..8]
                pass = 0;
                px = sx; py = sy; pz = sz;
#pragma unroll
                for (int k = 0; k < 9; ++k) fr[k] = S.init.frame[k];
                sl = cur;
                if (l == 0) { sl[0] = px; sl[1] = py; sl[2] = pz; }
                i = 1; qi = (step_frac == 1) ? 1 : 0; ri = (step_frac == 1) ? 0 : 1;
                have = true;
                break;
            }
            if (!have) break;  // the queues are empty
        }
        // One sub-step of the pass (tracker's loop body).  With `check` the
        // point is that of step i, already moved and stored, and its stop
        // check comes with the next sub-step; it passes before i counts on.
        const int ni = check ? i + 1 : i;  // the step to take now
        bool end = true;
        if (ni < nsub_max) {
            float dx = 0.0f, dy = 0.0f, dz = 0.0f;
            const int nd = ptt_flat_substep(P, B, S, fr, face, check, rng, px, py, pz, &dx, &dy, &dz);
            if (check && nd >= 0) {
                ++i;
                if (++ri == step_frac) { ri = 0; ++qi; }
            }
            if (nd > 0) {
                px = (float)__builtin_fma((double)(dx / 1.0f), sub, (double)px);
                py = (float)__builtin_fma((double)(dy / 1.0f), sub, (double)py);
                pz = (float)__builtin_fma((double)(dz / 1.0f), sub, (double)pz);
                if (l == 0 && ri == 0) {
                    float *o = sl + 3 * (size_t)qi;
                    o[0] = px; o[1] = py; o[2] = pz;
                }
                check = true;
                end = false;
            }
        } else if (check && slot_stop_end(P, wave_stop_begin(P, B.stop, px, py, pz)) == CUSLINES_TRACKPOINT) {
            ++i;
            if (++ri == step_frac) { ri = 0; ++qi; }
        }
        if (!end) continue;
        check = false;
        // the pass ends at step i (tracker's tail)
        int nsteps = qi;
        if (ri != 0 && i < step_frac * (MAXL - 1)) {
            ++nsteps;
            if (l == 0) {
                float *o = sl + 3 * (size_t)nsteps;
                o[0] = px; o[1] = py; o[2] = pz;
            }
        }
        const int off = si[4];
        float *cur = sline + (size_t)off * slot_f;
        if (pass == 0) {
            const int nb = nsteps;
            MEM_SYNC();
            for (int j = l; j < nb / 2; j += 32) {
                float *a = cur + 3 * (size_t)j, *b = cur + 3 * (size_t)(nb - 1 - j);
                const float a0 = a[0], a1 = a[1], a2 = a[2];
                a[0] = b[0]; a[1] = b[1]; a[2] = b[2];
                b[0] = a0; b[1] = a1; b[2] = a2;
            }
            MEM_SYNC();
            if (l == 0) si[5] = nb;
            // forward pass on the frame at [9..17], from the seed point at index nb - 1
            pass = 1;
            px = sf[0]; py = sf[1]; pz = sf[2];
#pragma unroll
            for (int k = 0; k < 9; ++k) fr[k] = S.init.frame[9 + k];
            sl = cur + 3 * (size_t)(nb - 1);
            if (l == 0) { sl[0] = px; sl[1] = py; sl[2] = pz; }
            i = 1; qi = (step_frac == 1) ? 1 : 0; ri = (step_frac == 1) ? 0 : 1;
            WAVE_SYNC();
        } else {
            if (l == 0) sline_len[off] = si[5] - 1 + nsteps;
            have = false;
        }
    }
}

__global__ void __launch_bounds__(256, PTT_WAVES)
    phase2_ptt_kernel(DevParams P, DevBufs B, const float *__restrict__ seeds, int nseeds, int rng_chunk,
                      const int *__restrict__ offsets, const int *__restrict__ dirs, int *__restrict__ sline_seed,
                      int *__restrict__ sline_len, float *__restrict__ sline, const int *__restrict__ order,
                      int *__restrict__ work) {
    extern __shared__ float4 smem4[];
    float *smem = reinterpret_cast<float *>(smem4);
    for (int i = threadIdx.x; i < DISC_VERT_CNT * 12; i += blockDim.x) {
        const int v = i / 12, k = i - 12 * v;
        smem[i] = (k < 9) ? B.vprop[9 * v + k] : 0.0f;
    }
    // per face: the curvatures of vertex 0 and the two edges from it
    for (int f = threadIdx.x; f < 32; f += blockDim.x) {
        float *o = smem + DISC_VERT_CNT * 12 + 8 * f;
        const int g = min(f, DISC_FACE_CNT - 1);
        const float *vk = B.vprop + VPROP_K;
        const int f0 = c_disc_face[g * 3], f1 = c_disc_face[g * 3 + 1], f2 = c_disc_face[g * 3 + 2];
        o[0] = vk[2 * f0];
        o[1] = vk[2 * f1] - vk[2 * f0];
        o[2] = vk[2 * f2] - vk[2 * f0];
        o[3] = vk[2 * f0 + 1];
        o[4] = vk[2 * f1 + 1] - vk[2 * f0 + 1];
        o[5] = vk[2 * f2 + 1] - vk[2 * f0 + 1];
        o[6] = o[7] = 0.0f;
    }
    __syncthreads();
    float *base = smem + PTT_TAB_FLOATS + (threadIdx.x >> 5) * PTT_FLAT_FLOATS;
    PttFlatLds S;
    S.init.frame = base;
    S.init.vert_pdf = base + 32;
    S.init.face_cdf = base + 64;
    S.init.act = nullptr;
    S.search = base + 96;
    S.entry = reinterpret_cast<float4 *>(base + 136);
    S.tap = base + 136 + 4 * PTT_ENTRIES;
    S.tab = smem;
    flat_slot_ptt(P, B, S, base + PTT_FLAT_FLOATS - FLAT_STATE_FLOATS, seeds, nseeds, rng_chunk, offsets, dirs,
                  sline_seed, sline_len, sline, order, work);
}

// One seed per 32-lane slot, static assignment.
template <int MODEL, int V = 0>
__global__ void __launch_bounds__(256) phase2_kernel(DevParams P, DevBufs B, const float *__restrict__ seeds,
                                                     int nseeds, int rng_chunk, const int *__restrict__ offsets,
                                                     const int *__restrict__ dirs, int *__restrict__ sline_seed,
                                                     int *__restrict__ sline_len, float *__restrict__ sline) {
    extern __shared__ float smem[];
    const float *sv = B.verts;
    int svf = 0;
    if (MODEL == CUSLINES_PROB) {  // the cone test reads every vertex at every step
        for (int i = threadIdx.x; i < 3 * P.nverts; i += blockDim.x) smem[i] = B.verts[i];
        sv = smem;
        svf = verts_floats(P);
    }
    DevBufs BL;
    svf += stage_network<V>(B, smem + svf, BL);
    __syncthreads();
    const int nslots = blockDim.x >> 5;
    const int slot = threadIdx.x >> 5;
    const int s = blockIdx.x * nslots + slot;
    if (s >= nseeds) return;
    SlotLds S;
    bind_slot<MODEL>(P, false, smem + svf + slot * slot_floats(MODEL, false, P.nv32, P.t32, P.hr32), S);
    track_seed<MODEL, V>(P, BL, sv, S, s, seeds, rng_chunk, offsets, dirs, sline_seed, sline_len, sline);
}

// Persistent work queue: a fixed grid of slots; each 32-lane slot takes the
// next seed from a counter as soon as its previous seed is done, so seeds of
// very uneven length keep every slot busy.  `order` lists the seeds in
// processing order and `work` holds WORK_INTS ints, the zeroed counters and
// where each class starts in that order (queue_range): both as spatial_order
// left them in the same call, since the class starts fit no other order.  The
// order changes no streamline: random streams and output slots follow the seed
// index.
// The per-seed nesting of plain PTT and of its tap count is held to 128 VGPRs
// (4 waves per SIMD): the few spills cost less than the latency hiding gained.
// The bootstrap getters likewise (4 waves per SIMD, which their 5 KB of LDS per
// slot allow), but for few seeds in flight (V == 6: 2 waves and 256 VGPRs, the
// products' loads in flight).  The flat loop of the learned proposal (V == 5)
// needs about 170 VGPRs and at 128 spills inside its loop, so it runs at 3 waves
// per SIMD (168 VGPRs, 17 spilled), in 768-thread workgroups (one staged copy of
// the network serves 24 slots).
template <int MODEL, int V = 0>
__global__ void __launch_bounds__((MODEL == CUSLINES_PTT && V == 1)   ? 512
                                  : (MODEL == CUSLINES_PTT && V == 5) ? 768
                                                                      : 256,
                                  (MODEL == CUSLINES_PTT && V == 5) ? 3
                                  : (MODEL == CUSLINES_PTT && V != 2)           ? 4
                                                                                : (V == 6                       ? 2
                                                                                 : MODEL <= CUSLINES_PROB ? 4
                                                                                                          : 1))
    phase2_queue_kernel(DevParams P, DevBufs B, const float *__restrict__ seeds,
                                                           int nseeds, int rng_chunk, const int *__restrict__ offsets,
                                                           const int *__restrict__ dirs, int *__restrict__ sline_seed,
                                                           int *__restrict__ sline_len, float *__restrict__ sline,
                                                           const int *__restrict__ order, int *__restrict__ work) {
    extern __shared__ float smem[];
    const float *sv = B.verts;
    int svf = 0;
    if (MODEL == CUSLINES_PROB) {  // the cone test reads every vertex at every step
        for (int i = threadIdx.x; i < 3 * P.nverts; i += blockDim.x) smem[i] = B.verts[i];
        sv = smem;
        svf = verts_floats(P);
    }
    DevBufs BL;
    svf += stage_network<V>(B, smem + svf, BL);
    __syncthreads();
    const int slot = threadIdx.x >> 5;
    const int l = lane32();
    SlotLds S;
    const int stride =
        slot_floats(MODEL, false, P.nv32, P.t32, P.hr32) + ((V >= 4) ? FLAT_STATE_FLOATS : 0);
    bind_slot<MODEL>(P, false, smem + svf + slot * stride, S);
    if constexpr (V >= 4) {
        flat_slot<MODEL, V == 5, V == 6>(P, BL, sv, S, smem + svf + slot * stride + stride - FLAT_STATE_FLOATS, seeds,
                                 nseeds, rng_chunk, offsets, dirs, sline_seed, sline_len, sline, order, work);
        return;
    }
    // Workgroups are dispatched to the 8 XCDs round-robin.  Each XCD first
    // drains its own eighth of the (spatially sorted) seed order, so an XCD's
    // L2 serves one region of the volume, then helps with the others.
    for (int k = 0; k < QUEUES; ++k) {
        const QueueRange qr = queue_range(work, k);
        const int lo = qr.lo, hi = qr.hi;
        for (;;) {
            int q = 0;
            if (l == 0 && lo < hi) q = atomicAdd(work + qr.counter, 1);
            q = shfl32(q, 0);
            if (lo + q >= hi) break;
            const int s = order[lo + q];
            track_seed<MODEL, V>(P, BL, sv, S, s, seeds, rng_chunk, offsets, dirs, sline_seed, sline_len, sline);
        }
    }
}

// -------------------------------------------------------------------------
// Bootstrap phase 2, batched on the matrix cores.
//
// Same algorithm as the scalar path above (get_direction_boot_d,
// boot.cu:393-608; tracker_boot_d, boot.cu:720-824; genStreamlinesMergeBoot_k,
// boot.cu:826-980), organised for MFMA: a 512-thread workgroup holds
// BB_SLOTS = 16 seed slots, one per 32-lane half-wave, that advance in
// lockstep -- every round, each active slot makes one getter attempt.  The
// per-slot work (gather, resampling, normalisation, peaks, closest peak, the
// step and its stop check) runs on the slot's own 32 lanes with the scalar
// path's code; the matrix products of the attempt run batched over the 16
// slots on v_mfma_f32_16x16x4_f32 (fp32 operands, fp32 accumulation):
//   phase B  [H; R] (2 hr16 x hr16) . X (hr16 x 16)    -> H.d, R.d
//   phase D  [dq | -db] (dn16 x 2 hr16) . [xf; msk]    -> model coefficients
//   phase E  S (nv16 x dn16) . C (dn16 x 16)           -> ODF on the sphere
//   phase F  the peak tests of every slot's vertices on all 8 waves, then each
//            slot's sort, closest peak and step on its own lanes
// Each matrix element read from L2 thus serves 16 seeds instead of one.  The
// products sum in another order than the reference's lane-strided dot
// products, so results agree with the scalar path within float rounding:
// peak indices are the same except at near-ties, and a streamline is
// identical up to the first step whose peak choice flips.
// What bounds it: a run lasts as long as its longest seed's chain of rounds
// (some 3000 of them), and a round is a chain of latencies -- barriers, L2
// reads of matrix rows, LDS -- of 54 k cycles for a lone slot when every phase
// ran on the slot's own lanes and one load was in flight at a time, about 40 k
// now; past some 50 000 seeds it is the vector work of 16 slots a workgroup.
// Measured with both variants below at their best, before | after: CSA 100
// seeds on 46x55x41 14.4 | 7.9 ms, 25 000 on 81x106x76 122 | 74 ms, 150 000
// 326 | 229 ms; 6001 seeds of 270 directions, order 8, 115 | 68 ms; OPDT
// 40 000 96 | 64 ms.
// Matrices (uploaded zero padded, row-major): hr_mat [2 hr16][hr16],
// fit_mat [dn16][2 hr16], odf_mat [nv16][dn16].  LDS per slot: the scalar
// slot's regions, the stride padded to 4 mod 32 floats so the 16 slots' rows
// sit in distinct LDS banks for the MFMA operand reads and result writes.
// -------------------------------------------------------------------------
constexpr int BB_SLOTS = 16, BB_THREADS = 512, BB_WAVES = BB_THREADS / 64;
constexpr int BB_ROWS = 320 / 32;  // rows of 32 DWI channels (boot_batch_fits)
constexpr int BB_MAX_ATTEMPTS = 5;  // NATTEMPTS of tracker_boot_d (boot.cu:757)

typedef float bb_v4 __attribute__((ext_vector_type(4)));

__host__ __device__ inline int bb_slot_stride(int nv32, int t32, int hr32) {
    return ((slot_floats(CUSLINES_CSA, false, nv32, t32, hr32) + 27) & ~31) + 4;
}

// Tiles t = wave, wave + 8, ... (t < ntiles) of Y = A . X over the 16 slots.
// A: global row-major [ntiles * 16][lda], K (<= lda) a multiple of 16, zero
// padded.  Slot n's operand is X[n * ss + k] (k < K), or X2[n * ss + k - ksplit]
// for k >= ksplit; its result rows go to Y[n * ss + row], or Y2[n * ss + row -
// ysplit] for row >= ysplit, rows >= ymax dropped.  Lane l of a wave supplies
// A[l % 16][k] and X_{l % 16}[k] of each step and holds Y rows 4 (l / 16) + r;
// within a 16-wide chunk of K, lane group q = l / 16 reads the contiguous k =
// 16 c + 4 q + (0..3) as one 16-byte load and MFMA step s takes component s.
// wmax, wmin (optional): this wave's maximum (NaN passed over) and minimum
// (NaN if any is) of each slot's result rows < ymax, written to
// wmax / wmin[wave * 16 + slot].
// UN steps of K have their loads in flight together (the wave index is made
// scalar, so that no tile's loads sit behind a divergent branch): a step's
// matrix rows come from L2, and one load round trip per step was most of
// these products' time.
template <int MAXT, int UN, bool CSA_ROW0 = false>
__device__ __forceinline__ void bb_gemm(const float *__restrict__ A, int lda, int K, int ntiles, const float *X,
                                        const float *X2, int ksplit, float *Y, float *Y2, int ysplit, int ymax,
                                        int ss, float *wmax = nullptr, float *wmin = nullptr) {
    int lane = threadIdx.x & 63;
    asm volatile("" : "+v"(lane));  // addresses are formed here, not kept in registers around the round
    const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int n = lane & 15, q = lane >> 4;
    bb_v4 acc[MAXT];
#pragma unroll
    for (int i = 0; i < MAXT; ++i) acc[i] = bb_v4{0.0f, 0.0f, 0.0f, 0.0f};
    if (w < ntiles) {
        const int aoff = n * lda + 4 * q;
        for (int k0 = 0; k0 < K; k0 += 16 * UN) {
            float4 a[UN][MAXT], b[UN];
#pragma unroll
            for (int u = 0; u < UN; ++u) {
                const int k = min(k0 + 16 * u, K - 16);  // past the end: re-read, not used
#pragma unroll
                for (int i = 0; i < MAXT; ++i) {
                    const int t = min(w + BB_WAVES * i, ntiles - 1);  // past the last tile: re-read, dropped below
                    a[u][i] = *reinterpret_cast<const float4 *>(A + (size_t)t * 16 * lda + k + aoff);
                }
                const float *xs = (k < ksplit) ? X + n * ss + k : X2 + n * ss + (k - ksplit);
                b[u] = *reinterpret_cast<const float4 *>(xs + 4 * q);
            }
#pragma unroll
            for (int u = 0; u < UN; ++u) {
                if (k0 + 16 * u < K) {
#pragma unroll
                    for (int i = 0; i < MAXT; ++i) {
                        acc[i] = __builtin_amdgcn_mfma_f32_16x16x4f32(a[u][i].x, b[u].x, acc[i], 0, 0, 0);
                        acc[i] = __builtin_amdgcn_mfma_f32_16x16x4f32(a[u][i].y, b[u].y, acc[i], 0, 0, 0);
                        acc[i] = __builtin_amdgcn_mfma_f32_16x16x4f32(a[u][i].z, b[u].z, acc[i], 0, 0, 0);
                        acc[i] = __builtin_amdgcn_mfma_f32_16x16x4f32(a[u][i].w, b[u].w, acc[i], 0, 0, 0);
                    }
                }
            }
        }
    }
    if (wmax) {
        float pm = REAL_MIN, mn = REAL_MAX;
#pragma unroll
        for (int i = 0; i < MAXT; ++i) {
            const int t = w + BB_WAVES * i;
            const int row = 16 * t + 4 * q;
            if (t < ntiles) {
#pragma unroll
                for (int r = 0; r < 4; ++r)
                    if (row + r < ymax) {
                        pm = fmaxf(pm, acc[i][r]);
                        mn = __builtin_elementwise_minimum(mn, acc[i][r]);
                    }
            }
        }
        pm = fmaxf(pm, __shfl_xor(pm, 16));
        pm = fmaxf(pm, __shfl_xor(pm, 32));
        mn = __builtin_elementwise_minimum(mn, __shfl_xor(mn, 16));
        mn = __builtin_elementwise_minimum(mn, __shfl_xor(mn, 32));
        if (q == 0) {
            wmax[w * 16 + n] = pm;
            wmin[w * 16 + n] = mn;
        }
    }
#pragma unroll
    for (int i = 0; i < MAXT; ++i) {
        const int t = w + BB_WAVES * i;
        if (t < ntiles) {
            int row = 16 * t + 4 * q;
            if (CSA_ROW0 && row == 0) acc[i].x = CSA_C0;  // CSA's constant term (boot.cu:363-368)
            float *y = Y + n * ss;
            if (row >= ysplit) { y = Y2 + n * ss; row -= ysplit; }
            if (row + 3 < ymax) {
                *reinterpret_cast<float4 *>(y + row) = float4{acc[i].x, acc[i].y, acc[i].z, acc[i].w};
            } else {
                if (row < ymax) y[row] = acc[i].x;
                if (row + 1 < ymax) y[row + 1] = acc[i].y;
                if (row + 2 < ymax) y[row + 2] = acc[i].z;
            }
        }
    }
}

// The models' transforms of the signal (gemv_xf) with the hardware base-2
// logarithm: the batched kernel's results already differ from the
// reference's in the last bits, and two series logarithms per channel (CSA)
// are a large share of its per-slot work.
template <int XF>
__device__ __forceinline__ float bb_xf(float x) {
    constexpr float LN2 = 0.693147180559945309f;
    if (XF == 1) {
        const float lx = __builtin_amdgcn_logf(x) * LN2;
        return ((-lx) * (1.5f + lx)) * x;
    }
    const float c = fminf(fmaxf(x, 0.001f), 0.999f);
    return __builtin_amdgcn_logf(-(__builtin_amdgcn_logf(c) * LN2)) * LN2;
}

// peak_directions_d on the ODF thresholded at `thr` (values below it read as
// 0, tracking_helpers.cu:75-245 after generate_streamlines_cuda.cu's
// threshold) without writing the thresholded array: the adjacency form of
// peak_directions with the threshold applied to every value it reads.  A
// peak is never below thr (its thresholded value would be 0 with no
// strictly smaller neighbour), so the kept candidates' values, the sort
// keys, are the raw ODF values.  Needs the adjacency table (PeakParams::nbr).
__device__ int bb_peaks_all(const PeakParams &P, const float *odf, float thr, uint16_t *cand, const float *sv) {
    const int l = lane32();
    const int nv = P.nverts;
    uint32_t pk = 0u;
    float mn = REAL_MAX, m = REAL_MIN;
    if (thr > 0.0f) {
        // With thr > 0 the thresholded test reduces to the raw values: a
        // vertex whose value x is below thr (or NaN) reads as 0 and has no
        // strictly smaller thresholded neighbour, so it is no peak; for x >=
        // thr, a neighbour y is smaller after thresholding iff y < x and
        // larger iff y > x.  So x is a peak iff x >= thr, the minimum of its
        // raw neighbours is below x and their maximum is not above it
        // (fminf / fmaxf pass over a NaN neighbour as the comparisons do).
        // The largest peak value is kept on the way: max(x + c) over the
        // peaks is max(x) + c, rounding being monotone.
        float pmax = REAL_MIN;
        for (int r0 = 0, j0 = l; j0 < nv; r0 += 4, j0 += 128) {
            uint4 qs[4];
#pragma unroll
            for (int u = 0; u < 4; ++u) {
                const int j = min(j0 + 32 * u, nv - 1);  // past the end: re-read a valid row, result dropped
                qs[u] = reinterpret_cast<const uint4 *>(P.nbr)[j];
            }
#pragma unroll
            for (int u = 0; u < 4; ++u) {
                const int j = j0 + 32 * u;
                if (j >= nv) break;
                const uint32_t w[4] = {qs[u].x, qs[u].y, qs[u].z, qs[u].w};
                const float x = odf[j];
                const float tx = (x < thr) ? 0.0f : x;
                mn = (mn < tx) ? mn : tx;
                float lo = odf[w[0] & 0xffffu], hi = lo;
#pragma unroll
                for (int k = 1; k < 8; ++k) {
                    const float y = odf[(w[k >> 1] >> (16 * (k & 1))) & 0xffffu];
                    lo = fminf(lo, y);
                    hi = fmaxf(hi, y);
                }
                if (x >= thr && lo < x && !(hi > x)) {
                    pk |= 1u << (r0 + u);
                    pmax = fmaxf(pmax, x);
                }
            }
        }
        mn = min32(mn);
        mn = (0.0f > mn) ? 0.0f : mn;
        pmax = max32(pmax);
        if (pmax != REAL_MIN) m = pmax + (-mn);
    } else {
        for (int r0 = 0, j0 = l; j0 < nv; r0 += 4, j0 += 128) {
            uint4 qs[4];
#pragma unroll
            for (int u = 0; u < 4; ++u) {
                const int j = min(j0 + 32 * u, nv - 1);
                qs[u] = reinterpret_cast<const uint4 *>(P.nbr)[j];
            }
#pragma unroll
            for (int u = 0; u < 4; ++u) {
                const int j = j0 + 32 * u;
                if (j >= nv) break;
                const uint32_t w[4] = {qs[u].x, qs[u].y, qs[u].z, qs[u].w};
                float x = odf[j];
                x = (x < thr) ? 0.0f : x;
                mn = (mn < x) ? mn : x;
                bool smaller = false, larger = false;
#pragma unroll
                for (int k = 0; k < 8; ++k) {
                    float y = odf[(w[k >> 1] >> (16 * (k & 1))) & 0xffffu];
                    y = (y < thr) ? 0.0f : y;
                    smaller = smaller || (y < x);
                    larger = larger || (x < y);
                }
                if (smaller && !larger) pk |= 1u << (r0 + u);
            }
        }
        mn = min32(mn);
        mn = (0.0f > mn) ? 0.0f : mn;
        for (int r = 0, j = l; j < nv; ++r, j += 32)
            if ((pk >> r) & 1u) {
                const float xm = odf[j] + (-mn);
                m = (m > xm) ? m : xm;
            }
        m = max32(m);
    }
    const float comp = (float)((double)P.rel_peak * (double)m);
    int n = 0;
    for (int r = 0, j0 = 0; j0 < nv; ++r, j0 += 32) {
        const int j = j0 + l;
        const bool keep = (j < nv) && ((pk >> r) & 1u) && ((odf[j] - mn) >= comp);
        const uint32_t msk = half_ballot(keep);
        if (keep) cand[n + __popc(msk & ((1u << l) - 1u))] = (uint16_t)j;
        n += __popc(msk);
    }
    WAVE_SYNC();
    return sort_dedup_peaks(P.sep, odf, cand, sv, n);
}

// bb_peaks_all, or the edge form without an adjacency table (out of line:
// rare, or a sphere with a vertex of more than 8 neighbours).
__device__ __noinline__ int bb_peaks_slow(PeakParams P, const float *verts, float *odf, float thr, uint32_t *marks,
                                          uint16_t *cand) {
    if (P.nbr) return bb_peaks_all(P, odf, thr, cand, verts);
    for (int j = lane32(); j < P.nverts; j += 32)
        if (odf[j] < thr) odf[j] = 0.0f;
    WAVE_SYNC();
    return peak_directions(P, odf, marks, cand, verts);
}

// sort_dedup_peaks out of line, for the kernels of 4 waves per SIMD: inlined
// in the batched one it costs 20 spilled vector registers, in the exact one 30.
__device__ __noinline__ int bb_tail(SepParams P, const float *odf, uint16_t *cand, const float *verts, int n) {
    return sort_dedup_peaks(P, odf, cand, verts, n);
}

// bb_peaks_all's kept candidates (before the sort), from the vertices that
// can pass its last test: x >= thr and x - mn >= rel_peak (pmax - mn), with
// the ODF's maximum mx in place of the largest peak value pmax.  The two are
// the same whenever a kept peak has the value mx; the caller checks that.
// The 64 lanes of every wave test 64 vertices of each slot in `todo` in turn,
// so the neighbour rows q0, q1 of the wave's vertices (64 w + lane, and 64 (w +
// 8) + lane) are the same for all slots, and a lone slot has 8 waves at work.
// thr, mn, comp: of slot (lane % 16).  One bit per vertex goes to the slot's
// marks, 64 at a time.  On each slot's own lanes, 24 compactions and the
// candidates' neighbour rows from L2 took 12.4 k of a lone slot's 54 k cycles
// (6000 CSA seeds 72 ms that way, 62 ms this way).
__device__ __forceinline__ void bb_peak_bits(uint32_t todo, int nv, int ss, float *smem, int off_marks, const uint4 &q0,
                                             const uint4 &q1, float thr, float mn, float comp) {
    int lane = threadIdx.x & 63;
    asm volatile("" : "+v"(lane));
    const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    while (todo) {
        const int s = __builtin_ctz(todo);
        todo &= todo - 1u;
        const float *odf = smem + s * ss;
        uint64_t *marks = reinterpret_cast<uint64_t *>(smem + s * ss + off_marks);
        const float st = __uint_as_float(__builtin_amdgcn_readlane(__float_as_uint(thr), s));
        const float sm = __uint_as_float(__builtin_amdgcn_readlane(__float_as_uint(mn), s));
        const float sc = __uint_as_float(__builtin_amdgcn_readlane(__float_as_uint(comp), s));
        const float x0 = odf[min(64 * w + lane, nv - 1)], x1 = odf[min(64 * (w + BB_WAVES) + lane, nv - 1)];
        auto peak = [&](const uint4 &q, float x, bool valid) {
            bool p = valid && x >= st && (x - sm) >= sc;
            if (p) {
                const uint32_t v[4] = {q.x, q.y, q.z, q.w};
                float y[8];
#pragma unroll
                for (int k = 0; k < 8; ++k) y[k] = odf[(v[k >> 1] >> (16 * (k & 1))) & 0xffffu];
                float lo = y[0], hi = y[0];
#pragma unroll
                for (int k = 1; k < 8; ++k) {
                    lo = fminf(lo, y[k]);
                    hi = fmaxf(hi, y[k]);
                }
                p = lo < x && !(hi > x);
            }
            return __ballot(p);
        };
        if (64 * w < nv) {
            const uint64_t m = peak(q0, x0, 64 * w + lane < nv);
            if (lane == 0) marks[w] = m;
        }
        if (64 * (w + BB_WAVES) < nv) {
            const uint64_t m = peak(q1, x1, 64 * (w + BB_WAVES) + lane < nv);
            if (lane == 0) marks[w + BB_WAVES] = m;
        }
    }
}

// The vertices marked by bb_peak_bits, in order, to cand; -1 if none has the value mx.
__device__ __forceinline__ int bb_peak_list(int nv, const float *odf, float mx, const uint32_t *marks, uint16_t *cand) {
    const int l = lane32();
    uint32_t m = (32 * l < nv) ? marks[l] : 0u;
    const int c = __popc(m);
    int e = c;
#pragma unroll
    for (int d = 1; d < 32; d <<= 1) {
        const int o = __shfl_up(e, d, 32);
        if (l >= d) e += o;
    }
    const int n = shfl32(e, 31);
    int pos = e - c;
    bool top = false;
    while (m) {
        const int j = 32 * l + __builtin_ctz(m);
        m &= m - 1u;
        top = top || odf[j] == mx;
        cand[pos++] = (uint16_t)j;
    }
    WAVE_SYNC();
    return half_ballot(top) ? n : -1;
}

// Per-slot state of the batched kernel (registers of the slot's 32 lanes).
struct BbSlot {
    int s;          // seed (-1: none yet)
    int qk;         // queue cursor: queues qk.. of this XCD's order still to drain
    int di, ndir;   // direction of the seed being tracked, directions of the seed
    int off;        // streamline index of direction di
    int pass;       // 0 backward, 1 forward
    int i, att;     // step index of the pass, attempt of the step
    int nb;         // backward points (pass 1)
    bool done;      // queues drained
    float sx, sy, sz, fx, fy, fz, px, py, pz, dx, dy, dz;
};

// Start pass `pass` of direction st.di: the tracker's loop head
// (boot.cu:738-745): the point at index 0 of the pass is the seed.
__device__ __forceinline__ void bb_start_pass(const DevParams &P, BbSlot &st, float *__restrict__ sline) {
    const float sg = st.pass ? 1.0f : -1.0f;
    st.px = st.sx; st.py = st.sy; st.pz = st.sz;
    st.dx = sg * st.fx; st.dy = sg * st.fy; st.dz = sg * st.fz;
    st.i = 1;
    st.att = 0;
    float *o = sline + (size_t)st.off * (2 * (size_t)P.max_sline_len * 3) + (st.pass ? 3 * (size_t)(st.nb - 1) : 0);
    if (lane32() == 0) { o[0] = st.px; o[1] = st.py; o[2] = st.pz; }
}

// Next seed with at least one direction from the XCD-ordered queues, or
// st.done.  Streamlines of seeds without directions need no work; in a
// bounded chunk (P.slot_cap) neither do seeds whose slots end past the cap.
__device__ void bb_next_seed(const DevParams &P, const DevBufs &B, BbSlot &st, Philox &rng, int nseeds,
                             const float *__restrict__ seeds, int rng_chunk, const int *__restrict__ offsets,
                             const int *__restrict__ dirs, const int *__restrict__ order, int *__restrict__ work,
                             float *__restrict__ sline) {
    const int l = lane32();
    while (st.qk < QUEUES) {
        const QueueRange qr = queue_range(work, st.qk);
        const int lo = qr.lo, hi = qr.hi;
        int q = 0;
        if (l == 0 && lo < hi) q = atomicAdd(work + qr.counter, 1);
        q = shfl32(q, 0);
        if (lo + q >= hi) { ++st.qk; continue; }
        const int s = order[lo + q];
        const int nd = (P.slot_cap > 0 && offsets[s + 1] > P.slot_cap) ? 0 : offsets[s + 1] - offsets[s];
        if (nd == 0) continue;
        st.s = s;
        st.ndir = nd;
        st.di = 0;
        st.off = offsets[s];
        st.sx = seeds[3 * s]; st.sy = seeds[3 * s + 1]; st.sz = seeds[3 * s + 2];
        rng.init(((uint64_t)P.seed_hi << 32) | P.seed_lo, (uint64_t)32 * (uint64_t)(s % rng_chunk) + l + 1);
        const int vi = dirs[(size_t)s * P.nverts];
        st.fx = B.verts[3 * vi]; st.fy = B.verts[3 * vi + 1]; st.fz = B.verts[3 * vi + 2];
        st.pass = 0;
        st.nb = 0;
        return;
    }
    st.done = true;
}

// A pass ended with `ns` points: reverse the backward half in place, start
// the forward pass, or close the streamline and move to the next direction
// or seed (genStreamlinesMergeBoot_k, boot.cu:855-979).
__device__ void bb_end_pass(const DevParams &P, const DevBufs &B, BbSlot &st, Philox &rng, int ns, int nseeds,
                            const float *__restrict__ seeds, int rng_chunk, const int *__restrict__ offsets,
                            const int *__restrict__ dirs, const int *__restrict__ order, int *__restrict__ work,
                            int *__restrict__ sline_seed, int *__restrict__ sline_len, float *__restrict__ sline) {
    const int l = lane32();
    const size_t slot_f = 2 * (size_t)P.max_sline_len * 3;
    float *cur = sline + (size_t)st.off * slot_f;
    if (st.pass == 0) {
        st.nb = ns;
        MEM_SYNC();
        for (int j = l; j < ns / 2; j += 32) {
            float *a = cur + 3 * (size_t)j, *b = cur + 3 * (size_t)(ns - 1 - j);
            const float a0 = a[0], a1 = a[1], a2 = a[2];
            a[0] = b[0]; a[1] = b[1]; a[2] = b[2];
            b[0] = a0; b[1] = a1; b[2] = a2;
        }
        MEM_SYNC();
        st.pass = 1;
        bb_start_pass(P, st, sline);
        return;
    }
    if (l == 0) {
        sline_seed[st.off] = st.s;
        sline_len[st.off] = st.nb - 1 + ns;
    }
    ++st.di;
    ++st.off;
    if (st.di < st.ndir) {
        const int vi = dirs[(size_t)st.s * P.nverts + st.di];
        st.fx = B.verts[3 * vi]; st.fy = B.verts[3 * vi + 1]; st.fz = B.verts[3 * vi + 2];
        st.pass = 0;
        st.nb = 0;
        bb_start_pass(P, st, sline);
        return;
    }
    bb_next_seed(P, B, st, rng, nseeds, seeds, rng_chunk, offsets, dirs, order, work, sline);
    if (!st.done) bb_start_pass(P, st, sline);
}

// OCC: waves per SIMD the kernel is compiled for (2: 185 VGPRs and one
// workgroup per CU; 4: 128 VGPRs, 40 spilled, and two workgroups per CU, whose
// lockstep phases overlap).  boot_waves has the rule and its figures.
// LR: the low-rank form of the [H; R] product (P.rk16 > 0), a separate
// instantiation so that each form's kernel carries only its own registers.
template <int MODEL, int OCC, bool LR>
__global__ void __launch_bounds__(BB_THREADS, OCC)
    phase2_boot_batch_kernel(DevParams P, DevBufs B, const float *__restrict__ seeds, int nseeds, int rng_chunk,
                             const int *__restrict__ offsets, const int *__restrict__ dirs,
                             int *__restrict__ sline_seed, int *__restrict__ sline_len, float *__restrict__ sline,
                             const int *__restrict__ order, int *__restrict__ work) {
    constexpr int UN_ODF = (OCC == 4) ? 1 : 2;
    extern __shared__ float smem[];
    const int ss = bb_slot_stride(P.nv32, P.t32, P.hr32);
    const int slot = threadIdx.x >> 5;
    const int l = lane32();
    SlotLds SL;
    bind_slot<MODEL>(P, false, smem + slot * ss, SL);
    BootLds &S = SL.boot;
    // Slot n's arrays are the same offsets from smem + n * ss.
    const int off_h = 0;
    const int off_vox = (int)(S.vox - smem) - slot * ss, off_msk = (int)(S.msk - smem) - slot * ss,
              off_r = (int)(S.r - smem) - slot * ss;
    const int hr = P.hr, T = P.dimt, nv = P.nverts;
    const int MAXL = P.max_sline_len;
    float *wmax = smem + BB_SLOTS * ss;  // [BB_WAVES][16] partial ODF maxima of phase E, and minima
    float *wmin = wmax + BB_WAVES * 16;
    int *live = reinterpret_cast<int *>(wmin + BB_WAVES * 16);  // [16] slots with a signal this round
    // the lane's rows of the signal: its DWI channels (two to a register) and which of its channels are b0
    uint32_t dwi2[BB_ROWS / 2];
#pragma unroll
    for (int r = 0; r < BB_ROWS; ++r) {
        const uint32_t d = (l + 32 * r < hr) ? (uint32_t)B.dwi_idx[l + 32 * r] : 0u;
        dwi2[r >> 1] = (r & 1) ? dwi2[r >> 1] | (d << 16) : d;
    }
    uint32_t b0_rows = 0u;
    for (int r = 0, j = l; r < 32 && j < T; ++r, j += 32) b0_rows |= (B.b0[j] ? 1u : 0u) << r;
    // floor(2^32 / hr), for hr 1 the largest 32-bit number: the high product of a draw is its quotient or one less
    const uint32_t hr_magic = (hr > 1) ? (uint32_t)(0x100000000ull / (uint32_t)hr) : 0xffffffffu;
    BbSlot st;
    st.s = -1; st.qk = 0; st.done = false; st.nb = 0; st.pass = 0;
    Philox rng;
    // fewer seeds than slots: spread over the workgroups, the rest of their slots idle
    if ((unsigned)slot * gridDim.x >= (unsigned)nseeds) st.done = true;
    else bb_next_seed(P, B, st, rng, nseeds, seeds, rng_chunk, offsets, dirs, order, work, sline);
    if (!st.done) bb_start_pass(P, st, sline);
    unsigned long long attempts = 0, rounds = 0;  // slot attempts and rounds of this workgroup
    for (;;) {
        // Formed anew each round: kept around it, the row tests of the
        // unrolled loops below take 90 scalar and their addresses as many
        // vector registers, and the 128 of 4 waves per SIMD spill.
        int l = lane32(), hr = P.hr, hr16 = P.hr16;
        asm volatile("" : "+v"(l), "+s"(hr), "+s"(hr16));
        // ---- phase A: gather the signal at the point -----------------------
        // The masked signal, and the normalisation by the b0 mean, which the
        // resampling does not touch.
        const bool active = !st.done;
        bool data = false;
        float inv = 0.0f;
        if (active) {
            data = bb_gather(P, B.data, st.px, st.py, st.pz, S.vox);
            WAVE_SYNC();
            if (data) {
                float part = 0.0f;
                for (int r = 0, j = l; j < T; ++r, j += 32) {
                    if ((r < 32) ? ((b0_rows >> r) & 1u) : (uint32_t)(B.b0[j] != 0)) {
                        float v = S.vox[j];
                        v = (P.min_signal > v) ? P.min_signal : v;
                        part = part + v;
                    }
                }
#pragma unroll
                for (int r = 0; r < BB_ROWS; ++r)
                    if (32 * r < hr16) {
                        const int m = l + 32 * r;
                        const float v = S.vox[(dwi2[r >> 1] >> (16 * (r & 1))) & 0xffffu];
                        if (m < hr16) S.msk[m] = (m < hr) ? v : 0.0f;
                    }
                inv = (float)(T - hr) / tree_sum32(part);
            }
        }
        if (l == 0) live[slot] = data;
        const int nact = __syncthreads_count(active) / 32;  // active slots (32 lanes each)
        if (nact == 0) break;
        attempts += (unsigned long long)nact;
        ++rounds;
        // ---- phase B: H.d and R.d for the 16 slots --------------------------
        if (LR) {
            // low-rank form: z = U^T d into the R.d region, then H.d = U z;
            // R.d follows in phase C
            bb_gemm<1, 5>(B.ut_mat, hr16, hr16, P.rk16 / 16, smem + off_msk, smem + off_msk, hr16, smem + off_r,
                          smem + off_r, 1 << 30, P.rk16, ss);
            __syncthreads();
            bb_gemm<(320 / 16 + BB_WAVES - 1) / BB_WAVES, 2>(B.u_mat, P.rk16, P.rk16, hr16 / 16, smem + off_r,
                                                             smem + off_r, 1 << 30, smem + off_h, smem + off_h,
                                                             1 << 30, hr16, ss);
        } else {
            bb_gemm<(2 * 320 / 16 + BB_WAVES - 1) / BB_WAVES, UN_ODF>(B.hr_mat, hr16, hr16, 2 * hr16 / 16,
                                                                      smem + off_msk, smem + off_msk, hr16,
                                                                      smem + off_h, smem + off_r, hr16, 2 * hr16, ss);
        }
        __syncthreads();
        // ---- phase C: residual bootstrap, normalisation, model transform -----
        if (active && data) {
            if (LR) {
                // R.d = v - mean(v), v = (d - H.d) / sqrt(1 - H_ii)
                float v[BB_ROWS], part = 0.0f;
#pragma unroll
                for (int r = 0; r < BB_ROWS; ++r) {
                    const int j = l + 32 * r;
                    v[r] = 0.0f;
                    if (j < hr) {
                        v[r] = (S.msk[j] - S.h[j]) * B.invlev[j];
                        part = part + v[r];
                    }
                }
                const float mean = tree_sum32(part) / (float)hr;
#pragma unroll
                for (int r = 0; r < BB_ROWS; ++r)
                    if (l + 32 * r < hr) S.r[l + 32 * r] = v[r] - mean;
                WAVE_SYNC();
            }
            float h[BB_ROWS];
#pragma unroll
            for (int r = 0; r < BB_ROWS; ++r) {
                const int j = l + 32 * r;
                h[r] = 0.0f;
                if (j < hr) {
                    // draw % hr: the high product is the quotient or one less
                    const uint32_t x = rng.next();
                    const uint32_t rem = x - __umulhi(x, hr_magic) * (uint32_t)hr;
                    h[r] = S.h[j] + S.r[min(rem, rem - (uint32_t)hr)];
                }
            }
            WAVE_SYNC();
#pragma unroll
            for (int r = 0; r < BB_ROWS; ++r) {
                const int m = l + 32 * r;
                if (m < hr16) {
                    const float c = (P.min_signal > h[r]) ? P.min_signal : h[r];
                    const float v = (m < hr) ? c * inv : 0.0f;
                    S.msk[m] = v;
                    S.h[m] = (m < hr) ? bb_xf<(MODEL == CUSLINES_OPDT) ? 1 : 2>(v) : 0.0f;
                }
            }
        }
        __syncthreads();
        // ---- phase D: model coefficients (CSA: dq.xf; OPDT: dq.xf - db.msk) --
        bb_gemm<1, 5, MODEL == CUSLINES_CSA>(B.fit_mat, 2 * hr16, (MODEL == CUSLINES_OPDT) ? 2 * hr16 : hr16,
                                             P.dn16 / 16, smem + off_h, smem + off_msk, hr16, smem + off_vox,
                                             smem + off_vox, 1 << 30, P.dn16, ss);
        __syncthreads();
        // ---- phase E: the ODF on the sphere ---------------------------------
        bb_gemm<(768 / 16 + BB_WAVES - 1) / BB_WAVES, UN_ODF>(B.odf_mat, P.dn16, P.dn16, P.nv16 / 16, smem + off_vox,
                                                              smem + off_vox, 1 << 30, smem + off_h, smem + off_h,
                                                              1 << 30, nv, ss, wmax, wmin);
        uint4 nb0 = uint4{0u, 0u, 0u, 0u}, nb1 = nb0;
        if (B.nbr) {
            int t = threadIdx.x;
            asm volatile("" : "+v"(t));
            nb0 = reinterpret_cast<const uint4 *>(B.nbr)[min(t, nv - 1)];
            nb1 = reinterpret_cast<const uint4 *>(B.nbr)[min(t + BB_THREADS, nv - 1)];
        }
        __syncthreads();
        // ---- phase F: peaks, closest peak, the step --------------------------
        uint32_t fast = 0u;  // slots whose peaks bb_peak_bits marks
        if (B.nbr) {
            // lane: slot lane % 16
            const int k = threadIdx.x & 63;
            float mx = fmaxf(wmax[k], wmax[k + 64]);
            float mn = __builtin_elementwise_minimum(wmin[k], wmin[k + 64]);
            mx = fmaxf(mx, __shfl_xor(mx, 16));
            mx = fmaxf(mx, __shfl_xor(mx, 32));
            mn = __builtin_elementwise_minimum(mn, __shfl_xor(mn, 16));
            mn = __builtin_elementwise_minimum(mn, __shfl_xor(mn, 32));
            const float thr = (float)(PMF_THRESHOLD_P * (double)mx);
            // a value below thr reads as 0 (and thr > 0), a NaN is left to bb_peaks_all
            fast = (uint32_t)__ballot(live[k & 15] && thr > 0.0f && mn == mn) & 0xffffu;
            mn = (mn < thr) ? 0.0f : mn;
            const float comp = (float)((double)P.rel_peak * (double)(mx + (-mn)));
            bb_peak_bits(fast, nv, ss, smem, (int)((float *)S.marks - smem) - slot * ss, nb0, nb1, thr, mn, comp);
            __syncthreads();
        }
        if (active) {
            int ns = -1;  // >= 0: the pass ends with ns points
            if (!data) {
                // the signal is zero at this point: every remaining attempt
                // fails the same way without a random draw
                ns = st.i;
            } else {
                // the ODF's maximum from the 8 waves' partial maxima of phase E
                float mx = (l < BB_WAVES) ? wmax[l * 16 + slot] : REAL_MIN;
                mx = max32(mx);
                const float thr = (float)(PMF_THRESHOLD_P * (double)mx);
                int npk = ((fast >> slot) & 1u) ? bb_peak_list(nv, S.h, mx, S.marks, S.cand) : -1;
                if (npk >= 0)
                    npk = (OCC == 4) ? bb_tail(sep_params(P), S.h, S.cand, B.verts, npk)
                                     : sort_dedup_peaks(sep_params(P), S.h, S.cand, B.verts, npk);
                else
                    npk = bb_peaks_slow(peak_params(P, B), B.verts, S.h, thr, S.marks, S.cand);
                float nx = 0.0f, ny = 0.0f, nz = 0.0f;
                const bool ok = npk > 0 && closest_peak(P, B.verts, st.dx, st.dy, st.dz, npk, S.cand, &nx, &ny, &nz);
                WAVE_SYNC();
                if (!ok) {
                    if (++st.att == BB_MAX_ATTEMPTS) ns = st.i;
                } else {
                    st.att = 0;
                    st.dx = nx; st.dy = ny; st.dz = nz;
                    st.px = (float)__builtin_fma((double)(nx / 1.0f), P.step_d, (double)st.px);
                    st.py = (float)__builtin_fma((double)(ny / 1.0f), P.step_d, (double)st.py);
                    st.pz = (float)__builtin_fma((double)(nz / 1.0f), P.step_d, (double)st.pz);
                    if (l == 0) {
                        float *o = sline + (size_t)st.off * (2 * (size_t)MAXL * 3) +
                                   (st.pass ? 3 * (size_t)(st.nb - 1) : 0) + 3 * (size_t)st.i;
                        o[0] = st.px; o[1] = st.py; o[2] = st.pz;
                    }
                    const int tissue = check_point(P, B.stop, st.px, st.py, st.pz);
                    if (tissue == CUSLINES_ENDPOINT || tissue == CUSLINES_INVALIDPOINT ||
                        tissue == CUSLINES_OUTSIDEIMAGE)
                        ns = st.i;
                    else if (++st.i == MAXL)
                        ns = MAXL;
                }
            }
            if (ns >= 0)
                bb_end_pass(P, B, st, rng, ns, nseeds, seeds, rng_chunk, offsets, dirs, order, work, sline_seed,
                            sline_len, sline);
        }
        // no barrier here: phase A writes only this slot's region A, which
        // phase E of every wave has finished reading (barrier above)
    }
    if (threadIdx.x == 0 && B.stats) {
        atomicAdd(B.stats, attempts);
        atomicAdd(B.stats + 1, rounds);
    }
}

__global__ void zero_ints(int *p, int n) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) p[i] = 0;
}

template <typename TO>
__global__ void zero_scalar(TO *p) {
    *p = 0;
}

// Processing order of the persistent queue: seeds bucketed by class and by the
// Morton code of their 2^brick_log2-voxel brick (counting sort).
__device__ __forceinline__ uint32_t spread3(uint32_t v) {  // bits 0..9 to every third bit
    v &= 0x3ffu;
    v = (v | (v << 16)) & 0x030000ffu;
    v = (v | (v << 8)) & 0x0300f00fu;
    v = (v | (v << 4)) & 0x030c30c3u;
    v = (v | (v << 2)) & 0x09249249u;
    return v;
}

// Class of a seed with n directions: the more, the earlier.  Without offsets
// every seed is in the first class: the order is then the spatial one alone.
__device__ __forceinline__ int seed_class(int n) {
    if (n >= 8) return 0;
    return (n >= 6) ? 1 : (n >= 1) ? 7 - n : SEED_CLASSES - 1;
}

__global__ void seed_keys(DevParams P, const float *__restrict__ seeds, const int *__restrict__ offsets, int n,
                          int brick_log2, int nbrick, int *__restrict__ key, int *__restrict__ count) {
    const int s = blockIdx.x * blockDim.x + threadIdx.x;
    if (s >= n) return;
    uint32_t c[3];
    const int dims[3] = {P.dimx, P.dimy, P.dimz};
    for (int a = 0; a < 3; ++a) {
        const float f = floorf(seeds[3 * s + a]);
        const int i = (f != f || f < 0.0f) ? 0 : (f > (float)(dims[a] - 1) ? dims[a] - 1 : (int)f);
        c[a] = (uint32_t)i >> brick_log2;
    }
    const int k = (offsets ? seed_class(offsets[s + 1] - offsets[s]) : 0) * nbrick +
                  (int)(spread3(c[0]) | (spread3(c[1]) << 1) | (spread3(c[2]) << 2));
    key[s] = k;
    atomicAdd(count + k, 1);
}

// Counters at zero and the classes' starts in the seed order.
__global__ void queue_init(int *__restrict__ work, const int *__restrict__ start, int nbrick) {
    const int i = threadIdx.x;
    if (i < WORK_INTS) work[i] = (i < QUEUES) ? 0 : start[(i - QUEUES) * nbrick];
}

__global__ void seed_scatter(const int *__restrict__ key, int n, const int *__restrict__ start, int *__restrict__ cursor,
                             int *__restrict__ order) {
    const int s = blockIdx.x * blockDim.x + threadIdx.x;
    if (s >= n) return;
    const int k = key[s];
    order[start[k] + atomicAdd(cursor + k, 1)] = s;
}

// -------------------------------------------------------------------------
// Training of the proposal network (no counterpart in the reference).
//
// One kernel for the forward and the backward pass and one that adds up its
// partial gradients.  A workgroup of 8 waves takes tiles of 16 pairs, keeps
// the three layers' weights (rounded to bf16) as MFMA operands and all weight
// gradients as MFMA accumulators in registers over its tiles, and writes the
// gradients once; activations stay in LDS.  The products run on
// v_mfma_f32_16x16x4_f32 (fp32 operands and sums); wave w owns hidden neurons
// 16 w .. 16 w + 15 of both layers.
// What bounds it at the default 4096 pairs is latency: reading the weights
// (10 us), seven short phases between barriers a tile (5-8 us, three tiles a
// workgroup), writing and re-reading the partials (11 MB).  Loss and gradient of
// 4096 pairs 361 -> 58 us with the copy to the host; the layer by layer,
// element by element kernels before took 13 launches and re-read the weights for
// every pair.  With room in the workspace for 256 partials, one tile each, it
// is 49 us.  60 000 pairs: 94 us, 15 tiles a workgroup at 5 us, where the matrix
// products alone are 3.6 us.
// -------------------------------------------------------------------------
__device__ __forceinline__ float bf16_round(float x) {  // to the nearest bf16, ties to even
    uint32_t b = __float_as_uint(x);
    if ((b & 0x7f800000u) == 0x7f800000u) return x;
    b += 0x7fffu + ((b >> 16) & 1u);
    return __uint_as_float(b & 0xffff0000u);
}

constexpr int MLP_TILE = 16, MLP_GROUPS = 256, MLP_THREADS = 512;
// A workgroup's partial gradients as its lanes hold them: 13 tiles (3 of the
// first layer, 8 of the second, 2 of the third) of 4 floats per thread, then the
// biases of the three layers and the loss.
constexpr int MLP_PART_B = 13 * 4 * MLP_THREADS, MLP_PART_LOSS = MLP_PART_B + 2 * MLP_H + MLP_OUT;
constexpr int MLP_PART = (MLP_PART_LOSS + 1 + 31) & ~31;
static_assert(MLP_H == 16 * MLP_THREADS / 64 && MLP_IN % 4 == 0 && MLP_OUT <= 32, "tiles of the training kernel");
// LDS row strides, 20 mod 64 floats: the rows of 16 pairs start in 16
// different groups of four banks (16-byte reads along a row), and 4 rows
// of 16 consecutive floats overlap little (reads across the rows).
constexpr int MLP_LDX = 84, MLP_LDH = 148, MLP_LDO = 36;

// The parameter that float `col` (before the loss) of a partial belongs to, -1
// for a tile's rows and columns past the layer's.
__device__ __forceinline__ int mlp_part_param(int col) {
    if (col >= MLP_PART_B) {
        const int j = col - MLP_PART_B;
        return (j < MLP_H) ? MLP_B1 + j : (j < 2 * MLP_H) ? MLP_B2 + j - MLP_H : MLP_B3 + j - 2 * MLP_H;
    }
    // tile k, thread (wave w, lane (i, q)), float r: row 4 q + r and column i of the tile
    const int k = col / (4 * MLP_THREADS), th = (col >> 2) & (MLP_THREADS - 1);
    const int w = th >> 6, i = th & 15, row = 4 * ((th >> 4) & 3) + (col & 3);
    if (k < 3) return (16 * k + i < MLP_IN) ? MLP_W1 + (16 * w + row) * MLP_IN + 16 * k + i : -1;
    if (k < 11) return MLP_W2 + (16 * w + row) * MLP_H + 16 * (k - 3) + i;
    return (16 * (k - 11) + row < MLP_OUT) ? MLP_W3 + (16 * (k - 11) + row) * MLP_H + 16 * w + i : -1;
}

struct __attribute__((packed, aligned(4))) FloatQuad {  // 16 bytes at any float's address
    float v[4];
};

__device__ __forceinline__ float row_sum16(float v) {  // sum over the 16 lanes of a DPP row
    v += dpp0<DPP_ROW_ROR + 8>(v);
    v += dpp0<DPP_ROW_ROR + 4>(v);
    v += dpp0<DPP_ROW_ROR + 2>(v);
    v += dpp0<DPP_ROW_ROR + 1>(v);
    return v;
}

__global__ void __launch_bounds__(MLP_THREADS, 2)
    mlp_train_kernel(const float *__restrict__ prm, const float *__restrict__ pairs, int n, float *__restrict__ part,
                     float *__restrict__ grad, float *__restrict__ mean_loss) {
    __shared__ __align__(16) float sx[2][MLP_TILE * MLP_LDX];  // pairs: 40 inputs, 24 targets
    __shared__ __align__(16) float sh1[MLP_TILE * MLP_LDH], sh2[MLP_TILE * MLP_LDH];
    __shared__ __align__(16) float sd1[MLP_TILE * MLP_LDH], sd2[MLP_TILE * MLP_LDH];  // gradients at the hidden layers
    __shared__ float so[4][32 * MLP_TILE];       // output sums over a quarter of the second hidden layer
    __shared__ float sdo[MLP_TILE * MLP_LDO];    // gradient at the outputs, rows 24..31 zero
    __shared__ float sred[MLP_THREADS / 16];
    typedef float v4 __attribute__((ext_vector_type(4)));
    const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6, i = lane & 15, q = lane >> 4;
    constexpr int H = MLP_H, K1 = MLP_IN / 4, NO = MLP_OUT;
    const int ntile = (n + MLP_TILE - 1) / MLP_TILE;
    auto fetch = [&](int t, float (&x)[2]) {
#pragma unroll
        for (int u = 0; u < 2; ++u) {
            const int e = tid + u * MLP_THREADS;
            const long long smp = (long long)t * MLP_TILE + (e >> 6);
            x[u] = (smp < n) ? pairs[smp * CUSLINES_PAIR_FLOATS + (e & 63)] : 0.0f;
        }
    };
    float xr[2];
    fetch(blockIdx.x, xr);
    // Operands: lane (i, q) holds row i; of a 16-wide chunk c of the sum, step
    // s takes index 16 c + 4 q + s, and with fewer terms index 4 s + q.
    float w1[K1], w2[32], w2t[32], w3[8], w3t[NO / 4];
    const int row = 16 * w + i;
#pragma unroll
    for (int s = 0; s < K1; ++s) w1[s] = bf16_round(prm[MLP_W1 + row * MLP_IN + 4 * s + q]);
#pragma unroll
    for (int c = 0; c < 8; ++c) {
        const FloatQuad f = *reinterpret_cast<const FloatQuad *>(prm + MLP_W2 + row * H + 16 * c + 4 * q);
#pragma unroll
        for (int s = 0; s < 4; ++s) {
            w2[4 * c + s] = bf16_round(f.v[s]);
            w2t[4 * c + s] = bf16_round(prm[MLP_W2 + (16 * c + 4 * q + s) * H + row]);
        }
    }
    const int ot = w & 1, kq = w >> 1;  // third layer: rows 16 ot.., columns 32 kq..
    uint32_t in3 = (16 * ot + i < NO) ? ~0u : 0u;
    asm volatile("" : "+v"(in3));  // a mask: as a branch, each of the loads waits for the one before
#pragma unroll
    for (int c = 0; c < 2; ++c) {
        const int j = 16 * ot + i;
        const FloatQuad f =
            *reinterpret_cast<const FloatQuad *>(prm + MLP_W3 + min(j, NO - 1) * H + 32 * kq + 16 * c + 4 * q);
#pragma unroll
        for (int s = 0; s < 4; ++s) w3[4 * c + s] = __uint_as_float(__float_as_uint(bf16_round(f.v[s])) & in3);
    }
#pragma unroll
    for (int s = 0; s < NO / 4; ++s) w3t[s] = bf16_round(prm[MLP_W3 + (4 * s + q) * H + row]);
    v4 b1, b2;
#pragma unroll
    for (int r = 0; r < 4; ++r) {
        b1[r] = bf16_round(prm[MLP_B1 + 16 * w + 4 * q + r]);
        b2[r] = bf16_round(prm[MLP_B2 + 16 * w + 4 * q + r]);
    }
    const int oj = tid >> 4;  // outputs: thread (output, pair i)
    const float b3 = bf16_round(prm[MLP_B3 + min(oj, NO - 1)]);
    const float scale = 2.0f / ((float)NO * (float)n);

    const v4 zero = {0.0f, 0.0f, 0.0f, 0.0f};
    v4 g1[3] = {zero, zero, zero}, g2[8], g3[2] = {zero, zero}, gb1 = zero, gb2 = zero;
#pragma unroll
    for (int k = 0; k < 8; ++k) g2[k] = zero;
    float gb3 = 0.0f, loss = 0.0f;

    int buf = 0;
    for (int t = blockIdx.x; t < ntile; t += gridDim.x, buf ^= 1) {
        float *X = sx[buf];
#pragma unroll
        for (int u = 0; u < 2; ++u) {
            const int e = tid + u * MLP_THREADS;
            X[(e >> 6) * MLP_LDX + (e & 63)] = xr[u];
        }
        if (t + (int)gridDim.x < ntile) fetch(t + gridDim.x, xr);
        const bool valid = (long long)t * MLP_TILE + i < n;  // pairs past the last one take no part
        __syncthreads();
        // first hidden layer
        v4 h1 = b1;
#pragma unroll
        for (int s = 0; s < K1; ++s)
            h1 = __builtin_amdgcn_mfma_f32_16x16x4f32(w1[s], X[i * MLP_LDX + 4 * s + q], h1, 0, 0, 0);
#pragma unroll
        for (int r = 0; r < 4; ++r) h1[r] = (valid && h1[r] > 0.0f) ? h1[r] : 0.0f;
        *reinterpret_cast<v4 *>(sh1 + i * MLP_LDH + 16 * w + 4 * q) = h1;
        __syncthreads();
        // second hidden layer
        v4 h2 = b2;
#pragma unroll
        for (int c = 0; c < 8; ++c) {
            const v4 x = *reinterpret_cast<const v4 *>(sh1 + i * MLP_LDH + 16 * c + 4 * q);
#pragma unroll
            for (int s = 0; s < 4; ++s) h2 = __builtin_amdgcn_mfma_f32_16x16x4f32(w2[4 * c + s], x[s], h2, 0, 0, 0);
        }
#pragma unroll
        for (int r = 0; r < 4; ++r) h2[r] = (valid && h2[r] > 0.0f) ? h2[r] : 0.0f;
        *reinterpret_cast<v4 *>(sh2 + i * MLP_LDH + 16 * w + 4 * q) = h2;
        __syncthreads();
        // outputs, a quarter of the sum per pair of waves
        {
            v4 o = zero;
#pragma unroll
            for (int c = 0; c < 2; ++c) {
                const v4 x = *reinterpret_cast<const v4 *>(sh2 + i * MLP_LDH + 32 * kq + 16 * c + 4 * q);
#pragma unroll
                for (int s = 0; s < 4; ++s) o = __builtin_amdgcn_mfma_f32_16x16x4f32(w3[4 * c + s], x[s], o, 0, 0, 0);
            }
#pragma unroll
            for (int r = 0; r < 4; ++r) so[kq][(16 * ot + 4 * q + r) * MLP_TILE + i] = o[r];
        }
        __syncthreads();
        // the error, the loss and the gradient at the outputs
        {
            float d = 0.0f;
            if (oj < NO && valid) {
                const float o = b3 + ((so[0][tid] + so[1][tid]) + (so[2][tid] + so[3][tid]));
                const float e = o - X[i * MLP_LDX + MLP_IN + oj];
                loss = __builtin_fmaf(e, e, loss);
                d = e * scale;
            }
            gb3 += d;
            sdo[i * MLP_LDO + oj] = d;
        }
        __syncthreads();
        // gradient at the second hidden layer
        v4 d2 = zero;
#pragma unroll
        for (int s = 0; s < NO / 4; ++s)
            d2 = __builtin_amdgcn_mfma_f32_16x16x4f32(w3t[s], sdo[i * MLP_LDO + 4 * s + q], d2, 0, 0, 0);
#pragma unroll
        for (int r = 0; r < 4; ++r) d2[r] = (h2[r] > 0.0f) ? d2[r] : 0.0f;
        gb2 += d2;
        *reinterpret_cast<v4 *>(sd2 + i * MLP_LDH + 16 * w + 4 * q) = d2;
        // third layer's weights: outputs x hidden neurons 16 w.., summed over the pairs
#pragma unroll
        for (int s = 0; s < 4; ++s) {
            const float x = sh2[(4 * s + q) * MLP_LDH + 16 * w + i];
#pragma unroll
            for (int k = 0; k < 2; ++k)
                g3[k] = __builtin_amdgcn_mfma_f32_16x16x4f32(sdo[(4 * s + q) * MLP_LDO + 16 * k + i], x, g3[k], 0, 0, 0);
        }
        __syncthreads();
        // gradient at the first hidden layer
        v4 d1 = zero;
#pragma unroll
        for (int c = 0; c < 8; ++c) {
            const v4 x = *reinterpret_cast<const v4 *>(sd2 + i * MLP_LDH + 16 * c + 4 * q);
#pragma unroll
            for (int s = 0; s < 4; ++s) d1 = __builtin_amdgcn_mfma_f32_16x16x4f32(w2t[4 * c + s], x[s], d1, 0, 0, 0);
        }
#pragma unroll
        for (int r = 0; r < 4; ++r) d1[r] = (h1[r] > 0.0f) ? d1[r] : 0.0f;
        gb1 += d1;
        *reinterpret_cast<v4 *>(sd1 + i * MLP_LDH + 16 * w + 4 * q) = d1;
        // second layer's weights
#pragma unroll
        for (int s = 0; s < 4; ++s) {
            const float d = sd2[(4 * s + q) * MLP_LDH + 16 * w + i];
#pragma unroll
            for (int k = 0; k < 8; ++k)
                g2[k] = __builtin_amdgcn_mfma_f32_16x16x4f32(d, sh1[(4 * s + q) * MLP_LDH + 16 * k + i], g2[k], 0, 0, 0);
        }
        WAVE_SYNC();  // sd1's columns 16 w.. are this wave's own
        // first layer's weights; columns 40.. are the targets' and dropped
#pragma unroll
        for (int s = 0; s < 4; ++s) {
            const float d = sd1[(4 * s + q) * MLP_LDH + 16 * w + i];
#pragma unroll
            for (int k = 0; k < 3; ++k)
                g1[k] = __builtin_amdgcn_mfma_f32_16x16x4f32(d, X[(4 * s + q) * MLP_LDX + 16 * k + i], g1[k], 0, 0, 0);
        }
        // the next tile's pairs go to the other buffer; sh1 is written after its barrier
    }

    // the lanes' tiles as they are; a lone workgroup's, and its sums, to their places
    const bool lone = gridDim.x == 1;
    float *P = part + (size_t)blockIdx.x * MLP_PART;
    auto put = [&](int k, const v4 &g) {
        if (!lone) {
            reinterpret_cast<FloatQuad *>(P)[k * MLP_THREADS + tid] = FloatQuad{{g[0], g[1], g[2], g[3]}};
        } else {
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const int at = mlp_part_param(4 * (k * MLP_THREADS + tid) + r);
                if (at >= 0) grad[at] = g[r];
            }
        }
    };
    auto put1 = [&](int at, float v) {
        if (lone) grad[mlp_part_param(at)] = v;
        else P[at] = v;
    };
#pragma unroll
    for (int k = 0; k < 3; ++k) put(k, g1[k]);
#pragma unroll
    for (int k = 0; k < 8; ++k) put(3 + k, g2[k]);
#pragma unroll
    for (int k = 0; k < 2; ++k) put(11 + k, g3[k]);
#pragma unroll
    for (int r = 0; r < 4; ++r) {
        const int j = 16 * w + 4 * q + r;
        const float s1 = row_sum16(gb1[r]), s2 = row_sum16(gb2[r]);
        if (i == 0) {
            put1(MLP_PART_B + j, s1);
            put1(MLP_PART_B + H + j, s2);
        }
    }
    gb3 = row_sum16(gb3);
    loss = row_sum16(loss);
    if (i == 0) {
        if (oj < NO) put1(MLP_PART_B + 2 * H + oj, gb3);
        sred[oj] = loss;
    }
    __syncthreads();
    if (tid == 0) {
        float l = 0.0f;
        for (int k = 0; k < MLP_THREADS / 16; ++k) l += sred[k];
        if (lone) mean_loss[0] = l / (float)NO / (float)n;
        else P[MLP_PART_LOSS] = l;
    }
}

// Sums of the workgroups' partials in a fixed order: thread (column c, quarter
// g) of a block adds its quarter of the workgroups.
constexpr int MLP_SUM_COLS = 64;
__global__ void __launch_bounds__(256)
    mlp_sum_kernel(const float *__restrict__ part, int groups, int n, float *__restrict__ grad, float *__restrict__ loss) {
    __shared__ float sp[4][MLP_SUM_COLS];
    const int c = threadIdx.x & (MLP_SUM_COLS - 1), g = threadIdx.x / MLP_SUM_COLS;
    const int col = blockIdx.x * MLP_SUM_COLS + c;
    const int per = (groups + 3) / 4, g0 = min(groups, g * per), g1 = min(groups, g0 + per);
    float acc = 0.0f;
    if (col <= MLP_PART_LOSS) {
        const float *p = part + col;
#pragma unroll 16
        for (int k = g0; k < g1; ++k) acc += p[(size_t)k * MLP_PART];
    }
    sp[g][c] = acc;
    __syncthreads();
    if (g != 0 || col > MLP_PART_LOSS) return;
    const float v = (sp[0][c] + sp[1][c]) + (sp[2][c] + sp[3][c]);
    if (col == MLP_PART_LOSS) {
        loss[0] = v / (float)MLP_OUT / (float)n;
    } else {
        const int at = mlp_part_param(col);
        if (at >= 0) grad[at] = v;
    }
}

// Adam (Kingma and Ba, 2015); c1 = 1 - beta1^step, c2 = 1 - beta2^step.
__global__ void adam_kernel(float *__restrict__ p, const float *__restrict__ g, float *__restrict__ m,
                            float *__restrict__ v, int n, float lr, float b1, float b2, float eps, float c1, float c2) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const float gi = g[i];
    const float mi = b1 * m[i] + (1.0f - b1) * gi;
    const float vi = b2 * v[i] + (1.0f - b2) * gi * gi;
    m[i] = mi;
    v[i] = vi;
    p[i] -= lr * (mi / c1) / (__builtin_sqrtf(vi / c2) + eps);
}

// Propagators of arc length FEAT_STEPS probe steps for the 24 disc vertices
// (the curves along which the learned proposal's inputs are tapped).
// Per disc vertex, the propagator of `steps` probe steps (FEAT_STEPS: the
// learned proposal's features; 1: the vertex phase's probes, followed at
// VPROP_K by the vertices' curvatures (k1, k2)).
__global__ void feature_propagators(DevParams P, int steps, float *__restrict__ out) {
    const int l = threadIdx.x;
    if (l < DISC_VERT_CNT) {
        const float k1 = (float)((double)c_disc_vert[2 * l] * (double)P.max_curv);
        const float k2 = (float)((double)c_disc_vert[2 * l + 1] * (double)P.max_curv);
        float p[9];
        prepare_propagator(k1, k2, (steps == 1) ? P.probe_step : (float)steps * P.probe_step, p);
        for (int i = 0; i < 9; ++i) out[9 * l + i] = p[i];
        if (steps == 1) {  // and the vertex's curvature, the disc scaled by MAX_CURVATURE
            out[VPROP_K + 2 * l] = k1;
            out[VPROP_K + 2 * l + 1] = k2;
        }
    }
}

// PTT corner blocks: for texel cell (cx,cy,cz) in [-1, D-1]^3 and direction
// rank r (vertex rank_vertex[r]), the 8 texels one linear-filtered tap of
// that vertex's tile reads (x fastest), with the tiling's bleed into
// neighbouring tiles and the clamp at the texture edge.  Block index =
// cell * nverts + r.
__global__ void build_corner_blocks(DevParams P, const float *__restrict__ odfv,
                                    const uint16_t *__restrict__ rank_vertex, float *__restrict__ blocks,
                                    long long ncells) {
    const long long idx = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    if (idx >= ncells) return;
    const int DX = P.dimx, DY = P.dimy, DZ = P.dimz;
    long long t = idx;
    const int v = (int)rank_vertex[t % P.nverts]; t /= P.nverts;
    const int cz = (int)(t % (DZ + 1)) - 1; t /= (DZ + 1);
    const int cy = (int)(t % (DY + 1)) - 1; t /= (DY + 1);
    const int cx = (int)(t % (DX + 1)) - 1;
    const int tx = v & (P.nx - 1), ty = (v >> P.log2x) & (P.ny - 1), tz = v >> (P.log2x + P.log2y);
    int txa, txb, lxa, lxb, tya, tyb, lya, lyb, tza, tzb, lza, lzb;
    axis_split(tx * DX + cx, DX, P.nx, tx, &txa, &lxa);
    axis_split(tx * DX + cx + 1, DX, P.nx, tx, &txb, &lxb);
    axis_split(ty * DY + cy, DY, P.ny, ty, &tya, &lya);
    axis_split(ty * DY + cy + 1, DY, P.ny, ty, &tyb, &lyb);
    axis_split(tz * DZ + cz, DZ, P.nz, tz, &tza, &lza);
    axis_split(tz * DZ + cz + 1, DZ, P.nz, tz, &tzb, &lzb);
    const int NV = P.nverts, nx = P.nx, ny = P.ny;
    auto fetch = [&](int ti, int li, int tj, int lj, int tk, int lk) -> float {
        const int w = ti + nx * (tj + ny * tk);
        if (w >= NV) return 0.0f;
        return odfv[(((size_t)w * DX + li) * DY + lj) * DZ + lk];
    };
    float4 lo, hi;
    lo.x = fetch(txa, lxa, tya, lya, tza, lza);
    lo.y = fetch(txb, lxb, tya, lya, tza, lza);
    lo.z = fetch(txa, lxa, tyb, lyb, tza, lza);
    lo.w = fetch(txb, lxb, tyb, lyb, tza, lza);
    hi.x = fetch(txa, lxa, tya, lya, tzb, lzb);
    hi.y = fetch(txb, lxb, tya, lya, tzb, lzb);
    hi.z = fetch(txa, lxa, tyb, lyb, tzb, lzb);
    hi.w = fetch(txb, lxb, tyb, lyb, tzb, lzb);
    float4 *out = reinterpret_cast<float4 *>(blocks + (size_t)idx * 8);
    out[0] = lo;
    out[1] = hi;
}

// PttDirectionGetter.prepare_data (cu_direction_getters.py:531-625) on the
// device, one thread per voxel, in the host recipe's order: clip at 0 (NaN
// kept and -0.0 made +0.0, as numpy's clip does), zero the voxel where the stop value is
// below the threshold, then divide by the voxel's maximum when it is > 0 (a
// NaN maximum, as numpy's max propagates it, leaves the voxel unchanged).
__global__ void ptt_normalise(float *__restrict__ odf, const float *__restrict__ stop, float thr, long long nvox,
                              int T) {
    const long long v = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    if (v >= nvox) return;
    float *o = odf + (size_t)v * T;
    const bool zero = stop[v] < thr;
    float mx = 0.0f;
    bool first = true;
    for (int t = 0; t < T; ++t) {
        float x = o[t];
        x = zero ? 0.0f : (x > 0.0f || x != x) ? x : 0.0f;  // -0.0 becomes +0.0, as in numpy
        o[t] = x;
        if (first || x != x || x > mx) { if (!(mx != mx)) mx = x; }
        first = false;
    }
    if (mx > 0.0f)
        for (int t = 0; t < T; ++t) o[t] = o[t] / mx;
}

// Sets *flag when some value of x[0..n) is not >= 0 (negative or NaN).
__global__ void flag_not_nonneg(const float *__restrict__ x, long long n, int *__restrict__ flag) {
    bool bad = false;
    for (long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (long long)gridDim.x * blockDim.x)
        bad |= !(x[i] >= 0.0f);
    if (__any(bad) && (threadIdx.x & 63) == 0) atomicOr(flag, 1);
}

// Nearest sphere vertex of every point of the linspace(-1, 1, res)^3 grid
// ([i0][i1][i2], i2 fastest), as PttDirectionGetter.prepare_data's KDTree
// query (cu_direction_getters.py:601-623): grid values i * (2 / (res - 1)) - 1
// in double with the last one exactly 1 (numpy's linspace), squared
// Euclidean distances in double, the first of equal minima; with sphere_symm
// the antipodes are candidates too, after all the vertices.
__global__ void ptt_lut_kernel(const float *__restrict__ verts, int nv, int res, int symm, int32_t *__restrict__ lut) {
    const long long idx = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    const long long n = (long long)res * res * res;
    if (idx >= n) return;
    const int i2 = (int)(idx % res), i1 = (int)((idx / res) % res), i0 = (int)(idx / ((long long)res * res));
    const double step = 2.0 / (double)(res - 1);
    auto coord = [&](int i) -> double {
        if (i == res - 1) return 1.0;
        const double y = (double)i * step;
        return y + (-1.0);
    };
    const double px = coord(i0), py = coord(i1), pz = coord(i2);
    double best = 0.0;
    int bi = -1;
    for (int pass = 0; pass < (symm ? 2 : 1); ++pass) {
        const double sg = pass ? -1.0 : 1.0;
        for (int v = 0; v < nv; ++v) {
            const double dx = px - sg * (double)verts[3 * v], dy = py - sg * (double)verts[3 * v + 1],
                         dz = pz - sg * (double)verts[3 * v + 2];
            const double d = (dx * dx + dy * dy) + dz * dz;
            if (bi < 0 || d < best) { best = d; bi = v; }
        }
    }
    lut[idx] = bi;
}

// PTT data: [X][Y][Z][T] -> vertex-major [T][X][Y][Z] (32x32 LDS tiles).
__global__ void transpose_vox_t(const float *__restrict__ src, float *__restrict__ dst, long long nvox, int T) {
    __shared__ float tile[32][33];
    const long long v0 = (long long)blockIdx.x * 32;
    const int t0 = blockIdx.y * 32;
    const int tx = threadIdx.x & 31, ty = threadIdx.x >> 5;  // 32 x 8
    for (int k = ty; k < 32; k += 8) {
        const long long v = v0 + k;
        const int t = t0 + tx;
        if (v < nvox && t < T) tile[k][tx] = src[v * T + t];
    }
    __syncthreads();
    for (int k = ty; k < 32; k += 8) {
        const int t = t0 + k;
        const long long v = v0 + tx;
        if (v < nvox && t < T) dst[(long long)t * nvox + v] = tile[tx][k];
    }
}

// Exclusive scans of int32 counts (1024 elements per block, three passes).
template <typename TO>
__device__ TO block_incl_scan(TO x, TO *wsum) {
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
#pragma unroll
    for (int d = 1; d < 64; d <<= 1) {
        const TO o = __shfl_up(x, d, 64);
        if (lane >= d) x += o;
    }
    if (lane == 63) wsum[w] = x;
    __syncthreads();
    if (w == 0) {
        TO y = (lane < (int)(blockDim.x >> 6)) ? wsum[lane] : (TO)0;
#pragma unroll
        for (int d = 1; d < 64; d <<= 1) {
            const TO o = __shfl_up(y, d, 64);
            if (lane >= d) y += o;
        }
        if (lane < (int)(blockDim.x >> 6)) wsum[lane] = y;
    }
    __syncthreads();
    if (w > 0) x += wsum[w - 1];
    __syncthreads();
    return x;
}

template <typename TO>
__global__ void __launch_bounds__(1024) scan_pass1(const int *__restrict__ in, int n, TO *__restrict__ bsum) {
    __shared__ TO wsum[16];
    const long long i = (long long)blockIdx.x * 1024 + threadIdx.x;
    const TO x = (i < n) ? (TO)in[i] : (TO)0;
    const TO inc = block_incl_scan<TO>(x, wsum);
    if (threadIdx.x == 1023) bsum[blockIdx.x] = inc;
}

template <typename TO>
__global__ void __launch_bounds__(1024) scan_pass2(TO *__restrict__ bsum, int nb) {
    __shared__ TO wsum[16];
    __shared__ TO carry;
    if (threadIdx.x == 0) carry = 0;
    __syncthreads();
    for (int b0 = 0; b0 < nb; b0 += 1024) {
        const int i = b0 + threadIdx.x;
        const TO x = (i < nb) ? bsum[i] : (TO)0;
        const TO inc = block_incl_scan<TO>(x, wsum);
        const TO c = carry;
        if (i < nb) bsum[i] = c + inc - x;  // exclusive
        __syncthreads();
        if (threadIdx.x == 1023) carry = c + inc;
        __syncthreads();
    }
}

template <typename TO>
__global__ void __launch_bounds__(1024) scan_pass3(const int *__restrict__ in, int n, const TO *__restrict__ bsum,
                                                   TO *__restrict__ out) {
    __shared__ TO wsum[16];
    const long long i = (long long)blockIdx.x * 1024 + threadIdx.x;
    const TO x = (i < n) ? (TO)in[i] : (TO)0;
    const TO inc = block_incl_scan<TO>(x, wsum);
    const TO base = bsum[blockIdx.x];
    if (i < n) out[i] = base + inc - x;
    if (i == n - 1) out[n] = base + inc;
}

// Copy each streamline's points from its padded slot into the packed array.
__global__ void compact_kernel(const int *__restrict__ len, int nsl, const float *__restrict__ sline,
                               size_t slot_f, const long long *__restrict__ off, float *__restrict__ pts) {
    const int lane = threadIdx.x & 63;
    const int w = (blockIdx.x * blockDim.x + threadIdx.x) >> 6;
    const int nw = (gridDim.x * blockDim.x) >> 6;
    for (int k = w; k < nsl; k += nw) {
        const int nf = 3 * len[k];
        const float *src = sline + (size_t)k * slot_f;
        float *dst = pts + 3 * (size_t)off[k];
        for (int p = lane; p < nf; p += 64) dst[p] = src[p];
    }
}

// Totals of a bounded chunk (one thread): the chunk's streamlines
// (offsets[n]), the slots phase 2 filled -- the largest offset <= cap, as
// the offsets never decrease and a seed is tracked when its last slot is
// below the cap -- and the points compacted (point_off[cap]).
__global__ void chunk_totals(const int *__restrict__ offsets, int n, int cap, const long long *__restrict__ point_off,
                             long long *__restrict__ totals) {
    int lo = 0, hi = n;
    while (lo < hi) {
        const int mid = (lo + hi + 1) >> 1;
        if (offsets[mid] <= cap) lo = mid; else hi = mid - 1;
    }
    totals[0] = offsets[n];
    totals[1] = offsets[lo];
    totals[2] = point_off[cap];
}

}  // namespace

// Workspace of cuslines_phase2_noalloc_async: the spatial seed order of at
// most CUSLINES_NOALLOC_MAX_SEEDS seeds (order and keys).  One copy per
// device for the life of the process, shared by every call on that device.
constexpr size_t SCRATCH_INTS = 2 * (size_t)CUSLINES_NOALLOC_MAX_SEEDS;
static __device__ __align__(256) int scratch[SCRATCH_INTS];

// =========================================================================
// Host side: C ABI
// =========================================================================
thread_local std::string g_last_error;

static int fail(int code, const std::string &msg) {
    g_last_error = msg;
    return code;
}

// roctx range over one C-ABI call (phases show up by name in rocprofv3
// --marker-trace timelines).
struct RoctxRange {
    explicit RoctxRange(const char *name) { roctxRangePushA(name); }
    ~RoctxRange() { roctxRangePop(); }
};

#define HIPC(expr)                                                                                  \
    do {                                                                                            \
        hipError_t e_ = (expr);                                                                     \
        if (e_ != hipSuccess) return fail(CUSLINES_EHIP, std::string(#expr) + ": " + hipGetErrorString(e_)); \
    } while (0)

struct cuslines_tracker {
    cuslines_params p{};
    DevParams dp{};
    int device = 0;
    hipStream_t stream = nullptr;
    float *d_data = nullptr, *d_stop = nullptr, *d_verts = nullptr;
    uint32_t *d_edges = nullptr;
    uint16_t *d_nbr = nullptr;  // vertex adjacency, 8 per vertex (nullptr: a degree above 8 or > 1024 vertices)
    float *d_H = nullptr, *d_R = nullptr, *d_db = nullptr, *d_dq = nullptr, *d_smat = nullptr;
    float *d_hrm = nullptr, *d_fitm = nullptr, *d_odfm = nullptr;  // batched bootstrap matrices
    float *d_ut = nullptr, *d_u = nullptr, *d_invlev = nullptr;   // low-rank form of [H; R] (rk16 > 0)
    int rk16 = 0, hrank = 0;                                      // rank of H and rounded to 16 (0: not that form)
    int boot_full = 0;                                            // batched bootstrap: always the [H; R] product
    int boot_mode = CUSLINES_BOOT_EXACT;
    int boot_occ = 0;  // bootstrap: waves per SIMD of the kernel variant (0: by the seeds in flight, boot_waves)
    int *d_b0 = nullptr, *d_dwi = nullptr;
    uint32_t *d_lut = nullptr;
    std::vector<uint16_t> rank_vertex;  // PTT: vertex of each direction rank (corner-block order)
    int *d_work = nullptr;      // work-queue counters and class starts of the persistent phase-2 kernels (WORK_INTS)
    int *d_sort = nullptr;      // seed order: bucket counts, starts and block sums (sort_ints)
    void *scratch = nullptr;    // device address of this device's `scratch` array
    float *d_blocks = nullptr;  // PTT corner blocks
    int use_blocks = 1;
    int schedule = CUSLINES_SCHED_QUEUE;
    int threads = 0;        // 0: per-getter default
    int blocks_per_cu = 0;  // 0: occupancy maximum
    int num_cu = 1;
    int ptt_lanes = 0;      // PTT: lanes per seed (8, 16, 32; 0 = shared 32-lane kernel)
    int flat = 1;           // phase 2 on the queue: one loop of steps per seed slot (flat_slot)
    float *d_fprop = nullptr;            // learned proposal: feature propagators [24][9]
    float *d_vprop = nullptr;            // PTT vertex-phase propagators [24][9]
    uint16_t *d_mlp = nullptr;           // learned proposal (nullptr: plain getter)
    unsigned long long *d_stats = nullptr;
    int count_taps = 0;  // PTT phase 2 counts its taps and sub-steps into d_stats
    float *rec = nullptr;                // caller's training-pair buffer (nullptr: no recording)
    int *rec_count = nullptr;
    bool has_data = false, has_stop = false, has_sphere = false, has_boot = false, has_lut = false;
    cuslines_tracker *parent = nullptr;  // fork: the tracker whose device data it shares
    int nforks = 0;                      // live forks of this tracker
    int ngraphs = 0;                     // live chunk graphs on this tracker (a parent: and on its forks)
};

// A captured chunk (cuslines_chunk_graph_create): its kernel nodes hold the
// tracker's device pointers and launch settings as they were at capture.
struct cuslines_graph {
    cuslines_tracker *t;
    hipGraph_t graph;
    hipGraphExec_t exec;
};

static float smallest_float_at_least(double x) {
    float f = (float)x;
    if ((double)f < x) f = std::nextafter(f, INFINITY);
    return f;
}

static int ceil32(int x) { return (x + 31) & ~31; }

static DevBufs bufs_of(const cuslines_tracker *t) {
    DevBufs b;
    b.data = t->d_data;
    b.stop = t->d_stop;
    b.verts = t->d_verts;
    b.edges = t->d_edges;
    b.nbr = t->d_nbr;
    b.H = t->d_H; b.R = t->d_R; b.db = t->d_db; b.dq = t->d_dq; b.smat = t->d_smat;
    b.hr_mat = t->d_hrm; b.fit_mat = t->d_fitm; b.odf_mat = t->d_odfm;
    b.ut_mat = t->d_ut; b.u_mat = t->d_u; b.invlev = t->d_invlev;
    b.b0 = t->d_b0;
    b.dwi_idx = t->d_dwi;
    b.lut = t->d_lut;
    b.blocks = t->use_blocks ? t->d_blocks : nullptr;
    b.fprop = t->d_fprop;
    b.vprop = t->d_vprop;
    b.mlp = t->d_mlp;
    b.rec = t->rec;
    b.rec_count = t->rec_count;
    b.stats = t->d_stats;
    return b;
}

static void dfree(void *p) {
    if (p) (void)hipFree(p);
}

// Device address of `scratch` on each device, looked up once per device with
// that device current (each device holds its own copy of the array).
static std::mutex g_scratch_mu;
static std::vector<void *> g_scratch_ptr;

static int scratch_of_device(int device, void **out) {
    std::lock_guard<std::mutex> lock(g_scratch_mu);
    if ((int)g_scratch_ptr.size() <= device) g_scratch_ptr.resize((size_t)device + 1, nullptr);
    if (!g_scratch_ptr[device]) {
        void *p = nullptr;
        const hipError_t e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
        if (e != hipSuccess || !p)
            return fail(CUSLINES_EHIP, std::string("hipGetSymbolAddress(scratch): ") + hipGetErrorString(e));
        g_scratch_ptr[device] = p;
    }
    *out = g_scratch_ptr[device];
    return CUSLINES_OK;
}

static int check_ready(const cuslines_tracker *t) {
    if (!t->has_data || !t->has_stop || !t->has_sphere)
        return fail(CUSLINES_ESTATE, "data, stop map and sphere must be uploaded first");
    if ((t->p.model_type == CUSLINES_OPDT || t->p.model_type == CUSLINES_CSA) && !t->has_boot)
        return fail(CUSLINES_ESTATE, "bootstrap matrices must be uploaded first");
    if (t->p.model_type == CUSLINES_PTT && !t->has_lut) return fail(CUSLINES_ESTATE, "PTT LUT must be uploaded first");
    return CUSLINES_OK;
}

// Setters that replace device data are refused on forks (they share their
// parent's buffers) and on trackers with live forks.
static int check_owner(const cuslines_tracker *t) {
    if (t->parent) return fail(CUSLINES_ESTATE, "a fork shares its parent's data: configure the parent");
    if (t->nforks) return fail(CUSLINES_ESTATE, "live forks share this tracker's data: destroy them first");
    if (t->ngraphs) return fail(CUSLINES_ESTATE, "live chunk graphs hold this tracker's data: destroy them first");
    return CUSLINES_OK;
}

template <int MODEL>
static int launch_phase1(cuslines_tracker *t, const float *seeds, int n, int chunk, int *counts, int *dirs) {
    const DevParams &d = t->dp;
    const int threads = 128;
    const int nslots = threads / 32;
    const size_t vf = verts_in_lds<MODEL>() ? (size_t)((3 * d.nverts + 3) & ~3) : 0;
    const size_t lds = sizeof(float) * (vf + (size_t)nslots * slot_floats(MODEL, true, d.nv32, d.t32, d.hr32));
    if (lds > 160 * 1024) return fail(CUSLINES_EINVAL, "sphere too large for LDS");
    HIPC(hipFuncSetAttribute((const void *)phase1_kernel<MODEL>, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds));
    const unsigned grid = (unsigned)((n + nslots - 1) / nslots);
    hipLaunchKernelGGL(phase1_kernel<MODEL>, dim3(grid), dim3(threads), lds, t->stream, d, bufs_of(t), seeds, n,
                       chunk, counts, dirs);
    HIPC(hipGetLastError());
    return CUSLINES_OK;
}

static int spatial_order(cuslines_tracker *t, const float *seeds, const int *offsets, int n, int **order, int *ws);

// PTT with L lanes per seed: with flat stepping (t->flat, the default) the
// flat grouped kernel over the XCD-ordered queues of the spatial seed order
// (`ws` as launch_phase2_v), else the per-seed kernel over one counter.
template <int L>
static int launch_ptt_l(cuslines_tracker *t, int threads, const float *seeds, int n, int chunk, const int *offsets,
                        const int *dirs, int *sseed, int *slen, float *sl, int *ws) {
    const DevParams &d = t->dp;
    const size_t lds = sizeof(float) * (size_t)(PTTC_FLOATS + (threads / L) * PTTG_FLOATS);
    const bool flat = t->flat != 0;
    const void *kfn = flat ? (const void *)phase2_ptt_flat_kernel<L> : (const void *)phase2_ptt_queue_kernel<L>;
    HIPC(hipFuncSetAttribute(kfn, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds));
    int per_cu = 0;
    HIPC(hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, kfn, threads, lds));
    if (per_cu < 1) per_cu = 1;
    if (t->blocks_per_cu > 0 && t->blocks_per_cu < per_cu) per_cu = t->blocks_per_cu;
    long long grid = (long long)per_cu * t->num_cu;
    const long long need = ((long long)n * L + threads - 1) / threads;
    if (grid > need) grid = need;
    if (grid < 1) grid = 1;
    int *order = nullptr;
    if (flat)
        if (int rc = spatial_order(t, seeds, offsets, n, &order, ws)) return rc;
    if (!flat) hipLaunchKernelGGL(zero_ints, dim3(1), dim3(64), 0, t->stream, t->d_work, 1);
    if (flat)
        hipLaunchKernelGGL(phase2_ptt_flat_kernel<L>, dim3((unsigned)grid), dim3(threads), lds, t->stream, d,
                           bufs_of(t), seeds, n, chunk, offsets, dirs, sseed, slen, sl, order, t->d_work);
    else
        hipLaunchKernelGGL(phase2_ptt_queue_kernel<L>, dim3((unsigned)grid), dim3(threads), lds, t->stream, d,
                           bufs_of(t), seeds, n, chunk, offsets, dirs, sseed, slen, sl, t->d_work);
    const hipError_t e = hipGetLastError();
    if (flat && !ws) (void)hipFreeAsync(order, t->stream);
    if (e != hipSuccess) return fail(CUSLINES_EHIP, std::string("phase 2 (PTT groups): ") + hipGetErrorString(e));
    return CUSLINES_OK;
}

static int launch_ptt_groups(cuslines_tracker *t, const float *seeds, int n, int chunk, const int *offsets,
                             const int *dirs, int *sseed, int *slen, float *sl, int *ws) {
    const int threads = t->threads > 0 ? t->threads : 256;
    switch (t->ptt_lanes) {
        case 8: return launch_ptt_l<8>(t, threads, seeds, n, chunk, offsets, dirs, sseed, slen, sl, ws);
        case 16: return launch_ptt_l<16>(t, threads, seeds, n, chunk, offsets, dirs, sseed, slen, sl, ws);
        default: return launch_ptt_l<32>(t, threads, seeds, n, chunk, offsets, dirs, sseed, slen, sl, ws);
    }
}

template <typename TO>
static int run_scan(cuslines_tracker *t, const int *in, int n, TO *out, TO *bsum_ws = nullptr);

// Buckets of the seed order: 4-voxel bricks (coarser when a dimension
// exceeds 256 voxels), at most 2^18 of them in each of the 8 classes.
static int order_buckets(const DevParams &d, int *brick_log2_out) {
    int mx = d.dimx > d.dimy ? d.dimx : d.dimy;
    mx = mx > d.dimz ? mx : d.dimz;
    int brick_log2 = 2;
    while (((mx - 1) >> brick_log2) >= 64) ++brick_log2;
    int bits = 0;
    while ((1 << bits) <= ((mx - 1) >> brick_log2)) ++bits;
    *brick_log2_out = brick_log2;
    return SEED_CLASSES << (3 * bits);
}

// ints of the counting sort's own arrays: bucket counts (nb), bucket starts
// (nb + 1) and the scan's block sums.  They are the handle's (2 MiB at
// 81x106x76, 16 MiB at the most), not part of a caller's workspace: their size
// follows how this library orders seeds, and a workspace that was large
// enough once stays so.
static size_t sort_ints(int nb) { return 2 * (size_t)nb + 1 + (size_t)((nb + 1023) / 1024); }

// ints of the seed-order workspace: order and keys.
static size_t order_ws_ints(int n) { return 2 * (size_t)n; }

// Seeds by class and, in a class, in Morton order of their brick, by a counting
// sort on the tracker's stream; the queue's counters and class starts in
// t->d_work.  Without offsets the seeds are one class.  With `ws`
// (order_ws_ints(n) ints of device memory) order and keys are carved from it
// and *order points into it; without, they are stream-ordered allocations and
// the caller frees *order with hipFreeAsync.
static int spatial_order(cuslines_tracker *t, const float *seeds, const int *offsets, int n, int **order, int *ws) {
    const DevParams &d = t->dp;
    int brick_log2 = 0;
    const int nb = order_buckets(d, &brick_log2);
    int *count = t->d_sort, *start = count + nb, *bsum = start + nb + 1;
    int *key = nullptr;
    if (ws) {
        *order = ws;
        key = ws + n;
    } else {
        *order = nullptr;
        hipError_t e = hipMallocAsync((void **)order, (size_t)n * sizeof(int), t->stream);
        if (e == hipSuccess) e = hipMallocAsync((void **)&key, (size_t)n * sizeof(int), t->stream);
        if (e != hipSuccess) {
            if (*order) (void)hipFreeAsync(*order, t->stream);
            *order = nullptr;
            return fail(CUSLINES_ENOMEM, std::string("seed order: ") + hipGetErrorString(e));
        }
    }
    const dim3 gb((unsigned)((nb + 255) / 256)), gs((unsigned)((n + 255) / 256));
    hipLaunchKernelGGL(zero_ints, gb, dim3(256), 0, t->stream, count, nb);
    hipLaunchKernelGGL(seed_keys, gs, dim3(256), 0, t->stream, d, seeds, offsets, n, brick_log2, nb / SEED_CLASSES, key,
                       count);
    int rc = run_scan<int>(t, count, nb, start, bsum);
    if (rc == CUSLINES_OK) {
        hipLaunchKernelGGL(zero_ints, gb, dim3(256), 0, t->stream, count, nb);
        hipLaunchKernelGGL(seed_scatter, gs, dim3(256), 0, t->stream, key, n, start, count, *order);
        hipLaunchKernelGGL(queue_init, dim3(1), dim3(64), 0, t->stream, t->d_work, start, nb / SEED_CLASSES);
    }
    hipError_t e = hipGetLastError();
    if (!ws) (void)hipFreeAsync(key, t->stream);
    if (rc) return rc;
    if (e != hipSuccess) return fail(CUSLINES_EHIP, std::string("seed order: ") + hipGetErrorString(e));
    return CUSLINES_OK;
}

template <int MODEL, int V>
static int launch_phase2_v(cuslines_tracker *t, const float *seeds, int n, int chunk, const int *offsets,
                           const int *dirs, int *sseed, int *slen, float *sl, int *ws) {
    const DevParams &d = t->dp;
    int threads = t->threads;
    if (threads <= 0) threads = (MODEL == CUSLINES_OPDT || MODEL == CUSLINES_CSA) ? 128 : 256;
    // learned: 512-thread workgroups of the queue kernel share one staged
    // copy of the network (50 KB of LDS) among 16 slots
    if (V == 1 && t->threads <= 0 && t->schedule != CUSLINES_SCHED_STATIC) threads = 512;
    if (V == 5 && t->threads <= 0) threads = 768;
    const int nslots = threads / 32;
    const size_t vf = ((MODEL == CUSLINES_PROB) ? (size_t)((3 * d.nverts + 3) & ~3) : 0) +
                      ((V == 1 || V == 5) ? (size_t)MLP_LDS_FLOATS : 0);
    const size_t lds = sizeof(float) * (vf + (size_t)nslots * (slot_floats(MODEL, false, d.nv32, d.t32, d.hr32) +
                                                             ((V >= 4) ? FLAT_STATE_FLOATS : 0)));
    if (lds > 160 * 1024) return fail(CUSLINES_EINVAL, "sphere too large for LDS");
    if constexpr (V < 4) {  // the flat loops are the queue's
        if (t->schedule == CUSLINES_SCHED_STATIC) {
            HIPC(hipFuncSetAttribute((const void *)phase2_kernel<MODEL, V>,
                                     hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds));
            const unsigned grid = (unsigned)((n + nslots - 1) / nslots);
            hipLaunchKernelGGL((phase2_kernel<MODEL, V>), dim3(grid), dim3(threads), lds, t->stream, d, bufs_of(t),
                               seeds, n, chunk, offsets, dirs, sseed, slen, sl);
            HIPC(hipGetLastError());
            return CUSLINES_OK;
        }
    }
    const void *kfn = (const void *)phase2_queue_kernel<MODEL, V>;
    HIPC(hipFuncSetAttribute(kfn, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds));
    int per_cu = 0;
    HIPC(hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, kfn, threads, lds));
    if (per_cu < 1) per_cu = 1;
    if (t->blocks_per_cu > 0 && t->blocks_per_cu < per_cu) per_cu = t->blocks_per_cu;
    long long grid = (long long)per_cu * t->num_cu;
    const long long need = (n + nslots - 1) / nslots;
    if (grid > need) grid = need;
    if (grid < 1) grid = 1;
    int *order = nullptr;
    // A recording run keeps the spatial order: its pairs are stored as they come
    // until the buffer is full, and by class a buffer smaller than the run would
    // hold those of the seeds with the most directions only.
    if (int rc = spatial_order(t, seeds, V == 2 ? nullptr : offsets, n, &order, ws)) return rc;
    hipLaunchKernelGGL((phase2_queue_kernel<MODEL, V>), dim3((unsigned)grid), dim3(threads), lds, t->stream, d,
                       bufs_of(t), seeds, n, chunk, offsets, dirs, sseed, slen, sl, order, t->d_work);
    hipError_t e = hipGetLastError();
    if (!ws) (void)hipFreeAsync(order, t->stream);
    if (e != hipSuccess) return fail(CUSLINES_EHIP, std::string("phase 2: ") + hipGetErrorString(e));
    return CUSLINES_OK;
}

// A persistent queue kernel over the spatial seed order, as launch_phase2_v:
// `threads` a workgroup, `nslots` seed slots in it, `lds` bytes.
template <typename K>
static int launch_queue(cuslines_tracker *t, K kernel, int threads, int nslots, size_t lds, const float *seeds, int n,
                        int chunk, const int *offsets, const int *dirs, int *sseed, int *slen, float *sl, int *ws) {
    const DevParams &d = t->dp;
    HIPC(hipFuncSetAttribute((const void *)kernel, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds));
    int per_cu = 0;
    HIPC(hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, (const void *)kernel, threads, lds));
    if (per_cu < 1) per_cu = 1;
    if (t->blocks_per_cu > 0 && t->blocks_per_cu < per_cu) per_cu = t->blocks_per_cu;
    long long grid = (long long)per_cu * t->num_cu;
    const long long need = (n + nslots - 1) / nslots;
    if (grid > need) grid = need;
    if (grid < 1) grid = 1;
    int *order = nullptr;
    if (int rc = spatial_order(t, seeds, offsets, n, &order, ws)) return rc;
    hipLaunchKernelGGL(kernel, dim3((unsigned)grid), dim3(threads), lds, t->stream, d, bufs_of(t), seeds, n, chunk,
                       offsets, dirs, sseed, slen, sl, order, t->d_work);
    hipError_t e = hipGetLastError();
    if (!ws) (void)hipFreeAsync(order, t->stream);
    if (e != hipSuccess) return fail(CUSLINES_EHIP, std::string("phase 2: ") + hipGetErrorString(e));
    return CUSLINES_OK;
}

// Probabilistic phase 2 with the cell in registers: NCH chunks of 256
// channels; one wave a workgroup, so that few seeds spread over the CUs.
template <int NCH>
static int launch_prob(cuslines_tracker *t, const float *seeds, int n, int chunk, const int *offsets, const int *dirs,
                       int *sseed, int *slen, float *sl, int *ws) {
    const int threads = t->threads > 0 ? t->threads : 64;
    const int nslots = threads / 64;
    const size_t lds = sizeof(float) * (3 * 256 * NCH + (size_t)nslots * prob_slot_floats(NCH));
    return launch_queue(t, phase2_prob_kernel<NCH>, threads, nslots, lds, seeds, n, chunk, offsets, dirs, sseed, slen,
                        sl, ws);
}

// Plain PTT phase 2; one wave a workgroup.
static int launch_ptt(cuslines_tracker *t, const float *seeds, int n, int chunk, const int *offsets, const int *dirs,
                      int *sseed, int *slen, float *sl, int *ws) {
    const int threads = t->threads > 0 ? t->threads : 64;
    const int nslots = threads / 32;
    const size_t lds = sizeof(float) * (PTT_TAB_FLOATS + (size_t)nslots * PTT_FLAT_FLOATS);
    return launch_queue(t, phase2_ptt_kernel, threads, nslots, lds, seeds, n, chunk, offsets, dirs, sseed, slen, sl, ws);
}

// Limits of the batched bootstrap kernel's tile counts per wave.
static bool boot_batch_fits(const DevParams &d) {
    return d.hr16 <= 320 && d.dn16 <= 128 && d.nv16 <= 768 && d.dn16 <= d.t32;
}

// Waves per SIMD of the bootstrap kernels' variant for a launch of n seeds:
// up to 8 seeds in flight for each slot of the 2-waves variant (16 a CU) the
// run lasts as long as its longest seeds, whose steps the larger register
// budget shortens; beyond, the other variant's second set of slots hides more.
// In ms at 2 | 4 waves (81x106x76, 160 directions):
//   batched CSA: 20 000 seeds 53 | 57, 32 000 80 | 88, 40 000 91 | 81, 60 000 111 | 93
//   exact CSA: 200 seeds 132 | 160, 3001 158 | 195, 20 000 170 | 206, 32 000 250 | 308, 40 000 281 | 275,
//   60 000 346 | 308, 200 000 996 | 745; exact OPDT: 20 000 190 | 238, 32 000 265 | 324, 40 000 300 | 355
// A handle with forks is one of a pipeline's: each of them is taken to have as
// many seeds in flight.  200,000 CSA seeds as chunks of 25,000 on 8 handles, end
// to end, by the launch's seeds | by all handles': exact 1,880 | 1,645 ms, batched
// 1,050 | 1,005 ms (OPDT exact 1,500 | 1,510, batched 782 | 769).
static int boot_waves(const cuslines_tracker *t, int n) {
    if (t->boot_occ) return t->boot_occ;
    const cuslines_tracker *root = t->parent ? t->parent : t;
    const long long handles = 1 + (long long)__atomic_load_n(&root->nforks, __ATOMIC_RELAXED);
    return (n * handles <= 8LL * BB_SLOTS * t->num_cu) ? 2 : 4;
}

template <int MODEL>
static int launch_boot_batch(cuslines_tracker *t, const float *seeds, int n, int chunk, const int *offsets,
                             const int *dirs, int *sseed, int *slen, float *sl, int *ws) {
    DevParams d = t->dp;
    d.rk16 = t->boot_full ? 0 : t->rk16;  // H.d = U (U^T d) and R.d from it
    if (!boot_batch_fits(d))
        return fail(CUSLINES_EINVAL, "batched bootstrap needs hr <= 320, delta_nr <= 128 and nverts <= 768");
    const size_t lds = sizeof(float) * ((size_t)BB_SLOTS * (size_t)bb_slot_stride(d.nv32, d.t32, d.hr32) +
                                        2 * (size_t)BB_WAVES * 16 + BB_SLOTS);
    if (lds > 160 * 1024) return fail(CUSLINES_EINVAL, "batched bootstrap slots too large for LDS");
    const bool lr = d.rk16 > 0;
    const int occ = boot_waves(t, n);
    const void *kfn = (occ == 4)
                          ? (lr ? (const void *)phase2_boot_batch_kernel<MODEL, 4, true>
                                : (const void *)phase2_boot_batch_kernel<MODEL, 4, false>)
                          : (lr ? (const void *)phase2_boot_batch_kernel<MODEL, 2, true>
                                : (const void *)phase2_boot_batch_kernel<MODEL, 2, false>);
    HIPC(hipFuncSetAttribute(kfn, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds));
    int per_cu = 0;
    HIPC(hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, kfn, BB_THREADS, lds));
    if (per_cu < 1) per_cu = 1;
    if (t->blocks_per_cu > 0 && t->blocks_per_cu < per_cu) per_cu = t->blocks_per_cu;
    long long grid = (long long)per_cu * t->num_cu;
    if (grid > n) grid = n;
    if (grid < 1) grid = 1;
    if (!t->d_stats && !ws) {  // the kernel's attempt and round counters (not allocated by the no-alloc entry)
        HIPC(hipMalloc(&t->d_stats, 4 * sizeof(unsigned long long)));
        HIPC(hipMemsetAsync(t->d_stats, 0, 4 * sizeof(unsigned long long), t->stream));
    }
    int *order = nullptr;
    if (int rc = spatial_order(t, seeds, offsets, n, &order, ws)) return rc;
    const DevBufs bb = bufs_of(t);
    const dim3 g((unsigned)grid), b(BB_THREADS);
    if (occ == 4 && lr)
        hipLaunchKernelGGL((phase2_boot_batch_kernel<MODEL, 4, true>), g, b, lds, t->stream, d, bb, seeds, n, chunk,
                           offsets, dirs, sseed, slen, sl, order, t->d_work);
    else if (occ == 4)
        hipLaunchKernelGGL((phase2_boot_batch_kernel<MODEL, 4, false>), g, b, lds, t->stream, d, bb, seeds, n, chunk,
                           offsets, dirs, sseed, slen, sl, order, t->d_work);
    else if (lr)
        hipLaunchKernelGGL((phase2_boot_batch_kernel<MODEL, 2, true>), g, b, lds, t->stream, d, bb, seeds, n, chunk,
                           offsets, dirs, sseed, slen, sl, order, t->d_work);
    else
        hipLaunchKernelGGL((phase2_boot_batch_kernel<MODEL, 2, false>), g, b, lds, t->stream, d, bb, seeds, n, chunk,
                           offsets, dirs, sseed, slen, sl, order, t->d_work);
    hipError_t e = hipGetLastError();
    if (!ws) (void)hipFreeAsync(order, t->stream);
    if (e != hipSuccess) return fail(CUSLINES_EHIP, std::string("phase 2 (batched): ") + hipGetErrorString(e));
    return CUSLINES_OK;
}

template <int MODEL>
static int launch_phase2(cuslines_tracker *t, const float *seeds, int n, int chunk, const int *offsets,
                         const int *dirs, int *sseed, int *slen, float *sl, int *ws) {
    if constexpr (MODEL == CUSLINES_OPDT || MODEL == CUSLINES_CSA) {
        if (t->boot_mode == CUSLINES_BOOT_MFMA && t->schedule != CUSLINES_SCHED_STATIC)
            return launch_boot_batch<MODEL>(t, seeds, n, chunk, offsets, dirs, sseed, slen, sl, ws);
    }
    if constexpr (MODEL == CUSLINES_PTT) {
        if (t->d_mlp && t->flat && t->schedule != CUSLINES_SCHED_STATIC)
            return launch_phase2_v<MODEL, 5>(t, seeds, n, chunk, offsets, dirs, sseed, slen, sl, ws);
        if (t->d_mlp)
            return launch_phase2_v<MODEL, 1>(t, seeds, n, chunk, offsets, dirs, sseed, slen, sl, ws);
        if (t->rec)
            return launch_phase2_v<MODEL, 2>(t, seeds, n, chunk, offsets, dirs, sseed, slen, sl, ws);
        if (t->count_taps)
            return launch_phase2_v<MODEL, 3>(t, seeds, n, chunk, offsets, dirs, sseed, slen, sl, ws);
        if (t->ptt_lanes > 0 && t->schedule != CUSLINES_SCHED_STATIC)
            return launch_ptt_groups(t, seeds, n, chunk, offsets, dirs, sseed, slen, sl, ws);
        if (t->flat && t->schedule != CUSLINES_SCHED_STATIC)
            return launch_ptt(t, seeds, n, chunk, offsets, dirs, sseed, slen, sl, ws);
    }
    if constexpr (MODEL == CUSLINES_PROB) {
        // a lane keeps 4 of a chunk's 256 channels, 8 corners each: 3 chunks fit the registers
        if (t->flat && t->schedule != CUSLINES_SCHED_STATIC) switch ((t->dp.t32 + 255) / 256) {
            case 1: return launch_prob<1>(t, seeds, n, chunk, offsets, dirs, sseed, slen, sl, ws);
            case 2: return launch_prob<2>(t, seeds, n, chunk, offsets, dirs, sseed, slen, sl, ws);
            case 3: return launch_prob<3>(t, seeds, n, chunk, offsets, dirs, sseed, slen, sl, ws);
            default: break;
        }
    }
    if constexpr (MODEL != CUSLINES_PTT) {
        if constexpr (MODEL != CUSLINES_PROB) {
            if (t->flat && t->schedule != CUSLINES_SCHED_STATIC && boot_waves(t, n) == 2)
                return launch_phase2_v<MODEL, 6>(t, seeds, n, chunk, offsets, dirs, sseed, slen, sl, ws);
        }
        if (t->flat && t->schedule != CUSLINES_SCHED_STATIC)
            return launch_phase2_v<MODEL, 4>(t, seeds, n, chunk, offsets, dirs, sseed, slen, sl, ws);
    }
    return launch_phase2_v<MODEL, 0>(t, seeds, n, chunk, offsets, dirs, sseed, slen, sl, ws);
}

template <typename TO>
static int run_scan(cuslines_tracker *t, const int *in, int n, TO *out, TO *bsum_ws) {
    if (n <= 0) {
        hipLaunchKernelGGL(zero_scalar<TO>, dim3(1), dim3(1), 0, t->stream, out);
        HIPC(hipGetLastError());
        return CUSLINES_OK;
    }
    const int nb = (n + 1023) / 1024;
    TO *bsum = bsum_ws;
    if (!bsum) HIPC(hipMallocAsync((void **)&bsum, (size_t)nb * sizeof(TO), t->stream));
    hipLaunchKernelGGL(scan_pass1<TO>, dim3(nb), dim3(1024), 0, t->stream, in, n, bsum);
    hipLaunchKernelGGL(scan_pass2<TO>, dim3(1), dim3(1024), 0, t->stream, bsum, nb);
    hipLaunchKernelGGL(scan_pass3<TO>, dim3(nb), dim3(1024), 0, t->stream, in, n, bsum, out);
    hipError_t e = hipGetLastError();
    if (!bsum_ws) (void)hipFreeAsync(bsum, t->stream);
    if (e != hipSuccess) return fail(CUSLINES_EHIP, std::string("scan: ") + hipGetErrorString(e));
    return CUSLINES_OK;
}

static int phase1_models(cuslines_tracker *t, const float *seeds, int n, int chunk, int *counts, int *dirs) {
    switch (t->p.model_type) {
        case CUSLINES_OPDT: return launch_phase1<CUSLINES_OPDT>(t, seeds, n, chunk, counts, dirs);
        case CUSLINES_CSA: return launch_phase1<CUSLINES_CSA>(t, seeds, n, chunk, counts, dirs);
        case CUSLINES_PROB: return launch_phase1<CUSLINES_PROB>(t, seeds, n, chunk, counts, dirs);
        default: return launch_phase1<CUSLINES_PTT>(t, seeds, n, chunk, counts, dirs);
    }
}

// Phase 2 of the handle's model; `ws` as launch_phase2_v (nullptr:
// stream-ordered allocations).
static int phase2_models(cuslines_tracker *t, const float *seeds, int n, int chunk, const int *offsets,
                         const int *dirs, int *sseed, int *slen, float *sl, int *ws) {
    switch (t->p.model_type) {
        case CUSLINES_OPDT:
            return launch_phase2<CUSLINES_OPDT>(t, seeds, n, chunk, offsets, dirs, sseed, slen, sl, ws);
        case CUSLINES_CSA:
            return launch_phase2<CUSLINES_CSA>(t, seeds, n, chunk, offsets, dirs, sseed, slen, sl, ws);
        case CUSLINES_PROB:
            return launch_phase2<CUSLINES_PROB>(t, seeds, n, chunk, offsets, dirs, sseed, slen, sl, ws);
        default:
            return launch_phase2<CUSLINES_PTT>(t, seeds, n, chunk, offsets, dirs, sseed, slen, sl, ws);
    }
}

static size_t align256(size_t x) { return (x + 255) & ~(size_t)255; }

// Workspace of a bounded chunk: the seed order's (order_ws_ints), then the
// block sums of the streamline-count scan (int) and of the point scan (int64).
static size_t chunk_ws_bytes(int n, int cap) {
    return align256(order_ws_ints(n) * sizeof(int)) +
           align256((size_t)((n + 1023) / 1024) * sizeof(int)) + (size_t)((cap + 1023) / 1024) * sizeof(long long);
}

// The stream work of cuslines_chunk_async (arguments already checked):
// phase 1, the scan, the lengths of the `cap` slots cleared, phase 2 of the
// seeds that fit (DevParams::slot_cap), the point scan and compaction over
// the `cap` slots and the totals.  No allocation and no host read.
static int chunk_enqueue(cuslines_tracker *t, const float *seeds, int n, int chunk, int *counts, int *dirs,
                         int *offsets, int cap, int *sseed, int *slen, float *sl, long long *poff, float *pts,
                         long long *totals, char *ws) {
    int *order_ws = reinterpret_cast<int *>(ws);
    char *p = ws + align256(order_ws_ints(n) * sizeof(int));
    int *scan_ws = reinterpret_cast<int *>(p);
    long long *pscan_ws = reinterpret_cast<long long *>(p + align256((size_t)((n + 1023) / 1024) * sizeof(int)));
    if (n > 0)
        if (int rc = phase1_models(t, seeds, n, chunk, counts, dirs)) return rc;
    if (int rc = run_scan<int>(t, counts, n, offsets, scan_ws)) return rc;
    hipLaunchKernelGGL(zero_ints, dim3((unsigned)((cap + 255) / 256)), dim3(256), 0, t->stream, slen, cap);
    HIPC(hipGetLastError());
    if (n > 0) {
        t->dp.slot_cap = cap;  // copied into the launches' arguments
        const int rc = phase2_models(t, seeds, n, chunk, offsets, dirs, sseed, slen, sl, order_ws);
        t->dp.slot_cap = 0;
        if (rc) return rc;
    }
    if (int rc = run_scan<long long>(t, slen, cap, poff, pscan_ws)) return rc;
    const size_t slot_f = (size_t)2 * t->dp.max_sline_len * 3;
    const unsigned grid = (unsigned)std::min<long long>(((long long)cap + 3) / 4, 65536);
    hipLaunchKernelGGL(compact_kernel, dim3(grid), dim3(256), 0, t->stream, slen, cap, sl, slot_f, poff, pts);
    hipLaunchKernelGGL(chunk_totals, dim3(1), dim3(1), 0, t->stream, offsets, n, cap, poff, totals);
    HIPC(hipGetLastError());
    return CUSLINES_OK;
}

struct chunk_args {
    const float *seeds;
    int n, chunk;
    int *counts, *dirs, *offsets;
    int cap;
    int *sseed, *slen;
    float *sl;
    long long *poff;
    float *pts;
    long long *totals;
    char *ws;
};

static int chunk_check(cuslines_tracker *t, const float *seeds_d, int32_t nseeds, int32_t rng_chunk, int32_t *counts_d,
                       int32_t *dirs_d, int32_t *offsets_d, int32_t slot_cap, int32_t *sline_seed_d,
                       int32_t *sline_len_d, float *sline_d, int64_t *point_off_d, float *points_d, int64_t *totals_d,
                       void *ws_d, size_t ws_bytes, chunk_args *a) {
    if (!t) return fail(CUSLINES_EINVAL, "null tracker");
    if (nseeds < 0 || rng_chunk < 0) return fail(CUSLINES_EINVAL, "negative size");
    if (slot_cap < 1) return fail(CUSLINES_EINVAL, "slot_cap must be at least 1");
    if ((nseeds > 0 && (!seeds_d || !counts_d || !dirs_d)) || !offsets_d || !sline_seed_d || !sline_len_d ||
        !sline_d || !point_off_d || !points_d || !totals_d || !ws_d)
        return fail(CUSLINES_EINVAL, "null buffer");
    if (int rc = check_ready(t)) return rc;
    const size_t need = chunk_ws_bytes(nseeds, slot_cap);
    if (ws_bytes < need)
        return fail(CUSLINES_EINVAL, "workspace of " + std::to_string(ws_bytes) + " bytes, " + std::to_string(need) +
                                         " needed (cuslines_chunk_workspace_bytes)");
    if ((reinterpret_cast<uintptr_t>(ws_d) & 255) != 0) return fail(CUSLINES_EINVAL, "workspace not 256-byte aligned");
    *a = chunk_args{seeds_d, nseeds, rng_chunk > 0 ? rng_chunk : nseeds, counts_d, dirs_d, offsets_d, slot_cap,
                    sline_seed_d, sline_len_d, sline_d, reinterpret_cast<long long *>(point_off_d), points_d,
                    reinterpret_cast<long long *>(totals_d), static_cast<char *>(ws_d)};
    return CUSLINES_OK;
}

static int chunk_run(cuslines_tracker *t, const chunk_args &a) {
    return chunk_enqueue(t, a.seeds, a.n, a.chunk, a.counts, a.dirs, a.offsets, a.cap, a.sseed, a.slen, a.sl, a.poff,
                         a.pts, a.totals, a.ws);
}

// Both phase-2 entry points.  noalloc: the seed-order workspace is this
// device's `scratch` array instead of stream-ordered allocations.
static int phase2_entry(cuslines_tracker *t, const float *seeds_d, int32_t nseeds, int32_t rng_chunk,
                        const int32_t *offsets_d, const int32_t *dirs_d, int32_t *sline_seed_d, int32_t *sline_len_d,
                        float *sline_d, bool noalloc) {
    RoctxRange range_("cuslines_phase2");
    if (!t) return fail(CUSLINES_EINVAL, "null tracker");
    if (nseeds < 0 || rng_chunk < 0) return fail(CUSLINES_EINVAL, "negative size");
    if (noalloc) {
        if (!t->scratch) return fail(CUSLINES_ESTATE, "no scratch array on this device");
        if (nseeds > CUSLINES_NOALLOC_MAX_SEEDS)
            return fail(CUSLINES_EINVAL, "nseeds exceeds CUSLINES_NOALLOC_MAX_SEEDS (" +
                                             std::to_string(CUSLINES_NOALLOC_MAX_SEEDS) + ")");
    }
    if (nseeds == 0) return CUSLINES_OK;
    if (!seeds_d || !offsets_d || !dirs_d || !sline_seed_d || !sline_len_d || !sline_d)
        return fail(CUSLINES_EINVAL, "null buffer");
    int rc = check_ready(t);
    if (rc) return rc;
    int *ws = noalloc ? static_cast<int *>(t->scratch) : nullptr;
    HIPC(hipSetDevice(t->device));
    const int chunk = rng_chunk > 0 ? rng_chunk : nseeds;
    return phase2_models(t, seeds_d, nseeds, chunk, offsets_d, dirs_d, sline_seed_d, sline_len_d, sline_d, ws);
}

extern "C" {

int cuslines_abi_version(void) { return CUSLINES_ABI_VERSION; }

int cuslines_last_error(char *buf, size_t len) {
    if (!buf || len == 0) return CUSLINES_EINVAL;
    const size_t n = std::min(len - 1, g_last_error.size());
    std::memcpy(buf, g_last_error.data(), n);
    buf[n] = '\0';
    return CUSLINES_OK;
}

int cuslines_device_count(int *count) {
    if (!count) return fail(CUSLINES_EINVAL, "count is null");
    int n = 0;
    HIPC(hipGetDeviceCount(&n));
    *count = n;
    return CUSLINES_OK;
}

int cuslines_tracker_create(const cuslines_params *p, int device, cuslines_tracker **out) {
    if (!p || !out) return fail(CUSLINES_EINVAL, "null argument");
    *out = nullptr;
    if (p->dimx <= 0 || p->dimy <= 0 || p->dimz <= 0 || p->dimt <= 0)
        return fail(CUSLINES_EINVAL, "volume dimensions must be positive");
    if (p->model_type < CUSLINES_OPDT || p->model_type > CUSLINES_PTT)
        return fail(CUSLINES_EINVAL, "invalid model type");
    if (p->nverts <= 0 || p->nverts > 65535 || p->nedges <= 0)
        return fail(CUSLINES_EINVAL, "sphere must have 1..65535 vertices and at least one edge");
    if (p->max_sline_len < 2) return fail(CUSLINES_EINVAL, "max_sline_len must be >= 2");
    if ((p->model_type == CUSLINES_PROB || p->model_type == CUSLINES_PTT) && p->nverts != p->dimt)
        return fail(CUSLINES_EINVAL, "prob/PTT data must hold one ODF value per sphere vertex");
    if (p->model_type == CUSLINES_PTT) {
        if (p->step_frac < 1 || p->probe_quality < 1 || p->lut_res < 2)
            return fail(CUSLINES_EINVAL, "invalid PTT parameters");
        const long long slots = 1LL << (p->tile_log2_x + p->tile_log2_y + p->tile_log2_z);
        if (slots < p->dimt) return fail(CUSLINES_EINVAL, "PTT tiling has fewer slots than vertices");
        // limits of the 24-bit index products in interp4
        const long long X1 = p->dimx + 1LL, Y1 = p->dimy + 1LL, Z1 = p->dimz + 1LL;
        if (p->lut_res > 1024 || X1 * Y1 >= (1LL << 24) || X1 * Y1 * Z1 >= (1LL << 32) ||
            (1LL << p->tile_log2_x) * p->dimx >= (1LL << 24) || (1LL << p->tile_log2_y) * p->dimy >= (1LL << 24) ||
            (1LL << p->tile_log2_z) * p->dimz >= (1LL << 24))
            return fail(CUSLINES_EINVAL, "PTT volume or LUT too large for the tap index arithmetic");
    }
    if ((p->model_type == CUSLINES_OPDT || p->model_type == CUSLINES_CSA) && p->delta_nr <= 0)
        return fail(CUSLINES_EINVAL, "bootstrap needs delta_nr > 0");
    int ndev = 0;
    HIPC(hipGetDeviceCount(&ndev));
    if (device < 0 || device >= ndev) return fail(CUSLINES_EINVAL, "device index out of range");
    HIPC(hipSetDevice(device));
    cuslines_tracker *t = new cuslines_tracker();
    t->p = *p;
    t->device = device;
    hipError_t e = hipStreamCreateWithFlags(&t->stream, hipStreamNonBlocking);
    if (e != hipSuccess) {
        delete t;
        return fail(CUSLINES_EHIP, std::string("hipStreamCreateWithFlags: ") + hipGetErrorString(e));
    }
    e = hipMalloc(&t->d_work, WORK_INTS * sizeof(int));
    if (e == hipSuccess) e = hipDeviceGetAttribute(&t->num_cu, hipDeviceAttributeMultiprocessorCount, device);
    if (e != hipSuccess) {
        dfree(t->d_work);
        (void)hipStreamDestroy(t->stream);
        delete t;
        return fail(CUSLINES_EHIP, std::string("tracker setup: ") + hipGetErrorString(e));
    }
    if (int rc = scratch_of_device(device, &t->scratch)) {
        dfree(t->d_work);
        (void)hipStreamDestroy(t->stream);
        delete t;
        return rc;
    }
    DevParams &d = t->dp;
    d.dimx = p->dimx; d.dimy = p->dimy; d.dimz = p->dimz; d.dimt = p->dimt; d.t32 = ceil32(p->dimt);
    d.nverts = p->nverts; d.nv32 = ceil32(p->nverts); d.nedges = p->nedges;
    d.sphere_symm = p->sphere_symm ? 1 : 0;
    d.max_sline_len = p->max_sline_len;
    d.model = p->model_type;
    d.hr = 0; d.hr32 = 0; d.delta_nr = p->delta_nr;
    d.seed_lo = (uint32_t)p->rng_seed; d.seed_hi = (uint32_t)(p->rng_seed >> 32);
    d.tc_threshold = p->tc_threshold;
    d.rel_peak = p->relative_peak_thresh;
    d.cos_max_angle = (float)std::cos((double)p->max_angle);
    d.cos_min_sep = (float)std::cos((double)p->min_separation_angle);
    d.min_signal = p->min_signal;
    d.step_d = (double)p->step_size;
    d.step_frac = (p->model_type == CUSLINES_PTT) ? p->step_frac : 1;
    d.probe_quality = p->probe_quality;
    d.lut_res = p->lut_res;
    d.log2x = p->tile_log2_x; d.log2y = p->tile_log2_y;
    d.nx = 1 << p->tile_log2_x; d.ny = 1 << p->tile_log2_y; d.nz = 1 << p->tile_log2_z;
    d.probe_step = p->probe_step_size;
    d.max_curv = p->max_curvature;
    d.min_support_f = smallest_float_at_least((double)p->probe_quality * PMF_THRESHOLD_P);
    d.ptt_seed_thr_f = smallest_float_at_least(PMF_THRESHOLD_P);
    d.ptt_sub_step = (float)(d.step_d / (double)d.step_frac);
    int brick_log2 = 0;
    e = hipMalloc(&t->d_sort, sort_ints(order_buckets(d, &brick_log2)) * sizeof(int));
    if (e != hipSuccess) {
        dfree(t->d_work);
        (void)hipStreamDestroy(t->stream);
        delete t;
        return fail(CUSLINES_ENOMEM, std::string("seed order: ") + hipGetErrorString(e));
    }
    *out = t;
    return CUSLINES_OK;
}

int cuslines_tracker_destroy(cuslines_tracker *t) {
    if (!t) return CUSLINES_OK;
    if (t->nforks) return fail(CUSLINES_ESTATE, "destroy the tracker's forks first");
    if (t->ngraphs) return fail(CUSLINES_ESTATE, "destroy the tracker's chunk graphs first");
    (void)hipSetDevice(t->device);
    if (t->stream) (void)hipStreamSynchronize(t->stream);
    if (t->parent) {  // a fork owns only its stream, its queue and its counters
        __atomic_fetch_sub(&t->parent->nforks, 1, __ATOMIC_RELAXED);
        dfree(t->d_work);
        dfree(t->d_sort);
        dfree(t->d_stats);
        if (t->stream) (void)hipStreamDestroy(t->stream);
        delete t;
        return CUSLINES_OK;
    }
    dfree(t->d_data); dfree(t->d_stop); dfree(t->d_verts); dfree(t->d_edges); dfree(t->d_nbr);
    dfree(t->d_H); dfree(t->d_R); dfree(t->d_db); dfree(t->d_dq); dfree(t->d_smat);
    dfree(t->d_hrm); dfree(t->d_fitm); dfree(t->d_odfm);
    dfree(t->d_ut); dfree(t->d_u); dfree(t->d_invlev);
    dfree(t->d_b0); dfree(t->d_dwi); dfree(t->d_lut); dfree(t->d_work); dfree(t->d_sort);
    dfree(t->d_blocks);
    dfree(t->d_fprop); dfree(t->d_vprop); dfree(t->d_mlp); dfree(t->d_stats);
    if (t->stream) (void)hipStreamDestroy(t->stream);
    delete t;
    return CUSLINES_OK;
}

int cuslines_tracker_fork(cuslines_tracker *t, cuslines_tracker **out) {
    if (!t || !out) return fail(CUSLINES_EINVAL, "null argument");
    *out = nullptr;
    if (t->parent) return fail(CUSLINES_EINVAL, "fork the parent tracker, not a fork");
    HIPC(hipSetDevice(t->device));
    cuslines_tracker *f = new cuslines_tracker(*t);  // shares every device buffer pointer
    f->parent = t;
    f->nforks = 0;
    f->ngraphs = 0;
    f->stream = nullptr;
    f->d_work = nullptr;
    f->d_sort = nullptr;
    f->d_stats = nullptr;  // learned statistics and tap counts stay with the parent
    f->rec = nullptr;
    f->rec_count = nullptr;
    f->count_taps = 0;
    hipError_t e = hipStreamCreateWithFlags(&f->stream, hipStreamNonBlocking);
    if (e == hipSuccess) e = hipMalloc(&f->d_work, WORK_INTS * sizeof(int));
    int brick_log2 = 0;
    if (e == hipSuccess) e = hipMalloc(&f->d_sort, sort_ints(order_buckets(f->dp, &brick_log2)) * sizeof(int));
    if (e != hipSuccess) {
        dfree(f->d_work);
        dfree(f->d_sort);
        if (f->stream) (void)hipStreamDestroy(f->stream);
        delete f;
        return fail(CUSLINES_EHIP, std::string("tracker fork: ") + hipGetErrorString(e));
    }
    __atomic_fetch_add(&t->nforks, 1, __ATOMIC_RELAXED);
    *out = f;
    return CUSLINES_OK;
}

// PTT corner blocks from the transposed ODF and the LUT's direction ranks
// (both must be present).  Without room for them taps gather their 8 texels.
// The low-rank form of the bootstrap's [H; R] products.  H is the hat
// matrix of the signal basis, a symmetric projection of rank r (the basis
// size): H = U U^T with U (hr x r) orthonormal, and R = lcr(H) =
// L (I - H) - 1 mu^T with L = diag(1 / sqrt(1 - H_ii)) (1 where H_ii >= 1)
// and mu the column means of L (I - H) (boot_utils.py:86-94, DIPY's
// lcr_matrix), so R.d = v - mean(v) with v = L (d - H.d).  U comes from
// Gram-Schmidt (twice, in double) over H's columns; the form is used only
// when U U^T and lcr(H) reproduce the given H and R to 1e-5.  Returns the
// rank (0 when the matrices do not have this form), U row-major [hr][r] and
// the leverage factors.
static int hat_lowrank(const float *H, const float *R, int hr, std::vector<double> &U, std::vector<double> &invlev) {
    std::vector<std::vector<double>> basis;
    double hmax = 0.0;
    for (size_t i = 0; i < (size_t)hr * hr; ++i) hmax = std::max(hmax, std::fabs((double)H[i]));
    if (hmax == 0.0) return 0;
    std::vector<double> v(hr);
    for (int j = 0; j < hr && (int)basis.size() < 64; ++j) {
        double n0 = 0.0;
        for (int i = 0; i < hr; ++i) { v[i] = H[(size_t)i * hr + j]; n0 += v[i] * v[i]; }
        if (n0 == 0.0) continue;
        for (int pass = 0; pass < 2; ++pass)
            for (const auto &u : basis) {
                double dot = 0.0;
                for (int i = 0; i < hr; ++i) dot += u[i] * v[i];
                for (int i = 0; i < hr; ++i) v[i] -= dot * u[i];
            }
        double n = 0.0;
        for (int i = 0; i < hr; ++i) n += v[i] * v[i];
        if (n > 1e-6 * n0 && n > 1e-12) {
            const double inv = 1.0 / std::sqrt(n);
            for (int i = 0; i < hr; ++i) v[i] *= inv;
            basis.push_back(v);
        }
    }
    const int r = (int)basis.size();
    if (r == 0 || r >= hr || r > 64) return 0;
    // A column added late can have a small residual, which the float32
    // rounding of H then dominates: refine the basis twice by U <- orth(H U)
    // (H is a projection, so H U lies in its range and is close to
    // orthonormal; Gram-Schmidt on it amplifies nothing)
    for (int it = 0; it < 2; ++it) {
        std::vector<std::vector<double>> nb;
        for (int k = 0; k < r; ++k) {
            for (int i = 0; i < hr; ++i) {
                double acc = 0.0;
                for (int j = 0; j < hr; ++j) acc += (double)H[(size_t)i * hr + j] * basis[k][j];
                v[i] = acc;
            }
            for (int pass = 0; pass < 2; ++pass)
                for (const auto &u : nb) {
                    double dot = 0.0;
                    for (int i = 0; i < hr; ++i) dot += u[i] * v[i];
                    for (int i = 0; i < hr; ++i) v[i] -= dot * u[i];
                }
            double n = 0.0;
            for (int i = 0; i < hr; ++i) n += v[i] * v[i];
            if (n < 0.25) return 0;  // H U lost a direction: not a projection
            const double inv = 1.0 / std::sqrt(n);
            for (int i = 0; i < hr; ++i) v[i] *= inv;
            nb.push_back(v);
        }
        basis.swap(nb);
    }
    // H = U U^T ?
    for (int i = 0; i < hr; ++i)
        for (int j = 0; j < hr; ++j) {
            double acc = 0.0;
            for (int k = 0; k < r; ++k) acc += basis[k][i] * basis[k][j];
            if (std::fabs(acc - (double)H[(size_t)i * hr + j]) > 1e-5 * hmax) return 0;
        }
    // R = lcr(H) ?
    invlev.assign(hr, 1.0);
    for (int i = 0; i < hr; ++i) {
        const double hii = H[(size_t)i * hr + i];
        if (hii < 1.0) invlev[i] = 1.0 / std::sqrt(1.0 - hii);
    }
    double rmax = 1.0;
    for (size_t i = 0; i < (size_t)hr * hr; ++i) rmax = std::max(rmax, std::fabs((double)R[i]));
    for (int j = 0; j < hr; ++j) {
        double mu = 0.0;
        for (int i = 0; i < hr; ++i) mu += ((i == j ? 1.0 : 0.0) - (double)H[(size_t)i * hr + j]) * invlev[i];
        mu /= hr;
        for (int i = 0; i < hr; ++i) {
            const double lij = ((i == j ? 1.0 : 0.0) - (double)H[(size_t)i * hr + j]) * invlev[i] - mu;
            if (std::fabs(lij - (double)R[(size_t)i * hr + j]) > 1e-5 * rmax) return 0;
        }
    }
    U.assign((size_t)hr * r, 0.0);
    for (int i = 0; i < hr; ++i)
        for (int k = 0; k < r; ++k) U[(size_t)i * r + k] = basis[k][i];
    return r;
}

static int build_blocks(cuslines_tracker *t) {
    const DevParams &d = t->dp;
    dfree(t->d_blocks);
    t->d_blocks = nullptr;
    const long long ncells = (long long)d.nverts * (d.dimx + 1) * (d.dimy + 1) * (d.dimz + 1);
    uint16_t *rv = nullptr;
    HIPC(hipMalloc(&rv, t->rank_vertex.size() * sizeof(uint16_t)));
    hipError_t e = hipMemcpy(rv, t->rank_vertex.data(), t->rank_vertex.size() * sizeof(uint16_t),
                             hipMemcpyHostToDevice);
    if (e == hipSuccess && hipMalloc(&t->d_blocks, (size_t)ncells * 8 * sizeof(float)) == hipSuccess) {
        hipLaunchKernelGGL(build_corner_blocks, dim3((unsigned)((ncells + 255) / 256)), dim3(256), 0, t->stream, d,
                           t->d_data, rv, t->d_blocks, ncells);
        e = hipGetLastError();
        if (e == hipSuccess) e = hipStreamSynchronize(t->stream);
    } else if (e == hipSuccess) {
        (void)hipGetLastError();
        t->d_blocks = nullptr;
    }
    dfree(rv);
    if (e != hipSuccess) return fail(CUSLINES_EHIP, std::string("PTT blocks: ") + hipGetErrorString(e));
    return CUSLINES_OK;
}

// PTT: the [X][Y][Z][T] ODF in device buffer `src` (left unchanged) becomes
// the tracker's vertex-major copy; corner blocks follow when the LUT is set.
static int ptt_take_data(cuslines_tracker *t, const float *src, int nonneg) {
    const DevParams &d = t->dp;
    const size_t nvox = (size_t)d.dimx * d.dimy * d.dimz;
    const size_t bytes = nvox * d.dimt * sizeof(float);
    dfree(t->d_data);
    t->d_data = nullptr;
    t->has_data = false;
    t->dp.ptt_nonneg = nonneg;
    if (hipMalloc(&t->d_data, bytes) != hipSuccess) {
        (void)hipGetLastError();
        t->d_data = nullptr;
        return fail(CUSLINES_ENOMEM, "PTT data allocation failed");
    }
    dim3 grid((unsigned)((nvox + 31) / 32), (unsigned)((d.dimt + 31) / 32));
    hipLaunchKernelGGL(transpose_vox_t, grid, dim3(256), 0, t->stream, src, t->d_data, (long long)nvox, d.dimt);
    hipError_t e = hipGetLastError();
    if (e == hipSuccess) e = hipStreamSynchronize(t->stream);
    if (e != hipSuccess) return fail(CUSLINES_EHIP, std::string("PTT data transpose: ") + hipGetErrorString(e));
    t->has_data = true;
    if (t->has_lut) return build_blocks(t);
    return CUSLINES_OK;
}

int cuslines_set_data(cuslines_tracker *t, const float *dataf) {
    RoctxRange range_("cuslines_set_data");
    if (!t || !dataf) return fail(CUSLINES_EINVAL, "null argument");
    if (int rc = check_owner(t)) return rc;
    HIPC(hipSetDevice(t->device));
    const DevParams &d = t->dp;
    const size_t nvox = (size_t)d.dimx * d.dimy * d.dimz;
    dfree(t->d_data);
    t->d_data = nullptr;
    t->has_data = false;
    if (t->p.model_type == CUSLINES_PTT) {
        // The early stop of rejection-round probes (data_support) relies on
        // taps >= 0; the reference's prepare_data clips the ODF at 0.
        const size_t nval = nvox * (size_t)d.dimt;
        // a NaN counts as negative: a NaN tap makes the full support NaN,
        // which fails the acceptance test, so no early stop may skip it
        const int nonneg = std::none_of(dataf, dataf + nval, [](float v) { return !(v >= 0.0f); }) ? 1 : 0;
        float *tmp = nullptr;
        HIPC(hipMalloc(&tmp, nval * sizeof(float)));
        hipError_t e = hipMemcpy(tmp, dataf, nval * sizeof(float), hipMemcpyHostToDevice);
        if (e != hipSuccess) { dfree(tmp); return fail(CUSLINES_EHIP, std::string("PTT data upload: ") + hipGetErrorString(e)); }
        const int rc = ptt_take_data(t, tmp, nonneg);
        dfree(tmp);
        return rc;
    } else {
        const size_t pitch = (size_t)d.t32 * sizeof(float);
        HIPC(hipMalloc(&t->d_data, nvox * pitch));
        HIPC(hipMemset(t->d_data, 0, nvox * pitch));
        HIPC(hipMemcpy2D(t->d_data, pitch, dataf, (size_t)d.dimt * sizeof(float), (size_t)d.dimt * sizeof(float),
                         nvox, hipMemcpyHostToDevice));
    }
    t->has_data = true;
    return CUSLINES_OK;
}

int cuslines_set_stop_map(cuslines_tracker *t, const float *stop_map) {
    if (!t || !stop_map) return fail(CUSLINES_EINVAL, "null argument");
    if (int rc = check_owner(t)) return rc;
    HIPC(hipSetDevice(t->device));
    const size_t n = (size_t)t->dp.dimx * t->dp.dimy * t->dp.dimz;
    // A failed re-upload must not leave the tracker ready with freed buffers.
    t->has_stop = false;
    dfree(t->d_stop);
    t->d_stop = nullptr;
    HIPC(hipMalloc(&t->d_stop, n * sizeof(float)));
    HIPC(hipMemcpy(t->d_stop, stop_map, n * sizeof(float), hipMemcpyHostToDevice));
    t->has_stop = true;
    return CUSLINES_OK;
}

int cuslines_set_sphere(cuslines_tracker *t, const float *vertices, const int32_t *edges) {
    if (!t || !vertices || !edges) return fail(CUSLINES_EINVAL, "null argument");
    if (int rc = check_owner(t)) return rc;
    HIPC(hipSetDevice(t->device));
    const int nv = t->dp.nverts, ne = t->dp.nedges;
    std::vector<uint32_t> packed(ne);
    for (int e = 0; e < ne; ++e) {
        const int u = edges[2 * e], v = edges[2 * e + 1];
        if (u < 0 || u >= nv || v < 0 || v >= nv) return fail(CUSLINES_EINVAL, "edge vertex index out of range");
        packed[e] = (uint32_t)u | ((uint32_t)v << 16);
    }
    t->has_sphere = false;
    dfree(t->d_verts); dfree(t->d_edges); dfree(t->d_nbr);
    t->d_verts = nullptr; t->d_edges = nullptr; t->d_nbr = nullptr;
    HIPC(hipMalloc(&t->d_verts, (size_t)nv * 3 * sizeof(float)));
    HIPC(hipMemcpy(t->d_verts, vertices, (size_t)nv * 3 * sizeof(float), hipMemcpyHostToDevice));
    HIPC(hipMalloc(&t->d_edges, (size_t)ne * sizeof(uint32_t)));
    HIPC(hipMemcpy(t->d_edges, packed.data(), (size_t)ne * sizeof(uint32_t), hipMemcpyHostToDevice));
    // Adjacency for the peak test (peak_directions): up to 8 distinct
    // neighbours per vertex, the rest of the row the vertex itself.
    std::vector<uint16_t> nbr((size_t)nv * 8);
    std::vector<int> deg(nv, 0);
    bool fits = nv <= 1024;
    for (int v = 0; v < nv; ++v)
        for (int k = 0; k < 8; ++k) nbr[(size_t)v * 8 + k] = (uint16_t)v;
    for (int e = 0; e < ne && fits; ++e) {
        const int a = edges[2 * e], b = edges[2 * e + 1];
        for (int side = 0; side < 2 && fits; ++side) {
            const int x = side ? b : a, y = side ? a : b;
            bool seen = false;
            for (int k = 0; k < deg[x]; ++k) seen = seen || nbr[(size_t)x * 8 + k] == y;
            if (seen) continue;
            if (deg[x] == 8) { fits = false; break; }
            nbr[(size_t)x * 8 + deg[x]++] = (uint16_t)y;
        }
    }
    if (fits) {
        HIPC(hipMalloc(&t->d_nbr, nbr.size() * sizeof(uint16_t)));
        HIPC(hipMemcpy(t->d_nbr, nbr.data(), nbr.size() * sizeof(uint16_t), hipMemcpyHostToDevice));
    }
    t->has_sphere = true;
    return CUSLINES_OK;
}

int cuslines_set_boot_matrices(cuslines_tracker *t, const float *H, const float *R, const float *delta_b,
                               const float *delta_q, const float *sampling_matrix, const int32_t *b0s_mask) {
    if (!t || !H || !R || !delta_b || !delta_q || !sampling_matrix || !b0s_mask)
        return fail(CUSLINES_EINVAL, "null argument");
    if (int rc = check_owner(t)) return rc;
    if (t->p.model_type != CUSLINES_OPDT && t->p.model_type != CUSLINES_CSA)
        return fail(CUSLINES_ESTATE, "bootstrap matrices need an OPDT or CSA tracker");
    HIPC(hipSetDevice(t->device));
    const int T = t->dp.dimt, dn = t->dp.delta_nr, nv = t->dp.nverts;
    std::vector<int> b0(T), dwi;
    int nb0 = 0;
    for (int j = 0; j < T; ++j) {
        b0[j] = b0s_mask[j] ? 1 : 0;
        if (b0[j]) ++nb0; else dwi.push_back(j);
    }
    const int hr = (int)dwi.size();
    if (hr == 0 || nb0 == 0) return fail(CUSLINES_EINVAL, "bootstrap needs at least one b0 and one DWI volume");
    t->has_boot = false;
    t->dp.hr = hr;
    t->dp.hr32 = ceil32(hr);
    float **dst[5] = {&t->d_H, &t->d_R, &t->d_db, &t->d_dq, &t->d_smat};
    const float *src[5] = {H, R, delta_b, delta_q, sampling_matrix};
    const int rows[5] = {hr, hr, dn, dn, nv}, cols[5] = {hr, hr, hr, hr, dn};
    for (int k = 0; k < 5; ++k) {
        // gemv_lanerow's layout: lane-interleaved when the row length is a
        // multiple of 4 (rows padded to a multiple of 32 with zeros), else row-major
        const int N = rows[k], M = cols[k];
        std::vector<float> h;
        if ((M & 3) == 0) {
            h.assign((size_t)ceil32(N) * M, 0.0f);
            for (int i = 0; i < N; ++i)
                for (int j = 0; j < M; ++j) h[mat_offset(M, i, j)] = src[k][(size_t)i * M + j];
        } else {
            h.assign(src[k], src[k] + (size_t)N * M);
        }
        dfree(*dst[k]);
        *dst[k] = nullptr;
        HIPC(hipMalloc(dst[k], h.size() * sizeof(float)));
        HIPC(hipMemcpy(*dst[k], h.data(), h.size() * sizeof(float), hipMemcpyHostToDevice));
    }
    // the batched kernel's zero-padded row-major copies: [H; R] [2 hr16][hr16],
    // [dq | -db] [dn16][2 hr16], sampling matrix [nv16][dn16]
    {
        const int hr16 = (hr + 15) & ~15, dn16 = (dn + 15) & ~15, nv16 = (nv + 15) & ~15;
        t->dp.hr16 = hr16; t->dp.dn16 = dn16; t->dp.nv16 = nv16;
        std::vector<float> hrm((size_t)2 * hr16 * hr16, 0.0f), fit((size_t)dn16 * 2 * hr16, 0.0f),
            odf((size_t)nv16 * dn16, 0.0f);
        for (int i = 0; i < hr; ++i)
            for (int j = 0; j < hr; ++j) {
                hrm[(size_t)i * hr16 + j] = H[(size_t)i * hr + j];
                hrm[(size_t)(hr16 + i) * hr16 + j] = R[(size_t)i * hr + j];
            }
        for (int i = 0; i < dn; ++i)
            for (int j = 0; j < hr; ++j) {
                fit[(size_t)i * 2 * hr16 + j] = delta_q[(size_t)i * hr + j];
                fit[(size_t)i * 2 * hr16 + hr16 + j] = -delta_b[(size_t)i * hr + j];
            }
        for (int i = 0; i < nv; ++i)
            for (int j = 0; j < dn; ++j) odf[(size_t)i * dn16 + j] = sampling_matrix[(size_t)i * dn + j];
        // low-rank form: U^T [rk16][hr16], U [hr16][rk16], 1/lev [hr16], zero padded
        std::vector<double> U, invlev;
        const int r = hat_lowrank(H, R, hr, U, invlev);
        const int rk16 = (r + 15) & ~15;
        std::vector<float> ut((size_t)std::max(rk16, 16) * hr16, 0.0f), um((size_t)hr16 * std::max(rk16, 16), 0.0f),
            il((size_t)hr16, 0.0f);
        for (int i = 0; i < hr && r > 0; ++i) {
            for (int k = 0; k < r; ++k) {
                ut[(size_t)k * hr16 + i] = (float)U[(size_t)i * r + k];
                um[(size_t)i * rk16 + k] = (float)U[(size_t)i * r + k];
            }
            il[i] = (float)invlev[i];
        }
        t->rk16 = r > 0 ? rk16 : 0;
        t->hrank = r;
        float **bdst[6] = {&t->d_hrm, &t->d_fitm, &t->d_odfm, &t->d_ut, &t->d_u, &t->d_invlev};
        const std::vector<float> *bsrc[6] = {&hrm, &fit, &odf, &ut, &um, &il};
        for (int k = 0; k < 6; ++k) {
            dfree(*bdst[k]);
            *bdst[k] = nullptr;
            HIPC(hipMalloc(bdst[k], bsrc[k]->size() * sizeof(float)));
            HIPC(hipMemcpy(*bdst[k], bsrc[k]->data(), bsrc[k]->size() * sizeof(float), hipMemcpyHostToDevice));
        }
    }
    dfree(t->d_b0); dfree(t->d_dwi);
    t->d_b0 = nullptr; t->d_dwi = nullptr;
    HIPC(hipMalloc(&t->d_b0, (size_t)T * sizeof(int)));
    HIPC(hipMemcpy(t->d_b0, b0.data(), (size_t)T * sizeof(int), hipMemcpyHostToDevice));
    HIPC(hipMalloc(&t->d_dwi, (size_t)hr * sizeof(int)));
    HIPC(hipMemcpy(t->d_dwi, dwi.data(), (size_t)hr * sizeof(int), hipMemcpyHostToDevice));
    t->has_boot = true;
    return CUSLINES_OK;
}

int cuslines_set_ptt_lut(cuslines_tracker *t, const int32_t *lut) {
    if (!t || !lut) return fail(CUSLINES_EINVAL, "null argument");
    if (int rc = check_owner(t)) return rc;
    if (t->p.model_type != CUSLINES_PTT) return fail(CUSLINES_ESTATE, "LUT needs a PTT tracker");
    HIPC(hipSetDevice(t->device));
    const size_t r = (size_t)t->dp.lut_res;
    const int nv = t->dp.nverts;
    std::vector<uint32_t> h(r * r * r);
    // Direction ranks: vertices numbered in the order they first appear along
    // a Morton traversal of the LUT grid, so consecutive ranks are
    // neighbouring directions; the corner blocks of a cell are stored in this
    // order (tap_sample).
    std::vector<int> rank(nv, -1);
    std::vector<uint16_t> rank_vertex;
    rank_vertex.reserve(nv);
    {
        int bits = 0;
        while ((size_t(1) << bits) < r) ++bits;
        const uint64_t ncode = uint64_t(1) << (3 * bits);
        for (uint64_t c = 0; c < ncode; ++c) {
            uint64_t a[3] = {0, 0, 0};
            for (int b = 0; b < bits; ++b)
                for (int k = 0; k < 3; ++k) a[k] |= ((c >> (3 * b + 2 - k)) & 1u) << b;
            if (a[0] >= r || a[1] >= r || a[2] >= r) continue;
            const int32_t v = lut[(a[0] * r + a[1]) * r + a[2]];
            if (v < 0 || v >= nv) return fail(CUSLINES_EINVAL, "LUT vertex index out of range");
            if (rank[v] < 0) { rank[v] = (int)rank_vertex.size(); rank_vertex.push_back((uint16_t)v); }
        }
        for (int v = 0; v < nv; ++v)
            if (rank[v] < 0) { rank[v] = (int)rank_vertex.size(); rank_vertex.push_back((uint16_t)v); }
    }
    // Unit directions touch a thin shell of the cube: with res % 4 == 0 the
    // table is stored as 4x4x4 bricks of 128 bytes (one cache line), so the
    // shell spans ~10x fewer lines than with rows along the last axis.
    const bool brick = (r % 4) == 0;
    const size_t nb = r / 4;
    for (size_t i0 = 0; i0 < r; ++i0)
        for (size_t i1 = 0; i1 < r; ++i1)
            for (size_t i2 = 0; i2 < r; ++i2) {
                const int32_t v = lut[(i0 * r + i1) * r + i2];
                const size_t dst = brick ? (((i0 >> 2) * nb + (i1 >> 2)) * nb + (i2 >> 2)) * 64 +
                                               ((i0 & 3) << 4) + ((i1 & 3) << 2) + (i2 & 3)
                                         : (i0 * r + i1) * r + i2;
                h[dst] = (uint32_t)v | ((uint32_t)rank[v] << 16);
            }
    t->has_lut = false;
    t->dp.lut_brick = brick ? 1 : 0;
    dfree(t->d_lut);
    t->d_lut = nullptr;
    HIPC(hipMalloc(&t->d_lut, h.size() * sizeof(uint32_t)));
    HIPC(hipMemcpy(t->d_lut, h.data(), h.size() * sizeof(uint32_t), hipMemcpyHostToDevice));
    t->rank_vertex.swap(rank_vertex);
    if (!t->d_vprop) {
        HIPC(hipMalloc(&t->d_vprop, VPROP_FLOATS * sizeof(float)));
        hipLaunchKernelGGL(feature_propagators, dim3(1), dim3(32), 0, t->stream, t->dp, 1, t->d_vprop);
        HIPC(hipGetLastError());
        HIPC(hipStreamSynchronize(t->stream));
    }
    t->has_lut = true;
    if (t->has_data) return build_blocks(t);
    return CUSLINES_OK;
}

int cuslines_device_alloc(cuslines_tracker *t, size_t bytes, void **dptr) {
    if (!t || !dptr) return fail(CUSLINES_EINVAL, "null argument");
    HIPC(hipSetDevice(t->device));
    *dptr = nullptr;
    if (bytes == 0) bytes = 4;
    hipError_t e = hipMalloc(dptr, bytes);
    if (e != hipSuccess) return fail(CUSLINES_ENOMEM, std::string("hipMalloc: ") + hipGetErrorString(e));
    return CUSLINES_OK;
}

int cuslines_device_free(cuslines_tracker *t, void *dptr) {
    if (!t) return fail(CUSLINES_EINVAL, "null tracker");
    HIPC(hipSetDevice(t->device));
    if (dptr) HIPC(hipFree(dptr));
    return CUSLINES_OK;
}

int cuslines_memcpy_htod(cuslines_tracker *t, void *dst, const void *src, size_t bytes) {
    if (!t || (bytes && (!dst || !src))) return fail(CUSLINES_EINVAL, "null argument");
    HIPC(hipSetDevice(t->device));
    if (bytes) HIPC(hipMemcpyAsync(dst, src, bytes, hipMemcpyHostToDevice, t->stream));
    HIPC(hipStreamSynchronize(t->stream));
    return CUSLINES_OK;
}

int cuslines_memcpy_dtoh(cuslines_tracker *t, void *dst, const void *src, size_t bytes) {
    if (!t || (bytes && (!dst || !src))) return fail(CUSLINES_EINVAL, "null argument");
    HIPC(hipSetDevice(t->device));
    if (bytes) HIPC(hipMemcpyAsync(dst, src, bytes, hipMemcpyDeviceToHost, t->stream));
    HIPC(hipStreamSynchronize(t->stream));
    return CUSLINES_OK;
}

int cuslines_synchronize(cuslines_tracker *t) {
    if (!t) return fail(CUSLINES_EINVAL, "null tracker");
    HIPC(hipSetDevice(t->device));
    HIPC(hipStreamSynchronize(t->stream));
    return CUSLINES_OK;
}

int cuslines_set_launch(cuslines_tracker *t, int schedule, int threads, int blocks_per_cu) {
    if (!t) return fail(CUSLINES_EINVAL, "null tracker");
    if (schedule != CUSLINES_SCHED_QUEUE && schedule != CUSLINES_SCHED_STATIC)
        return fail(CUSLINES_EINVAL, "unknown schedule");
    if (threads != 0 && (threads < 64 || threads > 256 || threads % 64 != 0))
        return fail(CUSLINES_EINVAL, "threads per block must be 0 or a multiple of 64 in [64, 256]");
    if (blocks_per_cu < 0) return fail(CUSLINES_EINVAL, "blocks_per_cu must be >= 0");
    t->schedule = schedule;
    t->threads = threads;
    t->blocks_per_cu = blocks_per_cu;
    return CUSLINES_OK;
}

int cuslines_set_boot_mode(cuslines_tracker *t, int mode) {
    if (!t) return fail(CUSLINES_EINVAL, "null tracker");
    if (t->p.model_type != CUSLINES_OPDT && t->p.model_type != CUSLINES_CSA)
        return fail(CUSLINES_EINVAL, "the bootstrap mode is for OPDT and CSA trackers");
    if ((mode & 0xff) != CUSLINES_BOOT_EXACT && (mode & 0xff) != CUSLINES_BOOT_MFMA)
        return fail(CUSLINES_EINVAL, "unknown mode");
    const int occ = (mode >> 8) & 0xff;
    if (occ != 0 && occ != 2 && occ != 4) return fail(CUSLINES_EINVAL, "waves per SIMD must be 2 or 4");
    if ((mode & ~(0xffff | CUSLINES_BOOT_FULL_PRODUCTS)) != 0) return fail(CUSLINES_EINVAL, "unknown mode flag");
    t->boot_mode = mode & 0xff;
    t->boot_occ = occ;
    t->boot_full = (mode & CUSLINES_BOOT_FULL_PRODUCTS) ? 1 : 0;
    return CUSLINES_OK;
}

int cuslines_hat_lowrank(const float *H, const float *R, int32_t hr, int32_t *rank) {
    if (!H || !R || !rank) return fail(CUSLINES_EINVAL, "null argument");
    if (hr < 1) return fail(CUSLINES_EINVAL, "hr must be positive");
    std::vector<double> U, invlev;
    *rank = hat_lowrank(H, R, hr, U, invlev);
    return CUSLINES_OK;
}

int cuslines_boot_lowrank(cuslines_tracker *t, int32_t *rank) {
    if (!t || !rank) return fail(CUSLINES_EINVAL, "null argument");
    *rank = (t->has_boot && !t->boot_full) ? t->hrank : 0;
    return CUSLINES_OK;
}

int cuslines_boot_waves(cuslines_tracker *t, int32_t nseeds, int32_t *waves) {
    if (!t || !waves) return fail(CUSLINES_EINVAL, "null argument");
    if (nseeds < 0) return fail(CUSLINES_EINVAL, "negative size");
    if (t->p.model_type != CUSLINES_OPDT && t->p.model_type != CUSLINES_CSA)
        return fail(CUSLINES_EINVAL, "bootstrap variants are for OPDT and CSA trackers");
    *waves = boot_waves(t, nseeds);
    return CUSLINES_OK;
}

int cuslines_set_stepping(cuslines_tracker *t, int flat) {
    if (!t) return fail(CUSLINES_EINVAL, "null tracker");
    if (flat != 0 && flat != 1) return fail(CUSLINES_EINVAL, "stepping must be 0 (per seed) or 1 (flat)");
    t->flat = flat;
    return CUSLINES_OK;
}

int cuslines_set_lanes_per_seed(cuslines_tracker *t, int lanes) {
    if (!t) return fail(CUSLINES_EINVAL, "null tracker");
    if (lanes != 0 && lanes != 8 && lanes != 16 && lanes != 32)
        return fail(CUSLINES_EINVAL, "lanes per seed must be 0, 8, 16 or 32");
    t->ptt_lanes = lanes;
    return CUSLINES_OK;
}

int cuslines_ptt_prepare(cuslines_tracker *t, const float *odf, const float *stop_map, float stop_threshold,
                         int sphere_symm, int32_t *lut_out) {
    RoctxRange range_("cuslines_ptt_prepare");
    if (!t || !odf || !stop_map) return fail(CUSLINES_EINVAL, "null argument");
    if (int rc = check_owner(t)) return rc;
    if (t->p.model_type != CUSLINES_PTT) return fail(CUSLINES_ESTATE, "PTT preparation needs a PTT tracker");
    if (!t->has_sphere) return fail(CUSLINES_ESTATE, "upload the sphere before preparing PTT data");
    if (t->dp.lut_res < 2) return fail(CUSLINES_EINVAL, "lut_res must be at least 2");
    HIPC(hipSetDevice(t->device));
    const DevParams &d = t->dp;
    const size_t nvox = (size_t)d.dimx * d.dimy * d.dimz;
    const size_t nval = nvox * (size_t)d.dimt;
    const size_t nlut = (size_t)d.lut_res * d.lut_res * d.lut_res;
    float *raw = nullptr, *stop = nullptr;
    int32_t *lut = nullptr;
    hipError_t e = hipMalloc(&raw, nval * sizeof(float));
    if (e == hipSuccess) e = hipMalloc(&stop, nvox * sizeof(float));
    if (e == hipSuccess) e = hipMalloc(&lut, nlut * sizeof(int32_t));
    if (e == hipSuccess) e = hipMemcpy(raw, odf, nval * sizeof(float), hipMemcpyHostToDevice);
    if (e == hipSuccess) e = hipMemcpy(stop, stop_map, nvox * sizeof(float), hipMemcpyHostToDevice);
    if (e == hipSuccess) {
        hipLaunchKernelGGL(ptt_normalise, dim3((unsigned)((nvox + 255) / 256)), dim3(256), 0, t->stream, raw, stop,
                           stop_threshold, (long long)nvox, d.dimt);
        hipLaunchKernelGGL(ptt_lut_kernel, dim3((unsigned)((nlut + 255) / 256)), dim3(256), 0, t->stream, t->d_verts,
                           d.nverts, d.lut_res, sphere_symm ? 1 : 0, lut);
        e = hipGetLastError();
    }
    if (e == hipSuccess) e = hipStreamSynchronize(t->stream);
    std::vector<int32_t> hl(nlut);
    if (e == hipSuccess) e = hipMemcpy(hl.data(), lut, nlut * sizeof(int32_t), hipMemcpyDeviceToHost);
    dfree(stop);
    dfree(lut);
    if (e != hipSuccess) {
        dfree(raw);
        return fail(CUSLINES_EHIP, std::string("PTT preparation: ") + hipGetErrorString(e));
    }
    // the clipped ODF has no negative value, but NaN inputs stay NaN
    int nonneg = 0;
    {
        int *flag = nullptr;
        e = hipMalloc(&flag, sizeof(int));
        if (e == hipSuccess) e = hipMemsetAsync(flag, 0, sizeof(int), t->stream);
        if (e == hipSuccess) {
            const size_t nb = std::min<size_t>((nval + 255) / 256, 65536);
            hipLaunchKernelGGL(flag_not_nonneg, dim3((unsigned)nb), dim3(256), 0, t->stream, raw, (long long)nval, flag);
            e = hipGetLastError();
        }
        int hf = 1;
        if (e == hipSuccess) e = hipMemcpyAsync(&hf, flag, sizeof(int), hipMemcpyDeviceToHost, t->stream);
        if (e == hipSuccess) e = hipStreamSynchronize(t->stream);
        dfree(flag);
        if (e != hipSuccess) {
            dfree(raw);
            return fail(CUSLINES_EHIP, std::string("PTT preparation: ") + hipGetErrorString(e));
        }
        nonneg = hf ? 0 : 1;
    }
    int rc = ptt_take_data(t, raw, nonneg);
    dfree(raw);
    if (rc) return rc;
    rc = cuslines_set_ptt_lut(t, hl.data());
    if (rc) return rc;
    if (lut_out) std::memcpy(lut_out, hl.data(), nlut * sizeof(int32_t));
    return CUSLINES_OK;
}

int cuslines_set_ptt_layout(cuslines_tracker *t, int corner_blocks) {
    if (!t) return fail(CUSLINES_EINVAL, "null tracker");
    if (int rc = check_owner(t)) return rc;
    t->use_blocks = corner_blocks ? 1 : 0;
    return CUSLINES_OK;
}

static int ensure_feature_propagators(cuslines_tracker *t) {
    if (t->d_fprop) return CUSLINES_OK;
    HIPC(hipMalloc(&t->d_fprop, DISC_VERT_CNT * 9 * sizeof(float)));
    hipLaunchKernelGGL(feature_propagators, dim3(1), dim3(32), 0, t->stream, t->dp, FEAT_STEPS, t->d_fprop);
    HIPC(hipGetLastError());
    HIPC(hipStreamSynchronize(t->stream));
    return CUSLINES_OK;
}

int cuslines_set_proposal(cuslines_tracker *t, const uint16_t *mlp_bf16) {
    if (!t) return fail(CUSLINES_EINVAL, "null tracker");
    if (int rc = check_owner(t)) return rc;
    HIPC(hipSetDevice(t->device));
    if (!mlp_bf16) {
        dfree(t->d_mlp);
        t->d_mlp = nullptr;
        return CUSLINES_OK;
    }
    if (t->p.model_type != CUSLINES_PTT) return fail(CUSLINES_EINVAL, "the learned proposal is for PTT");
    if (int rc = ensure_feature_propagators(t)) return rc;
    std::vector<uint16_t> il(IL_NPARAM, 0);
    auto put = [&](int dst, int src, int N, int K) {
        for (int j = 0; j < N; ++j)
            for (int k = 0; k < K; ++k) il[dst + mlp_il_offset(K, j, k)] = mlp_bf16[src + j * K + k];
    };
    put(IL_W1, MLP_W1, MLP_H, MLP_IN);
    put(IL_W2, MLP_W2, MLP_H, MLP_H);
    put(IL_W3, MLP_W3, MLP_OUT, MLP_H);
    for (int j = 0; j < MLP_H; ++j) { il[IL_B1 + j] = mlp_bf16[MLP_B1 + j]; il[IL_B2 + j] = mlp_bf16[MLP_B2 + j]; }
    for (int j = 0; j < MLP_OUT; ++j) il[IL_B3 + j] = mlp_bf16[MLP_B3 + j];
    if (!t->d_mlp) HIPC(hipMalloc(&t->d_mlp, IL_NPARAM * sizeof(uint16_t)));
    HIPC(hipMemcpy(t->d_mlp, il.data(), IL_NPARAM * sizeof(uint16_t), hipMemcpyHostToDevice));
    if (!t->d_stats) {
        HIPC(hipMalloc(&t->d_stats, 4 * sizeof(unsigned long long)));
        HIPC(hipMemset(t->d_stats, 0, 4 * sizeof(unsigned long long)));
    }
    return CUSLINES_OK;
}

int cuslines_set_recording(cuslines_tracker *t, float *pairs_d, int32_t capacity, int32_t *count_d, float rate) {
    if (!t) return fail(CUSLINES_EINVAL, "null tracker");
    if (int rc = check_owner(t)) return rc;
    if (!pairs_d) {
        t->rec = nullptr;
        t->rec_count = nullptr;
        return CUSLINES_OK;
    }
    if (!count_d || capacity <= 0 || !(rate > 0.0f && rate <= 1.0f))
        return fail(CUSLINES_EINVAL, "recording needs count_d, capacity > 0 and 0 < rate <= 1");
    if (t->p.model_type != CUSLINES_PTT) return fail(CUSLINES_EINVAL, "recording is for PTT");
    if (int rc = ensure_feature_propagators(t)) return rc;
    t->rec = pairs_d;
    t->rec_count = count_d;
    t->dp.rec_cap = capacity;
    const double th = (double)rate * 4294967296.0;
    t->dp.rec_thresh = (th >= 4294967295.0) ? 0xffffffffu : (uint32_t)th;
    return CUSLINES_OK;
}

int cuslines_proposal_stats(cuslines_tracker *t, int64_t *out3, int reset) {
    if (!t || !out3) return fail(CUSLINES_EINVAL, "null argument");
    HIPC(hipSetDevice(t->device));
    unsigned long long h[4] = {0, 0, 0, 0};
    if (t->d_stats) {
        HIPC(hipStreamSynchronize(t->stream));
        HIPC(hipMemcpy(h, t->d_stats, sizeof(h), hipMemcpyDeviceToHost));
        if (reset) HIPC(hipMemset(t->d_stats, 0, sizeof(h)));
    }
    for (int i = 0; i < 3; ++i) out3[i] = (int64_t)h[i];
    return CUSLINES_OK;
}

int cuslines_proposal_counters(cuslines_tracker *t, int64_t *out4, int reset) {
    if (!t || !out4) return fail(CUSLINES_EINVAL, "null argument");
    HIPC(hipSetDevice(t->device));
    unsigned long long h[4] = {0, 0, 0, 0};
    if (t->d_stats) {
        HIPC(hipStreamSynchronize(t->stream));
        HIPC(hipMemcpy(h, t->d_stats, sizeof(h), hipMemcpyDeviceToHost));
        if (reset) HIPC(hipMemset(t->d_stats, 0, sizeof(h)));
    }
    for (int i = 0; i < 4; ++i) out4[i] = (int64_t)h[i];
    return CUSLINES_OK;
}

int cuslines_boot_counters(cuslines_tracker *t, int64_t *out2, int reset) {
    if (!t || !out2) return fail(CUSLINES_EINVAL, "null argument");
    if (t->p.model_type != CUSLINES_OPDT && t->p.model_type != CUSLINES_CSA)
        return fail(CUSLINES_EINVAL, "bootstrap counters are for OPDT and CSA trackers");
    HIPC(hipSetDevice(t->device));
    unsigned long long h[4] = {0, 0, 0, 0};
    if (t->d_stats) {
        HIPC(hipStreamSynchronize(t->stream));
        HIPC(hipMemcpy(h, t->d_stats, sizeof(h), hipMemcpyDeviceToHost));
        if (reset) HIPC(hipMemset(t->d_stats, 0, sizeof(h)));
    }
    out2[0] = (int64_t)h[0];
    out2[1] = (int64_t)h[1];
    return CUSLINES_OK;
}

int cuslines_set_tap_count(cuslines_tracker *t, int enable) {
    if (!t) return fail(CUSLINES_EINVAL, "null tracker");
    if (t->p.model_type != CUSLINES_PTT) return fail(CUSLINES_EINVAL, "tap counting is for PTT");
    // Switched off: the instrumented phase-2 kernel stopped responding on
    // its first GPU run (48 seeds, 32x36x30 phantom) and the cause has not
    // been found, so it is never launched.
    if (enable) return fail(CUSLINES_ESTATE, "the instrumented PTT kernel (tap counting) is switched off");
    HIPC(hipSetDevice(t->device));
    if (enable && !t->d_stats) {
        HIPC(hipMalloc(&t->d_stats, 4 * sizeof(unsigned long long)));
        HIPC(hipMemset(t->d_stats, 0, 4 * sizeof(unsigned long long)));
    }
    t->count_taps = enable ? 1 : 0;
    return CUSLINES_OK;
}

int cuslines_tap_count(cuslines_tracker *t, int64_t *out2, int reset) {
    if (!t || !out2) return fail(CUSLINES_EINVAL, "null argument");
    if (t->d_mlp) return fail(CUSLINES_ESTATE, "the counters hold the learned proposal's statistics");
    HIPC(hipSetDevice(t->device));
    unsigned long long h[4] = {0, 0, 0, 0};
    if (t->d_stats) {
        HIPC(hipStreamSynchronize(t->stream));
        HIPC(hipMemcpy(h, t->d_stats, sizeof(h), hipMemcpyDeviceToHost));
        if (reset) HIPC(hipMemset(t->d_stats, 0, sizeof(h)));
    }
    out2[0] = (int64_t)h[0];
    out2[1] = (int64_t)h[1];
    return CUSLINES_OK;
}

// Floats of the caller's workspace: 561 a pair and 16,512 for every 128 pairs.
static size_t mlp_ws_floats(int n) {
    return (size_t)n * (4 * MLP_H + 2 * MLP_OUT + 1) + ((size_t)n + 127) / 128 * MLP_H * (MLP_H + 1);
}

// Workgroups of the training kernel: one per tile of pairs, up to one per CU
// and as many as the workspace has room for (105 at 4096 pairs); a lone one
// writes the gradient itself.
static int mlp_groups(int n) {
    const size_t room = std::max<size_t>(1, mlp_ws_floats(n) / MLP_PART);
    return (int)std::min<size_t>(room, (size_t)std::min((n + MLP_TILE - 1) / MLP_TILE, MLP_GROUPS));
}

constexpr int MLP_MAX_PAIRS = 65535 * 128;

int cuslines_mlp_workspace_bytes(int32_t n, size_t *bytes) {
    if (!bytes || n <= 0) return fail(CUSLINES_EINVAL, "n > 0 and bytes required");
    if (n > MLP_MAX_PAIRS) return fail(CUSLINES_EINVAL, "at most 8,388,480 pairs per training call");
    *bytes = mlp_ws_floats(n) * sizeof(float);
    return CUSLINES_OK;
}

int cuslines_mlp_loss_grad_async(cuslines_tracker *t, const float *params_d, const float *pairs_d, int32_t n,
                                 float *loss_d, float *grad_d, void *work_d) {
    if (!t || !params_d || !pairs_d || !loss_d || !grad_d || !work_d || n <= 0)
        return fail(CUSLINES_EINVAL, "null argument or n <= 0");
    if (n > MLP_MAX_PAIRS) return fail(CUSLINES_EINVAL, "at most 8,388,480 pairs per training call");
    HIPC(hipSetDevice(t->device));
    float *part = static_cast<float *>(work_d);
    const int groups = mlp_groups(n);
    hipLaunchKernelGGL(mlp_train_kernel, dim3((unsigned)groups), dim3(MLP_THREADS), 0, t->stream, params_d, pairs_d, n,
                       part, grad_d, loss_d);
    if (groups > 1)
        hipLaunchKernelGGL(mlp_sum_kernel, dim3(MLP_PART_LOSS / MLP_SUM_COLS + 1), dim3(256), 0, t->stream, part,
                           groups, n, grad_d, loss_d);
    HIPC(hipGetLastError());
    return CUSLINES_OK;
}

int cuslines_mlp_adam_async(cuslines_tracker *t, float *params_d, const float *grad_d, float *m_d, float *v_d,
                            int32_t step, float lr, float beta1, float beta2, float eps) {
    if (!t || !params_d || !grad_d || !m_d || !v_d || step < 1) return fail(CUSLINES_EINVAL, "bad Adam arguments");
    HIPC(hipSetDevice(t->device));
    const float c1 = (float)(1.0 - std::pow((double)beta1, (double)step));
    const float c2 = (float)(1.0 - std::pow((double)beta2, (double)step));
    hipLaunchKernelGGL(adam_kernel, dim3((MLP_NPARAM + 255) / 256), dim3(256), 0, t->stream, params_d, grad_d, m_d,
                       v_d, MLP_NPARAM, lr, beta1, beta2, eps, c1, c2);
    HIPC(hipGetLastError());
    return CUSLINES_OK;
}

int cuslines_get_stream(cuslines_tracker *t, void **stream) {
    if (!t || !stream) return fail(CUSLINES_EINVAL, "null argument");
    *stream = (void *)t->stream;
    return CUSLINES_OK;
}

int cuslines_phase1_async(cuslines_tracker *t, const float *seeds_d, int32_t nseeds, int32_t rng_chunk,
                          int32_t *counts_d, int32_t *dirs_d) {
    RoctxRange range_("cuslines_phase1");
    if (!t) return fail(CUSLINES_EINVAL, "null tracker");
    if (nseeds < 0 || rng_chunk < 0) return fail(CUSLINES_EINVAL, "negative size");
    if (nseeds == 0) return CUSLINES_OK;
    if (!seeds_d || !counts_d || !dirs_d) return fail(CUSLINES_EINVAL, "null buffer");
    int rc = check_ready(t);
    if (rc) return rc;
    HIPC(hipSetDevice(t->device));
    return phase1_models(t, seeds_d, nseeds, rng_chunk > 0 ? rng_chunk : nseeds, counts_d, dirs_d);
}

int cuslines_scan_async(cuslines_tracker *t, const int32_t *counts_d, int32_t nseeds, int32_t *offsets_d) {
    RoctxRange range_("cuslines_scan");
    if (!t || !offsets_d || (nseeds > 0 && !counts_d)) return fail(CUSLINES_EINVAL, "null argument");
    if (nseeds < 0) return fail(CUSLINES_EINVAL, "negative size");
    HIPC(hipSetDevice(t->device));
    return run_scan<int>(t, counts_d, nseeds, offsets_d);
}

int cuslines_phase2_async(cuslines_tracker *t, const float *seeds_d, int32_t nseeds, int32_t rng_chunk,
                          const int32_t *offsets_d, const int32_t *dirs_d, int32_t *sline_seed_d,
                          int32_t *sline_len_d, float *sline_d) {
    return phase2_entry(t, seeds_d, nseeds, rng_chunk, offsets_d, dirs_d, sline_seed_d, sline_len_d, sline_d, false);
}

int cuslines_phase2_noalloc_async(cuslines_tracker *t, const float *seeds_d, int32_t nseeds, int32_t rng_chunk,
                                  const int32_t *offsets_d, const int32_t *dirs_d, int32_t *sline_seed_d,
                                  int32_t *sline_len_d, float *sline_d) {
    return phase2_entry(t, seeds_d, nseeds, rng_chunk, offsets_d, dirs_d, sline_seed_d, sline_len_d, sline_d, true);
}

int cuslines_compact_async(cuslines_tracker *t, const int32_t *sline_len_d, int32_t nslines, const float *sline_d,
                           int64_t *point_off_d, float *points_d) {
    RoctxRange range_("cuslines_compact");
    if (!t || !point_off_d || (nslines > 0 && (!sline_len_d || !sline_d || !points_d)))
        return fail(CUSLINES_EINVAL, "null argument");
    if (nslines < 0) return fail(CUSLINES_EINVAL, "negative size");
    HIPC(hipSetDevice(t->device));
    int rc = run_scan<long long>(t, sline_len_d, nslines, reinterpret_cast<long long *>(point_off_d));
    if (rc) return rc;
    if (nslines == 0) return CUSLINES_OK;
    const size_t slot_f = (size_t)2 * t->dp.max_sline_len * 3;
    const unsigned grid = (unsigned)std::min<long long>(((long long)nslines + 3) / 4, 65536);
    hipLaunchKernelGGL(compact_kernel, dim3(grid), dim3(256), 0, t->stream, sline_len_d, nslines, sline_d, slot_f,
                       reinterpret_cast<const long long *>(point_off_d), points_d);
    HIPC(hipGetLastError());
    return CUSLINES_OK;
}

int cuslines_chunk_workspace_bytes(cuslines_tracker *t, int32_t nseeds, int32_t slot_cap, size_t *bytes) {
    if (!t || !bytes) return fail(CUSLINES_EINVAL, "null argument");
    if (nseeds < 0 || slot_cap < 1) return fail(CUSLINES_EINVAL, "negative size or slot_cap < 1");
    *bytes = chunk_ws_bytes(nseeds, slot_cap);
    return CUSLINES_OK;
}

int cuslines_chunk_async(cuslines_tracker *t, const float *seeds_d, int32_t nseeds, int32_t rng_chunk,
                         int32_t *counts_d, int32_t *dirs_d, int32_t *offsets_d, int32_t slot_cap,
                         int32_t *sline_seed_d, int32_t *sline_len_d, float *sline_d, int64_t *point_off_d,
                         float *points_d, int64_t *totals_d, void *ws_d, size_t ws_bytes) {
    RoctxRange range_("cuslines_chunk");
    chunk_args a;
    if (int rc = chunk_check(t, seeds_d, nseeds, rng_chunk, counts_d, dirs_d, offsets_d, slot_cap, sline_seed_d,
                             sline_len_d, sline_d, point_off_d, points_d, totals_d, ws_d, ws_bytes, &a))
        return rc;
    HIPC(hipSetDevice(t->device));
    return chunk_run(t, a);
}

int cuslines_chunk_graph_create(cuslines_tracker *t, const float *seeds_d, int32_t nseeds, int32_t rng_chunk,
                                int32_t *counts_d, int32_t *dirs_d, int32_t *offsets_d, int32_t slot_cap,
                                int32_t *sline_seed_d, int32_t *sline_len_d, float *sline_d, int64_t *point_off_d,
                                float *points_d, int64_t *totals_d, void *ws_d, size_t ws_bytes,
                                cuslines_graph **out) {
    RoctxRange range_("cuslines_chunk_graph_create");
    if (!out) return fail(CUSLINES_EINVAL, "null argument");
    *out = nullptr;
    chunk_args a;
    if (int rc = chunk_check(t, seeds_d, nseeds, rng_chunk, counts_d, dirs_d, offsets_d, slot_cap, sline_seed_d,
                             sline_len_d, sline_d, point_off_d, points_d, totals_d, ws_d, ws_bytes, &a))
        return rc;
    HIPC(hipSetDevice(t->device));
    HIPC(hipStreamBeginCapture(t->stream, hipStreamCaptureModeRelaxed));
    const int rc = chunk_run(t, a);
    hipGraph_t g = nullptr;
    const hipError_t e = hipStreamEndCapture(t->stream, &g);
    if (rc || e != hipSuccess) {
        if (g) (void)hipGraphDestroy(g);
        return rc ? rc : fail(CUSLINES_EHIP, std::string("hipStreamEndCapture: ") + hipGetErrorString(e));
    }
    hipGraphExec_t x = nullptr;
    const hipError_t ei = hipGraphInstantiate(&x, g, nullptr, nullptr, 0);
    if (ei != hipSuccess) {
        (void)hipGraphDestroy(g);
        return fail(CUSLINES_EHIP, std::string("hipGraphInstantiate: ") + hipGetErrorString(ei));
    }
    *out = new cuslines_graph{t, g, x};
    ++t->ngraphs;
    if (t->parent) ++t->parent->ngraphs;
    return CUSLINES_OK;
}

int cuslines_graph_launch(cuslines_graph *g) {
    if (!g) return fail(CUSLINES_EINVAL, "null graph");
    HIPC(hipSetDevice(g->t->device));
    HIPC(hipGraphLaunch(g->exec, g->t->stream));
    return CUSLINES_OK;
}

int cuslines_graph_destroy(cuslines_graph *g) {
    if (!g) return CUSLINES_OK;
    (void)hipSetDevice(g->t->device);
    (void)hipStreamSynchronize(g->t->stream);  // a launch may still run
    const hipError_t e1 = hipGraphExecDestroy(g->exec);
    const hipError_t e2 = hipGraphDestroy(g->graph);
    --g->t->ngraphs;
    if (g->t->parent) --g->t->parent->ngraphs;
    delete g;
    if (e1 != hipSuccess || e2 != hipSuccess) return fail(CUSLINES_EHIP, "hipGraph destroy failed");
    return CUSLINES_OK;
}

}  // extern "C"
