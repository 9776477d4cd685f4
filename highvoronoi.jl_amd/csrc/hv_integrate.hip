// hv_integrate.hip -- gfx950 kernels and host driver of cell volumes and interface areas.
//
// Exact polytope integrator (the reference's src/polyintegrator.jl:80-468 computes, cell by
// cell, each interface F_ik by a recursive cone decomposition and vol_i = sum_k A_ik h_ik/d,
// :296-312).  Here the same decomposition runs over all faces of the tessellation at once,
// one face dimension per pass:
//   * in general position every subset S of a vertex key that holds a generator is a
//     face; faces with |S| = m have dimension k = d + 1 - m and are identified by their
//     generator set, packed into 128 bits (21 bits per id);
//   * the (k-1)-faces of S are the faces T = S + {j}, so pass m takes the faces T of pass m + 1
//     (the vertices before the first pass, m = d), emits the pair (S, T) for each S = T - {j},
//     and groups the pairs by S: the groups are the faces of pass m, each with its list of T;
//   * edges (m = d) measure |v_a - v_b|; a face of dimension k > 1 is the union of cones
//     from one of its vertices p over its (k-1)-faces T that miss p:
//     |F_S| = (1/k) sum_T h(p, aff F_T) |F_T|, h measured inside aff F_S;
//   * p is the smallest vertex of S, so T holds it exactly when it is T's smallest vertex too;
//   * facets (m = 2) are the interfaces A_ik; volumes take the generator as apex.
// A face's T are read in a fixed order: no atomics, the result does not depend on scheduling.
//
// Grouping is what moves the most bytes, so it sorts 32-bit keys: the face's smallest id above 15
// bits of a hash of its ids (4 radix passes of 8 bytes per pair; the whole key in 42 .. 105
// bits took 6 .. 14 passes of 12).  About one face in a hundred shares its 32 bits with another
// of its cell; such runs are put in order by their full keys afterwards.  (More than 2^17 ids leave fewer
// hash bits: 11 for the nearly 2^21 of a 6D N=50k periodic mesh, whose runs hold many faces and take 2.5 of
// the 3.8 s to put in order, 4.9 s with the whole keys sorted.)  Pairs (S, T) instead of
// (S, vertex) are fewer from the 3-faces down and need no look-up of the sub-faces.
// 5D N=100k mixture (16.3M vertices): the integration's kernels 207 -> 77 ms (the sorts 70 -> 22,
// the measures 74 -> 20, the look-up tables of the former 31 -> 0).
//
// Monte-Carlo integrator (src/mcintegrator.jl:98-204): one workgroup per cell casts ndir
// rays from the generator (mc_raycast, :207-226) against the cell's neighbours (boundary
// planes through their mirror image of the generator), accumulates t^d and the facet
// hits, then the neighbour estimates are symmetrised (:176-200).  Each cell draws its own
// directions (counter-based splitmix64 + Box-Muller); the reference reuses one direction
// for every sample (the draw loop at :85-93 never re-enters), which is not carried over.
#include "hv_device.h"
#include "hv_internal.h"
#include <hipcub/hipcub.hpp>
#include <rocprim/rocprim.hpp>
#include <algorithm>
#include <climits>
#include <cmath>
#include <cstring>
#include <memory>
#include <numeric>
#include <set>

#define HVCK(call)                                                                 \
    do {                                                                           \
        hipError_t e_ = (call);                                                    \
        if (e_ != hipSuccess)                                                      \
            return hv_fail(c, HV_ERR_DEVICE, std::string(#call) + ": " + hipGetErrorString(e_)); \
    } while (0)

static inline unsigned nblk(int64_t n, int b) { return (unsigned)((n + b - 1) / b); }

template <typename T>
static T* iget(hv_ctx* c, const char* name, size_t count) {
    return (T*)c->pool->get(name, std::max<size_t>(1, count) * sizeof(T), false, c->stream);
}

constexpr uint64_t HV_F21 = 0x1FFFFFull;   // id field of a face key
// pairs one pass of a chunk may hold (a chunk of cells at a time beyond)
constexpr int64_t HV_INC_BUDGET = 1600000000ll;
constexpr int HV_GROUP_HASH = 15;          // hash bits of a grouping key
constexpr uint32_t HV_NO_FACE = 0xffffffffu;

// used ids of the mesh's keys (a first pass over the live vertices)
template <int D>
__global__ void k_mark_used(const int* __restrict__ ids, int nv, const int* __restrict__ key, int* __restrict__ used) {
    const int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= (int64_t)nv * (D + 1)) return;
    const int v = (int)(t / (D + 1)), j = (int)(t - (int64_t)v * (D + 1));
    used[key[(int64_t)ids[v] * (D + 1) + j]] = 1;
}

// word of the dense ids first .. first + count - 1 of each key (first id most significant), for
// the vertices in the order of perm (null: their own order, and perm0 receives 0, 1, ..)
template <int D>
__global__ void k_vkey_word(const int* __restrict__ ids, int nv, const int* __restrict__ key, const int* __restrict__ dense,
                            const int* __restrict__ perm, int first, int count, int bits, uint64_t* __restrict__ word,
                            int* __restrict__ perm0) {
    const int v = blockIdx.x * blockDim.x + threadIdx.x;
    if (v >= nv) return;
    const int* k = key + (int64_t)ids[perm ? perm[v] : v] * (D + 1);
    uint64_t w = 0;
    for (int j = 0; j < count; ++j) w = (w << bits) | (uint64_t)(uint32_t)dense[k[first + j]];
    word[v] = w;
    if (!perm) perm0[v] = v;
}

// the live vertices in the order of perm: keys in dense ids, coordinates
template <int D>
__global__ void k_int_permute(const int* __restrict__ perm, int nv, const int* __restrict__ ids, const int* __restrict__ key,
                              const int* __restrict__ dense, const double* __restrict__ x, int* __restrict__ vk,
                              double* __restrict__ vc) {
    const int v = blockIdx.x * blockDim.x + threadIdx.x;
    if (v >= nv) return;
    const int64_t s = ids[perm[v]];
#pragma unroll
    for (int j = 0; j <= D; ++j) vk[(int64_t)v * (D + 1) + j] = dense[key[s * (D + 1) + j]];
#pragma unroll
    for (int k = 0; k < D; ++k) vc[(int64_t)v * D + k] = x[s * D + k];
}

// ---- faces and their lists -------------------------------------------------------------------
// The faces of one pass: keys (ids 0 .. 2 of the sorted set in klo, 3 .. 5 in khi, 21 bits each),
// and per face its measure, its smallest vertex (canonical order) and its number of vertices.
struct HvFace {
    double meas;
    int vmin, nv;
};
struct HvFaces {
    uint64_t* klo;
    uint64_t* khi;
    HvFace* f;
};
// The pairs of pass m sorted by face: pair i belongs to T = pay[i] / (m + 1) with T's id jl[i]
// left out; face f holds the pairs start[f] .. start[f + 1] - 1 (the last one to *nvalid - 1).
struct HvPairs {
    const uint32_t* pay;
    const int* jl;
    const int* start;
    const int* nvalid;
    int nface;
};

// ids of T: a vertex (M == D: its key's row) or a face of pass M + 1
template <int D, int M>
__device__ __forceinline__ void hv_sub_ids(const int* __restrict__ vk, const HvFaces& F1, int64_t t, int* id) {
    if constexpr (M == D) {
#pragma unroll
        for (int j = 0; j <= M; ++j) id[j] = vk[t * (D + 1) + j];
    } else {
        const uint64_t lo = F1.klo[t];
        uint64_t hi = 0;
        if constexpr (M + 1 > 3) hi = F1.khi[t];
#pragma unroll
        for (int j = 0; j <= M; ++j) id[j] = (int)((j < 3 ? lo >> (21 * j) : hi >> (21 * (j - 3))) & HV_F21);
    }
}
// packed key of T without its p-th id, and that id
template <int M>
__device__ __forceinline__ int hv_face_key(const int* id, int p, uint64_t& lo, uint64_t& hi) {
    lo = hi = 0;
    int out = id[0];
#pragma unroll
    for (int j = 0; j < M; ++j) {
        const uint64_t v = (uint64_t)(uint32_t)(j < p ? id[j] : id[j + 1]);
        if (j < 3) lo |= v << (21 * j);
        else hi |= v << (21 * (j - 3));
    }
#pragma unroll
    for (int j = 1; j <= M; ++j) out = j == p ? id[j] : out;
    return out;
}

// hash of each dense id, from the id it stands for (the order of a face's T then does not depend
// on which cells a mesh or a chunk holds)
__global__ void k_id_hash(const int* __restrict__ gid, int n, uint32_t* __restrict__ hid) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) hid[i] = (uint32_t)(hv_mix64((uint64_t)gid[i] + 0x9e3779b97f4a7c15ull) >> 32);
}

// Grouping keys of the pairs (S = T - {its p-th id}, T), pair t (M + 1) + p, one thread per T: S's
// smallest id above hb bits of the hash of its ids (a sum over the ids, so that T's M + 1 subsets
// share it).  HV_NO_FACE, which sorts past the end, where S holds no cell of the chunk (cmask over
// the ids below N; null: every generator): such a face may be incomplete here.
template <int D, int M>
__global__ __launch_bounds__(256) void k_pair_emit(const int* __restrict__ vk, HvFaces F1, int nt, int N,
                                                   const uint8_t* __restrict__ cmask, const uint32_t* __restrict__ hid,
                                                   int hb, uint32_t* __restrict__ key) {
    const int t = blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= nt) return;
    int id[M + 1];
    hv_sub_ids<D, M>(vk, F1, t, id);
    uint32_t h[M + 1], sum = 0;
    int cells = 0, cell[M + 1];
#pragma unroll
    for (int j = 0; j <= M; ++j) {
        h[j] = hid[id[j]];
        sum += h[j];
        cell[j] = id[j] < N && (!cmask || cmask[id[j]] != 0) ? 1 : 0;
        cells += cell[j];
    }
#pragma unroll
    for (int p = 0; p <= M; ++p) {
        const uint32_t a = (uint32_t)(p == 0 ? id[1] : id[0]);
        const uint32_t hs = ((sum - h[p]) * 0x9E3779B1u) >> (32 - hb);
        key[(int64_t)t * (M + 1) + p] = cells > cell[p] ? ((a << hb) | hs) : HV_NO_FACE;
    }
}

// Sorted pairs -> first pair of every face, the id each pair leaves out, the number of pairs of
// real faces, and the runs of one grouping key that hold more than one face (runs: their first
// pairs, at their first change of face)
template <int D, int M>
__global__ __launch_bounds__(256) void k_pair_heads(const uint32_t* __restrict__ key, const uint32_t* __restrict__ pay,
                                                    int64_t n, const int* __restrict__ vk, HvFaces F1,
                                                    uint8_t* __restrict__ head, int* __restrict__ jl,
                                                    int* __restrict__ nvalid, int* __restrict__ runs,
                                                    int* __restrict__ nrun) {
    __shared__ uint64_t slo[257], shi[M > 3 ? 257 : 1];
    __shared__ uint32_t sk[257];
    __shared__ int cnt, base;
    const int64_t i0 = (int64_t)blockIdx.x * 256, i = i0 + threadIdx.x;
    if (threadIdx.x == 0) cnt = 0;
    auto stage = [&](int64_t q, int at) {   // pair q's grouping key and face key
        const uint32_t k = key[q];
        uint64_t lo = 0, hi = 0;
        int j = 0;
        if (k != HV_NO_FACE) {
            int id[M + 1];
            const uint32_t e = pay[q], t = e / (M + 1);
            hv_sub_ids<D, M>(vk, F1, t, id);
            j = hv_face_key<M>(id, (int)(e - t * (M + 1)), lo, hi);
        }
        sk[at] = k;
        slo[at] = lo;
        if constexpr (M > 3) shi[at] = hi;
        return j;
    };
    int j = 0;
    if (i < n) j = stage(i, threadIdx.x + 1);
    if (threadIdx.x == 0 && i0 > 0) stage(i0 - 1, 0);
    __syncthreads();
    int start = -1;
    if (i < n) {
        const uint32_t k = sk[threadIdx.x + 1];
        const bool prev = i > 0, samek = prev && sk[threadIdx.x] == k;
        auto differs = [&](int x) {   // pairs x and x + 1 of the staged ones
            bool d = slo[x] != slo[x + 1];
            if constexpr (M > 3) d = d || shi[x] != shi[x + 1];
            return d;
        };
        const bool change = !samek || differs(threadIdx.x);
        if (k == HV_NO_FACE) {
            head[i] = 0;
            if (!samek) *nvalid = (int)i;
        } else {
            head[i] = change ? 1 : 0;
            jl[i] = j;
            if (samek && change) {
                // the run's first change of face: none between the run's first pair and here
                int64_t q = i - 1;
                bool earlier = false;
                uint64_t plo = slo[threadIdx.x], phi = 0;
                if constexpr (M > 3) phi = shi[threadIdx.x];
                while (q > 0 && key[q - 1] == k && !earlier) {
                    --q;
                    uint64_t lo, hi;
                    int id[M + 1];
                    const uint32_t e = pay[q], t = e / (M + 1);
                    hv_sub_ids<D, M>(vk, F1, t, id);
                    hv_face_key<M>(id, (int)(e - t * (M + 1)), lo, hi);
                    earlier = lo != plo || hi != phi;
                }
                if (!earlier) start = (int)q;
            }
        }
    }
    int at = -1;
    if (start >= 0) at = atomicAdd(&cnt, 1);
    __syncthreads();
    if (threadIdx.x == 0) base = cnt ? atomicAdd(nrun, cnt) : 0;
    __syncthreads();
    if (at >= 0) runs[base + at] = start;
}

// A run of one grouping key with several faces: its pairs sorted by face (stably: each face's T
// stay ascending), one thread per run
template <int D, int M>
__global__ __launch_bounds__(64) void k_pair_fix(const uint32_t* __restrict__ key, int64_t n, const int* __restrict__ vk,
                                                 HvFaces F1, const int* __restrict__ runs, const int* __restrict__ nrun,
                                                 uint32_t* __restrict__ pay, uint8_t* __restrict__ head, int* __restrict__ jl) {
    const int nr = *nrun;
    for (int r = blockIdx.x * blockDim.x + threadIdx.x; r < nr; r += gridDim.x * blockDim.x) {
        const int64_t b = runs[r];
        const uint32_t k = key[b];
        auto face = [&](uint32_t e, uint64_t& lo, uint64_t& hi) {
            int id[M + 1];
            const uint32_t t = e / (M + 1);
            hv_sub_ids<D, M>(vk, F1, t, id);
            return hv_face_key<M>(id, (int)(e - t * (M + 1)), lo, hi);
        };
        int64_t e = b + 1;
        for (; e < n && key[e] == k; ++e) {
            const uint32_t x = pay[e];
            uint64_t xl, xh;
            face(x, xl, xh);
            int64_t q = e;
            while (q > b) {
                uint64_t yl, yh;
                face(pay[q - 1], yl, yh);
                if (!(yh > xh || (yh == xh && yl > xl))) break;
                pay[q] = pay[q - 1];
                --q;
            }
            pay[q] = x;
        }
        uint64_t pl = 0, ph = 0;
        for (int64_t q = b; q < e; ++q) {
            uint64_t lo, hi;
            jl[q] = face(pay[q], lo, hi);
            head[q] = (q == b || lo != pl || hi != ph) ? 1 : 0;
            pl = lo;
            ph = hi;
        }
    }
}

struct IntGeo {
    int N, P;
    int nreal;          // cells integrated: 0 .. nreal-1 (N - nreal periodic images follow)
    const double* xo;   // N x D, original order
    const double* pn;   // P x D outer normals
    const double* ph;   // P offsets <n_p, b_p>
};

// constraint normal of member b of a face whose first generator is a
template <int D>
__device__ __forceinline__ void hv_face_grad(const IntGeo& g, int a, int b, double* w) {
    if (b >= g.N) {
#pragma unroll
        for (int k = 0; k < D; ++k) w[k] = g.pn[(b - g.N) * D + k];
    } else {
#pragma unroll
        for (int k = 0; k < D; ++k) w[k] = g.xo[(int64_t)b * D + k] - g.xo[(int64_t)a * D + k];
    }
}

// w minus its components along the R orthonormal vectors Q (two Gram-Schmidt passes); its norm
template <int D, int R>
__device__ __forceinline__ double hv_project(double (*Q)[D], double* w) {
#pragma unroll
    for (int pass = 0; pass < 2; ++pass)
#pragma unroll
        for (int r = 0; r < R; ++r) {
            double cdot = 0.0;
#pragma unroll
            for (int k = 0; k < D; ++k) cdot = fma(w[k], Q[r][k], cdot);
#pragma unroll
            for (int k = 0; k < D; ++k) w[k] = fma(-cdot, Q[r][k], w[k]);
        }
    double nw = 0.0;
#pragma unroll
    for (int k = 0; k < D; ++k) nw = fma(w[k], w[k], nw);
    return sqrt(nw);
}

// orthonormal basis Q (M - 1 vectors) of the constraint normals of a face with the ids S
template <int D, int M, int S0 = 1>
__device__ __forceinline__ bool hv_face_basis(const IntGeo& g, const int* S, double (*Q)[D]) {
    if constexpr (S0 < M) {
        double w[D];
        hv_face_grad<D>(g, S[0], S[S0], w);
        const double nw = hv_project<D, S0 - 1>(Q, w);
        if (!(nw > 0.0)) return false;
#pragma unroll
        for (int k = 0; k < D; ++k) Q[S0 - 1][k] = w[k] / nw;
        return hv_face_basis<D, M, S0 + 1>(g, S, Q);
    }
    return true;
}

// distance within the face (basis Q, first generator a, da = |p - x_a|^2) of the point p from its
// sub-face on the bisector or plane of j
template <int D, int M>
__device__ __forceinline__ double hv_face_height(const IntGeo& g, double (*Q)[D], int a, int j, const double* p, double da) {
    double w[D];
    hv_face_grad<D>(g, a, j, w);
    const double nr = hv_project<D, M - 1>(Q, w);
    if (j >= g.N) {
        double np_ = 0.0;
#pragma unroll
        for (int k = 0; k < D; ++k) np_ = fma(g.pn[(j - g.N) * D + k], p[k], np_);
        return fabs(g.ph[j - g.N] - np_) / nr;
    }
    double dj = 0.0;
#pragma unroll
    for (int k = 0; k < D; ++k) {
        const double t = p[k] - g.xo[(int64_t)j * D + k];
        dj = fma(t, t, dj);
    }
    return fabs(dj - da) / (2.0 * nr);
}

// edges: pairs of vertices
template <int D>
__global__ void k_edge_measure(HvPairs L, const int* __restrict__ vk, const double* __restrict__ vc, HvFaces F,
                               int* __restrict__ bad) {
    const int f = blockIdx.x * blockDim.x + threadIdx.x;
    if (f >= L.nface) return;
    const int b = L.start[f], e = f + 1 < L.nface ? L.start[f + 1] : *L.nvalid;
    const uint32_t x = L.pay[b];
    const int va = (int)(x / (D + 1));
    int id[D + 1];
    hv_sub_ids<D, D>(vk, F, va, id);
    uint64_t lo, hi;
    hv_face_key<D>(id, (int)(x - (uint32_t)va * (D + 1)), lo, hi);
    F.klo[f] = lo;
    if constexpr (D > 3) F.khi[f] = hi;
    if (e - b != 2) {
        atomicOr(bad, 1);
        F.f[f] = HvFace{0.0, va, 2};
        return;
    }
    const int vb = (int)(L.pay[b + 1] / (D + 1));
    double s = 0.0;
#pragma unroll
    for (int k = 0; k < D; ++k) {
        const double t = vc[(int64_t)va * D + k] - vc[(int64_t)vb * D + k];
        s = fma(t, t, s);
    }
    F.f[f] = HvFace{sqrt(s), va, 2};   // pairs ascend by vertex: va is the smaller
}

// Faces of pass M < D from the faces of pass M + 1 (F1), `lanes` of a wavefront per face (W: a power
// of two), the partial sums combined in a fixed order.  Bound by the gathers of the sub-faces and
// the generators' coordinates; with W > 1 a face of many sub-faces is not one lane's serial chain.
template <int D, int M, int W>
__global__ __launch_bounds__(128) void k_face_measure(IntGeo g, HvPairs L, const int* __restrict__ vk,
                                                      const double* __restrict__ vc, HvFaces F1, HvFaces F,
                                                      int* __restrict__ bad) {
    const int64_t gt = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    const int lane = (int)(gt % W);
    // a dispatch holds at most 2^32 work-items: the faces are walked grid-stride
    for (int64_t f = gt / W; f < L.nface; f += (int64_t)gridDim.x * blockDim.x / W) {
        const int b = L.start[f], e = f + 1 < L.nface ? L.start[f + 1] : *L.nvalid;
        int S[M];
        {
            const uint32_t x = L.pay[b], t = x / (M + 1);
            int id[M + 1];
            hv_sub_ids<D, M>(vk, F1, t, id);
            const int p = (int)(x - t * (M + 1));
            uint64_t lo, hi;
            hv_face_key<M>(id, p, lo, hi);
#pragma unroll
            for (int s = 0; s < M; ++s) S[s] = s < p ? id[s] : id[s + 1];
            if (lane == 0) {
                F.klo[f] = lo;
                if constexpr (M > 3) F.khi[f] = hi;
            }
        }
        // the apex: the face's smallest vertex
        int apex = INT_MAX, nvs = 0;
        for (int i = b + lane; i < e; i += W) {
            const HvFace& T = F1.f[L.pay[i] / (M + 1)];
            apex = min(apex, T.vmin);
            nvs += T.nv;
        }
#pragma unroll
        for (int off = W / 2; off > 0; off >>= 1) {
            apex = min(apex, __shfl_xor(apex, off));
            nvs += __shfl_xor(nvs, off);
        }
        double Q[M > 1 ? M - 1 : 1][D];
        double sum = 0.0;
        if (hv_face_basis<D, M>(g, S, Q)) {
            double p[D], da = 0.0;
#pragma unroll
            for (int k = 0; k < D; ++k) {
                p[k] = vc[(int64_t)apex * D + k];
                const double t = p[k] - g.xo[(int64_t)S[0] * D + k];
                da = fma(t, t, da);
            }
            for (int i = b + lane; i < e; i += W) {
                const HvFace T = F1.f[L.pay[i] / (M + 1)];
                if (T.vmin == apex) continue;   // the sub-face holds the apex: zero height
                sum = fma(hv_face_height<D, M>(g, Q, S[0], L.jl[i], p, da), T.meas, sum);
            }
        } else if (lane == 0) {
            atomicOr(bad, 2);
        }
#pragma unroll
        for (int off = W / 2; off > 0; off >>= 1) sum += __shfl_xor(sum, off);
        constexpr int K = D + 1 - M;   // the face's dimension; a vertex of it lies in K of its T
        if (lane == 0) F.f[f] = HvFace{sum / (double)K, apex, nvs / K};
    }
}

// lanes per face of pass m, by the face dimension k = d + 1 - m: a polygon has 4 to 5 edges on
// average, a 3-face about 10 polygons, faces of higher dimension tens of sub-faces
constexpr int hv_face_lanes(int D, int M) { return D + 1 - M >= 4 ? 4 : 1; }

static inline unsigned hv_face_blocks(int nface, int lanes) {
    return (unsigned)std::min<int64_t>(std::max<int64_t>(((int64_t)nface * lanes + 127) / 128, 1), 1 << 20);
}

// ---- integrands (the reference's rule, src/polyintegrator.jl:174-353) -----------------------
// Every face G is cut into the simplices of the chains of face centres (the mean of a face's
// vertices) from G down to an edge; f enters only at the two ends of each edge:
//   J(edge) = |e| (f(v1) + f(v2)) / 2,   J(G) = sum over sub-faces H of h_H(c_G) J(H) / dim G,
// h_H(c_G) the distance within G from G's centre to H.  A facet F (dim d-1) then gets
//   I(F) = (d-1)/d J(F) + f(c_F) |F| / d,
// and a cell, with apex at its generator x,
//   bulk = f(x) vol / (d+1) + sum over facets F of dist(x, F) I(F) / (d+1).
// Exact for affine f.  nf <= HV_MAXF components per point.  Every vertex of a face of dimension
// k lies in k of its sub-faces, so the centre is the mean of theirs, weighted by their vertices.
constexpr int HV_MAXF = 8;

template <int D>
__global__ void k_edge_int(HvPairs L, HvFaces F, const double* __restrict__ vc, const double* __restrict__ fv, int nf,
                           double* __restrict__ cen, double* __restrict__ J) {
    const int f = blockIdx.x * blockDim.x + threadIdx.x;
    if (f >= L.nface) return;
    const int b = L.start[f], e = f + 1 < L.nface ? L.start[f + 1] : *L.nvalid;
    const int64_t va = L.pay[b] / (D + 1), vb = e - b == 2 ? L.pay[b + 1] / (D + 1) : va;   // flagged by k_edge_measure
#pragma unroll
    for (int k = 0; k < D; ++k) cen[(int64_t)f * D + k] = (vc[va * D + k] + vc[vb * D + k]) * 0.5;
    for (int c = 0; c < nf; ++c) J[(int64_t)f * nf + c] = F.f[f].meas * 0.5 * (fv[va * nf + c] + fv[vb * nf + c]);
}

// centre and J of each face of pass M from those of pass M + 1 (W lanes per face, as k_face_measure)
template <int D, int M, int W>
__global__ __launch_bounds__(128) void k_face_int(IntGeo g, HvPairs L, const int* __restrict__ vk, HvFaces F1,
                                                  const double* __restrict__ cen1, const double* __restrict__ J1, int nf,
                                                  double* __restrict__ cen, double* __restrict__ J, int* __restrict__ bad) {
    const int64_t gt = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    const int lane = (int)(gt % W);
    for (int64_t f = gt / W; f < L.nface; f += (int64_t)gridDim.x * blockDim.x / W) {
        const int b = L.start[f], e = f + 1 < L.nface ? L.start[f + 1] : *L.nvalid;
        int S[M];
        {
            const uint32_t x = L.pay[b], t = x / (M + 1);
            int id[M + 1];
            hv_sub_ids<D, M>(vk, F1, t, id);
            const int p = (int)(x - t * (M + 1));
#pragma unroll
            for (int s = 0; s < M; ++s) S[s] = s < p ? id[s] : id[s + 1];
        }
        double p[D], nvs = 0.0;
#pragma unroll
        for (int k = 0; k < D; ++k) p[k] = 0.0;
        for (int i = b + lane; i < e; i += W) {
            const int64_t t = L.pay[i] / (M + 1);
            const double w = (double)F1.f[t].nv;
            nvs += w;
#pragma unroll
            for (int k = 0; k < D; ++k) p[k] = fma(w, cen1[t * D + k], p[k]);
        }
#pragma unroll
        for (int off = W / 2; off > 0; off >>= 1) {
            nvs += __shfl_xor(nvs, off);
#pragma unroll
            for (int k = 0; k < D; ++k) p[k] += __shfl_xor(p[k], off);
        }
        double Q[M > 1 ? M - 1 : 1][D];
        double da = 0.0;
#pragma unroll
        for (int k = 0; k < D; ++k) {
            p[k] /= nvs;
            if (lane == 0) cen[f * D + k] = p[k];
            const double t = p[k] - g.xo[(int64_t)S[0] * D + k];
            da = fma(t, t, da);
        }
        double sum[HV_MAXF];
        for (int c = 0; c < nf; ++c) sum[c] = 0.0;
        if (hv_face_basis<D, M>(g, S, Q)) {
            for (int i = b + lane; i < e; i += W) {
                const double h = hv_face_height<D, M>(g, Q, S[0], L.jl[i], p, da);
                const int64_t t = L.pay[i] / (M + 1);
                for (int c = 0; c < nf; ++c) sum[c] = fma(h, J1[t * nf + c], sum[c]);
            }
        } else if (lane == 0) {
            atomicOr(bad, 2);
        }
        for (int c = 0; c < nf; ++c) {
#pragma unroll
            for (int off = W / 2; off > 0; off >>= 1) sum[c] += __shfl_xor(sum[c], off);
            if (lane == 0) J[f * nf + c] = sum[c] / (double)(D + 1 - M);
        }
    }
}

// facets: I(F) = (d-1)/d J(F) + f(c_F) |F| / d
template <int D>
__global__ void k_facet_int(int nface, const double* __restrict__ J, const double* __restrict__ fc,
                            const HvFace* __restrict__ face, int nf, double* __restrict__ I) {
    const int f = blockIdx.x * blockDim.x + threadIdx.x;
    if (f >= nface) return;
    for (int c = 0; c < nf; ++c)
        I[(int64_t)f * nf + c] = (double)(D - 1) / (double)D * J[(int64_t)f * nf + c] +
                                 fc[(int64_t)f * nf + c] * face[f].meas / (double)D;
}

// cells 0 .. nreal-1: f(x) vol / (d+1) + sum over rows of dist * I(row) / (d+1)
template <int D>
__global__ void k_cell_bulk(IntGeo g, const uint64_t* __restrict__ pkey, const int64_t* __restrict__ ptr,
                            const double* __restrict__ vol, const double* __restrict__ rint,
                            const double* __restrict__ fx, int nf, double* __restrict__ bulk) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= g.nreal) return;
    double y[HV_MAXF];
    for (int c = 0; c < nf; ++c) y[c] = fx[(int64_t)i * nf + c] * vol[i];
    for (int64_t t = ptr[i]; t < ptr[i + 1]; ++t) {
        const int k = (int)(pkey[t] & 0xffffffffull);
        double h;
        if (k >= g.N) {
            double nx = 0.0;
#pragma unroll
            for (int c = 0; c < D; ++c) nx = fma(g.pn[(k - g.N) * D + c], g.xo[(int64_t)i * D + c], nx);
            h = g.ph[k - g.N] - nx;
        } else {
            double s2 = 0.0;
#pragma unroll
            for (int c = 0; c < D; ++c) {
                const double t2 = g.xo[(int64_t)i * D + c] - g.xo[(int64_t)k * D + c];
                s2 = fma(t2, t2, s2);
            }
            h = 0.5 * sqrt(s2);
        }
        for (int c = 0; c < nf; ++c) y[c] = fma(h, rint[t * nf + c], y[c]);
    }
    for (int c = 0; c < nf; ++c) bulk[(int64_t)i * nf + c] = y[c] / (double)(D + 1);
}

// facets {a, b} -> rows (cell << bits | neighbour) at 2f and 2f + 1, one per side that is a cell of
// the chunk (~0, which sorts past the end, for the other), with their areas and interface integrals
__global__ void k_facet_rows(int nface, HvFaces F, int N, const uint8_t* __restrict__ cmask, int bits,
                             uint64_t* __restrict__ row, double* __restrict__ area, const double* __restrict__ I, int nf,
                             double* __restrict__ rint) {
    const int f = blockIdx.x * blockDim.x + threadIdx.x;
    if (f >= nface) return;
    const uint64_t a = F.klo[f] & HV_F21, b = (F.klo[f] >> 21) & HV_F21;
    const bool ra = a < (uint64_t)N && (!cmask || cmask[a] != 0), rb = b < (uint64_t)N && (!cmask || cmask[b] != 0);
    row[2 * (int64_t)f] = ra ? (a << bits) | b : ~0ull;
    row[2 * (int64_t)f + 1] = rb ? (b << bits) | a : ~0ull;
    const double m = F.f[f].meas;
    area[2 * (int64_t)f] = m;
    area[2 * (int64_t)f + 1] = m;
    for (int c = 0; c < nf; ++c) {
        const double v = I[(int64_t)f * nf + c];
        rint[2 * (int64_t)f * nf + c] = v;
        rint[(2 * (int64_t)f + 1) * nf + c] = v;
    }
}

__global__ void k_set_mask(const int* __restrict__ ids, int n, uint8_t* __restrict__ mask) {
    const int t = blockIdx.x * blockDim.x + threadIdx.x;
    if (t < n) mask[ids[t]] = 1;
}

// vertices holding a cell of the chunk
template <int D>
__global__ void k_vert_in_chunk(const int* __restrict__ vk, int nv, int N, const uint8_t* __restrict__ cmask,
                                uint8_t* __restrict__ flag) {
    const int v = blockIdx.x * blockDim.x + threadIdx.x;
    if (v >= nv) return;
    bool in = false;
#pragma unroll
    for (int j = 0; j <= D; ++j) {
        const int id = vk[(int64_t)v * (D + 1) + j];
        in = in || (id < N && cmask[id] != 0);
    }
    flag[v] = in ? 1 : 0;
}

template <int D>
__global__ __launch_bounds__(256) void k_count_in_chunk(const int* __restrict__ vk, int nv, int N,
                                                        const uint8_t* __restrict__ cmask, unsigned long long* __restrict__ cnt) {
    const int v = blockIdx.x * blockDim.x + threadIdx.x;
    bool in = false;
    if (v < nv)
#pragma unroll
        for (int j = 0; j <= D; ++j) {
            const int id = vk[(int64_t)v * (D + 1) + j];
            in = in || (id < N && cmask[id] != 0);
        }
    hv_wave_count(cnt, in);
}

template <int D>
__global__ void k_int_subset(const int* __restrict__ sel, int n, const int* __restrict__ vk, const double* __restrict__ vc,
                             const double* __restrict__ fv, int nf, int* __restrict__ vk2, double* __restrict__ vc2,
                             double* __restrict__ fv2) {
    const int t = blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= n) return;
    const int v = sel[t];
#pragma unroll
    for (int j = 0; j <= D; ++j) vk2[(int64_t)t * (D + 1) + j] = vk[(int64_t)v * (D + 1) + j];
#pragma unroll
    for (int k = 0; k < D; ++k) vc2[(int64_t)t * D + k] = vc[(int64_t)v * D + k];
    if (fv)
        for (int f = 0; f < nf; ++f) fv2[(int64_t)t * nf + f] = fv[(int64_t)v * nf + f];
}

// sorted rows (cell << bits | neighbour, dense ids) in the caller's ids (cell << 32 | neighbour; the
// map preserves the order) with their payloads; *npair: the number of real ones
__global__ void k_rows_out(const uint64_t* __restrict__ row, const int* __restrict__ perm, int64_t n, int bits,
                           const int* __restrict__ gid, const double* __restrict__ ra, const double* __restrict__ ri, int nf,
                           uint64_t* __restrict__ pkey, double* __restrict__ parea, double* __restrict__ rint,
                           int* __restrict__ npair) {
    const int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= n) return;
    const uint64_t r = row[t];
    if (r == ~0ull) {
        if (t == 0 || row[t - 1] != ~0ull) *npair = (int)t;
        return;
    }
    if (t == n - 1) *npair = (int)n;
    pkey[t] = ((uint64_t)gid[r >> bits] << 32) | (uint64_t)(uint32_t)gid[r & ((1ull << bits) - 1ull)];
    const int s = perm[t];
    parea[t] = ra[s];
    for (int f = 0; f < nf; ++f) rint[t * nf + f] = ri[(int64_t)s * nf + f];
}

template <int D>
__global__ void k_cell_volumes(IntGeo g, const uint64_t* __restrict__ pkey, const double* __restrict__ parea,
                               int64_t npair, double* __restrict__ vol, int64_t* __restrict__ ptr) {
    // one thread per cell: its rows are contiguous after the sort; binary search the range
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i > g.N) return;
    int64_t lo = 0, hi = npair;
    while (lo < hi) {
        const int64_t mid = (lo + hi) >> 1;
        if ((int)(pkey[mid] >> 32) < i) lo = mid + 1;
        else hi = mid;
    }
    ptr[i] = lo;
    if (i == g.N) return;
    double V = 0.0;
    for (int64_t t = lo; t < npair && (int)(pkey[t] >> 32) == i; ++t) {
        const int k = (int)(pkey[t] & 0xffffffffull);
        double h;
        if (k >= g.N) {
            double nx = 0.0;
#pragma unroll
            for (int c = 0; c < D; ++c) nx = fma(g.pn[(k - g.N) * D + c], g.xo[(int64_t)i * D + c], nx);
            h = g.ph[k - g.N] - nx;
        } else {
            double s = 0.0;
#pragma unroll
            for (int c = 0; c < D; ++c) {
                const double t2 = g.xo[(int64_t)i * D + c] - g.xo[(int64_t)k * D + c];
                s = fma(t2, t2, s);
            }
            h = 0.5 * sqrt(s);
        }
        V = fma(parea[t], h / (double)D, V);
    }
    vol[i] = V;
}

// ---- Monte-Carlo ------------------------------------------------------------------------

__device__ __forceinline__ uint64_t hv_sm64(uint64_t seed, uint64_t s) {
    uint64_t z = seed + (s + 1) * 0x9E3779B97F4A7C15ull;
    z = (z ^ (z >> 30)) * 0xBF58476D1CE4E5B9ull;
    z = (z ^ (z >> 27)) * 0x94D049BB133111EBull;
    return z ^ (z >> 31);
}
__device__ __forceinline__ double hv_unif(uint64_t seed, uint64_t s) {
    return (double)(hv_sm64(seed, s) >> 11) * (1.0 / 9007199254740992.0);
}

constexpr int HV_MC_MAXK = 512;

// One workgroup per cell, its neighbours in LDS as w = e - x (e the neighbour or its mirror image) and
// 1 / |w|^2.  A direction u ends at the neighbour of least t = |w|^2 / (2 <u, w>), that is of the largest
// <u, w> / |w|^2: a product and a comparison per neighbour where the quotient took 45 FP64 instructions,
// and t is formed once, for that neighbour.  A thread sweeps up to four directions together, so a
// row is read once for them.  Bound by the FP64 sweep and the directions' logarithms and sines; 4D
// N=20k, 1 000 directions a cell: 1.28 -> 0.61 ms.
template <int D, int NQ>
__device__ __forceinline__ double hv_mc_sweep(const double (*row)[D + 1], int K, double* acc, uint64_t first, int64_t q0, int64_t step,
                                              int64_t ndir, uint64_t seed) {
    constexpr int DP = (D + 1) & ~1;
    double u[NQ][D], best[NQ];
    int win[NQ];
#pragma unroll
    for (int z = 0; z < NQ; ++z) {
        const uint64_t base = (first + (uint64_t)(q0 + z * step)) * (uint64_t)DP;
        double uu = 0.0;
#pragma unroll
        for (int c = 0; c < D; c += 2) {
            const uint64_t p = (base + c) >> 1;
            const double u1 = fmax(hv_unif(seed, 2 * p), 1e-300), u2 = hv_unif(seed, 2 * p + 1);
            const double rad = sqrt(-2.0 * log(u1));
            double sn, cs;
            sincos(2.0 * M_PI * u2, &sn, &cs);
            u[z][c] = rad * cs;
            if (c + 1 < D) u[z][c + 1] = rad * sn;
        }
#pragma unroll
        for (int c = 0; c < D; ++c) uu = fma(u[z][c], u[z][c], uu);
        uu = sqrt(uu);
#pragma unroll
        for (int c = 0; c < D; ++c) u[z][c] /= uu;
        best[z] = 0.0;
        win[z] = -1;
    }
    for (int t = 0; t < K; ++t) {
        double w[D + 1];
#pragma unroll
        for (int c = 0; c <= D; ++c) w[c] = row[t][c];
#pragma unroll
        for (int z = 0; z < NQ; ++z) {
            double den = 0.0;
#pragma unroll
            for (int c = 0; c < D; ++c) den = fma(u[z][c], w[c], den);
            den *= w[D];
            const bool up = den > best[z];
            best[z] = up ? den : best[z];
            win[z] = up ? t : win[z];
        }
    }
    double V = 0.0;
#pragma unroll
    for (int z = 0; z < NQ; ++z) {
        if (q0 + z * step >= ndir) continue;
        double ts = INFINITY, cn = 0.0;
        if (win[z] >= 0) {
            double num = 0.0, den = 0.0;
#pragma unroll
            for (int c = 0; c < D; ++c) {
                const double w = row[win[z]][c];
                num = fma(w, w, num);
                den = fma(u[z][c], w, den);
            }
            ts = num / (2.0 * den);
            cn = den / sqrt(num);
        }
        double tp = 1.0;
#pragma unroll
        for (int c = 0; c < D - 1; ++c) tp *= ts;
        V += tp * ts;
        if (win[z] >= 0 && ts < INFINITY) atomicAdd(&acc[win[z]], tp / fabs(cn));
    }
    return V;
}

template <int D>
__global__ __launch_bounds__(256) void k_mc_cell(IntGeo g, const int64_t* __restrict__ ptr,
                                                 const uint64_t* __restrict__ pkey, int64_t ndir, uint64_t seed,
                                                 double cvol, double carea, double* __restrict__ vol,
                                                 double* __restrict__ area) {
    __shared__ double row[HV_MC_MAXK][D + 1];
    __shared__ double acc[HV_MC_MAXK];
    __shared__ double vred[256];
    const int i = blockIdx.x;
    const int64_t b = ptr[i];
    const int K = (int)(ptr[i + 1] - b);
    double x[D];
#pragma unroll
    for (int c = 0; c < D; ++c) x[c] = g.xo[(int64_t)i * D + c];
    for (int t = threadIdx.x; t < K; t += blockDim.x) {
        const int k = (int)(pkey[b + t] & 0xffffffffull);
        double e[D];
        if (k >= g.N) {
            // mirror image of the generator in the boundary plane (src/boundary.jl:206-211)
            double nx = 0.0;
#pragma unroll
            for (int c = 0; c < D; ++c) nx = fma(g.pn[(k - g.N) * D + c], x[c], nx);
            const double h = g.ph[k - g.N] - nx;
#pragma unroll
            for (int c = 0; c < D; ++c) e[c] = x[c] + 2.0 * h * g.pn[(k - g.N) * D + c];
        } else {
#pragma unroll
            for (int c = 0; c < D; ++c) e[c] = g.xo[(int64_t)k * D + c];
        }
        double s = 0.0;
#pragma unroll
        for (int c = 0; c < D; ++c) {
            row[t][c] = e[c] - x[c];
            s = fma(e[c] - x[c], e[c] - x[c], s);
        }
        row[t][D] = 1.0 / s;
        acc[t] = 0.0;
    }
    __syncthreads();
    double V = 0.0;
    const uint64_t first = (uint64_t)i * (uint64_t)ndir;
    const int64_t step = blockDim.x;
    for (int64_t q = 0; q < ndir;) {   // uniform over the workgroup
        const int64_t q0 = q + threadIdx.x, left = ndir - q;
        if (left > 2 * step) {
            V += hv_mc_sweep<D, 4>(row, K, acc, first, q0, step, ndir, seed);
            q += 4 * step;
        } else if (left > step) {
            V += hv_mc_sweep<D, 2>(row, K, acc, first, q0, step, ndir, seed);
            q += 2 * step;
        } else {
            if (q0 < ndir) V += hv_mc_sweep<D, 1>(row, K, acc, first, q0, step, ndir, seed);
            q += step;
        }
    }
    vred[threadIdx.x] = V;
    __syncthreads();
    for (int s = blockDim.x / 2; s > 0; s >>= 1) {
        if ((int)threadIdx.x < s) vred[threadIdx.x] += vred[threadIdx.x + s];
        __syncthreads();
    }
    if (threadIdx.x == 0) vol[i] = vred[0] * cvol / (double)ndir;
    for (int t = threadIdx.x; t < K; t += blockDim.x) area[b + t] = acc[t] * carea / (double)ndir;
}

// symmetrise each generator-generator interface with the neighbour's estimate (pairs k < i)
template <int D>
__global__ void k_mc_sym(IntGeo g, const int64_t* __restrict__ ptr, const uint64_t* __restrict__ pkey, int64_t npair,
                         double* __restrict__ vol, double* __restrict__ area) {
    const int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= npair) return;
    const int i = (int)(pkey[t] >> 32), k = (int)(pkey[t] & 0xffffffffull);
    if (k >= g.N || k >= i || i >= g.nreal) return;
    int64_t lo = ptr[k], hi = ptr[k + 1];
    while (lo < hi) {
        const int64_t mid = (lo + hi) >> 1;
        if ((int)(pkey[mid] & 0xffffffffull) < i) lo = mid + 1;
        else hi = mid;
    }
    if (lo >= ptr[k + 1] || (int)(pkey[lo] & 0xffffffffull) != i) return;
    const double old = area[t], neigh = area[lo];
    const double nw = fabs(neigh) < old * 1.0e-10 ? old : 0.5 * (old + neigh);
    double s = 0.0;
#pragma unroll
    for (int c = 0; c < D; ++c) {
        const double d2 = g.xo[(int64_t)i * D + c] - g.xo[(int64_t)k * D + c];
        s = fma(d2, d2, s);
    }
    const double factor = 0.5 * sqrt(s) / (double)D;
    atomicAdd(&vol[k], (nw - neigh) * factor);
    atomicAdd(&vol[i], (nw - old) * factor);
    area[t] = nw;
    area[lo] = nw;
}

// ---- dense ids -----------------------------------------------------------------------------
// Face keys pack 21 bits per id.  The face passes run on a dense numbering of the ids that
// occur in the mesh's keys (order-preserving, so sorted keys stay sorted): with periodic images
// the working set can exceed 2^21 generators while far fewer of them touch a walked cell.
// dense[i] (exclusive prefix sum of used) -> gid[dense] = i for the used ids
__global__ void k_dense_inverse(const int* __restrict__ used, const int* __restrict__ dense, int n, int* __restrict__ gid) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n && used[i]) gid[dense[i]] = i;
}

// generator rows and planes of the dense numbering: dense ids below ngen are generators
template <int D>
__global__ void k_dense_geo(const int* __restrict__ gid, int nused, int ngen, int N, const double* __restrict__ xo,
                            const double* __restrict__ pn, const double* __restrict__ ph, double* __restrict__ xd,
                            double* __restrict__ pnd, double* __restrict__ phd) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= nused) return;
    const int o = gid[i];
    if (i < ngen) {
#pragma unroll
        for (int k = 0; k < D; ++k) xd[(int64_t)i * D + k] = xo[(int64_t)o * D + k];
    } else {
        const int p = o - N, q = i - ngen;
#pragma unroll
        for (int k = 0; k < D; ++k) pnd[q * D + k] = pn[p * D + k];
        phd[q] = ph[p];
    }
}

// ---- host driver -------------------------------------------------------------------------

static int64_t binom(int n, int k) {
    int64_t r = 1;
    for (int i = 1; i <= k; ++i) r = r * (n - k + i) / i;
    return r;
}

struct Integrand {
    int nf;
    hv_integrand_fn fn;
    void* user;
};

// f at npts device points (D x npts) -> device values (nf x npts), through the caller's function
static int eval_integrand(hv_ctx* c, const Integrand* fi, int D, const double* dpts, int64_t npts, double* dvals) {
    if (npts == 0) return HV_OK;
    std::vector<double> hp((size_t)npts * D), hv((size_t)npts * fi->nf, 0.0);
    HVCK(hipMemcpyAsync(hp.data(), dpts, sizeof(double) * hp.size(), hipMemcpyDeviceToHost, c->stream));
    HVCK(hipStreamSynchronize(c->stream));
    fi->fn(fi->user, npts, hp.data(), hv.data());
    HVCK(hipMemcpyAsync(dvals, hv.data(), sizeof(double) * hv.size(), hipMemcpyHostToDevice, c->stream));
    HVCK(hipStreamSynchronize(c->stream));
    return HV_OK;
}

// Host state of one chunk's face passes.
struct FacePass {
    const int* vk = nullptr;        // the chunk's vertices, canonical order
    const double* vc = nullptr;
    const double* fv = nullptr;     // integrand at the vertices
    int nv = 0;
    const uint8_t* cmask = nullptr;
    const uint32_t* hid = nullptr;
    int hb = 0, zb = 0;             // hash and id bits of a grouping key
    int nf = 0;
    int* bad = nullptr;
    int* cnt = nullptr;             // device counters: pairs of real faces, faces, runs to fix
    // the faces of the last pass
    HvFaces F{};
    int nface = 0;
    double *cen = nullptr, *J = nullptr;
};

// Faces of pass M and their measures from those of pass M + 1 (the vertices for M == D)
template <int D, int M>
static int face_pass(hv_ctx* c, const IntGeo& g, FacePass& P) {
    const int nt = M == D ? P.nv : P.nface;
    const int64_t tot = (int64_t)nt * (M + 1);
    if (tot >= (1ll << 31)) return hv_fail(c, HV_ERR_CAPACITY, "too many face incidences for one pass");
    const size_t T = (size_t)std::max<int64_t>(tot, 1);
    uint32_t* key = iget<uint32_t>(c, "i_key", T);
    uint32_t* key2 = iget<uint32_t>(c, "i_key2", T);
    uint32_t* pay = iget<uint32_t>(c, "i_pay", T);
    uint8_t* head = iget<uint8_t>(c, "i_head", T);
    if (!key || !key2 || !pay || !head) return hv_fail(c, HV_ERR_DEVICE, "out of device memory (faces)");
    const HvFaces F1 = P.F;
    HVCK(hipMemsetAsync(P.cnt, 0, 4 * sizeof(int), c->stream));
    int nface = 0;
    HvPairs L{};
    if (tot > 0) {
        k_pair_emit<D, M><<<nblk(nt, 256), 256, 0, c->stream>>>(P.vk, F1, nt, g.N, P.cmask, P.hid, P.hb, key);
        HVCK(hipGetLastError());
        const unsigned nbits = (unsigned)(P.zb + P.hb);
        const rocprim::counting_iterator<uint32_t> it(0u);
        size_t tb = 0, tb2 = 0;
        HVCK(rocprim::radix_sort_pairs(nullptr, tb, key, key2, it, pay, T, 0u, nbits, c->stream));
        int* jl = (int*)key;   // free once sorted
        const hipcub::CountingInputIterator<int> pos(0);
        int* start0 = iget<int>(c, "i_start", T + 1);
        if (!start0) return hv_fail(c, HV_ERR_DEVICE, "out of device memory (faces)");
        HVCK(hipcub::DeviceSelect::Flagged(nullptr, tb2, pos, head, start0, P.cnt + 1, (int)tot, c->stream));
        void* tmp = c->pool->get("i_tmp", std::max(tb, tb2), false, c->stream);
        if (!tmp) return hv_fail(c, HV_ERR_DEVICE, "out of device memory (sort)");
        HVCK(rocprim::radix_sort_pairs(tmp, tb, key, key2, it, pay, T, 0u, nbits, c->stream));
        // HV_NO_FACE pairs lie at the end: their first position, or all of them real
        HVCK(hipMemsetD32Async((hipDeviceptr_t)P.cnt, (int)tot, 1, c->stream));
        int* runs = start0;    // room for one per pair, read before the faces' starts are written
        k_pair_heads<D, M><<<nblk(tot, 256), 256, 0, c->stream>>>(key2, pay, tot, P.vk, F1, head, jl, P.cnt, runs, P.cnt + 2);
        HVCK(hipGetLastError());
        k_pair_fix<D, M><<<1024, 64, 0, c->stream>>>(key2, tot, P.vk, F1, runs, P.cnt + 2, pay, head, jl);
        HVCK(hipGetLastError());
        HVCK(hipcub::DeviceSelect::Flagged(tmp, tb2, pos, head, start0, P.cnt + 1, (int)tot, c->stream));
        HVCK(hipMemcpyAsync(&nface, P.cnt + 1, sizeof(int), hipMemcpyDeviceToHost, c->stream));
        HVCK(hipStreamSynchronize(c->stream));
        L = HvPairs{pay, jl, start0, P.cnt, nface};
    }
    // tables of this pass and the one before alternate
    const std::string sfx = (M & 1) ? "a" : "b";
    auto nm = [&](const char* s) { return std::string(s) + sfx; };
    const size_t nfc = (size_t)std::max(nface, 1);
    HvFaces F;
    F.klo = iget<uint64_t>(c, nm("i_klo").c_str(), nfc);
    F.khi = M > 3 ? iget<uint64_t>(c, nm("i_khi").c_str(), nfc) : nullptr;
    F.f = iget<HvFace>(c, nm("i_face").c_str(), nfc);
    if (!F.klo || (M > 3 && !F.khi) || !F.f) return hv_fail(c, HV_ERR_DEVICE, "out of device memory (faces)");
    double *cen = nullptr, *J = nullptr;
    if (P.nf) {
        cen = iget<double>(c, nm("i_cen").c_str(), nfc * D);
        J = iget<double>(c, nm("i_J").c_str(), nfc * P.nf);
        if (!cen || !J) return hv_fail(c, HV_ERR_DEVICE, "out of device memory (integrand)");
    }
    if (nface > 0) {
        if constexpr (M == D) {
            k_edge_measure<D><<<nblk(nface, 256), 256, 0, c->stream>>>(L, P.vk, P.vc, F, P.bad);
            HVCK(hipGetLastError());
            if (P.nf) k_edge_int<D><<<nblk(nface, 256), 256, 0, c->stream>>>(L, F, P.vc, P.fv, P.nf, cen, J);
        } else {
            constexpr int W = hv_face_lanes(D, M);
            k_face_measure<D, M, W><<<hv_face_blocks(nface, W), 128, 0, c->stream>>>(g, L, P.vk, P.vc, F1, F, P.bad);
            HVCK(hipGetLastError());
            if (P.nf)
                k_face_int<D, M, W><<<hv_face_blocks(nface, W), 128, 0, c->stream>>>(g, L, P.vk, F1, P.cen, P.J, P.nf, cen, J,
                                                                                    P.bad);
        }
        HVCK(hipGetLastError());
    }
    P.F = F;
    P.nface = nface;
    P.cen = cen;
    P.J = J;
    if constexpr (M > 2) return face_pass<D, M - 1>(c, g, P);
    return HV_OK;
}

// pairs of the largest pass per vertex: C(d + 1, m + 1) faces T at most, each of at least
// (dimension of T) + 1 vertices, with m + 1 subsets
static double pairs_bound(int D) {
    double most = D + 1.0;
    for (int m = 2; m < D; ++m) most = std::max(most, (double)binom(D + 1, m + 1) * (m + 1) / (double)(D - m + 1));
    return most;
}

// faces of the tessellation, all passes; leaves the sorted (cell, neighbour) rows with areas.
// fi (optional): also the integrals of the rows' interfaces (*rint, npair x nf) by the
// reference's rule (see k_face_int)
template <int D>
static int facet_rows(hv_ctx* c, const hv_mesh* mesh, const IntGeo& g0, uint64_t*& pkey, double*& parea, int64_t& npair,
                      const Integrand* fi = nullptr, double** rint = nullptr) {
    const int nv = (int)mesh->nv;
    const size_t nv1 = (size_t)std::max(nv, 1);
    int* vk = iget<int>(c, "i_vk", nv1 * (D + 1));
    double* vc = iget<double>(c, "i_vc", nv1 * D);
    int* bad = iget<int>(c, "i_bad", 1);
    int* cnt = iget<int>(c, "i_cnt", 4);
    if (!vk || !vc || !bad || !cnt) return hv_fail(c, HV_ERR_DEVICE, "out of device memory (integration)");
    HVCK(hipMemsetAsync(bad, 0, sizeof(int), c->stream));
    const int* mids = (const int*)mesh->ids.p;
    const int* mkey = (const int*)mesh->key.p;
    IntGeo g = g0;          // the face passes' geometry, in dense ids
    int* gid = nullptr;     // dense id -> the caller's id
    int* dense = nullptr;   // caller's id -> dense id (exclusive prefix sum of used)
    uint32_t* hid = nullptr;
    const int nid = g0.N + g0.P;
    int ngen = 0, nused = 0, zb = 1;
    {
        // dense ids of the generators and planes that occur in the keys
        int* used = iget<int>(c, "i_used", (size_t)nid + 1);
        dense = iget<int>(c, "i_dense", (size_t)nid + 1);
        if (!used || !dense) return hv_fail(c, HV_ERR_DEVICE, "out of device memory (integration)");
        HVCK(hipMemsetAsync(used, 0, sizeof(int) * ((size_t)nid + 1), c->stream));
        if (nv) {
            k_mark_used<D><<<nblk((int64_t)nv * (D + 1), 256), 256, 0, c->stream>>>(mids, nv, mkey, used);
            HVCK(hipGetLastError());
        }
        size_t tbs = 0;
        HVCK(hipcub::DeviceScan::ExclusiveSum(nullptr, tbs, used, dense, nid + 1, c->stream));
        void* tmps = c->pool->get("i_stmp", tbs, false, c->stream);
        if (!tmps) return hv_fail(c, HV_ERR_DEVICE, "out of device memory (scan)");
        HVCK(hipcub::DeviceScan::ExclusiveSum(tmps, tbs, used, dense, nid + 1, c->stream));
        int hcnt[2] = {0, 0};   // used ids below N (generators), used ids in all
        HVCK(hipMemcpyAsync(&hcnt[0], dense + g0.N, sizeof(int), hipMemcpyDeviceToHost, c->stream));
        HVCK(hipMemcpyAsync(&hcnt[1], dense + nid, sizeof(int), hipMemcpyDeviceToHost, c->stream));
        HVCK(hipStreamSynchronize(c->stream));
        ngen = hcnt[0];
        nused = hcnt[1];
        if (nused >= (int)HV_F21)
            return hv_fail(c, HV_ERR_UNSUPPORTED, "more than 2^21 - 2 generators and planes occur in the mesh (21-bit face keys)");
        while ((1 << zb) < nused + 1) ++zb;   // every dense id is below 2^zb - 1
        gid = iget<int>(c, "i_gid", (size_t)std::max(1, nused));
        hid = iget<uint32_t>(c, "i_hid", (size_t)std::max(1, nused));
        double* xd = iget<double>(c, "i_xd", (size_t)std::max(1, ngen) * D);
        double* pnd = iget<double>(c, "i_pnd", (size_t)std::max(1, nused - ngen) * D);
        double* phd = iget<double>(c, "i_phd", (size_t)std::max(1, nused - ngen));
        if (!gid || !hid || !xd || !pnd || !phd) return hv_fail(c, HV_ERR_DEVICE, "out of device memory (integration)");
        k_dense_inverse<<<nblk(nid, 256), 256, 0, c->stream>>>(used, dense, nid, gid);
        HVCK(hipGetLastError());
        if (nused) {
            k_dense_geo<D><<<nblk(nused, 256), 256, 0, c->stream>>>(gid, nused, ngen, g0.N, g0.xo, g0.pn, g0.ph, xd, pnd, phd);
            HVCK(hipGetLastError());
            k_id_hash<<<nblk(nused, 256), 256, 0, c->stream>>>(gid, nused, hid);
            HVCK(hipGetLastError());
        }
        g.N = ngen;
        g.P = nused - ngen;
        g.nreal = g0.nreal;
        g.xo = xd;
        g.pn = pnd;
        g.ph = phd;
        // the live vertices in a numbering fixed by the vertex set (not by the walk's insertion
        // order), so that apexes and summation orders are reproducible: sorted by key, packed in
        // words of as many ids as fit, least significant word first
        uint64_t* w0 = iget<uint64_t>(c, "i_w0", nv1);
        uint64_t* w1 = iget<uint64_t>(c, "i_w1", nv1);
        int* pa = iget<int>(c, "i_vpa", nv1);
        int* pb = iget<int>(c, "i_vpb", nv1);
        if (!w0 || !w1 || !pa || !pb) return hv_fail(c, HV_ERR_DEVICE, "out of device memory (integration)");
        if (nv) {
            size_t tb = 0;
            HVCK(hipcub::DeviceRadixSort::SortPairs(nullptr, tb, w0, w1, pa, pb, nv, 0, 64, c->stream));
            void* tmp = c->pool->get("i_vtmp", tb, false, c->stream);
            if (!tmp) return hv_fail(c, HV_ERR_DEVICE, "out of device memory (sort)");
            const int per = 64 / zb;
            const int* order = nullptr;
            for (int e = D + 1; e > 0;) {
                const int n = order ? per : ((e % per) ? e % per : per);
                e -= n;
                k_vkey_word<D><<<nblk(nv, 256), 256, 0, c->stream>>>(mids, nv, mkey, dense, order, e, n, zb, w0, pa);
                HVCK(hipGetLastError());
                int* src = order ? pb : pa;
                int* dst = order ? pa : pb;
                HVCK(hipcub::DeviceRadixSort::SortPairs(tmp, tb, w0, w1, src, dst, nv, 0, n * zb, c->stream));
                pa = src;
                pb = dst;
                order = pb;
            }
            k_int_permute<D><<<nblk(nv, 256), 256, 0, c->stream>>>(order, nv, mids, mkey, dense, (const double*)mesh->x.p, vk, vc);
            HVCK(hipGetLastError());
        }
    }
    const int nf = fi ? fi->nf : 0;
    double* fv = nullptr;   // f at the vertices (edge ends)
    if (fi) {
        fv = iget<double>(c, "i_fv", nv1 * nf);
        if (!fv) return hv_fail(c, HV_ERR_DEVICE, "out of device memory (integrand)");
        int rc = eval_integrand(c, fi, D, vc, nv, fv);
        if (rc) return rc;
    }
    // Cells to integrate (dense ids), taken a chunk at a time.  A chunk's face passes hold the
    // vertices of its cells only: a face with one of the chunk's cells has all its vertices
    // there, and so do its sub-faces.  A facet of cells in two chunks is measured in both from
    // the same sub-faces in the same order (by their smallest id and hash), so the two values are
    // identical.  One chunk unless a pass would exceed HV_INC_BUDGET pairs.
    std::vector<int> hcell;
    {
        std::vector<int> hd((size_t)g0.nreal + 1);
        HVCK(hipMemcpyAsync(hd.data(), dense, sizeof(int) * ((size_t)g0.nreal + 1), hipMemcpyDeviceToHost, c->stream));
        HVCK(hipStreamSynchronize(c->stream));
        const auto add = [&](int i) -> bool {
            if (hd[(size_t)i + 1] == hd[(size_t)i]) return false;   // no vertex holds cell i
            hcell.push_back(hd[(size_t)i]);
            return true;
        };
        if (mesh->cells) {
            for (int i : *mesh->cells)
                if (!add(i)) return hv_fail(c, HV_ERR_STATE, "a listed cell of the mesh has no vertex");
        } else {
            hcell.reserve((size_t)g0.nreal);
            for (int i = 0; i < g0.nreal; ++i)
                if (!add(i)) return hv_fail(c, HV_ERR_STATE, "a cell of the mesh has no vertex");
        }
    }
    const int ncell = (int)hcell.size();
    const double cmax = pairs_bound(D);
    int nchunk = 1;
    if ((double)nv * cmax > (double)HV_INC_BUDGET)
        nchunk = (int)std::min<int64_t>(std::max(ncell, 1), (int64_t)std::ceil(1.3 * (double)nv * cmax / (double)HV_INC_BUDGET));
    if (nchunk > 1) {
        // chunks of nearby cells (Morton order of the generators), so that few vertices are in two
        std::vector<double> hx((size_t)std::max(1, ngen) * D);
        HVCK(hipMemcpyAsync(hx.data(), g.xo, sizeof(double) * (size_t)ngen * D, hipMemcpyDeviceToHost, c->stream));
        HVCK(hipStreamSynchronize(c->stream));
        double lo[D], hi[D];
        for (int k = 0; k < D; ++k) { lo[k] = INFINITY; hi[k] = -INFINITY; }
        for (int i : hcell)
            for (int k = 0; k < D; ++k) { lo[k] = std::min(lo[k], hx[(size_t)i * D + k]); hi[k] = std::max(hi[k], hx[(size_t)i * D + k]); }
        constexpr int B = 60 / D;
        std::vector<std::pair<uint64_t, int>> code(ncell);
        for (int q = 0; q < ncell; ++q) {
            const int i = hcell[q];
            uint64_t z = 0;
            uint32_t u[D];
            for (int k = 0; k < D; ++k) {
                const double w = hi[k] > lo[k] ? (hx[(size_t)i * D + k] - lo[k]) / (hi[k] - lo[k]) : 0.0;
                u[k] = (uint32_t)std::min(std::max(w, 0.0) * (double)((1u << B) - 1), (double)((1u << B) - 1));
            }
            for (int b = B - 1; b >= 0; --b)
                for (int k = 0; k < D; ++k) z = (z << 1) | ((u[k] >> b) & 1u);
            code[q] = {z, i};
        }
        std::sort(code.begin(), code.end());
        for (int q = 0; q < ncell; ++q) hcell[q] = code[q].second;
    }
    // no mask when every generator that occurs is a cell of the one chunk
    const bool whole = nchunk == 1 && !mesh->cells;   // every vertex takes part: no selection
    const bool every = whole && ncell == ngen;
    uint8_t* cmask = nullptr;
    int* dchunk = nullptr;
    if (!every) {
        cmask = iget<uint8_t>(c, "i_cmask", (size_t)std::max(1, nused));
        dchunk = iget<int>(c, "i_chunk", (size_t)std::max(1, ncell));
        if (!cmask || !dchunk) return hv_fail(c, HV_ERR_DEVICE, "out of device memory (integration)");
        if (ncell) HVCK(hipMemcpyAsync(dchunk, hcell.data(), sizeof(int) * ncell, hipMemcpyHostToDevice, c->stream));
    }
    auto set_chunk = [&](int q, int nch) -> int {
        if (every) return HV_OK;
        const int cb = (int)((int64_t)ncell * q / nch), ce = (int)((int64_t)ncell * (q + 1) / nch);
        HVCK(hipMemsetAsync(cmask, 0, (size_t)std::max(1, nused), c->stream));
        if (ce > cb) {
            k_set_mask<<<nblk(ce - cb, 256), 256, 0, c->stream>>>(dchunk + cb, ce - cb, cmask);
            HVCK(hipGetLastError());
        }
        return HV_OK;
    };
    int64_t nvc_max = nv;   // vertices of the largest chunk
    if (!whole && nchunk > 1) {
        // a vertex of cells in several chunks is in each of them: more chunks until every
        // chunk's passes fit (at most 2^31 - 1 pairs)
        unsigned long long* vcnt = iget<unsigned long long>(c, "i_vcnt", 1);
        if (!vcnt) return hv_fail(c, HV_ERR_DEVICE, "out of device memory (integration)");
        for (;;) {
            int64_t worst = 0;
            for (int q = 0; q < nchunk; ++q) {
                int rc = set_chunk(q, nchunk);
                if (rc) return rc;
                HVCK(hipMemsetAsync(vcnt, 0, sizeof(unsigned long long), c->stream));
                k_count_in_chunk<D><<<nblk(nv, 256), 256, 0, c->stream>>>(vk, nv, ngen, cmask, vcnt);
                HVCK(hipGetLastError());
                unsigned long long h = 0;
                HVCK(hipMemcpyAsync(&h, vcnt, sizeof(h), hipMemcpyDeviceToHost, c->stream));
                HVCK(hipStreamSynchronize(c->stream));
                worst = std::max<int64_t>(worst, (int64_t)h);
            }
            if ((double)worst * cmax < (double)(1ll << 31)) {
                nvc_max = worst;
                break;
            }
            if (nchunk >= ncell) return hv_fail(c, HV_ERR_CAPACITY, "too many face incidences for one cell");
            nchunk = std::min(ncell, 2 * nchunk);
        }
    }
    {
        // the per-pair buffers of the face passes at their largest size, once: growing them
        // between passes and chunks frees and maps tens of GB while the device idles
        if ((double)nvc_max * cmax >= (double)(1ll << 31)) return hv_fail(c, HV_ERR_CAPACITY, "too many face incidences for one pass");
        const size_t T = (size_t)std::max<int64_t>((int64_t)((double)nvc_max * cmax), 1);
        bool ok = true;
        for (const char* nmv : {"i_key", "i_key2", "i_pay"}) ok = ok && c->pool->reserve(nmv, 4 * T, c->stream);
        ok = ok && c->pool->reserve("i_head", T, c->stream) && c->pool->reserve("i_start", 4 * (T + 1), c->stream);
        if (!whole) {
            ok = ok && c->pool->reserve("i_vkc", sizeof(int) * (size_t)std::max<int64_t>(nvc_max, 1) * (D + 1), c->stream);
            ok = ok && c->pool->reserve("i_vcc", sizeof(double) * (size_t)std::max<int64_t>(nvc_max, 1) * D, c->stream);
        }
        if (!ok) return hv_fail(c, HV_ERR_DEVICE, "out of device memory (faces)");
        size_t tb = 0;
        const rocprim::counting_iterator<uint32_t> it(0u);
        HVCK(rocprim::radix_sort_pairs(nullptr, tb, (uint32_t*)nullptr, (uint32_t*)nullptr, it, (uint32_t*)nullptr, T, 0u, 32u,
                                       c->stream));
        if (!c->pool->reserve("i_tmp", tb, c->stream)) return hv_fail(c, HV_ERR_DEVICE, "out of device memory (sort)");
    }
    int64_t ntot = 0;   // row slots of the chunks so far
    uint64_t* rk = nullptr;
    double *ra = nullptr, *ri = nullptr;
    for (int q = 0; q < nchunk; ++q) {
        {
            int rc = set_chunk(q, nchunk);
            if (rc) return rc;
        }
        FacePass P;
        P.vk = vk;
        P.vc = vc;
        P.fv = fv;
        P.nv = nv;
        P.cmask = cmask;
        P.hid = hid;
        P.hb = std::min(HV_GROUP_HASH, 32 - zb);
        P.zb = zb;
        P.nf = nf;
        P.bad = bad;
        P.cnt = cnt;
        if (!whole) {
            // the vertices holding a cell of the chunk, in the canonical order
            uint8_t* vflag = iget<uint8_t>(c, "i_vflag", nv1);
            int* vsel = iget<int>(c, "i_vsel", nv1);
            if (!vflag || !vsel) return hv_fail(c, HV_ERR_DEVICE, "out of device memory (integration)");
            int nvc = 0;
            if (nv) {
                k_vert_in_chunk<D><<<nblk(nv, 256), 256, 0, c->stream>>>(vk, nv, ngen, cmask, vflag);
                HVCK(hipGetLastError());
                size_t tbf = 0;
                const hipcub::CountingInputIterator<int> pos(0);
                HVCK(hipcub::DeviceSelect::Flagged(nullptr, tbf, pos, vflag, vsel, cnt, nv, c->stream));
                void* tmpf = c->pool->get("i_tmpf", tbf, false, c->stream);
                if (!tmpf) return hv_fail(c, HV_ERR_DEVICE, "out of device memory (select)");
                HVCK(hipcub::DeviceSelect::Flagged(tmpf, tbf, pos, vflag, vsel, cnt, nv, c->stream));
                HVCK(hipMemcpyAsync(&nvc, cnt, sizeof(int), hipMemcpyDeviceToHost, c->stream));
                HVCK(hipStreamSynchronize(c->stream));
            }
            int* vk2 = iget<int>(c, "i_vkc", (size_t)std::max(1, nvc) * (D + 1));
            double* vc2 = iget<double>(c, "i_vcc", (size_t)std::max(1, nvc) * D);
            double* fv2 = fi ? iget<double>(c, "i_fvc", (size_t)std::max(1, nvc) * nf) : nullptr;
            if (!vk2 || !vc2 || (fi && !fv2)) return hv_fail(c, HV_ERR_DEVICE, "out of device memory (integration)");
            if (nvc) {
                k_int_subset<D><<<nblk(nvc, 256), 256, 0, c->stream>>>(vsel, nvc, vk, vc, fv, nf, vk2, vc2, fv2);
                HVCK(hipGetLastError());
            }
            P.vk = vk2;
            P.vc = vc2;
            P.fv = fv2;
            P.nv = nvc;
        }
        int rc = face_pass<D, D>(c, g, P);
        if (rc) return rc;
        const int nface = P.nface;   // facets
        double* I = nullptr;
        if (fi) {
            double* fc = iget<double>(c, "i_fc", (size_t)std::max(nface, 1) * nf);
            I = iget<double>(c, "i_If", (size_t)std::max(nface, 1) * nf);
            if (!fc || !I) return hv_fail(c, HV_ERR_DEVICE, "out of device memory (integrand)");
            rc = eval_integrand(c, fi, D, P.cen, nface, fc);
            if (rc) return rc;
            if (nface > 0) {
                k_facet_int<D><<<nblk(nface, 256), 256, 0, c->stream>>>(nface, P.J, fc, P.F.f, nf, I);
                HVCK(hipGetLastError());
            }
        }
        // this chunk's rows after the rows of the chunks before
        const size_t slots = (size_t)std::max<int64_t>(ntot + 2 * (int64_t)nface, 1);
        rk = (uint64_t*)c->pool->get("i_rk", sizeof(uint64_t) * slots, ntot > 0, c->stream);
        ra = (double*)c->pool->get("i_ra", sizeof(double) * slots, ntot > 0, c->stream);
        ri = fi ? (double*)c->pool->get("i_ri", sizeof(double) * slots * nf, ntot > 0, c->stream) : nullptr;
        if (!rk || !ra || (fi && !ri)) return hv_fail(c, HV_ERR_DEVICE, "out of device memory (rows)");
        if (nface > 0) {
            k_facet_rows<<<nblk(nface, 256), 256, 0, c->stream>>>(nface, P.F, ngen, cmask, zb, rk + ntot, ra + ntot, I, nf,
                                                                  fi ? ri + ntot * nf : nullptr);
            HVCK(hipGetLastError());
        }
        ntot += 2 * (int64_t)nface;
    }
    // rows of all chunks, sorted by (cell, neighbour), in the caller's ids
    if (ntot >= (1ll << 31)) return hv_fail(c, HV_ERR_CAPACITY, "too many rows");
    const size_t nr = (size_t)std::max<int64_t>(ntot, 1);
    uint64_t* rk2 = iget<uint64_t>(c, "i_rk2", nr);
    int* rpb = iget<int>(c, "i_rpb", nr);
    pkey = iget<uint64_t>(c, "i_pkey", nr);
    parea = iget<double>(c, "i_parea", nr);
    if (fi) *rint = iget<double>(c, "i_rint", nr * nf);
    if (!rk2 || !rpb || !pkey || !parea || (fi && !*rint)) return hv_fail(c, HV_ERR_DEVICE, "out of device memory (rows)");
    int hres[2] = {0, 0};   // flags, rows
    HVCK(hipMemsetAsync(cnt, 0, sizeof(int), c->stream));
    if (ntot > 0) {
        // 2 zb bits and the one above them, set in the slots of no row only
        size_t tbr = 0;
        const rocprim::counting_iterator<int> it(0);
        const unsigned nbits = (unsigned)std::min(2 * zb + 1, 64);
        HVCK(rocprim::radix_sort_pairs(nullptr, tbr, rk, rk2, it, rpb, (size_t)ntot, 0u, nbits, c->stream));
        void* tmpr = c->pool->get("i_tmpr", tbr, false, c->stream);
        if (!tmpr) return hv_fail(c, HV_ERR_DEVICE, "out of device memory (sort)");
        HVCK(rocprim::radix_sort_pairs(tmpr, tbr, rk, rk2, it, rpb, (size_t)ntot, 0u, nbits, c->stream));
        k_rows_out<<<nblk(ntot, 256), 256, 0, c->stream>>>(rk2, rpb, ntot, zb, gid, ra, ri, nf, pkey, parea,
                                                          fi ? *rint : nullptr, cnt);
        HVCK(hipGetLastError());
    }
    HVCK(hipMemcpyAsync(&hres[0], bad, sizeof(int), hipMemcpyDeviceToHost, c->stream));
    HVCK(hipMemcpyAsync(&hres[1], cnt, sizeof(int), hipMemcpyDeviceToHost, c->stream));
    HVCK(hipStreamSynchronize(c->stream));
    npair = hres[1];
    if (hres[0]) return hv_fail(c, HV_ERR_DEGENERATE, "a face is not in general position (integration)");
    return HV_OK;
}

// ---- neighbour rows without face measures (the Monte-Carlo integrators) -------------------
// Cells i and k are neighbours when i and k occur together in a vertex key (src/neighbors.jl:
// 219-251; general position).  Every unordered pair (a < b, a a generator) of every live
// vertex key goes into a device hash set; the set's pairs are counted by cell, (a, b) and (b, a),
// placed in the cells' segments and each segment put in order by a wavefront, which gives the rows
// facet_rows leaves (keys (cell << 32) | neighbour).  (Compacting, mirroring and sorting all rows
// together took some 30 launches and three more waits: 4D N=20k, 1 000 directions, 1.76 -> 1.55 ms a call.)
constexpr uint64_t HV_PAIR_EMPTY = ~0ull;

template <int D>
__global__ void k_pair_insert(const int* __restrict__ ids, int nv, const int* __restrict__ key, int N,
                              unsigned long long* __restrict__ tab, uint64_t mask, int* __restrict__ full) {
    const int t = blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= nv) return;
    const int* k = key + (int64_t)ids[t] * (D + 1);
    int kk[D + 1];
#pragma unroll
    for (int j = 0; j <= D; ++j) kk[j] = k[j];
#pragma unroll
    for (int a = 0; a < D; ++a) {
        if (kk[a] >= N) break;   // planes sort last
#pragma unroll
        for (int b = a + 1; b <= D; ++b) {
            const unsigned long long pk = ((unsigned long long)kk[a] << 32) | (unsigned)kk[b];
            uint64_t h = hv_mix64(pk) & mask;
            bool done = false;
            for (uint64_t probe = 0; probe <= mask && !done; ++probe) {
                const unsigned long long cur = tab[h];
                if (cur == pk) { done = true; break; }
                if (cur == HV_PAIR_EMPTY) {
                    const unsigned long long old = atomicCAS(&tab[h], HV_PAIR_EMPTY, pk);
                    if (old == HV_PAIR_EMPTY || old == pk) { done = true; break; }
                }
                h = (h + 1) & mask;
            }
            if (!done) atomicExch(full, 1);
        }
    }
}

// the counts as 64-bit numbers, for their running sum
struct CountRows {
    const int* cnt;
    struct Widen {
        const int* cnt;
        __host__ __device__ int64_t operator()(int i) const { return (int64_t)cnt[i]; }
    };
    hipcub::TransformInputIterator<int64_t, Widen, hipcub::CountingInputIterator<int>> begin() const {
        return {hipcub::CountingInputIterator<int>(0), Widen{cnt}};
    }
};

// host[0] set overflow, [1], [2] k_rows_most, [3] all rows
__global__ void k_rows_report(const int* __restrict__ res, const int64_t* __restrict__ total, unsigned long long* __restrict__ host) {
    if (threadIdx.x < 3) host[threadIdx.x] = (unsigned long long)res[threadIdx.x];
    if (threadIdx.x == 3) host[3] = (unsigned long long)*total;
}

// rows per cell of the set's pairs
__global__ __launch_bounds__(256) void k_rows_count(const unsigned long long* __restrict__ tab, int64_t n, int N,
                                                    int* __restrict__ cnt) {
    const int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= n || tab[t] == HV_PAIR_EMPTY) return;
    const int a = (int)(tab[t] >> 32), b = (int)(tab[t] & 0xffffffffull);
    atomicAdd(&cnt[a], 1);
    if (b < N) atomicAdd(&cnt[b], 1);
}

// the most rows of a cell: res[1] of all N, res[2] of the first nreal (the counts become the segments'
// cursors: zero)
__global__ __launch_bounds__(256) void k_rows_most(int* __restrict__ cnt, int N, int nreal, int* __restrict__ res) {
    int m = 0, r = 0;
    for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < N; i += gridDim.x * blockDim.x) {
        m = max(m, cnt[i]);
        if (i < nreal) r = max(r, cnt[i]);
        cnt[i] = 0;
    }
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) {
        m = max(m, __shfl_xor(m, off));
        r = max(r, __shfl_xor(r, off));
    }
    if ((threadIdx.x & 63) == 0) {
        if (m > 0) atomicMax(&res[1], m);
        if (r > 0) atomicMax(&res[2], r);
    }
}

__global__ __launch_bounds__(256) void k_rows_place(const unsigned long long* __restrict__ tab, int64_t n, int N,
                                                    const int64_t* __restrict__ ptr, int* __restrict__ cur,
                                                    uint64_t* __restrict__ rows) {
    const int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= n || tab[t] == HV_PAIR_EMPTY) return;
    const unsigned long long pk = tab[t];
    const int a = (int)(pk >> 32), b = (int)(pk & 0xffffffffull);
    rows[ptr[a] + atomicAdd(&cur[a], 1)] = pk;
    if (b < N) rows[ptr[b] + atomicAdd(&cur[b], 1)] = ((uint64_t)b << 32) | (unsigned)a;
}

// One wavefront per cell of at most HV_ROWS_SORT rows: distinct neighbours, so each one's place is the
// number of smaller ones.
constexpr int HV_ROWS_SORT = 512;
__global__ __launch_bounds__(256) void k_rows_sort(const int64_t* __restrict__ ptr, int N, uint64_t* __restrict__ rows) {
    __shared__ uint32_t list[4][HV_ROWS_SORT];
    const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
    const int i = blockIdx.x * 4 + wv;
    if (i >= N) return;   // no workgroup barrier below
    const int64_t b = ptr[i];
    const int K = (int)(ptr[i + 1] - b);
    for (int t = lane; t < K; t += 64) list[wv][t] = (uint32_t)rows[b + t];
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    for (int t = lane; t < K; t += 64) {
        const uint32_t k = list[wv][t];
        int at = 0;
        for (int q = 0; q < K; ++q) at += list[wv][q] < k ? 1 : 0;
        rows[b + at] = ((uint64_t)(uint32_t)i << 32) | k;
    }
}

// neighbours per cell, a generous bound for the hash-set size (d = 2..6, unit-cube densities)
static int64_t neighbours_bound(int D) {
    static const int nb[7] = {0, 0, 8, 24, 64, 160, 400};
    return nb[std::min(std::max(D, 2), 6)];
}

template <int D>
static int neighbor_rows(hv_ctx* c, const hv_mesh* mesh, uint64_t*& pkey, int64_t& npair, int64_t*& ptr, int* most = nullptr) {
    const int N = (int)c->N;
    const int nv = (int)mesh->nv;
    int* res = iget<int>(c, "n_full", 3);           // set overflow, k_rows_most
    int* cnt = iget<int>(c, "n_cnt", (size_t)N + 1);
    ptr = iget<int64_t>(c, "i_ptr", (size_t)N + 1);
    HvPinned pin(c->stream);
    if (!res || !cnt || !ptr || !pin.p) return hv_fail(c, HV_ERR_DEVICE, "out of device memory (neighbours)");
    size_t tb = 0;
    HVCK(hipcub::DeviceScan::ExclusiveSum(nullptr, tb, CountRows{cnt}.begin(), ptr, N + 1, c->stream));
    void* tmp = c->pool->get("n_tmp", tb, false, c->stream);
    if (!tmp) return hv_fail(c, HV_ERR_DEVICE, "out of device memory (neighbours)");
    // rows of the walked cells (images add the pairs of their vertices' other generators)
    const int64_t nrows = (int64_t)mesh->nreal * neighbours_bound(D) * (mesh->nreal < N ? 2 : 1);
    uint64_t tsize = 1024;
    while ((int64_t)tsize < nrows + 1024) tsize <<= 1;
    if (tsize > (1ull << 30)) return hv_fail(c, HV_ERR_CAPACITY, "too many cells for the neighbour set");
    unsigned long long* tab = nullptr;
    int hmost = 0;
    for (int attempt = 0;; ++attempt) {
        tab = iget<unsigned long long>(c, "n_tab", tsize);
        if (!tab) return hv_fail(c, HV_ERR_DEVICE, "out of device memory (neighbour set)");
        HVCK(hipMemsetAsync(tab, 0xff, tsize * sizeof(unsigned long long), c->stream));
        HVCK(hipMemsetAsync(cnt, 0, sizeof(int) * ((size_t)N + 1), c->stream));
        HVCK(hipMemsetAsync(res, 0, 3 * sizeof(int), c->stream));
        if (nv > 0) {
            k_pair_insert<D><<<nblk(nv, 256), 256, 0, c->stream>>>((const int*)mesh->ids.p, nv, (const int*)mesh->key.p,
                                                                   N, tab, tsize - 1, res);
            HVCK(hipGetLastError());
        }
        k_rows_count<<<nblk((int64_t)tsize, 256), 256, 0, c->stream>>>(tab, (int64_t)tsize, N, cnt);
        HVCK(hipGetLastError());
        HVCK(hipcub::DeviceScan::ExclusiveSum(tmp, tb, CountRows{cnt}.begin(), ptr, N + 1, c->stream));
        k_rows_most<<<std::min<unsigned>(nblk(N, 256), 256u), 256, 0, c->stream>>>(cnt, N, (int)mesh->nreal, res);
        HVCK(hipGetLastError());
        k_rows_report<<<1, 64, 0, c->stream>>>(res, ptr + N, pin.p);
        HVCK(hipGetLastError());
        HVCK(hipStreamSynchronize(c->stream));
        hmost = (int)pin.p[1];
        npair = (int64_t)pin.p[3];
        if (most) *most = (int)pin.p[2];
        if (!pin.p[0]) break;
        if (attempt >= 4 || tsize >= (1ull << 29)) return hv_fail(c, HV_ERR_CAPACITY, "neighbour set overflow");
        tsize <<= 2;
    }
    pin.settled();
    if (npair > (int64_t)INT32_MAX) return hv_fail(c, HV_ERR_CAPACITY, "more than 2^31 neighbour rows");
    uint64_t* rows = iget<uint64_t>(c, "n_rows", (size_t)std::max<int64_t>(npair, 1));
    if (!rows) return hv_fail(c, HV_ERR_DEVICE, "out of device memory (neighbours)");
    pkey = rows;
    if (npair > 0) {
        k_rows_place<<<nblk((int64_t)tsize, 256), 256, 0, c->stream>>>(tab, (int64_t)tsize, N, ptr, cnt, rows);
        HVCK(hipGetLastError());
        if (hmost <= HV_ROWS_SORT) {
            k_rows_sort<<<nblk(N, 4), 256, 0, c->stream>>>(ptr, N, rows);
            HVCK(hipGetLastError());
        } else {   // a cell of more neighbours than a wavefront sorts
            uint64_t* rows2 = iget<uint64_t>(c, "n_rows2", (size_t)npair);
            size_t ts = 0;
            HVCK(hipcub::DeviceRadixSort::SortKeys(nullptr, ts, rows, rows2, (int)npair, 0, 64, c->stream));
            tmp = c->pool->get("n_tmp", ts, false, c->stream);
            if (!rows2 || !tmp) return hv_fail(c, HV_ERR_DEVICE, "out of device memory (neighbours)");
            HVCK(hipcub::DeviceRadixSort::SortKeys(tmp, ts, rows, rows2, (int)npair, 0, 64, c->stream));
            pkey = rows2;
        }
    }
    return HV_OK;
}

template <int D>
static int make_geo(hv_ctx* c, const hv_mesh* mesh, IntGeo& g) {
    // the context is bound to the mesh's own working set and boundary (hv_bind_mesh)
    if (!mesh || mesh->D != D || mesh->N != c->N || !c->xw || c->xw != mesh->xw)
        return hv_fail(c, HV_ERR_STATE, "the context is not bound to the mesh's generators");
    {
        const char* why = nullptr;
        const int rc = hv_domain(c, D, &why);
        if (rc) return hv_fail(c, rc, why);
        if (c->dom_unbounded) return hv_fail(c, HV_ERR_UNSUPPORTED, "the integrators need a bounded domain");
    }
    g.N = (int)c->N;
    g.nreal = (int)mesh->nreal;
    g.P = c->P;
    g.xo = (const double*)c->xw->p;
    double* pn = iget<double>(c, "i_pn", (size_t)std::max(1, c->P) * D);
    double* ph = iget<double>(c, "i_ph", (size_t)std::max(1, c->P));
    if (!g.xo || !pn || !ph) return hv_fail(c, HV_ERR_DEVICE, "out of device memory (integration)");
    std::vector<double> hph(std::max(1, c->P), 0.0);
    for (int p = 0; p < c->P; ++p)
        for (int k = 0; k < D; ++k) hph[p] += c->pnormal[p * D + k] * c->pbase[p * D + k];
    if (c->P) {
        HVCK(hipMemcpyAsync(pn, c->pnormal.data(), sizeof(double) * c->P * D, hipMemcpyHostToDevice, c->stream));
        HVCK(hipMemcpyAsync(ph, hph.data(), sizeof(double) * c->P, hipMemcpyHostToDevice, c->stream));
    }
    g.pn = pn;
    g.ph = ph;
    return HV_OK;
}

// neighbours of the rows (cell << 32 | neighbour), 1-based
__global__ void k_row_nbr(const uint64_t* __restrict__ rows, int64_t n, int64_t* __restrict__ nbr) {
    const int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (t < n) nbr[t] = (int64_t)(rows[t] & 0xffffffffull) + 1;
}

template <int D>
static int finish(hv_ctx* c, int64_t ncell, const uint64_t* pkey, const double* area_d, const double* vol_d,
                  const int64_t* ptr_d, int64_t npair, float ms, hv_integral** out, int nf = 0,
                  const double* bulk_d = nullptr, const double* rint_d = nullptr) {
    // cells 0 .. ncell-1 (the originals) and their rows, which come first in the sorted order
    if (ncell < c->N) {
        HVCK(hipMemcpyAsync(&npair, ptr_d + ncell, sizeof(int64_t), hipMemcpyDeviceToHost, c->stream));
        HVCK(hipStreamSynchronize(c->stream));
    }
    std::unique_ptr<hv_integral> I(new hv_integral());
    I->N = ncell;
    I->rows = npair;
    I->device = c->device;
    I->nf = nf;
    I->ms = ms;
    size_t at = 0;
    auto part = [&](size_t bytes) { const size_t o = at; at += (bytes + 255) & ~(size_t)255; return o; };
    I->vol = part(sizeof(double) * ncell);
    I->ptr = part(sizeof(int64_t) * (ncell + 1));
    I->nbr = part(sizeof(int64_t) * npair);
    I->area = part(sizeof(double) * npair);
    I->bulk = part(sizeof(double) * ncell * nf);
    I->iface = part(sizeof(double) * npair * nf);
    I->bytes = at;
    I->dev.reset(new HvScratch(c->device, at, c->stream));
    hipMemcpyKind kind = hipMemcpyDeviceToDevice;
    if (I->dev->p) {
        I->base = (char*)I->dev->p;
    } else {
        I->dev.reset();
        I->host.resize(at);
        I->base = I->host.data();
        kind = hipMemcpyDeviceToHost;
    }
    auto put = [&](size_t off, const void* src, size_t bytes) {
        return bytes ? hipMemcpyAsync(I->base + off, src, bytes, kind, c->stream) : hipSuccess;
    };
    if (npair) {
        // in place for a host copy: the rows are this call's scratch
        int64_t* nbr = I->dev ? (int64_t*)(I->base + I->nbr) : (int64_t*)pkey;
        k_row_nbr<<<nblk(npair, 256), 256, 0, c->stream>>>(pkey, npair, nbr);
        HVCK(hipGetLastError());
        if (!I->dev) HVCK(put(I->nbr, nbr, sizeof(int64_t) * npair));
    }
    HVCK(put(I->area, area_d, sizeof(double) * npair));
    HVCK(put(I->vol, vol_d, sizeof(double) * ncell));
    HVCK(put(I->ptr, ptr_d, sizeof(int64_t) * (ncell + 1)));
    HVCK(put(I->bulk, bulk_d, sizeof(double) * ncell * nf));
    HVCK(put(I->iface, rint_d, sizeof(double) * npair * nf));
    HVCK(hipStreamSynchronize(c->stream));
    if (I->dev) I->dev->settled();   // it outlives the stream
    hv_integral_keep(I.get());
    *out = I.release();
    return HV_OK;
}

template <int D>
int hv_integrate_polytope_impl(hv_ctx* c, const hv_mesh* mesh, hv_integral** out) {
    return hv_integrate_polytope_f_impl<D>(c, mesh, 0, nullptr, nullptr, out);
}

template <int D>
int hv_integrate_polytope_f_impl(hv_ctx* c, const hv_mesh* mesh, int nf, hv_integrand_fn fn, void* user,
                                 hv_integral** out) {
    if (nf < 0 || nf > HV_MAXF || (nf > 0 && !fn)) return hv_fail(c, HV_ERR_ARG, "integrand: 0 < nf <= 8 and a function");
    IntGeo g;
    int rc = make_geo<D>(c, mesh, g);
    if (rc) return rc;
    HVCK(hipEventRecord(c->ev[0], c->stream));
    uint64_t* pkey = nullptr;
    double* parea = nullptr;
    int64_t npair = 0;
    Integrand spec{nf, fn, user};
    double* rint = nullptr;
    rc = facet_rows<D>(c, mesh, g, pkey, parea, npair, nf > 0 ? &spec : nullptr, &rint);
    if (rc) return rc;
    double* vol = iget<double>(c, "i_vol", c->N);
    int64_t* ptr = iget<int64_t>(c, "i_ptr", c->N + 1);
    if (!vol || !ptr) return hv_fail(c, HV_ERR_DEVICE, "out of device memory (volumes)");
    k_cell_volumes<D><<<nblk(c->N + 1, 256), 256, 0, c->stream>>>(g, pkey, parea, npair, vol, ptr);
    HVCK(hipGetLastError());
    double* bulk = nullptr;
    if (nf > 0) {
        // f at the generators (the cells' apexes), then the bulk integrals
        double* fx = iget<double>(c, "i_fx", (size_t)g.nreal * nf);
        bulk = iget<double>(c, "i_bulk", (size_t)g.nreal * nf);
        if (!fx || !bulk) return hv_fail(c, HV_ERR_DEVICE, "out of device memory (integrand)");
        rc = eval_integrand(c, &spec, D, g.xo, g.nreal, fx);
        if (rc) return rc;
        k_cell_bulk<D><<<nblk(g.nreal, 256), 256, 0, c->stream>>>(g, pkey, ptr, vol, rint, fx, nf, bulk);
        HVCK(hipGetLastError());
    }
    HVCK(hipEventRecord(c->ev[1], c->stream));
    HVCK(hipEventSynchronize(c->ev[1]));
    float ms = 0.f;
    HVCK(hipEventElapsedTime(&ms, c->ev[0], c->ev[1]));
    return finish<D>(c, g.nreal, pkey, parea, vol, ptr, npair, ms, out, nf, bulk, rint);
}

template <int D>
int hv_integrate_mc_impl(hv_ctx* c, const hv_mesh* mesh, int64_t ndir, uint64_t seed, hv_integral** out) {
    if (ndir < 1 || ndir > (1ll << 40)) return hv_fail(c, HV_ERR_ARG, "ndir must be positive");
    IntGeo g;
    int rc = make_geo<D>(c, mesh, g);
    if (rc) return rc;
    HVCK(hipEventRecord(c->ev[0], c->stream));
    uint64_t* pkey = nullptr;
    int64_t npair = 0;
    int64_t* ptr = nullptr;
    int most = 0;   // rows of a cell
    rc = neighbor_rows<D>(c, mesh, pkey, npair, ptr, &most);
    if (rc) return rc;
    double* vol = iget<double>(c, "i_vol", c->N);
    double* area = iget<double>(c, "i_marea", npair);
    if (!vol || !area) return hv_fail(c, HV_ERR_DEVICE, "out of device memory (volumes)");
    // one workgroup of 256 per cell, and a dispatch holds at most 2^32 work-items
    if ((int64_t)g.nreal > (1ll << 24) - 1)
        return hv_fail(c, HV_ERR_CAPACITY, "directional Monte Carlo: at most 2^24 - 1 cells per call");
    if (most > HV_MC_MAXK)
        return hv_fail(c, HV_ERR_CAPACITY, "a cell has more neighbours than the Monte-Carlo kernel holds");
    const double cvol = std::pow(M_PI, 0.5 * D) / std::tgamma(1.0 + 0.5 * D);
    HVCK(hipMemsetAsync(area, 0, sizeof(double) * std::max<int64_t>(npair, 1), c->stream));
    k_mc_cell<D><<<(unsigned)g.nreal, 256, 0, c->stream>>>(g, ptr, pkey, ndir, seed, cvol, D * cvol, vol, area);
    HVCK(hipGetLastError());
    k_mc_sym<D><<<nblk(npair, 256), 256, 0, c->stream>>>(g, ptr, pkey, npair, vol, area);
    HVCK(hipGetLastError());
    HVCK(hipEventRecord(c->ev[1], c->stream));
    HVCK(hipEventSynchronize(c->ev[1]));
    float ms = 0.f;
    HVCK(hipEventElapsedTime(&ms, c->ev[0], c->ev[1]));
    return finish<D>(c, g.nreal, pkey, area, vol, ptr, npair, ms, out);
}

// Point-sample counts -> volumes (sample fraction of the box) and interface areas.  A slab of
// width w beside an interface holds w * A - O(w^2) of volume (samples near the interface's
// own boundary see a third generator), so from the counts c1 (width eps) and c2 (width
// 2 eps): A = 2 A(eps) - A(2 eps) = V (2 c1 - c2 / 2) / (n eps), first order removed; a
// generator-generator interface averages the counts of its two sides.
__global__ void k_mcp_finish(int N, const int64_t* __restrict__ ptr, const uint64_t* __restrict__ pkey, int64_t npair,
                             const unsigned long long* __restrict__ ccnt, const unsigned long long* __restrict__ pcnt,
                             double n, double eps, double vbox, double* __restrict__ vol, double* __restrict__ area) {
    const int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (t < N) vol[t] = vbox * (double)ccnt[t] / n;
    if (t >= npair) return;
    const int i = (int)(pkey[t] >> 32), k = (int)(pkey[t] & 0xffffffffull);
    double c1 = (double)pcnt[2 * t], c2 = (double)pcnt[2 * t + 1];
    if (k < N) {
        int64_t lo = ptr[k], hi = ptr[k + 1];
        while (lo < hi) {
            const int64_t mid = (lo + hi) >> 1;
            if ((int)(pkey[mid] & 0xffffffffull) < i) lo = mid + 1;
            else hi = mid;
        }
        if (lo < ptr[k + 1] && (int)(pkey[lo] & 0xffffffffull) == i) {
            c1 = 0.5 * (c1 + (double)pcnt[2 * lo]);
            c2 = 0.5 * (c2 + (double)pcnt[2 * lo + 1]);
        }
    }
    area[t] = fmax(0.0, vbox * (2.0 * c1 - 0.5 * c2) / (n * eps));
}

template <int D>
int hv_integrate_mc_points_impl(hv_ctx* c, const hv_mesh* mesh, int64_t nsamples, uint64_t seed, double slab,
                                hv_integral** out) {
    if (nsamples < 1 || nsamples > (1ll << 40)) return hv_fail(c, HV_ERR_ARG, "nsamples must be positive");
    if (!(slab > 0.0)) slab = 0.03;
    IntGeo g;
    int rc = make_geo<D>(c, mesh, g);
    if (rc) return rc;
    HVCK(hipEventRecord(c->ev[0], c->stream));
    uint64_t* pkey = nullptr;
    int64_t npair = 0;
    int64_t* ptr = nullptr;
    rc = neighbor_rows<D>(c, mesh, pkey, npair, ptr);
    if (rc) return rc;
    double* vol = iget<double>(c, "i_vol", c->N);
    double* area = iget<double>(c, "i_marea", std::max<int64_t>(npair, 1));
    unsigned long long* ccnt = iget<unsigned long long>(c, "i_ccnt", c->N);
    unsigned long long* pcnt = iget<unsigned long long>(c, "i_pcnt", 2 * std::max<int64_t>(npair, 1));
    if (!vol || !area || !ccnt || !pcnt) return hv_fail(c, HV_ERR_DEVICE, "out of device memory (volumes)");
    HVCK(hipMemsetAsync(ccnt, 0, sizeof(unsigned long long) * c->N, c->stream));
    HVCK(hipMemsetAsync(pcnt, 0, sizeof(unsigned long long) * 2 * std::max<int64_t>(npair, 1), c->stream));
    int64_t n = 0;
    double eps = 0.0, vbox = 0.0;
    int64_t work = 0;
    double kms = 0.0;
    rc = hv_mc_points_impl<D>(c, nsamples, seed, slab, ptr, pkey, ccnt, pcnt, &n, &eps, &vbox, &work, &kms);
    if (rc) return rc;
    k_mcp_finish<<<nblk(std::max<int64_t>(c->N, npair), 256), 256, 0, c->stream>>>(
        g.nreal, ptr, pkey, npair, ccnt, pcnt, (double)n, eps, vbox, vol, area);
    HVCK(hipGetLastError());
    HVCK(hipEventRecord(c->ev[1], c->stream));
    HVCK(hipEventSynchronize(c->ev[1]));
    float ms = 0.f;
    HVCK(hipEventElapsedTime(&ms, c->ev[0], c->ev[1]));
    rc = finish<D>(c, g.nreal, pkey, area, vol, ptr, npair, ms, out);
    if (rc == HV_OK) {
        (*out)->work = work;
        (*out)->ms_kernel = kms;
    }
    return rc;
}

int hv_integral_work_impl(const hv_integral* I, int64_t* work, double* ms_kernel) {
    if (!I) return HV_ERR_ARG;
    if (work) *work = I->work;
    if (ms_kernel) *ms_kernel = I->ms_kernel;
    return HV_OK;
}

int hv_integral_counts_impl(const hv_integral* I, int64_t* ncells, int64_t* nnbr) {
    if (!I) return HV_ERR_ARG;
    if (ncells) *ncells = I->N;
    if (nnbr) *nnbr = I->rows;
    return HV_OK;
}

// Parts of the results, at offsets from their base, into the caller's memory (null: not wanted).  On
// the device they are adjacent: a small set comes in one copy through a pinned block.
struct IntegralPart {
    void* dst;
    size_t off, bytes;
};
static int integral_out(const hv_integral* I, const IntegralPart* part, int n) {
    std::lock_guard<std::mutex> own(I->mu);
    HvCopy list[4];
    int m = 0;
    size_t lo = ~(size_t)0, hi = 0;
    for (int k = 0; k < n; ++k) {
        if (!part[k].dst || part[k].bytes == 0) continue;
        list[m++] = {part[k].dst, I->base + part[k].off, part[k].bytes};
        lo = std::min(lo, part[k].off);
        hi = std::max(hi, part[k].off + part[k].bytes);
    }
    if (m == 0) return HV_OK;
    (void)hipSetDevice(I->device);
    if (!I->dev) {
        for (int k = 0; k < m; ++k) std::memcpy(list[k].dst, list[k].src, list[k].bytes);
        return HV_OK;
    }
    if (hi - lo <= HV_STAGE_BYTES) {
        HvLease pin(I->device);
        if (pin.base) {
            const hipStream_t st = hipStreamPerThread;
            if (hipMemcpyAsync(pin.base, I->base + lo, hi - lo, hipMemcpyDeviceToHost, st) != hipSuccess ||
                hipStreamSynchronize(st) != hipSuccess)
                return HV_ERR_DEVICE;
            for (int k = 0; k < m; ++k)
                std::memcpy(list[k].dst, pin.base + ((const char*)list[k].src - (I->base + lo)), list[k].bytes);
            return HV_OK;
        }
    }
    return hv_copies(I->device, true, list, m) == hipSuccess ? HV_OK : HV_ERR_DEVICE;
}

int hv_integral_export_f_impl(const hv_integral* I, int32_t* nf, double* bulk, double* iface) {
    if (!I) return HV_ERR_ARG;
    if (nf) *nf = I->nf;
    const IntegralPart part[2] = {{bulk, I->bulk, sizeof(double) * I->N * I->nf}, {iface, I->iface, sizeof(double) * I->rows * I->nf}};
    return integral_out(I, part, 2);
}

int hv_integral_export_impl(const hv_integral* I, double* vol, int64_t* nbr_ptr, int64_t* nbr, double* area,
                            double* ms) {
    if (!I) return HV_ERR_ARG;
    const IntegralPart part[4] = {{vol, I->vol, sizeof(double) * I->N},
                                  {nbr_ptr, I->ptr, sizeof(int64_t) * (I->N + 1)},
                                  {nbr, I->nbr, sizeof(int64_t) * I->rows},
                                  {area, I->area, sizeof(double) * I->rows}};
    if (ms) *ms = I->ms;
    return integral_out(I, part, 4);
}

// The integrals that may give their device memory back (never destroyed: one may be freed after this
// library's statics).  Whoever holds live_mu takes an integral's own lock by trying only.
static std::mutex live_mu;
static auto& live = *new std::set<hv_integral*>();

void hv_integral_keep(hv_integral* I) {
    std::lock_guard<std::mutex> lk(live_mu);
    live.insert(I);
}

void hv_integrals_to_host(int device) {
    std::lock_guard<std::mutex> lk(live_mu);
    for (hv_integral* I : live) {
        if (I->device != device) continue;
        std::unique_lock<std::mutex> own(I->mu, std::try_to_lock);
        if (!own.owns_lock() || !I->dev) continue;
        try {
            I->host.resize(I->bytes);
        } catch (...) {
            continue;   // no room there either
        }
        const HvCopy all{I->host.data(), I->base, I->bytes};
        if (hv_copies(device, true, &all, 1) != hipSuccess) {
            std::vector<char>().swap(I->host);
            continue;
        }
        I->base = I->host.data();
        I->dev.reset();
    }
}

void hv_integral_free_impl(hv_integral* I) {
    {
        std::lock_guard<std::mutex> lk(live_mu);
        live.erase(I);
    }
    delete I;
}

#define HV_IINST(D)                                                                                 \
    template int hv_integrate_polytope_impl<D>(hv_ctx*, const hv_mesh*, hv_integral**);          \
    template int hv_integrate_polytope_f_impl<D>(hv_ctx*, const hv_mesh*, int, hv_integrand_fn, void*, hv_integral**); \
    template int hv_integrate_mc_impl<D>(hv_ctx*, const hv_mesh*, int64_t, uint64_t, hv_integral**); \
    template int hv_integrate_mc_points_impl<D>(hv_ctx*, const hv_mesh*, int64_t, uint64_t, double, hv_integral**);
HV_IINST(2)
HV_IINST(3)
HV_IINST(4)
HV_IINST(5)
HV_IINST(6)
