// pkd.hip — treelets of P-k-d trees: the compact acceleration structure for very large scenes
// (plugins/optix_owl/src/TreeletsCreate.h:117-166 prePartition_inPlace, PKDCreate.h:86-160 recBuild,
// used by TreeletsRenderer.cpp:95-110).
//
// The spheres are sorted by Morton code (the first half of an LBVH build) and cut into treelets
// of M consecutive spheres (M a power of two; the last treelet is shorter). The reference cuts at
// spatial midpoints until a part holds at most `threshold` particles; a run of the Morton order is
// a cell of the same kind of midpoint subdivision, and a fixed M lets the traversal find a
// treelet by a shift. Each treelet becomes a left-balanced k-d tree over its own spheres in heap
// order (node i of treelet t at position t*M + i, children 2i+1 and 2i+2): node i's split axis
// is the widest extent of its cell (ties to the lower axis), its sphere the one of rank
// |left subtree| among its subtree's spheres ordered by the coordinate on that axis (ties: the
// lower Morton position), and the children's cells are the node's cell cut at that coordinate.
// The root cell is the treelet's sphere bounds. A complete binary tree of boxes over the treelets
// (64-byte nodes like the LBVH's, heap order, treelet t at leaf slot t) sits on top.
//
// Memory beyond the spheres in treelet order: one byte per sphere (the split axis), 28 bytes per
// treelet and 64 bytes per top node, against 64 bytes per stored LBVH node.
//
// One 256-thread workgroup builds one treelet in LDS. The spheres never move: three lists hold their
// local indices in the order of each coordinate (sorted once, stably, so that equal coordinates keep
// the Morton order). Level by level every segment's node takes the element of rank |left subtree| from
// the list of its axis, and the three lists are partitioned stably about it, so that each segment stays
// sorted on every axis. (Sorting the segments anew at every level, bitonically, 55 exchange steps for
// 1024 spheres, took 3.3 ms for 8M spheres; this takes 1.0 ms.)
#include <float.h>

#include <algorithm>

#include "ctx.hpp"

namespace mmhrt {
namespace {

constexpr float PKD_ABSENT = 3.0e38f;  // the box no ray reaches: an absent child of the top tree

__device__ __forceinline__ uint32_t ford(float f) {
    uint32_t u = __float_as_uint(f);
    return (u & 0x80000000u) ? ~u : (u | 0x80000000u);
}

// nodes of the subtree of heap node i in a left-balanced tree of m nodes
__device__ __forceinline__ uint32_t subtree_size(uint32_t i, uint32_t m) {
    uint32_t first = i, width = 1, cnt = 0;
    while (first < m) {
        uint32_t end = first + width;
        cnt += end <= m ? width : m - first;
        first = 2 * first + 1;
        width *= 2;
    }
    return cnt;
}

__device__ __forceinline__ float coord(const float4& s, int d) { return d == 0 ? s.x : (d == 1 ? s.y : s.z); }

__device__ __forceinline__ int widest_axis(const float* b) {
    float e0 = b[3] - b[0], e1 = b[4] - b[1], e2 = b[5] - b[2];
    int d = 0;
    float e = e0;
    if (e1 > e) {
        d = 1;
        e = e1;
    }
    if (e2 > e) d = 2;
    return d;
}

// Mask of the lanes whose (valid) 8-bit digit equals ours.
__device__ __forceinline__ uint64_t same_digit(uint32_t d, bool valid) {
    uint64_t m = __ballot(valid);
#pragma unroll
    for (int b = 0; b < 8; ++b) {
        const uint64_t bm = __ballot((d >> b) & 1u);
        m &= ((d >> b) & 1u) ? bm : ~bm;
    }
    return m;
}

template <int M>
__global__ __launch_bounds__(256) void k_pkd_treelet(const float4* __restrict__ sph, uint32_t* __restrict__ ids,
                                                     float4* __restrict__ out_sph, uint8_t* __restrict__ out_dim,
                                                     float* __restrict__ tl_box, float* __restrict__ tl_rmax,
                                                     uint64_t n) {
    constexpr int NT = M / 256;        // elements or positions per thread
    constexpr int HALF = M / 2 + 1;    // nodes that can have children
    struct Sort {                      // the initial sorts
        uint32_t key[M];
        uint16_t val[M];
        uint16_t wc[4][256];
        uint32_t wsum[4];
    };
    struct Level {                     // the levels
        float box[HALF * 6];           // cell of heap node i
        uint16_t pre[3][M];            // lefts before a position of a list, counted from its wavefront's first
        uint16_t mpos[3][HALF];        // where a list holds the median of a level's k-th node
        uint16_t wtot[3][4];           // lefts of each wavefront's positions
    };
    union Scratch {
        Sort s;
        Level l;
    };
    __shared__ float4 s_sph[M];
    __shared__ uint16_t s_list[3][M];
    __shared__ Scratch u;
    __shared__ uint16_t s_start[M];  // in-order start of node i's segment
    __shared__ uint16_t s_pos[M];    // segment (heap node) holding position p; bit 15: p is fixed
    __shared__ uint16_t s_elem[M];   // node i's sphere (local index)
    __shared__ uint8_t s_dim[M];
    __shared__ uint8_t s_side[M];    // an element's place about its segment's median: 0 left, 1 median, 2 right
    __shared__ float s_red[4][7];
    const uint32_t tid = threadIdx.x, lane = tid & 63u, wv = tid >> 6;
    const uint64_t lt = (1ull << lane) - 1ull;
    const uint64_t base = (uint64_t)blockIdx.x * M;
    const uint32_t m = (uint32_t)std::min<uint64_t>(M, n - base);
    // positions of a thread: wavefront w holds M / 4 consecutive ones and walks them 64 at a time
    const uint32_t pb = wv * (M / 4) + lane;
    float lo[3] = {FLT_MAX, FLT_MAX, FLT_MAX}, hi[3] = {-FLT_MAX, -FLT_MAX, -FLT_MAX};
    float rmax = 0.0f;
    uint32_t idv[NT];
#pragma unroll
    for (int k = 0; k < NT; ++k) {
        const uint32_t j = pb + 64u * k;
        idv[k] = j < m ? ids[base + j] : 0u;
    }
    float4 own[NT];
#pragma unroll
    for (int k = 0; k < NT; ++k) {
        const uint32_t j = pb + 64u * k;
        own[k] = make_float4(0.f, 0.f, 0.f, 0.f);
        s_pos[j] = j < m ? 0 : 0x8000u;
        if (j < m) {
            const float4 q = sph[idv[k]];
            own[k] = q;
            s_sph[j] = q;
            lo[0] = fminf(lo[0], q.x - q.w);
            lo[1] = fminf(lo[1], q.y - q.w);
            lo[2] = fminf(lo[2], q.z - q.w);
            hi[0] = fmaxf(hi[0], q.x + q.w);
            hi[1] = fmaxf(hi[1], q.y + q.w);
            hi[2] = fmaxf(hi[2], q.z + q.w);
            rmax = fmaxf(rmax, q.w);
        }
    }
    // treelet bounds: min / max are exact in any order
    for (int o = 32; o > 0; o >>= 1) {
        for (int a = 0; a < 3; ++a) {
            lo[a] = fminf(lo[a], __shfl_xor(lo[a], o, 64));
            hi[a] = fmaxf(hi[a], __shfl_xor(hi[a], o, 64));
        }
        rmax = fmaxf(rmax, __shfl_xor(rmax, o, 64));
    }
    if (lane == 0) {
        for (int a = 0; a < 3; ++a) {
            s_red[wv][a] = lo[a];
            s_red[wv][3 + a] = hi[a];
        }
        s_red[wv][6] = rmax;
    }
    // the three sorts: least significant digit first, ranked with ballots (wavefront, round and lane
    // order together are the input order, so each pass is stable)
    for (int ax = 0; ax < 3; ++ax) {
        uint32_t key[NT], val[NT], rank[NT];
#pragma unroll
        for (int k = 0; k < NT; ++k) {
            key[k] = ford(coord(own[k], ax));
            val[k] = pb + 64u * k;
        }
        for (int shift = 0; shift < 32; shift += 8) {
            for (uint32_t d = lane; d < 256; d += 64) u.s.wc[wv][d] = 0;
#pragma unroll
            for (int k = 0; k < NT; ++k) {
                const bool valid = pb + 64u * k < m;
                const uint32_t d = (key[k] >> shift) & 255u;
                const uint64_t peers = same_digit(d, valid);
                const uint32_t before = valid ? u.s.wc[wv][d] : 0u;
                rank[k] = before + (uint32_t)__popcll(peers & lt);
                if (valid && (peers & lt) == 0) u.s.wc[wv][d] = (uint16_t)(before + (uint32_t)__popcll(peers));
            }
            __syncthreads();
            uint32_t c[4], cnt = 0;  // thread = digit
#pragma unroll
            for (int w = 0; w < 4; ++w) {
                c[w] = u.s.wc[w][tid];
                cnt += c[w];
            }
            uint32_t inc = cnt;
#pragma unroll
            for (int o = 1; o < 64; o <<= 1) {
                const uint32_t y = __shfl_up(inc, o, 64);
                if (lane >= (uint32_t)o) inc += y;
            }
            if (lane == 63) u.s.wsum[wv] = inc;
            __syncthreads();
            uint32_t run = inc - cnt;
            for (uint32_t w = 0; w < wv; ++w) run += u.s.wsum[w];
#pragma unroll
            for (int w = 0; w < 4; ++w) {
                u.s.wc[w][tid] = (uint16_t)run;
                run += c[w];
            }
            __syncthreads();
            const bool last = shift == 24;
#pragma unroll
            for (int k = 0; k < NT; ++k)
                if (pb + 64u * k < m) {
                    const uint32_t pos = u.s.wc[wv][(key[k] >> shift) & 255u] + rank[k];
                    if (last) {
                        s_list[ax][pos] = (uint16_t)val[k];
                    } else {
                        u.s.key[pos] = key[k];
                        u.s.val[pos] = (uint16_t)val[k];
                    }
                }
            __syncthreads();
            if (!last) {
#pragma unroll
                for (int k = 0; k < NT; ++k) {
                    key[k] = u.s.key[pb + 64u * k];  // (past m: not used)
                    val[k] = u.s.val[pb + 64u * k];
                }
            }
        }
    }
    if (tid == 0) {
        float b[6];
        for (int a = 0; a < 3; ++a) {
            b[a] = fminf(fminf(s_red[0][a], s_red[1][a]), fminf(s_red[2][a], s_red[3][a]));
            b[3 + a] = fmaxf(fmaxf(s_red[0][3 + a], s_red[1][3 + a]), fmaxf(s_red[2][3 + a], s_red[3][3 + a]));
        }
        const float r = fmaxf(fmaxf(s_red[0][6], s_red[1][6]), fmaxf(s_red[2][6], s_red[3][6]));
        for (int a = 0; a < 6; ++a) {
            u.l.box[a] = b[a];
            tl_box[(size_t)blockIdx.x * 6 + a] = b[a];
        }
        tl_rmax[blockIdx.x] = r;
        s_dim[0] = (uint8_t)widest_axis(b);
        s_start[0] = 0;
    }
    __syncthreads();
    for (uint32_t first = 0; first < m; first = 2 * first + 1) {
        const uint32_t last = std::min(2 * first, m - 1);  // the nodes of this level
        const bool inner = 2 * first + 1 < m;              // some of them have children
        // each segment's median is where the list of its axis has it; the elements of that list know
        // their sides by their positions
        uint32_t code[NT], med[NT];
#pragma unroll
        for (int k = 0; k < NT; ++k) {
            const uint32_t p = pb + 64u * k;
            code[k] = s_pos[p];
            med[k] = 0;
            if (!(code[k] & 0x8000u)) {
                const uint32_t i = code[k];
                const uint32_t L = 2 * i + 1 < m ? subtree_size(2 * i + 1, m) : 0u;
                med[k] = s_start[i] + L;
                const uint32_t j = s_list[s_dim[i]][p];
                s_side[j] = p < med[k] ? 0 : (p == med[k] ? 1 : 2);
                if (p == med[k]) s_elem[i] = (uint16_t)j;
            }
        }
        __syncthreads();
        if (inner) {
            // stable partition of the three lists: lefts before each position, by ballots
            uint32_t el[3][NT];
#pragma unroll
            for (int a = 0; a < 3; ++a) {
                uint32_t run = 0;
#pragma unroll
                for (int k = 0; k < NT; ++k) {
                    const uint32_t p = pb + 64u * k;
                    const bool live = !(code[k] & 0x8000u);
                    el[a][k] = live ? s_list[a][p] : 0u;
                    const uint32_t sd = live ? s_side[el[a][k]] : 2u;
                    const uint64_t lefts = __ballot(sd == 0u);
                    u.l.pre[a][p] = (uint16_t)(run + (uint32_t)__popcll(lefts & lt));
                    run += (uint32_t)__popcll(lefts);
                    if (sd == 1u) u.l.mpos[a][code[k] - first] = (uint16_t)p;
                    el[a][k] |= sd << 16;
                }
                if (lane == 0) u.l.wtot[a][wv] = (uint16_t)run;
            }
            __syncthreads();
#pragma unroll
            for (int a = 0; a < 3; ++a) {
#pragma unroll
                for (int k = 0; k < NT; ++k) {
                    if (code[k] & 0x8000u) continue;
                    const uint32_t p = pb + 64u * k, i = code[k];
                    const uint32_t st = s_start[i], sw = st / (M / 4);  // the segment's start and its wavefront
                    uint32_t lefts = (uint32_t)u.l.pre[a][p] - (uint32_t)u.l.pre[a][st];
                    for (uint32_t w = sw; w < wv; ++w) lefts += u.l.wtot[a][w];
                    const uint32_t sd = el[a][k] >> 16;
                    const uint32_t np = sd == 0u ? st + lefts
                                       : sd == 1u ? med[k]
                                                  : med[k] + 1 + (p - st) - lefts - (u.l.mpos[a][i - first] < p ? 1u : 0u);
                    s_list[a][np] = (uint16_t)el[a][k];
                }
            }
        }
#pragma unroll
        for (int k = 0; k < NT; ++k) {
            if (code[k] & 0x8000u) continue;
            const uint32_t p = pb + 64u * k, i = code[k];
            s_pos[p] = (uint16_t)(p == med[k] ? (i | 0x8000u) : (p < med[k] ? 2 * i + 1 : 2 * i + 2));
        }
        __syncthreads();
        // the children's cells, axes and segment starts
        for (uint32_t i = first + tid; inner && i <= last; i += 256) {
            if (2 * i + 1 >= m) continue;
            const int d = s_dim[i];
            const float cv = coord(s_sph[s_elem[i]], d);
            const uint32_t L = subtree_size(2 * i + 1, m);
            float b[6];
            for (int a = 0; a < 6; ++a) b[a] = u.l.box[6 * i + a];
            for (uint32_t sd = 0; sd < 2; ++sd) {
                const uint32_t ch = 2 * i + 1 + sd;
                if (ch >= m) break;
                float c[6];
                for (int a = 0; a < 6; ++a) c[a] = b[a];
                c[sd ? d : 3 + d] = cv;
                if (2 * ch + 1 < m)  // (a leaf's cell is not read again)
                    for (int a = 0; a < 6; ++a) u.l.box[6 * ch + a] = c[a];
                s_dim[ch] = (uint8_t)widest_axis(c);
                s_start[ch] = (uint16_t)(sd ? s_start[i] + L + 1 : s_start[i]);
            }
        }
        __syncthreads();
    }
    // the ids are permuted in place: all are read before any is written
#pragma unroll
    for (int k = 0; k < NT; ++k) {
        const uint32_t i = tid + 256u * k;
        idv[k] = i < m ? ids[base + s_elem[i]] : 0u;
    }
    __syncthreads();
#pragma unroll
    for (int k = 0; k < NT; ++k) {
        const uint32_t i = tid + 256u * k;
        if (i < m) {
            out_sph[base + i] = s_sph[s_elem[i]];
            ids[base + i] = idv[k];
            out_dim[base + i] = s_dim[i];
        }
    }
}

// One level of the top tree (heap nodes first .. first + count - 1), bottom up: a child slot at or
// past L - 1 is treelet slot - (L - 1) (absent from T on); an internal child's box is the union of
// its present children.
__global__ __launch_bounds__(256) void k_pkd_top_level(Node* __restrict__ nodes, const float* __restrict__ tl_box,
                                                       uint32_t T, uint32_t L, uint32_t first, uint32_t count) {
    const uint32_t q = blockIdx.x * 256u + threadIdx.x;
    if (q >= count) return;
    const uint32_t k = first + q;
    float bx[2][6];
    int32_t ref[2];
    for (int c = 0; c < 2; ++c) {
        const uint32_t ch = 2 * k + 1 + (uint32_t)c;
        bool present = false;
        if (ch >= L - 1) {
            const uint32_t t = ch - (L - 1);
            if (t < T) {
                present = true;
                for (int a = 0; a < 6; ++a) bx[c][a] = tl_box[(size_t)t * 6 + a];
                ref[c] = ~(int32_t)t;
            }
        } else {
            const Node cn = nodes[ch];
            const float* f = reinterpret_cast<const float*>(&cn);
            const bool p0 = cn.d.x != INT32_MIN, p1 = cn.d.y != INT32_MIN;
            if (p0 || p1) {
                present = true;
                for (int a = 0; a < 3; ++a) {
                    const float l0 = f[a], h0 = f[3 + a], l1 = f[6 + a], h1 = f[9 + a];
                    bx[c][a] = p0 && p1 ? fminf(l0, l1) : (p0 ? l0 : l1);
                    bx[c][3 + a] = p0 && p1 ? fmaxf(h0, h1) : (p0 ? h0 : h1);
                }
                ref[c] = (int32_t)ch;
            }
        }
        if (!present) {
            for (int a = 0; a < 6; ++a) bx[c][a] = PKD_ABSENT;
            ref[c] = INT32_MIN;
        }
    }
    Node o;
    o.a = make_float4(bx[0][0], bx[0][1], bx[0][2], bx[0][3]);
    o.b = make_float4(bx[0][4], bx[0][5], bx[1][0], bx[1][1]);
    o.c = make_float4(bx[1][2], bx[1][3], bx[1][4], bx[1][5]);
    o.d = make_int4(ref[0], ref[1], 0, 0);
    nodes[k] = o;
}

}  // namespace

int build_pkd(mmhrt_ctx_s* c, int bits, bool reserve_only) {
    const int64_t M = c->opt_treelet;
    if (M != 256 && M != 512 && M != 1024)
        return fail(c, MMHRT_E_INVALID, "build: option treelet must be 256, 512 or 1024");
    if (int e = sort_spheres(c, bits, reserve_only)) return e;
    const uint64_t n = c->n;
    const uint32_t T = (uint32_t)((n + M - 1) / M);
    uint32_t L = 2;
    while (L < T) L *= 2;
    int e = 0;
    if ((e = ensure(c, c->leaf_sph, n, "leaf spheres"))) return e;
    if ((e = ensure(c, c->pkd_dim, n, "split axes"))) return e;
    if ((e = ensure(c, c->tl_box, (size_t)T * 6, "treelet boxes"))) return e;
    if ((e = ensure(c, c->tl_rmax, T, "treelet radii"))) return e;
    if ((e = ensure(c, c->nodes, L - 1, "top nodes"))) return e;
    if (reserve_only) {
        c->pkd_M = (uint32_t)M;
        c->pkd_T = T;
        c->pkd_L = L;
        c->accel = 1;
        return 0;
    }
    rec(c, 3);
    rec(c, 4);
    const float4* sph = cur_spheres(c);
    if (M == 256)
        hipLaunchKernelGGL(k_pkd_treelet<256>, dim3(T), dim3(256), 0, c->stream, sph, c->leaf_id.p, c->leaf_sph.p,
                           c->pkd_dim.p, c->tl_box.p, c->tl_rmax.p, n);
    else if (M == 512)
        hipLaunchKernelGGL(k_pkd_treelet<512>, dim3(T), dim3(256), 0, c->stream, sph, c->leaf_id.p, c->leaf_sph.p,
                           c->pkd_dim.p, c->tl_box.p, c->tl_rmax.p, n);
    else
        hipLaunchKernelGGL(k_pkd_treelet<1024>, dim3(T), dim3(256), 0, c->stream, sph, c->leaf_id.p, c->leaf_sph.p,
                           c->pkd_dim.p, c->tl_box.p, c->tl_rmax.p, n);
    for (uint32_t first = L / 2 - 1, count = L / 2;; first = (first - 1) / 2, count /= 2) {
        hipLaunchKernelGGL(k_pkd_top_level, dim3((count + 255) / 256), dim3(256), 0, c->stream, c->nodes.p,
                           c->tl_box.p, T, L, first, count);
        if (first == 0) break;
    }
    rec(c, 5);
    hipError_t he = hipGetLastError();
    if (he != hipSuccess) return hip_fail(c, he, "P-k-d build launch");
    c->pkd_M = (uint32_t)M;
    c->pkd_T = T;
    c->pkd_L = L;
    c->built = true;
    c->built_n = n;
    c->accel = 1;
    c->bvh_pairs = false;
    c->info_valid = false;
    return 0;
}

}  // namespace mmhrt
