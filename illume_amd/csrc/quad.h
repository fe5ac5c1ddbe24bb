/*
 * quad.h - closest-hit walk with four lanes per ray.
 *
 * A wave traces 16 rays at a time, each by a quad of neighbouring lanes: a node visit gives lane
 * k child k of an FP32 BVH4 node (FNode), a leaf visit gives lane k triangle k, and entering an
 * instance gives lane k row k of its inverse. Branches, the current node and the ray are uniform
 * over a quad; ranks, votes and broadcasts inside it are DPP quad permutations. The arithmetic of
 * every box test, triangle test and transform is that of traverse.h, and a closest hit does not
 * depend on the order of the walk, so the hits are the same bit for bit.
 */
#pragma once
#include "traverse.h"

#define QUADS 16                /* rays a wave walks at a time */
#define QSTACK ILM_QUAD_STACK   /* stack entries per quad, in LDS */

template <int CTRL>
__device__ inline int qperm_i(int v) { return __builtin_amdgcn_mov_dpp(v, CTRL, 0xf, 0xf, true); }
template <int CTRL>
__device__ inline float qperm_f(float v) { return __int_as_float(qperm_i<CTRL>(__float_as_int(v))); }
#define QP_ROT1 0x39            /* lane k takes lane k+1's value, 2: k+2, 3: k+3 (mod 4) */
#define QP_ROT2 0x4e
#define QP_ROT3 0x93
#define QP_XOR1 0xb1
#define QP_XOR2 0x4e
#define QP_B(k) ((k) * 0x55)    /* every lane takes lane k's value */
__device__ inline float quad_min_f(float v) {
    v = __builtin_fminf(v, qperm_f<QP_XOR1>(v));
    return __builtin_fminf(v, qperm_f<QP_XOR2>(v));
}
__device__ inline int quad_min_i(int v) {
    int o = qperm_i<QP_XOR1>(v);
    v = o < v ? o : v;
    o = qperm_i<QP_XOR2>(v);
    return o < v ? o : v;
}
__device__ inline int quad_or(int v) {
    v |= qperm_i<QP_XOR1>(v);
    return v | qperm_i<QP_XOR2>(v);
}
__device__ inline int quad_add(int v) {
    v += qperm_i<QP_XOR1>(v);
    return v + qperm_i<QP_XOR2>(v);
}

/* Between LDS accesses of different lanes of a wave: the LDS serves a wave's accesses in order, so
 * nothing has to be waited for, but the compiler, which follows one lane, must not move or forward
 * them across. No instruction. */
__device__ inline void wave_lds_order() {
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
}

/* A wave's rays and their hits in LDS: up to 64 rays staged by the lanes that own them and taken
 * by the quads one at a time; a finished quad leaves the hit in the ray's own columns. */
struct QuadLds {
    int stk[QSTACK * QUADS];    /* entry s of quad q at s * QUADS + q: quads never share a bank */
    float ray[6][64];           /* o, d; a hit leaves u, v, prim in columns 0..2 */
    float t[64];                /* closest hit so far (sphere or free-flight cap), then the hit's */
    int inst[64];
    int req[64];                /* request of the ray (chunks of several scenes) */
};

/* Stage a ray as entry j: its spheres are tested here, by the lane that owns it. */
__device__ inline void quad_stage(LDSAS QuadLds* L, int j, const GLOBAL DScene* S, V3 O, V3 D, float tmax0, int req) {
    Best B;
    best_init(B);
    B.t = tmax0;
    spheres_first(S, O, D, B);
    L->ray[0][j] = O.x; L->ray[1][j] = O.y; L->ray[2][j] = O.z;
    L->ray[3][j] = D.x; L->ray[4][j] = D.y; L->ray[5][j] = D.z;
    L->t[j] = B.t;
    L->inst[j] = B.inst;
    L->req[j] = req;
}

/* Walk rays 0..n-1 staged in L and leave their hits there. Every lane of the wave calls it. */
template <int TRI, int UNI>
__device__ inline void quad_walk(LDSAS QuadLds* L, int n, const GLOBAL DReq* reqs, const GLOBAL DScene* Su) {
    const int lane = threadIdx.x & 63;
    const int sub = lane & 3, quad = lane >> 2;
    LDSAS int* stk = L->stk + quad;
    const GLOBAL DScene* S = Su;
    const GLOBAL DInst* insts = nullptr;
    const GLOBAL FNode* tlas = nullptr;
    int root = ILM_NO_CHILD;
    if (UNI) {
        insts = uni_p(gp(Su->inst));
        tlas = uni_p(gp(Su->ftlas));
        root = uni_i(Su->ftlas_root);
    }
    int ridx = -1;
    V3 O, D, o, d, id;
    Best B;
    float qt = 0.0f;                    /* the quad's closest hit so far */
    const GLOBAL FNode* nodes = nullptr;
    const GLOBAL float4* tris = nullptr;
    WTRay wt;
    int node = 0, sp = 0, cur = 0, blas = 0;
    int next = 0;
    best_init(B);
    O = D = o = d = id = mk3(0.0f, 0.0f, 0.0f);
    for (;;) {
        wave_lds_order();   /* a stack entry is read by the lanes of its quad, written by one of them in an earlier trip */
        const unsigned long long idle = __ballot(ridx < 0);
        if (next < n) {
            if (idle) {
                const int rank = (int)(__builtin_amdgcn_mbcnt_hi((uint32_t)(idle >> 32),
                                                                 __builtin_amdgcn_mbcnt_lo((uint32_t)idle, 0u)) >> 2);
                if (ridx < 0 && next + rank < n) {
                    const int j = next + rank;
                    ridx = j;
                    O = mk3(L->ray[0][j], L->ray[1][j], L->ray[2][j]);
                    D = mk3(L->ray[3][j], L->ray[4][j], L->ray[5][j]);
                    B.t = qt = L->t[j];
                    B.u = B.v = 0.0f;
                    B.inst = L->inst[j];
                    B.prim = -1;
                    if (!UNI) {
                        S = gp(reqs[L->req[j]].scene);
                        insts = gp(S->inst);
                        tlas = gp(S->ftlas);
                        root = S->ftlas_root;
                    }
                    o = O;
                    d = D;
                    id = rcp3(D);
                    nodes = tlas;
                    node = root == ILM_NO_CHILD ? POP_MARK : root;
                    sp = 0;
                    blas = 0;
                    cur = -1;
                }
                next += __builtin_popcountll(idle) >> 2;
            }
        } else if (idle == ~0ull) {
            break;
        }
        if (ridx >= 0) {
            bool pop;
            if (node >= 0 && node != POP_MARK) {
                const GLOBAL float4* p = (const GLOBAL float4*)(nodes + node) + 2 * sub;
                const float4 a = p[0], b = p[1];
                const int code = __float_as_int(b.z);
                const float x0 = (a.x - o.x) * id.x, x1 = (a.y - o.x) * id.x;
                const float y0 = (a.z - o.y) * id.y, y1 = (a.w - o.y) * id.y;
                const float z0 = (b.x - o.z) * id.z, z1 = (b.y - o.z) * id.z;
                const float tn = __builtin_fmaxf(__builtin_fmaxf(__builtin_fminf(x0, x1), __builtin_fminf(y0, y1)),
                                                 __builtin_fmaxf(__builtin_fminf(z0, z1), 0.0f));
                const float tf = __builtin_fminf(__builtin_fminf(__builtin_fmaxf(x0, x1), __builtin_fmaxf(y0, y1)),
                                                 __builtin_fmaxf(z0, z1));
                const bool hit = (code != ILM_NO_CHILD) & (tn <= tf * BOX_K) & (tn <= qt * BOX_TMAX);
                /* distinct keys: entry distance (>= 0) with the lane in its low bits */
                const uint32_t key = hit ? ((f2u(tn) & 0x7ffffffcu) | (uint32_t)sub) : 0xffffffffu;
                const uint32_t k1 = (uint32_t)qperm_i<QP_ROT1>((int)key);
                const uint32_t k2 = (uint32_t)qperm_i<QP_ROT2>((int)key);
                const uint32_t k3 = (uint32_t)qperm_i<QP_ROT3>((int)key);
                const int rank = (int)(k1 < key) + (int)(k2 < key) + (int)(k3 < key);
                const int nhit = quad_add((int)hit);
                const int near = quad_or((hit & (rank == 0)) ? code : 0);
                if (hit & (rank > 0)) stk[(sp + nhit - 1 - rank) * QUADS] = code;
                pop = nhit == 0;
                if (!pop) {
                    sp += nhit - 1;
                    node = near;
                }
            } else if (node == POP_MARK) {
                pop = true;
            } else if (blas) {
                const int f = (int)ilm_leaf_first(node), cnt = (int)ilm_leaf_count(node);
                for (int q = sub; q < cnt; q += 4) {
                    const GLOBAL float4* tp = tris + 3 * (f + q);
                    const float4 A = tp[0], Bq = tp[1], C = tp[2];
                    float u = 0.0f, v = 0.0f, t;
                    if (TRI) t = tri_wt(wt, mk3(A.x, A.y, A.z), mk3(Bq.x, Bq.y, Bq.z), mk3(C.x, C.y, C.z), o, u, v);
                    else t = tri_mt(mk3(A.x, A.y, A.z), mk3(Bq.x, Bq.y, Bq.z), mk3(C.x, C.y, C.z), o, d, u, v);
                    const int prim = __float_as_int(A.w);
                    const bool tie = t == B.t && B.inst >= 0 && (cur < B.inst || (cur == B.inst && prim < B.prim));
                    if (t > 0.0f && (t < B.t || tie)) best_tri(B, t, u, v, cur, A);
                }
                qt = quad_min_f(B.t);
                pop = true;
            } else {
                /* entering instance k: lane j < 3 transforms component j, lane 3 brings the BLAS */
                const int k = (int)ilm_leaf_first(node);
                const GLOBAL DInst* I = insts + k;
                const GLOBAL float4* w = (const GLOBAL float4*)I + (sub == 3 ? 11 : sub);
                const float4 r = w[0];
                const GLOBAL float4* tr = gp(I->tris);
                const float oc = r.x * O.x + r.y * O.y + r.z * O.z + r.w * 1.0f;
                const float dc = r.x * D.x + r.y * D.y + r.z * D.z + r.w * 0.0f;
                const int broot = qperm_i<QP_B(3)>(__float_as_int(r.z));
                const uint32_t nl = (uint32_t)qperm_i<QP_B(3)>(__float_as_int(r.x));
                const uint32_t nh = (uint32_t)qperm_i<QP_B(3)>(__float_as_int(r.y));
                pop = broot == ILM_NO_CHILD;
                if (!pop) {
                    o = mk3(qperm_f<QP_B(0)>(oc), qperm_f<QP_B(1)>(oc), qperm_f<QP_B(2)>(oc));
                    d = mk3(qperm_f<QP_B(0)>(dc), qperm_f<QP_B(1)>(dc), qperm_f<QP_B(2)>(dc));
                    id = rcp3(d);
                    if (TRI) wt = wt_setup(d);
                    nodes = (const GLOBAL FNode*)(((uint64_t)nh << 32) | nl);
                    tris = tr;
                    stk[sp * QUADS] = STACK_SENTINEL;
                    sp++;
                    blas = 1;
                    cur = k;
                    node = broot;
                }
            }
            while (pop) {
                if (sp == 0) {
                    /* the ray is done: the lane that holds the closest hit writes it (equal
                     * distances: the smaller instance, then primitive, as leaf_tris keeps) */
                    const bool c = B.t == qt;
                    const int im = quad_min_i(c ? B.inst : 0x7fffffff);
                    const bool c2 = c & (B.inst == im);
                    const int pm = quad_min_i(c2 ? B.prim : 0x7fffffff);
                    if (c2 & (B.prim == pm)) {
                        L->t[ridx] = B.t;
                        L->inst[ridx] = B.inst;
                        L->ray[0][ridx] = B.u;
                        L->ray[1][ridx] = B.v;
                        L->ray[2][ridx] = __int_as_float(B.prim);
                    }
                    ridx = -1;
                    break;
                }
                sp--;
                node = stk[sp * QUADS];
                if (node != STACK_SENTINEL) break;
                o = O;
                d = D;
                id = rcp3(D);
                blas = 0;
                nodes = tlas;
            }
        }
    }
}

/* Closest hits of a short queue of one scene's rays. Each wave takes its share of the queue, 16
 * rays at least and 64 at a time. */
template <int TRI>
__global__ __launch_bounds__(64) __attribute__((amdgpu_waves_per_eu(6, 8))) void k_extend_quad(KParams P, int depth) {
    __shared__ QuadLds lds;
    LDSAS QuadLds* L = (LDSAS QuadLds*)&lds;
    const uint32_t count = gp(P.ctl)->count[depth];
    const int lane = threadIdx.x;
    const GLOBAL DReq* reqs = gp(P.chunk)->reqs;
    const GLOBAL DScene* S = uni_p(gp(reqs[0].scene));
    uint32_t per = ((count + gridDim.x - 1u) / gridDim.x + 15u) & ~15u;
    if (per > 64u) per = 64u;
    for (uint32_t base = blockIdx.x * per; base < count; base += gridDim.x * per) {
        const uint32_t n = count - base < per ? count - base : per;
        const uint32_t i = base + (uint32_t)lane;
        const bool own = (uint32_t)lane < n;
        if (own) {
            const float4 o4 = gp(P.in.o)[i], d4 = gp(P.in.d)[i];
            const uint2 rg = gp(P.in.rng)[i];
            quad_stage(L, lane, S, mk3(o4.x, o4.y, o4.z), mk3(d4.x, d4.y, d4.z),
                       medium_tmax(S, f2u(o4.w), rg, f2u(d4.w)), 0);
        }
        __syncthreads();
        quad_walk<TRI, 1>(L, (int)n, reqs, S);
        __syncthreads();
        if (own) {
            gpw(P.hits.h)[i] = make_float4(L->t[lane], L->ray[0][lane], L->ray[1][lane], L->ray[2][lane]);
            gpw(P.hits.inst)[i] = L->inst[lane];
        }
        __syncthreads();
    }
}
