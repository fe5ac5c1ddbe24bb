/*
 * engine.hip - host runtime behind the C ABI: context, device-resident scenes, the chunked
 * wavefront driver (direct launches, or hipGraphs by depth count and kind of chunk), the plain,
 * batched and served forms, and the parity hooks.
 *
 * Reference counterparts: Renderer::render_to_bitmap (src/renderer.cu:498-597) and
 * SceneRef (src/scene/sceneref.cpp:9-148). Differences by design: scenes stay on the device
 * across renders, path state is struct-of-arrays and compacted on the device, many passes
 * (and many requests) share one chunk of launches, and no depth synchronises with the host: its
 * launches are queued ahead of it.
 */
#include <algorithm>
#include <atomic>
#include <chrono>
#include <cmath>
#include <condition_variable>
#include <cstdio>
#include <cstring>
#include <deque>
#include <future>
#include <map>
#include <memory>
#include <mutex>
#include <string>
#include <system_error>
#include <thread>
#include <type_traits>
#include <vector>

#include "bvh.h"
#include "bvh_cache.h"
#include "engine.h"
#include "hostmath.h"
#include "kernels.h"

using namespace ilm;

static thread_local std::string g_err;

/* ======================= no-allocation scratch ======================= */

/* Device memory of ilm_render_noalloc: path state, hits, per-path results, control block, chunk
 * descriptor, traversal-stack spill area, Kahan sums and pixels of one render, all carved from
 * this array. Each GPU the library runs on holds its own copy until the process ends. In host
 * code the name is a host-side stand-in, never a device address: kernels and copies use the
 * address hipGetSymbolAddress gives for the current device (noalloc_scratch_of). The control
 * block's packet cursors and k_finish counts lie beyond ILM_NOALLOC_SCRATCH_BYTES, so that the
 * largest image the array takes does not depend on how many waves those kernels run. */
#define ILM_NOALLOC_CTL_BYTES (sizeof(DCtl::band) + sizeof(DCtl::tail))
#define ILM_NOALLOC_ARRAY_BYTES (ILM_NOALLOC_SCRATCH_BYTES + ILM_NOALLOC_CTL_BYTES)
static_assert(ILM_NOALLOC_CTL_BYTES % 256 == 0, "the blocks behind the control block keep their places in the documented bytes");
static __device__ __align__(256) unsigned char scratch[ILM_NOALLOC_ARRAY_BYTES];

#define ILM_MAX_DEVICES 64
static std::mutex g_scratch_mu;                     /* g_scratch_ptr */
static void* g_scratch_ptr[ILM_MAX_DEVICES];
/* held for the whole of an ilm_render_noalloc call: calls on one GPU share its array */
static std::mutex g_noalloc_mu[ILM_MAX_DEVICES];
/* held while a graph is captured on the device, and around the calls that wait for the whole
 * device (hipFree): the runtime refuses those while any stream of the device is capturing, and
 * contexts on one device may capture and free from different threads. A leaf lock. */
static std::mutex g_capture_mu[ILM_MAX_DEVICES];
static std::mutex& capture_mu(int device) { return g_capture_mu[device >= 0 && device < ILM_MAX_DEVICES ? device : 0]; }
static void dfree(int device, void* p) {
    if (!p) return;
    std::lock_guard<std::mutex> lk(capture_mu(device));
    (void)hipFree(p);
}

/* This device's address of the scratch array, looked up once per device with the device
 * current (the caller has made it current). */
static hipError_t noalloc_scratch_of(int device, void** out) {
    *out = nullptr;
    if (device < 0 || device >= ILM_MAX_DEVICES) return hipErrorInvalidDevice;
    std::lock_guard<std::mutex> lk(g_scratch_mu);
    if (!g_scratch_ptr[device]) {
        void* ptr = nullptr;
        hipError_t e = hipGetSymbolAddress((void**)&ptr, HIP_SYMBOL(scratch));
        if (e != hipSuccess) return e;
        if (!ptr) return hipErrorInvalidSymbol;
        g_scratch_ptr[device] = ptr;
    }
    *out = g_scratch_ptr[device];
    return hipSuccess;
}

const char* ilm_global_error(void) { return g_err.c_str(); }
int ilm_version(void) { return ILM_ABI_VERSION; }

static int fail(ilm_ctx* ctx, int code, const std::string& msg) {
    g_err = msg;
    if (ctx) {
        std::lock_guard<std::mutex> lk(ctx->err_mu);
        ctx->err = msg;
    }
    return code;
}
#define HIPTRY(ctx, call)                                                                          \
    do {                                                                                           \
        hipError_t e_ = (call);                                                                    \
        if (e_ != hipSuccess)                                                                      \
            return fail((ctx), ILM_E_DEVICE, std::string(#call ": ") + hipGetErrorString(e_));     \
    } while (0)

static double now_ms(const ilm_ctx* ctx) {
    return std::chrono::duration<double, std::milli>(std::chrono::steady_clock::now() - ctx->t0).count();
}

/* ======================= scenes ======================= */

static hipError_t dalloc(ilm_scene* s, void** p, size_t bytes) {
    *p = nullptr;
    if (bytes == 0) return hipSuccess;
    hipError_t e = hipMalloc(p, bytes);
    if (e == hipSuccess) {
        s->allocs.push_back(*p);
        s->bytes += (int64_t)bytes;
    }
    return e;
}
/* Blocking copy through the context's copy stream (never the legacy stream). */
static hipError_t copy_sync(ilm_ctx* ctx, void* dst, const void* src, size_t bytes, hipMemcpyKind kind) {
    hipError_t e = hipMemcpyAsync(dst, src, bytes, kind, ctx->copy_stream);
    if (e != hipSuccess) return e;
    return hipStreamSynchronize(ctx->copy_stream);
}
template <class T>
static hipError_t dupload(ilm_scene* s, T** dst, const T* src, size_t count) {
    *dst = nullptr;
    if (count == 0) return hipSuccess;
    hipError_t e = dalloc(s, (void**)dst, count * sizeof(T));
    if (e != hipSuccess) return e;
    return copy_sync(s->ctx, *dst, src, count * sizeof(T), hipMemcpyHostToDevice);
}

/* Two arrays in one allocation (the second 256-byte aligned), their copies waited for together: an
 * allocation and a wait take some 15 us, which a scene of a few triangles spends its upload on. */
template <class A, class B>
static hipError_t dupload2(ilm_scene* s, A** da, const A* a, size_t na, B** db, const B* b, size_t nb) {
    *da = nullptr;
    *db = nullptr;
    const size_t off = (na * sizeof(A) + 255) & ~(size_t)255;
    char* p = nullptr;
    hipError_t e = dalloc(s, (void**)&p, off + nb * sizeof(B));
    if (e != hipSuccess || !p) return e;
    if (na) *da = (A*)p;
    if (nb) *db = (B*)(p + off);
    const hipStream_t st = s->ctx->copy_stream;
    if (na) e = hipMemcpyAsync(p, a, na * sizeof(A), hipMemcpyHostToDevice, st);
    if (nb && e == hipSuccess) e = hipMemcpyAsync(p + off, b, nb * sizeof(B), hipMemcpyHostToDevice, st);
    const hipError_t w = hipStreamSynchronize(st);   /* the first copy too when the second failed */
    return e != hipSuccess ? e : w;
}

static int upload_texture(ilm_ctx* ctx, ilm_scene* s, const ilm_texture_desc& t, DTex& d) {
    std::memset(&d, 0, sizeof(d));
    d.type = t.type;
    if (t.type == ILM_TEX_CONSTANT) {
        for (int i = 0; i < 3; i++) d.a[i] = t.color[i];
    } else if (t.type == ILM_TEX_CHECKERBOARD) {
        for (int i = 0; i < 3; i++) { d.a[i] = t.on[i]; d.b[i] = t.off[i]; }
    } else if (t.type == ILM_TEX_BITMAP) {
        if (t.width <= 0 || t.height <= 0) return fail(ctx, ILM_E_INVALID, "bitmap texture without size");
        d.w = t.width; d.h = t.height; d.hdr = t.is_hdr;
        size_t n = (size_t)t.width * t.height;
        if (t.is_hdr) {
            if (!t.texels_f32) return fail(ctx, ILM_E_INVALID, "HDR bitmap without texels");
            float4* p;
            HIPTRY(ctx, dupload(s, &p, (const float4*)t.texels_f32, n));
            d.f = p;
        } else {
            if (!t.texels_u8) return fail(ctx, ILM_E_INVALID, "LDR bitmap without texels");
            uchar4* p;
            HIPTRY(ctx, dupload(s, &p, (const uchar4*)t.texels_u8, n));
            d.u8 = p;
        }
    } else {
        return fail(ctx, ILM_E_INVALID, "unknown texture type");
    }
    d.scale[0] = t.scale[0];
    d.scale[1] = t.scale[1];
    return ILM_OK;
}

static void m4_rows(const hm::M4& m, float* out12) {
    for (int i = 0; i < 3; i++) for (int j = 0; j < 4; j++) out12[4 * i + j] = m.m[i][j];
}

/* outward rounding of a double bound to float */
static float round_down(double v) { float f = (float)v; return (double)f > v ? std::nextafter(f, -INFINITY) : f; }
static float round_up(double v) { float f = (float)v; return (double)f < v ? std::nextafter(f, INFINITY) : f; }

/* f's result for a mesh of n triangles, made by a thread of its own; by the one that asks for it when
 * the mesh is small (a thread costs some 20 us, 16384 triangles 0.5 ms) or there can be no more
 * threads. A future that is dropped waits for its thread. */
template <class F>
static std::future<std::invoke_result_t<F>> beside(int n, F f) {
    if (n >= 16384) {
        try {
            return std::async(std::launch::async, f);
        } catch (const std::system_error&) {
        }
    }
    return std::async(std::launch::deferred, f);
}

int ilm_scene_upload(ilm_ctx* ctx, const ilm_scene_desc* d, ilm_scene** out) {
    if (!ctx || !d || !out) return fail(ctx, ILM_E_INVALID, "null argument");
    *out = nullptr;
    std::unique_ptr<ilm_scene> s(new ilm_scene());
    s->ctx = ctx;
    HIPTRY(ctx, hipSetDevice(ctx->device));

    /* ---- validation ---- */
    for (int i = 0; i < d->num_meshes; i++) {
        const ilm_mesh_desc& m = d->meshes[i];
        if (m.num_vertices < 0 || m.num_triangles < 0 || (m.num_triangles > 0 && (!m.indices || !m.positions)))
            return fail(ctx, ILM_E_INVALID, "mesh " + std::to_string(i) + ": bad arrays");
        if (!m.face_normals && !m.normals) return fail(ctx, ILM_E_INVALID, "mesh needs normals when face_normals=0");
        if (m.has_texcoords && !m.texcoords) return fail(ctx, ILM_E_INVALID, "mesh needs texcoords");
        if ((int64_t)m.num_triangles >= (1 << 27)) return fail(ctx, ILM_E_UNSUPPORTED, "mesh too large (2^27 triangles)");
        for (int64_t k = 0; k < 3LL * m.num_triangles; k++)
            if (m.indices[k] < 0 || m.indices[k] >= m.num_vertices)
                return fail(ctx, ILM_E_INVALID, "mesh " + std::to_string(i) + ": index out of range");
    }
    for (int i = 0; i < d->num_instances; i++) {
        if (d->instances[i].mesh < 0 || d->instances[i].mesh >= d->num_meshes)
            return fail(ctx, ILM_E_INVALID, "instance mesh out of range");
        if (d->instances[i].material < 0 || d->instances[i].material >= d->num_materials)
            return fail(ctx, ILM_E_INVALID, "instance material out of range");
    }
    for (int i = 0; i < d->num_spheres; i++)
        if (d->spheres[i].material < 0 || d->spheres[i].material >= d->num_materials)
            return fail(ctx, ILM_E_INVALID, "sphere material out of range");
    for (int i = 0; i < d->num_materials; i++)
        if (d->materials[i].medium < -1 || d->materials[i].medium >= d->num_mediums)
            return fail(ctx, ILM_E_INVALID, "material medium out of range");
    if (d->num_instances >= 65536) return fail(ctx, ILM_E_UNSUPPORTED, "too many instances");

    DScene hs;
    std::memset(&hs, 0, sizeof(hs));

    /* ---- meshes: BVH, layouts, triangle slots ---- */
    std::vector<DMesh> dmeshes(d->num_meshes);
    std::vector<Box> mesh_bounds(d->num_meshes);
    int blas_depth = 0, blas_qdepth = 0, blas_flevels = 0;
    BuildOpts bo;
    for (int i = 0; i < d->num_meshes; i++) {
        const ilm_mesh_desc& m = d->meshes[i];
        MeshBVH bvh;
        bool cached = false;
        uint64_t key = 0;
        if (!ctx->bvh_cache_dir.empty()) {
            key = mesh_key(m.positions, m.num_vertices, m.indices, m.num_triangles, bo);
            cached = cache_load(ctx->bvh_cache_dir, key, m.num_triangles, bvh);
        }
        if (!cached) {
            bvh = build_mesh_bvh(m.positions, m.indices, m.num_triangles, bo);
            if (!ctx->bvh_cache_dir.empty()) (void)cache_store(ctx->bvh_cache_dir, key, bvh);
        }
        if (!ctx->bvh_cache_dir.empty()) {
            std::lock_guard<std::mutex> lk(ctx->stat_mu);
            (cached ? ctx->stat_bvh_hits : ctx->stat_bvh_misses)++;
        }
        blas_depth = std::max(blas_depth, bvh.depth);
        blas_qdepth = std::max(blas_qdepth, bvh.qdepth);
        s->quant_max_exp = std::max(s->quant_max_exp, qnodes_max_exponent(bvh.qnodes));
        /* The FNode layout and the shading vertices are made beside the rest of the mesh's upload, so
         * that a mesh whose other layouts come from the cache waits for neither: a cached upload of
         * 722k triangles takes 60 ms, of 101k 5.0 (64.7 and 4.9 without FNodes, 85 and 6.3 with both made
         * in turn; 62 to 66 and 6.4 with the mesh's bounds taken before the threads start). */
        std::future<LayoutF> flayout = beside(m.num_triangles, [&bvh] { return make_layout_f(bvh.nodes, bvh.root); });
        /* shading vertices by original triangle index: the same floats the kernel would gather
         * through the index array */
        std::future<std::vector<float4>> sverts = beside(m.num_triangles, [&m] {
            std::vector<float4> sv(3 * (size_t)m.num_triangles);
            const float* va = m.face_normals ? m.positions : m.normals;
            for (int t = 0; t < m.num_triangles; t++)
                for (int k = 0; k < 3; k++) {
                    const float* v = &va[3 * (size_t)m.indices[3 * t + k]];
                    sv[3 * (size_t)t + k] = make_float4(v[0], v[1], v[2], 0.0f);
                }
            return sv;
        });
        Box mb;
        mb.reset();
        for (int64_t k = 0; k < 3LL * m.num_triangles; k++) mb.grow(&m.positions[3 * m.indices[k]]);
        mesh_bounds[i] = mb;
        std::vector<float4> tris(3 * (size_t)m.num_triangles);
        for (int k = 0; k < m.num_triangles; k++) {
            int t = bvh.order[k];
            const float* p0 = &m.positions[3 * m.indices[3 * t]];
            const float* p1 = &m.positions[3 * m.indices[3 * t + 1]];
            const float* p2 = &m.positions[3 * m.indices[3 * t + 2]];
            float tb;
            int32_t ti = t;
            std::memcpy(&tb, &ti, 4);
            tris[3 * k] = make_float4(p0[0], p0[1], p0[2], tb);
            tris[3 * k + 1] = make_float4(p1[0], p1[1], p1[2], 0.0f);
            tris[3 * k + 2] = make_float4(p2[0], p2[1], p2[2], 0.0f);
        }
        DMesh& dm = dmeshes[i];
        std::memset(&dm, 0, sizeof(dm));
        BNode* bn; QNode* qn; float4* tp; int* ip; float* pp; float* np; float* up;
        HIPTRY(ctx, dupload(s.get(), &bn, bvh.nodes.data(), bvh.nodes.size()));
        HIPTRY(ctx, dupload(s.get(), &qn, bvh.qnodes.data(), bvh.qnodes.size()));
        HIPTRY(ctx, dupload(s.get(), &tp, tris.data(), tris.size()));
        HIPTRY(ctx, dupload(s.get(), &ip, m.indices, 3 * (size_t)m.num_triangles));
        HIPTRY(ctx, dupload(s.get(), &pp, m.positions, 3 * (size_t)m.num_vertices));
        np = nullptr;
        up = nullptr;
        if (!m.face_normals) HIPTRY(ctx, dupload(s.get(), &np, m.normals, 3 * (size_t)m.num_vertices));
        if (m.has_texcoords) HIPTRY(ctx, dupload(s.get(), &up, m.texcoords, 2 * (size_t)m.num_vertices));
        const LayoutF lf = flayout.get();
        blas_flevels = std::max(blas_flevels, lf.levels);
        const std::vector<float4> sv = sverts.get();
        FNode* fn;
        float4* svp;
        HIPTRY(ctx, dupload2(s.get(), &fn, lf.nodes.data(), lf.nodes.size(), &svp, sv.data(), sv.size()));
        dm.nodes = bn; dm.qnodes = qn; dm.tris = tp; dm.idx = ip; dm.pos = pp; dm.nrm = np; dm.uv = up;
        dm.svert = svp;
        dm.fnodes = fn;
        dm.froot = lf.root;
        dm.root = bvh.root;
        dm.qroot = bvh.qroot;
        dm.face_normals = m.face_normals != 0;
        dm.has_texcoords = m.has_texcoords != 0;
        s->mesh_tris += m.num_triangles;
    }

    /* ---- instances and TLAS ---- */
    std::vector<DInst> dinst(d->num_instances);
    std::vector<Box> inst_boxes(d->num_instances);
    s->inst_mats.resize(48 * (size_t)d->num_instances);
    for (int i = 0; i < d->num_instances; i++) {
        hm::M4 mat, inv, tinv;
        hm::build_transform(d->instances[i].transform, mat, inv, tinv);
        DInst& di = dinst[i];
        std::memset(&di, 0, sizeof(di));
        m4_rows(inv, di.inv);
        m4_rows(tinv, di.tinv);
        di.mesh = d->instances[i].mesh;
        s->inst_tris += d->meshes[di.mesh].num_triangles;
        di.material = d->instances[i].material;
        di.nodes = dmeshes[di.mesh].nodes;
        di.qnodes = dmeshes[di.mesh].qnodes;
        di.tris = dmeshes[di.mesh].tris;
        di.root = dmeshes[di.mesh].root;
        di.qroot = dmeshes[di.mesh].qroot;
        di.svert = dmeshes[di.mesh].svert;
        di.uv = dmeshes[di.mesh].uv;
        di.idx = dmeshes[di.mesh].idx;
        di.pos = dmeshes[di.mesh].pos;
        di.fnodes = dmeshes[di.mesh].fnodes;
        di.froot = dmeshes[di.mesh].froot;
        di.flags = (d->meshes[di.mesh].face_normals ? ILM_INST_FACE_NORMALS : 0) |
                   (d->meshes[di.mesh].has_texcoords ? ILM_INST_TEXCOORDS : 0);
        for (int k = 0; k < 16; k++) {
            s->inst_mats[48 * i + k] = mat.m[k / 4][k % 4];
            s->inst_mats[48 * i + 16 + k] = inv.m[k / 4][k % 4];
            s->inst_mats[48 * i + 32 + k] = tinv.m[k / 4][k % 4];
        }
        /* conservative world box: 8 transformed corners in double, widened by a relative
         * margin that covers the float inverse used by the traversal */
        const Box& mb = mesh_bounds[di.mesh];
        double lo[3] = {1e300, 1e300, 1e300}, hi[3] = {-1e300, -1e300, -1e300};
        bool empty = d->meshes[di.mesh].num_triangles == 0;
        for (int c = 0; c < 8 && !empty; c++) {
            double p[3] = {(c & 1) ? mb.hi[0] : mb.lo[0], (c & 2) ? mb.hi[1] : mb.lo[1], (c & 4) ? mb.hi[2] : mb.lo[2]};
            for (int a = 0; a < 3; a++) {
                double w = (double)mat.m[a][0] * p[0] + (double)mat.m[a][1] * p[1] + (double)mat.m[a][2] * p[2] + (double)mat.m[a][3];
                lo[a] = std::min(lo[a], w);
                hi[a] = std::max(hi[a], w);
            }
        }
        Box& ib = inst_boxes[i];
        if (empty) { ib.reset(); continue; }
        double ext = std::max({hi[0] - lo[0], hi[1] - lo[1], hi[2] - lo[2], 1e-30});
        for (int a = 0; a < 3; a++) {
            double mag = std::max(std::fabs(lo[a]), std::fabs(hi[a]));
            double pad = 1e-5 * ext + 1e-6 * mag;
            ib.lo[a] = round_down(lo[a] - pad);
            ib.hi[a] = round_up(hi[a] + pad);
        }
    }
    int tlas_depth = 0, tlas_qdepth = 0, tlas_flevels = 0;
    hs.tlas_root = ILM_NO_CHILD;
    hs.ftlas_root = ILM_NO_CHILD;
    hs.qtlas_root = ILM_NO_CHILD;
    if (d->num_instances > 0) {
        BuildOpts to;
        to.max_leaf = 1;
        Tree tt = build_tree(inst_boxes, to);
        Layout2 T2 = make_layout2(tt);
        LayoutQ TQ = make_layout_q(tt);
        tlas_depth = tt.max_depth;
        tlas_qdepth = TQ.max_depth;
        s->quant_max_exp = std::max(s->quant_max_exp, qnodes_max_exponent(TQ.nodes));
        /* TLAS leaves hold one instance each: store the instance index itself as the leaf's
         * `first`, so that an entry reads the DInst record directly */
        auto direct = [&tt](int32_t c) {
            if (c == ILM_NO_CHILD || c >= 0) return c;
            return ilm_leaf_code((uint32_t)tt.order[ilm_leaf_first(c)], 1u);
        };
        for (BNode& n : T2.nodes) {
            n.d.x = direct(n.d.x);
            n.d.y = direct(n.d.y);
        }
        for (QNode& n : TQ.nodes)
            for (int k = 0; k < 4; k++) n.child[k] = direct(n.child[k]);
        BNode* bn; QNode* qn;
        HIPTRY(ctx, dupload(s.get(), &bn, T2.nodes.data(), T2.nodes.size()));
        hs.tlas_root = direct(T2.root);
        const LayoutF tf = make_layout_f(T2.nodes, hs.tlas_root);
        FNode* fn;
        HIPTRY(ctx, dupload2(s.get(), &fn, tf.nodes.data(), tf.nodes.size(), &qn, TQ.nodes.data(), TQ.nodes.size()));
        hs.tlas = bn; hs.qtlas = qn;
        hs.ftlas = fn;
        hs.ftlas_root = tf.root;
        tlas_flevels = tf.levels;
        hs.qtlas_root = direct(TQ.root);
    }
    /* device stack bound: pushes never exceed the depth of the current node per level */
    const int cap = ilm_k_lds_stack() + ilm_k_ovf_stack();
    s->stack_bound_fp32 = tlas_depth + 1 + blas_depth;
    s->stack_bound_q = 3 * (tlas_qdepth + 1) + 1 + 3 * (blas_qdepth + 1);
    /* quad walk: a node leaves at most three entries, an instance entry one */
    s->stack_bound_f = 3 * tlas_flevels + 1 + 3 * blas_flevels;
    if (s->stack_bound_fp32 > cap || (ctx->opts.bvh_layout == ILM_BVH_QUANT8 && s->stack_bound_q > cap))
        return fail(ctx, ILM_E_UNSUPPORTED, "BVH too deep for the traversal stack");
    if (ctx->opts.bvh_layout == ILM_BVH_QUANT8 && s->quant_max_exp > ILM_QUANT_MAX_EXP)
        return fail(ctx, ILM_E_UNSUPPORTED, "scene extent too large for 8-bit child boxes");

    /* ---- materials, mediums, spheres, environment, camera ---- */
    std::vector<DMat> dmats(d->num_materials);
    for (int i = 0; i < d->num_materials; i++) {
        const ilm_material_desc& m = d->materials[i];
        DMat& dm = dmats[i];
        std::memset(&dm, 0, sizeof(dm));
        if (m.type < ILM_MAT_EMISSIVE || m.type > ILM_MAT_PLASTIC) return fail(ctx, ILM_E_INVALID, "bad material type");
        dm.type = m.type;
        dm.medium = m.medium;
        dm.distribution = m.distribution;
        dm.ior = m.ior;
        for (int k = 0; k < 3; k++) { dm.eta[k] = m.eta[k]; dm.k[k] = m.k[k]; }
        if (m.type == ILM_MAT_PLASTIC) dm.diffuse_fresnel = hm::diffuse_fresnel(1.0f / m.ior, 1000000);  /* src/material.cu:176 */
        int rc = upload_texture(ctx, s.get(), m.albedo, dm.albedo);
        if (rc) return rc;
        rc = upload_texture(ctx, s.get(), m.roughness, dm.roughness);
        if (rc) return rc;
    }
    std::vector<DMedium> dmed(d->num_mediums);
    for (int i = 0; i < d->num_mediums; i++) {
        const ilm_medium_desc& m = d->mediums[i];
        DMedium& dm = dmed[i];
        std::memset(&dm, 0, sizeof(dm));
        for (int k = 0; k < 3; k++) dm.absorption[k] = m.sigma_a[k];
        dm.scattering = m.sigma_s;
        dm.g = m.g;
        float l2 = (m.sigma_a[0] * m.sigma_a[0]) + (m.sigma_a[1] * m.sigma_a[1]) + (m.sigma_a[2] * m.sigma_a[2]);
        dm.active = ((double)l2 > 1e-5 || m.sigma_s > 0);   /* src/medium.cu:12 */
    }
    std::vector<DSphere> dsph(d->num_spheres);
    for (int i = 0; i < d->num_spheres; i++) {
        std::memset(&dsph[i], 0, sizeof(DSphere));
        for (int k = 0; k < 3; k++) dsph[i].c[k] = d->spheres[i].center[k];
        dsph[i].r = d->spheres[i].radius;
        dsph[i].material = d->spheres[i].material;
    }
    if (d->has_environment) {
        int rc = upload_texture(ctx, s.get(), d->environment, hs.env);
        if (rc) return rc;
    } else {
        std::memset(&hs.env, 0, sizeof(hs.env));
        hs.env.type = ILM_TEX_CONSTANT;   /* black (src/texture.h:39-43) */
    }
    {
        hm::M4 mat, inv, tinv;
        hm::build_transform(d->camera.transform, mat, inv, tinv);
        m4_rows(mat, hs.cam);
        hs.dof = d->camera.dof;
        hs.aperture = d->camera.aperture;
        s->camera = d->camera;
    }
    DInst* di; DMesh* dmp; DSphere* dsp; DMat* dma; DMedium* dme;
    HIPTRY(ctx, dupload(s.get(), &di, dinst.data(), dinst.size()));
    HIPTRY(ctx, dupload(s.get(), &dmp, dmeshes.data(), dmeshes.size()));
    HIPTRY(ctx, dupload(s.get(), &dsp, dsph.data(), dsph.size()));
    HIPTRY(ctx, dupload(s.get(), &dma, dmats.data(), dmats.size()));
    HIPTRY(ctx, dupload(s.get(), &dme, dmed.data(), dmed.size()));
    hs.inst = di; hs.meshes = dmp; hs.spheres = dsp; hs.mats = dma; hs.mediums = dme;
    hs.n_inst = d->num_instances;
    hs.n_spheres = d->num_spheres;
    DScene* ds;
    HIPTRY(ctx, dupload(s.get(), &ds, &hs, 1));
    s->d_scene = ds;
    s->h_scene = hs;
    s->num_instances = d->num_instances;
    s->refs.store(1);
    {
        std::lock_guard<std::mutex> lk(ctx->sched_mu);
        ctx->in_use += s->bytes;
    }
    ctx->refs.fetch_add(1);
    *out = s.release();
    return ILM_OK;
}

void ctx_unref(ilm_ctx* ctx);

/* Drops one reference; the last frees the scene's device memory. sched_locked: the caller holds
 * the context's sched_mu (the scheduler's own release paths). */
static void scene_release(ilm_scene* s, bool sched_locked = false) {
    if (!s) return;
    if (s->refs.fetch_sub(1) != 1) return;
    ilm_ctx* ctx = s->ctx;
    (void)hipSetDevice(ctx->device);
    for (void* p : s->allocs) dfree(ctx->device, p);
    s->allocs.clear();
    (void)hipGetLastError();
    if (sched_locked) {
        ctx->in_use -= s->bytes;
    } else {
        std::lock_guard<std::mutex> lk(ctx->sched_mu);
        ctx->in_use -= s->bytes;
    }
    delete s;
    /* the scheduler thread never holds the last context reference (ilm_close joins it first) */
    ctx_unref(ctx);
}

void ilm_scene_free(ilm_scene* s) { scene_release(s); }
int64_t ilm_scene_device_bytes(const ilm_scene* s) { return s ? s->bytes : -1; }

int ilm_debug_instance_matrices(const ilm_scene* s, int32_t i, float* out48) {
    if (!s || !out48 || i < 0 || i >= s->num_instances) return fail(nullptr, ILM_E_INVALID, "bad instance");
    std::memcpy(out48, &s->inst_mats[48 * (size_t)i], 48 * sizeof(float));
    return ILM_OK;
}

/* ======================= context ======================= */

static void ctx_free_paths(ilm_ctx* ctx) {
    for (void* p : ctx->path_allocs) dfree(ctx->device, p);
    ctx->path_allocs.clear();
    ctx->own_bytes -= ctx->path_bytes;
    ctx->path_bytes = 0;
    ctx->A = DPaths{};
    ctx->B = DPaths{};
    ctx->hits = DHits{};
    ctx->contrib = nullptr;
    ctx->cap = 0;
}

static int ctx_alloc_paths(ilm_ctx* ctx, int64_t cap) {
    auto A = [&](void** p, size_t b) -> hipError_t {
        hipError_t e = hipMalloc(p, b);
        if (e == hipSuccess) { ctx->path_allocs.push_back(*p); ctx->own_bytes += (int64_t)b; ctx->path_bytes += (int64_t)b; }
        return e;
    };
    for (int k = 0; k < ctx->npipes; k++) {
        for (DPaths* P : {k ? &ctx->A2 : &ctx->A, k ? &ctx->B2 : &ctx->B}) {
            HIPTRY(ctx, A((void**)&P->o, cap * sizeof(float4)));
            HIPTRY(ctx, A((void**)&P->d, cap * sizeof(float4)));
            HIPTRY(ctx, A((void**)&P->c, cap * sizeof(float4)));
            HIPTRY(ctx, A((void**)&P->rng, cap * sizeof(uint2)));
        }
        DHits& h = k ? ctx->hits2 : ctx->hits;
        HIPTRY(ctx, A((void**)&h.h, cap * sizeof(float4)));
        HIPTRY(ctx, A((void**)&h.inst, cap * sizeof(int)));
        HIPTRY(ctx, A((void**)(k ? &ctx->contrib2 : &ctx->contrib), cap * sizeof(float4)));
    }
    ctx->cap = cap;
    return ILM_OK;
}

static bool opts_valid(const ilm_opts& o) {
    const bool sg_ok = o.sample_group >= 0 && o.sample_group <= 4096 && (o.sample_group & (o.sample_group - 1)) == 0;
    return !(o.bvh_layout < 0 || o.bvh_layout > ILM_BVH_QUANT8 || o.tri_test < 0 || o.tri_test > ILM_TRI_WATERTIGHT ||
             o.extend_mode < 0 || o.extend_mode > ILM_EXTEND_STEP_REFILL || !sg_ok || o.tile_rows < 0 || o.tile_rows > 256 ||
             o.refill_min < 0 || o.refill_min > 64 || o.ext_fetch < 0 || o.ext_fetch > 65536 || (o.ext_fetch & 63) != 0 ||
             o.leaf_wait_pct < 0 || o.leaf_wait_pct > 10000 || o.shade_sort < 0 || o.shade_sort > 2 ||
             o.sched_fair < 0 || o.sched_fair > 1 || o.camera_packets < 0 || o.camera_packets > 2 ||
             o.chunk_passes < 0 || o.paths_in_flight < 0 || o.hbm_budget_bytes < 0 || o.max_queued < 0 ||
             o.pipes < 0 || o.pipes > 2 || o.lone_split < 0 || o.lone_split > 2);
}

/* extend scheduling actually used (ILM_EXTEND_DEFAULT is the per-step refill) */
static int ext_mode_of(const ilm_opts& o) {
    return o.extend_mode == ILM_EXTEND_DEFAULT ? ILM_EXTEND_STEP_REFILL : o.extend_mode;
}

static int64_t cap_of(const ilm_opts& o) {
    /* 2^26 paths (~9.5 GB of path state) hold a whole 1024x1024x64 render in one chunk: every
     * depth is one launch over all live paths, so launch tails are amortised */
    int64_t cap = o.paths_in_flight > 0 ? o.paths_in_flight : (int64_t)1 << 26;
    cap = std::max<int64_t>(cap, 4096);
    return std::min<int64_t>(cap, (int64_t)1 << 30);
}

/* the traversal-stack spill area: one half per chunk pipeline */
static size_t ovf_pipe_ints(const ilm_ctx* ctx) {
    return (size_t)ctx->ovf_grid * ilm_k_ext_block() * ilm_k_ovf_stack();
}
static size_t ovf_bytes(const ilm_ctx* ctx) {
    return (size_t)ctx->npipes * ovf_pipe_ints(ctx) * sizeof(int);
}

int ilm_open(int device, const ilm_opts* opts, ilm_ctx** out) {
    if (!out) return fail(nullptr, ILM_E_INVALID, "null out");
    *out = nullptr;
    if (opts && !opts_valid(*opts)) return fail(nullptr, ILM_E_INVALID, "bad ilm_opts field");
    int n = 0;
    hipError_t e = hipGetDeviceCount(&n);
    if (e != hipSuccess || n == 0) return fail(nullptr, ILM_E_DEVICE, "no HIP device available");
    if (device < 0 || device >= n) return fail(nullptr, ILM_E_INVALID, "device index out of range");
    std::unique_ptr<ilm_ctx> c(new ilm_ctx());
    ilm_ctx* ctx = c.get();
    ctx->device = device;
    ctx->t0 = std::chrono::steady_clock::now();
    std::memset(&ctx->opts, 0, sizeof(ctx->opts));
    ctx->opts.use_graphs = 1;
    if (opts) ctx->opts = *opts;
    if (ctx->opts.bvh_cache_dir) ctx->bvh_cache_dir = ctx->opts.bvh_cache_dir;
    ctx->opts.bvh_cache_dir = nullptr;   /* the caller's string is not kept */
    HIPTRY(ctx, hipSetDevice(device));
    hipDeviceProp_t prop;
    HIPTRY(ctx, hipGetDeviceProperties(&prop, device));
    ctx->n_cu = prop.multiProcessorCount;
    HIPTRY(ctx, hipStreamCreateWithFlags(&ctx->stream, hipStreamNonBlocking));
    HIPTRY(ctx, hipStreamCreateWithFlags(&ctx->copy_stream, hipStreamNonBlocking));
    ctx->npipes = ctx->opts.pipes == 1 ? 1 : 2;
    if (ctx->npipes == 2) HIPTRY(ctx, hipStreamCreateWithFlags(&ctx->stream2, hipStreamNonBlocking));
    for (int i = 0; i < 2; i++) HIPTRY(ctx, hipEventCreateWithFlags(&ctx->acc_ev[i], hipEventDisableTiming));
    HIPTRY(ctx, hipEventCreateWithFlags(&ctx->fill_ev, hipEventDisableTiming));
    int occ = ilm_k_extend_occupancy(ctx->opts.tri_test, ctx->opts.bvh_layout, ext_mode_of(ctx->opts));
    ctx->ext_grid = ctx->n_cu * std::max(1, occ);
    ctx->gen_grid = ctx->n_cu * 8;
    ctx->fin_grid = std::min(ILM_TAIL_WAVES, ctx->n_cu * ilm_k_finish_occupancy());
    /* 512-thread blocks, block-stride loop: one resident wave of blocks, no stragglers */
    ctx->shade_grid = ctx->n_cu * ilm_k_shade_occupancy(ctx->opts.shade_sort != 2);
    int rc = ctx_alloc_paths(ctx, cap_of(ctx->opts));
    if (rc) return rc;
    auto A = [&](void** p, size_t b) -> hipError_t {
        hipError_t e2 = hipMalloc(p, b);
        if (e2 == hipSuccess) { ctx->allocs.push_back(*p); ctx->own_bytes += (int64_t)b; }
        return e2;
    };
    ctx->ovf_grid = ctx->ext_grid;
    HIPTRY(ctx, hipMalloc((void**)&ctx->ovf, ovf_bytes(ctx)));
    ctx->own_bytes += (int64_t)ovf_bytes(ctx);
    HIPTRY(ctx, A((void**)&ctx->ctl, sizeof(DCtl)));
    HIPTRY(ctx, A((void**)&ctx->d_chunk, sizeof(DChunk)));
    if (ctx->npipes == 2) {
        HIPTRY(ctx, A((void**)&ctx->ctl2, sizeof(DCtl)));
        HIPTRY(ctx, A((void**)&ctx->d_chunk2, sizeof(DChunk)));
    }
    HIPTRY(ctx, A((void**)&ctx->d_seg_total, 2 * sizeof(unsigned long long)));
    HIPTRY(ctx, A((void**)&ctx->d_trav, 2 * sizeof(unsigned long long)));
    HIPTRY(ctx, hipMemsetAsync(ctx->d_seg_total, 0, 2 * sizeof(unsigned long long), ctx->stream));
    HIPTRY(ctx, hipMemsetAsync(ctx->d_trav, 0, 2 * sizeof(unsigned long long), ctx->stream));
    HIPTRY(ctx, hipStreamSynchronize(ctx->stream));
    for (int i = 0; i < ILM_RING; i++) {
        HIPTRY(ctx, hipHostMalloc((void**)&ctx->h_chunk[i], sizeof(DChunk), hipHostMallocDefault));
        HIPTRY(ctx, hipEventCreateWithFlags(&ctx->ring_ev[i], hipEventDisableTiming));
    }
    HIPTRY(ctx, hipHostMalloc((void**)&ctx->h_report, ILM_MAX_DEPTH * sizeof(unsigned long long), hipHostMallocDefault));
    std::memset(ctx->h_report, 0, ILM_MAX_DEPTH * sizeof(unsigned long long));
    HIPTRY(ctx, hipHostMalloc((void**)&ctx->h_u64, 4 * sizeof(unsigned long long), hipHostMallocDefault));
    HIPTRY(ctx, hipHostMalloc((void**)&ctx->h_seg_ring, ILM_RING * sizeof(unsigned long long), hipHostMallocDefault));
    for (int i = 0; i < 2; i++) HIPTRY(ctx, hipEventCreate(&ctx->na_ev[i]));
    for (int i = 0; i < 2; i++) HIPTRY(ctx, hipEventCreate(&ctx->rend_ev[i]));
    HIPTRY(ctx, noalloc_scratch_of(device, &ctx->noalloc_scratch));
    size_t free_b = 0, total_b = 0;
    HIPTRY(ctx, hipMemGetInfo(&free_b, &total_b));
    ctx->budget = ctx->opts.hbm_budget_bytes > 0 ? ctx->opts.hbm_budget_bytes : (int64_t)(0.9 * (double)free_b);
    *out = c.release();
    return ILM_OK;
}

static void server_stop(ilm_ctx* ctx);
static void stage_trim(ilm_ctx* ctx);

static void ctx_destroy(ilm_ctx* ctx) {
    (void)hipSetDevice(ctx->device);
    (void)hipStreamSynchronize(ctx->stream);
    if (ctx->stream2) (void)hipStreamSynchronize(ctx->stream2);
    for (auto& kv : ctx->graphs) (void)hipGraphExecDestroy(kv.second);
    ctx_free_paths(ctx);
    dfree(ctx->device, ctx->ovf);
    for (auto& kv : ctx->bufs.free) dfree(ctx->device, kv.second);
    ctx->bufs.free.clear();
    stage_trim(ctx);
    for (void* p : ctx->allocs) dfree(ctx->device, p);
    dfree(ctx->device, ctx->seg_count);
    for (int i = 0; i < ILM_RING; i++) {
        if (ctx->h_chunk[i]) (void)hipHostFree(ctx->h_chunk[i]);
        if (ctx->ring_ev[i]) (void)hipEventDestroy(ctx->ring_ev[i]);
    }
    if (ctx->h_report) (void)hipHostFree(ctx->h_report);
    if (ctx->h_u64) (void)hipHostFree(ctx->h_u64);
    if (ctx->h_seg_ring) (void)hipHostFree(ctx->h_seg_ring);
    for (int i = 0; i < 2; i++) {
        if (ctx->na_ev[i]) (void)hipEventDestroy(ctx->na_ev[i]);
        if (ctx->rend_ev[i]) (void)hipEventDestroy(ctx->rend_ev[i]);
        if (ctx->acc_ev[i]) (void)hipEventDestroy(ctx->acc_ev[i]);
    }
    if (ctx->fill_ev) (void)hipEventDestroy(ctx->fill_ev);
    if (ctx->stream2) (void)hipStreamDestroy(ctx->stream2);
    if (ctx->copy_stream) (void)hipStreamDestroy(ctx->copy_stream);
    (void)hipStreamDestroy(ctx->stream);
    (void)hipGetLastError();
    delete ctx;
}

void ctx_unref(ilm_ctx* ctx) {
    if (ctx->refs.fetch_sub(1) == 1) ctx_destroy(ctx);
}

/* Stops the scheduler (queued and running requests end cancelled) and drops the caller's
 * reference; scenes and request handles still alive keep the device resources until freed. */
void ilm_close(ilm_ctx* ctx) {
    if (!ctx) return;
    server_stop(ctx);
    {
        std::lock_guard<std::mutex> dev(ctx->dev_mu);
        (void)hipSetDevice(ctx->device);
        (void)hipStreamSynchronize(ctx->stream);
        if (ctx->stream2) (void)hipStreamSynchronize(ctx->stream2);
    }
    ctx_unref(ctx);
}

/* Retune an idle context: bvh_layout, extend_mode, refill_min, ext_fetch, leaf_wait_pct, shade_sort,
 * sched_fair, camera_packets, sample_group, tile_rows, chunk_passes, paths_in_flight and lone_split take the values in *o (the
 * other fields are ignored). Every scene carries both node layouts, so a layout change needs no
 * upload. Path buffers are reallocated when the chunk size changes; captured graphs are dropped. */
int ilm_tune(ilm_ctx* ctx, const ilm_opts* o) {
    if (!ctx || !o) return fail(ctx, ILM_E_INVALID, "null argument");
    if (!opts_valid(*o)) return fail(ctx, ILM_E_INVALID, "bad ilm_opts field");
    std::lock_guard<std::mutex> sched(ctx->sched_mu);
    if (!ctx->pending.empty() || !ctx->active.empty()) return fail(ctx, ILM_E_BUSY, "requests in flight");
    std::lock_guard<std::mutex> dev(ctx->dev_mu);
    HIPTRY(ctx, hipSetDevice(ctx->device));
    HIPTRY(ctx, hipStreamSynchronize(ctx->stream));
    if (ctx->stream2) HIPTRY(ctx, hipStreamSynchronize(ctx->stream2));
    for (auto& kv : ctx->graphs) (void)hipGraphExecDestroy(kv.second);
    ctx->graphs.clear();
    if (ext_mode_of(*o) != ext_mode_of(ctx->opts) || o->bvh_layout != ctx->opts.bvh_layout) {
        const int occ = ilm_k_extend_occupancy(ctx->opts.tri_test, o->bvh_layout, ext_mode_of(*o));
        const int grid = ctx->n_cu * std::max(1, occ);
        if (grid > ctx->ovf_grid) {
            /* the spill area is sized for the grid: grow it before the grid grows (on failure
             * the context keeps its old mode, grid and buffer) */
            const size_t nb = (size_t)ctx->npipes * grid * ilm_k_ext_block() * ilm_k_ovf_stack() * sizeof(int);
            int* fresh = nullptr;
            HIPTRY(ctx, hipMalloc((void**)&fresh, nb));
            dfree(ctx->device, ctx->ovf);
            ctx->own_bytes += (int64_t)nb - (int64_t)ovf_bytes(ctx);
            ctx->ovf = fresh;
            ctx->ovf_grid = grid;
        }
        ctx->ext_grid = grid;
    }
    ctx->opts.bvh_layout = o->bvh_layout;
    ctx->opts.extend_mode = o->extend_mode;
    ctx->opts.sample_group = o->sample_group;
    ctx->opts.tile_rows = o->tile_rows;
    ctx->opts.refill_min = o->refill_min;
    ctx->opts.ext_fetch = o->ext_fetch;
    ctx->opts.leaf_wait_pct = o->leaf_wait_pct;
    ctx->opts.shade_sort = o->shade_sort;
    ctx->opts.sched_fair = o->sched_fair;
    ctx->opts.camera_packets = o->camera_packets;
    ctx->shade_grid = ctx->n_cu * ilm_k_shade_occupancy(ctx->opts.shade_sort != 2);
    ctx->opts.chunk_passes = o->chunk_passes;
    ctx->opts.lone_split = o->lone_split;
    const int64_t cap = cap_of(*o);
    if (cap != ctx->cap) {
        ctx_free_paths(ctx);
        int rc = ctx_alloc_paths(ctx, cap);
        if (rc) {
            ctx_free_paths(ctx);
            if (ctx_alloc_paths(ctx, 4096) != ILM_OK) return fail(ctx, ILM_E_NOMEM, "path buffers lost after a failed resize");
            return rc;
        }
    }
    ctx->opts.paths_in_flight = o->paths_in_flight;
    return ILM_OK;
}

const char* ilm_last_error(ilm_ctx* ctx) {
    if (!ctx) return g_err.c_str();
    std::lock_guard<std::mutex> lk(ctx->err_mu);
    ctx->err_copy = ctx->err;
    return ctx->err_copy.c_str();
}

/* ======================= chunk pipeline ======================= */

/* whether a scene needs the spilling traversal stack under this context's layout */
static bool scene_needs_ovf(const ilm_ctx* ctx, const ilm_scene* s) {
    const int bound = ctx->opts.bvh_layout == ILM_BVH_QUANT8 ? s->stack_bound_q : s->stack_bound_fp32;
    return bound > ilm_k_lds_stack();
}
/* whether the scene's FNode trees fit the quad walk's stacks */
static bool scene_fits_quad(const ilm_scene* s) { return s->stack_bound_f <= ILM_QUAD_STACK; }
static bool jobs_fit_quad(const std::vector<Job*>& jobs) {
    for (const Job* j : jobs)
        if (!scene_fits_quad(j->scene)) return false;
    return true;
}
static bool jobs_need_ovf(const ilm_ctx* ctx, const std::vector<Job*>& jobs) {
    for (const Job* j : jobs)
        if (scene_needs_ovf(ctx, j->scene)) return true;
    return false;
}

/* The context's own chunk pipeline k (0, or 1 when npipes == 2). */
static Pipe ctx_pipe(const ilm_ctx* ctx, int k = 0) {
    Pipe q;
    q.idx = k;
    q.stream = k ? ctx->stream2 : ctx->stream;
    q.A = k ? ctx->A2 : ctx->A;
    q.B = k ? ctx->B2 : ctx->B;
    q.hits = k ? ctx->hits2 : ctx->hits;
    q.contrib = k ? ctx->contrib2 : ctx->contrib;
    q.ctl = k ? ctx->ctl2 : ctx->ctl;
    q.chunk = k ? ctx->d_chunk2 : ctx->d_chunk;
    q.ovf = ctx->ovf + (k ? ovf_pipe_ints(ctx) : 0);
    q.ext_grid = ctx->ext_grid;
    q.seg_total = ctx->d_seg_total;
    return q;
}

static KParams base_params(ilm_ctx* ctx, const Pipe& q) {
    KParams P;
    std::memset(&P, 0, sizeof(P));
    P.chunk = q.chunk;
    P.ctl = q.ctl;
    P.in = q.A;
    P.out = q.B;
    P.hits = q.hits;
    P.contrib = q.contrib;
    P.bvh_layout = ctx->opts.bvh_layout;
    P.tri_test = ctx->opts.tri_test;
    P.extend_mode = ext_mode_of(ctx->opts);
    P.tile_rows = ctx->opts.tile_rows > 0 ? ctx->opts.tile_rows : 4;
    P.refill_min = ctx->opts.refill_min > 0 ? ctx->opts.refill_min : 24;
    P.ext_fetch = ctx->opts.ext_fetch > 0 ? ctx->opts.ext_fetch : 256;
    P.leaf_pct = ctx->opts.leaf_wait_pct > 0 ? ctx->opts.leaf_wait_pct : 60;
    P.shade_sort = ctx->opts.shade_sort == 2 ? 0 : 1;
    P.packet0 = ctx->opts.camera_packets == 2 ? 0 : 1;
    P.trav_stats = ctx->opts.count_tests ? ctx->d_trav : nullptr;
    return P;
}
static KParams base_params(ilm_ctx* ctx) { return base_params(ctx, ctx_pipe(ctx)); }

/* Queues of at most this many paths are finished by k_finish in one launch instead of two launches
 * per remaining depth. A depth of a short queue costs the per-depth kernels some 110 us however
 * few its paths are: the slowest of its walks, of one lane, and the launches (a 100k-triangle
 * mesh, 1920x1080, 1 spp: 90 us per depth past the fifth). k_finish keeps 5120 waves of 64
 * paths resident; past that a wave runs share after share, and its quads trace a long queue at
 * 0.4 of the per-lane kernel's rate. Measured over limits of 50k to 1.4M: 320x240, 8 spp, depth 45
 * in a medium 5.75 ms without, 3.49 at 50k, 2.82 at 200k, 2.76 at 330k, 3.06 at 700k; 960x720,
 * 32 spp 27.9, 27.8, 27.0, 27.4, 30.6; 640x480, 32 spp, depth 16 5.63, 5.55, 5.03, 4.93, 5.13. */
#define ILM_TAIL_PATHS (1 << 18)

/* How this chunk's launches trace it: short queues go to k_finish when every scene's FNode trees
 * fit its stacks (not while every depth's extend launch is timed or its tests counted, nor when
 * the caller asked for an extend kernel by name). */
static void chunk_choices(const ilm_ctx* ctx, uint32_t total_paths, bool quad_fits, KParams& P) {
    const bool quad = quad_fits && ctx->opts.extend_mode == ILM_EXTEND_DEFAULT && !ctx->opts.profile && !ctx->opts.count_tests;
    P.quad_max = quad ? ILM_TAIL_PATHS : 0;
    P.packet_f = quad_fits && P.uni_scene ? 1 : 0;
    P.tail_only = (int64_t)total_paths <= (int64_t)P.quad_max ? 1 : 0;
}

/* Whether a request's camera rays are traced as packets by default. A packet visits the union of
 * its 64 rays' walks, and one wave carries it to its end, so it pays while the 64 / sgroup pixels
 * it covers show few triangles; the scene's triangles per image pixel stand for that. First-depth
 * time as packets over FNodes / per lane with 8-bit nodes, by triangles in the footprint: 100k
 * triangles at 1920x1080 0.74 (0.4, 8 samples), 0.76 (1.6, 2), 0.88 (3.1, 1); at 640x480 0.67 (2.6,
 * 8), 0.72 (5, 4), 0.90 (10, 2), 1.09 (21, 1); 11 small meshes 0.70 (4.4, 8), 0.83 (8.8, 4), 0.94
 * (18, 2), 1.23 (35, 1); 32k triangles at 320x240 0.82 (6.7, 4), 0.94 (13, 2), 0.95 (27, 1); 12
 * instances of 722k 0.69 (9.4, 64), 0.80 (19, 32), 1.04 (38, 16), 1.32 (75, 8), 4.0 (600, 1). At one
 * sample the 64 pixels differ more (32k triangles at 400x300, three passes: 1.11 at 17), so the line
 * lies at half the triangles there; packets over the other layouts (several scenes in a chunk, very
 * deep trees) cost about a fifth more and lose at one sample. */
#define ILM_PACKET_MAX_TRIS 20
static bool packet_pays(const ilm_scene* s, const ilm_render_params& p, uint32_t sgroup, bool fnodes) {
    if (sgroup < 2 && !fnodes) return false;
    const double limit = sgroup < 2 ? 0.5 * ILM_PACKET_MAX_TRIS : ILM_PACKET_MAX_TRIS;
    return (double)s->inst_tris * 64.0 <= limit * (double)sgroup * p.width * p.height;
}

/* Stage a chunk descriptor: pinned ring slot -> pipeline q's device copy, on its stream, with the
 * pipeline's queue counters (k_stage reads the slot itself). */
static int stage_slot(ilm_ctx* ctx, int slot, int n_req, const Pipe& q) {
    HIPTRY(ctx, ilm_k_stage(q.ctl, q.chunk, ctx->h_chunk[slot], n_req, ctx->h_chunk[slot]->n_work, q.stream));
    HIPTRY(ctx, hipEventRecord(ctx->ring_ev[slot], q.stream));
    return ILM_OK;
}
static int stage_chunk(ilm_ctx* ctx, const DChunk& hc, int n_req, const Pipe& q) {
    int slot = ctx->ring_pos++ % ILM_RING;
    HIPTRY(ctx, hipEventSynchronize(ctx->ring_ev[slot]));
    DChunk* d = ctx->h_chunk[slot];
    std::memcpy(d, &hc, offsetof(DChunk, reqs));
    std::memcpy(d->reqs, hc.reqs, (size_t)n_req * sizeof(DReq));
    std::memcpy(d->work, hc.work, (size_t)hc.n_work * sizeof(DWork));
    return stage_slot(ctx, slot, n_req, q);
}

/* have the chunk's depths report their counts (see enqueue_depths) */
static void report_counts(ilm_ctx* ctx, KParams& P) {
    if (P.quad_max == 0 || P.tail_only) return;
    P.report = ctx->h_report;
    P.report_tag = ++ctx->report_tag;
}

/* A chunk's first launch after k_stage. With per-step refill the first depth's extend and
 * shade form the camera rays where they use them, so only the per-path results are cleared
 * (by the packet extend itself when the first depth runs as packets); the other extend modes
 * read the rays k_raygen writes out. */
static hipError_t start_paths(ilm_ctx* ctx, const Pipe& q, KParams& P, hipStream_t s) {
    P.in = q.A;
    P.cam0 = P.extend_mode == ILM_EXTEND_STEP_REFILL ? 1 : 0;
    if (P.cam0 && (P.packet0 || P.tail_only)) return hipSuccess;
    return P.cam0 ? ilm_k_path_clear(P, ctx->gen_grid, s) : ilm_k_raygen(P, ctx->gen_grid, s);
}

/* The count of the queue that k_shade found at `depth`, if it is there (in h_report with the chunk's
 * tag). */
static bool report_there(const KParams& P, int depth, uint32_t& count) {
    const unsigned long long v = __atomic_load_n(P.report + depth, __ATOMIC_RELAXED);
    count = (uint32_t)v;
    return (uint32_t)(v >> 32) == P.report_tag;
}
/* The same, waited for. The thread keeps its processor: what it waits for is at most one depth away
 * from leaving the GPU idle, and on a busy host a yield gives away several milliseconds. */
static int wait_report(ilm_ctx* ctx, const Pipe& q, const KParams& P, int depth, uint32_t& count) {
    for (unsigned spin = 1;; spin++) {
        const bool look = (spin & 255u) == 0;
        const hipError_t e = look ? hipStreamQuery(q.stream) : hipErrorNotReady;
        if (report_there(P, depth, count)) return ILM_OK;
        if (e == hipSuccess) return fail(ctx, ILM_E_DEVICE, "a depth ended without its count");
        if (e != hipErrorNotReady) HIPTRY(ctx, e);
        if (look) (void)hipGetLastError();
    }
}

/* How many of a chunk's D depths to have launched in all, when `launched` are and the first `known`
 * (two or more) have reported their counts. Once a queue is at most `limit`, no more. Otherwise at once
 * all whose queues are still longer than `limit` if each is shorter than the one before by the ratio
 * of the last two known, whose launches need no further word from the host, and the two after them
 * that would be launched while their counts are waited for. A host that finds every launched depth reported came late, the GPU is about to
 * run dry or has, and it will be late again: all of them, as if nothing were reported. */
static int depths_to_launch(const uint32_t* count, int known, int launched, int D, uint32_t limit) {
    const uint32_t last = count[known - 1];
    if (last <= limit) return launched;
    const double ratio = (double)last / (double)std::max(1u, count[known - 2]);
    if (known >= launched || ratio >= 1.0) return D;
    const double more = std::ceil(std::log((double)limit / last) / std::log(ratio)) - 1.0;
    return (int)std::min<double>(D, known + more + 2.0);
}
int ilm_debug_depths_to_launch(const uint32_t* counts, int32_t known, int32_t launched, int32_t depth_steps, uint32_t limit) {
    if (!counts || known < 2 || known > launched || launched > depth_steps || limit == 0) return ILM_E_INVALID;
    return depths_to_launch(counts, known, launched, depth_steps, limit);
}

/* The launch sequence of one chunk with depth_steps depth iterations, in two parts: the depths
 * (first rays, extend and shade per depth, k_finish), then the accumulation into the requests'
 * Kahan sums and the segment count.
 *
 * With P.report the depths are launched ahead of the counts that k_shade reports, and no more of them
 * once a queue is left to k_finish (depths_to_launch): the two launches of a depth with nothing to do
 * take 9 us, and a render of 45 depths whose queue is short after four spent 0.37 of its 2.5 ms on the
 * others. On a host whose processor is shared with one and with three busy threads that render takes 4.0
 * and 8.0 ms of wall time at the median (7.2 and 15.7 with all depths launched ahead through a graph,
 * 16 and 32 with two depths ahead and a thread that yields), a 1024x1024, 16 spp, depth 16 one 10.8 and
 * 19.3 (22 and 48, 20 and 40). */
static int enqueue_depths(ilm_ctx* ctx, const Pipe& q, const KParams& base, int depth_steps, ProfileSink* prof) {
    const bool follow = base.report != nullptr;
    hipStream_t s = q.stream;
    KParams P = base;
    HIPTRY(ctx, start_paths(ctx, q, P, s));
    int goal = base.tail_only ? 0 : follow ? std::min(3, depth_steps) : depth_steps;
    uint32_t counts[ILM_MAX_DEPTH];
    int known = 0;
    for (int d = 0;; d++) {
        if (d == goal) {
            if (!follow || goal == depth_steps) break;
            for (; known < d - 1; known++) {
                const int rc = wait_report(ctx, q, P, known, counts[known]);
                if (rc) return rc;
            }
            if (report_there(P, known, counts[known])) known++;
            goal = depths_to_launch(counts, known, d, depth_steps, (uint32_t)P.quad_max);
            if (goal == d) break;
        }
        P.in = (d & 1) ? q.B : q.A;
        P.out = (d & 1) ? q.A : q.B;
        if (prof) {
            hipEvent_t a, b;
            HIPTRY(ctx, hipEventCreate(&a));
            HIPTRY(ctx, hipEventCreate(&b));
            HIPTRY(ctx, hipEventRecord(a, s));
            HIPTRY(ctx, ilm_k_extend(P, d, q.ovf, q.ext_grid, s));
            HIPTRY(ctx, hipEventRecord(b, s));
            prof->ev.push_back({a, b});
        } else {
            HIPTRY(ctx, ilm_k_extend(P, d, q.ovf, q.ext_grid, s));
        }
        HIPTRY(ctx, ilm_k_shade(P, d, ctx->shade_grid, s));
    }
    if (base.quad_max > 0) {
        P.in = q.A;
        P.out = q.B;
        HIPTRY(ctx, ilm_k_finish(P, ctx->fin_grid, s));
    }
    return ILM_OK;
}
/* blocks: enough for the chunk's pixels, 64 each (a captured graph serves chunks of any size) */
static int acc_grid(const ilm_ctx* ctx, int64_t total_px) {
    return (int)std::max<int64_t>(1, std::min<int64_t>((total_px + 63) / 64, ctx->gen_grid * 4));
}
static int enqueue_finish(ilm_ctx* ctx, const Pipe& q, const KParams& base, int64_t total_px) {
    HIPTRY(ctx, ilm_k_accumulate(base, acc_grid(ctx, total_px), q.seg_total, q.stream));
    return ILM_OK;
}
/* both parts, on one stream (debug paths and the allocation-free render) */
static int enqueue_pipeline(ilm_ctx* ctx, const Pipe& q, const KParams& base, int depth_steps, int64_t total_px, ProfileSink* prof) {
    int rc = enqueue_depths(ctx, q, base, depth_steps, prof);
    return rc ? rc : enqueue_finish(ctx, q, base, total_px);
}

/* whether every request of the chunk renders the same scene (the extend kernel then reads it
 * once from the chunk descriptor, so a graph captured for it serves any later single-scene chunk) */
static bool chunk_uni_scene(const DChunk& hc) {
    bool uni = hc.n_work > 0;
    for (int k = 1; k < hc.n_work && uni; k++) uni = hc.reqs[hc.work[k].req].scene == hc.reqs[hc.work[0].req].scene;
    return uni && hc.work[0].req == 0;
}

/* Replay (capturing on first use) the graph of one part of a chunk's launch sequence. */
static int run_graph(ilm_ctx* ctx, int key, const Pipe& q, const KParams& P, int D, bool finish) {
    auto it = ctx->graphs.find(key);
    if (it == ctx->graphs.end()) {
        hipGraph_t g = nullptr;
        hipGraphExec_t ge = nullptr;
        {
            std::lock_guard<std::mutex> cap(capture_mu(ctx->device));
            HIPTRY(ctx, hipStreamBeginCapture(q.stream, hipStreamCaptureModeThreadLocal));
            int rc2 = finish ? enqueue_finish(ctx, q, P, (int64_t)1 << 40) : enqueue_depths(ctx, q, P, D, nullptr);
            hipError_t ec = hipStreamEndCapture(q.stream, &g);
            if (rc2) return rc2;
            if (ec != hipSuccess) return fail(ctx, ILM_E_DEVICE, std::string("graph capture: ") + hipGetErrorString(ec));
        }
        HIPTRY(ctx, hipGraphInstantiate(&ge, g, nullptr, nullptr, 0));
        (void)hipGraphDestroy(g);
        it = ctx->graphs.emplace(key, ge).first;
    }
    HIPTRY(ctx, hipGraphLaunch(it->second, q.stream));
    return ILM_OK;
}

/* Launch a chunk on the next pipeline. Its depths start at once, beside whatever the other
 * pipeline still runs; its accumulation waits for the previous chunk's (acc_ev of the other
 * pipeline) and for the latest clear of request buffers (fill_ev), so every pixel's sums grow
 * in pass order. Profiling and test counting keep one pipeline. Sets *pipe_used. */
static int launch_chunk(ilm_ctx* ctx, const DChunk& hc, const std::vector<Job*>& jobs, ProfileSink* prof, bool alone, int* pipe_used = nullptr) {
    const bool two = ctx->npipes == 2 && !prof && !ctx->opts.count_tests;
    const int k = two ? ctx->next_pipe : 0;
    if (two) ctx->next_pipe ^= 1;
    const Pipe q = ctx_pipe(ctx, k);
    int rc = stage_chunk(ctx, hc, (int)jobs.size(), q);
    if (rc) return rc;
    KParams P = base_params(ctx, q);
    const bool ovf = jobs_need_ovf(ctx, jobs);
    P.use_ovf = ovf ? 1 : 0;
    const bool uni = chunk_uni_scene(hc);
    P.uni_scene = uni ? 1 : 0;
    chunk_choices(ctx, hc.total_paths, jobs_fit_quad(jobs), P);
    if (ctx->opts.camera_packets == 0)
        for (int w = 0; w < hc.n_work && P.packet0; w++) {
            const Job* j = jobs[hc.work[w].req];
            P.packet0 = packet_pays(j->scene, j->p, hc.work[w].sgroup, P.packet_f) ? 1 : 0;
        }
    const int D = hc.depth_steps;
    /* the only chunk of a call: its thread has nothing else to launch and follows its counts */
    if (alone) report_counts(ctx, P);
    /* a chunk that k_finish does alone is two launches: launched directly, without the 15 us or so
     * that starting two graphs takes */
    const bool graphs = ctx->opts.use_graphs && !prof && !ctx->opts.count_tests && !P.tail_only && !P.report;
    if (graphs) rc = run_graph(ctx, 2 * (64 * D + 32 * P.packet_f + 16 * P.packet0 + 8 * (P.quad_max > 0) + 4 * k + (uni ? 2 : 0) + (ovf ? 1 : 0)), q, P, D, false);
    else rc = enqueue_depths(ctx, q, P, D, prof);
    if (rc) return rc;
    if (ctx->npipes == 2) {
        HIPTRY(ctx, hipStreamWaitEvent(q.stream, ctx->acc_ev[k ^ 1], 0));
        if (k == 1) HIPTRY(ctx, hipStreamWaitEvent(q.stream, ctx->fill_ev, 0));
    }
    if (graphs) rc = run_graph(ctx, 2 * (2 * (P.quad_max > 0) + k) + 1, q, P, D, true);
    else rc = enqueue_finish(ctx, q, P, hc.total_px);
    if (rc) return rc;
    HIPTRY(ctx, hipEventRecord(ctx->acc_ev[k], q.stream));
    ctx->last_pipe = k;
    if (pipe_used) *pipe_used = k;
    return ILM_OK;
}

/* ======================= jobs ======================= */

/* The request's device descriptor, over its Kahan buffer d_accum (2*W*H float4: sums, then
 * compensations); the issue cursor starts at pass 0. */
static void job_fill_req(Job* j) {
    const ilm_render_params& p = j->p;
    const int64_t wh = (int64_t)p.width * p.height;
    std::memset(&j->dreq, 0, sizeof(j->dreq));
    j->dreq.scene = j->scene->d_scene;
    j->dreq.width = p.width;
    j->dreq.height = p.height;
    j->dreq.max_depth = p.max_depth;
    j->dreq.ray_bias = p.ray_bias;
    j->dreq.tonemap = p.tonemap;
    j->dreq.spp = p.spp;
    hm::render_info(j->scene->camera, p.width, p.height, j->dreq.image_width, j->dreq.pixel_size, j->dreq.left, j->dreq.top);
    j->dreq.accum = j->d_accum;
    j->dreq.comp = j->d_accum + wh;
    j->next_pass = 0;
    j->next_px = 0;
}

/* begin: the first request of a plain or batched render, whose clear also starts the render's
 * counters (k_begin). */
static int job_prepare(ilm_ctx* ctx, Job* j, bool begin) {
    const ilm_render_params& p = j->p;
    const int64_t wh = (int64_t)p.width * p.height;
    const size_t ab = 2 * wh * sizeof(float4), pb = wh * sizeof(uint32_t);
    j->pool = &ctx->bufs;
    j->d_accum = (float4*)ctx->bufs.take(ab, &j->accum_cap);
    if (!j->d_accum) {
        HIPTRY(ctx, hipMalloc((void**)&j->d_accum, ab));
        j->accum_cap = ab;
    }
    j->d_px = (uint32_t*)ctx->bufs.take(pb, &j->px_cap);
    if (!j->d_px) {
        HIPTRY(ctx, hipMalloc((void**)&j->d_px, pb));
        j->px_cap = pb;
    }
    if (begin) HIPTRY(ctx, ilm_k_begin(j->d_accum, 2 * wh, ctx->d_seg_total, ctx->d_trav, ctx->h_u64, ctx->stream));
    else HIPTRY(ctx, ilm_k_fill_zero4(j->d_accum, 2 * wh, ctx->stream));
    HIPTRY(ctx, hipEventRecord(ctx->fill_ev, ctx->stream));
    job_fill_req(j);
    return ILM_OK;
}

/* Return the request's buffers to the pool (stream order keeps a later user of the same buffer
 * behind every kernel already queued on it). */
static void job_release_device(Job* j) {
    const int dev = j->scene ? j->scene->ctx->device : 0;
    if (j->d_accum && !(j->pool && j->pool->give(j->d_accum, j->accum_cap))) dfree(dev, j->d_accum);
    if (j->d_px && !(j->pool && j->pool->give(j->d_px, j->px_cap))) dfree(dev, j->d_px);
    j->d_accum = nullptr;
    j->d_px = nullptr;
}

static bool job_has_work(const Job* j) { return j->next_pass < j->p.spp; }

/* Fill a chunk from jobs in priority order. Each job contributes at most one slice per chunk
 * (all pixels x several passes, or a pixel range of one pass), so no pixel appears twice in a
 * chunk and every pixel's passes are accumulated in pass order. */
static int64_t job_demand(const Job* j) {
    const int64_t wh = (int64_t)j->p.width * j->p.height;
    return (int64_t)(j->p.spp - j->next_pass) * wh - j->next_px;
}

/* Fair-share quotas (water filling): jobs needing less than an equal share of the chunk get
 * what they need, the others split the rest equally. */
static void fair_quotas(const std::vector<Job*>& jobs, int64_t cap, std::vector<int64_t>& quota) {
    std::vector<std::pair<int64_t, size_t>> d;
    for (size_t k = 0; k < jobs.size(); k++) {
        quota[k] = 0;
        if (job_has_work(jobs[k]) && !jobs[k]->cancel.load()) d.push_back({job_demand(jobs[k]), k});
    }
    std::sort(d.begin(), d.end());
    int64_t left = cap;
    size_t n = d.size();
    for (auto& e : d) {
        const int64_t level = left / (int64_t)std::max<size_t>(n, 1);
        const int64_t q = std::min(e.first, std::max<int64_t>(level, 1));
        quota[e.second] = q;
        left -= q;
        n--;
    }
}

/* The divisors a request's pixel walk needs on the device (tile_pixel with th rows). */
static void req_divs(DReq& R, int th) {
    const uint32_t w = (uint32_t)R.width, h = (uint32_t)R.height, t = th > 1 ? (uint32_t)th : 1u;
    R.tile_th = t;
    R.tile_full = (h / t) * (t * w);
    R.w_div = udiv_make(w);
    R.band_div = udiv_make(t * w);
    R.th_div = udiv_make(t);
}

static void chunk_reset(DChunk& c) {
    c.total_paths = 0;
    c.total_px = 0;
    c.n_work = 0;
    c.depth_steps = 0;
}

/* Samples of a pixel that are consecutive path ids, at most, by default. Camera packets of one pixel
 * (64) walk the fewest nodes; at 16 a wave's rays still share them while the triangles are large
 * against the pixels, and the later depths, whose blocks then hold survivors of four times the pixels,
 * are faster. Device time with 16 / with 64, by triangles in a 4-pixel packet: 0.07 (metal spheres)
 * 0.95, 0.2 0.99, 0.3 (11 small meshes) 0.98, 0.4 0.97, 1.1 0.96, 1.3 0.99, 1.6 1.00, 3.8 (instances)
 * 1.02, 37 1.10; a 0.4 of instances 1.01; 8 samples within 0.02 of 16, never better by more. */
#define ILM_GROUP16_MAX_TRIS 1.5
static uint32_t sample_group_max(const ilm_ctx* ctx, const Job* j) {
    if (ctx->opts.sample_group > 0) return (uint32_t)ctx->opts.sample_group;
    const double px = (double)j->p.width * j->p.height;
    return (double)j->scene->inst_tris * 4.0 <= ILM_GROUP16_MAX_TRIS * px ? 16u : 64u;
}

/* Append job j's next slice, at most lim paths, as request nreq of chunk c: all pixels x as
 * many whole passes as fit, or a pixel range of one pass. Advances j's issue cursor. */
static void add_slice(const ilm_ctx* ctx, Job* j, int64_t lim, int nreq, DChunk& c) {
    const int64_t wh = (int64_t)j->p.width * j->p.height;
    DWork w;
    std::memset(&w, 0, sizeof(w));
    w.req = nreq;
    w.pass0 = j->next_pass;
    if (j->split_npx > 0) {
        /* a range of pixel slots with all of the request's passes (lim is not binding: the
         * caller chose split_npx so that one range fills at most a chunk) */
        const int64_t npx = std::min<int64_t>(wh - j->next_px, j->split_npx);
        w.npass = j->p.spp;
        w.px0 = (uint32_t)j->next_px;
        w.npx = (uint32_t)npx;
        j->next_px += npx;
        if (j->next_px >= wh) { j->next_px = 0; j->next_pass = j->p.spp; }
    } else if (j->next_px == 0 && wh <= lim) {
        int64_t np = std::min<int64_t>(j->p.spp - j->next_pass, lim / wh);
        if (ctx->opts.chunk_passes > 0) np = std::min<int64_t>(np, ctx->opts.chunk_passes);
        w.npass = (int)np;
        w.px0 = 0;
        w.npx = (uint32_t)wh;
        j->next_pass += (int)np;
    } else {
        int64_t npx = std::min<int64_t>(wh - j->next_px, lim);
        w.npass = 1;
        w.px0 = (uint32_t)j->next_px;
        w.npx = (uint32_t)npx;
        j->next_px += npx;
        if (j->next_px >= wh) { j->next_px = 0; j->next_pass += 1; }
    }
    w.sgroup = 1;
    {
        const uint32_t sg_max = sample_group_max(ctx, j);
        while (w.sgroup * 2 <= sg_max && w.npass % (w.sgroup * 2) == 0) w.sgroup *= 2;
    }
    w.sg_log2 = (uint32_t)__builtin_ctz(w.sgroup);
    w.span_div = udiv_make(w.npx * w.sgroup);
    w.pid_base = c.total_paths;
    w.acc_base = c.total_px;
    c.total_paths += (uint32_t)((int64_t)w.npass * w.npx);
    c.total_px += w.npx;
    c.reqs[nreq] = j->dreq;
    req_divs(c.reqs[nreq], ctx->opts.tile_rows > 0 ? ctx->opts.tile_rows : 4);
    c.work[c.n_work++] = w;
    c.depth_steps = std::max(c.depth_steps, j->p.max_depth);
}

/* How many paths of one scene make a chunk that requests of other scenes don't join, while n scenes
 * have work. A chunk of one scene reads that scene's values once per wave, walks its camera rays as
 * packets over FNodes and runs to its own depth; each further chunk has last depths of its own, which
 * the two pipelines overlap for a few chunks only. Wall time, chunks by scene / one chunk, requests of
 * 0.6 M, 1.2 M, 3.1 M and 12.4 M paths each: 2 scenes 0.98, 0.86, 0.93, 0.92; 4 scenes 0.92, 0.83, 0.90,
 * 0.91; 5 scenes 0.97, 0.85, 0.91, 0.89; 6 scenes 1.06, 0.95, 1.05, 0.90; 8 scenes 1.17, 1.00, 1.02,
 * 0.89. With fair shares or a pass limit a request's slice is not all its work, and one pipeline
 * overlaps nothing: there the other scenes join until the chunk is half full. */
#define ILM_FEW_SCENES 5
static int64_t own_chunk_paths(const ilm_ctx* ctx, const std::vector<Job*>& jobs) {
    if (ctx->npipes != 2 || ctx->opts.sched_fair || ctx->opts.chunk_passes > 0) return INT64_MAX;
    const ilm_scene* seen[ILM_FEW_SCENES];
    int n = 0;
    for (const Job* j : jobs) {
        if (!job_has_work(j) || j->cancel.load() || std::find(seen, seen + n, j->scene) != seen + n) continue;
        if (n == ILM_FEW_SCENES) return (int64_t)1 << 23;
        seen[n++] = j->scene;
    }
    return (int64_t)1 << 19;
}

static void build_chunk(ilm_ctx* ctx, const std::vector<Job*>& jobs, DChunk& c, std::vector<Job*>& in_chunk) {
    chunk_reset(c);
    in_chunk.clear();
    int64_t left = ctx->cap;
    int nreq = 0;
    std::vector<int64_t> quota(jobs.size(), ctx->cap);
    if (ctx->opts.sched_fair && jobs.size() > 1) fair_quotas(jobs, ctx->cap, quota);
    /* First the requests that render the scene of the first request with work, so that a chunk
     * usually holds one scene; requests of other scenes join only a chunk that would otherwise stay
     * under half full, and short for a chunk of its own (own_chunk_paths). */
    const int64_t own = std::min<int64_t>((ctx->cap + 1) / 2, own_chunk_paths(ctx, jobs));
    const ilm_scene* s0 = nullptr;
    for (Job* j : jobs)
        if (job_has_work(j) && !j->cancel.load()) { s0 = j->scene; break; }
    for (int round = 0; round < 2; round++) {
        if (round == 1 && (int64_t)c.total_paths >= own) break;
        for (size_t jk = 0; jk < jobs.size(); jk++) {
            Job* j = jobs[jk];
            if (!job_has_work(j) || j->cancel.load()) continue;
            if ((j->scene == s0) != (round == 0)) continue;
            if (nreq >= ILM_MAX_JOBS || c.n_work >= ILM_MAX_WORK || left <= 0) break;
            const int64_t lim = std::min(left, std::max<int64_t>(quota[jk], 1));
            const uint32_t before = c.total_paths;
            add_slice(ctx, j, lim, nreq, c);
            left -= (int64_t)(c.total_paths - before);
            nreq++;
            in_chunk.push_back(j);
        }
    }
}

static int validate_params(ilm_ctx* ctx, const ilm_render_params* p) {
    if (!p) return fail(ctx, ILM_E_INVALID, "null params");
    if (p->width <= 0 || p->height <= 0 || p->spp <= 0 || p->max_depth <= 0)
        return fail(ctx, ILM_E_INVALID, "width, height, spp and max_depth must be positive");
    if (p->max_depth > ILM_MAX_DEPTH) return fail(ctx, ILM_E_INVALID, "max_depth above 256");
    if ((int64_t)p->width * p->height >= (1LL << 31)) return fail(ctx, ILM_E_INVALID, "image too large");
    if (p->tonemap < 0 || p->tonemap > ILM_TONEMAP_UNCHARTED) return fail(ctx, ILM_E_INVALID, "bad tonemap");
    if (p->first_sample < 0) return fail(ctx, ILM_E_INVALID, "negative first_sample");
    return ILM_OK;
}

/* A scene uploaded under one layout may not suit the other (ilm_tune can switch layouts after
 * the upload): a BLAS too deep for its stack, or 8-bit child boxes past the largest quantum. */
static int check_scene_stack(ilm_ctx* ctx, const ilm_scene* s) {
    const int cap = ilm_k_lds_stack() + ilm_k_ovf_stack();
    const bool q = ctx->opts.bvh_layout == ILM_BVH_QUANT8;
    if ((q ? s->stack_bound_q : s->stack_bound_fp32) > cap)
        return fail(ctx, ILM_E_UNSUPPORTED, "BVH too deep for the traversal stack");
    if (q && s->quant_max_exp > ILM_QUANT_MAX_EXP)
        return fail(ctx, ILM_E_UNSUPPORTED, "scene extent too large for 8-bit child boxes");
    return ILM_OK;
}

/* ======================= results ======================= */

/* A result of n pixels in staging memory: packed RGB sums, then pixel words (k_send), each with
 * room for n rounded up to four. */
static int64_t stage_round(int64_t n) { return (n + 3) & ~(int64_t)3; }
static size_t stage_bytes(int64_t n) { return (size_t)stage_round(n) * 16; }

static void stage_free(ilm_ctx* ctx, Staging* g) {
    if (!g) return;
    {
        std::lock_guard<std::mutex> cap(capture_mu(ctx->device));
        if (g->p) (void)hipHostFree(g->p);
    }
    for (hipEvent_t e : g->ev)
        if (e) (void)hipEventDestroy(e);
    delete g;
}
/* gives the pool's idle buffers back to the system */
static void stage_trim(ilm_ctx* ctx) {
    std::vector<Staging*> idle;
    {
        std::lock_guard<std::mutex> lk(ctx->stages.mu);
        idle.swap(ctx->stages.free);
        ctx->stages.bytes = 0;
    }
    for (Staging* g : idle) stage_free(ctx, g);
}
static hipError_t stage_alloc(ilm_ctx* ctx, void** p, size_t bytes) {
    if ((int64_t)bytes > ctx->stages.largest.load()) return hipErrorOutOfMemory;
    std::lock_guard<std::mutex> cap(capture_mu(ctx->device));
    return hipHostMalloc(p, bytes, hipHostMallocDefault);
}
/* null when the system has no pinned memory of that size, not even in place of the idle buffers */
static Staging* stage_take(ilm_ctx* ctx, size_t bytes) {
    {
        std::lock_guard<std::mutex> lk(ctx->stages.mu);
        std::vector<Staging*>& f = ctx->stages.free;
        size_t best = f.size();
        for (size_t k = 0; k < f.size(); k++)
            if (f[k]->cap >= bytes && f[k]->cap / 2 <= bytes + (1 << 20) && (best == f.size() || f[k]->cap < f[best]->cap)) best = k;
        if (best < f.size()) {
            Staging* g = f[best];
            f.erase(f.begin() + best);
            ctx->stages.bytes -= g->cap;
            return g;
        }
    }
    std::unique_ptr<Staging> g(new (std::nothrow) Staging());
    if (!g) return nullptr;
    if (stage_alloc(ctx, &g->p, bytes) != hipSuccess) {
        (void)hipGetLastError();
        stage_trim(ctx);
        if (stage_alloc(ctx, &g->p, bytes) != hipSuccess) {
            (void)hipGetLastError();
            return nullptr;
        }
    }
    g->cap = bytes;
    return g.release();
}
static void stage_give(ilm_ctx* ctx, Staging* g) {
    if (!g) return;
    {
        std::lock_guard<std::mutex> lk(ctx->stages.mu);
        if (ctx->stages.bytes + g->cap <= ctx->stages.cap) {
            ctx->stages.free.push_back(g);
            ctx->stages.bytes += g->cap;
            return;
        }
    }
    stage_free(ctx, g);
}

/* A run of one result's pixels on its way to the caller: sent to the staging buffer's bytes at
 * off by one k_send, complete once the event is. */
struct Piece {
    const float4* d_sums;
    const uint32_t* d_px;
    int64_t n;
    size_t off;
    hipEvent_t ev;          /* null: already complete */
    float* rgb;             /* the caller's arrays at the piece's first pixel; either may be null */
    ilm_pixel* px;
};
static void words_to_pixels(const uint32_t* px, ilm_pixel* out, int64_t lo, int64_t hi) {
    for (int64_t i = lo; i < hi; i++) {
        const uint32_t v = px[i];
        out[i].r = v & 255u;
        out[i].g = (v >> 8) & 255u;
        out[i].b = (v >> 16) & 255u;
    }
}
static void piece_unpack(const Staging* g, const Piece& p, int64_t lo, int64_t hi) {
    const float* rgb = (const float*)((const char*)g->p + p.off);
    const uint32_t* px = (const uint32_t*)(rgb + 3 * stage_round(p.n));
    if (p.rgb) std::memcpy(p.rgb + 3 * lo, rgb + 3 * lo, (size_t)(hi - lo) * 3 * sizeof(float));
    if (p.px) words_to_pixels(px, p.px, lo, hi);
}

/* Unpack the pieces into the caller's arrays as they arrive. The caller's memory is usually fresh,
 * so this is bound by its page faults and stores: 1920x1080 takes one thread 4.9 to 12 ms, two
 * 2.7, four 1.5, eight 1.1. Small results stay on the calling thread (a thread costs some 20 us). */
#define ILM_UNPACK_PX 16384
static int unpack_pieces(ilm_ctx* ctx, const Staging* g, const std::vector<Piece>& pieces) {
    struct Item { int piece; int64_t lo, hi; };
    std::vector<Item> items;
    for (size_t k = 0; k < pieces.size(); k++)
        for (int64_t lo = 0; lo < pieces[k].n; lo += ILM_UNPACK_PX)
            items.push_back({(int)k, lo, std::min<int64_t>(pieces[k].n, lo + ILM_UNPACK_PX)});
    std::atomic<size_t> next{0};
    std::atomic<int> bad{(int)hipSuccess};
    auto work = [&] {
        int seen = -1;
        for (size_t i; (i = next.fetch_add(1)) < items.size();) {
            const Item& it = items[i];
            if (it.piece > seen) {
                if (pieces[it.piece].ev) {
                    const hipError_t e = hipEventSynchronize(pieces[it.piece].ev);
                    if (e != hipSuccess) { bad.store((int)e); return; }
                }
                seen = it.piece;
            }
            piece_unpack(g, pieces[it.piece], it.lo, it.hi);
        }
    };
    const unsigned hw = std::thread::hardware_concurrency();
    const size_t helpers = std::min<size_t>({(size_t)7, items.size() / 2, (size_t)(hw / 2)});
    std::vector<std::thread> th;
    try {
        th.reserve(helpers);
        for (size_t k = 0; k < helpers; k++) th.emplace_back(work);
    } catch (...) {   /* no more threads: those there are, and this one, do the rest */
    }
    work();
    for (std::thread& t : th) t.join();
    const hipError_t e = (hipError_t)bad.load();
    if (e != hipSuccess) return fail(ctx, ILM_E_DEVICE, std::string("result transfer: ") + hipGetErrorString(e));
    return ILM_OK;
}

/* Results of a plain or batched call, sent and unpacked in rounds of at most ILM_STAGE_ROUND bytes
 * of staging memory. The first round is queued on the render's stream right behind it, the others
 * (large batches) on the copy stream. Where no staging memory can be had, what is left is copied
 * into pageable memory, piece by piece (a 1920x1080 call of 3.2 ms takes 11.0). */
#define ILM_STAGE_ROUND ((size_t)64 << 20)
#define ILM_PIECE_PX (1 << 18)
struct Delivery {
    std::vector<Piece> all;     /* every piece of the call */
    size_t done = 0;            /* pieces unpacked */
    std::vector<Piece> round;   /* the round in flight */
    Staging* g = nullptr;
    bool pageable = false;      /* no staging memory: the pieces from `done` on are copied */
};
static void delivery_plan(Delivery& d, Job* j, float* rgb, ilm_pixel* px) {
    if (!rgb && !px) return;
    const int64_t wh = (int64_t)j->p.width * j->p.height;
    for (int64_t p0 = 0; p0 < wh; p0 += ILM_PIECE_PX) {
        Piece p = {j->d_accum + p0, j->d_px + p0, std::min<int64_t>(wh - p0, ILM_PIECE_PX), 0, nullptr,
                   rgb ? rgb + 3 * p0 : nullptr, px ? px + p0 : nullptr};
        d.all.push_back(p);
    }
}
static int delivery_send(ilm_ctx* ctx, Delivery& d, hipStream_t s) {
    d.round.clear();
    size_t bytes = 0;
    while (d.done + d.round.size() < d.all.size() && d.round.size() < ILM_STAGE_EVENTS) {
        Piece p = d.all[d.done + d.round.size()];
        const size_t b = stage_bytes(p.n);
        if (!d.round.empty() && bytes + b > ILM_STAGE_ROUND) break;
        p.off = bytes;
        bytes += b;
        d.round.push_back(p);
    }
    if (d.round.empty()) return ILM_OK;
    if (!d.g || d.g->cap < bytes) {
        stage_give(ctx, d.g);
        d.g = stage_take(ctx, bytes);
        if (!d.g) {
            d.pageable = true;
            d.round.clear();
            return ILM_OK;
        }
    }
    for (size_t k = 0; k < d.round.size(); k++) {
        Piece& p = d.round[k];
        float* rgb = (float*)((char*)d.g->p + p.off);
        uint32_t* px = (uint32_t*)(rgb + 3 * stage_round(p.n));
        HIPTRY(ctx, ilm_k_send(p.d_sums, p.d_px, p.rgb ? rgb : nullptr, p.px ? px : nullptr, (int)p.n, s));
        if (!d.g->ev[k]) HIPTRY(ctx, hipEventCreateWithFlags(&d.g->ev[k], hipEventDisableTiming));
        HIPTRY(ctx, hipEventRecord(d.g->ev[k], s));
        p.ev = d.g->ev[k];
    }
    return ILM_OK;
}
/* Unpack the round in flight, then send and unpack the rest. */
static int delivery_finish(ilm_ctx* ctx, Delivery& d) {
    int rc = ILM_OK;
    while (!rc && !d.round.empty()) {
        rc = unpack_pieces(ctx, d.g, d.round);
        d.done += d.round.size();
        if (!rc) rc = delivery_send(ctx, d, ctx->copy_stream);
    }
    if (!rc && d.pageable) {
        std::vector<float4> sums;
        std::vector<uint32_t> px;
        for (; d.done < d.all.size(); d.done++) {
            const Piece& p = d.all[d.done];
            if (p.rgb) {
                sums.resize(p.n);
                HIPTRY(ctx, copy_sync(ctx, sums.data(), p.d_sums, p.n * sizeof(float4), hipMemcpyDeviceToHost));
                for (int64_t i = 0; i < p.n; i++) {
                    p.rgb[3 * i] = sums[i].x;
                    p.rgb[3 * i + 1] = sums[i].y;
                    p.rgb[3 * i + 2] = sums[i].z;
                }
            }
            if (p.px) {
                px.resize(p.n);
                HIPTRY(ctx, copy_sync(ctx, px.data(), p.d_px, p.n * sizeof(uint32_t), hipMemcpyDeviceToHost));
                words_to_pixels(px.data(), p.px, 0, p.n);
            }
        }
    }
    return rc;
}
/* Give the staging buffer back; nothing may still be writing to it. */
static void delivery_end(ilm_ctx* ctx, Delivery& d, bool failed) {
    if (failed) {
        (void)hipStreamSynchronize(ctx->stream);
        (void)hipStreamSynchronize(ctx->copy_stream);
    }
    stage_give(ctx, d.g);
    d.g = nullptr;
}

/* a lone request of at least this many paths is rendered as two chunks (run_jobs_sync) */
#define ILM_SPLIT_MIN_PATHS (1LL << 22)
#define ILM_SPLIT_MIN_DEPTH 24

/* Run jobs on the calling thread (plain and batched forms). On return every kernel of the renders
 * is done and dl's first round of results is on its way. */
static int run_jobs_sync(ilm_ctx* ctx, std::vector<Job*>& jobs, float* const* accum_rgb, ilm_pixel* const* out, Delivery& dl,
                         ilm_render_info* info) {
    std::lock_guard<std::mutex> dev(ctx->dev_mu);
    HIPTRY(ctx, hipSetDevice(ctx->device));
    for (Job* j : jobs) {
        int rc = job_prepare(ctx, j, j == jobs[0]);
        if (rc) return rc;
        /* pass i of the render seeds wang_hash(first_sample + i) */
        j->next_pass = 0;
    }
    /* A lone request that fits one chunk may run as two chunks of half its pixels (all passes
     * each) on the two pipelines, so that each chunk's latency-bound last launches run beside
     * the other's (lone_split). Splitting by pixels keeps a pixel's samples together in the path
     * order, which the first depth's camera packets rely on; splitting by passes would halve the
     * sample group. Each pixel's passes stay in one chunk, so the sums are unchanged. Deep
     * renders gain (960x720, 32 spp, depth 45 in a subsurface medium: +3 %); shallow ones lose
     * a little to the two chunks' full launches competing (1024x1024, 64 spp, depth 16: -1.6 %),
     * hence the default's depth test. */
    if (jobs.size() == 1 && ctx->npipes == 2 && !ctx->opts.profile && !ctx->opts.count_tests &&
        ctx->opts.chunk_passes == 0 && ctx->opts.lone_split != 1) {
        Job* j = jobs[0];
        const int64_t wh = (int64_t)j->p.width * j->p.height;
        const int64_t paths = wh * j->p.spp;
        const bool deep = ctx->opts.lone_split == 2 || j->p.max_depth >= ILM_SPLIT_MIN_DEPTH;
        if (deep && paths <= ctx->cap && paths >= ILM_SPLIT_MIN_PATHS)
            j->split_npx = (((wh + 1) / 2) + 63) & ~(int64_t)63;
    }
    ProfileSink prof;
    const hipEvent_t e0 = ctx->rend_ev[0], e1 = ctx->rend_ev[1];
    HIPTRY(ctx, hipEventRecord(e0, ctx->stream));
    if (ctx->stream2) HIPTRY(ctx, hipStreamWaitEvent(ctx->stream2, e0, 0));
    DChunk* hc = &ctx->build;
    std::vector<Job*> in_chunk;
    int chunks = 0;
    int64_t max_paths = 0;
    for (;;) {
        build_chunk(ctx, jobs, *hc, in_chunk);
        if (in_chunk.empty()) break;
        /* pass offsets: first_sample shifts every pass of the request */
        for (int w = 0; w < hc->n_work; w++) hc->work[w].pass0 += in_chunk[hc->work[w].req]->p.first_sample;
        const bool alone = chunks == 0 && std::none_of(jobs.begin(), jobs.end(), job_has_work);
        int rc = launch_chunk(ctx, *hc, in_chunk, ctx->opts.profile ? &prof : nullptr, alone);
        if (rc) return rc;
        chunks++;
        max_paths = std::max<int64_t>(max_paths, hc->total_paths);
    }
    /* the latest accumulation follows every earlier one, and each chunk's depths precede its
     * accumulation on its stream */
    if (chunks && ctx->last_pipe != 0) HIPTRY(ctx, hipStreamWaitEvent(ctx->stream, ctx->acc_ev[ctx->last_pipe], 0));
    for (size_t k = 0; k < jobs.size(); k++) {
        Job* j = jobs[k];
        const int64_t wh = (int64_t)j->p.width * j->p.height;
        /* the last one leaves the counters (the segment counter is cumulative: k_begin's value off) */
        HIPTRY(ctx, ilm_k_tonemap8(j->d_accum, j->d_px, (int)wh, j->p.spp, j->p.tonemap, ctx->d_seg_total, ctx->d_trav,
                                   k + 1 == jobs.size() ? ctx->h_u64 : nullptr, ctx->stream));
    }
    HIPTRY(ctx, hipEventRecord(e1, ctx->stream));   /* device_ms: every kernel of the render, tonemap included */
    for (size_t k = 0; k < jobs.size(); k++) delivery_plan(dl, jobs[k], accum_rgb ? accum_rgb[k] : nullptr, out ? out[k] : nullptr);
    int rc = delivery_send(ctx, dl, ctx->stream);
    if (rc) return rc;
    HIPTRY(ctx, hipEventSynchronize(e1));
    float ms = 0.0f;
    HIPTRY(ctx, hipEventElapsedTime(&ms, e0, e1));
    double ext_ms = 0.0;
    for (auto& pr : prof.ev) {
        float m = 0.0f;
        (void)hipEventElapsedTime(&m, pr.first, pr.second);
        ext_ms += m;
        (void)hipEventDestroy(pr.first);
        (void)hipEventDestroy(pr.second);
    }
    const unsigned long long segs = ctx->h_u64[0] - ctx->h_u64[3];
    if (info) {
        info->segments = segs;
        info->device_ms = ms;
        info->extend_ms = ext_ms;
        info->extend_launches = (int32_t)prof.ev.size();
        info->chunks = chunks;
        info->paths_per_chunk = max_paths;
        info->box_tests = ctx->h_u64[1];
        info->tri_tests = ctx->h_u64[2];
    }
    {
        std::lock_guard<std::mutex> lk(ctx->stat_mu);   /* dev_mu is held: never sched_mu here */
        ctx->stat_busy_ms += ms;
        ctx->stat_segments += segs;
    }
    return ILM_OK;
}

int ilm_render(ilm_ctx* ctx, ilm_scene* scene, const ilm_render_params* params, float* accum_rgb, ilm_pixel* out,
               ilm_render_info* info) {
    if (!ctx || !scene) return fail(ctx, ILM_E_INVALID, "null context or scene");
    int rc = validate_params(ctx, params);
    if (!rc) rc = check_scene_stack(ctx, scene);
    if (rc) return rc;
    Job j;
    j.scene = scene;
    j.p = *params;
    std::vector<Job*> jobs = {&j};
    if (info) std::memset(info, 0, sizeof(*info));
    Delivery dl;
    rc = run_jobs_sync(ctx, jobs, &accum_rgb, &out, dl, info);
    if (!rc) rc = delivery_finish(ctx, dl);
    delivery_end(ctx, dl, rc != ILM_OK);
    job_release_device(&j);
    return rc;
}

int ilm_render_batch(ilm_ctx* ctx, int32_t n, ilm_scene* const* scenes, const ilm_render_params* params,
                     float* const* accum_rgb, ilm_pixel* const* out, ilm_render_info* info) {
    if (!ctx || n <= 0 || !scenes || !params) return fail(ctx, ILM_E_INVALID, "bad batch arguments");
    std::vector<Job> js(n);
    std::vector<Job*> jobs(n);
    for (int i = 0; i < n; i++) {
        int rc = validate_params(ctx, &params[i]);
        if (rc) return rc;
        if (!scenes[i]) return fail(ctx, ILM_E_INVALID, "null scene in batch");
        rc = check_scene_stack(ctx, scenes[i]);
        if (rc) return rc;
        js[i].scene = scenes[i];
        js[i].p = params[i];
        jobs[i] = &js[i];
    }
    if (info) std::memset(info, 0, sizeof(*info));
    int rc = ILM_OK;
    /* requests beyond one chunk's job table run in consecutive groups */
    for (int g = 0; g < n && !rc; g += ILM_MAX_JOBS) {
        std::vector<Job*> grp(jobs.begin() + g, jobs.begin() + std::min(n, g + ILM_MAX_JOBS));
        ilm_render_info gi;
        std::memset(&gi, 0, sizeof(gi));
        Delivery dl;
        rc = run_jobs_sync(ctx, grp, accum_rgb ? accum_rgb + g : nullptr, out ? out + g : nullptr, dl, &gi);
        if (!rc) rc = delivery_finish(ctx, dl);
        delivery_end(ctx, dl, rc != ILM_OK);
        if (info) {
            info->segments += gi.segments;
            info->device_ms += gi.device_ms;
            info->extend_ms += gi.extend_ms;
            info->extend_launches += gi.extend_launches;
            info->chunks += gi.chunks;
            info->paths_per_chunk = std::max(info->paths_per_chunk, gi.paths_per_chunk);
            info->box_tests += gi.box_tests;
            info->tri_tests += gi.tri_tests;
        }
        for (Job* j : grp) job_release_device(j);
    }
    return rc;
}

/* ======================= render without allocation ======================= */

static size_t align256(size_t x) { return (x + 255) & ~(size_t)255; }

/* bytes per path of the pipeline buffers: two copies of o, d, c (float4) and rng (uint2), the
 * hit record (float4 + int) and the per-path result (float4) */
#define ILM_PATH_BYTES (2 * (3 * sizeof(float4) + sizeof(uint2)) + sizeof(float4) + sizeof(int) + sizeof(float4))
/* spill area of a scene whose stack bound exceeds the LDS stack: at most this many extend
 * workgroups (one wave each) run when the scratch array holds it */
#define ILM_NOALLOC_SPILL_BLOCKS 1024

/* The scratch array's carving for one render: fixed blocks, the spill area (spill_blocks > 0
 * when the scene needs it), Kahan sums and compensations (2*W*H float4), pixels, then path
 * state for cap paths. Returns false when it does not fit with at least 4096 paths. */
struct NoallocLayout {
    size_t off_ctl, off_chunk, off_seg, off_ovf, off_accum, off_px, off_paths;
    int spill_blocks;
    int64_t cap;
};
static bool noalloc_layout(const ilm_ctx* ctx, int64_t wh, bool spill, NoallocLayout& L) {
    size_t o = 0;
    L.off_ctl = o;    o = align256(o + sizeof(DCtl));
    L.off_chunk = o;  o = align256(o + sizeof(DChunk));
    L.off_seg = o;    o = align256(o + sizeof(float4));
    L.off_ovf = o;
    L.spill_blocks = spill ? std::min(ctx->ext_grid, ILM_NOALLOC_SPILL_BLOCKS) : 0;
    o = align256(o + (size_t)L.spill_blocks * ilm_k_ext_block() * ilm_k_ovf_stack() * sizeof(int));
    L.off_accum = o;  o = align256(o + 2 * (size_t)wh * sizeof(float4));
    L.off_px = o;     o = align256(o + (size_t)wh * sizeof(ilm_pixel));
    L.off_paths = o;
    if (o >= ILM_NOALLOC_ARRAY_BYTES) return false;
    /* 9 arrays, each rounded up to 256 B */
    const size_t room = ILM_NOALLOC_ARRAY_BYTES - o;
    if (room < 9 * 256) return false;
    int64_t cap = (int64_t)((room - 9 * 256) / ILM_PATH_BYTES);
    cap = std::min<int64_t>(cap & ~(int64_t)63, cap_of(ctx->opts));
    L.cap = cap;
    return cap >= 4096;
}

int ilm_render_noalloc(ilm_ctx* ctx, ilm_scene* scene, const ilm_render_params* params, float* accum_rgb,
                       ilm_pixel* out, ilm_render_info* info) {
    if (!ctx || !scene) return fail(ctx, ILM_E_INVALID, "null context or scene");
    int rc = validate_params(ctx, params);
    if (!rc) rc = check_scene_stack(ctx, scene);
    if (rc) return rc;
    if (!ctx->noalloc_scratch) return fail(ctx, ILM_E_DEVICE, "no scratch address for this device");
    const int64_t wh = (int64_t)params->width * params->height;
    const bool spill = scene_needs_ovf(ctx, scene);
    NoallocLayout L;
    if (!noalloc_layout(ctx, wh, spill, L))
        return fail(ctx, ILM_E_UNSUPPORTED,
                    "image too large for ilm_render_noalloc: " + std::to_string(wh) + " pixels x 56 B plus 4096 paths x " +
                        std::to_string((int)ILM_PATH_BYTES) + " B" + (spill ? " and the traversal-stack spill area" : "") +
                        " exceed the " + std::to_string((long long)ILM_NOALLOC_SCRATCH_BYTES) + "-byte scratch array");
    std::lock_guard<std::mutex> na(g_noalloc_mu[ctx->device]);
    std::lock_guard<std::mutex> dev(ctx->dev_mu);
    HIPTRY(ctx, hipSetDevice(ctx->device));
    unsigned char* base = (unsigned char*)ctx->noalloc_scratch;
    Pipe q;
    q.stream = ctx->stream;
    q.ctl = (DCtl*)(base + L.off_ctl);
    q.chunk = (DChunk*)(base + L.off_chunk);
    q.seg_total = (unsigned long long*)(base + L.off_seg);
    q.ovf = spill ? (int*)(base + L.off_ovf) : nullptr;
    q.ext_grid = spill ? L.spill_blocks : ctx->ext_grid;
    {
        unsigned char* pp = base + L.off_paths;
        auto take = [&](size_t bytes) { void* r = pp; pp += align256(bytes); return r; };
        const size_t n = (size_t)L.cap;
        for (DPaths* D : {&q.A, &q.B}) {
            D->o = (float4*)take(n * sizeof(float4));
            D->d = (float4*)take(n * sizeof(float4));
            D->c = (float4*)take(n * sizeof(float4));
            D->rng = (uint2*)take(n * sizeof(uint2));
        }
        q.hits.h = (float4*)take(n * sizeof(float4));
        q.hits.inst = (int*)take(n * sizeof(int));
        q.contrib = (float4*)take(n * sizeof(float4));
        if (pp > base + ILM_NOALLOC_ARRAY_BYTES) return fail(ctx, ILM_E_DEVICE, "scratch carving overflow");
    }
    /* the array keeps the previous call's contents: the Kahan buffer and the segment counter
     * start at zero; the control block is cleared by every chunk's first kernel */
    float4* d_accum = (float4*)(base + L.off_accum);
    ilm_pixel* d_px = (ilm_pixel*)(base + L.off_px);
    HIPTRY(ctx, ilm_k_fill_zero4(d_accum, 2 * (size_t)wh, ctx->stream));
    HIPTRY(ctx, ilm_k_fill_zero4((float4*)q.seg_total, 1, ctx->stream));
    Job j;
    j.scene = scene;
    j.p = *params;
    j.d_accum = d_accum;
    job_fill_req(&j);
    HIPTRY(ctx, hipEventRecord(ctx->na_ev[0], ctx->stream));
    int chunks = 0;
    int64_t max_paths = 0;
    for (;;) {
        /* the descriptor is built in the pinned staging slot itself (no host allocation) */
        const int slot = ctx->ring_pos++ % ILM_RING;
        HIPTRY(ctx, hipEventSynchronize(ctx->ring_ev[slot]));
        DChunk& hc = *ctx->h_chunk[slot];
        chunk_reset(hc);
        if (!job_has_work(&j)) break;
        add_slice(ctx, &j, L.cap, 0, hc);
        hc.work[0].pass0 += params->first_sample;
        if ((rc = stage_slot(ctx, slot, 1, q))) return rc;
        KParams P = base_params(ctx, q);
        P.trav_stats = nullptr;
        P.use_ovf = spill ? 1 : 0;
        P.uni_scene = 1;
        chunk_choices(ctx, hc.total_paths, scene_fits_quad(scene), P);
        if (ctx->opts.camera_packets == 0) P.packet0 = packet_pays(scene, *params, hc.work[0].sgroup, P.packet_f) ? 1 : 0;
        report_counts(ctx, P);
        rc = enqueue_pipeline(ctx, q, P, hc.depth_steps, hc.total_px, nullptr);
        if (rc) return rc;
        chunks++;
        max_paths = std::max<int64_t>(max_paths, hc.total_paths);
    }
    HIPTRY(ctx, ilm_k_tonemap(d_accum, d_px, (int)wh, params->spp, params->tonemap, ctx->stream));
    HIPTRY(ctx, hipEventRecord(ctx->na_ev[1], ctx->stream));
    /* packed RGB into the compensation half of the Kahan buffer, no longer needed */
    float* d_rgb = (float*)(d_accum + wh);
    if (accum_rgb) HIPTRY(ctx, ilm_k_sums_to_rgb(d_accum, d_rgb, (int)wh, ctx->stream));
    unsigned long long segs = 0;
    HIPTRY(ctx, hipMemcpyAsync(&segs, q.seg_total, sizeof(segs), hipMemcpyDeviceToHost, ctx->stream));
    if (accum_rgb) HIPTRY(ctx, hipMemcpyAsync(accum_rgb, d_rgb, (size_t)wh * 3 * sizeof(float), hipMemcpyDeviceToHost, ctx->stream));
    if (out) HIPTRY(ctx, hipMemcpyAsync(out, d_px, (size_t)wh * sizeof(ilm_pixel), hipMemcpyDeviceToHost, ctx->stream));
    HIPTRY(ctx, hipStreamSynchronize(ctx->stream));
    float ms = 0.0f;
    HIPTRY(ctx, hipEventElapsedTime(&ms, ctx->na_ev[0], ctx->na_ev[1]));
    if (info) {
        std::memset(info, 0, sizeof(*info));
        info->segments = segs;
        info->device_ms = ms;
        info->chunks = chunks;
        info->paths_per_chunk = max_paths;
    }
    {
        std::lock_guard<std::mutex> lk(ctx->stat_mu);
        ctx->stat_busy_ms += ms;
        ctx->stat_segments += segs;
    }
    return ILM_OK;
}

/* ======================= parity hooks ======================= */

/* quad: by the walk of short queues (quad.h); otherwise by the extend kernel of the context's options */
static int closest_hits(ilm_ctx* ctx, ilm_scene* scene, const float* rays, int32_t n, int32_t* inst, int32_t* prim, float* t,
                        bool quad) {
    if (!ctx || !scene || !rays || n < 0 || !inst || !prim || !t) return fail(ctx, ILM_E_INVALID, "bad arguments");
    if (int rc = check_scene_stack(ctx, scene)) return rc;
    if (quad && !scene_fits_quad(scene)) return fail(ctx, ILM_E_UNSUPPORTED, "BVH too deep for the walk with four lanes per ray");
    std::lock_guard<std::mutex> dev(ctx->dev_mu);
    HIPTRY(ctx, hipSetDevice(ctx->device));
    std::unique_ptr<DChunk> hc(new DChunk());
    std::memset(hc.get(), 0, sizeof(DChunk));
    hc->reqs[0].scene = scene->d_scene;
    std::vector<float4> o4, d4, h4;
    std::vector<int> hi;
    for (int64_t base = 0; base < n; base += ctx->cap) {
        int64_t m = std::min<int64_t>(ctx->cap, n - base);
        o4.resize(m);
        d4.resize(m);
        for (int64_t i = 0; i < m; i++) {
            const float* r = rays + 6 * (base + i);
            o4[i] = make_float4(r[0], r[1], r[2], 0.0f);
            d4[i] = make_float4(r[3], r[4], r[5], 0.0f);
        }
        hc->total_paths = (uint32_t)m;
        hc->depth_steps = 1;
        int rc = stage_chunk(ctx, *hc, 1, ctx_pipe(ctx));
        if (rc) return rc;
        HIPTRY(ctx, hipMemcpyAsync(ctx->A.o, o4.data(), m * sizeof(float4), hipMemcpyHostToDevice, ctx->stream));
        HIPTRY(ctx, hipMemcpyAsync(ctx->A.d, d4.data(), m * sizeof(float4), hipMemcpyHostToDevice, ctx->stream));
        KParams P = base_params(ctx);
        P.trav_stats = nullptr;
        P.use_ovf = scene_needs_ovf(ctx, scene) ? 1 : 0;
        if (quad) HIPTRY(ctx, ilm_k_extend_quad(P, 0, ctx->fin_grid, ctx->stream));
        else HIPTRY(ctx, ilm_k_extend(P, 0, ctx->ovf, ctx->ext_grid, ctx->stream));
        h4.resize(m);
        hi.resize(m);
        HIPTRY(ctx, hipMemcpyAsync(h4.data(), ctx->hits.h, m * sizeof(float4), hipMemcpyDeviceToHost, ctx->stream));
        HIPTRY(ctx, hipMemcpyAsync(hi.data(), ctx->hits.inst, m * sizeof(int), hipMemcpyDeviceToHost, ctx->stream));
        HIPTRY(ctx, hipStreamSynchronize(ctx->stream));
        for (int64_t i = 0; i < m; i++) {
            int32_t pr;
            std::memcpy(&pr, &h4[i].w, 4);
            inst[base + i] = hi[i];
            prim[base + i] = hi[i] >= 0 ? pr : -1;
            t[base + i] = hi[i] == -1 ? 3.402823466e+38f : h4[i].x;
        }
    }
    return ILM_OK;
}

int ilm_debug_closest_hit(ilm_ctx* ctx, ilm_scene* scene, const float* rays, int32_t n, int32_t* inst, int32_t* prim, float* t) {
    return closest_hits(ctx, scene, rays, n, inst, prim, t, false);
}
int ilm_debug_closest_hit_quad(ilm_ctx* ctx, ilm_scene* scene, const float* rays, int32_t n, int32_t* inst, int32_t* prim, float* t) {
    return closest_hits(ctx, scene, rays, n, inst, prim, t, true);
}

int ilm_debug_pinned_limit(ilm_ctx* ctx, int64_t bytes) {
    if (!ctx || bytes < 0) return fail(ctx, ILM_E_INVALID, "bad argument");
    ctx->stages.largest.store(bytes);
    stage_trim(ctx);
    return ILM_OK;
}

int ilm_debug_path_radiance(ilm_ctx* ctx, ilm_scene* scene, const ilm_render_params* params,
                            const uint32_t* pixel_pass, int32_t n, float* rgb, int32_t* segments) {
    if (!ctx || !scene || !pixel_pass || n < 0 || !rgb) return fail(ctx, ILM_E_INVALID, "bad arguments");
    int rc = validate_params(ctx, params);
    if (!rc) rc = check_scene_stack(ctx, scene);
    if (rc) return rc;
    std::lock_guard<std::mutex> dev(ctx->dev_mu);
    HIPTRY(ctx, hipSetDevice(ctx->device));
    if (!ctx->seg_count) HIPTRY(ctx, hipMalloc((void**)&ctx->seg_count, ctx->cap * sizeof(int)));
    uint32_t* d_list = nullptr;
    HIPTRY(ctx, hipMalloc((void**)&d_list, 2 * std::min<int64_t>(ctx->cap, n) * sizeof(uint32_t) + 8));
    std::unique_ptr<DChunk> hc(new DChunk());
    std::memset(hc.get(), 0, sizeof(DChunk));
    DReq& R = hc->reqs[0];
    R.scene = scene->d_scene;
    R.width = params->width;
    R.height = params->height;
    R.max_depth = params->max_depth;
    R.ray_bias = params->ray_bias;
    R.tonemap = params->tonemap;
    R.spp = params->spp;
    hm::render_info(scene->camera, params->width, params->height, R.image_width, R.pixel_size, R.left, R.top);
    req_divs(R, 1);
    std::vector<float4> c4;
    std::vector<int> sc;
    for (int64_t base = 0; base < n; base += ctx->cap) {
        int64_t m = std::min<int64_t>(ctx->cap, n - base);
        hc->total_paths = (uint32_t)m;
        hc->depth_steps = params->max_depth;
        rc = stage_chunk(ctx, *hc, 1, ctx_pipe(ctx));
        if (rc) break;
        if (hipMemcpyAsync(d_list, pixel_pass + 2 * base, 2 * m * sizeof(uint32_t), hipMemcpyHostToDevice, ctx->stream) != hipSuccess) {
            rc = fail(ctx, ILM_E_DEVICE, "list upload");
            break;
        }
        KParams P = base_params(ctx);
        P.trav_stats = nullptr;
        P.use_ovf = scene_needs_ovf(ctx, scene) ? 1 : 0;
        P.list = d_list;
        P.seg_count = ctx->seg_count;
        chunk_choices(ctx, (uint32_t)m, scene_fits_quad(scene), P);
        if ((rc = enqueue_depths(ctx, ctx_pipe(ctx), P, params->max_depth, nullptr))) break;
        c4.resize(m);
        sc.resize(m);
        if (hipMemcpyAsync(c4.data(), ctx->contrib, m * sizeof(float4), hipMemcpyDeviceToHost, ctx->stream) != hipSuccess ||
            hipMemcpyAsync(sc.data(), ctx->seg_count, m * sizeof(int), hipMemcpyDeviceToHost, ctx->stream) != hipSuccess ||
            hipStreamSynchronize(ctx->stream) != hipSuccess) {
            rc = fail(ctx, ILM_E_DEVICE, "readback");
            break;
        }
        for (int64_t i = 0; i < m; i++) {
            rgb[3 * (base + i)] = c4[i].x;
            rgb[3 * (base + i) + 1] = c4[i].y;
            rgb[3 * (base + i) + 2] = c4[i].z;
            if (segments) segments[base + i] = sc[i];
        }
    }
    dfree(ctx->device, d_list);
    return rc;
}

/* ======================= served form ======================= */

static void admit_select_locked(ilm_ctx* ctx, std::vector<Job*>& picked);
static void admit_prepare(ilm_ctx* ctx, std::vector<Job*>& picked);

static void latency_record_locked(ilm_ctx* ctx, double ms) {
    if (ctx->latencies.size() < ILM_LATENCY_WINDOW) {
        ctx->latencies.push_back(ms);
    } else {
        ctx->latencies[ctx->lat_next] = ms;
        ctx->lat_next = (ctx->lat_next + 1) % ILM_LATENCY_WINDOW;
    }
}

/* Ends a job the scheduler holds (finished, failed or cancelled with nothing in flight). Its
 * device buffers go back first, outside sched_mu (a hipFree, when the pool is full, waits for the
 * device); then, under sched_mu, it leaves the active set, its state changes and the scheduler's
 * reference drops. The caller holds no lock. */
static void sched_finish(ilm_ctx* ctx, Job* j, int state, double t) {
    job_release_device(j);
    std::lock_guard<std::mutex> lk(ctx->sched_mu);
    ctx->in_use -= j->bytes;
    auto it = std::find(ctx->active.begin(), ctx->active.end(), j);
    if (it != ctx->active.end()) ctx->active.erase(it);
    j->end_ms = t;
    if (state == ILM_REQ_CANCELLED) {
        ctx->stat_cancelled++;
    } else {
        latency_record_locked(ctx, t - j->submit_ms);
        ctx->stat_done++;
        j->samples_done = j->p.spp;
    }
    j->state.store(state);
    j->cv.notify_all();
    if (--j->refs == 0) { scene_release(j->scene, true); delete j; }
}

static void server_loop(ilm_ctx* ctx) {
    (void)hipSetDevice(ctx->device);
    std::unique_ptr<DChunk> hc(new DChunk());
    std::vector<Job*> in_chunk;
    /* a chunk in flight: its completion event, the jobs it finishes and the pinned slot its
     * segment count is copied into */
    struct Inflight { hipEvent_t ev; std::vector<Job*> finishing; int seg_slot; };
    std::deque<Inflight> inflight;
    for (;;) {
        std::vector<Job*> active, picked;
        {
            std::unique_lock<std::mutex> lk(ctx->sched_mu);
            ctx->sched_cv.wait(lk, [&] {
                return ctx->stop || !ctx->pending.empty() || !ctx->active.empty() || !inflight.empty();
            });
            if (ctx->stop && ctx->pending.empty() && ctx->active.empty() && inflight.empty()) break;
            admit_select_locked(ctx, picked);
        }
        /* device buffers of newly admitted jobs: dev_mu only, never inside sched_mu */
        admit_prepare(ctx, picked);
        {
            std::lock_guard<std::mutex> lk(ctx->sched_mu);
            active = ctx->active;
        }
        bool launched = false;
        {
            std::lock_guard<std::mutex> dev(ctx->dev_mu);
            std::vector<Job*> issuable;
            for (Job* j : active)
                if (job_has_work(j) && !j->cancel.load()) issuable.push_back(j);
            if (!issuable.empty() && inflight.size() < 2) {
                build_chunk(ctx, issuable, *hc, in_chunk);
                for (int w = 0; w < hc->n_work; w++) hc->work[w].pass0 += in_chunk[hc->work[w].req]->p.first_sample;
                int pk = 0;
                int rc = launch_chunk(ctx, *hc, in_chunk, nullptr, false, &pk);
                const Pipe q = ctx_pipe(ctx, pk);
                Inflight f;
                f.seg_slot = ctx->seg_ring_pos++ % ILM_RING;   /* at most two chunks in flight */
                ctx->h_seg_ring[f.seg_slot] = 0;
                (void)hipMemcpyAsync(ctx->h_seg_ring + f.seg_slot, &q.ctl->segments, sizeof(unsigned long long),
                                     hipMemcpyDeviceToHost, q.stream);
                (void)hipEventCreateWithFlags(&f.ev, hipEventDisableTiming);
                for (Job* j : in_chunk) {
                    if (!job_has_work(j)) {
                        const int64_t wh = (int64_t)j->p.width * j->p.height;
                        float* rgb = (float*)j->stage->p;
                        if (ilm_k_tonemap8(j->d_accum, j->d_px, (int)wh, j->p.spp, j->p.tonemap, nullptr, nullptr, nullptr,
                                           q.stream) != hipSuccess ||
                            ilm_k_send(j->d_accum, j->d_px, rgb, (uint32_t*)(rgb + 3 * stage_round(wh)), (int)wh, q.stream) != hipSuccess)
                            j->failed = true;
                        f.finishing.push_back(j);
                    }
                }
                (void)hipEventRecord(f.ev, q.stream);
                for (Job* j : in_chunk) j->last_ev_seq = ctx->chunk_seq;
                ctx->chunk_seq++;
                if (rc) {
                    for (Job* j : in_chunk) j->failed = true;
                }
                inflight.push_back(f);
                launched = true;
            }
        }
        /* retire finished chunks; block on the oldest when nothing new could be launched */
        while (!inflight.empty()) {
            Inflight& f = inflight.front();
            hipError_t q = launched ? hipEventQuery(f.ev) : hipEventSynchronize(f.ev);
            if (q == hipErrorNotReady) break;
            double t = now_ms(ctx);
            std::vector<Job*> done = f.finishing;
            {
                std::lock_guard<std::mutex> lk(ctx->stat_mu);
                ctx->stat_segments += ctx->h_seg_ring[f.seg_slot];
            }
            (void)hipEventDestroy(f.ev);
            inflight.pop_front();
            ctx->chunks_retired++;
            for (Job* j : done) sched_finish(ctx, j, j->failed ? ILM_REQ_FAILED : ILM_REQ_DONE, t);
            launched = false;
        }
        /* cancelled jobs: release once no chunk that used them is still in flight (stream order
         * keeps any later user of their pooled buffers behind the kernels already queued) */
        std::vector<Job*> cancelled;
        {
            std::lock_guard<std::mutex> lk(ctx->sched_mu);
            for (Job* j : ctx->active) {
                bool busy = j->last_ev_seq >= ctx->chunk_seq - (int64_t)inflight.size();
                if (j->cancel.load() && !busy) cancelled.push_back(j);
            }
        }
        for (Job* j : cancelled) sched_finish(ctx, j, ILM_REQ_CANCELLED, now_ms(ctx));
    }
}

/* Take queued jobs out of the queue while the HBM budget allows, reserving their bytes; the
 * caller holds sched_mu. Cancelled queued jobs end here. */
static void admit_select_locked(ilm_ctx* ctx, std::vector<Job*>& picked) {
    while (!ctx->pending.empty() && (int)(ctx->active.size() + picked.size()) < ILM_MAX_JOBS) {
        Job* j = ctx->pending.front();
        if (j->cancel.load()) {
            ctx->pending.pop_front();
            j->state.store(ILM_REQ_CANCELLED);
            j->end_ms = now_ms(ctx);
            ctx->stat_cancelled++;
            j->cv.notify_all();
            if (--j->refs == 0) { scene_release(j->scene, true); delete j; }
            continue;
        }
        if (ctx->in_use + j->bytes > ctx->budget && !(ctx->active.empty() && picked.empty())) break;
        ctx->pending.pop_front();
        ctx->in_use += j->bytes;
        picked.push_back(j);
    }
}

/* Allocate and clear the picked jobs' device buffers (under dev_mu), then make them active
 * (under sched_mu); the two locks are never held together. */
static void admit_prepare(ilm_ctx* ctx, std::vector<Job*>& picked) {
    for (Job* j : picked) {
        int rc;
        {
            std::lock_guard<std::mutex> dev(ctx->dev_mu);
            rc = job_prepare(ctx, j, false);
            if (rc != ILM_OK) job_release_device(j);
        }
        std::lock_guard<std::mutex> lk(ctx->sched_mu);
        if (rc != ILM_OK) {
            ctx->in_use -= j->bytes;
            j->end_ms = now_ms(ctx);
            j->state.store(ILM_REQ_FAILED);
            j->cv.notify_all();
            if (--j->refs == 0) { scene_release(j->scene, true); delete j; }
            continue;
        }
        if (ctx->stop) j->cancel.store(true);
        j->start_ms = now_ms(ctx);
        j->state.store(ILM_REQ_RUNNING);
        ctx->active.push_back(j);
    }
    picked.clear();
}

static void server_start(ilm_ctx* ctx) {
    if (ctx->server.joinable()) return;
    ctx->stop = false;
    ctx->server = std::thread(server_loop, ctx);
}

static void server_stop(ilm_ctx* ctx) {
    {
        std::lock_guard<std::mutex> lk(ctx->sched_mu);
        ctx->stop = true;
        for (Job* j : ctx->pending) j->cancel.store(true);
        for (Job* j : ctx->active) j->cancel.store(true);
    }
    ctx->sched_cv.notify_all();
    if (ctx->server.joinable()) ctx->server.join();
}

int ilm_submit(ilm_ctx* ctx, ilm_scene* scene, const ilm_render_params* params, ilm_req** out) {
    if (!ctx || !scene || !out) return fail(ctx, ILM_E_INVALID, "null argument");
    *out = nullptr;
    int rc = validate_params(ctx, params);
    if (!rc) rc = check_scene_stack(ctx, scene);
    if (rc) return rc;
    const int64_t wh = (int64_t)params->width * params->height;
    Job* j = new Job();
    j->scene = scene;
    j->p = *params;
    /* what admission charges: sums, compensations and a whole ilm_pixel, 56 B a pixel, although the
     * device holds the pixel as a 4-byte word; what fits a budget and what is refused stays as it was */
    j->bytes = wh * (2 * (int64_t)sizeof(float4) + (int64_t)sizeof(ilm_pixel));
    j->ctx = ctx;
    j->stage = stage_take(ctx, stage_bytes(wh));
    if (!j->stage) {
        delete j;
        return fail(ctx, ILM_E_NOMEM, "pinned result buffers");
    }
    {
        std::lock_guard<std::mutex> lk(ctx->sched_mu);
        int maxq = ctx->opts.max_queued > 0 ? ctx->opts.max_queued : 4096;
        if ((int)ctx->pending.size() >= maxq) {
            ctx->stat_rejected++;
            delete j;
            return fail(ctx, ILM_E_BUSY, "admission queue full");
        }
        if (j->bytes > ctx->budget) {
            ctx->stat_rejected++;
            delete j;
            return fail(ctx, ILM_E_NOMEM, "request exceeds the HBM budget");
        }
        scene->refs.fetch_add(1);
        j->refs = 2;   /* scheduler + caller handle */
        j->submit_ms = now_ms(ctx);
        j->state.store(ILM_REQ_QUEUED);
        ctx->pending.push_back(j);
        server_start(ctx);
    }
    ctx->sched_cv.notify_all();
    ilm_req* r = new ilm_req();
    r->job = j;
    r->ctx = ctx;
    ctx->refs.fetch_add(1);
    *out = r;
    return ILM_OK;
}

int ilm_poll(ilm_req* r, ilm_req_status* st) {
    if (!r || !st) return fail(nullptr, ILM_E_INVALID, "null argument");
    Job* j = r->job;
    std::lock_guard<std::mutex> lk(r->ctx->sched_mu);
    st->state = j->state.load();
    st->samples_done = j->state.load() == ILM_REQ_DONE ? j->p.spp : j->next_pass;
    st->segments = 0;
    st->submit_ms = j->submit_ms;
    st->start_ms = j->start_ms;
    st->end_ms = j->end_ms;
    return ILM_OK;
}

int ilm_wait(ilm_req* r, int32_t timeout_ms) {
    if (!r) return fail(nullptr, ILM_E_INVALID, "null request");
    Job* j = r->job;
    std::unique_lock<std::mutex> lk(r->ctx->sched_mu);
    auto done = [&] { int s = j->state.load(); return s == ILM_REQ_DONE || s == ILM_REQ_CANCELLED || s == ILM_REQ_FAILED; };
    if (timeout_ms < 0) j->cv.wait(lk, done);
    else if (!j->cv.wait_for(lk, std::chrono::milliseconds(timeout_ms), done)) return fail(r->ctx, ILM_E_TIMEOUT, "wait timed out");
    int s = j->state.load();
    if (s == ILM_REQ_CANCELLED) return fail(r->ctx, ILM_E_CANCELLED, "request cancelled");
    if (s == ILM_REQ_FAILED) return fail(r->ctx, ILM_E_DEVICE, "request failed");
    return ILM_OK;
}

int ilm_result(ilm_req* r, float* accum_rgb, ilm_pixel* out) {
    if (!r) return fail(nullptr, ILM_E_INVALID, "null request");
    Job* j = r->job;
    if (j->state.load() != ILM_REQ_DONE) return fail(r->ctx, ILM_E_STATE, "request not done");
    const int64_t wh = (int64_t)j->p.width * j->p.height;
    const std::vector<Piece> whole = {{nullptr, nullptr, wh, 0, nullptr, accum_rgb, out}};
    return unpack_pieces(r->ctx, j->stage, whole);
}

int ilm_cancel(ilm_req* r) {
    if (!r) return fail(nullptr, ILM_E_INVALID, "null request");
    r->job->cancel.store(true);
    r->ctx->sched_cv.notify_all();
    return ILM_OK;
}

void ilm_req_free(ilm_req* r) {
    if (!r) return;
    Job* j = r->job;
    ilm_ctx* ctx = r->ctx;
    bool del = false;
    {
        std::lock_guard<std::mutex> lk(ctx->sched_mu);
        j->cancel.store(true);
        del = (--j->refs == 0);
    }
    ctx->sched_cv.notify_all();
    if (del) {
        scene_release(j->scene);
        delete j;
    }
    delete r;
    ctx_unref(ctx);
}

Job::~Job() {
    if (stage) stage_give(ctx, stage);
}

/* Reads host-side counters only (no device call, so a poll never waits behind a chunk in
 * flight): segments as of the last completed chunk or render, p50/p99 over the last
 * ILM_LATENCY_WINDOW completed requests. */
int ilm_stats_get(ilm_ctx* ctx, ilm_stats* st) {
    if (!ctx || !st) return fail(ctx, ILM_E_INVALID, "null argument");
    double lat[ILM_LATENCY_WINDOW];
    size_t n = 0;
    std::lock_guard<std::mutex> lk(ctx->sched_mu);
    std::memset(st, 0, sizeof(*st));
    st->requests_done = ctx->stat_done;
    st->requests_rejected = ctx->stat_rejected;
    st->requests_cancelled = ctx->stat_cancelled;
    {
        std::lock_guard<std::mutex> sl(ctx->stat_mu);
        st->segments = ctx->stat_segments;
        st->busy_ms = ctx->stat_busy_ms;
        st->bvh_cache_hits = ctx->stat_bvh_hits;
        st->bvh_cache_misses = ctx->stat_bvh_misses;
    }
    n = ctx->latencies.size();
    std::copy(ctx->latencies.begin(), ctx->latencies.end(), lat);
    st->hbm_budget_bytes = ctx->budget;
    st->hbm_in_use_bytes = ctx->in_use;
    if (n) {
        std::sort(lat, lat + n);
        auto q = [&](double f) {
            double pos = f * (double)(n - 1);
            size_t i = (size_t)pos;
            double fr = pos - (double)i;
            return i + 1 < n ? lat[i] * (1 - fr) + lat[i + 1] * fr : lat[i];
        };
        st->p50_ms = q(0.50);
        st->p99_ms = q(0.99);
    }
    return ILM_OK;
}
