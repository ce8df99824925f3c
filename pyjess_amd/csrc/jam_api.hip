// jam_api.hip -- host side of the C ABI declared in include/jess_amd.h.
//
// A query runs as one asynchronous chain on the context's stream:
//   k_candidates<count> -> exclusive scan -> k_candidates<fill> -> k_kd*
//   -> k_join -> k_super
// followed by one copy of the counters. Buffers are sized from the previous
// query; a kernel that would overflow one skips its writes (the counters keep
// counting) and the host grows the buffer to the exact size and re-runs the
// chain, so results never depend on capacities.
#include <hip/hip_ext.h>
#include <hip/hip_runtime.h>

#include <algorithm>
#include <atomic>
#include <cmath>
#include <cstdio>
#include <cstring>
#include <map>
#include <memory>
#include <mutex>
#include <numeric>
#include <thread>
#include <string>
#include <tuple>
#include <vector>

#include "../../include/jess_amd.h"
#include "jam_common.h"
#include "jam_grad.h"
#include "jam_ingest.h"
#include "jam_kernels.h"
#include "jam_sort.h"

namespace {

thread_local std::string g_error;

int32_t fail(int32_t code, const std::string &msg)
{
    g_error = msg;
    return code;
}

#define HIP_TRY(expr)                                                                   \
    do {                                                                                \
        hipError_t _e = (expr);                                                         \
        if (_e != hipSuccess)                                                           \
            return fail(JAM_EDEVICE, std::string(#expr) + ": " + hipGetErrorString(_e)); \
    } while (0)

// A device allocation that grows (never shrinks) and frees itself; or a view
// of a part of another one, which must outlive it.
struct DBuf {
    void *ptr = nullptr;
    size_t bytes = 0;
    bool owned = true;
    DBuf() = default;
    DBuf(const DBuf &) = delete;
    DBuf &operator=(const DBuf &) = delete;
    ~DBuf() { release(); }
    void release()
    {
        if (ptr && owned) (void)hipFree(ptr);
        ptr = nullptr;
        bytes = 0;
        owned = true;
    }
    void view(void *p, size_t n)
    {
        release();
        ptr = p;
        bytes = n;
        owned = false;
    }
    hipError_t reserve(size_t n)
    {
        if (n <= bytes && ptr) return hipSuccess;
        release();
        size_t want = std::max<size_t>(n, 256);
        hipError_t e = hipMalloc(&ptr, want);
        if (e == hipSuccess) bytes = want;
        else ptr = nullptr;
        return e;
    }
    template <class T> T *as() const { return static_cast<T *>(ptr); }
};

template <class T>
hipError_t upload(DBuf &b, const std::vector<T> &v, hipStream_t s)
{
    hipError_t e = b.reserve(std::max<size_t>(1, v.size()) * sizeof(T));
    if (e != hipSuccess || v.empty()) return e;
    e = hipMemcpyAsync(b.ptr, v.data(), v.size() * sizeof(T), hipMemcpyHostToDevice, s);
    if (e != hipSuccess) return e;
    return hipStreamSynchronize(s);
}

uint32_t pack4(const char *p)
{
    return (uint32_t)(uint8_t)p[0] | ((uint32_t)(uint8_t)p[1] << 8) | ((uint32_t)(uint8_t)p[2] << 16) |
           ((uint32_t)(uint8_t)p[3] << 24);
}

}  // namespace

// ---------------------------------------------------------------------------
// device scratch of the allocation-free entry point
// ---------------------------------------------------------------------------

// jam_superpose_batch_noalloc stages its inputs and outputs here instead of in
// buffers the library allocates: one copy of the array per device, held
// until the process ends. In host code `scratch` only names the symbol; its
// address on each device comes from hipGetSymbolAddress at context creation
// (g_scratch), and only that address is ever handed to the device.
static __device__ __align__(256) unsigned char scratch[JAM_NOALLOC_SCRATCH_BYTES];

namespace {
constexpr int JAM_MAX_DEVICES = 64;
void *g_scratch[JAM_MAX_DEVICES] = {};
std::mutex g_scratch_init;                    // guards g_scratch
std::mutex g_scratch_busy[JAM_MAX_DEVICES];   // one call at a time uses a device's array
}  // namespace

// ---------------------------------------------------------------------------
// objects
// ---------------------------------------------------------------------------

struct jam_context {
    int device = 0;
    hipStream_t stream = nullptr;
    hipEvent_t ev[6] = {};
    // start/stop events around every k_join launch (one per join level), for
    // the join kernels' own duration
    hipEvent_t xev[2 * JAM_MAX_LEVELS] = {};
    bool profile = false;       // join launches carry start/stop events (xev)
    // per-query workspace
    DBuf cnt, off, list, kidx, l2k, kent, katom, bbox, sbox, kscr, kd_bucket, kd_tied, kd_count;
    DBuf p_ord, p_lvl, p_nchunk, p_n1, p_base, p_cm, p_first;
    // join: two frontiers (pair + stride entries per row), complete matches,
    // counters (rows per level, complete matches, overflow flag)
    DBuf j_pair[2], j_ent[2], d_pair, d_ent, j_count;
    int64_t front_cap = 0, done_cap = 0;
    int front_stride = 0, done_stride = 0;
    int join_grid[8] = {};          // resident workgroups of the join kernel's variants
    int kd_grid[KD_GRIDS] = {};   // resident workgroups of the kd kernels
    // side streams of the kd passes (kd_launches), beside the main stream (all
    // streams at the default priority)
    hipStream_t kd_side[KD_SIDES] = {};
    hipEvent_t kd_fast[KD_SIDES] = {}, kd_joined[KD_SIDES] = {};
    bool kd_pending = false;    // side-stream work of the last kd launch may still run
    unsigned kd_used = 0;       // bit k: the last kd launch uses side stream k
    // sort of the complete matches
    DBuf s_key[2], s_perm[2], s_pkey[2];
    // groups of level-0 rows: matches, first position; each match's group, the
    // sorted matches, the positions of large groups
    DBuf sg_count, sg_start, sg_seg[2], sg_perm, sg_list;
    DBuf s_starts;   // per template size: complete matches of at most that many atoms
    // radix-sort histograms and their scan; scan temporaries of the query
    DBuf rs_hist, rs_off;
    std::vector<std::unique_ptr<DBuf>> q_scan;
    int64_t sort_cap = 0;
    DBuf e_all;  // the events of the last query, event_layout(count, stride)
    DBuf keep_d, keep_i;  // superpositions kept between the two k_super passes (few matches)
    int64_t set_cap = 0, blk_cap = 0, sblk_cap = 0, event_cap = 0;
    int nsets_cap = 0, npairs_cap = 0;
    int event_stride = 0;
    // incremented by every query: a result's events live in e_* until the
    // next query on the context
    uint64_t query_gen = 0;
    // pinned host staging for event copies: stage_slots slots of
    // JAM_STAGE_BYTES; one copy at a time uses them
    std::mutex stage_mutex;
    void *hstage = nullptr;
    int stage_slots = 0;
    hipEvent_t stage_ev[16] = {};
    // pinned host words the device's counters are read back into
    unsigned long long *hsmall = nullptr;
    int64_t hsmall_cap = 0;
    // standalone superposition buffers
    DBuf sa, sb, srmsd, srot, sc0, sc1;
    // standalone kd order: points, per-set offsets, zero chain/resSeq words
    DBuf o_xyz, o_aoff, o_zero;
    // per-pair hit counts and digests of jam_result_pair_digests
    DBuf dig;
    // temporary buffers of jam_molecules_parse_pdb, kept for the next parse
    DBuf g_buf, g_blk, g_blkoff, g_starts, g_kind, g_textof, g_back, g_lineatom, g_atomline;
    DBuf g_err, g_firsterr;
    std::vector<std::unique_ptr<DBuf>> g_scan;
    // jam_molecules_create: two pinned halves of up_half bytes, one packed
    // while the other is on its way to the device, and the index's temporary
    // buffers; one call at a time uses them
    std::mutex up_mutex;
    void *up_stage = nullptr;
    size_t up_half = 0;
    hipEvent_t up_ev[2] = {};
    DBuf u_keys, u_starts, u_nnames, u_names, u_order, u_skey, u_sval, u_hist, u_off;
    std::vector<std::unique_ptr<DBuf>> u_scan;
};

struct jam_templates {
    jam_context *ctx = nullptr;
    int n_templates = 0, n_types = 0, stride = 1;
    DBuf atom_off, atom_type, chain, resseq, pos, weight, dist_off, dist;
    DBuf type_mode, type_name_off, type_names, type_rn_off, type_rns;
    DevTpls dev() const
    {
        DevTpls d;
        d.n_templates = n_templates;
        d.n_types = n_types;
        d.stride = stride;
        d.atom_off = atom_off.as<int>();
        d.atom_type = atom_type.as<int>();
        d.chain = chain.as<int>();
        d.resseq = resseq.as<int>();
        d.pos = pos.as<double>();
        d.weight = weight.as<double>();
        d.dist_off = dist_off.as<int>();
        d.dist = dist.as<double>();
        d.type_mode = type_mode.as<int>();
        d.type_name_off = type_name_off.as<int>();
        d.type_names = type_names.as<uint32_t>();
        d.type_rn_off = type_rn_off.as<int>();
        d.type_rns = type_rns.as<uint32_t>();
        return d;
    }
};

struct jam_molecules {
    jam_context *ctx = nullptr;
    int n_mols = 0;
    int64_t n_atoms = 0;
    int64_t n_buckets = 0;
    DBuf block;   // holds the arrays of a batch made by jam_molecules_create
    DBuf atom_off, xyz, name, resname, chain, resseq, perm, res_off, res_key, res_begin, res_end;
    // the other atom fields, kept by jam_molecules_parse_pdb for the host's copy
    bool parsed = false;
    // of the parsed texts: no byte above 0x7F; HEADER records read (text,
    // offset in it), if there were few enough to keep
    bool ascii = true, headers_known = true;
    std::vector<std::pair<int, long long>> headers;
    DBuf serial, chains, altloc, icode, occupancy, tempfactor, segid, element, charge;
    DevMols dev() const
    {
        DevMols d;
        d.n_mols = n_mols;
        d.atom_off = atom_off.as<int>();
        d.xyz = xyz.as<double>();
        d.name = name.as<uint32_t>();
        d.resname = resname.as<uint32_t>();
        d.chain = chain.as<int>();
        d.resseq = resseq.as<int>();
        d.perm = perm.as<int>();
        d.res_off = res_off.as<int>();
        d.res_key = res_key.as<uint32_t>();
        d.res_begin = res_begin.as<int>();
        d.res_end = res_end.as<int>();
        return d;
    }
};

struct jam_result {
    int n_pairs = 0;
    int stride = 1;
    // the events stay in the context's device buffers (copied out on demand)
    jam_context *ctx = nullptr;
    uint64_t gen = 0;
    int64_t n_events = 0;
    std::vector<int64_t> pair_cm;
    double ms[5] = {0, 0, 0, 0, 0};
    double expand_ms = 0.0;     // summed duration of the k_join launches
    int64_t level_partials[JAM_MAX_LEVELS] = {};   // partial matches expanded per join level
    int expand_launches = 0;
};

// ---------------------------------------------------------------------------
// superposition RMSD and its gradient on device arrays
// ---------------------------------------------------------------------------

extern "C" int32_t jam_rmsd_forward(const double *a, const double *b, const int64_t *off, int64_t n_sets,
                                    int64_t n_points, double *rmsd, double *rot9, void *stream)
{
    if (n_sets < 0 || n_points < 0) return fail(JAM_EINVAL, "invalid sizes");
    if (n_sets == 0) return JAM_OK;
    if (!off || !rmsd || (n_points > 0 && (!a || !b))) return fail(JAM_EINVAL, "NULL argument");
    const int64_t tiles = (n_sets + RG_SETS - 1) / RG_SETS;
    auto *kernel = tiles <= RG_FEW_TILES ? jam::k_rmsd_fwd<false> : jam::k_rmsd_fwd<true>;
    hipLaunchKernelGGL(kernel, dim3((unsigned)tiles), dim3(RG_SETS), 0, (hipStream_t)stream, a, b, off,
                       (long long)n_sets, (long long)n_points, rmsd, rot9);
    HIP_TRY(hipGetLastError());
    return JAM_OK;
}

extern "C" int32_t jam_rmsd_backward(const double *a, const double *b, const int64_t *off, int64_t n_sets,
                                     int64_t n_points, const double *rmsd, const double *rot9,
                                     const double *grad_rmsd, double *grad_a, double *grad_b, void *stream)
{
    if (n_sets < 0 || n_points < 0) return fail(JAM_EINVAL, "invalid sizes");
    if (n_sets == 0) return JAM_OK;
    if (!off || !rmsd || !grad_rmsd || (!grad_a && !grad_b) || (n_points > 0 && (!a || !b)))
        return fail(JAM_EINVAL, "NULL argument");
    const int64_t tiles = (n_sets + RG_SETS - 1) / RG_SETS;
    auto *kernel = tiles <= RG_FEW_TILES ? jam::k_rmsd_bwd<false> : jam::k_rmsd_bwd<true>;
    hipLaunchKernelGGL(kernel, dim3((unsigned)tiles), dim3(RG_SETS), 0, (hipStream_t)stream, a, b, off,
                       (long long)n_sets, (long long)n_points, rmsd, rot9, grad_rmsd, grad_a, grad_b);
    HIP_TRY(hipGetLastError());
    return JAM_OK;
}

// ---------------------------------------------------------------------------
// misc
// ---------------------------------------------------------------------------

extern "C" const char *jam_last_error(void) { return g_error.c_str(); }

extern "C" const char *jam_version(void) { return "pyjess-amd 0.1.0 (gfx950)"; }

static bool is_gfx950(int dev)
{
    hipDeviceProp_t p;
    if (hipGetDeviceProperties(&p, dev) != hipSuccess) return false;
    return std::strncmp(p.gcnArchName, "gfx950", 6) == 0;
}

extern "C" int32_t jam_device_available(void)
{
    int n = 0;
    if (hipGetDeviceCount(&n) != hipSuccess || n <= 0) return 0;
    for (int i = 0; i < n; i++)
        if (is_gfx950(i)) return 1;
    return 0;
}

// ---------------------------------------------------------------------------
// context
// ---------------------------------------------------------------------------

extern "C" int32_t jam_context_create(int32_t device, jam_context **out)
{
    if (!out) return fail(JAM_EINVAL, "out is NULL");
    *out = nullptr;
    int n = 0;
    hipError_t e = hipGetDeviceCount(&n);
    if (e != hipSuccess || n <= 0) return fail(JAM_EDEVICE, "no HIP device visible");
    if (device < 0 || device >= n) return fail(JAM_EINVAL, "device ordinal out of range");
    if (!is_gfx950(device)) return fail(JAM_EDEVICE, "device is not a gfx950 (MI355X) GPU");
    HIP_TRY(hipSetDevice(device));
    if (device < JAM_MAX_DEVICES) {
        // the device address of this device's scratch array, once per device
        std::lock_guard<std::mutex> g(g_scratch_init);
        if (!g_scratch[device]) {
            void *p = nullptr;
            HIP_TRY(hipGetSymbolAddress(&p, HIP_SYMBOL(scratch)));
            g_scratch[device] = p;
        }
    }
    std::unique_ptr<jam_context> c(new jam_context());
    c->device = device;
    HIP_TRY(hipStreamCreateWithFlags(&c->stream, hipStreamNonBlocking));
    for (auto &ev : c->ev) HIP_TRY(hipEventCreate(&ev));
    for (auto &ev : c->xev) HIP_TRY(hipEventCreate(&ev));
    for (int k = 0; k < KD_SIDES; k++) {
        HIP_TRY(hipStreamCreateWithFlags(&c->kd_side[k], hipStreamNonBlocking));
        HIP_TRY(hipEventCreateWithFlags(&c->kd_fast[k], hipEventDisableTiming));
        HIP_TRY(hipEventCreateWithFlags(&c->kd_joined[k], hipEventDisableTiming));
    }
    *out = c.release();
    return JAM_OK;
}

extern "C" int32_t jam_synchronize(jam_context *ctx)
{
    if (!ctx) return fail(JAM_EINVAL, "NULL context");
    HIP_TRY(hipSetDevice(ctx->device));
    HIP_TRY(hipDeviceSynchronize());
    return JAM_OK;
}

extern "C" void jam_context_free(jam_context *ctx)
{
    if (!ctx) return;
    (void)hipSetDevice(ctx->device);
    if (ctx->stream) (void)hipStreamSynchronize(ctx->stream);
    for (auto &ev : ctx->ev)
        if (ev) (void)hipEventDestroy(ev);
    for (auto &ev : ctx->xev)
        if (ev) (void)hipEventDestroy(ev);
    if (ctx->hstage) (void)hipHostFree(ctx->hstage);
    if (ctx->hsmall) (void)hipHostFree(ctx->hsmall);
    if (ctx->up_stage) (void)hipHostFree(ctx->up_stage);
    for (auto &ev : ctx->up_ev)
        if (ev) (void)hipEventDestroy(ev);
    for (auto &ev : ctx->stage_ev)
        if (ev) (void)hipEventDestroy(ev);
    for (int k = 0; k < KD_SIDES; k++) {
        if (ctx->kd_side[k]) (void)hipStreamSynchronize(ctx->kd_side[k]);
        if (ctx->kd_fast[k]) (void)hipEventDestroy(ctx->kd_fast[k]);
        if (ctx->kd_joined[k]) (void)hipEventDestroy(ctx->kd_joined[k]);
        if (ctx->kd_side[k]) (void)hipStreamDestroy(ctx->kd_side[k]);
    }
    if (ctx->stream) (void)hipStreamDestroy(ctx->stream);
    delete ctx;
}

// ---------------------------------------------------------------------------
// templates
// ---------------------------------------------------------------------------

extern "C" int32_t jam_templates_create(jam_context *ctx, const jam_template_desc *d, jam_templates **out)
{
    if (!ctx || !d || !out) return fail(JAM_EINVAL, "NULL argument");
    *out = nullptr;
    if (d->n_templates < 0) return fail(JAM_EINVAL, "negative template count");
    const int T = d->n_templates;
    const int A = T > 0 ? d->atom_off[T] : 0;
    for (int t = 0; t < T; t++) {
        int n = d->atom_off[t + 1] - d->atom_off[t];
        if (n < 0) return fail(JAM_EINVAL, "atom offsets are not increasing");
        if (n > JAM_MAX_TEMPLATE_ATOMS)
            return fail(JAM_ETOOBIG, "template " + std::to_string(t) + " has " + std::to_string(n) +
                                         " atoms, more than JAM_MAX_TEMPLATE_ATOMS");
    }
    for (int a = 0; a < A; a++) {
        int m = d->mode[a];
        if (m != 0 && m != 1 && m != 3)
            return fail(JAM_EMODE, "match mode " + std::to_string(m) +
                                       " is not implemented on the device (implemented: 0, 1, 3)");
    }
    // atom types: (mode, names, residue names in order), deduplicated
    std::map<std::tuple<int, std::vector<uint32_t>, std::vector<uint32_t>>, int> types;
    std::vector<int> atom_type(A), type_mode, type_name_off{0}, type_rn_off{0};
    std::vector<uint32_t> type_names, type_rns;
    for (int a = 0; a < A; a++) {
        std::vector<uint32_t> nm, rn;
        for (int k = d->name_off[a]; k < d->name_off[a + 1]; k++) nm.push_back(pack4(d->names + 4 * k));
        for (int k = d->resname_off[a]; k < d->resname_off[a + 1]; k++)
            rn.push_back(jam_upper4(pack4(d->resnames + 4 * k)));
        auto key = std::make_tuple(d->mode[a], nm, rn);
        auto it = types.find(key);
        if (it == types.end()) {
            int id = (int)type_mode.size();
            types.emplace(key, id);
            type_mode.push_back(d->mode[a]);
            type_names.insert(type_names.end(), nm.begin(), nm.end());
            type_name_off.push_back((int)type_names.size());
            type_rns.insert(type_rns.end(), rn.begin(), rn.end());
            type_rn_off.push_back((int)type_rns.size());
            atom_type[a] = id;
        } else {
            atom_type[a] = it->second;
        }
    }
    std::vector<int> atom_off(d->atom_off, d->atom_off + T + 1), chain(A), resseq(A), dist_off(T);
    std::vector<double> pos(d->pos, d->pos + 3 * (size_t)A), weight(d->weight, d->weight + A), dist;
    int stride = 1;
    for (int a = 0; a < A; a++) {
        chain[a] = (int)(signed char)d->chain2[a];
        resseq[a] = d->resseq[a];
    }
    // template distances: TessAtom_distance, sqrt of squared differences summed x, y, z
    for (int t = 0; t < T; t++) {
        int b = atom_off[t], n = atom_off[t + 1] - b;
        stride = std::max(stride, n);
        dist_off[t] = (int)dist.size();
        for (int i = 0; i < n; i++)
            for (int k = 0; k < n; k++) {
                double s = 0.0;
                for (int q = 0; q < 3; q++) {
                    double v = pos[3 * (b + i) + q] - pos[3 * (b + k) + q];
                    s += v * v;
                }
                dist.push_back(i == k ? 0.0 : std::sqrt(s));
            }
    }
    HIP_TRY(hipSetDevice(ctx->device));
    std::unique_ptr<jam_templates> t(new jam_templates());
    t->ctx = ctx;
    t->n_templates = T;
    t->n_types = (int)type_mode.size();
    t->stride = stride;
    hipStream_t s = ctx->stream;
    HIP_TRY(upload(t->atom_off, atom_off, s));
    HIP_TRY(upload(t->atom_type, atom_type, s));
    HIP_TRY(upload(t->chain, chain, s));
    HIP_TRY(upload(t->resseq, resseq, s));
    HIP_TRY(upload(t->pos, pos, s));
    HIP_TRY(upload(t->weight, weight, s));
    HIP_TRY(upload(t->dist_off, dist_off, s));
    HIP_TRY(upload(t->dist, dist, s));
    HIP_TRY(upload(t->type_mode, type_mode, s));
    HIP_TRY(upload(t->type_name_off, type_name_off, s));
    HIP_TRY(upload(t->type_names, type_names, s));
    HIP_TRY(upload(t->type_rn_off, type_rn_off, s));
    HIP_TRY(upload(t->type_rns, type_rns, s));
    *out = t.release();
    return JAM_OK;
}

extern "C" void jam_templates_free(jam_templates *t)
{
    if (!t) return;
    (void)hipSetDevice(t->ctx->device);
    delete t;
}

// ---------------------------------------------------------------------------
// molecules
// ---------------------------------------------------------------------------

namespace {
int32_t order_by_serial(jam_context *c, int n, size_t na, const int *atom_off, const int *serial, const int *down,
                        unsigned long long n_down, hipStream_t s, const int *&order);
int32_t residue_index(jam_context *c, jam_molecules *M, const int *order, void *perm, void *res_off, hipStream_t s,
                      int &refused);
}

// ---------------------------------------------------------------------------
// molecules from host arrays
// ---------------------------------------------------------------------------

namespace {

// a stretch of host memory and where it goes in the device block
struct UploadPart {
    size_t at;
    const void *src;
    size_t bytes;
};

// bytes [lo, hi) of the image that `parts` (ascending, disjoint) make up, to dst
void pack_range(const std::vector<UploadPart> &parts, size_t lo, size_t hi, char *dst)
{
    auto it = std::upper_bound(parts.begin(), parts.end(), lo, [](size_t x, const UploadPart &p) { return x < p.at; });
    if (it != parts.begin()) --it;
    for (; it != parts.end() && it->at < hi; ++it) {
        const size_t a = std::max(lo, it->at), b = std::min(hi, it->at + it->bytes);
        if (a < b) std::memcpy(dst + (a - lo), (const char *)it->src + (a - it->at), b - a);
    }
}

// The same by up to 8 host threads, each at least 1 MB of it.
void pack_range_mt(const std::vector<UploadPart> &parts, size_t lo, size_t hi, char *dst)
{
    const size_t nt = std::min<size_t>(8, (hi - lo) >> 20);
    std::vector<std::thread> th;
    size_t done = lo;
    if (nt > 1) {
        const size_t per = ((hi - lo) / nt) & ~(size_t)63;
        try {
            th.reserve(nt);
            for (size_t k = 0; k + 1 < nt; k++, done += per)
                th.emplace_back([&parts, done, per, lo, dst] { pack_range(parts, done, done + per, dst + (done - lo)); });
        } catch (...) {
            // no more threads: the rest is done here
        }
    }
    pack_range(parts, done, hi, dst + (done - lo));
    for (auto &x : th) x.join();
}

constexpr size_t UP_HALF_MAX = size_t(16) << 20;

// Sends the image of `bytes` bytes to dev on stream s through the pinned
// halves (the caller holds up_mutex). Pinned halves because a copy from
// pageable memory moves at 10 GB/s here, a pinned one at 50, and its packing
// runs beside the transfer before it.
int32_t upload_parts(jam_context *c, const std::vector<UploadPart> &parts, size_t bytes, char *dev, hipStream_t s)
{
    const size_t want = std::min(UP_HALF_MAX, std::max<size_t>(bytes, size_t(1) << 18));
    if (want > c->up_half) {
        if (c->up_stage) HIP_TRY(hipHostFree(c->up_stage));
        c->up_stage = nullptr;
        c->up_half = 0;
        HIP_TRY(hipHostMalloc(&c->up_stage, 2 * want, hipHostMallocDefault));
        c->up_half = want;
    }
    for (auto &ev : c->up_ev)
        if (!ev) HIP_TRY(hipEventCreateWithFlags(&ev, hipEventDisableTiming));
    size_t k = 0;
    for (size_t lo = 0; lo < bytes; lo += c->up_half, k++) {
        const size_t hi = std::min(bytes, lo + c->up_half);
        char *h = (char *)c->up_stage + (k & 1) * c->up_half;
        if (k >= 2) HIP_TRY(hipEventSynchronize(c->up_ev[k & 1]));
        pack_range_mt(parts, lo, hi, h);
        HIP_TRY(hipMemcpyAsync(dev + lo, h, hi - lo, hipMemcpyHostToDevice, s));
        HIP_TRY(hipEventRecord(c->up_ev[k & 1], s));
    }
    return JAM_OK;
}

// The residue-name index of a batch on the host, for molecules with more
// names than the device kernel holds (ResIndex_create,
// patches/ResIndex.c.patch:34-119): atoms grouped by case-insensitive residue
// name, each group by serial, ties in input order, groups by key value.
int32_t host_residue_index(const jam_molecule_desc *mols, int32_t n, jam_molecules *M, hipStream_t s)
{
    std::vector<int> perm, res_off{0}, res_begin, res_end;
    std::vector<uint32_t> res_key;
    for (int m = 0; m < n; m++) {
        const jam_molecule_desc &D = mols[m];
        const int N = D.n_atoms;
        std::vector<uint32_t> upkey(N);
        for (int i = 0; i < N; i++) upkey[i] = jam_upper4(pack4(D.resnames + 4 * (size_t)i));
        std::vector<int> p(N);
        std::iota(p.begin(), p.end(), 0);
        std::stable_sort(p.begin(), p.end(), [&](int a, int b) {
            if (upkey[a] != upkey[b]) return upkey[a] < upkey[b];
            return D.serial[a] < D.serial[b];
        });
        perm.insert(perm.end(), p.begin(), p.end());
        for (int i = 0; i < N; i++) {
            if (i == 0 || upkey[p[i]] != upkey[p[i - 1]]) {
                if (i > 0) res_end.push_back(i);
                res_key.push_back(upkey[p[i]]);
                res_begin.push_back(i);
            }
        }
        if (N > 0) res_end.push_back(N);
        res_off.push_back((int)res_key.size());
    }
    HIP_TRY(upload(M->perm, perm, s));
    HIP_TRY(upload(M->res_off, res_off, s));
    HIP_TRY(upload(M->res_key, res_key, s));
    HIP_TRY(upload(M->res_begin, res_begin, s));
    HIP_TRY(upload(M->res_end, res_end, s));
    M->n_buckets = (int64_t)res_key.size();
    return JAM_OK;
}

// serial numbers that never descend
bool ascending(const int32_t *v, int n)
{
    int down = 0;
    for (int i = 1; i < n; i++) down |= v[i] < v[i - 1];
    return down == 0;
}

constexpr size_t HOST_SORT_ATOMS = 4096;

int32_t create_molecules(jam_context *ctx, const jam_molecule_desc *mols, int32_t n, jam_molecules **out)
{
    std::vector<int> atom_off(1, 0);
    atom_off.reserve((size_t)n + 1);
    for (int m = 0; m < n; m++) {
        if (mols[m].n_atoms < 0) return fail(JAM_EINVAL, "negative atom count");
        if ((int64_t)atom_off.back() + mols[m].n_atoms > INT32_MAX)
            return fail(JAM_ETOOBIG, "too many atoms in one batch");
        atom_off.push_back(atom_off.back() + mols[m].n_atoms);
    }
    const size_t na = (size_t)atom_off.back();
    // atoms at which serial numbers descend (five columns of a PDB text wrap
    // after 99,999 atoms), one more than k_run_order takes at the most
    std::vector<int> down;
    for (int m = 0; m < n && down.size() <= ING_RUNS; m++) {
        const int32_t *sr = mols[m].serial;
        if (ascending(sr, mols[m].n_atoms)) continue;
        for (int i = 1; i < mols[m].n_atoms && down.size() <= ING_RUNS; i++)
            if (sr[i] < sr[i - 1]) down.push_back(atom_off[m] + i);
    }
    // descending at many atoms of a small batch: sorted here, which takes less than
    // the launches of a sort on the device (2,000 atoms: 0.06 against 0.11 ms;
    // 90,000 atoms: 4.5 against 0.1 ms)
    std::vector<int> sorted;
    if (down.size() > ING_RUNS && na <= HOST_SORT_ATOMS) {
        sorted.resize(na);
        for (int m = 0; m < n; m++) {
            const auto from = sorted.begin() + atom_off[m], to = sorted.begin() + atom_off[m + 1];
            std::iota(from, to, 0);
            const int32_t *sr = mols[m].serial;
            std::stable_sort(from, to, [sr](int a, int b) { return sr[a] < sr[b]; });
        }
    }
    HIP_TRY(hipSetDevice(ctx->device));
    std::lock_guard<std::mutex> guard(ctx->up_mutex);
    std::unique_ptr<jam_molecules> M(new jam_molecules());
    M->ctx = ctx;
    M->n_mols = n;
    M->n_atoms = (int64_t)na;
    hipStream_t s = ctx->stream;
    // one block: the uploaded arrays first, as one image, then those made on
    // the device
    size_t bytes = 0;
    auto place = [&](size_t b) {
        const size_t at = bytes;
        bytes += (std::max<size_t>(b, 1) + 255) & ~(size_t)255;
        return at;
    };
    const size_t o_off = place(sizeof(int) * ((size_t)n + 1)), o_xyz = place(sizeof(double) * 3 * na);
    const size_t o_name = place(4 * na), o_resname = place(4 * na), o_resseq = place(sizeof(int) * na);
    const size_t o_chain8 = place(na), o_serial = down.empty() ? bytes : place(sizeof(int) * na);
    const size_t o_down = down.empty() ? bytes : place(sizeof(int) * down.size());
    const size_t image = bytes;
    const size_t o_chain = place(sizeof(int) * na), o_perm = place(sizeof(int) * na);
    const size_t o_resoff = place(sizeof(int) * ((size_t)n + 1));
    HIP_TRY(M->block.reserve(bytes));
    char *base = M->block.as<char>();
    M->atom_off.view(base + o_off, sizeof(int) * ((size_t)n + 1));
    M->xyz.view(base + o_xyz, sizeof(double) * 3 * na);
    M->name.view(base + o_name, 4 * na);
    M->resname.view(base + o_resname, 4 * na);
    M->resseq.view(base + o_resseq, sizeof(int) * na);
    M->chain.view(base + o_chain, sizeof(int) * na);
    std::vector<UploadPart> parts;
    parts.reserve(6 * (size_t)n + 3);
    parts.push_back({o_off, atom_off.data(), sizeof(int) * ((size_t)n + 1)});
    auto add = [&](size_t at, size_t width, auto src) {
        for (int m = 0; m < n; m++)
            if (mols[m].n_atoms > 0)
                parts.push_back({at + width * (size_t)atom_off[m], src(mols[m]), width * (size_t)mols[m].n_atoms});
    };
    add(o_xyz, sizeof(double) * 3, [](const jam_molecule_desc &d) { return (const void *)d.xyz; });
    add(o_name, 4, [](const jam_molecule_desc &d) { return (const void *)d.names; });
    add(o_resname, 4, [](const jam_molecule_desc &d) { return (const void *)d.resnames; });
    add(o_resseq, sizeof(int), [](const jam_molecule_desc &d) { return (const void *)d.resseq; });
    add(o_chain8, 1, [](const jam_molecule_desc &d) { return (const void *)d.chain2; });
    if (!sorted.empty()) {
        parts.push_back({o_serial, sorted.data(), sizeof(int) * na});
    } else if (!down.empty()) {
        add(o_serial, sizeof(int), [](const jam_molecule_desc &d) { return (const void *)d.serial; });
        parts.push_back({o_down, down.data(), sizeof(int) * down.size()});
    }
    int32_t rc = upload_parts(ctx, parts, image, base, s);
    int refused = 0;   // a batch without molecules has nothing to launch
    if (rc == JAM_OK && n > 0) {
        if (na > 0)
            hipLaunchKernelGGL(jam::k_chain_words, dim3((unsigned)((na + ING_THREADS - 1) / ING_THREADS)),
                               dim3(ING_THREADS), 0, s, (const signed char *)(base + o_chain8), (long long)na,
                               M->chain.as<int>());
        const int *order = (const int *)(base + o_serial);   // where it was sorted here
        if (sorted.empty())
            rc = order_by_serial(ctx, n, na, M->atom_off.as<const int>(), (const int *)(base + o_serial),
                                 (const int *)(base + o_down), down.size(), s, order);
        if (rc == JAM_OK) rc = residue_index(ctx, M.get(), order, base + o_perm, base + o_resoff, s, refused);
    }
    if (rc == JAM_OK && refused >= 0) rc = host_residue_index(mols, n, M.get(), s);
    // the pinned halves are free again, and so is the memory of a batch that
    // is given up, only once its transfers are over
    const hipError_t e = hipStreamSynchronize(s);
    if (rc != JAM_OK) return rc;
    HIP_TRY(e);
    *out = M.release();
    return JAM_OK;
}

}  // namespace

extern "C" int32_t jam_molecules_create(jam_context *ctx, const jam_molecule_desc *mols, int32_t n,
                                        jam_molecules **out)
{
    if (!ctx || !out || (n > 0 && !mols)) return fail(JAM_EINVAL, "NULL argument");
    if (n < 0) return fail(JAM_EINVAL, "negative molecule count");
    *out = nullptr;
    try {
        return create_molecules(ctx, mols, n, out);
    } catch (const std::bad_alloc &) {
        return fail(JAM_ENOMEM, "out of host memory");
    }
}

extern "C" void jam_molecules_free(jam_molecules *m)
{
    if (!m) return;
    (void)hipSetDevice(m->ctx->device);
    delete m;
}

// ---------------------------------------------------------------------------
// copies to the host
// ---------------------------------------------------------------------------

namespace {

// Copies to the caller's memory go through pinned slots of JAM_STAGE_BYTES, two per host thread:
// a thread unpacks one while the other is on its way from the device. 4 MB:
// about 80 us of transfer, well above what issuing one takes, and small enough
// that 64 MB keep eight threads unpacking while they arrive (two
// halves of 64 MB had the unpacking of most copies wait for the whole
// transfer).
constexpr size_t JAM_STAGE_BYTES = size_t(4) << 20;
constexpr int JAM_STAGE_THREADS = 8;

struct CopyPiece {
    void *dst;
    const char *src;
    size_t bytes;
};

// a field of `bytes` bytes at `src` for `dst` (may be NULL), cut into pieces of
// at most one slot
void add_pieces(std::vector<CopyPiece> &pieces, void *dst, const char *src, size_t bytes)
{
    if (!dst) return;
    for (size_t o = 0; o < bytes; o += JAM_STAGE_BYTES)
        pieces.push_back({(char *)dst + o, src + o, std::min(JAM_STAGE_BYTES, bytes - o)});
}

// pinned slots and their events, grown to `n` slots
int32_t grow_stage(jam_context *c, int n)
{
    if (n <= c->stage_slots) return JAM_OK;
    if (c->hstage) HIP_TRY(hipHostFree(c->hstage));
    c->hstage = nullptr;
    c->stage_slots = 0;
    for (int k = 0; k < n; k++)
        if (!c->stage_ev[k]) HIP_TRY(hipEventCreateWithFlags(&c->stage_ev[k], hipEventDisableTiming));
    HIP_TRY(hipHostMalloc(&c->hstage, JAM_STAGE_BYTES * (size_t)n, hipHostMallocDefault));
    c->stage_slots = n;
    return JAM_OK;
}

// Copies the pieces (device to host) through the context's pinned slots, on
// the context's stream, and waits for them.
int32_t copy_out(jam_context *c, const std::vector<CopyPiece> &pieces)
{
    hipStream_t s = c->stream;
    // batches of consecutive pieces, one slot each
    struct Batch {
        size_t first, last;
    };
    std::vector<Batch> batches;
    for (size_t i = 0; i < pieces.size();) {
        size_t used = 0, j = i;
        while (j < pieces.size() && used + pieces[j].bytes <= JAM_STAGE_BYTES) used += pieces[j++].bytes;
        batches.push_back({i, j});
        i = j;
    }
    if (batches.empty()) return JAM_OK;
    std::lock_guard<std::mutex> guard(c->stage_mutex);
    const int nt = (int)std::min<size_t>(JAM_STAGE_THREADS, (batches.size() + 1) / 2);
    int32_t rc = grow_stage(c, (int)std::min<size_t>(batches.size(), 2 * (size_t)nt));
    if (rc != JAM_OK) return rc;
    auto issue = [&](const Batch &b, int slot) -> hipError_t {
        char *h = (char *)c->hstage + (size_t)slot * JAM_STAGE_BYTES;
        size_t o = 0;
        for (size_t i = b.first; i < b.last;) {
            // one transfer for every run of pieces contiguous on the device
            size_t j = i + 1, bytes = pieces[i].bytes;
            while (j < b.last && pieces[j].src == pieces[j - 1].src + pieces[j - 1].bytes) bytes += pieces[j++].bytes;
            hipError_t e = hipMemcpyAsync(h + o, pieces[i].src, bytes, hipMemcpyDeviceToHost, s);
            if (e != hipSuccess) return e;
            o += bytes;
            i = j;
        }
        return hipEventRecord(c->stage_ev[slot], s);
    };
    // thread w takes the batches w, w + nt, ...: its k-th in slot
    // w + nt * (k & 1), issued two of its turns ahead (the first ones here, in
    // order)
    for (size_t k = 0; k < std::min<size_t>(batches.size(), 2 * (size_t)nt); k++) HIP_TRY(issue(batches[k], (int)k));
    std::atomic<int> failed{(int)hipSuccess};
    auto work = [&](size_t w) {
        hipError_t e = hipSetDevice(c->device);
        int turn = 0;
        for (size_t k = w; k < batches.size() && e == hipSuccess; k += (size_t)nt, turn ^= 1) {
            const int slot = (int)w + nt * turn;
            e = hipEventSynchronize(c->stage_ev[slot]);
            if (e != hipSuccess) break;
            const char *h = (const char *)c->hstage + (size_t)slot * JAM_STAGE_BYTES;
            size_t o = 0;
            for (size_t i = batches[k].first; i < batches[k].last; i++) {
                std::memcpy(pieces[i].dst, h + o, pieces[i].bytes);
                o += pieces[i].bytes;
            }
            if (k + 2 * (size_t)nt < batches.size()) e = issue(batches[k + 2 * (size_t)nt], slot);
        }
        if (e != hipSuccess) failed.store((int)e);
    };
    std::vector<std::thread> th;
    int started = 1;
    try {
        th.reserve((size_t)nt);
        for (; started < nt; started++) th.emplace_back(work, (size_t)started);
    } catch (...) {
        // no more threads: their batches are done here
    }
    work(0);
    for (int w = started; w < nt; w++) work((size_t)w);
    for (auto &x : th) x.join();
    HIP_TRY((hipError_t)failed.load());
    return JAM_OK;
}

}  // namespace

// ---------------------------------------------------------------------------
// PDB ingestion on the device
// ---------------------------------------------------------------------------

namespace {

constexpr int SCAN_BLOCK = 1024;
// arrays of at most this many SCAN_BLOCK-element blocks are scanned by one
// workgroup in one launch
constexpr long long SCAN_ONE_BLOCKS = 32;

// Exclusive scan of 1024-element blocks of `in` into `out`, each block's
// total into `sums` (sums in 64 bits).
template <class T, class O>
__global__ void __launch_bounds__(SCAN_BLOCK) k_scan_blocks(const T *in, long long n, O *out, long long *sums)
{
    __shared__ long long w[SCAN_BLOCK / JAM_WAVE];
    const long long i = (long long)blockIdx.x * SCAN_BLOCK + threadIdx.x;
    const long long v = i < n ? (long long)in[i] : 0;
    const int lane = jam::lane_id(), wv = threadIdx.x / JAM_WAVE;
    long long x = v;
    for (int sh = 1; sh < JAM_WAVE; sh <<= 1) {
        const long long y = __shfl_up(x, sh, JAM_WAVE);
        if (lane >= sh) x += y;
    }
    if (lane == JAM_WAVE - 1) w[wv] = x;
    __syncthreads();
    long long base = 0, total = 0;
    for (int k = 0; k < SCAN_BLOCK / JAM_WAVE; k++) {
        if (k < wv) base += w[k];
        total += w[k];
    }
    if (i < n) out[i] = (O)(base + x - v);
    if (threadIdx.x == 0) sums[blockIdx.x] = total;
}

// The whole exclusive scan in one workgroup, SCAN_BLOCK elements at a time
// with a running carry, the total into out[n]: for small arrays, where the
// launches of the multi-block scan would dominate. The largest element (at
// least 0, of 32 bits) and the total in 64 bits too, where they are asked for.
template <class T, class O>
__global__ void __launch_bounds__(SCAN_BLOCK) k_scan_one(const T *in, long long n, O *out, int *largest,
                                                        unsigned long long *total64)
{
    __shared__ long long w[SCAN_BLOCK / JAM_WAVE];
    __shared__ int top;
    int most = 0;
    if (threadIdx.x == 0) top = 0;
    const int lane = jam::lane_id(), wv = threadIdx.x / JAM_WAVE;
    long long carry = 0;
    for (long long b0 = 0; b0 < n; b0 += SCAN_BLOCK) {
        const long long i = b0 + threadIdx.x;
        const long long v = i < n ? (long long)in[i] : 0;
        long long x = v;
        for (int sh = 1; sh < JAM_WAVE; sh <<= 1) {
            const long long y = __shfl_up(x, sh, JAM_WAVE);
            if (lane >= sh) x += y;
        }
        if (lane == JAM_WAVE - 1) w[wv] = x;
        __syncthreads();
        long long base = 0, total = 0;
        for (int k = 0; k < SCAN_BLOCK / JAM_WAVE; k++) {
            if (k < wv) base += w[k];
            total += w[k];
        }
        if (i < n) out[i] = (O)(carry + base + x - v);
        carry += total;
        most = max(most, (int)v);
        __syncthreads();
    }
    if (threadIdx.x == 0) {
        out[n] = (O)carry;
        if (total64) *total64 = (unsigned long long)carry;
    }
    if (largest) {
        __syncthreads();
        atomicMax(&top, most);
        __syncthreads();
        if (threadIdx.x == 0) *largest = top;
    }
}

// Adds the blocks' offsets; the total (offs[blocks]) goes after the scan.
template <class O>
__global__ void __launch_bounds__(SCAN_BLOCK) k_scan_add(O *out, long long n, const long long *offs,
                                                        unsigned long long *total64)
{
    const long long i = (long long)blockIdx.x * SCAN_BLOCK + threadIdx.x;
    if (i < n) out[i] += (O)offs[blockIdx.x];
    if (i == 0) {
        out[n] = (O)offs[gridDim.x];
        if (total64) *total64 = (unsigned long long)offs[gridDim.x];
    }
}

__global__ void k_fill_u64(unsigned long long *v, long long n, unsigned long long x)
{
    for (long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (long long)gridDim.x * blockDim.x)
        v[i] = x;
}

__global__ void k_fill_i32(int *v, long long n, int x)
{
    for (long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (long long)gridDim.x * blockDim.x)
        v[i] = x;
}

// *out = the largest of in[0, n) (0 when n = 0): one workgroup
__global__ void __launch_bounds__(1024) k_max_i32(const int *in, long long n, int *out)
{
    __shared__ int w[1024 / JAM_WAVE];
    int m = 0;
    for (long long i = threadIdx.x; i < n; i += 1024) m = max(m, in[i]);
    for (int sh = JAM_WAVE / 2; sh >= 1; sh >>= 1) m = max(m, __shfl_xor(m, sh, JAM_WAVE));
    if (jam::lane_id() == 0) w[threadIdx.x / JAM_WAVE] = m;
    __syncthreads();
    if (threadIdx.x == 0) {
        for (int k = 1; k < 1024 / JAM_WAVE; k++) m = max(m, w[k]);
        *out = max(m, w[0]);
    }
}

// out[0, n] = exclusive scan of in[0, n) followed by the total (n + 1
// values), on stream s; temporary space from `tmp`, grown as needed. `largest`,
// `total64`: the largest element (of int arrays) and the total in 64 bits
template <class T, class O>
int32_t device_scan(const T *in, long long n, O *out, std::vector<std::unique_ptr<DBuf>> &tmp, size_t level,
                    hipStream_t s, int *largest = nullptr, unsigned long long *total64 = nullptr)
{
    const long long blocks = std::max<long long>(1, (n + SCAN_BLOCK - 1) / SCAN_BLOCK);
    if (blocks <= SCAN_ONE_BLOCKS) {
        hipLaunchKernelGGL((k_scan_one<T, O>), dim3(1), dim3(SCAN_BLOCK), 0, s, in, n, out, largest, total64);
        HIP_TRY(hipGetLastError());
        return JAM_OK;
    }
    while (tmp.size() <= level + 1) tmp.emplace_back(new DBuf());
    HIP_TRY(tmp[level]->reserve(sizeof(long long) * (size_t)(blocks + 1)));
    long long *sums = tmp[level]->as<long long>();
    hipLaunchKernelGGL((k_scan_blocks<T, O>), dim3((unsigned)blocks), dim3(SCAN_BLOCK), 0, s, in, n, out, sums);
    HIP_TRY(hipGetLastError());
    // scan of the block totals (with their total at [blocks]), added back
    HIP_TRY(tmp[level + 1]->reserve(sizeof(long long) * (size_t)(blocks + 1)));
    long long *offs = tmp[level + 1]->as<long long>();
    int32_t rc = device_scan<long long, long long>(sums, blocks, offs, tmp, level + 2, s);
    if (rc != JAM_OK) return rc;
    hipLaunchKernelGGL(k_scan_add<O>, dim3((unsigned)blocks), dim3(SCAN_BLOCK), 0, s, out, n,
                       (const long long *)offs, total64);
    if (largest) hipLaunchKernelGGL(k_max_i32, dim3(1), dim3(1024), 0, s, (const int *)in, n, largest);
    HIP_TRY(hipGetLastError());
    return JAM_OK;
}

// Stable LSD radix sort of n (key, value) pairs by bits [0, bits) of the
// keys, 8 bits per pass, between the buffer pairs (k0, v0) -- the input --
// and (k1, v1); `which` is set to the pair holding the result (0 or 1).
template <class K>
int32_t radix_sort(K *k0, int *v0, K *k1, int *v1, long long n, int bits, DBuf &hist, DBuf &offs,
                   std::vector<std::unique_ptr<DBuf>> &tmp, hipStream_t s, int &which)
{
    which = 0;
    if (n <= 1 || bits <= 0) return JAM_OK;
    if (n >= INT32_MAX) return fail(JAM_ETOOBIG, "more than 2^31 keys in one sort");
    const long long tiles = (n + RS_TILE - 1) / RS_TILE;
    HIP_TRY(hist.reserve(sizeof(int) * (size_t)(RS_THREADS * tiles)));
    HIP_TRY(offs.reserve(sizeof(int) * (size_t)(RS_THREADS * tiles + 1)));
    K *ki = k0, *ko = k1;
    int *vi = v0, *vo = v1;
    for (int shift = 0; shift < bits; shift += 8) {
        hipLaunchKernelGGL(jam::k_rs_hist<K>, dim3((unsigned)tiles), dim3(RS_THREADS), 0, s, (const K *)ki, n, shift,
                           hist.as<int>(), tiles);
        int32_t rc = device_scan<int, int>(hist.as<const int>(), RS_THREADS * tiles, offs.as<int>(), tmp, 0, s);
        if (rc != JAM_OK) return rc;
        hipLaunchKernelGGL(jam::k_rs_scatter<K>, dim3((unsigned)tiles), dim3(RS_THREADS), 0, s, (const K *)ki,
                           (const int *)vi, n, shift, offs.as<const int>(), tiles, ko, vo);
        HIP_TRY(hipGetLastError());
        std::swap(ki, ko);
        std::swap(vi, vo);
        which ^= 1;
    }
    return JAM_OK;
}

template <class T>
int32_t read_one(const T *dev, T &host, hipStream_t s)
{
    HIP_TRY(hipMemcpyAsync(&host, dev, sizeof(T), hipMemcpyDeviceToHost, s));
    HIP_TRY(hipStreamSynchronize(s));
    return JAM_OK;
}

// The order in which k_residue_index visits the atoms of n molecules (na atoms
// in all): by serial number, ties in input order; null where serial numbers do
// not descend. They descend at n_down atoms, of which down holds the first
// ING_RUNS: up to so many, each atom is ranked in every ascending run, beyond
// that all are sorted. The order is valid until the next call; the caller holds
// up_mutex.
int32_t order_by_serial(jam_context *c, int n, size_t na, const int *atom_off, const int *serial, const int *down,
                        unsigned long long n_down, hipStream_t s, const int *&order)
{
    order = nullptr;
    if (n_down == 0) return JAM_OK;
    const dim3 blocks((unsigned)((na + ING_THREADS - 1) / ING_THREADS));
    HIP_TRY(c->u_order.reserve(sizeof(int) * na));
    if (n_down <= ING_RUNS) {
        hipLaunchKernelGGL(jam::k_run_order, blocks, dim3(ING_THREADS), 0, s, atom_off, n, serial, down, (int)n_down,
                           c->u_order.as<int>());
    } else {
        HIP_TRY(c->u_skey.reserve(sizeof(unsigned long long) * 2 * na));
        HIP_TRY(c->u_sval.reserve(sizeof(int) * 2 * na));
        unsigned long long *k0 = c->u_skey.as<unsigned long long>(), *k1 = k0 + na;
        int *v0 = c->u_sval.as<int>(), *v1 = v0 + na;
        hipLaunchKernelGGL(jam::k_serial_keys, blocks, dim3(ING_THREADS), 0, s, atom_off, n, serial, k0, v0);
        int bits = 32, which = 0;
        while ((1ll << (bits - 32)) < n) bits++;
        const int32_t rc = radix_sort<unsigned long long>(k0, v0, k1, v1, (long long)na, bits, c->u_hist, c->u_off,
                                                          c->u_scan, s, which);
        if (rc != JAM_OK) return rc;
        hipLaunchKernelGGL(jam::k_sorted_order, blocks, dim3(ING_THREADS), 0, s, atom_off, n,
                           (const int *)(which ? v1 : v0), c->u_order.as<int>());
    }
    HIP_TRY(hipGetLastError());
    order = c->u_order.as<const int>();
    return JAM_OK;
}

// The residue-name index of M (atom_off and resname on the device, n_mols > 0)
// by k_residue_index, into `perm` and `res_off` (space in M's block) and arrays
// of the exact size. `refused`: a molecule with more than ING_MAX_NAMES names
// (or with a name the kernel cannot hold), -1 if there is none and the index
// is made. Synchronises, for the number of groups. The caller holds up_mutex.
int32_t residue_index(jam_context *c, jam_molecules *M, const int *order, void *perm, void *res_off, hipStream_t s,
                      int &refused)
{
    const int n = M->n_mols;
    const size_t na = (size_t)std::max<int64_t>(M->n_atoms, 1);
    M->perm.view(perm, sizeof(int) * na);
    M->res_off.view(res_off, sizeof(int) * ((size_t)n + 1));
    HIP_TRY(c->u_keys.reserve(sizeof(uint32_t) * na));
    HIP_TRY(c->u_starts.reserve(sizeof(int) * na));
    HIP_TRY(c->u_nnames.reserve(sizeof(int) * (size_t)n));
    const int *aoff = M->atom_off.as<const int>();
    const uint32_t *visited = M->resname.as<const uint32_t>();
    if (order && M->n_atoms > 0) {
        HIP_TRY(c->u_names.reserve(sizeof(uint32_t) * na));
        hipLaunchKernelGGL(jam::k_visited_names, dim3((unsigned)((na + ING_THREADS - 1) / ING_THREADS)),
                           dim3(ING_THREADS), 0, s, aoff, n, visited, order, c->u_names.as<uint32_t>());
        visited = c->u_names.as<const uint32_t>();
    }
    std::vector<int> names((size_t)n);
    int64_t total = 0;
    refused = -1;
    for (int big = 0; big < 2; big++) {
        auto *index = big ? jam::k_residue_index<ING_MAX_NAMES> : jam::k_residue_index<IDX_MAX_NAMES>;
        hipLaunchKernelGGL(index, dim3((unsigned)n), dim3(IDX_THREADS), 0, s, aoff, M->resname.as<const uint32_t>(),
                           visited, order, M->perm.as<int>(), c->u_keys.as<uint32_t>(), c->u_starts.as<int>(), c->u_nnames.as<int>());
        HIP_TRY(hipGetLastError());
        HIP_TRY(hipMemcpyAsync(names.data(), c->u_nnames.ptr, sizeof(int) * (size_t)n, hipMemcpyDeviceToHost, s));
        const int32_t rc = device_scan<int, int>(c->u_nnames.as<const int>(), n, M->res_off.as<int>(), c->u_scan, 0, s);
        HIP_TRY(hipStreamSynchronize(s));
        if (rc != JAM_OK) return rc;
        refused = -1;
        total = 0;
        for (int m = 0; m < n && refused < 0; m++) {
            if (names[m] < 0) refused = m;
            total += names[m];
        }
        if (refused < 0) break;
    }
    if (refused >= 0) return JAM_OK;
    M->n_buckets = total;
    const size_t nb = (size_t)std::max<int64_t>(total, 1);
    HIP_TRY(M->res_key.reserve(3 * sizeof(uint32_t) * nb));
    M->res_begin.view(M->res_key.as<int>() + nb, sizeof(int) * nb);
    M->res_end.view(M->res_key.as<int>() + 2 * nb, sizeof(int) * nb);
    hipLaunchKernelGGL(jam::k_index_ranges, dim3((unsigned)n), dim3(ING_THREADS), 0, s, aoff,
                       c->u_keys.as<const uint32_t>(), c->u_starts.as<const int>(), M->res_off.as<const int>(),
                       M->res_key.as<uint32_t>(), M->res_begin.as<int>(), M->res_end.as<int>());
    HIP_TRY(hipGetLastError());
    return JAM_OK;
}

}  // namespace

extern "C" int32_t jam_molecules_parse_pdb(jam_context *c, const char *const *texts, const int64_t *lengths,
                                           int32_t n, int32_t flags, jam_molecules **out)
{
    if (!c || !out || n < 0 || (n > 0 && (!texts || !lengths))) return fail(JAM_EINVAL, "invalid argument");
    *out = nullptr;
    if (flags & ~(JAM_PDB_SKIP_HETATM | JAM_PDB_IGNORE_ENDMDL)) return fail(JAM_EINVAL, "unknown flags");
    // where the texts go on the device: each one's bytes, then a line feed
    // when it does not end with one (its last line ends there)
    std::vector<long long> toff(n + 1, 0);
    for (int32_t k = 0; k < n; k++) {
        if (lengths[k] < 0 || (lengths[k] > 0 && !texts[k]))
            return fail(JAM_EINVAL, "text " + std::to_string(k) + ": negative length or NULL text");
        toff[k + 1] = toff[k] + lengths[k];
        if (lengths[k] > 0 && texts[k][lengths[k] - 1] != '\n') toff[k + 1]++;
    }
    HIP_TRY(hipSetDevice(c->device));
    hipStream_t s = c->stream;
    std::unique_ptr<jam_molecules> M(new jam_molecules());
    M->ctx = c;
    M->n_mols = n;
    M->parsed = true;
    std::vector<std::unique_ptr<DBuf>> &tmp = c->g_scan;
    // the texts, then (aligned) their offsets, through the pinned halves, which
    // are free again after the first read-back below; line feeds that are
    // missing as parts of their own
    const size_t toff_at = ((size_t)toff[n] + 255) & ~(size_t)255;
    const size_t image = toff_at + sizeof(long long) * toff.size();
    HIP_TRY(c->g_buf.reserve(image));
    std::unique_lock<std::mutex> guard(c->up_mutex);
    {
        static const char newline = '\n';
        std::vector<UploadPart> parts;
        for (int32_t k = 0; k < n; k++) {
            if (lengths[k] > 0) parts.push_back({(size_t)toff[k], texts[k], (size_t)lengths[k]});
            if (toff[k + 1] - toff[k] > lengths[k]) parts.push_back({(size_t)(toff[k + 1] - 1), &newline, 1});
        }
        parts.push_back({toff_at, toff.data(), sizeof(long long) * toff.size()});
        const int32_t up = upload_parts(c, parts, image, c->g_buf.as<char>(), s);
        if (up != JAM_OK) {
            (void)hipStreamSynchronize(s);
            return up;
        }
    }
    jam::IngText tx;
    tx.buf = c->g_buf.as<const unsigned char>();
    tx.n_bytes = toff[n];
    tx.text_off = (const long long *)(c->g_buf.as<const char>() + toff_at);
    tx.n_texts = n;
    tx.flags = flags;
    const long long per_block = (long long)ING_THREADS * ING_BPT;
    const long long byte_blocks = std::max<long long>(1, (tx.n_bytes + per_block - 1) / per_block);
    // what the host reads back, one array: the info words, the texts' ranges,
    // their first ENDMDL and mmCIF lines
    const size_t nt = (size_t)std::max(n, 1);
    const size_t w_line = ING_INFO_WORDS, w_atom = w_line + (size_t)n + 1, w_first = w_atom + (size_t)n + 1;
    const size_t words = w_first + 2 * nt;
    HIP_TRY(c->g_back.reserve(sizeof(unsigned long long) * words));
    unsigned long long *info = c->g_back.as<unsigned long long>();
    long long *text_line = (long long *)info + w_line, *text_atom = (long long *)info + w_atom;
    unsigned long long *first_endmdl = info + w_first, *first_mmcif = first_endmdl + nt;
    hipLaunchKernelGGL(k_fill_u64, dim3(1), dim3(256), 0, s, info, 2ll, 0ull);
    // ---- lines
    HIP_TRY(c->g_blk.reserve(sizeof(long long) * (size_t)byte_blocks));
    HIP_TRY(c->g_blkoff.reserve(sizeof(long long) * (size_t)(byte_blocks + 1)));
    hipLaunchKernelGGL(jam::k_ing_count, dim3((unsigned)byte_blocks), dim3(ING_THREADS), 0, s, tx,
                       c->g_blk.as<long long>(), info);
    int32_t rc;
    if ((rc = device_scan<long long>(c->g_blk.as<long long>(), byte_blocks, c->g_blkoff.as<long long>(), tmp, 0, s)) != JAM_OK)
        return rc;
    long long n_lines = 0;
    if ((rc = read_one(c->g_blkoff.as<long long>() + byte_blocks, n_lines, s)) != JAM_OK) return rc;
    guard.unlock();   // the upload is over
    if (tx.n_bytes == 0) n_lines = 0;
    const long long lines_cap = std::max<long long>(n_lines, 1);
    HIP_TRY(c->g_starts.reserve(sizeof(long long) * (size_t)lines_cap));
    if (n_lines > 0)
        hipLaunchKernelGGL(jam::k_ing_starts, dim3((unsigned)byte_blocks), dim3(ING_THREADS), 0, s, tx,
                           c->g_blkoff.as<const long long>(), c->g_starts.as<long long>());
    // ---- record kinds, first ENDMDL / mmCIF tag per text
    HIP_TRY(c->g_kind.reserve((size_t)lines_cap));
    HIP_TRY(c->g_textof.reserve(sizeof(int) * (size_t)lines_cap));
    hipLaunchKernelGGL(k_fill_u64, dim3(16), dim3(256), 0, s, first_endmdl, 2 * (long long)nt,
                       (unsigned long long)n_lines);
    const long long line_blocks = std::max<long long>(1, (n_lines + ING_THREADS - 1) / ING_THREADS);
    if (n_lines > 0)
        hipLaunchKernelGGL(jam::k_ing_classify, dim3((unsigned)line_blocks), dim3(ING_THREADS), 0, s, tx,
                           c->g_starts.as<const long long>(), n_lines, c->g_kind.as<unsigned char>(), c->g_textof.as<int>(),
                           first_endmdl, first_mmcif, info);
    // ---- atom records
    HIP_TRY(c->g_blk.reserve(sizeof(long long) * (size_t)line_blocks));
    HIP_TRY(c->g_blkoff.reserve(sizeof(long long) * (size_t)(line_blocks + 1)));
    HIP_TRY(c->g_lineatom.reserve(sizeof(long long) * (size_t)lines_cap));
    HIP_TRY(c->g_atomline.reserve(sizeof(long long) * (size_t)lines_cap));
    if (n_lines > 0) {
        hipLaunchKernelGGL(jam::k_ing_select_count, dim3((unsigned)line_blocks), dim3(ING_THREADS), 0, s, tx,
                           c->g_kind.as<const unsigned char>(), c->g_textof.as<const int>(),
                           (const unsigned long long *)first_endmdl, n_lines, c->g_blk.as<long long>());
        if ((rc = device_scan<long long>(c->g_blk.as<long long>(), line_blocks, c->g_blkoff.as<long long>(), tmp, 0, s)) !=
            JAM_OK)
            return rc;
        hipLaunchKernelGGL(jam::k_ing_select, dim3((unsigned)line_blocks), dim3(ING_THREADS), 0, s, tx,
                           c->g_kind.as<const unsigned char>(), c->g_textof.as<const int>(),
                           (const unsigned long long *)first_endmdl, n_lines, c->g_blkoff.as<const long long>(),
                           c->g_atomline.as<long long>(), c->g_lineatom.as<long long>());
    }
    hipLaunchKernelGGL(jam::k_ing_text_ranges, dim3((unsigned)((n + 1 + 63) / 64)), dim3(64), 0, s, tx,
                       c->g_starts.as<const long long>(), n_lines, c->g_lineatom.as<const long long>(),
                       c->g_blkoff.as<const long long>() + line_blocks, text_line, text_atom);
    HIP_TRY(hipGetLastError());
    std::vector<long long> back(words);
    HIP_TRY(hipMemcpyAsync(back.data(), info, sizeof(long long) * words, hipMemcpyDeviceToHost, s));
    HIP_TRY(hipStreamSynchronize(s));
    const long long *h_line = back.data() + w_line, *h_atom = back.data() + w_atom;
    const long long *h_endmdl = back.data() + w_first, *h_mmcif = h_endmdl + nt;
    // an mmCIF tag before the parse stops (PDBMoleculeParser raises)
    for (int32_t k = 0; k < n; k++) {
        if (h_mmcif[k] < n_lines && ((flags & JAM_PDB_IGNORE_ENDMDL) || h_mmcif[k] < h_endmdl[k]))
            return fail(JAM_EINVAL, "text " + std::to_string(k) + ": mmCIF data tags found, file is not in PDB format");
    }
    const long long n_atoms = h_atom[n];
    if (n_atoms >= INT32_MAX) return fail(JAM_ETOOBIG, "too many atoms in one batch");
    // HEADER records read before the parse stops, in order
    M->ascii = back[0] == 0;
    M->headers_known = back[1] <= ING_HEADERS;
    for (long long h = 0; M->headers_known && h < back[1]; h++) {
        const long long li = back[2 + 2 * h];
        const int t = (int)(std::upper_bound(toff.begin(), toff.end(), back[3 + 2 * h]) - toff.begin()) - 1;
        if ((flags & JAM_PDB_IGNORE_ENDMDL) || li < h_endmdl[t])
            M->headers.push_back({t, back[3 + 2 * h] - toff[t]});
    }
    std::sort(M->headers.begin(), M->headers.end());
    M->n_atoms = n_atoms;
    // ---- fields: one block, those that the host copies side by side
    const size_t na = (size_t)std::max<long long>(n_atoms, 1);
    size_t bytes = 0;
    auto place = [&](size_t b, size_t align) {
        bytes = (bytes + align - 1) / align * align;
        const size_t at = bytes;
        bytes += b;
        return at;
    };
    DBuf *const f8[] = {&M->xyz};
    DBuf *const f4[] = {&M->name, &M->resname, &M->resseq, &M->serial, &M->occupancy, &M->tempfactor, &M->segid, &M->charge};
    DBuf *const f2[] = {&M->chains, &M->element};
    DBuf *const f1[] = {&M->altloc, &M->icode};
    std::vector<std::tuple<DBuf *, size_t, size_t>> at_of;
    auto field = [&](DBuf *f, size_t width, size_t align) { at_of.emplace_back(f, place(width * na, align), width * na); };
    for (DBuf *f : f8) field(f, 24, 8);
    for (DBuf *f : f4) field(f, 4, 4);
    for (DBuf *f : f2) field(f, 2, 2);
    for (DBuf *f : f1) field(f, 1, 1);
    field(&M->chain, 4, 256);
    const size_t o_perm = place(4 * na, 256), o_resoff = place(sizeof(int) * ((size_t)n + 1), 256);
    const size_t o_off = place(sizeof(int) * ((size_t)n + 1), 256);
    HIP_TRY(M->block.reserve(bytes));
    char *blk = M->block.as<char>();
    for (auto &x : at_of) std::get<0>(x)->view(blk + std::get<1>(x), std::get<2>(x));
    M->atom_off.view(blk + o_off, sizeof(int) * ((size_t)n + 1));
    hipLaunchKernelGGL(jam::k_ing_narrow, dim3((unsigned)((n + 1 + 255) / 256)), dim3(256), 0, s,
                       (const long long *)text_atom, n + 1, M->atom_off.as<int>());
    HIP_TRY(c->g_err.reserve(sizeof(unsigned int) * na));
    HIP_TRY(c->g_firsterr.reserve(2 * sizeof(unsigned long long) + sizeof(int) * ING_RUNS));
    // first atom in error; atoms at which serial numbers descend, and the first of them
    unsigned long long *state = c->g_firsterr.as<unsigned long long>();
    hipLaunchKernelGGL(k_fill_u64, dim3(1), dim3(64), 0, s, state, 1ll, (unsigned long long)n_atoms);
    hipLaunchKernelGGL(k_fill_u64, dim3(1), dim3(64), 0, s, state + 1, 1ll, 0ull);
    jam::IngAtoms at;
    at.xyz = M->xyz.as<double>();
    at.name = M->name.as<uint32_t>();
    at.resname = M->resname.as<uint32_t>();
    at.chain = M->chain.as<int>();
    at.chains = M->chains.as<unsigned char>();
    at.resseq = M->resseq.as<int>();
    at.serial = M->serial.as<int>();
    at.altloc = M->altloc.as<unsigned char>();
    at.icode = M->icode.as<unsigned char>();
    at.occupancy = M->occupancy.as<float>();
    at.tempfactor = M->tempfactor.as<float>();
    at.segid = M->segid.as<uint32_t>();
    at.element = M->element.as<unsigned short>();
    at.charge = M->charge.as<int>();
    at.err = c->g_err.as<unsigned int>();
    at.first_err = state;
    const unsigned ablocks = (unsigned)((n_atoms + ING_THREADS - 1) / ING_THREADS);
    if (n_atoms > 0) {
        hipLaunchKernelGGL(jam::k_ing_parse, dim3(ablocks), dim3(ING_THREADS), 0, s, tx, c->g_starts.as<const long long>(),
                           n_lines, c->g_atomline.as<const long long>(), n_atoms, at);
        hipLaunchKernelGGL(jam::k_ing_descends, dim3(ablocks), dim3(ING_THREADS), 0, s, n_atoms, M->serial.as<const int>(),
                           c->g_atomline.as<const long long>(), c->g_textof.as<const int>(), state + 1,
                           (int *)(state + 2));
    }
    HIP_TRY(hipGetLastError());
    unsigned long long h_state[2] = {0, 0};
    HIP_TRY(hipMemcpyAsync(h_state, state, sizeof(h_state), hipMemcpyDeviceToHost, s));
    HIP_TRY(hipStreamSynchronize(s));
    if ((long long)h_state[0] < n_atoms) {
        long long li = 0;
        unsigned int kind = 0;
        HIP_TRY(hipMemcpyAsync(&li, c->g_atomline.as<long long>() + h_state[0], sizeof(li), hipMemcpyDeviceToHost, s));
        HIP_TRY(hipMemcpyAsync(&kind, c->g_err.as<unsigned int>() + h_state[0], sizeof(kind), hipMemcpyDeviceToHost, s));
        HIP_TRY(hipStreamSynchronize(s));
        int t = 0;
        while (t + 1 < n && h_line[t + 1] <= li) t++;
        return fail(JAM_EINVAL, "text " + std::to_string(t) + ", line " + std::to_string(li - h_line[t] + 1) +
                                    ": failed to parse atom (" +
                                    ((kind & ING_ENONASCII) ? "a non-ASCII character in the first 80 columns"
                                                            : "a numeric field does not parse") +
                                    ")");
    }
    // ---- residue-name index
    guard.lock();
    const int *order = nullptr;
    if ((rc = order_by_serial(c, n, na, M->atom_off.as<const int>(), M->serial.as<const int>(), (const int *)(state + 2),
                              h_state[1], s, order)) != JAM_OK)
        return rc;
    if (n > 0) {
        int refused = -1;
        if ((rc = residue_index(c, M.get(), order, blk + o_perm, blk + o_resoff, s, refused)) != JAM_OK) return rc;
        if (refused >= 0)
            return fail(JAM_ETOOBIG, "text " + std::to_string(refused) + " has more than " +
                                         std::to_string(ING_MAX_NAMES) + " distinct residue names");
    } else {
        M->perm.view(blk + o_perm, 4);
        M->res_off.view(blk + o_resoff, sizeof(int));
        HIP_TRY(M->res_key.reserve(4));
        HIP_TRY(M->res_begin.reserve(4));
        HIP_TRY(M->res_end.reserve(4));
        hipLaunchKernelGGL(k_fill_i32, dim3(1), dim3(64), 0, s, M->res_off.as<int>(), 1ll, 0);
    }
    HIP_TRY(hipStreamSynchronize(s));
    *out = M.release();
    return JAM_OK;
}

extern "C" int32_t jam_molecules_pdb_headers(const jam_molecules *m, int32_t *ascii, int32_t *known, int32_t *text,
                                             int64_t *offset, int32_t cap, int32_t *n)
{
    if (!m || !m->parsed || cap < 0 || (cap > 0 && (!text || !offset)))
        return fail(JAM_EINVAL, "not a batch of parsed molecules, or NULL argument");
    if (ascii) *ascii = m->ascii ? 1 : 0;
    if (known) *known = m->headers_known ? 1 : 0;
    if (n) *n = (int32_t)m->headers.size();
    for (size_t k = 0; k < m->headers.size() && k < (size_t)cap; k++) {
        text[k] = m->headers[k].first;
        offset[k] = m->headers[k].second;
    }
    return JAM_OK;
}

extern "C" int32_t jam_molecules_sizes(const jam_molecules *m, int64_t *atom_off, int64_t *n_buckets)
{
    if (!m) return fail(JAM_EINVAL, "NULL molecules");
    if (n_buckets) *n_buckets = m->n_buckets;
    if (atom_off) {
        std::vector<int> a((size_t)m->n_mols + 1, 0);
        if (m->n_mols > 0) {
            HIP_TRY(hipSetDevice(m->ctx->device));
            HIP_TRY(hipMemcpy(a.data(), m->atom_off.ptr, sizeof(int) * a.size(), hipMemcpyDeviceToHost));
        }
        for (size_t k = 0; k < a.size(); k++) atom_off[k] = a[k];
    }
    return JAM_OK;
}

extern "C" int32_t jam_molecules_copy_atoms(const jam_molecules *m, const jam_atom_fields *f)
{
    if (!m || !f) return fail(JAM_EINVAL, "NULL argument");
    const size_t na = (size_t)m->n_atoms;
    if (na == 0) return JAM_OK;
    const bool extra = f->serial || f->chains || f->altloc || f->icode || f->occupancy || f->tempfactor || f->segid ||
                       f->element || f->charge;
    if (extra && !m->parsed) return fail(JAM_EINVAL, "only molecules parsed on the device keep every atom field");
    HIP_TRY(hipSetDevice(m->ctx->device));
    std::vector<CopyPiece> pieces;
    auto get = [&](void *dst, const DBuf &src, size_t bytes) { add_pieces(pieces, dst, src.as<const char>(), bytes); };
    // in the order in which a parsed batch holds them
    get(f->xyz, m->xyz, sizeof(double) * 3 * na);
    get(f->names, m->name, 4 * na);
    get(f->resnames, m->resname, 4 * na);
    get(f->resseq, m->resseq, sizeof(int) * na);
    get(f->serial, m->serial, sizeof(int) * na);
    get(f->occupancy, m->occupancy, sizeof(float) * na);
    get(f->tempfactor, m->tempfactor, sizeof(float) * na);
    get(f->segid, m->segid, 4 * na);
    get(f->charge, m->charge, sizeof(int) * na);
    get(f->chains, m->chains, 2 * na);
    get(f->element, m->element, 2 * na);
    get(f->altloc, m->altloc, na);
    get(f->icode, m->icode, na);
    return copy_out(m->ctx, pieces);
}

extern "C" int32_t jam_molecules_residue_index(const jam_molecules *m, int32_t *perm, int32_t *res_off,
                                               uint32_t *res_key, int32_t *res_begin, int32_t *res_end)
{
    if (!m) return fail(JAM_EINVAL, "NULL molecules");
    HIP_TRY(hipSetDevice(m->ctx->device));
    hipStream_t s = m->ctx->stream;
    const size_t na = (size_t)m->n_atoms, nb = (size_t)m->n_buckets;
    if (perm && na) HIP_TRY(hipMemcpyAsync(perm, m->perm.ptr, sizeof(int) * na, hipMemcpyDeviceToHost, s));
    if (res_off) HIP_TRY(hipMemcpyAsync(res_off, m->res_off.ptr, sizeof(int) * ((size_t)m->n_mols + 1),
                                        hipMemcpyDeviceToHost, s));
    if (res_key && nb) HIP_TRY(hipMemcpyAsync(res_key, m->res_key.ptr, 4 * nb, hipMemcpyDeviceToHost, s));
    if (res_begin && nb) HIP_TRY(hipMemcpyAsync(res_begin, m->res_begin.ptr, 4 * nb, hipMemcpyDeviceToHost, s));
    if (res_end && nb) HIP_TRY(hipMemcpyAsync(res_end, m->res_end.ptr, 4 * nb, hipMemcpyDeviceToHost, s));
    HIP_TRY(hipStreamSynchronize(s));
    return JAM_OK;
}

// ---------------------------------------------------------------------------
// query
// ---------------------------------------------------------------------------

namespace {

int32_t grow_sets(jam_context *c, int64_t cap, int n_sets)
{
    if (n_sets > c->nsets_cap) {
        HIP_TRY(c->cnt.reserve(sizeof(int) * (size_t)n_sets));
        HIP_TRY(c->off.reserve(sizeof(int64_t) * ((size_t)n_sets + 1)));   // + the total
        HIP_TRY(c->kd_bucket.reserve(sizeof(int) * KD_TIERS * (size_t)n_sets));
        HIP_TRY(c->kd_tied.reserve(sizeof(int) * KD_TIERS * (size_t)n_sets));
        c->nsets_cap = n_sets;
    }
    const int64_t blk = cap / JAM_WAVE + n_sets + 1;
    if (cap > c->set_cap) {
        cap = std::max<int64_t>(cap, 1024);
        HIP_TRY(c->list.reserve(sizeof(int) * cap));
        HIP_TRY(c->kidx.reserve(sizeof(int) * cap));
        HIP_TRY(c->l2k.reserve(sizeof(int) * cap));
        HIP_TRY(c->kent.reserve(sizeof(SetEnt) * cap));
        HIP_TRY(c->katom.reserve(sizeof(int) * cap));
        HIP_TRY(c->kscr.reserve((size_t)KD_SCRATCH_BYTES_PER_ENTRY * cap));
        c->set_cap = cap;
    }
    // block and sub-block boxes: set s's boxes start at off[s] / size + s
    const int64_t blk_need = c->set_cap / JAM_WAVE + n_sets + 1;
    if (blk_need > c->blk_cap || blk > c->blk_cap) {
        c->blk_cap = std::max(blk, blk_need);
        HIP_TRY(c->bbox.reserve(sizeof(double) * 6 * (size_t)c->blk_cap));
    }
    const int64_t sblk_need = c->set_cap / JAM_SUB + n_sets + 1;
    if (sblk_need > c->sblk_cap) {
        c->sblk_cap = sblk_need;
        HIP_TRY(c->sbox.reserve(sizeof(double) * 6 * (size_t)c->sblk_cap));
    }
    // per tier: sets, tied sets; then an error word for jam_kd_order
    HIP_TRY(c->kd_count.reserve(sizeof(unsigned int) * (2 * KD_TIERS + 1)));
    return JAM_OK;
}

// Waits for the side-stream work of the last kd launch (before buffers it
// uses are grown, or when a query stops early).
void drain_kd(jam_context *c)
{
    if (!c->kd_pending) return;
    for (int k = 0; k < KD_SIDES; k++) (void)hipStreamSynchronize(c->kd_side[k]);
    c->kd_pending = false;
}

int32_t grow_pairs(jam_context *c, int n_pairs)
{
    if (n_pairs <= c->npairs_cap) return JAM_OK;
    HIP_TRY(c->p_ord.reserve((size_t)JAM_MAX_LEVELS * n_pairs));
    HIP_TRY(c->p_lvl.reserve(sizeof(PairLevel) * (size_t)JAM_MAX_LEVELS * n_pairs));
    HIP_TRY(c->p_nchunk.reserve(sizeof(int) * (size_t)n_pairs));
    HIP_TRY(c->p_base.reserve(sizeof(long long) * ((size_t)n_pairs + 1)));   // + the total
    // [0]: event count, [1, n_pairs]: complete matches per pair, then the kd
    // passes' error word
    HIP_TRY(c->p_cm.reserve(sizeof(long long) * ((size_t)n_pairs + 2)));
    HIP_TRY(c->p_first.reserve(sizeof(long long) * (size_t)n_pairs));
    HIP_TRY(c->p_n1.reserve(sizeof(int) * (size_t)n_pairs));
    c->npairs_cap = n_pairs;
    return JAM_OK;
}

// pinned host words for counter read-backs
int32_t grow_hsmall(jam_context *c, int64_t words)
{
    if (words <= c->hsmall_cap) return JAM_OK;
    words = std::max<int64_t>(words, 1024);
    if (c->hsmall) HIP_TRY(hipHostFree(c->hsmall));
    c->hsmall = nullptr;
    c->hsmall_cap = 0;
    HIP_TRY(hipHostMalloc((void **)&c->hsmall, sizeof(unsigned long long) * (size_t)words, hipHostMallocDefault));
    c->hsmall_cap = words;
    return JAM_OK;
}

// join frontiers (both buffers), rows of `stride` entries
int32_t grow_front(jam_context *c, int64_t rows, int stride)
{
    if (rows <= c->front_cap && stride <= c->front_stride) return JAM_OK;
    rows = std::max<int64_t>(std::max<int64_t>(rows, c->front_cap), 1 << 16);
    stride = std::max(stride, c->front_stride);
    for (int b = 0; b < 2; b++) {
        HIP_TRY(c->j_pair[b].reserve(sizeof(int) * (size_t)rows));
        HIP_TRY(c->j_ent[b].reserve(sizeof(int) * (size_t)rows * stride));
    }
    c->front_cap = rows;
    c->front_stride = stride;
    return JAM_OK;
}

int32_t grow_done(jam_context *c, int64_t rows, int stride)
{
    if (rows <= c->done_cap && stride <= c->done_stride) return JAM_OK;
    rows = std::max<int64_t>(std::max<int64_t>(rows, c->done_cap), 1 << 14);
    stride = std::max(stride, c->done_stride);
    HIP_TRY(c->d_pair.reserve(sizeof(int) * (size_t)rows));
    HIP_TRY(c->d_ent.reserve(sizeof(int) * (size_t)rows * stride));
    c->done_cap = rows;
    c->done_stride = stride;
    return JAM_OK;
}

// keys and permutations of the sort of n matches
int32_t grow_sort(jam_context *c, int64_t n)
{
    if (n <= c->sort_cap) return JAM_OK;
    n = std::max<int64_t>(n, 1 << 14);
    for (int b = 0; b < 2; b++) {
        HIP_TRY(c->s_key[b].reserve(sizeof(unsigned long long) * (size_t)n));
        HIP_TRY(c->s_perm[b].reserve(sizeof(int) * (size_t)n));
        HIP_TRY(c->s_pkey[b].reserve(sizeof(unsigned int) * (size_t)n));
    }
    c->sort_cap = n;
    return JAM_OK;
}

int32_t grow_events(jam_context *c, int64_t cap, int stride)
{
    if (cap > c->event_cap || stride > c->event_stride) {
        cap = std::max<int64_t>(cap, std::max<int64_t>(c->event_cap, 1024));
        stride = std::max(stride, c->event_stride);
        HIP_TRY(c->e_all.reserve(event_layout(cap, stride).bytes));
        c->event_cap = cap;
        c->event_stride = stride;
    }
    return JAM_OK;
}

__global__ void k_zero_u64(unsigned long long *v, long long n)
{
    for (long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (long long)gridDim.x * blockDim.x)
        v[i] = 0ull;
}

// Sorting the complete matches by groups of level-0 rows. Up to
// GROUP_RANK_MATCHES matches with up to GROUP_RANK_WORK comparisons (halved)
// every group is ranked by comparison: the LDS sort's tiles would leave most
// CUs idle (49,000 matches: 46 us in 4 passes). Above, groups of up to
// GROUP_TILE / 2 matches are sorted in LDS (470,000 matches: 0.25 ms) and larger
// ones ranked, about 1.8 us per million comparisons (halved) and pass: past
// group_work_max of them the radix passes are faster (470,000 matches of a
// 100,000-atom assembly, 28 M in large groups: 0.56 ms against 1.7 ms by radix
// passes; 6.3 M matches, 550 M in large groups: 3.2 against 2.4 ms). More than
// GROUP_MATCHES_MAX matches go by radix passes at once, although not all of
// them have large groups: finding out costs 0.3 ms for 6.3 M matches and 2.5 ms
// for the 51 M of 16 assemblies x 7,000 symmetric templates, in vain where the
// groups are large; where they are small it would gain 0.3 to 0.5 ms of 3.8 to
// 5.6 ms (sort and superposition of 5.1 to 6.1 M matches, 8 to 1,024 to a group:
// 3.4 against 3.8, 4.4 against 4.7, 4.8 against 5.3 ms).
#ifndef GROUP_RANK_WORK
#define GROUP_RANK_WORK 8000000ull
#endif
#ifndef GROUP_RANK_MATCHES
#define GROUP_RANK_MATCHES 131072
#endif
constexpr int64_t GROUP_MATCHES_MAX = int64_t(1) << 22;
unsigned long long group_work_max(int64_t n) { return 200000000ull + 16ull * (unsigned long long)n; }

// workgroups of `kernel` (with `threads` threads) that stay resident on the device
template <class K>
int resident_grid(K kernel, int threads, int device)
{
    int per_cu = 0, cus = 0;
    if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, kernel, threads, 0) != hipSuccess ||
        hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, device) != hipSuccess)
        return 1024;
    return std::max(1, per_cu) * std::max(1, cus);
}

typedef void (*join_kernel)(DevMols, DevTpls, DevSets, DevPairs, DevJoin, QueryParams);

// The k_join variant of join level L: what a wave keeps in LDS and registers
// grows with the placed atoms that it has room for, and up to four of them the
// loops over them are unrolled: the first four levels of 6 assemblies x 2,000
// templates 7.9 -> 6.7 ms, of 768 proteins x 200 templates 2.07 -> 1.70 ms,
// against one variant by the largest template (24 placed atoms). All variants
// run five waves per SIMD (94 to 96 registers; six spill, and were 6 to 20%
// slower).
constexpr int JOIN_VARIANTS = 8;
int join_variant(int L) { return L <= 4 ? L - 1 : L <= 8 ? 4 : L <= 16 ? 5 : L <= 24 ? 6 : 7; }
const join_kernel JOIN_KERNELS[JOIN_VARIANTS] = {
    jam::k_join<4, JOIN_TW, 1>, jam::k_join<4, JOIN_TW, 2>,  jam::k_join<4, JOIN_TW, 3>,  jam::k_join<4, JOIN_TW, 4>,
    jam::k_join<8, JOIN_TW, 0>, jam::k_join<16, JOIN_TW, 0>, jam::k_join<24, JOIN_TW, 0>, jam::k_join<32, JOIN_TW, 0>};

// one join level; the grid is the number of workgroups that stay resident
// e0, e1 (profiling, else null): events the runtime records at the
// dispatch's own start and end
void launch_join(jam_context *c, hipStream_t s, const DevMols &dm, const DevTpls &dt, const DevSets &st,
                 const DevPairs &pr, const DevJoin &jn, const QueryParams &qp, hipEvent_t e0, hipEvent_t e1)
{
    const int v = join_variant(jn.level);
    if (c->join_grid[v] == 0) c->join_grid[v] = resident_grid(JOIN_KERNELS[v], JOIN_WAVES * JAM_WAVE, c->device);
    hipExtLaunchKernelGGL(JOIN_KERNELS[v], dim3((unsigned)c->join_grid[v]), dim3(JOIN_WAVES * JAM_WAVE), 0, s, e0, e1, 0,
                          dm, dt, st, pr, jn, qp);
}


// Where kd_launches puts its kernels: side stream k is kd_side[k], KD_MAIN `s`.
struct KdQueue {
    jam_context *c;
    hipStream_t s;
    int n_sets;
    hipError_t error = hipSuccess;

    void check(hipError_t e)
    {
        if (error == hipSuccess) error = e;
    }
    // at most as many workgroups as there are sets and as stay resident
    template <class... K, class... A>
    void run(int k, int slot, void (*kernel)(K...), int threads, A... args)
    {
        if (c->kd_grid[slot] == 0) c->kd_grid[slot] = resident_grid(kernel, threads, c->device);
        run_grid(k, std::min(n_sets, c->kd_grid[slot]), kernel, threads, args...);
    }
    template <class... K, class... A>
    void run_grid(int k, int blocks, void (*kernel)(K...), int threads, A... args)
    {
        if (error != hipSuccess) return;   // nothing runs out of order
        hipLaunchKernelGGL(kernel, dim3((unsigned)blocks), dim3((unsigned)threads), 0, k == KD_MAIN ? s : c->kd_side[k],
                           args...);
        check(hipGetLastError());
    }
    void fork(int k, int from)
    {
        if (k == from) check(hipEventRecord(c->kd_fast[k], s));
        check(hipStreamWaitEvent(c->kd_side[k], c->kd_fast[from], 0));
    }
    void joined(int k)
    {
        c->kd_used |= 1u << k;
        check(hipEventRecord(c->kd_joined[k], c->kd_side[k]));
    }
};

// Launches the kd passes over the candidate sets of `st` (kd_launches); the
// caller has cleared *st.kd_err.
int32_t launch_kd(jam_context *c, const DevMols &dm, const DevTpls &dt, const DevSets &st, hipStream_t s,
                  bool one_molecule, int64_t n_atoms)
{
    c->kd_pending = true;
    c->kd_used = 0u;
    KdQueue q{c, s, st.n_sets};
    jam::kd_launches(q, dm, dt, st, c->kscr.as<unsigned char>(), c->kd_bucket.as<int>(), c->kd_tied.as<int>(),
                     c->kd_count.as<unsigned int>(), one_molecule, n_atoms);
    HIP_TRY(q.error);
    return JAM_OK;
}

// `s` waits for the side streams of the last launch_kd
hipError_t kd_join(jam_context *c, hipStream_t s)
{
    for (int k = 0; k < KD_SIDES; k++) {
        if (!((c->kd_used >> k) & 1u)) continue;
        const hipError_t e = hipStreamWaitEvent(s, c->kd_joined[k], 0);
        if (e != hipSuccess) return e;
    }
    return hipSuccess;
}

// The complete matches in report order by LSD radix passes: first by template
// size, then over the level positions (`bits` bits each, `per` levels per
// 64-bit key), the last levels first, then the pair. The result is in
// s_perm[cur].
int32_t sort_radix(jam_context *c, const DevSets &st, const DevTpls &dt, const DevPairs &pr, const DevJoin &jn,
                   int64_t n_done, int stride, int bits, int pbits, hipStream_t s, int &cur)
{
    const int T = dt.n_templates;
    const unsigned gs = (unsigned)((n_done + 255) / 256);
    int32_t rc;
    cur = 0;
    const int per = std::max(1, 64 / bits);
    const int nt = stride;
    // the matches by template size (stably): a match's levels at or
    // past its template's size are 0, so a group of levels starting
    // at l0 needs sorting only over the matches of more than l0
    // atoms, a suffix; that suffix's order is the only one to change,
    // so both permutation buffers keep the rest as it was
    hipLaunchKernelGGL(jam::k_iota, dim3(gs), dim3(256), 0, s, c->s_perm[0].as<int>(), (long long)n_done);
    hipLaunchKernelGGL(jam::k_sizekey, dim3(gs), dim3(256), 0, s, dt, jn, (long long)n_done,
                       c->s_pkey[0].as<unsigned int>());
    {
        int which = 0;
        if ((rc = radix_sort<unsigned int>(c->s_pkey[0].as<unsigned int>(), c->s_perm[0].as<int>(),
                                           c->s_pkey[1].as<unsigned int>(), c->s_perm[1].as<int>(),
                                           (long long)n_done, 6, c->rs_hist, c->rs_off, c->q_scan, s,
                                           which)) != JAM_OK)
            return rc;
        cur = which;
        HIP_TRY(c->s_starts.reserve(sizeof(long long) * (JAM_MAX_LEVELS + 1)));
        hipLaunchKernelGGL(jam::k_size_starts, dim3(1), dim3(64), 0, s, c->s_pkey[which].as<const unsigned int>(),
                           (long long)n_done, nt, c->s_starts.as<long long>());
        HIP_TRY(hipGetLastError());
        HIP_TRY(hipMemcpyAsync(c->s_perm[cur ^ 1].as<int>(), c->s_perm[cur].as<const int>(),
                               sizeof(int) * (size_t)n_done, hipMemcpyDeviceToDevice, s));
        HIP_TRY(hipMemcpyAsync(c->hsmall, c->s_starts.as<const long long>(), sizeof(long long) * (size_t)(nt + 1),
                               hipMemcpyDeviceToHost, s));
        HIP_TRY(hipStreamSynchronize(s));
    }
    long long size_le[JAM_MAX_LEVELS + 1];
    std::memcpy(size_le, c->hsmall, sizeof(long long) * (size_t)(nt + 1));
    for (int l0 = ((nt - 1) / per) * per; l0 >= 0; l0 -= per) {
        const int cnt_l = std::min(per, nt - l0);
        const long long a = l0 == 0 ? 0 : size_le[l0];   // matches of at most l0 atoms stay put
        const long long m = (long long)n_done - a;
        if (m <= 1) continue;
        // levels [l0, l0 + cnt_l) packed into cnt_l * bits bits
        hipLaunchKernelGGL(jam::k_sortkey, dim3((unsigned)((m + 255) / 256)), dim3(256), 0, s, st, dt, pr, jn,
                           c->s_perm[cur].as<const int>() + a, m, l0, cnt_l, bits,
                           c->s_key[0].as<unsigned long long>() + a);
        int which = 0;
        if ((rc = radix_sort<unsigned long long>(c->s_key[0].as<unsigned long long>() + a,
                                                 c->s_perm[cur].as<int>() + a,
                                                 c->s_key[1].as<unsigned long long>() + a,
                                                 c->s_perm[cur ^ 1].as<int>() + a, m, cnt_l * bits,
                                                 c->rs_hist, c->rs_off, c->q_scan, s, which)) != JAM_OK)
            return rc;
        cur ^= which;
    }
    hipLaunchKernelGGL(jam::k_pairkey, dim3(gs), dim3(256), 0, s, jn, T, c->s_perm[cur].as<const int>(),
                       (long long)n_done, c->s_pkey[0].as<unsigned int>());
    int which = 0;
    if ((rc = radix_sort<unsigned int>(c->s_pkey[0].as<unsigned int>(), c->s_perm[cur].as<int>(),
                                       c->s_pkey[1].as<unsigned int>(), c->s_perm[cur ^ 1].as<int>(),
                                       (long long)n_done, pbits, c->rs_hist, c->rs_off, c->q_scan, s,
                                       which)) != JAM_OK)
        return rc;
    cur ^= which;
    HIP_TRY(hipGetLastError());
    return JAM_OK;
}

// The same by groups of level-0 rows (k_group_count ... k_group_tile); the
// result is `perm`. `perm` stays null, with nothing sorted, where the rows
// cannot be numbered in 32 bits, or the matches are too many or their groups
// too large.
int32_t sort_groups(jam_context *c, const DevSets &st, const DevTpls &dt, const DevPairs &pr, const DevJoin &jn,
                    int64_t n_done, int64_t n_rows, int stride, int bits, hipStream_t s, const int *&perm)
{
    perm = nullptr;
    if (n_rows > (int64_t)UINT32_MAX || n_done > GROUP_MATCHES_MAX) return JAM_OK;
    // about as many groups as matches: fewer would mean more comparisons,
    // more a longer scan
    int shift = 0;
    while ((n_rows >> shift) > std::max<int64_t>(2 * n_done, 1 << 16)) shift++;
    const int64_t groups = (n_rows >> shift) + 1;
    if (c->sg_count.reserve(sizeof(int) * (size_t)groups) != hipSuccess ||
        c->sg_start.reserve(sizeof(int) * ((size_t)groups + 1)) != hipSuccess ||
        c->sg_seg[0].reserve(sizeof(jam::GroupSeg) * (size_t)n_done) != hipSuccess ||
        c->sg_seg[1].reserve(sizeof(jam::GroupSeg) * (size_t)n_done) != hipSuccess ||
        c->sg_perm.reserve(sizeof(int) * (size_t)n_done) != hipSuccess ||
        c->sg_list.reserve(sizeof(int) * (size_t)n_done) != hipSuccess) {
        (void)hipGetLastError();   // no room for them: the radix passes need less
        return JAM_OK;
    }
    HIP_TRY(c->s_starts.reserve(sizeof(long long) * (JAM_MAX_LEVELS + 1)));
    const unsigned gs = (unsigned)((n_done + 255) / 256);
    unsigned int *row = c->s_pkey[0].as<unsigned int>();
    int *slot = c->s_pkey[1].as<int>();
    unsigned long long *work = c->s_starts.as<unsigned long long>();
    hipLaunchKernelGGL(k_fill_i32, dim3((unsigned)std::min<int64_t>(2048, (groups + 255) / 256)), dim3(256), 0, s,
                       c->sg_count.as<int>(), (long long)groups, 0);
    hipLaunchKernelGGL(k_zero_u64, dim3(1), dim3(64), 0, s, work, 4ll);
    hipLaunchKernelGGL(jam::k_group_count, dim3(std::min(gs, 2048u)), dim3(256), 0, s, st, dt, pr, jn, (long long)n_done,
                       shift, row, slot, c->sg_count.as<int>(), work);
    HIP_TRY(hipGetLastError());
    HIP_TRY(hipMemcpyAsync(c->hsmall, work, 3 * sizeof(unsigned long long), hipMemcpyDeviceToHost, s));
    const int32_t rc = device_scan<int, int>(c->sg_count.as<const int>(), groups, c->sg_start.as<int>(), c->q_scan, 0, s);
    HIP_TRY(hipStreamSynchronize(s));
    if (rc != JAM_OK) return rc;
    const unsigned long long all = c->hsmall[0], most = c->hsmall[1] + 1, big = c->hsmall[2];
    if (big > group_work_max(n_done)) return JAM_OK;
    // groups of at least `least` matches by ranking, the others in LDS
    const bool rank_all = all <= GROUP_RANK_WORK && n_done <= GROUP_RANK_MATCHES;
    const int half = GROUP_TILE / 2, least = rank_all ? 1 : half + 1;
    int *list = rank_all ? nullptr : c->sg_list.as<int>();
    unsigned long long *n_list = work + 3;
    hipLaunchKernelGGL(jam::k_group_scatter, dim3(gs), dim3(256), 0, s, dt, pr, jn, (long long)n_done, shift, least,
                       (const unsigned int *)row, (const int *)slot, c->sg_start.as<const int>(),
                       c->s_perm[0].as<int>(), c->s_key[0].as<unsigned long long>(), c->sg_seg[0].as<jam::GroupSeg>());
    if (!rank_all)
        hipLaunchKernelGGL(jam::k_group_tile, dim3((unsigned)((n_done + half - 1) / half)), dim3(1024), 0, s, dt, pr, jn,
                           (long long)n_done, shift, (const unsigned int *)row, c->s_perm[0].as<const int>(),
                           c->sg_seg[0].as<const jam::GroupSeg>(), c->sg_perm.as<int>());
    if (!rank_all && most >= (unsigned long long)least)
        hipLaunchKernelGGL(jam::k_group_list, dim3(gs), dim3(256), 0, s, c->sg_seg[0].as<const jam::GroupSeg>(),
                           (long long)n_done, least, list, n_list);
    if (rank_all || most >= (unsigned long long)least) {
        const int words = jam::group_passes(stride, shift, bits);
        const unsigned waves = (unsigned)std::min<int64_t>(8192, (n_done + 3) / 4);
        int cur = 0;
        for (int w = 0; w < words; w++, cur ^= 1)
            hipLaunchKernelGGL(jam::k_group_rank, dim3(waves), dim3(256), 0, s, dt, pr, jn, (long long)n_done,
                               (const int *)list, (const unsigned long long *)n_list, c->s_perm[cur].as<const int>(),
                               c->s_key[cur].as<const unsigned long long>(), c->sg_seg[cur].as<const jam::GroupSeg>(),
                               w + 1 < words ? c->s_perm[cur ^ 1].as<int>() : c->sg_perm.as<int>(),
                               c->s_key[cur ^ 1].as<unsigned long long>(), c->sg_seg[cur ^ 1].as<jam::GroupSeg>());
    }
    HIP_TRY(hipGetLastError());
    perm = c->sg_perm.as<const int>();
    return JAM_OK;
}

}  // namespace

// One device array of counters, read back in one copy after the join: rows
// per join level, complete matches, the overflow flag, then the sizes phase A
// finds (candidate-set entries, level-0 items, largest set).
constexpr int CNT_DONE = JAM_MAX_LEVELS;
constexpr int CNT_OVF = JAM_MAX_LEVELS + 1;
constexpr int CNT_TOTAL = JAM_MAX_LEVELS + 2;
constexpr int CNT_ITEMS = JAM_MAX_LEVELS + 3;
constexpr int CNT_MAXCNT = JAM_MAX_LEVELS + 4;
constexpr int CNT_WORDS = JAM_MAX_LEVELS + 5;

extern "C" int32_t jam_query(jam_context *c, const jam_templates *tp, const jam_molecules *ms,
                             const jam_params *p, jam_result **out)
{
    if (!c || !tp || !ms || !p || !out) return fail(JAM_EINVAL, "NULL argument");
    if (tp->ctx != c || ms->ctx != c) return fail(JAM_EINVAL, "objects belong to another context");
    if (p->ignore_chain < 0 || p->ignore_chain > 2) return fail(JAM_EINVAL, "invalid ignore_chain");
    *out = nullptr;
    HIP_TRY(hipSetDevice(c->device));
    drain_kd(c);
    std::unique_ptr<jam_result> R(new jam_result());
    R->ctx = c;
    R->gen = ++c->query_gen;
    const int T = tp->n_templates, M = ms->n_mols, U = tp->n_types;
    const int64_t n_pairs64 = (int64_t)T * M;
    if (n_pairs64 > INT32_MAX / 64) return fail(JAM_ETOOBIG, "too many (template, molecule) pairs");
    if ((int64_t)M * U > INT32_MAX / 64) return fail(JAM_ETOOBIG, "too many (molecule, atom type) sets");
    const int n_pairs = (int)n_pairs64;
    R->n_pairs = n_pairs;
    R->stride = tp->stride;
    R->pair_cm.assign(n_pairs, 0);
    if (n_pairs == 0 || U == 0) {
        *out = R.release();
        return JAM_OK;
    }
    const int n_sets = M * U;
    hipStream_t s = c->stream;
    QueryParams qp;
    qp.rmsd_threshold = p->rmsd_threshold;
    qp.distance_cutoff = p->distance_cutoff;
    qp.max_dynamic_distance = p->max_dynamic_distance;
    qp.ignore_chain = p->ignore_chain;
    qp.reorder = p->reorder ? 1 : 0;
    qp.chunk = 1;
    const int stride = tp->stride;

    int32_t rc;
    if ((rc = grow_sets(c, std::max<int64_t>(c->set_cap, 1 << 16), n_sets)) != JAM_OK) return rc;
    if ((rc = grow_events(c, std::max<int64_t>(c->event_cap, 1 << 12), stride)) != JAM_OK) return rc;
    if ((rc = grow_pairs(c, n_pairs)) != JAM_OK) return rc;
    if ((rc = grow_hsmall(c, std::max<int64_t>(CNT_WORDS, (int64_t)n_pairs + 2))) != JAM_OK) return rc;
    HIP_TRY(c->j_count.reserve(sizeof(unsigned long long) * CNT_WORDS));
    DevMols dm = ms->dev();
    DevTpls dt = tp->dev();

    for (int attempt = 0; attempt < 8; attempt++) {
        DevSets st;
        st.n_sets = n_sets;
        st.cap = c->set_cap;
        st.blk_cap = c->blk_cap;
        st.cnt = c->cnt.as<int>();
        st.off = c->off.as<int64_t>();
        st.list = c->list.as<int>();
        st.kidx = c->kidx.as<int>();
        st.l2k = c->l2k.as<int>();
        st.kent = c->kent.as<SetEnt>();
        st.katom = c->katom.as<int>();
        st.bbox = c->bbox.as<double>();
        st.sbox = c->sbox.as<double>();
        unsigned long long *cnts = c->j_count.as<unsigned long long>();
        st.total = (int64_t *)(cnts + CNT_TOTAL);
        st.maxcnt = (int *)(cnts + CNT_MAXCNT);
        // the kd error word sits after the per-pair counts, which are read
        // back at the end of the query
        unsigned long long *pcm = (unsigned long long *)c->p_cm.ptr;
        st.kd_err = (unsigned int *)(pcm + (size_t)n_pairs + 1);
        DevPairs pr;
        pr.n_pairs = n_pairs;
        pr.n_items = (const long long *)(cnts + CNT_ITEMS);
        pr.ord = c->p_ord.as<unsigned char>();
        pr.lvl = c->p_lvl.as<PairLevel>();
        pr.nchunk = c->p_nchunk.as<int>();
        pr.n1 = c->p_n1.as<int>();
        pr.item_base = c->p_base.as<long long>();

        const int wpb = 4;  // waves per block of the per-set candidate kernels
        const int set_blocks = (n_sets + wpb - 1) / wpb;
        HIP_TRY(hipEventRecord(c->ev[0], s));
        hipLaunchKernelGGL(jam::k_candidates<false>, dim3(set_blocks), dim3(64 * wpb), 0, s, dm, dt, st, pr,
                           (long long *)nullptr, (unsigned long long *)nullptr, 0);
        HIP_TRY(hipGetLastError());
        if ((rc = device_scan<int, int64_t>(st.cnt, n_sets, st.off, c->q_scan, 0, s, st.maxcnt)) != JAM_OK) return rc;
        hipLaunchKernelGGL(jam::k_pairs, dim3((unsigned)((n_pairs + 7) / 8)), dim3(256), 0, s, dt, st, pr, qp, pcm + 1);
        HIP_TRY(hipGetLastError());
        if ((rc = device_scan<int, long long>(pr.nchunk, n_pairs, pr.item_base, c->q_scan, 0, s)) != JAM_OK)
            return rc;
        // no read-back here: the buffers keep the sizes of earlier queries,
        // every kernel below checks the sizes on the device, and the host
        // reads them with the join's counters, growing and running the query
        // again when something did not fit
        hipLaunchKernelGGL(jam::k_candidates<true>, dim3(set_blocks), dim3(64 * wpb), 0, s, dm, dt, st, pr,
                           (long long *)(cnts + CNT_ITEMS), cnts, CNT_TOTAL);
        HIP_TRY(hipGetLastError());
        HIP_TRY(hipEventRecord(c->ev[1], s));
        if ((rc = launch_kd(c, dm, dt, st, s, M == 1, ms->n_atoms)) != JAM_OK) {
            drain_kd(c);
            return rc;
        }
        HIP_TRY(kd_join(c, s));
        c->kd_pending = false;   // the rest of the query is ordered after every kd pass
        HIP_TRY(hipGetLastError());
        HIP_TRY(hipEventRecord(c->ev[2], s));

        // ---- the join: one launch per level, back to back; the counters
        // stay on the device until the end
        const int levels = std::max(1, stride - 1);
        if ((rc = grow_front(c, std::max<int64_t>(c->front_cap, 1 << 14), stride)) != JAM_OK) return rc;
        if ((rc = grow_done(c, std::max<int64_t>(c->done_cap, 1 << 14), stride)) != JAM_OK) return rc;
        unsigned long long *fcount = cnts;   // rows per level
        unsigned long long *n_done_dev = cnts + CNT_DONE;
        unsigned int *overflow = (unsigned int *)(cnts + CNT_OVF);
        DevJoin jn{};
        jn.stride = c->front_stride;
        jn.in_stride = 1;
        jn.out_stride = 1;
        jn.n_done = n_done_dev;
        jn.done_cap = c->done_cap;
        jn.done_pair = c->d_pair.as<int>();
        jn.done_ent = c->d_ent.as<int>();
        jn.overflow = overflow;
        if (c->done_stride != c->front_stride) {
            if ((rc = grow_done(c, c->done_cap, c->front_stride)) != JAM_OK) return rc;
            jn.done_pair = c->d_pair.as<int>();
            jn.done_ent = c->d_ent.as<int>();
        }
        {
            jn.level = 0;
            jn.n_out = fcount;
            jn.out_cap = c->front_cap;
            jn.out_pair = c->j_pair[0].as<int>();
            jn.out_ent = c->j_ent[0].as<int>();
            const int team = n_pairs > 4096 ? JAM_WAVE : 256, teams = 256 / team;
            hipLaunchKernelGGL(jam::k_level0, dim3((unsigned)((n_pairs + teams - 1) / teams)), dim3(256), 0, s, st, pr,
                               jn, team);
            HIP_TRY(hipGetLastError());
            for (int L = 1; L <= levels; L++) {
                const int bi = (L - 1) & 1, bo = L & 1;
                jn.level = L;
                jn.n_in = fcount + (L - 1);
                jn.in_cap = c->front_cap;
                jn.in_pair = c->j_pair[bi].as<int>();
                jn.in_ent = c->j_ent[bi].as<int>();
                // the frontier of level L - 1 holds L entries per row (a
                // child of level L exists only for templates of more than
                // L + 1 atoms, so L + 1 never exceeds the row buffers' width)
                jn.in_stride = L;
                jn.out_stride = std::min(L + 1, jn.stride);
                jn.n_out = fcount + L;
                jn.out_cap = c->front_cap;
                jn.out_pair = c->j_pair[bo].as<int>();
                jn.out_ent = c->j_ent[bo].as<int>();
                launch_join(c, s, dm, dt, st, pr, jn, qp, c->profile ? c->xev[2 * (L - 1) + 0] : nullptr,
                            c->profile ? c->xev[2 * (L - 1) + 1] : nullptr);
                HIP_TRY(hipGetLastError());
            }
        }
        unsigned long long *jc = c->hsmall;
        HIP_TRY(hipMemcpyAsync(jc, cnts, sizeof(unsigned long long) * CNT_WORDS, hipMemcpyDeviceToHost, s));
        HIP_TRY(hipStreamSynchronize(s));
        const int64_t total = (int64_t)jc[CNT_TOTAL];
        const int64_t n0 = (int64_t)jc[CNT_ITEMS];
        int maxcnt = 0;
        std::memcpy(&maxcnt, jc + CNT_MAXCNT, sizeof(int));
        if (total >= INT32_MAX) return fail(JAM_ETOOBIG, "more than 2^31 candidate-set entries in one query");
        const unsigned int ovf = (unsigned int)(jc[CNT_OVF] & 0xFFFFFFFFull);
        const int64_t n_done = (int64_t)jc[CNT_DONE];
        const bool regrow = total > c->set_cap || n0 > c->front_cap;
        if (regrow) {
            if (total > c->set_cap && (rc = grow_sets(c, total, n_sets)) != JAM_OK) return rc;
            if (n0 > c->front_cap && (rc = grow_front(c, std::max<int64_t>(2 * c->front_cap, n0), stride)) != JAM_OK)
                return rc;
            continue;
        }
        unsigned long long rows[JAM_MAX_LEVELS];   // the read-back area is reused below
        std::memcpy(rows, jc, sizeof(rows));
        if (ovf || n_done > c->done_cap) {
            // rows that did not fit: grow to what was seen (deeper levels saw
            // truncated inputs, so this may take another round)
            int64_t need = 0;
            for (int L = 0; L < JAM_MAX_LEVELS; L++) need = std::max<int64_t>(need, (int64_t)jc[L]);
            if ((rc = grow_front(c, std::max<int64_t>(2 * c->front_cap, need), stride)) != JAM_OK) return rc;
            if ((rc = grow_done(c, std::max<int64_t>(c->done_cap, 2 * n_done), c->front_stride)) != JAM_OK)
                return rc;
            continue;
        }
        HIP_TRY(hipEventRecord(c->ev[3], s));

        // ---- reference order of the complete matches: the order of the key
        // (pair, level 0 position, level 1 position, ...), by rank counting
        // when the matches are few, else by LSD radix passes over the level
        // positions (`bits` bits each, `per` levels per 64-bit key), the last
        // levels first, then the pair
        if ((rc = grow_sort(c, n_done)) != JAM_OK) return rc;
        if ((rc = grow_events(c, n_done, stride)) != JAM_OK) return rc;
        int cur = 0;
        const int *grouped = nullptr;
        const unsigned gs = (unsigned)((n_done + 255) / 256);
        int pbits = 1;
        while ((1ll << pbits) < (long long)n_pairs) pbits++;
        int bits = 1;
        while ((1ll << bits) <= (long long)maxcnt) bits++;
        const int words = (pbits + stride * bits + 63) / 64;
        if (n_done > 0 && n_done <= SORT_RANK_MAX && words <= SORT_RANK_WORDS) {
            // rank counting: same permutation as the radix passes below
            HIP_TRY(c->s_key[0].reserve(sizeof(unsigned long long) * (size_t)n_done * words));
            unsigned long long *fk = c->s_key[0].as<unsigned long long>();
            int *rank = c->s_perm[1].as<int>();
            const dim3 tiles((unsigned)((n_done + 255) / 256), (unsigned)((n_done + SORT_RANK_TJ - 1) / SORT_RANK_TJ));
            switch (words) {
#define JAM_RANK_SORT(W)                                                                                        \
    case W:                                                                                                     \
        hipLaunchKernelGGL(jam::k_fullkey<W>, dim3(gs), dim3(256), 0, s, st, dt, pr, jn, (long long)n_done, stride, \
                           bits, pbits, fk, rank);                                                              \
        hipLaunchKernelGGL(jam::k_rank<W>, tiles, dim3(256), 0, s, (const unsigned long long *)fk,                \
                           (long long)n_done, rank);                                                            \
        break;
                JAM_RANK_SORT(1)
                JAM_RANK_SORT(2)
                JAM_RANK_SORT(3)
                JAM_RANK_SORT(4)
#undef JAM_RANK_SORT
            }
            hipLaunchKernelGGL(jam::k_rank_scatter, dim3(gs), dim3(256), 0, s, (const int *)rank, (long long)n_done,
                               c->s_perm[0].as<int>());
            HIP_TRY(hipGetLastError());
        } else if (n_done > 0) {
            if ((rc = sort_groups(c, st, dt, pr, jn, n_done, n0, stride, bits, s, grouped)) != JAM_OK) return rc;
            if (!grouped && (rc = sort_radix(c, st, dt, pr, jn, n_done, stride, bits, pbits, s, cur)) != JAM_OK)
                return rc;
        }
        const int *perm = grouped ? grouped : c->s_perm[cur].as<const int>();

        // ---- superposition of every complete match; events in that order
        DevEvents ev;
        ev.cap = c->event_cap;
        ev.stride = stride;
        ev.base = c->e_all.as<unsigned char>();
        // the event count, then the complete matches of every pair and the kd
        // error word: read back in one copy
        ev.count = pcm;
        // marks and their scan reuse the (now free) 64-bit sort keys
        int *sel = c->s_key[0].as<int>();
        int *pos = c->s_key[1].as<int>();
        if (n_done > 0) {
            const long long *first = c->p_first.as<long long>();
            // few matches: the mark pass keeps its superpositions for the emit
            // pass (each is a chain of dependent FP64 work, long next to
            // reading it back)
            double *keep_d = nullptr;
            int *keep_i = nullptr;
            if (n_done <= SORT_RANK_MAX) {
                HIP_TRY(c->keep_d.reserve(sizeof(double) * 16 * (size_t)n_done));
                HIP_TRY(c->keep_i.reserve(sizeof(int) * (size_t)(stride + 2) * (size_t)n_done));
                keep_d = c->keep_d.as<double>();
                keep_i = c->keep_i.as<int>();
            }
            hipLaunchKernelGGL(jam::k_first, dim3(gs), dim3(256), 0, s, jn, perm, (long long)n_done,
                               c->p_first.as<long long>());
            hipLaunchKernelGGL(jam::k_super<false>, dim3(gs), dim3(256), 0, s, dm, dt, st, pr, jn, ev, qp, perm,
                               (long long)n_done, first, sel, (const int *)pos, keep_d, keep_i, (long long *)(pcm + 1));
            if ((rc = device_scan<int, int>((const int *)sel, (long long)n_done, pos, c->q_scan, 0, s, nullptr,
                                            ev.count)) != JAM_OK)
                return rc;
            hipLaunchKernelGGL(jam::k_super<true>, dim3(gs), dim3(256), 0, s, dm, dt, st, pr, jn, ev, qp, perm,
                               (long long)n_done, first, sel, (const int *)pos, keep_d, keep_i, (long long *)(pcm + 1));
            HIP_TRY(hipGetLastError());
        }
        HIP_TRY(hipEventRecord(c->ev[4], s));
        HIP_TRY(hipMemcpyAsync(c->hsmall, pcm, sizeof(unsigned long long) * ((size_t)n_pairs + 2),
                               hipMemcpyDeviceToHost, s));
        HIP_TRY(hipStreamSynchronize(s));
        // the error word is the low 32 bits of that slot (only they are
        // cleared and set on the device)
        if ((c->hsmall[(size_t)n_pairs + 1] & 0xFFFFFFFFull) != 0ull)
            return fail(JAM_EDEVICE, "a kd pass reached its round bound (broken QuickSelect invariant)");
        const unsigned long long ne_dev = c->hsmall[0];
        std::memcpy(R->pair_cm.data(), c->hsmall + 1, sizeof(long long) * (size_t)n_pairs);
        if ((int64_t)ne_dev > c->event_cap || (int64_t)ne_dev > n_done)
            return fail(JAM_EDEVICE, "event count exceeds the complete matches");
        float ms_k[5] = {0, 0, 0, 0, 0};
        HIP_TRY(hipEventElapsedTime(&ms_k[0], c->ev[0], c->ev[1]));
        HIP_TRY(hipEventElapsedTime(&ms_k[1], c->ev[1], c->ev[2]));
        HIP_TRY(hipEventElapsedTime(&ms_k[2], c->ev[2], c->ev[3]));
        HIP_TRY(hipEventElapsedTime(&ms_k[3], c->ev[3], c->ev[4]));
        HIP_TRY(hipEventElapsedTime(&ms_k[4], c->ev[0], c->ev[4]));
        for (int k = 0; k < 5; k++) R->ms[k] = ms_k[k];
        const int n_launched = levels;
        R->expand_ms = c->profile ? 0.0 : -1.0;
        for (int q = 0; c->profile && q < n_launched; q++) {
            float x = 0.f;
            HIP_TRY(hipEventElapsedTime(&x, c->xev[2 * q], c->xev[2 * q + 1]));
            R->expand_ms += x;
        }
        R->expand_launches = c->profile ? n_launched : 0;
        for (int q = 0; q < JAM_MAX_LEVELS; q++) R->level_partials[q] = 0;
        for (int L = 1; L < JAM_MAX_LEVELS && L <= n_launched; L++) R->level_partials[L] = (int64_t)rows[L - 1];
        R->n_events = (int64_t)ne_dev;
        HIP_TRY(hipStreamSynchronize(s));
        *out = R.release();
        return JAM_OK;
    }
    return fail(JAM_EDEVICE, "query did not converge after growing its buffers");
}

// ---------------------------------------------------------------------------
// results
// ---------------------------------------------------------------------------

extern "C" int64_t jam_result_n_events(const jam_result *r) { return r ? r->n_events : 0; }

extern "C" int32_t jam_result_stride(const jam_result *r) { return r ? r->stride : 0; }

extern "C" int32_t jam_result_n_pairs(const jam_result *r) { return r ? r->n_pairs : 0; }

// Copies the fields of n events packed at `base` (device memory, the layout
// of event_layout(n, stride)) to host buffers (any may be NULL) through the
// context's pinned slots, on the context's stream.
static int32_t copy_event_fields(jam_context *c, const char *base, size_t n, int stride, int32_t *pair,
                                 int64_t *rank, int32_t *flag, double *rmsd, double *rot, double *c0, double *c1,
                                 int32_t *atoms)
{
    HIP_TRY(hipSetDevice(c->device));
    // in the order of the packed layout, so that neighbouring pieces are
    // contiguous on the device
    std::vector<CopyPiece> pieces;
    const EventLayout L = event_layout((int64_t)n, stride);
    auto add = [&](void *dst, size_t at, size_t bytes) { add_pieces(pieces, dst, base + at, bytes); };
    add(rank, L.rank, sizeof(int64_t) * n);
    add(rmsd, L.rmsd, sizeof(double) * n);
    add(rot, L.rot, sizeof(double) * 9 * n);
    add(c0, L.c0, sizeof(double) * 3 * n);
    add(c1, L.c1, sizeof(double) * 3 * n);
    add(pair, L.pair, sizeof(int32_t) * n);
    add(flag, L.flag, sizeof(int32_t) * n);
    add(atoms, L.atoms, sizeof(int32_t) * (size_t)stride * n);
    return copy_out(c, pieces);
}

extern "C" int32_t jam_result_copy(const jam_result *r, int32_t *pair, int64_t *rank, int32_t *flag,
                                   double *rmsd, double *rot, double *c0, double *c1, int32_t *atoms)
{
    if (!r) return fail(JAM_EINVAL, "NULL result");
    const size_t n = (size_t)r->n_events;
    if (n == 0) return JAM_OK;
    jam_context *c = r->ctx;
    if (!c || c->query_gen != r->gen)
        return fail(JAM_ESTALE, "the events of this result were overwritten by a later query on its context");
    return copy_event_fields(c, c->e_all.as<const char>(), n, r->stride, pair, rank, flag, rmsd, rot, c0, c1,
                             atoms);
}

// events kept in device memory of their own (jam_result_keep)
struct jam_events {
    jam_context *ctx = nullptr;
    int64_t n = 0;
    int stride = 1;
    void *dev = nullptr;
};

extern "C" int32_t jam_result_keep(const jam_result *r, jam_events **out)
{
    if (!r || !out) return fail(JAM_EINVAL, "NULL argument");
    *out = nullptr;
    jam_context *c = r->ctx;
    if (!c || c->query_gen != r->gen)
        return fail(JAM_ESTALE, "the events of this result were overwritten by a later query on its context");
    HIP_TRY(hipSetDevice(c->device));
    std::unique_ptr<jam_events> e(new jam_events());
    e->ctx = c;
    e->n = r->n_events;
    e->stride = r->stride;
    const size_t bytes = event_layout(e->n, e->stride).bytes;
    if (bytes > 0) {
        HIP_TRY(hipMalloc(&e->dev, bytes));
        // ordered before the context's next query, which overwrites the source
        const hipError_t err = hipMemcpyAsync(e->dev, c->e_all.ptr, bytes, hipMemcpyDeviceToDevice, c->stream);
        if (err != hipSuccess) {
            (void)hipFree(e->dev);
            return fail(JAM_EDEVICE, std::string("hipMemcpyAsync: ") + hipGetErrorString(err));
        }
    }
    *out = e.release();
    return JAM_OK;
}

extern "C" int32_t jam_events_copy(const jam_events *e, int32_t *pair, int64_t *rank, int32_t *flag, double *rmsd,
                                   double *rot, double *c0, double *c1, int32_t *atoms)
{
    if (!e) return fail(JAM_EINVAL, "NULL events");
    if (e->n == 0) return JAM_OK;
    return copy_event_fields(e->ctx, (const char *)e->dev, (size_t)e->n, e->stride, pair, rank, flag, rmsd, rot, c0,
                             c1, atoms);
}

extern "C" void jam_events_free(jam_events *e)
{
    if (!e) return;
    (void)hipSetDevice(e->ctx->device);
    if (e->dev) (void)hipFree(e->dev);
    delete e;
}

extern "C" int32_t jam_result_pair_matches(const jam_result *r, int64_t *counts)
{
    if (!r || !counts) return fail(JAM_EINVAL, "NULL argument");
    std::memcpy(counts, r->pair_cm.data(), sizeof(int64_t) * r->pair_cm.size());
    return JAM_OK;
}

extern "C" int32_t jam_result_pair_digests(const jam_result *r, int32_t mol_base, int32_t n_templates,
                                           int64_t *hit_counts, uint64_t *digests)
{
    if (!r || !hit_counts || !digests) return fail(JAM_EINVAL, "NULL argument");
    if (n_templates < 1 || r->n_pairs % n_templates != 0) return fail(JAM_EINVAL, "invalid template count");
    jam_context *c = r->ctx;
    if (!c || c->query_gen != r->gen)
        return fail(JAM_ESTALE, "the events of this result were overwritten by a later query on its context");
    const size_t np = (size_t)r->n_pairs;
    if (np == 0) return JAM_OK;
    HIP_TRY(hipSetDevice(c->device));
    hipStream_t s = c->stream;
    HIP_TRY(c->dig.reserve(2 * sizeof(unsigned long long) * np));
    unsigned long long *d = c->dig.as<unsigned long long>();
    hipLaunchKernelGGL(k_zero_u64, dim3((unsigned)std::min<size_t>(1024, (2 * np + 255) / 256)), dim3(256), 0, s, d,
                       (long long)(2 * np));
    if (r->n_events > 0)
        hipLaunchKernelGGL(jam::k_pair_digest, dim3((unsigned)((r->n_events + 255) / 256)), dim3(256), 0, s,
                           c->e_all.as<const unsigned char>(), (long long)r->n_events, r->stride, n_templates,
                           mol_base, d, d + np);
    HIP_TRY(hipGetLastError());
    HIP_TRY(hipMemcpyAsync(hit_counts, d, sizeof(int64_t) * np, hipMemcpyDeviceToHost, s));
    HIP_TRY(hipMemcpyAsync(digests, d + np, sizeof(uint64_t) * np, hipMemcpyDeviceToHost, s));
    HIP_TRY(hipStreamSynchronize(s));
    return JAM_OK;
}

extern "C" int32_t jam_result_timings(const jam_result *r, double *ms5)
{
    if (!r || !ms5) return fail(JAM_EINVAL, "NULL argument");
    std::memcpy(ms5, r->ms, sizeof(r->ms));
    return JAM_OK;
}

extern "C" int32_t jam_result_level_partials(const jam_result *r, int64_t *counts)
{
    if (!r || !counts) return fail(JAM_EINVAL, "NULL argument");
    std::memcpy(counts, r->level_partials, sizeof(r->level_partials));
    return JAM_OK;
}

extern "C" int32_t jam_context_set_profiling(jam_context *c, int32_t on)
{
    if (!c) return fail(JAM_EINVAL, "NULL context");
    c->profile = on != 0;
    return JAM_OK;
}

extern "C" int32_t jam_result_join_kernels(const jam_result *r, double *ms, int32_t *launches)
{
    if (!r || !ms || !launches) return fail(JAM_EINVAL, "NULL argument");
    *ms = r->expand_ms;
    *launches = r->expand_launches;
    return JAM_OK;
}

extern "C" void jam_result_free(jam_result *r) { delete r; }

// ---------------------------------------------------------------------------
// standalone superposition
// ---------------------------------------------------------------------------

namespace {

// k_superpose_batch over device arrays, on stream s
int32_t superpose_launch(hipStream_t s, const double *da, const double *db, int k, int64_t n_sets, double *drmsd,
                         double *drot, double *dc0, double *dc1)
{
    const int tb = 256;
    hipLaunchKernelGGL(jam::k_superpose_batch, dim3((unsigned)((n_sets + tb - 1) / tb)), dim3(tb), 0, s, da, db, k,
                       (long long)n_sets, drmsd, drot, dc0, dc1);
    HIP_TRY(hipGetLastError());
    return JAM_OK;
}

// copies the outputs back and waits for them
int32_t superpose_fetch(hipStream_t s, int64_t n_sets, const void *drmsd, const void *drot, const void *dc0,
                        const void *dc1, double *rmsd, double *rot, double *c0, double *c1)
{
    HIP_TRY(hipMemcpyAsync(rmsd, drmsd, sizeof(double) * n_sets, hipMemcpyDeviceToHost, s));
    HIP_TRY(hipMemcpyAsync(rot, drot, sizeof(double) * 9 * n_sets, hipMemcpyDeviceToHost, s));
    HIP_TRY(hipMemcpyAsync(c0, dc0, sizeof(double) * 3 * n_sets, hipMemcpyDeviceToHost, s));
    HIP_TRY(hipMemcpyAsync(c1, dc1, sizeof(double) * 3 * n_sets, hipMemcpyDeviceToHost, s));
    HIP_TRY(hipStreamSynchronize(s));
    return JAM_OK;
}

}  // namespace

extern "C" int32_t jam_superpose_batch(jam_context *c, const double *a, const double *b, int32_t k,
                                       int64_t n_sets, double *rmsd, double *rot, double *c0, double *c1)
{
    if (!c || !a || !b || !rmsd || !rot || !c0 || !c1) return fail(JAM_EINVAL, "NULL argument");
    if (k < 1 || n_sets < 0) return fail(JAM_EINVAL, "invalid sizes");
    if (n_sets == 0) return JAM_OK;
    HIP_TRY(hipSetDevice(c->device));
    hipStream_t s = c->stream;
    const size_t pts = (size_t)n_sets * k * 3;
    HIP_TRY(c->sa.reserve(sizeof(double) * pts));
    HIP_TRY(c->sb.reserve(sizeof(double) * pts));
    HIP_TRY(c->srmsd.reserve(sizeof(double) * n_sets));
    HIP_TRY(c->srot.reserve(sizeof(double) * 9 * n_sets));
    HIP_TRY(c->sc0.reserve(sizeof(double) * 3 * n_sets));
    HIP_TRY(c->sc1.reserve(sizeof(double) * 3 * n_sets));
    HIP_TRY(hipMemcpyAsync(c->sa.ptr, a, sizeof(double) * pts, hipMemcpyHostToDevice, s));
    HIP_TRY(hipMemcpyAsync(c->sb.ptr, b, sizeof(double) * pts, hipMemcpyHostToDevice, s));
    int32_t rc = superpose_launch(s, c->sa.as<double>(), c->sb.as<double>(), k, n_sets, c->srmsd.as<double>(),
                                  c->srot.as<double>(), c->sc0.as<double>(), c->sc1.as<double>());
    if (rc != JAM_OK) return rc;
    return superpose_fetch(s, n_sets, c->srmsd.ptr, c->srot.ptr, c->sc0.ptr, c->sc1.ptr, rmsd, rot, c0, c1);
}

extern "C" int32_t jam_superpose_batch_noalloc(jam_context *c, const double *a, const double *b, int32_t k,
                                               int64_t n_sets, double *rmsd, double *rot, double *c0, double *c1)
{
    if (!c || !a || !b || !rmsd || !rot || !c0 || !c1) return fail(JAM_EINVAL, "NULL argument");
    if (k < 1 || n_sets < 0) return fail(JAM_EINVAL, "invalid sizes");
    if (n_sets == 0) return JAM_OK;
    // the array, cut into 256-byte aligned pieces: a, b, rmsd, rotations, centroids
    auto up = [](size_t x) { return (x + 255) & ~(size_t)255; };
    const size_t per_set = sizeof(double) * (6 * (size_t)k + 16);
    if ((size_t)n_sets > JAM_NOALLOC_SCRATCH_BYTES / per_set)
        return fail(JAM_ETOOBIG, "batch larger than the scratch of jam_superpose_batch_noalloc");
    const size_t pts = (size_t)n_sets * k * 3;
    const size_t o_a = 0, o_b = o_a + up(sizeof(double) * pts), o_r = o_b + up(sizeof(double) * pts);
    const size_t o_m = o_r + up(sizeof(double) * n_sets), o_c0 = o_m + up(sizeof(double) * 9 * n_sets);
    const size_t o_c1 = o_c0 + up(sizeof(double) * 3 * n_sets), end = o_c1 + up(sizeof(double) * 3 * n_sets);
    if (end > JAM_NOALLOC_SCRATCH_BYTES)
        return fail(JAM_ETOOBIG, "batch larger than the scratch of jam_superpose_batch_noalloc");
    if (c->device < 0 || c->device >= JAM_MAX_DEVICES) return fail(JAM_EDEVICE, "device ordinal has no scratch");
    void *base = nullptr;
    {
        std::lock_guard<std::mutex> g(g_scratch_init);
        base = g_scratch[c->device];
    }
    if (!base) return fail(JAM_EDEVICE, "the device's scratch address is unknown");
    std::lock_guard<std::mutex> busy(g_scratch_busy[c->device]);
    HIP_TRY(hipSetDevice(c->device));
    hipStream_t s = c->stream;
    unsigned char *w = static_cast<unsigned char *>(base);
    double *da = (double *)(w + o_a), *db = (double *)(w + o_b), *dr = (double *)(w + o_r);
    double *dm = (double *)(w + o_m), *d0 = (double *)(w + o_c0), *d1 = (double *)(w + o_c1);
    HIP_TRY(hipMemcpyAsync(da, a, sizeof(double) * pts, hipMemcpyHostToDevice, s));
    HIP_TRY(hipMemcpyAsync(db, b, sizeof(double) * pts, hipMemcpyHostToDevice, s));
    int32_t rc = superpose_launch(s, da, db, k, n_sets, dr, dm, d0, d1);
    if (rc != JAM_OK) {
        (void)hipStreamSynchronize(s);
        return rc;
    }
    return superpose_fetch(s, n_sets, dr, dm, d0, d1, rmsd, rot, c0, c1);
}

// ---------------------------------------------------------------------------
// standalone kd-tree leaf order
// ---------------------------------------------------------------------------

extern "C" int32_t jam_kd_order(jam_context *c, const double *xyz, const int64_t *off, int32_t n_sets,
                                int32_t *order)
{
    if (!c || !off || (n_sets > 0 && (!xyz || !order))) return fail(JAM_EINVAL, "NULL argument");
    if (n_sets < 0) return fail(JAM_EINVAL, "negative set count");
    if (off[0] != 0) return fail(JAM_EINVAL, "off[0] must be 0");
    for (int32_t k = 0; k < n_sets; k++)
        if (off[k + 1] < off[k]) return fail(JAM_EINVAL, "set offsets decrease");
    const int64_t total = off[n_sets];
    if (total >= INT32_MAX) return fail(JAM_ETOOBIG, "more than 2^31 points");
    if (n_sets == 0 || total == 0) return JAM_OK;
    HIP_TRY(hipSetDevice(c->device));
    drain_kd(c);
    hipStream_t s = c->stream;
    // every set is a molecule of its own whose candidate list is its points
    // in input order; chains and residue numbers are zero
    std::vector<int> aoff(n_sets + 1), cnt(n_sets), list((size_t)total);
    for (int32_t k = 0; k <= n_sets; k++) aoff[k] = (int)off[k];
    for (int32_t k = 0; k < n_sets; k++) {
        cnt[k] = (int)(off[k + 1] - off[k]);
        for (int i = 0; i < cnt[k]; i++) list[(size_t)off[k] + i] = i;
    }
    int32_t rc;
    if ((rc = grow_sets(c, std::max<int64_t>(total, c->set_cap), n_sets)) != JAM_OK) return rc;
    HIP_TRY(c->j_count.reserve(sizeof(unsigned long long) * CNT_WORDS));
    HIP_TRY(c->o_xyz.reserve(sizeof(double) * 3 * (size_t)total));
    HIP_TRY(c->o_zero.reserve(sizeof(int) * (size_t)total));
    HIP_TRY(upload(c->o_aoff, aoff, s));
    HIP_TRY(upload(c->cnt, cnt, s));
    HIP_TRY(upload(c->list, list, s));
    HIP_TRY(hipMemcpyAsync(c->off.ptr, off, sizeof(int64_t) * (size_t)n_sets, hipMemcpyHostToDevice, s));
    HIP_TRY(hipMemcpyAsync(c->o_xyz.ptr, xyz, sizeof(double) * 3 * (size_t)total, hipMemcpyHostToDevice, s));
    HIP_TRY(hipMemsetAsync(c->o_zero.ptr, 0, sizeof(int) * (size_t)total, s));
    unsigned long long *cnts = c->j_count.as<unsigned long long>();
    const unsigned long long tot = (unsigned long long)total;
    HIP_TRY(hipMemcpyAsync(cnts + CNT_TOTAL, &tot, sizeof(tot), hipMemcpyHostToDevice, s));
    DevMols dm{};
    dm.n_mols = n_sets;
    dm.atom_off = c->o_aoff.as<int>();
    dm.xyz = c->o_xyz.as<double>();
    dm.chain = c->o_zero.as<int>();
    dm.resseq = c->o_zero.as<int>();
    DevTpls dt{};
    dt.n_types = 1;
    DevSets st{};
    st.n_sets = n_sets;
    st.cap = c->set_cap;
    st.blk_cap = c->blk_cap;
    st.cnt = c->cnt.as<int>();
    st.off = c->off.as<int64_t>();
    st.list = c->list.as<int>();
    st.kidx = c->kidx.as<int>();
    st.l2k = c->l2k.as<int>();
    st.kent = c->kent.as<SetEnt>();
    st.katom = c->katom.as<int>();
    st.bbox = c->bbox.as<double>();
    st.sbox = c->sbox.as<double>();
    st.total = (int64_t *)(cnts + CNT_TOTAL);
    st.maxcnt = (int *)(cnts + CNT_MAXCNT);
    st.kd_err = c->kd_count.as<unsigned int>() + 2 * KD_TIERS;
    hipLaunchKernelGGL(jam::k_kd_setup, dim3(1), dim3(64), 0, s, st.kd_err, 1);
    if ((rc = launch_kd(c, dm, dt, st, s, n_sets == 1, total)) != JAM_OK) {
        drain_kd(c);
        return rc;
    }
    HIP_TRY(kd_join(c, s));
    std::vector<int> kidx((size_t)total);
    unsigned int err = 0;
    HIP_TRY(hipMemcpyAsync(kidx.data(), st.kidx, sizeof(int) * (size_t)total, hipMemcpyDeviceToHost, s));
    HIP_TRY(hipMemcpyAsync(&err, st.kd_err, sizeof(err), hipMemcpyDeviceToHost, s));
    HIP_TRY(hipStreamSynchronize(s));
    c->kd_pending = false;
    if (err) return fail(JAM_EDEVICE, "a kd pass reached its round bound (broken QuickSelect invariant)");
    // DFS position p (right child first) holds list element kidx[p] and is
    // leaf n-1-p
    for (int32_t k = 0; k < n_sets; k++) {
        const int64_t o = off[k];
        const int n = cnt[k];
        for (int p = 0; p < n; p++) order[(size_t)o + (n - 1 - p)] = kidx[(size_t)o + p];
    }
    return JAM_OK;
}
