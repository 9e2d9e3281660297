// rtc8x_slots.hpp -- the full-image launches (PATH_TRACE and PATH_TRACE_WITH_NRC), single and batched, as a
// scheduler of path slots: renderer/gpu_kernels/optix_pathtracing_kernels.cu:31-448 for volume-only scenes.
//
// One persistent workgroup per CU keeps about a thousand paths ("slots") in LDS, one dword per field and
// slot.  A slot is ready for exactly one kind of work -- a density lookup, a region walk, an escape, the end
// of a shadow ray, a real collision, a new path -- and a bit in that kind's mask says so.  A wavefront claims
// up to 64 slots that are ready for the same kind (the kind with the most), loads the fields the kind needs,
// runs it with full lanes, stores what changed and marks the slots ready for what comes next.  No path is
// bound to a lane, so no lane waits for its neighbours' events.
//
// What bounds the tracer is VALU issue and, next to it, the latency of the lookups.  With a path per lane for
// its whole life, 14 of 64 lanes did work per VALU instruction with the local majorants and 24 with the global
// one, and a third of the time went to vertex events with a few lanes each; here it is 26 and 44, in 10.3 G
// and 10.8 G instead of 18-19 G instructions per frame.  512^3 cloud, 1080p, 16 samples: 35.3 -> 24.9 ms (local), 36.5
// -> 29.2 ms (global); dense 128^3 cloud, 256 x 256, 4 samples: 1.17 -> 0.71 ms; 203 x 117, 1 sample, with the
// work order and tone map: 521 -> 271 us.
//
// Progress and exit.  The masks are taken and set with LDS atomics only; nothing is locked.  A claimed slot is
// always published again or retired by the wavefront that claimed it, and a wavefront that finds nothing
// ready sleeps and looks again until `active`, the number of slots that still have work, is zero.
#pragma once

namespace rtc8x {
namespace dev {

enum : uint32_t {
    kWorkLookup = 0,   // a tentative collision to look up (global majorant: tracking steps)
    kWorkWalk = 1,     // local majorants: a walk to the next tentative collision
    kWorkEscape = 2,   // a path that left the volume
    kWorkNeeDone = 3,  // a shadow ray that reached its end
    kWorkScatter = 4,  // a real collision
    kWorkStart = 5,    // a slot without a path
    kWorkKinds = 6,
    kWorkNone = 7      // a slot without work left
};

// Fields of a slot, one dword each.  Fields that are never alive together share a dword (the transmittance
// of the shadow ray and the direction's density), what follows from others is computed again (a shadow ray's
// origin, the walk's boundaries), and the throughput, whose channels are equal in a medium of one albedo,
// is kept once: a CU then holds about a thousand paths.
enum : uint32_t {
    kPix,      // lx | ly << 14 | flags
    kSample,   // sample of the pixel
    kCost,     // lookups of the pixel so far
    kIdxLen,   // region of the walk | path length << 15
    kRngLo, kRngHi,
    kOx, kOy, kOz,   // the segment's origin; from a collision on its position
    kDx, kDy, kDz,   // the path's direction
    kTp,             // throughput
    kCr, kCg, kCb,   // contribution
    kDirPd,          // density of the direction; during a shadow ray the transmittance
    kVis = kDirPd,
    kImp,            // initial importance
    kT, kT1,         // where the segment stands and ends
    kSx, kSy, kSz,   // the shadow ray's direction
    kNr, kNg, kNb, kK1, kK3,  // the NEE estimate's factors
    kCommonFields
};
constexpr uint32_t kPixShadow = 1u << 28, kPixSun = 1u << 29, kPixMask = 0x0FFFFFFFu, kPixNone = 0xFFFFFFFFu;
constexpr uint32_t kIdxBits = 15;  // RTC8X_MAX_REGIONS regions
static_assert(RTC8X_MAX_REGIONS <= 1u << kIdxBits && kHardMaxPathLength < 1u << (32 - kIdxBits), "kIdxLen");

constexpr uint32_t kDealt = 8;          // pixels of a workgroup's turn when they are dealt out
constexpr uint32_t kLdsBytes = 163840;  // of a CU
// REGION_BYTES: room for the region table (local majorants); SLOTS: at most this many
template <int ENTRY, int TRACKING, uint32_t REGION_BYTES, uint32_t SLOTS>
struct SlotLayout {
    static constexpr bool kLocal = TRACKING == RTC8X_TRACKING_LOCAL_MAJORANT;
    static constexpr bool kNrc = ENTRY == RTC8X_ENTRY_PATH_TRACE_WITH_NRC;
    // the region walk: optical depth (or the pending collision's majorant), 1 / direction in index space; then
    // the NRC's path spreads
    static constexpr uint32_t kTau = kCommonFields, kIv = kTau + 1;
    static constexpr uint32_t kSpread = kLocal ? kTau + 4 : kCommonFields;
    static constexpr uint32_t kFields = kSpread + (kNrc ? 2u : 0u);
    static constexpr uint32_t kFit = (kLdsBytes - REGION_BYTES - 4096u) / (4u * kFields) & ~63u;
    static constexpr uint32_t kSlots = kFit < SLOTS ? kFit : SLOTS;
};

template <int ENTRY, int TRACKING, uint32_t REGION_BYTES, uint32_t WAVES, uint32_t SLOTS>
struct SlotMem {
    using Lay = SlotLayout<ENTRY, TRACKING, REGION_BYTES, SLOTS>;
    uint32_t f[Lay::kFields][Lay::kSlots];
    uint32_t ready[kWorkKinds][64];  // bit b of word w: slot 64 b + w
    int32_t count[8];                // slots ready per kind (a hint: the masks decide)
    uint32_t active;                 // slots with work left
    uint32_t pad[3];
    uint16_t ids[WAVES][64];
    alignas(16) uint8_t regions[REGION_BYTES ? REGION_BYTES : 16];
};

// The region walk of Seg<RTC8X_TRACKING_LOCAL_MAJORANT> with what a visit needs held ready: the walk's
// linear region index and, per axis, the integer boundary ahead and what a step adds to it.  Positions,
// boundaries and decisions are Dda's, bit for bit.
struct RegionWalk {
    uint32_t idx;
    int32_t b0, b1, b2;        // boundary ahead (index space); kFarBoundary on an axis the ray does not move along
    int32_t ss0, ss1, ss2;     // +- region size, 0
    int32_t sg0, sg1, sg2;     // what a step adds to idx
    int32_t e0, e1, e2;        // boundary at which the ray leaves the grid
    float io0, io1, io2, iv0, iv1, iv2, id0, id1, id2, tn0, tn1, tn2;
    static constexpr int32_t kFarBoundary = 1 << 30;
    // values, not fields, are selected: a select of fields becomes one access through a selected address, and
    // the walk then lives in scratch memory
    static __device__ __forceinline__ int32_t pick(bool c, int32_t a, int32_t b) { return c ? a : b; }
    static __device__ __forceinline__ float pick(bool c, float a, float b) { return c ? a : b; }

    static __device__ __forceinline__ void axis_of(float id, int32_t stride, int32_t origin, int32_t size, int32_t dims,
                                                   int32_t c, int32_t& b, int32_t& ss, int32_t& sg, int32_t& e, float& iv)
    {
        ss = id > 0.0f ? size : (id < 0.0f ? -size : 0);
        sg = id > 0.0f ? stride : -stride;
        e = id > 0.0f ? origin + size * dims : origin;
        b = boundary(c, ss, origin, size);
        // an axis without motion never comes first: (far - origin) * inf
        iv = ss == 0 ? __builtin_huge_valf() : iv;
    }
    static __device__ __forceinline__ int32_t boundary(int32_t c, int32_t ss, int32_t origin, int32_t size)
    {
        const int32_t b = origin + __mul24(size, c) + (ss > 0 ? size : 0);
        return ss == 0 ? kFarBoundary : b;
    }
    __device__ __forceinline__ void refresh()
    {
        tn0 = ((float)b0 - io0) * iv0;
        tn1 = ((float)b1 - io1) * iv1;
        tn2 = ((float)b2 - io2) * iv2;
    }
    // the walk of the ray o + t d in region idx_, iv_ as Dda::init computed it; inv1, inv2: 1 / region_dims[1, 2]
    __device__ __forceinline__ void load(const rtc8x_grid& g, V3 o, V3 d, V3 iv_, uint32_t idx_, float inv1, float inv2)
    {
        const float* mm = g.inv_mat;
        const float x = o.x - g.vec[0], y = o.y - g.vec[1], z = o.z - g.vec[2];
        io0 = fmaf(x, mm[0], fmaf(y, mm[1], z * mm[2]));
        io1 = fmaf(x, mm[3], fmaf(y, mm[4], z * mm[5]));
        io2 = fmaf(x, mm[6], fmaf(y, mm[7], z * mm[8]));
        const V3 id = Dda::index_dir(g, d);
        id0 = id.x, id1 = id.y, id2 = id.z;
        iv0 = iv_.x, iv1 = iv_.y, iv2 = iv_.z;
        idx = idx_;
        // idx < 2^15: the half keeps the rounded quotient on the right side of every integer
        const int32_t c01 = (int32_t)(((float)idx_ + 0.5f) * inv2), c2 = (int32_t)idx_ - __mul24(c01, g.region_dims[2]);
        const int32_t c0 = (int32_t)(((float)c01 + 0.5f) * inv1), c1 = c01 - __mul24(c0, g.region_dims[1]);
        const int32_t size = region_size(g);
        axis_of(id0, g.region_dims[1] * g.region_dims[2], g.cell_origin[0], size, g.region_dims[0], c0, b0, ss0, sg0, e0, iv0);
        axis_of(id1, g.region_dims[2], g.cell_origin[1], size, g.region_dims[1], c1, b1, ss1, sg1, e1, iv1);
        axis_of(id2, 1, g.cell_origin[2], size, g.region_dims[2], c2, b2, ss2, sg2, e2, iv2);
        refresh();
    }
    static __device__ __forceinline__ int32_t cell_at(float t, float id, float io, int32_t origin, float inv_size, int32_t dims)
    {
        const float cf = floorf((fmaf(t, id, io) - (float)origin) * inv_size);
        return cf < 0.0f ? 0 : (cf > (float)(dims - 1) ? dims - 1 : (int32_t)cf);
    }
    // One visit, as Seg::visit_region.
    __device__ __forceinline__ int visit(const rtc8x_grid& g, const Medium& m, float& t, float t1, float& tau, float& mu,
                                         const uint8_t* __restrict__ table)
    {
        const uint32_t code = table[idx];
        if (code > RTC8X_REGION_EMPTY) {
            const int32_t k = (int32_t)(code - RTC8X_REGION_EMPTY);
            const float tx = fminf(fminf(fminf(__builtin_huge_valf(), ((float)(b0 + __mul24(k, ss0)) - io0) * iv0),
                                         ((float)(b1 + __mul24(k, ss1)) - io1) * iv1),
                                   ((float)(b2 + __mul24(k, ss2)) - io2) * iv2);
            if (tx > t) {
                if (!(tx < t1)) return kAdvanceEnd;
                t = tx;
                const int32_t size = region_size(g);
                const float inv_size = 1.0f / (float)size;
                const int32_t c0 = cell_at(t, id0, io0, g.cell_origin[0], inv_size, g.region_dims[0]);
                const int32_t c1 = cell_at(t, id1, io1, g.cell_origin[1], inv_size, g.region_dims[1]);
                const int32_t c2 = cell_at(t, id2, io2, g.cell_origin[2], inv_size, g.region_dims[2]);
                idx = (uint32_t)(__mul24(__mul24(c0, g.region_dims[1]) + c1, g.region_dims[2]) + c2);
                b0 = boundary(c0, ss0, g.cell_origin[0], size);
                b1 = boundary(c1, ss1, g.cell_origin[1], size);
                b2 = boundary(c2, ss2, g.cell_origin[2], size);
                refresh();
                return kAdvanceBudget;
            }
        }
        const bool m1 = tn1 < tn0;
        const float t01 = pick(m1, tn1, tn0);
        const bool is2 = tn2 < t01, is1 = !is2 & m1, is0 = !(is2 | m1);
        const float tna = pick(is2, tn2, t01);
        const float tend = tna < t1 ? tna : t1;
        mu = region_majorant(g, m, code);
        if (mu > 0.0f) {
            const float need = mu * (tend - t);
            if (tau < need) return kAdvanceCollision;
            tau = tau - need;
        }
        if (!(tna < t1)) return kAdvanceEnd;
        t = tend;
        if ((is0 & (b0 == e0)) | (is1 & (b1 == e1)) | (is2 & (b2 == e2))) return kAdvanceEnd;
        b0 += pick(is0, ss0, 0);
        b1 += pick(is1, ss1, 0);
        b2 += pick(is2, ss2, 0);
        idx += (uint32_t)pick(is2, sg2, pick(is1, sg1, sg0));
        refresh();
        return kAdvanceBudget;
    }
};

// The frame parameters are read anew for each chunk of work: held in registers from chunk to chunk, the
// parameters of every kind together spill (130 SGPRs, a quarter of the VALU instructions to move them).
typedef const __attribute__((address_space(4))) rtc8x_frame_params* ParamsPtr;

// One image by workgroup wg of its wgs; helper: a workgroup of another image of the batch, which takes pixels
// from this one's work counter only.
template <int ENTRY, int TRACKING, uint32_t REGION_BYTES, uint32_t WAVES, uint32_t SLOTS>
__device__ __forceinline__ void slots_body(ParamsPtr params, uint32_t W, uint32_t H, uint32_t num_samples, uint32_t ctr,
                                           uint32_t wg, uint32_t wgs, bool helper,
                                           SlotMem<ENTRY, TRACKING, REGION_BYTES, WAVES, SLOTS>& mem)
{
    using Lay = SlotLayout<ENTRY, TRACKING, REGION_BYTES, SLOTS>;
    constexpr bool kLocal = Lay::kLocal, kNrc = Lay::kNrc;
    const rtc8x_frame_params& p = *(const rtc8x_frame_params*)params;
    const uint32_t lane = threadIdx.x & 63u, wave = threadIdx.x >> 6;

    uint32_t total, tile_w, tiles_x;
    {
        tile_w = p.tile_shape == 1 ? 16u : (p.tile_shape == 2 ? 32u : (p.tile_shape == 3 ? 4u : 8u));
        const uint32_t tile_h = 64u / tile_w;
        tiles_x = (W + tile_w - 1) / tile_w;
        total = p.work_order ? W * H : tiles_x * ((H + tile_h - 1) / tile_h) * 64;
    }
    const size_t p_stride = (size_t)W * H, q_stride = (p_stride + 127u) & ~(size_t)127u;

    // Pixels come from the work counter.  Fewer than fill the slots are dealt out instead, eight at a time to
    // each workgroup in turn: the counter's atomics go through one address, and three thousand wavefronts
    // asking at once waited 30 us for their first pixel.  (With more pixels than slots, dealing out the first
    // ones costs more than the wait: 30.2 against 29.2 ms per global-majorant frame of the 512^3 cloud.)
    const uint32_t share = (total + wgs - 1) / wgs;
    const bool few = share < Lay::kSlots;
    if (helper) {
        // nothing to do here unless pixels are counted out and some are left
        if (few) return;
        if (threadIdx.x == 0) mem.active = __hip_atomic_load(&g_work_counter[ctr], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        __syncthreads();
        const bool left = mem.active < total;
        __syncthreads();
        if (!left) return;
    }
    const uint32_t n0 = few ? (share + kDealt - 1) / kDealt * kDealt : Lay::kSlots;
    const uint32_t waves = blockDim.x >> 6;
    for (uint32_t i = threadIdx.x; i < kWorkKinds * 64u; i += blockDim.x) {
        const uint32_t k = i / 64u, w = i % 64u;
        // slots 64 b + w below n0
        const uint32_t bits = w < n0 ? (n0 - w + 63u) / 64u : 0u;
        mem.ready[k][w] = k == kWorkStart && bits ? 0xFFFFFFFFu >> (32u - bits) : 0u;
    }
    if (threadIdx.x < 8) mem.count[threadIdx.x] = threadIdx.x == kWorkStart ? (int32_t)n0 : 0;
    if (threadIdx.x == 0) mem.active = n0;
    for (uint32_t i = threadIdx.x; i < n0; i += blockDim.x) {
        mem.f[kPix][i] = kPixNone;
        mem.f[kSample][i] = num_samples;
    }
    if constexpr (kLocal) {
        const uint32_t n16 = ((uint32_t)p.grid.region_dims[0] * (uint32_t)p.grid.region_dims[1] *
                                  (uint32_t)p.grid.region_dims[2] + 15u) / 16u;
        const uint4* src = reinterpret_cast<const uint4*>(p.grid.region_majorants);
        for (uint32_t i = threadIdx.x; i < n16; i += blockDim.x) reinterpret_cast<uint4*>(mem.regions)[i] = src[i];
    }
    __syncthreads();

    float inv1 = 0.0f, inv2 = 0.0f;
    if constexpr (kLocal) {
        inv1 = 1.0f / (float)p.grid.region_dims[1];
        inv2 = 1.0f / (float)p.grid.region_dims[2];
    }
    const bool bricks = has_bricks(p.grid);
    uint32_t paths = 0, vertices = 0, lookups = 0, scatters = 0;

    for (;;) {
        // ---- choose the kind with the most ready slots (always the fullest chunk there is)
        const int32_t my_count = lane < kWorkKinds ? __hip_atomic_load(&mem.count[lane], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP) : 0;
        uint32_t kind = 0;
        int32_t best = __builtin_amdgcn_readlane(my_count, 0);
#pragma unroll
        for (uint32_t k = 1; k < kWorkKinds; ++k) {
            const int32_t c = __builtin_amdgcn_readlane(my_count, (int)k);
            if (c > best) {
                best = c;
                kind = k;
            }
        }
        const uint32_t active = (uint32_t)__builtin_amdgcn_readfirstlane(
            (int)__hip_atomic_load(&mem.active, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP));
        if (active == 0) break;
        if (best <= 0) {
            // every slot is in another wavefront's hands: it publishes them, or retires them, when done
            __builtin_amdgcn_s_sleep(8);
            continue;
        }
        // few paths: at most twice a wavefront's share, so that every wavefront finds work
        const uint32_t even = 2u * (active + waves - 1) / waves;
        const uint32_t most = even < 64u ? even : 64u;

        // ---- claim up to `most` of its slots: every lane takes its word, ranks its bits behind the lanes'
        // before it (their counts added bit plane by bit plane), keeps those below `most` and returns the rest
        uint32_t got = __hip_atomic_exchange(&mem.ready[kind][lane], 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
        const uint32_t have = (uint32_t)__popc(got);
        uint32_t rank = 0, cnt = 0;
#pragma unroll
        for (uint32_t b = 0; b < 5; ++b) {
            const uint64_t plane = __ballot((have >> b) & 1u);
            rank += __builtin_amdgcn_mbcnt_hi((uint32_t)(plane >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)plane, 0u)) << b;
            cnt += (uint32_t)__popcll(plane) << b;
        }
        for (uint32_t slot = lane; __ballot(got != 0u && rank < most);) {
            if (got != 0u && rank < most) {
                mem.ids[wave][rank] = (uint16_t)(slot + 64u * (uint32_t)__builtin_ctz(got));
                got &= got - 1u;
                rank++;
            }
        }
        if (got != 0u)
            __hip_atomic_fetch_or(&mem.ready[kind][lane], got, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
        cnt = cnt < most ? cnt : most;
        if (cnt == 0) {
            __builtin_amdgcn_s_sleep(1);
            continue;
        }
        if (lane == 0)
            __hip_atomic_fetch_add(&mem.count[kind], -(int32_t)cnt, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "workgroup");
        const bool valid = lane < cnt;
        const uint32_t slot = valid ? mem.ids[wave][lane] : 0u;
        uint32_t next = kWorkNone;
        uint64_t fresh_params = (uint64_t)params;
        asm volatile("" : "+s"(fresh_params));
        const rtc8x_frame_params& p = *(const rtc8x_frame_params*)(ParamsPtr)fresh_params;
        const rtc8x_nrc_buffers& nb = p.nrc;
        Medium med;
        med.init(p.grid, p.density_coeff, bricks);

        auto U = [&](uint32_t f) -> uint32_t { return mem.f[f][slot]; };
        auto F = [&](uint32_t f) -> float { return __uint_as_float(mem.f[f][slot]); };
        auto SU = [&](uint32_t f, uint32_t v) { mem.f[f][slot] = v; };
        auto SF = [&](uint32_t f, float v) { mem.f[f][slot] = __float_as_uint(v); };
        auto V = [&](uint32_t f) -> V3 { return V3{F(f), F(f + 1), F(f + 2)}; };
        auto SV = [&](uint32_t f, V3 v) { SF(f, v.x); SF(f + 1, v.y); SF(f + 2, v.z); };
        auto load_rng = [&]() -> Pcg { Pcg r; r.state = ((uint64_t)U(kRngHi) << 32) | U(kRngLo); return r; };
        auto store_rng = [&](const Pcg& r) { SU(kRngLo, (uint32_t)r.state); SU(kRngHi, (uint32_t)(r.state >> 32)); };
        // the fields of a new segment; returns its region
        auto store_segment = [&](const Seg<TRACKING>& sg) -> uint32_t {
            SF(kT, sg.t);
            SF(kT1, sg.t1);
            if constexpr (kLocal) {
                SF(Lay::kTau, sg.tau);
                SV(Lay::kIv, V3{sg.s.iv0, sg.s.iv1, sg.s.iv2});
                return (uint32_t)(__mul24(__mul24(sg.s.c0, p.grid.region_dims[1]) + sg.s.c1, p.grid.region_dims[2]) + sg.s.c2);
            }
            return 0u;
        };
        // starts the segment o + t d of a path of `len` vertices; returns the kind of work that follows (`none`
        // without a segment)
        auto begin_segment = [&](Pcg& rng, V3 o, V3 d, float tmax, uint32_t len, uint32_t none) -> uint32_t {
            Seg<TRACKING> sg;
            if (!start_segment<TRACKING>(p.grid, med, sg, rng, o, d, tmax)) {
                SU(kIdxLen, len << kIdxBits);
                return none;
            }
            SU(kIdxLen, store_segment(sg) | len << kIdxBits);
            return kLocal ? kWorkWalk : kWorkLookup;
        };
        auto path_end = [&](uint32_t pix, uint32_t len, uint32_t sample, RGB c) {
            paths++;
            vertices += len;
            const size_t lin = (size_t)((pix >> 14) & 16383u) * W + (pix & 16383u);
            const bool ok = all_nonneg_finite(c);
            if constexpr (!kNrc) {
                if (ok) {
                    double* a = p.accum + 3 * lin;
                    a[0] += (double)c.r;
                    a[1] += (double)c.g;
                    a[2] += (double)c.b;
                }
            } else {
                float* pf = nb.per_frame_contribution + 3 * ((size_t)sample * p_stride + lin);
                pf[0] = ok ? c.r : 0.0f;
                pf[1] = ok ? c.g : 0.0f;
                pf[2] = ok ? c.b : 0.0f;
            }
            if (p.path_vertices) p.path_vertices[lin] += len;
        };

        if (kind == kWorkLookup || kind == kWorkWalk) {
            // ---------------------------------------------------------------- tracking and shadow steps
            uint32_t pix = 0;
            Pcg rng{0};
            float vis = 1.0f;
            bool shadow = false;
            Seg<TRACKING> sg{};
            if (valid) {
                pix = U(kPix);
                shadow = (pix & kPixShadow) != 0u;
                rng = load_rng();
                const V3 org = V(kOx);
                if (shadow) {
                    const V3 sd = V(kSx);
                    const float trace_len = 2.0f * p.world_radius;
                    sg.o = V3{org.x + trace_len * -sd.x, org.y + trace_len * -sd.y, org.z + trace_len * -sd.z};
                    sg.d = sd;
                    vis = F(kVis);
                } else {
                    sg.o = org;
                    sg.d = V(kDx);
                }
                sg.t = F(kT);
                sg.t1 = F(kT1);
            }
            uint32_t looked = 0;
            if constexpr (kLocal) {
                float mu = 0.0f, tau = 0.0f;
                enum : uint32_t { kIdle, kPending, kWalking };
                uint32_t st = kIdle, idx_len = 0;
                RegionWalk w{};
                if (valid) {
                    idx_len = U(kIdxLen);
                    w.load(p.grid, sg.o, sg.d, V(Lay::kIv), idx_len & ((1u << kIdxBits) - 1u), inv1, inv2);
                    tau = mu = F(Lay::kTau);
                    st = kind == kWorkLookup ? kPending : kWalking;
                }
                for (;;) {
                    if (st == kPending) {
                        const float sig = density_at(p.grid, med, sg.o, sg.d, sg.t);
                        looked++;
                        st = kWalking;
                        if (shadow) {
                            vis *= 1.0f - med.over(sig, mu);
                        } else if (rng.uni() < med.over(sig, mu)) {
                            st = kIdle;
                            next = kWorkScatter;
                        }
                        if (st == kWalking) tau = neg_log_1m(rng.uni());
                    }
                    // region visits until most lanes that walk have reached a collision or their end: the last
                    // fifth goes on in a later chunk (1/2, 1/4, 1/8: 35.4, 30.2, 28.6 ms per frame with 12
                    // wavefronts; with 16 and the threshold below 24.2 at 1/5, 24.5 at 1/8, 26.5 at 1/16)
                    const uint32_t walkers = (uint32_t)__popcll(__ballot(st == kWalking));
#pragma unroll 1
                    for (;;) {
                        if (st == kWalking) {
                            const int r = w.visit(p.grid, med, sg.t, sg.t1, tau, mu, mem.regions);
                            if (r == kAdvanceCollision) {
                                sg.t = sg.t + med.distance(tau, mu);
                                st = kPending;
                            } else if (r == kAdvanceEnd) {
                                st = kIdle;
                                next = shadow ? kWorkNeeDone : kWorkEscape;
                            }
                        }
                        const uint32_t left = (uint32_t)__popcll(__ballot(st == kWalking));
                        if (5u * left <= walkers) break;
                    }
                    // on with the lookups in registers while 3/8 of the lanes have one (3/4, 1/2, 3/8, 1/4: 26.9,
                    // 24.5, 24.2, 25.5 ms)
                    const uint32_t pending = (uint32_t)__popcll(__ballot(st == kPending));
                    if (8u * pending < 3u * cnt) break;
                }
                if (st == kPending) next = kWorkLookup;
                if (st == kWalking) next = kWorkWalk;
                if (valid) {
                    SU(kCost, U(kCost) + looked);
                    store_rng(rng);
                    SF(kT, sg.t);
                    if (shadow) SF(kVis, vis);
                    SF(Lay::kTau, st == kPending ? mu : tau);
                    SU(kIdxLen, w.idx | (idx_len & ~((1u << kIdxBits) - 1u)));
                }
            } else {
                Lane L;
                L.rng = rng;
                L.vis = vis;
                L.mode = valid ? (shadow ? kModeShadow : kModeTrack) : kModeIdle;
                med.lookups = 0;
                if (cnt <= kCoopClaim) {
                    coop_segments(p.grid, med, sg, L, __ballot(valid), lane);
                } else {
                    for (;;) {
                        if (L.mode == kModeTrack || L.mode == kModeShadow)
                            speculate_global<kSpeculate>(p.grid, med, sg, L, L.mode == kModeTrack);
                        const uint32_t left = (uint32_t)__popcll(__ballot(L.mode == kModeTrack || L.mode == kModeShadow));
                        if (4u * left < 3u * cnt) break;
                    }
                }
                if (valid) {
                    next = L.mode == kModeScatter ? kWorkScatter
                                                  : (L.mode == kModeEscape ? kWorkEscape
                                                                           : (L.mode == kModeNeeDone ? kWorkNeeDone : kWorkLookup));
                    SU(kCost, U(kCost) + med.lookups);
                    store_rng(L.rng);
                    SF(kT, sg.t);
                    if (shadow) SF(kVis, L.vis);
                }
            }
        } else if (kind == kWorkEscape || kind == kWorkStart) {
            // ---------------------------------------------------------------- path ends and starts
            uint32_t pix = 0, sample = 0;
            if (valid) {
                pix = U(kPix);
                sample = U(kSample);
            }
            if (kind == kWorkEscape && valid) {
                // escaped to the environment (optix_pathtracing_kernels.cu:130-174)
                const uint32_t len = U(kIdxLen) >> kIdxBits;
                RGB c{F(kCr), F(kCg), F(kCb)};
                const float tp1 = F(kTp);
                const RGB tp{tp1, tp1, tp1};
                const float prob_env = (p.sun.enabled && p.env.kind != RTC8X_ENV_NONE) ? 1.0f - p.sun.select_prob : 1.0f;
                if (p.env.kind != RTC8X_ENV_NONE) {
                    float hyp_pd;
                    const RGB radiance = env_evaluate(p.env, V(kDx), hyp_pd);
                    float mis = 1.0f;
                    if (len > 1) {
                        const float light_pd = prob_env * hyp_pd;
                        const float bsdf_pd = F(kDirPd);
                        mis = bsdf_pd * bsdf_pd / (bsdf_pd * bsdf_pd + light_pd * light_pd);
                    }
                    c = add(c, mul(tp, scale(radiance, mis)));
                }
                if constexpr (kNrc) {
                    const size_t lin = (size_t)((pix >> 14) & 16383u) * W + (pix & 16383u);
                    rtc8x_terminal_info ti;
                    ti.throughput[0] = tp.r;
                    ti.throughput[1] = tp.g;
                    ti.throughput[2] = tp.b;
                    ti.has_query = (len & 0xFFu) << 8;
                    nb.inference_terminals[(size_t)sample * p_stride + lin] = ti;
                }
                path_end(pix, len, sample, c);
                sample++;
            }
            Pcg rng{0};
            if (valid && pix != kPixNone) rng = load_rng();
            bool need = valid && sample >= num_samples, gone = false;
            if (need && pix != kPixNone) {
                const uint32_t lx = pix & 16383u, ly = (pix >> 14) & 16383u;
                p.rng_states[(size_t)ly * W + lx] = rng.state;
                const uint32_t cost = U(kCost);
                lookups += cost;
                if (p.pixel_cost) p.pixel_cost[(size_t)ly * W + lx] = cost;
            }
            const bool fresh = need;
            // the pixel of work item w
            auto take = [&](uint32_t w) {
                uint32_t lx, ly;
                bool in;
                if (p.work_order) {
                    const uint32_t lin = p.work_order[w];
                    in = lin < W * H;
                    lx = lin % W;
                    ly = lin / W;
                } else {
                    const uint32_t tile = w >> 6, within = w & 63u;
                    lx = (tile % tiles_x) * tile_w + within % tile_w;
                    ly = (tile / tiles_x) * (64u / tile_w) + within / tile_w;
                    in = lx < W && ly < H;
                }
                if (in) {
                    need = false;
                    pix = lx | ly << 14;
                }
            };
            if (need && few && pix == kPixNone) {
                const uint32_t w = (slot / kDealt * wgs + wg) * kDealt + slot % kDealt;
                if (w < total) take(w);
            }
            if (need && few) {
                need = false;
                gone = true;
            }
            // the next pixels from the work counter, one atomic per wavefront and round
            for (uint64_t ask = __ballot(need); ask; ask = __ballot(need)) {
                const uint32_t leader = (uint32_t)__ffsll((long long)ask) - 1u;
                uint32_t base = 0;
                if (lane == leader) base = atomicAdd(&g_work_counter[ctr], (uint32_t)__popcll(ask));
                base = (uint32_t)__builtin_amdgcn_readlane((int)base, (int)leader);
                if (need) {
                    const uint32_t w = base + (uint32_t)__popcll(ask & ((1ull << lane) - 1ull));
                    if (w >= total) {
                        need = false;
                        gone = true;
                    } else {
                        take(w);
                    }
                }
            }
            const uint64_t out = __ballot(gone);
            if (out && lane == 0)
                __hip_atomic_fetch_add(&mem.active, 0u - (uint32_t)__popcll(out), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
            if (valid && !gone) {
                const uint32_t lx = pix & 16383u, ly = (pix >> 14) & 16383u;
                if (fresh) {
                    rng.state = p.rng_states[(size_t)ly * W + lx];
                    sample = 0;
                    SU(kCost, 0u);
                }
                // camera ray (optix_pathtracing_kernels.cu:43-55)
                const float px = ((float)lx + rng.uni()) / (float)W;
                const float py = ((float)ly + rng.uni()) / (float)H;
                const float vh = p.camera.vh, vw = p.camera.vw;
                const float sensor_area = vw * vh;
                const V3 org{p.camera.position[0], p.camera.position[1], p.camera.position[2]};
                const V3 ldir = normalize(V3{vw * (-0.5f + px), vh * (0.5f - py), -1.0f});
                const float* M = p.camera.orientation;
                const V3 dir = normalize(V3{dot(V3{M[0], M[1], M[2]}, ldir), dot(V3{M[3], M[4], M[5]}, ldir),
                                            dot(V3{M[6], M[7], M[8]}, ldir)});
                const float az = ldir.z < 0.0f ? -ldir.z : ldir.z;
                const float dir_pd = 1.0f / (az * (az * az) * sensor_area);
                const float rinv = 1.0f / dir_pd;
                next = begin_segment(rng, org, dir, 1e10f, 1u, kWorkEscape);
                SU(kPix, pix & kPixMask);
                SU(kSample, sample);
                SV(kOx, org);
                SV(kDx, dir);
                SF(kTp, rinv);
                SV(kCr, V3{0.0f, 0.0f, 0.0f});
                SF(kDirPd, dir_pd);
                SF(kImp, luminance(RGB{rinv, rinv, rinv}));
                if constexpr (kNrc) {
                    SF(Lay::kSpread, 0.0f);
                    SF(Lay::kSpread + 1, 0.0f);
                }
                store_rng(rng);
            }
        } else if (kind == kWorkScatter) {
            // ---------------------------------------------------------------- real collisions
            if (valid) {
                // medium interaction at t (optix_pathtracing_kernels.cu:176-268)
                scatters++;
                uint32_t pix = U(kPix);
                const uint32_t len = U(kIdxLen) >> kIdxBits;
                Pcg rng = load_rng();
                const float th = F(kT);
                const V3 org = V(kOx), dir = V(kDx);
                const float tp1 = F(kTp);
                const RGB tp{tp1, tp1, tp1};
                const V3 pos{org.x + th * dir.x, org.y + th * dir.y, org.z + th * dir.z};
                const size_t lin = (size_t)((pix >> 14) & 16383u) * W + (pix & 16383u);
                float primary = 0.0f, cur = 0.0f;
                if constexpr (kNrc) {
                    // path spread (optix_pathtracing_kernels.cu:200-210)
                    primary = F(Lay::kSpread);
                    cur = F(Lay::kSpread + 1);
                    const float ddx = pos.x - org.x, ddy = pos.y - org.y, ddz = pos.z - org.z;
                    const float dist2 = ddx * ddx + ddy * ddy + ddz * ddz;
                    if (len == 1) {
                        primary = dist2 / (4.0f * RTC8X_PI_F * 1.0f);
                        SF(Lay::kSpread, primary);
                    } else {
                        cur += sqrtf(dist2 / (F(kDirPd) * 1.0f));
                        SF(Lay::kSpread + 1, cur);
                    }
                }
                // Russian roulette (optix_pathtracing_kernels.cu:254-268)
                float continue_prob = 1.0f;
                bool end = false;
                if (len > p.rr_after_path_length) {
                    const float q = luminance(tp) / F(kImp);
                    continue_prob = fminf(q, 1.0f);
                    if (rng.uni() >= continue_prob) end = true;
                }
                if constexpr (kNrc) {
                    // termination into the cache (optix_pathtracing_kernels.cu:282-330)
                    end |= cur * cur > nb.path_termination_factor * primary;
                    if (end) {
                        const uint32_t sample = U(kSample);
                        make_query(p, pos, V3{-dir.x, -dir.y, -dir.z}, &nb.inference_queries[(size_t)sample * q_stride + lin]);
                        rtc8x_terminal_info ti;
                        ti.throughput[0] = tp.r;
                        ti.throughput[1] = tp.g;
                        ti.throughput[2] = tp.b;
                        ti.has_query = 1u | ((len & 0xFFu) << 8);
                        nb.inference_terminals[(size_t)sample * p_stride + lin] = ti;
                    }
                }
                if (end) {
                    const uint32_t sample = U(kSample);
                    path_end(pix, len, sample, RGB{F(kCr), F(kCg), F(kCb)});
                    SU(kSample, sample + 1u);
                    next = kWorkStart;
                } else {
                    SF(kTp, tp1 * (1.0f / continue_prob));
                    SV(kOx, pos);
                    // NEE set-up: light choice and sample, everything of the estimate except visibility
                    const bool have_env = p.env.kind != RTC8X_ENV_NONE, have_sun = p.sun.enabled != 0;
                    const float u_light = rng.uni();
                    bool use_sun = false;
                    float prob_cur = 1.0f;
                    if (have_env && have_sun) {
                        if (u_light < p.sun.select_prob) {
                            use_sun = true;
                            prob_cur = p.sun.select_prob;
                        } else {
                            prob_cur = 1.0f - p.sun.select_prob;
                        }
                    } else if (have_sun) {
                        use_sun = true;
                    }
                    const float u0 = rng.uni();
                    const float u1 = rng.uni();
                    bool zero = !have_env && !have_sun;
                    V3 lpos{0.0f, 0.0f, 0.0f};
                    RGB emittance{0.0f, 0.0f, 0.0f};
                    float area_pd = 0.0f;
                    if (!zero) {
                        if (use_sun) {
                            lpos = V3{p.sun.direction[0], p.sun.direction[1], p.sun.direction[2]};
                            emittance = RGB{p.sun.irradiance[0], p.sun.irradiance[1], p.sun.irradiance[2]};
                        } else {
                            float ldir_pd;
                            const RGB radiance = env_sample(p.env, u0, u1, lpos, ldir_pd);
                            emittance = scale(radiance, RTC8X_PI_F);
                            area_pd = ldir_pd;
                            if (area_pd == 0.0f) zero = true;
                            area_pd *= prob_cur;
                        }
                    }
                    const V3 sdir{-lpos.x, -lpos.y, -lpos.z};
                    const float lp_cos = dot(sdir, sdir);
                    if (!zero && lp_cos <= 0.0f) zero = true;
                    if (zero) {
                        // no light: as a shadow ray that nothing came through
                        SF(kVis, 0.0f);
                        next = kWorkNeeDone;
                    } else {
                        const Frame fr = make_frame(V3{-dir.x, -dir.y, -dir.z});
                        const V3 vin = to_local(fr, V3{-sdir.x, -sdir.y, -sdir.z});
                        const float pval = phase_value(p.phase, p.scattering_forwardness, -vin.z);
                        const float alb = p.scattering_albedo;
                        const RGB fs{alb * pval, alb * pval, alb * pval};
                        RGB nee_f;
                        if (use_sun) {
                            nee_f = mul(fs, emittance);
                            SF(kK1, prob_cur);
                            pix |= kPixSun;
                        } else {
                            float bsdf_pd = pval * lp_cos / 1.0f;
                            if (!isfinite(bsdf_pd)) bsdf_pd = 0.0f;
                            const float light_pd = area_pd;
                            SF(kK1, light_pd * light_pd / (bsdf_pd * bsdf_pd + light_pd * light_pd));
                            nee_f = mul(fs, scale(emittance, 1.0f / RTC8X_PI_F));
                            SF(kK3, area_pd);
                            pix &= ~kPixSun;
                        }
                        SV(kNr, V3{nee_f.r, nee_f.g, nee_f.b});
                        SV(kSx, sdir);
                        SF(kVis, 1.0f);
                        SU(kPix, pix | kPixShadow);
                        const float trace_len = 2.0f * p.world_radius;
                        const V3 lpoint{pos.x + trace_len * -sdir.x, pos.y + trace_len * -sdir.y,
                                        pos.z + trace_len * -sdir.z};
                        next = begin_segment(rng, lpoint, sdir, trace_len, len, kWorkNeeDone);
                    }
                }
                store_rng(rng);
            }
        } else {
            // ---------------------------------------------------------------- shadow rays' ends
            if (valid) {
                // performNextEventEstimation (renderer_kernel_common.h:297-403)
                const uint32_t pix = U(kPix), len = U(kIdxLen) >> kIdxBits;
                Pcg rng = load_rng();
                const float tp1 = F(kTp);
                const RGB tp{tp1, tp1, tp1};
                RGB c{F(kCr), F(kCg), F(kCb)};
                uint32_t max_len = (!kNrc && p.max_path_length) ? p.max_path_length : kHardMaxPathLength;
                if (max_len > kHardMaxPathLength) max_len = kHardMaxPathLength;
                RGB nee_c{0.0f, 0.0f, 0.0f};
                const float vis = F(kVis);
                if (vis > 0.0f) {
                    const RGB nee_f{F(kNr), F(kNg), F(kNb)};
                    const V3 sdir = V(kSx);
                    const float k1 = F(kK1);
                    nee_c = (pix & kPixSun) ? scale(nee_f, vis / k1) : scale(nee_f, vis * k1 * dot(sdir, sdir) / F(kK3));
                }
                c = add(c, mul(tp, nee_c));
                bool end = len >= max_len;
                if (!end) {
                    // phase sampling (optix_pathtracing_kernels.cu:341-356)
                    const float us0 = rng.uni();
                    const float us1 = rng.uni();
                    V3 dl;
                    const float pdf = phase_sample(p.phase, p.scattering_forwardness, us0, us1, dl);
                    if (pdf == 0.0f) {
                        end = true;
                    } else {
                        const V3 dir = V(kDx), pos = V(kOx);
                        const Frame fr = make_frame(V3{-dir.x, -dir.y, -dir.z});
                        const float alb = p.scattering_albedo;
                        const V3 nd = from_local(fr, dl);
                        SV(kDx, nd);
                        SF(kTp, tp1 * (alb * pdf * (1.0f / pdf)));
                        SV(kCr, V3{c.r, c.g, c.b});
                        SF(kDirPd, pdf);
                        SU(kPix, pix & kPixMask);
                        next = begin_segment(rng, pos, nd, 1e10f, len + 1u, kWorkEscape);
                    }
                }
                if (end) {
                    const uint32_t sample = U(kSample);
                    path_end(pix, len, sample, c);
                    SU(kSample, sample + 1u);
                    next = kWorkStart;
                }
                store_rng(rng);
            }
        }

        // ---- publish: the fields first, then the ready bits
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup");
        if (next < kWorkKinds)
            __hip_atomic_fetch_or(&mem.ready[next][slot & 63u], 1u << (slot >> 6), __ATOMIC_RELAXED,
                                  __HIP_MEMORY_SCOPE_WORKGROUP);
        int32_t add_n = 0;
#pragma unroll
        for (uint32_t k = 0; k < kWorkKinds; ++k) {
            const int32_t n = (int32_t)__popcll(__ballot(next == k));
            if (lane == k) add_n = n;
        }
        if (add_n) __hip_atomic_fetch_add(&mem.count[lane], add_n, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
    }
    if (p.stats) {
        const uint64_t v[4] = {paths, vertices, lookups, scatters};
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            uint64_t x = v[i];
            for (int o = 32; o > 0; o >>= 1) x += __shfl_xor(x, o, 64);
            if (lane == 0) atomicAdd((unsigned long long*)&p.stats[i], (unsigned long long)x);
        }
    }
}

template <int ENTRY, int TRACKING, uint32_t REGION_BYTES, uint32_t WAVES, uint32_t SLOTS>
__global__ __launch_bounds__(64 * WAVES) void slots_kernel(const rtc8x_frame_params p, uint32_t W, uint32_t H,
                                                           uint32_t num_samples, uint32_t ctr)
{
    (void)p;  // the first kernel argument, read through the argument segment
    __shared__ SlotMem<ENTRY, TRACKING, REGION_BYTES, WAVES, SLOTS> mem;
    slots_body<ENTRY, TRACKING, REGION_BYTES, WAVES, SLOTS>((ParamsPtr)__builtin_amdgcn_kernarg_segment_ptr(), W, H, num_samples, ctr,
                                                     blockIdx.x, gridDim.x, false, mem);
}

// Several images (instances: their own volume, camera, sky, buffers and, with the NRC entry, cache buffers) in one
// persistent launch.  Workgroup b starts on the instance whose workgroup range [wg_end[i-1], wg_end[i]) holds b
// (the ranges are the caller's shares of the device, rtc8x_trace_batch); once its instance's last paths are
// done it moves on to the following instances and helps with what is left of them.
struct BatchArgs {
    const rtc8x_frame_params* params;  // device copy, count entries
    uint32_t count, ctr;               // instance i counts its work at g_work_counter[ctr + i]
    uint32_t wg_end[kMaxBatch];
    uint32_t num_samples[kMaxBatch];
};

template <int ENTRY, int TRACKING, uint32_t REGION_BYTES, uint32_t WAVES, uint32_t SLOTS>
__global__ __launch_bounds__(64 * WAVES) void slots_batch_kernel(const BatchArgs b)
{
    __shared__ SlotMem<ENTRY, TRACKING, REGION_BYTES, WAVES, SLOTS> mem;
    uint32_t first = 0;
    while (first + 1 < b.count && blockIdx.x >= b.wg_end[first]) ++first;
    for (uint32_t k = 0; k < b.count; ++k) {
        const uint32_t inst = first + k < b.count ? first + k : first + k - b.count;
        const uint32_t wg0 = inst ? b.wg_end[inst - 1] : 0u;
        const rtc8x_frame_params* pp = b.params + inst;
        slots_body<ENTRY, TRACKING, REGION_BYTES, WAVES, SLOTS>((ParamsPtr)(uint64_t)pp, pp->image_width, pp->image_height,
                                                         b.num_samples[inst], b.ctr + inst, blockIdx.x - wg0,
                                                         b.wg_end[inst] - wg0, k != 0, mem);
        __syncthreads();  // the LDS is free for the next instance
    }
}

}  // namespace dev
}  // namespace rtc8x
