// kernels.hip -- gfx950 kernels of the bead-spring MD step.
//
// Per-atom kernels run one wave64 per 64-slot tile.  Per-replica kernels run
// one workgroup (or lane) per replica.  Every kernel reads the replica's
// RepState to decide whether it has work (active / rebuild flags), so a fixed
// launch sequence can be captured once into a hipGraph and replayed while
// replicas rebuild, stop or fail independently.
//
// Step sequence (src/main.cu:403-630, one launch each, all replicas at once):
//   pre       kick + drift (+ Langevin O step, NH/NPT scaling), wrap, skin max
//   decide    per replica: rebuild if max displacement > (skin/2)^2 or every 20;
//             small replicas also sort their atoms here
//   bin/scan/scatter/rank   Morton-ordered cell sort of the larger ones
//             (rebuilding only)
//   build     Verlet list + bonded slot tables (rebuilding only)
//   force     LJ + FENE/WCA + angle, post-force kick, FP64 wave partials
//   boundary  per replica: FP64 reductions, NH chain / barostat, thermo record
#include "kernels.h"

#include <climits>

namespace fmd {

// ---------------------------------------------------------------------------
// wave64 helpers
// ---------------------------------------------------------------------------
__device__ inline int wave_in_grid() {
    return __builtin_amdgcn_readfirstlane(blockIdx.x * (blockDim.x >> 6) + (threadIdx.x >> 6));
}
__device__ inline int waves_in_grid() { return gridDim.x * (blockDim.x >> 6); }
// Workgroups are dispatched round-robin over the 8 XCDs, each with its own L2.
// Renumbering block b to (b % 8) * (G / 8) + b / 8 (for the first G - G % 8
// blocks) gives each XCD one contiguous range of tiles, so a replica's
// positions are gathered through one L2 instead of eight.
constexpr int kXcds = 8;
__device__ inline int xcd_block() {
    const int b = blockIdx.x, g = gridDim.x, g8 = g - g % kXcds;
    return b < g8 ? (b % kXcds) * (g8 / kXcds) + b / kXcds : b;
}
__device__ inline int xcd_wave_in_grid() {
    return __builtin_amdgcn_readfirstlane(xcd_block() * (blockDim.x >> 6) + (threadIdx.x >> 6));
}
__device__ inline int lane_id() { return threadIdx.x & 63; }
// set bits of m below this lane
__device__ inline int lane_prefix(unsigned long long m) {
    return (int)__builtin_amdgcn_mbcnt_hi((unsigned)(m >> 32), __builtin_amdgcn_mbcnt_lo((unsigned)m, 0u));
}

__device__ inline float wave_max(float x) {
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) x = fmaxf(x, __shfl_xor(x, o, 64));
    return x;
}
__device__ inline double wave_sum(double x) {
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) x += __shfl_xor(x, o, 64);
    return x;
}
// The sum over the wave in lane 63 (other lanes hold partial sums), by DPP
// moves on the VALU instead of LDS permutes: pairs, quads (quad_perm), 8 and
// 16 lanes (row_shr 4, 8), then rows 0+1 and 2+3 (row_bcast 15) and all four
// (row_bcast 31).  Every lane of the wave must be active.
template <int CTRL, int ROWS>
__device__ inline double dpp_move(double x) {
    const unsigned long long b = (unsigned long long)__double_as_longlong(x);
    const unsigned lo = (unsigned)__builtin_amdgcn_update_dpp(0, (int)(unsigned)b, CTRL, ROWS, 0xF, false);
    const unsigned hi = (unsigned)__builtin_amdgcn_update_dpp(0, (int)(unsigned)(b >> 32), CTRL, ROWS, 0xF, false);
    return __longlong_as_double((long long)(((unsigned long long)hi << 32) | lo));
}
__device__ inline double wave_sum_last(double x) {
    x += dpp_move<0xB1, 0xF>(x);   // quad_perm [1, 0, 3, 2]
    x += dpp_move<0x4E, 0xF>(x);   // quad_perm [2, 3, 0, 1]
    x += dpp_move<0x114, 0xF>(x);  // row_shr 4
    x += dpp_move<0x118, 0xF>(x);  // row_shr 8
    x += dpp_move<0x142, 0xA>(x);  // row_bcast 15 into rows 1 and 3
    x += dpp_move<0x143, 0xC>(x);  // row_bcast 31 into rows 2 and 3
    return x;
}
// The largest value of the wave in lane 63 (non-negative inputs: the lanes a
// DPP move leaves without a source read 0).
__device__ inline double wave_max_last(double x) {
    x = fmax(x, dpp_move<0xB1, 0xF>(x));
    x = fmax(x, dpp_move<0x4E, 0xF>(x));
    x = fmax(x, dpp_move<0x114, 0xF>(x));
    x = fmax(x, dpp_move<0x118, 0xF>(x));
    x = fmax(x, dpp_move<0x142, 0xA>(x));
    x = fmax(x, dpp_move<0x143, 0xC>(x));
    return x;
}
__device__ inline int wave_min_i(int x) {
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) x = min(x, __shfl_xor(x, o, 64));
    return x;
}
__device__ inline int wave_max_i(int x) {
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) x = max(x, __shfl_xor(x, o, 64));
    return x;
}
__device__ inline int wave_or(int x) {
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) x |= __shfl_xor(x, o, 64);
    return x;
}

// Global address-space views of descriptor pointers, so the hot loops issue
// global_load instead of flat_load.
#if defined(__HIP_DEVICE_COMPILE__)
#define FMD_GLOBAL __attribute__((address_space(1)))
#else
#define FMD_GLOBAL
#endif
template <class T> __device__ inline const FMD_GLOBAL T* gview(const T* p) {
    return (const FMD_GLOBAL T*)p;
}
// The same for stores.  A flat store also counts against the LDS wait
// counter, so a flat store ahead of LDS reads makes their wait include the
// store's trip to memory; a global store does not.
template <class T> __device__ inline FMD_GLOBAL T* gmut(T* p) { return (FMD_GLOBAL T*)p; }

constexpr int kMaxBlockK = 256;  // launch bound of k_force
constexpr int kLJChunk = 8;      // neighbors per software-pipelined chunk (kcap % 8 == 0)
constexpr int kLJTail = 4;       // rows are padded to multiples of this; a last chunk may be this short
constexpr int kBuildChunk = 8;   // list-build candidates whose loads are issued together
constexpr int kBndThreads = 256;  // workgroup of the per-replica boundary reduction
constexpr int kFusedChunks = 4;   // chunks a replica may have to be summed by that workgroup alone

#pragma clang fp contract(off)
__device__ inline float sq3(float x, float y, float z) { return x * x + y * y + z * z; }
#pragma clang fp contract(fast)

// Word 3 of a raw buffer resource on gfx9 parts: 32-bit data format, no swizzle.
constexpr int kBufferWord3 = 0x00020000;

// Indexed ("structured") buffer load of one 16-byte record: the resource
// carries the stride, the hardware forms index * stride (buffer_load_dwordx4
// ... idxen), and an index at or past the record count reads zeros.
typedef unsigned u32x4 __attribute__((ext_vector_type(4)));
__device__ u32x4 struct_load_b128(__amdgpu_buffer_rsrc_t rsrc, unsigned vindex, unsigned voffset,
                                  unsigned soffset, int aux) __asm("llvm.amdgcn.struct.ptr.buffer.load.v4i32");

// ---------------------------------------------------------------------------
// FP64 Nose-Hoover chain (src/integrate/nose_hoover.cu:86-178 / :356-447) and
// NPT barostat (src/integrate/nose_hoover.cu:185-305), one lane per replica.
// ---------------------------------------------------------------------------
// The chain's loops are unrolled to kMaxChain under uniform conditions, so its
// variables are registers (indexed at run time they would live in scratch).
__device__ double nh_chain(RepState* st, double KE, double kT, int natoms, double half_dt) {
    const int M = st->M;
    double xi[kMaxChain], v[kMaxChain], dd[kMaxChain];
#pragma unroll
    for (int k = 0; k < kMaxChain; k++) { xi[k] = st->xi[k]; v[k] = st->vxi[k]; dd[k] = 0.0; }
    const double Nf = 3.0 * (double)natoms, Q1 = st->Q1, Qr = st->Qr;
    const double dt2 = half_dt, dt4 = 0.5 * half_dt, dt8 = 0.25 * half_dt;
    double T = 2.0 * KE / Nf;
    if (Q1 > 0.0) dd[0] = (Nf * T - Nf * kT) / Q1;
#pragma unroll
    for (int ich = kMaxChain - 1; ich > 0; ich--)
        if (ich < M) {
            double e = 1.0;
            if (ich + 1 < kMaxChain && ich + 1 < M) e = exp(-dt8 * v[min(ich + 1, kMaxChain - 1)]);
            v[ich] = (v[ich] * e + dd[ich] * dt4) * e;
        }
    double e0 = (M > 1) ? exp(-dt8 * v[1]) : 1.0;
    v[0] = (v[0] * e0 + dd[0] * dt4) * e0;
    double scale = exp(-dt2 * v[0]);
    T *= scale * scale;
    if (Q1 > 0.0) dd[0] = (Nf * T - Nf * kT) / Q1;
#pragma unroll
    for (int k = 0; k < kMaxChain; k++)
        if (k < M) xi[k] += dt2 * v[k];
    v[0] = (v[0] * e0 + dd[0] * dt4) * e0;
#pragma unroll
    for (int ich = 1; ich < kMaxChain; ich++)
        if (ich < M) {
            double e = 1.0;
            if (ich + 1 < kMaxChain && ich + 1 < M) e = exp(-dt8 * v[min(ich + 1, kMaxChain - 1)]);
            double Qp = (ich == 1) ? Q1 : Qr;
            dd[ich] = (Qp * v[ich - 1] * v[ich - 1] - kT) / Qr;
            v[ich] = (v[ich] * e + dd[ich] * dt4) * e;
        }
#pragma unroll
    for (int k = 0; k < kMaxChain; k++) { st->xi[k] = xi[k]; st->vxi[k] = v[k]; }
    return scale;
}

struct BaroOut {
    double L, baro_scale, exp_vW, veps_W_dt, nh_scale, KE_scaled;
};
__device__ BaroOut npt_chain_baro(RepState* st, double KE, double vir_trace, bool advance,
                                  double kT, double Pt, int natoms, double half_dt, double dt) {
    BaroOut o;
    const double Nf = 3.0 * (double)natoms;
    double V = st->V0 * exp(3.0 * st->eps);
    if (advance) {
        double P = (2.0 * KE + vir_trace) / (3.0 * V);
        double cb = cbrt(2.0);
        double w[3] = {1.0 / (2.0 - cb), -cb / (2.0 - cb), 1.0 / (2.0 - cb)};
        for (int s = 0; s < 3; s++) {
            double ws = w[s] * dt;
            double dv = 3.0 * V * (P - Pt) * ws;
            double vh = st->veps + 0.5 * dv;
            st->eps += vh * ws / st->W;
            dv = 3.0 * st->V0 * exp(3.0 * st->eps) * (P - Pt) * ws;
            st->veps += dv;
        }
        V = st->V0 * exp(3.0 * st->eps);
    }
    o.L = cbrt(V);
    double vW = st->veps / st->W;
    o.baro_scale = exp(-(1.0 + 3.0 / Nf) * vW * half_dt);
    o.exp_vW = exp(vW * dt);
    o.veps_W_dt = vW * dt;
    o.KE_scaled = KE * o.baro_scale * o.baro_scale;
    o.nh_scale = nh_chain(st, o.KE_scaled, kT, natoms, half_dt);
    return o;
}

__device__ inline double sinch(double x) {
    if (fabs(x) < 1e-6) return 1.0 + x * x / 6.0;
    return sinh(x) / x;
}

// Cell grid of the current box (src/neighbor/verlet_list.cu:8-13), recomputed
// at every rebuild so the grid follows the box under NPT.
__device__ void set_grid(const RepDesc& d, RepState* st) {
    int n = (int)(st->Lp / d.rcs);
    int nx = n < 1 ? 1 : n;
    float cs = st->Lp / (float)nx;
    int cb = 0;
    while ((1 << cb) < nx) cb++;
    if ((1 << (3 * cb)) > d.ncell_cap) {
        st->err |= ERR_CELL;
        st->active = 0;
        return;
    }
    st->nx = nx;
    st->inv_cs = 1.0f / cs;
    st->cbits = cb;
}

// Start-of-step scalars for step s (T/P ramp, NH chain, barostat factors).
__device__ void start_step(const RepDesc& d, RepState* st, int64_t s) {
    float frac = (float)(s - 1) / (float)st->ramp_n;  // src/main.cu:407-409
    float T = (float)st->T_start + ((float)st->T_stop - (float)st->T_start) * frac;
    float P = (float)st->P_start + ((float)st->P_stop - (float)st->P_start) * frac;
    const double hdt = 0.5 * (double)d.dt, dt = (double)d.dt;
    // observables on NPT steps (the barostat needs the virial), thermo steps and
    // the last step of a run (its result is read back)
    st->want_obs = (d.ensemble == 2) || (st->thermo_freq > 0 && (s % st->thermo_freq) == 0) ||
                   (st->stress_freq > 0 && (s % st->stress_freq) == 0) || (s == st->stop);
    if (d.ensemble == 0) {
        st->kT = T;
        st->vscale = 1.0f;
    } else if (d.ensemble == 1) {
        double nh = nh_chain(st, st->ke_carry, (double)T, d.natoms, hdt);
        st->vscale = (float)((double)st->v_pending * nh);
    } else {
        BaroOut o = npt_chain_baro(st, st->ke_carry, 0.0, false, (double)T, (double)P, d.natoms,
                                   hdt, dt);
        st->vscale = (float)((double)st->v_pending * o.nh_scale * o.baro_scale);
        st->exp_vW = (float)o.exp_vW;
        double h = 0.5 * o.veps_W_dt;
        st->fpos = (float)(dt * exp(h) * sinch(h));
        st->L = (float)o.L;
        st->invL = 1.0f / st->L;
    }
    st->pre_ready = 1;
}

// Push-off speed limit (the displacement cap of a soft push-off): rescales v
// so that |v| <= vlim.
__device__ inline float4 limit_speed(float4 v, float vlim) {
    const float s2 = v.x * v.x + v.y * v.y + v.z * v.z;
    if (s2 > vlim * vlim) {
        const float f = vlim * rsqrtf(s2);
        v.x *= f; v.y *= f; v.z *= f;
    }
    return v;
}

// ---------------------------------------------------------------------------
// pre-force: kick, drift, (O), wrap, image, skin displacement
// (src/integrate/langevin.cu:34-94, src/integrate/nose_hoover.cu:606-757,
//  src/neighbor/skin_trigger.cuh:5-16)
// ---------------------------------------------------------------------------
__global__ void __launch_bounds__(256) k_pre(const RepDesc* __restrict__ descs,
                                             const Tile* __restrict__ tiles, int ntl, int* __restrict__ nrt) {
    if (blockIdx.x == 0 && threadIdx.x == 0) *nrt = 0;  // k_decide lists this step's rebuilding tiles
    const int w = wave_in_grid();
    if (w >= ntl) return;
    const Tile t = tiles[w];
    const RepDesc& d = descs[t.rep];
    RepState* st = d.st;
    if (!st->active || st->err) return;
    const int i = t.lt * kTile + lane_id();
    float d2 = 0.0f;
    int bad = 0;
    if (i < d.natoms) {
        float4 r = d.pos[i], v = d.vel[i];
        float4 ref = d.pos_ref[i];
        const float m = d.mass[type_of(r.w)];
        const float hdtm = d.half_dt / m;
        const float L = st->L, invL = st->invL;
        if (d.ensemble == 0) {
            if (!st->kicked) {  // else the last force pass gave this half kick
                const float4 f = d.force[i];
                // explicit FMAs: the force kernel's kick ahead computes the same bits
                v.x = fmaf(hdtm, f.x, v.x); v.y = fmaf(hdtm, f.y, v.y); v.z = fmaf(hdtm, f.z, v.z);
                if (d.vlim > 0.0f) v = limit_speed(v, d.vlim);
            }
            r.x += d.half_dt * v.x; r.y += d.half_dt * v.y; r.z += d.half_dt * v.z;
            const float3 z = normal3(d.seed_lo, d.seed_hi, (uint32_t)d.gid[i], st->step + 1);
            const float ns = d.c2 * sqrtf(st->kT / m);
            v.x = d.c1 * v.x + ns * z.x; v.y = d.c1 * v.y + ns * z.y; v.z = d.c1 * v.z + ns * z.z;
            if (d.vlim > 0.0f) v = limit_speed(v, d.vlim);
            r.x += d.half_dt * v.x; r.y += d.half_dt * v.y; r.z += d.half_dt * v.z;
        } else {
            const float sc = st->vscale;
            const float4 f = d.force[i];
            v.x *= sc; v.y *= sc; v.z *= sc;
            v.x += hdtm * f.x; v.y += hdtm * f.y; v.z += hdtm * f.z;
            if (d.ensemble == 1) {
                r.x += d.dt * v.x; r.y += d.dt * v.y; r.z += d.dt * v.z;
            } else {
                const float ew = st->exp_vW, fp = st->fpos;
                r.x = r.x * ew + v.x * fp; r.y = r.y * ew + v.y * fp; r.z = r.z * ew + v.z * fp;
                ref.x *= ew; ref.y *= ew; ref.z *= ew;
                d.pos_ref[i] = ref;
            }
        }
        const int ix = (int)floorf(r.x * invL), iy = (int)floorf(r.y * invL),
                  iz = (int)floorf(r.z * invL);
        r.x -= (float)ix * L; r.y -= (float)iy * L; r.z -= (float)iz * L;

        float dx = r.x - ref.x, dy = r.y - ref.y, dz = r.z - ref.z;
        dx -= L * roundf(dx * invL); dy -= L * roundf(dy * invL); dz -= L * roundf(dz * invL);
        d2 = dx * dx + dy * dy + dz * dz;
        bad = !(isfinite(r.x) && isfinite(r.y) && isfinite(r.z) && isfinite(v.x) &&
                isfinite(v.y) && isfinite(v.z));
        d.pos[i] = r;
        d.vel[i] = v;
        if (ix | iy | iz) {  // image counts change only on a wrap
            int4 im = d.img[i];
            im.x += ix; im.y += iy; im.z += iz;
            d.img[i] = im;
        }
        const double sc = 4294967296.0 / (double)L;
        d.ipos[i] = make_int4((int)fix_coord(r.x, sc), (int)fix_coord(r.y, sc), (int)fix_coord(r.z, sc),
                              __float_as_int(r.w));
    }
    // the tile's largest squared displacement since the last rebuild (-1: a
    // non-finite position or velocity), reduced per replica by k_decide; a
    // per-tile record instead of an atomic on one word per replica, which
    // serializes a large replica's waves
    const float m = wave_max(bad ? 0.0f : d2);
    const int b = wave_or(bad);
    if (lane_id() == 0) d.tdisp[t.lt] = b ? -1.0f : m;
}

// ---------------------------------------------------------------------------
// The Morton-ordered cell sort (below, k_bin to k_rank) of one replica by one
// workgroup of 1024 threads: the same order, in one kernel and with the cell
// counts in LDS, two 16-bit counts a word (at most kWgSortKeys cell keys; the
// engine lets it sort kSortInDecide atoms at most).  One CU moves the replica's
// state, so its time grows with the atoms, while the four kernels cost their
// launches on every step, rebuilding or not (1.5 us each).
// ---------------------------------------------------------------------------
constexpr int kSortThreads = 1024;
constexpr int kWgSortNear = 16384;
// a 16-byte record of any of the state arrays, moved as it is
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef float f32x2 __attribute__((ext_vector_type(2)));
template <class T> __device__ inline FMD_GLOBAL f32x4* raw4(T* p) { return (FMD_GLOBAL f32x4*)p; }
struct SortLds {
    unsigned h[kWgSortKeys / 2];       // counts, then first slots, of keys 2k and 2k + 1
    int wsum[kSortThreads / 64];
    int sx[kWgSortNear];               // the atoms' x sort keys in cell order
    unsigned lo[32];                   // lower bound floor(c 2^32 / nx) of each cell coordinate
};
__device__ void sort_wg(const RepDesc& d, int nx, float ics, int cbits, float Lp, SortLds& s) {
    const int tid = threadIdx.x, n = d.natoms, nkeys = 1 << (3 * cbits), nw = max(nkeys >> 1, 1);
    for (int j = tid; j < nw; j += kSortThreads) s.h[j] = 0u;
    if (tid < nx) s.lo[tid] = (unsigned)(((unsigned long long)tid << 32) / (unsigned)nx);
    __syncthreads();
    const double sc = 4294967296.0 / (double)Lp;
    // kB atoms per thread and pass, their loads in flight together
    constexpr int kB = 4;
    for (int i0 = tid; i0 < n; i0 += kB * kSortThreads) {
        f32x4 r[kB], v[kB], im[kB];
#pragma unroll
        for (int k = 0; k < kB; k++) {
            const int i = min(i0 + k * kSortThreads, n - 1);
            r[k] = raw4(d.pos)[i];
            v[k] = raw4(d.vel)[i];
            im[k] = raw4(d.img)[i];
        }
#pragma unroll
        for (int k = 0; k < kB; k++) {
            const int i = i0 + k * kSortThreads;
            if (i < n) {
                const int cx = cell_coord(r[k].x, ics, nx);
                const int key = (int)cell_key(cx, cell_coord(r[k].y, ics, nx), cell_coord(r[k].z, ics, nx));
                const int sh = (key & 1) * 16;
                gmut(d.rank)[i] = (int)((atomicAdd(&s.h[key >> 1], 1u << sh) >> sh) & 0xFFFFu);
                gmut(d.cell_of)[i] = key;
                gmut(d.sortx)[i] = (int)(fix_coord(r[k].x, sc) - s.lo[cx]);
                raw4(d.tmp_pos)[i] = r[k];
                raw4(d.tmp_vel)[i] = v[k];
                raw4(d.tmp_img)[i] = im[k];
            }
        }
    }
    __syncthreads();
    {  // exclusive scan of the counts; thread t holds the words [t per, (t + 1) per)
        const int per = (nw + kSortThreads - 1) / kSortThreads, w0 = tid * per, lane = lane_id();
        int sum = 0;
        for (int w = w0; w < min(w0 + per, nw); w++) sum += (int)(s.h[w] & 0xFFFFu) + (int)(s.h[w] >> 16);
        int x = sum;
#pragma unroll
        for (int o = 1; o < 64; o <<= 1) {
            const int y = __shfl_up(x, o, 64);
            if (lane >= o) x += y;
        }
        if (lane == 63) s.wsum[tid >> 6] = x;
        __syncthreads();
        int run = x - sum;
        for (int w = 0; w < (tid >> 6); w++) run += s.wsum[w];
        for (int w = w0; w < min(w0 + per, nw); w++) {
            const unsigned c = s.h[w];
            const int a = run, b = run + (int)(c & 0xFFFFu);
            run = b + (int)(c >> 16);
            s.h[w] = (unsigned)a | (unsigned)b << 16;
            gmut(d.cell_start)[2 * w] = a;
            gmut(d.cell_start)[2 * w + 1] = b;
        }
        if (tid == 0) gmut(d.cell_start)[nkeys] = n;
    }
    __syncthreads();
    auto first = [&](int key) { return (int)((s.h[key >> 1] >> ((key & 1) * 16)) & 0xFFFFu); };
    const bool near = n <= kWgSortNear;  // the sort keys in LDS, else in order2
    for (int i0 = tid; i0 < n; i0 += kB * kSortThreads) {
        int key[kB], rk[kB], sx[kB];
#pragma unroll
        for (int k = 0; k < kB; k++) {
            const int i = min(i0 + k * kSortThreads, n - 1);
            key[k] = gview(d.cell_of)[i];
            rk[k] = gview(d.rank)[i];
            sx[k] = gview(d.sortx)[i];
        }
#pragma unroll
        for (int k = 0; k < kB; k++) {
            const int i = i0 + k * kSortThreads;
            if (i < n) {
                const int dst = first(key[k]) + rk[k];
                gmut(d.order)[dst] = i;
                if (near) s.sx[dst] = sx[k];
                else gmut(d.order2)[dst] = sx[k];
            }
        }
    }
    __syncthreads();
    // rank inside the cell by x, then global id, and the move to the final slot
    auto sx = [&](int c) __attribute__((always_inline)) { return near ? s.sx[c] : gview(d.order2)[c]; };
    auto move = [&](int q, int key, f32x4 p, f32x4 v, f32x4 im) __attribute__((always_inline)) {
        const int b = first(key), e = key + 1 < nkeys ? first(key + 1) : n, rx = sx(q);
        const int gid = __float_as_int(im[3]);
        int to = b;
        for (int c = b; c < e; c++) {
            const int rc = sx(c);
            to += (rc < rx) || (rc == rx && c != q && gview(d.tmp_img)[gview(d.order)[c]].w < gid);
        }
        raw4(d.pos)[to] = p;
        raw4(d.pos_ref)[to] = p;
        raw4(d.vel)[to] = v;
        raw4(d.img)[to] = im;
        gmut(d.gid)[to] = gid;
        gmut(d.slot_of)[gid] = to;
        raw4(d.ipos)[to] = f32x4{__uint_as_float(fix_coord(p.x, sc)), __uint_as_float(fix_coord(p.y, sc)),
                                 __uint_as_float(fix_coord(p.z, sc)), p.w};
    };
    for (int q0 = tid; q0 < n; q0 += 2 * kSortThreads) {  // two atoms, their loads in flight together
        const int q1 = q0 + kSortThreads;
        const int s0 = gview(d.order)[q0], s1 = gview(d.order)[min(q1, n - 1)];
        const int k0 = gview(d.cell_of)[s0], k1 = gview(d.cell_of)[s1];
        const f32x4 p0 = raw4(d.tmp_pos)[s0], p1 = raw4(d.tmp_pos)[s1];
        const f32x4 v0 = raw4(d.tmp_vel)[s0], v1 = raw4(d.tmp_vel)[s1];
        const f32x4 m0 = raw4(d.tmp_img)[s0], m1 = raw4(d.tmp_img)[s1];
        move(q0, k0, p0, v0, m0);
        if (q1 < n) move(q1, k1, p1, v1, m1);
    }
}

// ---------------------------------------------------------------------------
// per-replica rebuild decision (src/main.cu:486-496, skin_trigger.cuh:18-33),
// with SORT also the cell sort of a replica that rebuilds
// ---------------------------------------------------------------------------
template <bool SORT>
__global__ void __launch_bounds__(1024) k_decide(const RepDesc* __restrict__ descs,
                                                 const int* __restrict__ reps, int nr,
                                                 const int* __restrict__ rep_t0, int* __restrict__ rlist,
                                                 int* __restrict__ nrt) {
    __shared__ float s_max[16];
    __shared__ int s_bad[16];
    __shared__ int s_base, s_nx, s_cb;
    __shared__ float s_ics, s_L;
    const RepDesc& d = descs[reps[blockIdx.x]];
    RepState* st = d.st;
    if (!st->active) return;
    float m = 0.0f;
    int bad = 0;
    for (int tl = threadIdx.x; tl < d.ntiles; tl += blockDim.x) {
        const float x = d.tdisp[tl];
        bad |= (x < 0.0f);
        m = fmaxf(m, x);
    }
    m = wave_max(m);
    bad = wave_or(bad);
    if (lane_id() == 0) {
        s_max[threadIdx.x >> 6] = m;
        s_bad[threadIdx.x >> 6] = bad;
    }
    __syncthreads();
    if (threadIdx.x == 0) {
        s_base = -1;
        for (int w = 1; w < (int)(blockDim.x >> 6); w++) {
            m = fmaxf(m, s_max[w]);
            bad |= s_bad[w];
        }
        m = fmaxf(m, s_max[0]);
        bad |= s_bad[0];
        if (bad) st->err |= ERR_NAN;
        if (st->err) {
            st->active = 0;
            st->rebuild = 0;
        } else {
            // k_pre of this step placed the positions in the box st->L
            st->Lp = st->L;
            st->invLp = st->invL;
            set_grid_consts(st, d.rc2);
            const float md = fmaxf(__int_as_float(st->maxdisp_bits), m);  // largest since the last rebuild
            const int since = st->since_rebuild + 1;
            const int rb = (md > d.half_skin2) || (since >= kRebuildEvery);
            st->rebuild = rb;
            if (rb) {
                st->since_rebuild = 0;
                st->maxdisp_bits = 0;
                st->nrebuilds++;
                set_grid(d, st);
                if (st->err) {  // the box outgrew the cell arrays: the replica has stopped
                    st->rebuild = 0;
                } else {
                    s_nx = st->nx; s_cb = st->cbits; s_ics = st->inv_cs; s_L = st->Lp;
                    s_base = atomicAdd(nrt, d.ntiles);  // this replica's run of the rebuild tile list
                }
            } else {
                st->since_rebuild = since;
                st->maxdisp_bits = __float_as_int(md);
            }
        }
    }
    __syncthreads();
    // the replica's tiles in the rebuild tile list (whole groups, in any
    // order of replicas: every consumer treats each group alone)
    const int base = s_base;
    if (base >= 0)
        for (int k = threadIdx.x; k < d.ntiles; k += blockDim.x) rlist[base + k] = rep_t0[blockIdx.x] + k;
    if constexpr (SORT) {
        __shared__ SortLds s_sort;
        if (base >= 0) sort_wg(d, s_nx, s_ics, s_cb, s_L, s_sort);
    }
}

// Radius of gyration of each chain (src/analysis/rg.cu:3-69): unwrapped
// positions x + image * L over the chain's beads (global-id order, through
// slot_of), centre of mass, then sqrt of the mean squared distance from it.
// One wave per chain, FP64 sums by wave shuffles.
__global__ void __launch_bounds__(64) k_rg(const RepDesc* __restrict__ d, double* __restrict__ out) {
    const int c = blockIdx.x;
    if (c >= d->nchains) return;
    const int g0 = d->t_choff[c], g1 = d->t_choff[c + 1], len = g1 - g0;
    const double L = (double)d->st->Lp;
    double sx = 0.0, sy = 0.0, sz = 0.0;
    for (int g = g0 + lane_id(); g < g1; g += 64) {
        const int q = d->slot_of[g];
        const float4 p = d->pos[q];
        const int4 im = d->img[q];
        sx += (double)p.x + im.x * L; sy += (double)p.y + im.y * L; sz += (double)p.z + im.z * L;
    }
    const double cx = wave_sum(sx) / len, cy = wave_sum(sy) / len, cz = wave_sum(sz) / len;
    double r2 = 0.0;
    for (int g = g0 + lane_id(); g < g1; g += 64) {
        const int q = d->slot_of[g];
        const float4 p = d->pos[q];
        const int4 im = d->img[q];
        const double dx = (double)p.x + im.x * L - cx, dy = (double)p.y + im.y * L - cy,
                     dz = (double)p.z + im.z * L - cz;
        r2 += dx * dx + dy * dy + dz * dz;
    }
    r2 = wave_sum(r2);
    if (lane_id() == 0) out[c] = sqrt(r2 / len);
}

// Mean of the per-chain values k_rg wrote to vals, summed in chain order by
// one lane (the order the host sum of the per-chain read uses).
__global__ void __launch_bounds__(64) k_rg_mean(const RepDesc* __restrict__ d, const double* __restrict__ vals,
                                                double* __restrict__ out) {
    if (threadIdx.x != 0) return;
    const int nc = d->nchains;
    double s = 0.0;
    for (int c = 0; c < nc; c++) s += vals[c];
    out[0] = nc > 0 ? s / nc : 0.0;
}

// Status of each listed replica for one host read per batch.
__global__ void k_status(const RepDesc* __restrict__ descs, const int* __restrict__ reps, int nr,
                         int4* __restrict__ out) {
    const int k = blockIdx.x * blockDim.x + threadIdx.x;
    if (k >= nr) return;
    const RepState* st = descs[reps[k]].st;
    const uint64_t s = (uint64_t)st->step;
    out[k] = make_int4(st->err, st->active, (int)(uint32_t)s, (int)(uint32_t)(s >> 32));
}

// Steps since each listed replica's last list build (-1: inactive), for the
// host's choice of step structure.
__global__ void k_phase(const RepDesc* __restrict__ descs, const int* __restrict__ reps, int nr,
                        int* __restrict__ out) {
    const int k = blockIdx.x * blockDim.x + threadIdx.x;
    if (k >= nr) return;
    const RepState* st = descs[reps[k]].st;
    out[k] = st->active ? st->since_rebuild : -1;
}

// Host-requested state changes.
__global__ void k_control(const RepDesc* __restrict__ descs, const int* __restrict__ reps, int nr,
                          int op, int64_t arg) {
    const int k = blockIdx.x * blockDim.x + threadIdx.x;
    if (k >= nr) return;
    const RepDesc& d = descs[reps[k]];
    RepState* st = d.st;
    if (op == CTL_RUN) {
        st->stop = st->step + arg;
        st->active = (st->err == 0 && arg > 0) ? 1 : 0;
    } else if (op == CTL_FORCE_REBUILD) {
        st->rebuild = 1;
        st->since_rebuild = 0;
        st->maxdisp_bits = 0;
        st->nrebuilds++;
        set_grid(d, st);
    }
}

// ---------------------------------------------------------------------------
// Morton-ordered cell sort.  Cells have side >= rc+skin on the reference grid;
// the cell key is the 3-D Morton interleave of the cell coordinates, so the
// slot order is a Morton curve over cells, and within a cell atoms are ordered
// by their grid coordinate along x, then global id (deterministic; the list
// build searches a cell's atoms by x).
// ---------------------------------------------------------------------------
// The rebuild kernels walk the batch's compact list of rebuilding tiles
// (k_rebuild_list), so their cost follows the replicas that rebuild.
#define REBUILD_PROLOGUE                                      \
    const Tile t = tiles[rlist[v]];                           \
    const RepDesc& d = descs[t.rep];                          \
    RepState* st = d.st;                                      \
    (void)st;                                                 \
    const int i = t.lt * kTile + lane_id();
#define REBUILD_LOOP for (int v = wave_in_grid(), nv = *nrt; v < nv; v += waves_in_grid())
#define REBUILD_ARGS const RepDesc* __restrict__ descs, const Tile* __restrict__ tiles, \
                     const int* __restrict__ rlist, const int* __restrict__ nrt

// Compact list of the tiles of rebuilding replicas (all replicas if `always`):
// one workgroup scans the per-replica tile counts and writes tile indices.
__global__ void __launch_bounds__(1024) k_rebuild_list(const RepDesc* __restrict__ descs,
                                                       const int* __restrict__ reps,
                                                       const int* __restrict__ rep_t0, int nr,
                                                       int always, int* __restrict__ rlist,
                                                       int* __restrict__ nrt) {
    __shared__ int wsum[16];
    __shared__ int s_off[kMaxReplicas];  // exclusive prefix of the listed tile counts
    __shared__ int s_carry;
    const int lane = lane_id(), wv = threadIdx.x >> 6;
    if (threadIdx.x == 0) s_carry = 0;
    __syncthreads();
    // one replica per thread and pass, a block prefix per pass of 1024
    for (int r0 = 0; r0 < nr; r0 += 1024) {
        const int r = r0 + threadIdx.x;
        int c = 0;
        if (r < nr) {
            const RepDesc& d = descs[reps[r]];
            const RepState* st = d.st;
            if (always || (st->active && st->rebuild)) c = d.ntiles;
        }
        int x = c;
#pragma unroll
        for (int o = 1; o < 64; o <<= 1) {
            const int y = __shfl_up(x, o, 64);
            if (lane >= o) x += y;
        }
        if (lane == 63) wsum[wv] = x;
        __syncthreads();
        int before = 0, all = 0;
        for (int w = 0; w < 16; w++) {
            const int ws = wsum[w];
            before += (w < wv) ? ws : 0;
            all += ws;
        }
        const int carry = s_carry;
        if (r < nr) s_off[r] = carry + before + x - c;
        __syncthreads();
        if (threadIdx.x == 0) s_carry = carry + all;
        __syncthreads();
    }
    const int total = s_carry;
    if (threadIdx.x == 0) *nrt = total;
    // each wave writes the tiles of replicas wv, wv + 16, ... (coalesced runs)
    for (int r = wv; r < nr; r += 16) {
        const int o = s_off[r];
        const int n = ((r + 1 < nr) ? s_off[r + 1] : total) - o;
        if (n == 0) continue;
        const int t0 = rep_t0[r];
        for (int v = lane; v < n; v += 64) rlist[o + v] = t0 + v;
    }
}

// Cell key of each atom and a unique position inside its cell.  The lanes of
// a wave (Morton-sorted atoms) fall in a few cells: one atomic per distinct
// key and wave reserves the positions, handed out in lane order.
__global__ void __launch_bounds__(256) k_bin(REBUILD_ARGS) {
    REBUILD_LOOP {
        REBUILD_PROLOGUE
        const bool valid = i < d.natoms;
        uint32_t key = 0xffffffffu;
        if (valid) {
            const float4 r = d.pos[i];
            const int nx = st->nx;
            const float ics = st->inv_cs;
            const int cx = cell_coord(r.x, ics, nx);
            key = cell_key(cx, cell_coord(r.y, ics, nx), cell_coord(r.z, ics, nx));
            d.cell_of[i] = (int)key;
            // the within-cell sort key (k_rank): the x grid coordinate
            // floor(x 2^32 / L) modulo 2^32, relative to the cell's lower bound
            // floor(cx 2^32 / nx)
            const unsigned lo = (unsigned)(((unsigned long long)cx << 32) / (unsigned)nx);
            d.sortx[i] = (int)(fix_coord(r.x, 4294967296.0 / (double)st->Lp) - lo);
        }
        unsigned long long todo = __ballot(valid);
        while (todo) {  // wave-uniform: one pass per distinct key
            const int lead = __builtin_ctzll(todo);
            const uint32_t k = __shfl(key, lead, 64);
            const unsigned long long same = __ballot(valid && key == k);
            int base = 0;
            if (lane_id() == lead) base = atomicAdd(&d.cell_cnt[k], __popcll(same));
            base = __shfl(base, lead, 64);
            if (valid && key == k) d.rank[i] = base + lane_prefix(same);
            todo &= ~same;
        }
    }
}

// Exclusive scan of the cell counts (k_scatter clears them for the next
// rebuild).  Workgroup (replica, y) of 1024 threads scans a run of keys in
// passes of kScanKeys, four consecutive ones a thread, from the sum of all the
// counts before it.  With up to kScanBlocks workgroups it forms that sum itself
// (1M beads, 262,144 keys: 195.5 us per step; one workgroup that carries the sum
// through all keys 200.1).  What is read so grows with the square of the keys,
// so for boxes of more keys the runs' totals are formed first (k_scan_totals,
// into the replica's `order`, which the sort writes later) and each workgroup
// sums those.  A list rebuild of 4,000 beads by one workgroup / by 64 / with
// totals: 2,097,152 keys 910 / 317 / 132 us, 16.8M 6.2 / 1.6 / 0.27 ms.
constexpr int kScanKeys = 4096;
constexpr int kScanBlocks = 64;   // workgroups a replica without totals
constexpr int kScanTotals = 256;  // and with: `order` holds at least a group's slots
static_assert(kScanTotals <= kGroupSlots, "a replica has at least a group of slots");
__device__ inline int scan_run(int nkeys) {  // keys of one workgroup
    const int pass = (int)gridDim.y * kScanKeys;
    return (nkeys + pass - 1) / pass * kScanKeys;
}
typedef int i32x4 __attribute__((ext_vector_type(4)));
__global__ void __launch_bounds__(1024) k_scan_totals(const RepDesc* __restrict__ descs,
                                                      const int* __restrict__ reps, int nr, int always) {
    __shared__ int wsum[16];
    const RepDesc& d = descs[reps[blockIdx.x]];
    const RepState* st = d.st;
    if (!always && !(st->active && st->rebuild)) return;
    const int nkeys = 1 << (3 * st->cbits), run = scan_run(nkeys), k0 = blockIdx.y * run;
    if (k0 >= nkeys || nkeys < 4) return;  // 1 key, or a multiple of 4
    const FMD_GLOBAL int* cnt = gview(d.cell_cnt);
    const int end = min(k0 + run, nkeys);
    int sum = 0;
#pragma unroll 4
    for (int k = k0 + 4 * threadIdx.x; k < end; k += kScanKeys) {
        const i32x4 v = *(const FMD_GLOBAL i32x4*)(cnt + k);
        sum += v.x + v.y + v.z + v.w;
    }
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) sum += __shfl_xor(sum, o, 64);
    if (lane_id() == 0) wsum[threadIdx.x >> 6] = sum;
    __syncthreads();
    if (threadIdx.x == 0) {
        int total = 0;
#pragma unroll
        for (int w = 0; w < 16; w++) total += wsum[w];
        gmut(d.order)[blockIdx.y] = total;
    }
}
// ONE: no workgroup has more than one pass.  At most 40 VGPRs: in the forked step
// a workgroup waits for its 16 waves' registers to come free beside the force
// pass (256 replicas: 33 us with 33 VGPRs, 167 with 50).
template <bool ONE, bool TOTALS>
__global__ void __launch_bounds__(1024) k_scan(const RepDesc* __restrict__ descs,
                                               const int* __restrict__ reps, int nr, int always) {
    __shared__ int wsum[16], wbase[16];
    const RepDesc& d = descs[reps[blockIdx.x]];
    RepState* st = d.st;
    if (!always && !(st->active && st->rebuild)) return;
    const int nkeys = 1 << (3 * st->cbits), run = scan_run(nkeys), k0 = blockIdx.y * run;
    if (k0 >= nkeys) return;
    const int lane = lane_id(), wv = threadIdx.x >> 6, end = min(k0 + run, nkeys);
    const FMD_GLOBAL int* cnt = gview(d.cell_cnt);
    int before = 0;
    if (TOTALS) {
        if (threadIdx.x < blockIdx.y) before = gview(d.order)[threadIdx.x];
    } else {
#pragma unroll 4
        for (int k = 4 * threadIdx.x; k < k0; k += kScanKeys) {  // k0 is a multiple of kScanKeys
            const i32x4 v = *(const FMD_GLOBAL i32x4*)(cnt + k);
            before += v.x + v.y + v.z + v.w;
        }
    }
    int c0 = k0 + 4 * threadIdx.x, v[4];
    auto load = [&]() __attribute__((always_inline)) {
        if (c0 + 3 < nkeys) {
            const i32x4 q = *(const FMD_GLOBAL i32x4*)(cnt + c0);
            v[0] = q.x; v[1] = q.y; v[2] = q.z; v[3] = q.w;
        } else {
#pragma unroll
            for (int k = 0; k < 4; k++) v[k] = c0 + k < nkeys ? cnt[c0 + k] : 0;
        }
    };
    load();
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) before += __shfl_xor(before, o, 64);
    if (lane == 0) wbase[wv] = before;
    int carry = 0;  // the counts before this pass, less those in wbase if there is one pass only
    if (!ONE) {
        __syncthreads();
#pragma unroll
        for (int w = 0; w < 16; w++) carry += wbase[w];
    }
    for (int p0 = k0;; p0 += kScanKeys) {
        const int local = v[0] + v[1] + v[2] + v[3];
        int x = local;
#pragma unroll
        for (int o = 1; o < 64; o <<= 1) {
            const int y = __shfl_up(x, o, 64);
            if (lane >= o) x += y;
        }
        if (lane == 63) wsum[wv] = x;
        __syncthreads();
        int at = carry + x - local;
#pragma unroll
        for (int w = 0; w < 16; w++) {
            const int ws = wsum[w];
            at += (ONE ? wbase[w] : 0) + (w < wv ? ws : 0);
            if (!ONE) carry += ws;
        }
        FMD_GLOBAL int* out = gmut(d.cell_start) + c0;
        if (c0 + 3 < nkeys) {
            *(FMD_GLOBAL i32x4*)out = i32x4{at, at + v[0], at + v[0] + v[1], at + v[0] + v[1] + v[2]};
        } else {
#pragma unroll
            for (int k = 0; k < 4; k++) {
                if (c0 + k < nkeys) out[k] = at;
                at += v[k];
            }
        }
        if (c0 < nkeys && c0 + 4 >= nkeys) gmut(d.cell_start)[nkeys] = d.natoms;
        if (ONE || p0 + kScanKeys >= end) break;
        c0 += kScanKeys;
        load();
        __syncthreads();  // wsum is rewritten by the next pass
    }
}

// Atoms, their keys (order) and sort keys (order2) stored in cell order, a
// cell's atoms in the order of their arrival: the rank then reads a cell's sort
// keys contiguously and its own atom's fields coalesced, instead of through the
// order (128 uneven replicas that rebuild together 343 -> 339 us per step, 1M
// beads 193.4 -> 192.9).
__global__ void __launch_bounds__(256) k_scatter(REBUILD_ARGS) {
    REBUILD_LOOP {
        REBUILD_PROLOGUE
        if (i < d.natoms) {
            const int key = d.cell_of[i], dst = d.cell_start[key] + d.rank[i];
            d.order[dst] = key;
            d.order2[dst] = d.sortx[i];
            d.tmp_pos[dst] = d.pos[i];
            d.tmp_vel[dst] = d.vel[i];
            d.tmp_img[dst] = d.img[i];
        }
        // the tile's share of the cell counts, cleared for the next rebuild
        const int nkeys = 1 << (3 * st->cbits), per = (nkeys + d.ntiles - 1) / d.ntiles;
        for (int k = t.lt * per + lane_id(); k < min((t.lt + 1) * per, nkeys); k += kTile) d.cell_cnt[k] = 0;
    }
}

// Rank inside the cell by x, then global id: a deterministic order
// independent of the atomic arrival order of k_bin, in which the list build
// finds the atoms of a row of cells within reach along x by binary search.
// x is the grid coordinate floor(x 2^32 / L) taken modulo 2^32 relative to the
// cell's lower bound floor(cx 2^32 / nx) (k_bin's sortx): the list build
// compares grid coordinates modulo 2^32, and a position a rounding step
// outside [0, L) (at -0 or L itself) stands at the cell's end where the grid
// coordinate puts it.
//
// The atom is moved to its slot here, from k_scatter's copy.  The stores land
// permuted within each cell, so they fill their lines less evenly than those of
// a kernel of its own that goes by the new slots, but that kernel is a launch
// in every step and reads the copy and the order once more.  Per step against
// it: 30,000 beads 40.4 -> 38.9 us, 60,000 41.4 -> 39.7, 250,000 72.2 -> 70.4,
// 1M 195.3 -> 193.8, 128 uneven replicas that rebuild together 355 -> 345.
__global__ void __launch_bounds__(256) k_rank(REBUILD_ARGS) {
    REBUILD_LOOP {
        REBUILD_PROLOGUE
        if (i < d.natoms) {
            const int key = d.order[i];
            const int s = d.cell_start[key], e = d.cell_start[key + 1];
            const int4 im = d.tmp_img[i];
            const int rx = d.order2[i];
            int r = 0;
            for (int q = s; q < e; q++) {
                const int ro = d.order2[q];
                r += (ro < rx) || (ro == rx && d.tmp_img[q].w < im.w);
            }
            const int dst = s + r;
            const float4 p = d.tmp_pos[i];
            d.pos[dst] = p;
            d.pos_ref[dst] = p;
            d.vel[dst] = d.tmp_vel[i];
            d.img[dst] = im;
            d.gid[dst] = im.w;
            d.slot_of[im.w] = dst;
            const double sc = 4294967296.0 / (double)st->Lp;
            d.ipos[dst] = make_int4((int)fix_coord(p.x, sc), (int)fix_coord(p.y, sc), (int)fix_coord(p.z, sc),
                                    __float_as_int(p.w));
        }
    }
}

// ---------------------------------------------------------------------------
// Verlet list + bonded slot tables (src/neighbor/verlet_list.cu:108-335).
// Full list, r^2 < (rc+skin)^2 on the reference FP32 distance, i != j, 1-2
// bonded partners excluded; stored tile-major nbr[tile][k][lane] so the force
// kernel streams one contiguous row per neighbor index.  A count above kcap is
// reported as ERR_NBR_OVERFLOW, never silently truncated.
//
// One workgroup of kGroupTiles waves per group of tiles.  The group's atoms lie
// in a few Morton-consecutive cells; the union of those cells' 27-neighborhoods
// (typically 90-140 cells, about 2000-2900 atoms) is staged in LDS with
// coalesced loads (the top 16 bits of each grid coordinate: a prefilter that
// sends the few candidates near the radius to the exact FP32 test), and each
// lane scans its own 27 cells from LDS in
// (dz, dy, dx) order, candidates in ascending slot order, exactly as the
// global-memory scan that serves groups whose union does not fit.  Both give
// the same rows.  The atoms the group's rows reference (its neighbor set, about
// 1400) are then numbered in slot order and listed in gstage; the rows are
// rewritten to those atoms' byte offsets in the force kernel's LDS copy of the
// set (or to slots when the set exceeds kGroupStage).
// ---------------------------------------------------------------------------
constexpr int kMaxWin = 1024;      // cells of a group's neighbor window (bitmap words <= 32)
constexpr int kPlaceBand = 16;     // row entries moved per pass of the placement

// cell coordinate offset by o in -1..1 with periodic wrap
__device__ inline int wrap_cell(int c, int o, int nx) {
    c += o;
    c += (c < 0) ? nx : 0;
    c -= (c >= nx) ? nx : 0;
    return c;
}

// The bits of candidates q0 + k that are the atom itself or a bonded partner.
__device__ __forceinline__ unsigned excluded_mask(unsigned m, int q0, int i, const int (&ex)[4], int nb, int bcap,
                                                  const FMD_GLOBAL int* bt) {
    unsigned x = 0u;
    auto drop = [&](int e) {
        const unsigned o = (unsigned)(e - q0);
        x |= (o < (unsigned)kBuildChunk) ? (1u << o) : 0u;
    };
    drop(i); drop(ex[0]); drop(ex[1]); drop(ex[2]); drop(ex[3]);
    for (int b = 4; b < nb && b < bcap; b++) drop(bt[b * kTile] & kSlotMask);
    return m & x;
}

// One chunk of kBuildChunk candidates (slots q0 + k, k < n) of the global scan
// by the reference FP32 distance: the tests give a bit mask, then the set bits
// are appended in slot order, skipping the atom itself and its bonded partners.
// W16 rows hold 16-bit entries (replicas of at most 65536 slots), others 32-bit.
template <bool W16>
__device__ __forceinline__ void build_chunk(const float4 (&pj)[kBuildChunk], int q0, int n, int i, float4 pi,
                                            float L, float invL, float rcs2, const int (&ex)[4], int nb,
                                            int bcap, const FMD_GLOBAL int* bt, FMD_GLOBAL int* out,
                                            FMD_GLOBAL unsigned short* out16, int kcap, int& cnt) {
    unsigned m = 0;
#pragma unroll
    for (int k = 0; k < kBuildChunk; k++) {
        const float r2 = dist2_ref(pi, pj[k], L, invL);  // every k: no per-candidate branch
        m |= ((k < n) & (r2 < rcs2)) ? (1u << k) : 0u;
    }
    m &= ~excluded_mask(m, q0, i, ex, nb, bcap, bt);
    while (m) {
        const int k = __builtin_ctz(m);
        m &= m - 1u;
        if (cnt < kcap) {
            if (W16) out16[cnt * kTile] = (unsigned short)(q0 + k);
            else out[cnt * kTile] = q0 + k;
        }
        cnt++;
    }
}

// The same decision with a coarse fixed-point prefilter.  The staged
// positions keep the top 16 bits of each grid coordinate, x and y packed in
// one word and z in the low half of another, so one packed 16-bit subtract per
// word gives the minimum-image differences (modulo 2^16, as the full grid
// wraps modulo 2^32) and two 16-bit dot products give their squared length
// qc.  Truncation moves each coordinate by less than one coarse unit, so
// |sqrt(qc) - r| < sqrt(3) units: qc below clo is certainly inside the list
// radius and qc above chi certainly outside (both bounds also allow for the
// band the exact FP32 test may differ by).  The few candidates in between --
// about 1e-3 sigma either side of the radius -- are decided by the reference
// FP32 formula on their positions.
template <bool B> struct BoolC { static constexpr bool value = B; };
typedef short fmd_s16x2 __attribute__((ext_vector_type(2)));
typedef unsigned short fmd_u16x2 __attribute__((ext_vector_type(2)));
__device__ __forceinline__ fmd_s16x2 coarse_diff(unsigned a, unsigned b) {  // two 16-bit lanes, modulo 2^16
    return __builtin_bit_cast(fmd_s16x2, __builtin_bit_cast(fmd_u16x2, a) - __builtin_bit_cast(fmd_u16x2, b));
}
// qc + acc for the two packed coordinate words of each atom, saturating (a
// sum past INT_MAX is far outside any radius); acc enters the first product
__device__ __forceinline__ int coarse_t(unsigned axy, unsigned az, unsigned bxy, unsigned bz, int acc) {
    const fmd_s16x2 dxy = coarse_diff(axy, bxy), dz = coarse_diff(az, bz);
    return __builtin_amdgcn_sdot2(dz, dz, __builtin_amdgcn_sdot2(dxy, dxy, acc, true), true);
}
__device__ __forceinline__ unsigned coarse_xy(int4 p) {
    return ((unsigned)p.x >> 16) | ((unsigned)p.y & 0xFFFF0000u);
}
__device__ __forceinline__ unsigned coarse_z(int4 p) { return (unsigned)p.z >> 16; }
// Rows are scanned in words of kWord candidates: a lane's hits among one word
// are a 32-bit mask, kept with the word's first staged index until the rows
// are placed.  At most kMaskWords words a tile, at the end of the tile's row
// area (kMaskBytes; kMaskRows rows of 32-bit entries): far more than the
// 9 rows x 2 words of a melt need, and a group with more takes the
// global-memory scan.
constexpr int kWord = 32;
constexpr int kMaskWords = 64;
constexpr int kMaskBytes = kMaskWords * kTile * 6;
constexpr int kMaskRows = kMaskBytes / (kTile * 4);
constexpr int kColWords = 18;  // words a row in the placement by columns

// The list build of one group by kGroupTiles x SPLIT waves.  Phases: the
// union of the group's neighbor cells and its staging, the bonded tables, the
// scan (hit masks), the neighbor set and the row lengths, the placement of the
// rows from the masks.  Wave w works on tile w % kGroupTiles; with SPLIT > 1
// each tile's nine rows of cells are shared out over its SPLIT waves (part
// w / kGroupTiles), which keeps the order of the entries.
//
// What bounds it: the groups' chains of dependent LDS reads, compares and
// barriers.  With every CU holding four groups (1M beads) the waves still wait
// 62% of their time, VALU instructions are issued in 59% of the cycles, and HBM
// moves 1.4 GB in 460 us, 65% of the copy rate; with one group a slot (a step of
// staggered replicas) VALU issue is 35%, and where fewer groups than CUs are
// built it is one group's latency (52 us).  Of a group's 119 us at 1M beads the
// scan takes 37, the placement 28, the bonded tables 11, the window and union
// 20.  Masks instead of appending each hit
// as it is found: the rows are written once, whole 128-byte rows at a time
// (appended, each lane's 2-byte stores fell in a row of their own, and the
// rows were then read back and moved: 165 us a group), and the parts of a
// split scan need not know their first entry.  Together per step: 1M beads
// 230 -> 206 us, 128 uneven replicas 411 -> 364, 30,000 beads 49.0 -> 44.3.
//
// At most 128 VGPRs (four waves per SIMD: four workgroups of one wave per
// tile, or one of four, per CU with the LDS below).
template <int SPLIT>
__global__ void __launch_bounds__(kGroupSlots * SPLIT) __attribute__((amdgpu_waves_per_eu(4, 8)))
k_build(REBUILD_ARGS) {
    constexpr int NT = kGroupSlots * SPLIT;
    constexpr int WP = kMaskWords / SPLIT;  // words of one part
    // During the scan s_raw holds
    //   s_pj    staged union, coarse fixed point: x | y << 16 and z of each atom side
    //           by side (one chunk of padding: a range's last chunk reads whole)
    //   s_cell  union cells: (first slot, count, LDS offset, -)
    //   s_seg   staged atom -> union cell
    //   s_wmap  window cell -> union index
    // and for the placement of a group whose neighbor set fits
    //   s_cidx  LDS byte offset of a used atom
    //   s_m, s_q  the hit masks and their first staged indices, by column
    constexpr int kPj = (kBuildStage + kBuildChunk) * 8, kCell = kMaxUnion * 16, kSeg = kBuildStage * 2;
    constexpr int kCidx = kBuildStage * 2, kMs = kColWords * kGroupSlots * 4, kQs = kColWords * kGroupSlots * 2;
    static_assert(kCidx + kMs + kQs <= kPj + kCell + kSeg + kMaxWin, "the masks fit the scan's arrays");
    __shared__ __align__(16) char s_raw[kPj + kCell + kSeg + kMaxWin];
    uint2* const s_pj = (uint2*)s_raw;
    int4* const s_cell = (int4*)(s_raw + kPj);
    unsigned short* const s_seg = (unsigned short*)(s_raw + kPj + kCell);
    unsigned char* const s_wmap = (unsigned char*)(s_raw + kPj + kCell + kSeg);
    unsigned short* const s_cidx = (unsigned short*)s_raw;
    unsigned* const s_m = (unsigned*)(s_raw + kCidx);
    unsigned short* const s_q = (unsigned short*)(s_raw + kCidx + kMs);
    __shared__ uint2 s_used[kBuildStage / 32 + 1];  // staged atoms in a row of the group: bits, set bits before
    __shared__ unsigned int s_bits[kMaxWin / 32];  // union cells of the window
    __shared__ int s_wpre[kMaxWin / 32];           // union cells before each word of the window
    __shared__ int s_red[6][kGroupTiles];          // per-wave window bounds
    __shared__ int s_c0[3], s_nu, s_nstage, s_ncomp, s_flag;
    __shared__ int s_cnt[SPLIT][kGroupSlots];      // hits of each atom, by part
    __shared__ unsigned char s_words[SPLIT][kGroupSlots];  // and words
    __shared__ unsigned s_col[kGroupSlots];        // by column: row entries | padding entry << 16
    __shared__ int s_hist[kGroupTiles][64];        // rows of each padded length (in kLJTail), by tile
    __shared__ int s_tlen[kGroupTiles];
    __shared__ unsigned short s_rank[kGroupSlots];  // column of each atom's row
    // s_flag: a partner outside the set; too many words or hits; too many words for the column form
    constexpr int kMiss = 1, kOver = 2, kMany = 4;
    // the wave index as a scalar: each wave's tile and replica fields are uniform
    const int wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = lane_id(), tid = threadIdx.x;
    const int tl = wv % kGroupTiles, part = wv / kGroupTiles, at = tl * kTile + lane;
    for (int gb = blockIdx.x, ng = *nrt / kGroupTiles; gb < ng; gb += gridDim.x) {
        const Tile t = tiles[rlist[gb * kGroupTiles + tl]];
        const RepDesc& d = descs[t.rep];
        RepState* st = d.st;
        const int i = t.lt * kTile + lane;
        const int grp = t.lt / kGroupTiles;
        const bool valid = i < d.natoms;
        int err = 0;
        // the exclusion set: the first four bonded partners (slots), and their
        // entries in the topology
        int ex[4] = {-1, -1, -1, -1}, ent[4] = {0, 0, 0, 0};
        int nb = 0;
        float4 pi = make_float4(0.f, 0.f, 0.f, 0.f);
        int4 pf = make_int4(0, 0, 0, 0);
        if (valid) {
            pi = gview(d.pos)[i];
            pf = (int4)gview(d.ipos)[i];
            const int gid = gview(d.gid)[i], b0 = gview(d.t_boff)[gid];
            nb = gview(d.t_boff)[gid + 1] - b0;
#pragma unroll
            for (int b = 0; b < 4; b++)
                if (b < nb) ent[b] = gview(d.t_blst)[b0 + b];
#pragma unroll
            for (int b = 0; b < 4; b++)
                if (b < nb) ex[b] = gview(d.slot_of)[ent[b] & kSlotMask];
        }
        const int kcap = d.kcap;
        const float rcs2 = d.rcs2;
        auto uni = [](float x) { return __int_as_float(__builtin_amdgcn_readfirstlane(__float_as_int(x))); };
        const int nx = __builtin_amdgcn_readfirstlane(st->nx);
        const float ics = uni(st->inv_cs);
        const float L = uni(st->Lp), invL = uni(st->invLp);
        const FMD_GLOBAL float4* gpos = gview(d.pos);
        const FMD_GLOBAL int* cstart = gview(d.cell_start);
        int cx = 0, cy = 0, cz = 0;
        if (valid) {
            cx = cell_coord(pi.x, ics, nx); cy = cell_coord(pi.y, ics, nx); cz = cell_coord(pi.z, ics, nx);
        }
        // The group's cells lie in a small box of cell coordinates (taken
        // relative to the cell of the group's first atom, which is always a real
        // atom, modulo the box).  Their 27-neighborhoods fall in that box grown
        // by one cell per side (the whole axis if that wraps): a window of at
        // most kMaxWin cells.  A bitmap over the window marks the union, whose
        // cells are numbered in window order.
        if (tid == 0) { s_c0[0] = cx; s_c0[1] = cy; s_c0[2] = cz; s_flag = 0; }
        for (int j = tid; j < kMaxWin / 32; j += NT) s_bits[j] = 0u;
        for (int j = tid; j < kBuildStage / 32 + 1; j += NT) s_used[j].x = 0u;
        if (tid < kGroupTiles * 64) s_hist[tid / 64][tid % 64] = 0;
        if (tid < kGroupTiles) s_tlen[tid] = 0;
        __syncthreads();
        const int h = nx >> 1;
        auto rel = [&](int c, int c0) {
            int r = c - c0;
            r += (r < -h) ? nx : 0;
            r -= (r >= nx - h) ? nx : 0;
            return r;
        };
        const int c0x = __builtin_amdgcn_readfirstlane(s_c0[0]), c0y = __builtin_amdgcn_readfirstlane(s_c0[1]),
                  c0z = __builtin_amdgcn_readfirstlane(s_c0[2]);
        const int rx = valid ? rel(cx, c0x) : 0, ry = valid ? rel(cy, c0y) : 0, rz = valid ? rel(cz, c0z) : 0;
        if (part == 0) {
            const int lo_x = wave_min_i(valid ? rx : INT_MAX), hi_x = wave_max_i(valid ? rx : INT_MIN);
            const int lo_y = wave_min_i(valid ? ry : INT_MAX), hi_y = wave_max_i(valid ? ry : INT_MIN);
            const int lo_z = wave_min_i(valid ? rz : INT_MAX), hi_z = wave_max_i(valid ? rz : INT_MIN);
            if (lane == 0) {
                s_red[0][tl] = lo_x; s_red[1][tl] = hi_x; s_red[2][tl] = lo_y;
                s_red[3][tl] = hi_y; s_red[4][tl] = lo_z; s_red[5][tl] = hi_z;
            }
        }
        __syncthreads();
        int sx, sy, sz, ex_, ey_, ez_;
        auto window = [&](int a, int& s0, int& e0) {
            int lo = INT_MAX, hi = INT_MIN;
            for (int w = 0; w < kGroupTiles; w++) { lo = min(lo, s_red[2 * a][w]); hi = max(hi, s_red[2 * a + 1][w]); }
            s0 = __builtin_amdgcn_readfirstlane(lo - 1);
            e0 = __builtin_amdgcn_readfirstlane(min(hi - lo + 3, nx));  // the whole axis once the grown box wraps
        };
        window(0, sx, ex_);
        window(1, sy, ey_);
        window(2, sz, ez_);
        // window cell of this atom's neighbor cell (dx, dy, dz); the offset from
        // the window start is >= 0 and, on an axis the window wraps (extent nx),
        // taken modulo nx
        auto wmod = [](int v, int e) {  // v in [0, e + 1]: v mod e (e >= 1)
            v -= (v >= e) ? e : 0;
            v -= (v >= e) ? e : 0;
            return v;
        };
        auto win_at = [&](int dx, int dy, int dz) {
            return (wmod(rz + dz - sz, ez_) * ey_ + wmod(ry + dy - sy, ey_)) * ex_ + wmod(rx + dx - sx, ex_);
        };
        const int W = ex_ * ey_ * ez_;
        // staged scan: prefilter in fixed point; boxes of fewer than 3 cells per
        // axis (where a pair can sit near half the box) use the global scan
        bool staged = W <= kMaxWin && nx >= 3;  // uniform over the group
        const unsigned cxy = coarse_xy(pf), cz16 = coarse_z(pf);
        int clo, chi, rb2;
        {
            // radius in coarse units (L / 2^16), widened by the band the exact
            // FP32 test may differ by and by sqrt(3) units of truncation
            const double rc = (double)d.rcs * 65536.0 / (double)L;
            const double band = 3e-5 + 1e-6 * (double)L / (double)d.rcs;  // >> the two forms' difference
            const double rb = rc * sqrt(1.0 + band);  // above the true distance of any pair the FP32 test accepts
            const double rin = rc * sqrt(1.0 - band) - 1.7321 - 0.01, rout = rb + 1.7321 + 0.01;
            clo = __builtin_amdgcn_readfirstlane(rin > 0.0 ? (int)floor(rin * rin) : 0);
            chi = __builtin_amdgcn_readfirstlane((int)ceil(rout * rout));
            rb2 = __builtin_amdgcn_readfirstlane((int)fmin(ceil(rb * rb) + 1.0, 2147483647.0));
            // In a box of three cells an atom on a cell bound (its float cell
            // coordinate one low) has an outer cell's far side in reach along x:
            // there the rows are not cut short (the pair's y and z distances are
            // next to nothing, so more than two cells are left of this along x).
            // In bits: the same as a choice by nx costs 0.25 us per step of 48
            // small replicas, in scalar registers.
            rb2 |= (int)((unsigned)((nx - 4) >> 31) >> 1);  // the largest int if nx < 4
        }
        int nu = 0, nstage = 0;
        if (staged) {
            // each cell of the group marks its 27 neighbors (its first lane in a
            // wave does), a share of them in each part
            const int prev = __shfl_up(cx + nx * (cy + nx * cz), 1, 64);
            if (valid && (lane == 0 || prev != cx + nx * (cy + nx * cz)))
                #pragma unroll 1
                for (int c = part; c < 27; c += SPLIT) {
                    const int w = win_at(c % 3 - 1, (c / 3) % 3 - 1, c / 9 - 1);
                    atomicOr(&s_bits[w >> 5], 1u << (w & 31));
                }
            __syncthreads();
            if (wv == 0) {
                // marked cells before each word of the window
                const int nwords = (W + 31) >> 5;  // <= kMaxWin / 32 <= 64 lanes
                const int c = (lane < nwords) ? __popc(s_bits[lane]) : 0;
                int x = c;
#pragma unroll
                for (int o = 1; o < 64; o <<= 1) {
                    const int y = __shfl_up(x, o, 64);
                    if (lane >= o) x += y;
                }
                if (lane < nwords) s_wpre[lane] = x - c;
                if (lane == 63) s_nu = x;
            }
            __syncthreads();
            nu = __builtin_amdgcn_readfirstlane(s_nu);
            staged = nu <= kMaxUnion;
        }
        if (staged) {
            // number the marked cells in window order, with their slots
            auto wrapn = [&](int p) {  // p in [-nx, 2 nx)
                p += (p < 0) ? nx : 0;
                p -= (p >= nx) ? nx : 0;
                return p;
            };
            for (int w = tid; w < W; w += NT) {
                const unsigned wb = s_bits[w >> 5];
                if ((wb >> (w & 31)) & 1u) {
                    const int u = s_wpre[w >> 5] + __popc(wb & ((1u << (w & 31)) - 1u));
                    const int wx = w % ex_, wyz = w / ex_, wy = wyz % ey_, wz = wyz / ey_;
                    const int k = (int)cell_key(wrapn(c0x + sx + wx), wrapn(c0y + sy + wy), wrapn(c0z + sz + wz));
                    const int s0 = cstart[k];
                    s_wmap[w] = (unsigned char)u;
                    s_cell[u] = make_int4(s0, cstart[k + 1] - s0, 0, 0);
                }
            }
            __syncthreads();
            if (wv == 0) {  // LDS offsets of the union cells
                int ns = 0;
                for (int u0 = 0; u0 < nu; u0 += 64) {
                    const int u = u0 + lane;
                    const int c = (u < nu) ? s_cell[u].y : 0;
                    int y = c;
#pragma unroll
                    for (int o = 1; o < 64; o <<= 1) {
                        const int z = __shfl_up(y, o, 64);
                        if (lane >= o) y += z;
                    }
                    if (u < nu) s_cell[u].z = ns + y - c;
                    ns += __shfl(y, 63, 64);
                }
                if (lane == 0) s_nstage = ns;
            }
            __syncthreads();
            nstage = __builtin_amdgcn_readfirstlane(s_nstage);
            staged = nstage <= kBuildStage;
        }
        if (staged) {
            for (int u = tid; u < nu; u += NT) {
                const int4 ce = s_cell[u];
                for (int j = 0; j < ce.y; j++) s_seg[ce.z + j] = (unsigned short)u;
            }
            __syncthreads();
            const FMD_GLOBAL int4* gip = gview(d.ipos);
            constexpr int kAhead = SPLIT == 1 ? 4 : 2;  // positions in flight per thread
            for (int q0 = 0; q0 < nstage; q0 += kAhead * NT) {
                int4 v4[kAhead];
#pragma unroll
                for (int k = 0; k < kAhead; k++) {
                    const int q = min(q0 + k * NT + tid, nstage - 1);
                    const int4 ce = s_cell[s_seg[q]];
                    v4[k] = gip[ce.x + q - ce.z];
                }
#pragma unroll
                for (int k = 0; k < kAhead; k++) {
                    const int q = q0 + k * NT + tid;
                    if (q < nstage) s_pj[q] = make_uint2(coarse_xy(v4[k]), coarse_z(v4[k]));
                }
            }
            __syncthreads();
        }
        auto slot_of = [&](int q) __attribute__((always_inline)) {  // slot of a staged atom
            const int4 ce = s_cell[s_seg[q]];
            return ce.x + q - ce.z;
        };
        auto mark = [&](int q) __attribute__((always_inline)) { atomicOr(&s_used[q >> 5].x, 1u << (q & 31)); };
        // The staged index of a bonded partner (slot ps at position pp): its cell
        // is one of the 27 around this atom's (a bond is shorter than a cell),
        // found through the window; -1 if not (the group then keeps slots
        // everywhere).
        auto staged_of = [&](int ps, float4 pp) __attribute__((always_inline)) -> int {
            int dx = rel(cell_coord(pp.x, ics, nx), c0x) - rx, dy = rel(cell_coord(pp.y, ics, nx), c0y) - ry,
                dz = rel(cell_coord(pp.z, ics, nx), c0z) - rz;
            dx += (dx < -1) ? nx : 0; dx -= (dx > 1) ? nx : 0;
            dy += (dy < -1) ? nx : 0; dy -= (dy > 1) ? nx : 0;
            dz += (dz < -1) ? nx : 0; dz -= (dz > 1) ? nx : 0;
            if (dx < -1 || dx > 1 || dy < -1 || dy > 1 || dz < -1 || dz > 1) return -1;
            const int u = s_wmap[win_at(dx, dy, dz)];
            if (u >= nu) return -1;
            const int4 ce = s_cell[u];
            const int o = ps - ce.x;
            return (o >= 0 && o < ce.y) ? ce.z + o : -1;
        };
        // exclusions as staged indices: the first four bonded partners (none, or a
        // partner outside the 27 cells, which is no candidate: INT_MAX).  Their
        // positions are requested together, so the latencies overlap.
        int xs[4] = {INT_MAX, INT_MAX, INT_MAX, INT_MAX};
        if (staged && valid) {
            float4 pp[4];
#pragma unroll
            for (int b = 0; b < 4; b++) pp[b] = gpos[ex[b] >= 0 ? ex[b] : i];
#pragma unroll
            for (int b = 0; b < 4; b++) {
                const int q = ex[b] >= 0 ? staged_of(ex[b], pp[b]) : -1;
                xs[b] = q >= 0 ? q : INT_MAX;
            }
        }
        // The bonded tables, the bonds by part 0 and the angles by the last:
        // entries hold the partners' slots, or with `set` their staged indices
        // (marked as used), which become LDS byte offsets once the set is known.
        const bool do_bonds = part == 0, do_angles = part == SPLIT - 1;
        int miss = 0;
        auto use = [&](int q) __attribute__((always_inline)) {  // a partner's staged index as an entry
            const bool in = q >= 0 && q != INT_MAX;
            if (in) mark(q);
            else miss = 1;
            return in ? q : 0;
        };
        auto partner = [&](int b) __attribute__((always_inline)) {  // the slot of bonded partner b >= 4
            return (int)gview(d.slot_of)[gview(d.t_blst)[gview(d.t_boff)[gview(d.gid)[i]] + b] & kSlotMask];
        };
        auto bonded = [&](bool set) __attribute__((always_inline)) {
            const int gid = gview(d.gid)[i], a0 = gview(d.t_aoff)[gid], na = gview(d.t_aoff)[gid + 1] - a0;
            if (do_bonds) {
                FMD_GLOBAL int* bt = gmut(d.bnd) + (size_t)t.lt * d.bcap * kTile + lane;
                const int nbk = min(nb, d.bcap);
                gmut(d.bhdr)[i] = nbk | (min(na, d.acap) << 8);
                if (nb > d.bcap || na > d.acap) err |= ERR_BONDED;
#pragma unroll
                for (int b = 0; b < 4; b++)
                    if (b < nbk) bt[b * kTile] = (set ? use(xs[b]) : ex[b]) | (ent[b] & ~kSlotMask);
                for (int b = 4; b < nbk; b++) {
                    const int ps = partner(b);
                    bt[b * kTile] = (set ? use(staged_of(ps, gpos[ps])) : ps) |
                                    (gview(d.t_blst)[gview(d.t_boff)[gid] + b] & ~kSlotMask);
                }
            }
            if (do_angles) {
                // kAngles at a time, the loads of each step of their chains together
                constexpr int kAngles = 3;
                FMD_GLOBAL int2* an = gmut(d.ang) + (size_t)t.lt * d.acap * kTile + lane;
                const int nak = min(na, d.acap);
                for (int k0 = 0; k0 < nak; k0 += kAngles) {
                    int4 A[kAngles];
                    int s1[kAngles], s2[kAngles], role[kAngles];
#pragma unroll
                    for (int k = 0; k < kAngles; k++) A[k] = (int4)gview(d.t_alst)[a0 + min(k0 + k, nak - 1)];
#pragma unroll
                    for (int k = 0; k < kAngles; k++) {
                        role[k] = (A[k].x == gid) ? 0 : ((A[k].y == gid) ? 1 : 2);
                        s1[k] = gview(d.slot_of)[role[k] == 0 ? A[k].y : A[k].x];
                        s2[k] = gview(d.slot_of)[role[k] == 2 ? A[k].y : A[k].z];
                    }
                    float4 p1[kAngles], p2[kAngles];
                    if (set) {
#pragma unroll
                        for (int k = 0; k < kAngles; k++) { p1[k] = gpos[s1[k]]; p2[k] = gpos[s2[k]]; }
                    }
#pragma unroll
                    for (int k = 0; k < kAngles; k++)
                        if (k0 + k < nak) {
                            const int e1 = set ? use(staged_of(s1[k], p1[k])) : s1[k];
                            const int e2 = set ? use(staged_of(s2[k], p2[k])) : s2[k];
                            an[(k0 + k) * kTile] = make_int2(e1 | (role[k] << kSlotBits), e2 | (A[k].w << kSlotBits));
                        }
                }
            }
        };
        const bool want_set = staged && !d.nostage;  // uniform
        if (valid) bonded(want_set);
        // hit masks of this lane and part, in row order
        char* const area_end = (char*)(d.nbr + (size_t)(t.lt + 1) * d.kcap * kTile);
        FMD_GLOBAL unsigned* gm = gmut((unsigned*)(area_end - kMaskBytes)) + part * WP * kTile + lane;
        FMD_GLOBAL unsigned short* gq =
            gmut((unsigned short*)(area_end - kMaskBytes + kMaskWords * kTile * 4)) + part * WP * kTile + lane;
        int cnt = 0, qself = 0, nw = 0;
        if (staged) {
            int pend = -1, pq = 0, over = 0;
            if (valid) {
                {  // the atom's own staged index
                    const int us = s_wmap[win_at(0, 0, 0)];
                    if (us < nu) qself = s_cell[us].z + (i - s_cell[us].x);
                    if (us >= nu || qself < 0 || qself >= nstage) {
                        err |= ERR_INTERNAL;
                        qself = 0;
                    }
                    if (part == 0) mark(qself);
                }
                int nxu = 0;  // entries of xs from nxu on are INT_MAX in every lane of the wave
#pragma unroll
                for (int b = 0; b < 4; b++) nxu = __ballot(xs[b] != INT_MAX) ? b + 1 : nxu;
                // Lower bounds (coarse units) of the distance along y and z from
                // this atom to any atom of the cell below and above its own: its
                // offset from its cell's bounds floor(c 2^16 / nx), less 2 units
                // (the truncation of the atom's coordinate and of the bound, and
                // the rounding of the float cell coordinate).  These offsets are
                // less than two cells, so with 3 or more cells per axis they do not
                // wrap as signed 16-bit differences of at most one cell.
                int yb[2], zb[2];
                {
                    auto cb = [&](int c) { return (int)(((unsigned)c << 16) / (unsigned)nx); };
                    auto off16 = [](int a, int b) { return max(0, (int)(short)(unsigned short)(a - b) - 2); };
                    const int yc = (int)(cxy >> 16), zc = (int)cz16;
                    yb[0] = off16(yc, cb(cy)); yb[1] = off16(cb(cy + 1), yc);
                    zb[0] = off16(zc, cb(cz)); zb[1] = off16(cb(cz + 1), zc);
                }
                // First q in [lo, hi) whose x offset from this atom, less `by`, is
                // above v (coarse units).  A cell's atoms are in ascending x; their
                // offsets from an atom of the neighboring cell span two cells, which
                // may wrap as signed 16-bit numbers, but not those less one cell
                // (by = -cell or cell, the offset of the cell's middle).
                const int cell16 = (int)(65536u / (unsigned)nx);
                auto first_above = [&](int lo, int hi, int by, int v) {
                    const unsigned ref = (cxy & 0xFFFFu) + (unsigned)by;
                    while (lo < hi) {
                        const int mid = (lo + hi) >> 1;
                        if ((int)(short)(unsigned short)(s_pj[mid].x - ref) <= v) lo = mid + 1;
                        else hi = mid;
                    }
                    return lo;
                };
                const unsigned bw = (unsigned)(chi - clo);
                // the hits among the candidates q0 .. q0 + n - 1 (n <= kWord): chunks
                // of kBuildChunk by the coarse prefilter.  t = q - clo is negative for
                // a candidate certainly inside; its sign bit is shifted into m from the
                // last candidate down (alignbit of (m, t) by 31 is m << 1 | t >> 31),
                // so bit k of m is candidate k; the smallest t as an unsigned number is
                // the nearest candidate not certainly inside, and only when it lies in
                // the band [0, bw] are the band's candidates found one by one.
                auto word = [&](int q0, int n) __attribute__((always_inline)) {
                    unsigned m = 0u, band = 0u;
#pragma unroll
                    for (int c = 0; c < kWord; c += kBuildChunk) {
                        if (c >= n) break;
                        unsigned m8 = 0u, umin = ~0u;
                        int tt[kBuildChunk];
                        uint2 jp[kBuildChunk];
#pragma unroll
                        for (int k = 0; k < kBuildChunk; k++) jp[k] = s_pj[q0 + c + k];
#pragma unroll
                        for (int k = kBuildChunk - 1; k >= 0; k--) {
                            tt[k] = coarse_t(cxy, cz16, jp[k].x, jp[k].y, -clo);
                            m8 = __builtin_amdgcn_alignbit(m8, (unsigned)tt[k], 31);
                            umin = min(umin, (unsigned)tt[k]);
                        }
                        m |= m8 << c;
                        if (umin <= bw) {
#pragma unroll
                            for (int k = 0; k < kBuildChunk; k++) band |= ((unsigned)tt[k] <= bw) ? (1u << (c + k)) : 0u;
                        }
                    }
                    unsigned keep = n >= kWord ? ~0u : (1u << n) - 1u;
                    // leave out the atom itself and its bonded partners
                    auto drop = [&](int v) {
                        const unsigned o = (unsigned)(v - q0);
                        keep &= ~(o < (unsigned)kWord ? 1u << o : 0u);
                    };
                    drop(qself); drop(xs[0]); drop(xs[1]);
                    if (__builtin_expect(nxu > 2, 0)) { drop(xs[2]); drop(xs[3]); }
                    for (int b = 4; b < nb; b++) {  // partners past the first four
                        const int ps = partner(b), q = staged_of(ps, gpos[ps]);
                        if (q >= 0) drop(q);
                    }
                    m &= keep;
                    band &= keep;
                    if (band) {
                        // undecided: the reference distance on the float positions, a
                        // global load.  A lane's first one counts as inside for now and
                        // is decided after the scan, with one load round trip for the
                        // whole wave; further ones are decided at once.
                        if (pend < 0) {
                            const int k = __builtin_ctz(band);
                            band &= band - 1u;
                            pend = nw * kWord + k;
                            pq = q0 + k;
                            m |= 1u << k;
                        }
                        while (band) {
                            const int k = __builtin_ctz(band);
                            band &= band - 1u;
                            m |= (dist2_ref(pi, gpos[slot_of(q0 + k)], L, invL) < rcs2) ? (1u << k) : 0u;
                        }
                    }
                    if (m) {
                        if (nw < WP) {
                            gm[nw * kTile] = m;
                            gq[nw * kTile] = (unsigned short)q0;
                            nw++;
                        } else {
                            over = 1;
                        }
                        cnt += __popc(m);
                        const int s = q0 & 31;
                        atomicOr(&s_used[q0 >> 5].x, m << s);
                        const unsigned up = s ? m >> (32 - s) : 0u;
                        if (up) atomicOr(&s_used[(q0 >> 5) + 1].x, up);
                    }
                };
                // this part's rows of the 27 cells in (dz, dy, dx) order; the three
                // cells of a (dz, dy) row are consecutive union cells (hence one
                // contiguous staged range) unless the window wraps that axis
                const int w0 = wmod(rx - 1 - sx, ex_), w1 = wmod(rx - sx, ex_), w2 = wmod(rx + 1 - sx, ex_);
                const int r0 = part * (8 / SPLIT), r1 = part == SPLIT - 1 ? 9 : r0 + 8 / SPLIT;
                #pragma unroll 1
                for (int r = r0; r < r1; r++) {
                    const int iy = r % 3, iz = r / 3;
                    // Only atoms within xr of this atom along x can be in the
                    // list: the distance along y and z to the row's cells leaves
                    // at most sqrt(rb2 - dy^2 - dz^2) along x, and the coarse x
                    // difference is within one unit of the true one.  A row with
                    // nothing left is skipped whole.
                    const int dyb = (iy == 1) ? 0 : yb[iy >> 1], dzb = (iz == 1) ? 0 : zb[iz >> 1];
                    const int rem = rb2 - dyb * dyb - dzb * dzb;
                    if (rem < 0) continue;
                    const int xr = (int)ceilf(sqrtf((float)rem)) + 2;
                    const int wb = (wmod(rz + iz - 1 - sz, ez_) * ey_ + wmod(ry + iy - 1 - sy, ey_)) * ex_;
                    const int ua = s_wmap[wb + w0], ub = s_wmap[wb + w1], uc = s_wmap[wb + w2];
                    if (ua >= nu || ub >= nu || uc >= nu) {  // every neighbor cell was marked; guard regardless
                        err |= ERR_INTERNAL;
                        continue;
                    }
                    const int4 A = s_cell[ua], B = s_cell[ub], Cc = s_cell[uc];
                    const bool one = ub == ua + 1 && uc == ub + 1;
                    // the outer cells' atoms within reach: from za in the first cell,
                    // up to ec in the third
                    const int za = first_above(A.z, A.z + A.y, -cell16, cell16 - xr - 1),
                              ec = first_above(Cc.z, Cc.z + Cc.y, cell16, xr - cell16);
                    #pragma unroll 1
                    for (int k = 0; k < (one ? 1 : 3); k++) {
                        const int z = k == 0 ? za : (k == 1 ? B.z : Cc.z);
                        const int e = (one || k == 2) ? ec : (k == 0 ? A.z + A.y : B.z + B.y);
                        #pragma unroll 1
                        for (int q0 = z; q0 < e; q0 += kWord) word(q0, e - q0);
                    }
                }
                if (pend >= 0 && !over) {  // the deferred candidate
                    const bool in = dist2_ref(pi, gpos[slot_of(pq)], L, invL) < rcs2;
                    if (!in) {
                        const int w = pend / kWord;
                        gm[w * kTile] &= ~(1u << (pend % kWord));
                        cnt--;
                    }
                }
            }
            s_cnt[part][at] = cnt;
            s_words[part][at] = (unsigned char)nw;
            const int flag = (miss ? kMiss : 0) | (over ? kOver : 0);
            if (flag) atomicOr(&s_flag, flag);
            __syncthreads();
            if (!d.idx16) {  // 32-bit rows share the area with the masks
                int all = 0;
#pragma unroll
                for (int p = 0; p < SPLIT; p++) all += s_cnt[p][at];
                if (all > kcap - kMaskRows - kLJTail) atomicOr(&s_flag, kOver);
                __syncthreads();
            }
            if (s_flag & kOver) staged = false;
        }
        FMD_GLOBAL int* out = gmut(d.nbr) + (size_t)t.lt * d.kcap * kTile + lane;
        // 16-bit rows of the global scan are built in the upper half of the
        // tile's row area (which holds 2 kcap 16-bit entries per lane) and moved
        // to the lower half by the placement below; 32-bit rows are built in place
        FMD_GLOBAL unsigned short* out16 =
            (FMD_GLOBAL unsigned short*)(gmut(d.nbr) + (size_t)t.lt * d.kcap * kTile) + (size_t)d.kcap * kTile + lane;
        if (!staged) {
            if (want_set) {  // the scan was given up: slots in the bonded tables too
                if (valid) bonded(false);
            }
            cnt = 0;
            nw = 0;
            if (valid && part == 0) {
                // global-memory scan with the same visiting order
                auto key_of = [&](int c) {
                    return (int)cell_key(wrap_cell(cx, c % 3 - 1, nx), wrap_cell(cy, (c / 3) % 3 - 1, nx),
                                         wrap_cell(cz, c / 9 - 1, nx));
                };
                // bonded partners past the first four are read from the table
                // (slots), which this lane wrote
                const FMD_GLOBAL int* bt = gview(d.bnd) + (size_t)t.lt * d.bcap * kTile + lane;
                for (int c = 0; c < 27; c++) {
                    const int k = key_of(c);
                    bool seen = false;
                    if (nx < 3)
                        for (int v = 0; v < c; v++) seen |= (key_of(v) == k);
                    if (seen) continue;
                    const int s0 = cstart[k], e0 = cstart[k + 1];
                    for (int q0 = s0; q0 < e0; q0 += kBuildChunk) {
                        float4 pj[kBuildChunk];
#pragma unroll
                        for (int k2 = 0; k2 < kBuildChunk; k2++) pj[k2] = gpos[min(q0 + k2, e0 - 1)];
                        if (d.idx16)
                            build_chunk<true>(pj, q0, e0 - q0, i, pi, L, invL, rcs2, ex, nb, d.bcap, bt, out, out16, kcap, cnt);
                        else
                            build_chunk<false>(pj, q0, e0 - q0, i, pi, L, invL, rcs2, ex, nb, d.bcap, bt, out, out16, kcap, cnt);
                    }
                }
            }
            __syncthreads();  // s_cnt is read by every part above
            s_cnt[part][at] = cnt;
            __syncthreads();
        }
        // Row lengths: start = this part's first entry, total over the parts
        int start = 0, total = 0, wstart = 0, words = 0;
#pragma unroll
        for (int p = 0; p < SPLIT; p++) {
            const int c = s_cnt[p][at], n = staged ? s_words[p][at] : 0;
            start += p < part ? c : 0;
            wstart += p < part ? n : 0;
            total += c;
            words += n;
        }
        if (words > kColWords || total > kcap) atomicOr(&s_flag, kMany);
        const int stored = min(total, kcap);
        const int padded = valid ? ((stored + kLJTail - 1) / kLJTail) * kLJTail : 0;
        // Columns: the group's rows go to columns in descending order of their
        // padded length (ties by slot; lengths from 252 up count as one), so the
        // 64 rows a wave streams are of nearly equal length; gperm[column] names
        // the atom.  A counting sort: rows of the same length in the wave by
        // ballot, in the group through s_hist.
        const int bucket = min(padded / kLJTail, 63);
        int within = 0;
        if (part == 0) {
            unsigned long long todo = ~0ull;
            while (todo) {
                const int lead = __builtin_ctzll(todo);
                const int b = __builtin_amdgcn_readlane(bucket, lead);
                const unsigned long long same = __ballot(bucket == b);
                if (bucket == b) within = lane_prefix(same);
                if (lane == lead) s_hist[tl][b] = __popcll(same);
                todo &= ~same;
            }
        }
        if (staged && wv == kGroupTiles * SPLIT - 1) {
            // used atoms before each word of the staged set
            int base = 0;
            for (int w0 = 0; w0 < kBuildStage / 32; w0 += 64) {
                const int w = w0 + lane;
                const int c = w < kBuildStage / 32 ? __popc(s_used[w].x) : 0;
                int x = c;
#pragma unroll
                for (int o = 1; o < 64; o <<= 1) {
                    const int y = __shfl_up(x, o, 64);
                    if (lane >= o) x += y;
                }
                if (w < kBuildStage / 32) s_used[w].y = (unsigned)(base + x - c);
                base += __shfl(x, 63, 64);
            }
            if (lane == 0) s_ncomp = base;
        }
        __syncthreads();
        // the group's neighbor set: used staged atoms, every atom itself and its
        // bonded partners (the force kernel reads them from the set too),
        // numbered in staged (slot) order
        const int ncomp = staged ? s_ncomp : 0;
        const int flags = s_flag;
        const bool compact = staged && want_set && ncomp <= kGroupStage && !(flags & kMiss);  // uniform
        const bool bycol = compact && !(flags & kMany);
        if (part == 0) {
            int tot = 0;  // rows of length `lane` in the group, then of that length or more
#pragma unroll
            for (int w = 0; w < kGroupTiles; w++) tot += s_hist[w][lane];
            int suf = tot;
#pragma unroll
            for (int o = 1; o < 64; o <<= 1) {
                const int y = __shfl_down(suf, o, 64);
                if (lane + o < 64) suf += y;
            }
            int rank = __shfl(suf - tot, bucket, 64) + within;
#pragma unroll
            for (int w = 0; w < kGroupTiles - 1; w++) rank += w < tl ? s_hist[w][bucket] : 0;
            s_rank[at] = (unsigned short)rank;
            gmut(d.gperm)[(size_t)grp * kGroupSlots + rank] = (unsigned char)at;
            atomicMax(&s_tlen[rank / kTile], padded);
        }
        if (compact)
            for (int q = tid; q < nstage; q += NT) {
                const uint2 u = s_used[q >> 5];
                if ((u.x >> (q & 31)) & 1u) {
                    const int idx = (int)u.y + __popc(u.x & ((1u << (q & 31)) - 1u));
                    const int slot = slot_of(q);
                    const size_t p = (size_t)grp * kGroupStage + idx;
                    s_cidx[q] = (unsigned short)(idx << 4);
                    if (d.idx16) ((FMD_GLOBAL unsigned short*)gmut(d.gstage))[p] = (unsigned short)slot;
                    else gmut(d.gstage)[p] = slot;
                }
            }
        if (tid == 0) gmut(d.gcount)[grp] = compact ? ncomp : -1;
        __syncthreads();
        // every row of a wave is padded to the wave's longest, whose length the
        // force pass reads as one uniform bound
        const int rank = s_rank[at];
        const int wpad = s_tlen[rank / kTile];
        if (part == 0 && rank % kTile == 0) gmut(d.tlen)[grp * kGroupTiles + rank / kTile] = wpad;
        int selfent = i;  // the padding entry: the atom itself (rejected by r^2 = 0)
        if (valid && want_set) {
            if (compact) {
                // bonded entries of a staged group: LDS byte offsets of the partners
                // in the set instead of staged indices (role and type bits kept)
                if (do_bonds)
                    for (int b = 0; b < min(nb, d.bcap); b++) {
                        FMD_GLOBAL int* p = gmut(d.bnd) + ((size_t)t.lt * d.bcap + b) * kTile + lane;
                        const int e = *p;
                        *p = (int)s_cidx[e & kSlotMask] | (e & ~kSlotMask);
                    }
                if (do_angles)
                    for (int a = 0, na = (gview(d.bhdr)[i] >> 8) & 0xFF; a < na; a++) {
                        FMD_GLOBAL int2* p = gmut(d.ang) + ((size_t)t.lt * d.acap + a) * kTile + lane;
                        const int ex1 = p->x, ex2 = p->y;
                        p->x = (int)s_cidx[ex1 & kSlotMask] | (ex1 & ~kSlotMask);
                        p->y = (int)s_cidx[ex2 & kSlotMask] | (ex2 & ~kSlotMask);
                    }
                selfent = (int)s_cidx[qself];
            } else if (staged) {
                bonded(false);
            }
        }
        // Placement.  From the masks, each part from its first entry on: an
        // entry is its atom's LDS byte offset in the set (or its slot when the set
        // did not fit).
        FMD_GLOBAL int* dtile = gmut(d.nbr) + (size_t)(grp * kGroupTiles + rank / kTile) * d.kcap * kTile;
        if (bycol) {
            // One lane per column, every lane at the same row entry: a pass stores a
            // whole 128-byte row (with a lane per atom and a word at a time, the
            // lanes' stores fall in as many rows as lanes).  The atoms' masks go to
            // LDS by column; with SPLIT > 1 each part places a share of the rows.
            for (int w = 0; w < nw; w++) {
                s_m[(wstart + w) * kGroupSlots + rank] = gm[w * kTile];
                s_q[(wstart + w) * kGroupSlots + rank] = gq[w * kTile];
            }
            if (part == 0) s_col[rank] = (unsigned)total | (unsigned)(valid ? selfent : 0) << 16;
            __syncthreads();
            const unsigned cc = s_col[at];
            const int n = (int)(cc & 0xFFFFu), pad = (int)(cc >> 16);
            const int wp = __builtin_amdgcn_readfirstlane(s_tlen[tl]);
            const int share = ((wp / kLJTail + SPLIT - 1) / SPLIT) * kLJTail;
            const int k0 = part * share, k1 = min(wp, k0 + share);
            int left = n - k0;  // entries left in the row
            const unsigned* pm = s_m + at;
            const unsigned short* pq = s_q + at;
            unsigned m = 0u;
            int q0 = 0;
            if (left > 0) {
                int skip = k0;
                m = *pm;
                while (skip > 0) {  // to this part's first entry
                    const int c = __popc(m);
                    if (c > skip) {
                        for (; skip > 0; skip--) m &= m - 1u;
                    } else {
                        skip -= c;
                        pm += kGroupSlots;
                        pq += kGroupSlots;
                        m = *pm;
                    }
                }
                q0 = *pq;
            }
            auto emit = [&](auto* dst) __attribute__((always_inline)) {
                for (int k = k0; k < k1; k += kLJTail, dst += kLJTail * kTile) {
                    int q[kLJTail];
#pragma unroll
                    for (int j = 0; j < kLJTail; j++) {
                        q[j] = -1;
                        if (left > j) {
                            while (!m) {
                                pm += kGroupSlots;
                                pq += kGroupSlots;
                                m = *pm;
                                q0 = *pq;
                            }
                            q[j] = q0 + __builtin_ctz(m);
                            m &= m - 1u;
                        }
                    }
                    left -= kLJTail;
                    int e[kLJTail];
#pragma unroll
                    for (int j = 0; j < kLJTail; j++) e[j] = (int)s_cidx[max(q[j], 0)];
#pragma unroll
                    for (int j = 0; j < kLJTail; j++) dst[j * kTile] = q[j] >= 0 ? e[j] : pad;
                }
            };
            FMD_GLOBAL int* ctile = gmut(d.nbr) + (size_t)t.lt * d.kcap * kTile;
            if (d.idx16) emit((FMD_GLOBAL unsigned short*)ctile + k0 * kTile + lane);
            else emit(ctile + k0 * kTile + lane);
        } else if (staged) {
            if (total > kcap) {  // more hits than the row holds (an error): leave out the last ones
                int room = max(0, kcap - start);
                for (int w = 0; w < nw; w++) {
                    unsigned m = gm[w * kTile], keep = 0u;
                    for (; m && room > 0; room--) {
                        keep |= m & (0u - m);
                        m &= m - 1u;
                    }
                    gm[w * kTile] = keep;
                }
            }
            auto emit = [&](auto* dst, auto set) __attribute__((always_inline)) {
                auto entry = [&](int q) __attribute__((always_inline)) {
                    return decltype(set)::value ? (int)s_cidx[q] : slot_of(min(q, nstage - 1));
                };
                dst += start * kTile;
                unsigned m = nw > 0 ? gm[0] : 0u;
                int q0 = nw > 0 ? gq[0] : 0;
                for (int w = 0; w < nw; w++) {
                    unsigned mn = 0u;
                    int qn = 0;
                    if (w + 1 < nw) { mn = gm[(w + 1) * kTile]; qn = gq[(w + 1) * kTile]; }
                    // four hits per pass, their reads in flight together (the bit of a
                    // missing one reads entry 31 and is not stored)
                    auto* p = dst;
                    dst += __popc(m) * kTile;
                    while (m) {
                        const unsigned m1 = m & (m - 1u), m2 = m1 & (m1 - 1u), m3 = m2 & (m2 - 1u);
                        const int e0 = entry(q0 + __builtin_ctz(m)), e1 = entry(q0 + __builtin_ctz(m1 | 0x80000000u)),
                                  e2 = entry(q0 + __builtin_ctz(m2 | 0x80000000u)),
                                  e3 = entry(q0 + __builtin_ctz(m3 | 0x80000000u));
                        p[0] = e0;
                        if (m1) p[kTile] = e1;
                        if (m2) p[2 * kTile] = e2;
                        if (m3) p[3 * kTile] = e3;
                        p += 4 * kTile;
                        m = m3 & (m3 - 1u);
                    }
                    m = mn;
                    q0 = qn;
                }
                if (part == SPLIT - 1) {
                    const int end = min(total, kcap);
                    for (int k = end; k < wpad; k++, dst += kTile) *dst = selfent;
                }
            };
            if (d.idx16) {
                FMD_GLOBAL unsigned short* dst = (FMD_GLOBAL unsigned short*)dtile + (rank % kTile);
                if (compact) emit(dst, BoolC<true>{});
                else emit(dst, BoolC<false>{});
            } else {
                FMD_GLOBAL int* dst = dtile + (rank % kTile);
                if (compact) emit(dst, BoolC<true>{});
                else emit(dst, BoolC<false>{});
            }
        } else if (d.idx16) {
            // rows of the global scan, from this lane's row in the upper half to
            // its column in the lower half: no entry is both read and written
            FMD_GLOBAL unsigned short* dst = (FMD_GLOBAL unsigned short*)dtile + (rank % kTile);
            if (part == 0)
                for (int k = 0; k < wpad; k++)
                    dst[k * kTile] = (unsigned short)(k < stored ? (int)out16[k * kTile] : selfent);
        } else {
            // in place: rows are moved a band of kPlaceBand entries at a time
            // (every read of a band precedes every write)
            FMD_GLOBAL int* dst = dtile + (rank % kTile);
            int maxpad = 0;
#pragma unroll
            for (int w = 0; w < kGroupTiles; w++) maxpad = max(maxpad, s_tlen[w]);
            for (int k0 = 0; k0 < maxpad; k0 += kPlaceBand) {
                int v[kPlaceBand];
#pragma unroll
                for (int e = 0; e < kPlaceBand; e++) {
                    const int k = k0 + e;
                    v[e] = (part == 0 && k < stored) ? out[k * kTile] : selfent;
                }
                __syncthreads();
#pragma unroll
                for (int e = 0; e < kPlaceBand; e++)
                    if (part == 0 && k0 + e < wpad) dst[(k0 + e) * kTile] = v[e];
                __syncthreads();
            }
        }
        if (valid && part == 0) {
            if (total > kcap) err |= ERR_NBR_OVERFLOW;
            gmut(d.nnbr)[i] = stored;
        }
        err = wave_or(err);
        if (err && lane == 0) atomicOr(&st->err, err);
        __syncthreads();  // the next group reuses the LDS
    }
}

// LJ over this atom's Verlet rows (src/force/lj.cu:27-63), in grid units.
// With a = (float)(int)(Xi - Xj) the fixed-point displacement (grid step
// u = L * 2^-32), q = a.a - lo_g is (r^2 - 1e-10) / u^2: the cutoff test
// compares q with thresholds scaled by 1/u^2 (grid_s, grid_inside),
// 1/q = u^2 / r^2 (to a relative 1e-10 / r^2) feeds the LJ terms with
// sigma^2 / u^2 and 24 eps / u^2 folded in, and the force and virial sums are
// kept in grid units and scaled by u and u^2 once per atom.  Every row of a
// wave is padded with the atom itself (q = 0 is rejected) to the wave's
// longest row, a multiple of kLJTail (tlen), so the wave runs whole chunks of
// kLJChunk and at most one of kLJTail, loaded unconditionally, under one
// uniform bound; the next chunk's entries are in flight while the current
// chunk's positions are read.  The cutoff masks 1/q,
// so there is no per-pair branch.  OBS adds the per-atom PE and virial (thermo
// steps and NPT), CAP the push-off pair-force cap, ONE_TYPE a single
// (eps, sigma) pair with eps and sigma nonzero.  With LDS the entries are byte
// offsets into the group's neighbor set staged in LDS (sp); otherwise they are
// slots, read with indexed buffer loads (the hardware scales the slot by the
// 16-byte record).
struct LJSum {
    float fx, fy, fz, pe, w0, w1, w2, w3, w4, w5;  // force, PE and virial of one atom's rows
};

template <bool OBS, bool CAP, bool ONE_TYPE, bool W16, bool LDS>
__device__ __forceinline__ LJSum lj_loop(const RepDesc& d, int lt, int lane, int nw, int4 pi, float L,
                                         const int4* sp) {
    // the tile's rows as a raw buffer: entry k of this lane sits at byte
    // (k * kTile + lane) * entry size; the row offset goes in the scalar
    // offset, so fetching the next chunk costs no vector address arithmetic
    const __amdgpu_buffer_rsrc_t nrs = __builtin_amdgcn_make_buffer_rsrc(
        (void*)(d.nbr + (size_t)lt * d.kcap * kTile), (short)0, d.kcap * kTile * (int)sizeof(int), kBufferWord3);
    const unsigned vlane = (unsigned)lane * (W16 ? 2u : 4u);
    auto entry = [&](int k) -> unsigned {
        if constexpr (W16) return (unsigned)__builtin_amdgcn_raw_buffer_load_b16(nrs, vlane, k * kTile * 2, 0);
        else return __builtin_amdgcn_raw_buffer_load_b32(nrs, vlane, k * kTile * 4, 0);
    };
    const __amdgpu_buffer_rsrc_t prs =
        __builtin_amdgcn_make_buffer_rsrc((void*)d.ipos, (short)sizeof(int4), d.nslots, kBufferWord3);
    const float u = L * 2.3283064365386963e-10f;
    const GridCut gc = grid_cut(d.st);
    const float iu2 = d.st->giu2;
    const float2* ljrow = d.lj + pi.w * d.ntypes;
    const float2 p0 = ONE_TYPE ? d.lj[0] : ljrow[0];
    const float s2g0 = p0.y * p0.y * iu2, c24g0 = 24.0f * p0.x * iu2, c2e0 = 2.0f * p0.x;
    const float capg = CAP ? d.fcap / u : 0.0f;  // fcap / r = (fcap / u) / sqrt(q)
    // one (eps, sigma): force / r = K sr2 sr6 (2 sr6 - 1) with K = 24 eps / sigma^2,
    // summed without K (applied once per atom); the +-1000 clamp becomes +-1000 / K
    constexpr bool fold = ONE_TYPE && !CAP;  // ONE_TYPE only with eps, sigma != 0
    const float kf = fold ? d.lj_kf : 1.0f;
    const float fclamp = fold ? d.lj_fclamp : 1000.0f;
    float gx = 0.f, gy = 0.f, gz = 0.f, pe = 0.f;
    float v0 = 0.f, v1 = 0.f, v2 = 0.f, v3 = 0.f, v4 = 0.f, v5 = 0.f;
    auto pair = [&](const uint4 pj) __attribute__((always_inline)) {
        const float ax = grid_d(pi.x, pj.x), ay = grid_d(pi.y, pj.y), az = grid_d(pi.z, pj.z);
        const float q = grid_s(ax, ay, az, gc.lo_g);
        // forces only, one (eps, sigma): q == 0 may count as inside (its
        // force/r is the clamp and finite), one compare fewer per pair
        const bool in = (fold && !OBS) ? grid_inside0(q, gc.span) : grid_inside(q, gc.span);
        float s2g = s2g0, c24g = c24g0, c2e = c2e0;
        if (!ONE_TYPE) {
            const float2 p = ljrow[pj.w];
            s2g = p.y * p.y * iu2; c24g = 24.0f * p.x * iu2; c2e = 2.0f * p.x;
        }
        const float qinv = in ? __builtin_amdgcn_rcpf(q) : 0.0f;
        const float sr2 = s2g * qinv;
        const float sr6 = sr2 * sr2 * sr2;
        const float sr12 = sr6 * sr6;
        float fr;
        if constexpr (fold) fr = (sr2 * sr6) * fmaf(sr6, 2.0f, -1.0f);  // force / r over K
        else fr = c24g * qinv * (2.0f * sr12 - sr6);        // force / r in real units
        fr = __builtin_amdgcn_fmed3f(fr, -fclamp, fclamp);  // src/force/lj.cu:48
        if (CAP) {
            const float cap = capg * __builtin_amdgcn_rsqf(q);
            fr = fminf(fmaxf(fr, -cap), cap);
        }
        gx += fr * ax; gy += fr * ay; gz += fr * az;
        // keep the type word live so the neighbor read stays 16 bytes:
        // gfx950 serves randomly addressed 12-byte LDS reads at about half
        // the rate of 16-byte ones (the empty asm emits no instruction)
        if constexpr (LDS && ONE_TYPE) asm volatile("" ::"v"(pj.w));
        if (OBS) {
            const float hx = fr * ax, hy = fr * ay, hz = fr * az;
            pe += c2e * (sr12 - sr6);
            v0 += hx * ax; v1 += hx * ay; v2 += hx * az;
            v3 += hy * ay; v4 += hy * az; v5 += hz * az;
        }
    };
    auto neighbor = [&](unsigned e) __attribute__((always_inline)) -> uint4 {
        if constexpr (LDS) {  // the row holds the LDS byte offset of the staged neighbor
            const int4 v = *(const int4*)((const char*)sp + e);
            return make_uint4((unsigned)v.x, (unsigned)v.y, (unsigned)v.z, (unsigned)v.w);
        } else {
            const u32x4 v = struct_load_b128(prs, e, 0, 0, 0);
            return make_uint4(v[0], v[1], v[2], v[3]);
        }
    };
    // nw, the wave's padded row length (a multiple of kLJTail, the same for
    // every lane: the list build pads each row of a wave to it), bounds whole
    // chunks of kLJChunk and a last chunk of kLJTail; entries fetched past nw
    // (within the row area, or zero from the bounded buffer) are never used
    unsigned nxt[kLJChunk];
    if (nw > 0) {
#pragma unroll
        for (int k = 0; k < kLJChunk; k++) nxt[k] = entry(k);
    }
    int k0 = 0;
    for (; k0 + kLJChunk <= nw; k0 += kLJChunk) {
        uint4 pjs[kLJChunk];
#pragma unroll
        for (int k = 0; k < kLJChunk; k++) pjs[k] = neighbor(nxt[k]);
        if (k0 + kLJChunk < nw) {
#pragma unroll
            for (int k = 0; k < kLJChunk; k++) nxt[k] = entry(k0 + kLJChunk + k);
        }
#pragma unroll
        for (int k = 0; k < kLJChunk; k++) pair(pjs[k]);
    }
    if (k0 < nw) {  // nw - k0 == kLJTail
        uint4 pjs[kLJTail];
#pragma unroll
        for (int k = 0; k < kLJTail; k++) pjs[k] = neighbor(nxt[k]);
#pragma unroll
        for (int k = 0; k < kLJTail; k++) pair(pjs[k]);
    }
    const float fu = kf * u, hu2 = 0.5f * kf * u * u;
    return LJSum{gx * fu, gy * fu, gz * fu, pe, v0 * hu2, v1 * hu2, v2 * hu2, v3 * hu2, v4 * hu2, v5 * hu2};
}

#define LJ_ARGS d, t.lt, lane, nw, pi, L, sp
template <bool W16, bool LDS>
__device__ __forceinline__ LJSum lj_variants(const RepDesc& d, const Tile& t, int lane, int nw, int4 pi,
                                             float L, bool obs, const int4* sp) {
    const bool cap = d.fcap > 0.0f, one = d.lj_kf != 0.0f;  // set for one (eps, sigma), neither zero
    if (!cap && one)
        return obs ? lj_loop<true, false, true, W16, LDS>(LJ_ARGS) : lj_loop<false, false, true, W16, LDS>(LJ_ARGS);
    if (!cap)
        return obs ? lj_loop<true, false, false, W16, LDS>(LJ_ARGS)
                   : lj_loop<false, false, false, W16, LDS>(LJ_ARGS);
    return obs ? lj_loop<true, true, false, W16, LDS>(LJ_ARGS) : lj_loop<false, true, false, W16, LDS>(LJ_ARGS);
}
#undef LJ_ARGS

// Tabulated pairs over the same Verlet rows (src/force/table.cu:58-118).  A
// pair inside the cutoff (the grid-unit test of the LJ loop) whose types have a
// table gets the linear interpolant of force / r and energy at r clamped to
// [rmin, rmax]: node k sits at rmin + k dr, k = (int)((r - rmin) / dr) clamped
// to [0, n - 2], weight t = (r - (rmin + k dr)) / dr.  Half the pair energy and
// half the pair virial go to this atom, as in the LJ loop.
// What bounds it is the chain of loads of a pair (its entry, the neighbor, the
// table of the types, the two nodes), so kTabChunk pairs go through each step
// together, pairs that do not count included, the next ones' entries requested
// meanwhile.
constexpr int kTabChunk = 4;
template <bool W16, bool LDS>
__device__ __forceinline__ LJSum table_loop(const RepDesc& d, int lt, int lane, int i, int4 pi, float L,
                                            const int4* sp) {
    const int nn = d.nnbr[i];
    const FMD_GLOBAL int* nl = gview(d.nbr) + (size_t)lt * d.kcap * kTile + lane;
    const FMD_GLOBAL unsigned short* nl16 =
        (const FMD_GLOBAL unsigned short*)(gview(d.nbr) + (size_t)lt * d.kcap * kTile) + lane;
    const float u = L * 2.3283064365386963e-10f;
    const GridCut gc = grid_cut(d.st);
    const FMD_GLOBAL int* trow = gview(d.tab_idx) + pi.w * d.ntypes;
    // nodes k and k + 1 in one load (8-byte aligned)
    typedef f32x4 f32x4_8 __attribute__((aligned(8)));
    const FMD_GLOBAL char* fe = (const FMD_GLOBAL char*)gview(d.tab_fe);
    LJSum s{0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
    int nxt[kTabChunk];
    auto fetch = [&](int k0) __attribute__((always_inline)) {
#pragma unroll
        for (int k = 0; k < kTabChunk; k++) {
            const int q = min(k0 + k, nn - 1);
            nxt[k] = W16 ? (int)nl16[q * kTile] : nl[q * kTile];
        }
    };
    if (nn > 0) fetch(0);
    for (int k0 = 0; k0 < nn; k0 += kTabChunk) {
        int tb[kTabChunk];
        float r[kTabChunk], dx[kTabChunk], dy[kTabChunk], dz[kTabChunk];
        unsigned in = 0u;
#pragma unroll
        for (int k = 0; k < kTabChunk; k++) {
            // LDS byte offset or slot
            const f32x4 v = LDS ? *(const f32x4*)((const char*)sp + nxt[k]) : raw4(d.ipos)[nxt[k]];
            const float ax = grid_d(pi.x, __float_as_uint(v.x)), ay = grid_d(pi.y, __float_as_uint(v.y)),
                        az = grid_d(pi.z, __float_as_uint(v.z));
            in |= (k0 + k < nn && grid_inside(grid_s(ax, ay, az, gc.lo_g), gc.span)) ? 1u << k : 0u;
            dx[k] = ax * u; dy[k] = ay * u; dz[k] = az * u;
            tb[k] = trow[__float_as_int(v.w)];
        }
        if (k0 + kTabChunk < nn) fetch(k0 + kTabChunk);
        f32x4 p[kTabChunk];
        float t[kTabChunk];
#pragma unroll
        for (int k = 0; k < kTabChunk; k++) {
            if (tb[k] < 0) in &= ~(1u << k);
            const int tab = max(tb[k], 0);
            const f32x4 tp = raw4(d.tab_parm)[tab];
            const f32x2 tn = ((const FMD_GLOBAL f32x2*)gview(d.tab_no))[tab];  // (points, offset)
            r[k] = fminf(fmaxf(sqrtf(sq3(dx[k], dy[k], dz[k])), tp.x), tp.y);
            const int idx = min(max((int)((r[k] - tp.x) * tp.w), 0), __float_as_int(tn.x) - 2);
            t[k] = (r[k] - (tp.x + (float)idx * tp.z)) * tp.w;
            p[k] = *(const FMD_GLOBAL f32x4_8*)(fe + (size_t)(__float_as_int(tn.y) + idx) * 8);
        }
#pragma unroll
        for (int k = 0; k < kTabChunk; k++)
            if ((in >> k) & 1u) {
                const float fs = p[k].x + t[k] * (p[k].z - p[k].x);
                const float e = p[k].y + t[k] * (p[k].w - p[k].y);
                const float hx = 0.5f * fs * dx[k], hy = 0.5f * fs * dy[k], hz = 0.5f * fs * dz[k];
                s.fx += fs * dx[k]; s.fy += fs * dy[k]; s.fz += fs * dz[k];
                s.pe += 0.5f * e;
                s.w0 += hx * dx[k]; s.w1 += hx * dy[k]; s.w2 += hx * dz[k];
                s.w3 += hy * dy[k]; s.w4 += hy * dz[k]; s.w5 += hz * dz[k];
            }
    }
    return s;
}

// atan2(y, x) for y >= 0, the angle between two bond vectors in [0, pi], by
// the range reduction and polynomial of the Cephes atanf (S. L. Moshier): the
// ratio r = min(|x|, y) / max(|x|, y) in [0, 1] becomes t = (r - 1) / (r + 1)
// above tan(pi/8), atan(t) = t + t z P(z) with z = t^2, then the octant is
// undone.  Within 4 ulp of an FP64 atan2 on random pairs; near a straight
// angle (small y, x < 0) within one ulp of pi.
__device__ __forceinline__ float angle_atan2(float y, float x) {
    const float ax = fabsf(x);
    const float mn = fminf(ax, y), mx = fmaxf(ax, y);
    const float r = mx > 0.0f ? mn * __builtin_amdgcn_rcpf(mx) : 0.0f;
    const bool big = r > 0.41421356237f;  // tan(pi/8)
    const float t = big ? (r - 1.0f) * __builtin_amdgcn_rcpf(r + 1.0f) : r;
    const float z = t * t;
    const float p = fmaf(fmaf(fmaf(8.05374449538e-2f, z, -1.38776856032e-1f), z, 1.99777106478e-1f), z,
                         -3.33329491539e-1f);
    float a = fmaf(p * z, t, t);
    if (big) a += 0.78539816339744831f;     // pi/4
    if (y > ax) a = 1.5707963267948966f - a;  // pi/2
    if (x < 0.0f) a = 3.1415926535897931f - a;
    return a;
}

// ---------------------------------------------------------------------------
// Force kernel: LJ over the Verlet list (src/force/lj.cu:27-63), FENE+WCA
// (src/force/fene.cu:21-65) and harmonic angle (src/force/angle.cu:22-79) as
// per-atom gathers (no float atomics), then the post-force half kick
// (src/integrate/langevin.cu:109-130).  Writes force[i] = (F, pe_i) and 13
// FP64 partials per wave: pe, virial[6], kinetic tensor[6] (after the kick).
// ---------------------------------------------------------------------------
//
// TAB includes the tabulated pairs, for batches with such a replica: they need
// more registers than the 80 of six waves per SIMD, which the others keep.
// 9,000 beads with a table on half the pairs: 97.4 us per step with the pairs
// one after the other in the one kernel, 67.9 in this form (four at a time; two
// 73, eight spill: 102); without the table code the others' kernel is also
// shorter (128 uneven replicas 355 -> 350 us per step, NPT 120,000 68.3 -> 66.8).
template <int TERMS, bool LIST = false, bool TAB = false>
__global__ void __launch_bounds__(kMaxBlockK) __attribute__((amdgpu_waves_per_eu(TAB ? 4 : 6, 8)))
k_force(const RepDesc* __restrict__ descs, const Tile* __restrict__ tiles, int t0, int ntl, int kick, int mode,
        int sel, const int* __restrict__ rlist, const int* __restrict__ nrt) {
    constexpr int terms = TERMS;
    __shared__ int4 s_pos[(TERMS & 1) ? kGroupStage : 1];  // the group's neighbor set
    // One tile per wave.  t0 and ntl are whole groups and a workgroup (1, 2 or
    // 4 waves) lies in one group, so the returns below are uniform over the
    // workgroup.
    auto tile = [&](int w) __attribute__((always_inline)) {
        const Tile t = tiles[w];
        const RepDesc& d = descs[t.rep];
        RepState* st = d.st;
        const int lane = lane_id();
        const int grp = t.lt / kGroupTiles;
        // requested together, before the replica's flags are looked at
        const int active = st->active, rebuild = st->rebuild;
        const int perm = gview(d.gperm)[t.lt * kTile + lane];
        const int nst = (terms & 1) ? gview(d.gcount)[grp] : -1;
        const int nw = (terms & 1) ? __builtin_amdgcn_readfirstlane(gview(d.tlen)[t.lt]) : 0;  // uniform: scalar loop control
        if (mode == FM_STEP && !active) return;
        if (sel == FS_STAYING && rebuild) return;
        // this lane computes the atom whose row the list build placed in its column
        const int i = grp * kGroupSlots + perm;
        // stage the group's neighbor set (coalesced slot list, one 16-byte position each)
        if (nst >= 0) {
            const int nth = blockDim.x, last = nst - 1;
            const FMD_GLOBAL int4* gp = gview(d.ipos);
            auto stage = [&](auto gs) {  // four slots, then four positions, in flight at once
                for (int q = threadIdx.x; q < nst; q += 4 * nth) {
                    const int qb = q + nth, qc = q + 2 * nth, qd = q + 3 * nth;
                    const int sa = gs[q], sb = gs[min(qb, last)], sc = gs[min(qc, last)], sd = gs[min(qd, last)];
                    const int4 va = gp[sa], vb = gp[sb], vc = gp[sc], vd = gp[sd];
                    s_pos[q] = va;
                    if (qb < nst) s_pos[qb] = vb;
                    if (qc < nst) s_pos[qc] = vc;
                    if (qd < nst) s_pos[qd] = vd;
                }
            };
            if (d.idx16) stage((const FMD_GLOBAL unsigned short*)gview(d.gstage) + (size_t)grp * kGroupStage);
            else stage(gview(d.gstage) + (size_t)grp * kGroupStage);
            __syncthreads();
        }
        const int4* sp = nst >= 0 ? s_pos : nullptr;
        float fx = 0.f, fy = 0.f, fz = 0.f, pe = 0.f;
        float w0 = 0.f, w1 = 0.f, w2 = 0.f, w3 = 0.f, w4 = 0.f, w5 = 0.f;
        // Langevin steps that record nothing need none of the FP64 partials (no
        // thermostat reads the kinetic energy; the host reevaluates unobserved
        // steps on request), and neither does a forces-only launch
        const bool partials = mode == FM_OBS || (mode == FM_STEP && (d.ensemble != 0 || st->want_obs));
        double k0 = 0, k1 = 0, k2 = 0, k3 = 0, k4 = 0, k5 = 0;
        double vkey = 0.0, fkey = 0.0;  // max_key of |v|^2 and |F|^2 (src/analysis/thermo.cu:26-75)
        int err = 0;
        if (i < d.natoms) {
            const int4 pi = d.ipos[i];
            const int ti = pi.w;
            const float L = st->Lp;
            const float ulen = L * 2.3283064365386963e-10f;  // fixed-point step, L * 2^-32
            const bool obs = (mode == FM_OBS) || (mode == FM_STEP && st->want_obs);
            if (terms & 1) {
                LJSum a;
                if (sp) {  // the array itself: its LDS address is a constant of the kernel
                    if (d.idx16) a = lj_variants<true, true>(d, t, lane, nw, pi, L, obs, s_pos);
                    else a = lj_variants<false, true>(d, t, lane, nw, pi, L, obs, s_pos);
                } else {
                    if (d.idx16) a = lj_variants<true, false>(d, t, lane, nw, pi, L, obs, sp);
                    else a = lj_variants<false, false>(d, t, lane, nw, pi, L, obs, sp);
                }
                fx = a.fx; fy = a.fy; fz = a.fz; pe = a.pe;
                w0 = a.w0; w1 = a.w1; w2 = a.w2; w3 = a.w3; w4 = a.w4; w5 = a.w5;
                if (TAB && d.ntables) {
                    const LJSum b = sp ? (d.idx16 ? table_loop<true, true>(d, t.lt, lane, i, pi, L, s_pos)
                                                  : table_loop<false, true>(d, t.lt, lane, i, pi, L, s_pos))
                                       : (d.idx16 ? table_loop<true, false>(d, t.lt, lane, i, pi, L, sp)
                                                  : table_loop<false, false>(d, t.lt, lane, i, pi, L, sp));
                    fx += b.fx; fy += b.fy; fz += b.fz; pe += b.pe;
                    w0 += b.w0; w1 += b.w1; w2 += b.w2; w3 += b.w3; w4 += b.w4; w5 += b.w5;
                }
            }
            const int hdr = (terms & 6) ? d.bhdr[i] : 0;
            // a bonded entry of a staged group is the partner's LDS byte offset in
            // the group's neighbor set (read from the set, or through its slot
            // list when this variant did not stage it); otherwise a slot
            const bool bstaged = (terms & 6) && (sp || d.gcount[grp] >= 0);
            const FMD_GLOBAL unsigned short* gs16 =
                (const FMD_GLOBAL unsigned short*)gview(d.gstage) + (size_t)grp * kGroupStage;
            const FMD_GLOBAL int* gs32 = gview(d.gstage) + (size_t)grp * kGroupStage;
            auto partner = [&](int e) __attribute__((always_inline)) -> int4 {
                const int v = e & kSlotMask;
                if (sp) return *(const int4*)((const char*)s_pos + v);
                if (bstaged) return d.ipos[d.idx16 ? (int)gs16[v >> 4] : gs32[v >> 4]];
                return d.ipos[v];
            };
            // The bonded terms in the order bonds, then angles, each over its rows;
            // the entries and partner positions of the first kBondAhead bonds and
            // kAngleAhead angles (all of a Kremer-Grest bead's) are requested
            // together, so their latencies overlap instead of forming one chain per
            // term.
            const int nb = (terms & 2) ? (hdr & 0xFF) : 0;
            const int na = (terms & 4) ? ((hdr >> 8) & 0xFF) : 0;
            const int* bt = d.bnd + (size_t)(i / kTile) * d.bcap * kTile + (i % kTile);
            const int2* at = d.ang + (size_t)(i / kTile) * d.acap * kTile + (i % kTile);
            auto bond_term = [&](int e, int4 pj) __attribute__((always_inline)) {
                const float4 bp = d.bparm[(unsigned)e >> kSlotBits];
                const float dx = fix_diff(pi.x, pj.x, ulen);
                const float dy = fix_diff(pi.y, pj.y, ulen);
                const float dz = fix_diff(pi.z, pj.z, ulen);
                float r2 = sq3(dx, dy, dz);
                const float R02 = bp.y * bp.y;
                // a bond at or beyond R0 is a failure of the run, except during the
                // capped soft push-off, where the clamp below keeps it finite
                if (!(r2 < R02) && !(d.fcap > 0.0f)) err |= ERR_STRETCH;
                r2 = fminf(fmaxf(r2, 1e-6f), R02 * 0.9999f);  // src/force/fene.cu:33
                // divisions as hardware reciprocals (1 ulp), as the reference's
                // fast-math build does; PE and virial only where observed
                float ff = -bp.x * R02 * __builtin_amdgcn_rcpf(R02 - r2);
                const float sig2 = bp.w * bp.w;
                const bool wca = r2 < sig2 * 1.2599210498948732f;
                float sr6 = 0.0f, sr12 = 0.0f;
                if (wca) {
                    const float r2inv = __builtin_amdgcn_rcpf(r2);
                    const float sr2 = sig2 * r2inv;
                    sr6 = sr2 * sr2 * sr2;
                    sr12 = sr6 * sr6;
                    ff += 24.0f * bp.z * r2inv * (2.0f * sr12 - sr6);
                }
                fx += ff * dx; fy += ff * dy; fz += ff * dz;
                if (obs) {
                    float bpe = -0.5f * bp.x * R02 * logf(1.0f - r2 / R02);
                    if (wca) bpe += 4.0f * bp.z * (sr12 - sr6) + bp.z;
                    const float hx = 0.5f * ff * dx, hy = 0.5f * ff * dy, hz = 0.5f * ff * dz;
                    pe += 0.5f * bpe;
                    w0 += hx * dx; w1 += hx * dy; w2 += hx * dz;
                    w3 += hy * dy; w4 += hy * dz; w5 += hz * dz;
                }
            };
            auto angle_term = [&](int2 e, int4 q1, int4 q2) __attribute__((always_inline)) {
                const int role = (unsigned)e.x >> kSlotBits;
                const float2 ap = d.aparm[(unsigned)e.y >> kSlotBits];
                // angle atoms (A, B=center, C) from this atom's role
                // (assignments, not conditionals of two lvalues: a select of
                // addresses would keep pi in scratch memory)
                int4 pa = q1, pb = q1, pc = q2;
                if (role == 0) pa = pi;
                if (role == 1) pb = pi;
                else if (role == 2) pb = q2;
                if (role == 2) pc = pi;
                const float ax = fix_diff(pa.x, pb.x, ulen);
                const float ay = fix_diff(pa.y, pb.y, ulen);
                const float az = fix_diff(pa.z, pb.z, ulen);
                const float bx = fix_diff(pc.x, pb.x, ulen);
                const float by = fix_diff(pc.y, pb.y, ulen);
                const float bz = fix_diff(pc.z, pb.z, ulen);
                const float ra2 = ax * ax + ay * ay + az * az;
                const float rb2 = bx * bx + by * by + bz * bz;
                const float cxp = ay * bz - az * by, cyp = az * bx - ax * bz, czp = ax * by - ay * bx;
                const float cr = sqrtf(cxp * cxp + cyp * cyp + czp * czp);
                const float dot = ax * bx + ay * by + az * bz;
                const float theta = angle_atan2(cr, dot);
                const float inv_ab = rsqrtf(ra2) * rsqrtf(rb2);
                const float c = dot * inv_ab;
                const float s = fmaxf(cr * inv_ab, 1e-6f);
                const float dth = theta - ap.y;
                const float pref = 2.0f * ap.x * dth * __builtin_amdgcn_rcpf(s);
                const float ia2 = __builtin_amdgcn_rcpf(ra2), ib2 = __builtin_amdgcn_rcpf(rb2);
                const float fix = pref * (bx * inv_ab - c * ax * ia2);
                const float fiy = pref * (by * inv_ab - c * ay * ia2);
                const float fiz = pref * (bz * inv_ab - c * az * ia2);
                const float fkx = pref * (ax * inv_ab - c * bx * ib2);
                const float fky = pref * (ay * inv_ab - c * by * ib2);
                const float fkz = pref * (az * inv_ab - c * bz * ib2);
                if (role == 0) { fx += fix; fy += fiy; fz += fiz; }
                else if (role == 2) { fx += fkx; fy += fky; fz += fkz; }
                else { fx -= fix + fkx; fy -= fiy + fky; fz -= fiz + fkz; }
                if (obs) {
                    const float third = 1.0f / 3.0f;
                    pe += ap.x * dth * dth * third;
                    w0 += (fix * ax + fkx * bx) * third;
                    w1 += (fix * ay + fkx * by) * third;
                    w2 += (fix * az + fkx * bz) * third;
                    w3 += (fiy * ay + fky * by) * third;
                    w4 += (fiy * az + fky * bz) * third;
                    w5 += (fiz * az + fkz * bz) * third;
                }
            };
            constexpr int kBondAhead = 2, kAngleAhead = 3;
            const int eb0 = (nb > 0) ? bt[0] : 0, eb1 = (nb > 1) ? bt[kTile] : 0;
            const int2 ea0 = (na > 0) ? at[0] : make_int2(0, 0), ea1 = (na > 1) ? at[kTile] : make_int2(0, 0),
                       ea2 = (na > 2) ? at[2 * kTile] : make_int2(0, 0);
            int4 pb0 = pi, pb1 = pi, qa0 = pi, qc0 = pi, qa1 = pi, qc1 = pi, qa2 = pi, qc2 = pi;
            if (nb > 0) pb0 = partner(eb0);
            if (nb > 1) pb1 = partner(eb1);
            if (na > 0) { qa0 = partner(ea0.x); qc0 = partner(ea0.y); }
            if (na > 1) { qa1 = partner(ea1.x); qc1 = partner(ea1.y); }
            if (na > 2) { qa2 = partner(ea2.x); qc2 = partner(ea2.y); }
            if (nb > 0) bond_term(eb0, pb0);
            if (nb > 1) bond_term(eb1, pb1);
            for (int b = kBondAhead; b < nb; b++) {
                const int e = bt[b * kTile];
                bond_term(e, partner(e));
            }
            if (na > 0) angle_term(ea0, qa0, qc0);
            if (na > 1) angle_term(ea1, qa1, qc1);
            if (na > 2) angle_term(ea2, qa2, qc2);
            for (int a = kAngleAhead; a < na; a++) {
                const int2 e = at[a * kTile];
                angle_term(e, partner(e.x), partner(e.y));
            }
            // Langevin steps followed by another step of the run also give that
            // step's pre-force half kick (the same force, the same operations as
            // k_pre), so the force need not be stored and read back; the kinetic
            // partials are taken between the two kicks
            const bool ahead = kick && mode == FM_STEP && d.ensemble == 0 && st->step + 1 < st->stop;
            if (!ahead) d.force[i] = make_float4(fx, fy, fz, pe);
            float4 v = d.vel[i];
            const float m = d.mass[ti];
            const float hdtm = d.half_dt / m;
            if (kick) { v.x = fmaf(hdtm, fx, v.x); v.y = fmaf(hdtm, fy, v.y); v.z = fmaf(hdtm, fz, v.z); }
            if (partials) {
                const double md = m, vx = v.x, vy = v.y, vz = v.z;
                k0 = md * vx * vx; k1 = md * vx * vy; k2 = md * vx * vz;
                k3 = md * vy * vy; k4 = md * vy * vz; k5 = md * vz * vz;
                const int g = d.gid[i];
                vkey = max_key(v.x * v.x + v.y * v.y + v.z * v.z, g);
                fkey = max_key(fx * fx + fy * fy + fz * fz, g);
            }
            if (ahead) {  // bit for bit the kick of k_pre (explicit FMAs there too)
                v.x = fmaf(hdtm, fx, v.x); v.y = fmaf(hdtm, fy, v.y); v.z = fmaf(hdtm, fz, v.z);
                if (d.vlim > 0.0f) v = limit_speed(v, d.vlim);
            }
            if (kick) d.vel[i] = v;
        }
        if (partials) {
            double part[kNumSum] = {(double)pe, (double)w0, (double)w1, (double)w2, (double)w3, (double)w4,
                                    (double)w5, k0, k1, k2, k3, k4, k5};
#pragma unroll
            for (int c = 0; c < kNumSum; c++) part[c] = wave_sum_last(part[c]);
            vkey = wave_max_last(vkey);
            fkey = wave_max_last(fkey);
            if (lane == 63) {
#pragma unroll
                for (int c = 0; c < kNumSum; c++) d.wpart[(size_t)t.lt * kNumPart + c] = part[c];
                d.wpart[(size_t)t.lt * kNumPart + kNumSum] = vkey;
                d.wpart[(size_t)t.lt * kNumPart + kNumSum + 1] = fkey;
            }
        }
        if (err) atomicOr(&st->err, err);  // failures only
    };
    if constexpr (LIST) {
        // the listed tiles (the rebuild phases' list): each workgroup (four
        // waves: one group) takes listed groups in turn, the workgroups of one
        // XCD (a multiple of kXcds in the grid) from one contiguous eighth of
        // the list, so a replica's positions are gathered through one L2
        const int ng = *nrt / kGroupTiles, per = (ng + kXcds - 1) / kXcds, x = blockIdx.x % kXcds;
        const int g1 = min((x + 1) * per, ng), gs = gridDim.x / kXcds;
        for (int g = x * per + blockIdx.x / kXcds; g < g1; g += gs) {
            tile(rlist[g * kGroupTiles + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6)]);
            __syncthreads();  // the next group's staging reuses s_pos
        }
    } else {
        // the grid's wave w takes tile t0 + w
        const int w = t0 + xcd_wave_in_grid();
        if (w < t0 + ntl) tile(w);
    }
}

// First reduction level: one workgroup sums the FP64 partials of kChunkTiles
// tiles of one replica in a fixed order (thread t takes tile t, then the DPP
// wave sum, then the four waves in order), so a large replica's sum is spread
// over many CUs.
// The sum of one chunk, by a workgroup of 256 threads, to out[0 .. kNumSum + 1].
__device__ __forceinline__ void chunk_sum(const RepDesc& d, int chunk, double (*red)[4], double* out) {
    constexpr int kN = kNumSum + 2;
    const int tl = chunk * kChunkTiles + threadIdx.x;
    double a[kN];
#pragma unroll
    for (int c = 0; c < kN; c++) a[c] = 0.0;
    if (tl < d.ntiles)
#pragma unroll
        for (int c = 0; c < kN; c++) a[c] = gview(d.wpart)[(size_t)tl * kNumPart + c];
#pragma unroll
    for (int c = 0; c < kN; c++) a[c] = c < kNumSum ? wave_sum_last(a[c]) : wave_max_last(a[c]);
    if (lane_id() == 63)
#pragma unroll
        for (int c = 0; c < kN; c++) red[c][threadIdx.x >> 6] = a[c];
    __syncthreads();
    if (threadIdx.x < kN) {
        const int c = threadIdx.x;
        out[c] = c < kNumSum ? ((red[c][0] + red[c][1]) + red[c][2]) + red[c][3]
                             : fmax(fmax(red[c][0], red[c][1]), fmax(red[c][2], red[c][3]));
    }
}
__global__ void __launch_bounds__(256) k_chunk(const RepDesc* __restrict__ descs,
                                              const Tile* __restrict__ chunks, int nch, int mode) {
    __shared__ double red[kNumSum + 2][4];
    const Tile ch = chunks[blockIdx.x];
    const RepDesc& d = descs[ch.rep];
    if (mode == BND_STEP && (!d.st->active || (d.ensemble == 0 && !d.st->want_obs))) return;  // nothing to sum
    chunk_sum(d, ch.lt, red, d.cpart + (size_t)ch.lt * kNumPart);
}

// Multiple-tau correlator push (src/analysis/correlator.cu:33-92), by the
// whole block: at each level thread (lag, c) adds sample * the sample lag
// pushes back (lags up to the ring's insert position, as the reference
// counts them), then thread 0 advances the ring and the block accumulator,
// which hands its mean to the next level every kCorrPoints samples.  smp is
// the sample (shared) and is replaced by the block mean on the way up.
__device__ void corr_push(CorrState* cs, double* smp) {
    __shared__ int cont;
    const int t = threadIdx.x, lag = t / 6, c = t % 6;
    for (int lv = 0; lv < kCorrLevels; lv++) {
        const int idx = cs->ins[lv];
        if (t < kCorrPoints * 6) {
            const double x = smp[c];
            const int base = lv * kCorrPoints;
            if (lag == 0) cs->buf[(base + idx) * 6 + c] = x;
            if (lag <= idx) {
                const double o = (lag == 0) ? x : cs->buf[(base + idx - lag) * 6 + c];
                cs->corr[(base + lag) * 6 + c] += x * o;
                if (c == 0) cs->counts[base + lag]++;
            }
        }
        __syncthreads();
        if (t == 0) {
            cs->ins[lv] = (idx + 1) % kCorrPoints;
            const int n = cs->bcount[lv] + 1;
            for (int k = 0; k < 6; k++) cs->acc[lv * 6 + k] += smp[k];
            cont = n >= kCorrPoints;
            if (cont) {
                for (int k = 0; k < 6; k++) {
                    smp[k] = cs->acc[lv * 6 + k] / (double)kCorrPoints;
                    cs->acc[lv * 6 + k] = 0.0;
                }
            }
            cs->bcount[lv] = cont ? 0 : n;
        }
        __syncthreads();
        if (!cont) break;
    }
}

__global__ void __launch_bounds__(128) k_corr_push(const RepDesc* __restrict__ d, Sample6 x) {
    __shared__ double smp[6];
    if (threadIdx.x < 6) smp[threadIdx.x] = x.v[threadIdx.x];
    __syncthreads();
    corr_push(d->corr, smp);
}

// The step's chain applications on a stream of kinetic energies, one lane,
// state carried from draw to draw (the device chain of nh_propagate_chain_kernel,
// src/integrate/nose_hoover.cu:86-178, as tests/test_nose_hoover.cu:343-439
// drives it).  carry = 0: one application per draw with KE ke[t]; carry = 1:
// two per draw, the post-force one with ke[t] and then the next pre-force one
// with the scaled kinetic energy ke[t] s^2 it leaves (chain_KE_carry).
__global__ void __launch_bounds__(64) k_nh_chain_run(RepState* st, const double* __restrict__ ke, int n,
                                                     int carry, double kT, int natoms, double half_dt,
                                                     double* __restrict__ scales) {
    if (threadIdx.x != 0) return;
    for (int t = 0; t < n; t++) {
        const double s = nh_chain(st, ke[t], kT, natoms, half_dt);
        if (carry) {
            scales[2 * t] = s;
            scales[2 * t + 1] = nh_chain(st, ke[t] * s * s, kT, natoms, half_dt);
        } else {
            scales[t] = s;
        }
    }
}

// Scalar tail of the per-replica boundary (thread 0): the post-force chain /
// barostat of this step, start-of-step scalars of the next, thermo record,
// step counter.  Returns 1 when this step's pressure tensor is a correlator
// sample (written to smp).
__device__ int boundary_tail(const RepDesc& d, RepState* st, int mode, const double (*red)[kBndThreads / 64],
                             double* smp) {
    double tot[kNumSum + 2];
#pragma unroll
    for (int c = 0; c < kNumSum + 2; c++) {
        tot[c] = 0.0;
#pragma unroll
        for (int w = 0; w < kBndThreads / 64; w++) tot[c] = c < kNumSum ? tot[c] + red[c][w] : fmax(tot[c], red[c][w]);
    }
    const double pe = tot[0];
    double W[6], K[6];
#pragma unroll
    for (int c = 0; c < 6; c++) { W[c] = tot[1 + c]; K[c] = tot[7 + c]; }
    const double KE = 0.5 * (K[0] + K[3] + K[5]);
    const bool reduced = !(mode == BND_STEP && d.ensemble == 0 && !st->want_obs);
    if (reduced) {
        st->vkey = tot[kNumSum];
        st->fkey = tot[kNumSum + 1];
    }
    if (mode == BND_REDUCE) {
        st->obs_step = st->step;
        st->pe = pe;
        for (int c = 0; c < 6; c++) { st->vir[c] = W[c]; st->kin[c] = K[c] * (double)st->v_pending * (double)st->v_pending; }
        return 0;
    }
    if (mode == BND_PRIME) {
        st->obs_step = st->step;
        st->pe = pe;
        for (int c = 0; c < 6; c++) { st->vir[c] = W[c]; st->kin[c] = K[c]; }
        st->ke_carry = KE;  // src/main.cu:373-386
        st->v_pending = 1.0f;
        st->rec_step = st->step;
        st->pre_ready = 0;
        return 0;
    }
    // BND_STEP: end of step cur
    const int64_t cur = st->step + 1;
    const double hdt = 0.5 * (double)d.dt, dt = (double)d.dt;
    double ks = 1.0;
    if (d.ensemble == 1) {
        const float frac = (float)(cur - 1) / (float)st->ramp_n;
        const float T = (float)st->T_start + ((float)st->T_stop - (float)st->T_start) * frac;
        const double s = nh_chain(st, KE, (double)T, d.natoms, hdt);
        st->ke_carry = KE * s * s;
        ks = s;
    } else if (d.ensemble == 2) {
        const float frac = (float)(cur - 1) / (float)st->ramp_n;
        const float T = (float)st->T_start + ((float)st->T_stop - (float)st->T_start) * frac;
        const float P = (float)st->P_start + ((float)st->P_stop - (float)st->P_start) * frac;
        const BaroOut o = npt_chain_baro(st, KE, W[0] + W[3] + W[5], true, (double)T, (double)P,
                                         d.natoms, hdt, dt);
        st->ke_carry = o.KE_scaled * o.nh_scale * o.nh_scale;
        ks = o.baro_scale * o.nh_scale;
        st->L = (float)o.L;
        st->invL = 1.0f / st->L;
    }
    st->v_pending = (float)ks;
    const double ks2 = (double)st->v_pending * (double)st->v_pending;
    if (d.ensemble != 0 || st->want_obs)  // else this step reduced no partials
        for (int c = 0; c < 6; c++) st->kin[c] = K[c] * ks2;
    if (st->want_obs) {
        st->pe = pe;
        for (int c = 0; c < 6; c++) st->vir[c] = W[c];
        st->obs_step = cur;
    }
    st->step = cur;
    st->rec_step = cur;
    const double Ld = (double)st->L, V = Ld * Ld * Ld;
    if (st->want_obs && st->thermo_freq > 0 && (cur % st->thermo_freq) == 0 && st->thermo_cap > 0) {
        ThermoRec r;
        const double N = (double)d.natoms;
        r.step = cur;
        r.ke = 0.5 * (st->kin[0] + st->kin[3] + st->kin[5]) / N;
        r.pe = pe / N;
        r.temp = 2.0 * r.ke / 3.0;  // src/analysis/thermo.cu:178
        for (int c = 0; c < 6; c++) r.press[c] = (st->kin[c] + W[c]) / V;
        r.L = Ld;
        float m2;
        int g;
        max_key_split(st->vkey, &m2, &g);
        r.maxv = sqrt((double)m2) * (double)st->v_pending;
        r.maxv_id = g;
        max_key_split(st->fkey, &m2, &g);
        r.maxf = sqrt((double)m2);
        r.maxf_id = g;
        d.thermo[st->thermo_written % st->thermo_cap] = r;
        st->thermo_written++;
    }
    // stress sample: the pressure tensor of the thermo record (src/main.cu:633,658-664)
    const int sample = d.corr && st->stress_freq > 0 && (cur % st->stress_freq) == 0;
    if (sample)
        for (int c = 0; c < 6; c++) smp[c] = (st->kin[c] + W[c]) / V;
    // the force pass of this step kicked ahead exactly when another step follows
    st->kicked = (d.ensemble == 0 && cur < st->stop) ? 1 : 0;
    // a neighbor overflow (list build) or an overstretched bond (force pass)
    // found during this step stops the replica at the end of it
    if (cur >= st->stop || st->err) {
        st->active = 0;
        st->pre_ready = 0;
    } else {
        start_step(d, st, cur + 1);
    }
    return sample;
}

// ---------------------------------------------------------------------------
// Per-replica boundary: fixed-order FP64 reduction of the wave partials, then
// the scalar integrator work and records (boundary_tail), then the stress
// correlator push on sample steps.
// ---------------------------------------------------------------------------
// The scalar part is one lane's chain of FP64 arithmetic: it works on a copy of
// the replica's state in LDS, read and written back by the whole workgroup (one
// trip to memory each way instead of one per dependent field).  With FUSED (a
// batch of replicas of at most kFusedChunks chunks) the first reduction level
// is done here too, chunk after chunk, instead of by a k_chunk launch: worth the
// launch for one chunk, or for several where most steps sum nothing (no chain
// reads the kinetic energy, no record or sample on every step), but two chunks
// one after the other take longer than the launch (30,000 beads NVT 50.4 us per
// step against 49.2; four with a record a step, 60,000 beads, 49.6 against
// 45.1).  Together per step: 2,000 beads 31.5 -> 28.6 us, 30,000 44.5 -> 41.7,
// NPT 120,000 72.1 -> 69.1, 48 small replicas 70.1 -> 63.2.
template <bool FUSED>
__global__ void __launch_bounds__(kBndThreads) k_boundary(const RepDesc* __restrict__ descs,
                                                          const int* __restrict__ reps, int nr, int mode) {
    static_assert(kBndThreads == kChunkTiles, "a workgroup sums a chunk");
    constexpr int kStWords = (int)(sizeof(RepState) / 4);
    static_assert(sizeof(RepState) % 4 == 0 && kStWords <= kBndThreads, "one word of the state per thread");
    __shared__ double red[kNumSum + 2][kBndThreads / 64];
    __shared__ double s_cp[FUSED ? kFusedChunks * kNumPart : 1];
    __shared__ double smp[6];
    __shared__ int push;
    __shared__ __align__(16) char s_state[sizeof(RepState)];
    const RepDesc& d = descs[reps[blockIdx.x]];
    RepState* const gst = d.st;
    RepState* const st = (RepState*)s_state;
    // The flags that the branches below go by are read by every wave ahead of the
    // barrier, and written (by thread 0: start_step sets all of them for the next
    // step) only behind it, so they are uniform over the workgroup.
    const int active = __builtin_amdgcn_readfirstlane(gst->active);
    const int ready = __builtin_amdgcn_readfirstlane(gst->pre_ready);
    const int want_obs = __builtin_amdgcn_readfirstlane(gst->want_obs);
    const bool quiet = mode == BND_STEP && d.ensemble == 0 && !want_obs;
    if (!quiet && threadIdx.x < kStWords) ((int*)s_state)[threadIdx.x] = gview((const int*)gst)[threadIdx.x];
    __syncthreads();
    if (mode == BND_START ? (!active || ready) : (mode == BND_STEP && !active)) return;
    if (quiet) {
        // a Langevin step that records nothing reduced no partials (k_force): the
        // step count and the next step's target only
        if (threadIdx.x == 0) {
            const int64_t cur = gst->step + 1, stop = gst->stop;
            const int err = gst->err;
            gst->v_pending = 1.0f;
            gst->step = cur;
            gst->rec_step = cur;
            gst->kicked = cur < stop ? 1 : 0;
            if (cur >= stop || err) {
                gst->active = 0;
                gst->pre_ready = 0;
            } else {
                start_step(d, gst, cur + 1);
            }
        }
        return;
    }
    if (mode == BND_START) {
        if (threadIdx.x == 0) {
            start_step(d, st, st->step + 1);
            push = 0;
        }
    } else {
        // fixed-order reduction: per-thread strided sums, wave shuffles, then the
        // waves in order (the same order whatever else is in the batch)
        // second level: lane l of a wave reads component l % 16 of chunk 4 w + l / 16
        // (+ 4 x waves per pass), the chunks in a fixed order
        if constexpr (FUSED) {
            for (int ck = 0; ck < d.nchunks; ck++) {
                chunk_sum(d, ck, red, s_cp + ck * kNumPart);
                __syncthreads();
            }
        }
        const int lane = lane_id(), wv = threadIdx.x >> 6, c = lane & 15;
        const bool mx = c >= kNumSum;  // the two maximum keys
        double a = 0.0;
        for (int ck = 4 * wv + (lane >> 4); ck < d.nchunks; ck += 4 * (kBndThreads / 64)) {
            const double x = FUSED ? s_cp[FUSED ? ck * kNumPart + c : 0] : d.cpart[(size_t)ck * kNumPart + c];
            a = mx ? fmax(a, x) : a + x;
        }
        double o = __shfl_xor(a, 16, 64);
        a = mx ? fmax(a, o) : a + o;
        o = __shfl_xor(a, 32, 64);
        a = mx ? fmax(a, o) : a + o;
        if (lane < kNumSum + 2) red[lane][wv] = a;
        __syncthreads();
        if (threadIdx.x == 0) push = boundary_tail(d, st, mode, red, smp);
    }
    __syncthreads();
    if (threadIdx.x < kStWords) gmut((int*)gst)[threadIdx.x] = ((const int*)s_state)[threadIdx.x];
    if (push) corr_push(d.corr, smp);
}

// Readback: a range of atoms by global id, written straight to pinned host
// memory.  One thread per global id (slot_of gives its slot), so the gathers
// are random in HBM and the stores to the host are whole lines in order; the
// three-component arrays go through LDS to be stored 16 bytes at a time.  Bound
// by the host: 1M beads (40 MB) 2.2 ms, most of it the copy into the caller's
// arrays (by copies of the slot arrays and a permutation on the host, 18.9 ms);
// 30,000 beads 76 us (159), 2,000 beads 21 us (96).
__global__ void __launch_bounds__(256) k_read_atoms(const RepDesc* __restrict__ dp, int g0, int n,
                                                    f32x4* __restrict__ pos, float* __restrict__ vel,
                                                    float* __restrict__ img) {
    __shared__ __align__(16) float s_v[768], s_i[768];
    const RepDesc& d = *dp;
    const int t = threadIdx.x, i = blockIdx.x * 256 + t, m = min(256, n - (int)blockIdx.x * 256);
    if (i < n) {
        const int s = gview(d.slot_of)[g0 + i];
        const float vs = d.st->v_pending;  // post-force scale not yet applied to vel[]
        const f32x4 v = raw4(d.vel)[s], im = raw4(d.img)[s];
        if (pos) pos[i] = raw4(d.pos)[s];
        s_v[3 * t] = v.x * vs; s_v[3 * t + 1] = v.y * vs; s_v[3 * t + 2] = v.z * vs;
        s_i[3 * t] = im.x; s_i[3 * t + 1] = im.y; s_i[3 * t + 2] = im.z;
    }
    __syncthreads();
    auto store = [&](float* out, const float* src) {
        float* o = out + (size_t)blockIdx.x * 768;
        if (m == 256) {
            if (t < 192) ((f32x4*)o)[t] = ((const f32x4*)src)[t];
        } else {
            for (int k = t; k < 3 * m; k += 256) o[k] = src[k];
        }
    };
    if (vel) store(vel, s_v);
    if (img) store(img, s_i);
}
// Forces by global id and the replica's state, to pinned host memory.
__global__ void __launch_bounds__(256) k_read_force(const RepDesc* __restrict__ dp, int g0, int n,
                                                    f32x4* __restrict__ force, int* __restrict__ state) {
    const RepDesc& d = *dp;
    const int i = blockIdx.x * 256 + threadIdx.x;
    if (force && i < n) force[i] = raw4(d.force)[gview(d.slot_of)[g0 + i]];
    if (state && blockIdx.x == 0 && threadIdx.x < sizeof(RepState) / 4)
        state[threadIdx.x] = gview((const int*)d.st)[threadIdx.x];
}

// Reference cell id and Morton key by global id (parity entry points).
__global__ void k_ref_cells(const RepDesc* __restrict__ dp, int natoms, int* __restrict__ out) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= natoms) return;
    const RepDesc& d = *dp;
    const RepState* st = d.st;
    int n = (int)(st->Lp / d.rcs);
    const int nx = n < 1 ? 1 : n;
    const float ics = 1.0f / (st->Lp / (float)nx);
    const float4 r = d.pos[i];
    out[d.img[i].w] = (cell_coord(r.z, ics, nx) * nx + cell_coord(r.y, ics, nx)) * nx +
                      cell_coord(r.x, ics, nx);
}

#pragma clang fp contract(off)
__device__ inline uint32_t quant1024(float x, float invL) {
    const float q = x * invL * 1024.0f;
    const uint32_t u = (q > 0.0f) ? (uint32_t)q : 0u;  // truncation, saturating at 0
    return u > 1023u ? 1023u : u;
}
#pragma clang fp contract(fast)

__global__ void k_morton_keys(const RepDesc* __restrict__ dp, int natoms, uint32_t* __restrict__ out) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= natoms) return;
    const RepDesc& d = *dp;
    const float invL = d.st->invLp;
    const float4 r = d.pos[i];
    out[d.img[i].w] = (expand_bits(quant1024(r.z, invL)) << 2) |
                      (expand_bits(quant1024(r.y, invL)) << 1) | expand_bits(quant1024(r.x, invL));
}

// ---------------------------------------------------------------------------
// launchers
// ---------------------------------------------------------------------------
static inline int cdiv(int a, int b) { return (a + b - 1) / b; }
// grid cap of the grid-stride rebuild kernels: a step's rebuild list (about
// 4,000 tiles) in one pass, without thousands of waves that find no tile
static constexpr int kStrideBlocks = 1024;
static constexpr int kBuildBlocks = 8192;   // grid cap of the list-build workgroups (one group each)
// Up to this many groups in the launch (one per CU) each group's scan is shared
// by four waves a tile; with more the CUs are full anyway and four only add
// barriers and a second group's wait.  Measured per step, four waves against
// one: 2,000 beads 40.1 / 41.6 us, 30,000 44.4 / 45.4, 60,000 45.6 / 46.8,
// 100,000 60.7 / 59.5, 250,000 80.6 / 75.3.
static constexpr int kSplitGroups = 256;
static constexpr int kForceListBlocks = 1280;  // workgroups of a listed force pass (five per CU; a multiple of kXcds)
static_assert(kForceListBlocks % kXcds == 0, "the listed force pass splits its grid evenly over the XCDs");

void launch_pre(const Launch& l) {
    if (l.ntl <= 0) return;
    k_pre<<<cdiv(l.ntl, 4), 256, 0, l.stream>>>(l.descs, l.tiles, l.ntl, l.nrt);
}
void launch_decide(const Launch& l, bool sort) {
    if (l.nr <= 0) return;
    if (sort) k_decide<true><<<l.nr, kSortThreads, 0, l.stream>>>(l.descs, l.reps, l.nr, l.rep_t0, l.rlist, l.nrt);
    else k_decide<false><<<l.nr, kSortThreads, 0, l.stream>>>(l.descs, l.reps, l.nr, l.rep_t0, l.rlist, l.nrt);
}
void launch_rg(const RepDesc* d, int nchains, double* out, hipStream_t s) {
    if (nchains <= 0) return;
    k_rg<<<nchains, 64, 0, s>>>(d, out);
}
void launch_rg_mean(const RepDesc* d, const double* vals, double* out, hipStream_t s) {
    k_rg_mean<<<1, 64, 0, s>>>(d, vals, out);
}
void launch_corr_push(const RepDesc* d, const Sample6& x, hipStream_t s) {
    k_corr_push<<<1, 128, 0, s>>>(d, x);
}
void launch_nh_chain_run(RepState* st, const double* ke, int n, int carry, double kT, int natoms,
                         double half_dt, double* scales, hipStream_t s) {
    if (n <= 0) return;
    k_nh_chain_run<<<1, 64, 0, s>>>(st, ke, n, carry, kT, natoms, half_dt, scales);
}
void launch_status(const Launch& l, int4* out) {
    if (l.nr <= 0) return;
    k_status<<<cdiv(l.nr, 256), 256, 0, l.stream>>>(l.descs, l.reps, l.nr, out);
}
void launch_phase(const Launch& l, int* out) {
    if (l.nr <= 0) return;
    k_phase<<<cdiv(l.nr, 256), 256, 0, l.stream>>>(l.descs, l.reps, l.nr, out);
}
void launch_control(const Launch& l, int op, int64_t arg) {
    if (l.nr <= 0) return;
    k_control<<<cdiv(l.nr, 64), 64, 0, l.stream>>>(l.descs, l.reps, l.nr, op, arg);
}
// k_force is compiled for at most kMaxBlock threads per block; any other request
// runs at the default shape.
static constexpr int kMaxBlock = kMaxBlockK;
static inline int valid_block(int b) { return (b == 64 || b == 128 || b == 256) ? b : kMaxBlock; }

// The workgroups of the scan: one a pass of keys of the largest replica, as far
// as their limits and kScanGrid for the whole batch go.  Those of replicas that
// do not rebuild, or have fewer keys, return at once, but they are launched in
// every step (1,023 small replicas and one of 2,097,152 keys: 680 us per step
// with a workgroup a pass for each replica, 145 with two a replica).
static constexpr int kScanGrid = 2048;
static void launch_scan(const Launch& l, int always) {
    const int passes = cdiv(l.max_keys, kScanKeys), share = max(1, kScanGrid / l.nr);
    const bool totals = min(passes, share) > kScanBlocks;
    const dim3 g(l.nr, min(min(passes, share), totals ? kScanTotals : kScanBlocks));
    if (totals) {
        k_scan_totals<<<g, 1024, 0, l.stream>>>(l.descs, l.reps, l.nr, always);
        k_scan<false, true><<<g, 1024, 0, l.stream>>>(l.descs, l.reps, l.nr, always);
    } else if (passes <= (int)g.y) {
        k_scan<true, false><<<g, 1024, 0, l.stream>>>(l.descs, l.reps, l.nr, always);
    } else {
        k_scan<false, false><<<g, 1024, 0, l.stream>>>(l.descs, l.reps, l.nr, always);
    }
}
void launch_rebuild(const Launch& l, int always, int build) {
    if (l.ntl <= 0) return;
    // a step's rebuild tile list is k_decide's; otherwise list the tiles here
    if (always) k_rebuild_list<<<1, 1024, 0, l.stream>>>(l.descs, l.reps, l.rep_t0, l.nr, always, l.rlist, l.nrt);
    int g = cdiv(l.ntl, 4);
    if (g > kStrideBlocks) g = kStrideBlocks;
    k_bin<<<g, 256, 0, l.stream>>>(l.descs, l.tiles, l.rlist, l.nrt);
    launch_scan(l, always);
    k_scatter<<<g, 256, 0, l.stream>>>(l.descs, l.tiles, l.rlist, l.nrt);
    k_rank<<<g, 256, 0, l.stream>>>(l.descs, l.tiles, l.rlist, l.nrt);
    if (build) launch_build(l);
}
void launch_build(const Launch& l, int max_blocks) {
    if (l.ntl <= 0) return;
    int gb = cdiv(l.ntl, kGroupTiles);
    const int cap = max_blocks > 0 ? max_blocks : kBuildBlocks;
    if (gb > cap) gb = cap;
    if (cdiv(l.ntl, kGroupTiles) <= kSplitGroups)
        k_build<4><<<gb, kGroupSlots * 4, 0, l.stream>>>(l.descs, l.tiles, l.rlist, l.nrt);
    else
        k_build<1><<<gb, kGroupSlots, 0, l.stream>>>(l.descs, l.tiles, l.rlist, l.nrt);
}
static void force_kernel(const Launch& l, int g, int block, int t0, int nt, int terms, int kick, int mode,
                         int sel) {
    const size_t lds = 0;
#define FMD_FORCE_ARGS l.descs, l.tiles, t0, nt, kick, mode, sel, l.rlist, l.nrt
    switch ((terms & 7) | (l.any_tab && (terms & 1) ? 8 : 0)) {
        case 1: k_force<1><<<g, block, lds, l.stream>>>(FMD_FORCE_ARGS); break;
        case 2: k_force<2><<<g, block, lds, l.stream>>>(FMD_FORCE_ARGS); break;
        case 3: k_force<3><<<g, block, lds, l.stream>>>(FMD_FORCE_ARGS); break;
        case 4: k_force<4><<<g, block, lds, l.stream>>>(FMD_FORCE_ARGS); break;
        case 5: k_force<5><<<g, block, lds, l.stream>>>(FMD_FORCE_ARGS); break;
        case 6: k_force<6><<<g, block, lds, l.stream>>>(FMD_FORCE_ARGS); break;
        case 7: k_force<7><<<g, block, lds, l.stream>>>(FMD_FORCE_ARGS); break;
        case 9: k_force<1, false, true><<<g, block, lds, l.stream>>>(FMD_FORCE_ARGS); break;
        case 11: k_force<3, false, true><<<g, block, lds, l.stream>>>(FMD_FORCE_ARGS); break;
        case 13: k_force<5, false, true><<<g, block, lds, l.stream>>>(FMD_FORCE_ARGS); break;
        case 15: k_force<7, false, true><<<g, block, lds, l.stream>>>(FMD_FORCE_ARGS); break;
        default: k_force<0><<<g, block, lds, l.stream>>>(FMD_FORCE_ARGS); break;
    }
#undef FMD_FORCE_ARGS
}
void launch_force(const Launch& l, int t0, int nt, int block, int terms, int kick, int mode, int sel) {
    if (nt <= 0) return;
    block = valid_block(block);
    force_kernel(l, cdiv(nt, block / 64), block, t0, nt, terms, kick, mode, sel);
}
void launch_force_listed(const Launch& l, int kick, int mode) {
    if (l.ntl <= 0) return;
    if (l.any_tab)
        k_force<7, true, true><<<kForceListBlocks, kGroupSlots, 0, l.stream>>>(l.descs, l.tiles, 0, 0, kick, mode,
                                                                                FS_ALL, l.rlist, l.nrt);
    else
        k_force<7, true><<<kForceListBlocks, kGroupSlots, 0, l.stream>>>(l.descs, l.tiles, 0, 0, kick, mode, FS_ALL,
                                                                          l.rlist, l.nrt);
}
void launch_boundary(const Launch& l, int mode) {
    if (l.nr <= 0) return;
    if (mode == BND_START || l.max_chunks <= (l.sums_always ? 1 : kFusedChunks)) {
        k_boundary<true><<<l.nr, kBndThreads, 0, l.stream>>>(l.descs, l.reps, l.nr, mode);
        return;
    }
    if (l.nch > 0) k_chunk<<<l.nch, 256, 0, l.stream>>>(l.descs, l.chunks, l.nch, mode);
    k_boundary<false><<<l.nr, kBndThreads, 0, l.stream>>>(l.descs, l.reps, l.nr, mode);
}
void launch_read_atoms(const RepDesc* d, int g0, int n, float* pos, float* vel, int* img, hipStream_t s) {
    if (n <= 0) return;
    k_read_atoms<<<cdiv(n, 256), 256, 0, s>>>(d, g0, n, (f32x4*)pos, vel, (float*)img);
}
void launch_read_force(const RepDesc* d, int g0, int n, float* force, void* state, hipStream_t s) {
    k_read_force<<<max(1, cdiv(n, 256)), 256, 0, s>>>(d, g0, n, (f32x4*)force, (int*)state);
}
void launch_ref_cells(const RepDesc* d, int natoms, int* out, hipStream_t s) {
    if (natoms <= 0) return;
    k_ref_cells<<<cdiv(natoms, 256), 256, 0, s>>>(d, natoms, out);
}
void launch_morton_keys(const RepDesc* d, int natoms, uint32_t* out, hipStream_t s) {
    if (natoms <= 0) return;
    k_morton_keys<<<cdiv(natoms, 256), 256, 0, s>>>(d, natoms, out);
}

}  // namespace fmd
