// fm_kernels.hip -- gfx950 kernels of the force / neighbour / integration path.
//
// Parity-critical FP64 arithmetic (cell index, image coordinates, squared distances, velocity
// Verlet) is written in the reference's operation order and compiled without fused multiply-add
// (file-wide fp contract off), so it is bit-identical to the reference's FP64 operations.
// The mixed-precision pair law re-enables contraction locally.
#include "fm_internal.h"

#include <limits.h>
#include <math.h>

#include <mutex>

#pragma clang fp contract(off)

namespace {

struct St {  // molecule state in slot order
    double *x, *y, *z, *vx, *vy, *vz, *ax, *ay, *az;
};

__host__ __device__ inline St state_of(double* base, int cap) {
    St s;
    s.x = base;
    s.y = base + (size_t)cap;
    s.z = base + 2 * (size_t)cap;
    s.vx = base + 3 * (size_t)cap;
    s.vy = base + 4 * (size_t)cap;
    s.vz = base + 5 * (size_t)cap;
    s.ax = base + 6 * (size_t)cap;
    s.ay = base + 7 * (size_t)cap;
    s.az = base + 8 * (size_t)cap;
    return s;
}

inline int nblocks(size_t n) { return (int)((n + FM_BLOCK - 1) / FM_BLOCK); }

__device__ inline void set_err(int* flags, int code, int mol) {
    if (atomicCAS(&flags[FLAG_ERROR], 0, code) == 0) flags[FLAG_ERROR_MOL] = mol;
}

// gcc __builtin_powi expansion (what gfortran emits for x**n): x7 = (x*x2)*(x2*x2) ...
__device__ inline double p3(double x) { return x * (x * x); }
__device__ inline double p4(double x) { double x2 = x * x; return x2 * x2; }
__device__ inline double p6(double x) { double x3 = x * (x * x); return x3 * x3; }
__device__ inline double p7(double x) { double x2 = x * x; return (x * x2) * (x2 * x2); }

__device__ inline int shift_code(int sx, int sy, int sz) { return (sx + 1) * 9 + (sy + 1) * 3 + (sz + 1); }
__device__ inline void decode_shift(int code, int& sx, int& sy, int& sz) {
    sx = code / 9 - 1;
    sy = (code / 3) % 3 - 1;
    sz = code % 3 - 1;
}
// image coordinate r + s*L, one add per shifted component (the reference's halo copy)
__device__ inline double img(double r, int s, double L) { return s == 0 ? r : r + (double)s * L; }

// ---------------------------------------------------------------------------------------------
__global__ void k_fill_i32(int* p, int v, size_t n) {
    size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) p[i] = v;
}
__global__ void k_fill_f64(double* p, double v, size_t n) {
    size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) p[i] = v;
}

// ---- velocity Verlet, src/simulation_move_particles_vv.f90:64-69 (pass 1), 132-135 (pass 2) ---
// halt: flag words of a conditional launch (does nothing while FLAG_HALT is set), or null
__global__ __launch_bounds__(FM_BLOCK) void k_pass1(St s, int np, double dt, double hdt2, double hdt, const int* halt) {
    if (halt && halt[FLAG_HALT] != 0) return;  // whole workgroup
    int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= np) return;
    double ax = s.ax[i], ay = s.ay[i], az = s.az[i];
    double vx = s.vx[i], vy = s.vy[i], vz = s.vz[i];
    s.x[i] = s.x[i] + dt * vx + hdt2 * ax;
    s.y[i] = s.y[i] + dt * vy + hdt2 * ay;
    s.z[i] = s.z[i] + dt * vz + hdt2 * az;
    s.vx[i] = vx + hdt * ax;
    s.vy[i] = vy + hdt * ay;
    s.vz[i] = vz + hdt * az;
}

__global__ __launch_bounds__(FM_BLOCK) void k_pass2(St s, int np, double hdt) {
    int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= np) return;
    s.vx[i] = s.vx[i] + hdt * s.ax[i];
    s.vy[i] = s.vy[i] + hdt * s.ay[i];
    s.vz[i] = s.vz[i] + hdt * s.az[i];
}

// ---- simulation_move_particles_lfv, src/simulation_move_particles_lfv.f90:38-177 ---------------
// NVE, or tag_move through simulation_move_particles_lfv_tag (308-490) for the tags without a
// thermostat; tethered molecules get tether_force (src/molecular_properties.f90:833-915) here,
// inside the move.  With disp != 0 the displacement update of simulation_checkrebuild (rebuild
// criterion 2) follows in the same pass.
__global__ __launch_bounds__(FM_BLOCK) void k_move_lfv(St s, const int* tag, double* teth, const int* ext, int np,
                                                        int cap, double dt, double k2, double k4, double k6,
                                                        double* rd, double thresh, int disp, int fresh,
                                                        int* flags, int cond) {
    if (cond && flags[FLAG_HALT] != 0) return;  // whole launch: a queued rebuild is pending
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    bool hit = false;
    if (i < np) {
        const int tg = tag ? tag[i] : FM_TAG_FREE;
        double r[3] = {s.x[i], s.y[i], s.z[i]};
        double v[3] = {s.vx[i], s.vy[i], s.vz[i]};
        double a[3] = {s.ax[i], s.ay[i], s.az[i]};
        const size_t c = (size_t)cap;
        if (tg == FM_TAG_TETH || tg == FM_TAG_TETH_SLIDE) {
            double rio[3];
            for (int d = 0; d < 3; ++d) rio[d] = r[d] - teth[i + d * c];
            const double mag = sqrt((rio[0] * rio[0] + rio[1] * rio[1]) + rio[2] * rio[2]);
            const double am = -2.0 * k2 * mag - 4.0 * k4 * (mag * mag) - 6.0 * k6 * pow(mag, 4.0);
            for (int d = 0; d < 3; ++d) a[d] = a[d] + am * rio[d];
            for (int d = 0; d < 3; ++d) teth[i + d * c] = teth[i + d * c] + teth[i + (3 + d) * c] * dt;
            s.ax[i] = a[0];
            s.ay[i] = a[1];
            s.az[i] = a[2];
        }
        switch (tg) {
        case FM_TAG_FREE:
        case FM_TAG_TETH:
            for (int d = 0; d < 3; ++d) v[d] = v[d] + dt * a[d];
            for (int d = 0; d < 3; ++d) r[d] = r[d] + dt * v[d];
            break;
        case FM_TAG_TETH_SLIDE:
            for (int d = 0; d < 3; ++d) v[d] = v[d] + dt * a[d];
            for (int d = 0; d < 3; ++d) r[d] = r[d] + dt * v[d] + dt * teth[i + (3 + d) * c];
            break;
        case FM_TAG_FIXED_SLIDE:
            for (int d = 0; d < 3; ++d) r[d] = r[d] + dt * teth[i + (3 + d) * c];
            break;
        case FM_TAG_FIXED:
            break;
        default:
            set_err(flags, FM_EINVAL, ext[i]);
        }
        s.x[i] = r[0];
        s.y[i] = r[1];
        s.z[i] = r[2];
        s.vx[i] = v[0];
        s.vy[i] = v[1];
        s.vz[i] = v[2];
        if (disp) {
            double d0 = fresh ? 0.0 : rd[i];
            double d1 = fresh ? 0.0 : rd[i + c];
            double d2 = fresh ? 0.0 : rd[i + 2 * c];
            d0 = d0 + v[0] * dt;
            d1 = d1 + v[1] * dt;
            d2 = d2 + v[2] * dt;
            rd[i] = d0;
            rd[i + c] = d1;
            rd[i + 2 * c] = d2;
            hit = fabs(d0) > thresh || fabs(d1) > thresh || fabs(d2) > thresh;
        }
    }
    unsigned long long m = __ballot(hit);
    if (m != 0ull && (int)(threadIdx.x & 63) == __ffsll((long long)m) - 1 &&
        __atomic_load_n(&flags[FLAG_REBUILD], __ATOMIC_RELAXED) == 0)
        atomicOr(&flags[FLAG_REBUILD], 1);
}

// ---- rebuild criterion 2, src/simulation_checkrebuild.f90:105-121 ----------------------------
__global__ __launch_bounds__(FM_BLOCK) void k_check_disp(St s, double* rd, int np, int cap, double dt,
                                                          double thresh, int fresh, int* flags) {
    int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= np) return;
    double d0 = fresh ? 0.0 : rd[i];
    double d1 = fresh ? 0.0 : rd[i + cap];
    double d2 = fresh ? 0.0 : rd[i + 2 * (size_t)cap];
    d0 = d0 + s.vx[i] * dt;
    d1 = d1 + s.vy[i] * dt;
    d2 = d2 + s.vz[i] * dt;
    rd[i] = d0;
    rd[i + cap] = d1;
    rd[i + 2 * (size_t)cap] = d2;
    bool hit = fabs(d0) > thresh || fabs(d1) > thresh || fabs(d2) > thresh;
    unsigned long long m = __ballot(hit);
    if (m != 0ull && (int)(threadIdx.x & 63) == __ffsll((long long)m) - 1 &&
        __atomic_load_n(&flags[FLAG_REBUILD], __ATOMIC_RELAXED) == 0)
        atomicOr(&flags[FLAG_REBUILD], 1);
}

// simulation_move_particles_vv(1) followed by the displacement update of simulation_checkrebuild,
// in one pass over the state (same operations as k_pass1 then k_check_disp)
// cond: a launch queued ahead of the host's check; it does nothing when an earlier step of the
// queue asked for a rebuild (FLAG_HALT), and records its step when it asks for one itself.
__global__ __launch_bounds__(FM_BLOCK) void k_pass1_disp(St s, double* rd, int np, int cap, double dt, double hdt2,
                                                          double hdt, double thresh, int fresh, int* flags, int cond,
                                                          int step) {
    if (cond && flags[FLAG_HALT] != 0) return;  // whole workgroup
    int i = blockIdx.x * blockDim.x + threadIdx.x;
    bool hit = false;
    if (i < np) {
        const double ax = s.ax[i], ay = s.ay[i], az = s.az[i];
        double vx = s.vx[i], vy = s.vy[i], vz = s.vz[i];
        s.x[i] = s.x[i] + dt * vx + hdt2 * ax;
        s.y[i] = s.y[i] + dt * vy + hdt2 * ay;
        s.z[i] = s.z[i] + dt * vz + hdt2 * az;
        vx = vx + hdt * ax;
        vy = vy + hdt * ay;
        vz = vz + hdt * az;
        s.vx[i] = vx;
        s.vy[i] = vy;
        s.vz[i] = vz;
        double d0 = fresh ? 0.0 : rd[i];
        double d1 = fresh ? 0.0 : rd[i + cap];
        double d2 = fresh ? 0.0 : rd[i + 2 * (size_t)cap];
        d0 = d0 + vx * dt;
        d1 = d1 + vy * dt;
        d2 = d2 + vz * dt;
        rd[i] = d0;
        rd[i + cap] = d1;
        rd[i + 2 * (size_t)cap] = d2;
        hit = fabs(d0) > thresh || fabs(d1) > thresh || fabs(d2) > thresh;
    }
    unsigned long long m = __ballot(hit);
    if (m != 0ull && (int)(threadIdx.x & 63) == __ffsll((long long)m) - 1 &&
        __atomic_load_n(&flags[FLAG_REBUILD], __ATOMIC_RELAXED) == 0) {
        atomicOr(&flags[FLAG_REBUILD], 1);
        if (cond) atomicExch(&flags[FLAG_RB_STEP], step);
    }
}

// ---- rebuild criterion 0 (Rapaport vmax), src/simulation_checkrebuild.f90:84-99 --------------
__global__ __launch_bounds__(FM_BLOCK) void k_vmax(St s, int np, unsigned long long* vmax_bits) {
    __shared__ double red[FM_BLOCK / 64];
    int i = blockIdx.x * blockDim.x + threadIdx.x;
    double m = 0.0;
    if (i < np) {
        double vx = s.vx[i], vy = s.vy[i], vz = s.vz[i];
        m = (vx * vx + vy * vy) + vz * vz;
    }
    for (int off = 32; off > 0; off >>= 1) m = fmax(m, __shfl_down(m, off, 64));
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = m;
    __syncthreads();
    if (threadIdx.x == 0) {
        double b = red[0];
        for (int w = 1; w < FM_BLOCK / 64; ++w) b = fmax(b, red[w]);
        // non-negative doubles order like their bit patterns
        const unsigned long long bits = (unsigned long long)__double_as_longlong(b);
        if (bits > __atomic_load_n(vmax_bits, __ATOMIC_RELAXED)) atomicMax(vmax_bits, bits);
    }
}

__global__ void k_vmax_finish(unsigned long long* vmax_bits, double* rmax, double dt, double thresh,
                              int forced, int* flags) {
    double vmax = sqrt(__longlong_as_double((long long)*vmax_bits));
    double r = *rmax + vmax * dt;
    int rb = forced || r > thresh;
    if (rb) {
        flags[FLAG_REBUILD] = 1;
        r = 0.0;
    }
    *rmax = r;
    *vmax_bits = 0ull;
}

// ---- sendmols on one periodic rank, src/messenger.MPI.f90:1383-1904 ---------------------------
// zero the listed flag words
struct FlagList {
    int n;
    int w[8];
};

// zero one flag word; a reset of FLAG_REBUILD also returns FLAG_RB_STEP to "no step" (INT_MAX),
// which the halt rule of conditional force launches relies on
__device__ inline void reset_flag(int* flags, int w) {
    flags[w] = 0;
    if (w == FLAG_REBUILD) flags[FLAG_RB_STEP] = 0x7fffffff;
    if (w == FLAG_HALT) flags[FLAG_HALT_STEP] = 0x7fffffff;
}

// The 3 x (3 axes x 2 directions) exchange passes of sendmols (checksendbuild, sendrecvface,
// reorderdata): in each pass the molecules beyond that face, in ascending molecule number, are
// wrapped by -dir*domain and their numbers reversed among them.  Where a molecule leaves depends on
// its own position alone, so every molecule runs its 18 passes by itself (wrap_molecule) and keeps
// them as bits; the numbers are then exchanged among the leavers by one workgroup (renumber).
struct WrapArgs {
    St s;
    const int* ext;
    const int* tag;        // null without tag_move
    double* teth;
    int np, cap;
    double L[3], ws[3];    // domain, wallslidev
    int* mask;             // per slot: the passes a leaver left in (written for leavers only)
    unsigned* bits;        // one bit per molecule number: leavers
    int* flags;
    FlagList reset;        // flag words zeroed by workgroup 0 (the resets of a queued rebuild)
};

// positions after the passes (r), stored where they changed
__device__ __forceinline__ void wrap_molecule(const WrapArgs& a, int i, double r[3]) {
    const double h[3] = {0.5 * a.L[0], 0.5 * a.L[1], 0.5 * a.L[2]};
    const bool out = (r[0] < -h[0]) | (r[0] >= h[0]) | (r[1] < -h[1]) | (r[1] >= h[1]) | (r[2] < -h[2]) | (r[2] >= h[2]);
    if (!out) return;
    const int tg = a.tag ? a.tag[i] : FM_TAG_FREE;
    const bool held = tg == FM_TAG_TETH || tg == FM_TAG_TETH_SLIDE;
    int m = 0;
    for (int it = 0; it < 3; ++it)
#pragma unroll
        for (int ax = 0; ax < 3; ++ax)
#pragma unroll
            for (int dir = -1; dir <= 1; dir += 2)
                if (dir == -1 ? r[ax] < -h[ax] : r[ax] >= h[ax]) {
                    r[ax] = r[ax] - (double)dir * a.L[ax];
                    if (held) a.teth[i + (size_t)ax * a.cap] = a.teth[i + (size_t)ax * a.cap] - (double)dir * a.L[ax];
                    m |= 1 << (it * 6 + ax * 2 + (dir + 1) / 2);
                }
    a.s.x[i] = r[0];
    a.s.y[i] = r[1];
    a.s.z[i] = r[2];
    if (a.tag) {
        // read_tag on the renumbered molecule (the last pass it left in saw its final y)
        const double sg = tg == FM_TAG_TETH_SLIDE ? copysign(1.0, r[1]) : tg == FM_TAG_FIXED_SLIDE ? 1.0 : 0.0;
#pragma unroll
        for (int d = 0; d < 3; ++d) a.teth[i + (size_t)(3 + d) * a.cap] = sg != 0.0 ? a.ws[d] * sg : 0.0;
    }
    a.mask[i] = m;
    const int e = a.ext[i];
    atomicOr(&a.bits[e >> 5], 1u << (e & 31));
}

__global__ __launch_bounds__(FM_BLOCK) void k_wrap(WrapArgs a) {
    if (blockIdx.x == 0 && (int)threadIdx.x < a.reset.n) reset_flag(a.flags, a.reset.w[threadIdx.x]);
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= a.np) return;
    double r[3] = {a.s.x[i], a.s.y[i], a.s.z[i]};
    wrap_molecule(a, i, r);
}

// Exclusive prefix of v over the workgroup's threads (1024 of them); *total: the sum.  wsum: 16 ints.
__device__ __forceinline__ int block_prefix(int v, int* wsum, int* total) {
    const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6, nw = blockDim.x >> 6;
    int x = v;
    for (int d = 1; d < 64; d <<= 1) {
        const int y = __shfl_up(x, d, 64);
        if (lane >= d) x += y;
    }
    __syncthreads();  // (wsum may still be read from the call before)
    if (lane == 63) wsum[wid] = x;
    __syncthreads();
    int pre = x - v, tot = 0;
    for (int w = 0; w < nw; ++w) {
        const int t = wsum[w];
        if (w < wid) pre += t;
        tot += t;
    }
    *total = tot;
    return pre;
}

// The passes over n leavers by list position q: number V[q] (ascending, fixed), the slot S[q] that
// carries it and that molecule's passes M[q].  lst, tS, tM: scratch of n each.
__device__ __forceinline__ void renumber_passes(int n, int passes, int* S, int* M, int* lst, int* tS, int* tM, int* wsum) {
    const int tid = threadIdx.x, nt = blockDim.x;
    for (; passes; passes &= passes - 1) {
        const int bit = passes & -passes;
        int k = 0;
        for (int base = 0; base < n; base += nt) {
            const int q = base + tid;
            const int lv = q < n && (M[q] & bit) ? 1 : 0;
            int tot;
            const int p = block_prefix(lv, wsum, &tot);
            if (lv) lst[k + p] = q;
            k += tot;
        }
        __syncthreads();
        for (int m = tid; m < k; m += nt) {
            const int q = lst[k - 1 - m];
            tS[m] = S[q];
            tM[m] = M[q];
        }
        __syncthreads();
        for (int m = tid; m < k; m += nt) {
            S[lst[m]] = tS[m];
            M[lst[m]] = tM[m];
        }
        __syncthreads();
    }
}

struct RenumArgs {
    int np;
    unsigned* bits;
    const int* mask;
    int *ext, *slot_of;
    int* scratch;          // 6 x cap ints, for more than RENUM_LDS leavers
    int cap;
    int set_slots;         // write slot_of too (a binning that follows rewrites it)
    int* flags;
};
#define RENUM_LDS 2048

// sendmols' numbers: one workgroup of 1024 threads.  The leavers are read off the bit map in
// ascending molecule number (each thread a contiguous range of its words, cleared as they are read).
// When every leaver left in one pass only, no pass moves a number that another one looks at, so all
// of them are done at once: the position of each leaver among those of its pass, and the slot of the
// one as far from that pass's end.  A molecule that left in two (an edge of the box: one rebuild in
// some) makes it the passes in turn, those that some molecule left in.
// Bound: one workgroup's chain of dependent loads (bits, slots, masks) and barriers.  In a queued
// rebuild it is one workgroup of the scan's launch.  With the selection it replaced a one-workgroup
// kernel of 18 passes and a launch that read every position through slot_of (23.6 + 12.1 us a
// rebuild at 1,048,576 molecules, 17.5 + 3.3 us at 2,048).
__device__ void renumber(const RenumArgs& a) {
    constexpr int NW = RENUM_LDS / 64;  // wavefronts' worth of leavers
    __shared__ int wsum[16], lds[6][RENUM_LDS], cnt[18 * NW + 1], all, multi;
    const int tid = threadIdx.x, lane = tid & 63, wid = tid >> 6;
    // 16-byte words, a contiguous run of them per thread
    const int nv = (a.np + 127) >> 7, per = (nv + (int)blockDim.x - 1) / (int)blockDim.x;
    const int v0 = min(nv, tid * per), v1 = min(nv, v0 + per);
    uint4* const B = (uint4*)a.bits;
    int mine = 0;
#pragma unroll 8
    for (int v = v0; v < v1; ++v) {
        const uint4 w = B[v];
        mine += __popc(w.x) + __popc(w.y) + __popc(w.z) + __popc(w.w);
    }
    if (tid == 0) all = multi = 0;
    int n;
    int pos = block_prefix(mine, wsum, &n);
    const bool small = n <= RENUM_LDS;
    int* V = small ? lds[0] : a.scratch;
    int* S = small ? lds[1] : a.scratch + a.cap;
    int* M = small ? lds[2] : a.scratch + 2 * (size_t)a.cap;
    for (int u = v0; mine && u < v1; u += 8) {
        uint4 w[8];
#pragma unroll
        for (int k = 0; k < 8; ++k) w[k] = B[min(u + k, v1 - 1)];
#pragma unroll
        for (int k = 0; k < 8; ++k) {
            const unsigned c[4] = {w[k].x, w[k].y, w[k].z, w[k].w};
            if (u + k >= v1 || (c[0] | c[1] | c[2] | c[3]) == 0u) continue;
#pragma unroll
            for (int d = 0; d < 4; ++d)
                for (unsigned m = c[d]; m; m &= m - 1) V[pos++] = ((u + k) << 7) + (d << 5) + __ffs((int)m) - 1;
            B[u + k] = make_uint4(0u, 0u, 0u, 0u);
        }
    }
    __syncthreads();
    int o = 0;
    bool two = false;
    for (int q = tid; q < n; q += blockDim.x) {
        const int slot = a.slot_of[V[q]], m = a.mask[slot];
        S[q] = slot;
        M[q] = m;
        o |= m;
        two = two || (m & (m - 1)) != 0;
    }
    if (o) atomicOr(&all, o);
    if (two) multi = 1;
    __syncthreads();
    if (!small) {
        renumber_passes(n, all, S, M, a.scratch + 3 * (size_t)a.cap, a.scratch + 4 * (size_t)a.cap,
                        a.scratch + 5 * (size_t)a.cap, wsum);
    } else if (multi) {
        renumber_passes(n, all, S, M, lds[3], lds[4], lds[5], wsum);
    } else {
        // cnt[pass][wavefront]: leavers, then their exclusive prefix in that order
        int rank[RENUM_LDS / 1024];
        for (int k = tid; k <= 18 * NW; k += blockDim.x) cnt[k] = 0;
        __syncthreads();
#pragma unroll
        for (int c = 0; c < RENUM_LDS / 1024; ++c) {
            const int q = c * 1024 + tid, m = q < n ? M[q] : 0;
            rank[c] = 0;
            for (int ps = all; ps; ps &= ps - 1) {
                const unsigned long long in = __ballot(m & ps & -ps);
                if (m & ps & -ps) rank[c] = __popcll(in & ((1ull << lane) - 1ull));
                if (lane == 0) cnt[(__ffs(ps) - 1) * NW + c * 16 + wid] = __popcll(in);
            }
        }
        __syncthreads();
        static_assert(18 * NW <= 1024, "a count per thread");
        int tot;
        const int pre = block_prefix(tid < 18 * NW ? cnt[tid] : 0, wsum, &tot);
        if (tid <= 18 * NW) cnt[tid] = pre;
        __syncthreads();
        int* lst = lds[3];
        int* out = lds[4];
        int p[RENUM_LDS / 1024];
#pragma unroll
        for (int c = 0; c < RENUM_LDS / 1024; ++c) {
            const int q = c * 1024 + tid;
            p[c] = 0;
            if (q < n) {
                const int b = __ffs(M[q]) - 1, at = cnt[b * NW + c * 16 + wid] + rank[c];
                lst[at] = q;
                p[c] = cnt[b * NW] + cnt[(b + 1) * NW] - 1 - at;
            }
        }
        __syncthreads();
#pragma unroll
        for (int c = 0; c < RENUM_LDS / 1024; ++c)
            if (c * 1024 + tid < n) out[c * 1024 + tid] = S[lst[p[c]]];
        S = out;  // (each thread reads its own below)
    }
    for (int q = tid; q < n; q += blockDim.x) {
        a.ext[S[q]] = V[q];
        if (a.set_slots) a.slot_of[V[q]] = S[q];
    }
    __syncthreads();
    // an escaped molecule met by k_bin_count before the renumbering: its slot, as ~slot
    if (tid == 0 && a.flags[FLAG_ERROR] == FM_EESCAPE && a.flags[FLAG_ERROR_MOL] < 0)
        a.flags[FLAG_ERROR_MOL] = a.ext[~a.flags[FLAG_ERROR_MOL]];
}

__global__ __launch_bounds__(1024) void k_renumber(RenumArgs a) { renumber(a); }

// Each active lane's position among the additions to its counter.  Lanes of a wavefront with the
// same counter are served by one atomic (consecutive slots mostly share a cell), and the wavefront's
// atomics go out together after the lanes are grouped: one round trip, where an atomic inside the
// grouping loop made it one per distinct cell (16.5 us for the 2,048 molecules of a WCA box with 2.8
// a cell).
__device__ inline int wave_aggregated_add(int* counters, int key, bool active) {
    const int lane = threadIdx.x & 63;
    unsigned long long todo = __ballot(active);
    int leader = lane, rank = 0, cnt = 0;
    while (todo) {
        const int l = __ffsll((long long)todo) - 1;
        const unsigned long long same = __ballot(active && key == __builtin_amdgcn_readlane(key, l));
        if ((same >> lane) & 1ull) {
            leader = l;
            rank = __popcll(same & ((1ull << lane) - 1ull));
            cnt = __popcll(same);
        }
        todo &= ~same;
    }
    int base = 0;
    if (active && lane == leader) base = atomicAdd(&counters[key], cnt);
    return __shfl(base, leader, 64) + rank;
}

// ---- assign_to_cell as a counting sort, src/linklist.f90:2645-2676 -----------------------------
struct BinArgs {
    double h[3], cs[3];
    int nc[3];
    int *cell_of, *count, *pos;
};

// WRAP: sendmols' wrap first (a queued rebuild: one pass over the positions for both)
template <bool WRAP>
__global__ __launch_bounds__(FM_BLOCK) void k_bin_count(WrapArgs a, BinArgs b) {
    if (WRAP && blockIdx.x == 0 && (int)threadIdx.x < a.reset.n) reset_flag(a.flags, a.reset.w[threadIdx.x]);
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    int cell = -1;
    if (i < a.np) {
        double r[3] = {a.s.x[i], a.s.y[i], a.s.z[i]};
        if (WRAP) wrap_molecule(a, i, r);
        int c[3] = {0, 0, 0};
        bool ok = true;
#pragma unroll
        for (int d = 0; d < 3; ++d) {
            double t = r[d] + b.h[d];
            ok = ok && t > -b.cs[d] && t < (double)(b.nc[d] + 1) * b.cs[d];  // also rejects NaN
            int ic = ok ? (int)ceil(t / b.cs[d]) + 1 : 0;  // 1-based with one halo layer
            if (ic == 1 && t == 0.0) {  // exactly on the lower face: the reference's ceiling() gives the halo
                atomicAdd(&a.flags[FLAG_EDGE], 1);
                ic = 2;
            }
            ok = ok && ic >= 2 && ic <= b.nc[d] + 1;
            c[d] = ic - 2;
        }
        if (ok) {
            cell = c[0] + b.nc[0] * (c[1] + b.nc[1] * c[2]);
        } else {
            // counted in some cell so that the permutation stays complete; the error stops the run.
            // (All over the box: k_bin_order ranks a cell in n^2 / 64 steps of one wavefront, a minute
            // for a million molecules in one cell)
            // (WRAP: the renumbering that follows turns ~slot into the molecule's number)
            set_err(a.flags, FM_EESCAPE, WRAP ? ~i : a.ext[i]);
            cell = i % (b.nc[0] * b.nc[1] * b.nc[2]);
        }
        b.cell_of[i] = cell;
    }
    // the molecule's place among its cell's molecules (the order within a cell is arbitrary
    // here: k_bin_order orders each cell by x, ties by molecule number)
    const int pos = wave_aggregated_add(b.count, cell, cell >= 0);
    if (i < a.np) b.pos[i] = pos;
}

// start[0..n) = exclusive prefix of the cells' counts, CELL_CH cells a workgroup.  A workgroup adds
// up the counts before its own: by itself from the counts (part null: up to CELL_DIRECT cells, where
// the last workgroup's read of them all costs less than the launch that would sum the chunks), or
// from the chunk sums of k_cell_part.  The counts stay (k_bin_order zeroes them).  One more
// workgroup, when asked, does sendmols' renumbering, which nothing before k_bin_order reads.
#define CELL_CH 4096
#define CELL_DIRECT (1 << 18)
__global__ __launch_bounds__(1024) void k_cell_part(const int* count, int* part, int n) {
    __shared__ int wsum[16];
    int v = 0, tot;
    for (int k = 0; k < 4; ++k) {
        const int i = blockIdx.x * CELL_CH + 4 * threadIdx.x + k;
        v += i < n ? count[i] : 0;
    }
    block_prefix(v, wsum, &tot);
    if (threadIdx.x == 0) part[blockIdx.x] = tot;
}

__global__ __launch_bounds__(1024) void k_cell_scan(const int* count, int* start, const int* part, int n, int nscan,
                                                    RenumArgs ra) {
    __shared__ int wsum[16];
    if ((int)blockIdx.x == nscan) {
        renumber(ra);
        return;
    }
    const int tid = threadIdx.x;
    int before = 0, v[4], s = 0, tot;
    if (part) {
        for (int b = tid; b < (int)blockIdx.x; b += blockDim.x) before += part[b];
    } else {
        const int4* c4 = (const int4*)count;  // (whole chunks: in range)
#pragma unroll 4
        for (int b = 0; b < (int)blockIdx.x; ++b) {
            const int4 w = c4[b * (CELL_CH / 4) + tid];
            before += (w.x + w.y) + (w.z + w.w);
        }
    }
    const int i0 = blockIdx.x * CELL_CH + 4 * tid;
#pragma unroll
    for (int k = 0; k < 4; ++k) {
        v[k] = i0 + k < n ? count[i0 + k] : 0;
        s += v[k];
    }
    int off;
    block_prefix(before, wsum, &off);
    int pre = off + block_prefix(s, wsum, &tot);
#pragma unroll
    for (int k = 0; k < 4; ++k)
        if (i0 + k < n) {
            start[i0 + k] = pre;
            pre += v[k];
        }
}

// start[0..n) = exclusive prefix of count[0..n), in chunks of SCAN_CH counts (FM_BLOCK threads,
// four consecutive counts each): k_scan_part sums each chunk; k_scan_fin adds up the sums of the
// chunks before its own, scans its chunk (by thread, wavefront and workgroup) and writes the
// prefixes (the radix sort's digit counts).
#define SCAN_CH (4 * FM_BLOCK)
__device__ inline int block_sum(int v, int* wsum) {
    const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
    for (int d = 32; d > 0; d >>= 1) v += __shfl_xor(v, d, 64);
    if (lane == 0) wsum[wid] = v;
    __syncthreads();
    int t = 0;
    for (int w = 0; w < FM_BLOCK / 64; ++w) t += wsum[w];
    return t;
}

__global__ __launch_bounds__(FM_BLOCK) void k_scan_part(const int* count, int* part, int n) {
    __shared__ int wsum[FM_BLOCK / 64];
    const int i0 = blockIdx.x * SCAN_CH + 4 * threadIdx.x;
    int v = 0;
#pragma unroll
    for (int k = 0; k < 4; ++k) v += i0 + k < n ? count[i0 + k] : 0;
    const int t = block_sum(v, wsum);
    if (threadIdx.x == 0) part[blockIdx.x] = t;
}

__global__ __launch_bounds__(FM_BLOCK) void k_scan_fin(const int* count, int* start, const int* part, int n) {
    __shared__ int wsum[FM_BLOCK / 64];
    const int tid = threadIdx.x, lane = tid & 63, wid = tid >> 6;
    // the sums of the chunks before this one
    int off = 0;
    for (int b = tid; b < (int)blockIdx.x; b += FM_BLOCK) off += part[b];
    off = block_sum(off, wsum);
    __syncthreads();  // (wsum is used again below)
    const int i0 = blockIdx.x * SCAN_CH + 4 * tid;
    int v[4], s = 0;
#pragma unroll
    for (int k = 0; k < 4; ++k) {
        v[k] = i0 + k < n ? count[i0 + k] : 0;
        s += v[k];
    }
    int x = s;
    for (int d = 1; d < 64; d <<= 1) {
        const int y = __shfl_up(x, d, 64);
        if (lane >= d) x += y;
    }
    if (lane == 63) wsum[wid] = x;
    __syncthreads();
    int pre = off + x - s;
    for (int w = 0; w < wid; ++w) pre += wsum[w];
#pragma unroll
    for (int k = 0; k < 4; ++k)
        if (i0 + k < n) {
            start[i0 + k] = pre;
            pre += v[k];
        }
}

__global__ __launch_bounds__(FM_BLOCK) void k_bin_scatter(const int* cell_of, const int* start, const int* pos,
                                                          int* perm, int np) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < np) perm[start[cell_of[i]] + pos[i]] = i;
}

// ---- order within a cell and the permutation of the state, in one pass ---------------------------
// Each cell's molecules are ordered by increasing x (ties: molecule number), which lets the list
// build window its candidate runs by x, and moved to their new slots.  A molecule's rank is the
// number of its cell's keys below its own; keys are distinct, so the ranks are a permutation.  The
// state goes to the other buffer, so nothing here overwrites what another lane still reads.
// Bound: HBM and the latency of each wavefront's chain (cell start, slots, state), so the state is
// loaded before the ranking and the keys are ranked from LDS.  One launch in place of a sort and a
// permutation: a binning of 1,048,576 molecules 79.5 -> 62 us, of 4,000,000 234 -> 174 us.  Cells
// above 64 molecules (long cutoffs) are ranked by the whole wavefront too, where an insertion sort
// by one lane took 1,000 us at 76 molecules a cell (55,296 molecules, rc 4): now 30 us.
// The key of x is its bits as an integer in the order of the doubles (-0 as +0): a total order, so
// the ranks stay a permutation even with the NaN of an escaped molecule among them.
__device__ inline long long xkey(double x) {
    const long long b = __double_as_longlong(x + 0.0);
    return b ^ ((b >> 63) & 0x7fffffffffffffffll);
}
__device__ inline bool xkey_less(long long xa, int ea, long long xb, int eb) {
    return xa < xb || (xa == xb && ea < eb);
}

struct PermArgs {
    const double* src;
    double* dst;
    const int *ext_src, *mt_src, *tag_src, *mono_src;
    int *ext_dst, *cell_dst, *mt_dst, *tag_dst, *mono_dst;
    const double* teth_src;
    double* teth_dst;
    int* slot_of;
    const int *start, *perm;
    int* count;          // zeroed for the next binning
    int ncell, maxcell, cap;
    int* flags;
    int nf;  // state fields moved: 9, or 6 when the accelerations are about to be recomputed
};

// A molecule's state fields, loaded before its rank is known (the loads run under the ranking) and
// stored at its new slot.
struct Moved {
    int o, e;      // old slot, molecule number
    double f[9];
};
__device__ __forceinline__ void load_molecule(const PermArgs& a, int at, Moved& m) {
    m.o = a.perm[at];
    m.e = a.ext_src[m.o];
#pragma unroll
    for (int f = 0; f < 9; ++f) m.f[f] = f < a.nf ? a.src[m.o + f * (size_t)a.cap] : 0.0;
}
__device__ __forceinline__ void store_molecule(const PermArgs& a, const Moved& m, int k, int c) {
    const size_t cap = a.cap;
#pragma unroll
    for (int f = 0; f < 9; ++f)
        if (f < a.nf) a.dst[k + f * cap] = m.f[f];
    a.ext_dst[k] = m.e;
    a.slot_of[m.e] = k;
    a.cell_dst[k] = c;
    if (a.mt_dst) a.mt_dst[k] = a.mt_src[m.o];
    if (a.tag_dst) {
        a.tag_dst[k] = a.tag_src[m.o];
        double t[6];
#pragma unroll
        for (int f = 0; f < 6; ++f) t[f] = a.teth_src[m.o + f * cap];
#pragma unroll
        for (int f = 0; f < 6; ++f) a.teth_dst[k + f * cap] = t[f];
    }
    if (a.mono_dst) {
        int t[8];
#pragma unroll
        for (int f = 0; f < 8; ++f) t[f] = a.mono_src[m.o + f * cap];
#pragma unroll
        for (int f = 0; f < 8; ++f) a.mono_dst[k + f * cap] = t[f];
    }
}

// orders a wavefront's LDS writes before the reads of its other lanes (and reads before later writes)
__device__ __forceinline__ void wave_sync() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// keys among keys[0..n) below `key`; `same` counts the equal ones
__device__ __forceinline__ int rank_among(const long long* keys, int n, long long key, int& same) {
    int rank = 0;
    for (int k = 0; k < n; ++k) {
        const long long o = keys[k];
        rank += o < key ? 1 : 0;
        same += o == key ? 1 : 0;
    }
    return rank;
}
// the equal keys whose molecule number is below e
__device__ __forceinline__ int rank_ties(const long long* keys, const int* exts, int n, long long key, int e) {
    int rank = 0;
    for (int k = 0; k < n; ++k) rank += (keys[k] == key && exts[k] < e) ? 1 : 0;
    return rank;
}

// One cell by a whole wavefront, 64 molecules at a time against all of the cell's keys, which pass
// through the wavefront's 64 LDS keys in turn.  Any cell size.
__device__ inline void order_cell(const PermArgs& a, int c, long long* keys, int* exts) {
    const int b = a.start[c], n = a.start[c + 1] - b, lane = threadIdx.x & 63;
    for (int q0 = 0; q0 < n; q0 += 64) {
        const bool own = q0 + lane < n;
        Moved m;
        load_molecule(a, b + min(q0 + lane, n - 1), m);
        const long long key = xkey(m.f[0]);
        int rank = 0;
        for (int p0 = 0; p0 < n; p0 += 64) {
            const int u = a.perm[b + min(p0 + lane, n - 1)], cnt = min(64, n - p0);
            wave_sync();
            keys[lane] = p0 == q0 ? key : xkey(a.src[u]);
            exts[lane] = a.ext_src[u];
            wave_sync();
            int same = 0;
            rank += rank_among(keys, cnt, key, same);
            if (__builtin_amdgcn_ballot_w64(same > (p0 == q0 ? 1 : 0)) != 0ull) rank += rank_ties(keys, exts, cnt, key, m.e);
        }
        if (own) store_molecule(a, m, b + rank, c);
    }
}

// PER cells per wavefront.  PER = 2: cells 2w and 2w + 1 side by side on its halves when both hold
// at most 32 molecules, else one after the other.
template <int PER>
__global__ __launch_bounds__(FM_BLOCK) void k_bin_order(PermArgs a) {
    __shared__ long long lkey[FM_BLOCK];
    __shared__ int lext[FM_BLOCK];
    const int lane = threadIdx.x & 63, w0 = threadIdx.x & ~63;
    const int c0 = PER * (int)((blockIdx.x * (size_t)blockDim.x + threadIdx.x) >> 6);
    if (c0 >= a.ncell) return;  // whole wavefront (each keeps to its own 64 LDS keys)
    const int hl = PER == 2 ? lane & 31 : lane, c = c0 + (PER == 2 ? lane >> 5 : 0);
    const int b = c < a.ncell ? a.start[c] : 0, n = c < a.ncell ? a.start[c + 1] - b : 0;
    if (hl == 0 && c < a.ncell) a.count[c] = 0;
    if (n > a.maxcell && hl == 0) set_err(a.flags, FM_EOVERFLOW, c);
    if (PER == 2 && __builtin_amdgcn_ballot_w64(n > 32) == 0ull) {
        const bool own = hl < n;
        Moved m;
        m.e = 0;
        m.f[0] = 0.0;
        if (own) load_molecule(a, b + hl, m);
        const long long key = xkey(m.f[0]);
        lkey[threadIdx.x] = key;
        lext[threadIdx.x] = m.e;
        wave_sync();
        const long long* keys = lkey + w0 + (lane & 32);
        int same = 0, rank = rank_among(keys, n, key, same);
        if (__builtin_amdgcn_ballot_w64(own && same > 1) != 0ull) rank += rank_ties(keys, lext + w0 + (lane & 32), n, key, m.e);
        if (own) store_molecule(a, m, b + rank, c);
        return;
    }
    order_cell(a, c0, lkey + w0, lext + w0);
    if (PER == 2 && c0 + 1 < a.ncell) order_cell(a, c0 + 1, lkey + w0, lext + w0);
}

// Cells of few molecules: a thread per molecule, which reads the keys of its cell's others itself (any cell
// size).  A wavefront of k_bin_order would hold two of these cells and move their molecules with a few of
// its lanes.  A binning, us by k_bin_order and by this: 1,048,576 molecules at 0.22 a cell 728 and 110, 1.1
// 272 and 90, 4.4 115 and 79, 7.5 89 and 76, 10.1 81 and 77, 13 73 and 81, 17.7 68 and 83; 4,000,000 WCA (2.3)
// 635 and 262; but 108,000 at 10 a cell 25 and 32, 32,000 WCA 26 and 28, 2,048 (2.8) 21 and 23.5, where a
// launch has few wavefronts either way.  So up to eleven a cell from SPARSE_CELLS cells on (108,000 at 6.1 a
// cell, 17,576 cells: 27.5 and 27.9).
#define SPARSE_OCC 11
#define SPARSE_CELLS 16384
__global__ __launch_bounds__(FM_BLOCK) void k_bin_order_sparse(PermArgs a, const int* cell_of, int np) {
    const int k = blockIdx.x * blockDim.x + threadIdx.x;
    if (k >= np) return;
    Moved m;
    load_molecule(a, k, m);
    const int c = cell_of[m.o], b = a.start[c], n = a.start[c + 1] - b;
    if (k == b) {
        a.count[c] = 0;  // (an empty cell's is zero)
        if (n > a.maxcell) set_err(a.flags, FM_EOVERFLOW, c);
    }
    const long long key = xkey(m.f[0]);
    int rank = 0;
    for (int q = 0; q < n; ++q) {
        const int u = a.perm[b + q];
        const long long o = xkey(a.src[u]);
        if (o < key || (o == key && u != m.o && a.ext_src[u] < m.e)) ++rank;
    }
    store_molecule(a, m, b + rank, c);
}

// ---- macroscopic sums, src/simulation_record.f90:1205-1314 ------------------------------------
// 7 sums per block: pe_lj, pe_poly, pe_lj+pe_poly, vir, mv2, vsum, msum ; + max(pe).  Each thread
// sums MACRO_MPT molecules a grid apart (in that order), then the wavefront and the workgroup.
#define NRED 8
#define MACRO_MPT 4
__global__ __launch_bounds__(FM_BLOCK) void k_macros_partial(St s, const double* pe_lj, const double* pe_poly,
                                                             const double* vir, const int* moltype,
                                                             const double* mass, int np, int lfv, double dt,
                                                             double* part) {
    __shared__ double red[NRED][FM_BLOCK / 64];
    double v[NRED] = {0, 0, 0, 0, 0, 0, 0, -1.0e300};
    const int stride = gridDim.x * blockDim.x;
#pragma unroll
    for (int k = 0; k < MACRO_MPT; ++k) {
        const int i = blockIdx.x * blockDim.x + threadIdx.x + k * stride;
        if (i >= np) break;
        double m = moltype ? mass[moltype[i]] : 1.0;
        double pl = pe_lj[i], pp = pe_poly ? pe_poly[i] : 0.0;
        v[0] = v[0] + pl;
        v[1] = v[1] + pp;
        v[2] = v[2] + (pl + pp);
        v[3] = v[3] + vir[i];
        double vx = s.vx[i], vy = s.vy[i], vz = s.vz[i];
        if (lfv) {  // leap-frog: velocity shifted half a step, src/simulation_record.f90:1238-1247
            vx = vx + 0.5 * s.ax[i] * dt;
            vy = vy + 0.5 * s.ay[i] * dt;
            vz = vz + 0.5 * s.az[i] * dt;
        }
        v[4] = v[4] + ((m * (vx * vx) + m * (vy * vy)) + m * (vz * vz));
        v[5] = v[5] + ((m * vx + m * vy) + m * vz);
        v[6] = v[6] + m;
        v[7] = fmax(v[7], pl + pp);
    }
    for (int q = 0; q < NRED; ++q) {
        double x = v[q];
        for (int off = 32; off > 0; off >>= 1) {
            double o = __shfl_down(x, off, 64);
            x = q == 7 ? fmax(x, o) : x + o;
        }
        if ((threadIdx.x & 63) == 0) red[q][threadIdx.x >> 6] = x;
    }
    __syncthreads();
    if (threadIdx.x < NRED) {
        int q = threadIdx.x;
        double x = red[q][0];
        for (int w = 1; w < FM_BLOCK / 64; ++w) x = q == 7 ? fmax(x, red[q][w]) : x + red[q][w];
        part[(size_t)blockIdx.x * NRED + q] = x;
    }
}

// one workgroup: thread t sums partials t, t+256, ... in that order, then a fixed tree over the
// threads (deterministic; the partial count is the number of k_macros_partial workgroups)
__global__ __launch_bounds__(256) void k_macros_final(const double* part, int nb, double* out) {
    __shared__ double red[NRED][256];
    const int t = threadIdx.x;
    double x[NRED];
#pragma unroll
    for (int q = 0; q < NRED; ++q) x[q] = q == 7 ? -1.0e300 : 0.0;
    for (int b = t; b < nb; b += 256) {
#pragma unroll
        for (int q = 0; q < NRED; ++q) {
            const double o = part[(size_t)b * NRED + q];
            x[q] = q == 7 ? fmax(x[q], o) : x[q] + o;
        }
    }
#pragma unroll
    for (int q = 0; q < NRED; ++q) red[q][t] = x[q];
    __syncthreads();
    for (int h = 128; h > 0; h >>= 1) {
        if (t < h)
#pragma unroll
            for (int q = 0; q < NRED; ++q) red[q][t] = q == 7 ? fmax(red[q][t], red[q][t + h]) : red[q][t] + red[q][t + h];
        __syncthreads();
    }
    if (t < NRED) out[t] = red[t][0];
}

// ---- host-order staging ---------------------------------------------------------------------
__global__ __launch_bounds__(FM_BLOCK) void k_to_host(St s, const int* ext, int np, double* out) {
    int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= np) return;
    size_t e = ext[i];
    const size_t n3 = 3 * (size_t)np;
    out[3 * e] = s.x[i];
    out[3 * e + 1] = s.y[i];
    out[3 * e + 2] = s.z[i];
    out[n3 + 3 * e] = s.vx[i];
    out[n3 + 3 * e + 1] = s.vy[i];
    out[n3 + 3 * e + 2] = s.vz[i];
    out[2 * n3 + 3 * e] = s.ax[i];
    out[2 * n3 + 3 * e + 1] = s.ay[i];
    out[2 * n3 + 3 * e + 2] = s.az[i];
}

// host (molecule-number) order <-> slot order
__global__ __launch_bounds__(FM_BLOCK) void k_from_host(St s, int* ext, int* slot_of, int np, const double* in) {
    int e = blockIdx.x * blockDim.x + threadIdx.x;
    if (e >= np) return;
    const size_t n3 = 3 * (size_t)np;
    s.x[e] = in[3 * (size_t)e];
    s.y[e] = in[3 * (size_t)e + 1];
    s.z[e] = in[3 * (size_t)e + 2];
    s.vx[e] = in[n3 + 3 * (size_t)e];
    s.vy[e] = in[n3 + 3 * (size_t)e + 1];
    s.vz[e] = in[n3 + 3 * (size_t)e + 2];
    s.ax[e] = in[2 * n3 + 3 * (size_t)e];
    s.ay[e] = in[2 * n3 + 3 * (size_t)e + 1];
    s.az[e] = in[2 * n3 + 3 * (size_t)e + 2];
    ext[e] = e;
    slot_of[e] = e;
}

// dst[s + f*cap] = src[ext[s]*nf + f]
template <typename T>
__global__ __launch_bounds__(FM_BLOCK) void k_ext_to_slot(T* dst, int cap, const T* src, int nf, const int* ext, int np) {
    int s = blockIdx.x * blockDim.x + threadIdx.x;
    if (s >= np) return;
    size_t e = ext[s];
    for (int f = 0; f < nf; ++f) dst[s + (size_t)f * cap] = src[e * nf + f];
}

// dst[ext[s]*nf + f] = src[s + f*cap]
template <typename T>
__global__ __launch_bounds__(FM_BLOCK) void k_slot_to_ext(T* dst, const T* src, int cap, int nf, const int* ext, int np) {
    int s = blockIdx.x * blockDim.x + threadIdx.x;
    if (s >= np) return;
    size_t e = ext[s];
    for (int f = 0; f < nf; ++f) dst[e * nf + f] = src[s + (size_t)f * cap];
}

// packed VV pass 1 (+ displacement check) over many domains: block b handles molecules
// table[b].y*FM_BLOCK .. of domain table[b].x (same operations as k_pass1 / k_pass1_disp).  A
// domain's pass does nothing when it has no step in this launch, or when a rebuild is pending
// for an earlier step (FLAG_HALT, or FLAG_REBUILD with FLAG_RB_STEP below this step: a check of
// this same launch stores this step, so its other workgroups still run); a check that fires
// records this step.
__global__ __launch_bounds__(FM_BLOCK) void k_pass1_multi(const P1Desc* descs, const int2* table) {
    const int2 t = table[blockIdx.x];
    const P1Desc& d = descs[t.x];
    if (!d.active) return;
    int* f = d.flags;
    if (f[FLAG_HALT] != 0 || (__atomic_load_n(&f[FLAG_REBUILD], __ATOMIC_RELAXED) != 0 &&
                              __atomic_load_n(&f[FLAG_RB_STEP], __ATOMIC_RELAXED) < d.step))
        return;
    const int i = t.y * FM_BLOCK + threadIdx.x;
    bool hit = false;
    if (i < d.np) {
        St s = state_of(d.st, d.cap);
        const double ax = s.ax[i], ay = s.ay[i], az = s.az[i];
        double vx = s.vx[i], vy = s.vy[i], vz = s.vz[i];
        s.x[i] = s.x[i] + d.dt * vx + d.hdt2 * ax;
        s.y[i] = s.y[i] + d.dt * vy + d.hdt2 * ay;
        s.z[i] = s.z[i] + d.dt * vz + d.hdt2 * az;
        vx = vx + d.hdt * ax;
        vy = vy + d.hdt * ay;
        vz = vz + d.hdt * az;
        s.vx[i] = vx;
        s.vy[i] = vy;
        s.vz[i] = vz;
        if (d.check) {
            const size_t cap = d.cap;
            double d0 = d.fresh ? 0.0 : d.rd[i];
            double d1 = d.fresh ? 0.0 : d.rd[i + cap];
            double d2 = d.fresh ? 0.0 : d.rd[i + 2 * cap];
            d0 = d0 + vx * d.dt;
            d1 = d1 + vy * d.dt;
            d2 = d2 + vz * d.dt;
            d.rd[i] = d0;
            d.rd[i + cap] = d1;
            d.rd[i + 2 * cap] = d2;
            hit = fabs(d0) > d.thresh || fabs(d1) > d.thresh || fabs(d2) > d.thresh;
        }
    }
    unsigned long long m = __ballot(hit);
    if (m != 0ull && (int)(threadIdx.x & 63) == __ffsll((long long)m) - 1 &&
        __atomic_load_n(&f[FLAG_REBUILD], __ATOMIC_RELAXED) == 0) {
        atomicOr(&f[FLAG_REBUILD], 1);
        atomicExch(&f[FLAG_RB_STEP], d.step);
    }
}

}  // namespace

// =============================================================================================
// launchers
#define LAUNCH_CHECK()                                                                       \
    do {                                                                                     \
        hipError_t _e = hipGetLastError();                                                   \
        if (_e != hipSuccess) return fm_set_error(FM_EHIP, "kernel launch: %s (%s:%d)",       \
                                                  hipGetErrorString(_e), __FILE__, __LINE__); \
    } while (0)

int launch_fill_i32(fm_ctx* c, int* p, int v, size_t n) {
    if (n == 0) return 0;
    k_fill_i32<<<nblocks(n), FM_BLOCK, 0, c->stream>>>(p, v, n);
    LAUNCH_CHECK();
    return 0;
}

int launch_fill_f64(fm_ctx* c, double* p, double v, size_t n) {
    if (n == 0) return 0;
    k_fill_f64<<<nblocks(n), FM_BLOCK, 0, c->stream>>>(p, v, n);
    LAUNCH_CHECK();
    return 0;
}

int launch_pass1(fm_ctx* c, bool cond) {
    if (c->np == 0) return 0;
    double dt = c->p.delta_t;
    ktimer_begin(c, KT_PASS1);
    k_pass1<<<nblocks(c->np), FM_BLOCK, 0, c->stream>>>(state_of(c->x(), c->cap), c->np, dt, 0.5 * (dt * dt),
                                                         0.5 * dt, cond ? c->d_flags : nullptr);
    ktimer_end(c, KT_PASS1);
    LAUNCH_CHECK();
    return 0;
}

int launch_pass2(fm_ctx* c) {
    if (c->np == 0) return 0;
    ktimer_begin(c, KT_PASS2);
    k_pass2<<<nblocks(c->np), FM_BLOCK, 0, c->stream>>>(state_of(c->x(), c->cap), c->np, 0.5 * c->p.delta_t);
    ktimer_end(c, KT_PASS2);
    LAUNCH_CHECK();
    return 0;
}

int launch_check_disp(fm_ctx* c) {
    if (c->np == 0) return 0;
    ktimer_begin(c, KT_CHECK);
    k_check_disp<<<nblocks(c->np), FM_BLOCK, 0, c->stream>>>(state_of(c->x(), c->cap), c->rdisp, c->np, c->cap,
                                                              c->p.delta_t, 0.5 * c->dmin,
                                                              c->rdisp_valid ? 0 : 1, c->d_flags);
    ktimer_end(c, KT_CHECK);
    LAUNCH_CHECK();
    c->rdisp_valid = true;
    return 0;
}

// zero the listed flag words (one launch for the resets before a queued stage)
__global__ void k_reset_flags(int* flags, FlagList l) {
    if ((int)threadIdx.x < l.n) reset_flag(flags, l.w[threadIdx.x]);
}

int launch_reset_flags(fm_ctx* c, const int* which, int n) {
    if (n < 1 || n > 8) return fm_set_error(FM_EINVAL, "reset of %d flag words", n);
    FlagList l;
    l.n = n;
    for (int k = 0; k < n; ++k) l.w[k] = which[k];
    k_reset_flags<<<1, 64, 0, c->stream>>>(c->d_flags, l);
    LAUNCH_CHECK();
    return 0;
}

// ---- sort_mols, src/linklist.f90:2744-2865 ------------------------------------------------------
// key[e] = curve position of molecule e's block, val[e] = e; cnt[key] counts the block
__global__ __launch_bounds__(FM_BLOCK) void k_sort_keys(St s, const int* slot_of, int np, const int* hcurve,
                                                         int nb0, int nb1, int nb2, double b0, double b1, double b2,
                                                         double h0, double h1, double h2, int* key, int* val,
                                                         int* cnt, int* flags) {
    const int e = blockIdx.x * blockDim.x + threadIdx.x;
    if (e >= np) return;
    const int slot = slot_of[e];
    const int i = (int)ceil((s.x[slot] + h0) / b0), j = (int)ceil((s.y[slot] + h1) / b1),
              k = (int)ceil((s.z[slot] + h2) / b2);
    if (i < 1 || i > nb0 || j < 1 || j > nb1 || k < 1 || k > nb2) {
        set_err(flags, FM_EESCAPE, e);
        key[e] = 0;
        val[e] = e;
        return;
    }
    const int c = hcurve[(i - 1) + nb0 * ((j - 1) + nb1 * (k - 1))];
    key[e] = c;
    val[e] = e;
    atomicAdd(&cnt[c], 1);
}

// order[k] = old number of the molecule that becomes number k -> relabel the slots
__global__ __launch_bounds__(FM_BLOCK) void k_sort_newof(const int* order, int np, int* newof) {
    const int k = blockIdx.x * blockDim.x + threadIdx.x;
    if (k < np) newof[order[k]] = k;
}

__global__ __launch_bounds__(FM_BLOCK) void k_sort_relabel(St s, int* ext, int* slot_of, const int* newof, int np,
                                                            const int* tag, double* teth, int cap, double w0,
                                                            double w1, double w2) {
    const int slot = blockIdx.x * blockDim.x + threadIdx.x;
    if (slot >= np) return;
    const int e = newof[ext[slot]];
    ext[slot] = e;
    slot_of[e] = slot;
    if (tag) {  // read_tag on every renumbered molecule
        const int tg = tag[slot];
        const double sg = tg == FM_TAG_TETH_SLIDE ? copysign(1.0, s.y[slot]) : tg == FM_TAG_FIXED_SLIDE ? 1.0 : 0.0;
        teth[slot + 3 * (size_t)cap] = sg != 0.0 ? w0 * sg : 0.0;
        teth[slot + 4 * (size_t)cap] = sg != 0.0 ? w1 * sg : 0.0;
        teth[slot + 5 * (size_t)cap] = sg != 0.0 ? w2 * sg : 0.0;
    }
}

// flags[flag] = max(flags[flag], v[0..n)) for an arbitrary array
__global__ __launch_bounds__(FM_BLOCK) void k_max_of(const int* v, int n, int* flag) {
    __shared__ int sm[FM_BLOCK / 64];
    int m = INT_MIN;
    for (int k = threadIdx.x; k < n; k += blockDim.x) m = max(m, v[k]);
    for (int off = 32; off > 0; off >>= 1) m = max(m, __shfl_xor(m, off, 64));
    if ((threadIdx.x & 63) == 0) sm[threadIdx.x >> 6] = m;
    __syncthreads();
    if (threadIdx.x == 0) {
        for (int w = 1; w < FM_BLOCK / 64; ++w) m = max(m, sm[w]);
        m = max(m, sm[0]);
        *flag = m;
    }
}

// ---- stable LSD radix sort of (key, value) pairs, 8 bits a pass ---------------------------------
// Each workgroup takes a tile of FM_BLOCK consecutive pairs.  k_radix_hist counts the tile's digits
// into hist[digit * ntiles + tile]: digit-major, so the exclusive prefix of the whole array (the
// chunked scan above) is, for each tile and digit, the first output position of that tile's pairs
// with that digit.  k_radix_scatter places each pair after the pairs of its digit that come before
// it in its tile: the lanes of its wavefront below it whose digit matches (eight ballots, one per
// digit bit) and the matching counts of the wavefronts before its own.  Tiles, wavefronts and lanes
// keep the input order, so every pass is stable.
static_assert(FM_BLOCK == 256, "one 8-bit digit bucket per thread of the tile");

__global__ __launch_bounds__(FM_BLOCK) void k_radix_hist(const int* key, int n, int shift, int* hist, int ntiles) {
    __shared__ int h[256];
    h[threadIdx.x] = 0;
    __syncthreads();
    const int i = blockIdx.x * FM_BLOCK + threadIdx.x;
    if (i < n) atomicAdd(&h[(key[i] >> shift) & 255], 1);
    __syncthreads();
    hist[(size_t)threadIdx.x * ntiles + blockIdx.x] = h[threadIdx.x];
}

__global__ __launch_bounds__(FM_BLOCK) void k_radix_scatter(const int* kin, const int* vin, int* kout, int* vout,
                                                             int n, int shift, const int* start, int ntiles) {
    __shared__ int wc[FM_BLOCK / 64][256];
    const int tid = threadIdx.x, lane = tid & 63, wid = tid >> 6;
    for (int w = 0; w < FM_BLOCK / 64; ++w) wc[w][tid] = 0;
    __syncthreads();
    const int i = blockIdx.x * FM_BLOCK + tid;
    const bool active = i < n;
    const int k = active ? kin[i] : 0;
    const int d = (k >> shift) & 255;
    uint64_t m = __ballot(active);
#pragma unroll
    for (int b = 0; b < 8; ++b) {
        const uint64_t on = __ballot((d >> b) & 1);
        m &= ((d >> b) & 1) ? on : ~on;
    }
    const int rank = __popcll(m & ((1ull << lane) - 1ull));
    if (active && rank == 0) wc[wid][d] = __popcll(m);
    __syncthreads();
    if (!active) return;
    int pos = start[(size_t)d * ntiles + blockIdx.x] + rank;
    for (int w = 0; w < wid; ++w) pos += wc[w][d];
    kout[pos] = k;
    vout[pos] = vin[i];
}

size_t radix_sort_bytes(int n) {
    const size_t nt = ((size_t)std::max(n, 1) + FM_BLOCK - 1) / FM_BLOCK, nh = 256 * nt;
    return (2 * nh + nh / SCAN_CH + 2) * sizeof(int);
}

// Sorts the pairs (k0, v0)[0..n) by key bits [0, end_bit), stably, with (k1, v1) as the other
// buffer of each pass; *vals is the buffer that ends with the sorted values.
int radix_sort_pairs(fm_ctx* c, int* k0, int* v0, int* k1, int* v1, int n, int end_bit, int** vals) {
    const int nt = (n + FM_BLOCK - 1) / FM_BLOCK, nh = 256 * nt, nscan = (nh + SCAN_CH - 1) / SCAN_CH;
    if ((size_t)(2 * (size_t)nh + nh / SCAN_CH + 2) * sizeof(int) > c->sort_tmp_bytes)
        return fm_set_error(FM_EOVERFLOW, "radix sort of %d pairs exceeds its temporary", n);
    int* hist = (int*)c->sort_tmp;
    int* start = hist + nh;
    int* part = start + nh;
    for (int shift = 0; shift < end_bit; shift += 8) {
        k_radix_hist<<<nt, FM_BLOCK, 0, c->stream>>>(k0, n, shift, hist, nt);
        k_scan_part<<<nscan, FM_BLOCK, 0, c->stream>>>(hist, part, nh);
        k_scan_fin<<<nscan, FM_BLOCK, 0, c->stream>>>(hist, start, part, nh);
        k_radix_scatter<<<nt, FM_BLOCK, 0, c->stream>>>(k0, v0, k1, v1, n, shift, start, nt);
        LAUNCH_CHECK();
        std::swap(k0, k1);
        std::swap(v0, v1);
    }
    *vals = v0;
    return 0;
}

// One sort_mols renumbering (the caller handles the call counter).  *overflow_out = 1 when a
// block exceeds the estimate and the round is skipped, as the reference does.
int launch_sort_mols(fm_ctx* c, int* overflow_out) {
    *overflow_out = 0;
    if (c->np == 0) return 0;
    const int blocks = c->sort_nb[0] * c->sort_nb[1] * c->sort_nb[2];
    int ave = c->np / blocks;
    ave = (int)ceil(ave * c->sort_sf1 + c->sort_sf2);
    if (int rc = launch_fill_i32(c, c->sort_cnt, 0, (size_t)blocks + 1)) return rc;
    St s = state_of(c->x(), c->cap);
    k_sort_keys<<<nblocks(c->np), FM_BLOCK, 0, c->stream>>>(
        s, c->slot_of, c->np, c->hcurve, c->sort_nb[0], c->sort_nb[1], c->sort_nb[2], c->sort_bsl[0], c->sort_bsl[1],
        c->sort_bsl[2], c->half[0], c->half[1], c->half[2], c->sort_key, c->sort_val, c->sort_cnt, c->d_flags);
    LAUNCH_CHECK();
    k_max_of<<<1, FM_BLOCK, 0, c->stream>>>(c->sort_cnt, blocks + 1, c->d_flags + FLAG_SORT_MAX);
    LAUNCH_CHECK();
    if (int rc = ctx_sync_flags(c)) return rc;
    if (c->h_flags[FLAG_SORT_MAX] > ave) {  // "Miss this round of sorting"
        c->sort_sf1 = c->sort_sf1 + 0.1;
        c->sort_sf2 = c->sort_sf2 + 5;
        *overflow_out = 1;
        return 0;
    }
    int end_bit = 1;
    while ((1 << end_bit) <= blocks) ++end_bit;
    int* order = nullptr;
    if (int rc = radix_sort_pairs(c, c->sort_key, c->sort_val, c->sort_key2, c->sort_val2, c->np, end_bit, &order))
        return rc;
    // the keys are spent: sort_key takes the new numbers (order is a value buffer)
    k_sort_newof<<<nblocks(c->np), FM_BLOCK, 0, c->stream>>>(order, c->np, c->sort_key);
    LAUNCH_CHECK();
    const bool tm = c->p.ensemble == FM_ENSEMBLE_TAG_MOVE && c->has_tags;
    k_sort_relabel<<<nblocks(c->np), FM_BLOCK, 0, c->stream>>>(
        s, c->ext[c->cur], c->slot_of, c->sort_key, c->np, tm ? c->tag[c->cur] : nullptr,
        tm ? c->teth[c->cur] : nullptr, c->cap, c->p.wallslidev[0], c->p.wallslidev[1], c->p.wallslidev[2]);
    LAUNCH_CHECK();
    return 0;
}

// simulation_move_particles_lfv; check_disp: fused displacement update of rebuild criterion 2
int launch_move_lfv(fm_ctx* c, bool check_disp, bool cond) {
    if (c->np == 0) return 0;
    const bool tm = c->p.ensemble == FM_ENSEMBLE_TAG_MOVE;
    ktimer_begin(c, KT_PASS1);
    k_move_lfv<<<nblocks(c->np), FM_BLOCK, 0, c->stream>>>(
        state_of(c->x(), c->cap), tm ? c->tag[c->cur] : nullptr, tm ? c->teth[c->cur] : nullptr, c->ext[c->cur],
        c->np, c->cap, c->p.delta_t, c->p.teth_k2, c->p.teth_k4, c->p.teth_k6, c->rdisp, 0.5 * c->dmin,
        check_disp ? 1 : 0, c->rdisp_valid ? 0 : 1, c->d_flags, cond ? 1 : 0);
    ktimer_end(c, KT_PASS1);
    LAUNCH_CHECK();
    if (check_disp) c->rdisp_valid = true;
    return 0;
}

int launch_check_vmax(fm_ctx* c) {
    ktimer_begin(c, KT_CHECK);
    if (c->np > 0) k_vmax<<<nblocks(c->np), FM_BLOCK, 0, c->stream>>>(state_of(c->x(), c->cap), c->np, c->d_vmax);
    k_vmax_finish<<<1, 1, 0, c->stream>>>(c->d_vmax, c->d_rmax, c->p.delta_t, 0.5 * c->dmin, 0, c->d_flags);
    ktimer_end(c, KT_CHECK);
    LAUNCH_CHECK();
    return 0;
}

static int make_wrap(fm_ctx* c, WrapArgs& a, const int* reset, int nreset) {
    if (nreset > 8) return fm_set_error(FM_EINVAL, "reset of %d flag words", nreset);
    const bool tm = c->p.ensemble == FM_ENSEMBLE_TAG_MOVE && c->has_tags;
    a.s = state_of(c->x(), c->cap);
    a.ext = c->ext[c->cur];
    a.tag = tm ? c->tag[c->cur] : nullptr;
    a.teth = tm ? c->teth[c->cur] : nullptr;
    a.np = c->np;
    a.cap = c->cap;
    for (int d = 0; d < 3; ++d) {
        a.L[d] = c->p.domain[d];
        a.ws[d] = c->p.wallslidev[d];
    }
    a.mask = c->out_mask;
    a.bits = c->out_bits;
    a.flags = c->d_flags;
    a.reset.n = nreset;
    for (int k = 0; k < nreset; ++k) a.reset.w[k] = reset[k];
    return 0;
}

static RenumArgs make_renum(fm_ctx* c, bool set_slots) {
    RenumArgs r;
    r.np = c->np;
    r.bits = c->out_bits;
    r.mask = c->out_mask;
    r.ext = c->ext[c->cur];
    r.slot_of = c->slot_of;
    r.scratch = (int*)c->stage;  // 9*cap doubles, used by host transfers only
    r.cap = c->cap;
    r.set_slots = set_slots ? 1 : 0;
    r.flags = c->d_flags;
    return r;
}

int launch_sendmols(fm_ctx* c, const int* reset, int nreset) {
    if (c->np == 0) return nreset ? launch_reset_flags(c, reset, nreset) : 0;
    WrapArgs w;
    if (int rc = make_wrap(c, w, reset, nreset)) return rc;
    ktimer_begin(c, KT_SENDMOLS);
    k_wrap<<<nblocks(c->np), FM_BLOCK, 0, c->stream>>>(w);
    LAUNCH_CHECK();
    k_renumber<<<1, 1024, 0, c->stream>>>(make_renum(c, true));
    ktimer_end(c, KT_SENDMOLS);
    LAUNCH_CHECK();
    return 0;
}

// send: sendmols first, in the binning's own launches (its wrap with the cell counts, its
// renumbering beside the scan), zeroing the listed flags.  sort_mols, which renumbers between the
// two, needs them apart.
int launch_bin(fm_ctx* c, bool keep_acc, bool send, const int* reset, int nreset) {
    c->btab_valid = false;  // new cells: the staging tables wait for the next list build
    if (c->np == 0) return nreset ? launch_reset_flags(c, reset, nreset) : 0;
    WrapArgs w;
    if (int rc = make_wrap(c, w, reset, nreset)) return rc;
    ktimer_begin(c, KT_BIN);
    const int nxt = 1 - c->cur;
    int* cell_tmp = c->out_flag;  // cell index in old slot order
    BinArgs b;
    for (int d = 0; d < 3; ++d) {
        b.h[d] = c->half[d];
        b.cs[d] = c->cs[d];
        b.nc[d] = c->nc[d];
    }
    b.cell_of = cell_tmp;
    b.count = c->cell_count;
    b.pos = c->bin_pos;
    if (send) k_bin_count<true><<<nblocks(c->np), FM_BLOCK, 0, c->stream>>>(w, b);
    else k_bin_count<false><<<nblocks(c->np), FM_BLOCK, 0, c->stream>>>(w, b);
    LAUNCH_CHECK();
    const int n = c->ncell + 1, nscan = (n + CELL_CH - 1) / CELL_CH;
    const bool part = n > CELL_DIRECT;
    if (part) {
        k_cell_part<<<nscan, 1024, 0, c->stream>>>(c->cell_count, c->scan_part, n);
        LAUNCH_CHECK();
    }
    k_cell_scan<<<nscan + (send ? 1 : 0), 1024, 0, c->stream>>>(c->cell_count, c->cell_start, part ? c->scan_part : nullptr,
                                                                n, nscan, make_renum(c, false));
    LAUNCH_CHECK();
    k_bin_scatter<<<nblocks(c->np), FM_BLOCK, 0, c->stream>>>(cell_tmp, c->cell_start, c->bin_pos, c->perm,
                                                               c->np);
    LAUNCH_CHECK();
    PermArgs a;
    a.src = c->st[c->scur];
    a.dst = c->st[1 - c->scur];
    a.ext_src = c->ext[c->cur];
    a.ext_dst = c->ext[nxt];
    a.cell_dst = c->cell_of;
    a.mt_src = c->has_moltype ? c->moltype[c->cur] : nullptr;
    a.mt_dst = c->has_moltype ? c->moltype[nxt] : nullptr;
    a.tag_src = c->has_tags ? c->tag[c->cur] : nullptr;
    a.tag_dst = c->has_tags ? c->tag[nxt] : nullptr;
    a.teth_src = c->has_tags ? c->teth[c->cur] : nullptr;
    a.teth_dst = c->has_tags ? c->teth[nxt] : nullptr;
    a.mono_src = c->has_mono ? c->mono[c->cur] : nullptr;
    a.mono_dst = c->has_mono ? c->mono[nxt] : nullptr;
    a.slot_of = c->slot_of;
    a.start = c->cell_start;
    a.perm = c->perm;
    a.count = c->cell_count;
    a.ncell = c->ncell;
    a.maxcell = c->p.max_cell_np > 0 ? c->p.max_cell_np : (1 << 26);
    a.cap = c->cap;
    a.flags = c->d_flags;
    a.nf = keep_acc ? 9 : 6;
    // two cells per wavefront while most cells fit its halves (a mean of 24 keeps nearly all
    // below 32), one above that
    const int per = (size_t)c->np <= 24 * (size_t)c->ncell ? 2 : 1;
    const int nsort = nblocks((size_t)((c->ncell + per - 1) / per) * 64);
    if (c->ncell >= SPARSE_CELLS && (size_t)c->np <= SPARSE_OCC * (size_t)c->ncell)
        k_bin_order_sparse<<<nblocks(c->np), FM_BLOCK, 0, c->stream>>>(a, cell_tmp, c->np);
    else if (per == 2) k_bin_order<2><<<nsort, FM_BLOCK, 0, c->stream>>>(a);
    else k_bin_order<1><<<nsort, FM_BLOCK, 0, c->stream>>>(a);
    ktimer_end(c, KT_BIN);
    LAUNCH_CHECK();
    c->cur = nxt;
    c->scur = 1 - c->scur;
    return 0;
}

int launch_macros(fm_ctx* c, int buf, double* out) {
    int nb = nblocks((c->np + MACRO_MPT - 1) / MACRO_MPT);
    if (nb == 0) nb = 1;
    if (buf < 0) buf = c->scur;
    ktimer_begin(c, KT_MACROS);
    const bool mie = c->p.mie_potential == 1;
    const bool poly = c->p.potential_flag == 1 && c->has_mono;
    k_macros_partial<<<nb, FM_BLOCK, 0, c->stream>>>(state_of(c->st[buf], c->cap), c->pe_lj, poly ? c->pe_poly : nullptr,
                                                      c->vir, mie ? c->moltype[c->cur] : nullptr,
                                                      c->d_mie + 7 * FM_MAX_TYPES * FM_MAX_TYPES,
                                                      c->np, c->p.integration_algorithm == FM_INTEGRATION_LFV ? 1 : 0,
                                                      c->p.delta_t, c->red);
    k_macros_final<<<1, 256, 0, c->stream>>>(c->red, nb, out ? out : c->d_macros);
    ktimer_end(c, KT_MACROS);
    LAUNCH_CHECK();
    return 0;
}

int launch_scatter_state_to_host_order(fm_ctx* c, double* d_out9, double*) {
    if (c->np == 0) return 0;
    k_to_host<<<nblocks(c->np), FM_BLOCK, 0, c->stream>>>(state_of(c->x(), c->cap), c->ext[c->cur], c->np, d_out9);
    LAUNCH_CHECK();
    return 0;
}

int launch_from_host(fm_ctx* c, const double* d_in9) {
    if (c->np == 0) return 0;
    k_from_host<<<nblocks(c->np), FM_BLOCK, 0, c->stream>>>(state_of(c->x(), c->cap), c->ext[c->cur], c->slot_of,
                                                             c->np, d_in9);
    LAUNCH_CHECK();
    return 0;
}

int launch_ext_to_slot_i32(fm_ctx* c, int* dst, const int* src, int nf) {
    if (c->np == 0) return 0;
    k_ext_to_slot<int><<<nblocks(c->np), FM_BLOCK, 0, c->stream>>>(dst, c->cap, src, nf, c->ext[c->cur], c->np);
    LAUNCH_CHECK();
    return 0;
}

int launch_ext_to_slot_f64(fm_ctx* c, double* dst, const double* src, int nf) {
    if (c->np == 0) return 0;
    k_ext_to_slot<double><<<nblocks(c->np), FM_BLOCK, 0, c->stream>>>(dst, c->cap, src, nf, c->ext[c->cur], c->np);
    LAUNCH_CHECK();
    return 0;
}

int launch_slot_to_ext_f64(fm_ctx* c, double* dst, const double* src, int nf) {
    if (c->np == 0) return 0;
    k_slot_to_ext<double><<<nblocks(c->np), FM_BLOCK, 0, c->stream>>>(dst, src, c->cap, nf, c->ext[c->cur], c->np);
    LAUNCH_CHECK();
    return 0;
}

int launch_slot_to_ext_i32(fm_ctx* c, int* dst, const int* src, int nf) {
    if (c->np == 0) return 0;
    k_slot_to_ext<int><<<nblocks(c->np), FM_BLOCK, 0, c->stream>>>(dst, src, c->cap, nf, c->ext[c->cur], c->np);
    LAUNCH_CHECK();
    return 0;
}

int launch_pass1_check_disp(fm_ctx* c, bool cond, int step) {
    if (c->np == 0) return 0;
    const double dt = c->p.delta_t;
    ktimer_begin(c, KT_PASS1);
    k_pass1_disp<<<nblocks(c->np), FM_BLOCK, 0, c->stream>>>(state_of(c->x(), c->cap), c->rdisp, c->np, c->cap, dt,
                                                              0.5 * (dt * dt), 0.5 * dt, 0.5 * c->dmin,
                                                              c->rdisp_valid ? 0 : 1, c->d_flags, cond ? 1 : 0, step);
    ktimer_end(c, KT_PASS1);
    LAUNCH_CHECK();
    c->rdisp_valid = true;
    return 0;
}

int launch_pass1_multi(hipStream_t st, const P1Desc* d_descs, const int2* d_table, int nblk) {
    if (nblk == 0) return 0;
    k_pass1_multi<<<nblk, FM_BLOCK, 0, st>>>(d_descs, d_table);
    LAUNCH_CHECK();
    return 0;
}

// =============================================================================================
// Record-step sums of caller-held device arrays without any allocation (fm_macros_sums_noalloc).
// The partial sums live in a file-scope device array; each device's copy is found once with
// hipGetSymbolAddress and its address is what the kernels receive.
#define FM_NOALLOC_MAX_NP (1 << 24)
#define FM_NOALLOC_BLOCKS ((FM_NOALLOC_MAX_NP + FM_BLOCK - 1) / FM_BLOCK)
static __device__ __align__(256) double scratch[FM_NOALLOC_BLOCKS * NRED];

namespace {
// the sums of k_macros_partial for (3,np) arrays in molecule order; a (leap-frog) shifts v by
// half a step, m = per-molecule masses (null: 1)
__global__ __launch_bounds__(FM_BLOCK) void k_macros_partial_aos(const double* v, const double* a, double dt,
                                                                 const double* pe_lj, const double* pe_poly,
                                                                 const double* vir, const double* mass, int np,
                                                                 double* part) {
    __shared__ double red[NRED][FM_BLOCK / 64];
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    double s[NRED] = {0, 0, 0, 0, 0, 0, 0, -1.0e300};
    if (i < np) {
        const double m = mass ? mass[i] : 1.0;
        const double pl = pe_lj[i], pp = pe_poly ? pe_poly[i] : 0.0;
        s[0] = pl;
        s[1] = pp;
        s[2] = pl + pp;
        s[3] = vir[i];
        double vx = v[3 * (size_t)i], vy = v[3 * (size_t)i + 1], vz = v[3 * (size_t)i + 2];
        if (a) {
            vx = vx + 0.5 * a[3 * (size_t)i] * dt;
            vy = vy + 0.5 * a[3 * (size_t)i + 1] * dt;
            vz = vz + 0.5 * a[3 * (size_t)i + 2] * dt;
        }
        s[4] = (m * (vx * vx) + m * (vy * vy)) + m * (vz * vz);
        s[5] = (m * vx + m * vy) + m * vz;
        s[6] = m;
        s[7] = pl + pp;
    }
    for (int q = 0; q < NRED; ++q) {
        double x = s[q];
        for (int off = 32; off > 0; off >>= 1) {
            const double o = __shfl_down(x, off, 64);
            x = q == 7 ? fmax(x, o) : x + o;
        }
        if ((threadIdx.x & 63) == 0) red[q][threadIdx.x >> 6] = x;
    }
    __syncthreads();
    if (threadIdx.x < NRED) {
        const int q = threadIdx.x;
        double x = red[q][0];
        for (int w = 1; w < FM_BLOCK / 64; ++w) x = q == 7 ? fmax(x, red[q][w]) : x + red[q][w];
        part[(size_t)blockIdx.x * NRED + q] = x;
    }
}
}  // namespace

// device address of `scratch` per device, looked up at each device's first call
static std::mutex g_scratch_mu;
static double* g_scratch_ptr[64] = {nullptr};

extern "C" int fm_macros_sums_noalloc(int32_t np, const double* v, const double* a, double delta_t,
                                      const double* potenergymol_LJ, const double* potenergymol_POLY,
                                      const double* virialmol, const double* mass, double* sums, void* stream) {
    if (np < 1 || np > FM_NOALLOC_MAX_NP)
        return fm_set_error(FM_EINVAL, "fm_macros_sums_noalloc: np %d outside 1..%d (the size of its static scratch)",
                            np, FM_NOALLOC_MAX_NP);
    if (!v || !potenergymol_LJ || !virialmol || !sums) return fm_set_error(FM_EINVAL, "fm_macros_sums_noalloc: null array");
    int dev = -1;
    if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= 64)
        return fm_set_error(FM_EHIP, "fm_macros_sums_noalloc: no current device");
    double* ptr;
    {
        std::lock_guard<std::mutex> lock(g_scratch_mu);
        if (!g_scratch_ptr[dev]) {
            void* p = nullptr;
            const hipError_t e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
            if (e != hipSuccess || !p)
                return fm_set_error(FM_EHIP, "hipGetSymbolAddress(scratch): %s", hipGetErrorString(e));
            g_scratch_ptr[dev] = (double*)p;
        }
        ptr = g_scratch_ptr[dev];
    }
    const hipStream_t st = (hipStream_t)stream;
    const int nb = (np + FM_BLOCK - 1) / FM_BLOCK;
    k_macros_partial_aos<<<nb, FM_BLOCK, 0, st>>>(v, a, delta_t, potenergymol_LJ, potenergymol_POLY, virialmol, mass,
                                                 np, ptr);
    k_macros_final<<<1, 256, 0, st>>>(ptr, nb, sums);
    LAUNCH_CHECK();
    return 0;
}
