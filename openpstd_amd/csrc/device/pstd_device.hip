// MI355X (gfx950) device solver for openPSTD's PSTD update loop.
//
// Implements the pstd_ctx_* C ABI of include/openpstd_amd.h: the GPU solver
// slot of openPSTD (GPUSingleThreadSolver / GPUMultiThreadSolver,
// kernel/Solver.cpp:153-160).
//
// State per domain lives in four arenas with identical layout (fields vx, vy,
// px, py at per-domain offsets):
//   TN  - values at t_n after PML attenuation (openPSTD's previous_values)
//   S0, S1 - raw outputs of the RK stages (ping-pong)
//   P0I - p0 (px slot) and its transpose (py slot): an explicit p0 (initial
//         state / host-written p0), and with `p0_pass` every stage's p0
// vx and px, which only X lines derive and update, are stored row-major; vy and
// py, which only Y lines do, column-major (transposed).  Every line of both
// directions is then contiguous in the field it derives, in t_n and in its
// output; only p0 = px + py (kernel/Solver.cpp:114-116) brings the two layouts
// together.  Large scenes form it in a pass of its own after every stage
// (p0_pass_kernel, both layouts); small ones, where a further launch costs more
// than it saves, add the other layout's field on the fly, strided.  The first
// stage of a step reads p0 from the raw stage-5 outputs of the previous step,
// which is openPSTD's p0 left stale by the PML attenuation (kernel/Solver.cpp:85).
//
// One RK stage = one launch of the fused line kernel: for each line of each
// segment it gathers the windowed line (spatderp3, kernel/core/
// kernel_functions.cpp:191-307), applies the spectral derivative with two
// complex FFTs in LDS (two real lines per complex transform), and writes the
// stage update of Solver::update_field_values (kernel/Solver.cpp:174-181).  The
// last stage also writes TN = output * PML factor (Domain::apply_pml_matrices,
// kernel/core/Domain.cpp:716-725).
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <complex>
#include <condition_variable>
#include <cstdio>
#include <cstring>
#include <map>
#include <mutex>
#include <string>
#include <tuple>
#include <type_traits>
#include <vector>

#include "../../../include/openpstd_amd.h"
#include "../host/plan_tables.h"
#include "fft_line.h"

using namespace pstdamd::dev;

// Scratch of the allocation-free advance (pstd_ctx_advance_static): the
// GEMM form's per-scene maxima, 2 classes x kStaticScenes scenes (8 KiB), one copy per device (each device has its own address, resolved
// with hipGetSymbolAddress), shared by every call on that device.
constexpr int kStaticScenes = 1024;
static __device__ __align__(256) unsigned scratch[2 * kStaticScenes];

namespace {

constexpr int kPassChunk = 2048;    // elements per passthrough tile
constexpr int kMaxDomainFloats = 1 << 29;  // one domain block (4 fields) per buffer resource

// A domain's four fields (vx, px row-major, vy, py column-major) form one block
// at the same offset of every arena (TN, S0, S1, P0I and the PML factors).
struct DomainDev {
    int nx, ny;
    long long base;                 // element offset of the block in an arena
    int size;                       // elements of the block
    int f_vx, f_vy, f_px, f_py;     // field offsets within the block
    float rho;
    int is_pml;
};

// One workgroup of a stage launch: `count` lines from line0 on of a line segment
// of a domain (Domain::calc, kernel/core/Domain.cpp:149-370), with everything the
// workgroup needs in one scalar-loadable record.  Caches are cold when a launch
// begins, and a small scene's stage is a chain of memory latencies: a record per
// workgroup is one of them, a reference to a record shared by the segment's tiles
// two (100 x 50 room 6.0 against 5.8 us per stage, three rooms of 333 000 cells 12.1
// / 11.5, 12 scenes of 64..600 a side 95.2 / 93.6, 16 sources of 512 x 1024 twice 350 /
// 351 with the launch arguments' first words in registers, kernel arguments below).
//  kind 0: derivative lines: gather, derivative, update.
//  kind 1: passthrough: a field that no segment updates (rigid domains,
//          directions openPSTD skips); lines are elements.
//  kind 2: receiver sampling (first stage of a step).
//  kind 3: the segment addressing of a GEMM-form tile (GemmTile::t).
// Memory is addressed through buffer resources over one domain block (base
// `*_dom`, `*_size` elements): value (line, pos) of a source field is element
// a + line*ls + pos of the block; where p0 = px + py is formed on the fly, plus
// element b + line + pos*bp (the field of the other layout).  Offsets past the
// block read 0 and drop stores, which is how absent neighbours, the zero padding
// and partial tiles are expressed.
struct TileDesc {
    int kind;
    int F;
    int line0, count;
    int wlen, n_main, n_out, vel, dir;
    int h_off, tw_off, win_off;
    long long m_dom, s1_dom, s2_dom;
    int m_size, s1_size, s2_size;
    int m_a, m_b, m_ls, m_bp;
    int s1_a, s1_b, s1_ls, s1_bp, s1_line, s1_len;  // s1_len < 0: no neighbour (zeros)
    int s2_a, s2_b, s2_ls, s2_bp, s2_line, s2_len;
    float c_s1, c_m1, c_s2, c_m2;
    int o_f, o_ls;        // output field (vx, px, vy or py) within the main block
    float coef;           // 1/rho (velocity update) or rho*c1^2 (pressure update)
    int is_pml;
    int scene;            // scene of the batch (per-scene maxima of the GEMM form's scaling)
    int slot;             // GEMM form: of the first wavefront's maximum (track_max)
};
static_assert(sizeof(TileDesc) == 192, "three 64-byte lines");

struct ReceiverCell {
    long long px, py;  // arena element offsets of the cell's px0 and py0; px < 0: spectral receiver
};

struct StageArgs {
    const float2 *ctab;
    const float *ftab;
    const float *p0;   // p0 arena: P0I, or (p0_two) a stage arena whose px + py it is
    int p0_two;
    const float *vsrc; // current vx / vy
    float *tn;
    float *out;
    const float *pml;  // PML factor arena (same layout); 1 for non-PML domains
    float s;           // dt * alpha_k
    int last;          // last RK stage: also write tn = out * pml
    // receiver sampling of the previous step (first stage of a step): p0 = px + py
    // of the previous step's raw stage-5 output (kernel/Solver.cpp:86-91)
    const ReceiverCell *cells;
    int nrec;
    float *samples;    // samples[slot * nrec + r], slot < 0: no sampling in this launch
    int slot;
    // GEMM form (wmax == nullptr otherwise): the largest |value| each wavefront
    // wrote, and what the previous stage's came to per scene (max_reduce)
    float *wmax;
    const unsigned *umax;
    const void *dmat;  // derivative matrices (2-byte elements)
    int f8;            // longest lines with 8 values per thread (pstd_ctx::values)
};

// ------------------------------------------------------------- device code

typedef __amdgpu_buffer_rsrc_t Rsrc;
constexpr int kOOB = (int)0x80000000u;  // byte offset past every block: loads 0, drops stores

__device__ __forceinline__ Rsrc block_rsrc(const float *arena, long long dom, int size) {
    // raw buffer (stride 0) over `size` floats; word 3 as for every gfx9 raw buffer
    return __builtin_amdgcn_make_buffer_rsrc((void *)(arena + dom), (short)0, size * 4, 0x00020000);
}
// per-lane byte offset, and a uniform one that the block's bounds need not know
// (kLead floats of padding cover what it adds)
__device__ __forceinline__ float bload(Rsrc r, int off_bytes, int uniform = 0) {
    return __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(r, off_bytes, uniform, 0));
}
__device__ __forceinline__ void bstore(Rsrc r, int off_bytes, int uniform, float v) {
    __builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(unsigned, v), r, off_bytes, uniform, 0);
}
// A block with the 32 floats before it: positions a halo length before a line's
// first value have non-negative offsets (they read the values before the line,
// which every user replaces).  kLead floats precede the first block of an arena and
// follow the last one: a row of threads that begins inside a line may end up to
// 512 floats past it.
constexpr int kLead = 576, kShift = 32;
__device__ __forceinline__ Rsrc lead_rsrc(const float *arena, long long dom, int size) {
    return block_rsrc(arena, dom - kShift, size + kShift);
}
// A uniform value anew: what is computed or loaded from it is computed again
// rather than kept in registers.
__device__ __forceinline__ int again(int x) {
    asm volatile("" : "+v"(x));
    return __builtin_amdgcn_readfirstlane(x);
}
// two adjacent floats (4-byte aligned suffices for buffer accesses)
__device__ __forceinline__ float2 bload2(Rsrc r, int off_bytes) {
    return __builtin_bit_cast(float2, __builtin_amdgcn_raw_buffer_load_b64(r, off_bytes, 0, 0));
}

// The GEMM form scales its operands by the largest |value| of a scene's pressure
// (class 0) and velocity fields (class 1) after a stage.  Every wavefront stores
// the largest value it wrote into a slot of its own, and max_reduce brings the
// slots of a scene and class, which lie together, to umax[scene * 2 + class]
// (float bits).  (With atomic maxima into the scene's word the strips' tiles of 16
// scenes took 200 us in the GEMM form, against 100 without them.)
__device__ __forceinline__ void track_max(const StageArgs &a, int slot, float m) {
    if (!a.wmax) return;
#pragma unroll
    for (int o = 32; o >= 1; o >>= 1) m = fmaxf(m, __shfl_xor(m, o));
    if ((threadIdx.x & 63) == 0) a.wmax[slot + (threadIdx.x >> 6)] = m;
}

// The derivative's input arena.  (Chosen between values: a conditional of two
// struct members is one of their addresses, and keeps the struct in memory.)
__device__ __forceinline__ const float *pick(bool c, const float *x, const float *y) { return c ? x : y; }
__device__ __forceinline__ const float *source(const StageArgs &a, int vel) { return pick(vel != 0, a.vsrc, a.p0); }

// Descriptors are read through the constant address space: by scalar loads,
// wherever they are needed, also after stores.
typedef const __attribute__((address_space(4))) TileDesc *Seg;

// A derivative tile: F-point lines, T = F/V threads per line pair; thread (p, t)
// holds the values at positions t + m*T (m = 0..V-1) of lines 2p and 2p+1 as one
// complex sequence (V: fft_line.h).  The code before and after the transforms is
// shared by all F of one V (few copies keep the kernel inside the instruction
// cache), the transforms are specialised.
//
// gather: the windowed lines (spatderp3, kernel/core/kernel_functions.cpp:210-216
// pressure, :263-269 velocity) [dom1 | main | dom3 | 0], where dom1[j] =
// (side1[tail + j] * c_s1 + main[reflected] * c_m1) * window[j] and dom3 likewise.
// Main values are loaded where they are transformed, a wavefront along the line;
// positions outside the main piece read whatever lies beside the line and are
// replaced.  The 2w halo values are formed where they are transformed too: each
// of T >= 32 threads holds at most one of a side's w <= 32 positions (the 16
// threads of a 128-point pair, SHORT: two), and loads its side value, its
// reflected main value (the line itself, a cache hit) and its window coefficient
// directly.  All loads are issued before the first
// wait, and no LDS staging or barrier precedes the transform.
//
// With p0_two, p0 = px + py is formed on the fly.  Across the other layout a line
// is strided and the tile's lines are adjacent: the workgroup reads position
// after position, all of the tile's lines at once (32 bytes of 8 lines; a thread
// reading its own pair touches 8 bytes per cache sector, which made up a quarter
// of the time of a 333 000-cell scene), and turns them through the pairs' LDS
// buffers.
struct Tile {
    int T, logT, p, t;  // threads per pair; this thread's pair and position
    int pitch;          // of the pairs' LDS buffers
    int line, count;    // first line of the pair; lines of the pair inside the tile (0, 1, 2 or more)
    // thread rows that positions [0, n) reach into
    __device__ __forceinline__ int rows(int n) const { return (n + T - 1) >> logT; }
};

// A line fills more than half of its F points (F is the next power of two), less
// 32 of the halo: rows of threads that lie inside it for sure.
template <int V, bool SHORT>
constexpr int kFull = SHORT ? 2 : V / 2 - 1;

template <int V, int NT, bool SHORT>
__device__ __forceinline__ void gather(const StageArgs &a, Seg td, const Tile &x, float2 *lds, float2 (&v)[V]) {
    constexpr int NI = SHORT ? 2 : 1, FULL = kFull<V, SHORT>;
    const int w = td->wlen, nm = td->n_main, vel = td->vel, end = w + nm, T = x.T, t = x.t, T4 = T * 4;
    __builtin_assume(w > 0 && w <= 32);
    const int rows = x.rows(end);
    const float *A = source(a, vel);
    const Rsrc rm = lead_rsrc(A, td->m_dom, td->m_size);
    const bool ok0 = x.count > 0, ok1 = x.count > 1;
    const int ls4 = td->m_ls * 4;
    const int row = (td->m_a + x.line * td->m_ls + kShift) * 4;  // the line's first main value
    const int off0 = ok0 ? row + (t - w) * 4 : kOOB, off1 = ok1 ? row + ls4 + (t - w) * 4 : kOOB;
#pragma unroll
    for (int m = 0; m < V; ++m) {
        v[m] = make_float2(0.f, 0.f);
        if (m < FULL || m < rows) v[m] = make_float2(bload(rm, off0, m * T4), bload(rm, off1, m * T4));
    }
    // halo item c of this thread: left position t + cT, right offset j0 + cT
    const int col = end & (T - 1), j0 = (t - col) & (T - 1);
    const Rsrc r1 = block_rsrc(A, td->s1_dom, td->s1_size), r2 = block_rsrc(A, td->s2_dom, td->s2_size);
    const int s1 = td->s1_len - w - vel, l1 = x.line + td->s1_line, l2 = x.line + td->s2_line;
    const bool has1 = ok0 && td->s1_len >= 0, has2 = ok0 && td->s2_len >= 0;
    float2 ls[NI], rs[NI], lr[NI], rr[NI];
    float lw[NI], rw[NI];
#pragma unroll
    for (int c = 0; c < NI; ++c) {
        const int i = t + c * T, j = j0 + c * T;
        const bool li = i < w, ri = j < w;
        lw[c] = a.ftab[td->win_off + (li ? i : 0)];
        rw[c] = a.ftab[td->win_off + w + 1 + (ri ? j : 0)];
        const int o1 = li && has1 ? (td->s1_a + l1 * td->s1_ls + s1 + i) * 4 : kOOB;
        const int o2 = ri && has2 ? (td->s2_a + l2 * td->s2_ls + j + vel) * 4 : kOOB;
        const int ol = li && ok0 ? row + (w - 1 + vel - i) * 4 : kOOB, orr = ri && ok0 ? row + (nm - 1 - vel - j) * 4 : kOOB;
        ls[c] = make_float2(bload(r1, o1), bload(r1, ok1 ? o1 + td->s1_ls * 4 : kOOB));
        rs[c] = make_float2(bload(r2, o2), bload(r2, ok1 ? o2 + td->s2_ls * 4 : kOOB));
        lr[c] = make_float2(bload(rm, ol), bload(rm, ok1 ? ol + ls4 : kOOB));
        rr[c] = make_float2(bload(rm, orr), bload(rm, ok1 ? orr + ls4 : kOOB));
    }
    if (!vel && a.p0_two) {
        const unsigned keep = ok1 ? ~0u : 0u;  // a lone last line's partner stays zero
        auto add = [&](float2 &u, float2 y) __attribute__((always_inline)) {
            u.x += y.x;
            u.y += __uint_as_float(__float_as_uint(y.y) & keep);
        };
        const int logP = __builtin_ctz(NT) - x.logT, P = 1 << logP, bp4 = td->m_bp * 4;
        // item (pair, position) = (i mod P, i / P), i = thread + k NT
        const int pair = threadIdx.x & (P - 1), pos = threadIdx.x >> logP, step = NT >> logP;
        const int lines = x.count + 2 * x.p - 2 * pair, b0 = (td->m_b + x.line - 2 * x.p + 2 * pair + kShift) * 4;
        float2 b[V];
#pragma unroll
        for (int k = 0; k < V; ++k)
            if (k == 0 || k * step < nm)
                b[k] = bload2(rm, lines > 0 && pos + k * step < nm ? b0 + (pos + k * step) * bp4 : kOOB);
        float2 y1[NI], y2[NI];
#pragma unroll
        for (int c = 0; c < NI; ++c) {
            y1[c] = bload2(r1, t + c * T < w && has1 ? (td->s1_b + l1 + (s1 + t + c * T) * td->s1_bp) * 4 : kOOB);
            y2[c] = bload2(r2, j0 + c * T < w && has2 ? (td->s2_b + l2 + (j0 + c * T) * td->s2_bp) * 4 : kOOB);
        }
        float2 *to = lds + pair * x.pitch;
        const int nm2 = again(nm);
#pragma unroll
        for (int k = 0; k < V; ++k)
            if ((k == 0 || k * step < nm2) && pos + k * step < nm) to[lds_slot(w + pos + k * step)] = b[k];
        __syncthreads();
        const float2 *buf = lds + x.p * x.pitch;
        const int rows2 = again(rows);
#pragma unroll
        for (int m = 0; m < V; ++m)
            if (m < FULL || m < rows2) add(v[m], buf[lds_slot(t + m * T)]);
#pragma unroll
        for (int c = 0; c < NI; ++c) {
            const int i = t + c * T, j = j0 + c * T;
            add(ls[c], y1[c]);
            add(rs[c], y2[c]);
            if (i < w) add(lr[c], buf[lds_slot(2 * w - 1 - i)]);
            if (j < w) add(rr[c], buf[lds_slot(end - 1 - j)]);
        }
    }
    float2 hr[NI];
#pragma unroll
    for (int c = 0; c < NI; ++c) {
        const float2 hl = make_float2(__builtin_fmaf(ls[c].x, td->c_s1, lr[c].x * td->c_m1) * lw[c],
                                      __builtin_fmaf(ls[c].y, td->c_s1, lr[c].y * td->c_m1) * lw[c]);
        hr[c] = make_float2(__builtin_fmaf(rs[c].x, td->c_s2, rr[c].x * td->c_m2) * rw[c],
                            __builtin_fmaf(rs[c].y, td->c_s2, rr[c].y * td->c_m2) * rw[c]);
        if (j0 + c * T >= w) hr[c] = make_float2(0.f, 0.f);
        if (t + c * T < w) v[c] = hl;
    }
    // thread row lo + c holds right item c from column `col` on, item c - 1 before it
    const int lo = again(end >> x.logT);
    const bool at_end = t >= col;
#pragma unroll
    for (int m = FULL; m < V; ++m)
#pragma unroll
        for (int c = 0; c <= NI; ++c)
            if (m == lo + c) {
                const float2 from = c < NI ? hr[c < NI ? c : 0] : make_float2(0.f, 0.f);
                v[m] = at_end ? from : c == 0 ? v[m] : hr[c > 0 ? c - 1 : 0];
            }
}

// Solver::update_field_values (kernel/Solver.cpp:174-181): out = t_n - s*L*coef,
// the last stage also t_n = out * PML factor.
struct OutAddr {
    int off0, off1, end, rows;
    __device__ __forceinline__ OutAddr(Seg td, const Tile &x) {
        const int off = (td->o_f + x.line * td->o_ls + x.t - td->wlen + kShift) * 4;
        off0 = x.count > 0 ? off : kOOB;
        off1 = x.count > 1 ? off + td->o_ls * 4 : kOOB;
        end = td->wlen + td->n_out;
        rows = x.rows(end);
    }
};

template <int V, bool SHORT>
__device__ __forceinline__ void update_loads(const StageArgs &a, Seg td, const Tile &x, float2 (&tn)[V]) {
    const OutAddr o(td, x);
    const Rsrc rt = lead_rsrc(a.tn, td->m_dom, td->m_size);
#pragma unroll
    for (int m = 0; m < V; ++m)
        if (m < kFull<V, SHORT> || m < o.rows)
            tn[m] = make_float2(bload(rt, o.off0, m * x.T * 4), bload(rt, o.off1, m * x.T * 4));
}

// v: the conjugate of the derivative (two real lines: the second one negated)
template <int V, bool SHORT>
__device__ __forceinline__ void update_stores(const StageArgs &a, Seg td, const Tile &x, float2 (&v)[V],
                                              const float2 (&tn)[V], int slot) {
    const OutAddr o(td, x);
    const int w = td->wlen, T4 = x.T * 4;
    const float sc = a.s * td->coef;
    const Rsrc ro = lead_rsrc(a.out, td->m_dom, td->m_size);
    float mx = 0.f;
    // the first rows hold the left halo (w <= 32), rows from kFull on can leave the line
    auto inside = [&](int m) __attribute__((always_inline)) {
        const int pos = x.t + m * x.T;
        return (m > (SHORT ? 1 : 0) || pos >= w) && (m < kFull<V, SHORT> || pos < o.end);
    };
#pragma unroll
    for (int m = 0; m < V; ++m) {
        if ((m < kFull<V, SHORT> || m < o.rows) && inside(m)) {
            v[m] = make_float2(__builtin_fmaf(-sc, v[m].x, tn[m].x), __builtin_fmaf(sc, v[m].y, tn[m].y));
            bstore(ro, o.off0, m * T4, v[m].x);
            bstore(ro, o.off1, m * T4, v[m].y);
            mx = fmaxf(mx, fmaxf(fabsf(v[m].x), fabsf(v[m].y)));
        }
    }
    if (a.last) {
        const Rsrc rt = lead_rsrc(a.tn, td->m_dom, td->m_size);
        if (td->is_pml) {
            const Rsrc rp = lead_rsrc(a.pml, td->m_dom, td->m_size);
            // four rows of threads at a time: few registers
#pragma unroll
            for (int m0 = 0; m0 < V; m0 += 4) {
                if (m0 >= kFull<V, SHORT> && m0 >= o.rows) break;
                float2 pm[4];
#pragma unroll
                for (int m = 0; m < 4; ++m)
                    if (m0 + m < kFull<V, SHORT> || m0 + m < o.rows)
                        pm[m] = make_float2(bload(rp, o.off0, (m0 + m) * T4), bload(rp, o.off1, (m0 + m) * T4));
#pragma unroll
                for (int m = 0; m < 4; ++m) v[m0 + m] = make_float2(v[m0 + m].x * pm[m].x, v[m0 + m].y * pm[m].y);
            }
        }
#pragma unroll
        for (int m = 0; m < V; ++m) {
            if ((m < kFull<V, SHORT> || m < o.rows) && inside(m)) {
                bstore(rt, o.off0, m * T4, v[m].x);
                bstore(rt, o.off1, m * T4, v[m].y);
            }
        }
    }
    track_max(a, slot, mx);
}

// SHORT: F = 128; SPLIT: F = 8192 (fft_line.h's two sequences)
template <int V, int NT, bool SHORT, bool SPLIT>
__device__ __forceinline__ void derivative_tile(const StageArgs &a, Seg td, float2 *lds) {
    constexpr int kLogV = V == 16 ? 4 : 3;
    const int F = td->F, logT = 31 - kLogV - __builtin_clz(F);
    Tile x;
    x.logT = logT;
    x.T = 1 << logT;
    x.p = threadIdx.x >> logT;
    x.t = threadIdx.x & (x.T - 1);
    x.line = td->line0 + 2 * x.p;
    x.count = td->count - 2 * x.p;
    x.pitch = lds_pitch(F);
    float2 *buf = lds + x.p * x.pitch;
    // the tables through a buffer resource: one lane offset, the rest in scalar registers
    const Table tab{__builtin_amdgcn_make_buffer_rsrc((void *)a.ctab, (short)0, 0x7fffffff, 0x00020000)};
    const int t = x.t;
    // 8 values per thread leave the registers to load t_n and the filter with the
    // lines (two memory latencies less); with 16 they are loaded where they are used
    constexpr bool kTnEarly = V == 8;
    float2 v[V], tn[V], h[V];
    // pairs of the filter's values as the transforms leave them: m and m + 1, or
    // (8192) the even and the odd bin of value m
    auto filter_loads = [&]() __attribute__((always_inline)) {
        const int h_off = td->h_off * 8;
#pragma unroll
        for (int m = 0; m < V; m += 2) tab.pair(h[m], h[m + 1], t * 16, h_off + (m << (logT + 3)));
    };
    gather<V, NT, SHORT>(a, td, x, lds, v);
    if constexpr (kTnEarly) update_loads<V, SHORT>(a, td, x, tn);
    if constexpr (kTnEarly) filter_loads();
    if constexpr (SPLIT) split_first(v, t, tab, td->tw_off * 8);
    // forward transform; spectral derivative: the Hermitian filter, which carries
    // the 1/F of kernel/core/kernel_functions.cpp:243,306; conjugate; the forward
    // transform again (the conjugate of the inverse)
#pragma unroll 1
    for (int dir = 0; dir < 2; ++dir) {
        const int tw = again(td->tw_off * 8);
        int ti = t;
        asm volatile("" : "+v"(ti));  // LDS addresses per pass, not kept for all lengths across the loop
#define PSTD_FFT_CASE(FV)                                                                            \
    case FV:                                                                                         \
        if constexpr ((fft_values(FV) == V || (FV <= 2048 && V == 8)) && FV <= V * NT && (FV == 128) == SHORT && (FV == 8192) == SPLIT) \
            fft_run<FV, V>(v, ti, buf, tab, tw);                                                        \
        break;
        switch (F) {
            PSTD_FFT_CASE(128)
            PSTD_FFT_CASE(256)
            PSTD_FFT_CASE(512)
            PSTD_FFT_CASE(1024)
            PSTD_FFT_CASE(2048)
            PSTD_FFT_CASE(4096)
            PSTD_FFT_CASE(8192)
            default: break;
        }
#undef PSTD_FFT_CASE
        if (dir == 0) {
            if constexpr (!kTnEarly) filter_loads();
#pragma unroll
            for (int m = 0; m < V; ++m) {
                const float2 y = cmul(v[m], h[SPLIT ? 2 * (m & 7) + (m >> 3) : m]);
                v[m] = make_float2(y.x, -y.y);
            }
        }
    }
    if constexpr (SPLIT) split_last(v, t, tab, td->tw_off * 8);
    // the descriptor again: the gather's fields need not stay in scalar registers
    const Seg to = td + again(0);
    if constexpr (!kTnEarly) update_loads<V, SHORT>(a, to, x, tn);
    update_stores<V, SHORT>(a, to, x, v, tn, to->slot);
}

// One extra workgroup of a launch samples the receivers (p0 of the previous
// step, read from the arena the first stage reads it from).
__device__ void sample_receivers(const StageArgs &a) {
    if (a.slot < 0) return;
    for (int r = threadIdx.x; r < a.nrec; r += blockDim.x) {
        const ReceiverCell c = a.cells[r];
        if (c.px < 0) continue;  // spectral receiver
        a.samples[(size_t)a.slot * a.nrec + r] = a.p0_two ? a.p0[c.px] + a.p0[c.py] : a.p0[c.px];
    }
}

// Fields no segment updates keep their t_n value (openPSTD leaves their L at 0,
// kernel/Solver.cpp:174-181); the last stage applies the PML factor.  Each
// thread issues all of its loads before its stores.
template <int NT>
__device__ __forceinline__ void passthrough_tile(const StageArgs &a, Seg td) {
    constexpr int PER = kPassChunk / NT;
    const Rsrc rt = block_rsrc(a.tn, td->m_dom, td->m_size);
    const Rsrc rp = block_rsrc(a.pml, td->m_dom, td->m_size);
    const Rsrc ro = block_rsrc(a.out, td->m_dom, td->m_size);
    const bool use_pml = a.last && td->is_pml;
    float v[PER], f[PER];
    int off[PER];
#pragma unroll
    for (int k = 0; k < PER; ++k) {
        const int e = threadIdx.x + k * NT;
        off[k] = e < td->count ? (td->o_f + td->line0 + e) * 4 : kOOB;
        v[k] = bload(rt, off[k]);
        f[k] = use_pml ? bload(rp, off[k]) : 1.f;
    }
#pragma unroll
    for (int k = 0; k < PER; ++k) {
        bstore(ro, off[k], 0, v[k]);
        if (use_pml) bstore(rt, off[k], 0, v[k] * f[k]);
    }
    float mx = 0.f;
#pragma unroll
    for (int k = 0; k < PER; ++k) mx = fmaxf(mx, fabsf(v[k]));
    track_max(a, td->slot, mx);
}

// Workgroups are dispatched to the 8 XCDs round-robin (workgroup b runs on XCD
// b % 8) and every XCD has its own L2.  With `remap`, XCD x works through a
// contiguous run of the tile list instead of every 8th tile, so tiles of
// neighbouring lines (which share the cache lines of the other layout's field)
// share that L2.  A bijection of [0, n).
__device__ __forceinline__ int tile_index(int b, int n, int remap) {
    if (!remap) return b;
    constexpr int X = 8;
    const int x = b % X, l = b / X, q = n / X, r = n % X;
    return x * q + min(x, r) + l;
}

// One launch per RK stage covers every FFT-form line: NT = 128, 256 or 512
// threads, lines of F <= 16 NT, about 17 NT complex values of LDS.  Pairs of F <=
// 1024 are one wavefront's (or a part's) business whatever NT is; the block size
// decides how long the lines may be (8192-point ones take a 512-thread block),
// how many adjacent lines a tile has and how finely a small scene spreads over
// the CUs.  Bound by the VALU and the L1 together (16 sources of 512 x 1024 twice:
// VALU 63 % and L1 address units 67 % busy, 275 us of the 346 us stage, 200 of them
// also without the transforms, which is what its memory traffic takes; one launch
// of 8-value tiles, 568 us per stage, had each column access touch 8-16 bytes of a
// cache line).
constexpr size_t stage_lds(int nt) { return (size_t)(16 * nt / 256) * lds_pitch(256) * sizeof(float2); }

// At most 128 VGPRs: four wavefronts per SIMD, what the LDS allows too.  What finds
// the record comes first: the build has the first eight words of kernel arguments
// in scalar registers when a wavefront starts, which saves another latency before
// the record's (100 x 50 room 6.05 -> 5.94 us per stage, 1024^2 31.0 -> 30.7).
template <int NT>
__global__ void __launch_bounds__(NT) __attribute__((amdgpu_waves_per_eu(4)))
stage_fft_kernel(const TileDesc *tiles, int ntiles, int remap, StageArgs a) {
    extern __shared__ float2 lds_dyn[];
    const Seg td = (Seg)tiles + tile_index(blockIdx.x, ntiles, remap);
    // one word of each of the record's 64-byte lines: fetched together, not one
    // after the other as the code comes to need them
    asm volatile("" ::"s"(td->kind), "s"(td->m_size), "s"(td->is_pml));
    switch (td->kind) {
        case 0:
            if (td->F == 128) derivative_tile<8, NT, true, false>(a, td, lds_dyn);
            else if (td->F <= a.f8) derivative_tile<8, NT, false, false>(a, td, lds_dyn);
            else if (NT == 512 && td->F == 8192) derivative_tile<16, NT, false, NT == 512>(a, td, lds_dyn);
            else derivative_tile<16, NT, false, false>(a, td, lds_dyn);
            break;
        case 1: passthrough_tile<NT>(a, td); break;
        case 2: sample_receivers(a); break;
        default: break;
    }
}

__global__ void receiver_kernel(const float *__restrict__ arena, const ReceiverCell *__restrict__ cells, int nrec,
                                float *__restrict__ samples, int slot) {
    // p0 = px0 + py0 (kernel/Solver.cpp:114-116)
    for (int r = threadIdx.x; r < nrec; r += blockDim.x) {
        const ReceiverCell c = cells[r];
        if (c.px < 0) continue;  // spectral receiver: sampled by the interpolation passes
        samples[(size_t)slot * nrec + r] = arena[c.px] + arena[c.py];
    }
}

// Spectral-interpolation receivers (Receiver::compute_with_si,
// kernel/core/Receiver.cpp:85-121), two passes after each step.  The
// fractional shift of one pressure line, read at one output, is a fixed linear
// function of the line's K = n + 2w raw values [side-1 tail | main | side-2
// head] (p0 = px + py): the row of the line operator (shift filter composed
// with the window and reflections) built in double on the host.  Pass 1: one
// wave per line of the domains the receiver's Y line reads, the dot product
// of its values with its X-shift row, into the receiver's column buffer
// [side-1 tail | domain rows | side-2 head].  Pass 2: one wave per receiver,
// the column buffer against the Y-shift row of the receiver's row.
struct SILine {
    long long m_px, m_py;    // arena offsets of the line's first main value in px0 (or p0), py0
    long long s1_px, s1_py;  // first of the w side-1 tail values; -1: no neighbour (zeros)
    long long s2_px, s2_py;  // first of the w side-2 head values; -1: zeros
    int m_ld, s1_ld, s2_ld;  // py0 is column-major: elements from one value to the next
    int n_main, w;
    int coef;                // first of the line's K weights in the weight table
    int dst;                 // element of the column buffer
};

struct SIPoint {
    int coef, K;             // Y-shift weights of the receiver's row
    int col;                 // first element of the receiver's column buffer
    int rec;                 // receiver index (sample position)
};

__device__ __forceinline__ float wave_sum(float v) {
    for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o);
    return v;
}

__global__ __launch_bounds__(256) void si_line_kernel(const float *__restrict__ arena, const SILine *__restrict__ lines,
                                                      int nlines, int two, const float *__restrict__ coef,
                                                      float *__restrict__ col) {
    // two: p0 = px + py of a stage arena; otherwise the arena holds p0 in the px slots
    // jobs are sorted by line: the receivers reading one line are neighbours,
    // and XCD-contiguous runs of blocks put them on one XCD (its L2 serves the
    // line after the first read)
    const int lane = threadIdx.x & 63, j = tile_index(blockIdx.x, gridDim.x, 1) * 4 + (threadIdx.x >> 6);
    if (j >= nlines) return;
    const SILine L = lines[j];
    const int w = L.w, n = L.n_main, K = n + 2 * w;
    const float *cf = coef + L.coef;
    float acc = 0.f;
    for (int k = lane; k < K; k += 64) {
        float u = 0.f;
        if (k < w) {
            if (L.s1_px >= 0) {
                u = arena[L.s1_px + k];
                if (two) u += arena[L.s1_py + (long long)k * L.s1_ld];
            }
        } else if (k < w + n) {
            u = arena[L.m_px + (k - w)];
            if (two) u += arena[L.m_py + (long long)(k - w) * L.m_ld];
        } else if (L.s2_px >= 0) {
            u = arena[L.s2_px + (k - w - n)];
            if (two) u += arena[L.s2_py + (long long)(k - w - n) * L.s2_ld];
        }
        acc = fmaf(cf[k], u, acc);
    }
    acc = wave_sum(acc);
    if (lane == 0) col[L.dst] = acc;
}

__global__ __launch_bounds__(64) void si_point_kernel(const float *__restrict__ col, const SIPoint *__restrict__ pts,
                                                      const float *__restrict__ coef, float *__restrict__ samples,
                                                      int nrec, int slot) {
    const SIPoint P = pts[blockIdx.x];
    float acc = 0.f;
    for (int k = threadIdx.x; k < P.K; k += 64) acc = fmaf(coef[P.coef + k], col[P.col + k], acc);
    acc = wave_sum(acc);
    if (threadIdx.x == 0) samples[(size_t)slot * nrec + P.rec] = acc;
}

// One 64 x 64-cell piece of a domain for the passes between the two layouts.
struct P0Tile {
    long long px, py;  // arena offsets of the domain's px (row-major) and py (column-major) fields
    int nx, ny, x0, y0;
};
constexpr int kP0Side = 64;

// p0 = px0 + py0 (kernel/Solver.cpp:114-116) of every cell in both layouts: the
// px slots of `p0` row-major, the py slots column-major.  Bound by HBM (16
// bytes per cell); a tile of 64 x 64 is turned through LDS so that all four
// accesses run along 256-byte pieces of a row (pitch 65: the turned read is
// free of bank conflicts).
// `py_src` false: p0's px slots hold p0 already, only its transpose is written.
// In the GEMM form the first blocks bring the stage's maxima together, one per
// scene and class (`mx`).
struct MaxArgs {
    const float *wmax;
    const int2 *first;  // group g's slots: first[g].x .. first[g + 1].x of the FFT-form tiles, .y of the GEMM tiles
    unsigned *umax;
    int n;              // groups (0: none)
};
__device__ void max_reduce(const MaxArgs &x, int g) {
    __shared__ float part[4];
    const int2 b = x.first[g], e = x.first[g + 1];
    float m = 0.f;
    for (int i = b.x + threadIdx.x; i < e.x; i += 256) m = fmaxf(m, x.wmax[i]);
    for (int i = b.y + threadIdx.x; i < e.y; i += 256) m = fmaxf(m, x.wmax[i]);
#pragma unroll
    for (int o = 32; o >= 1; o >>= 1) m = fmaxf(m, __shfl_xor(m, o));
    if ((threadIdx.x & 63) == 0) part[threadIdx.x >> 6] = m;
    __syncthreads();
    if (threadIdx.x == 0) x.umax[g] = __float_as_uint(fmaxf(fmaxf(part[0], part[1]), fmaxf(part[2], part[3])));
}

__global__ void __launch_bounds__(256) p0_pass_kernel(const float *__restrict__ src, float *__restrict__ p0,
                                                      const P0Tile *__restrict__ tiles, int py_src, MaxArgs mx) {
    __shared__ float turn[kP0Side][kP0Side + 1];
    if ((int)blockIdx.x < mx.n) {
        max_reduce(mx, blockIdx.x);
        return;
    }
    const P0Tile T = tiles[blockIdx.x - mx.n];
    const int lane = threadIdx.x & 63, row0 = threadIdx.x >> 6;
    const int w = min(kP0Side, T.nx - T.x0), h = min(kP0Side, T.ny - T.y0);
    float v[kP0Side / 4];
    // row-major side: rows y0 + r, columns x0 + lane
    const float *row = (py_src ? src : p0) + T.px + (long long)T.y0 * T.nx + T.x0 + lane;
#pragma unroll
    for (int i = 0; i < kP0Side / 4; ++i) {
        const int r = row0 + 4 * i;
        v[i] = r < h && lane < w ? row[(long long)r * T.nx] : 0.f;
    }
    if (py_src) {
        // column-major side: columns x0 + c, rows y0 + lane
        const float *col = src + T.py + (long long)T.x0 * T.ny + T.y0 + lane;
#pragma unroll
        for (int i = 0; i < kP0Side / 4; ++i) {
            const int c = row0 + 4 * i;
            turn[lane][c] = c < w && lane < h ? col[(long long)c * T.ny] : 0.f;
        }
        __syncthreads();
        float *out = p0 + T.px + (long long)T.y0 * T.nx + T.x0 + lane;
#pragma unroll
        for (int i = 0; i < kP0Side / 4; ++i) {
            const int r = row0 + 4 * i;
            v[i] += turn[r][lane];
            if (r < h && lane < w) out[(long long)r * T.nx] = v[i];
        }
        // every thread rewrites the slots that it alone has read
    }
#pragma unroll
    for (int i = 0; i < kP0Side / 4; ++i) turn[row0 + 4 * i][lane] = v[i];
    __syncthreads();
    float *out = p0 + T.py + (long long)T.x0 * T.ny + T.y0 + lane;
#pragma unroll
    for (int i = 0; i < kP0Side / 4; ++i) {
        const int c = row0 + 4 * i;
        if (c < w && lane < h) out[(long long)c * T.ny] = turn[lane][c];
    }
}

// Fields between the host's layout and the device's: host fields are row-major, vy
// and py are stored column-major.  dst (cols x rows) = transpose of src (rows x
// cols), for up to N fields in one launch (a launch costs what turning a field of a
// small scene does several times over).
struct TurnField {
    const float *src;
    float *dst;
    int rows, cols;
    unsigned first;  // the field's first workgroup
};
template <int N>
struct TurnFields {
    TurnField f[N];
    int n;
};
template <int N>
__global__ void __launch_bounds__(256) turn_kernel(TurnFields<N> fields) {
    __shared__ float turn[kP0Side][kP0Side + 1];
    int k = 0;
    while (k + 1 < fields.n && blockIdx.x >= fields.f[k + 1].first) ++k;
    const float *src = fields.f[k].src;
    float *dst = fields.f[k].dst;
    const int rows = fields.f[k].rows, cols = fields.f[k].cols, across = (cols + kP0Side - 1) / kP0Side;
    const int b = blockIdx.x - fields.f[k].first;
    const int lane = threadIdx.x & 63, row0 = threadIdx.x >> 6;
    const int x0 = b % across * kP0Side, y0 = b / across * kP0Side;
#pragma unroll
    for (int i = 0; i < kP0Side / 4; ++i) {
        const int r = y0 + row0 + 4 * i;
        if (r < rows && x0 + lane < cols) turn[row0 + 4 * i][lane] = src[(long long)r * cols + x0 + lane];
    }
    __syncthreads();
#pragma unroll
    for (int i = 0; i < kP0Side / 4; ++i) {
        const int c = x0 + row0 + 4 * i;
        if (c < cols && y0 + lane < rows) dst[(long long)c * rows + y0 + lane] = turn[lane][row0 + 4 * i];
    }
}

// A column-major field of one domain, row-major (py and vy), or p0 = px + py of it
// (px: row-major), for the caller of a short read: `out` is pinned host memory.  An
// element per thread: the read waits for one access to memory and one to the host,
// where turn_kernel's pieces do 16 after each other (a py of 100 x 50 cells in 13.4
// us against 15.7, of 255 x 250 in 22.0 against 25.1).
__global__ void __launch_bounds__(256) rows_kernel(const float *__restrict__ px, const float *__restrict__ py,
                                                   float *__restrict__ out, int nx, int rows) {
    const int i = blockIdx.x * 256 + threadIdx.x;
    if (i >= nx * rows) return;
    const float y = py[i % nx * rows + i / nx];
    out[i] = px ? px[i] + y : y;
}

// ------------------------------------------------------------- GEMM form
// The windowed line derivative of a segment is a fixed linear operator: the
// dense matrix D (n_out x K) of plan_tables.h, applied to the raw line
// u = [side1 tail | main | side2 head] (K values).  One workgroup (4 waves,
// two per CU) computes 128 lines x 128 outputs of C = U D^T on MFMA and
// applies the RK update:
//  * the input lines are read as FP32 (p0 as the pass after each stage left it,
//    vx and vy straight from the stage state), scaled by the scene's power of
//    two 2^e and split into two
//    16-bit parts while they are staged into LDS (U = hi + lo: FP16 keeps 22
//    bits when every scaled value is below 2^15, BF16 16 bits at any scale);
//  * D is stored split the same way (one power of two per matrix), in the order
//    of the MFMA operands, and goes from memory to registers: every wave has 32
//    outputs of its own and all of the tile's lines, so no part of D is loaded
//    twice, and the LDS (reads and writes took as many of its cycles as the
//    multiplication takes when D passed through it too) holds the lines only;
//  * C = U_hi D_hi + U_hi D_lo + U_lo D_hi with v_mfma_f32_32x32x16_{f16,bf16},
//    FP32 accumulation, over k-chunks of 32 through double-buffered LDS (one
//    workgroup barrier per chunk, which waits for no load in flight);
//  * the scene's scale comes from the largest |value| every wavefront of the
//    previous stage wrote (track_max, max_reduce), so no pass over the inputs
//    precedes the multiplication;
//  * pressure lines have n+1 outputs: the multiplication covers the first n,
//    the last is an FP32 dot product of the raw line with D's last row,
//    accumulated by the threads while they stage the line (its 128-wide
//    output tiles then fit n exactly instead of wasting most of a tile).
// U is on the MFMA A side (rows of C = lines, columns = outputs): consecutive
// lanes store consecutive floats of a line, in both directions (vy and py are
// stored column-major).
// Measured (launch alone, D through the LDS -> D straight to registers and the
// lines two chunks ahead): 1024^2 in BF16 53.6 -> 47.3 us, 16 scenes of 512 x 1024
// twice in FP16 536 -> 492 us (335 GFLOP of products: 680 TFLOP/s); 256 such sources in
// 6.22 ms (863 TFLOP/s, and 4.6 TB/s beyond the L2).  Neither bounds it alone: without
// its MFMAs it takes three quarters of the time, without its stores and t_n four
// fifths.  Three workgroups per CU (168 registers, one chunk ahead) do the 16 scenes in
// 502 us and the one scene, which has one workgroup per CU, in 62.
typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef unsigned u32x4 __attribute__((ext_vector_type(4)));

template <typename E>
struct MfmaOps;
template <>
struct MfmaOps<_Float16> {
    typedef _Float16 v8 __attribute__((ext_vector_type(8)));
    typedef _Float16 v4 __attribute__((ext_vector_type(4)));
    __device__ static f32x16 mfma(v8 a, v8 b, f32x16 c) { return __builtin_amdgcn_mfma_f32_32x32x16_f16(a, b, c, 0, 0, 0); }
};
template <>
struct MfmaOps<__bf16> {
    typedef __bf16 v8 __attribute__((ext_vector_type(8)));
    typedef __bf16 v4 __attribute__((ext_vector_type(4)));
    __device__ static f32x16 mfma(v8 a, v8 b, f32x16 c) { return __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, b, c, 0, 0, 0); }
};

constexpr int kGemmThreads = 256;  // 4 waves, each all lines x 32 outputs
constexpr int kGL = 128;           // lines per tile
constexpr int kGN = 128;           // outputs per tile
// (line, 8-k group) pieces of a chunk each thread stages: 2
constexpr int kGSlots = kGL * 32 / 8 / kGemmThreads;
constexpr int kGK = 32;            // k per LDS chunk (two MFMA k-steps)
constexpr int kGPart = kGL * kGK;            // elements of one part (hi or lo) of a chunk of U
constexpr int kGemmDChunk = 2 * kGN * kGK;   // elements of one chunk of D (both parts)
constexpr size_t kGemmLdsBytes = (size_t)2 * 2 * kGPart * 2;  // U: [buffer][part][line][k], 32 KiB
// Element of (row, 8-k group g) in a part: rows of 64 bytes, the groups of a row
// permuted so that 8 rows (32 banks) or 16 rows (64 banks) read with one group
// touch every bank once.
__host__ __device__ constexpr int gemm_slot(int row, int g) {
    return row * kGK + ((g ^ ((row >> 1) & 3) ^ ((row >> 3) & 1)) * 8);
}
// Element of D's value (output, k) of a tile: the operands of one MFMA (32 outputs,
// 16 k, one part) lie together in the order of the lanes that read them, as
// [chunk][k-step][part][output / 32][lane][k % 8].
__host__ __device__ constexpr long long gemm_d_at(int output, int k, int part) {
    return (((long long)(k / 16) * 2 + part) * (kGN / 32) + output / 32) * 512 + (k / 8 % 2 * 32 + output % 32) * 8 + k % 8;
}
static_assert(kGSlots == 2, "staging map assumes two slots per thread");

struct GemmTile {
    TileDesc t;            // segment addressing; line0/count: the tile's lines (count <= 128)
    // D of the tile's 128 outputs (2-byte elements): value (output, k, part hi or
    // lo) at element d_img + gemm_d_at(); d_len elements in all
    long long d_img, d_len;
    int n_rows, k_pad;     // rows of D (multiple of kGN) and columns (multiple of kGK)
    int n0;                // first output of the tile
    int n_g;               // outputs the multiplication produces (n_out, or n_out - 1 with the dot row)
    int d_exp;             // D was stored as D * 2^d_exp
    int K;                 // line length
    int dot_off;           // >= 0: ftab offset of D's last row (FP32): this tile writes output n_out - 1
};
typedef const __attribute__((address_space(4))) GemmTile *GTile;

// Power of two that brings a line whose values are bounded by m below 2^15
// (FP16 keeps both parts normal down to 2^-3 of that bound).
__device__ __forceinline__ int gemm_scale_exp(const StageArgs &a, int scene, int vel) {
    const unsigned bits = a.umax[scene * 2 + (vel ? 1 : 0)];
    const float m = __uint_as_float(bits) * (vel ? 1.f : 2.f);  // p0 = px + py
    return m > 0.f ? min(max(14 - ilogbf(m), -100), 100) : 0;
}

// Raw input values of one chunk held by a thread: 8 consecutive k of two lines
// (4 threads per line, so 4 lanes read 128 contiguous bytes).
struct UChunk {
    float a[kGSlots][8];
};

// Staging map of slot q: 4 threads per line, lines tid/4 and tid/4 + 64.
__device__ __forceinline__ int stage_line(int tid, int q) { return (tid >> 2) + q * (kGemmThreads / 4); }
__device__ __forceinline__ int stage_kq(int tid) { return (tid & 3) * 8; }

// raw buffer over `bytes` bytes at byte offset `byte_off` of `base`
__device__ __forceinline__ Rsrc bytes_rsrc(const void *base, long long byte_off, int bytes) {
    return __builtin_amdgcn_make_buffer_rsrc((void *)((const char *)base + byte_off), (short)0, bytes, 0x00020000);
}

// Line `line` (absolute) of a tile: byte offsets of position k of its raw
// input line in the three blocks it comes from (main, side1, side2).
struct LineAddr {
    int w, nm, K;
    int m_base, s1_base, s2_base;  // offset of k = 0 of each piece (4 bytes per k)
    bool s1, s2;
    __device__ __forceinline__ LineAddr(Seg td, int line, int K_) {
        const int vel = td->vel;
        w = td->wlen;
        nm = td->n_main;
        K = K_;
        m_base = (td->m_a + line * td->m_ls - w) * 4;
        s1 = td->s1_len >= 0;
        s2 = td->s2_len >= 0;
        s1_base = (td->s1_a + (line + td->s1_line) * td->s1_ls + td->s1_len - w - vel) * 4;
        s2_base = (td->s2_a + (line + td->s2_line) * td->s2_ls + vel - w - nm) * 4;
    }
    __device__ int main_off(int k) const { return k >= w && k < w + nm ? m_base + k * 4 : kOOB; }
    __device__ int s1_off(int k) const { return s1 && k < w ? s1_base + k * 4 : kOOB; }
    __device__ int s2_off(int k) const { return s2 && k >= w + nm && k < K ? s2_base + k * 4 : kOOB; }
};

// Which piece of the line a whole chunk [k0, k0 + kGK) lies in (the same for
// every line of a tile).  kPieceS2 chunks may run past K: positions from K on
// read zero (a value from past the halo could be another field, outside the
// range the scene's scale was chosen for).
constexpr int kPieceMain = 0, kPieceS1 = 1, kPieceS2 = 2, kPieceMixed = 3, kPieceNone = 4;
__device__ __forceinline__ int chunk_piece(Seg td, int K, int k0) {
    const int w = td->wlen, nm = td->n_main;
    return k0 >= K                              ? kPieceNone
           : k0 >= w && k0 + kGK <= w + nm      ? kPieceMain
           : k0 + kGK <= w                      ? kPieceS1
           : k0 >= w + nm                       ? kPieceS2
                                                : kPieceMixed;
}

// (Selections are between values, never between struct members: a select of
// member lvalues keeps the struct in scratch memory.)
template <class T>
__device__ __forceinline__ T pick3(int piece, T main, T s1, T s2) {
    return piece == kPieceMain ? main : piece == kPieceS1 ? s1 : s2;
}
// Buffer resource of one piece's domain block.
__device__ __forceinline__ Rsrc piece_rsrc(const float *src, Seg td, int piece) {
    return block_rsrc(src, pick3<long long>(piece, td->m_dom, td->s1_dom, td->s2_dom),
                      pick3<int>(piece, td->m_size, td->s1_size, td->s2_size));
}

// A chunk that is not all main values (one or two at either end of a line).
__device__ __forceinline__ void gemm_load_ends(const float *src, Seg td, int K, const bool (&ok)[kGSlots], int k0,
                                               UChunk &u) {
    const int kb = k0 + stage_kq(threadIdx.x);
    const int piece = chunk_piece(td, K, k0);
#pragma unroll
    for (int q = 0; q < kGSlots; ++q) {
        const LineAddr L(td, td->line0 + stage_line(threadIdx.x, q), K);
        if (piece == kPieceMixed) {
            // a chunk across a piece boundary: each value from whichever block holds it
            const Rsrc m = piece_rsrc(src, td, kPieceMain), s1 = piece_rsrc(src, td, kPieceS1),
                       s2 = piece_rsrc(src, td, kPieceS2);
#pragma unroll
            for (int j = 0; j < 8; ++j) {
                const int k = kb + j;
                const int om = ok[q] ? L.main_off(k) : kOOB, o1 = ok[q] ? L.s1_off(k) : kOOB,
                          o2 = ok[q] ? L.s2_off(k) : kOOB;
                u.a[q][j] = bload(m, om) + bload(s1, o1) + bload(s2, o2);
            }
        } else {
            // one block for the whole chunk; side-2 chunks may run to the end of the
            // block: 4-byte loads
            const Rsrc r = piece_rsrc(src, td, piece);
            const bool in = ok[q] && ((piece == kPieceS1 && L.s1) || (piece == kPieceS2 && L.s2));
            const int base = piece == kPieceS1 ? L.s1_base : L.s2_base;
#pragma unroll
            for (int j = 0; j < 8; ++j) u.a[q][j] = bload(r, in && kb + j < K ? base + (kb + j) * 4 : kOOB);
        }
    }
}

// The input lines of a tile.  In a chunk of main values every k lies in the
// line's own block: a per-lane part of the byte offset (line and k-group; kOOB
// for lanes past the tile's lines) and a uniform part (the chunk's k), both
// non-negative.
struct GemmLines {
    const float *src;
    Seg td;
    int K;
    bool ok[kGSlots];
    Rsrc r;
    int voff[kGSlots];
    __device__ __forceinline__ void load_main(int c, UChunk &u) const {
        const int so = (c * kGK - td->wlen) * 4;
#pragma unroll
        for (int q = 0; q < kGSlots; ++q) {
            const float4 x0 = __builtin_bit_cast(float4, __builtin_amdgcn_raw_buffer_load_b128(r, voff[q], so, 0));
            const float4 x1 = __builtin_bit_cast(float4, __builtin_amdgcn_raw_buffer_load_b128(r, voff[q] + 16, so, 0));
            u.a[q][0] = x0.x; u.a[q][1] = x0.y; u.a[q][2] = x0.z; u.a[q][3] = x0.w;
            u.a[q][4] = x1.x; u.a[q][5] = x1.y; u.a[q][6] = x1.z; u.a[q][7] = x1.w;
        }
    }
    __device__ __forceinline__ void load(int c, UChunk &u) const {
        if (chunk_piece(td, K, c * kGK) == kPieceMain) load_main(c, u);
        else gemm_load_ends(src, td, K, ok, c * kGK, u);
    }
};

// A wave's operands of a chunk of D: 32 outputs, straight from memory to
// registers (1 KiB per load; the matrix stays in the caches).
template <typename E>
struct DChunk {
    typename MfmaOps<E>::v8 b[2][2];  // [k-step][part]
    __device__ __forceinline__ void load(Rsrc dr, int voff, int c) {
#pragma unroll
        for (int s = 0; s < 2; ++s)
#pragma unroll
            for (int p = 0; p < 2; ++p)
                b[s][p] = __builtin_bit_cast(typename MfmaOps<E>::v8, __builtin_amdgcn_raw_buffer_load_b128(
                                                 dr, voff, c * kGemmDChunk * 2 + (s * 2 + p) * (kGN / 32) * 1024, 0));
    }
};

// Converts and writes one chunk into LDS buffer `buf` (8 k of one line per
// thread as one 16-byte write per part).
template <typename E>
__device__ __forceinline__ void gemm_stage(E *ulds, int buf, const UChunk &u, float sc) {
    using V8 = typename MfmaOps<E>::v8;
    const int tid = threadIdx.x;
    E *U0 = ulds + buf * 2 * kGPart, *U1 = U0 + kGPart;
#pragma unroll
    for (int q = 0; q < kGSlots; ++q) {
        // (a slot's rows lie 64 apart: the same permutation)
        const int at = gemm_slot(stage_line(tid, 0), tid & 3) + q * (kGemmThreads / 4) * kGK;
        V8 hi, lo;
#pragma unroll
        for (int j = 0; j < 8; ++j) {
            const float x = u.a[q][j] * sc;
            const E h = (E)x;
            hi[j] = h;
            lo[j] = (E)(x - (float)h);
        }
        *reinterpret_cast<V8 *>(U0 + at) = hi;
        *reinterpret_cast<V8 *>(U1 + at) = lo;
    }
}

// The chunk's part of the lines' FP32 dot products with the last output row
// (dotr; only in the last output tile of a line block).
__device__ __forceinline__ void gemm_dot(const UChunk &u, Rsrc dotr, int c, float (&gv)[kGSlots]) {
    float dk[8];
#pragma unroll
    for (int j = 0; j < 8; ++j) dk[j] = bload(dotr, (c * kGK + stage_kq(threadIdx.x) + j) * 4);  // zero from K on
#pragma unroll
    for (int q = 0; q < kGSlots; ++q)
#pragma unroll
        for (int j = 0; j < 8; ++j) gv[q] = __builtin_fmaf(u.a[q][j], dk[j], gv[q]);
}

// The MFMAs of one chunk (U0: its buffer): the tile's 128 lines (4 blocks of 32)
// x the wave's 32 outputs.
template <typename E, int DIR>
__device__ __forceinline__ void gemm_chunk(const E *U0, const DChunk<E> &d, f32x16 (&acc)[4]) {
    using V8 = typename MfmaOps<E>::v8;
    const int lane = threadIdx.x & 63;
#pragma unroll
    for (int s = 0; s < kGK / 16; ++s) {
        // (rows 32 apart: the same permutation)
        const int at = gemm_slot(lane & 31, 2 * s + (lane >> 5));
        V8 ah[4], al[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            ah[i] = *reinterpret_cast<const V8 *>(U0 + at + 32 * i * kGK);
            al[i] = *reinterpret_cast<const V8 *>(U0 + kGPart + at + 32 * i * kGK);
        }
        // each product over the four independent accumulators in turn (no
        // back-to-back MFMAs on one accumulator); the low parts of D first for X
        // lines, those of U for Y lines (a fixed order of the sums per direction)
        auto product = [&](const V8 (&x)[4], const V8 &y) __attribute__((always_inline)) {
#pragma unroll
            for (int i = 0; i < 4; ++i) acc[i] = MfmaOps<E>::mfma(x[i], y, acc[i]);
        };
        product(ah, d.b[s][0]);
        if constexpr (DIR == 0) {
            product(ah, d.b[s][1]);
            product(al, d.b[s][0]);
        } else {
            product(al, d.b[s][0]);
            product(ah, d.b[s][1]);
        }
    }
}

// The workgroup's LDS writes become visible; loads in flight are not waited for.
__device__ __forceinline__ void lds_barrier() {
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
}

template <typename E, int DIR>
__device__ __forceinline__ void gemm_tile(const StageArgs &a, GTile gt, const float *ftab, unsigned char *gemm_lds) {
    E *ulds = reinterpret_cast<E *>(gemm_lds);
    const Seg td = &gt->t;
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int e = gemm_scale_exp(a, td->scene, td->vel);
    const float sc = ldexpf(1.f, e);
    const Rsrc dr = bytes_rsrc(a.dmat, gt->d_img * 2, (int)(gt->d_len * 2));
    const bool dot = gt->dot_off >= 0;
    const int nch = gt->k_pad / kGK;
    GemmLines in;
    in.src = source(a, td->vel);
    in.td = td;
    in.K = gt->K;
    in.r = block_rsrc(in.src, td->m_dom, td->m_size);
#pragma unroll
    for (int q = 0; q < kGSlots; ++q) {
        in.ok[q] = stage_line(tid, q) < td->count;
        in.voff[q] = in.ok[q] ? (td->m_a + (td->line0 + stage_line(tid, q)) * td->m_ls + stage_kq(tid)) * 4 : kOOB;
    }
    const Rsrc dotr = bytes_rsrc(ftab, dot ? (long long)gt->dot_off * 4 : 0, dot ? in.K * 4 : 0);
    // waves whose outputs lie outside the tile skip their MFMAs
    const bool active = 32 * wave < gt->n_g - gt->n0;
    f32x16 acc[4];
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int q = 0; q < 16; ++q) acc[i][q] = 0.f;
    float gv[kGSlots] = {0.f, 0.f};
    // While chunk c is multiplied, the lines of chunk c + 2 and D of chunk c + 1 are
    // on their way to registers, and the lines of chunk c + 1, requested an iteration
    // before, are then converted into the other LDS buffer.
    UChunk u0, u1;
    DChunk<E> da, db;
    const int dv = (wave * 64 + lane) * 16;
    in.load(0, u0);
    da.load(dr, dv, 0);
    if (nch > 1) in.load(1, u1);
    gemm_stage<E>(ulds, 0, u0, sc);
    if (dot) gemm_dot(u0, dotr, 0, gv);
    lds_barrier();
    int c = 0;
    // chunk c + 2 is of main values: no branch between its loads and their use
    auto step_main = [&](auto mult, auto parity, const DChunk<E> &d, DChunk<E> &next) __attribute__((always_inline)) {
        constexpr int buf = decltype(parity)::value;
        UChunk &cur = buf ? u0 : u1, &after = buf ? u1 : u0;
        if constexpr (decltype(mult)::value) next.load(dr, dv, c + 1);
        in.load_main(c + 2, after);
        if constexpr (decltype(mult)::value) {
            gemm_chunk<E, DIR>(ulds + buf * 2 * kGPart, d, acc);
        }
        gemm_stage<E>(ulds, buf ^ 1, cur, sc);
        if (dot) gemm_dot(cur, dotr, c + 1, gv);
        lds_barrier();
        ++c;
    };
    auto step_end = [&](auto parity, const DChunk<E> &d, DChunk<E> &next) __attribute__((always_inline)) {
        constexpr int buf = decltype(parity)::value;
        const bool more = c + 1 < nch;
        UChunk &cur = buf ? u0 : u1, &after = buf ? u1 : u0;
        if (more) next.load(dr, dv, c + 1);
        if (c + 2 < nch) in.load(c + 2, after);
        if (active) gemm_chunk<E, DIR>(ulds + buf * 2 * kGPart, d, acc);
        if (more) {
            gemm_stage<E>(ulds, buf ^ 1, cur, sc);
            if (dot) gemm_dot(cur, dotr, c + 1, gv);
            lds_barrier();
        }
        ++c;
    };
    using P0 = std::integral_constant<int, 0>;
    using P1 = std::integral_constant<int, 1>;
    // main chunks: [1, cm1) (a halo is at most 32 long)
    const int cm1 = (td->wlen + td->n_main) / kGK;
    if (active) {
#pragma unroll 1
        while (c + 3 < cm1) {
            step_main(P1{}, P0{}, da, db);
            step_main(P1{}, P1{}, db, da);
        }
    } else {
#pragma unroll 1
        while (c + 3 < cm1) {
            step_main(P0{}, P0{}, da, db);
            step_main(P0{}, P1{}, db, da);
        }
    }
#pragma unroll 1
    while (true) {
        step_end(P0{}, da, db);
        if (c >= nch) break;
        step_end(P1{}, db, da);
        if (c >= nch) break;
    }
    // epilogue: L = C / (2^e 2^d_exp); out = t_n - s*coef*L (Solver::update_field_values)
    const float sc_upd = a.s * td->coef, inv = ldexpf(1.f, -(e + gt->d_exp));
    const bool use_pml = a.last && td->is_pml;
    const Rsrc rt = block_rsrc(a.tn, td->m_dom, td->m_size);
    const Rsrc rp = block_rsrc(a.pml, td->m_dom, td->m_size);
    const Rsrc ro = block_rsrc(a.out, td->m_dom, td->m_size);
    float mx = 0.f;
    if (active) {
        // value q of block i: line 32 i + 8 (q >> 2) + 4 (lane >> 5) + (q & 3), output 32 wave + (lane & 31)
        // of the tile; all t_n loads are issued before the first is used.  A per-lane
        // offset and, per value, a uniform one (the buffer instruction's scalar offset;
        // no address arithmetic on the vector unit) — lines past the tile's last by
        // their own condition
        const int line0 = 4 * (lane >> 5), n = gt->n0 + 32 * wave + (lane & 31);
        const int base = n < gt->n_g ? (td->o_f + (td->line0 + line0) * td->o_ls + n) * 4 : kOOB;
        auto line = [](int i, int q) { return 32 * i + 8 * (q >> 2) + (q & 3); };
        // (what a block of 16 values is addressed with, anew for each pass over them)
        struct Rows {
            int left, ls4;  // lines from this lane's first on; bytes from line to line
        };
        auto rows = [&]() __attribute__((always_inline)) {
            Rows r{td->count - line0, again(td->o_ls) * 4};
            asm volatile("" : "+v"(r.left));
            return r;
        };
        auto offset = [&](const Rows &r, int i, int q) __attribute__((always_inline)) {
            return line(i, q) < r.left ? base : kOOB;
        };
        float y[4][16];
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const Rows r = rows();
#pragma unroll
            for (int q = 0; q < 16; ++q) y[i][q] = bload(rt, offset(r, i, q), line(i, q) * r.ls4);
        }
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const Rows r = rows();
#pragma unroll
            for (int q = 0; q < 16; ++q) {
                y[i][q] = __builtin_fmaf(-sc_upd, acc[i][q] * inv, y[i][q]);
                const int o = offset(r, i, q);
                bstore(ro, o, line(i, q) * r.ls4, y[i][q]);
                mx = fmaxf(mx, o == kOOB ? 0.f : fabsf(y[i][q]));
            }
        }
        if (a.last) {
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const Rows r = rows();
                if (use_pml) {
                    float pm[16];
#pragma unroll
                    for (int q = 0; q < 16; ++q) pm[q] = bload(rp, offset(r, i, q), line(i, q) * r.ls4);
#pragma unroll
                    for (int q = 0; q < 16; ++q) y[i][q] *= pm[q];
                }
#pragma unroll
                for (int q = 0; q < 16; ++q) bstore(rt, offset(r, i, q), line(i, q) * r.ls4, y[i][q]);
            }
        }
    }
    if (dot) {
        // output n_out - 1 of every line: the FP32 dot products (no scaling)
        const int n = gt->n_g;
        auto write_dot = [&](int line, float Ldot) {
            if (line < 0 || line >= td->count) return;
            const int off = (td->o_f + (td->line0 + line) * td->o_ls + n) * 4;
            const float tnv = bload(rt, off), pm = use_pml ? bload(rp, off) : 1.f;
            const float nv = __builtin_fmaf(-sc_upd, Ldot, tnv);
            bstore(ro, off, 0, nv);
            if (a.last) bstore(rt, off, 0, nv * pm);
            mx = fmaxf(mx, fabsf(nv));
        };
        // the 4 threads of a line are adjacent lanes; slot q holds line tid/4 + 64 q
#pragma unroll
        for (int q = 0; q < kGSlots; ++q) {
            float g = gv[q];
            g += __shfl_xor(g, DIR == 0 ? 1 : 2);
            g += __shfl_xor(g, DIR == 0 ? 2 : 1);
            write_dot((tid & 3) == 0 ? stage_line(tid, q) : -1, g);
        }
    }
    track_max(a, td->slot, mx);
}

template <typename E>
__global__ void __launch_bounds__(kGemmThreads) __attribute__((amdgpu_waves_per_eu(2)))
stage_gemm_kernel(StageArgs a, const GemmTile *__restrict__ tiles, const float *__restrict__ ftab) {
    extern __shared__ __attribute__((aligned(16))) unsigned char gemm_lds[];
    // XCD-contiguous runs of tiles always (the tiles of one matrix and of one
    // line block share an XCD's L2), whatever order the FFT-form tiles use
    const GTile gt = (GTile)tiles + tile_index(blockIdx.x, gridDim.x, 1);
    if (gt->t.dir == 0) gemm_tile<E, 0>(a, gt, ftab, gemm_lds);
    else gemm_tile<E, 1>(a, gt, ftab, gemm_lds);
}

// Largest |p0| and |vx|, |vy| of every scene in the state a first stage reads
// after the host wrote fields (it has no previous stage).
struct MaxRange {
    long long off;  // element offset from the arena base
    long long n;
    int idx;        // scene * 2 + class
};

__global__ void fill_zero_kernel(unsigned *__restrict__ p, int n) {
    for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += gridDim.x * blockDim.x) p[i] = 0u;
}

__global__ void state_max_kernel(const float *__restrict__ arena, unsigned *__restrict__ umax,
                                 const MaxRange *__restrict__ ranges, int nr) {
    for (int k = blockIdx.y; k < nr; k += gridDim.y) {
        const MaxRange r = ranges[k];
        float m = 0.f;
        for (long long e = blockIdx.x * (long long)blockDim.x + threadIdx.x; e < r.n; e += (long long)gridDim.x * blockDim.x)
            m = fmaxf(m, fabsf(arena[r.off + e]));
#pragma unroll
        for (int o = 32; o >= 1; o >>= 1) m = fmaxf(m, __shfl_xor(m, o));
        if ((threadIdx.x & 63) == 0 && m > 0.f) atomicMax(&umax[r.idx], __float_as_uint(m));
    }
}

// ------------------------------------------------------------- host side

#define HIP_TRY(expr)                                                                   \
    do {                                                                                \
        hipError_t _e = (expr);                                                         \
        if (_e != hipSuccess) {                                                         \
            ctx->err = std::string(#expr) + ": " + hipGetErrorString(_e);               \
            return PSTD_ERR_DEVICE;                                                     \
        }                                                                               \
    } while (0)

int next_pow2(int n) {
    int p = 1;
    while (p < n) p <<= 1;
    return p;
}

}  // namespace

// Time steps per captured hipGraph unless pstd_ctx_set_graph_steps says otherwise.
constexpr int kDefaultGraphSteps = 20;

// p0 on the fly or in a pass of its own: the pass moves 16 bytes per cell and costs
// a launch (5 us); on the fly, a tile of n adjacent lines reads 4 n bytes of every
// 64-byte sector the other layout's field has in it.  The pass is taken where the
// fly moves this many bytes per stage more (about 5 us at 4 TB/s).  Measured, us
// per stage on the fly / with the pass: L-shape 7.7 / 14.2, 333 000 cells 11.8 / 19.2,
// one 900^2 domain 22.1 / 26.0, 1024^2 30.3 / 32.8, 1200^2 37.0 / 36.3, 1900^2 59.5 /
// 55.3, 2501 x 1237 69.1 / 55.7, 4096^2 465 / 394; twelve scenes of lines up to 600 (at
// least 8 lines per tile) 93.5 / 106.  Far above the line the two can be level: 16
// sources of 512 x 1024 twice, 133 MB more by this count, take 344 / 346.
constexpr long long kP0PassBytes = 20000000;
// 64-byte sectors read per 64 bytes used by a tile's strided reads (256 threads)
static int strided_factor(int F) {
    return std::max(1, 16 / std::max(2, 2 * 256 / (F / fft_values(F))));
}

// 1024- and 2048-point lines take 16 values per thread (one and two wavefronts per
// pair) or 8 (two and four): half the chain of arithmetic, t_n and the filter loaded
// with the lines, for a barrier per exchange and twice the twiddle loads.  A scene
// of few wavefronts (counted with 16; the chip holds 4096) is bound by that chain.
// Measured with 16 / 8, us per stage, wavefronts in brackets: 623 x 182 (1132) 11.0 /
// 9.2, 500^2 (1792) 13.8 / 12.6, 1500 x 150 (2214) 15.4 / 12.2, 700^2 (2392) 16.9 / 15.4,
// rooms of 333, 141, 477 x 217 (2508) 11.7 / 11.0, 1198 x 206 (2702) 14.8 / 14.1, 850^2
// (2844) 18.9 / 20.0, 900^2 (2992) 19.5 / 20.6, 1268 x 303 (3048) 15.9 / 15.7, two of 480^2
// (3472) 17.7 / 16.6, 600 x 1073 (3504) 20.9 / 21.5, 1024^2 (5616) 29.8 / 30.9, six of 480^2
// (10416) 35.2 / 36.3; the line tiles beside the matrix form of 1024^2 (1520) 63.4 / 60.4 with
// that form's launch.  No count separates the gains from the losses between 2700 and 3500:
// the line lies below the first loss, and what it gives away there is at most 6 %.
constexpr long long kFewWaves = 2750;

// Results of at most kPinBytes reach the caller's (pageable) memory through pinned
// memory of the context: a copy to pinned memory needs no staging by the runtime,
// and a kernel that has to run first writes there itself (100 x 50 room: one
// step's samples 5 us instead of 21, p0 13.5 instead of 36, vy0 13.4 instead of 29).
// A runtime copy that follows a kernel waits for it on the host, 16 us: through
// pinned memory / by the runtime, p0 of 257 x 256 cells takes 23 / 139 us, py 22 / 36;
// of 400 x 301 32 / 48 and 31 / 46; of 500 x 501 53 / 72 and 53 / 68; of 700 x 700 (1.9
// MiB) 125 / 126 and 115 / 123, but its px 114 / 106; of 1000 x 1001 254 / 238.  Longer
// results go through the runtime's staging (eight threads copying 256-KiB pieces
// from pinned memory took 420 us for 4 MiB, against 320 into untouched pages).
constexpr size_t kPinBytes = 1 << 20;

// A context takes its pinned memory at the first short result and gives it back when
// it is destroyed.  A program that makes a solver per run (PSTDKernel::run) paid 70 to
// 120 us for it each time (run() of 121 steps of the L-shape 7400 -> 7285 us, of two
// steps of 18 domains 1680 -> 1610): up to kPinKept buffers wait for the next
// context, of any device (portable), the others are freed.
constexpr size_t kPinKept = 4;
static std::mutex g_pinned_mu;
static std::vector<char *> g_pinned;

static char *take_pinned() {
    {
        std::lock_guard<std::mutex> lock(g_pinned_mu);
        if (!g_pinned.empty()) {
            char *p = g_pinned.back();
            g_pinned.pop_back();
            return p;
        }
    }
    void *p = nullptr;
    if (hipHostMalloc(&p, kPinBytes, hipHostMallocPortable) == hipSuccess) return (char *)p;
    (void)hipGetLastError();  // the runtime's staging then
    return nullptr;
}

// (no work that uses it is in flight)
static void give_pinned(char *p) {
    if (!p) return;
    {
        std::lock_guard<std::mutex> lock(g_pinned_mu);
        if (g_pinned.size() < kPinKept) {
            g_pinned.push_back(p);
            return;
        }
    }
    (void)hipHostFree(p);
}

// Calls on one context take turns, in the order of their arrival: a thread that
// advances in a loop does not keep one that reads frames from its turn (a plain
// mutex is taken again before a thread woken up by its release can run).
class TurnLock {
public:
    void lock() {
        std::unique_lock<std::mutex> l(mu);
        const uint64_t mine = next++;
        cv.wait(l, [&] { return serving == mine; });
    }
    void unlock() {
        {
            std::lock_guard<std::mutex> l(mu);
            ++serving;
        }
        cv.notify_all();
    }

private:
    std::mutex mu;
    std::condition_variable cv;
    uint64_t next = 0, serving = 0;
};

struct pstd_ctx {
    // Held by every call that issues work or changes the context, until the work
    // that the call waits for is done: reads share the pinned memory and turn vy and
    // py through S0, which is free between time steps only, and a captured step
    // graph must hold nothing else.
    TurnLock turn;
    int device = 0;
    hipStream_t stream = nullptr;
    // with `overlap`, GEMM-form stages run their FFT-form tiles on `side`,
    // concurrently with the GEMM kernel on `stream` (fork and join through the
    // two events; both streams at the default priority).  Off by default: two
    // wavefronts of the GEMM kernel leave 112 of a SIMD's 512 registers, one of an
    // FFT-form tile takes 128, so the two kernels only trade places, and the events
    // cost.  In order / overlapped, us per stage in the FP16 form: 1024^2 60.4 / 64.6
    // (one workgroup per CU, where both would fit), 4096^2 1566 / 1638, 16 sources of
    // 512 x 1024 twice 532 / 536, 64 scenes 1822 / 1849
    hipStream_t side = nullptr;
    hipEvent_t ev_fork = nullptr, ev_join = nullptr;
    bool overlap = false;
    std::string err;
    bool planned = false;
    // plan
    std::vector<DomainDev> doms;
    std::vector<pstd_plan_domain> plan_domains;
    // FFT-form segments (line0/count = the segment's line range), passthrough
    // fields and the receivers: the tile list is cut from them for the block size
    // (stage_threads)
    std::vector<TileDesc> fft_segs;
    int n_tiles = 0;
    int small_nt = 256;  // block size where the lines leave the choice (autotuned: 128 or 256)
    int small_fmax = 0;  // largest F of the F <= 2048 class (128 threads need F <= 1024)
    int fmax = 0;        // largest F
    // block size of the stage launch: the threads of one line pair
    int stage_threads() const { return std::max(small_nt, fmax / values(fmax)); }
    int f8 = 512;  // longest lines with 8 values per thread (kFewWaves)
    int values(int F) const { return F <= f8 ? 8 : 16; }
    std::vector<GemmTile> tiles_gemm;
    int n_scenes = 1;
    std::vector<MaxRange> max_ranges;  // state read by a first stage after host writes (GEMM form)
    int form = PSTD_FORM_FFT;      // the form the uploaded plan runs in
    int form_req = PSTD_FORM_FFT;  // as requested (PSTD_FORM_AUTO: chosen at upload)
    double gemm_flops = 0;   // algorithmic MFMA flops of one stage (3 split products)
    long long gemm_cells = 0;
    size_t arena_floats = 0;
    float dt = 0, c1 = 0;
    float alpha[6] = {0};
    int nrec = 0;
    // device buffers
    float *arena = nullptr;  // 4 arenas back to back: TN, S0, S1, P0I
    float *pml = nullptr;
    float2 *ctab = nullptr;
    float *ftab = nullptr;
    TileDesc *d_tiles = nullptr;
    GemmTile *d_gemm = nullptr;
    void *dmat = nullptr;         // derivative matrices of the GEMM form (hi, lo parts; 2-byte elements)
    unsigned *umax = nullptr;     // maxima of the written values, scenes x 2 classes
    float *wmax = nullptr;        // per wavefront (track_max): the FFT-form tiles' slots, then the GEMM tiles'
    int2 *d_max_first = nullptr;
    std::vector<int> gemm_first;  // first GEMM slot of every group (scene, class), then their number
    MaxRange *d_max_ranges = nullptr;
    ReceiverCell *d_cells = nullptr;
    // spectral receivers: line jobs, per-receiver jobs, weights, column buffer
    SILine *d_si_lines = nullptr;
    SIPoint *d_si_points = nullptr;
    float *d_si_coef = nullptr;
    float *d_si_col = nullptr;
    int n_si_lines = 0, n_si = 0;
    P0Tile *d_p0_tiles = nullptr;
    std::vector<int> p0_first;   // first tile of every domain, then the number of tiles
    // p0 is formed by p0_pass_kernel after every stage (P0I then always holds the
    // current p0), otherwise by the tiles that read it
    bool p0_pass = false;
    float *d_samples = nullptr;
    int sample_cap = 0;
    int steps_done = 0;
    bool p0_explicit = true;
    bool p0_turn = false;  // explicit p0 written since its transpose was
    // vy (even) and py (odd) of every domain written by the host and not turned yet:
    // row-major in S0 (turn_written)
    std::vector<char> written;
    bool any_written = false;
    int xcd_remap = 1;
    // stage kernel flavour as set (0 early, 1 late, 2 mid) and reported back: one kernel
    // serves them all
    int lean = 1;
    float tuned_stage_ms = 0;
    // the GEMM form's maxima in `umax` no longer describe the state (an
    // allocation-free advance used the shared array): recompute before the next step
    bool max_stale = false;
    // per-kernel-class timing (pstd_ctx_profile_kernels): event pairs around
    // every launch of a class while `prof` is set
    bool prof = false;
    std::vector<std::pair<int, std::pair<hipEvent_t, hipEvent_t>>> prof_events;
    // hipGraph of `graph_steps` whole time steps (0: launches are issued one by
    // one).  The graph writes its receiver samples into `d_gsamples`; each replay
    // is followed by a device-side copy to its place in `d_samples`.
    int graph_steps = kDefaultGraphSteps;
    hipGraph_t graph = nullptr;
    hipGraphExec_t graph_exec = nullptr;
    float *d_gsamples = nullptr;
    // autotuner bookkeeping: time steps its trials ran, and whether the launch
    // shape came from the per-(device, plan) cache instead
    int trial_steps = 0;
    bool tune_cached = false;

    // Pinned memory that short results pass through on their way to the caller
    // (short_result), taken by the first of them.
    char *pin = nullptr;

    void drop_graph() {
        if (graph_exec) (void)hipGraphExecDestroy(graph_exec);
        if (graph) (void)hipGraphDestroy(graph);
        if (d_gsamples) (void)hipFree(d_gsamples);
        graph_exec = nullptr;
        graph = nullptr;
        d_gsamples = nullptr;
    }

    float *TN() const { return arena; }
    float *S(int i) const { return arena + (1 + i) * arena_floats; }
    float *P0I() const { return arena + 3 * arena_floats; }

    void release() {
        drop_graph();
        (void)hipFree(arena);
        (void)hipFree(pml);
        (void)hipFree(ctab);
        (void)hipFree(ftab);
        (void)hipFree(d_tiles);
        (void)hipFree(d_gemm);
        (void)hipFree(dmat);
        (void)hipFree(umax);
        (void)hipFree(wmax);
        (void)hipFree(d_max_first);
        wmax = nullptr;
        d_max_first = nullptr;
        (void)hipFree(d_max_ranges);
        d_gemm = nullptr;
        dmat = nullptr;
        umax = nullptr;
        d_max_ranges = nullptr;
        (void)hipFree(d_cells);
        (void)hipFree(d_si_lines);
        (void)hipFree(d_si_points);
        (void)hipFree(d_si_coef);
        (void)hipFree(d_si_col);
        d_si_lines = nullptr;
        d_si_points = nullptr;
        d_si_coef = d_si_col = nullptr;
        n_si_lines = n_si = 0;
        (void)hipFree(d_p0_tiles);
        (void)hipFree(d_samples);
        arena = pml = ftab = d_samples = nullptr;
        ctab = nullptr;
        d_tiles = nullptr;
        d_cells = nullptr;
        d_p0_tiles = nullptr;
        planned = false;
    }
};

namespace {

// Device plan cache entries: the tables of plan_tables.h rounded once to float.
void build_filter(int F, int L, int field, double dx, int values, std::vector<float2> &out) {
    const std::vector<std::complex<double>> h = pstdamd::derivative_filter(F, L, field, dx);
    out.resize(F);
    // thread t's values t + m T in pairs of m, [m / 2][t][m % 2]; length 8192: the even
    // and the odd bin of t + 512 m, [m][t][bin % 2]
    const int T = F / values;
    for (int k = 0; k < F; ++k) {
        const int m = k / T, t = k % T;
        out[F == 8192 ? k : ((m / 2) * T + t) * 2 + m % 2] = make_float2((float)h[k].real(), (float)h[k].imag());
    }
}

// The tables of fft_line.h.
void build_twiddles(int F, std::vector<float2> &out) {
    out.clear();
    auto root = [](int i, int n) {
        const double a = -2.0 * M_PI * (double)i / (double)n;
        return make_float2((float)std::cos(a), (float)std::sin(a));
    };
    const int Fp = std::min(F, 4096);
    for (int p = 1; p < fft_npasses(Fp); ++p)
        for (int r = 0; r < fft_radix(Fp, p); r += 2)
            for (int k = 0; k < fft_span(Fp, p); ++k)
                for (int q = r; q < r + 2; ++q) out.push_back(root(q * k * (Fp / (fft_span(Fp, p) * fft_radix(Fp, p))), Fp));
    if (F == 8192)
        for (int m = 0; m < 8; m += 2)
            for (int t = 0; t < 512; ++t)
                for (int q = m; q < m + 2; ++q) out.push_back(root(t + 512 * q, F));
}

void build_window(int w, int patch_error, std::vector<float> &out) {
    const std::vector<double> win = pstdamd::window_coefficients(w, patch_error);
    out.assign(win.begin(), win.end());
}

// Kernel classes of pstd_ctx_profile_kernels: the FFT-form launch counts for the
// class of its longest lines.
constexpr int kClassSmall = 0, kClass4096 = 1, kClass8192 = 2, kClassGemm = 3, kClasses = 4;

typedef void (*StageKernel)(const TileDesc *, int, int, StageArgs);
StageKernel stage_kernel(int nt) {
    return nt <= 128 ? stage_fft_kernel<128> : nt <= 256 ? stage_fft_kernel<256> : stage_fft_kernel<512>;
}

// Brackets the launches issued by `launch` with an event pair when profiling.
template <class Fn>
void timed_launch(pstd_ctx *ctx, hipStream_t st, int cls, Fn launch) {
    if (!ctx->prof) {
        launch();
        return;
    }
    hipEvent_t e0 = nullptr, e1 = nullptr;
    if (hipEventCreate(&e0) != hipSuccess || hipEventCreate(&e1) != hipSuccess) {
        launch();
        return;
    }
    (void)hipEventRecord(e0, st);
    launch();
    (void)hipEventRecord(e1, st);
    ctx->prof_events.push_back({cls, {e0, e1}});
}

// One RK stage.  sample_slot >= 0 (first stage only): the launch also records
// the receivers of the previous step into that sample slot.
int launch_p0(pstd_ctx *ctx, int d, bool from_stage);

int launch_stage(pstd_ctx *ctx, int k, int sample_slot) {
    if (k == 0 && ctx->p0_turn) {
        const int rc = launch_p0(ctx, -1, false);
        if (rc) return rc;
        ctx->p0_turn = false;
    }
    StageArgs a{};
    a.ctab = ctx->ctab;
    a.ftab = ctx->ftab;
    const int in = (k + 1) & 1, outi = k & 1;
    a.p0_two = !ctx->p0_pass && !(k == 0 && ctx->p0_explicit);
    a.p0 = a.p0_two ? ctx->S(in) : ctx->P0I();
    a.vsrc = k == 0 ? ctx->TN() : ctx->S(in);
    a.cells = ctx->d_cells;
    a.nrec = ctx->nrec;
    a.samples = ctx->d_samples;
    a.slot = (k == 0 && !ctx->p0_explicit && ctx->nrec > 0) ? sample_slot : -1;
    a.tn = ctx->TN();
    a.out = ctx->S(outi);
    a.pml = ctx->pml;
    a.s = ctx->dt * ctx->alpha[k];
    a.f8 = ctx->f8;
    a.last = k == 5;
    const int ng = (int)ctx->tiles_gemm.size();
    if (ng) {
        a.wmax = ctx->wmax;
        a.umax = ctx->umax;
        a.dmat = ctx->dmat;
        if (k == 0 && ctx->p0_explicit && !ctx->max_ranges.empty()) {
            const int nr = (int)ctx->max_ranges.size();
            const int n = 2 * ctx->n_scenes;
            hipLaunchKernelGGL(fill_zero_kernel, dim3((n + 255) / 256), dim3(256), 0, ctx->stream, ctx->umax, n);
            hipLaunchKernelGGL(state_max_kernel, dim3(16, std::min(nr, 4096)), dim3(256), 0, ctx->stream, ctx->arena,
                               ctx->umax, ctx->d_max_ranges, nr);
        }
    }
    const int ns = ctx->n_tiles;
    const int nt = ctx->stage_threads();
    // FFT-form tiles beside a GEMM launch: on the side stream, forked after
    // everything issued so far and joined before anything issued later
    const bool fork = ng && ns && ctx->overlap && ctx->side;
    const hipStream_t fs = fork ? ctx->side : ctx->stream;
    if (fork) {
        HIP_TRY(hipEventRecord(ctx->ev_fork, ctx->stream));
        HIP_TRY(hipStreamWaitEvent(ctx->side, ctx->ev_fork, 0));
    }
    if (ns) timed_launch(ctx, fs, ctx->fmax >= 8192 ? kClass8192 : ctx->fmax >= 4096 ? kClass4096 : kClassSmall, [&] {
        hipLaunchKernelGGL(stage_kernel(nt), dim3(ns), dim3(nt), stage_lds(nt), fs, (const TileDesc *)ctx->d_tiles, ns, ctx->xcd_remap, a);
    });
    if (fork) HIP_TRY(hipEventRecord(ctx->ev_join, ctx->side));
    if (ng) timed_launch(ctx, ctx->stream, kClassGemm, [&] {
        if (ctx->form == PSTD_FORM_GEMM_BF16)
            hipLaunchKernelGGL(stage_gemm_kernel<__bf16>, dim3(ng), dim3(kGemmThreads), kGemmLdsBytes, ctx->stream, a,
                               ctx->d_gemm, ctx->ftab);
        else
            hipLaunchKernelGGL(stage_gemm_kernel<_Float16>, dim3(ng), dim3(kGemmThreads), kGemmLdsBytes, ctx->stream, a,
                               ctx->d_gemm, ctx->ftab);
    });
    if (fork) HIP_TRY(hipStreamWaitEvent(ctx->stream, ctx->ev_join, 0));
    if (ctx->p0_pass) {
        const MaxArgs mx{ctx->wmax, ctx->d_max_first, ctx->umax, ng ? 2 * ctx->n_scenes : 0};
        hipLaunchKernelGGL(p0_pass_kernel, dim3(mx.n + ctx->p0_first.back()), dim3(256), 0, ctx->stream, ctx->S(outi),
                           ctx->P0I(), ctx->d_p0_tiles, 1, mx);
    }
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) {
        ctx->err = std::string("stage launch: ") + hipGetErrorString(e);
        return PSTD_ERR_DEVICE;
    }
    return PSTD_OK;
}

int field_size(const pstd_plan_domain &d, int f) {
    switch (f) {
        case PSTD_FIELD_VX: return d.ny * (d.nx + 1);
        case PSTD_FIELD_VY: return (d.ny + 1) * d.nx;
        default: return d.nx * d.ny;
    }
}

// arena element offset of a field (p0 lives in the px slot of P0I)
long long field_off(const DomainDev &d, int f) {
    switch (f) {
        case PSTD_FIELD_VX: return d.base + d.f_vx;
        case PSTD_FIELD_VY: return d.base + d.f_vy;
        case PSTD_FIELD_PY: return d.base + d.f_py;
        default: return d.base + d.f_px;
    }
}

// P0I's slots of domain d (all domains: d < 0) from S1, or (px slots set) the
// transposed ones alone.
int launch_p0(pstd_ctx *ctx, int d, bool from_stage) {
    const int t0 = d < 0 ? 0 : ctx->p0_first[d], t1 = d < 0 ? ctx->p0_first.back() : ctx->p0_first[d + 1];
    hipLaunchKernelGGL(p0_pass_kernel, dim3(t1 - t0), dim3(256), 0, ctx->stream, ctx->S(1), ctx->P0I(),
                       ctx->d_p0_tiles + t0, from_stage ? 1 : 0, MaxArgs{});
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) {
        ctx->err = std::string("p0 launch: ") + hipGetErrorString(e);
        return PSTD_ERR_DEVICE;
    }
    return PSTD_OK;
}

int materialise_p0(pstd_ctx *ctx) {
    // P0I <- S1.px + S1.py for every domain (the current, stale p0)
    if (ctx->p0_explicit) return PSTD_OK;
    if (ctx->steps_done == 0) return PSTD_OK;
    if (!ctx->p0_pass) {
        const int rc = launch_p0(ctx, -1, true);
        if (rc) return rc;
    }
    ctx->p0_explicit = true;
    return PSTD_OK;
}

// Workgroups of turn_kernel for a rows x cols field.
unsigned turn_blocks(int rows, int cols) {
    return (unsigned)((rows + kP0Side - 1) / kP0Side) * (unsigned)((cols + kP0Side - 1) / kP0Side);
}

// Row-major rows x cols field <-> column-major: the host's and the device's
// layout of vy and py.
int launch_turn(pstd_ctx *ctx, const float *src, float *dst, int rows, int cols) {
    hipLaunchKernelGGL(turn_kernel<1>, dim3(turn_blocks(rows, cols)), dim3(256), 0, ctx->stream,
                       TurnFields<1>{{{src, dst, rows, cols, 0}}, 1});
    HIP_TRY(hipGetLastError());
    return PSTD_OK;
}

// The same for many fields.
constexpr int kTurnFields = 64;  // 2 KiB of kernel arguments
int launch_turns(pstd_ctx *ctx, const std::vector<TurnField> &fields) {
    for (size_t at = 0; at < fields.size(); at += kTurnFields) {
        TurnFields<kTurnFields> t;
        t.n = (int)std::min<size_t>(kTurnFields, fields.size() - at);
        unsigned blocks = 0;
        for (int k = 0; k < t.n; ++k) {
            t.f[k] = fields[at + k];
            t.f[k].first = blocks;
            blocks += turn_blocks(t.f[k].rows, t.f[k].cols);
        }
        hipLaunchKernelGGL(turn_kernel<kTurnFields>, dim3(blocks), dim3(256), 0, ctx->stream, t);
        HIP_TRY(hipGetLastError());
    }
    return PSTD_OK;
}

// The vy and py that the host wrote since the last time step, from S0 to TN.  A
// program writes the fields of all domains before it advances: they are turned
// together, in one launch per 64 fields (a launch and a wait per field took 12 us of
// the 26 us that writing a py of an 18-domain scene took, and made a run() of two
// steps of it 0.92 of the speed it has without).
int turn_written(pstd_ctx *ctx) {
    if (!ctx->any_written) return PSTD_OK;
    std::vector<TurnField> fields;
    for (size_t d = 0; d < ctx->doms.size(); ++d)
        for (int f : {PSTD_FIELD_VY, PSTD_FIELD_PY}) {
            if (!ctx->written[2 * d + (f == PSTD_FIELD_PY)]) continue;
            const pstd_plan_domain &p = ctx->plan_domains[d];
            const long long off = field_off(ctx->doms[d], f);
            fields.push_back({ctx->S(0) + off, ctx->TN() + off, field_size(p, f) / p.nx, p.nx, 0});
        }
    const int rc = launch_turns(ctx, fields);
    if (rc) return rc;
    std::fill(ctx->written.begin(), ctx->written.end(), 0);
    ctx->any_written = false;
    return PSTD_OK;
}

}  // namespace

extern "C" {

// Device address of `scratch` per device (the array's name is a host-side
// stand-in: kernels get this address).  Resolved once per device with that
// device current.
namespace {
std::mutex g_scratch_mu;
std::map<int, unsigned *> g_scratch;

int resolve_scratch(int device, unsigned **out) {
    std::lock_guard<std::mutex> lock(g_scratch_mu);
    auto it = g_scratch.find(device);
    if (it == g_scratch.end()) {
        void *ptr = nullptr;
        if (hipGetSymbolAddress(&ptr, HIP_SYMBOL(scratch)) != hipSuccess || !ptr) return PSTD_ERR_DEVICE;
        it = g_scratch.emplace(device, static_cast<unsigned *>(ptr)).first;
    }
    *out = it->second;
    return PSTD_OK;
}
}  // namespace

int pstd_ctx_create(int device, pstd_ctx **out) {
    if (!out) return PSTD_ERR_INVALID;
    *out = nullptr;
    int n = 0;
    if (hipGetDeviceCount(&n) != hipSuccess || n == 0) return PSTD_ERR_DEVICE;
    if (device < 0 || device >= n) return PSTD_ERR_INVALID;
    pstd_ctx *ctx = new pstd_ctx();
    ctx->device = device;
    if (hipSetDevice(device) != hipSuccess || hipStreamCreateWithFlags(&ctx->stream, hipStreamNonBlocking) != hipSuccess) {
        delete ctx;
        return PSTD_ERR_DEVICE;
    }
    // the side stream and its events (pstd_ctx_set_stage_overlap refuses to
    // turn the overlap on if one of them could not be created)
    if (hipStreamCreateWithFlags(&ctx->side, hipStreamNonBlocking) != hipSuccess) ctx->side = nullptr;
    if (hipEventCreateWithFlags(&ctx->ev_fork, hipEventDisableTiming) != hipSuccess) ctx->ev_fork = nullptr;
    if (hipEventCreateWithFlags(&ctx->ev_join, hipEventDisableTiming) != hipSuccess) ctx->ev_join = nullptr;
    // more than 64 KiB of LDS per workgroup: 512-thread stage blocks
    const hipFuncAttribute attr = hipFuncAttributeMaxDynamicSharedMemorySize;
    if (hipFuncSetAttribute((const void *)stage_kernel(512), attr, stage_lds(512)) != hipSuccess) {
        ctx->err = "cannot reserve LDS for the long-line kernels";
    }
    unsigned *sp = nullptr;
    if (resolve_scratch(device, &sp) != PSTD_OK) {
        (void)hipStreamDestroy(ctx->stream);
        delete ctx;
        return PSTD_ERR_DEVICE;
    }
    *out = ctx;
    return PSTD_OK;
}

void pstd_ctx_destroy(pstd_ctx *ctx) {
    if (!ctx) return;
    (void)hipSetDevice(ctx->device);
    if (ctx->stream) (void)hipStreamSynchronize(ctx->stream);
    ctx->release();
    if (ctx->side) (void)hipStreamSynchronize(ctx->side);
    if (ctx->ev_fork) (void)hipEventDestroy(ctx->ev_fork);
    if (ctx->ev_join) (void)hipEventDestroy(ctx->ev_join);
    if (ctx->side) (void)hipStreamDestroy(ctx->side);
    if (ctx->stream) (void)hipStreamDestroy(ctx->stream);
    give_pinned(ctx->pin);
    delete ctx;
}

const char *pstd_ctx_last_error(const pstd_ctx *ctx) { return ctx ? ctx->err.c_str() : "null context"; }

// Enqueues `chunk` time steps: 6 stage launches per step (the first stage of
// step s > 0 also samples step s-1 into sample slot base+s-1) and the sampling
// of the chunk's last step into slot base+chunk-1.
static int enqueue_steps(pstd_ctx *ctx, int chunk, int base = 0) {
    for (int s = 0; s < chunk; ++s) {
        for (int k = 0; k < 6; ++k) {
            int rc = launch_stage(ctx, k, s == 0 ? -1 : base + s - 1);
            if (rc) return rc;
            if (k == 0) ctx->p0_explicit = false;
        }
        if (ctx->n_si > 0) {
            // spectral receivers of this step, from its raw stage-5 output
            hipLaunchKernelGGL(si_line_kernel, dim3((ctx->n_si_lines + 3) / 4), dim3(256), 0, ctx->stream,
                               ctx->p0_pass ? ctx->P0I() : ctx->S(1), ctx->d_si_lines, ctx->n_si_lines,
                               ctx->p0_pass ? 0 : 1, ctx->d_si_coef, ctx->d_si_col);
            hipLaunchKernelGGL(si_point_kernel, dim3(ctx->n_si), dim3(64), 0, ctx->stream, ctx->d_si_col,
                               ctx->d_si_points, ctx->d_si_coef, ctx->d_samples, ctx->nrec, base + s);
            HIP_TRY(hipGetLastError());
        }
    }
    if (ctx->nrec > 0) {
        hipLaunchKernelGGL(receiver_kernel, dim3(1), dim3(64), 0, ctx->stream, ctx->S(1), ctx->d_cells, ctx->nrec,
                           ctx->d_samples, base + chunk - 1);
        HIP_TRY(hipGetLastError());
    }
    return PSTD_OK;
}

// The tile list for the current block size NT: a segment's lines in tiles of 2 P
// lines (P = NT / T pairs), passthrough fields in chunks.  The pairs (line0 + 2p,
// line0 + 2p + 1) are the same for every NT, so results do not depend on it.
static int upload_tiles(pstd_ctx *ctx) {
    const int nt = ctx->stage_threads();
    std::vector<TileDesc> tiles;
    // the longest tiles first, so that none of them starts last, but in the smallest
    // scenes, whose kinds of tiles stay mixed over the CUs.  (A batch of many lengths would
    // gain 3 % mixed, but the wavefront count is on the side of the single scenes that gain
    // 8 to 21 % sorted.)  Measured mixed / sorted, us
    // per stage: L-shape 8.1 / 8.2, rooms of 333, 141, 477 x 217 11.7 / 12.3 (11.0 / 11.0
    // with 8 values per thread), 1500 x 150 18.1 / 15.4, 900^2 22.1 / 19.5, 1268 x 303 20.1 /
    // 15.9, 1200^2 37.2 / 36.0, 1900^2 59.5 / 55.0, 4096^2 399 / 393, twelve scenes 91.0 / 93.6
    long long waves = 0;
    for (const TileDesc &g : ctx->fft_segs)
        if (g.kind == 0) waves += (long long)g.count / 2 * (g.F / ctx->values(g.F)) / 64;
    std::vector<int> order(ctx->fft_segs.size());
    for (size_t k = 0; k < order.size(); ++k) order[k] = (int)k;
    auto length = [&](int k) { return ctx->fft_segs[k].kind == 0 ? ctx->fft_segs[k].F : 0; };
    if (waves > 2048) std::stable_sort(order.begin(), order.end(), [&](int x, int y) { return length(x) > length(y); });
    for (int k : order) {
        const TileDesc &g = ctx->fft_segs[k];
        const int per = g.kind == 0 ? 2 * nt / (g.F / ctx->values(g.F)) : kPassChunk;
        for (int l = 0; l < g.count; l += per) {
            tiles.push_back(g);
            tiles.back().line0 = g.line0 + l;
            tiles.back().count = std::min(per, g.count - l);
        }
    }
    ctx->n_tiles = (int)tiles.size();
    HIP_TRY(hipStreamSynchronize(ctx->stream));
    if (!ctx->tiles_gemm.empty()) {
        // maxima slots: a group (scene, class) after the other
        const int groups = 2 * ctx->n_scenes;
        auto group = [](const TileDesc &t) { return 2 * t.scene + (t.vel ? 0 : 1); };
        std::vector<int2> first(groups + 1, make_int2(0, 0));
        auto writes = [](const TileDesc &t) { return t.kind != 2; };  // (receivers store no maximum)
        for (const TileDesc &t : tiles)
            if (writes(t)) first[group(t) + 1].x += nt / 64;
        for (int i = 0; i < groups; ++i) first[i + 1].x += first[i].x;
        std::vector<int2> next = first;
        for (TileDesc &t : tiles) {
            if (!writes(t)) continue;
            int &n = next[group(t)].x;
            t.slot = n;
            n += nt / 64;
        }
        const int base = first[groups].x;
        for (int i = 0; i <= groups; ++i) first[i].y = base + ctx->gemm_first[i];
        std::vector<GemmTile> gemm = ctx->tiles_gemm;
        for (GemmTile &t : gemm) t.t.slot += base;
        if (ctx->wmax) HIP_TRY(hipFree(ctx->wmax));
        ctx->wmax = nullptr;
        HIP_TRY(hipMalloc(&ctx->wmax, (size_t)(base + ctx->gemm_first.back()) * sizeof(float)));
        HIP_TRY(hipMemcpyAsync(ctx->d_gemm, gemm.data(), gemm.size() * sizeof(GemmTile), hipMemcpyHostToDevice, ctx->stream));
        HIP_TRY(hipMemcpyAsync(ctx->d_max_first, first.data(), first.size() * sizeof(int2), hipMemcpyHostToDevice,
                               ctx->stream));
        HIP_TRY(hipStreamSynchronize(ctx->stream));
    }
    if (ctx->d_tiles) HIP_TRY(hipFree(ctx->d_tiles));
    ctx->d_tiles = nullptr;
    HIP_TRY(hipMalloc(&ctx->d_tiles, std::max<size_t>(1, tiles.size()) * sizeof(TileDesc)));
    if (!tiles.empty()) {
        HIP_TRY(hipMemcpyAsync(ctx->d_tiles, tiles.data(), tiles.size() * sizeof(TileDesc), hipMemcpyHostToDevice,
                               ctx->stream));
        HIP_TRY(hipStreamSynchronize(ctx->stream));
    }
    return PSTD_OK;
}

// Launch-shape autotuner.  Times every (block size, tile order) candidate on the
// freshly uploaded (all-zero) state and keeps the fastest.  Zero fields stay
// exactly zero under the update, and the arenas are cleared again afterwards, so
// tuning leaves no trace in the results.
// The autotuner's choices, per (device, plan signature): a later context with a
// plan of the same launch geometry on the same device takes the choice and
// runs no trials.
struct TuneChoice {
    int xcd_remap, small_nt;
    float stage_ms;
};
std::mutex g_tune_mu;
std::map<std::pair<int, uint64_t>, TuneChoice> g_tune;
// PSTD_FORM_AUTO's choice per (device, signature of the plan's FFT-form upload)
std::map<std::pair<int, uint64_t>, int> g_form;

// FNV-1a over what the launches' timing depends on: the form, the scene count,
// the paths that the plan's sizes chose, every tile's line class, line count and
// direction, and the arena size.  Two plans that hash alike launch the same grids of
// the same kernels.
uint64_t plan_signature(const pstd_ctx *ctx) {
    uint64_t h = 1469598103934665603ull;
    auto mix = [&h](long long v) {
        for (int i = 0; i < 8; ++i) {
            h ^= (uint64_t)((v >> (8 * i)) & 0xff);
            h *= 1099511628211ull;
        }
    };
    mix(ctx->form);
    mix(ctx->n_scenes);
    mix(ctx->p0_pass);
    mix(ctx->f8);
    mix((long long)ctx->arena_floats);
    mix((long long)ctx->fft_segs.size());
    for (const TileDesc &t : ctx->fft_segs) {
        mix(t.kind);
        mix(t.F);
        mix(t.count);
        mix(t.dir);
        mix(t.vel);
        mix(t.n_out);
    }
    mix((long long)ctx->tiles_gemm.size());
    for (const GemmTile &g : ctx->tiles_gemm) {
        mix(g.t.dir);
        mix(g.t.vel);
        mix(g.t.count);
        mix(g.n_rows);
        mix(g.k_pad);
    }
    return h;
}

// The block size an earlier plan of the same signature was tuned to, before the
// tile list is cut for it.
static void take_tuned_threads(pstd_ctx *ctx) {
    std::lock_guard<std::mutex> lock(g_tune_mu);
    auto it = g_tune.find({ctx->device, plan_signature(ctx)});
    if (it != g_tune.end()) ctx->small_nt = it->second.small_nt;
}

static int autotune(pstd_ctx *ctx) {
    const std::pair<int, uint64_t> key(ctx->device, plan_signature(ctx));
    ctx->trial_steps = 0;
    ctx->tune_cached = false;
    {
        std::lock_guard<std::mutex> lock(g_tune_mu);
        auto it = g_tune.find(key);
        if (it != g_tune.end()) {
            ctx->xcd_remap = it->second.xcd_remap;
            ctx->tuned_stage_ms = it->second.stage_ms;
            ctx->tune_cached = true;
            if (it->second.small_nt != ctx->small_nt) {
                ctx->small_nt = it->second.small_nt;
                const int rc = upload_tiles(ctx);
                if (rc) return rc;
            }
            HIP_TRY(hipStreamSynchronize(ctx->stream));
            return PSTD_OK;
        }
    }
    hipEvent_t e0 = nullptr, e1 = nullptr;
    HIP_TRY(hipEventCreate(&e0));
    HIP_TRY(hipEventCreate(&e1));
    // one warm-up step, then GPU ms of n steps
    int n = 3;
    auto time_steps = [&](float &ms) -> int {
        ctx->trial_steps += 1 + n;
        int rc = enqueue_steps(ctx, 1);
        if (rc == PSTD_OK && hipEventRecord(e0, ctx->stream) != hipSuccess) rc = PSTD_ERR_DEVICE;
        if (rc == PSTD_OK) rc = enqueue_steps(ctx, n);
        if (rc == PSTD_OK && hipEventRecord(e1, ctx->stream) != hipSuccess) rc = PSTD_ERR_DEVICE;
        if (rc == PSTD_OK && hipEventSynchronize(e1) != hipSuccess) rc = PSTD_ERR_DEVICE;
        if (rc == PSTD_OK && hipEventElapsedTime(&ms, e0, e1) != hipSuccess) rc = PSTD_ERR_DEVICE;
        return rc;
    };
    float best = 0;
    int bi = 0, bnt = ctx->small_nt, rc = PSTD_OK;
    bool first = true;
    {
        // small (latency-bound) scenes get more timed steps per candidate
        // (about 2 ms of GPU time each), so that run-to-run noise does not
        // pick the shape; large ones keep 3
        float ms = 0;
        rc = time_steps(ms);
        if (rc == PSTD_OK && ms > 0.f) n = std::min(50, std::max(3, (int)std::ceil(2.0f / (ms / 3.0f))));
    }
    // block sizes, where the lines leave a choice
    std::vector<int> nts = {ctx->small_nt};
    if (ctx->small_fmax > 0 && ctx->fmax <= 2048)
        for (int nt : {128, 256})
            if (nt != ctx->small_nt && (nt >= 256 || ctx->small_fmax <= 1024)) nts.push_back(nt);
    for (int nt : nts) {
        if (rc != PSTD_OK) break;
        if (nt != ctx->small_nt) {
            ctx->small_nt = nt;
            rc = upload_tiles(ctx);
        }
        for (int c = 1; c >= 0 && rc == PSTD_OK; --c) {
            ctx->xcd_remap = c;
            float ms = 0;
            rc = time_steps(ms);
            if (rc == PSTD_OK && (first || ms < best)) {
                best = ms;
                bi = c;
                bnt = nt;
                first = false;
            }
        }
    }
    if (rc == PSTD_OK) {
        ctx->xcd_remap = bi;
        if (bnt != ctx->small_nt) {
            ctx->small_nt = bnt;
            rc = upload_tiles(ctx);
        }
    }
    (void)hipEventDestroy(e0);
    (void)hipEventDestroy(e1);
    if (rc) {
        if (ctx->err.empty()) ctx->err = "autotune: HIP event failure";
        return rc;
    }
    ctx->tuned_stage_ms = best / (6.0 * n);
    {
        std::lock_guard<std::mutex> lock(g_tune_mu);
        g_tune[key] = {ctx->xcd_remap, ctx->small_nt, ctx->tuned_stage_ms};
    }
    HIP_TRY(hipMemsetAsync(ctx->arena, 0, 4 * (size_t)ctx->arena_floats * sizeof(float), ctx->stream));
    if (ctx->umax) HIP_TRY(hipMemsetAsync(ctx->umax, 0, 2 * (size_t)ctx->n_scenes * sizeof(unsigned), ctx->stream));
    HIP_TRY(hipStreamSynchronize(ctx->stream));
    ctx->steps_done = 0;
    ctx->p0_explicit = true;
    return PSTD_OK;
}

// 16-bit parts of the GEMM form, from double, rounded to nearest even.
static uint16_t to_f16_bits(double v) {
    const _Float16 h = (_Float16)v;
    uint16_t b;
    std::memcpy(&b, &h, 2);
    return b;
}
static double from_f16_bits(uint16_t b) {
    _Float16 h;
    std::memcpy(&h, &b, 2);
    return (double)h;
}
static uint16_t to_bf16_bits(double v) {
    if (v == 0.0) return 0;
    int e = 0;
    const double m = std::frexp(v, &e);                        // |m| in [0.5, 1)
    const double q = std::nearbyint(std::ldexp(m, 8));         // 8 significant bits, ties to even
    const float f = (float)std::ldexp(q, e - 8);               // exact in float
    uint32_t u;
    std::memcpy(&u, &f, 4);
    return (uint16_t)(u >> 16);
}
static double from_bf16_bits(uint16_t b) {
    const uint32_t u = (uint32_t)b << 16;
    float f;
    std::memcpy(&f, &u, 4);
    return (double)f;
}

// Whether a segment runs in the GEMM form: its lines and outputs fill blocks of
// 128 lines x 256 outputs at least to 3/4 (thin PML strips keep the FFT form).
static bool gemm_fills(int lines, int n_g) {
    constexpr int kFillN = 256;
    const double cap = (double)((lines + kGL - 1) / kGL * kGL) * (double)((n_g + kFillN - 1) / kFillN * kFillN);
    return 4.0 * lines * (double)n_g >= 3.0 * cap;
}

// GEMM form of one segment: its derivative matrix (built once per distinct
// segment shape and stencil, split into 16-bit hi + lo parts of D * 2^d_exp;
// for pressure lines the last row kept apart in FP32 for the dot product) and
// its 128-line x 128-output tiles.
static int add_gemm_tiles(pstd_ctx *ctx, const pstd_plan_desc *plan, const pstd_plan_segment &s, const TileDesc &g,
                          std::vector<uint16_t> &dmat, std::vector<float> &ftab,
                          std::map<std::string, std::tuple<long long, int, int>> &dcache) {
    pstdamd::SegmentShape sh{g.F, s.table_len, s.field, (double)plan->dx, s.wlen, g.n_main, (double)plan->patch_error,
                             (double)s.c_side1, (double)s.c_main1, (double)s.c_side2, (double)s.c_main2};
    const int K = sh.K(), n_out = sh.n_out();
    const bool dot_row = s.field == 0;  // n + 1 outputs: the last one as an FP32 dot product
    const int n_g = n_out - (dot_row ? 1 : 0);
    const int k_pad = (K + kGK - 1) / kGK * kGK, n_rows = (n_g + kGN - 1) / kGN * kGN, nch = k_pad / kGK;
    const bool bf16 = ctx->form == PSTD_FORM_GEMM_BF16;
    char key[256];
    std::snprintf(key, sizeof key, "%d/%d/%d/%d/%d/%a/%a/%a/%a", sh.F, sh.table_len, sh.field, sh.w, sh.n_main,
                  sh.c_s1, sh.c_m1, sh.c_s2, sh.c_m2);
    auto it = dcache.find(key);
    if (it == dcache.end()) {
        std::vector<double> D;
        try {
            D = pstdamd::derivative_matrix(sh);
        } catch (const std::exception &e) {
            ctx->err = std::string("GEMM form: ") + e.what();
            return PSTD_ERR_INVALID;
        }
        double dm = 0;
        for (int i = 0; i < n_g; ++i)
            for (int k = 0; k < K; ++k) dm = std::max(dm, std::fabs(D[(size_t)i * K + k]));
        const int d_exp = dm > 0 ? 14 - std::ilogb(dm) : 0;
        // for every 128-output block, its chunks (gemm_d_at)
        const long long hi = (long long)dmat.size();
        dmat.resize(dmat.size() + (size_t)(n_rows / kGN) * nch * kGemmDChunk, 0);
        for (int i = 0; i < n_g; ++i)
            for (int k = 0; k < K; ++k) {
                const double v = std::ldexp(D[(size_t)i * K + k], d_exp);
                const uint16_t h = bf16 ? to_bf16_bits(v) : to_f16_bits(v);
                const double hv = bf16 ? from_bf16_bits(h) : from_f16_bits(h);
                const size_t tile = hi + (size_t)(i / kGN) * nch * kGemmDChunk;
                dmat[tile + gemm_d_at(i % kGN, k, 0)] = h;
                dmat[tile + gemm_d_at(i % kGN, k, 1)] = bf16 ? to_bf16_bits(v - hv) : to_f16_bits(v - hv);
            }
        int dot_off = -1;
        if (dot_row) {
            dot_off = (int)ftab.size();
            for (int k = 0; k < K; ++k) ftab.push_back((float)D[(size_t)(n_out - 1) * K + k]);
        }
        it = dcache.emplace(key, std::make_tuple(hi, d_exp, dot_off)).first;
    }
    const long long d_base = std::get<0>(it->second), d_len = (long long)nch * kGemmDChunk;
    ctx->gemm_flops += 3.0 * 2.0 * K * (double)n_out * (s.line_end - s.line_begin);
    ctx->gemm_cells += (long long)n_out * (s.line_end - s.line_begin);
    for (int l = s.line_begin; l < s.line_end; l += kGL) {
        GemmTile gt{};
        gt.t = g;
        gt.t.kind = 3;
        gt.t.line0 = l;
        gt.t.count = std::min(kGL, s.line_end - l);
        gt.d_len = d_len;
        gt.n_rows = n_rows;
        gt.k_pad = k_pad;
        gt.n_g = n_g;
        gt.d_exp = std::get<1>(it->second);
        gt.K = K;
        for (int n0 = 0; n0 < n_g; n0 += kGN) {
            gt.n0 = n0;
            gt.d_img = d_base + (long long)(n0 / kGN) * d_len;
            gt.dot_off = n0 + kGN >= n_g ? std::get<2>(it->second) : -1;  // the last output tile
            ctx->tiles_gemm.push_back(gt);
        }
    }
    return PSTD_OK;
}

// dom_scene: scene of every domain (a batch of scenes), or nullptr (one scene).
// Line jobs and weights of the spectral receivers (Receiver::compute_with_si,
// kernel/core/Receiver.cpp:85-121): for each, the Y pressure segment of its
// domain through its column gives the Y line (neighbours, stencil, window);
// every row of the domain and the w window rows of each Y neighbour are
// shifted along X with the X pressure segment holding that row; the weights
// are rows of the segments' line operators with the shift filter
// (plan_tables.h), rounded once to float.
static int build_spectral_receivers(pstd_ctx *ctx, const pstd_plan_desc *plan) {
    std::vector<SILine> lines;
    std::vector<SIPoint> points;
    std::vector<float> coef;
    int col_total = 0;
    std::map<std::pair<int, int>, int> row_cache;  // (segment, output column) -> weights, per receiver
    auto find_segment = [&](int dom, int dir, int line) -> int {
        for (int k = 0; k < plan->n_segments; ++k) {
            const pstd_plan_segment &s = plan->segments[k];
            if (s.domain == dom && s.direction == dir && s.field == 0 && s.line_begin <= line && line < s.line_end)
                return k;
        }
        return -1;
    };
    auto shape_of = [&](const pstd_plan_segment &s) {
        const DomainDev &d = ctx->doms[s.domain];
        const int n = s.direction == 0 ? d.nx : d.ny;
        return pstdamd::SegmentShape{next_pow2(n + 2 * s.wlen), s.table_len, 0, (double)plan->dx, s.wlen, n,
                                     (double)plan->patch_error, (double)s.c_side1, (double)s.c_main1,
                                     (double)s.c_side2, (double)s.c_main2};
    };
    auto add_weights = [&](const pstd_plan_segment &s, double offset, int out) {
        const pstdamd::SegmentShape sh = shape_of(s);
        const std::vector<double> row = pstdamd::operator_row(sh, pstdamd::shift_filter(sh.F, sh.table_len, offset), out);
        const int at = (int)coef.size();
        for (double v : row) coef.push_back((float)v);
        return at;
    };
    for (int r = 0; r < plan->n_receivers; ++r) {
        const pstd_plan_receiver &rc = plan->receivers[r];
        if (!rc.spectral) continue;
        if (!(rc.offset_x >= 0.f && rc.offset_x < 1.f && rc.offset_y >= 0.f && rc.offset_y < 1.f)) {
            ctx->err = "spectral receiver " + std::to_string(r) + ": offsets outside [0, 1)";
            return PSTD_ERR_INVALID;
        }
        const DomainDev &c = ctx->doms[rc.domain];
        const int cx = rc.index % c.nx, cy = rc.index / c.nx;
        const int ky = find_segment(rc.domain, 1, cx);
        if (ky < 0) {
            ctx->err = "spectral receiver " + std::to_string(r) + ": no Y pressure segment through its column";
            return PSTD_ERR_INVALID;
        }
        const pstd_plan_segment &sy = plan->segments[ky];
        const int w = sy.wlen, col0 = col_total;
        row_cache.clear();
        // the rows to shift along X: (domain, row, output column, column buffer element)
        struct Row {
            int dom, row, out, dst;
        };
        std::vector<Row> rows;
        for (int y = 0; y < c.ny; ++y) rows.push_back({rc.domain, y, cx, col0 + w + y});
        if (sy.side1 >= 0) {
            const DomainDev &n1 = ctx->doms[sy.side1];
            for (int j = 0; j < w; ++j) rows.push_back({sy.side1, n1.ny - w + j, cx + sy.side1_offset, col0 + j});
        }
        if (sy.side2 >= 0)
            for (int j = 0; j < w; ++j) rows.push_back({sy.side2, j, cx + sy.side2_offset, col0 + w + c.ny + j});
        for (const Row &q : rows) {
            const int kx = find_segment(q.dom, 0, q.row);
            if (kx < 0) {
                ctx->err = "spectral receiver " + std::to_string(r) + ": domain " + std::to_string(q.dom) +
                           " has no X pressure segment through row " + std::to_string(q.row);
                return PSTD_ERR_INVALID;
            }
            const pstd_plan_segment &sx = plan->segments[kx];
            const DomainDev &d = ctx->doms[q.dom];
            if (q.out < 0 || q.out >= d.nx) {
                ctx->err = "spectral receiver " + std::to_string(r) + ": column outside a neighbour";
                return PSTD_ERR_INVALID;
            }
            auto it = row_cache.find({kx, q.out});
            if (it == row_cache.end()) {
                int at;
                try {
                    at = add_weights(sx, (double)rc.offset_x, q.out);
                } catch (const std::exception &e) {
                    ctx->err = std::string("spectral receiver: ") + e.what();
                    return PSTD_ERR_INVALID;
                }
                it = row_cache.emplace(std::make_pair(kx, q.out), at).first;
            }
            SILine L{};
            L.m_px = d.base + d.f_px + (long long)q.row * d.nx;
            L.m_py = d.base + d.f_py + q.row;
            L.m_ld = d.ny;
            L.s1_px = L.s1_py = L.s2_px = L.s2_py = -1;
            if (sx.side1 >= 0) {
                const DomainDev &n = ctx->doms[sx.side1];
                const int row = q.row + sx.side1_offset, col = n.nx - sx.wlen;
                L.s1_px = n.base + n.f_px + (long long)row * n.nx + col;
                L.s1_py = n.base + n.f_py + (long long)col * n.ny + row;
                L.s1_ld = n.ny;
            }
            if (sx.side2 >= 0) {
                const DomainDev &n = ctx->doms[sx.side2];
                const int row = q.row + sx.side2_offset;
                L.s2_px = n.base + n.f_px + (long long)row * n.nx;
                L.s2_py = n.base + n.f_py + row;
                L.s2_ld = n.ny;
            }
            L.n_main = d.nx;
            L.w = sx.wlen;
            L.coef = it->second;
            L.dst = q.dst;
            lines.push_back(L);
        }
        SIPoint P{};
        try {
            P.coef = add_weights(sy, (double)rc.offset_y, cy);
        } catch (const std::exception &e) {
            ctx->err = std::string("spectral receiver: ") + e.what();
            return PSTD_ERR_INVALID;
        }
        P.K = c.ny + 2 * w;
        P.col = col0;
        P.rec = r;
        points.push_back(P);
        col_total += P.K;
    }
    if (points.empty()) return PSTD_OK;
    std::stable_sort(lines.begin(), lines.end(), [](const SILine &x, const SILine &y) { return x.m_px < y.m_px; });
    HIP_TRY(hipMalloc(&ctx->d_si_lines, lines.size() * sizeof(SILine)));
    HIP_TRY(hipMalloc(&ctx->d_si_points, points.size() * sizeof(SIPoint)));
    HIP_TRY(hipMalloc(&ctx->d_si_coef, coef.size() * sizeof(float)));
    HIP_TRY(hipMalloc(&ctx->d_si_col, (size_t)col_total * sizeof(float)));
    HIP_TRY(hipMemcpyAsync(ctx->d_si_lines, lines.data(), lines.size() * sizeof(SILine), hipMemcpyHostToDevice,
                           ctx->stream));
    HIP_TRY(hipMemcpyAsync(ctx->d_si_points, points.data(), points.size() * sizeof(SIPoint), hipMemcpyHostToDevice,
                           ctx->stream));
    HIP_TRY(hipMemcpyAsync(ctx->d_si_coef, coef.data(), coef.size() * sizeof(float), hipMemcpyHostToDevice,
                           ctx->stream));
    // window rows of missing neighbours are never written: zeros
    HIP_TRY(hipMemsetAsync(ctx->d_si_col, 0, (size_t)col_total * sizeof(float), ctx->stream));
    ctx->n_si_lines = (int)lines.size();
    ctx->n_si = (int)points.size();
    return PSTD_OK;
}

static int upload_impl(pstd_ctx *ctx, const pstd_plan_desc *plan, const std::vector<int> *dom_scene = nullptr) {
    if (plan->n_domains < 0) {
        ctx->err = "negative number of domains";
        return PSTD_ERR_INVALID;
    }
    HIP_TRY(hipSetDevice(ctx->device));
    HIP_TRY(hipStreamSynchronize(ctx->stream));
    ctx->release();
    ctx->doms.clear();
    ctx->small_fmax = 0;
    ctx->fmax = 0;
    ctx->small_nt = 256;
    ctx->fft_segs.clear();
    ctx->tiles_gemm.clear();
    ctx->max_ranges.clear();
    ctx->n_scenes = 1;
    if (dom_scene)
        for (int sc : *dom_scene) ctx->n_scenes = std::max(ctx->n_scenes, sc + 1);
    auto scene_of = [&](int d) { return dom_scene ? (*dom_scene)[d] : 0; };
    ctx->gemm_flops = 0;
    ctx->gemm_cells = 0;
    ctx->plan_domains.assign(plan->domains, plan->domains + plan->n_domains);
    ctx->written.assign(2 * (size_t)plan->n_domains, 0);
    ctx->any_written = false;
    // arena layout: one block per domain (vx, vy, px, py), 256 B aligned
    long long off = kLead;  // zeros before the first block
    auto align = [](long long v) { return (v + 63) & ~63LL; };
    for (int i = 0; i < plan->n_domains; ++i) {
        const pstd_plan_domain &p = plan->domains[i];
        if (p.nx <= 0 || p.ny <= 0) {
            ctx->err = "domain with empty extent";
            return PSTD_ERR_INVALID;
        }
        // (four times the cells of the largest extents do not fit 64 bits)
        const long long cells = (long long)p.nx * p.ny;
        if (cells > kMaxDomainFloats / 4 || 4 * cells + p.nx + p.ny + 4 * 64 > kMaxDomainFloats) {
            ctx->err = "domain of " + std::to_string(cells) + " cells exceeds one buffer block";
            return PSTD_ERR_UNSUPPORTED;
        }
        DomainDev d{};
        d.nx = p.nx;
        d.ny = p.ny;
        d.rho = p.rho;
        d.is_pml = p.is_pml;
        d.base = off;
        long long f = 0;
        d.f_vx = (int)f;
        f = align(f + (long long)p.ny * (p.nx + 1));
        d.f_vy = (int)f;
        f = align(f + (long long)(p.ny + 1) * p.nx);
        d.f_px = (int)f;
        f = align(f + cells);
        d.f_py = (int)f;
        f = align(f + cells + 1);  // a spare float after py (8-byte accesses of line pairs)
        d.size = (int)f;
        off += f;
        ctx->doms.push_back(d);
    }
    ctx->arena_floats = (size_t)(off + kLead);  // a matrix tile reads up to 3 floats past a block
    ctx->dt = plan->dt;
    ctx->c1 = plan->c1;
    for (int k = 0; k < 6; ++k) ctx->alpha[k] = plan->rk_alpha[k];
    // device plan cache: filters, twiddles, windows
    std::vector<float2> ctab;
    std::vector<float> ftab;
    std::map<std::tuple<int, int, int>, int> filt_cache;
    std::map<int, int> tw_cache;
    std::map<int, int> win_cache;
    const double dx = plan->dx;
    // source addressing of a domain's derivative input for (direction, field):
    // pressure reads p0 (px slot row-major for X, py slot column-major for Y; on
    // the fly plus the other field across its layout), velocity vx (X) or vy (Y)
    // (field offsets within the domain block)
    auto src_addr = [&](const DomainDev &d, int dir, int field, int &a, int &b, int &ls, int &bp) {
        const int n = dir == 0 ? d.nx : d.ny;
        if (field == 0) {
            a = dir == 0 ? d.f_px : d.f_py;
            b = dir == 0 ? d.f_py : d.f_px;
            ls = n;
            bp = dir == 0 ? d.ny : d.nx;
        } else {
            a = b = dir == 0 ? d.f_vx : d.f_vy;
            ls = n + 1;
            bp = 0;
        }
    };
    long long strided_bytes = 0, pass_cells = 0;  // p0 on the fly, or by the pass
    for (const DomainDev &d : ctx->doms) pass_cells += (long long)d.nx * d.ny;
    std::vector<std::vector<char>> covered(plan->n_domains, std::vector<char>(4, 0));
    std::vector<uint16_t> dmat;
    std::map<std::string, std::tuple<long long, int, int>> dcache;  // matrix key -> (hi offset, d_exp, dot row)
    // the segments as tiles' records (without tables yet), each checked before anything
    // is computed from it
    struct Line {
        const pstd_plan_segment *s;
        TileDesc g;
        bool gemm;
    };
    std::vector<Line> checked;
    long long waves = 0;
    for (int si = 0; si < plan->n_segments; ++si) {
        const pstd_plan_segment &s = plan->segments[si];
        if (s.domain < 0 || s.domain >= plan->n_domains || s.side1 >= plan->n_domains || s.side2 >= plan->n_domains ||
            (s.direction != 0 && s.direction != 1) || (s.field != 0 && s.field != 1) || s.wlen <= 0) {
            ctx->err = "invalid segment " + std::to_string(si);
            return PSTD_ERR_INVALID;
        }
        if (s.wlen > 32) {
            ctx->err = "window half-length " + std::to_string(s.wlen) + " above 32 (patch error above ~72 dB)";
            return PSTD_ERR_UNSUPPORTED;
        }
        const DomainDev &dm = ctx->doms[s.domain];
        const int n = s.direction == 0 ? dm.nx : dm.ny;
        const int nlines = s.direction == 0 ? dm.ny : dm.nx;
        if (s.line_begin < 0 || s.line_end > nlines || s.line_begin >= s.line_end) {
            ctx->err = "segment line range outside its domain";
            return PSTD_ERR_INVALID;
        }
        TileDesc g{};
        g.kind = 0;
        g.dir = s.direction;
        g.vel = s.field;
        g.wlen = s.wlen;
        g.n_main = s.field == 0 ? n : n + 1;
        g.n_out = s.field == 0 ? n + 1 : n;
        g.F = next_pow2(g.n_main + 2 * s.wlen);
        g.c_s1 = s.c_side1;
        g.c_m1 = s.c_main1;
        g.c_s2 = s.c_side2;
        g.c_m2 = s.c_main2;
        // update factor of Solver::update_field_values (kernel/Solver.cpp:174-181),
        // in double: 1/rho for the velocity fields, rho*c1^2 for the pressure fields
        g.coef = s.field == 0 ? (float)(1.0 / (double)dm.rho) : (float)((double)dm.rho * plan->c1 * plan->c1);
        g.is_pml = dm.is_pml;
        g.m_dom = g.s1_dom = g.s2_dom = dm.base;
        g.m_size = g.s1_size = g.s2_size = dm.size;
        if (g.F < 128 || g.F > 8192) {
            ctx->err = "FFT length " + std::to_string(g.F) + " outside 128..8192";
            return PSTD_ERR_UNSUPPORTED;
        }
        if (s.table_len < g.F || (s.table_len & (s.table_len - 1))) {
            ctx->err = "wavenumber table shorter than the FFT length";
            return PSTD_ERR_INVALID;
        }
        if (s.wlen > n) {
            ctx->err = "window longer than the domain";
            return PSTD_ERR_INVALID;
        }
        src_addr(dm, s.direction, s.field, g.m_a, g.m_b, g.m_ls, g.m_bp);
        g.s1_len = g.s2_len = -1;
        // neighbour bounds: lines and halo columns must exist in the neighbour
        for (int side = 0; side < 2; ++side) {
            int nb = side == 0 ? s.side1 : s.side2;
            const long long o = side == 0 ? s.side1_offset : s.side2_offset;  // a line + any 32-bit offset
            if (nb < 0) continue;
            const DomainDev &dn = ctx->doms[nb];
            int nlen = (s.direction == 0 ? dn.nx : dn.ny) + (s.field == 1 ? 1 : 0);
            int nlin = s.direction == 0 ? dn.ny : dn.nx;
            if (s.line_begin + o < 0 || s.line_end + o > nlin || nlen < s.wlen + (s.field == 1 ? 1 : 0)) {
                ctx->err = "segment reads outside its neighbour domain";
                return PSTD_ERR_INVALID;
            }
            if (side == 0) {
                src_addr(dn, s.direction, s.field, g.s1_a, g.s1_b, g.s1_ls, g.s1_bp);
                g.s1_line = (int)o;
                g.s1_len = nlen;
                g.s1_dom = dn.base;
                g.s1_size = dn.size;
            } else {
                src_addr(dn, s.direction, s.field, g.s2_a, g.s2_b, g.s2_ls, g.s2_bp);
                g.s2_line = (int)o;
                g.s2_len = nlen;
                g.s2_dom = dn.base;
                g.s2_size = dn.size;
            }
        }
        if (s.interp_only) {
            if (s.direction != 0 || s.field != 0) {
                ctx->err = "interpolation-only segment " + std::to_string(si) + " is not an X pressure segment";
                return PSTD_ERR_INVALID;
            }
            continue;  // read by the spectral receivers only
        }
        // output field: X pressure -> vx, X velocity -> px, Y pressure -> vy, Y velocity -> py
        g.o_f = s.direction == 0 ? (s.field == 0 ? dm.f_vx : dm.f_px) : (s.field == 0 ? dm.f_vy : dm.f_py);
        g.o_ls = s.field == 0 ? n + 1 : n;
        covered[s.domain][s.direction == 0 ? (s.field == 0 ? 2 : 0) : (s.field == 0 ? 3 : 1)] = 1;
        g.scene = scene_of(s.domain);
        if (s.field == 0) strided_bytes += 4LL * (s.line_end - s.line_begin) * n * strided_factor(g.F);
        g.line0 = s.line_begin;
        g.count = s.line_end - s.line_begin;
        // GEMM form: segments that fill the 128 x 256 tiles at least to 3/4
        // become GEMM tiles; thin ones (PML strips) stay FFT tiles
        const bool gemm = (ctx->form == PSTD_FORM_GEMM_F16 || ctx->form == PSTD_FORM_GEMM_BF16) &&
                          gemm_fills(g.count, s.field == 0 ? g.n_out - 1 : g.n_out);
        // of the lines this plan's stage launch runs
        if (!gemm) waves += (long long)g.count / 2 * (g.F / fft_values(g.F)) / 64;
        checked.push_back({&s, g, gemm});
    }
    ctx->f8 = waves <= kFewWaves ? 2048 : 512;
    for (Line &l : checked) {
        const pstd_plan_segment &s = *l.s;
        TileDesc &g = l.g;
        auto fk = std::make_tuple(g.F, s.table_len, s.field);
        auto it = filt_cache.find(fk);
        if (it == filt_cache.end()) {
            std::vector<float2> h;
            build_filter(g.F, s.table_len, s.field, dx, ctx->values(g.F), h);
            it = filt_cache.emplace(fk, (int)ctab.size()).first;
            ctab.insert(ctab.end(), h.begin(), h.end());
        }
        g.h_off = it->second;
        auto tt = tw_cache.find(g.F);
        if (tt == tw_cache.end()) {
            std::vector<float2> tw;
            build_twiddles(g.F, tw);
            tt = tw_cache.emplace(g.F, (int)ctab.size()).first;
            ctab.insert(ctab.end(), tw.begin(), tw.end());
        }
        g.tw_off = tt->second;
        auto wt = win_cache.find(s.wlen);
        if (wt == win_cache.end()) {
            std::vector<float> w;
            build_window(s.wlen, (int)plan->patch_error, w);
            wt = win_cache.emplace(s.wlen, (int)ftab.size()).first;
            ftab.insert(ftab.end(), w.begin(), w.end());
        }
        g.win_off = wt->second;
        if (l.gemm) {
            int rc = add_gemm_tiles(ctx, plan, s, g, dmat, ftab, dcache);
            if (rc) return rc;
            continue;
        }
        ctx->fmax = std::max(ctx->fmax, g.F);
        if (g.F <= 2048) ctx->small_fmax = std::max(ctx->small_fmax, g.F);
        ctx->fft_segs.push_back(g);
    }
    // passthrough tiles for fields no segment updates (rigid domains, directions
    // openPSTD does not update).  covered[] index: 0 px, 1 py, 2 vx, 3 vy
    for (int i = 0; i < plan->n_domains; ++i) {
        const DomainDev &d = ctx->doms[i];
        const int offs[4] = {d.f_px, d.f_py, d.f_vx, d.f_vy};
        const int sizes[4] = {d.nx * d.ny, d.nx * d.ny, d.ny * (d.nx + 1), (d.ny + 1) * d.nx};
        for (int f = 0; f < 4; ++f) {
            if (covered[i][f]) continue;
            TileDesc t{};
            t.kind = 1;
            t.count = sizes[f];
            t.m_dom = d.base;
            t.m_size = d.size;
            t.o_f = offs[f];
            t.is_pml = d.is_pml;
            t.scene = scene_of(i);
            t.vel = f < 2 ? 1 : 0;  // maxima class: px/py as written by velocity lines
            ctx->fft_segs.push_back(t);
        }
    }
    if (plan->n_receivers > 0) {
        TileDesc t{};
        t.kind = 2;  // receiver sampling of the previous step (first stage only)
        t.count = 1;
        ctx->fft_segs.push_back(t);
    }
    if (ctab.empty()) ctab.push_back(make_float2(0, 0));
    if (ftab.empty()) ftab.push_back(0);
    // PML factor arena (1 where no PML), vy and py row-major as they come: the device
    // turns them
    std::vector<float> pml(ctx->arena_floats, 1.f);
    std::vector<TurnField> pml_turned;  // vy and py of the PML domains (src, dst: below)
    std::vector<long long> pml_off;
    for (int i = 0; i < plan->n_domains; ++i) {
        const pstd_plan_domain &p = plan->domains[i];
        if (!p.is_pml) continue;
        const DomainDev &d = ctx->doms[i];
        const float *src[4] = {p.pml_vx, p.pml_vy, p.pml_px, p.pml_py};
        const long long offs[4] = {d.base + d.f_vx, d.base + d.f_vy, d.base + d.f_px, d.base + d.f_py};
        const int sizes[4] = {field_size(p, PSTD_FIELD_VX), field_size(p, PSTD_FIELD_VY), field_size(p, PSTD_FIELD_PX),
                              field_size(p, PSTD_FIELD_PY)};
        for (int f = 0; f < 4; ++f) {
            if (!src[f]) {
                ctx->err = "PML domain without factor arrays";
                return PSTD_ERR_INVALID;
            }
            std::memcpy(pml.data() + offs[f], src[f], sizeof(float) * sizes[f]);
            if (f == 1 || f == 3) {
                pml_turned.push_back({nullptr, nullptr, sizes[f] / p.nx, p.nx, 0});
                pml_off.push_back(offs[f]);
            }
        }
    }
    // receivers
    std::vector<ReceiverCell> cells;
    for (int r = 0; r < plan->n_receivers; ++r) {
        const pstd_plan_receiver &rc = plan->receivers[r];
        if (rc.domain < 0 || rc.domain >= plan->n_domains || rc.index < 0 ||
            rc.index >= plan->domains[rc.domain].nx * plan->domains[rc.domain].ny) {
            ctx->err = "receiver outside its domain";
            return PSTD_ERR_INVALID;
        }
        const DomainDev &d = ctx->doms[rc.domain];
        if (rc.spectral) cells.push_back({-1, -1});
        else cells.push_back({d.base + d.f_px + rc.index, d.base + d.f_py + (long long)(rc.index % d.nx) * d.ny + rc.index / d.nx});
    }
    ctx->nrec = (int)cells.size();
    {
        int rc = build_spectral_receivers(ctx, plan);
        if (rc) return rc;
    }
    std::vector<P0Tile> p0_tiles;
    ctx->p0_first.clear();
    for (const DomainDev &d : ctx->doms) {
        ctx->p0_first.push_back((int)p0_tiles.size());
        for (int y = 0; y < d.ny; y += kP0Side)
            for (int x = 0; x < d.nx; x += kP0Side) p0_tiles.push_back({d.base + d.f_px, d.base + d.f_py, d.nx, d.ny, x, y});
    }
    ctx->p0_first.push_back((int)p0_tiles.size());
    ctx->p0_pass = !ctx->tiles_gemm.empty() || strided_bytes - 16 * pass_cells > kP0PassBytes;
    if (!ctx->tiles_gemm.empty()) {
        // what a first stage after host writes reads: p0 (P0I) and vx, vy (TN)
        for (int i = 0; i < plan->n_domains; ++i) {
            const DomainDev &d = ctx->doms[i];
            const int sc = scene_of(i);
            ctx->max_ranges.push_back({3LL * (long long)ctx->arena_floats + d.base + d.f_px, (long long)d.nx * d.ny, 2 * sc});
            ctx->max_ranges.push_back({d.base + d.f_vx, (long long)d.ny * (d.nx + 1), 2 * sc + 1});
            ctx->max_ranges.push_back({d.base + d.f_vy, (long long)(d.ny + 1) * d.nx, 2 * sc + 1});
        }
    }
    // allocate + upload
    const size_t af = ctx->arena_floats;
    HIP_TRY(hipMalloc(&ctx->arena, 4 * af * sizeof(float)));
    HIP_TRY(hipMalloc(&ctx->pml, af * sizeof(float)));
    // the PML factors by way of S0, whose vy and py are turned over them (on the host
    // that took 30 to 100 us of the set-up of a small scene); then the arenas are zeroed
    HIP_TRY(hipMemcpyAsync(ctx->S(0), pml.data(), af * sizeof(float), hipMemcpyHostToDevice, ctx->stream));
    HIP_TRY(hipMemcpyAsync(ctx->pml, ctx->S(0), af * sizeof(float), hipMemcpyDeviceToDevice, ctx->stream));
    for (size_t k = 0; k < pml_turned.size(); ++k) {
        pml_turned[k].src = ctx->S(0) + pml_off[k];
        pml_turned[k].dst = ctx->pml + pml_off[k];
    }
    {
        const int rc = launch_turns(ctx, pml_turned);
        if (rc) return rc;
    }
    HIP_TRY(hipMemsetAsync(ctx->arena, 0, 4 * af * sizeof(float), ctx->stream));
    HIP_TRY(hipMalloc(&ctx->ctab, ctab.size() * sizeof(float2)));
    HIP_TRY(hipMemcpyAsync(ctx->ctab, ctab.data(), ctab.size() * sizeof(float2), hipMemcpyHostToDevice, ctx->stream));
    HIP_TRY(hipMalloc(&ctx->ftab, ftab.size() * sizeof(float)));
    HIP_TRY(hipMemcpyAsync(ctx->ftab, ftab.data(), ftab.size() * sizeof(float), hipMemcpyHostToDevice, ctx->stream));
    if (!ctx->tiles_gemm.empty()) {
        // the GEMM tiles' maxima slots, numbered like those of upload_tiles
        const int groups = 2 * ctx->n_scenes;
        ctx->gemm_first.assign(groups + 1, 0);
        auto group = [](const GemmTile &t) { return 2 * t.t.scene + (t.t.vel ? 0 : 1); };
        for (const GemmTile &t : ctx->tiles_gemm) ctx->gemm_first[group(t) + 1] += kGemmThreads / 64;
        for (int i = 0; i < groups; ++i) ctx->gemm_first[i + 1] += ctx->gemm_first[i];
        std::vector<int> next = ctx->gemm_first;
        for (GemmTile &t : ctx->tiles_gemm) {
            t.t.slot = next[group(t)];
            next[group(t)] += kGemmThreads / 64;
        }
        // segment order (a scene's segments together, a line block's output
        // tiles adjacent): measured faster than grouping the tiles by matrix
        HIP_TRY(hipMalloc(&ctx->d_gemm, ctx->tiles_gemm.size() * sizeof(GemmTile)));
        HIP_TRY(hipMalloc(&ctx->d_max_first, (size_t)(groups + 1) * sizeof(int2)));
        HIP_TRY(hipMalloc(&ctx->dmat, std::max<size_t>(1, dmat.size()) * sizeof(uint16_t)));
        HIP_TRY(hipMemcpyAsync(ctx->dmat, dmat.data(), dmat.size() * sizeof(uint16_t), hipMemcpyHostToDevice,
                               ctx->stream));
        const size_t nmax = 2 * (size_t)ctx->n_scenes;
        HIP_TRY(hipMalloc(&ctx->umax, nmax * sizeof(unsigned)));
        HIP_TRY(hipMemsetAsync(ctx->umax, 0, nmax * sizeof(unsigned), ctx->stream));
        HIP_TRY(hipMalloc(&ctx->d_max_ranges, ctx->max_ranges.size() * sizeof(MaxRange)));
        HIP_TRY(hipMemcpyAsync(ctx->d_max_ranges, ctx->max_ranges.data(), ctx->max_ranges.size() * sizeof(MaxRange),
                               hipMemcpyHostToDevice, ctx->stream));
    }
    {
        take_tuned_threads(ctx);
        const int rc = upload_tiles(ctx);
        if (rc) return rc;
    }
    HIP_TRY(hipMalloc(&ctx->d_cells, std::max<size_t>(1, cells.size()) * sizeof(ReceiverCell)));
    if (!cells.empty())
        HIP_TRY(hipMemcpyAsync(ctx->d_cells, cells.data(), cells.size() * sizeof(ReceiverCell), hipMemcpyHostToDevice,
                               ctx->stream));
    HIP_TRY(hipMalloc(&ctx->d_p0_tiles, std::max<size_t>(1, p0_tiles.size()) * sizeof(P0Tile)));
    if (!p0_tiles.empty())
        HIP_TRY(hipMemcpyAsync(ctx->d_p0_tiles, p0_tiles.data(), p0_tiles.size() * sizeof(P0Tile), hipMemcpyHostToDevice,
                               ctx->stream));
    ctx->sample_cap = 4096;
    HIP_TRY(hipMalloc(&ctx->d_samples, (size_t)ctx->sample_cap * std::max(1, ctx->nrec) * sizeof(float)));
    HIP_TRY(hipStreamSynchronize(ctx->stream));
    ctx->steps_done = 0;
    ctx->p0_explicit = true;
    ctx->planned = true;
    const int rc = autotune(ctx);
    if (rc) ctx->planned = false;  // a failed trial run leaves no usable launch state
    return rc;
}

// PSTD_FORM_AUTO: the plan uploaded (and autotuned) in the FFT form and in the
// FP16 GEMM form, the one with the shorter tuned stage kept; the choice is
// remembered per (device, plan signature), so a later upload of a plan of
// the same geometry uploads once.
static int upload_form(pstd_ctx *ctx, const pstd_plan_desc *plan, const std::vector<int> *dom_scene) {
    if (ctx->form_req != PSTD_FORM_AUTO) {
        ctx->form = ctx->form_req;
        return upload_impl(ctx, plan, dom_scene);
    }
    ctx->form = PSTD_FORM_FFT;
    int rc = upload_impl(ctx, plan, dom_scene);
    if (rc) return rc;
    const std::pair<int, uint64_t> key(ctx->device, plan_signature(ctx));
    int chosen = -1;
    {
        std::lock_guard<std::mutex> lock(g_tune_mu);
        auto it = g_form.find(key);
        if (it != g_form.end()) chosen = it->second;
    }
    if (chosen < 0) {
        const float fft_ms = ctx->tuned_stage_ms;
        const int trials = ctx->trial_steps;
        ctx->form = PSTD_FORM_GEMM_F16;
        rc = upload_impl(ctx, plan, dom_scene);
        if (rc) return rc;
        const bool gemm_better = !ctx->tiles_gemm.empty() && ctx->tuned_stage_ms < fft_ms;
        chosen = gemm_better ? PSTD_FORM_GEMM_F16 : PSTD_FORM_FFT;
        ctx->trial_steps += trials;
        {
            std::lock_guard<std::mutex> lock(g_tune_mu);
            g_form[key] = chosen;
        }
        if (gemm_better) return PSTD_OK;
        const int t = ctx->trial_steps;
        ctx->form = PSTD_FORM_FFT;
        rc = upload_impl(ctx, plan, dom_scene);  // its launch shape comes from the autotune cache
        ctx->trial_steps += t;
        return rc;
    }
    if (chosen == PSTD_FORM_FFT) return PSTD_OK;
    ctx->form = chosen;
    return upload_impl(ctx, plan, dom_scene);
}

int pstd_ctx_upload_plan(pstd_ctx *ctx, const pstd_plan_desc *plan) {
    if (!ctx || !plan) return PSTD_ERR_INVALID;
    std::lock_guard<TurnLock> turn(ctx->turn);
    return upload_form(ctx, plan, nullptr);
}

int pstd_ctx_upload_plans(pstd_ctx *ctx, const pstd_plan_desc *plans, int n_plans) {
    if (!ctx || !plans || n_plans <= 0) return PSTD_ERR_INVALID;
    std::lock_guard<TurnLock> turn(ctx->turn);
    if (n_plans == 1) return upload_form(ctx, plans, nullptr);
    // independent scenes: one plan with the domain lists concatenated; scenes
    // share the time step, the RK coefficients and the grid (one launch per
    // stage advances all of them)
    std::vector<pstd_plan_domain> doms;
    std::vector<pstd_plan_segment> segs;
    std::vector<pstd_plan_receiver> rcv;
    std::vector<int> dom_scene;
    const pstd_plan_desc &p0 = plans[0];
    for (int i = 0; i < n_plans; ++i) {
        const pstd_plan_desc &p = plans[i];
        bool same = p.dx == p0.dx && p.dt == p0.dt && p.c1 == p0.c1 && p.patch_error == p0.patch_error;
        for (int k = 0; k < 6; ++k) same = same && p.rk_alpha[k] == p0.rk_alpha[k];
        if (!same) {
            ctx->err = "batched scenes must share dx, dt, c1, patch error and RK coefficients (scene " +
                       std::to_string(i) + " differs)";
            return PSTD_ERR_INVALID;
        }
        if (p.n_domains < 0 || p.n_segments < 0 || p.n_receivers < 0) return PSTD_ERR_INVALID;
        const int base = (int)doms.size();
        for (int d = 0; d < p.n_domains; ++d) {
            doms.push_back(p.domains[d]);
            dom_scene.push_back(i);
        }
        for (int k = 0; k < p.n_segments; ++k) {
            pstd_plan_segment s = p.segments[k];
            const bool bad = s.domain < 0 || s.domain >= p.n_domains || s.side1 >= p.n_domains || s.side2 >= p.n_domains;
            if (bad) {
                ctx->err = "segment of scene " + std::to_string(i) + " names a domain outside its scene";
                return PSTD_ERR_INVALID;
            }
            s.domain += base;
            if (s.side1 >= 0) s.side1 += base;
            if (s.side2 >= 0) s.side2 += base;
            segs.push_back(s);
        }
        for (int r = 0; r < p.n_receivers; ++r) {
            pstd_plan_receiver c = p.receivers[r];
            if (c.domain < 0 || c.domain >= p.n_domains) {
                ctx->err = "receiver of scene " + std::to_string(i) + " outside its scene";
                return PSTD_ERR_INVALID;
            }
            c.domain += base;
            rcv.push_back(c);
        }
    }
    pstd_plan_desc m = p0;
    m.n_domains = (int)doms.size();
    m.domains = doms.data();
    m.n_segments = (int)segs.size();
    m.segments = segs.data();
    m.n_receivers = (int)rcv.size();
    m.receivers = rcv.data();
    return upload_form(ctx, &m, &dom_scene);
}

int pstd_ctx_set_field(pstd_ctx *ctx, int domain, int field, const float *host, size_t count) {
    if (!ctx) return PSTD_ERR_INVALID;
    std::lock_guard<TurnLock> turn(ctx->turn);
    if (!ctx->planned || !host) return PSTD_ERR_INVALID;
    if (domain < 0 || domain >= (int)ctx->doms.size() || field < 0 || field > 4) return PSTD_ERR_INVALID;
    const pstd_plan_domain &p = ctx->plan_domains[domain];
    if (count != (size_t)field_size(p, field)) {
        ctx->err = "field size mismatch";
        return PSTD_ERR_INVALID;
    }
    HIP_TRY(hipSetDevice(ctx->device));
    const DomainDev &d = ctx->doms[domain];
    const size_t bytes = count * sizeof(float);
    if (field == PSTD_FIELD_P0 || ctx->umax) {
        // GEMM form: the next first stage recomputes the scaling maxima from
        // the state, which needs p0 in its explicit array
        int rc = materialise_p0(ctx);
        if (rc) return rc;
    }
    if (field == PSTD_FIELD_P0) {
        HIP_TRY(hipMemcpyAsync(ctx->P0I() + field_off(d, PSTD_FIELD_PX), host, bytes, hipMemcpyHostToDevice, ctx->stream));
        ctx->p0_turn = true;  // for all domains at once, by the next first stage
    } else if (field == PSTD_FIELD_VY || field == PSTD_FIELD_PY) {
        // column-major on the device: turned from S0, which holds nothing else between
        // time steps, before the next step or read of such a field
        HIP_TRY(hipMemcpyAsync(ctx->S(0) + field_off(d, field), host, bytes, hipMemcpyHostToDevice, ctx->stream));
        ctx->written[2 * domain + (field == PSTD_FIELD_PY)] = 1;
        ctx->any_written = true;
    } else {
        HIP_TRY(hipMemcpyAsync(ctx->TN() + field_off(d, field), host, bytes, hipMemcpyHostToDevice, ctx->stream));
    }
    HIP_TRY(hipStreamSynchronize(ctx->stream));
    return PSTD_OK;
}

static bool short_result(pstd_ctx *ctx, size_t bytes) {
    if (bytes > kPinBytes) return false;
    if (!ctx->pin) ctx->pin = take_pinned();
    return ctx->pin != nullptr;
}

int pstd_ctx_get_field(pstd_ctx *ctx, int domain, int field, float *host, size_t count) {
    if (!ctx) return PSTD_ERR_INVALID;
    std::lock_guard<TurnLock> turn(ctx->turn);
    if (!ctx->planned || !host) return PSTD_ERR_INVALID;
    if (domain < 0 || domain >= (int)ctx->doms.size() || field < 0 || field > 4) return PSTD_ERR_INVALID;
    const pstd_plan_domain &p = ctx->plan_domains[domain];
    if (count != (size_t)field_size(p, field)) {
        ctx->err = "field size mismatch";
        return PSTD_ERR_INVALID;
    }
    HIP_TRY(hipSetDevice(ctx->device));
    const DomainDev &d = ctx->doms[domain];
    const float *src = ctx->TN() + field_off(d, field);
    if (field == PSTD_FIELD_VY || field == PSTD_FIELD_PY) {
        const int rc = turn_written(ctx);
        if (rc) return rc;
    }
    if (short_result(ctx, count * sizeof(float))) {
        if (field == PSTD_FIELD_P0 && !ctx->p0_explicit && !ctx->p0_pass) {
            hipLaunchKernelGGL(rows_kernel, dim3((unsigned)((count + 255) / 256)), dim3(256), 0, ctx->stream,
                               ctx->S(1) + field_off(d, PSTD_FIELD_PX), ctx->S(1) + field_off(d, PSTD_FIELD_PY),
                               (float *)ctx->pin, d.nx, d.ny);
            HIP_TRY(hipGetLastError());
        } else if (field == PSTD_FIELD_VY || field == PSTD_FIELD_PY) {
            hipLaunchKernelGGL(rows_kernel, dim3((unsigned)((count + 255) / 256)), dim3(256), 0, ctx->stream,
                               (const float *)nullptr, src, (float *)ctx->pin, d.nx, (int)(count / d.nx));
            HIP_TRY(hipGetLastError());
        } else {
            if (field == PSTD_FIELD_P0) src = ctx->P0I() + field_off(d, PSTD_FIELD_PX);
            HIP_TRY(hipMemcpyAsync(ctx->pin, src, count * sizeof(float), hipMemcpyDeviceToHost, ctx->stream));
        }
        HIP_TRY(hipStreamSynchronize(ctx->stream));
        std::memcpy(host, ctx->pin, count * sizeof(float));
        return PSTD_OK;
    }
    if (field == PSTD_FIELD_P0) {
        // P0I's slots are free where the tiles form p0 on the fly
        if (!ctx->p0_explicit && !ctx->p0_pass) {
            int rc = launch_p0(ctx, domain, true);
            if (rc) return rc;
        }
        src = ctx->P0I() + field_off(d, PSTD_FIELD_PX);
    } else if (field == PSTD_FIELD_VY || field == PSTD_FIELD_PY) {
        // row-major for the host; S0 holds nothing between time steps
        float *rows = ctx->S(0) + field_off(d, field);
        int rc = launch_turn(ctx, src, rows, d.nx, (int)(count / d.nx));
        if (rc) return rc;
        src = rows;
    }
    HIP_TRY(hipMemcpyAsync(host, src, count * sizeof(float), hipMemcpyDeviceToHost, ctx->stream));
    HIP_TRY(hipStreamSynchronize(ctx->stream));
    return PSTD_OK;
}

int pstd_ctx_read_frame(pstd_ctx *ctx, int domain, float *out, size_t count) {
    return pstd_ctx_get_field(ctx, domain, PSTD_FIELD_P0, out, count);
}

// Captures enqueue_steps(graph_steps) into a graph.  Only valid once p0 comes
// from the stage outputs (after the first step), which every replay keeps.
static int build_graph(pstd_ctx *ctx) {
    ctx->drop_graph();
    if (ctx->nrec > 0)
        HIP_TRY(hipMalloc(&ctx->d_gsamples, (size_t)ctx->graph_steps * ctx->nrec * sizeof(float)));
    float *const samples = ctx->d_samples;
    ctx->d_samples = ctx->d_gsamples;  // captured: the graph's own sample slots 0 .. graph_steps-1
    HIP_TRY(hipStreamBeginCapture(ctx->stream, hipStreamCaptureModeThreadLocal));
    int rc = enqueue_steps(ctx, ctx->graph_steps);
    hipGraph_t g = nullptr;
    hipError_t e = hipStreamEndCapture(ctx->stream, &g);
    ctx->d_samples = samples;
    if (rc) {
        if (g) (void)hipGraphDestroy(g);
        return rc;
    }
    if (e != hipSuccess) {
        ctx->err = std::string("graph capture: ") + hipGetErrorString(e);
        return PSTD_ERR_DEVICE;
    }
    ctx->graph = g;
    HIP_TRY(hipGraphInstantiate(&ctx->graph_exec, ctx->graph, nullptr, nullptr, 0));
    return PSTD_OK;
}

static int advance_impl(pstd_ctx *ctx, int steps, float *samples) {
    if (!ctx->planned || steps < 0) return PSTD_ERR_INVALID;
    HIP_TRY(hipSetDevice(ctx->device));
    {
        const int rc = turn_written(ctx);
        if (rc) return rc;
    }
    if (ctx->max_stale) {
        // the next first stage recomputes the maxima from the state (explicit p0)
        const int rc = materialise_p0(ctx);
        if (rc) return rc;
        ctx->max_stale = false;
    }
    int done = 0;
    const int gs = ctx->graph_steps;
    while (done < steps) {
        // one chunk of at most sample_cap steps fills sample slots 0 .. chunk-1:
        // graph replays where a whole graph fits (each copies its samples into
        // place on the device), eager launches for the rest and for a first step
        // after host writes (the graph reads p0 from the stage outputs)
        const int chunk = std::min(steps - done, ctx->sample_cap);
        int pos = 0;
        while (pos < chunk) {
            const int left = chunk - pos;
            if (gs > 0 && !ctx->p0_explicit && left >= gs) {
                if (!ctx->graph_exec) {
                    int rc = build_graph(ctx);
                    if (rc) return rc;
                }
                HIP_TRY(hipGraphLaunch(ctx->graph_exec, ctx->stream));
                if (samples && ctx->nrec > 0)
                    HIP_TRY(hipMemcpyAsync(ctx->d_samples + (size_t)pos * ctx->nrec, ctx->d_gsamples,
                                           (size_t)gs * ctx->nrec * sizeof(float), hipMemcpyDeviceToDevice,
                                           ctx->stream));
                pos += gs;
            } else {
                const int n = (gs > 0 && ctx->p0_explicit && left > gs) ? 1 : (gs > 0 && left >= gs ? gs : left);
                int rc = enqueue_steps(ctx, n, pos);
                if (rc) return rc;
                pos += n;
            }
        }
        ctx->steps_done += chunk;
        if (samples && ctx->nrec > 0) {
            float *const to = samples + (size_t)done * ctx->nrec;
            const size_t bytes = (size_t)chunk * ctx->nrec * sizeof(float);
            const bool pinned = short_result(ctx, bytes);
            HIP_TRY(hipMemcpyAsync(pinned ? (void *)ctx->pin : to, ctx->d_samples, bytes, hipMemcpyDeviceToHost, ctx->stream));
            HIP_TRY(hipStreamSynchronize(ctx->stream));
            if (pinned) std::memcpy(to, ctx->pin, bytes);
        }
        done += chunk;
    }
    return PSTD_OK;
}

int pstd_ctx_advance(pstd_ctx *ctx, int steps, float *samples) {
    if (!ctx) return PSTD_ERR_INVALID;
    std::lock_guard<TurnLock> turn(ctx->turn);
    int rc = advance_impl(ctx, steps, samples);
    if (rc) return rc;
    HIP_TRY(hipStreamSynchronize(ctx->stream));
    return PSTD_OK;
}

int pstd_ctx_advance_async(pstd_ctx *ctx, int steps) {
    if (!ctx) return PSTD_ERR_INVALID;
    std::lock_guard<TurnLock> turn(ctx->turn);
    return advance_impl(ctx, steps, nullptr);
}

int pstd_ctx_synchronize(pstd_ctx *ctx) {
    if (!ctx) return PSTD_ERR_INVALID;
    std::lock_guard<TurnLock> turn(ctx->turn);
    HIP_TRY(hipSetDevice(ctx->device));
    HIP_TRY(hipStreamSynchronize(ctx->stream));
    return PSTD_OK;
}

int pstd_ctx_steps_done(const pstd_ctx *ctx) { return ctx ? ctx->steps_done : -1; }

int pstd_ctx_set_stage_overlap(pstd_ctx *ctx, int on) {
    if (!ctx) return PSTD_ERR_INVALID;
    std::lock_guard<TurnLock> turn(ctx->turn);
    if (on && !(ctx->side && ctx->ev_fork && ctx->ev_join)) {
        ctx->err = "no side stream for overlapped stages";
        return PSTD_ERR_DEVICE;
    }
    HIP_TRY(hipSetDevice(ctx->device));
    HIP_TRY(hipStreamSynchronize(ctx->stream));
    ctx->drop_graph();
    ctx->overlap = on != 0;
    return PSTD_OK;
}

int pstd_ctx_capture_graph(pstd_ctx *ctx) {
    if (!ctx) return PSTD_ERR_INVALID;
    std::lock_guard<TurnLock> turn(ctx->turn);
    if (!ctx->planned) return PSTD_ERR_INVALID;
    if (ctx->graph_steps <= 0 || ctx->graph_exec) return PSTD_OK;
    if (ctx->p0_explicit) {
        ctx->err = "the step graph is captured once p0 comes from the stage outputs (after a time step)";
        return PSTD_ERR_INVALID;
    }
    HIP_TRY(hipSetDevice(ctx->device));
    HIP_TRY(hipStreamSynchronize(ctx->stream));
    return build_graph(ctx);
}

int pstd_ctx_set_graph_steps(pstd_ctx *ctx, int steps) {
    if (!ctx || steps < 0) return PSTD_ERR_INVALID;
    std::lock_guard<TurnLock> turn(ctx->turn);
    if (ctx->planned && steps > ctx->sample_cap) {
        ctx->err = "graph longer than the sample buffer (" + std::to_string(ctx->sample_cap) + " steps)";
        return PSTD_ERR_INVALID;
    }
    HIP_TRY(hipSetDevice(ctx->device));
    HIP_TRY(hipStreamSynchronize(ctx->stream));
    ctx->drop_graph();
    ctx->graph_steps = steps;
    return PSTD_OK;
}

int pstd_ctx_set_form(pstd_ctx *ctx, int form) {
    if (!ctx || (form != PSTD_FORM_FFT && form != PSTD_FORM_GEMM_F16 && form != PSTD_FORM_GEMM_BF16 &&
                 form != PSTD_FORM_AUTO))
        return PSTD_ERR_INVALID;
    std::lock_guard<TurnLock> turn(ctx->turn);
    if (ctx->planned) {
        ctx->err = "the derivative form is chosen before the plan is uploaded";
        return PSTD_ERR_INVALID;
    }
    ctx->form_req = form;
    ctx->form = form == PSTD_FORM_AUTO ? PSTD_FORM_FFT : form;
    return PSTD_OK;
}

int pstd_ctx_get_form(const pstd_ctx *ctx) { return ctx ? ctx->form : PSTD_ERR_INVALID; }

int pstd_ctx_set_kernel_flavour(pstd_ctx *ctx, int flavour) {
    if (!ctx || flavour < 0 || flavour > 2) return PSTD_ERR_INVALID;
    std::lock_guard<TurnLock> turn(ctx->turn);
    ctx->lean = flavour;
    return PSTD_OK;
}

int pstd_ctx_get_tuning(const pstd_ctx *ctx, int32_t *lean, int32_t *xcd_contiguous, double *stage_ms) {
    if (!ctx || !ctx->planned) return PSTD_ERR_INVALID;
    if (lean) *lean = ctx->lean;
    if (xcd_contiguous) *xcd_contiguous = ctx->xcd_remap;
    if (stage_ms) *stage_ms = ctx->tuned_stage_ms;
    return PSTD_OK;
}

int pstd_ctx_get_autotune(const pstd_ctx *ctx, int32_t *trial_steps, int32_t *from_cache) {
    if (!ctx || !ctx->planned) return PSTD_ERR_INVALID;
    if (trial_steps) *trial_steps = ctx->trial_steps;
    if (from_cache) *from_cache = ctx->tune_cached ? 1 : 0;
    return PSTD_OK;
}

int pstd_ctx_get_stage_paths(const pstd_ctx *ctx, int32_t *p0_pass, int32_t *eight_value_points) {
    if (!ctx || !ctx->planned) return PSTD_ERR_INVALID;
    if (p0_pass) *p0_pass = ctx->p0_pass ? 1 : 0;
    if (eight_value_points) *eight_value_points = ctx->f8;
    return PSTD_OK;
}

int pstd_ctx_set_tile_threads(pstd_ctx *ctx, int threads) {
    if (!ctx) return PSTD_ERR_INVALID;
    std::lock_guard<TurnLock> turn(ctx->turn);
    if (!ctx->planned || (threads != 128 && threads != 256 && threads != 512)) return PSTD_ERR_INVALID;
    if (threads == 128 && ctx->small_fmax > 1024) {
        ctx->err = "128-thread tiles need every line of the F <= 2048 class to have F <= 1024";
        return PSTD_ERR_INVALID;
    }
    HIP_TRY(hipSetDevice(ctx->device));
    HIP_TRY(hipStreamSynchronize(ctx->stream));
    ctx->drop_graph();
    ctx->small_nt = threads;
    const int rc = upload_tiles(ctx);
    if (rc) {
        ctx->planned = false;  // the tile lists are gone with the failed upload
        return rc;
    }
    HIP_TRY(hipStreamSynchronize(ctx->stream));
    return PSTD_OK;
}

int pstd_ctx_get_tile_threads(const pstd_ctx *ctx) {
    if (!ctx || !ctx->planned) return PSTD_ERR_INVALID;
    return ctx->small_nt;
}

int pstd_ctx_set_tile_order(pstd_ctx *ctx, int xcd_contiguous) {
    if (!ctx) return PSTD_ERR_INVALID;
    std::lock_guard<TurnLock> turn(ctx->turn);
    HIP_TRY(hipSetDevice(ctx->device));
    HIP_TRY(hipStreamSynchronize(ctx->stream));
    ctx->drop_graph();
    ctx->xcd_remap = xcd_contiguous ? 1 : 0;
    return PSTD_OK;
}

int pstd_ctx_profile_stages(pstd_ctx *ctx, int steps, double *mean_stage_ms, int *launches) {
    if (!ctx || steps <= 0 || !mean_stage_ms) return PSTD_ERR_INVALID;
    std::lock_guard<TurnLock> turn(ctx->turn);
    if (!ctx->planned) return PSTD_ERR_INVALID;
    HIP_TRY(hipSetDevice(ctx->device));
    hipEvent_t ev[2];
    HIP_TRY(hipEventCreate(&ev[0]));
    HIP_TRY(hipEventCreate(&ev[1]));
    int rc = PSTD_OK;
    float ms = 0;
    if (hipEventRecord(ev[0], ctx->stream) != hipSuccess) rc = PSTD_ERR_DEVICE;
    if (rc == PSTD_OK) rc = advance_impl(ctx, steps, nullptr);
    if (rc == PSTD_OK && hipEventRecord(ev[1], ctx->stream) != hipSuccess) rc = PSTD_ERR_DEVICE;
    if (rc == PSTD_OK && hipEventSynchronize(ev[1]) != hipSuccess) rc = PSTD_ERR_DEVICE;
    if (rc == PSTD_OK && hipEventElapsedTime(&ms, ev[0], ev[1]) != hipSuccess) rc = PSTD_ERR_DEVICE;
    (void)hipEventDestroy(ev[0]);
    (void)hipEventDestroy(ev[1]);
    if (rc) return rc;
    *mean_stage_ms = (double)ms / (6.0 * steps);
    if (launches) *launches = 6 * steps;
    return PSTD_OK;
}

int pstd_ctx_advance_static(pstd_ctx *ctx, int steps) {
    if (!ctx || steps < 0) return PSTD_ERR_INVALID;
    std::lock_guard<TurnLock> turn(ctx->turn);
    if (!ctx->planned) return PSTD_ERR_INVALID;
    const bool gemm = !ctx->tiles_gemm.empty();
    if (gemm && ctx->n_scenes > kStaticScenes) {
        ctx->err = "allocation-free advance: " + std::to_string(ctx->n_scenes) + " scenes, at most " +
                   std::to_string(kStaticScenes);
        return PSTD_ERR_INVALID;
    }
    HIP_TRY(hipSetDevice(ctx->device));
    unsigned *sp = nullptr;
    if (gemm) {
        if (resolve_scratch(ctx->device, &sp) != PSTD_OK) {
            ctx->err = "allocation-free advance: no device address for the scratch array";
            return PSTD_ERR_DEVICE;
        }
        // the shared array starts from the maxima of the current state (explicit
        // p0, then the first stage's reduction), as after host writes
        int rc = materialise_p0(ctx);
        if (rc) return rc;
    }
    {
        const int rc = turn_written(ctx);
        if (rc) return rc;
    }
    unsigned *own = ctx->umax;
    if (gemm) ctx->umax = sp;
    int rc = PSTD_OK, done = 0;
    while (rc == PSTD_OK && done < steps) {  // eager launches only: nothing to instantiate
        const int chunk = std::min(steps - done, ctx->sample_cap);
        rc = enqueue_steps(ctx, chunk);
        if (rc == PSTD_OK) {
            ctx->steps_done += chunk;
            done += chunk;
        }
    }
    ctx->umax = own;
    if (gemm) ctx->max_stale = true;
    return rc;
}

int pstd_ctx_profile_kernels(pstd_ctx *ctx, int steps, double *ms, int *launches) {
    if (!ctx || steps <= 0 || !ms || !launches) return PSTD_ERR_INVALID;
    std::lock_guard<TurnLock> turn(ctx->turn);
    if (!ctx->planned) return PSTD_ERR_INVALID;
    HIP_TRY(hipSetDevice(ctx->device));
    HIP_TRY(hipStreamSynchronize(ctx->stream));
    hipEvent_t ev[2];
    HIP_TRY(hipEventCreate(&ev[0]));
    HIP_TRY(hipEventCreate(&ev[1]));
    const int graph_steps = ctx->graph_steps;
    ctx->graph_steps = 0;  // eager launches: events cannot be recorded into the replayed graph
    ctx->prof = true;
    ctx->prof_events.clear();
    int rc = PSTD_OK;
    float total = 0;
    if (hipEventRecord(ev[0], ctx->stream) != hipSuccess) rc = PSTD_ERR_DEVICE;
    if (rc == PSTD_OK) rc = advance_impl(ctx, steps, nullptr);
    if (rc == PSTD_OK && hipEventRecord(ev[1], ctx->stream) != hipSuccess) rc = PSTD_ERR_DEVICE;
    if (rc == PSTD_OK && hipEventSynchronize(ev[1]) != hipSuccess) rc = PSTD_ERR_DEVICE;
    if (rc == PSTD_OK && hipEventElapsedTime(&total, ev[0], ev[1]) != hipSuccess) rc = PSTD_ERR_DEVICE;
    ctx->prof = false;
    ctx->graph_steps = graph_steps;
    for (int c = 0; c <= kClasses; ++c) {
        ms[c] = 0;
        launches[c] = 0;
    }
    for (auto &pe : ctx->prof_events) {
        float t = 0;
        if (rc == PSTD_OK && hipEventElapsedTime(&t, pe.second.first, pe.second.second) != hipSuccess) rc = PSTD_ERR_DEVICE;
        ms[pe.first] += t;
        launches[pe.first] += 1;
        (void)hipEventDestroy(pe.second.first);
        (void)hipEventDestroy(pe.second.second);
    }
    ctx->prof_events.clear();
    (void)hipEventDestroy(ev[0]);
    (void)hipEventDestroy(ev[1]);
    if (rc) {
        if (ctx->err.empty()) ctx->err = "profile_kernels: HIP event failure";
        return rc;
    }
    ms[kClasses] = total;
    launches[kClasses] = 6 * steps;
    return PSTD_OK;
}

int pstd_ctx_gemm_work(const pstd_ctx *ctx, double *flops_per_stage, long long *outputs_per_stage) {
    if (!ctx || !ctx->planned) return PSTD_ERR_INVALID;
    if (flops_per_stage) *flops_per_stage = ctx->gemm_flops;
    if (outputs_per_stage) *outputs_per_stage = ctx->gemm_cells;
    return PSTD_OK;
}

long long pstd_ctx_cells_per_stage(const pstd_ctx *ctx) {
    if (!ctx || !ctx->planned) return -1;
    long long n = 0;
    for (const pstd_plan_domain &d : ctx->plan_domains)
        if (!d.is_rigid) n += (long long)d.nx * d.ny;
    return n;
}

}  // extern "C"
