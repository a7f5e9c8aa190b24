// Triangular sweeps of 5-point grid factors, one grid line per lane.
//
// A compute wavefront owns a strip of 64 lines along i.  At step s, lane l
// finishes cell i = s - l of its line (up to a constant), so the two values a
// row depends on are the lane's own last result (i - 1) and the last result of
// lane l - 1 (j - 1): a step is the row's dependent arithmetic and one DPP lane
// shift, and no value of the recurrence goes through memory inside a strip.
// The rows' entries are applied in the order of the reference's loops
// (lower_trisolve.hpp:172-209, upper_trisolve.hpp:131-176), so results equal
// the general sweep's bit for bit.
//
// Upper sweeps run the same code on mirrored coordinates: row r of the grid is
// row n - 1 - r of the mirrored one, where its dependencies come first.
//
// Cells outside the grid (before a line's start, after its end, lines past the
// last) have coefficients +0 and right-hand side +0.  A cell that a row inside
// the grid reads without an entry for it lies before its line's start or in the
// zeros read in place of a strip before the first, and gives exactly +0:
// rr - (+0) * (+0) leaves rr unchanged.  What cells after a line's end or past
// the last line give is read by such cells only.
//
// What bounds it: the compute wavefront's instructions, 41 ns a step (18 ns of
// them the dependent chain: lane shift and four FP64 operations) for nx + 63
// steps a strip, and 3.9 (64 x 700) to 5.1 us (1000 x 1000) from strip to strip, of
// which the 64 steps between their first lines are 2.6 us; HBM traffic, 24 *
// steps / nx + 16 bytes a row in double (40 on long lines, 70 with nx = 64), is far
// below.  One wavefront per strip and workgroup, because two in one workgroup slowed
// each other (60 against 78 ns a step).  Per sweep in double, against the
// general sweep's tiles: 256 x 256 28 to 32 us (88), 301 x 173 28 us (80), 700 x 64
// 35 us, 64 x 64 9.2 us (27), 64 x 700 47 us, 1000 x 1000 125 us, 8000 x 66 381 us.
// A sweep that also forms dot(w, y) is bound by its loader: 58 us at 256 x 256.
// The same scheme with 16 x 4 lines of a 7-point grid per wavefront took 117 us
// at 128^3 with the factors in the Infinity Cache but 150 us without, no better
// than the general sweep's 140 us: 22 strips on the critical path, 198 cycles a step
// for the second lane shift and its imports, and only 16 steps of coefficients in
// flight.
#include "buffer_dev.hpp"
#include "m4g_device.hpp"
#include "lines.hpp"
#include "sentinel.hpp"

#include <algorithm>

namespace m4g {

constexpr int kLineBlock = 8;       // steps a compute wavefront runs between two looks at its imports
constexpr int kLineGroup = 4;       // steps whose coefficients are packed together
constexpr int kLineDepth = 16;      // steps of coefficients in flight (the unrolling)
constexpr int kLineRing = 32;       // steps of right-hand side, and of results, held in LDS
constexpr int kLineRow = kLineRing + 2;   // ring entries per lane: 16 lanes that read 16 bytes of theirs use all 64 banks
constexpr int kLineHeader = 128;    // bytes: counters of the workgroup
constexpr int kLineZeros = 16;      // zeros read in place of imports by the first strip
constexpr int kLineLead = 63;       // steps by which the strip before is ahead when it has the value a step needs
constexpr int kLineWaves = 8;
constexpr int kLinePollsPerSpin = 5;   // polls in half a microsecond and a little more (one takes 0.12 us, three in flight)
constexpr int kDone = 1 << 30;

// A strip's first line starts at step `line_phase`, chosen so that the imports
// of a block come from one block of the strip before: 63 is 7 modulo 8.
__host__ __device__ inline int line_phase(int strip) { return 7 * strip & 7; }

// Dynamic LDS: header, rings, zeros, then the imports, one value per step.
struct LineLds {
    size_t vring, yring, zeros, west, total;
};
__host__ __device__ inline LineLds line_lds(int steps, int vbytes)
{
    LineLds l;
    l.vring = kLineHeader;
    l.yring = l.vring + size_t(kWave) * kLineRow * vbytes;
    l.zeros = l.yring + size_t(kWave) * kLineRow * vbytes;
    l.west = l.zeros + size_t(kLineZeros) * vbytes;
    l.total = l.west + size_t(steps + kLineBlock) * vbytes;   // the last look ahead reads a block past the end
    return l;
}

// A strip holds coefficients for the lanes' skew as well: 24 * steps / nx bytes a
// row in double, 54 with nx = 64, 960 with nx = 2, where the general sweep's records take
// 64.  More than that is given for the speed (2 x 50 000: 5.7 against 12.1 ms an
// application) up to this size; a larger narrow grid takes the general sweep, so
// that whatever fits the card with records fits.
constexpr int64_t kLinePadBytes = int64_t(256) << 20;
constexpr int64_t kRecordRowBytes = 64;

LineGeom line_geometry(const GridInfo& g, size_t lds_budget)
{
    LineGeom G;
    // (the kernel addresses a vector with 32-bit byte offsets, a strip's coefficients likewise)
    if (g.nz != 1 || g.nx < 2 || g.ny < 2 || g.nx * g.ny >= (int64_t(1) << 29) - 64) return G;
    const int64_t steps = (g.nx + 63 + 7 + kLineDepth - 1) / kLineDepth * kLineDepth;   // the lanes' skew and the phase
    if (steps >= (1 << 20) || line_lds(int(steps), 8).total > lds_budget) return G;
    const int64_t strips = (g.ny + 63) / 64;
    if (strips * steps * kWave * 24 > std::max(kLinePadBytes, g.nx * g.ny * kRecordRowBytes)) return G;
    G.nx = int32_t(g.nx);
    G.ny = int32_t(g.ny);
    G.steps = int32_t(steps);
    G.strips = int32_t(strips);
    return G;
}

// ---------------------------------------------------------------------------
// coefficients
// ---------------------------------------------------------------------------
// Values of a step and lane: the two entries in the order they are subtracted,
// then 1/d unless the diagonal is one.  Those of a group's four steps lie
// together, 16 bytes of all lanes at a time: 1.5 loads a step in double.
template <typename FV, bool UNIT>
struct LinePack {
    static constexpr int K = UNIT ? 2 : 3;
    static constexpr int per = 16 / int(sizeof(FV));                    // values of a chunk
    static constexpr int chunks = kLineGroup * K / per;                 // of a group
    static constexpr int group_bytes = chunks * kWave * 16;
};

template <typename FV, bool UNIT>
__global__ __launch_bounds__(256) void k_line_pack(LineGeom G, int kind, const int32_t* __restrict__ fs,
                                                   const double* __restrict__ f, FV* __restrict__ out)
{
    using P = LinePack<FV, UNIT>;
    const int64_t x = blockIdx.x * int64_t(256) + threadIdx.x;   // (strip, step, lane)
    if (x >= int64_t(G.strips) * G.steps * kWave) return;
    const bool mirror = line_upper(kind), upper_storage = kind == kLineIc0Lower || kind == kLineIc0Upper;
    const int lane = int(x % kWave), s = int(x / kWave % G.steps), strip = int(x / kWave / G.steps);
    int i = s - lane - line_phase(strip), j = strip * kWave + lane;
    FV c[3] = {FV(0), FV(0), FV(0)};
    if (i >= 0 && i < G.nx && j < G.ny) {
        if (mirror) {
            i = G.nx - 1 - i;
            j = G.ny - 1 - j;
        }
        // storage position of the entry of row (ri, rj) towards axis a (0 i, 1 j), before or after its diagonal
        auto pos = [&](int ri, int rj, int a, bool after) {
            const int p = fs[ri + G.nx * rj];
            if (!after) return p + (a == 1 ? 0 : int(rj > 0));
            return p + (upper_storage ? 0 : int(rj > 0) + int(ri > 0)) + 1 + (a == 1 ? int(ri < G.nx - 1) : 0);
        };
        const bool own = kind == kLineIc0Upper || kind == kLineIluLower || kind == kLineIluUpper;
        const bool far_first = kind != kLineIc0Upper && kind != kLineIluUpper;   // j then i (else i then j)
        const int d = mirror ? 1 : -1;   // the dependency is the neighbour at +1 or -1
        for (int e = 0; e < 2; e++) {
            const int a = far_first ? 1 - e : e;
            const int ni = i + (a == 0 ? d : 0), nj = j + (a == 1 ? d : 0);
            if (ni < 0 || ni >= G.nx || nj < 0 || nj >= G.ny) continue;
            c[e] = FV(f[own ? pos(i, j, a, d > 0) : pos(ni, nj, a, d < 0)]);
        }
        if (!UNIT) c[2] = FV(f[fs[i + G.nx * j] + (upper_storage ? 0 : int(j > 0) + int(i > 0))]);
    }
    FV* o = out + (int64_t(strip) * G.steps + s) / kLineGroup * (P::group_bytes / int64_t(sizeof(FV)));
#pragma unroll
    for (int k = 0; k < P::K; k++) {
        const int e = s % kLineGroup * P::K + k;
        o[e / P::per * (kWave * P::per) + lane * P::per + e % P::per] = c[k];
    }
}

template <typename T>
__global__ void k_line_sentinel(int64_t count, T* __restrict__ x)
{
    for (int64_t e = blockIdx.x * int64_t(256) + threadIdx.x; e < count; e += int64_t(gridDim.x) * 256)
        x[e] = Sentinel<T>::value();
}

// ---------------------------------------------------------------------------
// device helpers
// ---------------------------------------------------------------------------
// Lane l receives lane l - 1's value, lane 0 its own `old`.
__device__ inline double lane_shift(double old, double v)
{
    const long long o = __double_as_longlong(old), b = __double_as_longlong(v);
    const int lo = __builtin_amdgcn_update_dpp(int(o), int(b), 0x138, 0xF, 0xF, false);
    const int hi = __builtin_amdgcn_update_dpp(int(o >> 32), int(b >> 32), 0x138, 0xF, 0xF, false);
    return __longlong_as_double((long long)(((unsigned long long)(unsigned)hi << 32) | (unsigned)lo));
}
__device__ inline float lane_shift(float old, float v)
{
    return __int_as_float(__builtin_amdgcn_update_dpp(__float_as_int(old), __float_as_int(v), 0x138, 0xF, 0xF, false));
}

// Waits for all but the newest `newer` global loads of the wavefront.
template <int newer>
__device__ inline void wait_loads()
{
    static_assert(newer < 64);
    __builtin_amdgcn_s_waitcnt((newer & 15) | 0x0F70 | (newer >> 4) << 14);
}
// Waits for the wavefront's LDS operations.  At the end of a seldom taken path
// it keeps the compiler from waiting for that path's reads, and for everything
// issued since, on the usual one.
__device__ inline void lds_settle() { __builtin_amdgcn_s_waitcnt(0xC07F); }

template <typename T>
__device__ inline T lds_read(const T* p)
{
    return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
}
template <typename T>
__device__ inline void lds_write(T* p, T v)
{
    __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
}

template <typename FV>
__device__ inline FV word_of(u32x4 c, int e)   // value e of 16 bytes
{
    if constexpr (sizeof(FV) == 4) {
        return __builtin_bit_cast(FV, unsigned(c[e]));
    } else {
        const u32x2 h = {c[2 * e], c[2 * e + 1]};
        return __builtin_bit_cast(FV, h);
    }
}

// ---------------------------------------------------------------------------
// the sweep
// ---------------------------------------------------------------------------
struct LineArgs {
    LineGeom G;
    int mirror;
    unsigned* tickets;           // [0] next ticket, [1] finished strips
    int* fault;
    int64_t other_count;         // entries of the other direction's exchange buffer
    int64_t poll_limit;          // fruitless polls of a strip's importer
    double* dot_partials;        // [strips], or null
};

// Roles of a workgroup's wavefronts: one computes, one loads the right-hand
// side into an LDS ring, one stores the results from another, one imports the
// last line of the strip before, one exports the own last line.  Loads and
// stores are in different wavefronts because a wavefront's loads do not count
// as done before its earlier stores are acknowledged.  Strips go out in order
// by ticket, so every wait is for a workgroup that has started or for another
// role of the same one.
//
// The partials of dot(w, y) are formed by the loader.  A lane of it meets about
// one cell for every step of its strip, far more than a thread of the general
// sweep does (26 at most), so products are added up in double whatever the
// vectors' type is, eight sums of one level to one of the next (DotSum): the
// longest chain of additions stays as short.
//
// The compute wavefront's pace is its number of instructions (about 7 cycles
// each, alone on its SIMD), so it does nothing else.  The other roles go to wavefronts on
// other SIMDs, as in the general sweep, though fixed roles measure the same here
// (64 x 700: 47.6 and 48.0 us, 1000 x 1000: 123.9 and 123.7).
enum LineRole { kLineCompute, kLineLoad, kLineStore, kLineImport, kLineExport, kLineIdle };

__device__ inline LineRole line_role(const int* simd, int wave)
{
    if (wave == 0) return kLineCompute;
    int before = 0;   // wavefronts that choose first: those away from wavefront 0, in order
    for (int x = 1; x < kLineWaves; x++) {
        const bool away_x = simd[x] != simd[0], away = simd[wave] != simd[0];
        before += away_x == away ? x < wave : away_x;
    }
    return before < 4 ? LineRole(kLineLoad + before) : kLineIdle;
}

// Progress of the roles in blocks of eight steps; a role that is done or has
// nothing to do says kDone.  The compute wavefront runs block b when all four
// are past it.
struct alignas(16) LineFlags {
    int loaded;     // blocks of right-hand side in the ring less one (it reads one ahead)
    int west;       // blocks of imports
    int stored;     // blocks of results taken by the storer, and a ring's
    int exported;   // blocks of results taken by the exporter, and a ring's
    int finished;   // blocks the compute wavefront has finished
};

struct DotSum {
    double level[4] = {0, 0, 0, 0};
    __device__ void add(double block, int b)   // the sum of block b's products; b from 0 up
    {
        level[0] += block;
        if ((b & 7) == 7) carry(0);
        if ((b & 63) == 63) carry(1);
        if ((b & 511) == 511) carry(2);
    }
    __device__ void carry(int k)
    {
        level[k + 1] += level[k];
        level[k] = 0;
    }
    __device__ double total() const { return ((level[0] + level[1]) + level[2]) + level[3]; }
};

template <typename FV, typename VT, bool UNIT, bool FAR_FIRST>
__global__ __launch_bounds__(kLineWaves * kWave) void k_line_sweep(LineArgs a, const FV* __restrict__ coef,
                                                                   const VT* __restrict__ v, VT* __restrict__ y, VT* xbuf,
                                                                   VT* xbuf_other, const VT* __restrict__ dot_with,
                                                                   const int* skip)
{
    using P = LinePack<FV, UNIT>;
    constexpr int B = kLineBlock, D = kLineDepth, RB = kLineRing / B;
    if (skip && *skip) return;   // the solve this sweep belongs to has finished
    struct alignas(2 * sizeof(VT)) VT2 {
        VT x, y;
    };
    extern __shared__ unsigned char lds_raw[];
    const LineGeom G = a.G;
    const int S = G.steps, nb = S / B;
    const LineLds L = line_lds(S, int(sizeof(VT)));
    LineFlags* flags = reinterpret_cast<LineFlags*>(lds_raw);
    int* ticket = reinterpret_cast<int*>(lds_raw + 32);
    int* simds = reinterpret_cast<int*>(lds_raw + 64);
    VT* vring_all = reinterpret_cast<VT*>(lds_raw + L.vring);
    VT* yring_all = reinterpret_cast<VT*>(lds_raw + L.yring);
    VT* zeros = reinterpret_cast<VT*>(lds_raw + L.zeros);
    VT* west = reinterpret_cast<VT*>(lds_raw + L.west);
    const int tid = threadIdx.x, lane = tid % kWave;
    const int wave = __builtin_amdgcn_readfirstlane(tid / kWave);
    // workgroup 0, dispatched first, takes the first strip without a ticket
    if (tid == 0) *ticket = blockIdx.x != 0 ? 1 + int(atomicAdd(&a.tickets[0], 1u)) : 0;
    if (lane == 0) simds[wave] = simd_id();
    if (tid < kLineZeros) zeros[tid] = VT(0);
    __syncthreads();
    const LineRole role = LineRole(__builtin_amdgcn_readfirstlane(line_role(simds, wave)));
    const int strip = __builtin_amdgcn_readfirstlane(*ticket);
    const int phase = line_phase(strip);
    const bool first = strip == 0, last = strip + 1 == G.strips;
    if (tid == 0) *flags = LineFlags{-1, first ? kDone : 0, RB, last ? kDone : RB, 0};

    double dacc = 0;
    if (role == kLineCompute) {
        // ---- compute ----
        VT* vring = vring_all + lane * kLineRow;
        VT* yring = yring_all + lane * kLineRow;
        const auto cres = buffer_of(reinterpret_cast<const char*>(coef) + int64_t(strip) * (S / kLineGroup) * P::group_bytes,
                                    unsigned(S / kLineGroup + 2 * D / kLineGroup) * P::group_bytes);
        u32x4 cv[D / kLineGroup][P::chunks];
        const int off = lane * 16;
        auto load = [&](int g, int s) {   // the coefficients of steps s..s+3 (a multiple of 4)
#pragma unroll
            for (int c = 0; c < P::chunks; c++)
                cv[g][c] = __builtin_amdgcn_raw_buffer_load_b128(cres, off + c % 4 * 1024,
                                                                 s / kLineGroup * P::group_bytes + c / 4 * 4096, 0);
        };
        // in this order: the loop waits for the oldest, and a later place of its load in this sequence would make it
        // wait for all of them on every turn
#pragma unroll
        for (int g = 0; g < D / kLineGroup; g++) {
            load(g, g * kLineGroup);
            __builtin_amdgcn_sched_barrier(0);
        }
        lds_barrier();
        __builtin_amdgcn_s_setprio(3);
        auto read8 = [](const VT* p, VT (&x)[B]) {
#pragma unroll
            for (int e = 0; e < B / 2; e++) {
                const VT2 t = reinterpret_cast<const VT2*>(p)[e];
                x[2 * e] = t.x;
                x[2 * e + 1] = t.y;
            }
        };
        // imports: lane 0 needs them, the others read along and ignore them
        const VT* wp = first ? zeros : west;
        const int wstep = first ? 0 : 1;
        typedef __attribute__((address_space(3))) const volatile i32x4 lds_i32x4;
        lds_i32x4* fp = (lds_i32x4*)(reinterpret_cast<const i32x4*>(flags));
        VT out = VT(0);
        VT vq[2][B], wq[2][B], res[B];   // this block's operands and the next one's
        i32x4 ready = fp[0];
        while (ready.x < 0) ready = fp[0];
        __atomic_signal_fence(__ATOMIC_SEQ_CST);
        read8(vring, vq[0]);
        auto look = [&](int s, int p) {   // the progress first, then the imports it covers
            ready = fp[0];
            __atomic_signal_fence(__ATOMIC_SEQ_CST);
            read8(wp + s * wstep, wq[p]);
        };
        look(0, 0);
        lds_settle();
        for (int s0 = 0; s0 < S; s0 += D) {
#pragma unroll
            for (int u0 = 0; u0 < D; u0 += B) {
                const int p = u0 / B & 1, s = s0 + u0, b = s / B;
                auto behind = [&] { return min(min(ready.x, ready.y), min(ready.z, ready.w)) <= b; };
                if (__builtin_expect(__any(behind()), 0)) {
                    do {
                        look(s, p);
                        lds_settle();
                    } while (__any(behind()));
                }
                __atomic_signal_fence(__ATOMIC_SEQ_CST);
                read8(vring + ((s + B) & (kLineRing - 1)), vq[1 - p]);
#pragma unroll
                for (int q = 0; q < B; q++) {
                    const int g = (u0 + q) / kLineGroup, e = (u0 + q) % kLineGroup * P::K;
                    if (e == 0) wait_loads<(D / kLineGroup - 1) * P::chunks>();
                    const VT c0 = VT(word_of<FV>(cv[g][e / P::per], e % P::per));
                    const VT c1 = VT(word_of<FV>(cv[g][(e + 1) / P::per], (e + 1) % P::per));
                    const VT vy = lane_shift(wq[p][q], out);
                    // rr -= c * y in the order of the reference's row, then the diagonal
                    VT rr = vq[p][q] - c0 * (FAR_FIRST ? vy : out);
                    rr = rr - c1 * (FAR_FIRST ? out : vy);
                    if constexpr (!UNIT) rr = rr * VT(word_of<FV>(cv[g][(e + 2) / P::per], (e + 2) % P::per));
                    out = rr;
                    res[q] = rr;
                    if ((u0 + q) % kLineGroup == kLineGroup - 1) load(g, s0 + D + g * kLineGroup);
                    if (q == B / 2 - 1) {
                        __builtin_amdgcn_sched_barrier(0);
                        look(s + B, 1 - p);
                        __builtin_amdgcn_sched_barrier(0);
                    }
                }
                VT2* yo = reinterpret_cast<VT2*>(yring + (s & (kLineRing - 1)));
#pragma unroll
                for (int e = 0; e < B / 2; e++) yo[e] = VT2{res[2 * e], res[2 * e + 1]};
                // LDS serves a wavefront's operations in order: whoever sees this count sees the results
                __atomic_signal_fence(__ATOMIC_SEQ_CST);
                lds_write(&flags->finished, b + 1);
            }
        }
        __builtin_amdgcn_s_setprio(0);
        __builtin_amdgcn_s_waitcnt(0);
    } else if (role == kLineLoad || role == kLineStore) {
        // ---- loader and storer ----
        // Lane 8 * m + c holds step c of a block of lines m, m + 8, ..., so a line's eight cells are one contiguous span.
        const int c = lane & 7;
        const unsigned bytes = unsigned(G.n()) * unsigned(sizeof(VT));
        const int delta = a.mirror ? -B * int(sizeof(VT)) : B * int(sizeof(VT));   // of a block
        int i0[8];         // cell of the lane's lines at block 0
        unsigned o0[8];    // and its offset in the vectors
#pragma unroll
        for (int q = 0; q < 8; q++) {
            const int l = 8 * q + (lane >> 3), j = strip * kWave + l;
            const int i = c - l - phase, r = i + G.nx * j;
            i0[q] = j < G.ny ? i : -(1 << 28);   // no cell is in range on a line outside
            o0[q] = unsigned(a.mirror ? G.n() - 1 - r : r) * unsigned(sizeof(VT));
        }
        auto offset = [&](int q, int b) {
            return unsigned(i0[q] + B * b) < unsigned(G.nx) ? o0[q] + unsigned(delta * b) : kNoCell;
        };
        auto wait_finished = [&](int b) {
            while (lds_read(&flags->finished) <= b) __builtin_amdgcn_s_sleep(1);
            __atomic_signal_fence(__ATOMIC_SEQ_CST);
        };
        VT* vring = vring_all + (lane >> 3) * kLineRow + c;
        const VT* yring = yring_all + (lane >> 3) * kLineRow + c;
        if (role == kLineLoad) {
            constexpr int F = RB;   // blocks in flight
            VT buf[F][8], wbuf[F][8];
            const auto vres = buffer_of(v, bytes), wres = buffer_of(dot_with, dot_with ? bytes : 0);
            auto fetch = [&](__amdgpu_buffer_rsrc_t from, VT (&x)[8], int b) {   // (no cell from block nb on)
#pragma unroll
                for (int q = 0; q < 8; q++) x[q] = buffer_load<VT, 0>(from, offset(q, b));
            };
#pragma unroll
            for (int f = 0; f < F; f++) {
                fetch(vres, buf[f], f);
                __builtin_amdgcn_sched_barrier(0);
            }
            lds_barrier();
            DotSum sum;
            // block b takes the place of block b - RB once that one is finished (and, for the dot, its results read)
            auto run = [&](auto with_dot) {
                constexpr bool dot = decltype(with_dot)::value;
                for (int b0 = 0; b0 < nb + (dot ? RB : 0); b0 += F) {
#pragma unroll
                    for (int f = 0; f < F; f++) {
                        const int b = b0 + f, d = b - RB;
                        if (d >= 0 && d < nb) {
                            wait_finished(d);
                            if constexpr (dot) {
                                const VT* p = yring + (d * B & (kLineRing - 1));
                                double t[8];   // (a cell outside the grid may hold anything)
#pragma unroll
                                for (int q = 0; q < 8; q++) {
                                    const double prod = double(wbuf[f][q]) * double(p[8 * q * kLineRow]);
                                    t[q] = offset(q, d) != kNoCell ? prod : 0.0;
                                }
                                sum.add(((t[0] + t[1]) + (t[2] + t[3])) + ((t[4] + t[5]) + (t[6] + t[7])), d);
                            }
                        }
                        if (b < nb) {
                            VT* p = vring + (b * B & (kLineRing - 1));
#pragma unroll
                            for (int q = 0; q < 8; q++) p[8 * q * kLineRow] = buf[f][q];
                            __atomic_signal_fence(__ATOMIC_SEQ_CST);
                            if (lane == 0) lds_write(&flags->loaded, b + 1 < nb ? b : kDone);
                        }
                        fetch(vres, buf[f], b + F);
                        if constexpr (dot) fetch(wres, wbuf[f], b);
                    }
                }
            };
            if (dot_with) run(std::true_type());
            else run(std::false_type());
            dacc = sum.total();
        } else {
            lds_barrier();
            const auto yres = buffer_of(y, bytes);
            for (int b = 0; b < nb; b++) {
                wait_finished(b);
                const VT* p = yring + (b * B & (kLineRing - 1));
                VT yv[8];
#pragma unroll
                for (int q = 0; q < 8; q++) yv[q] = p[8 * q * kLineRow];
                // (LDS serves these reads before the write of the count)
                __atomic_signal_fence(__ATOMIC_SEQ_CST);
                if (lane == 0) lds_write(&flags->stored, b + 1 + RB);
#pragma unroll
                for (int q = 0; q < 8; q++) buffer_store(yres, yv[q], offset(q, b));
            }
        }
    } else if (role == kLineImport) {
        // ---- importer ----
        // The strip before publishes its last line in order.  kPolls polls of the 64 entries after the first missing one
        // are in flight: a consumer that runs at its producer's pace ends up behind by the longest time a value takes,
        // and that includes the time between two polls (64 x 700: 47.6 us, with one in flight 48.9).
        lds_barrier();
        if (!first) {
            constexpr int kPolls = 3;
            const int lead = kLineLead + line_phase(strip - 1) - phase, count = S - lead;   // multiples of eight
            const auto src = buffer_of(xbuf + int64_t(strip - 1) * S + lead, unsigned(count) * unsigned(sizeof(VT)));
            int head = 0, from[kPolls];
            VT val[kPolls];
            BoundedWait wait{a.poll_limit, a.fault};
            auto poll = [&](int k) {   // (past the end: 0)
                from[k] = head;
                val[k] = buffer_load<VT, 0x10>(src, unsigned(head + lane) * unsigned(sizeof(VT)));
            };
            auto publish = [&] {
                __atomic_signal_fence(__ATOMIC_SEQ_CST);
                lds_write(&flags->west, head >= count ? kDone : head / B);
            };
#pragma unroll
            for (int k = 0; k < kPolls; k++) poll(k);
            while (head < count) {
#pragma unroll
                for (int k = 0; k < kPolls; k++) {
                    const unsigned long long miss = __ballot(Sentinel<VT>::is(val[k]));
                    const int got = min(count, from[k] + (miss ? int(__builtin_ctzll(miss)) : kWave));
                    if (got > head) {
                        if (from[k] + lane < got) west[from[k] + lane] = val[k];
                        head = got;
                        publish();
                    } else if (head < count) {
                        if (wait.over()) {
                            // give up: the host reports the fault, the results are meaningless
                            if (lane == 0) __hip_atomic_store(a.fault, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                            head = count;
                            publish();
                        }
                        __builtin_amdgcn_s_sleep(1);
                    }
                    poll(k);
                }
            }
        }
    } else if (role == kLineExport) {
        // ---- exporter ----
        // Stores lane 63's values as its blocks are finished, up to a ring's at a time.
        lds_barrier();
        if (!last) {
            const VT* p = yring_all + 63 * kLineRow;
            VT* dst = xbuf + int64_t(strip) * S + lane;
            for (int head = 0; head < nb;) {
                const int fin = __builtin_amdgcn_readfirstlane(lds_read(&flags->finished));
                if (fin == head) {
                    __builtin_amdgcn_s_sleep(1);
                    continue;
                }
                __atomic_signal_fence(__ATOMIC_SEQ_CST);
                const VT val = p[(head * B + lane) & (kLineRing - 1)];
                const int got = min(fin - head, RB);
                if (lane < got * B)
                    __hip_atomic_store(dst + head * B, val, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                head += got;
                __atomic_signal_fence(__ATOMIC_SEQ_CST);
                lds_write(&flags->exported, head + RB);
            }
        }
        // the other direction's exchange buffer is free: reset it for its next use
        for (int64_t x = strip * int64_t(kWave) + lane; x < a.other_count; x += int64_t(G.strips) * kWave)
            xbuf_other[x] = Sentinel<VT>::value();
    } else {
        lds_barrier();
    }
    __syncthreads();
    if (dot_with) {
        double* scratch = reinterpret_cast<double*>(lds_raw + L.vring);
        const double tot = block_sum<kLineWaves * kWave>(dacc, scratch);
        if (tid == 0) a.dot_partials[strip] = tot;
    }
    if (tid == 0) {
        const unsigned done = atomicAdd(&a.tickets[1], 1u);
        if (done == unsigned(G.strips) - 1) {   // every strip has started: reset for the next launch
            a.tickets[0] = 0;
            a.tickets[1] = 0;
        }
    }
}

// ---------------------------------------------------------------------------
// host side
// ---------------------------------------------------------------------------
void LineSweep::init(const LineGeom& g, int kd, int ftype, const double* f, const int32_t* rows)
{
    G = g;
    kind = kd;
    factor_type = ftype;
    fstore = f;
    frows = rows;
    stale = true;
    xbuf_type = -1;
    hipStream_t s = current_stream();
    tickets.reset(2);
    M4G_HIP(hipMemsetAsync(tickets.ptr, 0, 2 * sizeof(unsigned), s));
    fault.reset(1);
    M4G_HIP(hipMemsetAsync(fault.ptr, 0, sizeof(int), s));
}

template <typename FV, bool UNIT>
static void pack_lines(LineSweep& d, hipStream_t s)
{
    const int64_t groups = int64_t(d.G.strips) * (d.G.steps / kLineGroup);
    // the sweep reads up to kLineDepth steps past a strip's last
    const size_t bytes = size_t(groups + 2 * kLineDepth / kLineGroup) * LinePack<FV, UNIT>::group_bytes;
    if (d.coef.count != bytes) d.coef.reset(bytes);
    const int64_t count = groups * kLineGroup * kWave;
    hipLaunchKernelGGL((k_line_pack<FV, UNIT>), dim3(unsigned((count + 255) / 256)), dim3(256), 0, s, d.G, d.kind, d.frows,
                       d.fstore, (FV*)d.coef.ptr);
    M4G_HIP(hipGetLastError());
}

template <typename VT>
static void clear_exchange(LineSweep& d, hipStream_t s)
{
    const int64_t count = d.exchange_count();
    d.xbuf.reset(size_t(count) * sizeof(VT));
    hipLaunchKernelGGL(k_line_sentinel<VT>, dim3(unsigned(std::min<int64_t>(4096, (count + 255) / 256))), dim3(256), 0, s,
                       count, (VT*)d.xbuf.ptr);
    M4G_HIP(hipGetLastError());
}

void LineSweep::prepare(int vtype, hipStream_t s)
{
    if (stale) {
        const bool unit = line_unit(kind);
        if (factor_type == M4G_F64) unit ? pack_lines<double, true>(*this, s) : pack_lines<double, false>(*this, s);
        else unit ? pack_lines<float, true>(*this, s) : pack_lines<float, false>(*this, s);
        stale = false;
    }
    if (xbuf_type != vtype) {
        vtype == M4G_F64 ? clear_exchange<double>(*this, s) : clear_exchange<float>(*this, s);
        xbuf_type = vtype;
    }
}

template <typename FV, typename VT, bool UNIT, bool FAR_FIRST>
static void launch_line(LineSweep& d, LineSweep& other, const LineArgs& a, const void* v, void* y, const int* skip,
                        const void* dot_with, hipStream_t s)
{
    auto kern = k_line_sweep<FV, VT, UNIT, FAR_FIRST>;
    const size_t lds = line_lds(d.G.steps, int(sizeof(VT))).total;
    // beyond 64 KB of dynamic LDS must be requested, once per kernel and size
    static size_t granted = 0;
    if (lds > 65536 && lds > granted) {
        M4G_HIP(hipFuncSetAttribute(reinterpret_cast<const void*>(kern), hipFuncAttributeMaxDynamicSharedMemorySize,
                                    int(lds)));
        granted = lds;
    }
    hipLaunchKernelGGL(kern, dim3(unsigned(d.G.strips)), dim3(kLineWaves * kWave), lds, s, a, (const FV*)d.coef.ptr,
                       (const VT*)v, (VT*)y, (VT*)d.xbuf.ptr, (VT*)other.xbuf.ptr, (const VT*)dot_with, skip);
    M4G_HIP(hipGetLastError());
}

template <typename FV, typename VT>
static void launch_line_t(LineSweep& d, LineSweep& other, const LineArgs& a, const void* v, void* y, const int* skip,
                          const void* dot_with, hipStream_t s)
{
    if (line_unit(d.kind)) launch_line<FV, VT, true, true>(d, other, a, v, y, skip, dot_with, s);
    else if (d.kind == kLineIc0Upper || d.kind == kLineIluUpper)
        launch_line<FV, VT, false, false>(d, other, a, v, y, skip, dot_with, s);
    else launch_line<FV, VT, false, true>(d, other, a, v, y, skip, dot_with, s);
}

void LineSweep::launch(LineSweep& other, const void* v, void* y, int vtype, const int* skip, int64_t spin_limit,
                       const void* dot_with, double* dot_partials, hipStream_t s)
{
    LineArgs a;
    a.G = G;
    a.mirror = line_upper(kind);
    a.tickets = tickets.ptr;
    a.fault = fault.ptr;
    a.other_count = other.exchange_count();
    a.poll_limit = spin_limit * kLinePollsPerSpin;
    a.dot_partials = dot_partials;
    if (factor_type == M4G_F64) launch_line_t<double, double>(*this, other, a, v, y, skip, dot_with, s);
    else if (vtype == M4G_F64) launch_line_t<float, double>(*this, other, a, v, y, skip, dot_with, s);
    else launch_line_t<float, float>(*this, other, a, v, y, skip, dot_with, s);
}

}  // namespace m4g
