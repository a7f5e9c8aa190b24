// Triangular sweeps of 5-point grid factors, one grid line per lane.
#pragma once

#include "m4g_internal.hpp"
#include "schedule.hpp"

namespace m4g {

// The triangular solves of the preconditioners, named by the factor they read
// (storage: IC(0) the upper part of A's pattern, diagonal first; ILU(0) A's
// whole pattern; the diagonal inverted in both).
enum LineKind {
    kLineIc0Lower,   // L = trans(U): entries U[r-o][r], times 1/d
    kLineIc0Upper,   // U
    kLineIluLower,   // L, unit diagonal
    kLineIluUpper,   // U
    kLineAdjLower,   // trans(U)
    kLineAdjUpper    // trans(L), unit diagonal
};
inline __host__ __device__ bool line_upper(int kind)
{
    return kind == kLineIc0Upper || kind == kLineIluUpper || kind == kLineAdjUpper;
}
inline __host__ __device__ bool line_unit(int kind) { return kind == kLineIluLower || kind == kLineAdjUpper; }

// An nx x ny grid in strips of 64 lines (a line runs along i), one workgroup
// and one compute wavefront each.
struct LineGeom {
    int32_t nx = 0, ny = 0;
    int32_t strips = 0;       // 0: the sweep is not a line sweep
    int32_t steps = 0;        // steps of a strip, a multiple of the kernel's unrolling
    __host__ __device__ int32_t n() const { return nx * ny; }
};

// The geometry for a grid (strips 0 when it is not 2D, its lines are too long, or it is large and
// so narrow that the coefficients would take more memory than the general sweep's records).
LineGeom line_geometry(const GridInfo& g, size_t lds_budget);

struct LineSweep {
    LineGeom G;
    int kind = kLineIc0Lower;
    int factor_type = M4G_F64;
    const double* fstore = nullptr;      // factor values, in the storage's order
    const int32_t* frows = nullptr;      // [n+1] row starts of the storage (device, shared by the handle's sweeps)
    bool stale = true;                   // coefficients to be packed again
    DevBuf<unsigned char> coef;          // packed per strip, four steps and lane
    DevBuf<unsigned char> xbuf;          // exchange: the last line's values of every strip
    int xbuf_type = -1;
    DevBuf<unsigned> tickets;
    DevBuf<int> fault;

    void init(const LineGeom& g, int kind, int ftype, const double* f, const int32_t* rows);
    int64_t exchange_count() const { return int64_t(G.steps) * G.strips; }   // entries of xbuf
    void prepare(int vtype, hipStream_t s);
    void launch(LineSweep& other, const void* v, void* y, int vtype, const int* skip, int64_t spin_limit,
                const void* dot_with, double* dot_partials, hipStream_t s);
};

}  // namespace m4g
