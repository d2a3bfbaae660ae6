// Geometry set-up kernels (ibtfo_geom.hip).
#pragma once
#include "ibtfo_internal.h"

namespace ibtfo {

// shape record: {type (0 circle, 1 convex polygon), cx, cy, r, nverts, x0, y0, ... x7, y7}
constexpr int SHAPE_STRIDE = 21;

struct GeomArgs {
    Layout L;
    double Li, Hi, dx;      // first cell centre (with ghosts) and spacing, Psy_coord.cpp:21-26
    int kind;               // level-set hook
    double p[8];            // hook constants (evaluated on the host)
    const double* phi_in;   // kind 3: per-cell phi in reference cell order (null: phi holds it)
    const double* shapes;   // kind 5: nshapes records of SHAPE_STRIDE doubles
    int nshapes;
    double *phi, *nx, *ny;  // planes
    uint8_t* type;
    int bc;
    int unit_normals;       // corrected mode: normals scaled to unit length
    // cut cells (bc = IDW fill with active donors = types 0 and 3)
    int cut;
    double cdx, cdy;        // cell sizes (Psy_L / N_x, Psy_H / N_y)
    uint8_t* cmark;         // plane: merge direction and zero apertures (k_cut_cells, k_cut_target)
    CutCell* cuts;          // compact records of the type-3 cells (null: counting)
    int* cut_index;         // plane: record of each type-3 cell
    unsigned int* ccount;   // {cut cells, merge groups}
    int ccap;
    MergeGroup* groups;
    int gcap;
    uint8_t* stype;         // plane: the step kernel's types, a copy of type before the filling pass
    Ghost* ghosts;
    unsigned int* count;
    int cap;
};

// Mask level set (Test/PNGGeo/Level_Set.cpp:31-149): phi per cell from an RGBA image
struct MaskArgs {
    const unsigned* rgba;       // W x H pixels of four bytes, top row first
    int W, H;
    int M, N;                   // cells with ghosts
    double Li, Hi, dxc;         // cell centres (Psy_coord)
    double exo, eyo, dxp, dyp;  // edge pixel x: exo + dxp * x, y: eyo + dyp * y
    int nseg;                   // 32-row segments per pixel column
    unsigned* bits;             // nseg x W: edge pixels of each segment
    int *before, *after;        // nseg x W: last edge row below / first above each segment (-1: none)
    Layout L;
    double* phi;                // plane
};
constexpr int MASK_SEG = 32;
// The row search (k_edt_rows): cells per bounded interval, intervals, LDS bytes
constexpr int EDT_MAX_INTERVALS = 1024;
inline int edt_stride(int M) { return 64 * ((M + 64 * EDT_MAX_INTERVALS - 1) / (64 * EDT_MAX_INTERVALS)); }
inline int edt_intervals(int M) { return (M + edt_stride(M) - 1) / edt_stride(M); }
inline size_t mask_lds_bytes(int W, int M) { return (size_t)W * 16 + (edt_intervals(M) + 1) * sizeof(int); }
constexpr size_t MASK_LDS_MAX = 158 * 1024;  // beside a little static LDS

hipError_t geom_run(GeomArgs& g, hipStream_t s);
// lds: the row search stages its columns in LDS (mask_lds_bytes of it; the kernel's
// attribute is set by the caller), else it reads them from memory
hipError_t mask_run(MaskArgs& m, bool lds, hipStream_t s);
const void* mask_rows_kernel();  // the LDS form
// cut-cell geometry on top of geom_run's phi and normals: types, merge targets and
// ghosts, then the records (counting while g.cuts is null, then filling)
hipError_t cut_run(GeomArgs& g, hipStream_t s);
hipError_t cut_records(GeomArgs& g, hipStream_t s);
hipError_t geom_ghosts(GeomArgs& g, hipStream_t s);

}  // namespace ibtfo
