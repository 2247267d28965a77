// pg_sph.h -- the three-dimensional disk (ndim 3: spherical radius, azimuth,
// polar angle; adiabatic gas), host entry points called by the C ABI in
// pg_host.cpp when a handle is created with ndim = 3.
#pragma once

#include <cstddef>

#include "../../include/pg_params.h"

namespace pg {

struct Sph;

constexpr int SPH_BT2 = 512;     // threads per block of the sweeps (about one element each)

// Tile of the radial sweep: xr rows x a segment of tx cells.  The row is cut
// into equal segments, and as many rows as fit SPH_BT2 threads (one per slot,
// segment + 2 PAD slots a row; half as many in FP64, whose PEM4 sweep needs
// 160 VGPRs: 84 us against 127 on a 96x192x32 disk) make a block; of all cuts
// the one that puts the most cells into a block's threads, so that few lanes
// issue instructions for halo cells or for nothing (a 384-radius row: five rows
// of four 102-slot segments fill 480 of 512 lanes with cells, one row's two
// 198-slot segments 192 of 256: radial sweep of the 384x1536x64 disk 1210 ->
// 1140 us).  A small disk takes fewer rows, down to one, so that the blocks
// still cover the chip's 256 CUs eight times (a 101x190x33 disk is 1 % slower
// with four rows in 1568 blocks than with three in 2090).  Chosen once, when
// the disk is made: the search looks at every number of segments.
struct RadialTile {
    int tx, xr;
    int xm;   // slot t is in row t / (tx + 2 PAD) = (t * xm) >> 20, for t < SPH_BT2
};
inline RadialTile radial_tile(int nx, long rows, int es) {
    constexpr int PAD = 3;   // ghost cells a side
    const int most_threads = es == 8 ? SPH_BT2 / 2 : SPH_BT2;
    RadialTile best{0, 0, 0};
    double most = 0.0;
    for (int parts = (nx + most_threads - 2 * PAD - 1) / (most_threads - 2 * PAD); parts <= nx; ++parts) {
        const int tx = (nx + parts - 1) / parts;
        if (best.tx && tx < 32) break;   // the halo alone is 16 % there
        const long nseg = (nx + tx - 1) / tx;
        int xr = most_threads / (tx + 2 * PAD);
        while (xr > 1 && nseg * ((rows + xr - 1) / xr) < 2048) --xr;
        const int threads = (xr * (tx + 2 * PAD) + 63) / 64 * 64;
        const double use = (double)nx * xr / ((double)nseg * threads);
        if (use > most) {
            most = use;
            best = RadialTile{tx, xr, (1 << 20) / (tx + 2 * PAD) + 1};
        }
    }
    return best;
}

// error reporting shared with pg_host.cpp (pg_last_error)
int report_error(int code, const char* fmt, ...);
// axis edges with ghosts and cell volumes (make_grid, init.cu:472-500) and the
// 4th-order slope weights of a cell from its five neighbours' edges
void host_make_axis(double* a, double* v, double amin, double amax, int res, int pad, int geom, int grid);
void host_slope_weights(int geom, const double* x6, double wl[3], double wr[3]);

int sph_validate(const pg_params& P);
int sph_create(const pg_params& P, Sph** out);
void sph_destroy(Sph* s);
int sph_get_state(Sph* s, double* gas);
void sph_ghost_x(const Sph* s, int g, int k, double* f5);
void sph_dims(const Sph* s, int* nx, int* ny, int* nz);
int sph_set_state(Sph* s, const double* gas);
int sph_global_dt(Sph* s, double dt_prev, double* dt_out);
int sph_solve(Sph* s, double t, double dt);
int sph_run(Sph* s, int nsteps, double* t_io, double* dt_io, double* dts);
int sph_sweep(Sph* s, int dir, double dt);   // 0 radius, 1 azimuth, 2 polar angle
int sph_orbital_advection(Sph* s, double dt, int* inc, double* res);
int sph_sources(Sph* s, double t_planet, double mdt, double dt, int inplace);
int sph_viscosity(Sph* s, int on_T, double* vis);
int sph_planet(Sph* s, double t, double* body10);
int sph_write_snapshot(Sph* s, const char* filename, double t);
int sph_read_snapshot(Sph* s, const char* filename, double* t_out);
int sph_profile_enable(Sph* s, int on);
int sph_profile_get(Sph* s, const char* kernel, double* avg_us, int* count);
int sph_device_bytes(Sph* s, size_t* bytes);
void* sph_stream(Sph* s);

}  // namespace pg
