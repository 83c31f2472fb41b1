// dmx_tiling.h -- how the z-marching kernels cut a domain into column
// tiles and blocks of planes.  Plain integer code for host and device;
// tests/tiling_check.cpp compiles it on the host and checks that the tiles
// cover every column and plane exactly once within their limits,
// tests/launch_check.cpp the limits and choices of the launches.
#pragma once

#ifndef __HIPCC__
#ifndef __host__
#define __host__
#endif
#ifndef __device__
#define __device__
#endif
#ifndef __forceinline__
#define __forceinline__ inline
#endif
#endif

namespace dmx {

// A run of n columns cut into the fewest tiles of at most wmax: nt tiles,
// the first nt - nwide of them w wide, the last nwide w + 1 wide.  With
// wmax one more than a power-of-two tile width, the 2^m + 1 faces or
// 2^m + 2 cells of a power-of-two domain need no tile of one or two
// columns, which would cost a z-marching block as much as a full one.
struct Part { int nt, w, nwide; };
__host__ __device__ __forceinline__ Part make_part(int n, int wmax)
{
    Part p;
    p.nt = n > 0 ? (n + wmax - 1) / wmax : 1;
    p.w = n / p.nt;
    p.nwide = n - p.w * p.nt;
    return p;
}
__host__ __device__ __forceinline__ void part_tile(const Part& p, int t, int& start, int& width)
{
    const int nn = p.nt - p.nwide;
    start = t * p.w + (t > nn ? t - nn : 0);
    width = p.w + (t >= nn ? 1 : 0);
}

// The columns [0, nxc) x [0, nyc) of a plane in tiles of at most fc
// columns, at most fxm wide and fym high: x strips of the fewest tiles
// (make_part), each cut into rows of at most min(fym, fc / width).  Tiles
// are numbered strip by strip, rows fastest; nz blocks of planes, the
// fewest of at least kt planes (between kt and 2 kt - 1), follow one
// another.
struct Tiling {
    Part px, pyn, pyw, pz;
    int tz;   // tiles of one block of planes
};
__host__ __device__ __forceinline__ Tiling make_tiling(int nxc, int nyc, int nzc, int fxm, int fym, int fc, int kt)
{
    Tiling t;
    t.px = make_part(nxc, fxm);
    const int wn = t.px.w > 0 ? t.px.w : 1, ww = wn + 1;
    t.pyn = make_part(nyc, fc / wn < fym ? fc / wn : fym);
    t.pyw = make_part(nyc, fc / ww < fym ? fc / ww : fym);
    t.tz = (t.px.nt - t.px.nwide) * t.pyn.nt + t.px.nwide * t.pyw.nt;
    const int nzb = nzc / kt > 0 ? nzc / kt : 1;
    t.pz = make_part(nzc, (nzc + nzb - 1) / nzb);
    return t;
}
// tile l of block of planes zb: its first column, row and plane (from 0)
// and its extents
__host__ __device__ __forceinline__ void tiling_tile(const Tiling& t, int l, int zb, int& x0, int& fx, int& y0, int& fy,
                                                     int& z0, int& fz)
{
    const int nn = t.px.nt - t.px.nwide;
    int xt, yt;
    if (l < nn * t.pyn.nt) {
        xt = l / t.pyn.nt;
        yt = l - xt * t.pyn.nt;
        part_tile(t.pyn, yt, y0, fy);
    } else {
        l -= nn * t.pyn.nt;
        xt = nn + l / t.pyw.nt;
        yt = l - (xt - nn) * t.pyw.nt;
        part_tile(t.pyw, yt, y0, fy);
    }
    part_tile(t.px, xt, x0, fx);
    part_tile(t.pz, zb, z0, fz);
}

// Whether the face/edge stage over one plane per block, a grid of x * y * z
// blocks, may be launched as one block per Riemann problem of a cell: at most
// `most` blocks (kSplitMax in dmx_step.inc), and 6 z blocks along z, which
// counts planes times problems, within the 65535 that a grid has along y and z
// (float32 domains of nx <= 60 and ny = 3 reach 6 x 16384 otherwise).
inline bool split_fits(long long x, long long y, long long z, long long most)
{
    return x * y * z <= most && 6 * z <= 65535;
}

// Planes per block of the fused float64 kernel where it is not tuned: 16 where
// that gives 768 blocks (1.5 rounds of the 512 that the chip holds), else 4.
inline int fused_planes(int nx, int ny, int nz, int fxm, int fym, int fc)
{
    const Tiling t = make_tiling(nx + 1, ny + 1, nz + 1, fxm, fym, fc, 16);
    return (long long)t.tz * t.pz.nt >= 768 ? 16 : 4;
}

// Whether the fused float64 kernel over the tiles t is the faster form of the
// trace and the face/edge stage, by what the two take (us).  Fused: a block
// marches its planes and the one before them, 512 blocks (two per CU) at a time,
// 12.5 us a plane for each round begun, or 13.5 for a full one and 6 for the
// end of the last where the rounds run into one another.  Separate: 36 ns a
// block of 64 x 4 columns of a plane and 0.283 ns a cell.  So thin boxes and
// few blocks, which pay the extra plane and a second round that is nearly
// empty, keep the separate kernels.  Over 67 domains of 3 to 1000 cells a side
// with HLLD, and the other solvers over 13 of them, the choice is at most
// 5.8% from the faster one; measured (us, fused / separate): 101 x 50 x 37 133
// / 89, 118 x 60 x 30 134 / 94, 224 x 224 x 6 197 / 149, 128 x 256 x 8 160 / 139,
// 48^3 91 / 67, but 64^3 144 / 161, 512 x 512 x 8 940 / 1011, 80 x 48 x 243 418 /
// 517, 150 x 93 x 117 655 / 722 and 192^3 2617 / 3135.
inline bool fused_pays(const Tiling& t, int nx, int ny, int nz)
{
    const long long blocks = (long long)t.tz * t.pz.nt, begun = (blocks + 511) / 512;
    const double drift = 13.5 * (double)blocks / 512.0 + 6.0;
    const double fused = ((double)(nz + 1) / t.pz.nt + 1.0) * (12.5 * begun > drift ? 12.5 * begun : drift);
    const double nb = (double)((nx + 4 + 63) / 64) * ((ny + 1 + 3) / 4) * (nz + 1);
    const double separate = 4.0 + 0.036 * nb + 0.283e-3 * (nx + 1) * (ny + 1) * (nz + 1);
    return fused < separate;
}

// Planes per block (4, 8, 16 or 32) with which the fused float32 kernel, one
// block per CU, marches the fewest planes one after another: rounds of 256
// blocks times the planes of a block and the one before them, the fewer planes
// if it is the same within 1%.  A round takes 9.0 to 9.7 us a plane at any size
// from 96^3 on, so this is the fastest count or within 2% of it: 4, 8, 16, 32
// planes measured 216, 188, 167, 302 us at 96^3, 332, 355, 321, 354 at 112^3, 440, 442, 474, 602
// at 128^3, 782, 739, 785, 902 at 160^3, 1346, 1285, 1274, 1234 at 192^3 and
// 3080, 2857, 2717, 2764 at 256^3.
inline int fewest_plane_rounds(int nx, int ny, int nz, int fxm, int fym, int fc)
{
    int pick = 4;
    double least = 0.0;
    for (int kt = 4; kt <= 32; kt *= 2) {
        const Tiling t = make_tiling(nx + 1, ny + 1, nz + 1, fxm, fym, fc, kt);
        const long long rounds = ((long long)t.tz * t.pz.nt + 255) / 256;
        const double planes = (double)rounds * ((double)(nz + 1) / t.pz.nt + 1.0);
        if (kt == 4 || planes < 0.99 * least) {
            least = planes;
            pick = kt;
        }
    }
    return pick;
}

// A batch's launch shapes from context 0's: face/edge stage (mode 0 or 2 over
// 4 << kzi planes, 3 over 8 << kzi), trace (mode, z-march over 8 << kti planes).
// Shapes that were asked for (by the tuner, dmx_set_shape or the environment)
// are taken over, or the nearest that a batch has: 1 and 2 planes are 4, the
// separate face and edge kernels mode 0.  A context's own shapes are made for
// one box: a batch fills the chip with the separate kernels over 4 planes and
// the 3D tile of the trace.  Measured (ms a step, float64 / float32): 6 boxes of
// 128^3 6.7 / 3.61, over 8 planes 6.8 / 3.64, with the z-march of the trace 7.1 /
// 3.94, fused in float64 10.2; 16 of 64^3 2.64 / 1.49, 2.82 / 1.52, 2.76 / 1.59,
// 3.8; 48 of 32^3 1.30 / 0.70, 1.33 / 0.73, 1.37 / 0.78.  4 float64 boxes of
// 150 x 93 x 117, whose own trace is the z-march, take 3.36 with the tile, 3.47
// with the z-march.
struct BatchShape { int flux_mode, kzi, trace_mode, kti; };
inline BatchShape batch_shape(int flux_mode, int kz, bool flux_asked, int trace_mode, int kt, bool trace_asked)
{
    auto near = [](int k) { return k <= 11 ? 0 : (k <= 23 ? 1 : 2); };   // of 8, 16, 32
    BatchShape b = {0, 0, 0, 1};
    if (flux_asked) {
        b.flux_mode = flux_mode == 1 ? 0 : flux_mode;
        b.kzi = flux_mode == 3 ? near(kz) : (kz <= 4 ? 0 : (kz == 16 ? 2 : (kz == 32 ? 3 : 1)));
    }
    if (trace_asked) {
        b.trace_mode = trace_mode;
        b.kti = near(kt);
    }
    return b;
}

} // namespace dmx
