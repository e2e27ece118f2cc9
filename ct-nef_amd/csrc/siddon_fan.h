// The exact Siddon pair on fan planes (included by siddon.hip).
//
// The rays of one detector column of one view lie in one plane that contains
// the axis direction z: their paths in x, y are the same.  That path, the
// list of in-plane cells with the length of each, is worked out once per
// column in FP64 (one lane per slab) into an LDS table of pieces; a lane then
// walks one ray of the column through the list and is left with z alone.
// Where no ray steps more than one z cell per slab (fan_ok) a piece meets at
// most two z cells, the one the ray enters the slab in and the next one:
//
//   z = kz t + Zc at the slab's face,  fz = (p - fract(z)) / kz  (p = 1 rising, 0 falling)
//   clamp(fz - f0, 0, dt) in cell floor(z), the rest of dt in the next cell
//
// for a piece that covers [f0, f0 + dt] of its slab.  About 10 (forward) and
// 14 (adjoint) vector instructions per in-plane piece and ray, against 22 and
// 34 per voxel when every lane walks its own three coordinates: 512 x 512 x
// 256 voxels, 1024 x 768 cells, 720 views, forward 97.1 -> 78.6 ms, adjoint
// 262.4 -> 181.8 ms.  What bounds them now: the forward's two gathers per
// piece keep the CU's texture address unit busy 97 % of the time and its vector
// issue is nearly full as well; the adjoint fills 84 % of its vector issue
// slots and 56 % of its LDS cycles (two 64-bit additions per piece, 6.4 clocks
// of the CU each, and half a table read).
// Forward and adjoint evaluate the same functions below, a column by its own
// rules whichever others a wavefront takes with it, so the pair holds one
// matrix up to the rounding of a piece; the pieces do not depend on the block
// they are walked from, so the fixed-point adjoint's bits do not depend on how
// the volume or the views are split.  (walks_fan_planes may send one direction
// of a scan to the per-ray walk: then the two differ by a crossing's rounding.)
#pragma once

constexpr int FAN_ZPAD = 2;     // zero border of the z-fastest copy's rows

// In-plane path of a detector column in one view: walk axis m (the larger
// in-plane step in voxels), slabs [s0, s1) inside the box (none when it
// misses), the transverse coordinate a(t) = Aa + ka t at slab face t; and what
// its rays have in common: kz = b dk cells per slab and, above the view's
// z0, Zc = b dz cells at the slab tz for detector height b (mm).  (From b itself, which is exactly 0 in a middle row: its ray stays in the source's
// plane.)  One record per column and view is worked out once per call where
// the workspace has room: the adjoint reads it in every block it passes.
struct __align__(16) FanCol {
    double ka, ika, Aa, dk, dz;
    double l2;       // squared in-plane source-detector distance in x voxels (1/L^2 scale)
    double p2;       // squared in-plane mm per slab
    unsigned slabs;  // s0, s1 (15 bits each: grid sides are at most 16384), walk axis (bit 30)
    int tz;          // origin of z along the path (see FanRay)
    __device__ int s0() const { return slabs & 0x7fff; }
    __device__ int s1() const { return (slabs >> 15) & 0x7fff; }
    __device__ int m() const { return slabs >> 30; }
    __device__ int tc() const { return (s0() + s1()) >> 1; }        // middle slab
};
static_assert(sizeof(FanCol) == 64, "read as four 16-byte words");

// True when no ray of the geometry steps more than one z cell per slab of its
// in-plane walk: the in-plane source-detector distance is at least SAD, its
// larger component in voxels at least 1/sqrt(2) of that.
__host__ __device__ inline bool fan_ok(const VolDev& V, const DetDev& G, unsigned flags)
{
    if (flags & NEFCT_F_REF_SLAB) return false;
    const double b0 = G.bi * G.db - G.nb * G.db * 0.5, b1 = (G.bi + G.nb - 1) * G.db - G.nb * G.db * 0.5;
    const double bmax = fmax(fabs(b0), fabs(b1));
    return G.na < (1 << 24) && bmax * V.inv_vs[2] < 0.7 * G.sad * fmin(V.inv_vs[0], V.inv_vs[1]);
}

__device__ __forceinline__ FanCol fan_column(const VolDev& V, const DetDev& G, double c, double s, int ia)
{
#pragma clang fp contract(off)
    FanCol C;
    const double a = fma(G.ai + ia, G.da, -(G.na * G.da * 0.5));
    double lx, ly;
    if (G.cyl) {
        lx = G.sad * cos(a) - G.sid;
        ly = G.sad * sin(a);
    } else {
        lx = G.sad - G.sid;
        ly = a;
    }
    const double S0 = -G.sid * c, S1 = -G.sid * s;
    const double e0 = fma(lx, c, -(ly * s)) - S0, e1 = fma(lx, s, ly * c) - S1;
    const double d0 = e0 * V.inv_vs[0], d1 = e1 * V.inv_vs[1];
    const double u0 = (S0 - V.lo[0]) * V.inv_vs[0], u1 = (S1 - V.lo[1]) * V.inv_vs[1];
    const bool x = fabs(d0) >= fabs(d1);
    const double dm = x ? d0 : d1, dt = x ? d1 : d0, um = x ? u0 : u1, ut = x ? u1 : u0;
    const double vm = x ? V.vs[0] : V.vs[1], vt = x ? V.vs[1] : V.vs[0];
    const int nm = x ? V.n[0] : V.n[1], nt = x ? V.n[1] : V.n[0];
    const double idm = rcp64(dm);
    C.ka = dt * idm;
    C.ika = (dt != 0.0) ? dm * rcp64(dt) : 0.0;
    C.Aa = fma(-C.ka, um, ut);
    double tin = 0.0, tout = (double)nm;
    clip_axis(C.ka, C.ika, C.Aa, 0.0, (double)nt, tin, tout);
    const bool hit = dm != 0.0 && tout > tin;
    const int s0 = max((int)floor(tin), 0), s1 = min((int)ceil(tout), nm);
    const int b = hit ? s0 : 0, e = hit && s1 > s0 ? s1 : b;
    C.slabs = (unsigned)b | (unsigned)e << 15 | (x ? 0u : 1u << 30);
    const int near = dm > 0.0 ? b : e;      // the path's end towards the source
    C.tz = fabs((double)C.tc() - um) > 2.0 * fabs((double)near - um) ? near : C.tc();
    C.dk = V.inv_vs[2] * idm;
    C.dz = C.dk * ((double)C.tz - um);
    const double kt = C.ka * vt;
    C.p2 = fma(kt, kt, vm * vm);
    const double x0 = e0 * V.inv_vs[0], x1 = e1 * V.inv_vs[0];
    C.l2 = fma(x1, x1, x0 * x0);
    return C;
}

// z cells (from the volume's middle one) of a view's source
__device__ __forceinline__ double fan_z0(const VolDev& V, double lift)
{
#pragma clang fp contract(off)
    return (lift - V.lo[2]) * V.inv_vs[2] - (double)(V.n[2] >> 1);
}

// z of a ray over its column's path: z(t) = kz (t - tz) + Zc, in cells from
// the volume's middle cell (nz / 2); ink = 1 / |kz| (capped: a level ray
// never reaches the next cell); scale = mm per slab.
// z carries the rounding of numbers of the size of Zc.  The origin tz is the
// middle of the column's path, or its end towards the source where the middle
// is more than twice as far from the source as that: a steep ray that meets the
// volume near the source is far outside it at the middle, while at the near
// end it is between the source's height and its own.  (The per-ray walk takes
// the middle of each ray's own path.  256 x 256 x 16 voxels, source 62 voxels
// from the volume's face, slopes above 0.2: 4.0e-7 cells rms, about the middle
// 1.4e-6, per ray 4.1e-7; up to a factor of two, as in usual scans, the middle
// costs 1 to 12 %.)  Slope, reciprocal and length per slab are rounded once,
// from FP64.
struct FanRay {
    float kz, Zc, ink, scale;
};

__device__ __forceinline__ FanRay fan_ray(const VolDev& V, const DetDev& G, const FanCol& C, double z0, int ib,
                                          unsigned flags)
{
#pragma clang fp contract(off)
    FanRay r;
    const double b = fma(G.bi + ib, G.db, -(G.nb * G.db * 0.5));
    const double kz = b * C.dk, kv = kz * V.vs[2];
    r.kz = (float)kz;
    r.Zc = (float)fma(b, C.dz, z0);
    // the hardware reciprocal of the FP32 slope and one step towards 1 / |kz|
    const float rough = fminf(__builtin_amdgcn_rcpf(fabsf(r.kz)), 0x1p40f);
    r.ink = fmaf(rough, (float)fma(-fabs(kz), (double)rough, 1.0), rough);
    r.scale = __builtin_amdgcn_sqrtf((float)fma(kv, kv, C.p2));
    if (flags & NEFCT_F_INV_L2) {
        const double zd = b * V.inv_vs[0];
        r.scale = (float)((double)r.scale / fma(zd, zd, C.l2));
    }
    return r;
}

// Paths within 1/64 of a grid axis cross a face so slowly that the rounding of
// an FP32 coordinate (4e-6 cells at 64 cells from the middle) moves the
// crossing by 1e-3 slabs and more.  A ray's own coordinates are rounded about
// the middle of its own path, which differs from its column's where the ray
// leaves the volume in z, so on these paths (2 % of them) the rays work out
// their crossings themselves (FanOwn) and the table holds slabs: f0 = the
// cell before the crossing, dt = which part of the slab (FAN_WHOLE ...).  A
// slab whose faces come within FAN_REACH (relative) of a cell face gets both of
// its parts: a ray may cross there although its column does in the next slab.
constexpr double FAN_SLOW = 1.0 / 64.0;
constexpr float FAN_REACH = 0x1p-20f;   // the two coordinates differ by 4 * 2^-24 of the largest at most
constexpr float FAN_WHOLE = 0.0f, FAN_FIRST = 1.0f, FAN_SECOND = 2.0f, FAN_EMPTY = 3.0f;
__device__ __forceinline__ bool fan_slow(const FanCol& C) { return fabs(C.ka) < FAN_SLOW && C.ka != 0.0; }

// The one or two in-plane pieces of slab t (transverse cells c0 and, past a
// crossing, c1), their lengths and the slab's coordinate (from tz).  A piece of
// no length is dropped.  ha = half the transverse extent.
// The arithmetic is the per-ray walk's (slab_exact: FP32 coordinates from the
// middle of the volume and of the path), so the two walks agree to the last
// bits on a ray that stays inside the volume in z.  Paths near 45 degrees
// (near_unit_slope), whose FP32 face cells can skip one, take FP64 faces; where
// rounding still makes them differ by two, the first piece ends at the first
// boundary and the second takes the rest.
struct FanSlab {
    int c0, c1;
    float d0, d1;
    float ts;
    bool v0, v1;
};

__device__ __forceinline__ FanSlab fan_slab(const FanCol& C, int t, int ha)
{
#pragma clang fp contract(off)
    FanSlab s;
    const float tr = (float)(t - C.tc());
    bool cross;
    if (fabs(C.ka) > (double)K_NEAR_ONE) {
        const double a0 = fma(C.ka, (double)t, C.Aa), a1 = fma(C.ka, (double)(t + 1), C.Aa);
        const double f0 = floor(a0), f1 = floor(a1);
        cross = f0 != f1;
        const double bound = C.ka > 0.0 ? f0 + 1.0 : f0;
        const double fa = cross ? fmin(fmax((bound - a0) * C.ika, 0.0), 1.0) : 1.0;
        s.c0 = (int)f0;
        s.c1 = (int)f1;
        s.d0 = (float)fa;
        s.d1 = (float)(1.0 - fa);
    } else {
        const float ka = (float)C.ka, ika = (float)C.ika, Ac = (float)(fma(C.ka, (double)C.tc(), C.Aa) - ha);
        const float a0 = fmaf(ka, tr, Ac), a1 = fmaf(ka, tr + 1.0f, Ac);
        s.c0 = cell_floor(a0) + ha;
        s.c1 = cell_floor(a1) + ha;
        if (fan_slow(C)) {
            const float reach = FAN_REACH * (fmaxf(fabsf(a0), fabsf(Ac)) + 1.0f);
            const float face = floorf(fmaxf(a0, a1) + reach);
            if (face >= fminf(a0, a1) - reach) {
                s.c0 = (int)face + ha - (ka > 0.0f ? 1 : 0);
                s.c1 = (int)face + ha - (ka > 0.0f ? 0 : 1);
            }
        }
        cross = s.c0 != s.c1;
        s.d0 = cross ? cross_frac(cell_frac(a0), ika, ka > 0.0f ? ika : 0.0f) : 1.0f;
        s.d1 = 1.0f - s.d0;
    }
    s.ts = (float)(t - C.tz);
    const bool in = t >= C.s0() && t < C.s1();
    const bool parts = cross && fan_slow(C);    // both, whatever the column's own lengths
    s.v0 = in && (parts || s.d0 > 0.0f);
    s.v1 = in && cross && (parts || s.d1 > 0.0f);
    return s;
}

// A ray's own in-plane coordinate: a(t) = ka (t - tz - shift) + Ac.
struct FanOwn {
    float ka, ika, pia, Ac, shift;
};

__device__ __forceinline__ FanOwn fan_own(const VolDev& V, const DetDev& G, const FanCol& C, double z0, int ib, int ha)
{
#pragma clang fp contract(off)
    FanOwn w;
    const double b = fma(G.bi + ib, G.db, -(G.nb * G.db * 0.5));
    const double kz = b * C.dk, uz = z0 + (double)(V.n[2] >> 1);
    const double A = fma(b, fma(-C.dk, (double)C.tz, C.dz), uz);      // z at slab face 0
    double tin = 0.0, tout = 16384.0;
    clip_axis(kz, kz != 0.0 ? rcp64(kz) : 0.0, A, 0.0, (double)V.n[2], tin, tout);
    const int s0 = max(C.s0(), (int)floor(fmin(tin, 16384.0))), s1 = min(C.s1(), (int)ceil(fmax(tout, 0.0)));
    const int tc = (s0 + s1) >> 1;
    w.shift = (float)(tc - C.tz);
    w.Ac = (float)(fma(C.ka, (double)tc, C.Aa) - ha);
    w.ka = (float)C.ka;
    w.ika = (float)C.ika;
    w.pia = w.ka > 0.0f ? w.ika : 0.0f;
    return w;
}

// Column records of every view, if the call has room for them, else null.
__device__ __forceinline__ FanCol fan_col(const Launch& P, int iv, int ia)
{
    if (P.cols) return ((const FanCol*)P.cols)[(size_t)iv * P.G.na + ia];
    return fan_column(P.V, P.G, P.trig[2 * iv], P.trig[2 * iv + 1], ia);
}

__global__ __launch_bounds__(256) void k_fan_cols(Launch P, FanCol* __restrict__ cols)
{
    const int ia = blockIdx.x * 256 + threadIdx.x, iv = blockIdx.y;
    if (ia < P.G.na) cols[(size_t)iv * P.G.na + ia] = fan_column(P.V, P.G, P.trig[2 * iv], P.trig[2 * iv + 1], ia);
}

// Fills the records at p (which has `room` bytes) and points the launch at them.
void launch_fan_cols(Launch& L, char* p, size_t room, hipStream_t s)
{
    L.cols = nullptr;
    if (!p || sizeof(FanCol) * (size_t)L.G.na * (size_t)L.nv > room) return;
    hipLaunchKernelGGL(k_fan_cols, dim3((L.G.na + 255) / 256, L.nv), dim3(256), 0, s, L, (FanCol*)p);
    L.cols = p;
}

// A piece in LDS: its slab's coordinate, the part [f0, f0 + dt] of the slab,
// the byte offset of its cell's z row.
struct __align__(16) FanSeg {
    float ts, f0, dt;
    int off;
};

// The entry of a slab's part on a slow path (see FAN_SLOW), and a ray's own
// piece from it.
__device__ __forceinline__ FanSeg fan_seg(const FanSlab& s, bool second, bool slow, int ha, int off)
{
    if (slow)
        return FanSeg{s.ts, (float)(s.c0 - ha), second ? FAN_SECOND : s.c0 == s.c1 ? FAN_WHOLE : FAN_FIRST, off};
    return FanSeg{s.ts, second ? s.d0 : 0.0f, second ? s.d1 : s.d0, off};
}

// (slow: this lane's column; the entry of another column is a piece already)
__device__ __forceinline__ FanSeg fan_own_seg(const FanSeg& e, const FanOwn& w, bool slow)
{
    // (by the cells of the slab's two faces, as the per-ray walk finds a crossing)
    const float a0 = fmaf(w.ka, e.ts - w.shift, w.Ac), a1 = fmaf(w.ka, e.ts - w.shift + 1.0f, w.Ac);
    const float fa = e.dt == FAN_WHOLE || floorf(a1) == e.f0 ? 1.0f
                     : floorf(a0) != e.f0                    ? 0.0f
                                                             : cross_frac(a0 - e.f0, w.ika, w.pia);
    FanSeg r;
    r.ts = e.ts;
    r.f0 = !slow ? e.f0 : e.dt == FAN_SECOND ? fa : 0.0f;
    r.dt = !slow ? e.dt : e.dt == FAN_EMPTY ? 0.0f : e.dt == FAN_SECOND ? 1.0f - fa : fa;
    r.off = e.off;
    return r;
}

// The fraction of a slab that a ray takes to its next z face, from z at the
// slab's face (unclamped).  SIGN: rising (1), falling (-1) or either (0).
template <int SIGN>
__device__ __forceinline__ float fan_z_frac(float z, float kz, float ink)
{
    const float fr = cell_frac(z);
    if (SIGN > 0) return fmaf(fr, -ink, ink);
    if (SIGN < 0) return fr * ink;
    return fmaf(fr, kz < 0.0f ? ink : -ink, kz < 0.0f ? 0.0f : ink);
}

// ---------------------------------------------------------------------------
// Forward
// ---------------------------------------------------------------------------
// z-fastest copy of the volume: cell (x, y) at (x + nx y) (nz + 4) floats,
// its z row inside a border of two zeros on either side, so that the clamped
// cells -2 .. nz and the cell above each need no test.
__host__ __device__ inline int fan_row(int nz) { return nz + 2 * FAN_ZPAD; }

// Builds the copy through 64 x 64 LDS tiles (x and z of one y) and, in its
// first blocks, the view table.
__global__ __launch_bounds__(256) void k_fan_prep(const float* __restrict__ img, int nx, int ny, int nz,
                                                  float* __restrict__ out, int tx, int tz,
                                                  const float* __restrict__ angles, int nv, double* __restrict__ trig,
                                                  int trig_blocks)
{
    if ((int)blockIdx.x < trig_blocks) {
        const int i = blockIdx.x * 256 + threadIdx.x;
        if (i < nv) {
            const double a = (double)angles[i];
            trig[2 * i] = cos(a);
            trig[2 * i + 1] = sin(a);
        }
        return;
    }
    __shared__ float tile[64][65];
    const int b = (int)blockIdx.x - trig_blocks;
    const int bx = b % tx, by = (b / tx) % ny, bz = b / (tx * ny);
    const int lx = threadIdx.x & 63, ly = threadIdx.x >> 6;
    const int ix = bx * 64 + lx;
    const int row = fan_row(nz);
#pragma unroll 4
    for (int r = ly; r < 64; r += 4) {
        const int iz = bz * 64 + r - FAN_ZPAD;
        float v = 0.0f;
        if (ix < nx && iz >= 0 && iz < nz) v = img[(size_t)ix + (size_t)nx * ((size_t)by + (size_t)ny * iz)];
        tile[r][lx] = v;
    }
    __syncthreads();
#pragma unroll 4
    for (int r = ly; r < 64; r += 4) {
        const int x = bx * 64 + r, p = bz * 64 + lx;
        if (x < nx && p < row) out[((size_t)x + (size_t)nx * by) * row + p] = tile[lx][r];
    }
}

void launch_fan_prep(const float* image, const int grid[3], float* copy, const float* angles, int nv, double* trig,
                     hipStream_t s)
{
    const int tx = (grid[0] + 63) / 64, tz = (fan_row(grid[2]) + 63) / 64;
    const int tb = trig ? (nv + 255) / 256 : 0;
    hipLaunchKernelGGL(k_fan_prep, dim3((unsigned)(tb + (long long)tx * grid[1] * tz)), dim3(256), 0, s, image,
                       grid[0], grid[1], grid[2], copy, tx, tz, angles, nv, trig, tb);
}

constexpr int FAN_TAB = 128 + 4;    // pieces of 64 slabs, and a tail of empty ones
constexpr int FAN_U = 4;            // pieces per trip: their loads are in flight together
constexpr int FAN_FW = 4;           // forward: wavefronts (= detector columns) per workgroup

// acc += the z integrals of the table's n pieces.
// CLAMP: rays may leave the volume in z (z clamped into the zero border).
// rs1 is the copy from its second value on, or (SIGN < 0) rs is and rs1 is the
// copy: the next cell through a resource of its own keeps the two loads apart
// (as one 8-byte load they take 16 clocks of the CU's vector cache against 5
// for each 4-byte load of a wavefront).
// CAREFUL: a cell met with no length is not read into the sum (0 x NaN).
// SIGN: the wavefront's rays all rise (1), all fall (-1) or both (0).
// SLOW: the table holds slabs, the ray its own crossings.
template <bool CLAMP, bool CAREFUL, int SIGN, bool SLOW>
__device__ __forceinline__ float fan_forward_pieces(const FanSeg* __restrict__ tab, int n, float kz, float Zc,
                                                    float ink, float zlo, float zhi, __amdgpu_buffer_rsrc_t rs,
                                                    __amdgpu_buffer_rsrc_t rs1, const FanOwn& own, float acc)
{
    for (int j = 0; j < n; j += FAN_U) {
        float v0[FAN_U], v1[FAN_U], l[FAN_U], h[FAN_U];
#pragma unroll
        for (int u = 0; u < FAN_U; ++u) {
            FanSeg s = tab[j + u];
            if (SLOW) s = fan_own_seg(s, own, true);
            float z = fmaf(kz, s.ts, Zc);
            if (CLAMP) z = __builtin_amdgcn_fmed3f(z, zlo, zhi);
            // (falling: from the cell below, the first of the two in memory)
            const int o = s.off + (cell_floor(z) << 2) - (SIGN < 0 ? 4 : 0);
            l[u] = __builtin_amdgcn_fmed3f(fan_z_frac<SIGN>(z, kz, ink) - s.f0, 0.0f, s.dt);
            h[u] = s.dt - l[u];
            v0[u] = buf_load(rs, o);
            v1[u] = buf_load(rs1, SIGN == 0 ? o + (kz < 0.0f ? -8 : 0) : o);
        }
#pragma unroll
        for (int u = 0; u < FAN_U; ++u) {
            if (CAREFUL) {
                // selected as integers: the compiler may take float data to be no NaN
                const int w0 = l[u] > 0.0f ? __builtin_bit_cast(int, v0[u]) : 0;
                const int w1 = h[u] > 0.0f ? __builtin_bit_cast(int, v1[u]) : 0;
                acc = fmaf(l[u], __builtin_bit_cast(float, w0), acc);
                acc = fmaf(h[u], __builtin_bit_cast(float, w1), acc);
            } else {
                acc = fmaf(l[u], v0[u], acc);
                acc = fmaf(h[u], v1[u], acc);
            }
        }
    }
    return acc;
}

// One wavefront: detector column ia, rows ib0 + lane of view iv.
__device__ __forceinline__ void fan_forward_wave(const Launch& P, int ia, int ib0, int iv, FanSeg* __restrict__ tab,
                                                 float* __restrict__ out)
{
    const int lane = threadIdx.x & 63;
    const VolDev& V = P.V;
    const DetDev& G = P.G;
    const FanCol C = fan_col(P, iv, ia);
    const int nx = V.n[0], ny = V.n[1], nz = V.n[2], hz = nz >> 1, row4 = 4 * fan_row(nz);
    const int ib = ib0 + lane;
    const double vz0 = fan_z0(V, view_lift(P, iv));
    const FanRay q = fan_ray(V, G, C, vz0, min(ib, G.nb - 1), P.flags);
    const int ha = (C.m() == 0 ? ny : nx) >> 1;
    const bool slow = fan_slow(C);
    FanOwn own = {};
    if (slow) own = fan_own(V, G, C, vz0, min(ib, G.nb - 1), ha);
    float kz = q.kz, Zc = q.Zc, ink = q.ink;
    float lo = 3.0e38f, hi = -3.0e38f;      // slabs (from tz) that some ray spends inside the volume
    bool rests = false;
    const float e0 = (float)(C.s0() - C.tz), e1 = (float)(C.s1() - C.tz);
    const float zlo = (float)(-hz) - 0.0625f, zhi = (float)(nz - hz) + 0.0625f;
    {
        const float za = fmaf(kz, e0, Zc), zb = fmaf(kz, e1, Zc);
        if (C.s1() > C.s0() && ib < G.nb && fmaxf(za, zb) > zlo && fminf(za, zb) < zhi) {
            // slab coordinates where z passes the (widened) faces; |kz| < 2^-20 stays inside or outside
            lo = e0;
            hi = e1;
            if (fabsf(kz) > 0x1p-20f) {
                const float k = kz < 0.0f ? -ink : ink;
                const float ta = (zlo - Zc) * k, tb = (zhi - Zc) * k;
                lo = fmaxf(lo, fminf(ta, tb) - 1.0f);
                hi = fminf(hi, fmaxf(ta, tb) + 1.0f);
            }
        } else {            // rests in the zero border
            rests = true;
            kz = 0.0f;
            Zc = (float)(-hz - FAN_ZPAD);
            ink = 0x1p40f;
        }
    }
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) {
        lo = fminf(lo, __shfl_xor(lo, o, 64));
        hi = fmaxf(hi, __shfl_xor(hi, o, 64));
    }
    lo = __builtin_bit_cast(float, __builtin_amdgcn_readfirstlane(__builtin_bit_cast(int, lo)));
    hi = __builtin_bit_cast(float, __builtin_amdgcn_readfirstlane(__builtin_bit_cast(int, hi)));
    float acc = 0.0f;
    if (lo < hi) {
        const int t0 = __builtin_amdgcn_readfirstlane(max(C.s0(), C.tz + (int)floorf(lo)));
        const int t1 = __builtin_amdgcn_readfirstlane(min(C.s1(), C.tz + (int)ceilf(hi)));
        const float w0 = (float)(t0 - C.tz), w1 = (float)(t1 - C.tz);
        const float za = fmaf(kz, w0, Zc), zb = fmaf(kz, w1, Zc);
        // no ray's two cells leave -2 .. nz + 1 over [t0, t1]: no clamp
        const float down = kz < 0.0f ? 1.0f : 0.0f;
        const float clo = (float)(-hz - FAN_ZPAD) + down, chi = (float)(nz - hz) + 0.5f + down;
        const bool clamp = !__all(fminf(za, zb) >= clo && fmaxf(za, zb) < chi);
        const bool rise = __all(kz >= 0.0f), fall = __all(kz < 0.0f || rests);     // (a level ray rises)
        const uint32_t bytes = (uint32_t)nx * (uint32_t)ny * (uint32_t)row4;
        const __amdgpu_buffer_rsrc_t rs = make_rsrc(P.Ly.xf, bytes), rs1 = make_rsrc(P.Ly.xf + 1, bytes - 4);
        auto walk = [&](auto careful_tag) {
            constexpr bool CAREFUL = decltype(careful_tag)::value;
            acc = 0.0f;
            for (int tb = t0; tb < t1; tb += 64) {
                // the pieces of slabs tb .. tb + 63, one lane per slab
                const int t = tb + lane;
                FanSlab s = fan_slab(C, t, ha);
                const bool mx = C.m() == 0;
                const int na = mx ? ny : nx;
                s.v0 = s.v0 && t < t1 && (unsigned)s.c0 < (unsigned)na;
                s.v1 = s.v1 && t < t1 && (unsigned)s.c1 < (unsigned)na;
                const unsigned long long b0 = __builtin_amdgcn_ballot_w64(s.v0), b1 = __builtin_amdgcn_ballot_w64(s.v1);
                const unsigned long long below = (1ull << lane) - 1ull;
                int p = __popcll(b0 & below) + __popcll(b1 & below);
                const int n = __popcll(b0) + __popcll(b1);
                const int base = 4 * (hz + FAN_ZPAD);
                const int ct = mx ? nx : 1, mt = mx ? 1 : nx;      // cell strides of a and of t
                __builtin_amdgcn_wave_barrier();
                const int o0 = (s.c0 * ct + t * mt) * row4 + base, o1 = (s.c1 * ct + t * mt) * row4 + base;
                if (s.v0) tab[p++] = fan_seg(s, false, slow, ha, o0);
                if (s.v1) tab[p++] = fan_seg(s, true, slow, ha, o1);
                // the lane of the last piece adds empty ones in its slab, up to whole trips
                if ((s.v0 || s.v1) && p == n) {
#pragma unroll
                    for (int u = 0; u < FAN_U - 1; ++u) tab[n + u] = FanSeg{s.ts, 0.0f, slow ? FAN_EMPTY : 0.0f, base};
                }
                __builtin_amdgcn_wave_barrier();
                auto pieces = [&](auto clamp_tag, auto sign_tag) {
                    constexpr int SIGN = decltype(sign_tag)::value;
                    acc = fan_forward_pieces<decltype(clamp_tag)::value, CAREFUL, SIGN, false>(
                        tab, n, kz, Zc, ink, clo, chi, SIGN < 0 ? rs1 : rs, SIGN < 0 ? rs : rs1, own, acc);
                };
                using Mixed = std::integral_constant<int, 0>;
                using Rise = std::integral_constant<int, 1>;
                using Fall = std::integral_constant<int, -1>;
                if (slow)
                    acc = fan_forward_pieces<true, CAREFUL, 0, true>(tab, n, kz, Zc, ink, clo, chi, rs, rs1, own, acc);
                else if (CAREFUL || !(rise || fall))
                    pieces(std::true_type{}, Mixed{});
                else if (clamp)
                    rise ? pieces(std::true_type{}, Rise{}) : pieces(std::true_type{}, Fall{});
                else
                    rise ? pieces(std::false_type{}, Rise{}) : pieces(std::false_type{}, Fall{});
            }
        };
        walk(std::false_type{});
        // An infinity or NaN in a cell that a ray only touches (a product 0 x
        // Inf) must not reach its sum: a wavefront that ends with a non-finite
        // sum walks again, reading only cells met with some length.
        unsigned bits = __builtin_bit_cast(unsigned, acc);
        asm("" : "+v"(bits));       // (opaque: the compiler may take a float to be no NaN)
        if (__any((bits & 0x7f800000u) == 0x7f800000u)) walk(std::true_type{});
    }
    if (ib < G.nb) out[(size_t)ia + (size_t)G.na * ((size_t)ib + (size_t)G.nb * (size_t)iv)] = acc * q.scale;
}

// Task order as k_siddon's, with tiles of FAN_FW columns x 64 rows.  Held to
// eight wavefronts per SIMD (64 registers; with 68 the 512 x 512 x 256 forward
// takes 4 % longer).
__global__ __launch_bounds__(64 * FAN_FW, 8) void k_fan_fwd(Launch P, float* __restrict__ out, int tiles_a, int tiles_b,
                                                           int v0, int nvc, int vg_log2)
{
    __shared__ FanSeg tabs[FAN_FW][FAN_TAB];
    const unsigned per_xcd = gridDim.x >> 3;
    const unsigned task = (blockIdx.x & 7u) * per_xcd + (blockIdx.x >> 3);
    const unsigned tiles = (unsigned)tiles_a * (unsigned)tiles_b;
    const unsigned vin = task & ((1u << vg_log2) - 1u), rest = task >> vg_log2;
    const unsigned tile = rest % tiles, group = rest / tiles;
    const int iv = (int)((group << vg_log2) + vin);
    const int wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int ia = (int)(tile % (unsigned)tiles_a) * FAN_FW + wv;
    if (iv >= nvc || ia >= P.G.na) return;      // no barrier in this kernel
    fan_forward_wave(P, ia, (int)(tile / (unsigned)tiles_a) * 64, v0 + iv, tabs[wv], out);
}

void launch_fan_fwd(const Launch& L, float* out, int vgl, hipStream_t s)
{
    const int ta = (L.G.na + FAN_FW - 1) / FAN_FW, tb = (L.G.nb + 63) / 64;
    const long long tiles = (long long)ta * tb;
    const int vg = 1 << vgl;
    // 1-D grids below 2^31 work-items
    long long max_groups = (0x7fffffffll / (64 * FAN_FW)) / (tiles * vg);
    if (max_groups < 1) max_groups = 1;
    const int chunk = (int)std::min<long long>(L.nv, max_groups * vg);
    for (int v0 = 0; v0 < L.nv; v0 += chunk) {
        const int nvc = std::min(chunk, L.nv - v0);
        const long long groups = (nvc + vg - 1) / vg;
        const long long blocks = (tiles * groups * vg + 7) / 8 * 8;
        hipLaunchKernelGGL(k_fan_fwd, dim3((unsigned)blocks), dim3(64 * FAN_FW), 0, s, L, out, ta, tb, v0, nvc, vgl);
    }
}

// ---------------------------------------------------------------------------
// Adjoint
// ---------------------------------------------------------------------------
// A workgroup owns FB x FB columns of voxels, at most TZ tall (TZ x 256 words
// beside the tables fill the LDS), in LDS (64-bit
// fixed point, z fastest, FAN_HALO spare words on either side of a column's z
// run, shared with the neighbouring columns', for deposits that leave the
// block: a ray drifts a few cells in z over a block's width).
// Its wavefronts take four neighbouring detector columns of a view at a time:
// first 16 lanes per column tabulate the column's pieces inside the block
// (one lane per slab), then the lanes deal out the rows that can reach the
// block, 16 rows of each of the four columns at once, and walk their rays.
// No barrier is needed between views: a table belongs to its wavefront.
constexpr int FB = 16;
constexpr int FAN_ENT = 2 * FB;     // table entries per column: two per slab at most, and an empty one after an odd count

constexpr int FAN_HALO = 6;

template <int TZ, typename T>
struct FanAcc {
    static constexpr int ROW = TZ + FAN_HALO;           // words per column
    static constexpr int NEL = FB * FB * ROW + FAN_HALO;
    T v[NEL];
};

// z extent of the block's columns: the volume's height in equal parts of at most tz
__host__ __device__ inline int fan_zblocks(int nz, int tz) { return (nz + tz - 1) / tz; }

template <bool FIX, int TZ, int NW>
__device__ __forceinline__ void fan_adjoint_block(const Launch& P, const float* __restrict__ pv,
                                                  float* __restrict__ image, unsigned long long* __restrict__ sums,
                                                  int bx, int by, int bz, int nbz, int v0, int v1,
                                                  FanAcc<TZ, acc_t<FIX>>& acc, FanSeg (&tabs)[NW][4][FAN_ENT],
                                                  int4 (&shadows)[SHV], int2 (&deals)[SHV], int es)
{
    using T = acc_t<FIX>;
    constexpr int ROW = FanAcc<TZ, T>::ROW;
    constexpr int ES = (int)sizeof(T);
    const VolDev& V = P.V;
    const DetDev& G = P.G;
    const int tid = threadIdx.x, lane = tid & 63;
    const int wv = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int nx = V.n[0], ny = V.n[1], nz = V.n[2], hz = nz >> 1;
    const int x0 = bx * FB, y0 = by * FB, z0 = (int)((long long)nz * bz / nbz), z1 = (int)((long long)nz * (bz + 1) / nbz);
    const int b0[3] = {x0, y0, z0}, b1[3] = {min(x0 + FB, nx), min(y0 + FB, ny), z1};
    for (int i = tid; i < FanAcc<TZ, T>::NEL; i += 64 * NW) acc.v[i] = (T)0;
    const int col = lane >> 4, sl = lane & 15;
    FanSeg* const tab = tabs[wv][col];
    char* const ab = reinterpret_cast<char*>(acc.v);
    // byte offset of centred cell 0 of the block's first column
    const int org = ES * (FAN_HALO - (z0 - hz));
    // z range of a pair's lower cell within the spare words (no test), and as
    // a range of cells
    const float clo = (float)(z0 - hz - FAN_HALO), chi = (float)(z1 - hz + FAN_HALO - 1);
    const int ilo = z0 - hz - 1;
    const unsigned span = (unsigned)(z1 - z0);      // lower cells -1 .. height - 1 of the block
    // where a lane without a ray adds its zeros: a word of its own among 16
    const float rest = fminf(clo + (float)sl, chi - 0.5f);
    const float zlo = (float)(z0 - hz) - 0.0625f, zhi = (float)(z1 - hz) + 0.0625f;
    int turn = 0;       // units dealt out so far, modulo NW
    for (int iv = v0; iv < v1; ++iv) {
        const int slot = (iv - v0) % SHV;
        if (slot == 0) {
            __syncthreads();    // (and the accumulators' clearing, the first time)
            const int n = min(SHV, v1 - iv);
            for (int e = tid >> 3; e < n; e += 8 * NW) {
                const int4 sh = shadow_of_box(V, G, P.trig[2 * (iv + e)], P.trig[2 * (iv + e) + 1], b0, b1, true,
                                              tid & 7, view_lift(P, iv + e));
                if ((tid & 7) == 0) {
                    shadows[e] = sh;
                    const int H = max(sh.w - sh.z + 1, 1), cs = min(max((H + z1 - z0 - 4) / (z1 - z0), 1), H);
                    deals[e] = make_int2(cs, (H + cs - 1) / cs);
                }
            }
            __syncthreads();
        }
        const int4 sh = shadows[slot];
        const int ia0 = __builtin_amdgcn_readfirstlane(sh.x), ia1 = __builtin_amdgcn_readfirstlane(sh.y);
        const int ib0 = __builtin_amdgcn_readfirstlane(sh.z), ib1 = __builtin_amdgcn_readfirstlane(sh.w);
        if (ia1 < ia0 || ib1 < ib0) continue;
        const int units = (ia1 - ia0 + 4) >> 2;
        int g = wv - turn;
        g = g < 0 ? g + NW : g;
        turn = (turn + units) % NW;
        if (g >= units) continue;
        const double vz0 = fan_z0(V, view_lift(P, iv));
        // Rows are dealt with at least a voxel (at most two) between
        // neighbouring lanes: two of 16 lanes that deposit into one word
        // double the time of the whole addition (12.3 against 6.4 clocks of
        // the CU per wavefront; strides of one to two words cost 6.4 to 8.3).
        // Row index f = phase * HC + q is row q * cs + phase.
        const int cs = __builtin_amdgcn_readfirstlane(deals[slot].x), HC = __builtin_amdgcn_readfirstlane(deals[slot].y);
        const int nf = HC * cs;
        const float* __restrict__ pvv = pv + (size_t)G.na * (size_t)G.nb * (size_t)iv;
        for (; g < units; g += NW) {
            const int ia = ia0 + 4 * g + col;
            const FanCol C = fan_col(P, iv, min(ia, G.na - 1));
            const int ha = (C.m() == 0 ? ny : nx) >> 1;
            // the group walks as its slow columns need; every column keeps its
            // own rule, whichever neighbours a block deals it with
            const bool slow = fan_slow(C), any_slow = __any(slow);
            int n;
            float ta, tb;       // slab coordinates of the path's ends inside the block
            {
                // pieces of four columns, one lane per column and slab
                const int m0 = C.m() == 0 ? x0 : y0, m1 = C.m() == 0 ? b1[0] : b1[1];
                const int a0 = C.m() == 0 ? y0 : x0, a1 = C.m() == 0 ? b1[1] : b1[0];
                const int t = m0 + sl;
                FanSlab q = fan_slab(C, t, ha);
                const bool on = ia <= ia1 && t < m1;
                q.v0 = q.v0 && on && q.c0 >= a0 && q.c0 < a1;
                q.v1 = q.v1 && on && q.c1 >= a0 && q.c1 < a1;
                const unsigned long long w0 = __builtin_amdgcn_ballot_w64(q.v0), w1 = __builtin_amdgcn_ballot_w64(q.v1);
                const unsigned k0 = (unsigned)(w0 >> (lane & 48)) & 0xffffu, k1 = (unsigned)(w1 >> (lane & 48)) & 0xffffu;
                const unsigned below = (1u << sl) - 1u;
                int p = __popc(k0 & below) + __popc(k1 & below);
                n = __popc(k0) + __popc(k1);
                const int ct = C.m() == 0 ? FB : 1, mt = C.m() == 0 ? 1 : FB;
                const int cell0 = ((q.c0 - a0) * ct + sl * mt) * (ROW * ES) + org;
                const int cell1 = ((q.c1 - a0) * ct + sl * mt) * (ROW * ES) + org;
                __builtin_amdgcn_wave_barrier();
                if (q.v0) tab[p++] = fan_seg(q, false, slow, ha, cell0);
                if (q.v1) tab[p++] = fan_seg(q, true, slow, ha, cell1);
                // an empty piece in the last one's slab makes the count even
                if ((q.v0 || q.v1) && p == n && n < FAN_ENT)
                    tab[n] = FanSeg{q.ts, 0.0f, slow ? FAN_EMPTY : 0.0f, q.v1 ? cell1 : cell0};
                __builtin_amdgcn_wave_barrier();
                ta = tab[0].ts;
                tb = tab[max(n - 1, 0)].ts + 1.0f;
            }
            const float* __restrict__ pc = pvv + min(ia, G.na - 1);
            // the lane's place in the dealing: q of its phase, detector row
            int q = sl, ib = ib0 + sl * cs;
            {
                auto rays = [&](int f0, auto rows_tag, auto slow_tag) {
                    constexpr int R = decltype(rows_tag)::value;
                    constexpr bool SLOW = decltype(slow_tag)::value;
                    float kz[R], Zc[R], ik[R], sv[R];
                    FanOwn own[SLOW ? R : 1];
                    bool any = false, in = true, nonneg = true, rise = true, fall = true;
#pragma unroll
                    for (int r = 0; r < R; ++r) {
                        while (__any(q >= HC)) {    // the next phase
                            ib = q >= HC ? ib + 1 - HC * cs : ib;
                            q = q >= HC ? q - HC : q;
                        }
                        bool live = f0 + 16 * r + sl < nf && ib <= ib1 && n > 0;
                        const float pval = live ? pc[__umul24((unsigned)ib, (unsigned)G.na)] : 0.0f;
                        const FanRay y = fan_ray(V, G, C, vz0, ib, P.flags);
                        if constexpr (SLOW) own[r] = fan_own(V, G, C, vz0, ib, ha);
                        q += 16;
                        ib += 16 * cs;
                        const float za = fmaf(y.kz, ta, y.Zc), zb = fmaf(y.kz, tb, y.Zc);
                        const float z_lo = fminf(za, zb), z_hi = fmaxf(za, zb);
                        sv[r] = FIX ? ldexpf(pval * y.scale, es) : pval * y.scale;
                        live = live && z_hi > zlo && z_lo < zhi && sv[r] != 0.0f;
                        sv[r] = live ? sv[r] : 0.0f;
                        kz[r] = live ? y.kz : 0.0f;
                        Zc[r] = live ? y.Zc : rest;
                        ik[r] = FIX ? y.ink * sv[r] : y.ink;
                        // every deposit of the ray within the spare words: no test
                        in = in && (!live || (z_lo >= clo + 1.0f && z_hi < chi));
                        nonneg = nonneg && sv[r] >= 0.0f;
                        rise = rise && kz[r] >= 0.0f;
                        fall = fall && (kz[r] < 0.0f || !live);     // (a level ray rises)
                        any = any || live;
                    }
                    if (!__any(any)) return;
                    // SIGN: the rays all rise (1) or fall (-1) in z, or both (0)
                    auto walk = [&](auto nonneg_tag, auto test_tag, auto sign_tag) {
                        constexpr bool NONNEG = decltype(nonneg_tag)::value;
                        constexpr bool TEST = decltype(test_tag)::value;
                        constexpr int SIGN = decltype(sign_tag)::value;
                        auto deposit = [&](int o, int q) {
                            if constexpr (NONNEG) lds_deposit_q(ab, o, q, 0);
                            else lds_deposit_s(ab, o, q);
                        };
                        auto piece = [&](const FanSeg& entry) {
#pragma unroll
                            for (int r = 0; r < R; ++r) {
                                FanSeg e = entry;
                                if constexpr (SLOW) e = fan_own_seg(entry, own[r], slow);
                                const float z = fmaf(kz[r], e.ts, Zc[r]);
                                const int cz = cell_floor(z);
                                const int o = e.off + cz * ES;
                                const bool down = SIGN < 0 || (SIGN == 0 && kz[r] < 0.0f);
                                const int next = down ? -ES : ES;
                                // (masked, not clamped to a spare word, which
                                // would put many lanes on one word)
                                const bool ok = !TEST || (unsigned)(cz - ilo - (down ? 1 : 0)) <= span;
                                if constexpr (FIX) {
                                    // units of the whole piece to the nearest, the
                                    // first cell's cut, the rest to the next cell:
                                    // a piece keeps its length (cut apart, the two
                                    // lost up to a unit each, and with one value 1e5
                                    // times the others the image was 1.6e-4 too small)
                                    const float half = NONNEG ? 0.5f : copysignf(0.5f, sv[r]);
                                    const float whole = fmaf(e.dt, sv[r], half);
                                    const float raw = fmaf(-e.f0, sv[r], fan_z_frac<SIGN>(z, kz[r], ik[r]));
                                    const float part = __builtin_amdgcn_fmed3f(raw, half, whole);
                                    const int q = (int)part;
                                    if (ok) deposit(o, q);
                                    if (ok && part != whole) deposit(o + next, (int)whole - q);
                                } else {
                                    const float raw = fan_z_frac<SIGN>(z, kz[r], ik[r]) - e.f0;
                                    const float l = __builtin_amdgcn_fmed3f(raw, 0.0f, e.dt), h = e.dt - l;
                                    if (ok && l > 0.0f) lds_deposit<FIX>(ab, o, l * sv[r]);
                                    if (ok && h > 0.0f) lds_deposit<FIX>(ab, o + next, h * sv[r]);
                                }
                            }
                        };
                        for (int j = 0; j < n; j += 2) {
                            const FanSeg e0 = tab[j], e1 = tab[j + 1];
                            piece(e0);
                            piece(e1);
                        }
                    };
                    using Rise = std::integral_constant<int, 1>;
                    using Fall = std::integral_constant<int, -1>;
                    auto walk_sign = [&](auto nonneg_tag, auto sign_tag) {
                        if (__all(in)) walk(nonneg_tag, std::false_type{}, sign_tag);
                        else walk(nonneg_tag, std::true_type{}, sign_tag);
                    };
                    if (!FIX || SLOW || !(__all(rise) || __all(fall))) {
                        walk(std::false_type{}, std::true_type{}, std::integral_constant<int, 0>{});
                    } else if (__all(nonneg)) {
                        if (__all(rise)) walk_sign(std::true_type{}, Rise{});
                        else walk_sign(std::true_type{}, Fall{});
                    } else {
                        if (__all(rise)) walk_sign(std::false_type{}, Rise{});
                        else walk_sign(std::false_type{}, Fall{});
                    }
                };
                int f0 = 0;
                using R1 = std::integral_constant<int, 1>;
                using R2 = std::integral_constant<int, 2>;
                using R4 = std::integral_constant<int, 4>;
                if (any_slow) {
                    for (; f0 < nf; f0 += 16) rays(f0, R1{}, std::true_type{});
                } else {
                    for (; nf - f0 > 48; f0 += 64) rays(f0, R4{}, std::false_type{});
                    for (; nf - f0 > 16; f0 += 32) rays(f0, R2{}, std::false_type{});
                    if (f0 < nf) rays(f0, R1{}, std::false_type{});
                }
            }
        }
    }
    __syncthreads();
    const bool poisoned = FIX && es == FIX_POISON;
    const double inv_s = (FIX && !poisoned) ? ldexp(1.0, -es) : 1.0;
    const int bh = z1 - z0;
    for (int i = tid; i < FB * FB * bh; i += 64 * NW) {
        const int lx = i % FB, ly = (i / FB) % FB, lz = i / (FB * FB);
        if (x0 + lx >= nx || y0 + ly >= ny) continue;
        const size_t o = (size_t)(x0 + lx) + (size_t)nx * ((size_t)(y0 + ly) + (size_t)ny * (size_t)(z0 + lz));
        const T v = acc.v[(ly * FB + lx) * ROW + FAN_HALO + lz];
        if constexpr (FIX) {
            if (sums) {     // one of several view ranges: integer sums, whose order does not matter
                if (v != 0ull) atomicAdd(sums + o, v);
                continue;
            }
            if (poisoned)
                reinterpret_cast<unsigned*>(image)[o] = 0x7fc00000u;
            else
                image[o] = (float)((double)(long long)v * inv_s);
        } else {
            image[o] = v;
        }
    }
}

template <bool FIX, int TZ, int NW>
__global__ __launch_bounds__(64 * NW, 4) void k_fan_adj(Launch P, const float* __restrict__ pv,
                                                       float* __restrict__ image,
                                                       unsigned long long* __restrict__ sums, int nsplit,
                                                       const unsigned* __restrict__ maxbits)
{
    __shared__ FanAcc<TZ, acc_t<FIX>> acc;
    __shared__ FanSeg tabs[NW][4][FAN_ENT];
    __shared__ int4 shadows[SHV];
    __shared__ int2 deals[SHV];     // row spacing and rows per phase of each view's dealing
    const int es = FIX ? fixed_exp(*maxbits, P.sbound) : 0;
    const int nbz = gridDim.z / nsplit;
    const int bz = blockIdx.z % nbz, part = blockIdx.z / nbz;
    const int v0 = (int)((long long)P.nv * part / nsplit), v1 = (int)((long long)P.nv * (part + 1) / nsplit);
    fan_adjoint_block<FIX, TZ, NW>(P, pv, image, sums, blockIdx.x, blockIdx.y, bz, nbz, v0, v1, acc, tabs, shadows,
                                   deals, es);
}

constexpr int FAN_TZ = 52;      // tallest block of the fixed-point and float adjoints
constexpr int FAN_NW = 16;

// sums: a split's scratch (cleared by k_absmax), or null without one
void launch_fan_adj(const Launch& L, const float* pv, float* image, unsigned long long* sums, int nsplit,
                    const unsigned* maxbits, hipStream_t s)
{
    const int nbz = fan_zblocks(L.V.n[2], FAN_TZ);
    const dim3 g((L.V.n[0] + FB - 1) / FB, (L.V.n[1] + FB - 1) / FB, nbz * nsplit);
    if (L.flags & NEFCT_F_ADJ_FLOAT_ATOMIC) {
        hipLaunchKernelGGL((k_fan_adj<false, FAN_TZ, FAN_NW>), g, dim3(64 * FAN_NW), 0, s, L, pv, image, nullptr, 1,
                           maxbits);
        return;
    }
    hipLaunchKernelGGL((k_fan_adj<true, FAN_TZ, FAN_NW>), g, dim3(64 * FAN_NW), 0, s, L, pv, image,
                       sums, nsplit, maxbits);
    if (sums) launch_split_sums(L, sums, maxbits, image, s);
}
