// 2.5-D z-marching kernels of the 3-D acoustic path (fixed orders 2..8).
//
// A workgroup of 256 lanes (4 wave64s) owns a 64 (x) by TY (y) tile of
// columns and marches down a segment of z planes.  Each lane keeps, for each
// of its RY = TY/4 rows, the column's 2M+1 z-taps in a register queue; the
// current (x, y) plane of the tile plus an M-cell halo on each side sits in
// LDS for the x- and y-taps.  The LDS plane is double-buffered, so one
// workgroup barrier per plane orders its writes against the reads of the
// plane before.  The loads of plane z+1 (queue head, halos, the other
// fields) are issued before plane z is computed.  Per cell that is one HBM
// read per field read and one write per field written; halo cells come from
// L2.
//
// The computed box is cut into a lean interior -- [lo + M + 1, hi - M - 1)
// per axis: no forward CPML term, no strip cell, no adjoint CPML term (the
// adjoint's pure region) -- and the margins around it, grouped by the axes
// whose CPML margin they lie in (eight types, the interior included).  One
// launch per step runs every type: a workgroup looks its tile up in the plan
// and takes the code compiled for its type.  The types were a launch each
// before; on a volume of a few million cells each of those sixteen launches a
// step (forward and adjoint) ran for its own 30 to 60 us however few cells it
// held (97 x 110 x 131, order 8, one shot: 0.77 ms a step, per-cell kernels
// 0.56 ms, one launch 0.37 ms); at 256 x 512 x 512 the two are equal.
// Workgroup numbers are remapped so that each XCD (workgroups go round-robin
// over the eight) takes a contiguous run of each type's tiles, whose halos
// then meet in the same L2.
//
// The arithmetic is that of the per-cell kernels (acoustic3d.hip), which
// follow the reference's expression trees (csrc/cuda/equations/acoustic3d/
// forward_split.cu:81-328, adjoint_split.cu:56-318).
#include "acoustic3d_zm.h"
#include "fd.h"

#include <algorithm>

namespace swp {
namespace a3d {

using fd::d1_taps;
using fd::lap_taps;

namespace {

constexpr int kRectMax = 8;

// A box of cells [x0, x1) x [y0, y1) x [z0, z1) cut into tiles of 64 x TY
// columns (partial tiles masked) and z segments of tz planes.
// Tiles start at xs <= x0 (x0 rounded down to a 128-byte line when rows are
// line-aligned), so each wave row covers whole lines; lanes outside [x0, x1)
// are masked.
struct ZRect {
    int x0, x1, y0, y1, z0, z1, tz;
    int xs;
    int ntx, nty, nseg, nblk;
};

struct ZSet {
    ZRect r[kRectMax];
    int n;
    int per_shot;   // blocks per shot
};

// Calls f(integral_constant<int, I>) for I = B..N-1 in order while it returns true.
template <int I, int N, class F>
__device__ __forceinline__ void static_for(F &&f)
{
    if constexpr (I < N) {
        if (f(std::integral_constant<int, I>{})) static_for<I + 1, N>(f);
    }
}

// One shot's field seen from plane zbase on.  An access takes the lane's
// in-plane byte offset (a loop-invariant VGPR) and the plane's byte offset (an
// SGPR); the caller keeps (planes used) * sxy * 4 below 2^32 and every row,
// column and plane in the grid.  Two forms of the same access:
// Buf, a raw buffer resource (four SGPRs, base and extent; past the field's
// end loads read 0 and stores write nothing), where a plane step costs no
// vector instruction -- the forward step and the reconstruction, which have
// SGPRs for it (record of 128 x 256 x 256, order 8: 35.7 ms, with Ptr 36.9);
struct Buf {
    __amdgpu_buffer_rsrc_t r;
    __device__ __forceinline__ Buf(const float *field, int64_t base_cell, int64_t end_cell)
    {
        const int64_t bytes = (end_cell - base_cell) * 4;
        r = __builtin_amdgcn_make_buffer_rsrc(const_cast<float *>(field + base_cell), short(0),
                                              int(uint32_t(bytes < 0xffffffffLL ? bytes : 0xffffffffLL)),
                                              0x00020000);   // gfx9 dword 3: 32-bit raw data
    }
    __device__ __forceinline__ float ld(uint32_t voff, uint32_t soff) const
    {
        return __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(r, voff, soff, 0));
    }
    __device__ __forceinline__ void st(float v, uint32_t voff, uint32_t soff) const
    {
        __builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(uint32_t, v), r, voff, soff, 0);
    }
};
// Ptr, a base pointer (two SGPRs) and one 32-bit add a row and plane that all
// fields share -- the adjoint, whose nineteen fields as resources spilled up
// to 360 SGPRs to VGPR lanes (gradient of 256 x 512 x 512, two shots, 100
// steps: 556 ms, with Buf 561).
struct Ptr {
    char *p;
    __device__ __forceinline__ Ptr(const float *field, int64_t base_cell)
        : p(reinterpret_cast<char *>(const_cast<float *>(field) + base_cell))
    {
    }
    __device__ __forceinline__ float ld(uint32_t voff, uint32_t soff) const
    {
        return *reinterpret_cast<const float *>(p + uint32_t(voff + soff));
    }
    __device__ __forceinline__ void st(float v, uint32_t voff, uint32_t soff) const
    {
        *reinterpret_cast<float *>(p + uint32_t(voff + soff)) = v;
    }
};

// One workgroup's tile: its rectangle, shot, tile origin and z segment.
struct ZTile {
    ZRect r;
    int b, xo, yo, zb, ze;
};

// Tile t of one shot's tiles over n rectangles (TY rows each); false past the last.
__device__ __forceinline__ bool ztile(const ZRect *rs, int n, int TY, int t, ZTile &out)
{
    for (int k = 0; k < n; ++k) {
        const ZRect &R = rs[k];
        if (t < R.nblk) {
            const int tx = t % R.ntx;
            const int ty = (t / R.ntx) % R.nty;
            const int sg = t / (R.ntx * R.nty);
            out.r = R;
            out.xo = R.xs + 64 * tx;
            out.yo = R.y0 + TY * ty;
            out.zb = R.z0 + sg * R.tz;
            out.ze = min(out.zb + R.tz, R.z1);
            return true;
        }
        t -= R.nblk;
    }
    return false;
}

// The tile of a launch over one set, in the XCD-local order.
template <int TY>
__device__ __forceinline__ bool zcoords(const ZSet &s, ZTile &out)
{
    const int f = int(xcd_local_id(blockIdx.x, gridDim.x));
    out.b = f / s.per_shot;
    return ztile(s.r, s.n, TY, f % s.per_shot, out);
}

// The regions of a step in one launch.  Entry k is a region type (bit 0 BX,
// bit 1 BY, bit 2 BZ) with its rectangles r[r0[k] .. r0[k + 1]) and the
// workgroups [first[k], first[k + 1]): a multiple of eight, the last few
// idle, so that every type is spread over the XCDs and numbered XCD-locally
// by itself.
struct ZPlan {
    ZRect r[27];
    int r0[9], first[9], type[8], per_shot[8], ty[8];
    int n;
};

__device__ __forceinline__ bool zplan_tile(const ZPlan &zp, int B, int &type, ZTile &out)
{
    const int f = int(blockIdx.x);
    int k = 0;
    while (k + 1 < zp.n && f >= zp.first[k + 1]) ++k;
    const int t = int(xcd_local_id(unsigned(f - zp.first[k]), unsigned(zp.first[k + 1] - zp.first[k])));
    type = zp.type[k];
    out.b = t / zp.per_shot[k];
    return out.b < B && ztile(zp.r + zp.r0[k], zp.r0[k + 1] - zp.r0[k], zp.ty[k], t % zp.per_shot[k], out);
}

// ---------------------------------------------------------------- plane I/O
// The halo duties of a lane: y-halo rows j = w + 4t (t < YH) of the 2M rows
// above and below the tile, x-halo columns for lanes < 2M on each of its rows.
template <int M, int TY, int NW>
struct PlaneMap {
    static constexpr int LW = 64 + 2 * M;
    static constexpr int LH = TY + 2 * M;
    static constexpr int YH = (2 * M + NW - 1) / NW;
    int yh_row[YH];      // global row of each y-halo duty (clamped), or -1
    int yh_slot[YH];     // LDS row of each duty
    int xh_col, xh_slot; // x-halo column (clamped) and LDS column, xh_slot < 0: none
    __device__ PlaneMap(int lane, int w, int xo, int yo, int nx, int ny)
    {
#pragma unroll
        for (int t = 0; t < YH; ++t) {
            const int j = w + NW * t;
            if (j < 2 * M) {
                const int gy = j < M ? yo - M + j : yo + TY + (j - M);
                yh_row[t] = min(max(gy, 0), ny - 1);
                yh_slot[t] = j < M ? j : TY + M + (j - M);
            } else {
                yh_row[t] = -1;
                yh_slot[t] = 0;
            }
        }
        if (lane < M) {
            xh_col = xo - M + lane;
            xh_slot = lane;
        } else if (lane < 2 * M) {
            xh_col = xo + 64 + (lane - M);
            xh_slot = 64 + M + (lane - M);
        } else {
            xh_col = xo;
            xh_slot = -1;
        }
        xh_col = min(max(xh_col, 0), nx - 1);
    }
};

template <int M, int RY, int NW>
struct Lanes {
    int x, xc;
    bool xa;
    int y[RY], yc[RY];
    bool act[RY];
    __device__ Lanes(const ZRect &R, int lane, int w, int xo, int yo, int nx, int ny)
    {
        x = xo + lane;
        xa = x >= R.x0 && x < R.x1;
        xc = min(x, nx - 1);
#pragma unroll
        for (int r = 0; r < RY; ++r) {
            y[r] = yo + w + NW * r;
            yc[r] = min(y[r], ny - 1);
            act[r] = xa && y[r] < R.y1;
        }
    }
};

// ---------------------------------------------------------------- halo duties
// The x-halo of a tile plane is RY rows x 2M columns per wave; lane l < 2M RY
// of wave w takes row w + 4 (l / 2M) and halo column l mod 2M of it (M on the
// left of the tile, then M on the right), so each lane holds at most one
// x-halo value per plane.  The y-halo rows are spread as in
// PlaneMap (rows j = w + 4t of the 2M rows above and below the tile).
template <int M, int RY, int NW>
struct XHalo {
    static_assert(2 * M * RY <= 64, "x-halo duties exceed one wave");
    uint32_t off;   // in-plane byte offset (clamped into the grid)
    int col;        // global column (clamped)
    int lds;        // index in the LDS plane, -1: no duty
    __device__ XHalo(int lane, int w, int xo, int yo, int nx, int px, int ny)
    {
        if (lane < 2 * M * RY) {
            const int r = lane / (2 * M), c = lane % (2 * M);
            const int row = w + NW * r;
            const int gx = c < M ? xo - M + c : xo + 64 + (c - M);
            const int gy = min(yo + row, ny - 1);
            col = min(max(gx, 0), nx - 1);
            off = uint32_t(gy * px + col) * 4u;
            lds = (row + M) * (64 + 2 * M) + (c < M ? c : 64 + M + (c - M));
        } else {
            col = 0;
            off = 0;
            lds = -1;
        }
    }
};

// ---------------------------------------------------------------- forward
// One template for every region of the computed box: BX/BY/BZ switch on the
// CPML machinery of an axis (the region lies in that axis' CPML margin);
// the lean interior runs it with all three off.  With an axis on, its psi
// taps come from an LDS plane (x, y; halo on that axis only) or a register
// queue (z), so each psi is read once per step; each cell then applies the
// product-rule update on the axes whose band holds it (pos < lo + 1 or
// pos >= hi - 1), the plain second derivative on the others, and saves its
// strip cells.
//
// The z loop runs in rounds of R = 2M + 2 planes with every queue slot fixed
// at compile time.  At step S of a round (plane z), the u queue slot
// (S + M + d) mod R holds plane z + d for |d| <= M, and the free slot takes
// the head z + M + 1.  The x/y halo of u is fetched together with the head
// (when the neighbouring tiles fetch that plane as their own head, so the
// shared lines are still in L2) and waits in an (M + 1)-deep queue until the
// plane is staged in LDS; halo slot p mod (M + 1) holds plane zb + p.
// One axis' CPML update of a cell: its term of w_sum, and psi and zeta after
// the step.  Which products are fused is written out, not left to the
// compiler, so that a record's bits depend neither on the code around the sum
// nor, below kBigCells3, on the kernel family (there every plain second
// derivative enters the sum rounded and b du is the fused product of psi, as
// in the per-cell kernel; see BIG in fwd3_tile for the sizes above).
template <bool FUSE_APSI>
__device__ __forceinline__ float cpml_axis(float L, float a, float b, float db, float da, float du, float dpsi,
                                           float psi0, float zeta0, float &psi1, float &zeta1)
{
    const float tmp = fd::fused(da, psi0, fd::fused(dpsi, a, fd::fused(L, 1.0f + b, fd::rounded(db * du))));
    const float az = fd::rounded(a * zeta0);
    psi1 = FUSE_APSI ? fd::fused(a, psi0, fd::rounded(b * du)) : fd::fused(du, b, fd::rounded(a * psi0));
    zeta1 = fd::fused(b, tmp, az);
    return fd::rounded(fd::fused(1.0f + b, tmp, az));
}

template <int M, int RY, bool BX, bool BY, int NW>
constexpr int fwd_plane() { return (1 + (BX ? 1 : 0) + (BY ? 1 : 0)) * (NW * RY + 2 * M) * (64 + 2 * M); }

template <int M, int RY, bool BX, bool BY, bool BZ, int NW, bool BIG>
__device__ __forceinline__ void fwd3_tile(const Geo &g, const Coef &c, const Prof &pr, const StepFields &f,
                                          float *__restrict__ u_this, float *__restrict__ strip, const ZTile &tile,
                                          float *lds_mem)
{
    constexpr bool SHELL = BX || BY || BZ;
    constexpr bool TAIL_Y = BIG && !BY && !BZ, TAIL_Z = BIG && !BZ;
    constexpr int TY = NW * RY;
    using PM = PlaneMap<M, TY, NW>;
    constexpr int LW = PM::LW, PS = PM::LH * PM::LW, YH = PM::YH;
    constexpr int SX = 1, SY = BX ? 2 : 1;   // plane slots of psi_x, psi_y
    constexpr int R = 2 * M + 2, H = M + 1;
    float *const lds[2] = {lds_mem, lds_mem + fwd_plane<M, RY, BX, BY, NW>()};
    const int b = tile.b, xo = tile.xo, yo = tile.yo, zb = tile.zb, ze = tile.ze;
    const ZRect &Rc = tile.r;
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    const int nx = g.nx, ny = g.ny;
    const int64_t sxy = g.sxy;
    const Lanes<M, RY, NW> L(Rc, lane, w, xo, yo, nx, ny);
    const PM pm(lane, w, xo, yo, nx, ny);
    const XHalo<M, RY, NW> xh(lane, w, xo, yo, nx, g.px, ny);
    const int64_t off = int64_t(b) * g.n;
    const float dt = g.dt;
    // fields from plane zb - M on; plane z sits at byte offset pl(z)
    const int zbase = zb - M;
    const int64_t fb = off + int64_t(zbase) * sxy, fe = off + g.n;
    const int64_t mb = int64_t(b) * g.mstride + int64_t(zbase) * sxy, me = int64_t(b) * g.mstride + g.n;
    const uint32_t sxy4 = uint32_t(sxy) * 4u;
    auto pl = [&](int z) { return uint32_t(z - zbase) * sxy4; };
    const Buf un(f.u_now, fb, fe), up(f.u_prev, fb, fe), unx(f.u_next, fb, fe), vp(f.vp, mb, me);
    const Buf psx(f.psi[0], fb, fe), psy(f.psi[1], fb, fe), psz(f.psi[2], fb, fe);
    const Buf pnx(f.psin[0], fb, fe), pny(f.psin[1], fb, fe), pnz(f.psin[2], fb, fe);
    const Buf zex(f.zeta[0], fb, fe), zey(f.zeta[1], fb, fe), zez(f.zeta[2], fb, fe);

    uint32_t col[RY], yhc[YH];   // in-plane byte offsets
#pragma unroll
    for (int r = 0; r < RY; ++r) col[r] = uint32_t(L.yc[r] * g.px + L.xc) * 4u;
#pragma unroll
    for (int t = 0; t < YH; ++t) yhc[t] = uint32_t((pm.yh_row[t] >= 0 ? pm.yh_row[t] : 0) * g.px + L.xc) * 4u;

    float ax = 0.f, bx = 0.f, dbx = 0.f, dax = 0.f;
    bool inbx = false;
    float ay[RY], by[RY], dby[RY], day[RY];
    bool inby[RY];
    if constexpr (BX) {
        const int xs = min(max(L.x, M), nx - 1 - M);
        inbx = L.x < g.X0 + 1 || L.x >= g.X1 - 1;
        ax = pr.a[0][xs];
        bx = pr.b[0][xs];
        dbx = pr.db[0][xs];
        dax = d1_taps<M>(c, [&](int q) { return pr.a[0][xs + q]; }, g.inv_dx);
    }
    if constexpr (BY) {
#pragma unroll
        for (int r = 0; r < RY; ++r) {
            const int ys = min(max(L.y[r], M), ny - 1 - M);
            inby[r] = L.y[r] < g.Y0 + 1 || L.y[r] >= g.Y1 - 1;
            ay[r] = pr.a[1][ys];
            by[r] = pr.b[1][ys];
            dby[r] = pr.db[1][ys];
            day[r] = d1_taps<M>(c, [&](int q) { return pr.a[1][ys + q]; }, g.inv_dy);
        }
    }

    float q[RY][R], qp[RY][BZ ? R : 1];   // u and psi_z z-queues
    float hx[H], hy[H][YH];               // u halo queue
    // plane-(z+1) registers (single-use fields, fetched one plane ahead)
    float nup[RY], nv[RY], npx[RY], nzx[RY], npy[RY], nzy[RY], nzz[RY];
    float npxh = 0.f, npyh[YH];           // psi_x x-halo, psi_y y-halo

    auto load_halo = [&](int zh, int slot) {   // the u halo of plane zh into halo slot `slot`
        const uint32_t so = pl(zh);
        if (xh.lds >= 0) hx[slot] = un.ld(xh.off, so);
#pragma unroll
        for (int t = 0; t < YH; ++t)
            if (pm.yh_row[t] >= 0) hy[slot][t] = un.ld(yhc[t], so);
    };
    auto load_plane = [&](int zn) {   // the single-use fields of plane zn
        const uint32_t so = pl(zn);
#pragma unroll
        for (int r = 0; r < RY; ++r) {
            nup[r] = up.ld(col[r], so);
            nv[r] = vp.ld(col[r], so);
            if constexpr (BX) {
                npx[r] = psx.ld(col[r], so);
                nzx[r] = zex.ld(col[r], so);
            }
            if constexpr (BY) {
                npy[r] = psy.ld(col[r], so);
                nzy[r] = zey.ld(col[r], so);
            }
            if constexpr (BZ) nzz[r] = zez.ld(col[r], so);
        }
        if constexpr (BX)
            if (xh.lds >= 0) npxh = psx.ld(xh.off, so);
        if constexpr (BY) {
#pragma unroll
            for (int t = 0; t < YH; ++t)
                if (pm.yh_row[t] >= 0) npyh[t] = psy.ld(yhc[t], so);
        }
    };
    // stage plane z: its u from queue slot cs, its u halo from halo slot hs
    auto store_plane = [&](float *P, int cs, int hs) {
#pragma unroll
        for (int r = 0; r < RY; ++r) {
            const int row = (w + NW * r + M) * LW;
            P[row + lane + M] = q[r][cs];
            if constexpr (BX) P[SX * PS + row + lane + M] = npx[r];
            if constexpr (BY) P[SY * PS + row + lane + M] = npy[r];
        }
        if (xh.lds >= 0) {
            P[xh.lds] = hx[hs];
            if constexpr (BX) P[SX * PS + xh.lds] = npxh;
        }
#pragma unroll
        for (int t = 0; t < YH; ++t) {
            if (pm.yh_row[t] >= 0) {
                P[pm.yh_slot[t] * LW + lane + M] = hy[hs][t];
                if constexpr (BY) P[SY * PS + pm.yh_slot[t] * LW + lane + M] = npyh[t];
            }
        }
    };

    // prologue: u slots t = 0..2M hold planes zb - M + t, halo slots p hold
    // planes zb + p (p <= M), plane zb staged in buffer 0
#pragma unroll
    for (int r = 0; r < RY; ++r) {
#pragma unroll
        for (int t = 0; t <= 2 * M; ++t) {
            q[r][t] = un.ld(col[r], pl(zb - M + t));
            if constexpr (BZ) qp[r][t] = psz.ld(col[r], pl(zb - M + t));
        }
    }
#pragma unroll
    for (int p = 0; p < H; ++p) load_halo(min(zb + p, ze - 1 + M), p);
    load_plane(zb);
    store_plane(lds[0], M, 0);
    __syncthreads();

    for (int z0 = zb; z0 < ze; z0 += R) {
        static_for<0, R>([&](auto Sc) -> bool {
        constexpr int S = decltype(Sc)::value;
        constexpr int C = (S + M) % R;       // slot of plane z
        const int z = z0 + S;
        if (z >= ze) return false;
        const float *P = lds[S & 1];
        float cup[RY], cv[RY], czx[RY], czy[RY], czz[RY], cpx[RY], cpy[RY];
#pragma unroll
        for (int r = 0; r < RY; ++r) {
            cup[r] = nup[r];
            cv[r] = nv[r];
            czx[r] = nzx[r];
            czy[r] = nzy[r];
            czz[r] = nzz[r];
            cpx[r] = npx[r];
            cpy[r] = npy[r];
        }
        {   // plane z + M + 1: u head and u halo; plane z + 1: the rest
            // (clamped at the segment end, where they are not used)
            const int zh = min(z + M + 1, ze - 1 + M);
            const uint32_t so = pl(zh);
#pragma unroll
            for (int r = 0; r < RY; ++r) {
                q[r][(S + 2 * M + 1) % R] = un.ld(col[r], so);
                if constexpr (BZ) qp[r][(S + 2 * M + 1) % R] = psz.ld(col[r], so);
            }
            load_halo(zh, S % H);
            load_plane(min(z + 1, ze - 1));
        }
        const uint32_t so = pl(z);
        bool inbz = false;
        float az = 0.f, bz = 0.f, dbz = 0.f, daz = 0.f;
        if constexpr (BZ) {
            inbz = z < g.Z0 + 1 || z >= g.Z1 - 1;
            az = pr.a[2][z];
            bz = pr.b[2][z];
            dbz = pr.db[2][z];
            daz = d1_taps<M>(c, [&](int t) { return pr.a[2][z + t]; }, g.inv_dz);
        }
#pragma unroll
        for (int r = 0; r < RY; ++r) {
            if (!L.act[r]) continue;
            const int row = (w + NW * r + M) * LW + lane + M;
            const float *Rw = P + row;
            const float u0 = q[r][C];
            auto qz = [&](int t) { return q[r][(C + t + R) % R]; };
            const float acc_x = lap_taps<M>(c, [&](int t) { return Rw[t]; }, 1.0f), lx = fd::rounded(fd::scaled(acc_x, g.inv_dx2));
            const float acc_y = lap_taps<M>(c, [&](int t) { return Rw[t * LW]; }, 1.0f), ly = fd::rounded(fd::scaled(acc_y, g.inv_dy2));
            const float acc_z = lap_taps<M>(c, qz, 1.0f), lz = fd::rounded(fd::scaled(acc_z, g.inv_dz2));
            float w_sum;
            if constexpr (!SHELL) {
                w_sum = BIG ? fd::plus_scaled<true>(fd::plus_scaled<true>(ly, acc_x, g.inv_dx2), acc_z, g.inv_dz2) : lx + ly + lz;
            } else {
                if (strip) save_strips(g, strip + int64_t(b) * g.ns, L.x, L.y[r], z, u0);
                const bool bandx = BX && inbx, bandy = BY && inby[r], bandz = BZ && inbz;
                if (!bandx && !bandy && !bandz) {
                    w_sum = fd::plus_scaled<TAIL_Z>(fd::plus_scaled<TAIL_Y>(lx, acc_y, g.inv_dy2), acc_z, g.inv_dz2);
                } else {
                    w_sum = 0.f;
                    float psi1, z1v;
                    if (bandx) {
                        const float *Px = P + SX * PS + row;
                        const float du = d1_taps<M>(c, [&](int t) { return Rw[t]; }, g.inv_dx);
                        const float dpsi = d1_taps<M>(c, [&](int t) { return Px[t]; }, g.inv_dx);
                        const float psi0 = cpx[r];
                        const float z0v = czx[r];
                        w_sum += cpml_axis<BIG>(lx, ax, bx, dbx, dax, du, dpsi, psi0, z0v, psi1, z1v);
                        pnx.st(psi1, col[r], so);
                        zex.st(z1v, col[r], so);
                    } else {
                        w_sum += lx;
                    }
                    if (bandy) {
                        const float *Py = P + SY * PS + row;
                        const float du = d1_taps<M>(c, [&](int t) { return Rw[t * LW]; }, g.inv_dy);
                        const float dpsi = d1_taps<M>(c, [&](int t) { return Py[t * LW]; }, g.inv_dy);
                        const float psi0 = cpy[r];
                        const float z0v = czy[r];
                        w_sum += cpml_axis<BIG && (BX || BZ)>(ly, ay[r], by[r], dby[r], day[r], du, dpsi, psi0, z0v, psi1, z1v);
                        pny.st(psi1, col[r], so);
                        zey.st(z1v, col[r], so);
                    } else {
                        w_sum = fd::plus_scaled<TAIL_Y>(w_sum, acc_y, g.inv_dy2);
                    }
                    if constexpr (BZ) {
                        if (bandz) {
                            auto qpz = [&](int t) { return qp[r][(C + t + R) % R]; };
                            const float du = d1_taps<M>(c, qz, g.inv_dz);
                            const float dpsi = d1_taps<M>(c, qpz, g.inv_dz);
                            const float psi0 = qp[r][C];
                            const float z0v = czz[r];
                            w_sum += cpml_axis<false>(lz, az, bz, dbz, daz, du, dpsi, psi0, z0v, psi1, z1v);
                            pnz.st(psi1, col[r], so);
                            zez.st(z1v, col[r], so);
                        } else {
                            w_sum = fd::plus_scaled<TAIL_Z>(w_sum, acc_z, g.inv_dz2);
                        }
                    } else {
                        w_sum = fd::plus_scaled<TAIL_Z>(w_sum, acc_z, g.inv_dz2);
                    }
                }
            }
            const float v = cv[r];
            unx.st(fd::fused((v * v) * dt * dt, w_sum, 2.0f * u0 - cup[r]), col[r], so);
            if (u_this) u_this[off + int64_t(z) * sxy + col[r] / 4u] = (v * v) * w_sum;
        }
        if (z + 1 < ze) store_plane(lds[(S + 1) & 1], (C + 1) % R, (S + 1) % H);
        __syncthreads();
        return true;
        });
    }
}

// ---------------------------------------------------------------- adjoint
// The LDS plane G and the z queue hold gw = v^2 dt^2 lambda; a FIFO keeps
// lambda for the centre.  With an axis on (the region lies in that axis'
// adjoint band, outside phys_box(M + 1)), the transposed CPML update of
// that axis is taken through three per-cell fields of the neighbours,
//   T = b zeta + (1 + b) gw,  U = (1 + b) T,  V = b psi + db T,  W = a T,
// (profiles at the neighbour's own position), staged in LDS planes (x, y)
// or register queues (z):
//   L = sum_k lap_k ((U(+k) - U(0)) + (U(-k) - U(0))),
//   Dg = sum_k grad_k (V(+k) - V(-k)),  Dq = sum_k grad_k (W(+k) - W(-k)),
//   psi' = a psi + (da) T(0) - Dq,  zeta' = a (zeta + gw)
// -- the expression tree of the per-cell adjoint (adjoint_split.cu:56-318)
// with each neighbour's T formed once.  img != nullptr fuses the lagged
// full-mode imaging grad += 2 dt^2 img lambda / v.
template <int M, int RY, bool BX, bool BY, int NW>
constexpr int adj_plane() { return (1 + (BX ? 3 : 0) + (BY ? 3 : 0)) * (NW * RY + 2 * M) * (64 + 2 * M); }

template <int M, int RY, bool BX, bool BY, bool BZ, int NW>
__device__ __forceinline__ void adj3_tile(const Geo &g, const Coef &c, const Prof &pr, const AdjFields &f,
                                          const float *__restrict__ img, float *__restrict__ grad, const ZTile &tile,
                                          float *lds_mem)
{
    constexpr bool SHELL = BX || BY || BZ;
    constexpr int TY = NW * RY;
    using PM = PlaneMap<M, TY, NW>;
    constexpr int LW = PM::LW, PS = PM::LH * PM::LW, YH = PM::YH;
    constexpr int SX = 1, SY = BX ? 4 : 1;   // first plane slot of (U, V, W) for x, y
    constexpr int R = 2 * M + 2, H = M + 1;
    float *const lds[2] = {lds_mem, lds_mem + adj_plane<M, RY, BX, BY, NW>()};
    const int b = tile.b, xo = tile.xo, yo = tile.yo, zb = tile.zb, ze = tile.ze;
    const ZRect &Rc = tile.r;
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    const int nx = g.nx, ny = g.ny;
    const int64_t sxy = g.sxy;
    const Lanes<M, RY, NW> L(Rc, lane, w, xo, yo, nx, ny);
    const PM pm(lane, w, xo, yo, nx, ny);
    const XHalo<M, RY, NW> xh(lane, w, xo, yo, nx, g.px, ny);
    const int64_t off = int64_t(b) * g.n;
    const float dt2 = g.dt2;
    // fields from plane zb - M on; plane z sits at byte offset pl(z)
    const int zbase = zb - M;
    const int64_t fb = off + int64_t(zbase) * sxy;
    const int64_t mb = int64_t(b) * g.mstride + int64_t(zbase) * sxy;
    const uint32_t sxy4 = uint32_t(sxy) * 4u;
    auto pl = [&](int z) { return uint32_t(z - zbase) * sxy4; };
    const Ptr ln(f.l_now, fb), lp(f.l_prev, fb), lnx(f.l_next, fb), vp(f.vp, mb);
    const Ptr psx(f.psi[0], fb), psy(f.psi[1], fb), psz(f.psi[2], fb);
    const Ptr zex(f.zeta[0], fb), zey(f.zeta[1], fb), zez(f.zeta[2], fb);
    const Ptr pox(f.psio[0], fb), poy(f.psio[1], fb), poz(f.psio[2], fb);
    const Ptr zox(f.zetao[0], fb), zoy(f.zetao[1], fb), zoz(f.zetao[2], fb);

    uint32_t col[RY], yhc[YH];   // in-plane byte offsets
#pragma unroll
    for (int r = 0; r < RY; ++r) col[r] = uint32_t(L.yc[r] * g.px + L.xc) * 4u;
#pragma unroll
    for (int t = 0; t < YH; ++t) yhc[t] = uint32_t((pm.yh_row[t] >= 0 ? pm.yh_row[t] : 0) * g.px + L.xc) * 4u;

    // profiles: the lane's column / x-halo duty column (x), rows / halo rows (y)
    float ax = 0.f, bx = 0.f, dbx = 0.f, dax = 0.f, hax = 0.f, hbx = 0.f, hdbx = 0.f;
    float ay[RY], by[RY], dby[RY], day[RY], hay[YH], hby[YH], hdby[YH];
    if constexpr (BX) {
        const int xs = min(max(L.x, M), nx - 1 - M);
        ax = pr.a[0][L.xc];
        bx = pr.b[0][L.xc];
        dbx = pr.db[0][L.xc];
        dax = d1_taps<M>(c, [&](int q) { return pr.a[0][xs + q]; }, g.inv_dx);
        hax = pr.a[0][xh.col];
        hbx = pr.b[0][xh.col];
        hdbx = pr.db[0][xh.col];
    }
    if constexpr (BY) {
#pragma unroll
        for (int r = 0; r < RY; ++r) {
            const int ys = min(max(L.y[r], M), ny - 1 - M);
            ay[r] = pr.a[1][L.yc[r]];
            by[r] = pr.b[1][L.yc[r]];
            dby[r] = pr.db[1][L.yc[r]];
            day[r] = d1_taps<M>(c, [&](int q) { return pr.a[1][ys + q]; }, g.inv_dy);
        }
#pragma unroll
        for (int t = 0; t < YH; ++t) {
            const int yr = pm.yh_row[t] >= 0 ? pm.yh_row[t] : 0;
            hay[t] = pr.a[1][yr];
            hby[t] = pr.b[1][yr];
            hdby[t] = pr.db[1][yr];
        }
    }
    auto gwof = [&](float lv, float v) { return v * v * dt2 * lv; };
    // U, V, W of one cell from its raw values and its profile (b, db, a)
    auto uvw = [&](float zeta, float psi, float gwv, float bb, float dd, float aa, float &U, float &V, float &W) {
        const float T = bb * zeta + (1.0f + bb) * gwv;
        U = (1.0f + bb) * T;
        V = bb * psi + dd * T;
        W = aa * T;
    };

    // z queues over rounds of R = 2M + 2 planes (slot (S + M + d) mod R holds
    // plane z + d): gw (z taps), lambda (centre), U/V/W of the z axis; the gw
    // halo of a plane is formed with its queue head and waits in an
    // (M + 1)-deep queue (slot p mod (M + 1) holds plane zb + p) until staged.
    float qg[RY][R], ql[RY][R];
    float qu[RY][BZ ? R : 1], qv[RY][BZ ? R : 1], qw[RY][BZ ? R : 1];
    float hgx[H], hgy[H][YH];
    // heads of plane z + M + 1 in flight
    float nl[RY], nvh[RY], nzh[RY], nph[RY], nhl = 0.f, nhv = 0.f, nyl[YH], nyv[YH];
    // single-use fields of plane z + 1 in flight
    float nlp[RY], nzx[RY], npx[RY], nzxh = 0.f, npxh = 0.f, nzy[RY], npy[RY], nzyh[YH], npyh[YH], nzz[RY], npz[RY];

    auto load_head = [&](int zh) {   // queue heads and the lambda / vp halo of plane zh
        const uint32_t so = pl(zh);
#pragma unroll
        for (int r = 0; r < RY; ++r) {
            nl[r] = ln.ld(col[r], so);
            nvh[r] = vp.ld(col[r], so);
            if constexpr (BZ) {
                nzh[r] = zez.ld(col[r], so);
                nph[r] = psz.ld(col[r], so);
            }
        }
        if (xh.lds >= 0) {
            nhl = ln.ld(xh.off, so);
            nhv = vp.ld(xh.off, so);
        }
#pragma unroll
        for (int t = 0; t < YH; ++t) {
            if (pm.yh_row[t] >= 0) {
                nyl[t] = ln.ld(yhc[t], so);
                nyv[t] = vp.ld(yhc[t], so);
            }
        }
    };
    auto push_head = [&](int zh, int slot, int hslot) {   // the heads of plane zh into their queue slots
        float bz_ = 0.f, dbz_ = 0.f, az_ = 0.f;
        if constexpr (BZ) {
            bz_ = pr.b[2][zh];
            dbz_ = pr.db[2][zh];
            az_ = pr.a[2][zh];
        }
#pragma unroll
        for (int r = 0; r < RY; ++r) {
            const float gh = gwof(nl[r], nvh[r]);
            qg[r][slot] = gh;
            ql[r][slot] = nl[r];
            if constexpr (BZ) uvw(nzh[r], nph[r], gh, bz_, dbz_, az_, qu[r][slot], qv[r][slot], qw[r][slot]);
        }
        hgx[hslot] = gwof(nhl, nhv);
#pragma unroll
        for (int t = 0; t < YH; ++t) hgy[hslot][t] = gwof(nyl[t], nyv[t]);
    };
    auto load_plane = [&](int zn) {   // single-use fields of plane zn
        const uint32_t so = pl(zn);
#pragma unroll
        for (int r = 0; r < RY; ++r) {
            nlp[r] = lp.ld(col[r], so);
            if constexpr (BX) {
                nzx[r] = zex.ld(col[r], so);
                npx[r] = psx.ld(col[r], so);
            }
            if constexpr (BY) {
                nzy[r] = zey.ld(col[r], so);
                npy[r] = psy.ld(col[r], so);
            }
            if constexpr (BZ) {
                nzz[r] = zez.ld(col[r], so);
                npz[r] = psz.ld(col[r], so);
            }
        }
        if constexpr (BX) {
            if (xh.lds >= 0) {
                nzxh = zex.ld(xh.off, so);
                npxh = psx.ld(xh.off, so);
            }
        }
        if constexpr (BY) {
#pragma unroll
            for (int t = 0; t < YH; ++t) {
                if (pm.yh_row[t] >= 0) {
                    nzyh[t] = zey.ld(yhc[t], so);
                    npyh[t] = psy.ld(yhc[t], so);
                }
            }
        }
    };
    // stage plane z: centre gw from queue slot cs, gw halo from halo slot hs
    auto store_plane = [&](float *P, int cs, int hs) {
#pragma unroll
        for (int r = 0; r < RY; ++r) {
            const int row = (w + NW * r + M) * LW;
            const float gc = qg[r][cs];
            P[row + lane + M] = gc;
            if constexpr (BX) {
                float U, V, W;
                uvw(nzx[r], npx[r], gc, bx, dbx, ax, U, V, W);
                P[SX * PS + row + lane + M] = U;
                P[(SX + 1) * PS + row + lane + M] = V;
                P[(SX + 2) * PS + row + lane + M] = W;
            }
            if constexpr (BY) {
                float U, V, W;
                uvw(nzy[r], npy[r], gc, by[r], dby[r], ay[r], U, V, W);
                P[SY * PS + row + lane + M] = U;
                P[(SY + 1) * PS + row + lane + M] = V;
                P[(SY + 2) * PS + row + lane + M] = W;
            }
        }
        if (xh.lds >= 0) {
            const float gh = hgx[hs];
            P[xh.lds] = gh;
            if constexpr (BX) {
                float U, V, W;
                uvw(nzxh, npxh, gh, hbx, hdbx, hax, U, V, W);
                P[SX * PS + xh.lds] = U;
                P[(SX + 1) * PS + xh.lds] = V;
                P[(SX + 2) * PS + xh.lds] = W;
            }
        }
#pragma unroll
        for (int t = 0; t < YH; ++t) {
            if (pm.yh_row[t] >= 0) {
                const int row = pm.yh_slot[t] * LW + lane + M;
                const float gh = hgy[hs][t];
                P[row] = gh;
                if constexpr (BY) {
                    float U, V, W;
                    uvw(nzyh[t], npyh[t], gh, hby[t], hdby[t], hay[t], U, V, W);
                    P[SY * PS + row] = U;
                    P[(SY + 1) * PS + row] = V;
                    P[(SY + 2) * PS + row] = W;
                }
            }
        }
    };

    // prologue: queue slot t holds plane zb - M + t (t <= 2M), halo slot p
    // plane zb + p (p <= M); plane zb staged in buffer 0
#pragma unroll
    for (int t = 0; t <= 2 * M; ++t) {
        load_head(min(zb - M + t, ze - 1 + M));
        push_head(min(zb - M + t, ze - 1 + M), t, t >= M ? t - M : 0);
    }
    load_plane(zb);
    store_plane(lds[0], M, 0);
    __syncthreads();

    for (int z0 = zb; z0 < ze; z0 += R) {
        static_for<0, R>([&](auto Sc) -> bool {
        constexpr int S = decltype(Sc)::value;
        constexpr int C = (S + M) % R;
        const int z = z0 + S;
        if (z >= ze) return false;
        const float *P = lds[S & 1];
        float clp[RY], czx[RY], cpx[RY], czy[RY], cpy[RY], czz[RY], cpz[RY];
#pragma unroll
        for (int r = 0; r < RY; ++r) {
            clp[r] = nlp[r];
            czx[r] = nzx[r];
            cpx[r] = npx[r];
            czy[r] = nzy[r];
            cpy[r] = npy[r];
            czz[r] = nzz[r];
            cpz[r] = npz[r];
        }
        const int zh = min(z + M + 1, ze - 1 + M);   // clamped at the segment end, unused there
        load_head(zh);
        load_plane(min(z + 1, ze - 1));
        const uint32_t so = pl(z);
        float az = 0.f, bz = 0.f, daz = 0.f;
        if constexpr (BZ) {
            az = pr.a[2][z];
            bz = pr.b[2][z];
            daz = d1_taps<M>(c, [&](int t) { return pr.a[2][z + t]; }, g.inv_dz);
        }
#pragma unroll
        for (int r = 0; r < RY; ++r) {
            if (!L.act[r]) continue;
            const int row = (w + NW * r + M) * LW + lane + M;
            const float *Gw = P + row;
            const float gun = ql[r][C];
            const float gw = qg[r][C];
            auto zq = [&](const float (&qq)[R], int t) { return qq[(C + t + R) % R]; };
            if (grad && img && L.x >= g.X0 && L.x < g.X1 && L.y[r] >= g.Y0 && L.y[r] < g.Y1 && z >= g.Z0 &&
                z < g.Z1) {
                const int64_t i = off + int64_t(z) * sxy + col[r] / 4u;
                grad[i] += 2.f * g.dt * g.dt * img[i] * gun / vp.ld(col[r], so);
            }
            float out;
            if constexpr (!SHELL) {
                float lx = 0.f, ly = 0.f, lz = 0.f;
#pragma unroll
                for (int t = 1; t <= M; ++t) {
                    lx += c.lap[t] * ((Gw[t] - gw) + (Gw[-t] - gw));
                    ly += c.lap[t] * ((Gw[t * LW] - gw) + (Gw[-t * LW] - gw));
                    lz += c.lap[t] * ((zq(qg[r], t) - gw) + (zq(qg[r], -t) - gw));
                }
                out = 2.0f * gun - clp[r] + lx * g.inv_dx2.inv + ly * g.inv_dy2.inv + lz * g.inv_dz2.inv;
            } else {
                float Lt[3], Dg[3];
                if constexpr (BX) {
                    const float *Ux = P + SX * PS + row, *Vx = P + (SX + 1) * PS + row, *Wx = P + (SX + 2) * PS + row;
                    const float gt0 = bx * czx[r] + (1.0f + bx) * gw;
                    const float l0 = (1.0f + bx) * gt0;
                    float Ls = 0.f, Dgg = 0.f, Dq = 0.f;
#pragma unroll
                    for (int t = 1; t <= M; ++t) {
                        Ls += c.lap[t] * ((Ux[t] - l0) + (Ux[-t] - l0));
                        Dgg += c.grad[t] * (Vx[t] - Vx[-t]);
                        Dq += c.grad[t] * (Wx[t] - Wx[-t]);
                    }
                    Lt[0] = Ls * g.inv_dx2.inv;
                    Dg[0] = Dgg * g.inv_dx.inv;
                    Dq *= g.inv_dx.inv;
                    pox.st(ax * cpx[r] + dax * gt0 - Dq, col[r], so);
                    zox.st(ax * (czx[r] + gw), col[r], so);
                } else {
                    float Ls = 0.f;
#pragma unroll
                    for (int t = 1; t <= M; ++t) Ls += c.lap[t] * ((Gw[t] - gw) + (Gw[-t] - gw));
                    Lt[0] = Ls * g.inv_dx2.inv;
                    Dg[0] = 0.f;
                }
                if constexpr (BY) {
                    const float *Uy = P + SY * PS + row, *Vy = P + (SY + 1) * PS + row, *Wy = P + (SY + 2) * PS + row;
                    const float gt0 = by[r] * czy[r] + (1.0f + by[r]) * gw;
                    const float l0 = (1.0f + by[r]) * gt0;
                    float Ls = 0.f, Dgg = 0.f, Dq = 0.f;
#pragma unroll
                    for (int t = 1; t <= M; ++t) {
                        Ls += c.lap[t] * ((Uy[t * LW] - l0) + (Uy[-t * LW] - l0));
                        Dgg += c.grad[t] * (Vy[t * LW] - Vy[-t * LW]);
                        Dq += c.grad[t] * (Wy[t * LW] - Wy[-t * LW]);
                    }
                    Lt[1] = Ls * g.inv_dy2.inv;
                    Dg[1] = Dgg * g.inv_dy.inv;
                    Dq *= g.inv_dy.inv;
                    poy.st(ay[r] * cpy[r] + day[r] * gt0 - Dq, col[r], so);
                    zoy.st(ay[r] * (czy[r] + gw), col[r], so);
                } else {
                    float Ls = 0.f;
#pragma unroll
                    for (int t = 1; t <= M; ++t) Ls += c.lap[t] * ((Gw[t * LW] - gw) + (Gw[-t * LW] - gw));
                    Lt[1] = Ls * g.inv_dy2.inv;
                    Dg[1] = 0.f;
                }
                if constexpr (BZ) {
                    const float gt0 = bz * czz[r] + (1.0f + bz) * gw;
                    const float l0 = (1.0f + bz) * gt0;
                    float Ls = 0.f, Dgg = 0.f, Dq = 0.f;
#pragma unroll
                    for (int t = 1; t <= M; ++t) {
                        Ls += c.lap[t] * ((zq(qu[r], t) - l0) + (zq(qu[r], -t) - l0));
                        Dgg += c.grad[t] * (zq(qv[r], t) - zq(qv[r], -t));
                        Dq += c.grad[t] * (zq(qw[r], t) - zq(qw[r], -t));
                    }
                    Lt[2] = Ls * g.inv_dz2.inv;
                    Dg[2] = Dgg * g.inv_dz.inv;
                    Dq *= g.inv_dz.inv;
                    poz.st(az * cpz[r] + daz * gt0 - Dq, col[r], so);
                    zoz.st(az * (czz[r] + gw), col[r], so);
                } else {
                    float Ls = 0.f;
#pragma unroll
                    for (int t = 1; t <= M; ++t) Ls += c.lap[t] * ((zq(qg[r], t) - gw) + (zq(qg[r], -t) - gw));
                    Lt[2] = Ls * g.inv_dz2.inv;
                    Dg[2] = 0.f;
                }
                out = 2.0f * gun - clp[r] + (Lt[0] + Lt[1] + Lt[2] - Dg[0] - Dg[1] - Dg[2]);
            }
            lnx.st(out, col[r], so);
        }
        push_head(zh, (S + 2 * M + 1) % R, S % H);
        if (z + 1 < ze) store_plane(lds[(S + 1) & 1], (C + 1) % R, (S + 1) % H);
        __syncthreads();
        return true;
        });
    }
}

// ---------------------------------------------------------------- step kernels
// Rows per lane and waves per workgroup of the reconstruction (a block's tile
// is 64 x NW*RY cells; each plane re-reads 2M halo rows per tile, so a taller
// tile of more waves cuts the y-halo share without more registers per lane).
constexpr int kRyRecon = 4;
constexpr int kNwRecon = 8;

// Rows per lane of a region type (bits BX, BY, BZ); the step kernels run 4
// waves a workgroup, so a tile is 64 x 4 ry_of(type) cells.
constexpr int ry_of(int type)
{
    const int axes = (type & 1) + (type >> 1 & 1) + (type >> 2 & 1);
    return axes == 0 ? 4 : axes == 1 ? 2 : 1;
}

template <int M, int T>
constexpr int fwd_lds() { return fwd_plane<M, ry_of(T), (T & 1) != 0, (T & 2) != 0, 4>(); }
template <int M, int T>
constexpr int adj_lds() { return adj_plane<M, ry_of(T), (T & 1) != 0, (T & 2) != 0, 4>(); }
constexpr int max4(int a, int b, int c, int d) { return std::max(std::max(a, b), std::max(c, d)); }

template <int M, bool BIG>
__global__ void __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(4)))
fwd3_kernel(Geo g, Coef c, Prof pr, StepFields f, float *__restrict__ u_this, float *__restrict__ strip, ZPlan zp)
{
    __shared__ float lds[2 * max4(fwd_lds<M, 0>(), fwd_lds<M, 1>(), fwd_lds<M, 2>(), fwd_lds<M, 3>())];
    int type;
    ZTile tile;
    if (!zplan_tile(zp, g.B, type, tile)) return;
    switch (type) {
#define SWP_FWD3(T) \
    case T: fwd3_tile<M, ry_of(T), (T & 1) != 0, (T & 2) != 0, (T & 4) != 0, 4, BIG>(g, c, pr, f, u_this, strip, tile, lds); break
        SWP_FWD3(0);
        SWP_FWD3(1);
        SWP_FWD3(2);
        SWP_FWD3(3);
        SWP_FWD3(4);
        SWP_FWD3(5);
        SWP_FWD3(6);
        SWP_FWD3(7);
#undef SWP_FWD3
    }
}

// Three waves per SIMD: left alone the widest type takes 212 VGPRs and two
// (256 x 512 x 512, two shots, 100 steps: 571 against 556 ms; 97 x 110 x 131:
// 47.9 against 44.3 ms).
template <int M>
__global__ void __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(3)))
adj3_kernel(Geo g, Coef c, Prof pr, AdjFields f, const float *__restrict__ img, float *__restrict__ grad, ZPlan zp)
{
    __shared__ float lds[2 * max4(adj_lds<M, 0>(), adj_lds<M, 1>(), adj_lds<M, 2>(), adj_lds<M, 3>())];
    int type;
    ZTile tile;
    if (!zplan_tile(zp, g.B, type, tile)) return;
    switch (type) {
#define SWP_ADJ3(T) \
    case T: adj3_tile<M, ry_of(T), (T & 1) != 0, (T & 2) != 0, (T & 4) != 0, 4>(g, c, pr, f, img, grad, tile, lds); break
        SWP_ADJ3(0);
        SWP_ADJ3(1);
        SWP_ADJ3(2);
        SWP_ADJ3(3);
        SWP_ADJ3(4);
        SWP_ADJ3(5);
        SWP_ADJ3(6);
        SWP_ADJ3(7);
#undef SWP_ADJ3
    }
}

// ---------------------------------------------------------------- BS recon
// Reverse leapfrog without PML over one box, fused u_tt imaging on the cells
// of [lo + W, hi - W) per axis (the cells the strip restore leaves alone).
template <int M, int RY, int NW>
__global__ void __launch_bounds__(64 * NW) recon_zm_kernel(Geo g, Coef c, const float *__restrict__ vpb,
                                                       const float *__restrict__ u_prev, const float *__restrict__ u_now,
                                                       float *__restrict__ u_next, const float *__restrict__ adj,
                                                       float *__restrict__ grad, ZSet zs)
{
    constexpr int TY = NW * RY;
    using PM = PlaneMap<M, TY, NW>;
    constexpr int LW = PM::LW;
    __shared__ float lds[2][PM::LH * PM::LW];
    ZTile tile;
    if (!zcoords<TY>(zs, tile)) return;
    const ZRect &R = tile.r;
    const int b = tile.b, xo = tile.xo, yo = tile.yo, zb = tile.zb, ze = tile.ze;
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    const int nx = g.nx, ny = g.ny;
    const int64_t sxy = g.sxy;
    const Lanes<M, RY, NW> L(R, lane, w, xo, yo, nx, ny);
    const PM pm(lane, w, xo, yo, nx, ny);
    const int64_t off = int64_t(b) * g.n;
    const float dt = g.dt;
    const int zbase = zb - M;
    const int64_t fb = off + int64_t(zbase) * sxy, fe = off + g.n;
    const int64_t mb = int64_t(b) * g.mstride + int64_t(zbase) * sxy, me = int64_t(b) * g.mstride + g.n;
    const uint32_t sxy4 = uint32_t(sxy) * 4u;
    auto pl = [&](int z) { return uint32_t(z - zbase) * sxy4; };
    const Buf un(u_now, fb, fe), up(u_prev, fb, fe), unx(u_next, fb, fe), vp(vpb, mb, me);
    const Buf ad(adj, fb, fe), gr(grad, fb, fe);   // unused without grad
    const bool img_x = L.x >= g.X0 + g.W && L.x < g.X1 - g.W;
    bool img_y[RY];
    uint32_t col[RY], xhc[RY], yhc[PM::YH];   // in-plane byte offsets
#pragma unroll
    for (int r = 0; r < RY; ++r) {
        col[r] = uint32_t(L.yc[r] * g.px + L.xc) * 4u;
        xhc[r] = uint32_t(L.yc[r] * g.px + pm.xh_col) * 4u;
        img_y[r] = L.y[r] >= g.Y0 + g.W && L.y[r] < g.Y1 - g.W;
    }
#pragma unroll
    for (int t = 0; t < PM::YH; ++t) yhc[t] = uint32_t((pm.yh_row[t] >= 0 ? pm.yh_row[t] : 0) * g.px + L.xc) * 4u;

    constexpr int Q = 2 * M + 1;
    float q[RY][Q];
    float nq[RY], nup[RY], nv[RY], nxh[RY], na[RY], ng[RY];
    float nyh[PM::YH];
    auto load_plane = [&](int zn) {
        const uint32_t so = pl(zn);
#pragma unroll
        for (int r = 0; r < RY; ++r) {
            nup[r] = up.ld(col[r], so);
            nv[r] = vp.ld(col[r], so);
            if (grad) {
                na[r] = ad.ld(col[r], so);
                ng[r] = gr.ld(col[r], so);
            }
            nxh[r] = un.ld(xhc[r], so);
        }
#pragma unroll
        for (int t = 0; t < PM::YH; ++t)
            if (pm.yh_row[t] >= 0) nyh[t] = un.ld(yhc[t], so);
    };
    auto store_plane = [&](float *P, int cs) {
#pragma unroll
        for (int r = 0; r < RY; ++r) {
            P[(w + NW * r + M) * LW + lane + M] = q[r][cs];
            if (pm.xh_slot >= 0) P[(w + NW * r + M) * LW + pm.xh_slot] = nxh[r];
        }
#pragma unroll
        for (int t = 0; t < PM::YH; ++t)
            if (pm.yh_row[t] >= 0) P[pm.yh_slot[t] * LW + lane + M] = nyh[t];
    };
#pragma unroll
    for (int r = 0; r < RY; ++r) {
        na[r] = ng[r] = 0.f;
#pragma unroll
        for (int t = 0; t < Q; ++t) q[r][t] = un.ld(col[r], pl(zb - M + t));
    }
    load_plane(zb);
    store_plane(lds[zb & 1], M);
    __syncthreads();

    // rounds of Q planes with compile-time queue slots (as in fwd3_kernel)
    for (int z0 = zb; z0 < ze; z0 += Q) {
        static_for<0, Q>([&](auto Sc) -> bool {
        constexpr int S = decltype(Sc)::value;
        constexpr int C = (S + M) % Q;
        const int z = z0 + S;
        if (z >= ze) return false;
        const float *P = lds[z & 1];
        float cup[RY], cv[RY], ca[RY], cg[RY];
#pragma unroll
        for (int r = 0; r < RY; ++r) {
            cup[r] = nup[r];
            cv[r] = nv[r];
            ca[r] = na[r];
            cg[r] = ng[r];
        }
        {
            const int zn = min(z + 1, ze - 1);
            const uint32_t so = pl(zn + M);
#pragma unroll
            for (int r = 0; r < RY; ++r) nq[r] = un.ld(col[r], so);
            load_plane(zn);
        }
        const uint32_t so = pl(z);
        const bool img_z = z >= g.Z0 + g.W && z < g.Z1 - g.W;
#pragma unroll
        for (int r = 0; r < RY; ++r) {
            if (!L.act[r]) continue;
            const float *Rw = P + (w + NW * r + M) * LW + lane + M;
            const float u0 = q[r][C];
            const float w_sum = lap_taps<M>(c, [&](int t) { return Rw[t]; }, g.inv_dx2) +
                                lap_taps<M>(c, [&](int t) { return Rw[t * LW]; }, g.inv_dy2) +
                                lap_taps<M>(c, [&](int t) { return q[r][(C + t + Q) % Q]; }, g.inv_dz2);
            const float v = cv[r];
            const float unxt = 2.0f * u0 - cup[r] + (v * v) * dt * dt * w_sum;
            unx.st(unxt, col[r], so);
            if (grad && img_x && img_y[r] && img_z) {
                const float u_tt = fd::scaled(unxt - 2 * u0 + cup[r], g.inv_dt2);
                gr.st(cg[r] + 2.f * dt * dt * u_tt * ca[r] / v, col[r], so);
            }
        }
#pragma unroll
        for (int r = 0; r < RY; ++r) q[r][S] = nq[r];
        if (z + 1 < ze) store_plane(lds[(z + 1) & 1], (C + 1) % Q);
        __syncthreads();
        return true;
        });
    }
}

// ---------------------------------------------------------------- host plans
ZRect make_rect(int x0, int x1, int y0, int y1, int z0, int z1, int tz, int TY, int px)
{
    ZRect R{};
    R.x0 = x0; R.x1 = x1; R.y0 = y0; R.y1 = y1; R.z0 = z0; R.z1 = z1; R.tz = tz;
    // line-aligned tile origin unless that costs an extra column of tiles
    const int xa = px % 32 == 0 ? x0 - x0 % 32 : x0;
    R.xs = (x1 - xa + 63) / 64 <= (x1 - x0 + 63) / 64 ? xa : x0;
    R.ntx = (x1 - R.xs + 63) / 64;
    R.nty = (y1 - y0 + TY - 1) / TY;
    R.nseg = (z1 - z0 + tz - 1) / tz;
    R.nblk = R.ntx * R.nty * R.nseg;
    return R;
}

void add_rect(ZSet &s, int x0, int x1, int y0, int y1, int z0, int z1, int tz, int TY, int px)
{
    if (x1 <= x0 || y1 <= y0 || z1 <= z0) return;
    SWP_CHECK(s.n < kRectMax, "acoustic3d: too many block rectangles");
    s.r[s.n] = make_rect(x0, x1, y0, y1, z0, z1, tz, TY, px);
    s.per_shot += s.r[s.n].nblk;
    ++s.n;
}

// Per axis, the computed range [M, n-M) cut at the lean interior
// [lo + M + 1, hi - M - 1): low margin [c0, a), middle [a, b), high margin
// [b, c1).  The margins are exactly the cells in that axis' adjoint CPML band
// and hold its forward band and strip cells.
struct Cuts {
    int c0, a, b, c1;
};

// align > 1 (the x axis on line-aligned rows): the interior starts at the
// next multiple of align, so its tiles cover whole 128-byte lines; the low
// margin takes the few extra cells (its kernels run them without CPML terms).
Cuts cuts(int n, int M, int lo, int hi, int align = 1)
{
    Cuts k;
    k.c0 = M;
    k.c1 = n - M;
    k.a = std::min(std::max(lo + M + 1, k.c0), k.c1);
    k.b = std::min(std::max(hi - M - 1, k.a), k.c1);
    if (align > 1) k.a = std::min((k.a + align - 1) / align * align, k.b);
    return k;
}

// The regions whose axes lie in a margin exactly where (ex, ey, ez) say so.
ZSet region_set(const Geo &g, bool ex, bool ey, bool ez, int tz, int TY)
{
    const Cuts X = cuts(g.nx, g.M, g.X0, g.X1, 32), Y = cuts(g.ny, g.M, g.Y0, g.Y1), Z = cuts(g.nz, g.M, g.Z0, g.Z1);
    int xs[2][2], ys[2][2], zs[2][2];
    int nxr = 0, nyr = 0, nzr = 0;
    auto fill = [](const Cuts &k, bool edge, int out[2][2], int &n) {
        if (edge) {
            out[0][0] = k.c0; out[0][1] = k.a;
            out[1][0] = k.b; out[1][1] = k.c1;
            n = 2;
        } else {
            out[0][0] = k.a; out[0][1] = k.b;
            n = 1;
        }
    };
    fill(X, ex, xs, nxr);
    fill(Y, ey, ys, nyr);
    fill(Z, ez, zs, nzr);
    ZSet s{};
    for (int i = 0; i < nzr; ++i)
        for (int j = 0; j < nyr; ++j)
            for (int l = 0; l < nxr; ++l)
                add_rect(s, xs[l][0], xs[l][1], ys[j][0], ys[j][1], zs[i][0], zs[i][1], tz, TY, g.px);
    return s;
}

template <class K>
void by_order(int M, K &&k)
{
    switch (M) {
    case 1: k(std::integral_constant<int, 1>{}); break;
    case 2: k(std::integral_constant<int, 2>{}); break;
    case 3: k(std::integral_constant<int, 3>{}); break;
    case 4: k(std::integral_constant<int, 4>{}); break;
    default: fail("acoustic3d z-march: order ", 2 * M, " not instantiated");
    }
}

dim3 grid_of(const ZSet &s, int B)
{
    const int64_t n = int64_t(s.per_shot) * B;
    SWP_CHECK(n < (int64_t(1) << 31), "acoustic3d: launch too large");
    return dim3(unsigned(n));
}

void census_region(const char *what, int type, int64_t blocks)
{
    if (!census_on() || !blocks) return;
    const char site[] = {'a', '3', 'd', '.', what[0], what[1], what[2], '3', '.', char('0' + (type & 1)),
                         char('0' + (type >> 1 & 1)), char('0' + (type >> 2 & 1)), 0};
    census_add(site, blocks);
}

// Whether a launch takes z segments of half the height: while it would have
// fewer than kMinWaves waves (SWP_REGION_WAVES overrides, 1 keeps tz) and half
// of tz is still kMinTz planes or more.  A workgroup walks its segment one plane
// (one load latency) at a time, so a launch of few workgroups takes about tz
// plane latencies however few cells it holds; a shorter segment repeats its
// 2M + 1 plane prologue more often.  Measured per gradient at 40 x 36 x 44 (two shots, order 4), 97 x 110
// x 131 and, records only, 128 x 256 x 256 (order 8): 8 planes / 16384 waves
// 41.5, 41.8 and 35.7 ms; 16 planes / 8192 waves 43.7, 44.6 and 36.2 ms.
constexpr int64_t kMinWaves = 16384;
constexpr int kMinTz = 8;

bool halve_tz(int tz, int64_t waves)
{
    return tz / 2 >= kMinTz && waves < tuning(-1, "SWP_REGION_WAVES", kMinWaves);
}

// The plan of the region types in `mask` (bit t: type t).
ZPlan make_zplan(const Geo &g, unsigned mask, int tz)
{
    for (;; tz /= 2) {
        ZPlan p{};
        int64_t blocks = 0;
        for (int t : {7, 3, 5, 6, 1, 2, 4, 0}) {
            if (!(mask >> t & 1)) continue;
            const ZSet s = region_set(g, t & 1, t & 2, t & 4, tz, 4 * ry_of(t));
            if (!s.per_shot) continue;
            const int k = p.n++;
            p.type[k] = t;
            p.ty[k] = 4 * ry_of(t);
            p.per_shot[k] = s.per_shot;
            for (int j = 0; j < s.n; ++j) p.r[p.r0[k] + j] = s.r[j];
            p.r0[k + 1] = p.r0[k] + s.n;
            blocks += (int64_t(s.per_shot) * g.B + 7) / 8 * 8;
            SWP_CHECK(blocks < (int64_t(1) << 31), "acoustic3d: launch too large");
            p.first[k + 1] = int(blocks);
        }
        if (!halve_tz(tz, blocks * 4)) return p;
    }
}

}  // namespace

bool zm_supported(const Geo &g, int &tz)
{
    if (g.M < 1 || g.M > 4) return false;
    const int64_t planes = ((int64_t(1) << 32) - 1) / (4 * g.sxy);   // planes addressable from a segment base
    const int64_t fit = planes - 2 * g.M - 1;
    if (fit < 1) return false;
    tz = int(std::min<int64_t>(tz, fit));
    return true;
}

double zm_lane_ratio(const Geo &g)
{
    int64_t lanes = 0;
    for (int t = 0; t < 8; ++t) {
        const int TY = 4 * ry_of(t);
        const ZSet s = region_set(g, t & 1, t & 2, t & 4, g.nz, TY);
        for (int j = 0; j < s.n; ++j) lanes += int64_t(64) * s.r[j].ntx * TY * s.r[j].nty * (s.r[j].z1 - s.r[j].z0);
    }
    const int64_t cols = int64_t(g.nx - 2 * g.M + 63) / 64 * 64, rows = int64_t(g.ny - 2 * g.M + 3) / 4 * 4;
    return double(lanes) / double(cols * rows * (g.nz - 2 * g.M));
}

int shell_boxes(const Geo &g, Box out[6])
{
    // the six slabs around the lean interior (per-cell shell launches)
    const Cuts X = cuts(g.nx, g.M, g.X0, g.X1, 32), Y = cuts(g.ny, g.M, g.Y0, g.Y1), Z = cuts(g.nz, g.M, g.Z0, g.Z1);
    const Box cand[6] = {
        {X.c0, X.c1, Y.c0, Y.c1, Z.c0, Z.a}, {X.c0, X.c1, Y.c0, Y.c1, Z.b, Z.c1},
        {X.c0, X.c1, Y.c0, Y.a, Z.a, Z.b},   {X.c0, X.c1, Y.b, Y.c1, Z.a, Z.b},
        {X.c0, X.a, Y.a, Y.b, Z.a, Z.b},     {X.b, X.c1, Y.a, Y.b, Z.a, Z.b},
    };
    int n = 0;
    for (const Box &b : cand)
        if (b.x1 > b.x0 && b.y1 > b.y0 && b.z1 > b.z0) out[n++] = b;
    return n;
}

void launch_fwd_zm(const Ctx &x, const StepFields &f, float *u_this, float *strip, bool shell)
{
    const Geo &g = x.g;
    const ZPlan p = make_zplan(g, shell ? 0xffu : 1u, x.tz);
    if (!p.n) return;
    for (int k = 0; k < p.n; ++k) census_region("fwd", p.type[k], int64_t(p.per_shot[k]) * g.B);
    by_order(g.M, [&](auto ms) {
        constexpr int M = decltype(ms)::value;
        hipLaunchKernelGGL((x.big ? fwd3_kernel<M, true> : fwd3_kernel<M, false>), dim3(unsigned(p.first[p.n])), dim3(256),
                           0, stream(), g, x.c, x.pr, f, u_this, strip, p);
    });
    SWP_LAUNCHED();
}

void launch_adj_zm(const Ctx &x, const AdjFields &f, const float *img, float *grad, bool shell)
{
    const Geo &g = x.g;
    const ZPlan p = make_zplan(g, shell ? 0xffu : 1u, x.tz);
    if (!p.n) return;
    for (int k = 0; k < p.n; ++k) census_region("adj", p.type[k], int64_t(p.per_shot[k]) * g.B);
    by_order(g.M, [&](auto ms) {
        hipLaunchKernelGGL(adj3_kernel<decltype(ms)::value>, dim3(unsigned(p.first[p.n])), dim3(256), 0, stream(), g,
                           x.c, x.pr, f, img, grad, p);
    });
    SWP_LAUNCHED();
}

void launch_recon_zm(const Ctx &x, const float *vp, const float *u_prev, const float *u_now, float *u_next,
                     const float *adj, float *grad, int x0, int x1, int y0, int y1, int z0, int z1)
{
    const Geo &g = x.g;
    ZSet s;
    for (int tz = x.tz;; tz /= 2) {
        s = ZSet{};
        add_rect(s, x0, x1, y0, y1, z0, z1, tz, kNwRecon * kRyRecon, x.g.px);
        if (!s.per_shot) return;
        if (!halve_tz(tz, int64_t(s.per_shot) * g.B * kNwRecon)) break;
    }
    census_add("a3d.recon_zm", int64_t(s.per_shot) * g.B);
    by_order(g.M, [&](auto ms) {
        constexpr int M = decltype(ms)::value;
        hipLaunchKernelGGL((recon_zm_kernel<M, kRyRecon, kNwRecon>), grid_of(s, g.B), dim3(64 * kNwRecon), 0, stream(), g, x.c, vp, u_prev,
                           u_now, u_next, adj, grad, s);
    });
    SWP_LAUNCHED();
}

}  // namespace a3d
}  // namespace swp
