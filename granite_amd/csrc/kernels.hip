// gfx950 kernels of the CCZ4 RHS + SSP-RK3 stage engine.
//
// Stage kernel layout: one workgroup per part of a launch tile, one thread per cell. The 22
// fields are streamed one at a time through an LDS box holding the part plus the stencil halo (4
// cells along each axis, 1 cell on the edges used by the mixed second derivatives). The per-cell
// arithmetic is ccz4_cell.hpp; the RK3 combine, the floors and (last stage) the algebraic
// constraints are applied to each value before it is stored, so one launch per stage reads the
// stage input and u^n and writes the new stage state.
#include "kernels.hpp"

#include <cstdint>

// tile shape (overridable at build time): a tile of GR_TILE_X x Y x Z cells is the unit of
// the launch bookkeeping and of the mixed form's choice of precision; the kernels run each tile as
// parts (FP64_PARTS below), one thread per cell
#ifndef GR_TILE_X
#define GR_TILE_X 16
#endif
#ifndef GR_TILE_Y
#define GR_TILE_Y 4
#endif
#ifndef GR_TILE_Z
#define GR_TILE_Z 8
#endif
#ifndef GR_FP64_KO_EXACT
#define GR_FP64_KO_EXACT 1
#endif
// default field groups (second grid dimension) of the ghost fill (1, 2, 4 or 11)
#ifndef GR_GHOST_GROUPS
#define GR_GHOST_GROUPS 4
#endif
// field groups (second grid dimension) of the prolongation and restriction kernels
#ifndef GR_TRANSFER_GROUPS
#define GR_TRANSFER_GROUPS 4
#endif

namespace gr {

// Device buffers reached through tables (block descriptors, stage selectors) are generic
// pointers to the compiler, which would access them with flat instructions; flat accesses
// also count against the LDS wait counter, so every LDS wait would wait for the in-flight
// prefetch of the next field as well. The stage kernels access HBM through this type instead.
typedef __attribute__((address_space(1))) double gdouble;
typedef __attribute__((address_space(1))) char gchar;

// element at byte offset `off` (< 4 GiB) from a workgroup-uniform base
__device__ __forceinline__ double gload(const gdouble* base, unsigned off) {
    return *(const gdouble*)((const gchar*)base + off);
}
__device__ __forceinline__ void gstore(gdouble* base, unsigned off, double v) {
    *(gdouble*)((gchar*)base + off) = v;
}
namespace {

constexpr int HALO = 4;

// ------------------------------------------------------------------------------------
// exact (contraction-free) pointwise pieces shared with the reference
// ------------------------------------------------------------------------------------

// d = a1*s1 + a2*s2 + a3*dt*r, src/main.cpp:328-329
__device__ __forceinline__ double combine_exact(double a1, double s1, double a2, double s2, double a3dt, double r) {
#pragma clang fp contract(off)
    return a1 * s1 + a2 * s2 + a3dt * r;
}

__device__ __forceinline__ double floor_chi(double c) {
    // src/main.cpp:598-602
    if (!__builtin_isfinite(c) || c < 1.0e-4) c = 1.0e-4;
    if (c > 1.5) c = 1.5;
    return c;
}

__device__ __forceinline__ double floor_alpha(double a) {
    // src/main.cpp:603-605
    if (!__builtin_isfinite(a) || a < 1.0e-6) a = 1.0e-6;
    return a;
}

// det(gt) -> 1 by a cube-root rescale (or reset to identity), then remove the trace of A~
// with the cofactors of the rescaled metric, src/main.cpp:622-668
__device__ __forceinline__ void algebraic_exact(double g[6], double A[6]) {
#pragma clang fp contract(off)
    double &xx = g[0], &xy = g[1], &xz = g[2], &yy = g[3], &yz = g[4], &zz = g[5];
    const double det = xx * (yy * zz - yz * yz) - xy * (xy * zz - yz * xz) + xz * (xy * yz - yy * xz);
    if (__builtin_isfinite(det) && det > 1.0e-10) {
        const double s = cbrt(1.0 / det);
        for (int a = 0; a < 6; ++a) g[a] *= s;
    } else {
        xx = 1.0; xy = 0.0; xz = 0.0; yy = 1.0; yz = 0.0; zz = 1.0;
    }
    const double cxx = yy * zz - yz * yz;
    const double cxy = xz * yz - xy * zz;
    const double cxz = xy * yz - xz * yy;
    const double cyy = xx * zz - xz * xz;
    const double cyz = xz * xy - xx * yz;
    const double czz = xx * yy - xy * xy;
    const double tr = cxx * A[0] + cyy * A[3] + czz * A[5] + 2.0 * (cxy * A[1] + cxz * A[2] + cyz * A[4]);
    const double t3 = tr / 3.0;
    for (int a = 0; a < 6; ++a) A[a] -= t3 * g[a];
}

// ------------------------------------------------------------------------------------
// parts of a tile and their LDS boxes
// ------------------------------------------------------------------------------------
// Lane -> cell map of the parts (16 x 4 x TZ): lane bits 0-3 are x, bit 4 the low bit of z, bit
// 5 the low bit of y, and the wave index supplies the rest of y, then of z. A 64-bit read then
// takes each 16-lane group from one row and the 32 lanes of two groups from two planes, which
// are conflict-free where a plane spans 16 doubles modulo 32.
template <int TZ>
struct LaneMap {
    __host__ __device__ static constexpr void cell(int tid, int& x, int& y, int& z) {
        const int w = tid >> 6;
        x = tid & 15;
        z = ((tid >> 4) & 1) + 2 * (w >> 1);
        y = ((tid >> 5) & 1) + 2 * (w & 1);
    }
};

// whether a wave's reads of its cells (doubles, row pitch P, plane stride Q) are free of bank
// conflicts, modelled both as 16-lane groups of 32 four-byte banks and as 32-lane groups of 64
template <int TZ>
constexpr bool lds_conflict_free(int P, int Q) {
    for (int lanes = 16; lanes <= 32; lanes *= 2)
        for (int base = 0; base < 64 * TZ; base += lanes) {
            bool used[32] = {};
            for (int t = base; t < base + lanes; ++t) {
                int x = 0, y = 0, z = 0;
                LaneMap<TZ>::cell(t, x, y, z);
                const int bank = (z * Q + y * P + x) % lanes;
                if (used[bank]) return false;
                used[bank] = true;
            }
        }
    return true;
}

// LDS layout of one field's halo box of a 16 x 4 x TZ part: little more than what some stencil
// reads. Planes z = -1 .. TZ lie one after the other in 12 rows of 24 doubles (x = -4 .. 19) and 16
// doubles of padding, cut to rows y = -1 .. 4 on the two outer ones. Of the planes beyond (z = -4 ..
// -2, TZ + 1 .. TZ + 3) only the z axis reads the part's own 16 x 4 columns: their rows go, two to a block
// of 32 doubles, into the hole of the lower outer plane (A) and after the end (TE: even rows, TO:
// odd rows), each at the place modulo 32 doubles it would have in a plane of its own, so that the
// z taps stay free of bank conflicts. Parts of 16 x 4 x 4 take 16 KiB
// a field (a whole box 27) and, with the rows 64-byte aligned, 158 cache lines (8 x 4 x 8 parts of the
// same size: 188). 128^3, stages 1-2: 8x4x8 whole boxes 570 us, packed 535, 16x4x4 packed 508. Lines are one
// cost among several: the kernel without its loads took 75 us less, without its stores 92, without its
// LDS reads 87, and 16x4x8 parts, with a fifth fewer lines a cell, gained nothing.
template <int TZ>
struct PackedBox {
    static constexpr int TX = 16, TY = 4;
    static constexpr int ROW = TX + 2 * HALO, PL = 304, NP = TZ + 2 * HALO;
    static constexpr int LO = PL * (HALO - 1) + ROW * (HALO - 1) + HALO; // x = 0 of row y = -1 of plane z = -1
    static constexpr int up(int e, int r) { return (e - r + 31) / 32 * 32 + r; } // next e = r modulo 32
    static constexpr int A = up(PL * (HALO - 1) + ROW * (HALO + TY) + TX + HALO, 4);
    static constexpr int TE = up(PL * (NP - HALO) + ROW * (HALO + TY) + TX + HALO, 4);
    static constexpr int TO = up(TE + 5 * 32, 12);
    static constexpr int SIZE = TO + 6 * 32 - LO;
    static_assert(NP % 2 == 0 && PL % 32 == 16 && LO % 2 == 0, "parity of the far planes, residue of a plane");

    // whether some stencil reads (x, y, z): the axes reach 4 cells, the mixed derivatives 1 on edges
    __host__ __device__ static constexpr bool read(int x, int y, int z) {
        const bool xi = x >= 0 && x < TX, yi = y >= 0 && y < TY, zi = z >= 0 && z < TZ;
        const bool xe = x >= -1 && x <= TX, ye = y >= -1 && y <= TY, ze = z >= -1 && z <= TZ;
        return (yi && zi) || (xi && zi) || (xi && yi) || (xe && ye && zi) || (xe && yi && ze) || (xi && ye && ze);
    }
    // planes (0, 1), (2, NP - 3), (NP - 2, NP - 1) share blocks
    __host__ __device__ static constexpr int far(int x, int y, int p) {
        const int j = 3 * (y >> 1) + (p < 2 ? 0 : (p >= NP - 2 ? 2 : 1));
        const int odd = y & 1, u = (16 * p + 24 * y - 8 * odd) & 31;
        return (odd ? TO + 32 * j : (j ? TE - 32 + 32 * j : A)) + u + x;
    }
    // double of the buffer that holds (x, y, z), for every point some stencil reads
    __host__ __device__ static constexpr int pos(int x, int y, int z) {
        const int p = z + HALO;
        return (p < 3 || p > NP - HALO ? far(x, y, p) : PL * p + ROW * (y + HALO) + x + HALO) - LO;
    }
    // the point (x even) that fills double e (even) of the buffer. Doubles no stencil reads (row
    // ends of the y halo, padding, holes) name the nearest point read of their row or the row
    // before, so that the lane that fills them adds no cache line to its load
    __host__ __device__ static constexpr void point(int e, int& x, int& y, int& z) {
        e += LO;
        const bool inA = e >= A && e < A + 32;
        if (inA || e >= TE) {
            const int odd = e >= TO ? 1 : 0, t = inA ? e - A : (odd ? e - TO : e - TE + 32);
            const int b = t >> 5 > 5 ? 5 : t >> 5, h = b >= 3 ? 1 : 0, j = b - 3 * h;
            x = t & 15;
            y = 2 * h + odd;
            const int half = (t >> 4) & 1, even = ((24 * y - 8 * odd) >> 4) & 1; // the half of the even plane
            const int pe = j == 0 ? 0 : (j == 1 ? 2 : NP - 2), po = j == 0 ? 1 : (j == 1 ? NP - 3 : NP - 1);
            z = (half == even ? pe : po) - HALO;
            return;
        }
        const int pl = e / PL, r = e % PL;
        const bool outer = pl < HALO || pl >= NP - HALO; // planes z = -1 and z = TZ
        const int row = r / ROW - HALO, ylo = outer ? -1 : -HALO, yhi = outer ? TY : TY + HALO - 1;
        y = row < ylo ? ylo : (row > yhi ? yhi : row);
        z = pl > NP - HALO ? TZ : pl - HALO;
        const bool own = y >= 0 && y < TY, edge = y >= -1 && y <= TY;
        const int m = (own && !outer) ? HALO : ((own || (edge && !outer)) ? 2 : 0); // x reach (even)
        x = r % ROW - HALO;
        x = x < -m ? -m : (x > TX - 2 + m ? TX - 2 + m : x);
    }
    // every point read has a place of its own, in the bank of its place in a whole box, and the
    // place knows its point
    static constexpr bool consistent() {
        for (int z = -HALO; z < TZ + HALO; ++z)
            for (int y = -HALO; y < TY + HALO; ++y)
                for (int x = -HALO; x < TX + HALO; ++x) {
                    if (!read(x, y, z)) continue;
                    const int e = pos(x, y, z);
                    if (e < 0 || e >= SIZE || (e - pos(x & ~1, y, z)) != (x & 1)) return false;
                    int u = 99, v = 99, w = 99;
                    point(e & ~1, u, v, w);
                    if (u != (x & ~1) || v != y || w != z) return false;
                    const int natural = PL * (z + HALO) + ROW * (y + HALO) + x + HALO - LO;
                    if ((e - natural) % 32 != 0) return false;
                }
        return true;
    }
};
// Taps of a packed box. The z taps two cells off and more have an address of their own per lane; the
// others are reached from three bases per buffer, below the taps of the cell's own plane and of
// the planes next to it, each near enough for the paired LDS reads' 8-bit offsets: from the cell
// itself the compiler adds an address for nearly every pair, 228 instructions a part (128^3,
// stages 1-2: 504 -> 497 us; the uneven 64 blocks 772 -> 762).
template <class Box, typename R>
struct PackedTaps {
    typedef const __attribute__((address_space(3))) R* LdsPtr;
    static constexpr int NB = 4; // buffers, at most
    LdsPtr z[6];        // z - 4, - 3, - 2, + 2, + 3, + 4 in buffer 0
    LdsPtr base[NB][3]; // per buffer: planes z - 1, z, z + 1
    int buf, ofs;       // the current field's buffer and its first double
    // the small parts run one wave per SIMD, with no other to cover a wait: all LDS reads of a field
    // ahead of its arithmetic (a 16^3 stage 23.4 -> 21.3 us, 32^3 25.3 -> 23.4). With two waves
    // the registers that costs are worth more (128^3: 519 us against 508 without).
    static constexpr bool READS_FIRST = Box::NP == 2 + 2 * HALO;
    __device__ static constexpr int low(int p) { return p == 1 ? -HALO * Box::ROW : (p - 1) * Box::PL - Box::ROW; }
    __device__ __forceinline__ void place(LdsPtr lds, int lx, int ly, int lz, int nbuf, int size) {
#pragma unroll
        for (int k = 0; k < 6; ++k) z[k] = lds + Box::pos(lx, ly, lz + (k < 3 ? k - 4 : k - 1));
#pragma unroll
        for (int b = 0; b < NB; ++b)
#pragma unroll
            for (int p = 0; p < 3; ++p) {
                if (b >= nbuf) continue;
                base[b][p] = lds + Box::pos(lx, ly, lz) + b * size + low(p);
#ifdef __HIP_DEVICE_COMPILE__
                asm("" : "+v"(base[b][p])); // kept as one address: offsets from it fit the reads
#endif
            }
    }
    __device__ __forceinline__ R near(int dz, int q) const { return base[buf][dz + 1][q - low(dz + 1) + dz * Box::PL]; }
    __device__ __forceinline__ R at(const R*, int d, int k) const {
        if (d == 2 && (k >= 2 || k <= -2)) return z[k < 0 ? k + 4 : k + 1][ofs];
        return d == 2 ? near(k, 0) : near(0, d == 1 ? k * Box::ROW : k);
    }
    __device__ __forceinline__ R centre(const R*) const { return near(0, 0); }
    // i cells along axis a and j along axis b > a (i, j = -1 or 1)
    __device__ __forceinline__ R edge(const R*, int a, int b, int i, int j) const {
        const int q = a == 0 ? i : i * Box::ROW;
        return b == 2 ? near(j, q) : near(0, q + j * Box::ROW);
    }
};

// Order in which a kernel stages the fields: N fields, field(pos) at position pos.
struct RhsOrder {
    static constexpr int N = NV;
    __host__ __device__ static constexpr int field(int pos) { return FIELD_ORDER[pos]; }
    __host__ __device__ static constexpr int pos(int v) { return field_pos(v); }
};
// The constraint monitor's: metric, chi, Gamma-hat for H; with the momentum constraint also K and A~.
template <bool MOM>
struct MonitorOrder {
    static constexpr int N = MOM ? 17 : 10;
    __host__ __device__ static constexpr int field(int pos) {
        return pos < 6 ? GXX + pos : (pos == 6 ? CHI : (pos < 10 ? GHX + pos - 7 : (pos == 10 ? KTR : AXX + pos - 11)));
    }
    __host__ __device__ static constexpr int pos(int v) {
        int p = 0;
        while (field(p) != v) ++p;
        return p;
    }
};

// byte offset of the pair at (x, y, z) of the part, or of the part's first pair where it lies
// beyond the block (a pair at the end of an odd row takes the next row's first cell along)
__device__ __forceinline__ unsigned pair_offset(int x, int y, int z, int ox, int oy, int oz, const BlockDesc& b) {
    const int gx = ox + x, gy = oy + y, gz = oz + z;
    const int i = gx + b.nt[0] * (gy + b.nt[1] * gz);
    const bool ok = gx < b.nt[0] && gy < b.nt[1] && gz < b.nt[2] && i + 1 < b.nt[0] * b.nt[1] * b.nt[2];
    return 8u * (unsigned)(ok ? i : ox + b.nt[0] * (oy + b.nt[1] * oz));
}

// Per-thread input/output of one cell of an FP64 part: stages the fields into LDS for the
// stencils (Stager interface of ccz4_cell) and combines/stores the results (Sink interface).
//
// The halo goes straight from global memory to LDS, into a packed box: lane l of a wave's load of
// chunk c writes doubles 128 c + 2 l, + 1 of the buffer, fetched from the pair of x-neighbours the
// layout puts there (slots beyond the block fetch the part's first pair and are never read by an
// active cell); u^n of the cells is staged beside it. With NBUF field buffers, field p + NBUF - 1 is
// loaded while field p is evaluated. A load's LDS data is complete once the wave's vector memory
// counter has counted it back; the counter drains in issue order (loads and stores alike), so the
// barrier that starts field p waits until no more of this wave's operations are outstanding than it
// has issued since the loads of field p: the loads of the fields after p stay in flight across it.
// No vector register is loaded from memory between the first barrier and the last: the compiler does
// not count such a load's turn among the direct ones and would drain them all at its use (nine times
// a part when u^n went through registers).
// The 16-byte loads are aligned to 8 bytes only where rows are of odd length.
// UN_IN: u^n is the stage input itself (the first stage, chosen at launch), so its value at the
// cell is the centre value the combine already receives and is not loaded again (526 us against 590
// for the two stages of a 128^3 block, 8x4x8 parts).
template <int TZ, int MODE, bool UN_IN, class Order = RhsOrder>
struct TileIODma {
    typedef __attribute__((address_space(3))) double* LdsPtr;
    using Box = PackedBox<TZ>;
    static constexpr int NT = Box::TX * Box::TY * TZ;
    static_assert(Box::consistent() && lds_conflict_free<TZ>(Box::ROW, Box::PL), "packed box of the part");
    static constexpr int CH = 128; // doubles per chunk (64 lanes x 16 bytes)
    static constexpr int NCH = (Box::SIZE + CH - 1) / CH;
    static constexpr int LBUF = NCH * CH; // doubles per buffer
    static constexpr int NW = NT / 64; // waves
    static constexpr int KW = NCH / NW; // chunk loads per wave
    static_assert(NT % 64 == 0 && NCH % NW == 0, "whole waves, the same number of chunks for each");
    // doubles per buffer of the cells' own u^n values, staged beside the field (slot = thread)
    static constexpr int UNB = MODE == MODE_RHS || UN_IN ? 0 : NT;
    // in the last stage the new metric of every cell waits in LDS from its combine to the
    // algebraic constraints at the end
    static constexpr int METRIC = MODE == MODE_FINAL ? 6 * NT : 0;
    // field buffers: as many as fit (4 at most) while two workgroups share the CU's 160 KB
    static constexpr int fits(int n) { return (n * (LBUF + UNB) + METRIC) * 8 * 2 <= 163840; }
    static constexpr int NBUF = fits(4) ? 4 : 3;
    static_assert(fits(NBUF), "field buffers");
    // first double of each region (u^n first, so that every LDS address is a lane's own plus an
    // immediate offset of 16 bits)
    static constexpr int BUF0 = NBUF * UNB, METRIC0 = BUF0 + NBUF * LBUF;
    static constexpr int LDS_DOUBLES = METRIC0 + METRIC;
    // vector memory operations a wave issues after its loads of field `pos` and before the
    // barrier of that field, at least: in each turn between, the loads of one more field with its
    // u^n; for the first fields the loads issued at the start. (Results are stored too, but a
    // wave outside the block stores none.)
    __host__ __device__ static constexpr int younger(int pos) {
        int n = 0;
        for (int f = pos + 1; f <= pos + NBUF - 2 && f < Order::N; ++f) n += KW + (UNB && f >= NBUF - 1 ? 1 : 0);
        return n;
    }

    double* lds; // LDS_DOUBLES doubles
    const gdouble* in;
    const gdouble* un;
    gdouble* out;
    long stride;
    unsigned cb; // byte offset of the thread's cell inside one field
    int wave;
    bool active;
    bool ko_on;
    StageCoef cf;
    unsigned doff[KW]; // byte offset of this lane's pair in each of its wave's chunks
    unsigned uoff; // byte offset of the u^n pair this lane stages (lanes 0-31: the wave's 64 cells)
    int tid;
    PackedTaps<Box, double> taps;
    double unA[6]; // u^n of A~, whose results come after the last field
    double hA[6];

    __device__ __forceinline__ void place(int lx, int ly, int lz) {
        taps.place((LdsPtr)lds + BUF0, lx, ly, lz, NBUF, LBUF);
    }

    __device__ void init(int tid_, int ox, int oy, int oz, const BlockDesc& b) {
        tid = tid_;
        wave = __builtin_amdgcn_readfirstlane(tid / 64); // uniform: LDS bases go to M0 from scalars
        const int lane = tid % 64;
        int x = 0, y = 0, z = 0;
#pragma unroll
        for (int k = 0; k < KW; ++k) {
            Box::point((wave + k * NW) * CH + 2 * lane, x, y, z);
            doff[k] = pair_offset(x, y, z, ox, oy, oz, b);
        }
        LaneMap<TZ>::cell(wave * 64 + 2 * (lane % 32), x, y, z);
        uoff = pair_offset(x, y, z, ox, oy, oz, b);
#pragma unroll
        for (int p = 0; p < NBUF - 1; ++p) prefetch(p);
    }

    __device__ __forceinline__ void prefetch(int pos) {
        if (pos >= Order::N) return;
        const int v = Order::field(pos);
        const gchar* f = (const gchar*)(in + v * stride);
        // the LDS base is made opaque at every field, so the chunk addresses (M0 values) are
        // recomputed from it with one scalar add each instead of being kept (and spilled) as
        // 2 x KW live scalars across the whole kernel
        unsigned base = __builtin_amdgcn_readfirstlane((unsigned)(uintptr_t)(LdsPtr)lds);
#ifdef __HIP_DEVICE_COMPILE__
        asm volatile("" : "+s"(base));
#endif
        LdsPtr L = (LdsPtr)(uintptr_t)base;
        const LdsPtr U = L + (pos % NBUF) * UNB + wave * 64;
        L += BUF0 + (pos % NBUF) * LBUF;
#pragma unroll
        for (int k = 0; k < KW; ++k) {
            const int c = wave + k * NW; // uniform over the wave
#ifdef __HIP_DEVICE_COMPILE__
            // keeps the 32-bit offset at the load (scalar base + offset), in place
            asm volatile("" : "+v"(doff[k]));
#endif
            __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void*)(f + doff[k]),
                                             (__attribute__((address_space(3))) void*)(L + c * CH), 16, 0, 0);
        }
        // u^n of the wave's own cells (which only this wave overwrites, in the last stage)
        if (UNB && tid % 64 < 32) {
#ifdef __HIP_DEVICE_COMPILE__
            asm volatile("" : "+v"(uoff));
#endif
            __builtin_amdgcn_global_load_lds(
                (const __attribute__((address_space(1))) void*)((const gchar*)(un + v * stride) + uoff),
                (__attribute__((address_space(3))) void*)U, 16, 0, 0);
        }
    }
    __device__ __forceinline__ double staged_un(int v) const {
        return lds[(Order::pos(v) % NBUF) * UNB + tid];
    }

    // at most n of this wave's vector memory operations outstanding (n a constant after
    // inlining), its LDS accesses done
    static __device__ __forceinline__ void wait_outstanding(int n) {
#ifdef __HIP_DEVICE_COMPILE__
        asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" ::"i"(n) : "memory");
#endif
    }
    // ---- Stager
    __device__ double centre(int v) const { return gload(in + v * stride, cb); }
    __device__ void metric64(double g[6]) const {
#pragma unroll
        for (int a = 0; a < 6; ++a) g[a] = gload(in + (GXX + a) * stride, cb);
    }
    __device__ const PackedTaps<Box, double>& strides() const { return taps; }
    __device__ const double* field(int v) {
        const int pos = Order::pos(v);
        // this wave's loads of field pos have landed and its LDS accesses are done; then the
        // barrier: every wave's loads of pos have landed and every thread is done with field
        // pos - 1, whose buffer the prefetch refills. Written as statements that may touch any
        // memory, so the compiler keeps every access on its side; a workgroup fence would also
        // drain the loads of the fields after pos (they write LDS)
        wait_outstanding(younger(pos));
#ifdef __HIP_DEVICE_COMPILE__
        asm volatile("s_barrier" ::: "memory");
#endif
        prefetch(pos + NBUF - 1);
        if (UNB && v >= AXX && v < AXX + 6) unA[v - AXX] = staged_un(v);
        taps.buf = pos % NBUF;
        taps.ofs = (pos % NBUF) * LBUF;
        return lds; // the taps know the cell
    }

    // ---- Sink
    __device__ __forceinline__ void put(int v, double r, double ko, double uin) {
        const double rr = ko_on ? r + ko : r;
        if (MODE == MODE_RHS) {
            if (active) gstore(out + v * stride, cb, rr);
            return;
        }
        const double u0 = UN_IN ? uin : (v >= AXX && v < AXX + 6 ? unA[v - AXX] : staged_un(v));
        double val = combine_exact(cf.a1, u0, cf.a2, uin, cf.a3dt, rr);
        if (v == CHI) val = floor_chi(val);
        if (v == ALPHA) val = floor_alpha(val);
        // last stage: the new metric waits in LDS (this thread's own slots) for the algebraic
        // constraints, instead of in registers across the rest of the RHS; A~ comes last and is
        // held in registers
        if (MODE == MODE_FINAL && v >= GXX && v < GXX + 6) {
            lds[METRIC0 + (v - GXX) * NT + tid] = val;
            return;
        }
        if (MODE == MODE_FINAL && v >= AXX && v < AXX + 6) {
            hA[v - AXX] = val;
            return;
        }
        if (active) gstore(out + v * stride, cb, val);
    }

    __device__ __forceinline__ void finish() {
        if (MODE != MODE_FINAL) return;
        double hg[6];
#pragma unroll
        for (int a = 0; a < 6; ++a) hg[a] = lds[METRIC0 + a * NT + tid];
        algebraic_exact(hg, hA);
        if (!active) return;
#pragma unroll
        for (int a = 0; a < 6; ++a) {
            gstore(out + (GXX + a) * stride, cb, hg[a]);
            gstore(out + (AXX + a) * stride, cb, hA[a]);
        }
    }
};

// Mixed-precision counterpart of TileIODma: the stencils and the RHS algebra see FP32
// values, the RK3 combine, the floors and the algebraic constraints are done in FP64 on
// the FP64 state. Each field is staged as FP32 deltas from one FP64 reference value per
// tile (the field at the tile's first cell): every stencil's weights sum to zero, so
// derivatives of the deltas are derivatives of the field, while small structure on top of
// an O(1) field (1e-8 noise on the metric) keeps FP32 relative precision of the delta.
// The box is the packed one of the FP64 parts in floats, filled through registers one field ahead (the
// deltas are formed on the way), by the pairs each lane would load directly: four 16-byte loads
// and four 8-byte LDS writes a thread and field. 16x4x4 parts of 256 threads against whole 16x4x8
// tiles of 512 with a box of single values and its corners: two or three independent workgroups per
// CU instead of one (128^3: stages 1-2 516 -> 485 us,
// stage 3 557 -> 521; 192^3 1665 -> 1551, 1800 -> 1673). At three waves per SIMD (168 registers) stage
// 3 gains 2% at 128^3 and loses 7% at 101x77x59, where FP64 tiles are a larger share.
// UN_IN: u^n is the stage input itself (the first stage, chosen at launch): its value at the
// cell is the stage input's centre value, so it is not loaded separately
template <int TZ, int MODE, bool UN_IN = false>
struct TileIO32 {
    using Box = PackedBox<TZ>;
    typedef __attribute__((address_space(3))) float* LdsPtr;
    typedef double pair __attribute__((ext_vector_type(2), aligned(8)));
    typedef float pair32 __attribute__((ext_vector_type(2)));
    static constexpr int NT = Box::TX * Box::TY * TZ, CH = 128, NCH = (Box::SIZE + CH - 1) / CH;
    static constexpr int LBUF = NCH * CH, KW = NCH / (NT / 64);
    static_assert(Box::consistent() && NCH % (NT / 64) == 0, "packed box, the same number of chunks for each wave");

    float* lds; // 2 * LBUF floats
    const gdouble* in; // global address space: loads/stores wait on vmcnt only, never on LDS waits
    const gdouble* un;
    gdouble* out;
    long stride;
    unsigned cb; // byte offset of the thread's cell inside one field
    long ridx; // the tile's reference cell
    bool active;
    bool ko_on;
    StageCoef cf;
    int tid;
    unsigned doff[KW]; // byte offset of the thread's pairs of the halo box
    PackedTaps<Box, float> taps;
    pair buf[KW];
    double refb, unb, inb;
    double unv[NV], inv[NV];
    double* metric; // last stage: the new metric waits in LDS (6 * NT doubles) for the algebraic constraints
    double hA[6];

    __device__ void init(int tid_, int lx, int ly, int lz, int ox, int oy, int oz, const BlockDesc& b) {
        tid = tid_;
        taps.place((LdsPtr)lds, lx, ly, lz, 2, LBUF);
#pragma unroll
        for (int k = 0; k < KW; ++k) {
            int x = 0, y = 0, z = 0;
            Box::point(2 * (tid + k * NT), x, y, z);
            doff[k] = pair_offset(x, y, z, ox, oy, oz, b);
        }
        prefetch(0);
        stage_to_lds(0);
        prefetch(1);
    }

    __device__ __forceinline__ void prefetch(int pos) {
        if (pos >= NV) return;
        const int v = FIELD_ORDER[pos];
        const gdouble* f = in + v * stride;
#pragma unroll
        for (int k = 0; k < KW; ++k)
            buf[k] = *(const __attribute__((address_space(1))) pair*)((const gchar*)f + doff[k]);
        refb = f[ridx];
        inb = gload(f, cb);
        if (MODE != MODE_RHS && !UN_IN) unb = gload(un + v * stride, cb);
    }

    __device__ __forceinline__ void stage_to_lds(int pos) {
        if (pos >= NV) return;
        float* L = lds + (pos & 1) * LBUF;
        const double r = refb;
#pragma unroll
        for (int k = 0; k < KW; ++k)
            *(pair32*)(L + 2 * (tid + k * NT)) = pair32{(float)(buf[k].x - r), (float)(buf[k].y - r)};
        const int v = FIELD_ORDER[pos];
        inv[v] = inb;
        if (MODE != MODE_RHS) unv[v] = UN_IN ? inb : unb;
    }

    // ---- Stager
    __device__ float centre(int v) const { return (float)gload(in + v * stride, cb); }
    __device__ void metric64(double g[6]) const {
#pragma unroll
        for (int a = 0; a < 6; ++a) g[a] = gload(in + (GXX + a) * stride, cb);
    }
    __device__ const PackedTaps<Box, float>& strides() const { return taps; }
    __device__ const float* field(int v) {
        const int pos = field_pos(v);
        __syncthreads();
        stage_to_lds(pos + 1);
        prefetch(pos + 2);
        taps.buf = pos & 1;
        taps.ofs = (pos & 1) * LBUF;
        return lds; // the taps know the cell
    }

    // ---- Sink (FP64 combine on the FP64 stage input and u^n)
    __device__ __forceinline__ void put(int v, float r, float ko, float) {
        const double rr = ko_on ? (double)r + (double)ko : (double)r;
        if (MODE == MODE_RHS) {
            if (active) gstore(out + v * stride, cb, rr);
            return;
        }
        double val = combine_exact(cf.a1, unv[v], cf.a2, inv[v], cf.a3dt, rr);
        if (v == CHI) val = floor_chi(val);
        if (v == ALPHA) val = floor_alpha(val);
        if (MODE == MODE_FINAL && v >= GXX && v < GXX + 6) {
            metric[(v - GXX) * NT + tid] = val;
            return;
        }
        if (MODE == MODE_FINAL && v >= AXX && v < AXX + 6) {
            hA[v - AXX] = val;
            return;
        }
        if (active) gstore(out + v * stride, cb, val);
    }

    __device__ __forceinline__ void finish() {
        if (MODE != MODE_FINAL) return;
        double hg[6];
#pragma unroll
        for (int a = 0; a < 6; ++a) hg[a] = metric[a * NT + tid];
        algebraic_exact(hg, hA);
        if (!active) return;
#pragma unroll
        for (int a = 0; a < 6; ++a) {
            gstore(out + (GXX + a) * stride, cb, hg[a]);
            gstore(out + (AXX + a) * stride, cb, hA[a]);
        }
    }
};

struct StageArgs {
    Batch batch;
    int sel_in, sel_un, sel_out;
    int ntiles;
    int xcd_remap;
    Stencil<double> K;
    Stencil<float> K32;
    CellParams P;
    StageCoef cf;
    int ko_on;
    // tiles whose flag differs from `want` are left to the other precision's kernel
    const unsigned char* flags;
    int want;
    // scan != 0: launched as stage_kernel_scan over a small grid
    int scan;
};

// workgroup id -> tile id: consecutive tiles go to the same XCD (workgroups are dealt
// round-robin over the 8 XCDs), so that halo rows shared by neighbouring tiles are
// found in that XCD's L2.
__device__ __forceinline__ int tile_of_block(int bid, int ntiles, int remap) {
    if (!remap) return bid;
    // XCD x = bid % 8 takes ntiles / 8 consecutive slots, one more for the first ntiles % 8
    const int q = ntiles >> 3, r = ntiles & 7, x = bid & 7;
    return x * q + (x < r ? x : r) + (bid >> 3);
}

// a value the whole workgroup holds alike, moved to scalar registers
__device__ __forceinline__ unsigned long long wg_uniform(unsigned long long v) {
    const unsigned lo = __builtin_amdgcn_readfirstlane((unsigned)v);
    const unsigned hi = __builtin_amdgcn_readfirstlane((unsigned)(v >> 32));
    return ((unsigned long long)hi << 32) | lo;
}
template <class P>
__device__ __forceinline__ P* wg_uniform(P* p) {
    return (P*)wg_uniform((unsigned long long)p);
}

// the block and local tile coordinates of global tile t (uniform per workgroup)
struct TileRef {
    BlockDesc b;
    const gdouble* in; // global address space: loads/stores wait on vmcnt only, never on LDS waits
    const gdouble* un;
    gdouble* out;
    Sources src;
    int tix, tiy, tiz;
};

__device__ __forceinline__ TileRef resolve_tile(const StageArgs& A, int t) {
    TileRef r;
    int tile0, tiles0, tiles1;
    const double *b0, *b1, *b2;
    if (A.batch.table) {
        const BatchBlock& BB = A.batch.table[A.batch.tile_block[t]];
        r.b = BB.b;
        r.src = BB.src;
        b0 = BB.buf[0];
        b1 = BB.buf[1];
        b2 = BB.buf[2];
        tile0 = BB.tile0;
        tiles0 = BB.tiles[0];
        tiles1 = BB.tiles[1];
    } else {
        r.b = A.batch.one.b;
        r.src = A.batch.one.src;
        b0 = A.batch.one.buf[0];
        b1 = A.batch.one.buf[1];
        b2 = A.batch.one.buf[2];
        tile0 = 0;
        tiles0 = A.batch.one.tiles[0];
        tiles1 = A.batch.one.tiles[1];
    }
    const double* bufs[3] = {b0, b1, b2};
    // t is the same for the whole workgroup, and so is everything read for it
    r.in = wg_uniform((const gdouble*)bufs[A.sel_in]);
    r.un = wg_uniform((const gdouble*)bufs[A.sel_un]);
    r.out = wg_uniform((gdouble*)const_cast<double*>(bufs[A.sel_out]));
    r.b.stride = (long)wg_uniform((unsigned long long)r.b.stride);
    const int lt = t - tile0;
    // Tile order: x fastest, then z inside groups of 4 layers, then y, then the groups. The
    // workgroups that run together on one XCD (consecutive tiles) then cover a brick of
    // tiles whose y and z halo rows they share in that XCD's L2 (x, y, z order: 5% slower
    // at 128^3, where the stage input does not fit the memory-side cache).
    {
        constexpr int G = 4;
        const int tiles2 = (r.b.n[2] + GR_TILE_Z - 1) / GR_TILE_Z;
        const int row = lt / tiles0; // (y, z) row of tiles
        const int grp = row / (G * tiles1), in = row % (G * tiles1);
        const int gz = min(G, tiles2 - grp * G); // z layers in this group
        r.tix = lt % tiles0;
        r.tiz = grp * G + in % gz;
        r.tiy = in / gz;
    }
    return r;
}

// matter sources of the cell (zero for a block without sources: a vacuum block of a batch
// that has sources elsewhere; zero sources give the vacuum RHS bit for bit)
__device__ __forceinline__ void load_sources(const Sources& S, long cidx, CellSources& src) {
    if (!S.rho) { // uniform over the workgroup
        src.rho = src.S = 0.0;
#pragma unroll
        for (int a = 0; a < 3; ++a) src.Si[a] = 0.0;
#pragma unroll
        for (int a = 0; a < 6; ++a) src.Sij[a] = 0.0;
        return;
    }
    const gdouble *rho = (const gdouble*)S.rho, *Si = (const gdouble*)S.Si, *Sij = (const gdouble*)S.Sij,
                  *St = (const gdouble*)S.S;
    src.rho = rho[cidx];
    src.S = St[cidx];
#pragma unroll
    for (int a = 0; a < 3; ++a) src.Si[a] = Si[3 * cidx + a];
#pragma unroll
    for (int a = 0; a < 6; ++a) src.Sij[a] = Sij[6 * cidx + a];
}

static_assert(GR_TILE_X == 16 && GR_TILE_Y == 4 && GR_TILE_Z % 4 == 0, "the FP64 parts (16 x 4 x TZ) tile the launch tiles");
constexpr int TILE_X = GR_TILE_X, TILE_Y = GR_TILE_Y, TILE_Z = GR_TILE_Z;
// parts of a tile of TZ layers, one workgroup of 64 TZ threads each
template <int TZ>
constexpr int FP64_PARTS = TILE_Z / TZ;

// part `part` of a tile: layers part * TZ .. of it
template <int TZ, int MODE, bool HAS_SRC, bool KO_EXACT, bool UN_IN>
__device__ __forceinline__ void stage_tile(const StageArgs& A, const TileRef& R, int part, double* lds) {
    const BlockDesc& b = R.b;
    const int tid = threadIdx.x;
    int lx = 0, ly = 0, lz = 0;
    LaneMap<TZ>::cell(tid, lx, ly, lz);
    const int x0 = R.tix * TILE_X, y0 = R.tiy * TILE_Y, z0 = R.tiz * TILE_Z + part * TZ;
    const int ix = x0 + lx, iy = y0 + ly, iz = z0 + lz; // interior-relative
    const bool active = ix < b.n[0] && iy < b.n[1] && iz < b.n[2];
    const int gi = b.ng + (active ? ix : 0), gj = b.ng + (active ? iy : 0), gk = b.ng + (active ? iz : 0);
    const long cidx = gi + (long)b.nt[0] * (gj + (long)b.nt[1] * gk);

    TileIODma<TZ, MODE, UN_IN> io;
    io.lds = lds;
    io.in = R.in;
    io.un = R.un;
    io.out = R.out;
    io.stride = b.stride;
    io.cb = 8u * (unsigned)cidx;
    io.place(lx, ly, lz);
    io.active = active;
    io.ko_on = A.ko_on != 0;
    io.cf = A.cf;
    io.init(tid, b.ng + x0, b.ng + y0, b.ng + z0, b);

    CellSources src{};
    if (HAS_SRC) load_sources(R.src, cidx, src);
    ccz4_cell<double, HAS_SRC, KO_EXACT>(io, io, A.K, A.P, src);
}

// whether part `part` of tile R holds no cell of the block (uniform over the workgroup)
template <int TZ>
__device__ __forceinline__ bool part_outside(const TileRef& R, int part) {
    return R.tiz * TILE_Z + part * TZ >= R.b.n[2];
}

// one part of one tile per workgroup (FP64_PARTS consecutive workgroups per tile); two waves per
// SIMD (256 registers) for the large parts
template <int TZ, int MODE, bool HAS_SRC, bool KO_EXACT, bool UN_IN>
__global__ __launch_bounds__(64 * TZ, TZ / 2) void stage_kernel(StageArgs A) {
    constexpr int NP = FP64_PARTS<TZ>;
    __shared__ __align__(16) double lds[TileIODma<TZ, MODE, UN_IN>::LDS_DOUBLES];
    const int slot = tile_of_block(blockIdx.x, A.ntiles * NP, A.xcd_remap);
    const int tile = slot / NP, part = slot % NP;
    const TileRef R = resolve_tile(A, tile);
    if (part_outside<TZ>(R, part)) return; // whole workgroup leaves before any barrier
    stage_tile<TZ, MODE, HAS_SRC, KO_EXACT, UN_IN>(A, R, part, lds);
}

// the parts of the flagged tiles only, from a small grid: each workgroup gathers those with
// flags == want among parts blockIdx.x + k * gridDim.x and runs them one after the other. By part
// and not by tile, so that the parts of a tile run beside each other: small blocks, whose few FP64
// tiles take longer than all others, wait for one part instead of two (with the FP32 parts, mixed
// 32^3 step 244 -> 196 us, 64^3 332 -> 292, 101x77x59 711 -> 620).
// (every thread takes the same trip counts, so the barriers are uniform)
template <int TZ, int MODE, bool HAS_SRC, bool KO_EXACT, bool UN_IN>
__global__ __launch_bounds__(64 * TZ) void stage_kernel_scan(StageArgs A) {
    constexpr int NT = 64 * TZ;
    __shared__ __align__(16) double lds[TileIODma<TZ, MODE, UN_IN>::LDS_DOUBLES];
    __shared__ int list[NT];
    __shared__ int nlist;
    constexpr int NP = FP64_PARTS<TZ>;
    const int per = (int)gridDim.x * NT, nparts = A.ntiles * NP;
    for (int base = 0; base < nparts; base += per) {
        if (threadIdx.x == 0) nlist = 0;
        __syncthreads();
        const int t = base + (int)blockIdx.x + (int)threadIdx.x * (int)gridDim.x;
        if (t < nparts && A.flags[t / NP] == A.want) list[atomicAdd(&nlist, 1)] = t;
        __syncthreads();
        const int n = nlist;
        __syncthreads();
        for (int item = 0; item < n; ++item) {
            const int unit = list[item], part = unit % NP;
            const TileRef R = resolve_tile(A, unit / NP);
            if (part_outside<TZ>(R, part)) continue; // uniform over the workgroup
            stage_tile<TZ, MODE, HAS_SRC, KO_EXACT, UN_IN>(A, R, part, lds);
            __syncthreads(); // the next part reuses the LDS buffers
        }
    }
}

// Layers of the parts of large and of small launches, and the tiles from which a launch is large.
// Larger parts load less halo per cell; a launch whose small parts find a CU each takes as long
// as one part, and a small part is the shorter (stages 1-2 / 3, us, 2 against 4 layers: 16^3
// 21.3 / 23.0 against 23.9 / 24.9, 32^3, 64 tiles, 23.4 / 25.5 against 25.2 / 26.7; 37x29x23, 72
// tiles, 29.2 / 25.8 against 25.1 / 26.2).
constexpr int TZ_LARGE = 4, TZ_SMALL = 2;
constexpr int LARGE_TILES = 256 / FP64_PARTS<TZ_SMALL> + 1; // small parts outnumber the 256 CUs
// workgroups of the FP64 pass of the mixed form: one per CU
constexpr int FP64_SCAN_GRID = 256;

// one part of TZ layers of a launch tile per workgroup; the tile is the unit of the FP32 / FP64
// choice and of the reference value of the deltas
template <int TZ, int MODE, bool HAS_SRC, bool UN_IN = false>
__global__ __launch_bounds__(64 * TZ, 2) void stage_kernel_mixed(StageArgs A) {
    using IO = TileIO32<TZ, MODE, UN_IN>;
    constexpr int NP = FP64_PARTS<TZ>;
    __shared__ __align__(16) float lds[2 * IO::LBUF];
    __shared__ double metric[MODE == MODE_FINAL ? 6 * IO::NT : 1];

    const int slot = tile_of_block(blockIdx.x, A.ntiles * NP, A.xcd_remap);
    const int tile = slot / NP, part = slot % NP;
    if (A.flags && A.flags[tile] != A.want) return;
    const TileRef R = resolve_tile(A, tile);
    if (part_outside<TZ>(R, part)) return; // whole workgroup, before any barrier
    const BlockDesc& b = R.b;
    const int x0 = R.tix * TILE_X, y0 = R.tiy * TILE_Y, z0 = R.tiz * TILE_Z + part * TZ;
    const int tid = threadIdx.x;
    int lx = 0, ly = 0, lz = 0;
    LaneMap<TZ>::cell(tid, lx, ly, lz);
    const int ix = x0 + lx, iy = y0 + ly, iz = z0 + lz;
    const bool active = ix < b.n[0] && iy < b.n[1] && iz < b.n[2];
    const int gi = b.ng + (active ? ix : 0), gj = b.ng + (active ? iy : 0), gk = b.ng + (active ? iz : 0);
    const long cidx = gi + (long)b.nt[0] * (gj + (long)b.nt[1] * gk);

    IO io;
    io.lds = lds;
    io.metric = metric;
    io.in = R.in;
    io.un = R.un;
    io.out = R.out;
    io.stride = b.stride;
    io.cb = 8u * (unsigned)cidx;
    io.ridx = (b.ng + x0) + (long)b.nt[0] * ((b.ng + y0) + (long)b.nt[1] * (b.ng + R.tiz * TILE_Z));
    io.active = active;
    io.ko_on = A.ko_on != 0;
    io.cf = A.cf;
    io.init(tid, lx, ly, lz, b.ng + x0, b.ng + y0, b.ng + z0, b);

    CellSources src{};
    if (HAS_SRC) load_sources(R.src, cidx, src);
    ccz4_cell<float, HAS_SRC, false>(io, io, A.K32, A.P, src);
}

// flags[tile] = 1 where the tile needs the FP64 kernel in the mixed form: its smallest chi
// (interior cells of the stage input) is below chi_min or not finite.
template <int TX, int TY, int TZ>
__global__ __launch_bounds__(TX* TY* TZ) void classify_tiles_kernel(StageArgs A, double chi_min, unsigned char* flags) {
    __shared__ int bad;
    const int tile = blockIdx.x;
    const TileRef R = resolve_tile(A, tile);
    const BlockDesc& b = R.b;
    const int tid = threadIdx.x;
    const int ix = R.tix * TX + tid % TX, iy = R.tiy * TY + (tid / TX) % TY, iz = R.tiz * TZ + tid / (TX * TY);
    if (tid == 0) bad = 0;
    __syncthreads();
    if (ix < b.n[0] && iy < b.n[1] && iz < b.n[2]) {
        const double c =
            R.in[CHI * b.stride + (b.ng + ix) + (long)b.nt[0] * ((b.ng + iy) + (long)b.nt[1] * (b.ng + iz))];
        if (!(c >= chi_min)) bad = 1; // benign race: every writer stores 1
    }
    __syncthreads();
    if (tid == 0) flags[tile] = (unsigned char)bad;
}

template <int MODE, bool HAS_SRC, bool UN_IN>
hipError_t launch_stage_form(const StageArgs& A, int scan_grid, bool large, hipStream_t s) {
    constexpr bool KO = GR_FP64_KO_EXACT != 0;
    if (A.scan) // the flagged tiles, gathered by a small grid
        stage_kernel_scan<TZ_LARGE, MODE, HAS_SRC, KO, UN_IN><<<dim3(scan_grid), dim3(64 * TZ_LARGE), 0, s>>>(A);
    else if (A.ntiles > 0 && large)
        stage_kernel<TZ_LARGE, MODE, HAS_SRC, KO, UN_IN>
            <<<dim3(A.ntiles * FP64_PARTS<TZ_LARGE>), dim3(64 * TZ_LARGE), 0, s>>>(A);
    else if (A.ntiles > 0)
        stage_kernel<TZ_SMALL, MODE, HAS_SRC, KO, UN_IN>
            <<<dim3(A.ntiles * FP64_PARTS<TZ_SMALL>), dim3(64 * TZ_SMALL), 0, s>>>(A);
    return hipGetLastError();
}

template <int MODE, bool HAS_SRC>
hipError_t launch_stage_t(const StageArgs& A, int scan_grid, bool large, hipStream_t s) {
    // the first stage (u^n is the stage input) has an instance of its own: no u^n loads
    if (MODE == MODE_STAGE && A.sel_un == A.sel_in)
        return launch_stage_form<MODE, HAS_SRC, MODE == MODE_STAGE>(A, scan_grid, large, s);
    return launch_stage_form<MODE, HAS_SRC, false>(A, scan_grid, large, s);
}

// ------------------------------------------------------------------------------------
// ghost fill
// ------------------------------------------------------------------------------------
__device__ __forceinline__ double coord(const BlockDesc& b, int d, int idx) {
#pragma clang fp contract(off)
    // GridBlock::x, include/granite/core/grid.hpp:92-94
    return b.lo[d] + ((double)idx - (double)b.ng + 0.5) * b.dx[d];
}

__device__ __forceinline__ double radius(double x, double y, double z) {
#pragma clang fp contract(off)
    return sqrt(x * x + y * y + z * z) + 1e-30;
}

__device__ __forceinline__ double f_inf(int v) {
    return (v == 0 || v == 1 || v == 4 || v == 6 || v == 18) ? 1.0 : 0.0;
}

// a / b from inv = 1 / b, correctly rounded unless tiny_quotient(a, b): the quotient, its exact remainder
// and one correction (Markstein's theorem), with the hardware's rule for zeros, infinities and NaN. Four
// instructions where a division by itself takes eleven.
__device__ __forceinline__ double quotient(double a, double b, double inv) {
    const double q = a * inv;
    return __builtin_amdgcn_div_fixup(fma(fma(-q, b, a), inv, q), b, a);
}
// whether a / b may be subnormal (rounded twice above) or its remainder inexact
__device__ __forceinline__ bool tiny_quotient(double a, double b) {
    return (fabs(a) < 0x1p-900 && a != 0.0) || b > 0x1p100;
}

// Final value of a ghost cell after the reference's three passes: each pass over axis d
// rewrites the ghost layers of d over the full transverse extent from the boundary layer,
// so a cell that is a ghost along a set of axes ends with the chain of 1/r fall-offs from
// its interior anchor, applied in X, Y, Z order at the intermediate positions
// (src/main.cpp:395-483).
__device__ __forceinline__ long ghost_count(const BlockDesc& b) {
    return 2L * b.ng * b.nt[1] * b.nt[0] + (long)b.n[2] * 2 * b.ng * b.nt[0] + (long)b.n[2] * b.n[1] * 2 * b.ng;
}

// ghost cell number t of block b (z slabs, then y rows of interior z, then x columns).
// For the outflow copy (mode 2) only the faces whose bit is set in `faces` are filled
// (bit 2d: low side of axis d, bit 2d+1: high side); the others keep their values, as
// fillGhostZones leaves the faces covered by a parent level to prolongation
// (src/amr/amr.cpp:412-480).
// Fields g, g + G, ... of the cell: the G field groups run as separate workgroups (second
// grid dimension), so a small ghost region still fills the machine.
// Bound by memory: at 192^3 92 us for 290 MB read and 159 MB written, 4.9 TB/s, 56 us of them (6 of
// these the launch's) the x columns, whose anchors cost a 128-byte line per row end and field. With
// the division by a shared reciprocal and each such line written by neighbouring lanes at once:
// 192^3 95 -> 92 us, 128^3 42.4 -> 41.5, the 64 uneven blocks (four launches) 206 -> 200.
template <int G>
__device__ void fill_ghost_cell(const BlockDesc& b, gdouble* u, long t_, int mode, int faces, int g) {
#pragma clang fp contract(off)
    // ghost cells number fewer than 2^29 (the block limit): 32-bit index arithmetic
    const int t = (int)t_;
    const int nt0 = b.nt[0], nt1 = b.nt[1];
    const int nA = 2 * b.ng * nt1 * nt0;
    const int nB = b.n[2] * 2 * b.ng * nt0;
    const int ng = b.ng, g2 = 2 * ng;
    int i, j, k;
    if (t < nA) {
        i = t % nt0;
        const int r = t / nt0;
        j = r % nt1;
        const int kk = r / nt1;
        k = kk < ng ? kk : b.n[2] + kk;
    } else if (t < nA + nB) {
        const int q = t - nA;
        i = q % nt0;
        const int r = q / nt0;
        const int jj = r % g2;
        k = ng + r / g2;
        j = jj < ng ? jj : b.n[1] + jj;
    } else {
        // 2 * ng threads per row: the high ghosts of the row before (of the plane's last row at its
        // first) and the low ghosts of this one, which are neighbours in memory
        const int q = t - nA - nB;
        const int ii = q % g2;
        const int r = q / g2;
        const int row = r % b.n[1];
        k = ng + r / b.n[1];
        const bool hi = ii < ng;
        i = hi ? b.nt[0] - ng + ii : ii - ng;
        j = ng + (hi ? (row > 0 ? row : b.n[1]) - 1 : row);
    }
    const int I[3] = {i, j, k};
    int A[3];
    bool gh[3];
#pragma unroll
    for (int d = 0; d < 3; ++d) {
        gh[d] = I[d] < ng || I[d] >= ng + b.n[d];
        if (mode == 1) {
            int r = (I[d] - ng) % b.n[d];
            if (r < 0) r += b.n[d];
            A[d] = ng + r;
        } else {
            const bool lo = I[d] < ng, hi = I[d] >= ng + b.n[d];
            const bool fill = mode != 2 || (lo && ((faces >> (2 * d)) & 1)) || (hi && ((faces >> (2 * d + 1)) & 1));
            A[d] = (lo && fill) ? ng : ((hi && fill) ? ng + b.n[d] - 1 : I[d]);
        }
    }
    const long dst = I[0] + (long)nt0 * (I[1] + (long)nt1 * I[2]);
    const long src = A[0] + (long)nt0 * (A[1] + (long)nt1 * A[2]);
    // the anchor is never a cell this launch writes, so all loads go out before any store
    constexpr int NF = (NV + G - 1) / G;
    double val[NF];
#pragma unroll
    for (int m = 0; m < NF; ++m) {
        const int v = g + G * m;
        val[m] = v < NV ? u[v * b.stride + src] : 0.0;
    }
    if (mode == 0) {
        // (r_int, r_gh) of each step of the chain: start at the anchor, move one ghost axis
        // at a time in X, Y, Z order
        double Q[3] = {coord(b, 0, A[0]), coord(b, 1, A[1]), coord(b, 2, A[2])};
        bool tiny = false;
#pragma unroll
        for (int d = 0; d < 3; ++d) {
            if (!gh[d]) continue;
            const double rin = radius(Q[0], Q[1], Q[2]);
            Q[d] = coord(b, d, I[d]);
            const double rgh = radius(Q[0], Q[1], Q[2]);
            const double inv = 1.0 / rgh;
#pragma unroll
            for (int m = 0; m < NF; ++m) {
                const double fi = f_inf(g + G * m), a = (val[m] - fi) * rin;
                tiny = tiny || tiny_quotient(a, rgh);
                val[m] = fi + quotient(a, rgh, inv);
            }
        }
        // once more by divisions (same launch: the anchor still holds its value)
        if (tiny) {
#pragma unroll 1
            for (int v = g; v < NV; v += G) {
                const double fi = f_inf(v);
                double x = u[v * b.stride + src];
                double P[3] = {coord(b, 0, A[0]), coord(b, 1, A[1]), coord(b, 2, A[2])};
#pragma unroll
                for (int d = 0; d < 3; ++d) {
                    if (!gh[d]) continue;
                    const double rin = radius(P[0], P[1], P[2]);
                    P[d] = coord(b, d, I[d]);
                    x = fi + ((x - fi) * rin) / radius(P[0], P[1], P[2]);
                }
                u[v * b.stride + dst] = x;
            }
            return;
        }
    }
#pragma unroll
    for (int m = 0; m < NF; ++m) {
        const int v = g + G * m;
        if (v < NV) u[v * b.stride + dst] = val[m];
    }
}

template <int G>
__global__ __launch_bounds__(GHOST_WG) void fill_ghosts_kernel(BlockDesc b, double* u, int mode, int faces) {
    const long t = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= ghost_count(b)) return;
    fill_ghost_cell<G>(b, (gdouble*)u, t, mode, faces, blockIdx.y);
}

// ------------------------------------------------------------------------------------
// AMR transfer between a coarse and a fine block (one block per level)
// ------------------------------------------------------------------------------------

// Per-axis part of the trilinear coarse -> fine stencil, with the reference's index rounding
// and clamping (src/amr/amr.cpp:484-564): entry e < f.nt[0] is x index e, then the y indices,
// then the z indices. The stencil is separable, so the prolongation itself reads three entries
// per fine cell instead of repeating three divisions for every field group.
__global__ void prolong_axes_kernel(BlockDesc c, BlockDesc f, ProlongAxis* __restrict__ tab) {
#pragma clang fp contract(off)
    const int t = (int)(blockIdx.x * blockDim.x + threadIdx.x);
    if (t >= f.nt[0] + f.nt[1] + f.nt[2]) return;
    const int d = t < f.nt[0] ? 0 : (t < f.nt[0] + f.nt[1] ? 1 : 2);
    const int i = t - (d > 0 ? f.nt[0] : 0) - (d > 1 ? f.nt[1] : 0);
    const double x = coord(f, d, i);
    const double cf = (x - coord(c, d, c.ng)) / c.dx[d] + (double)c.ng;
    int ci = (int)round(cf);
    ci = ci < 0 ? 0 : (ci > c.nt[d] - 1 ? c.nt[d] - 1 : ci);
    const double fr = cf - (double)ci;
    int cj = ci + (fr >= 0.0 ? 1 : -1);
    cj = cj > c.nt[d] - 1 ? c.nt[d] - 1 : cj;
    cj = cj < 0 ? 0 : cj;
    tab[t] = ProlongAxis{ci, cj, fabs(fr)};
}

// Trilinear coarse -> fine into every fine cell, ghosts included (src/amr/amr.cpp:484-564),
// from the per-axis stencil table of this (coarse, fine) pair. One workgroup per fine tile of
// PT_X x PT_Y x PT_Z cells (a thread per (x, y) column of PT_Z cells): per field, the coarse
// box the tile's stencils reach is staged in LDS (double-buffered, one barrier per field) and
// the eight taps are read from there, so the coarse field is read from memory once per tile
// instead of eight times per fine cell. A tile whose stencils reach beyond the box capacity
// (a fine block not at half the parent's spacing) reads the taps from memory directly.
#ifndef GR_PT_X
#define GR_PT_X 32
#endif
#ifndef GR_PT_Y
#define GR_PT_Y 8
#endif
#ifndef GR_PT_Z
#define GR_PT_Z 8
#endif
#ifndef GR_PROLONG_PREFETCH
#define GR_PROLONG_PREFETCH 1
#endif
constexpr int PT_X = GR_PT_X, PT_Y = GR_PT_Y, PT_Z = GR_PT_Z, PT_N = PT_X * PT_Y;
constexpr int PB_X = PT_X / 2 + 2, PB_Y = PT_Y / 2 + 2, PB_Z = PT_Z / 2 + 2, PB_N = PB_X * PB_Y * PB_Z;
constexpr int PB_PER_THREAD = (PB_N + PT_N - 1) / PT_N;

__global__ __launch_bounds__(PT_N) void prolong_kernel(BlockDesc c, const double* __restrict__ cu, BlockDesc f,
                                                             double* __restrict__ fu,
                                                             const ProlongAxis* __restrict__ tab, int ntx, int nty) {
#pragma clang fp contract(off)
    __shared__ double box[2][PB_N];
    __shared__ int lim[6]; // per axis: lowest, highest coarse index any stencil of the tile reads
    const int tile = blockIdx.x;
    const int i0 = (tile % ntx) * PT_X, j0 = ((tile / ntx) % nty) * PT_Y, k0 = (tile / (ntx * nty)) * PT_Z;
    const int tid = threadIdx.x;
    if (tid < 6) lim[tid] = (tid & 1) ? -1 : 0x7fffffff;
    __syncthreads();
    if (tid < PT_X + PT_Y + PT_Z) {
        const int d = tid < PT_X ? 0 : (tid < PT_X + PT_Y ? 1 : 2);
        const int e = d == 0 ? i0 + tid : (d == 1 ? j0 + tid - PT_X : k0 + tid - PT_X - PT_Y);
        if (e < f.nt[d]) {
            const ProlongAxis A = tab[(d > 0 ? f.nt[0] : 0) + (d > 1 ? f.nt[1] : 0) + e];
            atomicMin(&lim[2 * d], A.c0 < A.c1 ? A.c0 : A.c1);
            atomicMax(&lim[2 * d + 1], A.c0 > A.c1 ? A.c0 : A.c1);
        }
    }
    __syncthreads();
    const int bx = lim[0], by = lim[2], bz = lim[4];
    const int ex = lim[1] - bx + 1, ey = lim[3] - by + 1, ez = lim[5] - bz + 1;
    const bool staged = ex <= PB_X && ey <= PB_Y && ez <= PB_Z; // uniform over the workgroup

    const int i = i0 + tid % PT_X, j = j0 + tid / PT_X;
    const bool live = i < f.nt[0] && j < f.nt[1];
    const ProlongAxis X = tab[live ? i : 0], Y = tab[f.nt[0] + (live ? j : 0)];
    // leading (x, y) factors of the reference's weight products, (wx * wy) * wz
    const double p00 = (1 - X.ax) * (1 - Y.ax), p10 = X.ax * (1 - Y.ax), p01 = (1 - X.ax) * Y.ax, p11 = X.ax * Y.ax;
    const ProlongAxis* Ztab = tab + f.nt[0] + f.nt[1];
    const int kn = f.nt[2] - k0 < PT_Z ? f.nt[2] - k0 : PT_Z;
    const int fplane = f.nt[0] * f.nt[1], fcol = i + f.nt[0] * j;
    if (staged) {
        const int q00 = (X.c0 - bx) + PB_X * (Y.c0 - by), q10 = (X.c1 - bx) + PB_X * (Y.c0 - by),
                  q01 = (X.c0 - bx) + PB_X * (Y.c1 - by), q11 = (X.c1 - bx) + PB_X * (Y.c1 - by);
        // coarse offsets of this thread's box elements (-1: none)
        int src[PB_PER_THREAD];
#pragma unroll
        for (int r = 0; r < PB_PER_THREAD; ++r) {
            const int e = tid + r * PT_N;
            const int a = e % PB_X, b = (e / PB_X) % PB_Y, z = e / (PB_X * PB_Y);
            src[r] = (e < PB_N && a < ex && b < ey && z < ez) ? (bx + a) + c.nt[0] * ((by + b) + c.nt[1] * (bz + z)) : -1;
        }
        double next[PB_PER_THREAD];
#if GR_PROLONG_PREFETCH
#pragma unroll
        for (int r = 0; r < PB_PER_THREAD; ++r)
            if (src[r] >= 0) next[r] = cu[(long)blockIdx.y * c.stride + src[r]];
#endif
        int buf = 0;
        for (int v = blockIdx.y; v < NV; v += gridDim.y) {
#if GR_PROLONG_PREFETCH
            // stage field v, then start loading field v + gridDim.y
#pragma unroll
            for (int r = 0; r < PB_PER_THREAD; ++r)
                if (src[r] >= 0) box[buf][tid + r * PT_N] = next[r];
            if (v + (int)gridDim.y < NV) {
                const double* Un = cu + (long)(v + gridDim.y) * c.stride;
#pragma unroll
                for (int r = 0; r < PB_PER_THREAD; ++r)
                    if (src[r] >= 0) next[r] = Un[src[r]];
            }
#else
            const double* U = cu + (long)v * c.stride;
#pragma unroll
            for (int r = 0; r < PB_PER_THREAD; ++r)
                if (src[r] >= 0) next[r] = U[src[r]];
#pragma unroll
            for (int r = 0; r < PB_PER_THREAD; ++r)
                if (src[r] >= 0) box[buf][tid + r * PT_N] = next[r];
#endif
            __syncthreads();
            if (live) {
                const double* B = box[buf];
                double* out = fu + (long)v * f.stride + fcol;
                for (int kk = 0; kk < kn; ++kk) {
                    const ProlongAxis Z = Ztab[k0 + kk];
                    const int z0 = PB_X * PB_Y * (Z.c0 - bz), z1 = PB_X * PB_Y * (Z.c1 - bz);
                    const double az = Z.ax, bz1 = 1 - Z.ax;
                    // the reference's term order: 000, 100, 010, 001, 110, 101, 011, 111
                    out[(long)fplane * (k0 + kk)] = p00 * bz1 * B[q00 + z0] + p10 * bz1 * B[q10 + z0] +
                        p01 * bz1 * B[q01 + z0] + p00 * az * B[q00 + z1] + p11 * bz1 * B[q11 + z0] +
                        p10 * az * B[q10 + z1] + p01 * az * B[q01 + z1] + p11 * az * B[q11 + z1];
                }
            }
            buf ^= 1;
        }
    } else if (live) {
        const int r00 = X.c0 + c.nt[0] * Y.c0, r10 = X.c1 + c.nt[0] * Y.c0, r01 = X.c0 + c.nt[0] * Y.c1,
                  r11 = X.c1 + c.nt[0] * Y.c1;
        const int cplane = c.nt[0] * c.nt[1];
        for (int v = blockIdx.y; v < NV; v += gridDim.y) {
            const double* U = cu + (long)v * c.stride;
            double* out = fu + (long)v * f.stride + fcol;
            for (int kk = 0; kk < kn; ++kk) {
                const ProlongAxis Z = Ztab[k0 + kk];
                const int z0 = cplane * Z.c0, z1 = cplane * Z.c1;
                const double az = Z.ax, bz1 = 1 - Z.ax;
                out[(long)fplane * (k0 + kk)] = p00 * bz1 * U[r00 + z0] + p10 * bz1 * U[r10 + z0] +
                    p01 * bz1 * U[r01 + z0] + p00 * az * U[r00 + z1] + p11 * bz1 * U[r11 + z0] +
                    p10 * az * U[r10 + z1] + p01 * az * U[r01 + z1] + p11 * az * U[r11 + z1];
            }
        }
    }
}

// 2x2x2 average of fine cells into the covered coarse interior cells
// (src/amr/amr.cpp:566-626, refinement ratio 2).
__global__ void restrict_kernel(BlockDesc f, const double* __restrict__ fu, BlockDesc c, double* __restrict__ cu) {
#pragma clang fp contract(off)
    const int t = (int)(blockIdx.x * blockDim.x + threadIdx.x); // interior cells < 2^29
    const int ncell = c.n[0] * c.n[1] * c.n[2];
    if (t >= ncell) return;
    const int C[3] = {c.ng + t % c.n[0], c.ng + (t / c.n[0]) % c.n[1], c.ng + t / (c.n[0] * c.n[1])};
    int b[3];
#pragma unroll
    for (int d = 0; d < 3; ++d) {
        b[d] = (int)round((coord(c, d, C[d]) - coord(f, d, 0)) / f.dx[d]) - 1;
        if (!(b[d] >= f.ng && b[d] + 2 <= f.ng + f.n[d] + f.ng)) return;
    }
    const long dst = C[0] + (long)c.nt[0] * (C[1] + (long)c.nt[1] * C[2]);
    for (int v = blockIdx.y; v < NV; v += gridDim.y) {
        const double* F = fu + v * f.stride;
        double s = 0.0;
        for (int rk = 0; rk < 2; ++rk)
            for (int rj = 0; rj < 2; ++rj)
                for (int ri = 0; ri < 2; ++ri) s += F[(b[0] + ri) + (long)f.nt[0] * ((b[1] + rj) + (long)f.nt[1] * (b[2] + rk))];
        cu[v * c.stride + dst] = s / 8;
    }
}

// interior cells of `r`, field by field, without the ghosts between them
__global__ void pack_interior_kernel(BlockDesc b, const double* __restrict__ r, double* __restrict__ out) {
    const int t = (int)(blockIdx.x * blockDim.x + threadIdx.x); // interior cells < 2^29
    const int ncell = b.n[0] * b.n[1] * b.n[2];
    if (t >= ncell) return;
    const int i = t % b.n[0], q = t / b.n[0], j = q % b.n[1], k = q / b.n[1];
    const long src = (b.ng + i) + (long)b.nt[0] * ((b.ng + j) + (long)b.nt[1] * (b.ng + k));
    const int v = blockIdx.y;
    out[(long)v * ncell + t] = r[v * b.stride + src];
}

// every ghost cell of buffer `sel` of every block of a table; ofs[i] = first ghost cell of
// block i (nblocks + 1 entries)
template <int G>
__global__ __launch_bounds__(GHOST_WG) void fill_ghosts_batch_kernel(const BatchBlock* __restrict__ table, const int* __restrict__ wg_block,
                                         int sel, int mode) {
    const BatchBlock& B = table[wg_block[blockIdx.x]]; // one block per workgroup
    const long t = (long)(blockIdx.x - B.ghost_wg0) * GHOST_WG + threadIdx.x;
    const BlockDesc b = B.b; // (not read again behind the stores)
    if (t >= ghost_count(b)) return;
    fill_ghost_cell<G>(b, (gdouble*)B.buf[sel], t, mode, 0x3f, blockIdx.y);
}

// ------------------------------------------------------------------------------------
// Kreiss-Oliger only (applyDissipation), global-memory stencils, reference order
// ------------------------------------------------------------------------------------
__global__ void dissipation_kernel(BlockDesc b, const double* __restrict__ u, double* rhs, Stencil<double> K) {
#pragma clang fp contract(off)
    const long t = (long)blockIdx.x * blockDim.x + threadIdx.x;
    const long ncell = (long)b.n[0] * b.n[1] * b.n[2];
    if (t >= ncell) return;
    const int i = b.ng + (int)(t % b.n[0]);
    const int j = b.ng + (int)((t / b.n[0]) % b.n[1]);
    const int k = b.ng + (int)(t / ((long)b.n[0] * b.n[1]));
    const long c = i + (long)b.nt[0] * (j + (long)b.nt[1] * k);
    const long st[3] = {1, b.nt[0], (long)b.nt[0] * b.nt[1]};
    for (int v = 0; v < NV; ++v) {
        const double* f = u + v * b.stride + c;
        double acc = 0.0;
        for (int d = 0; d < 3; ++d)
            acc = ko_axis_ordered(d == 0, acc, K.kw[d], f[-3 * st[d]], f[-2 * st[d]], f[-st[d]], f[0], f[st[d]], f[2 * st[d]],
                                  f[3 * st[d]]);
        rhs[v * b.stride + c] += acc;
    }
}

// ------------------------------------------------------------------------------------
// constraint monitor (src/spacetime/ccz4.cpp:941-1159)
// ------------------------------------------------------------------------------------

// 4th-order first and (D2) second derivatives of one staged field
template <bool D2, class ST>
__device__ __forceinline__ void field_derivs(const double* s, const Stencil<double>& K, const ST& st, double d1[3],
                                             double dd[6]) {
    const double c = st.centre(s);
#pragma unroll
    for (int d = 0; d < 3; ++d) {
        const double m1 = st.at(s, d, -1), p1 = st.at(s, d, 1), m2 = st.at(s, d, -2), p2 = st.at(s, d, 2);
        d1[d] = K.ih[d] * (-p2 + 8.0 * p1 - 8.0 * m1 + m2);
        if (D2) dd[sym(d, d)] = K.ih2[d] * (-p2 + 16.0 * p1 - 30.0 * c + 16.0 * m1 - m2);
        pin(d1[d]);
    }
    if (D2) {
        auto mixed = [&](int a, int b) {
            return st.edge(s, a, b, 1, 1) - st.edge(s, a, b, 1, -1) - st.edge(s, a, b, -1, 1) + st.edge(s, a, b, -1, -1);
        };
        dd[1] = K.ihh[0] * mixed(0, 1);
        dd[2] = K.ihh[1] * mixed(0, 2);
        dd[4] = K.ihh[2] * mixed(1, 2);
#pragma unroll
        for (int q = 0; q < 6; ++q) pin(dd[q]);
    }
}

// H of one cell and, with MOM, M_i into mom[0..2]; the fields come staged one by one, each folded
// into the Ricci tensor (or M_i) as it arrives
template <bool MOM, class Stager>
__device__ __forceinline__ double constraint_cell(Stager& S, const Stencil<double>& K, double mom[3]) {
    const double chi = S.centre(CHI), Ktr = S.centre(KTR);
    double gt[6], At[6], Gh[3];
#pragma unroll
    for (int a = 0; a < 6; ++a) {
        gt[a] = S.centre(GXX + a);
        At[a] = S.centre(AXX + a);
    }
#pragma unroll
    for (int a = 0; a < 3; ++a) Gh[a] = S.centre(GHX + a);
    const double det = gt[0] * (gt[3] * gt[5] - gt[4] * gt[4]) - gt[1] * (gt[1] * gt[5] - gt[4] * gt[2]) +
        gt[2] * (gt[1] * gt[4] - gt[3] * gt[2]);
    const double idet = 1.0 / (det + 1.0e-30);
    const double gu[6] = {(gt[3] * gt[5] - gt[4] * gt[4]) * idet, (gt[2] * gt[4] - gt[1] * gt[5]) * idet,
                          (gt[1] * gt[4] - gt[2] * gt[3]) * idet, (gt[0] * gt[5] - gt[2] * gt[2]) * idet,
                          (gt[1] * gt[2] - gt[0] * gt[4]) * idet, (gt[0] * gt[3] - gt[1] * gt[1]) * idet};
    double AA = 0.0;
    {
        double Au[3][3];
#pragma unroll
        for (int a = 0; a < 3; ++a)
#pragma unroll
            for (int c = 0; c < 3; ++c)
                Au[a][c] = gu[sym(a, 0)] * At[sym(0, c)] + gu[sym(a, 1)] * At[sym(1, c)] + gu[sym(a, 2)] * At[sym(2, c)];
#pragma unroll
        for (int a = 0; a < 3; ++a)
#pragma unroll
            for (int c = 0; c < 3; ++c) AA += Au[a][c] * Au[c][a];
        pin(AA);
    }

    // metric: Ricci term -1/2 g^lm d_l d_m gt_ij, first derivatives kept for the Christoffels
    double dgt[6][3], dd[6], Rt[6];
#pragma unroll
    for (int p = 0; p < 6; ++p) {
        field_derivs<true>(S.field(GXX + p), K, S.strides(), dgt[p], dd);
        double r = 0.0;
#pragma unroll
        for (int q = 0; q < 6; ++q) r += ((q == 0 || q == 3 || q == 5) ? -0.5 : -1.0) * gu[q] * dd[q];
        Rt[p] = r;
        pin(Rt[p]);
    }
    double chr[3][6];
#pragma unroll
    for (int q = 0; q < 3; ++q)
#pragma unroll
        for (int p = 0; p < 6; ++p) {
            const int a = sym_a(p), c = sym_b(p);
            double v = 0.0;
#pragma unroll
            for (int m = 0; m < 3; ++m) v += gu[sym(q, m)] * (dgt[sym(m, a)][c] + dgt[sym(m, c)][a] - dgt[p][m]);
            chr[q][p] = 0.5 * v;
            pin(chr[q][p]);
        }

    // chi: the conformal-factor part of the Ricci tensor
    double dchi[3];
    field_derivs<true>(S.field(CHI), K, S.strides(), dchi, dd);
    {
        double D[6], lapchi = 0.0, gradchi2 = 0.0;
#pragma unroll
        for (int p = 0; p < 6; ++p) {
            const int l = sym_a(p), m = sym_b(p);
            const double f = (l == m) ? 1.0 : 2.0;
            D[p] = dd[p] - chr[0][p] * dchi[0] - chr[1][p] * dchi[1] - chr[2][p] * dchi[2];
            lapchi += f * gu[p] * D[p];
            gradchi2 += f * gu[p] * dchi[l] * dchi[m];
        }
#pragma unroll
        for (int p = 0; p < 6; ++p)
            Rt[p] += (0.5 / (chi + 1e-30)) * (D[p] + gt[p] * lapchi) -
                (0.25 / ((chi * chi) + 1e-30)) * (dchi[sym_a(p)] * dchi[sym_b(p)] - 3.0 * gt[p] * gradchi2);
    }

    // products of Christoffel symbols, factored per k as in ccz4_cell
#pragma unroll
    for (int k = 0; k < 3; ++k) {
        double Gk[6], Gd = 0.0;
#pragma unroll
        for (int p = 0; p < 6; ++p) {
            Gk[p] = gt[sym(k, 0)] * chr[0][p] + gt[sym(k, 1)] * chr[1][p] + gt[sym(k, 2)] * chr[2][p];
            Gd += ((p == 0 || p == 3 || p == 5) ? 1.0 : 2.0) * gu[p] * chr[k][p];
        }
#pragma unroll
        for (int p = 0; p < 6; ++p) Rt[p] += (Gh[k] - Gd) * Gk[p];
#pragma unroll
        for (int l = 0; l < 3; ++l) {
            double H[3];
#pragma unroll
            for (int j = 0; j < 3; ++j)
                H[j] = gu[sym(l, 0)] * Gk[sym(j, 0)] + gu[sym(l, 1)] * Gk[sym(j, 1)] + gu[sym(l, 2)] * Gk[sym(j, 2)];
#pragma unroll
            for (int p = 0; p < 6; ++p) {
                const int a = sym_a(p), b = sym_b(p);
                Rt[p] += chr[k][sym(l, a)] * H[b] + chr[k][sym(l, b)] * H[a];
            }
        }
    }
#pragma unroll
    for (int p = 0; p < 6; ++p) pin(Rt[p]);

    double d1[3];
#pragma unroll
    for (int q = 0; q < 3; ++q) {
        field_derivs<false>(S.field(GHX + q), K, S.strides(), d1, dd);
#pragma unroll
        for (int p = 0; p < 6; ++p) {
            const int a = sym_a(p), b = sym_b(p);
            Rt[p] += 0.5 * (gt[sym(q, a)] * d1[b] + gt[sym(q, b)] * d1[a]);
            pin(Rt[p]);
        }
    }
    double Rs = 0.0;
#pragma unroll
    for (int p = 0; p < 6; ++p) Rs += ((p == 0 || p == 3 || p == 5) ? 1.0 : 2.0) * gu[p] * Rt[p];
    Rs *= chi;
    double H = Rs + (2.0 / 3.0) * Ktr * Ktr - AA;
    pin(H);
    if (!MOM) return H;

    // M_a = g^cq (d_c A_qa - chr^m_cq A_ma - chr^m_ca A_qm - 3 / (2 chi) A_ac d_q chi) - 2/3 d_a K:
    // the terms of the cell itself, then K's and A~'s derivatives as the fields arrive
    const double c3 = 3.0 / (2.0 * chi + 1e-30);
#pragma unroll
    for (int a = 0; a < 3; ++a) {
        double M = 0.0;
#pragma unroll
        for (int c = 0; c < 3; ++c)
#pragma unroll
            for (int q = 0; q < 3; ++q) {
                double DA = -c3 * At[sym(a, c)] * dchi[q];
#pragma unroll
                for (int m = 0; m < 3; ++m) DA -= chr[m][sym(c, q)] * At[sym(m, a)] + chr[m][sym(c, a)] * At[sym(q, m)];
                M += gu[sym(c, q)] * DA;
            }
        mom[a] = M;
        pin(mom[a]);
    }
    field_derivs<false>(S.field(KTR), K, S.strides(), d1, dd);
#pragma unroll
    for (int a = 0; a < 3; ++a) mom[a] -= (2.0 / 3.0) * d1[a];
#pragma unroll
    for (int p = 0; p < 6; ++p) {
        const int i = sym_a(p), j = sym_b(p);
        field_derivs<false>(S.field(AXX + p), K, S.strides(), d1, dd);
        mom[j] += gu[sym(0, i)] * d1[0] + gu[sym(1, i)] * d1[1] + gu[sym(2, i)] * d1[2];
        if (i != j) mom[i] += gu[sym(0, j)] * d1[0] + gu[sym(1, j)] * d1[1] + gu[sym(2, j)] * d1[2];
#pragma unroll
        for (int a = 0; a < 3; ++a) pin(mom[a]);
    }
    return H;
}

__device__ __forceinline__ double part_sum(double v, double* sh, int n) {
    sh[threadIdx.x] = v;
    __syncthreads();
    for (int o = n / 2; o > 0; o >>= 1) {
        if ((int)threadIdx.x < o) sh[threadIdx.x] += sh[threadIdx.x + o];
        __syncthreads();
    }
    const double s = sh[0];
    __syncthreads();
    return s;
}

// H (and, with MOM, M_i) over one block, in the stage kernel's parts and staging: each workgroup
// takes `per` consecutive parts. ham / mom (may be null): the values per interior cell, mom cell-major;
// partial (may be null): per workgroup the sum of H^2 and, gridDim.x further on, of |M|^2. 183 us for H
// and M_i of 10^6 cells (132x96x96, 17 fields of the state at 0.8 TB/s: bound as the stage kernel is,
// by the cache lines of the halo and the arithmetic); with the stencils read from memory by every
// cell and 1.9 KB of scratch per lane it took 1463 us.
template <bool MOM>
__global__ __launch_bounds__(64 * TZ_LARGE, 2) void constraints_kernel(StageArgs A, double* ham, double* mom,
                                                                       double* partial, int per) {
    constexpr int TZ = TZ_LARGE, NT = 64 * TZ;
    using IO = TileIODma<TZ, MODE_RHS, false, MonitorOrder<MOM>>;
    __shared__ __align__(16) double lds[IO::LDS_DOUBLES];
    const int tid = threadIdx.x;
    const int nparts = A.ntiles * FP64_PARTS<TZ>;
    const int first = tile_of_block(blockIdx.x, gridDim.x, A.xcd_remap) * per;
    const int last = first + per < nparts ? first + per : nparts;
    int lx = 0, ly = 0, lz = 0;
    LaneMap<TZ>::cell(tid, lx, ly, lz);
    double h2 = 0.0, m2 = 0.0;
    for (int part = first; part < last; ++part) {
        const TileRef R = resolve_tile(A, part / FP64_PARTS<TZ>);
        const BlockDesc& b = R.b;
        const int x0 = R.tix * TILE_X, y0 = R.tiy * TILE_Y, z0 = R.tiz * TILE_Z + part % FP64_PARTS<TZ> * TZ;
        if (z0 >= b.n[2]) continue; // uniform over the workgroup
        const int ix = x0 + lx, iy = y0 + ly, iz = z0 + lz;
        const bool active = ix < b.n[0] && iy < b.n[1] && iz < b.n[2];
        const int gi = b.ng + (active ? ix : 0), gj = b.ng + (active ? iy : 0), gk = b.ng + (active ? iz : 0);
        const long cidx = gi + (long)b.nt[0] * (gj + (long)b.nt[1] * gk);
        IO io;
        io.lds = lds;
        io.in = R.in;
        io.stride = b.stride;
        io.cb = 8u * (unsigned)cidx;
        io.place(lx, ly, lz);
        io.init(tid, b.ng + x0, b.ng + y0, b.ng + z0, b);
        double M[3] = {0.0, 0.0, 0.0};
        const double H = constraint_cell<MOM>(io, A.K, M);
        if (active) {
            h2 += H * H;
            if (MOM) m2 += M[0] * M[0] + M[1] * M[1] + M[2] * M[2];
            if (ham) ham[cidx] = H;
            if (MOM && mom)
#pragma unroll
                for (int a = 0; a < 3; ++a) mom[3 * cidx + a] = M[a];
        }
        __syncthreads(); // the next part reuses the buffers
    }
    if (!partial) return;
    const double sh2 = part_sum(h2, lds, NT);
    const double sm2 = MOM ? part_sum(m2, lds, NT) : 0.0;
    if (tid == 0) {
        partial[blockIdx.x] = sh2;
        if (MOM) partial[gridDim.x + blockIdx.x] = sm2;
    }
}

__global__ void zero_kernel(double* p, long n) {
    for (long t = (long)blockIdx.x * blockDim.x + threadIdx.x; t < n; t += (long)gridDim.x * blockDim.x) p[t] = 0.0;
}

// ------------------------------------------------------------------------------------
// initial data and noise
// ------------------------------------------------------------------------------------
__global__ void init_bl_kernel(BlockDesc b, double* u, int nbh, const double* mass, const double* pos) {
#pragma clang fp contract(off)
    const long t = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= b.stride) return;
    const int i = (int)(t % b.nt[0]);
    const int j = (int)((t / b.nt[0]) % b.nt[1]);
    const int k = (int)(t / ((long)b.nt[0] * b.nt[1]));
    const double x = coord(b, 0, i), y = coord(b, 1, j), z = coord(b, 2, k);
    // flat background (src/spacetime/ccz4.cpp:1165-1188) then the BL conformal factor
    // (src/initial_data/initial_data.cpp:79-158)
    for (int v = 0; v < NV; ++v) u[v * b.stride + t] = 0.0;
    u[(GXX + 0) * b.stride + t] = 1.0;
    u[(GXX + 3) * b.stride + t] = 1.0;
    u[(GXX + 5) * b.stride + t] = 1.0;
    double psi = 1.0;
    for (int h = 0; h < nbh; ++h) {
        const double ax = x - pos[3 * h], ay = y - pos[3 * h + 1], az = z - pos[3 * h + 2];
        const double r = sqrt(ax * ax + ay * ay + az * az + 1.0e-30);
        psi += mass[h] / (2.0 * r);
    }
    const double p2 = psi * psi;
    const double chi = 1.0 / (p2 * p2);
    u[CHI * b.stride + t] = chi;
    u[ALPHA * b.stride + t] = sqrt(chi);
    double dp[3] = {0.0, 0.0, 0.0};
    for (int h = 0; h < nbh; ++h) {
        const double rx = x - pos[3 * h], ry = y - pos[3 * h + 1], rz = z - pos[3 * h + 2];
        const double r2 = rx * rx + ry * ry + rz * rz + 1.0e-20;
        const double r3 = r2 * sqrt(r2);
        const double c = -mass[h] / (2.0 * r3);
        dp[0] += c * rx;
        dp[1] += c * ry;
        dp[2] += c * rz;
    }
    const double gf = 8.0 / (3.0 * psi);
    for (int a = 0; a < 3; ++a) u[(GHX + a) * b.stride + t] = gf * dp[a];
}

__device__ __forceinline__ uint64_t sm64(uint64_t s) {
    s += 0x9E3779B97F4A7C15ull;
    s = (s ^ (s >> 30)) * 0xBF58476D1CE4E5B9ull;
    s = (s ^ (s >> 27)) * 0x94D049BB133111EBull;
    return s ^ (s >> 31);
}

__global__ void add_noise_kernel(BlockDesc b, double* u, uint64_t seed, double amp, unsigned mask) {
    const long t = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= b.stride) return;
    for (int v = 0; v < NV; ++v) {
        if (!((mask >> v) & 1u)) continue;
        const uint64_t q = (uint64_t)v * (uint64_t)b.stride + (uint64_t)t;
        const uint64_t z1 = sm64(seed + (2 * q) * 0x9E3779B97F4A7C15ull);
        const uint64_t z2 = sm64(seed + (2 * q + 1) * 0x9E3779B97F4A7C15ull);
        const double u1 = ((double)(z1 >> 11) + 0.5) * (1.0 / 9007199254740992.0);
        const double u2 = (double)(z2 >> 11) * (1.0 / 9007199254740992.0);
        u[v * b.stride + t] += amp * (sqrt(-2.0 * log(u1)) * cos(2.0 * PI * u2));
    }
}

// ------------------------------------------------------------------------------------
// reductions (fixed order: per-workgroup tree, then one workgroup over the partials)
// ------------------------------------------------------------------------------------
constexpr int RED_T = 256;

__device__ __forceinline__ double block_sum(double v, double* sh) {
    sh[threadIdx.x] = v;
    __syncthreads();
    for (int o = RED_T / 2; o > 0; o >>= 1) {
        if ((int)threadIdx.x < o) sh[threadIdx.x] += sh[threadIdx.x + o];
        __syncthreads();
    }
    return sh[0];
}

__global__ __launch_bounds__(RED_T) void nonfinite_kernel(BlockDesc b, const double* u, double* partial, long per) {
    __shared__ double sh[RED_T];
    const long ncell = (long)b.n[0] * b.n[1] * b.n[2];
    const long beg = (long)blockIdx.x * per;
    const long end = beg + per < ncell ? beg + per : ncell;
    double acc = 0.0;
    for (long t = beg + threadIdx.x; t < end; t += RED_T) {
        const int i = b.ng + (int)(t % b.n[0]);
        const int j = b.ng + (int)((t / b.n[0]) % b.n[1]);
        const int k = b.ng + (int)(t / ((long)b.n[0] * b.n[1]));
        const long c = i + (long)b.nt[0] * (j + (long)b.nt[1] * k);
        for (int v = 0; v < NV; ++v) acc += __builtin_isfinite(u[v * b.stride + c]) ? 0.0 : 1.0;
    }
    const double s = block_sum(acc, sh);
    if (threadIdx.x == 0) partial[blockIdx.x] = s;
}

// out[g] = sum of the n partials of group g (one workgroup per group)
__global__ __launch_bounds__(RED_T) void sum_partials_kernel(const double* partial, int n, double* out) {
    __shared__ double sh[RED_T];
    double acc = 0.0;
    for (int t = threadIdx.x; t < n; t += RED_T) acc += partial[(long)blockIdx.x * n + t];
    const double s = block_sum(acc, sh);
    if (threadIdx.x == 0) out[blockIdx.x] = s;
}

// First non-finite interior value in the order of the reference's NaN scan
// (src/main.cpp:1192-1214: field v, then k, j, i over the interior). Position q of field v
// at interior cell (i', j', k') is v * ncell + (k' * n1 + j') * n0 + i'; each workgroup
// takes the contiguous range [blockIdx.x * per, ...) of positions (consecutive threads on
// consecutive x: coalesced) and writes the smallest non-finite position in it, or ~0.
__global__ __launch_bounds__(RED_T) void first_nonfinite_kernel(BlockDesc b, const double* u,
                                                                unsigned long long* partial, long per) {
    __shared__ unsigned long long sh[RED_T];
    const long ncell = (long)b.n[0] * b.n[1] * b.n[2];
    const long total = NV * ncell;
    const long beg = (long)blockIdx.x * per;
    const long end = beg + per < total ? beg + per : total;
    unsigned long long best = ~0ull;
    for (long q = beg + threadIdx.x; q < end; q += RED_T) {
        const int v = (int)(q / ncell);
        const long t = q - v * ncell;
        const int i = b.ng + (int)(t % b.n[0]);
        const int j = b.ng + (int)((t / b.n[0]) % b.n[1]);
        const int k = b.ng + (int)(t / ((long)b.n[0] * b.n[1]));
        const double x = u[v * b.stride + i + (long)b.nt[0] * (j + (long)b.nt[1] * k)];
        if (!__builtin_isfinite(x)) {
            best = (unsigned long long)q; // the thread's positions rise: the first is its smallest
            break;
        }
    }
    sh[threadIdx.x] = best;
    __syncthreads();
    for (int o = RED_T / 2; o > 0; o >>= 1) {
        if ((int)threadIdx.x < o && sh[threadIdx.x + o] < sh[threadIdx.x]) sh[threadIdx.x] = sh[threadIdx.x + o];
        __syncthreads();
    }
    if (threadIdx.x == 0) partial[blockIdx.x] = sh[0];
}

__global__ __launch_bounds__(RED_T) void min_partials_kernel(const unsigned long long* partial, int n,
                                                             unsigned long long* out) {
    __shared__ unsigned long long sh[RED_T];
    unsigned long long m = ~0ull;
    for (int t = threadIdx.x; t < n; t += RED_T) m = partial[t] < m ? partial[t] : m;
    sh[threadIdx.x] = m;
    __syncthreads();
    for (int o = RED_T / 2; o > 0; o >>= 1) {
        if ((int)threadIdx.x < o && sh[threadIdx.x + o] < sh[threadIdx.x]) sh[threadIdx.x] = sh[threadIdx.x + o];
        __syncthreads();
    }
    if (threadIdx.x == 0) out[0] = sh[0];
}

// the reference's max_adv_cfl = std::max(max_adv_cfl, local) keeps the running value when
// local is NaN (the comparison is false), so NaN never enters the maximum
__device__ __forceinline__ double cfl_max2(double a, double b) { return (a < b) ? b : a; }

// per-substep advective CFL guard (src/main.cpp:1155-1176): over the interior,
// |bx| * dt / dx0 + |by| * dt / dx1 + |bz| * dt / dx2, maximum per workgroup
__global__ __launch_bounds__(RED_T) void cfl_max_kernel(BlockDesc b, const double* u, double dt, double* partial,
                                                        long per) {
#pragma clang fp contract(off)
    __shared__ double sh[RED_T];
    const long ncell = (long)b.n[0] * b.n[1] * b.n[2];
    const long beg = (long)blockIdx.x * per;
    const long end = beg + per < ncell ? beg + per : ncell;
    double m = 0.0;
    for (long t = beg + threadIdx.x; t < end; t += RED_T) {
        const int i = b.ng + (int)(t % b.n[0]);
        const int j = b.ng + (int)((t / b.n[0]) % b.n[1]);
        const int k = b.ng + (int)(t / ((long)b.n[0] * b.n[1]));
        const long c = i + (long)b.nt[0] * (j + (long)b.nt[1] * k);
        const double bx = fabs(u[BX * b.stride + c]), by = fabs(u[(BX + 1) * b.stride + c]),
                     bz = fabs(u[(BX + 2) * b.stride + c]);
        const double local = bx * dt / b.dx[0] + by * dt / b.dx[1] + bz * dt / b.dx[2];
        m = cfl_max2(m, local);
    }
    sh[threadIdx.x] = m;
    __syncthreads();
    for (int o = RED_T / 2; o > 0; o >>= 1) {
        if ((int)threadIdx.x < o) sh[threadIdx.x] = cfl_max2(sh[threadIdx.x], sh[threadIdx.x + o]);
        __syncthreads();
    }
    if (threadIdx.x == 0) partial[blockIdx.x] = sh[0];
}

__global__ __launch_bounds__(RED_T) void max_partials_kernel(const double* partial, int n, double* out) {
    __shared__ double sh[RED_T];
    double m = 0.0;
    for (int t = threadIdx.x; t < n; t += RED_T) m = cfl_max2(m, partial[t]);
    sh[threadIdx.x] = m;
    __syncthreads();
    for (int o = RED_T / 2; o > 0; o >>= 1) {
        if ((int)threadIdx.x < o) sh[threadIdx.x] = cfl_max2(sh[threadIdx.x], sh[threadIdx.x + o]);
        __syncthreads();
    }
    if (threadIdx.x == 0) out[0] = sh[0];
}

// setGaugeWaveData (src/spacetime/ccz4.cpp:1190-1221): H = A sin(2 pi x / L) (the product
// 2 pi x formed left to right, then divided by L), chi = (1 + H)^(-1/3), gt_xx = (1 + H) chi,
// gt_yy = gt_zz = chi, alpha = sqrt(1 + H); the fields it does not set are 0, as on a
// freshly constructed GridBlock
__global__ void init_gauge_wave_kernel(BlockDesc b, double* u, double A, double L) {
#pragma clang fp contract(off)
    const long t = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= b.stride) return;
    const int i = (int)(t % b.nt[0]);
    const double x = coord(b, 0, i);
    const double H = A * sin(2.0 * PI * x / L);
    const double detg = 1.0 + H;
    const double chi = pow(detg, -1.0 / 3.0);
    for (int v = 0; v < NV; ++v) u[v * b.stride + t] = 0.0;
    u[CHI * b.stride + t] = chi;
    u[(GXX + 0) * b.stride + t] = (1.0 + H) * chi;
    u[(GXX + 3) * b.stride + t] = chi;
    u[(GXX + 5) * b.stride + t] = chi;
    u[ALPHA * b.stride + t] = sqrt(1.0 + H);
}

inline unsigned grid_for(long n, int threads) { return (unsigned)((n + threads - 1) / threads); }

} // namespace

Stencil<double> make_stencil(const BlockDesc& b, double ko_sigma) {
    Stencil<double> K;
    static const double wts[4] = {1.0, -6.0, 15.0, -20.0};
    for (int d = 0; d < 3; ++d) {
        K.ih[d] = 1.0 / (12.0 * b.dx[d]);
        K.ih2[d] = 1.0 / (12.0 * b.dx[d] * b.dx[d]);
        K.ko[d] = ko_sigma / (64.0 * b.dx[d]);
        for (int s = 0; s < 4; ++s) K.kw[d][s] = K.ko[d] * wts[s];
    }
    K.ihh[0] = 1.0 / (4.0 * b.dx[0] * b.dx[1]);
    K.ihh[1] = 1.0 / (4.0 * b.dx[0] * b.dx[2]);
    K.ihh[2] = 1.0 / (4.0 * b.dx[1] * b.dx[2]);
    return K;
}

void stage_tile_fp64(int* t3) {
    t3[0] = TILE_X;
    t3[1] = TILE_Y;
    t3[2] = TZ_LARGE;
}

void stage_tile_mixed(int* t3) {
    t3[0] = TILE_X;
    t3[1] = TILE_Y;
    t3[2] = TILE_Z;
}

#ifndef GR_XCD_REMAP
#define GR_XCD_REMAP 1
#endif

static StageArgs stage_args(const Batch& B, const int sel[3], const CellParams& P, double ko_sigma,
                            const StageCoef& cf, const unsigned char* flags, int want) {
    StageArgs A;
    A.batch = B;
    A.sel_in = sel[0];
    A.sel_un = sel[1];
    A.sel_out = sel[2];
    A.ntiles = B.ntiles;
    A.xcd_remap = GR_XCD_REMAP ? 1 : 0;
    BlockDesc g;
    for (int d = 0; d < 3; ++d) g.dx[d] = B.dx[d];
    A.K = make_stencil(g, ko_sigma);
    for (int d = 0; d < 3; ++d) {
        A.K32.ih[d] = (float)A.K.ih[d];
        A.K32.ih2[d] = (float)A.K.ih2[d];
        A.K32.ihh[d] = (float)A.K.ihh[d];
        A.K32.ko[d] = (float)A.K.ko[d];
        for (int t = 0; t < 4; ++t) A.K32.kw[d][t] = (float)A.K.kw[d][t];
    }
    A.P = P;
    A.cf = cf;
    A.ko_on = ko_sigma <= 0.0 ? 0 : 1; // applyDissipation returns early only for sigma <= 0 (NaN dissipates)
    A.flags = flags;
    A.want = want;
    A.scan = 0;
    return A;
}

int stage_tiles(const BlockDesc& b) {
    return ((b.n[0] + TILE_X - 1) / TILE_X) * ((b.n[1] + TILE_Y - 1) / TILE_Y) * ((b.n[2] + TILE_Z - 1) / TILE_Z);
}

static long host_ghost_count(const BlockDesc& b) {
    return 2L * b.ng * b.nt[1] * b.nt[0] + (long)b.n[2] * 2 * b.ng * b.nt[0] + (long)b.n[2] * b.n[1] * 2 * b.ng;
}

int batch_layout(std::vector<BatchBlock>& blocks, std::vector<int>& tile_block, std::vector<int>& ghost_wg_block) {
    int t = 0;
    tile_block.clear();
    ghost_wg_block.clear();
    for (size_t i = 0; i < blocks.size(); ++i) {
        BatchBlock& B = blocks[i];
        B.tiles[0] = (B.b.n[0] + TILE_X - 1) / TILE_X;
        B.tiles[1] = (B.b.n[1] + TILE_Y - 1) / TILE_Y;
        B.tiles[2] = (B.b.n[2] + TILE_Z - 1) / TILE_Z;
        B.tile0 = t;
        const int nt = B.tiles[0] * B.tiles[1] * B.tiles[2];
        tile_block.insert(tile_block.end(), nt, (int)i);
        t += nt;
        B.ghost_wg0 = (int)ghost_wg_block.size();
        ghost_wg_block.insert(ghost_wg_block.end(), grid_for(host_ghost_count(B.b), GHOST_WG), (int)i);
    }
    return t;
}

bool pairs_aligned(const BlockDesc& b, const void* p) {
    return b.nt[0] % 2 == 0 && (reinterpret_cast<uintptr_t>(p) & 15) == 0;
}

Batch single_batch(const BlockDesc& b, const double* in, const double* un, double* out, const Sources& src) {
    Batch B;
    B.pairs_ok = pairs_aligned(b, in) && pairs_aligned(b, un) && pairs_aligned(b, out);
    B.variant = 0;
    B.ghost_groups = GR_GHOST_GROUPS;
    B.table = nullptr;
    B.tile_block = nullptr;
    B.ghost_wg_block = nullptr;
    B.nblocks = 1;
    B.one.b = b;
    B.one.buf[0] = const_cast<double*>(in);
    B.one.buf[1] = const_cast<double*>(un);
    B.one.buf[2] = out;
    B.one.src = src;
    B.one.tile0 = 0;
    B.one.tiles[0] = (b.n[0] + TILE_X - 1) / TILE_X;
    B.one.tiles[1] = (b.n[1] + TILE_Y - 1) / TILE_Y;
    B.one.tiles[2] = (b.n[2] + TILE_Z - 1) / TILE_Z;
    B.ntiles = B.one.tiles[0] * B.one.tiles[1] * B.one.tiles[2];
    B.one.ghost_wg0 = 0;
    B.ghost_wgs = (int)grid_for(host_ghost_count(b), GHOST_WG);
    for (int d = 0; d < 3; ++d) B.dx[d] = b.dx[d];
    return B;
}

bool stage_parts_large(const Batch& B) {
    const int form = B.pairs_ok ? B.variant : 0;
    return form == 2 || (form == 0 && B.ntiles >= LARGE_TILES);
}

hipError_t launch_stage_fp64(const Batch& B, const int sel[3], bool has_src, const CellParams& P,
                             double ko_sigma, int mode, const StageCoef& cf, hipStream_t s,
                             const unsigned char* flags) {
    const bool large = stage_parts_large(B);
    StageArgs A = stage_args(B, sel, P, ko_sigma, cf, flags, 1);
    // with flags (the FP64 tiles of the mixed form: few, near the puncture) a small grid
    // gathers them instead of launching one workgroup per part of every tile of the level
    int nblk = 0;
    if (flags) {
        A.scan = 1;
        nblk = A.ntiles * FP64_PARTS<TZ_LARGE>;
        if (nblk > FP64_SCAN_GRID) nblk = FP64_SCAN_GRID;
    }
    if (has_src) {
        if (mode == MODE_RHS) return launch_stage_t<MODE_RHS, true>(A, nblk, large, s);
        if (mode == MODE_STAGE) return launch_stage_t<MODE_STAGE, true>(A, nblk, large, s);
        return launch_stage_t<MODE_FINAL, true>(A, nblk, large, s);
    }
    if (mode == MODE_RHS) return launch_stage_t<MODE_RHS, false>(A, nblk, large, s);
    if (mode == MODE_STAGE) return launch_stage_t<MODE_STAGE, false>(A, nblk, large, s);
    return launch_stage_t<MODE_FINAL, false>(A, nblk, large, s);
}

template <int MODE, bool HAS_SRC>
static hipError_t launch_mixed_t(const StageArgs& A, hipStream_t s) {
    const dim3 grid(A.ntiles * FP64_PARTS<TZ_LARGE>), wg(64 * TZ_LARGE);
    // the first stage (u^n is the stage input) has an instance of its own, so that no load
    // of the kernel's register prefetch is conditional
    if (MODE == MODE_STAGE && A.sel_un == A.sel_in)
        stage_kernel_mixed<TZ_LARGE, MODE, HAS_SRC, MODE == MODE_STAGE><<<grid, wg, 0, s>>>(A);
    else
        stage_kernel_mixed<TZ_LARGE, MODE, HAS_SRC><<<grid, wg, 0, s>>>(A);
    return hipGetLastError();
}

hipError_t launch_stage_mixed(const Batch& B, const int sel[3], bool has_src, const CellParams& P,
                              double ko_sigma, int mode, const StageCoef& cf, hipStream_t s, unsigned char* flags,
                              double chi_fp64_below, const AuxStream* aux) {
    const StageArgs A = stage_args(B, sel, P, ko_sigma, cf, flags, 0);
    classify_tiles_kernel<TILE_X, TILE_Y, TILE_Z>
        <<<dim3(A.ntiles), dim3(TILE_X * TILE_Y * TILE_Z), 0, s>>>(A, chi_fp64_below, flags);
    hipError_t st = hipGetLastError();
    if (st != hipSuccess) return st;
    // the FP64 tiles (flag 1) run beside the FP32 kernel on the auxiliary stream: both read
    // the stage input and write disjoint tiles of the output
    if (aux) {
        if ((st = hipEventRecord(aux->fork, s)) != hipSuccess) return st;
        if ((st = hipStreamWaitEvent(aux->stream, aux->fork, 0)) != hipSuccess) return st;
        if ((st = launch_stage_fp64(B, sel, has_src, P, ko_sigma, mode, cf, aux->stream, flags)) != hipSuccess)
            return st;
        if ((st = hipEventRecord(aux->join, aux->stream)) != hipSuccess) return st;
    }
    // FP32 tiles (flag 0)
    if (has_src) {
        if (mode == MODE_RHS) st = launch_mixed_t<MODE_RHS, true>(A, s);
        else if (mode == MODE_STAGE) st = launch_mixed_t<MODE_STAGE, true>(A, s);
        else st = launch_mixed_t<MODE_FINAL, true>(A, s);
    } else {
        if (mode == MODE_RHS) st = launch_mixed_t<MODE_RHS, false>(A, s);
        else if (mode == MODE_STAGE) st = launch_mixed_t<MODE_STAGE, false>(A, s);
        else st = launch_mixed_t<MODE_FINAL, false>(A, s);
    }
    if (st != hipSuccess) return st;
    if (aux) return hipStreamWaitEvent(s, aux->join, 0);
    // FP64 tiles near the puncture (flag 1)
    return launch_stage_fp64(B, sel, has_src, P, ko_sigma, mode, cf, s, flags);
}

bool ghost_groups_valid(int g) { return g == 1 || g == 2 || g == 4 || g == 11; }

template <int G>
static void fill_batch_g(const Batch& B, int sel, int mode, hipStream_t s) {
    fill_ghosts_batch_kernel<G><<<dim3(B.ghost_wgs, G), GHOST_WG, 0, s>>>(B.table, B.ghost_wg_block, sel, mode);
}

hipError_t launch_fill_ghosts_batch(const Batch& B, int sel, int mode, hipStream_t s) {
    if (!B.table) return launch_fill_ghosts(B.one.b, B.one.buf[sel], mode, s, 0x3f, B.ghost_groups);
    switch (B.ghost_groups) {
    case 1: fill_batch_g<1>(B, sel, mode, s); break;
    case 2: fill_batch_g<2>(B, sel, mode, s); break;
    case 11: fill_batch_g<11>(B, sel, mode, s); break;
    default: fill_batch_g<4>(B, sel, mode, s); break;
    }
    return hipGetLastError();
}

template <int G>
static void fill_one_g(const BlockDesc& b, double* u, int mode, hipStream_t s, int faces, long n) {
    fill_ghosts_kernel<G><<<dim3(grid_for(n, GHOST_WG), G), GHOST_WG, 0, s>>>(b, u, mode, faces);
}

hipError_t launch_fill_ghosts(const BlockDesc& b, double* u, int mode, hipStream_t s, int faces, int groups) {
    const long nA = 2L * b.ng * b.nt[1] * b.nt[0];
    const long nB = (long)b.n[2] * 2 * b.ng * b.nt[0];
    const long nC = (long)b.n[2] * b.n[1] * 2 * b.ng;
    const long n = nA + nB + nC;
    switch (groups) {
    case 1: fill_one_g<1>(b, u, mode, s, faces, n); break;
    case 2: fill_one_g<2>(b, u, mode, s, faces, n); break;
    case 11: fill_one_g<11>(b, u, mode, s, faces, n); break;
    default: fill_one_g<4>(b, u, mode, s, faces, n); break;
    }
    return hipGetLastError();
}

hipError_t launch_prolong_axes(const BlockDesc& c, const BlockDesc& f, ProlongAxis* tab, hipStream_t s) {
    prolong_axes_kernel<<<grid_for(f.nt[0] + f.nt[1] + f.nt[2], 256), 256, 0, s>>>(c, f, tab);
    return hipGetLastError();
}

hipError_t launch_prolongate(const BlockDesc& c, const double* cu, const BlockDesc& f, double* fu,
                             const ProlongAxis* tab, hipStream_t s, int groups) {
    const int ntx = (f.nt[0] + PT_X - 1) / PT_X, nty = (f.nt[1] + PT_Y - 1) / PT_Y, ntz = (f.nt[2] + PT_Z - 1) / PT_Z;
    const int g = groups > 0 && groups <= NV ? groups : GR_TRANSFER_GROUPS;
    prolong_kernel<<<dim3(ntx * nty * ntz, g), PT_N, 0, s>>>(c, cu, f, fu, tab, ntx, nty);
    return hipGetLastError();
}

hipError_t launch_restrict(const BlockDesc& f, const double* fu, const BlockDesc& c, double* cu, hipStream_t s,
                           int groups) {
    const long n = (long)c.n[0] * c.n[1] * c.n[2];
    const int g = groups > 0 && groups <= NV ? groups : GR_TRANSFER_GROUPS;
    restrict_kernel<<<dim3(grid_for(n, 256), g), 256, 0, s>>>(f, fu, c, cu);
    return hipGetLastError();
}

hipError_t launch_pack_interior(const BlockDesc& b, const double* r, double* out, hipStream_t s) {
    const long n = (long)b.n[0] * b.n[1] * b.n[2];
    pack_interior_kernel<<<dim3(grid_for(n, 256), NV), 256, 0, s>>>(b, r, out);
    return hipGetLastError();
}

hipError_t launch_dissipation(const BlockDesc& b, const double* u, double* rhs, double ko_sigma, hipStream_t s) {
    if (ko_sigma <= 0.0) return hipSuccess;
    const long n = (long)b.n[0] * b.n[1] * b.n[2];
    dissipation_kernel<<<grid_for(n, 256), 256, 0, s>>>(b, u, rhs, make_stencil(b, ko_sigma));
    return hipGetLastError();
}

// workgroups and parts per workgroup of a monitor launch with at most `cap` workgroups; sums take
// the 512 that run together (two per CU), so that each has the same number of parts but one
constexpr int MONITOR_GROUPS = 512;
static int monitor_split(int ntiles, int cap, int* per) {
    const int nparts = ntiles * FP64_PARTS<TZ_LARGE>;
    *per = (nparts + cap - 1) / cap;
    return (nparts + *per - 1) / *per;
}

static hipError_t launch_monitor(const BlockDesc& b, const double* u, double* ham, double* mom, bool with_mom,
                                 double* partial, int cap, int* groups, hipStream_t s) {
    static const int sel[3] = {0, 0, 0};
    const StageArgs A = stage_args(single_batch(b, u, u, nullptr), sel, CellParams{}, 0.0, StageCoef{0.0, 0.0, 0.0},
                                   nullptr, 0);
    int per = 1;
    *groups = monitor_split(A.ntiles, cap, &per);
    if (with_mom)
        constraints_kernel<true><<<*groups, 64 * TZ_LARGE, 0, s>>>(A, ham, mom, partial, per);
    else
        constraints_kernel<false><<<*groups, 64 * TZ_LARGE, 0, s>>>(A, ham, nullptr, partial, per);
    return hipGetLastError();
}

hipError_t launch_constraints(const BlockDesc& b, const double* u, double* ham, double* mom, hipStream_t s) {
    zero_kernel<<<grid_for(b.stride, 256 * 4), 256, 0, s>>>(ham, b.stride);
    if (mom) zero_kernel<<<grid_for(3 * b.stride, 256 * 4), 256, 0, s>>>(mom, 3 * b.stride);
    int groups = 0;
    return launch_monitor(b, u, ham, mom, mom != nullptr, nullptr, 1 << 30, &groups, s);
}

hipError_t launch_constraint_sums(const BlockDesc& b, const double* u, bool with_mom, double* partial, int cap,
                                  double* out, hipStream_t s) {
    int groups = 0;
    const hipError_t st = launch_monitor(b, u, nullptr, nullptr, with_mom, partial,
                                         cap < MONITOR_GROUPS ? cap : MONITOR_GROUPS, &groups, s);
    if (st != hipSuccess) return st;
    sum_partials_kernel<<<with_mom ? 2 : 1, RED_T, 0, s>>>(partial, groups, out);
    return hipGetLastError();
}

hipError_t launch_init_bl(const BlockDesc& b, double* u, int nbh, const double* mass, const double* pos,
                          hipStream_t s) {
    init_bl_kernel<<<grid_for(b.stride, 256), 256, 0, s>>>(b, u, nbh, mass, pos);
    return hipGetLastError();
}

hipError_t launch_add_noise(const BlockDesc& b, double* u, unsigned long long seed, double amp, unsigned mask,
                            hipStream_t s) {
    add_noise_kernel<<<grid_for(b.stride, 256), 256, 0, s>>>(b, u, seed, amp, mask);
    return hipGetLastError();
}

static long reduce_split(const BlockDesc& b, int cap, int* nparts) {
    const long ncell = (long)b.n[0] * b.n[1] * b.n[2];
    long per = (ncell + cap - 1) / cap;
    if (per < RED_T) per = RED_T;
    *nparts = (int)((ncell + per - 1) / per);
    return per;
}

hipError_t launch_count_nonfinite(const BlockDesc& b, const double* u, double* partial, int cap, int* nparts,
                                  hipStream_t s) {
    const long per = reduce_split(b, cap, nparts);
    nonfinite_kernel<<<*nparts, RED_T, 0, s>>>(b, u, partial, per);
    return hipGetLastError();
}

hipError_t launch_first_nonfinite(const BlockDesc& b, const double* u, unsigned long long* partial, int cap,
                                  int* nparts, hipStream_t s) {
    const long total = NV * (long)b.n[0] * b.n[1] * b.n[2];
    long per = (total + cap - 1) / cap;
    if (per < RED_T) per = RED_T;
    *nparts = (int)((total + per - 1) / per);
    first_nonfinite_kernel<<<*nparts, RED_T, 0, s>>>(b, u, partial, per);
    return hipGetLastError();
}

hipError_t launch_min_partials(const unsigned long long* partial, int n, unsigned long long* out, hipStream_t s) {
    min_partials_kernel<<<1, RED_T, 0, s>>>(partial, n, out);
    return hipGetLastError();
}

hipError_t launch_cfl_max(const BlockDesc& b, const double* u, double dt, double* partial, int cap, int* nparts,
                          hipStream_t s) {
    const long per = reduce_split(b, cap, nparts);
    cfl_max_kernel<<<*nparts, RED_T, 0, s>>>(b, u, dt, partial, per);
    return hipGetLastError();
}

hipError_t launch_max_partials(const double* partial, int n, double* out, hipStream_t s) {
    max_partials_kernel<<<1, RED_T, 0, s>>>(partial, n, out);
    return hipGetLastError();
}

hipError_t launch_init_gauge_wave(const BlockDesc& b, double* u, double A, double L, hipStream_t s) {
    init_gauge_wave_kernel<<<grid_for(b.stride, 256), 256, 0, s>>>(b, u, A, L);
    return hipGetLastError();
}

hipError_t launch_sum_partials(const double* partial, int n, double* out, hipStream_t s) {
    sum_partials_kernel<<<1, RED_T, 0, s>>>(partial, n, out);
    return hipGetLastError();
}

} // namespace gr
