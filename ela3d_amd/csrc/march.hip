// march.hip -- one whole time step (stress and velocity half-steps of every cell, the
// absorbing layers included) in a single launch, double-buffered field sets.
//
// A workgroup owns `rows` consecutive rows of a chunk of up to 64 columns and marches them
// through a z segment.  One wave per row, one column per lane.  One more wave holds both
// halo rows: the row below gives sigma_xy and sigma_yz, the row above sigma_yy, each only
// what the own rows' velocities read.  Every field and model array is read once per cell
// of the region (12 loads a plane, 7 on a halo row); nothing is loaded for a neighbour:
//  * x neighbours: DPP wave shifts (a chunk inside the grid holds one more column per side);
//  * y neighbours: LDS.  A wave publishes what the rows beside it read -- velocities and
//    material of the plane to come, new stresses of this plane -- in one of two alternating
//    sets of row buffers, so one LDS barrier per plane orders everything;
//  * z neighbours: registers, carried from plane to plane.
// 24 (FP64 16) waves per compute unit with no spilled register are what hides the loads:
// variants with two or four columns per lane (half the waves, misaligned vectors) and with
// streaming loads or stores were 5 to 30 % slower at 401 x 401 x 301, the next plane's loads
// issued before the barrier (73 registers for 67) 2 %, 32 waves (spills) 5 %.  The halo rows
// share a wave: one each would be idle for half a plane (101^3: 47 -> 41 us a step).
// dt over the averaged densities is the IEEE division, for every density that is accepted: the
// hardware reciprocal and one correction saved 0.1 to 0.4 us of a step of 33^3 to 113x97x85 and
// nothing from 201^3 on, but gave NaN below 1.2e-38.
//
// Time per step, FP32, two passes of two launches and a tail against this: 33^3 19 -> 10 us,
// 64^3 23 -> 15, 101^3 43 -> 35, 201^3 244 -> 228, 401x401x301 1305 -> 1173, 480x500x360
// 2250 -> 1950; FP64 81x61x75 39 -> 30, 192x200x188 423 -> 353.  The small grids are bound by a
// chain of latencies: the tables, the plane below, each plane, the plane above.  The large
// ones move 5.5 GB a step at 401x401x301 (two passes 6.4), 1.2 times one read and one write of
// every array, at 4.7 TB/s, where a copy with as many streams reaches 5.6: a segment's ends are
// read again, and rows beside a tile where workgroups have drifted apart.
//
// Updates follow the reference CPU loops (seismicCPML_3d_isotropic_simpelmodel.cpp):
// normal stress CPU:377-413, sigma_xy CPU:415-442, sigma_xz/yz CPU:444-499,
// vx/vy CPU:501-560, vz CPU:562-590.
#include "geom.hpp"
#include "tail_util.hpp"

// Every multiply-add is written out: a cell's result is then the same bits whichever wave
// computes it (own or halo row, general or plain code).
#pragma clang fp contract(off)

namespace ela3d {
namespace {

constexpr int kLead = 8;  // workgroups before the grid's own, one per die
// roles of a wave
constexpr int kOwn = 0, kLow = 1, kHigh = 2;
// phases of a plane: below the segment (sigma_xz and sigma_yz only), in it, above it (sigma_zz only)
constexpr int kBelow = 0, kIn = 1, kAbove = 2;

// the value of the lane below (west) or above (east); lanes 0 and 63 get 0 there, which no
// result that is kept reads
template <int CTRL>
__device__ __forceinline__ float lane_shift(float x)
{
    return __uint_as_float(unsigned(__builtin_amdgcn_update_dpp(0, (int)__float_as_uint(x), CTRL, 0xf, 0xf, true)));
}
template <int CTRL>
__device__ __forceinline__ double lane_shift(double x)
{
    const unsigned long long b = (unsigned long long)__double_as_longlong(x);
    const unsigned lo = (unsigned)__builtin_amdgcn_update_dpp(0, (int)(unsigned)b, CTRL, 0xf, 0xf, true);
    const unsigned hi = (unsigned)__builtin_amdgcn_update_dpp(0, (int)(unsigned)(b >> 32), CTRL, 0xf, 0xf, true);
    return __longlong_as_double((long long)(((unsigned long long)hi << 32) | lo));
}
template <typename R>
__device__ __forceinline__ R west(R x) { return lane_shift<0x138>(x); }  // wave_shr:1
template <typename R>
__device__ __forceinline__ R east(R x) { return lane_shift<0x130>(x); }  // wave_shl:1

// a value that is the same in every lane, moved to scalar registers
__device__ __forceinline__ float scalar(float x) { return __int_as_float(__builtin_amdgcn_readfirstlane(__float_as_int(x))); }
__device__ __forceinline__ double scalar(double x)
{
    const unsigned long long b = (unsigned long long)__double_as_longlong(x);
    const unsigned lo = (unsigned)__builtin_amdgcn_readfirstlane((int)(unsigned)b);
    const unsigned hi = (unsigned)__builtin_amdgcn_readfirstlane((int)(unsigned)(b >> 32));
    return __longlong_as_double((long long)(((unsigned long long)hi << 32) | lo));
}

// A uniform value the compiler takes for a new one at every use, so that what is derived from
// it is computed there (scalar, or one vector add) and not kept in vector registers over the loop.
__device__ __forceinline__ int fresh(int x)
{
    asm volatile("" : "+s"(x));
    return x;
}

// a where the mask is all ones, b where it is 0: one v_bfi_b32.  (A select on a lane
// condition becomes a branch around the arithmetic of its operands, one per use.)
__device__ __forceinline__ float pick(unsigned m, float a, float b)
{
    return __uint_as_float((m & __float_as_uint(a)) | (~m & __float_as_uint(b)));
}
__device__ __forceinline__ double pick(unsigned m, double a, double b)
{
    const unsigned long long x = (unsigned long long)__double_as_longlong(a), y = (unsigned long long)__double_as_longlong(b);
    const unsigned lo = (m & unsigned(x)) | (~m & unsigned(y)), hi = (m & unsigned(x >> 32)) | (~m & unsigned(y >> 32));
    return __longlong_as_double((long long)(((unsigned long long)hi << 32) | lo));
}
__device__ __forceinline__ unsigned ones(bool b) { return b ? ~0u : 0u; }

// The kernel's arguments, for the array pointers: read again in every phase of a plane.
// Held over the loop, 57 pointers overflow the scalar registers, and each spilled one
// comes back through VALU lane reads; a scalar load costs no vector slot.
template <typename T>
using KArgs = const __attribute__((address_space(4))) StepArgs<T>;
template <typename T>
__device__ __forceinline__ KArgs<T>* kargs()
{
    auto p = (KArgs<T>*)__builtin_amdgcn_kernarg_segment_ptr();
    asm volatile("" : "+s"(p));  // a new value every time, so that no pointer is kept
    return p;
}

// Row buffers of a set: kU* hold the plane to come, kS* this plane's new stresses.
constexpr int kUvx = 0, kUvy = 1, kUvz = 2, kUcs = 3, kUrho = 4, kSxy = 5, kSyy = 6, kSyz = 7;
constexpr int kSlot = 8 * 64;  // elements of a row's buffers in one set
// Column tables after them: a, b, 1/K on the full grid, then on the half grid; dt where
// i <= nx-2 and where i >= 1, else 0, which leaves the old value outside an update's range.
// Then masks: not a rigid x face; in an x layer.  Then a, b, 1/K (full, half grid) of the
// rows' y layers and of the planes' z layers.
constexpr int kCdtN = 6, kCdtS = 7, kMfree = 0, kMin = 1;

template <typename T>
struct March {
    typedef typename Arith<T>::R R;
    const StepArgs<T>& A;
    R* lds;          // [2][slots][8][64]; the column tables R [8][64], unsigned [2][64] (in R [2][64]);
                     // the row and plane tables R [slots][6], [zseg + 2][6]
    int slots, slot, lane;
    int j, kb, ke, xs, xe;
    unsigned o0;     // element offset of the lane's cell at plane 0 (an idle lane's: the last column's)
    unsigned ox;     // x memory-variable offset at plane 0 (lanes in an x layer)
    bool own, inx;   // the lane's column is own; lies in an x layer
    bool hasx;       // some lane of the wave lies in an x layer
    int cy;
    bool edge;       // the row has a y layer, or is the grid's first or last
    R dt, idx, idy, idz;

    // this row's buffers in set b: rows beside it at -kSlot and +kSlot
    __device__ __forceinline__ R* rows(int b) const { return lds + fresh((b * slots + slot) * kSlot) + lane; }
    __device__ __forceinline__ const R* cols() const { return lds + fresh(2 * slots * kSlot) + lane; }
    __device__ __forceinline__ unsigned mask(int q) const
    {
        return reinterpret_cast<const unsigned*>(lds + fresh((2 * slots + 1) * kSlot))[q * 64 + lane];
    }
    __device__ __forceinline__ unsigned cell(int k) const { return o0 + unsigned(fresh(k * A.nxyp)); }
    __device__ __forceinline__ unsigned xoff(int k) const
    {
        const unsigned o = ox + unsigned(fresh(k * A.ny * A.w[0]));
        return inx ? o : 0u;
    }
    __device__ __forceinline__ int column() const { return fresh(xs) + lane; }
    // whether plane m of this row needs the general code: a y or z layer, or the grid's faces
    __device__ __forceinline__ bool general(int m) const
    {
        return edge || m == 0 || m == A.nz - 1 || m < A.lo[2] || m >= A.hi[2];
    }
    // The x recurrence on derivative d: psi becomes the new memory variable.  Outside the
    // layers psi = 0, a = 0, 1/K = 1 leave d as it is; where the update does not reach
    // (column 0 with the full-grid table, nx-1 with the half-grid one), a = 0 and b = 1 in
    // the workgroup's copy of the tables leave psi.  GEN: psi stays too where `on` is 0.
    template <bool HALF, bool GEN>
    __device__ __forceinline__ void xpml(R& psi, unsigned on, R& d) const
    {
        const R* c = cols() + (HALF ? 3 * 64 : 0);
        const R p = pick(mask(kMin), psi, (R)0), v = recur(p, c[0], c[64], c[128], d);
        psi = GEN ? pick(on, v, p) : v;
    }
};

// What a wave loads for plane m: the plane above's velocities and material, this plane's
// cp and stresses, the x memory variables of the stress update.
template <typename R>
struct MLoad {
    R vx, vy, vz, cs, rho, cp;
    R s[6];   // xx yy zz xy xz yz
    R mx[3];  // dvx_dx, dvy_dx, dvz_dx
};

template <int ROLE, int PH, bool HASX, typename T, typename R>
__device__ __forceinline__ void march_load(const March<T>& M, int m, MLoad<R>& L)
{
    KArgs<T>* K = kargs<T>();
    const unsigned o = M.cell(m);
    if constexpr (PH != kAbove) {
        const unsigned u = o + (m == M.A.nz - 1 ? 0u : unsigned(M.A.nxyp));
        L.vx = el(K->fi[0], u);
        L.vy = el(K->fi[1], u);
        L.vz = el(K->fi[2], u);
        L.cs = (R)el(K->cs, u);
        L.rho = (R)el(K->rho, u);
    }
    if constexpr ((ROLE == kOwn && PH != kBelow) || ROLE == kHigh) L.cp = (R)el(K->cp, o);
    if constexpr (ROLE == kOwn && PH == kIn) L.s[0] = el(K->fi[3], o);
    if constexpr ((ROLE == kOwn && PH == kIn) || ROLE == kHigh) L.s[1] = el(K->fi[4], o);
    if constexpr (ROLE == kOwn && PH != kBelow) L.s[2] = el(K->fi[5], o);
    if constexpr ((ROLE == kOwn && PH == kIn) || ROLE == kLow) L.s[3] = el(K->fi[6], o);
    if constexpr (ROLE == kOwn && PH != kAbove) L.s[4] = el(K->fi[7], o);
    if constexpr ((ROLE == kOwn && PH != kAbove) || ROLE == kLow) L.s[5] = el(K->fi[8], o);
    if constexpr (HASX) {
        const unsigned x = M.xoff(m);
        if constexpr ((ROLE == kOwn && PH != kBelow) || ROLE == kHigh) L.mx[0] = el(K->mi[0], x);
        if constexpr ((ROLE == kOwn && PH == kIn) || ROLE == kLow) L.mx[1] = el(K->mi[3], x);
        if constexpr (ROLE == kOwn && PH != kAbove) L.mx[2] = el(K->mi[5], x);
    }
}

// acc + diff * inv; in a layer, whose memory variable changes the derivative, acc + the changed one
template <bool GEN, typename R>
__device__ __forceinline__ R add_axis(R acc, R diff, R inv, bool layer, unsigned on, R& psi, const R* t)
{
    if constexpr (GEN) {
        if (layer) {
            R d = diff * inv;
            psi = pick(on, recur(psi, t[0], t[1], t[2], d), psi);
            return acc + d;
        }
    }
    return fma_r(diff, inv, acc);
}

// Absorbing layers of a general plane along y and z: memory-variable offsets and tables
// (a, b, 1/K on the full grid, then on the half grid).  cy, cz < 0: no layer.
template <typename T>
struct Layers {
    typedef typename Arith<T>::R R;
    int cy = -1, cz = -1;
    unsigned y = 0, z = 0;
    const R *Y = nullptr, *Z = nullptr;
    __device__ __forceinline__ void at(const March<T>& M, KArgs<T>* K, int m)
    {
        const int ic = min(M.column(), M.xe - 1);
        const R* t = M.lds + fresh((2 * M.slots + 1) * kSlot + 128);
        cy = M.cy;
        cz = layer_index(m, K->lo[2], K->hi[2]);
        y = ymem_offset(m, cy, ic, K->nx, K->w[1]);
        z = zmem_offset(cz, M.j, ic, K->nx, K->ny);
        Y = t + M.slot * 6;
        Z = t + (M.slots + m - M.kb + 1) * 6;
    }
};

// One row of a wave: its state and its share of a plane.
template <typename T, bool ENERGY, int ROLE, bool HASX>
struct Row {
    typedef typename Arith<T>::R R;
    const March<T>& M;
    // the plane whose stresses come next: its velocities and material, vz below it
    R vx, vy, vz, cs, rho, vzm;
    R sxx, szz, sxz, pxz, rhoN, rhoW, cpc;  // of the last stress update; pxz: sigma_xz one plane below
    R hz, hq, hs, hr;   // vz of the plane below: in-plane part, dt/rho, sigma_zz, rho
    R mv[3];            // the velocity update's x memory variables
    MLoad<R> L;

    __device__ __forceinline__ explicit Row(const March<T>& m) : M(m) {}

    // the queue at plane m, from memory
    __device__ __forceinline__ void head(int m)
    {
        KArgs<T>* K = kargs<T>();
        const unsigned o = M.cell(m);
        vx = el(K->fi[0], o);
        vy = el(K->fi[1], o);
        vz = el(K->fi[2], o);
        cs = (R)el(K->cs, o);
        rho = (R)el(K->rho, o);
    }
    // velocities and material of plane m, for the rows beside this one
    __device__ __forceinline__ void publish(int m)
    {
        R* r = M.rows(m & 1);
        if constexpr (ROLE != kLow) {
            r[kUvx * 64] = vx;
            r[kUvz * 64] = vz;
            r[kUcs * 64] = cs;
            r[kUrho * 64] = rho;
        }
        if constexpr (ROLE != kHigh) r[kUvy * 64] = vy;
    }
    // energy box of the lane's column (own rows)
    __device__ __forceinline__ unsigned in_box(int k) const
    {
        const StepArgs<T>& A = M.A;
        const int em = A.emargin, i = M.column(), j = M.j;
        return ones(M.own && i >= em && i < A.nx - 1 - em && j >= em && j < A.ny - 1 - em && k >= A.ek0 && k < A.ek1);
    }

    // New stresses of plane m (those the role and phase need): own rows in the segment store
    // them, and all publish what the rows beside read.  Then the queue advances to plane m+1.
    // GEN: the row or the plane lies in a layer or on a face; elsewhere every j and k
    // condition of the loops holds.
    template <int PH, bool GEN>
    __device__ __forceinline__ void stress(int m)
    {
        constexpr bool ST = ROLE == kOwn && PH == kIn;
        constexpr bool NORMAL = (ROLE == kOwn && PH != kBelow) || ROLE == kHigh;
        constexpr bool XY = (ROLE == kOwn && PH == kIn) || ROLE == kLow;
        constexpr bool XZ = ROLE == kOwn && PH != kAbove;
        constexpr bool YZ = (ROLE == kOwn && PH != kAbove) || ROLE == kLow;
        const int j = M.j, nz = M.A.nz;
        const R idx = M.idx, idy = M.idy, idz = M.idz;
        KArgs<T>* K = kargs<T>();
        R* const r = M.rows(m & 1);
        const R* const c = M.cols();
        R my[3] = {0, 0, 0}, mz[3] = {0, 0, 0};  // memory variables along y (1, 4, 7) and z (2, 6, 8)
        Layers<T> G;
        if constexpr (GEN) {
            G.at(M, K, m);
            if (G.cy >= 0) {
                if constexpr (NORMAL) my[0] = el(K->mi[1], G.y);
                if constexpr (XY) my[1] = el(K->mi[4], G.y);
                if constexpr (YZ) my[2] = el(K->mi[7], G.y);
            }
            if (G.cz >= 0) {
                if constexpr (NORMAL) mz[0] = el(K->mi[2], G.z);
                if constexpr (XZ) mz[1] = el(K->mi[6], G.z);
                if constexpr (YZ) mz[2] = el(K->mi[8], G.z);
            }
            if (PH != kAbove && m == nz - 1)  // zero ghost plane above the top (read with the ghost quirk only)
                L.vx = L.vy = L.cs = L.rho = 0;
        }
        if constexpr (ST && HASX) {
            const unsigned x = M.xoff(m);
            mv[0] = el(K->mi[9], x);
            mv[1] = el(K->mi[12], x);
            mv[2] = el(K->mi[15], x);
        }
        const bool surface = GEN && K->fs && m == 0;
        const unsigned iN = GEN ? ones(M.column() <= K->nx - 2) : ~0u, iS = GEN ? ones(M.column() >= 1) : ~0u;
        R csW = 0, csN = 0, syy = 0, sxy = 0, syz = 0;
        if constexpr (XY || XZ) {
            csW = west(cs);
            rhoW = west(rho);
        }
        if constexpr (XY || YZ) {
            csN = r[kSlot + kUcs * 64];
            rhoN = r[kSlot + kUrho * 64];
        }
        if constexpr (NORMAL) {  // CPU:377-413
            const R dtN = c[kCdtN * 64];
            const unsigned on = GEN ? ones(j >= 1 && (m >= 1 || surface)) & iN : ~0u;
            R exx = (east(vx) - vx) * idx, eyy = (vy - r[-kSlot + kUvy * 64]) * idy, ezz = (vz - vzm) * idz;
            if constexpr (HASX) M.template xpml<true, GEN>(L.mx[0], on, exx);
            if constexpr (GEN) {
                if (G.cy >= 0) my[0] = pick(on, recur(my[0], G.Y[0], G.Y[1], G.Y[2], eyy), my[0]);
                if (G.cz >= 0) mz[0] = pick(on, recur(mz[0], G.Z[0], G.Z[1], G.Z[2], ezz), mz[0]);
            }
            const R vp = L.cp;
            const R lambda = rho * fma_r(vp, vp, (R)-2 * cs * cs);
            const R l2m = rho * vp * vp;
            const R DT_l2m = dtN * l2m, DT_l = dtN * lambda;
            if constexpr (GEN) {  // traction-free surface: sigma_zz = 0 there gives the vertical strain rate
                if (surface) ezz = -(lambda / l2m) * (exx + eyy);
            }
            if constexpr (ST) {
                const R v = fma_r(DT_l2m, exx, DT_l * (eyy + ezz)) + L.s[0];
                sxx = GEN ? pick(on, v, L.s[0]) : v;
            }
            if constexpr (ROLE == kHigh || ST) {
                const R v = fma_r(DT_l2m, eyy, DT_l * (exx + ezz)) + L.s[1];
                syy = GEN ? pick(on, v, L.s[1]) : v;
            }
            if constexpr (ROLE == kOwn) {
                const R v = fma_r(DT_l2m, ezz, DT_l * (exx + eyy)) + L.s[2];
                szz = GEN ? pick(on & ones(!surface), v, L.s[2]) : v;
            }
        }
        if constexpr (XY) {  // mu averaged over (i-1,j), (i,j+1) (CPU:415-442)
            const unsigned on = GEN ? ones(j <= K->ny - 2) & iS : ~0u;
            R dx = (vy - west(vy)) * idx;
            if constexpr (HASX) M.template xpml<false, GEN>(L.mx[1], on, dx);
            const R d = add_axis<GEN>(dx, r[kSlot + kUvx * 64] - vx, idy, G.cy >= 0, on, my[1], G.Y + 3);
            const R vs = (csW + csN) * (R)0.5, rh = (rhoW + rhoN) * (R)0.5;
            const R v = fma_r(c[kCdtS * 64] * (rh * vs * vs), d, L.s[3]);
            sxy = GEN ? pick(on, v, L.s[3]) : v;
        }
        if constexpr (XZ) {  // mu averaged over (i-1,k), (i,k+1) (CPU:444-470)
            const unsigned on = GEN ? ones(m <= K->kmax_shear) & iS : ~0u;
            R dx = (vz - west(vz)) * idx;
            if constexpr (HASX) M.template xpml<false, GEN>(L.mx[2], on, dx);
            const R d = add_axis<GEN>(dx, L.vx - vx, idz, G.cz >= 0, on, mz[1], G.Z + 3);
            const R vs = (csW + L.cs) * (R)0.5, rh = (rhoW + L.rho) * (R)0.5;
            const R v = fma_r(c[kCdtS * 64] * (rh * vs * vs), d, L.s[4]);
            sxz = GEN ? pick(on, v, L.s[4]) : v;
        }
        if constexpr (YZ) {  // mu averaged over (j+1,k), (j,k+1) (CPU:472-497)
            const unsigned on = GEN ? ones(m <= K->kmax_shear && j <= K->ny - 2) : ~0u;
            R dy = (r[kSlot + kUvz * 64] - vz) * idy;
            if constexpr (GEN) {
                if (G.cy >= 0) my[2] = pick(on, recur(my[2], G.Y[3], G.Y[4], G.Y[5], dy), my[2]);
            }
            const R d = add_axis<GEN>(dy, L.vy - vy, idz, G.cz >= 0, on, mz[2], G.Z + 3);
            const R vs = (csN + L.cs) * (R)0.5, rh = (rhoN + L.rho) * (R)0.5;
            const R v = fma_r(M.dt * (rh * vs * vs), d, L.s[5]);
            syz = GEN ? pick(on, v, L.s[5]) : v;
        }
        if constexpr (ST) {
            if (M.own) {
                const unsigned o = M.cell(m);
                el(K->fo[3], o) = sxx;
                el(K->fo[4], o) = syy;
                el(K->fo[5], o) = szz;
                el(K->fo[6], o) = sxy;
                el(K->fo[7], o) = sxz;
                el(K->fo[8], o) = syz;
                if constexpr (GEN) {
                    if (G.cy >= 0) {
                        el(K->mo[1], G.y) = my[0];
                        el(K->mo[4], G.y) = my[1];
                        el(K->mo[7], G.y) = my[2];
                    }
                    if (G.cz >= 0) {
                        el(K->mo[2], G.z) = mz[0];
                        el(K->mo[6], G.z) = mz[1];
                        el(K->mo[8], G.z) = mz[2];
                    }
                }
                if constexpr (HASX) {
                    if (M.inx) {
                        const unsigned x = M.xoff(m);
                        el(K->mo[0], x) = L.mx[0];
                        el(K->mo[3], x) = L.mx[1];
                        el(K->mo[5], x) = L.mx[2];
                    }
                }
            }
            if (ENERGY) cpc = L.cp;
        }
        if constexpr (XY) r[kSxy * 64] = sxy;
        if constexpr (ROLE == kHigh || ST) r[kSyy * 64] = syy;
        if constexpr (YZ) r[kSyz * 64] = syz;  // below the segment too: the first velocities read it
        if constexpr (PH == kBelow) pxz = sxz;
        if constexpr (PH != kAbove) {  // the queue moves up a plane
            vzm = vz;
            vx = L.vx;
            vy = L.vy;
            vz = L.vz;
            cs = L.cs;
            rho = L.rho;
        }
    }

    // vz of plane k once sigma_zz above it is known (CPU:562-590)
    template <bool GEN>
    __device__ __forceinline__ void finish_vz(int k, double& ek)
    {
        const int j = M.j, nz = M.A.nz;
        KArgs<T>* K = kargs<T>();
        const R hv = M.rows(k & 1)[kUvz * 64];  // the old value, still in this wave's row
        const unsigned free = M.mask(kMfree);
        R psi = 0;
        unsigned keep = ~0u, on = ~0u;
        Layers<T> G;
        if constexpr (GEN) {
            on = ones(j >= 1 && k <= nz - 2 && M.column() <= K->nx - 2);
            keep = ones(!(K->dirichlet && (j == 0 || j == K->ny - 1 || (k == 0 && !K->fs) || k == nz - 1)));
            G.at(M, K, k);
            if (G.cz >= 0) psi = el(K->mi[17], G.z);
        }
        const R u = fma_r(hq, add_axis<GEN>(hz, szz - hs, M.idz, G.cz >= 0, on, psi, G.Z + 3), hv);
        const R v = pick(free & keep, GEN ? pick(on, u, hv) : u, (R)0);
        if (M.own) {
            el(K->fo[2], M.cell(k)) = v;
            if constexpr (GEN) {
                if (G.cz >= 0) el(K->mo[17], G.z) = psi;
            }
        }
        if constexpr (ENERGY) ek += (double)pick(in_box(k), ((R)0.5 * hr * v) * v, (R)0);
    }

    // vx, vy of plane m, and what vz needs later, from the new stresses (own rows in the
    // segment).  The old velocities and density of the plane, sigma_yz below it and the new
    // stresses that were published are still in this wave's rows: read back from there.
    template <bool GEN>
    __device__ __forceinline__ void velocity(int m, double& ek, double& ep)
    {
        const int j = M.j, nz = M.A.nz;
        const R idx = M.idx, idy = M.idy, idz = M.idz;
        KArgs<T>* K = kargs<T>();
        const R* const r = M.rows(m & 1);
        const R* const c = M.cols();
        R my[3] = {0, 0, 0}, mz[2] = {0, 0};  // memory variables along y (10, 13, 16) and z (11, 14)
        Layers<T> G;
        if constexpr (GEN) {
            G.at(M, K, m);
            if (G.cy >= 0) {
                my[0] = el(K->mi[10], G.y);
                my[1] = el(K->mi[13], G.y);
                my[2] = el(K->mi[16], G.y);
            }
            if (G.cz >= 0) {
                mz[0] = el(K->mi[11], G.z);
                mz[1] = el(K->mi[14], G.z);
            }
        }
        const bool surface = GEN && K->fs && m == 0;
        const bool kon = !GEN || m >= 1 || surface;
        const unsigned iN = GEN ? ones(M.column() <= K->nx - 2) : ~0u, iS = GEN ? ones(M.column() >= 1) : ~0u;
        const unsigned free =
            M.mask(kMfree) &
            (GEN ? ones(!(K->dirichlet && (j == 0 || j == K->ny - 1 || (m == 0 && !surface) || m == nz - 1))) : ~0u);
        const R rhoc = r[kUrho * 64], sxy = r[kSxy * 64], syz = r[kSyz * 64];
        R nvx, nvy;
        {  // vx (CPU:502-529); at a free surface the image sigma_xz(k-1/2) = -sigma_xz(k+1/2)
            const unsigned on = GEN ? ones(j >= 1 && kon) & iS : ~0u;
            const R old = r[kUvx * 64];
            R d = (sxx - west(sxx)) * idx;
            if constexpr (HASX) M.template xpml<false, GEN>(mv[0], on, d);
            d = add_axis<GEN>(d, sxy - r[-kSlot + kSxy * 64], idy, G.cy >= 0, on, my[0], G.Y);
            d = add_axis<GEN>(d, sxz - (surface ? -sxz : pxz), idz, G.cz >= 0, on, mz[0], G.Z);
            const R v = fma_r(c[kCdtS * 64] / ((rhoc + rhoW) * (R)0.5), d, old);
            nvx = pick(free, GEN ? pick(on, v, old) : v, (R)0);
        }
        {  // vy (CPU:531-558)
            const unsigned on = GEN ? ones(j <= K->ny - 2 && kon) & iN : ~0u;
            const R old = r[kUvy * 64], below = M.rows((m & 1) ^ 1)[kSyz * 64];
            R d = (east(sxy) - sxy) * idx;
            if constexpr (HASX) M.template xpml<true, GEN>(mv[1], on, d);
            d = add_axis<GEN>(d, r[kSlot + kSyy * 64] - r[kSyy * 64], idy, G.cy >= 0, on, my[1], G.Y + 3);
            d = add_axis<GEN>(d, syz - (surface ? -syz : below), idz, G.cz >= 0, on, mz[1], G.Z);
            const R v = fma_r(c[kCdtN * 64] / ((rhoc + rhoN) * (R)0.5), d, old);
            nvy = pick(free, GEN ? pick(on, v, old) : v, (R)0);
        }
        {  // vz: the in-plane derivatives (CPU:562-590)
            const unsigned on = GEN ? ones(j >= 1 && m <= nz - 2) & iN : ~0u;
            R d = (east(sxz) - sxz) * idx;
            if constexpr (HASX) M.template xpml<true, GEN>(mv[2], on, d);
            hz = add_axis<GEN>(d, syz - r[-kSlot + kSyz * 64], idy, G.cy >= 0, on, my[2], G.Y);
            hq = c[kCdtN * 64] / ((rhoc + rho) * (R)0.5);  // rho: of plane m+1 by now
            hs = szz;
            if (ENERGY) hr = rhoc;
        }
        if (M.own) {
            const unsigned o = M.cell(m);
            el(K->fo[0], o) = nvx;
            el(K->fo[1], o) = nvy;
            if constexpr (GEN) {
                if (G.cy >= 0) {
                    el(K->mo[10], G.y) = my[0];
                    el(K->mo[13], G.y) = my[1];
                    el(K->mo[16], G.y) = my[2];
                }
                if (G.cz >= 0) {
                    el(K->mo[11], G.z) = mz[0];
                    el(K->mo[14], G.z) = mz[1];
                }
            }
            if constexpr (HASX) {
                if (M.inx) {
                    const unsigned x = M.xoff(m);
                    el(K->mo[9], x) = mv[0];
                    el(K->mo[12], x) = mv[1];
                    el(K->mo[15], x) = mv[2];
                }
            }
        }
        if constexpr (ENERGY) {
            const unsigned in = in_box(m);
            const R k2 = kinetic_energy<T>(rhoc, nvx, nvy, (R)0);
            const R p2 = strain_energy<T>(rhoc, cpc, (R)r[kUcs * 64], sxx, (R)r[kSyy * 64], szz, sxy, sxz, syz);
            ek += (double)pick(in, k2, (R)0);
            ep += (double)pick(in, p2, (R)0);
        }
        pxz = sxz;
    }
};

// An own row's march over planes [kb, ke) of the segment, one plane below and one above it.
template <typename T, bool ENERGY, bool HASX>
__device__ __forceinline__ void march_own(const March<T>& M, double& ek, double& ep)
{
    const int kb = M.kb, ke = M.ke, nz = M.A.nz;
    Row<T, ENERGY, kOwn, HASX> w(M);
    w.head(kb > 0 ? kb - 1 : 0);
    w.vzm = 0;
    w.pxz = 0;
    if (kb > 0) {
        march_load<kOwn, kBelow, HASX>(M, kb - 1, w.L);
        w.publish(kb - 1);
        lds_barrier();
        w.template stress<kBelow, true>(kb - 1);
    } else {
        M.rows(1)[kSyz * 64] = 0;  // nothing below plane 0
    }
    w.publish(kb);
    lds_barrier();
    for (int m = kb; m < ke; ++m) {
        march_load<kOwn, kIn, HASX>(M, m, w.L);
        const bool g = M.general(m);
        if (g)
            w.template stress<kIn, true>(m);
        else
            w.template stress<kIn, false>(m);
        if (m > kb) {
            if (M.general(m - 1))
                w.template finish_vz<true>(m - 1, ek);
            else
                w.template finish_vz<false>(m - 1, ek);
        }
        if (m + 1 < nz) w.publish(m + 1);
        lds_barrier();
        if (g)
            w.template velocity<true>(m, ek, ep);
        else
            w.template velocity<false>(m, ek, ep);
    }
    if (ke < nz) {
        march_load<kOwn, kAbove, HASX>(M, ke, w.L);
        w.template stress<kAbove, true>(ke);
    }
    w.template finish_vz<true>(ke - 1, ek);
}

// Both halo rows (lo, hi: whether the grid has them), with the own rows' barriers.
template <typename T, bool HASX>
__device__ __forceinline__ void march_halo(const March<T>& ML, const March<T>& MH, bool lo, bool hi)
{
    const int kb = ML.kb, ke = ML.ke, nz = ML.A.nz;
    Row<T, false, kLow, HASX> a(ML);
    Row<T, false, kHigh, HASX> b(MH);
    const int ms = kb > 0 ? kb - 1 : 0;
    if (lo) a.head(ms);
    if (hi) b.head(ms);
    b.vzm = 0;
    if (kb > 0) {
        if (lo) a.publish(ms);
        if (hi) b.publish(ms);
        lds_barrier();
        const auto z = b.vz;
        if (lo) a.head(kb);
        if (hi) b.head(kb);
        b.vzm = z;
    }
    if (lo) a.publish(kb);
    if (hi) b.publish(kb);
    lds_barrier();
    for (int m = kb; m < ke; ++m) {
        if (lo) march_load<kLow, kIn, HASX>(ML, m, a.L);
        if (hi) march_load<kHigh, kIn, HASX>(MH, m, b.L);
        if (lo) {
            if (ML.general(m))
                a.template stress<kIn, true>(m);
            else
                a.template stress<kIn, false>(m);
            if (m + 1 < nz) a.publish(m + 1);
        }
        if (hi) {
            if (MH.general(m))
                b.template stress<kIn, true>(m);
            else
                b.template stress<kIn, false>(m);
            if (m + 1 < nz) b.publish(m + 1);
        }
        lds_barrier();
    }
}

template <typename T, bool ENERGY, int NT, int WPE>
__global__ void __launch_bounds__(NT) __attribute__((amdgpu_waves_per_eu(WPE))) k_march(const StepArgs<T> A, const TailArgs<T> E)
{
    typedef typename Arith<T>::R R;
    extern __shared__ double march_smem[];
    const Box B = A.box[0];
    const int nx = A.nx, ny = A.ny;
    int chunk, zs;
    // A leading workgroup records the step before this one meanwhile (a tail kernel after every
    // step took 4 us: 64^3 18.0 -> 15.3 us a step, 101^3 37.8 -> 35.1).  Seven idle ones beside it
    // keep the others on the dies they would be on: moved by one die each, the two that march
    // through one strip no longer neighbour each other (401x401x301: 1176 -> 1207 us).
    if (blockIdx.x < kLead) {
        if (blockIdx.x > 0) return;
        const int done = *E.step;
        if (E.record) record_step(E, done, march_smem);
        if (threadIdx.x == 0) *E.step_out = done + 1;
        return;
    }
    const int nb = int(gridDim.x) - kLead, blk = turned(int(blockIdx.x) - kLead, nb, A.back);
    tile_of(B, xcd_block(blk, nb), chunk, zs);
    const int wave = __builtin_amdgcn_readfirstlane(int(threadIdx.x) >> 6);
    const MarchTile t = march_tile(nx, ny, A.rows, A.xch, A.xw, chunk);
    March<T> M{A};
    M.lds = reinterpret_cast<R*>(march_smem);
    M.slots = A.rows + 2;
    M.lane = int(threadIdx.x) & 63;
    segment_planes(B, zs, M.kb, M.ke);
    M.xs = t.xs;
    M.xe = t.xe;
    const int i = t.xs + M.lane, cx = layer_index(i, A.lo[0], A.hi[0]);
    M.own = i >= t.x0 && i < t.x1;
    M.inx = i < t.xe && cx >= 0;
    M.hasx = __ballot(M.inx) != 0;
    M.dt = scalar((R)A.dt); M.idx = scalar((R)A.idx); M.idy = scalar((R)A.idy); M.idz = scalar((R)A.idz);
    auto at_row = [&](March<T>& m, int slot) {
        m.slot = slot;
        m.j = t.j0 - 1 + slot;
        m.o0 = cell_offset(A.g0, A.nxyp, 0, m.j * nx + min(i, t.xe - 1));
        m.ox = m.inx ? xmem_offset(0, m.j, cx, ny, A.w[0]) : 0u;
        m.cy = layer_index(m.j, A.lo[1], A.hi[1]);
        m.edge = m.cy >= 0 || m.j == 0 || m.j == ny - 1;
    };
    at_row(M, wave + 1);
    // column tables of the chunk; a = 0, b = 1/K = 1 past the grid and where an update's
    // range ends (see xpml)
    {
        R* xt = M.lds + 2 * M.slots * kSlot;
        unsigned* xm = reinterpret_cast<unsigned*>(xt + kSlot);
        R* yt = xt + kSlot + 128;
        for (int q = int(threadIdx.x); q < 10 * 64; q += blockDim.x) {
            const int f = q / 64, c = t.xs + q % 64;
            if (f < 6) {
                const bool out = c >= nx || (f < 3 ? c == 0 : c == nx - 1);
                xt[q] = out ? (R)(f % 3 == 0 ? 0 : 1) : (R)A.tab[0][f * nx + c];
            } else if (f < 8) {
                xt[q] = (f == kCdtN ? c <= nx - 2 : c >= 1) ? M.dt : (R)0;
            } else {
                xm[q - kSlot] = ones(f == 8 ? !(A.dirichlet && (c == 0 || c == nx - 1))
                                            : c < t.xe && layer_index(c, A.lo[0], A.hi[0]) >= 0);
            }
        }
        // rows j0-1 .. and planes kb-1 .. ke
        for (int q = int(threadIdx.x); q < M.slots * 6; q += blockDim.x) {
            const int j = min(max(t.j0 - 1 + q / 6, 0), ny - 1);
            yt[q] = (R)A.tab[1][(q % 6) * ny + j];
        }
        for (int q = int(threadIdx.x); q < (M.ke - M.kb + 2) * 6; q += blockDim.x) {
            const int k = min(max(M.kb - 1 + q / 6, 0), A.nz - 1);
            yt[M.slots * 6 + q] = (R)A.tab[2][(q % 6) * A.nz + k];
        }
    }
    __syncthreads();
    double ek = 0.0, ep = 0.0;
    if (wave < t.n) {
        if (M.hasx)
            march_own<T, ENERGY, true>(M, ek, ep);
        else
            march_own<T, ENERGY, false>(M, ek, ep);
    } else if (wave == A.rows) {
        March<T> H = M;
        at_row(M, 0);
        at_row(H, t.n + 1);
        if (M.hasx)
            march_halo<T, true>(M, H, M.j >= 0, H.j < ny);
        else
            march_halo<T, false>(M, H, M.j >= 0, H.j < ny);
    } else {  // a wave without a row passes the workgroup's barriers
        const int nb = M.ke - M.kb + (M.kb > 0 ? 2 : 1);
        for (int q = 0; q < nb; ++q) lds_barrier();
    }
    if constexpr (ENERGY) {  // per-block FP64 partials, summed by whoever records the step (record_step)
        __shared__ double red[2][NT / 64];
        ek = wave_sum(ek);
        ep = wave_sum(ep);
        if (M.lane == 0) {
            red[0][wave] = ek;
            red[1][wave] = ep;
        }
        __syncthreads();
        if (threadIdx.x == 0) {
            double a = 0.0, b = 0.0;
            for (int q = 0; q < int(blockDim.x >> 6); ++q) {
                a += red[0][q];
                b += red[1][q];
            }
            A.epart[2 * blk] = a;
            A.epart[2 * blk + 1] = b;
        }
    }
    // the source, once its workgroup has stored every cell
    if (E.is >= t.x0 && E.is < t.x1 && E.js >= t.j0 && E.js < t.j0 + t.n && E.ks >= M.kb && E.ks < M.ke) {
        __syncthreads();
        if (threadIdx.x == 0) {
            for (int q = 0; q < 3; ++q) E.pre_out[q] = (double)E.f[q][E.src];
            inject_source(E, *E.step + 1, static_cast<float*>(nullptr));
        }
    }
}

template <typename T>
__global__ void __launch_bounds__(kMarchThreads) k_record(const TailArgs<T> E)
{
    __shared__ double red[2 * kMarchThreads / 64];
    record_step(E, *E.step, red);
}

}  // namespace

template <typename T>
void launch_march(const StepArgs<T>& a, const TailArgs<T>& tail, bool energy, hipStream_t s)
{
    constexpr int NT = kMarchThreads / (sizeof(T) / 4), WPE = sizeof(T) == 4 ? 6 : 4;
    const size_t lds = march_lds_bytes(int(sizeof(T)), a.rows, a.box[0].zseg);
    if (a.nblocks <= 0 || a.block != 64 * (a.rows + 1) || a.block > NT || lds > kMarchLds) return;  // refused on the host first
    if (energy)
        hipLaunchKernelGGL((k_march<T, true, NT, WPE>), dim3(a.nblocks + kLead), dim3(a.block), lds, s, a, tail);
    else
        hipLaunchKernelGGL((k_march<T, false, NT, WPE>), dim3(a.nblocks + kLead), dim3(a.block), lds, s, a, tail);
}
template <typename T>
void launch_record(const TailArgs<T>& a, int block, hipStream_t s)
{
    hipLaunchKernelGGL((k_record<T>), dim3(1), dim3(block), 0, s, a);
}
template void launch_march<float>(const StepArgs<float>&, const TailArgs<float>&, bool, hipStream_t);
template void launch_march<double>(const StepArgs<double>&, const TailArgs<double>&, bool, hipStream_t);
template void launch_record<float>(const TailArgs<float>&, int, hipStream_t);
template void launch_record<double>(const TailArgs<double>&, int, hipStream_t);

}  // namespace ela3d
