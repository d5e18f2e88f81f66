// kernels.hip -- HIP kernels of one MHIT36 timestep for gfx950 (CDNA4).
//
// Fields are N^3 FP64 arrays, x fastest, periodic in all three directions by
// index wrap (the y/z halo planes of the reference's X-pencils hold periodic
// copies at a 1x1 decomposition, so wrap reads the same values).  Every
// expression is evaluated in the order the reference's Fortran writes it
// (multi/main.f90), and the library is compiled with -ffp-contract=off.
#include "internal.h"
#include "devmath.h"

#include <mutex>
#include <type_traits>

namespace mhit {

#define IDX(i, j, k) ((size_t)(i) + (size_t)n * ((size_t)(j) + (size_t)n * (size_t)(k)))

constexpr int BLK = 256;

// A kernel of a halted run writes nothing.  The FFT passes, the projection and
// the sums read the flag at the start and test it just before the first store,
// so that no load waits for it: 0.2-0.4 us of a 64^3 box's 4 to 7 us kernels.
// (The marching passes gain nothing by it and their main loops compile worse.)
__device__ __forceinline__ bool halted(const Scalars *sc) { return sc->halted != 0; }

static inline unsigned nblocks(size_t work, int blk) { return (unsigned)((work + blk - 1) / blk); }

// Workgroups are dispatched round-robin over the 8 XCDs, each with its own L2.
// Renumber them so that XCD x works on the x-th contiguous eighth of the grid:
// neighbouring tiles, which share halo cells, then meet in the same L2.
__device__ __forceinline__ uint3 xcd_block()
{
    const unsigned gx = gridDim.x, gy = gridDim.y, gz = gridDim.z;
    const unsigned nb = gx * gy * gz;
    unsigned b = blockIdx.x + gx * (blockIdx.y + gy * blockIdx.z);
    if (nb % 8 == 0) b = (b % 8) * (nb / 8) + b / 8;
    return make_uint3(b % gx, (b / gx) % gy, b / (gx * gy));
}

// ---------------------------------------------------------------------------
// Phase field, main.f90:338-486, fused into one pass.
//
// A block owns an ATX x ATY column of cells and marches kz planes in z; thread
// t owns the cell (t % ATX, t / ATX) of the tile in every plane.  What a cell
// needs from its own column (psi at k-1..k+1 for the z part of the normal, phi
// at k-1..k+1, the z sharpening flux at k-1 and k+1) stays in the owning
// thread's registers; only what x/y neighbours share goes through LDS, one
// plane of each, double-buffered by plane parity:
//   psi on the tile plus a 2-cell ring (the 12 outer corners are never
//   read), for the x/y parts of the normal;
//   s_x, s_y of the sharpening flux s = a*n (a = 0.25(1 -
//   tanh^2(psi/(2 eps))), n the normalised undivided normal) on the tile plus
//   a 1-cell ring without corners, for the flux divergence;
//   phi on the same cells, for the convective and diffusive stencils.
// The ring cells are extra work items: the 96 cells of the 1-cell ring (psi,
// the normal and s_x or s_y) go to threads HS0.., the 100 further psi-only
// cells to threads HP0..; each such thread keeps its ring cell's column in
// registers the way it keeps its own.
// Iteration k: psi(k+2) from phi loaded one iteration earlier; s(k+1); the
// output plane k: convective and diffusive terms, the sharpening
// divergence and phi^{n+1} = phi + dt*rhs written to a second buffer;
// then psi(k+2) and phi(k+1) into LDS, and one barrier.  u, v of plane k+1, w
// of plane k+2 and phi of plane k+3 are loaded at the start of iteration k, a
// whole iteration ahead of their use.  HBM traffic:
// u, v, w, phi read once (plus halos), phi^{n+1} written once; psi and s
// never leave the chip.
// ---------------------------------------------------------------------------
constexpr int ATX = 32, ATY = 16;
constexpr int APX = ATX + 4, APY = ATY + 4;       // psi box
constexpr int ASX = ATX + 2, ASY = ATY + 2;       // s / phi box
constexpr int ATHREADS = ATX * ATY;
constexpr int NHS = 2 * ATY + 2 * ATX;            // 1-cell ring without corners: psi, normal, s_x or s_y
constexpr int NHP = 4 + 2 * ATY + 2 * ATX;        // its 4 corners and the 2-cell ring's sides: psi only
constexpr int HS0 = ATHREADS / 2, HP0 = 3 * ATHREADS / 4;   // first thread of each ring's work
static_assert(HS0 + NHS <= HP0 && HP0 + NHP <= ATHREADS, "one ring cell per thread at most");

__device__ __forceinline__ int wrap(int a, int n) { a %= n; return a < 0 ? a + n : a; }
// The same for an index less than one period outside.
__device__ __forceinline__ int wrap_once(int a, int n) { return a < 0 ? a + n : a >= n ? a - n : a; }

// FP64: the project's own table-driven log (bit-identical to the oracle;
// `tab` is the block's LDS copy of the table) and IEEE division.  FP32 (the
// mixed-precision pass, compared with FP64 by tolerance): the hardware log2
// and sqrt approximations (v_log_f32, v_sqrt_f32) and quotients as a product
// with the hardware reciprocal (v_rcp_f32): a few ulp of FP32, far below the
// FP32 storage error of the state, in 1-2 instructions where the correctly
// rounded forms take 8-10.  (HIP's __logf and __fdividef are the correctly
// rounded forms unless fast math is on.)  The arguments are positive normal
// numbers or moderate in size: log's is (phi + 1e-16) / (1 - phi + 1e-16)
// for phi clamped to [0, 1], the divisor |grad psi| + 1e-16.
__device__ __forceinline__ double tlog(double x, const double *tab) { return dlog(x, tab); }
__device__ __forceinline__ float tlog(float x, const double *)
{
    return __builtin_amdgcn_logf(x) * 0.6931471805599453f;       // log2(x) ln 2
}
__device__ __forceinline__ double tdiv(double a, double b) { return a / b; }
__device__ __forceinline__ float tdiv(float a, float b) { return a * __builtin_amdgcn_rcpf(b); }
__device__ __forceinline__ double tsqrt(double x) { return __builtin_sqrt(x); }
__device__ __forceinline__ float tsqrt(float x) { return __builtin_amdgcn_sqrtf(x); }

// Tile coordinates (x in -2..ATX+1, y in -2..ATY+1) of ring work item h:
// s ring (S) or psi-only ring (P).
__device__ __forceinline__ int2 ring_s_cell(int h)
{
    if (h < ATY) return make_int2(-1, h);
    if (h < 2 * ATY) return make_int2(ATX, h - ATY);
    if (h < 2 * ATY + ATX) return make_int2(h - 2 * ATY, -1);
    return make_int2(h - 2 * ATY - ATX, ATY);
}
__device__ __forceinline__ int2 ring_p_cell(int h)
{
    if (h < 4) return make_int2((h & 1) ? ATX : -1, (h & 2) ? ATY : -1);
    h -= 4;
    if (h < ATY) return make_int2(-2, h);
    if (h < 2 * ATY) return make_int2(ATX + 1, h - ATY);
    if (h < 2 * ATY + ATX) return make_int2(h - 2 * ATY, -2);
    return make_int2(h - 2 * ATY - ATX, ATY + 1);
}

// base[off] with a 32-bit byte offset (off * sizeof(T) < 2^32): the load takes
// the uniform base in scalar registers and the offset in one vector register.
template <typename T>
__device__ __forceinline__ T ld_off(const T *base, unsigned off)
{
    return *reinterpret_cast<const T *>(reinterpret_cast<const char *>(base) + off * (unsigned)sizeof(T));
}
template <typename T>
__device__ __forceinline__ T *at_off(T *base, unsigned off)
{
    return reinterpret_cast<T *>(reinterpret_cast<char *>(base) + off * (unsigned)sizeof(T));
}

// psi = eps log(phi / (1 - phi))
template <typename T>
__device__ __forceinline__ T acdi_psi(T f, T eps, T en, const double *tab)
{
    T val = f < (T)1.0 ? f : (T)1.0;
    if constexpr (sizeof(T) == 4) val = val > (T)0.0 ? val : (T)0.0;   // FP32 phi: no log of a negative
    return eps * tlog(tdiv(val + en, ((T)1.0 - val) + en), tab);
}
// The sharpening flux a(psi) n at a cell: g* the undivided gradient of psi, pc0
// psi and f phi at the cell.  The factor 1/4 (1 - tanh^2(psi/(2 eps))) of the flux
// comes from the cell's phi, no tanh: psi = eps log(A/B), A = val + enum,
// B = (1 - val) + enum, so it is A B / (A + B)^2 exactly (and, like the
// tanh form, goes to 0 with A as phi nears -enum).  A NaN psi (phi below
// -enum) stays NaN, as tanh(NaN) would.
template <typename T>
__device__ __forceinline__ void acdi_flux(T gx, T gy, T gz, T pc0, T f, T en, T tiny, T &sx, T &sy, T &sz)
{
    T normod = tdiv((T)1.0, tsqrt((gx * gx + gy * gy) + gz * gz) + tiny);
    T val = f < (T)1.0 ? f : (T)1.0;
    if constexpr (sizeof(T) == 4) val = val > (T)0.0 ? val : (T)0.0;   // as psi's FP32 clamp
    const T A = val + en, B = ((T)1.0 - val) + en, S = A + B;
    const T a = pc0 != pc0 ? pc0 : tdiv(A * B, S * S);
    sx = a * (gx * normod);
    sy = a * (gy * normod);
    sz = a * (gz * normod);
}
// phi^{n+1} at a cell: phi there (f0) and at its neighbours, the velocity at the
// cell's faces and the differences of the flux components over two cells.  The
// expressions of the march's output stencil, which has them in place: through
// this function its FP64 form spills 20 values instead of 14 (512^3: 1.59 against
// 1.44 ms).
template <typename T>
__device__ __forceinline__ T acdi_advance(T f0, T fxp, T fxm, T fyp, T fym, T fzp, T fzm, T uip, T u0, T vjp, T v0,
                                          T wkp, T w0, T dsx, T dsy, T dsz, T gamma, T eps, T dxi, T ddxi, T dt)
{
    if constexpr (sizeof(T) == 4) {
        const T hd = (T)0.5 * dxi;
        const T A = __builtin_fmaf(uip, fxp + f0, -(u0 * (f0 + fxm)));
        const T B = __builtin_fmaf(vjp, fyp + f0, -(v0 * (f0 + fym)));
        const T C = __builtin_fmaf(wkp, fzp + f0, -(w0 * (f0 + fzm)));
        const T lap = ((fxp + fxm) + (fyp + fym)) + __builtin_fmaf((T)-6.0, f0, fzp + fzm);
        const T sdiv = (dsx + dsy) + dsz;
        const T r2 = __builtin_fmaf(gamma * eps * ddxi, lap, -hd * (((A + B) + C) + gamma * sdiv));
        return __builtin_fmaf(dt, r2, f0);
    } else {
        T A = uip * (T)0.5 * (fxp + f0) - u0 * (T)0.5 * (f0 + fxm);
        T B = vjp * (T)0.5 * (fyp + f0) - v0 * (T)0.5 * (f0 + fym);
        T C = wkp * (T)0.5 * (fzp + f0) - w0 * (T)0.5 * (f0 + fzm);
        T r = (-(A * dxi) - B * dxi) - C * dxi;
        T dxx = eps * ((fxp - (T)2.0 * f0) + fxm) * ddxi;
        T dyy = eps * ((fyp - (T)2.0 * f0) + fym) * ddxi;
        T dzz = eps * ((fzp - (T)2.0 * f0) + fzm) * ddxi;
        T rphi = r + gamma * ((dxx + dyy) + dzz);
        T X = dsx * (T)0.5 * dxi;
        T Y = dsy * (T)0.5 * dxi;
        T Z = dsz * (T)0.5 * dxi;
        T r2 = rphi - gamma * ((X + Y) + Z);
        return f0 + dt * r2;
    }
}

// MARCH3: the march unrolled by three planes (the one-box FP64 pass); else
// one plane per iteration with the registers copied forward (FP32, and the
// gang pass, whose per-box addressing would not fit the unrolled march in 128
// VGPRs).
template <typename T, bool MARCH3 = (sizeof(T) == 8)>
__device__ __forceinline__ void k_acdi_body(uint3 blk,
    const T *__restrict__ u, const T *__restrict__ v, const T *__restrict__ w,
    const T *__restrict__ phi, T *__restrict__ phin, const Scalars *__restrict__ sc, const double *__restrict__ mtab,
    Consts c, int kz)
{
    if (halted(sc)) return;
    constexpr int NTAB = sizeof(T) == 8 ? TAB_LHI + 2 * 129 : 1;   // the log part of the table
    __shared__ double tabL[NTAB];
    __shared__ T psiL[2][APY * APX];
    __shared__ T sxL[2][ASY * ASX];
    __shared__ T syL[2][ASY * ASX];
    __shared__ T phL[2][ASY * ASX];
    const int n = c.n;
    const int tid = threadIdx.x;
    const int i0 = blk.x * ATX, j0 = blk.y * ATY, k0 = blk.z * kz;
    const T eps = c.eps, en = c.enumr, dxi = c.dxi, ddxi = c.ddxi;
    const T um = sc->umean, vm = sc->vmean, wm = sc->wmean;
    const T gamma = c.gamma_factor * sc->gumax;
    const T tiny = (T)1.0E-16f;
    const size_t nn = (size_t)n * n;

    // own cell
    const int tx = tid % ATX, ty = tid / ATX;
    const int i = i0 + tx, j = j0 + ty;
    const bool active = (i < n) && (j < n);
    // in-plane offsets (< n^2): the plane's base address is uniform, so loads
    // take a scalar base and a 32-bit vector offset
    const unsigned own = (unsigned)wrap(i, n) + (unsigned)n * (unsigned)wrap(j, n);   // ghost cells wrap
    const int pI = (ty + 2) * APX + (tx + 2), sI = (ty + 1) * ASX + (tx + 1);
    // ring cell: kind 1 = s ring with s_x, 2 = s ring with s_y, 3 = psi only
    int hk = 0;
    int2 hc = make_int2(0, 0);
    if (tid >= HS0 && tid < HS0 + NHS) { hk = tid - HS0 < 2 * ATY ? 1 : 2; hc = ring_s_cell(tid - HS0); }
    else if (tid >= HP0 && tid < HP0 + NHP) { hk = 3; hc = ring_p_cell(tid - HP0); }
    const unsigned hoff = (unsigned)wrap(i0 + hc.x, n) + (unsigned)n * (unsigned)wrap(j0 + hc.y, n);
    const int hP = (hc.y + 2) * APX + (hc.x + 2), hS = (hc.y + 1) * ASX + (hc.x + 1);

    auto ld_phi = [&](unsigned off, int m) { return ld_off(phi + nn * (size_t)wrap(m, n), off); };
    auto psi_of = [&](T f) { return acdi_psi(f, eps, en, tabL); };
    auto sharp = [&](T gx, T gy, T gz, T pc0, T f, T &sx, T &sy, T &sz) {
        acdi_flux(gx, gy, gz, pc0, f, en, tiny, sx, sy, sz);
    };

    if constexpr (sizeof(T) == 8) {
        for (int q = tid; q < NTAB; q += ATHREADS) tabL[q] = mtab[q];
        __syncthreads();
    }

    // Column registers of the march.  It is unrolled by three planes, and each
    // register's role (plane - k) is a compile-time index into a 3-element
    // array, so planes rotate through the registers without copies: a copy of
    // a register that a load is still filling would wait for that load, and
    // cap every load's lead at the end of the iteration that issued it.
    //   fr: phi of the own cell, hr: of the ring cell (planes not yet in LDS);
    //   zr: z flux of the own cell; U: u, u(x+1), v, v(y+1) of a plane and w
    //   of the plane above it (two planes live: the output plane and the next,
    //   in flight); wk: w of the output plane.
    // psi(k), psi(k+1) and phi(k-1), phi(k) of a thread's own cells are read
    // back from the LDS slots it wrote itself.  Every thread issues every load
    // of a plane (the offsets wrap, so a thread outside the box or without a
    // ring cell reads a valid cell it does not use): the count of loads per
    // plane is then fixed, and a wait for one plane's data leaves the later
    // planes' loads in flight.
    T fr[3] = {0, 0, 0}, hr[3] = {0, 0, 0}, zr[3] = {0, 0, 0};
    T U[3][5] = {};
    T wk = 0;
    const int kend = min(k0 + kz, n);
    // the x+1 and y+1 neighbours of the own cell, as offsets from it (periodic)
    const unsigned xpo = (unsigned)wrap(i + 1, n) + (unsigned)n * (unsigned)wrap(j, n);
    const unsigned ypo = (unsigned)wrap(i, n) + (unsigned)n * (unsigned)wrap(j + 1, n);
    // u, v of plane m < n and w of plane m+1 into the registers of one plane
    auto fetch_uvw = [&](int m, T (&d)[5]) {
        // the plane offsets are opaque: otherwise the compiler hoists base +
        // own out of the march as 64-bit vector pointers, which spill
        size_t z = nn * (size_t)m, zp = nn * (size_t)(m + 1 == n ? 0 : m + 1);
        asm volatile("" : "+s"(z), "+s"(zp));
        const T *up = u + z, *vp = v + z;
        d[0] = ld_off(up, own); d[1] = ld_off(up, xpo);
        d[2] = ld_off(vp, own); d[3] = ld_off(vp, ypo);
        d[4] = ld_off(w + zp, own);
    };

    // prologue: psi(k0-1), psi(k0) in LDS -> z flux of k0-1, s(k0), phi(k0-1),
    // phi(k0) in LDS -> psi(k0+1) in LDS; the registers in the roles of the
    // march's first plane.
    {
        const T fm2 = ld_phi(own, k0 - 2), fm1 = ld_phi(own, k0 - 1), f0 = ld_phi(own, k0);
        fr[1] = ld_phi(own, k0 + 1); fr[2] = ld_phi(own, k0 + 2);
        T hfm1 = 0, hf0 = 0;
        if (hk) {
            hfm1 = ld_phi(hoff, k0 - 1); hf0 = ld_phi(hoff, k0); hr[1] = ld_phi(hoff, k0 + 1);
            hr[2] = ld_phi(hoff, k0 + 2);
        }
        wk = ld_off(w + nn * (size_t)k0, own);
        fetch_uvw(k0, U[0]);
        const T qm2 = psi_of(fm2), qm1 = psi_of(fm1), q0 = psi_of(f0), qp1 = psi_of(fr[1]);
        T hqm1 = 0, hq0 = 0, hqp1 = 0;
        if (hk) { hqm1 = psi_of(hfm1); hq0 = psi_of(hf0); hqp1 = psi_of(hr[1]); }
        const int sm1 = (k0 - 1) & 1, s0 = k0 & 1;
        psiL[sm1][pI] = qm1; psiL[s0][pI] = q0;
        if (hk) { psiL[sm1][hP] = hqm1; psiL[s0][hP] = hq0; }
        __syncthreads();
        T sx, sy;
        sharp(psiL[sm1][pI + 1] - psiL[sm1][pI - 1], psiL[sm1][pI + APX] - psiL[sm1][pI - APX], q0 - qm2, qm1,
              fm1, sx, sy, zr[0]);
        sharp(psiL[s0][pI + 1] - psiL[s0][pI - 1], psiL[s0][pI + APX] - psiL[s0][pI - APX], qp1 - qm1, q0, f0,
              sx, sy, zr[1]);
        sxL[s0][sI] = sx; syL[s0][sI] = sy;
        phL[s0][sI] = f0; phL[sm1][sI] = fm1;
        if (hk == 1 || hk == 2) {
            T hx, hy, hz;
            sharp(psiL[s0][hP + 1] - psiL[s0][hP - 1], psiL[s0][hP + APX] - psiL[s0][hP - APX], hqp1 - hqm1, hq0,
                  hf0, hx, hy, hz);
            if (hk == 1) sxL[s0][hS] = hx; else syL[s0][hS] = hy;
            phL[s0][hS] = hf0;
        }
        __syncthreads();
        psiL[sm1][pI] = qp1;                 // the slot of plane k0+1
        if (hk) psiL[sm1][hP] = hqp1;
        __syncthreads();
    }

    // Output plane k, the march's plane R0 of three.  Roles: fr/hr [R1] phi(k+1),
    // [R2] phi(k+2), [R0] <- phi(k+3); zr [R0] flux(k-1), [R1] flux(k),
    // [R2] <- flux(k+1); U[R0] plane k, U[R1] <- plane k+1.
    auto plane = [&](auto PHC, int k) {
        constexpr int R0 = decltype(PHC)::value, R1 = (R0 + 1) % 3, R2 = (R0 + 2) % 3;
        const T f_p1 = fr[R1], f_p2 = fr[R2], hf_p1 = hr[R1], hf_p2 = hr[R2];
        const T z_m1 = zr[R0];
        const int s0 = k & 1, s1 = (k + 1) & 1;
        // phi(k+3) (psi of the next plane waits for it), psi(k+2), then u, v, w
        // of the next output plane (issued after psi: fewer registers live
        // through it)
        fr[R0] = ld_phi(own, k + 3);
        hr[R0] = ld_phi(hoff, k + 3);
        const T q_p2 = psi_of(f_p2);
        T hq_p2 = 0;
        if (hk) hq_p2 = psi_of(hf_p2);
        fetch_uvw(min(k + 1, n - 1), U[R1]);  // the next output plane (past the slab: unused)
        const T nu0 = U[R0][0], nuxp = U[R0][1], nv0 = U[R0][2], nvyp = U[R0][3], nwp = U[R0][4], nw0 = wk;
        // s(k+1): x/y parts of the normal from psi(k+1) in LDS, z part from the
        // column (psi(k) from the own slot, psi(k+2) just formed)
        T sx, sy, z_p1;
        sharp(psiL[s1][pI + 1] - psiL[s1][pI - 1], psiL[s1][pI + APX] - psiL[s1][pI - APX], q_p2 - psiL[s0][pI],
              psiL[s1][pI], f_p1, sx, sy, z_p1);
        zr[R2] = z_p1;
        sxL[s1][sI] = sx; syL[s1][sI] = sy;
        if (hk == 1 || hk == 2) {
            T hx, hy, hz;
            sharp(psiL[s1][hP + 1] - psiL[s1][hP - 1], psiL[s1][hP + APX] - psiL[s1][hP - APX],
                  hq_p2 - psiL[s0][hP], psiL[s1][hP], hf_p1, hx, hy, hz);
            if (hk == 1) sxL[s1][hS] = hx; else syL[s1][hS] = hy;
        }
        // the output plane k
        if (active) {
            const T f0 = phL[s0][sI];
            T fxp = phL[s0][sI + 1], fxm = phL[s0][sI - 1];
            T fyp = phL[s0][sI + ASX], fym = phL[s0][sI - ASX];
            T fzp = f_p1, fzm = phL[s1][sI];
            const T wkp_raw = nwp;
            T uip = nuxp - um, u0 = nu0 - um;
            T vjp = nvyp - vm, v0 = nv0 - vm;
            T wkp = wkp_raw - wm, w0 = nw0 - wm;
            if constexpr (sizeof(T) == 4) {
                // FP32 (mixed precision, held to the FP64 result by tolerance):
                // the same discretisation with the constant factors gathered
                // and fused multiply-adds, about half the instructions of the
                // operand-by-operand form below.
                const T hd = (T)0.5 * dxi;
                const T A = __builtin_fmaf(uip, fxp + f0, -(u0 * (f0 + fxm)));
                const T B = __builtin_fmaf(vjp, fyp + f0, -(v0 * (f0 + fym)));
                const T C = __builtin_fmaf(wkp, fzp + f0, -(w0 * (f0 + fzm)));
                const T lap = ((fxp + fxm) + (fyp + fym)) + __builtin_fmaf((T)-6.0, f0, fzp + fzm);
                const T sdiv = ((sxL[s0][sI + 1] - sxL[s0][sI - 1]) + (syL[s0][sI + ASX] - syL[s0][sI - ASX])) +
                               (z_p1 - z_m1);
                const T r2 = __builtin_fmaf(gamma * eps * ddxi, lap, -hd * (((A + B) + C) + gamma * sdiv));
                __builtin_nontemporal_store(__builtin_fmaf((T)c.dt, r2, f0), at_off(phin + nn * (size_t)k, own));
            } else {
                T A = uip * (T)0.5 * (fxp + f0) - u0 * (T)0.5 * (f0 + fxm);
                T B = vjp * (T)0.5 * (fyp + f0) - v0 * (T)0.5 * (f0 + fym);
                T C = wkp * (T)0.5 * (fzp + f0) - w0 * (T)0.5 * (f0 + fzm);
                T r = (-(A * dxi) - B * dxi) - C * dxi;
                T dxx = eps * ((fxp - (T)2.0 * f0) + fxm) * ddxi;
                T dyy = eps * ((fyp - (T)2.0 * f0) + fym) * ddxi;
                T dzz = eps * ((fzp - (T)2.0 * f0) + fzm) * ddxi;
                T rphi = r + gamma * ((dxx + dyy) + dzz);
                T X = (sxL[s0][sI + 1] - sxL[s0][sI - 1]) * (T)0.5 * dxi;
                T Y = (syL[s0][sI + ASX] - syL[s0][sI - ASX]) * (T)0.5 * dxi;
                T Z = (z_p1 - z_m1) * (T)0.5 * dxi;
                T r2 = rphi - gamma * ((X + Y) + Z);
                __builtin_nontemporal_store(f0 + (T)c.dt * r2, at_off(phin + nn * (size_t)k, own));
            }
        }
        // psi(k+2) and phi(k+1) for the x/y neighbours of the next plane
        psiL[s0][pI] = q_p2;
        phL[s1][sI] = f_p1;
        if (hk) psiL[s0][hP] = hq_p2;
        if (hk == 1 || hk == 2) phL[s1][hS] = hf_p1;
        wk = nwp;
        __syncthreads();
    };
    if constexpr (MARCH3) {
        for (int k = k0; k < kend; k += 3) {
            plane(std::integral_constant<int, 0>(), k);
            if (k + 1 < kend) plane(std::integral_constant<int, 1>(), k + 1);
            if (k + 2 < kend) plane(std::integral_constant<int, 2>(), k + 2);
        }
    } else {
        // one plane per iteration with the roles fixed and the registers copied
        // forward (FP32: within the 64 VGPRs of eight waves per SIMD, where
        // the three-plane form spills)
        for (int k = k0; k < kend; k++) {
            plane(std::integral_constant<int, 0>(), k);
            fr[1] = fr[2]; fr[2] = fr[0];
            hr[1] = hr[2]; hr[2] = hr[0];
            zr[0] = zr[1]; zr[1] = zr[2];
#pragma unroll
            for (int q = 0; q < 5; q++) U[0][q] = U[1][q];
        }
    }
}

// FP32: 8 waves per SIMD (63 VGPRs).  FP64: held to the 128 VGPRs of 4 waves
// per SIMD (two blocks per CU), with 14 spills by the compiler's count, in 12
// bytes of scratch per lane.  Held to the 80 VGPRs of
// 6 waves (three blocks, which the 44 KB of LDS would allow) the pass spills
// in the march and runs 2.3x slower.
template <typename T>
__global__ void __launch_bounds__(ATHREADS, sizeof(T) == 4 ? 8 : 4) k_acdi(
    const T *__restrict__ u, const T *__restrict__ v, const T *__restrict__ w,
    const T *__restrict__ phi, T *__restrict__ phin, const Scalars *__restrict__ sc, const double *__restrict__ mtab,
    Consts c, int kz)
{
    k_acdi_body<T>(xcd_block(), u, v, w, phi, phin, sc, mtab, c, kz);
}


// ---------------------------------------------------------------------------
// The phase field of a small box, where a march of a few planes is bound by its
// serial chain (four planes of psi before the first output, 1.6 us per plane):
// a block owns BTX x BTY x BTZ cells, forms psi on them and two cells around,
// then the flux on them and the face neighbours, then the output: three steps
// with a barrier between, in exchange for psi at 3 cells per cell instead of
// 1.4 plus the prologue.  March / box, us (event times): FP64 32^3 12.0 / 8.5,
// 64^3 12.8 / 11.6, 72^3 22.3 / 17.8, 96^3 22.7 / 25.2; FP32 32^3 8.5 / 6.7,
// 72^3 12.2 / 11.4, 96^3 12.9 / 15.3: used up to 72^3.
// ---------------------------------------------------------------------------
constexpr int BTX = 16, BTY = 8, BTZ = 4, BTHREADS = BTX * BTY * BTZ;
constexpr int BPX = BTX + 4, BPY = BTY + 4, BPZ = BTZ + 4, BPSI = BPX * BPY * BPZ;
constexpr int BRX = 2 * BTY * BTZ, BRY = 2 * BTX * BTZ, BRZ = 2 * BTX * BTY;      // face neighbours
static_assert(BRX + BRY + BRZ <= BTHREADS, "one face neighbour per thread at most");

template <typename T>
__global__ void __launch_bounds__(BTHREADS) k_acdi_box(
    const T *__restrict__ u, const T *__restrict__ v, const T *__restrict__ w,
    const T *__restrict__ phi, T *__restrict__ phin, const Scalars *__restrict__ sc, const double *__restrict__ mtab,
    Consts c)
{
    constexpr int NTAB = sizeof(T) == 8 ? TAB_LHI + 2 * 129 : 1, Q = (BPSI + BTHREADS - 1) / BTHREADS;
    static_assert(NTAB <= BTHREADS, "one table entry per thread");
    __shared__ double tabL[NTAB];
    __shared__ T psiL[BPSI], phL[BPSI];
    __shared__ T sxL[BTZ * BTY * (BTX + 2)], syL[BTZ * (BTY + 2) * BTX], szL[(BTZ + 2) * BTY * BTX];
    const bool stop = halted(sc);
    const int n = c.n, tid = threadIdx.x;
    const int i0 = blockIdx.x * BTX, j0 = blockIdx.y * BTY, k0 = blockIdx.z * BTZ;
    const T eps = c.eps, en = c.enumr, dxi = c.dxi, ddxi = c.ddxi, tiny = (T)1.0E-16f;
    const T um = sc->umean, vm = sc->vmean, wm = sc->wmean, gamma = c.gamma_factor * sc->gumax;
    const unsigned nn = (unsigned)n * n;
    // a tile reaches BTX + 1 past its first cell: below 2n from n = 18 on
    auto per = [&](int a) { return n >= BTX + 2 ? wrap_once(a, n) : wrap(a, n); };
    auto off = [&](int x, int y, int z) {
        return (unsigned)per(i0 + x) + (unsigned)n * (unsigned)per(j0 + y) + nn * (unsigned)per(k0 + z);
    };
    // this thread's cell, and every load of the pass
    const int x = tid % BTX, y = tid / BTX % BTY, z = tid / (BTX * BTY);
    const unsigned own = off(x, y, z);
    const T u0 = ld_off(u, own), v0 = ld_off(v, own), w0 = ld_off(w, own);
    const T uip = ld_off(u, off(x + 1, y, z)), vjp = ld_off(v, off(x, y + 1, z)), wkp = ld_off(w, off(x, y, z + 1));
    T f[Q];
    bool need[Q];
#pragma unroll
    for (int q = 0; q < Q; q++) {
        const int e = tid + q * BTHREADS, px = e % BPX - 2, py = e / BPX % BPY - 2, pz = e / (BPX * BPY) - 2;
        // psi is read up to two cells away in all: face neighbours of the face neighbours
        const int d = max(max(-px, px - (BTX - 1)), 0) + max(max(-py, py - (BTY - 1)), 0) + max(max(-pz, pz - (BTZ - 1)), 0);
        need[q] = e < BPSI && d <= 2;
        f[q] = need[q] ? ld_off(phi, off(px, py, pz)) : (T)0.0;
    }
    if constexpr (sizeof(T) == 8) {
        if (tid < NTAB) tabL[tid] = mtab[tid];
        __syncthreads();
    }
#pragma unroll
    for (int q = 0; q < Q; q++)
        if (need[q]) {
            psiL[tid + q * BTHREADS] = acdi_psi(f[q], eps, en, tabL);
            phL[tid + q * BTHREADS] = f[q];
        }
    __syncthreads();
    auto at = [&](int a, int b, int d) { return a + 2 + BPX * (b + 2 + BPY * (d + 2)); };
    auto flux = [&](int e, T &sx, T &sy, T &sz) {
        acdi_flux(psiL[e + 1] - psiL[e - 1], psiL[e + BPX] - psiL[e - BPX], psiL[e + BPX * BPY] - psiL[e - BPX * BPY],
                  psiL[e], phL[e], en, tiny, sx, sy, sz);
    };
    const int e0 = at(x, y, z);
    {
        T sx, sy, sz;
        flux(e0, sx, sy, sz);
        sxL[x + 1 + (BTX + 2) * (y + BTY * z)] = sx;
        syL[x + BTX * (y + 1 + (BTY + 2) * z)] = sy;
        szL[x + BTX * (y + BTY * (z + 1))] = sz;
    }
    if (tid < BRX + BRY + BRZ) {
        int h = tid;
        T sx, sy, sz;
        if (h < BRX) {
            const int a = h & 1 ? BTX : -1, b = (h >> 1) % BTY, d = (h >> 1) / BTY;
            flux(at(a, b, d), sx, sy, sz);
            sxL[a + 1 + (BTX + 2) * (b + BTY * d)] = sx;
        } else if (h < BRX + BRY) {
            h -= BRX;
            const int b = h & 1 ? BTY : -1, a = (h >> 1) % BTX, d = (h >> 1) / BTX;
            flux(at(a, b, d), sx, sy, sz);
            syL[a + BTX * (b + 1 + (BTY + 2) * d)] = sy;
        } else {
            h -= BRX + BRY;
            const int d = h & 1 ? BTZ : -1, a = (h >> 1) % BTX, b = (h >> 1) / BTX;
            flux(at(a, b, d), sx, sy, sz);
            szL[a + BTX * (b + BTY * (d + 1))] = sz;
        }
    }
    __syncthreads();
    if (stop || i0 + x >= n || j0 + y >= n || k0 + z >= n) return;
    const int ex = x + 1 + (BTX + 2) * (y + BTY * z), ey = x + BTX * (y + 1 + (BTY + 2) * z),
              ez = x + BTX * (y + BTY * (z + 1));
    const T r = acdi_advance(phL[e0], phL[e0 + 1], phL[e0 - 1], phL[e0 + BPX], phL[e0 - BPX], phL[e0 + BPX * BPY],
                             phL[e0 - BPX * BPY], uip - um, u0 - um, vjp - vm, v0 - vm, wkp - wm, w0 - wm,
                             sxL[ex + 1] - sxL[ex - 1], syL[ey + BTX] - syL[ey - BTX], szL[ez + BTX * BTY] - szL[ez - BTX * BTY],
                             gamma, eps, dxi, ddxi, (T)c.dt);
    __builtin_nontemporal_store(r, at_off(phin, own));
}


// ---------------------------------------------------------------------------
// Momentum, main.f90:513-681: convection, viscous term, ABC forcing,
// CSF force (phi^{n+1}) interpolated to the faces, AB2/Euler advance
// and rhs_o <- rhs, in one pass.
//
// A block owns an MTX x MTY column and marches kz planes in z.  LDS rings hold
// u, v, w on an (MTX+2) x (MTY+2) box and phi on an (MTX+3) x (MTY+3) box,
// three planes each, so every input is read from memory once per block (plus
// the halo).  What a point needs of plane k-1 (its u, v, w, u(i+1), v(j+1), its
// phi and the z force) it has seen at that plane and keeps in registers, so
// the slot of plane k-1 is free for the plane being stored and one barrier a
// plane is enough.  A thread forms the CSF force of its own cell, and MTX + MTY
// threads one of the cells before the tile in x or y too; the face averages
// take the neighbour's part from the lane before (x) or from LDS (y).
// Bound by memory: 13 values a point.  512 threads, because a taller tile reads
// less halo (rows of u: 18/16 instead of 10/8) and with one barrier the two
// blocks of a CU still cover each other's waits.  256^3 and 512^3 with phi:
// 394 and 3056 us (8 rows, two barriers a plane) -> 360 and 2907 (8 rows, one
// barrier) -> 348 and 2730 (16 rows; 2490-2820 at 512^3 on other boxes); 351 and
// 2742 with 32 rows.  128 VGPRs with phi, 2 values spilled.  Without phi:
// 345 and 2588 -> 325 and 2638 -> 308 and 2435.  13 (12) values at the 5.4 TB/s
// of a large copy are 2585 (2390) us at 512^3.
// ---------------------------------------------------------------------------
template <typename T>
struct MomK {
    T dxi, ddxi, mu, rhoi, f1, f2, f3, dt, alpha, beta;
};

// The momentum point, main.f90:513-696.  U0..W0: plane
// k, Up..Wp: plane k+1, with row stride SX; uzm..wzm, uxpm (u at k-1, i+1)
// and vypm (v at k-1, j+1) from plane k-1; FX/FY/FZ the force of plane k and
// fzm its z part at plane k-1 (row stride FXS).
template <int PHI, int SX, int FXS, typename T>
__device__ __forceinline__ void mom_point(const T *U0, const T *V0, const T *W0, const T *Up, const T *Vp,
                                          const T *Wp, int uc, T uzm, T vzm, T wzm, T uxpm, T vypm, const T *FX,
                                          const T *FY, const T *FZ, T fzm, int fc, T sk, T cj, T si, T ck, T sj, T ci,
                                          T ro0, T ro1, T ro2, const MomK<T> &q, T *out)
{
    const T dxi = q.dxi, ddxi = q.ddxi, mu = q.mu, rhoi = q.rhoi, f1 = q.f1, f2 = q.f2, f3 = q.f3;
    const T u0 = U0[uc], v0 = V0[uc], w0 = W0[uc];
    const T uxp = U0[uc + 1], uxm = U0[uc - 1], uyp = U0[uc + SX], uym = U0[uc - SX];
    const T uzp = Up[uc];
    const T vxp = V0[uc + 1], vxm = V0[uc - 1], vyp = V0[uc + SX], vym = V0[uc - SX];
    const T vzp = Vp[uc];
    const T wxp = W0[uc + 1], wxm = W0[uc - 1], wyp = W0[uc + SX], wym = W0[uc - SX];
    const T wzp = Wp[uc];
    T h11 = (uxp + u0) * (uxp + u0) - (u0 + uxm) * (u0 + uxm);
    T h12 = (uyp + u0) * (vyp + V0[uc + SX - 1]) - (u0 + uym) * (v0 + vxm);
    T h13 = (uzp + u0) * (wzp + Wp[uc - 1]) - (u0 + uzm) * (w0 + wxm);
    T h21 = (uxp + U0[uc + 1 - SX]) * (vxp + v0) - (u0 + uym) * (v0 + vxm);
    T h22 = (vyp + v0) * (vyp + v0) - (v0 + vym) * (v0 + vym);
    T h23 = (wzp + Wp[uc - SX]) * (vzp + v0) - (w0 + wym) * (v0 + vzm);
    T h31 = (wxp + w0) * (uxp + uxpm) - (w0 + wxm) * (u0 + uzm);
    T h32 = (vyp + vypm) * (wyp + w0) - (v0 + vzm) * (w0 + wym);
    T h33 = (wzp + w0) * (wzp + w0) - (w0 + wzm) * (w0 + wzm);
    h11 = h11 * (T)0.25 * dxi; h12 = h12 * (T)0.25 * dxi; h13 = h13 * (T)0.25 * dxi;
    h21 = h21 * (T)0.25 * dxi; h22 = h22 * (T)0.25 * dxi; h23 = h23 * (T)0.25 * dxi;
    h31 = h31 * (T)0.25 * dxi; h32 = h32 * (T)0.25 * dxi; h33 = h33 * (T)0.25 * dxi;
    T ru = -((h11 + h12) + h13);
    T rv = -((h21 + h22) + h23);
    T rw = -((h31 + h32) + h33);
    h11 = mu * ((uxp - (T)2.0 * u0) + uxm) * ddxi;
    h12 = mu * ((uyp - (T)2.0 * u0) + uym) * ddxi;
    h13 = mu * ((uzp - (T)2.0 * u0) + uzm) * ddxi;
    h21 = mu * ((vxp - (T)2.0 * v0) + vxm) * ddxi;
    h22 = mu * ((vyp - (T)2.0 * v0) + vym) * ddxi;
    h23 = mu * ((vzp - (T)2.0 * v0) + vzm) * ddxi;
    h31 = mu * ((wxp - (T)2.0 * w0) + wxm) * ddxi;
    h32 = mu * ((wyp - (T)2.0 * w0) + wym) * ddxi;
    h33 = mu * ((wzp - (T)2.0 * w0) + wzm) * ddxi;
    ru = ru + ((h11 + h12) + h13) * rhoi;
    rv = rv + ((h21 + h22) + h23) * rhoi;
    rw = rw + ((h31 + h32) + h33) * rhoi;
    ru = (ru + f3 * sk) + f2 * cj;
    rv = (rv + f1 * si) + f3 * ck;
    rw = (rw + f2 * sj) + f1 * ci;
    if constexpr (PHI) {
        ru = ru + (T)0.5 * (FX[fc - 1] + FX[fc]) * rhoi;
        rv = rv + (T)0.5 * (FY[fc - FXS] + FY[fc]) * rhoi;
        rw = rw + (T)0.5 * (fzm + FZ[fc]) * rhoi;
    }
    const T dt = q.dt, alpha = q.alpha, beta = q.beta;
    out[0] = u0 + dt * (alpha * ru - beta * ro0);
    out[1] = v0 + dt * (alpha * rv - beta * ro1);
    out[2] = w0 + dt * (alpha * rw - beta * ro2);
    out[3] = ru;
    out[4] = rv;
    out[5] = rw;
}

constexpr int MTX = 32, MTY = 16, MTHREADS = MTX * MTY;
constexpr int MUX = MTX + 2, MUY = MTY + 2;       // u/v/w box
constexpr int MPX = MTX + 3, MPY = MTY + 3;       // phi box
static_assert(MUX * MUY <= 2 * MTHREADS && MPX * MPY <= 2 * MTHREADS, "box loads assume <= 2 elements per thread");
static_assert(MTX == 32 && MTX + MTY <= MTHREADS, "two tile rows per wavefront; one edge cell per thread");

// The value of the previous lane (x - 1 in the tile; lane 0 gets 0).
__device__ __forceinline__ double prev_lane(double x)
{
    const int lo = __builtin_amdgcn_update_dpp(0, __double2loint(x), 0x138, 0xf, 0xf, true);     // wave_shr:1
    const int hi = __builtin_amdgcn_update_dpp(0, __double2hiint(x), 0x138, 0xf, 0xf, true);
    return __hiloint2double(hi, lo);
}
__device__ __forceinline__ float prev_lane(float x)
{
    return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(x), 0x138, 0xf, 0xf, true));
}

template <int PHI, typename T>
__device__ __forceinline__ void k_momentum_body(uint3 blk,
    const T *__restrict__ u, const T *__restrict__ v, const T *__restrict__ w,
    const T *__restrict__ phi,
    T *__restrict__ us, T *__restrict__ vs, T *__restrict__ ws,
    T *__restrict__ ruo, T *__restrict__ rvo, T *__restrict__ rwo,
    const double *__restrict__ sinf, const double *__restrict__ cosf, const Scalars *__restrict__ sc,
    Consts c, double ALPHA, double BETA, int kz)
{
    if (halted(sc)) return;
    __shared__ T UL[3][3][MUY * MUX];
    __shared__ T PL[PHI ? 3 : 1][PHI ? MPY * MPX : 1];
    __shared__ T FXL[PHI ? 2 : 1][PHI ? MTY : 1];
    __shared__ T FYL[PHI ? 2 : 1][PHI ? (MTY + 1) * MTX : 1];
    const int n = c.n;
    const int tid = threadIdx.x;
    const int i0 = blk.x * MTX, j0 = blk.y * MTY, k0 = blk.z * kz;
    const T um = sc->umean, vm = sc->vmean, wm = sc->wmean;
    MomK<T> q;
    q.dxi = (T)c.dxi; q.ddxi = (T)c.ddxi; q.mu = (T)c.mu; q.rhoi = (T)c.rhoi;
    q.f1 = (T)c.f1; q.f2 = (T)c.f2; q.f3 = (T)c.f3;
    q.dt = (T)c.dt; q.alpha = (T)ALPHA; q.beta = (T)BETA;

    // Box elements of this thread (<= 2 per box) and their x/y offsets.
    unsigned uoff[2], foff[2];
#pragma unroll
    for (int r = 0; r < 2; r++) {
        const int e = tid + r * MTHREADS;
        uoff[r] = (unsigned)wrap(i0 - 1 + e % MUX, n) + (unsigned)n * wrap(j0 - 1 + e / MUX, n);
        foff[r] = (unsigned)wrap(i0 - 2 + e % MPX, n) + (unsigned)n * wrap(j0 - 2 + e / MPX, n);
    }
    const size_t nn = (size_t)n * n;
    // Loads run one plane ahead into registers (pu, pp) and are stored into
    // the LDS rings an iteration later, so their latency overlaps compute.
    T pu[2][3], pp[2];
    auto fetch_u = [&](int m) {
        const size_t zoff = nn * (size_t)wrap(m, n);
#pragma unroll
        for (int r = 0; r < 2; r++) {
            if (tid + r * MTHREADS < MUX * MUY) {
                const size_t g = uoff[r] + zoff;
                pu[r][0] = u[g]; pu[r][1] = v[g]; pu[r][2] = w[g];
            }
        }
    };
    auto store_u = [&](int slot) {
#pragma unroll
        for (int r = 0; r < 2; r++) {
            const int e = tid + r * MTHREADS;
            if (e < MUX * MUY) {
                UL[slot][0][e] = pu[r][0] - um;
                UL[slot][1][e] = pu[r][1] - vm;
                UL[slot][2][e] = pu[r][2] - wm;
            }
        }
    };
    auto fetch_phi = [&](int m) {
        if constexpr (PHI) {
            const size_t zoff = nn * (size_t)wrap(m, n);
#pragma unroll
            for (int r = 0; r < 2; r++)
                if (tid + r * MTHREADS < MPX * MPY) pp[r] = phi[foff[r] + zoff];
        }
    };
    auto store_phi = [&](int slot) {
        if constexpr (PHI) {
#pragma unroll
            for (int r = 0; r < 2; r++) {
                const int e = tid + r * MTHREADS;
                if (e < MPX * MPY) PL[slot][e] = pp[r];
            }
        }
    };
    const int tx = tid % MTX, ty = tid / MTX;
    const int i = i0 + tx, j = j0 + ty;
    const bool active = (i < n) && (j < n);
    const int kend = min(k0 + kz, n);
    const int uc = (ty + 1) * MUX + (tx + 1), pc = (ty + 2) * MPX + (tx + 2);
    // The cell before the tile in x (row tid) or y (column tid - MTY) whose force this thread forms too.
    const bool edge_x = tid < MTY, edge = tid < MTX + MTY;
    const int ec = edge_x ? (tid + 2) * MPX + 1 : MPX + (tid - MTY + 2);
    const T sig6 = (T)((T)6.0 * c.sigma), eps = (T)c.eps, epsi = (T)c.epsi;
    auto chem = [&](const T *P0, const T *Pp, int e, T fzm) {
        const T f0 = P0[e];
        T t1 = f0 * ((T)1.0 - f0) * ((T)1.0 - (T)2.0 * f0) * epsi;
        T s6 = (((((P0[e + 1] + P0[e - 1]) + P0[e + MPX]) + P0[e - MPX]) + Pp[e]) + fzm) - (T)6.0 * f0;
        return t1 - eps * s6 * q.ddxi;
    };
    auto part = [&](T ch, T fp, T fm) { return sig6 * ch * ((T)0.5 * (fp - fm) * q.dxi); };
    // phi of the plane below at the thread's own and edge cell; its own forces
    // at the plane and, in z, at the plane below
    T fown = (T)0.0, fedge = (T)0.0, FX[9] = {}, FY[9] = {}, FZ[9] = {}, fzm = (T)0.0;
    auto force = [&](int s0, int sp, int buf) {
        if constexpr (PHI) {
            const T *P0 = PL[s0], *Pp = PL[sp];
            {
                const T ch = chem(P0, Pp, pc, fown);
                FX[4] = part(ch, P0[pc + 1], P0[pc - 1]);
                FY[4] = part(ch, P0[pc + MPX], P0[pc - MPX]);
                FZ[4] = part(ch, Pp[pc], fown);
                FYL[buf][(ty + 1) * MTX + tx] = FY[4];
                fown = P0[pc];
            }
            if (edge) {
                const T ch = chem(P0, Pp, ec, fedge);
                if (edge_x) FXL[buf][tid] = part(ch, P0[ec + 1], P0[ec - 1]);
                else FYL[buf][tid - MTY] = part(ch, P0[ec + MPX], P0[ec - MPX]);
                fedge = P0[ec];
            }
        }
    };
    const size_t cxy = (size_t)(i < n ? i : 0) + (size_t)n * (j < n ? j : 0);
    const int ic = i < n ? i : 0, jc = j < n ? j : 0;

    // prologue: slot of plane m in either ring: (m - k0) % 3
    fetch_u(k0);
    T um1[5];           // at plane k - 1: u, v, w, u(i+1), v(j+1)
    {
        const size_t zm = nn * (size_t)wrap(k0 - 1, n);
        um1[0] = u[cxy + zm] - um;
        um1[1] = v[cxy + zm] - vm;
        um1[2] = w[cxy + zm] - wm;
        um1[3] = u[zm + (size_t)n * jc + (ic + 1 == n ? 0 : ic + 1)] - um;
        um1[4] = v[zm + (size_t)n * (jc + 1 == n ? 0 : jc + 1) + ic] - vm;
    }
    T fzz = (T)0.0;
    if constexpr (PHI) {
        fzz = phi[cxy + nn * (size_t)wrap(k0 - 2, n)];
        fetch_phi(k0 - 1); store_phi(2);
        fetch_phi(k0); store_phi(0);
        fetch_phi(k0 + 1); store_phi(1);
    }
    store_u(0);
    fetch_u(k0 + 1);
    if (k0 + 1 < kend) fetch_phi(k0 + 2);
    T ro[3] = {(T)0.0, (T)0.0, (T)0.0};
    if (active) {
        ro[0] = ruo[cxy + nn * (size_t)k0];
        ro[1] = rvo[cxy + nn * (size_t)k0];
        ro[2] = rwo[cxy + nn * (size_t)k0];
    }
    __syncthreads();
    if constexpr (PHI) {
        fzm = part(chem(PL[2], PL[0], pc, fzz), PL[0][pc], fzz);
        fown = PL[2][pc];
        if (edge) fedge = PL[2][ec];
    }
    force(0, 1, 0);
    if constexpr (PHI) __syncthreads();        // the first plane's store takes slot 2, read above
    // One barrier a plane.  What is stored before the barrier of plane k (u of
    // k+1, phi of k+2) takes the slots of u(k-2) and phi(k-1), last read before
    // the barrier of plane k-1; force(k+1) writes the buffer that output(k-1)
    // read, before this barrier too.
    int sa = 0, sb = 1, sn = 2, buf = 0;       // slots of planes k, k+1 and the free one
    const T sj = (T)sinf[jc], cj = (T)cosf[jc], si = (T)sinf[ic], ci = (T)cosf[ic];
    for (int k = k0; k < kend; k++) {
        const bool more = k + 1 < kend;
        store_u(sb);
        if (more) {
            if constexpr (PHI) {
                store_phi(sn);
                if (k + 2 < kend) fetch_phi(k + 3);
            }
            fetch_u(k + 2);
        }
        const T ro0 = ro[0], ro1 = ro[1], ro2 = ro[2];
        if (active && more) {
            ro[0] = __builtin_nontemporal_load(&ruo[cxy + nn * (size_t)(k + 1)]);
            ro[1] = __builtin_nontemporal_load(&rvo[cxy + nn * (size_t)(k + 1)]);
            ro[2] = __builtin_nontemporal_load(&rwo[cxy + nn * (size_t)(k + 1)]);
        }
        __syncthreads();
        if constexpr (PHI) {
            FX[3] = prev_lane(FX[4]);
            if (tx == 0) FX[3] = FXL[buf][ty];
            FY[1] = FYL[buf][ty * MTX + tx];
        }
        const T *U0 = UL[sa][0], *V0 = UL[sa][1], *W0 = UL[sa][2];
        T o[6];
        mom_point<PHI, MUX, 3>(U0, V0, W0, UL[sb][0], UL[sb][1], UL[sb][2], uc, um1[0], um1[1], um1[2], um1[3],
                               um1[4], FX, FY, FZ, fzm, 4, (T)sinf[k], cj, si, (T)cosf[k], sj, ci, ro0, ro1, ro2, q, o);
        um1[0] = U0[uc]; um1[1] = V0[uc]; um1[2] = W0[uc]; um1[3] = U0[uc + 1]; um1[4] = V0[uc + MUX];
        fzm = FZ[4];
        if (active) {
            const size_t t = cxy + nn * (size_t)k;
            __builtin_nontemporal_store(o[0], &us[t]);
            __builtin_nontemporal_store(o[1], &vs[t]);
            __builtin_nontemporal_store(o[2], &ws[t]);
            __builtin_nontemporal_store(o[3], &ruo[t]);
            __builtin_nontemporal_store(o[4], &rvo[t]);
            __builtin_nontemporal_store(o[5], &rwo[t]);
        }
        buf ^= 1;
        if (more) force(sb, sn, buf);
        const int t = sa;
        sa = sb; sb = sn; sn = t;
    }
}

template <int PHI, typename T>
__global__ void __launch_bounds__(MTHREADS, 4) k_momentum(
    const T *__restrict__ u, const T *__restrict__ v, const T *__restrict__ w,
    const T *__restrict__ phi,
    T *__restrict__ us, T *__restrict__ vs, T *__restrict__ ws,
    T *__restrict__ ruo, T *__restrict__ rvo, T *__restrict__ rwo,
    const double *__restrict__ sinf, const double *__restrict__ cosf, const Scalars *__restrict__ sc,
    Consts c, double ALPHA, double BETA, int kz)
{
    k_momentum_body<PHI, T>(xcd_block(), u, v, w, phi, us, vs, ws, ruo, rvo, rwo, sinf, cosf, sc, c, ALPHA, BETA, kz);
}


// ---------------------------------------------------------------------------
// The same pass with two x-points per thread, used for FP32 state (in FP64
// the pair needs 220 VGPRs and 95 KB of LDS: one wave per SIMD): 64 x 8 points
// per block, every global load and store a float2 (the u/v/w and phi boxes
// start at the even column i0-2, so pairs never straddle the periodic seam),
// half the memory instructions per byte of the one-point form.  Each point's
// arithmetic is mom_point, as in k_momentum, so the results are those of
// k_momentum<PHI, T> bit for bit.  One barrier a plane as there: with phi
// 192^3 102 -> 88 us, 256^3 211 -> 185, 512^3 1450 -> 1414; without it the
// same as before (512^3 1.41-1.47 ms on other boxes).  Eight rows: with phi a thread takes 147 VGPRs (three waves
// per SIMD), of which 16 rows leave one block per CU or, held to 128, 47
// spills (512^3 2020 us); 12 rows 1582 us.
// ---------------------------------------------------------------------------
constexpr int PTX = 32, PTY = 8, PTHREADS = PTX * PTY;  // threads; 2 points each in x
constexpr int PBX = 2 * PTX + 4, PUY = PTY + 2;           // u/v/w box row (68) and rows
constexpr int PPY = PTY + 3;                              // phi box rows, same row as u/v/w
static_assert((PBX / 2) * PUY <= 2 * PTHREADS && (PBX / 2) * PPY <= 2 * PTHREADS, "two pairs per thread");
static_assert(PTX == 32 && 2 * PTX + PTY <= PTHREADS, "two tile rows per wavefront; one edge cell per thread");

template <typename T> struct Pair2;
template <> struct Pair2<float> { typedef float2 type; };
template <> struct Pair2<double> { typedef double2 type; };

template <typename T>
__device__ __forceinline__ typename Pair2<T>::type ld2(const T *p)
{
    return *reinterpret_cast<const typename Pair2<T>::type *>(p);
}
template <typename T>
__device__ __forceinline__ void st2nt(T *p, T a, T b)
{
    typedef T nt_pair __attribute__((ext_vector_type(2)));
    nt_pair v = {a, b};
    __builtin_nontemporal_store(v, reinterpret_cast<nt_pair *>(p));
}

template <int PHI, typename T>
__device__ __forceinline__ void k_momentum_x2_body(uint3 blk,
    const T *__restrict__ u, const T *__restrict__ v, const T *__restrict__ w,
    const T *__restrict__ phi, T *__restrict__ us, T *__restrict__ vs, T *__restrict__ ws,
    T *__restrict__ ruo, T *__restrict__ rvo, T *__restrict__ rwo,
    const double *__restrict__ sinf, const double *__restrict__ cosf, const Scalars *__restrict__ sc,
    Consts c, double ALPHA, double BETA, int kz)
{
    using P2 = typename Pair2<T>::type;
    if (halted(sc)) return;
    __shared__ T UL[3][3][PUY * PBX];
    __shared__ T PL[PHI ? 3 : 1][PHI ? PPY * PBX : 1];
    __shared__ T FXL[PHI ? 2 : 1][PHI ? PTY : 1];
    __shared__ T FYL[PHI ? 2 : 1][PHI ? (PTY + 1) * 2 * PTX : 1];
    const int n = c.n;
    const int tid = threadIdx.x;
    const int i0 = blk.x * (2 * PTX), j0 = blk.y * PTY, k0 = blk.z * kz;
    const T um = sc->umean, vm = sc->vmean, wm = sc->wmean;
    MomK<T> q;
    q.dxi = (T)c.dxi; q.ddxi = (T)c.ddxi; q.mu = (T)c.mu; q.rhoi = (T)c.rhoi;
    q.f1 = (T)c.f1; q.f2 = (T)c.f2; q.f3 = (T)c.f3;
    q.dt = (T)c.dt; q.alpha = (T)ALPHA; q.beta = (T)BETA;
    constexpr int NP = PBX / 2;                    // pairs per box row (34)

    // pairs of this thread in the u/v/w box (rows j0-1 ..) and the phi box (rows j0-2 ..)
    unsigned uoff[2], foff[2];
#pragma unroll
    for (int r = 0; r < 2; r++) {
        const int e = tid + r * PTHREADS;
        const int x = wrap(i0 - 2 + 2 * (e % NP), n);
        uoff[r] = (unsigned)x + (unsigned)n * wrap(j0 - 1 + e / NP, n);
        foff[r] = (unsigned)x + (unsigned)n * wrap(j0 - 2 + e / NP, n);
    }
    const size_t nn = (size_t)n * n;
    P2 pu[2][3], pp[2];
    auto fetch_u = [&](int m) {
        const size_t zoff = nn * (size_t)wrap(m, n);
#pragma unroll
        for (int r = 0; r < 2; r++)
            if (tid + r * PTHREADS < NP * PUY) {
                const size_t g = uoff[r] + zoff;
                pu[r][0] = ld2(u + g); pu[r][1] = ld2(v + g); pu[r][2] = ld2(w + g);
            }
    };
    auto store_u = [&](int slot) {
#pragma unroll
        for (int r = 0; r < 2; r++) {
            const int e = tid + r * PTHREADS;              // pair e of the box is elements 2e, 2e + 1
            if (e < NP * PUY) {
                UL[slot][0][2 * e] = pu[r][0].x - um; UL[slot][0][2 * e + 1] = pu[r][0].y - um;
                UL[slot][1][2 * e] = pu[r][1].x - vm; UL[slot][1][2 * e + 1] = pu[r][1].y - vm;
                UL[slot][2][2 * e] = pu[r][2].x - wm; UL[slot][2][2 * e + 1] = pu[r][2].y - wm;
            }
        }
    };
    auto fetch_phi = [&](int m) {
        if constexpr (PHI) {
            const size_t zoff = nn * (size_t)wrap(m, n);
#pragma unroll
            for (int r = 0; r < 2; r++)
                if (tid + r * PTHREADS < NP * PPY) pp[r] = ld2(phi + foff[r] + zoff);
        }
    };
    auto store_phi = [&](int slot) {
        if constexpr (PHI) {
#pragma unroll
            for (int r = 0; r < 2; r++) {
                const int e = tid + r * PTHREADS;
                if (e < NP * PPY) {
                    PL[slot][2 * e] = pp[r].x;
                    PL[slot][2 * e + 1] = pp[r].y;
                }
            }
        }
    };
    const int tx = tid % PTX, ty = tid / PTX;
    const int i = i0 + 2 * tx, j = j0 + ty;
    const bool active = (i < n) && (j < n);        // n even: i+1 < n with i
    const int kend = min(k0 + kz, n);
    const int uc = (ty + 1) * PBX + (2 * tx + 2), pc = (ty + 2) * PBX + (2 * tx + 2);
    // The cell before the tile in x (row tid) or y (column tid - PTY) whose force this thread forms too.
    const bool edge_x = tid < PTY, edge = tid < 2 * PTX + PTY;
    const int ec = edge_x ? (tid + 2) * PBX + 1 : PBX + (tid - PTY + 2);
    const T sig6 = (T)((T)6.0 * c.sigma), eps = (T)c.eps, epsi = (T)c.epsi;
    auto chem = [&](const T *P0, const T *Pp, int e, T fm) {
        const T f0 = P0[e];
        T t1 = f0 * ((T)1.0 - f0) * ((T)1.0 - (T)2.0 * f0) * epsi;
        T s6 = (((((P0[e + 1] + P0[e - 1]) + P0[e + PBX]) + P0[e - PBX]) + Pp[e]) + fm) - (T)6.0 * f0;
        return t1 - eps * s6 * q.ddxi;
    };
    auto part = [&](T ch, T fp, T fm) { return sig6 * ch * ((T)0.5 * (fp - fm) * q.dxi); };
    // as in k_momentum, for the thread's two points
    T fown[2] = {}, fedge = (T)0.0, FX[2][9] = {}, FY[2][9] = {}, FZ[2][9] = {}, fzm[2] = {};
    auto force = [&](int s0, int sp, int buf) {
        if constexpr (PHI) {
            const T *P0 = PL[s0], *Pp = PL[sp];
#pragma unroll
            for (int h = 0; h < 2; h++) {
                const int e = pc + h;
                const T ch = chem(P0, Pp, e, fown[h]);
                FX[h][4] = part(ch, P0[e + 1], P0[e - 1]);
                FY[h][4] = part(ch, P0[e + PBX], P0[e - PBX]);
                FZ[h][4] = part(ch, Pp[e], fown[h]);
                FYL[buf][(ty + 1) * 2 * PTX + 2 * tx + h] = FY[h][4];
                fown[h] = P0[e];
            }
            if (edge) {
                const T ch = chem(P0, Pp, ec, fedge);
                if (edge_x) FXL[buf][tid] = part(ch, P0[ec + 1], P0[ec - 1]);
                else FYL[buf][tid - PTY] = part(ch, P0[ec + PBX], P0[ec - PBX]);
                fedge = P0[ec];
            }
        }
    };
    const int ic = i < n ? i : 0, jc = j < n ? j : 0;
    const size_t cxy = (size_t)ic + (size_t)n * jc;

    // prologue: slot of plane m in either ring: (m - k0) % 3
    fetch_u(k0);
    T u1[3], v1[2], v1p[2], w1[2];      // plane k-1: u at i .. i+2, v at j and j+1, w
    {
        const size_t zm = nn * (size_t)wrap(k0 - 1, n), row = zm + (size_t)n * jc;
        const P2 a = ld2(u + row + ic), b = ld2(v + row + ic), d = ld2(w + row + ic),
                 e = ld2(v + zm + (size_t)n * (jc + 1 == n ? 0 : jc + 1) + ic);
        u1[0] = a.x - um; u1[1] = a.y - um;
        u1[2] = u[row + (ic + 2 == n ? 0 : ic + 2)] - um;
        v1[0] = b.x - vm; v1[1] = b.y - vm;
        v1p[0] = e.x - vm; v1p[1] = e.y - vm;
        w1[0] = d.x - wm; w1[1] = d.y - wm;
    }
    P2 fzz;
    fzz.x = fzz.y = (T)0.0;
    if constexpr (PHI) {
        fzz = ld2(phi + cxy + nn * (size_t)wrap(k0 - 2, n));
        fetch_phi(k0 - 1); store_phi(2);
        fetch_phi(k0); store_phi(0);
        fetch_phi(k0 + 1); store_phi(1);
    }
    store_u(0);
    fetch_u(k0 + 1);
    if (k0 + 1 < kend) fetch_phi(k0 + 2);
    const T sj = (T)sinf[jc], cj = (T)cosf[jc];
    const T sia = (T)sinf[ic], cia = (T)cosf[ic], sib = (T)sinf[ic + 1], cib = (T)cosf[ic + 1];
    P2 ro[3];
    ro[0].x = ro[0].y = ro[1].x = ro[1].y = ro[2].x = ro[2].y = (T)0.0;
    if (active) {
        ro[0] = ld2(ruo + cxy + nn * (size_t)k0);
        ro[1] = ld2(rvo + cxy + nn * (size_t)k0);
        ro[2] = ld2(rwo + cxy + nn * (size_t)k0);
    }
    __syncthreads();
    if constexpr (PHI) {
        fzm[0] = part(chem(PL[2], PL[0], pc, fzz.x), PL[0][pc], fzz.x);
        fzm[1] = part(chem(PL[2], PL[0], pc + 1, fzz.y), PL[0][pc + 1], fzz.y);
        fown[0] = PL[2][pc];
        fown[1] = PL[2][pc + 1];
        if (edge) fedge = PL[2][ec];
    }
    force(0, 1, 0);
    if constexpr (PHI) __syncthreads();        // the first plane's store takes slot 2, read above
    int sa = 0, sb = 1, sn = 2, buf = 0;       // slots of planes k, k+1 and the free one
    for (int k = k0; k < kend; k++) {
        const bool more = k + 1 < kend;
        store_u(sb);
        if (more) {
            if constexpr (PHI) {
                store_phi(sn);
                if (k + 2 < kend) fetch_phi(k + 3);
            }
            fetch_u(k + 2);
        }
        const P2 r0 = ro[0], r1 = ro[1], r2 = ro[2];
        if (active && more) {
            ro[0] = ld2(ruo + cxy + nn * (size_t)(k + 1));
            ro[1] = ld2(rvo + cxy + nn * (size_t)(k + 1));
            ro[2] = ld2(rwo + cxy + nn * (size_t)(k + 1));
        }
        __syncthreads();
        if constexpr (PHI) {
            FX[0][3] = prev_lane(FX[1][4]);
            if (tx == 0) FX[0][3] = FXL[buf][ty];
            FX[1][3] = FX[0][4];
            FY[0][1] = FYL[buf][ty * 2 * PTX + 2 * tx];
            FY[1][1] = FYL[buf][ty * 2 * PTX + 2 * tx + 1];
        }
        const T *U0 = UL[sa][0], *V0 = UL[sa][1], *W0 = UL[sa][2];
        const T *Up = UL[sb][0], *Vp = UL[sb][1], *Wp = UL[sb][2];
        const T sk = (T)sinf[k], ck = (T)cosf[k];
        T oa[6], ob[6];
        mom_point<PHI, PBX, 3>(U0, V0, W0, Up, Vp, Wp, uc, u1[0], v1[0], w1[0], u1[1], v1p[0], FX[0], FY[0], FZ[0],
                               fzm[0], 4, sk, cj, sia, ck, sj, cia, r0.x, r1.x, r2.x, q, oa);
        mom_point<PHI, PBX, 3>(U0, V0, W0, Up, Vp, Wp, uc + 1, u1[1], v1[1], w1[1], u1[2], v1p[1], FX[1], FY[1], FZ[1],
                               fzm[1], 4, sk, cj, sib, ck, sj, cib, r0.y, r1.y, r2.y, q, ob);
#pragma unroll
        for (int h = 0; h < 3; h++) u1[h] = U0[uc + h];
#pragma unroll
        for (int h = 0; h < 2; h++) {
            v1[h] = V0[uc + h]; v1p[h] = V0[uc + PBX + h]; w1[h] = W0[uc + h];
            fzm[h] = FZ[h][4];
        }
        if (active) {
            const size_t t = cxy + nn * (size_t)k;
            st2nt(us + t, oa[0], ob[0]);
            st2nt(vs + t, oa[1], ob[1]);
            st2nt(ws + t, oa[2], ob[2]);
            st2nt(ruo + t, oa[3], ob[3]);
            st2nt(rvo + t, oa[4], ob[4]);
            st2nt(rwo + t, oa[5], ob[5]);
        }
        buf ^= 1;
        if (more) force(sb, sn, buf);
        const int t = sa;
        sa = sb; sb = sn; sn = t;
    }
}

template <int PHI, typename T>
__global__ void __launch_bounds__(PTHREADS) k_momentum_x2(
    const T *__restrict__ u, const T *__restrict__ v, const T *__restrict__ w,
    const T *__restrict__ phi, T *__restrict__ us, T *__restrict__ vs, T *__restrict__ ws,
    T *__restrict__ ruo, T *__restrict__ rvo, T *__restrict__ rwo,
    const double *__restrict__ sinf, const double *__restrict__ cosf, const Scalars *__restrict__ sc,
    Consts c, double ALPHA, double BETA, int kz)
{
    k_momentum_x2_body<PHI, T>(xcd_block(), u, v, w, phi, us, vs, ws, ruo, rvo, rwo, sinf, cosf, sc, c, ALPHA, BETA, kz);
}


// ---------------------------------------------------------------------------
// The same pass without a march, for boxes whose march is a few planes long and
// then bound by its chain of barriers, not by memory: one point per thread,
// every neighbour loaded from the caches, the CSF force formed at the point and
// at its three lower neighbours.  49 loads per point, all in flight at once,
// and no barrier.  mom_point on 3 x 3 neighbourhoods (row stride 3, the point
// at 4): the results are those of k_momentum bit for bit.  March at its best
// slab / point, with the phase field, us (event times): FP64 32^3 10.2 / 6.6,
// 48^3 10.8 / 10.2, 54^3 11.2 / 11.3, 64^3 12.0 / 12.8, 72^3 22.0 / 20.0, 96^3
// 26.4 / 32.9; FP32 32^3 9.9 / 6.5, 64^3 10.5 / 8.3, 72^3 13.5 / 12.3, 96^3 17.7 /
// 17.7, 108^3 22.7 / 29.5.  Used up to 64^3 and 96^3: the lines were drawn
// against a march with two barriers a plane (64^3 FP64 14.3, 96^3 FP32 22.1 us);
// with one the two are level there.  72^3 FP64 stays with the march, which
// without the phase field is level too (19.2 / 18.0) at two planes a slab,
// though kz_momentum gives it four (24.3 us).
// Bound by the L1: 49 loads of 512 bytes per wavefront.
// At most 4 waves per SIMD, or the compiler saves registers and waits for
// the loads in groups (FP64 32^3 7.9 us).
// ---------------------------------------------------------------------------
constexpr int DTX = 32, DTY = 8;

template <int PHI, typename T>
__device__ __forceinline__ void k_momentum_point_body(uint3 blk,
    const T *__restrict__ u, const T *__restrict__ v, const T *__restrict__ w, const T *__restrict__ phi,
    T *__restrict__ us, T *__restrict__ vs, T *__restrict__ ws,
    T *__restrict__ ruo, T *__restrict__ rvo, T *__restrict__ rwo,
    const double *__restrict__ sinf, const double *__restrict__ cosf, const Scalars *__restrict__ sc,
    const Consts &c, double ALPHA, double BETA)
{
    const bool stop = halted(sc);
    const int n = c.n;
    const int i = blk.x * DTX + threadIdx.x % DTX, j = blk.y * DTY + threadIdx.x / DTX, k = blk.z;
    if (i >= n || j >= n) return;
    // periodic neighbours: columns, rows and planes -1 (and -2 for phi), 0, +1, as offsets
    const int im = i == 0 ? n - 1 : i - 1, ip = i + 1 == n ? 0 : i + 1;
    const int jm = j == 0 ? n - 1 : j - 1, jp = j + 1 == n ? 0 : j + 1;
    const int km = k == 0 ? n - 1 : k - 1, kp = k + 1 == n ? 0 : k + 1;
    const unsigned nn = (unsigned)n * n;
    const unsigned r0 = (unsigned)n * j, rm = (unsigned)n * jm, rp = (unsigned)n * jp;
    const unsigned z0 = nn * k, zm = nn * km, zp = nn * kp;
    const T um = sc->umean, vm = sc->vmean, wm = sc->wmean;
    T U0[9] = {}, V0[9] = {}, W0[9] = {}, Up[9] = {}, Vp[9] = {}, Wp[9] = {};
    auto at = [](const T *f, unsigned off) { return ld_off(f, off); };
    U0[4] = at(u, z0 + r0 + i) - um; U0[5] = at(u, z0 + r0 + ip) - um; U0[3] = at(u, z0 + r0 + im) - um;
    U0[7] = at(u, z0 + rp + i) - um; U0[1] = at(u, z0 + rm + i) - um; U0[2] = at(u, z0 + rm + ip) - um;
    V0[4] = at(v, z0 + r0 + i) - vm; V0[5] = at(v, z0 + r0 + ip) - vm; V0[3] = at(v, z0 + r0 + im) - vm;
    V0[7] = at(v, z0 + rp + i) - vm; V0[1] = at(v, z0 + rm + i) - vm; V0[6] = at(v, z0 + rp + im) - vm;
    W0[4] = at(w, z0 + r0 + i) - wm; W0[5] = at(w, z0 + r0 + ip) - wm; W0[3] = at(w, z0 + r0 + im) - wm;
    W0[7] = at(w, z0 + rp + i) - wm; W0[1] = at(w, z0 + rm + i) - wm;
    Up[4] = at(u, zp + r0 + i) - um;
    Vp[4] = at(v, zp + r0 + i) - vm;
    Wp[4] = at(w, zp + r0 + i) - wm; Wp[3] = at(w, zp + r0 + im) - wm; Wp[1] = at(w, zp + rm + i) - wm;
    const T uzm = at(u, zm + r0 + i) - um, uxpm = at(u, zm + r0 + ip) - um;
    const T vzm = at(v, zm + r0 + i) - vm, vypm = at(v, zm + rp + i) - vm;
    const T wzm = at(w, zm + r0 + i) - wm;
    const unsigned t = z0 + r0 + i;
    const T ro0 = ruo[t], ro1 = rvo[t], ro2 = rwo[t];
    MomK<T> q;
    q.dxi = (T)c.dxi; q.ddxi = (T)c.ddxi; q.mu = (T)c.mu; q.rhoi = (T)c.rhoi;
    q.f1 = (T)c.f1; q.f2 = (T)c.f2; q.f3 = (T)c.f3;
    q.dt = (T)c.dt; q.alpha = (T)ALPHA; q.beta = (T)BETA;
    T FX[9] = {}, FY[9] = {}, FZ[9] = {}, fzm = 0;
    if constexpr (PHI) {
        const T sig6 = (T)((T)6.0 * c.sigma), eps = (T)c.eps, epsi = (T)c.epsi, dxi = q.dxi, ddxi = q.ddxi;
        const int imm = im == 0 ? n - 1 : im - 1, jmm = jm == 0 ? n - 1 : jm - 1, kmm = km == 0 ? n - 1 : km - 1;
        const unsigned rmm = (unsigned)n * jmm, zmm = nn * kmm;
        // CSF force at a cell centre: sigma 6 chem times half the difference of the pair (p, m) / dx
        auto chem = [&](T f0, T fxp, T fxm, T fyp, T fym, T fzp, T fzm_) {
            T t1 = f0 * ((T)1.0 - f0) * ((T)1.0 - (T)2.0 * f0) * epsi;
            T s6 = (((((fxp + fxm) + fyp) + fym) + fzp) + fzm_) - (T)6.0 * f0;
            return t1 - eps * s6 * ddxi;
        };
        auto part = [&](T ch, T fp, T fm) { return sig6 * ch * ((T)0.5 * (fp - fm) * dxi); };
        const T f0 = at(phi, z0 + r0 + i), fx = at(phi, z0 + r0 + ip), fX = at(phi, z0 + r0 + im);
        const T fy = at(phi, z0 + rp + i), fY = at(phi, z0 + rm + i), fz = at(phi, zp + r0 + i), fZ = at(phi, zm + r0 + i);
        const T fXX = at(phi, z0 + r0 + imm), fXy = at(phi, z0 + rp + im), fXY = at(phi, z0 + rm + im),
                fXz = at(phi, zp + r0 + im), fXZ = at(phi, zm + r0 + im);
        const T fYY = at(phi, z0 + rmm + i), fYx = at(phi, z0 + rm + ip), fYz = at(phi, zp + rm + i),
                fYZ = at(phi, zm + rm + i);
        const T fZZ = at(phi, zmm + r0 + i), fZx = at(phi, zm + r0 + ip), fZy = at(phi, zm + rp + i);
        const T c0 = chem(f0, fx, fX, fy, fY, fz, fZ);
        FX[4] = part(c0, fx, fX);
        FY[4] = part(c0, fy, fY);
        FZ[4] = part(c0, fz, fZ);
        FX[3] = part(chem(fX, f0, fXX, fXy, fXY, fXz, fXZ), f0, fXX);
        FY[1] = part(chem(fY, fYx, fXY, f0, fYY, fYz, fYZ), f0, fYY);
        fzm = part(chem(fZ, fZx, fXZ, fZy, fYZ, f0, fZZ), f0, fZZ);
    }
    T o[6];
    mom_point<PHI, 3, 3>(U0, V0, W0, Up, Vp, Wp, 4, uzm, vzm, wzm, uxpm, vypm, FX, FY, FZ, fzm, 4, (T)sinf[k], (T)cosf[j],
                         (T)sinf[i], (T)cosf[k], (T)sinf[j], (T)cosf[i], ro0, ro1, ro2, q, o);
    if (stop) return;
    __builtin_nontemporal_store(o[0], &us[t]);
    __builtin_nontemporal_store(o[1], &vs[t]);
    __builtin_nontemporal_store(o[2], &ws[t]);
    __builtin_nontemporal_store(o[3], &ruo[t]);
    __builtin_nontemporal_store(o[4], &rvo[t]);
    __builtin_nontemporal_store(o[5], &rwo[t]);
}

template <int PHI, typename T>
__global__ void __launch_bounds__(DTX * DTY) __attribute__((amdgpu_waves_per_eu(1, 4))) k_momentum_point(
    const T *__restrict__ u, const T *__restrict__ v, const T *__restrict__ w, const T *__restrict__ phi,
    T *__restrict__ us, T *__restrict__ vs, T *__restrict__ ws,
    T *__restrict__ ruo, T *__restrict__ rvo, T *__restrict__ rwo,
    const double *__restrict__ sinf, const double *__restrict__ cosf, const Scalars *__restrict__ sc,
    Consts c, double ALPHA, double BETA)
{
    k_momentum_point_body<PHI, T>(xcd_block(), u, v, w, phi, us, vs, ws, ruo, rvo, rwo, sinf, cosf, sc, c, ALPHA, BETA);
}


// ---------------------------------------------------------------------------
// FFT machinery: mixed-radix Stockham autosort in LDS (Govindaraju et al.,
// SC'08), unnormalised.  A block holds `nlines` lines of length n; element p of
// line l sits at lds[l*lstride + p*pstride].  Each thread owns at most one
// radix-R butterfly per stage (the block has >= nlines*n/Rmin threads);
// consecutive threads take consecutive lines so that LDS accesses of a
// wavefront are contiguous for column tiles.
// ---------------------------------------------------------------------------
constexpr int FFT_MAX_THREADS = 1024;
constexpr size_t LDS_CAP = 65536;   // dynamic LDS bytes per block of the heuristic shapes (2 blocks per CU;
                                    // register-path column tiles up to twice that, 1 block per CU)
constexpr size_t LDS_MAX = 163840;  // what a gfx950 workgroup may allocate (tunable shapes)

template <int R, int SG>
__device__ __forceinline__ void fft_stage(double2 *lds, int n, int nlines, int lstride, int pstride,
                                          int Ns, const double2 *__restrict__ tw, bool first)
{
    const int L = n / R;
    const int total = nlines * L;
    const int t = threadIdx.x;
    const bool active = t < total;
    double2 v[R];
    int line = 0, j = 0;
    if (active) {
        line = t % nlines;
        j = t / nlines;
        const double2 *base = lds + line * lstride;
#pragma unroll
        for (int r = 0; r < R; r++) v[r] = base[(j + r * L) * pstride];
    }
    __syncthreads();
    if (active) {
        const int k = j % Ns;
        if (!first) {
#pragma unroll
            for (int r = 1; r < R; r++) {
                double2 wv = tw[k * (R - 1) + r - 1];
                double wi = SG < 0 ? -wv.y : wv.y;
                double xr = v[r].x, xi = v[r].y;
                v[r] = make_double2(xr * wv.x - xi * wi, xr * wi + xi * wv.x);
            }
        }
        dft<R, SG>(v);
        const int base_idx = (j / Ns) * Ns * R + k;
        double2 *base = lds + line * lstride;
#pragma unroll
        for (int r = 0; r < R; r++) base[(base_idx + r * Ns) * pstride] = v[r];
    }
    __syncthreads();
}

template <int SG>
__device__ void fft_lds(double2 *lds, int nlines, int lstride, int pstride, const FftPlan &pl,
                        const double2 *__restrict__ tw)
{
    for (int s = 0; s < pl.nst; s++) {
        const double2 *t = tw + pl.twoff[s];
        const bool first = (s == 0);
        switch (pl.R[s]) {
        case 8: fft_stage<8, SG>(lds, pl.n, nlines, lstride, pstride, pl.Ns[s], t, first); break;
        case 4: fft_stage<4, SG>(lds, pl.n, nlines, lstride, pstride, pl.Ns[s], t, first); break;
        case 3: fft_stage<3, SG>(lds, pl.n, nlines, lstride, pstride, pl.Ns[s], t, first); break;
        default: fft_stage<2, SG>(lds, pl.n, nlines, lstride, pstride, pl.Ns[s], t, first); break;
        }
    }
}

// Forward x pass with the Poisson right-hand side: divergence of u*, REAL(4) rounding of the
// Poisson RHS, then one complex FFT per pair of x-lines (j, j+1) whose
// spectrum is split into the two half spectra (main.f90:715-750).
template <typename T>
__device__ __forceinline__ void k_xfwd_body(uint3 blk, const T *__restrict__ us, const T *__restrict__ vs, const T *__restrict__ ws,
    double2 *__restrict__ spec, const double2 *__restrict__ tw, const Scalars *__restrict__ sc,
    Consts c, FftPlan pl, int ppb, int ld)
{
    if (halted(sc)) return;
    extern __shared__ double2 lds[];
    const int n = c.n, half = n / 2, nh = n / 2 + 1;
    const int lstride = n + 1;
    const int pair0 = blk.x * ppb;
    const double cdiv = c.rho * c.dxi / c.dt;
    for (int e = threadIdx.x; e < ppb * n; e += blockDim.x) {
        int pl_ = e / n, i = e - pl_ * n;
        int pair = pair0 + pl_;
        int k = pair / half, j = 2 * (pair - k * half);
        int ip = i + 1 == n ? 0 : i + 1;
        int kp = k + 1 == n ? 0 : k + 1;
        double rr[2];
#pragma unroll
        for (int h = 0; h < 2; h++) {
            int jj = j + h;
            int jp = jj + 1 == n ? 0 : jj + 1;
            size_t id = IDX(i, jj, k);
            double r = cdiv * ((double)us[IDX(ip, jj, k)] - (double)us[id]);
            r = r + cdiv * ((double)vs[IDX(i, jp, k)] - (double)vs[id]);
            r = r + cdiv * ((double)ws[IDX(i, jj, kp)] - (double)ws[id]);
            if (c.fp32_rhs) r = (double)(float)r;
            rr[h] = r;
        }
        lds[pl_ * lstride + i] = make_double2(rr[0], rr[1]);
    }
    __syncthreads();
    fft_lds<-1>(lds, ppb, lstride, 1, pl, tw);
    for (int e = threadIdx.x; e < ppb * nh; e += blockDim.x) {
        int pl_ = e / nh, q = e - pl_ * nh;
        int pair = pair0 + pl_;
        int k = pair / half, j = 2 * (pair - k * half);
        int m = q == 0 ? 0 : n - q;
        double2 zq = lds[pl_ * lstride + q], zm = lds[pl_ * lstride + m];
        double a = zq.x, b = zq.y, cc = zm.x, d = zm.y;
        spec[spec_row(k, j, n, ld) + q] = make_double2((a + cc) * 0.5, (b - d) * 0.5);
        spec[spec_row(k, j + 1, n, ld) + q] = make_double2((b + d) * 0.5, (cc - a) * 0.5);
    }
}

template <typename T>
__global__ void __launch_bounds__(FFT_MAX_THREADS) k_xfwd(
    const T *__restrict__ us, const T *__restrict__ vs, const T *__restrict__ ws,
    double2 *__restrict__ spec, const double2 *__restrict__ tw, const Scalars *__restrict__ sc,
    Consts c, FftPlan pl, int ppb, int ld)
{
    k_xfwd_body<T>(make_uint3(blockIdx.x, blockIdx.y, blockIdx.z), us, vs, ws, spec, tw, sc, c, pl, ppb, ld);
}


// Column pass along y (forward or inverse), in place.  Block = (kx tile, k).
template <int SG>
__device__ __forceinline__ void k_ypass_body(uint3 blk, double2 *__restrict__ spec,
                                                           const double2 *__restrict__ tw,
                                                           const Scalars *__restrict__ sc, FftPlan pl, int ld,
                                                           int tkx)
{
    if (halted(sc)) return;
    extern __shared__ double2 lds[];
    const int n = pl.n, nh = n / 2 + 1;
    const int q0 = blk.x * tkx, k = blk.y;
    const int nq = min(tkx, nh - q0);
    double2 *base = spec + spec_row(k, 0, n, ld) + q0;
    for (int e = threadIdx.x; e < n * tkx; e += blockDim.x) {
        int r = e / tkx, ql = e - r * tkx;
        lds[r * tkx + ql] = ql < nq ? base[(size_t)r * ld + ql] : make_double2(0.0, 0.0);
    }
    __syncthreads();
    fft_lds<SG>(lds, tkx, 1, tkx, pl, tw);
    for (int e = threadIdx.x; e < n * tkx; e += blockDim.x) {
        int r = e / tkx, ql = e - r * tkx;
        if (ql < nq) base[(size_t)r * ld + ql] = lds[r * tkx + ql];
    }
}

template <int SG>
__global__ void __launch_bounds__(FFT_MAX_THREADS) k_ypass(double2 *__restrict__ spec,
                                                           const double2 *__restrict__ tw,
                                                           const Scalars *__restrict__ sc, FftPlan pl, int ld,
                                                           int tkx)
{
    k_ypass_body<SG>(make_uint3(blockIdx.x, blockIdx.y, blockIdx.z), spec, tw, sc, pl, ld, tkx);
}


// Column pass along z: forward FFT, division by -k^2 and N^3 with the mean
// mode set to zero (main.f90:765-798), inverse FFT.  Block = (kx tile, j).
// INV_ONLY: the inverse z transform alone (no forward transform, no divide),
// for the initial-condition generator.
template <bool INV_ONLY = false>
__device__ __forceinline__ void k_zpoisson_body(uint3 blk, double2 *__restrict__ spec,
                                                              const double2 *__restrict__ tw,
                                                              const double *__restrict__ ktab,
                                                              const Scalars *__restrict__ sc, FftPlan pl, int ld,
                                                              int tkx)
{
    if (halted(sc)) return;
    extern __shared__ double2 lds[];
    const int n = pl.n, nh = n / 2 + 1;
    const int q0 = blk.x * tkx, j = blk.y;
    const int nq = min(tkx, nh - q0);
    const size_t rs = spec_plane(n, ld);
    double2 *base = spec + (size_t)j * ld + q0;
    for (int e = threadIdx.x; e < n * tkx; e += blockDim.x) {
        int r = e / tkx, ql = e - r * tkx;
        lds[r * tkx + ql] = ql < nq ? base[(size_t)r * rs + ql] : make_double2(0.0, 0.0);
    }
    __syncthreads();
    if constexpr (!INV_ONLY) {
        fft_lds<-1>(lds, tkx, 1, tkx, pl, tw);
        const double nnn = (double)((long long)n * (long long)n * (long long)n);
        const double ky = ktab[j];
        for (int e = threadIdx.x; e < n * tkx; e += blockDim.x) {
            int r = e / tkx, ql = e - r * tkx;
            int q = q0 + ql;
            if (ql < nq) {
                double kx = ktab[q], kz = ktab[r];
                double k2 = (kx * kx + ky * ky) + kz * kz;
                double2 z = lds[r * tkx + ql];
                z = make_double2(((-z.x) / k2) / nnn, ((-z.y) / k2) / nnn);
                if (q == 0 && j == 0 && r == 0) z = make_double2(0.0, 0.0);
                lds[r * tkx + ql] = z;
            }
        }
        __syncthreads();
    }
    fft_lds<1>(lds, tkx, 1, tkx, pl, tw);
    for (int e = threadIdx.x; e < n * tkx; e += blockDim.x) {
        int r = e / tkx, ql = e - r * tkx;
        if (ql < nq) base[(size_t)r * rs + ql] = lds[r * tkx + ql];
    }
}

__global__ void __launch_bounds__(FFT_MAX_THREADS) k_zpoisson(double2 *__restrict__ spec,
                                                              const double2 *__restrict__ tw,
                                                              const double *__restrict__ ktab,
                                                              const Scalars *__restrict__ sc, FftPlan pl, int ld,
                                                              int tkx)
{
    k_zpoisson_body<false>(make_uint3(blockIdx.x, blockIdx.y, blockIdx.z), spec, tw, ktab, sc, pl, ld, tkx);
}


// Inverse x pass: Hermitian extension of the half spectra of lines j and j+1,
// one complex inverse FFT per pair, p(.,j) = Re, p(.,j+1) = Im.
__device__ __forceinline__ void k_xinv_body(uint3 blk, const double2 *__restrict__ spec,
                                                          double *__restrict__ p, const double2 *__restrict__ tw,
                                                          const Scalars *__restrict__ sc, FftPlan pl, int ppb,
                                                          int ld)
{
    if (halted(sc)) return;
    extern __shared__ double2 lds[];
    const int n = pl.n, half = n / 2;
    const int lstride = n + 1;
    const int pair0 = blk.x * ppb;
    for (int e = threadIdx.x; e < ppb * n; e += blockDim.x) {
        int pl_ = e / n, q = e - pl_ * n;
        int pair = pair0 + pl_;
        int k = pair / half, j = 2 * (pair - k * half);
        const double2 *s1 = spec + spec_row(k, j, n, ld);
        const double2 *s2 = spec + spec_row(k, j + 1, n, ld);
        double2 z;
        if (q == 0 || q == half) {
            z = make_double2(s1[q].x, s2[q].x);
        } else if (q < half) {
            double2 a = s1[q], b = s2[q];
            z = make_double2(a.x - b.y, a.y + b.x);
        } else {
            int m = n - q;
            double2 a = s1[m], b = s2[m];
            z = make_double2(a.x + b.y, b.x - a.y);
        }
        lds[pl_ * lstride + q] = z;
    }
    __syncthreads();
    fft_lds<1>(lds, ppb, lstride, 1, pl, tw);
    for (int e = threadIdx.x; e < ppb * n; e += blockDim.x) {
        int pl_ = e / n, i = e - pl_ * n;
        int pair = pair0 + pl_;
        int k = pair / half, j = 2 * (pair - k * half);
        double2 z = lds[pl_ * lstride + i];
        p[IDX(i, j, k)] = z.x;
        p[IDX(i, j + 1, k)] = z.y;
    }
}

__global__ void __launch_bounds__(FFT_MAX_THREADS) k_xinv(const double2 *__restrict__ spec,
                                                          double *__restrict__ p, const double2 *__restrict__ tw,
                                                          const Scalars *__restrict__ sc, FftPlan pl, int ppb,
                                                          int ld)
{
    k_xinv_body(make_uint3(blockIdx.x, blockIdx.y, blockIdx.z), spec, p, tw, sc, pl, ppb, ld);
}


// ---------------------------------------------------------------------------
// Register-resident variant of the same Stockham FFT, for plans whose radices
// are 8, 4 and 2.  A line of length n is owned by LM = n/8 threads; thread tj
// holds the 8 elements at positions tj + m*LM (m = 0..7), which are exactly
// the inputs of its radix-8 butterfly (or of its 8/R radix-R butterflies, the
// q-th using m = q + r*8/R), and also exactly the outputs of the last stage.
// Hence the first stage reads straight from global memory, the last stage
// writes straight to global memory (or feeds the inverse transform), and LDS
// only carries the exchanges between stages.  Every butterfly, twiddle and
// operation order is the one of fft_stage, so results are bit-identical.
// ---------------------------------------------------------------------------
template <bool XL>
__device__ __forceinline__ int rlds(int line, int p, int lstride, int pstride)
{
    return XL ? line * lstride + p + (p >> 3) : line + p * pstride;
}

template <int R, int SG>
__device__ __forceinline__ void stage_regs(double2 (&v)[8], int tj, int LM, int Ns, const double2 *__restrict__ tw,
                                           bool first)
{
    constexpr int Q = 8 / R;
#pragma unroll
    for (int q = 0; q < Q; q++) {
        const unsigned jj = (unsigned)(tj + q * LM);
        const int k = (int)(jj % (unsigned)Ns);
        double2 x[R];
#pragma unroll
        for (int r = 0; r < R; r++) x[r] = v[q + r * Q];
        if (!first) {
#pragma unroll
            for (int r = 1; r < R; r++) {
                double2 wv = tw[k * (R - 1) + r - 1];
                double wi = SG < 0 ? -wv.y : wv.y;
                double xr = x[r].x, xi = x[r].y;
                x[r] = make_double2(xr * wv.x - xi * wi, xr * wi + xi * wv.x);
            }
        }
        dft<R, SG>(x);
#pragma unroll
        for (int r = 0; r < R; r++) v[q + r * Q] = x[r];
    }
}

template <int R, bool XL>
__device__ __forceinline__ void store_stage(const double2 (&v)[8], double2 *lds, int line, int tj, int LM, int Ns,
                                            int lstride, int pstride)
{
    constexpr int Q = 8 / R;
#pragma unroll
    for (int q = 0; q < Q; q++) {
        const unsigned jj = (unsigned)(tj + q * LM), k = jj % (unsigned)Ns;
        const int base = (int)((jj - k) * R + k);
#pragma unroll
        for (int r = 0; r < R; r++) lds[rlds<XL>(line, base + r * Ns, lstride, pstride)] = v[q + r * Q];
    }
}

// All stages of one line; v holds positions tj + m*LM on entry and on exit.
template <int SG, bool XL>
__device__ void fft_regs(double2 (&v)[8], int tj, int line, double2 *lds, int lstride, int pstride,
                         const FftPlan &pl, const double2 *__restrict__ tw)
{
    const int LM = pl.n / 8;
    for (int s = 0; s < pl.nst; s++) {
        if (s > 0) {
#pragma unroll
            for (int m = 0; m < 8; m++) v[m] = lds[rlds<XL>(line, tj + m * LM, lstride, pstride)];
            __syncthreads();
        }
        const double2 *t = tw + pl.twoff[s];
        const int R = pl.R[s], Ns = pl.Ns[s];
        if (R == 8) stage_regs<8, SG>(v, tj, LM, Ns, t, s == 0);
        else if (R == 4) stage_regs<4, SG>(v, tj, LM, Ns, t, s == 0);
        else stage_regs<2, SG>(v, tj, LM, Ns, t, s == 0);
        if (s < pl.nst - 1) {
            if (R == 8) store_stage<8, XL>(v, lds, line, tj, LM, Ns, lstride, pstride);
            else if (R == 4) store_stage<4, XL>(v, lds, line, tj, LM, Ns, lstride, pstride);
            else store_stage<2, XL>(v, lds, line, tj, LM, Ns, lstride, pstride);
            __syncthreads();
        }
    }
}

// The stage plan of a length N at compile time: the radices of the host plan
// builder (plan_radices), with the sub-lengths Ns and twiddle offsets that the
// host derives from them.  With N known the stage loop unrolls and every index
// of the exchanges (jj / Ns, jj % Ns, the line strides) becomes shifts, masks
// or a multiplication; fft_regs computes them from the runtime plan with
// integer divides.
struct CPlan {
    int nst, R[MAXSTAGES], Ns[MAXSTAGES], off[MAXSTAGES];
};
__host__ __device__ constexpr CPlan cplan(int n)
{
    CPlan p = {};
    p.nst = plan_radices(n, p.R);
    int ns = 1, off = 0;
    for (int s = 0; s < p.nst; s++) {
        p.Ns[s] = ns;
        p.off[s] = off;
        off += ns * (p.R[s] - 1);
        ns *= p.R[s];
    }
    return p;
}
constexpr bool is_pow2(int n) { return (n & (n - 1)) == 0; }
// Threads per line.  A power of two, or any plan with a radix-8 stage: n/8, one
// radix-8 butterfly each (a radix-3 stage then takes 2 2/3 per thread, the
// third for two threads of three).  Radices 4, 3 and 2 only: n/3, or n/6 with
// two butterflies each from 144 on (FFT passes of a step at 108^3 FP64 63 against
// 66 us, at 144^3 106 against 99 us).
__host__ __device__ constexpr int line_threads(int n)
{
    if (is_pow2(n)) return n / 8;
    const CPlan p = cplan(n);
    return p.R[0] == 8 ? n / 8 : n < 144 ? n / 3 : n / 6;
}

template <int SG, bool XL, int N, int S = 0>
__device__ __forceinline__ void fft_regs_c(double2 (&v)[8], int tj, int line, double2 *lds, int lstride,
                                           int pstride, const double2 *__restrict__ tw)
{
    constexpr CPlan P = cplan(N);
    constexpr int LM = N / 8, R = P.R[S], Ns = P.Ns[S];
    static_assert(is_pow2(N) && N >= 16, "8 elements per thread");
    if constexpr (S > 0) {
#pragma unroll
        for (int m = 0; m < 8; m++) v[m] = lds[rlds<XL>(line, tj + m * LM, lstride, pstride)];
        __syncthreads();
    }
    stage_regs<R, SG>(v, tj, LM, Ns, tw + P.off[S], S == 0);
    if constexpr (S + 1 < P.nst) {
        store_stage<R, XL>(v, lds, line, tj, LM, Ns, lstride, pstride);
        __syncthreads();
        fft_regs_c<SG, XL, N, S + 1>(v, tj, line, lds, lstride, pstride, tw);
    }
}

// The same for a length with a factor 3, whose stages do not share one set of
// positions per thread: thread tj of the line's T takes butterflies tj, tj + T,
// ... of each stage.  The first stage reads position p through ld(p), the last
// writes through st(p, value); LDS carries the exchanges between stages and may
// also be what ld reads (FROM_LDS: a barrier before the first write to it).
// Against the LDS form above, whose threads hold one butterfly of the smallest
// radix: no staging of input and output, indices known at compile time, and
// threads that all work in the radix-8 stages (of n/3 per line, 3/8 did).  The
// FFT passes of a mixed-precision step, us: 96^3 64 -> 54, 192^3 242 -> 164,
// 384^3 2025 -> 1160, 432^3 4272 -> 1880 (bound by memory from 192^3 on: 3.9-5.3
// TB/s in the y passes).  Holding the least common multiple of the radices
// per thread (24 points, no exchange between forward and inverse in the z pass)
// left too few wavefronts: 192^3 186, 384^3 1258 us.
template <int SG, bool XL, int N, bool FROM_LDS, int S = 0, typename LD, typename ST>
__device__ __forceinline__ void fft_threes(int tj, int line, double2 *lds, int lstride, int pstride,
                                           const double2 *__restrict__ tw, LD &&ld, ST &&st)
{
    constexpr CPlan P = cplan(N);
    constexpr int T = line_threads(N), R = P.R[S], Ns = P.Ns[S], L = N / R, Q = (L + T - 1) / T;
    constexpr bool last = S + 1 == P.nst;
    double2 x[Q][R];
#pragma unroll
    for (int q = 0; q < Q; q++) {
        const int j = tj + q * T;
        if (L % T == 0 || j < L)
#pragma unroll
            for (int r = 0; r < R; r++) {
                if constexpr (S == 0) x[q][r] = ld(j + r * L);
                else x[q][r] = lds[rlds<XL>(line, j + r * L, lstride, pstride)];
            }
    }
    if (S > 0 || FROM_LDS) __syncthreads();
#pragma unroll
    for (int q = 0; q < Q; q++) {
        const int j = tj + q * T;
        if (L % T == 0 || j < L) {
            const unsigned k = (unsigned)j % (unsigned)Ns;
            if constexpr (S > 0)
#pragma unroll
                for (int r = 1; r < R; r++) {
                    const double2 wv = tw[P.off[S] + (int)k * (R - 1) + r - 1];
                    const double wi = SG < 0 ? -wv.y : wv.y;
                    const double xr = x[q][r].x, xi = x[q][r].y;
                    x[q][r] = make_double2(xr * wv.x - xi * wi, xr * wi + xi * wv.x);
                }
            dft<R, SG>(x[q]);
            const int base = (int)(((unsigned)j - k) * R + k);
#pragma unroll
            for (int r = 0; r < R; r++) {
                if constexpr (last) st(base + r * Ns, x[q][r]);
                else lds[rlds<XL>(line, base + r * Ns, lstride, pstride)] = x[q][r];
            }
        }
    }
    if constexpr (!last) {
        __syncthreads();
        fft_threes<SG, XL, N, false, S + 1>(tj, line, lds, lstride, pstride, tw, ld, st);
    }
}

// All stages of one line of a power of two: the compile-time plan for N > 0,
// else the runtime plan pl.
template <int SG, bool XL, int N>
__device__ __forceinline__ void fft_lines(double2 (&v)[8], int tj, int line, double2 *lds, int lstride,
                                          int pstride, const FftPlan &pl, const double2 *__restrict__ tw)
{
    if constexpr (N > 0) fft_regs_c<SG, XL, N>(v, tj, line, lds, lstride, pstride, tw);
    else fft_regs<SG, XL>(v, tj, line, lds, lstride, pstride, pl, tw);
}

__host__ __device__ constexpr int rline_stride(int n) { return n + n / 8 + 1; }

// Default launch shapes of the register kernels: columns per block of the y/z
// passes and x-line pairs per block (threads = shape * line_threads <= 1024, pairs
// dividing n*n/2).  A column tile keeps whole 128-byte lines (8 columns) up to
// 2*LDS_CAP of LDS, one block per CU: at 1024 rows that beats two blocks of
// 4-column tiles, whose 64-byte row pieces half-use each line (z pass 5.9 ->
// 5.4 ms at 1024^3).  Line pairs stay within LDS_CAP; with a factor 3 within
// 28 KB, five blocks per CU (forward x pass of 384^3 FP64 with 8, 4, 2 pairs:
// 404, 372, 415 us; 432^3 with 4, 2, 1: 704, 614, 670 us).
static constexpr int rtile_n(int n)
{
    int t = 8;
    while (t > 1 && t * line_threads(n) > FFT_MAX_THREADS) t >>= 1;
    while (t > 1 && (size_t)t * n * sizeof(double2) > 2 * LDS_CAP) t >>= 1;
    return t;
}
static constexpr int rpairs_n(int n)
{
    int p = 8;
    while (p > 1 && p * line_threads(n) > FFT_MAX_THREADS) p >>= 1;
    const size_t cap = is_pow2(n) ? LDS_CAP : 28 * 1024;
    while (p > 1 && (size_t)p * rline_stride(n) * sizeof(double2) > cap) p >>= 1;
    while (p > 1 && (n * n / 2) % p != 0) p >>= 1;
    return p;
}
// Most threads a block of the kernel for N is launched with (N = 0: any power
// of two): x passes up to 16 pairs, column passes their default tile.
static constexpr int x_threads(int n)
{
    return n == 0 || is_pow2(n) ? FFT_MAX_THREADS : std::min(FFT_MAX_THREADS, (16 * line_threads(n) + 63) / 64 * 64);
}
static constexpr int col_threads(int n)
{
    return n == 0 || is_pow2(n) ? FFT_MAX_THREADS : (rtile_n(n) * line_threads(n) + 63) / 64 * 64;
}

// 16-byte streaming store of one complex value (written once, not re-read by this kernel).
typedef double nt_double2 __attribute__((ext_vector_type(2)));
__device__ __forceinline__ void nt_store2(double2 *dst, double re, double im)
{
    nt_double2 v = {re, im};
    __builtin_nontemporal_store(v, reinterpret_cast<nt_double2 *>(dst));
}

// The value `x` of lane `src` of this wavefront: a cross-lane permute
// (ds_bpermute over the LDS crossbar; no LDS allocation, no barrier).
__device__ __forceinline__ double2 lane_get2(double2 x, int src)
{
    return make_double2(__shfl(x.x, src, 64), __shfl(x.y, src, 64));
}

// The x passes pair position q of a line with its Hermitian mirror n - q.  A
// line of n <= 512 points sits in LM = n/8 consecutive lanes of one
// wavefront, thread tj holding positions tj + m*LM; for tj > 0 the mirror of
// tj + m*LM is (LM - tj) + (7 - m)*LM, held by lane LM - tj of the line in
// slot 7 - m, and for tj = 0 the mirror of m*LM is (8 - m)*LM, the thread's
// own slot 8 - m.  So the mirror comes from one permute of slot 7 - m.
__device__ __forceinline__ int mirror_lane(int tj, int LM)
{
    return (int)(threadIdx.x & 63) - tj + ((LM - tj) & (LM - 1));
}

// Poisson right-hand side (main.f90:715-750) at points (i, j, k) and (i, j+1, k).
template <typename T>
__device__ __forceinline__ double2 poisson_rhs(const T *__restrict__ us, const T *__restrict__ vs,
                                               const T *__restrict__ ws, int i, int j, int k, int kp, int n, double cdiv,
                                               int fp32)
{
    const int ip = i + 1 == n ? 0 : i + 1;
    double rr[2];
#pragma unroll
    for (int h = 0; h < 2; h++) {
        int jj = j + h;
        int jp = jj + 1 == n ? 0 : jj + 1;
        size_t id = IDX(i, jj, k);
        double r = cdiv * ((double)us[IDX(ip, jj, k)] - (double)us[id]);
        r = r + cdiv * ((double)vs[IDX(i, jp, k)] - (double)vs[id]);
        r = r + cdiv * ((double)ws[IDX(i, jj, kp)] - (double)ws[id]);
        if (fp32) r = (double)(float)r;
        rr[h] = r;
    }
    return make_double2(rr[0], rr[1]);
}

// The spectrum of two real lines transformed as one, a thread's 8 positions of
// it in v, split into the lines' half spectra (q = 0 .. n/2); z[n-q] comes from
// the mirror lane.  put(line, q, re, im).
template <typename Put>
__device__ __forceinline__ void split_pair(const double2 (&v)[8], int tj, int LM, int half, Put &&put)
{
    const int src = mirror_lane(tj, LM);
#pragma unroll
    for (int m = 0; m < 4; m++) {
        const int q = tj + m * LM;
        double2 zm = lane_get2(v[7 - m], src);
        if (tj == 0) zm = v[(8 - m) & 7];
        const double a = v[m].x, b = v[m].y, cc = zm.x, d = zm.y;
        put(0, q, (a + cc) * 0.5, (b - d) * 0.5);
        put(1, q, (b + d) * 0.5, (cc - a) * 0.5);
    }
    if (tj == 0) {                        // q = n/2, its own mirror
        const double a = v[4].x, b = v[4].y, cc = v[4].x, d = v[4].y;
        put(0, half, (a + cc) * 0.5, (b - d) * 0.5);
        put(1, half, (b + d) * 0.5, (cc - a) * 0.5);
    }
}

// The reverse: a thread's 8 positions of the joint spectrum of the half spectra
// s1, s2.  Each value is loaded once: positions below n/2 directly, their
// mirrors (slots 4..7) from the mirror lane by a permute.
__device__ __forceinline__ void join_pair(const double2 *s1, const double2 *s2, double2 (&v)[8], int tj, int LM, int half)
{
    double2 A[4], B[4];
#pragma unroll
    for (int m = 0; m < 4; m++) {
        A[m] = s1[tj + m * LM];
        B[m] = s2[tj + m * LM];
    }
    const int src = mirror_lane(tj, LM);
#pragma unroll
    for (int m = 0; m < 4; m++) {
        const double2 a = A[m], b = B[m];
        v[m] = tj + m * LM == 0 ? make_double2(a.x, b.x) : make_double2(a.x - b.y, a.y + b.x);
    }
#pragma unroll
    for (int m = 4; m < 8; m++) {
        double2 a = lane_get2(A[7 - m], src), b = lane_get2(B[7 - m], src);
        if (tj == 0) {
            if (m == 4) { a = s1[half]; b = s2[half]; }
            else { a = A[8 - m]; b = B[8 - m]; }
        }
        v[m] = (tj == 0 && m == 4) ? make_double2(a.x, b.x) : make_double2(a.x + b.y, b.x - a.y);
    }
}

template <typename T, int N = 0>
__device__ __forceinline__ void k_xfwd_r_body(uint3 blk,
    const T *__restrict__ us, const T *__restrict__ vs, const T *__restrict__ ws,
    double2 *__restrict__ spec, const double2 *__restrict__ tw, const Scalars *__restrict__ sc,
    Consts c, FftPlan pl, int ppb, int ld)
{
    const bool stop = halted(sc);
    extern __shared__ double2 lds[];
    const int n = N ? N : c.n, half = n / 2, nh = n / 2 + 1, LM = N ? line_threads(N) : n / 8;
    const int lstride = rline_stride(n);
    const int t = threadIdx.x, pl_ = t / LM, tj = t - pl_ * LM;
    const int pair = blk.x * ppb + pl_;
    const int k = pair / half, j = 2 * (pair - k * half);
    const int kp = k + 1 == n ? 0 : k + 1;
    const double cdiv = c.rho * c.dxi / c.dt;
    auto rhs = [&](int i) { return poisson_rhs(us, vs, ws, i, j, k, kp, n, cdiv, c.fp32_rhs); };
    double2 v[8];
    if constexpr (N > 0 && !is_pow2(N)) {
        fft_threes<-1, true, N, false>(tj, pl_, lds, lstride, 1, tw, rhs, [&](int p, double2 z) {
            lds[rlds<true>(pl_, p, lstride, 1)] = z;
        });
        __syncthreads();
    } else {
#pragma unroll
        for (int m = 0; m < 8; m++) v[m] = rhs(tj + m * LM);
        fft_lines<-1, true, N>(v, tj, pl_, lds, lstride, 1, pl, tw);
        if (stop) return;
        if (LM <= 64) {
            double2 *r1 = spec + spec_row(k, j, n, ld), *r2 = spec + spec_row(k, j + 1, n, ld);
            split_pair(v, tj, LM, half, [&](int h, int q, double re, double im) { nt_store2(&(h ? r2 : r1)[q], re, im); });
            return;
        }
#pragma unroll
        for (int m = 0; m < 8; m++) lds[rlds<true>(pl_, tj + m * LM, lstride, 1)] = v[m];
        __syncthreads();
    }
    if (stop) return;
    for (int e = t; e < ppb * nh; e += blockDim.x) {
        int pq = e / nh, q = e - pq * nh;
        int pr = blk.x * ppb + pq;
        int kk = pr / half, jj = 2 * (pr - kk * half);
        int mq = q == 0 ? 0 : n - q;
        double2 zq = lds[rlds<true>(pq, q, lstride, 1)], zm = lds[rlds<true>(pq, mq, lstride, 1)];
        double a = zq.x, b = zq.y, cc = zm.x, d = zm.y;
        nt_store2(&spec[spec_row(kk, jj, n, ld) + q], (a + cc) * 0.5, (b - d) * 0.5);
        nt_store2(&spec[spec_row(kk, jj + 1, n, ld) + q], (b + d) * 0.5, (cc - a) * 0.5);
    }
}

// With a factor 3, at most 4 waves per SIMD: left to itself the compiler holds
// some lengths to 46 VGPRs and waits for each load (48^3 FP64: 13.3 -> 7.2 us).
template <typename T, int N>
__global__ void __launch_bounds__(x_threads(N)) __attribute__((amdgpu_waves_per_eu(1, N && !is_pow2(N) ? 4 : 8))) k_xfwd_r(
    const T *__restrict__ us, const T *__restrict__ vs, const T *__restrict__ ws,
    double2 *__restrict__ spec, const double2 *__restrict__ tw, const Scalars *__restrict__ sc,
    Consts c, FftPlan pl, int ppb, int ld)
{
    k_xfwd_r_body<T, N>(make_uint3(blockIdx.x, blockIdx.y, blockIdx.z), us, vs, ws, spec, tw, sc, c, pl, ppb, ld);
}


// N > 0: n = N and TK columns per block, both compile-time
template <int SG, int N = 0, int TK = 0>
__device__ __forceinline__ void k_ypass_r_body(uint3 blk, double2 *__restrict__ spec,
                                                             const double2 *__restrict__ tw,
                                                             const Scalars *__restrict__ sc, FftPlan pl, int ld,
                                                             int tkx_)
{
    const bool stop = halted(sc);
    extern __shared__ double2 lds[];
    const int n = N ? N : pl.n, nh = n / 2 + 1, LM = n / 8, tkx = TK ? TK : tkx_;
    const int q0 = blk.x * tkx, k = blk.y;
    const int t = threadIdx.x, line = t % tkx, tj = t / tkx;
    const bool ok = q0 + line < nh;
    double2 *base = spec + spec_row(k, 0, n, ld) + q0 + line;
    if constexpr (N > 0 && !is_pow2(N)) {
        fft_threes<SG, false, N, false>(
            tj, line, lds, 1, tkx, tw,
            [&](int p) { return ok ? base[(size_t)p * ld] : make_double2(0.0, 0.0); },
            [&](int p, double2 z) { if (ok && !stop) nt_store2(&base[(size_t)p * ld], z.x, z.y); });
        return;
    }
    double2 v[8];
#pragma unroll
    for (int m = 0; m < 8; m++) v[m] = ok ? base[(size_t)(tj + m * LM) * ld] : make_double2(0.0, 0.0);
    if constexpr (N == 0 || is_pow2(N)) fft_lines<SG, false, N>(v, tj, line, lds, 1, tkx, pl, tw);
    if (ok && !stop) {
#pragma unroll
        for (int m = 0; m < 8; m++) nt_store2(&base[(size_t)(tj + m * LM) * ld], v[m].x, v[m].y);
    }
}

template <int SG, int N, int TK>
__global__ void __launch_bounds__(col_threads(N)) k_ypass_r(double2 *__restrict__ spec,
                                                             const double2 *__restrict__ tw,
                                                             const Scalars *__restrict__ sc, FftPlan pl, int ld,
                                                             int tkx)
{
    k_ypass_r_body<SG, N, TK>(make_uint3(blockIdx.x, blockIdx.y, blockIdx.z), spec, tw, sc, pl, ld, tkx);
}


template <bool INV_ONLY = false, int N = 0, int TK = 0>
__device__ __forceinline__ void k_zpoisson_r_body(uint3 blk, double2 *__restrict__ spec,
                                                                const double2 *__restrict__ tw,
                                                                const double *__restrict__ ktab,
                                                                const Scalars *__restrict__ sc, FftPlan pl, int ld,
                                                                int tkx_)
{
    const bool stop = halted(sc);
    extern __shared__ double2 lds[];
    const int n = N ? N : pl.n, nh = n / 2 + 1, LM = n / 8, tkx = TK ? TK : tkx_;
    const int q0 = blk.x * tkx, j = blk.y;
    const int t = threadIdx.x, line = t % tkx, tj = t / tkx;
    const int q = q0 + line;
    const bool ok = q < nh;
    const size_t rs = spec_plane(n, ld);
    double2 *base = spec + (size_t)j * ld + q;
    const double nnn = (double)((long long)n * (long long)n * (long long)n);
    const double ky = ktab[j], kx = ktab[ok ? q : 0];
    auto solve = [&](int r, double2 z) {        // the divide by -k^2 and N^3 at row r
        double kz = ktab[r];
        double k2 = (kx * kx + ky * ky) + kz * kz;
        z = make_double2(((-z.x) / k2) / nnn, ((-z.y) / k2) / nnn);
        if (q == 0 && j == 0 && r == 0) z = make_double2(0.0, 0.0);
        return z;
    };
    if constexpr (N > 0 && !is_pow2(N)) {
        static_assert(!INV_ONLY, "the generator's inverse runs the other forms");
        fft_threes<-1, false, N, false>(
            tj, line, lds, 1, tkx, tw,
            [&](int p) { return ok ? base[(size_t)p * rs] : make_double2(0.0, 0.0); },
            [&](int p, double2 z) { lds[rlds<false>(line, p, 1, tkx)] = solve(p, z); });
        __syncthreads();
        fft_threes<1, false, N, true>(
            tj, line, lds, 1, tkx, tw, [&](int p) { return lds[rlds<false>(line, p, 1, tkx)]; },
            [&](int p, double2 z) { if (ok && !stop) nt_store2(&base[(size_t)p * rs], z.x, z.y); });
    } else {
        double2 v[8];
#pragma unroll
        for (int m = 0; m < 8; m++) v[m] = ok ? base[(size_t)(tj + m * LM) * rs] : make_double2(0.0, 0.0);
        if constexpr (!INV_ONLY) {
            fft_lines<-1, false, N>(v, tj, line, lds, 1, tkx, pl, tw);
#pragma unroll
            for (int m = 0; m < 8; m++) v[m] = solve(tj + m * LM, v[m]);
        }
        fft_lines<1, false, N>(v, tj, line, lds, 1, tkx, pl, tw);
        if (ok && !stop) {
#pragma unroll
            for (int m = 0; m < 8; m++) nt_store2(&base[(size_t)(tj + m * LM) * rs], v[m].x, v[m].y);
        }
    }
}

__global__ void __launch_bounds__(FFT_MAX_THREADS) k_zinv_r(double2 *__restrict__ spec,
                                                            const double2 *__restrict__ tw,
                                                            const double *__restrict__ ktab,
                                                            const Scalars *__restrict__ sc, FftPlan pl, int ld,
                                                            int tkx)
{
    k_zpoisson_r_body<true>(make_uint3(blockIdx.x, blockIdx.y, blockIdx.z), spec, tw, ktab, sc, pl, ld, tkx);
}

__global__ void __launch_bounds__(FFT_MAX_THREADS) k_zinv(double2 *__restrict__ spec,
                                                          const double2 *__restrict__ tw,
                                                          const double *__restrict__ ktab,
                                                          const Scalars *__restrict__ sc, FftPlan pl, int ld,
                                                          int tkx)
{
    k_zpoisson_body<true>(make_uint3(blockIdx.x, blockIdx.y, blockIdx.z), spec, tw, ktab, sc, pl, ld, tkx);
}

template <int N, int TK>
__global__ void __launch_bounds__(col_threads(N)) k_zpoisson_r(double2 *__restrict__ spec,
                                                                const double2 *__restrict__ tw,
                                                                const double *__restrict__ ktab,
                                                                const Scalars *__restrict__ sc, FftPlan pl, int ld,
                                                                int tkx)
{
    k_zpoisson_r_body<false, N, TK>(make_uint3(blockIdx.x, blockIdx.y, blockIdx.z), spec, tw, ktab, sc, pl, ld,
                                    tkx);
}


template <int N = 0>
__device__ __forceinline__ void k_xinv_r_body(uint3 blk, const double2 *__restrict__ spec,
                                                            double *__restrict__ p, const double2 *__restrict__ tw,
                                                            const Scalars *__restrict__ sc, FftPlan pl, int ppb,
                                                            int ld)
{
    const bool stop = halted(sc);
    extern __shared__ double2 lds[];
    const int n = N ? N : pl.n, half = n / 2, LM = N ? line_threads(N) : n / 8;
    const int lstride = rline_stride(n);
    const int t = threadIdx.x, pl_ = t / LM, tj = t - pl_ * LM;
    const int pair = blk.x * ppb + pl_;
    const int k = pair / half, j = 2 * (pair - k * half);
    const double2 *s1 = spec + spec_row(k, j, n, ld);
    const double2 *s2 = spec + spec_row(k, j + 1, n, ld);
    if constexpr (N > 0 && !is_pow2(N)) {
        // the half spectra of the block's pairs into LDS, each value read once
        for (int e = t; e < ppb * (half + 1); e += blockDim.x) {
            const int pq = e / (half + 1), q = e - pq * (half + 1);
            const int pr = blk.x * ppb + pq, kk = pr / half, jj = 2 * (pr - kk * half);
            const double2 a = spec[spec_row(kk, jj, n, ld) + q], b = spec[spec_row(kk, jj + 1, n, ld) + q];
            const bool own = q == 0 || q == half;                  // its own mirror
            lds[rlds<true>(pq, q, lstride, 1)] = own ? make_double2(a.x, b.x) : make_double2(a.x - b.y, a.y + b.x);
            if (!own) lds[rlds<true>(pq, n - q, lstride, 1)] = make_double2(a.x + b.y, b.x - a.y);
        }
        __syncthreads();
        fft_threes<1, true, N, true>(
            tj, pl_, lds, lstride, 1, tw, [&](int q) { return lds[rlds<true>(pl_, q, lstride, 1)]; },
            [&](int i, double2 z) {
                if (stop) return;
                __builtin_nontemporal_store(z.x, &p[IDX(i, j, k)]);
                __builtin_nontemporal_store(z.y, &p[IDX(i, j + 1, k)]);
            });
        return;
    }
    double2 v[8];
    if (LM <= 64) {
        join_pair(s1, s2, v, tj, LM, half);
    } else {
#pragma unroll
        for (int m = 0; m < 8; m++) {
            const int q = tj + m * LM;
            double2 z;
            if (q == 0 || q == half) {
                z = make_double2(s1[q].x, s2[q].x);
            } else if (q < half) {
                double2 a = s1[q], b = s2[q];
                z = make_double2(a.x - b.y, a.y + b.x);
            } else {
                int mm = n - q;
                double2 a = s1[mm], b = s2[mm];
                z = make_double2(a.x + b.y, b.x - a.y);
            }
            v[m] = z;
        }
    }
    if constexpr (N == 0 || is_pow2(N)) fft_lines<1, true, N>(v, tj, pl_, lds, lstride, 1, pl, tw);
    if (stop) return;
#pragma unroll
    for (int m = 0; m < 8; m++) {
        const int i = tj + m * LM;
        __builtin_nontemporal_store(v[m].x, &p[IDX(i, j, k)]);
        __builtin_nontemporal_store(v[m].y, &p[IDX(i, j + 1, k)]);
    }
}

template <int N>
__global__ void __launch_bounds__(x_threads(N)) k_xinv_r(const double2 *__restrict__ spec,
                                                            double *__restrict__ p, const double2 *__restrict__ tw,
                                                            const Scalars *__restrict__ sc, FftPlan pl, int ppb,
                                                            int ld)
{
    // last pairs first: the y inverse pass wrote the highest planes last, and
    // some of them are still in the memory-side cache
    k_xinv_r_body<N>(make_uint3(gridDim.x - 1 - blockIdx.x, blockIdx.y, blockIdx.z), spec, p, tw, sc, pl, ppb, ld);
}


// ---------------------------------------------------------------------------
// Small boxes (n <= PLANE_MAX): the x and y passes of a plane in one block, the
// plane's half spectrum (n rows of n/2+1) in LDS between them.  These passes are
// bound by the latency of a launch and a memory round trip each, not by what
// they move (times at plane_fwd_alone).  Arithmetic and its order are those of
// the separate passes.  Threads past the last line repeat the last line's work
// and store nothing to memory.
// ---------------------------------------------------------------------------
constexpr int PLANE_MAX = 64;
__host__ __device__ constexpr int plane_threads(int n) { return ((n / 2 + 1) * line_threads(n) + 63) / 64 * 64; }
__host__ __device__ constexpr size_t plane_lds(int n)     // x lines in exchange order, then the spectrum rows
{
    return sizeof(double2) * ((size_t)(n / 2) * rline_stride(n) + (size_t)n * (n / 2 + 1));
}

template <typename T, int N>
__device__ __forceinline__ void k_plane_fwd_body(int k, const T *__restrict__ us, const T *__restrict__ vs,
                                                 const T *__restrict__ ws, double2 *__restrict__ spec,
                                                 const double2 *__restrict__ tw, const Scalars *__restrict__ sc,
                                                 const Consts &c, int ld)
{
    const bool stop = halted(sc);
    extern __shared__ double2 lds[];
    constexpr int n = N, half = N / 2, nh = half + 1, LM = line_threads(N), lstride = rline_stride(N);
    double2 *xl = lds, *rows = lds + half * lstride;
    const int t = threadIdx.x;
    {
        const int pl_ = min(t / LM, half - 1), tj = t % LM, j = 2 * pl_;
        const int kp = k + 1 == n ? 0 : k + 1;
        const double cdiv = c.rho * c.dxi / c.dt;
        auto rhs = [&](int i) { return poisson_rhs(us, vs, ws, i, j, k, kp, n, cdiv, c.fp32_rhs); };
        if constexpr (is_pow2(N)) {
            double2 v[8];
#pragma unroll
            for (int m = 0; m < 8; m++) v[m] = rhs(tj + m * LM);
            fft_regs_c<-1, true, N>(v, tj, pl_, xl, lstride, 1, tw);
            split_pair(v, tj, LM, half, [&](int h, int q, double re, double im) {
                rows[(j + h) * nh + q] = make_double2(re, im);
            });
        } else {
            fft_threes<-1, true, N, false>(tj, pl_, xl, lstride, 1, tw, rhs, [&](int p, double2 z) {
                xl[rlds<true>(pl_, p, lstride, 1)] = z;
            });
            __syncthreads();
            for (int e = t; e < half * nh; e += blockDim.x) {
                const int pq = e / nh, q = e - pq * nh, mq = q == 0 ? 0 : n - q;
                const double2 zq = xl[rlds<true>(pq, q, lstride, 1)], zm = xl[rlds<true>(pq, mq, lstride, 1)];
                const double a = zq.x, b = zq.y, cc = zm.x, d = zm.y;
                rows[2 * pq * nh + q] = make_double2((a + cc) * 0.5, (b - d) * 0.5);
                rows[(2 * pq + 1) * nh + q] = make_double2((b + d) * 0.5, (cc - a) * 0.5);
            }
        }
    }
    __syncthreads();
    const int line = t % nh, tj = min(t / nh, LM - 1);
    const bool ok = t < nh * LM && !stop;
    double2 *out = spec + spec_row(k, 0, n, ld) + line;
    if constexpr (is_pow2(N)) {
        double2 v[8];
#pragma unroll
        for (int m = 0; m < 8; m++) v[m] = rows[(tj + m * LM) * nh + line];
        __syncthreads();
        fft_regs_c<-1, false, N>(v, tj, line, rows, 1, nh, tw);
        if (ok) {
#pragma unroll
            for (int m = 0; m < 8; m++) nt_store2(&out[(size_t)(tj + m * LM) * ld], v[m].x, v[m].y);
        }
    } else {
        fft_threes<-1, false, N, true>(
            tj, line, rows, 1, nh, tw, [&](int p) { return rows[p * nh + line]; },
            [&](int p, double2 z) { if (ok) nt_store2(&out[(size_t)p * ld], z.x, z.y); });
    }
}

template <int N>
__device__ __forceinline__ void k_plane_inv_body(int k, const double2 *__restrict__ spec, double *__restrict__ p,
                                                 const double2 *__restrict__ tw, const Scalars *__restrict__ sc, int ld)
{
    const bool stop = halted(sc);
    extern __shared__ double2 lds[];
    constexpr int n = N, half = N / 2, nh = half + 1, LM = line_threads(N), lstride = rline_stride(N);
    double2 *xl = lds, *rows = lds + half * lstride;
    const int t = threadIdx.x;
    {
        const int line = t % nh, tj = min(t / nh, LM - 1);
        const double2 *in = spec + spec_row(k, 0, n, ld) + line;
        if constexpr (is_pow2(N)) {
            double2 v[8];
#pragma unroll
            for (int m = 0; m < 8; m++) v[m] = in[(size_t)(tj + m * LM) * ld];
            fft_regs_c<1, false, N>(v, tj, line, rows, 1, nh, tw);
#pragma unroll
            for (int m = 0; m < 8; m++) rows[(tj + m * LM) * nh + line] = v[m];
        } else {
            fft_threes<1, false, N, false>(
                tj, line, rows, 1, nh, tw, [&](int r) { return in[(size_t)r * ld]; },
                [&](int r, double2 z) { rows[r * nh + line] = z; });
        }
    }
    __syncthreads();
    const int pl_ = min(t / LM, half - 1), tj = t % LM, j = 2 * pl_;
    const bool ok = t < half * LM && !stop;
    if constexpr (is_pow2(N)) {
        double2 v[8];
        join_pair(rows + j * nh, rows + (j + 1) * nh, v, tj, LM, half);
        fft_regs_c<1, true, N>(v, tj, pl_, xl, lstride, 1, tw);
        if (ok) {
#pragma unroll
            for (int m = 0; m < 8; m++) {
                const int i = tj + m * LM;
                __builtin_nontemporal_store(v[m].x, &p[IDX(i, j, k)]);
                __builtin_nontemporal_store(v[m].y, &p[IDX(i, j + 1, k)]);
            }
        }
    } else {
        for (int e = t; e < half * nh; e += blockDim.x) {
            const int pq = e / nh, q = e - pq * nh;
            const double2 a = rows[2 * pq * nh + q], b = rows[(2 * pq + 1) * nh + q];
            const bool own = q == 0 || q == half;
            xl[rlds<true>(pq, q, lstride, 1)] = own ? make_double2(a.x, b.x) : make_double2(a.x - b.y, a.y + b.x);
            if (!own) xl[rlds<true>(pq, n - q, lstride, 1)] = make_double2(a.x + b.y, b.x - a.y);
        }
        __syncthreads();
        fft_threes<1, true, N, true>(
            tj, pl_, xl, lstride, 1, tw, [&](int q) { return xl[rlds<true>(pl_, q, lstride, 1)]; },
            [&](int i, double2 z) {
                if (!ok) return;
                __builtin_nontemporal_store(z.x, &p[IDX(i, j, k)]);
                __builtin_nontemporal_store(z.y, &p[IDX(i, j + 1, k)]);
            });
    }
}

template <typename T, int N>
__global__ void __launch_bounds__(plane_threads(N)) k_plane_fwd(
    const T *__restrict__ us, const T *__restrict__ vs, const T *__restrict__ ws,
    double2 *__restrict__ spec, const double2 *__restrict__ tw, const Scalars *__restrict__ sc, Consts c, int ld)
{
    k_plane_fwd_body<T, N>(blockIdx.x, us, vs, ws, spec, tw, sc, c, ld);
}

template <int N>
__global__ void __launch_bounds__(plane_threads(N)) k_plane_inv(const double2 *__restrict__ spec,
                                                                double *__restrict__ p, const double2 *__restrict__ tw,
                                                                const Scalars *__restrict__ sc, int ld)
{
    k_plane_inv_body<N>(blockIdx.x, spec, p, tw, sc, ld);
}


// ---------------------------------------------------------------------------
// Projection (main.f90:873-887) with the per-x-line partial sums and
// maxima behind the mean removal and umax.  One 64-wide wavefront per x-line: lane l owns
// i = l, l+64, ..., adds them in that order, then a xor-butterfly combines the
// 64 lanes.  That fixed order is what the oracle's lane-64 sum restates.
// ---------------------------------------------------------------------------
__device__ __forceinline__ double nanmax(double a, double b)
{
    if (a != a) return a;
    if (b != b) return b;
    return a > b ? a : b;
}

// Neumaier's compensated summation step (s, c) += x.
__device__ __forceinline__ void neumaier(double &s, double &c, double x)
{
    double t = s + x;
    if (__builtin_fabs(s) >= __builtin_fabs(x)) c += (s - t) + x;
    else c += (x - t) + s;
    s = t;
}

// The value of lane (this lane XOR OFF) of the wavefront, without a trip
// through the LDS crossbar where the hardware has a direct form: the gfx950
// lane-half swaps for 32 and 16 (each returns both halves; a lane keeps the
// other half's value), DPP row_ror:8 for 8, quad permutes for 2 and 1, and a
// swizzle for 4.
template <int OFF>
__device__ __forceinline__ unsigned lane_xor32(unsigned x)
{
    const unsigned l = threadIdx.x & 63;
    if constexpr (OFF == 32) {
        const auto p = __builtin_amdgcn_permlane32_swap(x, x, false, false);
        return l < 32 ? p[1] : p[0];
    } else if constexpr (OFF == 16) {
        const auto p = __builtin_amdgcn_permlane16_swap(x, x, false, false);
        return (l & 16) ? p[0] : p[1];
    } else if constexpr (OFF == 8) {
        return (unsigned)__builtin_amdgcn_update_dpp(0, (int)x, 0x128, 0xf, 0xf, false);   // row_ror:8
    } else if constexpr (OFF == 4) {
        return (unsigned)__builtin_amdgcn_ds_swizzle((int)x, (4 << 10) | 0x1f);            // xor 4
    } else if constexpr (OFF == 2) {
        return (unsigned)__builtin_amdgcn_update_dpp(0, (int)x, 0x4e, 0xf, 0xf, false);    // quad_perm [2,3,0,1]
    } else {
        static_assert(OFF == 1, "lane_xor: 32, 16, 8, 4, 2 or 1");
        return (unsigned)__builtin_amdgcn_update_dpp(0, (int)x, 0xb1, 0xf, 0xf, false);    // quad_perm [1,0,3,2]
    }
}
template <int OFF>
__device__ __forceinline__ double lane_xor(double x)
{
    const unsigned long long b = (unsigned long long)__double_as_longlong(x);
    const unsigned lo = lane_xor32<OFF>((unsigned)b), hi = lane_xor32<OFF>((unsigned)(b >> 32));
    return __longlong_as_double((long long)(((unsigned long long)hi << 32) | lo));
}

// Sum and max over the 64 lanes in the xor-butterfly order 32, 16, ..., 1
// (every lane ends with the result).  DIRECT: through lane_xor, the form for
// reductions on the critical path (a projection line of 64 points, the plane
// and total sums); otherwise through the LDS crossbar (__shfl_xor), fewer
// VALU instructions where a lane has several points to add first.
template <bool DIRECT = true>
__device__ __forceinline__ double wave_sum(double x)
{
    if constexpr (DIRECT) {
        x = x + lane_xor<32>(x);
        x = x + lane_xor<16>(x);
        x = x + lane_xor<8>(x);
        x = x + lane_xor<4>(x);
        x = x + lane_xor<2>(x);
        x = x + lane_xor<1>(x);
    } else {
#pragma unroll
        for (int off = 32; off >= 1; off >>= 1) x = x + __shfl_xor(x, off, 64);
    }
    return x;
}

template <bool DIRECT = true>
__device__ __forceinline__ double wave_max(double x)
{
    if constexpr (DIRECT) {
        x = nanmax(x, lane_xor<32>(x));
        x = nanmax(x, lane_xor<16>(x));
        x = nanmax(x, lane_xor<8>(x));
        x = nanmax(x, lane_xor<4>(x));
        x = nanmax(x, lane_xor<2>(x));
        x = nanmax(x, lane_xor<1>(x));
    } else {
#pragma unroll
        for (int off = 32; off >= 1; off >>= 1) x = nanmax(x, __shfl_xor(x, off, 64));
    }
    return x;
}

// Four (or two) reductions over the 64 lanes at once, each in the order of
// wave_sum / wave_max: the first exchange puts two lines' halves side by side
// in one register and the next four lines' quarters, so the later steps run
// once for all of them.  On return the 16 lanes of row r hold line
// reduced_line(r): a quarter of the instructions of four butterflies.
template <typename Op>
__device__ __forceinline__ double halves(double x, double y, Op op)      // lanes 0-31 x, 32-63 y
{
    const unsigned long long a = (unsigned long long)__double_as_longlong(x), b = (unsigned long long)__double_as_longlong(y);
    const auto lo = __builtin_amdgcn_permlane32_swap((unsigned)a, (unsigned)b, false, false);
    const auto hi = __builtin_amdgcn_permlane32_swap((unsigned)(a >> 32), (unsigned)(b >> 32), false, false);
    return op(__longlong_as_double((long long)(((unsigned long long)hi[0] << 32) | lo[0])),
              __longlong_as_double((long long)(((unsigned long long)hi[1] << 32) | lo[1])));
}
template <typename Op>
__device__ __forceinline__ double quarters(double x, double y, Op op)    // even rows of 16 lanes x, odd y
{
    const unsigned long long a = (unsigned long long)__double_as_longlong(x), b = (unsigned long long)__double_as_longlong(y);
    const auto lo = __builtin_amdgcn_permlane16_swap((unsigned)a, (unsigned)b, false, false);
    const auto hi = __builtin_amdgcn_permlane16_swap((unsigned)(a >> 32), (unsigned)(b >> 32), false, false);
    return op(__longlong_as_double((long long)(((unsigned long long)hi[0] << 32) | lo[0])),
              __longlong_as_double((long long)(((unsigned long long)hi[1] << 32) | lo[1])));
}
template <int LPW, typename Op>
__device__ __forceinline__ double reduce_lines(const double (&x)[LPW], Op op)
{
    static_assert(LPW == 2 || LPW == 4, "two halves or four quarters");
    double r = halves(x[0], x[1], op);
    if constexpr (LPW == 4) r = quarters(r, halves(x[2], x[3], op), op);
    else r = op(r, lane_xor<16>(r));
    r = op(r, lane_xor<8>(r));
    r = op(r, lane_xor<4>(r));
    r = op(r, lane_xor<2>(r));
    return op(r, lane_xor<1>(r));
}
template <int LPW>
__device__ __forceinline__ int reduced_line(int lane)
{
    return LPW == 4 ? 2 * ((lane >> 4) & 1) + (lane >> 5) : lane >> 5;
}

// A wavefront owns LPW consecutive x-lines of a plane, whose p(j-1) is mostly
// the line before, and reduces them together.  ONE: lines of at most 64 points,
// one per lane (without a loop over the line a lane's value is its sum and
// maximum, and four lines fit the registers; two do otherwise).  PLANE (with
// ONE): a block owns a whole plane and forms its plane sums too, in the order of
// k_reduce_planes.
template <typename T, int LPW, bool ONE, bool PLANE>
__device__ __forceinline__ void k_project_lines(uint3 blk,
    const T *__restrict__ us, const T *__restrict__ vs, const T *__restrict__ ws,
    const double *__restrict__ p, T *__restrict__ u, T *__restrict__ v, T *__restrict__ w,
    double *__restrict__ lsum, double *__restrict__ lmax, const Scalars *__restrict__ sc, Consts c)
{
    const bool stop = halted(sc);
    const int n = c.n;
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, per = n / LPW;
    int j0, k;
    if constexpr (PLANE) {
        j0 = wave * LPW;
        k = blk.x;
    } else {
        const unsigned g = blk.x * (BLK / 64) + wave;
        if (g >= (unsigned)(per * n)) return;
        k = g / per;
        j0 = (g - k * per) * LPW;
    }
    const int km = k == 0 ? n - 1 : k - 1, jm = j0 == 0 ? n - 1 : j0 - 1;
    const double dtr = c.dt / c.rho, dxi = c.dxi;
    double sum[3][LPW], comp[3][LPW], top[3][LPW];     // comp: Neumaier compensation (FP32 storage only)
#pragma unroll
    for (int m = 0; m < 3; m++)
#pragma unroll
        for (int q = 0; q < LPW; q++) { sum[m][q] = comp[m][q] = 0.0; top[m][q] = -__builtin_inf(); }
    auto points = [&](int i) {
        const int im = i == 0 ? n - 1 : i - 1;
        T a[3][LPW];
        double pc[LPW + 1], px[LPW], pz[LPW];          // p at rows j0-1.., at i-1, at k-1
        pc[0] = p[IDX(i, jm, k)];
#pragma unroll
        for (int q = 0; q < LPW; q++) {
            const size_t id = IDX(i, j0 + q, k);
            a[0][q] = us[id]; a[1][q] = vs[id]; a[2][q] = ws[id];
            pc[q + 1] = p[id];
            px[q] = p[IDX(im, j0 + q, k)];
            pz[q] = p[IDX(i, j0 + q, km)];
        }
#pragma unroll
        for (int q = 0; q < LPW; q++) {
            const double p0 = pc[q + 1];
            const T t[3] = {(T)((double)a[0][q] - dtr * (p0 - px[q]) * dxi),
                            (T)((double)a[1][q] - dtr * (p0 - pc[q]) * dxi),
                            (T)((double)a[2][q] - dtr * (p0 - pz[q]) * dxi)};
            const size_t id = IDX(i, j0 + q, k);
            if (!stop) {
                __builtin_nontemporal_store(t[0], &u[id]);
                __builtin_nontemporal_store(t[1], &v[id]);
                __builtin_nontemporal_store(t[2], &w[id]);
            }
#pragma unroll
            for (int m = 0; m < 3; m++) {
                const double x = t[m];
                if constexpr (sizeof(T) == 4) neumaier(sum[m][q], comp[m][q], x);
                else sum[m][q] = sum[m][q] + x;
                top[m][q] = ONE ? x : nanmax(top[m][q], x);
                if constexpr (ONE && sizeof(T) == 4) sum[m][q] = sum[m][q] + comp[m][q];
            }
        }
    };
    if constexpr (ONE) {
        if (lane < n) points(lane);
    } else {
        for (int i = lane; i < n; i += 64) points(i);
    }
    if (stop) return;
    const auto add = [](double x, double y) { return x + y; };
    const auto most = [](double x, double y) { return nanmax(x, y); };
    const size_t nn = (size_t)n * n;
    __shared__ double plane[PLANE ? 6 : 1][PLANE ? 64 : 1];
#pragma unroll
    for (int m = 0; m < 3; m++) {
        if constexpr (!ONE && sizeof(T) == 4)
#pragma unroll
            for (int q = 0; q < LPW; q++) sum[m][q] = sum[m][q] + comp[m][q];
        const double a = reduce_lines(sum[m], add), b = reduce_lines(top[m], most);
        if ((lane & (LPW == 4 ? 15 : 31)) == 0) {
            const int j = j0 + reduced_line<LPW>(lane);
            if constexpr (PLANE) {
                plane[m][j] = a;
                plane[3 + m][j] = b;
            } else {
                lsum[m * nn + (size_t)k * n + j] = a;
                lmax[m * nn + (size_t)k * n + j] = b;
            }
        }
    }
    if constexpr (PLANE) {                     // lsum, lmax: the plane sums and maxima here
        __syncthreads();
        for (int m = wave; m < 6; m += (int)(blockDim.x >> 6)) {
            if (m < 3) {
                const double a = wave_sum(lane < n ? 0.0 + plane[m][lane] : 0.0);
                if (lane == 0) lsum[m * n + k] = a;
            } else {
                const double b = wave_max(lane < n ? plane[m][lane] : -__builtin_inf());
                if (lane == 0) lmax[(m - 3) * n + k] = b;
            }
        }
    }
}

template <typename T>
__device__ __forceinline__ void k_project_body(uint3 blk,
    const T *__restrict__ us, const T *__restrict__ vs, const T *__restrict__ ws,
    const double *__restrict__ p, T *__restrict__ u, T *__restrict__ v, T *__restrict__ w,
    double *__restrict__ lsum, double *__restrict__ lmax, const Scalars *__restrict__ sc, Consts c)
{
    const bool stop = halted(sc);
    const int n = c.n;
    const int lane = threadIdx.x & 63;
    const size_t line = ((size_t)blk.x * BLK + threadIdx.x) >> 6;
    if (line >= (size_t)n * n) return;
    const int j = (int)(line % n), k = (int)(line / n);
    const int jm = j == 0 ? n - 1 : j - 1, km = k == 0 ? n - 1 : k - 1;
    const double dtr = c.dt / c.rho, dxi = c.dxi;
    double su = 0.0, sv = 0.0, sw = 0.0;
    double cu = 0.0, cv = 0.0, cw = 0.0;     // Neumaier compensation (FP32 storage only)
    double mu_ = -__builtin_inf(), mv = -__builtin_inf(), mw = -__builtin_inf();
    for (int i = lane; i < n; i += 64) {
        int im = i == 0 ? n - 1 : i - 1;
        size_t id = IDX(i, j, k);
        double p0 = p[id];
        const T tu = (T)((double)us[id] - dtr * (p0 - p[IDX(im, j, k)]) * dxi);
        const T tv = (T)((double)vs[id] - dtr * (p0 - p[IDX(i, jm, k)]) * dxi);
        const T tw = (T)((double)ws[id] - dtr * (p0 - p[IDX(i, j, km)]) * dxi);
        if (stop) return;
        __builtin_nontemporal_store(tu, &u[id]);
        __builtin_nontemporal_store(tv, &v[id]);
        __builtin_nontemporal_store(tw, &w[id]);
        const double uu = tu, vv = tv, ww = tw;
        if constexpr (sizeof(T) == 4) {
            neumaier(su, cu, uu); neumaier(sv, cv, vv); neumaier(sw, cw, ww);
        } else {
            su = su + uu; sv = sv + vv; sw = sw + ww;
        }
        mu_ = nanmax(mu_, uu); mv = nanmax(mv, vv); mw = nanmax(mw, ww);
    }
    if constexpr (sizeof(T) == 4) { su = su + cu; sv = sv + cv; sw = sw + cw; }
    su = wave_sum<false>(su); sv = wave_sum<false>(sv); sw = wave_sum<false>(sw);
    mu_ = wave_max<false>(mu_); mv = wave_max<false>(mv); mw = wave_max<false>(mw);
    if (lane == 0) {
        const size_t nn = (size_t)n * n;
        lsum[line] = su; lsum[nn + line] = sv; lsum[2 * nn + line] = sw;
        lmax[line] = mu_; lmax[nn + line] = mv; lmax[2 * nn + line] = mw;
    }
}

// The forms of the projection: lines per wavefront, and whether a block forms
// its plane's sums (small boxes; lsum, lmax are then psum, pmax).
struct ProjectForm {
    int lpw;
    bool plane;
};
__host__ __device__ constexpr ProjectForm project_form(int n)
{
    return n <= 48 && n % 4 == 0 ? ProjectForm{4, true} : n <= 128 ? ProjectForm{2, false} : ProjectForm{0, false};
}
__host__ __device__ constexpr int gang_lpw(int n) { return n <= 64 && n % 4 == 0 ? 4 : 2; }
__host__ __device__ constexpr unsigned project_blocks(int n)
{
    const ProjectForm f = project_form(n);
    return f.plane ? n : f.lpw ? (unsigned)((n / f.lpw * n + BLK / 64 - 1) / (BLK / 64)) : (unsigned)(((size_t)n * n * 64 + BLK - 1) / BLK);
}

template <typename T, int LPW, bool PLANE>
__global__ void __launch_bounds__(PLANE ? 1024 : BLK) k_project(
    const T *__restrict__ us, const T *__restrict__ vs, const T *__restrict__ ws,
    const double *__restrict__ p, T *__restrict__ u, T *__restrict__ v, T *__restrict__ w,
    double *__restrict__ lsum, double *__restrict__ lmax, const Scalars *__restrict__ sc, Consts c)
{
    const uint3 b = make_uint3(blockIdx.x, blockIdx.y, blockIdx.z);
    if constexpr (LPW > 0) k_project_lines<T, LPW, PLANE, PLANE>(b, us, vs, ws, p, u, v, w, lsum, lmax, sc, c);
    else k_project_body<T>(b, us, vs, ws, p, u, v, w, lsum, lmax, sc, c);
}


// Per z-plane: lane-64 sum over the n line sums of the plane (y direction).
// One wavefront per (plane, component).
__device__ __forceinline__ void k_reduce_planes_body(uint3 blk, const double *__restrict__ lsum, const double *__restrict__ lmax,
                                                      double *__restrict__ psum, double *__restrict__ pmax,
                                                      const Scalars *__restrict__ sc, int n)
{
    const bool stop = halted(sc);
    const int k = blk.x, comp = blk.y, lane = threadIdx.x;
    const size_t nn = (size_t)n * n;
    const double *ls = lsum + comp * nn + (size_t)k * n;
    const double *lm = lmax + comp * nn + (size_t)k * n;
    double s = 0.0, m = -__builtin_inf();
#pragma unroll 4
    for (int j = lane; j < n; j += 64) {
        s = s + ls[j];
        m = nanmax(m, lm[j]);
    }
    s = wave_sum(s);
    m = wave_max(m);
    if (lane == 0 && !stop) {
        psum[comp * n + k] = s;
        pmax[comp * n + k] = m;
    }
}

__global__ void __launch_bounds__(64) k_reduce_planes(const double *__restrict__ lsum, const double *__restrict__ lmax,
                                                      double *__restrict__ psum, double *__restrict__ pmax,
                                                      const Scalars *__restrict__ sc, int n)
{
    k_reduce_planes_body(make_uint3(blockIdx.x, blockIdx.y, blockIdx.z), lsum, lmax, psum, pmax, sc, n);
}


// Means (main.f90:906-913), signed umax (937-941), CFL (942-945), halt flag.
// One wavefront per sum and maximum.  publish: the last step of a call, which
// the host waits for through the mirror (a write to host memory and the fence
// behind it cost about 1 us).
constexpr int FIN_THREADS = 6 * 64;
__device__ __forceinline__ void k_finalize_body(const double *__restrict__ psum, const double *__restrict__ pmax,
                                                Scalars *__restrict__ sc, const Consts &c, Scalars *mirror, EnsSlot *slot,
                                                int publish)
{
    const bool stop = sc->halted != 0;
    const int n = c.n, lane = threadIdx.x & 63, q = threadIdx.x >> 6;
    __shared__ double part[6];
    if (q < 3) {
        double a = 0.0;
#pragma unroll 4
        for (int k = lane; k < n; k += 64) a = a + psum[q * n + k];
        a = wave_sum(a);
        if (lane == 0) part[q] = a;
    } else {
        double b = -__builtin_inf();
#pragma unroll 4
        for (int k = lane; k < n; k += 64) b = nanmax(b, pmax[(q - 3) * n + k]);
        b = wave_max(b);
        if (lane == 0) part[q] = b;
    }
    __syncthreads();
    if (stop) return;
    if (threadIdx.x == 0) {
        const double s[3] = {part[0], part[1], part[2]}, m[3] = {part[3], part[4], part[5]};
        const double dn = (double)n;
        double gu = s[0] / dn / dn / dn;
        double gv = s[1] / dn / dn / dn;
        double gw = s[2] / dn / dn / dn;
        // max(fl(x - g)) over x equals fl(max(x) - g): rounding is monotone.
        double uc = m[0] - gu, vc = m[1] - gv, wc = m[2] - gw;
        bool nan = (uc != uc) || (vc != vc) || (wc != wc);
        double mx = uc > vc ? uc : vc;
        double gumax = wc > mx ? wc : mx;
        double cou = gumax * c.dt * c.dxi;
        sc->umean = gu;
        sc->vmean = gv;
        sc->wmean = gw;
        sc->gumax = gumax;
        sc->cou = cou;
        const int steps = sc->steps + 1;
        sc->steps = steps;
        const int status = nan ? 6 : cou > 7.0 ? 5 : 0, halt = status != 0;
        if (halt) {
            sc->halted = 1;
            sc->status = status;
        }
        if (publish || halt) {             // the host's copy, its step count last
            mirror->umean = gu;
            mirror->vmean = gv;
            mirror->wmean = gw;
            mirror->gumax = gumax;
            mirror->cou = cou;
            mirror->halted = halt;
            mirror->status = status;
            __threadfence_system();
            *(volatile int *)&mirror->steps = steps;
        }
        if (slot) {
            slot->clk[steps % CLK_RING] = wall_clock64();
            if (halt) slot->halted = 1;
            __threadfence_system();
            slot->steps = steps;
        }
    }
}

__global__ void __launch_bounds__(FIN_THREADS) k_finalize(const double *__restrict__ psum, const double *__restrict__ pmax,
                                                         Scalars *__restrict__ sc, Consts c, Scalars *mirror,
                                                         EnsSlot *slot, int publish)
{
    k_finalize_body(psum, pmax, sc, c, mirror, slot, publish);
}

// ---------------------------------------------------------------------------
// Gang launches: one pass of one step for up to GANG_MAX boxes of the same n,
// precision and phiflag in a single launch.  The box is one more grid
// dimension (folded into z for the marching kernels, so that the XCD-aware
// block order hands each XCD whole boxes); every block loads its box's
// buffers and constants from the descriptor array g and runs the one-box code
// unchanged, so a box gives the same bits in a gang as alone.
// ---------------------------------------------------------------------------
// The place of this block in a gang's shared launch (a 1-D grid): its box,
// the last one whose first block is at or below the block's index, and its
// index among that box's blocks.  Indices run XCD-first (as in xcd_block), so
// each XCD works through consecutive blocks, mostly of one box.
__device__ __forceinline__ unsigned gang_block(const GangGrid &gg, int nbox, unsigned &local)
{
    const unsigned nb = gridDim.x;
    unsigned b = blockIdx.x;
    if (nb % 8 == 0) b = (b % 8) * (nb / 8) + b / 8;
    unsigned box = 0;
    for (int q = 1; q < nbox; q++)
        if ((unsigned)gg.first[q] <= b) box = (unsigned)q;
    local = b - (unsigned)gg.first[box];
    return box;
}

// A pointer field of a descriptor, read as one to device memory: a kernel's own
// pointer arguments are known to be that, one that is read from memory is not,
// and its accesses are flat ones, each with a 64-bit address in VGPRs, and never
// scalar loads.
template <typename T, typename F>
__device__ __forceinline__ T *global_ptr(F *const &field)
{
    return (T *)*reinterpret_cast<__attribute__((address_space(1))) T *const *>((uintptr_t)&field);
}

// Tile coordinates of a box's block `l` in a grid of gx x gy tiles per slab.
__device__ __forceinline__ uint3 tile_of(unsigned l, unsigned gx, unsigned gy)
{
    return make_uint3(l % gx, (l / gx) % gy, l / (gx * gy));
}

template <typename T>
__global__ void __launch_bounds__(ATHREADS, sizeof(T) == 4 ? 8 : 4) kg_acdi(const GangBox *__restrict__ g, int nbox,
                                                                           GangGrid gg)
{
    unsigned l;
    const unsigned box = gang_block(gg, nbox, l);
    const GangBox &B = g[box];
    const unsigned n = (unsigned)B.c.n;
    k_acdi_body<T, false>(tile_of(l, (n + ATX - 1) / ATX, (n + ATY - 1) / ATY), (const T *)B.f.u, (const T *)B.f.v,
                          (const T *)B.f.w, (const T *)B.f.phi, (T *)B.f.phin, B.f.sc, B.f.mtab, B.c, gg.kz[box]);
}

// euler: bit b set when box b takes its first (Euler) step, main.f90:323-324.
// The CSF force uses phi^{n+1} (main.f90:604-658): the buffer the phase pass
// of this step has just written, phin in the step's descriptor.
// At most 128 VGPRs (4 waves per SIMD), as in the one-box kernel, and 2 values
// spilled as there.  With the descriptor's pointers taken as they are (flat
// accesses, the means in VGPRs) it spilled 13, and a step of 8 boxes FP64 with
// phi took 55.0 / 125 / 170 / 589 / 1152 us at 32 / 48 / 64 / 96 / 128^3 instead
// of 52.5 / 115 / 159 / 555 / 1095 (8 rows, two barriers: 55.8 / 125 / 163 / 577 / 1128).
template <int PHI, typename T>
__global__ void __launch_bounds__(MTHREADS, 4) kg_momentum(const GangBox *__restrict__ g, int nbox, unsigned euler,
                                                        GangGrid gg)
{
    unsigned l;
    const unsigned box = gang_block(gg, nbox, l);
    const GangBox &B = g[box];
    const bool eu = (euler >> box) & 1u;
    const unsigned n = (unsigned)B.c.n;
    const int kz = gg.kz[box];
    k_momentum_body<PHI, T>(tile_of(l, (n + MTX - 1) / MTX, (n + MTY - 1) / MTY), global_ptr<const T>(B.f.u),
                            global_ptr<const T>(B.f.v), global_ptr<const T>(B.f.w), global_ptr<const T>(B.f.phin),
                            global_ptr<T>(B.f.us), global_ptr<T>(B.f.vs), global_ptr<T>(B.f.ws), global_ptr<T>(B.f.ruo),
                            global_ptr<T>(B.f.rvo), global_ptr<T>(B.f.rwo), global_ptr<const double>(B.f.sinf),
                            global_ptr<const double>(B.f.cosf), global_ptr<const Scalars>(B.f.sc), B.c, eu ? 1.0 : 1.5, eu ? 0.0 : 0.5, kz);
}

template <int PHI, typename T>
__global__ void __launch_bounds__(PTHREADS) kg_momentum_x2(const GangBox *__restrict__ g, int nbox, unsigned euler,
                                                           GangGrid gg)
{
    unsigned l;
    const unsigned box = gang_block(gg, nbox, l);
    const GangBox &B = g[box];
    const bool eu = (euler >> box) & 1u;
    const unsigned n = (unsigned)B.c.n;
    const int kz = gg.kz[box];
    k_momentum_x2_body<PHI, T>(tile_of(l, (n + 2 * PTX - 1) / (2 * PTX), (n + PTY - 1) / PTY), (const T *)B.f.u,
                               (const T *)B.f.v, (const T *)B.f.w, (const T *)B.f.phin, (T *)B.f.us, (T *)B.f.vs,
                               (T *)B.f.ws, (T *)B.f.ruo, (T *)B.f.rvo, (T *)B.f.rwo, B.f.sinf, B.f.cosf, B.f.sc,
                               B.c, eu ? 1.0 : 1.5, eu ? 0.0 : 0.5, kz);
}

// FFT passes: box = the first grid dimension the one-box launch leaves unused.
template <typename T, bool REGS, int N>
__global__ void __launch_bounds__(x_threads(N)) kg_xfwd(const GangBox *__restrict__ g, FftPlan pl, int ppb, int ld)
{
    const GangBox &B = g[blockIdx.y];
    const uint3 b = make_uint3(blockIdx.x, 0, 0);
    if constexpr (REGS)
        k_xfwd_r_body<T, N>(b, (const T *)B.f.us, (const T *)B.f.vs, (const T *)B.f.ws, B.f.spec, B.f.tw, B.f.sc, B.c,
                         pl, ppb, ld);
    else
        k_xfwd_body<T>(b, (const T *)B.f.us, (const T *)B.f.vs, (const T *)B.f.ws, B.f.spec, B.f.tw, B.f.sc, B.c, pl,
                       ppb, ld);
}

template <int SG, bool REGS, int N>
__global__ void __launch_bounds__(col_threads(N)) kg_ypass(const GangBox *__restrict__ g, FftPlan pl, int ld, int tkx)
{
    const GangBox &B = g[blockIdx.z];
    const uint3 b = make_uint3(blockIdx.x, blockIdx.y, 0);
    if constexpr (REGS)
        k_ypass_r_body<SG, N, N ? rtile_n(N) : 0>(b, B.f.spec, B.f.tw, B.f.sc, pl, ld, tkx);
    else
        k_ypass_body<SG>(b, B.f.spec, B.f.tw, B.f.sc, pl, ld, tkx);
}

template <bool REGS, int N>
__global__ void __launch_bounds__(col_threads(N)) kg_zpoisson(const GangBox *__restrict__ g, FftPlan pl, int ld,
                                                               int tkx)
{
    const GangBox &B = g[blockIdx.z];
    const uint3 b = make_uint3(blockIdx.x, blockIdx.y, 0);
    if constexpr (REGS)
        k_zpoisson_r_body<false, N, N ? rtile_n(N) : 0>(b, B.f.spec, B.f.tw, B.f.ktab, B.f.sc, pl, ld, tkx);
    else
        k_zpoisson_body<false>(b, B.f.spec, B.f.tw, B.f.ktab, B.f.sc, pl, ld, tkx);
}

template <bool REGS, int N>
__global__ void __launch_bounds__(x_threads(N)) kg_xinv(const GangBox *__restrict__ g, FftPlan pl, int ppb, int ld)
{
    const GangBox &B = g[blockIdx.y];
    const uint3 b = make_uint3(blockIdx.x, 0, 0);
    if constexpr (REGS)
        k_xinv_r_body<N>(b, B.f.spec, B.f.p, B.f.tw, B.f.sc, pl, ppb, ld);
    else
        k_xinv_body(b, B.f.spec, B.f.p, B.f.tw, B.f.sc, pl, ppb, ld);
}

template <typename T, int N>
__global__ void __launch_bounds__(plane_threads(N)) kg_plane_fwd(const GangBox *__restrict__ g, int ld)
{
    const GangBox &B = g[blockIdx.y];
    k_plane_fwd_body<T, N>(blockIdx.x, (const T *)B.f.us, (const T *)B.f.vs, (const T *)B.f.ws, B.f.spec, B.f.tw, B.f.sc,
                           B.c, ld);
}

template <int N>
__global__ void __launch_bounds__(plane_threads(N)) kg_plane_inv(const GangBox *__restrict__ g, int ld)
{
    const GangBox &B = g[blockIdx.y];
    k_plane_inv_body<N>(blockIdx.x, B.f.spec, B.f.p, B.f.tw, B.f.sc, ld);
}

// A gang's boxes do not form their plane sums here (a launch has one block size).
template <typename T>
__global__ void __launch_bounds__(BLK) kg_project(const GangBox *__restrict__ g, int nbox, GangGrid gg)
{
    unsigned l;
    const GangBox &B = g[gang_block(gg, nbox, l)];
    const uint3 b = make_uint3(l, 0, 0);
    const T *us = (const T *)B.f.us, *vs = (const T *)B.f.vs, *ws = (const T *)B.f.ws;
    T *u = (T *)B.f.u, *v = (T *)B.f.v, *w = (T *)B.f.w;
    if (gang_lpw(B.c.n) == 4)
        k_project_lines<T, 4, true, false>(b, us, vs, ws, B.f.p, u, v, w, B.f.lsum, B.f.lmax, B.f.sc, B.c);
    else
        k_project_lines<T, 2, false, false>(b, us, vs, ws, B.f.p, u, v, w, B.f.lsum, B.f.lmax, B.f.sc, B.c);
}

__global__ void __launch_bounds__(64) kg_reduce_planes(const GangBox *__restrict__ g, int nbox, GangGrid gg)
{
    unsigned l;
    const GangBox &B = g[gang_block(gg, nbox, l)];
    const unsigned n = (unsigned)B.c.n;
    k_reduce_planes_body(make_uint3(l % n, l / n, 0), B.f.lsum, B.f.lmax, B.f.psum, B.f.pmax, B.f.sc,
                         B.c.n);
}

__global__ void __launch_bounds__(FIN_THREADS) kg_finalize(const GangBox *__restrict__ g, int publish)
{
    const GangBox &B = g[blockIdx.x];
    k_finalize_body(B.f.psum, B.f.pmax, B.f.sc, B.c, B.f.mirror, B.f.slot, publish);
}


// ---------------------------------------------------------------------------
// On-device diagnostics: kinetic energy 0.5<u.u>, the dissipation
// 2 nu <S_ij S_ij> of post/compute_diss/main.f90:61-117 (central differences
// on the collocated grid with a caller-given 1/dx) and the phase sum.  One
// wavefront per x-line, then per plane, then one for the total.
// ---------------------------------------------------------------------------
template <typename T>
__global__ void __launch_bounds__(BLK) k_diag_lines(const T *__restrict__ u, const T *__restrict__ v,
                                                    const T *__restrict__ w, const T *__restrict__ phi,
                                                    double *__restrict__ lsum, const Scalars *__restrict__ sc,
                                                    Consts c, double dxi)
{
    const int n = c.n;
    const int lane = threadIdx.x & 63;
    const size_t line = ((size_t)blockIdx.x * BLK + threadIdx.x) >> 6;
    if (line >= (size_t)n * n) return;
    const int j = (int)(line % n), k = (int)(line / n);
    const int jp = j + 1 == n ? 0 : j + 1, jm = j == 0 ? n - 1 : j - 1;
    const int kp = k + 1 == n ? 0 : k + 1, km = k == 0 ? n - 1 : k - 1;
    const double um = sc->umean, vm = sc->vmean, wm = sc->wmean;
    double ke = 0.0, ss = 0.0, ph = 0.0;
    for (int i = lane; i < n; i += 64) {
        const int ip = i + 1 == n ? 0 : i + 1, im = i == 0 ? n - 1 : i - 1;
#define DU(f, m, a, b, cc) ((double)f[IDX(a, b, cc)] - m)
        const double u0 = DU(u, um, i, j, k), v0 = DU(v, vm, i, j, k), w0 = DU(w, wm, i, j, k);
        const double dudx = (DU(u, um, ip, j, k) - DU(u, um, im, j, k)) * 0.5 * dxi;
        const double dudy = (DU(u, um, i, jp, k) - DU(u, um, i, jm, k)) * 0.5 * dxi;
        const double dudz = (DU(u, um, i, j, kp) - DU(u, um, i, j, km)) * 0.5 * dxi;
        const double dvdx = (DU(v, vm, ip, j, k) - DU(v, vm, im, j, k)) * 0.5 * dxi;
        const double dvdy = (DU(v, vm, i, jp, k) - DU(v, vm, i, jm, k)) * 0.5 * dxi;
        const double dvdz = (DU(v, vm, i, j, kp) - DU(v, vm, i, j, km)) * 0.5 * dxi;
        const double dwdx = (DU(w, wm, ip, j, k) - DU(w, wm, im, j, k)) * 0.5 * dxi;
        const double dwdy = (DU(w, wm, i, jp, k) - DU(w, wm, i, jm, k)) * 0.5 * dxi;
        const double dwdz = (DU(w, wm, i, j, kp) - DU(w, wm, i, j, km)) * 0.5 * dxi;
#undef DU
        const double s12 = 0.5 * (dudy + dvdx), s13 = 0.5 * (dudz + dwdx), s23 = 0.5 * (dvdz + dwdy);
        ss = ss + dudx * dudx + dvdy * dvdy + dwdz * dwdz + 2.0 * ((s12 * s12 + s13 * s13) + s23 * s23);
        ke = ke + ((u0 * u0 + v0 * v0) + w0 * w0);
        if (phi) ph = ph + (double)phi[IDX(i, j, k)];
    }
    ke = wave_sum(ke); ss = wave_sum(ss); ph = wave_sum(ph);
    if (lane == 0) {
        const size_t nn = (size_t)n * n;
        lsum[line] = ke; lsum[nn + line] = ss; lsum[2 * nn + line] = ph;
    }
}

__global__ void __launch_bounds__(64) k_diag_planes(const double *__restrict__ lsum, double *__restrict__ psum, int n)
{
    const int k = blockIdx.x, comp = blockIdx.y, lane = threadIdx.x;
    const double *ls = lsum + comp * (size_t)n * n + (size_t)k * n;
    double a = 0.0;
    for (int j = lane; j < n; j += 64) a = a + ls[j];
    a = wave_sum(a);
    if (lane == 0) psum[comp * n + k] = a;
}

__global__ void __launch_bounds__(64) k_diag_total(const double *__restrict__ psum, double *__restrict__ out, int n)
{
    const int lane = threadIdx.x;
#pragma unroll
    for (int comp = 0; comp < 3; comp++) {
        double a = 0.0;
        for (int k = lane; k < n; k += 64) a = a + psum[comp * n + k];
        a = wave_sum(a);
        if (lane == 0) out[comp] = a;
    }
}

// Diagnostic: the device's elementary functions on an array of arguments.
__global__ void k_debug_math(int op, size_t count, const double *__restrict__ x, double *__restrict__ y,
                             const double *__restrict__ mtab)
{
    size_t t = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= count) return;
    double a = x[t];
    double r;
    switch (op) {
    case 0: r = dlog(a, mtab); break;
    case 1: r = dtanh(a, mtab); break;
    case 2: r = sqrt(a); break;
    default: r = 1.0 / a; break;
    }
    y[t] = r;
}

// ---------------------------------------------------------------------------
// Drop counting (post/DropCountSize, get_interface.f90:11-47, flood_fill.f90):
// cells with phi >= 0.5, 26-connected with periodic wrap, one drop per
// connected set.  Connected-component labelling by lock-free union-find
// (labels link a larger index to a smaller one with atomicMin, so every set
// ends labelled by its smallest linear index -- the cell the reference's
// raster scan meets first -- whatever the order of the atomics).
//
// The passes work on runs, not cells.  A bitmask holds one bit per cell, rows
// of W = ceil(n/64) words; a run is a maximal stretch of set bits of one word,
// and only its first cell's label is ever followed (the other cells of a run
// point at the first).  After the one pass over phi every pass reads n^3/8
// bytes of mask and the labels of the runs alone, one word per lane, and
// skips empty words.  At 256^3 with 64 drops the
// passes take 0.14 ms together, against 8.44 ms with one 64-bit atomic and one
// binary search per cell (6.92 ms) and 13 unions per cell (1.42 ms).
// ---------------------------------------------------------------------------
// phi >= 0.5 into the mask, one wavefront per CCL_WPW words, a lane per cell;
// labels of the set cells: the first cell of their run.  Bound by the read of phi
// (256^3 FP64: 34 us, 3.9 TB/s).
constexpr int CCL_WPW = 4;

template <typename T>
__global__ void __launch_bounds__(BLK) k_ccl_init(const T *__restrict__ phi, unsigned *__restrict__ lab,
                                                  unsigned long long *__restrict__ mask, int n, int W)
{
    const int lane = threadIdx.x & 63;
    const unsigned words = (unsigned)W * n * n;
    const unsigned w0 = (blockIdx.x * (BLK / 64) + (threadIdx.x >> 6)) * CCL_WPW;
    bool set[CCL_WPW];
    size_t cell[CCL_WPW];
#pragma unroll
    for (int q = 0; q < CCL_WPW; q++) {
        const unsigned wd = w0 + q, row = wd / (unsigned)W;
        const int x = (int)(wd - row * W) * 64 + lane;
        cell[q] = (size_t)row * n + x;
        set[q] = wd < words && x < n && (double)phi[cell[q]] >= 0.5;
    }
#pragma unroll
    for (int q = 0; q < CCL_WPW; q++) {
        const unsigned long long m = __ballot(set[q]);
        if (w0 + q >= words) break;
        if (lane == 0) mask[w0 + q] = m;
        if (set[q]) {
            const unsigned long long gaps = ~m & ((1ull << lane) - 1ull);       // clear bits below this one
            const int start = gaps ? 64 - __clzll((long long)gaps) : 0;
            lab[cell[q]] = (unsigned)(cell[q] - (size_t)(lane - start));
        }
    }
}

// Root of x as this thread's caches have it.
__device__ __forceinline__ unsigned ccl_find(const unsigned *lab, unsigned x)
{
    unsigned p = lab[x];
    while (p != x) {
        x = p;
        p = lab[x];
    }
    return x;
}

// Join the sets of a and b.  The finds may read labels that another XCD has
// changed since; only the atomic decides: a was a root if it still held its
// own index, and otherwise its true label, which is smaller, is joined with b
// in its place, so the loop ends.  Linking a root to a cell that is no root
// any more is as good, its chain goes on to the root.
__device__ __forceinline__ void ccl_union(unsigned *lab, unsigned a, unsigned b)
{
    a = ccl_find(lab, a);
    b = ccl_find(lab, b);
    while (a != b) {
        if (a < b) { unsigned t = a; a = b; b = t; }
        const unsigned old = atomicMin(&lab[a], b);     // link the larger to the smaller
        if (old == a) return;
        a = old;
    }
}

// Word w of row `r` with its cells' x-1 and x+1 neighbours (periodic) as masks.
struct CclRow {
    unsigned long long m, l, r;
};
__device__ __forceinline__ CclRow ccl_row(const unsigned long long *__restrict__ mask, unsigned r, int w, int n, int W)
{
    const unsigned long long *row = mask + (size_t)r * W;
    CclRow q;
    q.m = row[w];
    const int last = w + 1 == W ? (n - 1) & 63 : 63;                            // last cell's bit in this word
    const unsigned long long before = w == 0 ? row[W - 1] >> ((n - 1) & 63) : row[w - 1] >> 63;
    const unsigned long long after = row[w + 1 == W ? 0 : w + 1];
    q.l = (q.m << 1) | (before & 1ull);
    q.r = (q.m >> 1) | ((after & 1ull) << last);
    return q;
}

// Union of each run with the runs it touches in the 4 forward rows (y+1, and
// y-1, y, y+1 of plane z+1; the 13 forward offsets of the 26-neighbourhood
// with the own row's).  Where two runs lie side by side, the first pair of
// cells joins them: a cell x with row[x] set leaves it to cell x-1 if that and
// row[x-1] are set (but at x = 0, so that two full rows join somewhere); a
// diagonal pair is joined only where no straight pair beside it is.  Bound by
// the chain of dependent label loads and atomics of one lane, so the four rows
// of a word go to four lanes (107 against 116 us
// at 256^3 with 64 drops; 74 us with finds through the caches, ccl_find).
__global__ void __launch_bounds__(BLK) k_ccl_merge(unsigned *__restrict__ lab,
                                                   const unsigned long long *__restrict__ mask, int n, int W)
{
    const unsigned wd = blockIdx.x * (BLK / 4) + threadIdx.x / 4;
    const int q = threadIdx.x & 3;
    if (wd >= (unsigned)W * n * n || mask[wd] == 0) return;
    const unsigned row = wd / (unsigned)W;
    const int w = (int)(wd - row * W), k = (int)(row / (unsigned)n), j = (int)row - k * n;
    const CclRow o = ccl_row(mask, row, w, n, W);
    const unsigned base = row * (unsigned)n, x0 = (unsigned)w * 64;
    if (q == 0 && (o.m & o.l & 1ull)) ccl_union(lab, base + x0, base + (w == 0 ? (unsigned)n : x0) - 1);
    const int jp = j + 1 == n ? 0 : j + 1, jm = j == 0 ? n - 1 : j - 1, kp = k + 1 == n ? 0 : k + 1;
    const unsigned nrow = (unsigned)((q == 0 ? k : kp) * n + (q == 1 ? jm : q == 2 ? j : jp));
    const CclRow t = ccl_row(mask, nrow, w, n, W);
    const unsigned nbase = nrow * (unsigned)n;
    unsigned long long mid = o.m & t.m & ~(o.l & t.l);
    if (w == 0) mid |= o.m & t.m & 1ull;
    unsigned long long right = o.m & ~t.m & t.r & ~o.r, left = o.m & ~t.m & t.l & ~o.l;
    for (; mid; mid &= mid - 1) {
        const unsigned x = x0 + (unsigned)__builtin_ctzll(mid);
        ccl_union(lab, base + x, nbase + x);
    }
    for (; right; right &= right - 1) {
        const unsigned x = x0 + (unsigned)__builtin_ctzll(right);
        ccl_union(lab, base + x, nbase + (x + 1 == (unsigned)n ? 0 : x + 1));
    }
    for (; left; left &= left - 1) {
        const unsigned x = x0 + (unsigned)__builtin_ctzll(left);
        ccl_union(lab, base + x, nbase + (x == 0 ? (unsigned)n : x) - 1);
    }
}

// fn(first cell, length) for every run of a mask word whose bit 0 is `cell0`.
template <typename Fn>
__device__ __forceinline__ void ccl_runs(unsigned long long m, unsigned cell0, Fn &&fn)
{
    while (m) {
        const int s = __builtin_ctzll(m);
        const unsigned long long rest = ~(m >> s);                              // the run ends at its lowest set bit
        const int len = rest ? __builtin_ctzll(rest) : 64;
        fn(cell0 + (unsigned)s, len);
        m = s + len < 64 ? m & (~0ull << (s + len)) : 0ull;
    }
}

// Roots in raster order, without a sort: the words are cut into `chunks`
// contiguous chunks (at most CCL_CHUNKS); pass 1 points every run at its root
// and counts the roots (runs labelled by their own first cell) of each chunk;
// pass 2 adds up the counts before its chunk and writes the chunk's roots from
// there in cell order, clearing their volumes.
__device__ __forceinline__ unsigned ccl_chunk_begin(unsigned words, unsigned b, unsigned chunks)
{
    return (unsigned)((unsigned long long)words * b / chunks);
}
__device__ __forceinline__ unsigned ccl_cell0(unsigned wd, int n, int W)
{
    const unsigned row = wd / (unsigned)W;
    return row * (unsigned)n + (wd - row * W) * 64u;
}

// Sum over the block's BLK threads (every thread gets it); `part` is BLK/64 values of LDS.
__device__ __forceinline__ unsigned block_sum(unsigned c, unsigned *part)
{
    for (int off = 32; off >= 1; off >>= 1) c += __shfl_xor(c, off, 64);
    __syncthreads();
    if ((threadIdx.x & 63) == 0) part[threadIdx.x >> 6] = c;
    __syncthreads();
    unsigned t = 0;
    for (int q = 0; q < BLK / 64; q++) t += part[q];
    return t;
}

__global__ void __launch_bounds__(BLK) k_ccl_roots(unsigned *__restrict__ lab,
                                                   const unsigned long long *__restrict__ mask, int n, int W,
                                                   unsigned *__restrict__ counts)
{
    __shared__ unsigned part[BLK / 64];
    const unsigned words = (unsigned)W * n * n;
    const unsigned lo = ccl_chunk_begin(words, blockIdx.x, gridDim.x), hi = ccl_chunk_begin(words, blockIdx.x + 1, gridDim.x);
    unsigned c = 0;
    for (unsigned wd = lo + threadIdx.x; wd < hi; wd += BLK)
        ccl_runs(mask[wd], ccl_cell0(wd, n, W), [&](unsigned x, int) {
            const unsigned r = ccl_find(lab, x);
            if (r == x) c++;
            else lab[x] = r;
        });
    c = block_sum(c, part);
    if (threadIdx.x == 0) counts[blockIdx.x] = c;
}

__global__ void __launch_bounds__(BLK) k_ccl_place(const unsigned *__restrict__ lab,
                                                   const unsigned long long *__restrict__ mask, int n, int W,
                                                   const unsigned *__restrict__ counts, unsigned *__restrict__ nroots,
                                                   unsigned *__restrict__ roots, unsigned long long *__restrict__ vol,
                                                   unsigned cap)
{
    __shared__ unsigned part[BLK / 64];
    const int b = blockIdx.x, chunks = gridDim.x;
    if (b == 0) {
        unsigned t = 0;
        for (int q = threadIdx.x; q < chunks; q += BLK) t += counts[q];
        t = block_sum(t, part);
        if (threadIdx.x == 0) *nroots = t;
    }
    if (counts[b] == 0) return;
    unsigned pos = 0;
    for (int q = threadIdx.x; q < b; q += BLK) pos += counts[q];
    pos = block_sum(pos, part);
    const unsigned words = (unsigned)W * n * n;
    const unsigned lo = ccl_chunk_begin(words, b, chunks), hi = ccl_chunk_begin(words, b + 1, chunks);
    const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
    for (unsigned t0 = lo; t0 < hi; t0 += BLK) {
        const unsigned wd = t0 + threadIdx.x;
        const unsigned long long m = wd < hi ? mask[wd] : 0ull;
        const unsigned cell0 = ccl_cell0(wd, n, W);
        unsigned c = 0;
        ccl_runs(m, cell0, [&](unsigned x, int) { c += lab[x] == x; });
        unsigned incl = c;                                                      // roots up to this lane
        for (int off = 1; off < 64; off <<= 1) {
            const unsigned o = __shfl_up(incl, off, 64);
            if (lane >= off) incl += o;
        }
        __syncthreads();
        if (lane == 63) part[wv] = incl;
        __syncthreads();
        unsigned before = 0, total = 0;
        for (int q = 0; q < BLK / 64; q++) {
            before += q < wv ? part[q] : 0u;
            total += part[q];
        }
        unsigned at = pos + before + incl - c;
        if (c)
            ccl_runs(m, cell0, [&](unsigned x, int) {
                if (lab[x] != x) return;
                if (at < cap) {
                    roots[at] = x;
                    vol[at] = 0;
                }
                at++;
            });
        pos += total;
    }
}

// Cells per drop.  A lane adds up the runs of one root until another root
// comes, a wavefront adds up its lanes of one root, and only then the root's
// place in the list is looked up and its volume added to: one atomic and one
// search per root and wavefront of contiguous rows.  Runs only when every root
// fit the list (*nroots <= cap).
__global__ void __launch_bounds__(BLK) k_ccl_volume(const unsigned *__restrict__ lab,
                                                    const unsigned long long *__restrict__ mask, int n, int W,
                                                    const unsigned *__restrict__ roots,
                                                    const unsigned *__restrict__ nroots, unsigned cap,
                                                    unsigned long long *__restrict__ vol)
{
    const unsigned nr = *nroots;
    if (nr == 0 || nr > cap) return;
    auto add = [&](unsigned root, unsigned cells) {
        unsigned lo = 0, hi = nr - 1;
        while (lo < hi) {
            const unsigned mid = (lo + hi) >> 1;
            if (roots[mid] < root) lo = mid + 1;
            else hi = mid;
        }
        atomicAdd(&vol[lo], (unsigned long long)cells);
    };
    const unsigned words = (unsigned)W * n * n;
    const unsigned lo = ccl_chunk_begin(words, blockIdx.x, gridDim.x), hi = ccl_chunk_begin(words, blockIdx.x + 1, gridDim.x);
    unsigned root = 0, cells = 0;                                               // this lane's pending root
    for (unsigned wd = lo + threadIdx.x; wd < hi; wd += BLK)
        ccl_runs(mask[wd], ccl_cell0(wd, n, W), [&](unsigned x, int len) {
            const unsigned r = lab[x];
            if (cells && r != root) {
                add(root, cells);
                cells = 0;
            }
            root = r;
            cells += (unsigned)len;
        });
    const int lane = threadIdx.x & 63;
    unsigned long long todo = __ballot(cells != 0);
    while (todo) {
        const int lead = __builtin_ctzll(todo);
        const unsigned r = __shfl(root, lead, 64);
        const bool mine = cells != 0 && root == r;
        todo &= ~__ballot(mine);
        unsigned sum = mine ? cells : 0;
        for (int off = 32; off >= 1; off >>= 1) sum += __shfl_xor(sum, off, 64);
        if (lane == lead) add(r, sum);
    }
}

// ---------------------------------------------------------------------------
// Random-phase initial velocity (the turbulent start the reference reads from
// input/{u,v,w}.dat, main.f90:234-239): a random vector potential A drawn on
// the half spectrum, brought to the grid by the inverse passes of the Poisson
// solver, and u = curl A with the staggered grid's forward differences, so
// the discrete divergence of main.f90:723-725 vanishes up to rounding.
// ---------------------------------------------------------------------------
__device__ __forceinline__ unsigned long long splitmix64(unsigned long long x)
{
    // SplitMix64 (Steele, Lea and Flood, OOPSLA 2014): a counter-based hash, so
    // each spectral coefficient depends only on (seed, component, position).
    unsigned long long z = x + 0x9E3779B97F4A7C15ull;
    z = (z ^ (z >> 30)) * 0xBF58476D1CE4E5B9ull;
    z = (z ^ (z >> 27)) * 0x94D049BB133111EBull;
    return z ^ (z >> 31);
}

__device__ __forceinline__ double unit53(unsigned long long h) { return (double)(h >> 11) * (1.0 / 9007199254740992.0); }

// A_comp(q, ky, kz) = amp(k) g e^{i theta}: amp = sqrt(exp(-2 (k/kp)^2) / (4 pi))
// for 0 < k <= kmax, g standard normal (Box-Muller), theta uniform.
__global__ void __launch_bounds__(BLK) k_ic_spectrum(double2 *__restrict__ spec, int n, int ld, int comp,
                                                     unsigned long long seedmix, double kp, double kmax)
{
    const int nh = n / 2 + 1;
    const size_t total = (size_t)nh * n * n;
    const double twopi = 6.283185307179586;
    for (size_t e = (size_t)blockIdx.x * BLK + threadIdx.x; e < total; e += (size_t)gridDim.x * BLK) {
        const int q = (int)(e % nh);
        const int j = (int)((e / nh) % n);
        const int k = (int)(e / ((size_t)nh * n));
        const double kq = q, ky = j < n / 2 ? j : j - n, kz = k < n / 2 ? k : k - n;
        const double kk = __builtin_sqrt((kq * kq + ky * ky) + kz * kz);
        const unsigned long long idx = (((unsigned long long)comp * n + k) * n + j) * nh + q;
        const unsigned long long key = seedmix ^ (idx * 4ull);
        const double u1 = unit53(splitmix64(key)), u2 = unit53(splitmix64(key + 1ull)),
                     u3 = unit53(splitmix64(key + 2ull));
        const double g = sqrt(-2.0 * log(1.0 - u1)) * cos(twopi * u2);
        const double th = twopi * u3;
        const double amp = (kk > 0.0 && kk <= kmax) ? sqrt(exp(-2.0 * ((kk / kp) * (kk / kp))) / (4.0 * 3.141592653589793)) : 0.0;
        const double a = amp * g;
        spec[spec_row(k, j, n, ld) + q] = make_double2(a * cos(th), a * sin(th));
    }
}

// u = d_y A_z - d_z A_y, v = d_z A_x - d_x A_z, w = d_x A_y - d_y A_x (forward
// differences / dx).  SUM: per-x-line sums of u^2 + v^2 + w^2 into lsum;
// otherwise write s*u, s*v, s*w.
template <typename T, bool SUM>
__global__ void __launch_bounds__(BLK) k_ic_curl(const double *__restrict__ ax, const double *__restrict__ ay,
                                                 const double *__restrict__ az, T *__restrict__ u, T *__restrict__ v,
                                                 T *__restrict__ w, double *__restrict__ lsum, int n, double dx,
                                                 double s)
{
    const int lane = threadIdx.x & 63;
    const size_t line = ((size_t)blockIdx.x * BLK + threadIdx.x) >> 6;
    if (line >= (size_t)n * n) return;
    const int j = (int)(line % n), k = (int)(line / n);
    const int jp = j + 1 == n ? 0 : j + 1, kp = k + 1 == n ? 0 : k + 1;
    double acc = 0.0;
    for (int i = lane; i < n; i += 64) {
        const int ip = i + 1 == n ? 0 : i + 1;
        const size_t id = IDX(i, j, k);
        const double a0x = ax[id], a0y = ay[id], a0z = az[id];
        const double uu = (az[IDX(i, jp, k)] - a0z) / dx - (ay[IDX(i, j, kp)] - a0y) / dx;
        const double vv = (ax[IDX(i, j, kp)] - a0x) / dx - (az[IDX(ip, j, k)] - a0z) / dx;
        const double ww = (ay[IDX(ip, j, k)] - a0y) / dx - (ax[IDX(i, jp, k)] - a0x) / dx;
        if constexpr (SUM) {
            acc = acc + ((uu * uu + vv * vv) + ww * ww);
        } else {
            u[id] = (T)(uu * s);
            v[id] = (T)(vv * s);
            w[id] = (T)(ww * s);
        }
    }
    if constexpr (SUM) {
        acc = wave_sum(acc);
        if (lane == 0) lsum[line] = acc;
    }
}

// ---------------------------------------------------------------------------
// Launch helpers
// ---------------------------------------------------------------------------
void launch_diagnostics(const Fields &f, const Consts &c, double dxi, double *out, hipStream_t s)
{
    const size_t threads = (size_t)c.n * c.n * 64;
    if (c.mixed)
        hipLaunchKernelGGL(k_diag_lines<float>, dim3(nblocks(threads, BLK)), dim3(BLK), 0, s, (const float *)f.u,
                           (const float *)f.v, (const float *)f.w, (const float *)f.phi, f.lsum, f.sc, c, dxi);
    else
        hipLaunchKernelGGL(k_diag_lines<double>, dim3(nblocks(threads, BLK)), dim3(BLK), 0, s, f.u, f.v, f.w, f.phi,
                           f.lsum, f.sc, c, dxi);
    hipLaunchKernelGGL(k_diag_planes, dim3(c.n, 3), dim3(64), 0, s, f.lsum, f.psum, c.n);
    hipLaunchKernelGGL(k_diag_total, dim3(1), dim3(64), 0, s, f.psum, out, c.n);
}

// Scratch of the allocation-free drop count: a file-scope device array, one
// copy per GPU, held until the process ends.  Host code never passes the
// array's name to a kernel or copy (on the host it is a stand-in, not a device
// address); it uses the address hipGetSymbolAddress gives for each device.
static __device__ __align__(256) unsigned char scratch[NOALLOC_SCRATCH_BYTES];

void *noalloc_scratch(int device)
{
    static std::mutex mu;
    static void *addr[NOALLOC_MAX_DEVICES] = {};
    if (device < 0 || device >= NOALLOC_MAX_DEVICES) return nullptr;
    std::lock_guard<std::mutex> lock(mu);
    if (!addr[device]) {
        int cur = 0;
        if (hipGetDevice(&cur) != hipSuccess) return nullptr;
        if (cur != device && hipSetDevice(device) != hipSuccess) return nullptr;
        void *ptr = nullptr;
        const hipError_t e = hipGetSymbolAddress(&ptr, HIP_SYMBOL(scratch));
        if (cur != device) (void)hipSetDevice(cur);
        if (e != hipSuccess || !ptr) {
            (void)hipGetLastError();
            return nullptr;
        }
        addr[device] = ptr;
    }
    return addr[device];
}

CclWork ccl_carve(void *base, int n)
{
    const size_t n3 = (size_t)n * n * n;
    const size_t cap = ccl_cap(n3);
    auto up = ccl_up;
    char *p = (char *)base;
    CclWork w;
    w.lab = (unsigned *)p;                   p += up(n3 * 4);
    w.roots = (unsigned *)p;                 p += up(cap * 4);
    w.vol = (unsigned long long *)p;         p += up(cap * 8);
    w.mask = (unsigned long long *)p;        p += up(ccl_words(n) * 8);
    w.counts = (unsigned *)p;                p += up(CCL_CHUNKS * 4);
    w.nroots = (unsigned *)p;
    w.cap = (unsigned)cap;
    return w;
}

void launch_ccl_count(const Fields &f, const Consts &c, const CclWork &w, hipStream_t s)
{
    const int n = c.n, W = (n + 63) / 64;
    const size_t words = ccl_words(n);
    const dim3 gi(nblocks(words, BLK / 64 * CCL_WPW)), gw(nblocks(words, BLK));
    if (c.mixed)
        hipLaunchKernelGGL(k_ccl_init<float>, gi, dim3(BLK), 0, s, (const float *)f.phi, w.lab, w.mask, n, W);
    else
        hipLaunchKernelGGL(k_ccl_init<double>, gi, dim3(BLK), 0, s, f.phi, w.lab, w.mask, n, W);
    hipLaunchKernelGGL(k_ccl_merge, dim3(nblocks(words, BLK / 4)), dim3(BLK), 0, s, w.lab, w.mask, n, W);
    // a chunk per block's worth of words, up to CCL_CHUNKS
    const dim3 gc(gw.x < (unsigned)CCL_CHUNKS ? gw.x : (unsigned)CCL_CHUNKS);
    hipLaunchKernelGGL(k_ccl_roots, gc, dim3(BLK), 0, s, w.lab, w.mask, n, W, w.counts);
    hipLaunchKernelGGL(k_ccl_place, gc, dim3(BLK), 0, s, w.lab, w.mask, n, W, w.counts, w.nroots, w.roots, w.vol,
                       w.cap);
    hipLaunchKernelGGL(k_ccl_volume, gc, dim3(BLK), 0, s, w.lab, w.mask, n, W, w.roots, w.nroots, w.cap, w.vol);
}

void launch_debug_math(int op, size_t count, const double *x, double *y, const double *mtab, hipStream_t s)
{
    if (count == 0) return;
    hipLaunchKernelGGL(k_debug_math, dim3(nblocks(count, BLK)), dim3(BLK), 0, s, op, count, x, y, mtab);
}

static inline double F(const Consts &c) { return 8.0 * (double)c.n * c.n * c.n; }

// Planes per block for the z-marching kernels: of the powers of two dividing n,
// the one of least cost rounds (kz + extra), the rounds of resident blocks
// times the planes each works through; up to two rounds count whole, beyond
// that blocks end at different times and the rounds blur.  A thicker slab has
// to gain 2%.  `boxes` boxes launched together count as so many times the blocks.
static int march_kz(int n, int tiles, int slots, int extra, int most, int boxes = 1)
{
    int best = 1;
    double least = 0.0;
    for (int kz = 2; kz <= most && n % kz == 0; kz *= 2) {
        const double r = (double)boxes * tiles * (n / kz) / slots;
        const double cost = (r <= 1.0 ? 1.0 : r <= 2.0 ? 2.0 : r) * (kz + extra);
        if (best == 1 || cost < 0.98 * least) {
            best = kz;
            least = cost;
        }
    }
    return best;
}
// The constants are fitted to sweeps of kz at 16^3 to 512^3 (16, 32, 48, 64,
// 96, 108, 128, 192, 256, 384, 512).  This rule / the best power of two, us, with
// the phase field and the momentum march of one barrier a plane (16 rows FP64):
//   phase field FP64   96^3 22.5 / 22.4   128^3 33.0 / 33.0   192^3 95.2 / 94.9   256^3 182 / 182
//   phase field FP32   96^3 12.7 / 12.7   128^3 17.7 / 17.7   192^3 42.6 / 42.6   256^3 85.7 / 85.7
//   momentum FP64      72^3 24.3 / 22.0   128^3 46.2 / 46.1   192^3 152 / 152     256^3 340 / 340
//   momentum FP32     108^3 26.0 / 22.7   128^3 29.0 / 29.0   192^3 82.9 / 82.8   256^3 175 / 175
// (with a target of 2048 blocks instead: phase field FP64 128^3 54.9, 256^3 195).
// Only powers of two that divide n are tried: 54, 162 and 486 get two planes.
// A phase-field block recomputes 4 planes of psi in its prologue; two FP64
// blocks are resident per CU (as of the momentum pass), of FP32's four the last adds little.  A momentum
// block's prologue reads planes that its neighbour has just read.
static int kz_acdi(int n, int mixed, int boxes = 1)
{
    return march_kz(n, ((n + ATX - 1) / ATX) * ((n + ATY - 1) / ATY), mixed ? 768 : 512, 4, 64, boxes);
}
static int kz_momentum(int n, int mixed, int boxes = 1)
{
    const int tx = mixed ? 2 * PTX : MTX, ty = mixed ? PTY : MTY;
    return march_kz(n, ((n + tx - 1) / tx) * ((n + ty - 1) / ty), mixed ? 768 : 512, mixed ? 3 : 1, 32, boxes);
}

// The forms of small boxes take no slab height: they run unless one was set by hand.
static bool acdi_in_boxes(const Consts &c, const Tuning &tu) { return c.n <= 72 && tu.v[KNOB_KZ_ACDI] == 0; }
static bool momentum_by_point(const Consts &c, const Tuning &tu)
{
    return c.n <= (c.mixed ? 96 : 64) && tu.v[KNOB_KZ_MOM] == 0;
}

template <typename T>
static void launch_acdi_t(const Fields &f, const Consts &c, int kz, bool boxes, hipStream_t s)
{
    const int n = c.n;
    const T *u = (const T *)f.u, *v = (const T *)f.v, *w = (const T *)f.w, *phi = (const T *)f.phi;
    if (boxes)
        hipLaunchKernelGGL(k_acdi_box<T>, dim3((n + BTX - 1) / BTX, (n + BTY - 1) / BTY, (n + BTZ - 1) / BTZ),
                           dim3(BTHREADS), 0, s, u, v, w, phi, (T *)f.phin, f.sc, f.mtab, c);
    else
        hipLaunchKernelGGL(k_acdi<T>, dim3((n + ATX - 1) / ATX, (n + ATY - 1) / ATY, n / kz), dim3(ATHREADS), 0, s, u, v, w,
                           phi, (T *)f.phin, f.sc, f.mtab, c, kz);
}

void launch_acdi(const Fields &f, const Consts &c, const Tuning &tu, hipStream_t s, LaunchInfo *li)
{
    const int kz = tu.v[KNOB_KZ_ACDI] ? tu.v[KNOB_KZ_ACDI] : kz_acdi(c.n, c.mixed);
    const bool boxes = acdi_in_boxes(c, tu);
    if (c.mixed) launch_acdi_t<float>(f, c, kz, boxes, s);
    else launch_acdi_t<double>(f, c, kz, boxes, s);
    li->name = "acdi"; li->bytes = (c.mixed ? 2.5 : 5.0) * F(c);
}

template <int PHI, typename T>
static void launch_momentum_t(const Fields &f, const Consts &c, int kz, bool point, double alpha, double beta,
                              hipStream_t s)
{
    const int n = c.n;
    const T *u = (const T *)f.u, *v = (const T *)f.v, *w = (const T *)f.w, *ph = (const T *)f.phi;
    T *us = (T *)f.us, *vs = (T *)f.vs, *ws = (T *)f.ws, *ru = (T *)f.ruo, *rv = (T *)f.rvo, *rw = (T *)f.rwo;
    if (point)
        hipLaunchKernelGGL((k_momentum_point<PHI, T>), dim3((n + DTX - 1) / DTX, (n + DTY - 1) / DTY, n), dim3(DTX * DTY),
                           0, s, u, v, w, ph, us, vs, ws, ru, rv, rw, f.sinf, f.cosf, f.sc, c, alpha, beta);
    else if constexpr (sizeof(T) == 4)
        hipLaunchKernelGGL((k_momentum_x2<PHI, T>), dim3((n + 2 * PTX - 1) / (2 * PTX), (n + PTY - 1) / PTY, n / kz),
                           dim3(PTHREADS), 0, s, u, v, w, ph, us, vs, ws, ru, rv, rw, f.sinf, f.cosf, f.sc, c, alpha, beta,
                           kz);
    else
        hipLaunchKernelGGL((k_momentum<PHI, T>), dim3((n + MTX - 1) / MTX, (n + MTY - 1) / MTY, n / kz), dim3(MTHREADS), 0,
                           s, u, v, w, ph, us, vs, ws, ru, rv, rw, f.sinf, f.cosf, f.sc, c, alpha, beta, kz);
}

void launch_momentum(const Fields &f, const Consts &c, const Tuning &tu, double alpha, double beta, hipStream_t s,
                     LaunchInfo *li)
{
    const int kz = tu.v[KNOB_KZ_MOM] ? tu.v[KNOB_KZ_MOM] : kz_momentum(c.n, c.mixed);
    const bool point = momentum_by_point(c, tu);
    auto launch = c.mixed ? (c.phiflag ? launch_momentum_t<1, float> : launch_momentum_t<0, float>)
                          : (c.phiflag ? launch_momentum_t<1, double> : launch_momentum_t<0, double>);
    launch(f, c, kz, point, alpha, beta, s);
    li->name = "momentum"; li->bytes = (c.mixed ? (c.phiflag ? 6.5 : 6.0) : (c.phiflag ? 13.0 : 12.0)) * F(c);
}

static int plan_rmin(const FftPlan &pl)
{
    int rmin = 8;
    for (int s = 0; s < pl.nst; s++) rmin = pl.R[s] < rmin ? pl.R[s] : rmin;
    return rmin;
}

// Lines per block for the x passes: a power of two p <= 8 with one butterfly
// per thread (p*n/Rmin <= 1024 threads), LDS within LDS_CAP, dividing n*n/2.
static int pairs_per_block(const FftPlan &pl)
{
    const int rmin = plan_rmin(pl);
    int p = 8;
    while (p > 1 && p * (pl.n / rmin) > FFT_MAX_THREADS) p >>= 1;
    while (p > 1 && (size_t)p * (pl.n + 1) * sizeof(double2) > LDS_CAP) p >>= 1;
    const int pairs = pl.n * pl.n / 2;
    while (p > 1 && pairs % p != 0) p >>= 1;
    return p;
}

// kx columns per block for the y/z passes.
static int col_tile(const FftPlan &pl)
{
    const int rmin = plan_rmin(pl);
    int t = 8;
    while (t > 1 && t * (pl.n / rmin) > FFT_MAX_THREADS) t >>= 1;
    while (t > 1 && (size_t)t * pl.n * sizeof(double2) > LDS_CAP) t >>= 1;
    return t;
}

// The lengths the register kernels are compiled for, with the stage plan as
// constants: the column passes for their default tile (rtile_n) alone, the x
// passes for any number of line pairs per block.  FFT_SIZES_GANG: also in gang
// launches (boxes of up to 128^3).  The turbulent start's z pass is compiled for none.
#define FFT_SIZES_PLANE(X) X(32) X(36) X(48) X(54) X(64)
#define FFT_SIZES_GANG(X) FFT_SIZES_PLANE(X) X(72) X(96) X(108) X(128)
#define FFT_SIZES(X) FFT_SIZES_GANG(X) X(144) X(162) X(192) X(216) X(256) X(288) X(324) X(384) X(432) X(486) X(512) X(1024)

static bool compiled_n(int n, FftUse use)
{
    if (use == FFT_START) return false;
#define FFT_CASE(N) case N:
    switch (n) {
    FFT_SIZES_GANG(FFT_CASE)
        return true;
    default: break;
    }
    if (use == FFT_GANG) return false;
    switch (n) {
    FFT_SIZES(FFT_CASE)
        return true;
    default: return false;
    }
#undef FFT_CASE
}
// Calls fn(std::integral_constant<int, N>) for a compiled n, or with 0 for any other.
template <bool GANG, typename Fn>
static void with_n(int n, Fn &&fn)
{
#define FFT_CASE(N) case N: fn(std::integral_constant<int, N>()); return;
    if constexpr (GANG) {
        switch (n) {
        FFT_SIZES_GANG(FFT_CASE)
        default: break;
        }
    } else {
        switch (n) {
        FFT_SIZES(FFT_CASE)
        default: break;
        }
    }
#undef FFT_CASE
    fn(std::integral_constant<int, 0>());
}

template <typename Fn>
static void with_plane_n(int n, Fn &&fn)
{
#define FFT_CASE(N) case N: static_assert(N <= PLANE_MAX, "a plane fits one block"); fn(std::integral_constant<int, N>()); return;
    switch (n) {
    FFT_SIZES_PLANE(FFT_CASE)
    default: return;
    }
#undef FFT_CASE
}

// A power of two the runtime-plan register kernels take (radices 8/4/2, one
// thread per 8 elements).
static bool pow2_regs(const FftPlan &pl) { return pl.n >= 16 && is_pow2(pl.n); }

static int fft_threads(const FftPlan &pl, int nlines)
{
    int t = nlines * (pl.n / plan_rmin(pl));
    t = ((t + 63) / 64) * 64;
    return t < 64 ? 64 : t;
}

// How an x pass and a column pass are launched for a shape set by hand (0: the
// default): the register kernels where n is compiled (a column pass also needs
// its default tile) or a power of two, else the LDS-staged kernels.  A shape is
// chosen for the one-box passes, and another use of it may run the other form:
// the default column tile of the register kernels (8 at 432 and 486) gives the
// LDS-staged ones up to 1984 threads, so they take their own where it does not fit.
struct FftPass {
    int lines, threads;                  // pairs or columns, and threads, of a block
    size_t lds;
    bool regs;
    int n;                               // the length it is compiled for, or 0 (in with_n's list or not)
};
static FftPass x_pass(const FftPlan &pl, int set, FftUse use)
{
    FftPass q;
    q.regs = compiled_n(pl.n, use) || pow2_regs(pl);
    q.lines = set ? set : q.regs ? rpairs_n(pl.n) : pairs_per_block(pl);
    q.threads = q.regs ? q.lines * line_threads(pl.n) : fft_threads(pl, q.lines);
    q.lds = sizeof(double2) * (size_t)q.lines * (q.regs ? rline_stride(pl.n) : pl.n + 1);
    q.n = pl.n;
    return q;
}
static FftPass col_pass(const FftPlan &pl, int set, FftUse use)
{
    const bool compiled = compiled_n(pl.n, use), pow2 = pow2_regs(pl);
    FftPass q;
    q.lines = set ? set : compiled || pow2 ? rtile_n(pl.n) : col_tile(pl);
    q.regs = pow2 || (compiled && q.lines == rtile_n(pl.n));
    if (!q.regs && fft_threads(pl, q.lines) > FFT_MAX_THREADS) q.lines = col_tile(pl);
    q.threads = q.regs ? q.lines * line_threads(pl.n) : fft_threads(pl, q.lines);
    q.lds = sizeof(double2) * (size_t)q.lines * pl.n;
    q.n = q.lines == rtile_n(pl.n) ? pl.n : 0;
    return q;
}
static int default_pairs(const FftPlan &pl) { return x_pass(pl, 0, FFT_BOX).lines; }
static int default_tile(const FftPlan &pl) { return col_pass(pl, 0, FFT_BOX).lines; }

// Whether a box's x and y passes run plane by plane in one block: a small
// compiled length with no x or y shape set by hand (one asks for the separate
// passes).
// One box: n blocks leave most CUs idle, and the forward passes, whose threads
// load eleven values per point pair, gain only at 32^3 and in FP32 up to 48^3
// (forward pair / in one, us: 32^3 11.1 / 9.2, 48^3 FP32 9.7 / 8.7, FP64 9.7 /
// 14.9, 64^3 FP32 10.6 / 12.0, FP64 12.3 / 16.1); the inverse passes gain at every
// size (64^3 10.0 / 8.1).  36^3 and 54^3, by the time of the step with either:
// FP64 level or separate faster, FP32 within 6% either way.  A gang fills the CUs: 8 boxes of 64^3 20.4 / 15.6 and
// 18.1 / 10.1.
bool plane_fwd_alone(const Consts &c) { return c.n <= 32 || (c.mixed && c.n <= 48); }
bool plane_passes(const Consts &c, const Tuning &tu)
{
    return c.n <= PLANE_MAX && compiled_n(c.n, FFT_GANG) && tu.v[KNOB_XPAIRS] == 0 && tu.v[KNOB_XIPAIRS] == 0 &&
           tu.v[KNOB_YTILE] == 0;
}

// Tunable launch shapes.  Every candidate satisfies what the kernels assume:
// z planes per block divide n; blocks have at most FFT_MAX_THREADS threads and
// LDS_MAX bytes of LDS; pairs per block divide the n^2/2 line pairs.
int knob_default(int knob, const Consts &c, const FftPlan &pl)
{
    switch (knob) {
    case KNOB_KZ_ACDI: return kz_acdi(c.n, c.mixed);
    case KNOB_KZ_MOM: return kz_momentum(c.n, c.mixed);
    case KNOB_XPAIRS:
    case KNOB_XIPAIRS: return default_pairs(pl);
    default: return default_tile(pl);
    }
}

bool knob_unused(int knob, const Consts &c)
{
    switch (knob) {
    case KNOB_KZ_ACDI: return acdi_in_boxes(c, Tuning());
    case KNOB_KZ_MOM: return momentum_by_point(c, Tuning());
    case KNOB_ZTILE: return false;
    default: return plane_passes(c, Tuning());
    }
}

int knob_candidates(int knob, const Consts &c, const FftPlan &pl, int *out, int cap)
{
    const int n = c.n;
    const bool regs = pow2_regs(pl);
    const int per_line = regs ? n / 8 : n / plan_rmin(pl);   // most threads per line (the LDS-staged form's)
    int k = 0;
    for (int v = 1; v <= 1024 && k < cap; v *= 2) {
        bool ok;
        if (knob == KNOB_KZ_ACDI || knob == KNOB_KZ_MOM) {
            ok = v >= 2 && v <= n && n % v == 0;
        } else if (knob == KNOB_XPAIRS || knob == KNOB_XIPAIRS) {
            const size_t lds = sizeof(double2) * (size_t)v * (regs ? rline_stride(n) : n + 1);
            ok = v <= 16 && v * per_line <= FFT_MAX_THREADS && lds <= LDS_MAX && (n * n / 2) % v == 0;
        } else {
            const size_t lds = sizeof(double2) * (size_t)v * n;
            ok = v <= 16 && v * per_line <= FFT_MAX_THREADS && lds <= LDS_MAX && v <= n / 2 + 1;
        }
        if (ok || v == knob_default(knob, c, pl)) out[k++] = v;
    }
    return k;
}

LaunchShape launch_shape(int knob, FftUse use, const Consts &c, const FftPlan &pl, const Tuning &tu)
{
    if (knob == KNOB_KZ_ACDI) {
        const int kz = tu.v[knob] ? tu.v[knob] : kz_acdi(c.n, c.mixed);
        if (use == FFT_BOX && acdi_in_boxes(c, tu)) return {FORM_SMALL, 0, BTHREADS, 0};
        return {FORM_MARCH, kz, ATHREADS, 0};
    }
    if (knob == KNOB_KZ_MOM) {
        const int kz = tu.v[knob] ? tu.v[knob] : kz_momentum(c.n, c.mixed);
        if (use == FFT_BOX && momentum_by_point(c, tu)) return {FORM_SMALL, 0, DTX * DTY, 0};
        return {FORM_MARCH, kz, c.mixed ? PTHREADS : MTHREADS, 0};
    }
    const bool planes = use != FFT_START && knob != KNOB_ZTILE && plane_passes(c, tu);
    if (planes && (use == FFT_GANG || knob == KNOB_XIPAIRS || plane_fwd_alone(c)))
        return {FORM_SMALL, 0, plane_threads(c.n), plane_lds(c.n)};
    const bool x = knob == KNOB_XPAIRS || knob == KNOB_XIPAIRS;
    // the turbulent start's y and x passes are the one-box ones
    const FftPass q = x ? x_pass(pl, tu.v[knob], use == FFT_START ? FFT_BOX : use)
                        : col_pass(pl, tu.v[knob], use == FFT_START && knob == KNOB_YTILE ? FFT_BOX : use);
    return {q.regs ? FORM_REGS : FORM_LDS, q.lines, q.threads, q.lds};
}

void launch_xfwd(const Fields &f, const Consts &c, const FftPlan &pl, const Tuning &tu, hipStream_t s,
                 LaunchInfo *li)
{
    const FftPass q = x_pass(pl, tu.v[KNOB_XPAIRS], FFT_BOX);
    const int ppb = q.lines, pairs = c.n * c.n / 2;
    const dim3 grid(pairs / ppb), blk(q.threads);
    const float *us = (const float *)f.us, *vs = (const float *)f.vs, *ws = (const float *)f.ws;
    if (q.regs) {
        with_n<false>(q.n, [&](auto NC) {
            constexpr int N = decltype(NC)::value;
            if (c.mixed)
                hipLaunchKernelGGL((k_xfwd_r<float, N>), grid, blk, q.lds, s, us, vs, ws, f.spec, f.tw, f.sc, c, pl, ppb,
                                   f.ld);
            else
                hipLaunchKernelGGL((k_xfwd_r<double, N>), grid, blk, q.lds, s, f.us, f.vs, f.ws, f.spec, f.tw, f.sc, c,
                                   pl, ppb, f.ld);
        });
    } else if (c.mixed) {
        hipLaunchKernelGGL(k_xfwd<float>, grid, blk, q.lds, s, us, vs, ws, f.spec, f.tw, f.sc, c, pl, ppb, f.ld);
    } else {
        hipLaunchKernelGGL(k_xfwd<double>, grid, blk, q.lds, s, f.us, f.vs, f.ws, f.spec, f.tw, f.sc, c, pl, ppb, f.ld);
    }
    li->name = "xfwd_div"; li->bytes = (c.mixed ? 2.5 : 4.0) * F(c);
}

void launch_plane_fwd(const Fields &f, const Consts &c, hipStream_t s, LaunchInfo *li)
{
    with_plane_n(c.n, [&](auto NC) {
        constexpr int N = decltype(NC)::value;
        const dim3 grid(N), blk(plane_threads(N));
        if (c.mixed)
            hipLaunchKernelGGL((k_plane_fwd<float, N>), grid, blk, plane_lds(N), s, (const float *)f.us,
                               (const float *)f.vs, (const float *)f.ws, f.spec, f.tw, f.sc, c, f.ld);
        else
            hipLaunchKernelGGL((k_plane_fwd<double, N>), grid, blk, plane_lds(N), s, f.us, f.vs, f.ws, f.spec, f.tw, f.sc,
                               c, f.ld);
    });
    li->name = "plane_fwd"; li->bytes = (c.mixed ? 2.5 : 4.0) * F(c);
}

void launch_plane_inv(const Fields &f, const Consts &c, hipStream_t s, LaunchInfo *li)
{
    with_plane_n(c.n, [&](auto NC) {
        constexpr int N = decltype(NC)::value;
        hipLaunchKernelGGL(k_plane_inv<N>, dim3(N), dim3(plane_threads(N)), plane_lds(N), s, f.spec, f.p, f.tw, f.sc, f.ld);
    });
    li->name = "plane_inv"; li->bytes = 16.0 * (double)(c.n / 2 + 1) * c.n * c.n + F(c);
}

void launch_ypass(const Fields &f, const Consts &c, const FftPlan &pl, const Tuning &tu, int inverse,
                  hipStream_t s, LaunchInfo *li)
{
    const FftPass q = col_pass(pl, tu.v[KNOB_YTILE], FFT_BOX);
    const int tkx = q.lines, nh = c.n / 2 + 1;
    const dim3 grid((nh + tkx - 1) / tkx, c.n), blk(q.threads);
    if (q.regs) {
        with_n<false>(q.n, [&](auto NC) {
            constexpr int N = decltype(NC)::value, TK = N ? rtile_n(N) : 0;
            if (inverse)
                hipLaunchKernelGGL((k_ypass_r<1, N, TK>), grid, blk, q.lds, s, f.spec, f.tw, f.sc, pl, f.ld, tkx);
            else
                hipLaunchKernelGGL((k_ypass_r<-1, N, TK>), grid, blk, q.lds, s, f.spec, f.tw, f.sc, pl, f.ld, tkx);
        });
    } else if (inverse) {
        hipLaunchKernelGGL(k_ypass<1>, grid, blk, q.lds, s, f.spec, f.tw, f.sc, pl, f.ld, tkx);
    } else {
        hipLaunchKernelGGL(k_ypass<-1>, grid, blk, q.lds, s, f.spec, f.tw, f.sc, pl, f.ld, tkx);
    }
    li->name = inverse ? "y_inv" : "y_fwd";
    li->bytes = 2.0 * 16.0 * (double)nh * c.n * c.n;
}

void launch_zpoisson(const Fields &f, const Consts &c, const FftPlan &pl, const Tuning &tu, hipStream_t s,
                     LaunchInfo *li)
{
    const FftPass q = col_pass(pl, tu.v[KNOB_ZTILE], FFT_BOX);
    const int tkx = q.lines, nh = c.n / 2 + 1;
    const dim3 grid((nh + tkx - 1) / tkx, c.n), blk(q.threads);
    if (q.regs) {
        with_n<false>(q.n, [&](auto NC) {
            constexpr int N = decltype(NC)::value, TK = N ? rtile_n(N) : 0;
            hipLaunchKernelGGL((k_zpoisson_r<N, TK>), grid, blk, q.lds, s, f.spec, f.tw, f.ktab, f.sc, pl, f.ld, tkx);
        });
    } else {
        hipLaunchKernelGGL(k_zpoisson, grid, blk, q.lds, s, f.spec, f.tw, f.ktab, f.sc, pl, f.ld, tkx);
    }
    li->name = "z_poisson";
    li->bytes = 2.0 * 16.0 * (double)nh * c.n * c.n;
}

void launch_xinv(const Fields &f, const Consts &c, const FftPlan &pl, const Tuning &tu, hipStream_t s,
                 LaunchInfo *li)
{
    const FftPass q = x_pass(pl, tu.v[KNOB_XIPAIRS], FFT_BOX);
    const int ppb = q.lines, pairs = c.n * c.n / 2;
    const dim3 grid(pairs / ppb), blk(q.threads);
    if (q.regs) {
        with_n<false>(q.n, [&](auto NC) {
            hipLaunchKernelGGL((k_xinv_r<decltype(NC)::value>), grid, blk, q.lds, s, f.spec, f.p, f.tw, f.sc, pl, ppb, f.ld);
        });
    } else {
        hipLaunchKernelGGL(k_xinv, grid, blk, q.lds, s, f.spec, f.p, f.tw, f.sc, pl, ppb, f.ld);
    }
    li->name = "x_inv"; li->bytes = 16.0 * (double)(c.n / 2 + 1) * c.n * c.n + F(c);
}

template <typename T>
static void launch_project_t(const Fields &f, const Consts &c, hipStream_t s)
{
    const ProjectForm form = project_form(c.n);
    auto kern = form.plane ? k_project<T, 4, true> : form.lpw == 2 ? k_project<T, 2, false> : k_project<T, 0, false>;
    const dim3 grid(project_blocks(c.n)), blk(form.plane ? c.n / form.lpw * 64 : BLK);
    hipLaunchKernelGGL(kern, grid, blk, 0, s, (const T *)f.us, (const T *)f.vs, (const T *)f.ws, f.p, (T *)f.u, (T *)f.v,
                       (T *)f.w, form.plane ? f.psum : f.lsum, form.plane ? f.pmax : f.lmax, f.sc, c);
}

void launch_project(const Fields &f, const Consts &c, hipStream_t s, LaunchInfo *li)
{
    if (c.mixed) launch_project_t<float>(f, c, s);
    else launch_project_t<double>(f, c, s);
    li->name = "project"; li->bytes = (c.mixed ? 4.0 : 7.0) * F(c);
}

bool project_sums_planes(const Consts &c) { return project_form(c.n).plane; }

void launch_reduce(const Fields &f, const Consts &c, hipStream_t s, LaunchInfo *li)
{
    hipLaunchKernelGGL(k_reduce_planes, dim3(c.n, 3), dim3(64), 0, s, f.lsum, f.lmax, f.psum, f.pmax, f.sc, c.n);
    li->name = "reduce_planes"; li->bytes = 6.0 * 8.0 * c.n * c.n;
}

void launch_finalize(const Fields &f, const Consts &c, bool publish, hipStream_t s, LaunchInfo *li)
{
    hipLaunchKernelGGL(k_finalize, dim3(1), dim3(FIN_THREADS), 0, s, f.psum, f.pmax, f.sc, c, f.mirror, f.slot,
                       publish ? 1 : 0);
    li->name = "finalize"; li->bytes = 6.0 * 8.0 * c.n;
}

// Block layout of a gang step: each shared pass (phase field, momentum,
// projection, plane sums) is one 1-D launch over the blocks of every box, a
// box's blocks consecutive; the boxes' z slabs are sized from the gang's box
// count (more boxes, thicker slabs and fewer recomputed halo planes).  Boxes
// of one size form one entry of gl->size for the FFT passes.
void gang_layout(const GangBox *d, int nbox, const GangSize *sizes, GangLaunch *gl)
{
    *gl = GangLaunch{};
    gl->mixed = d[0].c.mixed;
    gl->phiflag = d[0].c.phiflag;
    for (int b = 0; b < nbox; b++) {
        const int n = d[b].c.n;
        const int ka = kz_acdi(n, gl->mixed, nbox), km = kz_momentum(n, gl->mixed, nbox);
        gl->grid[GP_ACDI].kz[b] = ka;
        gl->grid[GP_MOM].kz[b] = km;
        const int blocks[GP_COUNT] = {
            ((n + ATX - 1) / ATX) * ((n + ATY - 1) / ATY) * (n / ka),
            gl->mixed ? ((n + 2 * PTX - 1) / (2 * PTX)) * ((n + PTY - 1) / PTY) * (n / km)
                      : ((n + MTX - 1) / MTX) * ((n + MTY - 1) / MTY) * (n / km),
            (int)nblocks((size_t)n / gang_lpw(n) * n, BLK / 64), 3 * n};
        for (int q = 0; q < GP_COUNT; q++) gl->grid[q].first[b + 1] = gl->grid[q].first[b] + blocks[q];
        if (gl->nsize == 0 || gl->size[gl->nsize - 1].n != n) {
            GangSize &z = gl->size[gl->nsize++];
            z = sizes[b];
            z.off = b;
            z.cnt = 0;
            z.n = n;
            z.planes = plane_passes(d[b].c, z.tune);
        }
        gl->size[gl->nsize - 1].cnt++;
    }
}

// One step of a gang laid out by gang_layout (device descriptors g[0..nbox)),
// with the launch shapes of the one-box passes above: the shared passes once,
// the FFT passes once per size, on that size's boxes.
void launch_gang_step(const GangBox *g, int nbox, unsigned euler, bool publish, const GangLaunch &gl, hipStream_t s0,
                      const GangStreams *fs)
{
    const bool fork = fs && gl.nsize > 1 && fs->n >= gl.nsize - 1;
    hipStream_t s = s0;
    if (gl.phiflag) {
        const GangGrid &gg = gl.grid[GP_ACDI];
        const dim3 grid((unsigned)gg.first[nbox]);
        if (gl.mixed)
            hipLaunchKernelGGL(kg_acdi<float>, grid, dim3(ATHREADS), 0, s, g, nbox, gg);
        else
            hipLaunchKernelGGL(kg_acdi<double>, grid, dim3(ATHREADS), 0, s, g, nbox, gg);
    }
    {
        const GangGrid &gg = gl.grid[GP_MOM];
        const dim3 grid((unsigned)gg.first[nbox]);
        if (gl.mixed) {
            if (gl.phiflag)
                hipLaunchKernelGGL((kg_momentum_x2<1, float>), grid, dim3(PTHREADS), 0, s, g, nbox, euler, gg);
            else
                hipLaunchKernelGGL((kg_momentum_x2<0, float>), grid, dim3(PTHREADS), 0, s, g, nbox, euler, gg);
        } else {
            if (gl.phiflag)
                hipLaunchKernelGGL((kg_momentum<1, double>), grid, dim3(MTHREADS), 0, s, g, nbox, euler, gg);
            else
                hipLaunchKernelGGL((kg_momentum<0, double>), grid, dim3(MTHREADS), 0, s, g, nbox, euler, gg);
        }
    }
    if (fork) (void)hipEventRecord(fs->fork, s0);
    for (int q = 0; q < gl.nsize; q++) {
        s = fork && q > 0 ? fs->side[q - 1] : s0;
        if (fork && q > 0) (void)hipStreamWaitEvent(s, fs->fork, 0);
        const GangSize &z = gl.size[q];
        const GangBox *gs = g + z.off;
        const int nb = z.cnt, n = z.n, nh = n / 2 + 1, pairs = n * n / 2, ld = z.ld;
        const FftPlan &pl = z.plan;
        const Tuning &tu = z.tune;
        const FftPass xf = x_pass(pl, tu.v[KNOB_XPAIRS], FFT_GANG), xi = x_pass(pl, tu.v[KNOB_XIPAIRS], FFT_GANG);
        const FftPass yp = col_pass(pl, tu.v[KNOB_YTILE], FFT_GANG), zp = col_pass(pl, tu.v[KNOB_ZTILE], FFT_GANG);
        const int xp = xf.lines, xip = xi.lines, ty = yp.lines, tz = zp.lines;
        const dim3 gx(pairs / xp, nb), gxi(pairs / xip, nb), gy((nh + ty - 1) / ty, n, nb), gz((nh + tz - 1) / tz, n, nb);
        const bool planes = z.planes;
        if (planes) {
            with_plane_n(n, [&](auto NC) {
                constexpr int N = decltype(NC)::value;
                if (gl.mixed)
                    hipLaunchKernelGGL((kg_plane_fwd<float, N>), dim3(N, nb), dim3(plane_threads(N)), plane_lds(N), s, gs, ld);
                else
                    hipLaunchKernelGGL((kg_plane_fwd<double, N>), dim3(N, nb), dim3(plane_threads(N)), plane_lds(N), s, gs, ld);
            });
        } else if (xf.regs) {
            with_n<true>(xf.n, [&](auto NC) {
                constexpr int N = decltype(NC)::value;
                if (gl.mixed)
                    hipLaunchKernelGGL((kg_xfwd<float, true, N>), gx, dim3(xf.threads), xf.lds, s, gs, pl, xp, ld);
                else
                    hipLaunchKernelGGL((kg_xfwd<double, true, N>), gx, dim3(xf.threads), xf.lds, s, gs, pl, xp, ld);
            });
        } else if (gl.mixed) {
            hipLaunchKernelGGL((kg_xfwd<float, false, 0>), gx, dim3(xf.threads), xf.lds, s, gs, pl, xp, ld);
        } else {
            hipLaunchKernelGGL((kg_xfwd<double, false, 0>), gx, dim3(xf.threads), xf.lds, s, gs, pl, xp, ld);
        }
        auto ypass = [&](auto SGC) {
            constexpr int SG = decltype(SGC)::value;
            if (yp.regs)
                with_n<true>(yp.n, [&](auto NC) {
                    hipLaunchKernelGGL((kg_ypass<SG, true, decltype(NC)::value>), gy, dim3(yp.threads), yp.lds, s, gs, pl,
                                       ld, ty);
                });
            else
                hipLaunchKernelGGL((kg_ypass<SG, false, 0>), gy, dim3(yp.threads), yp.lds, s, gs, pl, ld, ty);
        };
        if (!planes) ypass(std::integral_constant<int, -1>());
        if (zp.regs)
            with_n<true>(zp.n, [&](auto NC) {
                hipLaunchKernelGGL((kg_zpoisson<true, decltype(NC)::value>), gz, dim3(zp.threads), zp.lds, s, gs, pl, ld,
                                   tz);
            });
        else
            hipLaunchKernelGGL((kg_zpoisson<false, 0>), gz, dim3(zp.threads), zp.lds, s, gs, pl, ld, tz);
        if (!planes) ypass(std::integral_constant<int, 1>());
        if (planes)
            with_plane_n(n, [&](auto NC) {
                constexpr int N = decltype(NC)::value;
                hipLaunchKernelGGL(kg_plane_inv<N>, dim3(N, nb), dim3(plane_threads(N)), plane_lds(N), s, gs, ld);
            });
        else if (xi.regs)
            with_n<true>(xi.n, [&](auto NC) {
                hipLaunchKernelGGL((kg_xinv<true, decltype(NC)::value>), gxi, dim3(xi.threads), xi.lds, s, gs, pl, xip, ld);
            });
        else
            hipLaunchKernelGGL((kg_xinv<false, 0>), gxi, dim3(xi.threads), xi.lds, s, gs, pl, xip, ld);
        if (fork && q > 0) (void)hipEventRecord(fs->join[q - 1], s);
    }
    s = s0;
    if (fork)
        for (int q = 1; q < gl.nsize; q++) (void)hipStreamWaitEvent(s0, fs->join[q - 1], 0);
    const GangGrid &gp = gl.grid[GP_PROJECT], &gr = gl.grid[GP_PLANES];
    if (gl.mixed)
        hipLaunchKernelGGL(kg_project<float>, dim3((unsigned)gp.first[nbox]), dim3(BLK), 0, s, g, nbox, gp);
    else
        hipLaunchKernelGGL(kg_project<double>, dim3((unsigned)gp.first[nbox]), dim3(BLK), 0, s, g, nbox, gp);
    hipLaunchKernelGGL(kg_reduce_planes, dim3((unsigned)gr.first[nbox]), dim3(64), 0, s, g, nbox, gr);
    hipLaunchKernelGGL(kg_finalize, dim3(nbox), dim3(FIN_THREADS), 0, s, g, publish ? 1 : 0);
}

// Inverse 3-D transform of the half spectrum into `out` (n^3, x fastest):
// z inverse, y inverse, x complex-to-real; unnormalised.
void launch_ic_potential(const Fields &f, const Consts &c, const FftPlan &pl, const Tuning &tu, int comp,
                         unsigned long long seedmix, double kp, double kmax, double *out, hipStream_t s)
{
    const size_t total = (size_t)(c.n / 2 + 1) * c.n * c.n;
    const unsigned g = nblocks(total, BLK) < 65536 ? nblocks(total, BLK) : 65536;
    hipLaunchKernelGGL(k_ic_spectrum, dim3(g), dim3(BLK), 0, s, f.spec, c.n, f.ld, comp, seedmix, kp, kmax);
    const int nh = c.n / 2 + 1;
    const FftPass q = col_pass(pl, tu.v[KNOB_ZTILE], FFT_START);
    hipLaunchKernelGGL(q.regs ? k_zinv_r : k_zinv, dim3((nh + q.lines - 1) / q.lines, c.n), dim3(q.threads), q.lds, s,
                       f.spec, f.tw, f.ktab, f.sc, pl, f.ld, q.lines);
    LaunchInfo li;
    launch_ypass(f, c, pl, tu, 1, s, &li);
    Fields g2 = f;
    g2.p = out;
    launch_xinv(g2, c, pl, tu, s, &li);
}

void launch_ic_curl(const Consts &c, const double *ax, const double *ay, const double *az, void *u, void *v,
                    void *w, double *lsum, double dx, double scale, bool sum, hipStream_t s)
{
    const dim3 grid(nblocks((size_t)c.n * c.n * 64, BLK));
    if (sum)
        hipLaunchKernelGGL((k_ic_curl<double, true>), grid, dim3(BLK), 0, s, ax, ay, az, (double *)nullptr,
                           (double *)nullptr, (double *)nullptr, lsum, c.n, dx, scale);
    else if (c.mixed)
        hipLaunchKernelGGL((k_ic_curl<float, false>), grid, dim3(BLK), 0, s, ax, ay, az, (float *)u, (float *)v,
                           (float *)w, lsum, c.n, dx, scale);
    else
        hipLaunchKernelGGL((k_ic_curl<double, false>), grid, dim3(BLK), 0, s, ax, ay, az, (double *)u, (double *)v,
                           (double *)w, lsum, c.n, dx, scale);
}

}  // namespace mhit
