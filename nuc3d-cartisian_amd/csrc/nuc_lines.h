// nuc_lines.h -- per-line interface computation shared by the production
// sweep kernels and the per-Field operator kernels.
//
// A line is held in LDS on [-HALO, NL R+HALO), with NL lanes for each sign: one
// wave owns it, lanes 0..31 reconstruct f^+ and lanes 32..63 f^- (NL = 32), or, for
// FP64 lines of 257-512 cells, two waves, one per sign (NL = 64); the reference
// does the two signs as separate sweeps (src/euler3d.cpp:334-387).  Lane h of a
// sign owns a chunk of R consecutive interfaces; f^- takes the chunks in mirrored
// order (lane h <-> chunk NL-1-h, rows reversed), which turns the f^- stencils and
// its tridiagonal system into the same shape as f^+, so both signs execute one
// instruction stream.
//
// Rank-local zones follow the reference's inner/boundary split per MPI block
// of length nloc (src/fieldOperator.cpp:387-465):
//   explicit boundary interfaces  ml in [0, ts-1] U [nloc-ts+1, nloc]
//   inner interfaces              ml in [ts, nloc-ts]
//   compact schemes: ml = ts and ml = nloc-ts are explicit closure rows,
//   ts < ml < nloc-ts are tridiagonal rows (src/crweno5.cpp:83-206).
#pragma once
#include "nuc_device.h"

#include <type_traits>

namespace nucdev {

constexpr int HALO = 4;

struct Zone {
    int nrows;    // interfaces on this line (n periodic, n+1 with ghost strips)
    int nloc;     // rank-local line length
    int ts;       // inviscid tilesize of the scheme
    int off = 0;  // position of interface 0 on the full line (a segment of a long line)
};

// Unnormalised WENO5 weights n_k ~ c_k / (eps + is_k)^2.  FP64 (b_k = 4 is_k)
// uses the division-free products c_k * s_i * s_j (one reciprocal per row in
// total); FP32 (b_k = is_k) uses c_k * rcp(s_k), since the products can leave
// FP32's range.
template <typename TW>
__device__ __forceinline__ void w5_weights(TW b0, TW b1, TW b2, TW c0, TW c1, TW c2, TW &n0, TW &n1, TW &n2)
{
    const TW eps = TW(sizeof(TW) == 8 ? 4.0e-6 : 1.0e-6);
    TW s0 = sq(eps + b0), s1 = sq(eps + b1), s2 = sq(eps + b2);
    if constexpr (sizeof(TW) == 8) {
        n0 = c0 * (s1 * s2); n1 = c1 * (s0 * s2); n2 = c2 * (s0 * s1);
    } else {
        n0 = c0 * frcp(s0); n1 = c1 * frcp(s1); n2 = c2 * frcp(s2);
    }
}

// upwind reach of a scheme's stencil, and the points it reads beyond the
// symmetric window (hccs78's 8-point central part)
template <int SCH> struct Radius {
    static constexpr int value = (SCH == WENO7JS || SCH == HCCS || SCH == HCCS78 || SCH == HCCS77) ? 3
                               : (SCH == WENO3JS || SCH == UPWIND1ST) ? 1 : 2;
};
template <int SCH> struct Extra { static constexpr int value = (SCH == HCCS78) ? 1 : 0; };

// Skewed LDS line layout: position y (y >= -B) lives at slot (y+B) + (y+B)/R,
// one pad slot after every R positions, B = HALO+2 rounded up to a multiple of
// R (the lowest position is that of the mirrored write-only dummy, cell NL R+HALO,
// y = -(HALO+2)).  The f^+ line stores cell x at y = x; the f^- line is stored mirrored,
// y = NL R-2-x (NL lanes per sign), so that both signs read their windows upwards from
// y = hR-RAD-1: the lane's window then starts at slot h*(R+1) + at(-RAD-1)
// and every window element is a compile-time offset from one base.  Lanes R
// positions apart sit R+1 slots apart (odd), so chunk reads and the
// consecutive-cell writes of the load phase hit distinct LDS banks.
// pitch(): line stride in slots, = 4 (mod 16): the y/z load mapping writes 4
// lines x 4 consecutive cells per 16 lanes, which then hit distinct banks
// (measured: y/z sweep bank-conflict cycles -79% against a pitch = 2 mod 16).
template <int R, int NL = 32> struct Skew {
    static constexpr int B = ((HALO + 2 + R - 1) / R) * R;
    __host__ __device__ static constexpr int at(int y) { return (y + B) + (y + B) / R; }
    __host__ __device__ static constexpr int mir(int x) { return at(NL * R - 2 - x); }
    // slots up to cell ncap+HALO: the last one is a write-only dummy (halo
    // writes of interior cells go there instead of branching)
    static constexpr int span(int ncap) { return at(ncap + HALO) + 1; }
    static constexpr int pitch(int ncap) { return span(ncap) + ((4 - span(ncap) % 16) + 16) % 16; }
};

// pitch of an unskewed line of ncap cells with HALO ghosts on each side and
// one dummy slot, = 4 (mod 16)
__host__ __device__ constexpr int plain_pitch(int ncap)
{
    return (ncap + 2 * HALO + 1) + ((4 - (ncap + 2 * HALO + 1) % 16) + 16) % 16;
}

// Distance-1 lane shifts as DPP moves (no LDS round trip): shr1 gives lane i
// the value of lane i-1, shl1 the value of lane i+1; the lanes without a source
// (0, resp. 63) read 0.  Across the boundary of the two half waves the values
// do move (lane 32 reads lane 31), so callers mask h == 0 / h == 31 as they
// do for the width-32 shuffles.
__device__ __forceinline__ int dpp_shr1(int x) { return __builtin_amdgcn_update_dpp(0, x, 0x138, 0xF, 0xF, true); }
__device__ __forceinline__ int dpp_shl1(int x) { return __builtin_amdgcn_update_dpp(0, x, 0x130, 0xF, 0xF, true); }
__device__ __forceinline__ double shr1(double x)
{
    return __hiloint2double(dpp_shr1(__double2hiint(x)), dpp_shr1(__double2loint(x)));
}
__device__ __forceinline__ double shl1(double x)
{
    return __hiloint2double(dpp_shl1(__double2hiint(x)), dpp_shl1(__double2loint(x)));
}
__device__ __forceinline__ float shr1(float x) { return __int_as_float(dpp_shr1(__float_as_int(x))); }
__device__ __forceinline__ float shl1(float x) { return __int_as_float(dpp_shl1(__float_as_int(x))); }

// Distance-16 exchange inside each half wave with one v_permlane16_swap per
// dword: swapping a value with itself leaves, in the first result, the lanes of
// the odd 16-lane rows holding the value of the lane 16 below (lane i-16), and,
// in the second, the lanes of the even rows holding the value of the lane 16
// above (lane i+16).  up16 is meaningful for h >= 16, dn16 for h < 16 (h = lane
// index within the half wave); the other lanes are masked by the callers.
__device__ __forceinline__ void swap16(unsigned x, unsigned &up, unsigned &dn)
{
    auto r = __builtin_amdgcn_permlane16_swap(x, x, false, false);
    up = r[0]; dn = r[1];
}
__device__ __forceinline__ void swap16(double x, double &up, double &dn)
{
    unsigned hu, hd, lu, ld;
    swap16((unsigned)__double2hiint(x), hu, hd);
    swap16((unsigned)__double2loint(x), lu, ld);
    up = __hiloint2double((int)hu, (int)lu);
    dn = __hiloint2double((int)hd, (int)ld);
}
__device__ __forceinline__ void swap16(float x, float &up, float &dn)
{
    unsigned u, d;
    swap16((unsigned)__float_as_int(x), u, d);
    up = __int_as_float((int)u); dn = __int_as_float((int)d);
}

// An empty asm that takes x and gives it back: the value must exist at this
// point, and code that uses the result cannot move above it (volatile asm
// statements keep their order).  Used to evaluate a lane's rows in order.
template <typename T> __device__ __forceinline__ void pin(T &x) { asm volatile("" : "+v"(x)); }

// Distance-32 exchange between the two halves of a wave (v_permlane32_swap):
// up is meaningful for lanes >= 32 (the value of lane i-32), dn for lanes < 32
// (lane i+32).
__device__ __forceinline__ void swap32(unsigned x, unsigned &up, unsigned &dn)
{
    auto r = __builtin_amdgcn_permlane32_swap(x, x, false, false);
    up = r[0]; dn = r[1];
}
__device__ __forceinline__ void swap32(double x, double &up, double &dn)
{
    unsigned hu, hd, lu, ld;
    swap32((unsigned)__double2hiint(x), hu, hd);
    swap32((unsigned)__double2loint(x), lu, ld);
    up = __hiloint2double((int)hu, (int)lu);
    dn = __hiloint2double((int)hd, (int)ld);
}

// normalised parallel cyclic reduction over the NL lanes (32 or 64) of one
// sign: row k: x_k + al*x_{k-1} + ga*x_{k+1} = de  ->  x_k = de on return
template <int NL, bool F32, typename T>
__device__ __forceinline__ void pcr(T &al, T &ga, T &de)
{
#pragma unroll
    for (int s = 1; s < NL; s <<= 1) {
        T alm, gam, dem, alp, gap, dep;
        if (s == 1) {
            alm = shr1(al); gam = shr1(ga); dem = shr1(de);
            alp = shl1(al); gap = shl1(ga); dep = shl1(de);
        } else if (s == 16 && NL == 32) {
            swap16(al, alm, alp); swap16(ga, gam, gap); swap16(de, dem, dep);
        } else if (s == 32) {
            swap32(al, alm, alp); swap32(ga, gam, gap); swap32(de, dem, dep);
        } else {
            alm = __shfl_up(al, s, NL); gam = __shfl_up(ga, s, NL); dem = __shfl_up(de, s, NL);
            alp = __shfl_down(al, s, NL); gap = __shfl_down(ga, s, NL); dep = __shfl_down(de, s, NL);
        }
        // no masks: lanes h < s hold al = 0 and lanes h + s >= NL hold ga = 0
        // exactly (the first and last rows do not couple outward, and each
        // level doubles those ranges), so the values they received from the
        // wrapped or neighbouring lanes, all finite, are multiplied by zero
        T r = frcp_for<F32>(T(1) - al * gam - ga * alp);
        T nal = -r * al * alm;
        T nga = -r * ga * gap;
        T nde = r * (de - al * dem - ga * dep);
        al = nal; ga = nga; de = nde;
    }
}

// Forward-eliminated rows of one lane's chunk (rows normalised):
//   r = 0: Af x_{-1} + x_0 + Cf x_1 = Df ;  r >= 1: Af x_0 + x_r + Cf x_{r+1} = Df
template <int R, typename T, int NL, bool F32 = false> struct Chunk {
    T Af[R], Cf[R], Df[R];
    __device__ __forceinline__ void row(int r, T a, T b, T c, T d)
    {
        if (r <= 1) {
            T rb = frcp_for<F32>(b);
            Af[r] = a * rb; Cf[r] = c * rb; Df[r] = d * rb;
        } else {
            T rr = frcp_for<F32>(b - a * Cf[r - 1]);
            Df[r] = rr * (d - a * Df[r - 1]);
            Af[r] = -rr * a * Af[r - 1];
            Cf[r] = rr * c;
        }
    }
    // Partition solve across the NL lanes of a sign (lane h holds chunk h in system
    // order; the first row of lane 0 and the last row of lane NL-1 must not
    // couple outward).  Solution returned in Df.  Equivalent to the
    // reference's Thomas sweep (src/crweno5.cpp:208-219) up to rounding.
    __device__ __forceinline__ void solve(int h)
    {
#pragma unroll
        for (int r = R - 3; r >= 1; r--) {
            T tD = Df[r] - Cf[r] * Df[r + 1];
            T tA = Af[r] - Cf[r] * Af[r + 1];
            Cf[r] = -Cf[r] * Cf[r + 1];
            Df[r] = tD; Af[r] = tA;
        }
        T A0, C0, D0;
        if constexpr (R == 2) {
            A0 = Af[0]; C0 = Cf[0]; D0 = Df[0];
        } else {
            T r0 = frcp_for<F32>(T(1) - Cf[0] * Af[1]);
            A0 = r0 * Af[0];
            C0 = -r0 * Cf[0] * Cf[1];
            D0 = r0 * (Df[0] - Cf[0] * Df[1]);
        }
        T A1 = Af[R - 1], C1 = Cf[R - 1], D1 = Df[R - 1];
        T A0n = shl1(A0), C0n = shl1(C0), D0n = shl1(D0);
        if (h == NL - 1) { A0n = T(0); C0n = T(0); D0n = T(0); }
        T rb = frcp_for<F32>(T(1) - A1 * C0 - C1 * A0n);
        T al = -rb * A1 * A0;
        T ga = -rb * C1 * C0n;
        T de = rb * (D1 - A1 * D0 - C1 * D0n);
        // the reduced system's first and last rows do not couple outward
        if (h == 0) al = T(0);
        if (h == NL - 1) ga = T(0);
        pcr<NL, F32>(al, ga, de);
        T X1 = de;
        T X1m = shr1(X1);
        if (h == 0) X1m = T(0);
        T X0 = D0 - A0 * X1m - C0 * X1;
#pragma unroll
        for (int r = 1; r <= R - 2; r++) Df[r] = Df[r] - Af[r] * X0 - Cf[r] * X1;
        Df[0] = X0;
        Df[R - 1] = X1;
    }
};

// WENO5 smoothness indicators and candidate values of a 5-point upwind stencil
// f0..f4 (src/weno5js.cpp, src/crweno5.cpp:87-129), computed from the
// stencil's differences d_j = f_j - f_{j-1} (j = 1..4) and second-difference
// terms e_k = 13/3 (d_{k+1} - d_k)^2 (k = 1..3), which a lane's consecutive
// rows share: f0-4f1+3f2 = 3d2-d1, f1-f3 = -(d2+d3), 3f2-4f3+f4 = d4-3d3,
// q0 = f2+(5d2-2d1)/6, q1 = f2+(d2+2d3)/6, q2 = f3-(2d3+d4)/6.  In FP64 the
// indicators come as b_k = e_k + (linear part)^2, four times is_k: the factor 1/4
// of the linear parts would be three more multiplications, and the weights only
// need the indicators' ratios (their eps is taken times four as well).  In FP32
// the linear parts are halved (b_k = is_k): the roundings of an FP32 stencil are
// seen in the results, so they stay what they were.
template <typename T> constexpr bool W5_FOUR = sizeof(T) == 8;   // b_k = 4 is_k
template <typename T> constexpr T w5_g() { return T(W5_FOUR<T> ? 13.0 / 3.0 : 13.0 / 12.0); }
// h2: the linear part of b2
template <typename T>
__device__ __forceinline__ void w5_diff(T f2, T f3, T d1, T d2, T d3, T d4, T e1, T e2, T e3, T &b0, T &b1, T &b2,
                                        T &q0, T &q1, T &q2, T &h2)
{
    if constexpr (W5_FOUR<T>) {
        const T h0 = T(3) * d2 - d1, h1 = d2 + d3;
        h2 = d4 - T(3) * d3;
        b0 = e1 + h0 * h0;
        b1 = e2 + h1 * h1;
        b2 = e3 + h2 * h2;
    } else {
        const T h0 = T(1.5) * d2 - T(0.5) * d1, h1 = T(0.5) * (d2 + d3);
        h2 = T(0.5) * d4 - T(1.5) * d3;
        b0 = e1 + h0 * h0;
        b1 = e2 + h1 * h1;
        b2 = e3 + h2 * h2;
    }
    q0 = f2 + (T(5.0 / 6.0) * d2 - T(1.0 / 3.0) * d1);
    q1 = f2 + (T(1.0 / 6.0) * d2 + T(1.0 / 3.0) * d3);
    q2 = f3 - (T(1.0 / 3.0) * d3 + T(1.0 / 6.0) * d4);
}

// The Z-type schemes multiply squared indicators (WENO5-Z and hccs rows: the 12th
// power of a flux, WENO7-Z the 4th) and hccs and its relatives square (tau/eps)^2
// once more, which leaves FP64's range from fluxes of about 1e17 on.  Their
// reconstruction scales with the line's values except for eps (1e-20, 1e-40), so a
// wave that holds a value of 2^45 (3.5e13) or more forms its rows of the values
// times a power of two that brings the largest there.  eps counts for more then,
// but against values 1e30 times smaller than the line's largest only.
// The test reads the values' high words as FP32 numbers, which order as the doubles
// do (infinities and NaN are numbers to neither, and pass): one instruction for two
// values, where a row has 75 to 210.  Rows formed twice, with a quotient for each
// indicator the second time, cost registers instead: 5 % on average, hccs78 twice
// the time in some forms; this is 0.6 %, at most 3 (kernels of hccs and WENO7).
template <int SCH> constexpr bool z_type()
{
    return SCH == WENO5Z || SCH == WENO7JS || SCH == HCCS || SCH == HCCS77 || SCH == HCCS78;
}
struct LineScale {
    int k = 0;   // of the wave, in the place of a double's exponent
    __device__ __forceinline__ double down() const { return __hiloint2double((1023 << 20) - k, 0); }
    __device__ __forceinline__ double up() const { return __hiloint2double((1023 << 20) + k, 0); }
    __device__ __forceinline__ bool on() const { return __builtin_expect(k != 0, 0); }
    // looks at f[FROM .. FROM + COUNT), which hold every value of the line in some lane
    template <int FROM, int COUNT, int N> __device__ __forceinline__ void apply(double (&f)[N])
    {
        float m = 0.f;
#pragma unroll
        for (int i = FROM; i < FROM + COUNT; i += 2)
            asm("v_max3_f32 %0, %1, |%2|, |%3|"
                : "=v"(m) : "v"(m), "v"(__double2hiint(f[i])), "v"(__double2hiint(f[i + 1 < FROM + COUNT ? i + 1 : i])));
        constexpr int TOP = (1023 + 45) << 20;
        if (__builtin_expect(__any(__float_as_int(m) >= TOP), 0)) {
            // the exponent of the wave's largest value above 2^45, bit by bit
#pragma unroll 1
            for (int b = 512 << 20; b >= 1 << 20; b >>= 1)
                if (__any(__float_as_int(m) >= TOP + k + b)) k += b;
#pragma unroll
            for (int i = 0; i < N; i++) f[i] *= down();
        }
    }
};

// The explicit rows of a compact line of one block (2 ts + 1 around interfaces
// 0 and nloc, ts the scheme's own tilesize), numbered k = 0 .. 2 (2 ts + 1) - 1:
// the interface m of row k; its place in row order is m of f^+, NL R - 1 - m of f^-.
template <int SCH> constexpr int edge_ts() { return SCH == HCCS ? 4 : 3; }
// Their values are kept in the pad slots of the line's buffer (one after every R
// positions, Skew<R>), which nothing else uses: row k in slot edge_slot(k).
template <int R, int NL> __host__ __device__ constexpr int edge_slot(int k)
{
    static_assert(17 * (R + 1) + R < Skew<R, NL>::span(NL * R), "a pad slot for every explicit row");
    return k * (R + 1) + R;
}
template <int SCH> __device__ __forceinline__ int edge_row(const Zone &z, int k)
{
    constexpr int ts = edge_ts<SCH>(), ne = 2 * ts + 1;
    return k < ne ? k - ts : z.nloc + k - ne - ts;
}
template <int SCH> __device__ __forceinline__ bool edge_mine(const Zone &z, int k, int m)
{
    return k < 2 * (2 * edge_ts<SCH>() + 1) && m >= 0 && m <= z.nloc;
}

// Reconstruct one sign of a line.  Lw points at the lane's window in the
// skewed line buffer (slot h*(R+1); the f^- buffer is mirrored, see Skew):
// win[t] = Lw[at(t-RAD-1)] in upwind order, row r uses win[r .. r+2*RAD] in
// upwind coordinates.  m0r is the interface index of row 0 and mstep its step
// (+1 for f^+, -1 for f^- whose rows run backwards).
// T is the type of the stencils (smoothness indicators, candidate values);
// TW the type of the nonlinear weights and compact rows; TS the type of the
// tridiagonal solve and of the result (FP64 in both precision paths).
// NL: lanes per sign, h in [0, NL).
// full: every row of every lane is an interface of the line (n = NL R).
// EDGE_AHEAD (the line is one block): the explicit rows of CRWENO5 and hccs are
// evaluated ahead.  They are then in slot edge_slot(k) of the wave's and sign's
// line buffer Lx, and out[] of those rows is meaningless.
// tails: rows past the line's last interface read defined (finite) cells.
// PERIODIC: cells outside the lanes' own R positions are images of cells inside.
enum { EDGE_IN_LOOP = 0, EDGE_AHEAD = 1 };
template <int SCH, int R, typename T, typename TW, typename TS, int NL = 32, int EDGE = EDGE_IN_LOOP, bool PERIODIC = false>
__device__ __forceinline__ void line_half(const T *Lw, int m0r, int mstep, const Zone &z, int h, bool neg,
                                          TS out[R], bool full = false, TS *Lx = nullptr, bool tails = false)
{
    constexpr int RAD = Radius<SCH>::value;
    constexpr int W = R + 2 * RAD + Extra<SCH>::value;
    T win[W];
    constexpr bool SCALED = z_type<SCH>() && sizeof(T) == 8;
    constexpr int LOOK = PERIODIC ? RAD + 1 : 0, LOOKS = PERIODIC ? R : W;   // LineScale
    LineScale sc;
    if constexpr (EDGE == EDGE_IN_LOOP) {
#pragma unroll
        for (int t = 0; t < W; t++) win[t] = Lw[Skew<R>::at(t - RAD - 1)];
        if constexpr (SCALED) sc.template apply<LOOK, LOOKS>(win);
    }
    // rank-local position of each row, without integer division in the loop
    int ml[R];
    {
        int m = m0r;
        int l = (m + z.off) % z.nloc;
#pragma unroll
        for (int r = 0; r < R; r++) {
            ml[r] = l;
            l += mstep;
            if (l >= z.nloc) l -= z.nloc;
            if (l < 0) l += z.nloc;
        }
    }
    if constexpr (SCH == WENO5JS) {
        // rows in order through a rolling window of differences (see CRWENO5)
        T f2 = win[2], f3 = win[3];
        T d1 = win[1] - win[0], d2 = f2 - win[1], d3 = f3 - f2;
        T e1 = w5_g<T>() * sq(d2 - d1), e2 = w5_g<T>() * sq(d3 - d2);
#pragma unroll
        for (int r = 0; r < R; r++) {
            T f4 = win[r + 4];
            T d4 = f4 - f3;
            T e3 = w5_g<T>() * sq(d4 - d3);
            T b0, b1, b2, q0, q1, q2, h2;
            w5_diff<T>(f2, f3, d1, d2, d3, d4, e1, e2, e3, b0, b1, b2, q0, q1, q2, h2);
            // alpha_k = c_k / s_k, normalised with a single reciprocal
            TW n0, n1, n2;
            w5_weights<TW>(TW(b0), TW(b1), TW(b2), TW(0.1), TW(0.6), TW(0.3), n0, n1, n2);
            TS o = TS((n0 * TW(q0) + n1 * TW(q1) + n2 * TW(q2)) * frcp(n0 + n1 + n2));
            pin(o); pin(f3); pin(f4); pin(d3); pin(d4); pin(e2); pin(e3);
            out[r] = o;
            f2 = f3; f3 = f4; d1 = d2; d2 = d3; d3 = d4; e1 = e2; e2 = e3;
        }
    } else if constexpr (SCH == WENO5Z) {
        // rows in order through a rolling window of differences (see CRWENO5)
        T f2 = win[2], f3 = win[3];
        T d1 = win[1] - win[0], d2 = f2 - win[1], d3 = f3 - f2;
        T e1 = w5_g<T>() * sq(d2 - d1), e2 = w5_g<T>() * sq(d3 - d2);
#pragma unroll
        for (int r = 0; r < R; r++) {
            T f4 = win[r + 4];
            T d4 = f4 - f3;
            T e3 = w5_g<T>() * sq(d4 - d3);
            T b0, b1, b2, q0, q1, q2, h2;
            w5_diff<T>(f2, f3, d1, d2, d3, d4, e1, e2, e3, b0, b1, b2, q0, q1, q2, h2);
            // the positive inner sweep's is2 reads f_{i+1} twice (src/weno5z.cpp:80):
            // (f2 - f3)^2 in place of its squared second difference
            bool typo = !neg && ml[r] >= z.ts && ml[r] <= z.nloc - z.ts;
            b2 = (typo ? w5_g<T>() * sq(d3) : e3) + h2 * h2;
            // alpha_k = c_k (1 + (tau/s_k)^2), s_k = is_k + eps (src/weno5z.cpp:84-92),
            // scaled by s_0^2 s_1^2 s_2^2: no quotient is left but the normalisation
            // (three IEEE quotients are 35 of the plain form's 75 instructions).  The
            // products hold fluxes up to about 1e21 (LineScale keeps them below).  FP32
            // stencils keep the plain form and its roundings (weno7z).
            const TW eps = TW(W5_FOUR<T> ? 4.0e-40 : 1.0e-40);
            const TW B0 = b0, B1 = b1, B2 = b2;
            TW a0, a1, a2;
            if constexpr (sizeof(T) == 8) {
                const TW S0 = sq(B0 + eps), S1 = sq(B1 + eps), S2 = sq(B2 + eps), T2 = sq(B2 - B0);
                a0 = TW(0.1) * ((S0 + T2) * (S1 * S2));
                a1 = TW(0.6) * ((S1 + T2) * (S0 * S2));
                a2 = TW(0.3) * ((S2 + T2) * (S0 * S1));
            } else {
                TW tau = fabs(B2 - B0);
                auto t = [&](TW s) {
                    const TW x = fmin(s, TW(1.0e280));   // an indicator beyond FP32's range
                    return fquot(tau, x, frcp_for<true>(x));
                };
                a0 = TW(0.1) * (TW(1) + sq(t(B0 + eps)));
                a1 = TW(0.6) * (TW(1) + sq(t(B1 + eps)));
                a2 = TW(0.3) * (TW(1) + sq(t(B2 + eps)));
            }
            TS o = TS((a0 * TW(q0) + a1 * TW(q1) + a2 * TW(q2)) * frcp_for<sizeof(T) == 4>(a0 + a1 + a2));
            pin(o); pin(f3); pin(f4); pin(d3); pin(d4); pin(e2); pin(e3);
            out[r] = o;
            f2 = f3; f3 = f4; d1 = d2; d2 = d3; d3 = d4; e1 = e2; e2 = e3;
        }
    } else if constexpr (SCH == WENO7JS) {
        // rows in order through a rolling 7-point window (see CRWENO5 below)
        T fw[7];
#pragma unroll
        for (int j = 0; j < 6; j++) fw[j] = win[j];
#pragma unroll
        for (int r = 0; r < R; r++) {
            fw[6] = win[r + 6];
            TS o = TS(weno7z<T, TW>(fw, TW(1.0e-20)));
            pin(o);
#pragma unroll
            for (int j = 1; j < 7; j++) pin(fw[j]);
            out[r] = o;
#pragma unroll
            for (int j = 0; j < 6; j++) fw[j] = fw[j + 1];
        }
    } else if constexpr (SCH == WENO3JS) {
#pragma unroll
        for (int r = 0; r < R; r++) out[r] = TS(weno3js<T, TW>(win + r));
    } else if constexpr (SCH == UPWIND1ST) {
        // src/upwind1st.cpp:56-113: the upwind cell itself
#pragma unroll
        for (int r = 0; r < R; r++) out[r] = TS(win[r + 1]);
    } else if constexpr (SCH == HCCS78) {
        // blend on the inner interfaces ts..nloc-ts (src/hccs78.cpp:56-60),
        // WENO7-Z on the edge interfaces (:207-304)
        T fw[8];
#pragma unroll
        for (int j = 0; j < 7; j++) fw[j] = win[j];
#pragma unroll
        for (int r = 0; r < R; r++) {
            fw[7] = win[r + 7];
            bool edge = ml[r] < z.ts || ml[r] > z.nloc - z.ts;
            TS o = TS(hccs78_value<T, TW>(fw, edge));
            pin(o);
#pragma unroll
            for (int j = 1; j < 8; j++) pin(fw[j]);
            out[r] = o;
#pragma unroll
            for (int j = 0; j < 7; j++) fw[j] = fw[j + 1];
        }
    } else if constexpr (SCH == CRWENO5 && sizeof(T) == 4) {
        // FP32 stencils: the explicit rows in place (see below; their FP32
        // arithmetic costs half, and no form of them ahead was faster)
        Chunk<R, TS, NL, true> ch;
        // Rows in order: a rolling window (f1..f4, the differences d1..d4 and
        // the second-difference terms e1..e3 of the current row), where the
        // values the next row reuses and the row's own coefficients pass
        // through an empty asm.  Left free,
        // the compiler evaluates every row's weights before the first
        // elimination step and holds about ten values per row (233 registers,
        // 2 waves per SIMD, against 164 and 3 waves in order).
        T f1 = win[1], f2 = win[2], f3 = win[3];
        T d1 = f1 - win[0], d2 = f2 - f1, d3 = f3 - f2;
        T e1 = w5_g<T>() * sq(d2 - d1), e2 = w5_g<T>() * sq(d3 - d2);
#pragma unroll
        for (int r = 0; r < R; r++) {
            T f4 = win[r + 4];
            T d4 = f4 - f3;
            T e3 = w5_g<T>() * sq(d4 - d3);
            T b0, b1, b2, q0, q1, q2, h2;
            w5_diff<T>(f2, f3, d1, d2, d3, d4, e1, e2, e3, b0, b1, b2, q0, q1, q2, h2);
            TW P0, P1, P2;   // weights with unit ideal weights
            w5_weights<TW>(TW(b0), TW(b1), TW(b2), TW(1), TW(1), TW(1), P0, P1, P2);
            // Every row is scaled by a factor of its own, which leaves the
            // tridiagonal solution unchanged.  The explicit WENO5-JS closure
            // (src/crweno5.cpp:87-129) becomes the row (sum n_k) x = sum n_k q_k
            // with the unnormalised JS weights n_k; the compact row
            // (src/crweno5.cpp:133-162) is scaled by 3 times the weight
            // denominator.
            TW n0 = TW(0.1) * P0, n1 = TW(0.6) * P1, n2 = TW(0.3) * P2;
            TW be = n0 + n1 + n2;
            TW de = n0 * TW(q0) + n1 * TW(q1) + n2 * TW(q2);
            TW m0 = TW(0.2) * P0, m1 = TW(0.5) * P1, m2 = TW(0.3) * P2;
            TW lo = TW(2) * m0 + m1;
            TW di = m0 + TW(2) * (m1 + m2);
            TW hi = m2;
            TW rhs = (m0 * TW(f1) + (TW(5) * (m0 + m1) + m2) * TW(f2) + (m1 + TW(5) * m2) * TW(f3)) * TW(0.5);
            int m = m0r + mstep * r;
            bool valid = full || m < z.nrows;
            bool expl = ml[r] <= z.ts || ml[r] >= z.nloc - z.ts;
            TS a = (valid && !expl) ? TS(lo) : TS(0);
            TS b = valid ? TS(expl ? be : di) : TS(1);
            TS c = (valid && !expl) ? TS(hi) : TS(0);
            TS d = valid ? TS(expl ? de : rhs) : TS(0);
            // the previous row's elimination step is done before this row's
            // coefficients are released, so that rows do not queue up for it
            if (r > 0) {
                pin(ch.Af[r - 1]); pin(ch.Cf[r - 1]); pin(ch.Df[r - 1]);
            }
            asm volatile("" : "+v"(f2), "+v"(f3), "+v"(f4), "+v"(d3), "+v"(d4), "+v"(e2), "+v"(e3),
                              "+v"(a), "+v"(b), "+v"(c), "+v"(d));
            ch.row(r, a, b, c, d);
            f1 = f2; f2 = f3; f3 = f4; d1 = d2; d2 = d3; d3 = d4; e1 = e2; e2 = e3;
        }
        ch.solve(h);
#pragma unroll
        for (int r = 0; r < R; r++) out[r] = ch.Df[r];
    } else if constexpr (SCH == CRWENO5 || SCH == HCCS) {
        // The explicit rows (2 ts + 1 around every block edge) lie in a few
        // lanes only, but evaluated in the row loop every row of every wave pays
        // for them: 27 of CRWENO5's 97 instructions a row (the candidate values,
        // the explicit row, the choice between the two), 150 of hccs's.  On a
        // line of one block lane h evaluates the h-th of them ahead, and the
        // rows next to them take their values to the right-hand side.  The rows
        // the loop still forms at their places are ordinary compact rows that no
        // other row reads.
        // Measured with the shorter indicators and reciprocals of the same rows, us
        // x/y/z: CRWENO5/LF 192^3 367/412/414 -> 361/400/385, 256^3 818/903/885 ->
        // 825/851/836 (the x sweep, which applies the update, spills 6 registers),
        // with AUSM 914/968/950 -> 862/914/890; hccs/LF 256^3 1220/1212/1184 ->
        // 1133/1130/1118.
        constexpr int RAD5 = 2;   // the 5-point stencil's window is win[O..]
        constexpr int O = RAD - RAD5;
        Chunk<R, TS, NL> ch;
        constexpr bool AHEAD = EDGE == EDGE_AHEAD;
        auto scale_edges = [&](TS f) {   // the explicit rows' values with the line's
            if (h < 2 * (2 * edge_ts<SCH>() + 1)) Lx[edge_slot<R, NL>(h)] *= f;
            __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
            __builtin_amdgcn_wave_barrier();
            __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
        };
        if constexpr (AHEAD) {
            const T *const Lb = Lw - h * (R + 1);
            const int m = edge_row<SCH>(z, h);
            const int y = !edge_mine<SCH>(z, h, m) ? 0 : (neg ? NL * R - 1 - m : m);
            T fe[2 * RAD + 1];
#pragma unroll
            for (int j = 0; j < 2 * RAD + 1; j++) fe[j] = Lb[Skew<R>::at(y - RAD - 1 + j)];
            TS x;
            if constexpr (SCH == HCCS) {
                LineScale se;
                if constexpr (SCALED) se.template apply<0, 2 * RAD + 1>(fe);
                x = TS(weno7z<T, TW>(fe, TW(1.0e-40)));
                if (se.on()) x *= se.up();
            } else {
                const T c1 = fe[1] - fe[0], c2 = fe[2] - fe[1], c3 = fe[3] - fe[2], c4 = fe[4] - fe[3];
                const T k1 = w5_g<T>() * sq(c2 - c1), k2 = w5_g<T>() * sq(c3 - c2), k3 = w5_g<T>() * sq(c4 - c3);
                T b0, b1, b2, q0, q1, q2, h2;
                w5_diff<T>(fe[2], fe[3], c1, c2, c3, c4, k1, k2, k3, b0, b1, b2, q0, q1, q2, h2);
                TW P0, P1, P2;
                w5_weights<TW>(TW(b0), TW(b1), TW(b2), TW(1), TW(1), TW(1), P0, P1, P2);
                const TW n0 = TW(0.1) * P0, n1 = TW(0.6) * P1, n2 = TW(0.3) * P2;
                x = TS(n0 * TW(q0) + n1 * TW(q1) + n2 * TW(q2)) * frcp(TS(n0 + n1 + n2));
            }
            if (h < 2 * (2 * edge_ts<SCH>() + 1)) Lx[edge_slot<R, NL>(h)] = x;
            __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
            __builtin_amdgcn_wave_barrier();
            __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
            // the window is read after the explicit rows, whose registers it takes
            asm volatile("; explicit rows ahead" ::: "memory");
#pragma unroll
            for (int t = 0; t < W; t++) win[t] = Lw[Skew<R>::at(t - RAD - 1)];
            if constexpr (SCALED) {
                sc.template apply<LOOK, LOOKS>(win);
                if (sc.on()) scale_edges(sc.down());
            }
        }
        // rows in order, as above
        T f1 = win[O + 1], f2 = win[O + 2], f3 = win[O + 3];
        T d1 = f1 - win[O], d2 = f2 - f1, d3 = f3 - f2;
        T e1 = w5_g<T>() * sq(d2 - d1), e2 = w5_g<T>() * sq(d3 - d2);
#pragma unroll
        for (int r = 0; r < R; r++) {
            T f4 = win[O + r + 4];
            T d4 = f4 - f3;
            T e3 = w5_g<T>() * sq(d4 - d3);
            T b0, b1, b2, q0, q1, q2, h2;
            w5_diff<T>(f2, f3, d1, d2, d3, d4, e1, e2, e3, b0, b1, b2, q0, q1, q2, h2);
            // Every row is scaled by a factor of its own, which leaves the
            // tridiagonal solution unchanged: the compact row
            // (src/crweno5.cpp:133-162) by 3 times the weight denominator, the
            // explicit WENO5-JS closure (src/crweno5.cpp:87-129) as the row
            // (sum n_k) x = sum n_k q_k with the unnormalised JS weights n_k.
            TW lo, di, hi, rhs;
            TW be = TW(0), de = TW(0);   // the explicit row, formed in place
            TW P0, P1, P2;   // weights with unit ideal weights
            if constexpr (SCH == HCCS) {
                hccs_row<T, TW>(f1 - d1, f1, f2, f3, f4, b0, b1, b2, lo, di, hi, rhs);
            } else {
                w5_weights<TW>(TW(b0), TW(b1), TW(b2), TW(1), TW(1), TW(1), P0, P1, P2);
                if constexpr (!AHEAD) {
                    const TW n0 = TW(0.1) * P0, n1 = TW(0.6) * P1, n2 = TW(0.3) * P2;
                    be = n0 + n1 + n2;
                    de = n0 * TW(q0) + n1 * TW(q1) + n2 * TW(q2);
                }
                TW m0 = TW(0.2) * P0, m1 = TW(0.5) * P1, m2 = TW(0.3) * P2;
                lo = TW(2) * m0 + m1;
                di = m0 + TW(2) * (m1 + m2);
                hi = m2;
                rhs = (m0 * TW(f1) + (TW(5) * (m0 + m1) + m2) * TW(f2) + (m1 + TW(5) * m2) * TW(f3)) * TW(0.5);
            }
            TS a = TS(lo), b = TS(di), c = TS(hi), d = TS(rhs);
            const bool valid = full || tails || m0r + mstep * r < z.nrows;
            if constexpr (AHEAD) {
                // the block's first and last compact rows, in row order: of a
                // full line (n = NL R) they can only be these r
                constexpr int ts = edge_ts<SCH>();
                if (!full || r == (ts + 1) % R || r == ts % R || r == (NL * R - ts - 1) % R || r == (NL * R - ts - 2) % R) {
                    const bool first = ml[r] == (neg ? z.nloc - ts - 1 : ts + 1);
                    const bool last = ml[r] == (neg ? ts + 1 : z.nloc - ts - 1);
                    // the explicit rows before and after, in row order
                    const TS xlo = Lx[edge_slot<R, NL>(2 * ts)], xhi = Lx[edge_slot<R, NL>(2 * ts + 1)];
                    const TS xp = neg ? xhi : xlo, xn = neg ? xlo : xhi;
                    d -= (first ? a : TS(0)) * xp + (last ? c : TS(0)) * xn;
                    if (first) a = TS(0);
                    if (last) c = TS(0);
                }
                if (!valid) { a = TS(0); b = TS(1); c = TS(0); d = TS(0); }
            } else {
                const bool expl = ml[r] <= z.ts || ml[r] >= z.nloc - z.ts;
                if constexpr (SCH == HCCS) {
                    // through the asm as well, so that the rows' WENO7 values
                    // are formed one after the other
                    T fw[7];
#pragma unroll
                    for (int j = 0; j < 7; j++) { fw[j] = win[r + j]; pin(fw[j]); }
                    TS x = TS(0);
                    if (expl) x = TS(weno7z<T, TW>(fw, TW(1.0e-40)));
                    pin(x);
                    if (expl) { a = TS(0); b = TS(1); c = TS(0); d = x; }
                    if (!valid) { a = TS(0); b = TS(1); c = TS(0); d = TS(0); }
                } else {
                    a = (valid && !expl) ? TS(lo) : TS(0);
                    b = valid ? TS(expl ? be : di) : TS(1);
                    c = (valid && !expl) ? TS(hi) : TS(0);
                    d = valid ? TS(expl ? de : rhs) : TS(0);
                }
            }
            // the previous row's elimination step is done before this row's
            // coefficients are released, so that rows do not queue up for it
            if (r > 0) {
                pin(ch.Af[r - 1]); pin(ch.Cf[r - 1]); pin(ch.Df[r - 1]);
            }
            asm volatile("" : "+v"(f2), "+v"(f3), "+v"(f4), "+v"(d3), "+v"(d4), "+v"(e2), "+v"(e3),
                              "+v"(a), "+v"(b), "+v"(c), "+v"(d));
            ch.row(r, a, b, c, d);
            f1 = f2; f2 = f3; f3 = f4; d1 = d2; d2 = d3; d3 = d4; e1 = e2; e2 = e3;
        }
        if constexpr (AHEAD && SCALED)
            if (sc.on()) scale_edges(sc.up());
        ch.solve(h);
#pragma unroll
        for (int r = 0; r < R; r++) out[r] = ch.Df[r];
    } else if constexpr (SCH == HCCS77) {
        // compact rows on ts+1..nloc-ts-1, WENO7-Z rows at ts and nloc-ts and
        // on the edges (src/hccs77.cpp:86-163, :349-455)
        Chunk<R, TS, NL> ch;
        T fw[7];
#pragma unroll
        for (int j = 0; j < 6; j++) fw[j] = win[j];
#pragma unroll
        for (int r = 0; r < R; r++) {
            fw[6] = win[r + 6];
            const T *f = fw;
            int m = m0r + mstep * r;
            bool valid = full || m < z.nrows;
            bool expl = ml[r] <= z.ts || ml[r] >= z.nloc - z.ts;
            TW a, b, c, d;
            hccs77_row<T, TW>(f, expl, a, b, c, d);
            if (!valid && !tails) { a = TW(0); b = TW(1); c = TW(0); d = TW(0); }
            TS as = TS(a), bs = TS(b), cs = TS(c), ds = TS(d);
            if (r > 0) {
                pin(ch.Af[r - 1]); pin(ch.Cf[r - 1]); pin(ch.Df[r - 1]);
            }
            pin(as); pin(bs); pin(cs); pin(ds);
#pragma unroll
            for (int j = 1; j < 7; j++) pin(fw[j]);
            ch.row(r, as, bs, cs, ds);
#pragma unroll
            for (int j = 0; j < 6; j++) fw[j] = fw[j + 1];
        }
        ch.solve(h);
#pragma unroll
        for (int r = 0; r < R; r++) out[r] = ch.Df[r];
    }
    if constexpr (SCALED) {
        if (sc.on()) {
#pragma unroll
            for (int r = 0; r < R; r++) out[r] *= sc.up();
        }
    }
}

// First derivative at cell c of a line buffer L (cd2 / cd6 / cd8); `inner` selects
// the inner-loop form of cd8 (src/centraldifference6th.cpp:42-48,
// src/centraldifference8th.cpp:52-66 inner, :127-131 edges).
template <typename T>
__device__ __forceinline__ T central_diff(const T *L, int c, bool inner, int vis, T inv_h)
{
    if (vis == VIS_CD2) return T(0.5) * (L[c + 1] - L[c - 1]) * inv_h;   // src/centraldifference2nd.cpp:38-40
    if (vis == VIS_CD6) {
        return (T(1.0 / 60.0) * (L[c + 3] - L[c - 3]) + T(-3.0 / 20.0) * (L[c + 2] - L[c - 2])
                + T(3.0 / 4.0) * (L[c + 1] - L[c - 1])) * inv_h;
    }
    if (inner) {
        T an = T(-1.0 / 280.0) * L[c - 4] + T(4.0 / 105.0) * L[c - 3] + T(-1.0 / 5.0) * L[c - 2] + T(4.0 / 5.0) * L[c - 1];
        T ap = T(4.0 / 5.0) * L[c + 1] + T(-1.0 / 5.0) * L[c + 2] + T(4.0 / 105.0) * L[c + 3] + T(-1.0 / 280.0) * L[c + 4];
        return (ap - an) * inv_h;
    }
    return (T(-1.0 / 280.0) * (L[c + 4] - L[c - 4]) + T(4.0 / 105.0) * (L[c + 3] - L[c - 3])
            + T(-1.0 / 5.0) * (L[c + 2] - L[c - 2]) + T(4.0 / 5.0) * (L[c + 1] - L[c - 1])) * inv_h;
}

}  // namespace nucdev
