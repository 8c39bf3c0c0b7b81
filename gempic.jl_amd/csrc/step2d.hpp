// step2d.hpp -- the 2D3V Strang step as one particle pass (split2d.hip).
//
// Within a step Hp1, Hp2 and Hp3 read only B, which none of them changes,
// and change only E, which none of them reads; the HE that ends a step and
// the HE that begins the next kick at the same positions. So between two
// field solves a particle's whole step runs in registers,
//   HE (with E of the step before's end and E of this step, summed), Hp3, Hp2, Hp1, Hp2, Hp3,
// and its currents are summed once: 88 bytes per particle and step (x1, x2,
// v1, v2, v3, w read, five written) where the seven passes of the operators
// move 472.
//
// A workgroup holds what its particles reach in LDS: E and B (six grids) and
// the three current grids, each of `hr` rows of `s` doubles with halos, so
// that a stencil is constant offsets from the cell. Where nine whole grids fit
// in 160 KB (48 x 36 at degree 3) every workgroup holds them all. Else
// (64 x 64: 9 x 37 KB) the grid is cut into strips of `h` rows; the particles
// are binned by strip every few steps, a workgroup works on one strip and
// holds it with `m` rows to spare on both sides, as particles drift between
// binnings. The few particles that leave the rows held, or cross more than one
// cell in a push, are put on a list and done from global memory by a kernel of
// its own (in the pass itself, the general form's registers made it spill).
//
// Bound by LDS: at degree 3, 127 reads per particle and 7 more for each of the
// three pushes that crosses a cell, 68 to 80 atomic adds; its pipe is busy 97 % of
// a CU's cycles, 50 per particle, 46 % of the cycles in bank conflicts of lanes at
// random nodes (VALU 26 %; counters at 16,777,216 particles, 64 x 64). The shared row sums below
// keep the reads down: B1's rows serve Hp3 and the neighbouring
// Hp2, and a path that stays in its cell deposits 3 rows, not 4.
#pragma once

// sub-steps of a pass; the last step of a call runs as two passes, because
// j_dofs end as the currents of its last Hp1, Hp2 and Hp3
enum F2Mode : int { F2_HE = 1, F2_HP3A = 2, F2_HP2A = 4, F2_HP1 = 8, F2_HP2B = 16, F2_HP3B = 32 };
constexpr int F2_FIRST = F2_HE | F2_HP3A | F2_HP2A, F2_SECOND = F2_HP1 | F2_HP2B | F2_HP3B;
constexpr int F2_ALL = F2_FIRST | F2_SECOND;

// threads of the pass: at degree 3 it needs more registers than 16 waves a CU
// leave it (128; it spilled 31)
constexpr int f2_threads(int p) { return p == 3 ? 768 : 1024; }
constexpr int kF2Lds = 163840;             // bytes of LDS of a CU
constexpr int kF2StripsMax = 64;

struct F2Args {
    int64_t n;
    int nx, ny;
    int s, hr;                      // LDS row stride (doubles) and rows held
    int strips, h, m;               // strips = 1: the whole grid (h, m unused)
    int64_t chunk;                  // strips = 1: particles per workgroup
    const int *wg;                  // strips > 1: {strip, begin, end} of every workgroup
    double xmin, ymin, dx, dy, rdx, rdy, Lx, Ly;
    double charge, cw, qm;
    double dt_half, dt;
    double *x1, *x2, *v1, *v2, *v3;
    const double *w;
    const double *e[3], *b[3];
    double *part;                   // [workgroups][3][hr][nx] current sums
    double *stray;                  // [3][nx * ny] currents of the listed particles; zero between steps
    int *list;                      // their indices (below 2^29), with the stage in the upper bits
    int *flags;                     // error bits, particles listed in this pass
};

// cell (ceil() - 1, not wrapped) and the degree-P and degree-(P-1) values
template <int P>
__device__ __forceinline__ bool f2_point(double pos, double lo, double d, double rd, int &cell,
                                         double (&b0)[P + 1], double (&b1)[P])
{
    const double xp = div_by(pos - lo, d, rd);
    const bool ok = fabs(xp) < 1.0e9;
    const double c = ok ? ceil(xp) : 1.0;
    bspline_pair_fast<P, P - 1>(ok ? xp - (c - 1.0) : 1.0, b0, b1);
    cell = (int)c - 1;
    return ok;
}

// suffix sums s[j] = sum_{i >= j} b[i], j = 1 .. P (s[0] = 1)
template <int P>
__device__ __forceinline__ void f2_suffix(const double (&b)[P + 1], double (&s)[P + 1])
{
    s[P] = b[P];
#pragma unroll
    for (int j = P - 1; j >= 1; --j) s[j] = s[j + 1] + b[j];
    s[0] = 1.0;
}

// Integrals d int N^{P-1} along a path that starts in a cell with suffix
// sums sa and ends in the cell + move (|move| <= 1) with sb, at the start
// cell's nodes 1 .. P (node k of cell c is c - P + k), and `extra` at node
// P + 1 (move = 1) or 0 (move = -1), from the antiderivative F (k_split2d):
// F is 1 below a cell's nodes, 0 above.
template <int P>
__device__ __forceinline__ void f2_path(const double (&sa)[P + 1], const double (&sb)[P + 1], int move, double d,
                                        double (&val)[P + 1], double &extra)
{
#pragma unroll
    for (int c = 1; c <= P; ++c) {
        const double up = sb[c - 1];                       // move = 1
        const double dn = c < P ? sb[c < P ? c + 1 : c] : 0.0;   // move = -1
        const double fe = move == 0 ? sb[c] : (move > 0 ? up : dn);
        val[c] = d * (fe - sa[c]);
    }
    val[0] = 0.0;
    extra = move == 0 ? 0.0 : (move > 0 ? d * sb[P] : d * (sb[1] - 1.0));
}

// The general form of a particle's sub-steps from `stage` on (0: all, 1: from
// Hp1, 2: from the second Hp2), on the grids in global memory: any cell, any
// path. Few particles come here.
template <int P, int MODE>
__device__ __forceinline__ int f2_general(const F2Args &a, int64_t i, int stage)
{
    const int nx = a.nx, ny = a.ny;
    int errs = 0;
    const int64_t nn = (int64_t)nx * ny;
    double x1 = a.x1[i], x2 = a.x2[i], v1 = a.v1[i], v2 = a.v2[i], v3 = a.v3[i];
    const double q = (a.w[i] * a.charge) * a.cw;
    int cx = 0, cy = 0;
    double bx0[P + 1], bx1[P], by0[P + 1], by1[P];
    auto shape = [&]() __attribute__((always_inline)) {
        bool ok = f2_point<P>(x1, a.xmin, a.dx, a.rdx, cx, bx0, bx1);
        ok = f2_point<P>(x2, a.ymin, a.dy, a.rdy, cy, by0, by1) && ok;
        return ok;
    };
    auto gather = [&](const double *f, int dgx, const double *bx, int dgy, const double *by) __attribute__((always_inline)) {
        double v = 0.0;
#pragma unroll
        for (int c = 0; c <= P; ++c) {
            if (c > dgy) break;
            const double *row = f + (int64_t)imod(cy - dgy + c, ny) * nx;
            double r = 0.0;
#pragma unroll
            for (int k = 0; k <= P; ++k)
                if (k <= dgx) r = __builtin_fma(row[imod(cx - dgx + k, nx)], bx[k], r);
            v = __builtin_fma(r, by[c], v);
        }
        return v;
    };
    auto hp3 = [&](double dt) __attribute__((always_inline)) {
        const double b1 = gather(a.b[0], P, bx0, P - 1, by1);
        const double b2 = gather(a.b[1], P - 1, bx1, P, by0);
        const double dv = (dt * a.qm) * v3;
        v1 = __builtin_fma(-dv, b2, v1);
        v2 = __builtin_fma(dv, b1, v2);
        const double wq = q * v3;
#pragma unroll
        for (int k = 0; k <= P; ++k)
#pragma unroll
            for (int c = 0; c <= P; ++c)
                unsafeAtomicAdd(&a.stray[2 * nn + imod(cx - P + k, nx) + (int64_t)imod(cy - P + c, ny) * nx],
                                (wq * bx0[k]) * by0[c]);
    };
    // Hp1 (along x) or Hp2: node by node of the path
    auto push = [&](bool along_x, double dt) __attribute__((always_inline)) {
        const double pos = along_x ? x1 : x2, vel = along_x ? v1 : v2;
        const double lo = along_x ? a.xmin : a.ymin, d = along_x ? a.dx : a.dy, rd = along_x ? a.rdx : a.rdy;
        const double pn = pos + dt * vel;
        double na[P + 1], nb[P];
        int ce = 0;
        const bool ok = f2_point<P>(pn, lo, d, rd, ce, na, nb);
        const int c0 = along_x ? cx : cy;
        const int64_t far = (int64_t)ce - c0;
        if (!ok || far > kMaxCross2 || far < -kMaxCross2) {
            errs |= E_FAR;
            return false;
        }
        double sa[P + 1], sb[P + 1];
        f2_suffix<P>(along_x ? bx0 : by0, sa);
        f2_suffix<P>(na, sb);
        auto F = [](const double (&sfx)[P + 1], int j) {
            double f = j <= 0 ? 1.0 : 0.0;
#pragma unroll
            for (int t = 1; t <= P; ++t) f = j == t ? sfx[t] : f;
            return f;
        };
        double s1 = 0.0, s3 = 0.0;
        const int clo = c0 < ce ? c0 : ce, chi = c0 < ce ? ce : c0;
        const double *fb = along_x ? a.b[1] : a.b[0];
        double *j = a.stray + (along_x ? 0 : nn);
        for (int node = clo - P + 1; node <= chi; ++node) {
            const double val = d * (F(sb, node - ce + P) - F(sa, node - c0 + P));
            const int na_ = imod(node, along_x ? nx : ny);
            double g = 0.0, g3 = 0.0;
#pragma unroll
            for (int c = 0; c <= P; ++c) {
                const int nc = along_x ? imod(cy - P + c, ny) : imod(cx - P + c, nx);
                const int64_t k = along_x ? na_ + (int64_t)nc * nx : nc + (int64_t)na_ * nx;
                const double wc = along_x ? by0[c] : bx0[c];
                g = __builtin_fma(fb[k], wc, g);
                if (c >= 1) g3 = __builtin_fma(a.b[2][k], along_x ? by1[c - 1] : bx1[c - 1], g3);
                unsafeAtomicAdd(&j[k], (q * val) * wc);
            }
            s1 = __builtin_fma(val, g, s1);
            s3 = __builtin_fma(val, g3, s3);
        }
        if (along_x) {
            v3 = __builtin_fma(a.qm, s1, v3);
            v2 = __builtin_fma(-a.qm, s3, v2);
            x1 = a.xmin + jl_mod(pn - a.xmin, a.Lx);
        } else {
            v3 = __builtin_fma(-a.qm, s1, v3);
            v1 = __builtin_fma(a.qm, s3, v1);
            x2 = a.ymin + jl_mod(pn - a.ymin, a.Ly);
        }
        return shape();
    };
    if (!shape()) {
        return E_INEXACT;
    }
    bool ok = true;
    if (stage == 0) {
        if (MODE & F2_HE) {
            const double dtqm = a.dt_half * a.qm;
            v1 = __builtin_fma(dtqm, gather(a.e[0], P - 1, bx1, P, by0), v1);
            v2 = __builtin_fma(dtqm, gather(a.e[1], P, bx0, P - 1, by1), v2);
            v3 = __builtin_fma(dtqm, gather(a.e[2], P, bx0, P, by0), v3);
        }
        if (MODE & F2_HP3A) hp3(a.dt_half);
        if (MODE & F2_HP2A) ok = push(false, a.dt_half);
    }
    if (ok && stage <= 1 && (MODE & F2_HP1)) ok = push(true, a.dt);
    if (ok && (MODE & F2_HP2B)) ok = push(false, a.dt_half);
    if (ok && (MODE & F2_HP3B)) hp3(a.dt_half);
    a.x1[i] = x1;
    a.x2[i] = x2;
    a.v1[i] = v1;
    a.v2[i] = v2;
    a.v3[i] = v3;
    return errs;
}

template <int P, int MODE>
__global__ void __launch_bounds__(f2_threads(P)) k_step2d(F2Args a)
{
    extern __shared__ __align__(16) double smem[];
    constexpr bool HE = (MODE & F2_HE) != 0, A = (MODE & F2_HP2A) != 0, HP1 = (MODE & F2_HP1) != 0;
    static_assert(HE == A && A == ((MODE & F2_HP3A) != 0) && HP1 == ((MODE & F2_HP2B) != 0) &&
                      HP1 == ((MODE & F2_HP3B) != 0),
                  "the first half, the second half, or both");
    constexpr int NE = HE ? 3 : 0, kThreads = f2_threads(P), kWaves = kThreads / kWave;
    const int nx = a.nx, ny = a.ny, S = a.s, HR = a.hr, fs = S * HR;
    const int lane = lane_id(), wave = threadIdx.x / kWave;
    double *sE = smem, *sB = smem + NE * fs, *sJ = sB + 3 * fs;

    // this workgroup's particles and rows: row r holds grid row jlo + r
    int64_t begin, end;
    int lo = 0, jlo = -P;
    if (a.strips == 1) {
        begin = (int64_t)blockIdx.x * a.chunk;
        end = begin + a.chunk < a.n ? begin + a.chunk : a.n;
    } else {
        lo = a.wg[3 * blockIdx.x] * a.h;
        begin = a.wg[3 * blockIdx.x + 1];
        end = a.wg[3 * blockIdx.x + 2];
        jlo = lo - a.m - P;
    }
    const int cols = nx + P + 1;
    for (int t = threadIdx.x; t < cols * HR; t += kThreads) {
        const int r = t / cols, c = t - r * cols;
        const int i = imod(c - P + nx, nx), j = imod(jlo + r + ny, ny);
        const int k = i + j * nx, o = r * S + c;
        double v[6];
#pragma unroll
        for (int f = 0; f < 3; ++f) {
            if (HE) v[f] = a.e[f][k];
            v[3 + f] = a.b[f][k];
        }
#pragma unroll
        for (int f = 0; f < 3; ++f) {
            if (HE) sE[f * fs + o] = v[f];
            sB[f * fs + o] = v[3 + f];
        }
    }
    for (int t = threadIdx.x; t < 3 * fs; t += kThreads) sJ[t] = 0.0;
    __syncthreads();
    const double *B1 = sB, *B2 = sB + fs, *B3 = sB + 2 * fs;
    double *J1 = sJ, *J2 = sJ + fs, *J3 = sJ + 2 * fs;

    // The wave's share, in whole waves of 64 particles: the first generation
    // of waves on a SIMD issues first, so its share is larger (as s2_args);
    // equal shares while they are a few rounds each.
    const int64_t len = end > begin ? (end - begin + kWave - 1) / kWave : 0;
    int64_t w0, w1;
    {
        auto bound = [&](int w) -> int64_t {
            if (len <= 4 * kWaves) return len * w / kWaves;
            constexpr int G = kWaves / 4;
            double sum = 0.0;
            for (int g = 0; g < G; ++g) {
                const int in = w - 4 * g < 0 ? 0 : (w - 4 * g > 4 ? 4 : w - 4 * g);
                sum += in * (1.0 + kS2GenSkew * (double)(G - 1 - 2 * g) / (double)(G - 1));
            }
            return w == kWaves ? len : (int64_t)((double)len * sum / kWaves);
        };
        w0 = bound(wave);
        w1 = bound(wave + 1);
    }

    // the LDS row of a cell's first node, cell in unwrapped grid rows; false
    // where the rows it reaches are not held
    auto row_of = [&](int cell, int &r) {
        if (a.strips == 1) {
            r = imod(cell, ny);
            return true;
        }
        r = imod(cell, ny) - lo;
        if (r < -a.m) r += ny;
        if (r >= ny - a.m) r -= ny;
        r += a.m;
        return r < a.h + 2 * a.m;
    };

    const double qm = a.qm, hdt = a.dt_half;
    int errs = 0;
    for (int64_t u = w0; u < w1; ++u) {
        const int64_t i = begin + u * kWave + lane;
        bool live = i < end;
        const int64_t ii = live ? i : end - 1;
        double x1 = a.x1[ii], x2 = a.x2[ii], v1 = a.v1[ii], v2 = a.v2[ii], v3 = a.v3[ii];
        const double q = (a.w[ii] * a.charge) * a.cw;
        int cx, cy, r = 0, stray = -1;        // stray: the stage to go on from, in the general form
        double bx0[P + 1], bx1[P], by0[P + 1], by1[P];
        bool ok = f2_point<P>(x1, a.xmin, a.dx, a.rdx, cx, bx0, bx1);
        ok = f2_point<P>(x2, a.ymin, a.dy, a.rdy, cy, by0, by1) && ok;
        if (live && !ok) {
            errs |= E_INEXACT;
            live = false;
        }
        if (live && !row_of(cy, r)) {
            stray = HE ? 0 : 1;
            live = false;
        }
        // Hp3's gather of B2 and Hp2's of B1 and B3 over rows: sums along x of
        // row k (0 .. P + 1) at a node offset o
        auto row_b1 = [&](int o, int k) {
            double g = 0.0;
#pragma unroll
            for (int c = 0; c <= P; ++c) g = __builtin_fma(B1[o + k * S + c], bx0[c], g);
            return g;
        };
        auto row_b3 = [&](int o, int k) {
            double g = 0.0;
#pragma unroll
            for (int c = 1; c <= P; ++c) g = __builtin_fma(B3[o + k * S + c], bx1[c - 1], g);
            return g;
        };
        auto b2_at = [&](int o) {
            double v = 0.0;
#pragma unroll
            for (int k = 0; k <= P; ++k) {
                double g = 0.0;
#pragma unroll
                for (int c = 1; c <= P; ++c) g = __builtin_fma(B2[o + k * S + c], bx1[c - 1], g);
                v = __builtin_fma(g, by0[k], v);
            }
            return v;
        };
        auto dep_j3 = [&](int o) {
            const double wq = q * v3;
#pragma unroll
            for (int k = 0; k <= P; ++k) {
                const double wk = wq * by0[k];
#pragma unroll
                for (int c = 0; c <= P; ++c) unsafeAtomicAdd(&J3[o + k * S + c], wk * bx0[c]);
            }
        };
        auto dep_j2_row = [&](int o, int k, double val) {
            const double qv = q * val;
#pragma unroll
            for (int c = 0; c <= P; ++c) unsafeAtomicAdd(&J2[o + k * S + c], qv * bx0[c]);
        };
        // the end of a push along x2 by dt: cell, values, suffix sums and the
        // move in cells; false where the general form has to take it
        double ey0[P + 1], ey1[P];
        int ce = 0, re = 0, move = 0;
        double pn = 0.0;
        auto end_y = [&](double dt) {
            pn = x2 + dt * v2;
            const bool fin = f2_point<P>(pn, a.ymin, a.dy, a.rdy, ce, ey0, ey1);
            move = ce - cy;
            return fin && move <= 1 && move >= -1 && row_of(ce, re);
        };
        auto take_y = [&] {
            x2 = a.ymin + jl_mod(pn - a.ymin, a.Ly);
            cy = imod(ce, ny);          // as of the position after the mod
            r = re;
#pragma unroll
            for (int k = 0; k <= P; ++k) by0[k] = ey0[k];
#pragma unroll
            for (int k = 0; k < P; ++k) by1[k] = ey1[k];
        };

        if constexpr (A) {
            if (live) {
                const int o = r * S + imod(cx, nx);
                if constexpr (HE) {
                    const double *E1 = sE + o, *E2 = sE + fs + o, *E3 = sE + 2 * fs + o;
                    double e1 = 0.0, e2 = 0.0, e3 = 0.0;
#pragma unroll
                    for (int k = 0; k <= P; ++k) {
                        double g1 = 0.0, g2 = 0.0, g3 = 0.0;
#pragma unroll
                        for (int c = 0; c <= P; ++c) {
                            if (c >= 1) g1 = __builtin_fma(E1[k * S + c], bx1[c >= 1 ? c - 1 : 0], g1);
                            if (k >= 1) g2 = __builtin_fma(E2[k * S + c], bx0[c], g2);
                            g3 = __builtin_fma(E3[k * S + c], bx0[c], g3);
                        }
                        e1 = __builtin_fma(g1, by0[k], e1);
                        if (k >= 1) e2 = __builtin_fma(g2, by1[k >= 1 ? k - 1 : 0], e2);
                        e3 = __builtin_fma(g3, by0[k], e3);
                    }
                    const double dtqm = hdt * qm;
                    v1 = __builtin_fma(dtqm, e1, v1);
                    v2 = __builtin_fma(dtqm, e2, v2);
                    v3 = __builtin_fma(dtqm, e3, v3);
                }
                // Hp3
                double g1[P + 1], b1 = 0.0;
#pragma unroll
                for (int k = 1; k <= P; ++k) {
                    g1[k] = row_b1(o, k);
                    b1 = __builtin_fma(g1[k], by1[k - 1], b1);
                }
                const double b2 = b2_at(o), dv = (hdt * qm) * v3;
                v1 = __builtin_fma(-dv, b2, v1);
                v2 = __builtin_fma(dv, b1, v2);
                if (!end_y(hdt)) {
                    stray = 0;          // nothing deposited or stored yet
                    live = false;
                } else {
                    dep_j3(o);
                    // Hp2
                    double sa[P + 1], sb[P + 1], val[P + 1], vx;
                    f2_suffix<P>(by0, sa);
                    f2_suffix<P>(ey0, sb);
                    f2_path<P>(sa, sb, move, a.dy, val, vx);
                    double s1 = 0.0, s3 = 0.0;
#pragma unroll
                    for (int k = 1; k <= P; ++k) {
                        s1 = __builtin_fma(val[k], g1[k], s1);
                        s3 = __builtin_fma(val[k], row_b3(o, k), s3);
                        dep_j2_row(o, k, val[k]);
                    }
                    if (move != 0) {
                        const int k = move > 0 ? P + 1 : 0;
                        s1 = __builtin_fma(vx, row_b1(o, k), s1);
                        s3 = __builtin_fma(vx, row_b3(o, k), s3);
                        dep_j2_row(o, k, vx);
                    }
                    v3 = __builtin_fma(-qm, s1, v3);
                    v1 = __builtin_fma(qm, s3, v1);
                    take_y();
                }
            }
        }
        if constexpr (HP1) {
            if (live) {
                const double xn = x1 + a.dt * v1;
                double ex0[P + 1], ex1[P];
                int cex = 0;
                const bool fin = f2_point<P>(xn, a.xmin, a.dx, a.rdx, cex, ex0, ex1);
                const int mx = cex - cx;
                if (!fin || mx > 1 || mx < -1) {
                    stray = 1;
                    live = false;
                } else {
                    const int o = r * S + imod(cx, nx);
                    double sa[P + 1], sb[P + 1], val[P + 1], vx;
                    f2_suffix<P>(bx0, sa);
                    f2_suffix<P>(ex0, sb);
                    f2_path<P>(sa, sb, mx, a.dx, val, vx);
                    double s2 = 0.0, s3 = 0.0;
#pragma unroll
                    for (int k = 0; k <= P; ++k) {
                        double g2 = 0.0, g3 = 0.0;
                        const double wk = q * by0[k];
#pragma unroll
                        for (int c = 1; c <= P; ++c) {
                            g2 = __builtin_fma(B2[o + k * S + c], val[c], g2);
                            if (k >= 1) g3 = __builtin_fma(B3[o + k * S + c], val[c], g3);
                            unsafeAtomicAdd(&J1[o + k * S + c], wk * val[c]);
                        }
                        s2 = __builtin_fma(g2, by0[k], s2);
                        if (k >= 1) s3 = __builtin_fma(g3, by1[k >= 1 ? k - 1 : 0], s3);
                    }
                    if (mx != 0) {
                        const int c = mx > 0 ? P + 1 : 0;
                        double g2 = 0.0, g3 = 0.0;
                        const double qv = q * vx;
#pragma unroll
                        for (int k = 0; k <= P; ++k) {
                            g2 = __builtin_fma(B2[o + k * S + c], by0[k], g2);
                            if (k >= 1) g3 = __builtin_fma(B3[o + k * S + c], by1[k >= 1 ? k - 1 : 0], g3);
                            unsafeAtomicAdd(&J1[o + k * S + c], qv * by0[k]);
                        }
                        s2 = __builtin_fma(vx, g2, s2);
                        s3 = __builtin_fma(vx, g3, s3);
                    }
                    v3 = __builtin_fma(qm, s2, v3);
                    v2 = __builtin_fma(-qm, s3, v2);
                    x1 = a.xmin + jl_mod(xn - a.xmin, a.Lx);
                    cx = cex;
#pragma unroll
                    for (int k = 0; k <= P; ++k) bx0[k] = ex0[k];
#pragma unroll
                    for (int k = 0; k < P; ++k) bx1[k] = ex1[k];
                    if (!end_y(hdt)) {
                        stray = 2;
                        live = false;
                    }
                }
                if (stray > 0) {        // go on from this state
                    a.x1[i] = x1;
                    a.x2[i] = x2;
                    a.v1[i] = v1;
                    a.v2[i] = v2;
                    a.v3[i] = v3;
                }
            }
            if (live) {
                // Hp2
                const int xc = imod(cx, nx), o = r * S + xc;
                double g1[P + 2];
                g1[0] = 0.0;
                g1[P + 1] = 0.0;
#pragma unroll
                for (int k = 1; k <= P; ++k) g1[k] = row_b1(o, k);
                double sa[P + 1], sb[P + 1], val[P + 1], vx;
                f2_suffix<P>(by0, sa);
                f2_suffix<P>(ey0, sb);
                f2_path<P>(sa, sb, move, a.dy, val, vx);
                double s1 = 0.0, s3 = 0.0;
#pragma unroll
                for (int k = 1; k <= P; ++k) {
                    s1 = __builtin_fma(val[k], g1[k], s1);
                    s3 = __builtin_fma(val[k], row_b3(o, k), s3);
                    dep_j2_row(o, k, val[k]);
                }
                if (move != 0) {
                    const int k = move > 0 ? P + 1 : 0;
                    const double g = row_b1(o, k);
                    if (move > 0) g1[P + 1] = g;
                    else g1[0] = g;
                    s1 = __builtin_fma(vx, g, s1);
                    s3 = __builtin_fma(vx, row_b3(o, k), s3);
                    dep_j2_row(o, k, vx);
                }
                v3 = __builtin_fma(-qm, s1, v3);
                v1 = __builtin_fma(qm, s3, v1);
                const int mv = move;
                take_y();
                // Hp3 at the end of the path: its rows of B1 are among those read
                double b1 = 0.0;
#pragma unroll
                for (int k = 1; k <= P; ++k)
                    b1 = __builtin_fma(mv == 0 ? g1[k] : (mv > 0 ? g1[k + 1] : g1[k - 1]), by1[k - 1], b1);
                const int oe = r * S + xc;
                const double b2 = b2_at(oe), dv = (hdt * qm) * v3;
                v1 = __builtin_fma(-dv, b2, v1);
                v2 = __builtin_fma(dv, b1, v2);
                dep_j3(oe);
            }
        }
        if (live) {
            if (HP1) a.x1[i] = x1;
            a.x2[i] = x2;
            a.v1[i] = v1;
            a.v2[i] = v2;
            a.v3[i] = v3;
        }
        const unsigned long long ms = __ballot(stray >= 0);
        if (ms) {
            const unsigned long long below = lane == 0 ? 0ull : (~0ull >> (kWave - lane));
            int at = 0;
            if (lane == 0) at = atomicAdd(&a.flags[1], __popcll(ms));
            at = __builtin_amdgcn_readfirstlane(at);
            if (stray >= 0) a.list[at + __popcll(ms & below)] = (int)i | (stray << 29);
        }
    }
    if (errs) atomicOr(a.flags, errs);
    __syncthreads();
    // columns folded onto the grid's (c = i + P for node i in [-P, nx])
    double *out = a.part + (size_t)blockIdx.x * 3 * HR * nx;
    for (int t = threadIdx.x; t < 3 * HR * nx; t += kThreads) {
        const int row = t / nx, i = t - row * nx;          // row: component and row
        const double *j = sJ + (row / HR) * fs + (row % HR) * S;
        double v = j[i + P];
        if (i >= nx - P) v += j[i + P - nx];
        if (i == 0) v += j[nx + P];
        out[t] = v;
    }
}

// After the pass. blockIdx.z = 0: the listed particles. z = 1 .. 3, component
// z - 1: part2[split][component][node] = sum over the split's workgroups, in
// order, of the rows they hold of the node's row. The two are independent (the
// listed particles' currents go to a.stray, which the next kernel adds), and
// the listed ones take the longer for all that they are few: one particle's
// gathers and pushes wait on memory one after another. In two launches, then in
// this one (us a step): 48 x 36, 150,000 particles 66.5, 64.5; 64 x 64,
// 2,000,000 particles 266, 256; 16,777,216 1639, 1622.
template <int P, int MODE>
__global__ void __launch_bounds__(256) k_f2_rest(F2Args a, int nblocks, double *part2)
{
    const int nn = a.nx * a.ny, splits = gridDim.y, sp = blockIdx.y;
    const int k = blockIdx.x * blockDim.x + threadIdx.x;
    if (blockIdx.z == 0) {
        const int n = a.flags[1], threads = gridDim.x * splits * blockDim.x;
        int errs = 0;
        for (int t = sp * gridDim.x * blockDim.x + k; t < n; t += threads) {
            const int it = a.list[t];
            errs |= f2_general<P, MODE>(a, it & 0x1fffffff, it >> 29);
        }
        if (errs) atomicOr(a.flags, errs);
        return;
    }
    if (k >= nn) return;
    const int c = blockIdx.z - 1, gy = k / a.nx, gx = k - gy * a.nx;
    const int b0 = (int)((int64_t)sp * nblocks / splits), b1 = (int)((int64_t)(sp + 1) * nblocks / splits);
    double t = 0.0;
    const size_t bs = (size_t)3 * a.hr * a.nx;
    if (a.strips == 1) {
        const double *q = a.part + ((size_t)c * a.hr + gy + P) * a.nx + gx;     // rows -P .. ny
        const int alias = gy >= a.ny - P ? -a.ny : (gy == 0 ? a.ny : 0);
#pragma unroll 8
        for (int b = b0; b < b1; ++b) {
            double v = q[b * bs];
            if (alias) v += q[b * bs + (ptrdiff_t)alias * a.nx];
            t += v;
        }
    } else {
        for (int b = b0; b < b1; ++b) {
            const int jlo = a.wg[3 * b] * a.h - a.m - P;
            for (int r = imod(gy - jlo, a.ny); r < a.hr; r += a.ny)
                t += a.part[b * bs + ((size_t)c * a.hr + r) * a.nx + gx];
        }
    }
    part2[((size_t)sp * 3 + c) * nn + k] = t;
}

// ---- how many particles a step would list ----
//
// Whether the one-pass step or the operators' passes are the faster way is
// decided ahead, from the particles as they are: a step that lists them all
// takes 45 times as long as the operators' passes (16,777,216 particles), so to
// try it and count is no way to find out. Each workgroup's out[blockIdx.x] is its
// part of sum over particles of how many of the next `steps` steps list
// it, with the present velocity: all of them where a push crosses more than one
// cell; with strips, binned now, those that begin after it has left the rows
// held. Groups of 64 neighbouring particles, every stride-th, stand for all: of
// 262,144 particles, 1 % to be listed are found to 4 % of that. Latency: 5 to 8 us
// (a million particles: 16), against the 2000 and more of the steps up to the next.
constexpr int kPredictBlocks = 256;
constexpr int64_t kPredictSample = (int64_t)1 << 18;

__global__ void __launch_bounds__(1024) k_f2_predict(F2Args a, int64_t groups, int64_t stride, int steps, int *out)
{
    __shared__ int part[1024 / kWave];
    const int lane = lane_id(), wave = threadIdx.x / kWave;
    int sum = 0;
    for (int64_t g = (int64_t)blockIdx.x * (1024 / kWave) + wave; g < groups; g += (int64_t)gridDim.x * (1024 / kWave)) {
        const int64_t i = g * stride * kWave + lane;
        if (i >= a.n) break;
        const double v2 = a.v2[i];
        const double xp = div_by(a.x1[i] - a.xmin, a.dx, a.rdx), yp = div_by(a.x2[i] - a.ymin, a.dy, a.rdy);
        const double mx = a.dt * a.v1[i] * a.rdx, my = a.dt * v2 * a.rdy;       // cells a step
        if (!(fabs(xp) < 1.0e9 && fabs(yp) < 1.0e9)) continue;                  // an error of the pass's
        if (!(fabs(ceil(xp + mx) - ceil(xp)) <= 1.0 && fabs(ceil(yp + 0.5 * my) - ceil(yp)) <= 1.0)) {
            sum += steps;
        } else if (a.strips > 1) {
            const double c = ceil(yp);
            const int r = imod((int)c - 1, a.ny) % a.h;
            const double lo = c - (double)(r + a.m), hi = c + (double)(a.h - 1 - r + a.m);      // ceil() of the rows held
            for (int k = 1; k <= steps; ++k) {
                const double e = ceil(yp + (double)k * my);
                sum += e < lo || e > hi;
            }
        }
    }
#pragma unroll
    for (int o = kWave / 2; o > 0; o >>= 1) sum += __shfl_xor(sum, o, kWave);
    if (lane == 0) part[wave] = sum;
    __syncthreads();
    if (threadIdx.x == 0) {
        int t = 0;
        for (int w = 0; w < 1024 / kWave; ++w) t += part[w];
        __hip_atomic_store(&out[blockIdx.x], t, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
    }
}

// ---- binning by strip ----
constexpr int kBinTile = 8192;                  // particles of a binning workgroup

__device__ __forceinline__ int strip_of(const F2Args &a, double x2)
{
    const double yp = div_by(x2 - a.ymin, a.dy, a.rdy);
    return fabs(yp) < 1.0e9 ? imod((int)ceil(yp) - 1, a.ny) / a.h : 0;
}

// counts[strip][tile]
__global__ void __launch_bounds__(1024) k_bin_count(F2Args a, int ntiles, int *counts)
{
    __shared__ int h[kF2StripsMax];
    if (threadIdx.x < kF2StripsMax) h[threadIdx.x] = 0;
    __syncthreads();
    const int64_t t0 = (int64_t)blockIdx.x * kBinTile;
    int mine[kBinTile / 1024];
#pragma unroll
    for (int u = 0; u < kBinTile / 1024; ++u) {
        const int64_t i = t0 + u * 1024 + threadIdx.x;
        mine[u] = i < a.n ? strip_of(a, a.x2[i]) : -1;
    }
#pragma unroll
    for (int u = 0; u < kBinTile / 1024; ++u)
        if (mine[u] >= 0) atomicAdd(&h[mine[u]], 1);
    __syncthreads();
    if ((int)threadIdx.x < a.strips) counts[(size_t)threadIdx.x * ntiles + blockIdx.x] = h[threadIdx.x];
}

// One workgroup: counts -> first positions (strip after strip, tile after
// tile), and the particle workgroups' ranges: a strip of c particles takes
// ceil(c / chunk) of them, chunk = ceil(n / (nblocks - strips)), so that all
// strips' fit; the rest are empty.
__global__ void __launch_bounds__(1024) k_bin_scan(F2Args a, int ntiles, int *counts, int nblocks, int64_t chunk,
                                                   int *wg)
{
    __shared__ int part[1024];
    __shared__ int first[kF2StripsMax + 1];
    const int t = threadIdx.x;
    const int64_t total = (int64_t)a.strips * ntiles;
    const int64_t per = (total + 1023) / 1024;
    const int64_t k0 = t * per < total ? t * per : total, k1 = k0 + per < total ? k0 + per : total;
    int s = 0;
    for (int64_t k = k0; k < k1; ++k) s += counts[k];
    part[t] = s;
    __syncthreads();
    for (int off = 1; off < 1024; off <<= 1) {
        const int v = t >= off ? part[t - off] : 0;
        __syncthreads();
        part[t] += v;
        __syncthreads();
    }
    int base = part[t] - s;
    for (int64_t k = k0; k < k1; ++k) {
        if (k % ntiles == 0) first[k / ntiles] = base;
        const int c = counts[k];
        counts[k] = base;
        base += c;
    }
    if (t == 0) first[a.strips] = (int)a.n;
    __syncthreads();
    if (t == 0) {
        int b = 0;
        for (int sp = 0; sp < a.strips; ++sp)
            for (int64_t p0 = first[sp]; p0 < first[sp + 1] && b < nblocks; p0 += chunk, ++b) {
                wg[3 * b] = sp;
                wg[3 * b + 1] = (int)p0;
                wg[3 * b + 2] = (int)(p0 + chunk < first[sp + 1] ? p0 + chunk : first[sp + 1]);
            }
        for (; b < nblocks; ++b) {
            wg[3 * b] = 0;
            wg[3 * b + 1] = 0;
            wg[3 * b + 2] = 0;
        }
    }
}

// the lanes of a strip take consecutive places from one LDS atomic
__global__ void __launch_bounds__(1024) k_bin_scatter(F2Args a, int ntiles, const int *counts, S2Perm pm)
{
    __shared__ int cur[kF2StripsMax];
    if ((int)threadIdx.x < a.strips) cur[threadIdx.x] = counts[(size_t)threadIdx.x * ntiles + blockIdx.x];
    __syncthreads();
    const int lane = lane_id();
    const unsigned long long below = lane == 0 ? 0ull : (~0ull >> (kWave - lane));
    const int64_t t0 = (int64_t)blockIdx.x * kBinTile;
    for (int u = 0; u < kBinTile / 1024; ++u) {
        const int64_t i = t0 + u * 1024 + threadIdx.x;
        if (i >= a.n) break;
        double v[6];
#pragma unroll
        for (int r = 0; r < 6; ++r) v[r] = pm.src[r][i];
        const int64_t id = pm.id[i];
        const int key = strip_of(a, v[1]);
        unsigned long long same = __ballot(true);
#pragma unroll
        for (int b = 0; b < 6; ++b) {
            const bool bit = (key >> b) & 1;
            const unsigned long long set = __ballot(bit);
            same &= bit ? set : ~set;
        }
        const int leader = __ffsll((long long)same) - 1;
        int base = 0;
        if (lane == leader) base = atomicAdd(&cur[key], __popcll(same));
        base = __shfl(base, leader, kWave);
        const int64_t d = (int64_t)base + __popcll(same & below);
#pragma unroll
        for (int r = 0; r < 6; ++r) pm.dst[r][d] = v[r];
        pm.id_dst[d] = id;
    }
}
