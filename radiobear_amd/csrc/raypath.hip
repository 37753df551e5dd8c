// Ray geometry in FP64: a ray's steps split over 32 lanes, or one thread per ray.
//
// Follows raypath.compute_ds / findEdge (raypath.py:60-273) and the ellipse
// branch of Shape (shape.py:223-298) step for step.  The reference converts
// latitude / longitude to degrees and back and rebuilds sines through
// arcsin/arccos; here the same quantities come from the vector components
// (sin lat = y/|v|, cos lat = sqrt(x^2+z^2)/|v|, cos lng = z/sqrt(x^2+z^2), ...),
// which is the same arithmetic up to rounding, with no transcendental calls in
// the loop, and a path after its one refraction is followed as a straight line.  Quirks kept: the latitude-0 substitution lat = 1e-6 rad
// (shape.py:231-233), the next-shell radius taken at the current point's
// latitude (raypath.py:182), refraction only at the first boundary
// (raypath.py:158, 257), the numpy arange trial grid and linear root of
// findEdge (raypath.py:64, 94-97), the ds < 0 truncation (raypath.py:212-216),
// NaN (not an exception) when a ray misses the next shell (raypath.py:190-209),
// and the loop end when layer + 1 runs past the last layer (raypath.py:255-264).
#include "common.hpp"

namespace rbx {

struct V3 {
    double x, y, z;
};
__device__ inline V3 operator+(V3 a, V3 b) { return {a.x + b.x, a.y + b.y, a.z + b.z}; }
__device__ inline V3 operator*(double s, V3 a) { return {s * a.x, s * a.y, s * a.z}; }
__device__ inline double dot(V3 a, V3 b) { return a.x * b.x + a.y * b.y + a.z * b.z; }
__device__ inline double norm(V3 a) { return sqrt(dot(a, a)); }

struct Geo {
    double ratio;   // Rpol/Req for 'ellipse', 1 for 'sphere'
    double M[9];    // rotate2planet = rotX(rotate) * rotZ(tip), row-major
};

__device__ inline V3 mat(const double *M, V3 v) {
    return {M[0] * v.x + M[1] * v.y + M[2] * v.z, M[3] * v.x + M[4] * v.y + M[5] * v.z,
            M[6] * v.x + M[7] * v.y + M[8] * v.z};
}

// sines/cosines of (planetocentric latitude, delta longitude) of vector v
struct LatLng {
    double slat, clat, slng, clng;
};

__device__ inline LatLng latlng(V3 v) {
    LatLng o;
    const double r = norm(v);
    const double h = sqrt(v.x * v.x + v.z * v.z);
    if (v.y == 0.0) {                 // lat == 0 -> 1e-6 rad (shape.py:231-233)
        o.slat = 9.999999999998333e-07;   // sin(1e-6)
        o.clat = 0.9999999999995;         // cos(1e-6)
    } else {
        o.slat = v.y / r;
        o.clat = h / r;
    }
    if (h > 0.0) {
        o.slng = v.x / h;
        o.clng = v.z / h;
    } else {                           // atan2(0, 0) = 0
        o.slng = 0.0;
        o.clng = 1.0;
    }
    return o;
}

// Shape._calcEllipse for equatorial radius a at (lat, lng): |r|, r and normal n
struct Surf {
    double rmag;
    V3 r, n;
};

__device__ inline Surf ellipse(const Geo &G, double a, const LatLng &q) {
    const double b = G.ratio * a;
    V3 nn = {0.0, a * q.slat, b * q.clat};
    const double inv = 1.0 / sqrt(nn.y * nn.y + nn.z * nn.z);
    nn.y *= inv;
    nn.z *= inv;
    Surf s;
    s.n = {q.slng * nn.z, nn.y, q.clng * nn.z};                      // rotY(lng, norm)
    const double rc = a * q.clat;
    s.r = {q.slng * rc, b * q.slat, q.clng * rc};                    // rotY(lng, r_vec)
    s.rmag = norm(s.r);
    return s;
}

// sqrt of a finite x >= 0 (NaN below 0, as sqrt): the hardware reciprocal square root refined
// by one coupled Newton step and one correction of the root, without the range scaling of the
// library's (arguments here are squared km, far from FP64's limits): about an ulp in 8
// dependent operations.
__device__ inline double sqrt_km2(double x) {
    const double y = __builtin_amdgcn_rsq(x);
    double g = x * y, h = 0.5 * y;
    const double e = fma(-h, g, 0.5);
    g = fma(g, e, g);
    h = fma(h, e, h);
    g = fma(fma(-g, g, x), h, g);
    return __builtin_amdgcn_class(x, 0x260) ? x : g;   // +-0 and +inf are their own roots
}

// 1 / x for a positive finite x: the hardware estimate refined twice
__device__ inline double rcp_pos(double x) {
    double r = __builtin_amdgcn_rcp(x);
    r = fma(r, fma(-x, r, 1.0), r);
    return fma(r, fma(-x, r, 1.0), r);
}

// f^2 of the shells at a point: a shell of equatorial radius a has radius a f at the point's
// latitude, f^2 = (X + ratio^2 Y) / (X + Y) = 1 - (1 - ratio^2) y^2 / |v|^2 with X = x^2 + z^2 and
// Y = y^2 (ellipse() with sin lat = y / |v|, cos lat = sqrt(X) / |v|).  y == 0 takes the
// reference's 1e-6 rad latitude (kLat0 = sin^2 of it).
constexpr double kLat0 = 9.999999999998333e-07 * 9.999999999998333e-07;
__device__ inline double shell_f2(double flat, double y, double q) {
    const double s2 = y == 0.0 ? kLat0 : y * y * rcp_pos(q);
    return fma(-flat, s2, 1.0);
}

// The direction after incidence past 90 degrees at r: the reference's arcsin(sin t_inc) folds the
// angle, which turns the direction by 2 cos n (n along (ratio x, y, ratio z)).
__device__ inline V3 reflected(const Geo &G, V3 r, V3 s) {
    V3 n = {G.ratio * r.x, r.y, G.ratio * r.z};
    n = (1.0 / norm(n)) * n;
    const double c = -dot(s, n), st = sqrt(1.0 - c * c);
    return s + (c - sqrt(1.0 - st * st)) * n;
}

constexpr int kRayThreads = 256;
constexpr int kWin = 8;   // shell radii fetched per window

struct RayArgs {
    Geo G;
    const double *R, *N;
    int nl;
    const double *b;
    int nray;
    int units;   // 0 km, 1 half step in cm
    double *ds;
    int ld;
    int *nsteps;
    int limb;
    // several atmospheres laid end to end (null: one atmosphere of nl layers):
    // ray r uses layers [layer_off[a], layer_off[a + 1]) with a = ray_atm[r]
    const int *ray_atm, *layer_off;
    int natm;
};

// A path from point r along s (any |s|^2 = 1) over the shells from `step` on, step by step: the
// path is the straight line r + t s, so a step is a chain in t alone: the point's y and |r|^2
// (for f^2 at its latitude), r.s, the root of the next shell.  The next shell's radius is taken
// at the current point's latitude (raypath.py:182), hence disc = (r.s)^2 - f^2 (R_k^2 - R_{k+1}^2).
// f2: f^2 for the first of the steps.  Returns the step count; `write`: this lane writes the steps.
// One step's chain is 0.17 us (it was 0.48 us carrying the point, two angles and four roots).
// SEC: limb 'sec' (raypath.py:218-219)
template <bool SEC>
__device__ inline int serial_steps(const RayArgs &A, const double *Rl, int nl, double *out, double flat, double unit,
                                   double mu, V3 r, V3 s, double f2, int step, bool write) {
    const Geo &G = A.G;
    double t = 0.0, y1 = r.y, q1 = dot(r, r), d1 = dot(r, s);
    int count = step;
    // Equatorial radii by windows of kWin steps, the next window's loads issued a window ahead: a
    // step is shorter than a load, and fetched one step ahead each step waited for one (1000
    // layers x 4 rays 256 us against 166 us).
    // A lane whose path has ended computes on (nothing it writes): the window has no exits.
    double win[kWin + 1], nxt[kWin];
#pragma unroll
    for (int u = 0; u <= kWin; ++u) win[u] = Rl[min(step + u, nl - 1)];
    bool alive = true;
    for (int k0 = step; alive; k0 += kWin) {
#pragma unroll
        for (int u = 0; u < kWin; ++u) nxt[u] = Rl[min(k0 + kWin + 1 + u, nl - 1)];
#pragma unroll
        for (int u = 0; u < kWin; ++u) {
            const double R0 = win[u], R1 = win[u + 1];
            const double rdots = d1 + t;
            const double disc = fma(rdots, rdots, -f2 * ((R0 - R1) * (R0 + R1)));
            double ds = -rdots - sqrt_km2(disc);         // NaN when the shell is missed
            // the path ends below a shell (raypath.py:212-216) or at the last one (the
            // IndexError on nr[layer + 1])
            alive = alive && !(ds < 0.0) && k0 + u < nl - 1;
            if constexpr (SEC) ds = fabs(R1 - R0) * sqrt(f2) / mu;
            if (alive && write) out[k0 + u] = ds * unit;
            count += alive ? 1 : 0;
            t += ds;
            const double y = fma(t, s.y, y1);
            f2 = shell_f2(flat, y, fma(t, fma(2.0, d1, t), q1));
            // incidence past 90 degrees, cos(t_inc) = -s.n < 0 with n along (ratio x, y, ratio z)
            const double ys = y * s.y, along = fma(G.ratio, (d1 + t) - ys, ys);
            if (__builtin_expect(alive && along > 0.0, 0)) {
                r = r + t * s;
                s = reflected(G, r, s);
                t = 0.0;
                y1 = r.y;
                q1 = dot(r, r);
                d1 = dot(r, s);
            }
        }
        win[0] = win[kWin];
#pragma unroll
        for (int u = 0; u < kWin; ++u) win[u + 1] = nxt[u];
    }
    return count;
}

// The same path by L lanes, each a run of consecutive steps.  With u_k = |r_k|^2 - |r_0|^2 a step
// is u_{k+1} = u_k - f^2(u_k) (R_k^2 - R_{k+1}^2), -r_k.s = S_k = sqrt((r_0.s)^2 + u_k) on the way
// in, and ds_k = (u_k - u_{k+1}) / (S_k + S_{k+1}).  f^2 changes slowly along a path, so lane c
// starts from a guess of its first u, walks its run, and tracks d(its last u)/d(its first u): the
// runs' affine maps composed over the lanes (a scan) give every lane a better first u.  The walk is
// repeated until no first u moves; each pass makes at least one more run exact, so L + 1 always
// suffice, and away from the limb 2 or 3 do.  Where a shell is missed, S and ds are NaN from there
// on, as in the serial steps.  Returns the step count, or -1 - k when the path meets incidence past
// 90 degrees at step k (reached with S in S_at): the caller goes on from there step by step.
template <int L>
__device__ inline int parallel_steps(const RayArgs &A, const double *Rl, int nl, double *out, double flat,
                                     double unit, V3 r, V3 s, double f2_first, int c, double (*stage)[kWin],
                                     double &S_at) {
    constexpr int W = kWin;
    const double ratio = A.G.ratio, sy = s.y, y1 = r.y, q1 = dot(r, r), d1 = dot(r, s), d1sq = d1 * d1;
    const int n = nl - 1, len = (n + L - 1) / L;
    const int kb = min(n, c * len), ke = min(n, kb + len);
    const int lane0 = (threadIdx.x % 64) / L * L;
    const unsigned long long group = (L == 64 ? ~0ull : ((1ull << (L % 64)) - 1ull)) << lane0;
    double u0 = 0.0;
    if (c > 0) {   // du/dB = -f^2(u) to second order in B = R_0^2 - R_k^2, the first step's own f^2 apart
        const double Ra = Rl[0], Rb = Rl[kb], R1 = Rl[1];
        const double B = (Ra - Rb) * (Ra + Rb), f = shell_f2(flat, y1, q1);
        const double g = flat * (y1 / q1) * (y1 / q1 - sy / d1);
        u0 = fma(-f, B, 0.5 * f * g * B * B) - (f2_first - f) * ((Ra - R1) * (Ra + R1));
    }
    int neg = n, refl = n;   // first step with ds < 0, first point past 90 degrees
    for (int pass = 0; pass <= L + 1; ++pass) {
        double u = u0, S = sqrt_km2(d1sq + u0), D = 1.0;
        double S_r = 0.0;
        neg = refl = n;
        double win[W + 1], nxt[W];
#pragma unroll
        for (int i = 0; i <= W; ++i) win[i] = Rl[min(kb + i, n)];
        for (int off = 0; off < len; off += W) {   // (the same trips for the ray's lanes)
            const int k0 = kb + off;
#pragma unroll
            for (int i = 0; i < W; ++i) nxt[i] = Rl[min(k0 + W + 1 + i, n)];
#pragma unroll
            for (int i = 0; i < W; ++i) {
                const int k = k0 + i;
                if (k < ke) {
                    const double y = fma(-(S + d1), sy, y1), q = q1 + u, ys = y * sy;
                    const double iq = rcp_pos(q);
                    const double f2 = k == 0 ? f2_first : fma(-flat, y == 0.0 ? kLat0 : y * y * iq, 1.0);
                    if (k > 0 && refl == n && fma(ratio, -S - ys, ys) > 0.0) {
                        refl = k;
                        S_r = S;
                    }
                    const double dR = (win[i] - win[i + 1]) * (win[i] + win[i + 1]);
                    const double v = f2 * dR, un = u - v, Sn = sqrt_km2(d1sq + un);
                    const double ds = v * rcp_pos(S + Sn);
                    if (neg == n && v < 0.0 && S >= 0.0) neg = k;   // ds < 0, also where un is infinite
                    stage[c][i] = ds * unit;
                    // 1 - d f^2/du dR (a derivative: the estimate of 1 / S will do)
                    D *= fma(-flat * dR * iq, fma(ys, __builtin_amdgcn_rcp(S), y * y * iq), 1.0);
                    u = un;
                    S = Sn;
                }
            }
            win[0] = win[W];
#pragma unroll
            for (int i = 0; i < W; ++i) win[i + 1] = nxt[i];
            // the window's steps leave through LDS: L consecutive lanes write whole pieces of the
            // lanes' runs (each lane writing its own step touches one line per lane and store).  The
            // first pass, a guess, writes nothing.
            if (pass > 0) {
                wave_sync();
#pragma unroll
                for (int j = 0; j < W; ++j) {
                    const int e = j * L + c, o = e / W, k = o * len + off + e % W;
                    if (off + e % W < len && k < n) out[k] = stage[o][e % W];
                }
                wave_sync();
            }
        }
        // how far lane c's first u moves: the end of the run before it against it, plus what the
        // moves of earlier runs do to that end (a difference, so that settled runs leave no noise)
        const bool bad = __builtin_isnan(u0);
        double e = __shfl_up(u, 1, L) - (bad ? 0.0 : u0), Dp = __shfl_up(D, 1, L);
        if (c == 0) e = Dp = 0.0;
#pragma unroll
        for (int m = 1; m < L; m <<= 1) {
            const double em = __shfl_up(e, m, L), Dm = __shfl_up(Dp, m, L);
            if (c >= m) {
                e = fma(Dp, em, e);
                Dp *= Dm;
            }
        }
        const double next = (bad ? 0.0 : u0) + e, w = d1sq + next;
        const bool missed = !(w >= 0.0) && !(d1sq + u0 >= 0.0);   // NaN steps before and after
        const bool settled = c == 0 || kb >= ke || missed ||
                             (!bad && fabs(e) <= 1.0e-13 * fabs(w) + 1.0e-15 * fabs(next));
        S_at = S_r;
        if (pass > 0 && (__builtin_amdgcn_ballot_w64(!settled) & group) == 0ull) break;
        if (c > 0) u0 = next;
    }
    int first = refl, at = neg;
#pragma unroll
    for (int m = 1; m < L; m <<= 1) {
        first = min(first, __shfl_xor(first, m, L));
        at = min(at, __shfl_xor(at, m, L));
    }
    if (first < at) {
        S_at = __shfl(S_at, first / len, L);
        return -1 - first;
    }
    return at;
}

// L lanes per ray (1: a thread walks its ray's steps).
template <bool SEC, int L>
__global__ __launch_bounds__(kRayThreads) void raypath_kernel(RayArgs A) {
    __shared__ double stage[L > 1 ? kRayThreads : 1][kWin];
    const long long id = static_cast<long long>(blockIdx.x) * blockDim.x + threadIdx.x;
    const int ray = static_cast<int>(id / L), c = static_cast<int>(id % L);
    if (ray >= A.nray) return;
    const double b0 = A.b[2 * ray], b1 = A.b[2 * ray + 1];
    double *out = A.ds + static_cast<size_t>(ray) * A.ld;
    const Geo &G = A.G;
    const double *Rl = A.R, *Nl = A.N;
    int nl = A.nl;
    if (A.ray_atm) {
        const int a = A.ray_atm[ray];
        const int l0 = (a >= 0 && a < A.natm) ? A.layer_off[a] : -1;
        const int l1 = (a >= 0 && a < A.natm) ? A.layer_off[a + 1] : -1;
        if (l0 < 0 || l1 > A.nl || l1 - l0 < 2 || l1 - l0 - 1 > A.ld) {   // bad index or offsets
            if (c == 0) A.nsteps[ray] = -2;
            return;
        }
        Rl += l0;
        Nl += l0;
        nl = l1 - l0;
    }
    const double rNorm = Rl[0];
    const double tmp = b0 * b0 + b1 * b1;
    if (!(tmp < 1.0)) {                                // raypath.py:126-127 (NaN b: off planet too)
        if (c == 0) A.nsteps[ray] = -1;
        return;
    }
    const double mu = sqrt(1.0 - tmp);

    // ---- findEdge: trial zQ = arange(1.01 sqrt(1-b^2), 0, -0.005) ----
    // a trial lies below the top shell when |v| < f, that is |v|^2 < f^2: no root per trial;
    // the distances of the two bracketing trials are formed once the bracket is known
    const double start = mu * 1.01;
    const int ntrial = static_cast<int>(ceil((0.0 - start) / -0.005));
    const double z1 = start + -0.005;
    const double dz = z1 - start;
    const double flat = 1.0 - G.ratio * G.ratio;
    const bool shell = rNorm != 0.0 && fabs(rNorm) < INFINITY;   // (else no trial is below it)
    auto trial = [&](int i) { return (i == 0) ? start : ((i == 1) ? z1 : start + i * dz); };
    int hit = -1;
    for (int i0 = 0; i0 < ntrial && hit < 0; i0 += L) {   // L trials at a time, the first below taken
        const int i = i0 + c;
        const V3 bv = mat(G.M, V3{b0, b1, trial(i)});
        const double q = dot(bv, bv), Y = bv.y * bv.y;
        // q < f^2 times q > 0 (1e-6 rad at y == 0)
        const bool below = shell && i < ntrial && q * q < fma(-flat, bv.y == 0.0 ? kLat0 * q : Y, q);
        if constexpr (L == 1) {
            if (below) hit = i;
        } else {
            const unsigned long long any =
                (__builtin_amdgcn_ballot_w64(below) >> (threadIdx.x % 64 / L * L)) & (~0ull >> (64 - L));
            if (any != 0ull) hit = i0 + __builtin_ctzll(any);
        }
    }
    if (hit < 0) {
        if (c == 0) A.nsteps[ray] = -1;
        return;
    }
    auto above = [&](double z) {   // |v| - top shell radius at v's latitude
        const V3 bv = mat(G.M, V3{b0, b1, z});
        return norm(bv) * rNorm - ellipse(G, rNorm, latlng(bv)).rmag;
    };
    const double zhit = trial(hit), dhit = above(zhit);
    const double zprev = hit > 0 ? trial(hit - 1) : 0.0, dprev = hit > 0 ? above(zprev) : 0.0;
    // np.interp(0, [dhit, dprev], [zhit, zprev]) on the two bracketing trials
    double zq;
    if (hit == 0 || dhit == 0.0) {
        zq = zhit;
    } else {
        const double slope = (zprev - zhit) / (dprev - dhit);
        zq = slope * (0.0 - dhit) + zhit;
        if (zq != zq) zq = slope * (0.0 - dprev) + zprev;
    }
    const V3 edge = rNorm * mat(G.M, V3{b0, b1, zq});

    // ---- compute_ds: start on the top shell at the edge's latitude ----
    const LatLng q0 = latlng(edge);
    const Surf geo = ellipse(G, rNorm, q0);
    V3 s = mat(G.M, V3{0.0, 0.0, -1.0});
    V3 r = geo.r;
    {
        // refraction at the first boundary (raypath.py:158, 179-180); every later one has
        // nratio = 1 (raypath.py:257), which leaves the direction as it is
        const double ci = -dot(s, geo.n);                // cos(t_inc)
        const double nratio = Nl[0] / Nl[1];
        const double st = nratio * sqrt(1.0 - ci * ci);  // sin(t_tran)
        s = nratio * s + (nratio * ci - sqrt(1.0 - st * st)) * geo.n;
    }
    double f2 = geo.rmag / rNorm;                        // the first step: at the edge's latitude
    f2 *= f2;
    const double unit = A.units == 1 ? 5.0E4 : 1.0;      // half steps in cm, or km
    int step = 0;
    if constexpr (L > 1) {
        if (dot(r, s) < 0.0) {
            double S;
            const int got = parallel_steps<L>(A, Rl, nl, out, flat, unit, r, s, f2, c, stage + (threadIdx.x - c), S);
            if (got >= 0) {
                if (c == 0) A.nsteps[ray] = got;
                return;
            }
            step = -1 - got;
            const double t = -S - dot(r, s);
            r = r + t * s;
            f2 = shell_f2(flat, r.y, dot(r, r));
            s = reflected(G, r, s);
        }
    }
    const int count = serial_steps<SEC>(A, Rl, nl, out, flat, unit, mu, r, s, f2, step, c == 0);
    if (c == 0) A.nsteps[ray] = count;
}

}  // namespace rbx

// planet shape, view and sizes shared by rbx_raypaths and rbx_raypaths_batch
static int fill_ray_args(rbx::RayArgs &A, const rbx_planet *planet, const double *R, const double *N, int nl,
                         const double *b, int nray, int out_units, double *ds, int ld, int *nsteps, const char *who) {
    RBX_CHECK_ARG(planet && R && N && b && ds && nsteps, "%s: null argument", who);
    RBX_CHECK_ARG(nl >= 2, "%s: need at least 2 layers (nl=%d)", who, nl);
    RBX_CHECK_ARG(nray >= 0, "%s: negative ray count", who);
    RBX_CHECK_ARG(out_units == 0 || out_units == 1, "%s: bad out_units %d", who, out_units);
    RBX_CHECK_ARG(planet->gtype == 0 || planet->gtype == 1, "%s: bad gtype %d", who, planet->gtype);
    RBX_CHECK_ARG(planet->limb == 0 || planet->limb == 1, "%s: bad limb %d", who, planet->limb);
    RBX_CHECK_ARG(planet->req > 0.0 && planet->rpol > 0.0, "%s: radii must be positive", who);
    // computeAspect (raypath.py:39-44)
    const double f = 1.0 - planet->rpol / planet->req;
    const double tip = -planet->orientation[0] * rbx::kPi / 180.0;
    const double rot = -std::atan(std::tan(planet->orientation[1] * rbx::kPi / 180.0) * (1.0 - f) * (1.0 - f));
    const double ct = std::cos(tip), st = std::sin(tip), cr = std::cos(rot), sr = std::sin(rot);
    // rotX(rot) * rotZ(tip)
    const double M[9] = {ct, -st, 0.0, cr * st, cr * ct, -sr, sr * st, sr * ct, cr};
    for (int i = 0; i < 9; ++i) A.G.M[i] = M[i];
    A.G.ratio = planet->gtype == 0 ? planet->rpol / planet->req : 1.0;
    A.R = R;
    A.N = N;
    A.nl = nl;
    A.b = b;
    A.nray = nray;
    A.units = out_units;
    A.ds = ds;
    A.ld = ld;
    A.nsteps = nsteps;
    A.limb = planet->limb;
    A.ray_atm = nullptr;
    A.layer_off = nullptr;
    A.natm = 0;
    return RBX_OK;
}

// Lanes per ray: a thread's chain of steps bounds a launch until its wavefronts fill the SIMDs, so a
// ray's steps are split over kRayLanes; past kSplitRays rays a thread per ray fills the device and
// the second walk over the steps only adds work.  One number of lanes up to there, so that a ray's
// path does not depend on the rays beside it.  Measured (us, 1 lane and 32): 1000 layers x 4 rays
// 183 -> 23, 500 x 256 100 -> 22, 400 x 4096 82 -> 23, 800 x 16384 150 -> 93, 800 x 32768 176 -> 173,
// 800 x 65536 233 against 330 (16 lanes 36, 24, 24, 87, 161, 298; 64 lanes 22, 21, 26, 106, 195).
constexpr int kRayLanes = 32, kSplitRays = 32768;

static int launch_rays(const rbx::RayArgs &A, void *stream) {
    const int threads = rbx::kRayThreads;
    const bool split = A.limb != 1 && A.nray <= kSplitRays;   // ('sec' steps leave the straight line)
    const long long lanes = static_cast<long long>(A.nray) * (split ? kRayLanes : 1);
    const dim3 grid(static_cast<unsigned>((lanes + threads - 1) / threads));
    hipStream_t st = static_cast<hipStream_t>(stream);
    if (split) hipLaunchKernelGGL((rbx::raypath_kernel<false, kRayLanes>), grid, dim3(threads), 0, st, A);
    else if (A.limb == 1) hipLaunchKernelGGL((rbx::raypath_kernel<true, 1>), grid, dim3(threads), 0, st, A);
    else hipLaunchKernelGGL((rbx::raypath_kernel<false, 1>), grid, dim3(threads), 0, st, A);
    return rbx::launch_status("raypath_kernel");
}

extern "C" int rbx_raypaths(const rbx_planet *planet, const double *R, const double *N, int nl, const double *b,
                            int nray, int out_units, double *ds, int ld, int *nsteps, void *stream) {
    rbx::RayArgs A;
    int rc = fill_ray_args(A, planet, R, N, nl, b, nray, out_units, ds, ld, nsteps, "rbx_raypaths");
    if (rc) return rc;
    RBX_CHECK_ARG(ld >= nl - 1, "rbx_raypaths: ld=%d < nl-1=%d", ld, nl - 1);
    if (nray == 0) return RBX_OK;
    return launch_rays(A, stream);
}

extern "C" int rbx_raypaths_batch(const rbx_planet *planet, const double *R, const double *N, int nl_total,
                                  const int *layer_off, int natm, const double *b, int nray, const int *ray_atm,
                                  int out_units, double *ds, int ld, int *nsteps, void *stream) {
    rbx::RayArgs A;
    int rc = fill_ray_args(A, planet, R, N, nl_total, b, nray, out_units, ds, ld, nsteps, "rbx_raypaths_batch");
    if (rc) return rc;
    RBX_CHECK_ARG(layer_off && ray_atm && natm > 0, "rbx_raypaths_batch: null offsets / ray map or natm=%d", natm);
    RBX_CHECK_ARG(ld >= 1, "rbx_raypaths_batch: ld=%d", ld);
    if (nray == 0) return RBX_OK;
    A.ray_atm = ray_atm;
    A.layer_off = layer_off;
    A.natm = natm;
    return launch_rays(A, stream);
}
