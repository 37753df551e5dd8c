// Ray geometry in FP64: one thread per ray.
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

// Rays per block.  One thread per ray: a ray's path is one dependent chain of FP64 steps, so
// the kernel is latency-bound and holds few wavefronts (256 for 16384 rays).  It runs beside the
// line sums (rbx_alpha) when a caller puts it on a second stream or graph branch; four
// wavefronts per block keep it on a quarter as many CUs as one per block, leaving the other
// CUs' slots whole for the line sums: 800 layers x 1024 frequencies x 16384 rays, graph step
// 3.71 -> 3.47 ms when the paths alone took 0.42 -> 0.45 ms (2 and 8 wavefronts per block: 3.59,
// 3.53 ms).
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

// SEC: limb 'sec' (raypath.py:218-219)
template <bool SEC>
__global__ __launch_bounds__(kRayThreads) void raypath_kernel(RayArgs A) {
    const int ray = blockIdx.x * blockDim.x + threadIdx.x;
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
            A.nsteps[ray] = -2;
            return;
        }
        Rl += l0;
        Nl += l0;
        nl = l1 - l0;
    }
    const double rNorm = Rl[0];
    const double tmp = b0 * b0 + b1 * b1;
    if (!(tmp < 1.0)) {                                // raypath.py:126-127 (NaN b: off planet too)
        A.nsteps[ray] = -1;
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
    auto trial = [&](int i) { return (i == 0) ? start : ((i == 1) ? z1 : start + i * dz); };
    int hit = -1;
    for (int i = 0; i < ntrial; ++i) {
        const V3 bv = mat(G.M, V3{b0, b1, trial(i)});
        const double q = dot(bv, bv), Y = bv.y * bv.y;
        // q < f^2 times q > 0 (1e-6 rad at y == 0)
        if (q * q < fma(-flat, bv.y == 0.0 ? kLat0 * q : Y, q)) {
            hit = i;
            break;
        }
    }
    if (hit < 0) {
        A.nsteps[ray] = -1;
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
        const double c = -dot(s, geo.n);                 // cos(t_inc)
        const double nratio = Nl[0] / Nl[1];
        const double st = nratio * sqrt(1.0 - c * c);    // sin(t_tran)
        s = nratio * s + (nratio * c - sqrt(1.0 - st * st)) * geo.n;
    }
    // The rest of the path is the straight line r + t s, so a step is a chain in t alone: the
    // point's y and |r|^2 (for f^2 at its latitude), r.s, the root of the next shell.  The next
    // shell's radius is taken at the current point's latitude (raypath.py:182), hence
    // disc = (r.s)^2 - f^2 (R_k^2 - R_{k+1}^2).  One thread's chain per ray bounds the kernel
    // (carrying the point, two angles and four roots it took 0.48 us a step; as a chain in t
    // 0.17 us: 1000 layers x 4 rays 480 -> 166 us, 800 layers x 16384 rays 440 -> 153 us).
    double t = 0.0, y1 = r.y, q1 = dot(r, r), d1 = dot(r, s);
    int count = 0;
    double f2 = geo.rmag / rNorm;                        // the first step: at the edge's latitude
    f2 *= f2;
    // Equatorial radii by windows of kWin steps, the next window's loads issued a window ahead: a
    // step is shorter than a load, and fetched one step ahead each step waited for one (1000
    // layers x 4 rays 256 us).
    // A lane whose path has ended computes on (nothing it writes): the window has no exits.
    const double unit = A.units == 1 ? 5.0E4 : 1.0;      // half steps in cm, or km
    double win[kWin + 1], nxt[kWin];
#pragma unroll
    for (int u = 0; u <= kWin; ++u) win[u] = Rl[min(u, nl - 1)];
    bool alive = true;
    for (int k0 = 0; alive; k0 += kWin) {
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
            if (alive) out[k0 + u] = ds * unit;
            count += alive ? 1 : 0;
            t += ds;
            const double y = fma(t, s.y, y1);
            f2 = shell_f2(flat, y, fma(t, fma(2.0, d1, t), q1));
            // incidence past 90 degrees, cos(t_inc) = -s.n < 0 with n along (ratio x, y, ratio z):
            // the reference's arcsin(sin t_inc) then folds the angle, which turns the direction
            // by 2 cos n
            const double ys = y * s.y, along = fma(G.ratio, (d1 + t) - ys, ys);
            if (__builtin_expect(alive && along > 0.0, 0)) {
                r = r + t * s;
                V3 n = {G.ratio * r.x, r.y, G.ratio * r.z};
                n = (1.0 / norm(n)) * n;
                const double c = -dot(s, n), st = sqrt(1.0 - c * c);
                s = s + (c - sqrt(1.0 - st * st)) * n;
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
    A.nsteps[ray] = count;
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

static int launch_rays(const rbx::RayArgs &A, void *stream) {
    const int threads = rbx::kRayThreads;
    const dim3 grid((A.nray + threads - 1) / threads);
    if (A.limb == 1)
        hipLaunchKernelGGL(rbx::raypath_kernel<true>, grid, dim3(threads), 0, static_cast<hipStream_t>(stream), A);
    else
        hipLaunchKernelGGL(rbx::raypath_kernel<false>, grid, dim3(threads), 0, static_cast<hipStream_t>(stream), A);
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
