// fsg_post.hip -- the potential and distance-estimate layers of a tile,
// computed on the GPU from the raw results while they are still in HBM.
//
// Restates, per pixel:
//   Continuous_iter_pp with kind "infinity" (src/fractalshades/postproc.py:
//   352-406, formula 1001-1009):
//     k = |a_d|^(1/(d-1)),  nu_frac = -log(log|z_n k| / log(M k)) / log d,
//     (div, mod) = divmod(-nu_frac, 1),  nu = (n - div - floor_iter) - mod
//   DEM_pp (postproc.py:684-731): |z_n| ln|z_n| / |dz_n/dc|, where for the
//   burning ship |dz_n/dc| is the larger singular value of the Jacobian,
//   (hypot(a + d, b - c) + hypot(a - d, b + c)) / 2, and values below
//   px_snap are snapped to 0.
//   Attr_normal_pp with kind "potential" / "infinity" (postproc.py:572-628):
//     holomorphic z_n / (dz_n/dc); burning ship J^T z_n with J the Jacobian
//     d(x, y)/d(a, b); then the transposed skew (apply_unskew_1d,
//     core.py:3147-3158) and division by the modulus.  The direction of
//     z_n / (dz_n/dc) is that of z_n conj(dz_n/dc), which is formed instead
//     (after a power-of-two scaling of the derivative, so that no product
//     overflows): the unit vector is the same.
//   Before the DEM and the normal, the derivatives take the loop's
//   dzndc_modifier (perturbation.py:1387-1388, which the tile kernels leave
//   to the host) and the projection's map at the pixel (get_dzndc,
//   postproc.py:184-206): dz/dc times df (apply_df, 972-978), the Jacobian
//   times the dfBS matrix (apply_dfBS, 980-998), the maps of the exponential
//   projection (projection.py:375-453).
// Each pixel takes layers_squares, or layers_general where a square would
// leave binary64's range.
// Computed in binary64, stored as binary32 (the reference's default
// post-processing dtype, settings.py:82).  Pixels that did not diverge get
// NaN in every layer: the reference's formulas have no meaning there and its
// layers mask them by stop reason.
#include "fsgpu.h"
#include "fsg_internal.hpp"

#include <cmath>
#include <string>

namespace fsg {
int set_error(int code, const std::string &msg);
}

using namespace fsg;

namespace {

struct PostArgs {
    const double *Z;
    const double *pix;
    int64_t n, ld;
    const int32_t *si;
    const int8_t *sr;
    float *nu, *dem, *nrm;
    int32_t holo, row_dc;
    double k, log_mk, log_d, floor_iter, px_snap;
    double s00, s01, s10, s11;
    int32_t proj, mod;
    double w_scale, mod_scale;
    // layers_squares' constants; skewed: the skew is not the identity; plain:
    // the constants are ones that it may take
    double log_k, inv_log_mk, inv_log_d;
    int32_t skewed, plain;
};

// The projection's map at pixel i, from its projected offset w = exp(h + t)
// (h real: the map's h_moy, or h_moy - h_band by bands): exp(t) = w e^-h,
// exp(i Im t) = w / |w|.  Holomorphic factor (fr, fi); burning-ship matrix
// (m00, m01, m10, m11) as projection.py:412-453 writes them.
__device__ void proj_map(const PostArgs &p, int64_t i, double &fr, double &fi, double m[4]) {
    const double wx = p.pix[2 * i], wy = p.pix[2 * i + 1];
    if (p.proj == 1) {                 // exp(t); (-Im e^t, -Re e^t, Re e^t, -Im e^t)
        const double cr = wx * p.w_scale, sr = wy * p.w_scale;
        fr = cr; fi = sr;
        m[0] = -sr; m[1] = -cr; m[2] = cr; m[3] = -sr;
    } else if (p.proj == 2) {          // exp(Re t)
        const double r = hypot(wx, wy) * p.w_scale;
        fr = r; fi = 0.;
        m[0] = r; m[1] = 0.; m[2] = 0.; m[3] = r;
    } else if (p.proj == 3) {          // exp(i Im t)
        const double a = hypot(wx, wy), c = wx / a, s = wy / a;
        fr = c; fi = s;
        m[0] = c; m[1] = -s; m[2] = s; m[3] = c;
    } else {
        fr = 1.; fi = 0.;
        m[0] = 1.; m[1] = 0.; m[2] = 0.; m[3] = 1.;
    }
}

// One pixel's layers in the form that takes every value: each logarithm,
// modulus and quotient by the math library.
template <bool HOLO> __device__ void layers_general(const PostArgs &p, double zr, double zi, const double J[4], double n_it, float out[4]) {
    if (p.nu) {
        const double azk = hypot(zr * p.k, zi * p.k);
        const double nu_frac = -(log(log(azk) / p.log_mk) / p.log_d);
        // numpy divmod(x, 1.): floor and the non-negative remainder
        const double x = -nu_frac;
        const double dv = floor(x);
        const double md = x - dv;
        out[0] = (float)(((n_it - dv) - p.floor_iter) - md);
    }
    const double dr = J[0], di = J[1], a = J[0], b = J[1], c = J[2], d = J[3];
    if (p.dem) {
        const double az = hypot(zr, zi);
        const double ad = HOLO ? hypot(dr, di) : 0.5 * (hypot(a + d, b - c) + hypot(a - d, b + c));
        double v = az * log(az) / ad;
        if (p.px_snap > 0. && v < p.px_snap) v = 0.;
        out[1] = (float)v;
    }
    if (p.nrm) {
        double nx, ny;
        if (HOLO) {
            const int sh = -__builtin_amdgcn_frexp_exp(fmax(fabs(dr), fabs(di)));
            const double er = ldexp(dr, sh), ei = ldexp(di, sh);
            nx = zr * er + zi * ei;          // z conj(dz/dc)
            ny = zi * er - zr * ei;
        } else {
            const int sh = -__builtin_amdgcn_frexp_exp(fmax(fmax(fabs(a), fabs(b)), fmax(fabs(c), fabs(d))));
            const double ea = ldexp(a, sh), eb = ldexp(b, sh), ec = ldexp(c, sh), ed = ldexp(d, sh);
            nx = ea * zr + ec * zi;          // J^T z
            ny = eb * zr + ed * zi;
        }
        const double ux = p.s00 * nx + p.s10 * ny, uy = p.s01 * nx + p.s11 * ny;
        const double m = hypot(ux, uy);
        out[2] = (float)(ux / m);
        out[3] = (float)(uy / m);
    }
}

// ln x of a positive normal x, within 2 ulp: x = 2^e m with m in [1/sqrt 2,
// sqrt 2), ln m = 2 atanh(s) = 2 s (1 + s^2/3 + s^4/5 + ...) at s = (m - 1) /
// (m + 1); |s| <= 0.172, so the term after s^18/19 is below 2^-55.
__device__ double log_pos(double x) {
    int e = __builtin_amdgcn_frexp_exp(x);
    double m = __builtin_amdgcn_frexp_mant(x);          // [0.5, 1)
    const int lo = m < 0.70710678118654752 ? 1 : 0;
    m = ldexp(m, lo);
    e -= lo;
    const double f = m - 1., g = m + 1.;
    double y = __builtin_amdgcn_rcp(g);
    y = fma(y, fma(-g, y, 1.), y);
    double s = f * y;
    s = fma(fma(-g, s, f), y, s);
    const double z = s * s;
    double t = 1. / 19;
    t = fma(t, z, 1. / 17);
    t = fma(t, z, 1. / 15);
    t = fma(t, z, 1. / 13);
    t = fma(t, z, 1. / 11);
    t = fma(t, z, 1. / 9);
    t = fma(t, z, 1. / 7);
    t = fma(t, z, 1. / 5);
    t = fma(t, z, 1. / 3);
    const double s2 = s + s;
    return fma((double)e, 0.69314718055994530942, fma(s2, z * t, s2));
}

// The same layers from squares, where none of them leaves binary64's range
// (false, and nothing said of out, elsewhere): one logarithm for both |z|'s,
// ln|z| = ln(q) / 2 with q = |z|^2; |z| / |d| = q rsqrt(q |d|^2); the normal
// is n rsqrt(|n|^2), where an unskewed holomorphic one has |n|^2 = q |d|^2.
template <bool HOLO> __device__ bool layers_squares(const PostArgs &p, double zr, double zi, const double J[4], double n_it, float out[4]) {
    const double q = zr * zr + zi * zi;
    const double L = 0.5 * log_pos(q);
    bool ok = q >= 2. && q <= 0x1p400;
    if (p.nu) {
        const double Lk = L + p.log_k;
        ok = ok && Lk >= 0.25;
        const double x = log_pos(Lk * p.inv_log_mk) * p.inv_log_d;
        const double dv = floor(x);
        const double md = x - dv;
        out[0] = (float)(((n_it - dv) - p.floor_iter) - md);
    }
    if (!p.dem && !p.nrm) return ok;
    double nx, ny, rs;
    if (HOLO) {
        const double dr = J[0], di = J[1];
        const double dd = dr * dr + di * di;
        ok = ok && dd >= 0x1p-400 && dd <= 0x1p400;
        rs = rsqrt(q * dd);
        if (p.dem) {
            double v = L * (q * rs);
            if (p.px_snap > 0. && v < p.px_snap) v = 0.;
            out[1] = (float)v;
        }
        nx = zr * dr + zi * di;          // z conj(dz/dc)
        ny = zi * dr - zr * di;
    } else {
        const double a = J[0], b = J[1], c = J[2], d = J[3];
        if (p.dem) {
            const double s = a + d, t = b - c, u = a - d, w = b + c;
            const double q1 = s * s + t * t, q2 = u * u + w * w;
            ok = ok && q1 + q2 >= 0x1p-800 && q1 + q2 <= 0x1p800;
            double v = sqrt(q) * L / (0.5 * (sqrt(q1) + sqrt(q2)));
            if (p.px_snap > 0. && v < p.px_snap) v = 0.;
            out[1] = (float)v;
        }
        nx = a * zr + c * zi;            // J^T z
        ny = b * zr + d * zi;
    }
    if (p.nrm) {
        if (!HOLO || p.skewed) {
            const double ux = p.s00 * nx + p.s10 * ny, uy = p.s01 * nx + p.s11 * ny;
            nx = ux; ny = uy;
            const double mm = nx * nx + ny * ny;
            ok = ok && mm >= 0x1p-800 && mm <= 0x1p800;
            rs = rsqrt(mm);
        }
        out[2] = (float)(nx * rs);
        out[3] = (float)(ny * rs);
    }
    return ok;
}

// Bound by memory: 53 bytes a pixel (69 with a Jacobian).  4096 x 4096 pixels,
// 889 MB, take 174 us, 5.1 TB/s, where a copy of 1 GiB reaches 5.2; a 2048 x 2048
// frame takes 42 (58) us, 5.3 TB/s: its 222 MB stay in part in the 256 MB cache
// behind the L2s.  The general form on every pixel takes 78 (86) us there, three
// 98-instruction logarithms, four moduli and five quotients of binary64 issue.  One kernel per form of derivative:
// its loads are then unconditional and all in flight together.
template <bool HOLO> __global__ void __launch_bounds__(256) k_postproc(const PostArgs p) {
    const int64_t stride = (int64_t)gridDim.x * blockDim.x;
    for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < p.n; i += stride) {
        // every load before the first use of one: a pixel's values do not
        // wait for its stop reason
        const int8_t reason = p.sr[i];
        const double n_it = (double)p.si[i];
        double zr, zi, J[4] = {0., 0., 0., 0.};  // dz/dc, or the Jacobian (dX/dA dX/dB; dY/dA dY/dB)
        if (HOLO) { zr = p.Z[2 * i]; zi = p.Z[2 * i + 1]; }
        else { zr = p.Z[i]; zi = p.Z[p.ld + i]; }
        if (p.dem || p.nrm) {
            if (HOLO) {
                const int64_t r = (int64_t)p.row_dc * p.ld + i;
                J[0] = p.Z[2 * r]; J[1] = p.Z[2 * r + 1];
            } else {
                const double *src = p.Z + (int64_t)p.row_dc * p.ld + i;
                for (int k = 0; k < 4; ++k) J[k] = src[k * p.ld];
            }
            if (p.mod != 0) {
                // the loop's dzndc_modifier at the pixel
                const double wx = p.pix[2 * i], wy = p.pix[2 * i + 1];
                const double f = (p.mod == 1 ? hypot(wx, wy) : hypot(wx + 1.e-6, wy)) * p.mod_scale;
                for (int k = 0; k < 4; ++k) J[k] *= f;
            }
            if (p.proj != 0) {
                double fr, fi, m[4];
                proj_map(p, i, fr, fi, m);
                const double a = J[0], b = J[1], c = J[2], d = J[3];
                if (HOLO) {
                    J[0] = fr * a - fi * b; J[1] = fr * b + fi * a;
                } else {
                    J[0] = a * m[0] + b * m[2]; J[1] = a * m[1] + b * m[3];
                    J[2] = c * m[0] + d * m[2]; J[3] = c * m[1] + d * m[3];
                }
            }
        }
        float out[4];
        const bool done = layers_squares<HOLO>(p, zr, zi, J, n_it, out) && p.plain;
        if (reason != 1) {
            for (int k = 0; k < 4; ++k) out[k] = __builtin_nanf("");
        } else if (!done) {
            layers_general<HOLO>(p, zr, zi, J, n_it, out);
        }
        if (p.nu) p.nu[i] = out[0];
        if (p.dem) p.dem[i] = out[1];
        if (p.nrm) { p.nrm[2 * i] = out[2]; p.nrm[2 * i + 1] = out[3]; }
    }
}

int fill_post(const fsg_post_desc *pp, PostArgs &a) {
    if (!pp) return set_error(FSG_E_INVALID, "null post-processing descriptor");
    if (!(pp->d > 1.) || !(pp->M > 0.)) return set_error(FSG_E_INVALID, "potential needs d > 1 and M > 0");
    a.holo = pp->holomorphic ? 1 : 0;
    a.row_dc = pp->dzndc_row;
    a.k = std::pow(std::fabs(pp->a_d), 1. / (pp->d - 1.));
    a.log_mk = std::log(pp->M * a.k);
    a.log_d = std::log(pp->d);
    a.floor_iter = pp->floor_iter;
    a.px_snap = pp->px_snap;
    const bool skew = pp->skew[0] != 0. || pp->skew[1] != 0. || pp->skew[2] != 0. || pp->skew[3] != 0.;
    a.s00 = skew ? pp->skew[0] : 1.; a.s01 = skew ? pp->skew[1] : 0.;
    a.s10 = skew ? pp->skew[2] : 0.; a.s11 = skew ? pp->skew[3] : 1.;
    if (pp->proj < 0 || pp->proj > 4) return set_error(FSG_E_INVALID, "unknown projection map");
    a.proj = pp->proj == 4 ? 0 : pp->proj;      // the map "one" changes nothing
    a.w_scale = pp->w_scale;
    if (pp->mod < 0 || pp->mod > 2) return set_error(FSG_E_INVALID, "unknown derivative modifier");
    a.mod = pp->mod; a.mod_scale = pp->mod_scale;
    a.skewed = a.s00 != 1. || a.s01 != 0. || a.s10 != 0. || a.s11 != 1.;
    a.log_k = std::log(a.k);
    a.inv_log_mk = 1. / a.log_mk;
    a.inv_log_d = 1. / a.log_d;
    // k = 0, M k <= 1 and non-finite constants are layers_general's
    a.plain = a.log_k >= -0x1p10 && a.log_k <= 0x1p10 && a.log_mk >= 0x1p-100 && a.log_mk <= 0x1p100;
    return 0;
}

}  // namespace

namespace fsg {

// enqueue the layers of n pixels whose raw results sit in Z (row stride ld)
int post_launch(const fsg_post_desc *pp, const double *Z, int64_t n, int64_t ld, const double *pix,
                const int32_t *si, const int8_t *sr, float *nu, float *dem, float *nrm, hipStream_t stream) {
    PostArgs a;
    int rc = fill_post(pp, a);
    if (rc) return rc;
    if ((dem || nrm) && pp->dzndc_row < 1)
        return set_error(FSG_E_INVALID, "DEM and normal need the dz/dc (Jacobian) rows");
    if ((a.proj != 0 || a.mod != 0) && (dem || nrm) && n > 0 && !pix)
        return set_error(FSG_E_INVALID, "the projection's map needs the pixels");
    a.Z = Z; a.pix = pix; a.n = n; a.ld = ld; a.si = si; a.sr = sr; a.nu = nu; a.dem = dem; a.nrm = nrm;
    if (n <= 0) return 0;
    int64_t blocks = (n + 255) / 256;
    if (blocks > 8192) blocks = 8192;
    hipLaunchKernelGGL(a.holo ? k_postproc<true> : k_postproc<false>, dim3((unsigned)blocks), dim3(256), 0, stream, a);
    if (hipGetLastError() != hipSuccess) return set_error(FSG_E_HIP, "post-processing launch failed");
    return 0;
}

}  // namespace fsg

extern "C" {

int fsg_postproc_device(const fsg_post_desc *pp, const double *d_Z, int64_t n, int64_t ld,
                        const double *d_c_pix, const int32_t *d_stop_iter, const int8_t *d_stop_reason,
                        float *d_nu, float *d_dem, float *d_normal, void *stream) {
    if (n < 0 || ld < n || (n > 0 && (!d_Z || !d_stop_iter || !d_stop_reason)))
        return set_error(FSG_E_INVALID, "bad post-processing buffers");
    return post_launch(pp, d_Z, n, ld, d_c_pix, d_stop_iter, d_stop_reason, d_nu, d_dem, d_normal,
                       static_cast<hipStream_t>(stream));
}

}  // extern "C"
