// The exponential-disk density model (optionally with a logarithmic spiral perturbation)
// normalised to a face-on optical depth: set up on the host, evaluated on the host (set-up,
// octree refinement, cell densities) and on the device (cell densities of a resident grid).
// ExpDiskGeometry (ExpDiskGeometry.cpp), SpiralStructureGeometryDecorator
// (SpiralStructureGeometryDecorator.cpp) and OpticalDepthMaterialNormalization.
#pragma once

#include <hip/hip_runtime.h>
#include <cmath>

#include "../../include/skirt_mi355x.h"
#include "philox.hpp"

namespace skg
{
    struct DiskModel
    {
        double hR, hz, rho0;
        bool spiral;
        double m, tanp, R0, phi0, w, cn;
        int N;
        double nnorm;  // number density per unit normalised geometric density
        // constants of geom_device: reciprocals of hR, hz and R0^2, and the spiral's phase
        // m gamma / 2 = phaseA log(R^2 / R0^2) + phaseB
        double ihR, ihz, iR02, phaseA, phaseB;

        explicit DiskModel(const skg_disk_model& d)
        {
            hR = d.scale_length;
            hz = d.scale_height;
            // ExpDiskGeometry::setupSelfBefore (no truncation): rho0 = 1 / (2 pi hR^2 * 2 hz)
            double intphi = 2.0 * M_PI;
            double intz = 2.0 * hz;
            double intR = hR * hR * (1.0 - 0.0);
            rho0 = 1.0 / (intR * intphi * intz);
            spiral = d.spiral_arms > 0;
            m = d.spiral_arms;
            N = d.spiral_index;
            tanp = std::tan(d.pitch_angle);
            R0 = d.radius_zero;
            phi0 = d.phase_zero;
            w = d.perturbation_weight;
            // SpiralStructureGeometryDecorator::setupSelfBefore: cn = sqrt(pi) Gamma(N+1) / Gamma(N+1/2)
            cn = std::sqrt(M_PI) * std::tgamma(N + 1.0) / std::tgamma(N + 0.5);
            // OpticalDepthMaterialNormalization along Z: number = tau / (sigma * SigmaZ), SigmaZ = 2 rho0 hz
            double sigmaZ = 2.0 * rho0 * hz;
            nnorm = d.tau_v / d.sext_v / sigmaZ;
            ihR = 1. / hR;
            ihz = 1. / hz;
            iR02 = 1. / (R0 * R0);
            phaseA = 0.25 * m / tanp;
            phaseB = 0.5 * m * phi0 + 0.25 * M_PI;
        }

        // normalised geometric density (integrates to one)
        double geom(double x, double y, double z) const
        {
            double R = sqrt(x * x + y * y);
            double v = rho0 * exp(-R / hR) * exp(-fabs(z) / hz);
            if (spiral)
            {
                double phi = atan2(y, x);
                double gamma = log(R / R0) / tanp + phi0 + 0.5 * M_PI / m;
                v *= (1.0 - w) + w * cn * pow(sin(0.5 * m * (gamma - phi)), 2 * N);
            }
            return v;
        }

        // The same on the device, where the transcendental functions bound the sampling kernels
        // (one evaluation per sample): one exponential of the summed exponents, no power function
        // (sin^2N by squaring), and the azimuth only as the cosine and sine of m phi / 2, from powers
        // of (x + i y) / R, so no arc tangent.  The sine of m (gamma - phi) / 2 as the difference of
        // two products keeps geom's relative accuracy near its zeros; over random models the errors
        // of cell averages against extended precision equal geom's (rms 1e-16 to 7e-15).
        __device__ __forceinline__ double geom_device(double x, double y, double z) const
        {
            const double R2 = fma(x, x, y * y), R = sqrt(R2);
            double v = rho0 * exp(-fma(R, ihR, fabs(z) * ihz));
            if (spiral)
            {
                double p = x / R, q = y / R;
                int e = static_cast<int>(m);
                if (e & 1)
                {
                    // half angles, the larger component by the root
                    const double a = sqrt(fma(0.5, fabs(p), 0.5)), b = 0.5 * fabs(q) / a;
                    q = copysign(p >= 0. ? b : a, q);
                    p = p >= 0. ? a : b;
                }
                else
                    e >>= 1;
                double c = 1., s = 0.;  // (p + i q)^e
                while (true)
                {
                    if (e & 1)
                    {
                        const double t = fma(c, p, -(s * q));
                        s = fma(c, q, s * p);
                        c = t;
                    }
                    if (!(e >>= 1)) break;
                    const double t = fma(p, p, -(q * q));
                    q = 2. * p * q;
                    p = t;
                }
                double sg, cg;
                sincos(fma(phaseA, log(R2 * iR02), phaseB), &sg, &cg);
                double f = fma(sg, c, -(cg * s));
                f *= f;
                double g = 1.;  // f^N
                for (int k = N; k > 0; k >>= 1)
                {
                    if (k & 1) g *= f;
                    f *= f;
                }
                v *= fma(w * cn, g, 1.0 - w);
            }
            return v;
        }
    };

    // The sum of f(u, v, w) over n points with three deviates each from the stream (seed, id, tag), or
    // over the share of lane `sub` of `lanes` lanes: two points per three blocks of the generator.
    template<typename F>
    __device__ __forceinline__ double sample_sum(int n, int sub, int lanes, uint64_t seed, uint64_t id, uint32_t tag, F f)
    {
        Philox a, b;
        a.init(seed, id, tag);
        b.init(seed, id, tag);
        double sum = 0.;
        for (int q = 2 * sub; q < n; q += 2 * lanes)
        {
            const uint32_t block = static_cast<uint32_t>(q / 2) * 3u;
            a.gen(block);
            b.gen(block + 1);
            sum += f(a.first(), a.second(), b.first());
            if (q + 1 == n) break;
            a.gen(block + 2);
            sum += f(b.second(), a.first(), a.second());
        }
        return sum;
    }
}
