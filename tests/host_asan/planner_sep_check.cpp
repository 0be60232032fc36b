// Host build of the planner's tables of the separable tiles (idi_amd/csrc/planner.hpp) for
// tests/test_planner_sep_cpu.py, with sanitizers.
//
// Input, one case per line (stdin):
//   n0 n1 pixelsize detz k off0 off1 nf scale secondorder rot m0 .. m8 tol_rev summode nrho rho_1 .. rho_nrho
// Output, one JSON object per case (stdout): the tables of the three rectangles, what an evaluation of
// every pixel in FP64 gives for each, the error of the kernel's series for the mixed remainder, and for
// every extent the bounds of tiles 17 .. 22, the eligible ones and the adjoint's side and bounds.
#include "../../idi_amd/csrc/checks.hpp"
#include "../../idi_amd/csrc/planner.hpp"

#include <cstdio>
#include <string>
#include <vector>

using namespace idisim;

static void put(const char* name, double v, bool last = false)
{
    if (std::isfinite(v))
        std::printf("\"%s\": %.17g%s", name, v, last ? "" : ", ");
    else
        std::printf("\"%s\": null%s", name, last ? "" : ", ");
}

static double norm(const double v[3]) { return std::sqrt(v[0] * v[0] + v[1] * v[1] + v[2] * v[2]); }

struct Brute {
    double line = 0, mixed = 0, rest = 0, off = 0, fourth = 0, du = 0, dR = 0, series = 0;
};

static Brute brute(const Geom& g, int TX, int TY)
{
    Brute b;
    const double hx = 0.5 * (TX - 1), hy = 0.5 * (TY - 1);
    for (int x0 = 0; x0 < g.n0; x0 += TX)
        for (int y0 = 0; y0 < g.n1; y0 += TY) {
            const double cx = x0 + hx, cy = y0 + hy;
            double r[3];
            pixel_pos(g, cx, cy, r);
            const SepFrame f = make_sep_frame(g, r);
            float e[2][3];
            sep_basis_of(f, e);
            double v3[2][3];
            sep_third(f, v3);
            const Frame c = make_frame(r);
            const Frame wc = pixel_frame(g, x0 / (2 * TX) * (2 * TX) + TX - 0.5, y0 / (2 * TY) * (2 * TY) + TY - 0.5);
            for (int j = 0; j < TY; ++j) {
                const Frame fy = pixel_frame(g, cx, y0 + j);
                double l[3];
                for (int k = 0; k < 3; ++k) l[k] = g.krev * (fy.u[k] - c.u[k]);
                b.line = std::max(b.line, norm(l));
            }
            for (int i = 0; i < TX; ++i) {
                const Frame fx = pixel_frame(g, x0 + i, cy);
                for (int j = 0; j < TY; ++j) {
                    const Frame p = pixel_frame(g, x0 + i, y0 + j), fy = pixel_frame(g, cx, y0 + j);
                    const double dx = i - hx, dy = j - hy;
                    double m[3], s[3], t[3], o[3], d[3], u[3];
                    float q[3];
                    sep_mixed(f, (float)dx, (float)dy, q);
                    for (int k = 0; k < 3; ++k) {
                        m[k] = -g.krev * ((p.u[k] - fx.u[k]) - (fy.u[k] - c.u[k]));
                        s[k] = m[k] - dx * dy * (double)f.mu[k];
                        t[k] = s[k] + g.krev * dx * dy * (dx * v3[0][k] + dy * v3[1][k]);
                        d[k] = m[k] - (double)q[k];
                        u[k] = p.u[k] - wc.u[k];
                    }
                    for (int k = 0; k < 3; ++k) {
                        o[k] = m[k];
                        for (int a = 0; a < 2; ++a)
                            o[k] -= (m[0] * e[a][0] + m[1] * e[a][1] + m[2] * e[a][2]) * (double)e[a][k];
                    }
                    b.mixed = std::max(b.mixed, norm(m));
                    b.rest = std::max(b.rest, norm(s));
                    b.fourth = std::max(b.fourth, norm(t));
                    b.off = std::max(b.off, norm(o));
                    b.series = std::max(b.series, norm(d));
                    b.du = std::max(b.du, norm(u));
                    b.dR = std::max(b.dR, std::fabs(p.R - wc.R));
                }
            }
        }
    return b;
}

int main()
{
    for (;;) {
        long n0, n1;
        double pix, detz, k, off0, off1, tol, M[9];
        int nf, scale, secondorder, rot, summode, nrho;
        if (std::scanf("%ld %ld %lf %lf %lf %lf %lf %d %d %d %d", &n0, &n1, &pix, &detz, &k, &off0, &off1, &nf, &scale,
                       &secondorder, &rot) != 11)
            break;
        for (double& m : M)
            if (std::scanf("%lf", &m) != 1) return 2;
        if (std::scanf("%lf %d %d", &tol, &summode, &nrho) != 3 || nrho < 0 || nrho > 64) return 2;
        std::vector<double> rhos((size_t)nrho);
        for (double& r : rhos)
            if (std::scanf("%lf", &r) != 1) return 2;
        idisim_geometry geom{};
        geom.n0 = n0;
        geom.n1 = n1;
        geom.pixelsize = pix;
        geom.detz = detz;
        geom.k = k;
        geom.detoffset[0] = off0;
        geom.detoffset[1] = off1;
        for (int i = 0; i < 9; ++i) geom.rot[i] = M[i];
        geom.flags = (nf ? IDISIM_NF : 0u) | (scale ? IDISIM_SCALE : 0u) | (secondorder ? IDISIM_SECONDORDER : 0u) |
                     (rot ? IDISIM_ROTATE : 0u);
        std::string msg;
        if (check_create(&geom, IDISIM_PREC_FP32SPLIT, &msg) != IDISIM_OK) return 3;
        Planner p;
        p.g = make_geom(geom);
        p.tol_rev = tol;
        p.summode = summode;
        planner_tables(&p);
        planner_sep_tables(&p);
        std::printf("{");
        put("krev", p.g.krev);
        std::printf("\"tables\": [");
        const int v0[3] = {kTileSep32, kTileSep32W, kTileSep16};
        for (int t = 0; t < 3; ++t) {
            std::printf("%s{", t ? ", " : "");
            put("line", p.sep_line_max[t]);
            put("mixed", p.sep_mixed_max[t]);
            put("rest", p.sep_rest_max[t]);
            put("off", p.sep_off_max[t]);
            put("fourth", p.sep_fourth_max[t]);
            put("du", p.du_max[v0[t]]);
            put("dR", p.dR_max[v0[t]], true);
            std::printf("}");
        }
        std::printf("], \"brute\": [");
        for (int t = 0; t < 3; ++t) {
            const Brute b = brute(p.g, tile_sep_rows(v0[t]), tile_sep_cols(v0[t]));
            std::printf("%s{", t ? ", " : "");
            put("line", b.line);
            put("mixed", b.mixed);
            put("rest", b.rest);
            put("off", b.off);
            put("fourth", b.fourth);
            put("du", b.du);
            put("dR", b.dR);
            put("series", b.series, true);
            std::printf("}");
        }
        std::printf("], \"extents\": [");
        for (size_t i = 0; i < rhos.size(); ++i) {
            std::printf("%s{", i ? ", " : "");
            for (int v = kTileSep32; v < kNumTilesAll; ++v) {
                put(("bound" + std::to_string(v)).c_str(), plan_bound(&p, v, rhos[i]));
                put(("trunc" + std::to_string(v)).c_str(), sep_trunc(&p, v, rhos[i]));
            }
            put("adjoint32", adjoint_sep_bound(&p, kTileSep32V, rhos[i]));
            put("adjoint16", adjoint_sep_bound(&p, kTileSep16Q, rhos[i]));
            std::printf("\"side\": %d, \"eligible\": [", adjoint_sep_side(&p, rhos[i]));
            const std::vector<int> ok = eligible_sep_tiles(&p, rhos[i]);
            for (size_t j = 0; j < ok.size(); ++j) std::printf(j ? ", %d" : "%d", ok[j]);
            std::printf("]}");
        }
        std::printf("], \"option\": [");
        for (int v = 0; v <= kNumTilesAll; ++v)
            std::printf("%s%d", v ? ", " : "", check_option(IDISIM_OPT_TILE, v, kNumTilesAll, &msg));
        std::printf("]}\n");
        std::fflush(stdout);
    }
    return 0;
}
