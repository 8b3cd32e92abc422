// CPU model of what a build's plan leaves room for, test infrastructure only (built and called by
// tests/plan_model.py): the library's own plan (dynamis_amd/csrc/dg_plan.hpp, host code without a
// GPU call), and the row words that the count pass makes of given atoms.  The model sweeps every
// target's stencil rows as search_kernel<0, 1 / 2> does (lower-triangular cells: rows trimmed to
// the cutoff, quarter-bin ends, pieces of at most 28 candidates that leave the target itself out,
// words of 20 mask bits), in 64 bits: it counts words and region-map entries, not edges.
#include <utility>
#include <vector>

namespace dg {
constexpr double kSelfThr = (double)1e-8f;
}
#include "../dynamis_amd/csrc/dg_plan.hpp"

using dg::Plan;

namespace {
constexpr int kWordBits = 20, kRowMax = 28;

bool make(Plan& p, const double* cell, const uint8_t* pbc, double r, int64_t n, int64_t nt, int f64)
{
    p = Plan();
    p.n = n;
    p.subset = nt >= 0;
    p.nt = nt >= 0 ? nt : n;
    p.f64 = f64;
    if (dg::plan_geometry(p, cell, pbc, r)) return false;
    dg::plan_grid(p);
    dg::plan_layout(p);
    return true;
}

int wrap(int x, int nb, bool periodic, bool* in)
{
    if (!periodic) {
        *in = x >= 0 && x < nb;
        return x;
    }
    *in = true;
    const int m = x % nb;
    return m < 0 ? m + nb : m;
}
}  // namespace

// out: nb[3], P[3], T[3], ntl[3], R[3], Kw, nrow, mapcap, ws_bytes, all-pairs, ws_bytes with the
// least lists, offset of the targets' word counts, pools of the map
extern "C" int plan_numbers(const double* cell, const uint8_t* pbc, double r, int64_t n, int64_t nt, int f64,
                            int64_t* out)
{
    Plan p;
    if (!make(p, cell, pbc, r, n, nt, f64)) return 1;
    for (int d = 0; d < 3; ++d) {
        out[d] = p.nb[d];
        out[3 + d] = p.P[d];
        out[6 + d] = p.T[d];
        out[9 + d] = p.ntl[d];
        out[12 + d] = p.R[d];
    }
    out[15] = p.Kw;
    out[16] = p.nrow;
    out[17] = p.mapcap;
    out[18] = (int64_t)p.ws_bytes;
    out[19] = p.brute;
    out[21] = (int64_t)p.o_nw;
    out[22] = p.npools;
    dg::plan_layout_lists(p, 2 * (size_t)p.K * (size_t)p.nrow);
    out[20] = (int64_t)p.ws_bytes;
    return 0;
}

// Row words of every target (all atoms), words[i], and the region-map entries of all tiles: their
// sum, and what each pool is asked for first, pools[64] (a tile asks pool ord mod npools, ord its
// place in the output: see tile_rank_kernel, xcd_tile_rank).
// pos: [n, 3]; the cell lower-triangular with a positive diagonal.
extern "C" int64_t count_words(const double* cell, const uint8_t* pbc, double r, int64_t n, const double* pos,
                               int f64, int32_t* words, int64_t* pools)
{
    Plan p;
    if (!make(p, cell, pbc, r, n, -1, f64) || p.brute) return -1;
    const int* nb = p.nb;
    struct Atom {
        double key;  // place along a in its bin, [0, 1)
        int id;
    };
    std::vector<std::vector<Atom>> bins((size_t)nb[0] * nb[1] * nb[2]);
    std::vector<int> bin(3 * n);
    std::vector<double> frac(3 * n);  // place in the bin, [0, 1)
    for (int64_t i = 0; i < n; ++i) {
        for (int d = 0; d < 3; ++d) {
            double f = 0;
            for (int c = 0; c < 3; ++c) f += pos[3 * i + c] * p.Cinv[3 * c + d];
            f = (f - floor(f)) * nb[d];
            const int b = std::min((int)f, nb[d] - 1);
            bin[3 * i + d] = b;
            frac[3 * i + d] = f - b;
        }
        bins[bin[3 * i] + (size_t)nb[0] * (bin[3 * i + 1] + (size_t)nb[1] * bin[3 * i + 2])].push_back(
            {frac[3 * i], (int)i});
    }
    for (auto& b : bins) std::sort(b.begin(), b.end(), [](const Atom& x, const Atom& y) { return x.key < y.key; });
    auto bin_at = [&](int x, int y, int z, bool* in) -> const std::vector<Atom>* {
        bool ix, iy, iz;
        x = wrap(x, nb[0], p.pbc[0], &ix);
        y = wrap(y, nb[1], p.pbc[1], &iy);
        z = wrap(z, nb[2], p.pbc[2], &iz);
        *in = ix && iy && iz;
        return *in ? &bins[x + (size_t)nb[0] * (y + (size_t)nb[1] * z)] : nullptr;
    };
    // tiles: entries of their regions, and whether the map and quarter-bin ends apply
    int64_t entries = 0;
    std::vector<int> region(p.ntiles);
    std::vector<int64_t> asks(p.ntiles);
    std::vector<std::pair<int64_t, int64_t>> order(p.ntiles);  // Morton code, tile
    for (int64_t t = 0; t < p.ntiles; ++t) {
        const int g[3] = {(int)(t % p.ntl[0]) * p.T[0], (int)(t / p.ntl[0] % p.ntl[1]) * p.T[1],
                          (int)(t / ((int64_t)p.ntl[0] * p.ntl[1])) * p.T[2]};
        int64_t total = 0, targets = 0;
        for (int z = 0; z < p.R[2]; ++z)
            for (int y = 0; y < p.R[1]; ++y)
                for (int x = 0; x < p.R[0]; ++x) {
                    bool in;
                    const auto* b = bin_at(g[0] - p.P[0] + x, g[1] - p.P[1] + y, g[2] - p.P[2] + z, &in);
                    if (in) total += (int64_t)b->size();
                }
        for (int z = g[2]; z < std::min(g[2] + p.T[2], nb[2]); ++z)
            for (int y = g[1]; y < std::min(g[1] + p.T[1], nb[1]); ++y)
                for (int x = g[0]; x < std::min(g[0] + p.T[0], nb[0]); ++x)
                    targets += (int64_t)bins[x + (size_t)nb[0] * (y + (size_t)nb[1] * z)].size();
        region[t] = (int)std::min<int64_t>(total, 1 << 30);
        asks[t] = targets > 0 && total <= 2 * dg::kCap ? total : 0;
        entries += asks[t];
        for (int k = 0, at = 0; k < 11; ++k)
            for (int d = 0; d < 3; ++d)
                if (k < p.mb[d]) {
                    const int64_t x = d == 0 ? t % p.ntl[0] : d == 1 ? t / p.ntl[0] % p.ntl[1] : t / ((int64_t)p.ntl[0] * p.ntl[1]);
                    order[t].first |= (x >> k & 1) << at++;
                }
        order[t].second = t;
    }
    std::sort(order.begin(), order.end());
    constexpr int64_t kRun = 16;
    for (int k = 0; k < 64; ++k) pools[k] = 0;
    for (int64_t b = 0, full = p.ntiles / (8 * kRun) * (8 * kRun); b < p.ntiles; ++b) {
        const int64_t j = b >> 3, rank = b < full ? ((j / kRun) * 8 + (b & 7)) * kRun + j % kRun : b;
        pools[b % p.npools] += asks[order[rank].second];
    }
    const double hax = p.C[0] / nb[0], hbx = p.C[3] / nb[1], hby = p.C[4] / nb[1], hcx = p.C[6] / nb[2],
                 hcy = p.C[7] / nb[2], hcz = p.C[8] / nb[2];
    const double pm = 1e-4 * r + 1e-3, rprune2 = (r + 2 * pm) * (r + 2 * pm);
    std::vector<char> edge;
    for (int64_t i = 0; i < n; ++i) {
        const int* b = &bin[3 * i];
        const double* u = &frac[3 * i];
        const int64_t t = b[0] / p.T[0] + p.ntl[0] * (b[1] / p.T[1] + (int64_t)p.ntl[1] * (b[2] / p.T[2]));
        const bool quarters = region[t] <= dg::kCap;
        int w = 0;
        auto piece = [&]() {
            const size_t m = edge.size(), low = m > kWordBits ? m - kWordBits : 0;
            bool a = false, c = false;
            for (size_t k = 0; k < m; ++k) (k < low ? a : c) |= edge[k] != 0;
            w += (int)a + (int)c;
            edge.clear();
        };
        for (int oz = -p.P[2]; oz <= p.P[2]; ++oz)
            for (int oy = -p.P[1]; oy <= p.P[1]; ++oy) {
                const double py = oy - u[1], pz = oz - u[2];
                const double zl = pz * hcz, zh = zl + hcz;
                const double yl = py * hby + std::min(pz * hcy, (pz + 1) * hcy),
                             yh = (py + 1) * hby + std::max(pz * hcy, (pz + 1) * hcy);
                const double gy = std::max(std::max({yl, -yh, 0.0}) - pm, 0.0),
                             gz = std::max(std::max({zl, -zh, 0.0}) - pm, 0.0);
                const double rem2 = rprune2 - gy * gy - gz * gz;
                if (rem2 < 0) continue;
                const double rem = sqrt(rem2);
                const double sl = std::min(py * hbx, (py + 1) * hbx) + std::min(pz * hcx, (pz + 1) * hcx),
                             sh = std::max(py * hbx, (py + 1) * hbx) + std::max(pz * hcx, (pz + 1) * hcx);
                const int ql = std::max((int)floor(4 * (u[0] + (-rem - sh) / hax)) + 4 * p.P[0], 0);
                const int qh = std::min((int)floor(4 * (u[0] + (rem - sl) / hax)) + 4 * p.P[0],
                                        4 * (2 * p.P[0] + 1) - 1);
                for (int x = ql >> 2; x <= qh >> 2; ++x) {
                    bool in;
                    const auto* list = bin_at(b[0] - p.P[0] + x, b[1] + oy, b[2] + oz, &in);
                    if (!in) continue;
                    for (const Atom& a : *list) {
                        const int q = 4 * x + std::min((int)(4 * a.key), 3);
                        if (quarters && (q < ql || q > qh)) continue;
                        if (a.id == i && x == p.P[0] && oy == 0 && oz == 0) {
                            piece();
                            continue;
                        }
                        const double* v = &frac[3 * (int64_t)a.id];
                        const double da = x - p.P[0] + v[0] - u[0], db = oy + v[1] - u[1], dc = oz + v[2] - u[2];
                        const double dx = da * hax + db * hbx + dc * hcx, dy = db * hby + dc * hcy, dz = dc * hcz;
                        edge.push_back(dx * dx + dy * dy + dz * dz <= r * r);
                        if (edge.size() == (size_t)kRowMax) piece();
                    }
                }
                piece();
            }
        words[i] = w;
    }
    return entries;
}
