// pzl_geometry.cpp -- search geometry and thresholds.
//
//   create_accelobs         accel_utils.c:1636-2037 (zmax/wmax rounding, r range,
//                           numindep, powcut, maxkernlen, fftlen, corr_uselen)
//   calc_fftlen             accel_utils.c:137-149
//   init_subharminfo        accel_utils.c:199-234 (per-harmonic zmax/wmax/grid)
//   rstep enumeration       accelsearch.c:183-188 (startr += rstep in double)
#include <algorithm>
#include <cmath>
#include <cstdarg>
#include <cstdio>
#include <cstring>

#include "pzl_math.h"
#include "pzl_plan.h"
#include "pzl_stats.h"

namespace pzl {

thread_local std::string g_err;

int fail(int code, const char *fmt, ...)
{
    char buf[512];
    va_list ap;
    va_start(ap, fmt);
    vsnprintf(buf, sizeof buf, fmt, ap);
    va_end(ap);
    g_err = buf;
    return code;
}

namespace {

int twon_to_index(int n)
{
    int x = 0;
    while (n > 1) {
        n >>= 1;
        x++;
    }
    return x;
}

int calc_fftlen(int numharm, int harmnum, int max_zfull, int max_wfull, int corr_uselen)
{
    const double hf = (double)harmnum / (double)numharm;
    const int bins_needed = (int)ceil(corr_uselen * hf) + 2;
    const int end_effects = 2 * PZL_NUMBETWEEN *
                            pzl_w_resp_halfwidth(pzl_calc_required_z(hf, max_zfull), pzl_calc_required_w(hf, max_wfull));
    return pzl_next_good_fftlen(bins_needed + end_effects);
}

}  // namespace

int compute_geometry(const PzlConfig &c, PzlGeometry &g, std::vector<PzlHarm> *harms_out,
                     std::vector<double> *startr_out)
{
    memset(&g, 0, sizeof g);
    int zmax = c.zmax, wmax = c.wmax;
    if (zmax < 0 || wmax < 0) return fail(PZL_ERR_ARG, "zmax and wmax must be >= 0");
    if (zmax % PZL_DZ) zmax = (zmax / PZL_DZ + 1) * PZL_DZ;
    const int nhm = c.numharm;
    if (nhm != 1 && nhm != 2 && nhm != 4 && nhm != 8 && nhm != 16 && nhm != 32)
        return fail(PZL_ERR_ARG, "'numharm' = %d must be a power-of-two (1..32)", c.numharm);
    if (c.numbins < 2 || c.N <= 0 || c.dt <= 0) return fail(PZL_ERR_ARG, "bad N/dt/numbins");
    g.N = (long long)c.N;
    g.numbins = c.numbins;
    g.lobin = c.lobin;
    g.numharmstages = twon_to_index(c.numharm) + 1;
    g.numz = (zmax / PZL_DZ) * 2 + 1;
    if (c.wmaxP) {
        if (wmax % PZL_DW) wmax = (wmax / PZL_DW + 1) * PZL_DW;
        g.whi = wmax;
        g.wlo = -wmax;
        g.numw = (wmax / PZL_DW) * 2 + 1;
        if (wmax == 0) g.numw = 0;
    } else {
        g.whi = g.wlo = 0.0;
        g.numw = 0;
        wmax = 0;
    }
    g.dt = c.dt;
    g.T = c.dt * c.N;
    g.rlo = c.floP ? floor(c.flo * g.T) : (c.rloP ? c.rlo : 1.0);
    if (g.rlo < g.lobin) g.rlo = (double)g.lobin;
    if (g.rlo > g.numbins - 1) return fail(PZL_ERR_ARG, "low frequency to search is above the highest bin");
    g.highestbin = g.numbins - 1;
    // The reference leaves rhi unset unless -fhi/-rhi is given; the default
    // command line always sets -fhi (accelsearch_cmd.c:59-62).
    g.rhi = (double)g.highestbin;
    if (c.fhiP || c.rhiP) {
        g.highestbin = c.fhiP ? (long long)ceil(c.fhi * g.T) : (long long)c.rhi;
        if (g.highestbin > g.numbins - 1) g.highestbin = g.numbins - 1;
        g.rhi = (double)g.highestbin;
        if (g.highestbin < g.rlo) return fail(PZL_ERR_ARG, "high frequency to search is below the low one");
    }
    g.zhi = zmax;
    g.zlo = -zmax;
    g.sigma = c.sigma;
    for (int ii = 0; ii < g.numharmstages; ii++) {
        const double dz = PZL_DZ, dw = PZL_DW;
        if (g.numz == 1 && g.numw == 0)
            g.numindep[ii] = (long long)((g.rhi - g.rlo) / (1 << ii));
        else if (g.numz > 1 && g.numw == 0)
            g.numindep[ii] = (long long)((g.rhi - g.rlo) * (g.numz + 1) * (dz / 6.95) / (1 << ii));
        else
            g.numindep[ii] =
                (long long)((g.rhi - g.rlo) * (g.numz + 1) * (dz / 6.95) * (g.numw + 1) * (dw / 44.2) / (1 << ii));
        g.powcut[ii] = (float)pzl_power_for_sigma(g.sigma, 1 << ii, (double)g.numindep[ii]);
    }
    g.maxkernlen = 2 * PZL_NUMBETWEEN * pzl_w_resp_halfwidth(g.zhi, g.whi);
    g.fftlen = pzl_fftlen_from_kernwidth(g.maxkernlen);
    if (g.fftlen < 2048) g.fftlen = 2048;
    g.corr_uselen = g.fftlen - g.maxkernlen;
    if (g.corr_uselen % PZL_RDR) g.corr_uselen = g.corr_uselen / PZL_RDR * PZL_RDR;
    if (g.corr_uselen <= 0 || g.corr_uselen > 65535) return fail(PZL_ERR_UNSUPPORTED, "corr_uselen out of range");

    std::vector<double> startr;
    const int rstep = (int)(g.corr_uselen * PZL_DR);
    for (double s = g.rlo; s + rstep < g.highestbin; s += rstep) startr.push_back(s);
    g.nrsteps = (long long)startr.size();

    // harmonics: fundamental, then stage order (accelsearch.c:199-211)
    std::vector<PzlHarm> harms;
    long long bank_off = 0, plane_off = 0, seg_off = 0;
    for (int stage = 0; stage < g.numharmstages; stage++) {
        const int numharm = 1 << stage;
        for (int harm = 1; harm < (stage ? numharm : 2); harm += 2) {
            PzlHarm H{};
            H.numharm = numharm;
            H.harmnum = harm;
            H.stage = stage;
            H.hf = (double)harm / (double)numharm;
            H.zmax = pzl_calc_required_z(H.hf, (int)g.zhi);
            H.wmax = pzl_calc_required_w(H.hf, (int)g.whi);
            H.numz = (H.zmax / PZL_DZ) * 2 + 1;
            H.numw = (H.wmax / PZL_DW) * 2 + 1;
            H.nrows = H.numz * H.numw;
            H.zlo = pzl_calc_required_z(H.hf, g.zlo);
            H.wlo = pzl_calc_required_w(H.hf, g.wlo);
            H.fftlen = (stage == 0) ? g.fftlen : calc_fftlen(numharm, harm, (int)g.zhi, (int)g.whi, g.corr_uselen);
            H.halfwidth = pzl_w_resp_halfwidth((double)-H.zmax, (double)-H.wmax);
            int maxrs = 0;
            for (double s : startr) {
                const PzlHarmR hr = pzl_harm_r(H.hf, stage == 0, s, s + rstep - PZL_DR, g.corr_uselen);
                maxrs = std::max(maxrs, hr.numrs);
            }
            if (startr.empty()) maxrs = g.corr_uselen;
            H.max_numrs = maxrs;
            H.rs_stride = (maxrs + 31) / 32 * 32;
            H.bank_off = bank_off;
            H.plane_off = plane_off;
            H.seg_off = seg_off;
            H.parent = (int)harms.size();
            H.ref_fftlen = H.fftlen;
            H.ref_halfwidth = H.halfwidth;
            bank_off += (long long)H.nrows * H.fftlen;
            plane_off += (long long)H.nrows * H.rs_stride;
            seg_off += H.fftlen / 2;
            harms.push_back(H);
        }
    }
    g.numharm_kernels = 0;
    for (auto &H : harms) g.numharm_kernels += H.nrows;
    g.bank_bytes = bank_off * 8;
    g.plane_bytes_per_rstep = plane_off * 4;
    if (harms_out) *harms_out = harms;
    if (startr_out) *startr_out = startr;
    return 0;
}

// A row's correlation length.  The reference gives every row of a harmonic the
// length of its widest kernel (calc_fftlen, accel_utils.c:137-149), but a
// kernel of half-width khw (z, w near 0: a third of the widest) only reaches
// 2 khw bins beyond each end of the wanted window, so a transform of numrs +
// 4 khw points gives the same outputs without wrap-around.  At zmax 200, wmax
// 300, 16 harmonics the points per rstep fall to 0.81 of the reference's
// lengths (with the lengths of the last correlation group).
bool compute_row_sets(const std::vector<PzlHarm> &harms, int corr_uselen, int (*has)(int n), std::vector<PzlHarm> *sets,
                      std::vector<int> *rows)
{
    sets->clear();
    rows->clear();
    long long bank_off = 0, seg_off = 0;
    // the half-widths of the whole (z, w) grid, of which every harmonic has a part
    // (a harmonic of 5000 rows has a few dozen different ones), and every held length
    int zmax = 0, wmax = 0, longest = 0;
    for (const PzlHarm &H : harms) {
        if (!has(H.fftlen)) return false;
        zmax = std::max(zmax, H.zmax);
        wmax = std::max(wmax, H.wmax);
        longest = std::max(longest, H.fftlen);
    }
    const int gz = zmax / PZL_DZ * 2 + 1, gw = wmax / PZL_DW * 2 + 1;
    std::vector<int> grid((size_t)gz * gw), held;
    for (int k = 0; k < gw; k++)
        for (int i = 0; i < gz; i++)
            grid[(size_t)k * gz + i] = pzl_w_resp_halfwidth(-zmax + i * PZL_DZ, -wmax + k * PZL_DW);
    for (int n = 2; n <= longest; n += 2)
        if (has(n)) held.push_back(n);
    std::vector<int> len_of;  // index in lens of each half-width's shortest length
    std::vector<int> row_len, count, widest;
    for (const PzlHarm &H : harms) {
        // held lengths up to the harmonic's own
        const std::vector<int> lens(held.begin(), std::upper_bound(held.begin(), held.end(), H.fftlen));
        // the widest window any start gives this harmonic (pzl_harm_r): its ends
        // round to half bins and then outwards to whole ones
        const double span = (corr_uselen / 2 - PZL_DR) * H.hf + 0.5;
        const int window = H.stage == 0 ? corr_uselen : std::max(H.max_numrs, 2 * ((int)floor(span + 1.0) + 1));
        const int last = (int)lens.size() - 1;
        len_of.resize(H.halfwidth + 1);
        for (int khw = 0, k = 0; khw <= H.halfwidth; khw++) {
            while (k < last && lens[k] < window + 4 * khw) k++;
            len_of[khw] = k;
        }
        row_len.resize(H.nrows);  // index in lens of each row, rows and widest row of each length
        count.assign(lens.size(), 0);
        widest.assign(lens.size(), 0);
        int row = 0;
        for (int wi = 0; wi < H.numw; wi++) {
            const int *khws = &grid[(size_t)(wi + (wmax - H.wmax) / PZL_DW) * gz + (zmax - H.zmax) / PZL_DZ];
            for (int zi = 0; zi < H.numz; zi++, row++) {
                const int khw = khws[zi], k = khw <= H.halfwidth ? len_of[khw] : last;
                row_len[row] = k;
                count[k]++;
                widest[k] = std::max(widest[k], khw);
            }
        }
        int at = (int)rows->size();
        rows->resize(rows->size() + H.nrows);
        for (int k = last; k >= 0; k--) {
            if (count[k] == 0) continue;
            PzlHarm S = H;
            S.fftlen = lens[k];
            // the full length keeps the harmonic's own segment, whatever its rows reach
            S.halfwidth = lens[k] == H.fftlen ? H.halfwidth : widest[k];
            S.nrows = count[k];
            S.bank_off = bank_off;
            S.seg_off = seg_off;
            bank_off += (long long)S.nrows * S.fftlen;
            seg_off += S.fftlen / 2;
            sets->push_back(S);
            count[k] = at;  // where the length's rows go
            at += S.nrows;
        }
        for (row = 0; row < H.nrows; row++) (*rows)[count[row_len[row]]++] = row;
    }
    return true;
}

}  // namespace pzl
