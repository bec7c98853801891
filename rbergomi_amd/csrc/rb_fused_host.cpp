// rb_fused_host.cpp -- host planning and launching of the fused mixed-precision kernel.
//
// plan_fused_request builds, from one request's deduplicated layout: the per-H tables of
// Toeplitz A fragments (hi + lo, or FP32), the per-H tables P_j = (j - off)^(2H), the group exponent
// coefficients, the payoff groups (group, rho), the option list and the assignment of 32-row
// output blocks to the four waves of a workgroup (balanced triangular work).
// FusedBatch concatenates any number of such requests into one launch: one table of requests,
// one list of work items (up to 1024 paths of one request each, about 1024 items per request
// where its tiles allow, the last eighth of a very large request in items an eighth of the
// size) ordered by decreasing cost and handed out through an atomic counter,
// and one ordered reduction of every request's option sums.
// A request's results depend only on its own items, so they are bit-identical alone and in any
// batch.
#include "rb_fused_host.h"
#include "rb_fft_lds.h"
#include "rb_path64.h"

#include <algorithm>
#include <array>
#include <cfloat>
#include <cstdio>
#include <cmath>
#include <cstdlib>
#include <cstring>
#include <map>
#include <mutex>
#include <numeric>
#include <string>
#include <vector>

#include "rb_engine.h"
#include "rb_kernels.h"

namespace rb {

// ---------------------------------------------------------------- tile shape choice
// Path blocks of 32 per tile (the tile is 32 PB paths by Np steps; the four waves split into
// 4 / PB per path block).  Measured on MI355X (split FP16, Romano-Touzi, 205 options, M = 2^21):
// N = 96: 2.96 / 2.58 / 2.31 ms for PB = 1 / 2 / 4; N = 128: 3.04 / 2.72 / 4.39; N = 160: 3.72 /
// 3.20 / 5.39; N = 192: 3.91 / 3.33 / 6.16; N = 256: 4.27 / 6.63 / 7.29; N >= 320: PB = 1 best.
// The default follows that; autotune_fused replaces it per (Np, mode, estimator) by timing.
namespace {
std::mutex g_tune_mu;
std::map<std::array<int, 3>, int> g_tune;  // (Np, mode, mc) -> PB
std::once_flag g_tune_env;
}  // namespace

int fused_default_pb(int NB) { return NB == 1 ? 4 : NB == 2 ? 2 : NB == 3 ? 4 : NB <= 6 ? 2 : 1; }

int fused_pb_choice(int Np, int mode, int mc) {
    std::call_once(g_tune_env, [] {
        // a cache file written by tune_save, loaded once per process
        if (const char* path = std::getenv("RBERGOMI_TUNE_CACHE")) {
            std::string err;
            (void)tune_load(path, err);
        }
    });
    std::lock_guard<std::mutex> lock(g_tune_mu);
    const auto it = g_tune.find({Np, mode, mc});
    return it != g_tune.end() ? it->second : fused_default_pb(Np / 32);
}

void tune_set(int Np, int mode, int mc, int pb) {
    std::lock_guard<std::mutex> lock(g_tune_mu);
    g_tune[{Np, mode, mc}] = pb;
}

void tune_clear() {
    std::lock_guard<std::mutex> lock(g_tune_mu);
    g_tune.clear();
}

// text file, one line per entry: "Np mode mc pb"
int tune_save(const char* path, std::string& err) {
    std::lock_guard<std::mutex> lock(g_tune_mu);
    FILE* f = std::fopen(path, "w");
    if (!f) {
        err = std::string("cannot write ") + path;
        return ST_ERR_ARG;
    }
    for (const auto& e : g_tune) std::fprintf(f, "%d %d %d %d\n", e.first[0], e.first[1], e.first[2], e.second);
    std::fclose(f);
    return ST_OK;
}

int tune_load(const char* path, std::string& err) {
    FILE* f = std::fopen(path, "r");
    if (!f) {
        err = std::string("cannot read ") + path;
        return ST_ERR_ARG;
    }
    std::vector<std::array<int, 4>> rows;
    int np, mode, mc, pb, line = 0;
    char buf[256];
    while (std::fgets(buf, sizeof buf, f)) {
        ++line;
        if (buf[0] == '#' || buf[0] == '\n') continue;
        if (std::sscanf(buf, "%d %d %d %d", &np, &mode, &mc, &pb) != 4 || np < 32 || np % 32 || mode < 0 ||
            mode > 2 || mc < 0 || mc > 1 || (pb != 1 && pb != 2 && pb != 4)) {
            std::fclose(f);
            err = std::string(path) + ": malformed entry on line " + std::to_string(line);
            return ST_ERR_ARG;
        }
        rows.push_back({np, mode, mc, pb});
    }
    std::fclose(f);
    std::lock_guard<std::mutex> lock(g_tune_mu);
    for (const auto& r : rows) g_tune[{r[0], r[1], r[2]}] = r[3];
    return ST_OK;
}

std::vector<std::array<int, 4>> tune_table() {
    std::lock_guard<std::mutex> lock(g_tune_mu);
    std::vector<std::array<int, 4>> t;
    for (const auto& e : g_tune) t.push_back({e.first[0], e.first[1], e.first[2], e.second});
    return t;
}

static uint16_t to_bf16_bits(float f) {
    uint32_t u;
    std::memcpy(&u, &f, 4);
    if ((u & 0x7F800000u) == 0x7F800000u) return uint16_t(u >> 16);  // inf / nan
    u += 0x7FFFu + ((u >> 16) & 1u);                                 // round to nearest even
    return uint16_t(u >> 16);
}
static float from_bf16_bits(uint16_t b) {
    const uint32_t u = uint32_t(b) << 16;
    float f;
    std::memcpy(&f, &u, 4);
    return f;
}

// hi + lo split of x in the operand type of the mode; returns the raw 16-bit patterns
static void split16(double x, int mode, uint16_t& hi, uint16_t& lo) {
    if (mode == 0) {
        const _Float16 h = (_Float16)(float)x;
        const _Float16 l = (_Float16)(float)(x - (double)(float)h);
        std::memcpy(&hi, &h, 2);
        std::memcpy(&lo, &l, 2);
    } else {
        hi = to_bf16_bits((float)x);
        lo = to_bf16_bits((float)(x - (double)from_bf16_bits(hi)));
    }
}

// Units, groups (sorted by unit), payoff groups (group, rho) and options (sorted by unit) of a
// request for the fused kernels, with the per-unit tables P_j = (j - off)^(2H) of Np entries,
// P_j at index j - pshift (1 <= j < N).  pgmax: payoff groups held at once; gmax: most groups of
// one unit.
void fused_tables(const Request& req, const Layout& lay, int Np, int frag_stride, int pshift, FusedHostReq& out,
                  int& pgmax, int& gmax) {
    const int nu = int(lay.units.size());
    out.fu.assign(nu, FusedUnit());
    out.fg.clear();
    out.fpg.clear();
    out.fo.clear();
    out.ptab.assign(size_t(nu) * Np, 0.f);  // Np = 0: no row tables
    const double log2e = 1.4426950408889634;
    const double off = req.comp == COMP_EXACT ? 0.0 : 1.0;
    pgmax = 1;
    gmax = 1;
    for (int u = 0; u < nu; ++u) {
        FusedUnit& U = out.fu[u];
        const double H = lay.units[u].H;
        U.b = float(lay.units[u].b);
        U.sc = float(lay.units[u].sc);
        U.frag_off = u * frag_stride;
        U.p_off = u * Np;
        for (int j = 1; Np > 0 && j < req.N; ++j)
            out.ptab[size_t(u) * Np + j - pshift] = float(std::pow(double(j) - off, 2.0 * H));
        U.g_begin = int(out.fg.size());
        U.pg_begin = int(out.fpg.size());
        U.o_begin = int(out.fo.size());
        for (size_t g = 0; g < lay.groups.size(); ++g) {
            const Group& G = lay.groups[g];
            if (G.unit != u) continue;
            FusedGroup F;
            F.c1 = float(0.5 * G.eta * G.TH * log2e);
            // at least FLT_MIN: the kernels zero a step's term by P = +inf (al P = +inf)
            F.al = std::max(float(0.25 * G.eta * G.eta * std::pow(G.dt, 2.0 * H) * log2e), FLT_MIN);
            F.be = float(-0.5 * std::log(G.xi) * log2e);
            F.xi = G.xi;
            F.sxi = std::sqrt(G.xi);
            F.dt = G.dt;
            F.sdt = G.sdt;
            F.pg_begin = int(out.fpg.size());
            F.o_begin = int(out.fo.size());
            const int fgi = int(out.fg.size());
            for (size_t I = 0; I < lay.options.size(); ++I) {
                const Option& o = lay.options[I];
                if (o.group != int(g)) continue;
                int pg = -1;
                for (int q = F.pg_begin; q < int(out.fpg.size()); ++q)
                    if (out.fpg[q].rho == o.rho) pg = q;
                if (pg < 0) {
                    pg = int(out.fpg.size());
                    out.fpg.push_back(FusedPG{fgi, 0, o.rho});
                }
                out.fo.push_back(FusedOption{pg, int(I), o.K, o.lnK});
            }
            F.pg_end = int(out.fpg.size());
            F.o_end = int(out.fo.size());
            out.fg.push_back(F);
        }
        U.g_end = int(out.fg.size());
        U.pg_end = int(out.fpg.size());
        U.o_end = int(out.fo.size());
        // payoff groups held at once: those of one pass (at most FUSED_GREG groups), so every
        // window of FUSED_GREG groups
        for (int g0 = U.g_begin; g0 < U.g_end; ++g0) {
            const int g1 = std::min(U.g_end, g0 + FUSED_GREG) - 1;
            pgmax = std::max(pgmax, out.fg[g1].pg_end - out.fg[g0].pg_begin);
        }
        gmax = std::max(gmax, U.g_end - U.g_begin);
    }
}

int plan_fused_request(const Request& req, const Layout& lay, int mode, FusedHostReq& out,
                       std::string& err, int pb, size_t bytes) {
    const int N = req.N;
    const int Np = (N + 31) / 32 * 32;
    if (Np > 1024) {
        err = "the split-precision kernel covers N <= 1024";
        return ST_ERR_LIMIT;
    }
    FusedReq& a = out.r;
    std::memset(&a, 0, sizeof(a));
    a.N = N;
    a.Np = Np;
    a.NK = Np / 16;
    a.chunk_u4 = fused_chunk_u4(mode);
    const int NB = Np / 32;
    // path blocks of 32 per tile: given, else the tuned or default choice for this shape
    a.PB = pb > 0 ? pb : fused_pb_choice(Np, mode, req.method == METHOD_MC ? 1 : 0);
    if (a.PB != 1 && a.PB != 2 && a.PB != 4) {
        err = "path blocks per tile must be 1, 2 or 4";
        return ST_ERR_ARG;
    }
    a.TP = 32 * a.PB;
    a.log2TP = a.PB == 1 ? 5 : (a.PB == 2 ? 6 : 7);
    // ---- waves: 4 / PB per path block; a block's output row blocks (cost rb + 1) go to its
    //      waves by longest-processing-time first
    std::vector<std::vector<int>> wrb(4);
    const int wpb = 4 / a.PB;
    for (int b = 0; b < a.PB; ++b) {
        std::vector<long> load(wpb, 0);
        for (int rb = NB - 1; rb >= 0; --rb) {
            const int w = int(std::min_element(load.begin(), load.end()) - load.begin());
            wrb[b * wpb + w].push_back(rb);
            load[w] += rb + 1;
        }
    }
    for (int w = 0; w < 4; ++w) a.wave_pb[w] = wrb[w].empty() ? -1 : w / wpb;
    size_t upw = 1;
    for (auto& v : wrb) upw = std::max(upw, v.size());
    if (upw > size_t(FUSED_MAX_UPW)) {
        err = "too many row blocks per wave for " + std::to_string(a.PB) + " path blocks per tile";
        return ST_ERR_LIMIT;
    }
    out.upw = upw <= 1 ? 1 : upw <= 2 ? 2 : upw <= 4 ? 4 : 8;
    for (int w = 0; w < 4; ++w) {
        // row blocks of a wave in decreasing order (the GEMM phases rely on it)
        std::sort(wrb[w].begin(), wrb[w].end(), [](int x, int y) { return x > y; });
        a.wave_nu[w] = int(wrb[w].size());
        for (int s = 0; s < FUSED_MAX_UPW; ++s) a.wave_rb[w][s] = s < int(wrb[w].size()) ? wrb[w][s] : -1;
    }
    int pgmax = 1, gmax = 1;
    // the GEMM kernel reads P_{j} at j - 1: a lane's four rows 8c + 4h + 0..3 are one aligned float4
    fused_tables(req, lay, Np, a.NK * 128, 1, out, pgmax, gmax);
    const int nu = int(lay.units.size());
    // rows j >= N of the last row block: P = +inf at index j - 1 and al >= FLT_MIN, so the
    // integrand exp2(c1 x - al P - be) is exactly 0 there (the kernel does not test rows)
    for (int u = 0; u < nu; ++u)
        for (int i = std::max(N - 1, 0); i < Np; ++i) out.ptab[size_t(u) * Np + i] = INFINITY;
    // the kernel reads each group's row terms al P_j + be (Np per group, the unit's groups in
    // order from p_off): one FP32 multiply-add rounded once, as the device's fmaf would give,
    // taken out of the kernel's (row, group) loop.  al P = +inf stays +inf.
    {
        std::vector<float> q;
        q.reserve(out.fg.size() * size_t(Np));
        for (int u = 0; u < nu; ++u) {
            FusedUnit& U = out.fu[u];
            const float* P = &out.ptab[size_t(u) * Np];
            U.p_off = int(q.size());
            for (int g = U.g_begin; g < U.g_end; ++g)
                for (int i = 0; i < Np; ++i) q.push_back(std::fmaf(out.fg[g].al, P[i], out.fg[g].be));
        }
        out.ptab.swap(q);
    }
    // ---- A fragments: entry (d, lane, slot j) = G[d + m - 8h - j], G[0] = a, G[t>0] = Gamma_t
    //      (0 outside [0, N)).  The table holds each G[t] about 64 times, so the operand split
    //      is computed once per t and the entries copied from it.
    out.frag.assign(size_t(nu) * a.NK * 128, uint4());
    std::vector<uint16_t> ghi(N), glo(N);
    std::vector<float> gf(N);
    for (int u = 0; u < nu; ++u) {
        const double* gam = &lay.gamma[size_t(u) * N];
        for (int t = 0; t < N; ++t) {
            const double g = t == 0 ? lay.units[u].a : gam[t];
            if (mode == 2)
                gf[t] = float(g);
            else
                split16(g, mode, ghi[t], glo[t]);
        }
        for (int f = 0; f < a.NK; ++f) {
            const int d = 16 * f - 16;
            uint4* e = &out.frag[(size_t(u) * a.NK + f) * 128];
            for (int lane = 0; lane < 64; ++lane) {
                const int m = lane & 31, hh = lane >> 5;
                uint16_t hi[8], lo[8];
                float g32[8];
                for (int j = 0; j < 8; ++j) {
                    const int t = d + m - 8 * hh - j;
                    const bool in = t >= 0 && t < N;
                    hi[j] = in ? ghi[t] : 0;
                    lo[j] = in ? glo[t] : 0;
                    g32[j] = in ? gf[t] : 0.0f;
                }
                if (mode == 2) {  // FP32 operands: slots 0..3, then 4..7
                    std::memcpy(&e[lane], g32, 16);
                    std::memcpy(&e[64 + lane], g32 + 4, 16);
                } else {
                    std::memcpy(&e[lane], hi, 16);
                    std::memcpy(&e[64 + lane], lo, 16);
                }
            }
        }
    }
    a.nunits = nu;
    a.pgmax = pgmax;
    a.out_size = int(lay.options.size());
    a.acc_in_lds = a.out_size > FUSED_MAX_REG_OPTS ? 1 : 0;
    // lanes per option in the payoff stage: the largest power of two S <= 32 with S*options <= 256
    a.log2slices = 0;
    while (!a.acc_in_lds && a.log2slices < 5 && (a.out_size << (a.log2slices + 1)) <= 256) ++a.log2slices;
    // with one lane per option (129 to 256 options) the lanes left over go to the first options,
    // two lanes each, in whole waves (32 options a wave), so that no wave prices with most of its
    // lanes idle: 205 options take 32 lane pairs and 173 single lanes
    a.pay2 = !a.acc_in_lds && a.log2slices == 0 ? std::min(a.out_size, (256 - a.out_size) / 32 * 32) : 0;
    a.mc = req.method == METHOD_MC ? 1 : 0;
    a.M = req.M;
    a.ntiles = (req.M + a.TP - 1) / a.TP;
    // Work items of at most 1024 paths, and 1024 or more per request where its tiles allow: three
    // workgroups on each CU take 768, and a request of some hundred items would leave a launch
    // of its own with one or two each (N = 512, M = 2^18, five maturities: 256 items 0.72 ms, 1024 items
    // 0.43, 2048 items 0.46; N = 365, M = 3e5, plain MC, BF16: 293 items 0.72, 938 items 0.49), but
    // beyond 256 items no less than 2^14 path steps each (a call of N = 64, M = 2^16: 256 items 0.108 ms, 512
    // items 0.118).  The item size depends on the request only, so its sums are added in the same order
    // alone and in any batch; only where the partial sums of so many items (16 bytes per option and
    // item) bring its memory above `bytes`, 256 items have to do.
    auto items = [&](long most) {
        const long steps = long(N) * a.TP;
        const long least = std::min((a.ntiles + 255) / 256, ((1L << 14) + steps - 1) / steps);
        a.tiles_per_item = int(std::max<long>(1, std::min<long>(1024 / a.TP, std::max((a.ntiles + most - 1) / most, least))));
        a.nitems = (a.ntiles + a.tiles_per_item - 1) / a.tiles_per_item;
        a.items_big = a.nitems;
        a.tiles_small = a.tiles_per_item;
        // a request of 4096 or more items is in practice a launch of its own: its last eighth of
        // tiles goes in items of an eighth of the size, handed out last (cheapest first in the
        // batch's order), so the workgroups finish together rather than one large item apart
        // (N = 512, M = 2^22, Romano-Touzi: 7.05 -> 6.70 ms with every item of 256 paths; plain
        // Monte Carlo, with no data-dependent branch, was even without it)
        if (a.nitems >= 4096 && a.tiles_per_item >= 8) {
            a.tiles_small = a.tiles_per_item / 8;
            a.items_big = (a.ntiles - a.ntiles / 8) / a.tiles_per_item;
            const long rest = a.ntiles - a.items_big * a.tiles_per_item;
            a.nitems = a.items_big + (rest + a.tiles_small - 1) / a.tiles_small;
        }
    };
    a.key = philox_key(req.seed.data(), int(req.seed.size()));
    a.gchunk = std::min(gmax, FUSED_GREG);
    out.gmax = gmax;
    out.ivopts = lay.options;
    items(1024);
    if (FusedBatch::footprint({&out}) > bytes) items(256);
    // cost of one item (relative): RNG + integrals ~ N * groups, GEMM ~ N^2 / 64, payoffs ~ options
    out.item_cost = double(a.tiles_per_item * a.TP) *
                    (double(N) * (2.0 + 2.0 * a.mc + gmax) + double(Np) * Np / 64.0 * nu + 4.0 * a.out_size);
    return ST_OK;
}

#define RB_TRY(expr)                                                         \
    do {                                                                     \
        hipError_t e_ = (expr);                                              \
        if (e_ != hipSuccess) {                                              \
            err = std::string(#expr) + ": " + hipGetErrorString(e_);         \
            return e_ == hipErrorOutOfMemory ? ST_ERR_NOMEM : ST_ERR_DEVICE; \
        }                                                                    \
    } while (0)

template <class T>
static hipError_t alloc_async(T** p, size_t n, hipStream_t st) {
    return hipMallocAsync(reinterpret_cast<void**>(p), std::max<size_t>(n, 1) * sizeof(T), st);
}

// n elements of T from the arena (256-byte aligned), or a stream-ordered allocation without one
template <class T>
static hipError_t batch_alloc(DevArena* ar, T** p, size_t n, hipStream_t st) {
    if (!ar) return alloc_async(p, n, st);
    const size_t bytes = (std::max<size_t>(n, 1) * sizeof(T) + 255) & ~size_t(255);
    if (ar->used + bytes > ar->size) return hipErrorOutOfMemory;
    *p = reinterpret_cast<T*>(ar->base + ar->used);
    ar->used += bytes;
    return hipSuccess;
}

size_t fused_batch_lds(const std::vector<const FusedHostReq*>& reqs, size_t lds_cu, FusedBatchArgs* a, int* cap) {
    int bf = 0, wp = 0, pg = 0, ac = 0, ns = 2, upw = 1;
    for (const FusedHostReq* q : reqs) {
        const FusedReq& r = q->r;
        upw = std::max(upw, q->upw);
        ns = r.mc ? 3 : 2;
        bf = std::max(bf, r.PB * r.NK * r.chunk_u4);
        wp = std::max(wp, 4 * r.gchunk * 32 * ns);
        pg = std::max(pg, r.TP * r.pgmax);
        ac = std::max(ac, r.acc_in_lds ? 2 * r.out_size : 0);
    }
    const size_t stat = sizeof(FusedReq) + 16;  // the kernel's static record and item index
    const size_t half = lds_cu / 2, third = lds_cu / 3;
    const size_t rest = size_t(bf) * 16 + size_t(pg) * sizeof(PathPG) + size_t(ac) * 8 + stat;
    int c_cap = 0;
    // chunks of half a pass's groups or more if that lets a third workgroup onto the CU (N = 512, FP16,
    // eight groups 2.09 -> 1.95 ms, N = 320, BF16, five groups 1.29 -> 1.20), of any size if it lets a second
    for (const size_t share : {third, half}) {
        if (share == third && upw > 4) continue;  // its registers do not fit three times
        if (rest + size_t(wp) * 8 <= share || c_cap > 0) break;
        const int c_min = share == third ? (wp / (4 * 32 * ns) + 1) / 2 : 1;
        for (int c = FUSED_GREG; c >= c_min && c_cap == 0; --c)
            if (rest + size_t(4 * c * 32 * ns) * 8 <= share) c_cap = c;
        if (c_cap > 0) {
            wp = 0;
            for (const FusedHostReq* q : reqs) wp = std::max(wp, 4 * std::min(q->r.gchunk, c_cap) * 32 * ns);
        }
    }
    if (a) {
        a->bf_u4 = bf;
        a->wpart_d = wp;
        a->pgd_n = pg;
        a->acc_d = ac;
    }
    if (cap) *cap = c_cap;
    return rest + size_t(wp) * 8;
}

bool fused_batch_accepts(const std::vector<const FusedHostReq*>& reqs, size_t lds_block, size_t lds_cu) {
    if (reqs.size() <= 1) return true;
    const size_t with = fused_batch_lds(reqs, lds_cu, nullptr, nullptr);
    if (with > lds_block) return false;
    if (with <= lds_cu / 2) return true;
    const std::vector<const FusedHostReq*> before(reqs.begin(), reqs.end() - 1);
    return fused_batch_lds(before, lds_cu, nullptr, nullptr) > lds_cu / 2;
}

std::vector<std::pair<int, int>> FusedBatch::split(const std::vector<const FusedHostReq*>& reqs, size_t lds_block,
                                                   size_t lds_cu, bool soft) {
    std::vector<std::pair<int, int>> runs;
    std::vector<const FusedHostReq*> cur;
    int begin = 0;
    for (int i = 0; i < int(reqs.size()); ++i) {
        cur.push_back(reqs[i]);
        const bool fits = soft ? fused_batch_accepts(cur, lds_block, lds_cu)
                               : cur.size() == 1 || fused_batch_lds(cur, lds_cu, nullptr, nullptr) <= lds_block;
        if (!fits) {
            runs.push_back({begin, i});
            begin = i;
            cur.assign(1, reqs[i]);
        }
    }
    if (!reqs.empty()) runs.push_back({begin, int(reqs.size())});
    return runs;
}

FusedBatch::~FusedBatch() { release(); }

void FusedBatch::release() {
    // the stream reads and writes the pinned blocks until it has passed the launch
    if (up.data() || out.data()) (void)hipStreamSynchronize(stream);
    up.release();
    out.release();
    if (d_block && !arena) (void)hipFreeAsync(d_block, stream);
    d_block = nullptr;
    d_reqs = nullptr;
    d_fu = nullptr;
    d_fg = nullptr;
    d_fpg = nullptr;
    d_fo = nullptr;
    d_frag = nullptr;
    d_ptab = nullptr;
    d_item_req = nullptr;
    d_item_local = nullptr;
    d_counter = nullptr;
    d_partial = nullptr;
    d_price = d_stat = d_iv = nullptr;
    d_ivopts = nullptr;
    d_row_off = d_row_n = d_row_M = nullptr;
}

size_t FusedBatch::footprint(const std::vector<const FusedHostReq*>& reqs) {
    size_t b = 0;
    for (const FusedHostReq* q : reqs) {
        b += q->frag.size() * 16 + q->ptab.size() * 4 + q->fo.size() * sizeof(FusedOption) +
             q->fg.size() * sizeof(FusedGroup) + q->fpg.size() * sizeof(FusedPG) +
             q->fu.size() * sizeof(FusedUnit) + sizeof(FusedReq);
        b += size_t(q->r.out_size) * q->r.nitems * 16 + size_t(q->r.nitems) * 8;
        b += size_t(q->r.out_size) * (3 * 8 + sizeof(Option) + 24);
    }
    return b;
}

// copies v into an existing device buffer of v.size() elements
template <class T>
static hipError_t batch_refill(T* p, const std::vector<T>& v, hipStream_t st) {
    if (v.empty()) return hipSuccess;
    return hipMemcpyAsync(p, v.data(), v.size() * sizeof(T), hipMemcpyHostToDevice, st);
}

int FusedBatch::build(const std::vector<const FusedHostReq*>& reqs, int mode_, int device,
                      hipStream_t st, std::string& err, bool refill, bool check_only) {
    if (refill && !d_reqs) {
        err = "no batch to refill";
        return ST_ERR_ARG;
    }
    if (!refill) release();
    // a refill that fails its check, or only checks, leaves the batch as it was
    struct Saved {
        FusedBatch& b;
        int mode, nreq, upw, greg, total_out;
        bool mc;
        hipStream_t stream;
        std::vector<long> out_off;
        FusedBatchArgs args;
        bool keep = false;
        ~Saved() {
            if (keep) return;
            b.mode = mode;
            b.nreq = nreq;
            b.upw = upw;
            b.greg = greg;
            b.total_out = total_out;
            b.mc = mc;
            b.stream = stream;
            b.out_off = out_off;
            b.args = args;
        }
    } saved{*this, mode, nreq, upw, greg, total_out, mc, stream, out_off, args};
    saved.keep = !refill;
    stream = st;
    mode = mode_;
    nreq = int(reqs.size());
    upw = 1;
    // concatenate the tables, fixing the offsets inside each request
    std::vector<FusedReq> R;
    std::vector<FusedUnit> fu;
    std::vector<FusedGroup> fg;
    std::vector<FusedPG> fpg;
    std::vector<FusedOption> fo;
    std::vector<uint4> frag;
    std::vector<float> ptab;
    std::vector<Option> ivo;
    std::vector<long> row_off, row_n, row_M;
    out_off.assign(nreq + 1, 0);
    long poff = 0;
    for (int q = 0; q < nreq; ++q) {
        const FusedHostReq& H = *reqs[q];
        FusedReq r = H.r;
        upw = std::max(upw, H.upw);
        const int u0 = int(fu.size()), g0 = int(fg.size()), pg0 = int(fpg.size()), o0 = int(fo.size());
        const int f0 = int(frag.size()), p0 = int(ptab.size());
        for (FusedUnit U : H.fu) {
            U.frag_off += f0;
            U.p_off += p0;
            U.g_begin += 0;
            fu.push_back(U);
        }
        for (const FusedGroup& G : H.fg) fg.push_back(G);
        for (FusedPG P : H.fpg) {
            P.group += 0;  // group indices are request-local
            fpg.push_back(P);
        }
        for (const FusedOption& O : H.fo) fo.push_back(O);
        frag.insert(frag.end(), H.frag.begin(), H.frag.end());
        ptab.insert(ptab.end(), H.ptab.begin(), H.ptab.end());
        // pointers are fixed after upload; keep the element offsets for now
        r.units = reinterpret_cast<const FusedUnit*>(size_t(u0));
        r.groups = reinterpret_cast<const FusedGroup*>(size_t(g0));
        r.pgs = reinterpret_cast<const FusedPG*>(size_t(pg0));
        r.opts = reinterpret_cast<const FusedOption*>(size_t(o0));
        r.partial = reinterpret_cast<double*>(size_t(poff));
        for (int I = 0; I < r.out_size; ++I) {
            row_off.push_back(poff + long(I) * r.nitems * 2);
            row_n.push_back(r.nitems);
            row_M.push_back(r.M);
        }
        poff += long(r.out_size) * r.nitems * 2;
        out_off[q + 1] = out_off[q] + r.out_size;
        ivo.insert(ivo.end(), H.ivopts.begin(), H.ivopts.end());
        if (q > 0 && r.mc != R[0].mc) {
            err = "a batch holds requests of one estimator (Romano-Touzi or plain Monte Carlo)";
            return ST_ERR_ARG;
        }
        R.push_back(r);
    }
    mc = nreq > 0 && R[0].mc != 0;
    {
        int gm = 1;
        for (int q = 0; q < nreq; ++q) gm = std::max(gm, reqs[q]->gmax);
        greg = fused_greg(gm);
    }
    total_out = int(out_off[nreq]);
    hipDeviceProp_t prop;
    RB_TRY(device_props(device, prop));
    if (!arena) keep_pool_cached(device);
    // Two or three workgroups per CU need at most half or a third of the CU's LDS each, the static request
    // record included; fused_batch_lds cuts the cross-wave partials' chunk of groups when that helps.
    const size_t lds_cu = size_t(prop.maxSharedMemoryPerMultiProcessor ? prop.maxSharedMemoryPerMultiProcessor
                                                                        : prop.sharedMemPerBlock);
    int cap = 0;
    const size_t lds_total = fused_batch_lds(reqs, lds_cu, &args, &cap);
    if (cap > 0)
        for (FusedReq& r : R) r.gchunk = std::min(r.gchunk, cap);
    if (lds_total > prop.sharedMemPerBlock) {
        err = "fused kernel needs " + std::to_string(lds_total) + " bytes of LDS (too many options or groups; "
              "a request that fits alone may not fit with others in one launch)";
        return ST_ERR_LIMIT;
    }
    // work items, most expensive first
    std::vector<std::pair<double, std::pair<int, int>>> items;
    for (int q = 0; q < nreq; ++q)
        for (long i = 0; i < R[q].nitems; ++i)
            items.push_back({i < R[q].items_big ? reqs[q]->item_cost
                                                : reqs[q]->item_cost * R[q].tiles_small / R[q].tiles_per_item,
                             {q, int(i)}});
    std::stable_sort(items.begin(), items.end(),
                     [](const std::pair<double, std::pair<int, int>>& x,
                        const std::pair<double, std::pair<int, int>>& y) { return x.first > y.first; });
    std::vector<int> item_req(items.size()), item_local(items.size());
    for (size_t i = 0; i < items.size(); ++i) {
        item_req[i] = items[i].second.first;
        item_local[i] = items[i].second.second;
    }
    args.total_items = long(items.size());
    const std::vector<size_t> shape = {fu.size(), fg.size(), fpg.size(), fo.size(), frag.size(), ptab.size(),
                                       ivo.size(), row_off.size(), item_req.size(), size_t(poff),
                                       size_t(total_out), size_t(mode_), size_t(upw), size_t(greg), size_t(mc),
                                       size_t(args.bf_u4), size_t(args.wpart_d), size_t(args.pgd_n),
                                       size_t(args.acc_d)};
    if (refill) {
        // new parameters of the same shapes into the same buffers: the request records keep their
        // pointers, so launches recorded in a graph stay valid
        if (shape != shape_) {
            err = "the new parameters change the batch's table layout (distinct H, maturities, rho, options "
                  "or tile shapes); build a new batch";
            return ST_ERR_ARG;
        }
        if (check_only) return ST_OK;
        saved.keep = true;
        RB_TRY(batch_refill(d_fu, fu, st));
        RB_TRY(batch_refill(d_fg, fg, st));
        RB_TRY(batch_refill(d_fpg, fpg, st));
        RB_TRY(batch_refill(d_fo, fo, st));
        RB_TRY(batch_refill(d_frag, frag, st));
        RB_TRY(batch_refill(d_ptab, ptab, st));
        RB_TRY(batch_refill(d_ivopts, ivo, st));
        RB_TRY(batch_refill(d_row_off, row_off, st));
        RB_TRY(batch_refill(d_row_n, row_n, st));
        RB_TRY(batch_refill(d_row_M, row_M, st));
        RB_TRY(batch_refill(d_item_req, item_req, st));
        RB_TRY(batch_refill(d_item_local, item_local, st));
        for (FusedReq& r : R) {
            r.units = d_fu + size_t(r.units);
            r.groups = d_fg + size_t(r.groups);
            r.pgs = d_fpg + size_t(r.pgs);
            r.opts = d_fo + size_t(r.opts);
            r.frag = d_frag;
            r.ptab = d_ptab;
            r.partial = d_partial + size_t(r.partial);
        }
        RB_TRY(batch_refill(d_reqs, R, st));
        RB_TRY(hipStreamSynchronize(st));
        return ST_OK;
    }
    shape_ = shape;
    // One device block: the tables, request records and item counter (one upload), then the
    // partial sums and the results price | iv | stat, adjacent so that one copy brings them back.
    // Pieces start on 256-byte boundaries.
    size_t off = 0;
    auto place = [&](size_t bytes) {
        const size_t o = off;
        off += (std::max<size_t>(bytes, 1) + 255) & ~size_t(255);
        return o;
    };
    const size_t o_fu = place(fu.size() * sizeof(FusedUnit)), o_fg = place(fg.size() * sizeof(FusedGroup)),
                 o_fpg = place(fpg.size() * sizeof(FusedPG)), o_fo = place(fo.size() * sizeof(FusedOption)),
                 o_frag = place(frag.size() * sizeof(uint4)), o_ptab = place(ptab.size() * sizeof(float)),
                 o_ivo = place(ivo.size() * sizeof(Option)), o_roff = place(row_off.size() * sizeof(long)),
                 o_rn = place(row_n.size() * sizeof(long)), o_rm = place(row_M.size() * sizeof(long)),
                 o_ireq = place(item_req.size() * sizeof(int)), o_iloc = place(item_local.size() * sizeof(int)),
                 o_reqs = place(R.size() * sizeof(FusedReq)), o_cnt = place(sizeof(int));
    const size_t up_bytes = off;
    const size_t res_bytes = std::max<size_t>(1, size_t(total_out) * 3 * sizeof(double));
    // results in the block where no pinned memory can be had
    double* host_out = to_host ? reinterpret_cast<double*>(out.reserve(res_bytes)) : nullptr;
    const size_t o_part = place(size_t(poff) * sizeof(double)), o_out = place(host_out ? 1 : res_bytes);
    RB_TRY(batch_alloc(arena, &d_block, off, st));
    d_fu = reinterpret_cast<FusedUnit*>(d_block + o_fu);
    d_fg = reinterpret_cast<FusedGroup*>(d_block + o_fg);
    d_fpg = reinterpret_cast<FusedPG*>(d_block + o_fpg);
    d_fo = reinterpret_cast<FusedOption*>(d_block + o_fo);
    d_frag = reinterpret_cast<uint4*>(d_block + o_frag);
    d_ptab = reinterpret_cast<float*>(d_block + o_ptab);
    d_ivopts = reinterpret_cast<Option*>(d_block + o_ivo);
    d_row_off = reinterpret_cast<long*>(d_block + o_roff);
    d_row_n = reinterpret_cast<long*>(d_block + o_rn);
    d_row_M = reinterpret_cast<long*>(d_block + o_rm);
    d_item_req = reinterpret_cast<int*>(d_block + o_ireq);
    d_item_local = reinterpret_cast<int*>(d_block + o_iloc);
    d_reqs = reinterpret_cast<FusedReq*>(d_block + o_reqs);
    d_counter = reinterpret_cast<int*>(d_block + o_cnt);
    counter_dirty = false;
    d_partial = reinterpret_cast<double*>(d_block + o_part);
    d_price = host_out ? host_out : reinterpret_cast<double*>(d_block + o_out);
    d_iv = d_price + total_out;
    d_stat = d_price + 2 * size_t(total_out);
    for (FusedReq& r : R) {
        r.units = d_fu + size_t(r.units);
        r.groups = d_fg + size_t(r.groups);
        r.pgs = d_fpg + size_t(r.pgs);
        r.opts = d_fo + size_t(r.opts);
        r.frag = d_frag;
        r.ptab = d_ptab;
        r.partial = d_partial + size_t(r.partial);
    }
    unsigned char* h = arena ? nullptr : up.reserve(up_bytes);
    const bool staged = h != nullptr;
    if (staged) {
        // packed into pinned memory: one copy, not waited for
        auto pack = [&](size_t o, const auto& v) {
            if (!v.empty()) std::memcpy(h + o, v.data(), v.size() * sizeof(v[0]));
        };
        pack(o_fu, fu);
        pack(o_fg, fg);
        pack(o_fpg, fpg);
        pack(o_fo, fo);
        pack(o_frag, frag);
        pack(o_ptab, ptab);
        pack(o_ivo, ivo);
        pack(o_roff, row_off);
        pack(o_rn, row_n);
        pack(o_rm, row_M);
        pack(o_ireq, item_req);
        pack(o_iloc, item_local);
        pack(o_reqs, R);
        std::memset(h + o_cnt, 0, sizeof(int));
        RB_TRY(hipMemcpyAsync(d_block, h, up_bytes, hipMemcpyHostToDevice, st));
    } else {
        // straight from the host tables (pageable memory: a packed copy would cost a host copy of
        // every table); the first launch zeroes the counter
        auto put = [&](size_t o, const auto& v) {
            return v.empty() ? hipSuccess
                             : hipMemcpyAsync(d_block + o, v.data(), v.size() * sizeof(v[0]), hipMemcpyHostToDevice, st);
        };
        RB_TRY(put(o_fu, fu));
        RB_TRY(put(o_fg, fg));
        RB_TRY(put(o_fpg, fpg));
        RB_TRY(put(o_fo, fo));
        RB_TRY(put(o_frag, frag));
        RB_TRY(put(o_ptab, ptab));
        RB_TRY(put(o_ivo, ivo));
        RB_TRY(put(o_roff, row_off));
        RB_TRY(put(o_rn, row_n));
        RB_TRY(put(o_rm, row_M));
        RB_TRY(put(o_ireq, item_req));
        RB_TRY(put(o_iloc, item_local));
        RB_TRY(put(o_reqs, R));
        counter_dirty = true;
    }
    args.reqs = d_reqs;
    args.item_req = d_item_req;
    args.item_local = d_item_local;
    args.counter = d_counter;
    // Three workgroups per CU where their LDS fits (and their registers: up to four row blocks per
    // wave).  Vector instructions of two waves per SIMD do not issue back to back: N = 512, M = 2^22, FP16,
    // five groups 6.51 -> 6.00 ms, M = 2^20, one group 1.24 -> 1.06, plain MC, two groups 1.13 -> 1.00,
    // N = 256, five groups 0.95 -> 0.81, 48 server requests 22.9 -> 20.6.  Where only two fit the
    // registers of three cost (N = 512, eight groups 2.08 -> 2.31, BF16, five groups 1.79 -> 1.93).
    args.per_cu = int(std::max<size_t>(1, std::min<size_t>(upw <= 4 ? 3 : 2, lds_cu / lds_total)));
    grid = int(std::min<long>(args.total_items, long(prop.multiProcessorCount) * args.per_cu));
    // pageable sources: the host tables die with this call
    if (!staged) RB_TRY(hipStreamSynchronize(st));
    return ST_OK;
}

int FusedBatch::launch(hipStream_t st, std::string& err, Plan* timing, hipEvent_t kbeg, hipEvent_t kend) {
    auto timed = [&](int id) { return timing ? timing->timed(id) : -1; };
    auto mark = [&](int slot) {
        if (timing) timing->mark(slot, nullptr, nullptr);
    };
    int s;
    // the upload and every complete launch leave the item counter at zero (the reduction resets
    // it); a launch that failed part-way may not have
    if (counter_dirty) RB_TRY(launch_zero_int(d_counter, 1, st));
    counter_dirty = true;
    if (kbeg) RB_TRY(hipEventRecord(kbeg, st));
    s = timed(K_FUSED);
    RB_TRY(launch_fused(mode, upw, mc, greg, args, grid, st));
    mark(s);
    if (kend) RB_TRY(hipEventRecord(kend, st));
    s = timed(K_REDUCE);
    RB_TRY(launch_reduce_iv(d_partial, ReduceRows{d_row_off, d_row_n, d_row_M, 0, 0}, d_ivopts, total_out, d_price,
                            d_stat, d_iv, d_counter, st));
    mark(s);
    counter_dirty = total_out < 1;
    return ST_OK;
}

hipError_t FusedBatch::fetch(int q, double* price, double* iv, double* stat) const {
    const long a = out_off[q], b = out_off[q + 1];
    const bool pinned = out.data() != nullptr;
    hipError_t e = fetch_results(price, d_price + a, size_t(b - a), pinned);
    if (!e) e = fetch_results(iv, d_iv + a, size_t(b - a), pinned);
    if (!e) e = fetch_results(stat, d_stat + a, size_t(b - a), pinned);
    return e;
}

int FusedBatch::results(int q, double* price, double* iv, double* stat, hipStream_t st,
                        std::string& err) {
    const size_t n = size_t(out_off[q + 1] - out_off[q]) * sizeof(double);
    if (price) RB_TRY(hipMemcpyAsync(price, d_price + out_off[q], n, hipMemcpyDeviceToHost, st));
    if (iv) RB_TRY(hipMemcpyAsync(iv, d_iv + out_off[q], n, hipMemcpyDeviceToHost, st));
    if (stat) RB_TRY(hipMemcpyAsync(stat, d_stat + out_off[q], n, hipMemcpyDeviceToHost, st));
    return ST_OK;
}

// ---------------------------------------------------------------- long paths: FFT kernel
FftFused::~FftFused() { release(); }

void FftFused::release() {
    // the stream reads and writes the pinned blocks until it has passed the launch
    if (up.data() || out.data()) (void)hipStreamSynchronize(stream);
    up.release();
    out.release();
    if (d_block) (void)hipFreeAsync(d_block, stream);
    d_block = nullptr;
    d_payjobs = nullptr;
    d_payopts = nullptr;
    d_partial = nullptr;
    d_price = d_stat = d_iv = nullptr;
    d_ivopts = nullptr;
}

// The request sizes of the long-path kernel, a limit of the interface: 16 bytes an option and 64 a (group, rho)
// of the H with the most, beside 8.25 a point of the transform, in 160 KiB less 1.5 (from the time when one
// workgroup's LDS held them; nothing in the present kernel needs it).
static int fft_request_fits(const FusedHostReq& tabs, int N, int nopt, std::string& err) {
    int log2L = 10;
    while ((1 << log2L) < 2 * N - 1) ++log2L;
    const long L = 1L << log2L, room = 160 * 1024 - 1536 - 8 * (L + L / 32);
    int pgu = 1;
    for (const FusedUnit& U : tabs.fu) pgu = std::max(pgu, U.pg_end - U.pg_begin);
    if (64L * pgu + 16L * nopt <= room) return ST_OK;
    err = "too many options for a request of N = " + std::to_string(N) + " on the long-path kernel: 16 for each of its " +
          std::to_string(nopt) + " options and 64 for each of the " + std::to_string(pgu) +
          " (maturity, eta, rho) of its largest H may come to " + std::to_string(room);
    return ST_ERR_LIMIT;
}

// Sizes of a request: paths per chunk, so that a chunk's integrals take about 4 MiB, and the block's
// pieces in bytes
struct FftSizes {
    int ppt;
    long nblk, chunk;
    size_t ptab, ghat, tw, gamma, tw64, ints, partial;
    FftSizes(const Request& req, int nunits, int ngroups, int nopt) {
        const int N = req.N, ns = req.method == METHOD_MC ? 3 : 2;
        const size_t L = size_t(1) << fused_fft_log2(N);
        ppt = payoff_paths_per_thread(req.M, nopt);
        const long pblk = 256L * ppt;
        nblk = (req.M + pblk - 1) / pblk;
        chunk = std::max<long>(1, (long(4) << 20) / (8L * ns * ngroups) / pblk) * pblk;
        chunk = std::min(chunk, nblk * pblk);
        ptab = nunits * (L / 2) * sizeof(float);
        ghat = nunits * L * sizeof(float2);
        tw = fused_fft_table(fused_fft_log2(N)) * sizeof(float2);
        gamma = N <= 4096 ? nunits * (L / 2) * sizeof(double) : 0;
        tw64 = N <= 4096 ? path64_fft_table(int(L / 2)) * sizeof(double2) : 0;
        ints = size_t(ngroups) * chunk * ns * sizeof(double);
        partial = size_t(nopt) * nblk * 2 * sizeof(double);
    }
    size_t total() const { return ptab + ghat + tw + gamma + tw64 + ints + partial; }
};

int FftFused::plan(const Request& req, const Layout& lay, size_t& footprint, std::string& err) {
    const int N = req.N;
    if (N <= 1024 || ((N + 3) / 4 + 255) / 256 > 8) {
        err = "the long-path kernel covers 1024 < N <= 8192";
        return ST_ERR_LIMIT;
    }
    FusedHostReq tabs;
    int pgmax = 1, gmax = 1;
    fused_tables(req, lay, 0, 0, 0, tabs, pgmax, gmax);
    const int rc = fft_request_fits(tabs, N, int(lay.options.size()), err);
    if (rc) return rc;
    footprint = FftSizes(req, int(lay.units.size()), int(tabs.fg.size()), int(lay.options.size())).total() +
                lay.options.size() * (sizeof(Option) + sizeof(PayOpt64) + sizeof(PayJob64)) +
                tabs.fg.size() * sizeof(FusedGroup) + tabs.fu.size() * (sizeof(FusedUnit) + sizeof(Unit));
    return ST_OK;
}

int FftFused::build(const Request& req, const Layout& lay, int device, hipStream_t st, std::string& err) {
    release();
    stream = st;
    const int N = req.N, nunits = int(lay.units.size());
    if (((N + 3) / 4 + 255) / 256 > 8) {
        err = "the long-path kernel covers N <= 8192";
        return ST_ERR_LIMIT;
    }
    FusedHostReq tabs;
    int pgmax = 1, gmax = 1;
    fused_tables(req, lay, 0, 0, 0, tabs, pgmax, gmax);
    total_out = int(lay.options.size());
    M = req.M;
    mc = req.method == METHOD_MC;
    hipDeviceProp_t prop;
    RB_TRY(device_props(device, prop));
    keep_pool_cached(device);
    cus = prop.multiProcessorCount;
    const int rc = fft_request_fits(tabs, N, total_out, err);
    if (rc) return rc;
    const FftSizes sz(req, nunits, int(tabs.fg.size()), total_out);
    ppt = sz.ppt;
    nblk = sz.nblk;
    chunk = sz.chunk;
    // beyond N = 4096 the FP64 transform of Gamma does not fit a workgroup's LDS: on the host
    const int log2L = fused_fft_log2(N), L = 1 << log2L;
    std::vector<float2> gh;
    if (!sz.gamma) {
        gh.resize(size_t(nunits) * L);
        for (int u = 0; u < nunits; ++u) {
            std::vector<std::complex<double>> g(L, 0.0);
            const double h = lay.units[u].H - 0.5 + 1.0;
            g[0] = lay.units[u].a;
            for (int k = 1; k < N; ++k) g[k] = (std::pow(k + 1.0, h) - std::pow(double(k), h)) / h;
            fft_host(g, -1);
            for (int k = 0; k < L; ++k) {
                const std::complex<double>& v = g[bit_reverse(k, log2L)];
                gh[size_t(u) * L + fft_spectrum_slot(log2L, k)] = make_float2(float(v.real()), float(v.imag()));
            }
        }
    }
    std::vector<PayRow> rows;
    for (const FusedOption& o : tabs.fo) {
        const FusedPG& pg = tabs.fpg[o.pg];
        rows.push_back(PayRow{pg.group, o.out, pg.rho, o.K, o.lnK});
    }
    std::stable_sort(rows.begin(), rows.end(), [](const PayRow& x, const PayRow& y) {
        return x.group != y.group ? x.group < y.group : x.rho < y.rho;
    });
    std::vector<PayJob64> jobs;
    std::vector<PayOpt64> opts;
    payoff_jobs(rows, nblk, cus, jobs, opts);
    npayjobs = int(jobs.size());
    // one device block: the tables (one upload from pinned memory, not waited for), what the device
    // forms from them, integrals, partial sums and results
    size_t off = 0;
    auto place = [&](size_t bytes) {
        const size_t o = off;
        off += (std::max<size_t>(bytes, 1) + 255) & ~size_t(255);
        return o;
    };
    const size_t o_un = place(nunits * sizeof(Unit)), o_fu = place(tabs.fu.size() * sizeof(FusedUnit)),
                 o_fg = place(tabs.fg.size() * sizeof(FusedGroup)), o_ivo = place(total_out * sizeof(Option)),
                 o_job = place(jobs.size() * sizeof(PayJob64)), o_opt = place(opts.size() * sizeof(PayOpt64)),
                 o_gh = place(sz.ghat);
    const size_t up_bytes = sz.gamma ? o_gh : off;
    const size_t o_tw = place(sz.tw), o_tw64 = place(sz.tw64), o_gamma = place(sz.gamma), o_ptab = place(sz.ptab),
                 o_ints = place(sz.ints), o_part = place(sz.partial);
    const size_t res_bytes = size_t(total_out) * 3 * sizeof(double);
    // results in the block where no pinned memory can be had, and large tables from pageable memory
    double* host_out = to_host ? reinterpret_cast<double*>(out.reserve(res_bytes)) : nullptr;
    const size_t o_out = place(host_out ? 1 : res_bytes);
    RB_TRY(alloc_async(&d_block, off, st));
    unsigned char* h = up_bytes <= PINNED_TABLES ? up.reserve(up_bytes) : nullptr;
    std::vector<unsigned char> pageable;
    if (!h) {
        pageable.resize(up_bytes);
        h = pageable.data();
    }
    d_price = host_out ? host_out : reinterpret_cast<double*>(d_block + o_out);
    d_iv = d_price + total_out;
    d_stat = d_iv + total_out;
    d_ivopts = reinterpret_cast<Option*>(d_block + o_ivo);
    d_payjobs = reinterpret_cast<PayJob64*>(d_block + o_job);
    d_payopts = reinterpret_cast<PayOpt64*>(d_block + o_opt);
    d_partial = reinterpret_cast<double*>(d_block + o_part);
    auto pack = [&](size_t o, const auto& v) {
        if (!v.empty()) std::memcpy(h + o, v.data(), v.size() * sizeof(v[0]));
    };
    pack(o_un, lay.units);
    pack(o_fu, tabs.fu);
    pack(o_fg, tabs.fg);
    pack(o_ivo, lay.options);
    pack(o_job, jobs);
    pack(o_opt, opts);
    pack(o_gh, gh);
    RB_TRY(hipMemcpyAsync(d_block, h, up_bytes, hipMemcpyHostToDevice, st));
    if (!pageable.empty()) RB_TRY(hipStreamSynchronize(st));
    FftFusedArgs& a = args;
    a = FftFusedArgs{};
    a.key = philox_key(req.seed.data(), int(req.seed.size()));
    a.N = N;
    a.nunits = nunits;
    a.mc = mc ? 1 : 0;
    a.units = reinterpret_cast<FusedUnit*>(d_block + o_fu);
    a.groups = reinterpret_cast<FusedGroup*>(d_block + o_fg);
    a.ptab = reinterpret_cast<float*>(d_block + o_ptab);
    a.ghat = reinterpret_cast<float2*>(d_block + o_gh);
    a.tw = reinterpret_cast<float2*>(d_block + o_tw);
    a.ints = reinterpret_cast<double*>(d_block + o_ints);
    RB_TRY(launch_fused_fft_tables(reinterpret_cast<const Unit*>(d_block + o_un), nunits, N,
                                   req.comp == COMP_EXACT ? 0.0 : 1.0,
                                   sz.gamma ? reinterpret_cast<double*>(d_block + o_gamma) : nullptr,
                                   sz.gamma ? reinterpret_cast<double2*>(d_block + o_tw64) : nullptr,
                                   reinterpret_cast<float*>(d_block + o_ptab), reinterpret_cast<float2*>(d_block + o_tw),
                                   reinterpret_cast<float2*>(d_block + o_gh), st));
    return ST_OK;
}

int FftFused::launch(hipStream_t st, std::string& err, Plan* timing, hipEvent_t kbeg, hipEvent_t kend) {
    auto timed = [&](int id) { return timing ? timing->timed(id) : -1; };
    auto mark = [&](int slot) {
        if (timing) timing->mark(slot, nullptr, nullptr);
    };
    int s;
    if (kbeg) RB_TRY(hipEventRecord(kbeg, st));
    for (long p0 = 0; p0 < M; p0 += chunk) {
        FftFusedArgs a = args;
        a.p0 = p0;
        a.np = std::min(chunk, M - p0);
        s = timed(K_FUSED);
        RB_TRY(launch_fused_fft(a, cus, st));
        mark(s);
        s = timed(K_PAYOFF);
        RB_TRY(launch_payoff64(a.ints, a.np, ppt, d_payjobs, npayjobs, d_payopts, total_out, mc ? PAY_MC_MIX : PAY_RT_MIX,
                               p0 / (256L * ppt), nblk, d_partial, nullptr, st));
        mark(s);
    }
    if (kend) RB_TRY(hipEventRecord(kend, st));
    s = timed(K_REDUCE);
    RB_TRY(launch_reduce_iv(d_partial, ReduceRows{nullptr, nullptr, nullptr, nblk, M}, d_ivopts, total_out, d_price,
                            d_stat, d_iv, nullptr, st));
    mark(s);
    return ST_OK;
}

hipError_t FftFused::fetch(double* price, double* iv, double* stat) const {
    const bool pinned = out.data() != nullptr;
    hipError_t e = fetch_results(price, d_price, total_out, pinned);
    if (!e) e = fetch_results(iv, d_iv, total_out, pinned);
    if (!e) e = fetch_results(stat, d_stat, total_out, pinned);
    return e;
}

int autotune_fused(const Request& shape, const std::vector<int>& Ns, int mode, int device,
                   std::vector<int>& chosen, std::vector<double>& best_ms, std::string& err) {
    chosen.assign(Ns.size(), 0);
    best_ms.assign(Ns.size(), 0.0);
    hipStream_t st = nullptr;
    hipEvent_t e0 = nullptr, e1 = nullptr;
    int rc = ST_OK;
    auto hip_ok = [&](hipError_t e, const char* what) {
        if (e == hipSuccess) return true;
        err = std::string(what) + ": " + hipGetErrorString(e);
        rc = e == hipErrorOutOfMemory ? ST_ERR_NOMEM : ST_ERR_DEVICE;
        return false;
    };
    if (!hip_ok(hipSetDevice(device), "hipSetDevice") ||
        !hip_ok(hipStreamCreateWithFlags(&st, hipStreamNonBlocking), "hipStreamCreate") ||
        !hip_ok(hipEventCreate(&e0), "hipEventCreate") || !hip_ok(hipEventCreate(&e1), "hipEventCreate"))
        goto done;
    for (size_t n = 0; n < Ns.size() && rc == ST_OK; ++n) {
        Request r = shape;
        r.N = Ns[n];
        rc = validate(r, err);
        if (rc) break;
        const Layout lay = make_layout(r);
        const int Np = (r.N + 31) / 32 * 32;
        double best = 0.0;
        int best_pb = 0;
        for (int pb : {1, 2, 4}) {
            FusedHostReq fh;
            std::string e2;
            if (plan_fused_request(r, lay, mode, fh, e2, pb) != ST_OK) continue;  // shape not valid
            FusedBatch B;
            if (B.build({&fh}, mode, device, st, e2) != ST_OK) continue;          // e.g. LDS
            // one untimed launch, then the fastest of three
            double ms = 0.0;
            for (int it = 0; it < 4 && rc == ST_OK; ++it) {
                if (!hip_ok(hipEventRecord(e0, st), "hipEventRecord")) break;
                if ((rc = B.launch(st, err)) != ST_OK) break;
                if (!hip_ok(hipEventRecord(e1, st), "hipEventRecord") ||
                    !hip_ok(hipEventSynchronize(e1), "hipEventSynchronize"))
                    break;
                float t = 0.f;
                if (!hip_ok(hipEventElapsedTime(&t, e0, e1), "hipEventElapsedTime")) break;
                if (it > 0 && (ms == 0.0 || t < ms)) ms = t;
            }
            B.release();
            (void)hipStreamSynchronize(st);
            if (rc != ST_OK) break;
            if (best_pb == 0 || ms < best) {
                best = ms;
                best_pb = pb;
            }
        }
        if (rc != ST_OK) break;
        if (best_pb == 0) {
            err = "no tile shape of the fused kernel fits N = " + std::to_string(r.N);
            rc = ST_ERR_LIMIT;
            break;
        }
        tune_set(Np, mode, r.method == METHOD_MC ? 1 : 0, best_pb);
        chosen[n] = best_pb;
        best_ms[n] = best;
    }
done:
    if (e0) (void)hipEventDestroy(e0);
    if (e1) (void)hipEventDestroy(e1);
    if (st) (void)hipStreamDestroy(st);
    return rc;
}

// ---------------------------------------------------------------- single-request plan
int Plan::init_fused(std::string& err) {
    fused_req.reset(new FusedHostReq());
    int rc = plan_fused_request(req, lay, fused_mode, *fused_req, err);
    if (rc) return rc;
    fused_batch.reset(new FusedBatch());
    fused_batch->to_host = true;
    rc = fused_batch->build({fused_req.get()}, fused_mode, device, stream, err);
    if (rc) return rc;
    nblk = fused_req->r.nitems;
    chunk = req.M;
    return ST_OK;
}

}  // namespace rb
