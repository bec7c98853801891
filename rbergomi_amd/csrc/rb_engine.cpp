// rb_engine.cpp -- host planner and executor.
//
// Replaces the driver layer of the reference: ComputePriceRTMT / ComputePriceMT
// (rBergLib/rBergomiMT.cpp:174-414), the single-thread class RBergomiST
// (rBergLib/RBergomi.cpp:157-370) and the ParamTot index algebra (rBergLib/ParamTot.h:20-50).
// Instead of walking the flat option index per path and recomputing on "triggers", the
// planner deduplicates the work once (units, groups, options; rb_types.h) and launches each
// stage over all paths of a chunk.
#include "rb_engine.h"

#include <algorithm>
#include <cmath>
#include <complex>
#include <cstdlib>
#include <cstring>
#include <deque>
#include <map>
#include <mutex>
#include <set>
#include <tuple>

#include "rb_kernels.h"

namespace rb {

static thread_local std::string g_last_error;
void set_last_error(const std::string& s) { g_last_error = s; }
const char* last_error() { return g_last_error.c_str(); }

const char* kernel_name(int id) {
    static const char* names[K_COUNT] = {"k_normals_f64", "k_volterra_f64", "k_scan_f64",
                                         "k_payoff64",    "k_reduce_iv",    "k_iv",
                                         "k_fused"};
    return id >= 0 && id < K_COUNT ? names[id] : "?";
}

hipError_t device_props(int device, hipDeviceProp_t& out) {
    static std::mutex mu;
    static std::map<int, hipDeviceProp_t> cache;
    std::lock_guard<std::mutex> lock(mu);
    const auto it = cache.find(device);
    if (it != cache.end()) {
        out = it->second;
        return hipSuccess;
    }
    const hipError_t e = hipGetDeviceProperties(&out, device);
    if (e == hipSuccess) cache[device] = out;
    return e;
}

void keep_pool_cached(int device) {
    static std::mutex mu;
    static std::set<int> done;
    std::lock_guard<std::mutex> lock(mu);
    if (!done.insert(device).second) return;
    hipMemPool_t pool;
    if (hipDeviceGetDefaultMemPool(&pool, device) == hipSuccess) {
        uint64_t keep = uint64_t(64) << 30;
        (void)hipMemPoolSetAttribute(pool, hipMemPoolAttrReleaseThreshold, &keep);
    }
}

int validate(const Request& r, std::string& err) {
    if (r.H.empty() || r.T.empty()) {
        err = "empty parameter or option arrays";
        return ST_ERR_ARG;
    }
    if (r.eta.size() != r.H.size() || r.rho.size() != r.H.size() || r.K.size() != r.T.size()) {
        err = "parameter arrays must be zipped: |H| = |eta| = |rho| and |T| = |K|";
        return ST_ERR_ARG;
    }
    if (r.rows && (r.T.size() != r.H.size() || r.xi_rows.size() != r.H.size())) {
        err = "unordered rows: every parameter array has one entry per row";
        return ST_ERR_ARG;
    }
    if (r.out_size() > 65535 || r.H.size() * (r.rows ? 1 : r.T.size()) > 65535) {
        err = "outputs above the supported maximum of 65535 per call";
        return ST_ERR_LIMIT;
    }
    if (r.scheme != SCHEME_HYBRID && r.scheme != SCHEME_CHOLESKY) {
        err = "unknown scheme";
        return ST_ERR_ARG;
    }
    if (r.N < 1 || r.M < 1) {
        err = "N and M must be positive";
        return ST_ERR_ARG;
    }
    if (r.N > 8192) {
        err = "N above the supported maximum of 8192 steps";
        return ST_ERR_LIMIT;
    }
    for (double h : r.H)
        if (!(h > 0.0 && h < 1.0)) {
            err = "H must lie in (0, 1)";
            return ST_ERR_ARG;
        }
    for (double t : r.T)
        if (!(t > 0.0)) {
            err = "maturities must be positive";
            return ST_ERR_ARG;
        }
    for (double k : r.K)
        if (!(k > 0.0)) {
            err = "strikes must be positive";
            return ST_ERR_ARG;
        }
    for (double x : r.rho)
        if (!(std::fabs(x) <= 1.0)) {
            err = "rho must lie in [-1, 1]";
            return ST_ERR_ARG;
        }
    if (!(r.xi >= 0.0)) {
        err = "xi must be non-negative";
        return ST_ERR_ARG;
    }
    for (double x : r.xi_rows)
        if (!(x >= 0.0)) {
            err = "xi must be non-negative";
            return ST_ERR_ARG;
        }
    return ST_OK;
}

Layout make_layout(const Request& r, bool gamma, bool comp) {
    Layout L;
    const int N = r.N;
    L.N = N;
    const long P = long(r.H.size()), O = long(r.T.size());
    // units: distinct H (getGamma per distinct H, rBergLib/rBergomiMT.cpp:318-324)
    std::map<double, int> unit_of;
    std::vector<int> unit_of_par(P);
    for (long h = 0; h < P; ++h) {
        auto it = unit_of.find(r.H[h]);
        if (it == unit_of.end()) {
            const int u = int(L.units.size());
            unit_of[r.H[h]] = u;
            const double H = r.H[h];
            const double s2H = std::sqrt(2.0 * H);
            const double rhoH = s2H / (H + 0.5);
            Unit un;
            un.H = H;
            un.a = rhoH / s2H;
            un.b = std::sqrt(1.0 - rhoH * rhoH) / s2H;
            un.sc = s2H * std::pow(1.0 / N, H);
            L.units.push_back(un);
            // Gamma_0 = 0, Gamma_k = ((k+1)^(a+1) - k^(a+1))/(a+1)  (getGamma :143-149)
            const double alpha = H - 0.5;
            if (gamma) L.gamma.push_back(0.0);
            for (int k = 1; gamma && k < N; ++k)
                L.gamma.push_back((std::pow(k + 1.0, alpha + 1.0) - std::pow(double(k), alpha + 1.0)) /
                                  (alpha + 1.0));
            unit_of_par[h] = u;
        } else {
            unit_of_par[h] = it->second;
        }
    }
    // groups: distinct (H, eta, T, xi) for RT; (H, eta, T, xi, rho) for plain MC.  Outputs in
    // order: I = h*|T| + t (tensor form, rBergLib/ParamTot.h:32-33), or I = row (unordered rows,
    // rBergomi/ParamTot.h:57-75, per-row xi as ML_console_ST/ParamTot.h:25-43)
    std::map<std::tuple<int, double, double, double, double>, int> group_of;
    const long nout = r.out_size();
    for (long I = 0; I < nout; ++I) {
        {
            const long h = r.rows ? I : I / O;
            const long t = r.rows ? I : I % O;
            const double xi = r.rows ? r.xi_rows[I] : r.xi;
            const int u = unit_of_par[h];
            const double rho_key = r.method == METHOD_MC ? r.rho[h] : 0.0;
            const auto key = std::make_tuple(u, r.eta[h], r.T[t], xi, rho_key);
            auto it = group_of.find(key);
            int g;
            if (it == group_of.end()) {
                g = int(L.groups.size());
                group_of[key] = g;
                const double H = r.H[h], T = r.T[t], eta = r.eta[h];
                Group G;
                G.unit = u;
                G.pad = 0;
                G.xi = xi;
                G.eta = eta;
                G.TH = std::pow(T, H);        // scaleWtilde :163-167
                G.dt = T / N;
                G.sdt = std::sqrt(G.dt);
                G.rho = r.rho[h];
                G.crho = std::sqrt(1.0 - r.rho[h] * r.rho[h]);
                L.groups.push_back(G);
                // compensator of updateV (:73-80): 0.5 eta^2 ((i-1) dt)^(2H), or (i dt) in exact mode
                if (comp) L.comp.push_back(0.0);
                for (int i = 1; comp && i < N; ++i) {
                    const double tc = r.comp == COMP_EXACT ? i * G.dt : (i - 1) * G.dt;
                    L.comp.push_back(0.5 * eta * eta * std::pow(tc, 2 * H));
                }
            } else {
                g = it->second;
            }
            Option o;
            o.group = g;
            o.pad = 0;
            o.rho = r.rho[h];
            o.K = r.K[t];
            o.lnK = std::log(r.K[t]);
            o.T = r.T[t];
            L.options.push_back(o);
        }
    }
    return L;
}

// splitmix64 finaliser (Steele, Lea, Flood, OOPSLA'14) folded over the seed words
static uint64_t splitmix64(uint64_t z) {
    z += 0x9E3779B97F4A7C15ULL;
    z = (z ^ (z >> 30)) * 0xBF58476D1CE4E5B9ULL;
    z = (z ^ (z >> 27)) * 0x94D049BB133111EBULL;
    return z ^ (z >> 31);
}

PhiloxKey philox_key(const uint64_t* seed, int n) {
    uint64_t h = splitmix64(0x243F6A8885A308D3ULL ^ uint64_t(n));
    for (int i = 0; i < n; ++i) h = splitmix64(h ^ seed[i]);
    PhiloxKey k;
    k.k0 = uint32_t(h);
    k.k1 = uint32_t(h >> 32);
    return k;
}

#define RB_TRY(expr)                                                                 \
    do {                                                                             \
        hipError_t e_ = (expr);                                                      \
        if (e_ != hipSuccess) {                                                      \
            err = std::string(#expr) + ": " + hipGetErrorString(e_);                 \
            return e_ == hipErrorOutOfMemory ? ST_ERR_NOMEM : ST_ERR_DEVICE;         \
        }                                                                            \
    } while (0)

// ---------------------------------------------------------------- workspace cache
// Device buffers of finished plans are kept for later plans: a one-shot call (rb_price_v2, the
// legacy symbols) otherwise spends far longer mapping and unmapping its staging buffers (up to
// ~6 GB) than computing with them -- measured 4 to 12 s against 0.36 s of kernels for 256
// small requests.  A request takes the smallest free block of its device that is at least its
// size and at most twice it, else allocates; freed blocks beyond WS_KEEP bytes are returned to
// the device, oldest first.  A block is reused only after the plan that released it has
// synchronized its stream.
namespace {
struct WsBlock {
    void* p;
    size_t bytes;
    int device;
};
std::mutex g_ws_mu;
std::deque<WsBlock> g_ws_free;          // released blocks, oldest first
std::map<void*, WsBlock> g_ws_used;
size_t g_ws_free_bytes = 0;
constexpr size_t WS_KEEP = size_t(48) << 30;
constexpr size_t WS_GRAIN = size_t(2) << 20;

// caller holds g_ws_mu
void ws_evict(size_t keep, int device) {
    for (auto it = g_ws_free.begin(); it != g_ws_free.end() && g_ws_free_bytes > keep;) {
        if (device >= 0 && it->device != device) {
            ++it;
            continue;
        }
        int cur = 0;
        (void)hipGetDevice(&cur);
        if (cur != it->device) (void)hipSetDevice(it->device);
        (void)hipFree(it->p);
        if (cur != it->device) (void)hipSetDevice(cur);
        g_ws_free_bytes -= it->bytes;
        it = g_ws_free.erase(it);
    }
}
}  // namespace

hipError_t ws_alloc(void** p, size_t bytes) {
    bytes = (std::max<size_t>(bytes, 1) + WS_GRAIN - 1) / WS_GRAIN * WS_GRAIN;
    int device = 0;
    hipError_t e = hipGetDevice(&device);
    if (e != hipSuccess) return e;
    std::lock_guard<std::mutex> lock(g_ws_mu);
    auto best = g_ws_free.end();
    for (auto it = g_ws_free.begin(); it != g_ws_free.end(); ++it)
        if (it->device == device && it->bytes >= bytes && it->bytes <= 2 * bytes &&
            (best == g_ws_free.end() || it->bytes < best->bytes))
            best = it;
    if (best != g_ws_free.end()) {
        *p = best->p;
        g_ws_used[best->p] = *best;
        g_ws_free_bytes -= best->bytes;
        g_ws_free.erase(best);
        return hipSuccess;
    }
    e = hipMalloc(p, bytes);
    if (e == hipErrorOutOfMemory) {  // give the device back what is cached, then try again
        (void)hipGetLastError();
        ws_evict(0, device);
        e = hipMalloc(p, bytes);
    }
    if (e == hipSuccess) g_ws_used[*p] = WsBlock{*p, bytes, device};
    return e;
}

void ws_free(void* p) {
    if (!p) return;
    std::lock_guard<std::mutex> lock(g_ws_mu);
    const auto it = g_ws_used.find(p);
    if (it == g_ws_used.end()) return;
    g_ws_free.push_back(it->second);
    g_ws_free_bytes += it->second.bytes;
    g_ws_used.erase(it);
    ws_evict(WS_KEEP, -1);
}

// A plan's device buffers are one workspace block, with everything to upload at its front: one
// allocation and, for tables of up to PINNED_TABLES, one copy per plan.
static size_t align256(size_t n) { return (n + 255) / 256 * 256; }

template <class T>
void Plan::dalloc(T** p, size_t n) {
    mem.push_back({reinterpret_cast<void**>(p), std::max<size_t>(n, 1) * sizeof(T)});
}

template <class T>
void Plan::upload(T** p, std::vector<T> v) {
    const auto held = std::make_shared<const std::vector<T>>(std::move(v));
    const size_t at = align256(up_bytes);
    up_bytes = at + held->size() * sizeof(T);
    up.push_back({reinterpret_cast<void**>(p), held, held->data(), held->size() * sizeof(T), at});
}

int Plan::commit(std::string& err) {
    // tables and results share a pinned block (the copy reads it and the last kernel writes it without
    // the host waiting); it is the plan's, and the plan waits for its stream before it goes.  Larger tables
    // are copied from where they are, and without pinned memory the results are too
    const size_t n = lay.options.size();
    size_t total = align256(up_bytes);
    const size_t front = up_bytes <= PINNED_TABLES ? total : 0;
    unsigned char* h = host.reserve(front + 3 * n * sizeof(double));
    if (!h) dalloc(&d_price, 3 * n);
    for (const auto& m : mem) total += align256(m.second);
    RB_TRY(ws_alloc(&d_block, total));
    char* base = static_cast<char*>(d_block);
    for (const Table& t : up) *t.p = base + t.at;
    size_t at = align256(up_bytes);
    for (const auto& m : mem) {
        *m.first = base + at;
        at += align256(m.second);
    }
    if (h) d_price = reinterpret_cast<double*>(h + front);
    d_stat = d_price + n;
    d_iv = d_stat + n;
    const bool packed = h && front > 0;
    for (const Table& t : up) {
        if (t.bytes == 0) continue;
        if (packed) std::memcpy(h + t.at, t.src, t.bytes);
        else RB_TRY(hipMemcpyAsync(base + t.at, t.src, t.bytes, hipMemcpyHostToDevice, stream));
    }
    if (packed && up_bytes > 0) RB_TRY(hipMemcpyAsync(base, h, up_bytes, hipMemcpyHostToDevice, stream));
    if (!packed) RB_TRY(hipStreamSynchronize(stream));  // the tables go now
    up.clear();
    return ST_OK;
}

Plan::~Plan() {
    if (stream) (void)hipStreamSynchronize(stream);
    if (gexec) (void)hipGraphExecDestroy(gexec);
    if (graph) (void)hipGraphDestroy(graph);
    fused_batch.reset();  // stream-ordered frees on this plan's stream
    fused_fft.reset();
    if (stream) (void)hipStreamSynchronize(stream);
    ws_free(d_block);  // the stream has synchronized above
    for (hipEvent_t e : ev_pool) (void)hipEventDestroy(e);
    if (own_stream && stream) stream_put(stream, device);
}

int Plan::init(const Request& r, hipStream_t st, bool quadrature, std::string& err) {
    int rc = validate(r, err);
    if (rc) return rc;
    req = r;
    path64 = r.precision == PREC_FP64 && r.scheme == SCHEME_HYBRID && r.N <= PATH64_FFT_MAX_N;
    // long paths on device Gaussians (or any N on request): the FFT kernel, which forms its own Gamma
    const bool split = fused_mode_of(r.precision) >= 0;  // a fused-kernel precision
    const bool fft1 = r.precision == PREC_FP32_FFT;      // the FFT kernel at every N
    const bool on_fft = (fft1 || (split && r.N > 1024)) && r.N <= 8192 && !quadrature && r.gauss == 0;
    // the staged scan's compensator table: the staged FP64 and FP32 paths, and caller's or Sobol'
    // Gaussians at a mixed precision
    lay = make_layout(r, !path64 && !on_fft, !path64 && (r.precision == PREC_FP64 || r.precision == PREC_FP32 || quadrature || r.gauss >= 1));
    int ndev = 0;
    RB_TRY(hipGetDeviceCount(&ndev));
    if (ndev < 1) {
        err = "no HIP device visible";
        return ST_ERR_DEVICE;
    }
    RB_TRY(hipGetDevice(&device));
    {
        hipDeviceProp_t prop;
        RB_TRY(device_props(device, prop));
        keep_pool_cached(device);
        lds_limit = prop.sharedMemPerBlock;
        cus = prop.multiProcessorCount;
        const size_t conv_lds = volterra_conv_mfma(r.N, lds_limit)
                                    ? volterra_mfma_long_lds_bytes(r.N, volterra_mfma_long_segment(r.N, lds_limit))
                                    : volterra_f64_lds_bytes(r.N);
        if (conv_lds > prop.sharedMemPerBlock) {
            err = "N = " + std::to_string(r.N) + " needs more LDS than one workgroup can hold";
            return ST_ERR_LIMIT;
        }
    }
    if (st) {
        stream = st;
    } else {
        RB_TRY(stream_get(&stream));
        own_stream = true;
    }
    if (r.turbo && (r.precision != PREC_FP64 || r.method != METHOD_RT || quadrature)) {
        err = "the turbo-charged estimator runs the Romano-Touzi FP64 path on device Gaussians";
        return ST_ERR_ARG;
    }
    if (r.scheme == SCHEME_CHOLESKY && r.precision != PREC_FP64) {
        err = "the Cholesky scheme runs on the FP64 path";
        return ST_ERR_ARG;
    }
    if (r.gauss >= 1 && (r.turbo || quadrature)) {
        err = "Sobol' points are not combined with caller Gaussians or the turbo-charged estimator";
        return ST_ERR_ARG;
    }
    if (r.gauss == 2 && (r.N & (r.N - 1)) != 0) {
        err = "the Brownian-bridge mapping needs N a power of two (hierarchical2increments)";
        return ST_ERR_ARG;
    }
    if (r.gauss >= 1 && r.M > 4294967294L) {
        err = "Sobol' points: M above 2^32 - 2";
        return ST_ERR_LIMIT;
    }
    if (r.scheme == SCHEME_CHOLESKY && r.N > 2048) {
        err = "the Cholesky scheme covers N <= 2048";
        return ST_ERR_LIMIT;
    }
    if (on_fft) {
        fused_fft.reset(new FftFused());
        fused_fft->to_host = true;
        const int rc = fused_fft->build(r, lay, device, stream, err);
        if (rc) return rc;
        nblk = fused_fft->nblk;
        chunk = fused_fft->chunk;
        return ST_OK;
    }
    if (r.precision == PREC_FP32 || ((split || fft1) && (r.N > 1024 || quadrature || r.gauss >= 1))) {
        // staged pipeline with the FP32 FFT convolution (long paths, user Gaussians)
        conv_fft = true;
    } else if (split) {
        if (quadrature) {
            err = "user-supplied Gaussians are priced on the FP64 path only";
            return ST_ERR_ARG;
        }
        fused = true;
        fused_mode = fused_mode_of(r.precision);
        return init_fused(err);
    }
    if (r.precision != PREC_FP64 && !conv_fft) {
        err = "precision not available in this build";
        return ST_ERR_ARG;
    }
    const int N = r.N;
    nstreams = r.method == METHOD_MC ? 3 : 2;
    const int nopt = int(lay.options.size());
    const long nunits = long(lay.units.size()), ngroups = long(lay.groups.size());
    // chunk the paths so that the staged buffers stay within ~6 GiB
    if (r.turbo) {
        if (r.precision != PREC_FP64 || r.method != METHOD_RT || quadrature) {
            err = "the turbo-charged estimator runs the Romano-Touzi FP64 path on device Gaussians";
            return ST_ERR_ARG;
        }
        if (r.m_control < 2 || !(r.q_max > 0.0)) {
            err = "turbo-charged estimator: m_control >= 2 and q_max > 0 required";
            return ST_ERR_ARG;
        }
    }
    const bool need_z = !path64 || quadrature || r.gauss >= 1;
    const double per_path = 8.0 * N * ((need_z ? nstreams : 0) + (path64 ? 0 : nunits)) + 16.0 * ngroups * (r.turbo ? 2 : 1) +
                            (quadrature ? 8.0 * nopt : 0.0);
    long ch = long(6.0e9 / per_path);
    // RBERGOMI_MAX_CHUNK caps the paths per chunk (used to test chunk boundaries)
    if (const char* env = std::getenv("RBERGOMI_MAX_CHUNK")) {
        const long cap = std::atol(env);
        if (cap > 0) ch = std::min(ch, cap);
    }
    // one path per payoff thread in the turbo-charged estimator, whose own payoff kernel sums 256
    ppt = r.turbo ? 1 : payoff_paths_per_thread(r.M, nopt);
    const long pblk = 256L * ppt;
    if (path64) {
        path64_fft = path64_uses_fft(N, int(nunits), int(ngroups), r.method == METHOD_MC);
        ch = std::min(ch, path64_fft ? path64_fft_max_paths(N) : path64_max_paths(N));
    }
    ch = std::max(pblk, ch / pblk * pblk);
    const long Mr = (r.M + pblk - 1) / pblk * pblk;
    chunk = std::min(ch, Mr);
    if (r.turbo) {
        // the pilot paths are priced as one chunk (two-pass covariances over all of them), of which the interface
        // allows as many as 6 GB hold with their Gaussians and Volterra processes beside the integrals
        const long mc = ((r.m_control + 255) / 256) * 256;
        const long fit = long(6.0e9 / (8.0 * N * (nstreams + nunits) + 32.0 * ngroups)) / 256 * 256;
        const long most = std::min(ch, std::max(256L, fit));
        if (mc > most) {
            err = "m_control above the paths one chunk holds (" + std::to_string(most) + ")";
            return ST_ERR_LIMIT;
        }
        chunk = std::max(chunk, mc);
    }
    nblk = (r.M + pblk - 1) / pblk;
    upload(&d_units, lay.units);
    upload(&d_opts, lay.options);
    init_payoffs();
    if (path64) {
        init_path64();
    } else {
        upload(&d_gamma, lay.gamma);
        upload(&d_groups, lay.groups);
        upload(&d_comp, lay.comp);
    }
    if (conv_fft) {
        rc = init_fft(err);
        if (rc) return rc;
    }
    if (r.gauss >= 1) {
        std::vector<uint32_t> V;
        sobol_directions(nstreams * N, V);
        upload(&d_sobol, V);
        if (!r.seed.empty()) {
            // digital shift: Philox block (0, dimension, 0, stream 7) of the seed's key
            const PhiloxKey key = philox_key(r.seed.data(), int(r.seed.size()));
            std::vector<uint32_t> sh(size_t(nstreams) * N);
            for (size_t d = 0; d < sh.size(); ++d) sh[d] = philox_block(key, uint64_t(d), 7u, 0u).x;
            upload(&d_shift, sh);
        }
    }
    if (r.scheme == SCHEME_CHOLESKY) {
        // host factor per unit (distinct H), then one upload
        std::vector<double> all, L;
        all.reserve(lay.units.size() * 2 * size_t(N) * N);
        for (const Unit& un : lay.units) {
            rc = chol_factor(un.H, N, L, err);
            if (rc) return rc;
            all.insert(all.end(), L.begin(), L.end());
        }
        upload(&d_chol, std::move(all));
    }
    if (need_z) dalloc(&d_Z, size_t(chunk) * nstreams * N);
    if (!path64) dalloc(&d_Wt, size_t(nunits) * chunk * N);
    dalloc(&d_ints, size_t(ngroups) * chunk * 2);
    dalloc(&d_partial, size_t(nopt) * nblk * 2);
    if (quadrature) dalloc(&d_payoff, size_t(chunk) * nopt);
    if (r.turbo) {
        dalloc(&d_ints2, size_t(ngroups) * chunk * 2);
        dalloc(&d_Qg, size_t(ngroups));
        dalloc(&d_alpha, size_t(nopt));
        dalloc(&d_exc, size_t(nopt) * nblk);
        dalloc(&d_count, size_t(nopt));
    }
    rc = commit(err);
    if (rc) return rc;
    if (path64) {
        p64.units = d_units;
        p64.groups = d_p64groups;
        p64.jobs = d_p64jobs;
        p64.gamma = d_p64tab;
        p64.ptab = d_p64tab + size_t(nunits) * p64.tlen;
        RB_TRY(launch_path64_tables(d_units, int(nunits), N, p64.tlen, r.comp == COMP_EXACT ? 0.0 : 1.0, d_p64tab,
                                    d_p64tab + size_t(nunits) * p64.tlen, stream));
        if (path64_fft) {
            p64.tw = d_p64fft;
            p64.ghat = d_p64fft + path64_fft_table(N);
            RB_TRY(launch_path64_fft_tables(p64.gamma, int(nunits), N, p64.tlen, d_p64fft,
                                            d_p64fft + path64_fft_table(N), stream));
        }
    }
    return ST_OK;
}

void Plan::begin_timing() {
    pending.clear();
    ev_used = 0;
    times.assign(K_COUNT, KernelTime());
    for (int i = 0; i < K_COUNT; ++i) times[i].name = kernel_name(i);
    if (fused_fft) times[K_FUSED].name = "k_fused_fft";
    // the convolution slot holds whichever kernel computes Wtilde
    if (req.scheme == SCHEME_CHOLESKY)
        times[K_VOLTERRA].name = "k_volterra_chol_f64";
    else if (conv_fft)
        times[K_VOLTERRA].name = "k_volterra_fft";
    else if (path64)
        times[K_VOLTERRA].name = path64_fft ? "k_path64_fft" : "k_path64";
    else if (volterra_conv_mfma(req.N, lds_limit))
        times[K_VOLTERRA].name = "k_volterra_mfma_long_f64";
}

int Plan::timed(int id) {
    if (!profile || capturing) return -1;
    while (ev_pool.size() < ev_used + 2) {
        hipEvent_t e;
        if (hipEventCreate(&e) != hipSuccess) return -1;
        ev_pool.push_back(e);
    }
    hipEvent_t a = ev_pool[ev_used], b = ev_pool[ev_used + 1];
    ev_used += 2;
    pending.push_back({id, {a, b}});
    (void)hipEventRecord(a, stream);
    return int(pending.size()) - 1;
}

void Plan::mark(int slot, hipEvent_t, hipEvent_t) {
    if (slot < 0) return;
    (void)hipEventRecord(pending[slot].second.second, stream);
}

void Plan::end_timing() {
    if (!profile) return;
    for (auto& p : pending) {
        float ms = 0.f;
        if (hipEventSynchronize(p.second.second) == hipSuccess &&
            hipEventElapsedTime(&ms, p.second.first, p.second.second) == hipSuccess) {
            times[p.first].total_ms += ms;
            times[p.first].launches += 1;
        }
    }
    pending.clear();
}

#define RB_LAUNCH(id, call)                  \
    do {                                     \
        const int slot_ = timed(id);         \
        RB_TRY(call);                        \
        mark(slot_, nullptr, nullptr);       \
    } while (0)

int Plan::integrals(uint64_t p0, long np, bool from_z, int signs, std::string& err) {
    const PhiloxKey key = philox_key(req.seed.data(), int(req.seed.size()));
    if (path64) {
        Path64Args a = p64;
        a.key = key;
        a.p0 = long(p0);
        a.np = np;
        a.src = !from_z ? P64_PHILOX : req.gauss >= 1 ? P64_MEMORY : P64_CALLER;
        a.signs = signs;
        a.Z = d_Z;
        a.zstride = long(nstreams) * req.N;
        a.ints = d_ints;
        a.ints2 = d_ints2;
        if (path64_fft) {
            path64_fft_shape(a, cus);
            RB_LAUNCH(K_VOLTERRA, launch_path64_fft(a, stream));
        } else {
            path64_shape(a, cus);
            RB_LAUNCH(K_VOLTERRA, launch_path64(a, stream));
        }
        return ST_OK;
    }
    const int N = req.N, ngroups = int(lay.groups.size());
    const long zs = long(nstreams) * N;
    if (!from_z) RB_LAUNCH(K_NORMALS, launch_normals_f64(key, long(p0), np, nstreams, N, d_Z, stream));
    RB_LAUNCH(K_VOLTERRA, conv(np, zs));
    RB_LAUNCH(K_SCAN, launch_scan_f64(req.method, d_Z, zs, d_Wt, np, N, d_groups, ngroups, d_comp, d_ints, stream));
    if (signs == 2)
        RB_LAUNCH(K_SCAN, launch_scan_f64(METHOD_RT, d_Z, zs, d_Wt, np, N, d_groups, ngroups, d_comp, d_ints2,
                                          stream, -1.0));
    return ST_OK;
}

// Enqueue one pricing run on the plan's stream (no synchronization).
int Plan::enqueue(std::string& err) {
    if (fused) return fused_batch->launch(stream, err, capturing ? nullptr : this);
    if (fused_fft) return fused_fft->launch(stream, err, capturing ? nullptr : this);
    const int N = req.N;
    const int nopt = int(lay.options.size());
    const int ngroups = int(lay.groups.size());
    if (req.turbo) {
        // pilot paths (counters TURBO_PILOT_BASE + m, disjoint from the main paths): Q and alpha
        const long mc = req.m_control;
        const int rc = integrals(TURBO_PILOT_BASE, mc, false, 1, err);
        if (rc) return rc;
        RB_LAUNCH(K_PAYOFF, launch_turbo_q(d_ints, mc, ngroups, d_Qg, stream));
        RB_LAUNCH(K_PAYOFF, launch_turbo_alpha(d_ints, mc, d_opts, nopt, d_Qg, d_alpha, stream));
    }
    for (long p0 = 0; p0 < req.M; p0 += chunk) {
        const long np = std::min(chunk, req.M - p0);
        if (req.gauss >= 1) {
            RB_LAUNCH(K_NORMALS, launch_normals_sobol_f64(d_sobol, d_shift, p0, np, nstreams, N, d_Z, stream));
            if (req.gauss == 2) RB_LAUNCH(K_NORMALS, launch_bridge_f64(d_Z, np * nstreams, N, stream));
        }
        const int rc = integrals(uint64_t(p0), np, req.gauss >= 1, req.turbo ? 2 : 1, err);
        if (rc) return rc;
        if (req.turbo) {
            RB_LAUNCH(K_PAYOFF, launch_turbo_payoff(d_ints, d_ints2, np, d_opts, nopt, d_Qg, d_alpha,
                                                    req.q_max, p0 / 256, nblk, d_partial, d_exc, stream));
        } else {
            RB_LAUNCH(K_PAYOFF, launch_payoff64(d_ints, np, ppt, d_payjobs, npayjobs, d_payopts, nopt,
                                                req.method == METHOD_MC ? PAY_MC64 : PAY_RT64,
                                                p0 / (256 * ppt), nblk, d_partial, nullptr, stream));
        }
    }
    RB_LAUNCH(K_REDUCE, launch_reduce_iv(d_partial, ReduceRows{nullptr, nullptr, nullptr, nblk, req.M}, d_opts, nopt,
                                         d_price, d_stat, req.turbo ? nullptr : d_iv, nullptr, stream));
    if (req.turbo) {
        RB_LAUNCH(K_REDUCE, launch_turbo_adjust(d_price, d_opts, nopt, d_Qg, d_alpha, req.q_max, d_exc,
                                                nblk, req.M, d_count, stream));
        RB_LAUNCH(K_IV, launch_iv(d_price, d_opts, nopt, d_iv, stream));
    }
    return ST_OK;
}

int Plan::run(std::string& err) {
    if (use_graph) {
        // first run: record the launches into a graph; every run replays it
        if (!gexec) {
            // one eager run first: kernel attributes are set outside the capture, and the
            // captured graph then replays the same launches
            RB_TRY(hipStreamSynchronize(stream));
            {
                const int rc = enqueue(err);
                if (rc) return rc;
            }
            RB_TRY(hipStreamSynchronize(stream));
            capturing = true;
            RB_TRY(hipStreamBeginCapture(stream, hipStreamCaptureModeThreadLocal));
            const int rc = enqueue(err);
            hipGraph_t g = nullptr;
            const hipError_t e = hipStreamEndCapture(stream, &g);
            capturing = false;
            if (rc) {
                if (g) (void)hipGraphDestroy(g);
                return rc;
            }
            RB_TRY(e);
            graph = g;
            RB_TRY(hipGraphInstantiate(&gexec, graph, nullptr, nullptr, 0));
        }
        RB_TRY(hipGraphLaunch(gexec, stream));
        RB_TRY(hipStreamSynchronize(stream));
        return ST_OK;
    }
    begin_timing();
    const int rc = enqueue(err);
    if (rc) return rc;
    RB_TRY(hipStreamSynchronize(stream));
    end_timing();
    return ST_OK;
}

int Plan::run_samples(const double* Z_host, double* payoff_host, std::string& err) {
    const int N = req.N;
    const int nopt = int(lay.options.size());
    begin_timing();
    for (long p0 = 0; p0 < req.M; p0 += chunk) {
        const long np = std::min(chunk, req.M - p0);
        RB_TRY(hipMemcpyAsync(d_Z, Z_host + size_t(p0) * nstreams * N,
                              size_t(np) * nstreams * N * sizeof(double), hipMemcpyHostToDevice, stream));
        const int rc = integrals(0, np, true, 1, err);
        if (rc) return rc;
        RB_LAUNCH(K_PAYOFF, launch_payoff64(d_ints, np, ppt, d_payjobs, npayjobs, d_payopts, nopt,
                                                req.method == METHOD_MC ? PAY_MC64 : PAY_RT64,
                                            p0 / (256 * ppt), nblk, d_partial, d_payoff, stream));
        RB_TRY(hipMemcpyAsync(payoff_host + size_t(p0) * nopt, d_payoff, size_t(np) * nopt * sizeof(double),
                              hipMemcpyDeviceToHost, stream));
        RB_TRY(hipStreamSynchronize(stream));
    }
    RB_LAUNCH(K_REDUCE, launch_reduce_iv(d_partial, ReduceRows{nullptr, nullptr, nullptr, nblk, req.M}, d_opts, nopt,
                                         d_price, d_stat, d_iv, nullptr, stream));
    RB_TRY(hipStreamSynchronize(stream));
    end_timing();
    return ST_OK;
}

// FFT in FP64 (iterative radix-2, sign -1 forward) for the host-side table FFT(Gamma)
void fft_host(std::vector<std::complex<double>>& a, int sign) {
    const int n = int(a.size());
    for (int i = 1, j = 0; i < n; ++i) {
        int bit = n >> 1;
        for (; j & bit; bit >>= 1) j ^= bit;
        j ^= bit;
        if (i < j) std::swap(a[i], a[j]);
    }
    for (int len = 2; len <= n; len <<= 1) {
        for (int i = 0; i < n; i += len)
            for (int k = 0; k < len / 2; ++k) {
                const double ang = sign * 2.0 * M_PI * k / len;
                const std::complex<double> w(std::cos(ang), std::sin(ang));
                const std::complex<double> u = a[i + k], v = a[i + k + len / 2] * w;
                a[i + k] = u + v;
                a[i + k + len / 2] = u - v;
            }
    }
}

int Plan::init_fft(std::string& err) {
    const int N = req.N;
    log2L = 0;
    while ((1 << log2L) < 2 * N - 1) ++log2L;
    if (log2L < 1) log2L = 1;
    const int L = 1 << log2L;
    hipDeviceProp_t prop;
    RB_TRY(device_props(device, prop));
    if (volterra_fft_lds_bytes(log2L) > prop.sharedMemPerBlock) {
        err = "N too large for the LDS FFT";
        return ST_ERR_LIMIT;
    }
    // twiddles computed in FP64, stored in FP32
    std::vector<float2> tw(L / 2);
    for (int k = 0; k < L / 2; ++k) {
        const double ang = -2.0 * M_PI * double(k) / double(L);
        tw[k] = make_float2(float(std::cos(ang)), float(std::sin(ang)));
    }
    std::vector<float2> gh(lay.units.size() * size_t(L));
    for (size_t u = 0; u < lay.units.size(); ++u) {
        std::vector<std::complex<double>> a(L, 0.0);
        for (int k = 0; k < N; ++k) a[k] = lay.gamma[u * N + k];
        fft_host(a, -1);
        for (int k = 0; k < L; ++k) gh[u * L + k] = make_float2(float(a[k].real()), float(a[k].imag()));
    }
    upload(&d_tw, tw);
    upload(&d_ghat, std::move(gh));
    return ST_OK;
}

void payoff_jobs(const std::vector<PayRow>& rows, long nblk, int cus, std::vector<PayJob64>& jobs,
                 std::vector<PayOpt64>& opts) {
    const int n = int(rows.size());
    int most = PAY64_OPTS;
    while (most > 1 && nblk * ((n + most - 1) / most) < 4L * cus) most /= 2;
    jobs.clear();
    opts.clear();
    for (int k = 0; k < n; ++k) {
        const PayRow& o = rows[k];
        opts.push_back(PayOpt64{o.K, o.lnK, o.out, 0});
        if (jobs.empty() || jobs.back().group != o.group || jobs.back().rho != o.rho || jobs.back().n == most)
            jobs.push_back(PayJob64{o.group, k, 0, 0, o.rho});
        ++jobs.back().n;
    }
}

void Plan::init_payoffs() {
    std::vector<PayRow> rows;
    for (size_t I = 0; I < lay.options.size(); ++I) {
        const Option& o = lay.options[I];
        rows.push_back(PayRow{o.group, int(I), o.rho, o.K, o.lnK});
    }
    std::stable_sort(rows.begin(), rows.end(),
                     [](const PayRow& a, const PayRow& b) { return a.group != b.group ? a.group < b.group : a.rho < b.rho; });
    std::vector<PayJob64> jobs;
    std::vector<PayOpt64> opts;
    payoff_jobs(rows, nblk, cus, jobs, opts);
    npayjobs = int(jobs.size());
    upload(&d_payjobs, jobs);
    upload(&d_payopts, opts);
}

// Tables of the single-pass FP64 path: groups ordered by unit with their exponent's coefficients,
// jobs of one unit and up to greg groups, and gamma and P of every unit, formed on the device.
void Plan::init_path64() {
    const int N = req.N, nunits = int(lay.units.size()), ngroups = int(lay.groups.size());
    std::vector<int> order(ngroups), count(nunits, 0);
    for (int g = 0; g < ngroups; ++g) {
        order[g] = g;
        ++count[lay.groups[g].unit];
    }
    std::stable_sort(order.begin(), order.end(), [&](int x, int y) { return lay.groups[x].unit < lay.groups[y].unit; });
    p64.N = N;
    p64.tlen = (N + 15) / 16 * 16;
    p64.mc = req.method == METHOD_MC;
    p64.greg = path64_greg(*std::max_element(count.begin(), count.end()), req.turbo ? 2 : 1);
    constexpr double L2E16 = 23.083120654223414192;  // 16 log2(e): half the exponent, in 32nds of an octave
    std::vector<Path64Group> groups(ngroups);
    std::vector<Path64Job> jobs;
    for (int k = 0; k < ngroups; ++k) {
        const Group& G = lay.groups[order[k]];
        const Unit& un = lay.units[G.unit];
        Path64Group& o = groups[k];
        o.c1 = L2E16 * G.eta * G.TH * un.sc;
        o.al = std::min(std::max(L2E16 * 0.5 * G.eta * G.eta * std::pow(G.dt, 2.0 * un.H), P64_AL_MIN), P64_AL_MAX);
        o.xi = G.xi;
        o.sxi = std::sqrt(G.xi);
        o.dt = G.dt;
        o.sdt = G.sdt;
        o.rho = G.rho;
        o.crho = G.crho;
        o.out = order[k];
        o.pad = 0;
        if (jobs.empty() || jobs.back().unit != G.unit || jobs.back().gn == p64.greg)
            jobs.push_back(Path64Job{G.unit, k, 0, 0});
        ++jobs.back().gn;
    }
    p64.njobs = int(jobs.size());
    upload(&d_units, lay.units);
    upload(&d_p64groups, groups);
    upload(&d_p64jobs, jobs);
    dalloc(&d_p64tab, size_t(2) * nunits * p64.tlen);
    if (path64_fft) dalloc(&d_p64fft, path64_fft_table(N) + (size_t(nunits) << path64_fft_log2(N)));
}

hipError_t Plan::conv(long np, long zstride) {
    if (req.scheme == SCHEME_CHOLESKY)
        return launch_volterra_chol(d_Z, zstride, np, req.N, int(lay.units.size()), d_chol, d_Wt, stream);
    if (conv_fft)
        return launch_volterra_fft(d_Z, zstride, np, req.N, log2L, int(lay.units.size()), d_units, d_ghat,
                                   d_tw, d_Wt, stream);
    return launch_volterra_conv_f64(d_Z, zstride, np, req.N, int(lay.units.size()), d_units, d_gamma, d_Wt,
                                    lds_limit, stream);
}

int Plan::turbo_results(double* alpha, double* Q, long* exceptions, std::string& err) {
    if (!req.turbo) {
        err = "not a turbo-charged plan";
        return ST_ERR_ARG;
    }
    const int nopt = int(lay.options.size());
    if (alpha) RB_TRY(hipMemcpyAsync(alpha, d_alpha, nopt * sizeof(double), hipMemcpyDeviceToHost, stream));
    if (exceptions)
        RB_TRY(hipMemcpyAsync(exceptions, d_count, nopt * sizeof(long), hipMemcpyDeviceToHost, stream));
    std::vector<double> qg(lay.groups.size());
    RB_TRY(hipMemcpyAsync(qg.data(), d_Qg, qg.size() * sizeof(double), hipMemcpyDeviceToHost, stream));
    RB_TRY(hipStreamSynchronize(stream));
    if (Q)
        for (int i = 0; i < nopt; ++i) Q[i] = qg[lay.options[i].group];
    return ST_OK;
}

int Plan::results(double* price, double* iv, double* stat, std::string& err) {
    RB_TRY(hipStreamSynchronize(stream));
    if (fused) {
        RB_TRY(fused_batch->fetch(0, price, iv, stat));
    } else if (fused_fft) {
        RB_TRY(fused_fft->fetch(price, iv, stat));
    } else {
        const size_t n = lay.options.size();
        const bool pinned = host.data() != nullptr;
        RB_TRY(fetch_results(price, d_price, n, pinned));
        RB_TRY(fetch_results(stat, d_stat, n, pinned));
        RB_TRY(fetch_results(iv, d_iv, n, pinned));
    }
    return ST_OK;
}

}  // namespace rb
