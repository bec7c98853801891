// CPU run of the transforms of k_fused_fft (rb_fused_fft.hip) as that kernel runs them: the merged first pass, the
// passes below it with the table ordered by pass, the spectrum in the middle pass's order, slots padded
// by 16, and the inverse top stage where the result is read.  A host runner walks the groups of every pass in
// order (on the device they are disjoint and barriers separate the passes); the first pass of all threads reads before
// any writes where half of the threads take each half.  Checked against a direct FP64 linear convolution of two
// real paths for every transform length, N at both ends of its range.  Exit status 0 when every case is within 2e-5
// relative of the direct sum, no pad slot was written and every slot was.
#include <hip/hip_runtime.h>

#include <cmath>
#include <complex>
#include <cstdio>
#include <random>
#include <vector>

#include "rb_fft_lds.h"
#include "rb_fused.h"

using namespace rb;
typedef std::complex<double> cd;

constexpr int PAD = 4;
static int slot(int i) { return i + (i >> PAD); }

struct HostRunner {
    template <int LOG2L, int SB, int R, int KIND, class TW, class GT>
    void pass(float2* z, TW tw, GT G) const {
        for (int t = 0; t < ((1 << LOG2L) >> R); ++t) fft_group<LOG2L, SB, R, KIND, PAD>(z, tw, G, t);
    }
};

static unsigned brev(unsigned i, int b) {
    unsigned r = 0;
    for (int k = 0; k < b; ++k) r |= ((i >> k) & 1u) << (b - 1 - k);
    return r;
}

// FP64 discrete Fourier transform, forward
static void dft(std::vector<cd>& a) {
    const size_t n = a.size();
    if (n == 1) return;
    std::vector<cd> e(n / 2), o(n / 2);
    for (size_t i = 0; i < n / 2; ++i) {
        e[i] = a[2 * i];
        o[i] = a[2 * i + 1];
    }
    dft(e);
    dft(o);
    for (size_t k = 0; k < n / 2; ++k) {
        const cd t = std::polar(1.0, -2.0 * M_PI * double(k) / double(n)) * o[k];
        a[k] = e[k] + t;
        a[k + n / 2] = e[k] - t;
    }
}

template <int LOG2L>
static int check(int N) {
    constexpr int L = 1 << LOG2L, H2 = L / 2, span = 1 << (LOG2L - 5);
    std::vector<float2> tw(fused_fft_table(LOG2L));
    for (size_t i = 0; i < tw.size(); ++i) {
        const double a = -2.0 * M_PI * fft_twiddle_power(LOG2L, int(i)) / L;
        tw[i] = make_float2(float(std::cos(a)), float(std::sin(a)));
    }
    std::mt19937 g(LOG2L * 7 + N);
    std::normal_distribution<double> nd;
    std::vector<double> xa(N), xb(N), gam(N), ra(N, 0.0), rb(N, 0.0);
    for (int i = 0; i < N; ++i) {
        xa[i] = nd(g);
        xb[i] = nd(g);
        gam[i] = 1.0 / (1.0 + i) + 0.1 * nd(g);
    }
    double scale = 0.0;
    for (int i = 0; i < N; ++i) {
        for (int k = 0; k <= i; ++k) {
            ra[i] += gam[k] * xa[i - k];
            rb[i] += gam[k] * xb[i - k];
        }
        scale = std::max(scale, std::max(std::abs(ra[i]), std::abs(rb[i])));
    }
    std::vector<cd> gh(L, 0.0);
    for (int i = 0; i < N; ++i) gh[i] = gam[i];
    dft(gh);
    std::vector<float2> G(L, make_float2(NAN, NAN));
    for (int i = 0; i < L; ++i) {  // element i of the bit-reversed order
        const cd v = gh[brev(unsigned(i), LOG2L)];
        G[fft_spectrum_slot(LOG2L, i)] = make_float2(float(v.real()), float(v.imag()));
    }
    std::vector<float2> z(L + (L >> PAD), make_float2(NAN, NAN));
    for (int i = 0; i < H2; ++i)
        z[slot(i)] = i < N ? make_float2(float(xa[i]), float(xb[i])) : make_float2(0.f, 0.f);
    // the first pass
    std::vector<float2> in(16 * span);
    for (int pos = 0; pos < span; ++pos) {
        float2 x[16];
        fft_first_load<LOG2L, PAD>(x, z.data(), pos);
        for (int k = 0; k < 16; ++k) in[16 * pos + k] = x[k];
    }
    for (int h = 0; h < 2; ++h)
        for (int pos = 0; pos < span; ++pos) {
            float2 x[16];
            for (int k = 0; k < 16; ++k) x[k] = in[16 * pos + k];
            if (h) fft_first_upper<LOG2L>(x, tw.data(), pos);
            fft_first_store<LOG2L, PAD>(x, z.data(), tw.data(), pos, h);
        }
    fft_nat_fwd<LOG2L, LOG2L - 6>(z.data(), FftPassTable{tw.data() + H2}, FftSpectrum{G.data()}, HostRunner{});
    double e = 0.0;
    for (int i = 0; i < N; ++i) {
        const float2 lo = z[slot(i)], hi = z[slot(i + H2)], w = tw[i];
        const float2 m = fft_mul<FFT_MUL_Y>(hi, make_float2(w.x, -w.y));
        e = std::max(e, std::max(std::abs(double(lo.x + m.x) / L - ra[i]), std::abs(double(lo.y + m.y) / L - rb[i])));
    }
    bool ok = e <= 2e-5 * scale;
    for (size_t i = 0; i < z.size(); ++i) ok &= (i % 17 == 16) == bool(std::isnan(z[i].x));
    std::printf("L=2^%d N=%5d max err %.2e (scale %.2f) %s\n", LOG2L, N, e, scale, ok ? "ok" : "FAIL");
    return !ok;
}

int main() {
    int bad = 0;
    bad += check<10>(1) + check<10>(33) + check<10>(512);
    bad += check<11>(513) + check<11>(1024);
    bad += check<12>(1025) + check<12>(2048);
    bad += check<13>(2049) + check<13>(4096);
    bad += check<14>(4097) + check<14>(8192);
    std::printf(bad ? "FAIL\n" : "OK\n");
    return bad ? 1 : 0;
}
