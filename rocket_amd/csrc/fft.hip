// FFT plans (radices, twiddle tables) shared by the Wiener filter, the spectral
// filter and PCE.
#include "prnu_internal.hpp"
#include "fft_device.hpp"
#include "fft_host.hpp"

#include <algorithm>
#include <cmath>
#include <new>
#include <vector>

namespace prnu {

struct FftPlan {
    FftDesc desc, basic;
    float2 *d_tw = nullptr;
};

// Radices whose product is n, as few as possible (a pass is an LDS round trip
// and a barrier), then with the smallest sum (the least arithmetic and the
// evenest split over the threads); the power-of-two ones first, so the twiddle
// exponent's j mod Ns stays a mask.  4000 = 20 20 10 instead of 8 4 5 5 5.
static bool fft_factor(int n, int *radix, int *passes) {
    static const int kRadices[] = {16, 8, 4, 2, 20, 12, 10, 6, 15, 9, 5, 3};
    std::vector<int> best, cur;
    int best_sum = 0;
    auto search = [&](auto &self, int left, int from, int sum, int depth) -> void {
        if (depth == 0) {
            if (left == 1 && (best.empty() || sum < best_sum)) {
                best = cur;
                best_sum = sum;
            }
            return;
        }
        int most = 1;  // what depth passes can reach
        for (int k = 0; k < depth; ++k) most *= 20;
        if (left > most) return;
        for (int i = from; i < (int)(sizeof(kRadices) / sizeof(int)); ++i) {
            if (left % kRadices[i]) continue;
            cur.push_back(kRadices[i]);
            self(self, left / kRadices[i], i, sum + kRadices[i], depth - 1);
            cur.pop_back();
        }
    };
    for (int depth = 1; depth <= std::min(kFftMaxPasses, 6) && best.empty(); ++depth) search(search, n, 0, 0, depth);
    if (best.empty()) return false;
    *passes = (int)best.size();
    std::copy(best.begin(), best.end(), radix);
    return true;
}

// Radices 8, 4, 2, then 3 and 5 alone (a power-of-two part 8^k * 2 becomes
// 8^(k-1) * 4 * 4): PCE's plan.  A score's error is the bias of the plane's
// energy, which its roundings do not average out: 4 spectra of 500x960 were
// 1.2e-7 off so, 2.0e-7 with the composite radices, 3 of 3375x96 2.1e-8 and
// 5.3e-8.
static void fft_factor_basic(int n, int *radix, int *passes) {
    int p = 0, e2 = 0;
    for (; n % 2 == 0; n /= 2) ++e2;
    int n8 = e2 / 3, n4 = e2 % 3 == 2 ? 1 : 0, n2 = 0;
    if (e2 % 3 == 1) {
        if (n8 > 0) {
            --n8;
            n4 = 2;
        } else {
            n2 = 1;
        }
    }
    while (n8-- > 0) radix[p++] = 8;
    while (n4-- > 0) radix[p++] = 4;
    while (n2-- > 0) radix[p++] = 2;
    for (; n % 3 == 0; n /= 3) radix[p++] = 3;
    for (; n % 5 == 0; n /= 5) radix[p++] = 5;
    *passes = p;
}

static void fft_steps(FftDesc &d) {
    int64_t Ns = 1;
    for (int k = 0; k < d.passes; ++k) {
        d.step[k] = (int)(d.n / (Ns * d.radix[k]));
        d.inv[k] = (Ns & (Ns - 1)) ? (uint32_t)((int64_t(1) << 32) / Ns + 1) : 0;
        Ns *= d.radix[k];
    }
}

int fft_plan_create(int n, FftPlan **out) {
    *out = nullptr;
    PRNU_REQUIRE(n >= 2 && n <= kFftMaxN, "fft: length %d outside [2, %d]", n, kFftMaxN);
    FftPlan *p = new (std::nothrow) FftPlan();
    if (!p) {
        set_error("fft: out of host memory");
        return PRNU_ENOMEM;
    }
    p->desc.n = n;
    if (!fft_factor(n, p->desc.radix, &p->desc.passes)) {
        delete p;
        set_error("fft: length %d has a prime factor other than 2, 3, 5", n);
        return PRNU_ENOTSUP;
    }
    p->basic.n = n;
    fft_factor_basic(n, p->basic.radix, &p->basic.passes);
    fft_steps(p->desc);
    fft_steps(p->basic);
    std::vector<float2> tw(n);
    const double two_pi = 6.283185307179586476925286766559;
    for (int t = 0; t < n; ++t) {
        const double a = -two_pi * (double)t / (double)n;
        tw[t] = make_float2((float)std::cos(a), (float)std::sin(a));
    }
    hipError_t e = hipMalloc(&p->d_tw, sizeof(float2) * n);
    if (e == hipSuccess) e = hipMemcpy(p->d_tw, tw.data(), sizeof(float2) * n, hipMemcpyHostToDevice);
    if (e != hipSuccess) {
        if (p->d_tw) (void)hipFree(p->d_tw);
        delete p;
        (void)hipGetLastError();
        set_error("fft: twiddle table: %s", hipGetErrorString(e));
        return PRNU_EDEVICE;
    }
    p->desc.tw = p->basic.tw = p->d_tw;
    *out = p;
    return PRNU_OK;
}

void fft_plan_destroy(FftPlan *p) {
    if (!p) return;
    if (p->d_tw) (void)hipFree(p->d_tw);
    delete p;
}

const FftDesc &fft_desc(const FftPlan *p) { return p->desc; }
const FftDesc &fft_desc_basic(const FftPlan *p) { return p->basic; }

int ensure_fft_plans(Context *c) {
    if (!c->fft_w) PRNU_TRY(fft_plan_create(c->w, &c->fft_w));
    if (!c->fft_h) {
        if (c->h == c->w) {
            c->fft_h = c->fft_w;
        } else {
            PRNU_TRY(fft_plan_create(c->h, &c->fft_h));
        }
    }
    return PRNU_OK;
}

}  // namespace prnu
