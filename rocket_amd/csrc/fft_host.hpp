// Host-side FFT plan helpers shared by the extraction and PCE translation units.
#pragma once

#include "fft_device.hpp"
#include "prnu_internal.hpp"

namespace prnu {

int fft_plan_create(int n, FftPlan **out);
void fft_plan_destroy(FftPlan *p);
const FftDesc &fft_desc(const FftPlan *p);
const FftDesc &fft_desc_basic(const FftPlan *p);  // radices 8, 4, 2, 3, 5 alone
// Create the context's length-w and length-h plans on first use.
int ensure_fft_plans(Context *c);

}  // namespace prnu
