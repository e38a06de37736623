// sc_dec_fed.hip -- the fed decode (sc_fed.h) for one head size (built with
// -DSC_FED_RT=1 or 2: 32 * SC_FED_RT chunks per head).
#include "sc_fed.h"

#ifndef SC_FED_RT
#error "build with -DSC_FED_RT=1 or 2"
#endif

namespace sc {

template <>
hipError_t launch_decompress_fed<SC_FED_RT>(const ModelDev &M, int32_t heads, int32_t sets, hipStream_t s,
                                            const uint32_t *words, const int64_t *woff, const int32_t *wcnt,
                                            const int32_t *len, int64_t count, uint8_t *tokens, const int64_t *toff,
                                            int32_t *st, uint8_t *xch, int32_t spin_max) {
    void *args[] = {(void *)&M, (void *)&words, (void *)&woff, (void *)&wcnt, (void *)&len, (void *)&count,
                    (void *)&tokens, (void *)&toff, (void *)&st, (void *)&heads, (void *)&sets, (void *)&xch,
                    (void *)&spin_max};
    // cooperative: heads and feeders wait for each other, so all must be resident
    return hipLaunchCooperativeKernel((const void *)k_decompress_fed<SC_FED_RT>,
                                      dim3((unsigned)(heads + sets * FED_SLICES)), dim3(THREADS), args, 0, s);
}

}  // namespace sc
