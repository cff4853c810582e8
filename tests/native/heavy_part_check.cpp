// The grouping of heavy keys by bin (k_heavy_part) on its own: with the bins' true
// counts every key arrives and no error is set; with counts that send keys past the
// call's end (the kernel checks every position) the error bit says so.
#include "../../qsketch_amd/csrc/qs_learned.hip"

#include <algorithm>
#include <cstdio>

// what the rest of that file calls in the others, never reached here
extern "C" int qs_create(const qs_params *, qs_sketch **) { return QS_ERR_PARAM; }
extern "C" void qs_destroy(qs_sketch *) {}
extern "C" int qs_clear(qs_sketch *) { return QS_ERR_PARAM; }
extern "C" int qs_insert(qs_sketch *, const void *, size_t) { return QS_ERR_PARAM; }
void qs_scan_digits(uint32_t *, uint32_t, uint32_t, uint32_t *, hipStream_t) {}
void qs_scan_u32(uint32_t *, uint32_t, uint32_t *, hipStream_t) {}
uint64_t qs_scan_sums(uint64_t) { return 0; }

#define OK(x)                                                                                                    \
    do {                                                                                                         \
        if ((x) != hipSuccess) {                                                                                 \
            printf("HIP call failed: %s\n", #x);                                                                 \
            return 1;                                                                                            \
        }                                                                                                        \
    } while (0)

int main()
{
    const uint32_t n = 5000, chunks = (n + ROUTE_CHUNK - 1) / ROUTE_CHUNK;
    std::vector<uint32_t> stage(chunks * ROUTE_CHUNK, 0u), keys, light(chunks, 0u), bins(2 * HBINS + 2, 0u);
    for (uint32_t c = 0; c < chunks; ++c) {
        const uint32_t in = std::min(ROUTE_CHUNK, n - c * ROUTE_CHUNK);
        light[c] = in / (c + 2u); // heavy keys lie at the back of a chunk's slots
        for (uint32_t i = ROUTE_CHUNK - (in - light[c]); i < ROUTE_CHUNK; ++i) {
            const uint32_t k = stage[c * ROUTE_CHUNK + i] = (c * ROUTE_CHUNK + i) % 700u * 2654435761u;
            keys.push_back(k);
            bins[(uint32_t)((k * 0x9E3779B97F4A7C15ull) >> 56)]++;
        }
    }
    uint32_t *d_stage, *d_light, *d_bins, *d_out;
    OK(hipMalloc(&d_stage, stage.size() * 4));
    OK(hipMalloc(&d_light, light.size() * 4));
    OK(hipMalloc(&d_bins, bins.size() * 4));
    OK(hipMalloc(&d_out, n * 4));
    OK(hipMemcpy(d_stage, stage.data(), stage.size() * 4, hipMemcpyHostToDevice));
    OK(hipMemcpy(d_light, light.data(), light.size() * 4, hipMemcpyHostToDevice));
    uint32_t err[2];
    for (int past = 0; past < 2; ++past) {
        std::vector<uint32_t> b = bins, out(n), want = keys;
        b[0] += past ? n : 0u; // all later bins start past the end
        OK(hipMemcpy(d_bins, b.data(), b.size() * 4, hipMemcpyHostToDevice));
        hipLaunchKernelGGL(k_heavy_part<4>, dim3((chunks + HP_WAVES - 1u) / HP_WAVES), dim3(64 * HP_WAVES), 0, 0, d_stage,
                           (uint64_t)n, chunks, d_light, d_bins, d_bins + HBINS, d_out, d_bins + 2 * HBINS);
        OK(hipGetLastError());
        OK(hipMemcpy(out.data(), d_out, n * 4, hipMemcpyDeviceToHost));
        OK(hipMemcpy(&err[past], d_bins + 2 * HBINS, 4, hipMemcpyDeviceToHost));
        if (!past) {
            out.resize(keys.size());
            std::sort(out.begin(), out.end());
            std::sort(want.begin(), want.end());
            if (out != want) {
                printf("keys lost\n");
                return 1;
            }
        }
    }
    printf("errors %u %u\n", err[0], err[1]);
    return err[0] == 0 && err[1] == LE_SORT ? 0 : 1;
}
