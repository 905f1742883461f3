// Plans direct convolutions on the host: every launch of ndc::launch_direct is
// recorded instead of made (LaunchContext::dry_run).  Arguments: dtype, then
// "n k dilation stride" for each axis.  Prints the status, and the dynamic LDS
// bytes, grid, block and form of each launch.
#include <cstdio>
#include <cstdlib>
#include <cstring>

#include "launch.hpp"

using namespace ndc;

struct Dry final : LaunchContext {
    int launches = 0;
    hipStream_t stream() override { return nullptr; }
    void* scratch(int, size_t) override { return nullptr; }
    const void* twiddles(int64_t, bool) override { return nullptr; }
    const void* constant_table(const std::string&, const void*, size_t) override { return nullptr; }
    std::string text;
    std::string& memo(const std::string&) override { return text; }
    const int32_t* border_maps(const Plan&, int64_t*) override { return nullptr; }
    int cu_count() override { return 256; }
    size_t max_lds() override { return 160 * 1024 - kStaticLdsReserve; }
    bool dry_run() override { return true; }
    void record_launch(const char* kernel, size_t smem, unsigned grid, unsigned block) override {
        std::printf("launch %zu %u %u %s\n", smem, grid, block, std::strstr(kernel, "matrix_conv") ? "matrix" : "vector");
        ++launches;
    }
};

int main(int argc, char** argv) {
    ndc_conv_desc d;
    std::memset(&d, 0, sizeof(d));
    d.dtype = std::atoi(argv[1]);
    d.rank = (argc - 2) / 4;
    d.reverse = 1;
    d.conv_mode.tag = NDC_CONV_EXPLICIT;
    for (int i = 0; i < d.rank; ++i) {
        d.x_shape[i] = std::atoll(argv[2 + 4 * i]);
        d.k_shape[i] = std::atoll(argv[3 + 4 * i]);
        d.dilation[i] = std::atoll(argv[4 + 4 * i]);
        d.conv_mode.strides[i] = std::atoll(argv[5 + 4 * i]);
    }
    Plan p;
    Dry ctx;
    int s = make_plan(&d, NDC_OP_CONV, &p, &ctx.err, true);
    if (s == NDC_OK) s = launch_direct(p, &ctx, &ctx, &ctx, ctx);
    std::printf("status %d %s\n", s, ctx.err.c_str());
    return 0;
}
