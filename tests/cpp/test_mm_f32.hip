// The fp32 products of many rows (k_mm_f32) against the few-row kernels,
// which other tests pin to the oracle, bit for bit: a head's gate, up and SiLU
// product (both matrices in one launch) and its down product added to its
// input, which no call returns by themselves.  Ends with status 1 on a
// difference, 2 without a GPU.
#include "../../pocketforge_amd/csrc/pf_gemv.hip"

#include <cstdio>
#include <cstring>
#include <random>
#include <vector>

using namespace pf;

static void hip(hipError_t e, const char* what) {
    if (e == hipSuccess) return;
    std::fprintf(stderr, "%s: %s\n", what, hipGetErrorString(e));
    std::exit(2);
}

template <class T>
struct Dev {
    T* p = nullptr;
    explicit Dev(size_t n) { hip(hipMalloc((void**)&p, n * sizeof(T)), "hipMalloc"); }
    explicit Dev(const std::vector<T>& v) : Dev(v.size()) {
        hip(hipMemcpy(p, v.data(), v.size() * sizeof(T), hipMemcpyHostToDevice), "hipMemcpy");
    }
    ~Dev() { (void)hipFree(p); }
    std::vector<T> host(size_t n) const {
        std::vector<T> v(n);
        hip(hipMemcpy(v.data(), p, n * sizeof(T), hipMemcpyDeviceToHost), "hipMemcpy");
        return v;
    }
};

// An N x K matrix: random codes, block scales of 2^-9 .. 2^-4.
struct Mat {
    Dev<uint8_t> codes;
    Dev<uint16_t> scales;
    static std::vector<uint8_t> bytes(std::mt19937& r, size_t n) {
        std::vector<uint8_t> v(n);
        for (auto& x : v) x = (uint8_t)r();
        return v;
    }
    static std::vector<uint16_t> halves(std::mt19937& r, size_t n) {
        std::vector<uint16_t> v(n);
        for (auto& x : v) x = (uint16_t)((6 + r() % 6) << 10 | r() % 1024);
        return v;
    }
    Mat(std::mt19937& r, uint32_t N, uint32_t K, int fmt)
        : codes(bytes(r, (size_t)N * K / (fmt == FMT_Q8 ? 1 : 2))), scales(halves(r, (size_t)N * K / 32)) {}
};

static int failures = 0;

static void same(const std::vector<float>& got, const std::vector<float>& ref, const char* what, uint32_t M, uint32_t N,
                 uint32_t K) {
    size_t bad = 0, zero = 0;
    for (size_t i = 0; i < ref.size(); i++) {
        bad += std::memcmp(&got[i], &ref[i], 4) != 0;
        zero += ref[i] == 0.0f;
    }
    const bool ok = bad == 0 && zero < ref.size() / 2;
    std::printf("%s %s: %u rows of %u x %u, %zu of %zu differ, %zu are 0\n", ok ? "ok" : "FAIL", what, M, N, K, bad,
                ref.size(), zero);
    std::fflush(stdout);
    failures += !ok;
}

template <int FMT, bool GLU, int KS>
static void tall(const Mat& a, const Mat* u, uint32_t M, uint32_t N, uint32_t K, const float* h, float* y,
                 const float* y_in) {
    const uint32_t mtiles = (M + 31) / 32, groups = (N / 32 + 4 / KS - 1) / (4 / KS);
    hipLaunchKernelGGL((k_mm_f32<FMT, GLU, KS>), dim3(8 * mtiles * ((groups + 7) / 8)), dim3(256), 0, 0, a.codes.p,
                       a.scales.p, u ? u->codes.p : nullptr, u ? u->scales.p : nullptr, N, K, M, mtiles, h, K, y, N, y_in);
    hip(hipGetLastError(), "k_mm_f32");
}

template <int FMT>
static void residual(std::mt19937& r, uint32_t M, uint32_t N, uint32_t K, const Dev<float>& h) {
    const Mat a(r, N, K, FMT);
    std::vector<float> in((size_t)M * N);
    std::normal_distribution<float> d;
    for (auto& x : in) x = d(r);
    const Dev<float> y_in(in), ref((size_t)M * N), y1((size_t)M * N), y4((size_t)M * N);
    hipLaunchKernelGGL((k_gemv_f32<1, FMT, 1>), dim3(N / 4, M), dim3(256), 0, 0, a.codes.p, a.scales.p, N, K, h.p, K, ref.p,
                       N, (const float*)y_in.p);
    hip(hipGetLastError(), "k_gemv_f32");
    tall<FMT, false, 1>(a, nullptr, M, N, K, h.p, y1.p, y_in.p);
    tall<FMT, false, 4>(a, nullptr, M, N, K, h.p, y4.p, y_in.p);
    const auto want = ref.host((size_t)M * N);
    same(y1.host((size_t)M * N), want, FMT == FMT_Q8 ? "Q8 down, a wave per tile" : "Q4 down, a wave per tile", M, N, K);
    same(y4.host((size_t)M * N), want, FMT == FMT_Q8 ? "Q8 down, K over four waves" : "Q4 down, K over four waves", M, N, K);
}

int main() {
    int n = 0;
    if (hipGetDeviceCount(&n) != hipSuccess || n == 0) {
        std::fprintf(stderr, "no GPU\n");
        return 2;
    }
    std::mt19937 r(7);
    const uint32_t shapes[][3] = {{12, 64, 256},   {17, 256, 256},  {18, 768, 768},   {27, 256, 256},  {28, 256, 256},
                                  {33, 1280, 1280}, {28, 2048, 2048}, {64, 2048, 2048}, {65, 320, 1792}, {320, 256, 512}};
    for (const auto& s : shapes) {
        const uint32_t M = s[0], N = s[1], K = s[2];
        std::vector<float> hv((size_t)M * K);
        std::normal_distribution<float> d;
        for (auto& x : hv) x = d(r);
        const Dev<float> h(hv), ref((size_t)M * N), y((size_t)M * N);
        const Mat g(r, N, K, FMT_Q4), u(r, N, K, FMT_Q4);
        hipLaunchKernelGGL(k_gemv_f32_glu<1>, dim3(N / 4, M), dim3(256), 0, 0, g.codes.p, g.scales.p, u.codes.p, u.scales.p, N,
                           K, h.p, K, ref.p, N);
        hip(hipGetLastError(), "k_gemv_f32_glu");
        tall<FMT_Q4, true, 4>(g, &u, M, N, K, h.p, y.p, nullptr);
        same(y.host((size_t)M * N), ref.host((size_t)M * N), "gate, up and SiLU", M, N, K);
        residual<FMT_Q4>(r, M, N, K, h);
        residual<FMT_Q8>(r, M, N, K, h);
    }
    std::printf("%d failed\n", failures);
    return failures ? 1 : 0;
}
