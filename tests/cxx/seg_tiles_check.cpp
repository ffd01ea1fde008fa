// Device check of the segmented products' bf16 tiles (moondream-zig_amd/csrc/seg_gemm.hip): every tile form gives the same bits in every
// segment, a sample of them is as close to sums in double as their type allows, and nothing outside the result is written.  And lm_silu
// against the quotient by the library's exponential, bit for bit.
#include "layer_list.hpp"
#include "lm_types.hpp"

#include <cmath>
#include <cstdio>
#include <cstring>
#include <random>
#include <vector>

static float widen(uint16_t v) {
    const uint32_t u = uint32_t(v) << 16;
    float f;
    memcpy(&f, &u, 4);
    return f;
}

// every f32 value; counts other bits (any NaN equals any)
__global__ void silu_check(unsigned *other) {
    const unsigned long long all = gridDim.x * 256ull;
    for (unsigned long long v = blockIdx.x * 256 + threadIdx.x; v <= 0xffffffffull; v += all) {
        const float z = __builtin_bit_cast(float, (unsigned)v), a = lm_silu(z), b = z / (1.0f + expf(-z));
        if (__builtin_bit_cast(unsigned, a) != __builtin_bit_cast(unsigned, b) && !(a != a && b != b)) atomicAdd(other, 1);
    }
}

int main() {
    moon_ctx ctx;
    if (hipSetDevice(0) != hipSuccess || hipStreamCreate(&ctx.stream) != hipSuccess) return printf("no device\n"), 2;
    ctx.cu_count = 256;
    struct Shape {
        int M, n16, n32, N, K, lda, splits, kb[SEG_MAX_SPLITS + 1], longest_first;
    };
    // edges of a tile's rows and columns, segments that meet inside a tile, one k-tile, two, an odd number; more tiles than compute units; ranges of k, with 38 wide
    // tiles each so that a die's last slots are empty and some workgroups' first tile is in their second round
    const Shape shapes[] = {
        {1, 64, 64, 64, 64, 64, 1, {}, 0},
        {63, 0, 0, 64, 128, 136, 1, {}, 0},
        {191, 64, 128, 256, 192, 192, 1, {}, 0},
        {192, 192, 256, 320, 256, 264, 1, {}, 0},
        {193, 128, 192, 448, 320, 320, 1, {}, 0},
        {255, 256, 256, 512, 64, 64, 1, {}, 0},
        {256, 0, 64, 256, 128, 128, 1, {}, 0},
        {257, 320, 384, 1024, 448, 448, 1, {}, 0},
        {385, 512, 512, 768, 2048, 2048, 1, {}, 0},
        {2000, 3072, 3136, 12352, 192, 192, 1, {}, 0},
        {300, 0, 640, 640, 704, 712, 3, {0, 128, 256, 704}, 1},
        {450, 0, 2048, 2048, 640, 640, 3, {0, 256, 512, 640}, 0},
        {300, 0, 4864, 4864, 640, 640, 8, {0, 128, 192, 320, 384, 448, 512, 576, 640}, 1},
    };
    int failures = 0, checked = 0;
    std::mt19937_64 rng(1);
    std::normal_distribution<float> normal;
    for (const Shape &s : shapes) {
        const int PAST = 4; // rows behind each result
        std::vector<uint16_t> a(size_t(s.M) * s.lda), w(size_t(s.N) * s.K);
        auto fill = [&](std::vector<uint16_t> &v, float scale) {
            for (auto &x : v) {
                const float f = normal(rng) * scale;
                uint32_t u;
                memcpy(&u, &f, 4);
                x = uint16_t(u >> 16);
            }
        };
        fill(a, 1.0f);
        fill(w, 2.0f / std::sqrt(float(s.K)));
        const int ld16 = s.n16 + 8, ld32 = s.n32 - s.n16 + 4, ldg = (s.N - s.n32) / 2 + 8;
        const size_t n16 = size_t(s.M + PAST) * ld16, n32 = size_t(s.M * s.splits + PAST) * ld32, ng = size_t(s.M + PAST) * ldg;
        void *da, *dw, *d16, *d32, *dg;
        if (hipMalloc(&da, a.size() * 2) || hipMalloc(&dw, w.size() * 2) || hipMalloc(&d16, n16 * 2) || hipMalloc(&d32, n32 * 4) || hipMalloc(&dg, ng * 2)) return printf("no memory\n"), 2;
        if (hipMemcpy(da, a.data(), a.size() * 2, hipMemcpyHostToDevice) || hipMemcpy(dw, w.data(), w.size() * 2, hipMemcpyHostToDevice)) return printf("copy\n"), 2;
        std::vector<uint16_t> first16, first_g, c16(n16), cg(ng);
        std::vector<uint32_t> first32, c32(n32);
        for (int tile : {2, 3, 4, SEG_BLOCK + 3, SEG_BLOCK + 4, SEG_THIN + 2}) {
            printf("%d x %d x %d, segments %d %d, %d ranges, tile %d\n", s.M, s.N, s.K, s.n16, s.n32, s.splits, tile);
            fflush(stdout);
            (void)hipMemset(d16, 0x5a, n16 * 2);
            (void)hipMemset(d32, 0x5a, n32 * 4);
            (void)hipMemset(dg, 0x5a, ng * 2);
            SegGemm p{};
            p.A = da;
            p.lda = s.lda;
            p.a_rows = s.M;
            p.W = dw;
            p.M = s.M;
            p.N = s.N;
            p.K = s.K;
            p.n16 = s.n16;
            p.n32 = s.n32;
            p.c16 = d16;
            p.c32 = (float *)d32;
            p.glu = dg;
            p.ld16 = ld16;
            p.ld32 = ld32;
            p.ldg = ldg;
            p.splits = s.splits;
            for (int i = 0; s.splits > 1 && i <= s.splits; i++) p.kb[i] = s.kb[i];
            p.longest_first = s.longest_first;
            p.c32_rows = s.M * s.splits;
            p.tile = tile;
            if (launch_seg_gemm(&ctx, MOON_DTYPE_BF16, p) != MOON_OK || hipStreamSynchronize(ctx.stream) != hipSuccess) return printf("launch: %s\n", ctx.err.c_str()), 2;
            (void)hipMemcpy(c16.data(), d16, n16 * 2, hipMemcpyDeviceToHost);
            (void)hipMemcpy(c32.data(), d32, n32 * 4, hipMemcpyDeviceToHost);
            (void)hipMemcpy(cg.data(), dg, ng * 2, hipMemcpyDeviceToHost);
            if (tile == 2) {
                first16 = c16;
                first32 = c32;
                first_g = cg;
            }
            checked++;
            if (c16 != first16 || c32 != first32 || cg != first_g) failures++, printf("FAILED: other bits than in 128-row tiles\n");
            auto outside = [&](auto &v, int rows, int ld, int used) {
                for (size_t i = 0; i < v.size(); i++)
                    if ((int(i / ld) >= rows || int(i % ld) >= used) && (v[i] & 0xffff) != 0x5a5a) return true;
                return false;
            };
            if (outside(c16, s.M, ld16, s.n16) || outside(c32, s.M * s.splits, ld32, s.n32 - s.n16) || outside(cg, s.M, ldg, (s.N - s.n32) / 2)) failures++, printf("FAILED: written outside of the result\n");
        }
        // bf16 results (8 bits): half a unit in the last place is at most 2^-8 of the value, and a little for the f32 sums; f32 ones 1e-6 of the sum of magnitudes
        for (int i = 0; i < 2000; i++) {
            const int m = i < 200 ? s.M - 1 - i % std::min(s.M, 7) : int(rng() % s.M), n = i % 5 ? int(rng() % s.N) : s.N - 1 - i % 64;
            auto dot = [&](int col, double &size) {
                double t = 0;
                size = 0;
                for (int k = 0; k < s.K; k++) {
                    const double x = double(widen(a[size_t(m) * s.lda + k])) * widen(w[size_t(col) * s.K + k]);
                    t += x;
                    size += std::fabs(x);
                }
                return t;
            };
            double size, size_up, want = dot(n, size), got = 0, limit;
            if (n < s.n16) {
                got = widen(first16[size_t(m) * ld16 + n]);
                limit = std::fabs(want) / 256 + 1e-6 * size;
            } else if (n < s.n32) {
                for (int r = 0; r < s.splits; r++) {
                    float f;
                    memcpy(&f, &first32[size_t(r * s.M + m) * ld32 + n - s.n16], 4);
                    got += f;
                }
                limit = 1e-6 * size;
            } else {
                const int at = n - s.n32, j = at / 64 * 32 + at % 32, gate = s.n32 + at / 64 * 64 + at % 32;
                const double g = dot(gate, size), u = dot(gate + 32, size_up);
                want = g / (1 + std::exp(-g)) * u;
                got = widen(first_g[size_t(m) * ldg + j]);
                limit = std::fabs(want) / 256 + 2e-6 * (size + 1) * (size_up + 1); // |silu'| < 1.1
            }
            checked++;
            if (!(std::fabs(got - want) <= limit) && failures++ < 20) printf("FAILED: (%d, %d) %g, should be %g\n", m, n, got, want);
        }
        (void)hipFree(da);
        (void)hipFree(dw);
        (void)hipFree(d16);
        (void)hipFree(d32);
        (void)hipFree(dg);
    }
    unsigned *other, n_other = 1;
    if (hipMalloc((void **)&other, 4) || hipMemset(other, 0, 4)) return printf("no memory\n"), 2;
    silu_check<<<4096, 256, 0, ctx.stream>>>(other);
    if (hipStreamSynchronize(ctx.stream) || hipMemcpy(&n_other, other, 4, hipMemcpyDeviceToHost)) return printf("silu\n"), 2;
    checked++;
    if (n_other) failures++, printf("FAILED: silu, %u values with other bits\n", n_other);
    printf("%d checks, %d failures\n", checked, failures);
    return failures != 0;
}
