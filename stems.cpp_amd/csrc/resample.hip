// resample.hip — band-limited resampling on gfx950.
//
// Reference: st::resample_planar (src/audio.h:17-59): a Kaiser-windowed sinc (beta 8.6, 32 zero
// crossings, cutoff 0.95 of the lower Nyquist), tabulated once over |x| in [0, half] at 2^15 + 2
// points and interpolated linearly; each output sample sums, in double and in input order, the
// weighted input samples within `half` of its position. Two kernels. The default one,
// resample_phase_kernel (below), weights each output by its exact phase, on the matrix cores; the per-tap one,
// resample_kernel, chosen by STX_RESAMPLE_EXACT=1 and for very short inputs, computes the table on the host with the
// reference's formula (so it is bit-identical), keeps it on the device, and does every per-tap
// operation as the reference's double operation in the reference's order, so its output is
// bit-identical. One thread per output sample and every channel; taps go in groups of eight
// whose loads are issued together (clamped addresses; a tap past the window, or one the
// reference skips, adds +0.0, an exact no-op on a sum that starts at +0.0). The per-tap
// division by `half` is done as a multiplication by r = RN(1/half) and one fma correction,
// q = RN(q0 + r RN(x - q0 half)) with q0 = RN(x r), which is the correctly rounded quotient
// (Markstein's theorem: r within half an ulp of 1/half, q0 within one ulp of x/half, residual
// exact by the fma), so bit-identical to IEEE division at a fraction of its cost.
#include <algorithm>
#include <cmath>
#include <cstdlib>
#include <numeric>
#include <type_traits>
#include <vector>

#include "common.hpp"
#include "resample.hpp"

struct stx_resampler {
    int src = 0, dst = 0;
    double ratio = 1.0, half = 0.0;
    double* d_table = nullptr;       // [kTableN + 2]
    // Phase tables (see resample_phase_kernel): dst = up * g, src = down * g, U = m up, D = m down.
    int U = 0, D = 0;
    int omin = 0;                    // offset of tap 0 from floor(c)
    int groups = 0, ks = 0;          // groups of 16 phases; products per group
    int width = 0, pitch = 0;        // staged row of one period
    long long lds_max = 0;           // LDS per workgroup of the device
    double* d_weights = nullptr;     // [groups][ks][64]
    int* d_goff = nullptr;           // [groups]
    int2* d_range = nullptr;         // [U]
};

namespace stx {
namespace {

constexpr int kTableN = 1 << 15;
constexpr int kTapGroup = 8;

struct ResampleArgs {
    const float* in;                 // [C][n]
    float* out;                      // [C][out_n]
    const double* table;
    double ratio, half, rhalf;       // rhalf = RN(1 / half)
    int n, out_n, C;
};


template <int NC>
__global__ __launch_bounds__(256) void resample_kernel(ResampleArgs a) {
#pragma clang fp contract(off)
    const int i = (int)(blockIdx.x * 256 + threadIdx.x);
    if (i >= a.out_n) return;
    const int C = NC > 0 ? NC : a.C;
    const double c = i / a.ratio;                                   // src/audio.h:43-46
    const int lo = max(0, (int)ceil(c - a.half)), hi = min(a.n - 1, (int)floor(c + a.half));
    constexpr int MC = NC > 0 ? NC : 8;
    double acc[MC];
#pragma unroll
    for (int k = 0; k < MC; k++) acc[k] = 0.0;
    for (int j0 = lo; j0 <= hi; j0 += kTapGroup) {
        double w[kTapGroup];
        bool use[kTapGroup];
        float x[kTapGroup][MC];
#pragma unroll
        for (int q = 0; q < kTapGroup; q++) {
            const int j = min(j0 + q, hi);
            const double pos = div_rn(fabs(j - c), a.half, a.rhalf) * kTableN;
            const int t = min((int)pos, kTableN);
            const double fr = pos - t;
            const double t0 = a.table[t], t1 = a.table[t + 1];
#pragma unroll
            for (int k = 0; k < MC; k++) x[q][k] = k < C ? a.in[(size_t)k * a.n + j] : 0.0f;
            w[q] = t0 + (t1 - t0) * fr;
            use[q] = j0 + q <= hi && (int)pos < kTableN;   // past the window, or t >= table_n (:49)
        }
#pragma unroll
        for (int q = 0; q < kTapGroup; q++)
#pragma unroll
            for (int k = 0; k < MC; k++) {
                const double p = w[q] * (double)x[q][k];
                acc[k] = acc[k] + (use[q] ? p : 0.0);
            }
    }
#pragma unroll
    for (int k = 0; k < MC; k++)
        if (k < C) store_stream(a.out + (size_t)k * a.out_n + i, (float)acc[k]);
}

// The same sums over weights that depend only on the output's phase, as products on the matrix
// cores. With dst = up g and src = down g, and U = m up, D = m down for a whole m, output
// i = q + M U sits at c = i down / up = fq + M D + p / up, where fq = floor(q down / up) and
// p = q down mod up, so its taps j = fq + M D + omin + k and their weights (the reference's table
// interpolation at |j - c|) are row p of a table of up rows computed once on the host. Those
// weights differ from the reference's, which it computes per output from c = i / ratio with ratio
// rounded to double, by the rounding of c (below 1e-9 for three hours of 48 kHz audio), so the
// output is within a few float ulps of the reference's (SNR above 160 dB) instead of bit-identical.
//
// Sixteen neighbouring outputs q = 16 g .. 16 g + 15 of a period read one window of 4 ks samples
// that starts at F = f(16 g) and holds all their taps, so for 16 periods M the outputs are
//   Y[M][q] = sum over s < 4 ks of X[M D + F + s] W_g[s][q],
// ks products v_mfma_f64_16x16x4_f64 (double operands and sums; W_g is zero outside a phase's own
// taps). A workgroup takes R = 16 T periods of one channel and stages in LDS one row of `width`
// samples per period (neighbouring rows overlap; rows are `pitch` floats apart, 2 mod 4, so that the
// 32 lanes that read 16 rows at two neighbouring samples touch 32 banks: no conflicts measured). A wave
// takes groups g and all T tiles of 16 periods: a weight operand (one double a lane, 512 contiguous
// bytes from the cache, a step of four ahead) feeds T products, a sample operand is one LDS read and
// one conversion.
//
// The double matrix rate (69 TFLOP/s measured) is a floor of 16 ceil(U / 16) / U more outputs and
// 4 ks / taps more taps than the sum needs (1.09 and 1.30 for 48 -> 44.1 kHz, 180 s stereo: 48 us); it
// takes 81 us there, staging, weights and stores sharing the vector memory pipe (47 us without the
// products). One fma per tap on the vector units, which this took the place of, issued a conversion
// for every two fmas and waited on LDS (115 us), left waves idle at ratios of few phases (2 : 1, 60 s
// stereo: 943 -> 52 us), and its tile of 64 whole periods did not fit at 44.1 -> 8 kHz (350 -> 34 us).
// Measured and dropped: ten waves (one a group) instead of eight at 44.1 -> 48 kHz, 70 against 61 us;
// rows staged through registers, 96 us; four tiles a wave, 92 us; weights held in registers by
// persistent workgroups with the next tile's rows on their way, 85 us (96 registers spill, and the
// compiler waits for the rows before the first LDS read).
//
// A zero weight times an infinity or NaN is NaN, where the phase's own window may have no such tap;
// finite samples never give a sum that is not finite (weights of at most 1, doubles). So where a sum
// is not finite the wave sums its outputs again, each over its own taps alone, in tap order.
struct PhaseArgs {
    const float* in;                 // [C][n]
    float* out;                      // [C][out_n]
    const double* w;                 // [groups][ks][64]: lane l holds tap 4 s + l / 16 of phase 16 g + l mod 16
    const int* goff;                 // [groups]: F
    const int2* range;               // [U]: first and last tap of each phase, counted from its group's F
    long long n, out_n;
    int U, D, omin, groups, ks;
    int width, pitch;                // staged samples per period; floats between rows (2 mod 4)
};

constexpr int kPhaseMaxWaves = 8;                    // a multiple of the CU's four SIMDs
constexpr long long kPhaseMaxWeights = 1 << 18;      // up * ntap above this: per-tap kernel
constexpr long long kPhaseMaxTable = 1 << 20;        // doubles of the groups' tables above this: per-tap kernel
constexpr int kPhaseUnroll = 4;                      // ks is a multiple of it

// The table does not change while the kernel runs: read through the constant address space, a
// wave-uniform load of it is a scalar load.
typedef const __attribute__((address_space(4))) int* ConstInts;
typedef __attribute__((address_space(1))) unsigned* GlobalWords;
typedef __attribute__((address_space(3))) unsigned* LocalWords;
typedef double stx_v4d __attribute__((ext_vector_type(4)));

// Stages rows [0, R) of the tile that starts at period m0: row l holds input (m0 + l) D + omin + r for
// r < width, zeros outside the input. Each wave takes whole rows. A row inside the input goes
// straight to LDS (64 samples an instruction, all in flight together; the caller waits for them),
// one at the input's ends through registers with a bounds test.
template <int R>
__device__ __forceinline__ void phase_stage(const PhaseArgs& a, const float* in, long long m0, float* xs, int wave, int waves,
                                            int lane) {
    for (int l = wave; l < R; l += waves) {
        const long long jb = (m0 + l) * a.D + a.omin;           // input index of r = 0
        const float* src = in + jb;
        float* dst = xs + l * a.pitch;
        if (jb >= 0 && jb + a.width <= a.n) {
            for (int r0 = 0; r0 < a.width; r0 += 64)
                if (r0 + lane < a.width)
                    __builtin_amdgcn_global_load_lds((GlobalWords)(src + r0 + lane), (LocalWords)(dst + r0), 4, 0, 0);
        } else {
            for (int r = lane; r < a.width; r += 64) {
                const long long j = jb + r;
                dst[r] = j >= 0 && j < a.n ? in[j] : 0.0f;
            }
        }
    }
}

// Writes group g's sums of T tiles of 16 periods (lane l's sums v are those of period
// l / 16 + 4 v of a tile, phase l mod 16); outp is output 0 of the first period, xg the group's
// window in its row and `left` the outputs from outp to the end.
template <int T>
__device__ __forceinline__ void phase_store(const PhaseArgs& a, const stx_v4d (&acc)[T], float* outp, int left, const float* xg,
                                            int g, int lane) {
    const int lm = lane & 15, lk = lane >> 4, q = 16 * g + lm;
    bool bad = false;
#pragma unroll
    for (int t = 0; t < T; t++)
#pragma unroll
        for (int v = 0; v < 4; v++) bad |= !isfinite(acc[t][v]);
    if (__ballot(bad) != 0) {
        // In a branch of its own, so that the stores of the usual case wait for nothing.
        if (q >= a.U) return;
        const int2 rg = a.range[q];
        const double* w = a.w + (size_t)g * a.ks * 64 + lm;
        for (int row = lk; row < 16 * T && row * a.U + q < left; row += 4) {
            const float* xw = xg + row * a.pitch;
            double y = 0.0;
            for (int k = rg.x; k <= rg.y; k++) y = fma(w[(k >> 2) * 64 + (k & 3) * 16], (double)xw[k], y);
            outp[row * a.U + q] = (float)y;
        }
        return;
    }
    if (q >= a.U) return;
#pragma unroll
    for (int t = 0; t < T; t++)
#pragma unroll
        for (int v = 0; v < 4; v++) {
            const int i = (16 * t + 4 * v + lk) * a.U + q;
            if (i < left) outp[i] = (float)acc[t][v];
        }
}

// Bounds of 128 registers keep the sums in architectural registers: with a larger budget the
// compiler moves them to accumulation registers and back around every loop step.
template <int T>
__global__ __launch_bounds__(kPhaseMaxWaves * 64) __attribute__((amdgpu_waves_per_eu(4))) void resample_phase_kernel(PhaseArgs a) {
    extern __shared__ float xs[];
    constexpr int R = 16 * T;
    const int c = (int)blockIdx.y;
    const long long m0 = (long long)blockIdx.x * R;
    const int lane = (int)threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
    const int waves = (int)blockDim.x >> 6;
    phase_stage<R>(a, a.in + (size_t)c * a.n, m0, xs, wave, waves, lane);
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");            // this wave's rows have landed
    __syncthreads();
    float* outp = a.out + (size_t)c * a.out_n + m0 * a.U;
    const int left = (int)min(a.out_n - m0 * a.U, (long long)R * a.U);
    for (int g = wave + waves * (int)blockIdx.z; g < a.groups; g += waves * (int)gridDim.z) {
        const int F = ((ConstInts)a.goff)[g];
        stx_v4d acc[T];
#pragma unroll
        for (int t = 0; t < T; t++) acc[t] = stx_v4d{0.0, 0.0, 0.0, 0.0};
        const float* xr = xs + (lane & 15) * a.pitch + F + (lane >> 4);
        const int tile = 16 * a.pitch;
        const double* wl = a.w + (size_t)g * a.ks * 64 + lane;
        double wn[kPhaseUnroll];
#pragma unroll
        for (int u = 0; u < kPhaseUnroll; u++) wn[u] = wl[64 * u];
        for (int s = 0; s < a.ks; s += kPhaseUnroll) {
            double wc[kPhaseUnroll];
            // The next step's weights in flight through this one's products (the last step
            // re-reads its own).
            const double* wx = wl + 64 * (s + kPhaseUnroll < a.ks ? s + kPhaseUnroll : s);
#pragma unroll
            for (int u = 0; u < kPhaseUnroll; u++) wc[u] = wn[u];
#pragma unroll
            for (int u = 0; u < kPhaseUnroll; u++) wn[u] = wx[64 * u];
            float x[kPhaseUnroll][T];
#pragma unroll
            for (int t = 0; t < T; t++)
#pragma unroll
                for (int u = 0; u < kPhaseUnroll; u++) x[u][t] = xr[t * tile + 4 * (s + u)];
#pragma unroll
            for (int u = 0; u < kPhaseUnroll; u++)
#pragma unroll
                for (int t = 0; t < T; t++)
                    acc[t] = __builtin_amdgcn_mfma_f64_16x16x4f64((double)x[u][t], wc[u], acc[t], 0, 0, 0);
        }
        phase_store(a, acc, outp, left, xs + F, g, lane);
    }
}

// The period multiple m and the shape of the tables for a ratio up / down with ntap taps a phase.
struct PhaseShape {
    int m = 0, groups = 0, ks = 0, width = 0, pitch = 0;
};

// f(q) = floor(q down / up).
inline int phase_floor(int q, int up, int down) { return (int)((long long)q * down / up); }

// m: more than one period where the period alone wastes columns of its last group (U not a
// multiple of 16) or has too few groups to give the waves of a workgroup one each (8), as long as
// the rows stay short enough for 32 of them in half the LDS (two workgroups a CU). The cost of each
// candidate is its padding times a factor for what it misses; the smallest m of least cost is
// taken. m = 0: no shape fits `budget` bytes of LDS with 16 rows.
PhaseShape phase_shape(int up, int down, int ntap, long long budget) {
    PhaseShape best;
    double least = 0.0;
    for (int m = 1; m <= 128; m++) {
        const long long U = (long long)m * up, D = (long long)m * down;
        if (m > 1 && (U > 1024 || D > 4096)) break;
        const int groups = (int)((U + 15) / 16);
        int span = 0, last = 0;
        for (int g = 0; g < groups; g++) {
            last = phase_floor(16 * g, up, down);
            span = std::max(span, phase_floor((int)std::min<long long>(16LL * g + 15, U - 1), up, down) - last);
        }
        const int ks = (ntap + span + 4 * kPhaseUnroll - 1) / (4 * kPhaseUnroll) * kPhaseUnroll;
        const int width = last + 4 * ks, pitch = width + (6 - width % 4) % 4;   // the next 2 mod 4
        if (16LL * pitch * 4 > budget) break;                  // rows only grow with m
        double cost = 16.0 * groups / (double)U;
        if (groups < 8) cost *= 1.0 + 0.05 * (8 - groups);
        if (32LL * pitch * 4 > budget / 2) cost *= 1.15;
        if (best.m == 0 || cost < least - 1e-9) {
            best = PhaseShape{m, groups, ks, width, pitch};
            least = cost;
        }
    }
    return best;
}

__global__ __launch_bounds__(256) void copy_kernel(const float* __restrict__ in, float* __restrict__ out, size_t n) {
    for (size_t e = (size_t)blockIdx.x * 256 + threadIdx.x; e < n; e += (size_t)gridDim.x * 256) out[e] = in[e];
}

double bessel_i0(double x) {
    double s = 1, t = 1;
    for (int k = 1; k < 30; k++) {
        t *= (x / (2 * k)) * (x / (2 * k));
        s += t;
    }
    return s;
}

void check_resampler(const stx_resampler* r) { STX_REQUIRE(r != nullptr, "null resampler"); }

}  // namespace

void resampler_rates(const stx_resampler* r, int& src, int& dst) {
    check_resampler(r);
    src = r->src;
    dst = r->dst;
}

}  // namespace stx

using namespace stx;

extern "C" {

STX_API stx_status stx_resampler_create(int src_rate, int dst_rate, stx_resampler** out) {
    return guard([&] {
        STX_REQUIRE(out != nullptr, "out is NULL");
        *out = nullptr;
        STX_REQUIRE(src_rate > 0 && dst_rate > 0, "sample rates must be positive");
        // LDS per workgroup of the current device: the phase kernel's staged tile must fit.
        int dev = 0, lds_max = 0;
        hip_check(hipGetDevice(&dev), "hipGetDevice");
        hip_check(hipDeviceGetAttribute(&lds_max, hipDeviceAttributeMaxSharedMemoryPerBlock, dev),
                  "hipDeviceGetAttribute");
        stx_resampler* r = new stx_resampler;
        r->src = src_rate;
        r->dst = dst_rate;
        r->ratio = (double)dst_rate / src_rate;
        if (src_rate != dst_rate) {                                  // src/audio.h:20-38
            const double cutoff = 0.95 * std::min(1.0, r->ratio);
            const int zc = 32;
            const double half = zc / cutoff;
            const double beta = 8.6;
            const double i0b = bessel_i0(beta);
            std::vector<double> table(kTableN + 2);
            for (int t = 0; t <= kTableN + 1; t++) {
                const double x = std::min((double)t / kTableN, 1.0) * half;
                const double rr = x / half;
                const double arg = M_PI * x * cutoff;
                const double sinc = arg < 1e-12 ? 1.0 : std::sin(arg) / arg;
                table[t] = rr >= 1 ? 0.0 : sinc * bessel_i0(beta * std::sqrt(1 - rr * rr)) / i0b * cutoff;
            }
            r->half = half;
            // Phase table: output i = q + M up has c = i down / up = floor(q down / up) + M down
            // + p / up with p = q down mod up; its taps are j = floor(c) + o for o in
            // [ceil(p/up - half), floor(p/up + half)], each weighted as the reference weights
            // |j - c| (src/audio.h:47-52), skipped where the table index reaches table_n.
            const int g = std::gcd(src_rate, dst_rate);
            const int up = dst_rate / g, down = src_rate / g;
            const int omin = -(int)std::floor(half), omax = (int)std::floor(half) + 1;
            const int ntap = omax - omin + 1;
            std::vector<double> weights;
            std::vector<int> goff;
            std::vector<int2> range;
            const long long budget = lds_max - 1024;                 // beside the kernel's static LDS
            PhaseShape shape;
            if ((long long)up * ntap <= kPhaseMaxWeights) shape = phase_shape(up, down, ntap, budget);
            // Above 64 KB a kernel is allowed that much dynamic LDS first.
            auto allow = [&](const void* k) {
                if (hipFuncSetAttribute(k, hipFuncAttributeMaxDynamicSharedMemorySize, (int)budget) == hipSuccess) return true;
                (void)hipGetLastError();
                return false;
            };
            if (shape.m > 0 && !(allow((const void*)resample_phase_kernel<1>) && allow((const void*)resample_phase_kernel<2>)))
                shape.m = 0;
            if (shape.m > 0 && (long long)shape.groups * shape.ks * 64 <= kPhaseMaxTable) {
                std::vector<double> phase((size_t)up * ntap, 0.0);
                std::vector<int2> taps(up, make_int2(0, -1));
                for (int p = 0; p < up; p++) {
                    const double frac = (double)p / up;
                    int lo = ntap, hi = -1;
                    for (int k = 0; k < ntap; k++) {
                        const int o = omin + k;
                        if (o < (int)std::ceil(frac - half) || o > (int)std::floor(frac + half)) continue;
                        const double pos = std::fabs(o - frac) / half * kTableN;
                        const int t = (int)pos;
                        if (t >= kTableN) continue;
                        phase[(size_t)p * ntap + k] = table[t] + (table[t + 1] - table[t]) * (pos - t);
                        lo = std::min(lo, k);
                        hi = std::max(hi, k);
                    }
                    taps[p] = make_int2(lo, hi);
                }
                const int U = shape.m * up;
                weights.assign((size_t)shape.groups * shape.ks * 64, 0.0);
                goff.resize(shape.groups);
                range.resize(U);
                for (int q = 0; q < U; q++) {
                    const int g = q / 16, F = phase_floor(16 * g, up, down), d = phase_floor(q, up, down) - F;
                    const int p = (int)((long long)q * down % up);
                    goff[g] = F;
                    range[q] = make_int2(taps[p].x + d, taps[p].y + d);
                    double* wg = weights.data() + (size_t)g * shape.ks * 64;
                    for (int k = taps[p].x; k <= taps[p].y; k++)
                        wg[(k + d) / 4 * 64 + (k + d) % 4 * 16 + q % 16] = phase[(size_t)p * ntap + k];
                }
                r->U = U;
                r->D = shape.m * down;
                r->omin = omin;
                r->groups = shape.groups;
                r->ks = shape.ks;
                r->width = shape.width;
                r->pitch = shape.pitch;
                r->lds_max = budget;
            }
            hipError_t e = hipMalloc(&r->d_table, sizeof(double) * table.size());
            if (e == hipSuccess)
                e = hipMemcpy(r->d_table, table.data(), sizeof(double) * table.size(), hipMemcpyHostToDevice);
            auto upload = [&](auto*& d, const auto& h) {
                if (e == hipSuccess) e = hipMalloc(&d, sizeof(h[0]) * h.size());
                if (e == hipSuccess) e = hipMemcpy(d, h.data(), sizeof(h[0]) * h.size(), hipMemcpyHostToDevice);
            };
            if (!weights.empty()) {
                upload(r->d_weights, weights);
                upload(r->d_goff, goff);
                upload(r->d_range, range);
            }
            if (e != hipSuccess) {
                stx_resampler_destroy(r);
                hip_check(e, "stx_resampler_create");
            }
        }
        *out = r;
    });
}

STX_API void stx_resampler_destroy(stx_resampler* r) {
    if (!r) return;
    if (r->d_table) (void)hipFree(r->d_table);
    if (r->d_weights) (void)hipFree(r->d_weights);
    if (r->d_goff) (void)hipFree(r->d_goff);
    if (r->d_range) (void)hipFree(r->d_range);
    delete r;
}

STX_API int64_t stx_resample_length(const stx_resampler* r, int64_t n) {
    if (!r || n < 0) return -1;
    if (r->src == r->dst) return n;
    return (int64_t)std::llround((double)n * r->ratio);              // src/audio.h:20: llround(n * ratio) with int n
}

STX_API stx_status stx_resample(const stx_resampler* r, const float* in, int channels, int64_t n, float* out,
                                stx_stream stream) {
    return guard([&] {
        check_resampler(r);
        STX_REQUIRE(channels >= 1 && n >= 0, "bad channels/n");
        STX_REQUIRE(n < (1LL << 31) && (long long)channels * n < (1LL << 40), "input too long");
        if (n == 0) return;
        STX_REQUIRE(in && out, "NULL buffer");
        const hipStream_t s = as_stream(stream);
        if (r->src == r->dst) {                                      // src/audio.h:19: the input as it is
            const size_t count = (size_t)channels * n;
            hipLaunchKernelGGL(copy_kernel, dim3((unsigned)std::min<size_t>((count + 255) / 256, 1 << 20)), dim3(256),
                               0, s, in, out, count);
            launch_check("copy_kernel");
            return;
        }
        const int64_t out_n = stx_resample_length(r, n);
        STX_REQUIRE(out_n < (1LL << 31), "output too long");
        if (out_n == 0) return;
        if (channels > 8) fail(STX_STATUS_UNSUPPORTED, "resample: more than 8 channels");
        // The phase table unless STX_RESAMPLE_EXACT=1 (read at each call) asks for the per-tap
        // kernel, which gives the reference's bits.
        const char* exact = std::getenv("STX_RESAMPLE_EXACT");
        // An input shorter than half a window (stereo: three eighths of one) has few taps in all, and the phase kernel
        // takes whole windows: 44.1 -> 8 kHz, 100 samples 9.8 us per tap, 14.6 by phases; 185 samples 14.5 and 14.6.
        const bool brief = channels <= 2 && (double)n <= r->half * (channels == 1 ? 1.0 : 0.75);
        if (r->d_weights && !brief && !(exact && exact[0] == '1')) {
            const PhaseArgs pa{in, out, r->d_weights, r->d_goff, r->d_range, n, out_n, r->U, r->D, r->omin, r->groups,
                               r->ks, r->width, r->pitch};
            const long long periods = (out_n + r->U - 1) / r->U;
            const int waves = std::min(r->groups, kPhaseMaxWaves);
            auto go = [&](auto tiles) {
                constexpr int T = decltype(tiles)::value;
                // Calls of fewer workgroups than CUs: waves that would take several groups in turn share them with further
                // workgroups on the same rows (192 -> 44.1 kHz, 1,000 samples: 33.7 -> 15.4 us).
                const long long blocks = (periods + 16 * T - 1) / (16 * T);
                const long long turns = (r->groups + waves - 1) / waves;
                const long long z = std::max(1LL, std::min(turns, device_cus() / (blocks * channels)));
                const dim3 grid((unsigned)blocks, (unsigned)channels, (unsigned)z);
                hipLaunchKernelGGL(resample_phase_kernel<T>, grid, dim3(waves * 64), (unsigned)(16 * T * r->pitch * 4), s, pa);
            };
            // Two tiles of 16 periods where their rows leave room for two workgroups a CU and there
            // are two workgroups for each CU of the device (a weight operand then feeds two products).
            if (32LL * r->pitch * 4 <= r->lds_max / 2 && (periods + 31) / 32 * channels >= 2LL * device_cus())
                go(std::integral_constant<int, 2>{});
            else
                go(std::integral_constant<int, 1>{});
            launch_check("resample_phase_kernel");
            return;
        }
        ResampleArgs a{in, out, r->d_table, r->ratio, r->half, 1.0 / r->half, (int)n, (int)out_n, channels};
        const dim3 grid((unsigned)((out_n + 255) / 256));
        if (channels == 1) hipLaunchKernelGGL(resample_kernel<1>, grid, dim3(256), 0, s, a);
        else if (channels == 2) hipLaunchKernelGGL(resample_kernel<2>, grid, dim3(256), 0, s, a);
        else hipLaunchKernelGGL(resample_kernel<0>, grid, dim3(256), 0, s, a);
        launch_check("resample_kernel");
    });
}

}  // extern "C"
