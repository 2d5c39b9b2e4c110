// The mel front end (Mel/MelSpectrogram.cpp) on gfx950: 16 kHz samples in,
// the normalised log-mel the encoder's first convolution reads out.
//
//   frames[f][t] = reflect-padded samples[f·hop + t - fft/2] · hann[t]
//   spectrum     = frames · basis^T          basis rows cos / -sin per bin
//   power[f][b]  = re^2 + im^2               (the non-redundant half)
//   mel[f][m]    = power · filters^T         the published filterbank
//   out[m][f]    = (max(log10 max(mel, 1e-10), peak - 8) + 4) / 4
//
// The transform is a product against a DFT basis built once in double on the
// host (as the reference's SpectrumProduct is); the window is the periodic
// Hann (Tests/Mel/ScalarMel.h:20-28) and the padding numpy's "reflect" folded
// into the frame index (Tests/Mel/ScalarMel.h:32-49). Everything up to the
// logarithm is one launch (spectrogram_kernel); transforms too long for its
// LDS run as launches over the library's products.
#include "../../include/wsp_hip.h"
#include "device_common.h"
#include "ops.h"

#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstdio>
#include <new>
#include <vector>

namespace wsp::mel
{
namespace
{
constexpr int kThreads = 256;
constexpr int kLogBlocks = 512; // blocks of the log pass, each leaving one maximum

__global__ void __launch_bounds__(kThreads) frames_kernel(const float* __restrict__ samples, int count,
                                                          const float* __restrict__ window, int fft, int hop,
                                                          float* __restrict__ frames)
{
    const int f = blockIdx.x;
    for (int t = threadIdx.x; t < fft; t += kThreads)
    {
        int x = f * hop + t - fft / 2;
        if (x < 0)
            x = -x;
        if (x >= count)
            x = 2 * (count - 1) - x;
        frames[(size_t) f * fft + t] = samples[x] * window[t];
    }
}

// Sixteen frames a block, from samples to log10 of the bands, in LDS: the
// windowed samples folded, the half- or quarter-length transforms on the
// matrix cores (v_mfma_f32_16x16x4_f32: 16 bins by 16 frames), the power, the
// filterbank as another such product, the logarithm and the block's largest
// value.
//
// Folding: cos(2πbn/N) is even about n = N/2 and sin odd, so re needs
// e[n] = x[n] + x[N-n] and im o[n] = x[n] - x[N-n] for n up to H = N/2 only.
// With N a multiple of four both fold once more about H/2, differently for
// even and odd bins: even ones take e[n] + e[H-n] and o[n] - o[H-n], odd ones
// e[n] - e[H-n] and o[n] + o[H-n] (at H/2 itself the cosine of an odd bin and
// the sine of an even one are zero). That leaves a quarter of the products of
// the whole transform and of the basis to read (200 KB a block at 400 points).
//
// A wave takes tiles of 16 bins of one parity, then tiles of 16 bands; the
// filterbank is copied to LDS meanwhile. Each product step sums four
// consecutive n (and bins), in order: position 16j + 4g + e of an LDS row, and
// of the basis, holds n = 16j + 4e + g. The basis is fragment-major, one
// contiguous kilobyte a load. The 30 s window: 53 us as seven launches with the
// products on the vector units, 38.8 with them on the matrix cores, 23.9 in
// this launch folded once with the filters read from memory, 17.3 now; two
// launches that do nothing but move the data take about 9.
constexpr int kSpectrogramThreads = 512;
constexpr int kSpectrogramFrames = 16;
constexpr int kRuns = 4;   // 16-value runs a wave loads at a time
constexpr int kRowPad = 4; // floats: rows of 16j + 4 land eight 16-byte reads on eight bank groups

typedef float f32x4 __attribute__((ext_vector_type(4)));

// Where an LDS row (and the basis) keeps value n.
__host__ __device__ constexpr int place(int n)
{
    return n / 16 * 16 + 4 * (n % 4) + n % 16 / 4;
}

// How a transform of `fft` points folds, and the tiles that leaves.
struct Folds
{
    int parities; // 2: even and odd bins apart
    int values;   // n of a folded row
    int tiles;    // 16-value runs of a folded row, and 16-bin tiles of a parity
    int bin_tiles; // 16-bin runs of a power row

    __host__ __device__ explicit Folds(int fft)
    {
        const int half = fft / 2;
        parities = fft % 4 == 0 ? 2 : 1;
        values = parities == 2 ? half / 2 + 1 : half + 1;
        tiles = (values + 15) / 16;
        bin_tiles = (half + 16) / 16;
    }
    __host__ __device__ int folded_stride() const { return 16 * tiles + kRowPad; }
    __host__ __device__ int power_stride() const { return 16 * bin_tiles + kRowPad; }
    // Floats of the folded rows ([parity][cosine, sine][frame]) and the power rows.
    __host__ __device__ int lds_floats() const
    {
        return kSpectrogramFrames * (2 * parities * folded_stride() + power_stride());
    }
};

template <bool STAGED>
__global__ void __launch_bounds__(kSpectrogramThreads) spectrogram_kernel(
    const float* __restrict__ samples, int count, const float* __restrict__ window, int fft, int hop, int frames,
    const float* __restrict__ basis, const float* __restrict__ filters, int mels, float* __restrict__ out,
    float* __restrict__ peaks)
{
    extern __shared__ __attribute__((aligned(16))) float rows[];
    __shared__ float scratch[kSpectrogramThreads / kWave];
    const Folds folds(fft);
    const int half = fft / 2, bins = half + 1, tiles = folds.tiles;
    const int stride = folds.folded_stride(), power_stride = folds.power_stride();
    float* const power = rows + 2 * folds.parities * kSpectrogramFrames * stride; // [frame][place(bin)]
    float* const staged = rows + folds.lds_floats();                             // the filterbank as it is
    const int f0 = blockIdx.x * kSpectrogramFrames;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave), lane = threadIdx.x % kWave;
    const int li = lane % 16, g = lane / 16;

    if constexpr (STAGED)
    {
        // In flight until the bands' tiles; the last few values by hand.
        const int total = mels * bins, whole = total / 4 * 4;
        const uint32_t base = lds_address(staged);
        for (int i = 256 * wave; i < whole; i += 256 * (kSpectrogramThreads / kWave))
            if (i + 4 * lane < whole)
                load_lds16(filters, 4 * (i + 4 * lane), __builtin_amdgcn_readfirstlane(base + 4 * i));
        if ((int) threadIdx.x < total - whole)
            staged[whole + threadIdx.x] = filters[whole + threadIdx.x];
    }

    // A thread folds value n of four frames (all their loads in flight at
    // once); values past the last are the padding.
    constexpr int kValues = 128, kFramesEach = kSpectrogramFrames * kValues / kSpectrogramThreads;
    const int first = threadIdx.x / kValues * kFramesEach;
    for (int n = threadIdx.x % kValues; n < 16 * tiles; n += kValues)
    {
        const bool in = n < folds.values, twice = folds.parities == 2;
        // x[n], x[N-n] and, folding twice, x[H-n], x[H+n]; without a partner the value itself
        const bool pair = in && n > 0 && 2 * n != fft;
        const int t[4] = {in ? n : 0, pair ? fft - n : in ? n : 0, in && twice ? half - n : 0,
                          pair && twice ? half + n : 0};
        float w[4], x[kFramesEach][4];
#pragma unroll
        for (int k = 0; k < 4; ++k)
            w[k] = window[t[k]];
#pragma unroll
        for (int i = 0; i < kFramesEach; ++i)
#pragma unroll
            for (int k = 0; k < 4; ++k)
            {
                const int at = abs(min(f0 + first + i, frames - 1) * hop - half + t[k]);
                x[i][k] = samples[at >= count ? 2 * (count - 1) - at : at];
            }
#pragma unroll
        for (int i = 0; i < kFramesEach; ++i)
        {
            const float a = x[i][0] * w[0], b = x[i][1] * w[1], c = x[i][2] * w[2], d = x[i][3] * w[3];
            const float en = !in ? 0.f : pair ? a + b : a, on = pair ? a - b : 0.f;
            float* const row = rows + (first + i) * stride + place(n);
            constexpr int kNext = kSpectrogramFrames; // rows between one folded row and the next kind
            if (!twice)
            {
                row[0] = en;
                row[kNext * stride] = on;
                continue;
            }
            const bool middle = 2 * n == half;
            const float em = !in ? 0.f : pair ? c + d : c, om = pair ? c - d : 0.f;
            row[0] = middle ? en : en + em;
            row[kNext * stride] = middle ? 0.f : on - om;
            row[2 * kNext * stride] = middle ? 0.f : en - em;
            row[3 * kNext * stride] = middle ? on : on + om;
        }
    }
    __syncthreads();

    // Runs of the basis (and of the filters) are loaded kRuns ahead of their
    // products; runs past the last repeat it and are not multiplied.
    for (int unit = wave; unit < folds.parities * tiles; unit += kSpectrogramThreads / kWave)
    {
        const int parity = unit % folds.parities, t = unit / folds.parities;
        const f32x4* from = reinterpret_cast<const f32x4*>(basis) + (size_t) (parity * tiles + t) * tiles * 2 * kWave
                            + lane;
        const float* even = rows + 2 * parity * kSpectrogramFrames * stride + li * stride + 4 * g;
        const float* odd = even + kSpectrogramFrames * stride;
        f32x4 re = {0.f, 0.f, 0.f, 0.f}, im = {0.f, 0.f, 0.f, 0.f};
        f32x4 c[2][kRuns], s[2][kRuns];
        auto load = [&](int j0, int set) {
#pragma unroll
            for (int i = 0; i < kRuns; ++i)
            {
                const int j = min(j0 + i, tiles - 1);
                c[set][i] = from[(size_t) (2 * j) * kWave];
                s[set][i] = from[(size_t) (2 * j + 1) * kWave];
            }
        };
        auto multiply = [&](int j0, int set) {
#pragma unroll
            for (int i = 0; i < kRuns; ++i)
            {
                if (j0 + i >= tiles)
                    break;
                const f32x4 e = *reinterpret_cast<const f32x4*>(even + 16 * (j0 + i));
                const f32x4 o = *reinterpret_cast<const f32x4*>(odd + 16 * (j0 + i));
#pragma unroll
                for (int k = 0; k < 4; ++k)
                {
                    re = __builtin_amdgcn_mfma_f32_16x16x4f32(c[set][i][k], e[k], re, 0, 0, 0);
                    im = __builtin_amdgcn_mfma_f32_16x16x4f32(s[set][i][k], o[k], im, 0, 0, 0);
                }
            }
        };
        load(0, 0);
        for (int j0 = 0; j0 < tiles; j0 += 2 * kRuns)
        {
            load(j0 + kRuns, 1);
            multiply(j0, 0);
            load(j0 + 2 * kRuns, 0);
            multiply(j0 + kRuns, 1);
        }
        // Lane (li, g) holds frame li's bins 16t + 4g + r of this parity.
#pragma unroll
        for (int r = 0; r < 4; ++r)
        {
            const int bin = folds.parities * (16 * t + 4 * g + r) + parity;
            if (bin < 16 * folds.bin_tiles)
                power[li * power_stride + place(bin)] = re[r] * re[r] + im[r] * im[r];
        }
    }
    if constexpr (STAGED)
        wait_loads<0>();
    __syncthreads();

    float best = -INFINITY;
    const int bands = (mels + 15) / 16;
    for (int t = wave; t < bands; t += kSpectrogramThreads / kWave)
    {
        const int from = min(16 * t + li, mels - 1) * bins;
        f32x4 sum = {0.f, 0.f, 0.f, 0.f};
        float w[2][kRuns][4];
        auto load = [&](int j0, int set) {
#pragma unroll
            for (int i = 0; i < kRuns; ++i)
#pragma unroll
                for (int k = 0; k < 4; ++k)
                {
                    const int at = from + min(16 * (j0 + i) + 4 * k + g, bins - 1);
                    w[set][i][k] = STAGED ? staged[at] : filters[at];
                }
        };
        auto multiply = [&](int j0, int set) {
#pragma unroll
            for (int i = 0; i < kRuns; ++i)
            {
                if (j0 + i >= folds.bin_tiles)
                    break;
                const f32x4 p = *reinterpret_cast<const f32x4*>(power + li * power_stride + 16 * (j0 + i) + 4 * g);
#pragma unroll
                for (int k = 0; k < 4; ++k)
                {
                    const bool in = 16 * (j0 + i) + 4 * k + g < bins; // (past the last bin both operands are zero)
                    sum = __builtin_amdgcn_mfma_f32_16x16x4f32(in ? w[set][i][k] : 0.f, in ? p[k] : 0.f, sum, 0, 0, 0);
                }
            }
        };
        load(0, 0);
        for (int j0 = 0; j0 < folds.bin_tiles; j0 += 2 * kRuns)
        {
            load(j0 + kRuns, 1);
            multiply(j0, 0);
            load(j0 + 2 * kRuns, 0);
            multiply(j0 + kRuns, 1);
        }
        const int f = f0 + li;
#pragma unroll
        for (int r = 0; r < 4; ++r)
        {
            const int m = 16 * t + 4 * g + r;
            if (m >= mels || f >= frames)
                continue;
            const float v = log10f(fmaxf(sum[r], 1e-10f));
            out[(size_t) m * frames + f] = v;
            best = fmaxf(best, v);
        }
    }
    best = block_max(best, scratch);
    if (threadIdx.x == 0)
        peaks[blockIdx.x] = best;
}

constexpr size_t kSpectrogramLds = 156 * 1024; // of a CU's 160 KB

size_t spectrogram_lds(int fft)
{
    return (size_t) Folds(fft).lds_floats() * sizeof(float);
}

// power rows have a stride of `padded` (bins rounded up to a multiple of 4,
// the padding left at zero) so the filterbank product takes vector loads.
__global__ void __launch_bounds__(kThreads) power_kernel(const float* __restrict__ spectrum, int bins, int padded,
                                                         int total, float* __restrict__ power)
{
    const int i = blockIdx.x * kThreads + threadIdx.x;
    if (i >= total)
        return;
    const int f = i / bins, b = i % bins;
    const float re = spectrum[(size_t) f * 2 * bins + 2 * b], im = spectrum[(size_t) f * 2 * bins + 2 * b + 1];
    power[(size_t) f * padded + b] = re * re + im * im;
}

// log10 of the [frames, mels] products into the band-major output, and each
// block's largest value into peaks[block].
__global__ void __launch_bounds__(kThreads) log_kernel(const float* __restrict__ rows, int frames, int mels,
                                                       float* __restrict__ out, float* __restrict__ peaks)
{
    __shared__ float scratch[kThreads / kWave];
    const int total = frames * mels;
    float best = -INFINITY;
    for (int i = blockIdx.x * kThreads + threadIdx.x; i < total; i += gridDim.x * kThreads)
    {
        const int m = i / frames, f = i % frames; // band-major index, so stores coalesce
        const float v = log10f(fmaxf(rows[(size_t) f * mels + m], 1e-10f));
        out[i] = v;
        best = fmaxf(best, v);
    }
    best = block_max(best, scratch);
    if (threadIdx.x == 0)
        peaks[blockIdx.x] = best;
}

__global__ void __launch_bounds__(kThreads) normalise_kernel(float* __restrict__ out, int total,
                                                             const float* __restrict__ peaks, int blocks)
{
    __shared__ float scratch[kThreads / kWave];
    float best = -INFINITY;
    for (int i = threadIdx.x; i < blocks; i += kThreads)
        best = fmaxf(best, peaks[i]);
    const float floor = block_max(best, scratch) - 8.f;
    for (int i = blockIdx.x * kThreads + threadIdx.x; i < total; i += gridDim.x * kThreads)
        out[i] = (fmaxf(out[i], floor) + 4.f) / 4.f;
}
} // namespace
} // namespace wsp::mel

struct wsp_mel
{
    wsp_mel_shape shape {};
    int device = 0;
    hipStream_t stream = nullptr;
    float* window = nullptr;   // [fft]
    float* folded = nullptr;   // spectrogram_kernel's basis: [bin tile][n / 16][cos, sin][lane][4]
    bool fused = false;        // one launch up to the logarithm; the rest of these then stay null
    float* basis = nullptr;    // [2 bins][fft]: cos, -sin
    float* frames = nullptr;   // [frames][fft]
    float* spectrum = nullptr; // [frames][2 bins]
    float* power = nullptr;    // [frames][padded bins], the padding zero
    float* filters = nullptr;  // [mels][padded bins]: the call's filterbank, the padding zero
    float* rows = nullptr;     // [frames][mels]
    float* peaks = nullptr;    // [kLogBlocks]
    std::vector<void*> owned;
    char error[512] = {0};
};

namespace
{
hipError_t mel_allocate(wsp_mel* m, float** out, size_t floats)
{
    void* p = nullptr;
    const hipError_t status = hipMalloc(&p, std::max<size_t>(floats, 1) * sizeof(float));
    if (status == hipSuccess)
    {
        m->owned.push_back(p);
        *out = static_cast<float*>(p);
    }
    return status;
}

int mel_hip(wsp_mel* m, hipError_t status, const char* what)
{
    if (status == hipSuccess)
        return WSP_OK;
    std::snprintf(m->error, sizeof m->error, "%s: %s", what, hipGetErrorString(status));
    return WSP_ERR_HIP;
}
} // namespace

extern "C" {

int wsp_mel_create(const wsp_mel_shape* shape, int device, void* stream, wsp_mel** out)
{
    if (shape == nullptr || out == nullptr)
        return WSP_ERR_ARGUMENT;
    *out = nullptr;
    const wsp_mel_shape& s = *shape;
    if (s.sample_count <= 0 || s.fft_length < 2 || s.hop_length <= 0 || s.frame_count <= 0 || s.mel_count <= 0)
        return WSP_ERR_ARGUMENT;
    // Reflect padding mirrors fft / 2 samples about each end, and the last
    // frame must start inside the padded signal.
    if (s.sample_count <= s.fft_length / 2 || (long long) (s.frame_count - 1) * s.hop_length > s.sample_count)
        return WSP_ERR_SHAPE;
    wsp_mel* m = new (std::nothrow) wsp_mel;
    if (m == nullptr)
        return WSP_ERR_HIP;
    m->shape = s;
    m->device = device;
    m->stream = static_cast<hipStream_t>(stream);
    const int fft = s.fft_length, bins = fft / 2 + 1;
    std::vector<float> window(fft), basis;
    const double two_pi = 2.0 * 3.14159265358979323846;
    for (int n = 0; n < fft; ++n)
        window[n] = (float) (0.5 * (1.0 - std::cos(two_pi * n / fft)));
    // the angle reduced modulo the period first, so it stays exact in double
    auto angle = [&](int b, int t) { return two_pi * (double) (((long long) b * t) % fft) / fft; };
    hipError_t status = hipSetDevice(device);
    if (status == hipSuccess)
        status = wsp::ops::prepare_split_products();
    if (status == hipSuccess)
        status = mel_allocate(m, &m->window, fft);
    if (status == hipSuccess)
        status = mel_allocate(m, &m->peaks, std::max(wsp::mel::kLogBlocks, (s.frame_count + 15) / 16));
    if (status == hipSuccess)
        status = hipMemcpy(m->window, window.data(), window.size() * sizeof(float), hipMemcpyHostToDevice);
    m->fused = wsp::mel::spectrogram_lds(fft) <= wsp::mel::kSpectrogramLds;
    if (m->fused)
    {
        const wsp::mel::Folds folds(fft);
        const int tiles = folds.tiles;
        basis.assign((size_t) folds.parities * tiles * tiles * 2 * 256, 0.f);
        for (int b = 0; b < bins; ++b)
            for (int n = 0; n < folds.values; ++n)
            {
                // lane (bin % 16, g), element e of run n / 16 stands for n = 16j + 4e + g
                const int parity = b % folds.parities, i = b / folds.parities;
                const size_t run = ((size_t) parity * tiles + i / 16) * tiles + n / 16;
                const size_t at = (run * 2 * 64 + 16 * (n % 4) + i % 16) * 4 + n % 16 / 4;
                basis[at] = (float) std::cos(angle(b, n));
                basis[at + 256] = (float) -std::sin(angle(b, n));
            }
        if (status == hipSuccess)
            status = mel_allocate(m, &m->folded, basis.size());
        if (status == hipSuccess)
            status = hipMemcpy(m->folded, basis.data(), basis.size() * sizeof(float), hipMemcpyHostToDevice);
        if (status == hipSuccess)
            status = hipFuncSetAttribute(reinterpret_cast<const void*>(&wsp::mel::spectrogram_kernel<true>),
                                         hipFuncAttributeMaxDynamicSharedMemorySize, (int) wsp::mel::kSpectrogramLds);
        if (status == hipSuccess)
            status = hipFuncSetAttribute(reinterpret_cast<const void*>(&wsp::mel::spectrogram_kernel<false>),
                                         hipFuncAttributeMaxDynamicSharedMemorySize, (int) wsp::mel::kSpectrogramLds);
    }
    else
    {
        basis.resize((size_t) 2 * bins * fft);
        for (int b = 0; b < bins; ++b)
            for (int t = 0; t < fft; ++t)
            {
                basis[(size_t) 2 * b * fft + t] = (float) std::cos(angle(b, t));
                basis[(size_t) (2 * b + 1) * fft + t] = (float) -std::sin(angle(b, t));
            }
        const int padded = (bins + 3) / 4 * 4;
        if (status == hipSuccess)
            status = mel_allocate(m, &m->basis, basis.size());
        if (status == hipSuccess)
            status = mel_allocate(m, &m->frames, (size_t) s.frame_count * fft);
        if (status == hipSuccess)
            status = mel_allocate(m, &m->spectrum, (size_t) s.frame_count * 2 * bins);
        if (status == hipSuccess)
            status = mel_allocate(m, &m->power, (size_t) s.frame_count * padded);
        if (status == hipSuccess)
            status = mel_allocate(m, &m->filters, (size_t) s.mel_count * padded);
        if (status == hipSuccess)
            status = hipMemset(m->power, 0, (size_t) s.frame_count * padded * sizeof(float));
        if (status == hipSuccess)
            status = hipMemset(m->filters, 0, (size_t) s.mel_count * padded * sizeof(float));
        if (status == hipSuccess)
            status = mel_allocate(m, &m->rows, (size_t) s.frame_count * s.mel_count);
        if (status == hipSuccess)
            status = hipMemcpy(m->basis, basis.data(), basis.size() * sizeof(float), hipMemcpyHostToDevice);
    }
    if (status != hipSuccess)
    {
        for (void* p : m->owned)
            (void) hipFree(p);
        delete m;
        return WSP_ERR_HIP;
    }
    *out = m;
    return WSP_OK;
}

void wsp_mel_destroy(wsp_mel* m)
{
    if (m == nullptr)
        return;
    (void) hipSetDevice(m->device);
    (void) hipStreamSynchronize(m->stream);
    for (void* p : m->owned)
        (void) hipFree(p);
    delete m;
}

const char* wsp_mel_last_error(const wsp_mel* m)
{
    return m == nullptr ? "null mel front end" : m->error;
}

int wsp_mel_encode(wsp_mel* m, const float* samples, const float* filters, float* output)
{
    using namespace wsp::mel;
    if (m == nullptr)
        return WSP_ERR_ARGUMENT;
    m->error[0] = 0;
    if (samples == nullptr || filters == nullptr || output == nullptr)
    {
        std::snprintf(m->error, sizeof m->error, "wsp_mel_encode: null samples, filters or output");
        return WSP_ERR_ARGUMENT;
    }
    const wsp_mel_shape& s = m->shape;
    const int fft = s.fft_length, bins = fft / 2 + 1, frames = s.frame_count, mels = s.mel_count;
    hipStream_t st = m->stream;
    (void) hipSetDevice(m->device);
    hipError_t status;
    const int total = frames * mels;
    if (m->fused)
    {
        const int blocks = (frames + kSpectrogramFrames - 1) / kSpectrogramFrames;
        // The filterbank goes through LDS where it fits and comes in whole 16-byte runs.
        const size_t lds = spectrogram_lds(fft), with_filters = lds + ((size_t) mels * bins + 3) / 4 * 16;
        const bool staged = with_filters <= kSpectrogramLds && reinterpret_cast<uintptr_t>(filters) % 16 == 0;
        if (staged)
            hipLaunchKernelGGL(spectrogram_kernel<true>, dim3(blocks), dim3(kSpectrogramThreads), with_filters, st,
                               samples, s.sample_count, m->window, fft, s.hop_length, frames, m->folded, filters, mels,
                               output, m->peaks);
        else
            hipLaunchKernelGGL(spectrogram_kernel<false>, dim3(blocks), dim3(kSpectrogramThreads), lds, st, samples,
                               s.sample_count, m->window, fft, s.hop_length, frames, m->folded, filters, mels, output,
                               m->peaks);
        if ((status = hipGetLastError()) != hipSuccess)
            return mel_hip(m, status, "spectrogram");
        hipLaunchKernelGGL(normalise_kernel, dim3(std::min(kLogBlocks, (total + kThreads - 1) / kThreads)),
                           dim3(kThreads), 0, st, output, total, m->peaks, blocks);
        if ((status = hipGetLastError()) != hipSuccess)
            return mel_hip(m, status, "normalise");
        return WSP_OK;
    }
    hipLaunchKernelGGL(frames_kernel, dim3(frames), dim3(kThreads), 0, st, samples, s.sample_count, m->window, fft,
                       s.hop_length, m->frames);
    if ((status = hipGetLastError()) != hipSuccess)
        return mel_hip(m, status, "framing");
    if ((status = wsp::ops::linear(st, m->frames, frames, fft, m->basis, WSP_F32, nullptr, m->spectrum, 2 * bins, 0))
        != hipSuccess)
        return mel_hip(m, status, "spectrum");
    const int cells = frames * bins, padded = (bins + 3) / 4 * 4;
    hipLaunchKernelGGL(power_kernel, dim3((cells + kThreads - 1) / kThreads), dim3(kThreads), 0, st, m->spectrum,
                       bins, padded, cells, m->power);
    if ((status = hipGetLastError()) != hipSuccess)
        return mel_hip(m, status, "power");
    // The filterbank into rows of the padded stride (the padding stays zero):
    // the product then sums the same terms in the same order, plus zeros.
    if ((status = hipMemcpy2DAsync(m->filters, (size_t) padded * sizeof(float), filters, (size_t) bins * sizeof(float),
                                   (size_t) bins * sizeof(float), mels, hipMemcpyDeviceToDevice, st))
        != hipSuccess)
        return mel_hip(m, status, "filterbank copy");
    if ((status = wsp::ops::linear(st, m->power, frames, padded, m->filters, WSP_F32, nullptr, m->rows, mels, 0))
        != hipSuccess)
        return mel_hip(m, status, "filterbank");
    const int blocks = std::min(kLogBlocks, (total + kThreads - 1) / kThreads);
    hipLaunchKernelGGL(log_kernel, dim3(blocks), dim3(kThreads), 0, st, m->rows, frames, mels, output, m->peaks);
    if ((status = hipGetLastError()) != hipSuccess)
        return mel_hip(m, status, "log");
    hipLaunchKernelGGL(normalise_kernel, dim3(blocks), dim3(kThreads), 0, st, output, total, m->peaks, blocks);
    if ((status = hipGetLastError()) != hipSuccess)
        return mel_hip(m, status, "normalise");
    return WSP_OK;
}

} // extern "C"
