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
// windowed samples folded about the frame's middle (cos(2πbn/N) is even and
// sin odd in n, so re needs x[n] + x[N-n] and im x[n] - x[N-n] for n up to N/2
// only: half the products), the two half-length products on the matrix cores
// (v_mfma_f32_16x16x4_f32: 16 bins by 16 frames), the power, the filterbank as
// another such product, the logarithm and the block's largest value. A wave
// takes 16-bin tiles, then 16-band tiles. Each product step sums four
// consecutive n (and bins), in order: position 16j + 4g + e of an LDS row, and
// of the basis, holds n = 16j + 4e + g. The basis is fragment-major, one
// contiguous kilobyte a load; each block reads all of it (346 KB at 400
// points), which with the 10.8 K matrix-core clocks of a CU's tiles is what
// bounds the launch. The 30 s window went from 38.8 us as seven launches
// (frames, spectrum 17, power, filterbank copy and product, log) and 53 with
// the products on the vector units to 23.5.
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

__global__ void __launch_bounds__(kSpectrogramThreads) spectrogram_kernel(
    const float* __restrict__ samples, int count, const float* __restrict__ window, int fft, int hop, int frames,
    const float* __restrict__ basis, const float* __restrict__ filters, int mels, float* __restrict__ out,
    float* __restrict__ peaks)
{
    extern __shared__ __attribute__((aligned(16))) float rows[];
    __shared__ float scratch[kSpectrogramThreads / kWave];
    const int half = fft / 2, bins = half + 1, tiles = (bins + 15) / 16, stride = 16 * tiles + kRowPad;
    float* const even = rows;                             // [frame][place(n)]
    float* const odd = even + kSpectrogramFrames * stride;
    float* const power = odd + kSpectrogramFrames * stride; // [frame][place(bin)]
    const int f0 = blockIdx.x * kSpectrogramFrames;

    // A thread folds value n of eight frames (all their loads in flight at
    // once); values past the middle are the padding.
    constexpr int kValues = 256, kFramesEach = kSpectrogramFrames * kValues / kSpectrogramThreads;
    const int first = threadIdx.x / kValues * kFramesEach;
    for (int n = threadIdx.x % kValues; n < 16 * tiles; n += kValues)
    {
        const bool in = n <= half, folded = in && n > 0 && 2 * n != fft;
        const int t = in ? n : 0, u = folded ? fft - n : t;
        const float wt = window[t], wu = window[u];
        float a[kFramesEach], b[kFramesEach];
#pragma unroll
        for (int i = 0; i < kFramesEach; ++i)
        {
            const int start = min(f0 + first + i, frames - 1) * hop - half;
            int x = abs(start + t), y = abs(start + u);
            x = x >= count ? 2 * (count - 1) - x : x;
            y = y >= count ? 2 * (count - 1) - y : y;
            a[i] = samples[x];
            b[i] = samples[y];
        }
#pragma unroll
        for (int i = 0; i < kFramesEach; ++i)
        {
            const float left = a[i] * wt, right = b[i] * wu;
            const int at = (first + i) * stride + place(n);
            even[at] = folded ? left + right : in ? left : 0.f;
            odd[at] = folded ? left - right : 0.f;
        }
    }
    __syncthreads();

    const int wave = threadIdx.x / kWave, lane = threadIdx.x % kWave, li = lane % 16, g = lane / 16;
    // Runs of the basis (and of the filters) are loaded kRuns ahead of their
    // products; runs past the last repeat it and are not multiplied.
    for (int t = wave; t < tiles; t += kSpectrogramThreads / kWave)
    {
        const f32x4* b = reinterpret_cast<const f32x4*>(basis) + (size_t) t * tiles * 2 * kWave + lane;
        f32x4 re = {0.f, 0.f, 0.f, 0.f}, im = {0.f, 0.f, 0.f, 0.f};
        f32x4 c[2][kRuns], s[2][kRuns];
        auto load = [&](int j0, int set) {
#pragma unroll
            for (int i = 0; i < kRuns; ++i)
            {
                const int j = min(j0 + i, tiles - 1);
                c[set][i] = b[(size_t) (2 * j) * kWave];
                s[set][i] = b[(size_t) (2 * j + 1) * kWave];
            }
        };
        auto multiply = [&](int j0, int set) {
#pragma unroll
            for (int i = 0; i < kRuns; ++i)
            {
                if (j0 + i >= tiles)
                    break;
                const f32x4 e = *reinterpret_cast<const f32x4*>(even + li * stride + 16 * (j0 + i) + 4 * g);
                const f32x4 o = *reinterpret_cast<const f32x4*>(odd + li * stride + 16 * (j0 + i) + 4 * g);
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
        // Lane (li, g) holds frame li's bins 16t + 4g + r.
#pragma unroll
        for (int r = 0; r < 4; ++r)
            power[li * stride + place(16 * t + 4 * g + r)] = re[r] * re[r] + im[r] * im[r];
    }
    __syncthreads();

    float best = -INFINITY;
    const int bands = (mels + 15) / 16;
    for (int t = wave; t < bands; t += kSpectrogramThreads / kWave)
    {
        const float* row = filters + (size_t) min(16 * t + li, mels - 1) * bins;
        f32x4 sum = {0.f, 0.f, 0.f, 0.f};
        float w[2][kRuns][4];
        auto load = [&](int j0, int set) {
#pragma unroll
            for (int i = 0; i < kRuns; ++i)
#pragma unroll
                for (int k = 0; k < 4; ++k)
                    w[set][i][k] = row[min(16 * (j0 + i) + 4 * k + g, bins - 1)];
        };
        auto multiply = [&](int j0, int set) {
#pragma unroll
            for (int i = 0; i < kRuns; ++i)
            {
                if (j0 + i >= tiles)
                    break;
                const f32x4 p = *reinterpret_cast<const f32x4*>(power + li * stride + 16 * (j0 + i) + 4 * g);
#pragma unroll
                for (int k = 0; k < 4; ++k)
                {
                    const bool in = 16 * (j0 + i) + 4 * k + g < bins; // (past the last bin both operands are zero)
                    sum = __builtin_amdgcn_mfma_f32_16x16x4f32(in ? w[set][i][k] : 0.f, in ? p[k] : 0.f, sum, 0, 0, 0);
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

size_t spectrogram_lds(int fft)
{
    return (size_t) 3 * kSpectrogramFrames * (16 * ((fft / 2 + 16) / 16) + kRowPad) * sizeof(float);
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
        status = mel_allocate(m, &m->window, fft);
    if (status == hipSuccess)
        status = mel_allocate(m, &m->peaks, std::max(wsp::mel::kLogBlocks, (s.frame_count + 15) / 16));
    if (status == hipSuccess)
        status = hipMemcpy(m->window, window.data(), window.size() * sizeof(float), hipMemcpyHostToDevice);
    m->fused = wsp::mel::spectrogram_lds(fft) <= 152 * 1024; // of a CU's 160 KB
    if (m->fused)
    {
        const int tiles = (bins + 15) / 16;
        basis.assign((size_t) tiles * tiles * 2 * 256, 0.f);
        for (int b = 0; b < bins; ++b)
            for (int n = 0; n < bins; ++n)
            {
                // lane (bin % 16, g), element e of run n / 16 stands for n = 16j + 4e + g
                const size_t at = (((size_t) (b / 16) * tiles + n / 16) * 2 * 64 + 16 * (n % 4) + b % 16) * 4 + n % 16 / 4;
                basis[at] = (float) std::cos(angle(b, n));
                basis[at + 256] = (float) -std::sin(angle(b, n));
            }
        if (status == hipSuccess)
            status = mel_allocate(m, &m->folded, basis.size());
        if (status == hipSuccess)
            status = hipMemcpy(m->folded, basis.data(), basis.size() * sizeof(float), hipMemcpyHostToDevice);
        if (status == hipSuccess)
            status = hipFuncSetAttribute(reinterpret_cast<const void*>(&wsp::mel::spectrogram_kernel),
                                         hipFuncAttributeMaxDynamicSharedMemorySize,
                                         (int) wsp::mel::spectrogram_lds(fft));
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
        hipLaunchKernelGGL(spectrogram_kernel, dim3(blocks), dim3(kSpectrogramThreads), spectrogram_lds(fft), st,
                           samples, s.sample_count, m->window, fft, s.hop_length, frames, m->folded, filters, mels,
                           output, m->peaks);
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
