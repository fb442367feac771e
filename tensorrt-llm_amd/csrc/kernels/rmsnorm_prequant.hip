// RMSNorm fused with the smoothing pass in front of the matmul:
//     normed = T(x * rsqrt(mean(x^2) + eps) * gamma [+ beta])              (one rounding to T)
//     out    = T_out(T(normed * pre_quant_scale))                          (T_out = T or fp8 e4m3)
// i.e. invokeGeneralRmsNorm (kernels/rmsnormKernels.cu:29-38, 83-124, 230-262: float32 sum of
// squares, rsqrtf, float32 products, cast to T) followed by apply_per_channel_scale
// (kernels/preQuantScaleKernel.cu:42-149: one multiply rounded to T, optional saturating cast to
// e4m3) in ONE pass over the activations: the normalised tensor never goes to memory, and with fp8
// output only half as many bytes are written.  pre_quant_scale may be NULL (plain RMSNorm, or
// RMSNorm + cast).
// One workgroup of 256 threads per row; a row of up to 16384 elements stays in registers between
// the two phases (longer rows are read again, from L2); 16-byte loads and stores; sum of squares by
// wavefront butterfly + one LDS step.
#include "dequant_math.h"

namespace woq
{

template <int DT, bool TO_FP8, int CHUNKS, bool AHEAD>
__global__ void __launch_bounds__(256) rmsnorm_prequant_kernel(void* out, void const* x, void const* gamma,
    void const* beta, void const* scale, float eps, int k)
{
    using E = Elem<DT>;
    long const row = blockIdx.x;
    uint16_t const* src = static_cast<uint16_t const*>(x) + row * k;
    int const n8 = k / 8; // 16-byte pieces of a row; thread t owns pieces t, t + 256, ...

    // AHEAD: the tables' pieces are requested together with the row's; read behind the sum of squares they cost a second
    // trip to memory (us, bf16 -> e4m3 with smoothing: 8 x 8192 3.80 -> 3.46, 1990 x 4096 7.64 -> 6.95, 4096 x 4096 13.6 ->
    // 12.4).  Long rows by the thousand are left as they were: the registers cost residency there (8192 x 8192 42.6 -> 44.4).
    u32x4 const zero = {0u, 0u, 0u, 0u};
    u32x4 v[CHUNKS];
    [[maybe_unused]] u32x4 gam[CHUNKS], sca[CHUNKS];
#pragma unroll
    for (int i = 0; i < CHUNKS; ++i)
    {
        int const piece = threadIdx.x + i * 256;
        bool const in = piece < n8;
        v[i] = in ? *reinterpret_cast<u32x4 const*>(src + (long) piece * 8) : zero;
        if constexpr (AHEAD)
        {
            gam[i] = in ? static_cast<u32x4 const*>(gamma)[piece] : zero;
            sca[i] = in && scale ? static_cast<u32x4 const*>(scale)[piece] : zero;
        }
    }
    float ss = 0.f;
#pragma unroll
    for (int i = 0; i < CHUNKS; ++i)
    {
#pragma unroll
        for (int r = 0; r < 4; ++r)
        {
            float const a = E::lo(v[i][r]), b = E::hi(v[i][r]);
            ss = __builtin_fmaf(a, a, ss);
            ss = __builtin_fmaf(b, b, ss);
        }
    }
    for (int piece = threadIdx.x + CHUNKS * 256; piece < n8; piece += 256) // rows longer than CHUNKS * 2048
    {
        u32x4 const w = *reinterpret_cast<u32x4 const*>(src + (long) piece * 8);
#pragma unroll
        for (int r = 0; r < 4; ++r)
        {
            float const a = E::lo(w[r]), b = E::hi(w[r]);
            ss = __builtin_fmaf(a, a, ss);
            ss = __builtin_fmaf(b, b, ss);
        }
    }
#pragma unroll
    for (int off = 32; off > 0; off >>= 1)
        ss += __shfl_xor(ss, off, 64);
    __shared__ float part[4];
    if ((threadIdx.x & 63) == 0)
        part[threadIdx.x >> 6] = ss;
    __syncthreads();
    float const inv = __frsqrt_rn((part[0] + part[1] + part[2] + part[3]) / (float) k + eps);

    auto finish = [&](u32x4 w, int piece, auto const& gamma_piece, auto const& scale_piece) __attribute__((always_inline))
    {
        u32x4 const g = gamma_piece(piece);
        u32x4 const b = beta ? static_cast<u32x4 const*>(beta)[piece] : u32x4{0u, 0u, 0u, 0u};
        u32x4 y;
#pragma unroll
        for (int r = 0; r < 4; ++r)
        {
            float lo = E::lo(w[r]) * inv * E::lo(g[r]), hi = E::hi(w[r]) * inv * E::hi(g[r]);
            if (beta)
            {
                lo += E::lo(b[r]);
                hi += E::hi(b[r]);
            }
            y[r] = E::pack(lo, hi);
        }
        if (scale)
        {
            u32x4 const sc = scale_piece(piece);
#pragma unroll
            for (int r = 0; r < 4; ++r)
                y[r] = E::mul2(y[r], sc[r]);
        }
        if constexpr (TO_FP8)
        {
            int lo = 0, hi = 0;
            lo = __builtin_amdgcn_cvt_pk_fp8_f32(clamp_e4m3(E::lo(y[0])), clamp_e4m3(E::hi(y[0])), lo, false);
            lo = __builtin_amdgcn_cvt_pk_fp8_f32(clamp_e4m3(E::lo(y[1])), clamp_e4m3(E::hi(y[1])), lo, true);
            hi = __builtin_amdgcn_cvt_pk_fp8_f32(clamp_e4m3(E::lo(y[2])), clamp_e4m3(E::hi(y[2])), hi, false);
            hi = __builtin_amdgcn_cvt_pk_fp8_f32(clamp_e4m3(E::lo(y[3])), clamp_e4m3(E::hi(y[3])), hi, true);
            u32x2 const o = {(uint32_t) lo, (uint32_t) hi};
            *reinterpret_cast<u32x2*>(static_cast<uint8_t*>(out) + row * k + (long) piece * 8) = o;
        }
        else
            *reinterpret_cast<u32x4*>(static_cast<uint16_t*>(out) + row * k + (long) piece * 8) = y;
    };
    auto const gamma_read = [&](int piece) { return static_cast<u32x4 const*>(gamma)[piece]; };
    auto const scale_read = [&](int piece) { return scale ? static_cast<u32x4 const*>(scale)[piece] : zero; };
    // Not AHEAD: the tables are read where they are used, or both at the top of a piece (us, bf16 -> e4m3 with smoothing: 4096 x 5120
    // 14.7 and 15.1, 2000 x 5120 7.74 and 7.89; with eight pieces a thread the other way about: 4096 x 14336 36.3 and 34.1, 2000 x 14336
    // 21.6 and 20.5)
    constexpr bool TOP = !AHEAD && CHUNKS == 8;
#pragma unroll
    for (int i = 0; i < CHUNKS; ++i)
    {
        int const piece = threadIdx.x + i * 256;
        if constexpr (TOP)
        {
            gam[i] = piece < n8 ? gamma_read(piece) : zero;
            sca[i] = piece < n8 ? scale_read(piece) : zero;
        }
        if (piece >= n8)
            continue;
        if constexpr (AHEAD || TOP)
            finish(v[i], piece, [&](int) { return gam[i]; }, [&](int) { return sca[i]; });
        else
            finish(v[i], piece, gamma_read, scale_read);
    }
    for (int piece = threadIdx.x + CHUNKS * 256; piece < n8; piece += 256)
    {
        u32x4 const g = gamma_read(piece), sc = scale_read(piece);
        finish(*reinterpret_cast<u32x4 const*>(src + (long) piece * 8), piece, [&](int) { return g; }, [&](int) { return sc; });
    }
}

template <int DT, bool TO_FP8>
static void launch_chunks(void* out, void const* x, void const* gamma, void const* beta, void const* scale, float eps,
    int m, int k, hipStream_t s)
{
    dim3 grid((unsigned) m), block(256);
    int const pieces_per_thread = (k / 8 + 255) / 256;
    bool const few = m <= 1024; // no more than four workgroups a CU
    if (pieces_per_thread <= 2)
        hipLaunchKernelGGL((rmsnorm_prequant_kernel<DT, TO_FP8, 2, true>), grid, block, 0, s, out, x, gamma, beta, scale, eps, k);
    else if (pieces_per_thread <= 4 && few)
        hipLaunchKernelGGL((rmsnorm_prequant_kernel<DT, TO_FP8, 4, true>), grid, block, 0, s, out, x, gamma, beta, scale, eps, k);
    else if (pieces_per_thread <= 4)
        hipLaunchKernelGGL((rmsnorm_prequant_kernel<DT, TO_FP8, 4, false>), grid, block, 0, s, out, x, gamma, beta, scale, eps, k);
    else if (few)
        hipLaunchKernelGGL((rmsnorm_prequant_kernel<DT, TO_FP8, 8, true>), grid, block, 0, s, out, x, gamma, beta, scale, eps, k);
    else
        hipLaunchKernelGGL((rmsnorm_prequant_kernel<DT, TO_FP8, 8, false>), grid, block, 0, s, out, x, gamma, beta, scale, eps, k);
}

int launch_rmsnorm_prequant(void* out, void const* x, void const* gamma, void const* beta, void const* scale, float eps,
    int m, int k, int dtype, int out_dtype, void* stream)
{
    auto s = static_cast<hipStream_t>(stream);
    bool const fp8 = out_dtype == WOQ_FP8_E4M3;
    if (dtype == WOQ_BF16)
        fp8 ? launch_chunks<WOQ_BF16, true>(out, x, gamma, beta, scale, eps, m, k, s)
            : launch_chunks<WOQ_BF16, false>(out, x, gamma, beta, scale, eps, m, k, s);
    else
        fp8 ? launch_chunks<WOQ_FP16, true>(out, x, gamma, beta, scale, eps, m, k, s)
            : launch_chunks<WOQ_FP16, false>(out, x, gamma, beta, scale, eps, m, k, s);
    hipError_t err = hipGetLastError();
    if (err != hipSuccess)
        return fail(WOQ_ERR_RUNTIME, "rmsnorm kernel launch failed: %s", hipGetErrorString(err));
    return WOQ_OK;
}

} // namespace woq
