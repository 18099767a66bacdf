// Epilogue of the fused gate/up projection: y = round16(silu(gate) * up) over two 16-bit [M, N] matrices, the arithmetic
// of the CUDA provider's paired kernel (onnx-runtime-ep-cuda/src/kernels/matmul_nbits.rs:4207-4233, 4375-4386): both
// projections arrive rounded to the 16-bit type (as the separate nodes would store them), silu is evaluated in f32 with
// the exponential taken in double and rounded to f32, and the product is rounded once. `decomposed` reproduces a graph
// that spelled silu as Sigmoid and Mul: the sigmoid and x * sigmoid are each rounded to the 16-bit type.
#include "swiglu.hiph"
#include "weights_ahead.hiph"

namespace mnb {

// Eight elements a lane (16-byte loads and stores) where all three matrices are 16-byte aligned; the remainder, and other alignments, one by
// one. Bound by vector instructions and memory about equally: 8192 x 14336 elements, f16, about 365 -> 189 us (3.7 TB/s), 777 rows 43 -> 24.
template <bool BF16>
__global__ __launch_bounds__(256) void swiglu_kernel(const uint16_t* __restrict__ gate, const uint16_t* __restrict__ up, int64_t count, int64_t pieces, int decomposed,
                                                     uint16_t* __restrict__ y)
{
    const int64_t first = blockIdx.x * static_cast<int64_t>(blockDim.x) + threadIdx.x, step = static_cast<int64_t>(gridDim.x) * blockDim.x;
    const bool dec = decomposed != 0;
    for (int64_t i = first; i < pieces; i += step) {
        const uint4 g = reinterpret_cast<const uint4*>(gate)[i], u = reinterpret_cast<const uint4*>(up)[i];
        const uint32_t gw[4] = {g.x, g.y, g.z, g.w}, uw[4] = {u.x, u.y, u.z, u.w};
        uint32_t o[4];
#pragma unroll
        for (int j = 0; j < 4; ++j)
            o[j] = swiglu16<BF16>(gw[j] & 0xffffu, uw[j] & 0xffffu, dec) | (static_cast<uint32_t>(swiglu16<BF16>(gw[j] >> 16, uw[j] >> 16, dec)) << 16);
        reinterpret_cast<uint4*>(y)[i] = make_uint4(o[0], o[1], o[2], o[3]);
    }
    for (int64_t i = pieces * 8 + first; i < count; i += step) y[i] = swiglu16<BF16>(gate[i], up[i], dec);
}

// RMS-normalization prologue (onnx-runtime-ep-cuda/src/kernels/matmul_nbits.rs:4125-4205): out = round16((a * inv_std) *
// gamma) per row, inv_std = 1 / sqrt(mean(a^2) + eps). The sum of squares follows the reference's order exactly - 32
// lanes, each with four running sums over its 4-element chunks, (s0 + s1) + (s2 + s3), then the shuffle tree over 32
// lanes. What bounds a call of few rows is the chain launch, trip to memory, sum, trip, store. So a workgroup of four waves takes
// one row, requests all of it and gamma at once (16 bytes a load; the pieces stay in registers up to kHeld a thread), passes the
// row through LDS, and every wave sums it from there - lanes 0..31 the running sums s0 and s1 of the reference's lanes, lanes 32..63
// s2 and s3 - so that nothing but one barrier lies between the row's arrival and its results. K = 3584, one / 16 rows, as a node of a
// recorded step: 6.2 / 8.0 us with one wave summing two rows straight from memory, 4.6 / 4.8 us so (3.0 with everything in a near cache).
constexpr int kHeld = 2;                     // 16-byte pieces of the row a thread keeps: 4096 elements a row

// Weights that a normalization launch brings to the near caches, at most: what fits the time that the launch takes anyway. (Bytes and no multiple of the CUs: the memory's rate sets them,
// and the eight caches of 4 MB that have to hold them.) 7B steps of 142 and 170 launches at
// one / 16 rows (29 and 57 normalizations), bytes read ahead 0, 2, 4, 8, 16 MB: 1,140 / 1,553, 1,133 / 1,545, 1,125 / 1,536, 1,113 / 1,519, 1,128 / 1,526 us.
constexpr uint32_t kAheadBytes = 8000000;

// x + (x of the lane `N` further on in its row of 16, cyclically)
template <int N>
__device__ __forceinline__ float add_rotated(float x)
{
    return __fadd_rn(x, __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(x), 0x120 + N, 0xf, 0xf, false)));
}

// STAGED: the row passes through LDS (K * 2 bytes of it); otherwise (rows beyond LDS) the sums read memory.
// Blocks from `rows` on read weights of the launch behind this one ahead: while a row is normalized the memory is idle.
template <bool BF16, bool STAGED>
__global__ __launch_bounds__(256) void rmsnorm16_kernel(const uint16_t* __restrict__ a, const void* __restrict__ gamma, uint16_t* __restrict__ out, int gamma_dtype, int64_t k, float epsilon,
                                                        uint32_t rows, WeightsAhead ahead)
{
    extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
    if (blockIdx.x >= rows) {
        read_ahead(ahead, blockIdx.x, 256);
        return;
    }
    const int t = threadIdx.x;
    const int64_t row = blockIdx.x;
    const uint16_t* const x = a + row * k;
    // eight elements of the row, from an 8-byte boundary
    auto load_piece = [&](int piece) {
        const uint2* const from = reinterpret_cast<const uint2*>(x) + 2 * piece;
        const uint2 lo = from[0], hi = from[1];
        return make_uint4(lo.x, lo.y, hi.x, hi.y);
    };
    const int pieces = static_cast<int>(k >> 3);
    const bool gf32 = gamma_dtype == ROCM_DT_F32;
    auto widen = [](uint32_t bits16) { return BF16 ? bf16_bits_to_f32(static_cast<uint16_t>(bits16)) : f16_bits_to_f32(static_cast<uint16_t>(bits16)); };
    struct Weights { uint4 lo, hi; };        // eight gamma values: 16-bit ones all in `lo`
    auto load_gamma = [&](int piece) {
        Weights w;
        w.lo = w.hi = make_uint4(0u, 0u, 0u, 0u);
        if (gf32) {
            w.lo = static_cast<const uint4*>(gamma)[2 * piece];
            w.hi = static_cast<const uint4*>(gamma)[2 * piece + 1];
        } else {
            const uint2* const g = static_cast<const uint2*>(gamma) + 2 * piece;               // (8-byte aligned only)
            const uint2 g0 = g[0], g1 = g[1];
            w.lo = make_uint4(g0.x, g0.y, g1.x, g1.y);
        }
        return w;
    };

    uint4 held[kHeld];
    Weights weights[kHeld];
#pragma unroll
    for (int i = 0; i < kHeld; ++i)
        if (t + i * 256 < pieces) held[i] = load_piece(t + i * 256);
#pragma unroll
    for (int i = 0; i < kHeld; ++i)
        if (t + i * 256 < pieces) weights[i] = load_gamma(t + i * 256);
    if constexpr (STAGED) {
#pragma unroll
        for (int i = 0; i < kHeld; ++i)
            if (t + i * 256 < pieces) reinterpret_cast<uint4*>(smem)[t + i * 256] = held[i];
        for (int piece = t + kHeld * 256; piece < pieces; piece += 256) reinterpret_cast<uint4*>(smem)[piece] = load_piece(piece);
        __syncthreads();
    }
    float inv_std;
    {
        const int lane = t & 63;
        // elements 2 (lane / 32) and + 1 of chunk (lane % 32) + 32 i
        const uint32_t* const pair = (STAGED ? reinterpret_cast<const uint32_t*>(smem) : reinterpret_cast<const uint32_t*>(x)) + (lane & 31) * 2 + (lane >> 5);
        const int items = static_cast<int>(k >> 7);
        float even = 0.f, odd = 0.f;
#pragma unroll 8
        for (int i = 0; i < items; ++i) {
            const uint32_t raw = pair[i * 64];
            const float v0 = widen(raw & 0xffffu), v1 = widen(raw >> 16);
            even = __fmaf_rn(v0, v0, even);
            odd = __fmaf_rn(v1, v1, odd);
        }
        float ss = __fadd_rn(even, odd);
        ss = __fadd_rn(ss, __shfl_xor(ss, 32, 64));         // (s0 + s1) + (s2 + s3)
        ss = __fadd_rn(ss, __shfl_xor(ss, 16, 64));         // the reference's tree: every lane ends with what its lane 0 has
        ss = add_rotated<8>(ss);
        ss = add_rotated<4>(ss);
        ss = add_rotated<2>(ss);
        ss = add_rotated<1>(ss);
        // sqrtf, not __fsqrt_rn: the latter is the hardware's approximate square root here; sqrtf and the division are
        // correctly rounded (the compiler's default for f32 divide and sqrt)
        inv_std = __fdiv_rn(1.0f, sqrtf(__fadd_rn(__fdiv_rn(ss, static_cast<float>(k)), epsilon)));
    }
    auto store = [&](int piece, const uint4& raw, const Weights& w) {
        const uint32_t d[4] = {raw.x, raw.y, raw.z, raw.w};
        const uint32_t g[8] = {w.lo.x, w.lo.y, w.lo.z, w.lo.w, w.hi.x, w.hi.y, w.hi.z, w.hi.w};
        uint32_t o[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const float g0 = gf32 ? __uint_as_float(g[2 * i]) : widen(g[i] & 0xffffu), g1 = gf32 ? __uint_as_float(g[2 * i + 1]) : widen(g[i] >> 16);
            const float y0 = as_f32(__fmul_rn(__fmul_rn(widen(d[i] & 0xffffu), inv_std), g0)), y1 = as_f32(__fmul_rn(__fmul_rn(widen(d[i] >> 16), inv_std), g1));
            o[i] = BF16 ? f32_to_bf16_bits(y0) | (static_cast<uint32_t>(f32_to_bf16_bits(y1)) << 16) : f32_to_f16_bits(y0) | (static_cast<uint32_t>(f32_to_f16_bits(y1)) << 16);
        }
        uint2* const y = reinterpret_cast<uint2*>(out + row * k) + 2 * piece;                  // (8-byte aligned only)
        y[0] = make_uint2(o[0], o[1]);
        y[1] = make_uint2(o[2], o[3]);
    };
#pragma unroll
    for (int i = 0; i < kHeld; ++i)
        if (t + i * 256 < pieces) store(t + i * 256, held[i], weights[i]);
    for (int piece = t + kHeld * 256; piece < pieces; piece += 256) store(piece, STAGED ? reinterpret_cast<const uint4*>(smem)[piece] : load_piece(piece), load_gamma(piece));
}

}  // namespace mnb

extern "C" int rocm_launch_rmsnorm16(const void* a, const void* gamma, int gamma_dtype, int64_t rows, int64_t k, float epsilon, int dtype, void* out,
                                     const RocmWeightsAhead* ahead, rocm_stream_t stream)
{
    if (rows <= 0 || k <= 0) return 0;
    if ((dtype != ROCM_DT_F16 && dtype != ROCM_DT_BF16) || k % 128 != 0) return static_cast<int>(hipErrorInvalidValue);
    // rows move four elements at a time: 8-byte pieces of a and out, 16- or 8-byte pieces of gamma
    const uintptr_t gamma_mask = gamma_dtype == ROCM_DT_F32 ? 15 : 7;
    if (((reinterpret_cast<uintptr_t>(a) | reinterpret_cast<uintptr_t>(out)) & 7) != 0 || (reinterpret_cast<uintptr_t>(gamma) & gamma_mask) != 0)
        return static_cast<int>(hipErrorInvalidValue);
    hipStream_t s = static_cast<hipStream_t>(stream);
    const bool staged = k <= 32768;          // what fits the 64 KiB a kernel gets without asking
    const size_t lds = staged ? static_cast<size_t>(k) * 2 : 0;
    mnb::WeightsAhead w{};
    unsigned blocks = static_cast<unsigned>(rows);
    if (ahead && rows <= 64) blocks = static_cast<unsigned>(mnb::plan_weights_ahead(*ahead, mnb::kAheadBytes, 256, blocks, 0, &w));
    auto go = [&](auto kernel) {
        hipLaunchKernelGGL(kernel, dim3(blocks), dim3(256), lds, s, static_cast<const uint16_t*>(a), gamma, static_cast<uint16_t*>(out), gamma_dtype, k, epsilon, static_cast<uint32_t>(rows), w);
        return static_cast<int>(hipGetLastError());
    };
    if (dtype == ROCM_DT_BF16) return staged ? go(mnb::rmsnorm16_kernel<true, true>) : go(mnb::rmsnorm16_kernel<true, false>);
    return staged ? go(mnb::rmsnorm16_kernel<false, true>) : go(mnb::rmsnorm16_kernel<false, false>);
}

extern "C" int rocm_launch_swiglu(const void* gate, const void* up, int64_t count, int dtype, int decomposed, void* y, rocm_stream_t stream)
{
    if (count <= 0) return 0;
    if (dtype != ROCM_DT_F16 && dtype != ROCM_DT_BF16) return static_cast<int>(hipErrorInvalidValue);
    const bool wide = ((reinterpret_cast<uintptr_t>(gate) | reinterpret_cast<uintptr_t>(up) | reinterpret_cast<uintptr_t>(y)) & 15) == 0;
    const int64_t pieces = wide ? count / 8 : 0;
    const int64_t items = wide && pieces > 0 ? pieces : count;
    int64_t blocks = (items + 255) / 256;
    if (blocks > 65536) blocks = 65536;
    const uint16_t* g = static_cast<const uint16_t*>(gate);
    const uint16_t* u = static_cast<const uint16_t*>(up);
    uint16_t* out = static_cast<uint16_t*>(y);
    hipStream_t s = static_cast<hipStream_t>(stream);
    if (dtype == ROCM_DT_BF16) hipLaunchKernelGGL(mnb::swiglu_kernel<true>, dim3(static_cast<unsigned>(blocks)), dim3(256), 0, s, g, u, count, pieces, decomposed, out);
    else hipLaunchKernelGGL(mnb::swiglu_kernel<false>, dim3(static_cast<unsigned>(blocks)), dim3(256), 0, s, g, u, count, pieces, decomposed, out);
    return static_cast<int>(hipGetLastError());
}
