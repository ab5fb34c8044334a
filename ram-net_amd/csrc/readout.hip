// Read-out of a RAM layer: RMSNorm of each head's read row, times a sigmoid
// gate (reference: ram_attn_block.py:326-334), in one pass:
//     out = sigmoid(gate) * y * rsqrt(mean(y^2) + eps) * weight.
//
// Bound by memory: y and the gate in, the product out. A wave holds whole
// rows, LPR lanes each (a power of two) of one 16-byte piece (VEC elements;
// one element where C or an address is not a multiple of the piece), so the
// row sum is a butterfly over registers, without LDS; each lane takes kRows
// rows at once, so their loads are in flight together. All in fp32, rounded
// once; or with the norm and the gate each rounded to the rows' type first
// (stepwise), as three kernels that store them would. 262144 rows of 128
// bf16: 192 us for torch's row norm alone (one block a row), 30 for its
// sigmoid and 30 for its product; 45 us here, 38 stepwise (which takes a
// reciprocal for a division).
#include "ramnet_device.hpp"
#include "ramnet_kernels.hpp"

namespace ramnet {

namespace {

constexpr int kRows = 4;

template<typename Scalar, int VEC>
__device__ __forceinline__ void load_piece(const Scalar *p, float (&out)[VEC]) {
    typedef uint32_t Words __attribute__((ext_vector_type(VEC * sizeof(Scalar) / 4 > 0 ? VEC * sizeof(Scalar) / 4 : 1)));
    if constexpr (VEC == 1) {
        out[0] = load_f32(p);
    } else {
        const Words w = *reinterpret_cast<const Words *>(p);
#pragma unroll
        for (int e = 0; e < VEC; ++e)
            out[e] = bits_f32<Scalar>(sizeof(Scalar) == 4 ? w[e] : (w[e / 2] >> (e % 2 * 16)) & 0xFFFFu);
    }
}

// v as it is stored in the rows' type (bf16 through the compiler's type, which
// rounds to nearest even with one instruction for two values).
template<typename Scalar>
__device__ __forceinline__ float stored(float v) {
    if constexpr (sizeof(Scalar) == 4)
        return v;
    else if constexpr (__is_same(Scalar, bf16_t))
        return static_cast<float>(static_cast<__bf16>(v));
    else
        return static_cast<float>(static_cast<_Float16>(v));
}

template<typename Scalar, int VEC, bool STEPWISE>
__global__ __launch_bounds__(256) void readout_kernel(const ReadoutJob job, int lpr_log) {
    const int lpr = 1 << lpr_log;
    const int lane = static_cast<int>(threadIdx.x) & (kWave - 1);
    const int sub = lane & (lpr - 1), c = sub * VEC;
    const bool on = c < job.C;  // past the row: a lane that adds nothing and stores nothing
    const int cc = on ? c : 0;
    const int64_t wave = (static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x) / kWave;
    const int per = kWave >> lpr_log;  // rows of a wave at a time
    const int64_t first = wave * per * kRows + (lane >> lpr_log);
    const Scalar *y = static_cast<const Scalar *>(job.y), *gate = static_cast<const Scalar *>(job.gate);
    float w[VEC], yv[kRows][VEC], gv[kRows][VEC];
    load_piece<Scalar, VEC>(static_cast<const Scalar *>(job.weight) + cc, w);
#pragma unroll
    for (int i = 0; i < kRows; ++i) {
        const int64_t row = first + i * per < job.rows ? first + i * per : job.rows - 1;
        load_piece<Scalar, VEC>(y + row * job.C + cc, yv[i]);
        load_piece<Scalar, VEC>(gate + row * job.C + cc, gv[i]);
    }
#pragma unroll
    for (int i = 0; i < kRows; ++i) {
        float sum = 0.f;
#pragma unroll
        for (int e = 0; e < VEC; ++e)
            sum += yv[i][e] * yv[i][e];
        sum = on ? sum : 0.f;
        for (int m = 1; m < lpr; m <<= 1)
            sum += __shfl_xor(sum, m);
        const float scale = 1.f / sqrtf(sum / static_cast<float>(job.C) + job.eps);
        const int64_t row = first + i * per;
        if (!on || row >= job.rows)
            continue;
        float o[VEC];
#pragma unroll
        for (int e = 0; e < VEC; ++e) {
            // (rounded to 16 bits next, the quotient takes the hardware's reciprocal, good to one unit of fp32)
            const float d = 1.f + expf(-gv[i][e]);
            if constexpr (STEPWISE)
                o[e] = stored<Scalar>(yv[i][e] * scale * w[e]) *
                       stored<Scalar>(sizeof(Scalar) == 4 ? 1.f / d : __builtin_amdgcn_rcpf(d));
            else
                o[e] = yv[i][e] * scale * w[e] / d;
        }
        Scalar *dst = static_cast<Scalar *>(job.out) + row * job.C + c;
        if constexpr (VEC == 1) {
            store_f32(dst, o[0]);
        } else {
            struct alignas(16) Out {
                Scalar v[VEC];
            } packed;
#pragma unroll
            for (int e = 0; e < VEC; ++e) {
                if constexpr (__is_same(Scalar, bf16_t))
                    packed.v[e].bits = __builtin_bit_cast(uint16_t, static_cast<__bf16>(o[e]));
                else
                    store_f32(&packed.v[e], o[e]);
            }
            *reinterpret_cast<Out *>(dst) = packed;
        }
    }
}

template<typename Scalar>
hipError_t launch_typed(const ReadoutJob &job, hipStream_t stream, const char **why) {
    constexpr int V = 16 / static_cast<int>(sizeof(Scalar));
    auto aligned = [](const void *p) { return reinterpret_cast<uintptr_t>(p) % 16 == 0; };
    const bool wide = job.C % V == 0 && aligned(job.y) && aligned(job.gate) && aligned(job.weight) && aligned(job.out);
    const int pieces = wide ? job.C / V : job.C;
    if (pieces > kWave) {
        *why = "readout: a row must fit one wave (64 pieces of 16 bytes, or 64 elements where unaligned)";
        return hipErrorInvalidValue;
    }
    int log = 0;
    while ((1 << log) < pieces)
        ++log;
    const int64_t per_block = static_cast<int64_t>(4 * kRows) * (kWave >> log);
    const int64_t blocks = (job.rows + per_block - 1) / per_block;
    if (blocks > 0x7fffffff) {
        *why = "readout: too many rows for one launch";
        return hipErrorInvalidValue;
    }
    const dim3 grid(static_cast<unsigned>(blocks));
#define RAMNET_READOUT(VEC, STEPWISE)                  \
    if (wide == (VEC > 1) && job.stepwise == STEPWISE) \
        hipLaunchKernelGGL((readout_kernel<Scalar, VEC, STEPWISE>), grid, dim3(256), 0, stream, job, log)
    RAMNET_READOUT(V, false);
    RAMNET_READOUT(V, true);
    RAMNET_READOUT(1, false);
    RAMNET_READOUT(1, true);
#undef RAMNET_READOUT
    return hipGetLastError();
}

}  // namespace

hipError_t launch_readout(const ReadoutJob &job, hipStream_t stream, const char **why) {
    if (job.rows == 0)
        return hipSuccess;
    switch (job.dtype) {
        case kF32: return launch_typed<float>(job, stream, why);
        case kF16: return launch_typed<_Float16>(job, stream, why);
        case kBF16: return launch_typed<bf16_t>(job, stream, why);
        default: *why = "readout: unsupported dtype"; return hipErrorInvalidValue;
    }
}

}  // namespace ramnet
