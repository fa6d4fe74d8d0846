// norm_rope.hip -- the stand-alone RMSNorm and RoPE ops of the path.
//
// RmsNormImpl<CPU> / rms_norm, src/backend/cpu/normalization.cpp:44-107,138-153,
// for any row width, in the reference's order exactly: running sum a < 32 of
// the CPU op takes the elements e with e % 32 == a of the whole 32-blocks
// (fused multiply-adds in increasing e), then (A[k]+A[8+k])+(A[16+k]+A[24+k])
// for k < 8, the remaining 8-blocks fused into those, ((T0+T4)+(T1+T5))+
// ((T2+T6)+(T3+T7)), and the scalar tail with fused multiply-adds.  Whole
// 8-blocks are stored by truncation, the tail by RNE (as the CPU op).
// Three forms (launch_rms_norm): whole 16-byte chunks and aligned pointers take
// rms_norm_head_kernel (rows of 64, 128 or 256: the head norms) or
// rms_norm_row_kernel (the hidden norms); the others rms_norm_kernel, one wave
// per row, lane a on sum a.
//
// ApplyRopeImpl<CPU>, src/backend/cpu/rope.cpp:76-119: NeoX pairs (i, i + D/2)
// of a head-major [H][S][D] row at position start_pos + s, eight pairs per
// thread (apply_rope_vec_kernel) or, for widths and pointers that do not allow
// 16-byte accesses and for small calls, one (apply_rope_kernel).
#include <algorithm>
#include <climits>

#include "common.hpp"
#include "kernels.hpp"

namespace genllm {

#pragma clang fp contract(off)

namespace {

__device__ __forceinline__ void unpack8(const uint4& u, float (&f)[8]) {
    f[0] = bf16_lo(u.x), f[1] = bf16_hi(u.x), f[2] = bf16_lo(u.y), f[3] = bf16_hi(u.y);
    f[4] = bf16_lo(u.z), f[5] = bf16_hi(u.z), f[6] = bf16_lo(u.w), f[7] = bf16_hi(u.w);
}

// Rows of 32 R elements: 8 lanes per row, lane j holds elements 4j + 32t +
// {0..3} and runs the CPU op's sums 4j .. 4j+3 itself; three 8-lane shuffles
// form the combine order.  Bound by memory: 48,000 + 12,000 rows of 128 (the
// head norms of 1500 tokens of 32 q and 8 kv heads) 6.4 and 2.8 us, 17.1 and
// 4.9 us in rms_norm_kernel.
template <int R>
__global__ __launch_bounds__(256) void rms_norm_head_kernel(uint16_t* out, const uint16_t* x, const float* w,
                                                            int64_t rows, float eps) {
    constexpr int H = 32 * R;
    const int lane = threadIdx.x & 63, j = lane & 7;
    const int64_t row = int64_t(blockIdx.x) * 32 + (threadIdx.x >> 3);
    const int64_t at = (row < rows ? row : rows - 1) * H + 4 * j;  // the last row again past the end: not stored
    uint2 u[R];
#pragma unroll
    for (int t = 0; t < R; ++t) u[t] = *reinterpret_cast<const uint2*>(x + at + 32 * t);
    float4 g[R];
#pragma unroll
    for (int t = 0; t < R; ++t) g[t] = *reinterpret_cast<const float4*>(w + 4 * j + 32 * t);
    float v[R][4], A[4] = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
    for (int t = 0; t < R; ++t) {
        v[t][0] = bf16_lo(u[t].x), v[t][1] = bf16_hi(u[t].x), v[t][2] = bf16_lo(u[t].y), v[t][3] = bf16_hi(u[t].y);
#pragma unroll
        for (int q = 0; q < 4; ++q) A[q] = __builtin_fmaf(v[t][q], v[t][q], A[q]);
    }
    float c[4];
#pragma unroll
    for (int q = 0; q < 4; ++q) A[q] += __shfl_down(A[q], 2, 8);  // A[k] + A[8+k]
#pragma unroll
    for (int q = 0; q < 4; ++q) A[q] += __shfl_down(A[q], 4, 8);  // + (A[16+k] + A[24+k])
#pragma unroll
    for (int q = 0; q < 4; ++q) c[q] = A[q] + __shfl_down(A[q], 1, 8);  // T[i] + T[i+4]
    const float ss = __shfl((c[0] + c[1]) + (c[2] + c[3]), 0, 8);
    const float r = 1.0f / __builtin_sqrtf(ss / float(H) + eps);
    if (row >= rows) return;
#pragma unroll
    for (int t = 0; t < R; ++t) {
        const float gv[4] = {g[t].x, g[t].y, g[t].z, g[t].w};
        uint32_t o[4];
#pragma unroll
        for (int q = 0; q < 4; ++q) o[q] = f32_to_bf16_trunc((v[t][q] * r) * gv[q]);
        *reinterpret_cast<uint2*>(out + at + 32 * t) = make_uint2(pack2(o[0], o[1]), pack2(o[2], o[3]));
    }
}

// One workgroup of NT threads per row of up to 8 NT NC elements (a multiple of
// 8): 16-byte loads of the row and its weights, the row through LDS, wave 0
// runs the sums from there.  Bound by latency for a few rows (the load, then
// the chain of hidden / 32 dependent fused multiply-adds, then the store) and
// by memory for many: 1 x 2560 2.8 us, 1500 x 2560 5.3 us, 4096 x 4096 13.4 us
// (5.0 TB/s); 13.4, 27.9 and 60.2 us in rms_norm_kernel, whose lanes wait for a
// two-byte load at every step of their sums.
template <int NT, int NC>
__global__ __launch_bounds__(NT) void rms_norm_row_kernel(uint16_t* out, const uint16_t* x, const float* w, int hidden,
                                                          float eps) {
    extern __shared__ __attribute__((aligned(16))) uint16_t s_row[];
    __shared__ float s_r;
    const int t = threadIdx.x, lane = t & 63;
    const int chunks = hidden >> 3;
    const uint16_t* const xr = x + int64_t(blockIdx.x) * hidden;
    uint16_t* const orow = out + int64_t(blockIdx.x) * hidden;
    uint4 u[NC];
    float4 g[NC][2];
#pragma unroll
    for (int i = 0; i < NC; ++i)
        if (t + NT * i < chunks) u[i] = *reinterpret_cast<const uint4*>(xr + 8 * (t + NT * i));
#pragma unroll
    for (int i = 0; i < NC; ++i)
        if (t + NT * i < chunks) {
            g[i][0] = *reinterpret_cast<const float4*>(w + 8 * (t + NT * i));
            g[i][1] = *reinterpret_cast<const float4*>(w + 8 * (t + NT * i) + 4);
        }
#pragma unroll
    for (int i = 0; i < NC; ++i)
        if (t + NT * i < chunks) *reinterpret_cast<uint4*>(s_row + 8 * (t + NT * i)) = u[i];
    __syncthreads();
    if (t < 64) {
        const int a = lane & 31, n32 = hidden >> 5;
        float A = 0.0f;
        int b = 0;
        for (; b + 16 <= n32; b += 16) {  // sixteen reads in flight, then their multiply-adds in order
            float v[16];
#pragma unroll
            for (int e = 0; e < 16; ++e) v[e] = bf16_to_f32(s_row[32 * (b + e) + a]);
#pragma unroll
            for (int e = 0; e < 16; ++e) A = __builtin_fmaf(v[e], v[e], A);
        }
        for (; b < n32; ++b) {
            const float v = bf16_to_f32(s_row[32 * b + a]);
            A = __builtin_fmaf(v, v, A);
        }
        const float a1 = __shfl(A, (a + 8) & 31), a2 = __shfl(A, (a + 16) & 31), a3 = __shfl(A, (a + 24) & 31);
        float T = (A + a1) + (a2 + a3);  // meaningful on lanes 0..7
        for (int e = 32 * n32; e < hidden; e += 8) {
            const float v = bf16_to_f32(s_row[e + (lane & 7)]);
            T = __builtin_fmaf(v, v, T);
        }
        const float c = T + __shfl(T, (lane + 4) & 63);  // lanes 0..3
        const float c1 = __shfl(c, 1), c2 = __shfl(c, 2), c3 = __shfl(c, 3);
        if (lane == 0) s_r = 1.0f / __builtin_sqrtf(((c + c1) + (c2 + c3)) / float(hidden) + eps);
    }
    __syncthreads();
    const float r = s_r;
#pragma unroll
    for (int i = 0; i < NC; ++i)
        if (t + NT * i < chunks) {
            float v[8];
            unpack8(u[i], v);
            const float gv[8] = {g[i][0].x, g[i][0].y, g[i][0].z, g[i][0].w, g[i][1].x, g[i][1].y, g[i][1].z, g[i][1].w};
            uint32_t o[8];
#pragma unroll
            for (int q = 0; q < 8; ++q) o[q] = f32_to_bf16_trunc((v[q] * r) * gv[q]);
            *reinterpret_cast<uint4*>(orow + 8 * (t + NT * i)) =
                make_uint4(pack2(o[0], o[1]), pack2(o[2], o[3]), pack2(o[4], o[5]), pack2(o[6], o[7]));
        }
}

}  // namespace

__global__ __launch_bounds__(256) void rms_norm_kernel(uint16_t* out, const uint16_t* x, const float* w,
                                                       int64_t rows, int hidden, float eps) {
    const int lane = threadIdx.x & 63;
    const int64_t row = int64_t(blockIdx.x) * 4 + (threadIdx.x >> 6);
    if (row >= rows) return;
    const uint16_t* xr = x + row * hidden;
    uint16_t* orow = out + row * hidden;
    const int n32 = hidden / 32;
    float A = 0.0f;
    if (lane < 32)
        for (int b = 0; b < n32; ++b) {
            const float v = bf16_to_f32(xr[32 * b + lane]);
            A = __builtin_fmaf(v, v, A);
        }
    const float a1 = __shfl(A, (lane + 8) & 63);
    const float a2 = __shfl(A, (lane + 16) & 63);
    const float a3 = __shfl(A, (lane + 24) & 63);
    float T = (A + a1) + (a2 + a3);  // meaningful on lanes 0..7
    int j = n32 * 32;
    for (; j + 8 <= hidden; j += 8)
        if (lane < 8) {
            const float v = bf16_to_f32(xr[j + lane]);
            T = __builtin_fmaf(v, v, T);
        }
    const float u = T + __shfl(T, (lane + 4) & 63);  // lanes 0..3: u[lane]
    const float u1 = __shfl(u, 1), u2 = __shfl(u, 2), u3 = __shfl(u, 3);
    float ss = (u + u1) + (u2 + u3);
    if (lane == 0)
        for (int t = j; t < hidden; ++t) {
            const float v = bf16_to_f32(xr[t]);
            ss = __builtin_fmaf(v, v, ss);
        }
    ss = __shfl(ss, 0);
    const float r = 1.0f / __builtin_sqrtf(ss / float(hidden) + eps);
    const int vec_end = (hidden / 8) * 8;
    for (int e = lane; e < hidden; e += 64) {
        const float y = (bf16_to_f32(xr[e]) * r) * w[e];
        orow[e] = uint16_t(e < vec_end ? f32_to_bf16_trunc(y) : f32_to_bf16_ref(y));
    }
}

// One thread per slot i < head_dim/2 of a row.  Slots below rope_dim/2 rotate
// the pair (i, i + rope_dim/2) with table entry [pos][i] (rows of rope_dim
// floats); slot i >= rope_dim/2 copies the two elements rope_dim + 2(i -
// rope_dim/2) + {0, 1} unchanged.  rope_dim == head_dim is the reference op.
// With `ctl` (a device-position decode step) the start position is the
// control block's pos; a step whose rows would pass the table's max_seq rows
// raises the block's error flag and writes nothing, as does any step after a
// refused one (the flag stays set until the host syncs the layer).
//
// Start position of a launch; false: a refused step, nothing to do.
template <bool kDevPos>
__device__ __forceinline__ bool rope_start(int32_t* ctl, int seq_len, int64_t max_seq, int64_t& start_pos) {
    if constexpr (kDevPos) {
        start_pos = __builtin_amdgcn_readfirstlane(
            __hip_atomic_load(ctl + kStepPos, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT));
        if (__hip_atomic_load(ctl + kStepError, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)) return false;
        if (start_pos < 0 || start_pos + seq_len > max_seq) {
            if (blockIdx.x == 0 && threadIdx.x == 0)
                __hip_atomic_store(ctl + kStepError, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            return false;
        }
    }
    return true;
}

template <bool kDevPos>
__global__ __launch_bounds__(256) void apply_rope_kernel(uint16_t* out, const uint16_t* x, const float* cos_tab,
                                                         const float* sin_tab, int64_t rows, int seq_len,
                                                         int head_dim, int rope_dim, int64_t start_pos,
                                                         int32_t* ctl, int64_t max_seq) {
    const int half = head_dim / 2, rhalf = rope_dim / 2;
    if (!rope_start<kDevPos>(ctl, seq_len, max_seq, start_pos)) return;
    const int64_t idx = int64_t(blockIdx.x) * blockDim.x + threadIdx.x;
    if (idx >= rows * half) return;
    const int64_t row = idx / half;
    const int i = int(idx - row * half);
    const uint16_t* xr = x + row * head_dim;
    uint16_t* orow = out + row * head_dim;
    if (i >= rhalf) {
        const int e = rope_dim + 2 * (i - rhalf);
        orow[e] = xr[e];
        orow[e + 1] = xr[e + 1];
        return;
    }
    const int64_t pos = start_pos + row % seq_len;
    const float c = cos_tab[pos * rope_dim + i], s = sin_tab[pos * rope_dim + i];
    const float x0 = bf16_to_f32(xr[i]);
    const float x1 = bf16_to_f32(xr[i + rhalf]);
    orow[i] = uint16_t(f32_to_bf16_ref(__builtin_fmaf(x0, c, -(x1 * s))));
    orow[i + rhalf] = uint16_t(f32_to_bf16_ref(__builtin_fmaf(x0, s, x1 * c)));
}

// The same pairs, eight per thread with 16-byte accesses: thread (s, slot) of
// HP heads, which share the position's table entries.  Slots below rope_dim/16
// rotate pairs 8 slot .. +7, the others copy eight elements.  Needs rope_dim a
// multiple of 16, head_dim of 8, 16-byte pointers.  Bound by memory (data, and
// the tables through L2): 32 heads of 128, 1500 tokens 7.0 us, 4096 tokens 12.3
// us (5.5 TB/s); 11.5 and 26.1 us in apply_rope_kernel.
template <bool kDevPos, int HP>
__global__ __launch_bounds__(256) void apply_rope_vec_kernel(uint16_t* out, const uint16_t* x, const float* cos_tab,
                                                             const float* sin_tab, int n_heads, int seq_len,
                                                             int head_dim, int rope_dim, int64_t start_pos,
                                                             int32_t* ctl, int64_t max_seq) {
    if (!rope_start<kDevPos>(ctl, seq_len, max_seq, start_pos)) return;
    const unsigned rot = unsigned(rope_dim) / 16, slots = rot + unsigned(head_dim - rope_dim) / 8;
    const unsigned idx = blockIdx.x * 256u + threadIdx.x;
    const unsigned sq = idx / slots, slot = idx - sq * slots;
    if (sq >= unsigned(seq_len)) return;
    const int h0 = int(blockIdx.y) * HP;
    const int n = min(HP, n_heads - h0);
    const int64_t hstride = int64_t(seq_len) * head_dim;
    const int64_t base = h0 * hstride + int64_t(sq) * head_dim;
    if (slot >= rot) {
        const int64_t at = base + rope_dim + 8 * (slot - rot);
#pragma unroll
        for (int i = 0; i < HP; ++i)
            if (i < n) *reinterpret_cast<uint4*>(out + at + i * hstride) = *reinterpret_cast<const uint4*>(x + at + i * hstride);
        return;
    }
    const int64_t at = base + 8 * slot;
    const int half = rope_dim / 2;
    uint4 lo[HP], hi[HP];
#pragma unroll
    for (int i = 0; i < HP; ++i)
        if (i < n) {
            lo[i] = *reinterpret_cast<const uint4*>(x + at + i * hstride);
            hi[i] = *reinterpret_cast<const uint4*>(x + at + i * hstride + half);
        }
    float c[8], s[8];
    {
        const int64_t tab = (start_pos + sq) * rope_dim + 8 * slot;
        const float4 c0 = *reinterpret_cast<const float4*>(cos_tab + tab), c1 = *reinterpret_cast<const float4*>(cos_tab + tab + 4);
        const float4 s0 = *reinterpret_cast<const float4*>(sin_tab + tab), s1 = *reinterpret_cast<const float4*>(sin_tab + tab + 4);
        c[0] = c0.x, c[1] = c0.y, c[2] = c0.z, c[3] = c0.w, c[4] = c1.x, c[5] = c1.y, c[6] = c1.z, c[7] = c1.w;
        s[0] = s0.x, s[1] = s0.y, s[2] = s0.z, s[3] = s0.w, s[4] = s1.x, s[5] = s1.y, s[6] = s1.z, s[7] = s1.w;
    }
#pragma unroll
    for (int i = 0; i < HP; ++i)
        if (i < n) {
            float x0[8], x1[8];
            unpack8(lo[i], x0);
            unpack8(hi[i], x1);
            float o0[8], o1[8];
#pragma unroll
            for (int e = 0; e < 8; ++e) {
                o0[e] = __builtin_fmaf(x0[e], c[e], -(x1[e] * s[e]));
                o1[e] = __builtin_fmaf(x0[e], s[e], x1[e] * c[e]);
            }
            *reinterpret_cast<uint4*>(out + at + i * hstride) =
                make_uint4(bf16_pair_out(o0[0], o0[1]), bf16_pair_out(o0[2], o0[3]), bf16_pair_out(o0[4], o0[5]),
                           bf16_pair_out(o0[6], o0[7]));
            *reinterpret_cast<uint4*>(out + at + i * hstride + half) =
                make_uint4(bf16_pair_out(o1[0], o1[1]), bf16_pair_out(o1[2], o1[3]), bf16_pair_out(o1[4], o1[5]),
                           bf16_pair_out(o1[6], o1[7]));
        }
}

static bool aligned16(const void* p) { return (reinterpret_cast<uintptr_t>(p) & 15) == 0; }

int launch_rms_norm(uint16_t* out, const uint16_t* x, const float* w, int64_t rows, int hidden, float eps,
                    hipStream_t stream) {
    if (rows <= 0) return GENLLM_OK;
    if (aligned16(out) && aligned16(x) && aligned16(w) && hidden % 8 == 0) {
        const unsigned hb = unsigned((rows + 31) / 32);
        if (hidden == 64 || hidden == 128 || hidden == 256) {
            auto* k = hidden == 64 ? rms_norm_head_kernel<2> : hidden == 128 ? rms_norm_head_kernel<4> : rms_norm_head_kernel<8>;
            hipLaunchKernelGGL(k, dim3(hb), dim3(256), 0, stream, out, x, w, rows, eps);
            GENLLM_LAUNCH_CHECK("rms_norm_head_kernel");
            return GENLLM_OK;
        }
        // rows of 8 to 32768 elements; a grid of at most 2^31 threads
        if (hidden <= 32768 && rows <= (int64_t(1) << 31) / 1024) {
            const int nt = hidden <= 512 ? 64 : hidden <= 1024 ? 128 : hidden <= 8192 ? 256 : 1024;
            auto* k = hidden <= 512    ? rms_norm_row_kernel<64, 1>
                      : hidden <= 1024 ? rms_norm_row_kernel<128, 1>
                      : hidden <= 2048 ? rms_norm_row_kernel<256, 1>
                      : hidden <= 4096 ? rms_norm_row_kernel<256, 2>
                      : hidden <= 8192 ? rms_norm_row_kernel<256, 4>
                                       : rms_norm_row_kernel<1024, 4>;
            hipLaunchKernelGGL(k, dim3(unsigned(rows)), dim3(nt), size_t(hidden) * 2, stream, out, x, w, hidden, eps);
            GENLLM_LAUNCH_CHECK("rms_norm_row_kernel");
            return GENLLM_OK;
        }
    }
    const int64_t blocks = (rows + 3) / 4;
    hipLaunchKernelGGL(rms_norm_kernel, dim3(unsigned(blocks)), dim3(256), 0, stream, out, x, w, rows, hidden, eps);
    GENLLM_LAUNCH_CHECK("rms_norm_kernel");
    return GENLLM_OK;
}

template <bool kDevPos>
static void launch_rope(uint16_t* out, const uint16_t* x, const float* cos_tab, const float* sin_tab, int n_heads,
                        int seq_len, int head_dim, int rope_dim, int64_t start_pos, hipStream_t stream, int32_t* ctl,
                        int64_t max_seq) {
    const int64_t rows = int64_t(n_heads) * seq_len;
    // below kRopeVecPairs pairs the one-pair kernel's shorter chain is as fast or
    // faster (32 heads: 1 token 2.19 against 2.36 us, 64 tokens 2.35 against
    // 2.38, 300 tokens 3.66 against 2.91)
    constexpr int64_t kRopeVecPairs = 1 << 18;
    if (rows * (head_dim / 2) >= kRopeVecPairs && rope_dim % 16 == 0 && head_dim % 8 == 0 && aligned16(out) && aligned16(x) && aligned16(cos_tab) && aligned16(sin_tab)) {
        const int64_t per = int64_t(rope_dim / 16 + (head_dim - rope_dim) / 8) * seq_len;
        // two heads share a thread's table reads in the largest calls (32 heads:
        // 4096 tokens 12.3 against 15.5 us, 1500 tokens 7.9 against 7.0)
        const int hp = per * n_heads >= int64_t(device_cu_count()) * 2048 ? 2 : 1;
        const int groups = (n_heads + hp - 1) / hp;
        if (per <= INT_MAX && groups <= 65535 && per * groups <= INT_MAX) {
            auto* k = hp == 2 ? apply_rope_vec_kernel<kDevPos, 2> : apply_rope_vec_kernel<kDevPos, 1>;
            hipLaunchKernelGGL(k, dim3(unsigned((per + 255) / 256), unsigned(groups)), dim3(256), 0, stream, out, x, cos_tab,
                               sin_tab, n_heads, seq_len, head_dim, rope_dim, start_pos, ctl, max_seq);
            return;
        }
    }
    const int64_t n = rows * (head_dim / 2);
    hipLaunchKernelGGL(apply_rope_kernel<kDevPos>, dim3(unsigned((n + 255) / 256)), dim3(256), 0, stream, out, x, cos_tab,
                       sin_tab, rows, seq_len, head_dim, rope_dim, start_pos, ctl, max_seq);
}

int launch_apply_rope(uint16_t* out, const uint16_t* x, const float* cos_tab, const float* sin_tab, int n_heads,
                      int seq_len, int head_dim, int rope_dim, int64_t start_pos, hipStream_t stream, int32_t* ctl,
                      int64_t max_seq) {
    if (int64_t(n_heads) * seq_len * (head_dim / 2) <= 0) return GENLLM_OK;
    if (ctl)
        launch_rope<true>(out, x, cos_tab, sin_tab, n_heads, seq_len, head_dim, rope_dim, 0, stream, ctl, max_seq);
    else
        launch_rope<false>(out, x, cos_tab, sin_tab, n_heads, seq_len, head_dim, rope_dim, start_pos, stream, ctl, max_seq);
    GENLLM_LAUNCH_CHECK("apply_rope kernel");
    return GENLLM_OK;
}

}  // namespace genllm
