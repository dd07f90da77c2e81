// pack.hip -- layout and degenerate-case kernels.
//
//   pack_tr, pack_copy, pack_kernel
//                    copy a strided operand into the kernels' k-contiguous
//                    layout (gemmkit's pack_panels role, src/pack.rs:28-117, but
//                    one plain row-per-row layout instead of micropanels):
//                    pack_tr a unit-row-stride operand (a row-major B, a
//                    column-major A), pack_copy a k-contiguous one that only
//                    misses the alignment, pack_kernel any other strides.
//   scale_c_kernel   C <- beta*C when the A*B term vanishes (scale_c_int,
//                    src/dispatch/int.rs:150-163; scale_c_float,
//                    src/dispatch.rs:484-497; the narrow twin for bf16).
//   requant_fill     the k == 0 requant fill (requant_degenerate,
//                    src/dispatch/int.rs:735-752).
//   fused_fill       C <- act(beta*C + bias) when the A*B term of a fused
//                    call vanishes (src/dispatch/float.rs:661-680).
//   split_reduce     sums the partial products of a split-K matrix-core launch
//                    and applies the call's epilogue.
#include <type_traits>

#include "epilogue.h"

namespace gk {

// A 16-byte access at any address: one global_load_dwordx4, whose address only
// has to be a byte address.
typedef uint32_t v4u_any __attribute__((ext_vector_type(4), aligned(1)));
typedef uint32_t v4u_p __attribute__((ext_vector_type(4)));

// Transposes the EPV x EPV elements of a thread (in[i] holds k = i of EPV
// consecutive rows) into out[j]: EPV consecutive k of row j.
template <int ESZ>
__device__ __forceinline__ void transpose_block(const v4u_p (&in)[16 / ESZ],
                                                v4u_p (&out)[16 / ESZ]) {
    if constexpr (ESZ == 4) {
#pragma unroll
        for (int j = 0; j < 4; ++j) out[j] = v4u_p{in[0][j], in[1][j], in[2][j], in[3][j]};
    } else if constexpr (ESZ == 2) {
#pragma unroll
        for (int j = 0; j < 8; ++j)
#pragma unroll
            for (int p = 0; p < 4; ++p)
                out[j][p] = __builtin_amdgcn_perm(in[2 * p + 1][j >> 1], in[2 * p][j >> 1],
                                                  (j & 1) ? 0x07060302u : 0x05040100u);
    } else {
#pragma unroll
        for (int c = 0; c < 4; ++c)
#pragma unroll
            for (int p = 0; p < 4; ++p) {
                const uint32_t i0 = in[4 * p][c], i1 = in[4 * p + 1][c];
                const uint32_t i2 = in[4 * p + 2][c], i3 = in[4 * p + 3][c];
                const uint32_t t0 = __builtin_amdgcn_perm(i1, i0, 0x05010400u);
                const uint32_t t1 = __builtin_amdgcn_perm(i1, i0, 0x07030602u);
                const uint32_t u0 = __builtin_amdgcn_perm(i3, i2, 0x05010400u);
                const uint32_t u1 = __builtin_amdgcn_perm(i3, i2, 0x07030602u);
                out[4 * c][p] = __builtin_amdgcn_perm(u0, t0, 0x05040100u);
                out[4 * c + 1][p] = __builtin_amdgcn_perm(u0, t0, 0x07060302u);
                out[4 * c + 2][p] = __builtin_amdgcn_perm(u1, t1, 0x05040100u);
                out[4 * c + 3][p] = __builtin_amdgcn_perm(u1, t1, 0x07060302u);
            }
    }
}

// Unit row stride (element (r, p) at r + p*cs): the transposing pack.  Bound by
// memory.  A lane owns a block of EPV rows x EPV k (16 bytes each way) and
// transposes it in registers, the wave's lanes lie 8 along the rows x 8 along
// k, so every load instruction reads 8 runs of 128 bytes and every store
// writes 8 runs of 128 bytes, with no LDS and no barrier, all EPV loads of a
// lane in flight at once.  bf16 4096 x 4096: 12.0 us (5.6 TB/s read + write, a
// large copy reaches 5.2) against 18.8 through pack_kernel's LDS tile with its
// element-wide accesses, 11008 x 4096 33.3 against 41.1, f32 2048 x 2048 8.0
// against 9.2.
template <typename T>
__global__ __launch_bounds__(256) void pack_tr(const T *__restrict__ src, int64_t cs, int64_t bs,
                                               int64_t rows, int64_t K, T *__restrict__ dst,
                                               int64_t ld, int64_t dbs, int tiles_r) {
    constexpr int ESZ = (int)sizeof(T), EPV = 16 / ESZ;
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    // A workgroup's four waves: 2 along the rows x 2 along k.  The last lanes
    // along the rows start EPV rows before the end (the caller ensures rows >=
    // EPV): rows their neighbours also pack, with the same values.
    int64_t r0 = ((int64_t)(blockIdx.x % tiles_r) * 16 + (wave & 1) * 8 + (lane & 7)) * EPV;
    const int64_t p0 = ((int64_t)(blockIdx.x / tiles_r) * 16 + (wave >> 1) * 8 + (lane >> 3)) * EPV;
    if (r0 >= rows || p0 >= ld) return;
    if (r0 + EPV > rows) r0 = rows - EPV;
    const T *s = src + (int64_t)blockIdx.y * bs + r0 + p0 * cs;
    dst += (int64_t)blockIdx.y * dbs;
    v4u_p in[EPV], out[EPV];
    if (p0 + EPV <= K) {
#pragma unroll
        for (int i = 0; i < EPV; ++i) in[i] = *(const v4u_any *)(s + i * cs);
    } else {  // zeros past K
#pragma unroll
        for (int i = 0; i < EPV; ++i) {
            in[i] = v4u_p{0, 0, 0, 0};
            if (p0 + i < K) in[i] = *(const v4u_any *)(s + i * cs);
        }
    }
    transpose_block<ESZ>(in, out);
    T *d = dst + r0 * ld + p0;
#pragma unroll
    for (int j = 0; j < EPV; ++j) *(v4u_p *)(d + j * ld) = out[j];
}

// The 16 bytes of v from byte `sh` (0..15) on, zeros behind them.
__device__ __forceinline__ v4u_p shift_down(v4u_p v, int sh) {
    const uint32_t w[8] = {v[0], v[1], v[2], v[3], 0, 0, 0, 0};
    const int d = sh >> 2;
    v4u_p o;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const uint32_t lo = d == 0 ? w[i] : (d == 1 ? w[i + 1] : (d == 2 ? w[i + 2] : w[i + 3]));
        const uint32_t hi = d == 0 ? w[i + 1] : (d == 1 ? w[i + 2] : (d == 2 ? w[i + 3] : w[i + 4]));
        o[i] = __builtin_amdgcn_alignbyte(hi, lo, (uint32_t)sh & 3u);
    }
    return o;
}

// k-contiguous rows (element (r, p) at r*rs + p) whose base, stride or length
// misses the 16-byte alignment: a copy of 16 bytes per lane.  Bound by memory,
// by latency below a few MB.  2^llog lanes (at most 64) walk a row's chunks, a
// lane takes four rows at a time, and a workgroup at most kCopyChunks chunks of
// its rows.  A row's last chunk is the 16 bytes before the row's end, shifted
// down (the caller ensures K >= EPV), so no lane goes element by element.
// i8 777 x 1001: 3.8 us against 4.6 through pack_kernel, 11008 x 4097: 22 against 38.
constexpr int kCopyChunks = 256, kCopyRows = 4;
template <typename T>
__global__ __launch_bounds__(256) void pack_copy(const T *__restrict__ src, int64_t rs, int64_t bs,
                                                 int64_t rows, int64_t K, T *__restrict__ dst,
                                                 int64_t ld, int64_t dbs, int llog, int blocks_c) {
    constexpr int EPV = 16 / (int)sizeof(T);
    src += (int64_t)blockIdx.y * bs;
    dst += (int64_t)blockIdx.y * dbs;
    const int lanes = 1 << llog, groups = 256 >> llog;
    const int64_t cpr = ld / EPV;
    const int64_t c0 = (int64_t)(blockIdx.x % blocks_c) * kCopyChunks;
    const int64_t c1 = c0 + kCopyChunks < cpr ? c0 + kCopyChunks : cpr;
    const int64_t r0 = (int64_t)(blockIdx.x / blocks_c) * groups * kCopyRows +
                       ((int)threadIdx.x >> llog);
    for (int64_t c = c0 + ((int)threadIdx.x & (lanes - 1)); c < c1; c += lanes) {
        const int64_t p = c * EPV < K - EPV ? c * EPV : K - EPV;  // first element loaded
        const int sh = (int)(c * EPV - p) * (int)sizeof(T);
        v4u_p v[kCopyRows];
#pragma unroll
        for (int u = 0; u < kCopyRows; ++u) {
            const int64_t r = r0 + u * groups;
            v[u] = *(const v4u_any *)(src + (r < rows ? r : rows - 1) * rs + p);
        }
#pragma unroll
        for (int u = 0; u < kCopyRows; ++u) {
            const int64_t r = r0 + u * groups;
            if (r < rows) *(v4u_p *)(dst + r * ld + c * EPV) = shift_down(v[u], sh);
        }
    }
}

// Any other strides: a 64 x 64 tile goes through LDS so both the strided read
// and the k-contiguous write are coalesced where the strides allow it.
template <typename T>
__global__ __launch_bounds__(256) void pack_kernel(const T *__restrict__ src, int64_t rs,
                                                   int64_t cs, int64_t bs, int64_t rows, int64_t K,
                                                   T *__restrict__ dst, int64_t ld, int64_t dbs) {
    __shared__ T tile[64][65];
    src += (int64_t)blockIdx.z * bs;
    dst += (int64_t)blockIdx.z * dbs;
    const int64_t r0 = (int64_t)blockIdx.y * 64;
    const int64_t p0 = (int64_t)blockIdx.x * 64;
    const int tx = threadIdx.x & 63, ty = threadIdx.x >> 6;  // 64 x 4
    // Read: let consecutive threads walk the operand's faster-moving index.
    // All 16 loads of a thread are issued before any is used (one memory
    // round trip per tile, not sixteen).
    const bool k_fast = (cs < 0 ? -cs : cs) <= (rs < 0 ? -rs : rs);
    T v[16];
#pragma unroll
    for (int i = 0; i < 16; ++i) {
        const int y = ty + 4 * i;
        int64_t r, p;
        if (k_fast) { r = r0 + y; p = p0 + tx; } else { r = r0 + tx; p = p0 + y; }
        v[i] = (r < rows && p < K) ? src[r * rs + p * cs] : T(0);
    }
#pragma unroll
    for (int i = 0; i < 16; ++i) {
        const int y = ty + 4 * i;
        if (k_fast) tile[y][tx] = v[i]; else tile[tx][y] = v[i];
    }
    __syncthreads();
    // Write: consecutive threads write consecutive k; columns [K, ld) get zeros.
#pragma unroll
    for (int i = 0; i < 16; ++i) {
        const int y = ty + 4 * i;
        int64_t r = r0 + y, p = p0 + tx;
        if (r < rows && p < ld) dst[r * ld + p] = (p < K) ? tile[y][tx] : T(0);
    }
}

template <typename T>
static hipError_t pack_go(const T *src, int64_t rs, int64_t cs, int64_t bs, int64_t rows,
                          int64_t K, T *dst, int64_t ld, int64_t dbs, int64_t batch,
                          hipStream_t stream) {
    constexpr int EPV = 16 / (int)sizeof(T);
    constexpr int64_t kMaxX = 1 << 24;  // workgroups of 256 in grid x
    if (cs == 1 && K >= EPV) {
        const int64_t cpr = ld / EPV;
        int llog = 0;
        while (llog < 6 && (1 << llog) < cpr) ++llog;
        const int64_t rpb = (int64_t)(256 >> llog) * kCopyRows;
        const int64_t bc = (cpr + kCopyChunks - 1) / kCopyChunks, br = (rows + rpb - 1) / rpb;
        if (bc * br < kMaxX) {
            hipLaunchKernelGGL(pack_copy<T>, dim3((unsigned)(bc * br), (unsigned)batch), dim3(256),
                               0, stream, src, rs, bs, rows, K, dst, ld, dbs, llog, (int)bc);
            return hipGetLastError();
        }
    } else if (rs == 1 && rows >= EPV) {
        const int64_t tr = (rows + 16 * EPV - 1) / (16 * EPV), tk = (ld + 16 * EPV - 1) / (16 * EPV);
        if (tr * tk < kMaxX) {
            hipLaunchKernelGGL(pack_tr<T>, dim3((unsigned)(tr * tk), (unsigned)batch), dim3(256), 0,
                               stream, src, cs, bs, rows, K, dst, ld, dbs, (int)tr);
            return hipGetLastError();
        }
    }
    const dim3 grid((unsigned)((ld + 63) / 64), (unsigned)((rows + 63) / 64), (unsigned)batch);
    hipLaunchKernelGGL(pack_kernel<T>, grid, dim3(256), 0, stream, src, rs, cs, bs, rows, K, dst,
                       ld, dbs);
    return hipGetLastError();
}

hipError_t launch_pack(InType in, const void *src, int64_t rs, int64_t cs, int64_t bs,
                       int64_t rows, int64_t K, void *dst, int64_t ld, int64_t batch,
                       hipStream_t stream) {
    if (batch < 1 || batch > kMaxGridZ) return hipErrorInvalidValue;
    switch (in_size(in)) {
    case 1:
        return pack_go((const uint8_t *)src, rs, cs, bs, rows, K, (uint8_t *)dst, ld, rows * ld,
                       batch, stream);
    case 2:
        return pack_go((const uint16_t *)src, rs, cs, bs, rows, K, (uint16_t *)dst, ld, rows * ld,
                       batch, stream);
    default:
        return pack_go((const uint32_t *)src, rs, cs, bs, rows, K, (uint32_t *)dst, ld, rows * ld,
                       batch, stream);
    }
}

// One thread per element of a (batch x) m x n view; beta == 1 never launches.
__global__ __launch_bounds__(256) void scale_c_kernel(int kind, void *c, int64_t m, int64_t n,
                                                      int64_t rsc, int64_t csc, int64_t bsc,
                                                      int32_t beta_i, float beta_f) {
    const int64_t idx = (int64_t)blockIdx.x * 256 + threadIdx.x;
    const int64_t z = blockIdx.y;
    if (idx >= m * n) return;
    const int64_t i = idx / n, j = idx % n;
    const int64_t off = z * bsc + i * rsc + j * csc;
    if (kind == (int)EpiKind::I32) {
        int32_t *p = (int32_t *)c + off;
        *p = beta_i == 0 ? 0 : (int32_t)((uint32_t)beta_i * (uint32_t)*p);
    } else if (kind == (int)EpiKind::F32) {
        float *p = (float *)c + off;
        *p = beta_f == 0.0f ? 0.0f : beta_f * *p;
    } else {
        uint16_t *p = (uint16_t *)c + off;
        *p = beta_f == 0.0f ? (uint16_t)0 : bf16_rne(beta_f * bf16_widen(*p));
    }
}

hipError_t launch_scale_c(EpiKind kind, void *c, int64_t m, int64_t n, int64_t rsc,
                          int64_t csc, int64_t batch, int64_t bsc, int32_t beta_i,
                          float beta_f, hipStream_t stream) {
    if (m == 0 || n == 0 || batch == 0) return hipSuccess;
    dim3 grid((unsigned)((m * n + 255) / 256), (unsigned)batch);
    hipLaunchKernelGGL(scale_c_kernel, grid, dim3(256), 0, stream, (int)kind, c, m, n, rsc, csc,
                       bsc, beta_i, beta_f);
    return hipGetLastError();
}

__global__ __launch_bounds__(256) void requant_fill_kernel(const EpiParams ep, int64_t m,
                                                           int64_t n) {
    const int64_t idx = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (idx >= m * n) return;
    Store<EpiKind::Q8>::apply(ep, 0, (int)(idx / n), (int)(idx % n), 0);
}

hipError_t launch_requant_fill(const EpiParams &ep, int64_t m, int64_t n, hipStream_t stream) {
    if (m == 0 || n == 0) return hipSuccess;
    dim3 grid((unsigned)((m * n + 255) / 256));
    hipLaunchKernelGGL(requant_fill_kernel, grid, dim3(256), 0, stream, ep, m, n);
    return hipGetLastError();
}

// Split-K reduction: one thread per 4 consecutive output elements of one
// batch element (blockIdx.y) when N % 4 == 0 (16-byte partial loads), else
// one per element.  The partial slabs are summed in K-range order (wrapping
// for i32), eight slabs' loads in flight at a time, then stored through the
// call's epilogue.
template <EpiKind E, typename A, int W>
__global__ __launch_bounds__(256) void split_reduce_kernel(const A *__restrict__ part, int splits,
                                                           int64_t M, int64_t N,
                                                           const EpiParams ep) {
    typedef A vec_t __attribute__((ext_vector_type(W)));
    const int64_t idx = ((int64_t)blockIdx.x * 256 + threadIdx.x) * W;
    const int64_t z = blockIdx.y;
    const int64_t slab = M * N;
    if (idx >= slab) return;
    const A *p = part + z * splits * slab + idx;
    vec_t acc = *(const vec_t *)p;
    for (int r0 = 1; r0 < splits; r0 += 8) {
        vec_t v[8];
#pragma unroll
        for (int u = 0; u < 8; ++u)
            if (r0 + u < splits) v[u] = *(const vec_t *)(p + (r0 + u) * slab);
#pragma unroll
        for (int u = 0; u < 8; ++u) {
            if (r0 + u < splits) {
                if constexpr (std::is_integral<A>::value) {
#pragma unroll
                    for (int e = 0; e < W; ++e) acc[e] = (A)((uint32_t)acc[e] + (uint32_t)v[u][e]);
                } else {
                    acc = acc + v[u];
                }
            }
        }
    }
    const int row = (int)(idx / N), col = (int)(idx % N);
#pragma unroll
    for (int e = 0; e < W; ++e) Store<E>::apply(ep, z, row, col + e, acc[e]);
}

template <EpiKind E, typename A>
static void split_reduce_go(const A *p, int splits, int64_t M, int64_t N, int64_t batch,
                            const EpiParams &ep, hipStream_t stream) {
    if (N % 4 == 0) {
        dim3 grid((unsigned)((M * N / 4 + 255) / 256), (unsigned)batch);
        hipLaunchKernelGGL((split_reduce_kernel<E, A, 4>), grid, dim3(256), 0, stream, p, splits,
                           M, N, ep);
    } else {
        dim3 grid((unsigned)((M * N + 255) / 256), (unsigned)batch);
        hipLaunchKernelGGL((split_reduce_kernel<E, A, 1>), grid, dim3(256), 0, stream, p, splits,
                           M, N, ep);
    }
}

hipError_t launch_split_reduce(InType in, const void *part, int splits, int64_t M, int64_t N,
                               int64_t batch, const EpiParams &ep, hipStream_t stream) {
    if (M == 0 || N == 0 || batch == 0) return hipSuccess;
    if (in == InType::I8) {
        const int32_t *p = (const int32_t *)part;
        if (ep.kind == EpiKind::I32)
            split_reduce_go<EpiKind::I32>(p, splits, M, N, batch, ep, stream);
        else if (ep.kind == EpiKind::Q8)
            split_reduce_go<EpiKind::Q8>(p, splits, M, N, batch, ep, stream);
        else
            return hipErrorInvalidValue;
    } else {
        const float *p = (const float *)part;
        if (ep.kind == EpiKind::F32)
            split_reduce_go<EpiKind::F32>(p, splits, M, N, batch, ep, stream);
        else if (ep.kind == EpiKind::BF16)
            split_reduce_go<EpiKind::BF16>(p, splits, M, N, batch, ep, stream);
        else
            return hipErrorInvalidValue;
    }
    return hipGetLastError();
}

// Fused degenerate map: one thread per element of a (batch x) m x n view in the
// user frame.  beta*C stays a separate rounding before the bias add, as in the
// reference's scalar loop.
__global__ __launch_bounds__(256) void fused_fill_kernel(const EpiParams ep, int64_t m,
                                                         int64_t n) {
#pragma clang fp contract(off)
    const int64_t idx = (int64_t)blockIdx.x * 256 + threadIdx.x;
    const int64_t z = blockIdx.y;
    if (idx >= m * n) return;
    const int i = (int)(idx / n), j = (int)(idx % n);
    const int64_t off = z * ep.bsc + (int64_t)i * ep.rsc + (int64_t)j * ep.csc;
    if (ep.kind == EpiKind::F32) {
        float *p = (float *)ep.c + off;
        const float base = ep.beta_f == 0.0f ? 0.0f : (ep.beta_f == 1.0f ? *p : ep.beta_f * *p);
        *p = fused_map<false>(ep, base, i, j);
    } else {
        uint16_t *p = (uint16_t *)ep.c + off;
        const float base = ep.beta_f == 0.0f
                               ? 0.0f
                               : (ep.beta_f == 1.0f ? bf16_widen(*p) : ep.beta_f * bf16_widen(*p));
        *p = bf16_rne(fused_map<true>(ep, base, i, j));
    }
}

hipError_t launch_fused_fill(const EpiParams &ep, int64_t m, int64_t n, int64_t batch,
                             hipStream_t stream) {
    if (m == 0 || n == 0 || batch == 0) return hipSuccess;
    dim3 grid((unsigned)((m * n + 255) / 256), (unsigned)batch);
    hipLaunchKernelGGL(fused_fill_kernel, grid, dim3(256), 0, stream, ep, m, n);
    return hipGetLastError();
}

}  // namespace gk
