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
#include <algorithm>
#include <type_traits>

#include "epilogue.h"

namespace gk {

// A 16-byte access at any address: one global_load_dwordx4, whose address only
// has to be a byte address.
typedef uint32_t v4u_any __attribute__((ext_vector_type(4), aligned(1)));
typedef uint32_t v4u_p __attribute__((ext_vector_type(4)));

// The words of a block's row: 16 bytes, or 8 for the 8 x 8 block of bytes.
typedef uint32_t v2u_any __attribute__((ext_vector_type(2), aligned(1)));
typedef uint32_t v2u_p __attribute__((ext_vector_type(2)));
template <int BYTES> struct PackVec { using any = v4u_any; using vec = v4u_p; };
template <> struct PackVec<8> { using any = v2u_any; using vec = v2u_p; };

// Transposes the B x B elements of a thread (in[i] holds k = i of B consecutive
// rows) into out[j]: B consecutive k of row j.
template <int ESZ, int B, typename V>
__device__ __forceinline__ void transpose_block(const V (&in)[B], V (&out)[B]) {
    if constexpr (ESZ == 4) {
#pragma unroll
        for (int j = 0; j < 4; ++j) out[j] = V{in[0][j], in[1][j], in[2][j], in[3][j]};
    } else if constexpr (ESZ == 2) {
#pragma unroll
        for (int j = 0; j < 8; ++j)
#pragma unroll
            for (int p = 0; p < 4; ++p)
                out[j][p] = __builtin_amdgcn_perm(in[2 * p + 1][j >> 1], in[2 * p][j >> 1],
                                                  (j & 1) ? 0x07060302u : 0x05040100u);
    } else {
#pragma unroll
        for (int c = 0; c < B / 4; ++c)
#pragma unroll
            for (int p = 0; p < B / 4; ++p) {
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
// memory, by latency below a few MB.  A lane owns a block of B rows x B k and
// transposes it in registers; the wave's lanes lie 8 along the rows x 8 along
// k, so every load instruction reads 8 runs of 8*B elements and every store
// writes as many, with no LDS and no barrier, all B loads of a lane in flight
// at once.  B fills 16 bytes (runs of 128), or is 8 for an i8 operand too small
// to give every CU a few waves that way (i8 1712 x 288 x 128 with A column-major
// 7.2 us in all against 8.5).  bf16 4096 x 4096: 12.0 us (5.6 TB/s read + write,
// a large copy reaches 5.2) against 18.8 through pack_kernel's LDS tile with its
// element-wide accesses, 11008 x 4096 33.3 against 41.1, f32 2048 x 2048 8.0
// against 9.2.
template <typename T, int B>
__device__ __forceinline__ void pack_tr(const PackJob &j, int block) {
    constexpr int ESZ = (int)sizeof(T);
    using Vec = typename PackVec<B * ESZ>::vec;
    using Any = typename PackVec<B * ESZ>::any;
    const T *src = (const T *)j.src + (int64_t)blockIdx.y * j.bs;
    T *dst = (T *)j.dst + (int64_t)blockIdx.y * j.rows * j.ld;
    const int64_t cs = j.cs, rows = j.rows, K = j.K, ld = j.ld;
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    // A workgroup's four waves: 2 along the rows x 2 along k.  The last lanes
    // along the rows start B rows before the end (the caller ensures rows >=
    // B): rows their neighbours also pack, with the same values.
    int64_t r0 = ((int64_t)(block % j.p0) * 16 + (wave & 1) * 8 + (lane & 7)) * B;
    const int64_t p0 = ((int64_t)(block / j.p0) * 16 + (wave >> 1) * 8 + (lane >> 3)) * B;
    if (r0 >= rows || p0 >= ld) return;
    if (r0 + B > rows) r0 = rows - B;
    const T *s = src + r0 + p0 * cs;
    Vec in[B], out[B];
    if (p0 + B <= K) {
#pragma unroll
        for (int i = 0; i < B; ++i) in[i] = *(const Any *)(s + i * cs);
    } else {  // zeros past K
#pragma unroll
        for (int i = 0; i < B; ++i) {
            in[i] = Vec{};
            if (p0 + i < K) in[i] = *(const Any *)(s + i * cs);
        }
    }
    transpose_block<ESZ, B>(in, out);
    T *d = dst + r0 * ld + p0;
#pragma unroll
    for (int i = 0; i < B; ++i) *(Vec *)(d + i * ld) = out[i];
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
// lane takes four rows at a time, and a workgroup at most j.copy chunks of its
// rows: kCopyChunks, or one per lane while that leaves fewer workgroups than CUs
// (a lane's chunks are round trips in series: i8 32 x 4665 times 4665 x 2 in all 11.6
// us with two workgroups, 9.6 with ten, as through pack_kernel; with a k-contiguous
// right side 8.2, 6.2 and 9.3).
// A row's last chunk is the 16 bytes before the row's end, shifted
// down (the caller ensures K >= EPV), so no lane goes element by element.
// i8 777 x 1001: 3.8 us against 4.6 through pack_kernel, 11008 x 4097: 22 against 38.
constexpr int kCopyChunks = 256, kCopyRows = 4;
template <typename T>
__device__ __forceinline__ void pack_copy(const PackJob &j, int block) {
    constexpr int EPV = 16 / (int)sizeof(T);
    const T *src = (const T *)j.src + (int64_t)blockIdx.y * j.bs;
    T *dst = (T *)j.dst + (int64_t)blockIdx.y * j.rows * j.ld;
    const int64_t rs = j.rs, rows = j.rows, K = j.K, ld = j.ld;
    const int blocks_c = j.p0, llog = j.p1;
    const int lanes = 1 << llog, groups = 256 >> llog;
    const int64_t cpr = ld / EPV;
    const int64_t c0 = (int64_t)(block % blocks_c) * j.copy;
    const int64_t c1 = c0 + j.copy < cpr ? c0 + j.copy : cpr;
    const int64_t r0 = (int64_t)(block / blocks_c) * groups * kCopyRows +
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

// One or two operands (the two of a product whose K is ragged) in one launch.
template <typename T>
__global__ __launch_bounds__(256) void pack_jobs(const PackJob a, const PackJob b) {
    const bool first = (int)blockIdx.x < a.blocks;
    const PackJob &j = first ? a : b;
    const int block = (int)blockIdx.x - (first ? 0 : a.blocks);
    if ((int)blockIdx.y >= j.batch) return;
    if (j.copy) {
        pack_copy<T>(j, block);
    } else if (sizeof(T) > 1 || j.p1) {
        pack_tr<T, 16 / (int)sizeof(T)>(j, block);
    } else {
        pack_tr<T, sizeof(T) == 1 ? 8 : 16 / (int)sizeof(T)>(j, block);
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

// Plans j for pack_jobs; false when its strides or sizes need pack_kernel.
static bool plan_pack(PackJob &j, int64_t epv) {
    constexpr int64_t kMaxX = 1 << 23;  // workgroups of 256 in grid x, two jobs together
    int64_t blocks;
    if (j.cs == 1 && j.K >= epv) {
        const int64_t cpr = j.ld / epv;
        int llog = 0;
        while (llog < 6 && (1 << llog) < cpr) ++llog;
        const int64_t rpb = (int64_t)(256 >> llog) * kCopyRows;
        const int64_t br = (j.rows + rpb - 1) / rpb;
        int64_t bc = (cpr + kCopyChunks - 1) / kCopyChunks;
        j.copy = kCopyChunks;
        if (bc * br * j.batch < 256) {
            j.copy = 64;
            bc = (cpr + 63) / 64;
        }
        blocks = bc * br;
        j.p0 = (int)bc;
        j.p1 = llog;
    } else if (j.rs == 1 && j.rows >= epv) {
        // 16-byte blocks; i8 takes 8 x 8 ones while they leave fewer than about
        // four waves per CU.
        j.copy = 0;
        j.p1 = epv < 16 || (double)j.rows * j.ld * j.batch >= 1024.0 * 64 * 256;
        const int64_t b = j.p1 ? epv : 8;
        const int64_t tr = (j.rows + 16 * b - 1) / (16 * b);
        blocks = tr * ((j.ld + 16 * b - 1) / (16 * b));
        j.p0 = (int)tr;
    } else {
        return false;
    }
    if (blocks >= kMaxX) return false;
    j.blocks = (int)blocks;
    return true;
}

template <typename T>
static hipError_t pack_go(PackJob *jobs, int n, hipStream_t stream) {
    PackJob run[2] = {};
    int nr = 0;
    for (int i = 0; i < n; ++i) {
        PackJob &j = jobs[i];
        if (plan_pack(j, 16 / (int)sizeof(T))) {
            run[nr++] = j;
            continue;
        }
        const dim3 grid((unsigned)((j.ld + 63) / 64), (unsigned)((j.rows + 63) / 64),
                        (unsigned)j.batch);
        hipLaunchKernelGGL(pack_kernel<T>, grid, dim3(256), 0, stream, (const T *)j.src, j.rs,
                           j.cs, j.bs, j.rows, j.K, (T *)j.dst, j.ld, j.rows * j.ld);
    }
    if (nr > 0)
        hipLaunchKernelGGL(pack_jobs<T>, dim3((unsigned)(run[0].blocks + run[1].blocks),
                                              (unsigned)std::max(run[0].batch, run[1].batch)),
                           dim3(256), 0, stream, run[0], run[1]);
    return hipGetLastError();
}

hipError_t launch_pack(InType in, PackJob *jobs, int n, hipStream_t stream) {
    if (n < 1 || n > 2) return hipErrorInvalidValue;
    for (int i = 0; i < n; ++i)
        if (jobs[i].batch < 1 || jobs[i].batch > kMaxGridZ) return hipErrorInvalidValue;
    switch (in_size(in)) {
    case 1: return pack_go<uint8_t>(jobs, n, stream);
    case 2: return pack_go<uint16_t>(jobs, n, stream);
    default: return pack_go<uint32_t>(jobs, n, stream);
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
