// gemv.hip -- HBM-bandwidth GEMV for skinny products (1..8 vectors).
//
// Replaces gemmkit's gemv route (src/special/gemv.rs:101-600, taken at
// m == 1 || n == 1 by src/dispatch/float.rs:81) and serves the i8 skinny shapes
// too (the reference has no i8 gemv: src/dispatch/int.rs:165-168; i8 results do
// not depend on the route because wrapping i32 addition is associative).
//
// out[j, r] = epi( sum_p mat[r, p] * vec[j, p] ),  r < R rows, j < nvec <= 8.
//
// The matrix streams from HBM exactly once, as 16-byte nontemporal loads; it is
// the only large operand, so the kernels are built around keeping enough of it
// in flight.  A row is split into 16-byte chunks; lane l of a wave owns chunks
// l, l+64, l+128, ... of every row it visits, so the vector chunks a lane
// multiplies are the same for every row.  Waves are persistent (a grid of a
// few workgroups per CU) and walk row groups with a grid stride:
//   * gemv_reg: rows of at most 64*CPL chunks.  Each lane loads its vector
//     chunks once into registers; the next row group's matrix loads are issued
//     before the current group is multiplied, so one group is always in flight
//     behind the arithmetic.
//   * gemv_wgrow: longer rows, one or two vectors.  The vectors are staged
//     once per workgroup in LDS and the whole workgroup reads one row at a
//     time, 32 KiB per batch, the next batch in flight behind the current.
//   * gemv_lds: longer rows, more vectors.  The vectors are staged in LDS and
//     each lane keeps UNROLL chunks per row in flight.
//   * gemv_cols: a matrix with unit row stride instead (x * W with W row-major),
//     read in place; sums in the order of whichever kernel above serves the
//     same shape.
// Per-lane partial sums of the RPW x NV outputs of a row group are combined by
// a butterfly over the 64 lanes that halves the number of values each lane
// carries at every step (V values cost V-1 + log2(64/V) shuffles instead of
// 6*V), leaving output v on lanes [v*64/V, (v+1)*64/V).
#include <stdio.h>
#include <stdlib.h>

#include "epilogue.h"

namespace gk {

typedef int v4i_g __attribute__((ext_vector_type(4)));
typedef float v4f_g __attribute__((ext_vector_type(4)));

template <InType T>
struct Dot16;

template <>
struct Dot16<InType::I8> {
    using acc_t = int32_t;
    __device__ __forceinline__ static acc_t dot(v4i_g m, v4i_g x, acc_t acc) {
        acc = __builtin_amdgcn_sdot4(m[0], x[0], acc, false);
        acc = __builtin_amdgcn_sdot4(m[1], x[1], acc, false);
        acc = __builtin_amdgcn_sdot4(m[2], x[2], acc, false);
        acc = __builtin_amdgcn_sdot4(m[3], x[3], acc, false);
        return acc;
    }
};

template <>
struct Dot16<InType::F32> {
    using acc_t = float;
    __device__ __forceinline__ static acc_t dot(v4i_g m, v4i_g x, acc_t acc) {
        v4f_g a = __builtin_bit_cast(v4f_g, m), b = __builtin_bit_cast(v4f_g, x);
        acc = __builtin_fmaf(a[0], b[0], acc);
        acc = __builtin_fmaf(a[1], b[1], acc);
        acc = __builtin_fmaf(a[2], b[2], acc);
        acc = __builtin_fmaf(a[3], b[3], acc);
        return acc;
    }
};

template <>
struct Dot16<InType::BF16> {
    using acc_t = float;
    __device__ __forceinline__ static acc_t dot(v4i_g m, v4i_g x, acc_t acc) {
#pragma unroll
        for (int w = 0; w < 4; ++w) {
            uint32_t mu = (uint32_t)m[w], xu = (uint32_t)x[w];
            acc = __builtin_fmaf(__uint_as_float(mu << 16), __uint_as_float(xu << 16), acc);
            acc = __builtin_fmaf(__uint_as_float(mu & 0xFFFF0000u), __uint_as_float(xu & 0xFFFF0000u), acc);
        }
        return acc;
    }
};

// Butterfly over the wave: on entry v[0..V) are this lane's partial sums of V
// outputs; on exit v[0] holds the wave total of output (lane >> (6 - log2 V)).
template <int V, typename A>
__device__ __forceinline__ void wave_reduce(A (&v)[V]) {
    static_assert(V >= 1 && V <= 64 && (V & (V - 1)) == 0, "V must be a power of two <= 64");
    const int lane = threadIdx.x & 63;
    int n = V;
#pragma unroll
    for (int off = 32; off >= 1; off >>= 1) {
        if (n > 1) {
            const bool hi = (lane & off) != 0;
            const int h = n / 2;
#pragma unroll
            for (int i = 0; i < V / 2; ++i) {
                if (i < h) {
                    A send = hi ? v[i] : v[i + h];
                    A keep = hi ? v[i + h] : v[i];
                    v[i] = keep + __shfl_xor(send, off, 64);
                }
            }
            n = h;
        } else {
            v[0] += __shfl_xor(v[0], off, 64);
        }
    }
}

constexpr int kGemvThreads = 256;
constexpr int kGemvWaves = kGemvThreads / 64;

template <int V>
constexpr int log2c() {
    return V <= 1 ? 0 : 1 + log2c<V / 2>();
}

// Stores the reduced outputs of row group [r0, r0 + RPW): output index
// v = r*NV + j lives on lanes [v*64/V, ...); its first lane stores it.
template <InType T, EpiKind E, int NV, int RPW, typename A>
__device__ __forceinline__ void store_group(const GemvArgs &g, const EpiParams &ep, int64_t r0,
                                            const A (&v)[RPW * NV]) {
    constexpr int V = RPW * NV;
    constexpr int SH = 6 - log2c<V>();
    const int lane = threadIdx.x & 63;
    if ((lane & ((1 << SH) - 1)) == 0) {
        const int idx = lane >> SH;
        const int r = idx / NV, j = idx % NV;
        if (j < g.nvec && r0 + r < g.R) Store<E>::apply(ep, blockIdx.y, j, (int)(r0 + r), v[0]);
    }
}

template <InType T, EpiKind E, int NV, int CPL, int RPW>
__global__ __launch_bounds__(kGemvThreads) void gemv_reg(const GemvArgs g, const EpiParams ep) {
    using D = Dot16<T>;
    using acc_t = typename D::acc_t;
    constexpr int esz = (T == InType::I8) ? 1 : (T == InType::BF16 ? 2 : 4);
    // A K*esz that is not a multiple of 16 only reaches this kernel through
    // the pack, which zero-fills both operands' rows up to the next 16 bytes.
    const int nch = (int)(((int64_t)g.K * esz + 15) / 16);
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int64_t zb = blockIdx.y;  // batch element
    const uint8_t *mat = (const uint8_t *)g.mat + zb * g.bsm * esz;
    const uint8_t *vec = (const uint8_t *)g.vec + zb * g.bsv * esz;
    const int64_t ld_b = g.ld * esz, vld_b = g.vld * esz;

    v4i_g x[NV][CPL];
#pragma unroll
    for (int j = 0; j < NV; ++j)
#pragma unroll
        for (int u = 0; u < CPL; ++u) {
            const int c = lane + 64 * u;
            x[j][u] = (j < g.nvec && c < nch) ? *(const v4i_g *)(vec + j * vld_b + (int64_t)c * 16)
                                              : v4i_g{0, 0, 0, 0};
        }

    const int64_t groups = ((int64_t)g.R + RPW - 1) / RPW;
    const int64_t stride = (int64_t)gridDim.x * kGemvWaves;
    auto load = [&](int64_t grp, v4i_g (&m)[RPW][CPL]) {
#pragma unroll
        for (int r = 0; r < RPW; ++r) {
            int64_t row = grp * RPW + r;
            row = row < g.R ? row : g.R - 1;
            const uint8_t *p = mat + row * ld_b;
#pragma unroll
            for (int u = 0; u < CPL; ++u) {
                const int c = lane + 64 * u;
                m[r][u] = c < nch ? __builtin_nontemporal_load((const v4i_g *)(p + (int64_t)c * 16))
                                  : v4i_g{0, 0, 0, 0};
            }
        }
    };

    int64_t grp = (int64_t)blockIdx.x * kGemvWaves + wave;
    if (grp >= groups) return;
    v4i_g cur[RPW][CPL], nxt[RPW][CPL];
    load(grp, nxt);
    for (; grp < groups; grp += stride) {
#pragma unroll
        for (int r = 0; r < RPW; ++r)
#pragma unroll
            for (int u = 0; u < CPL; ++u) cur[r][u] = nxt[r][u];
        if (grp + stride < groups) load(grp + stride, nxt);
        acc_t v[RPW * NV];
#pragma unroll
        for (int r = 0; r < RPW; ++r)
#pragma unroll
            for (int j = 0; j < NV; ++j) {
                acc_t a = acc_t(0);
#pragma unroll
                for (int u = 0; u < CPL; ++u) a = D::dot(cur[r][u], x[j][u], a);
                v[r * NV + j] = a;
            }
        wave_reduce(v);
        store_group<T, E, NV, RPW>(g, ep, grp * RPW, v);
    }
}

// Largest staged vector block (bytes) a workgroup keeps in LDS.
constexpr int kGemvLdsMax = 64 * 1024;
constexpr int kLdsUnroll = 8;

template <InType T, EpiKind E, int NV, int RPW>
__global__ __launch_bounds__(kGemvThreads) void gemv_lds(const GemvArgs g, const EpiParams ep) {
    using D = Dot16<T>;
    using acc_t = typename D::acc_t;
    extern __shared__ __attribute__((aligned(16))) uint8_t sv[];
    constexpr int esz = (T == InType::I8) ? 1 : (T == InType::BF16 ? 2 : 4);
    const int64_t nch = ((int64_t)g.K * esz + 15) / 16;
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int64_t zb = blockIdx.y;  // batch element
    const uint8_t *vec = (const uint8_t *)g.vec + zb * g.bsv * esz;
    const int64_t vld_b = g.vld * esz;
    // Vectors beyond nvec (up to NV) read as zeros; when the block does not
    // fit in LDS the vectors are read from global memory (L2-resident).
    const bool staged = (int64_t)NV * nch * 16 <= kGemvLdsMax;
    if (staged) {
        for (int64_t c = tid; c < NV * nch; c += kGemvThreads) {
            const int64_t j = c / nch, ch = c % nch;
            *(v4i_g *)(sv + c * 16) = j < g.nvec ? *(const v4i_g *)(vec + j * vld_b + ch * 16)
                                                 : v4i_g{0, 0, 0, 0};
        }
        __syncthreads();
    }
    auto xchunk = [&](int j, int64_t ch) -> v4i_g {
        if (staged) return *(const v4i_g *)(sv + (j * nch + ch) * 16);
        return j < g.nvec ? *(const v4i_g *)(vec + j * vld_b + ch * 16) : v4i_g{0, 0, 0, 0};
    };
    const uint8_t *mat = (const uint8_t *)g.mat + zb * g.bsm * esz;
    const int64_t ld_b = g.ld * esz;
    const int64_t groups = ((int64_t)g.R + RPW - 1) / RPW;
    const int64_t stride = (int64_t)gridDim.x * kGemvWaves;
    for (int64_t grp = (int64_t)blockIdx.x * kGemvWaves + wave; grp < groups; grp += stride) {
        const int64_t r0 = grp * RPW;
        const uint8_t *rowp[RPW];
#pragma unroll
        for (int r = 0; r < RPW; ++r) rowp[r] = mat + (r0 + r < g.R ? r0 + r : g.R - 1) * ld_b;
        acc_t acc[RPW][NV];
#pragma unroll
        for (int r = 0; r < RPW; ++r)
#pragma unroll
            for (int j = 0; j < NV; ++j) acc[r][j] = acc_t(0);
        int64_t ch = lane;
        for (; ch + 64 * (kLdsUnroll - 1) < nch; ch += 64 * kLdsUnroll) {
            v4i_g m[kLdsUnroll][RPW];
#pragma unroll
            for (int u = 0; u < kLdsUnroll; ++u)
#pragma unroll
                for (int r = 0; r < RPW; ++r)
                    m[u][r] = __builtin_nontemporal_load((const v4i_g *)(rowp[r] + (ch + 64 * u) * 16));
#pragma unroll
            for (int u = 0; u < kLdsUnroll; ++u)
#pragma unroll
                for (int j = 0; j < NV; ++j) {
                    const v4i_g xv = xchunk(j, ch + 64 * u);
#pragma unroll
                    for (int r = 0; r < RPW; ++r) acc[r][j] = D::dot(m[u][r], xv, acc[r][j]);
                }
        }
        for (; ch < nch; ch += 64) {
#pragma unroll
            for (int j = 0; j < NV; ++j) {
                const v4i_g xv = xchunk(j, ch);
#pragma unroll
                for (int r = 0; r < RPW; ++r)
                    acc[r][j] = D::dot(*(const v4i_g *)(rowp[r] + ch * 16), xv, acc[r][j]);
            }
        }
        acc_t v[RPW * NV];
#pragma unroll
        for (int r = 0; r < RPW; ++r)
#pragma unroll
            for (int j = 0; j < NV; ++j) v[r * NV + j] = acc[r][j];
        wave_reduce(v);
        store_group<T, E, NV, RPW>(g, ep, r0, v);
    }
}

// Long rows with one or two vectors: the workgroup takes one row at a time
// (rows blockIdx.x, + gridDim.x, ...), its 256 lanes reading 256*U
// consecutive 16-byte chunks per batch (thread t: chunks t + 256u), so each
// workgroup streams one contiguous 32..64 KiB window instead of four waves
// streaming four rows 8 KiB at a time (on a 16384^2 f32 matrix: 0.86 of HBM
// peak for this access pattern against 0.82 for a row per wave and 0.77 for
// two rows per wave, plain reads measured alone).  Batches run as one flat
// sequence over the workgroup's rows with the next batch's loads issued
// before the current one is multiplied; the last batch of a row is masked
// past the row's end.  At a row's end each wave reduces its lanes'
// partial sums, the four wave totals meet in LDS (two slots alternating by
// row, so one barrier per row suffices) and wave 0 adds them in wave order
// and stores.
template <InType T, EpiKind E, int NV, int U>
__global__ __launch_bounds__(kGemvThreads) void gemv_wgrow(const GemvArgs g, const EpiParams ep) {
    using D = Dot16<T>;
    using acc_t = typename D::acc_t;
    extern __shared__ __attribute__((aligned(16))) uint8_t sv[];
    constexpr int esz = (T == InType::I8) ? 1 : (T == InType::BF16 ? 2 : 4);
    const int64_t nch = ((int64_t)g.K * esz + 15) / 16;
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int64_t zb = blockIdx.y;  // batch element
    const uint8_t *vec = (const uint8_t *)g.vec + zb * g.bsv * esz;
    const int64_t vld_b = g.vld * esz;
    // The vectors are staged in LDS when they fit (else read from global
    // memory, L2-resident); the wave-total exchange follows them.
    const bool staged = (int64_t)NV * nch * 16 <= kGemvLdsMax;
    acc_t *comb = (acc_t *)(sv + (staged ? NV * nch * 16 : 0));
    if (staged) {
        for (int64_t c = tid; c < NV * nch; c += kGemvThreads) {
            const int64_t j = c / nch, ch = c % nch;
            *(v4i_g *)(sv + c * 16) = j < g.nvec ? *(const v4i_g *)(vec + j * vld_b + ch * 16)
                                                 : v4i_g{0, 0, 0, 0};
        }
    }
    __syncthreads();
    auto xchunk = [&](int j, int64_t ch) -> v4i_g {
        if (staged) return *(const v4i_g *)(sv + (j * nch + ch) * 16);
        return j < g.nvec ? *(const v4i_g *)(vec + j * vld_b + ch * 16) : v4i_g{0, 0, 0, 0};
    };
    const uint8_t *mat = (const uint8_t *)g.mat + zb * g.bsm * esz;
    const int64_t ld_b = g.ld * esz;
    constexpr int64_t kBatch = (int64_t)kGemvThreads * U;  // chunks per batch
    const int64_t nbr = (nch + kBatch - 1) / kBatch;       // batches per row
    int64_t irow = blockIdx.x, ib = 0;  // next batch to issue
    int64_t rrow = blockIdx.x, rb = 0;  // next batch to multiply
    int slot = 0;
    acc_t acc[NV];
    auto issue = [&](v4i_g (&m)[U]) {
        const uint8_t *rp = mat + irow * ld_b;
        const int64_t c0 = ib * kBatch + tid;
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const int64_t c = c0 + (int64_t)kGemvThreads * u;
            m[u] = c < nch ? __builtin_nontemporal_load((const v4i_g *)(rp + c * 16))
                           : v4i_g{0, 0, 0, 0};
        }
        if (++ib == nbr) {
            ib = 0;
            irow += gridDim.x;
        }
    };
    auto run = [&](const v4i_g (&m)[U]) {
        if (rb == 0) {
#pragma unroll
            for (int j = 0; j < NV; ++j) acc[j] = acc_t(0);
        }
        const int64_t c0 = rb * kBatch + tid;
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const int64_t c = c0 + (int64_t)kGemvThreads * u;
            if (c < nch) {
#pragma unroll
                for (int j = 0; j < NV; ++j) acc[j] = D::dot(m[u], xchunk(j, c), acc[j]);
            }
        }
        if (++rb < nbr) return;
        acc_t v[NV];
#pragma unroll
        for (int j = 0; j < NV; ++j) v[j] = acc[j];
        wave_reduce(v);
        constexpr int SH = 6 - log2c<NV>();
        if ((lane & ((1 << SH) - 1)) == 0)
            comb[(slot * kGemvWaves + wave) * NV + (lane >> SH)] = v[0];
        __syncthreads();
        if (wave == 0 && lane < NV) {
            acc_t s = comb[slot * kGemvWaves * NV + lane];
#pragma unroll
            for (int w = 1; w < kGemvWaves; ++w) s += comb[(slot * kGemvWaves + w) * NV + lane];
            if (lane < g.nvec) Store<E>::apply(ep, blockIdx.y, lane, (int)rrow, s);
        }
        slot ^= 1;
        rb = 0;
        rrow += gridDim.x;
    };
    v4i_g m0[U], m1[U];
    if (irow < g.R) issue(m0);
    while (rrow < g.R) {
        if (irow < g.R) issue(m1);
        run(m0);
        if (rrow >= g.R) break;
        if (irow < g.R) issue(m0);
        run(m1);
    }
}

// Persistent grid: enough workgroups to cover the row groups, at most
// `per_cu` per CU over all batch elements (grid y); every element gets at
// least one workgroup.
static dim3 gemv_grid(int64_t groups, int cus, int per_cu, int batch) {
    int64_t blocks = (groups + kGemvWaves - 1) / kGemvWaves;
    const int64_t nb = batch > 1 ? batch : 1;
    const int64_t cap = ((int64_t)(cus > 0 ? cus : 256) * per_cu + nb - 1) / nb;
    if (blocks > cap) blocks = cap;
    return dim3((unsigned)(blocks < 1 ? 1 : blocks), (unsigned)nb);
}

// Rows per wave iteration and workgroups per CU, from a graph-timed sweep over
// 1 KB..8 KB rows (i8, f32 and bf16, 4096..65536 rows, five rotating matrix
// copies so the Infinity Cache cannot serve them).  Rows of 4 KB or more want
// about 8 KB per wave iteration (2 rows of 4 KB, 1 of 8 KB) and 3 workgroups
// per CU: on a 58.7 MB i8 matrix that is 10.2 us against 11.4 us for 4 rows
// and up to 8 workgroups per CU, which keeps more bytes in flight but spends
// longer in each wave's reduction and store before its next loads.  Shorter
// rows keep 4 rows per iteration and up to 8 workgroups per CU.
template <int CPL>
constexpr int rows_per_wave() {
    return CPL >= 8 ? 1 : (CPL >= 4 ? 2 : 4);
}

template <int CPL>
constexpr int reg_per_cu() {
    return CPL >= 4 ? 3 : 8;
}

// GEMMKIT_HIP_GEMV_SHAPE="rows,wgs" overrides the register GEMV's launch shape:
// rows per wave iteration (1, 2 or 4; one vector only) and workgroups per CU.
// A tuning switch for the launch-shape sweep: i8 results do not change; float
// sums may round differently with the rows per iteration (the butterfly's
// tree depends on the number of values it reduces).
struct GemvShape {
    int rpw = 0, per_cu = 0;
};
static GemvShape gemv_shape_env() {
    GemvShape sh;
    const char *e = getenv("GEMMKIT_HIP_GEMV_SHAPE");
    if (e && sscanf(e, "%d,%d", &sh.rpw, &sh.per_cu) != 2) sh = GemvShape{};
    return sh;
}

template <InType T, EpiKind E, int NV, int CPL, int RPW>
static hipError_t go_reg_rpw(const GemvArgs &g, const EpiParams &ep, int per_cu,
                             hipStream_t stream) {
    const int64_t groups = ((int64_t)g.R + RPW - 1) / RPW;
    hipLaunchKernelGGL((gemv_reg<T, E, NV, CPL, RPW>), gemv_grid(groups, g.cus, per_cu, g.batch),
                       dim3(kGemvThreads), 0, stream, g, ep);
    return hipGetLastError();
}

template <InType T, EpiKind E, int NV, int CPL>
static hipError_t go_reg(const GemvArgs &g, const EpiParams &ep, hipStream_t stream) {
    const GemvShape sh = gemv_shape_env();
    const int per_cu = sh.per_cu > 0 ? sh.per_cu : reg_per_cu<CPL>();
    if constexpr (NV == 1) {
        if (sh.rpw == 1) return go_reg_rpw<T, E, NV, CPL, 1>(g, ep, per_cu, stream);
        if (sh.rpw == 2) return go_reg_rpw<T, E, NV, CPL, 2>(g, ep, per_cu, stream);
        if (sh.rpw == 4) return go_reg_rpw<T, E, NV, CPL, 4>(g, ep, per_cu, stream);
    }
    return go_reg_rpw<T, E, NV, CPL, rows_per_wave<CPL>()>(g, ep, per_cu, stream);
}

// Workgroup-per-row launch: as many workgroups per CU as LDS holds, at most
// 3 (2 and 3 measure alike; 4 or more contend in HBM), or the switch's count.
template <InType T, EpiKind E, int NV, int U>
static hipError_t go_wgrow(const GemvArgs &g, const EpiParams &ep, hipStream_t stream) {
    constexpr int esz = (T == InType::I8) ? 1 : (T == InType::BF16 ? 2 : 4);
    const int64_t vbytes = (int64_t)NV * (((int64_t)g.K * esz + 15) / 16) * 16;
    const size_t shm = (vbytes <= kGemvLdsMax ? (size_t)vbytes : 0) + 2 * kGemvWaves * NV * 4;
    const int fit = (int)(160 * 1024 / shm);
    int per_cu = fit < 3 ? (fit > 1 ? fit : 1) : 3;
    const GemvShape sh = gemv_shape_env();
    if (sh.per_cu > 0) per_cu = sh.per_cu < fit ? sh.per_cu : (fit > 1 ? fit : 1);
    const int64_t nb = g.batch > 1 ? g.batch : 1;
    int64_t blocks = ((int64_t)(g.cus > 0 ? g.cus : 256) * per_cu + nb - 1) / nb;
    if (blocks > g.R) blocks = g.R;
    hipLaunchKernelGGL((gemv_wgrow<T, E, NV, U>), dim3((unsigned)blocks, (unsigned)nb),
                       dim3(kGemvThreads), shm, stream, g, ep);
    return hipGetLastError();
}

template <InType T, EpiKind E, int NV>
static hipError_t go_lds(const GemvArgs &g, const EpiParams &ep, hipStream_t stream) {
    // one or two vectors (bf16: one, for registers): a workgroup per row
    if constexpr (T == InType::BF16 ? NV == 1 : NV <= 2) return go_wgrow<T, E, NV, 8>(g, ep, stream);
    constexpr int RPW = 1;
    constexpr int esz = (T == InType::I8) ? 1 : (T == InType::BF16 ? 2 : 4);
    const int64_t vbytes = (int64_t)NV * (((int64_t)g.K * esz + 15) / 16) * 16;
    const size_t shm = vbytes <= kGemvLdsMax ? (size_t)vbytes : 0;
    const int64_t groups = ((int64_t)g.R + RPW - 1) / RPW;
    hipLaunchKernelGGL((gemv_lds<T, E, NV, RPW>), gemv_grid(groups, g.cus, 2, g.batch),
                       dim3(kGemvThreads), shm, stream, g, ep);
    return hipGetLastError();
}

// Register-resident vectors while NV x CPL chunks per lane stay within the
// register budget (bf16 needs extra registers to widen its operands).
template <InType T, int NV, int CPL>
constexpr bool reg_fits() {
    return NV * CPL <= (T == InType::BF16 ? 16 : 32);
}

template <InType T, EpiKind E, int NV>
static hipError_t go_nv(const GemvArgs &g, const EpiParams &ep, hipStream_t stream) {
    constexpr int esz = (T == InType::I8) ? 1 : (T == InType::BF16 ? 2 : 4);
    const int64_t nch = ((int64_t)g.K * esz + 15) / 16;
    if (nch <= 64) return go_reg<T, E, NV, 1>(g, ep, stream);
    if (nch <= 128) return go_reg<T, E, NV, 2>(g, ep, stream);
    if constexpr (reg_fits<T, NV, 4>())
        if (nch <= 256) return go_reg<T, E, NV, 4>(g, ep, stream);
    if constexpr (reg_fits<T, NV, 8>())
        if (nch <= 512) return go_reg<T, E, NV, 8>(g, ep, stream);
    return go_lds<T, E, NV>(g, ep, stream);
}

template <InType T, EpiKind E>
static hipError_t gemv_nv(const GemvArgs &g, const EpiParams &ep, hipStream_t stream) {
    if (g.nvec <= 1) return go_nv<T, E, 1>(g, ep, stream);
    if (g.nvec <= 2) return go_nv<T, E, 2>(g, ep, stream);
    if (g.nvec <= 4) return go_nv<T, E, 4>(g, ep, stream);
    return go_nv<T, E, 8>(g, ep, stream);
}

// ---------------------------------------------------------- unit row stride

// A 16-byte load at any address (rows of a strided matrix need not be aligned).
typedef int v4i_any __attribute__((ext_vector_type(4), aligned(1)));

// x[k] of a staged chunk, widened, and the multiply of one matrix chunk row.
template <InType T>
struct ColStep;

template <>
struct ColStep<InType::F32> {
    static constexpr int EPC = 4;
    using acc_t = float;
    using elem_t = uint32_t;
    // m[e]: EPC consecutive matrix rows at k = e of the chunk; x: the chunk's EPC
    // vector elements.  Ascending k, one FMA each: Dot16's order.
    __device__ __forceinline__ static void mul(const v4i_g (&m)[4], v4i_g x, acc_t (&acc)[4]) {
        const v4f_g xf = __builtin_bit_cast(v4f_g, x);
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            const v4f_g mf = __builtin_bit_cast(v4f_g, m[e]);
#pragma unroll
            for (int r = 0; r < 4; ++r) acc[r] = __builtin_fmaf(mf[r], xf[e], acc[r]);
        }
    }
};

template <>
struct ColStep<InType::BF16> {
    static constexpr int EPC = 8;
    using acc_t = float;
    using elem_t = uint16_t;
    __device__ __forceinline__ static float at(const v4i_g &v, int i) {
        const uint32_t w = (uint32_t)v[i >> 1];
        return __uint_as_float((i & 1) ? (w & 0xFFFF0000u) : (w << 16));
    }
    __device__ __forceinline__ static void mul(const v4i_g (&m)[8], v4i_g x, acc_t (&acc)[8]) {
#pragma unroll
        for (int e = 0; e < 8; ++e) {
            const float xe = at(x, e);
#pragma unroll
            for (int r = 0; r < 8; ++r) acc[r] = __builtin_fmaf(at(m[e], r), xe, acc[r]);
        }
    }
};

template <>
struct ColStep<InType::I8> {
    static constexpr int EPC = 16;
    using acc_t = int32_t;
    using elem_t = uint8_t;
    // 4 x 4 byte transposes bring four k of one matrix row into a word.
    __device__ __forceinline__ static void mul(const v4i_g (&m)[16], v4i_g x, acc_t (&acc)[16]) {
#pragma unroll
        for (int p = 0; p < 4; ++p)
#pragma unroll
            for (int c = 0; c < 4; ++c) {
                const uint32_t i0 = m[4 * p][c], i1 = m[4 * p + 1][c];
                const uint32_t i2 = m[4 * p + 2][c], i3 = m[4 * p + 3][c];
                const uint32_t t0 = __builtin_amdgcn_perm(i1, i0, 0x05010400u);
                const uint32_t t1 = __builtin_amdgcn_perm(i1, i0, 0x07030602u);
                const uint32_t u0 = __builtin_amdgcn_perm(i3, i2, 0x05010400u);
                const uint32_t u1 = __builtin_amdgcn_perm(i3, i2, 0x07030602u);
                const uint32_t w[4] = {__builtin_amdgcn_perm(u0, t0, 0x05040100u),
                                       __builtin_amdgcn_perm(u0, t0, 0x07060302u),
                                       __builtin_amdgcn_perm(u1, t1, 0x05040100u),
                                       __builtin_amdgcn_perm(u1, t1, 0x07060302u)};
#pragma unroll
                for (int r = 0; r < 4; ++r)
                    acc[4 * c + r] = __builtin_amdgcn_sdot4((int)w[r], x[p], acc[4 * c + r], false);
            }
    }
};

// out[j, r] with a matrix of unit row stride (element (r, p) at r + p*mks, any
// mks and alignment) and k-contiguous vectors (any alignment).  Bound by
// streaming the matrix once: bf16 1 x 4096 x 11008 17.1 us (5.3 TB/s with three
// copies in turn, 20.6 from HBM alone) against 55 with the matrix packed first,
// f32 30.6 against 96, i8 12.0 against 44.  A lane loads 16 bytes of EPC consecutive matrix
// rows at one k; eight lanes side by side cover a run of 128 bytes (64-byte runs
// measured slower), and 64 slots split K by 16-byte chunks: slot s takes chunks
// s, s + 64, ... -- the chunks lane s of a row kernel multiplies, in the same
// order, so each slot's partial sum is that lane's.  The slots are then added in
// the row kernels' butterfly order (32, 16, 8, 4, 2, 1 apart) and, where those
// run 256 lanes per row (NCL = 4 chunk classes per slot), the four groups in
// wave order: results equal the row kernels' on a packed copy bit for bit.
// Slot s of a wave of 8 slots is s*8 + w, so the first three butterfly steps stay
// inside the wave and the eight waves w of a column group need one exchange: through
// LDS when one workgroup holds all eight, or (SPLIT, too few columns for the
// CUs) through global partial sums, a wave per workgroup and class group, that
// cols_combine adds.
constexpr int kColLanes = 8;

template <InType T>
__device__ __forceinline__ typename ColStep<T>::acc_t cols_tree(
    typename ColStep<T>::acc_t (&v)[kColLanes]) {
#pragma unroll
    for (int off = kColLanes / 2; off >= 1; off >>= 1)
#pragma unroll
        for (int w = 0; w < off; ++w) v[w] += v[w + off];
    return v[0];
}

template <InType T, EpiKind E, int NV, int NCL, int UNR, bool SPLIT>
__global__ __launch_bounds__(SPLIT ? 64 : kColLanes * 64) void gemv_cols(const GemvArgs g,
                                                                       const EpiParams ep) {
    using St = ColStep<T>;
    using acc_t = typename St::acc_t;
    using elem_t = typename St::elem_t;
    constexpr int EPC = St::EPC, COLS = kColLanes * EPC;
    __shared__ acc_t part[SPLIT ? 1 : NCL * NV][SPLIT ? 1 : kColLanes][SPLIT ? 1 : COLS];
    const int tid = threadIdx.x, lane = tid & 63;
    const int64_t zb = blockIdx.y;
    const elem_t *mat = (const elem_t *)g.mat + zb * g.bsm;
    const elem_t *vec = (const elem_t *)g.vec + zb * g.bsv;
    // SPLIT: workgroup = (column group, class group, wave), waves fastest.
    const int64_t blk = SPLIT ? blockIdx.x / (NCL * kColLanes) : blockIdx.x;
    const int wave = SPLIT ? (int)(blockIdx.x % kColLanes)
                           : __builtin_amdgcn_readfirstlane(tid >> 6);
    const int q0 = SPLIT ? (int)(blockIdx.x / kColLanes) % NCL : 0;
    const int cl = lane % kColLanes, slot = (lane / kColLanes) * kColLanes + wave;
    // The last column group's lanes start EPC rows before R at the latest (so
    // every load stays inside the matrix; the caller ensures R >= EPC); the
    // rows below their own range are another lane's to store.
    const int64_t rl = blk * COLS + cl * EPC;
    const int64_t r0 = rl + EPC <= g.R ? rl : g.R - EPC;
    constexpr int64_t STEP = 64 * NCL;
    const int64_t nfull = (int64_t)g.K / EPC;  // whole chunks (at least one: the caller's minimum K)

    auto load = [&](int64_t ch, v4i_g (&m)[EPC], v4i_g (&x)[NV]) {
        const elem_t *p = mat + r0 + ch * EPC * g.mks;
#pragma unroll
        for (int j = 0; j < NV; ++j)
            x[j] = *(const v4i_any *)(vec + (j < g.nvec ? j : 0) * g.vld + ch * EPC);
#pragma unroll
        for (int e = 0; e < EPC; ++e)
            m[e] = *(const v4i_any *)(p + e * g.mks);
    };
    for (int q = q0; q < (SPLIT ? q0 + 1 : NCL); ++q) {
        acc_t acc[NV][EPC] = {};
        int64_t ch = slot + 64 * q;
        // All loads of a batch are issued before any is used (the scheduler
        // would otherwise sink them to their uses to save registers); chunks
        // past the end load the last one again and are left out.
        for (int64_t c0 = 64 * q; c0 < nfull; c0 += STEP * UNR, ch += STEP * UNR) {
            v4i_g m[UNR][EPC], x[UNR][NV];
#pragma unroll
            for (int u = 0; u < UNR; ++u) {
                const int64_t c = ch + STEP * u;
                load(c < nfull ? c : nfull - 1, m[u], x[u]);
            }
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int u = 0; u < UNR; ++u)
                if (ch + STEP * u < nfull) {
#pragma unroll
                    for (int j = 0; j < NV; ++j) St::mul(m[u], x[u][j], acc[j]);
                }
        }
        if (nfull * EPC < g.K && nfull % STEP == slot + 64 * q) {  // the last chunk, zeros past K
            v4i_g m[EPC];
#pragma unroll
            for (int e = 0; e < EPC; ++e) {
                m[e] = v4i_g{0, 0, 0, 0};
                if (nfull * EPC + e < g.K)
                    m[e] = *(const v4i_any *)(mat + r0 + (nfull * EPC + e) * g.mks);
            }
#pragma unroll
            for (int j = 0; j < NV; ++j) {
                const elem_t *p = vec + (j < g.nvec ? j : 0) * g.vld + nfull * EPC;
                elem_t v[EPC];
#pragma unroll
                for (int e = 0; e < EPC; ++e) v[e] = nfull * EPC + e < g.K ? p[e] : elem_t(0);
                v4i_g x;
                __builtin_memcpy(&x, v, 16);
                St::mul(m, x, acc[j]);
            }
        }
#pragma unroll
        for (int j = 0; j < NV; ++j)
#pragma unroll
            for (int r = 0; r < EPC; ++r) {
#pragma unroll
                for (int off = 32; off >= kColLanes; off >>= 1)
                    acc[j][r] += __shfl_xor(acc[j][r], off, 64);
                if (lane < kColLanes && r0 + r >= rl) {
                    if constexpr (SPLIT) {
                        if (j < g.nvec)
                            ((acc_t *)g.part)[(((zb * NCL + q) * g.nvec + j) * kColLanes + wave) *
                                                  g.R + r0 + r] = acc[j][r];
                    } else {
                        part[q * NV + j][wave][r0 + r - blk * COLS] = acc[j][r];
                    }
                }
            }
    }
    if constexpr (!SPLIT) {
        __syncthreads();
        for (int o = tid; o < NV * COLS; o += kColLanes * 64) {
            const int j = o / COLS, c = o % COLS;
            acc_t sum = acc_t(0);
#pragma unroll
            for (int q = 0; q < NCL; ++q) {
                acc_t v[kColLanes];
#pragma unroll
                for (int w = 0; w < kColLanes; ++w) v[w] = part[q * NV + j][w][c];
                sum = q == 0 ? cols_tree<T>(v) : sum + cols_tree<T>(v);
            }
            const int64_t r = blk * COLS + c;
            if (j < g.nvec && r < g.R) Store<E>::apply(ep, zb, j, (int)r, sum);
        }
    }
}

// Adds SPLIT partial sums [element][class group][vector][wave][row] in the
// order above, one output per thread.
template <InType T, EpiKind E, int NCL>
__global__ __launch_bounds__(64) void cols_combine(const GemvArgs g, const EpiParams ep) {
    using acc_t = typename ColStep<T>::acc_t;
    const int64_t r = (int64_t)blockIdx.x * 64 + threadIdx.x;
    const int j = blockIdx.y;
    const int64_t zb = blockIdx.z;
    if (r >= g.R) return;
    acc_t v[NCL][kColLanes];
#pragma unroll
    for (int q = 0; q < NCL; ++q)
#pragma unroll
        for (int w = 0; w < kColLanes; ++w)
            v[q][w] = ((const acc_t *)g.part)[(((zb * NCL + q) * g.nvec + j) * kColLanes + w) *
                                                  g.R + r];
    acc_t sum = cols_tree<T>(v[0]);
#pragma unroll
    for (int q = 1; q < NCL; ++q) sum = sum + cols_tree<T>(v[q]);
    Store<E>::apply(ep, zb, j, (int)r, sum);
}

template <InType T, EpiKind E, int NV, int NCL, int UNR>
static hipError_t go_cols(const GemvArgs &g, const EpiParams &ep, hipStream_t stream) {
    constexpr int COLS = kColLanes * ColStep<T>::EPC;
    const int64_t blocks = ((int64_t)g.R + COLS - 1) / COLS;
    if (g.part) {
        hipLaunchKernelGGL((gemv_cols<T, E, NV, NCL, UNR, true>),
                           dim3((unsigned)(blocks * NCL * kColLanes), (unsigned)g.batch), dim3(64),
                           0, stream, g, ep);
        hipLaunchKernelGGL((cols_combine<T, E, NCL>),
                           dim3((unsigned)((g.R + 63) / 64), (unsigned)g.nvec, (unsigned)g.batch),
                           dim3(64), 0, stream, g, ep);
    } else {
        hipLaunchKernelGGL((gemv_cols<T, E, NV, NCL, UNR, false>),
                           dim3((unsigned)blocks, (unsigned)g.batch), dim3(kColLanes * 64), 0,
                           stream, g, ep);
    }
    return hipGetLastError();
}

// The summing order of the row kernel go_nv picks for the same shape: 256
// lanes per row where that is gemv_wgrow, 64 otherwise (i8 sums have no order).
static bool cols_wgrow(InType in, int nvec, int64_t K) {
    const int64_t nch = (K * (int64_t)in_size(in) + 15) / 16;
    return nch > 512 && (in == InType::F32 ? nvec <= 2 : (in == InType::BF16 && nvec == 1));
}

// Chunks per slot in one batch of loads: 16 matrix loads (64 registers) of a
// lane in flight, i8 32 (a chunk of i8 is 16 loads), half with more vectors.
constexpr int cols_unroll(InType in, int nv) {
    return (in == InType::F32 ? 4 : 2) / (nv <= 2 ? 1 : 2);
}

template <InType T, EpiKind E, int NV>
static hipError_t cols_nv(const GemvArgs &g, const EpiParams &ep, hipStream_t stream) {
    constexpr int UNR = cols_unroll(T, NV);
    if constexpr (T == InType::F32 ? NV <= 2 : (T == InType::BF16 && NV == 1)) {
        if (cols_wgrow(T, g.nvec, g.K)) return go_cols<T, E, NV, 4, UNR>(g, ep, stream);
    }
    return go_cols<T, E, NV, 1, UNR>(g, ep, stream);
}

template <InType T, EpiKind E>
static hipError_t gemv_cols_nv(const GemvArgs &g, const EpiParams &ep, hipStream_t stream) {
    if (g.nvec <= 1) return cols_nv<T, E, 1>(g, ep, stream);
    if (g.nvec <= 2) return cols_nv<T, E, 2>(g, ep, stream);
    return cols_nv<T, E, 4>(g, ep, stream);
}

int64_t gemv_cols_rounds(InType in, int64_t K, int nvec) {
    const int64_t epc = 16 / (int64_t)in_size(in);
    return K / epc / (64 * (cols_wgrow(in, nvec, K) ? 4 : 1) * cols_unroll(in, nvec));
}

// K is split over workgroups when a slot has more than one batch of loads and
// the column groups are few for the CUs: 1 x 4096 x 4096 (64 groups) 10.0 against
// 12.4 us in one workgroup per group, x 1024 (16 groups) 8.1 against 11.5, i8
// x 11008 (86) 14.7 against 17.9; bf16 x 11008 (172) 18.3 against 17.1 and 1 x
// 1024 x 16384 (256, one batch) 10.4 against 8.5 stay whole.  With four class
// groups there are four times as many waves to spread, and it pays up to two
// groups per CU (f32 1 x 4096 x 11008, 344 groups: 30.6 against 33.1 us).
int64_t gemv_cols_part_bytes(InType in, int64_t R, int64_t K, int nvec, int64_t batch, int cus) {
    const int64_t epc = 16 / (int64_t)in_size(in), cols = kColLanes * epc;
    const int ncl = cols_wgrow(in, nvec, K) ? 4 : 1;
    if (K / epc <= 64 * cols_unroll(in, nvec)) return 0;
    if ((R + cols - 1) / cols * batch > (int64_t)(cus > 0 ? cus : 256) * ncl / 2) return 0;
    return ncl * batch * nvec * kColLanes * R * 4;
}

hipError_t launch_gemv_cols(InType in, const GemvArgs &g, const EpiParams &ep,
                            hipStream_t stream) {
    if (g.nvec < 1 || g.nvec > kGemvColsMaxVec || g.R < 16 / (int)in_size(in) || g.ld != 1 || g.batch < 1 ||
        g.batch > kMaxGridZ)
        return hipErrorInvalidValue;
    switch (in) {
    case InType::I8:
        if (ep.kind == EpiKind::I32) return gemv_cols_nv<InType::I8, EpiKind::I32>(g, ep, stream);
        if (ep.kind == EpiKind::Q8) return gemv_cols_nv<InType::I8, EpiKind::Q8>(g, ep, stream);
        break;
    case InType::F32:
        if (ep.kind == EpiKind::F32) return gemv_cols_nv<InType::F32, EpiKind::F32>(g, ep, stream);
        break;
    case InType::BF16:
        if (ep.kind == EpiKind::F32) return gemv_cols_nv<InType::BF16, EpiKind::F32>(g, ep, stream);
        if (ep.kind == EpiKind::BF16)
            return gemv_cols_nv<InType::BF16, EpiKind::BF16>(g, ep, stream);
        break;
    }
    return hipErrorInvalidValue;
}

hipError_t launch_gemv(InType in, const GemvArgs &g, const EpiParams &ep, hipStream_t stream) {
    // Row addresses are formed in 64 bits (any non-negative row stride); the
    // host packs a matrix with a negative one.
    if (g.nvec < 1 || g.nvec > 8 || g.R < 1 || g.ld < 0 || g.batch < 1 || g.batch > kMaxGridZ)
        return hipErrorInvalidValue;
    switch (in) {
    case InType::I8:
        if (ep.kind == EpiKind::I32) return gemv_nv<InType::I8, EpiKind::I32>(g, ep, stream);
        if (ep.kind == EpiKind::Q8) return gemv_nv<InType::I8, EpiKind::Q8>(g, ep, stream);
        break;
    case InType::F32:
        if (ep.kind == EpiKind::F32) return gemv_nv<InType::F32, EpiKind::F32>(g, ep, stream);
        break;
    case InType::BF16:
        if (ep.kind == EpiKind::F32) return gemv_nv<InType::BF16, EpiKind::F32>(g, ep, stream);
        if (ep.kind == EpiKind::BF16) return gemv_nv<InType::BF16, EpiKind::BF16>(g, ep, stream);
        break;
    }
    return hipErrorInvalidValue;
}

}  // namespace gk
