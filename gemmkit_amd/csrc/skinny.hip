// skinny.hip -- matrix-core kernel for skinny products: 1..16 short-side rows
// (decode-shaped GEMV / small-batch linear layers), bound by streaming the
// long operand from HBM once.
//
// Serves the same route as gemv.hip (gemmkit's gemv, src/special/gemv.rs:101-600,
// and the i8 skinny shapes, src/dispatch/int.rs:165-168), for short sides up to
// 16: out[j, r] = epi( sum_p mat[r, p] * vec[j, p] ), r < R, j < nvec.
//
// Layout on the matrix cores: v_mfma_*_16x16x(64 i8 | 32 bf16 | 4x4 f32) with
// the (zero-padded) vectors as the instruction's 16 columns.  A load
// instruction reads 8 matrix rows x 128 contiguous bytes (a 128-byte k step):
// lane l (i = l%16, g = l/16) takes row i/2 of the 8, chunk c = 2g + i%2.  As
// MFMA operand, lane l is instruction row i with k group g, so row i pairs
// chunk 2g + i%2 of its matrix row with whatever chunk the vector operand
// holds for group g.  Two MFMAs per load, one with vector chunks 2g (h = 0)
// and one with 2g + 1 (h = 1), make the products of the even rows exact in
// the first and of the odd rows in the second; the other halves are ignored.
// Result (16x16 accumulator: register q of lane l is instruction row
// 4*(l/16) + q, vector l%16): matrix row 2*(l/16) + e of the block is
// acc_h0[2e] + acc_h1[2e+1], a per-lane add.  The vectors are staged once per
// workgroup in LDS (row stride padded so the 16 lanes of an LDS cycle hit
// distinct banks); the matrix goes global -> VGPRs through a buffer resource
// (rows past R and bytes past K read as zeros).
//
// Work item: BLK 8-row blocks (32 rows, or 8 when there are too few rows to
// give every CU an item) x all of K.  The 4 waves of a workgroup split K into
// 4 contiguous ranges; each keeps 4 k steps x BLK blocks of loads in flight
// behind its MFMAs, and the four partial sums are added through LDS, in wave
// order, before the epilogue.
// The vectors may have any strides: k-contiguous, 16-byte aligned rows are
// staged as 16-byte chunks, anything else element by element (so a strided
// activation needs no separate pack launch).
#include <stdio.h>
#include <stdlib.h>

#include <type_traits>

#include "epilogue.h"

namespace gk {

typedef int v4i_s __attribute__((ext_vector_type(4)));
typedef float v4f_s __attribute__((ext_vector_type(4)));
typedef __bf16 v8bf_s __attribute__((ext_vector_type(8)));

template <InType T>
struct Mma16;

template <>
struct Mma16<InType::I8> {
    using acc_t = v4i_s;
    using val_t = int32_t;
    __device__ __forceinline__ static acc_t step(v4i_s a, v4i_s b, acc_t c) {
        return __builtin_amdgcn_mfma_i32_16x16x64_i8(a, b, c, 0, 0, 0);
    }
};

template <>
struct Mma16<InType::BF16> {
    using acc_t = v4f_s;
    using val_t = float;
    __device__ __forceinline__ static acc_t step(v4i_s a, v4i_s b, acc_t c) {
        return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(v8bf_s, a),
                                                       __builtin_bit_cast(v8bf_s, b), c, 0, 0, 0);
    }
};

template <>
struct Mma16<InType::F32> {
    using acc_t = v4f_s;
    using val_t = float;
    __device__ __forceinline__ static acc_t step(v4i_s a, v4i_s b, acc_t c) {
        v4f_s af = __builtin_bit_cast(v4f_s, a), bf = __builtin_bit_cast(v4f_s, b);
        c = __builtin_amdgcn_mfma_f32_16x16x4f32(af[0], bf[0], c, 0, 0, 0);
        c = __builtin_amdgcn_mfma_f32_16x16x4f32(af[1], bf[1], c, 0, 0, 0);
        c = __builtin_amdgcn_mfma_f32_16x16x4f32(af[2], bf[2], c, 0, 0, 0);
        c = __builtin_amdgcn_mfma_f32_16x16x4f32(af[3], bf[3], c, 0, 0, 0);
        return c;
    }
};

constexpr int kSkThreads = 256;
constexpr int kSkWaves = 4;
constexpr int kSkBlocks = 4;               // 8-row blocks per work item (at most)
constexpr int kSkStep = 128;               // k bytes per step (one load per block)
constexpr int kSkPF = 4;                   // k steps per load batch
constexpr int kSkCombine = kSkWaves * kSkBlocks * 2 * 64 * 4;  // partial-sum exchange bytes
constexpr uint32_t kSkOut = 0x80000000u;   // out-of-range buffer offset (reads zeros)
constexpr int kSkRsrcWord3 = 0x00020000;   // raw buffer, 32-bit data format

// LDS row stride of a staged vector: K bytes rounded up to 256, plus 16, so
// the 16 vectors read in one LDS cycle start in distinct 16-byte bank groups.
__host__ __device__ constexpr int64_t skinny_xstride(int64_t kbytes) {
    return (kbytes + 255) / 256 * 256 + 16;
}

// A vector chunk: the default cache policy (every workgroup reads the vectors).
__device__ __forceinline__ v4i_s load16v(const uint8_t *base, uint32_t num, uint32_t off) {
    __amdgpu_buffer_rsrc_t r =
        __builtin_amdgcn_make_buffer_rsrc((void *)base, (short)0, (int)num, kSkRsrcWord3);
    return __builtin_bit_cast(v4i_s, __builtin_amdgcn_raw_buffer_load_b128(r, off, 0, 0));
}

__device__ __forceinline__ v4i_s load16(const uint8_t *base, uint32_t num, uint32_t off) {
    __amdgpu_buffer_rsrc_t r =
        __builtin_amdgcn_make_buffer_rsrc((void *)base, (short)0, (int)num, kSkRsrcWord3);
    // Cache policy 2 = nontemporal: the matrix is read once (12.6 against
    // 13.0 us with the default policy on the 14336x4096 i8 weight, 8 vectors).
    return __builtin_bit_cast(v4i_s, __builtin_amdgcn_raw_buffer_load_b128(r, off, 0, 2));
}

template <InType T, EpiKind E, int BLK>
__global__ __launch_bounds__(kSkThreads) void skinny_mfma(const GemvArgs g, const EpiParams ep) {
    constexpr int kSkRows = 8 * BLK;  // matrix rows per work item
    using Mm = Mma16<T>;
    using acc_t = typename Mm::acc_t;
    using val_t = typename Mm::val_t;
    constexpr int esz = (T == InType::I8) ? 1 : (T == InType::BF16 ? 2 : 4);
    extern __shared__ __attribute__((aligned(16))) uint8_t sh[];

    // Row bytes rounded up to whole 16-byte chunks: a K*esz that is not a
    // multiple of 16 only arrives through the pack, which zero-fills both
    // operands' rows up to the next 16 bytes.
    const int64_t kb = ((int64_t)g.K * esz + 15) / 16 * 16;
    const int nk = (int)((kb + kSkStep - 1) / kSkStep);
    const int64_t xs = skinny_xstride(kb);
    const int nvec = g.nvec;
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);

    const int li = lane & 15, lg = lane >> 4;
    const int chunk = 2 * lg + (li & 1);      // this lane's 16-byte chunk of a k step
    const bool lvec = li < nvec;
    const int64_t xaddr = (int64_t)(lvec ? li : 0) * xs + 32 * lg;  // + 16*h for MFMA h
    const int kseg = (nk + kSkWaves - 1) / kSkWaves;
    const int ks0 = wave * kseg, ks1 = ks0 + kseg < nk ? ks0 + kseg : nk;

    // This wave's load batches, in order: for each of the workgroup's items
    // (blockIdx.x, + gridDim.x, ...), nbw batches of kSkPF k steps of its K
    // range (at least one, all out of range when the range is empty, so every
    // wave takes part in every item's exchange).  Two register buffers
    // alternate: batch t+1 is in flight while batch t is multiplied, across
    // item boundaries too.  (Issuing batch 1 before the vector staging as
    // well measured slower: 14.3 against 12.6 us on the 14336x4096 i8
    // weight with 8 vectors.)
    const int64_t zb = blockIdx.y;  // batch element
    const uint8_t *mat = (const uint8_t *)g.mat + zb * g.bsm * esz;
    const int64_t ld_b = g.ld * esz;
    // (64-bit: R may be up to 2^31 - 1; every item's first row is below R)
    const int items = (int)(((int64_t)g.R + kSkRows - 1) / kSkRows);
    const int my_items = (int)blockIdx.x < items ? (items - 1 - (int)blockIdx.x) / (int)gridDim.x + 1 : 0;
    const int nbw = ks1 > ks0 ? (ks1 - ks0 + kSkPF - 1) / kSkPF : 1;
    const int total = my_items * nbw;
    uint32_t off[BLK];
#pragma unroll
    for (int b = 0; b < BLK; ++b) off[b] = (uint32_t)((8 * b + (li >> 1)) * ld_b + 16 * chunk);
    auto issue = [&](int t, v4i_s (&m)[kSkPF][BLK]) {
        const int r0 = ((int)blockIdx.x + (t / nbw) * (int)gridDim.x) * kSkRows;
        const int s0 = ks0 + (t % nbw) * kSkPF;
        const uint8_t *base = mat + (int64_t)r0 * ld_b;
        // Extent of the item's valid rows (rows may overlap: ld_b < kb is a
        // legal view); rows past R read zeros when they start past it and
        // otherwise produce outputs that are never stored.
        const bool live = t < total;  // batch 0 is issued even for a workgroup without items
        const int nrows = g.R - r0 < kSkRows ? g.R - r0 : kSkRows;
        const uint32_t num = live ? (uint32_t)((nrows - 1) * ld_b + kb) : 0u;
#pragma unroll
        for (int p = 0; p < kSkPF; ++p) {
            const int s = s0 + p;
            const bool in = live && s < ks1 && (int64_t)s * kSkStep + 16 * chunk < kb;
            // Out-of-range lanes get bit 31 set, past any resource size here
            // (an item spans at most 32 rows of at most 8 MiB, both for the
            // matrix's row stride and its row, so num and every in-range
            // offset stay below 2^31), without a select: every load is
            // issued on every path, so the wait counts after a batch are
            // exact.
            const uint32_t oor = (uint32_t)!in << 31;
#pragma unroll
            for (int b = 0; b < BLK; ++b)
                m[p][b] = load16(base, num, (off[b] + (uint32_t)s * kSkStep) | oor);
        }
    };
    v4i_s buf0[kSkPF][BLK], buf1[kSkPF][BLK];

    // Stage the vectors: nvec rows of kb bytes (zeros past K), 8 chunks or
    // elements per thread in flight at a time (one L2 round trip for up to
    // 32 KiB).
    const uint8_t *vec = (const uint8_t *)g.vec + zb * g.bsv * esz;
    const int64_t vld_b = g.vld * esz;
    if (g.vks == 1 && g.K * esz % 16 == 0 && vld_b % 16 == 0 && (uintptr_t)vec % 16 == 0) {
        // Chunk p of every vector (no index division), 8 loads in flight.
        // The first pass (chunk tid of vectors 0-7) is issued before the
        // matrix's batch 0 in straight-line code, so its LDS writes wait for
        // the vector loads only, not for batch 0 from HBM (8 vectors on the
        // 14336x4096 i8 weight: 11.95-11.98 against 12.54-12.59 us with
        // batch 0 first and a 64-bit index division per chunk).
        const int64_t cpr = kb / 16;
        // (A negative vector stride, legal on the unchecked tier, takes the
        // 64-bit pointer path: the buffer offsets below are unsigned.)
        if (vld_b >= 0 && (int64_t)(nvec - 1) * vld_b + kb <= 0x7FFFFFF0ll) {
            const uint32_t vnum = (uint32_t)((int64_t)(nvec - 1) * vld_b + kb);
            v4i_s tmp[8];
#pragma unroll
            for (int u = 0; u < 8; ++u)
                tmp[u] = load16v(vec, vnum, (tid < cpr && u < nvec)
                                                ? (uint32_t)(u * vld_b + (int64_t)tid * 16)
                                                : kSkOut);
            issue(0, buf0);
#pragma unroll
            for (int u = 0; u < 8; ++u)
                if (tid < cpr && u < nvec) *(v4i_s *)(sh + (int64_t)u * xs + (int64_t)tid * 16) = tmp[u];
        } else {
            issue(0, buf0);
            for (int j = 0; j < 8 && j < nvec; ++j)
                if (tid < cpr)
                    *(v4i_s *)(sh + (int64_t)j * xs + (int64_t)tid * 16) =
                        *(const v4i_s *)(vec + (int64_t)j * vld_b + (int64_t)tid * 16);
        }
        for (int64_t p = tid; p < cpr; p += kSkThreads) {
            for (int j0 = p == tid ? 8 : 0; j0 < nvec; j0 += 8) {
                v4i_s tmp[8];
#pragma unroll
                for (int u = 0; u < 8; ++u)
                    tmp[u] = j0 + u < nvec ? *(const v4i_s *)(vec + (int64_t)(j0 + u) * vld_b + p * 16)
                                           : v4i_s{0, 0, 0, 0};
#pragma unroll
                for (int u = 0; u < 8; ++u)
                    if (j0 + u < nvec) *(v4i_s *)(sh + (int64_t)(j0 + u) * xs + p * 16) = tmp[u];
            }
        }
    } else if (g.vld == 1 && g.vks >= nvec && (uintptr_t)vec % 4 == 0 &&
               (int64_t)(g.K - 1) * g.vks + nvec <= 0xFFFFFFFFll) {
        issue(0, buf0);
        // Column-major vectors (element (j, p) at p*vks + j): the span they
        // cover is read as aligned 4-byte words, 8 per thread in flight, and
        // each element is scattered to its vector's row.  A word never
        // straddles a page, so the bytes a last partial word reads past the
        // span are mapped; they are discarded.
        using elem_t = typename std::conditional<esz == 1, uint8_t,
                         typename std::conditional<esz == 2, uint16_t, uint32_t>::type>::type;
        constexpr int EPW = 4 / esz;  // elements per word
        const uint32_t vks = (uint32_t)g.vks;
        // idx / vks as a multiply-high (Granlund-Montgomery, exact for every
        // 32-bit idx): l = ceil(log2 vks), magic = 2^32 (2^l - vks) / vks + 1.
        const int dl = 32 - __builtin_clz(vks - 1);
        const uint32_t magic = (uint32_t)(((1ull << 32) * ((1ull << dl) - vks)) / vks + 1);
        const int64_t span = ((int64_t)(g.K - 1) * vks + nvec) * esz;
        const int64_t nw = (span + 3) / 4;
        const uint32_t *vw = (const uint32_t *)vec;
        for (int64_t w0 = tid; w0 < nw; w0 += kSkThreads * 8) {
            uint32_t tmp[8];
#pragma unroll
            for (int u = 0; u < 8; ++u) {
                const int64_t w = w0 + (int64_t)u * kSkThreads;
                tmp[u] = w < nw ? vw[w] : 0u;
            }
#pragma unroll
            for (int u = 0; u < 8; ++u) {
                const int64_t w = w0 + (int64_t)u * kSkThreads;
#pragma unroll
                for (int e = 0; e < EPW; ++e) {
                    const uint32_t idx = (uint32_t)(w * EPW + e);
                    const uint32_t hi = __umulhi(magic, idx);
                    const uint32_t p = (hi + ((idx - hi) >> 1)) >> (dl - 1), j = idx - p * vks;
                    if (w < nw && j < (uint32_t)nvec && p < (uint32_t)g.K)
                        *(elem_t *)(sh + j * xs + (int64_t)p * esz) =
                            (elem_t)(tmp[u] >> (8 * esz * e));
                }
            }
        }
        // Zero each vector's bytes from K up to the 16-byte padded length.
        const int64_t pad = kb - (int64_t)g.K * esz;
        if (tid < nvec * 16 && (tid & 15) < pad)
            sh[(tid >> 4) * xs + (int64_t)g.K * esz + (tid & 15)] = 0;
    } else {
        issue(0, buf0);
        using elem_t = typename std::conditional<esz == 1, uint8_t,
                         typename std::conditional<esz == 2, uint16_t, uint32_t>::type>::type;
        const elem_t *ve = (const elem_t *)vec;
        const int64_t epr = kb / esz, nel = nvec * epr;
        for (int64_t c0 = tid; c0 < nel; c0 += kSkThreads * 8) {
            elem_t tmp[8];
#pragma unroll
            for (int u = 0; u < 8; ++u) {
                const int64_t c = c0 + (int64_t)u * kSkThreads;
                const int64_t j = c / epr, p = c % epr;
                tmp[u] = (c < nel && p < g.K) ? ve[j * g.vld + p * g.vks] : (elem_t)0;
            }
#pragma unroll
            for (int u = 0; u < 8; ++u) {
                const int64_t c = c0 + (int64_t)u * kSkThreads;
                if (c < nel) *(elem_t *)(sh + (c / epr) * xs + (c % epr) * esz) = tmp[u];
            }
        }
    }
    val_t *comb = (val_t *)(sh + nvec * xs);
    __syncthreads();

    acc_t acc[2][BLK];
    // Multiplies batch t; after an item's last batch, forms each matrix row's
    // result from the two MFMAs, sums the four K ranges (wave order) through
    // LDS and applies the epilogue.
    auto run = [&](int t, const v4i_s (&m)[kSkPF][BLK]) {
        const int q = t % nbw;
        if (q == 0) {
#pragma unroll
            for (int b = 0; b < BLK; ++b) acc[0][b] = acc[1][b] = acc_t{};
        }
        const int s0 = ks0 + q * kSkPF;
#pragma unroll
        for (int p = 0; p < kSkPF; ++p) {
            const int s = s0 + p;
            if (s < ks1) {
#pragma unroll
                for (int h = 0; h < 2; ++h) {
                    v4i_s xv = *(const v4i_s *)(sh + xaddr + (int64_t)s * kSkStep + 16 * h);
                    if (!lvec || (int64_t)s * kSkStep + 16 * (2 * lg + h) >= kb) xv = v4i_s{0, 0, 0, 0};
#pragma unroll
                    for (int b = 0; b < BLK; ++b) acc[h][b] = Mm::step(m[p][b], xv, acc[h][b]);
                }
            }
        }
        if (q != nbw - 1) return;
        const int r0 = ((int)blockIdx.x + (t / nbw) * (int)gridDim.x) * kSkRows;
#pragma unroll
        for (int b = 0; b < BLK; ++b)
#pragma unroll
            for (int e = 0; e < 2; ++e)
                comb[((wave * BLK + b) * 2 + e) * 64 + lane] =
                    (val_t)acc[0][b][2 * e] + (val_t)acc[1][b][2 * e + 1];
        __syncthreads();
#pragma unroll
        for (int x = tid; x < BLK * 2 * 64; x += kSkThreads) {
            const int b = x / 128, e = (x / 64) % 2, ln = x % 64;
            val_t sum = comb[x];
#pragma unroll
            for (int w = 1; w < kSkWaves; ++w) sum += comb[w * BLK * 2 * 64 + x];
            const int64_t row = (int64_t)r0 + 8 * b + 2 * (ln >> 4) + e;
            const int j = ln & 15;
            if (j < nvec && row < g.R) Store<E>::apply(ep, zb, j, (int)row, sum);
        }
        __syncthreads();
    };
    for (int t = 0; t < total; t += 2) {
        if (t + 1 < total) issue(t + 1, buf1);
        run(t, buf0);
        if (t + 1 < total) {
            if (t + 2 < total) issue(t + 2, buf0);
            run(t + 1, buf1);
        }
    }
}

// Bytes of LDS the kernel needs (vectors + partial-sum exchange).
int64_t skinny_lds_bytes(InType in, int64_t K, int nvec) {
    const int64_t esz = in == InType::I8 ? 1 : (in == InType::BF16 ? 2 : 4);
    return nvec * skinny_xstride((K * esz + 15) / 16 * 16) + kSkCombine;
}

template <InType T, EpiKind E>
static hipError_t skinny_go(const GemvArgs &g, const EpiParams &ep, hipStream_t stream) {
    const int64_t shm = skinny_lds_bytes(T, g.K, g.nvec);
    const int cus = g.cus > 0 ? g.cus : 256;
    // 32-row items when there are enough of them for every CU, else 8-row
    // items (4x as many workgroups streaming the same bytes).
    const int64_t R = g.R;
    int rows = (R + 31) / 32 >= cus ? 32 : 8;
    // GEMMKIT_HIP_SKINNY_SHAPE="rows,wgs": rows per work item (8, 16 or 32)
    // and workgroups per CU, a tuning switch for the launch-shape sweep
    // (results do not change: each row's K ranges and their order are fixed
    // by K).
    int rows_env = 0, wgs_env = 0;
    if (const char *e = getenv("GEMMKIT_HIP_SKINNY_SHAPE"))
        if (sscanf(e, "%d,%d", &rows_env, &wgs_env) == 2 &&
            (rows_env == 8 || rows_env == 16 || rows_env == 32))
            rows = rows_env;
    const int64_t items = (R + rows - 1) / rows;
    // As many resident workgroups per CU as its 160 KiB of LDS holds (<= 4).
    const int fit = (int)(160 * 1024 / shm);
    int per_cu = fit < 4 ? (fit > 1 ? fit : 1) : 4;
    if (wgs_env > 0) per_cu = wgs_env < fit ? wgs_env : (fit > 1 ? fit : 1);
    // Batch elements share the persistent grid (grid y), each at least one
    // workgroup.
    const int64_t nb = g.batch > 1 ? g.batch : 1;
    int64_t blocks = ((int64_t)cus * per_cu + nb - 1) / nb;
    if (blocks > items) blocks = items;
    const dim3 grid((unsigned)blocks, (unsigned)nb);
    if (rows == 32)
        hipLaunchKernelGGL((skinny_mfma<T, E, 4>), grid, dim3(kSkThreads), (size_t)shm, stream, g,
                           ep);
    else if (rows == 16)
        hipLaunchKernelGGL((skinny_mfma<T, E, 2>), grid, dim3(kSkThreads), (size_t)shm, stream, g,
                           ep);
    else
        hipLaunchKernelGGL((skinny_mfma<T, E, 1>), grid, dim3(kSkThreads), (size_t)shm, stream, g,
                           ep);
    return hipGetLastError();
}

// ---- skinny_long ------------------------------------------------------------
// skinny_mfma's loads and matrix-core layout for vectors that would fill a CU's
// LDS: each wave reads its vector chunks beside the matrix's, from L2, so nothing
// is staged and the eight waves of a workgroup, one K range each, are the only
// limit on the loads in flight.  The vectors are k-contiguous with aligned rows.
// Every kSkPF steps the accumulators are added to running sums: a sum is then a
// chain of a few steps inside a chain of K / (8 waves * kSkPF steps): error against
// 64 bits 1.67e-7 rms at f32 8 x 11008 (standard normal times 1/sqrt(K)), 2.46e-7
// on the LDS GEMV that served it before.
// bf16 8 x 11008 x 4096 19.4 us against 73.7 there, 8 x 16384 x 1024 16.5 against
// 27, f32 8 x 11008 x 4096 38 (4.7 TB/s) against 97, 8 x 4096 x 4096 16 against 41.
constexpr int kSkLongWaves = 8;
constexpr int64_t kSkLongGrid = 1 << 22;  // workgroups per launch (2^31 threads)

template <InType T, EpiKind E, int BLK>
__global__ __launch_bounds__(kSkLongWaves * 64) void skinny_long(const GemvArgs g,
                                                                 const EpiParams ep, int row0) {
    constexpr int ROWS = 8 * BLK, NW = kSkLongWaves;
    using Mm = Mma16<T>;
    using acc_t = typename Mm::acc_t;
    using val_t = typename Mm::val_t;
    constexpr int esz = (T == InType::I8) ? 1 : (T == InType::BF16 ? 2 : 4);
    __shared__ val_t comb[NW][BLK * 2 * 64];
    const int64_t kb = ((int64_t)g.K * esz + 15) / 16 * 16;
    const int nk = (int)((kb + kSkStep - 1) / kSkStep);
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int li = lane & 15, lg = lane >> 4;
    const int chunk = 2 * lg + (li & 1);
    const int kseg = (nk + NW - 1) / NW;
    const int ks0 = wave * kseg, ks1 = ks0 + kseg < nk ? ks0 + kseg : nk;
    const int64_t zb = blockIdx.y;
    const int64_t ld_b = g.ld * esz, vld_b = g.vld * esz;
    const int r0 = row0 + (int)blockIdx.x * ROWS;
    const uint8_t *mat = (const uint8_t *)g.mat + zb * g.bsm * esz + (int64_t)r0 * ld_b;
    const uint8_t *vec = (const uint8_t *)g.vec + zb * g.bsv * esz;
    const int nrows = g.R - r0 < ROWS ? g.R - r0 : ROWS;
    const uint32_t num = (uint32_t)((nrows - 1) * ld_b + kb);
    const uint32_t vnum = (uint32_t)((g.nvec - 1) * vld_b + kb);
    uint32_t off[BLK];
#pragma unroll
    for (int b = 0; b < BLK; ++b) off[b] = (uint32_t)((8 * b + (li >> 1)) * ld_b + 16 * chunk);
    const uint32_t voff = (uint32_t)(li < g.nvec ? li : 0) * (uint32_t)vld_b + 32 * lg;
    const uint32_t vout = (uint32_t)(li >= g.nvec) << 31;  // columns past nvec: zeros
    // Chunks past K or the wave's range read zeros (bit 31 is past any extent here).
    auto issue = [&](int s0, v4i_s (&m)[kSkPF][BLK], v4i_s (&x)[kSkPF][2]) {
#pragma unroll
        for (int p = 0; p < kSkPF; ++p) {
            const int s = s0 + p;
            const uint32_t k = (uint32_t)s * kSkStep;
#pragma unroll
            for (int h = 0; h < 2; ++h) {
                const bool in = s < ks1 && (int64_t)k + 16 * (2 * lg + h) < kb;
                x[p][h] = load16v(vec, vnum, (voff + k + 16 * h) | vout | (uint32_t)!in << 31);
            }
            const bool in = s < ks1 && (int64_t)k + 16 * chunk < kb;
#pragma unroll
            for (int b = 0; b < BLK; ++b)
                m[p][b] = load16(mat, num, (off[b] + k) | (uint32_t)!in << 31);
        }
        __builtin_amdgcn_sched_barrier(0);
    };
    val_t sum[2][BLK][2] = {};  // [h][block][e]: the running sums of a matrix row's halves
    auto run = [&](int s0, const v4i_s (&m)[kSkPF][BLK], const v4i_s (&x)[kSkPF][2]) {
        acc_t acc[2][BLK] = {};
#pragma unroll
        for (int p = 0; p < kSkPF; ++p)
#pragma unroll
            for (int h = 0; h < 2; ++h)
#pragma unroll
                for (int b = 0; b < BLK; ++b) acc[h][b] = Mm::step(m[p][b], x[p][h], acc[h][b]);
#pragma unroll
        for (int b = 0; b < BLK; ++b)
#pragma unroll
            for (int e = 0; e < 2; ++e) {
                sum[0][b][e] += acc[0][b][2 * e];
                sum[1][b][e] += acc[1][b][2 * e + 1];
            }
        __builtin_amdgcn_sched_barrier(0);
    };
    v4i_s m0[kSkPF][BLK], m1[kSkPF][BLK], x0[kSkPF][2], x1[kSkPF][2];
    if (ks0 < ks1) {
        issue(ks0, m0, x0);
        for (int s = ks0; s < ks1; s += 2 * kSkPF) {
            if (s + kSkPF < ks1) issue(s + kSkPF, m1, x1);
            run(s, m0, x0);
            if (s + kSkPF >= ks1) break;
            if (s + 2 * kSkPF < ks1) issue(s + 2 * kSkPF, m0, x0);
            run(s + kSkPF, m1, x1);
        }
    }
#pragma unroll
    for (int b = 0; b < BLK; ++b)
#pragma unroll
        for (int e = 0; e < 2; ++e) comb[wave][(b * 2 + e) * 64 + lane] = sum[0][b][e] + sum[1][b][e];
    __syncthreads();
    for (int x = tid; x < BLK * 2 * 64; x += NW * 64) {
        val_t v = comb[0][x];
#pragma unroll
        for (int w = 1; w < NW; ++w) v += comb[w][x];
        const int b = x / 128, e = (x / 64) % 2, ln = x % 64;
        const int row = r0 + 8 * b + 2 * (ln >> 4) + e, j = ln & 15;
        if (j < g.nvec && row < g.R) Store<E>::apply(ep, zb, j, row, v);
    }
}

template <InType T, EpiKind E>
static hipError_t skinny_long_go(const GemvArgs &g, const EpiParams &ep, hipStream_t stream) {
    const int cus = g.cus > 0 ? g.cus : 256;
    const int64_t R = g.R, nb = g.batch;
    // A workgroup's rows (its registers leave room for one workgroup a CU): one round of
    // the CUs where that takes at most 32 rows, and no more rows than it takes (bf16
    // 16 x 8000, 16 rows in two rounds before: 4500 rows 26.5 us, 24 rows 19.9; 7000
    // rows 29.7, 32 rows 24.7).
    auto items = [&](int64_t rows) { return (R + rows - 1) / rows * nb; };
    const int rows = items(24) > cus ? 32 : (items(16) > cus ? 24 : (items(16) == cus ? 16 : 8));
    const dim3 block(kSkLongWaves * 64);
    for (int64_t r = 0; r < R; r += rows * kSkLongGrid) {
        const int64_t left = (R - r + rows - 1) / rows;
        const dim3 grid((unsigned)(left < kSkLongGrid ? left : kSkLongGrid), (unsigned)nb);
        if (rows == 32)
            hipLaunchKernelGGL((skinny_long<T, E, 4>), grid, block, 0, stream, g, ep, (int)r);
        else if (rows == 24)
            hipLaunchKernelGGL((skinny_long<T, E, 3>), grid, block, 0, stream, g, ep, (int)r);
        else if (rows == 16)
            hipLaunchKernelGGL((skinny_long<T, E, 2>), grid, block, 0, stream, g, ep, (int)r);
        else
            hipLaunchKernelGGL((skinny_long<T, E, 1>), grid, block, 0, stream, g, ep, (int)r);
    }
    return hipGetLastError();
}

hipError_t launch_skinny_long(InType in, const GemvArgs &g, const EpiParams &ep,
                              hipStream_t stream) {
    const int64_t esz = in == InType::I8 ? 1 : (in == InType::BF16 ? 2 : 4);
    // (32-bit offsets from an item's first row and the first vector; 16-byte
    // vector chunks)
    if (g.nvec < 1 || g.nvec > 16 || g.R < 1 || g.ld < 0 || g.vld < 0 || g.vks != 1 ||
        15 * g.vld * esz + g.K * esz >= 0x7FFFFF00ll || g.batch < 1 || g.batch > kMaxGridZ)
        return hipErrorInvalidValue;
    switch (in) {
    case InType::I8:
        if (ep.kind == EpiKind::I32) return skinny_long_go<InType::I8, EpiKind::I32>(g, ep, stream);
        if (ep.kind == EpiKind::Q8) return skinny_long_go<InType::I8, EpiKind::Q8>(g, ep, stream);
        break;
    case InType::F32:
        if (ep.kind == EpiKind::F32) return skinny_long_go<InType::F32, EpiKind::F32>(g, ep, stream);
        break;
    case InType::BF16:
        if (ep.kind == EpiKind::F32) return skinny_long_go<InType::BF16, EpiKind::F32>(g, ep, stream);
        if (ep.kind == EpiKind::BF16)
            return skinny_long_go<InType::BF16, EpiKind::BF16>(g, ep, stream);
        break;
    }
    return hipErrorInvalidValue;
}

bool skinny_is_long(InType in, int64_t K, int nvec) {
    return skinny_lds_bytes(in, K, nvec) > kSkinnyLdsMax;
}

// ---- skinny_cols ------------------------------------------------------------
// The same products with a matrix of unit row stride (element (r, p) at
// r + p*mks, any mks and alignment; x * W with W row-major) and k-contiguous
// vectors (any alignment), read in place.
//
// A lane loads 8 bytes, RPL rows, at one k (16 lanes side by side a run of 128
// bytes), for each k of its 16-byte chunk; byte permutes in registers turn them
// into RPL matrix-core operands, operand t holding rows RPL*i + t of the lanes
// i.  The kernel above sums a row in eight parts: four K ranges, each the sum
// of the even 16-byte chunks of its 128-byte steps (MFMA h = 0) and of the odd
// ones (h = 1).  Here every part is a wave of its own -- workgroup = (part, 16*RPL
// rows) -- which stores its sums, and cols_sum adds the parts in the order above:
// results equal that kernel's on a packed copy bit for bit.  i8, whose sums have no
// order, takes more ranges when the parts are few for the CUs.
//
// Bound by streaming the matrix once, against three passes when it is packed first
// (copies in turn, together beyond the caches; second launch included): bf16
// 8 x 4096 x 4096 10.6 us against 25.1, 4 x 4096 x 11008 18.4 (4.9 TB/s) against
// 51, 16 x 1024 x 1024 5.3 against 8.8; f32 4 x 4096 x 11008 36.1 (5.0 TB/s) against
// 122, 8 x 1024 x 16384 19.4 against 45; i8 8 x 11008 x 4096 13.0 against 36.5.
typedef int v2i_s __attribute__((ext_vector_type(2)));
typedef int v2i_sany __attribute__((ext_vector_type(2), aligned(1)));
typedef int v4i_sany __attribute__((ext_vector_type(4), aligned(1)));

template <InType T>
struct SkCols;

template <>
struct SkCols<InType::F32> {
    static constexpr int PF = 8;  // k steps per batch of loads (64 registers)
    using acc_t = v4f_s;
    using elem_t = uint32_t;
    // m[e]: the lane's RPL rows at k = e of its chunk; x: the chunk of its vector.
    __device__ __forceinline__ static void step(const v2i_s (&m)[4], v4i_s x, acc_t (&acc)[2]) {
        const v4f_s xf = __builtin_bit_cast(v4f_s, x);
#pragma unroll
        for (int e = 0; e < 4; ++e)
#pragma unroll
            for (int t = 0; t < 2; ++t)
                acc[t] = __builtin_amdgcn_mfma_f32_16x16x4f32(__int_as_float(m[e][t]), xf[e],
                                                              acc[t], 0, 0, 0);
    }
};

template <>
struct SkCols<InType::BF16> {
    static constexpr int PF = 4;
    using acc_t = v4f_s;
    using elem_t = uint16_t;
    __device__ __forceinline__ static void step(const v2i_s (&m)[8], v4i_s x, acc_t (&acc)[4]) {
#pragma unroll
        for (int t = 0; t < 4; ++t) {
            v4i_s w;
#pragma unroll
            for (int i = 0; i < 4; ++i)
                w[i] = (int)__builtin_amdgcn_perm((uint32_t)m[2 * i + 1][t / 2],
                                                  (uint32_t)m[2 * i][t / 2],
                                                  t % 2 ? 0x07060302u : 0x05040100u);
            acc[t] = Mma16<InType::BF16>::step(w, x, acc[t]);
        }
    }
};

template <>
struct SkCols<InType::I8> {
    static constexpr int PF = 2;
    using acc_t = v4i_s;
    using elem_t = uint8_t;
    __device__ __forceinline__ static void step(const v2i_s (&m)[16], v4i_s x, acc_t (&acc)[8]) {
#pragma unroll
        for (int c = 0; c < 2; ++c) {
            v4i_s w[4];  // 4 x 4 byte transposes: four k of a row side by side
#pragma unroll
            for (int p = 0; p < 4; ++p) {
                const uint32_t i0 = m[4 * p][c], i1 = m[4 * p + 1][c];
                const uint32_t i2 = m[4 * p + 2][c], i3 = m[4 * p + 3][c];
                const uint32_t t0 = __builtin_amdgcn_perm(i1, i0, 0x05010400u);
                const uint32_t t1 = __builtin_amdgcn_perm(i1, i0, 0x07030602u);
                const uint32_t u0 = __builtin_amdgcn_perm(i3, i2, 0x05010400u);
                const uint32_t u1 = __builtin_amdgcn_perm(i3, i2, 0x07030602u);
                w[0][p] = (int)__builtin_amdgcn_perm(u0, t0, 0x05040100u);
                w[1][p] = (int)__builtin_amdgcn_perm(u0, t0, 0x07060302u);
                w[2][p] = (int)__builtin_amdgcn_perm(u1, t1, 0x05040100u);
                w[3][p] = (int)__builtin_amdgcn_perm(u1, t1, 0x07060302u);
            }
#pragma unroll
            for (int t = 0; t < 4; ++t)
                acc[4 * c + t] = Mma16<InType::I8>::step(w[t], x, acc[4 * c + t]);
        }
    }
};

template <InType T, bool LONG>
__global__ __launch_bounds__(64) void skinny_cols(const GemvArgs g, int ranges) {
    using Sc = SkCols<T>;
    using elem_t = typename Sc::elem_t;
    using val_t = typename Mma16<T>::val_t;
    constexpr int EPC = 16 / (int)sizeof(elem_t), RPL = 8 / (int)sizeof(elem_t);
    constexpr int ROWS = 16 * RPL, STEPK = kSkStep / (int)sizeof(elem_t), PF = Sc::PF;
    const int lane = threadIdx.x, li = lane & 15, lg = lane >> 4;
    const unsigned groups = (unsigned)(((int64_t)g.R + ROWS - 1) / ROWS);
    const int unit = (int)(blockIdx.x / groups), h = unit & 1, range = unit >> 1;
    const int64_t rg = (int64_t)(blockIdx.x % groups) * ROWS, zb = blockIdx.y;
    // Rows start RPL before R at the latest, so every load stays inside the
    // matrix (the caller ensures R >= RPL); overlapping lanes form, and store,
    // the same sums.
    const auto row_of = [&](int i) {
        return rg + RPL * i + RPL <= g.R ? rg + RPL * i : (int64_t)g.R - RPL;
    };
    const int nk = (int)(((int64_t)g.K + STEPK - 1) / STEPK);
    const int kseg = (nk + ranges - 1) / ranges;
    const int ks0 = range * kseg, ks1 = ks0 + kseg < nk ? ks0 + kseg : nk;
    const int whole = g.K / STEPK, kfull = ks1 < whole ? ks1 : whole;  // whole steps: [ks0, kfull)
    const int64_t k0 = (2 * lg + h) * EPC;  // this lane's chunk of a step
    const elem_t *mat = (const elem_t *)g.mat + zb * g.bsm + row_of(li) + k0 * g.mks;
    // (columns past nvec repeat the last vector; they are not stored)
    const elem_t *vec = (const elem_t *)g.vec + zb * g.bsv +
                        (int64_t)(li < g.nvec ? li : g.nvec - 1) * g.vld + k0;

    typename Sc::acc_t acc[RPL] = {};
    // LONG (floats): skinny_long's running sums, every kSkPF steps of the range.
    typename Sc::acc_t sum[LONG ? RPL : 1] = {};
    auto step = [&](int s, const v2i_s (&m)[EPC], v4i_s x) {
        Sc::step(m, x, acc);
        if constexpr (LONG) {
            if ((s - ks0) % kSkPF == kSkPF - 1 || s == ks1 - 1) {
#pragma unroll
                for (int t = 0; t < RPL; ++t) {
                    sum[t] += acc[t];
                    acc[t] = typename Sc::acc_t{};
                }
            }
        }
    };
    // Two batches in turn, the next one's loads in flight while one is
    // multiplied.  All loads of a batch are issued before any is used; steps past
    // the end load the last one again and are left out.
    auto load = [&](int s, v2i_s (&m)[PF][EPC], v4i_s (&x)[PF]) {
#pragma unroll
        for (int u = 0; u < PF; ++u) {
            const int64_t k = (int64_t)(s + u < kfull ? s + u : kfull - 1) * STEPK;
            x[u] = *(const v4i_sany *)(vec + k);
#pragma unroll
            for (int e = 0; e < EPC; ++e) m[u][e] = *(const v2i_sany *)(mat + (k + e) * g.mks);
        }
        __builtin_amdgcn_sched_barrier(0);
    };
    auto mul = [&](int s, const v2i_s (&m)[PF][EPC], const v4i_s (&x)[PF]) {
#pragma unroll
        for (int u = 0; u < PF; ++u)
            if (s + u < kfull) step(s + u, m[u], x[u]);
        __builtin_amdgcn_sched_barrier(0);
    };
    if (ks0 < kfull) {
        v2i_s m0[PF][EPC], m1[PF][EPC];
        v4i_s x0[PF], x1[PF];
        load(ks0, m0, x0);
        for (int s = ks0; s < kfull; s += 2 * PF) {
            if (s + PF < kfull) load(s + PF, m1, x1);
            mul(s, m0, x0);
            if (s + PF >= kfull) break;
            if (s + 2 * PF < kfull) load(s + 2 * PF, m0, x0);
            mul(s + PF, m1, x1);
        }
    }
    if (whole >= ks0 && whole < ks1) {  // the last step, zeros past K
        v2i_s m[EPC];
        elem_t v[EPC];
        const int64_t k = (int64_t)whole * STEPK;
#pragma unroll
        for (int e = 0; e < EPC; ++e) {
            const bool in = k + k0 + e < g.K;
            m[e] = v2i_s{0, 0};
            v[e] = elem_t(0);
            if (in) {
                m[e] = *(const v2i_sany *)(mat + (k + e) * g.mks);
                v[e] = vec[k + e];
            }
        }
        v4i_s x;
        __builtin_memcpy(&x, v, 16);
        step(whole, m, x);
    }
    if (li < g.nvec) {
        val_t *out = (val_t *)g.part + ((zb * 2 * ranges + unit) * g.nvec + li) * g.R;
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            val_t v[RPL];
#pragma unroll
            for (int t = 0; t < RPL; ++t) v[t] = LONG ? sum[LONG ? t : 0][q] : acc[t][q];
            __builtin_memcpy(out + row_of(4 * lg + q), v, sizeof(v));
        }
    }
}

// Adds the parts [element][range][h][vector][row], one output per thread.
template <InType T, EpiKind E, int RANGES>
__global__ __launch_bounds__(64) void cols_sum(const GemvArgs g, const EpiParams ep) {
    using val_t = typename Mma16<T>::val_t;
    const int64_t r = (int64_t)blockIdx.x * 64 + threadIdx.x;
    const int j = blockIdx.y;
    const int64_t zb = blockIdx.z;
    if (r >= g.R) return;
    val_t v[2 * RANGES];
#pragma unroll
    for (int u = 0; u < 2 * RANGES; ++u)
        v[u] = ((const val_t *)g.part)[((zb * 2 * RANGES + u) * g.nvec + j) * g.R + r];
    val_t sum = v[0] + v[1];
#pragma unroll
    for (int u = 1; u < RANGES; ++u) sum += v[2 * u] + v[2 * u + 1];
    Store<E>::apply(ep, zb, j, (int)r, sum);
}

// K ranges: the row kernel's for floats (its order); i8 up to 16 while that leaves
// fewer than four waves per CU, half a batch of loads to each and a scratch no larger
// than a quarter of the matrix.
static int skinny_cols_ranges(InType in, int64_t R, int64_t K, int nvec, int64_t batch, int cus) {
    if (in != InType::I8) return skinny_is_long(in, K, nvec) ? kSkLongWaves : kSkWaves;
    int ranges = 4;
    const int64_t groups = (R + 127) / 128 * batch;
    while (ranges < 16 && groups * 2 * ranges < 4 * (int64_t)(cus > 0 ? cus : 256) &&
           K >= (int64_t)ranges * 128 * SkCols<InType::I8>::PF &&
           4 * ranges * nvec * 4 * 4 <= K)
        ranges *= 2;
    return ranges;
}

int64_t skinny_cols_part_bytes(InType in, int64_t R, int64_t K, int nvec, int64_t batch, int cus) {
    return 2 * skinny_cols_ranges(in, R, K, nvec, batch, cus) * batch * nvec * R * 4;
}

template <InType T, EpiKind E>
static hipError_t skinny_cols_go(const GemvArgs &g, const EpiParams &ep, hipStream_t stream) {
    constexpr int ROWS = 16 * 8 / (T == InType::I8 ? 1 : (T == InType::BF16 ? 2 : 4));
    const int ranges = skinny_cols_ranges(T, g.R, g.K, g.nvec, g.batch, g.cus);
    const int64_t groups = ((int64_t)g.R + ROWS - 1) / ROWS;
    const dim3 parts((unsigned)(groups * 2 * ranges), (unsigned)g.batch);
    const dim3 grid((unsigned)(((int64_t)g.R + 63) / 64), (unsigned)g.nvec, (unsigned)g.batch);
    if (T != InType::I8 && ranges == kSkLongWaves)
        hipLaunchKernelGGL((skinny_cols<T, T != InType::I8>), parts, dim3(64), 0, stream, g, ranges);
    else
        hipLaunchKernelGGL((skinny_cols<T, false>), parts, dim3(64), 0, stream, g, ranges);
    if constexpr (T == InType::I8) {
        if (ranges == 16)
            hipLaunchKernelGGL((cols_sum<T, E, 16>), grid, dim3(64), 0, stream, g, ep);
    }
    if (ranges == 8) hipLaunchKernelGGL((cols_sum<T, E, 8>), grid, dim3(64), 0, stream, g, ep);
    if (ranges == 4) hipLaunchKernelGGL((cols_sum<T, E, 4>), grid, dim3(64), 0, stream, g, ep);
    return hipGetLastError();
}

hipError_t launch_skinny_cols(InType in, const GemvArgs &g, const EpiParams &ep,
                              hipStream_t stream) {
    if (g.nvec < 1 || g.nvec > 16 || g.R < kSkinnyColsMinRows || g.ld != 1 || g.vks != 1 ||
        !g.part || g.batch < 1 || g.batch > kMaxGridZ)
        return hipErrorInvalidValue;
    switch (in) {
    case InType::I8:
        if (ep.kind == EpiKind::I32) return skinny_cols_go<InType::I8, EpiKind::I32>(g, ep, stream);
        if (ep.kind == EpiKind::Q8) return skinny_cols_go<InType::I8, EpiKind::Q8>(g, ep, stream);
        break;
    case InType::F32:
        if (ep.kind == EpiKind::F32) return skinny_cols_go<InType::F32, EpiKind::F32>(g, ep, stream);
        break;
    case InType::BF16:
        if (ep.kind == EpiKind::F32) return skinny_cols_go<InType::BF16, EpiKind::F32>(g, ep, stream);
        if (ep.kind == EpiKind::BF16)
            return skinny_cols_go<InType::BF16, EpiKind::BF16>(g, ep, stream);
        break;
    }
    return hipErrorInvalidValue;
}

hipError_t launch_skinny(InType in, const GemvArgs &g, const EpiParams &ep, hipStream_t stream) {
    // The matrix rows are addressed as unsigned 32-bit offsets from an item's
    // first row, so its row stride must be non-negative (the vectors may
    // have any strides).
    if (g.nvec < 1 || g.nvec > 16 || g.R < 1 || g.ld < 0 || g.batch < 1 || g.batch > kMaxGridZ ||
        skinny_lds_bytes(in, g.K, g.nvec) > kSkinnyLdsMax)
        return hipErrorInvalidValue;
    switch (in) {
    case InType::I8:
        if (ep.kind == EpiKind::I32) return skinny_go<InType::I8, EpiKind::I32>(g, ep, stream);
        if (ep.kind == EpiKind::Q8) return skinny_go<InType::I8, EpiKind::Q8>(g, ep, stream);
        break;
    case InType::F32:
        if (ep.kind == EpiKind::F32) return skinny_go<InType::F32, EpiKind::F32>(g, ep, stream);
        break;
    case InType::BF16:
        if (ep.kind == EpiKind::F32) return skinny_go<InType::BF16, EpiKind::F32>(g, ep, stream);
        if (ep.kind == EpiKind::BF16) return skinny_go<InType::BF16, EpiKind::BF16>(g, ep, stream);
        break;
    }
    return hipErrorInvalidValue;
}

}  // namespace gk
