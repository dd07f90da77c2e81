// f32x.hip -- f32 GEMM on the bf16 matrix cores, at f32 precision: every operand
// element is split into three bf16 parts and eight of the nine products of parts
// are summed in f32.
//
// Replaces the same layers as mma_kernel.h (src/driver.rs:402-944,
// src/kernel/float.rs:150-281) for f32 products with K of 128 or more beyond the
// small products of small.hip.
//
// Why.  CDNA4's f32 matrix rate is 1/16 of its bf16 rate (157 against 2500
// TFLOP/s), so eight bf16 products per f32 product leave twice the f32 rate.
// The split loses nothing: a = h + m + l with h = bf16(a), m = bf16(a - h),
// l = a - h - m is exact (24 significant bits in three times eight, both
// subtractions exact), and the products of parts are exact in f32 (pairs of 8-bit
// significands).  |m| <= 2^-8 |a| and |l| <= 2^-17 |a|, so the one product left
// out (ll) is at most 2^-34 of |a||b|.
//
// Sums.  The matrix cores cut the lower of two addends off at the result's last
// bit, so a small product added to a sum there costs up to an ulp.  The seven
// small products (2^-7 of the whole at most) of 32 k are therefore summed apart,
// smallest first, and added to the sum, which has taken the large ones (hh), in
// one rounded f32 addition: a sum of a single term is its correctly rounded value
// but within 2^-6 ulp of a tie (the f32 instructions': always).  With HL (the shapes
// small.hip would serve, whose sixteen partial sums round less) the small sum
// runs over all of K and is added once.  With ml and lm left out too, together up
// to 2^-24, and all products in one sum a single term erred by up to 1.4 ulp
// (2048^3: 93 us instead of 108).
// Measured (row-major, against the f32 tiles with B packed first): 2048^3 108 us =
// 159 TFLOP/s against 138, relative error on normal inputs 2.1e-7 against 8.1e-7;
// 1024^3 22.5 against 29.2, 1.5e-7 against 5.7e-7; 488 x 2512 x 3136 76 against 95.
// Bound by the matrix cores at the clock the chip's power limit leaves them: 1270
// TFLOP/s of bf16 products, where library products reach 1338 (4096^3) to 1610.
//
// Range.  Elements are scaled by 2^23 as they are split and the sums by 2^-46 at
// the end, both exact (a subnormal result is rounded once more): every part of
// every finite f32 below 2^105 is then a normal bf16 number or 0 (f32 values are
// multiples of 2^-149, so parts of 2^-126), and every product of parts that
// matters to a result of 2^-149 or more is a normal f32.  Larger elements,
// infinities and NaN leave a sum that is not finite, and so do results of 2^82 or
// more: a 16 x 16 block of the output with such a sum is computed again with the
// f32 instructions.  The blocks are cut at multiples of 16 whatever the tile, so an
// element's value does not depend on the tile that computed it.
// The second pass waits for the first and shares no operands between waves:
// 2048^3 with an infinity among 100,000 elements 280 us, with one in every block 360,
// against 108 without and 138 on the f32 tiles; zeros, subnormals and the smallest
// normal values cost nothing (unscaled parts below 2^-126 sent 64 x 64 blocks to
// such a pass: 380 us on 2048^3, 110 against 22 on 1024^3, with one element of
// 10,000 at 1e-35).
//
// Schedule.  One workgroup of two groups of four waves per BM x BN tile; a stage
// is 32 k, group g multiplies the stages of its parity (every wave of it a
// quarter of the tile) and the two partial tiles are added at the end.  The
// groups alternate, one wave of each per SIMD: while one multiplies stage n from
// fragments in registers, the other reads the fragments of stage n+1 from LDS,
// splits the elements of stage n+3 (loaded two slots before) into the slot
// stage n left, and issues the loads of stage n+5; then a barrier, and the roles
// change.  The matrix cores so always have a wave with nothing else to wait
// for, and the splitting, the LDS traffic and the memory latency run beside it.
// (All eight waves doing all of it in turn, with six products: 102 us on 2048^3
// against 85.)  A K that is no multiple of 32 has its short stage first, outside
// the loop.
//
// Operands are read in place with any strides (the caller packs those that this
// would read a cache line at a time): a k-contiguous operand as two 16-byte loads
// of 8 k of a row per thread, any other as 8 element loads with the lanes along the
// rows (coalesced when the rows are contiguous).
// LDS holds, per stage and part, 64-byte rows of 32 k; row r keeps its 16-byte
// chunk c in slot c ^ ((r >> 2) & 3), which spreads 16 consecutive rows (a
// fragment read, and the writes of either load form) over distinct banks.
// v_mfma_f32_16x16x32_bf16 takes B's fragment as its first operand, so
// register q of lane l is output row l%16, column 4*(l/16) + q of a block: four
// consecutive columns, one 16-byte store.
#include "epilogue.h"
#include "mma_kernel.h"

namespace gk {

typedef float v4f_x __attribute__((ext_vector_type(4)));
typedef float v4f_xu __attribute__((ext_vector_type(4), aligned(4)));
typedef uint32_t v4u_x __attribute__((ext_vector_type(4)));
typedef __bf16 v8bf_x __attribute__((ext_vector_type(8)));

constexpr int kXStage = 32;              // k per stage
constexpr int kXRow = kXStage * 2;       // LDS bytes of a row of one part
// Both operands are scaled by 2^23 as they are split, the sums by 2^-46 at the end.
constexpr float kXScale = 0x1p23f, kXUnscale = 0x1p-46f;

// The three bf16 parts of 8 consecutive k of a row.  (Forming the differences
// with v_dot2_f32_bf16, two instructions fewer per pair, doubled the time of a
// slot: it contends with the other group's MFMAs, plain VALU does not.)
__device__ __forceinline__ void x_split(const float (&v)[8], v4u_x &h, v4u_x &m, v4u_x &l) {
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const float a0 = v[2 * i] * kXScale, a1 = v[2 * i + 1] * kXScale;
        const uint32_t hp = bf16x2_rne(a0, a1);
        const float r0 = a0 - __uint_as_float(hp << 16);
        const float r1 = a1 - __uint_as_float(hp & 0xFFFF0000u);
        const uint32_t mp = bf16x2_rne(r0, r1);
        h[i] = hp;
        m[i] = mp;
        l[i] = bf16x2_rne(r0 - __uint_as_float(mp << 16), r1 - __uint_as_float(mp & 0xFFFF0000u));
    }
}

// AK / BK: the operand is k-contiguous.
constexpr int kXThreads = 512, kXGroup = 256;
// HL: the small products in accumulators of their own over all of K.
// WPE: waves per SIMD (128 registers each at 4, 256 at 2).
template <int BM, int BN, bool AK, bool BK, bool HL, int WPE>
__global__ __launch_bounds__(kXThreads)
__attribute__((amdgpu_waves_per_eu(WPE, WPE)))
void f32x_kernel(const SmallArgs g, const EpiParams ep) {
    constexpr int WTM = BM / 2, WTN = BN / 2;        // a wave's rows and columns
    constexpr int TM = WTM / 16, TN = WTN / 16;
    constexpr int IA = BM * 4 / kXGroup, IB = BN * 4 / kXGroup;  // 8-k chunks per thread and stage
    static_assert(IA >= 1 && IB >= 1 && 64 % WTM == 0 && 64 % WTN == 0, "tile");
    constexpr int PART = (BM + BN) * kXRow;          // one part of one stage
    constexpr int BUF = 3 * PART;
    static_assert(kXThreads * TM * TN * 2 * 4 <= 3 * BUF, "exchange of the partial tiles");
    __shared__ __attribute__((aligned(16))) uint8_t lds[3 * BUF];

    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int grp = wave >> 2, wm = (wave >> 1) & 1, wn = wave & 1, gt = tid & (kXGroup - 1);
    const int tiles_m = (g.M + BM - 1) / BM, tiles_n = (g.N + BN - 1) / BN;
    const int64_t pid = xcd_logical((int64_t)blockIdx.y * gridDim.x + blockIdx.x,
                                    (int64_t)gridDim.x * gridDim.y);
    const int64_t zb = pid / gridDim.x;
    int tm, tn;
    tile_coords((int)(pid % gridDim.x), tiles_m, tiles_n, tm, tn);
    const int m0 = tm * BM, n0 = tn * BN;
    const float *A = (const float *)g.a + zb * g.bsa;
    const float *B = (const float *)g.b + zb * g.bsb;

    // A thread's NC chunks of a stage, IA of A and the others of B: a row and eight
    // k, chunk c holding k 4c..4c+3 and 16+4c..16+4c+3 (both operands alike, so any
    // order pairs the right products).  k-contiguous: four threads side by side
    // read 64 bytes of a row at a time; otherwise the lanes lie along the rows.
    // Rows past the matrix edge read its last row (their outputs are not stored).
    constexpr int NC = IA + IB;
    auto of_a = [](int i) { return i < IA; };
    auto ks_of = [&](int i) { return of_a(i) ? g.ksa : g.ksb; };
    auto kc_of = [&](int i) { return of_a(i) ? AK : BK; };
    auto row_of = [&](int i) {
        const int c = gt + (of_a(i) ? i : i - IA) * kXGroup;
        return kc_of(i) ? c / 4 : c % (of_a(i) ? BM : BN);
    };
    auto chunk_of = [&](int i) {
        const int c = gt + (of_a(i) ? i : i - IA) * kXGroup;
        return kc_of(i) ? c % 4 : c / (of_a(i) ? BM : BN);
    };
    const float *src[NC];
#pragma unroll
    for (int i = 0; i < NC; ++i) {
        const int r = row_of(i), c = chunk_of(i);
        const int64_t o = of_a(i) ? (m0 + r < g.M ? m0 + r : g.M - 1) : (n0 + r < g.N ? n0 + r : g.N - 1);
        src[i] = (of_a(i) ? A + o * g.rsa : B + o * g.rsb) + 4 * c * ks_of(i);
    }
    // LDS byte offset of a chunk in a part: rows 64 further down keep their slot
    // (k-contiguous), chunks two further on flip one bit of it.
    auto slot_of = [&](int i) {
        const int r = row_of(i), c = chunk_of(i);
        return r * kXRow + ((c ^ ((r >> 2) & 3)) * 16);
    };
    const int dst_a = slot_of(0), dst_b = BM * kXRow + slot_of(IA);
    auto dst = [&](int i) {
        const int n = of_a(i) ? i : i - IA, d = of_a(i) ? dst_a : dst_b;
        return kc_of(i) ? d + n * 64 * kXRow : d ^ (n * (kXGroup / (of_a(i) ? BM : BN)) * 16);
    };
    // Stage t covers k from 32*(t - rag): the whole stages, after the short one
    // (the last K % 32 k) when there is one.
    const int rag = g.K % kXStage != 0, whole = g.K / kXStage, stages = whole + rag;

    float raw[NC][8];
    v4u_x ph[NC], pm[NC], pl[NC];
    auto load = [&](int i, int t) {  // a whole stage; past the last one, the last again
        const int64_t ks = ks_of(i);
        const float *p = src[i] + (int64_t)((t < stages ? t : stages - 1) - rag) * kXStage * ks;
        if (kc_of(i)) {
            const v4f_x lo = *(const v4f_xu *)p, hi = *(const v4f_xu *)(p + 16);
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                raw[i][e] = lo[e];
                raw[i][4 + e] = hi[e];
            }
        } else {
#pragma unroll
            for (int e = 0; e < 8; ++e) raw[i][e] = p[(e < 4 ? e : e + 12) * ks];
        }
    };
    auto load_short = [&](int i) {  // zeros past K
        const float *p = src[i] + (int64_t)whole * kXStage * ks_of(i);
        const int left = g.K - whole * kXStage - 4 * chunk_of(i);
#pragma unroll
        for (int e = 0; e < 8; ++e) {
            const int k = e < 4 ? e : e + 12;
            raw[i][e] = k < left ? p[k * ks_of(i)] : 0.0f;
        }
    };
    auto split = [&](int i) {
        x_split(raw[i], ph[i], pm[i], pl[i]);
        // (keeps the splitting in its slot: the compiler sinks it to the writes)
        asm volatile("" : "+v"(ph[i]), "+v"(pm[i]), "+v"(pl[i]));
    };
    auto put = [&](uint8_t *buf, int i) {
        *(v4u_x *)(buf + dst(i)) = ph[i];
        *(v4u_x *)(buf + PART + dst(i)) = pm[i];
        *(v4u_x *)(buf + 2 * PART + dst(i)) = pl[i];
    };

    // This lane's fragment offsets: row l%16 of a block, chunk l/16.
    const int fr = lane & 15, fc = lane >> 4;
    const int fsw = (fc ^ ((fr >> 2) & 3)) * 16;
    const int fa = (wm * WTM + fr) * kXRow + fsw, fb = (BM + wn * WTN + fr) * kXRow + fsw;
    v8bf_x a[3][TM], b[3][TN];
    // Part q of NC of a stage's fragments.
    constexpr int NF = 3 * (TM + TN) / NC;
    static_assert(3 * (TM + TN) % NC == 0, "fragments per chunk");
    auto frags = [&](const uint8_t *buf, int q) {
#pragma unroll
        for (int f = 0; f < NF; ++f) {
            const int x = q * NF + f, p = x / (TM + TN), o = x % (TM + TN);
            const int off = o < TM ? fa + o * 16 * kXRow : fb + (o - TM) * 16 * kXRow;
            const v8bf_x v = __builtin_bit_cast(v8bf_x, *(const v4u_x *)(buf + p * PART + off));
            if (o < TM) a[p][o < TM ? o : 0] = v; else b[p][o < TM ? 0 : o - TM] = v;
        }
    };
    v4f_x acc[TM][TN] = {};
    // Four blocks at a time: their large products into the sums, then the small
    // ones, smallest first, into four accumulators that start from zero and are
    // added to the sums behind the next four blocks' large products (by when the
    // last of them has left the matrix cores).  The group's next stage is split
    // beside the small products, a chunk of it at a time (a wave issues three VALU
    // instructions while one MFMA runs).
    constexpr int NB = TM * TN, NQ = NB / 4;
    static_assert(NB % 4 == 0 && (NQ == NC || NQ == 1) && !(HL && NQ != 1), "blocks");
    v4f_x t[4] = {};
    auto add = [&](int q) {
#pragma unroll
        for (int y = 0; y < 4; ++y) acc[(4 * q + y) / TN][(4 * q + y) % TN] += t[y];
        __builtin_amdgcn_sched_barrier(0);
    };
    auto mul = [&]() {
        constexpr int kSmall = 7;
        constexpr int kPart[kSmall][2] = {{2, 1}, {1, 2}, {2, 0}, {0, 2}, {1, 1}, {1, 0}, {0, 1}};
#pragma unroll
        for (int q = 0; q < NQ; ++q) {
#pragma unroll
            for (int y = 0; y < 4; ++y) {
                const int i = (4 * q + y) / TN, j = (4 * q + y) % TN;
                acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(b[0][j], a[0][i], acc[i][j], 0, 0, 0);
            }
            __builtin_amdgcn_sched_barrier(0);
            if (q > 0) add(q - 1);
#pragma unroll
            for (int s = 0; s < kSmall; ++s)
#pragma unroll
                for (int y = 0; y < 4; ++y) {
                    const int i = (4 * q + y) / TN, j = (4 * q + y) % TN;
                    t[y] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
                        b[kPart[s][0]][j], a[kPart[s][1]][i], s == 0 && !HL ? v4f_x{0, 0, 0, 0} : t[y], 0, 0, 0);
                }
#pragma unroll
            for (int c = 0; c < NC / NQ; ++c) split(q * (NC / NQ) + c);
#pragma unroll
            for (int x = 0; x < 4 * kSmall; ++x) {
                __builtin_amdgcn_sched_group_barrier(kSchedMfma, 1, 0);
                __builtin_amdgcn_sched_group_barrier(0x002, NQ == 1 ? 4 : 3, 0);
            }
            __builtin_amdgcn_sched_barrier(0);
        }
        if (!HL) add(NQ - 1);
    };
    // Ends a slot: this wave's LDS reads and writes are done, then the barrier
    // (loads of later stages stay in flight across it).  The scheduling barriers
    // keep the slot's MFMAs, which touch no memory, from moving past it: the
    // groups would take turns instead of running side by side.
    auto slot_end = [] {
        __builtin_amdgcn_sched_barrier(0);
        asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
        __builtin_amdgcn_sched_barrier(0);
    };
    // Beside the other group's stage n, which was in buffer `at`: reads the
    // fragments of stage n+1 from the next buffer, writes the parts of stage n+3
    // into this one and issues the loads of stage n+5, in turns (a wave issues
    // in order).  Past the last stage it reads and writes LDS that nobody uses.
    int at = 0;
    auto next = [&](int o) { return o == 2 * BUF ? 0 : o + BUF; };
    auto prep = [&](int n) {
#pragma unroll
        for (int i = 0; i < NC; ++i) {
            frags(lds + next(at), i);
            __builtin_amdgcn_sched_barrier(0);
            put(lds + at, i);
            load(i, n + 5);
            __builtin_amdgcn_sched_barrier(0);
        }
    };

    // Stages 0 and 2 (group 0) or 1 (group 1) into LDS; group 1's stage 3 split;
    // group 0's stage 4 loaded.
#pragma unroll
    for (int i = 0; i < NC; ++i) {
        if (grp == 0 && rag) load_short(i); else load(i, grp);
    }
#pragma unroll
    for (int i = 0; i < NC; ++i) {
        split(i);
        load(i, grp + 2);
        put(lds + grp * BUF, i);
    }
#pragma unroll
    for (int i = 0; i < NC; ++i) {
        split(i);
        if (grp == 0) {
            put(lds + 2 * BUF, i);
            load(i, 4);
        }
    }
    slot_end();
    if (grp == 0) {
#pragma unroll
        for (int i = 0; i < NC; ++i) frags(lds, i);
    }
    slot_end();
    if (grp == 1) {
        prep(0);
        at = next(at);
        slot_end();
    }
    for (int n = grp; n < stages; n += 2) {
        mul();
        at = next(at);
        slot_end();
        if (n + 1 >= stages) break;
        prep(n + 1);
        at = next(at);
        slot_end();
    }

    if constexpr (HL) add(0);
    // The groups exchange halves of their partial tiles: group 0 keeps rows
    // blocks [0, TM/2) of each wave's part, group 1 the others.
    constexpr int TH = TM / 2;
    v4f_x *ex = (v4f_x *)lds;
#pragma unroll
    for (int i = 0; i < TH; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j)
            ex[(i * TN + j) * kXThreads + tid] = grp == 0 ? acc[TH + i][j] : acc[i][j];
    __syncthreads();
    v4f_x out[TH][TN];
    unsigned odd = 0;  // blocks with a sum that is not finite, one bit each
#pragma unroll
    for (int i = 0; i < TH; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j) {
            const v4f_x o = ex[(i * TN + j) * kXThreads + (tid ^ kXGroup)];
            const v4f_x mine = grp == 0 ? acc[i][j] : acc[TH + i][j];
            bool bad = false;
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                const float v = mine[q] + o[q];
                bad = bad || (__float_as_uint(v) & 0x7F800000u) == 0x7F800000u;
                out[i][j][q] = v * kXUnscale;
            }
            odd |= (unsigned)(__builtin_amdgcn_ballot_w64(bad) != 0) << (i * TN + j);
        }
    const int mw = m0 + wm * WTM + grp * TH * 16, nw = n0 + wn * WTN;
    if (odd) {
        // Those blocks again on v_mfma_f32_16x16x4_f32, operands from memory, 16 k
        // a step (lane group c takes k 4c..4c+3 of it, one per instruction), the
        // next step's loads in flight beside one's products.
        constexpr int ND = TH + TN;
        const float *p[ND];
#pragma unroll
        for (int d = 0; d < ND; ++d) {
            const int64_t r = (d < TH ? mw + 16 * d : nw + 16 * (d - TH)) + fr;
            p[d] = d < TH ? A + (r < g.M ? r : g.M - 1) * g.rsa : B + (r < g.N ? r : g.N - 1) * g.rsb;
        }
        const int wsteps = g.K / 16;
        auto fetch = [&](int t, float (&v)[ND][4]) {  // past the last whole step, that step again
            const int64_t k = (int64_t)(t < wsteps ? t : wsteps - 1) * 16 + 4 * fc;
#pragma unroll
            for (int d = 0; d < ND; ++d) {
                if (d < TH ? AK : BK) {
                    const v4f_x x = *(const v4f_xu *)(p[d] + k);
#pragma unroll
                    for (int e = 0; e < 4; ++e) v[d][e] = x[e];
                } else {
#pragma unroll
                    for (int e = 0; e < 4; ++e) v[d][e] = p[d][(k + e) * (d < TH ? g.ksa : g.ksb)];
                }
            }
            __builtin_amdgcn_sched_barrier(0);
        };
        v4f_x again[TH][TN] = {};
        auto mul4 = [&](const float (&v)[ND][4]) {
#pragma unroll
            for (int e = 0; e < 4; ++e)
#pragma unroll
                for (int i = 0; i < TH; ++i)
#pragma unroll
                    for (int j = 0; j < TN; ++j)
                        again[i][j] = __builtin_amdgcn_mfma_f32_16x16x4f32(v[TH + j][e], v[i][e],
                                                                           again[i][j], 0, 0, 0);
            __builtin_amdgcn_sched_barrier(0);
        };
        float v0[ND][4], v1[ND][4];
        if (wsteps > 0) fetch(0, v0);
        for (int t = 0; t < wsteps; t += 2) {
            fetch(t + 1, v1);
            mul4(v0);
            if (t + 1 >= wsteps) break;
            fetch(t + 2, v0);
            mul4(v1);
        }
        if (g.K % 16 != 0) {  // the last, zeros past K
#pragma unroll
            for (int d = 0; d < ND; ++d)
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    const int64_t k = (int64_t)wsteps * 16 + 4 * fc + e;
                    v0[d][e] = k < g.K ? p[d][k * (d < TH ? g.ksa : g.ksb)] : 0.0f;
                }
            mul4(v0);
        }
#pragma unroll
        for (int i = 0; i < TH; ++i)
#pragma unroll
            for (int j = 0; j < TN; ++j)
                if (odd >> (i * TN + j) & 1) out[i][j] = again[i][j];
    }
#pragma unroll
    for (int i = 0; i < TH; ++i) {
        const int row = mw + 16 * i + fr;
#pragma unroll
        for (int j = 0; j < TN; ++j) {
            const int col = nw + 16 * j + 4 * fc;
            if (row >= g.M || col >= g.N) continue;
            const float v[4] = {out[i][j][0], out[i][j][1], out[i][j][2], out[i][j][3]};
            float f[4] = {0, 0, 0, 0};
            if (ep.fused) {
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    const int c = col + e < g.N ? col + e : g.N - 1;
                    f[e] = fused_bias<false>(ep, ep.axis ? c : row);
                }
            }
            store4<EpiKind::F32, float, StPol::Plain>(ep, zb, row, col, g.N, v, nullptr, nullptr, f);
        }
    }
}

template <int BM, int BN, bool HL, int WPE>
static hipError_t f32x_go(const SmallArgs &g, const EpiParams &ep, hipStream_t stream) {
    const int64_t tiles = ((int64_t)(g.M + BM - 1) / BM) * ((g.N + BN - 1) / BN);
    if (tiles * kXThreads > UINT32_MAX) return hipErrorInvalidValue;
    const dim3 grid((unsigned)tiles, (unsigned)g.batch), block(kXThreads);
    const bool ak = g.ksa == 1, bk = g.ksb == 1;
    if (ak && bk)
        hipLaunchKernelGGL((f32x_kernel<BM, BN, true, true, HL, WPE>), grid, block, 0, stream, g, ep);
    else if (ak)
        hipLaunchKernelGGL((f32x_kernel<BM, BN, true, false, HL, WPE>), grid, block, 0, stream, g, ep);
    else if (bk)
        hipLaunchKernelGGL((f32x_kernel<BM, BN, false, true, HL, WPE>), grid, block, 0, stream, g, ep);
    else
        hipLaunchKernelGGL((f32x_kernel<BM, BN, false, false, HL, WPE>), grid, block, 0, stream, g, ep);
    return hipGetLastError();
}

bool f32x_fits(int64_t M, int64_t N) {
    return ((M + 63) / 64) * ((N + 63) / 64) <= (int64_t)UINT32_MAX / kXThreads;
}

hipError_t launch_f32x(const SmallArgs &g, const EpiParams &ep, bool fine, int cus,
                       hipStream_t stream) {
    if (g.M < 1 || g.N < 1 || g.K < 1 || g.batch < 1 || g.batch > kMaxGridZ ||
        ep.kind != EpiKind::F32)
        return hipErrorInvalidValue;
    // 128 x 128 tiles, one per CU, against 64 x 64 ones, two per CU at a time: a round
    // of large tiles takes about 3 times a round of small ones (2048^3: 110 us in
    // one round against 142 in four; 1536 x 1000 x 1536 50 in one against 53 in three;
    // 3000 x 2000 x 3000 285 in three against 298 in nine; 2048 x 2048 x 2049, whose 272
    // large tiles take two rounds: 185 against 161 in five; 1024^3, a quarter of the
    // CUs: 46 against 22).
    const int64_t c = cus > 0 ? cus : 256;
    auto rounds = [&](int64_t t) {
        return (((g.M + t - 1) / t) * ((g.N + t - 1) / t) * g.batch + c - 1) / c;
    };
    // `fine` tiles of one round are alone on their CU and take the registers of two
    // waves per SIMD (with four, the loop's addresses go through scratch memory:
    // 2200 x 800 x 130 with A column-major 24.6 us against 17.7).
    if (fine)
        return rounds(64) == 1 ? f32x_go<64, 64, true, 2>(g, ep, stream)
                               : f32x_go<64, 64, true, 4>(g, ep, stream);
    if (3 * rounds(128) <= rounds(64))
        return f32x_go<128, 128, false, 2>(g, ep, stream);
    return f32x_go<64, 64, false, 4>(g, ep, stream);
}

}  // namespace gk
