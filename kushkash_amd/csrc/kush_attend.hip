// Attention of query rows over key / value rows in bf16 or fp16 for gfx950: what a prefill attends with, over
// an unpacked history and its own new rows, causal (a sequence's queries are its last keys) or not, one
// sequence length for a batch or ragged rows packed end to end. Reference contract: the varlen flash
// attention call of kushkash/vllm/backend.py:837-880 and the attention with log-sum-exp of
// kushkash/_ops.py:254-276.
//
// The path is a pair of matrix products with a softmax between: bound by the matrix cores, then by the
// VALU (the exponentials). Mapping:
//   - The G query heads of a kv head are folded into its query rows (row m = token m / G, head m % G), so K
//     and V are read once for all of them and a short chunk still fills a tile.
//   - A workgroup of NW waves takes 32 NW rows, 32 per wave, and walks the keys 64 at a time. K and V tiles
//     go to an LDS ring by buffer-to-LDS DMA, ST - 1 tiles ahead, one barrier per tile.
//   - S^T = K Q^T on 32x32x16 MFMA with Q^T in registers: a lane then holds 32 scores of one query row, so
//     the softmax needs one lane exchange per tile, and the scores' C layout is, key for key, the B operand
//     of O^T += V^T P^T (V^T by ds_read_b64_tr_b16): P goes from one product to the next in registers.
//   - The denominator sums P as rounded for the product (v_dot2, one per pair), and the running max is
//     exact, so a row's largest weight is 1, free of rounding: against 64 bits the output is as close as
//     torch's flash kernel's (1.84e-3 against 1.85e-3 at N(0, 2^2) keys, bf16); moving the max only when it
//     grows by 2^8 is 3 % faster and 10 % further off, and not taken.
//   - Two waves per SIMD (8 waves at D <= 128): one's exponentials run under the other's MFMAs.
// Measured (bf16, causal, device events): 2,048 tokens x 32 heads over 34,816 keys x 8 kv heads, D 128: 1,048 us,
// 1,082 TFLOP/s (1,081 us, 1,049 TFLOP/s on another card), where a large bf16 matrix product reaches 1,369 and torch's
// flash kernel 468.
#include <cmath>

#include "kush_common.h"
#include "kushkash_amd_attend.h"

namespace kush {

typedef float f16v __attribute__((ext_vector_type(16)));
typedef float f2 __attribute__((ext_vector_type(2)));
typedef __bf16 b8 __attribute__((ext_vector_type(8)));
typedef __bf16 b2 __attribute__((ext_vector_type(2)));
typedef _Float16 h2 __attribute__((ext_vector_type(2)));
typedef short s4 __attribute__((ext_vector_type(4)));
typedef short s8 __attribute__((ext_vector_type(8)));
typedef __attribute__((address_space(3))) s4 lds_s4;
typedef __attribute__((address_space(3))) void lds_void;

template <typename T>
__device__ __forceinline__ f16v mfma32(s8 a, s8 b, f16v c) {
    if constexpr (std::is_same<T, _Float16>::value)
        return __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(h8, a), __builtin_bit_cast(h8, b), c, 0, 0, 0);
    else
        return __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(b8, a), __builtin_bit_cast(b8, b), c, 0, 0, 0);
}

// two fp32 values rounded to T, packed (one v_cvt_pk)
template <typename T>
__device__ __forceinline__ uint32_t pack2(float a, float b) {
    if constexpr (std::is_same<T, _Float16>::value)
        return __builtin_bit_cast(uint32_t, __builtin_convertvector((f2{a, b}), h2));
    else
        return __builtin_bit_cast(uint32_t, __builtin_convertvector((f2{a, b}), b2));
}

// acc + both values of a packed pair, in fp32
template <typename T>
__device__ __forceinline__ float add_pair(uint32_t w, float acc) {
    if constexpr (std::is_same<T, _Float16>::value)
        return __builtin_amdgcn_fdot2(__builtin_bit_cast(h2, w), h2{(_Float16)1.0f, (_Float16)1.0f}, acc, false);
    else
        return __builtin_amdgcn_fdot2_f32_bf16(__builtin_bit_cast(b2, w), b2{(__bf16)1.0f, (__bf16)1.0f}, acc, false);
}

// Strides in elements; cu_q / cu_k (ragged rows: sequence b's rows start at cu[b], batch strides unused) or
// one (nq, nk) for every sequence. out is T, or fp32 (out_f32). Partials of split keys: part_o
// [split][query row][q head][D] unnormalized, part_ml [split][query row][q head][2] (max in log2 units, sum).
struct AttendArgs {
    const void *q, *k, *v;
    void* out;
    float* lse;
    int64_t q_batch, q_row, q_head, k_batch, k_row, k_head, v_batch, v_row, v_head, o_batch, o_row, o_head;
    int64_t lse_batch, lse_row, lse_head;
    const int32_t *cu_q, *cu_k;
    int nq, nk, H, G;
    float c;                 // scale log2 e
    int causal, out_f32;
    int chunk;               // key tiles a workgroup takes at most (0: all of them)
    int64_t total_q;         // query rows of all sequences
    float *part_o, *part_ml;
};

constexpr int KEYS = 64;     // keys per tile

// LDS: a stage holds a K and a V tile, rows of D elements in 16-byte chunks, chunk c of row r at position
// c ^ fk(r) (K) or c ^ fv(r) (V): the row-wise K reads (32 rows, one chunk column) and the transposing V reads
// (4 keys x 64 bytes per half wave) then cover the 64 banks evenly.
template <int D, int NW>
struct AttendTile {
    static constexpr int CPR = D / 8, BM = 32 * NW, TILE = KEYS * D * 2;
    static constexpr int ST = (D <= 128 && NW == 8) ? 3 : 2;
    static constexpr int NI = TILE / 1024 / NW;               // DMA instructions per wave and tile (K or V)
    static_assert(TILE % (1024 * NW) == 0, "whole DMA instructions per wave");
    __device__ static __forceinline__ int fk(int r) { return D == 64 ? (r >> 1) & 7 : r & 15; }
    __device__ static __forceinline__ int fv(int r) {
        return D == 64 ? (((r >> 1) & 1) << 2) | ((r >> 2) & 3) : ((r & 3) << 2) | ((r >> 2) & 3);
    }
};

// One sequence's rows and keys
struct Span {
    int T, N;                // query rows (tokens), keys
    int64_t q, k, v, o, lse; // element offsets of its first rows
    int64_t row0;            // its first query row among all
};

__device__ __forceinline__ Span span_of(const AttendArgs& a, int b) {
    if (a.cu_q != nullptr) {
        // wave-uniform, said so: the tiles' DMA descriptors are built from them in scalar registers
        const int x0 = __builtin_amdgcn_readfirstlane(a.cu_q[b]), x1 = __builtin_amdgcn_readfirstlane(a.cu_q[b + 1]);
        const int y0 = __builtin_amdgcn_readfirstlane(a.cu_k[b]), y1 = __builtin_amdgcn_readfirstlane(a.cu_k[b + 1]);
        return Span{x1 - x0, y1 - y0, x0 * a.q_row, y0 * a.k_row, y0 * a.v_row, x0 * a.o_row, x0 * a.lse_row, x0};
    }
    return Span{a.nq, a.nk, b * a.q_batch, b * a.k_batch, b * a.v_batch, b * a.o_batch, b * a.lse_batch,
                (int64_t)b * a.nq};
}

// key tiles that the rows of tile `tile` (bm rows) of a sequence see, and the splits they are cut into
__device__ __forceinline__ int key_tiles(const AttendArgs& a, const Span& s, int tile, int bm, int& nk) {
    const int rows = s.T * a.G;
    const int last = (min((tile + 1) * bm, rows) - 1) / a.G;
    nk = a.causal ? min(s.N, s.N - s.T + last + 1) : s.N;
    return (nk + KEYS - 1) / KEYS;
}
__device__ __forceinline__ int splits_of(const AttendArgs& a, int nt) { return a.chunk ? (nt + a.chunk - 1) / a.chunk : 1; }

// A 16-byte-per-lane load of 1 KB straight into LDS at `lds` (kush_decode.h, issue_page: m0 and its wait state)
__device__ __forceinline__ void dma_kb(uint32_t lds, uint32_t voff, u4 rsrc) {
#pragma clang diagnostic push
#pragma clang diagnostic ignored "-Winline-asm"
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tbuffer_load_dwordx4 %1, %2, 0 offen lds" ::"s"(lds), "v"(voff), "s"(rsrc)
                 : "memory", "m0");
#pragma clang diagnostic pop
}

// raw buffer descriptor of `bytes` bytes at p, in scalar registers
__device__ __forceinline__ u4 rows_desc(uint64_t p, uint32_t bytes) {
    return u4{(uint32_t)__builtin_amdgcn_readfirstlane((uint32_t)p),
              (uint32_t)__builtin_amdgcn_readfirstlane((uint32_t)(p >> 32) & 0xFFFFu),
              (uint32_t)__builtin_amdgcn_readfirstlane(bytes), 0x00020000u};
}

// vmcnt(N) and lgkmcnt(0): at most N DMAs outstanding, every LDS read of this wave done
template <int N>
__device__ __forceinline__ void wait_dma() {
    static_assert(N < 64, "vmcnt holds at most 63");
    __builtin_amdgcn_s_waitcnt((N & 15) | ((N >> 4) << 14) | (7 << 4));
    asm volatile("" ::: "memory");
}

// both halves' values of a query row folded: lanes l and l ^ 32 hold the same row
__device__ __forceinline__ float half_max(float x) {
    auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(x), false, false);
    return __builtin_fmaxf(__uint_as_float(r[0]), __uint_as_float(r[1]));
}
__device__ __forceinline__ float half_sum(float x) {
    auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(x), false, false);
    return __uint_as_float(r[0]) + __uint_as_float(r[1]);
}

__device__ __forceinline__ void store4(const AttendArgs& a, int64_t at, f4 v, _Float16) {
    *reinterpret_cast<u2*>((uint16_t*)a.out + at) = u2{pack2<_Float16>(v[0], v[1]), pack2<_Float16>(v[2], v[3])};
}
__device__ __forceinline__ void store4(const AttendArgs& a, int64_t at, f4 v, bf16_t) {
    *reinterpret_cast<u2*>((uint16_t*)a.out + at) = u2{pack2<bf16_t>(v[0], v[1]), pack2<bf16_t>(v[2], v[3])};
}
template <typename T>
__device__ __forceinline__ void emit4(const AttendArgs& a, int64_t at, f4 v) {
    if (a.out_f32)
        *reinterpret_cast<f4*>((float*)a.out + at) = v;
    else
        store4(a, at, v, T{});
}

// grid (Hkv * sequences, row tiles, splits), block 64 NW. Consecutive workgroups are the kv heads (and
// sequences) of one row tile: the dispatcher deals them to the 8 XCDs in turn, so the row tiles of one kv
// head tend to share an XCD's L2. The longest rows (the last tile) go first.
template <int D, typename T, int NW>
__global__ __launch_bounds__(NW * WAVE) void attend_kernel(const AttendArgs a) {
    using A = AttendTile<D, NW>;
    constexpr int KS = D / 16, DB = D / 32, ST = A::ST, NI = A::NI;
    __shared__ __align__(16) uint8_t ring[ST * 2 * A::TILE];
    const int lane = threadIdx.x & (WAVE - 1), w = __builtin_amdgcn_readfirstlane(threadIdx.x / WAVE);
    const int r32 = lane & 31, hh = lane >> 5;
    const int h = blockIdx.x % a.H, b = blockIdx.x / a.H;
    const int tile = gridDim.y - 1 - blockIdx.y, G = a.G;
    const Span s = span_of(a, b);
    const int rows = s.T * G;
    if (tile * A::BM >= rows) return;
    int nk;
    const int nt = key_tiles(a, s, tile, A::BM, nk), ns = splits_of(a, nt);
    if ((int)blockIdx.z >= ns) return;
    const int per = (nt + ns - 1) / ns, j0 = min(nt, per * (int)blockIdx.z), j1 = min(nt, j0 + per);

    const int first = tile * A::BM + w * 32, m = first + r32, mc = min(m, rows - 1);   // rows past the end: the last
    const int t = mc / G, g = mc - t * G;
    const int off = s.N - s.T;
    const int lim = a.causal ? off + t : s.N - 1;                        // the last key this lane's row sees
    const int wlo = a.causal ? off + min(first, rows - 1) / G : s.N - 1;   // and the wave's least and greatest
    const int whi = first >= rows ? -1 : (a.causal ? off + min(first + 31, rows - 1) / G : s.N - 1);

    s8 qf[KS];                                                           // B operand: row r32, dims 16 ks + 8 hh ..
    {
        const uint16_t* qp = (const uint16_t*)a.q + s.q + t * a.q_row + (int64_t)(h * G + g) * a.q_head + 8 * hh;
#pragma unroll
        for (int ks = 0; ks < KS; ++ks) qf[ks] = *reinterpret_cast<const s8*>(qp + 16 * ks);
    }
    const uint8_t* const kbase = (const uint8_t*)a.k + 2 * (s.k + h * a.k_head);
    const uint8_t* const vbase = (const uint8_t*)a.v + 2 * (s.v + h * a.v_head);
    const uint32_t krb = (uint32_t)(2 * a.k_row), vrb = (uint32_t)(2 * a.v_row);   // 64 of them fit 32 bits (host)
    uint32_t ko[NI], vo[NI];                                             // this lane's source offsets in a tile
#pragma unroll
    for (int i = 0; i < NI; ++i) {
        const int L = (w * NI + i) * WAVE + lane, r = L / A::CPR, p = L % A::CPR;
        ko[i] = r * krb + ((p ^ A::fk(r)) << 4);
        vo[i] = r * vrb + ((p ^ A::fv(r)) << 4);
    }
    const uint32_t lds0 = (uint32_t)(uintptr_t)(lds_void*)ring;
    // tile j into stage st: 2 NI instructions; rows past the keys (all of them past tile j1) lie outside the
    // buffer range, so they touch no memory and arrive as zeros
    const auto issue = [&](int j, int st) {
        const int left = j < j1 ? min(KEYS, nk - KEYS * j) : 0;
        const uint64_t ka = (uint64_t)(uintptr_t)(kbase + (int64_t)j * KEYS * krb);
        const uint64_t va = (uint64_t)(uintptr_t)(vbase + (int64_t)j * KEYS * vrb);
        const u4 kd = rows_desc(ka, left ? (left - 1) * krb + 2 * D : 0u);
        const u4 vd = rows_desc(va, left ? (left - 1) * vrb + 2 * D : 0u);
        const uint32_t base = lds0 + st * 2 * A::TILE + w * NI * 1024;
#pragma unroll
        for (int i = 0; i < NI; ++i) dma_kb(base + i * 1024, ko[i], kd);
#pragma unroll
        for (int i = 0; i < NI; ++i) dma_kb(base + A::TILE + i * 1024, vo[i], vd);
    };

    // LDS offsets: K chunk 2 ks + hh of row r32 (A operand); V^T pieces, where within a 16-lane group lane 4 k + c
    // supplies dims 4 c .. 4 c + 3 of key k and lane i receives dim i of the four keys: dims 32 db + lane % 32,
    // keys 8 half + 4 hh .. + 3, the keys that accumulator registers 4 half .. + 3 of this lane's scores stand for
    uint32_t kl[KS], vl[DB][2];
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) kl[ks] = r32 * (2 * D) + (((2 * ks + hh) ^ A::fk(r32)) << 4);
    {
        const int i16 = lane & 15, ds = (lane >> 4) & 1;
#pragma unroll
        for (int db = 0; db < DB; ++db)
#pragma unroll
            for (int half = 0; half < 2; ++half) {
                const int key = 8 * half + 4 * hh + (i16 >> 2);
                vl[db][half] = key * (2 * D) + (((4 * db + 2 * ds + ((i16 & 3) >> 1)) ^ A::fv(key)) << 4) + 8 * (i16 & 1);
            }
    }

    f16v o[DB];
#pragma unroll
    for (int db = 0; db < DB; ++db)
#pragma unroll
        for (int i = 0; i < 16; ++i) o[db][i] = 0.0f;
    float mr = -__builtin_inff(), l = 0.0f;                              // running max (log2 units), this half's sum

    __builtin_amdgcn_s_waitcnt(0x0F70);                                 // q is in: only DMAs count in vmcnt below
    asm volatile("" ::: "memory");
#pragma unroll
    for (int i = 0; i < ST - 1; ++i) issue(j0 + i, i);
    int st = 0;
    for (int j = j0; j < j1; ++j) {
        // tile j is in and, behind the barrier, in for every wave, and every wave has read tile j - 1, whose
        // stage takes tile j + ST - 1
        wait_dma<(ST - 2) * 2 * NI>();
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
        issue(j + ST - 1, st == 0 ? ST - 1 : st - 1);
        const uint8_t* const kt = ring + st * 2 * A::TILE;
        const uint8_t* const vt = kt + A::TILE;
        if (++st == ST) st = 0;
        if (KEYS * j > whi) continue;                                    // no row of this wave sees the tile
        f16v sc[2];                                                      // keys 32 kb + 8 (i / 4) + 4 hh + i % 4
#pragma unroll
        for (int kb = 0; kb < 2; ++kb) {
#pragma unroll
            for (int i = 0; i < 16; ++i) sc[kb][i] = 0.0f;
#pragma unroll
            for (int ks = 0; ks < KS; ++ks)
                sc[kb] = mfma32<T>(*reinterpret_cast<const s8*>(kt + kb * 64 * D + kl[ks]), qf[ks], sc[kb]);
        }
        if (KEYS * j + KEYS - 1 > wlo) {
#pragma unroll
            for (int kb = 0; kb < 2; ++kb)
#pragma unroll
                for (int i = 0; i < 16; ++i)
                    if (KEYS * j + 32 * kb + 8 * (i / 4) + 4 * hh + i % 4 > lim) sc[kb][i] = -__builtin_inff();
        }
        float mx = sc[0][0];
#pragma unroll
        for (int kb = 0; kb < 2; ++kb)
#pragma unroll
            for (int i = 0; i < 16; ++i) mx = __builtin_fmaxf(mx, sc[kb][i]);
        const float mn = __builtin_fmaxf(half_max(mx) * a.c, mr);
        // a row that has seen no key yet (a split's first tiles) keeps -inf; its weights are taken against 0
        const float mref = mn == -__builtin_inff() ? 0.0f : mn;
        if (__builtin_amdgcn_ballot_w64(mn != mr)) {                     // some row's max moved
            const float corr = __builtin_amdgcn_exp2f(mr - mref);
            l *= corr;
#pragma unroll
            for (int db = 0; db < DB; ++db) o[db] *= corr;
            mr = mn;
        }
        s8 p[4];                                                         // B operands of 16 keys each
        float sum = 0.0f;
#pragma unroll
        for (int kb = 0; kb < 2; ++kb)
#pragma unroll
            for (int e = 0; e < 2; ++e) {
                u4 wd;
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    wd[i] = pack2<T>(__builtin_amdgcn_exp2f(__builtin_fmaf(sc[kb][8 * e + 2 * i], a.c, -mref)),
                                     __builtin_amdgcn_exp2f(__builtin_fmaf(sc[kb][8 * e + 2 * i + 1], a.c, -mref)));
                    sum = add_pair<T>(wd[i], sum);
                }
                p[2 * kb + e] = __builtin_bit_cast(s8, wd);
            }
        l += sum;
#pragma unroll
        for (int s16 = 0; s16 < 4; ++s16)
#pragma unroll
            for (int db = 0; db < DB; ++db) {
                const s4 x = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s4*)(vt + s16 * 32 * D + vl[db][0]));
                const s4 y = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s4*)(vt + s16 * 32 * D + vl[db][1]));
                o[db] = mfma32<T>(__builtin_shufflevector(x, y, 0, 1, 2, 3, 4, 5, 6, 7), p[s16], o[db]);
            }
    }
    wait_dma<0>();                                                       // trailing (empty) DMAs: LDS is theirs until then
    if (m >= rows) return;
    l = half_sum(l);
    const int64_t head = h * G + g;
    if (ns > 1) {                                                        // a partial, for attend_merge_kernel
        const int64_t row = ((int64_t)blockIdx.z * a.total_q + s.row0 + t) * (a.H * G) + head;
        float* const op = a.part_o + row * D + 4 * hh;
#pragma unroll
        for (int db = 0; db < DB; ++db)
#pragma unroll
            for (int i = 0; i < 4; ++i)
                *reinterpret_cast<f4*>(op + 32 * db + 8 * i) = f4{o[db][4 * i], o[db][4 * i + 1], o[db][4 * i + 2], o[db][4 * i + 3]};
        if (hh == 0) *reinterpret_cast<f2*>(a.part_ml + 2 * row) = f2{mr, l};
        return;
    }
    const float inv = 1.0f / l;
    const int64_t at = s.o + t * a.o_row + head * a.o_head + 4 * hh;
#pragma unroll
    for (int db = 0; db < DB; ++db)
#pragma unroll
        for (int i = 0; i < 4; ++i)
            emit4<T>(a, at + 32 * db + 8 * i,
                     f4{o[db][4 * i], o[db][4 * i + 1], o[db][4 * i + 2], o[db][4 * i + 3]} * inv);
    if (a.lse != nullptr && hh == 0)
        a.lse[s.lse + t * a.lse_row + head * a.lse_head] = (mr + __builtin_log2f(l)) * 0.69314718055994530942f;
}

// grid (Hkv * sequences, query rows / MERGE_ROWS), block 256: the splits of each row merged by log-sum-exp, in
// split order. D / 4 threads per row; rows of tiles that were not split have nothing to do here. Latency-bound:
// a batch of splits is loaded before the first of it is used.
constexpr int MERGE_ROWS = 32;
template <int D, typename T>
__global__ __launch_bounds__(256) void attend_merge_kernel(const AttendArgs a, int bm) {
    constexpr int B = 8;
    const int h = blockIdx.x % a.H, b = blockIdx.x / a.H, G = a.G, first = blockIdx.y * MERGE_ROWS;
    const Span s = span_of(a, b);
    const int rows = s.T * G;
    if (first >= rows) return;
    int nk;
    const int ns = splits_of(a, key_tiles(a, s, first / bm, bm, nk));       // bm is a multiple of MERGE_ROWS
    if (ns <= 1) return;
    const int d = 4 * ((int)threadIdx.x % (D / 4));
    const int64_t stride = a.total_q * (a.H * G);                           // rows of one split
#pragma unroll
    for (int i = 0; i < MERGE_ROWS / (256 / (D / 4)); ++i) {
        const int m = first + (int)threadIdx.x / (D / 4) + i * (256 / (D / 4));
        if (m >= rows) break;
        const int t = m / G;
        const int64_t head = h * G + m - t * G, row = (s.row0 + t) * (a.H * G) + head;
        float M = -__builtin_inff();
        for (int z0 = 0; z0 < ns; z0 += B) {
            float mz[B];
#pragma unroll
            for (int u = 0; u < B; ++u) mz[u] = a.part_ml[2 * (row + min(z0 + u, ns - 1) * stride)];
#pragma unroll
            for (int u = 0; u < B; ++u) M = __builtin_fmaxf(M, mz[u]);
        }
        const float mref = M == -__builtin_inff() ? 0.0f : M;
        float L = 0.0f;
        f4 acc = f4{0.0f, 0.0f, 0.0f, 0.0f};
        for (int z0 = 0; z0 < ns; z0 += B) {
            f2 ml[B];
            f4 v[B];
#pragma unroll
            for (int u = 0; u < B; ++u) {
                const int64_t at = row + min(z0 + u, ns - 1) * stride;
                ml[u] = *reinterpret_cast<const f2*>(a.part_ml + 2 * at);
                v[u] = *reinterpret_cast<const f4*>(a.part_o + at * D + d);
            }
#pragma unroll
            for (int u = 0; u < B; ++u) {
                if (z0 + u >= ns) break;
                const float f = __builtin_amdgcn_exp2f(ml[u][0] - mref);
                L += f * ml[u][1];
                acc += f * v[u];
            }
        }
        emit4<T>(a, s.o + t * a.o_row + head * a.o_head + d, acc * (1.0f / L));
        if (a.lse != nullptr && d == 0)
            a.lse[s.lse + t * a.lse_row + head * a.lse_head] = (M + __builtin_log2f(L)) * 0.69314718055994530942f;
    }
}

template <int D, typename T, int NW>
static int launch_attend(const AttendArgs& a, int64_t n_seqs, int max_q, int max_k, hipStream_t stream) {
    constexpr int BM = AttendTile<D, NW>::BM;
    const int64_t tiles = ((int64_t)max_q * a.G + BM - 1) / BM, nt = ((int64_t)max_k + KEYS - 1) / KEYS;
    const int64_t splits = a.chunk ? (nt + a.chunk - 1) / a.chunk : 1;
    if (tiles > 65535 || splits > 65535 || n_seqs * a.H > 0x7fffffff)
        return kush_fail(-2, "kush_attend: %lld row tiles x %lld splits are too many", (long long)tiles, (long long)splits);
    attend_kernel<D, T, NW><<<dim3((unsigned)(n_seqs * a.H), (unsigned)tiles, (unsigned)splits), dim3(NW * WAVE), 0, stream>>>(a);
    if (splits > 1)
        attend_merge_kernel<D, T><<<dim3((unsigned)(n_seqs * a.H), (unsigned)(((int64_t)max_q * a.G + MERGE_ROWS - 1) / MERGE_ROWS)),
                                    dim3(256), 0, stream>>>(a, BM);
    return kush_check_launch("kush_attend");
}

}  // namespace kush

using namespace kush;

extern "C" int kush_attend(int head_dim, int dtype, const void* q, const void* k, const void* v, void* out, float* lse,
                           const int64_t* strides, const int32_t* cu_q, const int32_t* cu_k, int32_t n_q, int32_t n_k,
                           int64_t total_q, int32_t n_seqs, int32_t hkv, int32_t group, float scale, int32_t causal,
                           int32_t out_f32, int32_t waves, int32_t chunk, float* part_o, float* part_ml, void* stream) {
    if (n_seqs < 0 || hkv <= 0 || group <= 0 || n_q <= 0 || n_k <= 0 || chunk < 0 || (cu_q == nullptr) != (cu_k == nullptr))
        return kush_fail(-2, "kush_attend: bad n_seqs %d / hkv %d / group %d / n_q %d / n_k %d / chunk %d", n_seqs, hkv,
                         group, n_q, n_k, chunk);
    if (!(scale > 0.0f) || !std::isfinite(scale)) return kush_fail(-2, "kush_attend: scale must be positive");
    if (causal && cu_q == nullptr && n_k < n_q) return kush_fail(-2, "kush_attend: causal needs n_k >= n_q");
    if (dtype != 1 && dtype != 2) return kush_fail(-1, "kush_attend: dtype code %d (1 fp16, 2 bf16)", dtype);
    if (chunk > 0 && chunk < ((int64_t)n_k + KEYS - 1) / KEYS && (part_o == nullptr || part_ml == nullptr))
        return kush_fail(-2, "kush_attend: split keys need the partial buffers");
    const int64_t* st = strides;
    uint64_t align = (uintptr_t)q | (uintptr_t)k | (uintptr_t)v | (uintptr_t)out;
    for (int i = 0; i < 9; ++i) align |= 2 * (uint64_t)st[i];
    for (int i = 9; i < 12; ++i) align |= (out_f32 ? 4 : 2) * (uint64_t)st[i];
    if (align & 15) return kush_fail(-2, "kush_attend: rows must be 16-byte aligned (pointers and strides)");
    if (st[4] < head_dim || st[7] < head_dim || st[4] > (1 << 23) || st[7] > (1 << 23))
        return kush_fail(-2, "kush_attend: bad key / value row strides %lld, %lld", (long long)st[4], (long long)st[7]);
    if (n_seqs == 0) return 0;
    const AttendArgs a{q,      k,      v,      out,    lse,    st[0],  st[1],  st[2],  st[3],
                       st[4],  st[5],  st[6],  st[7],  st[8],  st[9],  st[10], st[11], st[12],
                       st[13], st[14], cu_q,   cu_k,   n_q,    n_k,    hkv,    group,
                       (float)((double)scale * 1.4426950408889634), causal != 0, out_f32 != 0, chunk, total_q, part_o,
                       part_ml};
    const auto go = [&](auto dd, auto in) -> int {
        constexpr int D = decltype(dd)::value;
        using T = decltype(in);
        if constexpr (D < 256) {
            if (waves == 8) return launch_attend<D, T, 8>(a, n_seqs, n_q, n_k, (hipStream_t)stream);
        }
        return launch_attend<D, T, 4>(a, n_seqs, n_q, n_k, (hipStream_t)stream);
    };
    const auto by_dtype = [&](auto dd) -> int { return dtype == 1 ? go(dd, _Float16{}) : go(dd, bf16_t{}); };
    switch (head_dim) {
        case 64: return by_dtype(ic<64>{});
        case 128: return by_dtype(ic<128>{});
        case 256: return by_dtype(ic<256>{});
    }
    return kush_fail(-1, "kush_attend: unsupported head_dim %d (64, 128 or 256)", head_dim);
}
