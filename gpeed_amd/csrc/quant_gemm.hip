// Products of many tokens over raw GGUF rows on the fp16 matrix cores
// (gfx950): Y[t][j] = sum_i W[j][i] X[t][i] for every block format, F16 and
// BF16 (F32 rows keep dot_f32's order, quant_rows.hip).
//
// Operands. A weight (at most 19 significant bits in every block format but
// Q2_K, whose weights are rounded to float32) times a power of two of its row
// is an fp16 hi plus an fp16 lo; F16 and BF16 weights need the hi alone. A
// float32 activation times a power of two of its token is hi plus lo as well
// (22 bits). A product is then three MFMAs, hi hi + hi lo + lo hi (two for
// F16 and BF16), where the fp32 MFMA has a sixteenth of the rate. The lo lo
// term left out is below 2^-22 of the product.
//
// Error against float64 (2-norm, 6144 columns): 2.5e-7 at 509 tokens (2.1e-7
// F16, BF16) where the fp32 MFMA GEMM has 1.4e-6 (it rounds its sums every 4
// columns, this path every 32), 1.7e-7 at 16 tokens where the 8-token slices
// have 2.0e-7.
//
// Measured, 6144 x 6144, us before (quant_rows.hip) and now:
//   tokens     8        20       64       256      509      1024
//   Q8_0    55 / 25  118 / 30  154 / 40  285 / 93  500 / 165  860 / 285
//   Q3_K    53 / 31  115 / 35  152 / 45  306 / 100 515 / 191  917 / 350
//   F16     75 / 25  131 / 29  149 / 37  285 / 77  483 / 134  848 / 225
// No single cost bounds the large sizes: of 376 us at 1024 tokens (Q3_K, 8 tiles), two
// of the three MFMAs take 83, the decode 29, the X reads from LDS 43, the
// barriers 34 (each left out alone).
//
// Non-finite values: every result that does not come out finite is summed
// again weight by weight in float32, so infinities and NaNs give what the
// float32 product gives.
#include "iq3_common.h"
#include "iq3_kernels.h"
#include "quant_decode.h"

#include <algorithm>
#include <climits>

namespace gpeed {

namespace {

typedef _Float16 half8_t __attribute__((ext_vector_type(8)));
typedef _Float16 half2v_t __attribute__((ext_vector_type(2)));
typedef float float2v_t __attribute__((ext_vector_type(2)));

constexpr int kBadRow = INT_MIN;  // in place of a scale exponent: the token holds a non-finite value
constexpr int kChunk = 128;       // columns of a chunk: one 32-weight sub-block for each lane group of 16
constexpr int kMaxIn = 1 << 20;    // (128 rows stay below 2 GiB)
constexpr int kFrag = 1024;       // bytes of one MFMA operand: 64 lanes of 8 fp16

// X in operand order. Fragment (token tile of 16, chunk, step s < 4, part):
// lane 16 k + i holds X[16 tile + i][128 chunk + 32 k + 8 s .. + 7], hi (part
// 0) or lo (part 1). Tokens past n_tok and columns past in_dim are zeros, a
// token with a non-finite value too (xexp = kBadRow). xexp[t]: the power of
// two token t was multiplied by. One workgroup per token; CPT > 0: the row is
// at most 256 CPT runs of 8 and stays in registers, read once.
template <int CPT>
__global__ __launch_bounds__(256) void k_prep_frag(const float* __restrict__ X, int n_tok, int in_dim, int n_chunk,
                                                   uint8_t* __restrict__ xf, int* __restrict__ xexp) {
    const int t = blockIdx.x, tid = threadIdx.x;
    const int n8 = t < n_tok ? in_dim >> 3 : 0;
    const u32x4_t* xr = reinterpret_cast<const u32x4_t*>(X + (size_t)min(t, n_tok - 1) * in_dim);
    __shared__ float red[4];
    float v[CPT > 0 ? CPT : 1][8];
    auto load8 = [&](int g, float (&o)[8]) {
        const u32x4_t a = xr[2 * g], b = xr[2 * g + 1];
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            o[i] = __uint_as_float(a[i]);
            o[4 + i] = __uint_as_float(b[i]);
        }
    };
    float mx = 0.0f;
    auto fold = [&](const float (&o)[8]) {
#pragma unroll
        for (int i = 0; i < 8; ++i) {
            const float a = fabsf(o[i]);
            mx = a < __builtin_inff() ? fmaxf(mx, a) : __builtin_inff();  // (a NaN or infinity stays: fmaxf with inf)
        }
    };
    if constexpr (CPT > 0) {
#pragma unroll
        for (int p = 0; p < CPT; ++p) {
            const int g = tid + 256 * p;
            if (g < n8) {
                load8(g, v[p]);
            } else {
#pragma unroll
                for (int i = 0; i < 8; ++i) v[p][i] = 0.0f;
            }
        }
#pragma unroll
        for (int p = 0; p < CPT; ++p) fold(v[p]);
    } else {
        for (int g = tid; g < n8; g += 256) {
            load8(g, v[0]);
            fold(v[0]);
        }
    }
    mx = wave_max(mx);
    if ((tid & 63) == 0) red[tid >> 6] = mx;
    __syncthreads();
    mx = fmaxf(fmaxf(red[0], red[1]), fmaxf(red[2], red[3]));
    const bool bad = !(mx < __builtin_inff());
    const int sc = pow2_scale_of_max(mx);
    if (tid == 0) xexp[t] = bad ? kBadRow : sc;
    auto store8 = [&](int g, const float (&o)[8]) {
        u32x4_t hi, lo;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const float a = bad ? 0.0f : ldexpf(o[2 * i], sc), b = bad ? 0.0f : ldexpf(o[2 * i + 1], sc);
            const half2v_t h = {(_Float16)a, (_Float16)b};
            const half2v_t l = {(_Float16)(a - (float)h[0]), (_Float16)(b - (float)h[1])};
            hi[i] = __builtin_bit_cast(uint32_t, h);
            lo[i] = __builtin_bit_cast(uint32_t, l);
        }
        // run g: chunk g / 16, lane group (g / 4) % 4, step g % 4
        uint8_t* d = xf + ((((size_t)(t >> 4) * n_chunk + (g >> 4)) * 4 + (g & 3)) * 2) * kFrag +
                     (((g >> 2) & 3) * 16 + (t & 15)) * 16;
        *reinterpret_cast<u32x4_t*>(d) = hi;
        *reinterpret_cast<u32x4_t*>(d + kFrag) = lo;
    };
    if constexpr (CPT > 0) {
#pragma unroll
        for (int p = 0; p < CPT; ++p)
            if (tid + 256 * p < n_chunk * 16) store8(tid + 256 * p, v[p]);
    } else {
        for (int g = tid; g < n_chunk * 16; g += 256) {
            if (g < n8) {
                load8(g, v[0]);
            } else {
#pragma unroll
                for (int i = 0; i < 8; ++i) v[0][i] = 0.0f;
            }
            store8(g, v[0]);
        }
    }
}

// Largest |weight| / |d| of a format, rounded up to a power of two (log2).
template <int DT>
constexpr int unit_bits() {
    return DT == kDtQ8_0 ? 7 : DT == kDtQ6_K || DT == kDtIQ4_XS ? 12 : DT == kDtQ2_K ? 6 : DT == kDtQ3_K ? 7
           : DT == kDtIQ2_S ? 8 : 9;
}

// b with every |weight| of a loaded sub-block below 2^b (fp16 d of exponent
// field E: |d| < 2^(E - 14); a non-finite scale counts as the largest one).
template <int DT>
__device__ __forceinline__ int sub_bound(const Sub<DT>& r) {
    if constexpr (DT == kDtBF16) {
        uint32_t m = 0;
#pragma unroll
        for (int i = 0; i < 16; ++i) m = max(m, max(r.w[i] & 0x7FFFu, (r.w[i] >> 16) & 0x7FFFu));
        return (int)min(m >> 7, 254u) - 126;
    } else {
        uint32_t m;
        if constexpr (DT == kDtQ8_0) m = r.w[8];
        else if constexpr (DT == kDtQ6_K) m = r.w[16] >> 16;
        else if constexpr (DT == kDtQ2_K) m = max(r.w[9] & 0x7FFFu, (r.w[9] >> 16) & 0x7FFFu);
        else if constexpr (DT == kDtQ3_K) m = r.w[17];
        else m = r.w[0];
        return (int)min((m >> 10) & 31u, 30u) - 14 + unit_bits<DT>();
    }
}

// One result in float32, weight by weight, over the wavefront's lanes.
template <int DT>
__device__ float dot_row(const uint8_t* __restrict__ row, const float* __restrict__ x, int in_dim,
                         const Tables<DT>& tb, int lane) {
    float acc = 0.0f;
    for (int s = lane; s < in_dim / 32; s += 64) {
        int sb;
        const uint8_t* blk = sub_block<DT>(row, s, sb);
        Sub<DT> r;
        load_sub<DT, true>(blk, sb, r);
        float y[32];
        decode_sub<DT>(r, sb, tb, 1.0f, y);
#pragma unroll
        for (int e = 0; e < 32; ++e) acc = fmaf(y[e], x[32 * s + e], acc);
    }
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) acc += __shfl_xor(acc, off);
    return acc;
}

// The four 8-weight operands (hi, and lo where the format has one) of a
// loaded sub-block, its weights times ds.
template <int DT>
struct Wops {
    static constexpr int kParts = DT == kDtF16 || DT == kDtBF16 ? 1 : 2;
    half8_t v[kParts][4];
};
// a - (float)(low or high half of h) in one instruction
template <int HI>
__device__ __forceinline__ float sub_half(float a, uint32_t h) {
    float d;
    if constexpr (HI) asm("v_fma_mix_f32 %0, %1, -1.0, %2 op_sel:[1,0,0] op_sel_hi:[1,0,0]" : "=v"(d) : "v"(h), "v"(a));
    else asm("v_fma_mix_f32 %0, %1, -1.0, %2 op_sel_hi:[1,0,0]" : "=v"(d) : "v"(h), "v"(a));
    return d;
}
template <int DT>
__device__ __forceinline__ void w_operands(const Sub<DT>& r, int sb, const Tables<DT>& tb, float ds, Wops<DT>& o) {
    if constexpr (DT == kDtF16) {
#pragma unroll
        for (int s = 0; s < 4; ++s) {
            const u32x4_t w = {r.w[4 * s], r.w[4 * s + 1], r.w[4 * s + 2], r.w[4 * s + 3]};
            o.v[0][s] = __builtin_bit_cast(half8_t, w);
        }
    } else {
        float y[32];
        decode_sub<DT>(r, sb, tb, ds, y);
#pragma unroll
        for (int s = 0; s < 4; ++s) {
            u32x4_t hi, lo;
#pragma unroll
            for (int k = 0; k < 4; ++k) {
                const float2v_t v = {y[8 * s + 2 * k], y[8 * s + 2 * k + 1]};
                hi[k] = __builtin_bit_cast(uint32_t, __builtin_convertvector(v, half2v_t));
                if constexpr (Wops<DT>::kParts == 2) {
                    const float2v_t l = {sub_half<0>(v[0], hi[k]), sub_half<1>(v[1], hi[k])};
                    lo[k] = __builtin_bit_cast(uint32_t, __builtin_convertvector(l, half2v_t));
                }
            }
            o.v[0][s] = __builtin_bit_cast(half8_t, hi);
            if constexpr (Wops<DT>::kParts == 2) o.v[1][s] = __builtin_bit_cast(half8_t, lo);
        }
    }
}

// 16 bytes a lane from global memory straight into LDS (the wavefront's 1 KiB at dst)
__device__ __forceinline__ void load_lds16(const uint8_t* src, uint8_t* dst) {
    __builtin_amdgcn_global_load_lds(src, dst, 16, 0, 0);
}


// the same from a buffer (past its end: zeros)
__device__ __forceinline__ void buffer_lds16(__amdgpu_buffer_rsrc_t rs, uint8_t* dst, uint32_t off) {
    __builtin_amdgcn_raw_ptr_buffer_load_lds(rs, dst, 16, (int)off, 0, 0, 0);
}
constexpr bool kWideLds = false;

// s_waitcnt vmcnt(N) lgkmcnt(0)
template <int N>
__device__ __forceinline__ void wait_vm() {
    static_assert(N >= 0 && N < 64, "vmcnt");
    __builtin_amdgcn_s_waitcnt((N & 15) | (7 << 4) | ((N >> 4) << 14));
}

// How a wavefront's 32 rows reach it. The block formats' bytes are copied to
// LDS, kGroup chunks (256 columns; Q8_0: 128) at a time: the 16-byte segments
// that cover a row's kBytes, consecutive lanes on consecutive segments, in
// kLoads copies of 1 KiB (a lane reading its own fields from memory touches
// sixteen rows with every load: 28 loads of a 256-column group took 135 of
// 425 us at 1024 tokens, 6144 x 6144, Q3_K). F16 and BF16 sub-blocks are 64
// contiguous bytes, four lanes side by side, and are loaded as they are.
template <int DT>
struct Stage {
    static constexpr bool kOn = DT != kDtF16 && DT != kDtBF16;
    static constexpr int kGroup = Fmt<DT>::kElems == 256 ? 2 : 1;
    static constexpr int kBytes = kGroup * kChunk / Fmt<DT>::kElems * Fmt<DT>::kBytes;
    static constexpr int kSegs = (kBytes + 14 + 15) / 16;  // (rows start at even addresses)
    static constexpr int kLoads = kOn ? (32 * kSegs + 63) / 64 : 0;
};

constexpr int kPerCu = 2;  // workgroups per CU that LDS and registers allow

// Tile of one workgroup: four wavefronts of 32 rows, 16 NT tokens, SPS steps
// of X a stage.
template <int DT, int NT>
struct SplitTile {
    static constexpr int kSps = NT > 4 ? 1 : NT == 4 ? 2 : 4;  // steps of X a stage
    static constexpr int kXb = NT >= 4 ? 3 : 2;                 // stages of X in LDS
    static constexpr int kStage = NT * kSps * 2 * kFrag;
    static constexpr int kCopies = (kStage / kFrag + 3) / 4;  // copies of a stage per wavefront
    static constexpr int kWBuf = Stage<DT>::kOn ? Stage<DT>::kLoads * 1024 : 16;
    // row groups in LDS per wavefront: two for few tokens, where they fit
    static constexpr int kWb = NT <= 2 && 8 * kWBuf + kXb * kStage + (int)sizeof(Tables<DT>) <= 80 * 1024 ? 2 : 1;
    static_assert(4 * kWb * kWBuf + kXb * kStage + (int)sizeof(Tables<DT>) <= 80 * 1024, "LDS of kPerCu workgroups");
};

// A workgroup of four wavefronts takes 128 rows x 16 NT tokens over the
// chunks of its K split: wavefront w rows 32 w .. + 31 for all tokens. A lane
// loads and decodes the sub-block of its row and lane group straight into
// operand registers, once per tile; the rows' bytes (each wavefront's own) and
// the X fragments (shared, double buffered) reach LDS by direct copies. Several
// workgroups share a CU, so one decodes or waits while the MFMAs of another
// run. n_split > 1: the split's sums go to part ([split][token][row], scaled)
// and k_sum_splits adds them.
//
// Row scale: the first chunk's bound with two bits to spare; where a later
// chunk passes it, the row's accumulators are brought down with it (an exact
// power of two; rare, as the scales of a row lie close together).
template <int DT, int NT>
__global__ __launch_bounds__(256, kPerCu) void k_gemm_split(
    const uint8_t* __restrict__ w, uint32_t rb, int in_dim, int out_dim, const uint8_t* __restrict__ xf,
    const int* __restrict__ xexp, const float* __restrict__ X, int n_tok, float* __restrict__ Y, int ldy,
    float* __restrict__ part, int tiles_m, int n_split) {
    using T = SplitTile<DT, NT>;
    using G = Stage<DT>;
    constexpr int kE = Fmt<DT>::kElems, kB = Fmt<DT>::kBytes, kSub = kE / 32, SPS = T::kSps;
    __shared__ Tables<DT> tb;
    __shared__ __attribute__((aligned(16))) uint8_t xs[T::kXb][T::kStage];
    __shared__ __attribute__((aligned(16))) uint8_t wsm[4][T::kWb][T::kWBuf];
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int li = lane & 15, lk = lane >> 4;
    // consecutive work of one XCD (workgroup id % 8): all token tiles, then
    // all splits, of a row band, whose rows then stay in that XCD's L2
    int tn, tm, sp;
    {
        const int n = gridDim.x, id = blockIdx.x, x = id & 7, q = n >> 3, rem = n & 7;
        const int lin = x * q + min(x, rem) + (id >> 3);
        const int t = lin / tiles_m;
        tm = lin - t * tiles_m;
        tn = t / n_split;
        sp = t - tn * n_split;
    }
    const int n_chunk = (in_dim + kChunk - 1) / kChunk, n_sub = in_dim / 32, tt_all = (n_tok + 15) >> 4;
    const int c0 = (int)((long long)n_chunk * sp / n_split), c1 = (int)((long long)n_chunk * (sp + 1) / n_split);
    const int j0 = tn * 128 + 32 * wave;
    // rows of this lane's two sub-blocks (past out_dim: the last row), byte offsets from w
    uint32_t row[2];
#pragma unroll
    for (int r = 0; r < 2; ++r) row[r] = (uint32_t)min(j0 + 16 * r + li, out_dim - 1) * rb;

    // F16 / BF16: this lane's fields of chunk c (sub-blocks past K are zeroed where they are decoded)
    Sub<DT> raw[2];
    auto load_raw = [&](int c) {
        const int sbi = min(c * 4 + lk, n_sub - 1);
#pragma unroll
        for (int r = 0; r < 2; ++r) load_sub<DT, true>(w + row[r] + (size_t)(sbi / kSub) * kB, sbi % kSub, raw[r]);
    };
    // the block formats: group g of the rows. Bytes past the tensor read as
    // zeros (they are not used); w itself may start inside a 16-byte segment.
    const uint32_t lead = (uint32_t)(reinterpret_cast<uintptr_t>(w) & 15);
    // (to the end of the last bytes' dword: a dword past the range in part reads as zero)
    const auto rs = __builtin_amdgcn_make_buffer_rsrc(const_cast<uint8_t*>(w) - lead, 0,
                                                      (int)((lead + (uint32_t)out_dim * rb + 3) & ~3u), 0x00020000);
    uint32_t srow[G::kOn ? G::kLoads : 1];  // row offset of each copy's lane
    if constexpr (G::kOn) {
#pragma unroll
        for (int k = 0; k < G::kLoads; ++k)
            srow[k] = lead + (uint32_t)min(j0 + (lane + 64 * k) / G::kSegs, out_dim - 1) * rb;
    }
    auto copy_w = [&](int g) {
#pragma unroll
        for (int k = 0; k < G::kLoads; ++k) {
            const uint32_t off = ((srow[k] + (uint32_t)g * G::kBytes) & ~15u) + 16u * ((lane + 64 * k) % G::kSegs);
            buffer_lds16(rs, wsm[wave][g % T::kWb] + k * 1024, off);
        }
    };
    // stage st (SPS steps) of X: 2 SPS fragments per token tile, a quarter of them per wavefront
    auto copy = [&](int st) {
        constexpr int kPer = 4 / SPS;
        const int c = c0 + st / kPer, s0 = (st % kPer) * SPS;
        uint8_t* dst = xs[st % T::kXb];
#pragma unroll
        for (int k = 0; k < T::kCopies; ++k) {
            const int f = min(wave + 4 * k, 2 * NT * SPS - 1), u = f / (2 * SPS), v = f % (2 * SPS);  // token tile, fragment of its steps
            const int tt = min(tm * NT + u, tt_all - 1);
            load_lds16(xf + (((size_t)tt * n_chunk + c) * 8 + 2 * s0 + v) * kFrag + lane * 16, dst + f * kFrag);
        }
    };
    const int g0 = c0 / G::kGroup, g1 = (c1 - 1) / G::kGroup + 1;
    if constexpr (G::kOn) {
#pragma unroll
        for (int k = 0; k < T::kWb; ++k)
            if (g0 + k < g1) copy_w(g0 + k);
    } else {
        load_raw(c0);
    }
    const int stages = (c1 - c0) * (4 / SPS);
#pragma unroll
    for (int k = 0; k < T::kXb - 1; ++k)
        if (k < stages) copy(k);
    tb.load(tid, 256);
    float4_t acc[2][NT], accx[2][NT];
    constexpr bool kTwoAcc = NT <= 2;  // the cross terms in sums of their own (fewer roundings of the large sum)
#pragma unroll
    for (int r = 0; r < 2; ++r)
#pragma unroll
        for (int u = 0; u < NT; ++u) acc[r][u] = accx[r][u] = float4_t{0.0f, 0.0f, 0.0f, 0.0f};
    int cur[2] = {-100000, -100000}, we[2] = {0, 0};  // row li: the bound its scale allows, the scale's exponent
    bool fresh = false;  // the newest copies in flight are a row group's
    for (int c = c0; c < c1; ++c) {
        Wops<DT> op[2];
#pragma unroll
        for (int q = 0; q < 4 / SPS; ++q) {
            // this stage's X and, at a group's first stage, its rows have
            // arrived; the next stage's X and a row group copied in the stage
            // before (and not needed yet) may still be on their way: they are
            // the newest copies. Every wavefront's reads of the stage before
            // are done (lgkmcnt), so the next copy may take its buffer.
            const int st = (c - c0) * (4 / SPS) + q;
            constexpr int kAhead = (T::kXb - 2) * T::kCopies;
            asm volatile("" ::: "memory");
            if (st + T::kXb - 2 >= stages) wait_vm<0>();
            else if ((T::kWb == 2 || q != 0) && fresh) wait_vm<kAhead + G::kLoads>();
            else wait_vm<kAhead>();
            __builtin_amdgcn_s_barrier();
            asm volatile("" ::: "memory");
            fresh = false;
            if (st + T::kXb - 1 < stages) copy(st + T::kXb - 1);
            if (q == 0) {
                const int sbi = c * 4 + lk;
#pragma unroll
                for (int r = 0; r < 2; ++r) {
                    if constexpr (G::kOn) {
                        const int g = c / G::kGroup, in_g = (c % G::kGroup) * 4 + lk;  // sub-block of the group
                        const uint32_t mis = (lead + row[r] + (uint32_t)g * G::kBytes) & 15u;
                        load_sub<DT, kWideLds>(wsm[wave][g % T::kWb] + (16 * r + li) * (G::kSegs * 16) + mis +
                                                   (in_g / kSub) * kB, in_g % kSub, raw[r]);
                    }
                    if (sbi >= n_sub) raw[r] = Sub<DT>{};  // past K: all-zero fields are zero weights
                    if constexpr (DT != kDtF16) {
                        const int b = sub_bound<DT>(raw[r]);
                        if (__any(b > cur[r])) {
                            int m = max(b, __shfl_xor(b, 16));
                            m = max(m, __shfl_xor(m, 32));
                            const int old = we[r];
                            if (m > cur[r]) {
                                const bool first = cur[r] == -100000;
                                cur[r] = first ? m + 2 : m;
                                we[r] = min(max(15 - cur[r], -120), 120);
                            }
                            const int dn = we[r] - old;  // (any value on the first chunk: the sums are zero)
#pragma unroll
                            for (int u = 0; u < NT; ++u) {
#pragma unroll
                                for (int i = 0; i < 4; ++i) {
                                    acc[r][u][i] = ldexpf(acc[r][u][i], dn);
                                    if constexpr (kTwoAcc) accx[r][u][i] = ldexpf(accx[r][u][i], dn);
                                }
                            }
                        }
                    }
                    w_operands<DT>(raw[r], sbi % kSub, tb, __uint_as_float((uint32_t)(127 + we[r]) << 23), op[r]);
                }
                if constexpr (G::kOn) {
                    const int g = c / G::kGroup;
                    if ((c + 1 == c1 || (c + 1) / G::kGroup != g) && g + T::kWb < g1) {
                        // the group's last fields are in registers: the next one takes its place
                        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
                        copy_w(g + T::kWb);
                        fresh = true;
                    }
                } else {
                    if (c + 1 < c1) load_raw(c + 1);
                }
            }
            const uint8_t* xb = xs[st % T::kXb] + lane * 16;
#pragma unroll
            for (int s2 = 0; s2 < SPS; ++s2) {
                const int s = q * SPS + s2;
#pragma unroll
                for (int u = 0; u < NT; ++u) {
                    const half8_t xh = *reinterpret_cast<const half8_t*>(xb + (u * SPS + s2) * 2 * kFrag);
                    const half8_t xl = *reinterpret_cast<const half8_t*>(xb + ((u * SPS + s2) * 2 + 1) * kFrag);
                    auto& ax = kTwoAcc ? accx : acc;
#pragma unroll
                    for (int r = 0; r < 2; ++r)
                        ax[r][u] = __builtin_amdgcn_mfma_f32_16x16x32_f16(xl, op[r].v[0][s], ax[r][u], 0, 0, 0);
                    if constexpr (Wops<DT>::kParts == 2) {
#pragma unroll
                        for (int r = 0; r < 2; ++r)
                            ax[r][u] = __builtin_amdgcn_mfma_f32_16x16x32_f16(xh, op[r].v[1][s], ax[r][u], 0, 0, 0);
                    }
#pragma unroll
                    for (int r = 0; r < 2; ++r)
                        acc[r][u] = __builtin_amdgcn_mfma_f32_16x16x32_f16(xh, op[r].v[0][s], acc[r][u], 0, 0, 0);
                }
            }
        }
    }
    // D: tokens 4 lk .. + 3 of the token tile, row li of the row tile (a store
    // takes 16 consecutive rows of four tokens). A result that is not finite
    // (a non-finite weight or activation, or a sum past float32) is summed
    // again weight by weight.
    float* yp = n_split > 1 ? part + (size_t)sp * n_tok * ldy : Y;
    bool bad = false;
#pragma unroll
    for (int u = 0; u < NT; ++u) {
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const int t = (tm * NT + u) * 16 + 4 * lk + i;
            const int xe = xexp[min(t, n_tok - 1)];
#pragma unroll
            for (int r = 0; r < 2; ++r) {
                const int j = j0 + 16 * r + li;
                const bool in = j < out_dim && t < n_tok;
                float v = acc[r][u][i];
                if constexpr (kTwoAcc) v += accx[r][u][i];
                v = xe == kBadRow ? __builtin_nanf("") : ldexpf(v, -(we[r] + xe));
                if (in) yp[(size_t)t * ldy + j] = v;
                bad |= in && !(fabsf(v) < __builtin_inff());
            }
        }
    }
    if (n_split > 1 || !__any(bad)) return;
    // (every result of the wavefront's 32 rows looked at again: its own stores)
    for (int q = 0; q < 8 * NT; ++q) {
        const int t = (tm * NT + (q >> 3)) * 16 + 4 * lk + ((q >> 1) & 3), jq = j0 + 16 * (q & 1) + li;
        const bool in = jq < out_dim && t < n_tok;
        const float v = in ? Y[(size_t)t * ldy + jq] : 0.0f;
        for (uint64_t m = __ballot(!(fabsf(v) < __builtin_inff())); m; m &= m - 1) {
            const int src = __builtin_ctzll(m);
            const int j = __shfl(jq, src), tk = __shfl(t, src);
            const float d = dot_row<DT>(w + (size_t)j * rb, X + (size_t)tk * in_dim, in_dim, tb, lane);
            if (lane == 0) Y[(size_t)tk * ldy + j] = d;
        }
    }
}

// Y[t][j] = the splits' sums in split order; results that are not finite are
// summed again weight by weight, as in k_gemm_split. One wavefront per 64
// rows of a token.
template <int DT>
__global__ __launch_bounds__(256) void k_sum_splits(const float* __restrict__ part, int n_split, int n_tok, int out_dim,
                                                    float* __restrict__ Y, int ldy, const uint8_t* __restrict__ w,
                                                    size_t rb, int in_dim, const float* __restrict__ X) {
    __shared__ Tables<DT> tb;
    const int lane = threadIdx.x & 63;
    const int j = blockIdx.x * 256 + threadIdx.x, t = blockIdx.y;
    const int jc = min(j, out_dim - 1);
    float v = 0.0f;
#pragma unroll 4
    for (int s = 0; s < n_split; ++s) v += part[((size_t)s * n_tok + t) * ldy + jc];
    if (j < out_dim) Y[(size_t)t * ldy + j] = v;
    const uint64_t bad = __ballot(j < out_dim && !(fabsf(v) < __builtin_inff()));
    if (!__syncthreads_or(bad != 0)) return;
    tb.load(threadIdx.x, 256);
    __syncthreads();
    for (uint64_t m = bad; m; m &= m - 1) {
        const int jj = j - lane + __builtin_ctzll(m);
        const float d = dot_row<DT>(w + (size_t)jj * rb, X + (size_t)t * in_dim, in_dim, tb, lane);
        if (lane == 0) Y[(size_t)t * ldy + jj] = d;
    }
}

size_t align256(size_t b) { return (b + 255) / 256 * 256; }
size_t frag_bytes(int in_dim, int n_tok) {
    return (size_t)((n_tok + 15) / 16) * ((in_dim + kChunk - 1) / kChunk) * 8 * kFrag;
}
// Tokens of one pass: all of them, or as many multiples of 128 as keep X in
// operand order near 1 GiB (its size in float32).
int pass_tokens(int in_dim, int n_tok) {
    const size_t per = frag_bytes(in_dim, 16) / 16;
    const long long fit = (long long)((1ull << 30) / per) / 128 * 128;
    return (int)std::min<long long>(n_tok, std::min<long long>(std::max<long long>(fit, 128), 32768));
}

// The launch of one product: 16 nt tokens per workgroup and splits of K.
// Up to 64 tokens the least of 1, 2, 4 tiles that holds them, fewer where the
// tiles and splits would not make a workgroup for each of 256 CUs. Above, of
// 4, 6, 7 and 8 tiles the one with the least time: rounds of the kPerCu slots
// of 256 CUs times chunks of a split times about 1.5 + 0.78 nt us (measured,
// Q3_K: 4.6 at 4 tiles, 7.7 at 8), and the splits' sums written and read.
// 6144 rows (Q3_K, us with 8 tiles and with the choice): 96 tokens 6 tiles 60
// and 54, 200 tokens 7 tiles 98 and 92, 509 tokens 7 tiles 204 and 193, 1024
// tokens 7 tiles 372 and 351.
constexpr int kMaxSplit = 16;
struct RowsPlan {
    int nt, splits;
};
RowsPlan rows_plan(int in_dim, int out_dim, int n_tok) {
    const int n_chunk = (in_dim + kChunk - 1) / kChunk;
    const long long tn = ((long long)out_dim + 127) / 128, most = std::max(1, std::min(kMaxSplit, n_chunk / 2));
    const auto groups = [&](int nt) { return tn * ((n_tok + 16 * nt - 1) / (16 * nt)); };
    const auto splits = [&](int nt) {
        return (int)std::max<long long>(1, std::min<long long>(most, 256ll * kPerCu / groups(nt)));
    };
    if (n_tok <= 64 || groups(4) * most < 256) {
        int nt = n_tok <= 16 ? 1 : n_tok <= 32 ? 2 : 4;
        while (nt > 1 && groups(nt) * most < 256) nt /= 2;
        return {nt, splits(nt)};
    }
    RowsPlan best{8, 1};
    double least = 0.0;
    for (int nt : {8, 7, 6, 4}) {
        const int s = splits(nt);
        const double rounds = (double)((groups(nt) * s + 256 * kPerCu - 1) / (256 * kPerCu));
        const double us = rounds * ((n_chunk + s - 1) / s) * (1.5 + 0.78 * nt) +
                          (s > 1 ? 3.0 + 8e-6 * s * (double)n_tok * out_dim / 4.0 : 0.0);
        if (least == 0.0 || us < 0.97 * least) best = {nt, s}, least = us;
    }
    return best;
}

struct RowsWs {  // the workspace of one pass
    const uint8_t* xf;
    const int* xexp;
    float* part;
};

template <int DT, int NT>
hipError_t gemm_split_nt(const uint8_t* w, size_t rb, int in_dim, int out_dim, const RowsWs& ws, const float* X,
                         int n_tok, float* Y, int n_split, hipStream_t s) {
    // row slabs of at most 2^20 workgroups (32-bit grids) and 2 GiB (32-bit offsets)
    const int tm = (n_tok + 16 * NT - 1) / (16 * NT);
    const int slab = (int)std::max<long long>(
        1, std::min<long long>((1 << 20) / (tm * n_split), ((1ll << 31) - 64) / (128ll * (long long)rb)));  // row tiles
    for (int j = 0; j < out_dim;) {
        const int rows = (int)std::min<long long>(out_dim - j, 128ll * slab);
        const int tn = (rows + 127) / 128;
        const uint8_t* wj = w + (size_t)j * rb;
        float* pj = n_split > 1 ? ws.part + j : nullptr;
        hipLaunchKernelGGL((k_gemm_split<DT, NT>), dim3((unsigned)(tm * tn * n_split)), dim3(256), 0, s, wj,
                           (uint32_t)rb, in_dim, rows, ws.xf, ws.xexp, X, n_tok, Y + j, out_dim, pj, tm, n_split);
        hipError_t e = hipGetLastError();
        if (e == hipSuccess && n_split > 1) {
            hipLaunchKernelGGL((k_sum_splits<DT>), dim3((unsigned)((rows + 255) / 256), (unsigned)n_tok), dim3(256), 0,
                               s, pj, n_split, n_tok, rows, Y + j, out_dim, wj, rb, in_dim, X);
            e = hipGetLastError();
        }
        if (e != hipSuccess) return e;
        j += rows;
    }
    return hipSuccess;
}

template <int DT>
hipError_t rows_gemm_dt(const uint8_t* w, size_t rb, int in_dim, int out_dim, const float* X, int n_tok, float* Y,
                        uint8_t* ws, hipStream_t s) {
    const int pass = pass_tokens(in_dim, n_tok), n_chunk = (in_dim + kChunk - 1) / kChunk;
    const size_t fb = align256(frag_bytes(in_dim, pass));
    int* xexp = reinterpret_cast<int*>(ws + fb);
    const RowsWs r{ws, xexp, reinterpret_cast<float*>(ws + fb + align256((size_t)(pass + 15) / 16 * 16 * sizeof(int)))};
    const RowsPlan pl = rows_plan(in_dim, out_dim, n_tok);
    for (int t = 0; t < n_tok; t += pass) {
        const int n = std::min(pass, n_tok - t), pad = (n + 15) / 16 * 16;
        const float* Xt = X + (size_t)t * in_dim;
        float* Yt = Y + (size_t)t * out_dim;
        if (n_chunk * 16 <= 1024)
            hipLaunchKernelGGL((k_prep_frag<4>), dim3(pad), dim3(256), 0, s, Xt, n, in_dim, n_chunk, ws, xexp);
        else
            hipLaunchKernelGGL((k_prep_frag<0>), dim3(pad), dim3(256), 0, s, Xt, n, in_dim, n_chunk, ws, xexp);
        hipError_t e = hipGetLastError();
        if (e != hipSuccess) return e;
        switch (pl.nt) {
            case 1: e = gemm_split_nt<DT, 1>(w, rb, in_dim, out_dim, r, Xt, n, Yt, pl.splits, s); break;
            case 2: e = gemm_split_nt<DT, 2>(w, rb, in_dim, out_dim, r, Xt, n, Yt, pl.splits, s); break;
            case 4: e = gemm_split_nt<DT, 4>(w, rb, in_dim, out_dim, r, Xt, n, Yt, pl.splits, s); break;
            case 6: e = gemm_split_nt<DT, 6>(w, rb, in_dim, out_dim, r, Xt, n, Yt, pl.splits, s); break;
            case 7: e = gemm_split_nt<DT, 7>(w, rb, in_dim, out_dim, r, Xt, n, Yt, pl.splits, s); break;
            default: e = gemm_split_nt<DT, 8>(w, rb, in_dim, out_dim, r, Xt, n, Yt, pl.splits, s); break;
        }
        if (e != hipSuccess) return e;
    }
    return hipSuccess;
}

}  // namespace

// Where this path takes a product over. Its three launches cost 9-13 us
// however small the product; the slices and the fp32 MFMA GEMM of
// quant_rows.hip cost by the row length and the token count. Measured, every
// format (here Q3_K, slices or fp32 GEMM against this path, us): in_dim 2048,
// 1024 rows, 4 tokens 10.6 / 13.5, 5 tokens 14.5 / 13.7; in_dim 1024, 5
// tokens 12.1 / 12.9, 16 tokens 14.3 / 13.0; in_dim 512, 1024 rows, 16 to 1000
// tokens 10.3-20.5 / 12.8-28.7, 12288 rows, 96 tokens 29.3 / 27.8.
bool rows_gemm_takes(int in_dim, int out_dim, int n_tok) {
    if (in_dim < 1024) return n_tok >= 5 && (long long)n_tok * out_dim >= 1 << 20;
    return n_tok >= (in_dim < 2048 ? 9 : 5);
}

size_t rows_gemm_ws_bytes(int dtype, int in_dim, int out_dim, int n_tok) {
    if (dtype == kDtF32 || in_dim > kMaxIn || !rows_gemm_takes(in_dim, out_dim, n_tok)) return 0;
    const int pass = pass_tokens(in_dim, n_tok), ns = rows_plan(in_dim, out_dim, n_tok).splits;
    return align256(frag_bytes(in_dim, pass)) + align256((size_t)((pass + 15) / 16 * 16) * sizeof(int)) +
           (ns > 1 ? align256((size_t)ns * pass * out_dim * sizeof(float)) : 0);
}

hipError_t launch_rows_gemm(int dtype, const uint8_t* w, size_t rb, unsigned long long row0, int in_dim, int out_dim,
                            const float* X, int n_tok, float* Y, uint8_t* ws, hipStream_t s) {
    switch (dtype) {
        case kDtF16: return rows_gemm_dt<kDtF16>(w + (size_t)row0 * rb, rb, in_dim, out_dim, X, n_tok, Y, ws, s);
        case kDtBF16: return rows_gemm_dt<kDtBF16>(w + (size_t)row0 * rb, rb, in_dim, out_dim, X, n_tok, Y, ws, s);
        case kDtQ8_0: return rows_gemm_dt<kDtQ8_0>(w + (size_t)row0 * rb, rb, in_dim, out_dim, X, n_tok, Y, ws, s);
        case kDtQ2_K: return rows_gemm_dt<kDtQ2_K>(w + (size_t)row0 * rb, rb, in_dim, out_dim, X, n_tok, Y, ws, s);
        case kDtQ3_K: return rows_gemm_dt<kDtQ3_K>(w + (size_t)row0 * rb, rb, in_dim, out_dim, X, n_tok, Y, ws, s);
        case kDtQ6_K: return rows_gemm_dt<kDtQ6_K>(w + (size_t)row0 * rb, rb, in_dim, out_dim, X, n_tok, Y, ws, s);
        case kDtIQ3_XXS: return rows_gemm_dt<kDtIQ3_XXS>(w + (size_t)row0 * rb, rb, in_dim, out_dim, X, n_tok, Y, ws, s);
        case kDtIQ3_S: return rows_gemm_dt<kDtIQ3_S>(w + (size_t)row0 * rb, rb, in_dim, out_dim, X, n_tok, Y, ws, s);
        case kDtIQ2_S: return rows_gemm_dt<kDtIQ2_S>(w + (size_t)row0 * rb, rb, in_dim, out_dim, X, n_tok, Y, ws, s);
        case kDtIQ4_XS: return rows_gemm_dt<kDtIQ4_XS>(w + (size_t)row0 * rb, rb, in_dim, out_dim, X, n_tok, Y, ws, s);
        default: return hipErrorInvalidValue;
    }
}

}  // namespace gpeed
