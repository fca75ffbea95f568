// preq2 GEMM of a prompt chunk and of batches of more than 16 columns: Y[n][:]
// = preq2(W) x_n for any number of activation columns, each column bit for bit what the single-column GEMV
// gives on it (plan_preq2's K split and lane layout), so that a prompt run in
// chunks leaves the K/V rows and logits of one step per token.  The reference
// feeds a prompt one forward_token per token
// (asdsl/kernels/native/unified_engine.cpp:1339-1688); it has no such kernel.
//
// The int32 dots of a 32-element slice come from v_mfma_i32_16x16x32_i8 (16
// rows x 16 columns, exact in any order).  The fp32 steps per (row, column)
// are the single-column kernel's:
//   acc = fma(d, s*xs, acc); acc = fma(-(z*s), xu, acc)
// in 16 accumulators per K range (one per lane position of a row):
//   GS 32:  group g belongs to accumulator g mod 16;
//   GS 128: slice t of group g belongs to accumulator (g mod 4, t);
// which then fold as slot_sum does.  A wave takes the accumulators four at a
// time (class w: GS 32 groups with (g mod 16) / 4 = w, GS 128 groups with g
// mod 4 = w): 4 MFMAs and 4 accumulators per (row, column) and step, class
// after class, R_w = the class's in-row fold, and a K range's sum is
// (R_0 + R_1) + (R_2 + R_3); the K ranges add in order.
//
// What bounds it: the fp32 steps.  Per MFMA each lane forms 4 values with 4
// conversions, 4 products s*xs (one in four of them for GS 128) and 8 fused
// multiply-adds on the vector unit, 13-16 instructions of 4 cycles against 16
// matrix cycles; decoding (s, -z*s), unpacking weights and addresses add
// 5 to 8.  So the kernel keeps what it can off the
// vector unit:
//  - the MFMA's rows are the weight rows and its columns the activation
//    columns: a lane holds one column's (xs, xu) and four rows' (s, z), and
//    one unpacked weight operand serves CB column blocks;
//  - the workgroup's waves take different rows of the same columns, so the
//    activation operands and scales of a step are staged once in LDS for all
//    of them (two buffers, the next step's loads in flight while the current
//    one computes; one barrier per step);
//    Both are laid out in LDS so that no two lanes of an operand read share
//    a bank (as first written, 41 % of the cycles of a gate_up launch were
//    bank conflicts; 6 % are left, the operands' stores among them, whose two
//    halves of a unit fall on the same banks);
//  - each wave's 16-row weight tile goes through its own LDS area (one 16-byte
//    load per lane and step, read back as each MFMA's operand dwords).
// Measured at 517 columns: gate_up 16384x3072 g128 166 us (313 T int8
// operations a second; 18.5 vector instructions beside each MFMA, 70 % of the
// issue slots taken), down 3072x8192 g128 100 us, qkv 5120x3072 g32 73 us (22.7 beside
// each MFMA), o_proj 3072x3072 g32 46 us; 33 times a launch of the 16-column exact
// kernel would be 386, 281, 290 and 182 us.
#include <cstdlib>

#include "abi_util.hpp"
#include "device_common.hpp"

namespace asdsl {
namespace {

typedef int v4i32 __attribute__((ext_vector_type(4)));

constexpr int kGemmWaves = 4;
constexpr int kGemmThreads = kGemmWaves * kWave;
constexpr int kGemmRows = 16 * kGemmWaves;  // rows of a workgroup's tile

// LDS bytes per column block and step: 4 slices of int8 operands, then the
// scales (GS 32: 4 groups x 16 pairs; GS 128: one group's 16 pairs and the 4
// slice sums of 16 columns).
constexpr int kOpBytes = 4 * 512;
__host__ __device__ constexpr int scale_bytes(int gs) { return gs == 32 ? 512 : 128 + 256; }
// a wave's weight tile of one step: 4 bands x 256 bytes, spaced so that the
// 64 lanes of an operand read (4 bands x 4 rows x 4 dwords; rows 16 bytes
// apart for GS 32, 64 for GS 128) fall on different banks, and its (s, z) pairs
__host__ __device__ constexpr int band_stride(int gs) { return 256 + (gs == 32 ? 64 : 16); }
__host__ __device__ constexpr int wave_stage(int gs) { return 4 * band_stride(gs) + 256; }

// SPLIT: the workgroup's waves take one class each of the same 16 rows, with
// operands, scales and weights all in the wave's own LDS area and no barrier
// but the one per K range that adds the classes.  A quarter of the steps per
// wave and four times the workgroups, for column counts that leave the other
// form with about one wave per SIMD: its time is then the steps' memory
// latency, 0.6 to 0.8 us each (down 3072x8192 g128 at 24 columns: 13.2 us split,
// 37.8 not).
template <int GS, int CB, bool SPLIT>
__global__ __launch_bounds__(kGemmThreads, 2) void preq2_gemm_exact_kernel(
    const uint32_t* __restrict__ meta, const uint8_t* __restrict__ quant, const uint8_t* __restrict__ image,
    float* __restrict__ Y, int M, int K, int ncols, int KS, int NU, int nrt, int nct, int per_xcd) {
#pragma clang fp contract(off)
    constexpr int UPS = GS / 32;
    constexpr int kGroupBytes = GS * 2;            // a band's group: 4 rows x UPS 16-byte slices
    constexpr int kStepGroups = GS == 32 ? 4 : 1;  // groups of a step
    constexpr int kClassStride = GS == 32 ? 16 : 4;  // groups between a class's steps
    constexpr int kScale = scale_bytes(GS);
    constexpr int kBandStride = band_stride(GS);
    constexpr int kBuf = CB * (kOpBytes + kScale);
    constexpr int kOpUnits = CB * kOpBytes / 16;       // 16-byte units of a step's operands
    constexpr int kScaleUnits = CB * kScale / 16;
    constexpr int kLoaders = SPLIT ? kWave : kGemmThreads;  // threads that stage one operand buffer
    constexpr int kOpLoads = (kOpUnits + kLoaders - 1) / kLoaders;
    static_assert(kScaleUnits <= kLoaders, "one scale unit per thread");
    __shared__ __align__(16) uint8_t s_bufs[SPLIT ? kGemmWaves : 2][kBuf];
    __shared__ __align__(16) uint8_t s_stage[kGemmWaves][wave_stage(GS)];
    __shared__ float s_red[SPLIT ? 2 : 1][SPLIT ? kGemmWaves : 1][SPLIT ? CB * 4 : 1][kWave];

    // Workgroup -> tile: ids go round the 8 XCDs in turn, so each XCD gets a
    // contiguous run of tiles, column tiles inside row tiles: the row tile's
    // weights and the chunk's image are then read from that XCD's L2.
    const int id = static_cast<int>(blockIdx.x);
    const int t = (id & 7) * per_xcd + (id >> 3);
    if (t >= nrt * nct) return;
    const int rt = t / nct;
    const int ct = t - rt * nct;

    const int G = K / GS;
    const int tid = static_cast<int>(threadIdx.x);
    const int lane = tid & (kWave - 1);
    const int wave = tid >> 6;
    const int r16 = lane & 15;
    const int q = lane >> 4;
    const int nbands = (M + 3) >> 2;
    const int nblk = (ncols + kImageCols - 1) / kImageCols;
    const int row0 = SPLIT ? rt * 16 : rt * kGemmRows + wave * 16;
    uint8_t* stage = s_stage[wave];
    uint8_t (*s_buf)[kBuf] = SPLIT ? s_bufs + wave : s_bufs;
    const int loader = SPLIT ? lane : tid;

    // rows past M read the last band / row and are never stored
    const uint8_t* wband = quant + static_cast<size_t>(min((row0 >> 2) + (lane >> 4), nbands - 1)) * G * kGroupBytes +
                           (lane & 15) * 16;
    const uint32_t* mrow = meta + static_cast<size_t>(min(row0 + r16, M - 1)) * G;
    const size_t fac_off = image_fac_offset(K);
    const size_t us_off = image_us_offset(K);

    // this thread's 16-byte units of a step's operands (at step group g: + g *
    // kOpStep) and of its scales; column blocks past the last read the last.
    // Threads past the units repeat the last one (the same bytes stored
    // twice), which keeps the step free of branches.
    const uint8_t* op_src[kOpLoads];
    int op_dst[kOpLoads];
#pragma unroll
    for (int i = 0; i < kOpLoads; ++i) {
        const int u = min(i * kLoaders + loader, kOpUnits - 1);
        const int cb = u / (kOpBytes / 16);
        const int blk = min(ct * CB + cb, nblk - 1);
        op_src[i] = image + static_cast<size_t>(blk) * image_bytes(K) + (u % (kOpBytes / 16)) * 16;
        // a unit is chunks 2h and 2h + 1 (h = u & 1) of a column's 32-element
        // slice; in LDS a slice is [chunk][column] (the image: [column][chunk]),
        // so that lane (r16, q) reads the 8 bytes at 8 * lane
        const int e = u % 32;
        op_dst[i] = cb * kOpBytes + (u % (kOpBytes / 16)) / 32 * 512 + (e & 1) * 256 + (e >> 1) * 8;
    }
    constexpr int kOpStep = UPS * 512;  // image bytes per group
    const uint8_t* sc_src;
    int sc_dst, sc_step;
    {
        const int u = min(loader, kScaleUnits - 1);
        const int cb = u / (kScale / 16);
        const int e = u % (kScale / 16);
        const int blk = min(ct * CB + cb, nblk - 1);
        const uint8_t* base = image + static_cast<size_t>(blk) * image_bytes(K);
        const bool pair = GS == 32 || e < 8;
        sc_src = base + (pair ? fac_off + e * 16 : us_off + (e - 8) * 16);
        sc_step = pair ? kImageCols * 8 : UPS * kImageCols * 4;  // bytes per group
        sc_dst = CB * kOpBytes + cb * kScale + e * 16;
    }

    uint4 ov[kOpLoads], sv, wv;
    uint32_t mv;
    auto load_step = [&](int g) __attribute__((always_inline)) {  // g: the step's first group
#pragma unroll
        for (int i = 0; i < kOpLoads; ++i)
            ov[i] = *reinterpret_cast<const uint4*>(op_src[i] + static_cast<size_t>(g) * kOpStep);
        sv = *reinterpret_cast<const uint4*>(sc_src + static_cast<size_t>(g) * sc_step);
        wv = *reinterpret_cast<const uint4*>(wband + static_cast<size_t>(g) * kGroupBytes);
        mv = mrow[g + (GS == 32 ? q : 0)];
    };
    auto store_shared = [&](int b) __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < kOpLoads; ++i) {
            *reinterpret_cast<uint2*>(s_buf[b] + op_dst[i]) = make_uint2(ov[i].x, ov[i].y);
            *reinterpret_cast<uint2*>(s_buf[b] + op_dst[i] + 128) = make_uint2(ov[i].z, ov[i].w);
        }
        *reinterpret_cast<uint4*>(s_buf[b] + sc_dst) = sv;
    };
    // the wave reads back only what it wrote; its LDS operations complete in order
    auto store_wave = [&]() {
        *reinterpret_cast<uint4*>(stage + (lane >> 4) * kBandStride + (lane & 15) * 16) = wv;
        if (GS == 32 || q == 0)
            *reinterpret_cast<uint32_t*>(stage + 4 * kBandStride + (GS == 32 ? (r16 * 4 + q) * 4 : r16 * 4)) = mv;
    };

    // the first group of step (ks, w, st): increasing over the classes' first
    // steps, so that once one is past the last group all later ones are
    auto group_of = [&](int ks, int w, int st) { return (ks * NU + st) * kClassStride + w * kStepGroups; };

    float tA[CB][4], tB[CB][4], sum[CB][4];
#pragma unroll
    for (int cb = 0; cb < CB; ++cb)
#pragma unroll
        for (int v = 0; v < 4; ++v) tA[cb][v] = tB[cb][v] = sum[cb][v] = 0.0f;

    const int w_begin = SPLIT ? wave : 0;
    const int w_end = SPLIT ? wave + 1 : 4;
    const int first = group_of(0, w_begin, 0);
    load_step(first < G ? first : 0);
    store_shared(0);
    int buf = 0;
    const v4i32 zero = {0, 0, 0, 0};
    for (int ks = 0; ks < KS; ++ks) {
        for (int w = w_begin; w < w_end; ++w) {
            float acc[CB][4][4];  // [column block][row 4q + v][accumulator j]
#pragma unroll
            for (int cb = 0; cb < CB; ++cb)
#pragma unroll
                for (int v = 0; v < 4; ++v)
#pragma unroll
                    for (int j = 0; j < 4; ++j) acc[cb][v][j] = 0.0f;
            for (int st = 0; st < NU; ++st) {  // uniform per workgroup
                const int g = group_of(ks, w, st);
                if (g >= G) break;
                store_wave();
                if constexpr (SPLIT) __builtin_amdgcn_wave_barrier();
                else __syncthreads();  // buffer `buf` is complete; the other one is free
                // the next step's loads (after the last step: this one's again)
                int gn = group_of(ks, w, st + 1);
                if (st + 1 == NU || gn >= G)
                    gn = w + 1 < w_end ? group_of(ks, w + 1, 0) : group_of(ks + 1, w_begin, 0);
                load_step(gn < G ? gn : g);
                __builtin_amdgcn_sched_barrier(0);

                const uint8_t* ops = s_buf[buf];
                uint4 m4[GS == 32 ? 4 : 1];  // GS 32: row 4q + v's four groups; GS 128: rows 4q..4q+3
#pragma unroll
                for (int v = 0; v < (GS == 32 ? 4 : 1); ++v)
                    m4[v] = *reinterpret_cast<const uint4*>(stage + 4 * kBandStride + (GS == 32 ? (4 * q + v) * 16 : q * 16));
                auto pair_of = [&](int v, int k) {
                    const uint4& m = m4[GS == 32 ? v : 0];
                    const int i = GS == 32 ? k : v;
                    return i == 0 ? m.x : i == 1 ? m.y : i == 2 ? m.z : m.w;
                };
                float sx[CB][4];  // GS 128: s*xs of the step's one group
                if constexpr (GS == 128) {
#pragma unroll
                    for (int cb = 0; cb < CB; ++cb) {
                        const float xs = *reinterpret_cast<const float*>(ops + CB * kOpBytes + cb * kScale + r16 * 8);
#pragma unroll
                        for (int v = 0; v < 4; ++v) sx[cb][v] = half_bits_to_float(pair_of(v, 0)) * xs;
                    }
                }
#pragma unroll
                for (int k = 0; k < 4; ++k) {
                    // GS 32: group k's row r16 & 3 of its band (unit 4k + r);
                    // GS 128: slice k of row r (unit 4r + k); dword q holds
                    // elements 8q..8q+7, split as the activation operand is
                    const int unit = GS == 32 ? 4 * k + (r16 & 3) : 4 * (r16 & 3) + k;
                    const uint32_t wd =
                        *reinterpret_cast<const uint32_t*>(stage + (r16 >> 2) * kBandStride + unit * 16 + q * 4);
                    const uint64_t a = static_cast<uint64_t>(wd & 0x0F0F0F0Fu) |
                                       (static_cast<uint64_t>((wd >> 4) & 0x0F0F0F0Fu) << 32);
                    float s[4], zs[4];
#pragma unroll
                    for (int v = 0; v < 4; ++v) {
                        const uint32_t p = pair_of(v, k);
                        s[v] = half_bits_to_float(p);
                        zs[v] = -(half_bits_to_float(p >> 16) * s[v]);
                    }
#pragma unroll
                    for (int cb = 0; cb < CB; ++cb) {
                        const uint64_t b =
                            *reinterpret_cast<const uint64_t*>(ops + cb * kOpBytes + k * 512 + lane * 8);
                        float xs = 0.0f, xu;
                        if constexpr (GS == 32) {
                            const float2 f = *reinterpret_cast<const float2*>(ops + CB * kOpBytes + cb * kScale +
                                                                              k * 128 + r16 * 8);
                            xs = f.x;
                            xu = f.y;
                        } else {
                            xu = *reinterpret_cast<const float*>(ops + CB * kOpBytes + cb * kScale + 128 + k * 64 +
                                                                 r16 * 4);
                        }
                        const v4i32 d = __builtin_amdgcn_mfma_i32_16x16x32_i8(static_cast<long>(a), static_cast<long>(b),
                                                                             zero, 0, 0, 0);
#pragma unroll
                        for (int v = 0; v < 4; ++v) {
                            const float p = GS == 32 ? s[v] * xs : sx[cb][v];
                            acc[cb][v][k] = fmaf(static_cast<float>(d[v]), p, acc[cb][v][k]);
                            acc[cb][v][k] = fmaf(zs[v], xu, acc[cb][v][k]);
                        }
                    }
                }
                __builtin_amdgcn_sched_barrier(0);
                if constexpr (!SPLIT) buf ^= 1;
                store_shared(buf);
            }
            // the class's in-row fold, then the classes and the K ranges
            float r[CB][4];
#pragma unroll
            for (int cb = 0; cb < CB; ++cb)
#pragma unroll
                for (int v = 0; v < 4; ++v) {
                    const float* a = acc[cb][v];
                    r[cb][v] = GS == 32 ? (a[0] + a[3]) + (a[2] + a[1]) : (a[0] + a[1]) + (a[2] + a[3]);
                }
            auto each = [&](auto&& f) {
#pragma unroll
                for (int cb = 0; cb < CB; ++cb)
#pragma unroll
                    for (int v = 0; v < 4; ++v) f(tA[cb][v], tB[cb][v], sum[cb][v], r[cb][v]);
            };
            if constexpr (SPLIT) {  // wave v adds the classes' value v of every block
                float (*red)[CB * 4][kWave] = s_red[ks & 1];
#pragma unroll
                for (int cb = 0; cb < CB; ++cb)
#pragma unroll
                    for (int v = 0; v < 4; ++v) red[wave][cb * 4 + v][lane] = r[cb][v];
                __syncthreads();  // every wave passes it once per K range
#pragma unroll
                for (int cb = 0; cb < CB; ++cb) {
                    const int i = cb * 4 + wave;
                    const float p = (red[0][i][lane] + red[1][i][lane]) + (red[2][i][lane] + red[3][i][lane]);
                    sum[cb][0] = ks == 0 ? p : sum[cb][0] + p;
                }
            } else if (w == 0) {
                each([](float& a, float&, float&, float x) { a = x; });
            } else if (w == 1) {
                each([](float& a, float&, float&, float x) { a = a + x; });
            } else if (w == 2) {
                each([](float&, float& b, float&, float x) { b = x; });
            } else if (ks == 0) {
                each([](float& a, float& b, float& t, float x) { t = a + (b + x); });
            } else {
                each([](float& a, float& b, float& t, float x) { t = t + (a + (b + x)); });
            }
        }
    }
    const int row = row0 + 4 * q + (SPLIT ? wave : 0);
#pragma unroll
    for (int cb = 0; cb < CB; ++cb) {
        const int n = (ct * CB + cb) * kImageCols + r16;
        if (n >= ncols) continue;
        float* y = Y + static_cast<size_t>(n) * M + row;
        if constexpr (SPLIT) {
            if (row < M) *y = sum[cb][0];
        } else if ((M & 3) == 0) {
            if (row < M) *reinterpret_cast<float4*>(y) = make_float4(sum[cb][0], sum[cb][1], sum[cb][2], sum[cb][3]);
        } else {
#pragma unroll
            for (int v = 0; v < 4; ++v)
                if (row + v < M) y[v] = sum[cb][v];
        }
    }
}

template <int GS, int CB, bool SPLIT = false>
asdsl_status launch_gemm(const uint8_t* meta, const uint8_t* quant, const void* image, float* Y, int M, int K,
                         int ncols, int ks, int nu, hipStream_t s) {
    const int rows = SPLIT ? 16 : kGemmRows;
    const int nrt = (M + rows - 1) / rows;
    const int nblk = (ncols + kImageCols - 1) / kImageCols;
    const int nct = (nblk + CB - 1) / CB;
    const int per_xcd = (nrt * nct + 7) / 8;
    return launch("preq2_gemm_exact_kernel", preq2_gemm_exact_kernel<GS, CB, SPLIT>, dim3(8 * per_xcd), dim3(kGemmThreads), 0,
                  s, reinterpret_cast<const uint32_t*>(meta), quant, static_cast<const uint8_t*>(image), Y, M, K,
                  ncols, ks, nu, nrt, nct, per_xcd);
}

}  // namespace
}  // namespace asdsl

using namespace asdsl;

asdsl_status asdsl::preq2_gemm_exact(const uint8_t* meta, const uint8_t* quant, const void* image, float* Y,
                                     int out_features, int in_features, int group_size, int n_cols,
                                     asdsl_stream_t stream) {
    const int M = out_features, K = in_features;
    ASDSL_CHECK_ARG(meta && quant && image && Y, "gemm_preq2_exact: null pointer");
    ASDSL_CHECK_ARG((group_size == 32 || group_size == 128) && M > 0 && K > 0 && K % 128 == 0 &&
                        K / 32 <= 640 && n_cols > 0,
                    "gemm_preq2_exact: invalid dimensions");
    ASDSL_CHECK_ARG(reinterpret_cast<uintptr_t>(image) % 16 == 0 && reinterpret_cast<uintptr_t>(quant) % 4 == 0 &&
                        reinterpret_cast<uintptr_t>(meta) % 4 == 0 && reinterpret_cast<uintptr_t>(Y) % 16 == 0,
                    "gemm_preq2_exact: misaligned operand");
    ASDSL_CU_COUNT(cus);
    int lks = 0, nu = 0, waves = 0;
    bool exact = false;
    preq2_plan_shape(M, K, cus, &lks, &nu, &waves, &exact);
    const int ks = 1 << lks;
    hipStream_t s = as_hip(stream);
    const int nrt = (M + kGemmRows - 1) / kGemmRows;
    const int nblk = (n_cols + kImageCols - 1) / kImageCols;
    // Up to 4.5 tiles of 64 rows x 16 columns per compute unit the split form
    // (us, split against not: o_proj 3072x3072 g32 at 80 columns, 0.9 tiles,
    // 13.2 / 18.3; down 3072x8192 g128 at 256, 3 tiles, 46.0 / 76.0; gate_up
    // 16384x3072 g128 at 64, 4 tiles, 27.6 / 33.0, at 80, 5 tiles, 36.8 /
    // 32.2; qkv 5120x3072 g32 at 256, 5 tiles, 35.7 / 36.5), with one block a
    // workgroup while four workgroups per compute unit hold them all (down at
    // 80 columns, 960 workgroups: 20.1 / 24.2 with two; at 128, 1536: 32.4 /
    // 24.6).
    if (2LL * nrt * nblk <= 9LL * cus) {
        const bool one = nblk == 1 || static_cast<long long>((M + 15) / 16) * nblk <= 4LL * cus;
        if (group_size == 32)
            return one ? launch_gemm<32, 1, true>(meta, quant, image, Y, M, K, n_cols, ks, nu, s)
                       : launch_gemm<32, 2, true>(meta, quant, image, Y, M, K, n_cols, ks, nu, s);
        return one ? launch_gemm<128, 1, true>(meta, quant, image, Y, M, K, n_cols, ks, nu, s)
                   : launch_gemm<128, 2, true>(meta, quant, image, Y, M, K, n_cols, ks, nu, s);
    }
    // Column blocks per workgroup otherwise: a block more shares the unpacked
    // weights and (s, z) pairs among more MFMAs (about 60 vector instructions
    // per step of 4 MFMAs per block, each 16) but leaves fewer workgroups;
    // taken is the smallest product of rounds over the compute units and cost.
    auto cost = [&](int cb) {
        const long long wgs = static_cast<long long>(nrt) * ((nblk + cb - 1) / cb);
        return ((wgs + cus - 1) / cus) * (60 + 64 * cb);
    };
    int cb = 4;
    for (int c = 3; c >= 1; --c)
        if (cost(c) < cost(cb)) cb = c;
    if (group_size == 32)
        return cb == 4   ? launch_gemm<32, 4>(meta, quant, image, Y, M, K, n_cols, ks, nu, s)
               : cb == 3 ? launch_gemm<32, 3>(meta, quant, image, Y, M, K, n_cols, ks, nu, s)
               : cb == 2 ? launch_gemm<32, 2>(meta, quant, image, Y, M, K, n_cols, ks, nu, s)
                         : launch_gemm<32, 1>(meta, quant, image, Y, M, K, n_cols, ks, nu, s);
    return cb == 4   ? launch_gemm<128, 4>(meta, quant, image, Y, M, K, n_cols, ks, nu, s)
           : cb == 3 ? launch_gemm<128, 3>(meta, quant, image, Y, M, K, n_cols, ks, nu, s)
           : cb == 2 ? launch_gemm<128, 2>(meta, quant, image, Y, M, K, n_cols, ks, nu, s)
                     : launch_gemm<128, 1>(meta, quant, image, Y, M, K, n_cols, ks, nu, s);
}
