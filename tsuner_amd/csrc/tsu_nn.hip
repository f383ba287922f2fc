// tsu_nn.hip -- BF16 MFMA kernels of the learned coarse-grid correction.
//
// Network: four 3x3 'same' convolutions (8 -> 32 -> 32 -> 32 -> 4 channels),
// ReLU after the first three.  Activations are NHWC BF16, weights BF16 with
// FP32 accumulation on v_mfma_f32_16x16x32_bf16, master weights and
// optimiser state FP32.
//
// Every convolution is computed transposed, D^T[m][p] = sum_k Wt[m][k] X^T[k][p]
// with m = output channel and p = pixel, so that both MFMA operands are
// 16-byte vectors along the channel axis of an NHWC row (weights [tap][m][k],
// activations [pixel][k]) and each lane's results are consecutive output
// channels of one pixel.  The K axis of an MFMA
// (32 values) is four "octets" of 8 channels; octet o of the flattened
// (tap, channel) axis is tap o / (K/8), channels 8*(o % (K/8)) + 0..7, so an
// 8-channel layer packs four taps into one MFMA and a 32-channel layer one
// tap.  The data-gradient is the same kernel with the tap offsets negated and
// the per-tap transposed weights; the weight gradient contracts over pixels.
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "tsu_nn.h"

namespace tsu {
namespace nn {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x4 __attribute__((ext_vector_type(4)));

__device__ __forceinline__ uint16_t to_bf16(float f)
{
    // round to nearest, ties to even (finite inputs)
    uint32_t u = __float_as_uint(f);
    u += 0x7FFFu + ((u >> 16) & 1u);
    return (uint16_t)(u >> 16);
}

__device__ __forceinline__ float from_bf16(uint16_t b) { return __uint_as_float((uint32_t)b << 16); }

__device__ __forceinline__ bf16x8 as_bf16x8(uint4 v) { return __builtin_bit_cast(bf16x8, v); }

__device__ __forceinline__ int tap_dy(int t) { return t / 3 - 1; }
__device__ __forceinline__ int tap_dx(int t) { return t % 3 - 1; }

// ---- walking down strips -----------------------------------------------------
//
// Every convolution kernel walks down strips of 64 columns, R rows per pass,
// with its input rows in an LDS ring: a row is loaded once per strip (plus two
// at the top of a stretch), and the next pass's rows are loaded into registers
// while the MFMAs run on the current ones.  The passes of all strips of all
// images, in order, are cut into one contiguous stretch per workgroup.
constexpr int kStripCols = 64;

// The stretch of one workgroup: `left` passes from image n, column c0, row r0.
struct StripWalk {
    long long left;
    int n, c0, r0;
    int H, W;
    __device__ StripWalk(int N, int H_, int W_, int R) : H(H_), W(W_)
    {
        const int segs = (W + kStripCols - 1) / kStripCols, passes = (H + R - 1) / R;
        const long long total = (long long)N * segs * passes;
        long long i = total * blockIdx.x / gridDim.x;
        left = total * (blockIdx.x + 1) / gridDim.x - i;
        r0 = (int)(i % passes) * R;
        i /= passes;
        c0 = (int)(i % segs) * kStripCols;
        n = (int)(i / segs);
    }
    // to the next pass; true if it continues the strip
    __device__ bool next(int R)
    {
        r0 += R;
        if (r0 < H) return true;
        r0 = 0;
        c0 += kStripCols;
        if (c0 >= W) {
            c0 = 0;
            n++;
        }
        return false;
    }
};

// Barrier for LDS only: the workgroup's waves share nothing in global memory,
// and __syncthreads() would wait for every store of the pass to reach memory
// (8 -> 64 channels, 32 images: 107 us with it).
__device__ __forceinline__ void lds_barrier()
{
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
}

// out[p][m] = post( sum_t sum_k in[p + SIGN*off(t)][k] * Wt[t][m][k] )
//   K: input channels (8, 32 or 64), MOUT: channels stored per output pixel,
//   M = 16 MTW MG: output channels held by the weights.
//   POST 0: + bias, ReLU, BF16 out.  1: + bias, FP32 out.  2: zero where
//   act[p][m] == 0 (ReLU derivative), BF16 out.
//
// A pass is R = 4 rows of 64 columns (more with 8 input channels, whose passes
// are short beside a load's latency, taken four rows at a time: 8 -> 64 for 32
// images 106 us with 4 rows, 70 with 8).  A wave covers
// 16 columns x RW = 4 / RG rows x 16 MTW output channels and keeps its weights of all nine taps in
// registers (144 for 64 channels in and 32 out), so that only the input is
// read from LDS, and each 16-byte read of an input row serves the output rows
// above, at and below it: one read per four MFMAs of 64 -> 64 and 32 -> 32
// channels.  The workgroup has 4 waves side by side, times MG groups of
// output channels, times RG groups of rows.  With two tiles of output
// channels, row 4g + e of tile a is channel 8g + 4a + e, so that a lane's
// results are eight consecutive channels of a pixel, one 16-byte store.
//
// Bound by the bytes of both tensors for the narrow layers and by how well the
// MFMAs, the epilogue and the loads of one workgroup overlap for 64 -> 64
// (matrix pipe 51 % busy; without its loads and stores 120 us).  Before
// (weights and a 10 x 66 pixel tile in LDS, one read per two MFMAs, the tile's
// loads and stores between barriers) and now, us:
//            8->32  32->32  32->4  8->64  64->64  64->4, and the data
//   32 images  41     89     48    106     200     95    gradients 4<-32 60,
//   of 256^2   27     50     30     68     140     62    32<-32 103, 4<-64 181,
//   8 images   14     25     14     28      55     27    64<-64 259 -> 54, 79,
//               9     16     11     15      36     18    123, 175 (32 images)
// 32 -> 32 moves 268 MB in 50 us, 5.4 TB/s of the copy kernel's 6.1.  Accumulation
// order and results are those of one tap after the other.
//
// LDS: the ring is three blocks of a pass's rows and copies of its first two
// rows behind them, so that the R + 2 rows of a pass lie in order wherever it
// starts and a read's row is an immediate.  A pixel's octets are XOR-ed with bits of its column:
// the 16 lanes of a read (one octet of 16 consecutive pixels) cover all banks.
template <int K>
__device__ __forceinline__ int octet_xor(int c)
{
    return K == 64 ? (c >> 1) & 7 : K == 32 ? (c >> 2) & 3 : 0;
}

typedef float f32x2 __attribute__((ext_vector_type(2)));
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));

// two floats -> packed BF16 pair, round to nearest even (v_cvt_pk_bf16_f32)
__device__ __forceinline__ uint32_t pack_bf16x2(float a, float b)
{
    return __builtin_bit_cast(uint32_t, __builtin_convertvector((f32x2){a, b}, bf16x2));
}

// max(x, 0), 0 for a NaN, in one instruction (fmaxf quiets its operand first)
__device__ __forceinline__ float relu(float x) { return __builtin_amdgcn_fmed3f(x, 0.f, __builtin_inff()); }

// waves per SIMD: what the registers allow (weights + accumulators + input)
template <int K>
constexpr int conv_waves() { return K == 8 ? 4 : 2; }

// rows of a pass, and of the ring: three blocks of them, and the copies
template <int K>
constexpr int conv_rows() { return K == 8 ? 8 : 4; }
constexpr int conv_ring(int rows) { return 3 * rows + 2; }

template <int K, int MTW, int MG, int RG, int MOUT, int SIGN, int POST>
__global__ __launch_bounds__(256 * MG * RG)
__attribute__((amdgpu_waves_per_eu(conv_waves<K>(), conv_waves<K>()))) void conv_kernel(
    const uint16_t* __restrict__ in, const uint16_t* __restrict__ Wt, const float* __restrict__ bias,
    const uint16_t* __restrict__ act, void* __restrict__ out, int N, int H, int W)
{
    constexpr int T = 256 * MG * RG, R = conv_rows<K>(), RW = 4 / RG, M = 16 * MTW * MG;
    constexpr int KO = K / 8, KK = K == 8 ? 1 : K / 32;
    constexpr int XCOL = kStripCols + 2, XROW = XCOL * KO;  // ring row, in uint4
    constexpr int SLOTS = kStripCols * KO;                  // a row's octets but for the last two columns'
    constexpr int SWEEP = T / SLOTS;                        // rows per sweep of the workgroup
    constexpr int LOADS = SWEEP >= R ? 1 : R / SWEEP;
    constexpr int STEPS = K == 8 ? 3 : 9 * KK;
    constexpr int READS = (K == 8 ? RW : RW + 2) * 3 * KK, AHEAD = K == 64 ? 2 : 0;
    constexpr bool EARLY = K == 64 || (K == 32 && POST == 2);   // see put
    static_assert(T % SLOTS == 0 && 2 * KO * R <= T, "one slot per thread and sweep");
    __shared__ uint4 ring[conv_ring(R) * XROW];
    const int tid = threadIdx.x, wv = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63;
    const int g = lane >> 4, li = lane & 15;
    const int seg = wv & 3, mg = (wv >> 2) % MG, rg = (wv >> 2) / MG;
    StripWalk walk(N, H, W, R);

    const int m0 = 16 * MTW * mg + 4 * MTW * g;             // this lane's 4 MTW consecutive output channels
    // of which MOUT = 4 has those of the first lane group only: the caller's
    // bias ends there
    static_assert(MOUT % (4 * MTW) == 0, "a lane's channels are all stored or none");
    f32x4 bias_of[MTW];
#pragma unroll
    for (int a = 0; a < MTW; a++)
#pragma unroll
        for (int e = 0; e < 4; e++) bias_of[a][e] = POST == 2 || m0 >= MOUT ? 0.f : bias[m0 + 4 * a + e];

    // staging: this thread's octet and column (and row, if a sweep takes
    // several), and one of the last two columns' for the first threads
    const int q = tid % KO, col = tid / KO % kStripCols, row = SWEEP > 1 ? tid / SLOTS : 0;
    const int put_at = row * XROW + col * KO + (q ^ octet_xor<K>(col));
    const bool has_edge = tid < 2 * KO * R;
    const int ecol = kStripCols + tid / KO % 2, erow = tid / (2 * KO);
    const int eput_at = erow * XROW + ecol * KO + (q ^ octet_xor<K>(ecol));
    uint4 stage[LOADS], estage;
    auto load = [&](int gr, int gc, int rows) {             // zeros outside the image's first rows
        uint4 v = make_uint4(0, 0, 0, 0);
        if (gr >= 0 && gr < rows && gc >= 0 && gc < W)
            v = *(const uint4*)((const char*)in + ((size_t)walk.n * H + gr) * W * (2 * K) +
                                (uint32_t)((gc * K + 8 * q) * 2));
        return v;
    };
    // the pass's new rows, r0 + 1 .. r0 + R (columns c0 - 1 .. c0 + 64), into registers
    auto fetch = [&](int rows) {
#pragma unroll
        for (int j = 0; j < LOADS; j++)
            if (SWEEP <= R || row < R) stage[j] = load(walk.r0 + 1 + j * SWEEP + row, walk.c0 - 1 + col, rows);
        if (has_edge) estage = load(walk.r0 + 1 + erow, walk.c0 - 1 + ecol, rows);
    };
    // ... and into ring rows R ph + 2 .. R ph + R + 1; the last two of block 2
    // are also the first two of block 0
    auto put = [&](int ph) {
#pragma unroll
        for (int j = 0; j < LOADS; j++) {
            const int r = j * SWEEP + row;
            if (SWEEP <= R || row < R) {
                ring[(R * ph + 2 + j * SWEEP) * XROW + put_at] = stage[j];
                if (ph == 2 && r >= R - 2) ring[(j * SWEEP - (R - 2)) * XROW + put_at] = stage[j];
            }
        }
        if (has_edge) {
            ring[(R * ph + 2) * XROW + eput_at] = estage;
            if (ph == 2 && erow >= R - 2) ring[-(R - 2) * XROW + eput_at] = estage;
        }
    };
    // at the top of a stretch or strip: rows r0 - 1 and r0, which go into ring
    // rows R ph and R ph + 1
    constexpr int TOP = 2 * XROW;
    auto load_top = [&](int idx) {
        const int o = idx % KO, c = idx / KO % XCOL, i = idx / XROW;
        const int gr = walk.r0 - 1 + i, gc = walk.c0 - 1 + c;
        uint4 v = make_uint4(0, 0, 0, 0);
        if (idx < TOP && gr >= 0 && gr < H && gc >= 0 && gc < W)
            v = *(const uint4*)(in + (((size_t)walk.n * H + gr) * W + gc) * K + 8 * o);
        return v;
    };
    auto put_top = [&](int ph, int idx, uint4 v) {
        const int o = idx % KO, c = idx / KO % XCOL, i = idx / XROW;
        if (idx < TOP) ring[(R * ph + i) * XROW + c * KO + (o ^ octet_xor<K>(c))] = v;
    };

    // this lane's reads in the first of the wave's rows: column 16 seg + li +
    // rx, octet 4 kk + g; with 8 channels, the offset of step rx and lane group g
    int at[3][KK];
#pragma unroll
    for (int rx = 0; rx < 3; rx++)
#pragma unroll
        for (int kk = 0; kk < KK; kk++) {
            const int o = 4 * rx + g < 9 ? 4 * rx + g : 8;
            const int cl = 16 * seg + li + (K == 8 ? o % 3 : rx);
            at[rx][kk] = (RW * rg + (K == 8 ? o / 3 : 0)) * XROW + cl * KO + ((K == 8 ? 0 : 4 * kk + g) ^ octet_xor<K>(cl));
        }

    // weights: step (offset ry, rx; 32 channels kk) of input offset (ry - 1,
    // rx - 1), tap 3 ry + rx, or its opposite for the data gradients.  With 8
    // channels a step holds four offsets, one per lane group.
    //
    // The weights of 64 input channels go through the ring, which is free yet: 16
    // lanes of a wave's own loads take 16 rows of weights, a cache line each, and
    // the four waves side by side the same ones.  64 -> 64, an image of 64^2: 13.5
    // us so, 7.7 here; 2 images of 256^2 19.7 and 14.0, 32 images 144 and 140.
    // With fewer channels the loads wait less than two more barriers take (32 ->
    // 32, an image of 64^2 4.3 and 4.7 us; training, 8 images, 193.5 and 196.6).
    constexpr bool BY_RING = K == 64;
    constexpr int WN = 9 * M * KO, WEIGHTS = (WN + T - 1) / T, TOPS = (TOP + T - 1) / T;
    static_assert(!BY_RING || WN <= conv_ring(R) * XROW, "the ring holds the weights");
    fetch(H);
    uint4 tops[TOPS];
#pragma unroll
    for (int j = 0; j < TOPS; j++) tops[j] = load_top(tid + T * j);
    if constexpr (BY_RING) {
        uint4 w[WEIGHTS];
#pragma unroll
        for (int j = 0; j < WEIGHTS; j++) w[j] = ((const uint4*)Wt)[min(tid + T * j, WN - 1)];
#pragma unroll
        for (int j = 0; j < WEIGHTS; j++) {
            const int idx = tid + T * j, row = idx / KO;    // row: of [tap][output channel]
            if (idx < WN) ring[row * KO + (idx % KO ^ octet_xor<K>(row))] = w[j];
        }
        lds_barrier();
    }
    bf16x8 A[STEPS][MTW];
#pragma unroll
    for (int s = 0; s < STEPS; s++)
#pragma unroll
        for (int a = 0; a < MTW; a++) {
            const int o = K == 8 ? 4 * s + g : s / KK, k = K == 8 ? 0 : 32 * (s % KK) + 8 * g;
            const int t = SIGN > 0 ? o : 8 - o;
            const int m = 16 * MTW * mg + (MTW == 2 ? 8 * (li >> 2) + 4 * a + (li & 3) : li);
            uint4 v = make_uint4(0, 0, 0, 0);
            if (BY_RING)
                v = ring[(t * M + m) * KO + (k / 8 ^ octet_xor<K>(m))];
            else if (o < 9)
                v = *(const uint4*)(Wt + ((size_t)(t * M + m) * K + k));
            A[s][a] = as_bf16x8(v);
        }
    if (BY_RING) lds_barrier();

    int ph = 0;                                             // ring row of input row r0 - 1, over R
#pragma unroll
    for (int j = 0; j < TOPS; j++) put_top(0, tid + T * j, tops[j]);
    put(0);
    lds_barrier();
    for (;;) {
        int cr0 = walk.r0 + RW * rg;                        // this pass: the wave's first row, this lane's column
        const int c = walk.c0 + 16 * seg + li;
        const int pass_n = walk.n;
        size_t p0 = ((size_t)walk.n * H + cr0) * W + c;
        const bool more = --walk.left > 0;                  // uniform over the workgroup
        bool down = false;                                  // the next pass continues this strip
        if (more) down = walk.next(R);
        if (EARLY || more) fetch(more ? H : 0);
        const int next_ph = ph == 2 ? 0 : ph + 1;           // the coming rows have ring rows of their own
        const uint4* rows = ring + R * ph * XROW;
#pragma unroll 1
        for (int part = 0; part < R / 4; part++) {
            f32x4 acc[RW][MTW];
#pragma unroll
            for (int r = 0; r < RW; r++)
#pragma unroll
                for (int a = 0; a < MTW; a++) acc[r][a] = f32x4{0.f, 0.f, 0.f, 0.f};
            // by input row: an output row then takes its taps in their order
            // (and with 8 channels, a row's steps, whose offsets the lanes
            // hold).  With 64 channels AHEAD reads are kept in flight: the
            // compiler, short of registers, issued each and waited for it by
            // itself.
            auto read = [&](int i) {
                const int j = i / (3 * KK), rx = i / KK % 3, kk = i % KK;
                uint4 v = rows[at[rx][kk] + j * XROW];
                if (K == 8 && rx == 2 && g > 0) v = make_uint4(0, 0, 0, 0);   // past the ninth offset
                return v;
            };
            uint4 ahead[AHEAD + 1];
#pragma unroll
            for (int i = 0; i < AHEAD; i++) ahead[i] = read(i);
#pragma unroll
            for (int i = 0; i < READS; i++) {
                if (i + AHEAD < READS) ahead[(i + AHEAD) % (AHEAD + 1)] = read(i + AHEAD);
                if (AHEAD > 0) __builtin_amdgcn_sched_barrier(0);
                const int j = i / (3 * KK), rx = i / KK % 3, kk = i % KK;
                const bf16x8 B = as_bf16x8(ahead[i % (AHEAD + 1)]);
#pragma unroll
                for (int ry = 0; ry < (K == 8 ? 1 : 3); ry++) {
                    const int r = j - ry;
                    if (r < 0 || r >= RW) continue;
#pragma unroll
                    for (int a = 0; a < MTW; a++)
                        acc[r][a] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
                            A[K == 8 ? rx : (3 * ry + rx) * KK + kk][a], B, acc[r][a], 0, 0, 0);
                }
            }
            // the activations of all rows at once (a row's load behind the
            // stores of the rows before it waits for them as well)
            uint4 mask[RW];
            if constexpr (POST == 2 && K != 8) {
#pragma unroll
                for (int r = 0; r < RW; r++)
                    mask[r] = *(const uint4*)(act + m0 +
                                              (((size_t)pass_n * H + min(cr0 + r, H - 1)) * W + min(c, W - 1)) * MOUT);
            }
            // EARLY: the coming rows go into the ring ahead of the results'
            // stores, in every pass.  A wait for these loads behind stores
            // that lanes may skip is a wait for the stores too: 64 -> 64, 32
            // images, 162 -> 150 us with the reads ahead.  Short passes have
            // the loads come later than the stores go: 8 -> 32, 8 images,
            // 9.2 us so and 10.0 early, 32 -> 32 16.9 and 17.7.
            if (EARLY) put(next_ph);
#pragma unroll
            for (int r = 0; r < RW; r++) {
                if (cr0 + r >= H || c >= W || m0 >= MOUT) continue;
                const size_t p = p0 + (size_t)r * W;
                float v[4 * MTW];
#pragma unroll
                for (int a = 0; a < MTW; a++)
#pragma unroll
                    for (int e = 0; e < 4; e++) {
                        const float o = POST == 2 ? acc[r][a][e] : acc[r][a][e] + bias_of[a][e];
                        v[4 * a + e] = POST == 0 ? relu(o) : o;
                    }
                if constexpr (POST == 1) {
                    static_assert(MTW == 1, "one tile of output channels");
                    *(float4*)((float*)out + p * MOUT + m0) = make_float4(v[0], v[1], v[2], v[3]);
                } else {
                    static_assert(MTW == 2, "16-byte stores");
                    if (POST == 2) {
                        if (K == 8) mask[r] = *(const uint4*)(act + p * MOUT + m0);
                        const uint32_t aw[4] = {mask[r].x, mask[r].y, mask[r].z, mask[r].w};
                        // ReLU outputs are >= 0: only +0 / -0 bit patterns mean inactive
#pragma unroll
                        for (int e = 0; e < 4; e++) {
                            if ((aw[e] & 0x7FFFu) == 0) v[2 * e] = 0.f;
                            if ((aw[e] & 0x7FFF0000u) == 0) v[2 * e + 1] = 0.f;
                        }
                    }
                    *(uint4*)((uint16_t*)out + p * MOUT + m0) =
                        make_uint4(pack_bf16x2(v[0], v[1]), pack_bf16x2(v[2], v[3]), pack_bf16x2(v[4], v[5]),
                                   pack_bf16x2(v[6], v[7]));
                }
            }
            rows += 4 * XROW;
            cr0 += 4;
            p0 += 4 * (size_t)W;
        }
        if (!more) break;
        if (!EARLY) put(next_ph);
        ph = next_ph;
        if (!down) {
            lds_barrier();                                // every wave is done with the rows above
            for (int idx = tid; idx < TOP; idx += T) put_top(ph, idx, load_top(idx));
        }
        lds_barrier();
    }
}

// ---- weight gradients --------------------------------------------------------
//
// dW[t][m][k] = sum_p dy[p][m] x[p + off(t)][k], contracted over pixels on the
// MFMA K axis (32 pixels of one row per MFMA).  Both operands lie in memory
// with the channel fastest while an MFMA operand wants eight pixels of one
// channel per lane, so the rows are staged in LDS and read with the
// transposing ds_read_b64_tr_b16: a group of 16 lanes reads four pixels x 16
// channels and each lane gets the four pixels of its channel.  (Gathering
// the operands with 2-byte global loads, one tap per workgroup, took 220 us
// for 64 -> 64 channels over 8 images of 256^2 and 109 us for 32 -> 32: nine
// passes over both tensors at two bytes a load.)
//
// A workgroup walks down a strip of 64 columns, R rows per pass: the rows of
// the shifted operand stay in an LDS ring, so that every row is loaded once
// per strip (plus two at the top of a stretch), and the next rows are loaded
// into registers while the MFMAs run on the current ones.  The passes of all
// strips of all images, in order, are cut into one contiguous stretch per
// workgroup; one workgroup per CU fits (its rings take most of the LDS) and
// kWgradWaves = 256 of them cover the chip.
//
// Measured, 8 images of 256^2, before and now (gradient + reduction):
//   64 -> 64  220 + 112 us -> 49 + 7 us (790 TFLOP/s; both tensors once are
//             134 MB, 22 us at the copy kernel's 6.1 TB/s, the MFMAs 15 us at
//             peak, the transposing reads 17 us of LDS time)
//   32 -> 32  109 + 110 us -> 21 + 4 us (67 MB, 11 us)
//   8 -> 64, 64 -> 4   145 and 118 + 112 us -> 21 + 5 us (76 MB, 12 us)
//   8 -> 32, 32 -> 4    84 and 82 + 110 us -> 13 + 4 us (42 MB, 7 us)
//
// Pixels: columns are pitched so that a row is a multiple of 8 pixels, and
// the 32-byte slots of a pixel (16 channels, what one transposing read takes)
// are XOR-ed with bits of its column: the 8 consecutive columns that half a
// wave reads then lie in different banks.  The eight pixels of lane group g
// in a 32-pixel step are 4g .. 4g+3 and 16+4g .. 16+4g+3, for both operands.
//
// The sum takes the pixels p of the image and zeros for x around it, also for
// values that are not finite (0 times an infinity is a NaN): a step's pixels
// past the image must meet zeros in both operands.  RAGGED: the image's width
// is no multiple of the strips' 64 columns (64 -> 64, 8 images of 250^2, 50.2
// -> 51.3 us with it, which widths without a remainder are spared).

constexpr int kWgradPitch = 72;            // LDS columns of the shifted operand's rows (66 used)

typedef short s16x4 __attribute__((ext_vector_type(4)));
typedef __attribute__((address_space(3))) s16x4 lds_s16x4;
typedef __attribute__((address_space(3))) uint4 lds_u4;

// eight pixels of one channel: the transposing reads at byte addresses a and b
__device__ __forceinline__ bf16x8 read_tr8(uint32_t a, uint32_t b)
{
    const s16x4 lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4*)(uintptr_t)a);
    const s16x4 hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4*)(uintptr_t)b);
    return __builtin_bit_cast(bf16x8, __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7));
}

// Eight channels of one pixel.  The weight gradients take operands of any
// element alignment (global loads need none on this hardware; 16-byte aligned
// rows are the fast case).
typedef uint32_t u32x4_any __attribute__((ext_vector_type(4), aligned(2)));
__device__ __forceinline__ uint4 load8(const uint16_t* p)
{
    const u32x4_any v = *(const u32x4_any*)p;
    return make_uint4(v.x, v.y, v.z, v.w);
}

// XOR of a pixel's 32-byte slots at column c: 64 channels have 4 slots and 2
// pixels per 256 bytes (all banks once), 32 channels 2 slots and 4 pixels.
template <int CH>
__device__ __forceinline__ int slot_xor(int c)
{
    return CH == 64 ? (c >> 1) & 3 : CH == 32 ? (c >> 2) & 1 : 0;
}

// Middle layers (x and dy of CH = 32 or 64 channels).  Each of 8 waves holds
// the nine taps of 32 x 32 channels (CH = 64: four such jobs, two waves of a
// job taking half of a pass's pixels each; CH = 32: one job, eight waves),
// and the waves of a job add their sums through LDS at the end.  Partial sums
// go to part[t][workgroup][m][k], the bias gradient (one MFMA per dy tile
// against ones, in the jobs of the first 32 input channels) to
// bpart[workgroup][m].
template <int CH, bool RAGGED>
__global__ __launch_bounds__(512) __attribute__((amdgpu_waves_per_eu(2, 2))) void wgrad_mid_kernel(
    const uint16_t* __restrict__ x, const uint16_t* __restrict__ dy, float* __restrict__ part,
    float* __restrict__ bpart, int N, int H, int W)
{
    constexpr int R = 4;                           // rows per pass
    constexpr int KO = CH / 8, PIX = CH * 2;
    constexpr int XR = 2 * R + 2, DR = 2 * R;      // ring rows: R + 2 in use and R coming, R and R
    constexpr int XROW = kWgradPitch * PIX, DROW = kStripCols * PIX;
    constexpr int JOBS = (CH / 32) * (CH / 32), GROUPS = 8 / JOBS;
    constexpr int STEPS = 2 * R / GROUPS;          // 32-pixel steps of a wave per pass
    constexpr int XPT = (R * 66 * KO + 511) / 512, DPT = R * 64 * KO / 512;
    constexpr int XN = XR * XROW / 16, DN = DR * DROW / 16;
    constexpr int AHEAD = 1;                       // operands read ahead of their MFMAs
    constexpr int TILES = 38;                      // accumulator tiles of a wave, bias included
    constexpr int RED = 4 * TILES * 64;            // those of half of the waves
    constexpr int LDS = XN + DN > RED ? XN + DN : RED;
    __shared__ uint4 lds[LDS];
    const uint32_t xbase = (uint32_t)(uintptr_t)(lds_u4*)lds, dbase = xbase + XN * 16;
    const int tid = threadIdx.x, wv = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63;
    const int g = lane >> 4, li = lane & 15;
    const int job = wv % JOBS, group = wv / JOBS;
    const int m0 = 2 * (job / (CH / 32)), k0 = 2 * (job % (CH / 32));   // first 16-channel tiles
    StripWalk walk(N, H, W, R);

    f32x4 acc[TILES];                              // [tap][k tile][m tile], then the bias of the m tiles
#pragma unroll
    for (int v = 0; v < TILES; v++) acc[v] = f32x4{0.f, 0.f, 0.f, 0.f};
    const uint32_t one2 = 0x3F803F80u;
    const bf16x8 ones = as_bf16x8(make_uint4(one2, one2, one2, one2));

    // lane addresses within a row: pixel 4g + (li >> 2), 8-byte chunk li & 3
    const int px = 4 * g + (li >> 2), chunk = (li & 3) * 8;
    uint32_t xa[3][2], da[2];
#pragma unroll
    for (int d = 0; d < 3; d++)
#pragma unroll
        for (int b = 0; b < 2; b++)
            xa[d][b] = xbase + (px + d) * PIX + (((k0 + b) ^ slot_xor<CH>(px + d)) * 32) + chunk;
#pragma unroll
    for (int a = 0; a < 2; a++) da[a] = dbase + px * PIX + (((m0 + a) ^ slot_xor<CH>(px)) * 32) + chunk;

    uint4 sx[XPT], sd[DPT];
    // x rows r0 + 1 .. r0 + R (columns c0 - 1 .. c0 + 64) and dy rows
    // r0 .. r0 + R - 1 of image n into registers, zeros outside the image
    auto fetch = [&](int n, int c0, int r0) {
#pragma unroll
        for (int j = 0; j < XPT; j++) {
            const int idx = tid + 512 * j;
            const int q = idx % KO, c = (idx / KO) % 66, i = idx / (KO * 66);
            const int gr = r0 + 1 + i, gc = c0 - 1 + c;
            sx[j] = make_uint4(0, 0, 0, 0);
            if (i < R && gr < H && gc >= 0 && gc < W)
                sx[j] = load8(x + (((size_t)n * H + gr) * W + gc) * CH + 8 * q);
        }
#pragma unroll
        for (int j = 0; j < DPT; j++) {
            const int idx = tid + 512 * j;
            const int q = idx % KO, c = (idx / KO) % 64, i = idx / (KO * 64);
            const int gr = r0 + i, gc = c0 + c;
            sd[j] = make_uint4(0, 0, 0, 0);
            if (gr < H && gc < W) sd[j] = load8(dy + (((size_t)n * H + gr) * W + gc) * CH + 8 * q);
        }
    };
    // the fetched rows into ring rows xs + 2, ... and ds, ...
    auto put = [&](int xs, int ds) {
#pragma unroll
        for (int j = 0; j < XPT; j++) {
            const int idx = tid + 512 * j;
            const int q = idx % KO, c = (idx / KO) % 66, i = idx / (KO * 66);
            int s = xs + 2 + i;
            s = s >= XR ? s - XR : s;
            if (i < R)
                lds[(s * XROW + c * PIX) / 16 + (((q >> 1) ^ slot_xor<CH>(c)) * 2 + (q & 1))] = sx[j];
        }
#pragma unroll
        for (int j = 0; j < DPT; j++) {
            const int idx = tid + 512 * j;
            const int q = idx % KO, c = (idx / KO) % 64, i = idx / (KO * 64);
            lds[XN + ((ds + i) * DROW + c * PIX) / 16 + (((q >> 1) ^ slot_xor<CH>(c)) * 2 + (q & 1))] = sd[j];
        }
    };

    // at the top of a stretch or strip: x rows r0 - 1 and r0 into ring rows 0, 1
    auto top = [&](int n, int c0, int r0) {
        for (int idx = tid; idx < 2 * 66 * KO; idx += 512) {
            const int q = idx % KO, c = (idx / KO) % 66, i = idx / (KO * 66);
            const int gr = r0 - 1 + i, gc = c0 - 1 + c;
            uint4 v = make_uint4(0, 0, 0, 0);
            if (gr >= 0 && gr < H && gc >= 0 && gc < W)
                v = load8(x + (((size_t)n * H + gr) * W + gc) * CH + 8 * q);
            lds[(i * XROW + c * PIX) / 16 + (((q >> 1) ^ slot_xor<CH>(c)) * 2 + (q & 1))] = v;
        }
    };

    // ring row of x row r0 - 1 and of dy row r0
    int xs = 0, ds = 0;
    fetch(walk.n, walk.c0, walk.r0);
    top(walk.n, walk.c0, walk.r0);
    put(xs, ds);
    __syncthreads();
    for (;;) {
        const int rows = H - walk.r0, cols = W - walk.c0;   // of the image, from this pass on
        const bool more = --walk.left > 0;                  // uniform over the workgroup
        bool down = false;                                  // the next pass continues this strip
        if (more) {
            down = walk.next(R);
            fetch(walk.n, walk.c0, walk.r0);
        }
#pragma unroll 1
        for (int s = 0; s < STEPS; s++) {
            const int st = group * STEPS + s;               // step of the pass: row st / 2, half row st % 2
            if ((st >> 1) >= rows) break;                   // past the image (see above)
            const uint32_t half = (uint32_t)(st & 1) * 32 * PIX;
            // the left neighbours of the first column past the image: from the
            // column itself, which holds zeros
            const int past = cols - (st & 1) * 32;
            uint32_t left[2][2];
#pragma unroll
            for (int b = 0; b < 2; b++) {
                left[b][0] = RAGGED && px == past ? xa[1][b] : xa[0][b];
                left[b][1] = RAGGED && px + 16 == past ? xa[1][b] : xa[0][b];
            }
            const uint32_t dof = (uint32_t)((ds + (st >> 1)) * DROW) + half;
            bf16x8 A[2];
#pragma unroll
            for (int a = 0; a < 2; a++) A[a] = read_tr8(da[a] + dof, da[a] + dof + 16 * PIX);
            uint32_t xo[3];
#pragma unroll
            for (int ty = 0; ty < 3; ty++) {
                int xrow = xs + (st >> 1) + ty;
                xrow = xrow >= XR ? xrow - XR : xrow;
                xo[ty] = (uint32_t)(xrow * XROW) + half;
            }
            // input operands (ty, d, b), each read while its predecessor's two
            // MFMAs run: the compiler, short of registers, waited for each read
            // (64 -> 64 60.5 us with its reduction, one ahead 56.7, two 57.3,
            // three, which spill, 59.2)
            auto read = [&](int i) {
                const int d = i / 2 % 3, b = i % 2;
                const uint32_t at = (d == 0 ? left[b][0] : xa[d][b]) + xo[i / 6];
                return read_tr8(at, (d == 0 ? left[b][1] + xo[i / 6] : at) + 16 * PIX);
            };
            bf16x8 B[AHEAD + 1];
#pragma unroll
            for (int i = 0; i < AHEAD; i++) B[i] = read(i);
            if (k0 == 0) {
#pragma unroll
                for (int a = 0; a < 2; a++)
                    acc[36 + a] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(A[a], ones, acc[36 + a], 0, 0, 0);
            }
#pragma unroll
            for (int i = 0; i < 18; i++) {
                if (i + AHEAD < 18) B[(i + AHEAD) % (AHEAD + 1)] = read(i + AHEAD);
                __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                for (int a = 0; a < 2; a++)
                    acc[2 * i + a] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(A[a], B[i % (AHEAD + 1)], acc[2 * i + a], 0,
                                                                             0, 0);
            }
        }
        if (!more) break;
        if (down) {
            // the coming rows have ring rows of their own
            xs = xs + R >= XR ? xs + R - XR : xs + R;
            ds = R - ds;
        } else {
            __syncthreads();                                // every wave is done with the rings
            xs = ds = 0;
            top(walk.n, walk.c0, walk.r0);
        }
        put(xs, ds);
        __syncthreads();
    }

    // the sums of a job's waves: halves added pairwise through LDS, in a fixed order
    f32x4* red = (f32x4*)lds;
#pragma unroll
    for (int o = 4; o >= JOBS; o >>= 1) {
        __syncthreads();
        if (wv >= o && wv < 2 * o) {
#pragma unroll
            for (int v = 0; v < TILES; v++) red[(v * 4 + wv - o) * 64 + lane] = acc[v];
        }
        __syncthreads();
        if (wv < o) {
#pragma unroll
            for (int v = 0; v < TILES; v++) acc[v] += red[(v * 4 + wv) * 64 + lane];
        }
    }
    if (wv >= JOBS) return;
    // D[m][k]: lane holds m = tile * 16 + 4 * g + e, k = tile * 16 + li
#pragma unroll
    for (int t = 0; t < 9; t++) {
        float* dst = part + ((size_t)t * gridDim.x + blockIdx.x) * CH * CH;
#pragma unroll
        for (int b = 0; b < 2; b++)
#pragma unroll
            for (int a = 0; a < 2; a++)
#pragma unroll
                for (int e = 0; e < 4; e++)
                    dst[((m0 + a) * 16 + 4 * g + e) * CH + (k0 + b) * 16 + li] = acc[(t * 2 + b) * 2 + a][e];
    }
    if (k0 == 0 && li == 0) {
#pragma unroll
        for (int a = 0; a < 2; a++)
#pragma unroll
            for (int e = 0; e < 4; e++)
                bpart[(size_t)blockIdx.x * CH + (m0 + a) * 16 + 4 * g + e] = acc[36 + a][e];
    }
}

__device__ __forceinline__ bool wave_any(bool b) { return __builtin_expect(__builtin_amdgcn_ballot_w64(b) != 0, 0); }

__device__ __forceinline__ bool not_finite16(uint32_t bits) { return (bits & 0x7F80u) == 0x7F80u; }

// any of eight values an infinity or a NaN: the largest magnitude bits
__device__ __forceinline__ bool not_finite(bf16x8 v)
{
    typedef uint16_t u16x2 __attribute__((ext_vector_type(2)));
    const uint4 u = __builtin_bit_cast(uint4, v);
    const uint32_t w[4] = {u.x, u.y, u.z, u.w};
    u16x2 most = {0, 0};
#pragma unroll
    for (int i = 0; i < 4; i++) most = __builtin_elementwise_max(most, __builtin_bit_cast(u16x2, w[i] & 0x7FFF7FFFu));
    return (most.x >= 0x7F80) | (most.y >= 0x7F80);
}

// A lane's eight pixels of the 32 from column c0 on (4g .. 4g + 3 and 16 + 4g
// ..), with a one of its sign for each value that is not finite and lies on the
// image's border (row: the whole row does).
__device__ __forceinline__ bf16x8 border_ones(bf16x8 v, bool row, int g, int c0, int W)
{
    typedef uint16_t u16x8 __attribute__((ext_vector_type(8)));
    u16x8 u = __builtin_bit_cast(u16x8, v);
#pragma unroll
    for (int i = 0; i < 8; i++) {
        const int c = c0 + 4 * g + (i & 3) + 4 * (i & 4);
        if ((row || c == 0 || c == W - 1) && not_finite16(u[i])) u[i] = (u[i] & 0x8000) | 0x3F80;
    }
    return __builtin_bit_cast(bf16x8, u);
}

// Input and output layers: a wide operand p (CH channels) against a narrow
// one q (8 channels) at nine shifts, G[s][a][b] = sum_p wide[p][a]
// narrow[p + off(s)][b].  The input layer is wide = dy, narrow = x, s = t;
// the output layer sums over x's pixels instead of dy's, wide = x, narrow =
// dy, s = 8 - t (the opposite offset).  Two shifts fill the 16 columns of an
// MFMA: five tiles, whose tenth half column is ones (the input layer's bias
// gradient, sum_p dy).  Every wave holds all shifts and channels; a pass is
// 8 rows, one per wave, and the waves' sums are added through LDS at the
// end.  Bound by the wide operand's bytes.
//
// The output layer's pixels of x at the image's border meet dy's zeros outside
// in products that are none of the sum's, and dy's border pixels x's zeros in
// products of the sum that it does not form.  Both are 0 unless a value there is
// not finite.  Then (a vote per half row and row of the border) such values of x
// are ones to the MFMAs, which keeps the products with infinities of dy, and
// the products that the sum has are added one by one, for such values of dy
// with x's zeros too: NaNs.  The votes cost 64 -> 4 0.8 us of 20.5 with its
// reduction (8 images of 256^2).
template <int CH, bool OUTL, bool RAGGED>
__global__ __launch_bounds__(512) __attribute__((amdgpu_waves_per_eu(2, 2))) void wgrad_edge_kernel(
    const uint16_t* __restrict__ wide, const uint16_t* __restrict__ narrow, float* __restrict__ part,
    float* __restrict__ bpart, int N, int H, int W)
{
    constexpr int R = 8;
    constexpr int KO = CH / 8, MT = CH / 16, PIX = CH * 2;
    constexpr int XR = 2 * R + 2, DR = 2 * R;
    constexpr int XROW = kWgradPitch * 16, DROW = kStripCols * PIX;
    constexpr int XPT = (R * 66 + 511) / 512, DPT = R * 64 * KO / 512;
    constexpr int XN = XR * XROW / 16, DN = DR * DROW / 16;
    __shared__ uint4 lds[XN + DN];
    const uint32_t xbase = (uint32_t)(uintptr_t)(lds_u4*)lds, dbase = xbase + XN * 16;
    const int tid = threadIdx.x, wv = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63;
    const int g = lane >> 4, li = lane & 15;
    StripWalk walk(N, H, W, R);

    f32x4 acc[5][MT], bacc;
#pragma unroll
    for (int j = 0; j < 5; j++)
#pragma unroll
        for (int a = 0; a < MT; a++) acc[j][a] = f32x4{0.f, 0.f, 0.f, 0.f};
    bacc = f32x4{0.f, 0.f, 0.f, 0.f};
    const uint32_t one2 = 0x3F803F80u;
    const bf16x8 ones = as_bf16x8(make_uint4(one2, one2, one2, one2));

    // lane addresses: pixel 4g + (li >> 2); chunks 0, 1 of a narrow tile hold
    // shift 2j's channels, chunks 2, 3 shift 2j + 1's (the tenth: shift 8's)
    const int px = 4 * g + (li >> 2), ch = li & 3;
    int xc[5], xr[5];
    uint32_t da[MT];
#pragma unroll
    for (int j = 0; j < 5; j++) {
        const int s0 = 2 * j, s1 = 2 * j + 1 < 9 ? 2 * j + 1 : 8;
        xc[j] = (px + (ch < 2 ? s0 % 3 : s1 % 3)) * 16 + (ch & 1) * 8;
        xr[j] = ch < 2 ? s0 / 3 : s1 / 3;
    }
#pragma unroll
    for (int a = 0; a < MT; a++) da[a] = dbase + px * PIX + ((a ^ slot_xor<CH>(px)) * 32) + ch * 8;

    uint4 sx[XPT], sd[DPT];
    auto fetch = [&](int n, int c0, int r0) {
#pragma unroll
        for (int j = 0; j < XPT; j++) {
            const int idx = tid + 512 * j;
            const int c = idx % 66, i = idx / 66;
            const int gr = r0 + 1 + i, gc = c0 - 1 + c;
            sx[j] = make_uint4(0, 0, 0, 0);
            if (i < R && gr < H && gc >= 0 && gc < W)
                sx[j] = load8(narrow + (((size_t)n * H + gr) * W + gc) * 8);
        }
#pragma unroll
        for (int j = 0; j < DPT; j++) {
            const int idx = tid + 512 * j;
            const int q = idx % KO, c = (idx / KO) % 64, i = idx / (KO * 64);
            const int gr = r0 + i, gc = c0 + c;
            sd[j] = make_uint4(0, 0, 0, 0);
            if (gr < H && gc < W) sd[j] = load8(wide + (((size_t)n * H + gr) * W + gc) * CH + 8 * q);
        }
    };
    auto put = [&](int xs, int ds) {
#pragma unroll
        for (int j = 0; j < XPT; j++) {
            const int idx = tid + 512 * j;
            const int c = idx % 66, i = idx / 66;
            int s = xs + 2 + i;
            s = s >= XR ? s - XR : s;
            if (i < R) lds[s * kWgradPitch + c] = sx[j];
        }
#pragma unroll
        for (int j = 0; j < DPT; j++) {
            const int idx = tid + 512 * j;
            const int q = idx % KO, c = (idx / KO) % 64, i = idx / (KO * 64);
            lds[XN + ((ds + i) * DROW + c * PIX) / 16 + (((q >> 1) ^ slot_xor<CH>(c)) * 2 + (q & 1))] = sd[j];
        }
    };

    auto top = [&](int n, int c0, int r0) {
        if (tid < 2 * 66) {
            const int c = tid % 66, i = tid / 66;
            const int gr = r0 - 1 + i, gc = c0 - 1 + c;
            uint4 v = make_uint4(0, 0, 0, 0);
            if (gr >= 0 && gr < H && gc >= 0 && gc < W)
                v = load8(narrow + (((size_t)n * H + gr) * W + gc) * 8);
            lds[i * kWgradPitch + c] = v;
        }
    };

    int xs = 0, ds = 0;
    fetch(walk.n, walk.c0, walk.r0);
    top(walk.n, walk.c0, walk.r0);
    put(xs, ds);
    __syncthreads();
    for (;;) {
        const int r = walk.r0 + wv, c0 = walk.c0;           // the wave's row, the strip's first column
        const bool more = --walk.left > 0;
        bool down = false;
        if (more) {
            down = walk.next(R);
            fetch(walk.n, walk.c0, walk.r0);
        }
        uint32_t xo[5];                                     // narrow row wv + (shift's row), per lane
#pragma unroll
        for (int j = 0; j < 5; j++) {
            int row = xs + wv + xr[j];
            row = row >= XR ? row - XR : row;
            xo[j] = xbase + row * XROW + xc[j];
        }
        const uint32_t dof = (uint32_t)((ds + wv) * DROW);
        // output layer, a row or strip at the image's border: a value of x or
        // dy that is not finite
        int own = xs + wv + 1;
        own = own >= XR ? own - XR : own;
        const uint4* mine = lds + own * kWgradPitch + 1;    // dy's pixels beside the wave's
        const bool at_border = r < H && (r == 0 || r == H - 1 || c0 == 0 || W - c0 <= kStripCols);
        bool bad = false;
        if (r < H) {                                        // (a row past the image has nothing to add)
            bf16x8 A[2][MT];
#pragma unroll
            for (int half = 0; half < 2; half++)
#pragma unroll
                for (int a = 0; a < MT; a++) {
                    const uint32_t p = da[a] + dof + half * 32 * PIX;
                    A[half][a] = read_tr8(p, p + 16 * PIX);
                }
            if (OUTL && at_border) {
                bad = not_finite(as_bf16x8(mine[lane]));
#pragma unroll
                for (int half = 0; half < 2; half++)
#pragma unroll
                    for (int a = 0; a < MT; a++) bad |= not_finite(A[half][a]);
                bad = wave_any(bad);
                if (bad) {
#pragma unroll
                    for (int half = 0; half < 2; half++)
#pragma unroll
                        for (int a = 0; a < MT; a++)
                            A[half][a] = border_ones(A[half][a], r == 0 || r == H - 1, g, c0 + 32 * half, W);
                }
            }
#pragma unroll
            for (int half = 0; half < 2; half++) {
                // input layer: the left neighbours of the first column past
                // the image from the column itself, which holds zeros (shifts
                // 0, 3 and 6: chunks 0, 1 of tiles 0 and 3, 2, 3 of tile 1)
                const int past = W - c0 - 32 * half;
                const uint32_t lo = RAGGED && px == past ? 16 : 0, hi = RAGGED && px + 16 == past ? 16 : 0;
#pragma unroll
                for (int j = 0; j < 5; j++) {
                    const bool to_left = !OUTL && RAGGED && (j == 1 ? ch >= 2 : (j == 0 || j == 3) && ch < 2);
                    const uint32_t p = xo[j] + half * 32 * 16;
                    bf16x8 B = read_tr8(p + (to_left ? lo : 0), p + (to_left ? hi : 0) + 16 * 16);
                    if (!OUTL && j == 4) B = li < 8 ? B : ones;
                    if (OUTL && j == 2) bacc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(ones, B, bacc, 0, 0, 0);
#pragma unroll
                    for (int a = 0; a < MT; a++)
                        acc[j][a] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(A[half][a], B, acc[j][a], 0, 0, 0);
                }
            }
        }
        if (OUTL && bad) {
#pragma unroll 1
            for (int i = 0; i < kStripCols && c0 + i < W; i++) {
                int ln = lane;                               // (no register is held for this by the passes)
                asm volatile("" : "+v"(ln));
                const int g = ln >> 4, li = ln & 15;
                const int c = c0 + i;
                const bool edge = r == 0 || r == H - 1 || c == 0 || c == W - 1;
                const bool bad_dy = not_finite16(((const uint16_t*)(mine + i))[li & 7]);
#pragma unroll
                for (int j = 0; j < 5; j++) {
                    const int s = 2 * j + (li >> 3), dr = s / 3 - 1, dc = s % 3 - 1;   // this column's shift
                    const bool in = r + dr >= 0 && r + dr < H && c + dc >= 0 && c + dc < W;
                    int row = xs + wv + 1 + dr;
                    row = row >= XR ? row - XR : row;
                    const uint16_t v = ((const uint16_t*)(lds + row * kWgradPitch + 1 + i + dc))[li & 7];
                    const bool out = r - dr < 0 || r - dr >= H || c - dc < 0 || c - dc >= W;
                    const float none = bad_dy && out ? __builtin_nanf("") : 0.f;
#pragma unroll
                    for (int a = 0; a < MT; a++) {
                        const uint16_t* at = (const uint16_t*)lds + (XN * 16 + (ds + wv) * DROW + i * PIX) / 2 +
                                             (a ^ slot_xor<CH>(i)) * 16 + 4 * g;
#pragma unroll
                        for (int e = 0; e < 4; e++) {
                            const bool add = edge && in && not_finite16(at[e]);
                            acc[j][a][e] += none + (add ? from_bf16(at[e]) * from_bf16(v) : 0.f);
                        }
                    }
                }
            }
        }
        if (!more) break;
        if (down) {
            xs = xs + R >= XR ? xs + R - XR : xs + R;
            ds = R - ds;
        } else {
            __syncthreads();
            xs = ds = 0;
            top(walk.n, walk.c0, walk.r0);
        }
        put(xs, ds);
        __syncthreads();
    }

    // the eight waves' sums: halves added pairwise through LDS, in a fixed order
    f32x4* red = (f32x4*)lds;
    static_assert(4 * (5 * MT + 1) * 64 <= XN + DN, "half of the waves' sums fit the LDS");
#pragma unroll
    for (int o = 4; o > 0; o >>= 1) {
        __syncthreads();
        if (wv >= o && wv < 2 * o) {
#pragma unroll
            for (int j = 0; j < 5; j++)
#pragma unroll
                for (int a = 0; a < MT; a++) red[((j * MT + a) * 4 + wv - o) * 64 + lane] = acc[j][a];
            red[(5 * MT * 4 + wv - o) * 64 + lane] = bacc;
        }
        __syncthreads();
        if (wv < o) {
#pragma unroll
            for (int j = 0; j < 5; j++)
#pragma unroll
                for (int a = 0; a < MT; a++) acc[j][a] += red[((j * MT + a) * 4 + wv) * 64 + lane];
            bacc += red[(5 * MT * 4 + wv) * 64 + lane];
        }
    }
    if (wv != 0) return;
    // D: lane holds wide channel a * 16 + 4 * g + e of shift 2j + (li >> 3),
    // narrow channel li & 7
#pragma unroll
    for (int j = 0; j < 5; j++) {
        const int s = 2 * j + (li >> 3);
#pragma unroll
        for (int a = 0; a < MT; a++)
#pragma unroll
            for (int e = 0; e < 4; e++) {
                const int m = a * 16 + 4 * g + e;
                if (s < 9) {
                    const int t = OUTL ? 8 - s : s;
                    const int i = OUTL ? (li & 7) * CH + m : m * 8 + (li & 7);
                    part[((size_t)t * gridDim.x + blockIdx.x) * CH * 8 + i] = acc[j][a][e];
                } else if (!OUTL && li == 8) {
                    bpart[(size_t)blockIdx.x * CH + m] = acc[j][a][e];
                }
            }
    }
    // the centre shift's columns of dy against ones: every row is the sum
    if (OUTL && g == 0 && li < 8) bpart[(size_t)blockIdx.x * 8 + li] = bacc[0];
}

// dw[t][m][k] = sum_w part[t][w][m][k]; dw has mrows >= my rows per tap
// (rows my .. mrows-1 are left untouched).  A workgroup of 1024 takes 64
// elements, 16 threads each over every sixteenth partial, added through LDS
// in a fixed order (one thread per element over all 256 partials was a chain
// of 256 loads: 110 us whatever the layer).  Grid row 9: the biases.
__global__ __launch_bounds__(1024) void wgrad_reduce_kernel(const float* __restrict__ part,
                                                            const float* __restrict__ bpart, float* __restrict__ dw,
                                                            float* __restrict__ db, int my, int kx, int mrows,
                                                            int waves)
{
    __shared__ float sh[16][64];
    const int t = blockIdx.y;
    const int n = t < 9 ? my * kx : my;
    const int e = threadIdx.x & 63, j = threadIdx.x >> 6;
    const int i = blockIdx.x * 64 + e;
    if (blockIdx.x * 64 >= n) return;                       // whole workgroup
    const float* src = t < 9 ? part + (size_t)t * waves * n : bpart;
    float s = 0.f;
    if (i < n) {
#pragma unroll 16
        for (int w = j; w < waves; w += 16) s += src[(size_t)w * n + i];
    }
    sh[j][e] = s;
    __syncthreads();
    if (j != 0 || i >= n) return;
#pragma unroll
    for (int o = 1; o < 16; o++) s += sh[o][e];
    if (t < 9)
        dw[((size_t)t * mrows + i / kx) * kx + i % kx] = s;
    else
        db[i] = s;
}

// Mean-squared-error gradient of the 4-channel FP32 output against the
// target: dy[p][0..3] = BF16(2 (out - target) / count), dy[p][4..7] = 0; the
// per-block partial sums of squared error go to loss_part (FP64).
__global__ __launch_bounds__(256) void mse_kernel(const float* __restrict__ out, const float* __restrict__ tgt,
                                                  uint16_t* __restrict__ dy, double* __restrict__ loss_part,
                                                  long long npix, float scale)
{
    __shared__ double sh[4];
    double acc = 0.0;
    for (long long p = blockIdx.x * (long long)blockDim.x + threadIdx.x; p < npix;
         p += (long long)gridDim.x * blockDim.x) {
        const float4 o = *(const float4*)(out + 4 * p);
        const float4 y = *(const float4*)(tgt + 4 * p);
        const float d0 = o.x - y.x, d1 = o.y - y.y, d2 = o.z - y.z, d3 = o.w - y.w;
        acc += (double)d0 * d0 + (double)d1 * d1 + (double)d2 * d2 + (double)d3 * d3;
        uint4 st;
        st.x = (uint32_t)to_bf16(scale * d0) | ((uint32_t)to_bf16(scale * d1) << 16);
        st.y = (uint32_t)to_bf16(scale * d2) | ((uint32_t)to_bf16(scale * d3) << 16);
        st.z = 0;
        st.w = 0;
        *(uint4*)(dy + 8 * p) = st;
    }
    for (int off = 32; off > 0; off >>= 1) acc += __shfl_xor(acc, off);
    if ((threadIdx.x & 63) == 0) sh[threadIdx.x >> 6] = acc;
    __syncthreads();
    if (threadIdx.x == 0) loss_part[blockIdx.x] = sh[0] + sh[1] + sh[2] + sh[3];
}

// Adam (Kingma & Ba 2015) with bias correction folded into the step size.
__device__ __forceinline__ float adam_one(float* __restrict__ p, const float* __restrict__ gr, float* __restrict__ m,
                                          float* __restrict__ v, long long i, float lr_t, float b1, float b2, float eps)
{
    const float gi = gr[i];
    const float mi = b1 * m[i] + (1.f - b1) * gi;
    const float vi = b2 * v[i] + (1.f - b2) * gi * gi;
    m[i] = mi;
    v[i] = vi;
    return p[i] -= lr_t * mi / (sqrtf(vi) + eps);
}

__global__ void adam_kernel(float* __restrict__ p, const float* __restrict__ gr, float* __restrict__ m,
                            float* __restrict__ v, long long n, float lr_t, float b1, float b2, float eps)
{
    for (long long i = blockIdx.x * (long long)blockDim.x + threadIdx.x; i < n; i += (long long)gridDim.x * blockDim.x) {
        adam_one(p, gr, m, v, i, lr_t, b1, b2, eps);
    }
}

// The step of a whole network's parameters (layer l's weights [9][m][k], then
// its bias) with every layer's BF16 copies, one parameter per thread: a launch
// for each layer's copies is all latency.  8 images of 256^2: a training step
// of the 32-wide network 206 -> 200 us; the 64-wide one takes the same 692.
//
// A wave takes 8 rows x 8 input channels of a tap, so that the transposed
// copies are written 16 bytes at a time (with a row of 64 channels per wave,
// 2-byte stores to 64 lines each, 697 us).
template <int W>
__global__ __launch_bounds__(256) void adam_pack_kernel(float* __restrict__ p, const float* __restrict__ gr,
                                                        float* __restrict__ m, float* __restrict__ v, float lr_t,
                                                        float b1, float b2, float eps, int mids,
                                                        uint16_t* __restrict__ wb, uint16_t* __restrict__ wt)
{
    constexpr int FIRST = 9 * W * 8, MID = 9 * W * W, LAST = 9 * 16 * W;   // weights of a layer
    const long long i = blockIdx.x * 256LL + threadIdx.x;
    const long long weights = FIRST + mids * (long long)MID + LAST;
    if (i >= weights) {                                                    // a bias
        const long long b = i - weights;
        const long long l = min(b / W, mids + 1LL);
        if (b < (mids + 1LL) * W + 16)
            adam_one(p, gr, m, v, (l <= mids ? FIRST + l * (long long)MID : weights) + b, lr_t, b1, b2, eps);
        return;
    }
    const int l = i < FIRST ? 0 : 1 + (int)min((i - FIRST) / MID, (long long)mids);
    const bool last = l == mids + 1;
    const long long base = l == 0 ? 0 : FIRST + (l - 1) * (long long)MID;  // of the layer in wb
    const int rows = last ? 16 : W, ks = l == 0 ? 8 : W;
    const int at = (int)(i - base), tile = at / 64, lane = at % 64;
    const int t = at / (rows * ks), in_tap = tile - t * (rows * ks / 64);
    const int row = in_tap / (ks / 8) * 8 + lane % 8, k = in_tap % (ks / 8) * 8 + lane / 8;
    const int w = (t * rows + row) * ks + k;
    const uint16_t b = to_bf16(adam_one(p, gr, m, v, base + l * (long long)W + w, lr_t, b1, b2, eps));
    wb[base + w] = b;
    const int mt = last ? 8 : W;
    if (l > 0 && row < mt) wt[base - FIRST + (t * W + k) * mt + row] = b;
}

__global__ void pack_kernel(const float* __restrict__ w, uint16_t* __restrict__ wb, uint16_t* __restrict__ wt, int m,
                            int k, int mt)
{
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= 9 * m * k) return;
    const int t = i / (m * k), rem = i % (m * k), mi = rem / k, ki = rem % k;
    const uint16_t b = to_bf16(w[i]);
    wb[i] = b;
    if (wt && mi < mt) wt[((size_t)t * k + ki) * mt + mi] = b;
}

// ---- ensemble-side kernels -------------------------------------------------
// State planes: h, qx, qy, H, hc (stride nvol); FP32 states add the low
// words of h, H, hc in planes 5, 6, 7.

template <typename S, bool COMP>
__device__ __forceinline__ double plane(const S* V, int f, long long nv, long long p)
{
    double v = (double)V[f * nv + p];
    if (COMP && (f == 0 || f == 3 || f == 4)) v += (double)V[(f == 0 ? 5 : f == 3 ? 6 : 7) * nv + p];
    return v;
}

template <typename S, bool COMP>
__device__ __forceinline__ void store_plane(S* V, int f, long long nv, long long p, double v)
{
    if (COMP && (f == 0 || f == 3 || f == 4)) {
        const float hi = (float)v;
        V[f * nv + p] = (S)hi;
        V[(f == 0 ? 5 : f == 3 ? 6 : 7) * nv + p] = (S)(float)(v - (double)hi);
    } else {
        V[f * nv + p] = (S)v;
    }
}

template <typename S, bool COMP>
__global__ __launch_bounds__(256) void features_kernel(const StageArgs* __restrict__ args, int npx, int npy,
                                                       NnScales sc, uint16_t* __restrict__ x)
{
    const int i = blockIdx.y;
    const S* V = (const S*)args[i].out;
    const double dx = args[i].P->dx, dy = args[i].P->dy;
    const long long nv = (long long)npx * npy;
    for (long long p = blockIdx.x * (long long)blockDim.x + threadIdx.x; p < nv; p += (long long)gridDim.x * blockDim.x) {
        const int r = (int)(p / npx), c = (int)(p % npx);
        const double h = plane<S, COMP>(V, 0, nv, p), H = plane<S, COMP>(V, 3, nv, p);
        const long long pl = c > 0 ? p - 1 : p, pr = c < npx - 1 ? p + 1 : p;
        const long long pd = r > 0 ? p - npx : p, pu = r < npy - 1 ? p + npx : p;
        const double sx = (double)((c > 0) + (c < npx - 1)) * dx, sy = (double)((r > 0) + (r < npy - 1)) * dy;
        const double dzdx = sx > 0 ? (plane<S, COMP>(V, 3, nv, pl) - plane<S, COMP>(V, 3, nv, pr)) / sx : 0.0;
        const double dzdy = sy > 0 ? (plane<S, COMP>(V, 3, nv, pd) - plane<S, COMP>(V, 3, nv, pu)) / sy : 0.0;
        const bool wet = h > sc.wet_h;
        float f[8];
        f[0] = (float)h * sc.in[0];
        f[1] = (float)V[nv + p] * sc.in[1];
        f[2] = (float)V[2 * nv + p] * sc.in[2];
        f[3] = (float)(-H) * sc.in[3];
        f[4] = (float)dzdx * sc.in[4];
        f[5] = (float)dzdy * sc.in[5];
        f[6] = wet ? (float)(h - H) * sc.in[6] : 0.f;
        f[7] = wet ? sc.in[7] : 0.f;
        uint4 st;
        st.x = (uint32_t)to_bf16(f[0]) | ((uint32_t)to_bf16(f[1]) << 16);
        st.y = (uint32_t)to_bf16(f[2]) | ((uint32_t)to_bf16(f[3]) << 16);
        st.z = (uint32_t)to_bf16(f[4]) | ((uint32_t)to_bf16(f[5]) << 16);
        st.w = (uint32_t)to_bf16(f[6]) | ((uint32_t)to_bf16(f[7]) << 16);
        *(uint4*)(x + ((size_t)i * nv + p) * 8) = st;
    }
}

// The correction changes depths and momenta, so the dt the last stage left
// for the next step (from the uncorrected state) no longer bounds it.  The
// corrected members' dt slots are re-armed and apply_kernel refills them from
// the corrected state, as the initial dt is computed (GPU/main_TSUNER.cu:
// 147-148), on the stream and without a host round trip.
__global__ void apply_dt_reset_kernel(const StageArgs* __restrict__ args, int n, long long expect)
{
    const int i = (blockIdx.x * blockDim.x + threadIdx.x) / kDtSlots, slot = threadIdx.x % kDtSlots;
    if (i >= n) return;
    if (args[i].ctrl->step == expect) args[i].dts->v[expect & 1][slot][0] = kInfBits;
}

// Bound by its memory accesses, up to 150 bytes of a cell with running
// maxima.  A cell's loads are issued before the first is used, and the time
// step's minimum is taken here: 32 members of 256^2 cells 94 us and 16 us for
// a pass of its own over the state, now 90 us.
template <typename S, bool COMP>
__global__ __launch_bounds__(256) void apply_kernel(const StageArgs* __restrict__ args, int npx, int npy, NnScales sc,
                                                    const float* __restrict__ out, long long expect,
                                                    float* __restrict__ resid, const uint16_t* __restrict__ x)
{
    const int i = blockIdx.y;
    const StageArgs& a = args[i];
    if (a.ctrl->step != expect) return;
    S* V = (S*)a.out;
    const DevParams& P = *a.P;
    const double eps_h = P.epsilon_h;
    const long long nv = (long long)npx * npy;
    // wet flag (input channel 7) of cell q before this correction
    auto wet_in = [&](long long q) -> bool { return x[((size_t)i * nv + q) * 8 + 7] != 0; };
    float rmax = 0.f;
    const double inf = __longlong_as_double((long long)kInfBits);
    double dt = inf;
    for (long long p = blockIdx.x * (long long)blockDim.x + threadIdx.x; p < nv; p += (long long)gridDim.x * blockDim.x) {
        // every load of the cell before its first use
        const float4 o = *(const float4*)(out + ((size_t)i * nv + p) * 4);
        S hs = V[p], qxs = V[nv + p], qys = V[2 * nv + p];
        const double h = plane<S, COMP>(V, 0, nv, p), H = plane<S, COMP>(V, 3, nv, p);
        double peak[3] = {0.0, 0.0, 0.0};
        if (a.ext)
            for (int j = 0; j < 3; j++) peak[j] = a.ext[j * nv + p];
        double h2 = h + (double)(o.x * sc.out[0]);
        double H2 = H;
        bool corrected = true;
        if (h > sc.wet_h) {
            // residual indicator: largest correction of the surface (h - H)
            rmax = fmaxf(rmax, fabsf(o.x * sc.out[0] - o.w * sc.out[3]));
            if (!(h2 > 0.0)) h2 = 0.0;
            H2 = H + (double)(o.w * sc.out[3]);
        } else {
            // a dry cell is wetted only on the shoreline (a wet neighbour in
            // the network's inputs) and only deeper than shore_h; the bed of
            // dry cells is left alone
            corrected = false;
            if (x && h2 > sc.shore_h) {
                const int r = (int)(p / npx), c = (int)(p % npx);
                corrected = (c > 0 && wet_in(p - 1)) || (c < npx - 1 && wet_in(p + 1)) ||
                            (r > 0 && wet_in(p - npx)) || (r < npy - 1 && wet_in(p + npx));
            }
        }
        if (corrected) {
            double qx = 0.0, qy = 0.0;
            if (h2 > 0.0) {
                qx = (double)qxs + (double)(o.y * sc.out[1]);
                qy = (double)qys + (double)(o.z * sc.out[2]);
            }
            store_plane<S, COMP>(V, 0, nv, p, h2);
            store_plane<S, COMP>(V, 1, nv, p, qx);
            store_plane<S, COMP>(V, 2, nv, p, qy);
            store_plane<S, COMP>(V, 3, nv, p, H2);
            if (h2 == 0.0) store_plane<S, COMP>(V, 4, nv, p, 0.0);
            // what the stage kernels fold and the time step reads: the stored
            // leading words (FP32: hi)
            hs = (S)h2;
            qxs = (S)qx;
            qys = (S)qy;
            if (a.ext) {
                const double hx = (double)hs, Hx = (double)(S)H2;
                if (hx > eps_h) {
                    a.ext[p] = fmax(peak[0], hx);
                    a.ext[2 * nv + p] = fmax(peak[2], hx - Hx);
                }
                a.ext[nv + p] = fmax(peak[1], Hx);
            }
        }
        dt = fmin(dt, (double)cell_dt(P, hs, qxs, qys));
    }
    for (int o = 32; o > 0; o >>= 1) dt = fmin(dt, __shfl_xor(dt, o, 64));
    if ((threadIdx.x & 63) == 0 && dt < inf)
        atomicMin(&a.dts->v[expect & 1][blockIdx.x & (kDtSlots - 1)][0],
                  (unsigned long long)__double_as_longlong(dt));
    if (resid) {
        // one atomic per workgroup (the early return above is uniform over
        // it: one member per grid row); non-negative floats order like their
        // bit patterns
        __shared__ float wmax[4];
        for (int off = 32; off > 0; off >>= 1) rmax = fmaxf(rmax, __shfl_xor(rmax, off));
        if ((threadIdx.x & 63) == 0) wmax[threadIdx.x >> 6] = rmax;
        __syncthreads();
        if (threadIdx.x == 0) {
            const float m = fmaxf(fmaxf(wmax[0], wmax[1]), fmaxf(wmax[2], wmax[3]));
            if (m > 0.f) atomicMax((unsigned int*)(resid + i), __float_as_uint(m));
        }
    }
}

// Free-surface restriction of the 4x4 block of fine cells under coarse cell
// (r, c): bed = block mean of H; surface = mean of h - H over the block's wet
// fine cells (h > kRestrictWetH), depth = max(surface + bed, 0) (0 when no
// fine cell is wet); discharge and suspended load = the block totals of q and
// hc scaled by depth / block total of h (mass-weighted velocity and
// concentration times the new depth).  A lake at rest restricts to a lake at
// rest: a block mean of h would lift the surface of every block that
// straddles the shoreline.
template <typename S, bool COMP>
__device__ __forceinline__ void restrict_block(const S* F, long long fnv, int fnx, int r, int c, double v[5])
{
    double sh = 0.0, sqx = 0.0, sqy = 0.0, sH = 0.0, shc = 0.0, seta = 0.0;
    int nw = 0;
    for (int dr = 0; dr < 4; dr++)
        for (int dc = 0; dc < 4; dc++) {
            const long long q = (long long)(4 * r + dr) * fnx + 4 * c + dc;
            const double h = plane<S, COMP>(F, 0, fnv, q), H = plane<S, COMP>(F, 3, fnv, q);
            sh += h;
            sqx += plane<S, COMP>(F, 1, fnv, q);
            sqy += plane<S, COMP>(F, 2, fnv, q);
            sH += H;
            shc += plane<S, COMP>(F, 4, fnv, q);
            if (h > kRestrictWetH) {
                seta += h - H;
                nw++;
            }
        }
    const double Hc = sH * 0.0625;
    const double hc = nw ? fmax(seta / (double)nw + Hc, 0.0) : 0.0;
    const double k = (hc > 0.0 && sh > 0.0) ? hc / sh : 0.0;
    v[0] = hc;
    v[1] = sqx * k;
    v[2] = sqy * k;
    v[3] = Hc;
    v[4] = shc * k;
}

template <typename S, bool COMP>
__global__ __launch_bounds__(256) void restrict_kernel(const StageArgs* __restrict__ fine,
                                                       const StageArgs* __restrict__ coarse, int npx, int npy)
{
    const int i = blockIdx.y;
    const S* F = (const S*)fine[i].out;
    S* Cs = (S*)coarse[i].out;
    const long long nv = (long long)npx * npy, fnv = 16 * nv;
    const int fnx = 4 * npx;
    for (long long p = blockIdx.x * (long long)blockDim.x + threadIdx.x; p < nv; p += (long long)gridDim.x * blockDim.x) {
        double v[5];
        restrict_block<S, COMP>(F, fnv, fnx, (int)(p / npx), (int)(p % npx), v);
        for (int f = 0; f < 5; f++) store_plane<S, COMP>(Cs, f, nv, p, v[f]);
    }
}

template <typename S, bool COMP>
__global__ __launch_bounds__(256) void target_kernel(const StageArgs* __restrict__ fine,
                                                     const StageArgs* __restrict__ coarse, int npx, int npy,
                                                     NnScales sc, float* __restrict__ target)
{
    const int i = blockIdx.y;
    const S* F = (const S*)fine[i].out;
    const S* Cs = (const S*)coarse[i].out;
    const long long nv = (long long)npx * npy, fnv = 16 * nv;
    const int fnx = 4 * npx;
    for (long long p = blockIdx.x * (long long)blockDim.x + threadIdx.x; p < nv; p += (long long)gridDim.x * blockDim.x) {
        double v[5];
        restrict_block<S, COMP>(F, fnv, fnx, (int)(p / npx), (int)(p % npx), v);
        float o[4];
        for (int j = 0; j < 4; j++) o[j] = (float)((v[j] - plane<S, COMP>(Cs, j, nv, p)) / (double)sc.out[j]);
        *(float4*)(target + ((size_t)i * nv + p) * 4) = make_float4(o[0], o[1], o[2], o[3]);
    }
}

}  // namespace nn

using namespace nn;

namespace {
dim3 member_grid(long long nv, int n)
{
    long long b = (nv + 255) / 256;
    if (b > 1024) b = 1024;
    return dim3((unsigned)b, (unsigned)n);
}
}  // namespace

hipError_t nn_launch_features(const StageArgs* args, int n, int npx, int npy, int precision, const NnScales& sc,
                              uint16_t* x, hipStream_t s)
{
    const dim3 g = member_grid((long long)npx * npy, n);
    if (precision == 0)
        features_kernel<double, false><<<g, 256, 0, s>>>(args, npx, npy, sc, x);
    else
        features_kernel<float, true><<<g, 256, 0, s>>>(args, npx, npy, sc, x);
    return hipGetLastError();
}

hipError_t nn_launch_apply(const StageArgs* args, int n, int npx, int npy, int precision, const NnScales& sc,
                           const float* out, long long expect_step, float* resid, const uint16_t* x,
                           hipStream_t s)
{
    const dim3 g = member_grid((long long)npx * npy, n);
    apply_dt_reset_kernel<<<(n * kDtSlots + 63) / 64, 64, 0, s>>>(args, n, expect_step);
    if (precision == 0)
        apply_kernel<double, false><<<g, 256, 0, s>>>(args, npx, npy, sc, out, expect_step, resid, x);
    else
        apply_kernel<float, true><<<g, 256, 0, s>>>(args, npx, npy, sc, out, expect_step, resid, x);
    return hipGetLastError();
}

hipError_t nn_launch_restrict(const StageArgs* fine, const StageArgs* coarse, int n, int npx, int npy,
                              int precision, hipStream_t s)
{
    const dim3 g = member_grid((long long)npx * npy, n);
    if (precision == 0)
        restrict_kernel<double, false><<<g, 256, 0, s>>>(fine, coarse, npx, npy);
    else
        restrict_kernel<float, true><<<g, 256, 0, s>>>(fine, coarse, npx, npy);
    return hipGetLastError();
}

hipError_t nn_launch_target(const StageArgs* fine, const StageArgs* coarse, int n, int npx, int npy, int precision,
                            const NnScales& sc, float* target, hipStream_t s)
{
    const dim3 g = member_grid((long long)npx * npy, n);
    if (precision == 0)
        target_kernel<double, false><<<g, 256, 0, s>>>(fine, coarse, npx, npy, sc, target);
    else
        target_kernel<float, true><<<g, 256, 0, s>>>(fine, coarse, npx, npy, sc, target);
    return hipGetLastError();
}

namespace {
// One workgroup per stretch of passes, as many as the chip holds at once.
template <int K, int MTW, int MG, int RG, int MOUT, int SIGN, int POST>
hipError_t launch_conv(const uint16_t* in, const uint16_t* w, const float* bias, const uint16_t* act, void* out, int N,
                       int H, int W, hipStream_t s)
{
    constexpr int R = conv_rows<K>(), lds = conv_ring(R) * (kStripCols + 2) * K * 2;
    // by LDS (160 KB) and by waves per SIMD
    constexpr int by_lds = 163840 / lds, by_waves = conv_waves<K>() / (MG * RG);
    constexpr int per_cu = by_lds < by_waves ? by_lds : (by_waves > 0 ? by_waves : 1);
    int dev = 0, cus = 0;
    if (hipGetDevice(&dev) != hipSuccess ||
        hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || cus < 1)
        cus = 256;
    const long long passes = (long long)N * ((W + kStripCols - 1) / kStripCols) * ((H + R - 1) / R);
    const long long most = (long long)cus * per_cu;
    conv_kernel<K, MTW, MG, RG, MOUT, SIGN, POST><<<(unsigned)(passes < most ? passes : most), 256 * MG * RG, 0, s>>>(
        in, w, bias, act, out, N, H, W);
    return hipGetLastError();
}
}  // namespace

hipError_t nn_launch_conv(int kind, const uint16_t* in, const uint16_t* w, const float* bias, const uint16_t* act,
                          void* out, int N, int H, int W, hipStream_t s)
{
    switch (kind) {
    case NN_FWD_IN:      // 8 -> 32, ReLU
        return launch_conv<8, 2, 1, 1, 32, 1, 0>(in, w, bias, act, out, N, H, W, s);
    case NN_FWD_MID:     // 32 -> 32, ReLU
        return launch_conv<32, 2, 1, 1, 32, 1, 0>(in, w, bias, act, out, N, H, W, s);
    case NN_FWD_OUT:     // 32 -> 4 (weights padded to 16 rows), FP32 out
        return launch_conv<32, 1, 1, 1, 4, 1, 1>(in, w, bias, act, out, N, H, W, s);
    case NN_DGRAD_OUT:   // dy 8 channels (4 used) -> dx 32, ReLU mask
        return launch_conv<8, 2, 1, 1, 32, -1, 2>(in, w, bias, act, out, N, H, W, s);
    case NN_DGRAD_MID:   // dy 32 -> dx 32, ReLU mask
        return launch_conv<32, 2, 1, 1, 32, -1, 2>(in, w, bias, act, out, N, H, W, s);
    case NN_FWD_IN | NN_W64:
        return launch_conv<8, 2, 2, 1, 64, 1, 0>(in, w, bias, act, out, N, H, W, s);
    case NN_FWD_MID | NN_W64:
        return launch_conv<64, 2, 2, 1, 64, 1, 0>(in, w, bias, act, out, N, H, W, s);
    case NN_FWD_OUT | NN_W64:
        return launch_conv<64, 1, 1, 2, 4, 1, 1>(in, w, bias, act, out, N, H, W, s);
    case NN_DGRAD_OUT | NN_W64:
        return launch_conv<8, 2, 2, 1, 64, -1, 2>(in, w, bias, act, out, N, H, W, s);
    case NN_DGRAD_MID | NN_W64:
        return launch_conv<64, 2, 2, 1, 64, -1, 2>(in, w, bias, act, out, N, H, W, s);
    default:
        return hipErrorInvalidValue;
    }
}

hipError_t nn_launch_wgrad(int kind, const uint16_t* x, const uint16_t* dy, float* part, float* bpart, float* dw,
                           float* db, int mrows, int N, int H, int W, hipStream_t s)
{
    // one workgroup per stretch of passes, at most kWgradWaves (the partial
    // sums the workspace holds)
    const int width = (kind & NN_W64) ? 64 : 32, base = kind & ~NN_W64;
    const bool mid = base == NN_WGRAD_MID;
    const int rows = mid ? 4 : 8;                       // rows per pass (R of the kernels)
    const long long passes = (long long)N * ((W + kStripCols - 1) / kStripCols) * ((H + rows - 1) / rows);
    const int waves = (int)(passes < kWgradWaves ? passes : kWgradWaves);
    int my = width, kx = width;
    // a: the kernel's first operand; ragged: for widths with a remainder
    typedef void (*Kernel)(const uint16_t*, const uint16_t*, float*, float*, int, int, int);
    auto launch = [&](Kernel whole, Kernel ragged, const uint16_t* a, const uint16_t* b) {
        (W % kStripCols ? ragged : whole)<<<waves, 512, 0, s>>>(a, b, part, bpart, N, H, W);
    };
    switch (kind) {
    case NN_WGRAD_IN:
        launch(wgrad_edge_kernel<32, false, false>, wgrad_edge_kernel<32, false, true>, dy, x);
        kx = 8;
        break;
    case NN_WGRAD_MID:
        launch(wgrad_mid_kernel<32, false>, wgrad_mid_kernel<32, true>, x, dy);
        break;
    case NN_WGRAD_OUT:
        launch(wgrad_edge_kernel<32, true, false>, wgrad_edge_kernel<32, true, false>, x, dy);
        my = 8;
        break;
    case NN_WGRAD_IN | NN_W64:
        launch(wgrad_edge_kernel<64, false, false>, wgrad_edge_kernel<64, false, true>, dy, x);
        kx = 8;
        break;
    case NN_WGRAD_MID | NN_W64:
        launch(wgrad_mid_kernel<64, false>, wgrad_mid_kernel<64, true>, x, dy);
        break;
    case NN_WGRAD_OUT | NN_W64:
        launch(wgrad_edge_kernel<64, true, false>, wgrad_edge_kernel<64, true, false>, x, dy);
        my = 8;
        break;
    default:
        return hipErrorInvalidValue;
    }
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;
    wgrad_reduce_kernel<<<dim3((my * kx + 63) / 64, 10), 1024, 0, s>>>(part, bpart, dw, db, my, kx, mrows, waves);
    return hipGetLastError();
}

hipError_t nn_launch_mse(const float* out, const float* tgt, uint16_t* dy, double* loss_part, int nblocks,
                         long long npix, float scale, hipStream_t s)
{
    mse_kernel<<<nblocks, 256, 0, s>>>(out, tgt, dy, loss_part, npix, scale);
    return hipGetLastError();
}

hipError_t nn_launch_adam(float* p, const float* g, float* m, float* v, long long n, float lr_t, float b1, float b2,
                          float eps, hipStream_t s)
{
    adam_kernel<<<(unsigned)((n + 255) / 256 < 1024 ? (n + 255) / 256 : 1024), 256, 0, s>>>(p, g, m, v, n, lr_t, b1,
                                                                                           b2, eps);
    return hipGetLastError();
}

hipError_t nn_launch_adam_pack(float* p, const float* g, float* m, float* v, float lr_t, float b1, float b2, float eps,
                               int width, int mids, uint16_t* wb, uint16_t* wt, hipStream_t s)
{
    const long long n = 9LL * width * 8 + width + mids * (9LL * width * width + width) + 9LL * 16 * width + 16;
    const unsigned blocks = (unsigned)((n + 255) / 256);
    if (width == 32)
        adam_pack_kernel<32><<<blocks, 256, 0, s>>>(p, g, m, v, lr_t, b1, b2, eps, mids, wb, wt);
    else
        adam_pack_kernel<64><<<blocks, 256, 0, s>>>(p, g, m, v, lr_t, b1, b2, eps, mids, wb, wt);
    return hipGetLastError();
}

hipError_t nn_launch_pack(const float* w, uint16_t* wb, uint16_t* wt, int m, int k, int mt, hipStream_t s)
{
    const int n = 9 * m * k;
    pack_kernel<<<(n + 255) / 256, 256, 0, s>>>(w, wb, wt, m, k, mt);
    return hipGetLastError();
}

}  // namespace tsu
