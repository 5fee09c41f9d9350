// Many rows against weights that have to be the CPU's, round(round(code * scale) + bias) (reference:
// crates/nuvec-core/src/kernels.rs:835-859; product kernels.rs:1091-1142): the weight is dequantized once into a workspace
// (affine_dequantize_kernel) and multiplied densely, in bfloat16 or float16 on v_mfma_f32_32x32x16.
//
// The tiled kernel that expands codes itself (qmk_kernel.h) does so for every 128 rows of x, and two roundings a weight make it bound by
// the vector unit: 517 rows, W[4096,4096] of 3 bits, 50 us.  A weight of N x K costs 2 N K bytes written and, from the chip's last
// cache, read.
//
// A block of four wavefronts owns BM x 128 of y, 128 or 256 rows of x, each wavefront BM / 2 x 64, and walks K in steps of 64
// through a ring of LDS stages that both operands reach by direct loads, as many as fit; layout, swizzle and order of K are
// those of qmm_kernel.h, whose x tile is either operand here.  Bound by LDS reads: one operand of 16 bytes a lane per matrix
// instruction at 128 rows, three per four at 256 (a step takes 0.5 and 0.85 us; operands laid out tile by tile beforehand, so
// that a load is 1 KB of consecutive bytes, took 0.55; eight wavefronts with a quarter of every window each, the two of a SIMD reading and
// multiplying by turns with a barrier each, 0.65).
// us, 4 bits, bfloat16, codes expanded in the product -> here: W[4096,4096] at 517 / 2048 rows 46 / 94 -> 41 / 72; W[6144,8192] at 768
// rows 134 -> 120; 3 bits W[4096,4096] at 517 rows 50 -> 40, 6 bits W[4064,7680] at 1519 rows 147 -> 110.
#include "qmm_kernel.h"

namespace nvq {
namespace {

using namespace qmm;

template <int TI_, int RING>
struct Dense {
    static constexpr int TI = TI_, TJ = 2, kRing = RING, BM = 64 * TI, BN = 128, kThreads = 256;
    static constexpr int kXBytes = BM * kRowBytes, kStageBytes = (BM + BN) * kRowBytes, kLdsBytes = kRing * kStageBytes;
    static constexpr int XP = BM * 8 / kThreads, WP = BN * 8 / kThreads, kParts = XP + WP;  // loads a step: of x, then of the weight
};
using Small = Dense<2, 5>;
using Big = Dense<4, 3>;

template <typename T, class D>
__global__ void __launch_bounds__(D::kThreads, 1) qmm_dense_kernel(const ProductArgs a, const int64_t ldy, const T *__restrict__ weights) {
    constexpr int TI = D::TI, TJ = D::TJ, XP = D::XP, kThreads = D::kThreads;
    constexpr int kAhead = D::kRing - 1;  // steps under way
    extern __shared__ __attribute__((aligned(16))) unsigned char lds[];
    const uint32_t lds0 = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) unsigned char *)lds;
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wm = wave >> 1, wn = wave & 1, h = lane >> 5, l32 = lane & 31;
    const int K = (int)a.k, N = (int)a.n, M = (int)a.m, steps = K / BK;  // K is a multiple of 64 (checked on the host)
    const int m0 = blockIdx.y * D::BM, n0 = blockIdx.x * D::BN;
    const char *xbase = reinterpret_cast<const char *>((const T *)a.x + (int64_t)m0 * K), *wbase = reinterpret_cast<const char *>(weights + (int64_t)n0 * K);

    // Instruction i of wavefront v fills the 64 consecutive 16-byte slots from slot i * kThreads + v * 64 on of its operand's
    // tile; slot S is row S / 8 and holds chunk S % 8 ^ swizzle(row).  Rows past the ends repeat the last one.
    uint32_t off[D::kParts];
#pragma unroll
    for (int i = 0; i < D::kParts; i++) {
        const bool is_x = i < XP;
        const int slot = (is_x ? i : i - XP) * kThreads + tid, row = slot >> 3, chunk = (slot & 7) ^ swizzle(row);
        const int last = is_x ? M - 1 - m0 : N - 1 - n0;
        off[i] = ((uint32_t)(row < last ? row : last) * (uint32_t)K + chunk * 8) * 2;
    }
    const uint32_t lds_wave = lds0 + wave * 64 * 16;
    // Load `i` of a step (past the end: the last step again, which keeps the wait counts uniform).
    auto issue = [&](int step, int stage, auto i_tag) {
        constexpr int i = decltype(i_tag)::value;
        const int sc = step < steps ? step : steps - 1;
        dma<4>((i < XP ? xbase : wbase) + sc * (BK * 2), off[i],
               lds_wave + stage * D::kStageBytes + (i < XP ? i * kThreads * 16 : D::kXBytes + (i - XP) * kThreads * 16));
    };
    // Item t of substep kk's operands, of the step in `stage`: TI of x, then TJ of the weights.
    uint4 af[2][TI], bf[2][TJ];
    auto read = [&](int stage, auto kk_tag, auto t_tag) {
        constexpr int kk = decltype(kk_tag)::value, t = decltype(t_tag)::value;
        const unsigned char *from = lds + stage * D::kStageBytes;
        if constexpr (t < TI) af[kk & 1][t] = *reinterpret_cast<const uint4 *>(from + lds_offset(wm * (32 * TI) + t * 32 + l32, 4 * h + kk));
        else bf[kk & 1][t - TI] = *reinterpret_cast<const uint4 *>(from + D::kXBytes + lds_offset(wn * (32 * TJ) + (t - TI) * 32 + l32, 4 * h + kk));
    };
    floatx16_t acc[TI][TJ];
#pragma unroll
    for (int i = 0; i < TI; i++)
#pragma unroll
        for (int j = 0; j < TJ; j++)
#pragma unroll
            for (int e = 0; e < 16; e++) acc[i][j][e] = 0.0f;

    static_for<kAhead>([&](auto s) { static_for<D::kParts>([&](auto i) { issue(decltype(s)::value, decltype(s)::value, i); }); });
    dma_wait<(kAhead - 1) * D::kParts>();
    __syncthreads();
    using c0 = std::integral_constant<int, 0>;
    static_for<TI + TJ>([&](auto t) { read(0, c0{}, t); });
    int stage = 0, last = kAhead;  // step % D::kRing, (step + kAhead) % D::kRing
    for (int step = 0; step < steps; step++) {
        const int stage1 = stage == kAhead ? 0 : stage + 1;
        static_for<4>([&](auto kk_tag) {
            constexpr int kk = decltype(kk_tag)::value, next = (kk + 1) & 3;
            // a quarter of the loads of step + kAhead, into the stage that everyone left at the last barrier
            static_for<D::kParts / 4>([&](auto p) { issue(step + kAhead, last, std::integral_constant<int, kk * (D::kParts / 4) + decltype(p)::value>{}); });
            if constexpr (kk == 3) {  // the next step has landed for everyone, and everyone is done reading this one
                dma_wait<(kAhead - 1) * D::kParts>();
                __syncthreads();
            }
            static_for<TI * TJ>([&](auto q_tag) {
                constexpr int q = decltype(q_tag)::value, i = q % TI, j = q / TI;
                acc[i][j] = Ops<T>::mfma(af[kk & 1][i], bf[kk & 1][j], acc[i][j]);
                static_for<TI + TJ>([&](auto t_tag) {
                    constexpr int t = decltype(t_tag)::value;
                    if constexpr (t >= q * (TI + TJ) / (TI * TJ) && t < (q + 1) * (TI + TJ) / (TI * TJ))
                        read(kk == 3 ? stage1 : stage, std::integral_constant<int, next>{}, t_tag);
                });
                pin();
            });
        });
        last = stage, stage = stage1;
    }
    dma_wait<0>();

    // Accumulator element e of a 32 x 32 tile is row 8 (e / 4) + 4 (lane / 32) + e % 4, column lane % 32.
    uint16_t *y = reinterpret_cast<uint16_t *>(a.y);
#pragma unroll
    for (int i = 0; i < TI; i++)
#pragma unroll
        for (int j = 0; j < TJ; j++) {
            const int col = n0 + wn * (32 * TJ) + j * 32 + l32, row0 = m0 + wm * (32 * TI) + i * 32 + 4 * h;
            if (col >= N) continue;
#pragma unroll
            for (int e = 0; e < 16; e += 2) {
                const uint32_t pair = Ops<T>::pack(add_row_bias<T>(a.row_bias, acc[i][j][e], col), add_row_bias<T>(a.row_bias, acc[i][j][e + 1], col));
                const int row = row0 + 8 * (e >> 2) + (e & 3);
                if (row < M) y[row * ldy + col] = (uint16_t)pair;
                if (row + 1 < M) y[(row + 1) * ldy + col] = (uint16_t)(pair >> 16);
            }
        }
}

template <typename T, class D>
int32_t run_tile(const ProductArgs &a, int64_t ldy, const void *weights, hipStream_t s) {
    static std::atomic<bool> configured = false;
    if (!configured) {
        NVQ_HIP_TRY(hipFuncSetAttribute(reinterpret_cast<const void *>(qmm_dense_kernel<T, D>), hipFuncAttributeMaxDynamicSharedMemorySize, D::kLdsBytes));
        configured = true;
    }
    const dim3 grid((unsigned)((a.n + D::BN - 1) / D::BN), (unsigned)((a.m + D::BM - 1) / D::BM));
    hipLaunchKernelGGL((qmm_dense_kernel<T, D>), grid, dim3(D::kThreads), D::kLdsBytes, s, a, ldy, (const T *)weights);
    NVQ_LAUNCH_CHECK("qmm_dense");
    return NVQ_OK;
}

// Microseconds of the dequantization and the product by tiles of either height: launches and ends of kernels, a weight written and read,
// more beyond what the caches keep, rounds of a tile per compute unit, outputs.  Fitted to 1400 timings of both heights (100 to 2048 rows, 1 to 8
// bits; 7 and 4 % off).
template <class D>
double dense_us(const ProductArgs &a) {
    const double tiles = (double)((a.m + D::BM - 1) / D::BM) * (double)((a.n + D::BN - 1) / D::BN), rounds = ceil(tiles / fmax(1.0, (double)compute_units()));
    const double steps = (double)(a.k / BK), weights = 1.0e-6 * (double)a.n * (double)a.k, outputs = 1.0e-6 * (double)a.m * (double)a.n;
    const double fill = (double)a.m / (double)((a.m + D::BM - 1) / D::BM * D::BM);  // (rows past the end are one row's bytes)
    const double beyond = fmax(0.0, weights - 25.0);
    return D::TI == 2 ? 5.9 + 0.465 * weights + 0.213 * beyond + rounds * (3.1 + (0.133 + 0.347 * fill) * steps) + 0.63 * outputs
                      : 4.6 + 0.39 * weights + 0.17 * beyond + rounds * (7.15 + (0.537 + 0.129 * fill) * steps) + 0.69 * outputs;
}

// The entry point without a workspace has the bits of the one with it.  It makes the copy in the library's scratch, a larger one in parts of weight
// rows unless run_tiled's tile that sums in this kernel's order, K whole, is estimated faster (few tiles a part).  us, that tile -> here: 4 bits
// W[4096,4096] at 517 rows 69 -> 44, 3 bits W[8035,6912] at 1702 rows 380 -> 222, 4 bits W[6144,8192] at 768 rows 198 -> 165; W[7786,11264] of
// 5 bits at 337 rows 205 there, 328 in parts.
constexpr size_t kScratch = NVQ_STATIC_SCRATCH_BYTES;
// Rows of a part: whole tiles, where they fit, and eight at least, whose codes are whole pieces of 16 bytes.
int64_t rows_of_a_part(const ProductArgs &a, size_t bytes) {
    const int64_t most = (int64_t)(bytes / (size_t)(2 * a.k)) / 8 * 8;
    if (most == 0) return 0;
    const int64_t parts = (a.n + most - 1) / most, rows = ((a.n + parts - 1) / parts + 127) / 128 * 128;
    return rows < most ? rows : most;
}
double parts_us(const ProductArgs &all) {
    ProductArgs a = all;
    a.n = rows_of_a_part(all, kScratch);
    return a.n == 0 ? HUGE_VAL : (double)((all.n + a.n - 1) / a.n) * fmin(dense_us<Small>(a), dense_us<Big>(a));
}
double whole_us(const ProductArgs &a) {
    const splits::Product p = split_product(a);
    return splits::qmm_tiles_us(p, splits::kSmall, splits::qmm_tiles(p, splits::kSmall), a.k / BK, 1, compute_units() < 1 ? 1 : compute_units());
}

}  // namespace

size_t qmm_dense_workspace_bytes(const ProductArgs &a) { return (size_t)a.n * (size_t)a.k * 2; }

// Half a gigabyte of workspace, W[8191,28672] and a little more: a weight that takes the CPU's values has fewer than 8192 rows.
constexpr int64_t kMostWeights = 1LL << 28;

// Among the products that the tiled kernels take with the CPU's weights: where it is estimated at most 4 % slower (705 products timed on both:
// 0.2 % above always taking the faster one, a dozen more than 5 %; without the 4 % twelve of 398 others of more than 640 rows are more than 5 %
// slower than before qmk_kernel, with it eight).  us here / there, 4 bits, on both sides of the line: W[4096,4096] at 517 / 576 / 640 / 768 rows
// 41 / 46, 44 / 43, 49 / 43, 49 / 44; W[6144,8192] at 640 / 768 rows 95 / 81 and 120 / 134; W[6144,4096] at 517 rows 48 / 47; W[4096,8192] at 768 rows
// 86 / 79; 3 bits W[6144,8192] at 517 rows 83 / 88.
bool qmm_dense_takes(const ProductArgs &a) {
    if (a.mode != NVQ_AFFINE || !a.exact_weights || a.row_exact || a.batch != 1 || a.batch_ndim != 0 || a.rhs != nullptr || a.lhs != nullptr || a.glu != 0)
        return false;
    if (a.k < BK || a.k % BK != 0 || a.k > 1 << 22 || (a.m + 127) / 128 > 65535) return false;  // (32-bit offsets in a tile)
    if (a.n * a.k > kMostWeights) return false;
    return fmin(dense_us<Small>(a), dense_us<Big>(a)) < 1.04 * qmm_estimate_us(a);
}

// The bytes of the copy that the kernel is given at a time where `most` are there; 0: run_tiled's tile is the faster one then.
size_t qmm_dense_bytes(const ProductArgs &a, size_t most) {
    const size_t all = qmm_dense_workspace_bytes(a);
    return all <= most ? all : parts_us(a) < whole_us(a) ? most : 0;
}

// Fewer bytes than the whole copy take it in parts, each multiplied before the next overwrites it: bit for bit the same.
int32_t launch_qmm_dense(const ProductArgs &all, void *workspace, size_t bytes, hipStream_t s) {
    const int64_t rows = bytes < qmm_dense_workspace_bytes(all) ? rows_of_a_part(all, bytes) : all.n;
    if (rows == 0) return fail(NVQ_BACKEND, "quantized_matmul: %zu bytes hold too few rows of K = %lld", bytes, (long long)all.k);
    const int64_t groups = all.k / all.group, words = all.k / 32 * all.bits;
    for (int64_t first = 0; first < all.n; first += rows) {
        ProductArgs a = all;
        a.n = all.n - first < rows ? all.n - first : rows;
        a.w = (const uint32_t *)all.w + first * words;
        a.scales = (const uint16_t *)all.scales + first * groups, a.biases = (const uint16_t *)all.biases + first * groups;
        a.y = (uint16_t *)all.y + first;
        if (all.row_bias != nullptr) a.row_bias = (const uint16_t *)all.row_bias + first;
        const int32_t rc = launch_affine_dequantize(a.dtype, a.group, a.bits, a.w, a.scales, a.biases, a.n * a.k, workspace, nullptr, a.k, a.n, s);
        if (rc != NVQ_OK) return rc;
        const bool big = dense_us<Big>(a) < dense_us<Small>(a);
        const int32_t done = a.dtype == NVQ_BF16 ? (big ? run_tile<bf16_t, Big>(a, all.n, workspace, s) : run_tile<bf16_t, Small>(a, all.n, workspace, s))
                                                 : (big ? run_tile<f16_t, Big>(a, all.n, workspace, s) : run_tile<f16_t, Small>(a, all.n, workspace, s));
        if (done != NVQ_OK) return done;
    }
    return NVQ_OK;
}

}  // namespace nvq
