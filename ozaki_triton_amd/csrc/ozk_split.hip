// ozk_split.hip -- the split planner (which kernel of ozk_split_kernels.h takes
// an operand) and the kernels without a slice type: exchange-word clears, the
// status of the cooperative launches, the transpose and the conversion of
// narrow inputs.
#include "ozk_common.h"
#include "ozk_internal.h"
#include "ozk_split_launch.h"

#include <atomic>
#include <stdlib.h>
#include <string.h>

namespace ozk {

__global__ __launch_bounds__(256) void zero_u64_kernel(uint64_t *p, int64_t n) {
    for (int64_t i = blockIdx.x * 256 + threadIdx.x; i < n; i += (int64_t)gridDim.x * 256) p[i] = 0;
}

// Sticky device status: bit 0 = a cooperative wait gave up since the last
// clear (read and cleared by read_device_status).
__device__ uint32_t g_device_status = 0;

// After a cooperative launch: if any member gave up its wait (status != 0),
// every scale of the split becomes NaN, so no entry of C computed from it can
// pass for a valid result, and the sticky device status records it.
__global__ __launch_bounds__(256) void poison_scales_kernel(const uint32_t *status, float *scales,
                                                            int64_t batch, int L, int64_t rows,
                                                            int64_t cs_b, int64_t cs_l,
                                                            int64_t cs_r) {
    if (*status == 0) return;
    const int64_t n = batch * L * rows;
    for (int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x; i < n;
         i += (int64_t)gridDim.x * 256) {
        const int64_t r = i % rows, l = (i / rows) % L, b = i / (rows * L);
        scales[b * cs_b + l * cs_l + r * cs_r] = __int_as_float(0x7fc00000);
    }
    if (blockIdx.x == 0 && threadIdx.x == 0)
        __hip_atomic_fetch_or(&g_device_status, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
}

// ---------------------------------------------------------------------------
// Transpose of a row-contiguous operand (xs_r == 1, the B^T view) into a
// K-contiguous workspace [batch, rows, K], for K too long for the column
// kernels; a row kernel then splits the workspace.  64 x 64 tiles through
// LDS: loads are 16 bytes per lane along the rows, stores 16 bytes along K.
// ---------------------------------------------------------------------------
template <typename XT>
__global__ __launch_bounds__(256) void transpose_kernel(const XT *__restrict__ X, int64_t batch,
                                                        int64_t rows, int64_t K, int64_t xs_b,
                                                        int64_t xs_k, XT *__restrict__ T) {
    constexpr int TILE = 64;
    constexpr int VEC = 16 / (int)sizeof(XT);
    // element alignment only: rows of any pitch, K of any length
    typedef XT vec_t __attribute__((ext_vector_type(VEC), aligned(sizeof(XT))));
    __shared__ XT tile[TILE][TILE + 1];
    const int64_t tiles_r = (rows + TILE - 1) / TILE;
    const int64_t tiles_k = (K + TILE - 1) / TILE;
    const int64_t tb = blockIdx.x;
    const int64_t b = tb / (tiles_r * tiles_k);
    const int64_t rem = tb % (tiles_r * tiles_k);
    const int64_t r0 = (rem % tiles_r) * TILE;
    const int64_t k0 = (rem / tiles_r) * TILE;
    const XT *xb = X + b * xs_b;
    // load: a lane covers VEC consecutive rows of one k (one 16-byte load where
    // they all exist)
    constexpr int LPR = TILE / VEC;              // lanes per k-row of the tile
    constexpr int KPP = 256 / LPR;               // k-rows per pass
    const int lr = threadIdx.x % LPR, lk = threadIdx.x / LPR;
#pragma unroll
    for (int kk = 0; kk < TILE; kk += KPP) {
        const int64_t k = k0 + kk + lk;
        const int64_t r = r0 + lr * VEC;
        XT v[VEC];
        if (k < K && r + VEC <= rows) {
            const vec_t w = *(const vec_t *)(xb + k * xs_k + r);
#pragma unroll
            for (int u = 0; u < VEC; ++u) v[u] = w[u];
        } else {
#pragma unroll
            for (int u = 0; u < VEC; ++u)
                v[u] = (k < K && r + u < rows) ? xb[k * xs_k + r + u] : (XT)0;
        }
#pragma unroll
        for (int u = 0; u < VEC; ++u) tile[kk + lk][lr * VEC + u] = v[u];
    }
    __syncthreads();
    // store: a lane covers VEC consecutive k of one row
    XT *tb_out = T + b * rows * K;
#pragma unroll
    for (int rr = 0; rr < TILE; rr += KPP) {
        const int64_t r = r0 + rr + lk;
        const int64_t k = k0 + lr * VEC;
        if (r < rows && k + VEC <= K) {
            vec_t w;
#pragma unroll
            for (int u = 0; u < VEC; ++u) w[u] = tile[lr * VEC + u][rr + lk];
            *(vec_t *)(tb_out + r * K + k) = w;
        } else if (r < rows) {
            for (int u = 0; u < VEC && k + u < K; ++u)
                tb_out[r * K + k + u] = tile[lr * VEC + u][rr + lk];
        }
    }
}

// ---------------------------------------------------------------------------
// Exact conversion of a narrow input (fp16 / bf16 / int8, any strides) into
// an fp32 copy [batch, rows, K] in the workspace.  A thread converts 4
// consecutive k of one row; rows run fastest when the operand's rows are
// contiguous (the B^T view), so loads stay coalesced either way.
// ---------------------------------------------------------------------------
template <typename XT>
__global__ __launch_bounds__(256) void convert_kernel(const XT *__restrict__ X, int64_t batch,
                                                      int64_t rows, int64_t K, int64_t xs_b,
                                                      int64_t xs_r, int64_t xs_k,
                                                      float *__restrict__ T, int rows_fast) {
    const int64_t kq = (K + 3) / 4;
    const int64_t total = batch * rows * kq;
    for (int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x; i < total;
         i += (int64_t)gridDim.x * 256) {
        int64_t r, q;
        if (rows_fast) {
            r = i % rows;
            q = (i / rows) % kq;
        } else {
            q = i % kq;
            r = (i / kq) % rows;
        }
        const int64_t b = i / (rows * kq);
        const XT *src = X + b * xs_b + r * xs_r;
        float *dst = T + (b * rows + r) * K;
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            const int64_t k = 4 * q + u;
            if (k < K) dst[k] = (float)src[k * xs_k];
        }
    }
}

// ---------------------------------------------------------------------------
// Planning and launch.  Rows and columns of K <= 8192 belong to the classes of
// split_fused_kernel; the variants after them are longer rows (one workgroup
// of 8 or 16 waves per row) and columns (16-byte strips).
// ---------------------------------------------------------------------------
static const int64_t kRowLimits[] = {256, 512, 1024, 2048, 4096, 8192, 16384, 32768, 65536};
static const int64_t kColLimits[] = {256, 512, 1024, 2048, 4096, 8192, 16384};
// the class or variant of a row / column of K elements, -1 if too long (fp64
// rows keep at most 32 values per lane)
static int row_variant(int64_t K, int xsz) {
    for (int i = 0; i < 9; ++i)
        if (K <= kRowLimits[i]) return i == 8 && xsz == 8 ? -1 : i;
    return -1;
}
static int col_variant(int64_t K) {
    for (int i = 0; i < 7; ++i)
        if (K <= kColLimits[i]) return i;
    return -1;
}

// exchange words plus the launch's status word (none without an exchange)
static size_t slot_bytes(int64_t nslots) { return nslots > 0 ? (size_t)(nslots + 1) * 8 : 0; }
static size_t rows_coop_slot_bytes(const SplitParams &p, int xsz) {
    return slot_bytes(rows_coop_slots(p, xsz));
}
static size_t round256(size_t x) { return (x + 255) / 256 * 256; }

static bool aligned(const void *ptr, int64_t bytes) {
    return ((uintptr_t)ptr % (uintptr_t)bytes) == 0;
}

static int dtype_size(int code) {
    switch (code) {
    case 0: return 8;           // f64
    case 1: return 4;           // f32
    case 2: case 3: return 2;   // f16, bf16
    default: return 1;          // i8
    }
}

// layout of the fp32 copy a narrow input (fp16 / bf16 / int8) is split from
static SplitParams converted_params(const SplitParams &p) {
    SplitParams q = p;
    q.xs_b = p.rows * p.K;
    q.xs_r = p.K;
    q.xs_k = 1;
    return q;
}

// ---------------------------------------------------------------------------
// Residency limit of the cooperative kernels.  The members of a group are
// consecutive workgroup ids and workgroups are dispatched in id order.  While
// the group of the oldest unfinished workgroup is not wholly resident, every
// workgroup that holds back the next id is a member of that group: the ids
// before it have finished, the next id is the group's own.  If the hardware
// sends each id to a fixed XCD, that XCD is full of members; if to any XCD
// with room, every XCD is.  Either way the group has more members than one
// XCD holds, so a group of at most that many (less a margin of 8) always
// becomes resident and its waits end.  One XCD holds the kernels' occupancy
// (the fewest workgroups per CU over every kernel that waits) times its CUs:
// 32 on gfx950, or all of a smaller partition.  Asked once per device; where
// the runtime cannot say (no device: a workspace query on a host without a
// GPU) MI355X's figure is assumed: 2 workgroups per CU (the kernels with
// up to 175 VGPRs, one wave per SIMD each, fit twice in 512), so 64 per XCD
// and at most 56 members (the row kernel's 64 chunks are cut to 56).
// ---------------------------------------------------------------------------
constexpr int kCusPerXcd = 32;
constexpr int kMi355xResident = 2 * kCusPerXcd;

int coop_resident_per_xcd() {
    if (debug_overrides().coop_resident > 0) return debug_overrides().coop_resident;
    static std::atomic<int> cached[64];
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= 64) return kMi355xResident;
    int r = cached[dev].load(std::memory_order_relaxed);
    if (r > 0) return r;
    int cus = 0, occ = 1 << 20;
    bool ok = hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) ==
                  hipSuccess && cus > 0;
    if (ok) {
        SplitLaunch<int8_t>::coop_occupancy(occ, ok);
        SplitLaunch<_Float16>::coop_occupancy(occ, ok);
        SplitLaunch<__bf16>::coop_occupancy(occ, ok);
        SplitLaunch<float>::coop_occupancy(occ, ok);
    }
    if (!ok) {
        (void)hipGetLastError();   // a failed query is not a launch error
        return kMi355xResident;
    }
    r = occ * (cus < kCusPerXcd ? cus : kCusPerXcd);
    cached[dev].store(r, std::memory_order_relaxed);
    return r;
}

// the most members a cooperative group may have on the current device (at
// least 1: a group of one never waits)
static int64_t coop_member_limit(int64_t kernel_max) {
    const int64_t r = (int64_t)coop_resident_per_xcd() - 8;
    return r < 1 ? 1 : (r < kernel_max ? r : kernel_max);
}

static SplitPlan plan_split_raw(const SplitParams &p, int x_dtype, int slice_dtype) {
    const int xsz = dtype_size(x_dtype);
    const int ssz = dtype_size(slice_dtype);
    const int force = debug_overrides().split;
    auto forced = [&](int which) { return force == which; };
    // everything but the generic kernel: slices along K from a base aligned to
    // four of them, element-aligned input, rows or columns contiguous
    const bool ok = p.ss_k == 1 && aligned(p.slices, 4 * ssz) && aligned(p.X, xsz);
    const bool rows_ok = ok && p.xs_k == 1, cols_ok = ok && !rows_ok && p.xs_r == 1;
    if (x_dtype >= 2) {
        // narrow inputs: converted as they are loaded (the fused kernel), else
        // into the workspace first and split as fp32 (X is replaced by the
        // workspace at launch, which is 16-byte aligned; the plan of the copy
        // is taken with that assumption).  A forced kernel is one of the fp32
        // copy's
        const int v = row_variant(p.Kp, 4);
        if (force == kForceSplitNone && (rows_ok || cols_ok) && v >= 0 && v < kFusedClasses)
            return {rows_ok ? kSplitRows : kSplitStrip, v};
        return {kSplitConvert, 0};
    }
    // the test hooks (include/ozaki_amd_debug.h) steer column operands to the
    // coop / strip / transpose / generic path, or force one of the two row
    // kernels; a path whose requirements fail is not taken
    // long rows: the row kernel shared by workgroups
    const bool rows_coop = rows_coop_members(p.K, xsz) <= coop_member_limit(kRowsCoopMaxP) &&
                           (forced(kForceSplitRowsCoop) || (!forced(kForceSplitRows) && p.K > kRowsCoopMinK));
    const int rv = row_variant(p.Kp, xsz);
    if (rows_ok && !forced(kForceSplitGeneric)) {
        if (rows_coop) return {kSplitRows, kRowsCoopVariant};
        if (rv >= 0) return {kSplitRows, rv};
    }
    // columns of 64 KB and more: the cooperative kernel.  Alone against one
    // workgroup's column groups, us, 2 int8 slices, 1024 / 2048 / 8192 columns:
    // f64 K = 8192 27.6 (26.9) / 41.3 (48.4) / 154 (250), K = 16384 45.8 (51.5) /
    // 108 (141) / 294 (542); f32 K = 16384 53.0 (34.6) / 81.4 (63.2) / 334 (382).
    // Shorter columns lose: f64 K = 2048 22.5 (14.3) / 21.3 (14.6) / 37.6 (31.9),
    // f32 K = 4096 21.4 (14.0) / 24.1 (15.8) / 59.6 (47.3), K = 8192 26.5 (20.0) /
    // 43.9 (33.1) / 154 (176).  The line lies where it lay against column groups one
    // 16-byte load wide, as does that of the 32 KB columns of fp64 into 1 or 2
    // int8 slices, 2048 or more: even those are no longer faster this way (27.0
    // against 22.2 at 2048 columns, 94.8 against 94.9 at 8192; the whole call, M x
    // N = 1024 x 4096, 2 slices, 114 against 97).  A forced coop takes it for any
    // length it holds
    const int64_t coop_max = coop_member_limit(kCoopMaxP);
    const bool coop_fits = cols_ok && coop_members(p.K, xsz, 8) <= coop_max;
    // columns too long for 32 chunks of 128-byte groups: 32-byte groups, whose
    // chunks hold 4x the rows, when the cooperative kernel is forced.  By
    // default such columns are transposed instead: at config 5 (fp32, K =
    // 65536, 32 chunks of 2048 rows) the 32-byte groups took 0.255-0.265 ms
    // against 0.216 ms for the transpose path, the exchange waiting on 32
    // members per group.
    const bool coop2_fits = cols_ok && !coop_fits && coop_members(p.K, xsz, 2) <= coop_max;
    const bool other = forced(kForceSplitStrip) || forced(kForceSplitTranspose) || forced(kForceSplitGeneric);
    const bool coop_long = p.K * xsz >= kCoopMinColumnBytes ||
                           (xsz == 8 && ssz == 1 && p.L <= 2 &&
                            p.K * xsz >= kCoopMinColumnBytes / 2 && p.batch * p.rows >= 2048);
    if (coop_fits && (forced(kForceSplitCoop) || (!other && coop_long))) return {kSplitCoop, 8};
    if (coop2_fits && forced(kForceSplitCoop)) return {kSplitCoop, 2};
    if (cols_ok && !forced(kForceSplitTranspose) && !forced(kForceSplitGeneric)) {
        const int v = col_variant(p.Kp);
        if (v >= 0) return {kSplitStrip, v};
    }
    // row-contiguous operand with a K too long for a resident strip: transpose
    // into the workspace, then the row kernel (if the row fits)
    if (cols_ok && !forced(kForceSplitGeneric)) {
        if (rows_coop) return {kSplitTransposeRows, kRowsCoopVariant};
        if (rv >= 0) return {kSplitTransposeRows, rv};
    }
    return {kSplitGeneric, 0};
}


// Operands that are not whole 16-byte pieces (K, row pitch, alignment) can do
// without scratch: long ones take a cooperative or transposing plan where there
// is scratch for it, else the generic kernel.  Callers that own a buffer of one
// size (ozk_matmul_static, or ozk_split without a workspace) need no room for
// them.  Whole operands must have what their plan needs.
static bool scratch_optional(const SplitParams &p, int x_dtype, int slice_dtype) {
    const int xsz = dtype_size(x_dtype), ssz = dtype_size(slice_dtype);
    const bool slices_whole = p.ss_k == 1 && aligned(p.slices, 4 * ssz) && p.ss_r % 4 == 0 &&
                              p.ss_l % 4 == 0 && p.ss_b % 4 == 0;
    if (p.K % 4 != 0 || !slices_whole) return true;
    if (x_dtype >= 2) return false;   // split from a whole fp32 copy
    return !aligned(p.X, 16) ||
           (p.xs_k == 1 && ((p.xs_r * xsz) % 16 != 0 || (p.xs_b * xsz) % 16 != 0));
}
// the plan without scratch of its own (a narrow input keeps its fp32 copy)
static SplitPlan plan_without_scratch(int x_dtype) {
    return x_dtype >= 2 ? SplitPlan{kSplitConvert, kConvertGeneric} : SplitPlan{kSplitGeneric, 0};
}

SplitPlan plan_split(const SplitParams &p, int x_dtype, int slice_dtype, size_t scratch) {
    const SplitPlan plan = plan_split_raw(p, x_dtype, slice_dtype);
    const size_t need = split_workspace_bytes(p, plan, x_dtype, slice_dtype);
    if (need > scratch && scratch_optional(p, x_dtype, slice_dtype))
        return plan_without_scratch(x_dtype);
    if (aligned(p.X, 16) && aligned(p.slices, 16)) return plan;   // the aligned plan
    // other pointers: no more scratch than the workspace queries reserve for
    // aligned ones, which see no pointers (the generic kernel needs none)
    SplitParams q = p;
    q.X = (const void *)(uintptr_t)256;
    q.slices = (void *)(uintptr_t)256;
    const SplitPlan ref = plan_split_raw(q, x_dtype, slice_dtype);
    if (need > split_workspace_bytes(q, ref, x_dtype, slice_dtype))
        return plan_without_scratch(x_dtype);
    return plan;
}

// plan of the fp32 copy of a narrow input (its X is the 16-byte aligned
// workspace: `aligned` in plan_split must see an aligned pointer)
static SplitPlan converted_plan(const SplitParams &p, const SplitPlan &plan, int slice_dtype) {
    if (plan.variant == kConvertGeneric) return {kSplitGeneric, 0};
    SplitParams q = converted_params(p);
    q.X = (const void *)(uintptr_t)256;
    return plan_split(q, 1, slice_dtype);
}

// What is transposed at a time: the whole operand, or where it could do without
// scratch at most kTransposePart bytes (so that such operands, which the generic
// kernel splits with none, do not take their own size of it): whole batches or
// rows of one, 64 rows or more.  Split alone, us, parts of 64 / 128 MiB / whole:
// 900 rows of 33001 f64 -> 1 int8 199 / 176 / 173, 4000 -> 4 1123 / 885 / 889,
// 1000 of 65535 f32 -> 3 285 / 231 / 243, 3000 of 20001 f32 -> 2 249 / 210 / 231.
constexpr int64_t kTransposePart = (int64_t)128 << 20;
static SplitParams transpose_part(const SplitParams &p, int x_dtype, int slice_dtype) {
    SplitParams q = p;
    if (p.K == 0 || !scratch_optional(p, x_dtype, slice_dtype)) return q;
    const int64_t n = kTransposePart / (p.K * dtype_size(x_dtype)) / 64 * 64;
    const int64_t rows = n > 64 ? n : 64;
    if (p.rows > rows) {
        q.batch = 1;
        q.rows = rows;
    } else if (p.batch * p.rows > rows) {
        q.batch = rows / p.rows;
    }
    return q;
}

size_t split_workspace_bytes(const SplitParams &p, const SplitPlan &plan, int x_dtype,
                             int slice_dtype) {
    const int64_t n = p.batch * p.rows * p.K;
    if (plan.path == kSplitConvert) {
        const SplitPlan inner = converted_plan(p, plan, slice_dtype);
        const size_t in = split_workspace_bytes(converted_params(p), inner, 1, slice_dtype);
        return in ? round256((size_t)(n * 4)) + in : (size_t)(n * 4);
    }
    // a narrow input the fused kernel converts as it loads it: the size of the
    // copy stays reserved, for other pointers and forced kernels
    if (x_dtype >= 2) return (size_t)(n * 4);
    if (plan.path == kSplitTransposeRows) {
        const SplitParams q = transpose_part(p, x_dtype, slice_dtype);
        const size_t tb = (size_t)(q.batch * q.rows * q.K * dtype_size(x_dtype));
        if (plan.variant != kRowsCoopVariant) return tb;
        return round256(tb) + rows_coop_slot_bytes(q, dtype_size(x_dtype));
    }
    if (plan.path == kSplitRows && plan.variant == kRowsCoopVariant)
        return rows_coop_slot_bytes(p, dtype_size(x_dtype));
    if (plan.path == kSplitCoop) return slot_bytes(coop_slots(p, dtype_size(x_dtype), plan.variant));
    return 0;
}

// Clears n exchange words and the status word after them.
hipError_t clear_slots(uint64_t *slot, int64_t n, hipStream_t st) {
    const int64_t zb = (n + 256) / 256 < 2048 ? (n + 256) / 256 : 2048;
    hipLaunchKernelGGL(zero_u64_kernel, dim3((unsigned)zb), dim3(256), 0, st, slot, n + 1);
    return hipGetLastError();
}

hipError_t launch_poison(const SplitParams &p, const uint64_t *status, hipStream_t st) {
    if (p.fail_out) {   // the cross-GEMM that follows checks the word instead
        *p.fail_out = (const uint32_t *)status;
        return hipSuccess;
    }
    const int64_t n = p.batch * p.L * p.rows;
    const int64_t nb = (n + 255) / 256 < 1024 ? (n + 255) / 256 : 1024;
    hipLaunchKernelGGL(poison_scales_kernel, dim3((unsigned)nb), dim3(256), 0, st,
                       (const uint32_t *)status, p.scales, p.batch, p.L, p.rows, p.cs_b, p.cs_l,
                       p.cs_r);
    return hipGetLastError();
}

WaitRule wait_rule() {
    const bool force = debug_overrides().coop_timeout != 0;
    return {(uint32_t)(kCoopTag >> 32) + (force ? 1u : 0u), force ? 0ull : kCoopTickLimit};
}

// calls SplitLaunch<ST>::f for the slice dtype
template <typename F> static hipError_t with_slice(int slice_dtype, F &&f) {
    switch (slice_dtype) {
    case 4: return f(SplitLaunch<int8_t>{});
    case 2: return f(SplitLaunch<_Float16>{});
    case 3: return f(SplitLaunch<__bf16>{});
    case 1: return f(SplitLaunch<float>{});
    }
    return hipErrorInvalidValue;
}

// a plan of split_fused_kernel
static bool fused_plan(const SplitPlan &plan) {
    return (plan.path == kSplitRows || plan.path == kSplitStrip) && plan.variant < kFusedClasses;
}
static SplitParams fused_params(const SplitParams &p, const SplitPlan &plan, int x_dtype) {
    SplitParams q = p;
    q.cols = plan.path == kSplitStrip;
    q.x_code = x_dtype;
    q.row_mul = 0;
    if (!q.cols && p.batch > 1 && p.rows > 1 && p.batch * p.rows < (int64_t)1 << 31) {
        // the smallest s with rows <= 2^s; 2^(31+s) / rows rounded up is exact
        // for every row below 2^31: row * (row_mul * rows - 2^(31+s)) < 2^(31+s)
        int s = 0;
        while (((int64_t)1 << s) < p.rows) ++s;
        q.row_mul = (uint32_t)((((uint64_t)1 << (31 + s)) + (uint64_t)p.rows - 1) / (uint64_t)p.rows);
        q.row_shift = s - 1;
    }
    return q;
}
// Width of the column groups (SplitLaunch::fused): wide ones where they are
// as many as MI355X's CUs or more (at K = 2048, twice as many): one step
// below, they measured 1.1-1.3x slower than the narrow ones, from there on
// 1.05-1.2x faster.
static int fused_width(const SplitParams &p, int cls, int x_dtype) {
    if (!p.cols) return 0;
    // columns of a wide group (0: none) and the fewest groups
    static const int kWide64[kFusedClasses][2] = {{0, 0}, {0, 0}, {8, 256}, {8, 512}, {4, 256}, {0, 0}};
    static const int kWide32[kFusedClasses][2] = {{0, 0}, {0, 0}, {0, 0}, {0, 0}, {8, 256}, {0, 0}};
    const int *w = x_dtype == 0 ? kWide64[cls] : kWide32[cls];
    return w[0] && p.batch * ((p.rows + w[0] - 1) / w[0]) >= w[1] ? 2 : 1;
}

template <typename XT>
static hipError_t launch_transpose(const SplitParams &p, XT *T, hipStream_t st) {
    const int64_t tiles = p.batch * ((p.rows + 63) / 64) * ((p.K + 63) / 64);
    hipLaunchKernelGGL((transpose_kernel<XT>), dim3((unsigned)tiles), dim3(256), 0, st,
                       (const XT *)p.X, p.batch, p.rows, p.K, p.xs_b, p.xs_k, T);
    return hipGetLastError();
}

template <typename XT>
static hipError_t launch_convert(const SplitParams &p, float *T, hipStream_t st) {
    const int64_t total = p.batch * p.rows * ((p.K + 3) / 4);
    if (total == 0) return hipSuccess;
    int64_t blocks = (total + 255) / 256;
    if (blocks > 65536) blocks = 65536;
    const int rows_fast = (p.xs_r == 1 && p.xs_k != 1);
    hipLaunchKernelGGL((convert_kernel<XT>), dim3((unsigned)blocks), dim3(256), 0, st,
                       (const XT *)p.X, p.batch, p.rows, p.K, p.xs_b, p.xs_r, p.xs_k, T,
                       rows_fast);
    return hipGetLastError();
}

// f on parts of an operand, `batch` batches of `rows` rows each or fewer.
template <typename F>
static hipError_t for_parts(const SplitParams &p, int64_t batch, int64_t rows, int x_dtype,
                            int slice_dtype, F &&f) {
    const int xsz = dtype_size(x_dtype), ssz = dtype_size(slice_dtype);
    for (int64_t b = 0; b < p.batch; b += batch)
        for (int64_t r = 0; r < p.rows; r += rows) {
            SplitParams q = p;
            q.batch = p.batch - b < batch ? p.batch - b : batch;
            q.rows = p.rows - r < rows ? p.rows - r : rows;
            q.X = (const char *)p.X + (b * p.xs_b + r * p.xs_r) * xsz;
            q.slices = (char *)p.slices + (b * p.ss_b + r * p.ss_r) * ssz;
            q.scales = p.scales + b * p.cs_b + r * p.cs_r;
            // the parts share one status word: each checks its own
            if (q.batch != p.batch || q.rows != p.rows) q.fail_out = nullptr;
            if (hipError_t e = f(q)) return e;
        }
    return hipSuccess;
}

// A launch counts its work-items in 32 bits, and split_fused_kernel takes up to
// 256 for a row: the rows of one launch, beside columns.
constexpr int64_t kFusedRows = (int64_t)1 << 23;
static bool fused_in_one(const SplitParams &p, const SplitPlan &plan) {
    return plan.path != kSplitRows || p.batch * p.rows <= kFusedRows;
}

hipError_t launch_split(const SplitParams &p, const SplitPlan &plan, int x_dtype,
                        int slice_dtype, hipStream_t st) {
    if (p.batch * p.rows == 0 || p.L == 0) return hipSuccess;
    if (fused_plan(plan) && !fused_in_one(p, plan)) {
        const int64_t rows = p.rows < kFusedRows ? p.rows : kFusedRows;
        return for_parts(p, kFusedRows / rows, rows, x_dtype, slice_dtype, [&](const SplitParams &q) {
            return launch_split(q, plan, x_dtype, slice_dtype, st);
        });
    }
    if (fused_plan(plan)) {
        const SplitParams q = fused_params(p, plan, x_dtype);
        return with_slice(slice_dtype, [&](auto s) {
            return s.fused(&q, nullptr, plan.variant, fused_width(q, plan.variant, x_dtype), x_dtype,
                           st);
        });
    }
    if (plan.path == kSplitConvert) {
        // narrow input: convert into the workspace, then split the fp32 copy
        // (any scratch that split needs follows the copy)
        float *T = p.resid;
        hipError_t e;
        if (x_dtype == 2) e = launch_convert<_Float16>(p, T, st);
        else if (x_dtype == 3) e = launch_convert<__bf16>(p, T, st);
        else e = launch_convert<int8_t>(p, T, st);
        if (e != hipSuccess) return e;
        SplitParams q = converted_params(p);
        q.X = T;
        q.resid = (float *)((char *)T + round256((size_t)(p.batch * p.rows * p.K) * 4));
        return launch_split(q, converted_plan(p, plan, slice_dtype), 1, slice_dtype, st);
    }
    if (plan.path == kSplitTransposeRows) {
        // workspace: [batch, rows, K] of a part, then the shared row kernel's
        // exchange words
        const SplitParams part = transpose_part(p, x_dtype, slice_dtype);
        const int xsz = dtype_size(x_dtype);
        const size_t tb = (size_t)(part.batch * part.rows * p.K) * xsz;
        return for_parts(p, part.batch, part.rows, x_dtype, slice_dtype, [&](SplitParams q) {
            const hipError_t e = x_dtype == 0 ? launch_transpose<double>(q, (double *)p.resid, st)
                                              : launch_transpose<float>(q, p.resid, st);
            if (e != hipSuccess) return e;
            q.X = p.resid;
            q.xs_b = q.rows * q.K;
            q.xs_r = q.K;
            q.xs_k = 1;
            q.resid = (float *)((char *)p.resid + round256(tb));
            return launch_split(q, {kSplitRows, plan.variant}, x_dtype, slice_dtype, st);
        });
    }
    return with_slice(slice_dtype, [&](auto s) { return s.one(p, plan, x_dtype, st); });
}

bool split_pair_ok(const SplitPlan &plan_a, const SplitPlan &plan_b, int x_dtype) {
    return x_dtype == 0 && pair_nc(plan_a) != 0 && plan_b.path == kSplitCoop &&
           plan_b.variant == 8 && debug_overrides().split == kForceSplitNone;
}

hipError_t launch_split_pair(const SplitParams &pa, const SplitPlan &plan_a,
                             const SplitParams &pb, const SplitPlan &plan_b, int x_dtype,
                             int slice_dtype, hipStream_t st) {
    if (!split_pair_ok(plan_a, plan_b, x_dtype)) return hipErrorInvalidValue;
    if (pa.batch * pa.rows == 0 || pb.batch * pb.rows == 0 || pa.L == 0) return hipSuccess;
    return with_slice(slice_dtype, [&](auto s) { return s.pair(pa, plan_a, pb, st); });
}

bool split_fused_ok(const SplitPlan &plan_a, const SplitPlan &plan_b) {
    return debug_overrides().split == kForceSplitNone && fused_plan(plan_a) && fused_plan(plan_b) &&
           plan_a.variant == plan_b.variant;
}

hipError_t launch_split_fused(const SplitParams &pa, const SplitPlan &plan_a, const SplitParams &pb,
                              const SplitPlan &plan_b, int x_dtype, int slice_dtype,
                              hipStream_t st) {
    if (!split_fused_ok(plan_a, plan_b)) return hipErrorInvalidValue;
    if (pa.batch * pa.rows == 0 || pb.batch * pb.rows == 0 || pa.L == 0) return hipSuccess;
    if (!fused_in_one(pa, plan_a) || !fused_in_one(pb, plan_b)) {
        if (hipError_t e = launch_split(pb, plan_b, x_dtype, slice_dtype, st)) return e;
        return launch_split(pa, plan_a, x_dtype, slice_dtype, st);
    }
    const SplitParams qa = fused_params(pa, plan_a, x_dtype), qb = fused_params(pb, plan_b, x_dtype);
    const int wa = fused_width(qa, plan_a.variant, x_dtype);
    const int wb = fused_width(qb, plan_b.variant, x_dtype);
    const int width = wa > wb ? wa : wb;
    return with_slice(slice_dtype, [&](auto s) {
        return s.fused(&qb, &qa, plan_a.variant, width, x_dtype, st);
    });
}

uint32_t *device_status_word() {
    static std::atomic<uint32_t *> cached[64];
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= 64) return nullptr;
    uint32_t *ptr = cached[dev].load(std::memory_order_acquire);
    if (!ptr) {
        void *addr = nullptr;
        if (hipGetSymbolAddress(&addr, HIP_SYMBOL(g_device_status)) != hipSuccess) return nullptr;
        ptr = (uint32_t *)addr;
        cached[dev].store(ptr, std::memory_order_release);
    }
    return ptr;
}

hipError_t read_device_status(unsigned *out, bool clear, hipStream_t st) {
    uint32_t v = 0;
    hipError_t e = hipMemcpyFromSymbolAsync(&v, HIP_SYMBOL(g_device_status), sizeof(v), 0,
                                            hipMemcpyDeviceToHost, st);
    if (e == hipSuccess) e = hipStreamSynchronize(st);
    if (e == hipSuccess && clear && v != 0) {
        const uint32_t zero = 0;
        e = hipMemcpyToSymbolAsync(HIP_SYMBOL(g_device_status), &zero, sizeof(zero), 0,
                                   hipMemcpyHostToDevice, st);
        if (e == hipSuccess) e = hipStreamSynchronize(st);
    }
    *out = v;
    return e;
}

}  // namespace ozk
