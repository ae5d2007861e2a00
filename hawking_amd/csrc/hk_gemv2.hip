// hk_gemv2.hip -- GEMV over sets of packed organs on the int8 matrix cores
// (engine in hk_mfma.h), plus the dense f32 GEMV used for the router.
//
// Grid: (workgroups per organ, organs).  A workgroup of 4 waves loads x once
// (ahead of its first weight loads), builds the x image in LDS, then each wave
// walks groups of R consecutive row tiles
// (16 rows each) of its slice of the organ; one LDS operand fetch feeds the R
// tiles' MFMAs and the next step's weight loads are in flight while the
// current step computes.
#include <type_traits>

#include "hk_mfma.h"
#include "hk_rice.h"

namespace hk {

// The item sequence of one wave: groups k = 0..ng-1 of R tiles starting at
// g0 + k*gstride, each over steps 0..S-1.
struct WaveItems {
    uint32_t g0, gstride, t1, steps, n;
    __device__ void at(uint32_t it, uint32_t* T, int R, int* nvalid, uint32_t* t) const {
        const uint32_t k = it / steps, g = g0 + k * gstride;
        *t = it % steps;
        for (int r = 0; r < R; ++r) T[r] = g + (uint32_t)r;
        *nvalid = (int)min((uint32_t)R, t1 - g);
    }
};

// A pipeline slot's walk over a wave's items: D items ahead at a time
// without a division per item (D / steps and D % steps once), clamped at
// the last item (past the end a slot re-reads it).  g = the slot's tile
// group start, t = its step.
template <int D>
struct ItemStride {
    uint32_t dq, dr, glast, tlast;
    __device__ __forceinline__ void init(const WaveItems& W, uint32_t last) {
        dq = (uint32_t)D / W.steps;
        dr = (uint32_t)D % W.steps;
        glast = W.g0 + (last / W.steps) * W.gstride;
        tlast = last % W.steps;
    }
    // slot (g, t) from item nx - D to item nx (nx > last: the last item)
    __device__ __forceinline__ void next(const WaveItems& W, uint32_t nx, uint32_t last, uint32_t* T, int R,
                                         int* nvalid, uint32_t* t) const {
        uint32_t g = T[0], s = *t + dr;
        g += dq * W.gstride;
        if (s >= W.steps) {
            s -= W.steps;
            g += W.gstride;
        }
        g = nx > last ? glast : g;
        s = nx > last ? tlast : s;
        *t = s;
        for (int r = 0; r < R; ++r) T[r] = g + (uint32_t)r;
        *nvalid = (int)min((uint32_t)R, W.t1 - g);
    }
};

// How a lane's terms of a row are summed, in every launch shape alike: in step
// order, and for Q4 and q8 (up to 56 and 112 steps a row) in blocks of four,
// the blocks' sums added up four at a time and those in order.  The shorter
// chains round less (relative error against 64 bits at 2048 x 7168, one chain
// -> blocks: Q4 2.1e-7 -> 1.75e-7, q8 2.3e-7 -> 1.5e-7; the same at 4 steps a
// row), and a wave of a split row adds a whole block by itself.
template <int KIND>
constexpr bool BLOCK_SUMS = KIND == HK_Q4 || KIND == HK_Q8;
struct BlockSum {
    float mid = 0.0f, tot = 0.0f;  // of blocks in the open group of four; of the groups
    __device__ __forceinline__ void add(uint32_t b, float v) {  // block b's sum
        mid += v;
        if ((b & 3u) == 3u) {
            tot += mid;
            mid = 0.0f;
        }
    }
};
// After step t: acc[r] into its block sums where t ends a block.
template <int KIND, int R>
__device__ __forceinline__ void end_step(uint32_t t, float* acc, BlockSum* bs) {
    if constexpr (BLOCK_SUMS<KIND>) {
        if ((t & 3u) != 3u) return;
#pragma unroll
        for (int r = 0; r < R; ++r) {
            bs[r].add(t >> 2, acc[r]);
            acc[r] = 0.0f;
        }
    }
}
// A finished row's total; the sums start again.
template <int KIND>
__device__ __forceinline__ float row_total(float& acc, BlockSum& bs) {
    float v = acc;
    if constexpr (BLOCK_SUMS<KIND>) v = bs.tot + (bs.mid + acc);
    acc = 0.0f;
    bs = BlockSum{};
    return v;
}

// Row totals of a finished group of R tiles into the workgroup's LDS row
// buffer (unscaled; tiles r >= nvalid alias T[0] and are skipped).
template <int KIND, int R>
__device__ __forceinline__ void flush_group(float* acc, BlockSum* bs, const uint32_t* T, int nvalid, uint32_t t0,
                                            int lane, float* ysh) {
#pragma unroll
    for (int r = 0; r < R; ++r) {
        const float v = tile_row_sum(row_total<KIND>(acc[r], bs[r]));
        if (r < nvalid && lane < 16) ysh[(T[r] - t0) * 16u + (uint32_t)lane] = v;
    }
}

constexpr size_t LOWRANK_LDS_LIMIT = 96 * 1024;  // of few pairs' launches (one workgroup per CU)

// Mixed step headers staged per workgroup: tiles x steps <= 32 x 24.
constexpr uint32_t GEMV_MAX_MIXED_TILES_PER_WG = 32;
constexpr int GEMV_HDR_PER_THREAD = 3;
constexpr uint32_t GEMV_MAX_MIXED_STEPS = GEMV_HDR_PER_THREAD * 256 / GEMV_MAX_MIXED_TILES_PER_WG;

// Tiles per workgroup of a launch: narrow 3-bit factors (<= 4 steps, e.g. the
// rank-160 left factor) take 128 tiles so the x image is built once per 128
// tiles; every other launch at most 32.
__host__ __device__ inline uint32_t gemv_max_tiles(int kind, uint32_t steps) {
    return kind == HK_U3 && steps <= 4 ? 128u : 32u;
}

// Dynamic LDS: x image, one quantization window (2048 columns), (mixed) the
// headers of the workgroup's tiles, then the workgroup's row outputs.
template <int KIND>
__host__ __device__ constexpr size_t gemv_hdr_offset(uint32_t steps) {
    return x_lds_bytes<KIND>(steps);
}

// The terminal head's extras (HEAD launches): x = RMSNorm(1+w)(h) is formed
// from the register chunks before the image is built (workgroup 0 also
// stores it), and the epilogue reduces the greedy key of the logits below
// n_valid into key[0] (one 64-bit atomic max per workgroup); a non-finite x
// sets the low word of key[1].
struct HeadArgs {
    const float* norm_w;
    bool norm_w4;  // 16-byte aligned
    float eps;
    float* xn;
    uint32_t n_valid;
    uint64_t* key;
};

// The greedy order of a logit: larger value first, then lower index; NaN
// never wins (key 0) and -0 ranks as +0.
__device__ __forceinline__ uint64_t greedy_key(float v, uint32_t i) {
    if (v != v) return 0ull;
    const uint32_t b = __float_as_uint(v == 0.0f ? 0.0f : v);
    const uint32_t ord = (b & 0x80000000u) ? ~b : (b | 0x80000000u);
    return ((uint64_t)ord << 32) | (uint64_t)(~i);
}

// The block's largest key into key[0], one atomic (every thread calls this;
// kred: one word per wave).
__device__ __forceinline__ void fold_key(uint64_t best, uint64_t* kred, uint64_t* key) {
    for (int off = 32; off; off >>= 1) best = max(best, (uint64_t)__shfl_xor((unsigned long long)best, off, 64));
    if ((threadIdx.x & 63) == 0) kred[threadIdx.x >> 6] = best;
    __syncthreads();
    if (threadIdx.x == 0) {
        for (uint32_t w = 1; w < (blockDim.x >> 6); ++w) best = max(best, kred[w]);
        if (best) atomicMax(reinterpret_cast<unsigned long long*>(key), (unsigned long long)best);
    }
}

// Block-wide sum (every thread gets it); red: one float per wave.
__device__ __forceinline__ float block_sum_f(float v, float* red) {
    v = wave_sum(v);
    __syncthreads();
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = v;
    __syncthreads();
    float t = 0.0f;
    for (uint32_t w = 0; w < (blockDim.x >> 6); ++w) t += red[w];
    __syncthreads();
    return t;
}

// load_x of a norm weight that is only 4-byte aligned (it has no alignment
// rule; the same kernel takes it, so xn and the logits are the same bits).
template <int NC>
__device__ __forceinline__ void load_norm_w(const float* w, uint32_t cols, XChunks<NC>& gw) {
#pragma unroll
    for (int j = 0; j < NC; ++j) {
        const uint32_t c0 = 8u * (threadIdx.x + blockDim.x * (uint32_t)j);
        const float* p = w + min(c0, cols - 8u);
#pragma unroll
        for (int k = 0; k < 2; ++k)
            gw.v[j][k] = make_float4(p[4 * k], p[4 * k + 1], p[4 * k + 2], p[4 * k + 3]);
    }
}

// xn = h * (1 / sqrt(mean(h^2) + eps)) * (1 + w) on this thread's register
// chunks of h (source_qwen80_residual_rms_norm,
// model/qwen80_complete_runtime.rs:6778-6797); every chunk of h must be in
// registers (cols <= 8 * block size * NC), and gw holds the same chunks of w
// (loaded with h, before the first weight steps: vector loads retire in
// issue order, so a w load issued after them would hold the norm until the
// weights land).
template <int NC>
__device__ __forceinline__ void head_norm_chunks(XChunks<NC>& xc, const XChunks<NC>& gw, uint32_t cols,
                                                 const HeadArgs& ha, float* red) {
    float ss = 0.0f;
#pragma unroll
    for (int j = 0; j < NC; ++j)
#pragma unroll
        for (int k = 0; k < 2; ++k) {
            const float4 v = xc.v[j][k];
            ss += v.x * v.x + v.y * v.y + v.z * v.z + v.w * v.w;
        }
    const float sum = block_sum_f(ss, red);
    const float inv = 1.0f / sqrtf(sum / (float)cols + ha.eps);
#pragma unroll
    for (int j = 0; j < NC; ++j) {
        const uint32_t c0 = 8u * (threadIdx.x + blockDim.x * (uint32_t)j);
        if (c0 < cols) {
#pragma unroll
            for (int k = 0; k < 2; ++k) {
                const float4 g = gw.v[j][k];
                float4& v = xc.v[j][k];
                v = make_float4(v.x * inv * (1.0f + g.x), v.y * inv * (1.0f + g.y), v.z * inv * (1.0f + g.z),
                                v.w * inv * (1.0f + g.w));
                if (blockIdx.x == 0) reinterpret_cast<float4*>(ha.xn + c0)[k] = v;
            }
        }
    }
}

// The HGRAVR02 residual added in the binary GEMV's epilogue (RES): views
// per organ, and the most 16-byte record pieces any workgroup's rows span.
struct ResArgs {
    const ResView* views;
    uint32_t pieces;
};
constexpr int GEMV_RES_NP = 12;  // record pieces per thread (pieces <= 12 * 256)

// Where the workgroup's row totals sit in LDS: after the x image (and the
// mixed headers), and with RES after the epilogue's residual table and
// records, which reuse the image's bytes.
template <int KIND, bool RES>
__host__ __device__ inline size_t gemv_ysh_offset(uint32_t steps, uint32_t tpw, uint32_t cols, uint32_t pieces) {
    size_t off = gemv_hdr_offset<KIND>(steps) + (KIND == HK_MIXED ? (size_t)tpw * steps * sizeof(uint4) : 0);
    if (RES) off = std::max(off, (rice_table3_bytes(cols) + (size_t)pieces * 16u + 15u) & ~(size_t)15);
    return off;
}

// D-deep software pipeline: D fetched steps are in flight while one is
// consumed; slot d of the rotating buffer holds item it+d.  The loop body is
// branch-free in memory operations (refetches are unconditional, past the end
// they re-read the last item; y goes out through LDS after the loop) so the
// compiler can wait for exactly the slot being consumed.
//
// RES (binary, at most 512 rows per workgroup): y = base + the HGRAVR02
// residual, to the bit what rice_apply does after the plain GEMV.  The row
// pointers load with the first weights; after the main loop the image's
// LDS takes the product table of three entries per column (from the x
// chunks still in registers) and the workgroup's byte-step record pieces
// (loaded in one round), and each row's thread steps through its records,
// adding its products to the row total in index order.
// Where a pipeline's fetches past its last item go: with the weights' loads
// non-temporal, a re-read of the last item (the refetches stay unconditional,
// a branch around them measured slower) would come from HBM again (6.5 %
// more read traffic on the headline stream); pointed at this small buffer,
// which every wave's refetches keep in the caches, they cost no HBM bytes.
// Nothing fetched from it is ever consumed.
__device__ __align__(256) uint8_t g_refetch_dummy[4096];

// fetch_step, or the same loads from g_refetch_dummy when past (uniform):
// tile 0, step 0 of a view whose sections start there (offsets below 4 KiB).
template <int KIND, int R, bool NT>
__device__ __forceinline__ void fetch_step_or_dummy(const OrganView& o, const uint32_t* T, int nvalid, uint32_t t,
                                                    int lane, Frag<KIND, R>& f, bool past) {
    OrganView op = o;
    op.data = past ? g_refetch_dummy : o.data;
    op.scales = past ? reinterpret_cast<const uint16_t*>(g_refetch_dummy) : o.scales;
    uint32_t Tz[R];
#pragma unroll
    for (int r = 0; r < R; ++r) Tz[r] = past ? 0u : T[r];
    fetch_step<KIND, R, NT>(op, Tz, nvalid, past ? 0u : t, lane, f);
}

template <int KIND, int R, int D, int NC, bool RES = false>
__global__ void __launch_bounds__(256)
gemv_tiled_kernel(const OrganView* __restrict__ organs, uint32_t n_organs, const float* __restrict__ xall,
                  size_t x_stride, float* __restrict__ yall, size_t y_stride, uint32_t tiles_per_wg, uint32_t parts,
                  ResArgs ra) {
    static_assert(!RES || (KIND == HK_BIN && NC == 1), "the fused residual is for binary organs");
    extern __shared__ __align__(16) uint8_t lds[];
    uint32_t oi, part;
    organ_part(blockIdx.x, parts, n_organs, &oi, &part);
    const OrganView o = organs[oi];
    const float* __restrict__ x = xall + (size_t)oi * x_stride;
    float* __restrict__ y = yall + (size_t)oi * y_stride;
    const int lane = threadIdx.x & 63, q = lane >> 4;
    const uint32_t wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const uint32_t t0 = part * tiles_per_wg, t1 = min(t0 + tiles_per_wg, o.n_tiles);
    WaveItems W{t0 + wave * R, 4u * R, t1, o.steps, 0};
    W.n = W.g0 < t1 ? ((t1 - W.g0 + W.gstride - 1) / W.gstride) * o.steps : 0;
    const uint32_t last = W.n ? W.n - 1u : 0u;

    // x first, then (mixed) this workgroup's
    // step headers, then the first D steps' weight loads, all before the
    // image build
    XChunks<NC> xc;
    load_x<NC>(BlockTeam{}, x, o.cols, xc);
    const uint32_t nh = (t1 - t0) * o.steps;
    uint4 hreg[GEMV_HDR_PER_THREAD];
    uint4* hsh = reinterpret_cast<uint4*>(lds + gemv_hdr_offset<KIND>(o.steps));
    float* ysh = reinterpret_cast<float*>(lds + gemv_ysh_offset<KIND, RES>(o.steps, tiles_per_wg, o.cols, ra.pieces));
    if constexpr (KIND == HK_MIXED) {
#pragma unroll
        for (int k = 0; k < GEMV_HDR_PER_THREAD; ++k) {
            const uint32_t i = threadIdx.x + 256u * k;
            if (i < nh) hreg[k] = ldg(o.hdr + (size_t)t0 * o.steps + i);
        }
    }
    Frag<KIND, R> f[D];
    uint32_t T[D][R], ts[D];
    int nv[D];
    {
        // unconditional, so the x wait below counts exactly these loads; a
        // wave without items re-reads the workgroup's first tile
        const WaveItems P = W.n ? W : WaveItems{t0, 4u * R, t0 + 1u, o.steps, 1u};
#pragma unroll
        for (int d = 0; d < D; ++d) {
            P.at(min((uint32_t)d, last), T[d], R, &nv[d], &ts[d]);
            if constexpr (KIND == HK_MIXED) fetch_step<KIND, R, true>(o, T[d], nv[d], ts[d], lane, f[d]);
            else fetch_step_or_dummy<KIND, R, true>(o, T[d], nv[d], ts[d], lane, f[d], (uint32_t)d > last);
        }
    }
    if constexpr (KIND == HK_MIXED) {
#pragma unroll
        for (int k = 0; k < GEMV_HDR_PER_THREAD; ++k) {
            const uint32_t i = threadIdx.x + 256u * k;
            if (i < nh) hsh[i] = hreg[k];
        }
    }
    // RES: the residual's view and the row pointers of this workgroup's rows
    // (two rows a thread), issued after the first weights
    ResView rv{};
    uint32_t rp0 = 0, my0[2] = {0u, 0u}, my1[2] = {0u, 0u};
    if constexpr (RES) {
        rv = ra.views[oi];
        const uint32_t r0 = t0 * 16u, r1 = min(t1 * 16u, o.rows);
        rp0 = ldg(rv.row_ptr8 + r0) / 16u;
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            const uint32_t row = min(r0 + threadIdx.x + 256u * (uint32_t)h, r1);
            my0[h] = ldg(rv.row_ptr8 + row);
            my1[h] = ldg(rv.row_ptr8 + min(row + 1u, r1));
        }
    }
    // the x image with E = 0: every thread scatters its own chunks (no
    // block-wide maximum, no gather pass); a unit's chunks are consecutive
    // threads, active together
    {
        const uint32_t nch = o.steps * (uint32_t)Kcfg<KIND>::STEP_COLS / 8u;
        float* sxw = reinterpret_cast<float*>(lds + (size_t)o.steps * Kcfg<KIND>::P * A_TILE_STRIDE);
        if (threadIdx.x < 64u) image_zero_blocks<KIND>(threadIdx.x, lds, o.steps);
#pragma unroll
        for (int j = 0; j < NC; ++j) {
            const uint32_t ch = threadIdx.x + 256u * (uint32_t)j;
            if (ch < nch) (void)image_chunk<KIND>(ch, xc.v[j], lds, sxw, 0u, 0u);
        }
        for (uint32_t ch = threadIdx.x + 256u * NC; ch < nch; ch += 256u) {
            float4 v[2];
            load_chunk(x, 8u * ch, o.cols, v);
            (void)image_chunk<KIND>(ch, v, lds, sxw, 0u, 0u);
        }
        __syncthreads();
    }
    const int E = 0;

    const ImageA A{lds, a_lane_offset(lane)};
    const float* SX = reinterpret_cast<const float*>(lds + (size_t)o.steps * Kcfg<KIND>::P * A_TILE_STRIDE);

    float acc[R];
    BlockSum bs[R];
#pragma unroll
    for (int r = 0; r < R; ++r) acc[r] = 0.0f;
    ItemStride<D> adv;
    adv.init(W, last);
    uint32_t it = 0;
    for (; it + D <= W.n; it += D) {
#pragma unroll
        for (int d = 0; d < D; ++d) {
            compute_step<KIND, R>(f[d], ts[d], A, SX, q, acc);
            end_step<KIND, R>(ts[d], acc, bs);
            if (ts[d] + 1 == o.steps) flush_group<KIND, R>(acc, bs, T[d], nv[d], t0, lane, ysh);
            adv.next(W, it + D + d, last, T[d], R, &nv[d], &ts[d]);
            if constexpr (KIND == HK_MIXED) {
                // headers from LDS: the data loads wait for an LDS read, not
                // for every load in flight before them
#pragma unroll
                for (int r = 0; r < R; ++r) {
                    const uint32_t Tr = r < nv[d] ? T[d][r] : T[d][0];
                    fetch_mixed<R>(o, hsh[(Tr - t0) * o.steps + ts[d]], lane, f[d], r);
                }
            } else {
                fetch_step_or_dummy<KIND, R, true>(o, T[d], nv[d], ts[d], lane, f[d], it + D + d > last);
            }
        }
    }
#pragma unroll
    for (int d = 0; d < D; ++d) {
        if (it + d >= W.n) break;
        compute_step<KIND, R>(f[d], ts[d], A, SX, q, acc);
        end_step<KIND, R>(ts[d], acc, bs);
        if (ts[d] + 1 == o.steps) flush_group<KIND, R>(acc, bs, T[d], nv[d], t0, lane, ysh);
    }
    __syncthreads();
    const uint32_t nrows = (t1 > t0 ? t1 - t0 : 0u) * 16u;
    if constexpr (RES) {
        // the image is dead: its bytes take the residual's table and records
        const uint32_t np = (ra.pieces + 255u) / 256u;
        const uint4* recs = reinterpret_cast<const uint4*>(rv.recs8);
        const uint32_t plast = (rv.count8 + 15u) / 16u - 1u;
        uint4 rr[GEMV_RES_NP];
#pragma unroll
        for (int j = 0; j < GEMV_RES_NP; ++j)
            if ((uint32_t)j < np) rr[j] = ldg(recs + min(rp0 + threadIdx.x + 256u * (uint32_t)j, plast));
        float* T3 = reinterpret_cast<float*>(lds);
        {
            const uint32_t c0 = 8u * threadIdx.x;
            if (c0 < o.cols) {
                const float xv[8] = {xc.v[0][0].x, xc.v[0][0].y, xc.v[0][0].z, xc.v[0][0].w,
                                     xc.v[0][1].x, xc.v[0][1].y, xc.v[0][1].z, xc.v[0][1].w};
#pragma unroll
                for (int k = 0; k < 8; ++k) {
                    const float p = rv.scale * xv[k];
                    T3[3u * (c0 + (uint32_t)k)] = -p;
                    T3[3u * (c0 + (uint32_t)k) + 1u] = p;
                    T3[3u * (c0 + (uint32_t)k) + 2u] = -0.0f;
                }
            }
        }
        if (threadIdx.x < 8u) T3[3u * o.cols + threadIdx.x] = -0.0f;
        uint4* Rr = reinterpret_cast<uint4*>(lds + rice_table3_bytes(o.cols));
#pragma unroll
        for (int j = 0; j < GEMV_RES_NP; ++j)
            if ((uint32_t)j < np && threadIdx.x + 256u * (uint32_t)j < ra.pieces) Rr[threadIdx.x + 256u * j] = rr[j];
        __syncthreads();
        const uint32_t* R4 = reinterpret_cast<const uint32_t*>(Rr);
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            const uint32_t i = threadIdx.x + 256u * (uint32_t)h, row = t0 * 16u + i;
            if (i < nrows && row < o.rows) {
                float acc = ldexpf(ysh[i], -E);
                uint32_t v = 0xFFFFFFFFu;  // -1: a row's first step lands on its first index
#pragma unroll 2
                for (uint32_t e = my0[h]; e < my1[h]; e += 4u) {
                    const uint32_t w = R4[(e - 16u * rp0) / 4u];
                    v += w & 0xFFu;
                    acc += T3[v];
                    v += (w >> 8) & 0xFFu;
                    acc += T3[v];
                    v += (w >> 16) & 0xFFu;
                    acc += T3[v];
                    v += w >> 24;
                    acc += T3[v];
                }
                y[row] = acc;
            }
        }
        return;
    }
    for (uint32_t i = threadIdx.x; i < nrows; i += blockDim.x) {
        const uint32_t row = t0 * 16u + i;
        if (row < o.rows) y[row] = ldexpf(ysh[i], -E);
    }
}

// One wave's walk over the row tiles [t0, t1) of organ o in groups of R tiles
// (stride 4R over the block's four waves), every step of each, D steps in
// flight -- the main loop of gemv_tiled_kernel for the non-mixed kinds.
// start() issues the first D fetches (before the caller builds its x image);
// run() consumes the walk against an x image, leaving the unscaled row totals
// in ysh[(tile - t0) * 16 + row].
template <int KIND, int R, int D>
struct TileWalk {
    WaveItems W;
    uint32_t last;
    Frag<KIND, R> f[D];
    uint32_t T[D][R], ts[D];
    int nv[D];

    __device__ __forceinline__ void start(const OrganView& o, uint32_t t0, uint32_t t1, uint32_t wave, int lane) {
        W = WaveItems{t0 + wave * R, 4u * R, t1, o.steps, 0};
        W.n = W.g0 < t1 ? ((t1 - W.g0 + W.gstride - 1) / W.gstride) * o.steps : 0;
        last = W.n ? W.n - 1u : 0u;
        // a wave without items re-reads tile t0 (its results are never used)
        const WaveItems P = W.n ? W : WaveItems{t0, 4u * R, t0 + 1u, o.steps, 1u};
#pragma unroll
        for (int d = 0; d < D; ++d) {
            P.at(min((uint32_t)d, last), T[d], R, &nv[d], &ts[d]);
            fetch_step<KIND, R>(o, T[d], nv[d], ts[d], lane, f[d]);
        }
    }

    __device__ __forceinline__ void run(const OrganView& o, uint32_t t0, const uint8_t* img, int lane, float* ysh) {
        const ImageA A{img, a_lane_offset(lane)};
        const float* SX = reinterpret_cast<const float*>(img + (size_t)o.steps * Kcfg<KIND>::P * A_TILE_STRIDE);
        const int q = lane >> 4;
        float acc[R];
        BlockSum bs[R];
#pragma unroll
        for (int r = 0; r < R; ++r) acc[r] = 0.0f;
        ItemStride<D> adv;
        adv.init(W, last);
        uint32_t it = 0;
        for (; it + D <= W.n; it += D) {
#pragma unroll
            for (int d = 0; d < D; ++d) {
                compute_step<KIND, R>(f[d], ts[d], A, SX, q, acc);
                end_step<KIND, R>(ts[d], acc, bs);
                if (ts[d] + 1 == o.steps) flush_group<KIND, R>(acc, bs, T[d], nv[d], t0, lane, ysh);
                adv.next(W, it + D + d, last, T[d], R, &nv[d], &ts[d]);
                fetch_step<KIND, R>(o, T[d], nv[d], ts[d], lane, f[d]);
            }
        }
#pragma unroll
        for (int d = 0; d < D; ++d) {
            if (it + d >= W.n) break;
            compute_step<KIND, R>(f[d], ts[d], A, SX, q, acc);
            end_step<KIND, R>(ts[d], acc, bs);
            if (ts[d] + 1 == o.steps) flush_group<KIND, R>(acc, bs, T[d], nv[d], t0, lane, ysh);
        }
    }
};

// LDS layout of the low-rank kernel: the right factor's x image, mid (16
// floats per right tile), the left factor's image, then the left rows.
struct LowrankLds {
    size_t img_r, win_r, mid, img_l, win_l, ysh, total;
};
__host__ __device__ inline LowrankLds lowrank_lds(const OrganView& l, const OrganView& r) {
    LowrankLds L{};
    L.img_r = 0;
    L.win_r = L.img_r + x_lds_bytes<HK_U3>(r.steps);
    L.mid = L.win_r;
    L.img_l = L.mid + ((size_t)r.n_tiles * 16u * 4u + 15u) / 16u * 16u;
    L.win_l = L.img_l + x_lds_bytes<HK_U3>(l.steps);
    L.ysh = L.win_l;
    L.total = L.ysh + (size_t)l.n_tiles * 16u * 4u;
    return L;
}

// (build-time overrides for launch-shape sweeps: tile groups and steps in
// flight of the right and the left factor's walks)
#ifndef HK_LR_RR
#define HK_LR_RR 1
#define HK_LR_RD 3
#define HK_LR_LR 2
#define HK_LR_LD 3
#endif

// HGRAVS01 pairs y_i = L_i (R_i x_i), one workgroup per pair: the right
// factor's rows (mid, kept in LDS) and then the left factor's, whose first
// weight steps are issued as soon as the right factor's walk ends (in flight
// while mid's x image is built).  Issued at the start instead, they hold
// their registers through the right walk: 74 VGPRs and 6 workgroups per CU
// against 56 and 8 (4,096 pairs then run in exactly two rounds; r160 pairs
// 164 against 161 us).  The arithmetic
// is that of two gemv_tiled_kernel launches (mid rounded to f32, then its own
// x image), so the result is the same bits.  mid_all (may be null) also
// receives mid.
#ifndef HK_LR_MINW
#define HK_LR_MINW 1
#endif
template <int NC>
__global__ void __launch_bounds__(256, HK_LR_MINW)
lowrank_kernel(const OrganView* __restrict__ lefts, const OrganView* __restrict__ rights, uint32_t n,
               const float* __restrict__ xall, size_t x_stride, float* __restrict__ mid_all, size_t mid_stride,
               float* __restrict__ yall, size_t y_stride) {
    extern __shared__ __align__(16) uint8_t lds[];
    uint32_t oi, part;
    organ_part(blockIdx.x, 1, n, &oi, &part);
    const OrganView rv = rights[oi], lv = lefts[oi];
    const float* __restrict__ x = xall + (size_t)oi * x_stride;
    float* __restrict__ y = yall + (size_t)oi * y_stride;
    const int lane = threadIdx.x & 63;
    const uint32_t wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const LowrankLds M = lowrank_lds(lv, rv);
    float* mid = reinterpret_cast<float*>(lds + M.mid);
    float* ysh = reinterpret_cast<float*>(lds + M.ysh);

    XChunks<NC> xc;
    load_x<NC>(BlockTeam{}, x, rv.cols, xc);
    TileWalk<HK_U3, HK_LR_RR, HK_LR_RD> wr;
    wr.start(rv, 0, rv.n_tiles, wave, lane);
    TileWalk<HK_U3, HK_LR_LR, HK_LR_LD> wl;
    // both x images with E = 0, scattered from each thread's chunks (the
    // two launches' images to the bit: the GEMV builds them the same way)
    {
        uint8_t* img = lds + M.img_r;
        float* sx = reinterpret_cast<float*>(img + (size_t)rv.steps * Kcfg<HK_U3>::P * A_TILE_STRIDE);
        const uint32_t nch = rv.steps * (uint32_t)Kcfg<HK_U3>::STEP_COLS / 8u;
        if (threadIdx.x < 64u) image_zero_blocks<HK_U3>(threadIdx.x, img, rv.steps);
#pragma unroll
        for (int j = 0; j < NC; ++j) {
            const uint32_t ch = threadIdx.x + 256u * (uint32_t)j;
            if (ch < nch) (void)image_chunk<HK_U3>(ch, xc.v[j], img, sx, 0u, 0u);
        }
        for (uint32_t ch = threadIdx.x + 256u * NC; ch < nch; ch += 256u) {
            float4 v[2];
            load_chunk(x, 8u * ch, rv.cols, v);
            (void)image_chunk<HK_U3>(ch, v, img, sx, 0u, 0u);
        }
        __syncthreads();
    }
    wr.run(rv, 0, lds + M.img_r, lane, mid);
    wl.start(lv, 0, lv.n_tiles, wave, lane);
    __syncthreads();
    if (mid_all)
        for (uint32_t i = threadIdx.x; i < rv.rows; i += blockDim.x) mid_all[(size_t)oi * mid_stride + i] = mid[i];
    {
        uint8_t* img = lds + M.img_l;
        float* sx = reinterpret_cast<float*>(img + (size_t)lv.steps * Kcfg<HK_U3>::P * A_TILE_STRIDE);
        const uint32_t nch = lv.steps * (uint32_t)Kcfg<HK_U3>::STEP_COLS / 8u;
        if (threadIdx.x < 64u) image_zero_blocks<HK_U3>(threadIdx.x, img, lv.steps);
        for (uint32_t ch = threadIdx.x; ch < nch; ch += 256u) {
            float4 v[2];
            load_chunk(mid, 8u * ch, rv.rows, v);
            (void)image_chunk<HK_U3>(ch, v, img, sx, 0u, 0u);
        }
        __syncthreads();
    }
    wl.run(lv, 0, lds + M.img_l, lane, ysh);
    __syncthreads();
    for (uint32_t i = threadIdx.x; i < lv.rows; i += blockDim.x) y[i] = ysh[i];
}

// The same pairs when there are too few of them for one workgroup each to
// fill the chip: P workgroups of 16 waves share a pair's left factor, each
// forming the whole mid itself (the right factor is the smaller one, and its
// re-reads are cache hits).  The right tiles go in rounds of at most 16: four
// waves split a tile's steps and leave their terms in LDS, then one wave per
// tile adds them in step order (the bits of a walk); the left tiles are one
// wave each, their first steps in flight while mid's image is built.
constexpr uint32_t LOWRANK_WAVES = 16, LOWRANK_ROUND = 16;
struct LowrankArgs {
    OrganView left, right;                // n = 1: the pair
    const OrganView *lefts, *rights;      // else the tables
    const float* x;
    float *mid, *y;                       // mid may be null
    size_t x_stride, mid_stride, y_stride;
    uint32_t n, parts;                    // pairs, workgroups per pair
    uint32_t tpw, round;                  // left tiles per workgroup, right tiles per round
};
struct LowrankSplitLds {
    size_t terms, mid, img_l, total;
    __host__ __device__ LowrankSplitLds(const OrganView& l, const OrganView& r, uint32_t round) {
        terms = (x_lds_bytes<HK_U3>(r.steps) + 15u) & ~(size_t)15;
        mid = terms + (size_t)round * r.steps * 512u;
        img_l = mid + (size_t)r.n_tiles * 64u;
        total = img_l + x_lds_bytes<HK_U3>(l.steps);
    }
};
__global__ void __launch_bounds__(64 * LOWRANK_WAVES) lowrank_split_kernel(LowrankArgs a) {
    extern __shared__ __align__(16) uint8_t lds[];
    constexpr int D = 4;
    constexpr uint32_t P3 = Kcfg<HK_U3>::P, KS = 4, TS = LOWRANK_WAVES / KS;
    uint32_t oi, part;
    organ_part(blockIdx.x, a.parts, a.n, &oi, &part);
    OrganView lv = a.left, rv = a.right;
    if (a.lefts) {
        lv = a.lefts[oi];
        rv = a.rights[oi];
    }
    const float* __restrict__ x = a.x + (size_t)oi * a.x_stride;
    float* __restrict__ y = a.y + (size_t)oi * a.y_stride;
    const int lane = threadIdx.x & 63, q = lane >> 4;
    const uint32_t wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), nthr = blockDim.x;
    const LowrankSplitLds M(lv, rv, a.round);
    float* mid = reinterpret_cast<float*>(lds + M.mid);
    float2* terms = reinterpret_cast<float2*>(lds + M.terms) + lane;
    const uint32_t S = rv.steps, ksl = wave & (KS - 1u), tsl = wave / KS;
    const uint32_t per = (S + KS - 1u) / KS, s0 = min(ksl * per, S), ns = min(per, S - s0);

    XChunks<1> xc;
    load_x<1>(BlockTeam{}, x, rv.cols, xc);  // cols <= 8192: one chunk a thread
    // this wave's items of the round of right tiles from b on
    uint32_t fT = 0, fs = 0, fi = 0, fn = 0;
    Frag<HK_U3, 1> f[D];
    auto next = [&]() {
        if (++fi < fn) {
            ++fs;
            if (fs == s0 + ns) {
                fs = s0;
                fT += TS;
            }
        }
    };
    auto start = [&](uint32_t b) {
        const uint32_t e = min(b + a.round, rv.n_tiles), t = b + tsl;
        fn = t < e ? (e - t + TS - 1u) / TS * ns : 0u;
        fT = fn ? t : b;
        fs = fn ? s0 : 0u;
        fi = 0;
#pragma unroll
        for (int d = 0; d < D; ++d) {
            fetch_one<HK_U3, 1>(rv, fT, fs, lane, f[d], 0);
            next();
        }
        return fn;
    };
    uint32_t n = start(0);
    auto image = [&](uint8_t* img, const OrganView& o, float4 (&v)[2], uint32_t ch) {
        float* sx = reinterpret_cast<float*>(img + (size_t)o.steps * P3 * A_TILE_STRIDE);
        if (ch < o.steps * 16u) (void)image_chunk<HK_U3>(ch, v, img, sx, 0u, 0u);
    };
    auto zero = [&](uint8_t* img, uint32_t steps) {
        for (uint32_t i = threadIdx.x; i < steps * P3; i += nthr)
            *reinterpret_cast<uint4*>(img + (size_t)i * A_TILE_STRIDE + 256u) = make_uint4(0u, 0u, 0u, 0u);
    };
    zero(lds, S);
    zero(lds + M.img_l, lv.steps);
    image(lds, rv, xc.v[0], threadIdx.x);
    __syncthreads();

    const ImageA AR{lds, a_lane_offset(lane)};
    const float* sxr = reinterpret_cast<const float*>(lds + (size_t)S * P3 * A_TILE_STRIDE);
    for (uint32_t b = 0; b < rv.n_tiles; b += a.round) {
        uint32_t cT = b + tsl, cs = s0;
        auto consume = [&](const Frag<HK_U3, 1>& fr) {
            float2* o = terms + ((cT - b) * S + cs) * 64u;
            compute_terms<HK_U3, 1>(fr, cs, AR, sxr, q, [&](int, float s, float v) { *o = make_float2(s, v); });
            ++cs;
            if (cs == s0 + ns) {
                cs = s0;
                cT += TS;
            }
        };
        uint32_t it = 0;
        for (; it + D < n; it += D) {
#pragma unroll
            for (int d = 0; d < D; ++d) {
                consume(f[d]);
                fetch_one<HK_U3, 1>(rv, fT, fs, lane, f[d], 0);
                next();
            }
        }
#pragma unroll
        for (int d = 0; d < D; ++d)
            if (it + (uint32_t)d < n) consume(f[d]);
        if (b + a.round < rv.n_tiles) n = start(b + a.round);
        __syncthreads();
        if (b + wave < min(b + a.round, rv.n_tiles)) {
            float v = 0.0f;
#pragma unroll 4
            for (uint32_t s = 0; s < S; ++s) {
                const float2 e = terms[(wave * S + s) * 64u];
                v = __builtin_fmaf(e.x, e.y, v);
            }
            v = tile_row_sum(v);
            if (lane < 16) mid[(b + wave) * 16u + (uint32_t)lane] = v;
        }
        __syncthreads();
    }

    // the left tiles: wave w takes t0 + w, t0 + w + 16, ..., every step
    const uint32_t t0 = part * a.tpw, t1 = min(t0 + a.tpw, lv.n_tiles), S2 = lv.steps;
    n = t0 + wave < t1 ? (t1 - t0 - wave + LOWRANK_WAVES - 1u) / LOWRANK_WAVES * S2 : 0u;
    fT = n ? t0 + wave : 0u;
    fs = 0;
    fi = 0;
    auto next_l = [&]() {
        if (++fi < n) {
            ++fs;
            if (fs == S2) {
                fs = 0;
                fT += LOWRANK_WAVES;
            }
        }
    };
#pragma unroll
    for (int d = 0; d < D; ++d) {
        fetch_one<HK_U3, 1>(lv, fT, fs, lane, f[d], 0);
        next_l();
    }
    if (a.mid && part == 0)
        for (uint32_t i = threadIdx.x; i < rv.rows; i += nthr) a.mid[(size_t)oi * a.mid_stride + i] = mid[i];
    {
        float4 v[2];
        load_chunk(mid, 8u * threadIdx.x, rv.rows, v);
        image(lds + M.img_l, lv, v, threadIdx.x);
    }
    __syncthreads();
    const ImageA AL{lds + M.img_l, a_lane_offset(lane)};
    const float* sxl = reinterpret_cast<const float*>(lds + M.img_l + (size_t)S2 * P3 * A_TILE_STRIDE);
    uint32_t cT = t0 + wave, cs = 0;
    float acc = 0.0f;
    auto consume = [&](const Frag<HK_U3, 1>& fr) {
        compute_step<HK_U3, 1>(fr, cs, AL, sxl, q, &acc);
        if (++cs == S2) {
            const float v = tile_row_sum(acc);
            const uint32_t row = cT * 16u + (uint32_t)lane;
            if (lane < 16 && row < lv.rows) y[row] = v;
            acc = 0.0f;
            cs = 0;
            cT += LOWRANK_WAVES;
        }
    };
    uint32_t it = 0;
    for (; it + D < n; it += D) {
#pragma unroll
        for (int d = 0; d < D; ++d) {
            consume(f[d]);
            fetch_one<HK_U3, 1>(lv, fT, fs, lane, f[d], 0);
            next_l();
        }
    }
#pragma unroll
    for (int d = 0; d < D; ++d)
        if (it + (uint32_t)d < n) consume(f[d]);
}

bool lowrank_fusable(const OrganView& l, const OrganView& r) {
    return l.kind == HK_U3 && r.kind == HK_U3 && r.rows == l.cols && r.cols <= 8192u && r.rows <= 2048u &&
           lowrank_lds(l, r).total <= GEMV_LDS_LIMIT;
}

hipError_t launch_lowrank(const OrganView* lefts, const OrganView* rights, uint32_t n, const OrganView& l,
                          const OrganView& r, const float* x, size_t x_stride, float* mid, size_t mid_stride, float* y,
                          size_t y_stride, hipStream_t s) {
    if (!lowrank_fusable(l, r)) return hipErrorInvalidValue;
    // One workgroup per CU over all pairs, at least 16 left tiles each (us in a
    // graph of one launch, against one 4-wave workgroup per pair): r160 2048 x
    // 768, 1 pair 17.9 -> 6.4, 64 pairs 18.3 -> 7.3, 256 pairs 18.8 -> 12.8, 512
    // pairs 23.3 -> 20.1, 1,024 pairs 34.7 against 37.7; r64 512 x 512, 1 pair
    // 6.2 -> 4.8, 256 pairs 6.6 -> 5.6, 512 pairs 7.5 against 7.8; r384 4096 x
    // 2048, 1 pair 53 -> 15.
    const uint32_t few = l.n_tiles >= 64u ? 512u : 256u;
    // (overlapping buffers: one workgroup a pair, which has read what it
    // overwrites)
    const bool shared = vectors_overlap(x, x_stride, r.cols, y, y_stride, l.rows, n) ||
                        vectors_overlap(x, x_stride, r.cols, mid, mid_stride, r.rows, n) ||
                        vectors_overlap(mid, mid_stride, r.rows, y, y_stride, l.rows, n);
    const uint32_t parts = n > few || shared
                               ? 0u
                               : std::min(std::max(256u / n, 1u), (l.n_tiles + LOWRANK_WAVES - 1u) / LOWRANK_WAVES);
    if (parts) {
        LowrankArgs a{};
        a.tpw = (l.n_tiles + parts - 1u) / parts;
        a.parts = (l.n_tiles + a.tpw - 1u) / a.tpw;
        a.round = std::min(std::min(LOWRANK_ROUND, r.n_tiles), 128u / r.steps);
        const size_t sl = LowrankSplitLds(l, r, a.round).total;
        if (a.round && sl <= LOWRANK_LDS_LIMIT) {
            a.left = l;
            a.right = r;
            a.lefts = n > 1 ? lefts : nullptr;
            a.rights = rights;
            a.x = x;
            a.mid = mid;
            a.y = y;
            a.x_stride = x_stride;
            a.mid_stride = mid_stride;
            a.y_stride = y_stride;
            a.n = n;
            hipLaunchKernelGGL(lowrank_split_kernel, dim3(a.parts * n), dim3(64u * LOWRANK_WAVES), sl, s, a);
            return hipGetLastError();
        }
    }
    const size_t lds = lowrank_lds(l, r).total;
    if (x_image_cols<HK_U3>(r.steps) <= 2048u)
        hipLaunchKernelGGL(lowrank_kernel<1>, dim3(n), dim3(256), lds, s, lefts, rights, n, x, x_stride, mid,
                           mid_stride, y, y_stride);
    else
        hipLaunchKernelGGL(lowrank_kernel<4>, dim3(n), dim3(256), lds, s, lefts, rights, n, x, x_stride, mid,
                           mid_stride, y, y_stride);
    return hipGetLastError();
}

// Dense f32 rows (router, shared-expert gate): one wave per row, float4 loads.
__global__ void __launch_bounds__(256) gemv_f32_kernel(const OrganView* __restrict__ organs,
                                                       const float* __restrict__ xall, size_t x_stride,
                                                       float* __restrict__ yall, size_t y_stride) {
    const OrganView o = organs[blockIdx.y];
    const int lane = threadIdx.x & 63;
    const uint32_t row = blockIdx.x * 4 + (threadIdx.x >> 6);
    if (row >= o.rows) return;
    const float4* w = reinterpret_cast<const float4*>(o.dense + (size_t)row * o.cols);
    const float4* xv = reinterpret_cast<const float4*>(xall + (size_t)blockIdx.y * x_stride);
    float acc = 0.f;
    for (uint32_t j = lane; j < o.cols / 4; j += 64) {
        const float4 a = w[j], b = xv[j];
        acc += a.x * b.x + a.y * b.y + a.z * b.z + a.w * b.w;
    }
    acc = wave_sum(acc);
    if (lane == 0) yall[(size_t)blockIdx.y * y_stride + row] = acc;
}

size_t gemv_lds_bytes(int kind, uint32_t cols) {
    const uint32_t S = n_steps_for(kind, cols);
    const size_t ysh = (size_t)gemv_max_tiles(kind, S) * 16u * sizeof(float);
    if (kind == HK_Q4) return gemv_hdr_offset<HK_Q4>(S) + ysh;
    if (kind == HK_U3) return gemv_hdr_offset<HK_U3>(S) + ysh;
    if (kind == HK_BIN) return gemv_hdr_offset<HK_BIN>(S) + ysh;
    if (kind == HK_Q8) return gemv_hdr_offset<HK_Q8>(S) + ysh;
    if (S > GEMV_MAX_MIXED_STEPS) return SIZE_MAX;
    return gemv_hdr_offset<HK_MIXED>(S) + (size_t)GEMV_MAX_MIXED_TILES_PER_WG * S * sizeof(uint4) + ysh;
}

template <int KIND, int R, int D, bool RES = false>
static hipError_t launch_kind(const OrganView* organs, uint32_t n, const OrganView& sh, const float* x,
                              size_t xs, float* y, size_t ys, uint32_t tpw, hipStream_t s, const ResArgs& ra = {}) {
    const uint32_t parts = (sh.n_tiles + tpw - 1) / tpw;
    const dim3 grid(parts * n);
    // image + one quantization window (2048 columns); x chunks held in
    // registers: one per thread up to 2048 columns, else four
    const uint32_t kc = x_image_cols<KIND>(sh.steps);
    const size_t lds = gemv_ysh_offset<KIND, RES>(sh.steps, tpw, sh.cols, ra.pieces) + (size_t)tpw * 16u * sizeof(float);
    if (kc <= 2048u)
        hipLaunchKernelGGL((gemv_tiled_kernel<KIND, R, D, 1, RES>), grid, dim3(256), lds, s, organs, n, x, xs, y, ys,
                           tpw, parts, ra);
    else if constexpr (!RES)
        hipLaunchKernelGGL((gemv_tiled_kernel<KIND, R, D, 4>), grid, dim3(256), lds, s, organs, n, x, xs, y, ys, tpw,
                           parts, ra);
    return hipGetLastError();
}

// ------------------------------------------------------------------ small launches
//
// One organ, or a set with too few row tiles to fill the chip: the time is a
// chain of memory round trips, not bandwidth.  gemv_split_kernel splits each
// row tile's steps over KS waves of its workgroup (TS = waves / KS tiles side
// by side), so a tile's weights are all in flight at once instead of two
// steps at a time in one wave, and every thread of the workgroup builds its
// part of the x image.  A single organ's view comes with the kernel
// arguments (one round trip fewer than a descriptor load).
struct SplitArgs {
    OrganView one;            // organs null: the one organ
    const OrganView* organs;  // else the table of the n organs
    ResView res_one;          // RES, the same way
    const ResView* res;
    const float* x;
    float* y;
    size_t x_stride, y_stride;
    uint32_t n, parts;        // organs, workgroups per organ
    uint32_t tpw;             // tiles per workgroup, a multiple of TS
    uint32_t ks_log, ts_log;  // log2 KS, log2 TS
    uint32_t bufs;            // KS > 1: buffers of a chunk's terms (one: a single chunk)
    HeadArgs ha;              // HEAD: the terminal head's prologue and epilogue
    uint32_t* status;
};

constexpr size_t SPLIT_LDS_LIMIT = 128 * 1024;

template <int KIND>
constexpr uint32_t split_depth = KIND == HK_MIXED ? 2 : 4;  // steps in flight per wave
enum { SPLIT_WALK, SPLIT_CHUNKS, SPLIT_ONCE };              // KS = 1; KS > 1; one round of at most split_depth items
// Steps of a tile that each of its KS waves runs (past the last: no work).
template <int KIND>
__host__ __device__ constexpr uint32_t split_per(uint32_t S, uint32_t ks_log) {
    return BLOCK_SUMS<KIND> ? (((S + 3u) / 4u + (1u << ks_log) - 1u) >> ks_log) * 4u
                            : (S + (1u << ks_log) - 1u) >> ks_log;
}

// LDS: the x image, then (RES) a copy of x and the residual's products, then
// (KS > 1) the {scale, v} terms or block sums of a chunk of steps of every tile
// of a round, then (RES) the rows' base sums.
template <int KIND, bool RES>
struct SplitLds {
    static constexpr uint32_t TERMS = KIND == HK_MIXED ? 2u : 1u;  // a step's
    // 256-byte words of a wave's item
    static constexpr uint32_t WORDS = BLOCK_SUMS<KIND> ? 1u : 2u * TERMS;
    uint32_t chunk;  // items of a wave between barriers (BLOCK_SUMS: one, of four steps)
    size_t xs, vals, terms, ysh, total;
    __host__ __device__ SplitLds(uint32_t S, uint32_t cols, uint32_t tpw, uint32_t waves, uint32_t per, uint32_t bufs)
        : chunk(BLOCK_SUMS<KIND> ? 1u : per < 4u ? per : 4u) {
        xs = (x_lds_bytes<KIND>(S) + 15u) & ~(size_t)15;
        vals = xs + (RES ? (size_t)cols * 4u : 0);
        terms = vals + (RES ? (size_t)RICE_BATCH * 4u : 0);
        ysh = terms + (size_t)bufs * waves * chunk * WORDS * 256u;  // (bufs 0: KS = 1)
        total = ysh + (RES ? (size_t)tpw * 64u : 0);
    }
};

// A row's terms are added as one wave walking the row adds them, whatever KS
// is, so an organ's sums are the same bits alone, in a set of any size and as
// an lm_head.  SPLIT_WALK (KS = 1): a wave walks its tiles (t0 + its index, +
// TS, ...).  Else (KS > 1) the workgroup takes TS tiles a round, wave k of a
// tile its steps k, k + KS, ... (BLOCK_SUMS: its blocks of four steps, the same
// way); the waves leave each lane's {scale, v} (the block's sum) in LDS and,
// every four items, one wave per tile (another each round) adds them in order,
// while the others are in the next items.  Every wave runs the same number of
// items, so all meet at each barrier; items past the tile's steps load a valid
// one and leave {-0, 0} (add nothing to the block), which changes no sum.  (The
// chain is in the code once: inlined after every item of the unrolled loop it
// cost up to 1 us of instruction fetches, 20 q8 512 x 2048 5.6 against 5.1.)
// SPLIT_ONCE: one round whose items are all in flight from the start
// (SPLIT_CHUNKS the rest): as straight code instead of the loops' it is 0.1-0.35
// us faster (20 mixed 512 x 2048 4.30 -> 4.12, 20 Q4 4.35 -> 4.03, 10 q8 4.08 ->
// 3.80).
// RES: the HGRAVR02 residual added to the base sums in the same launch (256
// threads; one round; records loaded before the image build).
// HEAD: x is the hidden state; the prologue forms RMSNorm(1+w) of it and the
// epilogue folds the rows' greedy keys (HeadArgs; cols <= 8192, 512 threads).
// NT: the weight loads carry the non-temporal hint.
template <int KIND, int MODE, bool RES, bool HEAD, bool NT = false>
__global__ void __launch_bounds__(RES ? 256 : 1024) gemv_split_kernel(SplitArgs a) {
    constexpr bool SPLIT = MODE != SPLIT_WALK;
    static_assert(!(RES && HEAD), "an lm_head has no fused residual");
    constexpr uint32_t D = split_depth<KIND>;
    constexpr uint32_t TERMS = SplitLds<KIND, RES>::TERMS;
    extern __shared__ __align__(16) uint8_t lds[];
    __shared__ float red[HEAD ? 16 : 1];
    __shared__ uint64_t kred[HEAD ? 16 : 1];
    uint32_t oi, part;
    organ_part(blockIdx.x, a.parts, a.n, &oi, &part);
    OrganView o = a.one;
    ResView rv = a.res_one;
    if (a.organs) {
        o = a.organs[oi];
        if constexpr (RES) rv = a.res[oi];
    }
    const float* __restrict__ x = a.x + (size_t)oi * a.x_stride;
    float* __restrict__ y = a.y + (size_t)oi * a.y_stride;
    const int lane = threadIdx.x & 63, q = lane >> 4;
    const uint32_t wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), nthr = blockDim.x;
    const uint32_t S = o.steps, KS = 1u << a.ks_log, TS = 1u << a.ts_log;
    const uint32_t ksl = wave & (KS - 1u), tsl = wave >> a.ks_log;
    const uint32_t t0 = part * a.tpw, t1 = min(t0 + a.tpw, o.n_tiles);
    // SPLIT: per items a tile and wave, D of them in flight
    const uint32_t per = SPLIT ? split_per<KIND>(S, a.ks_log) : S;
    // (KS = 1: a wave may have no tile)
    const uint32_t rounds = SPLIT || t0 + tsl < t1 ? (t1 - t0 - (SPLIT ? 0u : tsl) + TS - 1u) >> a.ts_log : 0u;
    const uint32_t n = rounds * per;
    const SplitLds<KIND, RES> M(S, o.cols, a.tpw, nthr >> 6, per, a.bufs);

    constexpr int NC = 2;  // (HEAD: 512 threads x 2 chunks = 8192 columns, all in registers)
    XChunks<NC> xc;
    load_x<NC>(BlockTeam{}, x, o.cols, xc);
    XChunks<HEAD ? NC : 1> gw;
    if constexpr (HEAD) {
        if (a.ha.norm_w4) load_x<NC>(BlockTeam{}, a.ha.norm_w, o.cols, gw);
        else load_norm_w<NC>(a.ha.norm_w, o.cols, gw);
    }
    RiceTile rt;
    const uint32_t r0 = t0 * 16u, r1 = min(t1 * 16u, o.rows);
    if constexpr (RES) rice_ranges(rv, r0, r1, rt);
    // the first D items, unconditionally (past its last a wave re-reads a valid
    // one)
    uint32_t fT = t0 + tsl, fj = 0, fi = 0;
    auto step_on = [&]() {
        if constexpr (SPLIT) {
            ++fj;
        } else if (++fi < n && ++fj == per) {
            fj = 0;
            fT += TS;
        }
    };
    auto f_tile = [&]() { return min(fT, t1 - 1u); };
    auto nth = [&](uint32_t j) {  // SPLIT: the step of this wave's item j
        return BLOCK_SUMS<KIND> ? 4u * (ksl + (j >> 2 << a.ks_log)) + (j & 3u) : ksl + (j << a.ks_log);
    };
    auto f_step = [&]() { return SPLIT ? min(nth(min(fj, per - 1u)), S - 1u) : fj; };
    Frag<KIND, 1> f[D];
    if constexpr (KIND == HK_MIXED) {
        uint4 h[D];
#pragma unroll
        for (uint32_t d = 0; d < D; ++d) {
            h[d] = ldg(o.hdr + (f_tile() * S + f_step()));
            step_on();
        }
#pragma unroll
        for (uint32_t d = 0; d < D; ++d) fetch_mixed<1>(o, h[d], lane, f[d], 0);
    } else {
#pragma unroll
        for (uint32_t d = 0; d < D; ++d) {
            fetch_one<KIND, 1, NT>(o, f_tile(), f_step(), lane, f[d], 0);
            step_on();
        }
    }
    if constexpr (RES) rice_first_records(rv, rt);
    if constexpr (HEAD) head_norm_chunks<NC>(xc, gw, o.cols, a.ha, red);

    const uint32_t nch = S * (uint32_t)Kcfg<KIND>::STEP_COLS / 8u;
    float* sx = reinterpret_cast<float*>(lds + (size_t)S * Kcfg<KIND>::P * A_TILE_STRIDE);
    float* xs = reinterpret_cast<float*>(lds + M.xs);
    for (uint32_t i = threadIdx.x; i < S * (uint32_t)Kcfg<KIND>::P; i += nthr)
        *reinterpret_cast<uint4*>(lds + (size_t)i * A_TILE_STRIDE + 256u) = make_uint4(0u, 0u, 0u, 0u);
    bool bad = false;  // (a plain GEMV's non-finite x gives zeroed units and no flag)
    auto image = [&](uint32_t ch, float4 (&v)[2]) {
        if constexpr (RES) {
            if (8u * ch < o.cols) {
                reinterpret_cast<float4*>(xs)[2u * ch] = v[0];
                reinterpret_cast<float4*>(xs)[2u * ch + 1u] = v[1];
            }
        }
        bad |= image_chunk<KIND>(ch, v, lds, sx, 0u, 0u);
    };
#pragma unroll
    for (int j = 0; j < NC; ++j) {
        const uint32_t ch = threadIdx.x + nthr * (uint32_t)j;
        if (ch < nch) image(ch, xc.v[j]);
    }
    if constexpr (!HEAD) for (uint32_t ch = threadIdx.x + nthr * NC; ch < nch; ch += nthr) {
        float4 v[2];
        load_chunk(x, 8u * ch, o.cols, v);
        image(ch, v);
    }
    __syncthreads();
    if constexpr (HEAD) {
        if (bad) {
            if (a.status) atomicOr(a.status, 1u);
            atomicOr(reinterpret_cast<uint32_t*>(a.ha.key + 1), 1u);
        }
    }

    const ImageA A{lds, a_lane_offset(lane)};
    float2* terms = reinterpret_cast<float2*>(lds + M.terms) + (uint32_t)lane * TERMS;  // + 64 TERMS a step
    float* sums = reinterpret_cast<float*>(lds + M.terms) + lane;                      // BLOCK_SUMS: + 64 a block
    float* ysh = reinterpret_cast<float*>(lds + M.ysh);
    uint64_t best = 0;
    auto put_tile = [&](uint32_t T, float v) {  // v: this lane's part of the tile's row sums
        v = tile_row_sum(v);
        const uint32_t row = T * 16u + (uint32_t)lane;
        if (lane >= 16) return;
        if constexpr (RES) {
            ysh[row - r0] = v;
        } else if (row < o.rows) {
            y[row] = v;
            if constexpr (HEAD)
                if (row < a.ha.n_valid) best = max(best, greedy_key(v, row));
        }
    };
    float acc = 0.0f;  // SPLIT: of the tile that this wave sums
    BlockSum bs;
    if constexpr (SPLIT) {
        uint32_t buf = 0;
        float blk = 0.0f;
        // adds up items jb .. jb + 3 of every wave of tile T (k-th of its
        // round), in order; last: and ends the row
        auto sum = [&](uint32_t T, uint32_t k, uint32_t jb, bool last) {
            if constexpr (BLOCK_SUMS<KIND>) {
                const float* t = sums + (((buf << a.ts_log) + k) << a.ks_log) * 64u;
                const uint32_t b0 = jb / 4u << a.ks_log;  // (KS > 2: a multiple of 4)
                auto add = [&](auto count) {
                    constexpr uint32_t N = decltype(count)::value;
                    float e[N];
#pragma unroll
                    for (uint32_t u = 0; u < N; ++u) e[u] = t[u * 64u];
#pragma unroll
                    for (uint32_t u = 0; u < N; ++u) bs.add(N > 2u ? u : b0 + u, e[u]);
                    t += N * 64u;
                };
                if (KS >= 8u)
                    for (uint32_t i = KS >> 3; i; --i) add(std::integral_constant<uint32_t, 8>{});
                else if (KS == 4u) add(std::integral_constant<uint32_t, 4>{});
                else add(std::integral_constant<uint32_t, 2>{});
            } else {
                const float2* t = terms + (((buf << a.ts_log) + k) * M.chunk << a.ks_log) * 64u * TERMS;
                const uint32_t m = (min(4u, per - jb) << a.ks_log) * TERMS;  // a multiple of 2
                auto add = [&](auto count) {
                    constexpr uint32_t N = decltype(count)::value;
                    float2 e[N];
#pragma unroll
                    for (uint32_t u = 0; u < N; ++u) e[u] = t[u / TERMS * 64u * TERMS + u % TERMS];
#pragma unroll
                    for (uint32_t u = 0; u < N; ++u) acc = __builtin_fmaf(e[u].x, e[u].y, acc);
                    t += N * 64u;
                };
                for (uint32_t i = m >> 4; i; --i) add(std::integral_constant<uint32_t, 16>{});
                if (m & 8u) add(std::integral_constant<uint32_t, 8>{});
                if (m & 4u) add(std::integral_constant<uint32_t, 4>{});
                if (m & 2u) add(std::integral_constant<uint32_t, 2>{});
            }
            if (last) put_tile(T, row_total<KIND>(acc, bs));
        };
        auto leave = [&](uint32_t j0, uint32_t d) {  // item j0 + d
            if (j0 + d >= per) return;
            const uint32_t cs = nth(j0 + d);
            if constexpr (BLOCK_SUMS<KIND>) {  // (D is a block)
                if (d == 0) blk = 0.0f;
                if (cs < S) compute_step<KIND, 1>(f[d], cs, A, sx, q, &blk);
                if (d == D - 1u) sums[((((buf << a.ts_log) + tsl) << a.ks_log) + ksl) * 64u] = blk;
                return;
            }
            float2* o2 =
                terms + (((((buf << a.ts_log) + tsl) * M.chunk + (j0 & 3u) + d) << a.ks_log) + ksl) * 64u * TERMS;
            if (cs < S) {
                compute_terms<KIND, 1>(f[d], cs, A, sx, q, [&](int, float s, float v) { *o2++ = make_float2(s, v); });
            } else {
#pragma unroll
                for (uint32_t u = 0; u < TERMS; ++u) o2[u] = make_float2(-0.0f, 0.0f);
            }
        };
        if constexpr (MODE == SPLIT_ONCE) {
#pragma unroll
            for (uint32_t d = 0; d < D; ++d) leave(0, d);
            __syncthreads();
            if (wave < TS && t0 + wave < t1) sum(t0 + wave, wave, 0, true);
        } else {
            for (uint32_t round = 0; round < rounds; ++round)
                for (uint32_t j0 = 0; j0 < per; j0 += D) {
                    // chunks of 4 items: this group's first slot
                    const uint32_t c0 = j0 & 3u;
                    const bool last = j0 + D >= per;  // of the tile
                    if (last) {
                        fj = 0;
                        fT += TS;
                    }
                    // (two bodies: a load under a condition would have every
                    // later item wait for all loads)
                    if (!last || round + 1u < rounds) {
#pragma unroll
                        for (uint32_t d = 0; d < D; ++d) {
                            leave(j0, d);
                            fetch_one<KIND, 1, NT>(o, f_tile(), f_step(), lane, f[d], 0);
                            step_on();
                        }
                    } else {
#pragma unroll
                        for (uint32_t d = 0; d < D; ++d) leave(j0, d);
                    }
                    if (!last && c0 + D < 4u) continue;
                    __syncthreads();
                    // the round's tiles, one tile per wave
                    const uint32_t k = (wave - (round << a.ts_log)) & ((nthr >> 6) - 1u), T = t0 + (round << a.ts_log) + k;
                    if (k < TS && T < t1) sum(T, k, j0 - c0, last);
                    buf ^= a.bufs - 1u;
                }
        }
    } else {
        uint32_t cT = t0 + tsl, cj = 0, it = 0;
        auto consume = [&](const Frag<KIND, 1>& fr) {
            compute_step<KIND, 1>(fr, cj, A, sx, q, &acc);
            end_step<KIND, 1>(cj, &acc, &bs);
            if (++cj < per) return;
            put_tile(cT, row_total<KIND>(acc, bs));
            cj = 0;
            cT += TS;
        };
        for (; it + D < n; it += D) {
#pragma unroll
            for (uint32_t d = 0; d < D; ++d) {
                consume(f[d]);
                fetch_one<KIND, 1, NT>(o, f_tile(), f_step(), lane, f[d], 0);
                step_on();
            }
        }
#pragma unroll
        for (uint32_t d = 0; d < D; ++d)
            if (it + d < n) consume(f[d]);
    }

    if constexpr (RES) {
        __syncthreads();
        float racc[2];
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            const uint32_t i = threadIdx.x + 256u * (uint32_t)h;
            racc[h] = r0 + i < r1 ? ysh[i] : 0.0f;
        }
        rice_batches_from(rv, rt, rt.e0 & ~7u, racc, xs, reinterpret_cast<float*>(lds + M.vals));
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            const uint32_t row = r0 + threadIdx.x + 256u * (uint32_t)h;
            if (row < r1) y[row] = racc[h];
        }
    }
    if constexpr (HEAD) fold_key(best, kred, a.ha.key);
}

// Launch shape (R tiles per wave group, D steps in flight, tiles per
// workgroup) by kind and size, from sweeps over the streamed workloads:
// binary 2-tile groups 5 deep, over 16 tiles when the organ has >= 4 steps
// (also with the fused residual), else over 32; Q4 and Q8 2 over 32, 3 deep;
// 3-bit factors 2 over 16, or over 128 when narrow; mixed (large fragments)
// 1 over 16 (1 over 32 and 1 over 64 measured 1.3 % slower on 6,144 organs of
// 512 x 2048).  With the weights' non-temporal loads (fetch_one) the wide
// binary shape moved from 4-tile groups 3 deep (0.73 of 8 TB/s with the hint,
// 0.756 without) to 2-tile groups 5 deep (0.78-0.80; 4 deep 0.70, 6 deep
// 0.71, 4-tile groups 4 deep 0.56), and the fused residual's with it (0.69
// -> 0.73).
// (build-time overrides for launch-shape sweeps)
#ifndef HK_BIN_NARROW_R
#define HK_BIN_NARROW_R 2
#define HK_BIN_NARROW_D 5
#define HK_BIN_NARROW_TPW 32
#endif
#ifndef HK_BIN_WIDE_R
#define HK_BIN_WIDE_R 2
#define HK_BIN_WIDE_D 5
#endif
#ifndef HK_Q_R
#define HK_Q_R 2
#define HK_Q_D 3
#endif
#ifndef HK_RES_R
#define HK_RES_R 2
#define HK_RES_D 5
#endif
#ifndef HK_BIN_WIDE_TPW
#define HK_BIN_WIDE_TPW 16
#endif
#ifndef HK_Q_TPW
#define HK_Q_TPW 32
#endif
#ifndef HK_MIX_R
#define HK_MIX_R 1
#define HK_MIX_D 3
#define HK_MIX_TPW 16
#endif
constexpr uint64_t MALL_BYTES = 256ull << 20;  // the Infinity Cache

struct SplitShape {
    uint32_t waves, ks, tpw;  // waves 0: the launch is not split
};

static uint32_t pow2_ceil(uint32_t v) {
    uint32_t p = 1;
    while (p < v) p *= 2u;
    return p;
}

// Where the split pays and its shape (us per launch, 20 launches in a graph;
// against the walk of gemv_tiled_kernel; organs of 512 x 2048 unless stated).
// A shape is waves / waves a tile / tiles a workgroup.
//   * one step (<= 512 binary columns): nothing to split (2.95 against 3.1-3.35);
//   * up to 1,024 row tiles the workgroups are what is scarce: about one per
//     CU, so tpw = tiles / 256 rounded up to a power of two, and as many waves
//     as the steps and the image (one chunk of 8 columns a thread) employ; Q4
//     and q8: as many waves a tile as the row has blocks (up to 16 / tpw), so
//     that every step is in flight at once.  One Q4 2048 x 7168: 14.2 -> 4.8, q8
//     4096 x 2048: 7.6 -> 3.4, q8 2048 x 7168: 21.8 -> 5.6, binary 4096 x 2048:
//     4.1 -> 3.35; 20 mixed organs (640 tiles): 5.35 -> 4.1; 20 Q4 organs: 6.8
//     -> 4.0; 10 Q4 organs of 23 steps 16/8/2 4.1, 8/4/2 4.7; one q8 organ of 36
//     steps 16/16/1 3.7, 8/8/1 4.35.  Rows of five to eight blocks in 513 to 704
//     tiles: 8/8/1 (23 q8 organs of 22 steps 4.5, 16/4/4 5.0);
//   * Q4 and q8 rows of eight blocks or more where three or five tiles a
//     workgroup give each CU one (a power of two leaves some idle): all waves
//     on one tile after the other (33 q8 organs 7.6 -> 7.25, with 7168 columns
//     21.3 -> 19.7; Q4 11,000 x 4096 6.7 -> 5.9, 23 Q4 organs of 36 steps 8.0 ->
//     6.6);
//   * up to 2,048 tiles one wave per tile, 8/1/8 (binary 4.4 -> 3.9, mixed 5.2 ->
//     4.6; 40 Q4 organs with 7168 columns: 25.4 -> 15.1), but up to five tiles a
//     CU 8/4/2 for rows of four blocks (Q4 20,000 x 2048 5.1 against 6.4) and
//     for five to eight 16/8/6 (40 Q4 organs of 26 steps 7.2, 8/8/1 8.0) or, q8,
//     8/8/1 (of 26 steps 6.3, 16/8/6 6.4);
//   * q8 rows whose blocks divide by eight, or long ones that about fill four
//     waves: 8/4/2 above 1,280 tiles (64 organs 12.3 against 14.3, with 7168
//     columns 36.1 against 38, 100 organs 18.1); others leave waves without a
//     block, 8/1/8 (64 organs of 22 steps 8.4 against 9.3, of 36 steps 12.05
//     against 13.1; 110 organs of 45 steps 22.8 against 23.7).  Q4 of more than 16 steps 8/1/8 up to 4,096 tiles
//     (100 organs with 7168 columns: 40 -> 31.5, 8/4/2 33.7); of up to 16 steps it
//     walks (80 organs: 9.4 against 9.8);
//   * the short kinds 4/1/4 up to 4,096 tiles (mixed 6.05 -> 5.63, binary 5.07 ->
//     4.88), mixed (8.9 -> 8.05) and q8 (200 organs: 42.7 -> 36.6) up to the
//     streamed shapes; the others' walk is faster there (binary 320 organs: 9.7
//     against 10.8; 200 Q4 organs: 20.1 against 19.9, with 7168 columns equal).
// HEAD: every workgroup ends in one atomic max on the same word, which the
// memory side takes at about 12 ns each (a binary 151,936 x 2048 lm_head: 15.1
// us over 256 workgroups, 16.2 over 594, 23.2 over 1,187), so one or two
// balanced workgroups per CU, 8 waves each.  One wave per tile for binary, for
// short rows (q8 32,000 x 1024 11.3 against 12.2 with four waves a tile) and for
// rows whose blocks do not divide by four (q8 16,536 x 1408 10.6 against 11.9,
// 65,000 x 2304 26.9 against 28.5, 151,936 x 3328 77.5 against 83.5; Q4 30,000 x
// 2304 12.5 against 15.0), four else (q8 151,936 x 2048 49.7 against 52; 65,000
// rows 25.3).  With at most two tiles a CU four waves, two for 17 to 23 steps
// (q8 8,000 x 1408 9.6, four 10.2, one 9.9; x 2880 10.7, 11.6, 13.2); eight
// where three tiles a workgroup give each CU one and the blocks divide (q8
// 11,409 x 2048 10.8, four 11.1, one 11.4).  A q8 lm_head larger than the
// Infinity Cache loads non-temporally with one workgroup per CU (128,256 x 4096:
// 96.2 -> 78; below, the hint and the fewer loads in flight cost: 65,000 rows
// 25.9 -> 34.8; Q4 of these sizes fits and gains nothing from it); tile counts
// that leave a nearly empty last round cost up to 30 %.
// RES (256 threads, at most 4 tiles a workgroup: a row's records are one
// thread's chain) replaces two launches: one organ 7.8 -> 5.0, 40 organs 8.8
// -> 6.6, 512 x 7168: 35.4 -> 8.7; above 4,096 tiles the two launches are
// faster (160 organs: 11.0 against 11.8).
static SplitShape split_shape(int kind, bool res, bool head, uint32_t n, uint32_t n_tiles, uint32_t S, uint32_t cols) {
    const uint64_t tiles = (uint64_t)n * n_tiles;
    const bool wide = kind == HK_Q4 || kind == HK_Q8;
    const uint32_t nb = (S + 3u) / 4u;  // blocks of a Q4 or q8 row
    if (head) {
        const uint32_t even = (uint32_t)((tiles + 255u) / 256u);
        uint32_t ks = nb % 4u == 0 && (S > 16 || tiles > 2048) ? 4u : 1u;
        if (tiles <= 512) ks = nb % 4u == 0 || S >= 24 ? 4u : 2u;
        else if (even == 3 && nb % 8u == 0) ks = 8;
        if (kind == HK_BIN || S <= 8) ks = 1;
        const uint32_t ts = 8u / ks;
        const bool past_mall = kind == HK_Q8 && tiles * 16u * cols > MALL_BYTES;
        const uint32_t wgs = kind == HK_BIN || tiles <= 4096 || past_mall ? 256u : 512u;
        const uint32_t per_wg = (uint32_t)((tiles + wgs - 1u) / wgs);
        return {8, ks, std::min((per_wg + ts - 1u) / ts * ts, 64u)};
    }
    const uint32_t tpw = std::min(pow2_ceil((uint32_t)((tiles + 255) / 256)), 4u);
    if (res) {
        if (tiles > 4096) return {0, 0, 0};
        const uint32_t ks = std::min(std::max(4u / tpw, 1u), pow2_ceil(S));
        return {4, ks, std::max(tpw, 4u / ks)};
    }
    if (S == 1 || tiles >= 16384) return {0, 0, 0};
    if (!wide) {
        if (tiles <= 1024) {
            const uint32_t w = cols > 4096 || (S >= 16 && tpw == 4) ? 16u : S < 16 && tpw == 1 ? 4u : 8u;
            const uint32_t ks = std::min(w / tpw, pow2_ceil(S));
            return {w, ks, std::max(tpw, w / ks)};
        }
        if (tiles <= 2048) return {8, 1, 8};
        return tiles <= 4096 || kind == HK_MIXED ? SplitShape{4, 1, 4} : SplitShape{0, 0, 0};
    }
    if (nb >= 8 && tiles > 512 && tiles <= 1280) {
        uint32_t even = 3;
        while (even < 5 && (uint64_t)n * ((n_tiles + even - 1u) / even) > 256u) ++even;
        const uint32_t w = nb > 8 ? 16u : 8u;
        const bool full = nb <= 16 || 4u * ((nb + 15u) / 16u) * 16u <= 5u * nb;  // (a wave's last block used)
        if (full && even != 4 && (uint64_t)n * ((n_tiles + even - 1u) / even) <= 256u) return {w, w, even};
    }
    if (nb >= 5 && nb <= 8 && ((tiles > 512 && tiles <= 704) || (tiles > 1024 && tiles <= 1280)))
        return kind == HK_Q4 && tiles > 1024 ? SplitShape{16, 8, 6} : SplitShape{8, 8, 1};
    if (tiles <= 1024) {
        const uint32_t w = nb <= 2 ? (tpw <= 2 ? 4u : 8u) : nb <= 4 ? (tpw == 4 ? 16u : 8u) : nb <= 8 && tpw == 1 ? 8u : 16u;
        const uint32_t ks = std::min(w / tpw, pow2_ceil(nb));
        return {w, ks, std::max(tpw, w / ks)};
    }
    if (nb == 4 && tiles <= 1280) return {8, 4, 2};
    const bool four = kind == HK_Q8 && (nb % 8u == 0 || (nb >= 16 && (nb + 3u) / 4u * 4u * 8u <= 9u * nb));
    if (tiles <= 2048 || (S > 16 && tiles <= 4096)) return four ? SplitShape{8, 4, 2} : SplitShape{8, 1, 8};
    if (kind == HK_Q8 && S >= 16 && tiles > 4096) return {8, 4, 2};
    return {0, 0, 0};
}

template <int KIND, bool RES, bool HEAD = false>
static hipError_t launch_split(const OrganView* organs, const ResView* res, const ResView* res_one, uint32_t n,
                               const OrganView& sh, const float* x, size_t xs, float* y, size_t ys, hipStream_t s,
                               bool* done, const HeadArgs& ha = {}, uint32_t* status = nullptr) {
    *done = false;
    const SplitShape c = split_shape(KIND, RES, HEAD, n, sh.n_tiles, sh.steps, sh.cols);
    if (!c.waves || (!HEAD && vectors_overlap(x, xs, sh.cols, y, ys, sh.rows, n))) return hipSuccess;
    const uint32_t waves = c.waves, ks = c.ks, tpw = c.tpw, ts = waves / ks;
    const uint32_t per = split_per<KIND>(sh.steps, (uint32_t)__builtin_ctz(ks));
    const uint32_t bufs = ks == 1u ? 0u : tpw == ts && per <= 4u ? 1u : 2u;
    const size_t lds = SplitLds<KIND, RES>(sh.steps, sh.cols, tpw, waves, per, bufs).total;
    if (lds > SPLIT_LDS_LIMIT) return hipSuccess;
    if (RES && (!organs || !res) && !(n == 1 && res_one)) return hipErrorInvalidValue;
    *done = true;
    SplitArgs a{};
    a.ks_log = (uint32_t)__builtin_ctz(ks);
    a.ts_log = (uint32_t)__builtin_ctz(ts);
    a.bufs = bufs;
    a.one = sh;
    // one organ's view comes with the arguments where the host has its
    // residual's too (a set of one has that only in its device table)
    a.organs = n > 1 || (RES && !res_one) ? organs : nullptr;
    if (res_one) a.res_one = *res_one;
    a.res = res;
    a.x = x;
    a.y = y;
    a.x_stride = xs;
    a.y_stride = ys;
    a.n = n;
    a.parts = (sh.n_tiles + tpw - 1) / tpw;
    a.tpw = tpw;
    a.ha = ha;
    a.status = status;
    const bool nt = HEAD && KIND == HK_Q8 && (uint64_t)sh.rows * sh.cols > MALL_BYTES;
    auto* k = ks > 1 ? nt ? gemv_split_kernel<KIND, SPLIT_CHUNKS, RES, HEAD, HEAD && KIND == HK_Q8>
                          : gemv_split_kernel<KIND, SPLIT_CHUNKS, RES, HEAD>
              : nt   ? gemv_split_kernel<KIND, SPLIT_WALK, RES, HEAD, HEAD && KIND == HK_Q8>
                     : gemv_split_kernel<KIND, SPLIT_WALK, RES, HEAD>;
    if constexpr (!HEAD)
        if (ks > 1 && tpw == ts && per <= split_depth<KIND>) k = gemv_split_kernel<KIND, SPLIT_ONCE, RES, HEAD>;
    hipLaunchKernelGGL(k, dim3(a.parts * n), dim3(64u * waves), lds, s, a);
    return hipGetLastError();
}

template <int KIND>
static hipError_t launch_r(const OrganView* organs, uint32_t n, const OrganView& sh, const float* x, size_t xs,
                           float* y, size_t ys, hipStream_t s) {
    const uint64_t tiles = (uint64_t)n * sh.n_tiles;
    bool done = false;
    const hipError_t e = launch_split<KIND, false>(organs, nullptr, nullptr, n, sh, x, xs, y, ys, s, &done);
    if (e != hipSuccess || done) return e;
    if (tiles >= 16384) {
        if constexpr (KIND == HK_BIN) {
            if (sh.steps >= 4)
                return launch_kind<KIND, HK_BIN_WIDE_R, HK_BIN_WIDE_D>(organs, n, sh, x, xs, y, ys, HK_BIN_WIDE_TPW, s);
            return launch_kind<KIND, HK_BIN_NARROW_R, HK_BIN_NARROW_D>(organs, n, sh, x, xs, y, ys, HK_BIN_NARROW_TPW, s);
        } else if constexpr (KIND == HK_U3) {
            // narrow factors: up to 128 tiles share an image, as long as 1,024
            // workgroups remain
            const bool one = vectors_overlap(x, xs, sh.cols, y, ys, sh.rows, n);  // (one workgroup an organ)
            const uint32_t share = one ? 128u : (uint32_t)std::min<uint64_t>(std::max<uint64_t>(tiles / 1024u, 16u), 128u) & ~7u;
            return launch_kind<KIND, 2, 3>(organs, n, sh, x, xs, y, ys, gemv_max_tiles(KIND, sh.steps) == 128u ? share : 16, s);
        } else if constexpr (KIND == HK_Q4 || KIND == HK_Q8) {
            return launch_kind<KIND, HK_Q_R, HK_Q_D>(organs, n, sh, x, xs, y, ys, HK_Q_TPW, s);
        } else {
            return launch_kind<KIND, HK_MIX_R, HK_MIX_D>(organs, n, sh, x, xs, y, ys, HK_MIX_TPW, s);
        }
    }
    if (tiles >= 4096) return launch_kind<KIND, 2, 2>(organs, n, sh, x, xs, y, ys, 8, s);
    const uint32_t tpw = (uint64_t)n * ((sh.n_tiles + 3) / 4) >= 256 ? 4 : 1;
    return launch_kind<KIND, 1, 2>(organs, n, sh, x, xs, y, ys, tpw, s);
}

// The terminal head on a packed lm_head of at most 8192 columns: one GEMV
// launch with the norm prologue and the greedy-key epilogue, then the
// one-thread pick (which also clears the key for the next call), against four
// launches of its parts.
__global__ void head_pick_fused_kernel(uint64_t* __restrict__ key, int32_t* __restrict__ token, uint32_t* status) {
    if (threadIdx.x == 0) {
        const uint64_t best = key[0];
        const uint32_t flag = reinterpret_cast<const uint32_t*>(key + 1)[0];
        const uint32_t ord = (uint32_t)(best >> 32);
        const float v = __uint_as_float((ord & 0x80000000u) ? (ord & 0x7FFFFFFFu) : ~ord);
        const bool ok = best != 0ull && isfinite(v) && flag == 0u;
        token[0] = ok ? (int32_t)(~(uint32_t)best) : -1;
        if (!ok) atomicOr(status, 1u);
        key[0] = 0ull;
        key[1] = 0ull;
    }
}

bool head_gemv_fusable(const OrganView& sh) {
    return (sh.kind == HK_Q8 || sh.kind == HK_Q4 || sh.kind == HK_BIN) &&
           sh.steps * tile_step_cols(sh.kind) <= 8192u;
}

template <int KIND>
static hipError_t launch_head_gemv(const OrganView& sh, const float* h, float* logits, const HeadArgs& ha,
                                   uint32_t* status, hipStream_t s) {
    bool done = false;
    const hipError_t e = launch_split<KIND, false, true>(nullptr, nullptr, nullptr, 1, sh, h, 0, logits, 0, s, &done, ha,
                                                         status);
    return e != hipSuccess || done ? e : hipErrorInvalidValue;  // (at most 55 KB of LDS: always done)
}

hipError_t launch_head_fused(const OrganView& sh, const float* h, const float* norm_w,
                             float eps, float* xn, float* logits, uint32_t n_valid, uint64_t* key, int32_t* token,
                             uint32_t* status, hipStream_t s) {
    if (!head_gemv_fusable(sh)) return hipErrorInvalidValue;
    const HeadArgs ha{norm_w, (reinterpret_cast<uintptr_t>(norm_w) & 15u) == 0, eps, xn, n_valid, key};
    const hipError_t e = sh.kind == HK_Q8   ? launch_head_gemv<HK_Q8>(sh, h, logits, ha, status, s)
                         : sh.kind == HK_Q4 ? launch_head_gemv<HK_Q4>(sh, h, logits, ha, status, s)
                                            : launch_head_gemv<HK_BIN>(sh, h, logits, ha, status, s);
    if (e != hipSuccess) return e;
    hipLaunchKernelGGL(head_pick_fused_kernel, dim3(1), dim3(64), 0, s, key, token, status);
    return hipGetLastError();
}

hipError_t launch_gemv_rice(const OrganView* organs_dev, const ResView* res_dev, const ResView* res_one, uint32_t n,
                            const OrganView& sh, uint32_t pieces256, uint32_t pieces512, const float* x,
                            size_t x_stride, float* y, size_t y_stride, hipStream_t s, bool* fused) {
    *fused = false;
    if (sh.kind == HK_BIN) {
        const hipError_t e = launch_split<HK_BIN, true>(organs_dev, res_dev, res_one, n, sh, x, x_stride, y, y_stride, s,
                                                        fused);
        if (e != hipSuccess || *fused) return e;
    }
    // the streamed binary shapes (launch_r), with x in one register chunk
    if (sh.kind != HK_BIN || (uint64_t)n * sh.n_tiles < 16384 || x_image_cols<HK_BIN>(sh.steps) > 2048u)
        return hipSuccess;
    const bool wide = sh.steps >= 4;
    const uint32_t tpw = wide ? HK_BIN_WIDE_TPW : HK_BIN_NARROW_TPW, pieces = wide ? pieces256 : pieces512;
    static_assert(HK_BIN_WIDE_TPW * 16 == 256 && HK_BIN_NARROW_TPW * 16 == 512, "RES rows per workgroup");
    // the fused kernel runs 4 workgroups per CU (its registers): LDS up to a
    // quarter of the CU's 160 KiB costs no occupancy
    if (pieces == 0 || pieces > 256u * GEMV_RES_NP ||
        gemv_ysh_offset<HK_BIN, true>(sh.steps, tpw, sh.cols, pieces) + (size_t)tpw * 64u > 40u * 1024u)
        return hipSuccess;
    const ResArgs ra{res_dev, pieces};
    *fused = true;
    if (wide)
        return launch_kind<HK_BIN, HK_RES_R, HK_RES_D, true>(organs_dev, n, sh, x, x_stride, y, y_stride, tpw, s, ra);
    return launch_kind<HK_BIN, HK_BIN_NARROW_R, HK_BIN_NARROW_D, true>(organs_dev, n, sh, x, x_stride, y, y_stride, tpw, s, ra);
}

hipError_t launch_gemv_tiled(const OrganView* organs_dev, uint32_t n, const OrganView& sh, const float* x,
                             size_t x_stride, float* y, size_t y_stride, hipStream_t s) {
    switch (sh.kind) {
    case HK_F32:
        hipLaunchKernelGGL(gemv_f32_kernel, dim3((sh.rows + 3) / 4, n), dim3(256), 0, s, organs_dev, x, x_stride,
                           y, y_stride);
        return hipGetLastError();
    case HK_BIN: return launch_r<HK_BIN>(organs_dev, n, sh, x, x_stride, y, y_stride, s);
    case HK_Q4: return launch_r<HK_Q4>(organs_dev, n, sh, x, x_stride, y, y_stride, s);
    case HK_MIXED: return launch_r<HK_MIXED>(organs_dev, n, sh, x, x_stride, y, y_stride, s);
    case HK_Q8: return launch_r<HK_Q8>(organs_dev, n, sh, x, x_stride, y, y_stride, s);
    case HK_U3: return launch_r<HK_U3>(organs_dev, n, sh, x, x_stride, y, y_stride, s);
    default: return hipErrorInvalidValue;
    }
}

}  // namespace hk
