// Tile rasterizer forward: one workgroup per work tile (of any view in
// a batch), front-to-back alpha compositing.
//
// Restates crates/gs-kernels/src/shaders/rasterize_fwd.wgsl:20-85 and
// evaluate_hit of raster_common.wgsl:69-95 (the oracle's forward.rs:207-246).
// MI355X layout: a TW x TW work tile (TW = 8, 16 or 32) is (TW/8)^2 wave64s.
// Surfel records are staged through LDS in batches of BATCH (gathered through
// the sorted payloads); each record's alpha >= 1/255 footprint (box clipped to
// its 16-px rect, screen disk and ellipse, computed at projection) is tested
// against parts of the tile, and every part walks its own order-preserving
// list. For TW = 8 and 16 a part is a 4x4 sub-block and a row of 16 lanes, for
// TW = 32 an 8x8 block and a wave. A wave leaves the batch once its pixels are
// saturated; the workgroup stops when every pixel's transmittance is below
// 1e-4.
//
// Outputs per pixel (same buffers as the reference Rasterizer):
//   color  = (sum w c, sum w),  aux = (T_final, sum w t, 0, 0),
//   normal = (sum w n, 0),      ncontrib = index (within the tile list) just
//   past the last contributing record.

#include "gs_internal.h"

namespace gs {

namespace {

// Locate the view owning a global tile id (views are few; tile_base ascends).
__device__ __forceinline__ uint32_t view_of_tile(const CamParams* cams, uint32_t n_views, uint32_t t) {
    uint32_t v = 0;
    for (uint32_t k = 1; k < n_views; ++k)
        if (cams[k].tile_base <= t) v = k;
    return v;
}

// 32-px work tiles: each wave owns an 8x8 block, and a batch is split into one
// list per block (colour outputs only).
template <int TW, int BATCH>
__global__ __launch_bounds__((TW / 8) * (TW / 8) * 64) void raster_fwd_kernel(
    const CamParams* __restrict__ cams, uint32_t n_views, const uint32_t* __restrict__ ranges,
    const uint32_t* __restrict__ payloads, const Record* __restrict__ recs, FwdOut out, bool cull,
    uint32_t total_tiles, TileQueue queue, uint32_t tile_begin) {
    constexpr int NC = TW / 8;             // blocks per tile row
    constexpr int NB = NC * NC;            // blocks (= waves) per tile
    constexpr int NT = NB * 64;            // threads
    constexpr int SW = BATCH / 64;         // staging waves per batch
    constexpr int SPT = (BATCH + NT - 1) / NT;  // batch slots per thread
    static_assert(BATCH % 64 == 0 && BATCH <= 1024, "batch of whole waves");
    __shared__ float4 s_m[BATCH], s_a[BATCH], s_b[BATCH], s_c[BATCH];
    __shared__ uint16_t s_list[NB][BATCH];
    __shared__ uint32_t s_qcnt[SW][NB];
    __shared__ uint32_t s_view, s_next;

    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const uint32_t all_blocks = NB == 32 ? ~0u : (1u << NB) - 1u;
    for (uint32_t iter = 0;; ++iter) {
        uint32_t pos;
        if (iter == 0) {
            pos = queue.cursor != nullptr ? blockIdx.x : xcd_swizzle(blockIdx.x, gridDim.x);
        } else if (queue.cursor != nullptr) {
            if (tid == 0) s_next = claim_position(queue);
            __syncthreads();
            pos = s_next;
            __syncthreads();  // every thread has pos before s_next is rewritten
        } else {
            pos = total_tiles;
        }
        if (pos >= total_tiles) break;
        const uint32_t gtile = queue.order != nullptr ? queue.order[pos] : tile_begin + pos;
        if (tid == 0) s_view = view_of_tile(cams, n_views, gtile);
        __syncthreads();
        const CamParams& cam = cams[s_view];
        const uint32_t local = gtile - cam.tile_base;
        const uint32_t tx = local % cam.tiles_x, ty = local / cam.tiles_x;
        const uint32_t x0 = tx * TW, y0 = ty * TW;
        const int px = (int)x0 + (wave % NC) * 8 + (lane & 7);
        const int py = (int)y0 + (wave / NC) * 8 + (lane >> 3);
        const bool inside = px < (int)cam.width && py < (int)cam.height;
        float sx, sy;
        pixel_s(cam, px, py, sx, sy);
        const float pxc = (float)px + 0.5f, pyc = (float)py + 0.5f;
        const uint64_t lt_mask = (lane == 0) ? 0ull : (~0ull >> (64 - lane));

        const uint32_t start = ranges[2 * (size_t)gtile], end = ranges[2 * (size_t)gtile + 1];
        // A pixel is done once T < kTTerminate (forward.rs stops there); T
        // only falls, so the test on T itself is the done flag, and pixels
        // outside the image start done (T = 0; nothing of theirs is written).
        float T = inside ? 1.0f : 0.0f;
        float cr = 0.f, cg = 0.f, cb = 0.f, wsum = 0.f;
        uint32_t last = 0;

        for (uint32_t base = start; base < end; base += BATCH) {
            const uint32_t cnt = min((uint32_t)BATCH, end - base);
            uint32_t qm[SPT];
            uint32_t qpos[SPT][NB];
#pragma unroll
            for (int m = 0; m < SPT; ++m) {
                const int slot = tid + m * NT;
                qm[m] = 0;
                if (slot >= BATCH) continue;  // whole waves (NT, BATCH multiples of 64)
                if ((uint32_t)slot < cnt) {
                    Record r = recs[payloads[base + slot]];
                    s_m[slot] = r.m_nt;
                    s_a[slot] = r.a_px;
                    s_b[slot] = r.b_py;
                    s_c[slot] = r.col_op;
                    qm[m] = cull ? block_mask<TW>(r, x0, y0) : all_blocks;
                }
                // Order-preserving split of the batch into per-block lists.
                const int sw = slot >> 6;
#pragma unroll
                for (int q = 0; q < NB; ++q) {
                    const uint64_t bal = __ballot((qm[m] >> q) & 1u);
                    qpos[m][q] = (uint32_t)__popcll(bal & lt_mask);
                    if (lane == 0) s_qcnt[sw][q] = (uint32_t)__popcll(bal);
                }
            }
            __syncthreads();
#pragma unroll
            for (int m = 0; m < SPT; ++m) {
                const int slot = tid + m * NT;
                if (slot >= BATCH) continue;
                const int sw = slot >> 6;
#pragma unroll
                for (int q = 0; q < NB; ++q) {
                    if ((qm[m] >> q) & 1u) {
                        uint32_t off = 0;
                        for (int w = 0; w < sw; ++w) off += s_qcnt[w][q];
                        s_list[q][off + qpos[m][q]] = (uint16_t)slot;
                    }
                }
            }
            uint32_t my_count = 0;
#pragma unroll
            for (int w = 0; w < SW; ++w) my_count += s_qcnt[w][wave];
            __syncthreads();
            if (__any(T >= kTTerminate)) {
                auto load = [&](uint32_t j, Record& r) {
                    r.m_nt = s_m[j];
                    r.a_px = s_a[j];
                    r.b_py = s_b[j];
                    r.col_op = s_c[j];
                    r.nrm_dep = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
                };
                auto composite = [&](uint32_t j, const Record& r) {
                    const HitEval h = eval_hit(r, sx, sy, pxc, pyc);
                    if (T >= kTTerminate && h.hit) {
                        const float w = T * h.a;
                        cr += r.col_op.x * w;
                        cg += r.col_op.y * w;
                        cb += r.col_op.z * w;
                        wsum += w;
                        T *= 1.0f - h.a;
                        last = base - start + j + 1u;
                    }
                };
                // Two records per round: both list entries and both records
                // are read from LDS together (one wait instead of two
                // dependent round trips each), then composited in list order
                // with the same per-record early exit.
                for (uint32_t k = 0; k < my_count; k += 2) {
                    const bool two = k + 1 < my_count;
                    const uint32_t j0 = s_list[wave][k];
                    const uint32_t j1 = two ? (uint32_t)s_list[wave][k + 1] : j0;
                    Record r0, r1;
                    load(j0, r0);
                    load(j1, r1);
                    // One saturation test per round: a wave done after j0
                    // walks j1 with every lane masked off (no contribution).
                    composite(j0, r0);
                    if (!two) break;
                    composite(j1, r1);
                    if (!__any(T >= kTTerminate)) break;
                }
            }
            if (__syncthreads_count(T >= kTTerminate) == 0) break;
        }
        if (inside) {
            const size_t pi = (size_t)cam.pix_base + (size_t)py * cam.width + (size_t)px;
            out.color[pi] = make_float4(cr, cg, cb, wsum);
            out.aux[pi] = make_float4(T, 0.0f, 0.0f, 0.0f);
            out.ncontrib[pi] = last;
        }
        __syncthreads();  // s_view and the LDS batch are reused by the next tile
    }
}

// Waves per SIMD the sub-block kernel is held to: four spilled registers (of
// the staging) at these, and at one more 15, in the walk as well: 1M surfels,
// four 1080p views 507 us at six and 509 at seven, 1283 x 717 79 and 88; with
// depth and normals, 300k at 720p 148 us at five and 200 at six.
template <bool AUX>
constexpr uint32_t kSubWaves = AUX ? 5 : 6;

// Work tiles of 8 or 16 px. Bound by VALU issue (1.25M surfels in sixteen
// 720p views: 823M wave instructions, 1.34 ms at 614 G/s, of 1.39 ms), so the
// lists are per 4x4 sub-block: a wave steps through the longest of its four
// rows' lists instead of the union of them, and a row whose pixels are
// saturated no longer counts. Against lists per 8x8 block and wave, with
// three barriers a batch: 650 -> 507 us for 1M surfels in four 1080p views,
// 1.82 -> 1.27 ms for 1.25M in sixteen 720p views; 8-px tiles 1.15 -> 0.94 ms
// (the first). A record in LDS is read by four rows at four addresses as fast
// as by a wave at one. 32-px tiles would need 64 lists (16 to 64 KB).
// AUX = false (training with colour losses only) skips the depth and normal
// accumulators: aux = (T_final, 0, 0, 0), normal is not written. TRACE
// additionally records every contribution of the trace window's pixels
// (FwdTrace; a verification variant, never used by training steps).
template <bool AUX, int TW, int BATCH, bool TRACE = false>
__global__ __launch_bounds__((TW / 8) * (TW / 8) * 64)
__attribute__((amdgpu_waves_per_eu(TW == 8 ? 4 : kSubWaves<AUX>))) void raster_fwd_sub_kernel(
    const CamParams* __restrict__ cams, uint32_t n_views, const uint32_t* __restrict__ ranges,
    const uint32_t* __restrict__ payloads, const Record* __restrict__ recs, FwdOut out, bool cull,
    uint32_t total_tiles, TileQueue queue, uint32_t tile_begin, FwdTrace trace) {
    constexpr int NC = TW / 8;             // waves per tile row
    constexpr int NT = NC * NC * 64;       // threads
    constexpr int NS = TW / 4;             // sub-blocks per tile row
    constexpr int SPT = (BATCH + NT - 1) / NT;  // batch slots per thread
    static_assert(BATCH % 64 == 0 && BATCH <= 256, "whole waves, 8-bit slots");
    __shared__ float4 s_m[BATCH], s_a[BATCH], s_b[BATCH], s_c[BATCH], s_n[AUX ? BATCH : 1];
    __shared__ uint16_t s_mask[BATCH];     // bit NS r + c: sub-block (c, r)
    __shared__ uint16_t s_list[NS * NS][BATCH / 2 + 1];  // slots, two a word; read one word ahead
    __shared__ uint32_t s_next;

    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    // Row g of the wave: lane p is pixel (p & 3, p >> 2) of sub-block (sc, sr).
    const int g = lane >> 4, p = lane & 15;
    const int sc = 2 * (wave % NC) + (g & 1), sr = 2 * (wave / NC) + (g >> 1);
    const uint64_t lt_mask = (lane == 0) ? 0ull : (~0ull >> (64 - lane));
    const uint16_t* const my_list = s_list[sr * NS + sc];
    for (uint32_t iter = 0;; ++iter) {
        uint32_t pos;
        if (iter == 0) {
            pos = queue.cursor != nullptr ? blockIdx.x : xcd_swizzle(blockIdx.x, gridDim.x);
        } else if (queue.cursor != nullptr) {
            if (tid == 0) s_next = claim_position(queue);
            __syncthreads();
            pos = __builtin_amdgcn_readfirstlane(s_next);
            __syncthreads();  // every thread has pos before s_next is rewritten
        } else {
            pos = total_tiles;
        }
        if (pos >= total_tiles) break;
        const uint32_t gtile = queue.order != nullptr ? queue.order[pos] : tile_begin + pos;
        const uint32_t view = view_of_tile(cams, n_views, gtile);
        const CamParams& cam = cams[view];
        const uint32_t local = gtile - cam.tile_base;
        const uint32_t x0 = local % cam.tiles_x * TW, y0 = local / cam.tiles_x * TW;
        const int px = (int)x0 + 4 * sc + (p & 3), py = (int)y0 + 4 * sr + (p >> 2);
        const bool inside = px < (int)cam.width && py < (int)cam.height;
        float sx, sy;
        pixel_s(cam, px, py, sx, sy);
        const float pxc = (float)px + 0.5f, pyc = (float)py + 0.5f;

        const uint32_t start = ranges[2 * (size_t)gtile], end = ranges[2 * (size_t)gtile + 1];
        // A pixel is done once T < kTTerminate (forward.rs stops there); T
        // only falls, so the test on T itself is the done flag, and pixels
        // outside the image start done (T = 0; nothing of theirs is written).
        float T = inside ? 1.0f : 0.0f;
        float cr = 0.f, cg = 0.f, cb = 0.f, wsum = 0.f, dsum = 0.f, nx = 0.f, ny = 0.f, nz = 0.f;
        uint32_t last = 0;
        // Trace window slot of this pixel (TRACE only).
        const bool traced = TRACE && inside && view == trace.view && (uint32_t)px >= trace.x0 &&
                            (uint32_t)px < trace.x0 + trace.w && (uint32_t)py >= trace.y0 &&
                            (uint32_t)py < trace.y0 + trace.h;
        const size_t tslot = traced ? (size_t)(py - trace.y0) * trace.w + (size_t)(px - trace.x0) : 0;
        uint32_t tcount = 0;

        for (uint32_t base = start; base < end; base += BATCH) {
            const uint32_t cnt = min((uint32_t)BATCH, end - base);
#pragma unroll
            for (int m = 0; m < SPT; ++m) {
                const int slot = tid + m * NT;
                if (slot >= BATCH) continue;  // whole waves (NT, BATCH multiples of 64)
                uint32_t mask = 0;
                if ((uint32_t)slot < cnt) {
                    const Record& r = recs[payloads[base + slot]];
                    const float4 a = r.a_px, b = r.b_py;
                    s_m[slot] = r.m_nt;
                    s_a[slot] = a;
                    s_b[slot] = b;
                    s_c[slot] = r.col_op;
                    if (AUX) s_n[slot] = r.nrm_dep;
                    mask = (1u << NS * NS) - 1u;
                    if (cull) {
                        const SubTest t = sub_test(r.box, r.ell0, r.ell1, a.w, b.w);
                        mask = 0;
#pragma unroll
                        for (int i = 0; i < NS; ++i)
                            mask |= (sub_row_mask(t, (float)x0, (float)(y0 + 4 * i)) & ((1u << NS) - 1u)) << NS * i;
                    }
                }
                s_mask[slot] = (uint16_t)mask;
            }
            __syncthreads();
            if (__any(T >= kTTerminate)) {
                // The wave's four lists, in slot order.
                uint32_t n[4] = {0, 0, 0, 0};
#pragma unroll
                for (int c = 0; c < BATCH / 64; ++c) {
                    const uint32_t slot = (uint32_t)(c * 64 + lane), mask = s_mask[slot];
#pragma unroll
                    for (int q = 0; q < 4; ++q) {
                        const int sub = (2 * (wave / NC) + (q >> 1)) * NS + 2 * (wave % NC) + (q & 1);
                        const bool hit = mask >> sub & 1u;
                        const uint64_t bal = __ballot(hit);
                        if (hit) ((uint8_t*)s_list[sub])[n[q] + (uint32_t)__popcll(bal & lt_mask)] = (uint8_t)slot;
                        n[q] += (uint32_t)__popcll(bal);
                    }
                }
                const uint32_t mine = g == 0 ? n[0] : g == 1 ? n[1] : g == 2 ? n[2] : n[3];
                // off: byte offset of a slot in each of the arrays.
                auto at = [](const float4* a, uint32_t off) { return *(const float4*)((const char*)a + off); };
                auto load = [&](uint32_t off, Record& r) {
                    r.m_nt = at(s_m, off);
                    r.a_px = at(s_a, off);
                    r.b_py = at(s_b, off);
                    r.col_op = at(s_c, off);
                    r.nrm_dep = AUX ? at(s_n, off) : make_float4(0.0f, 0.0f, 0.0f, 0.0f);
                };
                const uint32_t first = base - start + 1;
                auto composite = [&](uint32_t j, const Record& r, bool listed) {
                    const HitEval h = eval_hit(r, sx, sy, pxc, pyc);
                    if (listed & (T >= kTTerminate) & h.hit) {
                        const float w = T * h.a;
                        cr += r.col_op.x * w;
                        cg += r.col_op.y * w;
                        cb += r.col_op.z * w;
                        wsum += w;
                        if (AUX) {
                            dsum += h.t * w;
                            nx += r.nrm_dep.x * w;
                            ny += r.nrm_dep.y * w;
                            nz += r.nrm_dep.z * w;
                        }
                        T *= 1.0f - h.a;
                        last = first + j;
                        if (TRACE && traced) {
                            if (tcount < trace.cap)
                                trace.lists[tslot * trace.cap + tcount] =
                                    (payloads[base + j] & kTraceRecordMask) | (h.ray ? 1u << 30 : 0u) |
                                    (h.clamped ? 1u << 31 : 0u);
                            ++tcount;
                        }
                    }
                };
                // Two records of each row per round: their slots come as one
                // word, read a round ahead (a row past its end reads old
                // slots, below BATCH, and drops them).
                uint32_t jj = my_list[0];
                for (uint32_t k = 0; __any(T >= kTTerminate && k < mine); k += 2) {
                    const uint32_t j0 = jj & 0xFFu, j1 = jj >> 8;
                    Record r0, r1;
                    load((j0 & (BATCH - 1u)) << 4, r0);
                    load((j1 & (BATCH - 1u)) << 4, r1);
                    jj = my_list[k / 2 + 1];
                    composite(j0, r0, k < mine);
                    composite(j1, r1, k + 1 < mine);
                }
            }
            if (__syncthreads_count(T >= kTTerminate) == 0) break;
        }
        if (inside) {
            const size_t pi = (size_t)cam.pix_base + (size_t)py * cam.width + (size_t)px;
            out.color[pi] = make_float4(cr, cg, cb, wsum);
            out.aux[pi] = make_float4(T, dsum, 0.0f, 0.0f);
            if (AUX) out.normal[pi] = make_float4(nx, ny, nz, 0.0f);
            out.ncontrib[pi] = last;
            if (TRACE && traced) trace.counts[tslot] = tcount;
        }
    }
}

}  // namespace

hipError_t launch_raster_fwd(hipStream_t st, const CamParams* cams_dev, const CamParams* /*cams_host*/,
                             uint32_t n_views, uint32_t total_tiles, const uint32_t* ranges,
                             const uint32_t* payloads, const Record* recs, FwdOut out, bool cull,
                             TileQueue queue, bool aux_outputs, RasterShape shape, uint32_t tile_begin,
                             FwdTrace trace) {
    if (total_tiles == 0) return hipSuccess;
    const uint32_t t = shape.tile, b = shape.fwd_batch;
    // With a queue, positions below the grid size belong to workgroups that
    // should start at once, the longest lists among them: no more workgroups
    // than the CUs hold (`per_cu`). Eight for each CU where six fit leave the
    // last 512 of those lists to the end of the launch: 550 instead of 507 us
    // at 1M surfels in four 1080p views.
    auto go = [&](auto kernel, uint32_t threads, uint32_t waves_per_simd, auto... extra) {
        uint32_t grid = total_tiles;
        if (queue.cursor != nullptr) {
            const uint32_t per_cu = std::max(1u, waves_per_simd * 256u / threads);
            grid = std::min(grid, std::max(queue.grid_blocks, 1u));
            if (queue.cus != 0) grid = std::min(grid, per_cu * queue.cus);
        }
        hipLaunchKernelGGL(kernel, dim3(grid), dim3(threads), 0, st, cams_dev, n_views, ranges, payloads, recs,
                           out, cull, total_tiles, queue, tile_begin, extra...);
    };
    if (trace.lists != nullptr) {
        // The trace variant: depth / normal outputs, 16-px tiles, 256-record batches.
        if (!aux_outputs || t != 16 || b != 256 || trace.counts == nullptr) return hipErrorInvalidValue;
        go(raster_fwd_sub_kernel<true, 16, 256, true>, 256, kSubWaves<true>, trace);
    } else if (aux_outputs) {
        if (t != 16 || b != 256) return hipErrorInvalidValue;  // depth / normal outputs: 16-px tiles
        go(raster_fwd_sub_kernel<true, 16, 256>, 256, kSubWaves<true>, trace);
    } else if (t == 8 && b == 64) {
        go(raster_fwd_sub_kernel<false, 8, 64>, 64, kSubWaves<false>, trace);
    } else if (t == 8 && b == 128) {
        go(raster_fwd_sub_kernel<false, 8, 128>, 64, kSubWaves<false>, trace);
    } else if (t == 16 && b == 128) {
        go(raster_fwd_sub_kernel<false, 16, 128>, 256, kSubWaves<false>, trace);
    } else if (t == 16 && b == 256) {
        go(raster_fwd_sub_kernel<false, 16, 256>, 256, kSubWaves<false>, trace);
    } else if (t == 32 && b == 256) {
        go(raster_fwd_kernel<32, 256>, 1024, 4);
    } else if (t == 32 && b == 512) {
        go(raster_fwd_kernel<32, 512>, 1024, 4);
    } else {
        return hipErrorInvalidValue;
    }
    return hipGetLastError();
}

}  // namespace gs
