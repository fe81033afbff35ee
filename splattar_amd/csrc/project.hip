// Surfel projection with tile counting fused: one thread per
// (view, surfel). Restates crates/gs-kernels/src/shaders/surfel_prep_fwd.wgsl:
// 64-132 and count_tiles of tile_binning.wgsl:30-43, and additionally emits
// the per-surfel ray-splat setup (M, A, B, Nt) so the rasterizer's per-pixel
// intersection is three 2-FMA dot products instead of four triple products.
//
// HBM traffic per (view, surfel): reads 16+8+16+4+12*(d+1)^2 B of parameters,
// writes a 128-B record, a 16-B rect, a 4-B depth key and a 4-B count.
// The record's footprint box is clipped to the pixels of its 16-px tile rect
// (the forward model's coverage). With clip_to_box the emitted rect is the
// set of work tiles (cam.tile_size px) that clipped box reaches (tight
// binning); without it, the 16-px rect itself (work tiles must be 16 px).
// Surfels i >= cam.n_surfels are culled in that view. rects, depth_keys and
// counts may be null (callers that read only the presort and emit_info
// outputs).

#include "gs_internal.h"

namespace gs {

namespace {

__global__ __launch_bounds__(256) void project_kernel(
    const CamParams* __restrict__ cams, uint32_t n_views, uint32_t n, const float4* __restrict__ pos,
    const float2* __restrict__ scales, const float4* __restrict__ quats,
    const float* __restrict__ opac, const float* __restrict__ sh, Record* __restrict__ recs,
    uint4* __restrict__ rects, uint32_t* __restrict__ depth_keys, uint32_t* __restrict__ counts,
    uint32_t* __restrict__ ranges_to_clear, uint32_t num_ranges, uint32_t* __restrict__ presort_keys,
    uint32_t* __restrict__ presort_vals, uint32_t* __restrict__ item_count, bool clip_to_box,
    uint4* __restrict__ emit_info, bool pack_counts) {
    // Views vary fastest over the logical blocks and each XCD takes a
    // contiguous range of them, so the V blocks that read the same 256
    // surfels run on one XCD and the later ones find the parameters in its L2.
    const uint32_t lb = xcd_swizzle(blockIdx.x, gridDim.x);
    const uint32_t view = lb % n_views;
    const uint32_t sblocks = gridDim.x / n_views;
    const uint32_t i = (lb / n_views) * blockDim.x + threadIdx.x;
    // The tile-range table of the following binning stage starts cleared
    // (binning.rs:228); the first view's blocks do it (stream order makes it
    // visible to tile_ranges).
    if (view == 0 && ranges_to_clear != nullptr) {
        for (uint32_t k = i; k < num_ranges; k += sblocks * blockDim.x) ranges_to_clear[k] = 0u;
    }
    if (view == 0 && i == 0 && item_count != nullptr) *item_count = n * n_views;
    // Every thread of the block runs to the store of the records below; items
    // past n have none.
    const bool in_range = i < n;
    const CamParams cam = cams[view];
    const uint32_t g = view * n + i;
    // Per-item binning outputs, written on every path. The presort payload
    // carries the tile count in its low kPackBits bits when pack_counts (for
    // work tiles of 16 or 32 px a rect spans at most 9 x 9 tiles), so the
    // scan reads counts in depth order without a gather.
    // emit_info = (x0 | y0 << 16, x1 | y1 << 16, mask lo, mask hi): the rect
    // in 16-bit tile coordinates and the mask of its tiles the footprint
    // reaches (all ones = every tile).
    auto finish = [&](uint4 rect, uint32_t key, uint32_t count, uint64_t mask) {
        if (rects) rects[g] = rect;
        if (depth_keys) depth_keys[g] = key;
        if (counts) counts[g] = count;
        // Items without entries are left out by the presort's first pass.
        if (presort_keys) presort_keys[g] = count != 0u ? key : kDropKey;
        if (presort_vals) presort_vals[g] = pack_counts ? (g << kPackBits) | count : g;
        if (emit_info)
            emit_info[g] = make_uint4(rect.x | (rect.y << 16), rect.z | (rect.w << 16), (uint32_t)mask,
                                      (uint32_t)(mask >> 32));
    };

    uint4 rect = make_uint4(1u, 1u, 0u, 0u);
    bool live = in_range && i < cam.n_surfels;  // surfels past n_surfels are not part of this view
    CamFrame f;
    float depth = 0.0f;
    if (live) {
        f = cam_frame(cam, pos[i], scales[i], quats[i]);
        depth = -f.cz_;
        // Near cull (surfel_prep_fwd.wgsl:171-176); NaN culls too.
        live = depth >= kNearDepth;
    }
    Record rec;
    uint32_t count = 0u;
    uint64_t mask = ~0ull;
    bool masked = false;  // rect of at most 64 tiles: per-tile footprint test below
    float3 c = make_float3(0.0f, 0.0f, 0.0f), M = c;
    if (live) {
        const RectOut r = tile_rect(cam, f, depth);
        // Ray-splat setup.
        c = make_float3(f.cx_, f.cy_, f.cz_);
        const float3 tu = make_float3(f.tux, f.tuy, f.tuz);
        const float3 tv = make_float3(f.tvx, f.tvy, f.tvz);
        M = cross3(tu, tv);
        const float3 A = cross3(tv, c);
        const float3 B = cross3(c, tu);
        const float Nt = -dot3(M, c);
        rec.m_nt = make_float4(M.x, M.y, M.z, Nt);
        rec.a_px = make_float4(A.x, A.y, A.z, r.px);
        rec.b_py = make_float4(B.x, B.y, B.z, r.py);
        rec.col_op.w = opac[i];
        if (r.on_screen) {
            rect = make_uint4(r.x0, r.y0, r.x1, r.y1);
            record_footprint(rec, cam);
            rec.box = clip_box_to_rect(rec.box, rect);
            // Tight binning keeps only the work tiles the alpha >= 1/255
            // footprint reaches; the dropped entries would contribute nothing.
            if (clip_to_box) rect = box_tiles(rec.box, cam.tile_size, cam.tiles_x, cam.tiles_y);
            if (rect.x <= rect.z && rect.y <= rect.w) {
                count = (rect.z - rect.x + 1u) * (rect.w - rect.y + 1u);
                // Rects of at most 64 tiles get a per-tile footprint test (box,
                // disk, ellipse); larger ones keep every tile.
                masked = clip_to_box && count <= 64u;
            }
        }
    }

    // Per-tile footprint masks, bit t = row-major tile t of the rect: each lane
    // takes the rows of its item's rect, a column interval for each (a rect is
    // a few tiles; the wave takes as many steps as its tallest rect has rows).
    // Dealing (item, tile) pairs over the lanes, with an owner search and a
    // footprint test a pair, took half of the kernel's LDS accesses and a
    // quarter of its instructions. In all 367 -> 274 us for 4M items and 1200 ->
    // 983 us for 20M (where 128 B a record written and the parameters read take
    // 0.15 and 0.6 ms).
    if (masked) {
        const SubTest t = sub_test(rec.box, rec.ell0, rec.ell1, rec.a_px.w, rec.b_py.w);
        const uint32_t w = rect.z - rect.x + 1u;
        mask = 0ull;
        for (uint32_t y = rect.y, shift = 0u; y <= rect.w; ++y, shift += w)
            mask |= tile_row_mask(t, rect.x, w, y, cam.tile_size) << shift;
        count = (uint32_t)__popcll(mask);
    }
    // Binning outputs; a record only for items that reach a tile (no entry
    // ever reads the others).
    bool write_rec = false;
    if (in_range) {
        if (!live) {
            finish(make_uint4(1u, 1u, 0u, 0u), 0u, 0u, ~0ull);
        } else {
            if (count == 0u) {
                rect = make_uint4(1u, 1u, 0u, 0u);
                mask = ~0ull;
            }
            finish(rect, __float_as_uint(depth), count, mask);
            write_rec = count != 0u;
        }
    }
    if (write_rec) {
        // View-dependent colour (surfel_prep_fwd.wgsl:113-147, 183-186).
        const float inv_len = 1.0f / sqrtf(f.xx * f.xx + f.xy * f.xy + f.xz * f.xz);
        float basis[16];
        const int nb = sh_basis((int)cam.sh_degree, f.xx * inv_len, f.xy * inv_len, f.xz * inv_len, basis);
        // 16-B loads of the (48-float, 192-B aligned) coefficient row, only as
        // far as the degree needs; all at once: four at a time (80 registers
        // and six waves a SIMD instead of 103 and four) take 314 instead of
        // 274 us for 4M items.
        const float4* sh4 = reinterpret_cast<const float4*>(sh + (size_t)i * kShFloats);
        float shv[kShFloats];
#pragma unroll
        for (int q = 0; q < kShFloats / 4; ++q) {
            const float4 v = 4 * q < 3 * nb ? sh4[q] : make_float4(0.0f, 0.0f, 0.0f, 0.0f);
            shv[4 * q + 0] = v.x;
            shv[4 * q + 1] = v.y;
            shv[4 * q + 2] = v.z;
            shv[4 * q + 3] = v.w;
        }
        float cr = 0.5f, cg = 0.5f, cb = 0.5f;
#pragma unroll
        for (int k = 0; k < 16; ++k) {
            if (k < nb) {
                cr += basis[k] * shv[3 * k + 0];
                cg += basis[k] * shv[3 * k + 1];
                cb += basis[k] * shv[3 * k + 2];
            }
        }
        // Camera-facing unit normal (surfel_prep_fwd.wgsl:188-194).
        float3 nrm = M;
        const float mm = dot3(M, M);
        if (mm > 0.0f) {
            const float inv = 1.0f / sqrtf(mm);
            nrm = make_float3(M.x * inv, M.y * inv, M.z * inv);
            if (dot3(nrm, c) > 0.0f) nrm = make_float3(-nrm.x, -nrm.y, -nrm.z);
        }
        rec.col_op = make_float4(fmaxf(cr, 0.0f), fmaxf(cg, 0.0f), fmaxf(cb, 0.0f), opac[i]);
        rec.nrm_dep = make_float4(nrm.x, nrm.y, nrm.z, depth);
    }
    // The block's items are consecutive (one view, 256 consecutive surfels):
    // stage the records in LDS, half the block at a time, and store them as one
    // run, lane-consecutive 16-B stores instead of eight 16-B stores at a
    // 128-B stride per lane. Whole 128-B records, the normal also where nothing
    // reads it: a record with a 16-B hole costs a read of its line (4M records
    // 377 us against 310, 20M 1150 against 1020).
    constexpr int kRecRow = 9;  // float4 a row: one spare against LDS bank conflicts
    __shared__ float4 s_stage[128 * kRecRow];
    __shared__ uint32_t s_write[128];
    const uint32_t tid = threadIdx.x, i0 = i - tid;
    const uint32_t nrec = i0 < n ? min(256u, n - i0) : 0u;
#pragma unroll
    for (uint32_t half = 0; half < 2; ++half) {
        if (half == 1) __syncthreads();  // the first half's rows are stored
        if (tid >> 7 == half) {
            s_write[tid & 127u] = write_rec ? 1u : 0u;
            if (write_rec) {
                float4* row = s_stage + (tid & 127u) * kRecRow;
                row[0] = rec.m_nt;
                row[1] = rec.a_px;
                row[2] = rec.b_py;
                row[3] = rec.col_op;
                row[4] = rec.nrm_dep;
                row[5] = rec.box;
                row[6] = rec.ell0;
                row[7] = rec.ell1;
            }
        }
        __syncthreads();
        const uint32_t here = nrec > 128u * half ? min(128u, nrec - 128u * half) : 0u;
        float4* dst = reinterpret_cast<float4*>(recs + (size_t)view * n + i0 + 128u * half);
        for (uint32_t q = tid; q < here * 8u; q += 256u) {
            const uint32_t r = q >> 3, fld = q & 7u;
            if (s_write[r] == 0u) continue;
            const float4 v = s_stage[r * kRecRow + fld];
            typedef float f4v __attribute__((ext_vector_type(4)));
            __builtin_nontemporal_store(f4v{v.x, v.y, v.z, v.w}, reinterpret_cast<f4v*>(dst + q));
        }
    }
}

}  // namespace

hipError_t launch_project(hipStream_t st, const CamParams* cams_dev, uint32_t n_views, uint32_t n,
                          const float4* pos, const float2* scales, const float4* quats,
                          const float* opac, const float* sh, Record* recs, uint4* rects,
                          uint32_t* depth_keys, uint32_t* counts, uint32_t* ranges_to_clear,
                          uint32_t num_ranges, uint32_t* presort_keys, uint32_t* presort_vals,
                          uint32_t* item_count, bool clip_to_box, uint4* emit_info, bool pack_counts) {
    if (n == 0 && num_ranges == 0 && item_count == nullptr) return hipSuccess;
    if (n_views == 0) return hipSuccess;
    const uint32_t blocks = div_up(n > num_ranges ? (n ? n : 1) : num_ranges, 256);
    dim3 grid(blocks * n_views);
    hipLaunchKernelGGL(project_kernel, grid, dim3(256), 0, st, cams_dev, n_views, n, pos, scales, quats, opac,
                       sh, recs, rects, depth_keys, counts, ranges_to_clear, num_ranges, presort_keys,
                       presort_vals, item_count, clip_to_box, emit_info, pack_counts);
    return hipGetLastError();
}

}  // namespace gs
