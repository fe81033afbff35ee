// Tile rasterizer backward: the hand-written adjoint of raster_fwd.
//
// Restates crates/gs-kernels/src/shaders/rasterize_bwd.wgsl:113-312 (the
// oracle's backward.rs:67-173): per pixel, walk the tile list back to front
// from the stored final transmittance and last-contributor index, recover
// T_before = T / (1 - alpha) instead of storing per-fragment state, keep
// suffix sums, and differentiate the compositing and the ray-splat
// intersection. Differences from the reference, all MI355X-driven:
//   * gradients are taken w.r.t. the per-surfel record coefficients (A, B, M,
//     Nt, px, py, depth, colour, opacity, normal); the linear chain to
//     camera-space (c, tu, tv) happens once per surfel in geom_bwd instead of
//     four triple-product gradients per pixel-hit;
//   * a 16x16 work tile is one wave64 with four pixels per lane, one in each
//     8x8 block (raster_bwd_wave_kernel): a record is evaluated only in the
//     blocks its footprint reaches, its terms over the tile are summed in
//     registers, reduced once per (record, tile) and added to the record's
//     gradient with hardware global atomics, FP32 or FP64 (no CAS loops). A 32x32
//     tile is eight waves, each owning an 8-wide, 16-tall column of two
//     blocks (two pixels per lane), whose per-record reductions meet in LDS
//     slots (ds_add_f32) flushed once per batch, as do those of the two waves of
//     the depth / normal variant; an 8x8 tile is one wave with one pixel per
//     lane (raster_bwd_kernel). Records are staged BATCH at a time into
//     order-preserving lists that carry the blocks each reaches;
//   * each wave reduces its lanes' 16 values with a transposed butterfly (17
//     lane exchanges instead of 96, on permlane swaps and DPP rather than LDS
//     permutes);
//   * lists longer than a segment are split over depth: a state pass
//     (raster_state_kernel) leaves each pixel's walk state at the segment
//     boundaries, and the gradient pass takes segments as units.
// AUX = true (16-px tiles, raster_bwd_kernel) adds the depth / normal image
// losses and the in-walk depth distortion loss (backward.rs:126-153).

#include "gs_internal.h"

namespace gs {

namespace {

__device__ __forceinline__ uint32_t view_of_tile(const CamParams* cams, uint32_t n_views, uint32_t t) {
    uint32_t v = 0;
    for (uint32_t k = 1; k < n_views; ++k)
        if (cams[k].tile_base <= t) v = k;
    return v;
}

// Cross-lane exchange without the LDS crossbar: DPP for partners inside a
// 16-lane row, the gfx950 permlane swaps across rows. xlane<OFF>(x) returns x
// of a partner lane whose index differs from this lane's in bit OFF (and
// possibly in lower bits): row_mirror (i <-> 15-i) for 8, row_half_mirror
// (i <-> 7-i) for 4, quad permutations (xor) for 2 and 1.
template <int OFF>
__device__ __forceinline__ float xlane(float x) {
    static_assert(OFF == 8 || OFF == 4 || OFF == 2 || OFF == 1, "row-local exchange only");
    constexpr int ctrl = OFF == 8 ? 0x140 : OFF == 4 ? 0x141 : OFF == 2 ? 0x4E : 0xB1;
    return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(x), ctrl, 0xF, 0xF, false));
}

// The largest x of the wave, as a scalar.
__device__ __forceinline__ uint32_t wave_max(uint32_t x) {
    for (int o = 32; o >= 1; o >>= 1) x = max(x, (uint32_t)__shfl_xor((int)x, o));
    return __builtin_amdgcn_readfirstlane(x);
}

// Sums of values over the 64 lanes of a wave (every lane active) by halving: a
// transposition step at lane bit OFF leaves lanes with the bit clear with
// lo(self) + lo(partner) and lanes with it set with hi(self) + hi(partner), so
// each step halves the values a lane holds; when one is left, the remaining
// bits are summed. For bits 32 and 16 one permlane swap moves the upper half
// of lo and the lower half of hi across. Within a 16-lane row the partner's
// value comes by DPP (mirror, half mirror), and two adds that each write one
// bank half replace two selects and an add. Written out because a swap through
// the builtin copies an operand first: 16 values take 40 instructions instead
// of 55, 6 % of the gradient pass at 1M surfels. s_nop 1: a swap or DPP reads
// a register two waits after it is written.
__device__ __forceinline__ void swap32(float (&a)[8], float (&b)[8]) {
    asm("s_nop 1\n\t"
        "v_permlane32_swap_b32 %0, %8\n\tv_permlane32_swap_b32 %1, %9\n\t"
        "v_permlane32_swap_b32 %2, %10\n\tv_permlane32_swap_b32 %3, %11\n\t"
        "v_permlane32_swap_b32 %4, %12\n\tv_permlane32_swap_b32 %5, %13\n\t"
        "v_permlane32_swap_b32 %6, %14\n\tv_permlane32_swap_b32 %7, %15"
        : "+v"(a[0]), "+v"(a[1]), "+v"(a[2]), "+v"(a[3]), "+v"(a[4]), "+v"(a[5]), "+v"(a[6]), "+v"(a[7]),
          "+v"(b[0]), "+v"(b[1]), "+v"(b[2]), "+v"(b[3]), "+v"(b[4]), "+v"(b[5]), "+v"(b[6]), "+v"(b[7]));
}
__device__ __forceinline__ void swap16(float (&a)[4], float (&b)[4]) {
    asm("s_nop 1\n\t"
        "v_permlane16_swap_b32 %0, %4\n\tv_permlane16_swap_b32 %1, %5\n\t"
        "v_permlane16_swap_b32 %2, %6\n\tv_permlane16_swap_b32 %3, %7"
        : "+v"(a[0]), "+v"(a[1]), "+v"(a[2]), "+v"(a[3]), "+v"(b[0]), "+v"(b[1]), "+v"(b[2]), "+v"(b[3]));
}
// Lane l gets the total of value (l >> 2) & 15.
__device__ __forceinline__ float wave_sums16(const float (&v)[16]) {
    float a[8], b[8], c[4], d[4];
#pragma unroll
    for (int i = 0; i < 8; ++i) {
        a[i] = v[i];
        b[i] = v[8 + i];
    }
    swap32(a, b);
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        c[i] = a[i] + b[i];
        d[i] = a[4 + i] + b[4 + i];
    }
    swap16(c, d);
#pragma unroll
    for (int i = 0; i < 4; ++i) c[i] += d[i];
    float s, t;
    asm("s_nop 1\n\t"
        "v_add_f32_dpp %0, %2, %2 row_mirror row_mask:0xf bank_mask:0x3\n\t"
        "v_add_f32_dpp %1, %3, %3 row_mirror row_mask:0xf bank_mask:0x3\n\t"
        "v_add_f32_dpp %0, %4, %4 row_mirror row_mask:0xf bank_mask:0xc\n\t"
        "v_add_f32_dpp %1, %5, %5 row_mirror row_mask:0xf bank_mask:0xc\n\t"
        "s_nop 1\n\t"
        "v_add_f32_dpp %2, %0, %0 row_half_mirror row_mask:0xf bank_mask:0x5\n\t"
        "v_add_f32_dpp %2, %1, %1 row_half_mirror row_mask:0xf bank_mask:0xa\n\t"
        "s_nop 1\n\t"
        "v_add_f32_dpp %2, %2, %2 quad_perm:[2,3,0,1] row_mask:0xf bank_mask:0xf\n\t"
        "s_nop 1\n\t"
        "v_add_f32_dpp %2, %2, %2 quad_perm:[1,0,3,2] row_mask:0xf bank_mask:0xf"
        : "=&v"(s), "=&v"(t), "+v"(c[0])
        : "v"(c[1]), "v"(c[2]), "v"(c[3]));
    return c[0];
}
// Lane l gets the total of value (l >> 4) & 3.
__device__ __forceinline__ float wave_sums4(const float (&v)[4]) {
    auto swap = [](float lo, float hi, auto f) {
        const auto p = f(__float_as_uint(lo), __float_as_uint(hi));
        return __uint_as_float(p[0]) + __uint_as_float(p[1]);
    };
    auto s32 = [](uint32_t x, uint32_t y) { return __builtin_amdgcn_permlane32_swap(x, y, false, false); };
    auto s16 = [](uint32_t x, uint32_t y) { return __builtin_amdgcn_permlane16_swap(x, y, false, false); };
    float r = swap(swap(v[0], v[2], s32), swap(v[1], v[3], s32), s16);
    r += xlane<8>(r);
    r += xlane<4>(r);
    r += xlane<2>(r);
    return r + xlane<1>(r);
}

// Per-pixel state of the backward walk.
struct PixState {
    float sx, sy, pxc, pyc;
    float dlr, dlg, dlb, dld, dnx, dny, dnz;
    float T, w_total, wt_total;
    float suf_r, suf_g, suf_b, suf_d, suf_nx, suf_ny, suf_nz, suf_w, suf_cw;
    uint32_t last;
};

// Loads a pixel's incoming gradients and forward state; last = 0 when the
// pixel is outside the image or carries no loss gradient (nothing to walk).
template <bool AUX>
__device__ __forceinline__ void load_pixel(PixState& p, const CamParams& cam, int px, int py,
                                           const BwdIn& in, float lambda) {
    pixel_s(cam, px, py, p.sx, p.sy);
    p.pxc = (float)px + 0.5f;
    p.pyc = (float)py + 0.5f;
    p.dlr = p.dlg = p.dlb = p.dld = p.dnx = p.dny = p.dnz = 0.f;
    p.T = 1.0f;
    p.w_total = p.wt_total = 0.f;
    p.suf_r = p.suf_g = p.suf_b = p.suf_d = p.suf_nx = p.suf_ny = p.suf_nz = p.suf_w = p.suf_cw = 0.f;
    p.last = 0;
    const bool inside = px < (int)cam.width && py < (int)cam.height;
    if (!inside) return;
    const size_t pi = (size_t)cam.pix_base + (size_t)py * cam.width + (size_t)px;
    const float4 dl = in.dl_dcolor[pi];
    p.dlr = dl.x;
    p.dlg = dl.y;
    p.dlb = dl.z;
    const float4 aux = in.out_aux[pi];
    p.T = aux.x;
    uint32_t last = in.ncontrib[pi];
    bool has_loss = p.dlr != 0.f || p.dlg != 0.f || p.dlb != 0.f;
    if (AUX) {
        p.dld = dl.w;
        if (in.dl_dnormal) {
            const float4 dn = in.dl_dnormal[pi];
            p.dnx = dn.x;
            p.dny = dn.y;
            p.dnz = dn.z;
        }
        p.w_total = in.out_color[pi].w;
        p.wt_total = aux.y;
        has_loss = has_loss || p.dld != 0.f || p.dnx != 0.f || p.dny != 0.f || p.dnz != 0.f || lambda != 0.f;
    }
    p.last = has_loss ? last : 0u;
}

// The walk state's own arithmetic, shared by the gradient pass (add_hit) and
// the state pass (step_state), which has to reach the same bits: every
// multiply-add is explicit, nothing is left to contraction.
// Derivative of the distortion with respect to a hit's weight and, in
// dt_dist, its depth (backward.rs:126-153); lambda != 0.
__device__ __forceinline__ float distortion_coef(const PixState& p, float w, float t_hit, float lambda,
                                                 float& dt_dist) {
#pragma clang fp contract(off)
    const float a_pre = p.w_total - p.suf_w - w;
    const float b_pre = fmaf(-w, t_hit, p.wt_total - p.suf_d);
    dt_dist = lambda * 2.0f * w * (a_pre - p.suf_w);
    return lambda * fmaf(2.0f, fmaf(t_hit, a_pre, -b_pre), 2.0f * fmaf(-t_hit, p.suf_w, p.suf_d));
}
__device__ __forceinline__ void step_aux_sums(PixState& p, const Record& r, float w, float t_hit, float coef) {
#pragma clang fp contract(off)
    p.suf_d += t_hit * w;
    p.suf_nx = fmaf(r.nrm_dep.x, w, p.suf_nx);
    p.suf_ny = fmaf(r.nrm_dep.y, w, p.suf_ny);
    p.suf_nz = fmaf(r.nrm_dep.z, w, p.suf_nz);
    p.suf_w += w;
    p.suf_cw = fmaf(coef, w, p.suf_cw);
}
// One record's step of the walk without its gradient terms: what add_hit
// does to T and the suffix sums.
template <bool AUX>
__device__ __forceinline__ void step_state(PixState& p, const Record& r, const HitEval& h, bool act, float lambda) {
    const float alpha = act ? h.a : 0.0f;
    const float t_before = p.T * rcp_refined(1.0f - alpha);
    const float w = t_before * alpha;
    p.suf_r = fmaf(r.col_op.x, w, p.suf_r);
    p.suf_g = fmaf(r.col_op.y, w, p.suf_g);
    p.suf_b = fmaf(r.col_op.z, w, p.suf_b);
    if (AUX) {
        float dt_dist = 0.0f, coef = 0.0f;
        if (lambda != 0.0f) coef = distortion_coef(p, w, h.t, lambda, dt_dist);
        step_aux_sums(p, r, w, h.t, coef);
    }
    p.T = t_before;
}

// Walk states at segment boundaries (BwdSegments::state): pixel k of the
// tile (8x8 block k >> 6, row-major within it) of segment `at`.
template <bool AUX>
__device__ __forceinline__ void store_state(const BwdSegments& sg, uint32_t at, uint32_t k, const PixState& p) {
    const size_t j = (size_t)at * kSegmentPixels + k;
    sg.state[j] = make_float4(p.T, p.suf_r, p.suf_g, p.suf_b);
    if (AUX) {
        sg.state_aux[j] = make_float4(p.suf_d, p.suf_nx, p.suf_ny, p.suf_nz);
        sg.state_aux[(size_t)sg.pool * kSegmentPixels + j] = make_float4(p.suf_w, p.suf_cw, 0.0f, 0.0f);
    }
}
template <bool AUX>
__device__ __forceinline__ void load_state(const BwdSegments& sg, uint32_t at, uint32_t k, PixState& p) {
    const size_t j = (size_t)at * kSegmentPixels + k;
    const float4 a = sg.state[j];
    p.T = a.x;
    p.suf_r = a.y;
    p.suf_g = a.z;
    p.suf_b = a.w;
    if (AUX) {
        const float4 b = sg.state_aux[j], c = sg.state_aux[(size_t)sg.pool * kSegmentPixels + j];
        p.suf_d = b.x;
        p.suf_nx = b.y;
        p.suf_ny = b.z;
        p.suf_nz = b.w;
        p.suf_w = c.x;
        p.suf_cw = c.y;
    }
}

// One unit of the gradient pass: a tile, and either its whole list (seg ==
// kWholeTile) or one segment of it.
constexpr uint32_t kWholeTile = ~0u;
struct BwdItem {
    uint32_t tile, seg, at;  // at: the segment's slot (its boundary state)
    bool last;               // the tile's last segment: starts from the forward's end
};
// Position pos of the pass: the segments first (the largest units), then the
// tiles in the queue's order, of which the split ones are done already.
// False: nothing to do at this position.
__device__ __forceinline__ bool bwd_item(const BwdSegments& sg, uint32_t nseg, uint32_t pos, const TileQueue& queue,
                                         uint32_t tile_begin, BwdItem& it) {
    it.seg = kWholeTile;
    it.at = 0;
    it.last = true;
    if (pos < nseg) {
        const uint2 e = sg.table[pos];
        it.tile = e.x;
        it.seg = e.y & ~kSegmentLast;
        it.last = (e.y & kSegmentLast) != 0u;
        it.at = pos;
        return e.x != ~0u;
    }
    it.tile = queue.order != nullptr ? queue.order[pos - nseg] : tile_begin + (pos - nseg);
    return sg.state == nullptr || sg.split[it.tile] == 0u;
}

template <bool AUX, bool ACC>
__device__ __forceinline__ void put(float& dst, float v) {
    if constexpr (ACC) dst += v;
    else dst = v;
}

// Writes (ACC = false) or adds (ACC = true) one pixel-record hit's gradient
// terms into g / g2 and steps the pixel's walk, given the hit evaluation h and
// whether this lane contributes (act). Branch-free: a lane that does not
// contribute gets w = 0 and 1/(1-alpha) = 1 exactly, so its running sums and
// T are unchanged, and its gradient terms are selected to 0 (no NaN from
// 0 * inf); a wave with no contributing lane need not call it at all.
template <bool AUX, bool ACC>
__device__ __forceinline__ void add_hit(PixState& p, const Record& r, const HitEval& h, bool act,
                                        float lambda, float (&g)[16], float (&g2)[4]) {
    const float alpha = act ? h.a : 0.0f;
    const float inv_one_m = rcp_refined(1.0f - alpha);
    const float t_before = p.T * inv_one_m;
    const float w = t_before * alpha;
    const float t_hit = h.t;
    put<AUX, ACC>(g[kGCol + 0], p.dlr * w);
    put<AUX, ACC>(g[kGCol + 1], p.dlg * w);
    put<AUX, ACC>(g[kGCol + 2], p.dlb * w);
    float dl_dt = 0.0f;
    float dl_dalpha = (p.dlr * r.col_op.x + p.dlg * r.col_op.y + p.dlb * r.col_op.z) * t_before -
                      (p.dlr * p.suf_r + p.dlg * p.suf_g + p.dlb * p.suf_b) * inv_one_m;
    p.suf_r = fmaf(r.col_op.x, w, p.suf_r);
    p.suf_g = fmaf(r.col_op.y, w, p.suf_g);
    p.suf_b = fmaf(r.col_op.z, w, p.suf_b);
    if (AUX) {
        float dt_dist = 0.0f, coef = 0.0f;
        if (lambda != 0.0f) coef = distortion_coef(p, w, t_hit, lambda, dt_dist);
        put<AUX, ACC>(g2[kGNrm - 16 + 0], p.dnx * w);
        put<AUX, ACC>(g2[kGNrm - 16 + 1], p.dny * w);
        put<AUX, ACC>(g2[kGNrm - 16 + 2], p.dnz * w);
        dl_dt = p.dld * w + dt_dist;
        dl_dalpha += p.dld * (t_hit * t_before - p.suf_d * inv_one_m) +
                     (p.dnx * r.nrm_dep.x + p.dny * r.nrm_dep.y + p.dnz * r.nrm_dep.z) * t_before -
                     (p.dnx * p.suf_nx + p.dny * p.suf_ny + p.dnz * p.suf_nz) * inv_one_m +
                     coef * t_before - p.suf_cw * inv_one_m;
        step_aux_sums(p, r, w, t_hit, coef);
    }
    p.T = t_before;
    // Geometry terms exist only for contributing, unclamped hits, and the
    // plane terms only on the ray branch: the masks are applied once, to ghat
    // and to 1/D, so the terms derived from them are exact zeros (possibly
    // -0, which no sum tells apart) where the terms are absent. dl_dalpha,
    // u and v are finite (|1/D| <= 1e12 and finite record coefficients), so
    // no inf * 0 arises.
    const bool geo = act && !h.clamped;
    const float ghat_g = geo ? h.ghat : 0.0f;
    const float inv_r = h.ray ? h.inv_d : 0.0f;
    put<AUX, ACC>(g[kGOp], dl_dalpha * ghat_g);
    const float gd = ghat_g * (dl_dalpha * r.col_op.w);  // ghat dL/dghat
    const float dl_du = -h.u * gd;
    const float dl_dv = -h.v * gd;
    const float dnu = dl_du * inv_r;
    const float dnv = dl_dv * inv_r;
    // Colour-only (AUX = false): dl_dt = 0, and the record's depth is not
    // staged, so t_hit must not enter (it may hold anything).
    const float dD_num = AUX ? h.u * dl_du + h.v * dl_dv + t_hit * dl_dt : h.u * dl_du + h.v * dl_dv;
    const float dD = -dD_num * inv_r;
    put<AUX, ACC>(g[kGA + 0], dnu * p.sx);
    put<AUX, ACC>(g[kGA + 1], dnu * p.sy);
    put<AUX, ACC>(g[kGA + 2], dnu);
    put<AUX, ACC>(g[kGB + 0], dnv * p.sx);
    put<AUX, ACC>(g[kGB + 1], dnv * p.sy);
    put<AUX, ACC>(g[kGB + 2], dnv);
    put<AUX, ACC>(g[kGM + 0], dD * p.sx);
    put<AUX, ACC>(g[kGM + 1], dD * p.sy);
    put<AUX, ACC>(g[kGM + 2], dD);
    const float gs = h.ray ? 0.0f : 2.0f * gd;
    put<AUX, ACC>(g[kGPx], gs * (p.pxc - r.a_px.w));
    put<AUX, ACC>(g[kGPy], gs * (p.pyc - r.b_py.w));
    if (AUX) {
        put<AUX, ACC>(g[kGNt], (geo && h.ray) ? dl_dt * h.inv_d : 0.0f);
        put<AUX, ACC>(g2[kGDep - 16], (geo && !h.ray) ? dl_dt : 0.0f);
    }
}

// Waves per SIMD: with depth and normals three (168 registers), where the
// compiler's 174 leave two: a backward pass of 1M surfels at 1080p 1845 -> 1604
// us, 300k at 720p 877 -> 744, 20k at 321 x 243 160 -> 155; with no more
// workgroups than then fit (launch_raster_bwd) 1490, 739 and 153. A copy of the
// slots per wave instead of LDS adds takes 10 KB more, so five workgroups a CU
// instead of six: 1607, 791 and 155.
template <bool AUX, int TW, int BATCH, typename Slot>
__global__ __launch_bounds__(TW == 8 ? 64 : TW * TW / 2)
__attribute__((amdgpu_waves_per_eu(AUX ? 3 : 1))) void raster_bwd_kernel(
    const CamParams* __restrict__ cams, uint32_t n_views, const uint32_t* __restrict__ ranges,
    const uint32_t* __restrict__ payloads, const Record* __restrict__ recs, BwdIn in,
    Slot* __restrict__ grad_coef, bool cull, uint32_t total_tiles, TileQueue queue, uint32_t tile_begin,
    BwdSegments sg) {
    constexpr int NS = grad_stride(AUX);     // slots per record (LDS and grad_coef)
    constexpr bool TWO = TW >= 16;           // two pixels per lane (an 8x16 column per wave)
    constexpr int NC = TW / 8;               // 8x8 blocks per tile row
    constexpr int NW = TWO ? TW * TW / 128 : 1;  // waves
    constexpr int NT = NW * 64;
    constexpr int SW = BATCH / 64;           // staging waves per batch
    constexpr int SPT = (BATCH + NT - 1) / NT;
    constexpr int MB = 10;                   // list entry: slot | top << MB | bottom << (MB + 1)
    static_assert(BATCH % 64 == 0 && BATCH <= (1 << MB), "batch of whole waves");
    __shared__ float4 s_m[BATCH], s_a[BATCH], s_b[BATCH], s_c[BATCH], s_n[AUX ? BATCH : 1];
    __shared__ uint32_t s_pay[BATCH];        // the batch's surfel ids, for the flush
    __shared__ uint16_t s_list[NW][BATCH + 1];  // read one entry ahead
    __shared__ uint32_t s_wlast[NW][2];        // last contributors of each wave's blocks
    __shared__ uint32_t s_qcnt[SW][NW];      // [staging wave][list wave]
    __shared__ float s_grad[BATCH * NS];
    __shared__ uint32_t s_view, s_maxlast, s_next;

    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const uint64_t lt_mask = (lane == 0) ? 0ull : (~0ull >> (64 - lane));
    // Wave w owns block column c = w % NC, rows 16 (w / NC) .. + 15: blocks
    // top = (c, 2 (w / NC)) and bottom = (c, 2 (w / NC) + 1).
    const int col = wave % NC, hrow = wave / NC;
    const uint32_t nseg = sg.state != nullptr ? min(sg.ctl[0], sg.pool) : 0u;
    const uint32_t items = total_tiles + nseg;
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
            pos = items;
        }
        if (pos >= items) break;
        BwdItem it;
        if (!bwd_item(sg, nseg, pos, queue, tile_begin, it)) continue;
        const uint32_t gtile = it.tile;
        const uint32_t start = ranges[2 * (size_t)gtile], end = ranges[2 * (size_t)gtile + 1];
        if (end <= start) continue;
        if (tid == 0) {
            s_view = view_of_tile(cams, n_views, gtile);
            s_maxlast = 0u;
        }
        __syncthreads();
        const CamParams& cam = cams[s_view];
        const uint32_t local = gtile - cam.tile_base;
        const uint32_t tx = local % cam.tiles_x, ty = local / cam.tiles_x;
        const uint32_t x0 = tx * TW, y0 = ty * TW;
        const float lambda = AUX ? cam.lambda_dist : 0.0f;
        const int px = (int)x0 + col * 8 + (lane & 7);
        const int py = (int)y0 + hrow * 16 + (lane >> 3);
        PixState pa, pb;
        load_pixel<AUX>(pa, cam, px, py, in, lambda);
        if constexpr (TWO) load_pixel<AUX>(pb, cam, px, py + 8, in, lambda);
        else pb.last = 0u;
        const uint32_t last_a = wave_max(pa.last), last_b = wave_max(pb.last);
        if (lane == 0) {
            s_wlast[wave][0] = last_a;
            s_wlast[wave][1] = last_b;
            atomicMax(&s_maxlast, max(last_a, last_b));
        }
        __syncthreads();
        const uint32_t maxlast = s_maxlast;
        if (maxlast == 0) continue;
        // The list positions [k0, k1) of this item.
        uint32_t k0 = 0, k1 = maxlast;
        if (it.seg != kWholeTile) {
            k0 = it.seg * sg.ctl[1];
            if (!it.last) {
                k1 = k0 + sg.ctl[1];
                if constexpr (TW == 16) {
                    const uint32_t k = (uint32_t)(col + 2 * (2 * hrow)) * 64u + (uint32_t)lane;
                    load_state<AUX>(sg, it.at, k, pa);
                    load_state<AUX>(sg, it.at, k + 128u, pb);
                }
            }
        }

        const int nbatch = (int)((k1 - k0 + BATCH - 1) / BATCH);
        for (int b = nbatch - 1; b >= 0; --b) {
            const uint32_t first = k0 + (uint32_t)b * BATCH;
            const uint32_t base = start + first;
            const uint32_t cnt = min((uint32_t)BATCH, k1 - first);
            uint32_t memb[SPT][NW], qpos[SPT][NW];
#pragma unroll
            for (int m = 0; m < SPT; ++m) {
                const int slot = tid + m * NT;
                if (slot >= BATCH) continue;  // whole waves (NT, BATCH multiples of 64)
                uint32_t qmask = 0;
                if ((uint32_t)slot < cnt) {
                    const uint32_t pay = payloads[base + slot];
                    Record r = recs[pay];
                    s_pay[slot] = pay;
                    s_m[slot] = r.m_nt;
                    s_a[slot] = r.a_px;
                    s_b[slot] = r.b_py;
                    s_c[slot] = r.col_op;
                    if (AUX) s_n[slot] = r.nrm_dep;
                    qmask = cull ? block_mask<TW>(r, x0, y0) : ~0u;
                }
                // Order-preserving per-wave lists: wave w takes the records
                // that reach its top or bottom block.
                const int sw = slot >> 6;
#pragma unroll
                for (int w = 0; w < NW; ++w) {
                    const int bt = TWO ? (2 * (w / NC)) * NC + w % NC : 0;
                    // A block is walked only from its last contributor on.
                    const uint32_t rel = first + (uint32_t)slot;
                    const uint32_t top = rel < s_wlast[w][0] ? (qmask >> bt) & 1u : 0u;
                    const uint32_t bot = TWO && rel < s_wlast[w][1] ? (qmask >> (bt + NC)) & 1u : 0u;
                    memb[m][w] = top | (bot << 1);
                    const uint64_t bal = __ballot(memb[m][w] != 0u);
                    qpos[m][w] = (uint32_t)__popcll(bal & lt_mask);
                    if (lane == 0) s_qcnt[sw][w] = (uint32_t)__popcll(bal);
                }
            }
            for (int k = tid; k < (int)cnt * NS; k += NT) s_grad[k] = 0.0f;
            __syncthreads();
#pragma unroll
            for (int m = 0; m < SPT; ++m) {
                const int slot = tid + m * NT;
                if (slot >= BATCH) continue;
                const int sw = slot >> 6;
#pragma unroll
                for (int w = 0; w < NW; ++w) {
                    if (memb[m][w] != 0u) {
                        uint32_t off = 0;
                        for (int v = 0; v < sw; ++v) off += s_qcnt[v][w];
                        s_list[w][1 + off + qpos[m][w]] = (uint16_t)(slot | (memb[m][w] << MB));
                    }
                }
            }
            int my_count = 0;
#pragma unroll
            for (int v = 0; v < SW; ++v) my_count += (int)s_qcnt[v][wave];
            __syncthreads();

            uint32_t next = s_list[wave][my_count];
            for (int kk = my_count; kk > 0; --kk) {
                // The entry is the same for every lane: make it scalar, so the
                // block branches below are uniform.
                const uint32_t e = __builtin_amdgcn_readfirstlane(next);
                next = s_list[wave][kk - 1];
                const uint32_t j = e & ((1u << MB) - 1u);
                const bool need_a = (e >> MB) & 1u, need_b = TWO && ((e >> (MB + 1)) & 1u);
                const uint32_t rel = first + j;
                Record r;
                r.m_nt = s_m[j];
                r.a_px = s_a[j];
                r.b_py = s_b[j];
                r.col_op = s_c[j];
                r.nrm_dep = AUX ? s_n[AUX ? j : 0] : make_float4(0.0f, 0.0f, 0.0f, 0.0f);
                // Evaluate first; the gradient terms and the reduction run only
                // for blocks with a contributing lane (for the others the walk
                // state would not change).
                HitEval ha, hb;
                bool act_a = false, act_b = false;
                if (need_a) {
                    ha = eval_hit(r, pa.sx, pa.sy, pa.pxc, pa.pyc);
                    act_a = rel < pa.last && ha.hit;
                }
                if (need_b) {
                    hb = eval_hit(r, pb.sx, pb.sy, pb.pxc, pb.pyc);
                    act_b = rel < pb.last && hb.hit;
                }
                const bool go_a = need_a && __any(act_a);
                const bool go_b = need_b && __any(act_b);
                if (!go_a && !go_b) continue;
                float g[16];
                float g2[4];
#pragma unroll
                for (int k = 0; k < 16; ++k) asm volatile("" : "=v"(g[k]));  // defined here: else copied before the sums
                g[kGNt] = 0.0f;  // written only by the AUX terms
#pragma unroll
                for (int k = 0; k < 4; ++k) g2[k] = 0.0f;
                if (go_a && go_b) {
                    add_hit<AUX, false>(pa, r, ha, act_a, lambda, g, g2);
                    add_hit<AUX, true>(pb, r, hb, act_b, lambda, g, g2);
                } else if (go_a) {
                    add_hit<AUX, false>(pa, r, ha, act_a, lambda, g, g2);
                } else {
                    add_hit<AUX, false>(pb, r, hb, act_b, lambda, g, g2);
                }
                const float red = wave_sums16(g);
                if ((lane & 3) == 0) {
                    // One wave meets a record once per batch: no other adds.
                    float* const dst = &s_grad[j * NS + (lane >> 2)];
                    if constexpr (NW == 1) *dst = red;
                    else if (red != 0.0f) atomicAdd(dst, red);
                }
                if (AUX) {
                    const float red2 = wave_sums4(g2);
                    if ((lane & 15) == 0 && red2 != 0.0f) atomicAdd(&s_grad[j * NS + 16 + (lane >> 4)], red2);
                }
            }
            __syncthreads();
            for (int k = tid; k < (int)cnt * NS; k += NT) {
                const float v = s_grad[k];
                if (v != 0.0f) {
                    const int e = k / NS, slot = k - e * NS;
                    // A colour channel clamped at 0 in the forward passes no
                    // gradient to SH (surfel_prep_bwd.wgsl's clamp mask; the
                    // record stores such a channel as exactly 0).
                    if (slot >= kGCol && slot < kGCol + 3) {
                        const float4 c = s_c[e];
                        const float cc = slot == kGCol ? c.x : (slot == kGCol + 1 ? c.y : c.z);
                        if (cc == 0.0f) continue;
                    }
                    atomicAdd(&grad_coef[(size_t)s_pay[e] * NS + slot], (Slot)v);
                }
            }
            __syncthreads();
        }
    }
}

// Colour-only backward over 16-px work tiles with one wave per tile: lane l
// owns pixel (l & 7, l >> 3) of each of the tile's four 8x8 blocks, so a
// record's terms over the whole tile are summed in registers and reduced
// once per (record, tile) instead of once per half tile, and the reduced
// values go straight to the global FP32 atomics (no LDS accumulation slots:
// one wave is the only contributor of its tile). The records a batch stages
// form one order-preserving list carrying each record's 4-bit block mask.
template <int BATCH, typename Slot>
__global__ __launch_bounds__(64) __attribute__((amdgpu_waves_per_eu(4))) void raster_bwd_wave_kernel(
    const CamParams* __restrict__ cams, uint32_t n_views, const uint32_t* __restrict__ ranges,
    const uint32_t* __restrict__ payloads, const Record* __restrict__ recs, BwdIn in,
    Slot* __restrict__ grad_coef, bool cull, uint32_t total_tiles, TileQueue queue, uint32_t tile_begin,
    BwdSegments sg) {
    constexpr int NS = grad_stride(false);
    constexpr int SPT = BATCH / 64;          // staging rounds per batch
    // List entry: slot | block mask << 8 | channels at 0 (bits 12, 16, 20).
    static_assert(BATCH % 64 == 0 && BATCH <= 256, "batch of whole waves");
    __shared__ float4 s_m[BATCH], s_a[BATCH], s_b[BATCH], s_c[BATCH];
    __shared__ uint32_t s_pay[BATCH];
    __shared__ uint32_t s_list[BATCH + 1];  // read one entry ahead

    constexpr uint64_t kWriters = 0x1111111111111111ull;  // lane 4 k holds total k
    const int lane = threadIdx.x;
    const uint64_t lt_mask = (lane == 0) ? 0ull : (~0ull >> (64 - lane));
    const uint32_t nseg = sg.state != nullptr ? min(sg.ctl[0], sg.pool) : 0u;
    const uint32_t items = total_tiles + nseg;
    for (uint32_t iter = 0;; ++iter) {
        uint32_t pos;
        if (iter == 0) {
            pos = queue.cursor != nullptr ? blockIdx.x : xcd_swizzle(blockIdx.x, gridDim.x);
        } else if (queue.cursor != nullptr) {
            pos = __builtin_amdgcn_readfirstlane(lane == 0 ? claim_position(queue) : 0u);
        } else {
            pos = items;
        }
        if (pos >= items) break;
        BwdItem it;
        if (!bwd_item(sg, nseg, pos, queue, tile_begin, it)) continue;
        const uint32_t gtile = it.tile;
        const uint32_t start = ranges[2 * (size_t)gtile], end = ranges[2 * (size_t)gtile + 1];
        if (end <= start) continue;
        const uint32_t v = view_of_tile(cams, n_views, gtile);
        const CamParams& cam = cams[v];
        const uint32_t local = gtile - cam.tile_base;
        const uint32_t tx = local % cam.tiles_x, ty = local / cam.tiles_x;
        const uint32_t x0 = tx * 16, y0 = ty * 16;
        PixState p[4];
        uint32_t block_last[4], maxlast = 0;
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            load_pixel<false>(p[q], cam, (int)x0 + 8 * (q & 1) + (lane & 7), (int)y0 + 8 * (q >> 1) + (lane >> 3),
                              in, 0.0f);
            block_last[q] = wave_max(p[q].last);
            maxlast = max(maxlast, block_last[q]);
        }
        if (maxlast == 0) continue;
        // The list positions [k0, k1) of this item.
        uint32_t k0 = 0, k1 = maxlast;
        if (it.seg != kWholeTile) {
            k0 = it.seg * sg.ctl[1];
            if (!it.last) {
                k1 = k0 + sg.ctl[1];
#pragma unroll
                for (int q = 0; q < 4; ++q) load_state<false>(sg, it.at, (uint32_t)(q * 64 + lane), p[q]);
            }
        }

        const int nbatch = (int)((k1 - k0 + BATCH - 1) / BATCH);
        for (int b = nbatch - 1; b >= 0; --b) {
            const uint32_t first_k = k0 + (uint32_t)b * BATCH;
            const uint32_t base = start + first_k;
            const uint32_t cnt = min((uint32_t)BATCH, k1 - first_k);
            __syncthreads();  // the previous batch's walk has read its LDS
            uint32_t count = 0;
#pragma unroll
            for (int m = 0; m < SPT; ++m) {
                const int slot = lane + m * 64;
                uint32_t qmask = 0, dark = 0;
                if ((uint32_t)slot < cnt) {
                    const uint32_t pay = payloads[base + slot];
                    Record r = recs[pay];
                    s_pay[slot] = pay;
                    s_m[slot] = r.m_nt;
                    s_a[slot] = r.a_px;
                    s_b[slot] = r.b_py;
                    s_c[slot] = r.col_op;
                    qmask = cull ? block_mask<16>(r, x0, y0) : 0xFu;
                    // A block is walked only from its last contributor on.
#pragma unroll
                    for (int q = 0; q < 4; ++q)
                        if (first_k + (uint32_t)slot >= block_last[q]) qmask &= ~(1u << q);
                    // A colour channel clamped at 0 in the forward passes no
                    // gradient to SH (the record stores it as exactly 0).
                    dark = (r.col_op.x == 0.0f ? 1u : 0u) | (r.col_op.y == 0.0f ? 0x10u : 0u) |
                           (r.col_op.z == 0.0f ? 0x100u : 0u);
                }
                const uint64_t bal = __ballot(qmask != 0u);
                if (qmask != 0u)
                    s_list[1 + count + (uint32_t)__popcll(bal & lt_mask)] = (uint32_t)slot | (qmask << 8) | (dark << 12);
                count += (uint32_t)__popcll(bal);
            }
            __syncthreads();

            uint32_t next = s_list[count];
            for (uint32_t kk = count; kk > 0; --kk) {
                const uint32_t e = __builtin_amdgcn_readfirstlane(next);
                next = s_list[kk - 1];
                const uint32_t j = e & 0xFFu;
                const uint32_t rel = first_k + j;
                Record r;
                r.m_nt = s_m[j];
                r.a_px = s_a[j];
                r.b_py = s_b[j];
                r.col_op = s_c[j];
                r.nrm_dep = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
                float g[16];
                float g2[4];
#pragma unroll
                for (int k = 0; k < 16; ++k) asm volatile("" : "=v"(g[k]));  // defined here: else copied before the sums
                g[kGNt] = 0.0f;
                uint32_t blocks = 0;
#pragma unroll
                for (int q = 0; q < 4; ++q) {
                    if (((e >> (8 + q)) & 1u) == 0u) continue;
                    const HitEval h = eval_hit(r, p[q].sx, p[q].sy, p[q].pxc, p[q].pyc);
                    const bool act = rel < p[q].last && h.hit;
                    if (!__any(act)) continue;
                    if (blocks == 0u) add_hit<false, false>(p[q], r, h, act, 0.0f, g, g2);
                    else add_hit<false, true>(p[q], r, h, act, 0.0f, g, g2);
                    blocks = 1u;
                }
                if (blocks == 0u) continue;
                const float red = wave_sums16(g);
                const uint64_t writers = kWriters & ~((uint64_t)(e >> 12) << (4 * kGCol));
                Slot* const dst = grad_coef + (size_t)(uint32_t)__builtin_amdgcn_readfirstlane(s_pay[j]) * NS;
                if (__builtin_amdgcn_inverse_ballot_w64(writers) && red != 0.0f) atomicAdd(dst + (lane >> 2), (Slot)red);
            }
        }
    }
}

// Clears the gradient accumulator and the split flags, resets the cursors and
// the segment counter and sets the segment length: one launch per pass.
__global__ __launch_bounds__(256) void bwd_prepare_kernel(float4* __restrict__ grad_coef, size_t vecs,
                                                          uint32_t* __restrict__ cursor, BwdSegments sg,
                                                          uint32_t split_tiles,
                                                          const uint32_t* __restrict__ entries,
                                                          uint32_t min_len) {
    const size_t t = (size_t)blockIdx.x * 256 + threadIdx.x, step = (size_t)gridDim.x * 256;
    if (t == 0) {
        const uint32_t e = *entries;
        sg.ctl[0] = 0u;
        sg.ctl[1] = max(min_len, (e / kSegmentTarget + 31u) / 32u * 32u);
    }
    if (cursor != nullptr && t < kTileQueues) cursor[t * kCursorStride] = 0u;
    for (size_t k = t; k < split_tiles; k += step) sg.split[k] = 0u;
    for (size_t k = t; k < vecs; k += step) grad_coef[k] = make_float4(0.f, 0.f, 0.f, 0.f);
}

// State pass of the lists longer than a segment (16-px tiles; ctl[1] records
// per segment): claims the tile's segments, walks the records past the first
// segment back to front and stores every pixel's walk state at the segment
// boundaries. The arithmetic per (pixel, record) is the gradient pass's
// (step_state), so each segment continues with the bits the whole walk would
// have. A workgroup is four waves, one per 8x8 block; nothing is summed over
// pixels here, so each 16-lane row walks its own list of the records that
// reach its 4x4 sub-block: a list is about a third of the tile's, and a
// record's step has 45 instructions against ~230 with gradients and their
// reduction, which is what shortens the critical path. 250k surfels in two 1283
// x 717 views: 100 us for the state pass and 375 for the gradient pass, where a
// gradient pass over whole lists takes 679 us (its longest list); 200k surfels
// in six 640 x 360 views: 219 + 609 against 1373 us. Where no list is longer
// than a segment the pass is 10 us.
// Batches of 256 records that do not stop at segment boundaries, staged one
// record a thread: 281 -> 220 us for the six views, 105 -> 71 us with aux (20k
// surfels at 321 x 243), against batches of a segment (at most 128, two threads
// a record).
// Waves per SIMD: 220 us for the six views above at five, 235 at four, 295 at
// six (19 spilled registers); with aux 71 us at four, 84 at five.
template <bool AUX>
constexpr uint32_t kStateWaves = AUX ? 4 : 5;

template <bool AUX>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(kStateWaves<AUX>))) void raster_state_kernel(
    const CamParams* __restrict__ cams, uint32_t n_views, const uint32_t* __restrict__ ranges,
    const uint32_t* __restrict__ payloads, const Record* __restrict__ recs, BwdIn in, bool cull,
    uint32_t total_tiles, TileQueue queue, BwdSegments sg) {
    constexpr int BATCH = 256;               // records staged at a time, one a thread
    __shared__ float4 s_rec[4][BATCH];       // M Nt | A px | B py | colour opacity
    __shared__ float4 s_n[AUX ? BATCH : 1];
    __shared__ uint16_t s_mask[BATCH];       // bit 4 r + c: sub-block (c, r)
    __shared__ uint16_t s_list[16][BATCH / 2 + 1];  // slots, two a word, last record first; read one word ahead
    __shared__ uint32_t s_last[4], s_base;
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    // Row g of wave w: sub-block (2 (w & 1) + (g & 1), 2 (w >> 1) + (g >> 1)),
    // lane p its pixel (p & 3, p >> 2).
    const int g = lane >> 4, p = lane & 15;
    const int sc = 2 * (wave & 1) + (g & 1), sr = 2 * (wave >> 1) + (g >> 1);
    const uint64_t gt_mask = (lane == 63) ? 0ull : (~0ull << (lane + 1));
    const uint16_t* const my_list = s_list[sr * 4 + sc];
    // The pixel's index within the stored state: block, then row-major.
    const uint32_t pixel = (uint32_t)(wave * 64 + ((4 * (g >> 1) + (p >> 2)) * 8 + 4 * (g & 1) + (p & 3)));
    const uint32_t seg_len = sg.ctl[1];
    for (uint32_t pos = blockIdx.x; pos < total_tiles; pos += gridDim.x) {
        const uint32_t gtile = queue.order[pos];
        const uint32_t start = ranges[2 * (size_t)gtile], end = ranges[2 * (size_t)gtile + 1];
        // Longest lists first (keys saturate at 0xFFFF): no longer one follows.
        if (end - start <= min(seg_len, 0xFFFFu)) break;
        const CamParams& cam = cams[view_of_tile(cams, n_views, gtile)];
        const uint32_t local = gtile - cam.tile_base;
        const uint32_t x0 = (local % cam.tiles_x) * 16, y0 = (local / cam.tiles_x) * 16;
        const float lambda = AUX ? cam.lambda_dist : 0.0f;
        PixState ps;
        load_pixel<AUX>(ps, cam, (int)x0 + 4 * sc + (p & 3), (int)y0 + 4 * sr + (p >> 2), in, lambda);
        uint32_t row_last = ps.last;
        for (int o = 8; o >= 1; o >>= 1) row_last = max(row_last, (uint32_t)__shfl_xor((int)row_last, o));
        uint32_t rows_last[4], wave_last = 0;  // of the wave's rows
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            rows_last[q] = (uint32_t)__builtin_amdgcn_readlane((int)row_last, 16 * q);
            wave_last = max(wave_last, rows_last[q]);
        }
        if (lane == 0) s_last[wave] = wave_last;
        __syncthreads();
        const uint32_t maxlast =
            __builtin_amdgcn_readfirstlane(max(max(s_last[0], s_last[1]), max(s_last[2], s_last[3])));
        const uint32_t nseg = (maxlast + seg_len - 1) / seg_len;
        if (nseg < 2) {
            __syncthreads();  // s_last is rewritten by the next tile
            continue;
        }
        if (tid == 0) s_base = atomicAdd(sg.ctl, nseg);
        __syncthreads();
        const uint32_t at = __builtin_amdgcn_readfirstlane(s_base);
        const bool room = at + nseg <= sg.pool;  // always, unless the pool was capped
        for (uint32_t k = (uint32_t)tid; k < nseg && at + k < sg.pool; k += 256)
            sg.table[at + k] = make_uint2(room ? gtile : ~0u, k + 1 == nseg ? k | kSegmentLast : k);
        if (tid == 0 && room) sg.split[gtile] = 1u;
        if (!room) continue;  // walked whole by the gradient pass
        // The batches do not follow the segments: a row stores its pixels'
        // state whenever its walk passes a boundary (`bound`, the first record
        // of segment `s`).
        uint32_t s = nseg - 1, bound = s * seg_len;
        for (uint32_t top = maxlast; top > seg_len;) {
            const uint32_t first = top - seg_len > (uint32_t)BATCH ? top - BATCH : seg_len, cnt = top - first;
            __syncthreads();  // the previous walk has read the staged records
            if ((uint32_t)tid < cnt) {
                const Record& r = recs[payloads[start + first + (uint32_t)tid]];
                const float4 a = r.a_px, b = r.b_py;
                s_rec[0][tid] = r.m_nt;
                s_rec[1][tid] = a;
                s_rec[2][tid] = b;
                s_rec[3][tid] = r.col_op;
                if (AUX) s_n[tid] = r.nrm_dep;
                uint32_t mask = 0xFFFFu;
                if (cull) {
                    const SubTest t = sub_test(r.box, r.ell0, r.ell1, a.w, b.w);
                    mask = 0;
#pragma unroll
                    for (int i = 0; i < 4; ++i) mask |= sub_row_mask(t, (float)x0, (float)(y0 + 4 * i)) << 4 * i;
                }
                s_mask[tid] = (uint16_t)mask;
            }
            __syncthreads();
            if (wave_last > first) {
                // The wave's four lists, last record first: the records that
                // reach a row's sub-block before its last contributor.
                uint32_t n[4] = {0, 0, 0, 0};
#pragma unroll
                for (int c = BATCH / 64 - 1; c >= 0; --c) {
                    if ((uint32_t)(c * 64) >= cnt) continue;
                    const uint32_t slot = (uint32_t)(c * 64 + lane), mask = slot < cnt ? s_mask[slot] : 0u;
#pragma unroll
                    for (int q = 0; q < 4; ++q) {
                        const int sub = (2 * (wave >> 1) + (q >> 1)) * 4 + 2 * (wave & 1) + (q & 1);
                        const bool hit = (mask >> sub & 1u) && first + slot < rows_last[q];
                        const uint64_t bal = __ballot(hit);
                        if (hit) ((uint8_t*)s_list[sub])[n[q] + (uint32_t)__popcll(bal & gt_mask)] = (uint8_t)slot;
                        n[q] += (uint32_t)__popcll(bal);
                    }
                }
                const uint32_t mine = g == 0 ? n[0] : g == 1 ? n[1] : g == 2 ? n[2] : n[3];
                auto load = [&](uint32_t j, Record& r) {
                    r.m_nt = s_rec[0][j];
                    r.a_px = s_rec[1][j];
                    r.b_py = s_rec[2][j];
                    r.col_op = s_rec[3][j];
                    r.nrm_dep = AUX ? s_n[AUX ? j : 0] : make_float4(0.0f, 0.0f, 0.0f, 0.0f);
                };
                auto step = [&](uint32_t rel, const Record& r, const HitEval& h) {
                    while (rel < bound) {
                        store_state<AUX>(sg, at + s - 1, pixel, ps);
                        --s;
                        bound -= seg_len;
                    }
                    step_state<AUX>(ps, r, h, (rel < ps.last) & h.hit, lambda);
                };
                // Two records a round: their evaluations do not depend on the
                // walk state and overlap. Past a row's end: old slots, unused.
                uint32_t jj = my_list[0];
                for (uint32_t k = 0; __any(k < mine); k += 2) {
                    const uint32_t j0 = jj & 0xFFu, j1 = jj >> 8;
                    Record r0, r1;
                    load(j0, r0);
                    load(j1, r1);
                    jj = my_list[k / 2 + 1];
                    const HitEval h0 = eval_hit(r0, ps.sx, ps.sy, ps.pxc, ps.pyc);
                    const HitEval h1 = eval_hit(r1, ps.sx, ps.sy, ps.pxc, ps.pyc);
                    if (k < mine) step(first + j0, r0, h0);
                    if (k + 1 < mine) step(first + j1, r1, h1);
                }
            }
            top = first;
        }
        for (; s >= 1; --s) store_state<AUX>(sg, at + s - 1, pixel, ps);
        __syncthreads();  // s_last and s_base are rewritten by the next tile
    }
}

// Workgroups of a kernel that a CU holds.
template <auto Kernel>
uint32_t resident(uint32_t threads) {
    static const uint32_t fit = [threads] {
        int n = 0;
        const hipError_t e = hipOccupancyMaxActiveBlocksPerMultiprocessor(&n, Kernel, (int)threads, 0);
        return e == hipSuccess && n > 0 ? (uint32_t)n : 1u;
    }();
    return fit;
}

}  // namespace

hipError_t launch_bwd_prepare(hipStream_t st, CoefSlots grad_coef, size_t slots, uint32_t* cursor, BwdSegments sg,
                              uint32_t split_tiles, const uint32_t* entries, bool aux) {
    const size_t vecs = grad_coef.bytes(slots) / sizeof(float4);
    if (slots % 4 != 0) return hipErrorInvalidValue;
    uint64_t blocks = (std::max<size_t>(vecs, split_tiles) + 255) / 256;
    blocks = std::min<uint64_t>(std::max<uint64_t>(blocks, 1), 4096);
    hipLaunchKernelGGL(bwd_prepare_kernel, dim3((uint32_t)blocks), dim3(256), 0, st,
                       static_cast<float4*>(grad_coef.data), vecs, cursor, sg, split_tiles, entries,
                       aux ? kSegmentMinAux : kSegmentMin);
    return hipGetLastError();
}

hipError_t launch_raster_bwd(hipStream_t st, const CamParams* cams_dev, const CamParams* /*cams_host*/,
                             uint32_t n_views, uint32_t total_tiles, const uint32_t* ranges,
                             const uint32_t* payloads, const Record* recs, BwdIn in,
                             CoefSlots grad_coef, bool aux, bool cull, TileQueue queue, RasterShape shape,
                             uint32_t tile_begin, BwdSegments sg) {
    if (total_tiles == 0) return hipSuccess;
    const uint32_t t = shape.tile, b = shape.bwd_batch;
    // Segments need the queue (its order and cursors) and 16-px tiles.
    if (queue.cursor == nullptr || t != 16) sg = BwdSegments{};
    const uint32_t most = total_tiles + (sg.state != nullptr ? sg.pool : 0u);
    // With a queue, at most `times` workgroups for each that the schedule asks
    // for, and no more than the CUs hold (`fit`): positions below the grid size
    // belong to workgroups that should start at once.
    auto launch = [&](auto* kernel, auto* slots, uint32_t threads, uint32_t fit, uint32_t times) {
        uint32_t grid = total_tiles;
        if (queue.cursor != nullptr) {
            grid = std::min(most, std::max(times * queue.grid_blocks, 1u));
            if (queue.cus != 0) grid = std::min(grid, fit * queue.cus);
        }
        hipLaunchKernelGGL(kernel, dim3(grid), dim3(threads), 0, st, cams_dev, n_views, ranges, payloads, recs, in,
                           slots, cull, total_tiles, queue, tile_begin, sg);
    };
    auto go = [&](auto* narrow, auto* wide, uint32_t threads, uint32_t fit, uint32_t times = 1) {
        if (grad_coef.wide) launch(wide, static_cast<double*>(grad_coef.data), threads, fit, times);
        else launch(narrow, static_cast<float*>(grad_coef.data), threads, fit, times);
    };
    if (sg.state != nullptr) {
        // As many workgroups (four waves) as the CUs hold.
        const uint32_t fit = queue.cus * (aux ? kStateWaves<true> : kStateWaves<false>);
        const uint32_t g = std::min(total_tiles, std::max(fit != 0u ? fit : queue.grid_blocks / 2, 1u));
        if (aux)
            hipLaunchKernelGGL(raster_state_kernel<true>, dim3(g), dim3(256), 0, st, cams_dev, n_views, ranges,
                               payloads, recs, in, cull, total_tiles, queue, sg);
        else
            hipLaunchKernelGGL(raster_state_kernel<false>, dim3(g), dim3(256), 0, st, cams_dev, n_views, ranges,
                               payloads, recs, in, cull, total_tiles, queue, sg);
        const hipError_t e = hipGetLastError();
        if (e != hipSuccess) return e;
    }
    if (aux) {
        if (t != 16 || grad_coef.wide) return hipErrorInvalidValue;  // depth / normal losses: 16-px tiles, f32 slots
        launch(raster_bwd_kernel<true, 16, 128, float>, static_cast<float*>(grad_coef.data), 128,
               resident<raster_bwd_kernel<true, 16, 128, float>>(128), 1);
    } else if (t == 8 && b == 64) {
        go(raster_bwd_kernel<false, 8, 64, float>, raster_bwd_kernel<false, 8, 64, double>, 64,
           resident<raster_bwd_kernel<false, 8, 64, float>>(64));
    } else if (t == 8 && b == 128) {
        go(raster_bwd_kernel<false, 8, 128, float>, raster_bwd_kernel<false, 8, 128, double>, 64,
           resident<raster_bwd_kernel<false, 8, 128, float>>(64));
    } else if (t == 16 && b == 64) {
        // One wave per tile: twice the workgroups for the same waves per CU.
        go(raster_bwd_wave_kernel<64, float>, raster_bwd_wave_kernel<64, double>, 64,
           resident<raster_bwd_wave_kernel<64, float>>(64), 2);
    } else if (t == 16 && b == 128) {
        go(raster_bwd_wave_kernel<128, float>, raster_bwd_wave_kernel<128, double>, 64,
           resident<raster_bwd_wave_kernel<128, float>>(64), 2);
    } else if (t == 32 && b == 128) {
        go(raster_bwd_kernel<false, 32, 128, float>, raster_bwd_kernel<false, 32, 128, double>, 512,
           resident<raster_bwd_kernel<false, 32, 128, float>>(512));
    } else if (t == 32 && b == 256) {
        go(raster_bwd_kernel<false, 32, 256, float>, raster_bwd_kernel<false, 32, 256, double>, 512,
           resident<raster_bwd_kernel<false, 32, 256, float>>(512));
    } else {
        return hipErrorInvalidValue;
    }
    return hipGetLastError();
}

}  // namespace gs
