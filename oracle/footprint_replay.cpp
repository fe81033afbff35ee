/*
 * Replay of the rasterizer's footprint tests on the host (test infrastructure
 * only): the product's own record set-up, footprint, block, sub-block and tile
 * tests and hit evaluation (splattar_amd/csrc/gs_internal.h, compiled against
 * host_hip/), over every pixel of every record's 16-px rect. A test may keep
 * more than a record reaches; it may leave out nothing that the hit evaluation
 * (forward.rs:136-169) accepts.
 */
#include "../splattar_amd/csrc/gs_internal.h"

#include <random>
#include <vector>

using namespace gs;

namespace {

struct Counts {
    uint64_t hits = 0, misses[8] = {};
    uint64_t tests_hit = 0, tests = 0, bounded = 0, records = 0;
    double worst_radius = 0.0;
};

// Bits of the work tiles (ts px) that the projection's tight binning gives the
// record: the tiles its box meets, up to 64 of them masked by rows.
struct TileSet {
    uint4 rect;
    uint64_t mask;
    bool masked;
};
TileSet tight_tiles(const Record& r, uint32_t ts, uint32_t w, uint32_t h) {
    TileSet t{box_tiles(r.box, ts, (w + ts - 1) / ts, (h + ts - 1) / ts), ~0ull, false};
    if (t.rect.x > t.rect.z || t.rect.y > t.rect.w) return t;
    const uint32_t cols = t.rect.z - t.rect.x + 1u, rows = t.rect.w - t.rect.y + 1u;
    t.masked = cols * rows <= 64u;
    if (t.masked) {
        const SubTest s = sub_test(r.box, r.ell0, r.ell1, r.a_px.w, r.b_py.w);
        t.mask = 0ull;
        for (uint32_t y = t.rect.y, shift = 0u; y <= t.rect.w; ++y, shift += cols)
            t.mask |= tile_row_mask(s, t.rect.x, cols, y, ts) << shift;
    }
    return t;
}
bool has_tile(const TileSet& t, uint32_t tx, uint32_t ty) {
    if (tx < t.rect.x || tx > t.rect.z || ty < t.rect.y || ty > t.rect.w) return false;
    return !t.masked || (t.mask >> ((ty - t.rect.y) * (t.rect.z - t.rect.x + 1u) + tx - t.rect.x) & 1ull);
}

template <int TW>
void check_tile(const Record& r, const CamParams& cam, uint32_t x0, uint32_t y0, const TileSet& set, Counts& c,
                int slot) {
    const uint32_t blocks = block_mask<TW>(r, x0, y0);
    uint64_t subs = 0;
    constexpr int NS = TW / 4;
    const SubTest t = sub_test(r.box, r.ell0, r.ell1, r.a_px.w, r.b_py.w);
    if (TW <= 16)  // as the forward and the state pass do
        for (int i = 0; i < NS; ++i)
            subs |= (uint64_t)(sub_row_mask(t, (float)x0, (float)(y0 + 4 * i)) & ((1u << NS) - 1u)) << NS * i;
    const bool tile = has_tile(set, x0 / TW, y0 / TW);
    for (uint32_t y = y0; y < y0 + TW && y < cam.height; ++y)
        for (uint32_t x = x0; x < x0 + TW && x < cam.width; ++x) {
            float sx, sy;
            pixel_s(cam, (int)x, (int)y, sx, sy);
            if (!eval_hit(r, sx, sy, (float)x + 0.5f, (float)y + 0.5f).hit) continue;
            const uint32_t dx = x - x0, dy = y - y0;
            if (slot == 0) ++c.hits;
            if (!tile) ++c.misses[slot];
            if (!(blocks >> ((dy / 8) * (TW / 8) + dx / 8) & 1u)) ++c.misses[slot + 1];
            if (TW <= 16 && !(subs >> ((dy / 4) * NS + dx / 4) & 1u)) ++c.misses[slot + 2];
        }
    if (TW == 16) {
        c.tests += 16;
        c.tests_hit += (uint64_t)__builtin_popcountll(subs);
    }
}

}  // namespace

/*
 * n random surfels before a camera of w x h pixels. kind: 0 the usual
 * distribution, 1 thin surfels, 2 seen edge-on, 3 opacities at the threshold,
 * 4 large and near, 5 all of these mixed. out (16): accepted (pixel, record)
 * evaluations; those left out by the 16-px tile, 8x8 block and 4x4 sub-block
 * tests, the 8-px tile, its block and sub-block tests, the 32-px tile and block
 * tests; 4x4 tests that keep the record and all of them; records with a bounded
 * ellipse and all records; 0. radius_err: the largest relative error of a stored disk radius
 * against its f64 value rounded to f32.
 */
extern "C" int oref_footprint_replay(uint64_t seed, uint32_t n, uint32_t w, uint32_t h, int kind, uint64_t* out,
                                     double* radius_err) {
    if (n == 0 || w == 0 || h == 0 || out == nullptr || radius_err == nullptr) return 1;
    Counts total;
#pragma omp parallel
    {
        Counts c;
#pragma omp for schedule(dynamic, 64)
        for (uint32_t i = 0; i < n; ++i) {
            std::mt19937_64 rng(seed * 0x9E3779B97F4A7C15ull + i);
            std::normal_distribution<double> nrm;
            std::uniform_real_distribution<double> uni;
            const int k = kind == 5 ? (int)(rng() % 5) : kind;
            CamParams cam{};
            cam.rot[0] = cam.rot[4] = cam.rot[8] = 1.0f;
            cam.center[2] = 3.0f;
            cam.focal = (float)(0.5 * h / std::tan(0.5235987755982988) * std::exp(uni(rng) * 2.0 - 0.7));
            cam.cx = 0.5f * (float)w;
            cam.cy = 0.5f * (float)h;
            cam.width = w;
            cam.height = h;
            cam.rtiles_x = (w + 15) / 16;
            cam.rtiles_y = (h + 15) / 16;
            const double spread = k == 4 ? 2.5 : 1.2;
            const float4 p = make_float4((float)(spread * (2 * uni(rng) - 1)), (float)(spread * (2 * uni(rng) - 1)),
                                         (float)(spread * (2 * uni(rng) - 1)), 1.0f);
            double su = std::exp(-4.0 + 0.9 * nrm(rng)), sv = std::exp(-4.0 + 0.9 * nrm(rng));
            if (k == 1) sv = su * std::pow(10.0, -1.0 - 3.0 * uni(rng));
            if (k == 4) su *= 30.0, sv *= 30.0;
            float4 q = make_float4((float)nrm(rng), (float)nrm(rng), (float)nrm(rng), (float)nrm(rng));
            if (k == 2) {
                // Normal nearly at right angles to the viewing direction: z to
                // a direction in the image plane, tilted by 1e-1 to 1e-6.
                const double a = 6.283185307179586 * uni(rng);
                const double tilt = 1.5707963267948966 + (uni(rng) < 0.5 ? -1 : 1) * std::pow(10.0, -1.0 - 5.0 * uni(rng));
                q = make_float4((float)(std::sin(tilt / 2) * std::cos(a)), (float)(std::sin(tilt / 2) * std::sin(a)), 0.0f,
                                (float)std::cos(tilt / 2));
            }
            double op = 1.0 / (1.0 + std::exp(-nrm(rng)));
            if (k == 3) op = (1.0 + std::pow(10.0, -5.0 * uni(rng))) / 255.0;
            const CamFrame f = cam_frame(cam, p, float2{(float)su, (float)sv}, q);
            const float depth = -f.cz_;
            if (!(depth >= kNearDepth)) continue;
            const RectOut rect = tile_rect(cam, f, depth);
            if (!rect.on_screen) continue;
            // The record, as project.hip builds it.
            const float3 cc = make_float3(f.cx_, f.cy_, f.cz_), tu = make_float3(f.tux, f.tuy, f.tuz),
                         tv = make_float3(f.tvx, f.tvy, f.tvz);
            const float3 M = cross3(tu, tv), A = cross3(tv, cc), B = cross3(cc, tu);
            Record r{};
            r.m_nt = make_float4(M.x, M.y, M.z, -dot3(M, cc));
            r.a_px = make_float4(A.x, A.y, A.z, rect.px);
            r.b_py = make_float4(B.x, B.y, B.z, rect.py);
            r.col_op.w = (float)op;
            r.nrm_dep.w = depth;
            record_footprint(r, cam);
            ++c.records;
            if (r.ell1.y > 0.0f && r.ell0.x < 1e17f) ++c.bounded;
            if (r.col_op.w * 255.0f > 1.0f) {
                const float want = (float)(std::sqrt(std::log((double)r.col_op.w * 255.0) + 2e-3) + kMargin);
                c.worst_radius = std::max(c.worst_radius, std::fabs((double)r.ell1.w - want) / want);
            }
            r.box = clip_box_to_rect(r.box, make_uint4(rect.x0, rect.y0, rect.x1, rect.y1));
            const TileSet t8 = tight_tiles(r, 8, w, h), t16 = tight_tiles(r, 16, w, h), t32 = tight_tiles(r, 32, w, h);
            for (uint32_t ty = rect.y0; ty <= rect.y1; ++ty)
                for (uint32_t tx = rect.x0; tx <= rect.x1; ++tx) {
                    check_tile<16>(r, cam, 16 * tx, 16 * ty, t16, c, 0);
                    for (uint32_t b = 0; b < 4; ++b) check_tile<8>(r, cam, 16 * tx + 8 * (b & 1), 16 * ty + 8 * (b >> 1), t8, c, 3);
                }
            // A 32-px tile also holds pixels of 16-px tiles outside the rect,
            // which the clipped box keeps out of the model: only its own.
            for (uint32_t ty = rect.y0; ty <= rect.y1; ++ty)
                for (uint32_t tx = rect.x0; tx <= rect.x1; ++tx) {
                    const uint32_t x0 = tx / 2 * 32, y0 = ty / 2 * 32;
                    const uint32_t blocks = block_mask<32>(r, x0, y0);
                    const bool tile = has_tile(t32, tx / 2, ty / 2);
                    for (uint32_t y = 16 * ty; y < 16 * ty + 16 && y < h; ++y)
                        for (uint32_t x = 16 * tx; x < 16 * tx + 16 && x < w; ++x) {
                            float sx, sy;
                            pixel_s(cam, (int)x, (int)y, sx, sy);
                            if (!eval_hit(r, sx, sy, (float)x + 0.5f, (float)y + 0.5f).hit) continue;
                            if (!tile) ++c.misses[6];
                            if (!(blocks >> ((y - y0) / 8 * 4 + (x - x0) / 8) & 1u)) ++c.misses[7];
                        }
                }
        }
#pragma omp critical
        {
            total.hits += c.hits;
            for (int j = 0; j < 8; ++j) total.misses[j] += c.misses[j];
            total.tests += c.tests;
            total.tests_hit += c.tests_hit;
            total.bounded += c.bounded;
            total.records += c.records;
            total.worst_radius = std::max(total.worst_radius, c.worst_radius);
        }
    }
    out[0] = total.hits;
    for (int j = 0; j < 8; ++j) out[1 + j] = total.misses[j];
    out[9] = total.tests_hit;
    out[10] = total.tests;
    out[11] = total.bounded;
    out[12] = total.records;
    for (int j = 13; j < 16; ++j) out[j] = 0;
    *radius_err = total.worst_radius;
    return 0;
}
