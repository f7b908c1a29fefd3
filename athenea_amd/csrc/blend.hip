// blend.hip -- the per-tile front-to-back alpha blend for gfx950 and its
// adjoint.
//
// Forward: shaders/athenea/splat/splat_blend.slang:236-578 (splatBlend,
// blendPixel with composite, matte and trace off, contributionMode 0). One
// workgroup a tile of 8 or 16 pixels and four a tile of 32 (a 16 x 16 quarter
// each), one thread per pixel; the tile's Gaussians are staged in LDS a batch
// at a time (the reference stages 256, splat_blend.slang:300-311) and every
// pixel walks the ones that meet its own 4 x 4 block, from that block's list.
// A frame that keeps its walk for the adjoint stages listed pairs, `batch` at a
// time (blend_kernel); a plain one picks the tile's Gaussians out of its strip
// entries, in batches of its own (blend_entries_kernel); the variants and the
// contributions walk listed pairs that meet 8 x 8 pixels (blend_ex_kernel,
// contribution_kernel). A wavefront whose 64 pixels are all
// done stops walking at once; the group stops loading when every wavefront
// has stopped. Each pixel also keeps its final transmittance and how many of
// its tile's pairs it read, which is all the adjoint needs to replay the walk.
//
// Adjoint: no counterpart in the reference. It walks the same pairs back to
// front from the same block lists, recovering the transmittance before each
// Gaussian from the one after it (T_k = T_{k+1} / (1 - alpha_k); alpha <= 0.99
// keeps it stable), and accumulates per-slot gradients of the centre, conic,
// alpha and colour. The 16 lanes of a row walk one block's list, so a Gaussian's
// gradient is summed across the row first, then over the tile's blocks in LDS,
// and added to memory once a batch.
#include "athx_internal.h"
#include "bounds.h"

namespace athx {
namespace {

constexpr uint32_t kMaxBatch = 256;

__device__ inline uint32_t view_of_tile(const uint32_t* tile_bases, uint32_t nviews, uint32_t tile) {
    uint32_t lo = 0, hi = nviews;  // tile_bases[nviews] is the total
    while (hi - lo > 1) {
        const uint32_t mid = (lo + hi) >> 1;
        if (tile_bases[mid] <= tile) {
            lo = mid;
        } else {
            hi = mid;
        }
    }
    return lo;
}

struct LdsBatch {
    float4 xy_cut_op[kMaxBatch];  // centre x, y, cutoff, alpha
    float4 conic[kMaxBatch];      // a, 2b, c, view z
    float4 colour[kMaxBatch];     // r, g, b, conic b
};

__device__ inline void stage(LdsBatch& s, uint32_t k, const float* records, uint32_t slot) {
    const float4* rec = reinterpret_cast<const float4*>(records + (size_t)slot * kRecordFloats);
    const float4 screen = rec[0];
    const float4 conic = rec[1];
    const float4 col = rec[2];
    s.xy_cut_op[k] = make_float4(screen.x, screen.y, screen.w, conic.w);
    s.conic[k] = make_float4(conic.x, 2.0f * conic.y, conic.z, screen.z);
    s.colour[k] = make_float4(col.x, col.y, col.z, conic.y);
}

// A pair's record words.
struct Staged {
    float4 screen, conic, col;
};

__device__ inline Staged fetch(const float* records, uint32_t slot) {
    const float4* rec = reinterpret_cast<const float4*>(records + (size_t)slot * kRecordFloats);
    return Staged{rec[0], rec[1], rec[2]};
}

// e^(-power / 2) for a drawn pair: power <= the cut power <= 9, and above
// a tiny negative rounding floor for a positive definite conic, so the
// argument lies in [-4.5, 0+] where athx_expf_core equals athx_expf; the
// median only bounds it for inputs no record holds.
__device__ inline float blend_exp_of(float x) { return athx_expf_core(__builtin_amdgcn_fmed3f(x, -80.0f, 80.0f)); }
__device__ inline float blend_exp(float power) { return blend_exp_of(-0.5f * power); }

// A WAVEFRONT'S BAND. A tile's pairs are every Gaussian whose ellipse meets
// the tile; a wavefront's 64 pixels are an 8 x 8 block of it (its band: the
// squarest of 64 pixels, which the fewest ellipses meet -- against a band of
// 64 / TILE whole rows, 10 % fewer walked on the 60-view walk), and a small
// Gaussian often misses the band altogether, so that no
// lane of the wavefront could take it. Each wavefront tests its band against
// 64 staged Gaussians at once, a lane each, and walks only those that meet
// it: the walk and every result are the same, pair for pair, since a
// Gaussian skipped is one whose power exceeds the cut at every pixel centre
// of the band. The test is conservative: the least power over the band's box
// of pixel centres (zero when the box holds the centre, else the least over
// its edges, each at its clamped stationary point) must exceed the cut by
// kBandSlack * M, M = a X^2 + 2 |b| X Y + c Y^2 with X, Y the box's largest
// distances from the centre -- far above the rounding of both this float
// evaluation and the per-pixel one (a few units of 2^-24 M).
constexpr float kBandSlack = 256.0f * 0x1p-24f;

struct Band {
    float x0, x1, y0, y1;  // the band's first and last pixel centres
};

// Wavefront w of a TILE x TILE workgroup takes the 8 x 8 pixel block
// (w % (TILE / 8), w / (TILE / 8)) of the tile, lane l its pixel (l % 8, l / 8).
template <uint32_t TILE>
__device__ inline void block_pixel(uint32_t tid, uint32_t& lx, uint32_t& ly) {
    constexpr uint32_t kBx = TILE / 8;
    const uint32_t w = tid >> 6, l = tid & 63u;
    lx = (w % kBx) * 8u + (l & 7u);
    ly = (w / kBx) * 8u + (l >> 3);
}

template <uint32_t TILE>
__device__ inline Band wave_band(const DView& V, uint32_t tx, uint32_t ty, uint32_t wave) {
    constexpr uint32_t kBx = TILE / 8;
    const uint32_t c0 = tx * TILE + (wave % kBx) * 8u, r0 = ty * TILE + (wave / kBx) * 8u;
    // A block past the view's edge holds no pixel (its lanes never walk).
    const uint32_t c1 = min(c0 + 8u, V.width), r1 = min(r0 + 8u, V.height);
    Band b;
    b.x0 = (float)c0 + 0.5f;
    b.x1 = (float)(c1 > c0 ? c1 - 1u : c0) + 0.5f;
    b.y0 = (float)r0 + 0.5f;
    b.y1 = (float)(r1 > r0 ? r1 - 1u : r0) + 0.5f;
    return b;
}

__device__ inline bool band_meets(const Band& B, float cx, float cy, float a, float b, float c, float cut) {
    const float lox = B.x0 - cx, hix = B.x1 - cx, loy = B.y0 - cy, hiy = B.y1 - cy;
    if (lox <= 0.0f && hix >= 0.0f && loy <= 0.0f && hiy >= 0.0f) {
        return true;
    }
    if (!(a > 1e-12f) || !(c > 1e-12f)) {
        return true;
    }
    const float ia = __builtin_amdgcn_rcpf(a), ic = __builtin_amdgcn_rcpf(c);
    const auto at = [&](float x, float y) { return (a * x * x + 2.0f * b * x * y) + c * y * y; };
    const float ya = clamp_(-b * lox * ic, loy, hiy), yb = clamp_(-b * hix * ic, loy, hiy);
    const float xa = clamp_(-b * loy * ia, lox, hix), xb = clamp_(-b * hiy * ia, lox, hix);
    const float least = fmin_(fmin_(at(lox, ya), at(hix, yb)), fmin_(at(xa, loy), at(xb, hiy)));
    const float X = fmax_(fabsf(lox), fabsf(hix)), Y = fmax_(fabsf(loy), fabsf(hiy));
    const float M = (a * X * X + 2.0f * fabsf(b) * X * Y) + c * Y * Y;
    // Skipped only on a definite answer: a NaN anywhere keeps the Gaussian.
    return !(least > cut + kBandSlack * M);
}

// The staged Gaussians first .. first + 63 of the batch (count staged) that
// meet the band, as a mask of lanes: bit i for Gaussian first + i.
template <uint32_t TILE>
__device__ inline uint64_t band_mask(const LdsBatch& s, const Band& B, uint32_t first, uint32_t count, uint32_t lane) {
    if constexpr (TILE == 8) {
        // A wavefront is the whole tile, which every pair meets.
        const uint32_t n = count - first < 64u ? count - first : 64u;
        return n == 64u ? ~0ull : ((1ull << n) - 1ull);
    } else {
        const uint32_t j = first + lane;
        bool meets = false;
        if (j < count) {
            const float4 q = s.xy_cut_op[j];
            const float4 k = s.conic[j];
            meets = band_meets(B, q.x, q.y, k.x, s.colour[j].w, k.z, q.z);
        }
        return __ballot(meets);
    }
}

// A QUARTER WAVEFRONT'S BLOCK. The plain walk and its adjoint go finer than
// the band: each row of 16 lanes owns a 4 x 4 pixel block and walks its own
// list of the staged Gaussians that meet it, so the four rows of a wavefront
// are at four different Gaussians in the same step, and a wavefront's steps
// are the longest of its rows' lists instead of the union of what meets 8 x 8
// pixels. Both kernels are bound by the VALU's issue rate, so steps are time.
//
// Which blocks a Gaussian meets is found once, by the thread that staged it:
// the x-extent of the ellipse q <= C sliced by each row of blocks (the slice
// is convex, its ends a closed form) against the blocks' pixel centres, with
// C = cut + kBandSlack M over the whole tile, so a Gaussian left out of a
// block's list exceeds its cut at every pixel centre of it in any rounding
// (the strip classifier's rule, outer extent). A conic the extents do not
// handle meets every block. The answers are one ballot a block and 64
// Gaussians; each wavefront expands its own blocks' ballots into lists of
// LDS offsets.
//
// A 32 x 32 tile is walked by four workgroups of 16 x 16 pixels (SPLIT 2), each
// over the tile's pairs for its own quarter: one workgroup of 1024 lanes tests
// 64 blocks in the few wavefronts that stage, while the others wait (600 k at
// 1600 x 1100: 403 us a launch, against 8 x 8 pixels a step's 278).
//
// Measured against walking what meets a wavefront's 8 x 8 pixels, one Gaussian
// a step (us a launch, MI355X): 100 k Gaussians at 512 x 512 109 -> 61, 1.4 M
// at 1920 x 1080 244 -> 206, the 60-view walk 3 340 -> 2 420, 20 M in eight
// views 3 415 -> 2 045.
constexpr uint32_t kBlock = 4;  // a block's side, pixels

// A staged Gaussian as the walk reads it: three 16-byte words. The conic is
// stored times -1/2 (2 b times -1/2 is -b), an exact scaling, so the walk's
// sum is the exponent itself.
struct LdsRecord {
    float4 a;  // centre x, y, -a / 2, -b
    float4 b;  // -c / 2, -cut / 2, alpha, view z
    float4 c;  // r, g, b, conic b
};

template <uint32_t TILE, uint32_t BATCH>
struct LdsWalk {
    static constexpr uint32_t kSide = TILE / kBlock;       // blocks a tile's side
    static constexpr uint32_t kBlocks = kSide * kSide;
    static constexpr uint32_t kChunks = (BATCH + 63) / 64;  // a ballot's Gaussians each
    LdsRecord rec[BATCH + 1];  // and one that no pixel takes, which pads a list of odd length
    alignas(16) uint64_t meets[kChunks][kBlocks];
    uint16_t list[kBlocks][BATCH + 2];  // byte offsets of rec
};

__device__ inline void put(LdsRecord& d, const Staged& r) {
    d.a = make_float4(r.screen.x, r.screen.y, -0.5f * r.conic.x, -r.conic.y);
    d.b = make_float4(-0.5f * r.conic.z, -0.5f * r.screen.w, r.conic.w, r.screen.z);
    d.c = make_float4(r.col.x, r.col.y, r.col.z, r.conic.y);
}

// Lane l's pixel of wavefront w: row r = l / 16 of the wavefront takes block
// (r % 2, r / 2) of the wavefront's 8 x 8 pixels, its lanes the block's
// pixels row by row.
template <uint32_t TILE>
__device__ inline void quarter_pixel(uint32_t tid, uint32_t& lx, uint32_t& ly) {
    constexpr uint32_t kBx = TILE / 8;
    const uint32_t w = tid >> 6, row = (tid >> 4) & 3u, l = tid & 15u;
    lx = (w % kBx) * 8u + (row & 1u) * kBlock + (l & 3u);
    ly = (w / kBx) * 8u + (row >> 1) * kBlock + (l >> 2);
}

// The blocks of the tile (first pixel centre x0, y0) that each lane's
// Gaussian meets, one ballot a block written to out[block]: SLICES rows of
// blocks from the given one on. Every lane of the wavefront is active.
template <uint32_t TILE, uint32_t SLICES = TILE / kBlock>
__device__ inline void blocks_met(const Staged& r, bool valid, float x0, float y0, uint32_t lane, uint64_t* out,
                                  uint32_t slice = 0) {
    constexpr uint32_t kSide = TILE / kBlock;
    const float cx = r.screen.x, cy = r.screen.y, a = r.conic.x, b = r.conic.y, c = r.conic.z;
    const float xl = x0 - cx, yl = y0 - cy;
    const float X = fmaxf(fabsf(xl), fabsf(xl + (float)(TILE - 1u)));
    const float Y = fmaxf(fabsf(yl), fabsf(yl + (float)(TILE - 1u)));
    const float C = r.screen.w + kBandSlack * (a * X * X + 2.0f * fabsf(b) * X * Y + c * Y * Y);
    const float det = (float)((double)a * (double)c - (double)b * (double)b);
    const bool known = (a > 1e-9f) & (c > 1e-9f) & (det >= 0x1p-126f) & (det <= 0x1p126f) & (C > 0.0f);
    const float inv_det = __builtin_amdgcn_rcpf(det);
    const float ia = __builtin_amdgcn_rcpf(a), ic = __builtin_amdgcn_rcpf(c);
    // The ellipse's rows |y| <= ym; its widest points at y = -+yw.
    const float ym = __builtin_amdgcn_sqrtf(C * (a * inv_det));
    const float yw = (b * __builtin_amdgcn_sqrtf(C * (c * inv_det))) * ic;
    const float aC = a * C;
    uint64_t met[SLICES * kSide];
    const float ys = yl + (float)(slice * kBlock);
#pragma unroll
    for (uint32_t s = 0; s < SLICES; ++s) {
        const float b0 = ys + (float)(s * kBlock), b1 = ys + (float)(s * kBlock + kBlock - 1u);
        const float ya = fmaxf(b0, -ym), yb = fminf(b1, ym);
        const float yr = __builtin_amdgcn_fmed3f(-yw, ya, yb), yq = __builtin_amdgcn_fmed3f(yw, ya, yb);
        const float hr = fmaxf(__builtin_fmaf(-(det * yr), yr, aC), 0.0f);
        const float hq = fmaxf(__builtin_fmaf(-(det * yq), yq, aC), 0.0f);
        const float xb = __builtin_fmaf(-b, yr, __builtin_amdgcn_sqrtf(hr)) * ia;
        const float xa = -__builtin_fmaf(b, yq, __builtin_amdgcn_sqrtf(hq)) * ia;
        const bool none = ya > yb;
#pragma unroll
        for (uint32_t k = 0; k < kSide; ++k) {
            const float e0 = xl + (float)(k * kBlock), e1 = xl + (float)(k * kBlock + kBlock - 1u);
            // Left out only on a definite answer: a NaN anywhere keeps it.
            const bool apart = known & (none | (e1 < xa) | (e0 > xb));
            met[s * kSide + k] = __builtin_amdgcn_ballot_w64(valid & !apart);
        }
    }
    if (lane == 0) {
#pragma unroll
        for (uint32_t i = 0; i < SLICES * kSide; i += 2) {
            *reinterpret_cast<ulonglong2*>(out + slice * kSide + i) = make_ulonglong2(met[i], met[i + 1]);
        }
    }
}

// The sum, and the largest, over this lane's row of 16 lanes, in all of them
// (rotations within the row). Every lane of the row is active.
__device__ inline uint32_t row_sum(uint32_t x) {
    x += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)x, 0x121, 0xF, 0xF, true);
    x += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)x, 0x122, 0xF, 0xF, true);
    x += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)x, 0x124, 0xF, 0xF, true);
    return x + (uint32_t)__builtin_amdgcn_update_dpp(0, (int)x, 0x128, 0xF, 0xF, true);
}
__device__ inline uint32_t row_max(uint32_t x) {
    x = max(x, (uint32_t)__builtin_amdgcn_update_dpp(0, (int)x, 0x121, 0xF, 0xF, true));
    x = max(x, (uint32_t)__builtin_amdgcn_update_dpp(0, (int)x, 0x122, 0xF, 0xF, true));
    x = max(x, (uint32_t)__builtin_amdgcn_update_dpp(0, (int)x, 0x124, 0xF, 0xF, true));
    return max(x, (uint32_t)__builtin_amdgcn_update_dpp(0, (int)x, 0x128, 0xF, 0xF, true));
}

// Expands the ballots of this lane's row's block into its list, lane q of the
// row a sixteenth of the ballots' bits; of the batch the first `count`.
// Returns the list's length. Every lane of the wavefront is active.
template <uint32_t TILE, uint32_t BATCH>
__device__ inline uint32_t expand_list(LdsWalk<TILE, BATCH>& s, uint32_t block, uint32_t lane, uint32_t count) {
    constexpr uint32_t kBits = LdsWalk<TILE, BATCH>::kChunks * 4;  // a lane's
    static_assert(64 % kBits == 0, "a lane's bits lie in one ballot");
    const uint32_t q = lane & 15u, first = q * kBits;
    const uint32_t mine = count > first ? (count - first < kBits ? count - first : kBits) : 0u;
    // (A chunk of 64 past the count was not tested: its ballots are stale.)
    uint32_t bits = (uint32_t)(s.meets[first >> 6][block] >> (first & 63u)) & ((1u << mine) - 1u);
    const uint32_t here = (uint32_t)__popc(bits);
    uint32_t incl = here;
    incl += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)incl, 0x111, 0xF, 0xF, true);
    incl += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)incl, 0x112, 0xF, 0xF, true);
    incl += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)incl, 0x114, 0xF, 0xF, true);
    incl += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)incl, 0x118, 0xF, 0xF, true);
    uint16_t* out = s.list[block] + (incl - here);
    const uint32_t base = first * (uint32_t)sizeof(LdsRecord);
    for (; bits != 0; bits &= bits - 1u) {
        *out++ = (uint16_t)(base + __umul24((uint32_t)__builtin_ctz(bits), (uint32_t)sizeof(LdsRecord)));
    }
    if (q == 15u) {
        *out = (uint16_t)(BATCH * sizeof(LdsRecord));
    }
    return row_sum(here);
}

// The wavefront's own LDS writes seen by its own lanes (no other wavefront's
// are read).
__device__ inline void wave_lds_fence() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup");
}

// What a pixel's walk has gathered.
struct Pixel {
    float r = 0.0f, g = 0.0f, b = 0.0f, T = 1.0f, dsum = 0.0f, dat = -1.0f;
    bool done = false;
};

// The record that pads a list of odd length: the exponent 0 is below 1, so no
// pixel takes it.
__device__ inline void put_padding(LdsRecord& d) {
    d.a = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
    d.b = make_float4(0.0f, 1.0f, 0.0f, 0.0f);
    d.c = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
}

// Walks a block's list for this lane's pixel until it is done; returns the
// offset of the last Gaussian it took, or ~0. Two Gaussians a step: their
// exponents and alphas side by side (what a wavefront waits on where few are
// resident), then taken in order.
template <bool kThreshold>
__device__ inline uint32_t walk_list(const LdsRecord* rec, const uint16_t* list, uint32_t length, float pxc, float pyc,
                                     float depth_threshold, Pixel& p) {
    uint32_t last_at = ~0u;
    const auto record = [&](uint32_t at) -> const LdsRecord& {
        return *reinterpret_cast<const LdsRecord*>(reinterpret_cast<const char*>(rec) + at);
    };
    const auto take = [&](uint32_t at, float alpha, const float4& qb, const float4& qc) {
        const float w = p.T * alpha;
        p.r = p.r + w * qc.x;
        p.g = p.g + w * qc.y;
        p.b = p.b + w * qc.z;
        p.dsum = p.dsum + w * qb.w;
        p.T = p.T * (1.0f - alpha);
        if (kThreshold && p.dat < 0.0f && 1.0f - p.T >= depth_threshold) {
            p.dat = qb.w;
        }
        last_at = at;
        p.done = p.T < 1e-4f;
    };
    for (uint32_t i = 0; i < length && !p.done; i += 2) {
        const uint32_t two = *reinterpret_cast<const uint32_t*>(list + i);
        const uint32_t at0 = two & 0xFFFFu, at1 = two >> 16;
        const LdsRecord &k0 = record(at0), &k1 = record(at1);
        const float4 a0 = k0.a, b0 = k0.b, c0 = k0.c, a1 = k1.a, b1 = k1.b, c1 = k1.c;
        const float dx0 = pxc - a0.x, dy0 = pyc - a0.y, dx1 = pxc - a1.x, dy1 = pyc - a1.y;
        const float e0 = a0.z * dx0 * dx0 + a0.w * dx0 * dy0 + b0.x * dy0 * dy0;
        const float e1 = a1.z * dx1 * dx1 + a1.w * dx1 * dy1 + b1.x * dy1 * dy1;
        const float alpha0 = fminf(0.99f, b0.z * blend_exp_of(e0));
        const float alpha1 = fminf(0.99f, b1.z * blend_exp_of(e1));
        if (!(e0 < b0.y) & !(alpha0 < 1.0f / 255.0f)) {
            take(at0, alpha0, b0, c0);
        }
        if (!p.done & !(e1 < b1.y) & !(alpha1 < 1.0f / 255.0f)) {
            take(at1, alpha1, b1, c1);
        }
    }
    return last_at;
}

__device__ inline void finish_pixel(const DView& V, uint32_t px, uint32_t py, const Pixel& p, uint32_t last,
                                    uint32_t depth_mode) {
    const size_t pix = (size_t)py * V.width + px;
    const float coverage = 1.0f - p.T;
    float4 out;
    out.x = p.r + p.T * V.bg[0];
    out.y = p.g + p.T * V.bg[1];
    out.z = p.b + p.T * V.bg[2];
    out.w = coverage + p.T * V.bg[3];
    reinterpret_cast<float4*>(V.colour)[pix] = out;
    if (V.depth) {
        V.depth[pix] = depth_mode == 0 ? (coverage > 1e-6f ? p.dsum / coverage : 0.0f) : fmaxf(p.dat, 0.0f);
    }
    if (V.final_t) {
        V.final_t[pix] = p.T;
    }
    if (V.last) {
        V.last[pix] = last;
    }
}

template <uint32_t TILE, uint32_t SPLIT, bool kPiped, bool kThreshold>
__global__ void __launch_bounds__(TILE * TILE) blend_kernel(const DView* __restrict__ views,
                                                            const uint32_t* __restrict__ tile_bases, uint32_t nviews,
                                                            uint32_t batch, const uint32_t* __restrict__ ranges,
                                                            const uint32_t* __restrict__ pair_slots,
                                                            const float* __restrict__ records, uint32_t depth_mode,
                                                            float depth_threshold) {
    constexpr uint32_t kThreads = TILE * TILE;
    constexpr uint32_t kBx = TILE / 8, kSide = TILE / kBlock;
    __shared__ LdsWalk<TILE, kMaxBatch> s;
    // Tiles in dispatch order, not in bands an XCD: every XCD then walks the
    // same view at once, so the records gathered at any time are one view's
    // (a working set the 256 MB infinity cache holds, where eight views' do
    // not), and the views' unequal loads even out over the XCDs.
    const uint32_t gtile = blockIdx.x / (SPLIT * SPLIT), part = blockIdx.x % (SPLIT * SPLIT);
    const uint32_t v = view_of_tile(tile_bases, nviews, gtile);
    const DView& V = views[v];
    const uint32_t local = gtile - V.tile_base;
    // The workgroup's first pixel.
    const uint32_t ox = ((local % V.tiles_x) * SPLIT + part % SPLIT) * TILE;
    const uint32_t oy = ((local / V.tiles_x) * SPLIT + part / SPLIT) * TILE;
    const uint32_t tid = threadIdx.x;
    uint32_t lx, ly;
    quarter_pixel<TILE>(tid, lx, ly);
    const uint32_t px = ox + lx, py = oy + ly;
    const bool inside = px < V.width && py < V.height;
    const uint32_t start = ranges[2 * gtile], end = ranges[2 * gtile + 1];
    const float pxc = (float)px + 0.5f, pyc = (float)py + 0.5f;
    const float x0 = (float)ox + 0.5f, y0 = (float)oy + 0.5f;

    Pixel p;
    p.done = !inside;
    uint32_t last = 0;
    const uint32_t lane = tid & 63u, wave = tid >> 6, row = (tid >> 4) & 3u;
    const uint32_t block = ((wave / kBx) * 2u + (row >> 1)) * kSide + (wave % kBx) * 2u + (row & 1u);
    // With a batch of at most a record a thread (kPiped), the staging is
    // pipelined:
    // while a batch is walked, each thread already reads its record of the
    // next batch (its slot read during the batch before) and its slot of the
    // batch after, so a batch's staging waits on no memory.
    // The reads are unconditional (a thread with no pair reads the tile's
    // last one again, and its record is never staged), so no branch holds
    // them back.
    Staged ahead{};
    uint32_t slot_ahead = 0;
    if (kPiped && start < end) {
        ahead = fetch(records, pair_slots[min(start + tid, end - 1u)]);
        slot_ahead = pair_slots[min(start + batch + tid, end - 1u)];
    }
    if (tid == 0) {
        put_padding(s.rec[kMaxBatch]);
    }
    for (uint32_t first = start; first < end; first += batch) {
        if (!__syncthreads_or(!p.done)) {
            break;
        }
        const uint32_t count = end - first < batch ? end - first : batch;
        if constexpr (kPiped) {
            if (tid < count) {
                put(s.rec[tid], ahead);
            }
        }
        for (uint32_t c = wave; c * 64u < count; c += kThreads / 64u) {
            const uint32_t k = c * 64u + lane;
            if constexpr (!kPiped) {
                ahead = fetch(records, pair_slots[min(first + k, end - 1u)]);
                if (k < count) {
                    put(s.rec[k], ahead);
                }
            }
            blocks_met<TILE>(ahead, k < count, x0, y0, lane, s.meets[c]);
        }
        __syncthreads();
        if constexpr (kPiped) {
            ahead = fetch(records, slot_ahead);
            slot_ahead = pair_slots[min(first + 2u * batch + tid, end - 1u)];
        }
        if (__ballot(!p.done) == 0) {
            continue;  // the wavefront's pixels are done: it only stages
        }
        const uint32_t length = expand_list(s, block, lane, count);
        wave_lds_fence();
        const uint32_t last_at = walk_list<kThreshold>(s.rec, s.list[block], length, pxc, pyc, depth_threshold, p);
        // Pairs a pixel skipped after its last contribution are read again by
        // nobody: `last` is the walk's own extent.
        if (last_at != ~0u) {
            last = first - start + last_at / (uint32_t)sizeof(LdsRecord) + 1u;
        }
    }
    if (inside) {
        finish_pixel(V, px, py, p, last, depth_mode);
    }
}

// The same walk straight from the sorted strip entries, for a frame whose pairs
// nobody reads back: the tile's pairs are its strip's entries whose mask holds
// the tile, in the entries' order, so the workgroup picks them out itself --
// kPer entries a lane at a time, the hits' places appended in order to a ring,
// a batch staged from the ring. Nothing is counted, scanned or written a pair,
// and what lies behind an opaque tile is never read. Entries and records are
// loaded a step ahead of where they are used, as in blend_kernel. A batch waits
// for kEnough pairs while there are entries left: Gaussians of a tile or less
// hit one entry in sixteen, and a batch costs its barriers and its block tests
// whatever it holds.
// Measured against listing the pairs and blend_kernel over them (us a frame's
// GPU time, the other passes as they then were, MI355X): 4 k Gaussians at 203 x 117 137 -> 114, 100 k at 512 x 512
// 223 -> 190, 1.4 M at 1920 x 1080 924 -> 813, the 60-view walk 15 900 ->
// 14 634, 20 M in eight views 18 000 -> 16 550, 0.9 M at 294 x 262 (many
// entries a strip, most behind an opaque front) 583 -> 427.
constexpr uint32_t kPer = 8;              // entries a lane: one 16-byte word of masks, or two of keys
constexpr uint32_t kFill = kPer * 256u;   // a workgroup's
constexpr uint32_t kRing = kMaxBatch + kFill;
constexpr uint32_t kEnough = kMaxBatch / 2;

template <uint32_t SPLIT, bool kThreshold, bool kMasks>
__global__ void __launch_bounds__(256) blend_entries_kernel(const DView* __restrict__ views,
                                                            const uint32_t* __restrict__ tile_bases, uint32_t nviews,
                                                            EntryWalk entries, const float* __restrict__ records,
                                                            uint32_t depth_mode, float depth_threshold) {
    constexpr uint32_t TILE = 16, kThreads = 256, kWaves = kThreads / 64, kBx = TILE / 8, kSide = TILE / kBlock;
    __shared__ LdsWalk<TILE, kMaxBatch> s;
    __shared__ uint32_t s_ring[kRing];
    __shared__ uint32_t s_hits[kWaves];
    // Tiles in dispatch order (blend_kernel).
    const uint32_t gtile = blockIdx.x / (SPLIT * SPLIT), part = blockIdx.x % (SPLIT * SPLIT);
    const uint32_t v = view_of_tile(tile_bases, nviews, gtile);
    const DView& V = views[v];
    const uint32_t local = gtile - V.tile_base;
    const uint32_t ty = local / V.tiles_x, tx = local - ty * V.tiles_x;
    const uint32_t strip = V.strip_base + ty * V.strips_x + tx / kStripTiles, bit = tx % kStripTiles;
    const uint32_t ox = (tx * SPLIT + part % SPLIT) * TILE, oy = (ty * SPLIT + part / SPLIT) * TILE;
    const uint32_t tid = threadIdx.x;
    uint32_t lx, ly;
    quarter_pixel<TILE>(tid, lx, ly);
    const uint32_t px = ox + lx, py = oy + ly;
    const bool inside = px < V.width && py < V.height;
    const float pxc = (float)px + 0.5f, pyc = (float)py + 0.5f;
    const float x0 = (float)ox + 0.5f, y0 = (float)oy + 0.5f;
    Pixel p;
    p.done = !inside;
    uint32_t last = 0;
    const uint32_t lane = tid & 63u, wave = tid >> 6, row = (tid >> 4) & 3u;
    const uint32_t block = ((wave / kBx) * 2u + (row >> 1)) * kSide + (wave % kBx) * 2u + (row & 1u);
    if (tid == 0) {
        put_padding(s.rec[kMaxBatch]);
    }
    const uint32_t start = entries.ranges[2u * strip], end = entries.ranges[2u * strip + 1u];
    // Fills start at whole words; a lane past the end reads the last word
    // again (its last entries may lie past the end: the buffers are 32 bytes
    // longer than their entries) and finds nothing in it.
    uint32_t pos = start & ~(kPer - 1u);
    const uint32_t last_word = end != 0 ? (end - 1u) & ~(kPer - 1u) : 0u;
    uint4 word = make_uint4(0u, 0u, 0u, 0u), more = word;
    const auto load_entries = [&]() {
        const uint32_t e = min(pos + tid * kPer, last_word);
        if constexpr (kMasks) {
            word = *reinterpret_cast<const uint4*>(entries.masks + e);
        } else {
            word = *reinterpret_cast<const uint4*>(entries.keys + e);
            more = *reinterpret_cast<const uint4*>(entries.keys + e + 4u);
        }
    };
    bool held = start < end;  // entries loaded and not yet taken
    if (held) {
        load_entries();
    }
    uint32_t head = 0, queued = 0;  // the ring's
    uint32_t walked = 0, count = 0;  // the tile's pairs before the staged batch, and in it
    Staged ahead{};
    while (held || queued != 0 || count != 0) {
        if (!__syncthreads_or(!p.done)) {
            break;
        }
        if (tid < count) {
            put(s.rec[tid], ahead);
        }
        if (wave * 64u < count) {
            blocks_met<TILE>(ahead, tid < count, x0, y0, lane, s.meets[wave]);
        }
        const bool refill = held && queued < kMaxBatch;
        const uint32_t first = pos + tid * kPer;
        uint32_t bits = 0, before = 0;
        if (refill) {
            // The lane's entries that are the tile's, bit i for entry first + i.
            if constexpr (kMasks) {
                const uint32_t even = 0x00010001u;
                const uint32_t b = ((word.x >> bit) & even) | ((word.y >> bit) & even) << 2 |
                                   ((word.z >> bit) & even) << 4 | ((word.w >> bit) & even) << 6;
                bits = (b | b >> 15) & 0xFFu;
            } else {
                const uint32_t at = 16u + bit;
                bits = ((word.x >> at) & 1u) | ((word.y >> at) & 1u) << 1 | ((word.z >> at) & 1u) << 2 |
                       ((word.w >> at) & 1u) << 3 | ((more.x >> at) & 1u) << 4 | ((more.y >> at) & 1u) << 5 |
                       ((more.z >> at) & 1u) << 6 | ((more.w >> at) & 1u) << 7;
            }
            const uint32_t to = first < end ? min(end - first, kPer) : 0u;
            const uint32_t from = first < start ? start - first : 0u;
            bits &= ((1u << to) - 1u) & (~0u << from);
            const uint32_t here = (uint32_t)__popc(bits);
            uint32_t incl = here;
            incl += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)incl, 0x111, 0xF, 0xF, false);  // row_shr 1
            incl += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)incl, 0x112, 0xF, 0xF, false);  // row_shr 2
            incl += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)incl, 0x114, 0xF, 0xF, false);  // row_shr 4
            incl += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)incl, 0x118, 0xF, 0xF, false);  // row_shr 8
            incl += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)incl, 0x142, 0xA, 0xF, false);  // row_bcast 15
            incl += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)incl, 0x143, 0xC, 0xF, false);  // row_bcast 31
            before = incl - here;
            if (lane == 63) {
                s_hits[wave] = incl;
            }
        }
        __syncthreads();
        if (refill) {
            uint32_t all = 0;
#pragma unroll
            for (uint32_t w = 0; w < kWaves; ++w) {
                const uint32_t h = s_hits[w];
                before += w < wave ? h : 0u;
                all += h;
            }
            uint32_t at = head + queued + before;
            for (; bits != 0; bits &= bits - 1u, ++at) {
                s_ring[at >= kRing ? at - kRing : at] = first + (uint32_t)__builtin_ctz(bits);
            }
            queued += (uint32_t)__builtin_amdgcn_readfirstlane((int)all);
            pos += kFill;
            held = pos < end;
            if (held) {
                load_entries();
            }
        }
        __syncthreads();
        const uint32_t next = held && queued < kEnough ? 0u : queued < kMaxBatch ? queued : kMaxBatch;
        if (next != 0) {
            uint32_t at = head + min(tid, next - 1u);
            at -= at >= kRing ? kRing : 0u;
            ahead = fetch(records, entries.slots[s_ring[at]]);
            head += next;
            head -= head >= kRing ? kRing : 0u;
            queued -= next;
        }
        if (count != 0 && __ballot(!p.done) != 0) {
            const uint32_t length = expand_list(s, block, lane, count);
            wave_lds_fence();
            const uint32_t last_at = walk_list<kThreshold>(s.rec, s.list[block], length, pxc, pyc, depth_threshold, p);
            if (last_at != ~0u) {
                last = walked + last_at / (uint32_t)sizeof(LdsRecord) + 1u;
            }
        }
        walked += count;
        count = next;
    }
    if (inside) {
        finish_pixel(V, px, py, p, last, depth_mode);
    }
}

// The walk's variants (splat_blend.slang:236-578 with composite, matte and
// traced; athx_targets): the same walk as blend_kernel, and
//   under    an opaque layer under the splats (the view's under_colour and
//            under_depth): a splat at or behind its depth ends the pixel's
//            walk, and the layer takes the light left, as the background
//            would, its depth weighing in the mean (:287-300, 330-333,
//            512-566);
//   matte    the six heaviest Cryptomatte ids of the pixel with their
//            coverage, the layer's own id taking what the walk left
//            (:88-143, 421-423, 526-531);
//   traced   the four heaviest slots, their depths and weights, and what the
//            list left out and what closed the walk (splat_trace.slang).
// Both lists live in registers, every access to them unrolled, so they cost
// no memory; the flags are the frame's, uniform across the launch.
constexpr uint32_t kCryptoSlots = 6;

__device__ inline void crypto_add(uint32_t (&ids)[kCryptoSlots], float (&wts)[kCryptoSlots], uint32_t id,
                                  float weight) {
    if (weight <= 0.0f || id == 0u) {
        return;
    }
    uint32_t lightest = 0;
    float least = wts[0];
    bool merged = false;
#pragma unroll
    for (uint32_t k = 0; k < kCryptoSlots; ++k) {
        // The first rank naming this id takes the weight (splat_blend.slang:101-110).
        const bool same = !merged && ids[k] == id && wts[k] > 0.0f;
        if (same) {
            wts[k] = wts[k] + weight;
            merged = true;
        }
        if (!merged && wts[k] < least) {
            least = wts[k];
            lightest = k;
        }
    }
    if (!merged && weight > least) {
#pragma unroll
        for (uint32_t k = 0; k < kCryptoSlots; ++k) {
            if (k == lightest) {
                ids[k] = id;
                wts[k] = weight;
            }
        }
    }
}

// Ranks by descending weight, ties in list order (an insertion sort's).
template <uint32_t N>
__device__ inline void order_desc(const float (&w)[N], uint32_t (&order)[N]) {
#pragma unroll
    for (uint32_t k = 0; k < N; ++k) {
        uint32_t rank = 0;
#pragma unroll
        for (uint32_t m = 0; m < N; ++m) {
            rank += (w[m] > w[k] || (w[m] == w[k] && m < k)) ? 1u : 0u;
        }
#pragma unroll
        for (uint32_t r = 0; r < N; ++r) {
            if (r == rank) {
                order[r] = k;
            }
        }
    }
}

template <uint32_t N, typename T>
__device__ inline T pick(const T (&a)[N], uint32_t k) {
    T v = a[0];
#pragma unroll
    for (uint32_t m = 1; m < N; ++m) {
        v = m == k ? a[m] : v;
    }
    return v;
}

__device__ inline uint32_t half_of(float v) { return (uint32_t)__builtin_bit_cast(uint16_t, (_Float16)v); }

template <uint32_t TILE>
__global__ void __launch_bounds__(TILE * TILE) blend_ex_kernel(const DView* __restrict__ views,
                                                               const uint32_t* __restrict__ tile_bases,
                                                               uint32_t nviews, uint32_t batch,
                                                               const uint32_t* __restrict__ ranges,
                                                               const uint32_t* __restrict__ pair_slots,
                                                               const float* __restrict__ records,
                                                               const uint32_t* __restrict__ slot_ids,
                                                               uint32_t depth_mode, float depth_threshold) {
    constexpr uint32_t kThreads = TILE * TILE;
    __shared__ LdsBatch s;
    __shared__ uint32_t s_slot[kMaxBatch];
    __shared__ uint32_t s_id[kMaxBatch];
    const uint32_t gtile = blockIdx.x;
    const uint32_t v = view_of_tile(tile_bases, nviews, gtile);
    const DView& V = views[v];
    const uint32_t local = gtile - V.tile_base;
    const uint32_t tx = local % V.tiles_x, ty = local / V.tiles_x;
    const uint32_t tid = threadIdx.x;
    uint32_t lx, ly;
    block_pixel<TILE>(tid, lx, ly);
    const uint32_t px = tx * TILE + lx, py = ty * TILE + ly;
    const bool inside = px < V.width && py < V.height;
    const uint32_t start = ranges[2 * gtile], end = ranges[2 * gtile + 1];
    const float pxc = (float)px + 0.5f, pyc = (float)py + 0.5f;
    const uint32_t pixels = V.width * V.height;
    const size_t pix = inside ? (size_t)py * V.width + px : 0;
    const bool matte = V.crypto != nullptr, traced = V.trace != nullptr;
    const bool under = inside && V.under_colour != nullptr && V.under_depth != nullptr;
    const float under_z = under ? V.under_depth[pix] : 0.0f;
    const bool under_hit = under && under_z > 0.0f;

    float r = 0.0f, g = 0.0f, b = 0.0f, T = 1.0f, dsum = 0.0f, dat = -1.0f;
    uint32_t last = 0;
    uint32_t ids[kCryptoSlots];
    float cw[kCryptoSlots];
#pragma unroll
    for (uint32_t k = 0; k < kCryptoSlots; ++k) {
        ids[k] = 0u;
        cw[k] = 0.0f;
    }
    uint32_t tslot[ATHX_TRACE_SLOTS];
    float tw[ATHX_TRACE_SLOTS];
#pragma unroll
    for (uint32_t k = 0; k < ATHX_TRACE_SLOTS; ++k) {
        tslot[k] = ATHX_TRACE_NONE;
        tw[k] = 0.0f;
    }
    float ttotal = 0.0f, tfloor = 0.0f;
    uint32_t tlightest = 0;
    bool done = !inside;
    const uint32_t lane = tid & 63u;
    const Band band = wave_band<TILE>(V, tx, ty, tid >> 6);
    for (uint32_t first = start; first < end; first += batch) {
        if (!__syncthreads_or(!done)) {
            break;
        }
        const uint32_t count = end - first < batch ? end - first : batch;
        for (uint32_t k = tid; k < count; k += kThreads) {
            const uint32_t slot = pair_slots[first + k];
            stage(s, k, records, slot);
            s_slot[k] = slot;
            if (matte) {
                s_id[k] = slot_ids[slot];
            }
        }
        __syncthreads();
        // A pair the band skips holds nothing for these pixels; the under
        // layer's stop comes at the next pair walked, or none is left to stop:
        // pairs run front to back, so any later one lies behind the layer too.
        for (uint32_t c0 = 0; c0 < count && __ballot(!done) != 0; c0 += 64) {
          for (uint64_t mm = band_mask<TILE>(s, band, c0, count, lane); mm != 0 && !done; mm &= mm - 1ull) {
            const uint32_t j = c0 + (uint32_t)__builtin_ctzll(mm);
            const float4 q = s.xy_cut_op[j];
            const float4 k = s.conic[j];
            if (under_hit && k.w >= under_z) {
                done = true;
                break;
            }
            const float dx = pxc - q.x, dy = pyc - q.y;
            const float power = k.x * dx * dx + k.y * dx * dy + k.z * dy * dy;
            if (power > q.z) {
                continue;
            }
            const float alpha = fminf(0.99f, q.w * blend_exp(power));
            if (alpha < 1.0f / 255.0f) {
                continue;
            }
            const float4 c = s.colour[j];
            const float w = T * alpha;
            if (matte) {
                crypto_add(ids, cw, s_id[j], w);
            }
            if (traced) {
                ttotal = ttotal + w;
                if (w > tfloor) {
                    // TraceList::enter (splat_trace.slang:81-90)
                    const uint32_t slot = s_slot[j];
#pragma unroll
                    for (uint32_t m = 0; m < ATHX_TRACE_SLOTS; ++m) {
                        if (m == tlightest) {
                            tslot[m] = slot;
                            tw[m] = w;
                        }
                    }
                    tlightest = 0;
                    float least = tw[0];
#pragma unroll
                    for (uint32_t m = 1; m < ATHX_TRACE_SLOTS; ++m) {
                        if (tw[m] < least) {
                            least = tw[m];
                            tlightest = m;
                        }
                    }
                    tfloor = least;
                }
            }
            r = r + w * c.x;
            g = g + w * c.y;
            b = b + w * c.z;
            dsum = dsum + w * k.w;
            T = T * (1.0f - alpha);
            if (dat < 0.0f && 1.0f - T >= depth_threshold) {
                dat = k.w;
            }
            last = first - start + j + 1;
            if (T < 1e-4f) {
                done = true;
            }
          }
        }
        __syncthreads();
    }
    if (!inside) {
        return;
    }
    float4 behind = make_float4(V.bg[0], V.bg[1], V.bg[2], V.bg[3]);
    float opaque_z = 0.0f;
    uint32_t opaque_id = 0u;
    if (under_hit) {
        behind = reinterpret_cast<const float4*>(V.under_colour)[pix];
        opaque_z = under_z;
        opaque_id = matte && V.under_crypto ? V.under_crypto[pix] : 0u;
    }
    if (matte) {
        crypto_add(ids, cw, opaque_id, under_hit ? T : 0.0f);
        uint32_t order[kCryptoSlots];
        order_desc<kCryptoSlots>(cw, order);
#pragma unroll
        for (uint32_t layer = 0; layer < kCryptoSlots / 2; ++layer) {
            const uint32_t ka = order[layer * 2], kb = order[layer * 2 + 1];
            const float wa = pick(cw, ka), wb = pick(cw, kb);
            const uint32_t ia = pick(ids, ka), ib = pick(ids, kb);
            reinterpret_cast<float4*>(V.crypto)[(size_t)layer * pixels + pix] =
                make_float4(wa > 0.0f ? __builtin_bit_cast(float, ia) : 0.0f, fmaxf(wa, 0.0f),
                            wb > 0.0f ? __builtin_bit_cast(float, ib) : 0.0f, fmaxf(wb, 0.0f));
        }
    }
    if (traced) {
        const float under_w = under_hit ? T : 0.0f;
        if (!(ttotal > 0.0f) && !(under_w > 0.0f)) {
            V.trace[pix] = ATHX_TRACE_EMPTY;
        } else {
            uint32_t order[ATHX_TRACE_SLOTS];
            order_desc<ATHX_TRACE_SLOTS>(tw, order);
            float held = 0.0f;
            float sorted_w[ATHX_TRACE_SLOTS];
#pragma unroll
            for (uint32_t k = 0; k < ATHX_TRACE_SLOTS; ++k) {
                const float wk = pick(tw, order[k]);
                const uint32_t sk = pick(tslot, order[k]);
                const bool some = wk > 0.0f;
                sorted_w[k] = wk;
                V.trace[(size_t)k * pixels + pix] = some ? sk : ATHX_TRACE_NONE;
                V.trace[(size_t)(ATHX_TRACE_SLOTS + k) * pixels + pix] =
                    some ? __builtin_bit_cast(uint32_t, records[(size_t)sk * kRecordFloats + 2]) : 0u;
                held = held + wk;
            }
#pragma unroll
            for (uint32_t pr = 0; pr < ATHX_TRACE_SLOTS / 2; ++pr) {
                V.trace[(size_t)(ATHX_TRACE_SLOTS * 2 + pr) * pixels + pix] =
                    half_of(sorted_w[pr * 2]) | (half_of(sorted_w[pr * 2 + 1]) << 16);
            }
            V.trace[(size_t)(ATHX_TRACE_WORDS - 1) * pixels + pix] =
                half_of(fmaxf(ttotal - held, 0.0f)) | (half_of(fmaxf(under_w, 0.0f)) << 16);
        }
    }
    const float coverage = 1.0f - T;
    if (under_hit) {
        dsum = dsum + T * opaque_z;
        if (dat < 0.0f) {
            dat = opaque_z;
        }
    }
    const float total = under_hit ? 1.0f : coverage;
    float4 out;
    out.x = r + T * behind.x;
    out.y = g + T * behind.y;
    out.z = b + T * behind.z;
    out.w = coverage + T * behind.w;
    reinterpret_cast<float4*>(V.colour)[pix] = out;
    if (V.depth) {
        V.depth[pix] = depth_mode == 0 ? (total > 1e-6f ? dsum / total : 0.0f) : fmaxf(dat, 0.0f);
    }
    if (V.final_t) {
        V.final_t[pix] = T;
    }
    if (V.last) {
        V.last[pix] = last;
    }
}

// What each splat gave the last frame (splat_blend.slang:36-48, 364-398):
// the same walk as blend_kernel -- the same pairs, records, arithmetic and
// early stop -- counting at each pair's slot, with integer atomics (so in
// any order the same sum): mode 1 the blend weight T alpha in 1/4096 of a
// pixel, rounded; mode 4 NeuralFit's colour gradient, the weight times
// dL/dC (the view's dl_dcolour) in 1/256, each channel rounded down or up by
// color.slang's hash01 of (pixel, channel, slot) so that steps below one are
// kept on average, and the weight itself in 1/256 as a fourth word.
__device__ inline float hash01(uint32_t v) {
    const uint32_t state = v * 747796405u + 2891336453u;
    const uint32_t word = ((state >> ((state >> 28u) + 4u)) ^ state) * 277803737u;
    return (float)((word >> 22u) ^ word) / 4294967295.0f;
}

template <uint32_t TILE, uint32_t MODE>
__global__ void __launch_bounds__(TILE * TILE) contribution_kernel(const DView* __restrict__ views,
                                                                   const uint32_t* __restrict__ tile_bases,
                                                                   uint32_t nviews, uint32_t batch,
                                                                   const uint32_t* __restrict__ ranges,
                                                                   const uint32_t* __restrict__ pair_slots,
                                                                   const float* __restrict__ records,
                                                                   uint32_t* __restrict__ contribution) {
    constexpr uint32_t kThreads = TILE * TILE;
    __shared__ LdsBatch s;
    __shared__ uint32_t s_slot[kMaxBatch];
    const uint32_t gtile = blockIdx.x;
    const uint32_t v = view_of_tile(tile_bases, nviews, gtile);
    const DView& V = views[v];
    const uint32_t local = gtile - V.tile_base;
    const uint32_t tx = local % V.tiles_x, ty = local / V.tiles_x;
    const uint32_t tid = threadIdx.x;
    uint32_t lx, ly;
    block_pixel<TILE>(tid, lx, ly);
    const uint32_t px = tx * TILE + lx, py = ty * TILE + ly;
    const bool inside = px < V.width && py < V.height;
    const uint32_t start = ranges[2 * gtile], end = ranges[2 * gtile + 1];
    const float pxc = (float)px + 0.5f, pyc = (float)py + 0.5f;
    const uint32_t at = inside ? py * V.width + px : 0u;
    // The per-pixel input: mode 2 the pixel drawn whole, mode 3 the mask,
    // mode 4 dL/dC.
    float4 dl = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
    if ((MODE == 2 || MODE == 4) && inside) {
        dl = reinterpret_cast<const float4*>(V.dl_dcolour)[at];
    } else if (MODE == 3 && inside) {
        dl.x = fminf(fmaxf(V.dl_dcolour[at], 0.0f), 1.0f);
    }
    float T = 1.0f;
    float r = 0.0f, g = 0.0f, b = 0.0f;
    bool done = !inside;
    const uint32_t lane = tid & 63u;
    const Band band = wave_band<TILE>(V, tx, ty, tid >> 6);
    for (uint32_t first = start; first < end; first += batch) {
        if (!__syncthreads_or(!done)) {
            break;
        }
        const uint32_t count = end - first < batch ? end - first : batch;
        for (uint32_t k = tid; k < count; k += kThreads) {
            const uint32_t slot = pair_slots[first + k];
            stage(s, k, records, slot);
            s_slot[k] = slot;
        }
        __syncthreads();
        for (uint32_t c0 = 0; c0 < count && __ballot(!done) != 0; c0 += 64) {
          for (uint64_t mm = band_mask<TILE>(s, band, c0, count, lane); mm != 0 && !done; mm &= mm - 1ull) {
            const uint32_t j = c0 + (uint32_t)__builtin_ctzll(mm);
            const float4 q = s.xy_cut_op[j];
            const float4 k = s.conic[j];
            const float dx = pxc - q.x, dy = pyc - q.y;
            const float power = k.x * dx * dx + k.y * dx * dy + k.z * dy * dy;
            if (power > q.z) {
                continue;
            }
            const float alpha = fminf(0.99f, q.w * blend_exp(power));
            if (alpha < 1.0f / 255.0f) {
                continue;
            }
            const float w = T * alpha;
            const uint32_t slot = s_slot[j];
            if (MODE == 1) {
                atomicAdd(&contribution[slot], (uint32_t)(w * 4096.0f + 0.5f));
            } else if (MODE == 2) {
                // The pixel without this splat: what is behind it is
                // (C - P) / T' with P the walk once it is in, T' the
                // transmittance after it; the change is w (c - behind).
                const float4 c = s.colour[j];
                const float after = T * (1.0f - alpha);
                const float keep = fmaxf(after, 1.0e-4f);
                const float er = w * (c.x - (dl.x - (r + w * c.x)) / keep);
                const float eg = w * (c.y - (dl.y - (g + w * c.y)) / keep);
                const float eb = w * (c.z - (dl.z - (b + w * c.z)) / keep);
                const float e2 = fminf(er * er + eg * eg + eb * eb, 1.0f);
                const uint32_t add = (uint32_t)(e2 * 16777216.0f + 0.5f);
                const uint32_t before = atomicAdd(&contribution[(size_t)slot * 2], add);
                if (before + add < before) {
                    atomicAdd(&contribution[(size_t)slot * 2 + 1], 1u);
                }
                r = r + w * c.x;
                g = g + w * c.y;
                b = b + w * c.z;
            } else if (MODE == 3) {
                const uint32_t seen = (uint32_t)(w * 1024.0f + 0.5f);
                if (seen != 0u) {
                    atomicAdd(&contribution[(size_t)slot * 2 + 1], seen);
                    const uint32_t within = (uint32_t)(w * dl.x * 1024.0f + 0.5f);
                    if (within != 0u) {
                        atomicAdd(&contribution[(size_t)slot * 2], within);
                    }
                }
            } else {
                const float g[3] = {w * dl.x * 256.0f, w * dl.y * 256.0f, w * dl.z * 256.0f};
                for (uint32_t c = 0; c < 3; ++c) {
                    const int step = (int)floorf(g[c] + hash01((at * 3u + c) ^ (slot * 2654435761u)));
                    if (step != 0) {
                        atomicAdd(&contribution[(size_t)slot * 4 + c], (uint32_t)step);
                    }
                }
                atomicAdd(&contribution[(size_t)slot * 4 + 3], (uint32_t)(w * 256.0f + 0.5f));
            }
            T = T * (1.0f - alpha);
            if (T < 1e-4f) {
                done = true;
            }
          }
        }
        __syncthreads();
    }
}

__device__ inline float as_float(uint32_t u) { return __builtin_bit_cast(float, u); }
__device__ inline uint32_t as_uint(float f) { return __builtin_bit_cast(uint32_t, f); }

// Nine sums over each row of 16 lanes at once, the rows apart, every lane of
// the row active: the DPP adds that halve a value leave the sum in both
// halves, so where two values are at hand the second's add is written over the
// first's in half of the row's banks of four lanes (the bank mask), and one
// register goes on holding both. Bank k of the two registers ends with the
// sums 2 of its four lanes share: x0 those of v[0], v[2], v[4], v[6] in banks
// 0 to 3, x1 those of v[1], v[3], v[5], v[7], x2 v[8]'s in every lane: 20 VALU
// operations for four rows, where whole-wavefront sums of the nine took 39
// for one Gaussian.
template <int CTRL>
__device__ inline float dpp_sum(float x) {
    return x + as_float((uint32_t)__builtin_amdgcn_update_dpp(0, (int)as_uint(x), CTRL, 0xF, 0xF, true));
}
// dpp_sum(x) in the banks of BANKS, `keep` in the others.
template <int CTRL, int BANKS>
__device__ inline float dpp_sum_banks(float x, float keep) {
    const float sum = x + as_float((uint32_t)__builtin_amdgcn_update_dpp(0, (int)as_uint(x), CTRL, 0xF, 0xF, true));
    return as_float((uint32_t)__builtin_amdgcn_update_dpp((int)as_uint(keep), (int)as_uint(sum), 0xE4, 0xF, BANKS, false));
}

__device__ inline void row_sum9(const float (&v)[9], float& x0, float& x1, float& x2) {
    constexpr int kRor8 = 0x128, kHalfMirror = 0x141, kQuad2301 = 0x4E, kQuad1032 = 0xB1;
    // Lanes 8-15 (banks 2, 3) go on with v[k + 4].
    const float a0 = dpp_sum_banks<kRor8, 0xC>(v[4], dpp_sum<kRor8>(v[0]));
    const float a1 = dpp_sum_banks<kRor8, 0xC>(v[5], dpp_sum<kRor8>(v[1]));
    const float a2 = dpp_sum_banks<kRor8, 0xC>(v[6], dpp_sum<kRor8>(v[2]));
    const float a3 = dpp_sum_banks<kRor8, 0xC>(v[7], dpp_sum<kRor8>(v[3]));
    // Within each half, lanes 4-7 (banks 1, 3) with the value two on.
    x0 = dpp_sum_banks<kHalfMirror, 0xA>(a2, dpp_sum<kHalfMirror>(a0));
    x1 = dpp_sum_banks<kHalfMirror, 0xA>(a3, dpp_sum<kHalfMirror>(a1));
    x0 = dpp_sum<kQuad1032>(dpp_sum<kQuad2301>(x0));
    x1 = dpp_sum<kQuad1032>(dpp_sum<kQuad2301>(x1));
    x2 = dpp_sum<kQuad1032>(dpp_sum<kQuad2301>(dpp_sum<kHalfMirror>(dpp_sum<kRor8>(v[8]))));
}

// Gaussians staged at a time by the adjoint. Every (block, Gaussian) pair of a
// batch has nine words of LDS for its sums, which no other row writes, since
// an LDS float add takes some 3 cycles a lane of the CU's LDS pipe (measured:
// 109 for the 36 lanes of a step, against 7 for a plain write of them; with
// the adds the walk was bound by that pipe at 95 %): the batch is what leaves
// room for four workgroups a CU. Measured against the
// walk of 8 x 8 pixels a step with whole-wavefront sums (us a launch, MI355X):
// 100 k Gaussians at 512 x 512 293 -> 150, 1.4 M at 1920 x 1080 702 -> 501.
// Bound by the VALU's issue (0.51 of its rate) with the LDS pipe serving
// accesses in 0.28 of the clocks. Tiles in dispatch order: banded over the XCDs
// the first took 183 where it took 140 (the middle bands hold most of the work),
// the second the same.
template <uint32_t TILE>
constexpr uint32_t back_batch() {
    return TILE == 8 ? 32u : 56u;
}

template <uint32_t TILE, uint32_t SPLIT>
__global__ void __launch_bounds__(TILE * TILE) blend_backward_kernel(
    const DView* __restrict__ views, const uint32_t* __restrict__ tile_bases, uint32_t nviews,
    const uint32_t* __restrict__ ranges, const uint32_t* __restrict__ pair_slots, const float* __restrict__ records,
    float* __restrict__ grad2d) {
    constexpr uint32_t kThreads = TILE * TILE, kWaves = kThreads / 64;
    constexpr uint32_t kBx = TILE / 8, kSide = TILE / kBlock, kBlocks = kSide * kSide;
    constexpr uint32_t batch = back_batch<TILE>();
    constexpr uint32_t kOut = batch * kGrad2d;  // a block's words
    static_assert(batch <= 64, "a lane a Gaussian, one ballot");
    __shared__ LdsWalk<TILE, batch> s;
    __shared__ uint32_t s_slot[2][64];
    __shared__ alignas(16) float s_out[kBlocks * kOut];
    __shared__ float s_sum[kOut];
    __shared__ uint32_t s_max_last;
    const uint32_t gtile = blockIdx.x / (SPLIT * SPLIT), part = blockIdx.x % (SPLIT * SPLIT);
    const uint32_t v = view_of_tile(tile_bases, nviews, gtile);
    const DView& V = views[v];
    const uint32_t local = gtile - V.tile_base;
    const uint32_t ox = ((local % V.tiles_x) * SPLIT + part % SPLIT) * TILE;
    const uint32_t oy = ((local / V.tiles_x) * SPLIT + part / SPLIT) * TILE;
    const uint32_t tid = threadIdx.x;
    const uint32_t lane = tid & 63u, wave = tid >> 6, row = (tid >> 4) & 3u, q = tid & 15u;
    uint32_t lx, ly;
    quarter_pixel<TILE>(tid, lx, ly);
    const uint32_t px = ox + lx, py = oy + ly;
    const bool inside = px < V.width && py < V.height;
    const uint32_t start = ranges[2 * gtile];
    const uint32_t tile_pairs = ranges[2 * gtile + 1] - start;
    const float pxc = (float)px + 0.5f, pyc = (float)py + 0.5f;
    const float x0 = (float)ox + 0.5f, y0 = (float)oy + 0.5f;
    const size_t pix = inside ? (size_t)py * V.width + px : 0;
    const uint32_t block = ((wave / kBx) * 2u + (row >> 1)) * kSide + (wave % kBx) * 2u + (row & 1u);

    float T = 1.0f;
    uint32_t last = 0;
    float gr = 0.0f, gg = 0.0f, gb = 0.0f, ga = 0.0f;
    if (inside) {
        T = V.final_t[pix];
        // A walk never reads past its tile's pairs; the clamp keeps a stale
        // `last` from reading past them either.
        last = min(V.last[pix], tile_pairs);
        const float4 gc = reinterpret_cast<const float4*>(V.dl_dcolour)[pix];
        gr = gc.x; gg = gc.y; gb = gc.z; ga = gc.w;
    }
    // A pixel of the wavefront's has a dL/dC that is not finite.
    const bool infinite = __ballot(!(fabsf(gr) + fabsf(gg) + fabsf(gb) < INFINITY)) != 0;
    // dL/dC . (the colour of everything behind the current Gaussian, as seen
    // from just in front of it): the background, then each Gaussian over it.
    float br = V.bg[0], bgc = V.bg[1], bb = V.bg[2];
    // d(alpha out)/d(alpha_k) = T_N (1 - bg.a) / (1 - alpha_k).
    const float ga_scale = ga * T * (1.0f - V.bg[3]);
    if (tid == 0) {
        s_max_last = 0;
    }
    __syncthreads();
    // A row walks only the pairs below its own pixels' furthest.
    const uint32_t row_last = row_max(last);
    if (q == 0 && row_last != 0) {
        atomicMax(&s_max_last, row_last);
    }
    __syncthreads();
    const uint32_t max_last = s_max_last;
    // The lanes that write a row's sums: lanes 0 and 1 of each bank x0's and
    // x1's, lane 2 of the first x2's; their words within a Gaussian's: u, u dx,
    // u dx dx, u dx dy, u dy, u dy dy, then w dL/d(r, g, b).
    const bool writes = (q & 3u) < 2u || q == 2u;
    float* const out = s_out + block * kOut + (q == 2u ? 8u : (q >> 2) * 2u + (q & 1u));
    // The staging runs a batch ahead of the walk, as in the forward blend:
    // while a batch is walked each lane reads its record of the next (lower)
    // batch and its slot of the one after. Every wavefront reads them all, since
    // each tests rows of blocks of its own. The reads are unconditional, at
    // in-bounds pairs of the tile (the tile has max_last pairs or more).
    const auto pair_of = [&](uint32_t hi_b) {
        const uint32_t lo_b = hi_b > batch ? hi_b - batch : 0u;
        const uint32_t k = lo_b + lane;
        return start + (k < hi_b ? k : (hi_b != 0u ? hi_b - 1u : 0u));
    };
    uint32_t slot_now = 0, slot_ahead = 0;
    Staged rec_now{};
    if (max_last > 0) {
        slot_now = pair_slots[pair_of(max_last)];
        rec_now = fetch(records, slot_now);
        slot_ahead = pair_slots[pair_of(max_last > batch ? max_last - batch : 0u)];
    }
    const auto clear_out = [&]() {
        for (uint32_t k = tid; k < kBlocks * kOut / 4u; k += kThreads) {
            reinterpret_cast<float4*>(s_out)[k] = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
        }
    };
    static_assert(kBlocks * kOut % 4u == 0, "cleared by 16-byte words");
    clear_out();
    uint32_t turn = 0;
    for (uint32_t hi = max_last; hi > 0; turn ^= 1u) {
        const uint32_t lo = hi > batch ? hi - batch : 0;
        const uint32_t count = hi - lo;
        if (wave == 0 && lane < count) {
            s_slot[turn][lane] = slot_now;
            put(s.rec[lane], rec_now);
        }
        for (uint32_t slice = wave; slice < kSide; slice += kWaves) {
            blocks_met<TILE, 1>(rec_now, lane < count, x0, y0, lane, s.meets[0], slice);
        }
        __syncthreads();
        // The next batch is [lo - batch, lo); the one after it ends where that
        // one starts.
        slot_now = slot_ahead;
        rec_now = fetch(records, slot_ahead);
        slot_ahead = pair_slots[pair_of(lo > batch ? lo - batch : 0u)];
        // Back to front over the row's Gaussians below its furthest pair.
        const uint32_t length = expand_list(s, block, lane, bytes_below(row_last, lo, count, 1u));
        wave_lds_fence();
        const uint16_t* list = s.list[block];
        const uint32_t last_at = bytes_below(last, lo, count, (uint32_t)sizeof(LdsRecord));
        for (uint32_t i = length; i-- != 0;) {
            const uint32_t at = list[i];
            const LdsRecord& k = *reinterpret_cast<const LdsRecord*>(reinterpret_cast<const char*>(s.rec) + at);
            const float4 ka = k.a, kb = k.b, kc = k.c;
            const float dx = pxc - ka.x, dy = pyc - ka.y;
            const float x = ka.z * dx * dx + ka.w * dx * dy + kb.x * dy * dy;
            const float e = blend_exp_of(x);
            const float raw = kb.z * e;
            const float clamped = fminf(0.99f, raw);
            const bool took = (at < last_at) & !(x < kb.y) & !(clamped < 1.0f / 255.0f);
            // A lane that did not take the Gaussian goes through with an alpha
            // of 0 (T and the colour behind it unchanged, every term 0).
            const float alpha = took ? clamped : 0.0f;
            const float one_minus = 1.0f - alpha;
            // 1 / (1 - alpha), alpha <= 0.99: the hardware reciprocal and one
            // Newton step (within an ulp or so of the quotient), where an IEEE
            // divide takes a dozen operations. The adjoint answers to finite
            // differences at 1e-3, not to bits.
            float inv = __builtin_amdgcn_rcpf(one_minus);
            inv = __builtin_fmaf(inv, __builtin_fmaf(-one_minus, inv, 1.0f), inv);
            T = T * inv;
            const float or_ = took ? kc.x - br : 0.0f, og = took ? kc.y - bgc : 0.0f, ob = took ? kc.z - bb : 0.0f;
            const float over = __builtin_fmaf(or_, gr, __builtin_fmaf(og, gg, ob * gb));
            const float dl_dalpha = __builtin_fmaf(T, over, ga_scale * inv);
            br = __builtin_fmaf(alpha, or_, br);
            bgc = __builtin_fmaf(alpha, og, bgc);
            bb = __builtin_fmaf(alpha, ob, bb);
            // Zeroed by selection: an infinite or NaN dL/dC of a pixel reaches
            // the Gaussians that the pixel took and no others of its block.
            const float w = alpha * T;
            const float u = took & !(raw > 0.99f) ? dl_dalpha * e : 0.0f;
            float wr = w * gr, wg = w * gg, wb = w * gb;
            if (infinite) {
                // (Kept a branch: the three selects in every step are 3 % of
                // the walk, 513 us against 501 at 1920 x 1080.)
                asm volatile("" : "+v"(wr), "+v"(wg), "+v"(wb));
                wr = took ? wr : 0.0f;
                wg = took ? wg : 0.0f;
                wb = took ? wb : 0.0f;
            }
            const float ux = u * dx, uy = u * dy;
            // -2 x's derivatives along dx and dy, where a thin Gaussian's
            // terms cancel: taken a pixel, not from the pixels' sums.
            const float hx = __builtin_fmaf(-ka.w, dy, -2.0f * (ka.z * dx));
            const float hy = __builtin_fmaf(-ka.w, dx, -2.0f * (kb.x * dy));
            const float sums[9] = {u, u * hx, ux * dx, ux * dy, u * hy, uy * dy, wr, wg, wb};
            float s0, s1, s2;
            row_sum9(sums, s0, s1, s2);
            if (writes) {
                // (at is 48 bytes a Gaussian, its words 36.)
                static_assert(sizeof(LdsRecord) * 3 == kGrad2d * sizeof(float) * 4, "48 to 36");
                *reinterpret_cast<float*>(reinterpret_cast<char*>(out) + (at - (at >> 2))) =
                    q == 2u ? s2 : (q & 1u) ? s1 : s0;
            }
        }
        __syncthreads();
        // Each Gaussian's words summed over the tile's blocks.
        for (uint32_t k = tid; k < count * kGrad2d; k += kThreads) {
            float sum = 0.0f;
#pragma unroll 8
            for (uint32_t m = 0; m < kBlocks; ++m) {
                sum += s_out[m * kOut + k];
            }
            s_sum[k] = sum;
        }
        __syncthreads();
        clear_out();
        // The exponent x = -(a dx dx + 2 b dx dy + c dy dy) / 2 taken apart, in
        // place: to the centre, conic and alpha (kGrad2d's order).
        for (uint32_t k = tid; k < count; k += kThreads) {
            float* G = s_sum + k * kGrad2d;
            const LdsRecord& p = s.rec[k];
            const float op = p.b.z;
            const float u = G[0], ux = G[1], uxx = G[2], uxy = G[3], uy = G[4], uyy = G[5];
            G[0] = op * ux;
            G[1] = op * uy;
            G[2] = -0.5f * op * uxx;
            G[3] = -op * uxy;
            G[4] = -0.5f * op * uyy;
            G[5] = u;
        }
        __syncthreads();
        for (uint32_t k = tid; k < count * kGrad2d; k += kThreads) {
            const uint32_t j = k / kGrad2d;
            const float g = s_sum[k];
            if (g != 0.0f) {
                atomicAdd(&grad2d[(size_t)s_slot[turn][j] * kGrad2d + (k - j * kGrad2d)], g);
            }
        }
        hi = lo;
    }
}

template <uint32_t TILE, uint32_t SPLIT>
hipError_t blend_for(const DView* views, const uint32_t* tile_bases, uint32_t nviews, uint32_t tiles, uint32_t batch,
                     const uint32_t* ranges, const uint32_t* slots, const float* records, uint32_t depth_mode,
                     float depth_threshold, hipStream_t s) {
    using Kernel = void (*)(const DView*, const uint32_t*, uint32_t, uint32_t, const uint32_t*, const uint32_t*,
                            const float*, uint32_t, float);
    const bool piped = batch <= TILE * TILE, threshold = depth_mode != 0;
    const Kernel kernel =
        piped ? (threshold ? blend_kernel<TILE, SPLIT, true, true> : blend_kernel<TILE, SPLIT, true, false>)
              : (threshold ? blend_kernel<TILE, SPLIT, false, true> : blend_kernel<TILE, SPLIT, false, false>);
    hipLaunchKernelGGL(kernel, dim3(tiles * SPLIT * SPLIT), dim3(TILE * TILE), 0, s, views, tile_bases, nviews, batch,
                       ranges, slots, records, depth_mode, depth_threshold);
    return hipGetLastError();
}

template <uint32_t TILE, uint32_t SPLIT>
hipError_t blend_backward_for(const DView* views, const uint32_t* tile_bases, uint32_t nviews, uint32_t tiles,
                              const uint32_t* ranges, const uint32_t* slots, const float* records, float* grad2d,
                              hipStream_t s) {
    hipLaunchKernelGGL((blend_backward_kernel<TILE, SPLIT>), dim3(tiles * SPLIT * SPLIT), dim3(TILE * TILE), 0, s,
                       views, tile_bases, nviews, ranges, slots, records, grad2d);
    return hipGetLastError();
}

}  // namespace

hipError_t launch_blend(const DView* views_dev, const uint32_t* tile_bases, uint32_t nviews, uint32_t total_tiles,
                        uint32_t tile, uint32_t batch, const uint32_t* ranges, const uint32_t* pair_slots,
                        const float* records, uint32_t depth_mode, float depth_threshold, hipStream_t s,
                        bool variants, const uint32_t* slot_ids) {
    if (total_tiles == 0) {
        return hipSuccess;
    }
    if (batch == 0 || batch > kMaxBatch) {
        return hipErrorInvalidValue;
    }
    if (variants) {
        using Kernel = void (*)(const DView*, const uint32_t*, uint32_t, uint32_t, const uint32_t*, const uint32_t*,
                                const float*, const uint32_t*, uint32_t, float);
        const Kernel k = tile == 8 ? blend_ex_kernel<8> : tile == 16 ? blend_ex_kernel<16> : tile == 32 ? blend_ex_kernel<32>
                                                                                                          : nullptr;
        if (!k) {
            return hipErrorInvalidValue;
        }
        hipLaunchKernelGGL(k, dim3(total_tiles), dim3(tile * tile), 0, s, views_dev, tile_bases, nviews, batch, ranges,
                           pair_slots, records, slot_ids, depth_mode, depth_threshold);
        return hipGetLastError();
    }
    switch (tile) {
    case 8:
        return blend_for<8, 1>(views_dev, tile_bases, nviews, total_tiles, batch, ranges, pair_slots, records, depth_mode,
                            depth_threshold, s);
    case 16:
        return blend_for<16, 1>(views_dev, tile_bases, nviews, total_tiles, batch, ranges, pair_slots, records,
                             depth_mode, depth_threshold, s);
    case 32:
        return blend_for<16, 2>(views_dev, tile_bases, nviews, total_tiles, batch, ranges, pair_slots, records,
                             depth_mode, depth_threshold, s);
    default:
        return hipErrorInvalidValue;
    }
}

hipError_t launch_blend_entries(const DView* views_dev, const uint32_t* tile_bases, uint32_t nviews,
                                uint32_t total_tiles, uint32_t tile, const EntryWalk& entries, const float* records,
                                uint32_t depth_mode, float depth_threshold, hipStream_t s) {
    if (total_tiles == 0) {
        return hipSuccess;
    }
    if (tile != 16 && tile != 32) {
        return hipErrorInvalidValue;
    }
    using Kernel = void (*)(const DView*, const uint32_t*, uint32_t, EntryWalk, const float*, uint32_t, float);
    const bool threshold = depth_mode != 0;
    const Kernel kernels[2][2][2] = {
        {{blend_entries_kernel<1, false, false>, blend_entries_kernel<1, false, true>},
         {blend_entries_kernel<1, true, false>, blend_entries_kernel<1, true, true>}},
        {{blend_entries_kernel<2, false, false>, blend_entries_kernel<2, false, true>},
         {blend_entries_kernel<2, true, false>, blend_entries_kernel<2, true, true>}}};
    const Kernel kernel = kernels[tile == 32 ? 1 : 0][threshold ? 1 : 0][entries.masks ? 1 : 0];
    hipLaunchKernelGGL(kernel, dim3(total_tiles * (tile == 32 ? 4u : 1u)), dim3(256), 0, s, views_dev, tile_bases,
                       nviews, entries, records, depth_mode, depth_threshold);
    return hipGetLastError();
}

template <uint32_t TILE>
static hipError_t contribution_for(const DView* views, const uint32_t* tile_bases, uint32_t nviews, uint32_t tiles,
                            uint32_t batch, const uint32_t* ranges, const uint32_t* slots, const float* records,
                            uint32_t mode, uint32_t* out, hipStream_t s) {
    if (mode == 1) {
        hipLaunchKernelGGL((contribution_kernel<TILE, 1>), dim3(tiles), dim3(TILE * TILE), 0, s, views, tile_bases,
                           nviews, batch, ranges, slots, records, out);
    } else if (mode == 2) {
        hipLaunchKernelGGL((contribution_kernel<TILE, 2>), dim3(tiles), dim3(TILE * TILE), 0, s, views, tile_bases,
                           nviews, batch, ranges, slots, records, out);
    } else if (mode == 3) {
        hipLaunchKernelGGL((contribution_kernel<TILE, 3>), dim3(tiles), dim3(TILE * TILE), 0, s, views, tile_bases,
                           nviews, batch, ranges, slots, records, out);
    } else {
        hipLaunchKernelGGL((contribution_kernel<TILE, 4>), dim3(tiles), dim3(TILE * TILE), 0, s, views, tile_bases,
                           nviews, batch, ranges, slots, records, out);
    }
    return hipGetLastError();
}

hipError_t launch_contribution(const DView* views_dev, const uint32_t* tile_bases, uint32_t nviews,
                               uint32_t total_tiles, uint32_t tile, uint32_t batch, const uint32_t* ranges,
                               const uint32_t* pair_slots, const float* records, uint32_t mode, uint32_t* out,
                               hipStream_t s) {
    if (total_tiles == 0) {
        return hipSuccess;
    }
    if (batch == 0 || batch > kMaxBatch || mode < 1 || mode > 4) {
        return hipErrorInvalidValue;
    }
    switch (tile) {
    case 8:
        return contribution_for<8>(views_dev, tile_bases, nviews, total_tiles, batch, ranges, pair_slots, records,
                                   mode, out, s);
    case 16:
        return contribution_for<16>(views_dev, tile_bases, nviews, total_tiles, batch, ranges, pair_slots, records,
                                    mode, out, s);
    case 32:
        return contribution_for<32>(views_dev, tile_bases, nviews, total_tiles, batch, ranges, pair_slots, records,
                                    mode, out, s);
    default:
        return hipErrorInvalidValue;
    }
}

hipError_t launch_blend_backward(const DView* views_dev, const uint32_t* tile_bases, uint32_t nviews,
                                 uint32_t total_tiles, uint32_t tile, const uint32_t* ranges,
                                 const uint32_t* pair_slots, const float* records, float* grad2d, hipStream_t s) {
    if (total_tiles == 0) {
        return hipSuccess;
    }
    switch (tile) {
    case 8:
        return blend_backward_for<8, 1>(views_dev, tile_bases, nviews, total_tiles, ranges, pair_slots, records,
                                     grad2d, s);
    case 16:
        return blend_backward_for<16, 1>(views_dev, tile_bases, nviews, total_tiles, ranges, pair_slots, records,
                                      grad2d, s);
    case 32:
        return blend_backward_for<16, 2>(views_dev, tile_bases, nviews, total_tiles, ranges, pair_slots, records,
                                      grad2d, s);
    default:
        return hipErrorInvalidValue;
    }
}

}  // namespace athx
