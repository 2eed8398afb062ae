// Per-tile compositing and its derivative (train_forward.comp:38-100,
// train_backward.glsl:78-158). The lists are per tile (16x16 by default, or
// 8x8, 32x8 or 32x32); the pixels are worked in 8x8 blocks, one workgroup of one
// wave64 per block, lane l holding pixel (l & 7, l >> 3). A block reads its
// tile's list in batches of 64 entries: each lane stages one splat with the
// block's pixels it can touch already worked out, and only the splats that
// can touch a pixel of the block are kept, packed in list order. A block
// stops when its own pixels are done, with no barrier across the tile.
//
// Staging: for each splat, an 8-bit column mask and an 8-bit row mask of the
// pixels inside both its extent box (splat_pixels, train_types.glsl:43-48) and
// its radius square (the first test of splat_at): a pixel is a candidate iff
// its column and row bits are set. The masks are computed with the same float
// operations as the per-pixel tests they replace, so the set is the same.
// A wave skips a splat none of its lanes is a candidate for; otherwise every
// lane evaluates the Gaussian without branches and the result is selected.
// Every list shape has the same 8x8 blocks, so images and sums do not depend
// on the shape.
//
// Backward: for each splat the 12 non-zero of the 14 per-pixel sums are
// reduced over the wave by a transposed butterfly in which the steps halve the
// values a lane carries where they can: partner lanes l ^ 32 and l ^ 16
// through the permlane swaps, l ^ 15 and l ^ 7 through DPP row and half-row
// mirrors, then l ^ 2 and l ^ 1 through quad permutations. Twelve lanes end
// with one total each, which goes to global memory with one atomic: 64-bit
// fixed point (each wave total quantised, so the integer sums are the same in
// any order) or float.
#include "device.hpp"
#include "kernels.hpp"
#include "blockscan.hpp"
#include "tiles.hpp"

namespace vsplat {

namespace {

struct Staged {
  float qx, qy, qz, o;
  float r, g, b;
  uint32_t entry; // the splat's index in the tile's list
  float cx, cy;
  uint32_t cols, rows; // the block's columns (bits 0-7) and rows (bits 16-23) the splat can touch; rows unused
};
static_assert(sizeof(Staged) == 48, "48-byte staged splat");

// Splats the forward pass evaluates together before it blends them in turn: the
// evaluations do not depend on each other, so one wait for LDS and one branch
// serve four, and nothing but the blending is a chain. At 1M Gaussians and
// 1280x720 (32x32 lists) the kernel took 127.7 us one splat at a time with its
// loads waited for batch by batch (ListWalk), and takes 91.7 in groups of four,
// 92.6 in twos and 93.8 in eights; at 40k Gaussians and 333x251, where 1344
// blocks leave most of the chip idle and latency is all, 138.9 and 98.0 us
// (103.5 and 98.9). The backward pass evaluates in the same groups: 189.7 us one
// by one, 180.8 in twos, 178.8 in fours at 1M.
constexpr uint32_t kGroup = 4;
constexpr uint32_t kBlock = 64; // pixels of an 8x8 block, threads of its workgroup, entries per batch

struct BlockGeometry {
  uint32_t x0, y0, x1, y1;
  uint32_t block; // the block's number in its tile (its bit in the entries' block masks)
  bool reach;     // lists of tiles larger than the block: stage only the splats whose ellipse reaches it
};

// Workgroups are dealt to the chip's eight XCDs in turn (workgroup h runs on
// XCD h % 8), and each XCD has its own L2. Launch index h works 8x8 block q of
// list tile t such that a tile's blocks all run on one XCD, one after another,
// and read its list through one L2, while the tiles are still dealt over the
// XCDs in turn (XCD x works tiles x, x + 8, x + 16, ...): with u = h / 8,
// t = (u / blocks) * 8 + h % 8 and q = u % blocks, the tile's blocks row-major
// (TW / 8 across). A grid of raster_blocks(tiles) covers every (t, q) once;
// the blocks of the tiles past the last (t >= tiles) start below the image.
template <uint32_t TW, uint32_t TH>
__device__ __forceinline__ BlockGeometry block_geometry(uint32_t h, uint32_t gridW, uint32_t width, uint32_t height,
                                                        uint32_t &tile) {
  constexpr uint32_t kAcross = TW / 8u, kPerTile = (TW / 8u) * (TH / 8u);
  const uint32_t u = h / kRasterXcds;
  tile = (u / kPerTile) * kRasterXcds + h % kRasterXcds;
  const uint32_t q = u % kPerTile;
  const uint32_t x0 = (tile % gridW) * TW + (q % kAcross) * 8u, y0 = (tile / gridW) * TH + (q / kAcross) * 8u;
  return {x0, y0, x0 + 8u < width ? x0 + 8u : width, y0 + 8u < height ? y0 + 8u : height, q, TW * TH > 64u};
}

// Heaviest first: a block's work (entries) as one of kOrderKeys keys, 8 per
// octave (the exponent and the next 3 bits of work + 1), the largest work the
// smallest key.
constexpr uint32_t kOrderKeys = 256;
__device__ __forceinline__ uint32_t heavy_first(uint32_t work) {
  const uint32_t v = work < 0xFFFFFFFFu ? work + 1u : work;
  const uint32_t e = 31u - static_cast<uint32_t>(__builtin_clz(v));
  const uint32_t fraction = (e >= 3u ? v >> (e - 3u) : v << (3u - e)) & 7u;
  return kOrderKeys - 1u - (e * 8u + fraction);
}

// Whether the splat's 1/255 ellipse can reach a pixel centre of the block:
// the least of q = qx x^2 + 2 qy x y + qz y^2 over the block's square of pixel
// centres against 2 ln(255 o). That least lies on an edge facing the splat's
// centre (at the optimum an edge that holds the point back faces it), so on
// x = xn or y = yn, the square's coordinates nearest the centre (zero where the
// centre lies between the edges: a point of the square too). The reciprocals
// and the logarithm are the hardware's. The slack covers them and every
// rounding, here and in the pixels' own exponents, in proportion to the largest
// terms q has in the block: a splat some pixel would take is never left out.
// Staging was about a fifth of the forward's vector work: with this test in place
// of the lists' (four edges, correctly rounded divisions and logarithm), the
// masks from their ends instead of pixel by pixel, and exp_finite's shorter tail,
// the forward took 85.1 us for 91.7 at 1M Gaussians and 1280x720, and 179 for 195
// at 1M heavy-tailed ones and 1920x1080 (32x32 lists).
__device__ __forceinline__ bool reaches_block(const Splat &s, float x0, float y0) {
  const float lowx = (x0 + 0.5f) - s.cx, lowy = (y0 + 0.5f) - s.cy;
  const float highx = lowx + 7.0f, highy = lowy + 7.0f;
  const float xn = __builtin_amdgcn_fmed3f(lowx, highx, 0.0f), yn = __builtin_amdgcn_fmed3f(lowy, highy, 0.0f);
  const float y = __builtin_amdgcn_fmed3f(-(s.qy * xn) * __builtin_amdgcn_rcpf(s.qz), lowy, highy);
  const float x = __builtin_amdgcn_fmed3f(-(s.qy * yn) * __builtin_amdgcn_rcpf(s.qx), lowx, highx);
  const float vertical = fma32(s.qz * y, y, fma32(2.0f * s.qy * xn, y, s.qx * xn * xn));
  const float horizontal = fma32(s.qz * yn, yn, fma32(2.0f * s.qy * x, yn, s.qx * x * x));
  const float fx = __builtin_fmaxf(-lowx, highx), fy = __builtin_fmaxf(-lowy, highy); // the farthest pixel centres
  const float terms = fma32(s.qz * fy, fy, s.qx * fx * fx);
  const float reach = 1.3862944f * __builtin_amdgcn_logf(255.0f * s.o); // 2 ln(255 o), v_log_f32 being log2
  // A splat whose determinant overflows has a conic of zeros (or next to nothing, its
  // reciprocals infinite), with which the lists' test finds no edge that it reaches:
  // it is its centre's block's alone, in every tile shape.
  const bool conic = __builtin_fmaxf(s.qx, s.qz) > 0x1p-128f || s.qy != 0.0f;
  return __builtin_fminf(vertical, horizontal) <= fma32(1e-6f, terms, fma32(reach, 1.001f, 1e-3f)) &&
         (conic || (xn == 0.0f && yn == 0.0f));
}

// The bits lo .. hi - 1 (0 <= lo < hi <= 8) of pixels first + lo, ... (centres)
// that lie within `radius` of c, |d| <= radius in float. [lo, hi) is the extent
// box's pixels in the block, and the extent is at most the radius, so a pixel
// centre of it is at most extent + 1 away plus the box's own rounding: only the
// first two and the last two can fail.
__device__ __forceinline__ uint32_t span_mask(float first, uint32_t lo, uint32_t hi, float c, float radius) {
  float l = first + static_cast<float>(lo), h = first + static_cast<float>(hi - 1u);
#pragma unroll
  for (int k = 0; k < 2; ++k) {
    l = fabsf(l - c) > radius ? l + 1.0f : l;
    h = fabsf(h - c) > radius ? h - 1.0f : h;
  }
  const int from = static_cast<int>(l - first), to = static_cast<int>(h - first); // first and last, from > to for none
  return (0xFFu << from) & (0xFFu >> (7 - to)) & (from > to ? 0u : 0xFFu);
}

// The block's pixels a splat can touch: inside the extent box and within the
// radius (|d| <= r on both axes, d from the pixel centre). A larger tile's list
// holds every splat whose extent box meets the block (the block marks), and
// about a quarter of those (elongated, turned splats) have boxes that meet the
// block where their 1/255 ellipse does not: those are dropped here, so that every
// tile shape stages about the splats the lists of 8x8 tiles hold, and none that
// could take a pixel of the block.
__device__ __forceinline__ Staged stage(const Splat &s, const BlockGeometry &geo, uint32_t entry) {
  const uint32_t box = splat_box(s, geo.x0, geo.y0, geo.x1, geo.y1);
  const float x0 = static_cast<float>(geo.x0), y0 = static_cast<float>(geo.y0);
  uint32_t mask = 0;
  if (box != 0u && (!geo.reach || reaches_block(s, x0, y0))) {
    mask = span_mask(x0 + 0.5f, box & 0xFFu, (box >> 16) & 0xFFu, s.cx, s.radius) |
           (span_mask(y0 + 0.5f, (box >> 8) & 0xFFu, box >> 24, s.cy, s.radius) << 16);
  }
  return Staged{s.qx, s.qy, s.qz, s.o, s.r, s.g, s.b, entry, s.cx, s.cy, mask, 0u};
}

// Lane l's pixel in its block and its two mask bits.
__device__ __forceinline__ uint32_t lane_bits(uint32_t lx, uint32_t ly) { return (1u << lx) | (1u << (16u + ly)); }

// The wave votes as scalar masks: a ballot of one comparison is that
// comparison's lane mask, so the loops vote with the AND of the ballots of
// single comparisons (scalar work) rather than the ballot of a combined
// predicate (which costs vector instructions to form).
__device__ __forceinline__ uint64_t vote(bool p) { return __builtin_amdgcn_ballot_w64(p); }

// The calling lane's bit of a lane mask, as the condition of a selection (the
// mask itself is the selection's operand).
__device__ __forceinline__ bool lane_of(uint64_t mask) { return __builtin_amdgcn_inverse_ballot_w64(mask); }

// The position of set bit number k (from 0) of m, which has more than k.
__device__ __forceinline__ uint32_t kth_set_bit(uint64_t m, uint32_t k) {
  uint32_t at = 0;
#pragma unroll
  for (uint32_t w = 32; w >= 1; w >>= 1) {
    const uint32_t low = static_cast<uint32_t>(__popcll(m & ((1ull << w) - 1ull)));
    if (k >= low) {
      k -= low;
      m >>= w;
      at += w;
    }
  }
  return at;
}

// The Gaussian's exponent at offset (dx, dy) (splat_at, train_types.glsl:88).
__device__ __forceinline__ float power_at(const Staged &s, float dx, float dy) {
  return fma32(-0.5f, fma32(s.qx * dx, dx, (s.qz * dy) * dy), -((s.qy * dx) * dy));
}

// A block's walk over its tile's list in batches of up to kBlock entries that
// have the block's bit (blockBit) in their key, from pos towards limit (up: pos,
// pos + 1, ...; down: pos - 1, pos - 2, ...), with its loads in flight ahead of
// their use. A staged batch needs three loads that wait for each other: the
// keys, the wanted entries' Gaussians, and their splats. While a batch is
// worked, request() queues the next one's entries (from keys loaded before)
// and starts the load of their Gaussians, fetch(), half a batch later, that of
// their splats, and stage() uses them when the next batch's turn comes.
template <bool Down> struct ListWalk {
  const Splat *__restrict__ splats;
  const uint32_t *__restrict__ entryKeys;
  const uint32_t *__restrict__ entryValues;
  uint32_t blockBit, limit, pos;
  uint32_t key;             // this lane's key of the window at pos
  uint32_t queued, entry;   // the next batch: its size, this lane's entry
  uint32_t gaussian;
  float4 a, b, c;

  __device__ __forceinline__ uint32_t left() const { return Down ? pos - limit : limit - pos; }
  __device__ __forceinline__ uint32_t window_entry() const { return Down ? pos - 1u - threadIdx.x : pos + threadIdx.x; }
  __device__ __forceinline__ void load_window() { key = threadIdx.x < left() ? entryKeys[window_entry()] : 0u; }

  // Fills the queue for the next batch and loads its Gaussians' indices.
  __device__ __forceinline__ void request(uint32_t *queue) {
    const uint32_t lane = threadIdx.x;
    queued = 0;
    while (queued < kBlock && pos != limit) {
      const uint32_t n = left() < kBlock ? left() : kBlock;
      const bool wanted = lane < n && (key & blockBit) != 0u;
      const uint64_t m = __ballot(wanted);
      const uint32_t found = static_cast<uint32_t>(__popcll(m)), room = kBlock - queued;
      const uint32_t taken = found > room ? kth_set_bit(m, room) : n; // window entries used up
      if (wanted && lane < taken) queue[queued + static_cast<uint32_t>(__popcll(m & ((1ull << lane) - 1ull)))] = window_entry();
      queued += found < room ? found : room;
      pos = Down ? pos - taken : pos + taken;
      load_window();
    }
    __syncthreads();
    if (lane < queued) {
      entry = queue[lane];
      gaussian = entryValues[entry];
    }
  }
  // Loads the requested batch's splats.
  __device__ __forceinline__ void fetch() {
    if (threadIdx.x < queued) {
      const float4 *p = reinterpret_cast<const float4 *>(splats + gaussian);
      a = p[0];
      b = p[1];
      c = p[2];
    }
  }
  // The fetched batch: each lane stages one splat, and those that can touch a
  // pixel of the block are packed at the front of `batch` in walk order (with
  // the byte offsets of their rows of rowBytes, when rowOffset is given, and
  // their Gaussians marked in `touched`). Returns how many were kept.
  __device__ __forceinline__ uint32_t stage(const BlockGeometry &geo, Staged *batch, uint64_t *rowOffset, uint32_t rowBytes,
                                            uint8_t *__restrict__ touched) const {
    Staged st{};
    bool keep = false;
    if (threadIdx.x < queued) {
      st = vsplat::stage(Splat{a.x, a.y, a.z, a.w, b.x, b.y, b.z, b.w, c.x, c.y, c.z, c.w}, geo, entry);
      keep = (st.cols & 0xFFu) != 0u && (st.cols >> 16) != 0u;
    }
    const uint64_t kept = __ballot(keep);
    if (keep) {
      const uint32_t slot = static_cast<uint32_t>(__popcll(kept & ((1ull << threadIdx.x) - 1ull)));
      batch[slot] = st;
      if (rowOffset != nullptr) {
        rowOffset[slot] = static_cast<uint64_t>(gaussian) * rowBytes;
        touched[gaussian] = 1;
      }
    }
    return static_cast<uint32_t>(__popcll(kept));
  }
};

// Front to back over a tile's list (train_forward.comp:38-100): the colour
// (with Colour), the transmittance and its log, and the stop index of the
// calling lane's pixel. The forward pass and the backward pass that
// recomputes the transmittance both run this, so they agree bit for bit.
// A pixel stops at the splat that would take its transmittance, the product
// of 1 - alpha, under 1e-4; train_forward.comp:84-88 asks the same of the sum
// of the logs (log T < log 1e-4), which costs a log per pair, and rounds
// further from the exact product than the product does. The log of the
// final transmittance is taken once per pixel.
template <bool Colour>
__device__ __forceinline__ void composite_block(const Splat *__restrict__ splats, const uint32_t *__restrict__ entryKeys,
                                                const uint32_t *__restrict__ entryValues, uint32_t blockBit, uint2 range,
                                                const BlockGeometry &geo, Staged *batch, uint32_t *queue, bool inside, float px, float py,
                                                uint32_t bits, float &r, float &g, float &b, float &T, float &logT, uint32_t &stop) {
  stop = range.x;
  uint64_t doneLanes = ~vote(inside); // lanes whose pixel is finished (or outside the image)
  if (range.y > range.x && doneLanes != ~0ull) {
    ListWalk<true> walk{splats, entryKeys, entryValues, blockBit, range.x, range.y};
    walk.load_window();
    walk.request(queue);
    walk.fetch();
    while (walk.queued != 0) {
      const uint32_t kept = walk.stage(geo, batch, nullptr, 0u, nullptr);
      // Pad the last group with splats no pixel is a candidate for (their
      // colours, which a zero weight multiplies, finite).
      if (threadIdx.x < kGroup) batch[kept + threadIdx.x] = Staged{};
      __syncthreads();
      walk.request(queue);
      bool fetched = false;
      // The batch runs front to back already (the queue was filled walking down).
      for (uint32_t k = 0; k < kept && doneLanes != ~0ull; k += kGroup) {
        if (!fetched && k * 2u >= kept) {
          walk.fetch();
          fetched = true;
        }
        uint64_t oks[kGroup];
        float alpha[kGroup];
#pragma unroll
        for (uint32_t j = 0; j < kGroup; ++j) {
          const Staged &s = batch[k + j];
          const bool covered = (s.cols & bits) == bits;
          const float dx = px - s.cx, dy = py - s.cy;
          const float power = power_at(s, dx, dy);
          // Below -87 alpha is far under 1/255 either way, so the clamp in exp_finite decides nothing.
          const float a = s.o * exp_finite(power);
          alpha[j] = a < 0.99f ? a : 0.99f;
          oks[j] = vote(covered) & vote(!(power > 0.0f)) & vote(alpha[j] >= kMinAlpha);
        }
#pragma unroll
        for (uint32_t j = 0; j < kGroup; ++j) {
          const Staged &s = batch[k + j];
          const uint64_t ok = oks[j] & ~doneLanes;
          // Without branches: a lane that takes nothing adds a zero weight
          // (fma(0, c, r) is r) and keeps its transmittance by selection.
          const float Tnext = T * (1.0f - alpha[j]);
          const uint64_t stops = ok & vote(Tnext < kMinTransmittance);
          const bool take = lane_of(ok & ~stops);
          if constexpr (Colour) {
            const float w = take ? T * alpha[j] : 0.0f;
            r = fma32(w, s.r, r);
            g = fma32(w, s.g, g);
            b = fma32(w, s.b, b);
          }
          T = take ? Tnext : T;
          if (stops != 0) {
            stop = lane_of(stops) ? s.entry + 1u : stop;
            doneLanes |= stops;
          }
        }
      }
      if (doneLanes == ~0ull) break;
      if (!fetched) walk.fetch();
      __syncthreads(); // the batch is read
    }
  }
  logT = log_normal(T); // T in [1e-4, 1]: a normal float
}

// The forward pass of one 8x8 block (item) of a view.
template <uint32_t TW, uint32_t TH>
__device__ __forceinline__ void forward_block(uint32_t item, const Splat *__restrict__ splats, const uint32_t *__restrict__ entryKeys,
                                              const uint32_t *__restrict__ entryValues, uint32_t tileBits,
                                              const uint2 *__restrict__ ranges, uint32_t width, uint32_t height, uint32_t gridW,
                                              float bgR, float bgG, float bgB, float4 *__restrict__ image, uint32_t *__restrict__ stops,
                                              uint32_t *__restrict__ work, Staged *batch, uint32_t *queue) {
  uint32_t tile;
  const BlockGeometry geo = block_geometry<TW, TH>(item, gridW, width, height, tile);
  if (geo.x0 >= width || geo.y0 >= height) { // a block past the image's edge (uniform)
    if (work != nullptr && threadIdx.x == 0) work[item] = 0;
    return;
  }
  const uint32_t lx = threadIdx.x & 7u, ly = threadIdx.x >> 3;
  const uint32_t x = geo.x0 + lx, y = geo.y0 + ly;
  const bool inside = x < width && y < height;
  const float px = static_cast<float>(x) + 0.5f, py = static_cast<float>(y) + 0.5f;
  float r = 0.0f, g = 0.0f, b = 0.0f, T = 1.0f, logT = 0.0f;
  uint32_t stop;
  const uint2 range = ranges[tile];
  composite_block<true>(splats, entryKeys, entryValues, 1u << (tileBits + geo.block), range, geo, batch, queue, inside, px, py,
                        lane_bits(lx, ly), r, g, b, T, logT, stop);
  if (inside) {
    const uint32_t at = y * width + x;
    image[at] = make_float4(fma32(T, bgR, r), fma32(T, bgG, g), fma32(T, bgB, b), logT);
    if (stops != nullptr) stops[at] = stop; // none when the backward recomputes them
  }
  if (work != nullptr) {
    // The backward's walk over this block: the entries from its lowest stop to the list's end.
    uint32_t low = inside ? stop : range.y;
#pragma unroll
    for (uint32_t d = 32; d >= 1; d >>= 1) {
      const uint32_t other = static_cast<uint32_t>(__shfl_xor(static_cast<int>(low), static_cast<int>(d), 64));
      low = other < low ? other : low;
    }
    if (threadIdx.x == 0) work[item] = range.y - low;
  }
}

template <uint32_t TW, uint32_t TH>
__global__ __launch_bounds__(kBlock) void forward_kernel(const Splat *__restrict__ splats, const uint32_t *__restrict__ entryKeys,
                                                         const uint32_t *__restrict__ entryValues, uint32_t tileBits,
                                                         const uint2 *__restrict__ ranges, uint32_t width, uint32_t height,
                                                         uint32_t gridW, float bgR, float bgG, float bgB, float4 *__restrict__ image,
                                                         uint32_t *__restrict__ stops, uint32_t *__restrict__ work,
                                                         const uint32_t *__restrict__ order) {
  __shared__ Staged batch[kBlock + kGroup];
  __shared__ uint32_t queue[kBlock];
  const uint32_t item = order != nullptr ? order[blockIdx.x] : blockIdx.x;
  forward_block<TW, TH>(item, splats, entryKeys, entryValues, tileBits, ranges, width, height, gridW, bgR, bgG, bgB, image, stops, work,
                        batch, queue);
}

// The view of a batched launch that block `item` belongs to, and the block's
// index within it (the views' blocks follow each other in view order).
__device__ __forceinline__ uint32_t view_of(const RasterViews &views, uint32_t &item) {
  uint32_t v = 0;
  while (v + 1 < views.count && item >= views.view[v + 1].firstBlock) ++v;
  item -= views.view[v].firstBlock;
  return v;
}

// The forward pass of a batch's views in one launch: one workgroup per
// (view, 8x8 block) pair, the views' tile lists all of shape TW x TH.
template <uint32_t TW, uint32_t TH>
__global__ __launch_bounds__(kBlock) void forward_views_kernel(RasterViews views, float bgR, float bgG, float bgB) {
  __shared__ Staged batch[kBlock + kGroup];
  __shared__ uint32_t queue[kBlock];
  uint32_t item = blockIdx.x;
  const RasterView &w = views.view[view_of(views, item)];
  forward_block<TW, TH>(item, w.splats, w.entryKeys, w.entryValues, w.tileBits, w.ranges, w.width, w.height, w.gridW, bgR, bgG, bgB,
                        w.image, w.stops, nullptr, batch, queue);
}

// The fixed-point quantisation of a wave total (train_backward_fixed.comp:19-21),
// NaN as 0, widened to 64 bits: the scale carries 2^20 steps per unit where the
// reference's carries 64, and the clamp is the reference's 1e9 times the same
// 2^14, so a total spans the same range in units at 16384 times the resolution.
__device__ __forceinline__ int64_t quantise(float v, float scale) {
  float s = v * scale;
  if (s != s) s = 0.0f;
  s = s > kFixedClamp ? kFixedClamp : (s < -kFixedClamp ? -kFixedClamp : s);
  return static_cast<int64_t>(__builtin_rintf(s));
}

// The totals of a splat's values over the wave: each value through the same
// tree over the lanes (partners l ^ 32, 16, 15, 7, 2, 1 in turn; a + b and b + a
// are the same float). The first two steps are permlane swaps, each followed by
// one add for two values. (Moving the values through LDS instead, with no
// swaps, was slower: its traffic is more than the LDS carries.) The last four
// steps are DPP adds within 16-lane rows, two of them merging a pair of values
// by bank masks (lanes with bit 3, then bit 2, set keep the second) where a
// selection of what to keep and what to send took two instructions more each.

// A DPP add reads a register two wait states after a vector instruction wrote
// it, which the compiler does not see inside the block: hence the s_nops.
__device__ __forceinline__ float reduce_row3(float a, float b, float c) {
  float t, u, w;
  asm("s_nop 1\n\t"
      "v_add_f32_dpp %0, %3, %3 row_mirror row_mask:0xf bank_mask:0x3\n\t"
      "v_add_f32_dpp %1, %5, %5 row_mirror row_mask:0xf bank_mask:0xf\n\t"
      "v_add_f32_dpp %0, %4, %4 row_mirror row_mask:0xf bank_mask:0xc\n\t"
      "s_nop 0\n\t"
      "v_add_f32_dpp %2, %1, %1 row_half_mirror row_mask:0xf bank_mask:0xa\n\t"
      "v_add_f32_dpp %2, %0, %0 row_half_mirror row_mask:0xf bank_mask:0x5\n\t"
      "s_nop 1\n\t"
      "v_add_f32_dpp %2, %2, %2 quad_perm:[2,3,0,1] row_mask:0xf bank_mask:0xf\n\t"
      "s_nop 1\n\t"
      "v_add_f32_dpp %2, %2, %2 quad_perm:[1,0,3,2] row_mask:0xf bank_mask:0xf"
      : "=&v"(t), "=&v"(u), "=&v"(w)
      : "v"(a), "v"(b), "v"(c));
  return w;
}

__device__ __forceinline__ float swap32_add(float a, float b) {
  const auto p = __builtin_amdgcn_permlane32_swap(as_uint(a), as_uint(b), false, false);
  return as_float(p[0]) + as_float(p[1]);
}
__device__ __forceinline__ float swap16_add(float a, float b) {
  const auto p = __builtin_amdgcn_permlane16_swap(as_uint(a), as_uint(b), false, false);
  return as_float(p[0]) + as_float(p[1]);
}

// Twelve values per lane to the wave's twelve totals: lane l ends with the total
// of value reduced_value(l); wave_emits(l) picks one lane per value.
__device__ __forceinline__ float reduce_wave(const float (&v)[12]) {
  float u[6];
#pragma unroll
  for (int i = 0; i < 6; ++i) u[i] = swap32_add(v[i], v[i + 6]); // lanes 0-31 keep values 0-5
  return reduce_row3(swap16_add(u[0], u[3]), swap16_add(u[1], u[4]), swap16_add(u[2], u[5]));
}

// Sixteen values per lane, for the scored pass's fourteen sums: lane l ends with
// the total of value reduced_value16(l).
__device__ __forceinline__ float reduce_wave16(const float (&v)[16]) {
  float u[8];
#pragma unroll
  for (int i = 0; i < 8; ++i) u[i] = swap32_add(v[i], v[i + 8]);
  const float last = swap16_add(u[3], u[7]);
  const float w = reduce_row3(swap16_add(u[0], u[4]), swap16_add(u[1], u[5]), swap16_add(u[2], u[6]));
  const float z = reduce_row3(last, last, last);
  return (threadIdx.x & 12u) == 12u ? z : w;
}

// The value whose total lane l holds after reduce_wave: 3 (l / 16) + (b2 ? 2 : b3),
// with bk bit k of l.
__device__ __forceinline__ uint32_t reduced_value(uint32_t lane) {
  return 3u * (lane >> 4) + ((lane & 4u) != 0u ? 2u : (lane >> 3) & 1u);
}
// One lane per value: bits 0 and 1 clear, and not both bits 2 and 3 (those
// lanes hold the third value twice).
__device__ __forceinline__ bool wave_emits(uint32_t lane) { return (lane & 3u) == 0u && (lane & 12u) != 12u; }
// After reduce_wave16: 4 (l / 16) + the third or the fourth where bit 2 is set, by bit 3.
__device__ __forceinline__ uint32_t reduced_value16(uint32_t lane) {
  return 4u * (lane >> 4) + ((lane & 4u) != 0u ? ((lane & 8u) != 0u ? 3u : 2u) : (lane >> 3) & 1u);
}

// What a wave adds to a splat's row of raw sums, given the splat and the pixel's
// alpha (0 where it takes nothing), transmittance in front and colour behind.
// Lane l adds value `value` of the row, in fixed-point steps or as it is; values 3
// to 5 are reduced twice their size (an exact halving in the scale). Values 12 and
// 13 of the kRawPerSplat slots are zero without scoring.
template <bool Fixed, bool Score> struct Emitter {
  float4 adj;
  float perPixel, edgeWeight, scale;
  uint64_t lanes;
  uint8_t *base;

  __device__ __forceinline__ Emitter(const float4 &adjoint, float edge, float perPixelShare, float fixedScale,
                                     unsigned long long *rawFixed, float *rawFloat)
      : adj(adjoint), perPixel(perPixelShare), edgeWeight(edge) {
    const uint32_t lane = threadIdx.x & 63u;
    const uint32_t value = Score ? reduced_value16(lane) : reduced_value(lane);
    lanes = vote(Score ? (lane & 3u) == 0 && value < kRawPerSplat : wave_emits(lane));
    scale = (value >= 3u && value <= 5u ? 0.5f : 1.0f) * (Fixed ? fixedScale : 1.0f);
    base = Fixed ? reinterpret_cast<uint8_t *>(rawFixed + value) : reinterpret_cast<uint8_t *>(rawFloat + value);
  }

  // ok: the lanes that take something; free: those of them whose alpha is not
  // clamped (at the 0.99 clamp alpha no longer depends on the parameters).
  __device__ __forceinline__ void operator()(const Staged &s, float dx, float dy, float e, float alpha, float T, float Br, float Bg, float Bb,
                                             uint64_t ok, uint64_t free, uint64_t rowOffset) const {
    const float Ta = T * alpha;
    const float toward = T * fma32(adj.z, s.b - Bb, fma32(adj.y, s.g - Bg, adj.x * (s.r - Br)));
    const float dAlpha = lane_of(free) ? toward : 0.0f;
    const float dPower = dAlpha * alpha;
    const float vx = fma32(s.qy, dy, s.qx * dx), vy = fma32(s.qz, dy, s.qy * dx);
    const float g1 = dPower * vx, g2 = dPower * vy;
    constexpr int kValues = Score ? 16 : 12;
    float v[kValues];
    v[0] = dAlpha * e;
    v[1] = g1;
    v[2] = g2;
    v[3] = g1 * vx; // twice the sum (scale)
    v[4] = g1 * vy;
    v[5] = g2 * vy;
    v[6] = Ta * adj.x;
    v[7] = Ta * adj.y;
    v[8] = Ta * adj.z;
    v[9] = Ta * perPixel;
    v[10] = fabsf(g1);
    v[11] = fabsf(g2);
    if constexpr (Score) {
      v[12] = lane_of(ok) ? adj.w * perPixel : 0.0f;
      v[13] = (edgeWeight * Ta) * perPixel;
      v[14] = v[15] = 0.0f;
    }
    float total;
    if constexpr (Score) {
      total = reduce_wave16(v);
    } else {
      total = reduce_wave(v);
    }
    uint8_t *const slot = base + rowOffset;
    const float scaled = total * scale;
    if constexpr (Fixed) {
      // Totals under 2^31 steps (nearly all) round and convert in 32 bits,
      // exactly as quantise() would; the wave takes quantise() if any is larger.
      const float rounded = __builtin_rintf(scaled);
      int64_t q = static_cast<int32_t>(rounded);
      uint64_t send = lanes & vote(rounded != 0.0f);
      if ((lanes & vote(!(fabsf(scaled) < 2147483648.0f))) != 0u) {
        q = quantise(total, scale);
        send = lanes & vote(q != 0);
      }
      if (lane_of(send)) atomicAdd(reinterpret_cast<unsigned long long *>(slot), static_cast<unsigned long long>(q));
    } else {
      if (lane_of(lanes & vote(scaled != 0.0f))) atomicAdd(reinterpret_cast<float *>(slot), scaled);
    }
  }
};

// Back to front over the tile's list (train_backward.glsl:78-158), for the
// block's pixels, from the block's lowest stop. Bound by the vector unit: a
// splat's evaluation is 29 instructions, its gradient terms, reduction and emission
// where a pixel takes it 91 more, the permlane swaps and the reciprocal among them at
// a third of an fma's rate. At 1M Gaussians and 1280x720 (32x32 lists, fixed point) 205 us
// before the walk's loads ran ahead, the evaluations were grouped, the reduction
// merged by bank masks and the emission shortened (a row's byte offset staged
// once, the halves of sums 3 to 5 taken last); 179 us with them. With Recompute the pixel's log
// transmittance and stop come from a front-to-back sweep of its own instead
// of the forward pass's image and stops, which are then not read. With Score
// (a scored view) the last two sums are filled too: the pixel's high-error
// mark (the adjoint's fourth value) and its edge weight times the blending
// weight, each over 3 pixels of the image.
template <bool Fixed, bool Recompute, bool Score, uint32_t TW, uint32_t TH>
__device__ __forceinline__ void backward_block(uint32_t item, const Splat *__restrict__ splats, const uint32_t *__restrict__ entryKeys,
                                               const uint32_t *__restrict__ entryValues, uint32_t tileBits,
                                               const uint2 *__restrict__ ranges, uint32_t width, uint32_t height, uint32_t gridW,
                                               float bgR, float bgG, float bgB, const float4 *__restrict__ image,
                                               const float4 *__restrict__ adjoint, const uint32_t *__restrict__ stops,
                                               float fixedScale, unsigned long long *__restrict__ rawFixed,
                                               float *__restrict__ rawFloat, uint8_t *__restrict__ touched, const float *__restrict__ edge, Staged *batch,
                                               uint64_t *rowOffset, uint32_t *queue) {
  uint32_t tile;
  const BlockGeometry geo = block_geometry<TW, TH>(item, gridW, width, height, tile);
  if (geo.x0 >= width || geo.y0 >= height) return; // a block past the image's edge (uniform)
  const uint32_t lane = threadIdx.x, lx = lane & 7u, ly = lane >> 3;
  const uint32_t bits = lane_bits(lx, ly);
  const uint32_t x = geo.x0 + lx, y = geo.y0 + ly;
  const bool inside = x < width && y < height;
  const float px = static_cast<float>(x) + 0.5f, py = static_cast<float>(y) + 0.5f;
  const uint32_t at = inside ? y * width + x : 0u;
  const float4 adj = inside ? adjoint[at] : make_float4(0.0f, 0.0f, 0.0f, 0.0f);
  const float edgeWeight = Score && inside ? edge[at] : 0.0f;
  const float perPixel = 1.0f / (3.0f * static_cast<float>(width) * static_cast<float>(height));
  const uint2 range = ranges[tile];
  float logTotal;
  uint32_t stop;
  if constexpr (Recompute) {
    float r = 0.0f, g = 0.0f, b = 0.0f, T = 1.0f;
    logTotal = 0.0f;
    composite_block<false>(splats, entryKeys, entryValues, 1u << (tileBits + geo.block), range, geo, batch, queue, inside, px, py, bits, r,
                           g, b, T, logTotal, stop);
    if (!inside) stop = range.y;
  } else {
    logTotal = inside ? image[at].w : 0.0f;
    stop = inside ? stops[at] : range.y;
  }
  // The block's lowest stop: entries before it have no candidate lane here.
  uint32_t first = stop;
#pragma unroll
  for (uint32_t d = 32; d >= 1; d >>= 1) {
    const uint32_t other = static_cast<uint32_t>(__shfl_xor(static_cast<int>(first), static_cast<int>(d), 64));
    first = other < first ? other : first;
  }
  // The colour behind the splats visited so far, and the transmittance in
  // front of them: before any, the background and the pixel's final
  // transmittance. Walking back, a splat's own transmittance is the one in
  // front of those behind it over 1 - alpha, one rounding a step, where
  // train_backward.glsl:119 takes the exp of the difference of two log sums.
  float Br = bgR, Bg = bgG, Bb = bgB;
  float Tbehind = exp_finite(logTotal);

  const uint64_t insideLanes = vote(inside);
  const Emitter<Fixed, Score> emit(adj, edgeWeight, perPixel, fixedScale, rawFixed, rawFloat);
  if (first >= range.y) return;
  ListWalk<false> walk{splats, entryKeys, entryValues, 1u << (tileBits + geo.block), range.y, first};
  walk.load_window();
  walk.request(queue);
  walk.fetch();
  while (walk.queued != 0) {
    const uint32_t kept = walk.stage(geo, batch, rowOffset, kRawPerSplat * (Fixed ? 8u : 4u), touched);
    if (lane < kGroup) batch[kept + lane] = Staged{}; // the last group padded with splats no pixel is a candidate for
    __syncthreads();
    walk.request(queue);
    bool fetched = false;
    for (uint32_t k = 0; k < kept; k += kGroup) {
      if (!fetched && k * 2u >= kept) {
        walk.fetch();
        fetched = true;
      }
      uint64_t oks[kGroup];
      float falloff[kGroup];
#pragma unroll
      for (uint32_t j = 0; j < kGroup; ++j) {
        const Staged &s = batch[k + j];
        const float power = power_at(s, px - s.cx, py - s.cy);
        const float e = exp_finite(power);
        falloff[j] = e;
        oks[j] = insideLanes & vote(s.entry >= stop) & vote((s.cols & bits) == bits) & vote(!(power > 0.0f)) &
                 vote(!(s.o * e < kMinAlpha));
      }
#pragma unroll
      for (uint32_t j = 0; j < kGroup; ++j) {
        if (oks[j] == 0) continue;
        const Staged s = batch[k + j];
        const float dx = px - s.cx, dy = py - s.cy;
        const float e = falloff[j];
        const float a = s.o * e;
        // A lane that takes nothing from the splat has alpha 0: its
        // transmittance, the colour behind it and every sum below stay as they
        // are (T / 1 is T; every other factor is finite, and the sign of a zero
        // cannot change a total that is not zero). Else 0.01 <= 1 - alpha <= 1,
        // and the transmittance is at least the pixel's final one, which the
        // forward keeps at or above 1e-4, so the short division is exact
        // `Tbehind / (1 - alpha)`.
        const float alpha = lane_of(oks[j]) ? (a < 0.99f ? a : 0.99f) : 0.0f;
        const float T = div_in_range(Tbehind, 1.0f - alpha);
        emit(s, dx, dy, e, alpha, T, Br, Bg, Bb, oks[j], oks[j] & vote(a < 0.99f), rowOffset[k + j]);
        Br = fma32(alpha, s.r - Br, Br);
        Bg = fma32(alpha, s.g - Bg, Bg);
        Bb = fma32(alpha, s.b - Bb, Bb);
        Tbehind = T;
      }
    }
    if (!fetched) walk.fetch();
    __syncthreads(); // the batch is read
  }
}


template <bool Fixed, bool Recompute, bool Score, uint32_t TW, uint32_t TH>
__global__ __launch_bounds__(kBlock) void backward_kernel(const Splat *__restrict__ splats, const uint32_t *__restrict__ entryKeys,
                                                          const uint32_t *__restrict__ entryValues, uint32_t tileBits,
                                                          const uint2 *__restrict__ ranges, uint32_t width, uint32_t height, uint32_t gridW,
                                                          float bgR, float bgG, float bgB, const float4 *__restrict__ image,
                                                          const float4 *__restrict__ adjoint, const uint32_t *__restrict__ stops,
                                                          float fixedScale, unsigned long long *__restrict__ rawFixed,
                                                          float *__restrict__ rawFloat, uint8_t *__restrict__ touched, const float *__restrict__ edge,
                                                          const uint32_t *__restrict__ order) {
  __shared__ Staged batch[kBlock + kGroup];
  __shared__ uint64_t rowOffset[kBlock];
  __shared__ uint32_t queue[kBlock];
  const uint32_t item = order != nullptr ? order[blockIdx.x] : blockIdx.x;
  backward_block<Fixed, Recompute, Score, TW, TH>(item, splats, entryKeys, entryValues, tileBits, ranges, width, height, gridW, bgR,
                                                  bgG, bgB, image, adjoint, stops, fixedScale, rawFixed, rawFloat, touched, edge, batch, rowOffset,
                                                  queue);
}

// The backward pass of a batch's views in one launch, one workgroup per
// (view, 8x8 block) pair; each view's sums go to its own raw buffer.
template <bool Fixed, bool Recompute, uint32_t TW, uint32_t TH>
__global__ __launch_bounds__(kBlock) void backward_views_kernel(RasterViews views, float bgR, float bgG, float bgB) {
  __shared__ Staged batch[kBlock + kGroup];
  __shared__ uint64_t rowOffset[kBlock];
  __shared__ uint32_t queue[kBlock];
  uint32_t item = blockIdx.x;
  const RasterView &w = views.view[view_of(views, item)];
  backward_block<Fixed, Recompute, false, TW, TH>(item, w.splats, w.entryKeys, w.entryValues, w.tileBits, w.ranges, w.width, w.height,
                                                  w.gridW, bgR, bgG, bgB, w.image, w.adjoint, w.stops, w.fixedScale,
                                                  reinterpret_cast<unsigned long long *>(w.rawFixed), w.rawFloat, w.touched, nullptr, batch,
                                                  rowOffset, queue);
}

// ---- Small views: four waves a block.
//
// A view of few blocks leaves most SIMDs with one wave or none, and a lone wave
// issues at half the rate and waits out every latency: its time is the length of
// its heaviest block's chain of splats. There a block is worked by kWideWaves
// waves on the same 64 pixels, which share what does not depend on the order of
// the splats: a window of 256 entries is staged by 256 threads; of each chunk of
// kWideChunk staged splats every wave evaluates a quarter, leaving the alphas
// (0 where a pixel takes nothing) in LDS; then every wave follows the whole chain
// from the alphas, a few instructions a splat, the forward's waves for one colour
// channel each, the backward's emitting the sums of the splats they evaluated.
// Every float is formed as in the one-wave kernels, so the results are the same
// bits. It does more work in all (the chain four times over), so it is for views
// of few blocks (wide_blocks). Forward and backward against one wave a block:
// 10k Gaussians at 256x256 (1024 blocks) 18.5 and 40.5 us, before 32 and 59; a
// batch's 1504-block view of 10k 47 and 87 us, before 86 and 150.
constexpr uint32_t kWideWaves = 4, kWideThreads = kWideWaves * 64, kWideChunk = 32, kWideShare = kWideChunk / kWideWaves;

struct WideShared {
  Staged batch[kWideThreads + kWideChunk];
  uint64_t rowOffset[kWideThreads];
  float alpha[2][kWideChunk][64];
  uint32_t kept[kWideWaves];
};

// block_geometry for a tile shape known at run time.
__device__ __forceinline__ BlockGeometry wide_geometry(uint32_t h, uint32_t tileW, uint32_t tileH, uint32_t gridW, uint32_t width,
                                                       uint32_t height, uint32_t &tile) {
  const uint32_t across = tileW >> 3, perTile = across * (tileH >> 3), u = h / kRasterXcds;
  tile = (u / perTile) * kRasterXcds + h % kRasterXcds;
  const uint32_t q = u % perTile;
  const uint32_t x0 = (tile % gridW) * tileW + (q % across) * 8u, y0 = (tile / gridW) * tileH + (q / across) * 8u;
  return {x0, y0, x0 + 8u < width ? x0 + 8u : width, y0 + 8u < height ? y0 + 8u : height, q, perTile > 1u};
}

// The walk of a block's four waves over its tile's list, a window of 256 entries
// at a time: the next window's splats and the keys and Gaussians of the one
// after are in flight while a window is worked.
template <bool Down> struct WideWalk {
  const Splat *__restrict__ splats;
  const uint32_t *__restrict__ entryKeys;
  const uint32_t *__restrict__ entryValues;
  uint32_t blockBit, limit, pos;
  uint32_t entryNext, key, value; // this thread's entry of the window at pos
  uint32_t entry, gaussian;
  bool wanted, more;
  float4 a, b, c;

  __device__ __forceinline__ void load_window() {
    const uint32_t left = Down ? pos - limit : limit - pos;
    const bool valid = threadIdx.x < left;
    entryNext = Down ? pos - 1u - threadIdx.x : pos + threadIdx.x;
    key = valid ? entryKeys[entryNext] : 0u;
    value = valid ? entryValues[entryNext] : 0u;
  }
  // Takes the window at pos, starts the load of its splats and of the next window.
  __device__ __forceinline__ void take() {
    more = pos != limit;
    if (!more) return;
    wanted = (key & blockBit) != 0u;
    gaussian = value;
    entry = entryNext;
    if (wanted) {
      const float4 *p = reinterpret_cast<const float4 *>(splats + gaussian);
      a = p[0];
      b = p[1];
      c = p[2];
    }
    const uint32_t left = Down ? pos - limit : limit - pos, n = left < kWideThreads ? left : kWideThreads;
    pos = Down ? pos - n : pos + n;
    load_window();
  }
  // The taken window's splats staged, those that can touch the block packed in
  // walk order; padded to whole chunks. Returns how many. (Two barriers: every
  // thread calls it; the batch may be read after it.)
  __device__ __forceinline__ uint32_t stage(const BlockGeometry &geo, WideShared &shared, uint32_t rowBytes, uint8_t *__restrict__ touched) const {
    Staged st{};
    bool keep = false;
    if (wanted) {
      st = vsplat::stage(Splat{a.x, a.y, a.z, a.w, b.x, b.y, b.z, b.w, c.x, c.y, c.z, c.w}, geo, entry);
      keep = (st.cols & 0xFFu) != 0u && (st.cols >> 16) != 0u;
    }
    const uint64_t mine = __ballot(keep);
    const uint32_t lane = threadIdx.x & 63u, wave = threadIdx.x >> 6;
    if (lane == 0) shared.kept[wave] = static_cast<uint32_t>(__popcll(mine));
    __syncthreads();
    uint32_t before = 0, total = 0;
#pragma unroll
    for (uint32_t w = 0; w < kWideWaves; ++w) {
      const uint32_t n = shared.kept[w];
      before += w < wave ? n : 0u;
      total += n;
    }
    if (keep) {
      const uint32_t slot = before + static_cast<uint32_t>(__popcll(mine & ((1ull << lane) - 1ull)));
      shared.batch[slot] = st;
      shared.rowOffset[slot] = static_cast<uint64_t>(gaussian) * rowBytes;
      if (touched != nullptr) touched[gaussian] = 1;
    }
    if (threadIdx.x < kWideChunk) shared.batch[total + threadIdx.x] = Staged{};
    __syncthreads();
    return total;
  }
};

// This wave's share of a chunk of staged splats evaluated: the alphas of splats
// at + share .. into `out` rows, 0 where the lane's pixel (in `live`, with stop or
// beyond it when Stops) takes nothing, and each splat's falloff, 0 likewise.
template <bool Stops>
__device__ __forceinline__ void evaluate_share(const Staged *batch, uint32_t at, float (*out)[64], float px, float py, uint32_t bits,
                                               uint64_t live, uint32_t stop, float (&falloff)[kWideShare]) {
  const uint32_t lane = threadIdx.x & 63u, share = (threadIdx.x >> 6) * kWideShare;
#pragma unroll
  for (uint32_t j = 0; j < kWideShare; ++j) {
    const Staged &s = batch[at + share + j];
    const float power = power_at(s, px - s.cx, py - s.cy);
    const float e = exp_finite(power);
    const float a = s.o * e;
    uint64_t ok = live & vote((s.cols & bits) == bits) & vote(!(power > 0.0f)) & vote(!(a < kMinAlpha));
    if constexpr (Stops) ok &= vote(s.entry >= stop);
    falloff[j] = lane_of(ok) ? e : 0.0f;
    out[share + j][lane] = lane_of(ok) ? (a < 0.99f ? a : 0.99f) : 0.0f;
  }
}

// composite_block by four waves: every lane ends with its pixel's transmittance
// and stop; `colour` is the channel of the calling wave (0 to 2: r, g, b; the
// fourth wave's is not used).
__device__ __forceinline__ void composite_wide(const Splat *__restrict__ splats, const uint32_t *__restrict__ entryKeys,
                                               const uint32_t *__restrict__ entryValues, uint32_t blockBit, uint2 range,
                                               const BlockGeometry &geo, WideShared &shared, bool inside, float px, float py, uint32_t bits,
                                               float &colour, float &T, float &logT, uint32_t &stop) {
  const uint32_t lane = threadIdx.x & 63u, wave = threadIdx.x >> 6, channel = wave < 3u ? wave : 0u;
  stop = range.x;
  uint64_t doneLanes = ~vote(inside);
  colour = 0.0f;
  T = 1.0f;
  float Tlive = inside ? 1.0f : 0.0f; // T, or 0 once the pixel is finished
  WideWalk<true> walk{splats, entryKeys, entryValues, blockBit, range.x, range.y};
  walk.load_window();
  for (walk.take(); walk.more && doneLanes != ~0ull;) {
    const uint32_t kept = walk.stage(geo, shared, 0u, nullptr);
    walk.take();
    float falloff[kWideShare];
    uint32_t buffer = 0;
    if (kept != 0) evaluate_share<false>(shared.batch, 0, shared.alpha[0], px, py, bits, ~0ull, 0u, falloff);
    for (uint32_t at = 0; at < kept && doneLanes != ~0ull; at += kWideChunk, buffer ^= 1u) {
      __syncthreads(); // this chunk's alphas are in place, and the chunk before is read
      if (at + kWideChunk < kept) {
        evaluate_share<false>(shared.batch, at + kWideChunk, shared.alpha[buffer ^ 1u], px, py, bits, ~0ull, 0u, falloff);
      }
#pragma unroll 2
      for (uint32_t k = 0; k < kWideChunk; k += kGroup) {
        float alpha[kGroup], c[kGroup], front[kGroup + 1];
        front[0] = Tlive;
#pragma unroll
        for (uint32_t j = 0; j < kGroup; ++j) {
          alpha[j] = shared.alpha[buffer][k + j][lane];
          c[j] = (&shared.batch[at + k + j].r)[channel];
          front[j + 1] = front[j] * (1.0f - alpha[j]);
        }
        // The transmittance only falls: if no pixel is under the bound after the group, none stops in it.
        if ((vote(front[kGroup] < kMinTransmittance) & ~doneLanes) == 0) {
#pragma unroll
          for (uint32_t j = 0; j < kGroup; ++j) colour = fma32(front[j] * alpha[j], c[j], colour);
          Tlive = front[kGroup];
          continue;
        }
#pragma unroll
        for (uint32_t j = 0; j < kGroup; ++j) {
          const float Tnext = Tlive * (1.0f - alpha[j]);
          const uint64_t stops = vote(Tnext < kMinTransmittance) & ~doneLanes;
          // These lanes stop at the splat and do not take it.
          const bool stopped = lane_of(stops);
          const float w = stopped ? 0.0f : Tlive * alpha[j];
          T = stopped ? Tlive : T;
          stop = stopped ? shared.batch[at + k + j].entry + 1u : stop;
          Tlive = stopped ? 0.0f : Tnext;
          doneLanes |= stops;
          colour = fma32(w, c[j], colour);
        }
      }
    }
    __syncthreads(); // the batch is read
  }
  T = lane_of(doneLanes) ? T : Tlive;
  logT = log_normal(T); // T in [1e-4, 1]: a normal float
}

__global__ __launch_bounds__(kWideThreads) void forward_wide_kernel(const Splat *__restrict__ splats, const uint32_t *__restrict__ entryKeys,
                                                                    const uint32_t *__restrict__ entryValues, uint32_t tileBits,
                                                                    const uint2 *__restrict__ ranges, uint32_t width, uint32_t height,
                                                                    uint32_t tileW, uint32_t tileH, uint32_t gridW, float bgR, float bgG,
                                                                    float bgB, float *__restrict__ image, uint32_t *__restrict__ stops,
                                                                    uint32_t *__restrict__ work, const uint32_t *__restrict__ order) {
  __shared__ WideShared shared;
  const uint32_t item = order != nullptr ? order[blockIdx.x] : blockIdx.x;
  uint32_t tile;
  const BlockGeometry geo = wide_geometry(item, tileW, tileH, gridW, width, height, tile);
  if (geo.x0 >= width || geo.y0 >= height) { // a block past the image's edge (uniform)
    if (work != nullptr && threadIdx.x == 0) work[item] = 0;
    return;
  }
  const uint32_t lane = threadIdx.x & 63u, wave = threadIdx.x >> 6, lx = lane & 7u, ly = lane >> 3;
  const uint32_t x = geo.x0 + lx, y = geo.y0 + ly;
  const bool inside = x < width && y < height;
  float colour, T, logT;
  uint32_t stop;
  const uint2 range = ranges[tile];
  composite_wide(splats, entryKeys, entryValues, 1u << (tileBits + geo.block), range, geo, shared, inside, static_cast<float>(x) + 0.5f,
                 static_cast<float>(y) + 0.5f, lane_bits(lx, ly), colour, T, logT, stop);
  if (inside) {
    const uint32_t at = y * width + x;
    const float background = wave == 0u ? bgR : (wave == 1u ? bgG : bgB);
    image[at * 4u + wave] = wave < 3u ? fma32(T, background, colour) : logT;
    if (wave == 3u && stops != nullptr) stops[at] = stop;
  }
  if (work != nullptr && wave == 0u) {
    uint32_t low = inside ? stop : range.y;
#pragma unroll
    for (uint32_t d = 32; d >= 1; d >>= 1) {
      const uint32_t other = static_cast<uint32_t>(__shfl_xor(static_cast<int>(low), static_cast<int>(d), 64));
      low = other < low ? other : low;
    }
    if (lane == 0) work[item] = range.y - low;
  }
}

// backward_block by four waves.
template <bool Fixed, bool Recompute, bool Score>
__global__ __launch_bounds__(kWideThreads) void backward_wide_kernel(const Splat *__restrict__ splats, const uint32_t *__restrict__ entryKeys,
                                                                     const uint32_t *__restrict__ entryValues, uint32_t tileBits,
                                                                     const uint2 *__restrict__ ranges, uint32_t width, uint32_t height,
                                                                     uint32_t tileW, uint32_t tileH, uint32_t gridW, float bgR, float bgG,
                                                                     float bgB, const float4 *__restrict__ image,
                                                                     const float4 *__restrict__ adjoint, const uint32_t *__restrict__ stops,
                                                                     float fixedScale, unsigned long long *__restrict__ rawFixed,
                                                                     float *__restrict__ rawFloat, uint8_t *__restrict__ touched, const float *__restrict__ edge,
                                                                     const uint32_t *__restrict__ order) {
  __shared__ WideShared shared;
  uint32_t tile;
  const BlockGeometry geo = wide_geometry(order != nullptr ? order[blockIdx.x] : blockIdx.x, tileW, tileH, gridW, width, height, tile);
  if (geo.x0 >= width || geo.y0 >= height) return; // a block past the image's edge (uniform)
  const uint32_t lane = threadIdx.x & 63u, wave = threadIdx.x >> 6, lx = lane & 7u, ly = lane >> 3;
  const uint32_t bits = lane_bits(lx, ly);
  const uint32_t x = geo.x0 + lx, y = geo.y0 + ly;
  const bool inside = x < width && y < height;
  const float px = static_cast<float>(x) + 0.5f, py = static_cast<float>(y) + 0.5f;
  const uint32_t at = inside ? y * width + x : 0u;
  const float4 adj = inside ? adjoint[at] : make_float4(0.0f, 0.0f, 0.0f, 0.0f);
  const float edgeWeight = Score && inside ? edge[at] : 0.0f;
  const float perPixel = 1.0f / (3.0f * static_cast<float>(width) * static_cast<float>(height));
  const uint2 range = ranges[tile];
  const uint32_t blockBit = 1u << (tileBits + geo.block);
  float logTotal;
  uint32_t stop;
  if constexpr (Recompute) {
    float colour, T;
    composite_wide(splats, entryKeys, entryValues, blockBit, range, geo, shared, inside, px, py, bits, colour, T, logTotal, stop);
    if (!inside) {
      stop = range.y;
      logTotal = 0.0f;
    }
  } else {
    logTotal = inside ? image[at].w : 0.0f;
    stop = inside ? stops[at] : range.y;
  }
  uint32_t first = stop;
#pragma unroll
  for (uint32_t d = 32; d >= 1; d >>= 1) {
    const uint32_t other = static_cast<uint32_t>(__shfl_xor(static_cast<int>(first), static_cast<int>(d), 64));
    first = other < first ? other : first;
  }
  if (first >= range.y) return; // the same for the four waves
  float Br = bgR, Bg = bgG, Bb = bgB;
  float Tbehind = exp_finite(logTotal);
  const uint64_t insideLanes = vote(inside);
  const Emitter<Fixed, Score> emit(adj, edgeWeight, perPixel, fixedScale, rawFixed, rawFloat);
  WideWalk<false> walk{splats, entryKeys, entryValues, blockBit, range.y, first};
  walk.load_window();
  for (walk.take(); walk.more;) {
    const uint32_t kept = walk.stage(geo, shared, kRawPerSplat * (Fixed ? 8u : 4u), touched);
    walk.take();
    uint32_t buffer = 0;
    float falloff[kWideShare], next[kWideShare];
    if (kept != 0) evaluate_share<true>(shared.batch, 0, shared.alpha[0], px, py, bits, insideLanes, stop, next);
    for (uint32_t start = 0; start < kept; start += kWideChunk, buffer ^= 1u) {
      __syncthreads(); // this chunk's alphas are in place, and the chunk before is read
#pragma unroll
      for (uint32_t j = 0; j < kWideShare; ++j) falloff[j] = next[j];
      if (start + kWideChunk < kept) {
        evaluate_share<true>(shared.batch, start + kWideChunk, shared.alpha[buffer ^ 1u], px, py, bits, insideLanes, stop, next);
      }
      // The chain over the chunk, share by share; the sums of this wave's own on the way.
#pragma unroll 1
      for (uint32_t w = 0; w < kWideWaves; ++w) {
        const uint32_t share = w * kWideShare;
        float alpha[kWideShare];
#pragma unroll
        for (uint32_t j = 0; j < kWideShare; ++j) alpha[j] = shared.alpha[buffer][share + j][lane];
#pragma unroll
        for (uint32_t j = 0; j < kWideShare; ++j) {
          const Staged &s = shared.batch[start + share + j];
          const float T = div_in_range(Tbehind, 1.0f - alpha[j]);
          if (w == wave) {
            const uint64_t ok = vote(alpha[j] != 0.0f);
            if (ok != 0) {
              const Staged own = s;
              emit(own, px - own.cx, py - own.cy, falloff[j], alpha[j], T, Br, Bg, Bb, ok, ok & vote(alpha[j] < 0.99f),
                   shared.rowOffset[start + share + j]);
            }
          }
          Br = fma32(alpha[j], s.r - Br, Br);
          Bg = fma32(alpha[j], s.g - Bg, Bg);
          Bb = fma32(alpha[j], s.b - Bb, Bb);
          Tbehind = T;
        }
      }
    }
    __syncthreads(); // the batch is read
  }
}

constexpr uint32_t kOrderThreads = 1024;
// Keys kept in LDS between the two passes, up to this many items per XCD
// (a 2880x2880 view of 8x8 blocks); past it the second pass reads the work again.
constexpr uint32_t kOrderStaged = 16384;

// Adds each lane's item to its key's count, one atomic per distinct key of the
// wave (most blocks share a few small keys), and returns the lane's place
// among its key's items.
__device__ __forceinline__ uint32_t key_place(uint32_t *counts, uint32_t key, bool valid) {
  const uint32_t lane = threadIdx.x & 63u;
  uint64_t same = __ballot(valid);
#pragma unroll
  for (uint32_t b = 0; b < 8; ++b) { // key < kOrderKeys
    const uint64_t ones = __ballot((key >> b) & 1u);
    same &= ((key >> b) & 1u) ? ones : ~ones;
  }
  const uint32_t lower = static_cast<uint32_t>(__popcll(same & ((uint64_t{1} << lane) - 1u)));
  uint32_t base = 0;
  if (valid && lower == 0) base = atomicAdd(&counts[key], static_cast<uint32_t>(__popcll(same)));
  const int leader = valid ? __builtin_ctzll(same) : static_cast<int>(lane);
  return static_cast<uint32_t>(__shfl(static_cast<int>(base), leader, 64)) + lower;
}

// A raster launch order, heaviest first: one workgroup per XCD x sorts the
// launch indices h = 8 i + x of XCD x by key(h) (a counting sort over
// kOrderKeys keys in LDS) and gives the j-th to launch index 8 j + x, which
// runs on XCD x too (so a tile's blocks still share one L2). Items of one key
// land in any order, which changes nothing: each block's pixels are its own
// and its sums are added with atomics. `items` is a multiple of 8 (raster_blocks).
template <class Key>
__device__ __forceinline__ void xcd_order(const Key &key, uint32_t items, uint32_t *__restrict__ order) {
  __shared__ uint32_t counts[kOrderKeys];
  __shared__ uint32_t waveTotals[kOrderThreads / 64];
  __shared__ uint8_t staged[kOrderStaged];
  const uint32_t x = blockIdx.x, n = items / kRasterXcds;
  for (uint32_t k = threadIdx.x; k < kOrderKeys; k += kOrderThreads) counts[k] = 0;
  __syncthreads();
  // Every lane runs every trip, so that the ballots see whole waves.
  for (uint32_t start = 0; start < n; start += kOrderThreads) {
    const uint32_t i = start + threadIdx.x;
    const bool valid = i < n;
    const uint32_t k = valid ? key(i * kRasterXcds + x) : 0u;
    if (valid && i < kOrderStaged) staged[i] = static_cast<uint8_t>(k);
    (void)key_place(counts, k, valid);
  }
  __syncthreads();
  const uint32_t c = threadIdx.x < kOrderKeys ? counts[threadIdx.x] : 0u;
  uint32_t before;
  block_exclusive_sum(c, before, waveTotals);
  if (threadIdx.x < kOrderKeys) counts[threadIdx.x] = before;
  __syncthreads();
  for (uint32_t start = 0; start < n; start += kOrderThreads) {
    const uint32_t i = start + threadIdx.x;
    const bool valid = i < n;
    const uint32_t k = !valid ? 0u : i < kOrderStaged ? staged[i] : key(i * kRasterXcds + x);
    const uint32_t j = key_place(counts, k, valid);
    if (valid) order[j * kRasterXcds + x] = i * kRasterXcds + x;
  }
}

// The backward's key: the entries the forward found that block walks.
struct WorkKey {
  const uint32_t *work;
  __device__ uint32_t operator()(uint32_t h) const { return heavy_first(work[h]); }
};

// The forward's key: the length of the block's tile list (block_geometry's
// mapping from launch index to tile), which the forward's walk follows.
struct ListKey {
  const uint2 *ranges;
  uint32_t tiles, perTile;
  __device__ uint32_t operator()(uint32_t h) const {
    const uint32_t tile = (h / kRasterXcds / perTile) * kRasterXcds + h % kRasterXcds;
    if (tile >= tiles) return kOrderKeys - 1u;
    const uint2 r = ranges[tile];
    return heavy_first(r.y - r.x);
  }
};

__global__ __launch_bounds__(kOrderThreads) void work_order_kernel(const uint32_t *__restrict__ work, uint32_t items,
                                                                    uint32_t *__restrict__ order) {
  xcd_order(WorkKey{work}, items, order);
}

__global__ __launch_bounds__(kOrderThreads) void list_order_kernel(const uint2 *__restrict__ ranges, uint32_t tiles, uint32_t perTile,
                                                                    uint32_t items, uint32_t *__restrict__ order) {
  xcd_order(ListKey{ranges, tiles, perTile}, items, order);
}
} // namespace

void launch_work_order(hipStream_t stream, const uint32_t *work, uint32_t items, uint32_t *order) {
  if (items == 0) return;
  hipLaunchKernelGGL(work_order_kernel, dim3(kRasterXcds), dim3(kOrderThreads), 0, stream, work, items, order);
}

void launch_list_order(hipStream_t stream, const uint2 *ranges, uint32_t tiles, uint32_t tileW, uint32_t tileH, uint32_t *order) {
  const uint32_t items = raster_blocks(tiles, tileW, tileH);
  if (items == 0) return;
  hipLaunchKernelGGL(list_order_kernel, dim3(kRasterXcds), dim3(kOrderThreads), 0, stream, ranges, tiles, (tileW / 8u) * (tileH / 8u), items,
                     order);
}


// Calls LAUNCH(TW, TH) with the tile shape as compile-time constants.
#define VSPLAT_TILE_DISPATCH(tileW, tileH, LAUNCH)                                                                                 \
  if ((tileW) == 8 && (tileH) == 8) {                                                                                              \
    LAUNCH(8, 8);                                                                                                                  \
  } else if ((tileW) == 32 && (tileH) == 8) {                                                                                      \
    LAUNCH(32, 8);                                                                                                                 \
  } else if ((tileW) == 32 && (tileH) == 32) {                                                                                     \
    LAUNCH(32, 32);                                                                                                                \
  } else {                                                                                                                         \
    LAUNCH(16, 16);                                                                                                                \
  }

void launch_forward(hipStream_t stream, const Splat *splats, const uint32_t *entryKeys, const uint32_t *entryValues, uint32_t tileBits,
                    const uint2 *ranges, uint32_t width, uint32_t height, uint32_t tileW, uint32_t tileH, const float background[3],
                    float4 *image, uint32_t *stops, uint32_t *work, const uint32_t *order, bool batch) {
  const uint32_t gridW = (width + tileW - 1) / tileW, gridH = (height + tileH - 1) / tileH;
  if (wide_blocks(raster_blocks(gridW * gridH, tileW, tileH), batch)) {
    hipLaunchKernelGGL(forward_wide_kernel, dim3(raster_blocks(gridW * gridH, tileW, tileH)), dim3(kWideThreads), 0, stream, splats, entryKeys,
                       entryValues, tileBits, ranges, width, height, tileW, tileH, gridW, background[0], background[1], background[2],
                       reinterpret_cast<float *>(image), stops, work, order);
    return;
  }
#define VSPLAT_FORWARD(W, H)                                                                                                       \
  hipLaunchKernelGGL((forward_kernel<W, H>), dim3(raster_blocks(gridW * gridH, W, H)), dim3(kBlock), 0, stream, splats, entryKeys,   \
                     entryValues, tileBits, ranges, width, height, gridW, background[0], background[1], background[2], image, stops, work,  \
                     order)
  VSPLAT_TILE_DISPATCH(tileW, tileH, VSPLAT_FORWARD)
#undef VSPLAT_FORWARD
}

void launch_backward(hipStream_t stream, bool fixedPoint, bool recompute, const Splat *splats, const uint32_t *entryKeys,
                     const uint32_t *entryValues, uint32_t tileBits, const uint2 *ranges, uint32_t width, uint32_t height, uint32_t tileW,
                     uint32_t tileH, const float background[3], const float4 *image, const float4 *adjoint, const uint32_t *stops,
                     float fixedScale, int64_t *rawFixed, float *rawFloat, uint8_t *touched, const float *edge, const uint32_t *order,
                     bool batch) {
  const uint32_t gridW = (width + tileW - 1) / tileW, gridH = (height + tileH - 1) / tileH;
  const bool score = edge != nullptr;
  const int variant = (fixedPoint ? 4 : 0) | (recompute ? 2 : 0) | (score ? 1 : 0);
  if (wide_blocks(raster_blocks(gridW * gridH, tileW, tileH), batch)) {
#define VSPLAT_BACKWARD_WIDE(F, R, S)                                                                                               \
  hipLaunchKernelGGL((backward_wide_kernel<F, R, S>), dim3(raster_blocks(gridW * gridH, tileW, tileH)), dim3(kWideThreads), 0, stream, \
                     splats, entryKeys, entryValues, tileBits, ranges, width, height, tileW, tileH, gridW, background[0], background[1], \
                     background[2], image, adjoint, stops, fixedScale, reinterpret_cast<unsigned long long *>(rawFixed), rawFloat, touched, edge, order)
    switch (variant) {
    case 7: VSPLAT_BACKWARD_WIDE(true, true, true); break;
    case 6: VSPLAT_BACKWARD_WIDE(true, true, false); break;
    case 5: VSPLAT_BACKWARD_WIDE(true, false, true); break;
    case 4: VSPLAT_BACKWARD_WIDE(true, false, false); break;
    case 3: VSPLAT_BACKWARD_WIDE(false, true, true); break;
    case 2: VSPLAT_BACKWARD_WIDE(false, true, false); break;
    case 1: VSPLAT_BACKWARD_WIDE(false, false, true); break;
    default: VSPLAT_BACKWARD_WIDE(false, false, false); break;
    }
#undef VSPLAT_BACKWARD_WIDE
    return;
  }
#define VSPLAT_BACKWARD_SHAPE(F, R, S, W, H)                                                                                       \
  hipLaunchKernelGGL((backward_kernel<F, R, S, W, H>), dim3(raster_blocks(gridW * gridH, W, H)), dim3(kBlock), 0, stream, splats,   \
                     entryKeys, entryValues, tileBits, ranges, width, height, gridW, background[0], background[1], background[2], image, \
                     adjoint, stops, fixedScale, reinterpret_cast<unsigned long long *>(rawFixed), rawFloat, touched, edge, order)
#define VSPLAT_BACKWARD_TTT(W, H) VSPLAT_BACKWARD_SHAPE(true, true, true, W, H)
#define VSPLAT_BACKWARD_TTF(W, H) VSPLAT_BACKWARD_SHAPE(true, true, false, W, H)
#define VSPLAT_BACKWARD_TFT(W, H) VSPLAT_BACKWARD_SHAPE(true, false, true, W, H)
#define VSPLAT_BACKWARD_TFF(W, H) VSPLAT_BACKWARD_SHAPE(true, false, false, W, H)
#define VSPLAT_BACKWARD_FTT(W, H) VSPLAT_BACKWARD_SHAPE(false, true, true, W, H)
#define VSPLAT_BACKWARD_FTF(W, H) VSPLAT_BACKWARD_SHAPE(false, true, false, W, H)
#define VSPLAT_BACKWARD_FFT(W, H) VSPLAT_BACKWARD_SHAPE(false, false, true, W, H)
#define VSPLAT_BACKWARD_FFF(W, H) VSPLAT_BACKWARD_SHAPE(false, false, false, W, H)
  switch (variant) {
  case 7: VSPLAT_TILE_DISPATCH(tileW, tileH, VSPLAT_BACKWARD_TTT) break;
  case 6: VSPLAT_TILE_DISPATCH(tileW, tileH, VSPLAT_BACKWARD_TTF) break;
  case 5: VSPLAT_TILE_DISPATCH(tileW, tileH, VSPLAT_BACKWARD_TFT) break;
  case 4: VSPLAT_TILE_DISPATCH(tileW, tileH, VSPLAT_BACKWARD_TFF) break;
  case 3: VSPLAT_TILE_DISPATCH(tileW, tileH, VSPLAT_BACKWARD_FTT) break;
  case 2: VSPLAT_TILE_DISPATCH(tileW, tileH, VSPLAT_BACKWARD_FTF) break;
  case 1: VSPLAT_TILE_DISPATCH(tileW, tileH, VSPLAT_BACKWARD_FFT) break;
  default: VSPLAT_TILE_DISPATCH(tileW, tileH, VSPLAT_BACKWARD_FFF) break;
  }
#undef VSPLAT_BACKWARD_FFF
#undef VSPLAT_BACKWARD_FFT
#undef VSPLAT_BACKWARD_FTF
#undef VSPLAT_BACKWARD_FTT
#undef VSPLAT_BACKWARD_TFF
#undef VSPLAT_BACKWARD_TFT
#undef VSPLAT_BACKWARD_TTF
#undef VSPLAT_BACKWARD_TTT
#undef VSPLAT_BACKWARD_SHAPE
}

// The batched raster launches: one grid over every view's 8x8 blocks.
void launch_forward_views(hipStream_t stream, const RasterViews &views, uint32_t tileW, uint32_t tileH, const float background[3]) {
  if (views.count == 0) return;
  const uint32_t blocks = views.view[views.count - 1].firstBlock + views.view[views.count - 1].blocks;
#define VSPLAT_FORWARD_VIEWS(W, H)                                                                                                 \
  hipLaunchKernelGGL((forward_views_kernel<W, H>), dim3(blocks), dim3(kBlock), 0, stream, views, background[0], background[1],      \
                     background[2])
  VSPLAT_TILE_DISPATCH(tileW, tileH, VSPLAT_FORWARD_VIEWS)
#undef VSPLAT_FORWARD_VIEWS
}

void launch_backward_views(hipStream_t stream, bool fixedPoint, bool recompute, const RasterViews &views, uint32_t tileW, uint32_t tileH,
                           const float background[3]) {
  if (views.count == 0) return;
  const uint32_t blocks = views.view[views.count - 1].firstBlock + views.view[views.count - 1].blocks;
#define VSPLAT_BACKWARD_VIEWS_SHAPE(F, R, W, H)                                                                                     \
  hipLaunchKernelGGL((backward_views_kernel<F, R, W, H>), dim3(blocks), dim3(kBlock), 0, stream, views, background[0], background[1], \
                     background[2])
#define VSPLAT_BACKWARD_VIEWS_TT(W, H) VSPLAT_BACKWARD_VIEWS_SHAPE(true, true, W, H)
#define VSPLAT_BACKWARD_VIEWS_TF(W, H) VSPLAT_BACKWARD_VIEWS_SHAPE(true, false, W, H)
#define VSPLAT_BACKWARD_VIEWS_FT(W, H) VSPLAT_BACKWARD_VIEWS_SHAPE(false, true, W, H)
#define VSPLAT_BACKWARD_VIEWS_FF(W, H) VSPLAT_BACKWARD_VIEWS_SHAPE(false, false, W, H)
  if (fixedPoint && recompute) {
    VSPLAT_TILE_DISPATCH(tileW, tileH, VSPLAT_BACKWARD_VIEWS_TT)
  } else if (fixedPoint) {
    VSPLAT_TILE_DISPATCH(tileW, tileH, VSPLAT_BACKWARD_VIEWS_TF)
  } else if (recompute) {
    VSPLAT_TILE_DISPATCH(tileW, tileH, VSPLAT_BACKWARD_VIEWS_FT)
  } else {
    VSPLAT_TILE_DISPATCH(tileW, tileH, VSPLAT_BACKWARD_VIEWS_FF)
  }
#undef VSPLAT_BACKWARD_VIEWS_FF
#undef VSPLAT_BACKWARD_VIEWS_FT
#undef VSPLAT_BACKWARD_VIEWS_TF
#undef VSPLAT_BACKWARD_VIEWS_TT
#undef VSPLAT_BACKWARD_VIEWS_SHAPE
}

} // namespace vsplat
