// mpm_kernels.hip — gfx950 kernels of the MLS-MPM substep.
//
// One substep over every active scene of a world (device data in WorldDev):
//   k_clear         clear hash regions, block tables and counters, then
//   k_keys_touch    per particle: block key; per block that a workgroup meets, insertion
//                   of it and its 7 +1 neighbours (both only for the first substep
//                   and after the host changed the arena or the tables: otherwise the
//                   previous substep's k_g2p_update made the keys and insertions)
//   k_scan_slots    single-pass scan of occupied hash slots -> dense block ids
//   k_block_count   per block: dense ids of the 7 +1 and 7 -1 neighbours, collider mask;
//                   per particle: dense block id, wave-aggregated block counts and ranks
//   k_scan_counts   single-pass scan of block counts -> first particle of each block
//   k_scatter       per particle: sorted position (block-major permutation)
//   k_cell_order    now and then: the order of the particles inside their blocks
//   k_p2g           per block: LDS-staged scatter of its particles into a 6^3 node tile
//   k_grid_update   per node: sum of the tiles covering it, momentum -> velocity, gravity,
//                   clamp, cuboid colliders; empties the hash
//   k_g2p_update    per sorted particle: 27-node gather + deformation / constitutive update,
//                   written in sorted order to the output arena; then the next substep's
//                   block keys and insertions
// CPIC worlds add the contact fields (k_mesh_cdf, k_grid_cdf, k_particle_cdf) before P2G,
// the CPIC variants of the transfers, and k_g2p_contact before k_g2p_update.
// The reference runs the same stages as ~21 dispatches (src_mpm/pipeline.rs:385-526).
#include <type_traits>

#include <hip/hip_ext.h>

#include "mpm_kernels.h"

namespace nxm {

// ------------------------------------------------------------------------------------
// Wave helpers (wave64).

__device__ inline uint32_t lane_id() { return __lane_id(); }

__device__ inline uint64_t lanes_le(uint32_t l) { return l == 63 ? ~0ull : ((2ull << l) - 1ull); }

// Index of the run head at or below this lane given the 64-bit mask of run heads.
__device__ inline uint32_t run_head(uint64_t heads, uint32_t l)
{
    uint64_t m = heads & lanes_le(l);
    return 63u - (uint32_t)__clzll(m);
}

// Index one past the end of the run starting at head h.
__device__ inline uint32_t run_end(uint64_t heads, uint32_t h)
{
    uint64_t above = h == 63 ? 0ull : (heads & ~lanes_le(h));
    return above ? (uint32_t)__ffsll((unsigned long long)above) - 1u : 64u;
}

// XCD-contiguous work ranges.  Workgroups are dealt to the 8 XCDs round-robin
// (workgroup i runs on XCD i mod 8), and each XCD has its own L2.  Renumbering the
// workgroups so that those of one XCD are consecutive, and giving each a contiguous
// range of the (Morton-ordered) work, keeps neighbouring blocks and their particles in
// the same L2.  The grid must be a multiple of 8 workgroups.
constexpr uint32_t NUM_XCD = 8;

// Workgroup size of k_g2p_update (one particle per thread): two waves, measured fastest for
// the plain kernel (256: sand column G2P 1 us, clumped fluid 5-7 % slower; 192: the fluid 6 %
// slower; 64 and 512 slower too); CPIC worlds keep 256 (128: the
// same from 60,000 to 1M particles, 2 % faster at 262,144).
template <bool CPIC> constexpr int g2p_threads() { return CPIC ? 256 : 128; }

__device__ inline void xcd_range(uint32_t n, uint32_t &begin, uint32_t &end)
{
    const uint32_t g = gridDim.x, b = blockIdx.x;
    const uint32_t logical = (g % NUM_XCD == 0) ? (b % NUM_XCD) * (g / NUM_XCD) + b / NUM_XCD : b;
    // Balanced split: every workgroup gets floor(n / g) or ceil(n / g) items.
    const uint32_t q = n / g, more = n - q * g;
    begin = logical * q + min(logical, more);
    end = begin + q + (logical < more ? 1u : 0u);
}

// ------------------------------------------------------------------------------------
// Hash regions: open addressing, double hashing, 32-bit packed block keys
// (src_mpm_shaders/grid/grid.rs:447-536).  Values are dense block ids.

__device__ inline bool hash_insert(uint32_t *keys, uint32_t mask, uint32_t key, uint32_t &slot)
{
    const HashProbe p = hash_probe(key, mask);
    uint32_t s = p.slot;
    for (uint32_t probe = 0; probe <= mask; ++probe) {
        uint32_t prev = atomicCAS(keys + s, EMPTY_KEY, key);
        if (prev == EMPTY_KEY) { slot = s; return true; }
        if (prev == key) { slot = s; return false; }
        s = (s + p.stride) & mask;
    }
    slot = NONE;
    return false;
}

__device__ inline uint32_t hash_find(const uint32_t *keys, const uint32_t *vals, uint32_t mask, uint32_t key)
{
    const HashProbe p = hash_probe(key, mask);
    uint32_t s = p.slot;
    for (uint32_t probe = 0; probe <= mask; ++probe) {
        uint32_t k = keys[s];
        if (k == key) return vals[s];
        if (k == EMPTY_KEY) return NONE;
        s = (s + p.stride) & mask;
    }
    return NONE;
}

__device__ inline uint32_t find_block(const WorldDev &w, const SceneDev &sc, int32_t x, int32_t y, int32_t z)
{
    return hash_find(w.hkeys + sc.h_base, w.hvals + sc.h_base, sc.h_cap - 1u, pack_vid(x, y, z));
}

// Key of a particle that cannot get a block: the x field 0x7FF never occurs for
// in-range blocks or their +1 neighbours.
constexpr uint32_t OVERFLOW_KEY = 0x000007FFu;

// ------------------------------------------------------------------------------------
// Block building without counters: keys are inserted into the scenes' hash regions,
// then the occupied slots are compacted by a prefix scan into dense block ids.  Each
// region ends with one virtual slot, always occupied, that becomes the scene's
// overflow block, so the dense ids of a scene are contiguous and end with it.

__device__ inline uint32_t scene_of_slot(const WorldDev &w, uint32_t j)
{
    // last active region whose start is <= j
    uint32_t lo = 0, hi = w.n_regions;
    while (hi - lo > 1) {
        uint32_t mid = (lo + hi) >> 1;
        if (w.region_start[mid] <= j) lo = mid; else hi = mid;
    }
    return w.region_scene[lo];
}

__device__ inline int4 unpack_vid(uint32_t key)
{
    return make_int4((int)(key & 0x7FFu) - 0x3FF, (int)((key >> 11) & 0x3FFu) - 0x1FF, (int)(key >> 21) - 0x3FF, 0);
}

__host__ __device__ inline uint32_t clear_len(const WorldDev &w)
{
    const uint32_t a = w.h_total > w.b_total ? w.h_total : w.b_total;
    const uint32_t b = 2u * w.scan_stride > w.s_count ? 2u * w.scan_stride : w.s_count;
    return a > b ? a : b;
}
__device__ inline void clear_tables(const WorldDev &w)
{
    const uint32_t n = clear_len(w);
    for (uint32_t i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += gridDim.x * blockDim.x) {
        if (i < w.h_total) { w.hkeys[i] = EMPTY_KEY; w.hmark[i] = 0u; }
        if (i < w.b_total) w.bnp[i] = 0u;
        if (i < 2u * w.scan_stride) w.scan_state[i] = 0ull;
        if (i == 0) { w.g->p_out = 0u; w.g->n_blocks = 0u; w.g->ticket[0] = 0u; w.g->ticket[1] = 0u; }
        if (w.clock && i < w.s_count) w.clock[i].bound = NONE;   // recomputed by the key pass's bound
    }
}
__global__ void k_clear(WorldDev w) { clear_tables(w); }

// Row i of an array of three-component rows.
__device__ inline f3 load3(const float *p, size_t i) { return mk3(p[3 * i], p[3 * i + 1], p[3 * i + 2]); }
__device__ inline void store3(float *p, size_t i, f3 v)
{
    p[3 * i] = v.x;
    p[3 * i + 1] = v.y;
    p[3 * i + 2] = v.z;
}

// One particle's P2G inputs.
struct P2GIn {
    float px, py, pz, m;
    f3 v;
    m3 C;
    uint32_t flags;
};

__device__ inline P2GIn p2g_load(const WorldDev &w, uint32_t slot)
{
    const float4 q0 = w.in.quad(0)[slot], q1 = w.in.quad(1)[slot], q2 = w.in.quad(2)[slot], q3 = w.in.quad(3)[slot],
                 q4 = w.in.quad(4)[slot];
    P2GIn p;
    p.px = q0.x; p.py = q0.y; p.pz = q0.z;
    p.flags = __float_as_uint(q0.w);
    p.v = mk3(q1.x, q1.y, q1.z);
    p.C.c0 = mk3(q2.x, q2.y, q2.z);
    p.C.c1 = mk3(q2.w, q3.x, q3.y);
    p.C.c2 = mk3(q3.z, q3.w, q4.x);
    p.m = q4.y;
    return p;
}

// Bounds of a particle's P2G contributions, |m v + C dpt| (|dpt_j| <= 1.5 h) and m, as the
// exponents of the powers of two above them: the low half and the high half of one word, 0
// for none.  A bound that is not finite counts as none, so that a block's scale is that of
// its other particles (p2g_one checks every contribution of such a particle); NaN
// components are left out, as fmaxf does.  Made where a particle's key is made, from the
// state still in registers; the count kernel takes a block's maxima, so that P2G reads a
// block's particles once.
constexpr int CODE_BIAS = 200;
__device__ inline uint32_t bound_code(float b)
{
    if (!(b > 0.0f) || !isfinite(b)) return 0u;
    int e;
    (void)frexpf(b, &e);   // b = m 2^e, m in [0.5, 1): b < 2^e
    return (uint32_t)(e + CODE_BIAS);
}
__device__ inline uint32_t bound_codes(f3 v, const m3 &C, float m, float h)
{
    const float cmax = fmaxf(fmaxf(fabsf(C.c0.x), fmaxf(fabsf(C.c0.y), fabsf(C.c0.z))),
                             fmaxf(fmaxf(fabsf(C.c1.x), fmaxf(fabsf(C.c1.y), fabsf(C.c1.z))),
                                   fmaxf(fabsf(C.c2.x), fmaxf(fabsf(C.c2.y), fabsf(C.c2.z)))));
    const float vmax = fmaxf(fabsf(v.x), fmaxf(fabsf(v.y), fabsf(v.z)));
    const float am = fabsf(m);
    return bound_code(__builtin_fmaf(4.5f * h, cmax, am * vmax)) | (bound_code(am) << 16);
}

// Block key of particle slot i at position (x, y, z) of active scene s; its bound codes go
// to prank[i] and its scene to pdense[i].
__device__ inline uint32_t particle_key(const WorldDev &w, uint32_t i, bool valid, uint32_t s, float x, float y, float z,
                                        uint32_t codes)
{
    if (!valid) return EMPTY_KEY;
    const SceneDev sc = w.scenes[s];
    int32_t bx, by, bz;
    uint32_t lx, ly, lz, key = OVERFLOW_KEY;
    cell_of(x, sc.h, sc.inv_h, bx, lx);
    cell_of(y, sc.h, sc.inv_h, by, ly);
    cell_of(z, sc.h, sc.inv_h, bz, lz);
    if (vid_in_range(bx, by, bz)) key = pack_vid(bx, by, bz);
    else atomicOr(&w.ctr[s].err, ERR_DOMAIN);
    w.prank[i] = codes;
    w.pdense[i] = s;
    return key;
}

// The first lane of a run of neighbours in the wave with one (scene, key).  Invalid lanes
// are passed over: CPIC's contact particles, which another kernel keys, lie all through the
// waves of the plain ones.
__device__ inline bool run_starts(bool valid, uint32_t s, uint32_t key)
{
    const uint64_t before = __ballot(valid) & (lanes_le(lane_id()) >> 1);
    const int prev = before ? 63 - __clzll((long long)before) : 0;
    const uint32_t pk = __shfl(key, prev, WAVE), ps = __shfl(s, prev, WAVE);
    return valid && key != OVERFLOW_KEY && (!before || pk != key || ps != s);
}

// The key words of particle slot i (particle_key), its block's hash slot (to pslot[i]) and the wave's block insertions:
// adjacent lanes with the same (scene, key) form a run; each run inserts its block (marked primary) and the block's 7 +1
// neighbours (the active set is P + {0,1}^3, src_mpm/grid/grid.rs:193-200).  Called by
// every lane of a wave together (invalid lanes with valid = false), so that the lanes'
// neighbours in the wave are the particles' neighbours in the arena.
__device__ inline void touch_keys(const WorldDev &w, uint32_t i, bool valid, uint32_t s, float x, float y, float z,
                                  uint32_t codes)
{
    const uint32_t l = lane_id();
    const uint32_t key = particle_key(w, i, valid, s, x, y, z, codes);
    const bool head = run_starts(valid, s, key);
    // Up to 8 runs per round: lane l inserts neighbour (l mod 8) of run (l / 8), so a
    // wave's insertions overlap instead of waiting for each other's atomics.
    uint64_t heads = __ballot(head);
    const uint64_t up_to = heads & lanes_le(l);
    const uint32_t run = (uint32_t)__popcll(up_to) - 1u;   // this lane's run, if it has a key
    uint32_t mine = NONE;
    for (uint32_t first = 0; heads; first += 8u) {
        uint32_t hsrc[8];
        #pragma unroll
        for (int k = 0; k < 8; ++k) {
            hsrc[k] = heads ? (uint32_t)__ffsll((unsigned long long)heads) - 1u : 64u;
            heads = heads ? heads & (heads - 1ull) : 0ull;
        }
        const uint32_t r = l >> 3, j = l & 7u;
        uint32_t src = hsrc[0];
        #pragma unroll
        for (int k = 1; k < 8; ++k) src = r == (uint32_t)k ? hsrc[k] : src;
        const uint32_t hk = __shfl(key, (int)(src & 63u), WAVE);
        const uint32_t hs = __shfl(s, (int)(src & 63u), WAVE);
        uint32_t at = NONE;
        if (src < 64u) {
            const SceneDev hsc = w.scenes[hs];
            const int4 v = unpack_vid(hk);
            uint32_t slot;
            hash_insert(w.hkeys + hsc.h_base, hsc.h_cap - 1u,
                        pack_vid(v.x + ASSOC[j][0], v.y + ASSOC[j][1], v.z + ASSOC[j][2]), slot);
            if (slot == NONE) atomicOr(&w.ctr[hs].err, ERR_GRID_CAPACITY);
            else {
                at = hsc.h_base + slot;
                if (j == 0) w.hmark[at] = 1u;
            }
        }
        const uint32_t got = __shfl(at, (int)(((run - first) & 7u) * 8u), WAVE);
        if (run - first < 8u) mine = got;
    }
    if (valid) w.pslot[i] = key == OVERFLOW_KEY ? NONE : mine;
}

// The virtual overflow slot closing each active scene's hash region.
__device__ inline void mark_overflow_slots(const WorldDev &w)
{
    for (uint32_t s = blockIdx.x * blockDim.x + threadIdx.x; s < w.s_count; s += gridDim.x * blockDim.x) {
        const SceneDev sc = w.scenes[s];
        if (sc.active) w.hkeys[sc.h_base + sc.h_cap] = OVERFLOW_KEY;
    }
}

// Keys and block insertions of particles in the order the host or a caller has them.  Blocks
// come back every few lines of such an order, or all through it, and an insertion is an
// atomic on its slot: by runs, as touch_keys does them, one slot took thousands.  So a
// workgroup of KEY_GROUP takes consecutive particles and keeps the blocks it has met in a
// set in LDS.  A block new to the set is looked up, and one found marked is left alone (keys
// and marks only ever turn on, so a stale line can only send a workgroup the long way); the
// workgroup whose atomic marks it inserts its 7 neighbours.  Against eight insertions per
// run, with 256 threads: 1M particles in random order 496 -> 326 us, 2M in clumps 1322 -> 161.
// (Groups of 256 and 1024 took as long for the clumps, and a call of 1000 particles 1-2 us
// more with 1024.)
constexpr int KEY_GROUP = 512;
struct KeySet {
    static constexpr uint32_t SIZE = 2 * KEY_GROUP;
    static_assert(SIZE == 1024, "add() takes a 10-bit hash");
    static constexpr unsigned long long EMPTY = ~0ull;
    unsigned long long entry[SIZE];  // scene << 32 | key
    uint32_t slot[SIZE];             // its place in the hash
    uint16_t fresh[KEY_GROUP];       // entered since the last insert()
    uint16_t marked[KEY_GROUP];      // those of them that this workgroup marked
    uint32_t count, n_fresh, n_marked;
    __device__ void clear()
    {
        for (uint32_t k = threadIdx.x; k < SIZE; k += KEY_GROUP) entry[k] = EMPTY;
        if (threadIdx.x == 0) count = n_fresh = n_marked = 0u;
        __syncthreads();
    }
    // One (scene, key), by any lane; at most KEY_GROUP between two calls of insert().
    __device__ uint32_t add(uint32_t s, uint32_t key)
    {
        const unsigned long long e = ((unsigned long long)s << 32) | key;
        uint32_t at = (key ^ (key >> 11) * 0x9E3779B9u ^ s * 0x85EBCA6Bu) * 0x9E3779B9u >> 22;
        for (;; at = (at + 1u) % SIZE) {   // ends: the set is at most half full before a round
            const unsigned long long prev = atomicCAS(&entry[at], EMPTY, e);
            if (prev == e) return at;
            if (prev == EMPTY) break;
        }
        fresh[atomicAdd(&n_fresh, 1u)] = (uint16_t)at;
        return at;
    }
    // The new blocks, marked primary, and their +1 neighbours into the hash.
    __device__ void insert(const WorldDev &w)
    {
        __syncthreads();
        const uint32_t n = n_fresh;
        if (threadIdx.x < n) {
            const uint32_t at = fresh[threadIdx.x];
            const unsigned long long e = entry[at];
            const uint32_t s = (uint32_t)(e >> 32), key = (uint32_t)e;
            const SceneDev &sc = w.scenes[s];
            uint32_t *keys = w.hkeys + sc.h_base, *marks = w.hmark + sc.h_base;
            uint32_t to = hash_probe(key, sc.h_cap - 1u).slot;
            if (look(keys + to) != key || look(marks + to) == 0u) {
                hash_insert(keys, sc.h_cap - 1u, key, to);
                if (to == NONE) atomicOr(&w.ctr[s].err, ERR_GRID_CAPACITY);
                if (to == NONE || atomicExch(marks + to, 1u) == 0u) marked[atomicAdd(&n_marked, 1u)] = (uint16_t)at;
            }
            slot[at] = to == NONE ? NONE : sc.h_base + to;
        }
        __syncthreads();
        const uint32_t m = n_marked;
        for (uint32_t t = threadIdx.x; t < 8u * m; t += KEY_GROUP) {
            const uint32_t j = t & 7u;
            if (j == 0u) continue;
            const unsigned long long e = entry[marked[t >> 3]];
            const uint32_t s = (uint32_t)(e >> 32);
            const SceneDev &sc = w.scenes[s];
            const int4 v = unpack_vid((uint32_t)e);
            uint32_t to;
            hash_insert(w.hkeys + sc.h_base, sc.h_cap - 1u,
                        pack_vid(v.x + ASSOC[j][0], v.y + ASSOC[j][1], v.z + ASSOC[j][2]), to);
            if (to == NONE) atomicOr(&w.ctr[s].err, ERR_GRID_CAPACITY);
        }
    }
    // Between two rounds: the set empty if the next could fill it.
    __device__ void next()
    {
        __syncthreads();
        const bool full = count + n_fresh > SIZE / 2u;
        __syncthreads();
        if (threadIdx.x == 0) {
            count += n_fresh;
            n_fresh = n_marked = 0u;
        }
        __syncthreads();
        if (full) clear();
    }
    // One particle of a round (by every thread of the workgroup): its key words, block and
    // hash slot.
    __device__ void particle(const WorldDev &w, uint32_t i, bool valid, uint32_t s, f3 x, uint32_t codes)
    {
        const uint32_t key = particle_key(w, i, valid, s, x.x, x.y, x.z, codes);
        const bool head = run_starts(valid, s, key);
        uint32_t at = 0u;
        if (head) at = add(s, key);
        const uint64_t heads = __ballot(head) & lanes_le(lane_id());
        at = __shfl(at, heads ? 63 - __clzll((long long)heads) : 0, WAVE);
        insert(w);
        if (valid) w.pslot[i] = key == OVERFLOW_KEY ? NONE : slot[at];
        next();
    }
    __device__ static uint32_t look(const uint32_t *p)
    {
        return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WAVEFRONT);
    }
};
// The particles of a key workgroup: [begin, end), whole rounds of KEY_GROUP.
__device__ inline void key_range(uint32_t n, uint32_t &begin, uint32_t &end)
{
    const uint32_t rounds = (n + KEY_GROUP - 1u) / KEY_GROUP, per = (rounds + gridDim.x - 1u) / gridDim.x;
    const uint32_t r = min(blockIdx.x * per, rounds);
    begin = r * KEY_GROUP;
    end = min(min(r + per, rounds) * KEY_GROUP, (n + WAVE - 1u) / WAVE * WAVE);
}

// Keys and block insertions of every particle of the input arena.  Used for a substep
// whose keys the previous substep's G2P did not insert (the first one, and after the
// host changed the arena or the tables): k_clear has emptied the hash and the counters
// before it.
__global__ void __launch_bounds__(KEY_GROUP) k_keys_touch(WorldDev w)
{
    __shared__ KeySet set;
    mark_overflow_slots(w);
    set.clear();
    const uint32_t n = w.g->p_in;
    uint32_t begin, end;
    key_range(n, begin, end);
    for (uint32_t c = begin; c < end; c += KEY_GROUP) {
        const uint32_t i = c + threadIdx.x;
        bool valid = i < n;
        uint32_t s = 0;
        float x = 0.0f, y = 0.0f, z = 0.0f;
        uint32_t codes = 0u;
        if (valid) {
            const P2GIn p = p2g_load(w, i);
            s = flags_scene(p.flags);
            valid = w.scenes[s].active != 0u;
            if (!valid) w.pdense[i] = s;   // the count kernel leaves it out
            x = p.px;
            y = p.py;
            z = p.pz;
            if (p.flags & FLAG_ENABLED) codes = bound_codes(p.v, p.C, p.m, w.scenes[s].h);
        }
        set.particle(w, i, valid, s, mk3(x, y, z), codes);
    }
}

// Exclusive scans: k_scan_slots numbers the occupied hash slots (dense block ids), slot_tile
// slots per tile; k_scan_counts sums the particles of each block (the first sorted position
// of each block), SCAN_TILE blocks per tile.
enum Scan { SCAN_SLOTS = 0, SCAN_COUNTS = 1 };   // ticket and state words
template <int ROWS, int WAVES> constexpr uint32_t slot_tile() { return ROWS * WAVES * WAVE; }
static_assert(slot_tile<4, 4>() >= SCAN_TILE, "scan_stride is sized for tiles of SCAN_TILE");

// Runs of SCAN_TILE elements per scan tile for a scan of len elements (at most
// SCAN_MAX_TILES tiles).
constexpr uint32_t SCAN_MAX_TILES = 4096;
__host__ __device__ inline uint32_t scan_chunks(uint32_t len)
{
    const uint32_t per = (uint32_t)SCAN_TILE * SCAN_MAX_TILES;
    return len <= per ? 1u : (uint32_t)(((uint64_t)len + per - 1) / per);
}

__device__ inline uint32_t block_reduce_256(uint32_t v, uint32_t *sh)
{
    for (int o = 32; o > 0; o >>= 1) v += __shfl_down(v, o, WAVE);
    if (lane_id() == 0) sh[threadIdx.x / WAVE] = v;
    __syncthreads();
    uint32_t t = sh[0] + sh[1] + sh[2] + sh[3];
    __syncthreads();
    return t;
}

// Inclusive wave scan.
__device__ inline uint32_t wave_incl_scan(uint32_t v)
{
    uint32_t l = lane_id();
    for (int o = 1; o < WAVE; o <<= 1) {
        uint32_t u = __shfl_up(v, o, WAVE);
        if (l >= (uint32_t)o) v += u;
    }
    return v;
}

// Exclusive scan over a 256-thread block, one element per thread.
__device__ inline uint32_t block_excl_scan_256(uint32_t v, uint32_t *sh, uint32_t &total)
{
    uint32_t incl = wave_incl_scan(v);
    uint32_t wv = threadIdx.x / WAVE;
    if (lane_id() == WAVE - 1) sh[wv] = incl;
    __syncthreads();
    uint32_t off = 0;
    for (uint32_t k = 0; k < wv; ++k) off += sh[k];
    total = sh[0] + sh[1] + sh[2] + sh[3];
    __syncthreads();
    return off + incl - v;
}

// Single-pass exclusive scan with decoupled look-back (Merrill and Garland, "Single-pass
// Parallel Prefix Scan with Decoupled Look-back", 2016).  Workgroups take tiles in ticket
// order, publish the tile's aggregate, then add the published values of the preceding
// tiles until one carries an inclusive prefix.  Status and value share one 64-bit word
// (bits 32-33: 1 aggregate, 2 inclusive prefix), so a reader sees both or neither.  A
// tile waits only for tiles with smaller tickets; those belong to workgroups already
// running, which publish their aggregate before waiting themselves, so every wait ends.
constexpr unsigned long long ST_AGG = 1ull << 32, ST_PREFIX = 2ull << 32;

__device__ inline void advance_clocks(const WorldDev &w);

// The look-back of tile t with the given total, by one wave, 64 predecessors at a time: lane
// l reads tile hi - l; the nearest tile with an inclusive prefix ends the walk once every
// tile up to it has published.  Returns the tile's exclusive prefix, in every lane.
__device__ inline uint32_t look_back(unsigned long long *state, uint32_t t, uint32_t total)
{
    const uint32_t l = lane_id();
    uint32_t prefix = 0;
    if (t > 0u) {
        if (l == 0) __hip_atomic_store(&state[t], ST_AGG | total, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        int64_t hi = (int64_t)t - 1;
        for (;;) {
            const int64_t j = hi - (int64_t)l;
            // Below tile 0 (never needed: tile 0 carries a prefix) read as prefix 0.
            const unsigned long long st =
                j >= 0 ? __hip_atomic_load(&state[j], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) : ST_PREFIX;
            const unsigned long long flag = st & (3ull << 32);
            const uint64_t pmask = __ballot(flag == ST_PREFIX);
            const uint32_t stop = pmask ? (uint32_t)__ffsll((unsigned long long)pmask) - 1u : 64u;
            const uint64_t need = stop >= 63u ? ~0ull : ((2ull << stop) - 1ull);
            if (__ballot(flag == 0ull) & need) continue;   // a tile in range has not published yet
            uint32_t val = l <= stop ? (uint32_t)st : 0u;
            for (int o = 32; o > 0; o >>= 1) val += __shfl_xor(val, o, WAVE);
            prefix += val;
            if (stop < 64u) break;
            hi -= 64;                                         // 64 aggregates: walk further back
        }
    }
    if (l == 0)
        __hip_atomic_store(&state[t], ST_PREFIX | (unsigned long long)(prefix + total), __ATOMIC_RELAXED,
                           __HIP_MEMORY_SCOPE_AGENT);
    return prefix;
}

// Tickets: a workgroup past the last tile takes none, and one that has had its tile is done
// when there are workgroups for all of them (a launch covers the allocated blocks, many times
// the occupied ones: every ticket is an atomic on one word).
__device__ inline uint32_t take_ticket(const WorldDev &w, Scan which, uint32_t *shared)
{
    __syncthreads();
    if (threadIdx.x == 0) *shared = atomicAdd(&w.g->ticket[which], 1u);
    __syncthreads();
    return *shared;
}

// Dense block ids of the occupied slots, and what a block starts its substep with.  Bound by
// latency and, on a large hash, by the tickets (20-30 ns each): a wave has ROWS rows of 64
// slots in flight, a ballot counts a row, and a tile has one barrier on each side of its
// look-back.  The tiles are small for a small hash and large for a large one (SMALL_HASH).
// Against a slot count per thread, four slots in flight and 1024 slots a tile at every size:
// 50,000 particles 7.4 -> 5.5 us, 32 scenes 16.4 -> 10.8, 1M sand 9.7 -> 7.6, 2M clumped
// particles (2^22 slots) 71 -> 23.
template <int ROWS, int WAVES>
__global__ void __launch_bounds__(WAVES * WAVE) k_scan_slots(WorldDev w)
{
    constexpr uint32_t SLOT_TILE = slot_tile<ROWS, WAVES>();
    if (blockIdx.x == 0) advance_clocks(w);   // the substep's first kernel
    __shared__ uint32_t sh[WAVES], s_tile, s_prefix;
    const uint32_t len = w.h_total, l = lane_id(), wave = __builtin_amdgcn_readfirstlane(threadIdx.x / WAVE);
    const uint32_t ntiles = min((len + SLOT_TILE - 1u) / SLOT_TILE, w.scan_stride - 1u);
    if (blockIdx.x >= ntiles) return;
    do {
        const uint32_t t = take_ticket(w, SCAN_SLOTS, &s_tile);
        if (t >= ntiles) break;
        const uint32_t first = t * SLOT_TILE + wave * (ROWS * WAVE);
        uint32_t key[ROWS], mark[ROWS];
        #pragma unroll
        for (int r = 0; r < ROWS; ++r) {
            const uint32_t i = first + r * WAVE + l;
            key[r] = i < len ? w.hkeys[i] : EMPTY_KEY;
            mark[r] = i < len ? w.hmark[i] : 0u;
        }
        // The scene of the wave's first slot, and where the next one's slots start.
        uint32_t region = 0u;
        for (uint32_t hi = w.n_regions; hi - region > 1u;) {
            const uint32_t mid = (region + hi) / 2u;
            if (ld_uniform(w.region_start + mid) <= first) region = mid; else hi = mid;
        }
        const uint32_t scene = ld_uniform(w.region_scene + region);
        const uint32_t next = region + 1u < w.n_regions ? ld_uniform(w.region_start + region + 1u) : NONE;
        uint32_t n = 0u;
        #pragma unroll
        for (int r = 0; r < ROWS; ++r) n += (uint32_t)__popcll(__ballot(key[r] != EMPTY_KEY));
        if (l == 0) sh[wave] = n;
        __syncthreads();
        if (wave == 0u) {
            uint32_t total = 0u;
            for (int k = 0; k < WAVES; ++k) total += sh[k];
            const uint32_t prefix = look_back(w.scan_state, t, total);
            if (l == 0) {
                s_prefix = prefix;
                if (t == ntiles - 1u) w.g->n_blocks = min(prefix + total, w.b_total);
            }
        }
        __syncthreads();
        uint32_t before = s_prefix;
        for (uint32_t k = 0; k < wave; ++k) before += sh[k];
        #pragma unroll
        for (int r = 0; r < ROWS; ++r) {
            const uint32_t i = first + r * WAVE + l;
            const uint64_t on = __ballot(key[r] != EMPTY_KEY);
            const uint32_t d = before + (uint32_t)__popcll(on & (lanes_le(l) >> 1));
            before += (uint32_t)__popcll(on);
            if (i >= len) continue;
            const bool taken = key[r] != EMPTY_KEY;
            w.hvals[i] = taken && d >= w.b_total ? NONE : d;
            if (!taken) continue;
            const uint32_t s = i < next ? scene : scene_of_slot(w, i);
            if (d >= w.b_total) {
                atomicOr(&w.ctr[s].err, ERR_GRID_CAPACITY);
                continue;
            }
            w.bscene[d] = s;
            // vid.w and bprim take the block's bound codes while its particles are counted
            // (bprim stays nonzero for a primary block).
            w.bvid[d] = key[r] == OVERFLOW_KEY ? make_int4(OVERFLOW_VID, 0, 0, 0) : unpack_vid(key[r]);
            w.bprim[d] = mark[r];
            // This substep's count starts at zero (k_block_count adds to it; the previous
            // substep's stay readable until here; only the dense ids handed out are read).
            w.bnp[d] = 0u;
        }
    } while (gridDim.x < ntiles);
}

// First sorted position of each block (2M clumped particles 30 -> 8 us without the tickets of
// the workgroups that have no tile).
__global__ void __launch_bounds__(256) k_scan_counts(WorldDev w)
{
    constexpr int PER = SCAN_TILE / 256;
    __shared__ uint32_t sh[4];
    __shared__ uint32_t s_tile, s_prefix;
    const uint32_t len = min(w.g->n_blocks, w.b_total);
    // A tile is `chunks` runs of SCAN_TILE elements, so that there are at most
    // SCAN_MAX_TILES tiles: every tile takes a ticket, one same-address atomic, and with
    // millions of blocks those tickets, not the data, would set the time.  The state
    // array has scan_stride words per scan (the host sizes it for SCAN_TILE tiles); the bound
    // keeps every tile's word inside it whatever the host passed.
    const uint32_t chunks = scan_chunks(len);
    const uint32_t tile_len = SCAN_TILE * chunks;
    const uint32_t ntiles = min((len + tile_len - 1) / tile_len, w.scan_stride - 1u);
    if (blockIdx.x >= ntiles) return;
    do {
        const uint32_t t = take_ticket(w, SCAN_COUNTS, &s_tile);
        if (t >= ntiles) break;
        // One run: thread elements i1 .. i1 + PER - 1, one block scan.  Several runs: element
        // i0 + 256 k of each run (k < PER) belongs to this thread, row k of the run being 256
        // consecutive elements, so that loads and stores are coalesced; a row's exclusive
        // scan plus the rows before it give the rank.
        uint32_t v[PER], sum = 0;
        const uint32_t i0 = t * tile_len + threadIdx.x, i1 = t * tile_len + PER * threadIdx.x;
        uint32_t total = 0, ex = 0;
        if (chunks == 1u) {
            #pragma unroll
            for (int k = 0; k < PER; ++k) {
                v[k] = i1 + k < len ? w.bnp[i1 + k] : 0u;
                sum += v[k];
            }
            ex = block_excl_scan_256(sum, sh, total);
        } else {
            // First pass: the tile's total; the second (below) reads the runs again.
            for (uint32_t c = 0; c < chunks; ++c) {
                const uint32_t ic = i0 + c * SCAN_TILE;
                #pragma unroll
                for (int k = 0; k < PER; ++k) {
                    const uint32_t i = ic + 256u * k;
                    sum += i < len ? w.bnp[i] : 0u;
                }
            }
            total = block_reduce_256(sum, sh);
        }
        if (threadIdx.x < WAVE) {
            const uint32_t prefix = look_back(w.scan_state + w.scan_stride, t, total);
            if (threadIdx.x == 0) {
                s_prefix = prefix;
                if (t == ntiles - 1) w.g->p_out = prefix + total;
            }
        }
        __syncthreads();
        if (chunks == 1u) {
            uint32_t r = s_prefix + ex;
            for (int k = 0; k < PER; ++k) {
                if (i1 + k < len) w.bfirst[i1 + k] = r;
                r += v[k];
            }
        } else {
            uint32_t run = s_prefix;
            for (uint32_t c = 0; c < chunks; ++c) {
                const uint32_t ic = i0 + c * SCAN_TILE;
                #pragma unroll
                for (int k = 0; k < PER; ++k) {
                    const uint32_t i = ic + 256u * k;
                    v[k] = i < len ? w.bnp[i] : 0u;
                }
                #pragma unroll
                for (int k = 0; k < PER; ++k) {
                    uint32_t rt;
                    const uint32_t e = block_excl_scan_256(v[k], sh, rt);
                    const uint32_t i = ic + 256u * k;
                    if (i < len) w.bfirst[i] = run + e;
                    run += rt;
                }
            }
        }
    } while (gridDim.x < ntiles);
}

// Per block, 16 threads: threads 0..7 look up the 8 blocks vid - {0,1}^3 (grid update
// sources), threads 8..15 the 8 blocks vid + {0,1}^3 (G2P tile, primaries only); thread j
// also tests collider j against the block (bounding spheres) for the collider mask.
__device__ inline void block_info_part(const WorldDev &w, uint32_t group, uint32_t groups)
{
    // Per scene: its dense block range; the last block of the range is the overflow block.
    for (uint32_t s = group * blockDim.x + threadIdx.x; s < w.s_count; s += groups * blockDim.x) {
        const SceneDev sc = w.scenes[s];
        if (!sc.active) continue;
        const uint32_t first = w.hvals[sc.h_base];
        const uint32_t last = w.hvals[sc.h_base + sc.h_cap];
        w.ctr[s].b_start = first;
        w.ctr[s].b_count = last == NONE ? 0u : last + 1u - first;
        if (last != NONE && last - first > sc.b_cap) atomicOr(&w.ctr[s].err, ERR_GRID_CAPACITY);
    }
    const uint64_t n = (uint64_t)w.g->n_blocks * 16;
    for (uint64_t t = (uint64_t)group * blockDim.x + threadIdx.x; t < n; t += (uint64_t)groups * blockDim.x) {
        const uint32_t d = (uint32_t)(t >> 4), j = (uint32_t)(t & 15);
        if (j == 0 && w.breach) w.breach[d] = 0u;   // set by k_grid_cdf (CPIC worlds)
        const int4 v = w.bvid[d];
        if (v.x == OVERFLOW_VID) continue;
        const SceneDev sc = w.scenes[w.bscene[d]];
        if (j < 8) {
            // Sources of the grid update: only primary blocks have a P2G staging tile.
            const uint32_t src = j == 0 ? d : find_block(w, sc, v.x - ASSOC[j][0], v.y - ASSOC[j][1], v.z - ASSOC[j][2]);
            w.bdn[8 * d + j] = (src != NONE && w.bprim[src]) ? src : NONE;
        } else if (w.bprim[d]) {
            const uint32_t i = j - 8;
            w.bup[8 * d + i] = i == 0 ? d : find_block(w, sc, v.x + ASSOC[i][0], v.y + ASSOC[i][1], v.z + ASSOC[i][2]);
        }
        // Collider mask: collider j can touch a node of this block only if its bounding
        // sphere (radius reach about the body origin) comes within 1.5 h (the projection
        // reach) of the block's node sphere.
        bool hit = false;
        if (j < sc.col_count) {
            const ColliderDev &c = w.cols[sc.col_start + j];
            const float h = sc.h;
            const f3 center = mk3(((float)(4 * v.x) + 1.5f) * h, ((float)(4 * v.y) + 1.5f) * h, ((float)(4 * v.z) + 1.5f) * h);
            const float rb = 1.5f * h * 1.7320509f;                  // node sphere of the block
            const float rc = c.reach;
            const f3 dc = center - mk3(c.t[0], c.t[1], c.t[2]);
            const float reach = rb + rc + 1.5f * h * 1.7320509f + 2.0f * h;
            hit = dot(dc, dc) <= reach * reach;
        }
        // 16 consecutive lanes of a wave hold one block: combine their bits.
        const uint64_t bits = __ballot(hit);
        if (j == 0) {
            const uint32_t lane0 = __lane_id() & ~15u;
            w.bmask[d] = (uint32_t)((bits >> lane0) & 0xFFFFull);
        }
    }
}

// Particles of input slot i's block counted: its block id (d, written to pdense[i]) and the
// maxima of its run's bound codes.
struct CountRun {
    uint32_t d, codes, length, offset;   // codes, length: at the run's head
    bool valid, head;
    int first;                           // lane of the head
};
__device__ inline CountRun count_run(const WorldDev &w, uint32_t i, uint32_t n)
{
    const uint32_t l = lane_id();
    CountRun r;
    r.valid = i < n;
    r.d = NONE;
    r.codes = 0u;
    if (r.valid) {
        const uint32_t s = w.pdense[i];
        const SceneDev &sc = w.scenes[s];
        // (Words of a scene that has left may be of an older table: looked up in bounds.)
        const uint32_t at = w.pslot[i];
        if (at < w.h_total) r.d = w.hvals[at];
        r.codes = w.prank[i];
        r.valid = sc.active != 0u;
        if (!r.valid) {
            r.d = NONE;
        } else if (r.d == NONE) {
            r.d = w.hvals[sc.h_base + sc.h_cap];   // the overflow block: P2G does not take it
            r.codes = 0u;
        }
        w.pdense[i] = r.d;   // NONE: of a scene that has left
    }
    const uint32_t pd = __shfl_up(r.d, 1, WAVE);
    const bool pv = __shfl_up((int)r.valid, 1, WAVE) != 0;
    r.head = !r.valid || l == 0 || !pv || pd != r.d;
    const uint64_t heads = __ballot(r.head);
    const uint32_t h = run_head(heads, l), end = run_end(heads, h);
    // The run's maxima of the two code halves, at its head.
    for (uint32_t o = 1; o < WAVE; o <<= 1) {
        const uint32_t u = __shfl_down(r.codes, o, WAVE);
        if (l + o < end) r.codes = max(r.codes & 0xFFFFu, u & 0xFFFFu) | (max(r.codes >> 16, u >> 16) << 16);
    }
    r.head = r.head && r.valid;
    r.length = end - l;
    r.offset = l - h;
    r.first = (int)h;
    return r;
}

// Particles in the order of the last substep's blocks: an atomic per run.
__device__ inline void count_part(const WorldDev &w, uint32_t group, uint32_t groups)
{
    const uint32_t n = w.g->p_in;
    const uint32_t nr = (n + WAVE - 1) / WAVE * WAVE;
    for (uint32_t i = group * blockDim.x + threadIdx.x; i < nr; i += groups * blockDim.x) {
        const CountRun r = count_run(w, i, n);
        uint32_t base = 0;
        if (r.head) {
            base = atomicAdd(&w.bnp[r.d], r.length);
            if (r.codes) {
                atomicMax((uint32_t *)&w.bvid[r.d].w, r.codes & 0xFFFFu);
                atomicMax(&w.bprim[r.d], r.codes >> 16);
            }
        }
        base = __shfl(base, r.first, WAVE);
        if (r.valid) w.prank[i] = base + r.offset;
    }
}

// Particles in the order the host or a caller has them: a block comes back in many runs, so a
// workgroup first adds up its runs by block in LDS (120,001 particles line by line, the kernel
// 23.5 -> 10.7 us; 31,337 of four materials 11 -> 7).
struct CountSet {
    static constexpr uint32_t SIZE = 2 * KEY_GROUP;
    uint32_t block[SIZE], count[SIZE], codes[SIZE], mass_codes[SIZE];
};
__device__ inline void count_part_unsorted(const WorldDev &w, CountSet &set, uint32_t group, uint32_t groups)
{
    const uint32_t n = w.g->p_in;
    for (uint32_t c = group * KEY_GROUP; c < n; c += groups * KEY_GROUP) {
        for (uint32_t k = threadIdx.x; k < CountSet::SIZE; k += KEY_GROUP) {
            set.block[k] = NONE;
            set.count[k] = set.codes[k] = set.mass_codes[k] = 0u;
        }
        __syncthreads();
        const uint32_t i = c + threadIdx.x;
        const CountRun r = count_run(w, i, n);
        uint32_t at = 0u, base = 0u;
        if (r.head) {
            at = r.d * 0x9E3779B9u >> 22;
            for (;; at = (at + 1u) % CountSet::SIZE) {   // ends: at most half the places are taken
                const uint32_t prev = atomicCAS(&set.block[at], NONE, r.d);
                if (prev == NONE || prev == r.d) break;
            }
            base = atomicAdd(&set.count[at], r.length);
            atomicMax(&set.codes[at], r.codes & 0xFFFFu);
            atomicMax(&set.mass_codes[at], r.codes >> 16);
        }
        __syncthreads();
        for (uint32_t k = threadIdx.x; k < CountSet::SIZE; k += KEY_GROUP) {
            const uint32_t d = set.block[k];
            if (d == NONE) continue;
            if (set.codes[k]) atomicMax((uint32_t *)&w.bvid[d].w, set.codes[k]);
            if (set.mass_codes[k]) atomicMax(&w.bprim[d], set.mass_codes[k]);
            set.count[k] = atomicAdd(&w.bnp[d], set.count[k]);
        }
        __syncthreads();
        if (r.head) base += set.count[at];
        base = __shfl(base, r.first, WAVE);
        if (r.valid) w.prank[i] = base + r.offset;
        __syncthreads();
    }
}

// Block tables and particle counts, both needing only the dense block ids: side by side, by
// the first count_groups workgroups and the others (in one thread after the other the two
// chains of dependent reads add up).  The keys carry their hash slots, so a particle's block
// id is one read.  In sequence and with a hash search per particle: 50,000 particles 7.4 us,
// now 5.0; 32 scenes 22 and 19; the CPIC sand 8.9 and 6.8.
template <bool UNSORTED>
__global__ void __launch_bounds__(UNSORTED ? KEY_GROUP : 256) k_block_count(WorldDev w, uint32_t count_groups)
{
    if (blockIdx.x >= count_groups) {
        block_info_part(w, blockIdx.x - count_groups, gridDim.x - count_groups);
    } else if constexpr (UNSORTED) {
        __shared__ CountSet set;
        count_part_unsorted(w, set, blockIdx.x, count_groups);
    } else {
        count_part(w, blockIdx.x, count_groups);
    }
}

// P2G work split: workgroup g of the P2G grid takes blocks [p2g_start[g], p2g_start[g+1]),
// so that every workgroup gets about the same cost, counted as its particles plus
// w.p2g_block_cost per block (the tile clear and flush).  cost(d) = first particle of
// block d + p2g_block_cost d is non-decreasing; p2g_start[g] = min{d : cost(d) G >= g T},
// T the total cost, G the number of workgroups.

__device__ inline void p2g_split(const WorldDev &w)
{
    const uint32_t nb = w.g->n_blocks, G = w.p2g_groups;
    if (nb == 0u || G == 0u) return;
    const uint64_t K = w.p2g_block_cost;
    const uint64_t T = (uint64_t)w.g->p_out + K * nb;
    const uint32_t gid = blockIdx.x * blockDim.x + threadIdx.x, gsz = gridDim.x * blockDim.x;
    // 16 threads share a block's groups where there are several groups per block (few
    // blocks, or crowded ones: one thread wrote up to hundreds of starts, 51 us for 1000
    // particles); a thread per block otherwise, since each repeats the two divisions.
    const uint32_t J = G >= 4u * nb ? 16u : 1u;
    for (uint64_t t = gid; t < (uint64_t)nb * J; t += gsz) {
        const uint32_t d = (uint32_t)(t / J);
        const uint64_t g_hi = ((uint64_t)w.bfirst[d] + K * d) * G / T;   // last g with start d
        uint64_t g = 0;                                                  // first g with start d
        if (d > 0) g = (((uint64_t)w.bfirst[d - 1] + K * (d - 1)) * G) / T + 1;
        for (g += t % J; g <= g_hi && g < G; g += J) w.p2g_start[g] = d;
    }
    const uint64_t last = ((uint64_t)w.bfirst[nb - 1] + K * (nb - 1)) * G / T;
    for (uint64_t g = last + 1 + gid; g <= G; g += gsz) w.p2g_start[g] = nb;
}

__global__ void k_scatter(WorldDev w)
{
    const uint32_t n = w.g->p_in;
    for (uint32_t i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += gridDim.x * blockDim.x) {
        const uint32_t d = w.pdense[i];
        if (d == NONE) continue;
        uint32_t pos = w.bfirst[d] + w.prank[i];
        w.perm[pos] = i;
        w.sblock[pos] = d;
    }
    p2g_split(w);
}

// Order of the particles inside their blocks: by (rank among the particles of their cell,
// cell), in windows of ORDER_WINDOW.  A wave of P2G then holds particles of different
// cells, whose stencils meet different nodes at the same instruction: its LDS adds take 9
// cycles each against 17 in arrival order (8.4 without any conflict; 64 lanes on the 6^3
// tile).  No result depends on the order.  The output arena keeps it and the sort keeps
// the arrival order of a block's particles, so it lasts: the pass runs when the host has
// changed the arena and then once in ORDER_EVERY substeps (particles move about a
// hundredth of a cell per substep).  One wave per block.
constexpr int ORDER_PER = 8, ORDER_WINDOW = ORDER_PER * WAVE;
__global__ void __launch_bounds__(WAVE) k_cell_order(WorldDev w)
{
    __shared__ uint32_t count[NODES_PER_BLOCK], before[ORDER_WINDOW];
    __shared__ uint64_t cells[ORDER_WINDOW];
    const uint32_t l = threadIdx.x, nb = w.g->n_blocks;
    for (uint32_t d = blockIdx.x; d < nb; d += gridDim.x) {
        const int4 v = w.bvid[d];
        const uint32_t np = w.bnp[d];
        if (np < 4u || v.x == OVERFLOW_VID) continue;
        const SceneDev sc = w.scenes[w.bscene[d]];
        for (uint32_t c0 = 0; c0 < np; c0 += ORDER_WINDOW) {
            const uint32_t first = w.bfirst[d] + c0, n = min(np - c0, (uint32_t)ORDER_WINDOW);
            count[l] = 0u;
            __syncthreads();
            uint32_t slot[ORDER_PER], cell[ORDER_PER], rank[ORDER_PER];
            #pragma unroll
            for (int k = 0; k < ORDER_PER; ++k) slot[k] = k * WAVE + l < n ? w.perm[first + k * WAVE + l] : NONE;
            #pragma unroll
            for (int k = 0; k < ORDER_PER; ++k) {
                if (slot[k] == NONE) continue;
                const float4 q = w.in.quad(0)[slot[k]];
                const float x = q.x, y = q.y, z = q.z;
                // base cell in the block, 0..3 on each axis (a position without one: any cell)
                const int cx = (int)round_div(x, sc.h, sc.inv_h) - 1 - 4 * v.x;
                const int cy = (int)round_div(y, sc.h, sc.inv_h) - 1 - 4 * v.y;
                const int cz = (int)round_div(z, sc.h, sc.inv_h) - 1 - 4 * v.z;
                cell[k] = (uint32_t)(cx & 3) + 4u * (uint32_t)(cy & 3) + 16u * (uint32_t)(cz & 3);
                rank[k] = atomicAdd(&count[cell[k]], 1u);
            }
            __syncthreads();
            // cells[r]: the cells with more than r particles; before[r]: particles of rank < r.
            const uint32_t mine = count[l];
            uint32_t sum = 0u;
            for (uint32_t r = 0; sum < n; ++r) {
                const uint64_t m = __ballot(mine > r);
                if (l == 0) {
                    cells[r] = m;
                    before[r] = sum;
                }
                sum += (uint32_t)__popcll(m);
            }
            __syncthreads();
            #pragma unroll
            for (int k = 0; k < ORDER_PER; ++k)
                if (slot[k] != NONE)
                    w.perm[first + before[rank[k]] + (uint32_t)__popcll(cells[rank[k]] & ((1ull << cell[k]) - 1ull))] = slot[k];
            __syncthreads();
        }
    }
}

// ------------------------------------------------------------------------------------
// P2G: one wave per block, or a team of four waves per crowded block.  Each particle adds
// its 27-node quadratic-B-spline stencil (momentum m v + C dpt and mass, weighted) into a
// 6^3 LDS tile covering the block and its +1 halo; the tile is then written to the block's
// staging slot.  Same per-pair arithmetic as gpu_p2g_generic (p2g.rs:240-311): dpt = node -
// x, contribution (C dpt + m v) w and m w.
//
// The tile accumulates in 64-bit fixed point with integer LDS atomics (ds_add_u64):
// float LDS atomics serialize on gfx950 (~200 cycles per wave-op against ~8 for the
// 64-bit integer add).  The block's contributions are bounded by 2^e (bound_codes, reduced
// by the count kernel); a tile node receives at most np of them (one per particle of the
// block), so the scale 2^(62 - e - ceil(log2 np)) keeps every node sum below 2^62 while
// resolving contributions down to 2^-62 np of the largest.  Integer sums do not depend on
// the order of the adds, so the tile is bit-reproducible whatever the particle order.

// 64-bit fixed-point accumulator words of the P2G tile.
struct Fixed {
    using word = unsigned long long;
    // round(a w) as a two's-complement 64-bit integer, |a w| < 2^62: contributions are formed
    // in double and rounded once.  t = a w + 1.5 2^84 holds the high part H = round(a w / 2^32)
    // 2^32 in its low mantissa word; with it taken off exactly, r = a w - H + 1.5 2^52, where
    // |a w - H| <= 2^31, holds the rest in its mantissa.  The pattern of r plus H is the
    // integer plus that of 1.5 2^52, which ONE takes off (its low word is zero, so that it
    // can stand in t): three double operations and one 32-bit sum.  Doubles run at
    // the rate of floats here.  The product is exact before each rounding, so an integer
    // depends on a and w alone.
    // One rounding to a unit of 2^(e - 51) takes a third of the double operations (P2G 3-6 %
    // less: 1M sand 78 us against 82.6), but small contributions, such as the mass at the rim
    // of a stencil, then have up to 11 bits less.
    static constexpr int BITS = 62;
    static constexpr double ONE = (double)0x43380000u * 0x1p32, T = 0x1.8p84 - ONE, R = 0x1.8p52;
    __device__ static word of(double a, double w)
    {
        const double t = __builtin_fma(a, w, T);
        const double r = __builtin_fma(a, w, (T + R) - t);   // (T + R and the difference: exact)
        const uint32_t h = (uint32_t)__double_as_longlong(t);
        union { double d; uint32_t w[2]; word all; } u{r};
        // (written out: as plain sums the compiler makes two 64-bit ones of it)
        asm("v_add_u32 %0, %1, %2" : "=v"(u.w[1]) : "v"(u.w[1]), "v"(h));
        return u.all;
    }
    // scale is a power of two: multiplying by its reciprocal is exact
    __device__ static float back(word x, double inv_scale) { return (float)((double)(long long)x * inv_scale); }
};

__device__ inline int log2_up(uint32_t np) { return np > 1u ? 32 - __clz((int)(np - 1u)) : 0; }   // ceil(log2 np)

// The scale of a block whose contributions are bounded by 2^e, from the bound's code
// (bound_code).
__device__ inline float fixed_scale(uint32_t code, uint32_t np)
{
    const int e = code < 2u ? 0 : (int)code - CODE_BIAS;   // 0, 1: no bound (of a marked block)
    int k = Fixed::BITS - e - log2_up(np);
    k = k > 126 ? 126 : (k < -126 ? -126 : k);
    return ldexpf(1.0f, k);
}

// Staging tile regions, in the order of the +1 offsets e = 4 ex + 2 ey + ez (the
// reference's blocks_associated_to_block order): sizes 64, 32, 32, 16, 32, 16, 16, 8.
__device__ __constant__ const int REGION_OFFSET[8] = {0, 64, 96, 128, 144, 176, 192, 208};

// Words of the non-finite mask (one bit per tile word); the word after them flags any.
// The tile holds 4 fixed-point fields per node (momentum, mass).  CPIC blocks with
// particles that carry affinity bits fill it twice: the compatible contributions, flushed
// to the staging tiles, then the incompatible ones, flushed to the second staging tiles.
constexpr int TILE_FIELDS = 4;
constexpr int BAD_ANY = (TILE_FIELDS * TILE_NODES + 31) / 32;

// Which contributions a scatter pass adds: all (no affinity in the block), the compatible
// ones, or the incompatible ones.
constexpr int PART_ALL = 0, PART_COMPATIBLE = 1, PART_INCOMPATIBLE = 2;

struct d3 { double x, y, z; };
__device__ inline d3 scaled(f3 a, double s) { return d3{a.x * s, a.y * s, a.z * s}; }   // exact for 29-bit s
__device__ inline d3 step(d3 a, d3 h, double s)
{
    return d3{__builtin_fma(h.x, s, a.x), __builtin_fma(h.y, s, a.y), __builtin_fma(h.z, s, a.z)};
}
__device__ inline float pick(const float (&w)[3], int s) { return s == 0 ? w[0] : (s == 1 ? w[1] : w[2]); }

// One particle's stencil: C dpt + m v at node (sx, sy, sz) is base + sx hx + sy hy + sz hz
// (three fused steps per node instead of a matrix product), all in double with the block's
// scales folded in; the weights; the tile index of its base node.
struct Stencil {
    d3 base, hx, hy, hz;
    double mass;
    float wx[3], wy[3], wz[3];
    int t0;
};

// CPIC (p2g.rs:268-302): a particle not compatible with the node adds to the node's
// incompatible fields (the second pass of the block).
template <int PART>
__device__ __forceinline__ bool adds_to(const uint32_t *naff, int t, uint32_t pa)
{
    if (PART == PART_ALL) return true;
    const bool incomp = (pa & 0xFFFFu) != 0u && !aff_compatible(pa, naff[t]);
    return incomp == (PART == PART_INCOMPATIBLE);
}

__device__ __forceinline__ void add_node(unsigned long long *tile, int t, d3 a, double mass, double wgt)
{
    atomicAdd(&tile[t], Fixed::of(a.x, wgt));
    atomicAdd(&tile[TILE_NODES + t], Fixed::of(a.y, wgt));
    atomicAdd(&tile[2 * TILE_NODES + t], Fixed::of(a.z, wgt));
    atomicAdd(&tile[3 * TILE_NODES + t], Fixed::of(mass, wgt));
}

// K lanes share one particle: K = 1 scatters all 27 stencil nodes; K = 3 the 9 nodes of z
// slab sel; K = 9 the 3 nodes of row (sz, sy) = (sel / 3, sel % 3); K = 27 node (sel / 9,
// sel / 3 % 3, sel % 3).  Every node's contribution is computed by the same operations
// whatever K is (each step an explicit fused multiply-add; one with an offset of 0 is exact,
// and left out where the offset is known), so which lanes take a particle changes no bit.
template <int PART, int K>
__device__ __forceinline__ void p2g_scatter(unsigned long long *tile, const Stencil &q, int sel, const uint32_t *naff,
                                            uint32_t pa)
{
    constexpr int NZ = K == 1 ? 3 : 1, NY = K <= 3 ? 3 : 1, NX = K <= 9 ? 3 : 1;
    // The z slabs in a loop of nine nodes each: the code of all 27 is several times what the
    // instruction cache fetches in the time of a small launch.
    #pragma unroll 1
    for (int kz = 0; kz < NZ; ++kz) {
        const int sz = K == 1 ? kz : (K == 3 ? sel : (K == 9 ? sel / 3 : sel / 9));
        const d3 az = step(q.base, q.hz, (double)sz);
        const double wzs = (double)pick(q.wz, sz);
        #pragma unroll
        for (int ky = 0; ky < NY; ++ky) {
            const int sy = NY == 3 ? ky : (K == 9 ? sel % 3 : (sel / 3) % 3);
            const d3 ay = NY == 3 && ky == 0 ? az : step(az, q.hy, (double)sy);   // (a step of 0 adds nothing)
            const double wyz = (double)pick(q.wy, sy) * wzs;
            #pragma unroll
            for (int kx = 0; kx < NX; ++kx) {
                const int sx = NX == 3 ? kx : sel % 3;
                const int t = q.t0 + sx + TILE * sy + TILE * TILE * sz;
                const d3 a = NX == 3 && kx == 0 ? ay : step(ay, q.hx, (double)sx);
                if (adds_to<PART>(naff, t, pa)) add_node(tile, t, a, q.mass, (double)pick(q.wx, sx) * wyz);
            }
        }
    }
}

// The same for a particle whose bound is not finite (it is not in the block's): its
// contributions beyond the others' range (limit, np of which fit a word) are marked, and
// the node reads NaN.  Rare, so one loop over nodes [q0, q1) of the stencil.
template <int PART>
__device__ __forceinline__ void p2g_scatter_checked(unsigned long long *tile, uint32_t *bad, const Stencil &q, int q0,
                                                    int q1, double limit, const uint32_t *naff, uint32_t pa)
{
    #pragma unroll 1
    for (int n = q0; n < q1; ++n) {
        const int sz = n / 9, sy = n / 3 % 3, sx = n % 3;
        const int t = q.t0 + sx + TILE * sy + TILE * TILE * sz;
        if (!adds_to<PART>(naff, t, pa)) continue;
        const d3 a = step(step(step(q.base, q.hz, (double)sz), q.hy, (double)sy), q.hx, (double)sx);
        const double wgt = (double)pick(q.wx, sx) * ((double)pick(q.wy, sy) * (double)pick(q.wz, sz));
        add_node(tile, t, a, q.mass, wgt);
        auto off = [&](double v) { return !(fabs(v * wgt) < limit); };   // NaN too
        if (off(a.x) || off(a.y) || off(a.z) || off(q.mass)) {
            atomicOr(&bad[BAD_ANY], 1u);
            for (int c = 0; c < TILE_FIELDS; ++c) {
                const int k = c * TILE_NODES + t;
                atomicOr(&bad[k >> 5], 1u << (k & 31));
            }
        }
    }
}

// Flush: after the block's scatter pass, node t of the 6^3 tile goes to the region of the
// block it belongs to (offset e = (tx >= 4, ty >= 4, tz >= 4)), stored contiguously in that
// block's node order in the staging array st, so the consumer reads each region as one run
// of float4.  fdst, the kernel's LDS copy of FLUSH_CODE, gives each tile node's region e
// (bits 8..10) and its offset in the block's 216-node staging slot (bits 0..7).  Ends with
// the tile free for the next pass.
struct alignas(8) FlushCodes {
    uint16_t c[TILE_NODES];
};
constexpr FlushCodes flush_codes()
{
    FlushCodes f{};
    const int off[8] = {0, 64, 96, 128, 144, 176, 192, 208};   // REGION_OFFSET
    for (int t = 0; t < TILE_NODES; ++t) {
        const int tx = t % TILE, ty = (t / TILE) % TILE, tz = t / (TILE * TILE);
        const int ex = tx >> 2, ey = ty >> 2, ez = tz >> 2;
        const int e = 4 * ex + 2 * ey + ez;
        const int nx = ex ? 2 : 4, ny = ey ? 2 : 4;
        const int idx = (tx - 4 * ex) + nx * ((ty - 4 * ey) + ny * (tz - 4 * ez));
        f.c[t] = (uint16_t)((e << 8) | (off[e] + idx));
    }
    return f;
}
__device__ __constant__ const FlushCodes FLUSH_CODE = flush_codes();

// Copies FLUSH_CODE into the kernel's LDS table (54 lanes, 8 bytes each).
__device__ inline void load_flush_table(uint16_t *fdst, uint32_t l)
{
    static_assert(TILE_NODES * sizeof(uint16_t) == 54 * sizeof(uint64_t), "216 codes in 54 words");
    if (l < 54u) reinterpret_cast<uint64_t *>(fdst)[l] = reinterpret_cast<const uint64_t *>(FLUSH_CODE.c)[l];
}

// A team: the lanes that share one tile.  One wave (its LDS operations execute in order, so
// it only keeps the compiler from moving them), or the P2G_WAVES waves of a workgroup.
template <bool TEAM> constexpr int team_lanes() { return TEAM ? P2G_WAVES * WAVE : WAVE; }
template <bool TEAM> __device__ __forceinline__ void team_sync()
{
    if (TEAM) {
        __syncthreads();
    } else {
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    }
}

// With zero (a block whose particles do not reach every region), the flush also zeroes the
// words it reads, which are all the words the pass added to: the tile is then clean for the
// next pass without a full clear.
template <bool TEAM>
__device__ __forceinline__ void p2g_flush(unsigned long long *tile, const uint32_t *bad, float4 *stage,
                                          uint32_t d, float smom, float sm, uint32_t l, uint32_t touched,
                                          const uint16_t *fdst, bool zero)
{
    team_sync<TEAM>();
    const double inv_smom = 1.0 / (double)smom, inv_sm = 1.0 / (double)sm;   // exact: powers of two
    const bool any_bad = bad[BAD_ANY] != 0u;
    float4 *st = stage + (size_t)d * TILE_NODES;
    for (int t = (int)l; t < TILE_NODES; t += team_lanes<TEAM>()) {
        const uint32_t code = fdst[t];
        if (!((touched >> (code >> 8)) & 1u)) continue;   // no particle's stencil reaches region e
        float v4[4];
        #pragma unroll
        for (int c = 0; c < 4; ++c) v4[c] = Fixed::back(tile[c * TILE_NODES + t], c < 3 ? inv_smom : inv_sm);
        if (zero) {
            #pragma unroll
            for (int c = 0; c < 4; ++c) tile[c * TILE_NODES + t] = 0ull;
        }
        if (any_bad) {
            #pragma unroll
            for (int c = 0; c < 4; ++c) {
                const int q = c * TILE_NODES + t;
                if (bad[q >> 5] & (1u << (q & 31))) v4[c] = __builtin_nanf("");
            }
        }
        st[code & 0xFFu] = make_float4(v4[0], v4[1], v4[2], v4[3]);
    }
    team_sync<TEAM>();
}

// Empties the tile (unless the last flush left it clean) and its non-finite marks for the
// next scatter pass.  Blocks that reach all 8 regions (dense ones) clear here: one tight
// loop costs them less than zeroing inside the flush.
template <bool TEAM>
__device__ __forceinline__ void p2g_clear(unsigned long long *tile, uint32_t *bad, uint32_t l, bool dirty)
{
    if (dirty)
        for (int k = l; k < TILE_FIELDS * TILE_NODES; k += team_lanes<TEAM>()) tile[k] = 0;
    if (l <= (uint32_t)BAD_ANY) bad[l] = 0u;
}

// Staging regions of a block's tile that a particle with base cell (bx, by, bz) in the
// block reaches: region e = 4 ex + 2 ey + ez (the part of the +e neighbour in the tile)
// needs base cell coordinates >= 2 on the axes where e is 1 (the reference's spill rule,
// grid/sort.rs:322-328).
__device__ inline uint32_t spill_mask(int bx, int by, int bz)
{
    const bool sx = bx >= 2, sy = by >= 2, sz = bz >= 2;
    uint32_t m = 1u;
    if (sz) m |= 1u << 1;
    if (sy) m |= 1u << 2;
    if (sy && sz) m |= 1u << 3;
    if (sx) m |= 1u << 4;
    if (sx && sz) m |= 1u << 5;
    if (sx && sy) m |= 1u << 6;
    if (sx && sy && sz) m |= 1u << 7;
    return m;
}

// The quadratic B-spline weights of one axis, f in [0.5, 1.5] cells from the base node.
__device__ __forceinline__ void stencil_weights(float f, float (&w)[3])
{
    const float a = 1.5f - f, b = f - 1.0f, c = f - 0.5f;
    w[0] = 0.5f * a * a;
    w[1] = __builtin_fmaf(-b, b, 0.75f);
    w[2] = 0.5f * c * c;
}

// What a wave knows of the block it scatters.
struct BlockScales {
    int4 v;
    float h, ih, smom, sm;
    uint32_t np;
};
__device__ __forceinline__ BlockScales block_scales(const WorldDev &w, uint32_t s, int4 v, uint32_t mass_code, uint32_t np)
{
    BlockScales b;
    b.v = v;
    b.h = ld_uniform(&w.scenes[s].h);
    b.ih = ld_uniform(&w.scenes[s].inv_h);
    b.smom = fixed_scale((uint32_t)v.w, np);
    b.sm = fixed_scale(mass_code, np);
    b.np = np;
    return b;
}

// Scatter of one particle, by this lane as lane sel of the K that share it; returns the
// staging regions it reaches (0: its base cell is not in the block).  K = 0: as many as
// lanes says, with one copy of all but the scatter itself for every share.  (With a whole
// copy for each, 25 vector registers spilled: P2G of 2M clumped fluid 407 -> 337 us without
// them, of 1M sand 81 -> 73.8, of 100,003 21 -> 18.7.)
template <int PART, int K>
__device__ __forceinline__ uint32_t p2g_one(unsigned long long *tile, uint32_t *bad, const P2GIn &p, const BlockScales &b,
                                            uint32_t sel, const uint32_t *naff, uint32_t pa, uint32_t lanes = K)
{
    const float h = b.h, ih = b.ih;
    // A sum that bounds |m v + C dpt|: finite and far below FLT_MAX, it says that the bound
    // code did count this particle, so that its contributions fit the block's scale.  Any
    // other particle (a NaN or an infinity among its inputs, or a bound that overflows) takes
    // the checked scatter.
    const float vsum = fabsf(p.v.x) + fabsf(p.v.y) + fabsf(p.v.z);
    const float csum = fabsf(p.C.c0.x) + fabsf(p.C.c0.y) + fabsf(p.C.c0.z) + fabsf(p.C.c1.x) + fabsf(p.C.c1.y) +
                       fabsf(p.C.c1.z) + fabsf(p.C.c2.x) + fabsf(p.C.c2.y) + fabsf(p.C.c2.z);
    float sum = __builtin_fmaf(4.5f * h, csum, fabsf(p.m) * vsum);
    sum = __builtin_fmaf(p.px, 0.0f, __builtin_fmaf(p.py, 0.0f, __builtin_fmaf(p.pz, 0.0f, sum)));
    // Base node of the stencil and its offset from the particle.
    const float cx = round_div(p.px, h, ih) - 1.0f, cy = round_div(p.py, h, ih) - 1.0f, cz = round_div(p.pz, h, ih) - 1.0f;
    const int bx = (int)cx - 4 * b.v.x, by = (int)cy - 4 * b.v.y, bz = (int)cz - 4 * b.v.z;
    // A particle's primary block holds its base cell: bx, by, bz are in [0, 3] for every
    // finite position; anything else contributes nothing.
    if (!((unsigned)bx < 4u && (unsigned)by < 4u && (unsigned)bz < 4u)) return 0u;
    // Every operation that could be contracted is an explicit fused one: this function is
    // inlined once per way of taking a particle, and the copies must agree in every bit.
    const f3 d0 = mk3(__builtin_fmaf(cx, h, -p.px), __builtin_fmaf(cy, h, -p.py), __builtin_fmaf(cz, h, -p.pz));
    Stencil q;
    q.t0 = bx + TILE * by + TILE * TILE * bz;
    stencil_weights(-d0.x * ih, q.wx);
    stencil_weights(-d0.y * ih, q.wy);
    stencil_weights(-d0.z * ih, q.wz);
    // The scales are powers of two and products of two floats are exact in double.
    const double ds = (double)b.smom, hs = (double)h * ds;
    q.base = scaled(p.v, (double)p.m * ds);
    q.base = step(q.base, scaled(p.C.c0, ds), (double)d0.x);
    q.base = step(q.base, scaled(p.C.c1, ds), (double)d0.y);
    q.base = step(q.base, scaled(p.C.c2, ds), (double)d0.z);
    q.hx = scaled(p.C.c0, hs);
    q.hy = scaled(p.C.c1, hs);
    q.hz = scaled(p.C.c2, hs);
    q.mass = (double)p.m * (double)b.sm;
    const int share = 27 / (int)lanes, q0 = (int)sel * share;
    if (!(sum < 0x1p120f) || !(fabsf(p.m) < 0x1p120f))
        p2g_scatter_checked<PART>(tile, bad, q, q0, q0 + share, ldexp(1.0, Fixed::BITS - log2_up(b.np)), naff, pa);
    else if constexpr (K != 0)
        p2g_scatter<PART, K>(tile, q, (int)sel, naff, pa);
    else if (lanes == 1u)
        p2g_scatter<PART, 1>(tile, q, 0, naff, pa);
    else if (lanes == 3u)
        p2g_scatter<PART, 3>(tile, q, (int)sel, naff, pa);
    else if (lanes == 9u)
        p2g_scatter<PART, 9>(tile, q, (int)sel, naff, pa);
    else
        p2g_scatter<PART, 27>(tile, q, (int)sel, naff, pa);
    return spill_mask(bx, by, bz);
}

// Node affinity words of block d's 6^3 tile (CPIC scenes; zero, compatible with every
// particle, elsewhere and for missing blocks).
template <bool TEAM>
__device__ inline void load_tile_affinity(const WorldDev &w, uint32_t d, uint32_t *naff, uint32_t l)
{
    for (int t = l; t < TILE_NODES; t += team_lanes<TEAM>()) {
        const int tx = t % TILE, ty = (t / TILE) % TILE, tz = t / (TILE * TILE);
        const int e = 4 * (tx >> 2) + 2 * (ty >> 2) + (tz >> 2);
        const uint32_t blk = w.bup[8 * (size_t)d + e];
        naff[t] = blk == NONE ? 0u : w.ncdf[(size_t)blk * NODES_PER_BLOCK + (tx & 3) + 4 * (ty & 3) + 16 * (tz & 3)].y;
    }
}

// The union over the wave of the lanes' region masks.
__device__ inline uint32_t wave_or_mask8(uint32_t m)
{
    uint32_t out = 0u;
    #pragma unroll
    for (int e = 0; e < 8; ++e) out |= __ballot((m >> e) & 1u) ? (1u << e) : 0u;
    return out;
}

// Regions of block d that no particle reached are neither flushed nor read: the block
// receiving region e (bup[d][e]) stops listing d as its source e (bdn), so the grid update
// skips it.  Only block d writes that entry, and the grid update reads it after P2G.
__device__ inline void unlink_untouched(const WorldDev &w, uint32_t d, uint32_t touched, uint32_t l)
{
    if (l < 8u && !((touched >> l) & 1u)) {
        const uint32_t dst = w.bup[8 * (size_t)d + l];
        if (dst != NONE) w.bdn[8 * (size_t)dst + l] = NONE;
    }
}

// A particle of the input arena for P2G; off: none, or a disabled one.
struct P2GLane {
    P2GIn p;
    bool on;
};
__device__ __forceinline__ P2GLane p2g_fetch(const WorldDev &w, uint32_t slot)
{
    P2GLane r{};
    if (slot != NONE) {
        r.p = p2g_load(w, slot);
        r.on = (r.p.flags & FLAG_ENABLED) != 0u;
    }
    return r;
}

// One turn of a wave on a block: its particles [64 c, 64 c + 64), one per lane; the block's
// last turn, of r < 64 particles, with K lanes per particle: K = 27, 9, 3 or 1 for r <= 2,
// 7, 21 or more, so that a small remainder costs a fraction of a full 27-node pass.
struct Turn {
    uint32_t d, np, first, c, s, mass_code;   // np = 0: none
    int4 v;
};
__device__ __forceinline__ uint32_t turn_lanes(const Turn &t)
{
    const uint32_t r = t.np - WAVE * t.c;
    return r <= 2u ? 27u : (r <= 7u ? 9u : (r <= 21u ? 3u : 1u));
}
// The particle of its turn that lane l shares with k - 1 others.
__device__ __forceinline__ uint32_t shared_by(uint32_t l, uint32_t k)
{
    return k == 1u ? l : (k == 3u ? l / 3u : (k == 9u ? l / 9u : l / 27u));
}
__device__ __forceinline__ uint32_t turn_slot(const WorldDev &w, const Turn &t, uint32_t l)
{
    if (t.np == 0u) return NONE;
    const uint32_t i = WAVE * t.c + shared_by(l, turn_lanes(t));
    return i < t.np ? w.perm[t.first + i] : NONE;
}

// Staging regions reached, over a wave or a team.
template <bool TEAM>
__device__ __forceinline__ uint32_t team_touched(uint32_t *words, uint32_t l, uint32_t spill)
{
    uint32_t m = wave_or_mask8(spill);
    if (!TEAM) return m;
    if (l % WAVE == 0) words[l / WAVE] = m;
    __syncthreads();
    #pragma unroll
    for (int k = 0; k < P2G_WAVES; ++k) m |= words[k];
    return m;
}

// Scatter of a team's turns: a particle per lane, the next one's loads under the scatter of
// this one.
template <int PART>
__device__ __forceinline__ uint32_t p2g_turns(const WorldDev &w, unsigned long long *tile, uint32_t *bad, const BlockScales &b,
                                              uint32_t first, uint32_t np, uint32_t l, const uint32_t *naff)
{
    constexpr uint32_t LANES = team_lanes<true>();
    uint32_t spill = 0u;
    auto slot_of = [&](uint32_t i) { return i < np ? w.perm[first + i] : NONE; };
    auto aff_of = [&](uint32_t i) { return PART != PART_ALL && i < np ? w.out.uplane(PAFF)[first + i] : 0u; };
    uint32_t next = slot_of(l + LANES);
    P2GLane q = p2g_fetch(w, slot_of(l));
    for (uint32_t i = l; i - l % WAVE < np; i += LANES) {
        const uint32_t pa = aff_of(i);
        const P2GLane now = q;
        q = p2g_fetch(w, next);
        next = slot_of(i + 2 * LANES);
        if (now.on && (PART != PART_INCOMPATIBLE || (pa & 0xFFFFu) != 0u))
            spill |= p2g_one<PART, 1>(tile, bad, now.p, b, 0u, naff, pa);
    }
    return spill;
}

// One crowded block by a team.
template <bool CPIC>
__device__ __forceinline__ void p2g_team_block(const WorldDev &w, uint32_t d, uint32_t np, const int4 v,
                                               unsigned long long *tile, uint32_t *bad, uint32_t *naff, const uint16_t *fdst,
                                               uint32_t *words, bool &dirty)
{
    const uint32_t l = threadIdx.x, first = ld_uniform(w.bfirst + d);
    const BlockScales b = block_scales(w, ld_uniform(w.bscene + d), v, ld_uniform(w.bprim + d), np);
    bool inc = false;
    if (CPIC && ld_uniform(w.breach + d)) {
        for (uint32_t i = l; i < np; i += team_lanes<true>())
            inc |= (w.out.uplane(PAFF)[first + i] & 0xFFFFu) != 0u;   // (a disabled one: a second tile of zeros)
        inc = __ballot(inc) != 0ull;
        if (l % WAVE == 0) words[l / WAVE] = inc ? 1u : 0u;
        __syncthreads();
        for (int k = 0; k < P2G_WAVES; ++k) inc |= words[k] != 0u;
    }
    p2g_clear<true>(tile, bad, l, dirty);
    if (CPIC && inc) load_tile_affinity<true>(w, d, naff, l);
    team_sync<true>();
    uint32_t spill;
    if (CPIC && inc) spill = p2g_turns<PART_COMPATIBLE>(w, tile, bad, b, first, np, l, naff);
    else spill = p2g_turns<PART_ALL>(w, tile, bad, b, first, np, l, naff);
    const uint32_t touched = team_touched<true>(words, l, spill);
    p2g_flush<true>(tile, bad, reinterpret_cast<float4 *>(w.stage), d, b.smom, b.sm, l, touched, fdst, touched != 0xFFu);
    dirty = touched == 0xFFu;
    if (CPIC && inc) {
        // Second pass: the incompatible contributions of the particles with affinity.
        p2g_clear<true>(tile, bad, l, dirty);
        team_sync<true>();
        p2g_turns<PART_INCOMPATIBLE>(w, tile, bad, b, first, np, l, naff);
        p2g_flush<true>(tile, bad, reinterpret_cast<float4 *>(w.stage_i), d, b.smom, b.sm, l, touched, fdst, touched != 0xFFu);
        dirty = touched == 0xFFu;
    }
    unlink_untouched(w, d, touched, l);
    if (CPIC && l == 0) w.binc[d] = inc ? 1u : 0u;
}

// A particle of a turn and its affinity.
struct ReachLane {
    P2GLane q;
    uint32_t pa, lanes, sel;
};
__device__ __forceinline__ ReachLane reach_lane(const WorldDev &w, const Turn &t, uint32_t l)
{
    ReachLane r;
    r.lanes = turn_lanes(t);
    const uint32_t share = shared_by(l, r.lanes), i = WAVE * t.c + share;
    r.sel = l - r.lanes * share;
    r.q = p2g_fetch(w, turn_slot(w, t, l));
    r.pa = i < t.np ? w.out.uplane(PAFF)[t.first + i] : 0u;
    return r;
}
template <int PART>
__device__ __forceinline__ uint32_t reach_scatter(const ReachLane &r, unsigned long long *tile, uint32_t *bad,
                                                  const BlockScales &b, const uint32_t *naff)
{
    if (!r.q.on || (PART == PART_INCOMPATIBLE && (r.pa & 0xFFFFu) == 0u)) return 0u;
    return p2g_one<PART, 0>(tile, bad, r.q.p, b, r.sel, naff, r.pa, r.lanes);
}

// One CPIC block in reach of a collider by one wave, turn by turn; the particles of a block of
// one turn are read once for both passes.  With one lane per particle in the last turn, the
// affinities looked up through the slots first and the particles read anew for the second
// pass, P2G of 60,000 particles in 17,612 blocks took 72.7 us (now 55.9), of 262,144 in
// 6580 blocks 47.8 (45.9), of 1,048,576 in 21,764 blocks 114.6 (108.1).  Blocks of more than
// 64 by a team: 60,000 in 2024 blocks 25.3 us instead of 31.6, but 1,048,576 152 instead
// of 108.
__device__ __forceinline__ void p2g_reach_block(const WorldDev &w, Turn t, uint32_t l, unsigned long long *tile, uint32_t *bad,
                                                uint32_t *naff, const uint16_t *fdst, bool &dirty)
{
    ReachLane r = reach_lane(w, t, l);
    const BlockScales b = block_scales(w, t.s, t.v, t.mass_code, t.np);
    bool inc = (r.pa & 0xFFFFu) != 0u;   // (of a disabled particle alone: a second tile of zeros)
    for (uint32_t i = WAVE + l; i < t.np; i += WAVE) inc |= (w.out.uplane(PAFF)[t.first + i] & 0xFFFFu) != 0u;
    inc = __ballot(inc) != 0ull;
    p2g_clear<false>(tile, bad, l, dirty);
    if (inc) load_tile_affinity<false>(w, t.d, naff, l);
    team_sync<false>();
    uint32_t spill = 0u;
    for (;;) {
        spill |= inc ? reach_scatter<PART_COMPATIBLE>(r, tile, bad, b, naff) : reach_scatter<PART_ALL>(r, tile, bad, b, naff);
        if (WAVE * ++t.c >= t.np) break;
        r = reach_lane(w, t, l);
    }
    const uint32_t touched = wave_or_mask8(spill);
    p2g_flush<false>(tile, bad, reinterpret_cast<float4 *>(w.stage), t.d, b.smom, b.sm, l, touched, fdst, touched != 0xFFu);
    dirty = touched == 0xFFu;
    if (inc) {
        // Second pass: the incompatible contributions of the particles with affinity.
        p2g_clear<false>(tile, bad, l, dirty);
        team_sync<false>();
        t.c = 0u;
        if (t.np > (uint32_t)WAVE) r = reach_lane(w, t, l);
        for (;;) {
            reach_scatter<PART_INCOMPATIBLE>(r, tile, bad, b, naff);
            if (WAVE * ++t.c >= t.np) break;
            r = reach_lane(w, t, l);
        }
        p2g_flush<false>(tile, bad, reinterpret_cast<float4 *>(w.stage_i), t.d, b.smom, b.sm, l, touched, fdst, touched != 0xFFu);
        dirty = touched == 0xFFu;
    }
    unlink_untouched(w, t.d, touched, l);
    if (l == 0) w.binc[t.d] = inc ? 1u : 0u;
}

// Workgroups of P2G_WAVES waves, each with a cost-balanced range of blocks (p2g_split), the
// ranges of an XCD contiguous.  The waves take the range's blocks of up to TEAM_MIN
// particles one by one from a counter, each with a tile of its own; the crowded blocks are
// then taken by all the waves together on one tile: a block's particles are one serial
// chain otherwise (a block of 512 took 8 turns of 64, and a body of 32,768 particles at 8
// per cell kept 64 waves of the chip busy).
// Whether there are crowded ones the waves learn while they take the others, or each would
// go through the range again while the workgroup holds its tiles (P2G of 1M sand with CPIC
// 119.5 -> 113.7 us, of 2M clumped fluid 396 -> 387).
// A wave works ahead: while it scatters one turn, the next turn's particles (of the same
// block or the next) are being loaded and the slots of the one after are read, so that the
// chain slot -> particle -> LDS adds of a block is not waited for.
constexpr uint32_t TEAM_MIN = 128;
template <bool CPIC>
__global__ void __launch_bounds__(P2G_WAVES * WAVE) __attribute__((amdgpu_waves_per_eu(4))) k_p2g(WorldDev w)
{
    __shared__ typename Fixed::word tiles[P2G_WAVES][TILE_FIELDS * TILE_NODES];
    __shared__ uint32_t bads[P2G_WAVES][BAD_ANY + 1];   // non-finite contributions; last word: any at all
    __shared__ uint32_t naffs[CPIC ? P2G_WAVES : 1][CPIC ? TILE_NODES : 1];
    __shared__ __align__(8) uint16_t fdst[TILE_NODES];
    __shared__ uint32_t words[P2G_WAVES], queue[2], crowded;
    const uint32_t G = gridDim.x, bx = blockIdx.x;
    const uint32_t g = (G % NUM_XCD == 0) ? (bx % NUM_XCD) * (G / NUM_XCD) + bx / NUM_XCD : bx;
    const uint32_t begin = ld_uniform(w.p2g_start + g), end = ld_uniform(w.p2g_start + g + 1);
    if (begin == end) return;
    load_flush_table(fdst, threadIdx.x);
    if (threadIdx.x < 2u) queue[threadIdx.x] = begin;
    if (threadIdx.x == 0u) crowded = 0u;
    __syncthreads();
    const uint32_t wave = __builtin_amdgcn_readfirstlane(threadIdx.x / WAVE), l = lane_id();
    unsigned long long *tile = tiles[wave];
    uint32_t *bad = bads[wave], *naff = naffs[CPIC ? wave : 0];
    bool dirty = true;
    // Next block of a queue whose particles are taken by one wave (CPIC: those in reach of
    // a collider come from the second queue).
    auto pop = [&](int which, Turn &t) {
        for (;;) {
            uint32_t at = 0u;
            if (l == 0) at = atomicAdd(&queue[which], 1u);
            t.d = __builtin_amdgcn_readfirstlane(at);
            t.np = 0u;
            if (t.d >= end) return;
            const uint32_t np = ld_uniform(w.bnp + t.d);
            if (np > TEAM_MIN) crowded = 1u;   // (by whichever lanes: the same value)
            if (np == 0u || np > TEAM_MIN) continue;
            t.v = ld_uniform(w.bvid + t.d);
            if (t.v.x == OVERFLOW_VID) continue;
            if (CPIC && (ld_uniform(w.breach + t.d) != 0u) != (which == 1)) continue;
            t.np = np;
            t.c = 0u;
            t.first = ld_uniform(w.bfirst + t.d);
            t.s = ld_uniform(w.bscene + t.d);
            t.mass_code = ld_uniform(w.bprim + t.d);
            return;
        }
    };
    auto advance = [&](const Turn &t) {
        Turn n = t;
        if (WAVE * (t.c + 1u) < t.np) ++n.c;
        else if (t.np) pop(0, n);
        return n;
    };
    Turn t0;
    pop(0, t0);
    Turn t1 = advance(t0);
    P2GLane q = p2g_fetch(w, turn_slot(w, t0, l));
    uint32_t slot1 = turn_slot(w, t1, l), spill = 0u;
    while (t0.np) {
        const Turn t2 = advance(t1);
        const uint32_t slot2 = turn_slot(w, t2, l);
        const P2GLane q1 = p2g_fetch(w, slot1);
        const BlockScales b = block_scales(w, t0.s, t0.v, t0.mass_code, t0.np);
        if (t0.c == 0u) {
            p2g_clear<false>(tile, bad, l, dirty);
            team_sync<false>();
            spill = 0u;
        }
        const uint32_t k = turn_lanes(t0);
        if (q.on && l < (k == 27u ? 54u : (k == 1u ? 64u : 63u))) {
            spill |= p2g_one<PART_ALL, 0>(tile, bad, q.p, b, l - k * shared_by(l, k), naff, 0u, k);
        }
        if (WAVE * (t0.c + 1u) >= t0.np) {
            const uint32_t touched = wave_or_mask8(spill);
            p2g_flush<false>(tile, bad, reinterpret_cast<float4 *>(w.stage), t0.d, b.smom, b.sm, l, touched, fdst, touched != 0xFFu);
            dirty = touched == 0xFFu;
            unlink_untouched(w, t0.d, touched, l);
            if (CPIC && l == 0) w.binc[t0.d] = 0u;
        }
        t0 = t1;
        t1 = t2;
        q = q1;
        slot1 = slot2;
    }
    if (CPIC) {
        Turn t;
        for (pop(1, t); t.np; pop(1, t)) p2g_reach_block(w, t, l, tile, bad, naff, fdst, dirty);
    }
    __syncthreads();   // every block has been met, and the first wave has left its tile
    if (crowded == 0u) return;
    dirty = true;
    for (uint32_t d = begin; d < end; ++d) {
        const uint32_t np = ld_uniform(w.bnp + d);
        if (np <= TEAM_MIN) continue;
        const int4 v = ld_uniform(w.bvid + d);
        if (v.x == OVERFLOW_VID) continue;
        p2g_team_block<CPIC>(w, d, np, v, tiles[0], bads[0], naffs[0], fdst, words, dirty);
    }
}

// Empties the hash regions (keys and primary marks) for the next substep's insertions.
__device__ inline void clear_hash(const WorldDev &w)
{
    const uint32_t gid = blockIdx.x * blockDim.x + threadIdx.x, gsz = gridDim.x * blockDim.x;
    const uint32_t quads = w.h_total / 4u;   // (both arrays start on 16 bytes)
    for (uint32_t i = gid; i < quads; i += gsz) {
        reinterpret_cast<uint4 *>(w.hkeys)[i] = make_uint4(EMPTY_KEY, EMPTY_KEY, EMPTY_KEY, EMPTY_KEY);
        reinterpret_cast<uint4 *>(w.hmark)[i] = make_uint4(0u, 0u, 0u, 0u);
    }
    if (gid < w.h_total % 4u) {
        w.hkeys[4u * quads + gid] = EMPTY_KEY;
        w.hmark[4u * quads + gid] = 0u;
    }
}

// A block's staging tile as a buffer, empty without the block: the hardware's range check
// gives zero for a node outside it.
__device__ __forceinline__ __amdgpu_buffer_rsrc_t staged_tile(const float *stage, uint32_t block)
{
    const bool none = block == NONE;
    const float *at = stage + (none ? 0 : (size_t)block * (4 * TILE_NODES));
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<float *>(at), 0, none ? 0 : TILE_NODES * 16, 0x00020000);
}
__device__ __forceinline__ float4 staged_node(__amdgpu_buffer_rsrc_t tile, uint32_t offset)
{
    using u4 = uint32_t __attribute__((ext_vector_type(4)));
    const u4 q = __builtin_amdgcn_raw_buffer_load_b128(tile, (int)offset, 0, 0);
    return make_float4(__uint_as_float(q.x), __uint_as_float(q.y), __uint_as_float(q.z), __uint_as_float(q.w));
}

// ------------------------------------------------------------------------------------
// Grid update: gpu_grid_update + gpu_grid_update_collide (grid_update.rs:21-88,
// grid_update_collide.rs:105-183) on the summed tiles.  CPIC scenes update both velocity
// fields and skip the collider pass (solver/grid_update.rs:26-50).  MESH: the world has
// mesh colliders in scenes without CPIC, whose projection the collider pass then runs
// (its registers kept out of the common variant).
template <bool CPIC, bool MESH>
__global__ void __launch_bounds__(256) k_grid_update(WorldDev w)
{
    clear_hash(w);   // not read after the block tables (k_block_count, k_mesh_cdf) are built
    // Whole blocks per workgroup: a wave's 64 consecutive nodes are then one block, and the
    // per-block reads (scene, block id, tile sources, collider mask) are wave-uniform.
    uint32_t bbegin, bend;
    xcd_range(w.g->n_blocks, bbegin, bend);
    const uint32_t nend = bend * NODES_PER_BLOCK;
    // This lane's node in the eight source tiles: byte offset, out of range where the node is
    // not in the source's region.  The eight reads then go out together, without a branch.
    // Behind branches each waited for the one before: 1000 particles 7.4 us, now 5.6; 32 scenes
    // 17.8 and 12.7; 1M sand 20 and 17; 2M clumped particles 214 and 172 (2.9 TB/s of staged
    // tiles and nodes).  Reading the next block's words ahead costs more registers than it
    // saves (188 us there, 32 scenes 17.8).
    uint32_t node[8];
    #pragma unroll
    for (int e = 0; e < 8; ++e) {
        const int i = threadIdx.x & 3, j = (threadIdx.x >> 2) & 3, k = (threadIdx.x >> 4) & 3;
        const int ex = ASSOC[e][0], ey = ASSOC[e][1], ez = ASSOC[e][2];
        const int nx = ex ? 2 : 4, ny = ey ? 2 : 4;
        const bool out = (ex && i > 1) || (ey && j > 1) || (ez && k > 1);
        node[e] = out ? ~15u : 16u * (uint32_t)(REGION_OFFSET[e] + i + nx * (j + ny * k));
    }
    for (uint32_t n = bbegin * NODES_PER_BLOCK + threadIdx.x; n < nend; n += blockDim.x) {
        const uint32_t d = __builtin_amdgcn_readfirstlane(n >> 6);
        const uint32_t s = ld_uniform(w.bscene + d);
        const int4 v = ld_uniform(w.bvid + d);
        uint32_t src[8];
        #pragma unroll
        for (int e = 0; e < 8; ++e) src[e] = ld_uniform(w.bdn + 8 * (size_t)d + e);
        if (v.x == OVERFLOW_VID) continue;
        const uint32_t li = n & 63u;
        const int i = li & 3, j = (li >> 2) & 3, k = li >> 4;
        const SceneDev sc = ld_uniform(w.scenes + s);
        const bool cp = CPIC && sc.cpic;
        float mx = 0.0f, my = 0.0f, mz = 0.0f, m = 0.0f;
        float ix = 0.0f, iy = 0.0f, iz = 0.0f, im = 0.0f;
        float4 q[8];
        uint32_t inc[8];
        #pragma unroll
        for (int e = 0; e < 8; ++e) q[e] = staged_node(staged_tile(w.stage, src[e]), node[e]);
        if (cp) {
            // Only blocks with particles in reach of a collider have a second tile.
            #pragma unroll
            for (int e = 0; e < 8; ++e) inc[e] = ld_uniform(w.binc + (src[e] == NONE ? 0u : src[e]));
        }
        #pragma unroll
        for (int e = 0; e < 8; ++e) {
            mx += q[e].x;
            my += q[e].y;
            mz += q[e].z;
            m += q[e].w;
        }
        if (cp) {
            #pragma unroll
            for (int e = 0; e < 8; ++e) {
                q[e] = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
                if (src[e] != NONE && inc[e]) q[e] = staged_node(staged_tile(w.stage_i, src[e]), node[e]);
            }
            #pragma unroll
            for (int e = 0; e < 8; ++e) {
                ix += q[e].x;
                iy += q[e].y;
                iz += q[e].z;
                im += q[e].w;
            }
        }
        if (w.dbg_mom) {
            w.dbg_mom[3 * (size_t)n] = mx;
            w.dbg_mom[3 * (size_t)n + 1] = my;
            w.dbg_mom[3 * (size_t)n + 2] = mz;
        }
        const float inv_mass = m > 0.0f ? 1.0f / m : 0.0f;
        const float mdt = m * sc.dt;
        f3 vel = mk3((mx + sc.gx * mdt) * inv_mass, (my + sc.gy * mdt) * inv_mass, (mz + sc.gz * mdt) * inv_mass);
        const float lim = sc.vlim;
        vel.x = fminf(fmaxf(vel.x, -lim), lim);
        vel.y = fminf(fmaxf(vel.y, -lim), lim);
        vel.z = fminf(fmaxf(vel.z, -lim), lim);
        if (cp) {
            const float inv_mi = im > 0.0f ? 1.0f / im : 0.0f;
            const float midt = im * sc.dt;
            f3 vi = mk3((ix + sc.gx * midt) * inv_mi, (iy + sc.gy * midt) * inv_mi, (iz + sc.gz * midt) * inv_mi);
            vi.x = fminf(fmaxf(vi.x, -lim), lim);
            vi.y = fminf(fmaxf(vi.y, -lim), lim);
            vi.z = fminf(fmaxf(vi.z, -lim), lim);
            w.gridv_i[n] = make_float4(vi.x, vi.y, vi.z, im);
        }
        const uint32_t mask = cp ? 0u : ld_uniform(w.bmask + d);
        if (mask) {
            const f3 pt = mk3((float)(v.x * 4 + i), (float)(v.y * 4 + j), (float)(v.z * 4 + k)) * sc.h;
            const MeshSetDev ms{w.mesh_v, w.mesh_t, w.mesh_vn, w.mesh_en, w.mesh_grid, w.mesh_cell, w.mesh_ctri, w.col_mesh};
            vel = collide_node<MESH>(w.cols + sc.col_start, sc.col_count, mask, sc.h, sc.dt, pt, vel, ms, sc.col_start);
        }
        w.gridv[n] = make_float4(vel.x, vel.y, vel.z, m);
    }
}

// ------------------------------------------------------------------------------------
// G2P + particle update, one thread per sorted particle (g2p.rs:150-270,
// particle_update.rs:60-201, non-CPIC so the contact-distance terms vanish).

// NBH_SHIFTS (grid/kernel.rs:42-70), the reference's G2P summation order.
__device__ __constant__ const int8_t NBH[27][3] = {
    {2, 2, 2}, {2, 0, 2}, {2, 1, 2}, {0, 2, 2}, {0, 0, 2}, {0, 1, 2}, {1, 2, 2}, {1, 0, 2}, {1, 1, 2},
    {2, 2, 0}, {2, 0, 0}, {2, 1, 0}, {0, 2, 0}, {0, 0, 0}, {0, 1, 0}, {1, 2, 0}, {1, 0, 0}, {1, 1, 0},
    {2, 2, 1}, {2, 0, 1}, {2, 1, 1}, {0, 2, 1}, {0, 0, 1}, {0, 1, 1}, {1, 2, 1}, {1, 0, 1}, {1, 1, 1}};

// Node velocities of the particle's 6^3 stencil tile, read from the grid (the 8 blocks
// vid + {0,1}^3; missing blocks read as zero).
struct GatherGrid {
    const uint32_t *bup;
    const float4 *gridv;
    const float4 *gridv_i;                     // CPIC: incompatible velocities
    const uint4 *ncdf;                         // CPIC: node contact distance fields
    uint32_t n0, n1, n2, n3, n4, n5, n6, n7;   // vid + {0,1}^3 in ASSOC order (4 ox + 2 oy + oz)
    __device__ void prepare(uint32_t d)
    {
        const uint32_t *p = bup + 8 * (size_t)d;
        n0 = p[0]; n1 = p[1]; n2 = p[2]; n3 = p[3]; n4 = p[4]; n5 = p[5]; n6 = p[6]; n7 = p[7];
    }
    // Grid node of tile position (tx, ty, tz), NONE in a missing block.
    __device__ uint32_t index(int tx, int ty, int tz) const
    {
        // block of the node by selects on the three offset bits (no indexed register array)
        const bool ox = tx >= 4, oy = ty >= 4, oz = tz >= 4;
        const uint32_t z0 = oz ? n1 : n0, z1 = oz ? n3 : n2, z2 = oz ? n5 : n4, z3 = oz ? n7 : n6;
        const uint32_t y0 = oy ? z1 : z0, y1 = oy ? z3 : z2;
        const uint32_t blk = ox ? y1 : y0;
        if (blk == NONE) return NONE;
        return blk * NODES_PER_BLOCK + (tx & 3) + 4 * (ty & 3) + 16 * (tz & 3);
    }
    // The quadratic transfer over the 27 nodes at base position (bx, by, bz): vel = sum w v and
    // g_j = sum w v s_j over the offsets s, as sums along x, then y, then z of nine rows.  A
    // row's three nodes lie in at most two blocks, picked per row, so a node costs one select
    // and one add beside its load.  Missing blocks (a scene over its capacity) read as zero, in
    // a loop of its own.  Against 27 nodes one by one, each with its block picked from eight
    // and ten multiply-adds of its own, with the SVD copy without V: 141 -> 115 registers (4
    // waves a SIMD instead of 3), the 1M sand column's G2P 102 -> 90 us (2.1 TB/s of state),
    // 4 x 510k clumped fluid 251 -> 231, 32 mixed scenes 136 -> 123, the CPIC sand's plain
    // particles 34 -> 28.
    __device__ __forceinline__ void transfer(int bx, int by, int bz, const float (&wx)[3], const float (&wy)[3],
                                             const float (&wz)[3], f3 &vel, f3 &gx, f3 &gy, f3 &gz) const
    {
        const bool whole = n0 != NONE && n1 != NONE && n2 != NONE && n3 != NONE && n4 != NONE && n5 != NONE &&
                           n6 != NONE && n7 != NONE;
        if (whole) sum<true>(bx, by, bz, wx, wy, wz, vel, gx, gy, gz);
        else sum<false>(bx, by, bz, wx, wy, wz, vel, gx, gy, gz);
    }
    template <bool WHOLE>
    __device__ __forceinline__ void sum(int bx, int by, int bz, const float (&wx)[3], const float (&wy)[3],
                                        const float (&wz)[3], f3 &vel, f3 &gx, f3 &gy, f3 &gz) const
    {
        const bool x1 = bx == 3, x2 = bx >= 2;                       // offset 1, 2 beyond the block
        const uint32_t lx0 = bx, lx1 = (bx + 1) & 3, lx2 = (bx + 2) & 3;
        constexpr int WHOLLY = WHOLE ? 3 : 1;                        // (the rare case: a loop)
        #pragma unroll WHOLLY
        for (int sz = 0; sz < 3; ++sz) {
            const bool oz = bz + sz >= 4;
            const uint32_t a0 = oz ? n1 : n0, a1 = oz ? n3 : n2, b0 = oz ? n5 : n4, b1 = oz ? n7 : n6;
            const uint32_t lz = 16u * ((bz + sz) & 3);
            f3 s0 = mk3(0, 0, 0), sx = mk3(0, 0, 0), sy1 = mk3(0, 0, 0);
            #pragma unroll WHOLLY
            for (int sy = 0; sy < 3; ++sy) {
                const bool oy = by + sy >= 4;
                const uint32_t A = oy ? a1 : a0, B = oy ? b1 : b0, at = lz + 4u * ((by + sy) & 3);
                const uint32_t ra = A * NODES_PER_BLOCK + at, rb = B * NODES_PER_BLOCK + at;
                f3 v0, v1, v2;
                if (WHOLE) {
                    v0 = node(ra + lx0);
                    v1 = node((x1 ? rb : ra) + lx1);
                    v2 = node((x2 ? rb : ra) + lx2);
                } else {
                    v0 = A == NONE ? mk3(0, 0, 0) : node(ra + lx0);
                    v1 = (x1 ? B : A) == NONE ? mk3(0, 0, 0) : node((x1 ? rb : ra) + lx1);
                    v2 = (x2 ? B : A) == NONE ? mk3(0, 0, 0) : node((x2 ? rb : ra) + lx2);
                }
                const f3 c1 = v1 * wx[1], c2 = v2 * wx[2];
                const f3 r0 = v0 * wx[0] + c1 + c2, rx = c1 + c2 * 2.0f;
                const float wys = pick(wy, sy);
                const f3 t0 = r0 * wys;
                s0 = s0 + t0;
                sx = sx + rx * wys;
                sy1 = sy1 + t0 * (float)sy;
            }
            const float wzs = pick(wz, sz);
            const f3 u0 = s0 * wzs;
            vel = vel + u0;
            gx = gx + sx * wzs;
            gy = gy + sy1 * wzs;
            gz = gz + u0 * (float)sz;
        }
    }
    __device__ __forceinline__ f3 node(uint32_t i) const
    {
        const float4 g = gridv[i];
        return mk3(g.x, g.y, g.z);
    }
};

// Returns the position, flags and bound codes of what it wrote (xo, flo, codes), for the
// caller's key insertion.
template <class Gather, bool CPIC>
__device__ __forceinline__ void g2p_particle(const WorldDev &w, uint32_t pos, uint32_t d, Gather &gather, f3 &xo,
                                             uint32_t &flo, uint32_t &codes)
{
    {
        const uint32_t slot = w.perm[pos];
        const uint32_t s = w.bscene[d];
        const SceneDev sc = w.scenes[s];
        const int4 bv = w.bvid[d];
        const float4 q0 = w.in.quad(0)[slot], q4 = w.in.quad(4)[slot], q5 = w.in.quad(5)[slot], q6 = w.in.quad(6)[slot],
                     q7 = w.in.quad(7)[slot];
        uint32_t fl = __float_as_uint(q0.w);
        const float px = q0.x, py = q0.y, pz = q0.z;
        float mass = q4.y;
        const float vol0 = q4.z, id = q4.w;
        m3 F;
        F.c0 = mk3(q5.x, q5.y, q5.z);
        F.c1 = mk3(q5.w, q6.x, q6.y);
        F.c2 = mk3(q6.z, q6.w, q7.x);
        // Per-particle plastic state: three words for the sand tags, one for snow.
        float ps0 = q7.y, ps1 = q7.z, ps2 = q7.w;
        f3 vel;
        m3 C;
        f3 npos = mk3(px, py, pz);
        const ClassDev &cls = w.classes[sc.class_base + flags_class(fl)];
        const uint32_t tag = cls.tag;
        // CPIC: this substep's particle contact field (written at the sorted position).  A
        // particle without affinity bits is compatible with every node and its contact
        // field is zero (a regular fit needs a node sharing an affinity), so it takes the
        // plain path.
        uint32_t pa = 0u;
        if (CPIC && sc.cpic) pa = w.out.uplane(PAFF)[pos];
        const bool cp = CPIC && (pa & 0xFFFFu) != 0u;
        f3 rigid_vel = mk3(0, 0, 0);
        if (bv.x == OVERFLOW_VID) {
            // No block: keep the particle unchanged (the scene reports an error).
            vel = mk3(w.in.plane(PVX)[slot], w.in.plane(PVY)[slot], w.in.plane(PVZ)[slot]);
            C.c0 = mk3(w.in.plane(PC0)[slot], w.in.plane(PC1)[slot], w.in.plane(PC2)[slot]);
            C.c1 = mk3(w.in.plane(PC3)[slot], w.in.plane(PC4)[slot], w.in.plane(PC5)[slot]);
            C.c2 = mk3(w.in.plane(PC6)[slot], w.in.plane(PC7)[slot], w.in.plane(PC8)[slot]);
        } else {
            const float h = sc.h, dt = sc.dt, inv_d = sc.inv_d;
            vel = mk3(0, 0, 0);
            m3 gradv = mzero();
            float div = 0.0f;
            const float ih = sc.inv_h;
            const float cx = round_div(px, h, ih) - 1.0f, cy = round_div(py, h, ih) - 1.0f,
                        cz = round_div(pz, h, ih) - 1.0f;
            const int bx = (int)cx - 4 * bv.x, by = (int)cy - 4 * bv.y, bz = (int)cz - 4 * bv.z;
            const bool inside = (unsigned)bx < 4u && (unsigned)by < 4u && (unsigned)bz < 4u;
            if ((fl & FLAG_ENABLED) && inside) {
                const f3 ref = mk3(cx * h - px, cy * h - py, cz * h - pz);
                float wx[3], wy[3], wz[3];
                {
                    const float fx = -ref.x * ih, fy = -ref.y * ih, fz = -ref.z * ih;
                    wx[0] = 0.5f * (1.5f - fx) * (1.5f - fx); wx[1] = 0.75f - (fx - 1.0f) * (fx - 1.0f); wx[2] = 0.5f * (fx - 0.5f) * (fx - 0.5f);
                    wy[0] = 0.5f * (1.5f - fy) * (1.5f - fy); wy[1] = 0.75f - (fy - 1.0f) * (fy - 1.0f); wy[2] = 0.5f * (fy - 0.5f) * (fy - 0.5f);
                    wz[0] = 0.5f * (1.5f - fz) * (1.5f - fz); wz[1] = 0.75f - (fz - 1.0f) * (fz - 1.0f); wz[2] = 0.5f * (fz - 0.5f) * (fz - 0.5f);
                }
                gather.prepare(d);
                // With dpt = ref + s h (s in {0,1,2}^3): sum w v dpt^T = V ref^T + h [Gx Gy Gz],
                // V = sum w v and Gj = sum w v s_j, so each node costs a product and a few
                // adds instead of an outer product; the velocity gradient and its trace
                // (the divergence) follow after the loop.
                f3 gx = mk3(0, 0, 0), gy = mk3(0, 0, 0), gz = mk3(0, 0, 0);
                if (cp) {
                    // g2p.rs:206-233: a node the particle is not compatible with gives its
                    // incompatible velocity, seen through its closest collider's boundary
                    // condition (friction scaled by the particle's factor) relative to the
                    // body's velocity there.  Fully unrolled: the contact particles are few,
                    // so their kernel runs about one wave per SIMD and needs every load in
                    // flight rather than occupancy.
                    const f3 pn = mk3(w.out.plane(PNX)[pos], w.out.plane(PNY)[pos], w.out.plane(PNZ)[pos]);
                    #pragma unroll
                    for (int q = 0; q < 27; ++q) {
                        const int sx = NBH[q][0], sy = NBH[q][1], sz = NBH[q][2];
                        const uint32_t ni = gather.index(bx + sx, by + sy, bz + sz);
                        f3 cv = mk3(0, 0, 0);
                        if (ni != NONE) {
                            const uint4 nc = gather.ncdf[ni];
                            const bool comp = aff_compatible(pa, nc.y);
                            const float4 g = comp ? gather.gridv[ni] : gather.gridv_i[ni];
                            cv = mk3(g.x, g.y, g.z);
                            if (!comp && nc.z != NONE) {
                                // the closest body's velocity at the node and its boundary
                                // condition {type in ncdf.w, friction}, stored by k_grid_cdf
                                const float4 nb = w.nbody[ni];
                                const f3 bpv = mk3(nb.x, nb.y, nb.z);
                                cv = bpv + bc_project(nc.w, nb.w * cls.bfric, cv - bpv, pn);
                            }
                        }
                        const float wsx = sx == 0 ? wx[0] : (sx == 1 ? wx[1] : wx[2]);
                        const float wsy = sy == 0 ? wy[0] : (sy == 1 ? wy[1] : wy[2]);
                        const float wsz = sz == 0 ? wz[0] : (sz == 1 ? wz[1] : wz[2]);
                        const f3 cw = cv * (wsx * wsy * wsz);
                        vel = vel + cw;
                        gx = gx + cw * (float)sx;
                        gy = gy + cw * (float)sy;
                        gz = gz + cw * (float)sz;
                    }
                } else {
                    gather.transfer(bx, by, bz, wx, wy, wz, vel, gx, gy, gz);
                }
                gradv.c0 = (vel * ref.x + gx * h) * inv_d;
                gradv.c1 = (vel * ref.y + gy * h) * inv_d;
                gradv.c2 = (vel * ref.z + gz * h) * inv_d;
                div = gradv.c0.x + gradv.c1.y + gradv.c2.z;
                if (cp) {
                    // g2p.rs:248-258: the bodies' velocities at the particle over its affinities
                    for (uint32_t m = pa & ((1u << sc.col_count) - 1u); m != 0u; m &= m - 1u)   // col_count <= 16
                        rigid_vel = rigid_vel + body_point_velocity(w.cols[sc.col_start + (uint32_t)__ffs(m) - 1u], mk3(px, py, pz));
                }
            }
            // Particle update.  CPIC: a particle deeper than 0.05 h behind a surface is
            // reprojected (slip relative to the bodies) and pushed out by a penalty
            // impulse after the position update (particle_update.rs:92-136).
            // (The contact field is re-read here so that it is not live across the node loop.)
            f3 pn = mk3(0, 0, 0);
            float psd = 0.0f;
            if (cp) {
                pn = mk3(w.out.plane(PNX)[pos], w.out.plane(PNY)[pos], w.out.plane(PNZ)[pos]);
                psd = w.out.plane(PSD)[pos];
            }
            const bool pen = cp && psd < -0.05f * h;
            if (pen) vel = rigid_vel + bc_project(1u, 0.0f, vel - rigid_vel, pn);
            const float vl = length(vel);
            if (vl > sc.vlim) vel = vel / vl * h / dt;
            vel = vel * rcp_hw(1.0f + cls.damping * dt);
            if (fl & FLAG_FIXED) vel = mk3(0, 0, 0);
            npos = mk3(px, py, pz) + vel * dt;
            if (pen) {
                const float corrected = fmaxf(psd, -0.3f * h);
                vel = vel + pn * (dt * -corrected * 1.0e3f);
            }
            m3 tau = mzero();
            if (tag != 4u) {
                F = F + mul(gradv * dt, F);
            } else {
                const float f0 = F.c0.x;
                float rate = div * dt / 3.0f;
                rate = fminf(fmaxf(rate, -0.1f), 0.1f);
                float nd = f0 + rate * f0;
                nd = nd < 0.5f ? 0.5f : (nd > 2.0f ? 2.0f : nd);
                F = m3{{nd, 0, 0}, {0, nd, 0}, {0, 0, nd}};
            }
            if (tag == 1u) {
                tau = nh_stress(cls.w[0], cls.w[1], F);
            } else if (tag == 4u) {
                tau = fluid_stress(cls.w, F, gradv);
            } else if (tag <= 5u) {
                // Corotated linear, Drucker-Prager over either backbone, and snow: one copy of
                // the SVD without V and one with it (snow, and a sand projection that is wide).
                m3 U;
                f3 sv;
                const float *lame = cls.w;
                float hard = 1.0f;
                bool wide = tag == 5u;
                if (!wide) {
                    svd3_us(F, U, sv);
                    if (tag != 0u) {
                        wide = dp_project(cls.w + 3, ps0, ps1, ps2, F, U, sv);
                        lame += 10;
                    }
                }
                if (wide) {
                    const f3 projected = sv;
                    m3 V;
                    svd3(F, U, sv, V);
                    if (tag == 5u) {
                        hard = snow_project(cls.w + 1, ps0, F, U, sv, V);
                        lame += 4;
                    } else {
                        sv = projected;
                        F = recompose(U, sv, V);
                    }
                }
                tau = tag == 3u ? nh_stress(lame[0], lame[1], F) : linear_stress_svd(lame[0] * hard, lame[1] * hard, U, sv);
            }
            C = gradv * mass - tau * (vol0 * inv_d * dt);
            const bool nan_pos = npos.x != npos.x || npos.y != npos.y || npos.z != npos.z;
            if (nan_pos || !(det(F) > 0.0f)) {
                fl &= ~FLAG_ENABLED;
                vel = mk3(0, 0, 0);
                F = mident();
                C = mzero();
                mass = 0.0f;
                npos = mk3(px, py, pz);
            }
        }
        w.out.quad(0)[pos] = make_float4(npos.x, npos.y, npos.z, __uint_as_float(fl));
        // The affinity word beside the velocity is this substep's own (k_particle_cdf).
        *reinterpret_cast<f3 *>(&w.out.quad(1)[pos]) = vel;
        w.out.quad(2)[pos] = make_float4(C.c0.x, C.c0.y, C.c0.z, C.c1.x);
        w.out.quad(3)[pos] = make_float4(C.c1.y, C.c1.z, C.c2.x, C.c2.y);
        w.out.quad(4)[pos] = make_float4(C.c2.z, mass, vol0, id);
        w.out.quad(5)[pos] = make_float4(F.c0.x, F.c0.y, F.c0.z, F.c1.x);
        w.out.quad(6)[pos] = make_float4(F.c1.y, F.c1.z, F.c2.x, F.c2.y);
        w.out.quad(7)[pos] = make_float4(F.c2.z, ps0, ps1, ps2);
        xo = npos;
        flo = fl;
        codes = fl & FLAG_ENABLED ? bound_codes(vel, C, mass, sc.h) : 0u;
    }
}

// Body integration at the end of a substep (the reference's "Integrate bodies" pass,
// src_mpm/pipeline.rs:510-520, gpu_rigid_impulses_update in rigid_impulses.rs:66-140):
// MPM integrates its own copy of every coupled body (gpu_rigid_impulses_update,
// rigid_impulses.rs:66-140).  The particles' impulses on the bodies are compiled out in
// the reference (src_mpm_shaders/lib.rs:38), so the velocity is not changed by them and
// never capped; the pose advances about the world centre of mass c = pose * local_com:
// t' = c + exp(w dt) (t - c) + v dt, q' = normalize(exp(w dt) q) (Velocity::integrate,
// src_rbd_shaders/dynamics/body.rs:253-268, with glam's from_scaled_axis, quaternion
// product and normalize); then gravity is added to v along the axes where the body's
// inverse mass is nonzero (a dynamic body coupled two ways; zero for the others).
__device__ inline void integrate_collider(ColliderDev &c, float dt, f3 g)
{
    const f3 t0 = mk3(c.t[0], c.t[1], c.t[2]);
    const f3 com = collider_com(c);
    const f3 sa = mk3(c.angvel[0] * dt, c.angvel[1] * dt, c.angvel[2] * dt);
    const float len = sqrtf(sa.x * sa.x + sa.y * sa.y + sa.z * sa.z);
    float dx = 0.0f, dy = 0.0f, dz = 0.0f, dw = 1.0f;
    if (len != 0.0f) {
        float sn, cs;
        sincosf(len * 0.5f, &sn, &cs);
        dx = sa.x / len * sn;
        dy = sa.y / len * sn;
        dz = sa.z / len * sn;
        dw = cs;
    }
    const f3 arm = quat_rotate(dx, dy, dz, dw, t0 - com);
    c.t[0] = (com.x + arm.x) + c.linvel[0] * dt;
    c.t[1] = (com.y + arm.y) + c.linvel[1] * dt;
    c.t[2] = (com.z + arm.z) + c.linvel[2] * dt;
    const float qx = c.q[0], qy = c.q[1], qz = c.q[2], qw = c.q[3];
    const float nx = dw * qx + dx * qw + dy * qz - dz * qy;
    const float ny = dw * qy - dx * qz + dy * qw + dz * qx;
    const float nz = dw * qz + dx * qy - dy * qx + dz * qw;
    const float nw = dw * qw - dx * qx - dy * qy - dz * qz;
    const float r = 1.0f / sqrtf(nx * nx + ny * ny + nz * nz + nw * nw);
    c.q[0] = nx * r;
    c.q[1] = ny * r;
    c.q[2] = nz * r;
    c.q[3] = nw * r;
    c.linvel[0] = c.linvel[0] + (c.inv_mass[0] != 0.0f ? g.x : 0.0f) * dt;
    c.linvel[1] = c.linvel[1] + (c.inv_mass[1] != 0.0f ? g.y : 0.0f) * dt;
    c.linvel[2] = c.linvel[2] + (c.inv_mass[2] != 0.0f ? g.z : 0.0f) * dt;
}

// Every collider of every active scene, 16 slots per scene, grid-stride.  Runs inside the
// substep's last kernel (nothing after it in the substep reads the colliders).
__device__ inline void integrate_colliders_part(const WorldDev &w)
{
    const uint32_t n = w.s_count * 16u;
    for (uint32_t t = blockIdx.x * blockDim.x + threadIdx.x; t < n; t += gridDim.x * blockDim.x) {
        const SceneDev sc = w.scenes[t >> 4];
        const uint32_t c = t & 15u;
        if (!sc.active || c >= sc.col_count) continue;
        integrate_collider(w.cols[sc.col_start + c], sc.dt, mk3(sc.gx, sc.gy, sc.gz));
    }
}

// Contact particles of CPIC scenes: those with affinity bits (the others are compatible
// with every node and have a zero contact field, so the plain path is exact for them).
__device__ inline bool contact_particle(const WorldDev &w, uint32_t pos, uint32_t d)
{
    // breach is zero for the blocks of scenes without CPIC.
    return w.breach[d] && (w.out.uplane(PAFF)[pos] & 0xFFFFu) != 0u;
}

// ------------------------------------------------------------------------------------
// CFL timestep bound (timestep_bound.rs:61-111, models/default.rs:268-330,
// models/utils.rs:157-172) over the input arena: per enabled particle the smaller of the
// model's sound-speed bound and the velocity bound, as 1e-12 s units (saturating),
// min-reduced per scene.  Particles of one scene are contiguous, so a wave first
// reduces over the lanes that share a scene and issues one atomic per scene present.
__device__ inline uint32_t secs_to_int(float dt)
{
    const float x = dt * 1.0e12f;
    if (!(x > 0.0f)) return 0u;
    if (x >= 4294967295.0f) return 0xFFFFFFFFu;
    return (uint32_t)x;
}

__device__ inline float particle_dt_bound(const ClassDev &cls, float h, float mass, float vol0, const f3 &v,
                                          const m3 &F, const m3 &A, float pdet)
{
    const uint32_t tag = cls.tag;
    float bulk, shear, cfl;
    if (tag <= 1u) { bulk = cls.w[0] + 2.0f * cls.w[1] / 3.0f; shear = cls.w[1]; cfl = cls.w[2]; }
    else if (tag <= 3u) { bulk = cls.w[10] + 2.0f * cls.w[11] / 3.0f; shear = cls.w[11]; cfl = cls.w[12]; }
    else if (tag == 4u) { bulk = cls.w[0] * cls.w[1]; shear = 0.0f; cfl = cls.w[3]; }
    else if (tag == 5u) {
        // Snow: the linear elastic backbone with its moduli scaled by the hardening factor.
        const float hard = expf(cls.w[3] * (1.0f - pdet));
        bulk = (cls.w[4] + 2.0f * cls.w[5] / 3.0f) * hard; shear = cls.w[5] * hard; cfl = cls.w[6];
    }
    else { bulk = shear = cfl = 0.0f; }
    float dt = 0.0f;
    if (tag <= 5u) {
        const float density0 = mass / vol0;
        const float density = density0 / fmaxf(det(F), 1.0e-6f);
        const float c = sqrtf((bulk + shear * 4.0f / 3.0f) / density);
        dt = cfl * h / fmaxf(length(v), c);
    }
    const float na2 = dot(A.c0, A.c0) + dot(A.c1, A.c1) + dot(A.c2, A.c2);
    const float norm_b = (h * h) / 4.0f * sqrtf(na2) / mass;
    const float apic_v = norm_b * 6.0f * sqrtf(3.0f) / h;
    return fminf(dt, h / (length(v) + apic_v));
}

// The bound of arena slot i (flags fl, scene sc) in 1e-12 s units.
__device__ inline uint32_t arena_dt_bound(const Arena &a, uint32_t i, uint32_t fl, const SceneDev &sc,
                                          const ClassDev *classes)
{
    m3 F, A;
    F.c0 = mk3(a.plane(PF0)[i], a.plane(PF1)[i], a.plane(PF2)[i]);
    F.c1 = mk3(a.plane(PF3)[i], a.plane(PF4)[i], a.plane(PF5)[i]);
    F.c2 = mk3(a.plane(PF6)[i], a.plane(PF7)[i], a.plane(PF8)[i]);
    A.c0 = mk3(a.plane(PC0)[i], a.plane(PC1)[i], a.plane(PC2)[i]);
    A.c1 = mk3(a.plane(PC3)[i], a.plane(PC4)[i], a.plane(PC5)[i]);
    A.c2 = mk3(a.plane(PC6)[i], a.plane(PC7)[i], a.plane(PC8)[i]);
    const f3 v = mk3(a.plane(PVX)[i], a.plane(PVY)[i], a.plane(PVZ)[i]);
    const ClassDev &cls = classes[sc.class_base + flags_class(fl)];
    const float pdet = cls.tag == 5u ? a.plane(PS0)[i] : 1.0f;
    return secs_to_int(particle_dt_bound(cls, sc.h, a.plane(PMASS)[i], a.plane(PVOL0)[i], v, F, A, pdet));
}

// Wave reduction per scene of the lanes' running minima (cur_s = NONE: none): one
// atomicMin into out[s * stride] per distinct scene held by the wave's lanes.  Called by
// every lane of the wave.
__device__ inline void wave_scene_min(uint32_t cur_s, uint32_t cur_min, uint32_t *out, uint32_t stride)
{
    const uint32_t l = lane_id();
    uint64_t pending = __ballot(cur_s != NONE);
    while (pending) {
        const uint32_t leader = (uint32_t)__ffsll((unsigned long long)pending) - 1u;
        const uint32_t s = __shfl(cur_s, (int)leader, WAVE);
        uint32_t v = (cur_s == s) ? cur_min : 0xFFFFFFFFu;
        for (int o = 32; o > 0; o >>= 1) v = min(v, (uint32_t)__shfl_xor(v, o, WAVE));
        if (l == leader) atomicMin(&out[(size_t)s * stride], v);
        pending &= ~__ballot(cur_s == s);
    }
}

// Adaptive scenes: the CFL bound of the state a G2P kernel has just written at sorted
// position pos (valid lanes; every lane of the wave calls), min-reduced per scene into the
// scene's clock for the next substep.
__device__ inline void next_dt_bound(const WorldDev &w, uint32_t pos, bool valid, uint32_t s)
{
    uint32_t cand = NONE, cs = NONE;
    if (valid) {
        const SceneDev sc = w.scenes[s];
        const uint32_t fl = w.out.uplane(PFLAGS)[pos];
        if (sc.adaptive && (fl & FLAG_ENABLED)) {
            cand = arena_dt_bound(w.out, pos, fl, sc, w.classes);
            cs = s;
        }
    }
    wave_scene_min(cs, cand, &w.clock[0].bound, (uint32_t)(sizeof(SceneClock) / 4));
}

// Start of a substep (first workgroup of its first scan): each adaptive scene's substep
// length becomes min(dt_max, the bound of its state), written into the scene table for
// the substep's later kernels; every scene's clock advances by its substep length.
__device__ inline void advance_clocks(const WorldDev &w)
{
    if (!w.clock) return;
    for (uint32_t s = threadIdx.x; s < w.s_count; s += blockDim.x) {
        SceneDev &sc = const_cast<SceneDev &>(w.scenes[s]);
        if (!sc.active) continue;
        SceneClock &c = w.clock[s];
        float dt = sc.dt;
        if (sc.adaptive) {
            dt = sc.dt_max;
            // The bound in seconds as the reference's host converts it (timestep_bound.rs:45).
            const float b = (float)c.bound / 1.0e12f;
            if (c.bound != NONE && b < dt) dt = b;
            if (!(dt > 0.0f)) dt = sc.dt_max;   // a zero bound (no finite one) keeps the maximum
            sc.dt = dt;
            sc.vlim = sc.h / dt;
        }
        c.bound = NONE;
        c.dt = dt;
        c.steps += 1u;
        c.t += (double)dt;
    }
}

// After this substep's scans: their look-back state and tickets start empty for the next
// substep, whose keys the G2P kernels insert into the hash (emptied by the grid update).
__device__ inline void prepare_next_sort(const WorldDev &w)
{
    const uint32_t gid = blockIdx.x * blockDim.x + threadIdx.x, gsz = gridDim.x * blockDim.x;
    for (uint32_t i = gid; i < 2u * w.scan_stride; i += gsz) w.scan_state[i] = 0ull;
    if (gid == 0) { w.g->ticket[0] = 0u; w.g->ticket[1] = 0u; }
    mark_overflow_slots(w);
}

// One thread per sorted particle, nodes read from the grid: the launch (g2p_groups) gives
// every workgroup at most g2p_threads positions, and a thread takes at most one, so no loop keeps
// the addresses of both arenas' quads and of the tables live in scalar registers.  In CPIC worlds this kernel takes the
// plain particles and k_g2p_contact the contact ones, so that the contact code does not
// weigh on the register budget of the common path.  Then the new positions give
// the next substep's block keys and insertions (touch_keys): the output arena is the next
// input arena, in the same order, so the next substep starts at its scan.  The keys are
// taken by whole waves (lanes past the range are invalid) from the position and flags the
// thread has just written, still in its registers.
template <bool CPIC, bool ADAPT>
__global__ void __launch_bounds__(g2p_threads<CPIC>()) k_g2p_update(WorldDev w)
{
    uint32_t pbegin, pend;
    xcd_range(w.g->p_out, pbegin, pend);
    GatherGrid grid{w.bup, w.gridv, w.gridv_i, w.ncdf, NONE, NONE, NONE, NONE, NONE, NONE, NONE, NONE};
    const uint32_t pos = pbegin + threadIdx.x;
    bool valid = pos < pend;
    f3 xo = mk3(0, 0, 0);
    uint32_t flo = 0u, codes = 0u;
    if (valid) {
        const uint32_t d = w.sblock[pos];
        if (CPIC && contact_particle(w, pos, d)) valid = false;   // keyed by k_g2p_contact
        else g2p_particle<GatherGrid, false>(w, pos, d, grid, xo, flo, codes);
    }
    if (pbegin + (threadIdx.x & ~(uint32_t)(WAVE - 1)) < pend) {   // the wave holds positions
        const uint32_t s = valid ? flags_scene(flo) : 0u;
        touch_keys(w, pos, valid, s, xo.x, xo.y, xo.z, codes);
        if (ADAPT) next_dt_bound(w, pos, valid, s);
    }
    prepare_next_sort(w);
    integrate_colliders_part(w);   // their last reader (k_g2p_contact, in CPIC worlds) has run
}

// The contact particles listed by k_particle_cdf, then their keys (as in k_g2p_update).
template <bool ADAPT>
__global__ void __launch_bounds__(256) k_g2p_contact(WorldDev w)
{
    const uint32_t n = w.g->n_contact;
    GatherGrid grid{w.bup, w.gridv, w.gridv_i, w.ncdf, NONE, NONE, NONE, NONE, NONE, NONE, NONE, NONE};
    for (uint32_t i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += gridDim.x * blockDim.x) {
        const uint32_t pos = w.clist[i];
        f3 xo;
        uint32_t flo, codes;
        g2p_particle<GatherGrid, true>(w, pos, w.sblock[pos], grid, xo, flo, codes);
        w.prank[pos] = codes;   // touch_keys below writes it again
    }
    const uint32_t l = lane_id();
    for (uint32_t base = blockIdx.x * blockDim.x + (threadIdx.x & ~(uint32_t)(WAVE - 1)); base < n;
         base += gridDim.x * blockDim.x) {
        const uint32_t i = base + l;
        const bool valid = i < n;
        uint32_t pos = 0, s = 0, codes = 0u;
        float x = 0.0f, y = 0.0f, z = 0.0f;
        if (valid) {
            pos = w.clist[i];
            codes = w.prank[pos];
            s = w.bscene[w.sblock[pos]];
            x = w.out.plane(PX)[pos];
            y = w.out.plane(PY)[pos];
            z = w.out.plane(PZ)[pos];
        }
        touch_keys(w, pos, valid, s, x, y, z, codes);
        if (ADAPT) next_dt_bound(w, pos, valid, s);
    }
}

// ------------------------------------------------------------------------------------
// CPIC contact distance field.

// Per rigid particle of a CPIC scene's mesh colliders: gpu_p2g_cdf (p2g_cdf.rs:60-259)
// as a scatter.  The sample and its triangle take the body's pose of the substep's start
// (gpu_transform_sample_points / gpu_transform_shape_points, rigid_particle_update.rs:
// 10-55).  The nodes of the 3-cell range from the sample's associated cell
// round(x / h) - 1 that lie in active blocks get, where their projection onto the
// triangle's plane falls inside the triangle (edge tests with n = ab x ac), the
// collider's affinity bit with the side n . (x - a) < 0, and the candidate distance
// |n . (x - a)| / |n|.  Per node a 64-bit minimum of (distance bits << 32) | collider
// keeps the least distance, the lower collider on a tie (the distances are not
// negative, so their bits order like their values).  The reference reaches the same
// nodes through its rigid-particle sort (a primary block, extras in the +1 neighbours,
// grid/sort.rs:165-250, 493-680) and a per-block loop; here each block of the range is
// looked up in the scene's hash.
__global__ void __launch_bounds__(256) k_mesh_cdf(WorldDev w)
{
    for (uint32_t r = blockIdx.x * blockDim.x + threadIdx.x; r < w.n_rp; r += gridDim.x * blockDim.x) {
        const float4 rp = w.mesh_rp[r];
        const uint4 tri = w.mesh_t[__float_as_uint(rp.w)];
        const SceneDev sc = w.scenes[tri.w >> 4];
        if (!sc.active || !sc.cpic) continue;
        const uint32_t cid = tri.w & 15u;
        const ColliderDev &c = w.cols[sc.col_start + cid];
        const f3 t = mk3(c.t[0], c.t[1], c.t[2]);
        const float qx = c.q[0], qy = c.q[1], qz = c.q[2], qw = c.q[3];
        const float4 va = w.mesh_v[tri.x], vb = w.mesh_v[tri.y], vc = w.mesh_v[tri.z];
        const f3 p = quat_rotate(qx, qy, qz, qw, mk3(rp.x, rp.y, rp.z)) + t;
        const f3 a = quat_rotate(qx, qy, qz, qw, mk3(va.x, va.y, va.z)) + t;
        const f3 b = quat_rotate(qx, qy, qz, qw, mk3(vb.x, vb.y, vb.z)) + t;
        const f3 cc = quat_rotate(qx, qy, qz, qw, mk3(vc.x, vc.y, vc.z)) + t;
        const f3 ab = b - a, ac = cc - a, bc = cc - b;
        const f3 n = cross(ab, ac);
        const float nl = length(n);
        if (nl == 0.0f) continue;
        const f3 eab = cross(ab, n), ebc = cross(bc, n), eac = cross(ac, n);
        const float h = sc.h, ih = sc.inv_h;
        const float fx = round_div(p.x, h, ih) - 1.0f, fy = round_div(p.y, h, ih) - 1.0f,
                    fz = round_div(p.z, h, ih) - 1.0f;
        if (!(fabsf(fx) < 4000.0f && fabsf(fy) < 2000.0f && fabsf(fz) < 4000.0f)) continue;   // NaN too
        const int cx = (int)fx, cy = (int)fy, cz = (int)fz;
        for (int bz = cz >> 2; bz <= (cz + 2) >> 2; ++bz)
            for (int by = cy >> 2; by <= (cy + 2) >> 2; ++by)
                for (int bx = cx >> 2; bx <= (cx + 2) >> 2; ++bx) {
                    // Keys of blocks outside the packable range would alias others.
                    if (bx < -1023 || bx > 1023 || by < -511 || by > 511 || bz < -1023 || bz > 1023) continue;
                    const uint32_t d = find_block(w, sc, bx, by, bz);
                    if (d == NONE) continue;
                    const int x0 = max(cx, 4 * bx), x1 = min(cx + 2, 4 * bx + 3);
                    const int y0 = max(cy, 4 * by), y1 = min(cy + 2, 4 * by + 3);
                    const int z0 = max(cz, 4 * bz), z1 = min(cz + 2, 4 * bz + 3);
                    for (int z = z0; z <= z1; ++z)
                        for (int y = y0; y <= y1; ++y)
                            for (int x = x0; x <= x1; ++x) {
                                const f3 pt = mk3((float)x, (float)y, (float)z) * h;
                                const f3 ap = pt - a, bp = pt - b, cp = pt - cc;
                                if (!(dot(eab, ap) <= 0.0f && dot(ebc, bp) <= 0.0f && dot(eac, cp) >= 0.0f)) continue;
                                const float sd = dot(n, ap) / nl;
                                const size_t node = (size_t)d * NODES_PER_BLOCK + (size_t)((x - 4 * bx) + 4 * (y - 4 * by) + 16 * (z - 4 * bz));
                                atomicOr(&w.maff[node], (sd < 0.0f ? 0x00010001u : 0x00000001u) << cid);
                                atomicMin(&w.mkey[node], ((unsigned long long)__float_as_uint(fabsf(sd)) << 32) | cid);
                            }
                }
    }
}

// Per node of a CPIC scene's blocks: gpu_grid_update_cdf (grid_update_cdf.rs:60-132) for
// the cuboids, then the meshes' part left by k_mesh_cdf: its affinity bits are added and
// its closest collider replaces the cuboids' when strictly nearer (p2g_cdf.rs:241).  The
// mesh part is reset to empty for the next substep.
__global__ void __launch_bounds__(256) k_grid_cdf(WorldDev w)
{
    // One wave per block: lane = node; bany[d] records whether any node of block d is in
    // reach of a collider (the particle pass skips stencils without such nodes).
    const uint32_t waves = gridDim.x * (blockDim.x / WAVE);
    const uint32_t l = threadIdx.x % WAVE;
    if (blockIdx.x == 0 && threadIdx.x == 0) w.g->n_contact = 0u;   // contact list of this substep
    for (uint32_t d = blockIdx.x * (blockDim.x / WAVE) + threadIdx.x / WAVE; d < w.g->n_blocks; d += waves) {
        const SceneDev sc = w.scenes[w.bscene[d]];
        if (!sc.cpic) continue;
        const int4 v = w.bvid[d];
        float dist = MAX_FLT_REF;
        uint32_t aff = 0u, closest = NONE, bc = 0u;
        const uint32_t mask = v.x != OVERFLOW_VID ? w.bmask[d] : 0u;
        const size_t n = (size_t)d * NODES_PER_BLOCK + l;
        const int i = l & 3, j = (l >> 2) & 3, k = l >> 4;
        const int4 vb = v.x != OVERFLOW_VID ? v : make_int4(0, 0, 0, 0);   // no mesh reaches the overflow block
        const f3 pt = mk3((float)(vb.x * 4 + i), (float)(vb.y * 4 + j), (float)(vb.z * 4 + k)) * sc.h;
        if (mask) node_cdf(w.cols + sc.col_start, sc.col_count, mask, sc.h, pt, dist, aff, closest);
        if (w.n_rp) {
            const unsigned long long key = w.mkey[n];
            if (key != ~0ull) {
                w.mkey[n] = ~0ull;
                const float md = __uint_as_float((uint32_t)(key >> 32));
                if (md < dist) { dist = md; closest = (uint32_t)key & 15u; }
            }
            const uint32_t ma = w.maff[n];
            if (ma) { w.maff[n] = 0u; aff |= ma; }
        }
        if (closest != NONE) {
            // For G2P's incompatible nodes: the closest body's velocity at the node
            // (g2p.rs:214-231 evaluates it at the node position as dpt + x) and its
            // boundary condition.
            const ColliderDev &c = w.cols[sc.col_start + closest];
            const f3 bpv = body_point_velocity(c, pt);
            w.nbody[n] = make_float4(bpv.x, bpv.y, bpv.z, c.bc_friction);
            bc = c.bc_type;
        }
        w.ncdf[n] = make_uint4(__float_as_uint(dist), aff, closest, bc);
        const uint64_t any = __ballot(aff != 0u);
        if (l == 0) w.bany[d] = any != 0ull ? 1u : 0u;
        // The primary blocks whose particles' stencils include nodes of this block (block d
        // is their +e neighbour, e in {0,1}^3) have particles in reach of a collider.
        if (any && l < 8u) {
            const uint32_t src = w.bdn[8 * (size_t)d + l];
            if (src != NONE) w.breach[src] = 1u;
        }
    }
}

// Per particle of a CPIC scene: gpu_g2p_cdf (g2p_cdf.rs:150-331).  The affinity word is
// the union of the stencil nodes' affinities; a collider reached for the first time gets
// its side from the sign of the weighted signed node distances, a known one keeps its
// side.  Then the moving-least-squares fit d(x) = n . (x - x_p) + d_p over the nodes that
// share an affinity with the particle (distance negated where the node's side differs)
// gives the normal and the signed distance; when its matrix is singular (det <= 1e-8) the
// field is zero, affinity included.  Results go to the output arena at the sorted
// position, where P2G and G2P read them and where they stay as the next state.
__device__ __forceinline__ uint32_t particle_cdf_one(const WorldDev &w, uint32_t pos, uint32_t d, const SceneDev &sc)
{
    const uint32_t slot = w.perm[pos];
    const uint32_t prev = w.in.uplane(PAFF)[slot];
    uint32_t aff = prev;
    f3 nrm = mk3(0, 0, 0);
    float sd = 0.0f;
    const int4 bv = w.bvid[d];
    if (bv.x != OVERFLOW_VID) {
        const float px = w.in.plane(PX)[slot], py = w.in.plane(PY)[slot], pz = w.in.plane(PZ)[slot];
        const float h = sc.h, ih = sc.inv_h;
        const float cx = round_div(px, h, ih) - 1.0f, cy = round_div(py, h, ih) - 1.0f,
                    cz = round_div(pz, h, ih) - 1.0f;
        const int bx = (int)cx - 4 * bv.x, by = (int)cy - 4 * bv.y, bz = (int)cz - 4 * bv.z;
        if ((unsigned)bx < 4u && (unsigned)by < 4u && (unsigned)bz < 4u) {
            const f3 ref = mk3(cx * h - px, cy * h - py, cz * h - pz);
            float wx[3], wy[3], wz[3];
            {
                const float fx = -ref.x * ih, fy = -ref.y * ih, fz = -ref.z * ih;
                wx[0] = 0.5f * (1.5f - fx) * (1.5f - fx); wx[1] = 0.75f - (fx - 1.0f) * (fx - 1.0f); wx[2] = 0.5f * (fx - 0.5f) * (fx - 0.5f);
                wy[0] = 0.5f * (1.5f - fy) * (1.5f - fy); wy[1] = 0.75f - (fy - 1.0f) * (fy - 1.0f); wy[2] = 0.5f * (fy - 0.5f) * (fy - 0.5f);
                wz[0] = 0.5f * (1.5f - fz) * (1.5f - fz); wz[1] = 0.75f - (fz - 1.0f) * (fz - 1.0f); wz[2] = 0.5f * (fz - 0.5f) * (fz - 0.5f);
            }
            // No node of the 8 blocks of the stencil (block d and its +1 neighbours) is in
            // reach of a collider: every affinity is empty, the fit has no node and the
            // field is zero.
            if (!w.breach[d]) {
                w.out.uplane(PAFF)[pos] = 0u;
                return 0u;
            }
            GatherGrid gather{w.bup, w.gridv, w.gridv_i, w.ncdf, NONE, NONE, NONE, NONE, NONE, NONE, NONE, NONE};
            gather.prepare(d);
            float nd[27], wq[27];
            uint32_t na[27];
            uint32_t pa = 0u;
            #pragma unroll
            for (int q = 0; q < 27; ++q) {
                const int sx = NBH[q][0], sy = NBH[q][1], sz = NBH[q][2];
                const uint32_t ni = gather.index(bx + sx, by + sy, bz + sz);
                const uint4 nc = ni == NONE ? make_uint4(__float_as_uint(MAX_FLT_REF), 0u, NONE, 0u) : w.ncdf[ni];
                nd[q] = __uint_as_float(nc.x);
                na[q] = nc.y;
                wq[q] = wx[sx] * wy[sy] * wz[sz];
                pa |= nc.y & 0xFFFFu;
            }
            // Sides: kept for colliders known before, from the weighted signed
            // distances for newly reached ones.
            pa |= prev & ((prev & 0xFFFFu) << 16);
            // Only colliders some stencil node is affine to can give a side (for the others
            // every term is zero), and only those not known before need one.
            for (uint32_t todo = pa & ~prev & 0xFFFFu; todo != 0u; todo &= todo - 1u) {
                const uint32_t c = (uint32_t)__ffs(todo) - 1u;
                float acc = 0.0f;
                #pragma unroll
                for (int q = 0; q < 27; ++q) {
                    const float comp = (na[q] >> c) & 1u ? 1.0f : 0.0f;
                    const float sgn = (na[q] >> (16 + c)) & 1u ? -1.0f : 1.0f;
                    acc += comp * wq[q] * sgn * nd[q];
                }
                if (acc < 0.0f) pa |= 0x00010000u << c;
            }
            Sym4 m{0, 0, 0, 0, 0, 0, 0, 0, 0, 0};
            float u[4] = {0.0f, 0.0f, 0.0f, 0.0f};
            #pragma unroll
            for (int q = 0; q < 27; ++q) {
                const uint32_t comb = na[q] & pa & 0xFFFFu;
                if (comb == 0u) continue;
                const uint32_t sdiff = ((na[q] >> 16) ^ (pa >> 16)) & comb;
                const float sx = (float)NBH[q][0] * h, sy = (float)NBH[q][1] * h, sz = (float)NBH[q][2] * h;
                const float dx = ref.x + sx, dy = ref.y + sy, dz = ref.z + sz;
                const float wgt = wq[q];
                const float dd = sdiff == 0u ? nd[q] : -nd[q];
                m.q00 += dx * dx * wgt; m.q01 += dx * dy * wgt; m.q02 += dx * dz * wgt; m.q03 += dx * wgt;
                m.q11 += dy * dy * wgt; m.q12 += dy * dz * wgt; m.q13 += dy * wgt;
                m.q22 += dz * dz * wgt; m.q23 += dz * wgt;
                m.q33 += wgt;
                u[0] += dx * (wgt * dd); u[1] += dy * (wgt * dd); u[2] += dz * (wgt * dd); u[3] += wgt * dd;
            }
            float res[4];
            if (sym4_solve(m, u, res)) {
                const f3 g = mk3(res[0], res[1], res[2]);
                const float len = length(g);
                nrm = len > 1.0e-6f ? g / len : mk3(0, 0, 0);
                sd = res[3];
                aff = pa;
            } else {
                aff = 0u;
            }
        }
    }
    // The normal and signed distance are only read where the affinity is not empty.
    w.out.uplane(PAFF)[pos] = aff;
    if (aff == 0u) return 0u;
    w.out.plane(PNX)[pos] = nrm.x;
    w.out.plane(PNY)[pos] = nrm.y;
    w.out.plane(PNZ)[pos] = nrm.z;
    w.out.plane(PSD)[pos] = sd;
    return aff;
}

// Appends pos to a list (one counter atomic per wave; the order does not matter).
__device__ inline void wave_append(uint32_t *list, uint32_t *count, bool take, uint32_t pos)
{
    const uint32_t l = lane_id();
    const uint64_t active = __ballot(1), m = __ballot(take);
    if (!m) return;
    const uint32_t leader = (uint32_t)__ffsll((unsigned long long)active) - 1u;
    uint32_t base = 0u;
    if (l == leader) base = atomicAdd(count, (uint32_t)__popcll(m));
    base = __shfl(base, (int)leader, WAVE);
    if (take) list[base + (uint32_t)__popcll(m & ((1ull << l) - 1ull))] = pos;
}

// Per particle of a CPIC scene: its contact field (particle_cdf_one); the particles left
// with affinity bits go to the contact list that k_g2p_contact processes densely.
__global__ void __launch_bounds__(256) k_particle_cdf(WorldDev w)
{
    uint32_t pbegin, pend;
    xcd_range(w.g->p_out, pbegin, pend);
    for (uint32_t pos = pbegin + threadIdx.x; pos < pend; pos += blockDim.x) {
        const uint32_t d = w.sblock[pos];
        const SceneDev sc = w.scenes[w.bscene[d]];
        const bool contact = sc.cpic && (particle_cdf_one(w, pos, d, sc) & 0xFFFFu) != 0u;
        wave_append(w.clist, &w.g->n_contact, contact, pos);
    }
}

__global__ void __launch_bounds__(256) k_timestep_bound(WorldDev w, uint32_t n, uint32_t *out, uint32_t stride)
{
    const uint32_t nr = (n + WAVE - 1) / WAVE * WAVE;
    uint32_t cur_s = NONE, cur_min = 0xFFFFFFFFu;     // per lane: running minimum of one scene
    for (uint32_t i = blockIdx.x * blockDim.x + threadIdx.x; i < nr; i += gridDim.x * blockDim.x) {
        if (i >= n) continue;
        const uint32_t fl = w.in.uplane(PFLAGS)[i];
        const uint32_t s = flags_scene(fl);
        const SceneDev sc = w.scenes[s];
        if (!sc.active || !(fl & FLAG_ENABLED)) continue;
        const uint32_t cand = arena_dt_bound(w.in, i, fl, sc, w.classes);
        if (s != cur_s) {
            if (cur_s != NONE) atomicMin(&out[(size_t)cur_s * stride], cur_min);
            cur_s = s;
            cur_min = cand;
        } else {
            cur_min = min(cur_min, cand);
        }
    }
    wave_scene_min(cur_s, cur_min, out, stride);
}

// ------------------------------------------------------------------------------------
// Canonical sort readback (not on the hot path): per sorted particle its primary
// block and local cell, and the ten bucket counts of every block including the
// spilled extras (grid/sort.rs:287-349).
__global__ void k_canonical(WorldDev w, Arena prev, uint32_t *pcell_out, uint32_t *buckets)
{
    const uint32_t n = w.g->p_out;
    for (uint32_t pos = blockIdx.x * blockDim.x + threadIdx.x; pos < n; pos += gridDim.x * blockDim.x) {
        const uint32_t slot = w.perm[pos];
        const uint32_t d = w.sblock[pos];
        const int4 bv = w.bvid[d];
        const SceneDev sc = w.scenes[w.bscene[d]];
        if (bv.x == OVERFLOW_VID) { pcell_out[pos] = NONE; continue; }
        int32_t b[3];
        uint32_t loc[3];
        cell_of(prev.plane(PX)[slot], sc.h, sc.inv_h, b[0], loc[0]);
        cell_of(prev.plane(PY)[slot], sc.h, sc.inv_h, b[1], loc[1]);
        cell_of(prev.plane(PZ)[slot], sc.h, sc.inv_h, b[2], loc[2]);
        pcell_out[pos] = loc[0] + 4 * loc[1] + 16 * loc[2];
        atomicAdd(&buckets[10 * d + loc[2]], 1u);
        for (int i = 1; i < 8; ++i) {
            const int sx = ASSOC[i][0], sy = ASSOC[i][1], sz = ASSOC[i][2];
            if ((sx && loc[0] < 2) || (sy && loc[1] < 2) || (sz && loc[2] < 2)) continue;
            const uint32_t dn = w.bup[8 * d + i];
            if (dn == NONE) continue;
            int lz = (int)loc[2] - sz * 4;
            if (lz < -2) lz = -2;
            atomicAdd(&buckets[10 * dn + 4 + (lz + 2)], 1u);
        }
    }
}

// ------------------------------------------------------------------------------------
// Launch sequence.

static inline int grid_for(uint64_t n, int threads, int cap)
{
    uint64_t g = (n + threads - 1) / threads;
    if (g < 1) g = 1;
    if (g > (uint64_t)cap) g = cap;
    g = (g + NUM_XCD - 1) / NUM_XCD * NUM_XCD;   // whole XCD rounds (xcd_range)
    return (int)g;
}

// Workgroups of k_keys_touch: four a CU at most, each with consecutive particles.
static inline int key_groups(uint64_t n)
{
    return (int)std::min<uint64_t>(std::max<uint64_t>((n + KEY_GROUP - 1) / KEY_GROUP, 1), 1024);
}

// Workgroups of k_g2p_update: enough that xcd_range gives none more than `threads` (its
// workgroup size) of the at most p_hint sorted positions (one per thread).
static inline int g2p_groups(uint64_t p_hint, int threads)
{
    return grid_for(p_hint, threads, std::numeric_limits<int>::max() / 2);
}

// Slots up to which the hash is scanned in tiles of 1024 rather than 16,384: small tiles
// leave more waves to write the block tables, large ones take fewer tickets and shorter
// look-backs.  1024 and 16,384: 6.5 and 10 us at 120,000 particles, 7.6 and 12.3 at 1M
// (2^17 slots), 10.8 and 15.3 for 32 scenes, 80 and 23 at 2^22 slots.
constexpr uint32_t SMALL_HASH = 1u << 20;

// Particles from which an unsorted count goes through LDS: few particles have few runs per
// block, and its barriers show.  Calls without and with: 5000 of one material 69-70 and
// 71-72 us, 8000 75-77 and 74-77 (sand 78 and 73), 12,000 80-82 and 75-78, 32,000 sand 91 and 87.
constexpr uint64_t UNSORTED_MIN = 8192;

void launch_substep(const WorldDev &w, const LaunchConfig &lc, hipStream_t st, hipEvent_t *ev, bool keys)
{
    const int T = 256;
    const int cap = lc.persistent_blocks;
    if (ev) (void)hipEventRecord(ev[0], st);
    if (keys) k_keys_touch<<<key_groups(lc.p_hint), KEY_GROUP, 0, st>>>(w);
    // Adaptive scenes after a host change: the bound of the input state (otherwise the
    // previous substep's G2P left it in the clocks).
    if (keys && w.any_adaptive && w.clock)
        k_timestep_bound<<<grid_for(lc.p_hint, T, cap), T, 0, st>>>(w, (uint32_t)lc.p_hint, &w.clock[0].bound,
                                                                      (uint32_t)(sizeof(SceneClock) / 4));
    auto slots = [&](auto kernel, int threads, uint32_t tile) {
        const int tiles = std::min((int)((w.h_total + tile - 1) / tile), cap);
        kernel<<<std::max(tiles, 1), threads, 0, st>>>(w);
    };
    if (w.h_total <= SMALL_HASH) slots(k_scan_slots<4, 4>, 4 * WAVE, slot_tile<4, 4>());
    else slots(k_scan_slots<16, 16>, 16 * WAVE, slot_tile<16, 16>());
    auto count = [&](auto kernel, int threads) {
        const int counting = grid_for(lc.p_hint, threads, cap);
        kernel<<<counting + grid_for((uint64_t)w.b_total * 16, threads, cap), threads, 0, st>>>(w, (uint32_t)counting);
    };
    if ((keys || lc.unsorted) && lc.p_hint >= UNSORTED_MIN) count(k_block_count<true>, KEY_GROUP);
    else count(k_block_count<false>, T);
    const uint32_t btile = SCAN_TILE * scan_chunks(w.b_total);
    const int bscan = std::min((int)((w.b_total + btile - 1) / btile), cap);
    k_scan_counts<<<std::max(bscan, 1), 256, 0, st>>>(w);
    k_scatter<<<grid_for(lc.p_hint, T, cap), T, 0, st>>>(w);
    // Workgroups of one wave, one block each (blocks with 4 particles or more).
    if (lc.order) k_cell_order<<<grid_for(std::min<uint64_t>(w.b_total, lc.p_hint), 1, 16 * cap), WAVE, 0, st>>>(w);
    if (ev) (void)hipEventRecord(ev[1], st);
    const int pg = lc.p2g_blocks;
    if (w.any_cpic) {
        // CPIC worlds: the contact distance fields, then the CPIC variants of the
        // transfers (scenes without CPIC take the plain path inside them).
        if (w.n_rp) k_mesh_cdf<<<grid_for(w.n_rp, T, cap), T, 0, st>>>(w);
        k_grid_cdf<<<grid_for((uint64_t)w.b_total * 64, T, cap), T, 0, st>>>(w);   // one wave per block
        k_particle_cdf<<<grid_for(lc.p_hint, T, cap), T, 0, st>>>(w);
        if (ev) hipExtLaunchKernelGGL(k_p2g<true>, dim3(pg), dim3(P2G_WAVES * WAVE), 0, st, ev[5], ev[6], 0, w);
        else k_p2g<true><<<pg, P2G_WAVES * WAVE, 0, st>>>(w);
        if (ev) (void)hipEventRecord(ev[2], st);
        if (w.mesh_pass) k_grid_update<true, true><<<grid_for((uint64_t)w.b_total * 64, T, cap), T, 0, st>>>(w);
        else k_grid_update<true, false><<<grid_for((uint64_t)w.b_total * 64, T, cap), T, 0, st>>>(w);
        if (ev) (void)hipEventRecord(ev[3], st);
        // The contact particles' G2P, then the plain particles', which also integrates the
        // bodies.  (Side by side on two streams the fork, the join and a launch for the bodies
        // cost more than the overlap gave, frames of 20 substeps: 60,000 particles 2925 -> 2618
        // us, 262,144 3875 -> 3600, 1,048,576 7865 -> 7650, sand on a mesh ramp 3350 -> 3127.)
        // Adaptive worlds take the variants that also min-reduce the next substep's bound.
        if (w.any_adaptive) k_g2p_contact<true><<<grid_for(lc.p_hint, T, cap), T, 0, st>>>(w);
        else k_g2p_contact<false><<<grid_for(lc.p_hint, T, cap), T, 0, st>>>(w);
        auto g2p = w.any_adaptive ? k_g2p_update<true, true> : k_g2p_update<true, false>;
        constexpr int GT = g2p_threads<true>();
        if (ev) hipExtLaunchKernelGGL(g2p, dim3(g2p_groups(lc.p_hint, GT)), dim3(GT), 0, st, ev[7], ev[8], 0, w);
        else g2p<<<g2p_groups(lc.p_hint, GT), GT, 0, st>>>(w);
    } else {
        if (ev) hipExtLaunchKernelGGL(k_p2g<false>, dim3(pg), dim3(P2G_WAVES * WAVE), 0, st, ev[5], ev[6], 0, w);
        else k_p2g<false><<<pg, P2G_WAVES * WAVE, 0, st>>>(w);
        if (ev) (void)hipEventRecord(ev[2], st);
        if (w.mesh_pass) k_grid_update<false, true><<<grid_for((uint64_t)w.b_total * 64, T, cap), T, 0, st>>>(w);
        else k_grid_update<false, false><<<grid_for((uint64_t)w.b_total * 64, T, cap), T, 0, st>>>(w);
        if (ev) (void)hipEventRecord(ev[3], st);
        auto g2p = w.any_adaptive ? k_g2p_update<false, true> : k_g2p_update<false, false>;
        constexpr int GT = g2p_threads<false>();
        if (ev) hipExtLaunchKernelGGL(g2p, dim3(g2p_groups(lc.p_hint, GT)), dim3(GT), 0, st, ev[7], ev[8], 0, w);
        else g2p<<<g2p_groups(lc.p_hint, GT), GT, 0, st>>>(w);
    }
    if (ev) (void)hipEventRecord(ev[4], st);
}

__global__ void k_set_particles(Globals *g, uint32_t p_in) { g->p_in = p_in; }

void launch_set_particles(Globals *g, uint32_t p_in, hipStream_t st)
{
    k_set_particles<<<1, 1, 0, st>>>(g, p_in);
}

void launch_clear(const WorldDev &w, const LaunchConfig &lc, hipStream_t st)
{
    const int T = 256;
    k_clear<<<grid_for(clear_len(w), T, lc.persistent_blocks), T, 0, st>>>(w);
}

void launch_timestep_bound(const WorldDev &w, uint32_t n, uint32_t *out, uint32_t stride, int max_blocks, hipStream_t st)
{
    k_timestep_bound<<<grid_for(n, 256, max_blocks), 256, 0, st>>>(w, n, out, stride);
}

void launch_canonical(const WorldDev &w, const Arena &prev, uint32_t *pcell, uint32_t *buckets, uint32_t p_hint,
                      hipStream_t st)
{
    k_canonical<<<grid_for(p_hint, 256, 4096), 256, 0, st>>>(w, prev, pcell, buckets);
}

// ------------------------------------------------------------------------------------
// State readback: particles in id order, so that the host takes whole arrays by one copy
// (it copied and scattered every component by itself: 3.9 ms for the positions of 1M
// particles whose 20 substeps take 5 ms; 0.5 ms now, most of it the copy over the bus and
// the host's own).  Bound by the scattered row writes.
__global__ void __launch_bounds__(256) k_read_rows(Arena a, uint32_t start, uint32_t count, ReadList list, float *out)
{
    for (uint32_t i = blockIdx.x * blockDim.x + threadIdx.x; i < count; i += gridDim.x * blockDim.x) {
        const uint32_t slot = start + i;
        const size_t id = a.uplane(PID)[slot];
        for (int k = 0; k < list.n; ++k) {
            const ReadRows r = list.rows[k];
            for (int c = 0; c < r.comps; ++c) out[r.off + id * r.comps + c] = a.plane(r.plane + c)[slot];
        }
    }
}

void launch_read_rows(const Arena &a, uint32_t start, uint32_t count, const ReadList &list, float *out, int cap,
                      hipStream_t st)
{
    if (count == 0) return;
    k_read_rows<<<grid_for(count, 256, cap), 256, 0, st>>>(a, start, count, list, out);
}

// ------------------------------------------------------------------------------------
// Render readback: gpu_prep_readback (src_mpm_shaders/solver/prep_readback.rs:245-300)
// over arena positions [start, start + count) of one scene, written at each particle's id
// as 24 floats (ReadbackData: colour, deformation as a column-major 4x4 with the 3x3 in
// its upper left, position, padding).  group / phase / radius are the particles' constant
// properties by id; cdf says whether the scene's contact field is live (CPIC).
__global__ void __launch_bounds__(256) k_prep_readback(Arena a, uint32_t start, uint32_t count, const uint32_t *group,
                                                       const float *phase, const float *radius, const float4 *palette,
                                                       uint32_t npal, uint32_t mode, float h, float dt, uint32_t cdf,
                                                       float *out)
{
    for (uint32_t i = blockIdx.x * blockDim.x + threadIdx.x; i < count; i += gridDim.x * blockDim.x) {
        const uint32_t slot = start + i;
        const uint32_t id = a.uplane(PID)[slot];
        const uint32_t fl = a.uplane(PFLAGS)[slot];
        m3 F;
        F.c0 = mk3(a.plane(PF0)[slot], a.plane(PF1)[slot], a.plane(PF2)[slot]);
        F.c1 = mk3(a.plane(PF3)[slot], a.plane(PF4)[slot], a.plane(PF5)[slot]);
        F.c2 = mk3(a.plane(PF6)[slot], a.plane(PF7)[slot], a.plane(PF8)[slot]);
        const float4 base = palette[group[id] % npal];
        // compute_deformation (:97-118): diag(2 r) times F with entries clamped to [-4, 4].
        const float d = radius[id] * 2.0f;
        float *o = out + 24 * (size_t)id;
        const f3 cols[3] = {F.c0, F.c1, F.c2};
        #pragma unroll
        for (int c = 0; c < 3; ++c) {
            o[4 + 4 * c + 0] = d * fminf(fmaxf(cols[c].x, -4.0f), 4.0f);
            o[4 + 4 * c + 1] = d * fminf(fmaxf(cols[c].y, -4.0f), 4.0f);
            o[4 + 4 * c + 2] = d * fminf(fmaxf(cols[c].z, -4.0f), 4.0f);
            o[4 + 4 * c + 3] = 0.0f;
        }
        o[16] = 0.0f; o[17] = 0.0f; o[18] = 0.0f; o[19] = 1.0f;
        // compute_color (:170-243).
        float4 col = base;
        const uint32_t aff = cdf ? a.uplane(PAFF)[slot] : 0u;
        if (mode == 2u) {           // velocity
            const f3 v = mk3(a.plane(PVX)[slot], a.plane(PVY)[slot], a.plane(PVZ)[slot]);
            col = make_float4(fabsf(v.x) * dt * 100.0f + 0.2f, fabsf(v.y) * dt * 100.0f + 0.2f,
                              fabsf(v.z) * dt * 100.0f + 0.2f, base.w);
        } else if (mode == 1u) {    // volume: singular values of F, largest first
            m3 U, V;
            f3 sv;
            svd3(F, U, sv, V);
            float s0 = sv.x, s1 = sv.y, s2 = sv.z, t;
            if (s0 < s1) { t = s0; s0 = s1; s1 = t; }
            if (s1 < s2) { t = s1; s1 = s2; s2 = t; }
            if (s0 < s1) { t = s0; s0 = s1; s1 = t; }
            col = make_float4((1.0f - s0) / 0.005f + 0.2f, (1.0f - s1) / 0.005f + 0.2f, (1.0f - s2) / 0.005f + 0.2f,
                              base.w);
        } else if (mode == 3u) {    // phase
            const float ph = phase[id];
            col = make_float4(0.0f, 0.4f * ph, 0.4f * (1.0f - ph), base.w);
        } else if (mode == 4u) {    // contact normals
            const f3 n = aff ? mk3(a.plane(PNX)[slot], a.plane(PNY)[slot], a.plane(PNZ)[slot]) : mk3(0, 0, 0);
            col = n.x == 0.0f && n.y == 0.0f && n.z == 0.0f
                      ? make_float4(0.0f, 0.0f, 0.0f, base.w)
                      : make_float4((n.x + 1.0f) * 0.5f, (n.y + 1.0f) * 0.5f, (n.z + 1.0f) * 0.5f, base.w);
        } else if (mode == 5u) {    // contact signed distances
            const float sd = aff ? a.plane(PSD)[slot] : 0.0f;
            const float dd = sd / (h * 1.5f);
            col = dd > 0.0f ? make_float4(0.0f, fabsf(dd), 0.0f, base.w) : make_float4(fabsf(dd), 0.0f, 0.0f, base.w);
        } else if (mode == 6u) {    // contact sides
            const uint32_t inside = (aff >> 16) & (aff & 0xFFFFu);
            col = aff == 0u ? make_float4(0.0f, 0.0f, 0.0f, base.w)
                            : (inside == 0u ? make_float4(0.0f, 1.0f, 0.0f, base.w)
                                            : make_float4(1.0f, 0.0f, 0.0f, base.w));
        }
        if (!(fl & FLAG_ENABLED)) col = make_float4(1.0f, 0.0f, 0.0f, 1.0f);   // failed particles in red
        o[0] = col.x; o[1] = col.y; o[2] = col.z; o[3] = col.w;
        o[20] = a.plane(PX)[slot]; o[21] = a.plane(PY)[slot]; o[22] = a.plane(PZ)[slot]; o[23] = 0.0f;
    }
}

void launch_prep_readback(const Arena &a, uint32_t start, uint32_t count, const uint32_t *group, const float *phase,
                          const float *radius, const float4 *palette, uint32_t npal, uint32_t mode, float h, float dt,
                          bool cdf, float *out, int cap, hipStream_t st)
{
    if (count == 0) return;
    const int T = 256;
    k_prep_readback<<<grid_for(count, T, cap), T, 0, st>>>(a, start, count, group, phase, radius, palette, npal, mode,
                                                          h, dt, cdf ? 1u : 0u, out);
}

// ------------------------------------------------------------------------------------
// Substep without allocation: the world's tables and arenas live in a buffer the host
// carved up (the library's static scratch array); the particles come from and return to
// the caller's arrays in id order.

// Tables and counters (by the first workgroup), and the empty hash and scan states.
__global__ void __launch_bounds__(256) k_noalloc_setup(WorldDev w, NoallocTables t)
{
    clear_tables(w);
    if (blockIdx.x != 0) return;
    const uint32_t tid = threadIdx.x;
    if (tid == 0) {
        *const_cast<SceneDev *>(w.scenes) = t.scene;
        w.ctr[0] = SceneCtr{0u, 0u, 0u, 0u};
        const_cast<uint32_t *>(w.region_start)[0] = 0u;
        const_cast<uint32_t *>(w.region_scene)[0] = 0u;
        w.g->p_in = t.n;
        w.g->n_contact = 0u;
    }
    if (tid < t.n_classes) const_cast<ClassDev *>(w.classes)[tid] = t.classes[tid];
    if (tid < t.n_cols) {
        ColliderDev c{};
        float *words = reinterpret_cast<float *>(&c);
        for (int k = 0; k < COLLIDER_BODY_WORDS; ++k) words[k] = t.cols[tid].body[k];
        c.shape = SHAPE_CUBOID;
        c.reach = t.cols[tid].reach;
        w.cols[tid] = c;
    }
}

// The input arena from the caller's arrays, and the particles' keys and block insertions
// from the same registers (k_keys_touch's work).  Every array is read before the first
// store: the compiler must assume that they may overlap.  As two kernels, the keys by runs:
// 31,337 particles 6 + 37 us, 120,001 8 + 61; as one 9.5 and 12.5.
__global__ void __launch_bounds__(KEY_GROUP) k_noalloc_pack(WorldDev w, NoallocParticles p, uint32_t n, uint32_t n_classes)
{
    __shared__ KeySet set;
    mark_overflow_slots(w);
    set.clear();
    const Arena a = w.in;
    const float h = w.scenes[0].h;
    uint32_t begin, end;
    key_range(n, begin, end);
    for (uint32_t c = begin; c < end; c += KEY_GROUP) {
        const uint32_t i = c + threadIdx.x;
        const bool valid = i < n;
        f3 x = mk3(0, 0, 0);
        uint32_t codes = 0u;
        if (valid) {
            x = load3(p.x, i);
            const f3 v = load3(p.v, i);
            const f3 C0 = load3(p.C, 3 * (size_t)i), C1 = load3(p.C, 3 * (size_t)i + 1), C2 = load3(p.C, 3 * (size_t)i + 2);
            const f3 F0 = load3(p.F, 3 * (size_t)i), F1 = load3(p.F, 3 * (size_t)i + 1), F2 = load3(p.F, 3 * (size_t)i + 2);
            const float mass = p.mass[i], vol0 = p.vol0[i];
            const f3 given = p.pstate ? load3(p.pstate, i) : mk3(0, 0, 0);
            const uint32_t f = p.flags[i];
            uint32_t cls = flags_class(f);
            if (cls >= n_classes) {
                // A material index outside the table: reported, and the particle takes material 0.
                atomicOr(&w.ctr[0].err, ERR_MODEL);
                cls = 0u;
            }
            // Plastic state: the caller's, or the material's initial words (the sand tags'
            // three, snow's one), as an upload takes it from the particle's model words.
            const ClassDev &k = w.classes[cls];
            const uint32_t tag = k.tag;
            const int pw = (tag == 2u || tag == 3u) ? 3 : tag == 5u ? 1 : 0;
            const float ps0 = pw > 0 ? (p.pstate ? given.x : k.w[0]) : 0.0f;
            const float ps1 = pw > 1 ? (p.pstate ? given.y : k.w[1]) : 0.0f;
            const float ps2 = pw > 2 ? (p.pstate ? given.z : k.w[2]) : 0.0f;
            const uint32_t flags = make_flags((f & FLAG_ENABLED) != 0u, (f & FLAG_FIXED) != 0u, cls, 0u);
            a.quad(0)[i] = make_float4(x.x, x.y, x.z, __uint_as_float(flags));
            a.quad(1)[i] = make_float4(v.x, v.y, v.z, 0.0f);
            a.quad(2)[i] = make_float4(C0.x, C0.y, C0.z, C1.x);
            a.quad(3)[i] = make_float4(C1.y, C1.z, C2.x, C2.y);
            a.quad(4)[i] = make_float4(C2.z, mass, vol0, __uint_as_float(i));
            a.quad(5)[i] = make_float4(F0.x, F0.y, F0.z, F1.x);
            a.quad(6)[i] = make_float4(F1.y, F1.z, F2.x, F2.y);
            a.quad(7)[i] = make_float4(F2.z, ps0, ps1, ps2);
            a.quad(8)[i] = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
            if (flags & FLAG_ENABLED) codes = bound_codes(v, m3{C0, C1, C2}, mass, h);
        }
        set.particle(w, i, valid, 0u, x, codes);
    }
}

// The caller's arrays from the output arena, by particle id.  A particle's eight loads are
// issued before its first store (one word at a time, each load waiting for the store before
// it: 1000 particles 8 us, 120,001 18; now 3 and 10).
__global__ void __launch_bounds__(256) k_noalloc_unpack(WorldDev w, NoallocParticles p, uint32_t n)
{
    const Arena a = w.out;
    for (uint32_t pos = blockIdx.x * blockDim.x + threadIdx.x; pos < n; pos += gridDim.x * blockDim.x) {
        const float4 q0 = a.quad(0)[pos], q1 = a.quad(1)[pos], q2 = a.quad(2)[pos], q3 = a.quad(3)[pos],
                     q4 = a.quad(4)[pos], q5 = a.quad(5)[pos], q6 = a.quad(6)[pos], q7 = a.quad(7)[pos];
        const uint32_t id = __float_as_uint(q4.w);
        if (id >= n) continue;
        store3(p.x, id, mk3(q0.x, q0.y, q0.z));
        store3(p.v, id, mk3(q1.x, q1.y, q1.z));
        const size_t r = 3 * (size_t)id;
        store3(p.C, r, mk3(q2.x, q2.y, q2.z));
        store3(p.C, r + 1, mk3(q2.w, q3.x, q3.y));
        store3(p.C, r + 2, mk3(q3.z, q3.w, q4.x));
        store3(p.F, r, mk3(q5.x, q5.y, q5.z));
        store3(p.F, r + 1, mk3(q5.w, q6.x, q6.y));
        store3(p.F, r + 2, mk3(q6.z, q6.w, q7.x));
        p.mass[id] = q4.y;
        if (p.pstate) store3(p.pstate, id, mk3(q7.y, q7.z, q7.w));
        const uint32_t f = __float_as_uint(q0.w);
        p.flags[id] = (f & (FLAG_ENABLED | FLAG_FIXED)) | (flags_class(f) << 2);
    }
    if (blockIdx.x == 0 && threadIdx.x == 0 && p.errors) p.errors[0] = w.ctr[0].err;
}

void launch_noalloc_setup(const WorldDev &w, const NoallocTables &t, const NoallocParticles &p, int cap, hipStream_t st)
{
    const int T = 256;
    k_noalloc_setup<<<grid_for(clear_len(w), T, cap), T, 0, st>>>(w, t);
    k_noalloc_pack<<<key_groups(t.n), KEY_GROUP, 0, st>>>(w, p, t.n, t.n_classes);
}

void launch_noalloc_unpack(const WorldDev &w, const NoallocParticles &p, uint32_t n, int cap, hipStream_t st)
{
    const int T = 256;
    k_noalloc_unpack<<<grid_for(std::max<uint32_t>(n, 1u), T, cap), T, 0, st>>>(w, p, n);
}

}  // namespace nxm
