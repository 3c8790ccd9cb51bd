// Host-side bounds model of the hot kernels' fetch patterns (plain g++, no GPU): runs the address
// arithmetic of litenn_amd/csrc/fetch_model.hpp -- the very functions the kernels call -- for every
// thread of a launch over page-exact, ragged and minimal shapes, and checks
//   * every requested 16-byte piece is 16-byte aligned and holds at least one byte of its tensor
//     (so it lies in a page the tensor occupies);
//   * the pieces a kernel consumes are fetched from the right addresses and cover what it reads;
//   * rows, activation elements and cache rows are each covered, none outside its array.
// It also shows that the checker has teeth: the matrix-core GEMM's piece arithmetic as it was before
// its over-fetch was fixed (no redirection of a piece that holds no byte of its chunk) fails on the
// Q2_K 512 x 512 tensor that once faulted a GPU.
#include <cstdint>
#include <cstdio>
#include <cstdlib>
#include <map>
#include <vector>

#include "../../litenn_amd/csrc/fetch_model.hpp"
#include "../../litenn_amd/csrc/room.hpp"

namespace fm = litenn_hip::fetch;

static int g_failures = 0;
#define CHECK(cond, ...)                                                                                               \
	do                                                                                                                 \
	{                                                                                                                  \
		if (!(cond))                                                                                                   \
		{                                                                                                              \
			if (++g_failures <= 20)                                                                                    \
			{                                                                                                          \
				std::printf("FAIL %s:%d %s: ", __FILE__, __LINE__, #cond);                                             \
				std::printf(__VA_ARGS__);                                                                              \
				std::printf("\n");                                                                                     \
			}                                                                                                          \
		}                                                                                                              \
	} while (0)

struct Format
{
	const char* name;
	int chunk_bytes;   // bytes of 256 elements
	bool aligned16;    // the GEMM's view: chunks start on 16-byte boundaries
	int base_align;    // what the GEMM launcher demands of the tensor's address
	int stream_slice;  // bytes of 4096 elements (one wavefront's slice in the streaming GEMV)
};
static const Format kFormats[] = {
	{ "Q4_0", 144, true, 16, 2304 }, { "Q4_1", 160, true, 16, 2560 }, { "Q5_0", 176, true, 16, 2816 },
	{ "Q5_1", 192, true, 16, 3072 }, { "Q8_0", 272, true, 16, 4352 }, { "Q4_K", 144, true, 16, 2304 },
	{ "Q5_K", 176, true, 16, 2816 }, { "Q2_K", 84, false, 4, 1344 },  { "Q3_K", 110, false, 2, 1760 },
	{ "Q6_K", 210, false, 2, 3360 },
};

constexpr uintptr_t kPage = 4096;

// ---- matrix-core GEMM weight pieces -------------------------------------------------------------
typedef uintptr_t (*PieceFn)(uintptr_t, int, int, bool, int);

static uintptr_t piece_without_redirection(uintptr_t row_start, int c, int chunk_bytes, bool aligned16, int offset)
{
	const uintptr_t chunk = row_start + static_cast<size_t>(c) * chunk_bytes;
	return (aligned16 ? chunk : (chunk & ~uintptr_t{ 15 })) + offset;
}

// returns the number of pieces that touch no byte of [base, base + bytes)
// base_up != 0: the gated form (ng = 2), whose second weight group holds the same rows of a second
// n-row matrix at base_up
static long gemm_case(const Format& f, int ng, int waves, int n, int chunks, uintptr_t base, PieceFn piece_fn,
                      bool check_contents, uintptr_t base_up = 0)
{
	const bool gated = base_up != 0;
	const size_t row_bytes = static_cast<size_t>(chunks) * f.chunk_bytes;
	const size_t bytes = static_cast<size_t>(n) * row_bytes;
	const int pieces = fm::gemm_weight_pieces(f.chunk_bytes, f.aligned16);
	const int loads = (ng * 16 * pieces + 63) / 64;
	const int bn = gated ? 16 * waves : 16 * waves * ng;
	const auto matrix_of = [&](int slot_row) { return gated && slot_row >= 16 ? base_up : base; };
	const auto row_of = [&](int slot_row) { return gated ? (slot_row & 15) : slot_row; };
	long outside = 0;
	for (int block = 0; block < (n + bn - 1) / bn; ++block)
	{
		for (int wave = 0; wave < waves; ++wave)
		{
			const int n_base = (block * waves + wave) * 16 * (gated ? 1 : ng);
			for (int c = 0; c < chunks; ++c)
			{
				std::map<int, uintptr_t> slot; // slot byte offset of a piece -> where it was fetched from
				for (int i = 0; i < loads; ++i)
				{
					for (int lane = 0; lane < 64; ++lane)
					{
						const fm::GemmWeightRequest rq = fm::gemm_weight_request(i, lane, ng, pieces);
						if (!(64 * (i + 1) <= ng * 16 * pieces || rq.issued))
						{
							continue;
						}
						CHECK(rq.row >= 0 && rq.row < 16 * ng && rq.offset >= 0 && rq.offset < 16 * pieces, "%s row %d off %d",
						      f.name, rq.row, rq.offset);
						const uintptr_t mbase = matrix_of(rq.row), end = mbase + bytes;
						const uintptr_t row_start =
						    mbase + static_cast<size_t>(fm::gemm_weight_row(n_base, row_of(rq.row), n)) * row_bytes;
						const uintptr_t from = piece_fn(row_start, c, f.chunk_bytes, f.aligned16, rq.offset);
						if (check_contents)
						{
							CHECK(from % 16 == 0, "%s n %d: piece at %#zx is not aligned", f.name, n, static_cast<size_t>(from));
						}
						if (!(from < end && from + 16 > mbase))
						{
							++outside;
						}
						// the i-th instruction writes 1 KB of the slot: lane l at 1024 i + 16 l
						slot[1024 * i + 16 * lane] = from;
					}
				}
				if (!check_contents)
				{
					continue;
				}
				// what the decoders read: row r of the wavefront at slot offset r * 16 pieces + mis,
				// chunk_bytes bytes, which must be the chunk's own bytes
				for (int r = 0; r < 16 * ng; ++r)
				{
					const uintptr_t row_start =
					    matrix_of(r) + static_cast<size_t>(fm::gemm_weight_row(n_base, row_of(r), n)) * row_bytes;
					const uintptr_t chunk = row_start + static_cast<size_t>(c) * f.chunk_bytes;
					const int mis = fm::gemm_weight_misalignment(row_start, c, f.chunk_bytes, f.aligned16);
					for (int b = 0; b < f.chunk_bytes; ++b)
					{
						const int at = r * 16 * pieces + mis + b;
						const auto it = slot.find(at & ~15);
						CHECK(it != slot.end() && it->second + (at & 15) == chunk + b, "%s n %d chunk %d row %d byte %d", f.name, n, c,
						      r, b);
					}
				}
			}
		}
	}
	return outside;
}

static void test_gemm_weight_pieces()
{
	const int tiles[][2] = { { 2, 8 }, { 1, 8 }, { 1, 4 } }; // weight groups per wavefront, wavefronts
	long cases = 0;
	for (const Format& f : kFormats)
	{
		for (const auto& t : tiles)
		{
			for (int n : { 1, 15, 16, 17, 33, 128, 129, 512 })
			{
				for (int chunks : { 1, 2, 3, 8 })
				{
					const size_t bytes = static_cast<size_t>(n) * chunks * f.chunk_bytes;
					std::vector<uintptr_t> bases;
					for (int mis = 0; mis < 16; mis += f.base_align)
					{
						bases.push_back(64 * kPage + mis); // every misalignment the launcher accepts
					}
					const uintptr_t ends_on_page = 1024 * kPage - bytes; // the tensor's last byte is a page's last
					if (ends_on_page % f.base_align == 0)
					{
						bases.push_back(ends_on_page);
					}
					for (uintptr_t base : bases)
					{
						const long outside = gemm_case(f, t[0], t[1], n, chunks, base, fm::gemm_weight_piece, true);
						CHECK(outside == 0, "%s ng %d waves %d n %d chunks %d base %#zx: %ld pieces outside the tensor", f.name, t[0],
						      t[1], n, chunks, static_cast<size_t>(base), outside);
						++cases;
						// the gated form: the gate matrix at `base`, the up matrix ending on a page far behind it
						const uintptr_t up = 4096 * kPage - bytes;
						if (t[0] == 2 && up % f.base_align == 0)
						{
							const long out2 = gemm_case(f, 2, t[1], n, chunks, base, fm::gemm_weight_piece, true, up);
							CHECK(out2 == 0, "%s gated n %d chunks %d base %#zx: %ld pieces outside their matrix", f.name, n, chunks,
							      static_cast<size_t>(base), out2);
							++cases;
						}
					}
				}
			}
		}
	}
	std::printf("gemm weight pieces: %ld launches walked\n", cases);
	// the arithmetic as it was before the fix, on the tensor that faulted: Q2_K, 512 rows of 512
	// elements = 21 pages exactly; the last piece of the last rows' last chunk lies in the next page
	const Format& q2k = kFormats[7];
	const size_t bytes = 512 * 2 * 84;
	CHECK(bytes == 21 * kPage, "Q2_K 512 x 512 is 21 pages");
	const long before = gemm_case(q2k, 1, 4, 512, 2, 512 * kPage, piece_without_redirection, false);
	const long after = gemm_case(q2k, 1, 4, 512, 2, 512 * kPage, fm::gemm_weight_piece, false);
	CHECK(before > 0, "the pre-fix arithmetic must be caught");
	CHECK(after == 0, "the current arithmetic stays inside");
	std::printf("Q2_K 512 x 512, page-exact: %ld pieces behind the tensor before the fix, %ld now\n", before, after);
}

// ---- streaming GEMM for few activation rows -----------------------------------------------------
// A workgroup owns a run of consecutive rows and walks it in tiles of 16; wavefront w of eight or sixteen fetches
// the bytes of chunks [w cpw, (w + 1) cpw) of every row of a tile (its slice) with the matrix-core
// GEMM's piece arithmetic, the slice in the place of a chunk.
static void test_gemm_stream_pieces()
{
	long cases = 0;
	for (const Format& f : kFormats)
	{
		for (int geometry : { 801, 802, 804, 1601, 1602 }) // wavefronts x 100 + chunks per wavefront
		{
			const int waves = geometry / 100, cpw = geometry % 100;
			const int slice_bytes = cpw * f.chunk_bytes;
			const size_t row_bytes = static_cast<size_t>(waves) * slice_bytes;
			const int pieces = fm::gemm_weight_pieces(slice_bytes, f.aligned16);
			const int loads = (16 * pieces + 63) / 64;
			for (int n : { 1, 15, 16, 17, 56, 57, 100, 300 })
			{
				for (int cus : { 256, 8, 1 })
				{
					const size_t bytes = static_cast<size_t>(n) * row_bytes;
					std::vector<uintptr_t> bases;
					for (int mis = 0; mis < 16; mis += f.base_align)
					{
						bases.push_back(64 * kPage + mis);
					}
					const uintptr_t ends_on_page = 4096 * kPage - bytes;
					if (ends_on_page % f.base_align == 0)
					{
						bases.push_back(ends_on_page);
					}
					int rows = (n + cus - 1) / cus;
					rows = (rows + 3) / 4 * 4;
					const int blocks = (n + rows - 1) / rows;
					for (uintptr_t base : bases)
					{
						const uintptr_t end = base + bytes;
						std::vector<int> stored(n, 0);
						for (int block = 0; block < blocks; ++block)
						{
							const int row0 = block * rows;
							const int block_rows = rows < n - row0 ? rows : n - row0;
							CHECK(block_rows > 0, "%s n %d: empty workgroup %d", f.name, n, block);
							const int last_row = row0 + block_rows - 1;
							for (int t = 0; t < (block_rows + 15) / 16; ++t)
							{
								for (int wave = 0; wave < waves; ++wave)
								{
									std::vector<uintptr_t> slot(static_cast<size_t>(loads) * 64, 0); // by 16-byte piece of the slot
									for (int i = 0; i < loads; ++i)
									{
										for (int lane = 0; lane < 64; ++lane)
										{
											const fm::GemmWeightRequest rq = fm::gemm_weight_request(i, lane, 1, pieces);
											if (!(64 * (i + 1) <= 16 * pieces || rq.issued))
											{
												continue;
											}
											const int row = fm::gemm_weight_row(row0 + 16 * t, rq.row, last_row + 1);
											CHECK(row >= row0 && row <= last_row, "%s: row %d outside the run", f.name, row);
											const uintptr_t row_start = base + static_cast<size_t>(row) * row_bytes;
											const uintptr_t from = fm::gemm_weight_piece(row_start, wave, slice_bytes, f.aligned16, rq.offset);
											CHECK(from % 16 == 0, "%s: piece not aligned", f.name);
											CHECK(from < end && from + 16 > base, "%s cpw %d n %d base %#zx: piece outside the tensor", f.name, cpw,
											      n, static_cast<size_t>(base));
											slot[64 * i + lane] = from;
										}
									}
									for (int r = 0; r < 16; ++r)
									{
										const int row = fm::gemm_weight_row(row0 + 16 * t, r, last_row + 1);
										const uintptr_t row_start = base + static_cast<size_t>(row) * row_bytes;
										const uintptr_t slice = row_start + static_cast<size_t>(wave) * slice_bytes;
										const int mis = fm::gemm_weight_misalignment(row_start, wave, slice_bytes, f.aligned16);
										for (int b = 0; b < slice_bytes; ++b)
										{
											const int at = r * 16 * pieces + mis + b;
											const uintptr_t from = slot[at >> 4];
											CHECK(from != 0 && from + (at & 15) == slice + b, "%s cpw %d n %d row %d byte %d", f.name,
											      cpw, n, r, b);
										}
										if (wave == 0 && row0 + 16 * t + r <= last_row)
										{
											++stored[row0 + 16 * t + r];
										}
									}
								}
							}
						}
						for (int r = 0; r < n; ++r)
						{
							CHECK(stored[r] == 1, "%s n %d: row %d stored %d times", f.name, n, r, stored[r]);
						}
						++cases;
					}
				}
			}
		}
	}
	std::printf("streaming gemm: %ld launches walked\n", cases);
}

// ---- streaming GEMV ------------------------------------------------------------------------------
static void test_stream_rows_and_pieces()
{
	long cases = 0;
	for (const Format& f : kFormats)
	{
		for (int k : { 256, 512, 1024, 4096, 4352, 8192, 11008, 12288, 14336, 28672, 32768 })
		{
			const uint32_t row_bytes = static_cast<uint32_t>(k / 256 * f.chunk_bytes);
			const int slices = (k + 4095) / 4096;
			if (slices > 8 || row_bytes % 16 != 0)
			{
				continue; // the launcher sends such a shape to the register kernel
			}
			// three-slice rows also run with twelve wavefronts (four groups)
			for (int groups : { 8 / slices, slices == 3 ? 4 : 0 })
			{
			if (groups == 0 || k > 64 * slices * groups * 4 * 8)
			{
				continue; // more than eight 128-bit activation loads per thread: register kernel as well
			}
			const int loads = (f.stream_slice + 1023) / 1024;
			for (int whole = 0; whole < 2; ++whole)
			{
				if (whole && k != 4096)
				{
					continue; // the whole-slice instance exists for K = 4096 only
				}
				std::vector<int> covered(row_bytes, 0);
				for (int s = 0; s < slices; ++s)
				{
					const uint32_t slice_off = static_cast<uint32_t>(s) * f.stream_slice;
					CHECK(slice_off < row_bytes, "%s k %d slice %d starts behind the row", f.name, k, s);
					const uint32_t len = fm::stream_slice_len(whole != 0, f.stream_slice, row_bytes, slice_off);
					CHECK(len >= 16 && len % 16 == 0 && slice_off + len <= row_bytes, "%s k %d slice %d len %u", f.name, k, s, len);
					for (int i = 0; i < loads; ++i)
					{
						for (int lane = 0; lane < 64; ++lane)
						{
							const fm::StreamPiece p = fm::stream_row_piece(i, lane, len, whole != 0);
							if (!p.issued)
							{
								continue;
							}
							CHECK(p.offset + 16 <= len, "%s k %d: piece %u + 16 > %u", f.name, k, p.offset, len);
							if (1024u * i + 16u * lane < len) // a consumed piece sits where the unit reads it
							{
								CHECK(p.offset == 1024u * i + 16u * lane, "%s k %d: piece misplaced", f.name, k);
								for (int b = 0; b < 16; ++b)
								{
									++covered[slice_off + p.offset + b];
								}
							}
						}
					}
				}
				for (uint32_t b = 0; b < row_bytes; ++b)
				{
					CHECK(covered[b] == 1, "%s k %d: row byte %u fetched %d times", f.name, k, b, covered[b]);
				}
				// activations: 128-bit loads, clamped so that every thread issues every one of them
				const int threads = 64 * slices * groups;
				const int per_thread = (k / 4 + threads - 1) / threads;
				const int xp = per_thread <= 2 ? 2 : (per_thread <= 4 ? 4 : 8);
				CHECK(per_thread <= xp, "%s k %d: %d loads per thread", f.name, k, per_thread);
				std::vector<int> x_seen(k, 0);
				for (int tid = 0; tid < threads; ++tid)
				{
					for (int j = 0; j < xp; ++j)
					{
						const int at = fm::stream_x_index(tid, j, threads, k);
						CHECK(at >= 0 && at + 4 <= k && at % 4 == 0, "%s k %d: x load at %d", f.name, k, at);
						if ((tid + j * threads) * 4 < k)
						{
							for (int e = 0; e < 4; ++e)
							{
								++x_seen[at + e];
							}
						}
					}
				}
				for (int e = 0; e < k; ++e)
				{
					CHECK(x_seen[e] == 1, "%s k %d: activation %d staged %d times", f.name, k, e, x_seen[e]);
				}
				// rows: one round of workgroups, every row walked by exactly one wavefront group
				for (int n_total : { 1, 2, 7, 100, 4096, 11008, 32000, 128256 })
				{
					for (int max_blocks : { 256, 64, 1 })
					{
						int rows = (n_total + max_blocks * groups - 1) / (max_blocks * groups);
						rows = rows < 1 ? 1 : (rows > 64 ? 64 : rows);
						// every pair of runs the launcher may choose: the first half of the groups walk `run`
						// rows, the second half `run - diff` (an even number of groups, both at least one row)
						for (int diff = 0; diff < rows && (diff == 0 || groups % 2 == 0); ++diff)
						{
							const int block_rows = fm::stream_block_rows(groups, rows, diff);
							const int blocks = (n_total + block_rows - 1) / block_rows;
							std::vector<int> walked(n_total, 0);
							for (int block = 0; block < blocks; ++block)
							{
								int expect = block * block_rows; // the groups' runs follow each other
								for (int g = 0; g < groups; ++g)
								{
									const fm::StreamRows r = fm::stream_group_rows(block, g, groups, rows, diff, n_total);
									const int run = fm::stream_group_run(g, groups, rows, diff);
									CHECK(r.row0 == expect && run >= 1 && run <= rows, "run %d of group %d starts at %d, expected %d", run, g,
									      r.row0, expect);
									CHECK(r.count >= 0 && r.count <= run, "count %d", r.count);
									expect += run;
									for (int q = 0; q < r.count; ++q)
									{
										CHECK(r.row0 + q < n_total, "%s k %d n %d: row %d", f.name, k, n_total, r.row0 + q);
										if (r.row0 + q < n_total)
										{
											++walked[r.row0 + q];
										}
									}
								}
								CHECK(expect == (block + 1) * block_rows, "a workgroup's runs cover %d rows", expect - block * block_rows);
							}
							for (int r = 0; r < n_total; ++r)
							{
								CHECK(walked[r] == 1, "%s k %d n %d diff %d: row %d walked %d times", f.name, k, n_total, diff, r, walked[r]);
							}
							++cases;
						}
					}
				}
			}
			}
		}
	}
	std::printf("streaming gemv: %ld launch geometries walked\n", cases);
}

// ---- tiled prompt attention -----------------------------------------------------------------------
static void test_attention_tiles()
{
	constexpr int q_tile = 64, key_tile = 64;
	long cases = 0;
	for (int m : { 16, 17, 63, 64, 65, 100, 512, 2048 })
	{
		for (int past : { 0, 1, 5, 63, 64, 1000 })
		{
			const int cache_rows = past + m; // rows the cache is guaranteed to hold
			for (int tile = 0; tile < (m + q_tile - 1) / q_tile; ++tile)
			{
				const int kv_len = fm::attn_tile_kv_len(past, tile * q_tile, q_tile, m);
				CHECK(kv_len >= 1 && kv_len <= cache_rows, "m %d past %d tile %d: kv_len %d", m, past, tile, kv_len);
				// the last row of the tile sees keys 0 .. past + row
				const int last_row = (tile * q_tile + q_tile < m ? tile * q_tile + q_tile : m) - 1;
				CHECK(kv_len == past + last_row + 1, "kv_len %d", kv_len);
				const int n_key_tiles = (kv_len + key_tile - 1) / key_tile;
				std::vector<int> seen(kv_len, 0);
				for (int kt = 0; kt < n_key_tiles + 2; ++kt) // the kernel re-reads the last tile past the end
				{
					const int t = fm::imin(kt, n_key_tiles - 1);
					for (int idx = 0; idx < key_tile; ++idx)
					{
						const int key = fm::attn_tile_key(t, key_tile, idx, kv_len);
						CHECK(key >= 0 && key < kv_len, "m %d past %d: key %d of %d", m, past, key, kv_len);
						if (kt < n_key_tiles && t * key_tile + idx < kv_len)
						{
							++seen[key];
						}
					}
				}
				for (int key = 0; key < kv_len; ++key)
				{
					CHECK(seen[key] == 1, "m %d past %d: key %d staged %d times", m, past, key, seen[key]);
				}
				++cases;
			}
		}
	}
	std::printf("attention tiles: %ld query tiles walked\n", cases);
}

// ---- decoder-block kernel: rows dealt out per team, column segments of the output projection ----
static void test_team_rows_and_segments()
{
	long cases = 0;
	// first phase: every row of every matrix is walked exactly once over the eight teams
	for (int n0 : { 4096, 2048, 1024 })
	{
		for (int n1 : { 4096, 1024, 512, 0 })
		{
			const int n2 = n1;
			std::vector<int> seen0(n0, 0), seen1(n1, 0), seen2(n2, 0);
			const int per_team = (n0 >> 3) + (n1 >> 3) + (n2 >> 3);
			for (int team = 0; team < 8; ++team)
			{
				for (int v = 0; v < per_team; ++v)
				{
					const fm::TeamRow r = fm::team_row(v, team, n0, n1, n2);
					std::vector<int>& seen = r.m == 0 ? seen0 : (r.m == 1 ? seen1 : seen2);
					CHECK(r.m >= 0 && r.m <= 2 && r.local >= 0 && r.local < static_cast<int>(seen.size()),
					      "team %d row %d -> matrix %d row %d", team, v, r.m, r.local);
					if (r.local >= 0 && r.local < static_cast<int>(seen.size()))
					{
						++seen[r.local];
					}
					++cases;
				}
			}
			for (const std::vector<int>* seen : { &seen0, &seen1, &seen2 })
			{
				for (size_t i = 0; i < seen->size(); ++i)
				{
					CHECK((*seen)[i] == 1, "n %d %d: row %zu walked %d times", n0, n1, i, (*seen)[i]);
				}
			}
		}
	}
	// third phase: 4096 x 4096 output projection, team t owns 512 columns (two 256-element chunks) of
	// every row; a wavefront's fetch holds the segments of eight consecutive rows and must look like a
	// 4096-wide slice of a row made of those segments
	for (const Format& f : kFormats)
	{
		const int seg_bytes = 2 * f.chunk_bytes;
		if (seg_bytes % 16 != 0)
		{
			continue; // the launcher sends such a format down the separate launches
		}
		const int n = 4096, row_bytes = 16 * f.chunk_bytes, seg_pieces = seg_bytes / 16, rows_per_fetch = 8;
		CHECK(seg_pieces * rows_per_fetch * 16 == f.stream_slice, "%s: eight segments are not one slice", f.name);
		const int loads = (f.stream_slice + 1023) / 1024;
		const uintptr_t base = 7 * kPage; // page-exact tensor: 4096 rows x 16 chunks
		const uintptr_t end = base + static_cast<size_t>(n) * row_bytes;
		std::vector<unsigned char> covered(static_cast<size_t>(n) * row_bytes, 0);
		for (int block = 0; block < 256; ++block)
		{
			const int team = block & 7, place = block >> 3;
			for (int wave = 0; wave < 8; ++wave)
			{
				for (int fetch = 0; fetch < 2; ++fetch)
				{
					const int row0 = place * 128 + (wave * 2 + fetch) * rows_per_fetch;
					std::map<int, uintptr_t> slot;
					for (int i = 0; i < loads; ++i)
					{
						for (int lane = 0; lane < 64; ++lane)
						{
							const fm::SegmentPiece sp = fm::segment_piece(i, lane, seg_pieces, rows_per_fetch);
							if (!sp.issued)
							{
								continue;
							}
							CHECK(sp.row >= 0 && sp.row < rows_per_fetch && sp.offset + 16 <= static_cast<uint32_t>(seg_bytes),
							      "%s: piece row %d offset %u", f.name, sp.row, sp.offset);
							const uintptr_t from = base + static_cast<size_t>(row0 + sp.row) * row_bytes +
							                       static_cast<size_t>(team) * seg_bytes + sp.offset;
							CHECK(from % 16 == 0 && from >= base && from + 16 <= end, "%s: piece at %#zx outside the tensor", f.name,
							      static_cast<size_t>(from));
							slot[1024 * i + 16 * lane] = from;
							if (from >= base && from + 16 <= end)
							{
								for (int b = 0; b < 16; ++b)
								{
									++covered[from - base + b];
								}
							}
							++cases;
						}
					}
					// the slot, read as a slice: byte b of row r's segment sits at r * seg_bytes + b
					for (int r = 0; r < rows_per_fetch; ++r)
					{
						for (int b = 0; b < seg_bytes; b += 16)
						{
							const auto it = slot.find(r * seg_bytes + b);
							const uintptr_t want = base + static_cast<size_t>(row0 + r) * row_bytes + static_cast<size_t>(team) * seg_bytes + b;
							CHECK(it != slot.end() && it->second == want, "%s: slot byte %d of row %d", f.name, b, r);
						}
					}
				}
			}
		}
		for (size_t i = 0; i < covered.size(); ++i)
		{
			if (covered[i] != 1)
			{
				CHECK(false, "%s: byte %zu of the projection fetched %d times", f.name, i, covered[i]);
				break;
			}
		}
	}
	std::printf("team rows and column segments: %ld rows and pieces walked\n", cases);
}

// The K ranges of the tiled GEMM: whatever the split, the ranges tile [0, chunks) in order; and
// whenever the launcher's condition for several groups per workgroup holds, the groups of every
// workgroup walk equally many chunks (they pass one set of barriers per chunk: an unequal walk would
// leave a group waiting at a barrier the other never reaches).
static void test_gemm_chunk_ranges()
{
	using namespace litenn_hip::fetch;
	long walked = 0;
	for (int chunks = 1; chunks <= 96; ++chunks)
	{
		for (int grid_z = 1; grid_z <= 4; grid_z *= 2)
		{
			for (int groups = 1; groups <= 2; ++groups)
			{
				const int parts = grid_z * groups;
				int expect_begin = 0;
				for (int part = 0; part < parts; ++part)
				{
					const ChunkRange r = gemm_chunk_range(part, parts, chunks);
					CHECK(r.begin == expect_begin && r.end >= r.begin && r.end <= chunks, "chunks %d parts %d part %d: [%d, %d)",
					      chunks, parts, part, r.begin, r.end);
					expect_begin = r.end;
					walked += r.end - r.begin;
				}
				CHECK(expect_begin == chunks, "chunks %d parts %d: ranges end at %d", chunks, parts, expect_begin);
				if (groups > 1 && gemm_ranges_equal(chunks, parts))
				{
					for (int z = 0; z < grid_z; ++z)
					{
						const ChunkRange g0 = gemm_chunk_range(z * groups, parts, chunks);
						const ChunkRange g1 = gemm_chunk_range(z * groups + 1, parts, chunks);
						CHECK(g0.end - g0.begin == g1.end - g1.begin && g0.end > g0.begin,
						      "chunks %d grid z %d: groups of workgroup %d walk %d and %d chunks", chunks, grid_z, z,
						      g0.end - g0.begin, g1.end - g1.begin);
					}
				}
			}
		}
	}
	// an odd chunk count must not pass the launcher's condition
	CHECK(!gemm_ranges_equal(43, 2) && !gemm_ranges_equal(6, 4) && gemm_ranges_equal(16, 4) && !gemm_ranges_equal(1, 2),
	      "the condition for several groups per workgroup");
	std::printf("tiled GEMM K ranges: %ld chunks walked\n", walked);
}

// Products over bfloat16 weights: whatever the ranges of K and the groups of wavefronts, every tile of K is
// multiplied once, the groups of a workgroup make equally many rounds, and only tiles that are there are requested
// (up to a ring's buffers past the last round).
static void test_dense_walks()
{
	using namespace litenn_hip::fetch;
	long walked = 0;
	for (int all = 1; all <= 300; ++all)
	{
		for (int ranges = 1; ranges <= 4; ++ranges)
		{
			for (int groups = 1; groups <= 3; ++groups)
			{
				std::vector<int> times(all, 0);
				for (int range = 0; range < ranges; ++range)
				{
					for (int group = 0; group < groups; ++group)
					{
						const DenseWalk w = dense_walk(all, ranges, groups, range, group);
						CHECK(w.rounds == dense_walk(all, ranges, groups, range, 0).rounds, "%d tiles, %d ranges of %d groups", all, ranges, groups);
						for (int round = 0; round < w.rounds + kDenseMaxBuffers; ++round)
						{
							const int tile = w.tile(round);
							CHECK(tile >= 0 && tile < all, "%d tiles, %d ranges of %d groups: tile %d", all, ranges, groups, tile);
							if (round < w.rounds && w.multiplies(round))
							{
								++times[tile];
								++walked;
							}
						}
					}
				}
				for (int tile = 0; tile < all; ++tile)
				{
					CHECK(times[tile] == 1, "%d tiles, %d ranges of %d groups: tile %d %d times", all, ranges, groups, tile, times[tile]);
				}
			}
		}
	}
	std::printf("bfloat16 products: %ld tiles of K walked\n", walked);
}

// The form a product of bfloat16 operands takes against what all of them took (us on the card, weights from HBM, forms in
// the order of DenseForm, 0 not measured): never 5 % more than the fastest.
static void test_dense_forms()
{
	using namespace litenn_hip::fetch;
	struct Measured
	{
		int n, k, ranges, m;
		double us[kDenseForms];
	};
	const Measured measured[] = {
		{ 4096, 14336, 1, 639, { 313.1, 195.0, 201.1, 150.6, 160.5, 191.6, 132.7, 162.2, 168.8, 162.3, 195.9, 254.4 } },
		{ 4096, 14336, 3, 178, { 117.1, 72.4, 77.8, 60.2, 58.3, 68.3, 45.8, 55.3, 65.4, 63.8, 73.7, 88.5 } },
		{ 4096, 14336, 4, 33, { 79.5, 52.2, 55.6, 42.5, 41.9, 51.9, 34.5, 28.5, 32.0, 23.3, 28.5, 34.2 } },
		{ 4096, 4096, 4, 96, { 31.5, 22.2, 21.0, 17.6, 19.1, 19.6, 16.0, 13.6, 14.1, 14.4, 17.6, 21.7 } },
		{ 28672, 4096, 1, 178, { 105.7, 69.6, 75.2, 61.7, 98.6, 75.4, 83.2, 90.2, 87.8, 102.1, 129.7, 166.0 } },
		{ 28672, 4096, 1, 2048, { 450.6, 467.7, 467.8, 523.4, 529.0, 490.6, 573.0, 650.3, 669.8, 0, 0, 0 } },
		{ 13888, 4096, 1, 17, { 89.6, 57.6, 62.0, 46.8, 45.9, 58.5, 38.3, 32.2, 35.0, 26.8, 25.5, 25.6 } },
		{ 6160, 2048, 1, 320, { 58.4, 35.3, 37.2, 29.1, 29.6, 33.3, 24.0, 28.2, 21.4, 23.6, 30.3, 38.9 } },
		{ 6432, 2048, 1, 1280, { 62.4, 67.4, 46.1, 57.7, 59.4, 40.0, 51.8, 57.4, 57.7, 67.0, 84.5, 123.7 } },
		{ 11264, 2048, 1, 777, { 60.5, 66.6, 48.6, 56.7, 59.3, 68.7, 64.3, 63.2, 67.8, 75.8, 100.1, 140.9 } },
		{ 2048, 5632, 1, 777, { 131.8, 79.3, 83.3, 62.8, 63.7, 77.5, 49.8, 39.0, 42.3, 46.0, 61.6, 71.2 } },
		{ 2048, 5632, 2, 512, { 80.1, 48.4, 48.0, 37.8, 40.3, 44.0, 33.7, 26.2, 27.1, 29.6, 39.9, 51.1 } },
		{ 1024, 2816, 2, 48, { 34.6, 23.8, 24.2, 19.1, 19.6, 22.5, 16.3, 12.8, 15.0, 10.7, 8.9, 6.9 } },
	};
	for (const Measured& p : measured)
	{
		double least = p.us[0];
		for (double us : p.us)
		{
			least = us > 0.0 && us < least ? us : least;
		}
		const DenseForm form = dense_form(p.n, p.k / 64, p.m, p.ranges);
		CHECK(p.us[form] > 0.0 && p.us[form] <= 1.05 * least, "%d x %d x %d in %d ranges: form %d", p.m, p.n, p.k, p.ranges, static_cast<int>(form));
	}
	for (int m = 1; m <= 4096; m += 1 + m / 3) // any size has one
	{
		for (int n = 1; n <= 40000; n += 1 + n / 2)
		{
			for (int tiles : { 1, 2, 3, 7, 64, 300 })
			{
				const int form = dense_form(n, tiles, m, dense_ranges(n, tiles, m));
				CHECK(form >= 0 && form < kDenseForms, "%d x %d x %d tiles: form %d", m, n, tiles, form);
			}
		}
	}
}

// The ranges of K of a sublayer's last product, bfloat16 operands, against what it and the norm that adds its sums take in one
// to four of them (us on the card, weights from HBM, 0: fewer than 16 tiles of K each).
static void test_dense_ranges()
{
	using namespace litenn_hip::fetch;
	struct Measured
	{
		int n, k, m;
		double us[kDenseMaxRanges];
	};
	const Measured measured[] = {
		{ 4096, 14336, 33, { 40.0, 34.8, 34.9, 31.8 } }, { 4096, 14336, 100, { 49.5, 44.5, 46.8, 40.6 } }, { 4096, 14336, 178, { 70.4, 58.5, 54.8, 46.9 } },
		{ 4096, 14336, 300, { 93.6, 72.9, 68.3, 58.8 } }, { 4096, 14336, 400, { 95.6, 74.6, 81.7, 70.0 } }, { 4096, 14336, 500, { 104.8, 82.9, 85.3, 72.4 } },
		{ 4096, 14336, 639, { 141.9, 101.1, 91.4, 95.6 } }, { 4096, 14336, 777, { 129.2, 115.6, 116.9, 118.5 } }, { 4096, 14336, 900, { 131.6, 122.3, 119.6, 119.7 } },
		{ 4096, 14336, 1000, { 141.7, 122.1, 141.3, 124.2 } }, { 4096, 4096, 33, { 16.4, 18.9, 18.8, 18.1 } }, { 4096, 4096, 100, { 19.3, 21.9, 23.0, 21.0 } },
		{ 4096, 4096, 178, { 25.3, 27.1, 27.6, 25.6 } }, { 4096, 4096, 300, { 33.3, 32.9, 33.0, 30.6 } }, { 4096, 4096, 400, { 34.4, 34.2, 38.8, 34.9 } },
		{ 4096, 4096, 500, { 37.3, 35.7, 39.7, 37.2 } }, { 4096, 4096, 639, { 48.0, 43.0, 41.5, 43.6 } }, { 4096, 4096, 777, { 48.4, 49.6, 50.6, 59.2 } },
		{ 4096, 4096, 900, { 49.3, 50.5, 52.1, 60.5 } }, { 4096, 4096, 1000, { 50.6, 51.0, 67.3, 63.8 } }, { 2048, 5632, 33, { 18.8, 15.4, 15.0, 13.8 } },
		{ 2048, 5632, 100, { 19.2, 17.8, 18.0, 16.4 } }, { 2048, 5632, 178, { 24.4, 22.2, 22.5, 19.9 } }, { 2048, 5632, 300, { 30.4, 27.7, 24.8, 25.1 } },
		{ 2048, 5632, 400, { 29.2, 28.4, 28.8, 26.1 } }, { 2048, 5632, 500, { 32.1, 30.4, 31.0, 27.7 } }, { 2048, 5632, 640, { 45.0, 38.8, 32.2, 32.4 } },
		{ 2048, 5632, 777, { 43.0, 37.2, 37.3, 38.4 } }, { 2048, 5632, 900, { 43.3, 38.2, 38.0, 39.9 } }, { 2048, 5632, 1000, { 46.3, 40.4, 44.8, 40.6 } },
		{ 2048, 4096, 33, { 15.4, 13.7, 13.3, 12.5 } }, { 2048, 4096, 100, { 15.8, 15.4, 15.7, 14.7 } }, { 2048, 4096, 200, { 18.3, 18.1, 19.5, 17.6 } },
		{ 2048, 4096, 400, { 23.3, 23.8, 24.5, 22.8 } }, { 2048, 4096, 640, { 34.8, 31.0, 27.1, 28.1 } }, { 2048, 4096, 777, { 34.0, 31.5, 31.9, 32.6 } },
		{ 2048, 4096, 1000, { 36.6, 33.2, 37.9, 35.9 } }, { 2048, 2048, 33, { 10.9, 11.3, 0, 0 } }, { 2048, 2048, 100, { 11.2, 12.4, 0, 0 } },
		{ 2048, 2048, 200, { 12.9, 14.3, 0, 0 } }, { 2048, 2048, 400, { 16.0, 18.5, 0, 0 } }, { 2048, 2048, 640, { 22.2, 22.4, 0, 0 } },
		{ 2048, 2048, 777, { 21.6, 23.3, 0, 0 } }, { 2048, 2048, 1000, { 23.6, 24.4, 0, 0 } }, { 1024, 2816, 33, { 12.2, 10.6, 0, 0 } },
		{ 1024, 2816, 100, { 12.3, 10.9, 0, 0 } }, { 1024, 2816, 200, { 12.6, 12.1, 0, 0 } }, { 1024, 2816, 400, { 14.8, 14.4, 0, 0 } },
		{ 1024, 2816, 640, { 17.2, 17.2, 0, 0 } }, { 1024, 2816, 777, { 17.6, 17.9, 0, 0 } }, { 1024, 2816, 1000, { 18.6, 19.1, 0, 0 } },
	};
	double more = 0.0;
	int count = 0;
	for (const Measured& p : measured)
	{
		double least = p.us[0];
		for (double us : p.us)
		{
			least = us > 0.0 && us < least ? us : least;
		}
		const int ranges = dense_ranges(p.n, p.k / 64, p.m);
		const double chosen = p.us[ranges - 1];
		CHECK(chosen > 0.0 && chosen <= least + 1.8, "%d x %d x %d: %d ranges", p.m, p.n, p.k, ranges);
		const double by_tiles = p.us[dense_f32_ranges(p.n, p.k / 64, p.m) - 1]; // (enough for two workgroups a CU)
		CHECK(chosen <= by_tiles + 0.5, "%d x %d x %d: %d ranges %.1f us, by the number of tiles %.1f", p.m, p.n, p.k, ranges, chosen, by_tiles);
		more += chosen / least - 1.0;
		++count;
	}
	CHECK(more <= 0.01 * count, "ranges of K: %.3f of the fastest too much in the mean", more / count);
}

// The sums of a sublayer's last product lie in a buffer made for the longest pass so far: any shorter one's, in
// its ranges of K, must fit (widths and K of layered decoders, and small odd ones).
static void test_dense_sum_rows()
{
	using namespace litenn_hip::fetch;
	long passes = 0, ranged = 0;
	for (int cap = 1; cap <= 4300; cap += cap < 1000 || cap > 1030 ? 37 : 1)
	{
		const size_t room = dense_sum_rows(cap);
		for (int rows = 1; rows <= cap; ++rows)
		{
			for (int n : { 1, 50, 88, 640, 1024, 2048, 4096 })
			{
				for (int k : { 64, 1000, 2048, 2816, 5632, 14336 })
				{
					for (const int ranges : { dense_ranges(n, (k + 63) / 64, rows), dense_f32_ranges(n, (k + 63) / 64, rows) })
					{
						CHECK(ranges >= 1 && ranges <= kDenseMaxRanges && ranges <= (k + 63) / 64 && static_cast<size_t>(ranges) * rows <= room,
						      "%d ranges of %d rows (%d x %d) in room for %zu, made for passes of %d", ranges, rows, n, k, room, cap);
						++passes;
						ranged += ranges > 1;
					}
				}
			}
		}
	}
	std::printf("sums in ranges of K: %ld of %ld passes\n", ranged, passes);
}

// Attention of many rows over Float32 keys: the keys that a block of rows sees, and the form taken against what both take (us on
// the card): never 5 % more than the faster one, whether or not rows and keys are equally many.
static void test_rows_forms()
{
	using namespace litenn_hip::fetch;
	for (const RowsSeen a : { RowsSeen{ 70, 70, true, 0, 1ll << 62 }, RowsSeen{ 70, 71, true, 1, 1ll << 62 }, RowsSeen{ 33, 400, true, 367, 40 },
	                          RowsSeen{ 40, 300, false, 0, 1ll << 62 }, RowsSeen{ 40, 90, true, 100, 1ll << 62 }, RowsSeen{ 1, 1, true, 0, 1 } })
	{
		for (int first = 0; first < a.rows; first += 32)
		{
			int low = a.keys, high = -1;
			for (int i = first; i < a.rows && i < first + 32; ++i)
			{
				for (int key = 0; key < a.keys; ++key)
				{
					if (key > a.q_at + i - a.window && (!a.causal || key <= a.q_at + i))
					{
						low = imin(low, key);
						high = imax(high, key);
					}
				}
			}
			CHECK(a.tiles(first, 32) == (high - low + 32) / 32, "%d rows on %d keys, rows from %d: %d tiles", a.rows, a.keys, first, a.tiles(first, 32));
		}
	}
	struct Measured
	{
		int rows, keys, heads, dim;
		bool causal;
		double alone, pairs;
	};
	const Measured measured[] = {
		{ 300, 300, 32, 128, true, 28.9, 30.6 }, { 300, 301, 32, 128, true, 34.8, 31.8 }, { 300, 320, 32, 128, true, 34.6, 31.5 },
		{ 300, 350, 32, 128, true, 34.9, 35.4 }, { 300, 400, 32, 128, true, 41.3, 39.9 }, { 300, 500, 32, 128, true, 52.1, 44.8 },
		{ 300, 1000, 32, 128, true, 90.9, 79.2 }, { 512, 512, 32, 128, true, 45.7, 44.6 }, { 512, 513, 32, 128, true, 52.0, 49.7 },
		{ 512, 700, 32, 128, true, 63.4, 58.5 }, { 512, 1024, 32, 128, true, 89.6, 79.9 }, { 700, 700, 16, 128, true, 43.3, 56.9 },
		{ 700, 701, 16, 128, true, 46.9, 57.9 }, { 700, 1000, 16, 128, true, 69.5, 79.6 }, { 700, 1500, 16, 128, true, 111.5, 114.3 },
		{ 1024, 1024, 16, 128, true, 67.3, 79.2 }, { 1024, 1500, 16, 128, true, 112.5, 115.7 }, { 400, 400, 24, 128, true, 33.9, 38.4 },
		{ 400, 500, 24, 128, true, 46.5, 44.8 }, { 1200, 1200, 8, 128, true, 65.0, 91.2 }, { 1200, 2400, 8, 128, true, 145.8, 174.7 },
		{ 2000, 2000, 8, 128, true, 111.4, 148.1 }, { 2000, 3000, 8, 128, true, 201.6, 217.9 }, { 3000, 3000, 4, 128, true, 142.3, 213.3 },
		{ 3000, 4000, 4, 128, true, 206.4, 286.0 }, { 300, 300, 32, 128, false, 51.3, 31.4 }, { 512, 512, 24, 128, false, 61.3, 44.5 },
		{ 700, 700, 16, 128, false, 85.0, 57.9 }, { 700, 128, 16, 128, false, 28.1, 18.0 }, { 1100, 2000, 8, 128, false, 195.7, 149.9 },
		{ 1100, 1100, 8, 128, false, 118.3, 88.1 }, { 64, 300, 200, 128, false, 55.1, 32.6 }, { 64, 300, 200, 128, true, 54.9, 32.7 },
		{ 30, 300, 300, 128, true, 54.9, 59.2 }, { 200, 1000, 32, 128, true, 53.9, 78.6 }, { 512, 512, 16, 128, true, 32.0, 43.7 },
		{ 1000, 1000, 32, 128, true, 132.7, 92.6 }, { 600, 600, 32, 128, true, 63.8, 52.8 }, { 512, 512, 32, 64, true, 26.5, 29.6 },
		{ 512, 700, 32, 64, true, 37.1, 38.7 }, { 700, 700, 16, 64, true, 25.2, 37.8 }, { 700, 1000, 16, 64, true, 40.2, 53.1 },
		{ 300, 300, 32, 64, true, 17.0, 20.3 }, { 300, 1000, 32, 64, true, 52.6, 53.1 }, { 300, 400, 32, 64, true, 24.2, 26.6 },
		{ 1024, 1024, 16, 64, true, 39.4, 52.7 }, { 1024, 1500, 16, 64, true, 65.9, 76.5 }, { 2000, 3000, 8, 64, true, 114.9, 143.1 },
		{ 512, 1024, 32, 64, true, 52.4, 53.1 },
	};
	for (const Measured& p : measured)
	{
		const bool alone = rows_float_alone({ p.rows, p.keys, p.causal, p.causal ? p.keys - p.rows : 0, 1ll << 62 }, p.heads, p.dim);
		const double least = p.alone < p.pairs ? p.alone : p.pairs;
		CHECK((alone ? p.alone : p.pairs) <= 1.05 * least, "%d rows on %d keys, %d heads of %d, causal %d: alone %d", p.rows, p.keys, p.heads, p.dim, p.causal, alone);
	}
	for (int heads : { 1, 3, 8, 24, 255, 256, 257, 300, 512, 513 }) // any size has one
	{
		for (int rows = 1; rows <= 3000; rows += 1 + rows / 5)
		{
			for (bool causal : { false, true })
			{
				const RowsSeen a{ rows, rows + 7, causal, 7, 1ll << 62 };
				const long long groups = static_cast<long long>(heads) * ((rows + 31) / 32);
				CHECK(rows_float_alone(a, heads, 64) || groups > 256, "%d rows of %d heads", rows, heads);
				CHECK(groups > 512 || (rows_time(a, heads, 32, 4, { 98, 180, 55 }) > 98 && rows_time(a, heads, 64, 2, { 90, 160, 43 }) > 90), "%d rows of %d heads", rows, heads);
			}
		}
	}
}

// Attention with options, a key at a time or tiles, against what a call takes either way (us on the card, no soft cap): never 6 % more
// than the faster one.
static void test_options_forms()
{
	struct Measured
	{
		int rows, keys, heads, dim;
		bool f32;
		double row, tiles;
	};
	const Measured measured[] = {
		{ 1, 96, 32, 72, true, 8.7, 14.6 }, { 4, 128, 32, 72, true, 10.4, 14.8 }, { 12, 96, 32, 72, true, 9.1, 13.8 }, { 8, 300, 32, 72, true, 19.4, 25.8 },
		{ 8, 96, 128, 72, true, 13.6, 13.9 }, { 8, 128, 128, 72, true, 16.6, 13.9 }, { 12, 64, 128, 72, true, 15.0, 14.0 }, { 1, 160, 32, 80, true, 11.9, 20.1 },
		{ 4, 96, 32, 80, true, 8.8, 14.8 }, { 4, 200, 32, 80, true, 14.5, 20.5 }, { 2, 600, 32, 80, true, 34.1, 37.0 }, { 4, 1000, 32, 80, true, 54.3, 53.8 },
		{ 4, 300, 128, 80, true, 19.7, 26.4 }, { 4, 96, 128, 80, true, 9.4, 15.0 }, { 8, 64, 128, 80, true, 11.5, 13.9 }, { 8, 112, 128, 80, true, 16.6, 14.0 },
		{ 1, 112, 32, 96, true, 9.4, 14.6 }, { 2, 1000, 32, 96, true, 55.5, 53.4 }, { 8, 600, 32, 96, true, 33.5, 36.6 }, { 12, 200, 32, 96, true, 17.9, 19.7 },
		{ 12, 300, 32, 96, true, 24.3, 25.3 }, { 8, 64, 128, 96, true, 14.9, 13.7 }, { 4, 200, 128, 96, true, 21.7, 20.6 }, { 4, 400, 32, 104, true, 23.0, 31.9 },
		{ 2, 96, 128, 104, true, 8.9, 14.9 }, { 8, 128, 128, 104, true, 23.7, 13.9 }, { 16, 200, 32, 104, true, 19.5, 20.2 }, { 2, 64, 32, 72, false, 9.2, 10.8 },
		{ 4, 80, 32, 72, false, 10.5, 10.7 }, { 24, 64, 32, 72, false, 10.3, 10.1 }, { 8, 96, 32, 96, false, 12.5, 10.3 }, { 4, 80, 128, 104, false, 12.0, 10.8 },
		{ 12, 64, 128, 104, false, 21.7, 10.0 }, { 4, 64, 32, 64, true, 7.0, 9.1 }, { 4, 112, 32, 64, true, 9.2, 9.2 }, { 8, 96, 32, 64, true, 8.6, 8.8 },
		{ 24, 64, 32, 64, true, 9.0, 8.7 }, { 2, 200, 32, 64, true, 13.6, 12.3 }, { 2, 64, 32, 32, true, 7.2, 9.2 }, { 8, 128, 32, 32, true, 10.6, 8.9 },
		{ 2, 96, 32, 128, true, 14.9, 14.3 }, { 2, 64, 32, 128, true, 11.4, 14.3 }, { 8, 128, 32, 128, true, 18.6, 13.7 }, { 4, 112, 32, 120, true, 16.0, 15.0 },
		{ 2, 64, 32, 64, false, 8.7, 7.0 }, { 2, 64, 32, 128, false, 10.5, 9.8 }, { 8, 96, 32, 128, false, 13.9, 9.4 }, { 12, 64, 128, 64, false, 16.7, 6.4 },
	};
	for (const Measured& p : measured)
	{
		const bool tiles = litenn_hip::fetch::rows_options_tiles(p.rows, p.keys, p.heads, p.dim, p.f32);
		CHECK((tiles ? p.tiles : p.row) <= 1.06 * (p.row < p.tiles ? p.row : p.tiles), "%d rows on %d keys, %d heads of %d: tiles %d", p.rows, p.keys, p.heads, p.dim, tiles);
	}
	struct Window
	{
		int rows, keys, heads, dim, vdim;
		double row, tiles;
	};
	const Window windows[] = { // (10 %)
		{ 64, 66, 4, 128, 64, 11.3, 15.2 }, { 16, 80, 16, 128, 64, 11.9, 14.4 }, { 64, 80, 16, 128, 64, 14.0, 15.3 }, { 32, 80, 48, 128, 64, 19.7, 15.3 },
		{ 48, 80, 48, 128, 64, 25.6, 15.4 }, { 16, 66, 4, 80, 80, 13.1, 14.8 }, { 48, 66, 16, 80, 80, 13.6, 15.9 }, { 80, 80, 16, 80, 80, 16.3, 15.9 },
		{ 100, 80, 16, 80, 80, 18.2, 15.9 }, { 200, 66, 48, 80, 80, 61.3, 24.5 }, { 64, 66, 4, 128, 128, 14.3, 15.3 }, { 16, 80, 48, 128, 128, 25.2, 14.6 },
		{ 64, 84, 16, 128, 128, 18.0, 15.5 }, { 20, 66, 48, 64, 64, 10.4, 9.4 }, { 32, 66, 4, 64, 64, 9.4, 9.6 },
	};
	for (const Window& p : windows)
	{
		const bool tiles = litenn_hip::fetch::rows_window_tiles(p.rows, p.keys, p.heads, p.dim, p.vdim);
		const double least = p.row < p.tiles ? p.row : p.tiles;
		CHECK((tiles ? p.tiles : p.row) <= 1.1 * least, "window, %d rows on %d keys, %d heads of %d and %d: tiles %d", p.rows, p.keys, p.heads, p.dim, p.vdim, tiles);
	}
	// rows that are asked for alone go by the form that all would go by, with a block of 64 ahead of them at most
	for (int rows = 1; rows <= 900; ++rows)
	{
		for (int first = 0; first < rows; ++first)
		{
			for (int keys : { rows, rows < 65 ? rows : 65, rows < 90 ? rows : 90 })
			{
				for (int dim : { 64, 80, 128 })
				{
					const int from = litenn_hip::fetch::window_rows_from(rows, first, 64, keys, 8, dim, dim);
					const bool all = litenn_hip::fetch::rows_window_tiles(rows, keys, 8, dim, dim), some = litenn_hip::fetch::rows_window_tiles(rows - from, keys, 8, dim, dim);
					CHECK(from >= 0 && from <= first && first - from < 128 && from % 64 == 0, "%d of %d rows: from %d", rows - first, rows, from);
					CHECK(some == all || keys < 96, "%d of %d rows on %d keys: from %d", rows - first, rows, keys, from);
				}
			}
		}
	}
	CHECK(!litenn_hip::fetch::rows_window_tiles(15, 500, 16, 128, 128) && !litenn_hip::fetch::rows_window_tiles(500, 64, 16, 128, 128), "few rows or keys");
}

// Q6_K with Float32 operands, one tile of activations a wavefront or two, against what a call takes either way (us on the card,
// weights from HBM): up to 512 tiles never 5 % more than the faster one.
static void test_exact_forms()
{
	struct Measured
	{
		int n, k, m;
		double one, two;
	};
	const Measured measured[] = {
		{ 4096, 14336, 33, 50.7, 70.6 }, { 4096, 14336, 45, 50.7, 70.5 }, { 4096, 14336, 64, 51.3, 70.9 }, { 4096, 14336, 65, 81.1, 65.7 },
		{ 4096, 14336, 96, 81.7, 67.0 }, { 4096, 14336, 97, 82.3, 69.8 }, { 4096, 14336, 128, 83.4, 70.9 }, { 4096, 4096, 33, 24.8, 30.1 },
		{ 4096, 4096, 64, 25.0, 30.6 }, { 4096, 4096, 96, 33.4, 31.6 }, { 4096, 4096, 128, 34.1, 32.4 }, { 8192, 4096, 33, 33.8, 31.3 },
		{ 8192, 4096, 64, 34.2, 32.3 }, { 1024, 4096, 64, 23.8, 27.9 }, { 1024, 4096, 200, 25.5, 31.6 }, { 1024, 4096, 300, 34.1, 32.8 },
		{ 1024, 4096, 512, 37.6, 35.5 }, { 2048, 5632, 64, 28.1, 36.2 }, { 2048, 5632, 128, 30.1, 38.1 }, { 2048, 5632, 200, 42.8, 38.6 },
		{ 2720, 14336, 65, 49.7, 64.7 }, { 2720, 14336, 96, 50.0, 64.7 }, { 4128, 4096, 33, 32.2, 30.4 }, { 4128, 4096, 64, 32.5, 30.6 },
		{ 4128, 14336, 33, 78.1, 70.3 }, { 4128, 14336, 64, 78.5, 70.8 }, { 7000, 4096, 33, 34.2, 31.3 }, { 7000, 4096, 64, 34.4, 32.2 },
		{ 512, 2048, 600, 28.4, 27.9 }, { 512, 2048, 1000, 35.6, 31.7 }, { 1024, 11008, 270, 63.9, 58.0 }, { 1024, 11008, 400, 78.5, 62.0 },
		{ 2100, 4096, 128, 31.6, 30.6 }, { 2100, 4096, 150, 32.3, 31.5 }, { 2100, 4096, 200, 33.5, 50.4 },
	};
	for (const Measured& p : measured)
	{
		const bool two = litenn_hip::fetch::exact_two_tiles((p.n + 31) / 32, (p.m + 31) / 32);
		CHECK((two ? p.two : p.one) <= 1.05 * (p.one < p.two ? p.one : p.two), "%d x %d x %d: two tiles %d", p.m, p.n, p.k, two);
	}
	CHECK(!litenn_hip::fetch::exact_two_tiles(4000, 1) && litenn_hip::fetch::exact_two_tiles(448, 3), "one tile, and many");
}

// Whether K goes in ranges, against what a call takes by the forms without them and with them (us on the card, weights from HBM):
// never 3 % more than the faster one.
static void test_exact_ranges()
{
	struct Measured
	{
		bool by_step; // Q6_K, else Q4_K or Q5_K
		int n, k, m;
		double without, ranged;
	};
	const Measured measured[] = {
		{ true, 32800, 4096, 9, 72.5, 91.8 }, { true, 32800, 4096, 16, 72.5, 92.6 }, { true, 32800, 4096, 32, 74.8, 97.8 }, { true, 128256, 4096, 9, 211.5, 225.8 },
		{ true, 128256, 4096, 16, 214.4, 232.6 }, { true, 128256, 4096, 32, 221.1, 253.9 }, { true, 128256, 4096, 64, 373.3, 275.7 },
		{ false, 4096, 4096, 300, 55.7, 50.8 }, { false, 4096, 14336, 33, 39.1, 37.9 }, { false, 4096, 14336, 64, 40.3, 41.4 }, { false, 4096, 14336, 65, 60.2, 52.2 }, { false, 4096, 14336, 300, 159.7, 115.4 },
		{ false, 14336, 4096, 64, 40.3, 39.6 }, { false, 4096, 14336, 33, 40.6, 39.8 }, { false, 4096, 14336, 64, 41.7, 44.3 }, { true, 4096, 4096, 300, 73.4, 58.7 }, { true, 14336, 4096, 33, 47.5, 44.5 },
		{ false, 2048, 14336, 128, 41.9, 42.8 }, { false, 3072, 11008, 160, 54.1, 55.4 }, { false, 3072, 14336, 160, 66.1, 62.2 }, { false, 5120, 14336, 64, 59.7, 46.3 }, { false, 5120, 14336, 90, 63.0, 66.0 },
		{ false, 5120, 14336, 128, 89.1, 68.6 }, { false, 6144, 7168, 160, 64.9, 64.8 }, { false, 8192, 4096, 192, 58.2, 55.2 }, { false, 8192, 7168, 64, 38.2, 40.2 }, { false, 8192, 7168, 90, 51.3, 53.4 },
		{ false, 8192, 7168, 128, 65.0, 55.2 }, { false, 8192, 7168, 192, 93.3, 80.8 }, { false, 11008, 7168, 33, 49.0, 43.3 }, { false, 2048, 14336, 128, 43.5, 44.6 }, { false, 5120, 14336, 90, 67.3, 70.4 },
		{ false, 8192, 4096, 192, 62.3, 57.9 }, { false, 8192, 7168, 64, 40.7, 42.1 }, { true, 5120, 4096, 65, 31.0, 37.9 }, { true, 5120, 4096, 90, 31.3, 38.5 }, { true, 5120, 4096, 128, 47.9, 39.5 },
		{ true, 5120, 7168, 90, 44.9, 50.7 }, { true, 5120, 7168, 128, 69.9, 52.0 }, { true, 5120, 14336, 65, 78.7, 81.9 }, { true, 6144, 4096, 65, 46.8, 43.5 }, { true, 8192, 7168, 65, 68.4, 61.7 },
	};
	for (const Measured& p : measured)
	{
		const int ranges = litenn_hip::fetch::exact_ranges(p.by_step, p.n, p.m, p.k / 256);
		CHECK((ranges > 1 ? p.ranged : p.without) <= 1.03 * (p.without < p.ranged ? p.without : p.ranged), "%d x %d x %d: %d ranges", p.m, p.n, p.k, ranges);
	}
	// the rows that go at a time: pairs of tiles, all rows among them, and sums within bounds
	for (int n : { 1, 31, 1000, 4096, 14336, 28672, 65535, 65536, 128256, 262144, 600000, 1 << 20 })
	{
		for (int ranges : { 2, 3, 4, 16 })
		{
			for (int m = 1; m <= 1 << 20; m += 1 + m / 7)
			{
				const int rows = litenn_hip::fetch::ranged_rows(ranges, n, m), times = (m + rows - 1) / rows;
				const long long sums = static_cast<long long>(ranges) * rows * n, bound = rows > 256 ? 1ll << 25 : rows > 64 ? 1ll << 26 : 1ll << 62;
				CHECK(rows > 0 && rows <= m + 63 && (times == 1 || rows % 64 == 0) && sums <= bound, "%d ranges of %d, %d rows: %d at a time", ranges, n, m, rows);
				CHECK(rows <= litenn_hip::fetch::ranged_rows_whole(ranges, n) && (times == 1 ? rows == m : m - (times - 1) * rows > 0), "%d ranges of %d, %d rows: %d at a time", ranges, n, m, rows);
				const int chosen = litenn_hip::fetch::exact_ranges(true, n, m, 16);
				CHECK(chosen == 1 || static_cast<long long>(chosen) * litenn_hip::fetch::ranged_rows(chosen, n, m) * n <= 1ll << 27, "%d x %d: %d ranges", n, m, chosen);
			}
		}
	}
	// more rows than go at a time keep the ranges of fewer
	for (int m : { 2336, 2337, 2400, 4096, 100000 })
	{
		CHECK(litenn_hip::fetch::exact_ranges(true, 28672, m, 16) == 2, "28672 x 4096, %d rows", m);
	}
}

// Memory that a model holds: what it is faster with is left out where it cannot be had, and not asked for on every call.
static void test_room()
{
	size_t largest = 1000, held = 0, asked = 0;
	char memory;
	const auto allocate = [&](size_t bytes) -> void* {
		++asked;
		held = bytes <= largest ? bytes : 0;
		return held ? &memory : nullptr;
	};
	const auto release = [&](void* p) {
		CHECK(p == &memory && held > 0, "released what was held");
		held = 0;
	};
	litenn_hip::Room room;
	const auto grow = [&](size_t need, size_t want) { return litenn_hip::grow_room(room, need, want, allocate, release); };
	CHECK(grow(100, 300) && held == 300 && room.bytes == 300 && asked == 1, "the larger one");
	CHECK(grow(200, 300) && grow(100, 100) && asked == 1, "no less than is there");
	CHECK(grow(400, 5000) && held == 400 && room.bytes == 400 && asked == 3, "the lesser one where the larger is refused");
	CHECK(grow(400, 5000) && grow(300, 9000) && held == 400 && asked == 3, "a size that was refused is not asked for again");
	CHECK(grow(300, 700) && held == 700 && asked == 4, "a smaller one is");
	CHECK(grow(800, 6000) && held == 800 && asked == 5, "more than is there, the refused size not tried");
	CHECK(!grow(2000, 2000) && held == 0 && !room.data && room.bytes == 0 && asked == 6, "none");
	CHECK(grow(500, 900) && held == 900 && asked == 7, "and some again");
}

int main(int argc, char** argv)
{
	if (argc > 1) // n k m ...: the forms of these products, with bfloat16 and with Float32 operands
	{
		for (int i = 1; i + 2 < argc; i += 3)
		{
			const int n = std::atoi(argv[i]), k_tiles = (std::atoi(argv[i + 1]) + 63) / 64, m = std::atoi(argv[i + 2]);
			std::printf("%d %d\n", static_cast<int>(litenn_hip::fetch::dense_form(n, k_tiles, m, 1)),
			            static_cast<int>(litenn_hip::fetch::dense_f32_form(n, m, 1)));
		}
		return 0;
	}
	test_rows_forms();
	test_options_forms();
	test_exact_forms();
	test_exact_ranges();
	test_room();
	test_dense_walks();
	test_dense_forms();
	test_dense_ranges();
	test_dense_sum_rows();
	test_gemm_chunk_ranges();
	test_gemm_weight_pieces();
	test_gemm_stream_pieces();
	test_stream_rows_and_pieces();
	test_attention_tiles();
	test_team_rows_and_segments();
	if (g_failures)
	{
		std::printf("%d checks failed\n", g_failures);
		return 1;
	}
	std::printf("fetch bounds ok\n");
	return 0;
}
