// Which bytes of a weight tensor, an activation vector or a KV cache a launch may request: the address
// arithmetic of every fetch pattern of the hot kernels, as plain functions that the kernels call on
// the device and that tests/cpp/fetch_bounds_test.cpp calls on the host for every thread of a
// launch.  The test walks page-exact, ragged and minimal shapes and asserts that every requested
// 16-byte piece holds at least one byte of its tensor (an aligned 16-byte piece never crosses a page,
// so such a piece touches mapped memory only) and that the pieces that are consumed cover what the
// kernel needs.  An over-fetch is found there, on the CPU, not by a fault on the GPU.
//
// Nothing here depends on HIP: with a host compiler the functions are ordinary inline functions.
#pragma once

#include <cstddef>
#include <cstdint>

#if defined(__HIPCC__)
#define LITENN_FETCH_FN __host__ __device__ __forceinline__
#else
#define LITENN_FETCH_FN inline
#endif

namespace litenn_hip
{
	namespace fetch
	{
		LITENN_FETCH_FN int imin(int a, int b) { return a < b ? a : b; }
		LITENN_FETCH_FN int imax(int a, int b) { return a > b ? a : b; }

		// ---- products of quantised weights with Float32 operands ----------------------------------
		// Whether Q6_K takes two 32-row tiles of activations a wavefront, which saves a second decode, K in eight ranges and one workgroup
		// to a CU.  Not for up to 256 tiles, which have a CU each, nor where up to 512 of one tile are all on the card at once and these
		// are not.  us of a call, weights from HBM, one tile and two: 4096 x 14336, 64 rows 51 and 71, 96 rows 82 and 67, 160 115
		// and 118, 300 190 and 181; 4128 x 4096, 33 rows 32 and 30; 1024 x 11008, 400 rows 78 and 62; 2100 x 4096, 200 rows 34 and 50.
		// (From 512 on one tile would sometimes be faster, 14336 x 4096 at 96 rows 76 and 93, 45 56 and 53, but walks K in four
		// ranges, which rounds more: K = 14336 1.23e-7 of the result, eight 1.16e-7.)
		inline bool exact_two_tiles(int strips, int m_tiles)
		{
			const int ones = strips * m_tiles, twos = strips * ((m_tiles + 1) / 2);
			return m_tiles > 1 && (ones >= 512 || (ones > 256 && twos <= 256));
		}

		// Chunks that a range of `per` adds up before they join its sum: those for which the roundings, each as large as what has been
		// summed by then, come to least
		struct SumLength
		{
			int chunks;
			long long roundings;
		};
		inline SumLength chunks_a_sum(int per)
		{
			SumLength best{ 1, -1 };
			for (int count = 1; count <= per; ++count)
			{
				long long sizes = 0;
				for (int from = 0; from < per; from += count)
				{
					const long long here = imin(count, per - from);
					sizes += here * (here + 1) / 2 + (from ? from + here : 0);
				}
				if (best.roundings < 0 || sizes < best.roundings)
				{
					best = { count, sizes };
				}
			}
			return best;
		}

		constexpr int kMostRanges = 16;
		// Rows of activations that go through the form with ranges at a time: whole pairs of tiles, about equally many each time, whose
		// sums bound what a call or a model holds beside its rows.  128 MB of them, or 256 rows up to 256 MB: a launch of fewer rows has
		// its last round of workgroups and its weights from HBM to itself, one of more finds less in the caches.  us of a call of
		// Q6_K with 64 MB, 128 and 512: 14336 x 4096 at 700 rows 324, 297, 299, at 2000 834, 834, 878, 28672 x 4096 at 2400 1936, 1971,
		// 2050; 128256 x 4096 at 300 in three launches 1223, in one 1156.  (By the forms without ranges 28672 x 4096 at 2400 takes 4970.)
		constexpr long long kRangedFloats = 1ll << 25, kMostRangedFloats = 1ll << 27;
		inline int ranged_rows_whole(int ranges, int n)
		{
			const long long a_row = static_cast<long long>(ranges) * n, some = kRangedFloats / a_row, wide = 2 * kRangedFloats / a_row;
			const long long rows = some > 256 ? some : wide > 256 ? 256 : wide;
			return rows < 64 ? 64 : rows < (1 << 24) ? static_cast<int>(rows / 64 * 64) : 1 << 24;
		}
		inline int ranged_rows(int ranges, int n, int m)
		{
			const int whole = ranged_rows_whole(ranges, n), times = (m + whole - 1) / whole;
			return times > 1 ? ((m + times - 1) / times + 63) / 64 * 64 : m;
		}

		// Ranges of K for the form that shares activations, with grid z, 1 where it does not pay: up to 256 workgroups of 128 x 64 results
		// as many as leave every one its place on the card, two to a CU.  by_step: Q6_K, whose steps are scaled one by one (other
		// formats that take the form, Q4_K and Q5_K, scale chunks).
		inline int exact_ranges(bool by_step, int n, int m, int chunks)
		{
			const int strips = (n + 31) / 32, m_tiles = (m + 31) / 32, tiles = strips * m_tiles;
			const int workgroups = (strips + 3) / 4 * ((m_tiles + 1) / 2), most = imin(imin(512 / imax(workgroups, 1), chunks), kMostRanges);
			// One tile of activations leaves the second half of its 64 rows empty: us of a call of Q6_K at 32 rows by the forms without
			// ranges and by this, 32800 x 4096 75 and 98, 128256 x 4096 221 and 255, at 9 rows 72 and 92, 212 and 226.
			if (m_tiles < 2)
			{
				return 1;
			}
			// Q6_K on more workgroups: as few ranges as round no more than the eight of the form without, whose wavefronts each read their
			// activations from L2 (us of a call by that and by this: 4096 x 14336 at 700 rows 385 and 321, 1000 598 and 415, 2000 2051 and
			// 848, 8192 x 4096 at 300 rows 124 and 103, 14336 x 4096 207 and 155), some rows at a time where their sums are many.
			if (by_step && workgroups > 256 && chunks >= 16)
			{
				const long long r = (chunks + 7) / 8;
				for (int ranges = 2; ranges <= 4; ++ranges)
				{
					const int each = (chunks + ranges - 1) / ranges;
					if (static_cast<long long>(ranges) * imin(m, 64) * n > kMostRangedFloats)
					{
						return 1;
					}
					if (ranges * chunks_a_sum(each).roundings + chunks <= 4 * r * (r + 1) + 3 * chunks)
					{
						return (chunks + each - 1) / each;
					}
				}
				return 1;
			}
			if (most < 2)
			{
				return 1;
			}
			const int per = (chunks + most - 1) / most, ranges = (chunks + per - 1) / per;
			// Q6_K, us of a call by the forms without ranges and by this (K = 4096, by workgroups: 64 28 and 32, 96 46 and 43, 112 50 and 46,
			// 160 76 and 59, 240 101 and 74; K = 14336: 64 69 and 70, 96 118 and 99, 128 126 and 115, 160 186 and 147; K = 1024, 128 24 and
			// 27).  Not where up to 512 single tiles are all on the card at once, though 80 workgroups have a third of their rows empty
			// (5120 x 4096 at 65 to 96 rows 31 and 38, x 7168 44 and 50, x 14336 79 and 82; at 128 48 and 40, 70 and 52, 125 and 87).
			if (by_step)
			{
				return workgroups >= 80 && chunks >= 16 && tiles > 512 ? ranges : 1;
			}
			// Q4_K and Q5_K, below the 200 workgroups that have a form for themselves, in tenths of a us.  Without ranges tiles of 32 x 32 go
			// through the card 256 at a time; with them every workgroup has its chunks, and what they leave is written and read (fitted to
			// 214 calls, of which none is 2 % slower by the form this takes: K = 4096, by tiles: 768 34 and 36, 896 44 and 37 or 42 and 40, 960
			// 43 and 46, 1280 55 and 50; K = 14336: 256 of 33 rows 38.5 and 37.7, of 64 40 and 41, Q5_K 41 and 44, 480 63 and 66, 512 66 and
			// 58, 896 129 and 94, 1280 175 and 122; K = 7168: 512 38 and 40, 768 54 and 50 or 51 and 53; K = 1024, 1280 23 and 29).
			// The first line is an older fit, which keeps calls off that the second was not fitted to.
			const bool worth = 210 + 44 * per < 272ll * tiles * chunks / 10000;
			const long long ranged = 155 + 44 * per + 19ll * ranges * m * n / 1000000, plain = 135 + 45 * chunks * ((tiles + 255) / 256) / 10;
			return workgroups < 200 && worth && ranged < plain ? ranges : 1;
		}

		// ---- attention of many rows: what a block of 32 query rows sees ---------------------------
		struct RowsSeen
		{
			int rows, keys;
			bool causal;
			long long q_at, window; // query i sees keys max(0, q_at + i - window + 1) .. (causal: q_at + i)
			// tiles of 32 keys that rows first .. first + count - 1 see
			int tiles(int first, int count) const
			{
				const long long end = first + count < rows ? first + count : rows;
				const long long to = causal && q_at + end < keys ? q_at + end : keys;
				const long long from = q_at + first - window + 1 > 0 ? q_at + first - window + 1 : 0;
				return to > from ? static_cast<int>((to - from + 31) / 32) : 0;
			}
		};
		// What up to 512 workgroups of `block` rows take, one to a CU and the longest first: a fixed part and a step for every `per` tiles of
		// keys (tenths of a us).  From the 257th on one waits for the shortest that is left before it.
		struct RowsCost
		{
			int once, twice, step; // fixed parts of a workgroup and of two in a row
		};
		inline int rows_time(const RowsSeen& a, int heads, int block, int per, RowsCost c)
		{
			const int blocks = (a.rows + block - 1) / block;
			const auto steps = [&](int b) { return (a.tiles(block * b, block) + per - 1) / per; };
			int time = c.once + c.step * steps(blocks - 1);
			for (int b = blocks - 1 - 256 / heads; b >= 0; --b)
			{
				const int last = (blocks - b) * heads - 1; // of the block's workgroups, in the order of their start
				time = imax(time, c.twice + c.step * (steps(b) + steps(blocks - 1 - imax(0, 511 - last) / heads)));
			}
			return time;
		}
		// Whether Float32 tiles go through four wavefronts of a workgroup of 32 rows, each with keys of its own, or through two pairs
		// of 64 rows that share theirs: four tiles a step, or two in less time.  Up to 256 workgroups four wavefronts are the faster
		// form, beyond 512 pairs, between the two what the steps take.  us of four and of pairs, 32 heads of 128 unless said: 200
		// rows on 1000 keys 54 and 79, 1000 on 1000 133 and 93; causal, 300 on 300 28.9 and 30.6, on 301 34.8 and 31.8, on 1000 91 and
		// 79, 512 on 512 45.7 and 44.6, of 64 26.5 and 29.6, 700 of 16 heads on 700 43 and 57, on 1000 70 and 80; every key seen
		// by all, 300 on 300 51 and 31.
		inline bool rows_float_alone(const RowsSeen& a, int heads, int dim)
		{
			const long long groups = static_cast<long long>(heads) * ((a.rows + 31) / 32);
			if (groups <= 256 || groups > 512)
			{
				return groups <= 256;
			}
			return dim > 64 ? rows_time(a, heads, 32, 4, { 98, 180, 55 }) < rows_time(a, heads, 64, 2, { 90, 160, 43 })
			                : rows_time(a, heads, 32, 4, { 64, 123, 31 }) < rows_time(a, heads, 64, 2, { 61, 110, 29 });
		}

		// Whether a call with options takes the tiles, or the row kernel with options, a key at a time and a workgroup for each row of a
		// head, whose time grows from some 500 of them on (us of that kernel and of the tiles, 32 heads over 8 unless said).
		// Float16 keys of 128: 2 rows on 48 9.0 / 10.6, on 64 10.5 / 10.4, on 96 14 / 10, on 1000 130 / 20, 64 on 64 29 / 10; heads of
		// 64 on 64 keys 8.7 / 7.8; of 72 on 64 9.2 / 10.8, on 80 10.5 / 10.7.  Float32 keys: 2 rows on 96 14.9 / 14.9, of 64 8.5 / 9.1
		// and on 128 10.1 / 9.1, 24 on 64 24 / 14.5 and of 64 9.2 / 9.2, 64 on 1000 850 / 54, with a soft cap 20 on 100 35 / 15.
		// Float32 heads of 72 to 112 take the tiles of 128, and five to seven elements a lane in the row kernel: 4 rows of 80 on 96
		// 8.8 / 14.8, on 200 14.5 / 20.5, on 600 34.3 / 37.3, of 96 on 1000 54.3 / 53.4, 128 heads, 4 rows of 80 on 300 19.7 / 26.4, of 96
		// 29.8 / 26.1, 8 rows of 80 on 96 14.8 / 13.9, of 96 20.2 / 13.7 and on 64 14.9 / 13.7.  (From 16 rows
		// on 96 keys on they stay on the tiles, whose error against 64 bits is the smaller one, 1.4e-7 and 1.6.)
		inline bool rows_options_tiles(size_t rows, size_t keys, size_t heads, size_t dim, bool f32)
		{
			const size_t groups = rows * heads;
			if (dim <= 64 || dim > 112 || (rows >= 16 && keys >= 96))
			{
				return f32 ? keys >= 96 || (keys >= 64 && groups >= 768) : keys >= 64;
			}
			if (!f32)
			{
				return keys >= (groups >= 768 ? 64u : 80u);
			}
			const size_t load = dim > 80 ? groups + groups / 2 : groups;
			return keys >= (load >= 1536 ? 64u : load >= 1024 ? 112u : load > 512 ? 300u : 800u);
		}

		// The same for a window with Float32 keys, a row of which sees `keys`.  A layer of a prompt, 2048 wide, in both: 48 and 64 rows on
		// themselves equal, 80 7 to 13 us apart, 32 four us the other way.  Below 96 keys heads that leave much of the tiles of 128
		// empty want some 1400 rows of all heads (the call alone, us of the row kernel and of the tiles, 66 keys): 4 heads of 128 with
		// values of 64, 64 rows 11.3 / 15.2, 16 heads 13.2 / 15.3, 48 heads, 32 rows 16.3 / 15.3; of 80, 4 heads, 64 rows 13.1 / 15.7,
		// 16 heads, 80 rows 15.6 / 15.9, 100 17.1 / 15.9; of 128 14.3 / 15.3, 16.4 / 15.5, 22.9 / 15.5; of 64 9.5 / 9.6, 10.4 / 9.7.
		inline bool rows_window_tiles(size_t rows, size_t keys, size_t heads, size_t dim, size_t vdim)
		{
			const bool filled = (dim <= 64 && vdim <= 64) || dim + vdim > 224;
			return rows >= 16 && keys > 64 && (keys >= 96 || filled || rows * heads >= 1400);
		}
		// The first of a prompt's rows that such a call takes where rows `first` .. alone are asked for: that of their block, or of the one
		// before where what is left would go by the row kernel, whose rows walk all keys, and a block more does not.  us of a whole
		// prompt of two layers, two rows asked for, from their own block and now: Kulurax 1024 wide 200 tokens 305 -> 275, 456 388 -> 308,
		// 712 486 -> 356, Degedra 712 519 -> 409 (and with all rows taken 288, 327, 380, 448).
		inline int window_rows_from(int rows, int first, int block, size_t keys, size_t heads, size_t dim, size_t vdim)
		{
			const int from = first / block * block;
			const bool again = from > 0 && !rows_window_tiles(rows - from, keys, heads, dim, vdim) && rows_window_tiles(rows - from + block, keys, heads, dim, vdim);
			return again ? from - block : from;
		}

		// ---- products over bfloat16 weights: the K tiles of a group of wavefronts ----------------
		// K is cut into `ranges` times `groups` parts, in order, that differ by a tile at most; the groups of a
		// workgroup take neighbouring ones.  They pass one set of barriers, so all of them go through as many
		// rounds as the longest part has tiles, multiplying only in their own; a group by itself makes its own.
		struct DenseWalk
		{
			int first, steps, rounds, all;
			LITENN_FETCH_FN bool multiplies(int round) const { return round < steps; }
			// the tile of a round that is requested and staged (in rounds that multiply nothing, one that is there)
			LITENN_FETCH_FN int tile(int round) const { return imin(first + imax(0, imin(round, steps - 1)), all - 1); }
		};
		LITENN_FETCH_FN DenseWalk dense_walk(int all, int ranges, int groups, int range, int group)
		{
			const int parts = ranges * groups, part = range * groups + group;
			const int first = all * part / parts, steps = all * (part + 1) / parts - first;
			return { first, steps, groups == 1 ? steps : (all + parts - 1) / parts, all };
		}

		// buffers of a ring at most: a kernel asks for tiles that many rounds past the one it multiplies
		constexpr int kDenseMaxBuffers = 8;

		// The form a product of bfloat16 operands takes, activation rows x weight rows of a tile; the two with a digit behind
		// differ in the buffers of their ring.  (All give the same bits.)
		enum DenseForm
		{
			kDense256x256, kDense128x256, kDense192x128, kDense192x128x3, kDense128x192, kDense128x128, kDense128x128x3,
			kDense128x64, kDense64x128, kDense64x64, kDense32x64, kDense32x32, kDenseForms
		};
		// The form of least time, where a CU has r workgroups of it: ns of a workgroup by itself (a fixed part and one a tile of K) and
		// of two that share a CU, r / 2 pairs and the odd one; a form whose ring leaves room for one only takes them in a row.
		// Fitted to 925 products with weights from HBM (25 matrices of the layered decoders' widths, 37 numbers of rows
		// from 17 to 2048): 0.3 % slower than the fastest form in the mean, 15 % at most, and at matrices kept out of the fit 0.5 %.
		// With one time for a workgroup whether it shares its CU or not, and without 128 x 128, tiles in a row took up to 1.6 times
		// as long: us for 639 x 4096 x 14336 in 192 x 128 with two buffers 201, 128 x 128 with three 132; 178 rows in three
		// ranges 78, 45; 1100 x 2048 x 5632 85, 51.
		struct DenseChoice
		{
			DenseForm form;
			long long ns;
		};
		inline DenseChoice dense_choice(int n, int k_tiles, int m, int ranges)
		{
			struct Cost
			{
				int rows, columns, alone, alone_tile, pair, pair_tile;
			};
			constexpr Cost costs[kDenseForms] = {
				{ 256, 256, 19800, 1350, 0, 0 },     { 128, 256, 8760, 860, 0, 0 },    { 192, 128, 6580, 860, 10510, 1120 },
				{ 192, 128, 7380, 660, 0, 0 },       { 128, 192, 7370, 690, 0, 0 },    { 128, 128, 4350, 770, 8090, 900 },
				{ 128, 128, 5180, 560, 0, 0 },       { 128, 64, 3650, 420, 5360, 640 }, { 64, 128, 3570, 450, 5460, 720 },
				{ 64, 64, 3230, 290, 3570, 450 },    { 32, 64, 2830, 240, 3130, 330 }, { 32, 32, 2840, 170, 2820, 270 },
			};
			const int tiles_of_k = imax(1, k_tiles / ranges);
			int best = 0;
			long long least = -1;
			for (int form = 0; form < kDenseForms; ++form)
			{
				const Cost& c = costs[form];
				const long long workgroups = static_cast<long long>((m + c.rows - 1) / c.rows) * ((n + c.columns - 1) / c.columns) * ranges;
				const long long in_a_cu = (workgroups + 255) / 256;
				const long long alone = c.alone + static_cast<long long>(c.alone_tile) * tiles_of_k;
				const long long pair = c.pair + static_cast<long long>(c.pair_tile) * tiles_of_k;
				const long long time = c.pair ? in_a_cu / 2 * pair + in_a_cu % 2 * alone : in_a_cu * alone;
				if (least < 0 || time < least)
				{
					least = time;
					best = form;
				}
			}
			return { static_cast<DenseForm>(best), least };
		}
		inline DenseForm dense_form(int n, int k_tiles, int m, int ranges) { return dense_choice(n, k_tiles, m, ranges).form; }

		// The ranges of K a sublayer's last product of m rows is walked in at once, each with sums of its own [m, ld] behind the one
		// before, none shorter than 16 tiles of K.  Float32 operands: where there are few tiles, enough for about two workgroups per CU.
		// bfloat16: as many as take least time, a range's sums being written and read again at 4500 bytes a ns.  (By the rule of the
		// Float32 operands 777 x 2048 x 5632 had one range, whose 224 tiles of 128 x 64 wait for L2: 37.8 us, and 30.6 in three
		// with 2.9 for the sums; 777 x 2048 x 4096 28.8, and 24.8 in two with 2.3; a 4096-wide prompt of 639 tokens, two
		// layers, 1085 and 1008.)  And 1.5 us for sums being there at all, which is what two ranges that save nothing take longer in
		// the mean: 2048 x 2048 in one and in two, the norm behind it included, 400 rows 16.0 and 18.5, 777 21.6 and 23.3.
		constexpr int kDenseMaxRanges = 4, kDenseRangedRows = 1024;
		inline int dense_ranges(int n, int k_tiles, int m)
		{
			if (m > kDenseRangedRows)
			{
				return 1;
			}
			int best = 1;
			long long least = -1;
			for (int ranges = 1; ranges <= imax(1, imin(kDenseMaxRanges, k_tiles / 16)); ++ranges)
			{
				const long long sums = ranges > 1 ? 1500 + static_cast<long long>(ranges - 1) * m * n * 16 / 9000 : 0;
				const long long ns = dense_choice(n, k_tiles, m, ranges).ns + sums;
				if (least < 0 || ns < least)
				{
					least = ns;
					best = ranges;
				}
			}
			return best;
		}
		inline int dense_f32_ranges(int n, int k_tiles, int m)
		{
			if (m > kDenseRangedRows)
			{
				return 1;
			}
			const int tiles = ((m + (m <= 32 ? 31 : 63)) / (m <= 32 ? 32 : 64)) * ((n + 63) / 64);
			return imax(1, imin(kDenseMaxRanges, imin((512 + tiles / 2) / tiles, k_tiles / 16)));
		}
		// rows of sums that passes of up to `rows` rows write: a short pass in ranges may write more than a long one
		inline size_t dense_sum_rows(size_t rows)
		{
			const size_t ranged = kDenseMaxRanges * (rows < kDenseRangedRows ? rows : kDenseRangedRows);
			return rows > ranged ? rows : ranged;
		}

		// The form a product of Float32 operands takes.  Beyond 256 tiles of 64 x 128 it is one chain over K, up to there, and for
		// 32 rows and fewer, two halves: results hang on this alone.  Time is what a tile of K takes of each workgroup that a CU
		// has in a row, tens of ns, fitted to 16 shapes from 30 x 4096 x 2048 to 1000 x 11264 x 4096; us for 64 x 128 and 64 x 256: 512
		// rows by 11264 x 2048 75, 85, by 7200 x 2048 52, 46; for 64 x 128, 64 x 64, 32 x 64 in halves: 512 rows by 2048 x 5632 in two
		// ranges 44, 57, 59, 64 by 11264 x 2048 31, 23, 26, 96 by 2048 x 2048 in two ranges 18, 13, 11.
		enum DenseF32Form { kF32Chain64x128, kF32Chain64x256, kF32Halves32x64, kF32Halves64x128, kF32Halves64x64, kDenseF32Forms };
		inline DenseF32Form dense_f32_form(int n, int m, int ranges)
		{
			const auto workgroups = [&](int rows, int columns) { return ((m + rows - 1) / rows) * ((n + columns - 1) / columns) * ranges; };
			const auto in_a_row = [&](int rows, int columns) { return (workgroups(rows, columns) + 255) / 256; };
			if (m > 32 && workgroups(64, 128) > 256)
			{
				return 83 * in_a_row(64, 128) <= 147 * in_a_row(64, 256) ? kF32Chain64x128 : kF32Chain64x256;
			}
			const int tall = 88 * in_a_row(64, 128), square = 64 * in_a_row(64, 64), low = 37 * in_a_row(32, 64);
			if (m <= 32 || low <= imin(tall, square))
			{
				return kF32Halves32x64;
			}
			return tall <= square ? kF32Halves64x128 : kF32Halves64x64;
		}

		// ---- matrix-core GEMM: raw weight blocks of one 256-element chunk per row --------------
		// A wavefront owns 16 * ng consecutive rows; their chunks land in its LDS slot row after row
		// as `pieces` 16-byte pieces each.  Formats whose chunks start on 16-byte boundaries take
		// chunk_bytes / 16 pieces; the others (Q2_K 84, Q3_K 110, Q6_K 210 bytes per chunk) start at
		// the 16-byte boundary at or below the chunk and need one piece more for the worst case.
		constexpr int gemm_weight_pieces(int chunk_bytes, bool aligned16)
		{
			return aligned16 ? chunk_bytes / 16 : (chunk_bytes + 14 + 15) / 16;
		}

		struct GemmWeightRequest
		{
			int row;    // 0 .. 16 ng - 1 within the wavefront's rows
			int offset; // byte offset of the piece from the row's first piece: 16 j
			bool issued;
		};

		// load instruction i (0 .. ceil(16 ng pieces / 64) - 1) of `lane`
		LITENN_FETCH_FN GemmWeightRequest gemm_weight_request(int i, int lane, int ng, int pieces)
		{
			const int total = ng * 16 * pieces;
			const int piece = imin(64 * i + lane, total - 1);
			const int row = piece / pieces;
			return { row, 16 * (piece - row * pieces), 64 * (i + 1) <= total || 64 * i + lane < total };
		}

		// rows past the end of the matrix re-read its last row (their products are never stored)
		LITENN_FETCH_FN int gemm_weight_row(int n_base, int row, int n) { return imin(n_base + row, n - 1); }

		// Address of the piece at `offset` of chunk c of the row that starts at `row_start`.  With
		// unaligned chunks `pieces` counts the worst misalignment; with a smaller one the last piece
		// holds no byte of the chunk, and behind the tensor's last chunk it can be the first 16 bytes
		// of a page that is not mapped: such a piece fetches the chunk's first piece again (its slot
		// bytes are never read).
		LITENN_FETCH_FN uintptr_t gemm_weight_piece(uintptr_t row_start, int c, int chunk_bytes, bool aligned16,
		                                            int offset)
		{
			const uintptr_t chunk = row_start + static_cast<size_t>(c) * static_cast<size_t>(chunk_bytes);
			if (aligned16)
			{
				return chunk + static_cast<uintptr_t>(offset);
			}
			const uintptr_t base = chunk & ~uintptr_t{ 15 };
			const uintptr_t from = base + static_cast<uintptr_t>(offset);
			return from >= chunk + static_cast<uintptr_t>(chunk_bytes) ? base : from;
		}

		// where the decoders find the chunk's first byte inside the row's part of the slot
		LITENN_FETCH_FN int gemm_weight_misalignment(uintptr_t row_start, int c, int chunk_bytes, bool aligned16)
		{
			return aligned16
			           ? 0
			           : static_cast<int>((row_start + static_cast<size_t>(c) * static_cast<size_t>(chunk_bytes)) & 15);
		}

		// ---- streaming GEMV: rows HBM -> LDS --------------------------------------------------
		// Wavefront s of a row's `slices` fetches bytes [s * slice_bytes, s * slice_bytes + len) of
		// every row it walks, as loads of 1 KB (64 lanes x 16 bytes).
		LITENN_FETCH_FN uint32_t stream_slice_len(bool whole_slices, uint32_t slice_bytes, uint32_t row_bytes,
		                                          uint32_t slice_off)
		{
			return whole_slices ? slice_bytes : (slice_bytes < row_bytes - slice_off ? slice_bytes : row_bytes - slice_off);
		}

		struct StreamPiece
		{
			uint32_t offset; // from the slice's first byte
			bool issued;
		};

		// Load instruction i of a row, lane `lane`.  Every row takes the same number of instructions
		// whatever the slice's length (the vmcnt bookkeeping is fixed at compile time): an instruction
		// whose 1 KB lies wholly past a short slice still runs in lane 0, which fetches the slice's
		// first 16 bytes again into that (unused) part of the slot.
		LITENN_FETCH_FN StreamPiece stream_row_piece(int i, int lane, uint32_t slice_len, bool whole_slices)
		{
			const uint32_t off = static_cast<uint32_t>(i) * 1024u + static_cast<uint32_t>(lane) * 16u;
			const bool inside = off < slice_len;
			return { inside ? off : 0u, inside || (lane == 0 && !whole_slices) };
		}

		// rows [row0, row0 + count) of the launch that wavefront group g of workgroup `block` walks
		struct StreamRows
		{
			int row0, count;
		};
		// A workgroup's groups walk consecutive runs of its rows.  The first half of the groups walk
		// `run` rows each and the second half `run - diff` (diff > 0 only with an even number of
		// groups): of the two wavefronts that share a SIMD the one that arrived first (the lower
		// index) gets ahead of the other, and the longer run levels the two.
		LITENN_FETCH_FN int stream_group_run(int g, int groups, int run, int diff)
		{
			return 2 * g < groups ? run : run - diff;
		}
		LITENN_FETCH_FN int stream_group_first(int g, int groups, int run, int diff)
		{
			const int half = groups / 2;
			return 2 * g < groups ? g * run : g * run - (g - half) * diff;
		}
		LITENN_FETCH_FN int stream_block_rows(int groups, int run, int diff) { return groups * run - (groups / 2) * diff; }
		LITENN_FETCH_FN StreamRows stream_group_rows(int block, int g, int groups, int run, int diff, int n_total)
		{
			const int row0 = block * stream_block_rows(groups, run, diff) + stream_group_first(g, groups, run, diff);
			return { row0, imax(0, imin(stream_group_run(g, groups, run, diff), n_total - row0)) };
		}

		// first float of the 128-bit activation load j of thread `tid` (clamped: every lane issues
		// every load)
		LITENN_FETCH_FN int stream_x_index(int tid, int j, int threads, int k) { return imin((tid + j * threads) * 4, k - 4); }

		// ---- decoder-block kernel: rows dealt out per XCD, and the output projection's columns ---
		// The launch's 256 workgroups form eight teams of 32 (workgroup b: team b % 8, place b / 8;
		// the dispatcher deals workgroups to the card's eight XCDs in that order, so a team shares
		// an L2).  Team t takes an eighth of the rows of each of the up to three matrices of the
		// first phase: virtual row v of the team lies in matrix m at row t * (n[m] / 8) + r.
		struct TeamRow
		{
			int m, local;
		};
		LITENN_FETCH_FN TeamRow team_row(int v, int team, int n0, int n1, int n2)
		{
			const int r0 = n0 >> 3, r1 = n1 >> 3, r2 = n2 >> 3;
			if (v < r0)
			{
				return { 0, team * r0 + v };
			}
			if (v < r0 + r1)
			{
				return { 1, team * r1 + (v - r0) };
			}
			return { 2, team * r2 + imin(v - r0 - r1, r2 > 0 ? r2 - 1 : 0) };
		}

		// The third phase multiplies a column slice of the output projection: team t owns `seg_bytes`
		// bytes of every row (the blocks of its heads' columns), from byte t * seg_bytes of the row.
		// A wavefront fetches the segments of `rows_per_fetch` consecutive rows (4096 weights in all)
		// as one run of 16-byte pieces, piece p of the run being piece p % seg_pieces of row
		// p / seg_pieces; load instruction i moves pieces 64 i .. 64 i + 63 to consecutive LDS
		// addresses, so the slot holds what a 4096-wide slice of a row would.
		struct SegmentPiece
		{
			int row;         // 0 .. rows_per_fetch - 1
			uint32_t offset; // from the segment's first byte
			bool issued;
		};
		LITENN_FETCH_FN SegmentPiece segment_piece(int i, int lane, int seg_pieces, int rows_per_fetch)
		{
			const int total = seg_pieces * rows_per_fetch;
			const int p = 64 * i + lane;
			const int q = imin(p, total - 1);
			return { q / seg_pieces, static_cast<uint32_t>(q % seg_pieces) * 16u, p < total };
		}

		// ---- tiled GEMM: the chunks of K a group of wavefronts walks ------------------------------
		// K (in 256-element chunks) is cut into `parts` consecutive ranges: grid z x the K groups of a
		// workgroup, part = blockIdx.z * groups + group
		struct ChunkRange
		{
			int begin, end;
		};
		LITENN_FETCH_FN ChunkRange gemm_chunk_range(int part, int parts, int chunks)
		{
			return { part * chunks / parts, (part + 1) * chunks / parts };
		}
		// The K groups of one workgroup pass the same barriers, one set per chunk: a launch with more than
		// one group per workgroup is only made when this holds (every range is then equally long)
		LITENN_FETCH_FN bool gemm_ranges_equal(int chunks, int parts)
		{
			return parts > 0 && chunks >= parts && chunks % parts == 0;
		}

		// ---- tiled prompt attention: key / value rows of a 64-key tile -------------------------
		// keys any query row of the 64-row tile starting at q_first may see
		LITENN_FETCH_FN int attn_tile_kv_len(int past, int q_first, int q_tile, int m)
		{
			return past + imin(m, q_first + q_tile) - 1 + 1;
		}
		// cache row fetched for slot `idx` (0 .. 63) of key tile kt: past the end the last key is re-read
		LITENN_FETCH_FN int attn_tile_key(int kt, int key_tile, int idx, int kv_len)
		{
			return imin(kt * key_tile + idx, kv_len - 1);
		}
	} // namespace fetch
} // namespace litenn_hip
