// Linear layers over bfloat16 weights for gfx950: y[m, n] = sum_k x[m, k] W[n, k].
//
// One row (decode) streams the weights once through registers with Float32 activations in LDS; many
// rows (prompt) run on the matrix cores, either with bfloat16 operands or, where Float32 operands are
// asked for, with each activation taken apart exactly into three bfloat16 values.  Every accumulation is
// Float32.  The reference has no counterpart (its linears are f32 MatMul nodes,
// src/LiteNN/Layer/Linear.h:67-95).
#include "dense.hpp"

#include <algorithm>
#include <type_traits>

namespace litenn_hip
{
	namespace
	{
		typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
		typedef float floatx4 __attribute__((ext_vector_type(4)));
		typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));

		// ------------------------------------------------------------------
		// One activation row.  A wavefront owns R consecutive rows at a time and walks K in blocks of 512
		// (64 lanes x 8 weights, one 16-byte load each); kFlight blocks of every row are requested ahead,
		// the first ones before the activations are even looked at, so that the weights travel while the
		// prologue runs, and the next rows' first blocks while the current rows finish.
		// LDS: the activations as two planes (elements 0..3 and 4..7 of every group of eight), so that
		// consecutive lanes read consecutive 16-byte pieces.
		// ------------------------------------------------------------------
		constexpr int kRowThreads = 512, kRowWaves = kRowThreads / 64, kFlight = 4, kRowBlock = 512;

		struct RowArgs
		{
			DenseRow d;
			int groups; // steps of kFlight blocks that cover a row
		};

		__device__ __forceinline__ int row_slot(int k, int half)
		{
			return ((k >> 2) & 1) * half + (k >> 3) * 4 + (k & 3);
		}

		// elements i .. i + 3 of a vector of k, zero beyond (global loads take any 4-byte address)
		__device__ __forceinline__ floatx4 load_piece(const float* x, int i, int k)
		{
			typedef floatx4 floatx4_a4 __attribute__((aligned(4)));
			floatx4 v = { 0.0f, 0.0f, 0.0f, 0.0f };
			if (i + 3 < k)
			{
				v = *reinterpret_cast<const floatx4_a4*>(x + i);
			}
			else
			{
#pragma unroll
				for (int e = 0; e < 3; ++e)
				{
					v[e] = i + e < k ? x[i + e] : 0.0f;
				}
			}
			return v;
		}

		__device__ __forceinline__ floatx4 load_piece(const uint16_t* x, int i, int k)
		{
			floatx4 v = { 0.0f, 0.0f, 0.0f, 0.0f };
			if (i + 3 < k)
			{
				const uint2 w = *reinterpret_cast<const uint2*>(x + i);
				v = floatx4{ bf16_to_f32(w.x & 0xffffu), bf16_to_f32(w.x >> 16), bf16_to_f32(w.y & 0xffffu), bf16_to_f32(w.y >> 16) };
			}
			else
			{
#pragma unroll
				for (int e = 0; e < 3; ++e)
				{
					v[e] = i + e < k ? bf16_to_f32(x[i + e]) : 0.0f;
				}
			}
			return v;
		}

		__device__ __forceinline__ float square_sum(const floatx4& v, float acc)
		{
			acc = fmaf(v.x, v.x, acc);
			acc = fmaf(v.y, v.y, acc);
			acc = fmaf(v.z, v.z, acc);
			return fmaf(v.w, v.w, acc);
		}

		// sum over the workgroup; `red` holds one float per wavefront
		__device__ __forceinline__ float block_sum(float v, float* red)
		{
			v = wave_sum(v);
			__syncthreads();
			if ((threadIdx.x & 63) == 0)
			{
				red[threadIdx.x >> 6] = v;
			}
			__syncthreads();
			float t = 0.0f;
			for (int i = 0; i < static_cast<int>(blockDim.x >> 6); ++i)
			{
				t += red[i];
			}
			return t;
		}

		template <int R>
		__global__ __launch_bounds__(kRowThreads) void dense_row_kernel(const RowArgs args)
		{
			extern __shared__ __attribute__((aligned(16))) float row_lds[];
			__shared__ float red[kRowWaves];
			const DenseRow& d = args.d;
			const int lane = threadIdx.x & 63;
			const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
			const int n = d.w.n, k = d.w.k, pitch = d.w.pitch, groups = args.groups;
			const int row_groups = (n + R - 1) / R;
			const int stride = static_cast<int>(gridDim.x) * kRowWaves;
			int rg = static_cast<int>(blockIdx.x) * kRowWaves + wave;
			const bool busy = rg < row_groups;
			const int half = groups * kFlight * kRowBlock / 2;

			u32x4 cur[R][kFlight], nxt[R][kFlight];
			const auto request = [&](u32x4 (&dst)[R][kFlight], int group_of_rows, int step) {
#pragma unroll
				for (int r = 0; r < R; ++r)
				{
					const uint16_t* row = d.w.w + static_cast<size_t>(min(group_of_rows * R + r, n - 1)) * pitch;
#pragma unroll
					for (int p = 0; p < kFlight; ++p)
					{
						// past the row's end any of its weights will do: the activations there are zero
						const int at = (step * kFlight + p) * kRowBlock + lane * 8;
						dst[r][p] = __builtin_nontemporal_load(reinterpret_cast<const u32x4*>(row + (at < pitch ? at : 0)));
					}
				}
			};
			if (busy)
			{
				request(cur, rg, 0);
			}

			// activations, four at a time where k allows; a thread's first kKept pieces stay in registers
			const int pieces = half >> 1; // of four floats, zeros behind the k-th
			const auto put = [&](int piece, floatx4 v) {
				*reinterpret_cast<floatx4*>(row_lds + (piece & 1) * half + (piece >> 1) * 4) = v;
			};
			if (d.prologue == kRowAddNorm)
			{
				constexpr int kKept = 2;
				floatx4 x[kKept], sub[kKept], subw[kKept], nw[kKept];
#pragma unroll
				for (int e = 0; e < kKept; ++e)
				{
					const int i = 4 * (static_cast<int>(threadIdx.x) + kRowThreads * e);
					x[e] = load_piece(d.x, i, k);
					sub[e] = d.sub ? load_piece(d.sub, i, k) : floatx4{ 0.0f, 0.0f, 0.0f, 0.0f };
					subw[e] = d.sub ? load_piece(d.sub_w, i, k) : floatx4{ 0.0f, 0.0f, 0.0f, 0.0f };
					nw[e] = d.norm_w ? load_piece(d.norm_w, i, k) : floatx4{ 1.0f, 1.0f, 1.0f, 1.0f };
				}
				float scale_sub = 0.0f;
				if (d.sub)
				{
					float ss = 0.0f;
#pragma unroll
					for (int e = 0; e < kKept; ++e)
					{
						ss = square_sum(sub[e], ss);
					}
					for (int p = threadIdx.x + kRowThreads * kKept; p < pieces; p += kRowThreads)
					{
						ss = square_sum(load_piece(d.sub, 4 * p, k), ss);
					}
					scale_sub = 1.0f / sqrtf(block_sum(ss, red) / static_cast<float>(k) + d.eps);
				}
				float ss = 0.0f;
				const auto enter = [&](int p, floatx4 v, floatx4 s, floatx4 sw, floatx4 w) {
					if (d.sub)
					{
						v += s * scale_sub * sw;
					}
					if (d.x_out && blockIdx.x == 0)
					{
#pragma unroll
						for (int i = 0; i < 4; ++i)
						{
							if (4 * p + i < k)
							{
								d.x_out[4 * p + i] = v[i];
							}
						}
					}
					ss = square_sum(v, ss);
					return v * w;
				};
#pragma unroll
				for (int e = 0; e < kKept; ++e)
				{
					x[e] = enter(static_cast<int>(threadIdx.x) + kRowThreads * e, x[e], sub[e], subw[e], nw[e]);
				}
				for (int p = threadIdx.x + kRowThreads * kKept; p < pieces; p += kRowThreads)
				{
					put(p, enter(p, load_piece(d.x, 4 * p, k), d.sub ? load_piece(d.sub, 4 * p, k) : floatx4{ 0.0f, 0.0f, 0.0f, 0.0f },
					             d.sub ? load_piece(d.sub_w, 4 * p, k) : floatx4{ 0.0f, 0.0f, 0.0f, 0.0f },
					             d.norm_w ? load_piece(d.norm_w, 4 * p, k) : floatx4{ 1.0f, 1.0f, 1.0f, 1.0f }));
				}
				const float scale = d.norm_w ? 1.0f / sqrtf(block_sum(ss, red) / static_cast<float>(k) + d.eps) : 1.0f;
#pragma unroll
				for (int e = 0; e < kKept; ++e)
				{
					const int p = static_cast<int>(threadIdx.x) + kRowThreads * e;
					if (p < pieces)
					{
						put(p, x[e] * scale);
					}
				}
				for (int p = threadIdx.x + kRowThreads * kKept; p < pieces; p += kRowThreads)
				{
					floatx4* slot = reinterpret_cast<floatx4*>(row_lds + (p & 1) * half + (p >> 1) * 4);
					*slot = *slot * scale; // this thread's own
				}
			}
			else if (d.prologue == kRowHeadGate)
			{
				const int heads = k / d.vdim;
				for (int h = wave; h < heads; h += kRowWaves)
				{
					const float* o = d.x + static_cast<size_t>(h) * d.vdim;
					float ss = 0.0f;
					for (int e = lane; e < d.vdim; e += 64)
					{
						ss = fmaf(o[e], o[e], ss);
					}
					const float scale = 1.0f / sqrtf(wave_sum(ss) / static_cast<float>(d.vdim) + d.eps);
					for (int e = lane; e < d.vdim; e += 64)
					{
						const float g = d.gate[h * d.vdim + e];
						row_lds[row_slot(h * d.vdim + e, half)] = o[e] * scale * d.norm_w[e] * (g * sigmoid_f32(g));
					}
				}
				for (int i = k + threadIdx.x; i < 2 * half; i += kRowThreads)
				{
					row_lds[row_slot(i, half)] = 0.0f;
				}
			}
			else if (d.x16)
			{
#pragma unroll 4
				for (int p = threadIdx.x; p < pieces; p += kRowThreads)
				{
					put(p, load_piece(d.x16, 4 * p, k));
				}
			}
			else
			{
#pragma unroll 4
				for (int p = threadIdx.x; p < pieces; p += kRowThreads)
				{
					put(p, load_piece(d.x, 4 * p, k));
				}
			}
			__syncthreads();
			if (!busy)
			{
				return;
			}

			float acc[R];
#pragma unroll
			for (int r = 0; r < R; ++r)
			{
				acc[r] = 0.0f;
			}
			int step = 0;
			while (true)
			{
				// the step after this one, possibly of the next rows
				int next_rg = rg, next_step = step + 1;
				if (next_step == groups)
				{
					next_step = 0;
					next_rg = rg + stride;
				}
				const bool more = next_rg < row_groups;
				if (more)
				{
					request(nxt, next_rg, next_step);
				}
#pragma unroll
				for (int p = 0; p < kFlight; ++p)
				{
					const int piece = (step * kFlight + p) * (kRowBlock / 8) + lane;
					const floatx4 x0 = *reinterpret_cast<const floatx4*>(row_lds + piece * 4);
					const floatx4 x1 = *reinterpret_cast<const floatx4*>(row_lds + half + piece * 4);
#pragma unroll
					for (int r = 0; r < R; ++r)
					{
						const u32x4 w = cur[r][p];
						float a = acc[r];
						a = fmaf(__uint_as_float(w.x << 16), x0.x, a);
						a = fmaf(__uint_as_float(w.x & 0xffff0000u), x0.y, a);
						a = fmaf(__uint_as_float(w.y << 16), x0.z, a);
						a = fmaf(__uint_as_float(w.y & 0xffff0000u), x0.w, a);
						a = fmaf(__uint_as_float(w.z << 16), x1.x, a);
						a = fmaf(__uint_as_float(w.z & 0xffff0000u), x1.y, a);
						a = fmaf(__uint_as_float(w.w << 16), x1.z, a);
						a = fmaf(__uint_as_float(w.w & 0xffff0000u), x1.w, a);
						acc[r] = a;
					}
				}
				if (next_step == 0)
				{
#pragma unroll
					for (int r = 0; r < R; ++r)
					{
						acc[r] = wave_sum(acc[r]);
					}
					if (lane == 0)
					{
						if constexpr (R >= 2)
						{
							if (d.glu)
							{
#pragma unroll
								for (int r = 0; r < R; r += 2)
								{
									if (rg * R + r < n)
									{
										d.y[(rg * R + r) >> 1] = clamped_glu(acc[r], acc[r + 1], d.act);
									}
								}
							}
						}
						if (R < 2 || !d.glu)
						{
#pragma unroll
							for (int r = 0; r < R; ++r)
							{
								if (rg * R + r < n)
								{
									d.y[rg * R + r] = soft_cap(acc[r], d.softcap);
								}
							}
						}
					}
#pragma unroll
					for (int r = 0; r < R; ++r)
					{
						acc[r] = 0.0f;
					}
				}
				if (!more)
				{
					return;
				}
				rg = next_rg;
				step = next_step;
#pragma unroll
				for (int r = 0; r < R; ++r)
				{
#pragma unroll
					for (int p = 0; p < kFlight; ++p)
					{
						cur[r][p] = nxt[r][p];
					}
				}
			}
		}

		// ------------------------------------------------------------------
		// Many rows: BM activation rows x BN weight rows per workgroup, bfloat16 operands (Float32 ones:
		// below), K in tiles of 64 double-buffered in LDS (global -> registers tiles ahead -> LDS
		// while the previous tile is multiplied), v_mfma_f32_16x16x32_bf16 with the weights as the A operand, so that a lane
		// ends up with four consecutive outputs of one activation row.  The 16-byte pieces of a 128-byte
		// LDS row are permuted by the row's low three bits: the 16 rows a fragment read touches then fall
		// on different banks.
		// ------------------------------------------------------------------
		constexpr int kTileK = 64;

		struct TileArgs
		{
			DenseRows d;
			int m_tiles, n_tiles;
		};

		// Tile of this workgroup: the eight XCDs (workgroups are dealt to them round-robin) walk eight
		// consecutive ranges of tiles, and inside a range eight row tiles share a weight tile's L2 lines.
		__device__ __forceinline__ bool tile_of(const TileArgs& a, int& tm, int& tn)
		{
			const int total = a.m_tiles * a.n_tiles;
			const int per = static_cast<int>(gridDim.x) >> 3;
			const int t = static_cast<int>(blockIdx.x & 7) * per + static_cast<int>(blockIdx.x >> 3);
			if (t >= total)
			{
				return false;
			}
			constexpr int kGroup = 8;
			const int width = kGroup * a.n_tiles;
			const int first = t / width * kGroup, in = t % width;
			const int rows = min(kGroup, a.m_tiles - first);
			tm = first + in % rows;
			tn = in / rows;
			return true;
		}

		__device__ __forceinline__ int operand_row(const DenseRows& d, int m)
		{
			int r = min(m, d.m - 1);
			if (d.a_ring > 0)
			{
				r += d.a_first;
				r -= r >= d.a_ring ? d.a_ring : 0;
			}
			return r;
		}

		// four consecutive outputs n .. n + 3 of activation row m
		template <typename T>
		__device__ __forceinline__ void store_outputs(const DenseRows& d, int m, int n, const floatx4& v)
		{
			if (m >= d.m || n >= d.w.n)
			{
				return;
			}
			float f[4] = { v.x, v.y, v.z, v.w };
			if (d.out == kOutGlu)
			{
				T* c = static_cast<T*>(d.c) + static_cast<size_t>(m) * d.ldc + (n >> 1);
#pragma unroll
				for (int i = 0; i < 2; ++i)
				{
					if (n + 2 * i < d.w.n)
					{
						operand_store(c + i, clamped_glu(f[2 * i], f[2 * i + 1], d.act));
					}
				}
				return;
			}
			if (d.out == kOutOperand && sizeof(T) == 2)
			{
				uint16_t* c = static_cast<uint16_t*>(d.c) + static_cast<size_t>(m) * d.ldc + n;
				if (n + 3 < d.w.n)
				{
					*reinterpret_cast<uint2*>(c) = make_uint2(pack_bf16(f[0], f[1]), pack_bf16(f[2], f[3]));
				}
				else
				{
					for (int i = 0; i < 4 && n + i < d.w.n; ++i)
					{
						c[i] = to_bf16(f[i]);
					}
				}
				return;
			}
			if (d.softcap > 0.0f)
			{
#pragma unroll
				for (int i = 0; i < 4; ++i)
				{
					f[i] = soft_cap(f[i], d.softcap);
				}
			}
			float* c = static_cast<float*>(d.c) + blockIdx.y * d.split_stride + static_cast<size_t>(m) * d.ldc + n;
			if (n + 3 < d.w.n && (d.ldc & 3) == 0)
			{
				*reinterpret_cast<float4*>(c) = make_float4(f[0], f[1], f[2], f[3]);
			}
			else
			{
				for (int i = 0; i < 4 && n + i < d.w.n; ++i)
				{
					c[i] = f[i];
				}
			}
		}

		// A Float32 as three values whose upper halves are bfloat16 and whose sum it is: eight significant bits, the next
		// eight, the rest.  An infinity or a NaN is the first one, the others zero.
		template <bool FINITE>
		__device__ __forceinline__ void cut_in_three(uint32_t bits, uint32_t (&part)[3])
		{
			if constexpr (FINITE)
			{
				part[0] = bits & 0xffff0000u;
				const float rest = __uint_as_float(bits) - __uint_as_float(part[0]);
				part[1] = __float_as_uint(rest) & 0xffff0000u;
				part[2] = __float_as_uint(rest - __uint_as_float(part[1]));
				return;
			}
			const bool special = (bits & 0x7f800000u) == 0x7f800000u;
			const uint32_t quiet = (bits & 0x007fffffu) != 0u ? 0x00400000u : 0u;
			part[0] = (bits | (special ? quiet : 0u)) & 0xffff0000u;
			const float rest = special ? 0.0f : __uint_as_float(bits) - __uint_as_float(part[0]);
			part[1] = __float_as_uint(rest) & 0xffff0000u;
			part[2] = __float_as_uint(rest - __uint_as_float(part[1]));
		}

		// WM x WN wavefronts share the tile.
		//
		// F32: Float32 operands.  The weights are bfloat16 as they are; an activation is the sum of three bfloat16 values
		// of eight bits each, cut off its front one after the other, which is exact, so that three products per operand
		// pair give what one of Float32 operands gives, at 48 cycles per 32 elements of K where v_mfma_f32_16x16x4_f32
		// takes 256.  The activations are taken apart on their way into LDS, without a look at infinities where a piece's
		// magnitudes add up to a number (64 x 128 on 500 x 11264 x 2048 100 -> 88 us; eight wavefronts instead of four 88 -> 85).
		//
		// Two wavefronts a SIMD hide most of a step's chain of latencies (request, LDS, barrier, products that feed each other):
		// eight of them on 128 x 128 take 49 us for 2048 x 5632 at 1254 rows, four 70.  S tiles of K travel at any time.
		// Every output is one chain of products over K in order whatever the form, so that bfloat16 results hang on
		// the ranges of K alone.
		//
		// KG (Float32 operands only): groups of WM x WN wavefronts share the tile and cut its K walk into as many ranges,
		// each through buffers of its own; their sums meet in LDS at the end, in K order.
		template <int BM, int BN, int WM, int WN, int KG, int S, bool F32>
		__global__ __launch_bounds__(64 * WM * WN * KG) void dense_tile_kernel(const TileArgs args)
		{
			constexpr int T = 64 * WM * WN, kRowStep = T / 8; // threads of a group, rows they stage at once
			constexpr int P = F32 ? 3 : 1; // parts of an activation
			typedef std::conditional_t<F32, float, uint16_t> operand;
			constexpr int TM = BM / WM / 16, TN = BN / WN / 16;
			constexpr int LA = BM / kRowStep, LW = BN / kRowStep; // 16-byte pieces a thread stages per K tile
			static_assert(KG == 1 || F32, "one chain of products over K");
			static_assert(S % 2 == 0, "register sets and LDS buffers alternate together");
			static_assert(LA * kRowStep == BM && LW * kRowStep == BN && TM * WM * 16 == BM && TN * WN * 16 == BN, "tile");
			extern __shared__ __attribute__((aligned(16))) uint16_t tile_lds[]; // per group: activations [2][P][BM][64], weights [2][BN][64]
			const int group = KG == 1 ? 0 : __builtin_amdgcn_readfirstlane(threadIdx.x / T);
			uint16_t* const xs = tile_lds + group * (2 * kTileK * (P * BM + BN));
			uint16_t* const ws = xs + 2 * P * BM * kTileK;
			const DenseRows& d = args.d;
			int tm, tn;
			if (!tile_of(args, tm, tn))
			{
				return;
			}
			const int tid = threadIdx.x & (T - 1), lane = tid & 63, wave = tid >> 6;
			const int j = lane & 15, g = lane >> 4;
			const int wm = wave / WN, wn = wave % WN;
			const int m0 = tm * BM, n0 = tn * BN;
			const int k = d.w.k;
			const fetch::DenseWalk walk = fetch::dense_walk(d.w.pitch / kTileK, d.splits, KG, static_cast<int>(blockIdx.y), group);

			const int ch = tid & 7, row = tid >> 3; // this thread's piece column and first row
			const operand* xp[LA];
			const uint16_t* wp[LW];
#pragma unroll
			for (int i = 0; i < LA; ++i)
			{
				xp[i] = static_cast<const operand*>(d.a) + static_cast<size_t>(operand_row(d, m0 + row + kRowStep * i)) * d.lda + ch * 8;
			}
#pragma unroll
			for (int i = 0; i < LW; ++i)
			{
				wp[i] = d.w.w + static_cast<size_t>(min(n0 + row + kRowStep * i, d.w.n - 1)) * d.w.pitch + ch * 8;
			}
			// tile t of K is in register set t % S until it is staged, and then in LDS buffer t % 2
			constexpr int kWords = F32 ? 2 : 1; // of a piece of eight activations
			u32x4 rx[S][LA][kWords], rw[S][LW];
			const auto request = [&](int step, int set) {
#pragma unroll
				for (int i = 0; i < LA; ++i)
				{
#pragma unroll
					for (int w = 0; w < kWords; ++w)
					{
						rx[set][i][w] = *reinterpret_cast<const u32x4*>(xp[i] + step * kTileK + 4 * w);
					}
				}
#pragma unroll
				for (int i = 0; i < LW; ++i)
				{
					rw[set][i] = *reinterpret_cast<const u32x4*>(wp[i] + step * kTileK);
				}
			};
			const auto stage = [&](int step, int set) {
				const int left = k - step * kTileK - ch * 8; // valid elements of this thread's pieces
				if (left < 8)
				{
					// behind the k-th activation there may be anything: zero it
#pragma unroll
					for (int i = 0; i < LA; ++i)
					{
#pragma unroll
						for (int e = 0; e < 4 * kWords; ++e)
						{
							const uint32_t keep = F32 ? (e < left ? 0xffffffffu : 0u)
							                          : left >= 2 * e + 2 ? 0xffffffffu : left == 2 * e + 1 ? 0xffffu : 0u;
							rx[set][i][e / 4][e % 4] &= keep;
						}
					}
				}
				const int slot = (ch ^ (row & 7)) * 8;
#pragma unroll
				for (int i = 0; i < LA; ++i)
				{
					uint16_t* const dst = xs + (set & 1) * (P * BM * kTileK) + (row + kRowStep * i) * kTileK + slot;
					if constexpr (F32)
					{
						u32x4 part[3];
						const auto cut = [&](auto finite) {
#pragma unroll
							for (int e = 0; e < 4; ++e)
							{
								uint32_t lo[3], hi[3];
								cut_in_three<decltype(finite)::value>(rx[set][i][e / 2][2 * (e % 2)], lo);
								cut_in_three<decltype(finite)::value>(rx[set][i][e / 2][2 * (e % 2) + 1], hi);
#pragma unroll
								for (int p = 0; p < 3; ++p)
								{
									part[p][e] = __builtin_amdgcn_perm(hi[p], lo[p], 0x07060302u); // the upper halves
								}
							}
						};
						float sum = 0.0f; // of magnitudes: one that is no number or infinite shows in it
#pragma unroll
						for (int e = 0; e < 8; ++e)
						{
							sum += fabsf(__uint_as_float(rx[set][i][e / 4][e % 4]));
						}
						if (__builtin_expect(__any(!(sum <= 3.402823466e38f)), 0))
						{
							cut(std::false_type{});
						}
						else
						{
							cut(std::true_type{});
						}
#pragma unroll
						for (int p = 0; p < 3; ++p)
						{
							*reinterpret_cast<u32x4*>(dst + p * (BM * kTileK)) = part[p];
						}
					}
					else
					{
						*reinterpret_cast<u32x4*>(dst) = rx[set][i][0];
					}
				}
#pragma unroll
				for (int i = 0; i < LW; ++i)
				{
					*reinterpret_cast<u32x4*>(ws + (set & 1) * (BN * kTileK) + (row + kRowStep * i) * kTileK + slot) = rw[set][i];
				}
			};

			floatx4 acc[TN][TM];
#pragma unroll
			for (int a = 0; a < TN; ++a)
			{
#pragma unroll
				for (int b = 0; b < TM; ++b)
				{
					acc[a][b] = floatx4{ 0.0f, 0.0f, 0.0f, 0.0f };
				}
			}
			const auto multiply = [&](int buf) {
#pragma unroll
				for (int ks = 0; ks < 2; ++ks)
				{
					bf16x8 wf[TN], xf[P][TM];
#pragma unroll
					for (int a = 0; a < TN; ++a)
					{
						const int r = wn * (BN / WN) + 16 * a + j;
						wf[a] = *reinterpret_cast<const bf16x8*>(ws + buf * (BN * kTileK) + r * kTileK + (((4 * ks + g) ^ (r & 7)) * 8));
					}
#pragma unroll
					for (int b = 0; b < TM; ++b)
					{
						const int r = wm * (BM / WM) + 16 * b + j;
#pragma unroll
						for (int p = 0; p < P; ++p)
						{
							xf[p][b] = *reinterpret_cast<const bf16x8*>(xs + (buf * P + p) * (BM * kTileK) + r * kTileK + (((4 * ks + g) ^ (r & 7)) * 8));
						}
					}
#pragma unroll
					for (int p = P - 1; p >= 0; --p) // small parts first
					{
#pragma unroll
						for (int a = 0; a < TN; ++a)
						{
#pragma unroll
							for (int b = 0; b < TM; ++b)
							{
								acc[a][b] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wf[a], xf[p][b], acc[a][b], 0, 0, 0);
							}
						}
					}
				}
			};
			// past the last tile it is requested and staged again: a branch around the loads would make every
			// wait behind it a wait for all of them
#pragma unroll
			for (int t = 0; t < S; ++t)
			{
				request(walk.tile(t), t);
			}
			stage(walk.tile(0), 0);
			__syncthreads();
			// tile `step` is in LDS, the S - 1 behind it in their register sets
			const auto advance = [&](int step, int set) {
				request(walk.tile(step + S), set);
				if constexpr (BM * BN < 128 * 128 && !F32)
				{
					// on their way before the products, not behind them (the largest tile, whose products take
					// longer than the loads, runs better scheduled freely)
					__builtin_amdgcn_sched_barrier(0);
				}
				if (KG == 1 || walk.multiplies(step))
				{
					multiply(set & 1);
				}
				stage(walk.tile(step + 1), (set + 1) % S);
				__syncthreads();
			};
			int step = 0;
			for (; step + S <= walk.rounds; step += S)
			{
#pragma unroll
				for (int t = 0; t < S; ++t)
				{
					advance(step + t, t);
				}
			}
#pragma unroll
			for (int t = 0; t < S - 1; ++t)
			{
				if (step + t < walk.rounds)
				{
					advance(step + t, t);
				}
			}
			if constexpr (KG > 1)
			{
				floatx4* const handed = reinterpret_cast<floatx4*>(tile_lds);
				if (group > 0)
				{
#pragma unroll
					for (int a = 0; a < TN; ++a)
					{
#pragma unroll
						for (int b = 0; b < TM; ++b)
						{
							handed[((group - 1) * (WM * WN) + wave) * (TN * TM * 64) + (a * TM + b) * 64 + lane] = acc[a][b];
						}
					}
				}
				__syncthreads();
				if (group > 0)
				{
					return;
				}
#pragma unroll
				for (int other = 0; other < KG - 1; ++other)
				{
#pragma unroll
					for (int a = 0; a < TN; ++a)
					{
#pragma unroll
						for (int b = 0; b < TM; ++b)
						{
							acc[a][b] += handed[(other * (WM * WN) + wave) * (TN * TM * 64) + (a * TM + b) * 64 + lane];
						}
					}
				}
			}
#pragma unroll
			for (int b = 0; b < TM; ++b)
			{
				const int m = m0 + wm * (BM / WM) + 16 * b + j;
#pragma unroll
				for (int a = 0; a < TN; ++a)
				{
					store_outputs<operand>(d, m, n0 + wn * (BN / WN) + 16 * a + 4 * g, acc[a][b]);
				}
			}
		}

		// ------------------------------------------------------------------
		// The same product of bfloat16 operands that lie on 16 bytes: tiles of K go from memory into a ring of S buffers in LDS
		// directly (global_load_lds_dwordx4: 8 rows of 128 bytes at a time, lane l fills bytes 16 l, so it is the address that
		// is permuted), and a wavefront's fragments of half a tile are read while the other half is multiplied.  One barrier a
		// tile, in its middle: behind it the next tile is there and this one's buffer is free.  Outputs are the chains of
		// products over K that dense_tile_kernel forms, bit for bit.
		//
		// What bounds it: small tiles, the rate at which a CU takes operands from L2 (70 to 80 GB/s a CU, about 30 bytes a cycle; a
		// ring twice as deep changes nothing), and a tenth or two for weights that come from HBM (a wavefront that touches
		// them ahead of the others costs more than that); large ones, the products (256 x 256 on 2048 x 28672 x 4096: 1040 TFLOP/s
		// with the weights from HBM, 1125 without).
		// ------------------------------------------------------------------
		template <int BM, int BN, int WM, int WN, int S>
		__global__ __launch_bounds__(64 * WM * WN, 2) void dense_ring_kernel(const TileArgs args)
		{
			constexpr int W = WM * WN, TM = BM / WM / 16, TN = BN / WN / 16;
			constexpr int kRowBytes = 2 * kTileK, kStage = (BM + BN) * kRowBytes; // [BM activations, BN weights][64]
			constexpr int LA = BM / 8 / W, LW = BN / 8 / W, L = LA + LW;         // 1 KB pieces a wavefront moves per tile
			static_assert(LA * 8 * W == BM && LW * 8 * W == BN && TM * WM * 16 == BM && TN * WN * 16 == BN, "tile");
			static_assert((S - 1) * L < 64 && S <= fetch::kDenseMaxBuffers, "loads that a wait can count");
			extern __shared__ __attribute__((aligned(16))) uint8_t ring_lds[];
			const DenseRows& d = args.d;
			int tm, tn;
			if (!tile_of(args, tm, tn))
			{
				return;
			}
			const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
			const int j = lane & 15, g = lane >> 4;
			const int wm = wave / WN, wn = wave % WN;
			const int m0 = tm * BM, n0 = tn * BN;
			const fetch::DenseWalk walk = fetch::dense_walk(d.w.pitch / kTileK, d.splits, 1, static_cast<int>(blockIdx.y), 0);

			// piece i of a wavefront: rows 8 (i W + wave) .. + 7 of the activations, then of the weights
			uint32_t from[L];
			{
				const int row = lane >> 3, at = ((lane & 7) ^ row) * 16;
#pragma unroll
				for (int i = 0; i < LA; ++i)
				{
					from[i] = static_cast<uint32_t>(operand_row(d, m0 + 8 * (i * W + wave) + row)) * static_cast<uint32_t>(2 * d.lda) + at;
				}
#pragma unroll
				for (int i = 0; i < LW; ++i)
				{
					from[LA + i] = static_cast<uint32_t>(min(n0 + 8 * (i * W + wave) + row, d.w.n - 1)) * static_cast<uint32_t>(2 * d.w.pitch) + at;
				}
			}
			const uint32_t lds_base = static_cast<uint32_t>(reinterpret_cast<uintptr_t>((__attribute__((address_space(3))) const uint8_t*)(ring_lds)));
			const auto request = [&](int step, int buffer) {
				const size_t k_bytes = static_cast<size_t>(walk.tile(step)) * kRowBytes;
				const uint8_t* const a = static_cast<const uint8_t*>(d.a) + k_bytes;
				const uint8_t* const w = reinterpret_cast<const uint8_t*>(d.w.w) + k_bytes;
				const uint32_t to = lds_base + buffer * kStage + wave * 1024;
#pragma unroll
				for (int i = 0; i < L; ++i)
				{
#pragma clang diagnostic push
#pragma clang diagnostic ignored "-Winline-asm" // m0 is named as clobbered although it is reserved
					asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2"
					             :
					             : "s"(to + i * (W * 1024)), "v"(from[i]), "s"(i < LA ? a : w)
					             : "memory", "m0");
#pragma clang diagnostic pop
				}
			};
			// this lane's piece of the first fragment, by half of the tile
			const uint8_t* x_at[2];
			const uint8_t* w_at[2];
#pragma unroll
			for (int ks = 0; ks < 2; ++ks)
			{
				const int piece = ((4 * ks + g) ^ (j & 7)) * 16;
				x_at[ks] = ring_lds + (wm * (BM / WM) + j) * kRowBytes + piece;
				w_at[ks] = ring_lds + (BM + wn * (BN / WN) + j) * kRowBytes + piece;
			}
			bf16x8 wf[2][TN], xf[2][TM];
			const auto read = [&](int ks, int buffer) {
#pragma unroll
				for (int a = 0; a < TN; ++a)
				{
					wf[ks][a] = *reinterpret_cast<const bf16x8*>(w_at[ks] + buffer * kStage + a * (16 * kRowBytes));
				}
#pragma unroll
				for (int b = 0; b < TM; ++b)
				{
					xf[ks][b] = *reinterpret_cast<const bf16x8*>(x_at[ks] + buffer * kStage + b * (16 * kRowBytes));
				}
			};
			floatx4 acc[TN][TM];
#pragma unroll
			for (int a = 0; a < TN; ++a)
			{
#pragma unroll
				for (int b = 0; b < TM; ++b)
				{
					acc[a][b] = floatx4{ 0.0f, 0.0f, 0.0f, 0.0f };
				}
			}
			const auto multiply = [&](int ks) {
#pragma unroll
				for (int a = 0; a < TN; ++a)
				{
#pragma unroll
					for (int b = 0; b < TM; ++b)
					{
						acc[a][b] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wf[ks][a], xf[ks][b], acc[a][b], 0, 0, 0);
					}
				}
			};
			// behind the k-th activation there may be anything: the last tile's is zeroed once it is there
			const int last_tile = d.w.pitch / kTileK - 1, last_valid = d.w.k - last_tile * kTileK;
			const auto trim = [&](int step, int buffer) {
				if (last_valid == kTileK || step >= walk.rounds || walk.tile(step) != last_tile)
				{
					return;
				}
				for (int i = threadIdx.x; i < BM * 8; i += 64 * W)
				{
					const int row = i >> 3, left = last_valid - 8 * ((i & 7) ^ (row & 7));
					uint16_t* const piece = reinterpret_cast<uint16_t*>(ring_lds + buffer * kStage + i * 16);
					for (int e = max(left, 0); e < 8; ++e)
					{
						piece[e] = 0;
					}
				}
				__syncthreads();
			};
#pragma unroll
			for (int t = 0; t < S; ++t)
			{
				request(t, t); // (past the range's last tile that one comes again: every wait counts the same)
			}
			// all but the last N pieces have arrived, this wavefront's reads too; then the others say the same
			asm volatile("s_waitcnt vmcnt(%0)\n\ts_barrier" ::"n"((S - 1) * L) : "memory");
			trim(0, 0);
			read(0, 0);
			int buffer = 0;
			for (int step = 0; step < walk.rounds; ++step)
			{
				read(1, buffer);
				__builtin_amdgcn_sched_barrier(0);
				multiply(0);
				__builtin_amdgcn_sched_barrier(0);
				asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"((S - 2) * L) : "memory");
				request(step + S, buffer);
				buffer = buffer == S - 1 ? 0 : buffer + 1;
				trim(step + 1, buffer);
				read(0, buffer);
				__builtin_amdgcn_sched_barrier(0);
				multiply(1);
				__builtin_amdgcn_sched_barrier(0);
			}
			asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)" ::: "memory"); // (nothing may arrive in LDS that is another workgroup's)
#pragma unroll
			for (int b = 0; b < TM; ++b)
			{
				const int m = m0 + wm * (BM / WM) + 16 * b + j;
#pragma unroll
				for (int a = 0; a < TN; ++a)
				{
					store_outputs<uint16_t>(d, m, n0 + wn * (BN / WN) + 16 * a + 4 * g, acc[a][b]);
				}
			}
		}

		constexpr size_t kRowLdsLimit = 152 * 1024;

		size_t row_lds_bytes(int pitch, int& groups)
		{
			groups = (pitch + kFlight * kRowBlock - 1) / (kFlight * kRowBlock);
			return sizeof(float) * static_cast<size_t>(groups) * kFlight * kRowBlock;
		}

		template <int R>
		void launch_row(const RowArgs& args, size_t lds, hipStream_t s)
		{
			const int waves = (args.d.w.n + R - 1) / R;
			const int cap = lds > 72 * 1024 ? 256 : 512;
			const int rounds = (waves + cap * kRowWaves - 1) / (cap * kRowWaves);
			const int blocks = (waves + rounds * kRowWaves - 1) / (rounds * kRowWaves);
			allow_dynamic_lds(reinterpret_cast<const void*>(&dense_row_kernel<R>), kRowLdsLimit);
			dense_row_kernel<R><<<dim3(blocks), dim3(kRowThreads), lds, s>>>(args);
		}

		template <int BM, int BN, int WM, int WN, int KG, int S, bool F32>
		void launch_tile(TileArgs& args, hipStream_t s)
		{
			constexpr size_t lds = sizeof(uint16_t) * KG * 2 * kTileK * ((F32 ? 3 : 1) * BM + BN);
			static_assert(lds <= 160 * 1024 && sizeof(float) * (KG - 1) * BM * BN <= lds, "LDS");
			allow_dynamic_lds(reinterpret_cast<const void*>(&dense_tile_kernel<BM, BN, WM, WN, KG, S, F32>), lds);
			args.m_tiles = (args.d.m + BM - 1) / BM;
			args.n_tiles = (args.d.w.n + BN - 1) / BN;
			const int per = (args.m_tiles * args.n_tiles + 7) / 8;
			dense_tile_kernel<BM, BN, WM, WN, KG, S, F32><<<dim3(8 * per, args.d.splits), dim3(64 * WM * WN * KG), lds, s>>>(args);
		}

		template <int BM, int BN, int WM, int WN, int S>
		void launch_ring(TileArgs& args, hipStream_t s)
		{
			constexpr size_t lds = static_cast<size_t>(S) * (BM + BN) * kTileK * sizeof(uint16_t);
			static_assert(lds <= 160 * 1024, "LDS");
			allow_dynamic_lds(reinterpret_cast<const void*>(&dense_ring_kernel<BM, BN, WM, WN, S>), lds);
			args.m_tiles = (args.d.m + BM - 1) / BM;
			args.n_tiles = (args.d.w.n + BN - 1) / BN;
			const int per = (args.m_tiles * args.n_tiles + 7) / 8;
			dense_ring_kernel<BM, BN, WM, WN, S><<<dim3(8 * per, args.d.splits), dim3(64 * WM * WN), lds, s>>>(args);
		}

		int tiles(const DenseRows& d, int bm, int bn) { return ((d.m + bm - 1) / bm) * ((d.w.n + bn - 1) / bn); }
	} // namespace

	int dense_rows_splits(const DenseMatrix& w, int m, bool f32)
	{
		return f32 ? fetch::dense_f32_ranges(w.n, w.pitch / kTileK, m) : fetch::dense_ranges(w.n, w.pitch / kTileK, m);
	}

	size_t dense_row_max_k() { return kRowLdsLimit / sizeof(float) / (kFlight * kRowBlock) * (kFlight * kRowBlock); }

	bool launch_dense_row(const DenseRow& a, hipStream_t s)
	{
		if (a.w.n <= 0)
		{
			return true;
		}
		RowArgs args{ a, 0 };
		const size_t lds = row_lds_bytes(a.w.pitch, args.groups);
		if (lds > kRowLdsLimit)
		{
			return false;
		}
		// enough wavefronts to cover the card matters more than rows per wavefront
		if (a.glu || a.w.n >= 2048)
		{
			launch_row<2>(args, lds, s);
		}
		else
		{
			launch_row<1>(args, lds, s);
		}
		return true;
	}

	void launch_dense_rows(const DenseRows& a, hipStream_t s)
	{
		if (a.m <= 0 || a.w.n <= 0)
		{
			return;
		}
		TileArgs args{ a, 0, 0 };
		const auto work = [&](int bm, int bn) { return tiles(a, bm, bn) * a.splits; };
		if (a.f32)
		{
			switch (fetch::dense_f32_form(a.w.n, a.m, a.splits))
			{
			case fetch::kF32Chain64x128: return launch_tile<64, 128, 2, 4, 1, 2, true>(args, s);
			case fetch::kF32Chain64x256: return launch_tile<64, 256, 2, 4, 1, 2, true>(args, s);
			case fetch::kF32Halves64x128: return launch_tile<64, 128, 2, 4, 2, 2, true>(args, s);
			case fetch::kF32Halves64x64: return launch_tile<64, 64, 2, 4, 2, 2, true>(args, s);
			default: return launch_tile<32, 64, 1, 4, 2, 2, true>(args, s);
			}
		}
		// us, weights from HBM, for 256 x 256, 128 x 256, 192 x 128 (three buffers), 128 x 192, 128 x 128 (three), 128 x 64, 64 x 128,
		// 64 x 64, 32 x 64, 32 x 32 and the best of dense_tile_kernel: 2048 x 28672 x 4096 451, 468, 523, 529, 573, 650, 670, more, more, more and 528;
		// 639 x 4096 x 14336 313, 195, 151, 161, 133, 162, 169, 162, 196, 254 and 136; 777 x 2048 x 5632 132, 79, 63, 64, 50, 39, 42, 46,
		// 62, 71 and 44; 320 x 6160 x 2048 58, 35, 29, 30, 24, 28, 21, 24, 30, 39 and 22; 33 x 4096 x 14336 in four ranges 80, 52, 43, 42,
		// 35, 29, 32, 23, 29, 34 and 24; 17 x 13888 x 4096 90, 58, 47, 46, 38, 32, 35, 27, 26, 26 and 26.  Two buffers instead of
		// three: 1280 x 6432 x 2048 128 x 128 40 and 52, 192 x 128 46 (777 x 11264 x 2048 49 and 57).
		const auto on16 = [](const void* p) { return reinterpret_cast<uintptr_t>(p) % 16 == 0; };
		const auto reach = [](size_t rows, size_t pitch) { return rows * pitch * sizeof(uint16_t) <= 0xffffffffu; }; // 32-bit offsets
		if (on16(a.a) && on16(a.w.w) && a.lda % 8 == 0 && reach(std::max(a.m, a.a_ring), a.lda) && reach(a.w.n, a.w.pitch))
		{
			switch (fetch::dense_form(a.w.n, a.w.pitch / kTileK, a.m, a.splits))
			{
			case fetch::kDense256x256: return launch_ring<256, 256, 2, 4, 2>(args, s);
			case fetch::kDense128x256: return launch_ring<128, 256, 2, 4, 3>(args, s);
			case fetch::kDense192x128: return launch_ring<192, 128, 4, 2, 2>(args, s);
			case fetch::kDense192x128x3: return launch_ring<192, 128, 4, 2, 3>(args, s);
			case fetch::kDense128x192: return launch_ring<128, 192, 2, 4, 3>(args, s);
			case fetch::kDense128x128: return launch_ring<128, 128, 4, 2, 2>(args, s);
			case fetch::kDense128x128x3: return launch_ring<128, 128, 4, 2, 3>(args, s);
			case fetch::kDense128x64: return launch_ring<128, 64, 4, 2, 3>(args, s);
			case fetch::kDense64x128: return launch_ring<64, 128, 2, 4, 3>(args, s);
			case fetch::kDense64x64: return launch_ring<64, 64, 2, 2, 4>(args, s);
			case fetch::kDense32x64: return launch_ring<32, 64, 1, 4, 6>(args, s);
			default: return launch_ring<32, 32, 2, 2, 8>(args, s);
			}
		}
		// A K step of a form costs so many ns where a CU has r workgroups of it, fitted over 2048 x 5632, 4096 x 14336, 11264 x
		// 2048, 6432 x 2048 and 6144 x 4096 at 30 to 1254 rows; the form with the least is the fastest of eleven, or within 5 % of
		// it, at all of these (us for 128 x 128, 64 x 128, 64 x 64, 32 x 64: 2048 x 5632 at 777 rows 48, 40, 41, 51, at 500 rows
		// 48, 39, 26, 32; 11264 x 2048 at 777 rows 58, 66, 75, 92, at 30 rows 23, 19, 13, 13).  The small tiles, taken where a CU
		// has one or two, wait for memory: four tiles of K on their way instead of two make 6144 x 4096 27 -> 21 us at 100 rows,
		// 26 -> 19 at 30.
		const auto cost = [&](int bm, int bn, int fixed, int per) { return fixed + per * ((work(bm, bn) + 255) / 256); };
		const int c128 = cost(128, 128, 0, 570), c64 = cost(64, 128, 60, 360), c64n = cost(64, 64, 50, 220), c32 = cost(32, 64, 60, 140);
		const int least = std::min({ c128, c64, c64n, c32 });
		if (c128 == least)
		{
			launch_tile<128, 128, 4, 2, 1, 2, false>(args, s);
		}
		else if (c64 == least)
		{
			launch_tile<64, 128, 2, 4, 1, 2, false>(args, s);
		}
		else if (c64n == least)
		{
			launch_tile<64, 64, 2, 4, 1, 4, false>(args, s);
		}
		else
		{
			launch_tile<32, 64, 1, 4, 1, 4, false>(args, s);
		}
	}
} // namespace litenn_hip
