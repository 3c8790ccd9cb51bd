// Quantised matmul of several activation rows with Float32 operands on the matrix cores:
//   Y[M, N] = X[M, K] . deq(W)[N, K]^T  (+ residual)
// with the accuracy of the Float32 streaming kernel (csrc/gemv.hip), which would read the weights once
// per row.  No operand is rounded to 16 bits:
//
//   * A GGUF weight is a small integer times a scale.  The integers (or, for the K-quants with six-bit
//     sub-scales, integer times sub-scale: at most 63 * 16 and some) are exact in binary16 and are what
//     the matrix cores multiply; the block's Float32 scale is applied to the Float32 sum of its
//     products.
//   * An activation is scaled by a power of two (per row, for few rows per row and 256 elements) to at most 2^15 and
//     taken apart into two binary16 values, hi = half(x) and lo = half(4096 (x - hi)): off by 2^-24 of itself at most down
//     to 2^-28 of the largest, by 2^-52 of that below.  Both are multiplied by the integers, lo by the integers / 4096
//     (exact as well), and accumulate in the same Float32 registers.
//   * The minimum term of Q4_K and Q5_K, dmin * sum_j m_j (sum of sub-block j's activations), is one
//     more product per 256 elements: the eight sums, taken apart the same way, against the eight
//     six-bit minima.
//
// Against 64 bits the result is closer than the streaming kernel's in every format and form (relative L2 over K = 256 ..
// 14336, mean of six inputs, 0.7e-7 to 1.2e-7; the streaming kernel 0.9e-7 to 2.5e-7).
//
// What bounds it: few rows are the weights' stream and the launch; many rows, no unit alone (the forms below say more).  Row by
// row through the streaming kernel the same calls took, us, before -> now with the rows' pre-pass: Q6_K 4096 x 14336 at 45 rows
// 571 -> 43; 8B-shape prompt of 300 tokens, two blocks 28100 -> 650.
//
// v_mfma_f32_32x32x16_f16 but for few rows: D[i][j] += A[i][k] B[k][j] with the activations as A and the
// weights as B, so that a lane's sixteen results belong to one weight row, whose scale the lane holds.
#include "common.hpp"
#include "fetch_model.hpp"

#include <algorithm>

namespace litenn_hip
{
	namespace
	{
		typedef _Float16 half8 __attribute__((ext_vector_type(8)));
		typedef _Float16 half4 __attribute__((ext_vector_type(4)));
		typedef _Float16 half2v __attribute__((ext_vector_type(2)));
		typedef float floatx4 __attribute__((ext_vector_type(4)));
		typedef floatx4 floatx4_a4 __attribute__((aligned(4)));
		typedef float floatx16 __attribute__((ext_vector_type(16)));
		typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
		typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));

		constexpr int kTile = 32;     // activation rows and weight rows of one product
		constexpr int kChunk = 256;   // K elements of the outer loop's step: four stages of four MFMA steps
		constexpr int kFrag = 1024;   // bytes of an operand fragment: 64 lanes x 8 halves
		constexpr int kStageBytes = 8 * kFrag;           // one tile, 64 elements: (hi, lo) x 4 steps
		constexpr int kTileChunkBytes = 4 * kStageBytes; // one tile, 256 elements
		constexpr float kSumScale = 1.0f / 64.0f; // sums of 32 activations back into the binary16 range
		constexpr float kLowScale = 1.0f / 4096.0f; // of the low parts: small activations beside a large one keep their bits

		// ---- weight blocks -> binary16 integers -------------------------------------------------------
		// A wavefront copies the raw blocks of its 32 rows for one 256-element chunk into a slot of its own in
		// LDS, 16-byte pieces in a row's order (eight neighbouring lanes fetch one 128-byte line; a lane that
		// fetched its own row's bytes instead took 29 us for Q8_0 4096 x 4096, most of it in the vector memory
		// path).  From there lane (r, h) = (lane % 32, lane / 32) takes, of weight row r, elements 16 s + 8 h .. + 7
		// of step s (K in natural order).  A stage is 64 elements = steps 0..3.  Blocks are only 2-byte aligned.
		typedef const __attribute__((address_space(3))) uint8_t* lds_bytes_t;
		// `p` is on 8 bytes and `at` a constant once unrolled: LDS reads off their alignment are served lane by lane, which
		// was most of the time of Q6_K's and Q8_0's matmuls, so what lies on 2 bytes is put together from dwords
		__device__ __forceinline__ u32x2 load8(lds_bytes_t p, int at)
		{
			typedef const __attribute__((address_space(3))) uint32_t* words_t;
			if (at % 8 == 0)
			{
				return *(const __attribute__((address_space(3))) u32x2*)(p + at);
			}
			if (at % 4 == 0)
			{
				const words_t w = (words_t)(p + at);
				return { w[0], w[1] };
			}
			const words_t w = (words_t)(p + at - 2);
			return { __builtin_amdgcn_alignbit(w[1], w[0], 16), __builtin_amdgcn_alignbit(w[2], w[1], 16) };
		}
		__device__ __forceinline__ u32x4 load16(lds_bytes_t p) { return *(const __attribute__((address_space(3))) u32x4*)(p); }
		__device__ __forceinline__ uint32_t load2(lds_bytes_t p) { return *(const __attribute__((address_space(3))) uint16_t*)(p); }

		__device__ __forceinline__ half2v as_half2(uint32_t v) { return __builtin_bit_cast(half2v, v); }

		// bytes 0, 1 and 2, 3 of v as the halves 1024 + byte (0x6400 | byte)
		__device__ __forceinline__ half2v biased01(uint32_t v) { return as_half2(__builtin_amdgcn_perm(0x64646464u, v, 0x04010400u)); }
		__device__ __forceinline__ half2v biased23(uint32_t v) { return as_half2(__builtin_amdgcn_perm(0x64646464u, v, 0x04030402u)); }

		// the factors of the low parts
		__device__ __forceinline__ half8 lowered(half8 v) { return v * static_cast<_Float16>(kLowScale); }
		// factors of sub-block sums: lanes (r, 0) hold those of the high parts, lanes (r, 1) of the low ones
		__device__ __forceinline__ half8 for_sums(half8 v, int h) { return v * static_cast<_Float16>(h ? kLowScale : 1.0f); }

		__device__ __forceinline__ half8 join(half2v a, half2v b, half2v c, half2v d)
		{
			return half8{ a.x, a.y, b.x, b.y, c.x, c.y, d.x, d.y };
		}
		// eight unsigned bytes minus `bias`
		__device__ __forceinline__ half8 bytes_minus(uint32_t a, uint32_t b, float bias)
		{
			const _Float16 m = static_cast<_Float16>(-1024.0f - bias);
			const half2v off = { m, m };
			return join(biased01(a) + off, biased23(a) + off, biased01(b) + off, biased23(b) + off);
		}
		// Integer q times sub-scale s, less about kCentre s: (1024 + q) s + off with off = -(1024 + centre) s rounded to a half,
		// fused.  What is taken off is the integer -off - 1024 s = centred_by, exactly.
		__device__ __forceinline__ half2v centre_offset(half2v s, float centre)
		{
			const _Float16 m = static_cast<_Float16>(-1024.0f - centre);
			return s * half2v{ m, m };
		}
		__device__ __forceinline__ half2v centred_by(half2v s, float centre)
		{
			return -__builtin_elementwise_fma(s, half2v{ 1024, 1024 }, centre_offset(s, centre));
		}
		// eight unsigned bytes (at most 31) times the integer `scale` (at most 63), centred
		__device__ __forceinline__ half8 bytes_times(uint32_t a, uint32_t b, uint32_t scale, float centre)
		{
			const half2v s = as_half2(0x64006400u | (scale * 0x00010001u)) - half2v{ 1024, 1024 };
			const half2v off = centre_offset(s, centre);
			return join(__builtin_elementwise_fma(biased01(a), s, off), __builtin_elementwise_fma(biased23(a), s, off),
			            __builtin_elementwise_fma(biased01(b), s, off), __builtin_elementwise_fma(biased23(b), s, off));
		}
		// what that took off, for the eight scales a, b, as the factors of sums times kSumScale (at most 960 * 64: a half)
		__device__ __forceinline__ half8 centres(uint32_t a, uint32_t b, float centre)
		{
			const half2v off = { -1024, -1024 };
			const _Float16 f = static_cast<_Float16>(1.0f / kSumScale);
			return half8{ f, f, f, f, f, f, f, f } * join(centred_by(biased01(a) + off, centre), centred_by(biased23(a) + off, centre), centred_by(biased01(b) + off, centre),
			            centred_by(biased23(b) + off, centre));
		}

		// Formats:
		//   kBlock        elements of a block, kChunkBytes bytes of 256 elements
		//   kScaleSteps   steps whose products share one scale: after them the sum is scaled and added
		//   Head          what the lane needs of the chunk as a whole
		//   kMins         whether a minimum term follows each chunk.  The integers are then taken about kCentre, the middle of
		//                 their range, lower, and what that takes from the sum is added back per chunk, a product more over the
		//                 sub-blocks' sums, together with the minima, much of which it cancels: the sums on the way stay as small
		//                 as the result (relative error at Q5_K, 33 rows of 2048, 1.66e-7 without it)
		// Rows whose last chunk is not whole (blocks of 32 only) load their last block again in the missing blocks'
		// places and scale it by 0 (`blocks` whole blocks of the chunk are there).
		struct Q4_0X
		{
			static constexpr int kBlock = 32, kChunkBytes = 8 * 18, kScaleSteps = 2;
			static constexpr bool kMins = false;
			struct Head {};
			struct Raw { u32x2 q[2]; uint32_t d[2]; };
			static __device__ __forceinline__ Head head(lds_bytes_t, int) { return {}; }
			static __device__ __forceinline__ Raw load(lds_bytes_t chunk, int st, int h, int blocks)
			{
				Raw r;
#pragma unroll
				for (int b = 0; b < 2; ++b)
				{
					const int block = 2 * st + b;
					const uint32_t d = load2(chunk + 18 * block); // (there, whatever it is: not a branch)
					r.d[b] = block < blocks ? d : 0u;
					r.q[b] = load8(chunk + 8 * h, 18 * block + 2);
				}
				return r;
			}
			static __device__ __forceinline__ half8 frag(const Head&, const Raw& r, int, int t)
			{
				const u32x2 q = r.q[t >> 1];
				const int sh = 4 * (t & 1);
				return bytes_minus((q.x >> sh) & 0x0f0f0f0fu, (q.y >> sh) & 0x0f0f0f0fu, 8.0f);
			}
			static __device__ __forceinline__ float scale(const Head&, const Raw& r, int, int t) { return f16_bits_to_f32(r.d[t >> 1]); }
			static __device__ __forceinline__ float chunk_scale(const Head&) { return 1.0f; }
		};

		struct Q8_0X
		{
			static constexpr int kBlock = 32, kChunkBytes = 8 * 34, kScaleSteps = 2;
			static constexpr bool kMins = false;
			struct Head {};
			struct Raw { u32x2 q[4]; uint32_t d[2]; };
			static __device__ __forceinline__ Head head(lds_bytes_t, int) { return {}; }
			static __device__ __forceinline__ Raw load(lds_bytes_t chunk, int st, int h, int blocks)
			{
				Raw r;
#pragma unroll
				for (int b = 0; b < 2; ++b)
				{
					const int block = 2 * st + b;
					const uint32_t d = load2(chunk + 34 * block); // (there, whatever it is: not a branch)
					r.d[b] = block < blocks ? d : 0u;
					r.q[2 * b] = load8(chunk + 8 * h, 34 * block + 2);
					r.q[2 * b + 1] = load8(chunk + 8 * h, 34 * block + 18);
				}
				return r;
			}
			static __device__ __forceinline__ half8 frag(const Head&, const Raw& r, int, int t)
			{
				return bytes_minus(r.q[t].x ^ 0x80808080u, r.q[t].y ^ 0x80808080u, 128.0f);
			}
			static __device__ __forceinline__ float scale(const Head&, const Raw& r, int, int t) { return f16_bits_to_f32(r.d[t >> 1]); }
			static __device__ __forceinline__ float chunk_scale(const Head&) { return 1.0f; }
		};

		struct Q4_KX
		{
			static constexpr int kBlock = 256, kChunkBytes = 144, kScaleSteps = 16;
			static constexpr bool kMins = true;
			static constexpr float kCentre = 8.0f;
			struct Head { u32x4 w; }; // d, dmin, 12 bytes of six-bit scales and minima
			struct Raw { u32x2 q[2]; };
			static __device__ __forceinline__ Head head(lds_bytes_t chunk, int) { return { load16(chunk) }; }
			static __device__ __forceinline__ Raw load(lds_bytes_t chunk, int st, int h, int)
			{
				lds_bytes_t p = chunk + 16 + 32 * st + 8 * h;
				return { { load8(p, 0), load8(p, 16) } };
			}
			// get_scale_min_k4 of the ggml block definition, four sub-blocks to a dword
			static __device__ __forceinline__ uint32_t scales(const u32x4& w, int four)
			{
				return four == 0 ? w.y & 0x3f3f3f3fu : (w.w & 0x0f0f0f0fu) | ((w.y >> 2) & 0x30303030u);
			}
			static __device__ __forceinline__ uint32_t minima(const u32x4& w, int four)
			{
				return four == 0 ? w.z & 0x3f3f3f3fu : ((w.w >> 4) & 0x0f0f0f0fu) | ((w.z >> 2) & 0x30303030u);
			}
			// steps 0, 1: low nibbles (sub-block 2 st); steps 2, 3: high nibbles (2 st + 1)
			static __device__ __forceinline__ half8 frag(const Head& hd, const Raw& r, int st, int t)
			{
				const int sh = 4 * (t >> 1), sub = 2 * st + (t >> 1);
				const uint32_t s = (scales(hd.w, sub >> 2) >> (8 * (sub & 3))) & 0xffu;
				const u32x2 q = r.q[t & 1];
				return bytes_times((q.x >> sh) & 0x0f0f0f0fu, (q.y >> sh) & 0x0f0f0f0fu, s, kCentre);
			}
			static __device__ __forceinline__ float scale(const Head&, const Raw&, int, int) { return 1.0f; }
			static __device__ __forceinline__ float chunk_scale(const Head& hd) { return f16_bits_to_f32(hd.w.x); }
			// element l of sub-block j
			static __device__ __forceinline__ int code(const uint8_t* block, int j, int l)
			{
				return (block[16 + (j >> 1) * 32 + l] >> (4 * (j & 1))) & 15;
			}
			static __device__ __forceinline__ half8 min_frag(const Head& hd) { return bytes_minus(minima(hd.w, 0), minima(hd.w, 1), 0.0f); }
			static __device__ __forceinline__ half8 centre_frag(const Head& hd) { return centres(scales(hd.w, 0), scales(hd.w, 1), kCentre); }
			static __device__ __forceinline__ float min_scale(const Head& hd) { return -f16_bits_to_f32(hd.w.x >> 16); }
		};

		struct Q5_KX
		{
			static constexpr int kBlock = 256, kChunkBytes = 176, kScaleSteps = 16;
			static constexpr bool kMins = true;
			static constexpr float kCentre = 15.0f; // (1040 * 63 is no half)
			struct Head { u32x4 w; u32x2 fifth[2]; };
			struct Raw { u32x2 q[2]; };
			static __device__ __forceinline__ Head head(lds_bytes_t chunk, int h)
			{
				return { load16(chunk), { load8(chunk + 8 * h, 16), load8(chunk + 8 * h, 32) } };
			}
			static __device__ __forceinline__ Raw load(lds_bytes_t chunk, int st, int h, int)
			{
				lds_bytes_t p = chunk + 48 + 32 * st + 8 * h;
				return { { load8(p, 0), load8(p, 16) } };
			}
			static __device__ __forceinline__ half8 frag(const Head& hd, const Raw& r, int st, int t)
			{
				const int sh = 4 * (t >> 1), sub = 2 * st + (t >> 1);
				const uint32_t s = (Q4_KX::scales(hd.w, sub >> 2) >> (8 * (sub & 3))) & 0xffu;
				const u32x2 q = r.q[t & 1], f = hd.fifth[t & 1]; // bit `sub` of a byte is its element's fifth bit
				return bytes_times(((q.x >> sh) & 0x0f0f0f0fu) | (((f.x >> sub) & 0x01010101u) << 4),
				                   ((q.y >> sh) & 0x0f0f0f0fu) | (((f.y >> sub) & 0x01010101u) << 4), s, kCentre);
			}
			static __device__ __forceinline__ float scale(const Head&, const Raw&, int, int) { return 1.0f; }
			static __device__ __forceinline__ float chunk_scale(const Head& hd) { return f16_bits_to_f32(hd.w.x); }
			static __device__ __forceinline__ int code(const uint8_t* block, int j, int l)
			{
				return ((block[48 + (j >> 1) * 32 + l] >> (4 * (j & 1))) & 15) | ((block[16 + l] >> j) & 1) << 4;
			}
			static __device__ __forceinline__ half8 min_frag(const Head& hd)
			{
				return bytes_minus(Q4_KX::minima(hd.w, 0), Q4_KX::minima(hd.w, 1), 0.0f);
			}
			static __device__ __forceinline__ half8 centre_frag(const Head& hd) { return centres(Q4_KX::scales(hd.w, 0), Q4_KX::scales(hd.w, 1), kCentre); }
			static __device__ __forceinline__ float min_scale(const Head& hd) { return -f16_bits_to_f32(hd.w.x >> 16); }
		};

		struct Q6_KX
		{
			// six bits and a signed byte of sub-scale per 16 elements: their product does not fit a half, so every
			// step is scaled on its own
			static constexpr int kBlock = 256, kChunkBytes = 210, kScaleSteps = 1;
			static constexpr bool kMins = false;
			struct Head { u32x4 sc; uint32_t d; };
			struct Raw { u32x2 low[4], high[2]; }; // half st / 2 of the block: [32 x (first, second)] x 16-element runs
			static __device__ __forceinline__ Head head(lds_bytes_t chunk, int) { return { load16(chunk + 192), load2(chunk + 222) }; } // (the last piece ends with the block)
			static __device__ __forceinline__ Raw load(lds_bytes_t chunk, int st, int h, int)
			{
				lds_bytes_t ql = chunk + 64 * (st >> 1) + 8 * h;
				lds_bytes_t qh = chunk + 128 + 32 * (st >> 1) + 8 * h;
				return { { load8(ql, 0), load8(ql, 16), load8(ql, 32), load8(ql, 48) }, { load8(qh, 0), load8(qh, 16) } };
			}
			// quarter i = 2 (st % 2) + t / 2 of the half, elements 16 (t % 2) + 8 h .. of its 32
			static __device__ __forceinline__ half8 frag(const Head&, const Raw& r, int st, int t)
			{
				const int sh = 4 * (st & 1), top = 2 * (2 * (st & 1) + (t >> 1));
				const u32x2 q = r.low[2 * (t >> 1) + (t & 1)], f = r.high[t & 1];
				return bytes_minus(((q.x >> sh) & 0x0f0f0f0fu) | (((f.x >> top) & 0x03030303u) << 4),
				                   ((q.y >> sh) & 0x0f0f0f0fu) | (((f.y >> top) & 0x03030303u) << 4), 32.0f);
			}
			static __device__ __forceinline__ float scale(const Head& hd, const Raw&, int st, int t)
			{
				const int sub = 4 * st + t;
				const uint32_t w = sub < 4 ? hd.sc.x : sub < 8 ? hd.sc.y : sub < 12 ? hd.sc.z : hd.sc.w;
				return static_cast<float>(static_cast<int8_t>(w >> (8 * (sub & 3))));
			}
			static __device__ __forceinline__ float chunk_scale(const Head& hd) { return f16_bits_to_f32(hd.d); }
		};

		// A weight row times the activations x(k), the terms formed as the streaming kernel forms them: for results that an
		// infinite activation leaves infinite or NaN, which centred integers would give another sign or no number.
		template <typename F, typename X>
		__device__ __forceinline__ float plain_dot(const uint8_t* row, int chunks, X x)
		{
			float total = 0.0f;
#pragma unroll 1
			for (int c = 0; c < chunks; ++c, row += F::kChunkBytes)
			{
				const float d = f16_bits_to_f32(row[0] | row[1] << 8), dmin = f16_bits_to_f32(row[2] | row[3] << 8);
#pragma unroll 1
				for (int j = 0; j < 8; ++j)
				{
					const uint8_t* const sc = row + 4;
					const int s = j < 4 ? sc[j] & 63 : (sc[j + 4] & 15) | (sc[j - 4] >> 6) << 4;
					const int m = j < 4 ? sc[j + 4] & 63 : sc[j + 4] >> 4 | (sc[j] >> 6) << 4;
					float sum = 0.0f, off = 0.0f;
#pragma unroll 1
					for (int l = 0; l < 32; ++l)
					{
						const float v = x(kChunk * c + 32 * j + l);
						sum = fmaf(static_cast<float>(F::code(row, j, l)), v, sum);
						off += v;
					}
					total += d * (static_cast<float>(s) * sum) - dmin * (static_cast<float>(m) * off);
				}
			}
			return total;
		}

		// 16-byte pieces of a row's chunk, the last one moved back so that it ends with the chunk.  The rows of a slot are a
		// multiple of 16 bytes but not of 32 apart: 32 lanes then read over 64 banks two to a bank.
		template <typename F>
		constexpr int slot_pieces() { return (F::kChunkBytes + 15) / 16; }
		template <typename F>
		constexpr int slot_stride() { return 16 * (slot_pieces<F>() | 1); }

		// ---- activations -> fragments -----------------------------------------------------------------
		// [tile of 32 rows][chunk][step][hi, lo] fragments, then [tile][chunk] fragments of sub-block sums
		// (halves 0..7 of lane (r, 0): hi parts, of lane (r, 1): lo parts), then a factor per row.
		struct RowsLayout
		{
			size_t sums, factors, bytes;
			__host__ __device__ RowsLayout(size_t tiles, size_t chunks)
			{
				sums = tiles * chunks * kTileChunkBytes;
				factors = sums + tiles * chunks * kFrag;
				bytes = factors + tiles * kTile * sizeof(float);
			}
		};

		constexpr int kMostItems = 2048; // 8-element items of a row: rows up to 16384 wide

		// One workgroup per row.  The producers of csrc/gemm.hip's pre-pass may run first: RMSNorm with f64
		// accumulation (norm_w) or SwiGLU's silu(x) * up.
		template <int T>
		__global__ __launch_bounds__(T) void split_rows_kernel(const float* __restrict__ x, uint8_t* __restrict__ out,
		                                                         int m, int m_pad, int k, int chunks,
		                                                         const float* __restrict__ norm_w, double eps,
		                                                         const float* __restrict__ up)
		{
			constexpr int kHeldItems = kMostItems / T, kWaves = T / 64;
			__shared__ float red[kWaves];
			__shared__ double red64[kWaves];
			// eight rows share every 128-byte line of the layout: XCD x (workgroups are dealt out round-robin)
			// takes the row octets x, x + 8, ... so that its L2 puts whole lines together
			const int xcd = blockIdx.x & 7, nth = blockIdx.x >> 3;
			const int row = (((nth >> 3) << 3) + xcd) * 8 + (nth & 7);
			if (row >= m_pad)
			{
				return;
			}
			const RowsLayout at(m_pad / kTile, chunks);
			const int tile = row / kTile, r = row % kTile;
			uint8_t* frags = out + static_cast<size_t>(tile) * chunks * kTileChunkBytes + r * 16;
			uint8_t* sums = out + at.sums + static_cast<size_t>(tile) * chunks * kFrag + r * 16;
			float* factors = reinterpret_cast<float*>(out + at.factors);
			const int items = chunks * (kChunk / 8);
			float held[kHeldItems][8];
			double ss = 0.0;
			float mx = 0.0f;
#pragma unroll
			for (int u = 0; u < kHeldItems; ++u)
			{
				const int it = threadIdx.x + T * u;
#pragma unroll
				for (int e = 0; e < 8; ++e)
				{
					held[u][e] = 0.0f;
				}
				if (row < m && 8 * it < k)
				{
					const size_t o = static_cast<size_t>(row) * k + 8 * it;
					const float4 a = *reinterpret_cast<const float4*>(x + o);
					const float4 b = *reinterpret_cast<const float4*>(x + o + 4);
					held[u][0] = a.x, held[u][1] = a.y, held[u][2] = a.z, held[u][3] = a.w;
					held[u][4] = b.x, held[u][5] = b.y, held[u][6] = b.z, held[u][7] = b.w;
					if (up)
					{
						const float4 ua = *reinterpret_cast<const float4*>(up + o);
						const float4 ub = *reinterpret_cast<const float4*>(up + o + 4);
						const float uu[8] = { ua.x, ua.y, ua.z, ua.w, ub.x, ub.y, ub.z, ub.w };
#pragma unroll
						for (int e = 0; e < 8; ++e)
						{
							const float gv = held[u][e];
							const float sig = __fdiv_rn(1.0f, __fadd_rn(1.0f, expf(-gv)));
							held[u][e] = __fmul_rn(__fmul_rn(gv, sig), uu[e]);
						}
					}
#pragma unroll
					for (int e = 0; e < 8; ++e)
					{
						const double v = static_cast<double>(held[u][e]);
						ss += v * v;
					}
				}
			}
			if (norm_w)
			{
				for (int off = 32; off > 0; off >>= 1)
				{
					ss += __shfl_xor(ss, off, 64);
				}
				if ((threadIdx.x & 63) == 0)
				{
					red64[threadIdx.x >> 6] = ss;
				}
				__syncthreads();
				double total = red64[0];
#pragma unroll
				for (int i = 1; i < kWaves; ++i)
				{
					total += red64[i];
				}
				const double inv = 1.0 / sqrt(total / static_cast<double>(k) + eps);
#pragma unroll
				for (int u = 0; u < kHeldItems; ++u)
				{
					const int it = threadIdx.x + T * u;
					if (row < m && 8 * it < k)
					{
						const float4 wa = *reinterpret_cast<const float4*>(norm_w + 8 * it);
						const float4 wb = *reinterpret_cast<const float4*>(norm_w + 8 * it + 4);
						const float ww[8] = { wa.x, wa.y, wa.z, wa.w, wb.x, wb.y, wb.z, wb.w };
#pragma unroll
						for (int e = 0; e < 8; ++e)
						{
							held[u][e] = static_cast<float>(static_cast<double>(held[u][e]) * inv * static_cast<double>(ww[e]));
						}
					}
				}
			}
			// the largest finite magnitude (infinities and NaN keep their values below)
#pragma unroll
			for (int u = 0; u < kHeldItems; ++u)
			{
#pragma unroll
				for (int e = 0; e < 8; ++e)
				{
					const float a = fabsf(held[u][e]);
					mx = a <= 3.402823466e38f ? fmaxf(mx, a) : mx;
				}
			}
			mx = wave_max(mx);
			if ((threadIdx.x & 63) == 0)
			{
				red[threadIdx.x >> 6] = mx;
			}
			__syncthreads();
#pragma unroll
			for (int i = 0; i < kWaves; ++i)
			{
				mx = fmaxf(mx, red[i]);
			}
			// x 2^shift has its largest magnitude in [2^14, 2^15); the inverse stays a normal number
			const int shift = mx > 0.0f ? min(14 - ilogbf(mx), 126) : 0;
#pragma unroll
			for (int u = 0; u < kHeldItems; ++u)
			{
				const int it = threadIdx.x + T * u;
				double sum = 0.0;
				if (it < items)
				{
					half8 hi, lo;
#pragma unroll
					for (int e = 0; e < 8; ++e)
					{
						const float v = ldexpf(held[u][e], shift);
						hi[e] = static_cast<_Float16>(v);
						const float rest = v - static_cast<float>(hi[e]);
						lo[e] = static_cast<_Float16>(fabsf(v) <= 65504.0f ? rest * (1.0f / kLowScale) : 0.0f); // (inf - inf)
						sum += static_cast<double>(v);
					}
					uint8_t* dst = frags + static_cast<size_t>(it >> 1) * (2 * kFrag) + (it & 1) * 512;
					*reinterpret_cast<half8*>(dst) = hi;
					*reinterpret_cast<half8*>(dst + kFrag) = lo;
				}
				// four neighbouring threads hold one sub-block of 32 elements
				sum += __shfl_xor(sum, 1, 64);
				sum += __shfl_xor(sum, 2, 64);
				if (it < items && (threadIdx.x & 3) == 0)
				{
					const float v = static_cast<float>(sum * kSumScale);
					const _Float16 hi = static_cast<_Float16>(v);
					const double rest = sum * kSumScale - static_cast<double>(static_cast<float>(hi));
					const _Float16 lo = static_cast<_Float16>(fabsf(v) <= 65504.0f ? static_cast<float>(rest * (1.0f / kLowScale)) : 0.0f);
					uint8_t* dst = sums + static_cast<size_t>(it >> 5) * kFrag + ((it >> 2) & 7) * 2;
					*reinterpret_cast<_Float16*>(dst) = hi;
					*reinterpret_cast<_Float16*>(dst + 512) = lo;
				}
			}
			if (threadIdx.x == 0)
			{
				factors[row] = row < m ? ldexpf(1.0f, -shift) : 0.0f;
			}
		}

		// The sums of neighbouring ranges of K, then of neighbouring pairs: a shorter chain rounds less.  v[0] is the result.
		template <typename V, int N>
		__device__ __forceinline__ void add_in_pairs(V (&v)[N])
		{
#pragma unroll
			for (int apart = 1; apart < N; apart *= 2)
			{
#pragma unroll
				for (int i = 0; i + apart < N; i += 2 * apart)
				{
					v[i] += v[i + apart];
				}
			}
		}

		// ---- the product ------------------------------------------------------------------------------
		struct ExactMats
		{
			const uint8_t* w[3];
			float* y[3];
			int n[3];
			int first_block[3]; // grid x index of each matrix's first workgroup (INT_MAX when unused)
		};

		// Workgroups that share a strip of weight rows follow each other on one XCD (as in csrc/gemm.hip)
		__device__ __forceinline__ void exact_grid_position(int& grid_x, int& grid_y)
		{
			grid_x = blockIdx.x, grid_y = blockIdx.y;
			if (gridDim.y > 1)
			{
				const int gx = gridDim.x, gy = gridDim.y, full = gx & ~7, l = grid_x + gx * grid_y;
				if (l < full * gy)
				{
					grid_x = (l / (8 * gy)) * 8 + (l & 7);
					grid_y = (l >> 3) % gy;
				}
				else
				{
					grid_x = full + (l - full * gy) % (gx - full);
					grid_y = (l - full * gy) / (gx - full);
				}
			}
		}

		// A wavefront's share of the weights on their way: the raw blocks of 32 (or 16) rows for one chunk, from memory (where
		// they lie on 2 bytes) to the wavefront's slot in LDS (where a row's chunk begins on 16).  The P pieces of a row fall
		// into groups of 16, 8, 4, 2 and 1 (the bits of P); a load takes one group of as many rows as there are lanes for, so
		// that a lane's place in the row stays the same from load to load and its addresses are one sum.  Nothing behind
		// the matrix is fetched: rows behind the last are the last, and a row's chunk that is not whole comes element
		// by element, its missing part being the row's last two bytes.
		template <typename F, int ROWS = kTile>
		struct WeightPieces
		{
			static constexpr int P = slot_pieces<F>(), kStride = slot_stride<F>(), kRows = ROWS;
			static constexpr int loads_of(int width) { return (P & width) != 0 ? (kRows * width + 63) / 64 : 0; }
			static constexpr int kLoads = loads_of(16) + loads_of(8) + loads_of(4) + loads_of(2) + loads_of(1);
			static constexpr int kSlotBytes = kRows * kStride;
			static_assert(P < 32, "pieces");
			// (addresses of the global segment: a load through a generic pointer counts as an LDS access too, and every
			// wait for LDS would wait for it)
			typedef u32x4 u32x4_a2 __attribute__((aligned(2)));
			typedef const __attribute__((address_space(1))) uint8_t* global_bytes_t;
			typedef const __attribute__((address_space(1))) u32x4_a2* global_u32x4_t;
			typedef const __attribute__((address_space(1))) uint16_t* global_u16_t;
			global_bytes_t base; // the first row
			int row_bytes, rows_left;
			uint8_t* slot;

			__device__ __forceinline__ WeightPieces(uint8_t* slot_, const uint8_t* w, int n_base, int n, size_t row_bytes_)
			    : base((global_bytes_t)(w + static_cast<size_t>(min(n_base, n - 1)) * row_bytes_)), row_bytes(static_cast<int>(row_bytes_)),
			      rows_left(max(n - n_base, 1)), slot(slot_)
			{
			}
			// calls f(load, lane's row, lane's piece)
			template <typename Fn>
			static __device__ __forceinline__ void each(int lane, Fn f)
			{
				int load = 0, first = 0;
#pragma unroll
				for (int width = 16; width >= 1; width /= 2)
				{
#pragma unroll
					for (int i = 0; i < loads_of(width); ++i)
					{
						f(load++, (i * (64 / width) + lane / width) % kRows, first + lane % width);
					}
					first += P & width;
				}
			}
			__device__ __forceinline__ void request(u32x4 (&moving)[kLoads], int c, int lane) const
			{
				const int from = c * F::kChunkBytes;
				if (F::kBlock < kChunk && from + F::kChunkBytes > row_bytes)
				{
					each(lane, [&](int i, int row, int piece) {
#pragma unroll
						for (int e = 0; e < 8; ++e)
						{
							const global_u16_t at = (global_u16_t)(base + min(row, rows_left - 1) * row_bytes + min(from + 16 * piece + 2 * e, row_bytes - 2));
							moving[i][e / 2] = e % 2 == 0 ? *at : moving[i][e / 2] | static_cast<uint32_t>(*at) << 16;
						}
					});
					return;
				}
				each(lane, [&](int i, int row, int piece) {
					moving[i] = *(global_u32x4_t)(base + min(row, rows_left - 1) * row_bytes + (from + min(16 * piece, F::kChunkBytes - 16)));
				});
			}
			__device__ __forceinline__ void deposit(const u32x4 (&moving)[kLoads], int lane) const
			{
				each(lane, [&](int i, int row, int piece) { *reinterpret_cast<u32x4*>(slot + row * kStride + 16 * piece) = moving[i]; });
			}
			// the lane's row in the slot
			__device__ __forceinline__ lds_bytes_t chunk(int lane) const { return (lds_bytes_t)(slot) + (lane & (kRows - 1)) * kStride; }
		};

		// What of the product a workgroup and its wavefront take, and the way out of their sums: shared by both forms below.
		// A wavefront multiplies 32 weight rows by MT tiles of 32 activation rows over one of KS ranges of K; the KS sums meet in
		// LDS at the end, added in K order.  Two levels of sums, a chunk's and the range's, keep the rounding of long rows down.
		template <typename F, int MT, int WN, int KS>
		struct ExactPlace
		{
			const uint8_t* w;
			float* y;
			int n, lane, part, wv, n_base, mt_base, c_begin, c_end, per;

			__device__ __forceinline__ ExactPlace(const ExactMats& mats, int chunks)
			{
				int grid_x, grid_y;
				exact_grid_position(grid_x, grid_y);
				const int which = (grid_x >= mats.first_block[1]) + (grid_x >= mats.first_block[2]);
				w = which == 0 ? mats.w[0] : (which == 1 ? mats.w[1] : mats.w[2]);
				y = which == 0 ? mats.y[0] : (which == 1 ? mats.y[1] : mats.y[2]);
				n = which == 0 ? mats.n[0] : (which == 1 ? mats.n[1] : mats.n[2]);
				const int block_x = grid_x - (which == 0 ? 0 : (which == 1 ? mats.first_block[1] : mats.first_block[2]));
				lane = threadIdx.x & 63;
				const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
				part = wave / WN, wv = wave % WN;
				n_base = (block_x * WN + wv) * kTile;
				mt_base = grid_y * MT;
				per = (chunks + KS - 1) / KS;
				c_begin = part * per, c_end = min(c_begin + per, chunks);
			}

			// The sums of all ranges, scaled, go out (not `scaled`: those of one range of several, to which a launch more sees: times
			// a row's factor a range's sum may overflow where the result does not); every wavefront of the workgroup calls it
			__device__ __forceinline__ void finish(floatx16 (&acc)[MT], uint8_t* lds, const uint8_t* xs, const RowsLayout& at, const float* residual,
			                                       int m, int chunks, size_t row_bytes, bool scaled = true) const
			{
				const int r = lane & 31, h = lane >> 5;
				if constexpr (KS > 1)
				{
					// ranges 1 .. KS - 1 hand their sums to range 0
					__syncthreads();
					floatx16* const handed = reinterpret_cast<floatx16*>(lds);
					if (part > 0)
					{
#pragma unroll
						for (int t = 0; t < MT; ++t)
						{
#pragma unroll
							for (int e = 0; e < 16; e += 4)
							{
								float4* dst = reinterpret_cast<float4*>(handed + (((part - 1) * WN + wv) * MT + t) * 64) + (e / 4) * 64 + lane;
								*dst = float4{ acc[t][e], acc[t][e + 1], acc[t][e + 2], acc[t][e + 3] };
							}
						}
					}
					__syncthreads();
					if (part > 0)
					{
						return;
					}
#pragma unroll
					for (int t = 0; t < MT; ++t)
					{
#pragma unroll
						for (int e = 0; e < 16; e += 4)
						{
							floatx4 v[KS];
							v[0] = floatx4{ acc[t][e], acc[t][e + 1], acc[t][e + 2], acc[t][e + 3] };
#pragma unroll
							for (int other = 1; other < KS; ++other)
							{
								v[other] = *(reinterpret_cast<const floatx4*>(handed + (((other - 1) * WN + wv) * MT + t) * 64) + (e / 4) * 64 + lane);
							}
							add_in_pairs(v);
#pragma unroll
							for (int i = 0; i < 4; ++i)
							{
								acc[t][e + i] = v[0][i];
							}
						}
					}
				}

				// lane (r, h) holds weight row r and activation rows 8 (e / 4) + 4 h + e % 4.  Everything is asked for before the first
				// store: a factor and a residual at a time, each waited for, were 10 us of every workgroup.
				const float* factors = reinterpret_cast<const float*>(xs + at.factors);
				const int col = n_base + r;
				uint32_t again = 0; // results that are not finite
#pragma unroll
				for (int t = 0; t < MT; ++t)
				{
					const int first = (mt_base + t) * kTile + 4 * h;
					if ((mt_base + t) * kTile >= m)
					{
						break;
					}
					floatx4 us[4];
					float res[16];
#pragma unroll
					for (int e = 0; e < 16; e += 4)
					{
						us[e / 4] = scaled ? *reinterpret_cast<const floatx4*>(factors + first + 2 * e) : floatx4{ 1.0f, 1.0f, 1.0f, 1.0f };
					}
					if (residual)
					{
#pragma unroll
						for (int e = 0; e < 16; ++e)
						{
							res[e] = residual[static_cast<size_t>(min(first + 8 * (e / 4) + (e & 3), m - 1)) * n + min(col, n - 1)];
						}
					}
					if (col < n)
					{
#pragma unroll
						for (int e = 0; e < 16; ++e)
						{
							const int mm = first + 8 * (e / 4) + (e & 3);
							if (mm < m)
							{
								if (F::kMins && !(fabsf(acc[t][e]) <= 3.402823466e38f))
								{
									again |= 1u << (16 * t + e);
									continue;
								}
								const float v = acc[t][e] * us[e / 4][e & 3];
								y[static_cast<size_t>(mm) * n + col] = residual ? res[e] + v : v;
							}
						}
					}
				}
				if constexpr (F::kMins)
				{
					while (__builtin_expect(again != 0, 0))
					{
						const int i = __ffs(again) - 1, e = i & 15, mm = (mt_base + (i >> 4)) * kTile + 8 * (e / 4) + 4 * h + (e & 3);
						again &= again - 1;
						const uint8_t* const parts = xs + static_cast<size_t>(mm / kTile) * chunks * kTileChunkBytes + (mm % kTile) * 16;
						const float v = (scaled ? factors[mm] : 1.0f) * plain_dot<F>(w + static_cast<size_t>(col) * row_bytes, chunks, [&](int i) {
							const uint8_t* const at = parts + static_cast<size_t>(i >> 4) * (2 * kFrag) + ((i >> 3) & 1) * 512 + (i & 7) * 2;
							return fmaf(static_cast<float>(*reinterpret_cast<const _Float16*>(at + kFrag)), kLowScale, static_cast<float>(*reinterpret_cast<const _Float16*>(at)));
						});
						const size_t o = static_cast<size_t>(mm) * n + col;
						y[o] = residual ? residual[o] + v : v;
					}
				}
			}
		};

		// WN wavefronts side by side share the activation fragments of a range through LDS: a ring of 64-element stages that loads fill
		// directly, two stages ahead, which leaves registers for the sums and time for the blocks of the next chunk (they come from HBM,
		// and what was asked for behind them arrives behind them).  Those blocks travel through registers into the wavefront's slot.
		// What a step of 16 elements multiplies is in registers when it begins: the step before asks for its activations ahead of
		// its own products and decodes its weights behind them, and a stage's last products follow the barrier, so that they cover
		// the next stage's first reads.
		// KS = 1 gives every `flush` chunks a sum of their own: half of K's, which are added as the two ranges of KS = 2 are, or, with
		// RANGES of K over grid z, as many of the range's as round least.
		// Bound by no unit alone (matrix cores 38 % busy, VALU 39, LDS 26; 18 % of a wavefront's time are waits for operands and barriers)
		// and by a last round of few workgroups.  us, kernel alone, Q4_K 28672 x 4096 at 300 rows: stages through registers and two
		// buffers 221, ring 216, KS = 1 with two workgroups to a CU 190; Q6_K 4096 x 14336, by two tiles a wavefront on their own 172,
		// here in three ranges 130 and 5 for adding them.
		constexpr int kRing = 3; // stages: one is multiplied, two are on their way
		// all but the N youngest of the wavefront's loads are there
		template <int N>
		__device__ __forceinline__ void arrived() { asm volatile("s_waitcnt vmcnt(%0)" : : "n"(N) : "memory"); }

		template <typename F, int MT, int WN, int KS, bool RANGES>
		__global__ __launch_bounds__(64 * WN * KS, 2) void exact_shared_kernel(const ExactMats mats, const uint8_t* __restrict__ xs,
		                                                                    const float* residual, int k, int m, int m_tiles,
		                                                                    int chunks, size_t row_bytes, int flush, size_t range_stride, int first_row)
		{
			constexpr bool kScaled = F::kScaleSteps < 16; // sums of kScaleSteps steps are scaled and added to the chunk's
			static_assert(kScaled != F::kMins, "one scale for a chunk has minima beside it");
			constexpr int kPieces = MT * 8 / WN; // 1 KB pieces a wavefront stages
			static_assert(kPieces * WN == MT * 8, "activation pieces / wavefront split");
			typedef WeightPieces<F> W;
			constexpr int kBuffer = MT * kStageBytes, kRingBytes = KS * kRing * kBuffer;
			extern __shared__ __attribute__((aligned(16))) uint8_t lds[]; // [KS][kRing][MT][stage], [WN KS][slot]; later the KS sums
			ExactPlace<F, MT, WN, KS> place(mats, chunks);
			const int lane = place.lane, h = lane >> 5;
			if constexpr (RANGES)
			{
				static_assert(KS == 1, "ranges of K over workgroups");
				const int per = (chunks + static_cast<int>(gridDim.z) - 1) / static_cast<int>(gridDim.z);
				place.c_begin = static_cast<int>(blockIdx.z) * per, place.c_end = min(place.c_begin + per, chunks);
				place.mt_base += first_row / kTile;
				place.y += static_cast<ptrdiff_t>(blockIdx.z * range_stride) - static_cast<ptrdiff_t>(first_row) * place.n;
			}
			const int c_begin = place.c_begin, c_end = place.c_end;
			const W weights(lds + kRingBytes + (place.part * WN + place.wv) * W::kSlotBytes, place.w, place.n_base, place.n, row_bytes);
			u32x4 moving[W::kLoads];

			const RowsLayout at(m_tiles, chunks);
			const uint8_t* sum_tiles[MT];
#pragma unroll
			for (int t = 0; t < MT; ++t)
			{
				sum_tiles[t] = xs + at.sums + static_cast<size_t>(min(place.mt_base + t, m_tiles - 1)) * chunks * kFrag;
			}

			floatx16 acc[MT], p[MT];
			floatx16 held[MT]; // the chunk's first half; kScaled: its sum so far
			constexpr bool kFlushed = KS == 1 || kScaled; // every `flush` chunks' sums go to a sum of their own
			floatx16 total[kFlushed ? MT : 1];
#pragma unroll
			for (int t = 0; t < MT; ++t)
			{
				acc[t] = floatx16{};
			}

			const uint8_t* const ring = lds + place.part * kRingBytes / KS;
			const uint8_t* from[kPieces];
#pragma unroll
			for (int i = 0; i < kPieces; ++i)
			{
				const int piece = i * WN + place.wv;
				from[i] = xs + static_cast<size_t>(min(place.mt_base + (piece >> 3), m_tiles - 1)) * chunks * kTileChunkBytes + (piece & 7) * kFrag;
			}
			const uint32_t lane_at = lane * 16;
			const uint32_t ring_lds = static_cast<uint32_t>(reinterpret_cast<uintptr_t>((lds_bytes_t)(ring)));
			// (as inline assembly: a load into LDS that the compiler knew of would be waited for before every read of LDS)
			const auto request = [&](int c, int st, int buffer) {
#pragma unroll
				for (int i = 0; i < kPieces; ++i)
				{
					const uint8_t* const src = from[i] + static_cast<size_t>(c) * kTileChunkBytes + st * kStageBytes;
					const uint32_t dst = ring_lds + buffer * kBuffer + (i * WN + place.wv) * kFrag;
#pragma clang diagnostic push
#pragma clang diagnostic ignored "-Winline-asm" // m0 is named as clobbered although it is reserved
					asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2" : : "s"(dst), "v"(lane_at), "s"(src) : "memory", "m0");
#pragma clang diagnostic pop
				}
			};

			half8 a[2][MT][2], b[2]; // of this step and the next
			const auto read = [&](int buffer, int s, int into) {
#pragma unroll
				for (int t = 0; t < MT; ++t)
				{
#pragma unroll
					for (int e = 0; e < 2; ++e)
					{
						a[into][t][e] = *reinterpret_cast<const half8*>(ring + buffer * kBuffer + t * kStageBytes + (2 * s + e) * kFrag + lane * 16);
					}
				}
			};

			typename F::Head head, next_head;
			typename F::Raw raw, next_raw;
			const auto blocks_of = [&](int c) { return k / F::kBlock - c * (kChunk / F::kBlock); };
			if (c_begin < c_end)
			{
				weights.request(moving, c_begin, lane);
				request(c_begin, 0, 0);
				request(c_begin, 1, 1);
				weights.deposit(moving, lane);
				weights.request(moving, min(c_begin + 1, c_end - 1), lane);
				__builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
				arrived<kPieces + W::kLoads>(); // (behind the first stage's: the second's and the next chunk's blocks)
			}
			__syncthreads();
			int buffer = 0;
			const auto behind = [](int b, int by) { return b + by < kRing ? b + by : b + by - kRing; };
			if (c_begin < c_end)
			{
				head = F::head(weights.chunk(lane), h);
				raw = F::load(weights.chunk(lane), 0, h, blocks_of(c_begin));
				read(0, 0, 0);
				b[0] = F::frag(head, raw, 0, 0);
			}
			const auto walk = [&](int c_from, int c_to) {
				for (int c = c_from; c < c_to; ++c)
				{
					const int next = min(c + 1, c_end - 1);
					half8 sum_frag[MT];
#pragma unroll
					for (int st = 0; st < 4; ++st)
					{
#pragma unroll
						for (int s = 0; s < 4; ++s)
						{
							const int step = 4 * st + s, mine = s & 1, other = mine ^ 1;
							if (s < 3)
							{
								read(buffer, s + 1, other);
							}
							if (s == 0)
							{
								if (F::kMins && st == 2)
								{
#pragma unroll
									for (int t = 0; t < MT; ++t)
									{
										sum_frag[t] = *reinterpret_cast<const half8*>(sum_tiles[t] + static_cast<size_t>(c) * kFrag + lane_at);
									}
								}
								if (st == 3)
								{
									// (a wavefront's LDS accesses keep their order: the slot's reads, the next chunk, its reads)
									__builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
									weights.deposit(moving, lane);
									__builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
								}
								// (the buffer was read last before the barrier that this stage began with)
								request(st < 2 ? c : next, (st + 2) & 3, behind(buffer, 2));
								if (st == 3)
								{
									weights.request(moving, min(c + 2, c_end - 1), lane);
								}
							}
							if (s == 2)
							{
								if (st == 3)
								{
									next_head = F::head(weights.chunk(lane), h);
								}
								next_raw = F::load(weights.chunk(lane), (st + 1) & 3, h, blocks_of(st < 3 ? c : next));
							}
							if (s == 3)
							{
								// the wavefront's pieces of the next stage are there; behind them are those of the one after it and a chunk's blocks
								if (st == 3)
								{
									arrived<kPieces + W::kLoads>();
								}
								else
								{
									arrived<kPieces>();
								}
								__syncthreads();
								buffer = behind(buffer, 1);
								read(buffer, 0, other);
							}
							__builtin_amdgcn_sched_barrier(0);
							const half8 low = lowered(b[mine]);
							const bool fresh = step % (kScaled ? F::kScaleSteps : 8) == 0;
#pragma unroll
							for (int e = 0; e < 2; ++e)
							{
#pragma unroll
								for (int t = 0; t < MT; ++t)
								{
									p[t] = __builtin_amdgcn_mfma_f32_32x32x16_f16(a[mine][t][e], e == 0 ? b[mine] : low, fresh && e == 0 ? floatx16{} : p[t], 0, 0, 0);
								}
							}
							if (s < 3)
							{
								b[other] = F::frag(head, raw, st, s + 1);
							}
							else
							{
								b[other] = F::frag(st < 3 ? head : next_head, next_raw, (st + 1) & 3, 0);
							}
							if constexpr (kScaled)
							{
								if (step % F::kScaleSteps == F::kScaleSteps - 1)
								{
									const float d = F::scale(head, raw, st, s);
#pragma unroll
									for (int t = 0; t < MT; ++t)
									{
#pragma unroll
										for (int e = 0; e < 16; ++e)
										{
											held[t][e] = step == F::kScaleSteps - 1 ? d * p[t][e] : fmaf(d, p[t][e], held[t][e]);
										}
									}
								}
							}
							if (F::kMins && step == 7) // (two sums of eight steps each: a shorter chain rounds less)
							{
#pragma unroll
								for (int t = 0; t < MT; ++t)
								{
									held[t] = p[t];
								}
							}
							__builtin_amdgcn_sched_barrier(0);
						}
						raw = next_raw;
					}
					const float d = F::chunk_scale(head);
					if constexpr (F::kMins)
					{
						const half8 centres = for_sums(F::centre_frag(head), h), minima = for_sums(F::min_frag(head), h);
						const float dm = F::min_scale(head) * (1.0f / kSumScale);
#pragma unroll
						for (int t = 0; t < MT; ++t)
						{
							const floatx16 ce = __builtin_amdgcn_mfma_f32_32x32x16_f16(sum_frag[t], centres, floatx16{}, 0, 0, 0);
							const floatx16 mi = __builtin_amdgcn_mfma_f32_32x32x16_f16(sum_frag[t], minima, floatx16{}, 0, 0, 0);
#pragma unroll
							for (int e = 0; e < 16; ++e)
							{
								acc[t][e] += fmaf(d, held[t][e] + p[t][e], fmaf(d, ce[e], dm * mi[e]));
							}
						}
					}
					else
					{
#pragma unroll
						for (int t = 0; t < MT; ++t)
						{
#pragma unroll
							for (int e = 0; e < 16; ++e)
							{
								acc[t][e] = fmaf(d, held[t][e], acc[t][e]);
							}
						}
					}
					head = next_head;
				}
			};
			if constexpr (kFlushed)
			{
#pragma unroll
				for (int t = 0; t < MT; ++t)
				{
					total[t] = floatx16{};
				}
				for (int c = c_begin; c < c_end; c += flush)
				{
					walk(c, min(c + flush, c_end));
#pragma unroll
					for (int t = 0; t < MT; ++t)
					{
						total[t] += acc[t];
						acc[t] = floatx16{};
					}
				}
#pragma unroll
				for (int t = 0; t < MT; ++t)
				{
					acc[t] = total[t];
				}
			}
			else
			{
				walk(c_begin, c_end);
			}
			arrived<0>(); // (nothing may arrive in LDS that is the sums' or another workgroup's)
			// a shorter range only passes the barriers
			for (int i = max(c_end - c_begin, 0); KS > 1 && i < place.per; ++i)
			{
#pragma unroll
				for (int st = 0; st < 4; ++st)
				{
					__syncthreads();
				}
			}
			place.finish(acc, lds, xs, at, residual, m, chunks, row_bytes, !RANGES);
		}

		// The same with less held ahead.  WN > 1: the fragments pass through the same two buffers, two stages on their way; with WN =
		// 1 nobody shares them and they go to registers directly, each refilled for a later step once it has been used.  Nobody is
		// waited for there either: in one run (ONE_RUN) a wavefront walks its own range with no branch in a chunk's steps, which the
		// compiler orders as a whole; else stage by stage.  With two tiles only two steps' fragments are held (four: 32 more
		// registers, the sums' and scales' loads waited for in turn).  Q6_K 4096 x 14336, 1000 rows: 630 us with a branch a stage
		// and four steps, 608 with two, 595 without the branches; 14336 x 4096, 45 rows: 52.1 -> 50.0; one tile (Q4_0, Q8_0): 1 to 4 %.
		template <typename F, int MT, int WN, int KS, bool ONE_RUN>
		__global__ __launch_bounds__(64 * WN * KS) void exact_gemm_kernel(const ExactMats mats, const uint8_t* __restrict__ xs,
		                                                                  const float* residual, int k, int m, int m_tiles,
		                                                                  int chunks, size_t row_bytes)
		{
			constexpr bool kShared = WN > 1;
			constexpr int kPieces = kShared ? MT * 8 / WN : 1; // 1 KB pieces a wavefront stages
			static_assert(!kShared || kPieces * WN == MT * 8, "activation pieces / wavefront split");
			static_assert(kShared ? !ONE_RUN : ONE_RUN || MT == 1, "barriers; a stage held");
			typedef WeightPieces<F> W;
			constexpr int kRingBytes = kShared ? KS * 2 * MT * kStageBytes : 0;
			extern __shared__ __attribute__((aligned(16))) uint8_t lds[]; // [KS][2][MT][stage], [WN KS][slot]; later the KS sums
			const ExactPlace<F, MT, WN, KS> place(mats, chunks);
			const int lane = place.lane, part = place.part, wv = place.wv, h = lane >> 5, mt_base = place.mt_base;
			const int c_begin = place.c_begin, c_end = place.c_end, per = place.per;

			const W weights(lds + kRingBytes + (part * WN + wv) * W::kSlotBytes, place.w, place.n_base, place.n, row_bytes);
			u32x4 moving[W::kLoads];

			const RowsLayout at(m_tiles, chunks);
			const uint8_t* tiles[MT]; // this lane's 16 bytes of the tile's first fragment
			const uint8_t* sum_tiles[MT];
#pragma unroll
			for (int t = 0; t < MT; ++t)
			{
				const size_t tile = min(mt_base + t, m_tiles - 1);
				tiles[t] = xs + tile * chunks * kTileChunkBytes + lane * 16;
				sum_tiles[t] = xs + at.sums + tile * chunks * kFrag + lane * 16;
			}

			floatx16 acc[MT], p[MT], first[MT]; // first: of the chunk's first half, where kScaleSteps is 16
#pragma unroll
			for (int t = 0; t < MT; ++t)
			{
				acc[t] = floatx16{};
			}

			// ---- activations
			constexpr int kHeld = MT > 1 ? 2 : 4; // steps whose fragments are here or on their way, WN = 1
			half8 direct[kShared ? 1 : MT][kHeld][2];
			u32x4 staged[2][kPieces]; // WN > 1: the next two stages on their way
			uint8_t* const ring = lds + part * (2 * MT * kStageBytes);
			const auto request = [&](u32x4 (&into)[kPieces], int c, int st) {
#pragma unroll
				for (int i = 0; i < kPieces; ++i)
				{
					const int piece = i * WN + wv, t = piece >> 3;
					const size_t tile = min(mt_base + t, m_tiles - 1);
					into[i] = *reinterpret_cast<const u32x4*>(xs + (tile * chunks + c) * kTileChunkBytes + st * kStageBytes +
					                                            (piece & 7) * kFrag + lane * 16);
				}
			};
			const auto deposit = [&](const u32x4 (&from)[kPieces], int buffer) {
#pragma unroll
				for (int i = 0; i < kPieces; ++i)
				{
					*reinterpret_cast<u32x4*>(ring + buffer * (MT * kStageBytes) + (i * WN + wv) * kFrag + lane * 16) = from[i];
				}
			};
			const auto fetch_direct = [&](int c, int st, int s) {
#pragma unroll
				for (int t = 0; t < MT; ++t)
				{
#pragma unroll
					for (int e = 0; e < 2; ++e)
					{
						direct[t][s % kHeld][e] = *reinterpret_cast<const half8*>(tiles[t] + static_cast<size_t>(c) * kTileChunkBytes +
						                                                  st * kStageBytes + (2 * s + e) * kFrag);
					}
				}
			};

			half8 sum_frag[MT];
			if (c_begin < c_end)
			{
				weights.request(moving, c_begin, lane);
				if constexpr (kShared)
				{
					request(staged[0], c_begin, 0);
					request(staged[1], c_begin, 1);
				}
				else
				{
#pragma unroll
					for (int s = 0; s < kHeld; ++s)
					{
						fetch_direct(c_begin, 0, s);
					}
				}
				weights.deposit(moving, lane);
				__builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
				if constexpr (kShared)
				{
					deposit(staged[0], 0);
				}
			}
			if constexpr (kShared)
			{
				__syncthreads();
			}
			int buffer = 0;
			const int trips = ONE_RUN ? c_end - c_begin : per;
			for (int i = 0; i < trips; ++i)
			{
				const int c = c_begin + i;
				const bool live = ONE_RUN || c < c_end; // (uniform: a shorter range only passes the barriers)
				const int next = min(c + 1, c_end - 1);
				typename F::Head head;
				floatx16 sum[MT]; // the chunk's, where kScaleSteps is less
				const int blocks = k / F::kBlock - c * (kChunk / F::kBlock);
				if (live)
				{
					weights.request(moving, next, lane);
					head = F::head(weights.chunk(lane), h);
					if constexpr (F::kMins)
					{
#pragma unroll
						for (int t = 0; t < MT; ++t)
						{
							sum_frag[t] = *reinterpret_cast<const half8*>(sum_tiles[t] + static_cast<size_t>(c) * kFrag);
						}
					}
				}
#pragma unroll
				for (int st = 0; st < 4; ++st)
				{
					if (live)
					{
						const typename F::Raw raw = F::load(weights.chunk(lane), st, h, blocks);
						if constexpr (kShared)
						{
							request(staged[st & 1], st < 2 ? c : next, (st + 2) & 3);
						}
#pragma unroll
						for (int s = 0; s < 4; ++s)
						{
							const half8 b = F::frag(head, raw, st, s), b_low = lowered(b);
							const int step = 4 * st + s;
							const bool fresh = step % min(F::kScaleSteps, 8) == 0;
#pragma unroll
							for (int t = 0; t < MT; ++t)
							{
								half8 a[2];
#pragma unroll
								for (int e = 0; e < 2; ++e)
								{
									if constexpr (kShared)
									{
										a[e] = *reinterpret_cast<const half8*>(ring + buffer * (MT * kStageBytes) + t * kStageBytes +
										                                       (2 * s + e) * kFrag + lane * 16);
									}
									else
									{
										a[e] = direct[t][s % kHeld][e];
									}
								}
								p[t] = __builtin_amdgcn_mfma_f32_32x32x16_f16(a[0], b, fresh ? floatx16{} : p[t], 0, 0, 0);
								p[t] = __builtin_amdgcn_mfma_f32_32x32x16_f16(a[1], b_low, p[t], 0, 0, 0);
							}
							if constexpr (ONE_RUN)
							{
								fetch_direct(step + kHeld < 16 ? c : next, ((step + kHeld) & 15) / 4, (s + kHeld) % 4);
							}
							else if constexpr (!kShared) // (the next stage's same step, said so: Q4_0 in 164 registers instead of 186)
							{
								fetch_direct(st < 3 ? c : next, (st + 1) & 3, s);
							}
							if constexpr (F::kMins)
							{
								if (step == 7) // (two sums of eight steps each: a shorter chain rounds less)
								{
#pragma unroll
									for (int t = 0; t < MT; ++t)
									{
										first[t] = p[t];
									}
								}
							}
							if constexpr (F::kScaleSteps < 16)
							{
								if (step % F::kScaleSteps == F::kScaleSteps - 1)
								{
									const float d = F::scale(head, raw, st, s);
#pragma unroll
									for (int t = 0; t < MT; ++t)
									{
#pragma unroll
										for (int e = 0; e < 16; ++e)
										{
											sum[t][e] = step == F::kScaleSteps - 1 ? d * p[t][e] : fmaf(d, p[t][e], sum[t][e]);
										}
									}
								}
							}
						}
						if constexpr (kShared)
						{
							deposit(staged[(st + 1) & 1], buffer ^ 1);
						}
					}
					if constexpr (kShared)
					{
						__syncthreads();
					}
					buffer ^= 1;
				}
				if (live)
				{
					const float d = F::chunk_scale(head);
					if constexpr (F::kMins)
					{
						const half8 centres = for_sums(F::centre_frag(head), h), minima = for_sums(F::min_frag(head), h);
						const float dm = F::min_scale(head) * (1.0f / kSumScale);
#pragma unroll
						for (int t = 0; t < MT; ++t)
						{
							const floatx16 c = __builtin_amdgcn_mfma_f32_32x32x16_f16(sum_frag[t], centres, floatx16{}, 0, 0, 0);
							const floatx16 s = __builtin_amdgcn_mfma_f32_32x32x16_f16(sum_frag[t], minima, floatx16{}, 0, 0, 0);
#pragma unroll
							for (int e = 0; e < 16; ++e)
							{
								acc[t][e] += fmaf(d, first[t][e] + p[t][e], fmaf(d, c[e], dm * s[e]));
							}
						}
					}
					else
					{
#pragma unroll
						for (int t = 0; t < MT; ++t)
						{
#pragma unroll
							for (int e = 0; e < 16; ++e)
							{
								acc[t][e] = fmaf(d, sum[t][e], acc[t][e]);
							}
						}
					}
					// (a wavefront's LDS accesses keep their order: the slot's reads, the next chunk, its reads)
					__builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
					weights.deposit(moving, lane);
					__builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
				}
			}

			place.finish(acc, lds, xs, at, residual, m, chunks, row_bytes);
		}

		// Rows `first` .. of y_i = factor of the row times the sum over `ranges` of from_i (+ residual), in double, rounded once.  A
		// workgroup takes 1024 elements of a row (grid x) of one matrix (grid z), four a thread.  Bound by its bytes and the launch: three
		// ranges of 300 x 4096 in 4.6 us.
		constexpr int kMostRanges = fetch::kMostRanges;
		__global__ __launch_bounds__(256) void add_ranges_kernel(const ExactMats to, const ExactMats from, int ranges, size_t stride,
		                                                         const float* __restrict__ factors, const float* residual, int first)
		{
			const int row = first + static_cast<int>(blockIdx.x), which = blockIdx.z, n = to.n[which];
			const int column = (static_cast<int>(blockIdx.y) * 256 + static_cast<int>(threadIdx.x)) * 4;
			const size_t at = static_cast<size_t>(row) * n + column;
			const float* const part = from.y[which] + static_cast<size_t>(blockIdx.x) * n + column;
			float* const y = to.y[which] + at;
			const double factor = static_cast<double>(factors[row]);
			if (column + 4 <= n)
			{
				floatx4 v[kMostRanges];
#pragma unroll
				for (int i = 0; i < kMostRanges; ++i)
				{
					v[i] = i < ranges ? *reinterpret_cast<const floatx4_a4*>(part + i * stride) : floatx4{};
				}
				const floatx4 res = residual ? *reinterpret_cast<const floatx4_a4*>(residual + at) : floatx4{};
				floatx4 out;
#pragma unroll
				for (int e = 0; e < 4; ++e)
				{
					double sum = static_cast<double>(v[0][e]);
#pragma unroll
					for (int i = 1; i < kMostRanges; ++i)
					{
						sum += static_cast<double>(v[i][e]);
					}
					out[e] = static_cast<float>(fma(sum, factor, static_cast<double>(res[e])));
				}
				*reinterpret_cast<floatx4_a4*>(y) = out;
				return;
			}
			for (int e = 0; column + e < n; ++e)
			{
				double sum = 0.0;
				for (int i = 0; i < ranges; ++i)
				{
					sum += static_cast<double>(part[i * stride + e]);
				}
				y[e] = static_cast<float>(fma(sum, factor, residual ? static_cast<double>(residual[at + e]) : 0.0));
			}
		}

		// ---- few rows: up to MR activation rows, one launch, no scratch ---------------------------------
		// A workgroup takes 16 weight rows; its KS wavefronts take ranges of K and meet in LDS at the end.  Each takes
		// the activations apart by itself, a chunk of 256 at a time and with a power of two per chunk and row: a
		// lane holds four neighbouring elements of every row, and the parts go to fragments in the wavefront's LDS.
		// v_mfma_f32_16x16x32_f16 (16x16x16 where every 16 elements have a scale) with the activations as A, the high parts of row
		// i as its row i, the low ones as row 8 + i: lane (r, g) = (lane % 16, lane / 16) holds weight row r's results of
		// activation rows 4 (g % 2) .., the high parts' where g < 2 and the low ones' else, which are summed apart and meet at the end.
		// Bound by a wavefront's chain per chunk (blocks and activations into LDS, 8 products, 16 in Q6_K); a row more costs its
		// preparation, 32 instructions.  us against 32 weight rows a workgroup (below), which leave half the card idle here: Q8_0
		// 4096 x 4096 at 3 rows 10.3 -> 7.6, Q4_K 8.3 -> 6.9, Q6_K 4096 x 14336 at 2 rows 22.4 -> 15.0, at 8 rows 32.6 -> 24.5.  Error
		// against 64 bits up to 8 % lower.
		template <int MR>
		struct FewRows
		{
			static constexpr int kPart = MR * 16, kHalf = 2 * kPart + 16; // bytes of a step's part, of eight elements' parts (16: 64 banks)
			static constexpr int kSums = 32 * kHalf;                      // sub-block sums: [hi, lo][row][8 halves]
			static constexpr int kUnused = kSums + 2 * kPart; // what lanes with nothing to write write
			static constexpr int kBytes = kUnused + 256;
		};
		// A range's activations on their way into fragments in the wavefront's LDS
		template <typename F, int MR>
		struct FewActivations
		{
			typedef FewRows<MR> R;
			floatx4 xv[MR];
			const float* rows[MR];
			float unscale[MR];
			uint8_t* frags;
			uint8_t* frag_to;
			int lane, k, sum_at, sum_row, sum_low;

			__device__ __forceinline__ FewActivations(const float* x, int m, int k_, uint8_t* frags_, int lane_) : frags(frags_), lane(lane_), k(k_)
			{
#pragma unroll
				for (int i = 0; i < MR; ++i)
				{
					rows[i] = x + static_cast<size_t>(min(i, m - 1)) * k;
				}
				// lane l holds elements 4 l .. 4 l + 3: group of eight l / 2, its first or second four
				frag_to = frags + (lane >> 1) * R::kHalf + (lane & 1) * 8;
				// the sub-block sum of lanes 8 j .. 8 j + 7 is lane 8 j's to write, the others' go nowhere
				sum_at = (lane & 7) == 0 ? R::kSums + (lane >> 3) * 2 : R::kUnused + lane * 4;
				sum_row = (lane & 7) == 0 ? 16 : 0, sum_low = (lane & 7) == 0 ? R::kPart : 2;
			}
			// (nothing here may hang on a branch or look at what it loads: the next chunk's loads would be waited for at once)
			__device__ __forceinline__ void request(int c)
			{
				const int at = min(c * kChunk + 4 * lane, k - 4);
#pragma unroll
				for (int i = 0; i < MR; ++i)
				{
					xv[i] = *reinterpret_cast<const floatx4_a4*>(rows[i] + at);
				}
			}
			__device__ __forceinline__ void deposit(int c)
			{
				const bool there = F::kBlock == kChunk || c * kChunk + 4 * lane < k;
#pragma unroll
				for (int i = 0; i < MR; ++i)
				{
					float v[4];
#pragma unroll
					for (int e = 0; e < 4; ++e)
					{
						v[e] = there ? xv[i][e] : 0.0f;
					}
					// Times 2^shift the largest is in [2^14, 2^15); the inverse stays a normal number.  (An infinity leaves the row's
					// results infinite or NaN whatever becomes of the chunk's other elements, a NaN has no part in the largest.)
					const float mx = wave_max_nonnegative(fmaxf(fmaxf(fabsf(v[0]), fabsf(v[1])), fmaxf(fabsf(v[2]), fabsf(v[3]))));
					const int shift = min(141 - static_cast<int>(static_cast<uint32_t>(__float_as_int(mx)) >> 23), 126);
					const float scale = __int_as_float((127 + shift) << 23);
					unscale[i] = __int_as_float((127 - shift) << 23);
					half4 hi, lo;
					float sum = 0.0f;
#pragma unroll
					for (int e = 0; e < 4; ++e)
					{
						v[e] *= scale;
						hi[e] = static_cast<_Float16>(v[e]);
						lo[e] = static_cast<_Float16>(fmaxf((v[e] - static_cast<float>(hi[e])) * (1.0f / kLowScale), -32768.0f)); // (inf - inf: any number will do)
						sum += v[e];
					}
					*reinterpret_cast<half4*>(frag_to + 16 * i) = hi;
					*reinterpret_cast<half4*>(frag_to + R::kPart + 16 * i) = lo;
					if constexpr (F::kMins)
					{
						// eight neighbouring lanes hold one sub-block of 32 elements
						sum += dpp_f32<0xB1>(sum);
						sum += dpp_f32<0x4E>(sum);
						sum += dpp_f32<0x141>(sum);
						const float s = sum * kSumScale;
						const _Float16 high = static_cast<_Float16>(s);
						*reinterpret_cast<_Float16*>(frags + sum_at + sum_row * i) = high;
						*reinterpret_cast<_Float16*>(frags + sum_at + sum_row * i + sum_low) = static_cast<_Float16>(fmaxf((s - static_cast<float>(high)) * (1.0f / kLowScale), -32768.0f));
					}
				}
			}
		};

		constexpr int kFewTile = 16; // weight rows of a workgroup

		// What lane (r, g) multiplies of weight row r: of step s = 2 st + u elements 32 s + 8 g .. + 7, or, where kStep is 16, of step s
		// = 4 st + u elements 16 s + 4 g .. + 3.  `chunk` is the row's in the slot; st one of four stages of 64 elements.
		template <typename F>
		struct FewWeights;

		template <>
		struct FewWeights<Q4_0X>
		{
			static constexpr int kStep = 32;
			struct Head {};
			struct Raw { u32x2 q[2]; uint32_t d[2]; };
			static __device__ __forceinline__ Head head(lds_bytes_t, int) { return {}; }
			static __device__ __forceinline__ Raw load(lds_bytes_t chunk, int st, int g, int blocks)
			{
				Raw r;
#pragma unroll
				for (int u = 0; u < 2; ++u)
				{
					const int block = 2 * st + u;
					const uint32_t d = load2(chunk + 18 * block); // (there, whatever it is: not a branch)
					r.d[u] = block < blocks ? d : 0u;
					r.q[u] = load8(chunk + 8 * (g & 1), 18 * block + 2);
				}
				return r;
			}
			static __device__ __forceinline__ half8 frag(const Head&, const Raw& r, int, int u, int g)
			{
				const int sh = 4 * (g >> 1);
				return bytes_minus((r.q[u].x >> sh) & 0x0f0f0f0fu, (r.q[u].y >> sh) & 0x0f0f0f0fu, 8.0f);
			}
			static __device__ __forceinline__ float scale(const Head&, const Raw& r, int, int u) { return f16_bits_to_f32(r.d[u]); }
			static __device__ __forceinline__ float chunk_scale(const Head&) { return 1.0f; }
		};

		template <>
		struct FewWeights<Q8_0X>
		{
			static constexpr int kStep = 32;
			struct Head {};
			struct Raw { u32x2 q[2]; uint32_t d[2]; };
			static __device__ __forceinline__ Head head(lds_bytes_t, int) { return {}; }
			static __device__ __forceinline__ Raw load(lds_bytes_t chunk, int st, int g, int blocks)
			{
				Raw r;
#pragma unroll
				for (int u = 0; u < 2; ++u)
				{
					const int block = 2 * st + u;
					const uint32_t d = load2(chunk + 34 * block); // (there, whatever it is: not a branch)
					r.d[u] = block < blocks ? d : 0u;
					r.q[u] = load8(chunk + 8 * g, 34 * block + 2);
				}
				return r;
			}
			static __device__ __forceinline__ half8 frag(const Head&, const Raw& r, int, int u, int)
			{
				return bytes_minus(r.q[u].x ^ 0x80808080u, r.q[u].y ^ 0x80808080u, 128.0f);
			}
			static __device__ __forceinline__ float scale(const Head&, const Raw& r, int, int u) { return f16_bits_to_f32(r.d[u]); }
			static __device__ __forceinline__ float chunk_scale(const Head&) { return 1.0f; }
		};

		template <>
		struct FewWeights<Q4_KX>
		{
			static constexpr int kStep = 32;
			typedef Q4_KX::Head Head;
			struct Raw { u32x2 q; };
			static __device__ __forceinline__ Head head(lds_bytes_t chunk, int) { return { load16(chunk) }; }
			static __device__ __forceinline__ Raw load(lds_bytes_t chunk, int st, int g, int) { return { load8(chunk + 8 * g, 16 + 32 * st) }; }
			static __device__ __forceinline__ half8 frag(const Head& hd, const Raw& r, int st, int u, int)
			{
				const int sh = 4 * u, sub = 2 * st + u;
				const uint32_t s = (Q4_KX::scales(hd.w, sub >> 2) >> (8 * (sub & 3))) & 0xffu;
				return bytes_times((r.q.x >> sh) & 0x0f0f0f0fu, (r.q.y >> sh) & 0x0f0f0f0fu, s, Q4_KX::kCentre);
			}
			static __device__ __forceinline__ float scale(const Head&, const Raw&, int, int) { return 1.0f; }
			static __device__ __forceinline__ float chunk_scale(const Head& hd) { return Q4_KX::chunk_scale(hd); }
		};

		template <>
		struct FewWeights<Q5_KX>
		{
			static constexpr int kStep = 32;
			typedef Q5_KX::Head Head;
			struct Raw { u32x2 q; };
			static __device__ __forceinline__ Head head(lds_bytes_t chunk, int g)
			{
				const u32x2 fifth = load8(chunk + 8 * g, 16);
				return { load16(chunk), { fifth, fifth } };
			}
			static __device__ __forceinline__ Raw load(lds_bytes_t chunk, int st, int g, int) { return { load8(chunk + 8 * g, 48 + 32 * st) }; }
			static __device__ __forceinline__ half8 frag(const Head& hd, const Raw& r, int st, int u, int)
			{
				const int sh = 4 * u, sub = 2 * st + u;
				const uint32_t s = (Q4_KX::scales(hd.w, sub >> 2) >> (8 * (sub & 3))) & 0xffu;
				const u32x2 f = hd.fifth[0]; // bit `sub` of a byte is its element's fifth bit
				return bytes_times(((r.q.x >> sh) & 0x0f0f0f0fu) | (((f.x >> sub) & 0x01010101u) << 4),
				                   ((r.q.y >> sh) & 0x0f0f0f0fu) | (((f.y >> sub) & 0x01010101u) << 4), s, Q5_KX::kCentre);
			}
			static __device__ __forceinline__ float scale(const Head&, const Raw&, int, int) { return 1.0f; }
			static __device__ __forceinline__ float chunk_scale(const Head& hd) { return Q5_KX::chunk_scale(hd); }
		};

		template <>
		struct FewWeights<Q6_KX>
		{
			static constexpr int kStep = 16;
			typedef Q6_KX::Head Head;
			struct Raw { uint32_t low[2][2], high[2]; }; // half st / 2 of the block: [32 x (first, second)][16-element run]
			static __device__ __forceinline__ Head head(lds_bytes_t chunk, int) { return Q6_KX::head(chunk, 0); }
			static __device__ __forceinline__ Raw load(lds_bytes_t chunk, int st, int g, int)
			{
				typedef const __attribute__((address_space(3))) uint32_t* words_t;
				const words_t low = (words_t)(chunk + 64 * (st >> 1) + 4 * g), high = (words_t)(chunk + 128 + 32 * (st >> 1) + 4 * g);
				return { { { low[0], low[4] }, { low[8], low[12] } }, { high[0], high[4] } };
			}
			// quarter i = 2 (st % 2) + u / 2 of the half, elements 16 (u % 2) + 4 g .. of its 32
			static __device__ __forceinline__ half4 frag(const Head&, const Raw& r, int st, int u, int)
			{
				const int sh = 4 * (st & 1), top = 2 * (2 * (st & 1) + (u >> 1));
				const uint32_t v = ((r.low[u >> 1][u & 1] >> sh) & 0x0f0f0f0fu) | (((r.high[u & 1] >> top) & 0x03030303u) << 4);
				const _Float16 m = static_cast<_Float16>(-1024.0f - 32.0f);
				const half2v a = biased01(v) + half2v{ m, m }, b = biased23(v) + half2v{ m, m };
				return half4{ a.x, a.y, b.x, b.y };
			}
			static __device__ __forceinline__ float scale(const Head& hd, const Raw& r, int st, int u) { return Q6_KX::scale(hd, {}, st, u); }
			static __device__ __forceinline__ float chunk_scale(const Head& hd) { return Q6_KX::chunk_scale(hd); }
		};

		template <typename F, int MR, int KS>
		__global__ __launch_bounds__(64 * KS, 2) void exact_few_kernel(const uint8_t* __restrict__ w, const float* __restrict__ x, float* y,
		                                                            const float* residual, int n, int k, int m, int chunks, size_t row_bytes)
		{
			typedef FewRows<MR> R;
			typedef FewWeights<F> D;
			typedef WeightPieces<F, kFewTile> W;
			constexpr int NE = 4; // results of a lane
			constexpr int kSteps = 64 / D::kStep; // of a stage
			extern __shared__ __attribute__((aligned(16))) uint8_t lds[]; // [KS][slot, fragments]; later the KS sums
			const int lane = threadIdx.x & 63;
			const int part = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
			const int r = lane & 15, g = lane >> 4;
			const int n_base = blockIdx.x * kFewTile;
			const int per = (chunks + KS - 1) / KS;
			const int c_begin = part * per, c_end = min(c_begin + per, chunks);
			uint8_t* const mine = lds + part * (W::kSlotBytes + R::kBytes);
			uint8_t* const frags = mine + W::kSlotBytes;
			const W weights(mine, w, n_base, n, row_bytes);

			FewActivations<F, MR> xs(x, m, k, frags, lane);
			// A's row r: high parts of activation row r, low ones of row r - 8 (rows that are not there repeat the last)
			const uint8_t* const frag_row = frags + (r >> 3) * R::kPart + min(r & 7, m - 1) * 16;
			const uint8_t* const frag_from = D::kStep == 32 ? frag_row + g * R::kHalf : frag_row + (g >> 1) * R::kHalf + (g & 1) * 8;
			const uint8_t* const sums_from = frags + R::kSums + (r >> 3) * R::kPart + min(r & 7, m - 1) * 16;

			float acc[2][NE] = {}; // of every other chunk
			u32x4 moving[2][W::kLoads]; // the next two chunks
			if (c_begin < c_end)
			{
				weights.request(moving[0], c_begin, lane);
				xs.request(c_begin);
				weights.request(moving[1], min(c_begin + 1, c_end - 1), lane);
			}
			const auto step = [&](int c, u32x4 (&arrived)[W::kLoads], float (&acc)[NE]) {
				weights.deposit(arrived, lane);
				xs.deposit(c);
				xs.request(min(c + 1, c_end - 1));
				weights.request(arrived, min(c + 2, c_end - 1), lane);
				__builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront"); // (a wavefront's LDS accesses keep their order)
				const int blocks = k / F::kBlock - c * (kChunk / F::kBlock);
				lds_bytes_t const chunk = weights.chunk(lane);
				const typename D::Head head = D::head(chunk, g);
				floatx4 stage, sum[2]; // sum: of the chunk's halves (two shorter chains round less)
#pragma unroll
				for (int st = 0; st < 4; ++st)
				{
					const typename D::Raw raw = D::load(chunk, st, g, blocks);
					floatx4& half = sum[st >> 1];
#pragma unroll
					for (int u = 0; u < kSteps; ++u)
					{
						const int at = kSteps * st + u;
						floatx4 p;
						if constexpr (D::kStep == 32)
						{
							const half8 a = *reinterpret_cast<const half8*>(frag_from + 4 * at * R::kHalf);
							p = __builtin_amdgcn_mfma_f32_16x16x32_f16(a, D::frag(head, raw, st, u, g), floatx4{}, 0, 0, 0);
						}
						else
						{
							const half4 a = *reinterpret_cast<const half4*>(frag_from + 2 * at * R::kHalf);
							p = __builtin_amdgcn_mfma_f32_16x16x16f16(a, D::frag(head, raw, st, u, g), floatx4{}, 0, 0, 0);
						}
						if constexpr (F::kMins)
						{
							stage = u == 0 ? p : stage + p;
							if (u == kSteps - 1)
							{
								half = (st & 1) == 0 ? stage : half + stage;
							}
						}
						else
						{
							const float d = D::scale(head, raw, st, u);
#pragma unroll
							for (int e = 0; e < NE; ++e)
							{
								half[e] = (st & 1) == 0 && u == 0 ? d * p[e] : fmaf(d, p[e], half[e]);
							}
						}
					}
				}
				const float d = D::chunk_scale(head);
				floatx4 total = sum[0] + sum[1];
				if constexpr (F::kMins)
				{
					// eight sums of a row's high or low parts; the high ones' products are short enough to be summed exactly
					const half8 sums = g == 0 ? *reinterpret_cast<const half8*>(sums_from) : half8{};
					const floatx4 centre = __builtin_amdgcn_mfma_f32_16x16x32_f16(sums, F::centre_frag(head), floatx4{}, 0, 0, 0);
					const floatx4 s = __builtin_amdgcn_mfma_f32_16x16x32_f16(sums, F::min_frag(head), floatx4{}, 0, 0, 0);
					const float dm = F::min_scale(head) * (1.0f / kSumScale);
#pragma unroll
					for (int e = 0; e < NE; ++e)
					{
						total[e] = fmaf(d, total[e], fmaf(d, centre[e], dm * s[e]));
					}
				}
				else
				{
					total *= d;
				}
#pragma unroll
				for (int e = 0; e < NE; ++e)
				{
					const float even = xs.unscale[e < MR ? e : 0], odd = xs.unscale[e + 4 < MR ? e + 4 : 0]; // (values: a choice of places would keep them in memory)
					acc[e] = fmaf(total[e], g & 1 ? odd : even, acc[e]);
				}
				__builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
			};
			for (int c = c_begin; c < c_end; c += 2)
			{
				step(c, moving[0], acc[0]);
				if (c + 1 < c_end)
				{
					step(c + 1, moving[1], acc[1]);
				}
			}
			__syncthreads();
			float* const handed = reinterpret_cast<float*>(lds); // [KS][activation row][weight row]
#pragma unroll
			for (int e = 0; e < NE; ++e)
			{
				const int row = 4 * (g & 1) + e;
				const float high = acc[0][e] + acc[1][e], low = __shfl_xor(high, 32, 64);
				if (g < 2 && row < m)
				{
					handed[(part * MR + row) * kFewTile + r] = fmaf(low, kLowScale, high);
				}
			}
			__syncthreads();
			for (int i = threadIdx.x; i < m * kFewTile; i += 64 * KS)
			{
				const int row = i / kFewTile, col = n_base + i % kFewTile;
				float ranges[KS];
#pragma unroll
				for (int p = 0; p < KS; ++p)
				{
					ranges[p] = handed[p * MR * kFewTile + i];
				}
				add_in_pairs(ranges);
				float v = ranges[0];
				if (col < n)
				{
					if constexpr (F::kMins)
					{
						if (__builtin_expect(!(fabsf(v) <= 3.402823466e38f), 0))
						{
							const float* const from = x + static_cast<size_t>(row) * k;
							v = plain_dot<F>(w + static_cast<size_t>(col) * row_bytes, chunks, [&](int i) { return from[i]; });
						}
					}
					const size_t o = static_cast<size_t>(row) * n + col;
					y[o] = residual ? residual[o] + v : v;
				}
			}
		}

		// The same where there are many weight rows: 32 of them share a wavefront's preparation of the activations, on
		// v_mfma_f32_32x32x16_f16 with rows 0 .. MR - 1 of a fragment the high parts and 16 .. 16 + MR - 1 the low ones, so that one
		// product forms both; their sums lie in one lane (elements e and e + 8 of the result).  us at 3 rows, 16 rows a
		// workgroup and 32: 14336 x 4096 Q8_0 19.3 and 18.0, Q4_K 17.7 and 14.8, 12000 x 8192 24.9 and 23.6; 6000 x 2048 6.7 and 5.3.
		template <typename F, int MR, int KS>
		__global__ __launch_bounds__(64 * KS, 2) void exact_few_wide_kernel(const uint8_t* __restrict__ w, const float* __restrict__ x, float* y,
		                                                            const float* residual, int n, int k, int m, int chunks, size_t row_bytes)
		{
			typedef FewRows<MR> R;
			typedef WeightPieces<F> W;
			constexpr int NE = 4; // results of a lane
			extern __shared__ __attribute__((aligned(16))) uint8_t lds[]; // [KS][slot, fragments]; later the KS sums
			const int lane = threadIdx.x & 63;
			const int part = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
			const int r = lane & 31, h = lane >> 5;
			const int n_base = blockIdx.x * kTile;
			const int per = (chunks + KS - 1) / KS;
			const int c_begin = part * per, c_end = min(c_begin + per, chunks);
			uint8_t* const mine = lds + part * (W::kSlotBytes + R::kBytes);
			uint8_t* const frags = mine + W::kSlotBytes;
			const W weights(mine, w, n_base, n, row_bytes);

			FewActivations<F, MR> xs(x, m, k, frags, lane);
			const uint8_t* const frag_from = frags + h * R::kHalf + (r >> 4) * R::kPart + min(r & 15, m - 1) * 16;
			const uint8_t* const sums_from = frags + R::kSums + h * R::kPart + min(r & 15, m - 1) * 16;

			float acc[2][NE] = {}; // of every other chunk
			u32x4 moving[2][W::kLoads]; // the next two chunks
			if (c_begin < c_end)
			{
				weights.request(moving[0], c_begin, lane);
				xs.request(c_begin);
				weights.request(moving[1], min(c_begin + 1, c_end - 1), lane);
			}
			const auto step = [&](int c, u32x4 (&arrived)[W::kLoads], float (&acc)[NE]) {
				weights.deposit(arrived, lane);
				xs.deposit(c);
				xs.request(min(c + 1, c_end - 1));
				weights.request(arrived, min(c + 2, c_end - 1), lane);
				__builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront"); // (a wavefront's LDS accesses keep their order)
				lds_bytes_t const chunk = weights.chunk(lane);
				const typename F::Head head = F::head(chunk, h);
				const int blocks = k / F::kBlock - c * (kChunk / F::kBlock);
				floatx16 p;
				float sum[NE], low[NE]; // low: the low parts', where kScaleSteps is 16
#pragma unroll
				for (int st = 0; st < 4; ++st)
				{
					const typename F::Raw raw = F::load(chunk, st, h, blocks);
#pragma unroll
					for (int s = 0; s < 4; ++s)
					{
						const int at = 4 * st + s;
						const half8 a = *reinterpret_cast<const half8*>(frag_from + 2 * at * R::kHalf);
						p = __builtin_amdgcn_mfma_f32_32x32x16_f16(a, F::frag(head, raw, st, s), at % min(F::kScaleSteps, 4) == 0 ? floatx16{} : p, 0, 0, 0);
						if constexpr (F::kMins)
						{
							if (s == 3)
							{
#pragma unroll
								for (int e = 0; e < NE; ++e)
								{
									sum[e] = st == 0 ? p[e] : sum[e] + p[e];
									low[e] = st == 0 ? p[e + 8] : low[e] + p[e + 8];
								}
							}
						}
						if constexpr (F::kScaleSteps < 16)
						{
							if (at % F::kScaleSteps == F::kScaleSteps - 1)
							{
								const float d = F::scale(head, raw, st, s);
#pragma unroll
								for (int e = 0; e < NE; ++e)
								{
									const float both = fmaf(p[e + 8], kLowScale, p[e]);
									sum[e] = at == F::kScaleSteps - 1 ? d * both : fmaf(d, both, sum[e]);
								}
							}
						}
						if constexpr (F::kScaleSteps < 16)
						{
							// (the stage's sums now and not later: all stages' products at once are more than the registers hold)
							if (s == 3)
							{
#pragma unroll
								for (int e = 0; e < NE; ++e)
								{
									asm volatile("" : "+v"(sum[e]));
								}
							}
						}
					}
				}
				const float d = F::chunk_scale(head);
				if constexpr (F::kMins)
				{
					const half8 sums = r < 16 ? *reinterpret_cast<const half8*>(sums_from) : half8{}; // (into the high parts' rows alone)
					const floatx16 centre = __builtin_amdgcn_mfma_f32_32x32x16_f16(sums, for_sums(F::centre_frag(head), h), floatx16{}, 0, 0, 0);
					const floatx16 s = __builtin_amdgcn_mfma_f32_32x32x16_f16(sums, for_sums(F::min_frag(head), h), floatx16{}, 0, 0, 0);
					const float dm = F::min_scale(head) * (1.0f / kSumScale);
#pragma unroll
					for (int e = 0; e < NE; ++e)
					{
						sum[e] = fmaf(d, fmaf(low[e], kLowScale, sum[e]), fmaf(d, centre[e], dm * s[e]));
					}
				}
				else
				{
#pragma unroll
					for (int e = 0; e < NE; ++e)
					{
						sum[e] = d * sum[e];
					}
				}
				// lane (r, h) holds weight row r and activation rows 8 (e / 4) + 4 h + e % 4
#pragma unroll
				for (int e = 0; e < NE; ++e)
				{
					const int row = 8 * (e / 4) + (e & 3);
					const float low4 = xs.unscale[row < MR ? row : 0], high4 = xs.unscale[row + 4 < MR ? row + 4 : 0];
					acc[e] = fmaf(sum[e], h ? high4 : low4, acc[e]);
				}
				__builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
			};
			for (int c = c_begin; c < c_end; c += 2)
			{
				step(c, moving[0], acc[0]);
				if (c + 1 < c_end)
				{
					step(c + 1, moving[1], acc[1]);
				}
			}
			__syncthreads();
			float* const handed = reinterpret_cast<float*>(lds); // [KS][activation row][weight row]
#pragma unroll
			for (int e = 0; e < NE; ++e)
			{
				const int row = 8 * (e / 4) + 4 * h + (e & 3);
				if (row < m)
				{
					handed[(part * MR + row) * kTile + r] = acc[0][e] + acc[1][e];
				}
			}
			__syncthreads();
			for (int i = threadIdx.x; i < m * kTile; i += 64 * KS)
			{
				const int row = i / kTile, col = n_base + i % kTile;
				float ranges[KS];
#pragma unroll
				for (int p = 0; p < KS; ++p)
				{
					ranges[p] = handed[p * MR * kTile + i];
				}
				add_in_pairs(ranges);
				float v = ranges[0];
				if (col < n)
				{
					if constexpr (F::kMins)
					{
						if (__builtin_expect(!(fabsf(v) <= 3.402823466e38f), 0))
						{
							const float* const from = x + static_cast<size_t>(row) * k;
							v = plain_dot<F>(w + static_cast<size_t>(col) * row_bytes, chunks, [&](int i) { return from[i]; });
						}
					}
					const size_t o = static_cast<size_t>(row) * n + col;
					y[o] = residual ? residual[o] + v : v;
				}
			}
		}

		struct ExactCall
		{
			int count;
			const uint8_t* w[3];
			float* y[3];
			int n[3];
			int total_rows; // of all matrices
			const uint8_t* xs;
			const float* residual;
			int k, m, m_tiles, chunks;
			size_t row_bytes;
			hipStream_t stream;
			float* partial; // room for the sums of K's ranges, or null
			size_t partial_floats;
		};

		// the matrices, `rows` weight rows a workgroup, side by side in grid x
		ExactMats grid_mats(const ExactCall& c, int rows, int& blocks)
		{
			ExactMats mats{};
			blocks = 0;
			for (int i = 0; i < 3; ++i)
			{
				mats.first_block[i] = 0x7fffffff;
				if (i < c.count)
				{
					mats.w[i] = c.w[i];
					mats.y[i] = c.y[i];
					mats.n[i] = c.n[i];
					mats.first_block[i] = blocks;
					blocks += (c.n[i] + rows - 1) / rows;
				}
			}
			return mats;
		}

		template <typename F, int MT, int WN, int KS, bool ONE_RUN = WN == 1>
		void launch_variant(const ExactCall& c)
		{
			constexpr size_t rings = (WN > 1 ? static_cast<size_t>(KS) * 2 * MT * kStageBytes : 0) +
			                         static_cast<size_t>(WN) * KS * WeightPieces<F>::kSlotBytes;
			constexpr size_t sums = static_cast<size_t>(KS - 1) * WN * MT * 64 * 64;
			constexpr size_t lds = rings > sums ? rings : sums;
			static_assert(lds <= 160 * 1024, "LDS");
			int blocks;
			const ExactMats mats = grid_mats(c, WN * kTile, blocks);
			const auto kernel = &exact_gemm_kernel<F, MT, WN, KS, ONE_RUN>;
			allow_dynamic_lds(reinterpret_cast<const void*>(kernel), lds);
			kernel<<<dim3(blocks, (c.m_tiles + MT - 1) / MT), dim3(64 * WN * KS), lds, c.stream>>>(
			    mats, c.xs, c.residual, c.k, c.m, c.m_tiles, c.chunks, c.row_bytes);
		}

		// RANGES: `ranges` of K in grid z, none of them empty, leave their sums in c.partial, from where a launch more adds them, for
		// as many rows at a time as fetch::ranged_rows says
		template <typename F, int KS, bool RANGES = false>
		void launch_shared(const ExactCall& c, int flush, int ranges = 1)
		{
			constexpr int MT = 2, WN = 4;
			constexpr size_t rings = static_cast<size_t>(KS) * kRing * MT * kStageBytes + static_cast<size_t>(WN) * KS * WeightPieces<F>::kSlotBytes;
			constexpr size_t sums = static_cast<size_t>(KS - 1) * WN * MT * 64 * 64;
			constexpr size_t lds = rings > sums ? rings : sums;
			static_assert(lds <= (KS == 1 ? 80 : 160) * 1024, "LDS");
			int blocks;
			ExactMats mats = grid_mats(c, WN * kTile, blocks);
			constexpr auto kernel = &exact_shared_kernel<F, MT, WN, KS, RANGES>;
			allow_dynamic_lds(reinterpret_cast<const void*>(kernel), lds);
			if constexpr (!RANGES)
			{
				kernel<<<dim3(blocks, (c.m_tiles + MT - 1) / MT), dim3(64 * WN * KS), lds, c.stream>>>(
				    mats, c.xs, c.residual, c.k, c.m, c.m_tiles, c.chunks, c.row_bytes, flush, 0, 0);
				return;
			}
			const ExactMats out = mats;
			const int rows = fetch::ranged_rows(ranges, c.total_rows, c.m);
			const size_t stride = static_cast<size_t>(rows) * c.total_rows;
			size_t at = 0;
			for (int i = 0; i < c.count; ++i)
			{
				mats.y[i] = c.partial + at;
				at += static_cast<size_t>(rows) * c.n[i];
			}
			const unsigned widest = static_cast<unsigned>(*std::max_element(c.n, c.n + c.count));
			const float* const factors = reinterpret_cast<const float*>(c.xs + RowsLayout(c.m_tiles, c.chunks).factors);
			for (int first = 0; first < c.m; first += rows)
			{
				const int here = std::min(rows, c.m - first);
				kernel<<<dim3(blocks, (here + MT * kTile - 1) / (MT * kTile), ranges), dim3(64 * WN * KS), lds, c.stream>>>(
				    mats, c.xs, nullptr, c.k, c.m, c.m_tiles, c.chunks, c.row_bytes, flush, stride, first);
				add_ranges_kernel<<<dim3(here, (widest + 1023) / 1024, c.count), dim3(256), 0, c.stream>>>(out, mats, ranges, stride, factors, c.residual, first);
			}
		}

		// Formats whose weights' slots leave a CU room for two workgroups of the shared form.  (Q4_0 takes fewer bytes, but its sums,
		// scaled every other step, spill registers there: 104 -> 288 us.)
		template <typename F>
		constexpr bool kShares = F::kMins || F::kScaleSteps == 1;

		template <typename F>
		void launch_exact_format(const ExactCall& c)
		{
			const int strips = (c.total_rows + kTile - 1) / kTile, units = strips * c.m_tiles;
			const int workgroups = (strips + 3) / 4 * ((c.m_tiles + 1) / 2);
			// Where 128 x 64 tiles give most CUs a workgroup, four wavefronts share the activations and each decoded weight meets two
			// tiles (us, kernel alone, weights from HBM, here and below): Q4_K 28672 x 4096 at 300 rows 226 against 313 of the
			// forms below, at 64 rows 47 against 64; and from there on in one range of K, four wavefronts each, two workgroups to a CU:
			// one's barriers, sums and results go beside the other's products (672 workgroups of Q5_K 139 -> 131, 448 of Q4_K 83 -> 75,
			// 1120 217 -> 191; one to a CU they have nobody beside them: 240 47 and 49).  The same sums.
			if constexpr (kShares<F>)
			{
				const int ranges = fetch::exact_ranges(F::kScaleSteps == 1, c.total_rows, c.m, c.chunks);
				if (ranges > 1 && static_cast<size_t>(ranges) * fetch::ranged_rows(ranges, c.total_rows, c.m) * c.total_rows <= c.partial_floats)
				{
					return launch_shared<F, 1, true>(c, fetch::chunks_a_sum((c.chunks + ranges - 1) / ranges).chunks, ranges);
				}
			}
			if constexpr (F::kMins)
			{
				if (workgroups >= 200 && c.m_tiles > 1)
				{
					return workgroups > 256 ? launch_shared<F, 1>(c, (c.chunks + 1) / 2) : launch_shared<F, 2>(c, c.chunks);
				}
			}
			else if constexpr (F::kScaleSteps > 1)
			{
				if (workgroups >= 200 && c.m_tiles > 1)
				{
					return launch_variant<F, 2, 4, 2>(c);
				}
			}
			// Otherwise a wavefront keeps to itself and the ranges of K fill the card, in Q6_K with two tiles where these are enough.
			if constexpr (F::kScaleSteps == 1)
			{
				if (fetch::exact_two_tiles(strips, c.m_tiles))
				{
					return launch_variant<F, 2, 1, 8>(c);
				}
			}
			// Eight ranges while there are few tiles (Q6_K 4096 x 14336 at 45 rows 41 against 46 with four, at 16 43 against 47), four
			// from there on (Q4_K 14336 x 4096 at 45 rows 37 against 44 with eight, at 16 equal) and for short rows (Q8_0 1024 x 1024 at
			// 16 rows 5.8 against 6.0).
			if (units <= 256 && c.chunks >= 8)
			{
				return launch_variant<F, 1, 1, 8>(c);
			}
			// Stage by stage where many tiles of activations meet few strips: in one run wavefronts drift apart, and loads of what others
			// brought into L2 come too late (Q4_0 512 x 8192, 1000 rows: 2.6 and 4.0 million misses).  us of stages and of a run: that
			// one 78 and 100, Q4_K 1024 x 8192, 777 rows 106 and 129, 2048 x 8192, 640 rows 140 and 164, 4096 x 4096, 300 rows 60 and 59;
			// the other way round 14336 x 4096, 45 rows 41.6 and 39.9, Q8_0 45.7 and 44.0.
			if constexpr (F::kScaleSteps > 1)
			{
				if (units > 256 && 12 * c.m_tiles >= strips)
				{
					return launch_variant<F, 1, 1, 4, false>(c);
				}
			}
			launch_variant<F, 1, 1, 4>(c);
		}

		struct FewCall
		{
			const uint8_t* w;
			const float* x;
			float* y;
			const float* residual;
			int n, k, m, chunks;
			size_t row_bytes;
			hipStream_t stream;
		};

		// tile: weight rows of a workgroup
		template <typename F, int MR, int KS, int TILE>
		void launch_few(const FewCall& c)
		{
			constexpr size_t parts = static_cast<size_t>(KS) * (WeightPieces<F, TILE>::kSlotBytes + FewRows<MR>::kBytes);
			constexpr size_t sums = static_cast<size_t>(KS) * MR * TILE * sizeof(float);
			constexpr size_t lds = parts > sums ? parts : sums;
			static_assert(lds <= 160 * 1024, "LDS");
			constexpr auto kernel = TILE == kFewTile ? &exact_few_kernel<F, MR, KS> : &exact_few_wide_kernel<F, MR, KS>;
			allow_dynamic_lds(reinterpret_cast<const void*>(kernel), lds);
			kernel<<<dim3((c.n + TILE - 1) / TILE), dim3(64 * KS), lds, c.stream>>>(c.w, c.x, c.y, c.residual, c.n, c.k, c.m, c.chunks, c.row_bytes);
		}

		template <typename F, int MR>
		void launch_few_rows(const FewCall& c)
		{
			// Sixteen weight rows a workgroup while each has a CU to itself (us at 3 rows, sixteen and 32: Q8_0 4096 x 4096 7.6 and 10.3,
			// 1024 x 4096 6.1 and 8.2, Q6_K 4096 x 14336 16.8 and 24.8; in a second round not: 6000 x 2048 9.0 and 7.7), in eight ranges of K.
			if (c.n <= 256 * kFewTile)
			{
				launch_few<F, MR, 8, kFewTile>(c);
			}
			// Eight ranges of K where 8192 weight rows and fewer leave CUs idle, else four (Q4_0 11008 x 4096 16.4 and 14.3).
			else if (c.n <= 8192 && c.chunks >= 8)
			{
				launch_few<F, MR, 8, kTile>(c);
			}
			else
			{
				launch_few<F, MR, 4, kTile>(c);
			}
		}

		template <typename F>
		void launch_few_format(const FewCall& c)
		{
			switch (c.m)
			{
			case 2: launch_few_rows<F, 2>(c); break;
			case 3: launch_few_rows<F, 3>(c); break;
			case 4: launch_few_rows<F, 4>(c); break;
			case 5: case 6: launch_few_rows<F, 6>(c); break;
			default: launch_few_rows<F, 8>(c); break;
			}
		}
	} // namespace

	// bytes of scratch the rows of an m x k activation matrix take
	size_t exact_scratch_bytes(size_t m, size_t k)
	{
		const size_t tiles = (m + kTile - 1) / kTile, chunks = (k + kChunk - 1) / kChunk;
		return RowsLayout(tiles, chunks).bytes;
	}

	// Whether launch_exact_rows takes rows of this number and width.
	bool exact_rows_take(size_t m, size_t k)
	{
		return m > 0 && m <= (size_t{ 1 } << 20) && k > 0 && k % 32 == 0 && k <= static_cast<size_t>(kMostItems) * 8;
	}

	// Whether launch_exact_gemm takes a matrix: one of the formats above, rows that start on 2 bytes.
	bool exact_gemm_takes(int fmt, const void* wq, size_t n, size_t k)
	{
		switch (fmt)
		{
		case LITENN_FMT_Q4_0: case LITENN_FMT_Q8_0: case LITENN_FMT_Q4_K: case LITENN_FMT_Q5_K: case LITENN_FMT_Q6_K: break;
		default: return false;
		}
		return n > 0 && n <= 0x3fffffffu && row_bytes(fmt, k) != 0 && row_bytes(fmt, k) < (size_t{ 1 } << 25) && reinterpret_cast<uintptr_t>(wq) % 2 == 0;
	}

	// Takes the rows of X' = x, RMSNorm(x) * norm_w or silu(x) * up apart into `scratch` (exact_scratch_bytes,
	// 16-byte aligned) for any number of launch_exact_gemm calls of the same m and k.  Returns false, launching
	// nothing, for rows it does not take.
	bool launch_exact_rows(const float* x, size_t m, size_t k, const float* norm_w, double eps, const float* up, void* scratch,
	                       hipStream_t stream)
	{
		const auto aligned = [](const void* p) { return reinterpret_cast<uintptr_t>(p) % 16 == 0; };
		if (!scratch || !exact_rows_take(m, k) || !aligned(x) || !aligned(scratch) || !aligned(norm_w) || !aligned(up) || (norm_w && up))
		{
			return false;
		}
		const int chunks = static_cast<int>((k + kChunk - 1) / kChunk);
		const int m_pad = static_cast<int>((m + kTile - 1) / kTile * kTile);
		const auto launch = [&](auto kernel, int threads) {
			kernel<<<dim3(static_cast<unsigned>((m_pad + 63) / 64 * 64)), dim3(threads), 0, stream>>>(
			    x, static_cast<uint8_t*>(scratch), static_cast<int>(m), m_pad, static_cast<int>(k), chunks, norm_w, eps, up);
		};
		// Few rows leave a workgroup a CU to itself: more threads, fewer elements in a chain, and it pays at every width (us, 256 /
		// 512 / 1024 threads: 64 rows of 14336 10.8, 8.7, 8.3, of 4096 5.9, 5.0, 4.8, of 2048 5.0, 4.3, 4.0, of 1024 4.9, 4.1, 3.9; 9 of
		// 1024 4.2, 3.6, 3.5; 128 of 1024 5.1, 4.3, 4.1); beyond 256 rows they share a CU (300 rows of 14336 14.2, 13.0, 14.0, of 4096
		// 9.3, 9.2, 9.4, of 1024 6.6, 6.0, 6.7).  From 129 to 256 the two are 0.1 to 0.4 apart.
		if (m <= 128)
		{
			launch(&split_rows_kernel<1024>, 1024);
		}
		else
		{
			launch(&split_rows_kernel<512>, 512);
		}
		return true;
	}

	// ranges of K that launch_exact_gemm leaves sums of, where it has room for them
	static int exact_ranges(int fmt, size_t n, size_t k, size_t m)
	{
		return fmt == LITENN_FMT_Q4_K || fmt == LITENN_FMT_Q5_K || fmt == LITENN_FMT_Q6_K
		           ? fetch::exact_ranges(fmt == LITENN_FMT_Q6_K, static_cast<int>(n), static_cast<int>(m), static_cast<int>((k + kChunk - 1) / kChunk))
		           : 1;
	}

	// floats that it leaves them in (0: it takes K in one)
	size_t exact_partial_floats(int fmt, size_t n, size_t k, size_t m)
	{
		const int ranges = exact_ranges(fmt, n, k, m);
		return ranges > 1 ? static_cast<size_t>(ranges) * fetch::ranged_rows(ranges, static_cast<int>(n), static_cast<int>(m)) * n : 0;
	}

	// the same for any number of rows up to m
	size_t exact_most_partial_floats(int fmt, size_t n, size_t k, size_t m)
	{
		// beyond 256 workgroups of 128 x 64 results there is one number of ranges, and as many rows as go at a time take most; up to
		// there every number of tiles has its own, and the fewer rows it holds the sooner they pay
		const size_t blocks = (n + 4 * kTile - 1) / (4 * kTile), last = std::min(m, 64 * (256 / std::max<size_t>(blocks, 1)));
		size_t most = 0;
		if (const int ranges = exact_ranges(fmt, n, k, m); m > last && ranges > 1)
		{
			most = static_cast<size_t>(ranges) * std::min<size_t>(m, fetch::ranged_rows_whole(ranges, static_cast<int>(n))) * n;
		}
		for (size_t first = 1; first <= last; first += kTile)
		{
			const int ranges = exact_ranges(fmt, n, k, first);
			most = std::max(most, ranges > 1 ? static_cast<size_t>(ranges) * std::min(m, first + kTile - 1) * n : 0);
		}
		return most;
	}

	// y_i[M, n_i] = X' . deq(W_i)^T (+ residual, which may alias y; single matrix) for up to three matrices of
	// one format over rows that launch_exact_rows has taken apart.  partial: room for sums of ranges of K, or null.
	void launch_exact_gemm(int fmt, int count, const void* const* wq, const size_t* n, size_t k, size_t m, float* const* y,
	                       const float* residual, const void* scratch, float* partial, size_t partial_floats, hipStream_t stream)
	{
		ExactCall c{};
		c.partial = partial;
		c.partial_floats = partial ? partial_floats : 0;
		c.count = count;
		for (int i = 0; i < count; ++i)
		{
			c.w[i] = static_cast<const uint8_t*>(wq[i]);
			c.y[i] = y[i];
			c.n[i] = static_cast<int>(n[i]);
			c.total_rows += c.n[i];
		}
		c.xs = static_cast<const uint8_t*>(scratch);
		c.residual = residual;
		c.k = static_cast<int>(k);
		c.m = static_cast<int>(m);
		c.m_tiles = static_cast<int>((m + kTile - 1) / kTile);
		c.chunks = static_cast<int>((k + kChunk - 1) / kChunk);
		c.row_bytes = row_bytes(fmt, k);
		c.stream = stream;
		switch (fmt)
		{
		case LITENN_FMT_Q4_0: launch_exact_format<Q4_0X>(c); break;
		case LITENN_FMT_Q8_0: launch_exact_format<Q8_0X>(c); break;
		case LITENN_FMT_Q4_K: launch_exact_format<Q4_KX>(c); break;
		case LITENN_FMT_Q5_K: launch_exact_format<Q5_KX>(c); break;
		default: launch_exact_format<Q6_KX>(c); break;
		}
	}

	// Y[M, N] = X . deq(W)^T (+ residual, which may alias y) for 2 to 8 rows, a matrix that exact_gemm_takes.
	// Returns false, launching nothing, for others.
	bool launch_exact_few(int fmt, const void* wq, size_t n, size_t k, const float* x, size_t m, float* y, const float* residual,
	                      hipStream_t stream)
	{
		if (m < 2 || m > 8 || k < 4)
		{
			return false;
		}
		const FewCall c{ static_cast<const uint8_t*>(wq), x, y, residual, static_cast<int>(n), static_cast<int>(k), static_cast<int>(m),
			             static_cast<int>((k + kChunk - 1) / kChunk), row_bytes(fmt, k), stream };
		switch (fmt)
		{
		case LITENN_FMT_Q4_0: launch_few_format<Q4_0X>(c); break;
		case LITENN_FMT_Q8_0: launch_few_format<Q8_0X>(c); break;
		case LITENN_FMT_Q4_K: launch_few_format<Q4_KX>(c); break;
		case LITENN_FMT_Q5_K: launch_few_format<Q5_KX>(c); break;
		default: launch_few_format<Q6_KX>(c); break;
		}
		return true;
	}
} // namespace litenn_hip
