// Attention of many query rows with Float32 operands on the matrix cores: the prompt's attention under
// LITENN_HIP_MATMUL_PRECISE, the reference layer with its options (src/LiteNN/Layer/FlashAttnExt.h:100-228) and
// the layered decoders' windows in 32 bits.  The row kernels this stands beside read every key once per query row.
//
//   S^T[key, q]  = K[key, :] . Q[q, :]        A = keys (row-major in LDS), B = queries (registers)
//   O^T[d, q]   += V^T[d, key] . P^T[key, q]  A = values, read transposed from LDS, B = weights (registers)
//
// on v_mfma_f32_32x32x16: a query stays in its lane column through both products, so its running maximum and sum
// live beside its outputs, and the weights leave the first product in the registers the second one takes (the
// order of the keys inside a step is chosen to match; ds_read_b64_tr_b16 turns four keys' rows into the value
// operand).  No operand is rounded to 16 bits:
//   * Float16 keys and values are exact; a query (its row scaled to 2^14) and a softmax weight (times 2^14) are two halves
//     each, hi + lo / 4096, off by 2^-24 of itself at most down to 2^-27 of the row's largest (of a weight of 1), and by
//     2^-51 of that below: two products per operand pair, in a sum each.
//   * Float32 keys, values, queries and weights are three bfloat16 values each, exactly; of their nine products the three
//     below 2^-26 of the pair's, a quarter of what a Float32 rounding takes, are left out.
// Scores, softmax and sums are Float32 as in the row kernels.
//
// A tile is one chain in its wavefront (16 products, softmax, 16 products) that the vector ALUs bound: 600 instructions at four
// cycles beside 1024 cycles of products.  So what counts is how few there are (a whole tile's rows lie at one distance from a
// uniform address, weights take an exponential for arguments of one sign, places in LDS are a register and a constant), that two
// wavefronts fit a SIMD (256 registers: one of keys and values is in flight at a time, the second halves of the queries are in LDS
// where all wavefronts have the same), that no load hangs on a branch, and that every wavefront has its own keys, with no barrier.
// 200 rows on 1000 keys (32 heads of 128 over 8) with mask, slopes, soft cap and sinks take 27.6 us (38.5 with 1000 instructions a
// tile, 31 registers spilled and the groups merged by one of them), where the row kernel took 1365; causal, with Float32 keys and
// values (three times the products, one wavefront a SIMD), 57 (85 in pairs of wavefronts that share their keys, on half the SIMDs).
// Sums are short chains: scores in two sums, the parts' small products in one of their own, the weights' sum as a tree, outputs one
// addition per tile, which costs 4 us and leaves the error against 64 bits below the row kernel's (mean of six inputs, 1e-7:
// these rows 1.30 and, the tangent in the layer's form throughout, 3.78, 150 rows on 700 keys 1.86 and 2.02, with Float32 keys 1.64 and 2.03).
#include "common.hpp"
#include "attn_math.hpp"
#include "layer_device.hpp"
#include "attn_rows.hpp"
#include "fetch_model.hpp"

#include <cmath>

namespace litenn_hip
{
	namespace
	{
		typedef _Float16 half8 __attribute__((ext_vector_type(8)));
		typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
		typedef short short4v __attribute__((ext_vector_type(4)));
		typedef float floatx16 __attribute__((ext_vector_type(16)));
		typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
		typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));

		constexpr int kKeys = 32; // keys of a tile, queries of a wavefront

		// How a Float32 operand is taken apart, and which products of the parts are formed
		struct HalfOperands // keys and values as they are
		{
			typedef half8 frag;
			typedef uint16_t stored;
			static constexpr int kStored = 1, kSplit = 2, kProducts = 2; // pieces of a key or value, of a query or weight
			static constexpr int stored_of[2] = { 0, 0 }, split_of[2] = { 0, 1 };
			static constexpr float kWeightScale = 16384.0f, kLowScale = 1.0f / 4096.0f;
			static __device__ __forceinline__ void split(float v, int e, frag (&out)[2])
			{
				out[0][e] = static_cast<_Float16>(v);
				out[1][e] = static_cast<_Float16>((v - static_cast<float>(out[0][e])) * (1.0f / kLowScale));
			}
			static __device__ __forceinline__ floatx16 multiply(frag a, frag b, floatx16 c)
			{
				return __builtin_amdgcn_mfma_f32_32x32x16_f16(a, b, c, 0, 0, 0);
			}
		};
		struct FloatOperands
		{
			typedef bf16x8 frag;
			typedef float stored;
			static constexpr int kStored = 3, kSplit = 3, kProducts = 6;
			static constexpr int stored_of[6] = { 0, 0, 1, 1, 0, 2 }, split_of[6] = { 0, 1, 0, 1, 2, 0 };
			static constexpr float kWeightScale = 1.0f, kLowScale = 1.0f;
			static __device__ __forceinline__ void split(float v, int e, frag (&out)[3])
			{
				out[0][e] = static_cast<__bf16>(v);
				const float r1 = v - static_cast<float>(out[0][e]);
				out[1][e] = static_cast<__bf16>(r1);
				out[2][e] = static_cast<__bf16>(r1 - static_cast<float>(out[1][e]));
			}
			static __device__ __forceinline__ floatx16 multiply(frag a, frag b, floatx16 c)
			{
				return __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, b, c, 0, 0, 0);
			}
		};

		// Detail::ComputeALiBiSlope (FlashAttnExt.h:69-96), in double like the reference
		__device__ inline double row_alibi_slope(int head, int heads, double max_bias)
		{
			int head_log2 = 1;
			while ((head_log2 << 1) <= heads)
			{
				head_log2 <<= 1;
			}
			// (its powers of 2 to a power are one power of 2)
			const int times = head < head_log2 ? 2 * (head + 1) : 2 * (head - head_log2) + 1;
			return exp2(-(max_bias / 2.0) / static_cast<double>(head_log2) * static_cast<double>(times));
		}

		// exp(x) for x at most 0, or NaN: the product's rounding is put back behind the power of two, which below 2^-126 is 0.
		// Seven instructions where expf, which reduces its range and looks for its ends, takes thirteen.
		__device__ __forceinline__ float exp_of_nonpositive(float x)
		{
			constexpr float kLog2e = 1.44269504088896341f, kLog2eRest = 1.925963033e-8f, kLn2 = 0.69314718055994531f;
			x = __builtin_elementwise_maximum(x, -256.0f); // (an infinity would leave no number; a NaN stays one)
			const float high = x * kLog2e;
			const float low = fmaf(x, kLog2eRest, fmaf(x, kLog2e, -high));
			const float p = __builtin_amdgcn_exp2f(high);
			return fmaf(p * low, kLn2, p);
		}

		// Rows of keys lie 16 bytes further apart in LDS than they are long, rows of values 64, which spreads a piece of each of 16
		// keys, and 64 bytes of each of four values, over all 64 banks.  (Pieces permuted by their row want a register for each
		// place that is read: 31 of them spilled.)
		template <int D>
		constexpr int key_stride() { return 2 * D + 16; }
		template <int D>
		constexpr int value_stride() { return 2 * D + 64; }
		// A wavefront that shares its Float32 tiles with nobody puts the values where the keys were: four of them fit a CU's LDS
		template <typename O, int QW>
		constexpr bool one_buffer() { return O::kStored > 1 && QW == 1; }
		template <typename O, int D, int QW>
		constexpr int group_bytes() { return O::kStored * kKeys * (one_buffer<O, QW>() ? value_stride<D>() : key_stride<D>() + value_stride<D>()); }

		// The second half of the queries waits in LDS where every wavefront has the same ones and registers are short: behind all
		// buffers, or, where that keeps a second workgroup of four wavefronts off the CU (83968 bytes, and 75776 without), in the 64
		// bytes that set one row of values apart from the next.  (1000 rows on 1000 keys 67 and 49 us.)
		template <typename O, int D, int QW>
		constexpr bool queries_in_lds() { return O::kSplit == 2 && QW == 1 && D == 128; }
		template <typename O, int D, int QW, int KW>
		constexpr bool queries_between_values() { return queries_in_lds<O, D, QW>() && KW == 4; }

		// A workgroup takes 32 QW query rows of one head; its KW groups of QW wavefronts take the key tiles in turn,
		// each group with its own buffers, and merge at the end.
		template <typename O, int D, int QW, int KW>
		__global__ __launch_bounds__(64 * QW * KW, O::kStored == 1 ? 2 : 1) void attn_rows_kernel(const RowsAttn a)
		{
			typedef typename O::frag frag;
			typedef typename O::stored stored;
			constexpr int kKeyStride = key_stride<D>(), kValueStride = value_stride<D>();
			constexpr int kKeyBytes = kKeys * kKeyStride, kValueBytes = kKeys * kValueStride; // of one part of a tile
			constexpr bool kOneBuffer = one_buffer<O, QW>();
			constexpr int kGroupBytes = group_bytes<O, D, QW>();
			constexpr bool kQueriesInLds = queries_in_lds<O, D, QW>(), kQueriesBetween = queries_between_values<O, D, QW, KW>();
			extern __shared__ __attribute__((aligned(16))) uint8_t lds[]; // [KW][keys, values], queries; later the groups' results
			const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
			const int group = wave / QW, qw = wave % QW;
			const int tid = qw * 64 + lane; // within the group
			const int j = lane & 31, h = lane >> 5;
			// heads are dealt to the XCDs in runs, so that the query heads of one key/value head share an L2
			const int head = (a.heads & 7) == 0 ? static_cast<int>(blockIdx.x & 7) * (a.heads >> 3) + static_cast<int>(blockIdx.x >> 3)
			                                    : static_cast<int>(blockIdx.x);
			const int kv_head = head / a.share;
			const int q_first = (static_cast<int>(gridDim.y) - 1 - static_cast<int>(blockIdx.y)) * (32 * QW); // long runs first
			const int keys = a.keys;
			const long long q_at = a.q_at; // key index of query row 0's own position
			const int row = q_first + 32 * qw + j, row_c = min(row, a.rows - 1);
			// keys [lo, hi) a query sees; [first, last) any of the workgroup's
			const auto sees_from = [&](int i) { return static_cast<int>(max(0ll, q_at + i - a.window + 1)); };
			const auto sees_to = [&](int i) { return a.causal ? static_cast<int>(min(static_cast<long long>(keys), q_at + i + 1)) : keys; };
			const int lo = sees_from(row_c), hi = sees_to(row_c);
			// keys that all of the wavefront's queries see
			const int wave_lo = sees_from(min(q_first + 32 * qw + 31, a.rows - 1)), wave_hi = sees_to(min(q_first + 32 * qw, a.rows - 1));
			const int first = sees_from(q_first), last = sees_to(min(q_first + 32 * QW, a.rows) - 1);
			const int tiles = (last - first + kKeys - 1) / kKeys;
			const int steps = (tiles + KW - 1) / KW;

			const stored* const kb = static_cast<const stored*>(a.k) + kv_head * a.k_head;
			const stored* const vb = static_cast<const stored*>(a.v) + kv_head * a.v_head;
			const auto buffer_row = [&](int key) {
				key += a.ring_first;
				return a.ring > 0 && key >= a.ring ? key - a.ring : key;
			};

			// ---- the wavefront's queries: B operand of the first product, times 2^shift
			frag q[D / 16][O::kSplit];
			float unscale = 1.0f;
			floatx4 raw[D / 8]; // asked for ahead of the first tile's keys and values
			{
				// (whole groups of eight; one behind the head's last loads the first again and is dropped: the loads must not
				// hang on branches, or each waits for the one before)
				const float* src = a.q + static_cast<size_t>(row_c) * a.ldq + static_cast<size_t>(head) * a.dim;
#pragma unroll
				for (int s = 0; s < D / 16; ++s)
				{
					const int d = 16 * s + 8 * h;
					const floatx4_a4* at = reinterpret_cast<const floatx4_a4*>(src + (d < a.dim ? d : 0));
					raw[2 * s] = at[0], raw[2 * s + 1] = at[1];
				}
			}
			// ---- staging: a thread moves 8-element pieces of rows
			uint8_t* const k_lds = lds + group * kGroupBytes;
			uint8_t* const v_lds = kOneBuffer ? k_lds : k_lds + O::kStored * kKeyBytes;
			constexpr int kRowPieces = D / 8, kPieces = kKeys * kRowPieces / (64 * QW), kRowStep = 64 * QW / kRowPieces;
			static_assert(kPieces * 64 * QW == kKeys * kRowPieces && kRowStep * kRowPieces == 64 * QW, "pieces per thread");
			constexpr int kWords = sizeof(stored) / 2; // 16-byte words of a piece
			const int piece_row = tid / kRowPieces, piece = tid % kRowPieces; // first row, and the same column in all of them
			u32x4 kr[kPieces][kWords], vr[kPieces][kWords];
			const uint32_t ldk = static_cast<uint32_t>(a.ldk), ldv = static_cast<uint32_t>(a.ldv);
			// (a piece behind the head's last loads the first again and goes nowhere)
			const uint32_t k_off = static_cast<uint32_t>(piece_row) * ldk + (8 * piece < a.dim ? 8 * piece : 0);
			const uint32_t v_off = static_cast<uint32_t>(piece_row) * ldv + (8 * piece < a.vdim ? 8 * piece : 0);
			const auto request = [&](u32x4 (&into)[kPieces][kWords], const stored* from, uint32_t ld, uint32_t off, int tile) __attribute__((always_inline)) {
				// A whole tile that does not wrap lies at one distance from a uniform address; others go row by row
				const int key = first + tile * kKeys;
				const int at0 = buffer_row(key);
				if (key + kKeys <= last && (a.ring <= 0 || at0 + kKeys <= a.ring) && ld <= (1u << 26)) // (offsets of 32 bits)
				{
					const stored* const rows = from + static_cast<uint64_t>(static_cast<uint32_t>(at0)) * ld;
#pragma unroll
					for (int i = 0; i < kPieces; ++i)
					{
#pragma unroll
						for (int w = 0; w < kWords; ++w)
						{
							into[i][w] = *reinterpret_cast<const u32x4*>(rows + static_cast<uint64_t>(kRowStep * i) * ld + 4 * w + off);
						}
					}
					return;
				}
#pragma unroll
				for (int i = 0; i < kPieces; ++i)
				{
					const uint32_t at = buffer_row(min(key + piece_row + kRowStep * i, last - 1));
#pragma unroll
					for (int w = 0; w < kWords; ++w)
					{
						into[i][w] = *reinterpret_cast<const u32x4*>(from + static_cast<uint64_t>(at) * ld + 4 * w + (off - static_cast<uint32_t>(piece_row) * ld));
					}
				}
			};
			const auto store_piece = [&](uint8_t* dst, int part_bytes, const u32x4 (&v)[kWords]) __attribute__((always_inline)) {
				if constexpr (O::kStored == 1)
				{
					*reinterpret_cast<u32x4*>(dst) = v[0];
				}
				else
				{
					frag f[O::kStored];
#pragma unroll
					for (int e = 0; e < 8; ++e)
					{
						O::split(__uint_as_float(v[e / 4][e % 4]), e, f);
					}
#pragma unroll
					for (int p = 0; p < O::kStored; ++p)
					{
						*reinterpret_cast<frag*>(dst + p * part_bytes) = f[p];
					}
				}
			};
			const auto deposit = [&](u32x4 (&pieces)[kPieces][kWords], uint8_t* to, int stride, int part_bytes, int dim) __attribute__((always_inline)) {
				const bool there = 8 * piece < dim;
				if (kOneBuffer && !there) // (the buffer holds both in turn, and not in the same places)
				{
#pragma unroll
					for (int i = 0; i < kPieces; ++i)
					{
#pragma unroll
						for (int w = 0; w < kWords; ++w)
						{
							pieces[i][w] = u32x4{ 0u, 0u, 0u, 0u };
						}
					}
				}
				if (kOneBuffer || there)
				{
#pragma unroll
					for (int i = 0; i < kPieces; ++i)
					{
						store_piece(to + (piece_row + kRowStep * i) * stride + 16 * piece, part_bytes, pieces[i]);
					}
				}
			};
			const auto deposit_keys = [&]() { deposit(kr, k_lds, kKeyStride, kKeyBytes, a.dim); };
			const auto deposit_values = [&]() { deposit(vr, v_lds, kValueStride, kValueBytes, a.vdim); };
			if (!kOneBuffer && (a.dim < D || a.vdim < D)) // (uniform) pieces behind the head's last stay zero
			{
				for (int at = tid * 16; at < kGroupBytes; at += 64 * QW * 16)
				{
					*reinterpret_cast<u32x4*>(k_lds + at) = u32x4{ 0u, 0u, 0u, 0u };
				}
				if constexpr (QW > 1 || kQueriesBetween)
				{
					__syncthreads();
				}
			}
			const auto meet = [&]() {
				if constexpr (QW > 1)
				{
					__syncthreads();
				}
				else
				{
					__builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront"); // (a wavefront's LDS accesses keep their order)
					__builtin_amdgcn_wave_barrier();
				}
			};

			// Keys travel while the previous tile's values are used and go into LDS once its scores are formed, values the
			// other way round: one of the two is in registers at a time.
			const auto tile_at = [&](int step) { return min(step * KW + group, tiles - 1); };
			if (steps > 0)
			{
				request(kr, kb, ldk, k_off, tile_at(0));
				request(vr, vb, ldv, v_off, tile_at(0));
			}
			__builtin_amdgcn_sched_barrier(0); // (the first tile travels while the queries are taken apart)
			{
				if (a.dim < D) // (uniform)
				{
#pragma unroll
					for (int s = 0; s < D / 8; ++s)
					{
						raw[s] = 16 * (s >> 1) + 8 * h < a.dim ? raw[s] : floatx4{};
					}
				}
				float scale = 1.0f;
				if constexpr (O::kSplit == 2)
				{
					float mx = 0.0f;
#pragma unroll
					for (int s = 0; s < D / 8; ++s)
					{
						mx = fmaxf(mx, fmaxf(fmaxf(fabsf(raw[s].x), fabsf(raw[s].y)), fmaxf(fabsf(raw[s].z), fabsf(raw[s].w))));
					}
					if (__any(mx > 3.402823466e38f)) // (of the finite ones, then)
					{
						mx = 0.0f;
#pragma unroll
						for (int s = 0; s < D / 8; ++s)
						{
#pragma unroll
							for (int e = 0; e < 4; ++e)
							{
								const float m = fabsf(raw[s][e]);
								mx = m <= 3.402823466e38f ? fmaxf(mx, m) : mx;
							}
						}
					}
					mx = fmaxf(mx, __shfl_xor(mx, 32, 64));
					const int shift = mx > 0.0f ? min(14 - ilogbf(mx), 126) : 0;
					scale = ldexpf(1.0f, shift);
					unscale = ldexpf(1.0f, -shift);
				}
#pragma unroll
				for (int s = 0; s < D / 16; ++s)
				{
#pragma unroll
					for (int e = 0; e < 8; ++e)
					{
						O::split(raw[2 * s + e / 4][e & 3] * scale, e, q[s]);
					}
				}
			}
			uint8_t* const q_lds = kQueriesBetween ? lds + kKeyBytes + (lane >> 2) * kValueStride + 2 * D + 16 * (lane & 3) : lds + KW * kGroupBytes + 16 * lane;
			const auto q_step = [](int s) { return kQueriesBetween ? (s >> 1) * kGroupBytes + (s & 1) * 16 * kValueStride : 1024 * s; };
			if constexpr (kQueriesInLds)
			{
				static_assert(!kQueriesBetween || (kValueStride == 2 * D + 64 && D / 32 <= KW && kKeys == 32), "16 rows a step, two steps a group");
				if (group == 0)
				{
#pragma unroll
					for (int s = 0; s < D / 16; ++s)
					{
						*reinterpret_cast<frag*>(q_lds + q_step(s)) = q[s][1];
					}
				}
				__syncthreads();
			}
			const float slope = a.mask && a.max_bias > 0.0 ? static_cast<float>(row_alibi_slope(head, a.heads, a.max_bias)) : 1.0f;
			const float factor = a.apply_scale ? unscale * a.scale : unscale; // (a power of two and the scale: one rounding for both)
			const float* const mask_row = a.mask ? a.mask + static_cast<size_t>(row_c) * keys : nullptr;

			// a dot product's score (the causal mask and the window aside)
			const auto score_of = [&](float v, float mv) {
				if (a.apply_scale)
				{
					v = __fmul_rn(v, a.scale);
				}
				if (a.softcap != 0.0f)
				{
					v = capped_tanh(v);
					if (a.apply_cap)
					{
						v = __fmul_rn(v, a.softcap);
					}
				}
				if (a.mask)
				{
					v = __fadd_rn(v, __fmul_rn(mv, slope));
				}
				return v;
			};

			floatx16 o[D / 32];
#pragma unroll
			for (int b = 0; b < D / 32; ++b)
			{
				o[b] = floatx16{};
			}
			float run_m = -INFINITY, run_l = 0.0f; // run_l: of this lane's keys
			if (steps > 0)
			{
				deposit_keys();
			}
			for (int step = 0; step < steps; ++step)
			{
				const int tile = step * KW + group;
				const bool live = tile < tiles; // a group without a tile left goes through the motions on the last one
				const int base = first + min(tile, tiles - 1) * kKeys;
				// the tile's mask: four runs of four keys (at the mask's end the last whole run there is, shifted below)
				float mask[16];
				if (a.mask)
				{
#pragma unroll
					for (int e = 0; e < 16; e += 4)
					{
						const int key = base + 2 * e + 4 * h, from = max(0, min(key, keys - 4));
						const floatx4 x = *reinterpret_cast<const floatx4_a4*>(mask_row + from);
#pragma unroll
						for (int i = 0; i < 4; ++i)
						{
							mask[e + i] = x[i];
						}
						if (base + kKeys > keys)
						{
#pragma unroll
							for (int i = 0; i < 3; ++i)
							{
								const bool shifted = key - from > i;
								mask[e] = shifted ? mask[e + 1] : mask[e];
								mask[e + 1] = shifted ? mask[e + 2] : mask[e + 1];
								mask[e + 2] = shifted ? mask[e + 3] : mask[e + 2];
							}
						}
					}
				}
				meet(); // the tile's keys are there, the previous tile's values have been used
				floatx16 s = {}, s_odd = {}, s_low = {}; // the parts' small products apart: every addition to a large sum rounds
#pragma unroll
				for (int st = 0; st < D / 16; ++st)
				{
#pragma unroll
					for (int p = 0; p < O::kProducts; ++p)
					{
						const frag kf = *reinterpret_cast<const frag*>(k_lds + O::stored_of[p] * kKeyBytes + j * kKeyStride + 16 * (2 * st + h));
						floatx16& to = p > 0 ? s_low : st % 2 == 0 ? s : s_odd;
						if constexpr (kQueriesInLds)
						{
							to = O::multiply(kf, p == 0 ? q[st][0] : *reinterpret_cast<const frag*>(q_lds + q_step(st)), to);
						}
						else
						{
							to = O::multiply(kf, q[st][O::split_of[p]], to);
						}
					}
				}
				deposit_values();
				request(kr, kb, ldk, k_off, tile_at(step + 1));
				// lane (j, h) holds keys base + 8 (e / 4) + 4 h + e % 4 of query j
				float sc[16];
				float top = -INFINITY;
#pragma unroll
				for (int e = 0; e < 16; ++e)
				{
					sc[e] = fmaf(s_low[e], O::kLowScale, s[e] + s_odd[e]) * factor;
				}
				// (an option at a time over all sixteen: a branch for each score's options was a tenth of the tile)
				if (a.softcap != 0.0f)
				{
					// Capped scores are a small part of the cap as a rule: the series takes seven instructions, the layer's form 35 more
					// where a lane of the wavefront has a score that wants it (the call above with caps of 30 and 4: 34 and 39 us,
					// with Float32 keys and a cap of 0.5 107; error against 64 bits 1.3e-7 where the layer's form alone has 3.7e-7).
					float most = 0.0f;
#pragma unroll
					for (int e = 0; e < 16; ++e)
					{
						most = fmaxf(most, fabsf(sc[e])); // (a NaN stays one in either form)
					}
					if (__all(most <= kSmallTangent))
					{
#pragma unroll
						for (int e = 0; e < 16; ++e)
						{
							sc[e] = small_tanh(sc[e]);
						}
					}
					else
					{
#pragma unroll
						for (int e = 0; e < 16; ++e)
						{
							const float near = small_tanh(sc[e]);
							float far = layer_tanh(sc[e]);
							asm("" : "+v"(far)); // (a choice, not a branch for each score)
							sc[e] = fabsf(sc[e]) <= kSmallTangent ? near : far;
							if (e == 7)
							{
								__builtin_amdgcn_sched_barrier(0); // (sixteen at once want registers that spill)
							}
						}
					}
					if (a.apply_cap)
					{
#pragma unroll
						for (int e = 0; e < 16; ++e)
						{
							sc[e] = __fmul_rn(sc[e], a.softcap);
						}
					}
				}
				if (a.mask)
				{
#pragma unroll
					for (int e = 0; e < 16; ++e)
					{
						sc[e] = fmaf(mask[e], slope, sc[e]);
					}
				}
				if (!live || base < wave_lo || base + kKeys > wave_hi) // (a key that one of the wavefront's queries does not see)
				{
#pragma unroll
					for (int e = 0; e < 16; ++e)
					{
						const int key = base + 8 * (e / 4) + 4 * h + (e & 3);
						sc[e] = live && key >= lo && key < hi ? sc[e] : -INFINITY;
					}
				}
#pragma unroll
				for (int e = 0; e < 16; ++e)
				{
					top = fmaxf(top, sc[e]);
				}
				top = fmaxf(top, __shfl_xor(top, 32, 64));
				const float new_m = fmaxf(run_m, top);
				const float ref_m = new_m == -INFINITY ? 0.0f : new_m; // (no visible key yet: every exponent is -inf)
				const float corr = expf(run_m - ref_m);
				run_m = new_m;
				float sums[16];
				frag w[2][O::kSplit];
#pragma unroll
				for (int e = 0; e < 16; ++e)
				{
					const float p = exp_of_nonpositive(sc[e] - ref_m);
					sums[e] = p;
					O::split(p * O::kWeightScale, e & 7, w[e >> 3]);
				}
#pragma unroll
				for (int half = 8; half > 0; half /= 2)
				{
#pragma unroll
					for (int e = 0; e < half; ++e)
					{
						sums[e] += sums[e + half];
					}
				}
				run_l = fmaf(run_l, corr, sums[0]);
				// step u: keys 16 u + 4 h + 0..3 and 16 u + 8 + 4 h + 0..3.  Sixteen lanes read four keys' rows of
				// sixteen dimensions, eight bytes each, and get the four keys of one dimension
				meet(); // the tile's values are there, its keys have been used
				if constexpr (!kOneBuffer)
				{
					deposit_keys();
				}
				request(vr, vb, ldv, v_off, tile_at(step + 1));
				const int v_row = 4 * h + ((lane & 15) >> 2), v_col = ((lane >> 4) & 1) * 2 + ((lane & 3) >> 1), v_byte = (lane & 1) * 8;
#pragma unroll
				for (int b = 0; b < D / 32; ++b)
				{
					if constexpr (O::kSplit == 2)
					{
						__builtin_amdgcn_sched_barrier(0); // (one block of dimensions after the other: four at once are more than the registers hold)
					}
					// the tile's sum, the small products' first, added at once: the running sum rounds once per tile
					floatx16 t = {}, t_low = {};
					frag vf[2][O::kStored];
#pragma unroll
					for (int u = 0; u < 2; ++u)
					{
#pragma unroll
						for (int p = 0; p < O::kStored; ++p)
						{
							typedef __attribute__((address_space(3))) short4v* lds_short4;
							const uint8_t* const at = v_lds + p * kValueBytes + v_row * kValueStride + 16 * v_col + v_byte;
							const u32x2 x = __builtin_bit_cast(u32x2, __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_short4)(at + 16 * u * kValueStride + 64 * b)));
							const u32x2 y = __builtin_bit_cast(u32x2, __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_short4)(at + (16 * u + 8) * kValueStride + 64 * b)));
							vf[u][p] = __builtin_bit_cast(frag, u32x4{ x.x, x.y, y.x, y.y });
						}
#pragma unroll
						for (int p = O::kProducts - 1; p > 0; --p)
						{
							t_low = O::multiply(vf[u][O::stored_of[p]], w[u][O::split_of[p]], t_low);
						}
					}
					if constexpr (O::kSplit == 2)
					{
						t = t_low * O::kLowScale; // (and the large products go on top: no registers for two sums)
					}
#pragma unroll
					for (int u = 0; u < 2; ++u)
					{
						t = O::multiply(vf[u][0], w[u][0], t);
					}
					if constexpr (O::kSplit > 2)
					{
						t += t_low;
					}
#pragma unroll
					for (int e = 0; e < 16; ++e)
					{
						o[b][e] = fmaf(o[b][e], corr, t[e]);
					}
				}
				if constexpr (kOneBuffer)
				{
					meet();
					deposit_keys();
				}
			}
			run_l += __shfl_xor(run_l, 32, 64);

			// The groups hand (maximum, sum, outputs) over through LDS, and each takes a share of the dimensions: quads of them, as
			// they lie in o, group by group.  (One group that took all of them in turn: 1.2 us more of 39 with eight groups.)
			constexpr int kQuads = D / 8 / KW; // of this wavefront
			static_assert(kQuads * KW * 8 == D, "quads and groups");
			float r[kQuads][4];
			{
				float* const xch = reinterpret_cast<float*>(lds);
				constexpr int kWaveFloats = (D / 2 + 2) * 64; // of one wavefront: outputs, maximum, sum
				__syncthreads();
				float* const dst = xch + (group * QW + qw) * kWaveFloats;
#pragma unroll
				for (int b = 0; b < D / 32; ++b)
				{
#pragma unroll
					for (int e = 0; e < 16; e += 4)
					{
						*reinterpret_cast<float4*>(dst + ((b * 16 + e) / 4 * 64 + lane) * 4) = float4{ o[b][e], o[b][e + 1], o[b][e + 2], o[b][e + 3] };
					}
				}
				dst[D / 2 * 64 + lane] = run_m;
				dst[(D / 2 + 1) * 64 + lane] = run_l;
				__syncthreads();
				float m[KW], weight[KW];
#pragma unroll
				for (int i = 0; i < KW; ++i)
				{
					m[i] = xch[(i * QW + qw) * kWaveFloats + D / 2 * 64 + lane];
					run_m = i == 0 ? m[0] : fmaxf(run_m, m[i]);
				}
				const float ref_m = run_m == -INFINITY ? 0.0f : run_m;
#pragma unroll
				for (int i = 0; i < KW; ++i)
				{
					weight[i] = expf(m[i] - ref_m);
					const float l = xch[(i * QW + qw) * kWaveFloats + (D / 2 + 1) * 64 + lane] * weight[i];
					run_l = i == 0 ? l : run_l + l;
				}
#pragma unroll
				for (int i = 0; i < KW; ++i)
				{
#pragma unroll
					for (int n = 0; n < kQuads; ++n)
					{
						const float4 t = *reinterpret_cast<const float4*>(xch + (i * QW + qw) * kWaveFloats + ((group * kQuads + n) * 64 + lane) * 4);
						r[n][0] = i == 0 ? t.x * weight[0] : fmaf(t.x, weight[i], r[n][0]);
						r[n][1] = i == 0 ? t.y * weight[0] : fmaf(t.y, weight[i], r[n][1]);
						r[n][2] = i == 0 ? t.z * weight[0] : fmaf(t.z, weight[i], r[n][2]);
						r[n][3] = i == 0 ? t.w * weight[0] : fmaf(t.w, weight[i], r[n][3]);
					}
				}
			}
			// the first of the quad's dimensions
			const auto dim_of = [&](int n) {
				const int quad = group * kQuads + n;
				return 32 * (quad >> 2) + 8 * (quad & 3) + 4 * h;
			};
			if (row >= a.rows)
			{
				return;
			}
			// An infinity or a NaN reaches every query of a tile through a weight of zero, or comes out of an operand that
			// was taken apart.  A query whose result is not finite is computed again, key by key over its own keys alone,
			// so that it gets what Float32 arithmetic gives it.
			bool finite = fabsf(run_l) <= 3.402823466e38f;
#pragma unroll
			for (int n = 0; n < kQuads; ++n)
			{
#pragma unroll
				for (int i = 0; i < 4; ++i)
				{
					finite = finite && fabsf(r[n][i]) <= 3.402823466e38f;
				}
			}
			if (__builtin_expect(!finite, 0))
			{
				const auto widen = [](stored v) {
					if constexpr (O::kStored == 1)
					{
						return f16_bits_to_f32(v);
					}
					else
					{
						return v;
					}
				};
				const float* src = a.q + static_cast<size_t>(row) * a.ldq + static_cast<size_t>(head) * a.dim;
				run_m = -INFINITY;
				run_l = 0.0f;
#pragma unroll
				for (int n = 0; n < kQuads; ++n)
				{
#pragma unroll
					for (int i = 0; i < 4; ++i)
					{
						r[n][i] = 0.0f;
					}
				}
				for (int key = lo; key < hi; ++key)
				{
					const stored* kr0 = kb + static_cast<size_t>(buffer_row(key)) * a.ldk;
					const stored* vr0 = vb + static_cast<size_t>(buffer_row(key)) * a.ldv;
					float dot = 0.0f;
					for (int d = 0; d < a.dim; ++d)
					{
						dot = fmaf(src[d], widen(kr0[d]), dot);
					}
					const float v = score_of(dot, a.mask ? mask_row[key] : 0.0f);
					const float new_m = fmaxf(run_m, v), ref_m = new_m == -INFINITY ? 0.0f : new_m;
					const float corr = expf(run_m - ref_m), p = expf(v - ref_m);
					run_m = new_m;
					run_l = fmaf(run_l, corr, p);
#pragma unroll
					for (int n = 0; n < kQuads; ++n)
					{
#pragma unroll
						for (int i = 0; i < 4; ++i)
						{
							const int d = dim_of(n) + i;
							r[n][i] = fmaf(p * O::kWeightScale, d < a.vdim ? widen(vr0[d]) : 0.0f, r[n][i] * corr);
						}
					}
				}
			}
			float weight = 1.0f, total = run_l;
			if (a.sinks)
			{
				// the sink joins the row maximum and the denominator, not the values (FlashAttnExt.h:184-212)
				const float sink = a.sinks[head];
				const float all_m = fmaxf(run_m, sink);
				weight = expf(run_m - all_m);
				total = run_l * weight + expf(sink - all_m);
			}
			const float inv = weight / total * (a.out_scale / O::kWeightScale);
			float* const out = a.out + static_cast<size_t>(row) * a.ldo + static_cast<size_t>(head) * a.vdim;
			const float* const gate = a.gate ? a.gate + static_cast<size_t>(row) * a.ldg + static_cast<size_t>(head) * a.vdim : nullptr;
#pragma unroll
			for (int n = 0; n < kQuads; ++n)
			{
				const int d = dim_of(n);
				if (d < a.vdim) // (whole groups of eight)
				{
					float4 v = { r[n][0] * inv, r[n][1] * inv, r[n][2] * inv, r[n][3] * inv };
					if (gate)
					{
						v.x *= sigmoid_f32(gate[d]);
						v.y *= sigmoid_f32(gate[d + 1]);
						v.z *= sigmoid_f32(gate[d + 2]);
						v.w *= sigmoid_f32(gate[d + 3]);
					}
					*reinterpret_cast<float4*>(out + d) = v;
				}
			}
		}

		template <typename O, int D, int QW, int KW>
		void launch_form(const RowsAttn& a, hipStream_t s)
		{
			constexpr size_t tiles = static_cast<size_t>(KW) * group_bytes<O, D, QW>() + (queries_in_lds<O, D, QW>() && !queries_between_values<O, D, QW, KW>() ? 64 * D : 0);
			constexpr size_t merge = static_cast<size_t>(KW) * QW * (D / 2 + 2) * 64 * sizeof(float);
			constexpr size_t lds = tiles > merge ? tiles : merge;
			static_assert(lds <= 160 * 1024, "LDS");
			static_assert(O::kStored > 1 || KW > 4 || 2 * lds <= 160 * 1024, "two workgroups of four wavefronts a CU");
			allow_dynamic_lds(reinterpret_cast<const void*>(&attn_rows_kernel<O, D, QW, KW>), lds);
			attn_rows_kernel<O, D, QW, KW><<<dim3(a.heads, (a.rows + 32 * QW - 1) / (32 * QW)), dim3(64 * QW * KW), lds, s>>>(a);
		}

		template <int D>
		void launch_dim(const RowsAttn& a, bool f32, hipStream_t s)
		{
			if (f32)
			{
				if (fetch::rows_float_alone({ a.rows, a.keys, a.causal, a.q_at, a.window }, a.heads, D))
				{
					launch_form<FloatOperands, D, 1, 4>(a, s);
				}
				else
				{
					launch_form<FloatOperands, D, 2, 2>(a, s);
				}
			}
			else
			{
				const size_t groups = static_cast<size_t>(a.heads) * ((a.rows + 31) / 32);
				// Eight wavefronts on a head's rows, one workgroup to a CU, while all of them fit the 256 CUs at once and have more than
				// a tile or two each; four, two workgroups to a CU, for few keys and for many rows (us of eight and four, 32 heads over
				// 8, rows on keys: 200 on 1000 24 and 27, 16 on 2000 31 and 43, 128 on 400 17.3 and 18.1, on 300 17.3 and 15.9, on 128
				// 13.8 and 10.6, 512 on 512 29 and 20, on 1024 41 and 32, 1000 on 2000 121 and 98, 1500 on 4000 306 and 272; heads of 64,
				// 300 on 1000 26 and 19, 1000 on 4000 136 and 120).
				if (groups <= 256 && a.keys >= 384)
				{
					launch_form<HalfOperands, D, 1, 8>(a, s);
				}
				else
				{
					launch_form<HalfOperands, D, 1, 4>(a, s);
				}
			}
		}
	} // namespace

	// Causal attention of m rows at positions past .. past + m - 1 (operands as in launch_attn_decode)
	bool launch_attn_rows_causal(const float* q, const void* kcache, const void* vcache, int cache_dtype, size_t m,
	                             size_t past, size_t n_head, size_t n_kv_head, size_t head_dim, float* out, hipStream_t s)
	{
		if (!attn_rows_pay_causal(m, past + m, cache_dtype == LITENN_F32) || m > 0x3fffffffu || n_head > 65535 || past + m > 0x3fffffffu)
		{
			return false;
		}
		RowsAttn a;
		a.q = q;
		a.ldq = a.ldo = n_head * head_dim;
		a.k = kcache;
		a.v = vcache;
		a.ldk = a.ldv = n_kv_head * head_dim;
		a.k_head = a.v_head = head_dim;
		a.heads = static_cast<int>(n_head);
		a.share = static_cast<int>(n_head / n_kv_head);
		a.dim = a.vdim = static_cast<int>(head_dim);
		a.rows = static_cast<int>(m);
		a.q_at = static_cast<long long>(past);
		a.keys = static_cast<int>(a.q_at) + a.rows;
		a.apply_scale = true;
		a.scale = static_cast<float>(1.0 / sqrt(static_cast<double>(head_dim)));
		a.out = out;
		return launch_attn_rows(a, cache_dtype == LITENN_F32, s);
	}

	bool launch_attn_rows(const RowsAttn& a, bool f32, hipStream_t s)
	{
		const auto aligned = [](const void* p) { return (reinterpret_cast<uintptr_t>(p) & 15u) == 0; };
		const int piece = f32 ? 4 : 8; // elements of 16 bytes
		if (a.rows <= 0 || a.heads <= 0 || a.dim % 8 != 0 || a.vdim % 8 != 0 || a.dim <= 0 || a.vdim <= 0 || a.dim > 128 || a.vdim > 128 ||
		    a.ldk % piece != 0 || a.ldv % piece != 0 || a.k_head % piece != 0 || a.v_head % piece != 0 || a.ldo % 4 != 0 ||
		    a.ldk > 0xffffffffu || a.ldv > 0xffffffffu || (a.mask && a.keys < 4) || !aligned(a.k) || !aligned(a.v) || !aligned(a.out) || (a.rows + 31) / 32 > 65535)
		{
			return false;
		}
		if (a.dim <= 64 && a.vdim <= 64)
		{
			launch_dim<64>(a, f32, s);
		}
		else
		{
			launch_dim<128>(a, f32, s);
		}
		return true;
	}
} // namespace litenn_hip
