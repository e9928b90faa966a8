import sys, os, statistics, dataclasses, json
sys.path.insert(0, os.getcwd())
import torch
from xllm_service_amd.engine.metadata import AttnMetadata
from xllm_service_amd.models.config import get_config
from xllm_service_amd.models.llama import LlamaForCausalLM
dev='cuda'; res={}
def i32(v): return torch.tensor(v, dtype=torch.int32, device=dev)
def meta_of(prompts, decodes, cfg, L):
    P=len(prompts); n=P+len(decodes); pages=(2048+512)//16
    tables=torch.arange(n*pages,device=dev,dtype=torch.int32).view(n,pages)
    pos=[p for k in prompts for p in range(k)]+list(decodes)
    seq=[i for i,k in enumerate(prompts) for _ in range(k)]+list(range(P,n))
    slots=torch.tensor([s*pages*16+p for s,p in zip(seq,pos)],device=dev)
    cu=[0]
    for k in prompts: cu.append(cu[-1]+k)
    m=AttnMetadata(num_prefill_tokens=cu[-1],num_decode_tokens=len(decodes),slot_mapping=slots,
        cu_q=i32(cu) if P else None,prefill_seq_lens=i32(prompts) if P else None,prefill_block_tables=tables[:P].contiguous() if P else None,
        decode_seq_lens=i32([d+1 for d in decodes]) if decodes else None,decode_block_tables=tables[P:].contiguous() if decodes else None)
    return m,torch.tensor(pos,device=dev),n*pages
for name,bias in (('llama-2k',0),('llama-4k',0)):
    cfg=dataclasses.replace(get_config(name),num_layers=4,vocab_size=1024)
    torch.manual_seed(0)
    with torch.device(dev):
        model=LlamaForCausalLM(cfg,torch.bfloat16)
    model.random_init(0)
    if bias:
        for l in model.layers:
            l.attn.qkv_proj.bias=torch.nn.Parameter(torch.randn(l.attn.qkv_proj.weight.shape[0],device=dev).bfloat16()*.1)
    for tag,prompts,decodes in [(f'd{m}',[],[700]*m) for m in (1,4,8,12,16,24,32,48,64)]+[(f'p{t}',[t],[]) for t in (16,40,64,200)]:
        m,pos,np_=meta_of(prompts,decodes,cfg,4)
        caches=[tuple(torch.randn(np_,cfg.num_kv_heads,16,cfg.head_dim,device=dev).bfloat16() for _ in 'kv') for _ in range(4)]
        ids=torch.randint(0,1024,(len(pos),),device=dev)
        with torch.inference_mode():
            for _ in range(2): model(ids,pos,caches,m)
            torch.cuda.synchronize()
            g=torch.cuda.CUDAGraph()
            with torch.cuda.graph(g): model(ids,pos,caches,m)
            for _ in range(3): g.replay()
            torch.cuda.synchronize(); ts=[]
            for _ in range(15):
                a,b=torch.cuda.Event(True),torch.cuda.Event(True); a.record(); g.replay(); b.record(); torch.cuda.synchronize(); ts.append(a.elapsed_time(b)*1e3)
        res[f'{name} {tag}']=statistics.median(ts)
        del caches,g
    del model; torch.cuda.empty_cache(); print(name,flush=True)
json.dump(res,open(sys.argv[1],'w'))
